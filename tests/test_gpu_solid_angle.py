"""The plain solid angle's shortened square roots, quotients and arctangent against the general ones: one
triangle at sizes inside and outside the range they are used in, against FP64."""

import ctypes
import os

import numpy as np
import pytest

from smallgwn_amd import synth
from tests.test_gpu_build import build_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [2.0 ** -60, 2.0 ** -50, 2.0 ** -47, 1.0, 2.0 ** 46, 2.0 ** 49, 2.0 ** 60])
def test_plain_angle_in_and_out_of_the_usual_range(gwn, orc, dev, scale):
    """Squared lengths from 2^-120 to 2^120: the shortened forms serve 2^-96 to 2^96."""
    import torch

    v = np.array([[0.3, -0.2, 0.1], [1.0, 0.1, -0.3], [-0.2, 0.9, 0.4]], np.float32) * np.float32(scale)
    mesh = synth.Mesh(*(np.ascontiguousarray(v[:, k]) for k in range(3)), *(np.array([k], np.uint32) for k in range(3)))
    _, bvh = build_gpu(gwn, mesh)
    q = [a * np.float32(scale) for a in synth.uniform_box_points(9, 4096, (-1.5,) * 3, (1.5,) * 3)]
    out = torch.empty(4096, dtype=torch.float32, device=dev)
    gwn.gwn_compute_winding_number_exact_batch(bvh, *[torch.from_numpy(a).to(dev) for a in q], out).raise_if_error()
    ref = orc.winding_exact_mesh_f64(mesh, *q)
    # The angle is twice the arctangent of num / den.  Both are sums of six products of unit corners, 12 roundings of
    # at most 2^-24 in all, over their distance from zero; the arctangent adds 4 ulps of at most pi.
    corner = [(v[k].astype(np.float64) - np.stack(q, 1)) for k in range(3)]
    a, b, c = (u / np.linalg.norm(u, axis=1, keepdims=True) for u in corner)
    num = (a * np.cross(b - a, c - a)).sum(1)
    den = 1.0 + (a * b).sum(1) + (a * c).sum(1) + (b * c).sum(1)
    tol = (2 * 12 * 2.0 ** -24 / np.hypot(num, den) + 2 * 4 * 2.0 ** -22) / (4 * np.pi)
    got = out.cpu().numpy()
    assert np.all(np.abs(got - ref) <= tol)
    # A power of two changes no operation of either form (without subnormal squares), so both give the same bits.
    if scale < 2.0 ** -47:
        return
    _, unit = build_gpu(gwn, synth.Mesh(*(a / np.float32(scale) for a in (mesh.vx, mesh.vy, mesh.vz)), mesh.i0, mesh.i1, mesh.i2))
    one = torch.empty_like(out)
    gwn.gwn_compute_winding_number_exact_batch(unit, *[torch.from_numpy(a / np.float32(scale)).to(dev) for a in q], one).raise_if_error()
    assert torch.equal(out, one)


def test_plain_angle_on_the_triangle(gwn, dev):
    """At a vertex the angle is zero by definition, in the plane outside it zero, non-finite points give NaN."""
    import torch

    mesh = synth.Mesh(*(np.array(a, np.float32) for a in ([0, 1, 0], [0, 0, 1], [0, 0, 0])),
                      *(np.array([k], np.uint32) for k in range(3)))
    _, bvh = build_gpu(gwn, mesh)
    q = [np.array(a, np.float32) for a in ([0, 1, 3, np.nan, 0], [0, 0, 0, 0, np.inf], [0, 0, 0, 1, 0])]
    out = torch.empty(5, dtype=torch.float32, device=dev)
    gwn.gwn_compute_winding_number_exact_batch(bvh, *[torch.from_numpy(a).to(dev) for a in q], out).raise_if_error()
    w = out.cpu().numpy()
    assert w[0] == 0 and w[1] == 0 and w[2] == 0 and np.isnan(w[3]) and np.isnan(w[4])


@pytest.fixture(scope="module")
def angle(gwn):
    so = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "libgwn_point_api.so")
    if not os.path.exists(so):
        pytest.fail(f"{so} is not built (tests/cpp/build.py)")
    fn = ctypes.CDLL(so).gwn_angle_run
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_void_p] * 4 + [ctypes.c_uint64, ctypes.c_void_p, ctypes.c_void_p]
    return fn


def _spread(r, n, low, high):
    return (r.choice([-1.0, 1.0], n) * 2.0 ** r.uniform(low, high, n)).astype(np.float32)


def test_arctangent_to_four_ulps(angle, dev):
    """|t| <= 1 by a reciprocal of 1 ulp and a product, a fit of 2.1e-8 of the arctangent, the last operation of the
    polynomial and one of pi's differences: below 4 ulps in all, in every octant and over the whole range."""
    import torch

    r = np.random.default_rng(8)
    n = 1 << 22
    for low, high, near in ((-100, 100, False), (-3, 3, False), (0, 1, True)):
        x = _spread(r, n, low, high)
        y = (x * r.uniform(0.9, 1.1, n)).astype(np.float32) if near else _spread(r, n, low, high)
        dx, dy, out = torch.from_numpy(x).to(dev), torch.from_numpy(y).to(dev), torch.empty(n, device=dev)
        assert angle(None, dx.data_ptr(), dy.data_ptr(), None, n, out.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
        want = np.arctan2(y.astype(np.float64), x.astype(np.float64))
        usual = np.abs(want) > 2.0 ** -120
        off = np.abs(out.cpu().numpy().astype(np.float64) - want) / np.spacing(np.abs(want).astype(np.float32))
        assert off[usual].max() <= 4.0, (low, high, off[usual].max())


def test_normalisation_is_correctly_rounded(angle, dev):
    """The square root and the quotients equal the correctly rounded ones bit for bit, for squared lengths of the
    whole range that the form is used in and components down to 2^-100 of the length."""
    import torch

    r = np.random.default_rng(9)
    n = 1 << 22
    ss = (2.0 ** r.uniform(-96, 96, n)).astype(np.float32)
    length = np.sqrt(ss)
    v = [(length * (r.uniform(-1, 1, n) if k < 2 else _spread(r, n, -26, 0))).astype(np.float32) for k in range(3)]
    d = [torch.from_numpy(a).to(dev) for a in (ss, *v)]
    assert angle(*(t.data_ptr() for t in d), n, None, torch.cuda.current_stream().cuda_stream) == 0
    for a, t in zip(v, d[1:]):
        assert np.array_equal(t.cpu().numpy().view(np.uint32), (a / length).view(np.uint32))
