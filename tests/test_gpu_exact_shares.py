"""The exact batches' splits of the work: plain with 16, 4 and 1 lanes per query, split and FP64 with
the triangles shared out over blocks, at the edges of tiles, groups and blocks, and at coordinates near
the ends of the float range."""

import numpy as np
import pytest

from smallgwn_amd import synth
from tests.test_gpu_build import build_gpu

pytestmark = pytest.mark.gpu


def _first(mesh, n):
    return synth.Mesh(mesh.vx, mesh.vy, mesh.vz, mesh.i0[:n].copy(), mesh.i1[:n].copy(), mesh.i2[:n].copy())


def _run(gwn, dev, bvh, q, precision=None):
    import torch

    d = [torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in q]
    out = torch.full((q[0].shape[0],), 7.0, dtype=torch.float32 if precision is None else torch.float64, device=dev)
    if precision is None:
        gwn.gwn_compute_winding_number_exact_batch(bvh, *d, out).raise_if_error()
    else:
        gwn.gwn_compute_winding_number_exact_batch_ex(bvh, *d, out, precision).raise_if_error()
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("tris", [1, 15, 17, 255, 256, 257, 1000, 4097])
@pytest.mark.parametrize("queries", [1, 255, 257, 3001])
def test_exact_edges_match_oracle(gwn, orc, dev, tris, queries):
    mesh = _first(synth.displaced_sphere(64, 40), tris)
    _, bvh = build_gpu(gwn, mesh)
    q = synth.uniform_box_points(tris + queries, queries, (-1.5,) * 3, (1.5,) * 3)
    ref64 = orc.winding_exact_mesh_f64(mesh, *q)
    # The reference's float GPU-vs-CPU tolerance, and a tenth of it for FP64 near terms and sums.
    tol = 2e-5 + 2e-5 * np.abs(ref64)
    assert np.all(np.abs(_run(gwn, dev, bvh, q) - ref64) <= tol)
    assert np.all(np.abs(_run(gwn, dev, bvh, q, gwn.Precision.SPLIT) - ref64) <= 0.1 * tol)
    assert np.abs(_run(gwn, dev, bvh, q, gwn.Precision.FP64) - ref64).max() <= 1e-12


def test_exact_plain_is_one_ordered_sum_for_every_batch_size(gwn, dev):
    """16, 4 and 1 lanes per query add the same angles in the same order."""
    mesh = _first(synth.displaced_sphere(64, 40), 1003)
    _, bvh = build_gpu(gwn, mesh)
    q = synth.uniform_box_points(5, 530000, (-1.5,) * 3, (1.5,) * 3)
    want = _run(gwn, dev, bvh, q)
    for n in (700, 131073):
        got = _run(gwn, dev, bvh, [a[:n] for a in q])
        assert np.array_equal(got.view(np.uint32), want[:n].view(np.uint32)), n


@pytest.mark.parametrize("scale", [2.0 ** -45, 2.0 ** -42, 2.0 ** 40])
def test_exact_split_at_the_ends_of_the_float_range(gwn, orc, dev, scale):
    """Denominators (four cubed lengths) that leave the reciprocal's range but not the float range go
    through the arctangent: a power-of-two scale of mesh and queries changes no winding number."""
    base = _first(synth.displaced_sphere(32, 20), 700)
    mesh = synth.Mesh(*(a * np.float32(scale) for a in (base.vx, base.vy, base.vz)), base.i0, base.i1, base.i2)
    _, bvh = build_gpu(gwn, mesh)
    q = [a * np.float32(scale) for a in synth.uniform_box_points(3, 1000, (-1.5,) * 3, (1.5,) * 3)]
    ref64 = orc.winding_exact_mesh_f64(mesh, *q)
    # Far triangles lie at least 0.8 scale away, so a denominator is 2.1 (0.8 scale)^3 at least, and the products
    # of its numerator round to subnormals of 2^-149: at 2^-45 that is 3 2^-150 / 1.1 2^-135 = 8.5e-5 of half an angle a
    # triangle, 3.6e-4 of W for 700 of them with errors of both signs.  At 2^-42 it is 512 times less, and the usual
    # bound holds.
    err = np.abs(_run(gwn, dev, bvh, q, gwn.Precision.SPLIT) - ref64)
    assert np.all(err <= (2e-6 + 2e-6 * np.abs(ref64) if scale >= 2.0 ** -42 else 4e-4))


def test_exact_batch_under_capture(gwn, dev):
    """Captured, the split batch stays one launch; its replays equal the eager batch to FP64 rounding."""
    import torch

    mesh = synth.displaced_sphere(32, 20)
    _, bvh = build_gpu(gwn, mesh)
    d = [torch.from_numpy(a).to(dev) for a in synth.uniform_box_points(3, 1000, (-1.5,) * 3, (1.5,) * 3)]
    eager = torch.zeros(1000, dtype=torch.float64, device=dev)
    gwn.gwn_compute_winding_number_exact_batch_ex(bvh, *d, eager, gwn.Precision.SPLIT).raise_if_error()
    torch.cuda.synchronize()
    out = torch.zeros_like(eager)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gwn.gwn_compute_winding_number_exact_batch_ex(bvh, *d, out, gwn.Precision.SPLIT).raise_if_error()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.allclose(out, eager, rtol=1e-12, atol=1e-12)
