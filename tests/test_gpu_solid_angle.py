"""The plain solid angle's shortened square roots, quotients and arctangent against the general ones: one
triangle at sizes inside and outside the range they are used in, against FP64."""

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
    # Unit corners to 1 ulp each, six products of them in the numerator and denominator: the angle's error is
    # below 32 ulps over the (here at least 0.02) distance of the corners from cancelling, over 2 pi.
    assert np.abs(out.cpu().numpy() - ref).max() <= 32 * 2.0 ** -24 / 0.02 / (2 * np.pi)


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
