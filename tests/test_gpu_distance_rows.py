"""The row (16 lanes per point) and quad (4 lanes, points handed out within a wave) distance traversals
against the one-lane kernel: distances and nearest records equal bit for bit on both sides of the size
that chooses between them, with ties, axis-aligned faces, bands and non-finite points."""

import numpy as np
import pytest

from smallgwn_amd import synth
from tests.helpers import nested_octants
from tests.test_gpu_build import build_gpu

pytestmark = pytest.mark.gpu

ROW_POINTS = 1 << 16


def _meshes():
    yield "cube", synth.closed_cube()                    # faces on their boxes' sides, every distance tied
    yield "layers", synth.layered_triangles(37)          # flat boxes
    yield "sphere", synth.displaced_sphere(48, 32)
    yield "soup", synth.open_soup(64, 40)
    yield "octants", nested_octants(16)                  # stacks of more than 64 entries


def _run(gwn, dev, bvh, q, lanes, band, nearest):
    import torch

    n = q[0].shape[0]
    d = [torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in q]
    out = torch.full((n,), 7.0, dtype=torch.float32, device=dev)
    near = torch.full((n,), 7, dtype=torch.int32, device=dev) if nearest else None
    gwn.gwn_compute_unsigned_distance_batch(bvh, *d, out, culling_band=band, nearest=near,
                                            config=gwn.QueryConfig(lanes_per_point=lanes, stack_capacity=128)).raise_if_error()
    torch.cuda.synchronize()
    return out.cpu().numpy().view(np.uint32), near.cpu().numpy() if nearest else None


def _points(mesh, n, seed):
    q = list(synth.mixed_queries(mesh, n, seed=seed, band=0.2))
    k = min(n // 4, 500)
    if k:  # vertices, midpoints of two vertices and grid points: zero and tied distances
        r = np.random.default_rng(seed)
        v = mesh.vertices()
        a, b = v[r.integers(0, v.shape[0], k)], v[r.integers(0, v.shape[0], k)]
        for c in range(3):
            q[c][:k] = np.where(np.arange(k) % 3 == 0, a[:, c],
                                np.where(np.arange(k) % 3 == 1, (a[:, c] + b[:, c]) / 2, np.round(a[:, c])))
    return q


@pytest.mark.parametrize("name,mesh", list(_meshes()), ids=[m[0] for m in _meshes()])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 17, 1023, 20000, ROW_POINTS, ROW_POINTS + 1, 1 << 18, (1 << 18) + 1, 700001])
def test_rows_and_quads_equal_the_lane_kernel(gwn, dev, name, mesh, n):
    _, bvh = build_gpu(gwn, mesh)
    q = _points(mesh, n, seed=n)
    for band in (float("inf"), 0.15, 0.0):
        want, want_rec = _run(gwn, dev, bvh, q, 1, band, True)
        got, got_rec = _run(gwn, dev, bvh, q, 0, band, True)
        assert np.array_equal(got, want) and np.array_equal(got_rec, want_rec), (name, n, band)
        plain, _ = _run(gwn, dev, bvh, q, 0, band, False)
        assert np.array_equal(plain, want), (name, n, band)


@pytest.mark.parametrize("n", [64, ROW_POINTS + 64])
def test_non_finite_points_equal_the_lane_kernel(gwn, dev, n):
    mesh = synth.octahedron()
    _, bvh = build_gpu(gwn, mesh)
    q = _points(mesh, n, seed=3)
    q[0][5], q[1][6], q[2][7], q[0][40] = np.nan, np.inf, -np.inf, 1e30
    want, want_rec = _run(gwn, dev, bvh, q, 1, float("inf"), True)
    got, got_rec = _run(gwn, dev, bvh, q, 0, float("inf"), True)
    fw, fg = want.view(np.float32), got.view(np.float32)
    assert ((want == got) | (np.isnan(fw) & np.isnan(fg))).all() and np.array_equal(got_rec, want_rec)
