"""The four-lanes-per-ray traversals (packed and canonical) at the edges of quads, waves and blocks and
where a wave hands out further rays: records equal the oracle's bit for bit."""

import numpy as np
import pytest

from smallgwn_amd import synth
from tests.helpers import nested_octants
from tests.test_gpu_build import build_gpu
from tests.test_gpu_ray import _oracle, _rays, _same

pytestmark = pytest.mark.gpu

MESHES = {"cube": synth.closed_cube(), "layers": synth.layered_triangles(33), "soup": synth.open_soup(48, 32)}


def _set(mesh, n, seed):
    """Rays around the mesh: toward random points, along axes, from vertices, toward vertices and edges, zero
    and non-finite ones."""
    r = np.random.default_rng(seed)
    v = mesh.vertices()
    o = r.normal(size=(n, 3))
    o = o / np.linalg.norm(o, axis=1, keepdims=True) * 3.0
    at = v[r.integers(0, v.shape[0], n)]
    to = np.where((np.arange(n) % 3 == 0)[:, None], at, np.where((np.arange(n) % 3 == 1)[:, None],
                  (at + v[r.integers(0, v.shape[0], n)]) / 2, r.uniform(-1, 1, (n, 3))))
    o = np.where((np.arange(n) % 11 == 0)[:, None], at, o)
    d = to - o
    d[5::13, 0] = 0.0
    d[7::17, 1:] = 0.0
    d[::29] = 0.0
    if n > 40:
        d[40, 2], o[41 % n, 0] = np.nan, np.inf
    return o.astype(np.float32), d.astype(np.float32)


@pytest.mark.parametrize("canonical", [False, True])
@pytest.mark.parametrize("name", list(MESHES))
@pytest.mark.parametrize("n", [1, 3, 4, 17, 64, 257, 3001])
def test_quad_records_equal_the_oracle(gwn, orc, dev, name, n, canonical):
    mesh = MESHES[name]
    _, bvh = build_gpu(gwn, mesh)
    info = bvh.info()
    stack = info["internal_stack_bound"] if canonical else max(64, info["packed_stack_bound"])
    if canonical and info["packed_stack_bound"] <= stack:
        pytest.skip("the packed traversal fits this tree's smallest stack")
    o, d = _set(mesh, n, n)
    for t_min, t_max in ((0.0, float("inf")), (-1.0, 2.5), (1.0, 1.0)):
        _same(_rays(gwn, dev, bvh, o, d, t_min, t_max, stack=stack), _oracle(orc, mesh, o, d, t_min, t_max, stack=stack))


@pytest.mark.parametrize("canonical", [False, True])
def test_rays_handed_out_within_a_wave(gwn, orc, dev, canonical):
    """700,001 rays (a wave's quads take several each) equal the same rays in batches of 5,000."""
    mesh = MESHES["soup"]
    _, bvh = build_gpu(gwn, mesh)
    info = bvh.info()
    stack = info["internal_stack_bound"] if canonical else max(64, info["packed_stack_bound"])
    assert not canonical or info["packed_stack_bound"] > stack
    o, d = _set(mesh, 700001, 3)
    got = _rays(gwn, dev, bvh, o, d, stack=stack)
    for k in (0, 262140, 695001):
        _same(got[k:k + 5000], _rays(gwn, dev, bvh, o[k:k + 5000], d[k:k + 5000], stack=stack))
    _same(got[::997], _oracle(orc, mesh, o[::997], d[::997], stack=stack))


@pytest.mark.parametrize("canonical", [False, True])
@pytest.mark.parametrize("seed", [0, 2, 4, 10])
def test_directions_with_infinite_reciprocals(gwn, orc, dev, seed, canonical):
    """Subnormal direction components and origins in the planes of flat boxes: a child's slab test gives 0 * inf and
    meets the box at any t, so no entry beyond the best hit may be dropped by its own box's t."""
    r = np.random.default_rng(100 + seed)
    count, side = int(r.integers(40, 600)), int(r.integers(2, 6))
    tri = np.repeat(r.integers(0, side + 1, (count, 3))[:, None], 3, 1)
    axis = r.integers(0, 3, count)
    for k in (1, 2):
        off = r.integers(-2, 3, (count, 3))
        off[np.arange(count), axis] = 0
        tri[:, k] += off
    v, f = tri.reshape(-1, 3).astype(np.float32), np.arange(3 * count).reshape(-1, 3).astype(np.uint32)
    mesh = synth.Mesh(*(np.ascontiguousarray(v[:, k]) for k in range(3)), *(np.ascontiguousarray(f[:, k]) for k in range(3)))
    _, bvh = build_gpu(gwn, mesh)
    info = bvh.info()
    stack = info["internal_stack_bound"] if canonical else max(64, info["packed_stack_bound"])
    n = 300000
    o = r.integers(-4, 2 * side + 5, (n, 3)) / 2.0
    d = r.integers(-2, 3, (n, 3)).astype(np.float64)
    d = np.where(r.random((n, 3)) < 0.5, r.choice([1e-40, -1e-40, 3e-39, -1e-44], (n, 3)), d)
    o, d = o.astype(np.float32), d.astype(np.float32)
    for t_min in (0.0, -5.0, -float("inf")):
        _same(_rays(gwn, dev, bvh, o, d, t_min, stack=stack), _oracle(orc, mesh, o, d, t_min, stack=stack))


@pytest.mark.parametrize("canonical", [False, True])
@pytest.mark.parametrize("n", [1000, 100003])
def test_deep_stacks(gwn, orc, dev, n, canonical):
    """Stacks of more than 64 entries, with whole bounds (few rays) and 16-bit ones (more blocks than LDS holds with
    whole ones)."""
    mesh = nested_octants(16)
    _, bvh = build_gpu(gwn, mesh)
    info = bvh.info()
    assert info["packed_stack_bound"] > info["internal_stack_bound"] > 64
    stack = info["internal_stack_bound"] if canonical else 128
    r = np.random.default_rng(n)
    v = mesh.vertices()
    o = r.normal(size=(n, 3))
    o = (o / np.linalg.norm(o, axis=1, keepdims=True) * 2.0 ** -r.integers(0, 18, (n, 1))).astype(np.float32)
    d = (v[r.integers(0, v.shape[0], n)] - o).astype(np.float32)
    for t_min in (0.0, -1.0):
        _same(_rays(gwn, dev, bvh, o, d, t_min, stack=stack), _oracle(orc, mesh, o, d, t_min, stack=stack))


@pytest.mark.parametrize("triangles", [12, 64, 65])
def test_many_rays_of_a_few_triangles(gwn, orc, dev, triangles):
    """Both sides of the rule that gives large batches over a few triangles one lane per ray."""
    mesh = synth.open_soup(16, 8)
    mesh = synth.Mesh(mesh.vx, mesh.vy, mesh.vz, mesh.i0[:triangles].copy(), mesh.i1[:triangles].copy(), mesh.i2[:triangles].copy())
    _, bvh = build_gpu(gwn, mesh)
    o, d = _set(mesh, (1 << 19) + 5, triangles)
    for n in ((1 << 19) - 1, (1 << 19) + 5):
        got = _rays(gwn, dev, bvh, o[:n], d[:n])
        _same(got[-20000:], _oracle(orc, mesh, o[n - 20000:n], d[n - 20000:n]))
