"""The Taylor traversals with 16 and four lanes per query against the wave traversal: values, gradients and work
counters equal bit for bit, at the edges of rows, quads, waves and blocks and on both sides of the rules
that choose between them."""

import numpy as np
import pytest

from smallgwn_amd import synth
from tests.helpers import nested_octants
from tests.test_gpu_build import build_gpu

pytestmark = pytest.mark.gpu


def _first(q, n, dev):
    import torch

    return [torch.from_numpy(np.ascontiguousarray(a[:n])).to(dev) for a in q]


def _run(gwn, dev, bvh, mom, d, sort, precision, beta, grad):
    import torch

    n = d[0].numel()
    out = torch.full((n,), 7.0, dtype=torch.float32, device=dev)
    cnt = torch.zeros(3 * n, dtype=torch.int32, device=dev)
    cfg = gwn.QueryConfig(sort_queries=sort, stack_capacity=128)
    if grad:
        g = [torch.full_like(out, 7.0) for _ in range(3)]
        gwn.gwn_compute_winding_gradient_taylor_batch(bvh, mom, *d, *g, accuracy_scale=beta, config=cfg,
                                                      precision=precision, out=out, counters=cnt).raise_if_error()
    else:
        g = []
        gwn.gwn_compute_winding_number_taylor_batch(bvh, mom, *d, out, accuracy_scale=beta, config=cfg,
                                                    precision=precision, counters=cnt).raise_if_error()
    torch.cuda.synchronize()
    return [t.cpu().numpy().view(np.uint32) for t in (out, cnt, *g)]


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("order", [0, 1, 2])
def test_quad_equals_wave_bit_for_bit(gwn, dev, order, split, grad):
    precision = gwn.Precision.SPLIT if split else gwn.Precision.PLAIN
    # 8 triangles: dense from 12,728 queries at scale 2; 320: from one query at scale 1e6.
    for mesh, beta, n_wave in ((synth.octahedron(), 2.0, 66000), (synth.icosphere(2), 1e6, 66000)):
        _, bvh = build_gpu(gwn, mesh)
        mom = gwn.MomentObject(order)
        gwn.gwn_refit_bvh_moment(bvh, mom).raise_if_error()
        q = synth.mixed_queries(mesh, n_wave, seed=order + 11)
        q[0][5], q[1][6] = np.nan, np.inf
        want = _run(gwn, dev, bvh, mom, _first(q, n_wave, dev), 1, precision, beta, grad)
        for n in (1, 3, 4, 5, 15, 17, 65, 257, 65536, 65537):
            got = _run(gwn, dev, bvh, mom, _first(q, n, dev), 0, precision, beta, grad)
            for k, (a, b) in enumerate(zip(got, want)):
                b = b[:3 * n] if k == 1 else b[:n]
                fa, fb = a.view(np.float32), b.view(np.float32)
                same = (a == b) | (np.isnan(fa) & np.isnan(fb) if k != 1 else False)
                assert same.all(), (beta, n, k)


def test_quads_beyond_one_launch(gwn, dev):
    """2^28 + 77 unsorted queries (two launches): both ends equal the same queries in a batch of their own."""
    import torch

    mesh = synth.torus(40, 20)
    _, bvh = build_gpu(gwn, mesh)
    mom = gwn.MomentObject(0)
    gwn.gwn_refit_bvh_moment(bvh, mom).raise_if_error()
    n, k = (1 << 28) + 77, 70000
    g = torch.Generator(device=dev)
    g.manual_seed(1)
    d = [torch.rand(n, generator=g, device=dev) * 3 - 1.5 for _ in range(3)]
    out = torch.full((n,), 7.0, device=dev)
    cfg = gwn.QueryConfig(sort_queries=0)
    gwn.gwn_compute_winding_number_taylor_batch(bvh, mom, *d, out, accuracy_scale=2.0, config=cfg).raise_if_error()
    for part in (slice(0, k), slice(n - k, n)):
        e = [a[part].clone() for a in d]
        want = torch.empty(k, device=dev)
        gwn.gwn_compute_winding_number_taylor_batch(bvh, mom, *e, want, accuracy_scale=2.0, config=cfg).raise_if_error()
        assert torch.equal(out[part], want)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("triangles,beta", [(8, 2.0), (16, 2.0), (101, 2.0), (300, 6.25)])
def test_whole_waves_of_tiny_trees_in_any_order(gwn, dev, triangles, beta, grad):
    """Unsorted batches on both sides of the rule that walks a tree with whole waves where every query descends most
    of it: the same bits as rows (a smaller batch of the same queries), work counters too."""
    full = synth.torus(20, 10)
    mesh = synth.Mesh(full.vx, full.vy, full.vz, full.i0[:triangles].copy(), full.i1[:triangles].copy(), full.i2[:triangles].copy())
    _, bvh = build_gpu(gwn, mesh)
    for order, precision in ((1, gwn.Precision.PLAIN), (2, gwn.Precision.SPLIT)):
        mom = gwn.MomentObject(order)
        gwn.gwn_refit_bvh_moment(bvh, mom).raise_if_error()
        q = synth.mixed_queries(mesh, 70000, seed=triangles)
        q[0][5], q[1][6] = np.nan, np.inf
        small = [_run(gwn, dev, bvh, mom, _first([a[at:] for a in q], 7000, dev), 0, precision, beta, grad)
                 for at in range(0, 70000, 7000)]
        want = [np.concatenate(parts) for parts in zip(*small)]
        for n in (32767, 40768, 48767, 48768, 48769, 63487, 63488, 63489, 70000):
            got = _run(gwn, dev, bvh, mom, _first(q, n, dev), 0, precision, beta, grad)
            for k, (a, b) in enumerate(zip(got, want)):
                b = b[:a.shape[0]]
                fa, fb = a.view(np.float32), b.view(np.float32)
                assert ((a == b) | (np.isnan(fa) & np.isnan(fb) if k != 1 else False)).all(), (n, k)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("order", [0, 1, 2])
@pytest.mark.parametrize("name", ["sphere", "octants"])
def test_rows_and_quads_equal_waves_on_deep_trees(gwn, dev, name, order, split, grad):
    """Accepted terms, leaves and stacks of many entries (more than 64 allowed for the octants) together: a sorted
    batch dense enough for whole waves, the same queries unsorted in rows and in quads."""
    mesh = synth.displaced_sphere(40, 32) if name == "sphere" else nested_octants(16)
    precision = gwn.Precision.SPLIT if split else gwn.Precision.PLAIN
    _, bvh = build_gpu(gwn, mesh)
    assert name == "sphere" or bvh.info()["internal_stack_bound"] > 64
    mom = gwn.MomentObject(order)
    gwn.gwn_refit_bvh_moment(bvh, mom).raise_if_error()
    n_wave = 250000
    assert n_wave >= 4500 * np.sqrt(mesh.i0.shape[0])  # dense at scale 2
    q = synth.mixed_queries(mesh, n_wave, seed=order + 3)
    if name == "octants":
        for a in q:
            a[:40000] *= np.float32(2.0) ** -(np.arange(40000) % 18).astype(np.float32)
    want = _run(gwn, dev, bvh, mom, _first(q, n_wave, dev), 1, precision, 2.0, grad)
    for n in (1000, 65536, 65537):
        got = _run(gwn, dev, bvh, mom, _first(q, n, dev), 0, precision, 2.0, grad)
        for k, (a, b) in enumerate(zip(got, want)):
            assert np.array_equal(a, b[:a.shape[0]]), (n, k)
