"""Batched mode with four lanes per query beside whole waves in one launch: results equal the single-mesh
batch's bit for bit (same tests, same terms, same order per query) for meshes on both sides of the rule, at
counts around a quad, a wave and a chunk, with every block size, also when only the block size changes."""

import numpy as np
import pytest

from smallgwn_amd import synth

from .helpers import nested_octants
from .test_gpu_batch import _check, _queries

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [0, 2])
def test_sparse_and_dense_meshes_in_one_batch(gwn, dev, order):
    import torch

    items, refs = [], []
    # 288 triangles: whole waves from 9,216 queries on; 12,800: four lanes per query at every count here.
    for mesh in (synth.torus(16, 9), synth.torus(80, 80)):
        geom = gwn.GeometryObject()
        gwn.gwn_upload_geometry(geom, mesh.vx, mesh.vy, mesh.vz, mesh.i0, mesh.i1, mesh.i2).raise_if_error()
        for n in (1, 3, 15, 16, 17, 63, 64, 65, 255, 257, 1023, 1025, 9215, 9217):
            bvh, mom = gwn.BvhObject(), gwn.MomentObject(order)
            gwn.gwn_build_bvh(geom, bvh, gwn.BuildOptions(method=gwn.BuildMethod.HPLOC)).raise_if_error()
            gwn.gwn_refit_bvh_moment(bvh, mom).raise_if_error()
            q = [torch.from_numpy(a).to(dev) for a in _queries(mesh, n, n)]
            out = torch.full((n,), float("nan"), dtype=torch.float32, device=dev)
            ref = torch.empty_like(out)
            gwn.gwn_compute_winding_number_taylor_batch(bvh, mom, *q, ref, accuracy_scale=2.0).raise_if_error()
            items.append((bvh, mom, *q, out))
            refs.append((geom, ref))
    batch = gwn.BatchObject(items, accuracy_scale=2.0)
    for traversal in (0, 1, 2):
        for block in (64, 192, 256):
            for it in items:
                it[5].fill_(float("nan"))
            batch.set_tuning(block, 768, 2, traversal).raise_if_error()
            batch.query().raise_if_error()
            _check(items, refs)


@pytest.mark.parametrize("order", [0, 2])
def test_deep_stacks_in_a_batch(gwn, dev, order):
    """A tree whose stack bound needs more than 64 entries beside shallow ones, in quads, waves and both, with the
    LDS of every block size."""
    import torch

    items, refs = [], []
    for mesh, n in ((nested_octants(16), 3000), (synth.torus(16, 9), 20000), (synth.octahedron(), 777)):
        geom, bvh, mom = gwn.GeometryObject(), gwn.BvhObject(), gwn.MomentObject(order)
        gwn.gwn_upload_geometry(geom, mesh.vx, mesh.vy, mesh.vz, mesh.i0, mesh.i1, mesh.i2).raise_if_error()
        gwn.gwn_build_bvh(geom, bvh, gwn.BuildOptions(method=gwn.BuildMethod.HPLOC)).raise_if_error()
        gwn.gwn_refit_bvh_moment(bvh, mom).raise_if_error()
        q = [torch.from_numpy(a).to(dev) for a in _queries(mesh, n, n)]
        if n == 3000:  # toward the small end too
            assert bvh.info()["internal_stack_bound"] > 64
            for a in q:
                a[1000:].mul_(2.0 ** -8)
                a[2000:].mul_(2.0 ** -8)
        out = torch.full((n,), float("nan"), dtype=torch.float32, device=dev)
        ref = torch.empty_like(out)
        gwn.gwn_compute_winding_number_taylor_batch(bvh, mom, *q, ref, accuracy_scale=2.0,
                                                    config=gwn.QueryConfig(stack_capacity=128)).raise_if_error()
        items.append((bvh, mom, *q, out))
        refs.append((geom, ref))
    batch = gwn.BatchObject(items, accuracy_scale=2.0)
    for traversal, density in ((0, 1.0), (1, 1.0), (2, 1.0), (2, 0.01)):
        for block in (64, 192, 256):
            for it in items:
                it[5].fill_(float("nan"))
            batch.set_tuning(block, 768, 4, traversal, wave_queries_per_triangle=density).raise_if_error()
            batch.query().raise_if_error()
            _check(items, refs)
