"""Batched mode with four lanes per query beside whole waves in one launch: results equal the single-mesh
batch's bit for bit (same tests, same terms, same order per query) for meshes on both sides of the rule, at
counts around a quad, a wave and a chunk, with every block size, also when only the block size changes."""

import numpy as np
import pytest

from smallgwn_amd import synth

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
