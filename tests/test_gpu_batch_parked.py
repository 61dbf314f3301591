"""H-PLOC over a batch large enough (more than 6.3M leaves) that the global launch takes one parked range per
lane instead of one per half wave: trees, moments and results still equal the single-mesh build's bit for bit."""

import numpy as np
import pytest

from smallgwn_amd import synth

from .test_gpu_batch_build import _same_results, _same_tree, _sequential

pytestmark = pytest.mark.gpu


def test_one_parked_range_per_lane_equals_single_builds(gwn, dev):
    import torch

    geoms = []
    count = 84
    for mesh in [synth.torus(317, 158), synth.displaced_sphere(320, 160)] * (count // 2):  # about 100,000 triangles
        geom = gwn.GeometryObject()
        gwn.gwn_upload_geometry(geom, mesh.vx, mesh.vy, mesh.vz, mesh.i0, mesh.i1, mesh.i2).raise_if_error()
        geoms.append(geom)
    q = [torch.from_numpy(a).to(dev) for a in synth.uniform_box_points(4, 500, (-1.5,) * 3, (1.5,) * 3)]
    leaves = sum(g.triangle_count() for g in geoms)
    assert leaves > 8192 * 1024
    outs = [torch.full((500,), float("nan"), dtype=torch.float32, device=dev) for _ in range(count)]
    batch = gwn.BuiltBatchObject([(geoms[k], *q, outs[k]) for k in range(count)], order=0, accuracy_scale=2.0)
    batch.query().raise_if_error()
    torch.cuda.synchronize()
    assert batch.status().is_ok()
    for k in (0, 1, 41, 82, 83):
        want = _sequential(gwn, geoms[k], q, 4, 8, 0)
        _same_tree(k, batch.export(k), want[:2])
        _same_results(k, outs[k], want[2])
    assert all(np.array_equal(o.cpu().numpy(), outs[k % 2].cpu().numpy()) for k, o in enumerate(outs))
