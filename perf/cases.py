"""Performance cases of the geometric-query library: what its users have it do, over the real range.

A case is a dict of plain values.  ``prepare`` makes what a program has in hand before the call (a
mesh uploaded and built, query points on the GPU, output buffers), ``run`` is one pass through the
public entry points, ``exact`` the same outputs in 64 bits by brute force where that is affordable.

The kinds of case:

  taylor        Taylor winding numbers of a query batch over a built mesh (inside/outside tests)
  gradient      winding number and its gradient with respect to the query point (normals of the field)
  exact         brute-force winding numbers (every triangle for every query)
  distance      unsigned distance of a query batch (sampling a distance field)
  ray           first hits of a ray batch
  rebuild       a mesh whose triangles move freely: tree, moments, then a query batch
  refit         a mesh that deforms: new vertices, box and moment refit, then a query batch
  differentiate one optimisation step: winding and distance forward, loss, backward, SGD
  batch         many uneven meshes rebuilt and queried by one recorded graph

Meshes are closed bumpy latitude-longitude spheres (the library's own large workload), the exact case
an open soup (30 % of the faces missing); queries are half uniform in the box 1.5 times the unit
sphere and half within 0.01 of the surface, as in the library's benchmark, or a regular grid.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from smallgwn_amd import autograd, gwn

DEVICE = "cuda"


def listed():
    return [
        # The smallest call a program makes: a probe of some points against a small mesh, where the
        # launches and the latency of one traversal count.
        {"name": "taylor 1k of 5k", "kind": "taylor", "tris": 5120, "queries": 1000, "points": "mixed",
         "order": 1, "beta": 2.0, "split": False, "build": "lbvh"},
        # An ordinary inside/outside batch at the library's default scale.
        {"name": "taylor 500k of 131k", "kind": "taylor", "tris": 131072, "queries": 500009, "points": "mixed",
         "order": 2, "beta": 2.0, "split": False, "build": "hploc"},
        # The library's benchmark: accurate winding numbers (precision split) of 16.8M points over 1M triangles.
        {"name": "taylor 16m of 1m", "kind": "taylor", "tris": 1048576, "queries": 16777216, "points": "mixed",
         "order": 2, "beta": 6.25, "split": True, "build": "hploc"},
        # Field values and gradients on a regular grid of odd size (surface extraction).
        {"name": "gradient grid 97", "kind": "gradient", "tris": 131072, "queries": 97 ** 3, "points": "grid",
         "order": 1, "beta": 2.0, "split": False, "build": "hploc"},
        # Reference values for a quarter million points over an open soup, in the accurate form.
        {"name": "exact 32k of 100k", "kind": "exact", "tris": 100000, "queries": 32749, "points": "mixed",
         "split": True, "build": "lbvh"},
        # Distance samples of a fine mesh, near and far points mixed.
        {"name": "distance 1m of 1m", "kind": "distance", "tris": 1048576, "queries": 1000003, "points": "mixed",
         "build": "hploc"},
        # A distance field of a small part on a coarse grid.
        {"name": "distance grid 40", "kind": "distance", "tris": 20000, "queries": 40 ** 3, "points": "grid",
         "build": "hploc"},
        # Visibility: first hits of rays aimed at the mesh from around it.
        {"name": "ray 4m of 1m", "kind": "ray", "tris": 1048576, "queries": 4194304, "build": "hploc"},
        # A fine mesh replaced each frame: tree, moments and a few probes.
        {"name": "rebuild 1m", "kind": "rebuild", "tris": 1048576, "queries": 4096, "points": "mixed",
         "order": 2, "beta": 2.0, "split": False, "build": "hploc"},
        # A deforming mesh of ordinary size, refitted each frame.
        {"name": "refit 131k", "kind": "refit", "tris": 131072, "queries": 65536, "points": "mixed",
         "order": 1, "beta": 2.0, "split": False, "build": "hploc"},
        # The library's differentiation workload: one optimisation step over the vertices.
        {"name": "differentiate 131k", "kind": "differentiate", "tris": 131072, "queries": 1048576,
         "targets": 262144, "order": 1, "beta": 2.0, "build": "hploc"},
        # Many uneven meshes, every tree rebuilt, one graph replay.
        {"name": "batch 128", "kind": "batch", "meshes": 128, "max_tris": 100000, "max_queries": 400000,
         "order": 1, "beta": 2.0, "build": "hploc"},
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["taylor", "taylor", "taylor", "gradient", "exact", "distance", "distance", "ray", "rebuild",
                       "refit", "differentiate", "batch"])
    tris = _spread(rng, 500, 1048576)
    build = rng.choice(["hploc", "hploc", "lbvh"])
    if kind == "batch":
        return {"kind": kind, "meshes": _spread(rng, 8, 128), "max_tris": _spread(rng, 2000, 100000),
                "max_queries": _spread(rng, 4000, 400000), "order": rng.choice([0, 1, 2]), "beta": 2.0,
                "build": build}
    if kind == "ray":
        return {"kind": kind, "tris": tris, "queries": _spread(rng, 500, 4194304), "build": build}
    if kind == "exact":
        tris = _spread(rng, 500, 100000)
        # No more pairs than the listed case has.
        queries = min(_spread(rng, 500, 262144), 3_000_000_000 // tris)
        return {"kind": kind, "tris": tris, "queries": queries, "points": "mixed", "split": rng.random() < 0.5,
                "build": build}
    if kind == "differentiate":
        return {"kind": kind, "tris": _spread(rng, 500, 131072), "queries": _spread(rng, 2000, 1048576),
                "targets": _spread(rng, 500, 262144), "order": rng.choice([0, 1]), "beta": 2.0, "build": build}
    points = rng.choice(["mixed", "mixed", "grid"])
    queries = _spread(rng, 500, 1000003 if kind == "distance" else (65536 if kind in ("rebuild", "refit") else 4194304))
    if points == "grid":
        queries = int(round(queries ** (1.0 / 3.0))) ** 3
    case = {"kind": kind, "tris": tris, "queries": queries, "points": points, "build": build}
    if kind != "distance":
        case.update(order=rng.choice([0, 1, 2]), beta=rng.choice([2.0, 2.0, 4.0]), split=rng.random() < 0.4)
    return case


# ---------------------------------------------------------------------------------------------
# Meshes and points, made on the GPU from the seed
# ---------------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed) & 0x7fffffffffff)
    return g


def _rand(g, *shape):
    return torch.rand(shape, generator=g, device=DEVICE, dtype=torch.float64)


def _sphere(tris, g):
    """Closed outward-oriented latitude-longitude sphere with about ``tris`` triangles and r = 1 + bumps.

    Returns vertices (V, 3) float64 and faces (T, 3) int64 on the GPU.  The poles are single vertices,
    so one triangle of each pole quad has no area, as in the library's own meshes.
    """
    nlat = max(3, int(round(math.sqrt(tris / 4.0))))
    nlon = max(3, int(round(tris / (2.0 * nlat))))
    th = (torch.arange(1, nlat, device=DEVICE, dtype=torch.float64) * (math.pi / nlat)).repeat_interleave(nlon)
    ph = (torch.arange(nlon, device=DEVICE, dtype=torch.float64) * (2.0 * math.pi / nlon)).repeat(nlat - 1)
    pole = torch.tensor([[0.0, 0.0, 1.0], [0.0, 0.0, -1.0]], device=DEVICE, dtype=torch.float64)
    ring = torch.stack([th.sin() * ph.cos(), th.sin() * ph.sin(), th.cos()], 1)
    d = torch.cat([pole[:1], ring, pole[1:]])
    k = (_rand(g, 8, 3) * 2.0 - 1.0) * 9.0
    r = 1.0 + 0.02 * torch.sin(d @ k.t() + 2.0 * math.pi * _rand(g, 8)).sum(1)
    v = d * r[:, None]
    i = torch.arange(nlat, device=DEVICE).repeat_interleave(nlon)
    j = torch.arange(nlon, device=DEVICE).repeat(nlat)

    def vid(a, b):
        x = 1 + (a - 1) * nlon + b % nlon
        x = torch.where(a == 0, torch.zeros_like(x), x)
        return torch.where(a == nlat, torch.full_like(x, 1 + (nlat - 1) * nlon), x)

    a, b, c, e = vid(i, j), vid(i + 1, j), vid(i + 1, j + 1), vid(i, j + 1)
    return v, torch.stack([torch.stack([a, b, c], 1), torch.stack([a, c, e], 1)], 1).reshape(-1, 3)


def _mesh(case, g):
    if case["kind"] == "exact":  # about ``tris`` faces left of a sphere that lost 30 % of them
        v, f = _sphere(case["tris"] / 0.7, g)
        f = f[_rand(g, f.shape[0]) >= 0.3]
    else:
        v, f = _sphere(case["tris"], g)
    return v.to(torch.float32), f


def _near(v, f, n, g, band):
    """``n`` points within ``band`` of the surface, along the normals of random faces."""
    v = v.to(torch.float64)
    a, b, c = v[f[:, 0]], v[f[:, 1]], v[f[:, 2]]
    nrm = torch.linalg.cross(b - a, c - a)
    good = torch.nonzero(nrm.norm(dim=1) > 0)[:, 0]
    t = good[(_rand(g, n) * good.numel()).long().clamp_(max=good.numel() - 1)]
    s, w = _rand(g, n).sqrt()[:, None], _rand(g, n)[:, None]
    p = (1.0 - s) * a[t] + s * (1.0 - w) * b[t] + s * w * c[t]
    unit = nrm[t] / nrm[t].norm(dim=1, keepdim=True)
    return p + unit * ((_rand(g, n) * 2.0 - 1.0) * band)[:, None]


def _points(case, v, f, g):
    n = case["queries"]
    if case.get("points") == "grid":
        m = int(round(n ** (1.0 / 3.0)))
        # A grid over the box, its origin not the same for every seed.
        ax = [(torch.arange(m, device=DEVICE, dtype=torch.float64) + o) * (2.5 / m) - 1.25 for o in _rand(g, 3)]
        p = torch.stack(torch.meshgrid(*ax, indexing="ij"), -1).reshape(-1, 3)
    else:
        near = n // 2
        p = torch.cat([_rand(g, n - near, 3) * 3.0 - 1.5, _near(v, f, near, g, 0.01)])
    return _soa(p)


def _soa(p):
    p = p.to(torch.float32)
    return [p[:, k].contiguous() for k in range(3)]


def _upload(v, f):
    geo = gwn.GeometryObject()
    x, i = v.t().contiguous().cpu().numpy(), f.t().contiguous().to(torch.int32).cpu().numpy().astype(np.uint32)
    gwn.gwn_upload_geometry(geo, x[0], x[1], x[2], i[0], i[1], i[2]).raise_if_error()
    return geo


def _options(case):
    return gwn.BuildOptions(method=gwn.BuildMethod.LBVH if case["build"] == "lbvh" else gwn.BuildMethod.HPLOC)


def _precision(case):
    return gwn.Precision.SPLIT if case["split"] else gwn.Precision.PLAIN


class _Device:
    """An object's device storage as a tensor (no copy)."""

    def __init__(self, address, count, typestr):
        self.__cuda_array_interface__ = {"shape": (int(count),), "typestr": typestr, "data": (int(address), False),
                                         "version": 3}


def _view(owner, address, count, typestr):
    t = torch.as_tensor(_Device(address, count, typestr), device=DEVICE)
    t.owner = owner  # the storage lives as long as the object that it belongs to
    return t


def _tree(bvh):
    """The tree's public storage (primitive order, leaf triangles) and what a program reads of its nodes on
    the host.  The node array itself has another length for every mesh; the winding numbers go through it."""
    a = bvh.accessor()
    return {"primitives": _view(bvh, a["primitive_indices"], a["triangle_count"], "<i4"),
            "triangles": _view(bvh, a["triangles"], 9 * a["triangle_count"], "<f4"),
            "node_count": a["node_count"], "stack_bound": a["internal_stack_bound"], "root_bounds": a["root_bounds"]}


# ---------------------------------------------------------------------------------------------
# prepare, run
# ---------------------------------------------------------------------------------------------

def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "batch":
        return _prepare_batch(case, seed, g)
    v, f = _mesh(case, g)
    if kind == "differentiate":
        return _prepare_differentiate(case, v, f, g)
    s = {"case": case, "geometry": _upload(v, f), "bvh": gwn.BvhObject()}
    gwn.gwn_build_bvh(s["geometry"], s["bvh"], _options(case)).raise_if_error()
    n = case["queries"]
    if kind == "ray":
        s["rays"] = _rays(n, g)
        s["hits"] = torch.zeros(8 * n, dtype=torch.int32, device=DEVICE)
        return s
    if "order" in case:
        s["moment"] = gwn.MomentObject(case["order"])
        gwn.gwn_refit_bvh_moment(s["bvh"], s["moment"]).raise_if_error()
    s["q"] = _points(case, v, f, g)
    s["out"] = torch.zeros(n, dtype=torch.float64 if kind == "exact" and case["split"] else torch.float32,
                           device=DEVICE)
    if kind == "gradient":
        s["grad"] = [torch.zeros(n, dtype=torch.float32, device=DEVICE) for _ in range(3)]
    if kind == "refit":
        s["moved"] = _soa(_moved(v, g))
    return s


def _moved(v, g):
    """Vertices after a smooth deformation."""
    v = v.to(torch.float64)
    k = (_rand(g, 3, 3) * 2.0 - 1.0) * 4.0
    return v + 0.05 * torch.sin(v @ k + 2.0 * math.pi * _rand(g, 3))


def _rays(n, g):
    """Origins on a sphere of radius 3, directions toward points of the unit ball."""
    o = torch.randn((n, 3), generator=g, device=DEVICE, dtype=torch.float64)
    o = 3.0 * o / o.norm(dim=1, keepdim=True)
    t = torch.randn((n, 3), generator=g, device=DEVICE, dtype=torch.float64)
    t = t / t.norm(dim=1, keepdim=True) * _rand(g, n, 1) ** (1.0 / 3.0)
    d = t - o
    return _soa(o) + _soa(d / d.norm(dim=1, keepdim=True))


def _prepare_differentiate(case, v, f, g):
    verts = v.clone().requires_grad_(True)
    scene = autograd.MeshScene(f, verts, order=case["order"], method=_options(case).method,
                               accuracy_scale=case["beta"])
    queries = (_rand(g, case["queries"], 3) * 3.0 - 1.5).to(torch.float32)
    t = torch.randn((case["targets"], 3), generator=g, device=DEVICE, dtype=torch.float64)
    targets = (0.9 * t / t.norm(dim=1, keepdim=True)).to(torch.float32)
    return {"case": case, "vertices": verts, "scene": scene, "queries": queries, "targets": targets,
            "labels": (queries.norm(dim=1) < 0.9).to(torch.float32), "optimizer": torch.optim.SGD([verts], lr=1e-3)}


def _batch_sizes(case, seed):
    r = np.random.default_rng(seed)
    m = case["meshes"]
    tris = np.exp(r.uniform(math.log(200), math.log(case["max_tris"]), m)).astype(np.int64)
    queries = np.exp(r.uniform(math.log(64), math.log(case["max_queries"]), m)).astype(np.int64)
    return tris, queries


def _prepare_batch(case, seed, g):
    # Sizes come from the case, so that passes of other seeds cost the same.
    tris, queries = _batch_sizes(case, case["meshes"])
    out = torch.zeros(int(queries.sum()), dtype=torch.float32, device=DEVICE)
    items, at = [], 0
    for t, n in zip(tris.tolist(), queries.tolist()):
        v, f = _sphere(t, g)
        v = (v * (0.5 + _rand(g, 3)) + (_rand(g, 3) * 10.0 - 5.0)).to(torch.float32)
        lo, hi = v.amin(0), v.amax(0)
        q = _soa((lo + hi) / 2 + (_rand(g, n, 3) - 0.5) * (hi - lo) * 1.5)
        items.append((_upload(v, f), q[0], q[1], q[2], out[at:at + n]))
        at += n
    batch = gwn.BuiltBatchObject(items, width=4, hploc_radius=8, order=case["order"], accuracy_scale=case["beta"],
                                 method=_options(case).method)
    # The launch shape that the library's tuner settles on for such batches.
    batch.set_tuning(256, 1024, 8, traversal=1).raise_if_error()
    batch.capture(include_refit=True).raise_if_error()
    return {"case": case, "batch": batch, "out": out}


def _taylor(s):
    c = s["case"]
    gwn.gwn_compute_winding_number_taylor_batch(s["bvh"], s["moment"], *s["q"], s["out"], accuracy_scale=c["beta"],
                                                precision=_precision(c)).raise_if_error()
    return s["out"]


def run(state):
    s = state
    c = s["case"]
    kind = c["kind"]
    if kind == "taylor":
        return _taylor(s)
    if kind == "gradient":
        gwn.gwn_compute_winding_gradient_taylor_batch(s["bvh"], s["moment"], *s["q"], *s["grad"],
                                                      accuracy_scale=c["beta"], precision=_precision(c),
                                                      out=s["out"]).raise_if_error()
        return {"winding": s["out"], "gradient": s["grad"]}
    if kind == "exact":
        if c["split"]:
            gwn.gwn_compute_winding_number_exact_batch_ex(s["bvh"], *s["q"], s["out"],
                                                          gwn.Precision.SPLIT).raise_if_error()
        else:
            gwn.gwn_compute_winding_number_exact_batch(s["bvh"], *s["q"], s["out"]).raise_if_error()
        return s["out"]
    if kind == "distance":
        gwn.gwn_compute_unsigned_distance_batch(s["bvh"], *s["q"], s["out"]).raise_if_error()
        return s["out"]
    if kind == "ray":
        gwn.gwn_compute_ray_first_hit_batch(s["bvh"], *s["rays"], s["hits"]).raise_if_error()
        h = s["hits"].view(-1, 8)
        return {"hit": h[:, :6].view(torch.float32), "id": h[:, 6:]}
    if kind == "rebuild":
        gwn.gwn_build_bvh(s["geometry"], s["bvh"], _options(c)).raise_if_error()
        gwn.gwn_refit_bvh_moment(s["bvh"], s["moment"]).raise_if_error()
        return {"tree": _tree(s["bvh"]), "winding": _taylor(s)}
    if kind == "refit":
        gwn.gwn_update_geometry(s["geometry"], *s["moved"]).raise_if_error()
        gwn.gwn_refit_bvh(s["geometry"], s["bvh"]).raise_if_error()
        gwn.gwn_refit_bvh_moment(s["bvh"], s["moment"]).raise_if_error()
        return {"tree": _tree(s["bvh"]), "winding": _taylor(s)}
    if kind == "differentiate":
        s["optimizer"].zero_grad(set_to_none=True)
        w = autograd.taylor_winding(s["vertices"], s["queries"], s["scene"])
        d = autograd.unsigned_distance(s["vertices"], s["targets"], s["scene"])
        loss = ((torch.sigmoid(20.0 * (w - 0.5)) - s["labels"]) ** 2).mean() + d.mean()
        loss.backward()
        s["optimizer"].step()
        return {"winding": w.detach(), "distance": d.detach(), "gradient": s["vertices"].grad,
                "vertices": s["vertices"].detach(), "loss": loss.detach()}
    s["batch"].replay().raise_if_error()
    return s["out"]


# ---------------------------------------------------------------------------------------------
# work, tolerance, exact
# ---------------------------------------------------------------------------------------------

_TERM = {0: 12, 1: 34, 2: 55}          # operations of one accepted expansion
_FIELDS = {0: 7, 1: 13, 2: 23}         # coefficients of one child slot


def _taylor_flops(tris, queries, order, beta):
    # Accepted expansions of a query over a surface grow with beta^2 and the depth; each comes with
    # about 1.5 acceptance tests, and about an eighth as many near triangles.
    accepted = 1.8 * beta * beta * max(1.0, math.log2(tris))
    return queries * accepted * (1.5 * 10 + _TERM[order] + 87 / 8.0)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        tris, queries = _batch_sizes(case, case["meshes"])
        t, n = int(tris.sum()), int(queries.sum())
        flops = sum(_taylor_flops(int(a), int(b), case["order"], case["beta"]) for a, b in zip(tris, queries))
        return {"bytes": 18 * t + t * (36 + 4 + 64) + t * 2 * 4 * _FIELDS[case["order"]] + 16 * n, "flops": flops + 60.0 * t}
    t, n = case["tris"], case["queries"]
    depth = max(1.0, math.log2(t))
    records = 36 * t
    boxes = 64 * t                     # about half as many wide nodes as triangles, 128 bytes each
    if kind == "exact":
        return {"bytes": records + 20 * n, "flops": 87.0 * t * n}
    if kind == "distance":
        return {"bytes": records + boxes + 16 * n, "flops": n * depth * (4 * 18 + 2 * 60)}
    if kind == "ray":
        return {"bytes": records + boxes + 56 * n, "flops": n * depth * (4 * 20 + 50)}
    moments = 2 * t * 4 * _FIELDS[case["order"]]
    flops = _taylor_flops(t, n, case["order"], case["beta"])
    if kind == "taylor":
        return {"bytes": records + moments + 16 * n, "flops": flops}
    if kind == "gradient":
        return {"bytes": records + moments + 28 * n, "flops": 2 * flops}
    if kind == "rebuild":
        return {"bytes": 18 * t + records + 4 * t + boxes + moments + 16 * n, "flops": flops + 60.0 * t * depth}
    if kind == "refit":
        return {"bytes": 6 * t + 18 * t + records + 2 * boxes + moments + 16 * n, "flops": flops + 60.0 * t}
    m = case["targets"]
    return {"bytes": 18 * t + 2 * (records + moments) + 2 * boxes + 28 * n + 28 * m,
            "flops": 3 * flops + m * depth * (4 * 18 + 2 * 60)}


def tolerance(case):
    kind = case["kind"]
    if kind == "differentiate":
        # 32-bit atomic sums of the vertex gradients over up to a million queries.
        return {"rel": 1e-4, "max": 1e-2}
    if kind == "gradient":
        # Plain arithmetic close to a face: 3e-5 and 2.5e-2 against 64-bit sums and near triangles.
        return {"rel": 1e-4, "max": 1e-1} if not case["split"] else {"rel": 1e-5, "max": 1e-3}
    if kind == "exact":
        # Split: 64-bit sums, 32-bit angles of the far triangles (3e-8, 2.3e-7 measured against 64
        # bits); plain: one 32-bit sum over every triangle (1.7e-5, 7e-5).
        return {"rel": 1.2e-7, "max": 1e-6} if case["split"] else {"rel": 7e-5, "max": 1e-3}
    if kind == "distance":
        return {"rel": 1e-6, "max": 1e-5}  # the smallest of the triangles' distances, each in 32 bits
    if kind == "ray":
        # A ray through a shared edge has either face's id and normal: one in a million with another tree.
        return {"rel": 1e-4, "max": 0.9, "differ": 5e-6}
    # 32-bit sums of some hundred terms; plain arithmetic close to a face loses digits.
    return {"rel": 1e-5, "max": 1e-2}


_PAIRS = 12_000_000_000  # brute force in 64 bits stays under about 20 seconds


def _winding64(v, f, q):
    """Winding numbers of points q over all triangles, in 64 bits."""
    v = v.to(torch.float32).to(torch.float64)
    a, b, c = (v[f[:, k]].t().contiguous() for k in range(3))
    p = torch.stack(q, 0).to(torch.float64)
    n = p.shape[1]
    out = torch.empty(n, dtype=torch.float64, device=DEVICE)
    step = max(1, 16_000_000 // max(1, f.shape[0]))
    for i in range(0, n, step):
        x = p[:, i:i + step, None]
        d = [[m[k][None] - x[k] for k in range(3)] for m in (a, b, c)]
        ln = [(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]).sqrt() for u in d]

        def dot(u, w):
            return u[0] * w[0] + u[1] * w[1] + u[2] * w[2]

        num = (d[0][0] * (d[1][1] * d[2][2] - d[1][2] * d[2][1]) + d[0][1] * (d[1][2] * d[2][0] - d[1][0] * d[2][2])
               + d[0][2] * (d[1][0] * d[2][1] - d[1][1] * d[2][0]))
        den = (ln[0] * ln[1] * ln[2] + dot(d[0], d[1]) * ln[2] + dot(d[0], d[2]) * ln[1] + dot(d[1], d[2]) * ln[0])
        out[i:i + step] = torch.atan2(num, den).sum(1) / (2.0 * math.pi)
    return out


def _distance64(v, f, q):
    """Distances of points q to the nearest of all triangles, in 64 bits: the plane's foot where it
    lies in the triangle, the nearest edge elsewhere."""
    v = v.to(torch.float32).to(torch.float64)
    t = [v[f[:, k]].t().contiguous() for k in range(3)]
    p = torch.stack(q, 0).to(torch.float64)
    n = p.shape[1]
    out = torch.empty(n, dtype=torch.float64, device=DEVICE)
    step = max(1, 16_000_000 // max(1, f.shape[0]))
    e = [t[(k + 1) % 3] - t[k] for k in range(3)]
    nrm = torch.linalg.cross(e[0], e[1], dim=0)
    nn = (nrm * nrm).sum(0)
    for i in range(0, n, step):
        x = p[:, i:i + step, None]
        best = None
        inside = (nn > 0)[None]
        for k in range(3):
            r = [x[m] - t[k][m][None] for m in range(3)]
            ee = (e[k] * e[k]).sum(0)
            s = (r[0] * e[k][0] + r[1] * e[k][1] + r[2] * e[k][2]) / torch.where(ee > 0, ee, torch.ones_like(ee))
            s = s.clamp(0.0, 1.0)
            d = sum((r[m] - s * e[k][m][None]) ** 2 for m in range(3))
            best = d if best is None else torch.minimum(best, d)
            m = torch.linalg.cross(nrm, e[k], dim=0)  # toward the inside of this edge
            inside = inside & (r[0] * m[0] + r[1] * m[1] + r[2] * m[2] >= 0)
        h = r[0] * nrm[0] + r[1] * nrm[1] + r[2] * nrm[2]
        best = torch.where(inside, torch.minimum(best, h * h / torch.where(nn > 0, nn, torch.ones_like(nn))), best)
        out[i:i + step] = best.amin(1).sqrt()
    return out


def exact(case, seed):
    """The Taylor kinds against the winding number that they expand, distances against brute force."""
    kind = case["kind"]
    if kind in ("batch", "differentiate", "ray") or case["tris"] * case["queries"] > _PAIRS:
        return None
    g = _gen(seed)
    v, f = _mesh(case, g)
    q = _points(case, v, f, g)
    if kind == "refit":
        v = torch.stack(_soa(_moved(v, g)), 1)
    if kind == "distance":
        return _distance64(v, f, q)
    w = _winding64(v, f, q)
    if kind == "gradient":
        return {"winding": w, "gradient": [None, None, None]}
    if kind in ("rebuild", "refit"):
        return {"tree": {"primitives": None, "triangles": None, "node_count": None, "stack_bound": None, "root_bounds": None},
                "winding": w}
    return w
