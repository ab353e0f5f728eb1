"""Performance cases: points in, exact Delaunay tetrahedra and adjacency out, in the forms in which
programs call the library's C ABI (include/gstar4d.h).

Every case names one way of calling it (`call`):

  serve    g4d_triangulate_device_noalloc: points already on the GPU, the mesh written into the
           program's device buffers; small sets, where launches and host round trips count.
  host     g4d_triangulate: points in host memory, the mesh copied out of the context's buffers into
           the program's arrays.
  device   g4d_triangulate_device on HBM-resident points, plain or with the learned proposal, then
           g4d_copy_result into the program's page-locked buffers.
  batch    g4d_triangulate_batch: many independent sets in one call, host to host.

A program keeps one context and feeds it one input after another, so the states of one case share
a context; every state has inputs and output buffers of its own.  The number of tetrahedra depends
on the points, so output buffers have room to spare, whose rows stay -1.

Distributions (`points`): uniform in the unit cube; gauss, one Gaussian; clustered, 70 % in Gaussian
clusters of very different widths over a uniform background; hard, half in tight clusters and a
quarter each on a sphere and on a lattice, where spheres are degenerate and the exact predicates
and their tie-breaking decide.
"""
import ctypes
import json
import math

import numpy as np
import torch

import gstar4d_amd as g
from gstar4d_amd import proposal

TETS_PER_POINT = 6.7   # of a large set in three dimensions
INSPHERE_FLOPS = 111   # one filtered in-sphere test, one for each pair of neighbours


def listed():
    return [
        # The smallest mesh that a service is asked for: latency of the call.
        dict(name="serve_1k", call="serve", n=1000, grid=32, points="uniform", adjacency=True),
        # The most points that the allocation-free call takes, denser in the middle.
        dict(name="serve_16k", call="serve", n=16384, grid=64, points="gauss", adjacency=True),
        # A small odd-sized set in host memory, tetrahedra only.
        dict(name="host_7k", call="host", n=7321, grid=56, points="gauss", adjacency=False),
        # The 100,000-point uniform workload of the benchmark, from host memory and back.
        dict(name="host_100k", call="host", n=100000, grid=128, points="uniform", adjacency=True),
        # Scans and CAD points: spheres and lattices, degenerate throughout.
        dict(name="device_hard_30k", call="device", n=30000, grid=96, points="hard", adjacency=True, learned=False),
        # Ordinary sizes on the GPU, in Morton order, tetrahedra only.
        dict(name="device_300k", call="device", n=300007, grid=192, points="uniform", adjacency=False, learned=False,
             order="morton"),
        # Clustered points without the proposal network: stars grow far beyond their first neighbours.
        dict(name="device_clustered_1m", call="device", n=1000000, grid=256, points="clustered", adjacency=True,
             learned=False),
        # The 4,194,304-point uniform workload of the benchmark.
        dict(name="device_4m", call="device", n=4194304, grid=512, points="uniform", adjacency=True, learned=False),
        # Large clustered sets with the learned proposal.
        dict(name="device_clustered_4m_learned", call="device", n=4000000, grid=512, points="clustered", adjacency=True,
             learned=True),
        # Very many small sets at once.
        dict(name="batch_512x1k", call="batch", sets=512, lo=500, hi=2000, points="mixed", adjacency=True),
        # The benchmark's batch of sets of very different sizes, a part of it.
        dict(name="batch_64x200k", call="batch", sets=64, lo=1000, hi=200000, points="mixed", adjacency=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, n, lo, hi):
    """A grid of 8 to 48 voxels a point, as the benchmark's configurations and the autotuner choose."""
    return max(lo, min(hi, int(round((n * math.exp(rng.uniform(math.log(8), math.log(48)))) ** (1 / 3)))))


def draw(rng):
    call = rng.choice(("serve", "host", "device", "device", "learned", "batch"))
    if call == "serve":
        n = _log_uniform(rng, 1000, 16384)  # clusters of very different widths need more of its scratch
        return dict(call="serve", n=n, grid=_grid(rng, n, 24, 96),
                    points=rng.choice(("uniform", "gauss", "clustered") if n < 4000 else ("uniform", "gauss")),
                    adjacency=rng.random() < 0.7)
    if call == "host":
        n = _log_uniform(rng, 1000, 200000)
        return dict(call="host", n=n, grid=_grid(rng, n, 32, 160),
                    points=rng.choice(("uniform", "gauss", "clustered", "hard") if n < 30000 else
                                      ("uniform", "gauss", "clustered")), adjacency=rng.random() < 0.7)
    if call == "batch":
        lo = _log_uniform(rng, 200, 2000)
        hi = _log_uniform(rng, 2 * lo, 100 * lo)
        return dict(call="batch", sets=min(_log_uniform(rng, 16, 512), max(16, 4000000 // hi)), lo=lo, hi=hi,
                    points="mixed", adjacency=rng.random() < 0.7)
    n = _log_uniform(rng, 100000, 4000000)
    learned = call == "learned"
    points = "clustered" if learned else rng.choice(("uniform", "uniform", "gauss", "clustered"))
    if points in ("gauss", "clustered") and not learned:
        n = min(n, 1000000 - rng.randrange(300000))
    return dict(call="device", n=n, grid=_grid(rng, n, 96, 512), points=points, adjacency=rng.random() < 0.7,
                learned=learned, order=rng.choice(("input", "morton")))


# ---- inputs ----

def _clusters(n, centres, sigmas, gen):
    """n points of Gaussian clusters, drawn again until inside the unit cube."""
    which = torch.randint(centres.shape[0], (n,), generator=gen, device="cuda")
    out = torch.empty((n, 3), dtype=torch.float64, device="cuda")
    todo = torch.arange(n, device="cuda")
    while todo.numel():
        k = which[todo]
        p = centres[k] + sigmas[k, None] * torch.randn((todo.numel(), 3), generator=gen, dtype=torch.float64, device="cuda")
        ok = ((p >= 0) & (p < 1)).all(1)
        out[todo[ok]] = p[ok]
        todo = todo[~ok]
    return out


def _points(kind, n, gen):
    def uniform(*shape):
        return torch.rand(shape, generator=gen, dtype=torch.float64, device="cuda")

    if kind == "uniform":
        return uniform(n, 3)
    if kind == "gauss":
        return _clusters(n, torch.full((1, 3), 0.5, dtype=torch.float64, device="cuda"),
                         torch.full((1,), 0.1, dtype=torch.float64, device="cuda"), gen)
    if kind == "clustered":
        k = max(4, min(256, n // 4000))
        few = int(round(0.3 * n))
        sigmas = 0.002 * (0.05 / 0.002) ** uniform(k)
        return torch.cat([_clusters(n - few, uniform(k, 3), sigmas, gen), uniform(few, 3)])
    part = n // 4
    side = math.ceil((1.03 * part) ** (1 / 3))
    cell = torch.randperm(side ** 3, generator=gen, device="cuda")[:part]
    lattice = torch.stack([cell // (side * side), cell // side % side, cell % side], 1).double() / side
    ball = torch.randn((part, 3), generator=gen, dtype=torch.float64, device="cuda")
    ball = 0.5 + 0.4 * ball / ball.norm(dim=1, keepdim=True)
    tight = torch.full((64,), 0.01, dtype=torch.float64, device="cuda")
    return torch.cat([_clusters(n - 2 * part, uniform(64, 3), tight, gen), ball, lattice])


def _set_sizes(case):
    """Sizes of a batch's sets, spread evenly over the logarithm of their range."""
    s, r = case["sets"], math.log(case["hi"] / case["lo"])
    return [int(case["lo"] * math.exp(r * ((k * 0.6180339887498949) % 1.0))) for k in range(s)]


# ---- the program's side ----

def _ptr(a, kind=ctypes.c_int32):
    """A tensor's or an array's memory, for the C ABI; NULL for none."""
    at = None if a is None else a.ctypes.data if isinstance(a, np.ndarray) else a.data_ptr()
    return ctypes.cast(ctypes.c_void_p(at), ctypes.POINTER(kind))


def _view(at, shape):
    return torch.from_numpy(np.ctypeslib.as_array(at, shape=shape))


class Session:
    """A program's context."""

    def __init__(self, grid, adjacency, morton, learned):
        self.lib = g.load_library()
        opt = g.Options()
        self.lib.g4d_default_options(ctypes.byref(opt))
        opt.grid_size, opt.compute_adjacency, opt.index_space = grid, int(adjacency), int(morton)
        self.ctx = ctypes.c_void_p()
        if self.lib.g4d_create(ctypes.byref(self.ctx), ctypes.byref(opt)):
            raise RuntimeError("no context")
        if learned:
            params, threshold, _ = proposal.load_weights()
            p = np.ascontiguousarray(params, dtype=np.float32).reshape(-1)
            self.ok(self.lib.g4d_set_proposal(self.ctx, _ptr(p, ctypes.c_float), p.shape[0], float(threshold), 1))

    def ok(self, status):
        if status:
            raise RuntimeError(self.lib.g4d_last_error(self.ctx).decode())

    def room(self, nt, tets):
        if nt > tets.shape[0]:
            raise RuntimeError("%d tetrahedra, room for %d" % (nt, tets.shape[0]))
        return nt

    def serve(self, xyz, tets, opp, perm):
        nt = ctypes.c_int64(0)
        self.ok(self.lib.g4d_triangulate_device_noalloc(
            self.ctx, xyz.data_ptr(), xyz.shape[0], tets.data_ptr(), None if opp is None else opp.data_ptr(),
            tets.shape[0], perm.data_ptr(), ctypes.byref(nt), None))
        return nt.value, tets, opp, perm

    def device(self, xyz, tets, opp, perm):
        nt = ctypes.c_int64(0)
        self.ok(self.lib.g4d_triangulate_device(self.ctx, xyz.data_ptr(), xyz.shape[0], ctypes.byref(nt)))
        self.room(nt.value, tets)
        self.ok(self.lib.g4d_copy_result(self.ctx, _ptr(tets), _ptr(opp), _ptr(perm)))
        return nt.value, tets, opp, perm

    def host(self, xyz, tets, opp, perm):
        r = g.Result()
        self.ok(self.lib.g4d_triangulate(self.ctx, _ptr(xyz, ctypes.c_double), xyz.shape[0], ctypes.byref(r)))
        self.take(r, tets, opp)
        perm.copy_(_view(r.perm, tuple(perm.shape)))
        return r.num_tets, tets, opp, perm

    def batch(self, xyz, offsets, tets, opp, tet_offsets):
        r = g.BatchResult()
        self.ok(self.lib.g4d_triangulate_batch(self.ctx, _ptr(xyz, ctypes.c_double), _ptr(offsets, ctypes.c_int64),
                                               offsets.shape[0] - 1, None, ctypes.byref(r)))
        self.take(r, tets, opp)
        tet_offsets.copy_(_view(r.tet_offsets, tuple(tet_offsets.shape)))
        return r.num_tets, tets, opp, tet_offsets

    def take(self, r, tets, opp):
        """The result out of the context's memory, which its next call reuses."""
        nt = self.room(r.num_tets, tets)
        tets[:nt].copy_(_view(r.tets, (nt, 4)))
        if opp is not None:
            opp[:nt].copy_(_view(r.opp, (nt, 4)))

    def __del__(self):
        if self.ctx:
            self.lib.g4d_destroy(self.ctx)


_KEPT = {}  # the context of the case at hand


def _session(case):
    key = json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True)
    if key not in _KEPT:
        _KEPT.clear()
        _KEPT[key] = Session(case.get("grid", 64), case["adjacency"], case.get("order") == "morton",
                             case.get("learned", False))
    return _KEPT[key]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    call = case["call"]
    args = []
    if call == "batch":
        sizes = _set_sizes(case)
        xyz = torch.cat([_points("gauss" if k % 2 else "uniform", n, gen) for k, n in enumerate(sizes)])
        args = [np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)]
    else:
        xyz = _points(case["points"], case["n"], gen).contiguous()
    n = xyz.shape[0]
    room = 7 * n + 1024
    if call in ("host", "batch"):
        xyz = xyz.cpu().numpy()
    where = dict(device="cuda") if call == "serve" else dict(pin_memory=True) if call == "device" else {}
    tets = torch.empty((room, 4), dtype=torch.int32, **where).fill_(-1)
    opp = torch.empty((room, 4), dtype=torch.int32, **where).fill_(-1) if case["adjacency"] else None
    if call == "batch":
        last = torch.zeros(case["sets"] + 1, dtype=torch.int64)
    else:
        last = torch.empty(n, dtype=torch.int32, **where).fill_(-1)
    return dict(call=getattr(_session(case), call), args=[xyz] + args + [tets, opp, last])


def run(state):
    return state["call"](*state["args"])


def work(case):
    """Points read, mesh (and order) written; an in-sphere test for each pair of neighbours."""
    n = sum(_set_sizes(case)) if case["call"] == "batch" else case["n"]
    tets = TETS_PER_POINT * n
    order = 0 if case["call"] == "batch" else 4 * n
    return {"bytes": 24 * n + 16 * tets * (2 if case["adjacency"] else 1) + order, "flops": 2 * tets * INSPHERE_FLOPS}
