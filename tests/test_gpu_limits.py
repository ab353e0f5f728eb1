"""GPU: inputs at the edges of number ranges and sizes, through the C ABI."""
import numpy as np
import pytest

import gstar4d_amd as g

pytestmark = pytest.mark.gpu


# ---------------------------------------------------------------- coordinates that underflow

def _cubes(rng, count):
    """Tuples of five corners of the unit cube (cospherical, so that the filters leave them open), the
    position of a zero coordinate in each, and ids."""
    corners = np.array([[(k >> c) & 1 for c in range(3)] for k in range(8)], np.float64)
    t, at = [], []
    while len(t) < count:
        q = corners[rng.permutation(8)[:5]]
        i, c = rng.integers(5), rng.integers(3)
        if q[i, c] == 0.0:
            t.append(q)
            at.append((i, c))
    idx = np.array([rng.permutation(10 ** 6)[:5] for _ in t], np.int32)
    return np.array(t), at, idx


# the tuple's scale 2^big, and a coordinate 2^low in place of a zero: below 2^(big - 1135) it vanishes on
# the scale that makes the largest coordinate fit 61 bits
@pytest.mark.parametrize("big,low", [(62, -1074), (100, -1074), (200, -936), (200, -960), (200, -1074), (300, -900),
                                     (1000, -300), (1000, -1074), (0, -126), (0, -1074)])
@pytest.mark.parametrize("mode", [0, 1])
def test_coordinate_that_vanishes_on_the_common_scale_is_refused(tri, orc, mode, big, low):
    """Coordinates that span more than the exact arithmetic's 125 bits are refused, also when scaling
    the small one underflows to zero; the same tuple with a true zero there is decided."""
    t, at, idx = _cubes(np.random.default_rng(big), 40)
    ref = [orc.orient4_sos(t[j], idx[j]) for j in range(t.shape[0])]
    t = t * 2.0 ** big
    sign, depth = tri.diag_orient4(t.reshape(-1, 15), idx, mode=mode)
    assert (sign == np.array([r[0] for r in ref])).all()
    assert (depth == np.array([r[1] for r in ref])).all()
    for sgn in (1.0, -1.0):
        for j, (i, c) in enumerate(at):
            q = t[j].copy()
            q[i, c] = sgn * 2.0 ** low
            with pytest.raises(g.G4DError, match="PREDICATE_RANGE"):
                tri.diag_orient4(q.reshape(1, 15), idx[j:j + 1], mode=mode)


def test_triangulation_of_coordinates_that_underflow_is_refused():
    x = np.array([[i, j, k] for i in range(4) for j in range(4) for k in range(4)], np.float64) * 2.0 ** 200
    x[0, 1] = 2.0 ** -960
    with g.Triangulator(grid_size=16) as t:
        with pytest.raises(g.G4DError, match="PREDICATE_RANGE"):
            t.triangulate(x)


# ---------------------------------------------------------------- the plan of a splaying pass

def _plan(vnum, hnum, keys):
    """Stars with keys, and their sizes (vertices, triangle words, history), in whole numbers."""
    star, count = np.unique(keys >> np.uint64(32), return_counts=True)
    star = star.astype(np.int64)
    v = vnum[star].astype(np.int64) + count
    t = np.where(v >= 4, 2 * v - 4, 4)
    return star, v, np.where(v >= 512, 2 * t, t), hnum[star].astype(np.int64) + count


@pytest.mark.parametrize("stars,keys,small", [(1, 2, True), (1, 5000, False), (63, 130, True), (1025, 2050, True),
                                              (4095, 4096, True), (4096, 4096, True), (4096, 4096, False),
                                              (4097, 4100, False), (9000, 30000, False)])
@pytest.mark.parametrize("links", [20, 131073, 1 << 27])
def test_pass_plan_sizes(tri, stars, keys, small, links):
    """Regions of a pass's stars are next to each other, in some order, from the arenas' tops on, also
    where a tile's words pass 2^31 (4,096 stars of 131,074 vertices) and 2^41."""
    rng = np.random.default_rng(stars + links)
    n = stars + stars // 2 + 1
    own = rng.permutation(n)[:stars]
    k = np.concatenate([own, rng.choice(own, keys - stars)]).astype(np.uint64) << np.uint64(32)
    k = np.sort(k) + np.arange(keys, dtype=np.uint64)
    vnum = links + rng.integers(0, 20, n)
    hnum = 3 * vnum
    base = np.array([7, 1 << 33, 1 << 40])
    off, plan = tri.diag_pass_plan(vnum, hnum, k, base, small)
    star, v, t, h = _plan(vnum, hnum, k)
    assert plan[0] == star.shape[0]
    assert (plan[1:4] == [v.sum(), t.sum(), h.sum()]).all()
    for a, size in enumerate((v, t, h)):
        o = off[a][star]
        order = np.argsort(o)
        assert o[order[0]] == base[a]
        assert (np.diff(o[order]) == size[order][:-1]).all()
    rest = np.setdiff1d(np.arange(n), star)
    assert (off[:, rest] == -1).all()
    # a pass of at most 6,144 keys puts 64 and 128 vertices on the 256-vertex list
    merged = keys <= 6144
    tiers = [(32, 32), (32, 32), (32, 256)] if merged else [(32, 64), (64, 128), (128, 256)]
    tiers += [(256, 512), (512, 1024), (1024, 1 << 62)]
    assert list(plan[4:10]) == [int(((v > a) & (v <= b)).sum()) for a, b in tiers]
    assert plan[10] == (v > 64).sum()
    assert plan[11] == (v.max() if v.max() > 1024 else 0)


# ---------------------------------------------------------------- a full device

def _clumps(seed, count, each):
    rng = np.random.default_rng(seed)
    return np.concatenate([c + 1e-3 * rng.normal(size=(each, 3)) for c in rng.random((count, 3))])


def _bigger(kind):
    """A set after _clumps(5, 25, 1600) that needs larger buffers, with and without a repack."""
    return _clumps(6, 25, 3200) if kind == "clumps" else np.random.default_rng(6).random((120000, 3))


@pytest.mark.parametrize("kind", ["clumps", "uniform"])
def test_kept_arenas_are_given_back_when_the_device_is_full(kind):
    """After a repack a context keeps the arenas it has left.  An allocation that finds the memory full, at
    any place of the next call, gives them back and goes on: the same tetrahedra as a new context."""
    first, x = _clumps(5, 25, 1600), _bigger(kind)
    with g.Triangulator(grid_size=64) as t:
        want = t.triangulate(x)[:2]
    for at in range(1, 200, 3):
        with g.Triangulator(grid_size=64) as t:
            t.triangulate(first)
            assert t.stats()["store_repacks"] >= 1 and t.diag_fail_alloc(at)[1] > 0
            got = t.triangulate(x)[:2]
            left, _ = t.diag_fail_alloc(0)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), at
        if left:
            break  # the call allocates less often
    assert left and at > 10


def test_full_device_without_kept_arenas_is_an_error_once(orc):
    x = np.random.default_rng(8).random((4000, 3))
    ref, _, _ = orc.triangulate(x, 32)
    with g.Triangulator(grid_size=32) as t:
        for at in (1, 5, 20):
            assert t.diag_fail_alloc(at)[1] == 0
            with pytest.raises(g.G4DError) as e:
                t.triangulate(x)
            assert e.value.status == "OOM"
        tets, _, _ = t.triangulate(x)
        assert (g.canonical(tets) == ref).all()


# ---------------------------------------------------------------- statistics

def test_star_kernel_statistics_are_the_32_vertex_kernels():
    """Evaluations and cofactors of the 32-vertex kernel are the same whether the larger stars run in the
    LDS kernels or, by a lowered limit, in the global-memory kernel; the default variant leaves out
    the late passes, which share a launch."""
    x = np.concatenate([_clumps(9, 10, 800), np.random.default_rng(9).random((4000, 3))])
    def run(variant, limit):
        with g.Triangulator(grid_size=32, lds_star_limit=limit) as t:
            t.set_star_kernel(variant)
            t.triangulate(x)
            return t.stats()
    for variant in (0, 1, 2, 4):
        a, b = run(variant, 0), run(variant, 32)
        assert a["big_stars"] > 0 and b["huge_stars"] > a["huge_stars"]
        assert a["star_t0_launches"] == a["star_passes"] == b["star_passes"] == b["star_t0_launches"]
        assert a["star_t0_filter_evals"] == b["star_t0_filter_evals"] > 0
        assert a["star_t0_cofactors"] == b["star_t0_cofactors"] > 0
    c = run(-1, 0)
    assert 0 < c["star_t0_launches"] < c["star_passes"] == a["star_passes"]
    d = run(2, 0)
    assert 0 < c["star_t0_filter_evals"] < d["star_t0_filter_evals"]
    assert 0 < c["star_t0_cofactors"] < d["star_t0_cofactors"]


# ---------------------------------------------------------------- which kernel builds a star

@pytest.mark.parametrize("k,tier", [(16, "32"), (48, "64"), (96, "128"), (190, "256"), (380, "512"), (760, "1024"),
                                    (1500, "global")])
def test_star_of_each_size_is_built_by_its_kernel(orc, k, tier):
    """The centre of a shell of k points has most of them in its workset and the rest in its next passes:
    link and insertions come to k in one of them, k lies inside the tier, and no star needs more.
    Enough other points that the first pass does not merge its tiers."""
    rng = np.random.default_rng(k)
    shell = rng.normal(size=(k, 3))
    shell *= (0.3 + 0.001 * rng.random((k, 1))) / np.linalg.norm(shell, axis=1)[:, None]
    x = np.concatenate([[[0.5, 0.5, 0.5]], 0.5 + shell, rng.random((1500, 3)) * 0.15])
    with g.Triangulator(grid_size=128) as t:
        tets, _, _ = t.triangulate(x)
        n = t.diag_star_tiers()
        st = t.stats()
    ref, _, _ = orc.triangulate(x, 128)
    assert (g.canonical(tets) == ref).all()
    assert n[tier] >= 1
    wide = ("512", "1024", "global")
    assert st["huge_stars"] == sum(n[c] for c in wide)
    assert all(n[c] == 0 for c in wide[wide.index(tier) + 1 if tier in wide else 0:])


@pytest.mark.parametrize("norm,points,tier", [(314, 312, "512"), (614, 408, "512"), (1361, 720, "1024")])
def test_inconclusive_wide_star_is_handed_on(orc, norm, points, tier):
    """Whole points at one distance from the origin, and the origin: its star has a link of all of them and
    only zero determinants, so the wide kernel gives it to the global-memory one."""
    r = int(norm ** 0.5)
    a = np.arange(-r, r + 1)
    x = np.stack(np.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
    x = np.concatenate([x[(x * x).sum(1) == norm], [[0, 0, 0]]]).astype(np.float64)
    assert x.shape[0] == points + 1
    with g.Triangulator(grid_size=128) as t:
        tets, _, _ = t.triangulate(x)
        n = t.diag_star_tiers()
    ref, _, _ = orc.triangulate(x, 128)
    assert g.canonical(tets).shape == ref.shape and (g.canonical(tets) == ref).all()
    assert n[tier] >= 1 and n["wide_exact"] >= 1


def test_small_rounds_take_the_short_way(orc):
    """Late passes of a general set take one launch and are followed without the host's look; a set
    whose stars need exact predicates throughout never is."""
    rng = np.random.default_rng(3)
    with g.Triangulator(grid_size=32) as t:
        x = rng.random((1000, 3))
        tets, _, _ = t.triangulate(x)
        n = t.diag_star_tiers()
        assert (g.canonical(tets) == orc.triangulate(x, 32)[0]).all()
        assert n["ahead_passes"] >= 1 and n["exact"] == n["wide_exact"] == n["global"] == 0
        lattice = np.stack(np.meshgrid(*[np.arange(9.0)] * 3, indexing="ij"), -1).reshape(-1, 3)
        tets, _, _ = t.triangulate(lattice)
        n = t.diag_star_tiers()
        assert (g.canonical(tets) == orc.triangulate(lattice, 32)[0]).all()
        assert n["exact"] > 0
