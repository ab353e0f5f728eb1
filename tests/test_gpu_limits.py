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
