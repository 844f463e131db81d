"""Survey (s, mu) counts with squared distances |r|^2 that do not belong to the
coordinates: s^2 = |a|^2 + |b|^2 - 2 a.b comes out far below zero for some
pairs, which then belong to no bin and must leave every bin as it is."""
import numpy as np
import pytest

import fcfc_amd as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    with F.Engine() as e:
        yield e


@pytest.mark.parametrize("smin", [0, 3])
@pytest.mark.parametrize("tile", [0, 16, 1024])
def test_squares_too_low(eng, smin, tile):
    """Clumps 200 apart and 30 across; the |r|^2 of half of the objects is 5000
    (beyond the range of s^2) too low, so that only pairs of the others count."""
    rng = np.random.default_rng(3 + smin)
    b = F.Bins.linear(F.GEOM_SURVEY, F.BIN_SMU, smin, 40, 1, nmu=20)
    assert b.rescale == 1 and b.tabtype == 0
    cen = 1000.0 + 200.0 * np.stack(np.meshgrid(*[np.arange(3)] * 3), -1).reshape(-1, 3)
    p = (cen[:, None] + rng.uniform(-15, 15, (27, 40, 3)) / np.sqrt(3)).reshape(-1, 3)
    w = rng.uniform(0.5, 2, len(p))
    low = np.tile(np.arange(40) % 2 == 1, 27)
    s = np.einsum("ij,ij->i", p, p) - 5000.0 * low
    A = F.Catalog(b, *p.T, w, s=s)
    N = F.Catalog(b, *p[~low].T, w[~low])
    ob = O.oracle_bins(b.bintype, b.s2bin, b.nmu)
    ref = [O.count(1, None, (N.x, N.y, N.z, N.s, N.w if wt else None), None, True, ob, variant=0,
                   weighted=wt)[0] for wt in (False, True)]
    g = rng.uniform(-1, 1, b.ntot)
    try:
        eng.set_tuning(tile=tile)
        for prec in ("fp64", "plain"):
            print(f"case survey squares smin={smin} tile={tile} {prec}", flush=True)
            np.testing.assert_array_equal(eng.count_pairs(A, None, b, isauto=True, precision=prec), ref[0])
            np.testing.assert_array_equal(eng.count_pairs(A, A, b, precision=prec).sum(),
                                          2 * ref[0].sum() + (0 if smin else (~low).sum()))
            np.testing.assert_allclose(eng.count_pairs(A, None, b, isauto=True, withwt=True, precision=prec),
                                       ref[1], rtol=1e-12, atol=0)
        ga, _ = eng.count_backward(A, None, b, g, isauto=True)
        gn, _ = eng.count_backward(N, None, b, g, isauto=True)
        assert not ga[low].any()
        np.testing.assert_allclose(ga[~low], gn, rtol=0, atol=1e-12 * np.abs(g).max() * w.sum())
    finally:
        eng.set_tuning()
