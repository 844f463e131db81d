"""Pairs below a separation range that starts above zero: coincident objects
and pairs closer than the FP32 resolution belong to no bin and must leave
every bin as it is -- against the oracle (counts identical, weighted counts
within 1e-12 relative)."""
import numpy as np
import pytest

import fcfc_amd as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu
L = 1000.0


@pytest.fixture(scope="module")
def eng():
    with F.Engine() as e:
        yield e


def _bins(geom, hyb, ns, nmu):
    bs = L if geom == F.GEOM_BOX else None
    if hyb:
        return F.Bins.edges(geom, F.BIN_SMU, np.geomspace(20.2, 190, ns + 1), nmu=nmu, bsize=bs)
    return F.Bins.linear(geom, F.BIN_SMU, 20, 20 + 5 * ns, 5, nmu=nmu, bsize=bs)


def _oracle(b, A, B, weighted):
    ob = O.oracle_bins(b.bintype, b.s2bin, b.nmu)
    w = lambda c: (c.x, c.y, c.z, c.s, c.w if weighted else None)
    g, bs, var = (0, b.bsize_rescaled, 1) if b.geometry == F.GEOM_BOX else (1, None, 0)
    return O.count(g, bs, w(A), None if B is None else w(B), B is None, ob, variant=var,
                   weighted=weighted)[0]


@pytest.mark.parametrize("geom", [F.GEOM_BOX, F.GEOM_SURVEY])
@pytest.mark.parametrize("hyb", [False, True])
@pytest.mark.parametrize("ns,nmu", [(1, 2), (2, 126), (5, 9), (6, 20), (39, 100)])
def test_coincident_pairs(eng, geom, hyb, ns, nmu):
    """500 objects counted against themselves at the same places (as a second
    catalogue) and against copies 1e-9 apart: the FP32 (s, mu) forms cannot
    bin such a pair (its mu estimate is 0 * inf) and re-evaluate every one."""
    rng = np.random.default_rng(ns)
    b = _bins(geom, hyb, ns, nmu)
    assert b.tabtype == (1 if hyb else 0) and b._b.soff > 0
    n = 500
    o = 0.0 if geom == F.GEOM_BOX else 600.0
    p, w = o + rng.uniform(1, L - 1, (3, n)), rng.uniform(0.5, 2, n)
    A = F.Catalog(b, *p, w)
    B = F.Catalog(b, *p, w[::-1].copy())
    C = F.Catalog(b, *(p + 1e-9), w)
    D = F.Catalog(b, *np.concatenate([p, p], axis=1), np.concatenate([w, w]))
    for what, X, Y in (("same places", A, B), ("1e-9 apart", A, C), ("auto, every object twice", D, None)):
        ref, refw = _oracle(b, X, Y, False), _oracle(b, X, Y, True)
        for prec in ("fp64", "fp32", "plain"):
            print(f"case below range geom={geom} hyb={hyb} ns={ns} nmu={nmu} {what} {prec}", flush=True)
            got = eng.count_pairs(X, Y, b, isauto=Y is None, precision=prec)
            re = eng.stats()["rechecked"]
            np.testing.assert_array_equal(got, ref)
            gotw = eng.count_pairs(X, Y, b, isauto=Y is None, withwt=True, precision=prec)
            rew = eng.stats()["rechecked"]
            np.testing.assert_allclose(gotw, refw, rtol=1e-12, atol=0)
            if prec == "fp32":
                assert min(re, rew) >= n
