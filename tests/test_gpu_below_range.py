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


@pytest.mark.parametrize("tile", [0, 16])
@pytest.mark.parametrize("geom,bt", [(g, t) for g in (F.GEOM_BOX, F.GEOM_SURVEY)
                                     for t in (F.BIN_ISO, F.BIN_SMU, F.BIN_SPI)])
def test_gradient_of_infinite_weights(eng, geom, bt, tile):
    """A clump 8 across, counted from 20 on, whose objects have infinite
    weights: they are in no bin with anything, and neither their gradients nor
    the others' may notice."""
    rng = np.random.default_rng(8)
    b = F.Bins.linear(geom, bt, 20, 60, 5, nmu=9 if bt == F.BIN_SMU else 1,
                      pmin=10 if bt == F.BIN_SPI else 0, pmax=40 if bt == F.BIN_SPI else 0, dpi=5,
                      bsize=L if geom == F.GEOM_BOX else None)
    o = 0.0 if geom == F.GEOM_BOX else 600.0
    p = o + np.concatenate([rng.uniform(100, 250, (3, 800)), 800 + rng.uniform(0, 4.6, (3, 70))], axis=1)
    w = np.concatenate([rng.uniform(0.5, 2, 800), np.full(70, np.inf)])
    A, N = F.Catalog(b, *p, w), F.Catalog(b, *p[:, :800], w[:800])
    g = rng.uniform(-1, 1, b.ntot)
    try:
        eng.set_tuning(tile=tile)
        for X, Y in ((None, None), (A, N)):
            print(f"case gradient inf geom={geom} bt={bt} tile={tile} auto={X is None}", flush=True)
            ga, gb = eng.count_backward(A, X, b, g, isauto=X is None)
            na, nb = eng.count_backward(N, Y, b, g, isauto=Y is None)
            assert abs(na).max() > 0
            tol = 1e-12 * np.abs(g).max() * w[:800].sum()
            for got, ref in ((ga, na), (gb, nb)):
                if got is not None:
                    assert not got[800:].any()
                    np.testing.assert_allclose(got[:800], ref, rtol=0, atol=tol)
    finally:
        eng.set_tuning()
