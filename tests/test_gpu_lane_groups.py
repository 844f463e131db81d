"""Sparse catalogues, whose runs of 16 objects are held by four groups of lanes
(reported as tiles of 128), with every kind of table: integer, hybrid in LDS,
hybrid found by searching the edges, and too long for LDS beside the groups'
chunks -- against the oracle (counts identical, weighted counts within 1e-12
relative)."""
import numpy as np
import pytest

import fcfc_amd as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu
L = 1000.0
HYBRID = np.geomspace(20.2, 190, 11)               # 2232 table entries
SEARCHED = np.geomspace(0.1, 40, 25)               # 102400 or more: beyond LDS


@pytest.fixture(scope="module")
def eng():
    with F.Engine() as e:
        yield e


def _oracle(b, A, B, weighted):
    ob = O.oracle_bins(b.bintype, b.s2bin, b.nmu, b.pbin if b.bintype == F.BIN_SPI else None)
    w = lambda c: (c.x, c.y, c.z, c.s, c.w if weighted else None)
    g, bs, var, mask = (0, b.bsize_rescaled, 1, 0b11111) if b.geometry == F.GEOM_BOX else (1, None, 0, 0b111111)
    ref, cen = O.count(g, bs, w(A), None if B is None else w(B), B is None, ob, variant=var,
                       census_mask=0 if weighted else mask, weighted=weighted)
    assert weighted or cen == 0
    return ref


def _points(rng, n, o):
    """Half uniform, half in clumps of 30 (pairs at every separation)."""
    k = n // 60
    c = (rng.uniform(20, L - 20, (k, 1, 3)) + rng.normal(0, 6, (k, 30, 3))).reshape(-1, 3)
    p = np.concatenate([np.clip(c, 0, L - 1e-6), rng.uniform(0, L, (n - len(c), 3))])
    return (o + p).T


def _check(eng, b, A, B, tile, what):
    rng = np.random.default_rng(1)
    g = rng.uniform(-1, 1, b.ntot)
    for X in (None, B):
        ref, refw = _oracle(b, A, X, False), _oracle(b, A, X, True)
        for prec in ("fp64", "fp32"):
            print(f"case lane groups {what} auto={X is None} {prec}", flush=True)
            np.testing.assert_array_equal(eng.count_pairs(A, X, b, isauto=X is None, precision=prec), ref)
            assert eng.stats()["tile"] == tile
            np.testing.assert_allclose(eng.count_pairs(A, X, b, isauto=X is None, withwt=True, precision=prec),
                                       refw, rtol=1e-12, atol=0)
            assert eng.stats()["tile"] == tile
        ga, gb = eng.count_backward(A, X, b, g, isauto=X is None)
        # each pair weight appears in both sides' gradients
        tot, mag = (2 if X is None else 1) * (g @ refw), 2 * np.abs(g) @ refw
        np.testing.assert_allclose(ga @ A.w, tot, rtol=0, atol=1e-12 * mag)
        if X is not None:
            np.testing.assert_allclose(gb @ B.w, tot, rtol=0, atol=1e-12 * mag)


@pytest.mark.parametrize("geom,bt", [(F.GEOM_BOX, F.BIN_ISO), (F.GEOM_BOX, F.BIN_SMU), (F.GEOM_BOX, F.BIN_SPI),
                                     (F.GEOM_SURVEY, F.BIN_ISO), (F.GEOM_SURVEY, F.BIN_SMU)])
@pytest.mark.parametrize("kind", ["hybrid", "searched"])
def test_hybrid_tables(eng, geom, bt, kind):
    rng = np.random.default_rng(5)
    e = HYBRID if kind == "hybrid" else SEARCHED
    b = F.Bins.edges(geom, bt, e, nmu=12 if bt == F.BIN_SMU else 1,
                     pedges=np.linspace(0, 40, 11) if bt == F.BIN_SPI else None,
                     bsize=L if geom == F.GEOM_BOX else None)
    assert b.tabtype == 1 and (b._b.stab_len < 20000 if kind == "hybrid" else b._b.stab_len > 40000)
    o = 0.0 if geom == F.GEOM_BOX else 600.0
    A, B = (F.Catalog(b, *_points(rng, n, o), rng.uniform(0.5, 2, n)) for n in (1501, 2203))
    _check(eng, b, A, B, 128, f"geom={geom} bt={bt} {kind}")


@pytest.mark.parametrize("smax,tile", [(130, 128), (190, 512)])
def test_integer_tables(eng, smax, tile):
    """A table of 68 KB leaves room for the groups' chunks, one of 144 KB does
    not: runs of 64 objects then, and the table stays."""
    rng = np.random.default_rng(6)
    b = F.Bins.linear(F.GEOM_BOX, F.BIN_ISO, 0, smax, 1, bsize=L)
    assert b.tabtype == 0 and b._b.stab_len == smax ** 2
    A, B = (F.Catalog(b, *_points(rng, n, 0.0), rng.uniform(0.5, 2, n)) for n in (1501, 2203))
    ref = [_oracle(b, A, X, False) for X in (None, B)]
    for X, r in zip((None, B), ref):
        print(f"case lane groups integer smax={smax} auto={X is None}", flush=True)
        np.testing.assert_array_equal(eng.count_pairs(A, X, b, isauto=X is None), r)
        assert eng.stats()["tile"] == tile
