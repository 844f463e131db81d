"""Runs of A objects per wavefront: remainders of 16, 64 and 128 objects, long
sparse columns across the periodic boundary, 32-bit counters beyond 2^32 pairs
and job changes of few workgroups -- against the oracle (counts identical,
weighted counts within 1e-12 relative)."""
import numpy as np
import pytest

import fcfc_amd as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu
L = 1000.0
FORMS = ("fp64", "fp32", "plain")


@pytest.fixture(scope="module")
def eng():
    with F.Engine() as e:
        yield e


def _oracle(b, A, B, isauto, weighted, tied=False):
    ob = O.oracle_bins(b.bintype, b.s2bin, b.nmu, b.pbin if b.bintype == F.BIN_SPI else None)
    a = (A.x, A.y, A.z, A.s, A.w if weighted else None)
    c = None if isauto else (B.x, B.y, B.z, B.s, B.w if weighted else None)
    g, bs, var, mask = ((0, b.bsize_rescaled, 1, 0b11111) if b.geometry == F.GEOM_BOX
                        else (1, None, 0, 0b111111))
    ref, cen = O.count(g, bs, a, c, isauto, ob, variant=var, census_mask=0 if weighted else mask,
                       weighted=weighted)
    assert weighted or tied or cen == 0
    return ref


def _check(eng, b, A, B, what, tied=False):
    for isauto in (True, False):
        ref = _oracle(b, A, B, isauto, False, tied)
        refw = _oracle(b, A, B, isauto, True, tied)
        for prec in FORMS:
            print(f"case runs {what} auto={isauto} prec={prec}", flush=True)
            np.testing.assert_array_equal(
                eng.count_pairs(A, None if isauto else B, b, isauto=isauto, precision=prec), ref)
            np.testing.assert_allclose(
                eng.count_pairs(A, None if isauto else B, b, isauto=isauto, withwt=True,
                                precision=prec), refw, rtol=1e-12, atol=0)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128, 129, 255, 257, 1025])
@pytest.mark.parametrize("bt,hyb", [(F.BIN_SMU, False), (F.BIN_SPI, True)])
def test_run_remainders(eng, n, bt, hyb):
    """n objects in one cell column (a clump), so that the last run of the
    column holds the remainder, in one, two and four objects per lane."""
    rng = np.random.default_rng(n)
    ds = 7.3 if hyb else 5.0
    b = F.Bins.linear(F.GEOM_BOX, bt, 0, 20 * ds, ds, nmu=10 if bt == F.BIN_SMU else 1, pmin=0,
                      pmax=100 if bt == F.BIN_SPI else 0, dpi=5, bsize=L)
    A = F.Catalog(b, *(rng.uniform(500, 512, n) for _ in range(3)), rng.uniform(0.5, 2, n))
    B = F.Catalog(b, *(rng.uniform(430, 580, 300) for _ in range(3)), rng.uniform(0.5, 2, 300))
    try:
        for tile in (0, 40, 512, 1024, 2048):
            eng.set_tuning(tile=tile)
            _check(eng, b, A, B, f"n={n} bt={bt} tile={tile}")
    finally:
        eng.set_tuning()


@pytest.mark.parametrize("geom,bt,hyb", [(g, t, h) for g in (F.GEOM_BOX, F.GEOM_SURVEY)
                                         for t in (F.BIN_ISO, F.BIN_SMU, F.BIN_SPI)
                                         for h in (False, True)])
def test_groups_of_lanes(eng, geom, bt, hyb):
    """Runs of 16 and of 5 objects, each held by four groups of lanes, with
    numbers of objects that leave remainders of the runs and of the groups;
    counts, and the gradient by its linearity in the weights."""
    rng = np.random.default_rng(21)
    ds = 7.3 if hyb else 5.0
    box = geom == F.GEOM_BOX
    b = F.Bins.linear(geom, bt, 0, 20 * ds, ds, nmu=10 if bt == F.BIN_SMU else 1, pmin=0,
                      pmax=100 if bt == F.BIN_SPI else 0, dpi=5, bsize=L if box else None)
    o = 0.0 if box else 600.0
    A, B = (F.Catalog(b, *(rng.uniform(o, o + 400, n) for _ in range(3)), rng.uniform(0.5, 2, n))
            for n in (203, 1501))
    g = rng.uniform(-1, 1, b.ntot)
    try:
        for tile in (16, 5):
            eng.set_tuning(tile=tile)
            _check(eng, b, A, B, f"groups geom={geom} bt={bt} hyb={hyb} tile={tile}")
            for X in (None, B):
                ga, gb = eng.count_backward(A, X, b, g, isauto=X is None)
                cnt = eng.count_pairs(A, X, b, isauto=X is None, withwt=True)
                # each pair weight appears in both sides' gradients
                ref = (2 if X is None else 1) * (g @ cnt)
                mag = 2 * np.abs(g) @ cnt
                np.testing.assert_allclose(ga @ A.w, ref, rtol=0, atol=1e-12 * mag)
                if X is not None:
                    np.testing.assert_allclose(gb @ B.w, ref, rtol=0, atol=1e-12 * mag)
    finally:
        eng.set_tuning()


@pytest.mark.parametrize("geom", [F.GEOM_BOX, F.GEOM_SURVEY])
def test_run_spans_the_box(eng, geom):
    """A thin column of 200 objects along z: runs as long as the column, whose
    windows reach both periodic images."""
    rng = np.random.default_rng(7)
    box = geom == F.GEOM_BOX
    b = F.Bins.linear(geom, F.BIN_SMU, 0, 480, 10, nmu=20, bsize=L if box else None)
    o = 0.0 if box else 600.0
    A = F.Catalog(b, rng.uniform(0, 2, 200) + o, rng.uniform(0, 2, 200), rng.uniform(0, L, 200),
                  rng.uniform(0.5, 2, 200))
    B = F.Catalog(b, rng.uniform(0, L, 3000) + o, rng.uniform(0, L, 3000), rng.uniform(0, L, 3000),
                  rng.uniform(0.5, 2, 3000))
    try:
        for cd, zd in ((0, 0), (1, 1), (2, 16)):
            eng.set_tuning(cell_div=cd, zdiv=zd)
            _check(eng, b, A, B, f"span geom={geom} cd={cd} zd={zd}")
    finally:
        eng.set_tuning()


@pytest.mark.parametrize("geom", [F.GEOM_BOX, F.GEOM_SURVEY])
@pytest.mark.parametrize("bt,ns", [(F.BIN_ISO, 1), (F.BIN_ISO, 6), (F.BIN_SMU, 5), (F.BIN_SMU, 6),
                                   (F.BIN_SPI, 5), (F.BIN_SPI, 6)])
def test_ranges_from_above_zero(eng, geom, bt, ns):
    """Odd and even numbers of bins whose range begins above zero, of objects
    on a lattice of the bin width: pairs on both range edges, below and beyond
    them (the oracle's own roundings differ for some survey pairs there: the
    counts are those of its first)."""
    rng = np.random.default_rng(ns)
    b = F.Bins.linear(geom, bt, 20, 20 + 5 * ns, 5, nmu=9 if bt == F.BIN_SMU else 1,
                      pmin=10 if bt == F.BIN_SPI else 0, pmax=35 if bt == F.BIN_SPI else 0, dpi=5,
                      bsize=L if geom == F.GEOM_BOX else None)
    o = 0.0 if geom == F.GEOM_BOX else 600.0
    A, B = (F.Catalog(b, *(o + 5.0 * rng.integers(0, 18, n) for _ in range(3)),
                      rng.uniform(0.5, 2, n)) for n in (500, 1500))
    _check(eng, b, A, B, f"above zero geom={geom} bt={bt} ns={ns}", tied=True)
    # the count is linear in each side's weights: the gradient times them
    g = rng.uniform(-1, 1, b.ntot)
    ga, gb = eng.count_backward(A, B, b, g)
    tot = g @ eng.count_pairs(A, B, b, withwt=True)
    mag = np.abs(g) @ eng.count_pairs(A, B, b, withwt=True)
    np.testing.assert_allclose([ga @ A.w, gb @ B.w], [tot, tot], rtol=0, atol=1e-12 * mag)


def test_counters_beyond_32_bits(eng):
    """4.5e9 pairs of one bin counted by one workgroup: its 32-bit LDS counters
    are flushed before they overflow."""
    n = 95000
    rng = np.random.default_rng(8)
    b = F.Bins.linear(F.GEOM_BOX, F.BIN_ISO, 0, 100, 100, bsize=L)
    A = F.Catalog(b, *(rng.uniform(500, 510, n) for _ in range(3)))
    try:
        eng.set_tuning(nblock=1)
        print("case runs 32-bit counters", flush=True)
        cnt = eng.count_pairs(A, None, b, isauto=True)
    finally:
        eng.set_tuning()
    assert int(cnt.sum()) == n * (n - 1) // 2


@pytest.mark.parametrize("prec", FORMS)
def test_job_changes_of_few_workgroups(eng, prec):
    """Batched jobs of very different sizes (empty ones among them) counted by
    one and three workgroups, whose wavefronts change jobs at different
    times."""
    rng = np.random.default_rng(9)
    b = F.Bins.linear(F.GEOM_BOX, F.BIN_SMU, 0, 150, 5, nmu=20, bsize=L)
    cats = [F.Catalog(b, *(rng.uniform(0, L, n) for _ in range(3)), rng.uniform(0.5, 2, n))
            for n in (0, 1, 40, 700, 3000, 90, 0, 1500)]
    jobs, refs = [], []
    for k, c in enumerate(cats):
        d = cats[(k + 3) % len(cats)]
        for au, wt in ((True, False), (True, True), (False, True), (False, False)):
            jobs.append((c, None if au else d, au, wt))
            refs.append(_oracle(b, c, d, au, wt))
    try:
        for nb in (1, 3, 0):
            eng.set_tuning(nblock=nb)
            print(f"case runs job changes nblock={nb} prec={prec}", flush=True)
            for (c, d, au, wt), r, g in zip(jobs, refs, eng.count_batch(jobs, b, precision=prec)):
                if wt:
                    np.testing.assert_allclose(g, r, rtol=1e-12, atol=0)
                else:
                    np.testing.assert_array_equal(g, r)
    finally:
        eng.set_tuning()
