"""Survey catalogues in a plane and on a line: counts against the oracle, and
grids as coarse as their objects ask for."""
import numpy as np
import pytest

import fcfc_amd as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    with F.Engine() as e:
        yield e


def _check(eng, b, p, what):
    rng = np.random.default_rng(2)
    A = F.Catalog(b, *p, rng.uniform(0.5, 2, len(p[0])))
    ob = O.oracle_bins(b.bintype, b.s2bin, b.nmu)
    ref, refw = (O.count(1, None, (A.x, A.y, A.z, A.s, A.w if wt else None), None, True, ob, variant=0,
                         weighted=wt)[0] for wt in (False, True))
    assert ref.sum() > 0
    for prec in ("fp64", "fp32"):
        print(f"case flat {what} {prec}", flush=True)
        np.testing.assert_array_equal(eng.count_pairs(A, None, b, isauto=True, precision=prec), ref)
        np.testing.assert_allclose(eng.count_pairs(A, None, b, isauto=True, withwt=True, precision=prec),
                                   refw, rtol=1e-12, atol=0)
    return eng.stats()["cell_div"]


@pytest.mark.parametrize("bt", [F.BIN_ISO, F.BIN_SMU])
@pytest.mark.parametrize("flat", [(0,), (1,), (2,), (0, 1), (0, 2), (1, 2)])
def test_planes_and_lines(eng, bt, flat):
    """5000 objects in a plane of 500 x 500 or on a line of 5000, to 50: cells
    are sized for two runs of 16 (squares of 40, pieces of 32: one and two
    cells per separation)."""
    rng = np.random.default_rng(1)
    p = 700.0 + rng.uniform(0, 500 if len(flat) == 1 else 5000, (3, 5000))
    for k in flat:
        p[k] = 800.0
    b = F.Bins.linear(F.GEOM_SURVEY, bt, 0, 50, 5, nmu=10 if bt == F.BIN_SMU else 1)
    assert _check(eng, b, p, f"bt={bt} flat={flat}") == len(flat)


def test_plane_through_the_observer(eng):
    """A plane of 3000 x 3000 at z = 0 counted to 1: twelve cells per
    separation would be more than the grid may have."""
    rng = np.random.default_rng(4)
    p = np.stack([rng.uniform(-1500, 1500, 3000), rng.uniform(-1500, 1500, 3000), np.zeros(3000)])
    p[:, 1500:] = p[:, :1500] + rng.uniform(-0.5, 0.5, (3, 1500)) * [[1], [1], [0]]
    _check(eng, F.Bins.linear(F.GEOM_SURVEY, F.BIN_ISO, 0, 1, 0.1), p, "plane z=0")
