"""The statistic `evals`: distances evaluated, without the objects that the
bounding box of a wavefront's A objects drops."""
import numpy as np
import pytest

import fcfc_amd as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32", "plain"])
@pytest.mark.parametrize("tile", [16, 512, 1024])
def test_evals_of_a_point(prec, tile):
    """6400 objects within 1e-6 of a point against 5000 in the cube around the
    sphere of the largest separation: only those inside are evaluated."""
    rng = np.random.default_rng(1)
    b = F.Bins.linear(F.GEOM_BOX, F.BIN_ISO, 0, 100, 10, bsize=1000.0)
    B = 500 + rng.uniform(-100, 100, (3, 5000))
    r = np.sqrt(((B - 500) ** 2).sum(0))
    B = B[:, abs(r - 100) > 1e-3]
    n = int((abs(r) < 100 - 1e-3).sum())
    with F.Engine() as eng:
        eng.set_tuning(tile=tile)
        print(f"case evals tile={tile} {prec}", flush=True)
        A = F.Catalog(b, *(500 + rng.uniform(0, 1e-6, (3, 6400))))
        cnt = eng.count_pairs(A, F.Catalog(b, *B), b, precision=prec)
        assert cnt.sum() == 6400 * n
        assert eng.stats()["evals"] == 6400 * n
