"""Launches of one kernel with different amounts of LDS after each other: in
one engine, in two, and between the replays of a prepared plan."""
import numpy as np
import pytest

import fcfc_amd as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu
L = 1000.0


def _count(eng, b, x):
    c = F.Catalog(b, *x)
    return eng.count_pairs(c, None, b, isauto=True)


def test_lds_sizes_in_turn():
    import torch
    rng = np.random.default_rng(11)
    x = rng.uniform(0, L, (3, 3000))
    big, small = (F.Bins.linear(F.GEOM_BOX, F.BIN_ISO, 0, s, 1, bsize=L) for s in (190, 30))
    assert big._b.stab_len == 36100 and small._b.stab_len == 900     # 144 and 4 KB of LDS
    ref = {}
    for b in (big, small):
        c = F.Catalog(b, *x)
        ref[b] = O.count(0, b.bsize_rescaled, (c.x, c.y, c.z, None, None), None, True,
                         O.oracle_bins(b.bintype, b.s2bin), variant=1)[0]
    with F.Engine() as e1, F.Engine() as e2:
        for e in (e1, e2):
            e.set_tuning(tile=1024)               # the same kernel for all
        dev = [torch.from_numpy(v * big.rescale).cuda() for v in x]
        plan = e1.plan([(F.Catalog(big, *dev), None, True, False)], big)
        for k, (e, b) in enumerate([(e1, big), (e1, small), (e1, big), (e2, small), (e1, big),
                                    (e2, big), (e1, small), (e2, big)]):
            print(f"case lds sequence {k}", flush=True)
            np.testing.assert_array_equal(_count(e, b, x), ref[b])
            np.testing.assert_array_equal(np.asarray(plan.run()[0]), ref[big])
        plan.close()
