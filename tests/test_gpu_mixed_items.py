"""Mixed Plummer gravity at the sizes where its launch changes: one contiguous
unit of records per part or tiles of 256 dealt out to the parts, blocks that
take items from the queues or one block per item, and 2, 3, 4 or 6 of them per
CU.  Accelerations and potentials of sampled particles against an FP64 direct
sum over the same (split) positions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# tiles in place of units from 512 records per part on (8 parts below 8 192
# particles: 3 585; 24 parts above: 10 753); queues below 196 608
@pytest.mark.parametrize("n", [3, 64, 257, 1000, 3583, 3585, 8191, 8193, 10751, 10753, 20479, 20481, 28673, 57343, 57345, 65536, 196607,
                               196609])
def test_items_cover_every_pair(cs, n):
    print(f"mixed gravity items n={n}", flush=True)
    e = cs.make_engine("mixed", 2, n, 7, ph_sort=True)
    for _ in range(2):   # the second evaluation starts from cleared queues
        e.run_pass(cs.GRAVITY)
    got = e.get("grav")[:n].astype(np.float64)
    x = e.get("pos64")[:n, :3]
    m = e.get("vel")[:n, 3].astype(np.float64)
    eps2 = float(cs.preset_params(2, n).grav_eps) ** 2
    e.close()
    pick = np.unique(np.linspace(0, n - 1, min(n, 96)).astype(int))
    for i in pick:
        r = x[i] - x
        inv = 1.0 / np.sqrt((r * r).sum(1) + eps2)
        a = -(m * inv ** 3)[:, None] * r
        # a pair's FP32 arithmetic is within 16 roundings (2^-24 each: the
        # expanded r^2 loses up to 4 in each of its 3), and the sums are
        # compensated, so the error is within 2^-20 of the terms' magnitudes
        assert np.linalg.norm(got[i, :3] - a.sum(0)) <= 2.0 ** -20 * np.linalg.norm(a, axis=1).sum(), i
        assert abs(got[i, 3] + (m * inv).sum()) <= 2.0 ** -20 * (m * inv).sum(), i
