"""Mixed Plummer gravity at the sizes where its launch changes: one contiguous
unit of records per part or tiles of 256 dealt out to the parts; pairs taken
once, with odd and even counts of tiles of 512, a last tile with one particle,
and unequal masses.  Accelerations and potentials of sampled particles against
an FP64 direct sum over the same (split) positions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# tiles in place of units from 512 records per part on (3 585); pairs taken once
# from 8 192; 17, 18, 33 tiles
@pytest.mark.parametrize("masses", ["equal", "unequal"])
@pytest.mark.parametrize("n", [3, 64, 257, 1000, 3583, 3585, 8191, 8192, 8193, 8704, 9216, 9217, 16385, 65536, 81921])
def test_items_cover_every_pair(cs, n, masses):
    print(f"mixed gravity items n={n} {masses}", flush=True)
    e = cs.make_engine("mixed", 2, n, 7, ph_sort=True)
    if masses == "unequal":
        v = e.get("vel64")
        v[:n, 3] *= 10.0 ** np.random.default_rng(n).uniform(-1, 1, n)
        e.set("vel64", v)
    e.run_pass(cs.GRAVITY)
    got = e.get("grav")[:n].astype(np.float64)
    x = e.get("pos64")[:n, :3]
    m = e.get("vel64")[:n, 3]
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
