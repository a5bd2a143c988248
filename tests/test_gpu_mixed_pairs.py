"""Mixed Plummer gravity with each pair of particles evaluated once for both
(csrc/gravity.hip: k_gravity_mixed_pairs), beyond the sums themselves
(test_gpu_mixed_items.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def unequal(e, n):
    v = e.get("vel64")
    v[:n, 3] *= 10.0 ** np.random.default_rng(n).uniform(-1, 1, n)
    e.set("vel64", v)


def gravity_ms(cs, e):
    e.set_scalar("timing", 1)
    best = np.inf
    for _ in range(5):
        e.reset_timers()
        e.run_pass(cs.GRAVITY)
        best = min(best, e.timers()["gravity"][0])
    return best


@pytest.mark.parametrize("n", [30001, 65536])
def test_unequal_masses_cost_about_as_much_as_equal_ones(cs, n):
    """The body for unequal masses has 19 operations for a pair's two
    interactions where the one for equal masses has 16, and both have the same
    v_rsq_f32 and moves, so the pass takes at most about a fifth longer.  Twice
    is allowed: registers that do not suffice cost five times."""
    print(f"time of unequal masses n={n}", flush=True)
    e = cs.make_engine("mixed", 2, n, 7, ph_sort=True)
    equal = gravity_ms(cs, e)
    unequal(e, n)
    other = gravity_ms(cs, e)
    e.close()
    print(f"  equal {equal:.3f} ms, unequal {other:.3f} ms", flush=True)
    assert other <= 2 * equal


def test_few_tiles_take_no_longer_than_every_ordered_pair(cs):
    """8 192 particles are 16 tiles of 512, whose blocks leave half of the GPU idle:
    the pass takes what the kernel of every ordered pair does (which a measurement
    switch selects; its body is longer by one operation)."""
    n = 8192
    print(f"few tiles n={n}", flush=True)
    e = cs.make_engine("mixed", 2, n, 7, ph_sort=True)
    chosen = min(gravity_ms(cs, e), gravity_ms(cs, e))
    e.set_scalar("grav_expand", 0)
    ordered = min(gravity_ms(cs, e), gravity_ms(cs, e))
    e.close()
    print(f"  chosen {chosen:.3f} ms, every ordered pair {ordered:.3f} ms", flush=True)
    assert chosen <= 1.15 * ordered


@pytest.mark.parametrize("masses", ["equal", "unequal"])
@pytest.mark.parametrize("value", [np.nan, np.inf])
# records of the 12289: the origin record of a sub-tile of 64, another one, the
# last tile's only real record, which is its sub-tile's origin too
@pytest.mark.parametrize("at", [32, 4128, 100, 12288])
def test_a_lost_place_reaches_every_sum(cs, at, value, masses):
    """One particle at NaN or infinity: no particle's acceleration stays finite,
    as in a sum over all pairs."""
    n = 12289
    print(f"lost place at={at} {value} {masses}", flush=True)
    e = cs.make_engine("mixed", 2, n, 7, ph_sort=True)
    if masses == "unequal":
        unequal(e, n)
    x = e.get("pos64")
    x[at, 0] = value
    e.set("pos64", x)
    e.run_pass(cs.GRAVITY)
    a = e.get("grav")[:n, :3]
    e.close()
    assert not np.isfinite(a[:, 0]).any(), np.isfinite(a[:, 0]).sum()


def assert_sums(e, n, pick):
    """accelerations and potentials against FP64 over the same (split) places,
    with the bound of test_gpu_mixed_items.py"""
    got = e.get("grav")[:n].astype(np.float64)
    x = e.get("pos64")[:n, :3]
    m = e.get("vel64")[:n, 3].astype(np.float32).astype(np.float64)
    eps2 = float(e.params.grav_eps) ** 2
    for i in pick:
        r = x[i] - x
        inv = 1.0 / np.sqrt((r * r).sum(1) + eps2)
        a = -(m * inv ** 3)[:, None] * r
        assert np.linalg.norm(got[i, :3] - a.sum(0)) <= 2.0 ** -20 * np.linalg.norm(a, axis=1).sum(), i
        assert abs(got[i, 3] + (m * inv).sum()) <= 2.0 ** -20 * (m * inv).sum(), i


# the last size with every ordered pair, the first with pairs once (24 tiles),
# 25 tiles with one particle and full, 26 and 27
@pytest.mark.parametrize("masses", ["equal", "unequal"])
@pytest.mark.parametrize("n", [12032, 12287, 12288, 12289, 12800, 13312, 13313])
def test_tiles_around_the_first_size(cs, n, masses):
    print(f"first size n={n} {masses}", flush=True)
    e = cs.make_engine("mixed", 2, n, 7, ph_sort=True)
    if masses == "unequal":
        unequal(e, n)
    for parts in (0, 1, 3):
        e.set_scalar("grav_parts", parts)
        e.run_pass(cs.GRAVITY)
        assert_sums(e, n, np.unique(np.r_[0, 511, 512, n // 2, n - 1, np.linspace(0, n - 1, 60).astype(int)]))
    e.close()


# 733 and 734 tiles have 367 and 368 offsets, of which 2 GiB of reactions hold
# 357 (from 724 tiles on there are two chunks); the even count's opposite tiles
# meet in the second
@pytest.mark.parametrize("masses", ["equal", "unequal"])
@pytest.mark.parametrize("n", [733 * 512 - 100, 734 * 512 - 511])
def test_offsets_in_two_chunks(cs, n, masses):
    """Odd and even counts of tiles whose reactions do not fit at once: sampled
    sums against FP64, as in test_gpu_mixed_items.py."""
    print(f"two chunks n={n} {masses}", flush=True)
    e = cs.make_engine("mixed", 2, n, 7, ph_sort=True)
    tiles = -(-e.nd // 512)
    chunk = (2 << 30) // (16 * 512 * tiles)
    assert chunk < tiles // 2 + 1
    if masses == "unequal":
        unequal(e, n)
    e.run_pass(cs.GRAVITY)
    half = tiles // 2 * 512   # (a tile at most half way round: particles on both sides of it)
    assert_sums(e, n, np.unique(np.r_[0, 511, 512, half - 1, half, half + 512, n - 1,
                                      np.linspace(0, n - 1, 40).astype(int)]))
    e.close()
