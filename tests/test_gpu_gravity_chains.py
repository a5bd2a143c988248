"""The plain form's gravity sums (csrc/gravity.hip: k_gravity_chains,
k_gravity_lane): the shortened two-sum must be taken only where it is exact,
so the sums are the oracle's bits also where they cancel, start from zero or
meet terms larger than themselves, and at every edge of a batch or tile."""
import numpy as np
import pytest

from helpers import assert_bits, copy_state

pytestmark = pytest.mark.gpu


def gravity_pair(cs, orc, cfg, n, mode, change=None):
    p = cs.preset_params(cfg, n)
    p.grav_mode = mode
    pos, vel, hyd = cs.generate_ic(cfg, n, 31)
    if change is not None:
        change(pos, vel)
    e, o = cs.Engine("plain", p), orc.Oracle(32, p)
    for s in (e, o):
        s.load_ic(pos, vel, hyd)
    e.set_scalar("exact_rsqrt", 1)
    o.run_pass(cs.GRAVITY)
    return e, o


@pytest.mark.parametrize("sums", [0, 1])
@pytest.mark.parametrize("cfg,n", [(1, 1), (2, 15), (2, 16), (1, 17), (3, 63), (2, 65), (2, 511), (1, 513), (2, 4099)])
def test_spline_sums(cs, orc, cfg, n, sums):
    print(f"spline sums cfg={cfg} n={n} sums={sums}", flush=True)
    e, o = gravity_pair(cs, orc, cfg, n, 0)
    e.set_scalar("grav_sums", sums)
    e.run_pass(cs.GRAVITY)
    assert_sums(e, o, n)
    e.close()


def assert_sums(e, o, n):
    """the oracle's bits; a NaN (a padding record on a particle at the origin)
    is a NaN whatever its sign and payload"""
    a, b = e.get("grav")[:n], o.get("grav")[:n]
    assert np.array_equal(np.isnan(a), np.isnan(b))
    assert_bits(np.nan_to_num(a, nan=0.0), np.nan_to_num(b, nan=0.0), "grav")


def lattice(pos, vel):
    """a cubic lattice about the origin: sums that cancel exactly, equal terms"""
    n = len(pos)
    k = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(k) - (k - 1) / 2] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    pos[:, :3] = g * 0.125


def masses(pos, vel):
    """masses over 30 decades, some of them zero: terms far above the sum"""
    rng = np.random.default_rng(7)
    vel[:, 3] = 10.0 ** rng.uniform(-28, 2, len(vel))
    vel[::5, 3] = 0.0


def far_pairs(pos, vel):
    """two mirrored clumps far apart and a light particle between"""
    n = len(pos)
    pos[: n // 2, 0] += 1e4
    pos[n // 2:, 0] -= 1e4
    pos[0, :3] = 0.0


@pytest.mark.parametrize("sums", [0, 1])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("change", [lattice, masses, far_pairs])
@pytest.mark.parametrize("n", [1000, 4097])
def test_sums_that_cancel_or_jump(cs, orc, n, change, mode, sums):
    print(f"sums {change.__name__} n={n} mode={mode} sums={sums}", flush=True)
    e, o = gravity_pair(cs, orc, 2, n, mode, change)
    e.set_scalar("grav_sums", sums)
    e.run_pass(cs.GRAVITY)
    assert_sums(e, o, n)
    e.close()


@pytest.mark.parametrize("cfg,n", [(3, 524287), (2, 524289)])
def test_both_sides_of_the_large_size_rule(cs, cfg, n):
    """One lane per particle with and without the shortened two-sum (the rule
    at 2^19 particles, by padded count) against a wavefront per sum."""
    print(f"large sums cfg={cfg} n={n}", flush=True)
    e = cs.make_engine("plain", cfg, n, 3, ph_sort=True)
    out = []
    for sums in (-1, 1):
        e.set_scalar("grav_sums", sums)
        e.run_pass(cs.GRAVITY)
        out.append(e.get("grav")[:n].copy())
    assert_bits(out[0], out[1], "grav")
    e.close()
