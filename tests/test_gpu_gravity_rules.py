"""The plain form's gravity on both sides of each size at which its kernel
changes (csrc/gravity.hip, launch_gravity, by the padded count e.nd), and the
shortened two-sum of many particles on inputs that cancel or jump: the bits of
a wavefront per sum (checked against the oracle in test_gpu_gravity_chains.py)
and of a lane per particle."""
import numpy as np
import pytest

from helpers import assert_bits
from test_gpu_gravity_chains import far_pairs, lattice, masses

pytestmark = pytest.mark.gpu


def sums_of(cs, e, n, choices):
    out = []
    for sums in choices:
        e.set_scalar("grav_sums", sums)
        e.run_pass(cs.GRAVITY)
        out.append(e.get("grav")[:n].copy())
    return out


# Plummer: a wavefront per sum up to 94 208 records, one lane above, with the
# shortened two-sum from 2^19 on; spline: up to 81 920, then the last of these
@pytest.mark.parametrize("mode,n,rule", [(1, 94208, "chains"), (1, 94209, "lane"), (1, 524032, "lane"),
                                         (1, 524288, "fast lane"), (0, 81920, "chains"), (0, 81921, "fast lane")])
def test_both_sides_of_every_rule(cs, mode, n, rule):
    print(f"gravity rule mode={mode} n={n} {rule}", flush=True)
    p = cs.preset_params(3, n)
    p.grav_mode = mode
    e = cs.make_engine("plain", 3, n, 3, params=p, ph_sort=True)
    most = 94208 if mode else 81920
    assert rule == ("chains" if e.nd <= most else "lane" if mode and e.nd < 1 << 19 else "fast lane")
    auto, lane, chains = sums_of(cs, e, n, (-1, 0, 1))
    e.close()
    assert_bits(auto, lane, "automatic, one lane")
    assert_bits(auto, chains, "automatic, a wavefront per sum")


def same(a, b):
    """the same bits; a NaN (a padding record on a particle at the origin) is
    a NaN whatever its sign and payload"""
    assert np.array_equal(np.isnan(a), np.isnan(b))
    assert_bits(np.nan_to_num(a, nan=0.0), np.nan_to_num(b, nan=0.0), "grav")


@pytest.mark.parametrize("change", [lattice, masses, far_pairs])
def test_many_particles_that_cancel_or_jump(cs, change):
    """The bound on a group's terms that licenses the shortened two-sum, under
    Plummer softening, where only 2^19 records and more take that kernel."""
    n = 1 << 19
    print(f"fast lane {change.__name__}", flush=True)
    p = cs.preset_params(2, n)
    pos, vel, hyd = cs.generate_ic(2, n, 31)
    change(pos, vel)
    e = cs.Engine("plain", p)
    e.load_ic(pos, vel, hyd)
    auto, chains = sums_of(cs, e, n, (-1, 1))
    e.close()
    same(auto, chains)
