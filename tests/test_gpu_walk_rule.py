"""Which walk takes a particle (csrc/walks.hip, walk_alone): 16 lanes or one, by
the number of records (n_dev, a multiple of 256) and the neighbour target."""
import numpy as np
import pytest

from helpers import assert_bits, lists_of

pytestmark = pytest.mark.gpu


# targets of 45.2 (lists of 64) and 62 (lists of 89); with the second the lane
# takes over at 65 536 records
@pytest.mark.parametrize("n,target", [(65280, 62.0), (65536, 62.0), (65535, 45.2)])
def test_ranges_and_lists_on_both_sides(cs, orc, n, target):
    print(f"walk rule n={n} target={target}", flush=True)
    p = cs.preset_params(5, n)
    p.desired_ngb = target
    pos, vel, hyd = cs.generate_ic(5, n, 5)
    e, o = cs.Engine("plain", p), orc.Oracle(32, p)
    for s in (e, o):
        s.load_ic(pos, vel, hyd)
        for pid in (cs.TREE, cs.SOLVE, cs.OFFSETS, cs.FIND):
            s.run_pass(pid)
    assert_bits(e.get("pos")[:n], o.get("pos")[:n], "range")
    assert np.array_equal(e.get("ngb_count"), o.get("ngb_count"))
    le, lo = lists_of(e, n), lists_of(o, n)
    bad = [i for i in range(n) if not np.array_equal(le[i], lo[i])]
    assert not bad, f"{len(bad)} lists differ, first particle {bad[0]}"
    e.close()


# lists of 50 stay with 16 lanes up to 2^19 records
@pytest.mark.parametrize("n,alone", [(524032, False), (524288, True)])
def test_lists_on_both_sides_of_2_to_the_19(cs, n, alone):
    """The mixed form's lists are the particles within the range, by brute force
    over a sample."""
    print(f"sampled lists n={n}", flush=True)
    p = cs.preset_params(5, n)
    p.desired_ngb = 35.3
    p.eos_newton = 1
    e = cs.make_engine("mixed", 5, n, 3, params=p, ph_sort=True)
    assert (e.nd >= 1 << 19) == alone
    for pid in (cs.TREE, cs.SOLVE, cs.OFFSETS, cs.FIND):
        e.run_pass(pid)
    q = e.get("pos")[:n]
    off, cnt = e.get("ngb_offset"), e.get("ngb_count")
    lst = e.get("ngb_list", int(off[-1]))
    e.close()
    for i in range(0, n, n // 37):
        d = q[i, :3] - q[:, :3]
        d2 = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]
        want = np.nonzero(d2 < q[i, 3] * q[i, 3])[0]
        assert np.array_equal(np.sort(lst[off[i]:off[i] + cnt[i]]), want), i


@pytest.mark.parametrize("form", ["mixed", "fp64"])
def test_long_lists_cost_what_they_are_longer(cs, form):
    """h-solve and lists of 262 144 particles: lists 1.37 times as long take at
    most 2.5 times as long (walked in several passes of a group: 4)."""
    n, ms = 262144, {}
    print(f"time of long lists {form}", flush=True)
    for target in (45.2, 62.0):
        p = cs.preset_params(5, n)
        p.desired_ngb = target
        p.eos_newton = 1
        e = cs.make_engine(form, 5, n, 5, params=p, ph_sort=True)
        for pid in (cs.TREE, cs.SOLVE):
            e.run_pass(pid)
        e.set_scalar("timing", 1)
        best = np.inf
        for _ in range(4):
            e.reset_timers()
            for pid in (cs.SOLVE, cs.OFFSETS, cs.FIND):
                e.run_pass(pid)
            t = e.timers()
            best = min(best, t["solve_range"][0] + t["find_ngb"][0])
        ms[target] = best
        e.close()
    print("  ", ms, flush=True)
    assert ms[62.0] <= 2.5 * ms[45.2]
