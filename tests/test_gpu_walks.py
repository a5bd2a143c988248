"""The shared tree walks (csrc/walks.hip) where they can go wrong, against the
CPU oracle bit for bit: trees smaller than a group of lanes, lists that outgrow
one pass of a group's LDS, ranges the solver has to move far, and the two
sides of the rule that hands large particle numbers to a lane each."""
import numpy as np
import pytest

from helpers import assert_bits, copy_state, lists_of

pytestmark = pytest.mark.gpu


def pair(cs, orc, form, cfg, n, boxes):
    p = cs.preset_params(cfg, n)
    pos, vel, hyd = cs.generate_ic(cfg, n, 5)
    e = cs.Engine(form, p)
    e.set_scalar("walk_boxes", boxes)
    o = orc.Oracle(64 if form == "fp64" else 32, p)
    for s in (e, o):
        s.load_ic(pos, vel, hyd)
    o.init()
    copy_state(e, o)
    return e, o


def walk_lengths(sim):
    h = sim.get("hash")
    out = np.zeros(len(h), np.int64)
    out[h[:, 1]] = h[:, 0]
    return out


@pytest.mark.parametrize("form", ["plain", "fp64"])
@pytest.mark.parametrize("boxes", [0, 1])
@pytest.mark.parametrize("cfg,n", [(1, 1), (1, 2), (2, 15), (1, 16), (2, 17), (1, 256), (2, 1000), (2, 6000),
                                    (1, 6000)])
def test_lists_of_wide_ranges(cs, orc, form, boxes, cfg, n):
    """Every 40th particle's range widened 3.5 times (some hundred to all
    particles in its list): the same lists in the same order."""
    print(f"wide lists {form} boxes={boxes} cfg={cfg} n={n}", flush=True)
    e, o = pair(cs, orc, form, cfg, n, boxes)
    q = o.get("pos")
    q[:n:40, 3] *= 3.5
    for s in (e, o):
        s.set("pos", q)
        s.run_pass(cs.OFFSETS)
    d2 = ((q[:n, None, :3] - q[None, :n, :3]) ** 2).sum(2)
    slots = ((d2 < q[:n, None, 3] ** 2).sum(1) + 3) // 4 * 4
    if slots.sum() > 100 * e.nd:   # more than the lists' allocation: refused
        with pytest.raises(RuntimeError, match="overflow"):
            e.run_pass(cs.FIND)
        return
    o.run_pass(cs.FIND)
    e.run_pass(cs.FIND)
    assert np.array_equal(e.get("ngb_count"), o.get("ngb_count"))
    le, lo = lists_of(e, n), lists_of(o, n)
    bad = [i for i in range(n) if not np.array_equal(le[i], lo[i])]
    assert not bad, f"{len(bad)} lists differ, first particle {bad[0]}"
    if not boxes:
        assert np.array_equal(walk_lengths(e)[:n], walk_lengths(o)[:n])
    e.close()


@pytest.mark.parametrize("form", ["plain", "fp64"])
@pytest.mark.parametrize("cfg,n", [(1, 2), (2, 33), (1, 1000), (2, 5000)])
@pytest.mark.parametrize("scale", [0.25, 0.9, 1.02, 3.0])
def test_solve_from_a_far_range(cs, orc, form, cfg, n, scale):
    """The h-solve started `scale` times off: the same ranges and counts, with
    the kept distances, without them, and with the subtree boxes."""
    print(f"far solve {form} cfg={cfg} n={n} scale={scale}", flush=True)
    e, o = pair(cs, orc, form, cfg, n, 0)
    q = o.get("pos")
    q[:n, 3] *= scale
    o.set("pos", q)
    o.run_pass(cs.SOLVE)
    for cache, boxes in ((1, 0), (0, 0), (1, 1)):
        e.set_scalar("solve_cache", cache)
        e.set_scalar("walk_boxes", boxes)
        e.set("pos", q)
        e.run_pass(cs.SOLVE)
        assert_bits(e.get("pos")[:n], o.get("pos")[:n], f"range, cache {cache} boxes {boxes}")
        assert np.array_equal(e.get("n_ngb")[:n], o.get("n_ngb")[:n])
    e.close()


@pytest.mark.parametrize("n", [524287, 524288])
def test_both_walks_give_the_tree_s_lists(cs, n):
    """One lane or 16 per particle: the mixed form's lists are the particles
    within the range, by brute force over a sample."""
    print(f"sampled lists n={n}", flush=True)
    e = cs.make_engine("mixed", 5, n, 3, ph_sort=True)
    for pid in (cs.TREE, cs.SOLVE, cs.OFFSETS, cs.FIND):
        e.run_pass(pid)
    q = e.get("pos")[:n]
    off, cnt = e.get("ngb_offset"), e.get("ngb_count")
    lst = e.get("ngb_list", int(off[-1]))
    for i in range(0, n, n // 37):
        d = q[i, :3] - q[:, :3]
        d2 = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]
        want = np.nonzero(d2 < q[i, 3] * q[i, 3])[0]
        assert np.array_equal(np.sort(lst[off[i]:off[i] + cnt[i]]), want), i
    e.close()


@pytest.mark.parametrize("form", ["plain", "mixed", "fp64"])
def test_whole_evaluation_refuses_lists_beyond_the_allocation(cs, form):
    """A neighbour target of 100 needs more than the 100 slots per particle:
    init() refuses, as the offsets pass by itself, and no list was written."""
    n = 2000
    print(f"refusal {form}", flush=True)
    p = cs.preset_params(2, n)
    p.desired_ngb = 100.0
    e = cs.Engine(form, p)
    e.load_ic(*cs.generate_ic(2, n, 5))
    e.set("ngb_list", np.full_like(e.get("ngb_list"), 7))   # (allocated, not cleared)
    with pytest.raises(RuntimeError, match="overflow"):
        e.init()
    assert (e.get("ngb_list") == 7).all() and not e.get("ngb_count").any()
    with pytest.raises(RuntimeError, match="overflow"):
        e.run_pass(cs.OFFSETS)
    e.close()


@pytest.mark.parametrize("scale", [1.0, 1e21, 1e-21, 1e40])
@pytest.mark.parametrize("n,off,seed", [(256, 1.0, 1), (2048, 0.5, 1), (2048, 1.0, 3), (8192, 1.0, 1)])
def test_kept_distances_at_any_scale(cs, n, off, seed, scale):
    """FP64 lengths whose squares are no floats.  The reference's out-of-range
    record n+1 (at the origin) is placed beside its parent node, where some walks
    reach it at 17/16 of their range and not at the range itself."""
    print(f"kept distances n={n} off={off} seed={seed} scale={scale}", flush=True)
    p = cs.preset_params(1, n)
    assert p.fix_phantom == 0 and p.n_dev == n
    pos, vel, hyd = cs.generate_ic(1, n, seed)
    e = cs.Engine("fp64", p)
    e.load_ic(pos, vel, hyd)
    for pid in (cs.TREE, cs.SOLVE):
        e.run_pass(pid)
    r = e.get("pos")[:n, 3].copy()
    d = np.random.default_rng(seed).normal(size=3)
    pos[:n, :3] -= e.get("tree")[n // 2, :3] + off * r.mean() * d / np.linalg.norm(d)
    pos[:n, 3] = 1.1 * r
    pos[:n] *= scale
    out = []
    for cache in (0, 1):
        e.set_scalar("solve_cache", cache)
        e.load_ic(pos, vel, hyd)
        for pid in (cs.TREE, cs.SOLVE):
            e.run_pass(pid)
        out.append((e.get("pos")[:n, 3].copy(), e.get("n_ngb")[:n].copy()))
    e.close()
    assert_bits(out[1][0], out[0][0], "range")
    assert np.array_equal(out[1][1], out[0][1])
