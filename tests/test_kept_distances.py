"""The h-solve's kept distances (cudasph_amd/csrc/walks.hip: walk_pass with
REACH, Solver::eval) in numpy, operation for operation.

A walk at 17/16 of a range keeps the distances it accepts, and, beside each, the
largest distance to a split plane that its path's pushes crossed.  A later
evaluation at a smaller range r takes the kept distances below r, unless one lies
so close to r that the rounding of the push tests may decide (`sure`), or some
record's path bound is not below its distance; then it walks at r.  Whatever it
takes must be the walk's distances in the walk's order."""
import numpy as np
import pytest

from test_solve_cache_bounds import build


class Real:
    """one type's arithmetic"""

    def __init__(self, t):
        self.t = t
        self.eps = t(2.0 ** -24 if t is np.float32 else 2.0 ** -53)
        self.tiny = t(1e-30 if t is np.float32 else 1e-60)


REALS = [Real(np.float32), Real(np.float64)]


def visit(R, q, tree, phantom, node):
    """(children to push at range r -> their plane distances, distance^2) of a
    node; the record past the tree is the reference's out-of-range fetch, zeros"""
    t = R.t
    n = len(tree) - 1
    p, ax = tree[node] if node <= n else ((t(0), t(0), t(0)), 0)
    dx, dy, dz = (t(q[k] - p[k]) for k in range(3))
    ds2 = t(t(t(dx * dx) + t(dy * dy)) + t(dz * dz))

    def children(r):
        c, out = 2 * node, []
        if c <= n:
            qc, nc = q[ax], p[ax]
            if t(qc - r) < nc:
                out.append((c, np.float32(max(t(qc - nc), t(0)))))
            if t(qc + r) > nc and (phantom or c < n):
                out.append((c + 1, np.float32(max(t(nc - qc), t(0)))))
        return out
    return children, ds2


def walk(R, q, r, tree, phantom):
    """[(distance^2, path bound)] in the walk's order"""
    t = R.t
    r2 = t(r * r)
    out, stack = [], [(1, np.float32(0))]
    while stack:
        node, path = stack.pop()
        children, ds2 = visit(R, q, tree, phantom, node)
        if ds2 < r2:
            out.append((ds2, path))
        for c, m in children(r):   # (the right child, pushed last, is visited first)
            stack.append((c, max(path, m)))
    return out


def keep(R, q, r0, tree, phantom):
    t = R.t
    with np.errstate(over="ignore", under="ignore"):
        rec = walk(R, q, t(r0 * t(1.0625)), tree, phantom)
        for ds2, path in rec:
            if path > 0 and not (t(t(path) * t(path)) <= t(ds2 * t(1.00001)) and ds2 >= R.tiny):
                return None
    return [ds2 for ds2, _ in rec]


def evaluate(R, q, r, kept):
    """the kept distances that evaluation r takes, or None: it walks"""
    t = R.t
    pad = t(t(t(32) * R.eps) * max(abs(q[0]), abs(q[1]), abs(q[2])))
    sure = t(t(r - t(pad + t(t(t(32) * R.eps) * r))) * t(1.0 - 1.0 / 32768.0))
    sure2 = t(sure * sure) if sure > 0 else t(0)
    take = [d for d in kept if d < t(r * r)]
    return take if all(d < sure2 for d in take) else None


def check(R, q, r0, tree, phantom, ranges):
    taken = 0
    kept = keep(R, q, r0, tree, phantom)
    if kept is None:
        return 0
    for r in ranges:
        got = evaluate(R, q, r, kept)
        if got is not None:
            assert got == [d for d, _ in walk(R, q, r, tree, phantom)], (q, r)
            taken += 1
    return taken


# (squares of FP32 lengths of the other scales are no floats: no range has neighbours)
@pytest.mark.parametrize("R,scale", [(REALS[0], 1.0), (REALS[1], 1.0), (REALS[1], 1e21), (REALS[1], 1e-21)],
                         ids=["float", "double", "double-1e21", "double-1e-21"])
@pytest.mark.parametrize("grid", [0, 64])
@pytest.mark.parametrize("n,phantom", [(1000, False), (1000, True), (999, True)])
def test_kept_distances_are_the_walk_s(R, scale, grid, n, phantom):
    rng = np.random.default_rng(7)
    raw = rng.random((n, 3))
    if grid:
        raw = np.round(raw * grid) / grid   # many equal coordinates and distances
    pts = [tuple(R.t(v * scale) for v in row) for row in raw.astype(R.t)]
    taken = asked = 0
    for shift in range(2):
        if shift:   # the zero record beside its parent node n / 2
            tree = build(pts)
            o = tree[n // 2][0]
            pts = [tuple(R.t(p[k] - o[k] + R.t(0.05 * scale)) for k in range(3)) for p in pts]
        tree = build(pts)
        near = sorted(pts, key=lambda p: max(abs(v) for v in p))
        for trial in range(60):
            q = near[trial] if trial % 2 else pts[rng.integers(n)]
            r0 = R.t(rng.choice([0.0625, 0.09375, 0.1, 0.125]) * scale)
            ranges = [r0, R.t(r0 * R.t(0.9)), R.t(r0 * R.t(1.0625)), R.t(0.0625 * scale), R.t(r0 * R.t(1.01))]
            ranges = [r for r in ranges if r <= R.t(r0 * R.t(1.0625))]
            taken += check(R, q, r0, tree, phantom, ranges)
            asked += len(ranges)
    assert taken > asked / 4   # (grids put distances at the range itself)


@pytest.mark.parametrize("R", REALS, ids=["float", "double"])
def test_a_particle_that_rounding_prunes(R):
    """The left subtree's plane lies at nc = fl(qx - r), its particle at x = nc
    with the query's y and z.  fl(qx - r) < nc is false, so the walk at r prunes it,
    yet fl(qx - nc) < r puts it inside the range."""
    t = R.t
    qx, r = next((a, b) for a in map(t, np.linspace(0.3, 0.9, 400)) for b in map(t, (0.1, 0.13, 0.17))
                 if t(a - t(a - b)) < b)
    nc = t(qx - r)
    q = (qx, t(0.5), t(0.5))
    inside = (nc, t(0.5), t(0.5))
    tree = [None, ((nc, t(0.9), t(0.5)), 0), (inside, 1), ((t(0.95), t(0.5), t(0.5)), 1)]
    d = visit(R, q, tree, False, 2)[1]
    walked = [x for x, _ in walk(R, q, r, tree, False)]
    kept = keep(R, q, r, tree, False)
    assert d not in walked and d in kept and d < t(r * r)   # a bare filter is wrong here
    assert evaluate(R, q, r, kept) is None                  # the rule sends it to a walk
