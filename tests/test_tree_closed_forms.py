"""One level of the device kd-tree build (cudasph_amd/csrc/tree.hip:
k_tree_count, k_tree_move) in numpy, index for index: the closed forms of a
subtree's size and place (subtree_size, subtree_start, subtree_at, lefts_before)
against counting node by node, and the places that k_tree_move computes from
them and from the counts of its tiles.  Every write must land inside the next
list, every place of it must be written once, and the tree must be the recursive
build's (kd_tree.cpp:39-95)."""
import numpy as np
import pytest

from test_tree_levels import assert_kd_order, recursive_build
from test_tree_levels import subtree_size as size_by_levels
from test_tree_levels import subtree_start as start_by_levels


def floor_log2(x):
    return int(x).bit_length() - 1


def subtree_size(t, n):
    if t > n:
        return 0
    k = floor_log2(n) - floor_log2(t)
    last = n - (t << k) + 1
    return (1 << k) - 1 + min(max(last, 0), 1 << k)


def subtree_start(t, L, n):
    k = floor_log2(n) - L
    if k < 0:
        return 0
    m, fill = t - (1 << L), n + 1 - (1 << (k + L))
    return m * ((1 << k) - 1) + min(m << k, fill)


def lefts_before(t, L, n):
    k = floor_log2(n) - L - 1
    if k < 0:
        return 0
    m, fill = t - (1 << L), n + 1 - (1 << (k + 1 + L))
    filled = min(m << (k + 1), fill)
    part = filled & ((2 << k) - 1)
    return m * ((1 << k) - 1) + ((filled >> (k + 1)) << k) + min(part, 1 << k)


def subtree_at(idx, L, n):
    k = floor_log2(n) - L
    fill = n + 1 - (1 << (k + L))
    full, part = fill >> k, fill & ((1 << k) - 1)
    large, small = (2 << k) - 1, (1 << k) - 1
    if idx < full * large:
        return (1 << L) + idx // large
    idx -= full * large
    return (1 << L) + full + (0 if idx < small + part else 1 + (idx - small - part) // small)


SIZES = list(range(1, 70)) + [(1 << k) + d for k in (7, 9, 11) for d in (-2, -1, 0, 1, 2)] + [96, 1000, 1537]


@pytest.mark.parametrize("n", SIZES)
def test_closed_forms_count_the_nodes(n):
    for L in range(floor_log2(n) + 1):
        nodes = np.arange(1 << L, min(2 << L, n + 1))
        sizes = size_by_levels(nodes, n)
        starts = start_by_levels(nodes, L, n)
        at = 0
        lefts = 0
        for t, s, b in zip(nodes.tolist(), sizes.tolist(), starts.tolist()):
            assert subtree_size(t, n) == s and subtree_start(t, L, n) == b == at
            assert lefts_before(t, L, n) == lefts
            for idx in {at, at + s - 1, at + s // 2}:
                assert subtree_at(idx, L, n) == t, (idx, L)
            at += s
            lefts += subtree_size(2 * t, n)
        # one past the level's last node: where a run of all of them ends
        assert subtree_start(2 << L, L, n) == n - (1 << L) + 1 if n >= (2 << L) - 1 else True


def level_build(xyz, tile):
    """The build with tiles of `tile` places (1024 on the device)."""
    n = len(xyz)
    node_id = np.full(n + 1, -1, np.int64)
    lists = [np.argsort(xyz[:, a], kind="stable") for a in range(3)]
    rank = np.empty((3, n), np.int64)   # the order that `before` compares: (coordinate, id)
    for a in range(3):
        rank[a, lists[a]] = np.arange(n)
    m, L = n, 0
    while m > 0:
        a = L % 3
        la = lists[a]
        t_of = [subtree_at(i, L, n) for i in range(m)]
        placed = min(1 << L, n - ((1 << L) - 1))
        for k in range(3):
            l = lists[k]
            nxt = np.full(max(m - placed, 0), -1, np.int64)

            def write(to, i):
                assert 0 <= to < m - placed and nxt[to] == -1
                nxt[to] = l[i]

            if k == a:
                for i in range(m):
                    t = t_of[i]
                    p, lt, before = i - subtree_start(t, L, n), subtree_size(2 * t, n), t - (1 << L)
                    if p < lt:
                        write(i - before, i)
                    elif p > lt:
                        write(i - before - 1, i)
                    else:
                        assert node_id[t] == -1
                        node_id[t] = l[i]
            else:
                side = []
                for i in range(m):
                    t = t_of[i]
                    node = la[subtree_start(t, L, n) + subtree_size(2 * t, n)]
                    side.append(0 if l[i] == node else 1 if rank[a, l[i]] < rank[a, node] else 2)
                side = np.array(side)
                for b in range(0, m, tile):
                    bl, br = (side[:b] == 1).sum(), (side[:b] == 2).sum()   # the tiles before
                    nl = nr = 0
                    for i in range(b, min(b + tile, m)):
                        t = t_of[i]
                        base = subtree_start(t, L, n) - (t - (1 << L))
                        lb0 = lefts_before(t, L, n)
                        if side[i] == 1:
                            write(base + bl + nl - lb0, i)
                            nl += 1
                        elif side[i] == 2:
                            write(base + subtree_size(2 * t, n) + br + nr - (base - lb0), i)
                            nr += 1
            assert (nxt >= 0).all()
            lists[k] = nxt
        m -= placed
        L += 1
    return node_id


@pytest.mark.parametrize("n,tile", [(1, 4), (2, 4), (3, 1), (7, 2), (8, 3), (31, 4), (32, 5), (33, 8), (100, 16),
                                    (255, 32), (256, 7), (257, 64), (700, 128)])
def test_level_build_is_the_recursive_build(n, tile):
    xyz = np.random.default_rng(n).random((n, 3)).astype(np.float32)
    got = level_build(xyz, tile)
    assert_kd_order(xyz, got)
    if all(len(np.unique(xyz[:, k])) == n for k in range(3)):
        assert np.array_equal(got, recursive_build(xyz))


@pytest.mark.parametrize("n,cells", [(50, 2), (300, 3)])
def test_level_build_with_ties_is_a_kd_tree(n, cells):
    xyz = np.random.default_rng(n).integers(0, cells, (n, 3)).astype(np.float32)
    assert_kd_order(xyz, level_build(xyz, 16))
