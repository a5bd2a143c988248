"""The plain form's density, hydro and reaction sums by 16 lanes per particle, in
list order (OrderedSums): the oracle's bits with lists of every length around
16 and its multiples, from particles alone to hundreds of neighbours."""
import numpy as np
import pytest

from helpers import assert_bits, copy_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 33, 700])
@pytest.mark.parametrize("scale", [0.05, 0.6, 1.0, 1.3])
def test_sums_in_list_order(cs, orc, n, scale):
    print(f"ordered sums n={n} scale={scale}", flush=True)
    p = cs.preset_params(2, n)
    e, o = cs.Engine("plain", p), orc.Oracle(32, p)
    pos, vel, hyd = cs.generate_ic(2, n, 11)
    for s in (e, o):
        s.load_ic(pos, vel, hyd)
    o.init()
    copy_state(e, o)
    q = o.get("pos")
    q[:n, 3] *= scale * np.linspace(0.8, 1.2, n).astype(q.dtype)   # lengths that differ within a wavefront
    d2 = ((q[:n, None, :3] - q[None, :n, :3]) ** 2).sum(2)
    if (((d2 < q[:n, None, 3] ** 2).sum(1) + 3) // 4 * 4).sum() > 100 * e.nd:   # more than the lists' allocation
        e.set("pos", q)
        with pytest.raises(RuntimeError, match="overflow"):
            e.run_pass(cs.OFFSETS)
            e.run_pass(cs.FIND)
        return
    for s in (e, o):
        s.set("pos", q)
        for k in (cs.OFFSETS, cs.FIND, cs.DENSITY, cs.EOS, cs.HYDRO, cs.REACTION):
            s.run_pass(k)
    for name in ("hydro", "dots", "bdots", "hydro2"):
        a, b = e.get(name)[:n], o.get(name)[:n]
        nan = np.isnan(b)
        assert np.array_equal(np.isnan(a), nan), name
        assert_bits(np.where(nan, 0, a), np.where(nan, 0, b), name)
    e.close()
