"""FP64 gravity and its reverse pass where each pair of particles is evaluated
once for both (csrc/pairs64.h): odd and even tile counts, a last tile with one
particle, every part count; equal masses,
masses over a factor of 100, and one that differs."""
import numpy as np
import pytest

import adjoint_reference as ar

pytestmark = pytest.mark.gpu


# 8 192 is the first size, 12 287 the last with more parts; 16, 17, 18, 19, 24, 25
# and 129 tiles
@pytest.mark.parametrize("n", [8191, 8192, 8193, 8449, 8704, 9217, 12287, 12289, 65537])
@pytest.mark.parametrize("masses", ["equal", "unequal", "one differs"])
def test_pairs_give_the_direct_sum(cs, n, masses):
    print(f"fp64 pairs n={n} {masses}", flush=True)
    p = cs.preset_params(2, n)
    pos, vel, hyd = cs.generate_ic(2, n, 3)
    rng = np.random.default_rng(n)
    if masses == "unequal":
        vel[:n, 3] *= 10.0 ** rng.uniform(-1, 1, n).astype(vel.dtype)
    elif masses == "one differs":
        vel[n // 3, 3] *= 3
    e = cs.Engine("fp64", p)
    e.load_ic(pos, vel, hyd)
    x, m = pos[:n, :3].astype(np.float64), vel[:n, 3].astype(np.float64)
    eps2 = float(p.grav_eps) ** 2
    pick = np.unique(np.r_[0, 255, 256, n - 2, n - 1, np.linspace(0, n - 1, 64).astype(int)])
    terms = []
    for i in pick:
        r = x[i] - x
        inv = 1.0 / np.sqrt((r * r).sum(1) + eps2)
        terms.append((-(m * inv ** 3)[:, None] * r, -(m * inv)))
    for parts in (0, 1, 2, 3, 5, 8):
        e.set_scalar("grav_parts", parts)
        e.run_pass(cs.GRAVITY)
        got = e.get("grav")
        for i, (a, ph) in zip(pick, terms):
            # a term is within 16 roundings of 2^-53, a sum's chains are
            # shorter than 2^13 terms: 2^-40 of the terms' magnitudes
            assert np.linalg.norm(got[i, :3] - a.sum(0)) <= 2.0 ** -40 * np.linalg.norm(a, axis=1).sum(), (parts, i)
            assert abs(got[i, 3] - ph.sum()) <= 2.0 ** -40 * -ph.sum(), (parts, i)
    e.close()


def test_reverse_pass_against_the_cpu_reference(cs):
    """One step at 17 tiles, as test_adjoint_matches_fp64_cpu_reference_gradient
    (same tolerance)."""
    n, K = 8193, 1
    print(f"adjoint pairs n={n}", flush=True)
    p = cs.preset_params(4, n)
    pos, vel, hyd = cs.generate_ic(4, n, 3)
    e = cs.Engine("fp64", p)
    e.load_ic(pos, vel, hyd)
    loss = e.adjoint_forward(K, 1)
    g = np.concatenate([a.ravel() for a in e.adjoint_backward()])
    ranges, dts = e.adjoint_records()
    lref, *gr = ar.gradient(pos[:n], vel[:n], hyd[:n], ranges, dts, p)
    gr = np.concatenate([a.ravel() for a in gr])
    assert loss == pytest.approx(lref, rel=1e-11)
    err = np.linalg.norm(g - gr) / np.linalg.norm(gr)
    assert err <= 1e-8, err
    e.close()
