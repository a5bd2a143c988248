"""Device memory of the pair sums: only engines whose gravity takes pairs once
hold their reactions."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

N = 1 << 18
# FP32: 257 slots of 2^18 records of 16 bytes; FP64: 256 of 32
REACTIONS = {"mixed": 257 * N * 16, "fp64": 256 * N * 32}
SLACK = 64 << 20   # the driver's granularity, other buffers of the mode


def used(cs):
    L, free, total = cs.lib(), C.c_size_t(), C.c_size_t()   # (finds the HIP runtime it is linked with)
    assert L.hipDeviceSynchronize() == 0 and L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return total.value - free.value


@pytest.mark.parametrize("form", ["mixed", "fp64"])
def test_spline_softening_holds_no_reactions(cs, form):
    print(f"workspace spline {form}", flush=True)
    size = {}
    for mode in (1, 0, 1, 0):   # (the first ones bring the library's own memory)
        p = cs.preset_params(2, N)
        p.grav_mode = mode
        before = used(cs)
        e = cs.Engine(form, p)
        size[mode] = used(cs) - before
        e.close()
    assert size[1] - size[0] >= REACTIONS[form] - SLACK, size


def test_the_far_field_gives_the_reactions_back(cs):
    print("workspace far field", flush=True)
    e = cs.make_engine("mixed", 2, N, 3, ph_sort=True)
    e.run_pass(cs.GRAVITY)
    pairs, a = used(cs), e.get("grav")
    e.set_scalar("grav_far", 1)
    e.run_pass(cs.GRAVITY)
    assert pairs - used(cs) >= REACTIONS["mixed"] - SLACK
    e.set_scalar("grav_far", 0)
    e.run_pass(cs.GRAVITY)
    assert (e.get("grav") == a).all()
    e.close()
