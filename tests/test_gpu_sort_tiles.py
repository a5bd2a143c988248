"""The look-back radix sort (csrc/sort.hip) around its tile of 4096 records
and with few distinct digits, against numpy's stable sort bit for bit."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 4095, 4096, 4097, 8192, 12289, 300001])
@pytest.mark.parametrize("bits", [3, 8, 16, 24, 32])
@pytest.mark.parametrize("kind", ["random", "equal", "descending"])
def test_sort_around_tiles(cs, n, bits, kind):
    print(f"sort n={n} bits={bits} {kind}", flush=True)
    import torch
    rng = np.random.default_rng(n + bits)
    top = 1 << bits
    keys = {"random": rng.integers(0, top, n, dtype=np.uint64), "equal": np.full(n, top - 1, np.uint64),
            "descending": np.sort(rng.integers(0, top, n, dtype=np.uint64))[::-1]}[kind].astype(np.uint32)
    kv = np.stack([keys, np.arange(n, dtype=np.uint32)], 1)
    data = torch.from_numpy(kv.astype(np.int64).astype(np.uint32).view(np.int32).copy()).cuda()
    alt = torch.zeros_like(data)
    L = cs.lib()
    L.sph_radix_sort_noalloc.argtypes = [C.c_void_p, C.c_void_p, C.c_uint, C.c_uint, C.c_void_p]
    L.sph_radix_sort_noalloc.restype = C.c_int
    for _ in range(2):   # sorted input the second time
        assert L.sph_radix_sort_noalloc(data.data_ptr(), alt.data_ptr(), n, bits,
                                        torch.cuda.current_stream().cuda_stream) == 0
        got = data.cpu().numpy().view(np.uint32)
        assert np.array_equal(got, kv[np.argsort(keys, kind="stable")])


def test_more_records_of_one_digit_than_2_to_the_30(cs):
    """RadixSort takes any count up to 2^31 - 1: 2^30 + 2^20 + 3 records, all but
    the last 1000 with the same digit."""
    import torch
    n, few = (1 << 30) + (1 << 20) + 3, 1000
    print(f"sort n={n}", flush=True)
    data = torch.empty((n, 2), dtype=torch.int32, device="cuda")
    data[:, 0] = 5
    data[n - few:, 0] = 3
    torch.arange(n, dtype=torch.int32, out=data[:, 1])
    alt = torch.zeros_like(data)
    torch.cuda.synchronize()
    L = cs.lib()
    L.RadixSort.argtypes = [C.c_void_p, C.c_void_p, C.c_uint, C.c_uint]
    L.RadixSort.restype = None
    L.RadixSort(data.data_ptr(), alt.data_ptr(), n, 8)
    del alt
    torch.cuda.synchronize()
    first = data[:few].cpu().numpy()
    assert (first[:, 0] == 3).all() and np.array_equal(first[:, 1], np.arange(n - few, n))
    assert bool((data[few:, 0] == 5).all())
    assert torch.equal(data[few:, 1], torch.arange(n - few, dtype=torch.int32, device="cuda"))


@pytest.mark.parametrize("polls", [0, 3])
@pytest.mark.parametrize("n,bits,distinct", [(4097, 8, 256), (100001, 32, 1 << 32), (130000, 16, 5)])
def test_a_wait_cut_short_changes_nothing(cs, n, bits, distinct, polls):
    """A tile that stops waiting for an earlier one counts that one's records."""
    print(f"short waits n={n} bits={bits} polls={polls}", flush=True)
    import torch
    rng = np.random.default_rng(n)
    kv = np.stack([rng.integers(0, distinct, n, dtype=np.uint64).astype(np.uint32), np.arange(n, dtype=np.uint32)], 1)
    data = torch.from_numpy(kv.view(np.int32).copy()).cuda()
    alt = torch.zeros_like(data)
    torch.cuda.synchronize()
    L = cs.lib()
    L.sph_radix_sort_polls.argtypes = [C.c_void_p, C.c_void_p, C.c_uint, C.c_uint, C.c_int]
    assert L.sph_radix_sort_polls(data.data_ptr(), alt.data_ptr(), n, bits, polls) == 0
    assert np.array_equal(data.cpu().numpy().view(np.uint32), kv[np.argsort(kv[:, 0], kind="stable")])
