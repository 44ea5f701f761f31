"""The kernels of path preparation at the sizes where their tiles and packings end."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from eppgcn_amd import capi
    capi.load()
    assert torch.cuda.is_available()
    return capi


@pytest.mark.parametrize("n,length", [(1, 1), (31, 5), (32, 1023), (33, 1024), (8192, 1025), (8193, 40000),
                                      (70001, 4097), (1 << 18, 3), (5, 0)])
@pytest.mark.parametrize("shift", [0, 1])
def test_distinct_rows_with_and_without_scratch(api, n, length, shift):
    """`shift`: the list starts 4 bytes past a 16-byte boundary.  Half of the entries are one hub row."""
    rng = np.random.default_rng(n * 7 + length)
    rows = rng.integers(0, n, length + shift, dtype=np.int32)
    rows[rng.random(length + shift) < 0.5] = n // 2
    lst = torch.from_numpy(rows).cuda()[shift:]
    want = np.zeros((n + 31) // 32 * 32, np.uint8)
    want[rows[shift:]] = 1
    bits = np.packbits(want, bitorder="little").view(np.int32)
    got, count = api.mark_gathered_rows(lst, length, n)
    assert count == int(want.sum()) and np.array_equal(got.cpu().numpy(), bits)
    # the entry point without scratch memory
    lib, out = api.load(), torch.full(((n + 31) // 32 + 1,), -1, dtype=torch.int32, device="cuda")
    v = ctypes.c_int64(-1)
    rc = lib.eppgcn_mark_gathered_rows(lst.data_ptr() if length else None, length, n, out.data_ptr(), out[-1:].data_ptr(),
                                       ctypes.byref(v), torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and v.value == count and np.array_equal(out[:-1].cpu().numpy(), bits)


@pytest.mark.parametrize("n", [0, 1, 255, 4096, 4097, 300001])
def test_count_of_rows_with_kept_edges(api, n):
    deg = (np.arange(n) % 3).astype(np.int32)
    assert api.count_nonzero(torch.from_numpy(deg).cuda()) == int(np.count_nonzero(deg))
