"""The fused VLC exchange (words and decoded elements in one pass over the chunks) against the
per-chunk codec, bit for bit."""
import ctypes

import numpy as np
import pytest

from test_gpu_vlc import _arr, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("length", [
    8,                    # a tail and no vector row
    16,                   # one row
    31 * 16 + 2,          # a unit of 32 rows one short, and a tail
    32 * 16,              # one unit
    33 * 16 + 14,         # one row in the second unit
    4 * 32 * 16,          # one wave's units
    4 * 32 * 16 + 8,
    9 * 32 * 16 + 5 * 16 + 6,
])
def test_exchange_matches_per_chunk_codec(soi, torch_cuda, length):
    """Field widths from 56 bits down to none (a chunk 60 binades below the largest), an all-zero
    chunk among them.  Words and decoded doubles are equal bit for bit, and nothing is written
    past a chunk's words or elements."""
    torch = torch_cuda
    L = soi.lib()
    c_long, c_int, c_void = ctypes.c_long, ctypes.c_int, ctypes.c_void_p
    L.soik_max_exponent.argtypes = [c_void, c_int, c_int, c_void, c_void]
    L.soik_vlc_exchange.argtypes = [c_void, c_long, c_void, c_int, c_int, c_void, c_void, c_void]
    rng = np.random.default_rng(length)
    e = [3, 3, 2, -7, -18, -19, -20, -21, -27, -31, -45, -60, 1]
    nch, stride, mark = len(e), 2 * length + 16, 0x5A5A5A5A
    chunks = [_arr(rng, length, v) for v in e]
    chunks[-1][:] = 0.0
    xt = to_dev(torch, np.concatenate(chunks))
    i32 = dict(dtype=torch.int32, device="cuda")
    emi, nw = torch.zeros(nch, **i32), torch.zeros(nch, **i32)
    print(f"case exchange length={length}", flush=True)
    assert L.soik_max_exponent(xt.data_ptr(), length, nch, emi.data_ptr(), None) == 0
    torch.cuda.synchronize()
    e_max = emi.max().reshape(1).clone()
    words = [torch.full((nch * stride,), mark, **i32) for _ in range(2)]
    y_ref = torch.zeros(nch * length, dtype=torch.float64, device="cuda")
    assert L.soi_compress_batch(words[0].data_ptr(), stride, xt.data_ptr(), length, nch,
                                int(e_max), emi.data_ptr(), nw.data_ptr(), None) == 0
    assert L.soi_decompress_batch(y_ref.data_ptr(), words[0].data_ptr(), stride, length, nch,
                                  int(e_max), emi.data_ptr(), None) == 0
    y = torch.full((nch * length + 16,), 7.0, dtype=torch.float64, device="cuda")
    y[:-16] = xt
    assert L.soik_vlc_exchange(words[1].data_ptr(), stride, y.data_ptr(), length, nch,
                               e_max.data_ptr(), emi.data_ptr(), None) == 0
    torch.cuda.synchronize()
    n = nw.cpu().numpy()
    assert n[0] > 0 and n[-1] == 0
    ref, got = (w.cpu().numpy().reshape(nch, stride) for w in words)
    for c in range(nch):
        assert np.array_equal(got[c, :n[c]], ref[c, :n[c]]), c
        assert np.all(got[c, n[c]:] == mark), c
    assert torch.equal(y[:-16].view(torch.int64), y_ref.view(torch.int64))
    assert torch.all(y[-16:] == 7.0)
