"""The register passes of long complex64 transforms against the LDS kernels (k_fft_col,
k_fft_row): same radices, twiddles and roundings, so equal bit for bit."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Batch(ctypes.Structure):
    _fields_ = [("x", ctypes.c_void_p), ("at", ctypes.c_void_p), ("tb", ctypes.c_void_p),
                ("n", ctypes.c_int)]


def _table(torch, L, n, mult=1):
    a = (torch.arange(n, dtype=torch.float64, device="cuda") * mult) % L * (-2 * np.pi / L)
    return torch.complex(torch.cos(a), torch.sin(a)).to(torch.complex64)


def _noise(torch, n, dtype=None):
    return torch.view_as_complex(torch.randn((n, 2), device="cuda", dtype=dtype))


def _bits(torch, a):
    return torch.view_as_real(a).view(torch.int32)


COLS = [576, 600, 640, 720, 768, 800, 960, 1000, 1024, 1080, 1152, 1200, 1280, 1440, 1536, 1600,
        1920, 2000, 2048, 2160, 2304, 2400, 2560]
ROWS = COLS + [2880, 3072, 3200, 3456, 3840]


@pytest.mark.parametrize("L", COLS)
def test_columns_match_lds_kernel(soi, torch_cuda, L):
    """20 columns: a last tile of four, and enough rows that the twiddle exponents span the table."""
    torch, lib = torch_cuda, soi.lib()
    vp, ci, cl = ctypes.c_void_p, ctypes.c_int, ctypes.c_long
    lib.soik_fft_col_f32.argtypes = [vp] * 4 + [ci] * 4 + [cl, ci, Batch, vp]
    lib.soik_fft_longd_cols.argtypes = [vp] * 4 + [ci] * 3 + [cl, ci, vp, cl, Batch, vp]
    assert lib.soik_fft_longd_supported(L, 0)
    n2, S = 20, 3
    Mh = L * n2
    lb = max(6, (Mh - 1).bit_length() // 2)
    tw, thi, tlo = _table(torch, L, L), _table(torch, Mh, (Mh >> lb) + 1, 1 << lb), _table(torch, Mh, 1 << lb)
    torch.manual_seed(L)
    x = _noise(torch, S * Mh)
    ref, out = x.clone(), torch.zeros(S * Mh, dtype=torch.complex64, device="cuda")
    print(f"case columns L={L}", flush=True)
    b = Batch()
    assert lib.soik_fft_col_f32(ref.data_ptr(), tw.data_ptr(), thi.data_ptr(), tlo.data_ptr(), L, n2,
                                2, 1 << lb, Mh, S, b, None) == 0
    assert lib.soik_fft_longd_cols(x.data_ptr(), tw.data_ptr(), thi.data_ptr(), tlo.data_ptr(), L,
                                   n2, lb, Mh, S, out.data_ptr(), Mh, b, None) == 0
    torch.cuda.synchronize()
    got = out.view(S, L // 8, n2, 8).permute(0, 1, 3, 2).reshape(-1)  # 8-row tiles
    assert torch.equal(_bits(torch, got), _bits(torch, ref))


@pytest.mark.parametrize("L", ROWS)
def test_rows_match_lds_kernel(soi, torch_cuda, L):
    """40 rows in five segments (a last group of one segment), some outputs past M dropped."""
    torch, lib = torch_cuda, soi.lib()
    vp, ci, cl = ctypes.c_void_p, ctypes.c_int, ctypes.c_long
    lib.soik_fft_row_f32.argtypes = [vp] * 4 + [ci] * 3 + [cl, cl, ci, Batch, vp]
    lib.soik_fft_longd_rows.argtypes = [vp] * 4 + [ci] * 2 + [cl, cl, ci, Batch, vp]
    assert lib.soik_fft_longd_supported(L, 1)
    n1, S = 40, 5
    Mh = n1 * L
    M = Mh * 4 // 5
    torch.manual_seed(L)
    tw, winv, z = _table(torch, L, L), _noise(torch, M, torch.float64), _noise(torch, S * Mh)
    tiles = z.view(S, n1 // 8, 8, L).permute(0, 1, 3, 2).reshape(-1).contiguous()
    X = [torch.zeros(S * M + 8, dtype=torch.complex64, device="cuda") for _ in range(2)]
    print(f"case rows L={L}", flush=True)
    b = Batch()
    Tr = 2 if L <= 2560 else 1
    assert lib.soik_fft_row_f32(z.data_ptr(), X[0].data_ptr(), tw.data_ptr(), winv.data_ptr(), n1, L,
                                Tr, Mh, M, S, b, None) == 0
    assert lib.soik_fft_longd_rows(tiles.data_ptr(), X[1].data_ptr(), tw.data_ptr(),
                                   winv.data_ptr(), n1, L, Mh, M, S, b, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(_bits(torch, X[0]), _bits(torch, X[1]))
