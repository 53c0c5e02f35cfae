"""Every transform length of the register FFT passes, as columns, as rows and as a whole segment,
in both precisions, against torch's FP64 DFT of the same input.

The partner length is 100 (partial tiles: 100 is no multiple of 8 or 16).  Bounds: relative L2 <= 3e-14 (the default window's truncation and FP64
rounding, the bound of the plain form elsewhere) and 1e-6 for complex64 (its stated bound)."""
import os
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HEADER = os.path.join(os.path.dirname(__file__), "..", "soi_fft_amd", "csrc", "soi_fft_lengths.h")


def lengths(*lists):
    text = open(HEADER).read()
    out = []
    for name in lists:
        body = re.search(r"#define SOI_FFT_%s\(X\)((?:.*\\\n)*.*)" % name, text).group(1)
        out += [int(n) for n in re.findall(r"X\((\d+),", body)]
    return sorted(out)


def check(soi, torch, M_hat, P, k, single):
    M = M_hat * 4 // 5
    N = M * P * k
    assert 4 * M_hat % 5 == 0 and M % (4 * P) == 0 and M // P >= 72
    g = torch.Generator(device="cuda").manual_seed(M_hat)
    x = torch.view_as_complex(torch.rand((N, 2), generator=g, device="cuda", dtype=torch.float64) * 2 - 1)
    if single:
        x = x.to(torch.complex64)
    ref = torch.fft.fft(x.to(torch.complex128))
    y = x.clone()
    torch.cuda.synchronize()
    d = soi.make_descriptor(N, P, k, precision=soi.SOI_PREC_FP32 if single else soi.SOI_PREC_FP64)
    try:
        errs = []
        for v in range(soi.fft_variants(d)):
            soi.set_fft_variant(d, v)
            y.copy_(x)
            torch.cuda.synchronize()
            soi.compute_soi(d, y.data_ptr())
            errs.append((torch.linalg.norm(y - ref) / torch.linalg.norm(ref)).item())
    finally:
        soi.free_soi_descriptor(d)
    print(f"case M_hat={M_hat} N={N} P={P} k={k} single={single}: {errs}", flush=True)
    assert max(errs) < (1e-6 if single else 3e-14)


@pytest.mark.parametrize("L", lengths("SHORT", "LONG", "LONGEST"))
def test_columns_and_rows(soi, torch_cuda, monkeypatch, L):
    """L x 100 and 100 x L."""
    for n1 in (L, 100):
        monkeypatch.setenv("SOI_FFT_N1", str(n1))
        for single in (False, True):
            check(soi, torch_cuda, 100 * L, 4, 1, single)


@pytest.mark.parametrize("L", [n for n in lengths("ONE") if n % 5 == 0])
def test_one_pass(soi, torch_cuda, L):
    P, k = (4, 1) if L % 20 == 0 else (2, 2) if L % 10 == 0 else (1, 4)
    for single in (False, True):
        check(soi, torch_cuda, L, P, k, single)


@pytest.mark.parametrize("L", [n for n in lengths("ONE") if n % 32 == 0 and n % 5])
def test_one_pass_mu87(soi, orc, torch_cuda, L):
    """Whole-segment lengths without a factor 5, which mu = 8/7 gives, against the oracle: two FP64
    implementations agree to 2 eps max|W_inv| (that window's truncation, 4e-12 to 2e-11 for
    segments this short, is in both)."""
    torch = torch_cuda
    kw = dict(n_mu=8, d_mu=7, tau=0.7, sigma=360.0)
    N = L * 7 // 8 * 4
    p = orc.params(N, 4, **kw)
    x = orc.uniform_input(N, L)
    ref, _ = orc.compute_soi(p, x)
    xt = torch.from_numpy(x).cuda()
    d = soi.make_descriptor(N, 4, **kw)
    try:
        torch.cuda.synchronize()
        soi.compute_soi(d, xt.data_ptr())
    finally:
        soi.free_soi_descriptor(d)
    e = np.linalg.norm(xt.cpu().numpy() - ref) / np.linalg.norm(ref)
    print(f"case M_hat={L}: {e}", flush=True)
    assert e < 2 * 2.0 ** -52 * np.abs(orc.w_inv_table(p)).max()
