"""Which segment FFT passes a plan takes, and whole transforms through each of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def noise(torch, N, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.rand((N, 2), generator=g, device="cuda", dtype=torch.float64).mul_(2).sub_(1)
    return torch.view_as_complex(x).to(torch.complex64)


def dft(torch, x):
    return torch.fft.fft(x.to(torch.complex128))


def rel(torch, y, ref):
    return (torch.linalg.norm(y.to(torch.complex128) - ref) / torch.linalg.norm(ref)).item()


@pytest.mark.parametrize("N,P", [(2 ** 22, 4), (2 ** 20, 4), (3 * 2 ** 20, 4), (5 * 2 ** 18, 4), (9 * 2 ** 19, 4)])
def test_passes_follow_the_segment_length(soi, torch_cuda, N, P):
    """Complex64 plans of the same segment length, 4 and 32 segments (N below and from 2^24): the same
    alternatives, and the passes' error is the same."""
    torch, got = torch_cuda, []
    for n, p in ((N, P), (8 * N, 8 * P)):
        d = soi.make_descriptor(n, p, precision=soi.SOI_PREC_FP32)
        try:
            x = noise(torch, n, 3)
            ref = dft(torch, x)
            torch.cuda.synchronize()
            soi.compute_soi(d, x.data_ptr())
            got.append((soi.fft_variants(d), rel(torch, x, ref)))
        finally:
            soi.free_soi_descriptor(d)
    print(f"case N={N} P={P}: {got}", flush=True)
    assert got[0][0] == got[1][0]
    assert max(e for _, e in got) < 3.5e-7


CHAINS = [(3 * 2 ** 23, 8), (27 * 2 ** 20, 16), (75 * 2 ** 18, 16), (9 * 2 ** 21, 4), (3 * 2 ** 20, 4)]


@pytest.mark.parametrize("N,P", CHAINS)
def test_chains_whole_transform(soi, torch_cuda, N, P):
    """Complex64 through the chains of small radices with the tables and buffers of a real plan: split,
    twiddle table in LDS (2^9 to 2^12 entries), tile buffer, rows of more than 2560 points
    (9*2^21).  Bound: the largest error of complex64 transforms measured, 3.5e-7; and two members of a batch equal
    the single transform bit for bit."""
    torch = torch_cuda
    x = noise(torch, N, 5)
    ref = dft(torch, x)
    descs = [soi.make_descriptor(N, P, precision=soi.SOI_PREC_FP32) for _ in range(2)]
    try:
        assert soi.fft_variants(descs[0]) == 1
        y = x.clone()
        torch.cuda.synchronize()
        print(f"case N={N} P={P}", flush=True)
        soi.compute_soi(descs[0], y.data_ptr())
        e = rel(torch, y, ref)
        print(f"  {e:.3e}", flush=True)
        assert e < 3.5e-7
        bufs = [x.clone(), x.clone()]
        torch.cuda.synchronize()
        b = soi.Batch(descs, [t.data_ptr() for t in bufs], autotune=False)
        try:
            for _ in range(2):
                for t in bufs:
                    t.copy_(x)
                torch.cuda.synchronize()
                b.run()
                torch.cuda.synchronize()
                for t in bufs:
                    assert torch.equal(torch.view_as_real(t).view(torch.int32), torch.view_as_real(y).view(torch.int32))
        finally:
            b.close()
    finally:
        for d in descs:
            soi.free_soi_descriptor(d)


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("N,P,alternatives", [(2 ** 24, 8, 2), (2 ** 24, 4, 2), (5 * 2 ** 20, 8, 2), (2 ** 22, 16, 1)])
def test_every_alternative(soi, torch_cuda, N, P, alternatives, single):
    """Every alternative tile of a plan (two where a length has more than 640 points, but rows of 2048) against the
    FP64 DFT, and against alternative 0: the same stages in the same order, so within 1e-15 in
    complex128 and 1e-6 in complex64."""
    torch = torch_cuda
    g = torch.Generator(device="cuda").manual_seed(9)
    x = torch.view_as_complex(torch.rand((N, 2), generator=g, device="cuda", dtype=torch.float64).mul_(2).sub_(1))
    if single:
        x = x.to(torch.complex64)
    ref = dft(torch, x)
    d = soi.make_descriptor(N, P, precision=soi.SOI_PREC_FP32 if single else soi.SOI_PREC_FP64)
    try:
        nv, outs, errs = soi.fft_variants(d), [], []
        assert nv >= alternatives
        for v in range(nv):
            soi.set_fft_variant(d, v)
            y = x.clone()
            torch.cuda.synchronize()
            soi.compute_soi(d, y.data_ptr())
            errs.append(rel(torch, y, ref))
            outs.append(y)
        apart = [rel(torch, y, outs[0].to(torch.complex128)) for y in outs]
    finally:
        soi.free_soi_descriptor(d)
    print(f"case N={N} P={P} single={single}: {errs}, apart {apart}", flush=True)
    assert max(errs) < (3.5e-7 if single else 3e-14)
    assert max(apart) < (1e-6 if single else 1e-15)


@pytest.mark.parametrize("single", [False, True])
def test_forced_column_length(soi, torch_cuda, monkeypatch, single):
    """SOI_FFT_N1 takes another split (other roundings) of the same transform."""
    torch = torch_cuda
    N, P = 2 ** 24, 4
    x = noise(torch, N, 9) if single else noise(torch, N, 9).to(torch.complex128)
    ref, outs = dft(torch, x), []
    for n1 in (None, "2048", "2560"):
        if n1:
            monkeypatch.setenv("SOI_FFT_N1", n1)
        d = soi.make_descriptor(N, P, precision=soi.SOI_PREC_FP32 if single else soi.SOI_PREC_FP64)
        try:
            y = x.clone()
            torch.cuda.synchronize()
            soi.compute_soi(d, y.data_ptr())
        finally:
            soi.free_soi_descriptor(d)
        assert rel(torch, y, ref) < (3.5e-7 if single else 3e-14)
        outs.append(y)
    assert not torch.equal(outs[1], outs[2])
    assert torch.equal(outs[0], outs[1]) or torch.equal(outs[0], outs[2])
