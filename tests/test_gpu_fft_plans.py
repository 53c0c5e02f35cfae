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
