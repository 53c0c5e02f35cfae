"""How far the complex128 stages are from the exact result, in isolation, against long double: a form on
the matrix units or with larger radices is no less accurate than the plain one that it replaced."""
import ctypes

import numpy as np
import pytest

from gpu_util import d2h, to_dev

pytestmark = pytest.mark.gpu

LD = np.longdouble
PI = LD("3.14159265358979323846264338327950288")


def rel_rms(got, ref):
    e = got.astype(np.clongdouble) - ref
    return float(np.sqrt((np.abs(e) ** 2).sum() / (np.abs(ref) ** 2).sum()))


def cis(num, den):
    """e^{i pi num/den} of integers"""
    r = np.asarray(num) % (2 * den)
    a = PI * np.where(r > den, r - 2 * den, r).astype(LD) / LD(den)
    return np.cos(a) + 1j * np.sin(a)


def exact_filter(x, S, M, n_mu, d_mu, B, tau, sigma, w):
    """parallel_filter_subsampling in long double, [S][M_hat]: with the window's closed form, or with the
    table w of complex taps [theta][b][i]"""
    nJ, mu = M // d_mu, LD(n_mu) / d_mu
    rows = x.reshape(M, S).astype(np.clongdouble)
    i = np.arange(S)
    out = np.zeros((nJ, n_mu, S), np.clongdouble)
    for th in range(n_mu):
        for b in range(B):
            if w is None:
                num = 2 * th * d_mu * S + (B - d_mu) * n_mu * S - 2 * i * n_mu - 2 * b * n_mu * S
                t = num.astype(LD) / (2 * n_mu * S)
                a = PI * LD(tau) * t
                y = np.where(a == 0, LD(1), np.sin(a) / np.where(a == 0, LD(1), a))
                wb = cis(num, 2 * n_mu * S) * (y * np.exp(-PI * PI * t * t / LD(sigma)) / mu)
            else:
                wb = w[th, b].astype(np.clongdouble)
            out[:, th, :] += rows[(np.arange(nJ) * d_mu + b) % M] * wb
    return (out.reshape(nJ * n_mu, S) @ cis(-2 * np.outer(i, i), S)).T


WINDOWS = {
    "b72": dict(window_mode=2),
    "b76": dict(window_mode=2, B=76, tau=872 / 1024, sigma=313.1715),
    "b64": dict(window_mode=2, B=64, tau=818 / 1024, sigma=267.4513),
    "b60": dict(window_mode=2, B=60, tau=0.75, sigma=230.0),
    "mu87": dict(n_mu=8, d_mu=7, tau=0.7, sigma=360.0),
    "ct72": dict(window_mode=1),
    "ct52": dict(B=52, tau=0.6, sigma=180.0),
    "b44": dict(B=44, tau=0.5, sigma=121.0936),
    "b30": dict(B=30, tau=0.154, sigma=73.2102363),
}
# Error of the VALU form (FP64 FMAs in two slices of real taps, four of complex) on these inputs, 1e-16
VALU = {
    "b72": {64: 3.280}, "b64": {64: 3.183}, "b60": {64: 2.935},
    "b76": {4: 2.529, 16: 2.892, 32: 2.976, 64: 3.172},
    "mu87": {4: 1.737, 16: 1.990, 32: 2.094, 64: 2.221},
    "ct72": {4: 1.724, 16: 1.969, 32: 2.065, 64: 2.188},
    "ct52": {4: 1.978, 16: 2.184, 32: 2.273, 64: 2.393},
    "b44": {4: 1.506, 16: 1.785, 32: 1.877, 64: 2.024},
    "b30": {4: 1.594, 16: 1.826, 32: 1.929, 64: 2.069},
}


@pytest.mark.parametrize("name,S", [(n, S) for n, v in VALU.items() for S in v])
def test_filter_error(soi, torch_cuda, name, S):
    """The MFMA filter against the error of the VALU form, 3% for what depends on the inputs.  Real taps are
    judged by the window itself, complex ones (the reference's values) by the descriptor's table."""
    torch, kw = torch_cuda, WINDOWS[name]
    n_mu, d_mu, B = kw.get("n_mu", 5), kw.get("d_mu", 4), kw.get("B", 72)
    M = 1792 if n_mu == 8 else 1600
    rng = np.random.default_rng(S)
    x = rng.uniform(-1, 1, M * S) + 1j * rng.uniform(-1, 1, M * S)
    d = soi.SoiDesc()
    soi.set_default_soi_descriptor(d)
    d.N, d.P, d.k = M * S, 4, S // 4
    for f, v in kw.items():
        setattr(d, f, v)
    at = torch.zeros(S * n_mu * M // d_mu, dtype=torch.complex128, device="cuda")
    d.alpha_tilde = at.data_ptr()
    soi.init_soi_descriptor(d, S // 4)
    try:
        assert soi.filter_form(d) == soi.SOI_FILTER_MFMA_F64
        w = None if kw.get("window_mode") == 2 else d2h(ctypes.c_void_p(d.w), n_mu * B * S, np.complex128)
        xt = to_dev(torch, x)
        torch.cuda.synchronize()
        soi.parallel_filter_subsampling(d, xt.data_ptr())
        got = at.cpu().numpy().reshape(S, -1)
    finally:
        soi.free_soi_descriptor(d)
    ref = exact_filter(x, S, M, n_mu, d_mu, B, d.tau, d.sigma, None if w is None else w.reshape(n_mu, B, S))
    e = rel_rms(got, ref)
    print(f"case {name} S={S}: {e:.3e}, VALU form {VALU[name][S]}e-16", flush=True)
    assert e < 1.03e-16 * VALU[name][S]


class Batch(ctypes.Structure):
    _fields_ = [("x", ctypes.c_void_p), ("at", ctypes.c_void_p), ("tb", ctypes.c_void_p),
                ("n", ctypes.c_int)]


# Error, 1e-16, of the passes with stages of radix 10 and less or on the LDS kernels, their tables' too
PASSES = [("cols", 48, 2.067), ("cols", 240, 2.545), ("cols", 480, 2.651), ("rows", 64, 1.526),
          ("rows", 512, 1.984), ("one", 1152, 2.382), ("one", 1280, 2.276), ("one", 5120, 2.508)]


@pytest.mark.parametrize("kind,L,former", PASSES)
def test_pass_error(soi, torch_cuda, kind, L, former):
    """A complex128 FFT pass with the library's own twiddle tables against the error of the stages and
    tables before these, 4% for what depends on the inputs."""
    import scipy.fft
    torch, lib, vp, cl = torch_cuda, soi.lib(), ctypes.c_void_p, ctypes.c_long

    def table(n, mult, of):
        t = torch.zeros(n, dtype=torch.complex128, device="cuda")
        assert lib.soik_make_twiddles(vp(t.data_ptr()), cl(n), cl(of), cl(mult), None) == 0
        return t

    p = lambda t: vp(t.data_ptr())
    b, other, S = Batch(), 40, 4
    if kind == "one":
        other, S = 1, 32
    Mh = L * other
    rng = np.random.default_rng(L)
    shape = (S, L, other) if kind == "cols" else (S, other, L)
    x = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    y = to_dev(torch, x)
    out = torch.zeros(S * Mh, dtype=torch.complex128, device="cuda")
    one = torch.ones(Mh, dtype=torch.complex128, device="cuda")
    tw = table(L, 1, L)
    print(f"case {kind} L={L}", flush=True)
    ref = scipy.fft.fft(x.astype(np.clongdouble), axis=1 if kind == "cols" else 2)
    if kind == "cols":
        lb = max(6, (Mh - 1).bit_length() // 2)
        hi, lo = table((Mh >> lb) + 1, 1 << lb, Mh), table(1 << lb, 1, Mh)
        assert lib.soik_fft_cols(p(y), p(tw), p(hi), p(lo), L, other, lb, cl(Mh), S, 0, None, cl(0), b, None) == 0
        out, ref = y, ref * cis(-2 * np.outer(np.arange(L), np.arange(other)), Mh)
    elif kind == "rows":
        assert lib.soik_fft_rows(p(y), p(out), p(tw), p(one), other, L, cl(Mh), cl(Mh), S, 0, b, None) == 0
        ref = ref.transpose(0, 2, 1)
    else:
        assert lib.soik_fft_one(p(y), p(out), p(tw), p(one), L, cl(L), S, b, None) == 0
    torch.cuda.synchronize()
    e = rel_rms(out.cpu().numpy().reshape(ref.shape), ref)
    print(f"  {e:.3e}, before {former}e-16", flush=True)
    assert e < 1.04e-16 * former


# Error, 1e-7, of complex64 transforms of uniform noise on the LDS kernels' stages
SINGLE = [(40960, 8, 2.779), (9 * 2 ** 19, 8, 3.172), (27 * 2 ** 18, 8, 3.170), (27 * 2 ** 18, 32, 3.161),
          (3 * 2 ** 22, 8, 3.210)]


@pytest.mark.parametrize("N,P,former", SINGLE)
def test_single_precision_error(soi, torch_cuda, N, P, former):
    """Lengths with odd factors against the error of the kernels before the register passes, 0.5% for
    what depends on the inputs."""
    torch = torch_cuda
    g = torch.Generator(device="cuda").manual_seed(10)
    x = torch.rand((N, 2), generator=g, device="cuda", dtype=torch.float64).mul_(2).sub_(1)
    x = torch.view_as_complex(x).to(torch.complex64)
    ref = torch.fft.fft(x.to(torch.complex128))
    d = soi.make_descriptor(N, P, precision=soi.SOI_PREC_FP32)
    try:
        torch.cuda.synchronize()
        soi.compute_soi(d, x.data_ptr())
    finally:
        soi.free_soi_descriptor(d)
    e = (torch.linalg.norm(x.to(torch.complex128) - ref) / torch.linalg.norm(ref)).item()
    print(f"case N={N} P={P}: {e:.4e}, before {former}e-7", flush=True)
    assert e < 1.005e-7 * former
