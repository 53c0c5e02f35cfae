"""The complex128 MFMA filter (soi_filter_g.hpp) in every form against the oracle's
parallel_filter_subsampling: real and complex taps, both mu, every K length, every S; row group
counts with a partial last tile, and enough tiles that blocks walk several.

Bound: relative L2 <= 1e-13, the bound of the plain form's filter stage (the default window's exact
and reference values differ by less, and nothing has been amplified by the demodulation yet)."""
import numpy as np
import pytest

from gpu_util import rel, to_dev

pytestmark = pytest.mark.gpu

WINDOWS = {
    "rt72": dict(),                                                 # real taps, 20 K steps
    "rt76": dict(B=76, tau=872 / 1024, sigma=313.1715),             # 22
    "ct72": dict(window_mode=1),                                    # complex taps, 20
    "ct78": dict(B=78, tau=872 / 1024, sigma=313.1715, window_mode=1),  # 22
    "ct52": dict(B=52, tau=0.6, sigma=180.0),                       # 16
    "ct44": dict(B=44, tau=0.5, sigma=121.0936),                    # 13
    "ct30": dict(B=30, tau=0.154, sigma=73.2102363),                # 10
    "mu87_72": dict(n_mu=8, d_mu=7, tau=0.7, sigma=360.0),          # 20
    "mu87_50": dict(n_mu=8, d_mu=7, B=50, tau=0.5, sigma=200.0),    # 16
    "mu87_78": dict(n_mu=8, d_mu=7, B=78, tau=0.7, sigma=360.0),    # 22 (VALU form at S >= 32)
}


def run(soi, orc, torch, S, M, kw):
    P, k = 4, S // 4
    d = soi.SoiDesc()
    soi.set_default_soi_descriptor(d)
    d.N, d.P = M * S, P
    d.k = k
    for f, v in kw.items():
        setattr(d, f, v)
    at = torch.full((S * d.n_mu * M // d.d_mu,), float("nan"), dtype=torch.complex128, device="cuda")
    d.alpha_tilde = at.data_ptr()
    x = orc.uniform_input(M * S, S + M)
    soi.init_soi_descriptor(d, k)
    try:
        form = soi.filter_form(d)
        xt = to_dev(torch, x)
        soi.parallel_filter_subsampling(d, xt.data_ptr())
        got = at.cpu().numpy().reshape(S, -1)
    finally:
        soi.free_soi_descriptor(d)
    okw = {f: v for f, v in kw.items() if f != "window_mode"}
    ref = orc.filter_subsample(orc.params(M * S, P, k=k, **okw), x)
    e = rel(got, ref)
    print(f"case S={S} M={M} {kw} form={form}: {e:.2e}", flush=True)
    assert e < 1e-13
    return form


@pytest.mark.parametrize("name", WINDOWS)
@pytest.mark.parametrize("S", [4, 8, 16, 32, 64])
def test_filter_form(soi, orc, torch_cuda, S, name):
    kw = WINDOWS[name]
    for M in ((336, 756) if "mu87" in name else (320, 1600)):  # 3 tiles and a part, many and a part
        form = run(soi, orc, torch_cuda, S, M, kw)
        valu = name == "mu87_78" and S >= 32
        assert form == (soi.SOI_FILTER_VALU if valu else soi.SOI_FILTER_MFMA_F64)


@pytest.mark.parametrize("S,M,name", [(4, 100000, "rt72"), (64, 25600, "rt72"),
                                      (32, 25600, "ct44"), (64, 31500, "mu87_72")])
def test_several_tiles_a_block(soi, orc, torch_cuda, S, M, name):
    run(soi, orc, torch_cuda, S, M, WINDOWS[name])


@pytest.mark.parametrize("M", [320, 25600, 54000, 81920])
def test_four_row_buffers(soi, orc, torch_cuda, M):
    """S = 32, resident real taps: rows load three groups (of four a tile) ahead.  Blocks of one, two,
    three and four tiles, the last tile a part."""
    run(soi, orc, torch_cuda, 32, M, WINDOWS["rt72"])
