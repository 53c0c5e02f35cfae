"""The VLC planning kernel over cost ratios that the descriptor takes unchecked."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ratio", [0.0, 1.0, 50.0, -0.01, -1e9, float("inf"), float("nan")])
@pytest.mark.parametrize("P,k", [(4, 2), (64, 1), (1, 8)])
def test_boundaries(soi, orc, torch_cuda, P, k, ratio):
    """Every ratio ends with boundaries between 0 and the number of segments, the oracle's where its walk ends
    in them too (costs that grow from segment to segment); a target that no segment reaches (NaN costs) ends
    at the last one."""
    torch, lib = torch_cuda, soi.lib()
    vp, ci, cl, cd = ctypes.c_void_p, ctypes.c_int, ctypes.c_long, ctypes.c_double
    S, l = P * k, 1004
    e = np.random.default_rng(S).integers(1000, 1040, S).astype(np.int32)
    exps = torch.from_numpy(np.repeat(e, P)).cuda()
    i32 = dict(dtype=torch.int32, device="cuda")
    emi, nw, plan = torch.zeros(S * P, **i32), torch.zeros(S * P, **i32), torch.full((2 + 2 * S + P,), -7, **i32)
    pcs = torch.zeros(S + 1, dtype=torch.float64, device="cuda")
    p = lambda t: vp(t.data_ptr())
    print(f"case P={P} k={k} ratio={ratio}", flush=True)
    assert lib.soik_vlc_plan(p(exps), ci(S), ci(P), ci(k), cl(l), cl(P * l), cd(ratio), p(emi), p(plan),
                             p(pcs), None, p(nw), None) == 0
    torch.cuda.synchronize()
    plan = plan.cpu().numpy()
    bd = plan[1 + 2 * S:]
    assert bd[0] == 0 and bd[P] == S and np.all((bd >= 0) & (bd <= S))
    if np.isfinite(ratio) and ratio >= -0.01:
        counts, boundaries = orc.vlc_plan(P, k, l, P * l, ratio, e)
        assert np.array_equal(plan[1 + S:1 + 2 * S], counts) and np.array_equal(bd, boundaries)
    if np.isnan(ratio):
        assert np.all(bd[1:] == S)
