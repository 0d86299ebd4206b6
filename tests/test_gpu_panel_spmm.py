"""Products of two and four vectors over sorted-group column panels against the
FP64 oracle, one vector at a time: every entry within the roundings of two sums of
L products, 2 (L + 3) 2^-53 of alpha * sum |a x| + |beta y|.
Rows a panel: one group, a round of the waves and more (one pass of four
vectors), and too many for that (two passes of two).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

M, N = 2_499, 9_001  # the last row panel and the last window are part full


@pytest.mark.parametrize("rows", [64, 448, 896, 1024])
@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("k", [2, 4])
def test_panel_spmm(oracle, k, dtype, rows):
    import torch
    from hpda_sblas_pnnl_amd import gen as G
    from hpda_sblas_pnnl_amd.device import SpmvPlan
    rng = np.random.default_rng(rows + k)
    lens = rng.integers(250, 401, M)  # at least 1.5 windows of elements a slice, 4 at 1024 rows
    lens[rng.random(M) < 0.02] = 0
    rp = np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
    col = np.concatenate([np.sort(rng.integers(0, N, c)) for c in lens]).astype(np.int32)
    wide = rng.standard_normal(len(col))
    if dtype == "f64":
        val, dval = wide, torch.from_numpy(wide).cuda()
    elif dtype == "f32":
        val = wide.astype(np.float32).astype(np.float64)
        dval = torch.from_numpy(wide.astype(np.float32)).cuda()
    else:
        bits = G.to_bf16_bits(wide)
        val, dval = G.from_bf16_bits(bits), torch.from_numpy(bits.view(np.int16)).cuda()
    X, Y0 = rng.uniform(-1, 1, (N, k)), rng.uniform(-1, 1, (M, k))
    plan = SpmvPlan("csr", M, N, torch.from_numpy(rp).cuda(), torch.from_numpy(col).cuda(), dval,
                    chunks=3, part_mode="v1_numa", variant=3, panel_layout=2, panel_rows=rows)
    info = plan.info()
    assert (info["variant"], info["panel_layout"], info["panel_rows"]) == (3, 2, rows)
    for shift, alpha, beta in ((0, 1.0, 0.0), (1, -0.75, 0.5)):  # on and off 16 bytes
        dX = torch.empty(N * k + shift, dtype=torch.float64, device="cuda")[shift:].view(N, k)
        dY = torch.empty(M * k + shift, dtype=torch.float64, device="cuda")[shift:].view(M, k)
        dX.copy_(torch.from_numpy(X))
        dY.copy_(torch.from_numpy(Y0))
        plan.spmm(dX, dY, alpha, beta)
        got = dY.cpu().numpy()
        for j in range(k):
            x, y0 = np.ascontiguousarray(X[:, j]), np.ascontiguousarray(Y0[:, j])
            ref = oracle.csr_spmv(M, N, val, rp, col, x, alpha, beta, y0)
            scale = oracle.csr_spmv(M, N, np.abs(val), rp, col, np.abs(x), abs(alpha), abs(beta),
                                    np.abs(y0))
            assert (np.abs(got[:, j] - ref) <= 2 * (lens + 3) * 2.0 ** -53 * scale).all()
