"""Products of 2 and 4 vectors over column segments against the FP64 oracle,
vector by vector: segment counts on both sides of a mask word (32) and the most
(64; at 2 segments four vectors keep the row blocks), rows past the last whole
merge block, empty rows, rows cut across row blocks, Y read and not read, X and
Y 8 bytes off 16.  A result is two sums of L products and P pieces: within
2 (L + P + 3) 2^-53 of alpha * sum |a x| + |beta y|.
"""
import numpy as np
import pytest

from conftest import random_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [2, 7, 33, 64])
@pytest.mark.parametrize("k", [2, 4])
@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
def test_segment_vectors(oracle, monkeypatch, P, k, dtype):
    import torch
    from hpda_sblas_pnnl_amd import gen as G
    from hpda_sblas_pnnl_amd.device import SpmvPlan
    rng = np.random.default_rng(P * 10 + k)
    m, n = 6003, 5003
    rp, col, val = random_csr(rng, m, n, 40, empty_frac=0.25, long_rows=3, long_len=5000)
    if dtype == "f64":
        dval = torch.from_numpy(val).cuda()
    elif dtype == "f32":
        dval = torch.from_numpy(val.astype(np.float32)).cuda()
        val = val.astype(np.float32).astype(np.float64)
    else:
        bits = G.to_bf16_bits(val)
        dval, val = torch.from_numpy(bits.view(np.int16)).cuda(), G.from_bf16_bits(bits)
    monkeypatch.setenv("SBLAS_SEGMENTS", str(P))
    plan = SpmvPlan("csr", m, n, torch.from_numpy(rp).cuda(), torch.from_numpy(col).cuda(), dval,
                    kernel="vector", variant=6)
    assert plan.info()["variant"] == 6 and plan.info()["segments"] == P
    X, Y0 = rng.uniform(-1, 1, (n, k)), rng.uniform(-1, 1, (m, k))
    off = lambda a: torch.empty(a.size + 1, dtype=torch.float64, device="cuda")[1:].view(a.shape)
    dX, dY = off(X), off(Y0)
    dX.copy_(torch.from_numpy(X))
    length = np.diff(rp)
    for alpha, beta in ((1.0, 0.0), (-0.75, 0.5)):
        dY.copy_(torch.from_numpy(Y0))
        plan.spmm(dX, dY, alpha, beta)
        got = dY.cpu().numpy()
        for v in range(k):
            x, y0 = np.ascontiguousarray(X[:, v]), np.ascontiguousarray(Y0[:, v])
            ref = oracle.csr_spmv(m, n, val, rp, col, x, alpha, beta, y0)
            scale = oracle.csr_spmv(m, n, np.abs(val), rp, col, np.abs(x), abs(alpha), abs(beta),
                                    np.abs(y0))
            assert (np.abs(got[:, v] - ref) <= 2 * (length + P + 3) * 2.0 ** -53 * scale).all(), v
