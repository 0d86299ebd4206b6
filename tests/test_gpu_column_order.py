"""Column panels and segments asked for over rows whose columns ascend but for one
pair: refused (row blocks in their place) wherever the pair lies, also next to the
edges of a workgroup's elements; descents from one row to the next do not count."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROW = 1025
NNZ = 5 * ROW  # two workgroups' elements and a part of a third


@pytest.mark.parametrize("variant", [3, 6])
@pytest.mark.parametrize("at", [None, 1, 255, 256, 257, 2047, 2048, 2049, 4095, 4096, NNZ - 1])
def test_one_descent(oracle, variant, at):
    import torch
    from hpda_sblas_pnnl_amd.device import SpmvPlan
    rng = np.random.default_rng(0)
    rp = np.arange(0, NNZ + 1, ROW, dtype=np.int32)
    n = 3 * ROW
    col = np.concatenate([np.sort(rng.choice(n, ROW, replace=False)) for _ in range(5)])
    if at is not None:
        assert at % ROW  # inside a row
        col[[at - 1, at]] = col[[at, at - 1]]
    col = col.astype(np.int32)
    val, x = rng.standard_normal(NNZ), rng.uniform(-1, 1, n)
    plan = SpmvPlan("csr", 5, n, torch.from_numpy(rp).cuda(), torch.from_numpy(col).cuda(),
                    torch.from_numpy(val).cuda(), kernel="vector", variant=variant)
    assert plan.info()["variant"] == (variant if at is None else 2)
    dy = torch.empty(5, dtype=torch.float64, device="cuda")
    plan.spmv(torch.from_numpy(x).cuda(), dy)
    ref = oracle.csr_spmv(5, n, val, rp, col, x, 1.0, 0.0, np.zeros(5))
    scale = oracle.csr_spmv(5, n, np.abs(val), rp, col, np.abs(x), 1.0, 0.0, np.zeros(5))
    assert (np.abs(dy.cpu().numpy() - ref) <= 2 * (ROW + 3) * 2.0 ** -53 * scale).all()
