"""A plan over two column segments keeps sums of two vectors a virtual row, not of
four, which never run over its segments: with M virtual rows of 1.75 a row at three
elements a row, its format (12 bytes an element, 13 a virtual row), 16 M bytes of
sums and row blocks stay under 105 bytes a row; 32 M bytes of sums would pass 115."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_sums_of_two_vectors(monkeypatch):
    import torch
    from hpda_sblas_pnnl_amd.device import SpmvPlan
    monkeypatch.setenv("SBLAS_SEGMENTS", "2")
    rng = np.random.default_rng(0)
    m = 200_000
    rp = np.arange(0, 3 * m + 1, 3, dtype=np.int32)
    col = np.sort(rng.integers(0, m, (m, 3)), axis=1).astype(np.int32)
    plan = SpmvPlan("csr", m, m, torch.from_numpy(rp).cuda(), torch.from_numpy(col.ravel()).cuda(),
                    torch.from_numpy(rng.standard_normal(3 * m)).cuda(), kernel="vector", variant=6)
    info = plan.info()
    assert info["variant"] == 6 and 1.7 * m < info["virtual_rows"] < 1.8 * m
    assert info["workspace_bytes"] < 105 * m
