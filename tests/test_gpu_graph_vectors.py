"""Products of two and four vectors captured into a graph on a stream of its own,
over sorted column panels and over column segments: every replay, with eager
products on another stream between, gives the bits of the eager product."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FORMS = {"panels": dict(variant=3, panel_layout=2, panel_rows=448, chunks=3, part_mode="v1_numa"),
         "segments": dict(kernel="vector", variant=6)}


@pytest.mark.parametrize("k", [2, 4])
@pytest.mark.parametrize("form", list(FORMS))
def test_captured_vectors(monkeypatch, form, k):
    import torch
    from hpda_sblas_pnnl_amd.device import SpmvPlan
    monkeypatch.setenv("SBLAS_SEGMENTS", "7")
    rng = np.random.default_rng(k)
    M, N = 3001, 9001
    lens = rng.integers(250, 401, M)
    rp = np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
    col = np.concatenate([np.sort(rng.integers(0, N, c)) for c in lens]).astype(np.int32)
    plan = SpmvPlan("csr", M, N, torch.from_numpy(rp).cuda(), torch.from_numpy(col).cuda(),
                    torch.from_numpy(rng.standard_normal(len(col))).cuda(), **FORMS[form])
    assert plan.info()["variant"] == FORMS[form]["variant"]
    X, Y0 = (torch.from_numpy(rng.uniform(-1, 1, s)).cuda() for s in ((N, k), (M, k)))
    want = plan.spmm(X, Y0.clone(), -0.75, 0.5)
    Y = Y0.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.spmm(X, Y, -0.75, 0.5)
    for _ in range(3):
        Y.copy_(Y0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(Y, want)
        again = plan.spmm(X, Y0.clone(), -0.75, 0.5)
        torch.cuda.synchronize()
        assert torch.equal(again, want)
