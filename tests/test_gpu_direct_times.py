"""The times a drop-in call without a plan reports: part_time holds what a plan's
creation would do on the host, comm_time the copies alone.  Kernel 3 on a matrix of
2 M rows, nearly all empty, lists its empty rows on the host (two passes over the
rows, 16 MB written: no less than 1 ms at 16 GB/s), kernel 2 needs no list."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_host_analysis_is_part_time():
    from hpda_sblas_pnnl_amd import spmv
    m, n = 2_000_000, 1000
    lens = np.zeros(m, np.int64)
    lens[::50] = 1
    rp = np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
    nnz = int(rp[-1])
    rng = np.random.default_rng(0)
    col = rng.integers(0, n, nnz).astype(np.int32)
    val, x = rng.standard_normal(nnz), rng.uniform(-1, 1, n)
    part = {2: [], 3: []}
    for _ in range(4):
        for kernel in part:
            y = np.zeros(m)
            ret = spmv.spMV_mgpu_v1(m, n, nnz, 1.0, val, rp, col, x, 0.0, y, 1, kernel)
            assert np.array_equal(y[lens == 0], np.zeros(m - nnz))
            assert np.allclose(y[lens == 1], val * x[col], rtol=1e-15)
            assert min(ret.comm_time, ret.comp_time, ret.merg_time) > 0
            part[kernel].append(ret.part_time)
    assert min(part[3]) - min(part[2]) > 1e-3
