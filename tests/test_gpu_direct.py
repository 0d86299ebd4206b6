"""Drop-in calls without a plan (csrc/direct.cpp): every kernel, calls that
grow and reuse the call context, calls from several threads at once, refused
inputs.  Against the FP64 oracle within the roundings of two sums of L products
in different orders, 2 (L + 3) 2^-53 of alpha * sum |a x| + |beta y|."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(seed, m, n, mean, long_row=0):
    rng = np.random.default_rng(seed)
    lens = np.minimum(rng.geometric(1.0 / mean, m) - 1, n)
    if long_row:
        lens[m // 2] = min(long_row, n)
    rp = np.zeros(m + 1, np.int64)
    np.cumsum(lens, out=rp[1:])
    col = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lens]).astype(np.int32)
    return (rp.astype(np.int32), col, rng.standard_normal(len(col)), rng.uniform(-1, 1, n),
            rng.uniform(-1, 1, m))


def _check(oracle, mat, y, alpha, beta):
    rp, col, val, x, y0 = mat
    m, n = len(rp) - 1, len(x)
    ref = oracle.csr_spmv(m, n, val, rp, col, x, alpha, beta, y0)
    scale = oracle.csr_spmv(m, n, np.abs(val), rp, col, np.abs(x), abs(alpha), abs(beta),
                            np.abs(y0))
    return (np.abs(y - ref) <= 2 * (np.diff(rp) + 3) * 2.0 ** -53 * scale).all()


def _run(mat, kernel, alpha, beta):
    from hpda_sblas_pnnl_amd import spmv
    rp, col, val, x, y0 = mat
    y = y0.copy()
    ret = spmv.spMV_mgpu_v1(len(rp) - 1, len(x), len(val), alpha, val, rp, col, x, beta, y, 1,
                            kernel)
    assert ret.comp_time > 0 and ret.comm_time > 0
    return y


# one row; a row over several blocks; y beyond the pinned buffer; the staging
# ring's sizes
SIZES = [(1, 50, 20, 0), (300, 9000, 5, 7000), (140_001, 500, 2, 0), (60_000, 60_000, 14, 0)]


@pytest.mark.parametrize("kernel", [1, 2, 3])
def test_direct_sizes(oracle, kernel, monkeypatch):
    mats = [_matrix(i, *s) for i, s in enumerate(SIZES)]
    for mat in mats + mats[::-1]:  # the context grows, then is larger than needed
        if not len(mat[2]):
            continue
        for alpha, beta in ((1.0, 0.0), (-0.5, 2.0)):
            assert _check(oracle, mat, _run(mat, kernel, alpha, beta), alpha, beta)
    monkeypatch.setenv("SBLAS_CHUNKS", "7")
    assert _check(oracle, mats[1], _run(mats[1], kernel, 1.5, -1.0), 1.5, -1.0)


def test_direct_threads(oracle):
    mats = [_matrix(20 + i, 500 + 100 * i, 3000, 8) for i in range(4)]
    good = [True] * 4

    def work(i):
        for _ in range(10):
            good[i] &= bool(_check(oracle, mats[i], _run(mats[i], 1 + i % 3, 1.0, 0.5), 1.0, 0.5))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(good)


@pytest.mark.parametrize("kernel", [1, 2, 3])
def test_direct_refuses(kernel):
    from hpda_sblas_pnnl_amd import SblasError, _lib, spmv
    rp, col, val, x, y0 = _matrix(3, 200, 300, 6)
    for bad in ("column", "negative", "rows"):
        c, r = col.copy(), rp.copy()
        if bad == "rows":
            r[10], r[11] = r[11] + 1, r[10]
        else:
            c[len(c) // 2] = 300 if bad == "column" else -1
        y = y0.copy()
        with pytest.raises(SblasError) as e:
            spmv.spMV_mgpu_v1(200, 300, len(val), 1.0, val, r, c, x, 0.5, y, 1, kernel)
        assert e.value.status == _lib.SBLAS_ERR_ARGS and np.array_equal(y, y0)
