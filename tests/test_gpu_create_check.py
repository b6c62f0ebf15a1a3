"""The check of a CSR's columns at npbcg_create on both sides of the size that decides
whether host or device makes it: a column outside the matrix is refused wherever it lies,
descending columns are taken and solved on the CSR kernels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnz", [1, 64, 32767, 32768, 32769])
def test_columns(gpu, nnz):
    n = min(nnz, 300)   # a band, with what is left over in the first row
    per = nnz // n
    length = np.full(n, per)
    length[0] += nnz - per * n
    rowstr = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
    k = np.arange(nnz) - np.repeat(rowstr[:-1], length)
    colidx = ((np.repeat(np.arange(n), length) + k) % n).astype(np.int32)
    a = np.where(k == 0, 1000.0, 0.5)
    for at, bad in ((0, n), (nnz // 2, -1), (nnz - 1, 1 << 30)):
        ci = colidx.copy()
        ci[at] = bad
        with pytest.raises(gpu.NpbcgError) as e:
            gpu.Context(gpu.Matrix(n, rowstr, ci, a))
        assert e.value.code == gpu.ERR_INVALID
    sort = colidx.copy()
    for j in range(n):
        sort[rowstr[j]:rowstr[j + 1]].sort()
    with gpu.Context(gpu.Matrix(n, rowstr, sort, a), spmv_variant=5) as ctx:
        repeats = any(np.any(np.diff(sort[rowstr[j]:rowstr[j + 1]]) <= 0) for j in range(n))
        assert ctx.describe()["spmv_variant"] == (1 if repeats else 5)
    if nnz > n:
        with gpu.Context(gpu.Matrix(n, rowstr, colidx[::-1].copy(), a), spmv_variant=5) as ctx:
            assert ctx.describe()["spmv_variant"] == 1
