"""Products of an unstructured matrix in random numbering (no windows of
columns): entries dealt to the threads up to 262144 rows, a row per thread
above, its matrix loads non-temporal where x passes 5.5 MB (92^3 in FP64, 116^3
in the FP32 form).  Bit for bit against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(64, 64, 64), (64, 64, 65), (71, 73, 77), (92, 92, 93), (116, 116, 116)])
def test_products(cases, oracle, gpu, dims):
    s = cases.knn(*dims)
    print(f"scattered {dims} n={s.n} nnz={len(s.col)}", flush=True)
    nat = gpu.Native(s.row, s.col, s.dia)
    nat.reorder(gpu.ORDER_NATURAL)
    nat.spmv_select(5)
    A = oracle.Matrix(s.row, s.col, s.dia, s.val)
    rng = np.random.default_rng(8)
    p, b = rng.standard_normal(s.n), rng.standard_normal(s.n)
    dv, dp, db, dq = (gpu.DeviceArray(a) for a in (s.val, p, b, np.zeros(s.n)))
    nat.spmv(dv, dp, dq)
    assert np.array_equal(dq.download(), oracle.spmv(A, p))
    nat.residual(dv, db, dp, dq)
    assert np.array_equal(dq.download(), oracle.residual(A, b, p))
    fn = 1.0 / (s.val[s.dia - 1].sum() / s.n)
    x = rng.uniform(-1, 1, s.n).astype(np.float32)
    dx, dy = gpu.DeviceArray(x), gpu.DeviceArray(np.zeros(s.n, dtype=np.float32))
    nat.spmv_fp32(dv, fn, dx, dy)
    assert np.array_equal(dy.download(), oracle.lap32_spmv(A, oracle.lap32_form(A, fn), x))
