"""The CG update that carries x (NRMS over the x range), at 1048576 rows, where
a thread takes one pair per step, and just above, where it takes two: three
iterations against the oracle.  Only the order of the dot products differs, so
x agrees to a few roundings (1e-12)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(128, 128, 64), (17, 61681, 1)])
@pytest.mark.parametrize("prec", ["jacobi", "none"])
def test_three_iterations(cases, oracle, gpu, dims, prec):
    s = cases.hex_pressure(*dims, rho_out=10.0)
    print(f"update items {dims} n={s.n} {prec}", flush=True)
    x = np.random.default_rng(3).uniform(-1, 1, s.n)
    ref = x.copy()
    A = oracle.Matrix(s.row, s.col, s.dia, s.val.copy())
    oracle.solve("cg", prec, A, ref, s.b.copy(), 3, 1e-30)
    it, _ = gpu.Native(s.row, s.col, s.dia).solve_native("cg", prec, s.val, x, s.b, 3, 1e-30)
    assert it == 3 and np.linalg.norm(x - ref) <= 1e-12 * np.linalg.norm(ref)
