"""The element-wise kernels of CGS and BiCGSTAB where a thread takes one row, a
few, and several steps of four: two iterations against the oracle.  Only the
order of the dot products differs, so x agrees to a few roundings, which two
iterations' quotients of dot products magnify by no more than 1e4 (1e-11)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", [3, 7, 8, 33, 73, 74, 93, 101, 118])
@pytest.mark.parametrize("solver,prec", [("bcgs", "jacobi"), ("bcgs", "none"), ("cgs", "jacobi"),
                                         ("cgs", "none")])
def test_two_iterations(cases, oracle, gpu, side, solver, prec):
    s = cases.upwind(side)
    print(f"nonsym items {side}^3 {solver} {prec}", flush=True)
    x = np.random.default_rng(11).uniform(-1, 1, s.n)
    ref = x.copy()
    A = oracle.Matrix(s.row, s.col, s.dia, s.val.copy())
    it_ref, _ = oracle.solve(solver, prec, A, ref, s.b.copy(), 2, 1e-30, criterion="relres")
    nat = gpu.Native(s.row, s.col, s.dia)
    y = x.copy()
    it, _ = nat.solve_native(solver, prec, s.val, y, s.b, 2, 1e-30,
                             options=gpu.Options(criterion=gpu.CRIT_RELRES))
    assert it == it_ref and np.linalg.norm(y - ref) <= 1e-11 * np.linalg.norm(ref)
