"""The element-wise CG kernels where a thread takes more than one item: sizes
around one, two and several sweeps of the grid, odd and even, each stopping
test, both preconditioners.  Three iterations against the oracle: only the
order of the dot products differs, so x agrees to a few roundings (1e-12)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# rows: one pair per thread and sweep, 768 workgroups of 256 threads: 393216
SIZES = [(1, 1, 513), (13, 11, 9), (96, 64, 64), (64, 64, 97), (101, 103, 97), (128, 96, 100)]


@pytest.mark.parametrize("dims", SIZES)
@pytest.mark.parametrize("crit,norm,prec", [("relres", None, "jacobi"), ("relres", None, "none"),
                                            ("nrms", 1.0, "jacobi"), ("nrms", None, "jacobi")])
def test_three_iterations(cases, oracle, gpu, dims, crit, norm, prec):
    s = cases.hex_pressure(*dims, rho_out=10.0)
    print(f"items {dims} n={s.n} {crit} norm={norm} {prec}", flush=True)
    x = np.random.default_rng(3).uniform(-1, 1, s.n)
    ref = x.copy()
    A = oracle.Matrix(s.row, s.col, s.dia, s.val.copy())
    _, fin_ref = oracle.solve("cg", prec, A, ref, s.b.copy(), 3, 1e-30, norm=norm, criterion=crit)
    nat = gpu.Native(s.row, s.col, s.dia)
    for path in (gpu.PATH_AUTO, gpu.PATH_KERNELS):
        o = gpu.Options(criterion=gpu.CRIT_RELRES if crit == "relres" else gpu.CRIT_NRMS, path=path)
        y = x.copy()
        it, fin = nat.solve_native("cg", prec, s.val, y, s.b, 3, 1e-30, norm=norm, options=o)
        assert it == 3 and np.linalg.norm(y - ref) <= 1e-12 * np.linalg.norm(ref)
        assert abs(fin - fin_ref) <= 1e-10 * fin_ref
