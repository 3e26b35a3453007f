"""Batched vector kernels, a row block per wavefront: systems of one row, around
64 rows (a row per lane), 256 (a block) and more, in counts that leave
wavefronts of a workgroup without a block.  FP64: three iterations, x to a few
roundings (1e-12) of the oracle's; FP32 form: the true residual meets 1e-8."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIDES = [(1, 1, 1), (3, 3, 7), (4, 4, 4), (13, 5, 1), (17, 5, 3), (16, 4, 4), (257, 1, 1), (23, 11, 5)]


def _solve(gpu, systems, miter, tol, **opt):
    off = np.cumsum([0] + [s.n for s in systems])
    cat = lambda name: np.ascontiguousarray(np.concatenate([getattr(s, name) for s in systems]))
    bt = gpu.Batch([(s.row, s.col, s.dia) for s in systems])
    x = np.zeros(off[-1])
    niter, fin, _ = bt.solve("cg", "jacobi", cat("val"), x, cat("b"), miter, tol,
                             options=gpu.Options(criterion=gpu.CRIT_RELRES, **opt))
    bt.close()
    return niter, [x[a:b] for a, b in zip(off, off[1:])]


@pytest.mark.parametrize("count", [1, 2, 3, 5, 8, 33])
def test_wave_blocks(cases, oracle, gpu, monkeypatch, count):
    monkeypatch.setenv("TFG_BATCH_TUNE", "0")
    systems = [cases.hex_pressure(*SIDES[-1 - k % len(SIDES)], rho_out=10.0) for k in range(count)]
    print(f"batch waves {count} systems", flush=True)
    niter, xs = _solve(gpu, systems, 3, 1e-30)
    for s, x, it in zip(systems, xs, niter):
        if s.n < 256:
            continue  # may be solved, or stalled at rounding, by then
        ref = np.zeros(s.n)
        A = oracle.Matrix(s.row, s.col, s.dia, s.val.copy())
        oracle.solve("cg", "jacobi", A, ref, s.b.copy(), 3, 1e-30, criterion="relres")
        assert it == 3 and np.linalg.norm(x - ref) <= 1e-12 * np.linalg.norm(ref)
    for precision in (gpu.FP64, gpu.FP32_IR):
        niter, xs = _solve(gpu, systems, 5000, 1e-8, precision=precision)
        for s, x in zip(systems, xs):
            assert np.linalg.norm(s.b - s.scipy() @ x) <= 1.01e-8 * np.linalg.norm(s.b)
