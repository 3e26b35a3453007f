"""One-launch CG of small systems at the edges of its thread groups, row blocks
and slots: bit for bit the three-kernel form (the same sums in the same trees),
and x within a few roundings (1e-12) of the oracle after three iterations."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# rows: one, an odd few, around one block, one workgroup's 2048, blocks 9, 24,
# 25 (a product workgroup with two), 127 to 129, 250, 256, 257 (not taken)
SIZES = [(1, 1, 1), (1, 1, 3), (5, 17, 3), (16, 16, 1), (1, 257, 1), (16, 16, 4), (25, 41, 1),
         (89, 23, 1), (16, 16, 8), (683, 3, 1), (19, 11, 11), (32, 24, 8), (29, 13, 17),
         (127, 16, 16), (32, 32, 32), (47, 37, 19), (40, 40, 40), (64, 32, 32), (241, 17, 16)]


@pytest.mark.parametrize("dims", SIZES)
@pytest.mark.parametrize("crit,norm,prec", [("relres", None, "jacobi"), ("relres", None, "none"),
                                            ("nrms", 1.0, "jacobi"), ("nrms", None, "jacobi"),
                                            ("nrms", None, "none")])
def test_same_bits(cases, oracle, gpu, dims, crit, norm, prec):
    s = cases.hex_pressure(*dims, rho_out=10.0)
    print(f"small {dims} n={s.n} {crit} norm={norm} {prec}", flush=True)
    x = np.random.default_rng(5).uniform(-1, 1, s.n)
    nat = gpu.Native(s.row, s.col, s.dia)
    c = gpu.CRIT_RELRES if crit == "relres" else gpu.CRIT_NRMS
    for miter, tol in ((3, 1e-30), (400, 1e-7)):
        got = []
        for path in (gpu.PATH_AUTO, gpu.PATH_KERNELS):
            y = x.copy()
            it, fin = nat.solve_native("cg", prec, s.val, y, s.b, miter, tol, norm=norm,
                                       options=gpu.Options(criterion=c, path=path))
            got.append((it, fin, y))
        assert got[0][:2] == got[1][:2] and got[0][2].tobytes() == got[1][2].tobytes()
        if miter == 3 and s.n > 512:  # smaller ones may be solved by then
            ref = x.copy()
            A = oracle.Matrix(s.row, s.col, s.dia, s.val.copy())
            oracle.solve("cg", prec, A, ref, s.b.copy(), 3, 1e-30, norm=norm, criterion=crit)
            assert np.linalg.norm(got[0][2] - ref) <= 1e-12 * np.linalg.norm(ref)


def test_two_threads(cases, gpu):
    """Two solves at once: one of them finds the XCD taken, the bits are the same."""
    s = cases.hex_pressure(32, 32, 32, rho_out=10.0)
    ref = np.zeros(s.n)
    want = gpu.Native(s.row, s.col, s.dia).solve_native("cg", "jacobi", s.val, ref, s.b, 200, 1e-7)
    out = [[], []]

    def work(k):
        nat = gpu.Native(s.row, s.col, s.dia)
        for _ in range(5):
            x = np.zeros(s.n)
            out[k].append((nat.solve_native("cg", "jacobi", s.val, x, s.b, 200, 1e-7), x))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for got, x in out[0] + out[1]:
        assert got == want and x.tobytes() == ref.tobytes()
    assert len(out[0]) == len(out[1]) == 5
