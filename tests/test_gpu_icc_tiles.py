"""The tiled DIC sweeps at the edges of their tiles (8 x 8 x 16 cells) and of
the level loop's lanes: full tiles, one cell more and less along each axis,
single planes and lines.  z = M^-1 r is the oracle's to the bit, as every row
does the same operations in the same order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(8, 8, 16), (9, 8, 16), (8, 9, 16), (8, 8, 17), (7, 7, 15),
                                  (16, 16, 32), (17, 15, 33), (2, 2, 2), (3, 5, 1), (1, 1, 40),
                                  (1, 9, 1), (33, 1, 1), (8, 2, 31), (5, 3, 16), (25, 23, 50)])
def test_tile_edges(cases, oracle, gpu, dims):
    s = cases.hex_pressure(*dims, rho_out=1000.0)
    print(f"icc tiles {dims}", flush=True)
    r = np.random.default_rng(7).standard_normal(s.n)
    A = oracle.Matrix(s.row, s.col, s.dia, s.val)
    nat = gpu.Native(s.row, s.col, s.dia)
    assert nat.info()["icc_tiles"] > 0  # a line counts along z, whichever axis it is given on
    dv, dr, dz = gpu.DeviceArray(s.val), gpu.DeviceArray(r), gpu.DeviceArray(np.zeros(s.n))
    d, dinv = oracle.prec_form(A, "icc")
    nat.prec_apply("icc", dv, dr, dz)
    assert np.array_equal(dz.download(), oracle.prec_solve(A, d, dinv, r, "icc"))
