"""The per-cell walk of the Rhie-Chow fluxes where it can go wrong: block
remainders, boundary faces before, between and after the domain faces, faces
whose c1 is the larger cell, cells of many faces and of none, and a cell's
faces dealt to three threads, to two and to one (by the number of cells).  Bit for bit against the oracle's serial loop; every domain face is
written (NaN before), no boundary face is."""
import numpy as np
import pytest

from test_gpu_cell_faces import _case

pytestmark = pytest.mark.gpu

CASES = ["line255", "line256", "line257", "box3x5x17", "box9x8x7_ambient", "box16x16x4_shuffled", "star400",
         "complete64", "unset", (28, 28, 28), (34, 34, 33), (40, 40, 40), (40, 41, 41)]


@pytest.mark.parametrize("which", CASES, ids=str)
@pytest.mark.parametrize("choi,gu,vof", [(False, False, False), (True, True, True), (True, False, False),
                                         (False, True, True)])
def test_fluxes_bitexact(cases, oracle, gpu, which, choi, gu, vof):
    f = _case(cases, which) if isinstance(which, str) else cases.hex_faces(*which, shuffle=which[0] != 34)
    print(f"fluxes {which} n={f.n} faces={f.n_faces} {choi} {gu} {vof}", flush=True)
    rng = np.random.default_rng(9)
    cell = lambda: rng.uniform(-1.0, 1.0, f.n)  # noqa: E731
    face = lambda: rng.uniform(-1.0, 1.0, f.n_faces)  # noqa: E731
    at_face = {"f", "fc", "sx", "sy", "sz", "dx", "dy", "dz", "flux_o", "flux_oo", "face_fx", "face_fy", "face_fz"}
    rf = cases.RhieChowFields(**{k: face() if k in at_face else cell()
                                 for k in cases.RhieChowFields.__dataclass_fields__})
    kw = dict(choi=choi, dt=3e-3, w_o=2.0, w_oo=-0.5, gu=gu, vof=vof, sigma=0.07)
    base = np.where(f.c2 > 0, np.nan, face())
    nat = gpu.Native(f.row, f.col, f.dia)
    faces = gpu.Faces(nat, f.c1, f.c2, f.pos, f.diag_bc, f.b_region)
    dflux = gpu.DeviceArray(base)
    faces.rhie_chow(gpu.RhieChow(rf, **kw), dflux)
    got = dflux.download()
    assert np.isfinite(got).all() and np.array_equal(got, oracle.rhie_chow_fluxes(f, rf, base, **kw))
