"""The per-cell face walks of the device assembly (one workgroup per 256
cells, rows staged in LDS) where they can go wrong: block remainders, boundary
faces before, between and after the domain faces, cells without faces, rows
too long for the stage or for byte-sized places, entries no face sets.  Bit for
bit against the oracle's serial loops."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _graph(cases, n, edges, extra=(), seed=3):
    """Faces of a graph of n cells: one face per edge in a random order; the
    pairs `extra` are matrix entries that no face sets."""
    rng = np.random.default_rng(seed)
    nbrs = [set() for _ in range(n)]
    for a, b in list(edges) + list(extra):
        nbrs[a].add(b)
        nbrs[b].add(a)
    row, col, at = [1], [], {}
    for i in range(n):
        for c in [i] + sorted(nbrs[i]):
            at[i, c] = len(col) + 1
            col.append(c + 1)
        row.append(len(col) + 1)
    edges = [edges[k] for k in rng.permutation(len(edges))]
    nf = len(edges)
    z = np.zeros(nf, dtype=np.int32)
    return cases.Faces(
        row=np.array(row, np.int32), col=np.array(col, np.int32), dia=np.array(row[:-1], np.int32),
        c1=np.array([a + 1 for a, _ in edges], np.int32), c2=np.array([b + 1 for _, b in edges], np.int32),
        pos=np.array([p for a, b in edges for p in (at[a, b], at[b, a])], np.int32), diag_bc=z,
        b_region=z, fc=rng.uniform(0.5, 2.0, nf), fw=rng.uniform(0.3, 0.7, nf),
        vm=1e-3 * rng.uniform(0.5, 2.0, n), vflux=rng.uniform(-1.0, 1.0, nf), region=z)


def _case(cases, which):
    if which.startswith("line"):
        return cases.hex_faces(1, 1, int(which[4:]), ambient=True)
    return {
        "box3x5x17": lambda: cases.hex_faces(3, 5, 17, shuffle=False),
        "box9x8x7_ambient": lambda: cases.hex_faces(9, 8, 7, ambient=True),
        "box16x16x4_shuffled": lambda: cases.hex_faces(16, 16, 4),
        # a row of 400 entries: places above 255
        "star400": lambda: _graph(cases, 400, [(0, k) for k in range(1, 400)]),
        # 64 rows of 64 entries: one block's rows exceed the stage
        "complete64": lambda: _graph(cases, 64, [(a, b) for a in range(64) for b in range(a)]),
        # entries that no face sets, staged and not; cells without faces
        "unset": lambda: _graph(cases, 300, [(k, k + 1) for k in range(0, 200)], [(k, k + 2) for k in range(298)]),
        "unset_dense": lambda: _graph(cases, 80, [(k, k + 1) for k in range(0, 60)],
                                      [(a, b) for a in range(80) for b in range(a - 1)]),
    }[which]()


@pytest.mark.parametrize("which", ["line255", "line256", "line257", "box3x5x17", "box9x8x7_ambient",
                                   "box16x16x4_shuffled", "star400", "complete64", "unset", "unset_dense"])
def test_face_walks_bitexact(cases, oracle, gpu, which):
    f = _case(cases, which)
    print(f"face walk {which} n={f.n} faces={f.n_faces}", flush=True)
    nat = gpu.Native(f.row, f.col, f.dia)
    faces = gpu.Faces(nat, f.c1, f.c2, f.pos, f.diag_bc, f.b_region)
    d = {k: gpu.DeviceArray(getattr(f, k)) for k in ("fc", "fw", "vm", "vflux")}
    dpp = gpu.DeviceArray(f.pp) if f.pp is not None else None
    nan = lambda n: gpu.DeviceArray(np.full(n, np.nan))  # noqa: E731
    dval, db, dvm = nan(len(f.col)), nan(f.n), nan(f.n)
    faces.assemble(d["fc"], d["fw"], d["vm"], d["vflux"], dval, db, singular=True, dpp=dpp, n_bnd=f.n_bnd)
    val, b = oracle.pressure_assemble(f, singular=True)
    assert np.array_equal(dval.download(), val) and np.array_equal(db.download(), b)
    mf = cases.momentum_fields(f)
    for adv in ("minmod", "central"):
        dval, db = nan(len(f.col)), nan(f.n)
        faces.momentum(gpu.Momentum(mf, component=3, adv=adv), dval, db, dvm)
        ref = oracle.momentum_assemble(f, mf, component=3, adv=adv)
        for got, want in zip((dval, db, dvm), ref):
            assert np.array_equal(got.download(), want)
