"""The product engines of matrices without a row structure (entries dealt four
at a time; x gathered entry by entry, or once per row block through its list
of different columns): last chunks of 1..4 entries, blocks of one to many
rows, rows around the eight terms added at once, blocks with more columns than
the window (a few: entry by entry in those; most: no window), rows longer than
the stage.  Bit for bit against the oracle, in FP64 and in the FP32 row-excess
form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(n, near, far_rows, far, seed, extra=0, width=400):
    """Rows of 1 + near random neighbours within +-width (above 128: more column
    offsets than the coded engine takes, so the handle makes the window), the rows `far_rows` also
    `far` anywhere; symmetric in structure and values; `extra` more entries in
    the last row."""
    rng = np.random.default_rng(seed)
    pairs = set()
    for i in range(n):
        for j in rng.integers(max(0, i - width), min(n, i + width + 1), near):
            pairs.add((min(i, int(j)), max(i, int(j))))
    for i in far_rows:
        for j in rng.integers(0, n, far):
            pairs.add((min(i, int(j)), max(i, int(j))))
    for j in range(extra):
        pairs.add((j, n - 1))
    nbrs = [[] for _ in range(n)]
    for i, j in pairs:
        if i != j:
            v = -rng.uniform(0.5, 2.0)
            nbrs[i].append((j, v))
            nbrs[j].append((i, v))
    row, col, val = [1], [], []
    for i in range(n):
        nbrs[i].sort()
        col += [i + 1] + [j + 1 for j, _ in nbrs[i]]
        val += [1e-3 - sum(v for _, v in nbrs[i])] + [v for _, v in nbrs[i]]
        row.append(len(col) + 1)
    return (np.array(row, np.int32), np.array(col, np.int32), np.array(row[:-1], np.int32),
            np.array(val))


CASES = {
    **{f"tail{k}": lambda k=k: _matrix(500 + k // 2, 3, [], 0, 1, extra=k % 2) for k in range(4)},
    "one_block": lambda: _matrix(67, 3, [], 0, 1, width=40),
    "short_rows": lambda: _matrix(1000, 1, [], 0, 2),
    "eight_terms": lambda: _matrix(900, 4, [], 0, 3),
    "window": lambda: _matrix(3000, 9, [], 0, 4),
    "entrywise": lambda: _matrix(3000, 9, [], 0, 4, width=40),
    "few_wide_blocks": lambda: _matrix(6000, 9, range(100, 170), 40, 5, width=150),
    "no_window": lambda: _matrix(4000, 2, range(4000), 8, 6),
    "long_row": lambda: _matrix(5000, 6, [2500], 4000, 7),
}


@pytest.mark.parametrize("which", list(CASES))
def test_products_without_row_structure(oracle, gpu, which):
    row, col, dia, val = CASES[which]()
    n = len(dia)
    print(f"window {which} n={n} nnz={len(col)}", flush=True)
    nat = gpu.Native(row, col, dia)
    nat.spmv_select(5)
    A = oracle.Matrix(row, col, dia, val)
    rng = np.random.default_rng(8)
    p, b = rng.standard_normal(n), rng.standard_normal(n)
    dv, dp, db, dq = (gpu.DeviceArray(a) for a in (val, p, b, np.zeros(n)))
    long_rows = np.diff(row) > 2040      # summed by a tree, not in CSR order
    ref = oracle.spmv(A, p)
    nat.spmv(dv, dp, dq)
    q = dq.download()
    assert np.array_equal(q[~long_rows], ref[~long_rows])
    assert np.allclose(q[long_rows], ref[long_rows], rtol=1e-12)
    nat.residual(dv, db, dp, dq)
    assert np.array_equal(dq.download()[~long_rows], oracle.residual(A, b, p)[~long_rows])
    fn = 1.0 / (val[dia - 1].sum() / n)
    x = rng.uniform(-1, 1, n).astype(np.float32)
    dx, dy = gpu.DeviceArray(x), gpu.DeviceArray(np.zeros(n, dtype=np.float32))
    nat.spmv_fp32(dv, fn, dx, dy)
    y = oracle.lap32_spmv(A, oracle.lap32_form(A, fn), x)
    assert np.array_equal(dy.download()[~long_rows], y[~long_rows])
