"""The FP32 update of a batch by wavefront (2048 active blocks and more) and by
workgroup (fewer): each system's x has the same bits either
way, at one row, around 64 rows (a row per lane), 256 (a block) and more, in
counts around the line and with wavefronts of a workgroup left without a block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIDES = [(1, 1, 3), (3, 3, 7), (4, 4, 4), (13, 5, 1), (17, 5, 3), (16, 4, 4), (257, 1, 1), (23, 11, 5)]


def _solve(gpu, systems, prec):
    off = np.cumsum([0] + [s.n for s in systems])
    cat = lambda name: np.ascontiguousarray(np.concatenate([getattr(s, name) for s in systems]))
    bt = gpu.Batch([(s.row, s.col, s.dia) for s in systems])
    x = np.zeros(off[-1])
    with pytest.raises(gpu.TFlowsGpuError, match="breakdown"):  # the three rows are solved in three steps
        bt.solve("cg", prec, cat("val"), x, cat("b"), 400, 1e-8,
                 options=gpu.Options(criterion=gpu.CRIT_RELRES, precision=gpu.FP32_IR))
    blocks = bt.info()["blocks"]
    bt.close()
    return [x[a:b] for a, b in zip(off, off[1:])], blocks


@pytest.mark.parametrize("count,prec", [(1262, "jacobi"), (1263, "none"), (1264, "jacobi"), (1500, "none")])
def test_same_bits(cases, gpu, monkeypatch, count, prec):
    monkeypatch.setenv("TFG_BATCH_TUNE", "0")
    one = [cases.hex_pressure(*d, rho_out=10.0, seed=3 + k) for k, d in enumerate(SIDES)]
    systems = [one[k % len(one)] for k in range(count)]
    print(f"batch form {count} systems {prec}", flush=True)
    xs, blocks = _solve(gpu, systems, prec)
    assert (blocks >= 2048) == (count >= 1263), blocks
    want, few = _solve(gpu, one, prec)
    assert few < 2048
    for k in range(count):
        assert xs[k].tobytes() == want[k % len(one)].tobytes()
