"""The one-launch CG of small systems: that it runs where it should, that a
solve cut into many launches goes on where it stopped, that the tags of its
hand-overs start again, and that a solve whose launch gives up (its first wait
ended from the host by a bound of no reads; every kernel ends normally) is
solved again.  Each time the iterations, the residual and x have the bits of the
three-kernel form, from a non-zero x, on host and device operands."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one workgroup: an odd and an even number of rows; several: 8, 24, 25 and 128 blocks
TINY = [(5, 17, 3), (16, 16, 4)]
SMALL = [(683, 3, 1), (32, 24, 8), (29, 13, 17), (32, 32, 32)]
MODES = [("relres", None, "jacobi"), ("nrms", 1.0, "none"), ("nrms", None, "jacobi")]


def _solver(cases, gpu, dims, crit, norm, prec):
    s = cases.hex_pressure(*dims, rho_out=10.0)
    x = np.random.default_rng(5).uniform(-1, 1, s.n)
    nat = gpu.Native(s.row, s.col, s.dia)
    c = gpu.CRIT_RELRES if crit == "relres" else gpu.CRIT_NRMS
    dv, db = gpu.DeviceArray(s.val), gpu.DeviceArray(s.b)

    def solve(path, device=False, miter=60, tol=1e-7):
        opt = gpu.Options(criterion=c, path=path)
        if device:
            dx = gpu.DeviceArray(x)
            res = nat.solve_native_device("cg", prec, dv, dx, db, miter, tol, norm=norm, options=opt)
            return res, dx.download().tobytes()
        y = x.copy()
        return nat.solve_native("cg", prec, s.val, y, s.b, miter, tol, norm=norm, options=opt), y.tobytes()
    return nat, solve


@pytest.mark.parametrize("dims,workgroups", [
    ((1, 1, 3), -1),           # fewer than 64 entries: no row patterns
    ((16, 16, 8), 1), ((683, 3, 1), None), ((19, 11, 11), None), ((40, 40, 40), None),
    ((241, 17, 16), 0)])       # 257 row blocks
def test_form_taken(cases, gpu, dims, workgroups):
    nat, solve = _solver(cases, gpu, dims, *MODES[0])
    assert nat.small_info()["workgroups"] == -1
    solve(gpu.PATH_KERNELS)
    solve(gpu.PATH_GRAPH)
    assert nat.small_info() == dict(workgroups=-1, launches=0, solves=0, busy=0, given_up=0)
    assert solve(gpu.PATH_AUTO) == solve(gpu.PATH_KERNELS)
    i = nat.small_info()
    took = int(workgroups is None or workgroups > 0)
    assert (i["launches"], i["solves"], i["busy"], i["given_up"]) == (took, took, 0, 0)
    assert i["workgroups"] == workgroups if workgroups is not None else 2 <= i["workgroups"] <= 64


@pytest.mark.parametrize("dims", TINY + SMALL)
@pytest.mark.parametrize("mode", MODES, ids=str)
@pytest.mark.parametrize("length", [1, 2, 7])
def test_many_launches(cases, gpu, dims, mode, length):
    print(f"small launches {dims} {mode} of {length}", flush=True)
    nat, solve = _solver(cases, gpu, dims, *mode)
    want = solve(gpu.PATH_KERNELS)
    nat.small_limits(iterations=length)
    for device in (False, True):
        assert solve(gpu.PATH_AUTO, device) == want
    i = nat.small_info()
    assert i["solves"] == 2 and i["given_up"] == 0
    assert i["launches"] == 2 * -(-want[0][0] // length)


@pytest.mark.parametrize("dims", SMALL[:3])
@pytest.mark.parametrize("before", [0, 5, 64])
def test_tags_start_again(cases, gpu, dims, before):
    print(f"small tags {dims} {before} before the end", flush=True)
    nat, solve = _solver(cases, gpu, dims, *MODES[0])
    want = solve(gpu.PATH_KERNELS)
    assert solve(gpu.PATH_AUTO) == want          # the slots hold this solve's tags
    nat.small_limits(iterations=7, next_tag=0xf0000000 - before)
    for _ in range(3):
        assert solve(gpu.PATH_AUTO) == want
    i = nat.small_info()
    assert i["solves"] == 4 and i["given_up"] == 0
    nat.small_limits(next_tag=1 << 20)           # below it again
    with pytest.raises(gpu.TFlowsGpuError):
        nat.small_limits(next_tag=1 << 10)
    with pytest.raises(gpu.TFlowsGpuError):
        nat.small_limits(next_tag=0xf0000001)


@pytest.mark.parametrize("dims", SMALL)
@pytest.mark.parametrize("mode", MODES, ids=str)
@pytest.mark.parametrize("device,good", [(False, 0), (True, 0), (False, 3), (True, 2)])
def test_given_up(cases, gpu, dims, mode, device, good):
    """At the first launch, and after some launches of seven iterations."""
    print(f"small given up {dims} {mode} device={device} after {good}", flush=True)
    nat, solve = _solver(cases, gpu, dims, *mode)
    want = solve(gpu.PATH_KERNELS)
    assert want[0][0] > 7 * good
    nat.small_limits(iterations=7, launches=good)
    assert solve(gpu.PATH_AUTO, device) == want
    i = nat.small_info()
    assert (i["launches"], i["solves"], i["given_up"]) == (good + 1, 0, 1)


def test_tried_again(cases, gpu):
    """After a launch gave up, 16 solves go another way, 32 when the next one
    gives up too, then the one launch is back, and a later pause starts at 16."""
    nat, solve = _solver(cases, gpu, SMALL[0], *MODES[0])
    want = solve(gpu.PATH_KERNELS)

    def run(n):
        for _ in range(n):
            assert solve(gpu.PATH_AUTO) == want
        i = nat.small_info()
        return i["solves"], i["given_up"]

    nat.small_limits(launches=0)
    assert run(1) == (0, 1)
    assert run(16) == (0, 1) and run(1) == (0, 2)
    nat.small_limits()
    assert run(32) == (0, 2) and run(1) == (1, 2) and run(3) == (4, 2)
    nat.small_limits(launches=0)
    assert run(1) == (4, 3)
    nat.small_limits()
    assert run(16) == (4, 3) and run(1) == (5, 3)


def test_two_at_once(cases, gpu):
    """Each solve runs in the one launch or finds the device's XCD taken; none
    gives up, and the bits are the same."""
    made = [_solver(cases, gpu, SMALL[3], *MODES[0]) for _ in range(2)]
    want = made[0][1](gpu.PATH_KERNELS)
    got = [[], []]

    def work(k):
        for _ in range(8):
            got[k].append(made[k][1](gpu.PATH_AUTO))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert got[0] == got[1] == [want] * 8
    infos = [nat.small_info() for nat, _ in made]
    assert all(i["solves"] + i["busy"] == 8 and i["given_up"] == 0 for i in infos)
    assert sum(i["solves"] for i in infos) >= 1


def test_one_workgroup_never_waits(cases, gpu):
    nat, solve = _solver(cases, gpu, TINY[1], *MODES[0])
    nat.small_limits(launches=0)
    assert solve(gpu.PATH_AUTO) == solve(gpu.PATH_KERNELS)
    assert nat.small_info()["solves"] == 1


def test_limits_validation(gpu, cases):
    nat, _ = _solver(cases, gpu, TINY[0], *MODES[0])
    for n in (0, (1 << 14) + 1):
        with pytest.raises(gpu.TFlowsGpuError) as e:
            nat.small_limits(iterations=n)
        assert e.value.code == gpu.TFG_EINVAL
