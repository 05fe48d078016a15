"""Which steps a plan takes (host memory only: no device is needed)."""
import ctypes
import os
import subprocess
import sys
import time

import numpy as np
import pytest

from strawberryfields_amd import _lib, circuits, runtime

OP, DIAG, VECTOR, MATRIX = range(4)


class Plan:
    """A plan's steps (kind, operations) and the kinds of its forward-only steps."""

    def __init__(self, ops, n, D, mixed=False, dtype=_lib.C64, fuse=None):
        lib = _lib.load()
        arr = (_lib.OpDesc * len(ops))()
        for i, (name, modes) in enumerate(ops):
            arr[i].kind = _lib.OP_KINDS[name]
            arr[i].mode0 = modes[0]
            arr[i].mode1 = modes[1] if len(modes) > 1 else -1
        K = runtime.default_fuse(n, D) | _lib.FUSE_PAYING if fuse is None else fuse
        h = ctypes.c_void_p()
        assert lib.sfamd_prog_create(arr, len(ops), n, D, int(mixed), dtype, K | _lib.FUSE_MIXED, ctypes.byref(h)) == 0
        self.steps, self.run = [], []
        buf = (ctypes.c_int32 * len(ops))()
        while (k := lib.sfamd_prog_step_kind(h, 0, len(self.steps))) >= 0:
            m = lib.sfamd_prog_step_ops(h, len(self.steps), buf, len(ops))
            self.steps.append((k, buf[:m]))
        while (k := lib.sfamd_prog_step_kind(h, 1, len(self.run))) >= 0:
            self.run.append(k)
        lib.sfamd_prog_destroy(h)

    @property
    def kinds(self):
        return [k for k, _ in self.steps]


def _layered(n, layers=1, loss=False):
    return [o[:2] for o in circuits.layered(n, layers, np.random.default_rng(0), loss=loss)]


# --------------------------------------------------- stages that hold too few gates
@pytest.mark.parametrize("dtype", [_lib.C64, _lib.C128])
@pytest.mark.parametrize(
    "n,D,mixed,ops",
    [(6, 16, False, [("BS", (0, 1))]), (8, 8, False, [("S2", (0, 1))]), (4, 15, False, [("CK", (0, 3))]),
     (20, 2, False, [("MZ", (0, 1))]), (3, 9, True, [("D", (0,))]), (3, 16, True, [("S", (1,))]),
     (4, 6, True, [("D", (0,)), ("LOSS", (0,)), ("D", (1,)), ("LOSS", (1,))]), (7, 3, True, [("D", (0,)), ("S", (1,))])],
)
def test_gates_that_share_no_stage_run_alone(n, D, mixed, ops, dtype):
    """A stage of one or two gates costs more than the gates' own passes, forward
    only and with the adjoint; an explicit tile still asks for it."""
    plan = Plan(ops, n, D, mixed, dtype)
    if dtype == _lib.C64 or D not in (8, 15):
        assert set(plan.run) == {OP}
    if dtype == _lib.C64:
        assert set(plan.kinds) == {OP}
    if not mixed or D <= 12:
        assert MATRIX in Plan(ops, n, D, mixed, dtype, fuse=3).run


@pytest.mark.parametrize("D", [4, 9, 12, 17])
@pytest.mark.parametrize("kind", ["BS", "MZ", "S2", "CK"])
def test_pairs_followed_by_a_mode_run_in_one_pass(D, kind):
    """A two-mode gate on the first modes of a complex64 density matrix takes its own
    one-pass kernel, also by default."""
    for modes in [(0, 1), (1, 0)]:
        assert Plan([(kind, modes)], 3, D, True).run == [OP]


@pytest.mark.parametrize("dtype", [_lib.C64, _lib.C128])
@pytest.mark.parametrize("n,D,mixed", [(3, 8, False), (6, 8, False), (8, 5, False), (12, 2, False), (12, 3, False), (7, 16, False),
                                       (2, 8, True), (3, 9, True), (3, 12, True), (4, 6, True), (6, 3, True), (8, 2, True)])
def test_layers_still_run_in_stages(n, D, mixed, dtype):
    plan = Plan(_layered(n, 1, mixed), n, D, mixed, dtype)
    assert plan.run.count(MATRIX) >= len([k for k in plan.run if k == OP]) - n  # (a layer has n losses)
    assert MATRIX in plan.run


@pytest.mark.parametrize(
    "n,D,dtype,forward,adjoint",
    [(3, 18, _lib.C64, False, False), (3, 20, _lib.C64, False, False), (3, 20, _lib.C128, True, False), (2, 20, _lib.C64, True, False),
     (10, 2, _lib.C128, False, False), (8, 2, _lib.C128, True, True), (10, 2, _lib.C64, True, True), (7, 3, _lib.C128, True, False),
     (6, 3, _lib.C128, True, True), (5, 5, _lib.C128, True, False), (5, 5, _lib.C64, True, True), (4, 5, _lib.C128, True, True),
     (4, 9, _lib.C64, False, False), (4, 10, _lib.C128, False, False), (3, 10, _lib.C128, True, True), (4, 8, _lib.C128, True, True)],
)
def test_large_density_matrices_leave_stages_where_these_lose(n, D, dtype, forward, adjoint):
    """States past the caches where a stage's operands are mostly padding, and
    complex64 forwards above cutoff 16, run gate by gate."""
    plan = Plan(_layered(n, 1, True), n, D, True, dtype)
    assert (MATRIX in plan.run, MATRIX in plan.kinds) == (forward, adjoint)


@pytest.mark.parametrize(
    "n,D,dtype,forward,adjoint,steps",
    [(3, 9, _lib.C64, VECTOR, VECTOR, 2), (5, 9, _lib.C64, VECTOR, VECTOR, 8), (6, 9, _lib.C64, MATRIX, VECTOR, 15),
     (7, 9, _lib.C64, VECTOR, OP, 59), (4, 9, _lib.C128, MATRIX, VECTOR, 7), (4, 10, _lib.C64, MATRIX, VECTOR, 5),
     (5, 10, _lib.C64, MATRIX, VECTOR, 8), (3, 10, _lib.C64, MATRIX, VECTOR, 5), (4, 10, _lib.C128, MATRIX, VECTOR, 12),
     (9, 5, _lib.C128, MATRIX, VECTOR, 32), (8, 5, _lib.C128, MATRIX, MATRIX, 15), (8, 6, _lib.C128, MATRIX, VECTOR, 25)],
)
def test_stages_of_cutoffs_that_half_fill_an_operand(n, D, dtype, forward, adjoint, steps):
    plan = Plan(_layered(n), n, D, False, dtype)
    assert max(plan.run) == forward and len(plan.kinds) == steps
    assert set(plan.kinds) == {adjoint} if adjoint != OP else max(plan.kinds) <= DIAG


@pytest.mark.parametrize("n,D", [(2, 8), (3, 4), (5, 3), (6, 5), (8, 8), (4, 13), (3, 17), (4, 20), (3, 24), (1, 8)])
@pytest.mark.parametrize("mixed", [False, True])
def test_autotuner_candidates_are_tiles_that_the_planner_has(n, D, mixed):
    """And the default tile is one of them, or has the plan of one (a density
    matrix's stage of two modes has the tile of three axes)."""
    cands = runtime.Autotuner.candidates(n, D, mixed)
    want = runtime.default_fuse(n, D)
    assert (max(want, 3) if mixed and want else want) in cands
    for K in cands[1:]:
        plan = Plan([("BS", (0, 1))] * 8 + [("S2", (1, 0))], n, D, mixed, _lib.C64, fuse=K)
        big = D**n * 8 > 20e6 or (mixed and D > 16)
        assert big or max(plan.run) == (VECTOR if K == 2 else MATRIX)


@pytest.mark.parametrize("seed", range(12))
def test_default_plans_keep_every_gate_and_mode_order(seed):
    """Also where some gates of a run leave their stage."""
    rng = np.random.default_rng(seed)
    n, D = [(2, 8), (3, 9), (4, 4), (3, 16), (6, 3), (8, 2)][seed % 6]
    mixed = bool(seed // 6)
    ops = []
    for _ in range(60):
        kind = ["D", "S", "R", "K", "BS", "S2", "CK", "MZ", "LOSS" if mixed else "D"][rng.integers(9)]
        a, b = (int(v) for v in rng.choice(n, 2, replace=False))
        ops.append((kind, (a, b) if kind in ("BS", "S2", "CK", "MZ") else (a,)))
    for dtype in (_lib.C64, _lib.C128):
        flat = [i for _, st in Plan(ops, n, D, mixed, dtype).steps for i in st]
        assert sorted(flat) == list(range(len(ops)))
        for m in range(n):
            order = [i for i in flat if m in ops[i][1]]
            assert order == sorted(order)


def test_plans_of_many_modes_are_made_in_milliseconds():
    """A density matrix of 10 modes at cutoff 2 (252 sets of 5 modes): the search for its
    stages stays far below the 110 ms that one step of lookahead over all pairs of sets
    takes, about 2 ms here."""
    ops = _layered(10, 2, True)
    times = []
    for _ in range(3):
        t = time.perf_counter()
        plan = Plan(ops, 10, 2, True)
        times.append(time.perf_counter() - t)
    assert MATRIX in plan.kinds and min(times) < 0.04


def test_plans_that_do_not_fit_in_host_memory_are_refused():
    """An error code, not an exception through the C interface."""
    code = """
import ctypes, resource, sys
sys.path.insert(0, %r)
from strawberryfields_amd import _lib
lib = _lib.load()
n = 100000
arr = (_lib.OpDesc * n)()
for i in range(n):
    arr[i].kind, arr[i].mode0, arr[i].mode1 = _lib.OP_KINDS["D"], i %% 3, -1
h = ctypes.c_void_p()
assert lib.sfamd_prog_create(arr, n, 3, 24, 0, 0, 0, ctypes.byref(h)) == 0
lib.sfamd_prog_destroy(h)
h = ctypes.c_void_p()
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + (16 << 20), -1))
print(lib.sfamd_prog_create(arr, n, 3, 24, 0, 0, 0, ctypes.byref(h)), h.value)
""" % os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    assert res.stdout.split() == ["-1", "None"]
