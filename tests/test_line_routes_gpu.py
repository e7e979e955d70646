"""1D solves by one workgroup and by the grid path, and the widths of the batch
workgroup, at the sizes where the route or the width changes.  Add, multiply, divide
and square root only: every comparison is bit for bit."""

import ctypes
import math

import numpy as np
import pytest

import oracle_lib as O
from vanguard_amd import _lib
from vanguard_amd import solvers as S

pytestmark = pytest.mark.gpu

EULER = [1.4, 0, 25, 0, 0.25, 250]


def _euler(n):
    rng = np.random.default_rng(n)
    w = rng.uniform(-0.4, 0.4, (n, 6))
    w[:, 0], w[:, 4], w[:, 5] = rng.uniform(0.3, 1.5, n), rng.uniform(0.3, 1.5, n), 1.0
    return w


def _mhd(n, seed=0):
    rng = np.random.default_rng(n + 100000 * seed)
    w = rng.uniform(-0.4, 0.4, (n, 9))
    w[:, 0], w[:, 4] = rng.uniform(0.5, 1.5, n), rng.uniform(0.5, 1.5, n)
    return w


# 252 / 253: one tile of 256 threads or of 512; 508 / 509 (SLIC) and 1020 / 1021
# (FORCE): the last size of a long run in one workgroup and the first on the grid path;
# 60 / 124: MHD tiles.  Up to 12 steps (SLIC) the workgroup keeps an Euler line of two
# tiles; 11 steps of 2100 cells are launched one by one, 41 steps replayed.
@pytest.mark.parametrize("n", [60, 124, 125, 252, 253, 508, 509, 569, 1020, 1021, 2100])
@pytest.mark.parametrize("order", [2, 1])
@pytest.mark.parametrize("steps", [11, 41])
def test_1d_routes_match_oracle(vg_ctx, n, order, steps):
    kw = dict(order=order, dim=1, dx=1.0 / n, cfl=0.7, tfinal=math.inf, max_steps=steps, bias=0.0, limiter=0)
    for bc in (S.TRANSMISSIVE, S.PERIODIC):
        w = _euler(n)
        r = S.euler_solve(w, 1, 1.0 / n, 0.7, math.inf, order=order, limiter=0, max_steps=steps, bc=bc)
        ref, dts = O.euler_solve(w, params=EULER, bc=bc, **kw)
        O.assert_bitwise(r.dt, dts, f"euler n {n} dt")
        O.assert_bitwise(r.cells, ref, f"euler n {n} state")
        w = _mhd(n)
        r = S.mhd_solve(w, 1, 1.0 / n, 0.7, math.inf, order=order, limiter=0, max_steps=steps, bc=bc,
                        params=S.MHDMaterialParameters(5.0 / 3.0, 0.0, 0.7, 0.4))
        ref, dts = O.mhd_solve(w, gamma=5.0 / 3.0, ch=0.7, cp=0.4, bc=bc, **kw)
        O.assert_bitwise(r.dt, dts, f"mhd n {n} dt")
        O.assert_bitwise(r.cells, ref, f"mhd n {n} state")


@pytest.mark.parametrize("n", [300, 700, 2100])
def test_final_time_and_caps_on_both_routes(vg_ctx, n):
    w = _euler(n)
    kw = dict(order=2, dim=1, dx=1.0 / n, cfl=0.8, bias=0.0, limiter=1, params=EULER)
    ref, dts = O.euler_solve(w, tfinal=0.05, max_steps=0, **kw)
    r = S.euler_solve(w, 1, 1.0 / n, 0.8, 0.05, limiter=1)
    assert r.stats.t == 0.05 and r.stats.steps == len(dts)
    O.assert_bitwise(r.dt, dts, "dt to the final time")
    O.assert_bitwise(r.cells, ref, "state at the final time")
    for cap in (1, 8, 9, 23, 33, 40, 47):
        r = S.euler_solve(w, 1, 1.0 / n, 0.8, 0.05, limiter=1, max_steps=cap)
        assert r.stats.steps == min(cap, len(dts))
        O.assert_bitwise(r.dt, dts[:cap], "capped dt prefix")
    assert S.euler_solve(w, 1, 1.0 / n, 0.8, 0.0, limiter=1).stats.steps == 0


@pytest.mark.parametrize("n", [300, 700])
def test_a_step_that_cannot_advance_is_refused_on_both_routes(vg_ctx, n):
    for solve, w, p in ((S.euler_solve, _euler(n), None), (S.mhd_solve, _mhd(n), S.MHDMaterialParameters(1.4))):
        w[n // 2, 1] = math.inf          # an infinite wave speed: dt = 0
        r = solve(w, 1, 1.0 / n, 0.8, 1.0, params=p, raise_on_error=False)
        assert r.status == _lib.VG_ERR_NONFINITE and r.stats.steps == 0


# 3 instances fill a wide workgroup each, 300 a middle one, 700 the narrow one.
@pytest.mark.parametrize("n_inst", [3, 300, 700])
@pytest.mark.parametrize("mode", [S.EXACT, S.FAST])
def test_batch_widths_give_the_single_solves_bits(vg_ctx, n_inst, mode):
    sizes = np.array([600, 300, 125] + [17 + (7 * q) % 120 for q in range(n_inst - 3)])
    off = np.concatenate([[0], np.cumsum(sizes)])
    w = np.concatenate([_mhd(int(n), q) for q, n in enumerate(sizes)])
    r = S.mhd_solve_batch(w, off, 1.0 / sizes, np.full(n_inst, 5.0 / 3.0), 10.0, 0.6, max_steps=7, limiter=1, mode=mode)
    for q in (0, 1, 2, n_inst - 1):
        one = S.mhd_solve(w[off[q]:off[q + 1]], 1, 1.0 / sizes[q], 0.6, 10.0, limiter=1, max_steps=7, mode=mode,
                          params=S.MHDMaterialParameters(5.0 / 3.0))
        O.assert_bitwise(r.cells[off[q]:off[q + 1]], one.cells, f"instance {q}")


def _launches(ctx, w, t_final, max_steps, **kw):
    """batch_solve launches of one Euler line: 1 where the whole solve is one workgroup's."""
    ctx.reset_timing()
    r = S.euler_solve(w, 1, 1.0 / len(w), 0.8, t_final, max_steps=max_steps, limiter=1, ctx=ctx, **kw)
    return r, ctx.kernel_time("batch_solve")[0]


def test_few_steps_of_a_longer_line_stay_in_one_workgroup():
    """The grid path costs some tens of microseconds more a call, so by step cap or by
    final time a short run of 509 to about 1500 cells is one launch; its result is the
    long run's prefix either way."""
    ctx = S.Context(0)
    try:
        ctx.set_timing(True)
        for n, order in ((509, 2), (1016, 2), (1021, 1), (1530, 1)):
            w = _euler(n)
            long, launches = _launches(ctx, w, math.inf, 60, order=order)
            assert launches == 0, (n, order)
            short, launches = _launches(ctx, w, math.inf, 7, order=order)
            assert launches == 1 and short.stats.steps == 7, (n, order)
            O.assert_bitwise(short.dt, long.dt[:7], "capped dt")
            # six steps of a fifth of a length and two whole ones
            ended, launches = _launches(ctx, w, 0.999 * float(np.sum(long.dt[:8])), 0, order=order)
            assert launches == 1 and ended.stats.steps == 8, (n, order)
            O.assert_bitwise(ended.dt[:7], long.dt[:7], "dt to a final time")
            # an infinite wave speed predicts no number of steps
            w[n // 2, 0] = 0.0
            assert _launches(ctx, w, 1.0, 60, order=order, raise_on_error=False)[1] == 0
    finally:
        ctx.close()


@pytest.mark.parametrize("n", [300, 5000])
def test_a_rejected_call_leaves_the_run_statistics_alone(vg_ctx, n):
    """An unknown mode: no step is taken, and of the caller's statistics only the step
    counts and the time (MHD) are set."""
    for nf, name in ((6, "vg_euler_solve_1d"), (9, "vg_mhd_solve_1d")):
        w, out = np.ones((n, nf)), np.empty((n, nf))
        st = _lib.RunStats(first_nonfinite=-1, nonfinite_cells=3, dt_min=0.25, dt_max=0.5, device_ms=1.5, wall_ms=2.5)
        p = S.EulerMaterialParameters(1.4) if nf == 6 else S.MHDMaterialParameters(1.4)
        sub = [] if nf == 6 else [0]
        rc = getattr(vg_ctx.lib, name)(vg_ctx.handle, _lib.as_dptr(w), _lib.as_dptr(out), n, 1.0 / n, 0.5, 1.0, 5, 0.0,
                                       0, 2, 0, *sub, ctypes.byref(p.c_struct()), 9, None, 0, ctypes.byref(st))
        assert rc == _lib.VG_ERR_ARG
        assert (st.first_nonfinite, st.nonfinite_cells) == (-1, 3), name
        assert (st.dt_min, st.dt_max, st.device_ms, st.wall_ms) == (0.25, 0.5, 1.5, 2.5), name
        assert st.steps == 0 and st.t == 0.0


def test_a_long_euler_line_that_cannot_advance_is_returned_as_it_is(vg_ctx):
    """Euler lines of over 32,768 cells report a step that cannot advance t by their
    statistics only: no steps, the initial state (finite and admissible here)."""
    w = np.tile([1e-300, 0.0, 0.0, 0.0, 1e300, 1.0], (40000, 1))
    r = S.euler_solve(w, 1, 1e-3, 0.8, 1.0)
    assert r.status == _lib.VG_OK and r.stats.steps == 0 and r.stats.t == 0.0
    O.assert_bitwise(r.cells, w, "state")
    r = S.euler_solve(w[:32768], 1, 1e-3, 0.8, 1.0, raise_on_error=False)
    assert r.status == _lib.VG_ERR_NONFINITE


# Up to 256 instances take the limiter by selects, more by branches.
@pytest.mark.parametrize("n_inst", [256, 257])
@pytest.mark.parametrize("limiter,bias", [(0, 0.0), (1, -0.35), (2, 1.0), (1, 1.5)])
def test_batches_on_both_sides_of_the_limiter_rule_match_oracle(vg_ctx, n_inst, limiter, bias):
    sizes = 20 + (13 * np.arange(n_inst)) % 110
    off = np.concatenate([[0], np.cumsum(sizes)])
    kw = dict(order=2, dim=1, cfl=0.6, tfinal=10.0, max_steps=7, bias=bias, limiter=limiter)
    we = np.concatenate([_euler(int(n)) for n in sizes])
    wm = np.concatenate([_mhd(int(n)) for n in sizes])
    e = S.euler_solve_batch(we, off, 1.0 / sizes, [S.EulerMaterialParameters(*EULER)] * n_inst, np.full(n_inst, 10.0),
                            0.6, max_steps=7, bias=bias, limiter=limiter)
    m = S.mhd_solve_batch(wm, off, 1.0 / sizes, np.full(n_inst, 5.0 / 3.0), 10.0, 0.6, max_steps=7, bias=bias,
                          limiter=limiter)
    for q in range(0, n_inst, 32):
        a, b = off[q], off[q + 1]
        ref, _ = O.euler_solve(we[a:b], dx=1.0 / sizes[q], params=EULER, **kw)
        O.assert_bitwise(e.cells[a:b], ref, f"euler instance {q}")
        ref, _ = O.mhd_solve(wm[a:b], dx=1.0 / sizes[q], gamma=5.0 / 3.0, **kw)
        O.assert_bitwise(m.cells[a:b], ref, f"mhd instance {q}")
