"""The EXACT sweeps and source sub-cycles off the usual ranges, against the oracle: biases
outside [-1, 1] and slope differences beyond 2^600 (where the limiter takes IEEE
divisions), and distortions whose Gramian overflows."""

import numpy as np
import pytest

import oracle_lib as O
from test_hpr_gpu import mat_params, rel_l1
from vanguard_amd import solvers as S

pytestmark = pytest.mark.gpu

EULER = [1.4, 0, 25, 0.3, 0.25, 250]


def _state(nf, ny=23, nx=65):
    rng = np.random.default_rng(nf)
    w = rng.uniform(-0.3, 0.3, (ny, nx, nf))
    w[..., 0] = rng.uniform(0.5, 1.5, (ny, nx))
    w[..., 4] = rng.uniform(0.5, 1.5, (ny, nx))
    if nf == 17:
        w = rng.uniform(-0.03, 0.03, (ny, nx, nf))
        w[..., 0] += 1.0
        w[..., 1] += 1.0 / 1.4
        w[..., 2:11] += np.eye(3).ravel()
    return w, rng


def _ghosted(w, order):
    """Transmissive ghosts: g[-1] = c[0], g[-2] = c[1]."""
    return np.pad(w, ((order, order), (order, order), (0, 0)), mode="symmetric")


def _assert_alike(got, want, what):
    """The same bits, and NaN in the same places."""
    nan = np.isnan(want)
    assert (np.isnan(got) == nan).all(), what
    O.assert_bitwise(np.where(nan, 0.0, got), np.where(nan, 0.0, want), what)


def _sweeps(w, limiter, bias, dt):
    ny, nx, nf = w.shape
    for direction in (0, 1):
        kw = dict(order=2, dim=2, direction=direction, dx=1.0 / nx, ts=dt, bias=bias, limiter=limiter)
        if nf == 6:
            cls, p = S.SecondOrderSolver, S.EulerMaterialParameters(*EULER)
            ref = O.euler_sweep(w, params=EULER, **kw)
        else:
            cls, p = S.MHDSecondOrderSolver, S.MHDMaterialParameters(5.0 / 3.0, 0.0, 0.7, 0.4)
            ref = O.mhd_sweep(w, gamma=5.0 / 3.0, p_inf=0.0, ch=0.7, cp=0.4, **kw)
        cells = w.copy()
        fn = cls.computeXSLICTimeStep2D if direction == 0 else cls.computeYSLICTimeStep2D
        fn(cells, _ghosted(w, 2), 1.0 / nx, dt, bias, limiter, p)
        _assert_alike(cells, ref, f"{nf} fields, direction {direction}, limiter {limiter}, bias {bias}")


@pytest.mark.parametrize("limiter", [0, 1, 2])
@pytest.mark.parametrize("bias", [1.5, -2.0])
@pytest.mark.parametrize("nf", [6, 9])
def test_a_bias_outside_its_range_matches_oracle(vg_ctx, nf, bias, limiter):
    _sweeps(_state(nf)[0], limiter, bias, 2e-3)


@pytest.mark.parametrize("limiter", [0, 1, 2])
@pytest.mark.parametrize("nf", [6, 9])
def test_slope_differences_beyond_the_short_range_match_oracle(vg_ctx, nf, limiter):
    """One cell in nine holds a velocity (Euler) or a cleaning potential (MHD) of 2^590 to
    2^700; the time step keeps the products finite in most of the others."""
    w, rng = _state(nf)
    big = rng.choice([-1.0, 1.0], w.shape[:2]) * np.exp2(rng.uniform(590, 700, w.shape[:2]))
    field = 1 if nf == 6 else 8
    w[..., field] = np.where(rng.random(w.shape[:2]) < 1 / 9, big, w[..., field])
    _sweeps(w, limiter, 0.25, 1e-160)


@pytest.mark.parametrize("limiter", [0, 1, 2])
@pytest.mark.parametrize("bias", [1.5, -2.0])
def test_hpr_and_sub_cycles_with_a_bias_outside_its_range_match_oracle(vg_ctx, bias, limiter):
    w, _ = _state(17, 9, 33)
    dts = [1e-3, 2e-3]
    for thermal in (False, True):
        p = O.hpr_params(thermal)
        for sub in (0, 1):
            kw = dict(bias=bias, limiter=limiter, subcycles=sub, params=p)
            ref = O.hpr_fixed_dt(w, dts, dim=2, dx=1.0 / 33, **kw)
            got = S.hpr_solve_fixed_dt(w, 2, 1.0 / 33, dts, bias=bias, limiter=limiter, subcycles=sub,
                                       params=mat_params(p))
            if sub == 0:
                O.assert_bitwise(got, ref, f"thermal {thermal}")
            else:   # pow(det A, 5/3) may differ in its last bit between the GPU and glibc
                assert rel_l1(got, ref) <= 1e-10
    m, _ = _state(9)
    kw = dict(order=2, dim=2, dx=1.0 / 65, cfl=0.4, tfinal=np.inf, max_steps=3, bias=bias, limiter=limiter, subcycles=1)
    ref, dts = O.mhd_solve(m, gamma=5.0 / 3.0, **kw)
    r = S.mhd_solve(m, 2, 1.0 / 65, 0.4, np.inf, max_steps=3, bias=bias, limiter=limiter, subcycles=1,
                    params=S.MHDMaterialParameters(5.0 / 3.0))
    O.assert_bitwise(r.dt, dts, "MHD dt")
    O.assert_bitwise(r.cells, ref, "MHD state")


@pytest.mark.parametrize("thermal", [False, True])
@pytest.mark.parametrize("lo,hi", [(500, 520), (-520, -480)])
def test_distortions_whose_gramian_overflows_match_oracle(vg_ctx, lo, hi, thermal):
    """Distortions of 2^500 to 2^520 (an infinite trace, or one whose energy overflows) in
    one cell in nine, and of 2^-520 to 2^-480 (a trace below 2^-960)."""
    w, rng = _state(17, 12, 40)
    scale = np.exp2(rng.uniform(lo, hi, w.shape[:2]))
    scale = np.where(rng.random(w.shape[:2]) < 1 / 9, scale, 1.0)
    w[..., 2:11] *= scale[..., None]
    p = O.hpr_params(thermal)
    for dt in (1e-3, 1e-300):
        ref = O.hpr_fixed_dt(w, [dt], dim=2, dx=1.0 / 40, bias=0.0, limiter=1, subcycles=0, params=p)
        got = S.hpr_solve_fixed_dt(w, 2, 1.0 / 40, [dt], limiter=1, params=mat_params(p))
        _assert_alike(got, ref, f"dt {dt}")
