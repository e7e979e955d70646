"""The sweeps' two shapes -- tiles of one cell per thread on small grids, blocks
walking rows on large ones -- at the edges of their tiles and on both sides of the
rule that picks them.  Everything here is add, multiply, divide and square root, so
every comparison is bit for bit."""

import math

import numpy as np
import pytest

import oracle_lib as O
from vanguard_amd import _lib, problems
from vanguard_amd import solvers as S

pytestmark = pytest.mark.gpu

EULER = [1.4, 0, 25, 0.3, 0.25, 250]


def _state(physics, ny, nx):
    rng = np.random.default_rng(ny * 1000 + nx)
    shape = (ny, nx)
    if physics == "euler":
        w = rng.uniform(-0.3, 0.3, shape + (6,))
        w[..., 0] = rng.uniform(0.5, 1.5, shape)
        w[..., 4] = rng.uniform(0.5, 1.5, shape)
        w[..., 5] = rng.uniform(0.0, 1.0, shape)
    elif physics == "mhd":
        w = rng.uniform(-0.3, 0.3, shape + (9,))
        w[..., 0] = rng.uniform(0.5, 1.5, shape)
        w[..., 4] = rng.uniform(0.5, 1.5, shape)
    else:
        w = rng.uniform(-0.05, 0.05, shape + (17,))
        w[..., 0] += 1.0
        w[..., 1] += 1.0 / 1.4
        w[..., 2:11] += np.eye(3).ravel()
    return w


def _gpu(physics, w, dx, order, bc, steps, limiter=1, bias=0.0, **kw):
    kw.update(order=order, limiter=limiter, bias=bias, max_steps=steps, bc=bc)
    if physics == "euler":
        return S.euler_solve(w, 2, dx, 0.6, np.inf, params=S.EulerMaterialParameters(*EULER), **kw)
    if physics == "mhd":
        return S.mhd_solve(w, 2, dx, 0.6, np.inf, params=S.MHDMaterialParameters(5.0 / 3.0, 0.0, 0.7, 0.4), **kw)
    return S.hpr_solve(w, 2, dx, 0.4, np.inf, params=S.HPRMaterialParameters(is_thermal=False), **kw)


def _oracle(physics, w, dx, order, bc, steps, limiter=1, bias=0.0):
    kw = dict(order=order, dim=2, dx=dx, tfinal=np.inf, max_steps=steps, bias=bias, limiter=limiter, bc=bc)
    if physics == "euler":
        return O.euler_solve(w, cfl=0.6, params=EULER, **kw)
    if physics == "mhd":
        return O.mhd_solve(w, cfl=0.6, gamma=5.0 / 3.0, ch=0.7, cp=0.4, **kw)
    return O.hpr_solve(w, cfl=0.4, subcycles=0, params=O.hpr_params(False), **kw)


# Output rows of a y tile: 28 (SLIC; 60 for the 64-row shape), 30 (FORCE); output
# columns of an x tile: 60 (SLIC), 62 (FORCE); y tiles are 8 or 4 columns wide.  Eleven
# steps: a replay of eight, in which a step begins inside its first sweep, and three
# launched one by one.
@pytest.mark.parametrize("physics", ["euler", "mhd", "hpr"])
@pytest.mark.parametrize("ny,nx", [(2, 2), (28, 60), (29, 61), (30, 62), (31, 9), (57, 121), (61, 4)])
def test_tile_edges_match_oracle(vg_ctx, physics, ny, nx):
    w = _state(physics, ny, nx)
    for order in (2, 1):
        for bc in (S.TRANSMISSIVE, S.PERIODIC):
            r = _gpu(physics, w, 1.0 / nx, order, bc, 11)
            ref, dts = _oracle(physics, w, 1.0 / nx, order, bc, 11)
            O.assert_bitwise(r.dt, dts, f"{physics} {ny}x{nx} order {order} bc {bc} dt")
            O.assert_bitwise(r.cells, ref, f"{physics} {ny}x{nx} order {order} bc {bc} state")


@pytest.mark.parametrize("physics,ny,nx,rep", [("euler", 133, 134, 10), ("mhd", 109, 110, 10), ("hpr", 82, 83, 10)])
def test_large_grids_take_the_walking_sweeps_with_the_same_bits(vg_ctx, physics, ny, nx, rep):
    """A periodic state repeated over a grid beyond the small-tile rule (over 160 MB
    read and written per sweep; FORCE 48 MB) advances as its repeated unit does: the walking
    sweeps against the tiles (y: what the tuner picks)."""
    unit = _state(physics, ny, nx)
    big = np.ascontiguousarray(np.tile(unit, (rep, rep, 1)))
    assert 2 * big.nbytes > 160 << 20 > 2 * unit.nbytes
    for order in (2, 1):
        a = _gpu(physics, unit, 1.0 / nx, order, S.PERIODIC, 3)
        b = _gpu(physics, big, 1.0 / nx, order, S.PERIODIC, 3)
        O.assert_bitwise(b.dt, a.dt, f"{physics} order {order} dt")
        O.assert_bitwise(b.cells, np.tile(a.cells, (rep, rep, 1)), f"{physics} order {order} state")


# One x block a row is a key: 2 x 512 keys are the most a step that begins inside its
# first sweep reduces (columns 61 .. 120 take two tiles; FORCE 63 .. 124).
@pytest.mark.parametrize("ny,nx", [(512, 97), (513, 97)])
def test_steps_on_both_sides_of_the_key_limit_match_oracle(vg_ctx, ny, nx):
    w = _state("euler", ny, nx)
    for order in (2, 1):
        r = _gpu("euler", w, 1.0 / nx, order, S.TRANSMISSIVE, 11)
        ref, dts = _oracle("euler", w, 1.0 / nx, order, S.TRANSMISSIVE, 11)
        O.assert_bitwise(r.dt, dts, f"order {order} dt")
        O.assert_bitwise(r.cells, ref, f"order {order} state")


@pytest.fixture
def ctx():
    c = S.Context(0)
    yield c
    c.close()


def _pin(c, physics, order, mode, shape, x, y):
    """x: 0 walked rows, 1 tiles; y: a y variant."""
    names = ("euler", "euler_planar") if physics == "euler" else (physics,)
    for name in names:
        key = f"{name}/{order}/{int(mode)}/{shape[0]}/{shape[1]}"
        c.set_tuned_key(key, y)
        c.set_tuned_key(key + "/x", x)
        c.set_tuned_key("rgfm_" + key + "/x", x)


# Walked x blocks put out 252 columns by 4 rows (HPR 124 by 3; FORCE 2 more), walked y
# strips are 64 rows or 16 (HPR): partial ones of each.  Limiters 0 superbee, 1 van
# Leer, 2 minbee.
@pytest.mark.parametrize("limiter,bias", [(0, 0.0), (1, -0.35), (2, 1.0)])
@pytest.mark.parametrize("physics,ny,nx", [("euler", 70, 261), ("euler", 6, 505), ("mhd", 70, 255), ("hpr", 19, 131)])
def test_pinned_walks_and_tiles_match_oracle(ctx, physics, ny, nx, limiter, bias):
    w = _state(physics, ny, nx)
    for order in (2, 1):
        for bc in (S.TRANSMISSIVE, S.PERIODIC):
            ref, dts = _oracle(physics, w, 1.0 / nx, order, bc, 9, limiter, bias)
            for x, y in ((0, 0), (1, 4)):
                _pin(ctx, physics, order, S.EXACT, (ny, nx), x, y)
                r = _gpu(physics, w, 1.0 / nx, order, bc, 9, limiter, bias, ctx=ctx)
                what = f"{physics} order {order} bc {bc} shape {x}"
                O.assert_bitwise(r.dt, dts, what + " dt")
                O.assert_bitwise(r.cells, ref, what + " state")


@pytest.mark.parametrize("physics,ny,nx", [("euler", 70, 261), ("mhd", 70, 255), ("hpr", 19, 131)])
def test_pinned_walks_and_tiles_round_alike_in_fast_mode(ctx, physics, ny, nx):
    w = _state(physics, ny, nx)
    states = [w]
    if physics == "euler":   # the 4-field sweeps too
        planar = w.copy()
        planar[..., 3], planar[..., 5] = 0.0, 1.0
        states.append(planar)
    for w in states:
        for order in (2, 1):
            for limiter, bias, bc in ((0, 0.0, S.TRANSMISSIVE), (1, 0.4, S.PERIODIC), (2, -1.0, S.TRANSMISSIVE)):
                runs = []
                for x, y in ((0, 0), (1, 4)):
                    _pin(ctx, physics, order, S.FAST, (ny, nx), x, y)
                    runs.append(_gpu(physics, w, 1.0 / nx, order, bc, 9, limiter, bias, mode=S.FAST, ctx=ctx))
                O.assert_bitwise(runs[0].dt, runs[1].dt, f"{physics} order {order} limiter {limiter} dt")
                O.assert_bitwise(runs[0].cells, runs[1].cells, f"{physics} order {order} limiter {limiter} state")


@pytest.mark.parametrize("model", ["multiphysics", "reduced"])
def test_pinned_walks_and_tiles_of_the_two_material_models_match_oracle(ctx, model):
    kind = ("multiphysics", "reduced").index(model)
    ny, nx = 37, 135
    rng = np.random.default_rng(kind)
    nf = O.MP_NP[kind]
    w = np.zeros((ny, nx, nf))
    w[..., 0] = np.where(np.arange(nx) < nx // 2, 0.999, 0.001)[None, :]
    w[..., 1:3] = rng.uniform(-0.2, 0.2, (ny, nx, 2))
    w[..., 4:] = rng.uniform(0.5, 1.5, (ny, nx, nf - 4))
    p1, p2 = (1.4, 0.0, 25.0, 0.0, 0.25, 250.0), (3.0, 0.1, 25.0, 0.0, 0.25, 250.0)
    for order in (2, 1):
        ref, dts = O.mp_solve(kind, w, order=order, dim=2, dx=1 / nx, cfl=0.6, tfinal=math.inf, max_steps=9, bias=0.2,
                              limiter=0, reinit=2, p1=p1, p2=p2)
        for x, y in ((0, 0), (1, 4)):
            _pin(ctx, "euler_" + model, order, S.EXACT, (ny, nx), x, y)
            r = S.two_material_solve(model, w, 2, 1 / nx, 0.6, math.inf, order=order, limiter=0, bias=0.2,
                                     reinit_every=2, params1=S.EulerMaterialParameters(*p1),
                                     params2=S.EulerMaterialParameters(*p2), max_steps=9, ctx=ctx)
            O.assert_bitwise(r.dt, dts, f"order {order} shape {x} dt")
            O.assert_bitwise(r.cells, ref, f"order {order} shape {x} state")


@pytest.mark.parametrize("planar", [True, False])
def test_rgfm_steps_are_the_same_bits_in_every_shape(ctx, planar):
    """Each direction's pair launch (tiles) and its single launches (walks)."""
    ny, nx = 70, 261
    m1, m2, phi, dx, dy = problems.shock_bubble_2d(nx, ny)
    if not planar:
        m1[..., 3], m2[..., 3] = 0.1, -0.1
    runs = []
    for x, y in ((0, 0), (1, 4), (1, 5), (0, 4), (1, 0)):
        _pin(ctx, "euler", 2, S.EXACT, (ny, nx), x, y)
        runs.append(S.rgfm_solve(S.MultimaterialSystem(m1, m2, phi), dx, 0.6, math.inf,
                                 S.EulerMaterialParameters(*problems.HELIUM), S.EulerMaterialParameters(*problems.AIR),
                                 dy=dy, limiter=0, max_steps=11, ctx=ctx))
    for r in runs[1:]:
        O.assert_bitwise(r.dt, runs[0].dt, "dt")
        for a, b in ((r.system.material1, runs[0].system.material1), (r.system.material2, runs[0].system.material2),
                     (r.system.level_set, runs[0].system.level_set)):
            O.assert_bitwise(a, b, "state")


def test_pins_outside_a_keys_variants_are_refused(ctx):
    for key, last in (("euler/2/0/8/9/x", 1), ("euler/2/0/8/9", 7)):
        ctx.set_tuned_key(key, last)
        assert ctx.tuned_key(key) == last
        with pytest.raises(_lib.VanguardError):
            ctx.set_tuned_key(key, last + 1)
        ctx.set_tuned_key(key, -1)
        assert ctx.tuned_key(key) == -1
