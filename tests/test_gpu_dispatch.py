"""Launch shapes chosen by size (levels per block of the chunked stencils,
columns per block of the vertical solve) against the fixed large-grid shapes:
the states are equal bit for bit, whole chunks or not.
"""
from __future__ import annotations

import ctypes as C
import os

import numpy as np
import pytest

from common import HIP_D2H, HIP_H2D, STATE, earth_params, grid, hip_runtime

pytestmark = pytest.mark.gpu


def _run(capi, g, p, st, env, steps=2, variant=""):
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        d = capi.Dyn(g, p, variant=variant)  # the switches are read when the handle is created
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v
    d.set_state(st)
    d.run(steps)
    d.sync()
    out = d.get_state()
    d.close()
    return out


@pytest.mark.parametrize("glevel,nv", [(4, 3), (4, 23), (4, 63), (5, 33)])
@pytest.mark.parametrize("precision", [0, 1])
def test_shapes_by_size_equal_the_fixed_ones(built, glevel, nv, precision):
    capi = built
    print(f"case: g{glevel} L{nv} precision {precision}: chunks by size vs 16 levels, columns 16 vs 64", flush=True)
    g = grid(capi, glevel, nv)
    p = earth_params(capi, glevel, dt=600.0, ns=4, precision=precision)
    st = capi.ic_rest(g, p, seed=2040 + nv, temperature_noise=1e-3, wind_noise=1.0)
    # the default kernels, chunks by size or of 16 levels, in both builds; then the vertical
    # solve with one lane per column (the columns are set in both), 16 or 64 of them per block
    lane = {"THOR_THOMAS_SEG": "0", "THOR_THOMAS_ROWS": "0"} if precision else {}
    for x, y, build in (({}, {"THOR_STENCIL_LEVELS": "16"}, ""), ({}, {"THOR_STENCIL_LEVELS": "16"}, "pm"),
                        (dict(lane, THOR_THOMAS_COLUMNS="16"),
                         dict(lane, THOR_STENCIL_LEVELS="16", THOR_THOMAS_COLUMNS="64"), "")):
        a, b = _run(capi, g, p, st, x, variant=build), _run(capi, g, p, st, y, variant=build)
        for k in STATE:
            assert np.isfinite(a[k]).all(), (x, build, k)
            assert np.array_equal(a[k], b[k]), (x, build, k)


@pytest.mark.parametrize("nv,extra", [
    (3, {}), (20, {}), (33, dict(DeepModel=0, NonHydro=0)), (23, dict(HyDiffOrder=8)), (21, dict(thermo_equation=1)),
    (20, dict(DivDampP=0)), (20, dict(HyDiff=0)),
    (23, dict(DiffSponge=1, order_diff_sponge=2)), (20, dict(HyDiffOrder=6, DiffSponge=1, order_diff_sponge=4)),
])
def test_fp64_operator_weights_equal_the_triangle_walk(built, nv, extra):
    """FP64 operators as weights per point against the reference's walk over
    the triangles (THOR_FP64_MULTILEVEL), one step with every option that
    reaches them. An operator is a sum of at most 84 products: in another order
    it moves by at most 84 x 2^-53 = 9e-15 of its largest term, and ten substeps
    add that up; 1e-12 of the field's scale (rho c_s for the momenta), as for
    the production build against the oracle."""
    capi = built
    print(f"case: FP64 g4 L{nv} {extra}: operator weights vs triangle walk, 1 step", flush=True)
    g = grid(capi, 4, nv)
    p = earth_params(capi, 4, dt=600.0, ns=6, **extra)
    st = capi.ic_rest(g, p, seed=2140 + nv, temperature_noise=1e-3, wind_noise=1.0)
    a = _run(capi, g, p, st, {}, steps=1)
    b = _run(capi, g, p, st, {"THOR_FP64_MULTILEVEL": "1"}, steps=1)
    cs = np.sqrt(p.Cp / (p.Cp - p.Rd) * p.Rd * p.Tmean)
    for k in STATE:
        scale = np.abs(b["Rho"]).max() * cs if k in ("Mh", "Wh", "W") else np.abs(b[k]).max()
        err = np.abs(a[k] - b[k]).max() / scale
        print(f"  {k}: {err:.2e}")
        assert err < 1e-12, k


@pytest.mark.parametrize("nv,extra", [
    (3, {}), (16, {}), (17, {}), (18, dict(DeepModel=0)), (33, dict(DeepModel=0, NonHydro=0, GravHeightVar=1)),
    (34, dict(GravHeightVar=1)), (49, {}), (65, {}), (66, {}), (97, {}),
])
@pytest.mark.parametrize("precision", [0, 1])
def test_row_solve_equals_the_one_lane_solve(built, nv, extra, precision):
    """Vertical solve with the sweeps on all rows of the block (affine maps
    scanned over the rows), the level constants from a table and one power per
    cell, and in FP64 the split flux divergence, against the one-lane solve
    (THOR_THOMAS_COLUMNS; mixed THOR_THOMAS_SEG 0), one step, with and without a
    hook between solve and update; up to 65 levels (four interfaces per row);
    above them the mixed form's sweeps run on all rows of k_thomas_dp and in FP64
    both are the one-lane solve. Bound as above: the recurrences are
    the same numbers in another association, each power within the portable
    pow's 2.5 (1 + |y log x|) ulp; the mixed form rounds the momentum deviation
    that follows to FP32, so 1e-9 there."""
    capi = built
    print(f"case: precision {precision} g4 L{nv} {extra}: row solve vs one lane per column, 1 step", flush=True)
    g = grid(capi, 4, nv)
    p = earth_params(capi, 4, dt=600.0, ns=6, precision=precision, **extra)
    st = capi.ic_rest(g, p, seed=2240 + nv, temperature_noise=1e-3, wind_noise=1.0)
    a = _run(capi, g, p, st, {}, steps=1)
    b = _run(capi, g, p, st, {"THOR_THOMAS_COLUMNS": "16", "THOR_THOMAS_SEG": "0", "THOR_THOMAS_ROWS": "0"}, steps=1)
    d = capi.Dyn(g, p)
    d.set_hooks(fast_modes=lambda stream, nstep, times, view: 0)
    d.set_state(st)
    d.run(1)
    d.sync()
    c = d.get_state()
    d.close()
    cs = np.sqrt(p.Cp / (p.Cp - p.Rd) * p.Rd * p.Tmean)
    for k in STATE:
        scale = np.abs(b["Rho"]).max() * cs if k in ("Mh", "Wh", "W") else np.abs(b[k]).max()
        err = np.abs(a[k] - b[k]).max() / scale
        print(f"  {k}: {err:.2e}")
        assert err < (1e-9 if precision else 1e-12), k
        assert np.array_equal(a[k], c[k]), ("hook split", k)


@pytest.mark.parametrize("precision,nv,extra", [
    (0, 20, {}), (1, 20, {}), (0, 3, {}), (1, 33, dict(DeepModel=0, NonHydro=0, GravHeightVar=1)),
    (0, 33, dict(DeepModel=0, NonHydro=0, GravHeightVar=1)), (1, 23, dict(DivDampP=0)), (0, 23, dict(HyDiff=0)),
    (0, 21, dict(NonHydro=0)), (1, 21, dict(NonHydro=0, GravHeightVar=1)),
    (0, 21, dict(thermo_equation=1)), (0, 20, dict(VertHyDiff=1, VertHyDiffOrder=6, Diffc_v=2e-3)),
])
def test_slow_modes_equal_the_reference_order(built, precision, nv, extra):
    """k_slow_w (weights in registers, constants from a table, the first stage's
    momentum written with the slow tendencies) against the kernels in the
    reference's order (THOR_SLOW_CHUNKED), one step with given forcing arrays.
    FP64: sums of at most 21 products in another order, 1e-12 of the field's
    scale. Mixed: the first stage's momentum is rounded to FP32 once instead of
    twice, so 2^-24 of rho c_s in the momenta and what that moves, 1e-7."""
    capi = built
    print(f"case: precision {precision} g4 L{nv} {extra}: k_slow_w vs the reference order, 1 step", flush=True)
    g = grid(capi, 4, nv)
    p = earth_params(capi, 4, dt=600.0, ns=6, precision=precision, **extra)
    st = capi.ic_rest(g, p, seed=2340 + nv, temperature_noise=1e-3, wind_noise=1.0)
    rng = np.random.default_rng(nv)
    tend = {"profx_Qheat": 1e-3 * rng.standard_normal((g.P, nv)), "profx_dMh": 1e-5 * rng.standard_normal((g.P, nv, 3)),
            "profx_dWh": 1e-6 * rng.standard_normal((g.P, nv + 1))}
    out = []
    for env in ({}, {"THOR_SLOW_CHUNKED": "1"}):
        for k, v in env.items():
            os.environ[k] = v
        try:
            d = capi.Dyn(g, p)
        finally:
            for k in env:
                os.environ.pop(k, None)
        d.set_state(st)
        for k, v in tend.items():
            d.set_field(k, v)
        d.thor()
        d.sync()
        out.append(d.get_state())
        d.close()
    a, b = out
    cs = np.sqrt(p.Cp / (p.Cp - p.Rd) * p.Rd * p.Tmean)
    for k in STATE:
        scale = np.abs(b["Rho"]).max() * cs if k in ("Mh", "Wh", "W") else np.abs(b[k]).max()
        err = np.abs(a[k] - b[k]).max() / scale
        print(f"  {k}: {err:.2e}")
        assert err < (1e-7 if precision else 1e-12), k


@pytest.mark.parametrize("precision", [0, 1])
def test_known_zero_tendencies_equal_zeros_read(built, precision):
    """Arrays of forcing tendencies that are known to be zero are not read:
    the same states as with zeros written to them, before and after a forcing
    that fills them (double-gray heating), ProfX clearing them again."""
    from common import hj_grid, hj_params, rt_params
    capi = built
    print(f"case: precision {precision} g4 L20: known zero tendencies", flush=True)
    g, p = hj_grid(capi, 4, 20), hj_params(capi, 4, precision=precision)
    st = capi.ic_rest(g, p, seed=2440, temperature_noise=1.0, wind_noise=1.0)
    z = {"profx_Qheat": np.zeros((g.P, 20)), "profx_dMh": np.zeros((g.P, 20, 3)), "profx_dWh": np.zeros((g.P, 21))}
    nr = capi.NewtonianParams(1600.0, 600.0, 0.0, 1e2, 1e7, 1e6, 1e4, 1e7)
    out = []
    for written in (False, True):
        d = capi.Dyn(g, p)
        d.set_newtonian(nr)
        d.set_rt(rt_params(capi))
        d.set_state(st)
        res = []
        for forcing in (capi.FORCING_NONE, capi.FORCING_NEWTONIAN, capi.FORCING_DOUBLE_GRAY, capi.FORCING_NEWTONIAN,
                        capi.FORCING_NONE):
            d.profx(forcing)
            if written:
                for k, v in z.items():
                    d.set_field(k, d.get_field(k) if k == "profx_Qheat" else v)
            d.thor()
            d.sync()
            res.append(dict(d.get_state(), q=d.get_field("profx_Qheat")))
        out.append(res)
        d.close()
    for i, (a, b) in enumerate(zip(*out)):
        for k in a:
            assert np.array_equal(a[k], b[k]), (i, k)
    assert np.abs(out[0][2]["q"]).max() > 0 and np.abs(out[0][3]["q"]).max() == 0


@pytest.mark.parametrize("nv,extra", [
    (3, {}), (16, {}), (17, dict(DeepModel=0)), (31, dict(GravHeightVar=1)), (32, dict(NonHydro=0)),
    (33, dict(DeepModel=0, NonHydro=0, GravHeightVar=1)), (48, {}), (63, {}), (64, dict(GravHeightVar=1)), (65, {}),
    (20, dict(thermo_equation=1)),
])
@pytest.mark.parametrize("precision", [0, 1])
def test_column_kernel_equals_the_separate_kernels(built, nv, extra, precision):
    """Stage update, column preparation and factorisation in one kernel (rows of
    one to four cells, constants from a table, pivots by scanned Moebius maps)
    against the three kernels (THOR_COLPREP_LEVELS), one step; above 64 levels
    both are the three. Bound: a few FP64 roundings per value and the powers'
    2.5 (1 + |y log x|) ulp, 1e-12 of a field's scale (gtilh differences two
    pressures, H / dz <= 20 times that); mixed: the advection's FP32 rounding
    may fall the other way, 1e-9. The energy equation has the FP64 form only."""
    capi = built
    if precision and extra.get("thermo_equation"):
        return
    print(f"case: precision {precision} g4 L{nv} {extra}: column kernel vs separate kernels, 1 step", flush=True)
    g = grid(capi, 4, nv)
    p = earth_params(capi, 4, dt=600.0, ns=6, precision=precision, **extra)
    st = capi.ic_rest(g, p, seed=2540 + nv, temperature_noise=1e-3, wind_noise=1.0)
    out = []
    for env in ({}, {"THOR_COLPREP_LEVELS": "2"}):
        os.environ.update(env)
        try:
            d = capi.Dyn(g, p)
        finally:
            for k in env:
                os.environ.pop(k, None)
        d.set_state(st)
        d.run(1)
        d.sync()
        out.append(dict(d.get_state(), **{k: d.get_field(k) for k in ("temperature", "h", "pt", "hh", "pth", "gtilh")}))
        d.close()
    a, b = out
    cs = np.sqrt(p.Cp / (p.Cp - p.Rd) * p.Rd * p.Tmean)
    for k in a:
        scale = np.abs(b["Rho"]).max() * cs if k in ("Mh", "Wh", "W") else np.abs(b[k]).max()
        err = np.abs(a[k] - b[k]).max() / scale
        print(f"  {k}: {err:.2e}")
        assert err < (1e-9 if precision else 2e-11 if k == "gtilh" else 1e-12), k


@pytest.mark.parametrize("glevel,nv", [(4, 3), (4, 21), (4, 22), (4, 64), (4, 65), (5, 97)])
def test_device_layout_equals_the_host_one(built, glevel, nv):
    """The state between device arrays in THOR's layout and the planes (tiles of
    32 points x at most 64 values of a point's row: remainders of both, one to
    five chunks per field) equals the conversion on the host, bit for bit, in both
    directions."""
    capi = built
    print(f"case: g{glevel} L{nv}: device layout", flush=True)
    hip = hip_runtime()
    g = grid(capi, glevel, nv)
    d = capi.Dyn(g, earth_params(capi, glevel, dt=600.0, ns=4))
    rng = np.random.default_rng(nv)
    st = {k: rng.standard_normal((g.P, nv + (k == "Wh")) + ((3,) if k == "Mh" else ())) for k in STATE}
    ptrs = {}
    try:
        for k in STATE:
            ptr = C.c_void_p()
            assert hip.hipMalloc(C.byref(ptr), st[k].nbytes) == 0
            ptrs[k] = ptr.value
            assert hip.hipMemcpy(ptrs[k], st[k].ctypes.data, st[k].nbytes, HIP_H2D) == 0
        s = capi.State(1, *(C.cast(C.c_void_p(ptrs[k]), capi._dp) for k in STATE))
        d._chk(d.L.thor_dyn_set_state(d._h, C.byref(s)))
        back = d.get_state()
        d.set_state({k: -st[k] for k in STATE})
        d._chk(d.L.thor_dyn_get_state(d._h, C.byref(s)))
        for k in STATE:
            out = np.empty_like(st[k])
            assert hip.hipMemcpy(out.ctypes.data, ptrs[k], out.nbytes, HIP_D2H) == 0
            assert np.array_equal(back[k].reshape(st[k].shape), st[k]), ("set", k)
            assert np.array_equal(out, -st[k]), ("get", k)
    finally:
        d.close()
        for ptr in ptrs.values():
            hip.hipFree(ptr)


@pytest.mark.parametrize("ns", [0.0, 0.96, 0.99])
@pytest.mark.parametrize("mode,temp", [(0, 0), (0, 1), (1, 1), (3, 0)])
def test_sponge_from_any_level_bitwise(built, ns, mode, temp):
    """The sponge's zonal means are formed at the damped levels only (Alt / top >=
    ns): all of the levels, the top one, none. Parity build, two steps against the
    oracle, which forms them everywhere: bit for bit."""
    from common import hj_grid, hj_params, nr_params
    from oracle.oracle import Oracle
    capi = built
    print(f"case: parity build, hot Jupiter g4 L20, sponge above {ns}, mode {mode}, temperature {temp}", flush=True)
    g, p = hj_grid(capi, 4, 20), hj_params(capi, 4)
    st = capi.ic_rest(g, p, seed=2640, temperature_noise=1.0, wind_noise=20.0)
    q = capi.SpongeParams(ns, 2e-4, 1e-4, 16, 1, 1, temp, 3e-4 if temp else 0.0, mode)
    d, o = capi.Dyn(g, p, variant="pm"), Oracle(g, p, variant="pm")
    for x in (d, o):
        x.set_state(st)
        x.set_newtonian(nr_params(capi))
        x.set_sponge(q)
    d.run(2, capi.FORCING_NEWTONIAN)
    d.sync()
    o.run(2, capi.FORCING_NEWTONIAN)
    a, b = d.get_state(), o.get_state()
    d.close()
    for k in STATE:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("hooked", [False, True])
def test_row_solve_takes_a_cell_without_pressure(built, precision, hooked):
    """A cell whose pressure is exactly zero: the update of the row solve divides
    by a power of it, the reference's does not; the new pressure is the
    reference's all the same, P_Ref (-Rd flux dt / P_Ref)^(Cp/Cv). Against the FP64
    one-lane solve in the reference's order, one short step; bounds as
    test_row_solve_equals_the_one_lane_solve, mixed against the FP64 form 1e-4."""
    capi = built
    print(f"case: precision {precision} g4 L20: zero pressure in one cell, hook {hooked}", flush=True)
    g = grid(capi, 4, 20)
    st = capi.ic_rest(g, earth_params(capi, 4, dt=1.0, ns=6), seed=2740, temperature_noise=1e-3, wind_noise=1.0)
    st["pressure"][1000, 7] = 0.0
    p = earth_params(capi, 4, dt=1.0, ns=6, precision=precision)
    d = capi.Dyn(g, p)
    if hooked:
        d.set_hooks(fast_modes=lambda stream, nstep, times, view: 0)
    d.set_state(st)
    d.run(1, capi.FORCING_NONE)
    d.sync()
    a = d.get_state()
    d.close()
    q = earth_params(capi, 4, dt=1.0, ns=6)
    os.environ["THOR_THOMAS_COLUMNS"] = "16"
    try:
        d = capi.Dyn(g, q)
    finally:
        del os.environ["THOR_THOMAS_COLUMNS"]
    d.set_state(st)
    d.run(1, capi.FORCING_NONE)
    d.sync()
    b = d.get_state()
    d.close()
    cs = np.sqrt(p.Cp / (p.Cp - p.Rd) * p.Rd * p.Tmean)
    for k in STATE:
        assert np.isfinite(b[k]).all(), k
        scale = np.abs(b["Rho"]).max() * cs if k in ("Mh", "Wh", "W") else np.abs(b[k]).max()
        err = np.abs(a[k] - b[k]).max() / scale
        print(f"  {k}: {err:.2e}")
        assert err < (1e-4 if precision else 1e-12), k
