"""Physics-module hooks and RK-advanced module arrays on the GPU.

THOR calls its physics modules at four points of the dynamics step
(phy_modules.h:76-86; thor_driver.cu:116, 641, 1290, 1465) and advances the
arrays they register like the state (UpdateRK / UpdateRK2,
thor_auxiliary.h:376-387, 482-494). Checked here:
  * the call sequence and the `times` argument of every call;
  * a hook between the vertical solve and the density/pressure update
    (which splits the fused column kernel in two) leaves the step bit for
    bit unchanged;
  * a module array with a constant tendency S added in every acoustic
    substep ends the step at x0 + S * dt exactly as the RK3 combination
    implies (stage weights 1/3, 1/2 - 1/3 ... sum to one step), for both
    precision modes. Closed form: the stage deviations start at 0, then
    x_i - x_k, so after stage 3 x_k = x0 + S * (ns * dt / ns) = x0 + S dt;
  * what a hook sets through the library (forcing tendencies, the sponge)
    counts from the next kernel on that reads it.
"""
from __future__ import annotations

import numpy as np
import pytest

from common import earth_params, grid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup(built):
    capi = built
    g = grid(capi, 4, 20)
    return capi, g


def _state(capi, g, p):
    return capi.ic_rest(g, p, seed=1004, temperature_noise=1e-3, wind_noise=1.0)


def test_hook_sequence_and_times(setup):
    capi, g = setup
    ns, dt = 6, 600.0
    print(f"case: FP64 g4 L20, ns={ns}, dt={dt}: hook call sequence over 2 steps", flush=True)
    p = earth_params(capi, 4, dt=dt, ns=ns)
    d = capi.Dyn(g, p)
    d.set_state(_state(capi, g, p))
    calls = []

    def rec(kind):
        if kind in ("init", "end"):
            def f(stream, nstep, view):
                assert stream != 0 and view.nv == g.nv and view.point_num == g.P and view.mhs_fp32 == 0
                calls.append((kind, nstep, None))
                return 0
        else:
            def f(stream, nstep, times, view):
                assert view.Whs and view.Rhok and view.Mhs
                calls.append((kind, nstep, times))
                return 0
        return f

    d.set_hooks(init=rec("init"), slow_modes=rec("slow"), fast_modes=rec("fast"), end=rec("end"))
    d.thor()
    d.thor()
    d.sync()
    want = []
    for step in (1, 2):
        want.append(("init", step, None))
        for rk, nit in enumerate((1, ns // 2, ns)):
            times = dt / 3.0 if rk == 0 else dt / ns
            want.append(("slow", step, times))
            want += [("fast", step, times)] * nit
        want.append(("end", step, None))
    assert calls == want
    d.close()


def test_hook_split_step_is_bitwise_unchanged(setup):
    capi, g = setup
    print("case: FP64 and mixed g4 L20, 2 steps with a no-op fast-mode hook vs none", flush=True)
    for prec in (capi.PRECISION_FP64, capi.PRECISION_MIXED):
        p = earth_params(capi, 4, dt=600.0, ns=6, precision=prec)
        st = _state(capi, g, p)
        a, b = capi.Dyn(g, p), capi.Dyn(g, p)
        a.set_state(st)
        b.set_state(st)
        b.set_hooks(fast_modes=lambda stream, nstep, times, view: 0)
        for d in (a, b):
            d.run(2, capi.FORCING_HELD_SUAREZ)
            d.sync()
        sa, sb = a.get_state(), b.get_state()
        for k in sa:
            assert np.array_equal(sa[k], sb[k]), (prec, k)
        a.close()
        b.close()


def _hip():
    """The HIP runtime the library itself links (device buffers for the test module)."""
    import ctypes as C
    import os
    hip = C.CDLL(os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib", "libamdhip64.so"))
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipFree.argtypes = [C.c_void_p]
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    hip.hipMemcpyAsync.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int, C.c_void_p]
    hip.hipMemsetAsync.argtypes = [C.c_void_p, C.c_int, C.c_size_t, C.c_void_p]
    hip.hipStreamSynchronize.argtypes = [C.c_void_p]
    return hip


def test_rk_array_constant_tendency(setup):
    """A module in the style of THOR's chemistry module (chemistry.cu:335-345,
    494-502): init copies tracer -> tracerk and clears the deviation, the
    fast-mode hook adds S * times to the deviation, end copies tracerk back."""
    import ctypes as C
    capi, g = setup
    hip = _hip()
    H2D, D2H, D2D = 1, 2, 3
    ns, dt, S, dims = 6, 600.0, 2.5e-3, 2
    for prec in (capi.PRECISION_FP64, capi.PRECISION_MIXED):
        print(f"case: precision {prec}, g4 L20: module array with constant tendency S = {S}", flush=True)
        p = earth_params(capi, 4, dt=dt, ns=ns, precision=prec)
        d = capi.Dyn(g, p)
        d.set_state(_state(capi, g, p))
        n = g.P * g.nv * dims
        nb = n * 8
        x0 = np.linspace(-1.0, 1.0, n)
        bufs = {}
        for k in ("tracer", "tracerk", "tracers"):
            ptr = C.c_void_p()
            assert hip.hipMalloc(C.byref(ptr), nb) == 0
            bufs[k] = ptr.value
        assert hip.hipMemcpy(bufs["tracer"], x0.ctypes.data, nb, H2D) == 0
        d.register_rk_array(bufs["tracers"], bufs["tracerk"], bufs["tracer"], dims)
        host = np.empty(n)

        def init(stream, nstep, view):
            hip.hipMemcpyAsync(bufs["tracerk"], bufs["tracer"], nb, D2D, stream)
            return hip.hipMemsetAsync(bufs["tracers"], 0, nb, stream)

        def fast(stream, nstep, times, view):
            hip.hipStreamSynchronize(stream)
            hip.hipMemcpy(host.ctypes.data, bufs["tracers"], nb, D2H)
            host[:] += S * times
            return hip.hipMemcpy(bufs["tracers"], host.ctypes.data, nb, H2D)

        def end(stream, nstep, view):
            return hip.hipMemcpyAsync(bufs["tracer"], bufs["tracerk"], nb, D2D, stream)

        d.set_hooks(init=init, fast_modes=fast, end=end)
        out = np.empty(n)
        for step in (1, 2):
            d.thor()
            d.sync()
            assert hip.hipMemcpy(out.ctypes.data, bufs["tracer"], nb, D2H) == 0
            err = np.abs(out - (x0 + step * S * dt)).max()
            print(f"  after {step} step(s): max |x - (x0 + n S dt)| = {err:.2e}")
            assert err < 1e-12
        d.clear_hooks()
        d.clear_rk_arrays()
        d.close()
        for v in bufs.values():
            hip.hipFree(v)


def test_hook_error_stops_the_step(setup):
    capi, g = setup
    print("case: FP64 g4 L20: a slow-mode hook that fails", flush=True)
    p = earth_params(capi, 4)
    d = capi.Dyn(g, p)
    d.set_state(_state(capi, g, p))
    d.set_hooks(slow_modes=lambda stream, nstep, times, view: 1)
    with pytest.raises(capi.ThorError) as e:
        d.thor()
    assert e.value.code == capi.THOR_ERR_HOOK
    d.sync()
    d.close()


@pytest.mark.parametrize("precision,variant,extra", [
    (0, "", {}), (1, "", {}), (0, "pm", {}), (0, "", dict(thermo_equation=1)),
])
def test_tendencies_set_by_a_hook_count_at_once(setup, precision, variant, extra):
    """A hook that sets the forcing tendencies with thor_dyn_set_field acts from
    the next kernel on that reads them, whether the arrays held zeros known to
    the host (which the step does not read) or written ones: bit for bit the
    same states. At the first slow-mode hook nothing has read them yet, so that
    equals setting them before the step, also where Held-Suarez clears the
    heating in every ProfX; at a fast-mode hook the update of that very substep
    takes the heating."""
    capi, g = setup
    p = earth_params(capi, 4, dt=600.0, ns=6, precision=precision, **extra)
    st = _state(capi, g, p)
    rng = np.random.default_rng(17)
    tend = {"profx_Qheat": 1e-2 * rng.standard_normal((g.P, g.nv)),
            "profx_dMh": 1e-4 * rng.standard_normal((g.P, g.nv, 3)),
            "profx_dWh": 1e-5 * rng.standard_normal((g.P, g.nv + 1))}

    def run(when, written, forcing, steps):
        """when: (hook, its index within the step); written: zeros written to the arrays before."""
        d = capi.Dyn(g, p, variant=variant)
        d.set_state(st)
        if written:
            for k, v in tend.items():
                d.set_field(k, np.zeros_like(v))
        seen = {}

        def hook(kind):
            def f(stream, nstep, *rest):
                i = seen[kind, nstep] = seen.get((kind, nstep), -1) + 1
                if (kind, i) == when:
                    for k, v in tend.items():
                        d.set_field(k, v)
                return 0
            return f

        d.set_hooks(init=hook("init"), slow_modes=hook("slow"), fast_modes=hook("fast"))
        d.run(steps, forcing)
        d.sync()
        out = d.get_state()
        d.close()
        return out

    none, hs = capi.FORCING_NONE, capi.FORCING_HELD_SUAREZ
    print(f"case: precision {precision} {variant} {extra}: tendencies set by hooks", flush=True)
    quiet = run(None, False, none, 1)
    pairs = [("first slow-mode hook = init hook, Held-Suarez", run(("slow", 0), False, hs, 2), run(("init", 0), False, hs, 2))]
    for when in (("slow", 0), ("slow", 1), ("fast", 0), ("fast", 2)):
        pairs.append((when, run(when, False, none, 1), run(when, True, none, 1)))
        assert np.abs(pairs[-1][1]["pressure"] - quiet["pressure"]).max() > 0, when
    for name, a, b in pairs:
        for k in a:
            assert np.isfinite(a[k]).all(), (name, k)
            assert np.array_equal(a[k], b[k]), (name, k)


@pytest.mark.parametrize("precision", [0, 1])
def test_sponge_switched_on_by_a_hook(setup, precision):
    """The explicit sponge writes the tendencies of the stage. Switched on by the
    first slow-mode hook of a step it acts in that stage, as when it was
    switched on before the step: bit for bit the same states."""
    from common import hj_grid, hj_params
    capi, _ = setup
    g, p = hj_grid(capi, 4, 20), hj_params(capi, 4, precision=precision)
    st = capi.ic_rest(g, p, seed=1104, temperature_noise=1.0, wind_noise=20.0)
    q = capi.SpongeParams(0.5, 2e-4, 1e-4, 16, 1, 1, 1, 3e-4, 3)
    out = []
    for by_hook in (False, True):
        print(f"case: precision {precision} hot Jupiter g4 L20: explicit sponge, switched on by a hook: {by_hook}", flush=True)
        d = capi.Dyn(g, p)
        d.set_state(st)
        calls = []

        def slow(stream, nstep, times, view):
            if not calls:
                d.set_sponge(q)
            calls.append(nstep)
            return 0

        if by_hook:
            d.set_hooks(slow_modes=slow)
        else:
            d.set_sponge(q)
        d.thor()
        d.sync()
        out.append(dict(d.get_state(), **{k: d.get_field(k) for k in ("profx_Qheat", "profx_dMh", "profx_dWh")}))
        d.close()
    a, b = out
    assert np.abs(a["profx_dMh"]).max() > 0 and np.abs(a["profx_Qheat"]).max() > 0
    for k in a:
        assert np.isfinite(a[k]).all(), k
        assert np.array_equal(a[k], b[k]), k


def _with_env(capi, g, p, env):
    """A handle created under the switches env."""
    import os
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        return capi.Dyn(g, p)
    finally:
        for k, v in old.items():
            os.environ.pop(k) if v is None else os.environ.update({k: v})


def _agree(p, a, b, tol):
    cs = np.sqrt(p.Cp / (p.Cp - p.Rd) * p.Rd * p.Tmean)
    for k in a:
        scale = np.abs(b["Rho"]).max() * cs if k in ("Mh", "Wh", "W") else np.abs(b[k]).max()
        err = np.abs(a[k] - b[k]).max() / scale
        print(f"  {k}: {err:.2e}")
        assert err < tol, k


@pytest.mark.parametrize("field,factor", [("hh", 2.0), ("gtilh", 2.0)])
@pytest.mark.parametrize("precision", [0, 1])
def test_slow_mode_hook_reaches_the_vertical_solve(setup, precision, field, factor):
    """hh and gtilh set by a slow-mode hook enter the stage's factorisation, also
    where the column kernel has formed it before the hook: against the separate
    kernels (THOR_COLPREP_LEVELS), which form it after. Bound as for the column
    kernel without a hook: FP64 rounding, 1e-12 of a field's scale, mixed 1e-9."""
    capi, g = setup
    p = earth_params(capi, 4, dt=600.0, ns=6, precision=precision)
    st = _state(capi, g, p)
    out = []
    for env, hooked in (({}, True), ({"THOR_COLPREP_LEVELS": "2"}, True), ({}, False)):
        print(f"case: precision {precision} g4 L20: {field} x {factor} by a slow-mode hook: {hooked}, {env}", flush=True)
        d = _with_env(capi, g, p, env)
        d.set_state(st)
        if hooked:
            def slow(stream, nstep, times, view):
                d.set_field(field, factor * d.get_field(field))
                return 0
            d.set_hooks(slow_modes=slow)
        d.thor()
        d.sync()
        out.append(d.get_state())
        d.close()
    a, b, quiet = out
    assert np.abs(b["Wh"] - quiet["Wh"]).max() > 1e-4 * np.abs(b["Wh"]).max()  # the hook does something
    _agree(p, a, b, 1e-9 if precision else 1e-12)


@pytest.mark.parametrize("field", ["pt", "h", "pth"])
def test_fast_mode_hook_reaches_the_flux_divergences(setup, field):
    """FP64: what a fast-mode hook sets of pt, h and pth enters the later substeps
    of the stage whole, also where the stage part of the pressure flux
    divergence has been formed with the slow tendencies: against the kernels
    that form it anew in every substep (THOR_THOMAS_SEG64). Bound as for the row
    solve: FP64 rounding, 1e-12 of a field's scale."""
    capi, g = setup
    p = earth_params(capi, 4, dt=600.0, ns=6)
    st = capi.ic_rest(g, p, seed=1204, temperature_noise=1.0, wind_noise=20.0)
    out = []
    for env, hooked in (({}, True), ({"THOR_THOMAS_SEG64": "0"}, True), ({}, False)):
        print(f"case: FP64 g4 L20: {field} x 1.1 by a fast-mode hook: {hooked}, {env}", flush=True)
        d = _with_env(capi, g, p, env)
        d.set_state(st)
        calls = []

        def fast(stream, nstep, times, view):
            if len(calls) == 2:  # the second stage's second substep of three
                d.set_field(field, 1.1 * d.get_field(field))
            calls.append(times)
            return 0
        if hooked:
            d.set_hooks(fast_modes=fast)
        d.thor()
        d.sync()
        out.append(d.get_state())
        d.close()
    a, b, quiet = out
    assert np.abs(b["pressure"] - quiet["pressure"]).max() > 1e-9 * np.abs(b["pressure"]).max()
    _agree(p, a, b, 1e-12)
