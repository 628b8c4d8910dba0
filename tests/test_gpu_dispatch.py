"""Launch shapes chosen by size (levels per block of the chunked stencils,
columns per block of the vertical solve) against the fixed large-grid shapes:
the states are equal bit for bit, whole chunks or not.
"""
from __future__ import annotations

import os

import numpy as np
import pytest

from common import STATE, earth_params, grid

pytestmark = pytest.mark.gpu


def _run(capi, g, p, st, env, steps=2):
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        d = capi.Dyn(g, p)  # the switches are read when the handle is created
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
    print(f"case: g{glevel} L{nv} precision {precision}: shapes by size vs 16-level chunks, 64 columns", flush=True)
    g = grid(capi, glevel, nv)
    p = earth_params(capi, glevel, dt=600.0, ns=4, precision=precision)
    st = capi.ic_rest(g, p, seed=2040 + nv, temperature_noise=1e-3, wind_noise=1.0)
    a = _run(capi, g, p, st, {})
    b = _run(capi, g, p, st, {"THOR_STENCIL_LEVELS": "16", "THOR_THOMAS_COLUMNS": "64"})
    for k in STATE:
        assert np.isfinite(a[k]).all(), k
        assert np.array_equal(a[k], b[k]), k
