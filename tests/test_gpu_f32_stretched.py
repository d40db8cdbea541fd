"""FP32 on an azimuthal grid that is not uniform: interpolation coefficients per cell, widths per column,
and the planet's turn by the series instead of the rings' rotation rows."""
from __future__ import annotations

import numpy as np
import pytest

from penguin_2_0_amd import abi, configs

pytestmark = pytest.mark.gpu

VISC = dict(visc_flag=1, ss_alpha=3.0e-3, vis_nu=7.5e-6)
ADIA = dict(eos=3, gam=1.4, init_p_iso=1)


def stretched(grid, params):
    d = abi.init_disk(grid, params, 3, 1.0e-4)
    n = grid.jmax
    edges = np.linspace(0.0, 2.0 * np.pi, n + 1)
    edges = edges + 0.2 / n * np.sin(3.0 * edges) * 2.0 * np.pi   # widths vary by a fifth
    for a in (d.rings, d.lft, d.rgh):
        a["y"] = edges[:-1]
        a["dy"] = np.diff(edges)
        a["yc"] = edges[:-1] + 0.5 * np.diff(edges)
        a["yvol"] = np.diff(edges)
    return d


# azimuthal variants 0 and 1: windows of 116 kept columns; 2 and 3: of 244; 317 columns are a multiple of
# neither.  Viscous disks keep the short ones.
@pytest.mark.parametrize("over,var_y", [({}, 0), ({}, 1), ({}, 2), ({}, 3), (ADIA, 0), (ADIA, 3), (VISC, 1),
                                        ({**ADIA, **VISC}, 0)])
def test_stretched_azimuth_follows_fp64(over, var_y):
    """Each of 5 x 2 sweeps rounds a few hundred FP32 operations of the local state's size, 2^-24 of it
    each and of either sign: 1e-6 of it (of c_s for velocities) in the mean, and 1e-4 where a limiter chooses
    otherwise in a cell of the smooth start."""
    print("case: FP32 stretched azimuth", over, "variant", var_y, flush=True)
    grid, params = abi.PnGrid(48, 317, 1), configs.disk2d(48, 317, q=1.0e-3, fargo_flag=0, t_growth=0.0, **over)
    d = stretched(grid, params)
    out = []
    for prec in (abi.PN_FP32, abi.PN_FP64):
        with abi.Context(grid, params, prec) as ctx:
            ctx.load(d)
            if prec == abi.PN_FP32:
                ctx.set_variants(0, var_y)
            st = ctx.run_begin()
            ctx.run(5, st)
            out.append((ctx.store(), st.dt))
    (a, ta), (b, tb) = out
    assert abs(ta - tb) <= 1.0e-6 * tb
    cs = np.sqrt(b["p"] / b["r"])
    for f, scale in (("r", b["r"]), ("p", b["p"]), ("u", cs), ("v", cs)):
        e = np.abs(a[f] - b[f]) / scale
        print(f"  {f}: mean {e.mean():.2e} max {e.max():.2e}", flush=True)
        assert e.mean() <= 1.0e-6 and e.max() <= 1.0e-4, f
