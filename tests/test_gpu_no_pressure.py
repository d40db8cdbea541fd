"""FP64 cells without pressure: a loaded state may hold p = 0, whose sound speed is 0 and whose edge the
flattening sees as an unbounded jump.  The interface states are floored at 1e-15 (states.cu:45-68), so
the disk goes on; against the oracle, bars of 5 steps as in test_gpu_fp64_windows.py (3-D as there)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from penguin_2_0_amd import abi, configs

pytestmark = pytest.mark.gpu

HPI = 1.570796326794896619231321691639751442


@pytest.mark.parametrize("kind", ["isothermal", "viscous", "adiabatic", "spherical"])
def test_cells_without_pressure(kind):
    print("case: cells without pressure,", kind, flush=True)
    over = {"viscous": dict(visc_flag=1, ss_alpha=3.0e-3, vis_nu=7.5e-6),
            "adiabatic": dict(eos=3, gam=1.4, init_p_iso=1)}.get(kind, {})
    p = configs.disk2d(60, 130, **over)
    grid = abi.PnGrid(60, 130, 1)
    if kind == "spherical":
        p = p.replace(ndim=3, ngeomx=2, ngeomy=4, ngeomz=5, p_alpha=1.5, p_beta=1.0, zmin=HPI - 0.15, zmax=HPI + 0.15)
        grid = abi.PnGrid(24, 60, 14)
    d = abi.init_disk(grid, p, 3, 1.0e-4)
    o = oracle.OracleDisk(grid, p, 3, 1.0e-4)
    for s in (d, o):
        s.rings["p"][grid.imax // 3: grid.imax // 2, 20:40] = 0.0
    steps = 1 if kind == "adiabatic" else 2   # gas that streams into the void crosses cells in its second step
    so = o.run_begin()
    o.run(steps, so)
    with abi.Context(grid, p, abi.PN_FP64) as ctx:
        ctx.load(d)
        st = ctx.run_begin()
        ctx.run(steps, st)
        got = ctx.store()
    l1, linf = (1.0e-10, 1.0e-7) if kind == "spherical" else (1.0e-11, 1.0e-8)
    assert abs(st.dt - so.dt) <= 1.0e-9 * so.dt
    for f in "rpuv":
        e, s = np.abs(got[f] - o.rings[f]), np.abs(o.rings[f])
        print(f"  {f}: L1 {e.sum() / s.sum():.2e} Linf {e.max() / s.max():.2e}", flush=True)
        assert np.isfinite(o.rings[f]).all()
        assert e.sum() <= l1 * s.sum() and e.max() <= linf * s.max(), f
