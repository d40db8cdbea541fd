"""The time step of a frame that follows a planet off the circle: dt comes from the frame's rate after
the step that ended (timestep.cu:12-73 runs at the start of each step), not from the rate its sweeps
saw."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from penguin_2_0_amd import abi, configs

pytestmark = pytest.mark.gpu


def states(params, vx):
    grid = abi.PnGrid(40, 400, 1)
    d = abi.init_disk(grid, params, 3, 1.0e-4)
    o = oracle.OracleDisk(grid, params, 3, 1.0e-4)
    so = o.run_begin()
    so.planet.vx = vx
    return grid, d, o, so


# a radial velocity, given to the planet of a frame at rest before it; a radius whose circle does not
# close to the last bit (the frame's rate moves in its last bits only)
@pytest.mark.parametrize("vx,radius", [(0.02, 1.0), (0.0, 1.1), (0.0, 1.0)])
@pytest.mark.parametrize("steps,graph", [(5, False), (40, True)])
def test_dt_follows_the_frame(vx, radius, steps, graph):
    print("case: frame rate, vx", vx, "radius", radius, "steps", steps, "graph", graph, flush=True)
    params = configs.disk2d(40, 400, q=1.0e-4, plnt_flag=1, frrot_flag=1, R_p=radius)
    grid, d, o, so = states(params, vx)
    with abi.Context(grid, params, abi.PN_FP64) as ctx:
        ctx.load(d)
        st = ctx.run_begin()
        st.planet.vx = vx
        for _ in range(2):   # the second run starts from what the first one left
            o.run(steps, so)
            ctx.run(steps, st, graph=graph)
            print(f"  dt {st.dt!r} oracle {so.dt!r}, FrRot {st.FrRot!r} {so.FrRot!r}", flush=True)
            # equal arithmetic but for the disk's own differences (1e-11 of a cell after ten steps); the
            # rate of the step before moves dt by several 1e-3 where vx is 0.02 (the azimuthal width limits dt)
            assert abs(st.dt - so.dt) <= 1.0e-9 * so.dt
            assert abs(st.FrRot - so.FrRot) <= 1.0e-12
        got = ctx.store()
    assert np.array_equal(got["rot_j"], o.rings["rot_j"])


def test_frame_set_in_motion_between_runs():
    """One context, replayed steps kept: at rest, then moving, then at rest again."""
    print("case: frame set in motion between runs", flush=True)
    params = configs.disk2d(40, 400, q=1.0e-4, plnt_flag=1, frrot_flag=1)
    grid = abi.PnGrid(40, 400, 1)
    d = abi.init_disk(grid, params, 3, 1.0e-4)
    out = []
    for graph in (True, False):
        with abi.Context(grid, params, abi.PN_FP64) as ctx:
            ctx.load(d)
            st = ctx.run_begin()
            rest = (st.planet.x, st.planet.vx, st.planet.vy, st.planet.fx, st.planet.fy, st.FrRot)
            log = []
            for vx in (0.0, 0.01, 0.0):
                p = st.planet
                p.x, p.vx, p.vy, p.fx, p.fy, st.FrRot = rest
                p.vx = vx
                ctx.run(27, st, graph=graph)
                log += [st.dt, st.FrRot, st.simtime]
            out.append((log, ctx.store().tobytes()))
    assert out[0] == out[1]
