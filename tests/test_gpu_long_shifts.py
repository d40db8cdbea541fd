"""FARGO shifts of more than a turn: rot_j stays in [0, jmax), where the reference's single wrap
(ppm.cu:309-322) would leave it outside."""
from __future__ import annotations

import numpy as np
import pytest

from penguin_2_0_amd import abi, configs

pytestmark = pytest.mark.gpu


# rings rolled in the step's one workgroup and over the whole grid (more than 2048 slots)
@pytest.mark.parametrize("prec", [abi.PN_FP64, abi.PN_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("nr,nphi", [(40, 97), (2100, 24)])
def test_shifts_of_several_turns(nr, nphi, prec):
    print("case: shifts of several turns", nr, nphi, "precision", prec, flush=True)
    grid, params = abi.PnGrid(nr, nphi, 1), configs.disk2d(nr, nphi, q=1.0e-4)
    d = abi.init_disk(grid, params, 3, 1.0e-4)
    with abi.Context(grid, params, prec) as ctx:
        ctx.load(d)
        st = ctx.run_begin()
        mass = ctx.totals()[0]
        for _ in range(2):   # the second shift uses the rates the first one set
            ctx.index_shift(40.0, st.FrRot)
        inc = ctx.store()["inc_j"]
        assert np.abs(inc).max() > 3 * nphi and inc.min() < 0 < inc.max()
        for n in (1, 2, 3):
            ctx.sweep2d(1.0e-4, st.planet, st.FrRot)
            got = ctx.store()
            assert np.array_equal(got["rot_j"], (n * inc.astype(np.int64)) % nphi)
        assert all(np.isfinite(got[f]).all() for f in "rpuv")
        # three steps of 1e-4 move a cell by 1e-3 of its width at most
        assert abs(ctx.totals()[0] - mass) <= 1.0e-6 * mass


@pytest.mark.parametrize("graph", [False, True], ids=["launched", "replayed"])
def test_a_cold_disk_turns_many_times_a_step(graph):
    """Without sound speed and on Keplerian circles nothing limits dt (the first one is 1.1 times the run's
    end, 7e4, or 1e6 cells): the rings still roll to where their turns leave them."""
    print("case: cold disk, graph", graph, flush=True)
    grid, params = abi.PnGrid(30, 60, 1), configs.disk2d(30, 60, q=1.0e-4, plnt_flag=0).replace(sc_h=0.0)
    d = abi.init_disk(grid, params, 3, 1.0e-4)
    with abi.Context(grid, params, abi.PN_FP64) as ctx:
        ctx.load(d)
        st = ctx.run_begin()
        ctx.run(1, st, graph=False)
        one = ctx.store()
        assert np.abs(one["inc_j"].astype(np.int64)).max() > 60
        assert np.array_equal(one["rot_j"], one["inc_j"].astype(np.int64) % 60)
        ctx.run(5, st, graph=graph)
        got = ctx.store()
    assert got["rot_j"].min() >= 0 and got["rot_j"].max() < 60
