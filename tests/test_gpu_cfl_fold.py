"""A disk whose last sweep leaves more than 8192 CFL partials folds them in 256 chunks before the
step's single workgroup reads them: the post-step of a run's last step, and the mid-step of every
other one, also inside replayed graphs."""
from __future__ import annotations

import numpy as np
import pytest

from penguin_2_0_amd import abi, configs

pytestmark = pytest.mark.gpu

SPLIT = 8192   # partials a step kernel reads without the fold


def blocks_of_ring(ring: int, nwin: int, nring: int, waves: int):
    """The workgroups (of how many) that hold a ring's azimuthal windows: wave ring nwin + l, `waves` of
    them a workgroup, workgroup ids dealt round-robin over 8 XCDs that each walk a contiguous run."""
    nblk = -(-(nwin * nring) // waves)
    bid = np.arange(nblk)
    q, rem = divmod(nblk, 8)
    item = (bid % 8) * q + np.minimum(bid % 8, rem) + bid // 8
    mine = (ring * nwin + np.arange(nwin)) // waves
    return bid[np.isin(item, mine)], nblk


# FP32: the 1024 x 3072 disk with azimuthal variant 0, two 128-cell windows a workgroup; FP64: four,
# and more rings.  The ring's workgroups lie past partial 8192, so a step that read only the first
# ones would miss it.
@pytest.mark.parametrize("prec,nr,waves,ring", [(abi.PN_FP32, 1024, 2, 103), (abi.PN_FP64, 1300, 4, 160)],
                         ids=["fp32", "fp64"])
@pytest.mark.parametrize("graph", [False, True], ids=["launched", "replayed"])
def test_folded_partials_set_dt(prec, nr, waves, ring, graph):
    w = configs.Workload(f"disk_{nr}x3072", abi.PnGrid(nr, 3072, 1), configs.disk2d(nr, 3072), seed=5, steps=4)
    blocks, nblk = blocks_of_ring(ring, -(-3072 // 116), nr, waves)
    print("case: CFL fold,", w.name, "precision", prec, "partials", nblk, "ring's", blocks.min(), "..", blocks.max(),
          "graph", graph, flush=True)
    assert nblk > SPLIT and blocks.min() > SPLIT
    d = abi.init_disk(w.grid, w.params, w.seed, w.noise)
    d.rings["v"][ring, :] += 0.25   # super-Keplerian: its azimuthal signal speed sets dt
    dts = {}
    for n in (3, 4):
        with abi.Context(w.grid, w.params, prec) as ctx:
            ctx.load(d)
            if prec == abi.PN_FP32:
                ctx.set_variants(0, 0)
            st = ctx.run_begin()
            ctx.run(n, st, graph=graph)
            dts[n] = st.dt
            if n == 3:
                p, FrRot = ctx.store(), st.FrRot
    # timestep.cu:12-73 on the state after three steps
    r = p["xc"][:, None]
    cs = np.sqrt(w.params.gam * p["p"] / p["r"])
    rate = np.maximum((np.abs(p["u"]) + cs) / p["dx"][:, None],
                      (np.abs(p["v"] - p["rot_v"][:, None] - FrRot * r) + cs) / (r * p["dy"]))
    assert rate.max(axis=1).argmax() == ring
    want = min(1.1 * dts[3], w.params.courant / rate.max())
    print(f"  dt of step 4 {dts[4]!r}, from the state {want!r}", flush=True)
    # FP32 forms a rate in three roundings of 2^-24; FP64 agrees to its last bits
    assert abs(dts[4] - want) <= (1.0e-6 if prec == abi.PN_FP32 else 1.0e-14) * want
    assert want < 0.999 * 1.1 * dts[3]   # the signal speed limits dt, not its growth
