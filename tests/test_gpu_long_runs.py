"""Runs long enough for graphs of several steps: the first step apart, eight steps a replay,
single steps for the remainder, against the same steps launched one by one."""
from __future__ import annotations

import numpy as np
import pytest

from penguin_2_0_amd import abi, configs

pytestmark = pytest.mark.gpu

HPI = 1.570796326794896619231321691639751442


def say(*a):
    print(*a, flush=True)


def spherical(nr, nphi, nth):
    p = configs.disk2d(nr, nphi, q=3.0e-5).replace(
        ndim=3, ngeomx=2, ngeomy=4, ngeomz=5, p_alpha=1.5, p_beta=1.0, zmin=HPI - 0.15, zmax=HPI + 0.15)
    return configs.Workload(f"disk3d_{nr}x{nphi}x{nth}", abi.PnGrid(nr, nphi, nth), p, seed=11, steps=10)


# a small disk, one whose rings are shifted over the whole grid (more than 2048 slots), a 3-D disk
# (two steps to return to its buffer), damping (the CFL apart) and a planet that feels the disk
CASES = [configs.small(48, 144), configs.small(2100, 24), spherical(16, 48, 8), configs.small(60, 97, kill_flag=1),
         configs.small(40, 120, plnt_flag=2, M_p=1e-3)]


@pytest.mark.parametrize("prec", [abi.PN_FP64, abi.PN_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("w", CASES, ids=lambda w: f"{w.name}_{w.params.plnt_flag}{w.params.kill_flag}")
def test_graph_of_several_steps_gives_the_eager_bytes(w, prec):
    d = abi.init_disk(w.grid, w.params, w.seed, w.noise)
    out = []
    for graph in (True, False):
        say("case: long run", w.name, "precision", prec, "graph", graph)
        with abi.Context(w.grid, w.params, prec) as ctx:
            ctx.load(d)
            if prec == abi.PN_FP32:
                ctx.set_variants(0, 3)
            st = ctx.run_begin()
            for n in (29, 3, 18):   # graphs kept from one call to the next, and one made anew
                ctx.run(n, st, graph=graph)
            out.append((ctx.store(), st.dt, st.simtime, st.planet.x, st.planet.y, st.ncycle))
    assert out[0][1:] == out[1][1:]
    assert np.array_equal(out[0][0].view(np.uint8), out[1][0].view(np.uint8))


def test_batch_graph_of_several_steps_gives_the_eager_bytes():
    ws = [configs.small(48, 144), configs.small(72, 216, M_p=1e-4), configs.small(33, 97)]
    disks = [abi.init_disk(w.grid, w.params, w.seed + k, w.noise) for k, w in enumerate(ws)]
    out = []
    for graph in (True, False):
        say("case: long run of a batch, graph", graph)
        with abi.Batch([w.grid for w in ws], [w.params for w in ws]) as b:
            for ctx, d in zip(b.disks, disks):
                ctx.load(d)
            b.set_variants(0, 1)
            st = b.run_begin()
            for n in (21, 2, 11):
                b.run(n, st, graph=graph)
            out.append([(c.store().tobytes(), s.dt, s.simtime) for c, s in zip(b.disks, st)])
    assert out[0] == out[1]
