"""FP32 pencils: windows of every number of columns per wavefront, and states whose jumps leave
the series of the interface solver."""
from __future__ import annotations

import numpy as np
import pytest

from penguin_2_0_amd import abi, configs

pytestmark = pytest.mark.gpu

HPI = 1.570796326794896619231321691639751442


def say(*a):
    print(*a, flush=True)


def run(w, prec, d, n, pack=True, var_x=0, var_y=3):
    with abi.Context(w.grid, w.params, prec) as ctx:
        ctx.load(d)
        if prec == abi.PN_FP32:
            ctx.set_packing(pack)
            ctx.set_variants(var_x, var_y)
        st = ctx.run_begin()
        ctx.run(n, st)
        return ctx.store(), st


# a 128-cell window keeps 116: the last window keeps 1, 9, 20, 31 rings and runs 9, 5, 4, 2 columns
# per wavefront; theta pencils of 4, 9, 20, 31 and 52 cells run 8, 5, 4, 2 and 2
@pytest.mark.parametrize("nr,nth", [(117, 1), (125, 1), (136, 1), (147, 1), (20, 4), (15, 9), (12, 20), (12, 31), (12, 52)])
def test_columns_per_wavefront_give_the_same_bytes(nr, nth):
    p = configs.disk2d(nr, 97, q=1.0e-4)
    if nth > 1:
        p = p.replace(ndim=3, ngeomx=2, ngeomy=4, ngeomz=5, p_alpha=1.5, p_beta=1.0, zmin=HPI - 0.15, zmax=HPI + 0.15)
    w = configs.Workload(f"disk_{nr}x97x{nth}", abi.PnGrid(nr, 97, nth), p, seed=5, steps=5)
    d = abi.init_disk(w.grid, w.params, w.seed, w.noise)
    for vx in (0, 3):
        say("case: columns per wavefront", w.name, "radial variant", vx)
        a, sa = run(w, abi.PN_FP32, d, 5, True, vx)
        b, sb = run(w, abi.PN_FP32, d, 5, False, vx)
        assert sa.dt == sb.dt
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), (w.name, vx)


@pytest.mark.parametrize("eos", [0, 3])
@pytest.mark.parametrize("ratio", [1.15, 1.35, 3.0])
def test_strong_jumps_follow_fp64(eos, ratio):
    """Density steps along both directions: relative jumps below 1/5, between 1/5 and 1/2 and far
    above, so the interface logs and exponentials run by series, by both and by the library (and
    the steepest are flattened with EOS 3; without it v is constant along phi beside the steps, so
    whether a flow converges there, which switches the flattening of a cell on, is decided by the
    last bit of equal numbers, in FP32 and FP64 alike).  Each of the 3 x 2 sweeps rounds a few hundred FP32 operations of
    the local state's size (2^-24 of it each, so about 1e-6 if none cancel), and limiters may
    choose differently in single cells beside a step: 1e-5 in the mean, 2e-3 at most."""
    over = dict(eos=3, gam=1.4, init_p_iso=1) if eos == 3 else dict(flat_flag=0)
    w = configs.small(70, 200, **over)
    d = abi.init_disk(w.grid, w.params, w.seed, w.noise)
    f = np.ones((70, 200))
    f[20:45, 50:120] = ratio
    d.rings["r"] *= f
    d.rings["p"] *= f
    say("case: strong jumps, eos", eos, "ratio", ratio)
    a, sa = run(w, abi.PN_FP32, d, 3)
    b, sb = run(w, abi.PN_FP64, d, 3)
    cs = np.sqrt(b["p"] / b["r"])
    assert abs(sa.dt - sb.dt) <= 1e-5 * sb.dt
    for k, scale in (("r", b["r"]), ("p", b["p"]), ("u", cs), ("v", cs)):
        e = np.abs(a[k] - b[k]) / scale
        say(f"  {k}: mean {e.mean():.2e} max {e.max():.2e}")
        assert e.mean() <= 1e-5 and e.max() <= 2e-3, k
