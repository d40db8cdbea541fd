"""FP64 sweeps against the oracle where their windows and branches change: last windows of 64 and
65 cells (two columns a wavefront up to 64), column counts that leave part of a workgroup empty,
theta pencils on both sides of the same line, a stretched azimuthal grid (interpolation
coefficients and the planet's turn per cell), coarse rings whose shift leaves the short sine
series, and density jumps that leave the interface's series.

Bars as in test_gpu_parity.py's 10 steps: relative L1 1e-11, Linf 1e-8 (3-D: 1e-10, 1e-7, as in
test_gpu_parity_flags.py; v_theta's bar is derived where it is used)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from penguin_2_0_amd import abi, configs

pytestmark = pytest.mark.gpu


def close(got, ref, fields, l1, linf, what):
    for f in fields:
        d = np.abs(got[f] - ref[f])
        s1, si = np.abs(ref[f]).sum(), np.abs(ref[f]).max()
        print(f"  {what} {f}: L1 {d.sum() / s1:.2e} Linf {d.max() / si:.2e}", flush=True)
        assert d.sum() <= l1 * s1 and d.max() <= linf * si, (what, f)


def run_pair(grid, params, steps, change=None, noise=1.0e-4):
    d = abi.init_disk(grid, params, 3, noise)
    o = oracle.OracleDisk(grid, params, 3, noise)
    if change:
        change(d)
        change(o)
    st = o.run_begin()
    o.run(steps, st)
    with abi.Context(grid, params, abi.PN_FP64) as ctx:
        ctx.load(d)
        gst = ctx.run_begin()
        ctx.run(steps, gst)
        got = ctx.store()
    assert np.array_equal(got["rot_j"], o.rings["rot_j"])
    return got, o.rings


# last windows of 64 (52 and 168 rings), 65 (53, 169) and 13 cells (117); columns 0..7 past a
# multiple of 8
@pytest.mark.parametrize("nr,nphi", [(52, 104), (53, 101), (168, 97), (169, 106), (117, 99), (40, 13), (300, 143)])
@pytest.mark.parametrize("visc", [0, 1])
def test_radial_windows(nr, nphi, visc):
    print("case: radial windows", nr, nphi, "visc", visc, flush=True)
    over = {"visc_flag": 1, "ss_alpha": 3.0e-3, "vis_nu": 7.5e-6} if visc else {}
    got, ref = run_pair(abi.PnGrid(nr, nphi, 1), configs.disk2d(nr, nphi, **over), 5)
    close(got, ref, "ruv", 1.0e-11, 1.0e-8, f"{nr}x{nphi}")


@pytest.mark.parametrize("nth", [51, 52, 53, 120])
def test_theta_windows(nth):
    print("case: theta windows", nth, flush=True)
    got, ref = run_pair(abi.PnGrid(16, 37, nth), configs.c3().params.replace(zmin=1.42, zmax=1.72), 3)
    close(got, ref, "ruv", 1.0e-10, 1.0e-7, f"theta {nth}")
    # v_theta: the area factor (cos x0 - cos x) / (x - x0) of an edge moved by d = dt w / r carries
    # 2^-52 / d of the rounding of its cosines, so a step adds c_s^2 / (r dtheta) dt 2^-52 / d =
    # c_s^2 / dtheta 2^-52 / w to w; c_s^2 <= 0.0025 / 0.4, w its mean size
    size = np.abs(ref["w"]).mean()
    bar = 3 * (0.0025 / 0.4) / (0.3 / nth) * 2.0 ** -52 / size
    err = np.abs(got["w"] - ref["w"]).mean()
    print(f"  theta {nth} w: mean error {err:.2e}, bar {bar:.2e}", flush=True)
    assert err <= bar


def test_state_with_w_in_2d():
    """A 2-D state that carries w: it is advected by every sweep, packed windows included."""
    print("case: 2-D with w", flush=True)

    def add_w(d):
        for a in (d.rings, d.lft, d.rgh):
            a["w"] = 0.01 * a["r"]

    got, ref = run_pair(abi.PnGrid(130, 91, 1), configs.disk2d(130, 91), 5, add_w)
    close(got, ref, "ruvw", 1.0e-11, 1.0e-8, "w")


def test_stretched_azimuth():
    print("case: stretched azimuth", flush=True)
    nphi = 144
    edges = np.linspace(0.0, 2.0 * np.pi, nphi + 1)
    edges = edges + 0.2 / nphi * np.sin(3.0 * edges) * 2.0 * np.pi

    def stretch(d):
        for a in (d.rings, d.lft, d.rgh):
            a["y"] = edges[:-1]
            a["dy"] = np.diff(edges)
            a["yc"] = edges[:-1] + 0.5 * np.diff(edges)
            a["yvol"] = np.diff(edges)

    got, ref = run_pair(abi.PnGrid(48, nphi, 1), configs.disk2d(48, nphi, fargo_flag=0), 5, stretch)
    close(got, ref, "ruv", 1.0e-11, 1.0e-8, "stretched")


def test_coarse_rings_and_large_jumps():
    """24 columns and 1-in-2 density noise: turns past the sine series, jumps past the interface's
    (both take the library functions)."""
    print("case: coarse rings, large jumps", flush=True)
    p = configs.disk2d(20, 24, q=1.0e-3)
    got, ref = run_pair(abi.PnGrid(20, 24, 1), p, 5, noise=0.5)
    close(got, ref, "ruv", 1.0e-11, 1.0e-8, "jumps")


# jumps within the interface's series (1/8), on both sides of it in one wavefront, and far past it;
# bars of test_gpu_parity_flags.py's 10 steps of these closures
@pytest.mark.parametrize("eos", [2, 3])
@pytest.mark.parametrize("noise", [0.02, 0.15, 0.5])
def test_gamma_law_jumps(eos, noise):
    print("case: gamma-law jumps, eos", eos, "noise", noise, flush=True)
    p = configs.disk2d(50, 90, q=1.0e-3, eos=eos, gam=1.4, init_p_iso=1)
    got, ref = run_pair(abi.PnGrid(50, 90, 1), p, 5, noise=noise)
    close(got, ref, "rpuv", 1.0e-10, 1.0e-8, f"eos {eos}")
