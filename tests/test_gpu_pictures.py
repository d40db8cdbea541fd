"""Pictures fetched in pieces: the records of pn_store_rings against the state that was loaded,
at sizes where a piece holds one ring, ends inside a theta row, or spans rows with their ghost
slots, and small disks that fit one piece.  FP64 records come back byte for byte; FP32 ones hold
the background plus the deviation rounded once."""
from __future__ import annotations

import numpy as np
import pytest

from penguin_2_0_amd import abi, configs

pytestmark = pytest.mark.gpu

# (rings, columns, theta rows): one ring a piece (a ring of 150001 columns is 6 MB staged); a
# 3-D disk of several pieces that end inside rows; rows of one piece; one small piece
SIZES = [(3, 150001, 1), (24, 73, 41), (300, 128, 3), (13, 12, 1)]


def disk(nr, nphi, nth, **over):
    if nth > 1:
        p = configs.c3().params.replace(**over)
    else:
        p = configs.disk2d(nr, nphi, **over)
    grid = abi.PnGrid(nr, nphi, nth)
    d = abi.init_disk(grid, p, 11, 1.0e-4)
    rng = np.random.default_rng(5)
    for f in ("u", "v") + (("w",) if nth > 1 else ()):
        d.rings[f] += 1.0e-3 * rng.standard_normal(d.rings[f].shape)
    d.rings["rot_j"] = rng.integers(0, nphi, len(d.rings))
    d.rings["inc_j"] = rng.integers(-3, 4, len(d.rings))
    d.rings["rot_v"] = rng.standard_normal(len(d.rings))
    d.rings["res_v"] = rng.standard_normal(len(d.rings))
    return grid, p, d


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_fp64_pictures_are_the_loaded_bytes(size):
    print("case: FP64 picture", size, flush=True)
    grid, p, d = disk(*size)
    with abi.Context(grid, p, abi.PN_FP64) as ctx:
        ctx.load(d)
        assert np.array_equal(ctx.store().view(np.uint8), d.rings.view(np.uint8))
        if size[2] == 1:   # a state with w has a fifth field to fetch, in the same staging buffer
            d.rings["w"] = 1.0
            ctx.load(d)
            assert np.array_equal(ctx.store().view(np.uint8), d.rings.view(np.uint8))


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("eos", [0, 3])
def test_fp32_pictures_round_the_deviations_once(size, eos):
    if eos == 3 and size[2] > 1:
        pytest.skip("EOS 3 is a 2-D closure")
    print("case: FP32 picture", size, "eos", eos, flush=True)
    grid, p, d = disk(*size, **({"eos": 3, "gam": 1.4, "init_p_iso": 1} if eos else {}))
    bg = d.val_array()
    with abi.Context(grid, p, abi.PN_FP32) as ctx:
        ctx.load(d)
        got = ctx.store()

    def rounded(x):
        return x.astype(np.float32).astype(np.float64)

    want = d.rings.copy()
    rb, pb, vb = (bg[:, n, None] for n in (0, 1, 3))
    want["r"] = rb + rounded(d.rings["r"] - rb)
    want["u"] = rounded(d.rings["u"])
    want["v"] = vb + rounded(d.rings["v"] - vb)
    want["w"] = rounded(d.rings["w"])
    if eos == 3:
        qb = pb / rb
        want["p"] = want["r"] * (qb + rounded(d.rings["p"] / d.rings["r"] - qb))
        assert np.array_equal(got["p"], want["p"])
    else:   # c_s^2 Sigma, c_s^2 from libm's pow
        assert np.allclose(got["p"], d.rings["p"], rtol=1.0e-6, atol=0.0)
        want["p"] = got["p"]
    assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
