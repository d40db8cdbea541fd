"""The disk's pull on a moving planet: one pass over the state after each step's sweeps takes both
force sums, the damping zones and the place of the integer roll."""
from __future__ import annotations

import pytest

from penguin_2_0_amd import abi, configs

pytestmark = pytest.mark.gpu

SIGMA0 = 1.0 * 0.00019126835


def say(*a):
    print(*a, flush=True)


# rings of less than, exactly, just over and several of a workgroup's 256 columns; more than 2048
# slots (the roll in a launch of its own); more ring runs than partial sums
@pytest.mark.parametrize("prec", [abi.PN_FP64, abi.PN_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("kill", [0, 1])
@pytest.mark.parametrize("nr,nphi", [(40, 97), (33, 256), (33, 257), (60, 601), (2100, 24), (4200, 12)])
def test_forces_are_the_reductions_of_the_stored_state(nr, nphi, kill, prec):
    """After a step the planet's forces are those of modes 8 and 9 over the state it leaves: the
    sums differ by their order alone, a few tens of 2^-53 of the sum of magnitudes, which 1e-9 of
    the larger force covers a thousandfold."""
    w = configs.small(nr, nphi, plnt_flag=2, kill_flag=kill, M_p=1e-3, t_growth=0.0)
    d = abi.init_disk(w.grid, w.params, w.seed, w.noise)
    say("case: planet torque", nr, nphi, "kill", kill, "precision", prec)
    with abi.Context(w.grid, w.params, prec) as ctx:
        ctx.load(d)
        st = ctx.run_begin()
        ctx.run(3, st, graph=False)
        p = st.planet
        # the closing half kick has added fy to the planet's rate
        rate = p.vy + st.FrRot - 0.5 * st.dt * p.fy / p.x ** 2
        f8 = (p.fx + 1.0 / p.x ** 2 - p.x * rate ** 2) * p.m / SIGMA0
        f9 = p.fy * p.m / SIGMA0
        r8, r9 = ctx.reduce(p, 0.0, 8), ctx.reduce(p, 0.0, 9)
        say(f"  radial {f8!r} mode 8 {r8!r}; azimuthal {f9!r} mode 9 {r9!r}")
        tol = 1e-9 * max(abs(r8), abs(r9))
        assert abs(f9 - r9) <= tol
        assert abs(f8 - r8) <= tol + 1e-15 * p.m / SIGMA0   # 1/x^2 and x rate^2 are near 1
