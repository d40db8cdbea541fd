"""The FP32 sweeps round where they always have.

A disk's flow amplifies roundings (a start nudged by 1e-9 has moved v_r by 2e-3 after 3000 steps of
1024 x 3072), so two builds whose FP32 operations round differently show different disks in long
runs, without either being wrong by more than its own noise.  The words below are v_r of 24 cells
per disk as the sweeps left them before their divisors were taken as table reciprocals and their
limiters rewritten (EOS 3: with the quotients of its interface states corrected, which that form
had not); a sweep that rounds one operation otherwise changes most of them within these
steps.  Three quarters have to agree: a host whose libm rounds an entry of the tables otherwise
moves single cells."""
from __future__ import annotations

import numpy as np
import pytest

from penguin_2_0_amd import abi, configs

pytestmark = pytest.mark.gpu

HPI = 1.570796326794896619231321691639751442
VISC = dict(visc_flag=1, ss_alpha=3.0e-3, vis_nu=7.5e-6)
ADIA = dict(eos=3, gam=1.4, init_p_iso=1)


def flat(nr, nphi, **over):
    return abi.PnGrid(nr, nphi, 1), configs.disk2d(nr, nphi, q=1.0e-4, **over)


def ball(nr, nphi, nth, **over):
    p = configs.disk2d(nr, nphi, q=3.0e-5, **over)
    return abi.PnGrid(nr, nphi, nth), p.replace(ndim=3, ngeomx=2, ngeomy=4, ngeomz=5, p_alpha=1.5, p_beta=1.0,
                                                zmin=HPI - 0.15, zmax=HPI + 0.15)


# disk, steps, a density step of this height, radial and azimuthal variants
CASES = {
    "isothermal": (flat(125, 353), 40, 1.0, (0, 1)),
    "isothermal, long azimuthal windows": (flat(200, 601), 40, 1.0, (3, 3)),
    "viscous": (flat(117, 353, **VISC), 40, 1.0, (0, 0)),
    "adiabatic": (flat(96, 288, **ADIA), 40, 1.0, (0, 2)),
    "adiabatic, viscous": (flat(153, 276, **ADIA, **VISC), 40, 1.0, (1, 1)),
    "barycentric": (flat(100, 300, bary_flag=1), 40, 1.0, (2, 0)),
    "shocks": (flat(70, 200), 20, 3.0, (0, 1)),
    "adiabatic shocks": (flat(140, 200, **ADIA), 20, 9.0, (0, 1)),
    "spherical": (ball(48, 144, 20), 20, 1.0, (0, 1)),
    "spherical, viscous": (ball(40, 96, 53, **VISC), 20, 1.0, (3, 1)),
    "spherical shocks": (ball(40, 96, 24), 12, 3.0, (0, 1)),
}

PINS = {
    "isothermal":
        "55fb02b951b2a2ba113e1a398c4e0839151d6e390e41ec369ff29c384d3141b8a058d0b8621526b9fecb6db6d75da438"
        "f5fbf138217d85388350fdb7091150b7c756f93882fde03873d69b38b5b4e3386f8dea38d25204391afbd2382f2537b7",
    "isothermal, long azimuthal windows":
        "66652338158dd6b8e14a94b8a2a9e33756ff3cb98870e938e7f361b8540af4b76faa89b82a14bab837a08c381e9920b9"
        "f9544bb5aa53afb89f4781385fd296381498e8b8b204c636796d863841f1a838cd76d6b8e9c85d3730ff873684a30138",
    "viscous":
        "953da1b9e0152bb962501039489204b9afc822b9d4e4a9375f2df0b8789d4238151308b96e22063724bd0b39ddddbab8"
        "11710939701b1339400668b997ad30b90e8f1039175eacb9773a92bbcc5aebb87c1960baa64d88b9e5f726b9202e6838",
    "adiabatic":
        "acc034b9b52f3238d6f477b73a2a9db81b932fba2e83bc38c45455b99c4263b8d9adf0b81179d938f30c1eb96d1646b9"
        "f3746bb8ad3e2db9980c5c374f7407391e51ccb962c01ab928c0fc38397d11375927ea38122f02b9e8eb2db95752a1b8",
    "adiabatic, viscous":
        "d78e6738255c55ba4f7eacb88d8c43383f92ccb8411b8fb887f52038137c5d370252af3716b0f8b800ff08b9f99921b9"
        "04219d3790ed8e3832e71eb98644eeb9d9dec5379b3886b8f7dc87b85594a2389a66a539dbc866b744238db8cde0b8b8",
    "barycentric":
        "4915c6b77dc112b90ea156b95c4e71b8be131839149341b65873d437567b1cb92bc5d0b9daaecf37f216ed3743a84bb7"
        "5bd19f39dc9445bafe61b3b653363fb6298cc3b8d32fd1399c7cfeb837272b379fae2239c3580cb94a4294b8f77bf238",
    "shocks":
        "804f89b92410c9bac6d1bc3823d2c237bdb8833ba6a6e1362e6f4db9d8ddb6b83c569939c5e1ed38d7fd843c22fad538"
        "612dc3bcd836ffb60423a8385fc8b638bf3bc7b897bda13752cde1ba6ccc03b98ef160bc51ba7e38aa27fc386dc55bb8",
    "adiabatic shocks":
        "e60b4638ee4efeb69288abb954ea1938b6a9c1b71211f637f074b3b833cc883811b292b867db4b37e2c54438f8736bb7"
        "fcafe43c00f34238c5cdee3792c93c37daf604bafc495f379d7085b8297103388ab938380de08f3712004738f1d956b7",
    "spherical":
        "6199843900b9a5b850508f3880ee6c38813fe4b77e1eeb34375b1f379d8156381ec2b43657466338bbec54b79f038e37"
        "c32f9db7a2dd2337059f54387aefc0b671891638c24b2a37ed100fb754c19836008c253679e5de378c4a3b3824d851b9",
    "spherical, viscous":
        "200dbe3763dfb3b7fe4d093864539537a060a9b48368d9376218ecb7a4cad8b6aa8aa8372ce0e437756b4136f0bb3437"
        "2e065db73602dd371200173712c94eb88b4b44b76acf12b86e0adeb577c069b720d144b522031537592d09b7ee6bc037",
    "spherical shocks":
        "bdf9efb6b61415ba7b27b2371b0dc737ecd6773b634c10b7cfd80333a4bace37ca76c537692b2c37f7792eb85469deb5"
        "5c618738f35af6b56e360938b417c9351d4d0638577cc937bafdea3b40128e361f61e63b493bc8ba540ee437f96b5837",
}


def state(name):
    (grid, params), steps, jump, variants = CASES[name]
    d = abi.init_disk(grid, params, 7, 1.0e-4)
    rows = np.arange(grid.imax * grid.kmax) % grid.imax
    rows = (rows > grid.imax // 3) & (rows < 2 * grid.imax // 3)
    for f in ("r", "p"):
        d.rings[f][np.ix_(rows, np.arange(grid.jmax // 4, grid.jmax // 2))] *= jump
    with abi.Context(grid, params, abi.PN_FP32) as ctx:
        ctx.load(d)
        ctx.set_variants(*variants)
        st = ctx.run_begin()
        ctx.run(steps, st)
        u = ctx.store()["u"].ravel()
    return u[np.random.default_rng(0).integers(0, u.size, 24)].astype(np.float32)


@pytest.mark.parametrize("name", CASES)
def test_sweeps_round_where_they_did(name):
    print("case: FP32 rounding,", name, flush=True)
    got = state(name)
    want = np.frombuffer(bytes.fromhex(PINS[name]), "<f4")
    same = int((got.view(np.uint32) == want.view(np.uint32)).sum())
    print(f"  {same} of 24 cells with the same word, largest difference {np.abs(got - want).max():.1e}", flush=True)
    assert same >= 18
