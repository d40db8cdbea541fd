"""A batch whose disks' packing changes between runs: the radial order is laid out anew, with another
number of slots, and the replayed step has to run all of them."""
from __future__ import annotations

import numpy as np
import pytest

from penguin_2_0_amd import abi, configs

pytestmark = pytest.mark.gpu


def test_packing_changed_between_runs_of_a_batch():
    """Four disks, radial variant 2: 312 slots without packing, 400 with it, and room for 616 after
    tuning (the other variants' order), so the order array stays where it is."""
    ws = [configs.small(nr, 3 * nr, M_p=q) for nr, q in ((128, 1e-3), (48, 1e-4), (256, 3e-4), (192, 1e-5))]
    disks = [abi.init_disk(w.grid, w.params, 200 + d, w.noise) for d, w in enumerate(ws)]
    out = []
    for graph in (True, False):
        print("case: packing changed between runs of a batch, graph", graph, flush=True)
        with abi.Batch([w.grid for w in ws], [w.params for w in ws]) as b:
            for ctx, d in zip(b.disks, disks):
                ctx.load(d)
                ctx.set_packing(False)
            b.tune(2)
            b.set_variants(2, 1)
            st = b.run_begin()
            for pack in (False, True, False, True):
                for ctx in b.disks:
                    ctx.set_packing(pack)
                b.run(6, st, graph=graph)
            out.append([(s.dt, ctx.store()) for s, ctx in zip(st, b.disks)])
    for d, ((ta, a), (tb, c)) in enumerate(zip(*out)):
        assert ta == tb, d
        assert np.array_equal(a.view(np.uint8), c.view(np.uint8)), d
