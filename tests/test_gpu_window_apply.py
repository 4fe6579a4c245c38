"""The slice launch's update of G when a workgroup owns one or several 64 x 64 tiles (several from
129 tiles on), and a ragged last tile, gives the chain of one launch per window (one tile per
workgroup) bit for bit.  Runs across the boundary of the flavour blocks: test_gpu_tile_runs.py."""
import numpy as np
import pytest

from conftest import make_chain

pytestmark = pytest.mark.gpu


# (U > 0: one flavour)  n = 576: 81 tiles, one per workgroup; n = 729 (ragged), two flavours: 288
# tiles in runs of 3 down columns of 12; n = 784 (ragged): 169 tiles in runs of 2 across columns of 13
@pytest.mark.parametrize("L,U,W", [(24, 4.0, 32), (27, -4.0, 16), (28, 4.0, 0)])
def test_runs_of_tiles_equal_single_tiles(pkg, hip, L, U, W):
    chains = []
    try:
        for one in (True, False):
            g, model, par, field = make_chain(hip.HIPChain, pkg, L, U, 0.4, seed=3, delay_depth=W)
            chains.append(g)
            g.set_hopping(model.hopping_matrix())
            g.set_field(field.conf)
            g.set_seed(17)
            g.set_slice_launch(one)
            g.build_stack()
        gs, gw = chains
        for it in range(2):
            assert gs.sweep(1) == gw.sweep(1), it
            assert np.array_equal(gs.get_field(), gw.get_field()), it
            assert np.array_equal(gs.greens(), gw.greens()), it
        assert gs.counters()["device_errors"] == 0
    finally:
        for c in chains:
            c.close()
