"""Runs of 64 x 64 tiles in the slice launch's update of G that cross a column of tiles and the
boundary between the two flavour blocks give the chain of one launch per window (one tile per
workgroup) bit for bit."""
import numpy as np
import pytest

from conftest import make_chain

pytestmark = pytest.mark.gpu


def runs(n, flavors, workgroups=128):
    """Tiles per column, per block, and the runs [t0, t1) of the application workgroups."""
    nt = -(-n // 64)
    tiles = flavors * nt * nt
    per = -(-tiles // min(tiles, workgroups))
    return nt, nt * nt, [(t, min(t + per, tiles)) for t in range(0, tiles, per)]


# n = 576: 162 tiles in runs of 2 over columns of 9; n = 676 (ragged): 242 in runs of 2 over
# columns of 11; n = 784 (ragged): 338 in runs of 3 over columns of 13
@pytest.mark.parametrize("L,W", [(24, 32), (26, 16), (26, 32), (28, 16), (28, 0)])
def test_runs_across_columns_and_blocks_equal_single_tiles(pkg, hip, L, W):
    chains = []
    try:
        for one in (True, False):
            g, model, par, field = make_chain(hip.HIPChain, pkg, L, -4.0, 0.4, seed=3, delay_depth=W)
            chains.append(g)
            assert field.flavors == 2
            g.set_hopping(model.hopping_matrix())
            g.set_field(field.conf)
            g.set_seed(17)
            g.set_slice_launch(one)
            g.build_stack()
        column, block, rs = runs(L * L, 2)
        assert any(t0 // column != (t1 - 1) // column for t0, t1 in rs)
        assert any(t0 < block < t1 for t0, t1 in rs)
        gs, gw = chains
        for it in range(2):
            assert gs.sweep(1) == gw.sweep(1), it
            assert np.array_equal(gs.get_field(), gw.get_field()), it
            assert np.array_equal(gs.greens(), gw.greens()), it
        assert gs.counters()["device_errors"] == 0
    finally:
        for c in chains:
            c.close()
