"""Chains on both sides of the sizes where rdivp changes its kernel (256, 512, 640 sites) in one
batch: each gives what it gives alone, bit for bit."""
import numpy as np
import pytest

from conftest import make_chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[(8, -4.0), (24, 4.0), (16, 4.0)], [(20, -4.0), (26, -4.0), (24, 4.0), (6, 3.0)]])
def test_batch_of_small_and_large_chains_equals_chains_alone(pkg, hip, sizes):
    def mk(k, L, U):
        g, model, par, field = make_chain(hip.HIPChain, pkg, L, U, 0.8, safe_mult=4, seed=7 + k)
        g.set_hopping(model.hopping_matrix())
        g.set_field(field.conf)
        g.set_seed(70 + k)
        g.build_stack()
        return g

    alone, chains = [], []
    for k, (L, U) in enumerate(sizes):
        g = mk(k, L, U)
        acc = g.sweep(2)
        alone.append((acc, g.get_field(), g.greens()))
        g.close()
    try:
        for k, (L, U) in enumerate(sizes):
            chains.append(mk(k, L, U))
        accs = hip.batch_sweep(chains, 2)
        for (acc, f, G), g, a in zip(alone, chains, accs):
            assert a == acc
            assert np.array_equal(g.get_field(), f)
            assert np.array_equal(g.greens(), G)
    finally:
        for g in chains:
            g.close()
