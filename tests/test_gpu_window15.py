"""16-site windows whose last one has 15 sites (rings of 15, 31 and 47 sites), against the oracle:
one and two flavours, supplied uniforms and the counter stream."""
import numpy as np
import pytest

from conftest import assert_same_decisions, counter_stream, make_chain, rel_maxdiff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,U", [(15, 4.0), (15, -4.0), (31, 4.0), (31, -4.0), (47, -3.0)])
@pytest.mark.parametrize("stream", ["supplied", "counter"])
def test_last_window_of_15_sites_matches_the_oracle(pkg, hip, oracle, n, U, stream):
    kw = dict(lattice=pkg.Chain(n), seed=5)
    g, model, par, field = make_chain(hip.HIPChain, pkg, n, U, 1.5, delay_depth=16, **kw)
    o, *_ = make_chain(oracle.OracleChain, pkg, n, U, 1.5, **kw)
    assert len(model.l) == n and n % 16 == 15
    o.set_hopping(model.hopping_matrix())
    g.set_hopping_exp(*o.get_hopping_exp())
    cap = 2 * n * par.slices
    u = np.random.default_rng(31).random(cap) if stream == "supplied" else counter_stream(77, cap)
    for c in (g, o):
        c.set_field(field.conf)
        if stream == "supplied":
            c.set_uniforms(u)
        else:
            c.set_seed(77)
        c.set_log(cap)
        c.build_stack()
    ag, ao = g.sweep(1), o.sweep(1)
    (dg, pg), (do, po) = g.get_log(), o.get_log()
    if assert_same_decisions(dg, do, po, u):
        assert ag == ao and np.array_equal(g.get_field(), o.get_field())
        assert rel_maxdiff(g.greens(), o.greens()) < 1e-10
        assert g.counters()["uniforms_used"] == o.counters()["uniforms_used"]
    assert g.counters()["device_errors"] == 0
    g.close()
    o.close()
