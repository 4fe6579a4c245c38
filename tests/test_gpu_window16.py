"""16-site windows against the oracle: last windows of 1, 2 and 9 sites (15 sites:
test_gpu_window15.py), one and two flavours, supplied uniforms (so that a ragged window reads its
own) and the counter stream."""
import numpy as np
import pytest

from conftest import assert_same_decisions, counter_stream, make_chain, rel_maxdiff

pytestmark = pytest.mark.gpu


# sites modulo 16: 3^2 -> 9, 7^2 -> 1, 9^2 -> 1, 5^2 -> 9, honeycomb 5 (50) -> 2, honeycomb 9 (162)
# -> 2, 13^2 -> 9
@pytest.mark.parametrize("L,U,lattice", [(3, 4.0, None), (7, -4.0, None), (9, 4.0, None), (5, -3.0, None),
                                         (5, 2.0, "honeycomb"), (9, -2.0, "honeycomb"), (13, 4.0, None)])
@pytest.mark.parametrize("stream", ["supplied", "counter"])
def test_ragged_windows_match_the_oracle(pkg, hip, oracle, L, U, lattice, stream):
    lat = pkg.Honeycomb(L) if lattice == "honeycomb" else None
    kw = dict(lattice=lat, seed=5)
    g, model, par, field = make_chain(hip.HIPChain, pkg, L, U, 1.5, delay_depth=16, **kw)
    o, *_ = make_chain(oracle.OracleChain, pkg, L, U, 1.5, **kw)
    o.set_hopping(model.hopping_matrix())
    g.set_hopping_exp(*o.get_hopping_exp())
    n, M = len(model.l), par.slices
    cap = 2 * n * M
    if stream == "supplied":
        u = np.random.default_rng(31).random(cap)
    else:
        u = counter_stream(77, cap)
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
