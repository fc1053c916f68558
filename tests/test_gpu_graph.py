"""The graph stage at the sizes where its two forms begin and end (one workgroup up to
4,096 states, passes over sub-cubes of 64 beyond), bit for bit against the oracle."""
import numpy as np
import pytest

from oracle import pipeline as P
from oracle.bnet import read_bnet_text
from paraexastolog_amd import model_builder, synth, transition_graph, transition_table

pytestmark = pytest.mark.gpu

TINY = {"one": "targets, factors\nA, !A\n", "two": "targets, factors\nA, B\nB, !A\n",
        "three": "targets, factors\nA, B & C\nB, A | !C\nC, C\n"}
# nodes, inputs per node, seed, fixed nodes
NETS = [(4, 2, 0, 0), (6, 2, 1, 0), (7, 2, 2, 0), (10, 2, 1, 0), (10, 2, 3, 0), (11, 0, 5, 5), (12, 0, 1, 5), (13, 2, 4, 0),
        (13, 0, 3, 5), (14, 2, 0, 0), (14, 0, 2, 5), (15, 2, 3, 0), (15, 0, 2, 5)]


def check(ctx, text, rates):
    om = read_bnet_text(text)
    pm = model_builder().parse_model(text)
    t = transition_table(ctx, pm, rates)
    t.construct_table()
    g = transition_graph(ctx, t)
    g.reorganize_vertices()
    n = 1 << om.n_nodes
    ip, rows, cols = P.transition_table(om, rates)
    reord, off, T, ids = P.transition_graph(n, ip, rows)
    np.testing.assert_array_equal(g.scc_ids, ids)
    np.testing.assert_array_equal(g.reordered_vertices, reord)
    np.testing.assert_array_equal(g.sccs_offsets, off)
    assert g.terminals_count == T
    assert g.max_height == int(P.scc_heights(n, ip, rows, ids)[1].max())
    c = g.stage_counts()
    assert c["scc_rounds"] >= 1 and c["mask_passes"] > c["scc_rounds"] and c["host_round_trips"] >= 1


@pytest.mark.parametrize("name", sorted(TINY))
def test_tiny(ctx, name):
    N = TINY[name].count("\n") - 1
    check(ctx, TINY[name], np.ones(2 * N))


@pytest.mark.parametrize("N,K,seed,fixed", NETS)
@pytest.mark.parametrize("zeros", [0, 3])
def test_graph_bit_exact(ctx, N, K, seed, fixed, zeros):
    net, rng = synth.generate(N, K, seed, fixed)
    rates = synth.rate_sets(rng, N, 1)[0]
    rates[np.random.default_rng(seed).choice(2 * N, zeros, replace=False)] = 0.0  # edges taken out
    check(ctx, net.bnet(), rates)
