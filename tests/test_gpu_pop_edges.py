"""Pair branching's plan on either side of its two sorts (up to 1024 walkers ranks, more
a bitonic sort) and of its slots per thread, against the oracle, and weights that are
infinite: the map stays within the walkers."""

import numpy
import pytest

from oracle import pop_control as pc
from tests.test_gpu_pop import WTOL, _ctx, _plan, _rel, _weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw", [1, 3, 63, 65, 1023, 1025, 2049, 3500])
@pytest.mark.parametrize("kind", ["lognormal", "ties"])
def test_pair_branch_at_the_edges(nw, kind):
    print(f"[case] pair branch nw={nw} {kind}", flush=True)
    w = _weights(nw, 11 + nw, kind)
    u = numpy.random.RandomState(nw).rand(max(nw // 2, 1))
    src, nwt, total, npairs = _plan(_ctx(), "pair_branch", w, nw, u)
    tot, _, scaled = pc.rescale(w, nw)
    osrc, onw, opairs = pc.pair_branch_plan(scaled, 0.1, 4.0, u)
    assert npairs == opairs and numpy.array_equal(src, osrc)
    assert _rel(nwt, onw) <= WTOL and abs(total - tot) <= WTOL * abs(tot)


@pytest.mark.parametrize("nw", [64, 1100])
def test_infinite_weights_keep_the_map_in_range(nw):
    print(f"[case] infinite weights nw={nw}", flush=True)
    w = _weights(nw, 3, "lognormal")
    w[5] = numpy.inf
    src, _, _, _ = _plan(_ctx(), "pair_branch", w, nw, numpy.random.RandomState(1).rand(nw // 2))
    assert src.min() >= 0 and src.max() < nw
