"""Subtrees whose lists fit the register machine (at most 64 entries, |L| at
most 64) at the edges of what it takes, bit for bit against the oracle: lists
and L of 63, 64 and 65, alone and with every node handed to other waves."""
import pytest

import graphs
import oracle
from gmbe_amd import enumerate_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("knobs", [dict(), dict(late_share=1, share_work=1, share_queue=1 << 30),
                                   dict(prune=0), dict(dom_k=1)])
@pytest.mark.parametrize("nU,nV,p", [(2, 70, 0.6), (63, 64, 0.2), (64, 65, 0.2), (65, 66, 0.2),
                                     (64, 130, 0.12), (130, 65, 0.3), (300, 40, 0.3)])
def test_short_lists(gpu, nU, nV, p, knobs):
    g = graphs.random_graph(nU, nV, p, 77 + nU).derive(uvtrans=0, order=1, fast_mode=1)
    r = enumerate_graph(g, **knobs)
    assert r.overflow == 0
    assert r.digest() == oracle.gmbe(g.oracle_graph(), threads=8).digest()
