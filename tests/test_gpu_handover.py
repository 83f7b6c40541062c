"""Entries handed to waiting waves, bit for bit against the oracle: one block (its
own waves are all that can wait), a full grid, and queues of two slots a shard,
where what no waiting wave takes may not fit and runs where it is.  Nodes have
fewer items than an entry holds (15), about as many, and far more."""
import pytest

import graphs
import oracle
from gmbe_amd import enumerate_graph

pytestmark = pytest.mark.gpu

EAGER = dict(late_share=1, share_work=1, share_queue=1 << 30)


@pytest.mark.parametrize("knobs", [dict(), dict(blocks=1), dict(blocks=1, queue_log2=6),
                                   dict(queue_log2=6), dict(ctx_slots=1)])
@pytest.mark.parametrize("nU,nV,p", [(12, 16, 0.5), (40, 60, 0.3), (80, 400, 0.08), (200, 150, 0.1)])
def test_handover(gpu, nU, nV, p, knobs):
    g = graphs.random_graph(nU, nV, p, 31 + nV).derive(uvtrans=0, order=1, fast_mode=1)
    r = enumerate_graph(g, **EAGER, **knobs)
    assert r.overflow == 0
    assert r.digest() == oracle.gmbe(g.oracle_graph(), threads=8).digest()
