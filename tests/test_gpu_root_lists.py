"""Root lists built tile by tile in LDS, at the edges of what that takes, bit for
bit against the oracle: rows of 8, 16 and 32 neighbours and one more (the bits per
vertex change, or the general way takes over), V sides that end just before, at
and after a tile (3,072, 1,536 and 768 vertices in a 7 KB arena), arenas too small
for it, few and many different bitsets (the table holds 224), and graphs without
neighbourhoods that fill a tile."""
import numpy as np
import pytest

import oracle
from gmbe_amd import BiGraph, enumerate_graph

pytestmark = pytest.mark.gpu


def _graph(nV, heavy, light, seed, nU=40, n_heavy=24):
    """nV rows over nU columns: n_heavy rows of `heavy` entries among rows of `light`."""
    rng = np.random.default_rng(seed)
    rows = [sorted(rng.choice(nU, light, replace=False).tolist()) for _ in range(nV)]
    for v in rng.choice(nV, n_heavy, replace=False):
        rows[v] = sorted(rng.choice(nU, heavy, replace=False).tolist())
    return BiGraph.from_rows(nU, rows).derive(uvtrans=0, order=1, fast_mode=1)


def _check(g, **knobs):
    r = enumerate_graph(g, **knobs)
    assert r.overflow == 0
    assert r.digest() == oracle.gmbe(g.oracle_graph(), threads=8).digest()


@pytest.mark.parametrize("nV", [767, 768, 769, 1536, 1537, 3071, 3072, 3073, 6145])
@pytest.mark.parametrize("heavy", [8, 9, 16, 17, 32, 33])
def test_tiles(gpu, heavy, nV):
    _check(_graph(nV, heavy, 2, 1000 * heavy + nV))


@pytest.mark.parametrize("lds_kb", [0, 3, 7, 16])
def test_arenas(gpu, lds_kb):
    _check(_graph(2000, 12, 3, 5), lds_kb=lds_kb)


@pytest.mark.parametrize("light", [1, 3, 6])
def test_many_bitsets(gpu, light):
    _check(_graph(900, 14, light, 11, nU=30))


@pytest.mark.parametrize("knobs", [dict(group=0), dict(dom_skip=0), dict(recompute=1), dict(share=0)])
def test_general_way(gpu, knobs):
    _check(_graph(1000, 16, 3, 7), **knobs)


def test_thin_rows(gpu):
    """20,000 rows of one entry in groups of two: every tile holds almost nothing."""
    rows = [[i // 2] for i in range(20000)] + [[0, 9999], [5, 5000, 9998]]
    _check(BiGraph.from_rows(10000, rows).derive(uvtrans=0, order=1, fast_mode=1))
