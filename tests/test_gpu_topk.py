"""The device's top-k selection where its bound can go wrong: fewer candidates
than slots, waves and blocks without any, all scores equal (the ids decide),
the best scores all in one lane's entries or in a few lanes' and quads', and counts at the edges of a block's
2048 entries and of a second level of blocks.  Ids and scores bit for bit
against the oracle."""
import numpy as np
import pytest

from oracle import oracle as orc
import three_llm_amd.tlm as tlm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = tlm.Context(0)
    yield c
    c.close()


def scores(kind, n):
    rng = np.random.default_rng(n)
    if kind == "equal":
        return np.full(n, -1.5, np.float32)
    if kind == "ascending":
        return np.arange(n, dtype=np.float32)
    if kind == "one lane":  # every 64th entry, four blocks' worth of waves
        x = rng.standard_normal(n).astype(np.float32)
        x[::64] += 100
        return x
    if kind == "few":  # three candidates, the rest never take part
        x = np.full(n, -np.inf, np.float32)
        x[1::2] = np.nan
        x[[0, n // 2, n - 1]] = [-3.0, 2.0, 2.0]
        return x
    if kind.startswith("first"):  # scores in the first lanes of every 64 alone
        x = rng.standard_normal(n).astype(np.float32)
        x[np.arange(n) % 64 >= int(kind.split()[1])] = -np.inf
        return x
    if kind == "random":
        return rng.standard_normal(n).astype(np.float32)
    return np.full(n, -np.inf, np.float32)


@pytest.mark.parametrize("kind", ["equal", "ascending", "one lane", "few", "none"])
@pytest.mark.parametrize("n,k", [(5, 16), (64, 16), (2047, 3), (2049, 1), (4096, 16), (262145, 16)])
def test_topk_selection_edges(ctx, kind, n, k):
    x = scores(kind, n)
    assert tlm.topk(ctx, ctx.array(x), n, k) == orc.topk_candidates(x, k)


@pytest.mark.parametrize("kind", ["random", "first 60", "first 15", "first 12", "first 1", "ascending", "equal"])
@pytest.mark.parametrize("n,k", [(600, 16), (2048, 9), (32000, 4), (151936, 8), (151936, 16), (262144, 16)])
def test_topk_where_the_quads_bound_is_a_loose_one(ctx, kind, n, k):
    """Fewer quads (or lanes) than k hold a score, or the merged lists' ranks fall
    on the same quads: a closer bound from the lanes, the same result."""
    x = scores(kind, n)
    assert tlm.topk(ctx, ctx.array(x), n, k) == orc.topk_candidates(x, k)
