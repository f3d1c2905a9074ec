"""tlm_op_logits: the token is picked by the last block to finish or by a merge
kernel, so what is checked is the choice across blocks (ties, nothing above the
lowest score) and that one call leaves the next one a clean start."""
import numpy as np
import pytest

import three_llm_amd.tlm as tlm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = tlm.Context(0)
    yield c
    c.close()


# up to 128 blocks and from 128 MiB of weights on: the last block; between: the merge
@pytest.mark.parametrize("V", [1, 64, 65, 8192, 8193, 40000, 1050000])
def test_token_across_blocks(ctx, V):
    rng = np.random.default_rng(V)
    K = 64
    w = (rng.integers(-4, 5, (V, K)) / 8.0).astype(np.float16)
    best = sorted(rng.choice(V, min(V, 3), replace=False))
    w[best] = 1.0  # three equal rows, the best for x = ones: the lowest id wins
    L = tlm.Linear(ctx, tlm.FMT_F16, np.ascontiguousarray(w.view(np.uint16)))
    out, tok = ctx.buffer(4 * V), ctx.buffer(4)
    for x, token in ((np.ones(K), best[0]), (np.full(K, np.nan), 0), (np.full(K, -np.inf), None),
                     (-np.ones(K), None), (np.ones(K), best[0])):
        tlm.logits(L, ctx.array(x.astype(np.float32)), out, tok)
        lg = out.read()[:V]
        if token is None:  # the lowest id of the device's best score, 0 when there is none
            s = np.where(np.isnan(lg), -np.inf, lg)
            token = int(np.argmax(s)) if s.max() > -np.inf else 0
        assert int(tok.read(np.int32)[0]) == token
    L.close()
