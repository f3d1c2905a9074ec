"""Batched chunks whose GEMMs pick 128-row tiles with K slices (q4) or the fp16
ring tiles, at ragged row counts, against the replayed decode graph: an
independent path with the tolerances of the batched prefill (fp16 activations)."""
import dataclasses

import numpy as np
import pytest

from bridge import close
import three_llm_amd.runner as R
import three_llm_amd.tlm as tlm
import three_llm_amd.weights as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,n", [(None, 1001), (None, 1901), ("f16", 65), ("f16", 700)])
def test_ragged_chunks_match_replay(storage, n):
    print(f"[prefill slices] {storage or 'q4'} linears, {n} rows", flush=True)
    layers, base = 2, W.WORKLOADS["llama-3.2-1b"]
    store = base.storage if storage is None else dataclasses.replace(base.storage, linear=storage)
    cfg = dict(base.config, num_hidden_layers=layers, vocab_size=4096)
    wl = W.Workload(base.name + "-2l", cfg, store, n + 1, 6, n + 8, qkv_bias=base.qkv_bias)
    ctx = tlm.Context(0)
    runner = R.DecoderHIPRunner(W.synthetic(wl), {"maxTokens": n + 8, "prefillChunkSize": 2048}, ctx=ctx)
    m = runner.model
    prompt = [int(t) for t in np.random.default_rng(n).integers(0, 4096, n + 1)]
    res = []
    for least in (0, 64):  # no batched chunk, then one
        m.reset_cache()
        m.set_prefill(least, 2048)
        m.prefill(prompt, 0, n)
        m.compute_token(prompt[-1], n, True)
        res.append((m.read_logits(), [a.view(np.float16).astype(np.float32) for l in range(layers)
                                      for a in m.kv_read(l, 0, n)]))
    (ref, ref_kv), (got, got_kv) = res
    for a, b in zip(got_kv, ref_kv):
        close(a, b, 2e-2, 1e-2)
    close(got, ref, 2e-2, 1e-2)
    runner.close()
    ctx.close()


@pytest.mark.parametrize("storage,hidden", [(None, 1024), (None, 512), ("f16", 1024)])
def test_short_chunk_of_a_wide_mlp_matches_replay(storage, hidden):
    """64 rows through gate|up of 2 x 32768: the tiles for few rows over many columns, with SwiGLU."""
    base, n = W.WORKLOADS["llama-3.2-1b"], 64
    store = base.storage if storage is None else dataclasses.replace(base.storage, linear=storage)
    cfg = dict(base.config, num_hidden_layers=2, vocab_size=512, hidden_size=hidden, intermediate_size=32768,
               num_attention_heads=hidden // 64, num_key_value_heads=4, head_dim=64)
    wl = W.Workload("wide-mlp", cfg, store, n + 1, 6, n + 8, qkv_bias=False)
    ctx = tlm.Context(0)
    runner = R.DecoderHIPRunner(W.synthetic(wl), {"maxTokens": n + 8, "prefillChunkSize": 2048}, ctx=ctx)
    m = runner.model
    prompt = [int(t) for t in np.random.default_rng(n).integers(0, 512, n + 1)]
    res = []
    for least in (0, 64):
        m.reset_cache()
        m.set_prefill(least, 2048)
        m.prefill(prompt, 0, n)
        m.compute_token(prompt[-1], n, True)
        # the second layer's cache rows come from the first one's MLP
        res.append([m.read_logits()] + [a.view(np.float16).astype(np.float32) for a in m.kv_read(1, 0, n)])
    for a, b in zip(res[1], res[0]):
        close(a, b, 2e-2, 1e-2)
    runner.close()
    ctx.close()


def test_chunks_of_several_sizes_on_one_model_equal_fresh_models():
    """A captured chunk goes when a later one has the row buffers replaced: sizes
    in turn and again, over a first set of buffers for chunks of 128 rows and a
    second for 2048, give a fresh model's cache rows bit for bit."""
    layers, base, longest = 2, W.WORKLOADS["llama-3.2-1b"], 2048
    cfg = dict(base.config, num_hidden_layers=layers, vocab_size=4096)
    wl = W.Workload(base.name + "-2l", cfg, base.storage, longest + 1, 6, longest + 8, qkv_bias=base.qkv_bias)
    hw = W.synthetic(wl)
    hw.keep = True
    ctx = tlm.Context(0)
    prompt = [int(t) for t in np.random.default_rng(9).integers(0, 4096, longest)]

    def rows(m, n):
        print(f"[prefill sizes] {n} rows", flush=True)
        m.reset_cache()
        m.prefill(prompt, 0, n)
        return [a.copy() for l in range(layers) for a in m.kv_read(l, 0, n)]

    fresh = {}
    for n in (127, 1000, 1500, 2048):
        runner = R.DecoderHIPRunner(hw, {"maxTokens": longest + 8, "prefillChunkSize": 2048}, ctx=ctx)
        fresh[n] = rows(runner.model, n)
        runner.close()
    runner = R.DecoderHIPRunner(hw, {"maxTokens": longest + 8, "prefillChunkSize": 128}, ctx=ctx)
    for chunk, sizes in ((128, (127,)), (2048, (127, 1000, 127, 2048, 1500, 2048, 1000, 127))):
        runner.model.set_prefill(64, chunk)
        for n in sizes:
            for a, b in zip(rows(runner.model, n), fresh[n]):
                assert np.array_equal(a, b), f"{n} rows in chunks of up to {chunk}"
    runner.close()
    ctx.close()
