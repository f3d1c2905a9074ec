"""tlm_op_attention_rows where its kernel can go wrong: key and query tiles that
end inside a tile, a softmax reference that moves with every tile or never, rows
with nothing to see in a tile, and queries staged in the context's buffer or in one
of their own.

No rotation (frequencies of zero) and queries and keys on a coarse grid make
every score exact in fp32; what is left is fp16 probabilities (2^-11 each,
rounded to nearest) and the fp16 output, so 2e-3 bounds the error of a
weighted mean of values of unit scale."""
import math

import numpy as np
import pytest

import three_llm_amd.tlm as tlm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = tlm.Context(0)
    yield c
    c.close()


def inputs(rng, n, heads, kv, D, slope):
    """Rows whose scores change by about `slope` (log2) per key position."""
    q = rng.integers(-2, 3, (n, heads, D)) / 8.0
    k = rng.integers(-8, 9, (n, kv, D)) / 8.0
    q[:, :, 0] = 1.0
    k[:, :, 0] = np.round(np.arange(n) * slope * 8)[:, None] / 8.0
    v = rng.standard_normal((n, kv, D)).astype(np.float16).astype(np.float32)
    return np.concatenate([x.reshape(n, -1) for x in (q, k, v)], 1).astype(np.float32)


def expected(x, p0, heads, kv, D, window):
    n = x.shape[0]
    q = x[p0:, :heads * D].astype(np.float64).reshape(n - p0, heads, D)
    k = x[:, heads * D:(heads + kv) * D].astype(np.float64).reshape(n, kv, D)
    v = x[:, (heads + kv) * D:].astype(np.float64).reshape(n, kv, D)
    pos, key = np.arange(p0, n)[:, None], np.arange(n)[None, :]
    hidden = (key > pos) | ((key <= pos - window) if window else False)
    out = np.empty((n - p0, heads, D))
    for h in range(heads):
        s = np.where(hidden, -np.inf, q[:, h] @ k[:, h // (heads // kv)].T)
        p = np.exp2(s - s.max(1, keepdims=True))
        out[:, h] = (p / p.sum(1, keepdims=True)) @ v[:, h // (heads // kv)]
    return out.reshape(n - p0, heads * D)


@pytest.mark.parametrize("heads,kv,D", [(7, 1, 64), (4, 2, 64), (3, 1, 128)])
@pytest.mark.parametrize("p0,rows,window,slope", [
    (0, 1, 0, 0.0), (0, 33, 0, 1.0), (31, 34, 0, -1.0), (63, 1, 0, 1.0), (64, 65, 0, 0.5), (1, 127, 0, -0.25),
    (200, 161, 0, 4.0), (200, 161, 0, -4.0), (190, 100, 30, 1.0), (190, 100, 1, 0.0), (100, 200, 129, -2.0),
])
def test_rows_at_tile_edges_and_moving_references(ctx, heads, kv, D, p0, rows, window, slope):
    print(f"[attention rows] {heads}/{kv} x {D}, {rows} at {p0}, window {window}, slope {slope}", flush=True)
    rng = np.random.default_rng(heads * 1000 + p0 + rows)
    n = p0 + rows
    x = inputs(rng, n, heads, kv, D, slope)
    A = tlm.Attention(ctx, heads, kv, D, n, np.zeros(D // 2, np.float32), sliding_window=window,
                      attn_scale=math.log(2.0))
    if p0:
        A.rows(ctx.array(x[:p0]), p0, 0, ctx.buffer(2 * p0 * heads * D))
    got = A.rows(ctx.array(x[p0:]), rows, p0, ctx.buffer(2 * rows * heads * D)).read(np.uint16)
    A.close()
    got = got.view(np.float16).astype(np.float64).reshape(rows, heads * D)
    ref = expected(x, p0, heads, kv, D, window)
    assert np.abs(got - ref).max() <= 2e-3 * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("D", [64, 128])
def test_rows_written_over_their_projections_equal_rows_apart(ctx, D):
    """out inside qkv: the queries are staged first, so the result is the same."""
    heads, kv, rows = 6, 2, 70
    rng = np.random.default_rng(D)
    x = rng.standard_normal((rows, (heads + 2 * kv) * D)).astype(np.float32)
    inv = (1e4 ** (-np.arange(0, D, 2) / D)).astype(np.float32)
    outs = []
    for inside in (False, True):
        A = tlm.Attention(ctx, heads, kv, D, rows, inv)
        qkv = ctx.array(x)
        out = A.rows(qkv, rows, 0, qkv if inside else ctx.buffer(2 * rows * heads * D))
        outs.append(out.read(np.uint16)[:rows * heads * D].copy())
        A.close()
    assert np.array_equal(*outs)


@pytest.mark.parametrize("scale,q0,unit,dims", [(2.0 ** -24, 1.5, 2.0 ** 12, None), (2.0, 49984.0, 2.0 ** -14, 1)])
@pytest.mark.parametrize("rotary", [True, False])
@pytest.mark.parametrize("D", [64, 128])
def test_queries_round_before_the_softmax_scale(ctx, D, rotary, scale, q0, unit, dims):
    """The scale multiplies fp32 scores: query values that fp16 holds exactly keep
    every bit where query * scale is subnormal in fp16 (1.5 steps: 2 once rounded)
    or past its largest value."""
    print(f"[attention rows] D {D}, scale {scale}, queries {q0}", flush=True)
    rng = np.random.default_rng(D)
    n = 97
    c = rng.integers(-8, 9, (n, 1, 1)).astype(np.float64)
    q, k = np.zeros((n, 2, D)), np.zeros((n, 1, D))
    q[:, :, :dims], k[:, :, :dims] = q0, c * unit
    v = (c / 8 + 0.1 * rng.standard_normal((n, 1, D))).astype(np.float16)
    x = np.concatenate([t.reshape(n, -1) for t in (q, k, v)], 1).astype(np.float32)
    A = tlm.Attention(ctx, 2, 1, D, n, np.zeros(D // 2, np.float32) if rotary else None, rotary_dim=None if rotary else 0,
                      attn_scale=scale * math.log(2.0))
    got = A.rows(ctx.array(x), n, 0, ctx.buffer(2 * n * 2 * D)).read(np.uint16)
    A.close()
    got = got.view(np.float16).astype(np.float64).reshape(n, 2 * D)
    x64 = x.astype(np.float64)
    x64[:, :2 * D] *= scale
    ref = expected(x64, 0, 2, 1, D, 0)
    assert np.abs(got - ref).max() <= 2e-3 * max(1.0, np.abs(ref).max())


def test_rows_written_right_after_creation_stay(ctx):
    """The cache's first fill ends before its attention is handed out: 512 MiB
    each of K and V, and the rows of the first calls are there afterwards."""
    heads, kv, D, rows = 8, 8, 128, 64
    x = np.random.default_rng(5).standard_normal((rows, (heads + 2 * kv) * D)).astype(np.float16).astype(np.float32)
    qkv, out = ctx.array(x), ctx.buffer(2 * rows * heads * D)
    ctx.sync()
    for _ in range(3):
        A = tlm.Attention(ctx, heads, kv, D, 1 << 18)  # no rotary dims: the rows are the projection's
        A.rows_noalloc(qkv, rows, 0, out)
        k, v = A.read_cache(rows)
        A.close()
        assert np.array_equal(np.concatenate([k, v], 1), x[:, heads * D:])


def test_queries_past_the_contexts_buffer(ctx):
    """4100 rows of 32 x 128 queries (33.6 MB) get a buffer of their own: the same
    rows as in two calls that fit the context's."""
    heads, kv, D, rows = 32, 2, 128, 4100
    x = np.random.default_rng(3).standard_normal((rows, (heads + 2 * kv) * D)).astype(np.float32)
    inv = (1e4 ** (-np.arange(0, D, 2) / D)).astype(np.float32)
    outs = []
    for parts in ((rows,), (2048, rows - 2048)):
        A = tlm.Attention(ctx, heads, kv, D, rows, inv)
        done = []
        for n in parts:
            p = sum(len(d) for d in done)
            out = ctx.buffer(2 * n * heads * D)
            done.append(A.rows(ctx.array(x[p:p + n]), n, p, out).read(np.uint16).reshape(n, heads * D))
        outs.append(np.concatenate(done))
        A.close()
    a, b = (o.view(np.float16).astype(np.float64) for o in outs)
    assert np.abs(a - b).max() <= 2e-3 * np.abs(a).max()
