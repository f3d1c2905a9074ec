"""One decode attention call at the window lengths where its route changes: the
block per head (a wave per pass of 8 to 64 positions, 12 of them), the chunks with
their combine and, past 1024 positions, the matrix-core kernel, each one position
short of, at and past its edge, as prefix lengths and as sliding windows.

Inputs of unit scale, so the scores' softmax is neither flat nor a single row.
The reference attends to the cache rows that the device holds: a K element whose
fp32 rotation falls across an fp16 tie from the 64-bit one moves its score by up to
2^-10 |k| |q| scale, about 1e-3, which would hide what is tested; the rows
themselves are checked to one rounding of their own.  What is left is fp32 sums
and exponentials (past 1024 positions q enters the matrix cores as hi + lo fp16
pairs): 2e-5 of the output's scale, and 5e-6 with fp32 rows."""
import ctypes

import numpy as np
import pytest

import three_llm_amd.tlm as tlm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = tlm.Context(0)
    yield c
    c.close()


def rope(x, pos, inv):
    ang = pos[:, None] * inv[None, :].astype(np.float64)
    c, s = np.cos(ang)[:, None, :], np.sin(ang)[:, None, :]
    half = inv.size
    a, b = x[..., :half], x[..., half:2 * half]
    return np.concatenate([a * c - b * s, b * c + a * s, x[..., 2 * half:]], -1)


def run(ctx, hq, hkv, d, kv_fmt, positions, window=0, rotary=None):
    rng = np.random.default_rng(d * 1000 + hq + window)
    n, rd = max(positions) + 1, d if rotary is None else rotary
    inv = (1e4 ** (-np.arange(0, rd, 2) / rd)).astype(np.float32) if rd else None
    x = rng.standard_normal((n, hq + 2 * hkv, d)).astype(np.float32)
    q, k, v = x[:, :hq].astype(np.float64), x[:, hq:hq + hkv].astype(np.float64), x[:, hq + hkv:].astype(np.float64)
    if rd:
        q, k = rope(q, np.arange(n), inv), rope(k, np.arange(n), inv)
    if kv_fmt == tlm.FMT_F16:
        k, v = k.astype(np.float16).astype(np.float64), v.astype(np.float16).astype(np.float64)
    a = tlm.Attention(ctx, hq, hkv, d, n + 7, inv_freq=inv, rotary_dim=rd or None, sliding_window=window, kv_fmt=kv_fmt)
    buf, out = ctx.buffer(4 * (hq + 2 * hkv) * d), ctx.buffer(4 * hq * d)
    want = set(positions)
    for p in range(n):
        a(buf.write(x[p]), p, out)
        if p not in want:
            continue
        got = out.read().reshape(hq, d)
        kc, vc = (c.reshape(p + 1, hkv, d).astype(np.float64) for c in a.read_cache(p + 1))
        ulp = 2.0 ** -10 if kv_fmt == tlm.FMT_F16 else 1e-6
        assert np.array_equal(vc, v[:p + 1])
        assert np.all(np.abs(kc - k[:p + 1]) <= ulp * np.maximum(np.abs(k[:p + 1]), 2.0 ** -12) + 4e-7)
        first = max(0, p - window + 1) if window else 0
        for h in range(hq):
            kk, vv = kc[first:, h // (hq // hkv)], vc[first:, h // (hq // hkv)]
            s = kk @ q[p, h] / np.sqrt(d)
            e = np.exp(s - s.max())
            ref = (e / e.sum()) @ vv
            tol = 2e-5 if kv_fmt == tlm.FMT_F16 else 5e-6
            err = np.abs(got[h] - ref).max()
            assert err <= tol * max(1.0, np.abs(ref).max()), f"position {p} head {h}: {err}"
    a.close()
    buf.free()
    out.free()


@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (4, 4, 64), (24, 8, 128), (3, 1, 128), (16, 1, 64)])
def test_fp16_cache_routes(ctx, hq, hkv, d):
    # 192 | 193 (head_dim 128) and 384 | 385 (64): block per head -> chunks; 1024 | 1025
    # (prefix lengths): the matrix-core kernel
    run(ctx, hq, hkv, d, tlm.FMT_F16, [0, 1, 15, 16, 31, 32, 62, 63, 64, 65, 127, 190, 191, 192, 255, 256, 382, 383, 384,
                                       511, 512, 513, 767, 768, 769, 1023, 1024, 1025])


@pytest.mark.parametrize("d,positions", [(64, [0, 15, 16, 63, 190, 191, 192, 193, 300]), (128, [0, 7, 8, 94, 95, 96, 97, 200]),
                                         (32, [0, 31, 32, 382, 383, 384, 385]), (18, [0, 31, 32, 40])])
def test_fp32_cache_routes(ctx, d, positions):
    run(ctx, 6, 2, d, tlm.FMT_F32, positions)


@pytest.mark.parametrize("window", [1, 33, 64, 65, 513, 769])
def test_sliding_windows(ctx, window):
    run(ctx, 8, 2, 64, tlm.FMT_F16, [0, window - 1, window, window + 1, window + 40], window)


def test_without_the_matrix_core_kernel_and_partial_rotary(ctx):
    run(ctx, 4, 2, 32, tlm.FMT_F16, [0, 63, 64, 767, 768, 769, 1030], rotary=16)
    run(ctx, 8, 4, 64, tlm.FMT_F16, [0, 63, 64, 700], rotary=32)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("position", [70, 300, 500, 800, 1023])
def test_queries_past_the_fp16_range(ctx, d, position):
    """Windows up to 1024 positions keep q in 32 bits: q * attn_scale * log2 e is past
    fp16's largest value here, over cache rows small enough for scores of order ten.
    Their 32-bit sums of d terms are off by at most d 2^-24 of the terms' magnitudes
    (51 in all at d 64): 2e-4 of a probability."""
    hq, hkv = 4, 2
    rng = np.random.default_rng(d + position)
    n = position + 1
    x = np.zeros((n, hq + 2 * hkv, d), np.float32)
    x[:, hq:hq + hkv] = rng.integers(-32, 33, (n, hkv, d)) * 2.0 ** -20 * (64 / d)
    x[:, hq + hkv:] = rng.standard_normal((n, hkv, d)).astype(np.float16)
    a = tlm.Attention(ctx, hq, hkv, d, n, attn_scale=1.0)  # no rotary dims
    a.rows(ctx.array(x), n, 0, ctx.buffer(2 * n * hq * d))
    x[position, :hq] = rng.standard_normal((hq, d)) * 2.0 ** 16
    got = a(ctx.array(x[position]), position, ctx.buffer(4 * hq * d)).read().reshape(hq, d)
    kc, vc = (c.reshape(n, hkv, d).astype(np.float64) for c in a.read_cache(n))
    a.close()
    for h in range(hq):
        s = kc[:, h // 2] @ x[position, h].astype(np.float64)
        e = np.exp(s - s.max())
        ref = (e / e.sum()) @ vc[:, h // 2]
        assert np.abs(got[h] - ref).max() <= 2e-4 * max(1.0, np.abs(ref).max()), f"head {h}"


@pytest.mark.parametrize("kv_fmt", [tlm.FMT_F16, tlm.FMT_F32])
@pytest.mark.parametrize("d,position", [(64, 0), (64, 40), (64, 150), (128, 90), (20, 60)])
def test_out_inside_qkv(ctx, d, position, kv_fmt):
    """out over any part of qkv: over the queries alone, half over the keys, over the
    keys and values.  The sums may be taken in another order than with out apart."""
    hq, hkv = 16, 8
    rng = np.random.default_rng(d + position)
    x = rng.standard_normal((position + 1, (hq + 2 * hkv) * d)).astype(np.float32)
    a = tlm.Attention(ctx, hq, hkv, d, position + 1, kv_fmt=kv_fmt)
    qkv, out = ctx.buffer(x[0].nbytes), ctx.buffer(4 * hq * d)
    for p in range(position + 1):
        a(qkv.write(x[p]), p, out)
    ref = out.read().reshape(hq * d)
    for at in (0, hq * d // 2 + 1, hq * d):
        qkv.write(x[position])
        tlm.check(tlm.lib().tlm_op_attention(a.ptr, qkv.ptr, position, ctypes.c_void_p(qkv.ptr.value + 4 * at)))
        got = qkv.read().reshape(-1)[at:at + hq * d]
        assert np.abs(got - ref).max() <= 2e-6 * max(1.0, np.abs(ref).max()), f"out at {at}"
    a.close()
