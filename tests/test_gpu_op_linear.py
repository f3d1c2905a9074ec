"""The one-launch linear and gated MLP (op_gemv_kernel) where they can go wrong:
row counts at the edges of a block's rows (8, 16, 32 or 64 by the row count), one
chunk of K up to more than one slice of x in LDS (10624 k for q4, 10920 for fp16),
K that no float4 covers, and a result written over its own input.

Tolerance, per output: fp32 accumulation against the oracle's double sum,
4e-5 (|x| . |W|) + 1e-7, as for every linear op here (the q4 dot subtracts
8 sum(x), whose terms are bounded by the same magnitude sum)."""
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


def make(ctx, fmt, n, k, rng):
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    if fmt == tlm.FMT_Q4:
        packed, scales = orc.q4_quantize(w)
        return tlm.Linear(ctx, fmt, packed, scales), orc.q4_dequant(packed, scales)
    bits = w.astype(np.float16).view(np.uint16)
    return tlm.Linear(ctx, fmt, bits), bits.view(np.float16).astype(np.float32)


def check(y, x, w, b=None):
    ref = w.astype(np.float64) @ x.astype(np.float64)
    mag = np.abs(w).astype(np.float64) @ np.abs(x).astype(np.float64)
    if b is not None:
        ref, mag = ref + b, mag + np.abs(b)
    excess = np.abs(y.astype(np.float64) - ref) - (4e-5 * mag + 1e-7)
    assert excess.max() <= 0, f"row {int(excess.argmax())}: excess {excess.max()}"


Q4, F16 = tlm.FMT_Q4, tlm.FMT_F16


@pytest.mark.parametrize("fmt,n,k", [(Q4, 1, 32), (Q4, 9, 64), (Q4, 1535, 96), (Q4, 3071, 160), (Q4, 3073, 416),
                                     (Q4, 6145, 384), (Q4, 12289, 224), (Q4, 65, 10624), (Q4, 65, 10656),
                                     (Q4, 12300, 10688), (F16, 1, 1), (F16, 8, 8), (F16, 1537, 30), (F16, 3100, 136),
                                     (F16, 6200, 97), (F16, 12290, 40), (F16, 33, 10920), (F16, 33, 10931),
                                     # four blocks a CU and more: 4, 8 and 16 waves by the chunks
                                     (Q4, 65473, 736), (Q4, 65473, 768), (Q4, 65473, 1536), (F16, 65480, 190),
                                     (F16, 65480, 192), (F16, 65480, 385)])
def test_linear_at_block_and_slice_edges(ctx, fmt, n, k):
    rng = np.random.default_rng(n * 31 + k)
    lin, w = make(ctx, fmt, n, k, rng)
    x = rng.standard_normal(k).astype(np.float32)
    b = (rng.standard_normal(n) * 0.1).astype(np.float32)
    check(lin(ctx.array(x), ctx.buffer(4 * n), ctx.array(b)).read(), x, w, b)
    check(lin(ctx.array(x), ctx.buffer(4 * n)).read(), x, w)
    lin.close()


def test_linear_writes_over_its_input(ctx):
    rng = np.random.default_rng(5)
    lin, w = make(ctx, Q4, 896, 896, rng)
    x = rng.standard_normal(896).astype(np.float32)
    b = (rng.standard_normal(896) * 0.1).astype(np.float32)
    buf = ctx.array(x)
    check(lin(buf, buf, ctx.array(b)).read(), x, w, b)
    lin.close()


@pytest.mark.parametrize("fmt,hidden,inner", [(Q4, 64, 32), (Q4, 96, 1568), (Q4, 2080, 96), (F16, 24, 33),
                                              (F16, 257, 3137), (F16, 40, 6145)])
def test_gated_mlp_at_block_edges(ctx, fmt, hidden, inner):
    rng = np.random.default_rng(hidden + inner)
    gu, wgu = make(ctx, fmt, 2 * inner, hidden, rng)
    down, wd = make(ctx, fmt, hidden, inner, rng)
    x = (rng.standard_normal(hidden) * 4).astype(np.float32)
    y = tlm.gated_mlp(gu, down, ctx.array(x), ctx.buffer(4 * hidden)).read().astype(np.float64)
    z = wgu.astype(np.float64) @ x
    g, u = z[:inner], z[inner:]
    h = g / (1 + np.exp(-g)) * u
    # the bound of the first product goes through |silu'| <= 1.1 and the product with u, then both dots
    dz = 4e-5 * (np.abs(wgu).astype(np.float64) @ np.abs(x)) + 1e-7
    dh = 1.1 * dz[:inner] * (np.abs(u) + dz[inner:]) + np.abs(g) * dz[inner:] + 1e-6 * np.abs(h)
    bound = np.abs(wd).astype(np.float64) @ (dh + 4e-5 * np.abs(h)) + 1e-7
    excess = np.abs(y - wd.astype(np.float64) @ h) - bound
    assert excess.max() <= 0
    gu.close()
    down.close()
