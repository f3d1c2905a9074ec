"""tlm_op_linear_rows at the edges of its tiles and split counts, against the
float64 product of the fp16 operands the matrix cores see (weights rounded to
fp16 once, activations fp16).  fp32 sums of K products: an error bound of
2e-6 of the sum of magnitudes, as for any order of the same additions."""
import ctypes

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


def make_linear(ctx, fmt, w):
    if fmt == tlm.FMT_Q4:
        packed, scales = orc.q4_quantize(w)
        return tlm.Linear(ctx, fmt, packed, scales), orc.q4_dequant(packed, scales)
    h = w.astype(np.float16)
    return tlm.Linear(ctx, fmt, np.ascontiguousarray(h.view(np.uint16))), h.astype(np.float32)


# (format, rows, N, K, bias, the block's rows x columns, whether K goes in slices);
# test_rows_plan.py holds the planner to the last two without a GPU
CASES = [
    # four waves splitting K on 32 x 64 tiles: a wave without steps, a ring that
    # is never full, ragged rows and columns
    (tlm.FMT_F16, 1, 256, 32, True, (32, 64), False), (tlm.FMT_F16, 31, 65, 96, False, (32, 64), False),
    (tlm.FMT_F16, 33, 64, 416, True, (32, 64), False), (tlm.FMT_F16, 129, 1000, 1056, True, (32, 64), False),
    # the same in K slices that a second kernel adds; N % 4 != 0 there too
    (tlm.FMT_F16, 33, 192, 4096, True, (32, 64), True), (tlm.FMT_F16, 33, 195, 2080, True, (32, 64), True),
    (tlm.FMT_Q4, 31, 130, 4096, False, (32, 64), True), (tlm.FMT_Q4, 257, 300, 8192, True, (32, 64), True),
    # 128 x 128 tiles, whole and in slices
    (tlm.FMT_F16, 1030, 4100, 1024, True, (128, 128), False), (tlm.FMT_F16, 512, 2048, 4096, False, (128, 128), True),
    (tlm.FMT_F16, 700, 10000, 320, True, (128, 128), False),
    # 256 x 256 tiles: rows and columns past the last whole one, an odd step count
    (tlm.FMT_F16, 900, 12300, 608, True, (256, 256), False),
    # 128 x 256 tiles (q4), whole and in slices
    (tlm.FMT_Q4, 900, 8200, 256, True, (128, 256), False), (tlm.FMT_Q4, 257, 4100, 6048, False, (128, 256), True),
    # few rows over many columns: 64 x 256, 32 x 256 (one and two row tiles) and, fp16, 64 x 128
    (tlm.FMT_Q4, 61, 65600, 544, True, (64, 256), False), (tlm.FMT_Q4, 63, 65541, 64, False, (32, 256), False),
    (tlm.FMT_Q4, 17, 131100, 96, True, (32, 256), False), (tlm.FMT_F16, 50, 16450, 160, True, (64, 128), False),
    (tlm.FMT_F16, 32, 49200, 1056, False, (64, 128), False),
]


@pytest.mark.parametrize("fmt,M,N,K,bias", [c[:5] for c in CASES])
def test_rows_at_tile_edges(ctx, fmt, M, N, K, bias):
    print(f"[rows] fmt {fmt}, {M} x {N} x {K}", flush=True)
    rng = np.random.default_rng(M * 7 + N + K)
    w = (rng.standard_normal((N, K), dtype=np.float32) * 0.02).astype(np.float32)
    x = rng.standard_normal((M, K), dtype=np.float32).astype(np.float16)
    b = (rng.standard_normal(N) * 0.1).astype(np.float32)
    L, wd = make_linear(ctx, fmt, w)
    # two calls: the second finds the slices' buffer as the first left it
    out = ctx.array(np.full((M, N), np.nan, np.float32))
    for _ in range(2):
        y = L.rows(ctx.array(x.view(np.uint16)), M, out, ctx.array(b) if bias else None).read().reshape(M, N)
    L.close()
    xh, wh = x.astype(np.float64), wd.astype(np.float16).astype(np.float64)
    ref, mag = xh @ wh.T, np.abs(xh) @ np.abs(wh).T
    if bias:
        ref, mag = ref + b, mag + np.abs(b)
    excess = np.abs(y - ref) - (2e-6 * mag + 1e-7)
    assert excess.max() <= 0, f"max excess {excess.max()}"


@pytest.mark.parametrize("fmt", [tlm.FMT_F16, tlm.FMT_Q4])
@pytest.mark.parametrize("M,N,K", [(3, 100, 96), (130, 4200, 512), (40, 64, 1 << 19)])
def test_rows_from_any_alignment_of_x(ctx, fmt, M, N, K):
    """x at 2, 4 and 8 bytes past a 16-byte boundary: the rows are staged (the last
    shape in two parts) and give the aligned call's sums, of unsplit products."""
    print(f"[rows] unaligned x, fmt {fmt}, {M} x {N} x {K}", flush=True)
    rng = np.random.default_rng(M + N)
    w = (rng.standard_normal((N, K), dtype=np.float32) * 0.02).astype(np.float32)
    x = rng.standard_normal((M, K), dtype=np.float32).astype(np.float16)
    b = (rng.standard_normal(N) * 0.1).astype(np.float32)
    L, wd = make_linear(ctx, fmt, w)
    xh, wh = x.astype(np.float32), wd.astype(np.float16).astype(np.float32)
    ref, mag = xh.astype(np.float64) @ wh.T.astype(np.float64) + b, np.abs(xh) @ np.abs(wh).T + np.abs(b)
    bias, out = ctx.array(b), ctx.buffer(4 * M * N)
    for halves in (1, 2, 4):
        buf = ctx.array(np.concatenate([np.zeros(halves, np.uint16), x.view(np.uint16).reshape(-1)]))
        assert buf.ptr.value % 16 == 0
        out.write(np.full(M * N, np.nan, np.float32))
        tlm.check(tlm.lib().tlm_op_linear_rows(L.ptr, ctypes.c_void_p(buf.ptr.value + 2 * halves), M, bias.ptr, out.ptr))
        excess = np.abs(out.read().reshape(M, N) - ref) - (2e-6 * mag + 1e-7)
        assert excess.max() <= 0, f"{halves} halves: max excess {excess.max()}"
        buf.free()
    L.close()
