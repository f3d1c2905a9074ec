// One-call operators of the C ABI (tlm_op_linear, tlm_op_gated_mlp): one
// vector through a linear in one launch.
#include <stdint.h>

#include <algorithm>

#include "tlm_device.h"

namespace tlm {

// y = bias + W x, or with SWIGLU h[i] = silu(gate_i x) * (up_i x) over the
// plain row order gate [0, I), up [I, 2 I) (TSLLinear.ts:13-82,
// TSLGatedMLP.ts:17-90 for one token).
//
// A block owns R consecutive rows (of each half with SWIGLU) and the whole of
// K, so nothing is left for a second kernel to add up: the time of these
// calls is launches and latency.  A 64-row tile's chunk is 64 x 16 bytes; lane
// l reads row l % R, and the 64 / R lane groups read consecutive chunks, so a
// wave's load covers 64 / R runs of 16 R bytes (whole cache lines from R = 8
// up).  Waves take the chunk groups in turn; the lane groups and the waves are
// added at the end in a fixed order.  x sits in LDS once per block, with its
// q4 group sums; longer inputs go through in slices of `cps` chunks.
//
// Bound: an empty launch takes 2.3 us back to back, and the split-K kernel
// with a second kernel that adds its partials took two of them.  Back to back
// with rotating weights: 1152 x 896 q4 2.4 us, 3072 x 8192 q4 (14.2 MB) 5.8,
// SwiGLU 16384 x 3072 q4 (28.3 MB) 7.2, 16384 x 8192 q4 (75.5 MB) 12.9 (5.9
// TB/s), 16384 x 2048 fp16 (67 MB) 11.2 (6.0 TB/s).
template <int FMT, int R, int W, bool SWIGLU>
__global__ __launch_bounds__(W * 64) void op_gemv_kernel(OpGemvArgs a) {
  extern __shared__ float sm[];
  constexpr int CK = FMT == WF_Q4 ? 32 : 8;  // k per 16-byte chunk
  // floats between chunks of x in LDS: the lane groups' 16-byte reads of
  // consecutive chunks fall on different banks
  constexpr int XS = FMT == WF_Q4 ? 36 : 8;
  constexpr int NG = SWIGLU ? 2 : 1, NS = 64 / R, STEP = W * NS;
  constexpr int XV = 2;  // float4s of x a thread requests before the weights
  float* xl = sm;
  float* xsum = xl + a.cps * XS;
  float* red = xsum + a.cps;  // [NG][W][R]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane % R, sub = lane / R;
  const int rows = SWIGLU ? a.N / 2 : a.N;
  const int row = min((int)blockIdx.x * R + r, rows - 1);
  const uint4* wp[NG];
  const uint16_t* sp[NG];
#pragma unroll
  for (int g = 0; g < NG; g++) {
    const int n = row + g * rows;
    const size_t at = (size_t)(n / kTile) * a.C * kTile + n % kTile;
    wp[g] = a.w + at;
    sp[g] = FMT == WF_Q4 ? a.s + at : nullptr;
  }
  float acc[NG] = {};
  for (int c0 = 0; c0 < a.C; c0 += a.cps) {
    const int ncl = min(a.cps, a.C - c0), n4 = ncl * (CK / 4), k0 = c0 * CK;
    const int nw = wave * NS < ncl ? (ncl - wave * NS + STEP - 1) / STEP : 0;  // this wave's chunk groups
    if (c0) lds_barrier();  // the previous slice has been read
    auto load_x = [&](int f) -> float4 {
      const int k = k0 + 4 * f;
      if (a.x_vec) {
        const float4 v = ldg_f4(a.x + min(k, a.K - 4));
        return k < a.K ? v : make_float4(0.f, 0.f, 0.f, 0.f);
      }
      float4 v;
      v.x = k < a.K ? a.x[k] : 0.f;
      v.y = k + 1 < a.K ? a.x[k + 1] : 0.f;
      v.z = k + 2 < a.K ? a.x[k + 2] : 0.f;
      v.w = k + 3 < a.K ? a.x[k + 3] : 0.f;
      return v;
    };
    auto put_x = [&](int f, float4 v) {
      if (FMT == WF_Q4) {
        const float s = sum8(f < n4 ? (v.x + v.y) + (v.z + v.w) : 0.f);
        if (f < n4) {
          *reinterpret_cast<float4*>(xl + (f >> 3) * XS + (f & 7) * 4) = v;
          if ((f & 7) == 0) xsum[f >> 3] = s;
        }
      } else if (f < n4) {
        *reinterpret_cast<float4*>(xl + 4 * f) = v;
      }
    };
    float4 xv[XV];
#pragma unroll
    for (int u = 0; u < XV; u++)
      if (u * W * 64 < n4) xv[u] = load_x(min(tid + u * W * 64, n4 - 1));
    uint4 d[NG];
    uint16_t sc[NG];
    // chunk group b of this wave (clamped: loads stay unconditional)
    auto load_w = [&](int b) {
      const int c = c0 + min(wave * NS + sub + min(b, max(nw, 1) - 1) * STEP, ncl - 1);
#pragma unroll
      for (int g = 0; g < NG; g++) {
        d[g] = ldg_u4(wp[g] + (size_t)c * kTile);
        if (FMT == WF_Q4) sc[g] = gl(sp[g])[(size_t)c * kTile];
      }
    };
    load_w(0);
    __builtin_amdgcn_sched_barrier(0);  // every load issued before the first wait
#pragma unroll
    for (int u = 0; u < XV; u++)
      if (u * W * 64 < n4) put_x(tid + u * W * 64, xv[u]);
    for (int f = tid + XV * W * 64; f - tid < n4; f += W * 64) put_x(f, load_x(min(f, n4 - 1)));
    lds_barrier();
    for (int b = 0; b < nw; b++) {  // wave-uniform
      uint4 cur[NG];
      uint16_t cs[NG];
#pragma unroll
      for (int g = 0; g < NG; g++) {
        cur[g] = d[g];
        cs[g] = sc[g];
      }
      if (b + 1 < nw) load_w(b + 1);  // in flight during this group's dots
      const int cl = wave * NS + sub + b * STEP, cc = min(cl, ncl - 1);
#pragma unroll
      for (int g = 0; g < NG; g++) {
        const float v = FMT == WF_Q4 ? dot_q4(cur[g], xl + cc * XS, xsum[cc], h2f(cs[g])) : dot_f16(cur[g], xl + cc * XS);
        acc[g] += cl < ncl ? v : 0.f;
      }
    }
  }
#pragma unroll
  for (int g = 0; g < NG; g++) {
    float v = acc[g];
    if (R <= 32) v += lane_swap32(v);
    if (R <= 16) v += lane_swap16(v);
    if (R <= 8) v += dpp<0x128>(v);  // row_ror:8: lane ^ 8
    if (sub == 0) red[(g * W + wave) * R + r] = v;
  }
  lds_barrier();
  const int orow = blockIdx.x * R + tid;
  if (tid >= R || orow >= rows) return;
  float v[NG];
#pragma unroll
  for (int g = 0; g < NG; g++) {
    v[g] = 0.f;
#pragma unroll
    for (int w = 0; w < W; w++) v[g] += red[(g * W + w) * R + tid];
  }
  if (SWIGLU)
    a.y[orow] = v[0] / (1.f + __expf(-v[0])) * v[NG - 1];
  else
    a.y[orow] = v[0] + (a.bias ? a.bias[orow] : 0.f);
}

// Rows per block: the most that still give three blocks for every four CUs
// (more rows read x less often, fewer fill the chip: 8192 output rows at K
// 3072, SwiGLU: 7.2 us at 32 rows = 256 blocks, 8.5 at 16, 8.1 at 64 = 128; 2048
// at K 8192: 5.1 at 8 or 16, 7.0 at 32 = 64 blocks).  Waves: one for each chunk
// group of the block up to 16 (896 x 4864, 19 groups: 3.2 us with 16 waves, 3.4
// with 8, 4.4 with 4; 1152 x 896, 3.5 groups: 2.35 with 4, 2.65 with 16).  From
// four blocks a CU on the blocks fill the chip by themselves and a wave has at
// least three groups, as its start and the sum at the end cost more than what
// it hides: q4 151936 x 256 6.4 -> 5.3 us, x 896 16.2 -> 14.2, 65536 x 896 7.5 ->
// 6.1, fp16 65536 x 256 5.8 -> 4.3.
bool launch_op_gemv(int fmt, bool swiglu, const OpGemvArgs& aa, int cus, hipStream_t st) {
  OpGemvArgs a = aa;
  // x and its sums in at most 48 KB of LDS
  const size_t per_chunk = sizeof(float) * (fmt == WF_Q4 ? 37 : 9);
  a.cps = std::min(a.C, (int)(49152 / per_chunk));
  a.x_vec = a.K % 4 == 0 && (reinterpret_cast<uintptr_t>(a.x) & 15) == 0;
  const int rows = swiglu ? a.N / 2 : a.N;
  int R = 64;
  while (R > 8 && (rows + R - 1) / R < 3 * cus / 4) R /= 2;
  const dim3 grid((rows + R - 1) / R);
  const int groups = (a.cps * R + 63) / 64;
  const bool many = (int)grid.x >= 4 * cus;
  const int W = groups >= (many ? 48 : 12) ? 16 : groups >= (many ? 24 : 6) ? 8 : 4;
  const size_t smem = a.cps * per_chunk + sizeof(float) * (swiglu ? 2 : 1) * W * R;
#define OPG(F, RV, WV)                                                                                       \
  if (fmt == F && R == RV && W == WV) {                                                                      \
    if (swiglu) hipLaunchKernelGGL((op_gemv_kernel<F, RV, WV, true>), grid, dim3(WV * 64), smem, st, a);     \
    else hipLaunchKernelGGL((op_gemv_kernel<F, RV, WV, false>), grid, dim3(WV * 64), smem, st, a);           \
    return true;                                                                                             \
  }
#define OPG_W(F, RV) OPG(F, RV, 4) OPG(F, RV, 8) OPG(F, RV, 16)
#define OPG_R(F) OPG_W(F, 8) OPG_W(F, 16) OPG_W(F, 32) OPG_W(F, 64)
  OPG_R(WF_Q4) OPG_R(WF_F16)
#undef OPG_R
#undef OPG_W
#undef OPG
  return false;
}

}  // namespace tlm
