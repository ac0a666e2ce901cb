// neon_exact_attn.hip -- the canonical decode attention (see k_attn_split in
// neon_kernels.hip for its definition) on the fp32 matrix instruction
// v_mfma_f32_16x16x4_f32, whose four products join the accumulator one after
// the other with one rounding each: a chain of it is the canonical fmaf chain.
//
// A block of 4 waves serves one (row, kv head, key split): the G = Hq / Hkv query
// heads are the columns (lane j + 16 h: column j), so a score or an output of
// every head comes from one pass over K and V.  Per chunk of 64 keys:
//   scores    wave w takes keys 16 w .. 16 w + 15: A = 16 keys x 4 dims, B = q,
//             16 steps along the 64 dims.  Lane i + 16 kk holds dims 4 s + kk of
//             key i: loaded as 4 consecutive dims per lane and transposed 4 x 4
//             between the lanes' kk and the registers with two lane swaps.
//   softmax   the waves' maxima and then their weights meet in LDS (two barriers
//             per chunk); wave 0 forms the butterfly sum of the weights from
//             registers (off 32, 4, 2, 1) and lane exchanges (off 16, 8).
//   output    wave w takes dims 16 w .. 16 w + 15; o[kg] = the chain of keys kg +
//             8 i, i = 0 .. 7: two steps of A = 16 dims x 4 keys (V from LDS),
//             B = the weights.
// The next chunk's K and V are on their way meanwhile.  The splits that hold
// keys (min(S, chunks); the others add nothing to the merge) are numbered in
// order; each stores its partial and k_xa_merge joins them, or with one of them
// the block finishes the row.
// Bound: no unit alone.  T = 8192, B = 8: the address units are 54% busy (8-byte
// loads of K), the vector units 31%, the matrix units 20% (half of the 16 columns
// stand empty at G = 8), and waves wait 39% of their time, at the two barriers of
// a chunk among others; memory reads 1.1 times the cache, 2.6 TB/s.
// us, k_attn_split's vector chains -> this with the merge, 64 / 8 heads: B = 8, T =
// 2048 44.7 -> 21.6, T = 8192 83.4 -> 51.2, B = 32, T = 1024 79 -> 32; 333 prompt
// rows, 0.79 -> 0.06 ms per layer.
#include "neon_common.hpp"
#include "neon_internal.hpp"

namespace neon {

__device__ __forceinline__ xf4 xa_mfma(float a, float b, xf4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// exchanges the register pair's index bit with lane bit 5 / 4
__device__ __forceinline__ void swap32(float& a, float& b) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(p[0]);
  b = __uint_as_float(p[1]);
}
__device__ __forceinline__ void swap16(float& a, float& b) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(p[0]);
  b = __uint_as_float(p[1]);
}
// v[t] of lane kk -> v[kk'] of lane t: 4 x 4 transposition over lane bits 5, 4
__device__ __forceinline__ void xa_transpose(float (&v)[4]) {
  swap32(v[0], v[2]);
  swap32(v[1], v[3]);
  swap16(v[0], v[1]);
  swap16(v[2], v[3]);
}
__device__ __forceinline__ void xa_unpack(float (&v)[4], const uint2& w) {
  v[0] = bf_lo(w.x); v[1] = bf_hi(w.x); v[2] = bf_lo(w.y); v[3] = bf_hi(w.y);
}

constexpr int kXaVStride = 72;  // bf16 per key row in LDS: 16-byte rows, spread over the banks
struct XaLds {
  uint16_t v[2][64 * kXaVStride];
  float p[2][72 * 16];  // weight of (key, column) at (key + key / 8) 16 + column
  float mx[2][4][16];
  float l[16];
};

__global__ __launch_bounds__(256, 4) void k_xa_attn(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc,
    const uint16_t* __restrict__ vc, const int32_t* __restrict__ pos_arr,
    float* __restrict__ part_o, float* __restrict__ part_ml, const uint16_t* __restrict__ sinks,
    uint16_t* __restrict__ out, const int32_t* __restrict__ seq, int Hq, int Hkv, int G, int T_max,
    int key_mask, int window, int S, int q_stride) {
  __shared__ __align__(16) XaLds lds;
  const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, h4 = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = blockIdx.x % Hkv, s = blockIdx.x / Hkv, b = blockIdx.y;
  const int head = g * G + min(j, G - 1);
  // q of the lane's column, whatever the position
  const uint2* qp = reinterpret_cast<const uint2*>(q + (size_t)b * q_stride + (size_t)head * 64);
  uint2 qw[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) qw[m] = qp[4 * m + h4];
  const uint16_t sink_raw = load_pinned_u16(sinks + head);
  const int p = __builtin_amdgcn_readfirstlane(pos_arr[b]);
  const int sq = seq != nullptr ? __builtin_amdgcn_readfirstlane(seq[b]) : b;
  const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
  const int nch = (p - lo + 64) >> 6, ns = min(S, nch);
  if (s >= ns) return;
  const int c0 = nch <= S ? s : (int)((int64_t)s * nch / S);
  const int c1 = nch <= S ? s + 1 : (int)((int64_t)(s + 1) * nch / S);
  const size_t kv_base = ((size_t)sq * Hkv + g) * T_max * 64;
  const uint2* kp = reinterpret_cast<const uint2*>(kc + kv_base) + h4;      // dims 4 kk ..
  const uint4* vp = reinterpret_cast<const uint4*>(vc + kv_base) + (tid & 7);
  uint2 kw[4];
  uint4 vw[2];  // thread: 8 dims of keys tid / 8 and 32 + tid / 8
  auto load = [&](int cb) {
    const uint2* r = kp + (uint32_t)(min(cb + 16 * w + j, p) & key_mask) * 16u;
#pragma unroll
    for (int m = 0; m < 4; ++m) kw[m] = r[4 * m];
#pragma unroll
    for (int u = 0; u < 2; ++u)
      vw[u] = vp[(uint32_t)(min(cb + 32 * u + (tid >> 3), p) & key_mask) * 8u];
  };
  load(lo + 64 * c0);
  float qf[16];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    float v[4];
    xa_unpack(v, qw[m]);
    xa_transpose(v);
#pragma unroll
    for (int t = 0; t < 4; ++t) qf[4 * m + t] = v[t];
  }
  xf4 o[8];
#pragma unroll
  for (int kg = 0; kg < 8; ++kg) o[kg] = xf4{0.0f, 0.0f, 0.0f, 0.0f};
  float mx = -INFINITY, l = 0.0f;
  for (int c = c0; c < c1; ++c) {
    const int cb = lo + 64 * c, buf = c & 1;
    // V to LDS; keys past p as zero rows, as their weights are
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int key = 32 * u + (tid >> 3);
      const uint4 z = make_uint4(0, 0, 0, 0);
      *reinterpret_cast<uint4*>(&lds.v[buf][key * kXaVStride + 8 * (tid & 7)]) = cb + key <= p ? vw[u] : z;
    }
    // ---- scores of the wave's 16 keys ----
    float kv[16];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      float v[4];
      xa_unpack(v, kw[m]);
      xa_transpose(v);
      pin4(v);
#pragma unroll
      for (int t = 0; t < 4; ++t) kv[4 * m + t] = v[t];
    }
    __builtin_amdgcn_sched_barrier(0);
    if (c + 1 < c1) load(cb + 64);
    __builtin_amdgcn_sched_barrier(0);
    xf4 sc = xf4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < 16; ++t) sc = xa_mfma(kv[t], qf[t], sc);
    float cm = -INFINITY;
    bool valid[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      valid[r] = cb + 16 * w + 4 * h4 + r <= p;
      sc[r] = valid[r] ? __fmul_rn(sc[r], 0.125f) : -INFINITY;
      cm = fmaxf(cm, sc[r]);
    }
    cm = fmaxf(cm, xor_lane<32>(cm));
    cm = fmaxf(cm, xor_lane<16>(cm));
    if (h4 == 0) lds.mx[buf][w][j] = cm;
    lds_barrier();
    // ---- weights ----
    cm = fmaxf(fmaxf(lds.mx[buf][0][j], lds.mx[buf][1][j]), fmaxf(lds.mx[buf][2][j], lds.mx[buf][3][j]));
    const float mn = fmaxf(mx, cm);
    const float alpha = neon_expf(__fsub_rn(mx, mn));
    mx = mn;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = 16 * w + 4 * h4 + r;
      lds.p[buf][(key + (key >> 3)) * 16 + j] = valid[r] ? neon_expf(__fsub_rn(sc[r], mn)) : 0.0f;
    }
#pragma unroll
    for (int kg = 0; kg < 8; ++kg)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[kg][r] = __fmul_rn(o[kg][r], alpha);
    lds_barrier();
    // pb[s2][kg]: the weight of key kg + 8 (4 s2 + kk) for lane kk; va: its V at
    // the lane's dim
    float pb[2][8], va[2][8];
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int kg = 0; kg < 8; ++kg) {
        const int k8 = 4 * s2 + h4;
        pb[s2][kg] = lds.p[buf][(kg + 9 * k8) * 16 + j];
        va[s2][kg] = bf2f(lds.v[buf][(kg + 8 * k8) * kXaVStride + 16 * w + j]);
      }
    if (w == 0) {  // l: off 32 joins the steps, 16 and 8 the lanes, 4, 2, 1 the key groups
      float t[8];
#pragma unroll
      for (int kg = 0; kg < 8; ++kg) {
        t[kg] = __fadd_rn(pb[0][kg], pb[1][kg]);
        t[kg] = __fadd_rn(t[kg], xor_lane<32>(t[kg]));
        t[kg] = __fadd_rn(t[kg], xor_lane<16>(t[kg]));
      }
      const float a = __fadd_rn(__fadd_rn(t[0], t[4]), __fadd_rn(t[2], t[6]));
      const float d = __fadd_rn(__fadd_rn(t[1], t[5]), __fadd_rn(t[3], t[7]));
      l = __builtin_fmaf(l, alpha, __fadd_rn(a, d));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int kg = 0; kg < 8; ++kg) o[kg] = xa_mfma(va[s2][kg], pb[s2][kg], o[kg]);
  }
  // over the key groups: xor 8, 16, 32 of the lane form; dim 16 w + 4 h + r
  float r4[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    r4[r] = __fadd_rn(__fadd_rn(__fadd_rn(o[0][r], o[1][r]), __fadd_rn(o[2][r], o[3][r])),
                      __fadd_rn(__fadd_rn(o[4][r], o[5][r]), __fadd_rn(o[6][r], o[7][r])));
  if (ns == 1) {  // the only split with keys: the merge with the sink
    if (w == 0 && h4 == 0) lds.l[j] = l;
    lds_barrier();
    l = lds.l[j];
    const float sk = bf2f(sink_raw);
    const float M = fmaxf(sk, mx);
    float den = neon_expf(__fsub_rn(sk, M));
    const float f = (mx == -INFINITY) ? 0.0f : neon_expf(__fsub_rn(mx, M));
    den = __builtin_fmaf(l, f, den);
    const float inv = __fdiv_rn(1.0f, den);
    uint32_t w2[2];
#pragma unroll
    for (int e = 0; e < 2; ++e)
      w2[e] = pack_bf2(__fmul_rn(__builtin_fmaf(f, r4[2 * e], 0.0f), inv),
                       __fmul_rn(__builtin_fmaf(f, r4[2 * e + 1], 0.0f), inv));
    if (j < G)
      *reinterpret_cast<uint2*>(out + ((size_t)b * Hq + head) * 64 + 16 * w + 4 * h4) =
          make_uint2(w2[0], w2[1]);
    return;
  }
  if (j >= G) return;
  const size_t pi = ((size_t)b * Hq + head) * S + s;
  *reinterpret_cast<float4*>(part_o + pi * 64 + 16 * w + 4 * h4) = make_float4(r4[0], r4[1], r4[2], r4[3]);
  if (w == 0 && h4 == 0) *reinterpret_cast<float2*>(part_ml + pi * 2) = make_float2(mx, l);
}

// Joins a head's partials with the sink, lane = dim: attn_merge_head's
// operations over the splits that hold keys (the others' factor is 0).
constexpr int kXaMaxSplits = 32;
__global__ __launch_bounds__(64) void k_xa_merge(const float* __restrict__ part_o,
                                                 const float* __restrict__ part_ml,
                                                 const int32_t* __restrict__ pos_arr,
                                                 const uint16_t* __restrict__ sinks,
                                                 uint16_t* __restrict__ out, int Hq, int S,
                                                 int window) {
  const int h = blockIdx.x, b = blockIdx.y, lane = threadIdx.x;
  const int p = __builtin_amdgcn_readfirstlane(pos_arr[b]);
  const int n = min(S, ((window > 0 ? min(window, p + 1) : p + 1) + 63) >> 6);
  if (n == 1) return;  // finished by its wave
  const size_t pi = ((size_t)b * Hq + h) * S;
  float ov[kXaMaxSplits];
#pragma unroll
  for (int t = 0; t < kXaMaxSplits; ++t) ov[t] = part_o[(pi + min(t, n - 1)) * 64 + lane];
  const float2 ml = *reinterpret_cast<const float2*>(part_ml + (pi + min(lane, n - 1)) * 2);
  const float mt = lane < n ? ml.x : -INFINITY;
  const float sk = bf2f(sinks[h]);
  const float M = fmaxf(sk, wave_max(mt));
  const float f = (mt == -INFINITY) ? 0.0f : neon_expf(__fsub_rn(mt, M));
  float den = neon_expf(__fsub_rn(sk, M));
  float acc = 0.0f;
#pragma unroll
  for (int t = 0; t < kXaMaxSplits; ++t)
    if (t < n) {
      const float ft = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), t));
      const float lt = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(ml.y), t));
      den = __builtin_fmaf(lt, ft, den);
      acc = __builtin_fmaf(ft, ov[t], acc);
    }
  out[((size_t)b * Hq + h) * 64 + lane] = f2bf(__fmul_rn(acc, __fdiv_rn(1.0f, den)));
}

void launch_xa_attn(const AttnArgs& a, int max_keys, hipStream_t st) {
  const int G = a.Hq / a.Hkv;
  const int span = a.window > 0 && a.window < max_keys ? a.window : max_keys;
  const int ch = (span + 63) / 64, ns = ch < a.S ? ch : a.S;
  hipLaunchKernelGGL(k_xa_attn, dim3(a.Hkv * ns, a.B), dim3(256), 0, st, a.q, a.kc, a.vc, a.pos,
                     a.part_o, a.part_ml, a.sinks, a.out, a.seq, a.Hq, a.Hkv, G, a.T_max, a.key_mask,
                     a.window, a.S, a.q_stride);
  if (ns > 1)
    hipLaunchKernelGGL(k_xa_merge, dim3(a.Hq, a.B), dim3(64), 0, st, a.part_o, a.part_ml, a.pos,
                       a.sinks, a.out, a.Hq, a.S, a.window);
}

}  // namespace neon
