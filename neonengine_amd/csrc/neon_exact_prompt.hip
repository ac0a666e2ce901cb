// neon_exact_prompt.hip -- the exact prompt pass: many prompt rows at once with
// the canonical fp32 dot products on the fp32 matrix instructions.
//
// v_mfma_f32_16x16x4_f32 adds its four products to the accumulator one after
// the other, k = 0, 1, 2, 3, each with one correctly rounded fused multiply-add
// (compared with a v_fma_f32 chain on 16.8M operand sets of each of six kinds,
// denormals, infinities and NaN included).  A chain of them along K is the
// canonical chain of the one-row kernels for 16 weight rows x 16 input rows at
// once, so the results are bit-identical to prompt rows taken one at a time.
//
// Lanes: A (weights) lane i + 16 kk holds row i, element 4 s + kk of step s; B
// (inputs) lane j + 16 kk row j, element 4 s + kk; D's register r at lane
// j + 16 h is output row 4 h + r, column j.
//
// The canonical dot has 64 lane partials (chain l: the units u = l + 64 p in
// increasing p) summed by an xor butterfly, off = 32 .. 1.  Here the chains run
// one after the other with l in bit-reversed order, and their sums meet as in
// a binary counter: after chain t (l = bitrev6(t)) the sum merges with as many
// waiting partial sums as t has trailing ones.  The pairings are the
// butterfly's, and fp32 addition commutes, so the bits are too.
#include "neon_common.hpp"
#include "neon_internal.hpp"

namespace neon {

__device__ __forceinline__ xf4 xg_mfma(float a, float b, xf4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ int bitrev6(int t) { return (int)(__builtin_bitreverse32((uint32_t)t) >> 26); }

// The binary counter: S merges with m waiting sums, then waits itself (m < 6)
// or is the total (m = 6: p[0] .. p[5] all taken).
template <int NT, int LV = 0>
__device__ __forceinline__ void xg_merge(xf4 (&s)[NT], xf4 (&p)[6][NT], int m) {
  if constexpr (LV < 6) {
    if (m == LV) {
#pragma unroll
      for (int n = 0; n < NT; ++n) p[LV][n] = s[n];
      // (differs per level: the stores are not merged into one through an
      // index, which would put p in scratch memory)
      asm volatile("; waits at level %0" ::"n"(LV));
    } else {
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[n][r] = __fadd_rn(p[LV][n][r], s[n][r]);
      xg_merge<NT, LV + 1>(s, p, m);
    }
  }
}

// ===========================================================================
// Pairs by expert: pair[] holds the pairs q = row k + slot grouped by expert,
// off[e] the first of expert e's, toff[e] its first tile of 16 pairs (E + 1
// entries each), tile[t] = first pair | pair count << 16 (toff[E] tiles).  One block; the order of
// an expert's pairs is free (a pair's results go to its own place).  An id
// outside [0, E) joins no expert.
// ===========================================================================
__global__ __launch_bounds__(1024) void k_xg_group(const int32_t* __restrict__ idx, int nk, int E,
                                                   int32_t* __restrict__ pair,
                                                   int32_t* __restrict__ toff,
                                                   uint32_t* __restrict__ tile,
                                                   int32_t* __restrict__ err) {
  __shared__ int cnt[256], off[256], ws[4][2];
  constexpr int PT = kXgMaxPairs / 1024;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  if (tid < 256) cnt[tid] = 0;
  __syncthreads();
  int id[PT], rank[PT];
#pragma unroll
  for (int m = 0; m < PT; ++m) {
    const int q = tid + 1024 * m;
    id[m] = q < nk ? idx[q] : -1;
    if (q < nk && (unsigned)id[m] >= (unsigned)E) {
      flag_dev_err(err, kDevErrExpertId);
      id[m] = -1;
    }
    rank[m] = id[m] >= 0 ? atomicAdd(&cnt[id[m]], 1) : 0;
  }
  __syncthreads();
  const int c = tid < 256 ? cnt[tid] : 0, nt = (c + 15) >> 4;
  int pc = c, pt = nt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int a = __shfl_up(pc, o, 64), b = __shfl_up(pt, o, 64);
    if (lane >= o) { pc += a; pt += b; }
  }
  if (lane == 63 && w < 4) { ws[w][0] = pc; ws[w][1] = pt; }
  __syncthreads();
  if (tid < 256) {
    int bc = 0, bt = 0;
    for (int v = 0; v < w; ++v) { bc += ws[v][0]; bt += ws[v][1]; }
    const int o0 = bc + pc - c, t0 = bt + pt - nt;
    off[tid] = o0;
    if (tid <= E) toff[tid] = t0;  // experts from E on are empty
    if (tid == 255 && E == 256) toff[256] = bt + pt;
    for (int m = 0; m < nt; ++m)
      tile[t0 + m] = (uint32_t)(o0 + 16 * m) | ((uint32_t)min(16, c - 16 * m) << 16);
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < PT; ++m)
    if (id[m] >= 0) pair[off[id[m]] + rank[m]] = tid + 1024 * m;
}

// ===========================================================================
// Expert inputs in B operand order: xt[tile][unit][lane][8] bf16, lane j + 16 kk
// holding elements kk, 4 + kk, .. 28 + kk of the unit of the tile's pair j (a
// place past the tile's pairs repeats the last): one 16-byte load per lane and
// unit, 1 KB contiguous.  grid (max tiles, 4), 256 threads.
// ===========================================================================
__device__ __forceinline__ uint32_t xg_half(const uint4& v, int e) {
  const uint32_t w = e < 2 ? v.x : e < 4 ? v.y : e < 6 ? v.z : v.w;
  return (e & 1) ? w >> 16 : w & 0xFFFFu;
}
__global__ __launch_bounds__(256) void k_xg_pack_pairs(const uint16_t* __restrict__ x,
                                                       const int32_t* __restrict__ pair,
                                                       const int32_t* __restrict__ toff,
                                                       const uint32_t* __restrict__ tile, int E,
                                                       int k, int H, uint4* __restrict__ xt) {
  const int t = blockIdx.x, U = H / 32;
  if (t >= toff[E]) return;
  const uint32_t ti = tile[t];
  const int first = ti & 0xFFFF, cnt = ti >> 16;
  for (int it = blockIdx.y * 256 + threadIdx.x; it < 16 * U; it += gridDim.y * 256) {
    const int j = it / U, u = it % U;
    const uint4* src = reinterpret_cast<const uint4*>(
        x + (size_t)(pair[first + min(j, cnt - 1)] / k) * H) + 4 * u;
    uint4 v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = src[q];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      uint32_t o[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) o[q] = xg_half(v[q], kk) | (xg_half(v[q], 4 + kk) << 16);
      xt[((size_t)t * U + u) * 64 + kk * 16 + j] = make_uint4(o[0], o[1], o[2], o[3]);
    }
  }
}

// ===========================================================================
// The expert products: grid (rows / 32, E), 4 waves.  Block (x, e) holds rows
// 32 x .. 32 x + 31 of expert e in LDS (codes as stored, scales as bf16), and
// each wave takes every fourth tile of 16 pairs: two 16 x 16 outputs, the whole
// K.  Bound: the chains of a wave, 16 matrix instructions of 32 cycles per unit
// one after the other, and waves without a tile: the matrix units are 50% busy
// at 512 rows (4 or 5 tiles per expert; 960 us gate_up, 531 us down) and 40% at
// 240 rows (626, 354 us).  The inputs of the next three units are on their way.
//   GATE_UP: SwiGLU of the interleaved (gate, up) rows, which sit in adjacent
//            registers of a lane, stored as bf16 in the next product's tiles;
//   DOWN:    ybuf[pair][row] = dot + bias (fp32), combined by k_moe_combine.
// ===========================================================================
struct XgExpertArgs {
  const uint8_t *codes, *scales;   // [E][N][K/2], [E][N][K/32]
  const uint16_t* bias;            // [E][N]
  const uint4* xt;                 // input tiles
  const int32_t *pair, *toff;
  const uint32_t* tile;
  uint16_t* yt;                    // GATE_UP: output tiles (N / 2 columns)
  float* ybuf;                     // DOWN: [pair][N]
  int N, K;
  float alpha, limit;
};

// bytes of LDS for rows of U units
static size_t xg_expert_lds(int U) {
  return (size_t)32 * (U | 1) * 16 + (size_t)U * 32 * 2 + (size_t)(U + 4) * 4;
}

template <bool GATE_UP>
__global__ __launch_bounds__(256, 3) void k_xg_experts(XgExpertArgs a) {
  extern __shared__ __align__(16) char lds[];
  const int e = blockIdx.y, tb = a.toff[e], te = a.toff[e + 1];
  if (tb == te) return;
  const int U = a.K / 32, SU = U | 1;  // odd row stride in units: the 16 rows' reads hit all banks
  uint4* cs = reinterpret_cast<uint4*>(lds);
  uint16_t* sc = reinterpret_cast<uint16_t*>(lds + (size_t)32 * SU * 16);  // 2^(s - 127) as bf16
  int* tab = reinterpret_cast<int*>(sc + (size_t)U * 32);
  const int tid = threadIdx.x, lane = tid & 63;
  // tiles rotate over the waves from block to block (a wave sits on one SIMD)
  const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) + blockIdx.x) & 3;
  const size_t row0 = (size_t)e * a.N + (size_t)blockIdx.x * 32;
  const uint4* csrc = reinterpret_cast<const uint4*>(a.codes + row0 * (a.K / 2));
  for (int p = tid; p < 32 * U; p += 256) {
    const int r = p / U, u = p - r * U;
    cs[r * SU + u] = csrc[p];
    const uint32_t s = a.scales[row0 * U + p];
    sc[u * 32 + r] = s == 0 ? 0x0040 : s == 0xFF ? 0x7FC0 : (uint16_t)(s << 7);
  }
  // the units in chain order (requests run ahead by it)
  if (tid < 64) {
    const int l = bitrev6(tid);
    const int n = l < U ? (U - l + 63) / 64 : 0;
    int at = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(at, o, 64);
      if (lane >= o) at += v;
    }
    at -= n;
    for (int p = 0; p < n; ++p) tab[at + p] = l + 64 * p;
    if (tid < 4) tab[U + tid] = 0;  // past the end: a unit that exists, dropped
  }
  __syncthreads();
  const int i = lane & 15, kk = lane >> 4;
  const int UO = a.N / 64;          // GATE_UP: units of an output row
  const uint4* crow = cs + i * SU;
  const uint16_t* srow = sc + 4 * kk;
  for (int t = tb + wave; t < te; t += 4) {
    const uint4* xs = a.xt + (size_t)t * U * 64 + lane;
    // unit n: codes and scales from LDS one unit ahead, inputs three
    int n = 0, u1 = __builtin_amdgcn_readfirstlane(tab[1]);
    uint4 x0 = xs[(size_t)__builtin_amdgcn_readfirstlane(tab[0]) * 64];
    uint4 x1 = xs[(size_t)u1 * 64];
    uint4 x2 = xs[(size_t)__builtin_amdgcn_readfirstlane(tab[2]) * 64];
    int u3 = __builtin_amdgcn_readfirstlane(tab[3]);
    int u2 = __builtin_amdgcn_readfirstlane(tab[2]);
    uint4 c[2];
    uint2 f[2];
    auto rows = [&](int u) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        c[rt] = crow[rt * 16 * SU + u];
        f[rt] = *reinterpret_cast<const uint2*>(srow + u * 32 + rt * 16);
      }
    };
    rows(__builtin_amdgcn_readfirstlane(tab[0]));
    xf4 acc[2];
    // acc += scale * (the next unit's chain); acc starts a chain when `first`
    auto unit = [&](bool first) {
      float xv[8] = {bf_lo(x0.x), bf_hi(x0.x), bf_lo(x0.y), bf_hi(x0.y),
                     bf_lo(x0.z), bf_hi(x0.z), bf_lo(x0.w), bf_hi(x0.w)};
      float w[2][8];
      uint2 fc[2];
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const uint32_t cw[4] = {c[rt].x >> (4 * kk), c[rt].y >> (4 * kk), c[rt].z >> (4 * kk),
                                c[rt].w >> (4 * kk)};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          w[rt][2 * q] = fp4x2_to_f32<0>(cw[q]).x;
          w[rt][2 * q + 1] = fp4x2_to_f32<2>(cw[q]).x;
        }
        fc[rt] = f[rt];
        pin8(w[rt]);
      }
      pin8(xv);
      __builtin_amdgcn_sched_barrier(0);
      x0 = x1;
      x1 = x2;
      x2 = xs[(size_t)u3 * 64];
      rows(u1);
      u1 = u2;
      u2 = u3;
      ++n;
      u3 = tab[min(n + 3, U)];
      __builtin_amdgcn_sched_barrier(0);
      xf4 tt[2] = {xf4{0.0f, 0.0f, 0.0f, 0.0f}, xf4{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) tt[rt] = xg_mfma(w[rt][s], xv[s], tt[rt]);
      asm volatile("" ::"v"(tt[0]), "v"(tt[1]));
      __builtin_amdgcn_sched_barrier(0);
      u3 = __builtin_amdgcn_readfirstlane(u3);
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const float fv[4] = {bf_lo(fc[rt].x), bf_hi(fc[rt].x), bf_lo(fc[rt].y), bf_hi(fc[rt].y)};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[rt][r] = __fadd_rn(first ? 0.0f : acc[rt][r], __fmul_rn(tt[rt][r], fv[r]));
      }
    };
    xf4 p0[2], p1[2], p2[2], p3[2], p4[2], p5[2];
    auto add = [&](xf4 (&s)[2], const xf4 (&o)[2]) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[rt][r] = __fadd_rn(o[rt][r], s[rt][r]);
    };
    auto keep = [&](xf4 (&d)[2]) { d[0] = acc[0]; d[1] = acc[1]; };
    for (int tt = 0; tt < 8; ++tt) {
      const int lo = (tt & 1) * 4 + (tt & 2) + (tt >> 2);
      // eight chains, l = lo + 8 {0, 4, 2, 6, 1, 5, 3, 7}: off 32, 16, 8
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        const int l = lo + 8 * ((m & 1) * 4 + (m & 2) + (m >> 2));
        if (l < U) {
          unit(true);
          for (int u = l + 64; u < U; u += 64) unit(false);
        } else {  // a row of fewer than 64 units
          acc[0] = acc[1] = xf4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        if ((m & 1) == 0) { keep(p0); continue; }
        add(acc, p0);
        if ((m & 2) == 0) { keep(p1); continue; }
        add(acc, p1);
        if ((m & 4) == 0) { keep(p2); continue; }
        add(acc, p2);
      }
      // off 4, 2, 1
      if ((tt & 1) == 0) {
        keep(p3);
        asm volatile("; level 3");
      } else {
        add(acc, p3);
        if ((tt & 2) == 0) {
          keep(p4);
          asm volatile("; level 4");
        } else {
          add(acc, p4);
          if ((tt & 4) == 0) {
            keep(p5);
            asm volatile("; level 5");
          } else {
            add(acc, p5);
          }
        }
      }
    }
    // acc: the totals (the last chain merges all six waiting sums)
    const uint32_t ti = a.tile[t];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const int row = blockIdx.x * 32 + rt * 16 + 4 * kk;
      const uint2 bw = *reinterpret_cast<const uint2*>(a.bias + (size_t)e * a.N + row);
      const float b4[4] = {bf_lo(bw.x), bf_hi(bw.x), bf_lo(bw.y), bf_hi(bw.y)};
      if constexpr (GATE_UP) {
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2) {
          const int c = row / 2 + c2, uo = c >> 5, ee = c & 31;
          const float v = swiglu_clamp(__fadd_rn(acc[rt][2 * c2], b4[2 * c2]),
                                       __fadd_rn(acc[rt][2 * c2 + 1], b4[2 * c2 + 1]), a.alpha,
                                       a.limit);
          a.yt[((((size_t)t * UO + uo) * 64) + (ee & 3) * 16 + i) * 8 + (ee >> 2)] = f2bf(v);
        }
      } else {
        if (i < (int)(ti >> 16)) {
          const int q = a.pair[(ti & 0xFFFF) + i];
          *reinterpret_cast<float4*>(a.ybuf + (size_t)q * a.N + row) =
              make_float4(__fadd_rn(acc[rt][0], b4[0]), __fadd_rn(acc[rt][1], b4[1]),
                          __fadd_rn(acc[rt][2], b4[2]), __fadd_rn(acc[rt][3], b4[3]));
        }
      }
    }
  }
}

// ===========================================================================
// Dense rows (weights or inputs) in operand order: out[row tile][chain l][pp]
// [lane][2 units][2] bf16, lane i + 16 kk holding elements kk and 4 + kk of
// row i's units l + 64 (2 pp) and l + 64 (2 pp + 1).  A unit past K is `pad`
// (-0.0 for weights, +0 for inputs: their product -0 leaves every chain value
// as it is), rows past n re-read row n - 1.  One thread per lane of a piece.
// ===========================================================================
__global__ __launch_bounds__(256) void k_xg_pack_rows(const uint16_t* __restrict__ x, int n, int K,
                                                      int P2, uint32_t pad,
                                                      uint2* __restrict__ out) {
  const int U = K / 8, lane = threadIdx.x & 63, i = lane & 15, kk = lane >> 4;
  const int pieces = 64 * P2;
  const uint4* row = reinterpret_cast<const uint4*>(
      x + (size_t)min((int)blockIdx.x * 16 + i, n - 1) * K);
  uint2* o = out + (size_t)blockIdx.x * pieces * 64 + lane;
  // consecutive waves take consecutive chains of one pp: whole lines of a row
  for (int c = blockIdx.y * 4 + (threadIdx.x >> 6); c < pieces; c += gridDim.y * 4) {
    const int l = c & 63, pp = c >> 6;
    uint32_t w[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int u = l + 64 * (2 * pp + h);
      const uint4 v = row[min(u, U - 1)];
      const uint32_t lo = (kk & 2) ? v.y : v.x, hi = (kk & 2) ? v.w : v.z;
      const uint32_t a = (kk & 1) ? lo >> 16 : lo & 0xFFFFu;
      const uint32_t b = (kk & 1) ? hi & 0xFFFF0000u : hi << 16;
      w[h] = u < U ? a | b : pad;
    }
    o[((size_t)l * P2 + pp) * 64] = make_uint2(w[0], w[1]);
  }
}

// ===========================================================================
// Dense product of packed rows: y[m][n] = bf16(dot + bias[n]), or with RESID
// y = bf16(y + bf16(dot + bias)).  grid (N / 64, ceil(M / 32)), 4 waves: wave
// (w & 1) takes 32 of the block's 64 weight rows, (w >> 1) 16 of its 32 input
// rows.  A chain is 4 P2 matrix instructions per output tile; the next chain's
// operands are requested before it.
// ===========================================================================
template <int P2, bool RESID>
__global__ __launch_bounds__(256, 2) void k_xg_dense(const uint2* __restrict__ wp,
                                                     const uint2* __restrict__ xp,
                                                     const uint16_t* __restrict__ bias,
                                                     uint16_t* __restrict__ y, int M, int N) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nt = blockIdx.x * 4 + (wave & 1) * 2, mt = blockIdx.y * 2 + (wave >> 1);
  if (mt * 16 >= M || nt * 16 >= N) return;
  const bool two = (nt + 1) * 16 < N;
  constexpr size_t TS = (size_t)64 * P2 * 64;  // uint2 per tile
  const uint2* w0 = wp + (size_t)nt * TS + lane;
  const uint2* w1 = wp + (size_t)(two ? nt + 1 : nt) * TS + lane;
  const uint2* xr = xp + (size_t)mt * TS + lane;
  uint2 rw0[P2], rw1[P2], rx[P2];
  auto load = [&](int l) {
    const size_t o = (size_t)l * P2 * 64;
#pragma unroll
    for (int pp = 0; pp < P2; ++pp) {
      rw0[pp] = w0[o + pp * 64];
      rw1[pp] = w1[o + pp * 64];
      rx[pp] = xr[o + pp * 64];
    }
  };
  load(0);
  xf4 p[6][2], acc[2];
  for (int t = 0; t < 64; ++t) {
    float a0[4 * P2], a1[4 * P2], b[4 * P2];
#pragma unroll
    for (int pp = 0; pp < P2; ++pp) {
      asm volatile("" : "+v"(rw0[pp].x), "+v"(rw0[pp].y), "+v"(rw1[pp].x), "+v"(rw1[pp].y),
                        "+v"(rx[pp].x), "+v"(rx[pp].y));
      a0[4 * pp] = bf_lo(rw0[pp].x); a0[4 * pp + 1] = bf_hi(rw0[pp].x);
      a0[4 * pp + 2] = bf_lo(rw0[pp].y); a0[4 * pp + 3] = bf_hi(rw0[pp].y);
      a1[4 * pp] = bf_lo(rw1[pp].x); a1[4 * pp + 1] = bf_hi(rw1[pp].x);
      a1[4 * pp + 2] = bf_lo(rw1[pp].y); a1[4 * pp + 3] = bf_hi(rw1[pp].y);
      b[4 * pp] = bf_lo(rx[pp].x); b[4 * pp + 1] = bf_hi(rx[pp].x);
      b[4 * pp + 2] = bf_lo(rx[pp].y); b[4 * pp + 3] = bf_hi(rx[pp].y);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (t + 1 < 64) load(bitrev6(t + 1));
    __builtin_amdgcn_sched_barrier(0);
    acc[0] = acc[1] = xf4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 4 * P2; ++s) {
      acc[0] = xg_mfma(a0[s], b[s], acc[0]);
      acc[1] = xg_mfma(a1[s], b[s], acc[1]);
    }
    xg_merge<2>(acc, p, __builtin_ctz(~(uint32_t)t));
  }
  const int m = mt * 16 + (lane & 15);
  if (m >= M) return;
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    if (rt == 1 && !two) break;
    const int n = (nt + rt) * 16 + 4 * (lane >> 4);
    float v[4] = {acc[rt][0], acc[rt][1], acc[rt][2], acc[rt][3]};
    if (bias != nullptr) {
      const uint2 bw = *reinterpret_cast<const uint2*>(bias + n);
      v[0] = __fadd_rn(v[0], bf_lo(bw.x)); v[1] = __fadd_rn(v[1], bf_hi(bw.x));
      v[2] = __fadd_rn(v[2], bf_lo(bw.y)); v[3] = __fadd_rn(v[3], bf_hi(bw.y));
    }
    uint2* yp = reinterpret_cast<uint2*>(y + (size_t)m * N + n);
    uint32_t o0 = pack_bf2(v[0], v[1]), o1 = pack_bf2(v[2], v[3]);
    if (RESID) {
      const uint2 h = *yp;
      o0 = pack_bf2(__fadd_rn(bf_lo(h.x), bf_lo(o0)), __fadd_rn(bf_hi(h.x), bf_hi(o0)));
      o1 = pack_bf2(__fadd_rn(bf_lo(h.y), bf_lo(o1)), __fadd_rn(bf_hi(h.y), bf_hi(o1)));
    }
    *yp = make_uint2(o0, o1);
  }
}

// ---- launchers ------------------------------------------------------------
// chain passes in pairs; 0 when K is not covered
static int xg_p2(int K) {
  const int P2 = ((K / 8 + 63) / 64 + 1) / 2;
  return K % 8 == 0 && P2 >= 1 && P2 <= 4 ? P2 : 0;
}
size_t xg_packed_bytes(int rows, int K) {
  return (size_t)((rows + 15) / 16) * 64 * xg_p2(K) * 64 * sizeof(uint2);
}
int xg_max_tiles(int pairs, int E) { return (pairs + 15 * (E < pairs ? E : pairs)) / 16; }
size_t xg_tile_bytes(int pairs, int E, int K) {
  return (size_t)xg_max_tiles(pairs, E) * (K / 32) * 1024;
}
constexpr int kXgMaxK = 5120;  // expert reductions: 32 rows of codes and scales in LDS
bool xg_supported(int H, int I, int qd, int qkv_rows, int E) {
  return xg_p2(H) && xg_p2(qd) && H % 32 == 0 && I % 32 == 0 && H <= kXgMaxK && I <= kXgMaxK &&
         qkv_rows % 16 == 0 && H % 16 == 0 && E <= 256;
}
// opts the expert kernels in to the LDS of their longest rows
hipError_t xg_prepare() {
  const int lds = (int)xg_expert_lds(kXgMaxK / 32);
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_xg_experts<true>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e == hipSuccess)
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_xg_experts<false>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  return e;
}

void launch_xg_dense(const uint16_t* W, const uint16_t* bias, const uint16_t* x, uint16_t* y, int M,
                     int N, int K, bool resid, void* wp, void* xp, hipStream_t st) {
  const int P2 = xg_p2(K);
  uint2 *w = (uint2*)wp, *xx = (uint2*)xp;
  hipLaunchKernelGGL(k_xg_pack_rows, dim3((N + 15) / 16, 4), dim3(256), 0, st, W, N, K, P2,
                     0x80008000u, w);
  hipLaunchKernelGGL(k_xg_pack_rows, dim3((M + 15) / 16, 16), dim3(256), 0, st, x, M, K, P2, 0u, xx);
  const dim3 grid((N + 63) / 64, (M + 31) / 32);
#define XD(P)                                                                                  \
  if (resid) hipLaunchKernelGGL((k_xg_dense<P, true>), grid, dim3(256), 0, st, w, xx, bias, y, \
                                M, N);                                                         \
  else hipLaunchKernelGGL((k_xg_dense<P, false>), grid, dim3(256), 0, st, w, xx, bias, y, M, N)
  switch (P2) {
    case 1: XD(1); break;
    case 2: XD(2); break;
    case 3: XD(3); break;
    default: XD(4); break;
  }
#undef XD
}

void launch_xg_moe(const MoeArgs& a, const XgMoeScratch& s, hipStream_t st) {
  const int nk = a.B * a.k, tiles = xg_max_tiles(nk, a.E);
  hipLaunchKernelGGL(k_xg_group, dim3(1), dim3(1024), 0, st, a.idx, nk, a.E, s.pair, s.toff, s.tile,
                     a.err);
  hipLaunchKernelGGL(k_xg_pack_pairs, dim3(tiles, 4), dim3(256), 0, st, a.xn, s.pair, s.toff, s.tile,
                     a.E, a.k, a.H, (uint4*)s.xt);
  XgExpertArgs g{};
  g.codes = a.gu_codes; g.scales = a.gu_scales; g.bias = a.gu_bias; g.xt = (const uint4*)s.xt;
  g.pair = s.pair; g.toff = s.toff; g.tile = s.tile; g.yt = (uint16_t*)s.yt;
  g.N = 2 * a.I; g.K = a.H; g.alpha = a.alpha; g.limit = a.limit;
  hipLaunchKernelGGL(k_xg_experts<true>, dim3(g.N / 32, a.E), dim3(256), xg_expert_lds(g.K / 32), st, g);
  XgExpertArgs d = g;
  d.codes = a.dn_codes; d.scales = a.dn_scales; d.bias = a.dn_bias; d.xt = (const uint4*)s.yt;
  d.yt = nullptr; d.ybuf = s.ybuf; d.N = a.H; d.K = a.I;
  hipLaunchKernelGGL(k_xg_experts<false>, dim3(d.N / 32, a.E), dim3(256), xg_expert_lds(d.K / 32), st, d);
  launch_moe_combine(s.ybuf, a.score, a.idx, a.B, a.E, a.k, a.H, a.out, st);
}

}  // namespace neon
