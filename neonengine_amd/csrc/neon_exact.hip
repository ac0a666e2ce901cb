// neon_exact.hip -- the canonical fp32 dot products on the fp32 matrix
// instructions.
//
// v_mfma_f32_4x4x1_16b_f32 forms 16 independent 4 x 4 outer products and adds
// each product to its accumulator with one correctly rounded fused
// multiply-add: D = fmaf(a, b, C), bit for bit, denormals, infinities and
// NaN included (compared with v_fma_f32 on 16.8M operand triples of each of
// six kinds: E2M1 x bf16, bf16 x bf16, any bits, wide exponents, denormal
// inputs, denormal results).  So a chain of them is the canonical chain of
// the one-row kernels, with 4 weight rows x 4 input rows x 16 chains per
// instruction in place of 64 products, and every dot product here is
// bit-identical to theirs (the butterfly's pairings are kept as well).
//
// Lane layout: lane 4 b + i of the A operand holds row i of block b, lane
// 4 b + j of B column j, and D's register i at lane 4 b + j is output (i, j)
// of block b.  Block b is one canonical lane partial: in group g the lanes
// own the units u = 16 g + b, so a lane reads its own row's units straight
// from the stored row (256 contiguous bytes per row and group).
#include "neon_common.hpp"
#include "neon_exact_index.hpp"
#include "neon_exact_routes.hpp"
#include "neon_internal.hpp"

namespace neon {

__device__ __forceinline__ xf4 xm_mfma(float a, float b, xf4 c) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
}

// the value of lane I of the caller's quad (lanes 4 b .. 4 b + 3)
template <int I>
__device__ __forceinline__ float quad_bcast(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                                       0, __builtin_bit_cast(int, v), I * 0x55, 0xF, 0xF, true));
}

// 2^(s - 127) as fp32, NaN for 0xFF: t * it is e8m0_scale(t, s), one rounding
// of an exact power-of-two scaling.  ldexp of the denormal 2^-127 gives every
// finite one and +inf for 0xFF, and fma(f, 0, f) turns only that into NaN.
__device__ __forceinline__ float e8m0_f32(uint32_t s) {
  const float f = __builtin_amdgcn_ldexpf(__builtin_bit_cast(float, 0x00400000u), (int)s);
  return __builtin_fmaf(f, 0.0f, f);
}

// The last steps of the butterfly: N values per lane hold the sums over off =
// 32 and 16 already; block bits 3..0 (off 8, 4, 2, 1) sit in lane bits 5..2.
// While more than one value is left a lane keeps half of them (fp32 addition
// commutes, so the totals are those of N separate butterflies).  Value v ends
// in the lanes whose bits 5, 4, .. spell v from its top bit down.
template <int N, int OFF = 32>
__device__ __forceinline__ float xm_fold(const float (&a)[N], int lane) {
  if constexpr (N == 1) {
    const float v = __fadd_rn(a[0], xor_lane<OFF>(a[0]));
    if constexpr (OFF > 4) {
      const float w[1] = {v};
      return xm_fold<1, OFF / 2>(w, lane);
    } else {
      return v;
    }
  } else {
    static_assert(OFF >= 4, "xm_fold: at most 16 values");
    const bool up = (lane & OFF) != 0;
    float h[N / 2];
#pragma unroll
    for (int i = 0; i < N / 2; ++i)
      h[i] = __fadd_rn(up ? a[i + N / 2] : a[i], xor_lane<OFF>(up ? a[i] : a[i + N / 2]));
    if constexpr (N / 2 == 1 && OFF == 4) return h[0];
    else return xm_fold<N / 2, OFF / 2>(h, lane);
  }
}

// ---------------------------------------------------------------------------
// MXFP4 rows: RQ quads of 4 weight rows against 4 input rows.  NG groups of 16
// units cover the row's U = K / 32 units (a lane past U re-reads the last unit
// and its value is dropped).  The groups run in the order 0, 4, .. 2, 6, ..
// 1, 5, .. 3, 7, ..: groups of one residue mod 4 hold the units l, l + 64, ..
// of the same lanes l, off 32 pairs residues 0-2 and 1-3, off 16 their sums.
// ---------------------------------------------------------------------------
template <int NG>
__device__ constexpr int xm_order(int o) {
  int n = 0;
  for (int li = 0; li < 4; ++li) {
    const int lg = li == 1 ? 2 : li == 2 ? 1 : li;
    for (int g = lg; g < NG; g += 4, ++n)
      if (n == o) return g;
  }
  return 0;
}
// groups requested ahead: a divisor of NG
template <int NG>
constexpr int xm_depth() { return NG == 6 ? 3 : NG == 8 ? 4 : NG == 4 ? 2 : NG; }

// one work item of a wave: its first row's codes and scales (uniform) and the
// lane's input row; row quads from `quads` on re-read quad 0 (past the matrix)
struct XmItem {
  const uint8_t *codes, *scales;
  const uint16_t* x;
  int quads;
};

// The stream of a wave: the codes, scales and inputs of the next D groups are
// always on their way, across items (loads return in the order they were
// requested, so an input requested later than the rows would wait for them).
// Inputs come from LDS as fp32 (XL; xs, in the lanes' order: no conversion), or
// from rows in the order of xm_act_at.
template <int RQ, int NG, bool XL>
struct XmStream {
  static constexpr int D = xm_depth<NG>();
  uint4 c[D][RQ];
  uint32_t s[D][RQ];
  uint4 x[XL ? 1 : D][4];

  // (the lane goes through an empty asm: the addresses of all groups are not
  // kept in registers across the item loop)
  __device__ __forceinline__ void rows(const XmItem& it, int o, int U, int lane) {
    asm volatile("" : "+v"(lane));
    const uint32_t u = (uint32_t)((lane & 3) * U + min(16 * xm_order<NG>(o) + (lane >> 2), U - 1));
#pragma unroll
    for (int r = 0; r < RQ; ++r) {
      const uint32_t ur = (r < it.quads ? 4 * r : 0) * U;  // units before the quad
      c[o % D][r] = load_weight16(it.codes + (size_t)ur * 16 + u * 16);
      s[o % D][r] = load_weight1(it.scales + ur + u);
    }
  }
  __device__ __forceinline__ void input(const XmItem& it, int o, int U, int lane) {
    asm volatile("" : "+v"(lane));
    const XmPieces at = xm_pieces(xm_order<NG>(o), lane >> 2, U);
    const uint4* p = reinterpret_cast<const uint4*>(it.x) + at.first;
#pragma unroll
    for (int q = 0; q < 4; ++q) x[o % D][q] = p[q * at.step];
  }
  __device__ __forceinline__ void start(const XmItem& it, int U, int lane) {
#pragma unroll
    for (int o = 0; o < D; ++o) {
      if constexpr (!XL) input(it, o, U, lane);
      rows(it, o, U, lane);
    }
  }

  // The canonical partials of the item's rows, summed over off = 32 and 16:
  // block b's values in lanes 4 b + j.  Requests the first groups of `next`.
  // Per group: a quarter of the unit's conversions, then that quarter of its
  // chain, four times: a change between vector and matrix instructions costs
  // cycles, so each runs in bursts.
  __device__ __forceinline__ void item(float (&out)[4 * RQ], const XmItem& it,
                                       const XmItem& next, int U, int lane,
                                       const float4* xs = nullptr) {
    xf4 sum[RQ], half[RQ], a[RQ];
#pragma unroll
    for (int o = 0; o < NG; ++o) {
      const int g = xm_order<NG>(o), lg = g & 3;
      if (g < 4) {
#pragma unroll
        for (int r = 0; r < RQ; ++r) a[r] = xf4{0.0f, 0.0f, 0.0f, 0.0f};
      }
      xf4 t[RQ];
#pragma unroll
      for (int r = 0; r < RQ; ++r) t[r] = xf4{0.0f, 0.0f, 0.0f, 0.0f};
      float f[RQ];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float w[RQ][8];
        float xv[8];
        if constexpr (XL) {
          const float4 v0 = xs[(8 * g + 2 * q) * 64 + lane], v1 = xs[(8 * g + 2 * q + 1) * 64 + lane];
          xv[0] = v0.x; xv[1] = v0.y; xv[2] = v0.z; xv[3] = v0.w;
          xv[4] = v1.x; xv[5] = v1.y; xv[6] = v1.z; xv[7] = v1.w;
        } else {
          uint4 xw = x[o % D][q];
          asm volatile("" : "+v"(xw.x), "+v"(xw.y), "+v"(xw.z), "+v"(xw.w));
          xv[0] = bf_lo(xw.x); xv[1] = bf_hi(xw.x); xv[2] = bf_lo(xw.y); xv[3] = bf_hi(xw.y);
          xv[4] = bf_lo(xw.z); xv[5] = bf_hi(xw.z); xv[6] = bf_lo(xw.w); xv[7] = bf_hi(xw.w);
        }
#pragma unroll
        for (int r = 0; r < RQ; ++r) {
          const uint4& cc = c[o % D][r];
          uint32_t cw = q == 0 ? cc.x : q == 1 ? cc.y : q == 2 ? cc.z : cc.w;
          asm volatile("" : "+v"(cw));
          const float2_v v0 = fp4x2_to_f32<0>(cw), v1 = fp4x2_to_f32<1>(cw);
          const float2_v v2 = fp4x2_to_f32<2>(cw), v3 = fp4x2_to_f32<3>(cw);
          w[r][0] = v0.x; w[r][1] = v0.y; w[r][2] = v1.x; w[r][3] = v1.y;
          w[r][4] = v2.x; w[r][5] = v2.y; w[r][6] = v3.x; w[r][7] = v3.y;
          if (q == 3) {
            uint32_t sv = s[o % D][r];
            asm volatile("" : "+v"(sv));
            f[r] = e8m0_f32(sv);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (q == 3) {  // the words are converted: their places take what comes next
          const XmItem& from = o + D < NG ? it : next;
          if constexpr (!XL) input(from, (o + D) % NG, U, lane);
          rows(from, (o + D) % NG, U, lane);
          __builtin_amdgcn_sched_barrier(0);
        }
        // (empty asm statements keep the two kinds apart: the compiler would
        // otherwise float the matrix instructions to the end and hold every
        // converted value until then)
#pragma unroll
        for (int r = 0; r < RQ; ++r) pin8(w[r]);
        pin8(xv);
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int r = 0; r < RQ; ++r) t[r] = xm_mfma(w[r][e], xv[e], t[r]);
#pragma unroll
        for (int r = 0; r < RQ; ++r) asm volatile("" ::"v"(t[r]));
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int r = 0; r < RQ; ++r) {
        const float f4[4] = {quad_bcast<0>(f[r]), quad_bcast<1>(f[r]), quad_bcast<2>(f[r]),
                             quad_bcast<3>(f[r])};
#pragma unroll
        for (int i = 0; i < 4; ++i) t[r][i] = __fmul_rn(t[r][i], f4[i]);
      }
      if (16 * g + 16 > U) {  // padded units add +0: a partial is never -0
        const bool on = 16 * g + (lane >> 2) < U;
#pragma unroll
        for (int r = 0; r < RQ; ++r)
#pragma unroll
          for (int i = 0; i < 4; ++i) t[r][i] = on ? t[r][i] : 0.0f;
      }
#pragma unroll
      for (int r = 0; r < RQ; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) a[r][i] = __fadd_rn(a[r][i], t[r][i]);
      if (g + 4 >= NG) {  // the residue's last group (absent residues add +0 below)
#pragma unroll
        for (int r = 0; r < RQ; ++r)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (lg == 0) sum[r][i] = a[r][i];
            else if (lg == 2) sum[r][i] = __fadd_rn(sum[r][i], a[r][i]);
            else if (lg == 1) half[r][i] = a[r][i];
            else half[r][i] = __fadd_rn(half[r][i], a[r][i]);
          }
      }
    }
#pragma unroll
    for (int r = 0; r < RQ; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        out[4 * r + i] = NG > 1 ? __fadd_rn(sum[r][i], half[r][i]) : sum[r][i];
  }
};

// ===========================================================================
// Experts of a batch (2 rows and more), each used expert's rows read once for
// all the pairs (row b, slot s; pair q = b k + s) that chose it.
//
// gate_up: grid (ceil(tasks / (4 kXmGuTasks)), E), 4 waves.  Block (x, e)
// serves expert e; a task is 6 intermediate columns (12 rows, gate and up
// interleaved).  Four of the expert's pairs at a time sit in LDS as fp32, and
// each wave streams its tasks' rows against them.
// Bound: matrix instructions and the conversions around them, which do not
// overlap in a wave (B = 16: matrix units 30% busy, vector units 44%, waves
// waiting 39% of their time), beside 4.5 TB/s of memory reads, 1.6 times the
// bytes of the rows: a group's 16 scale bytes fetch a 128-byte line each time.
// A quad of pairs costs what 1.7 single ones cost the vector kernels; from two
// pairs per expert on that wins.  20b, B = 16 (64 pairs, 28 experts): gate_up
// 100 -> 88 us, down 57 -> 44 us; B = 64 616 -> 309 us per layer.
// ===========================================================================
constexpr int kXmGuRq = 3;     // row quads per gate_up task
constexpr int kXmGuTasks = 3;  // tasks per wave
static_assert(kXmGuColumns == 2 * kXmGuRq * 4 * kXmGuTasks, "columns of a block");

template <int NG>
__global__ __launch_bounds__(256, 2) void k_xm_gate_up(
    const uint8_t* __restrict__ gu_codes, const uint8_t* __restrict__ gu_scales,
    const uint16_t* __restrict__ gu_bias, const int32_t* __restrict__ idx,
    const uint16_t* __restrict__ xn, uint16_t* __restrict__ act, int nk, int H, int I, int k,
    float alpha, float limit) {
  constexpr int RQ = kXmGuRq, COLS = 2 * RQ;
  __shared__ uint16_t list[kXmMaxPairs];
  __shared__ __align__(16) float4 xs[8 * NG * 64];  // [8 g + e / 4][lane]: the quad's inputs
  const int U = H / 32, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 3, e = blockIdx.y;
  const int tasks = (I + COLS - 1) / COLS;
  const int t0 = blockIdx.x * 4 * kXmGuTasks + wave, t1 = min((int)(blockIdx.x + 1) * 4 * kXmGuTasks, tasks);
  int n = 0;
  for (int q0 = 0; q0 < nk; q0 += 64) {
    const bool mine = q0 + lane < nk && idx[min(q0 + lane, nk - 1)] == e;
    const uint64_t bal = __ballot(mine);
    if (mine && wave == 0) list[n + __popcll(bal & ((1ull << lane) - 1ull))] = (uint16_t)(q0 + lane);
    n += __popcll(bal);
  }
  if (n == 0) return;
  const size_t rows = (size_t)2 * I;
  const uint16_t* bias = gu_bias + (size_t)e * rows;
  const uint8_t* codes = gu_codes + (size_t)e * rows * (H / 2);
  const uint8_t* scales = gu_scales + (size_t)e * rows * U;
  auto fill = [&](XmItem& w, int t) {
    t = min(t, tasks - 1);  // a wave without tasks reads along and stores nothing
    w.codes = codes + (size_t)t * (2 * COLS) * (H / 2);
    w.scales = scales + (size_t)t * (2 * COLS) * U;
    w.quads = (2 * I - 2 * COLS * t) / 4;
    w.x = nullptr;
  };
  XmItem it;
  fill(it, t0);
  XmStream<RQ, NG, true> st;
  st.start(it, U, lane);
  for (int q0 = 0; q0 < n; q0 += 4) {
    lds_barrier();  // list written; the previous quad's inputs read
    // the quad's inputs as fp32: thread = one 16-byte piece (8 elements) of a row
    for (int p = tid; p < 4 * 4 * U; p += 256) {
      const int r = p / (4 * U), u = (p >> 2) % U, pc = p & 3;
      const int q = list[min(q0 + r, n - 1)];
      const uint4 v = reinterpret_cast<const uint4*>(xn + (size_t)(q / k) * H)[4 * u + pc];
      float4* d = xs + (8 * (u >> 4) + 2 * pc) * 64 + 4 * (u & 15) + r;
      d[0] = make_float4(bf_lo(v.x), bf_hi(v.x), bf_lo(v.y), bf_hi(v.y));
      d[64] = make_float4(bf_lo(v.z), bf_hi(v.z), bf_lo(v.w), bf_hi(v.w));
    }
    lds_barrier();
    const int q = list[min(q0 + i, n - 1)];  // the lane's pair (column i)
    for (int t = t0; t < t1; t += 4) {
      const int j = COLS * t + ((lane & 4) ? 4 + (lane >> 5) : lane >> 4);  // the lane's column below
      const uint32_t bgu = load_pinned_u32(
          reinterpret_cast<const uint32_t*>(bias + 2 * min(j, I - 1)));
      XmItem nx;
      fill(nx, t + 4 < t1 ? t + 4 : t0);  // the wave's next task, or the next quad's first
      float a[4 * RQ];
      st.item(a, it, nx, U, lane, xs);
      it = nx;
      // rows 0 .. 7 end in the lanes whose bits 5..3 spell them, rows 8 .. 11 in
      // bits 5, 4; the lowest of those bits tells up from gate
      float a8[8], a4[4];
#pragma unroll
      for (int v = 0; v < 8; ++v) a8[v] = a[v];
#pragma unroll
      for (int v = 0; v < 4; ++v) a4[v] = a[8 + v];
      const float s8 = xm_fold<8>(a8, lane), s4 = xm_fold<4>(a4, lane);
      const float u8 = xor_lane<8>(s8), u4 = xor_lane<16>(s4);
      // lanes with bit 2 clear take columns 0 .. 3 (lane >> 4), the others columns
      // 4, 5 (lane >> 5): one SwiGLU for both
      const bool hi = (lane & 4) != 0;
      const float gb = __fadd_rn(hi ? s4 : s8, bf_lo(bgu));
      const float ub = __fadd_rn(hi ? u4 : u8, bf_hi(bgu));
      if ((lane & (hi ? 24 : 8)) == 0 && q0 + i < n && j < I)
        act[(size_t)q * I + xm_act_at(j, I / 32)] = f2bf(swiglu_clamp(gb, ub, alpha, limit));
    }
  }
}

// ===========================================================================
// down + weighted sum (+ residual): grid ceil(H / 12), 8 waves.  A block serves
// 12 output rows for every pair: the pairs are grouped by expert in LDS, and
// each wave takes every eighth item (an expert's next four pairs).  Row b's
// slots are then combined in slot order as in k_moe_down.  12 rows: 240 blocks
// at H = 2880, one round of the 256 CUs.
// ===========================================================================
constexpr int kXmDnRq = 3, kXmDnWaves = 8;
struct XmDownLds {
  int cnt[256], off[256], item0[256];
  int wsum[4][2];
  int n_items;
  uint16_t pair[kXmMaxPairs];   // grouped by expert
  uint32_t item[kXmMaxPairs];   // expert | first << 8 | count << 24
  float red[kXmMaxPairs][4 * kXmDnRq + 1];  // [pair][row]: dot + bias
};

template <int NG>
__global__ __launch_bounds__(64 * kXmDnWaves, 1) void k_xm_down(
    const uint8_t* __restrict__ dn_codes, const uint8_t* __restrict__ dn_scales,
    const uint16_t* __restrict__ dn_bias, const int32_t* __restrict__ idx,
    const float* __restrict__ score, int E, const uint16_t* __restrict__ act,
    const uint16_t* residual, uint16_t* out, int B, int H, int I, int k,
    int32_t* __restrict__ err) {
  constexpr int RQ = kXmDnRq, ROWS = 4 * RQ, NT = 64 * kXmDnWaves;
  constexpr int PT = (kXmMaxPairs + NT - 1) / NT;  // pairs per thread
  __shared__ XmDownLds s;
  const int U = I / 32, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 3, n0 = blockIdx.x * ROWS, nk = B * k;
  if (tid < 256) s.cnt[tid] = 0;
  __syncthreads();
  // rank of each pair within its expert (any order: a pair's value goes to its
  // own place); an id outside [0, E) matches no expert and contributes 0
  int rank[PT];
#pragma unroll
  for (int m = 0; m < PT; ++m) {
    const int q = tid + NT * m;
    rank[m] = -1;
    if (NT * m < nk && q < nk) {
      const int id = idx[q];
      if ((unsigned)id < (unsigned)E) {
        rank[m] = (atomicAdd(&s.cnt[id], 1) << 8) | id;
      } else {
        if (blockIdx.x == 0) flag_dev_err(err, kDevErrExpertId);
#pragma unroll
        for (int r = 0; r < ROWS; ++r) s.red[q][r] = 0.0f;
      }
    }
  }
  __syncthreads();
  // thread t < 256: expert t's first pair and first item
  const int c = tid < 256 ? s.cnt[tid] : 0, ni = (c + 3) >> 2;
  int pc = c, pi = ni;  // inclusive scans over the wave
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int a = __shfl_up(pc, o, 64), d = __shfl_up(pi, o, 64);
    if (lane >= o) { pc += a; pi += d; }
  }
  if (lane == 63 && wave < 4) { s.wsum[wave][0] = pc; s.wsum[wave][1] = pi; }
  __syncthreads();
  if (tid < 256) {
    int bc = 0, bi = 0;
    for (int v = 0; v < wave; ++v) { bc += s.wsum[v][0]; bi += s.wsum[v][1]; }
    const int o0 = bc + pc - c, i0 = bi + pi - ni;
    s.off[tid] = o0;
    for (int m = 0; m < ni; ++m)
      s.item[i0 + m] = (uint32_t)tid | ((uint32_t)(o0 + 4 * m) << 8) | ((uint32_t)min(4, c - 4 * m) << 24);
    if (tid == 255) s.n_items = bi + pi;
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < PT; ++m)
    if (rank[m] >= 0) s.pair[s.off[rank[m] & 255] + (rank[m] >> 8)] = (uint16_t)(tid + NT * m);
  __syncthreads();
  const int n_items = __builtin_amdgcn_readfirstlane(s.n_items);
  if (wave < n_items) {
    int q;
    uint32_t bl[RQ];
    auto fill = [&](XmItem& w, int at) {
      const uint32_t item = __builtin_amdgcn_readfirstlane(s.item[at]);
      const int first = (item >> 8) & 0xFFFF, cn = item >> 24;
      const size_t er = (size_t)(item & 255) * H;
      q = s.pair[first + min(i, cn - 1)];
      q |= i < cn ? 0 : 0x10000;  // a column past the item's pairs
      w.codes = dn_codes + (er + n0) * (I / 2);
      w.scales = dn_scales + (er + n0) * U;
      w.quads = (H - n0) / 4;  // H % 4 == 0
      w.x = act + (size_t)(q & 0xFFFF) * I;
      // the biases of the rows this lane holds after the folds
      bl[0] = load_pinned_u16(dn_bias + er + min(n0 + (lane >> 3), H - 1));
      bl[1] = load_pinned_u16(dn_bias + er + min(n0 + 8 + (lane >> 4), H - 1));
    };
    XmItem it;
    fill(it, wave);
    XmStream<RQ, NG, false> st;
    st.start(it, U, lane);
    for (int at = wave; at < n_items; at += kXmDnWaves) {
      const int q_cur = q;
      const float b0 = bf2f((uint16_t)bl[0]), b1 = bf2f((uint16_t)bl[1]);
      XmItem nx = it;
      if (at + kXmDnWaves < n_items) fill(nx, at + kXmDnWaves);
      float a[4 * RQ], a8[8], a4[4];
      st.item(a, it, nx, U, lane);
#pragma unroll
      for (int v = 0; v < 8; ++v) a8[v] = a[v];
#pragma unroll
      for (int v = 0; v < 4; ++v) a4[v] = a[8 + v];
      const float t8 = xm_fold<8>(a8, lane);  // row lane >> 3
      const float t4 = xm_fold<4>(a4, lane);  // row 8 + (lane >> 4)
      if (q_cur < 0x10000) {
        if ((lane & 4) == 0) s.red[q_cur][lane >> 3] = __fadd_rn(t8, b0);
        if ((lane & 12) == 0) s.red[q_cur][8 + (lane >> 4)] = __fadd_rn(t4, b1);
      }
      it = nx;
    }
  }
  __syncthreads();
  // row b, output row n0 + r: y = fmaf(score_s, red_s, y) over the slots in order
  for (int t = tid; t < B * ROWS; t += NT) {
    const int bb = t / ROWS, r = t % ROWS, n = n0 + r;
    if (n >= H) continue;
    float y = 0.0f;
    for (int sl = 0; sl < k; ++sl) y = __builtin_fmaf(score[bb * k + sl], s.red[bb * k + sl][r], y);
    const uint16_t m = f2bf(y);
    const size_t o = (size_t)bb * H + n;
    out[o] = residual ? f2bf(__fadd_rn(bf2f(residual[o]), bf2f(m))) : m;
  }
}

bool xm_moe_supported(const MoeArgs& a) {
  return xm_moe_wanted(a.B, a.k, a.E, a.H, a.I) && a.idx != nullptr && a.score != nullptr &&
         a.router_lg == nullptr && xm_groups(a.H) != 0 && xm_groups(a.I) != 0;
}

void launch_xm_moe(const MoeArgs& a, hipStream_t st) {
  const int gu_blocks = (a.I + kXmGuColumns - 1) / kXmGuColumns;
#define GU(NG)                                                                               \
  hipLaunchKernelGGL(k_xm_gate_up<NG>, dim3(gu_blocks, a.E), dim3(256), 0, st,        \
                     a.gu_codes, a.gu_scales, a.gu_bias, a.idx, a.xn, a.act, a.B * a.k, a.H, \
                     a.I, a.k, a.alpha, a.limit)
#define DN(NG)                                                                               \
  hipLaunchKernelGGL(k_xm_down<NG>, dim3((a.H + 4 * kXmDnRq - 1) / (4 * kXmDnRq)), dim3(64 * kXmDnWaves), 0, st, a.dn_codes,      \
                     a.dn_scales, a.dn_bias, a.idx, a.score, a.E, a.act, a.residual, a.out,  \
                     a.B, a.H, a.I, a.k, a.err)
  switch (xm_groups(a.H)) {
    case 1: GU(1); break;
    case 2: GU(2); break;
    case 4: GU(4); break;
    case 6: GU(6); break;
    default: GU(8); break;
  }
  switch (xm_groups(a.I)) {
    case 1: DN(1); break;
    case 2: DN(2); break;
    case 4: DN(4); break;
    case 6: DN(6); break;
    default: DN(8); break;
  }
#undef GU
#undef DN
}

}  // namespace neon
