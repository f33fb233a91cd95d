// Products with unquantised matrices: y[M,N] = x[M,K] @ w[N,K]^T (+ bias), element type bf16 or
// float, float32 accumulation.  Row strides are multiples of 64 elements and the columns between
// K and the stride are zero in BOTH operands, so no kernel has a K tail and any K is taken.
//
//  * dense_gemv_kernel, up to 16 rows of x: 16 weight rows per workgroup, K dealt out over its
//    waves, weights straight from memory into the A operand of a 16x16 matrix product (16 rows x
//    64 bytes per load instruction), x rows as the 16 columns of B.  One batch of kBatch loads per
//    wave is in flight before anything is waited for.  Range-checked loads stand in for every
//    tail: rows past N, x rows past M and steps past a wave's range read as zero.  PAIR: a gate and
//    an up matrix, the gated unit as epilogue.  DUAL: two products with nothing in common but the
//    number of rows share the launch.  Few columns under few rows: Q = 2 or 4 parts of K side by
//    side in the product - A's 16 rows are 16 / Q weight rows times Q parts, B's 16 columns 16 / Q
//    rows of x times Q parts; of the products of every part with every other the Q of equal parts
//    count - so that a workgroup has 16 / Q columns and the launch Q times the workgroups: a CU
//    takes no more than about 25 GB/s from memory, so 6.4 TB/s need all 256.
//  * dense_gemm_kernel, any number of rows: a (64 MI) x (64 NJ) tile per workgroup of four waves
//    (2 x 2, each (32 MI) x (32 NJ) in 32x32 products), K steps of 128 bytes per row through two
//    LDS buffers, the next two steps' vectors in registers meanwhile; one barrier per step.  A row's
//    eight 16-byte chunks sit at slot chunk ^ (row / 2 % 8): the 16 rows of an operand read meet no
//    bank of the 64 twice (chunk ^ (row % 8): half of the LDS cycles were conflicts; 2048x6912
//    under 1004 rows 62.0 -> 58.2 us, pair of 6912x2048 80.1 -> 78.2).  PAIR: the weight tile holds
//    rows of a gate and an up matrix, 32 and 32, so that a wave's column tiles are (gate, up) of the
//    same outputs and the gated unit is its epilogue.
//    GROUPED: the rows are one expert's (token, slot) pairs, from exo_moe_group's tile list.
//  * dense_gemm_wide_kernel: 256 x 256 tiles for bf16 launches of enough of them.
// Either may send its last output columns to a second, float32 buffer: inputs of 32-bit arithmetic
// (step sizes, gates, decays) are rows of the same weight matrix as the bf16 projections.
#include "../../include/exo_mi355x.h"
#include "dense.h"

#include <algorithm>
#include <type_traits>

namespace {

// ------------------------------------------------------------------------------ GEMV
constexpr int kBatch = 8;

struct GemvParams {
  const void* x;
  const void* w;   // gate matrix in pair mode
  const void* w2;  // up matrix
  const float* bias;
  void* y;
  float* y2;       // columns from n1 on
  int M, N, n1, ldx, ldw, ldy, ldy2;
  int y_f32 : 2, cols : 6, tiles : 24;  // weight rows of a workgroup, at most 16 / Q; workgroups: ceil(N / cols)
  GluConst glu;
  Epilogue ep;
};
// Two products and a norm's arguments go to one kernel, each line of 64 bytes another 0.2 to 0.3 us of a small launch's way to its first request: four bytes
// more were 5 % of two products of 520x960 in float32 under one row (3.44 | 3.65 us), a division by cols in the kernel one more.
static_assert(sizeof(GemvParams) == 128, "whole lines");

template <typename T>
__device__ __forceinline__ void store_out(void* y, size_t i, float v, int y_f32) {
  if (y_f32)
    reinterpret_cast<float*>(y)[i] = v;
  else
    reinterpret_cast<T*>(y)[i] = Elem<T>::make(v);
}

// Norm of the previous sublayer's output and residual sum, in front of the product that reads the
// residual: every workgroup forms y = x + mult * gain * v / rms(v), or (sum) y = gain * norm(keep * x + v),
// for itself and from it the product's operand (in LDS, element type): y, or y / rms(y) * pre.  v is the
// branch, or half the sum of two branches that are normed each with a gain of its own.  `norm` divides by
// the RMS, after the mean was taken off if `center`; without `gain` there is no norm: y = x + mult * v.  x null: only the branch is normed.  Workgroup 0 also writes y out - to another
// buffer than x is read from, since the others may still be reading.
struct PostNorm {
  const float* x;        // [M][H], or null
  const float* branch;   // [M][ldb]
  const float* branch2;  // [M][ldb], or null
  const float* gain_a;   // [H] gains of two branches
  const float* gain_b;
  const float* gain;     // [H], or null: the branch is added as it is
  const float* pre;      // [H], or null
  float* x_out;          // [M][H] (null with x)
  void* xb_out;          // T [M][ldx] the operand, or null
  int H, ldb, sum, center;
  float eps, mult, keep;
};
constexpr int kPostPasses = 4;  // at most so many float4 per lane of a row's waves

__host__ __device__ inline int post_waves_per_row(int M, int NW) {
  int p = 1;
  while (p < M) p *= 2;
  return NW > p ? NW / p : 1;
}

// what the wpr waves (a power of two) that share a row have left at `part`, added up
template <int NW>
__device__ __forceinline__ float row_total(const float* part, int wave, int wpr, int lane) {
  float v = part[(wave & ~(wpr - 1)) + (lane & (wpr - 1))];
  if (wpr >= 2) v += dpp_get<0xB1, 0xf>(v);
  if (wpr >= 4) v += dpp_get<0x4E, 0xf>(v);
  if (wpr >= 8) v += dpp_get<0x141, 0xf>(v);
  if (wpr >= 16) v += dpp_get<0x140, 0xf>(v);
  return v;
}
// a workgroup's LDS writes before it are visible behind it; requests to memory stay in flight
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
// sum over those waves.  part: two buffers in turn, so that one barrier is enough
template <int NW>
__device__ __forceinline__ float row_sum(float a, float (&part)[4][NW], int& phase, int wave, int wpr, int lane) {
  a = wave_total(a);
  phase ^= 1;
  if (lane == 0) part[phase][wave] = a;
  lds_barrier();
  return row_total<NW>(part[phase], wave, wpr, lane);
}

// PP: float4 of a row per lane in front of the product (0: nothing there); NORMED: branches that are normed (0: one
// that is added as it is).  RING: operands that are used up are requested again at once, for the step a batch ahead, so that requests
// are in flight throughout (gemv_ring: where that is the faster one)
template <typename T, int NW, int PP, int NORMED, bool PAIR, bool DUAL, int Q = 1, int STEPS = kBatch, bool RING = (Q != 1 && !PAIR)>
__global__ __launch_bounds__(64 * NW) void dense_gemv_kernel(const GemvParams p0, const GemvParams p1, const PostNorm q) {
  constexpr bool POST = PP > 0, TWO = NORMED == 2;
  constexpr int NP = POST ? PP : 1, NU = TWO ? NP : 1;
  constexpr int NM = PAIR ? 2 : 1;
  constexpr int R = 16 / Q;  // weight rows, and rows of x
  constexpr int BATCH = PAIR ? STEPS / 2 : STEPS;
  __shared__ float red[NM][NW][256];
  __shared__ float part[4][NW];  // (the last two: sums of two branches)
  extern __shared__ __attribute__((aligned(16))) char xs[];  // POST: [M][ldx * sizeof(T) + 16]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int tiles0 = p0.tiles;
  const bool second = DUAL && (int)blockIdx.x >= tiles0;
  const GemvParams& p = second ? p1 : p0;
  const int n0 = ((int)blockIdx.x - (second ? tiles0 : 0)) * p.cols, rows = min(p.cols, p.N - n0);
  const uint32_t wrow = (uint32_t)p.ldw * sizeof(T), xrow = (uint32_t)p.ldx * sizeof(T);
  const int steps = (int)(wrow >> 6) / Q;  // (rows are multiples of 128 or 256 bytes)
  const uint32_t part_at = Q > 1 ? r / R * steps * 64 : 0;
  const int per = (steps + NW - 1) / NW, s0 = min(steps, wave * per), s1 = min(steps, s0 + per);
  const __amdgpu_buffer_rsrc_t rw =
      buf_of(reinterpret_cast<const char*>(p.w) + (size_t)n0 * wrow, (uint32_t)rows * wrow);
  const __amdgpu_buffer_rsrc_t ru =
      buf_of(reinterpret_cast<const char*>(PAIR ? p.w2 : p.w) + (size_t)n0 * wrow, (uint32_t)rows * wrow);
  const __amdgpu_buffer_rsrc_t rx = buf_of(p.x, (uint32_t)p.M * xrow);
  const uint32_t woff = r % R * wrow + part_at + g * 16;
  uint4 wv[NM][BATCH];
  auto load_w = [&](int i, int s) {
    const uint32_t o = s < s1 ? woff + s * 64 : kPastEnd;
    wv[0][i] = buf_load16(rw, o, 0);
    if (PAIR) wv[NM - 1][i] = buf_load16(ru, o, 0);
  };
  auto batch_of_weights = [&](int s) {
#pragma unroll
    for (int i = 0; i < BATCH; ++i) load_w(i, s + i);
  };
  if (POST) {
    // A row's columns over wpr waves.  Everything that the sums need is requested ahead of the first weights, without a branch
    // that the compiler could not count across: a wait for a row's inputs or gains then leaves the weights in flight.  (Behind branches
    // every wait was for all requests: the norm began when the weights were there, and its gains were two more latencies.  2048 -> 6912
    // columns bf16 with the norms: 1 row 10.5 -> 9.4 us, 4 rows 18.0 -> 14.4; 1024 -> 4384 float, 2 rows 12.0 -> 10.5.)
    const int wpr = post_waves_per_row(p.M, NW), rpi = NW / wpr;  // rows per iteration
    const uint32_t lrow = xrow + 16;
    const bool vec = q.H % 4 == 0 && q.ldb % 4 == 0;
    const __amdgpu_buffer_rsrc_t rv = buf_of(q.branch, (uint32_t)p.M * q.ldb * 4), rr = buf_of(q.x ? q.x : q.branch, q.x ? (uint32_t)p.M * q.H * 4 : 0),
                                 r2 = buf_of(TWO ? q.branch2 : q.branch, (uint32_t)p.M * q.ldb * 4);
    const uint32_t gbytes = (uint32_t)q.H * 4;
    const __amdgpu_buffer_rsrc_t ra = buf_of(TWO ? q.gain_a : q.branch, TWO ? gbytes : 0), rb = buf_of(TWO ? q.gain_b : q.branch, TWO ? gbytes : 0),
                                 rg = buf_of(NORMED ? q.gain : q.branch, NORMED ? gbytes : 0), rp = buf_of(q.pre ? q.pre : q.branch, q.pre ? gbytes : 0);
    floatx4 v[NP], x[NP], u[NU], ga[NU], gb[NU], gn[NP], gp[NP];
    int phase = 0;
    const int cfirst = ((wave % wpr) * 64 + lane) * 4, cs = wpr * 256;
    // four columns from c on of a row that starts at element `at`: zero past H, past the buffer and where `on` is not set
    auto four = [&](const __amdgpu_buffer_rsrc_t& r, uint32_t at, int c, bool on, auto whole) __attribute__((always_inline)) {
      if constexpr (decltype(whole)::value) {
        return __builtin_bit_cast(floatx4, buf_load16(r, on && c < q.H ? (at + c) * 4 : kPastEnd, 0));
      } else {
        floatx4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t w = __builtin_amdgcn_raw_buffer_load_b32(r, on && c + e < q.H ? (at + c + e) * 4 : kPastEnd, 0, 0);
          o[e] = __builtin_bit_cast(float, w);
        }
        return o;
      }
    };
    constexpr bool AHEAD = PP * NU <= 2 && PP <= 2;  // (beyond, the gains do not fit beside the weights: requested where they are used)
    auto branch_gains = [&](auto whole) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < NU; ++i) ga[i] = four(ra, 0, cfirst + i * cs, true, whole), gb[i] = four(rb, 0, cfirst + i * cs, true, whole);
    };
    auto gains = [&](auto whole) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < NP; ++i) gn[i] = four(rg, 0, cfirst + i * cs, true, whole);
    };
    auto pre_gains = [&](auto whole) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < NP; ++i) gp[i] = four(rp, 0, cfirst + i * cs, true, whole);
    };
    auto all_gains = [&](auto whole) __attribute__((always_inline)) {
      if (TWO) branch_gains(whole);
      if (NORMED) gains(whole);
      pre_gains(whole);
    };
    auto here = [&](auto f) __attribute__((always_inline)) {  // not ahead
      if (AHEAD) return;
      if (vec)
        f(std::true_type());
      else
        f(std::false_type());
    };
    auto inputs = [&](int m0, auto whole) __attribute__((always_inline)) {
      const int m = m0 + wave / wpr;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int c = cfirst + i * cs;
        v[i] = four(rv, (uint32_t)m * q.ldb, c, m < p.M, whole);
        if (TWO) u[TWO ? i : 0] = four(r2, (uint32_t)m * q.ldb, c, m < p.M, whole);
        x[i] = four(rr, (uint32_t)m * q.H, c, m < p.M, whole);
      }
    };
    auto request = [&](int m0) __attribute__((always_inline)) {
      if (vec) {
        inputs(m0, std::true_type());
        if (AHEAD && m0 == 0) all_gains(std::true_type());
      } else {
        inputs(m0, std::false_type());
        if (AHEAD && m0 == 0) all_gains(std::false_type());
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto normed = [&](int m0) __attribute__((always_inline)) {
      const int m = m0 + wave / wpr;
      const bool on = m < p.M;
      const size_t o = (size_t)m * q.H;
      float ss = 0.f, su = 0.f;
      if (TWO) {  // half the sum of the two normed branches
#pragma unroll
        for (int i = 0; i < NP; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) ss += v[i][e] * v[i][e], su += u[TWO ? i : 0][e] * u[TWO ? i : 0][e];
        ss = wave_total(ss), su = wave_total(su);
        if (lane == 0) part[2][wave] = ss, part[3][wave] = su;
        lds_barrier();
        ss = row_total<NW>(part[2], wave, wpr, lane), su = row_total<NW>(part[3], wave, wpr, lane);
        const float ia = 0.5f / sqrtf(ss / q.H + q.eps), ib = 0.5f / sqrtf(su / q.H + q.eps);
        here(branch_gains);
#pragma unroll
        for (int i = 0; i < NP; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[i][e] = v[i][e] * ia * ga[TWO ? i : 0][e] + u[TWO ? i : 0][e] * ib * gb[TWO ? i : 0][e];
        ss = su = 0.f;
      }
      if (NORMED && q.sum) {  // the sum itself is normed
#pragma unroll
        for (int i = 0; i < NP; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[i][e] = fmaf(q.keep, x[i][e], v[i][e]);
            x[i][e] = 0.f;
            su += v[i][e];
          }
        if (q.center) {
          const float mean = row_sum<NW>(su, part, phase, wave, wpr, lane) / q.H;
#pragma unroll
          for (int i = 0; i < NP; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (cfirst + i * cs + e < q.H) v[i][e] -= mean;
        }
        ss = su = 0.f;
      }
      float inv = q.mult;
      if (NORMED) {
#pragma unroll
        for (int i = 0; i < NP; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) ss += v[i][e] * v[i][e];
        ss = row_sum<NW>(ss, part, phase, wave, wpr, lane);
        inv = (q.sum ? 1.f : q.mult) / sqrtf(ss / q.H + q.eps);
      }
      ss = 0.f;
      if (NORMED) here(gains);
#pragma unroll
      for (int i = 0; i < NP; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[i][e] += v[i][e] * inv * (NORMED ? gn[i][e] : 1.f);  // zero past H
          ss += x[i][e] * x[i][e];
        }
      float pinv = 1.f;
      if (q.pre) {
        ss = row_sum<NW>(ss, part, phase, wave, wpr, lane);
        pinv = 1.f / sqrtf(ss / q.H + q.eps);
        here(pre_gains);
      }
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int c = cfirst + i * cs;
        if (!on || c >= p.ldx) continue;
        floatx4 y = x[i];
        if (q.pre) {
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = y[e] * pinv * gp[i][e];
        }
        T out[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          out[e] = Elem<T>::make(y[e]);
          if (blockIdx.x == 0 && c + e < q.H) {
            if (q.x_out) q.x_out[o + c + e] = x[i][e];
            if (q.xb_out) reinterpret_cast<T*>(q.xb_out)[(size_t)m * p.ldx + c + e] = out[e];
          }
        }
        T* dst = reinterpret_cast<T*>(xs + m * lrow) + c;
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[e] = out[e];
      }
    };
    request(0);
    batch_of_weights(s0);
    __builtin_amdgcn_sched_barrier(0);
    normed(0);
    for (int m0 = rpi; m0 < p.M; m0 += rpi) {
      request(m0);
      normed(m0);
    }
    lds_barrier();
  } else {
    batch_of_weights(s0);
  }
  floatx4 acc[NM];
#pragma unroll
  for (int k = 0; k < NM; ++k) acc[k] = floatx4{0.f, 0.f, 0.f, 0.f};
  uint4 xv[BATCH];
  auto load_x = [&](int i, int s) {
    if (POST)  // (steps past the range: any finite values, their weights are zero)
      xv[i] = *reinterpret_cast<const uint4*>(xs + min(r % R, p.M - 1) * (xrow + 16) + part_at + g * 16 + min(s, s1 - 1) * 64);
    else
      xv[i] = buf_load16(rx, s < s1 ? r % R * xrow + part_at + g * 16 + s * 64 : kPastEnd, 0);
  };
  auto product = [&](int i) {
#pragma unroll
    for (int k = 0; k < NM; ++k) acc[k] = Elem<T>::mma16(wv[k][i], xv[i], acc[k]);
  };
  if (RING) {
    int s = s0;
    if (s < s1) {
#pragma unroll
      for (int i = 0; i < BATCH; ++i) load_x(i, s + i);
      for (; s + BATCH < s1; s += BATCH) {
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
          product(i);
          load_w(i, s + BATCH + i);
          load_x(i, s + BATCH + i);
        }
      }
#pragma unroll
      for (int i = 0; i < BATCH; ++i) product(i);
    }
  } else {
    for (int s = s0; s < s1; s += BATCH) {
#pragma unroll
      for (int i = 0; i < BATCH; ++i) load_x(i, s + i);
#pragma unroll
      for (int i = 0; i < BATCH; ++i) product(i);
      if (s + BATCH < s1) batch_of_weights(s + BATCH);
    }
  }
#pragma unroll
  for (int k = 0; k < NM; ++k)
#pragma unroll
    for (int e = 0; e < 4; ++e) red[k][wave][r * 16 + 4 * g + e] = acc[k][e];  // [m][n]
  __syncthreads();
  for (int o = threadIdx.x; o < R * p.M; o += 64 * NW) {
    const int m = o / R, n = o % R;
    if (n >= rows) continue;
    float v = 0.f, u = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        const int at = (k * R + m) * 16 + k * R + n;
        v += red[0][w][at];
        if (PAIR) u += red[NM - 1][w][at];
      }
    if (PAIR) {
      store_out<T>(p.y, (size_t)m * p.ldy + n0 + n, clamped_glu(v, u, p.glu), p.y_f32);
      continue;
    }
    if (p.bias) v += p.bias[n0 + n];
    if (n0 + n < p.n1)
      store_out<T>(p.y, (size_t)m * p.ldy + n0 + n, finish<T>(v, m, n0 + n, p.ep), p.y_f32);
    else
      p.y2[(size_t)m * p.ldy2 + n0 + n - p.n1] = v;
  }
}

// ------------------------------------------------------------------------------ GEMM
struct GemmParams {
  const void* x;
  const void* w;   // gate matrix in pair mode
  const void* w2;  // up matrix
  const float* bias;
  void* y;
  float* y2;       // columns from n1 on
  int M, N, n1, ldx, ldw, ldy, ldy2, y_f32;
  GluConst glu;
  Epilogue ep;
  // grouped
  const int32_t* sorted;
  const int32_t* tiles;
  int x_div;           // x row of a pair = pair / x_div
  size_t w_stride;     // elements between experts
  // split over K
  int ksplit, ksteps;  // 128-byte steps per split
  float* part;         // [ksplit][M][N]
};

// A wave's results, accumulators acc[i][j] of the 32 x 32 tiles at row wm + 32 i, weight row wn + 32 j of the workgroup's tile;
// wcol: the wave's place among those side by side.
template <typename T, int MI, int NJ, bool GROUPED, bool PAIR>
__device__ __forceinline__ void store_tile(const GemmParams& p, floatx16 (&acc)[MI][NJ], int n0, int m0, int m_end, int wm, int wn,
                                           int wcol, int lane, const int* row_pair) {
  const int frow = lane & 31, half = lane >> 5;
  // ---- epilogue: element e of tile (i, j): row wm + 32 i + 8 (e / 4) + 4 half + e % 4, column lane
  // One plain output (its last columns may go to the float32 buffer), or a partial one: every store at 32-bit
  // offsets from the tile's first row, rows past the end dropped by the buffer's range, columns of the other
  // buffer and past N by an offset beyond it.  (The whole offset is in the vector register: the scalar one takes
  // no part in the range check.)  Element by element, as in the loop at the end, 13664 columns of K = 2048 with
  // 96 in the second buffer under 1004 rows took 108 us, here 78; 6208 columns 52.5, here 38.
  if (!GROUPED && !PAIR && (p.ksplit > 1 || (!p.ep.mul && (p.n1 == p.N || p.ldy2 < 1 << 22)))) {
    const bool part = p.ksplit > 1, f32 = part || p.y_f32 || sizeof(T) == 4;
    const uint32_t ld = part ? (uint32_t)p.N : (uint32_t)p.ldy, size = f32 ? 4 : 2;
    const int n1 = part ? p.N : p.n1, held = m_end - m0;
    char* base = part ? reinterpret_cast<char*>(p.part + ((size_t)blockIdx.z * p.M + m0) * p.N)
                      : reinterpret_cast<char*>(p.y) + (size_t)m0 * ld * size;
    const __amdgpu_buffer_rsrc_t ry = buf_of(base, (uint32_t)held * ld * size);
    const uint32_t ld2 = n1 < p.N ? (uint32_t)p.ldy2 : 0;
    const __amdgpu_buffer_rsrc_t ry2 = buf_of(p.y2 + (size_t)m0 * ld2, (uint32_t)held * ld2 * 4);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int c0 = n0 + wn + 32 * j, n = c0 + frow;
      if (!part && p.bias) {
        const float b = n < p.N ? p.bias[n] : 0.f;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] += b;
      }
      auto store = [&](uint32_t voff, uint32_t row_bytes, auto put) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) put(acc[i][j][e], voff + (uint32_t)(32 * i + 8 * (e >> 2) + (e & 3)) * row_bytes);
      };
      auto put32 = [](const __amdgpu_buffer_rsrc_t& to, float v, uint32_t at) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), to, at, 0, 0);
      };
      if (c0 + 32 > n1 && n1 < p.N)  // (uniform)
        store(n >= n1 && n < p.N ? ((uint32_t)(wm + 4 * half) * ld2 + (n - n1)) * 4 : kPastEnd, ld2 * 4,
              [&](float v, uint32_t at) __attribute__((always_inline)) { put32(ry2, v, at); });
      if (c0 >= n1) continue;
      if (!part && p.ep.act) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] = activated(acc[i][j][e], p.ep.act, p.ep.cap);
      }
      const uint32_t voff = n < n1 ? ((uint32_t)(wm + 4 * half) * ld + n) * size : kPastEnd;
      if (f32)
        store(voff, ld * size, [&](float v, uint32_t at) __attribute__((always_inline)) { put32(ry, v, at); });
      else
        store(voff, ld * size, [&](float v, uint32_t at) __attribute__((always_inline)) {
          __builtin_amdgcn_raw_buffer_store_b16(f2bf(v), ry, at, 0, 0);
        });
    }
    return;
  }
  // A range of K of a gated pair: the gate's sums, then the up matrix's
  if (!GROUPED && PAIR && p.ksplit > 1) {
    const uint32_t row = (uint32_t)p.N * 4;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const __amdgpu_buffer_rsrc_t to = buf_of(p.part + ((size_t)(blockIdx.z * 2 + (j & 1)) * p.M + m0) * p.N, (uint32_t)(m_end - m0) * row);
      const int n = n0 + wcol * (16 * NJ) + (j >> 1) * 32 + frow;
      const uint32_t voff = n < p.N ? (uint32_t)(wm + 4 * half) * row + n * 4 : kPastEnd;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float v = acc[i][j][e];
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), to, voff + (uint32_t)(32 * i + 8 * (e >> 2) + (e & 3)) * row, 0, 0);
        }
    }
    return;
  }
  // Gated pairs and an expert's rows, in the element type: the same with a row's offset from the list of
  // pairs (four consecutive tile rows at a time).
  if (GROUPED || PAIR) {
    const uint32_t ld = (uint32_t)p.ldy * sizeof(T);
    char* base = reinterpret_cast<char*>(p.y) + (GROUPED ? 0 : (size_t)m0 * ld);
    const __amdgpu_buffer_rsrc_t ry = buf_of(base, GROUPED ? kPastEnd : (uint32_t)(m_end - m0) * ld);
    constexpr int JS = PAIR ? 2 : 1;  // accumulators per output
    uint32_t coff[NJ / JS];
#pragma unroll
    for (int j = 0; j < NJ / JS; ++j) {
      const int n = PAIR ? n0 + wcol * (16 * NJ) + j * 32 + frow : n0 + wn + 32 * j + frow;
      coff[j] = n < p.N ? (uint32_t)n * sizeof(T) : kPastEnd;
    }
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int t0 = wm + 32 * i + 8 * k + 4 * half;
        int rows[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) rows[e] = GROUPED ? row_pair[t0 + e] : t0 + e;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool in = GROUPED ? t0 + e < m_end : true;  // (not grouped: by the range)
#pragma unroll
          for (int j = 0; j < NJ / JS; ++j) {
            float v = acc[i][JS * j][4 * k + e];
            if (PAIR) v = gated<T>(v, acc[i][JS * j + JS - 1][4 * k + e], p.glu);
            const uint32_t off = in && coff[j] != kPastEnd ? (uint32_t)rows[e] * ld + coff[j] : kPastEnd;
            if (sizeof(T) == 4)
              __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), ry, off, 0, 0);
            else
              __builtin_amdgcn_raw_buffer_store_b16(f2bf(v), ry, off, 0, 0);
          }
        }
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int tr = wm + 32 * i + 8 * (e >> 2) + 4 * half + (e & 3);
      if (m0 + tr >= m_end) continue;
      const size_t row = (size_t)(m0 + tr);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int n = n0 + wn + 32 * j + frow;
        if (n >= p.N) continue;
        const float v = acc[i][j][e] + (p.bias ? p.bias[n] : 0.f);
        if (n < p.n1)
          store_out<T>(p.y, row * p.ldy + n, finish<T>(v, row, n, p.ep), p.y_f32);
        else
          p.y2[row * p.ldy2 + n - p.n1] = v;
      }
    }
}

template <typename T, int MI, int NJ, bool GROUPED, bool PAIR>
__global__ __launch_bounds__(256, 2) void dense_gemm_kernel(const GemmParams p) {
  constexpr int BM = 64 * MI, BW = 64 * NJ;      // tile rows of x, of weights
  constexpr int BN = PAIR ? BW / 2 : BW;         // output columns
  constexpr int XV = BM * 8 / 256, WV = BW * 8 / 256;
  constexpr int PD = 2;
  extern __shared__ __attribute__((aligned(16))) char lds[];  // [2][(BM + BW) * 128]
  __shared__ int row_pair[GROUPED ? BM : 1];
  constexpr int BUF = (BM + BW) * 128;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave >> 1) * (32 * MI), wn = (wave & 1) * (32 * NJ);
  // Consecutive workgroups go to different XCDs: give each XCD a contiguous run of tiles, row
  // tiles innermost, so that it streams few weight columns through its own L2.
  int bx, by;
  {
    const int total = (int)(gridDim.x * gridDim.y), id = (int)(blockIdx.y * gridDim.x + blockIdx.x);
    const int q = total >> 3, rem = total & 7, xcd = id & 7, k = id >> 3;
    const int t = xcd * q + min(xcd, rem) + k;
    by = t % (int)gridDim.y;
    bx = t / (int)gridDim.y;
  }
  const int n0 = bx * BN;
  int m0 = by * BM, m_end = p.M;
  size_t w_off = 0;
  if (GROUPED) {
    const int32_t* ti = p.tiles + 3 * (size_t)by;
    const int e = ti[0];
    if (e < 0) return;  // whole workgroup: an unused entry of the tile list
    m0 = 0;
    m_end = ti[2];
    for (int i = tid; i < BM; i += 256) row_pair[i] = p.sorted[ti[1] + min(i, m_end - 1)];
    w_off = (size_t)e * p.w_stride * sizeof(T);
    __syncthreads();
  }
  const uint32_t wrow = (uint32_t)p.ldw * sizeof(T), xrow = (uint32_t)p.ldx * sizeof(T);
  const int all_steps = (int)(wrow >> 7);
  const int k0 = p.ksplit > 1 ? (int)blockIdx.z * p.ksteps : 0;
  const int steps = (p.ksplit > 1 ? min(all_steps, k0 + p.ksteps) : all_steps) - k0;

  const char* xbase = reinterpret_cast<const char*>(p.x);
  if (!GROUPED) xbase += (size_t)m0 * xrow;
  const char* wbase = reinterpret_cast<const char*>(p.w) + w_off + (size_t)n0 * wrow;
  const uint32_t wbytes = (uint32_t)min(BN, p.N - n0) * wrow;  // rows past N read as zero
  const __amdgpu_buffer_rsrc_t rx = buf_of(xbase, 0xFFFFFFFFu);
  __amdgpu_buffer_rsrc_t rw[PAIR ? 2 : 1];
  rw[0] = buf_of(wbase, wbytes);
  if (PAIR)
    rw[PAIR ? 1 : 0] = buf_of(reinterpret_cast<const char*>(p.w2) + w_off + (size_t)n0 * wrow, wbytes);
  uint32_t xoff[XV], woff[WV];
#pragma unroll
  for (int i = 0; i < XV; ++i) {
    const int id = tid + 256 * i, tr = id >> 3, c = id & 7;
    const uint32_t row = GROUPED ? (uint32_t)(row_pair[tr] / p.x_div) : (uint32_t)min(tr, m_end - 1 - m0);
    xoff[i] = row * xrow + c * 16;
  }
#pragma unroll
  for (int i = 0; i < WV; ++i) {
    const int id = tid + 256 * i, tr = id >> 3, c = id & 7;
    // A pass of 256 threads covers one 32-row tile of the weight block: tile i belongs to wave
    // column half i / NJ.  PAIR: its column tiles alternate gate / up over the same 32 outputs.
    const int n = PAIR ? (i / NJ) * (16 * NJ) + ((i % NJ) >> 1) * 32 + (tr & 31) : tr;
    woff[i] = (uint32_t)n * wrow + c * 16;
  }
  // PD steps of tiles in flight in registers.  Requests past the last step re-read it: every load
  // is unconditional, so the waits count exactly the loads in front of the ones they are for.
  uint4 xr[PD][XV], wr[PD][WV];
  auto load_regs = [&](uint4 (&x)[XV], uint4 (&w)[WV], int s) {
    const uint32_t so = (uint32_t)(k0 + min(s, steps - 1)) * 128;
#pragma unroll
    for (int i = 0; i < XV; ++i) x[i] = buf_load16(rx, xoff[i], so);
#pragma unroll
    for (int i = 0; i < WV; ++i) w[i] = buf_load16(rw[PAIR ? (i % NJ) & 1 : 0], woff[i], so);
  };
  auto store_lds = [&](const uint4 (&x)[XV], const uint4 (&w)[WV], int b) {
    char* xl = lds + b * BUF;
    char* wl = xl + BM * 128;
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const int id = tid + 256 * i, tr = id >> 3, c = id & 7;
      *reinterpret_cast<uint4*>(xl + tr * 128 + ((c ^ ((tr >> 1) & 7)) << 4)) = x[i];
    }
#pragma unroll
    for (int i = 0; i < WV; ++i) {
      const int id = tid + 256 * i, tr = id >> 3, c = id & 7;
      *reinterpret_cast<uint4*>(wl + tr * 128 + ((c ^ ((tr >> 1) & 7)) << 4)) = w[i];
    }
  };
  const int frow = lane & 31, half = lane >> 5;
  floatx16 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

#pragma unroll
  for (int u = 0; u < PD; ++u) load_regs(xr[u], wr[u], u);
  store_lds(xr[0], wr[0], 0);
  load_regs(xr[0], wr[0], PD);
  for (int s0 = 0; s0 < steps; s0 += PD) {
#pragma unroll
    for (int u = 0; u < PD; ++u) {
      const int s = s0 + u;
      if (s >= steps) break;
      __syncthreads();  // step s is complete in its buffer, the other buffer is no longer read
      const int v = (u + 1) % PD;
      store_lds(xr[v], wr[v], (s + 1) & 1);
      load_regs(xr[v], wr[v], s + 1 + PD);
      __builtin_amdgcn_sched_barrier(0);  // (left alone, the requests sink behind the products)
      const char* xl = lds + (s & 1) * BUF + (wm + frow) * 128;
      const char* wl = lds + (s & 1) * BUF + (BM + wn + frow) * 128;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int slot = ((2 * t + half) ^ ((frow >> 1) & 7)) << 4;
        uint4 a[MI], b[NJ];
#pragma unroll
        for (int i = 0; i < MI; ++i) a[i] = *reinterpret_cast<const uint4*>(xl + i * 4096 + slot);
#pragma unroll
        for (int j = 0; j < NJ; ++j) b[j] = *reinterpret_cast<const uint4*>(wl + j * 4096 + slot);
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) acc[i][j] = Elem<T>::mma32(a[i], b[j], acc[i][j]);
      }
    }
  }

  store_tile<T, MI, NJ, GROUPED, PAIR>(p, acc, n0, m0, GROUPED ? m_end : min(m_end, m0 + BM), wm, wn, wave & 1, lane, row_pair);
}

// The same product in bf16 on 256 x 256 tiles, one workgroup of eight waves (2 x 4, each 128 x 64) per CU.  On the 128 x 128 tile
// a wave reads as many bytes of LDS per product as the CU delivers meanwhile (64 x 64: 16 KB per 16 products of 32
// cycles on each of four SIMDs), and the vectors pass through registers on their way there; here it is three quarters of that.  K steps of 64
// bytes per row through four LDS buffers, requested into them directly three steps ahead, each request in a slot of its
// own behind a product; one barrier per step, which drains nothing.  A step's first operands are read in the step before it, so
// that no wave stands behind the barrier.  A row's four 16-byte chunks sit at chunk ^ (row / 4 % 4): no bank twice in
// an operand read.
// Pair of 6912x2048 under 1004 rows 76 -> 59 us (970 TFLOP/s), 4100 rows 292 -> 229, 32768x2048 under 1004 rows 169 -> 129,
// 4096x13824 in four ranges 153 -> 117.  What bounds it: a round of 256 tiles takes 41 to 57 us of K = 2048 by how many CUs
// it fills, where the matrix cores are busy for 28; the first tiles' latency, the stores and the step after the barrier.
// (256 x 128 tiles, four waves of the same size: 1.2 to 1.3 times the time where both fill the chip, 2 to 8 % less than
// the 128 x 128 tile where few tiles do: not kept.)
constexpr int kWideStage = 2 * 256 * 64;
template <bool PAIR>
__global__ __launch_bounds__(512) void dense_gemm_wide_kernel(const GemmParams p) {
  typedef bf16_t T;
  constexpr int MI = 4, NJ = 2, BN = PAIR ? 128 : 256;
  constexpr int RQ = 4;  // a wave's requests of a step: 2 x 16 rows of x, 2 x 16 weight rows (PAIR: of one matrix)
  extern __shared__ __attribute__((aligned(1024))) char lds[];  // [4][x 256 rows | weights 256 rows][64]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wm = (wave >> 2) * 128, wcol = wave & 3, wn = wcol * 64;
  int bx, by;  // (tiles by XCD, as above)
  {
    const int total = (int)(gridDim.x * gridDim.y), id = (int)(blockIdx.y * gridDim.x + blockIdx.x);
    const int q = total >> 3, rem = total & 7, xcd = id & 7, k = id >> 3;
    const int t = xcd * q + min(xcd, rem) + k;
    by = t % (int)gridDim.y;
    bx = t / (int)gridDim.y;
  }
  const int n0 = bx * BN, m0 = by * 256;
  const uint32_t wrow = (uint32_t)p.ldw * sizeof(T), xrow = (uint32_t)p.ldx * sizeof(T);
  const int all = (int)(wrow >> 6), k0 = p.ksplit > 1 ? (int)blockIdx.z * p.ksteps * 2 : 0;
  const int steps = (p.ksplit > 1 ? min(all, k0 + p.ksteps * 2) : all) - k0;
  auto rsrc = [](const void* base) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32)),
                 0xFFFFFFFFu, 0x00020000u};
  };
  // (rows past the end repeat the last one, their results are not stored)
  const u32x4 rx = rsrc(reinterpret_cast<const char*>(p.x) + (size_t)m0 * xrow);
  const u32x4 rw = rsrc(reinterpret_cast<const char*>(PAIR && (wave & 1) ? p.w2 : p.w) + (size_t)n0 * wrow);
  uint32_t xoff[2], woff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int tr = (wave * 2 + i) * 16 + (lane >> 2), c = (lane & 3) ^ ((tr >> 2) & 3);
    const int n = PAIR ? (wave >> 1) * 32 + (tr & 31) : tr;
    xoff[i] = (uint32_t)min(tr, p.M - 1 - m0) * xrow + c * 16;
    woff[i] = (uint32_t)min(n, p.N - 1 - n0) * wrow + c * 16;
  }
  auto request = [&](int which, int s) {  // one of the wave's of step s (past the end: of the last)
    const uint32_t so = (uint32_t)(k0 + min(s, steps - 1)) * 64;
    const bool x = which < 2;
    const int i = which & 1;
    char* to = lds + (s & 3) * kWideStage + (x ? 0 : 256 * 64) + (wave * 2 + i) * 1024;
    load_to_lds16_untracked(x ? rx : rw, (lds_char)to, x ? xoff[i] : woff[i], so);
  };
  const int frow = lane & 31, half = lane >> 5, swz = (frow >> 2) & 3;
  const char* const xl = lds + (wm + frow) * 64;
  const char* const wl = lds + 256 * 64 + (wn + frow) * 64;
  floatx16 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  uint4 a[2][MI], b[2][NJ];
  auto read = [&](int which, int s, int t) {  // one of the six operands of half t of step s
    const int at = (s & 3) * kWideStage + (((2 * t + half) ^ swz) << 4);
    if (which < NJ)
      b[t][which] = *reinterpret_cast<const uint4*>(wl + at + which * 32 * 64);
    else
      a[t][which - NJ] = *reinterpret_cast<const uint4*>(xl + at + (which - NJ) * 32 * 64);
  };
#pragma unroll
  for (int s = 0; s < 3; ++s)
#pragma unroll
    for (int i = 0; i < RQ; ++i) request(i, s);
  auto landed = [](bool first) {
    if (first)
      __builtin_amdgcn_s_waitcnt(0x0F70 | (2 * RQ));  // vmcnt: step 0 is here
    else
      __builtin_amdgcn_s_waitcnt(0x0F70 | RQ);  // vmcnt: the next step's tiles are here too
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  landed(true);
#pragma unroll
  for (int i = 0; i < MI + NJ; ++i) read(i, 0, 0);
  for (int s = 0; s < steps; ++s) {
    // every wave has read step s - 1: its buffer takes step s + 3
    landed(false);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int k = 0; k < MI * NJ; ++k) {
        const int i = k / NJ, j = k % NJ;
        acc[i][j] = Elem<T>::mma32(a[t][i], b[t][j], acc[i][j]);
        // (the other half's operands, first the ones that its first products need)
        if (k < MI + NJ) read(k, t ? s + 1 : s, t ^ 1);
        if (k >= MI * NJ - RQ / 2) request(t * (RQ / 2) + k - (MI * NJ - RQ / 2), s + 3);
        __builtin_amdgcn_sched_barrier(0);
      }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the repeated requests have landed
  store_tile<T, MI, NJ, false, PAIR>(p, acc, n0, m0, min(p.M, m0 + 256), wm, wn, wcol, lane, nullptr);
}

// adds the K ranges in their order.  VEC (columns in fours, no activation or factor): four neighbouring columns per thread
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void dense_reduce_kernel(const GemmParams p) {
  constexpr int C = VEC ? 4 : 1;
  const int n = (blockIdx.x * 256 + threadIdx.x) * C, m = blockIdx.y;
  if (n >= p.N) return;
  float v[C];
#pragma unroll
  for (int e = 0; e < C; ++e) v[e] = p.bias ? p.bias[n + e] : 0.f;
  for (int z = 0; z < p.ksplit; ++z) {
    const float* at = p.part + ((size_t)z * p.M + m) * p.N + n;
    if constexpr (VEC) {
      const floatx4 u = *reinterpret_cast<const floatx4*>(at);
#pragma unroll
      for (int e = 0; e < C; ++e) v[e] += u[e];
    } else {
      v[0] += *at;
    }
  }
#pragma unroll
  for (int e = 0; e < C; ++e) {
    if (n + e < p.n1)
      store_out<T>(p.y, (size_t)m * p.ldy + n + e, VEC ? v[e] : finish<T>(v[e], m, n + e, p.ep), p.y_f32);
    else
      p.y2[(size_t)m * p.ldy2 + n + e - p.n1] = v[e];
  }
}
// ... of a gated pair, and its unit
template <typename T>
__global__ __launch_bounds__(256) void dense_reduce_pair_kernel(const GemmParams p) {
  const int n = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
  if (n >= p.N) return;
  const size_t one = (size_t)p.M * p.N;
  const float* at = p.part + (size_t)m * p.N + n;
  float g = 0.f, u = 0.f;
  for (int z = 0; z < p.ksplit; ++z) g += at[2 * z * one], u += at[(2 * z + 1) * one];
  store_out<T>(p.y, (size_t)m * p.ldy + n, gated<T>(g, u, p.glu), p.y_f32);
}
template <typename T>
void launch_reduce(const GemmParams& p, hipStream_t st) {
  // (from 2 MB of results on; below, one column per thread is as fast or, 130 rows of 2048, 15.9 us of a product against 18.0, faster)
  if (p.N % 4 == 0 && !p.ep.act && !p.ep.mul && (int64_t)p.M * p.N >= 1 << 19 && ((uintptr_t)p.part & 15) == 0)
    dense_reduce_kernel<T, true><<<dim3(exo_ceil_div(p.N, 1024), p.M), 256, 0, st>>>(p);
  else
    dense_reduce_kernel<T, false><<<dim3(exo_ceil_div(p.N, 256), p.M), 256, 0, st>>>(p);
}

int raise_lds(const void* fn, int bytes, bool* done) {
  if (*done || bytes <= 64 * 1024) return EXO_OK;
  const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) {
    exo_set_error("cannot raise the dynamic LDS limit to %d bytes: %s", bytes, hipGetErrorString(e));
    return EXO_ERR_HIP;
  }
  *done = true;
  return EXO_OK;
}

template <typename T, int MI, int NJ, bool GROUPED, bool PAIR>
int launch_gemm(const GemmParams& p, int row_tiles, hipStream_t st) {
  constexpr int lds = 2 * (64 * MI + 64 * NJ) * 128;
  static bool done = false;
  const auto fn = dense_gemm_kernel<T, MI, NJ, GROUPED, PAIR>;
  const int rc = raise_lds(reinterpret_cast<const void*>(fn), lds, &done);
  if (rc) return rc;
  const int bn = PAIR ? 32 * NJ : 64 * NJ;
  const dim3 grid(exo_ceil_div(p.N, bn), row_tiles, p.ksplit);
  exo_note_variant("dense_gemm<%s,%d,%d,%s,%s> grid=%dx%dx%d", sizeof(T) == 2 ? "bf16" : "f32", MI, NJ,
                   GROUPED ? "grouped" : "plain", PAIR ? "pair" : "single", (int)grid.x, (int)grid.y, (int)grid.z);
  fn<<<grid, 256, lds, st>>>(p);
  return EXO_OK;
}

template <bool PAIR>
int launch_wide(const GemmParams& p, hipStream_t st) {
  static bool done = false;
  const auto fn = dense_gemm_wide_kernel<PAIR>;
  const int rc = raise_lds(reinterpret_cast<const void*>(fn), 4 * kWideStage, &done);
  if (rc) return rc;
  const dim3 grid(exo_ceil_div(p.N, PAIR ? 128 : 256), exo_ceil_div(p.M, 256), p.ksplit);
  exo_note_variant("dense_gemm_wide<%s> grid=%dx%dx%d", PAIR ? "pair" : "single", (int)grid.x, (int)grid.y, (int)grid.z);
  fn<<<grid, 512, 4 * kWideStage, st>>>(p);
  return EXO_OK;
}

// 256 rows of each output lie below kPastEnd, where store_tile sends what it drops (the checks of the entry points allow
// for the 128 rows of the other tiles: strides of float32 from 2097152 on stay with those)
bool wide_fits(const GemmParams& p) {
  const int64_t row = (int64_t)p.ldy * (p.y_f32 ? 4 : 2), row2 = p.n1 < p.N ? (int64_t)p.ldy2 * 4 : 0;
  return 256 * std::max(row, row2) < kPastEnd;
}

// Whether 256 x 256 tiles are the faster: rounds of 256 of them, the last one by its share, against rounds of 512 of 128 x 128, in
// units of such a round (37 us of K = 2048).  More than one round only from K = 1024 on, or where the output is more than the last cache
// takes in: there is one workgroup per CU, whose stores nothing covers (widths of 6912 to 65536 under 130 to 2000 rows, of the time of 128 x
// 128: one round 0.72 to 0.97 at K = 2048, 0.83 to 1.05 at 64 to 192; several 0.74 to 0.98 at 2048, up to 1.05 at 1024, 1.19 at 768 and 1.44 at
// 192; of 151936 columns of K = 64 under 520 to 1004 rows 0.74 to 0.85).
bool wide_is_faster(int64_t wide, int64_t narrow, int steps, int64_t out_bytes) {
  const int64_t last = wide % 256;
  if (wide > 256 && steps < 16 && out_bytes < 1 << 27) return false;
  const double tw = 1.5 * (wide / 256) + (last ? 1.15 + 0.35 * last / 256 : 0.0);
  const double tn = narrow <= 512 ? 1.0 : narrow / 512.0 + 0.4;
  return tw < tn;
}

constexpr int64_t kPairWorkspace = 1 << 24;  // floats: as much as a device's single products share
// Ranges of K of a gated pair whose tiles leave CUs without work, or few in flight on each.  us: a step of 128 bytes of K takes 0.6 in bf16 and 1.3 in
// float, 1.7 times that with two workgroups on a CU, which is a full round; the reduce launch 2.75 and 0.35 a range more, the
// sums' way through memory 2.5 MB / us.
// It has to promise 12 % of tiles that leave CUs idle, 18 % of more: of 710 shapes (17 to 700 rows, 300 to 40000 columns, K of 256 to 8192) that it would split for 3 %
// 5 of 475 and 36 of 235 took more than 1.02 of the time of one range, up to 1.11 (f32 194x11240x960 119 | 132 us, bf16 39x36830x6912 203 | 218), and with this line none;
// of idle CUs 0.64 of the time on average (0.63 without the line), of more tiles 0.91 (0.88).
// Pair of 2560x1024 float under 53 rows, 40 workgroups, 40 -> 17 us; of 6912x2048 bf16 under 60 24.3 -> 18.8; of 999x7424 under 206 69 -> 25.
int pair_ranges(int64_t tiles, int steps, int64_t outputs, bool tall, int elem, int64_t ws_floats) {
  const double step = (elem == 2 ? 0.6 : 1.3) * (tall ? 1.6 : 1.0);
  auto rounds = [](int64_t wgs) { return wgs / 512 * 1.7 + (wgs % 512 > 256 ? 1.7 : wgs % 512 ? 1.0 : 0.0); };
  int best = 1;
  double least = (tiles <= 256 ? 0.88 : 0.82) * step * steps * rounds(tiles);
  for (int ks = 2; ks <= 16 && steps / ks >= 2 && 2 * ks * outputs <= ws_floats; ++ks) {
    const int range = exo_ceil_div(steps, ks), used = exo_ceil_div(steps, range);
    const double us = step * range * rounds(tiles * used) + 2.75 + used * (0.35 + 8e-6 / 2.5 * outputs);
    if (us < least) least = us, best = ks;
  }
  return best;
}

// Tiles of a product: 256 rows high (wide), or 128 where those still leave most CUs a workgroup (tall), else 64
struct PlainTiles {
  int64_t t1, t2, w;
  int steps;
  bool tall, wide;
};
template <typename T, bool PAIR>
PlainTiles tiles_of(const GemmParams& p) {
  PlainTiles t;
  const int64_t cols = exo_ceil_div(p.N, PAIR ? 64 : 128);
  t.steps = (int)((int64_t)p.ldw * sizeof(T) / 128);
  t.t2 = cols * exo_ceil_div(p.M, 128), t.t1 = cols * exo_ceil_div(p.M, 64);
  t.w = (int64_t)exo_ceil_div(p.N, PAIR ? 128 : 256) * exo_ceil_div(p.M, 256);
  t.tall = p.M > 64 && t.t2 >= 192;
  t.wide = sizeof(T) == 2 && p.M > 128 && wide_fits(p) && wide_is_faster(t.w, t.t2, t.steps, (int64_t)p.M * p.N * (p.y_f32 ? 4 : 2));
  return t;
}
template <typename T>
int pair_ranges_of(const GemmParams& p, int64_t ws_floats) {
  const PlainTiles t = tiles_of<T, true>(p);
  if (t.wide || p.M > 65535) return 1;  // (the launch that adds them has a row per block of y)
  return pair_ranges(t.tall ? t.t2 : t.t1, t.steps, (int64_t)p.M * p.N, t.tall, (int)sizeof(T), ws_floats);
}

template <typename T, bool PAIR>
int launch_plain(GemmParams p, int64_t ws_floats, hipStream_t st) {
  const PlainTiles plan = tiles_of<T, PAIR>(p);
  const int64_t t1 = plan.t1, t2 = plan.t2;
  const int steps = plan.steps;
  const bool tall = plan.tall;
  p.ksplit = 1;
  p.ksteps = steps;
  if constexpr (sizeof(T) == 2) {
    const int64_t wide = plan.w;
    if (plan.wide) return launch_wide<PAIR>(p, st);
    // ... or of ranges of K, while they are long against the partial sums' way through memory (columns x K, rows, us before | now:
    // 4096x13824, 300 88 | 66, 700 150 | 105, 2000 271 | 222; 4096x8192, 1004 93 | 85; 3072x6144, 700 65 | 54; 2048x6912, 1500 77 | 66; but
    // in ranges of 864, 1004 rows 54 | 58, and 4096x4096, 1004 rows 51 | 59)
    if (!PAIR && p.part && p.M > 256 && steps >= 96) {
      int ks = 1;
      while (wide * ks * 2 <= 256 && steps / (ks * 2) >= 16) ks *= 2;
      while (ks > 1 && (int64_t)ks * p.M * p.N > ws_floats) ks /= 2;
      if (ks > 1 && wide * ks > 128) {
        p.ksteps = exo_ceil_div(steps, ks);
        p.ksplit = exo_ceil_div(steps, p.ksteps);
        const int rc = launch_wide<PAIR>(p, st);
        if (rc == EXO_OK) launch_reduce<T>(p, st);
        return rc;
      }
    }
  }
  // Few tiles: split K until the chip has about one workgroup per CU, and on long ranges of K two, which wait for
  // different loads: 24 steps where some CUs have none yet, 48 where each has one (2048 columns, bf16, us: 300 rows
  // of K = 6912, 160 -> 320 workgroups 32.9 -> 28.2; 700 rows 176 -> 352 53.6 -> 46.8; 1004 rows 256 -> 512 56.9 -> 51.6, but of
  // K = 4096, ranges of 32 steps, 34.8 -> 35.6; tall tiles lose, 2000 rows 78.9 -> 83.1).
  if (!PAIR && p.part) {
    const int64_t tiles = tall ? t2 : t1;
    int ks = 1;
    auto more = [&](int64_t wgs, int range) {
      return wgs * 2 <= 256 ? range >= 4 : !tall && wgs * 2 <= 512 && range >= (wgs <= 192 ? 24 : 48);
    };
    while (ks < 16 && more(tiles * ks, steps / (ks * 2))) ks *= 2;
    while (ks > 1 && (int64_t)ks * p.M * p.N > ws_floats) ks /= 2;
    if (ks > 1) {
      p.ksteps = exo_ceil_div(steps, ks);
      p.ksplit = exo_ceil_div(steps, p.ksteps);
    }
  }
  if (PAIR && p.part) {
    const int ks = pair_ranges_of<T>(p, ws_floats);
    if (ks > 1) {
      p.ksteps = exo_ceil_div(steps, ks);
      p.ksplit = exo_ceil_div(steps, p.ksteps);
    }
  }
  int rc;
  if (tall)
    rc = launch_gemm<T, 2, 2, false, PAIR>(p, exo_ceil_div(p.M, 128), st);
  else
    rc = launch_gemm<T, 1, 2, false, PAIR>(p, exo_ceil_div(p.M, 64), st);
  if (rc) return rc;
  if (p.ksplit > 1 && PAIR)
    dense_reduce_pair_kernel<T><<<dim3(exo_ceil_div(p.N, 256), p.M), 256, 0, st>>>(p);
  else if (p.ksplit > 1)
    launch_reduce<T>(p, st);
  return EXO_OK;
}

int gemv_waves(int N) {
  const int tiles = exo_ceil_div(N, 16);
  return tiles >= 1024 ? 4 : tiles >= 256 ? 8 : 16;
}
// the columns of a row fit its waves' registers, the rows fit the LDS
bool post_fits(int M, int N, int H, int ldx, int elem) {
  return M <= 16 && ldx <= post_waves_per_row(M, gemv_waves(N)) * 256 * kPostPasses && H <= ldx &&
         (int64_t)M * (ldx * elem + 16) <= 40 * 1024;
}

// Where a wave has more steps than one batch, the next batch was requested only when the last was used up, one memory latency after another.
// Requested in a ring, rows of x as well as weights, us: 4096 columns bf16 K = 14336 under 1 | 4 | 8 rows 28.1 | 29.4 | 30.6 -> 24.6 | 25.4 | 27.4, K =
// 4096 9.1 | 9.7 | 10.2 -> 8.4 | 8.8 | 9.4; 2048 columns of K = 6912 in two parts 8.2 | 9.0 | 9.8 -> 7.7 | 8.5 | 9.4; f32 4096 of 4096 under 2 rows 18.6 ->
// 15.3, 20000 of 4096 72.7 -> 63.6.  The ring takes 72 registers instead of 51, 6 waves per SIMD instead of 8, which costs where x takes
// longer than the weights' latency: 16 rows 0.89 to 1.03 of the speed, 6 and 8 rows in the many workgroups of 4 waves 0.96 to 1.03 (20000 of 4096 bf16
// 8 rows 37.3 -> 39.1; 4 rows 0.98 to 1.09), pairs, whose rings hold two matrices, 0.89 to 1.02.
// A wave whose steps are one batch has nothing to request again and only fewer neighbours: f32 10822 columns of K = 256 under 6 rows 7.5 | 9.4,
// 11765 of 384 under 7 8.2 | 10.2, 14550 of 448 under 5 9.4 | 10.3, bf16 22185 of 768 under one 9.5 | 9.9 with it.
bool gemv_ring(const GemvParams& p, const GemvParams* p1, int waves, int elem) {
  const int steps = std::max(p.ldw, p1 ? p1->ldw : 0) * elem / 64;
  return p.M <= (waves == 4 ? 4 : 8) && steps > waves * kBatch;
}
// Behind norms, where the ring's registers come on top of the norms': from two whole batches on (f32, one row of 2048 into 20480 columns 37.6 -> 34.3
// us, of 4096 81.7 -> 78.0; bf16 level), and not where a wave has one or one and a half (four rows of 1024 into 9216 13.6 | 14.3, one of 2048 into 3072 9.3 | 9.7).
bool gemv_ring_post(const GemvParams& p, int waves, int elem) { return p.ldw * elem / 64 >= 2 * waves * kBatch; }
template <typename T, int NW, int PP, int Q, bool RING>
void launch_gemv_post_as(const GemvParams& p, const PostNorm& q, hipStream_t st) {
  constexpr int one = Q > 1 ? kBatch / 2 : kBatch;  // (post_parts: a wave's share of a part; a pair has half of STEPS of each)
  const int tiles = exo_ceil_div(p.N, p.cols), lds = p.M * (p.ldx * (int)sizeof(T) + 16);
  const auto fn = q.branch2 ? dense_gemv_kernel<T, NW, PP, 2, false, false, Q, one, RING> : q.gain ? dense_gemv_kernel<T, NW, PP, 1, false, false, Q, one, RING>
                                                                                                   : dense_gemv_kernel<T, NW, PP, 0, false, false, Q, one, RING>;
  fn<<<tiles, 64 * NW, lds, st>>>(p, p, q);
}
template <typename T, int NW, int PP, int Q = 1>
void launch_gemv_post(const GemvParams& p, const PostNorm& q, hipStream_t st) {
  if (p.w2) {
    const auto fn = q.branch2 ? dense_gemv_kernel<T, NW, PP, 2, true, false, Q> : q.gain ? dense_gemv_kernel<T, NW, PP, 1, true, false, Q> : dense_gemv_kernel<T, NW, PP, 0, true, false, Q>;
    fn<<<exo_ceil_div(p.N, p.cols), 64 * NW, p.M * (p.ldx * (int)sizeof(T) + 16), st>>>(p, p, q);
  } else if (Q > 1 || gemv_ring_post(p, NW, (int)sizeof(T))) {
    launch_gemv_post_as<T, NW, PP, Q, true>(p, q, st);
  } else if constexpr (Q == 1) {
    launch_gemv_post_as<T, NW, PP, Q, false>(p, q, st);
  }
}
template <typename T, int NW>
void launch_gemv_nw(const GemvParams& p, const GemvParams* p1, const PostNorm* q, hipStream_t st) {
  const int tiles = exo_ceil_div(p.N, p.cols);
  const PostNorm none{};
  if (q) {
    const int passes = exo_ceil_div(p.ldx, post_waves_per_row(p.M, NW) * 256);  // (post_fits: at most kPostPasses)
    if (passes <= 1)
      launch_gemv_post<T, NW, 1>(p, *q, st);
    else if (passes <= 2)
      launch_gemv_post<T, NW, 2>(p, *q, st);
    else
      launch_gemv_post<T, NW, kPostPasses>(p, *q, st);
  } else if (p.w2)
    dense_gemv_kernel<T, NW, 0, 0, true, false><<<tiles, 64 * NW, 0, st>>>(p, p, none);
  else {
    const bool ring = gemv_ring(p, p1, NW, (int)sizeof(T));
    const auto fn = p1 ? (ring ? dense_gemv_kernel<T, NW, 0, 0, false, true, 1, kBatch, true> : dense_gemv_kernel<T, NW, 0, 0, false, true>)
                       : (ring ? dense_gemv_kernel<T, NW, 0, 0, false, false, 1, kBatch, true> : dense_gemv_kernel<T, NW, 0, 0, false, false>);
    fn<<<tiles + (p1 ? exo_ceil_div(p1->N, p1->cols) : 0), 64 * NW, 0, st>>>(p, p1 ? *p1 : p, none);
  }
}
// Parts of K side by side where 16 columns per workgroup leave CUs without work, as many rows of x as the
// product then holds, and rows of whole parts.  One part -> these, us: N = 2048 (128 workgroups -> 256) under
// 4 rows, bf16: K = 4096 8.0 -> 6.9, K = 6912 11.8 -> 9.1 (8 rows: 12.8 -> 9.8; with the ring 8.5 and 9.4); N = 1024 (64 -> 256) under
// 2 rows, f32: K = 1024 6.5 -> 4.2, K = 2560 11.0 -> 5.7.  Four parts at N = 2048 give no more than two (6.8, 9.8).
// From 128 tiles of 16 columns on - more than 256 workgroups of two parts - the smaller pieces fill the CUs more evenly, but each
// reads x and adds its sums again.  `even`: how much less uneven they are (the work of the fullest CU over the average, of one part
// over that of two); of 24 widths of 2100 to 40000 columns, ten row lengths, 1 to 8 rows, bf16 and f32 (2656 points) two parts take
//   0.77 to 0.95 of the time of one where even is 1.33, 0.80 to 1.08 at 1.2 and 1.0 to 1.3 at 1.0, the more the more rows of x there are and
//   the longer they are (4 | 8 rows of 8 KB 1.0 to 1.2 | 1.0 to 1.24); hence the line, which leaves 0.5 % of the points more than 2 % behind one part
//   rows of 2 to 4 KB under few rows of x at any width below 16384 columns 0.77 to 1.04, short ones where one part leaves CUs idle 0.86 to 1.02
// 16 waves instead of 8: 7.4 and 8.7 in place of 6.9 and 9.1, f32 6.9 in place of 5.7.
int gemv_parts(const GemvParams& p, const GemvParams* p1, int elem) {
  const int tiles = exo_ceil_div(p.N, 16) + (p1 ? exo_ceil_div(p1->N, 16) : 0);
  const int rows = p.ldw * elem | (p1 ? p1->ldw * elem : 0);
  if (tiles <= 96 && p.M <= 4 && rows % 256 == 0) return 4;
  if (p.M > 8 || rows % 128) return 1;
  if (tiles <= 128) return 2;
  const int longest = std::max(p.ldw, p1 ? p1->ldw : 0) * elem;
  const int halves = exo_ceil_div(p.N, 8) + (p1 ? exo_ceil_div(p1->N, 8) : 0);
  auto fullest = [](int n) { return exo_ceil_div(n, 256) * 256.0 / n; };  // of 256 CUs, over the average
  const double one = fullest(tiles), even = one / fullest(halves);
  const bool pair = p.w2, short_rows = longest <= 2048, up_to_4k = longest <= 4096;
  bool two;
  if (tiles < (pair ? 160 : 192))  // (one round's worth of CUs; beyond it rows of less than 1 KB have no step for every wave of a part)
    two = pair ? short_rows : up_to_4k;
  else if (longest < 1024)
    two = false;
  else if (tiles >= 1024)
    two = !pair && !short_rows && up_to_4k && p.M <= 2;
  else if (tiles < 256)
    two = !pair && up_to_4k;
  else if (!up_to_4k && !pair && p.M > 4)  // (0.9 to 1.3)
    two = false;
  else if (short_rows)
    two = even >= 1.02 + 0.02 * p.M || (!pair && p.M <= 2 && one >= 1.15);
  else if (up_to_4k)
    two = longest <= 3072 ? even >= 1.02 + 0.02 * p.M || p.M <= 2 : even >= 1.1 || p.M <= 4;
  else
    two = even >= 1.05 + (pair ? 0.02 : 0.05) * p.M || (!pair && p.M == 1 && longest <= 8192 && one >= 1.15);
  return two ? 2 : 1;
}
// The same behind norms, which every workgroup repeats: more workgroups than one round cost more of them.  Rows up to 4 KB whose
// columns are at most two float4 per lane; the times of two parts over those of one, from a sweep of 672 shapes of 1 to 4 rows:
//   up to 128 tiles of 16 columns 0.60 to 0.85 (1536 columns of K = 512 bf16 5.8 -> 4.3 us, 2048 of K = 1024 float 8.3 -> 5.6)
//   below 256: one float4 per lane 0.77 to 0.96 (2 rows of 1024 float, 3072 columns 9.0 -> 8.1), two 0.93 to 1.07, pairs 0.90 to 1.18
//   beyond, rows of 4 KB behind one branch: 0.87 to 0.95 up to 352 tiles, pairs 0.77 to 1.01; 0.92 to 1.33 with more columns,
//     1.01 to 1.34 for shorter rows, 0.96 to 1.5 behind two branches
int post_parts(const GemvParams& p, const PostNorm& q, int elem) {
  const int tiles = exo_ceil_div(p.N, 16), row = p.ldw * elem, passes = exo_ceil_div(p.ldx, post_waves_per_row(p.M, 8) * 256);
  if (p.M > 8 || row > 4096 || row % 128 || passes > 2) return 1;
  if (tiles <= 128) return 2;
  if (tiles < 256) return !p.w2 && passes == 1 ? 2 : 1;
  return row > 3072 && !q.branch2 && tiles > 256 && tiles < (p.w2 ? 1024 : 352) ? 2 : 1;
}
template <typename T, bool PAIR, bool DUAL, int Q>
void launch_gemv_parts(const GemvParams& p, const GemvParams* p1, hipStream_t st) {
  const int tiles = exo_ceil_div(p.N, p.cols) + (DUAL ? exo_ceil_div(p1->N, p1->cols) : 0);
  const PostNorm none{};
  // (half the requests at once where a wave's share of a part is no more: requests past it cost time as well)
  const int ldw = DUAL && p1->ldw > p.ldw ? p1->ldw : p.ldw;
  if (exo_ceil_div((int)((int64_t)ldw * sizeof(T) / 64) / Q, 8) <= (PAIR ? kBatch / 4 : kBatch / 2))
    dense_gemv_kernel<T, 8, 0, 0, PAIR, DUAL, Q, kBatch / 2><<<tiles, 512, 0, st>>>(p, DUAL ? *p1 : p, none);
  else
    dense_gemv_kernel<T, 8, 0, 0, PAIR, DUAL, Q><<<tiles, 512, 0, st>>>(p, DUAL ? *p1 : p, none);
}
// Weight rows of a workgroup and its waves.  All workgroups of a launch of up to about two rounds are resident together, so the CU
// that got the most rows ends last: 864 workgroups of 8 rows leave 96 CUs with 32 (27 on average), 988 of 7 none with more than 28.  Fewer
// rows than the product holds cost nothing but its empty lanes.  Fewer waves cost less where every workgroup repeats norms and
// adds its waves' sums, more of them keep more requests in flight.  gemv_us is a fit to 4873 shapes (64 to 14336 columns of K, 300 to
// 40000 columns, 1 to 16 rows, with and without norms, bf16 and f32, 12 settings each).  What is fastest by it takes, on average, 0.946 of the time of
// whole 16 / parts rows and waves by the number of columns (gemv_waves), pairs 0.948, behind norms 0.946 and 0.935 (the best setting of each shape 0.93 to
// 0.94); slower by more than 2 % are 0.2 to 0.9 %: the 4 % that it has to promise leave most of them out.  us: f32 under 2 rows behind norms, 6432
// columns of 1024 11.0 -> 9.6, pair of 2560 10.5 -> 9.1; bf16 under 4 rows pair of 6912x2048 13.5 -> 12.6, under 8 15.6 -> 13.9, one row
// behind a norm 6160x2048 9.8 -> 8.3.
struct GemvShape {
  int waves, cols;
};
double gemv_us(const GemvParams& p, const GemvParams* p1, const PostNorm* q, int elem, int parts, GemvShape c) {
  const int mats = p.w2 ? 2 : 1, row = std::max(p.ldw, p1 ? p1->ldw : 0) * elem;
  const int wgs = exo_ceil_div(p.N, c.cols) + (p1 ? exo_ceil_div(p1->N, c.cols) : 0), held = std::max(1, exo_ceil_div(wgs - 2, 256));  // by the fullest CU (one or two more make no round)
  const double total = ((double)p.N * p.ldw + (p1 ? (double)p1->N * p1->ldw : 0.0)) * elem * mats;
  const double cu = (double)c.cols * row * mats / 25e3;  // a workgroup's bytes at 25 GB/s
  const double fullest = std::max(held * cu, total / 6.4e6), average = wgs * cu / 256;
  const double x = (double)held * p.M * row / 64e3, waves = c.waves * wgs / 8192.0;  // rows of x read, waves beside one another
  const int steps = exo_ceil_div(row / 64 / parts, c.waves);
  const bool half = parts > 1 && (q ? !p.w2 : steps <= kBatch / mats / 2);  // (the instances of launch_gemv_post_as and launch_gemv_parts)
  const int batch = kBatch / mats / (half ? 2 : 1);
  const double empty = (double)(exo_ceil_div(steps, batch) * batch - steps) * c.waves * held / 64;  // requests past a wave's range
  if (!q)
    return p.w2 ? 2.29 + 0.65 * fullest + 0.41 * average + 1.42 * x + 0.25 * waves + 1.17 * empty + 0.15 * steps
                : 2.46 + 0.74 * fullest + 0.45 * average + 1.34 * x + 0.83 * empty + (0.002 * p.M + 0.027) * steps;
  const int passes = exo_ceil_div(p.ldx, post_waves_per_row(p.M, c.waves) * 256);
  const double norms = (q->branch2 ? 3.2 * waves : 0.0);
  return norms + (p.w2 ? 0.94 + 0.69 * fullest + 0.34 * average + 4.77 * x + 1.73 * waves + 2.19 * empty + 0.51 * passes + 0.14 * steps + 0.17 * c.waves
                       : 0.96 + 0.74 * fullest + 0.20 * average + 3.1 * x + 2.52 * waves + 0.51 * empty + 0.66 * passes + 0.083 * steps + 0.21 * c.waves);
}
GemvShape gemv_shape(const GemvParams& p, const GemvParams* p1, const PostNorm* q, int elem, int parts) {
  const int N = p.N + (p1 ? p1->N : 0), most = 16 / parts;
  auto passes = [&](int waves) { return exo_ceil_div(p.ldx, post_waves_per_row(p.M, waves) * 256); };
  const GemvShape usual{parts > 1 ? 8 : gemv_waves(N), most};
  GemvShape best = usual;
  double least = 0.96 * gemv_us(p, p1, q, elem, parts, usual);
  for (int waves = 4; waves <= 16; waves *= 2) {
    if (parts > 1 && waves != 8) continue;
    // (More are another instance, which the cost is no fit to.  Behind two branches the second pass already takes its gains where they are used and not
    // ahead; one pass for those gives 1.10 of the time over the 212 shapes of the sweep that it would change, 0.86 to 1.33.)
    if (q && passes(waves) > std::max(2, passes(usual.waves))) continue;
    auto weigh = [&](int cols) {
      // (more waves than usual: 8 %, which leaves out f32 57806x1856 under two rows 87 | 98 us, two products of 10756x2048 20.5 | 22.1)
      const double us = gemv_us(p, p1, q, elem, parts, {waves, cols}) * (waves > usual.waves ? 0.96 / 0.92 : 1.0);
      if (us < least) least = us, best = GemvShape{waves, cols};
    };
    weigh(most);
    // one, two ... workgroups a CU (two products: one workgroup more), down to half of the rows that a product holds
    for (int held = exo_ceil_div(N, 256 * most), cols = most; 2 * cols > most; ++held) {
      cols = exo_ceil_div(N, 256 * held - (p1 ? 1 : 0));
      if (cols <= most && 2 * cols >= most) weigh(cols);
    }
  }
  return best;
}
template <typename T>
int launch_gemv(GemvParams p, const GemvParams* second, const PostNorm* q, hipStream_t st) {
  GemvParams other{};
  const GemvParams* p1 = nullptr;
  if (second) other = *second, p1 = &other;
  const int parts = q ? post_parts(p, *q, (int)sizeof(T)) : gemv_parts(p, p1, (int)sizeof(T));
  const GemvShape shape = gemv_shape(p, p1, q, (int)sizeof(T), parts);
  p.cols = other.cols = shape.cols, p.tiles = exo_ceil_div(p.N, p.cols);
  if (q && parts == 2) {
    exo_note_variant("dense_gemv<%s,8,post,%s> M=%d N=%d parts=2 cols=%d", sizeof(T) == 2 ? "bf16" : "f32", p.w2 ? "pair" : "single", p.M, p.N, p.cols);
    if (p.ldx <= post_waves_per_row(p.M, 8) * 256)
      launch_gemv_post<T, 8, 1, 2>(p, *q, st);
    else
      launch_gemv_post<T, 8, 2, 2>(p, *q, st);
    return EXO_OK;
  }
  if (parts > 1) {
    exo_note_variant("dense_gemv<%s,8,plain,%s> M=%d N=%d parts=%d cols=%d", sizeof(T) == 2 ? "bf16" : "f32",
                     p1 ? "dual" : p.w2 ? "pair" : "single", p.M, p.N, parts, p.cols);
    const auto launch = parts == 4 ? p1     ? launch_gemv_parts<T, false, true, 4>
                                     : p.w2 ? launch_gemv_parts<T, true, false, 4>
                                            : launch_gemv_parts<T, false, false, 4>
                        : p1       ? launch_gemv_parts<T, false, true, 2>
                        : p.w2     ? launch_gemv_parts<T, true, false, 2>
                                   : launch_gemv_parts<T, false, false, 2>;
    launch(p, p1, st);
    return EXO_OK;
  }
  const int nw = shape.waves;
  exo_note_variant("dense_gemv<%s,%d,%s,%s> M=%d N=%d cols=%d", sizeof(T) == 2 ? "bf16" : "f32", nw, q ? "post" : "plain",
                   p1 ? "dual" : p.w2 ? "pair" : "single", p.M, p.N, p.cols);
  if (nw == 4)
    launch_gemv_nw<T, 4>(p, p1, q, st);
  else if (nw == 8)
    launch_gemv_nw<T, 8>(p, p1, q, st);
  else
    launch_gemv_nw<T, 16>(p, p1, q, st);
  return EXO_OK;
}

#define EXO_DENSE_ARGS(what)                                                                            \
  EXO_REQUIRE(dtype == 0 || dtype == 1, what ": dtype must be 0 (bf16) or 1 (float32)");                \
  EXO_REQUIRE(x && w && y, what ": null pointer");                                                      \
  EXO_REQUIRE(M > 0 && N > 0 && ldx > 0 && ldx == ldw && ldw % 64 == 0,                                 \
              what ": need M, N > 0 and equal row strides that are multiples of 64 (got M=%d N=%d %d/%d)", \
              M, N, ldx, ldw);                                                                          \
  EXO_REQUIRE((((uintptr_t)x | (uintptr_t)w) & 15) == 0, what ": operands must be 16-byte aligned");    \
  EXO_REQUIRE((int64_t)ldw * 256 * 4 < (1ll << 31), what ": row stride %d too large", ldw)

}  // namespace

// ---- the struct interface: one product (or gated pair), rows of any number
static int linear_check(const exo_linear* a, const char* what) {
  EXO_REQUIRE(a && (a->dtype == 0 || a->dtype == 1), "%s: dtype must be 0 (bf16) or 1 (float32)", what);
  EXO_REQUIRE(a->w && a->y, "%s: null pointer", what);
  EXO_REQUIRE(a->M > 0 && a->N > 0 && a->ldx > 0 && a->ldx == a->ldw && a->ldw % 64 == 0,
              "%s: need M, N > 0 and equal row strides that are multiples of 64 (got M=%d N=%d %d/%d)", what, a->M, a->N,
              a->ldx, a->ldw);
  EXO_REQUIRE((((uintptr_t)a->x | (uintptr_t)a->w | (uintptr_t)a->w_up) & 15) == 0, "%s: operands must be 16-byte aligned", what);
  EXO_REQUIRE((int64_t)a->ldw * 256 * 4 < (1ll << 31) && (int64_t)a->ldy * 512 < (1ll << 31), "%s: row strides %d / %d too large", what, a->ldw, a->ldy);
  EXO_REQUIRE(a->n1 > 0 && a->n1 <= a->N && a->ldy >= a->n1 && (a->n1 == a->N || (a->y2 && a->ldy2 >= a->N - a->n1)),
              "%s: outputs do not hold %d columns (%d in the first: %d, %d)", what, a->N, a->n1, a->ldy, a->ldy2);
  EXO_REQUIRE(!a->w_up || (a->n1 == a->N && !a->bias), "%s: a gated pair has one output and no bias", what);
  EXO_REQUIRE(a->act >= 0 && a->act <= 3 && (a->act != 3 || a->cap > 0.f) && (!a->mul || a->ldmul >= a->N) && (!(a->act || a->mul) || (!a->w_up && a->n1 == a->N)),
              "%s: an activation (%d) or factor belongs to one plain output", what, a->act);
  return EXO_OK;
}
static GemvParams gemv_of(const exo_linear* a) {
  GemvParams p{};
  p.x = a->x, p.w = a->w, p.w2 = a->w_up, p.bias = a->bias, p.y = a->y, p.y2 = a->y2;
  p.M = a->M, p.N = a->N, p.n1 = a->n1, p.ldx = a->ldx, p.ldw = a->ldw, p.ldy = a->ldy, p.ldy2 = a->ldy2, p.y_f32 = a->y_f32 != 0;
  p.glu = GluConst{a->limit, a->alpha, a->shift, a->cubic};
  p.ep = Epilogue{a->act, a->mul, a->mul_rows, a->ldmul, a->cap};
  return p;
}

extern "C" int exo_linear_rows(const exo_linear* a, const exo_linear* b, exo_stream_t stream) {
  int rc = linear_check(a, "exo_linear_rows");
  if (rc) return rc;
  EXO_REQUIRE(a->M <= 16 && a->x, "exo_linear_rows: M=%d must be <= 16, x not null", a->M);
  GemvParams second{};
  if (b) {
    rc = linear_check(b, "exo_linear_rows");
    if (rc) return rc;
    EXO_REQUIRE(b->x && b->M == a->M && b->dtype == a->dtype && !a->w_up && !b->w_up,
                "exo_linear_rows: two products of one launch need the same rows and no gated pair");
    second = gemv_of(b);
  }
  const GemvParams p = gemv_of(a);
  rc = EXO_BY_TYPE(a->dtype, launch_gemv<bf16_t>(p, b ? &second : nullptr, nullptr, (hipStream_t)stream),
                   launch_gemv<float>(p, b ? &second : nullptr, nullptr, (hipStream_t)stream));
  if (rc) return rc;
  EXO_CHECK_LAUNCH("exo_linear_rows");
  return EXO_OK;
}

extern "C" int exo_post_linear_fits(int M, int N, int H, int ldx, int dtype) {
  return M > 0 && N > 0 && H > 0 && post_fits(M, N, H, ldx, dtype == 0 ? 2 : 4);
}

// row m of the launch alone (of its arguments; the branches' row stride then has no use)
static exo_linear row_of(exo_linear a, int m) {
  const size_t elem = a.dtype ? 4 : 2;
  auto at = [](auto* p, size_t bytes) { return p ? reinterpret_cast<decltype(p)>((uintptr_t)p + bytes) : p; };
  a.y = at(a.y, (size_t)m * a.ldy * (a.y_f32 ? 4 : elem)), a.y2 = at(a.y2, (size_t)m * a.ldy2 * 4);
  a.mul = at(a.mul, a.mul_rows ? 0 : (size_t)m * a.ldmul * elem), a.mul_rows = at(a.mul_rows, (size_t)m * 4);
  a.M = 1;
  return a;
}
static exo_post_norm row_of(exo_post_norm q, const exo_linear& a, int m) {
  auto at = [](auto* p, size_t bytes) { return p ? reinterpret_cast<decltype(p)>((uintptr_t)p + bytes) : p; };
  q.x = at(q.x, (size_t)m * q.H * 4), q.x_out = at(q.x_out, (size_t)m * q.H * 4);
  q.branch = at(q.branch, (size_t)m * q.ldb * 4), q.branch2 = at(q.branch2, (size_t)m * q.ldb * 4);
  q.operand = at(q.operand, (size_t)m * a.ldx * (a.dtype ? 4 : 2));
  q.ldb = q.H;
  return q;
}

extern "C" int exo_post_linear(const exo_post_norm* q, const exo_linear* a, exo_stream_t stream) {
  int rc = linear_check(a, "exo_post_linear");
  if (rc) return rc;
  EXO_REQUIRE(q && q->branch && (q->x ? q->x_out && q->x_out != q->x : q->gain && !q->x_out && !q->sum),
              "exo_post_linear: null pointer or x_out == x");
  EXO_REQUIRE(q->gain || !(q->sum || q->branch2), "exo_post_linear: a branch without a norm is one, added as it is");
  EXO_REQUIRE(q->ldb >= q->H && !(q->sum && q->branch2) && (q->sum || !q->center),
              "exo_post_linear: branch stride %d of %d columns, or a norm of the sum of two branches", q->ldb, q->H);
  EXO_REQUIRE(!q->branch2 || (q->gain_a && q->gain_b), "exo_post_linear: two branches need a gain each");
  EXO_REQUIRE(post_fits(a->M, a->N, q->H, a->ldx, a->dtype == 0 ? 2 : 4), "exo_post_linear: %d rows of %d columns do not fit one launch",
              a->M, q->H);
  // (the kernel's offsets into all rows of a branch have 32 bits and stay below kPastEnd; rows further apart one by one)
  if ((int64_t)a->M * q->ldb * 4 >= kPastEnd && q->ldb > q->H) {
    for (int m = 0; m < a->M; ++m) {
      const exo_linear one = row_of(*a, m);
      const exo_post_norm norms = row_of(*q, *a, m);
      if ((rc = exo_post_linear(&norms, &one, stream))) return rc;
    }
    return EXO_OK;
  }
  const GemvParams p = gemv_of(a);
  const PostNorm n{q->x, q->branch, q->branch2, q->gain_a, q->gain_b, q->gain, q->pre, q->x_out, q->operand, q->H, q->ldb,
                   q->sum, q->center, q->eps, q->mult, q->keep};
  rc = EXO_BY_TYPE(a->dtype, launch_gemv<bf16_t>(p, nullptr, &n, (hipStream_t)stream),
                   launch_gemv<float>(p, nullptr, &n, (hipStream_t)stream));
  if (rc) return rc;
  EXO_CHECK_LAUNCH("exo_post_linear");
  return EXO_OK;
}

static GemmParams gemm_of(const exo_linear* a) {
  GemmParams p{};
  p.x = a->x, p.w = a->w, p.w2 = a->w_up, p.bias = a->bias, p.y = a->y, p.y2 = a->y2;
  p.M = a->M, p.N = a->N, p.n1 = a->n1, p.ldx = a->ldx, p.ldw = a->ldw, p.ldy = a->ldy, p.ldy2 = a->ldy2, p.y_f32 = a->y_f32;
  p.glu = GluConst{a->limit, a->alpha, a->shift, a->cubic};
  p.ep = Epilogue{a->act, a->mul, a->mul_rows, a->ldmul, a->cap};
  return p;
}

extern "C" int64_t exo_linear_pair_workspace(const exo_linear* a) {
  if (linear_check(a, "exo_linear_pair_workspace") || !a->w_up) return 0;
  const GemmParams p = gemm_of(a);
  const int ks = EXO_BY_TYPE(a->dtype, pair_ranges_of<bf16_t>(p, kPairWorkspace), pair_ranges_of<float>(p, kPairWorkspace));
  return ks > 1 ? 2 * (int64_t)ks * p.M * p.N : 0;
}

extern "C" int exo_linear_gemm(const exo_linear* a, float* workspace, int64_t workspace_floats, exo_stream_t stream) {
  int rc = linear_check(a, "exo_linear_gemm");
  if (rc) return rc;
  EXO_REQUIRE(a->x && a->M <= 65535 * 64, "exo_linear_gemm: null x or bad M=%d", a->M);
  GemmParams p = gemm_of(a);
  p.part = workspace;
  EXO_REQUIRE(!a->w_up || a->y_f32 == (a->dtype == 1), "exo_linear_gemm: a gated pair leaves in the element type");
  if (a->w_up)
    rc = EXO_BY_TYPE(a->dtype, (launch_plain<bf16_t, true>(p, workspace_floats, (hipStream_t)stream)),
                     (launch_plain<float, true>(p, workspace_floats, (hipStream_t)stream)));
  else
    rc = EXO_BY_TYPE(a->dtype, (launch_plain<bf16_t, false>(p, workspace_floats, (hipStream_t)stream)),
                     (launch_plain<float, false>(p, workspace_floats, (hipStream_t)stream)));
  if (rc) return rc;
  EXO_CHECK_LAUNCH("exo_linear_gemm");
  return EXO_OK;
}

// Experts of a prompt: x rows by (token, slot) pair through exo_moe_group's workspace.  w_up null:
// the plain product, else the gated pair.  y row = pair index.
extern "C" int exo_dense_grouped_gemm(const void* x, const void* w, const void* w_up, const void* group_ws, void* y,
                                      float limit, float alpha, float shift, int T, int topk, int x_per_pair, int E,
                                      int N, int ldx, int ldw, int ldy, int dtype, exo_stream_t stream) {
  const int M = T;
  EXO_DENSE_ARGS("exo_dense_grouped_gemm");
  EXO_REQUIRE(group_ws && topk > 0 && E > 0 && ldy >= N && (int64_t)T * topk < (1ll << 30),
              "exo_dense_grouped_gemm: bad arguments (T=%d topk=%d E=%d)", T, topk, E);
  EXO_REQUIRE((int64_t)T * (x_per_pair ? topk : 1) * ldx * (dtype ? 4 : 2) < (1ll << 32),
              "exo_dense_grouped_gemm: activations exceed 32-bit byte offsets");
  EXO_REQUIRE((int64_t)T * topk * ldy * (dtype ? 4 : 2) < kPastEnd, "exo_dense_grouped_gemm: outputs exceed 31-bit byte offsets");
  const int64_t pairs = (int64_t)T * topk;
  const int tiles = (int)((pairs + 127) / 128) + E;  // exo_moe_group's list length
  EXO_REQUIRE(tiles <= 65535, "exo_dense_grouped_gemm: %d row tiles exceed the grid limit", tiles);
  GemmParams p{};
  p.x = x, p.w = w, p.w2 = w_up, p.y = y, p.M = T, p.N = N, p.ldx = ldx, p.ldw = ldw, p.ldy = ldy;
  p.glu = GluConst{limit, alpha, shift, 0.f};
  p.sorted = reinterpret_cast<const int32_t*>(group_ws);
  p.tiles = p.sorted + pairs;
  p.x_div = x_per_pair ? 1 : topk;
  p.w_stride = (size_t)N * ldw;
  p.ksplit = 1;
  const hipStream_t st = (hipStream_t)stream;
  int rc;
  if (w_up)
    rc = EXO_BY_TYPE(dtype, (launch_gemm<bf16_t, 2, 2, true, true>(p, tiles, st)),
                     (launch_gemm<float, 2, 2, true, true>(p, tiles, st)));
  else
    rc = EXO_BY_TYPE(dtype, (launch_gemm<bf16_t, 2, 2, true, false>(p, tiles, st)),
                     (launch_gemm<float, 2, 2, true, false>(p, tiles, st)));
  if (rc) return rc;
  EXO_CHECK_LAUNCH("exo_dense_grouped_gemm");
  return EXO_OK;
}
