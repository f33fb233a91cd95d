// Bandwidth-bound small ops: residual+RMSNorm, RoPE + KV append (+ per-head norm),
// SwiGLU, MoE routing/combination, greedy sampling reductions.
#include "../../include/exo_mi355x.h"
#include "common.h"
#include "dense.h"
#include "route.h"
#include <cstring>

namespace {

// ---------------------------------------------------------------- the host's numbers
// In the launch's own arguments (a launch takes 4 KB of them): a copy from pageable memory returns when everything in
// front of it on the stream is done, and the next launches then start on an idle GPU.
struct PutInts {
  int32_t v[EXO_PUT_INTS];
};
__global__ __launch_bounds__(64) void put_i32_kernel(int32_t* __restrict__ dst, const PutInts src, int n) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  if (i < n) dst[i] = src.v[i];
}

// ---------------------------------------------------------------- add + RMSNorm
// One workgroup per row; each thread keeps up to 4 x 8 elements in registers.
constexpr int kNormThreads = 256;
constexpr int kNormMaxChunks = 4;  // H <= 256*8*4 = 8192

__device__ __forceinline__ float block_sum_256(float v, float* sh) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) sh[wave] = v;
  __syncthreads();
  float r = sh[0] + sh[1] + sh[2] + sh[3];
  __syncthreads();
  return r;
}

// TOGETHER: row, residual and weights are requested together, without a branch (past the row: nothing, as zeros); behind branches they are
// up to nine memory latencies in a chain.  Otherwise piece by piece, weights behind the sum (norm_together: where that is the faster one).
template <int CHUNKS, bool TOGETHER>
__global__ __launch_bounds__(kNormThreads) void add_rmsnorm_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ res,
    const bf16_t* __restrict__ w, bf16_t* __restrict__ h_out, bf16_t* __restrict__ n_out,
    int H, float eps) {
  __shared__ float sh[4];
  const size_t row = (size_t)blockIdx.x * H;
  uint4 a[CHUNKS], r[CHUNKS], wv[CHUNKS];
  if (TOGETHER) {
    const uint32_t bytes = (uint32_t)H * 2;
    const __amdgpu_buffer_rsrc_t rx = buf_of(x + row, bytes), rr = buf_of(res ? res + row : x, res ? bytes : 0), rw = buf_of(w, bytes);
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      const uint32_t at = (threadIdx.x + i * kNormThreads) * 16;
      a[i] = buf_load16(rx, at, 0);
      r[i] = buf_load16(rr, at, 0);
    }
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) wv[i] = buf_load16(rw, (threadIdx.x + i * kNormThreads) * 16, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
  float v[CHUNKS][8];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < CHUNKS; ++i) {
    const int e0 = (threadIdx.x + i * kNormThreads) * 8;
    if (TOGETHER || e0 < H) {
      if (!TOGETHER) {
        a[i] = *reinterpret_cast<const uint4*>(x + row + e0);
        if (res) r[i] = *reinterpret_cast<const uint4*>(res + row + e0);
      }
      const uint32_t a4[4] = {a[i].x, a[i].y, a[i].z, a[i].w}, r4[4] = {r[i].x, r[i].y, r[i].z, r[i].w};
      uint32_t o4[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o4[e] = res ? pack_bf2(bf_lo(a4[e]) + bf_lo(r4[e]), bf_hi(a4[e]) + bf_hi(r4[e])) : a4[e];
        v[i][2 * e] = bf_lo(o4[e]);
        v[i][2 * e + 1] = bf_hi(o4[e]);
      }
      if (h_out && e0 < H) *reinterpret_cast<uint4*>(h_out + row + e0) = make_uint4(o4[0], o4[1], o4[2], o4[3]);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(v[i][e], v[i][e], ss);
    }
  }
  ss = block_sum_256(ss, sh);
  const float inv = rsqrtf(ss / (float)H + eps);
#pragma unroll
  for (int i = 0; i < CHUNKS; ++i) {
    const int e0 = (threadIdx.x + i * kNormThreads) * 8;
    if (e0 < H) {
      if (!TOGETHER) wv[i] = *reinterpret_cast<const uint4*>(w + e0);
      const uint32_t w4[4] = {wv[i].x, wv[i].y, wv[i].z, wv[i].w};
      uint32_t o4[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o4[e] = pack_bf2(v[i][2 * e] * inv * bf_lo(w4[e]), v[i][2 * e + 1] * inv * bf_hi(w4[e]));
      *reinterpret_cast<uint4*>(n_out + row + e0) = make_uint4(o4[0], o4[1], o4[2], o4[3]);
    }
  }
}
// Few rows of two pieces and more wait for their latencies; between 800 and 2000 they keep the memory busier when the requests
// come one after another; beyond, those without a residual or of two or three pieces are together again the faster.  One piece is one chain either way; with a residual and more
// than the L2s hold, together (3000 of 2048 8.9 and 9.3).
// Without | with a residual, us, together and piece by piece: 61 rows of 4096 3.1 | 3.3 and 3.1 | 3.6, of 8192 3.5 | 3.9 and 3.9 | 4.9; 1023 of 3072
// 4.3 | 5.7 and 4.0 | 5.3, of 4096 4.6 | 6.4 and 4.5 | 6.1, of 8192 6.7 | 11.3 and 6.7 | 12.2; 3000 of 4096 8.7 | 15.8 and 9.6 | 16.4; 4096 of 1024 5.1 | 7.2 and
// 4.7 | 6.7.
bool norm_together(int rows, int H, bool residual) {
  const int chunks = exo_ceil_div(H, kNormThreads * 8);
  if (chunks == 1) return residual && (int64_t)rows * H >= 5000000;
  if (rows < 800) return true;
  if (chunks == 2) return rows >= 2100;
  return residual ? chunks == 3 || rows < 1800 : rows >= 1600;
}
template <bool TOGETHER>
void launch_add_rmsnorm(const bf16_t* x, const bf16_t* res, const bf16_t* w, bf16_t* h_out, bf16_t* n_out, int rows, int H, float eps, hipStream_t st) {
  const int chunks = exo_ceil_div(H, kNormThreads * 8);
  const auto fn = chunks <= 1 ? add_rmsnorm_kernel<1, TOGETHER> : chunks <= 2 ? add_rmsnorm_kernel<2, TOGETHER> :
                  chunks <= 3 ? add_rmsnorm_kernel<3, TOGETHER> : add_rmsnorm_kernel<kNormMaxChunks, TOGETHER>;
  fn<<<dim3(rows), kNormThreads, 0, st>>>(x, res, w, h_out, n_out, H, eps);
}

// ------------------------------------------------------ RoPE + KV append (+ head norm)
// blockIdx.x = token, blockIdx.y = a run of 4 * kRopeHeadsPerWave heads; each wave takes
// kRopeHeadsPerWave heads and requests all of them before it works on the first (a short
// prompt is one latency chain per wave: 12 heads in turn took 7.9 us at 126 tokens).  Lane
// i < D/2 owns the pair (i, i + D/2) of every head.  The angle's cosine and sine come from
// the table ((cos, sin) per position and pair, as the decode step uses) when the position is
// inside it, else from a precise sincosf (the angle reaches thousands of radians) of the
// same product - the table holds exactly those values.
constexpr int kRopeHeadsPerWave = 3;
__global__ __launch_bounds__(256) void rope_kv_kernel(
    const bf16_t* __restrict__ qkv, bf16_t* __restrict__ q_out, bf16_t* __restrict__ kc,
    bf16_t* __restrict__ vc, const int32_t* __restrict__ pos, const float* __restrict__ inv_freq,
    const float2* __restrict__ tab, int tab_rows, const bf16_t* __restrict__ qn,
    const bf16_t* __restrict__ kn, float eps, int T, int Hq, int Hkv, int D, int S_max) {
  const int tok = blockIdx.x;  // b*T + t
  const int b = tok / T, t = tok - b * T;
  const int i = threadIdx.x & 63, wave = threadIdx.x >> 6, half = D >> 1;
  const bool active = i < half;
  const int p = pos[b] + t;
  const int nh = Hq + 2 * Hkv;  // heads [0,Hq) are q, [Hq,Hq+Hkv) k, then v
  const int h0 = ((int)blockIdx.y * 4 + wave) * kRopeHeadsPerWave;
  bf16_t lo[kRopeHeadsPerWave], hi[kRopeHeadsPerWave];
#pragma unroll
  for (int u = 0; u < kRopeHeadsPerWave; ++u) {
    lo[u] = 0;
    hi[u] = 0;
    if (active && h0 + u < nh) {
      const bf16_t* src = qkv + (size_t)tok * nh * D + (size_t)(h0 + u) * D;
      lo[u] = src[i];
      hi[u] = src[i + half];
    }
  }
  float sn = 0.f, cs = 1.f;
  if (active) {
    if (tab && p < tab_rows) {
      const float2 v = tab[(size_t)p * half + i];
      cs = v.x;
      sn = v.y;
    } else {
      sincosf((float)p * inv_freq[i], &sn, &cs);
    }
  }
#pragma unroll
  for (int u = 0; u < kRopeHeadsPerWave; ++u) {
    const int head = h0 + u;
    if (head >= nh) break;
    if (head >= Hq + Hkv) {  // v: copy into the cache
      if (active && p < S_max) {
        bf16_t* dst = vc + (((size_t)b * Hkv + (head - Hq - Hkv)) * S_max + p) * D;
        dst[i] = lo[u];
        dst[i + half] = hi[u];
      }
      continue;
    }
    float x1 = bf2f(lo[u]), x2 = bf2f(hi[u]);
    const bool is_q = head < Hq;
    const bf16_t* nw = is_q ? qn : kn;
    if (nw) {  // per-head RMSNorm, rounded to bf16 like a separate rms_norm call
      const float ss = wave_sum(x1 * x1 + x2 * x2);
      const float inv = rsqrtf(ss / (float)D + eps);
      if (active) {
        x1 = bf2f(f2bf(x1 * inv * bf2f(nw[i])));
        x2 = bf2f(f2bf(x2 * inv * bf2f(nw[i + half])));
      }
    }
    if (!active) continue;
    const bf16_t o1 = f2bf(x1 * cs - x2 * sn);
    const bf16_t o2 = f2bf(x2 * cs + x1 * sn);
    if (is_q) {
      bf16_t* dst = q_out + (size_t)tok * Hq * D + (size_t)head * D;
      dst[i] = o1;
      dst[i + half] = o2;
    } else if (p < S_max) {
      bf16_t* dst = kc + (((size_t)b * Hkv + (head - Hq)) * S_max + p) * D;
      dst[i] = o1;
      dst[i + half] = o2;
    }
  }
}

// The same in pieces of 16 bytes where every operand begins at such a piece: D / 8 lanes hold a head, a thread kRopeHeadsPerThread heads of a
// token beside one piece of the table's row.  What bounds it is the memory (a token of 32 / 8 heads of 128 is 24 KB in and out, 4.8 TB/s of it from 4096
// tokens on); the kernel above moves 2 bytes a lane and sums a head's squares over the whole wave.  32 / 8 heads of 128, without | with norms, us: 61 tokens
// 3.5 | 4.4 -> 3.3 | 3.6, 1023 9.5 | 12.5 -> 7.3 | 7.7, 4096 27.3 | 37.8 -> 20.1 | 20.9; of 64, 1023 tokens 8.7 | 11.8 -> 5.5 | 5.7.
// Few heads leave most of 256 threads without one: as many threads as heads take (8000 tokens of 1 / 1 heads of 64 12.5 -> 5.8 us, of 5 / 1 13.3 -> 6.8).
constexpr int kRopeHeadsPerThread = 3;
template <int D, int THREADS>
__global__ __launch_bounds__(THREADS) void rope_kv_wide_kernel(
    const bf16_t* __restrict__ qkv, bf16_t* __restrict__ q_out, bf16_t* __restrict__ kc,
    bf16_t* __restrict__ vc, const int32_t* __restrict__ pos, const float* __restrict__ inv_freq,
    const float2* __restrict__ tab, int tab_rows, const bf16_t* __restrict__ qn,
    const bf16_t* __restrict__ kn, float eps, int T, int Hq, int Hkv, int S_max) {
  constexpr int LPH = D / 8, GROUPS = THREADS / LPH, U = kRopeHeadsPerThread;
  const int tok = blockIdx.x;  // b*T + t
  const int b = tok / T, t = tok - b * T;
  const int sl = threadIdx.x % LPH, h0 = (int)blockIdx.y * GROUPS * U + threadIdx.x / LPH;
  const int nh = Hq + 2 * Hkv;  // heads [0,Hq) are q, [Hq,Hq+Hkv) k, then v
  const bf16_t* const row = qkv + (size_t)tok * nh * D + sl * 8;
  uint4 raw[U], wq = make_uint4(0, 0, 0, 0), wk = wq;
#pragma unroll
  for (int u = 0; u < U; ++u) raw[u] = *reinterpret_cast<const uint4*>(row + (size_t)min(h0 + u * GROUPS, nh - 1) * D);
  if (qn) wq = *reinterpret_cast<const uint4*>(qn + sl * 8);
  if (kn) wk = *reinterpret_cast<const uint4*>(kn + sl * 8);
  const int p = pos[b] + t, pair = sl * 8 % (D / 2);
  float cs[8], sn[8];
  if (p < tab_rows) {
    const float4* tp = reinterpret_cast<const float4*>(tab + (size_t)p * (D / 2) + pair);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float4 v = tp[e];
      cs[2 * e] = v.x, sn[2 * e] = v.y, cs[2 * e + 1] = v.z, sn[2 * e + 1] = v.w;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) sincosf((float)p * inv_freq[pair + e], &sn[e], &cs[e]);
  }
  const bool first = sl < LPH / 2;  // elements of the first half
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int head = h0 + u * GROUPS;
    if (head >= nh) break;
    if (head >= Hq + Hkv) {  // v: copy into the cache
      if (p < S_max) *reinterpret_cast<uint4*>(vc + (((size_t)b * Hkv + (head - Hq - Hkv)) * S_max + p) * D + sl * 8) = raw[u];
      continue;
    }
    const bool is_q = head < Hq;
    const uint32_t r4[4] = {raw[u].x, raw[u].y, raw[u].z, raw[u].w};
    const uint4 w = is_q ? wq : wk;
    const uint32_t w4[4] = {w.x, w.y, w.z, w.w};
    float x[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[2 * e] = bf_lo(r4[e]), x[2 * e + 1] = bf_hi(r4[e]);
    if (is_q ? qn != nullptr : kn != nullptr) {  // per-head RMSNorm, rounded to bf16 like a separate rms_norm call
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(x[e], x[e], ss);
      const float inv = rsqrtf(run_sum<LPH>(ss) / (float)D + eps);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = bf2f(f2bf(x[e] * inv * ((e & 1) ? bf_hi(w4[e >> 1]) : bf_lo(w4[e >> 1]))));
    }
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {  // (the other half's element: half of the head's lanes further)
      const float other = LPH == 16 ? dpp_get<0x128, 0xf>(x[e]) : dpp_get<0x1B, 0xf>(dpp_get<0x141, 0xf>(x[e]));
      y[e] = first ? x[e] * cs[e] - other * sn[e] : x[e] * cs[e] + other * sn[e];
    }
    const uint4 out = make_uint4(pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3]), pack_bf2(y[4], y[5]), pack_bf2(y[6], y[7]));
    if (is_q)
      *reinterpret_cast<uint4*>(q_out + ((size_t)tok * Hq + head) * D + sl * 8) = out;
    else if (p < S_max)
      *reinterpret_cast<uint4*>(kc + (((size_t)b * Hkv + (head - Hq)) * S_max + p) * D + sl * 8) = out;
  }
}

// ------------------------------------------------------------------------ SwiGLU
__global__ __launch_bounds__(256) void swiglu_kernel(const bf16_t* __restrict__ g,
                                                     const bf16_t* __restrict__ u,
                                                     bf16_t* __restrict__ out, int64_t n) {
  int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 2;
  if (i + 1 < n) {
    const uint32_t gv = *reinterpret_cast<const uint32_t*>(g + i);
    const uint32_t uv = *reinterpret_cast<const uint32_t*>(u + i);
    const float g0 = bf_lo(gv), g1 = bf_hi(gv);
    *reinterpret_cast<uint32_t*>(out + i) = pack_bf2(
        g0 / (1.f + __expf(-g0)) * bf_lo(uv), g1 / (1.f + __expf(-g1)) * bf_hi(uv));
  } else if (i < n) {
    const float g0 = bf2f(g[i]);
    out[i] = f2bf(g0 / (1.f + __expf(-g0)) * bf2f(u[i]));
  }
}

// ------------------------------------------------------------------- MoE routing
// One wave per row (route.h).
__global__ __launch_bounds__(64) void router_topk_kernel(const bf16_t* __restrict__ logits,
                                                         int32_t* __restrict__ idx,
                                                         bf16_t* __restrict__ scores, int E,
                                                         int k, int renorm) {
  const int row = blockIdx.x, lane = threadIdx.x;
  int my_id;
  float my_p, tot;
  route_topk_wave(logits + (size_t)row * E, E, k, lane, my_id, my_p, tot);
  if (lane < k) {
    idx[(size_t)row * k + lane] = my_id;
    scores[(size_t)row * k + lane] = route_score(my_p, tot, renorm);
  }
}

// ------------------------------------------------------------------ MoE combine
__global__ __launch_bounds__(256) void moe_combine_kernel(const bf16_t* __restrict__ y,
                                                          const bf16_t* __restrict__ scores,
                                                          const bf16_t* __restrict__ res,
                                                          bf16_t* __restrict__ out, int topk,
                                                          int H) {
  const int t = blockIdx.y;
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= H) return;
  float acc = 0.f;
  for (int j = 0; j < topk; ++j) {
    const float s = bf2f(scores[(size_t)t * topk + j]);
    acc += bf2f(f2bf(bf2f(y[((size_t)t * topk + j) * H + e]) * s));
  }
  float o = bf2f(f2bf(acc));
  if (res) o += bf2f(res[(size_t)t * H + e]);
  out[(size_t)t * H + e] = f2bf(o);
}

// The same sums for H a multiple of 8 (16-byte aligned rows): 8 elements per thread, the
// expert rows of four slots requested together.  Slot order and rounding points as above.
__global__ __launch_bounds__(256) void moe_combine_vec_kernel(const bf16_t* __restrict__ y,
                                                              const bf16_t* __restrict__ scores,
                                                              const bf16_t* __restrict__ res,
                                                              bf16_t* __restrict__ out, int topk,
                                                              int H) {
  const int t = blockIdx.y;
  const int e = (blockIdx.x * 256 + threadIdx.x) * 8;
  if (e >= H) return;
  float acc[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) acc[k] = 0.f;
  const bf16_t* yt = y + (size_t)t * topk * H + e;
  for (int j0 = 0; j0 < topk; j0 += 4) {
    uint4 v[4];
    float sc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = min(j0 + u, topk - 1);
      v[u] = *reinterpret_cast<const uint4*>(yt + (size_t)j * H);
      sc[u] = bf2f(scores[(size_t)t * topk + j]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (j0 + u < topk) {
        const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          acc[2 * k] += bf2f(f2bf(bf_lo(w[k]) * sc[u]));
          acc[2 * k + 1] += bf2f(f2bf(bf_hi(w[k]) * sc[u]));
        }
      }
    }
  }
  float o[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) o[k] = bf2f(f2bf(acc[k]));
  if (res) {
    const uint4 rv = *reinterpret_cast<const uint4*>(res + (size_t)t * H + e);
    const uint32_t w[4] = {rv.x, rv.y, rv.z, rv.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      o[2 * k] += bf_lo(w[k]);
      o[2 * k + 1] += bf_hi(w[k]);
    }
  }
  uint4 ov;
  ov.x = pack_bf2(o[0], o[1]);
  ov.y = pack_bf2(o[2], o[3]);
  ov.z = pack_bf2(o[4], o[5]);
  ov.w = pack_bf2(o[6], o[7]);
  *reinterpret_cast<uint4*>(out + (size_t)t * H + e) = ov;
}

// -------------------------------------------------- argmax + logsumexp over logits
// Stage 1: grid (kArgBlocks, rows): per block (max, argmax, sum exp(x - max)).
// Stage 2: one wave per row merges the blocks.
constexpr int kArgBlocks = 64;

// the wave's largest value and, of equal ones, the first index, in every lane
template <int BIT = 32>
__device__ __forceinline__ void first_of_largest(float& mx, int& mi) {
  const float ov = lane_xor<BIT>(mx);
  const int oi = (int)lane_xor_bits<BIT>((uint32_t)mi);
  if (ov > mx || (ov == mx && oi < mi)) {
    mx = ov;
    mi = oi;
  }
  if constexpr (BIT > 1) first_of_largest<BIT / 2>(mx, mi);
}

__global__ __launch_bounds__(256) void argmax_stage1(const bf16_t* __restrict__ logits,
                                                     float* __restrict__ ws, int V) {
  __shared__ float smax[4], ssum[4];
  __shared__ int sidx[4];
  const int row = blockIdx.y;
  const bf16_t* src = logits + (size_t)row * V;
  // rows of 16-byte multiples (every vocabulary here): the block's share is whole 8-element
  // chunks, up to two per thread, which stay in registers for the second pass
  const bool vec = (V & 7) == 0 && (V >> 3) <= kArgBlocks * 512 && ((uintptr_t)logits & 15) == 0;
  const int per = vec ? (((V >> 3) + kArgBlocks - 1) / kArgBlocks) << 3 : (V + kArgBlocks - 1) / kArgBlocks;
  const int lo = min((int)blockIdx.x * per, V), hi = min(lo + per, V);
  float mx = -INFINITY;
  int mi = 0x7fffffff;
  float xv[16];
  if (vec) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i0 = lo + (threadIdx.x + 256 * u) * 8;
      uint4 v = make_uint4(0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u);  // -inf
      if (i0 < hi) v = *reinterpret_cast<const uint4*>(src + i0);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        xv[8 * u + 2 * k] = bf_lo(w[k]);
        xv[8 * u + 2 * k + 1] = bf_hi(w[k]);
      }
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (xv[8 * u + k] > mx) {
          mx = xv[8 * u + k];
          mi = i0 + k;
        }
    }
  } else {
    for (int i = lo + threadIdx.x; i < hi; i += 256) {
      const float x = bf2f(src[i]);
      if (x > mx) {
        mx = x;
        mi = i;
      }
    }
  }
  first_of_largest(mx, mi);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    smax[wave] = mx;
    sidx[wave] = mi;
  }
  __syncthreads();
  float bm = smax[0];
  int bi = sidx[0];
#pragma unroll
  for (int w = 1; w < 4; ++w)
    if (smax[w] > bm || (smax[w] == bm && sidx[w] < bi)) {
      bm = smax[w];
      bi = sidx[w];
    }
  float se = 0.f;
  if (bm > -INFINITY) {
    if (vec) {
#pragma unroll
      for (int k = 0; k < 16; ++k) se += expf(xv[k] - bm);  // padding is -inf: exp = 0
    } else {
      for (int i = lo + threadIdx.x; i < hi; i += 256) se += expf(bf2f(src[i]) - bm);
    }
  }
  se = wave_sum(se);
  if (lane == 0) ssum[wave] = se;
  __syncthreads();
  if (threadIdx.x == 0) {
    float* d = ws + ((size_t)row * kArgBlocks + blockIdx.x) * 4;
    d[0] = bm;
    d[1] = __int_as_float(bi);
    d[2] = ssum[0] + ssum[1] + ssum[2] + ssum[3];
  }
}

__global__ __launch_bounds__(64) void argmax_stage2(const float* __restrict__ ws,
                                                    int32_t* __restrict__ token,
                                                    float* __restrict__ lse,
                                                    float* __restrict__ logprob,
                                                    int32_t* __restrict__ pos_inc) {
  const int row = blockIdx.x, lane = threadIdx.x;
  const float* s = ws + ((size_t)row * kArgBlocks + lane) * 4;
  float mx = s[0];
  int mi = __float_as_int(s[1]);
  const float bm = mx, bs = s[2];
  first_of_largest(mx, mi);
  float se = (bm > -INFINITY) ? bs * expf(bm - mx) : 0.f;
  se = wave_sum(se);
  if (lane == 0) {
    const float l = mx + logf(se);
    token[row] = mi;
    if (lse) lse[row] = l;
    if (logprob) logprob[row] = mx - l;
    if (pos_inc) pos_inc[row] += 1;
  }
}

}  // namespace

extern "C" int exo_add_rmsnorm(const uint16_t* x, const uint16_t* residual,
                               const uint16_t* weight, uint16_t* h_out, uint16_t* n_out,
                               int rows, int H, float eps, exo_stream_t stream) {
  EXO_REQUIRE(x && weight && n_out, "exo_add_rmsnorm: null pointer");
  EXO_REQUIRE(rows >= 0 && H > 0 && H % 8 == 0 && H <= kNormThreads * 8 * kNormMaxChunks,
              "exo_add_rmsnorm: H=%d must be a multiple of 8 and <= %d", H,
              kNormThreads * 8 * kNormMaxChunks);
  if (rows == 0) return EXO_OK;
  const auto launch = norm_together(rows, H, residual != nullptr) ? launch_add_rmsnorm<true> : launch_add_rmsnorm<false>;
  launch(x, residual, weight, h_out, n_out, rows, H, eps, (hipStream_t)stream);
  EXO_CHECK_LAUNCH("exo_add_rmsnorm");
  return EXO_OK;
}

extern "C" int exo_rope_kv_append_tab(const uint16_t* qkv, uint16_t* q_out, uint16_t* k_cache,
                                      uint16_t* v_cache, const int32_t* pos,
                                      const float* inv_freq, const float* rope_table,
                                      int table_rows, const uint16_t* q_norm_w,
                                      const uint16_t* k_norm_w, float eps, int B, int T, int Hq,
                                      int Hkv, int D, int S_max, exo_stream_t stream) {
  EXO_REQUIRE(qkv && q_out && k_cache && v_cache && pos && inv_freq,
              "exo_rope_kv_append: null pointer");
  EXO_REQUIRE(B > 0 && T > 0 && Hq > 0 && Hkv > 0 && S_max > 0,
              "exo_rope_kv_append: non-positive size");
  EXO_REQUIRE(D == 64 || D == 128, "exo_rope_kv_append: head_dim %d not supported (64, 128)", D);
  EXO_REQUIRE(!rope_table || table_rows > 0, "exo_rope_kv_append: table without rows");
  EXO_REQUIRE((int64_t)B * T <= 0x7fffffff / 2, "exo_rope_kv_append: too many tokens");
  const uintptr_t all = (uintptr_t)qkv | (uintptr_t)q_out | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)rope_table | (uintptr_t)q_norm_w | (uintptr_t)k_norm_w;
  if (!rope_table) table_rows = 0;  // (no position is inside it)
  if ((all & 15) == 0) {
    const int heads = Hq + 2 * Hkv, lanes = heads * (D / 8), threads = lanes <= 64 ? 64 : lanes <= 128 ? 128 : 256;
    const auto fn = D == 128 ? (threads == 64 ? rope_kv_wide_kernel<128, 64> : threads == 128 ? rope_kv_wide_kernel<128, 128> : rope_kv_wide_kernel<128, 256>)
                             : (threads == 64 ? rope_kv_wide_kernel<64, 64> : threads == 128 ? rope_kv_wide_kernel<64, 128> : rope_kv_wide_kernel<64, 256>);
    fn<<<dim3(B * T, exo_ceil_div(heads, threads / (D / 8) * kRopeHeadsPerThread)), threads, 0, (hipStream_t)stream>>>(
        qkv, q_out, k_cache, v_cache, pos, inv_freq, reinterpret_cast<const float2*>(rope_table), table_rows, q_norm_w, k_norm_w, eps, T, Hq, Hkv, S_max);
    EXO_CHECK_LAUNCH("exo_rope_kv_append");
    return EXO_OK;
  }
  const int runs = exo_ceil_div(Hq + 2 * Hkv, 4 * kRopeHeadsPerWave);
  rope_kv_kernel<<<dim3(B * T, runs), 256, 0, (hipStream_t)stream>>>(
      qkv, q_out, k_cache, v_cache, pos, inv_freq, reinterpret_cast<const float2*>(rope_table),
      table_rows, q_norm_w, k_norm_w, eps, T, Hq, Hkv, D, S_max);
  EXO_CHECK_LAUNCH("exo_rope_kv_append");
  return EXO_OK;
}

extern "C" int exo_rope_kv_append(const uint16_t* qkv, uint16_t* q_out, uint16_t* k_cache,
                                  uint16_t* v_cache, const int32_t* pos, const float* inv_freq,
                                  const uint16_t* q_norm_w, const uint16_t* k_norm_w, float eps,
                                  int B, int T, int Hq, int Hkv, int D, int S_max,
                                  exo_stream_t stream) {
  return exo_rope_kv_append_tab(qkv, q_out, k_cache, v_cache, pos, inv_freq, nullptr, 0, q_norm_w,
                                k_norm_w, eps, B, T, Hq, Hkv, D, S_max, stream);
}

extern "C" int exo_swiglu(const uint16_t* gate, const uint16_t* up, uint16_t* out, int64_t n,
                          exo_stream_t stream) {
  EXO_REQUIRE(gate && up && out && n >= 0, "exo_swiglu: null pointer or negative size");
  if (n == 0) return EXO_OK;
  swiglu_kernel<<<dim3(exo_ceil_div((n + 1) / 2, 256)), 256, 0, (hipStream_t)stream>>>(
      gate, up, out, n);
  EXO_CHECK_LAUNCH("exo_swiglu");
  return EXO_OK;
}

extern "C" int exo_router_topk(const uint16_t* logits, int32_t* idx, uint16_t* scores, int rows,
                               int E, int k, int renorm, exo_stream_t stream) {
  EXO_REQUIRE(logits && idx && scores, "exo_router_topk: null pointer");
  EXO_REQUIRE(E > 0 && E <= 256 && k > 0 && k <= 16 && k <= E && rows >= 0,
              "exo_router_topk: need 0<E<=256, 0<k<=min(16,E); got E=%d k=%d", E, k);
  if (rows == 0) return EXO_OK;
  router_topk_kernel<<<dim3(rows), 64, 0, (hipStream_t)stream>>>(logits, idx, scores, E, k,
                                                                  renorm);
  EXO_CHECK_LAUNCH("exo_router_topk");
  return EXO_OK;
}

extern "C" int exo_moe_combine(const uint16_t* y, const uint16_t* scores,
                               const uint16_t* residual, uint16_t* out, int T, int topk, int H,
                               exo_stream_t stream) {
  EXO_REQUIRE(y && scores && out, "exo_moe_combine: null pointer");
  EXO_REQUIRE(T >= 0 && topk > 0 && H > 0 && T <= 65535, "exo_moe_combine: bad size");
  if (T == 0) return EXO_OK;
  const bool vec = H % 8 == 0 &&
                   (((uintptr_t)y | (uintptr_t)residual | (uintptr_t)out) & 15) == 0;
  if (vec)
    moe_combine_vec_kernel<<<dim3(exo_ceil_div(H / 8, 256), T), 256, 0, (hipStream_t)stream>>>(
        y, scores, residual, out, topk, H);
  else
    moe_combine_kernel<<<dim3(exo_ceil_div(H, 256), T), 256, 0, (hipStream_t)stream>>>(
        y, scores, residual, out, topk, H);
  EXO_CHECK_LAUNCH("exo_moe_combine");
  return EXO_OK;
}

extern "C" int exo_put_i32(int32_t* dst, const int32_t* values, int n, exo_stream_t stream) {
  EXO_REQUIRE(n >= 0, "exo_put_i32: n=%d is negative", n);
  EXO_REQUIRE(n == 0 || (dst && values), "exo_put_i32: null pointer");
  for (int i = 0; i < n; i += EXO_PUT_INTS) {
    PutInts v;
    const int m = n - i < EXO_PUT_INTS ? n - i : EXO_PUT_INTS;
    memcpy(v.v, values + i, m * sizeof(int32_t));
    put_i32_kernel<<<dim3(exo_ceil_div(m, 64)), 64, 0, (hipStream_t)stream>>>(dst + i, v, m);
  }
  EXO_CHECK_LAUNCH("exo_put_i32");
  return EXO_OK;
}

extern "C" int64_t exo_argmax_workspace(int rows) {
  return (int64_t)rows * kArgBlocks * 4 * (int64_t)sizeof(float);
}

extern "C" int exo_argmax_logsumexp(const uint16_t* logits, int32_t* token, float* lse,
                                    float* logprob, float* workspace, int32_t* pos_inc,
                                    int rows, int V, exo_stream_t stream) {
  EXO_REQUIRE(logits && token && workspace, "exo_argmax_logsumexp: null pointer");
  EXO_REQUIRE(rows >= 0 && rows <= 65535 && V > 0, "exo_argmax_logsumexp: bad size");
  if (rows == 0) return EXO_OK;
  argmax_stage1<<<dim3(kArgBlocks, rows), 256, 0, (hipStream_t)stream>>>(logits, workspace, V);
  argmax_stage2<<<dim3(rows), 64, 0, (hipStream_t)stream>>>(workspace, token, lse, logprob,
                                                           pos_inc);
  EXO_CHECK_LAUNCH("exo_argmax_logsumexp");
  return EXO_OK;
}
