// Recurrent mixers of layer-list decoders.  Per head, over a sequence, with S (keys x values) from zero:
//     S <- diag(a_t) S + k_t v_t^T,     o_t = S^T q_t
// Options, each a parameter of the layer: the decay per key channel (a low-rank product's output through
// a logarithm of the sigmoid) or per head (exp(-a dt), values scaled by dt), queries and keys per head or
// shared by a group of heads, a skip o_t += D v_t, a causal convolution per channel with silu in front
// of queries, keys and values.  Or exponential gates i_t, f_t per head, kept in range by their running
// maximum m_t = max(f_t + m_(t-1), i_t) (logarithms): decay exp(f_t + m_(t-1) - m_t), values scaled by
// exp(i_t - m_t), which to everything behind the gates is a decay per head and a step size.  Decays, step sizes, states and their products are float32; where a
// float32 factor enters a bf16 matrix product it goes in as two bf16 terms (value and remainder).
//
// A cache row owns a state slot (map: row -> slot): the states, and a ring of the convolution's latest
// `taps` inputs in which position p sits at p % taps - the entry a step writes is none that it reads.  A
// sequence at position 0 starts from zero whatever its slot holds.
//
// Single tokens: recur_step_kernel does it all, a workgroup per (row, head, range of value columns).
// Portions of prompts, cut into chunks of 64 tokens, c_t = sum of the binary logarithms of the decays of
// the chunk's tokens up to t (every exponent below is <= 0):
//   recur_prep / recur_conv / recur_gates   c, dt, and the convolved inputs, the maxima
//   recur_scores  per chunk   A[i][j] = sum_d q_i k_j 2^(c_i - c_j), j <= i; decay per head: q_i . k_j
//   recur_carry   per portion, tiles of the state in registers: leaves the state ahead of every chunk,
//                             S <- 2^c_end S + sum_t 2^(c_end - c_t) k_t v_t^T
//   recur_out     per chunk   o_i = 2^c_i q_i S + sum_j A[i][j] v_j (+ D v_i)
// A decay per channel does not factor out of a score without overflow, so its scores are formed for
// 16-token blocks: between blocks both factors are taken to the query block's start, between a block's
// halves to its middle, and inside a half each pair has its own exponentials.  That launch also leaves 2^c q and, transposed, 2^(c_end - c) k as
// matrix operands; recur_carry leaves the states as operands too (value columns x keys).
#include "../../include/exo_mi355x.h"
#include "dense.h"

#include <type_traits>

namespace {

typedef __attribute__((__vector_size__(4 * sizeof(int)))) int int4v;

constexpr int kChunk = 64;
constexpr int kRec = 8;  // ints of a chunk's record: row, cache row, position, tokens, portion's first position

// the arguments and where the parts of the workspace lie
struct Rec : exo_recurrence {
  float* scores;         // [chunk][group][64][64]
  void* states;          // T [terms][chunk][head][lds][dp]: the state ahead of a chunk, value columns x keys
  void *qhat, *khat;     // decay per channel: T [terms][chunk][head][64][dp], [terms][chunk][head][dp][64]
  size_t nstates, nhat;  // elements of a term
  int dp;                // dim rounded up to 64, zeros behind dim
};

constexpr float kLog2e = 1.4426950408889634f, kLn2 = 0.6931471805599453f;
__device__ __forceinline__ float pow2(float x) { return __builtin_amdgcn_exp2f(x); }
// max(z, 0) + log(1 + e), e = exp(-|z|).  u = 1 + e rounds, so log(u) belongs to u - 1 instead of e: taken
// times e / (u - 1) it keeps its relative precision for small e.
__device__ __forceinline__ float softplus(float z) {
  const float e = pow2(-fabsf(z) * kLog2e), u = 1.f + e, d = u - 1.f;
  const float l = d == 0.f ? e : __builtin_amdgcn_logf(u) * kLn2 * (e * __builtin_amdgcn_rcpf(d));
  return fmaxf(z, 0.f) + l;
}
__device__ __forceinline__ float sigmoidf(float z) { return 1.f / (1.f + expf(-z)); }

template <typename T>
__device__ __forceinline__ const T* as(const void* p) {
  return reinterpret_cast<const T*>(p);
}

// a float32 operand of a matrix product
template <typename T>
struct Split;
template <>
struct Split<bf16_t> {
  uint4 hi, lo;
  __device__ __forceinline__ void set(const float (&f)[8]) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      h[i] = pack_bf2(f[2 * i], f[2 * i + 1]);
      l[i] = pack_bf2(f[2 * i] - bf_lo(h[i]), f[2 * i + 1] - bf_hi(h[i]));
    }
    hi = uint4{h[0], h[1], h[2], h[3]};
    lo = uint4{l[0], l[1], l[2], l[3]};
  }
};
template <>
struct Split<float> {
  uint4 hi;
  __device__ __forceinline__ void set(const float (&f)[4]) { hi = __builtin_bit_cast(uint4, floatx4{f[0], f[1], f[2], f[3]}); }
};
// its value term from p, the remainder term (bf16) n elements behind
template <typename T>
__device__ __forceinline__ Split<T> split_at(const void* p, size_t at, size_t n) {
  Split<T> s;
  s.hi = *reinterpret_cast<const uint4*>(reinterpret_cast<const T*>(p) + at);
  if constexpr (sizeof(T) == 2) s.lo = *reinterpret_cast<const uint4*>(reinterpret_cast<const T*>(p) + n + at);
  return s;
}
// four consecutive elements of such an operand
template <typename T>
__device__ __forceinline__ void split_store(void* p, size_t at, size_t n, const float (&f)[4]) {
  if constexpr (sizeof(T) == 2) {
    const uint32_t h0 = pack_bf2(f[0], f[1]), h1 = pack_bf2(f[2], f[3]);
    *reinterpret_cast<uint2*>(reinterpret_cast<T*>(p) + at) = uint2{h0, h1};
    *reinterpret_cast<uint2*>(reinterpret_cast<T*>(p) + n + at) =
        uint2{pack_bf2(f[0] - bf_lo(h0), f[1] - bf_hi(h0)), pack_bf2(f[2] - bf_lo(h1), f[3] - bf_hi(h1))};
  } else {
    *reinterpret_cast<floatx4*>(reinterpret_cast<T*>(p) + at) = floatx4{f[0], f[1], f[2], f[3]};
  }
}
template <typename T>
__device__ __forceinline__ floatx4 mma(const Split<T>& a, const uint4& b, floatx4 c) {
  if constexpr (sizeof(T) == 2) c = Elem<T>::mma16(a.lo, b, c);
  return Elem<T>::mma16(a.hi, b, c);
}
template <typename T>
__device__ __forceinline__ floatx4 mma(const uint4& a, const Split<T>& b, floatx4 c) {
  if constexpr (sizeof(T) == 2) c = Elem<T>::mma16(a, b.lo, c);
  return Elem<T>::mma16(a, b.hi, c);
}
template <typename T>
__device__ __forceinline__ floatx4 mma(const Split<T>& a, const Split<T>& b, floatx4 c) {
  if constexpr (sizeof(T) == 2) {
    c = Elem<T>::mma16(a.lo, b.hi, c);
    c = Elem<T>::mma16(a.hi, b.lo, c);
  }
  return Elem<T>::mma16(a.hi, b.hi, c);
}

// N elements from p, zero from `left` on
template <typename T, int N>
__device__ __forceinline__ void load_n(const T* p, T (&f)[N], bool vec, int left) {
  if (vec && left >= N) {
    if constexpr (N * sizeof(T) >= 16) {
#pragma unroll
      for (int i = 0; i < (int)(N * sizeof(T) / 16); ++i)
        *reinterpret_cast<uint4*>(&f[i * 16 / sizeof(T)]) = *reinterpret_cast<const uint4*>(p + i * 16 / sizeof(T));
    } else {
      *reinterpret_cast<uint2*>(&f[0]) = *reinterpret_cast<const uint2*>(p);
    }
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) f[i] = i < left ? p[i] : T(0);
  }
}

struct Chunk {
  int row, crow, pos, n, pos0;
  __device__ __forceinline__ explicit Chunk(const int32_t* list, int i) {
    const int32_t* c = list + (size_t)i * kRec;
    row = c[0], crow = c[1], pos = c[2], n = min(c[3], kChunk), pos0 = c[4];
  }
};

// ------------------------------------------------------------------------------ what enters a recurrence
// c per key channel: z = low-rank product + bias, log decay = -softplus(-z) / tau, summed over the chunk
constexpr int kRankStep = 16, kSeg = kChunk / 4;

// 64 channels per workgroup; a wave takes a quarter of the tokens
__global__ __launch_bounds__(256) void recur_prep_channel_kernel(const Rec p) {
  __shared__ __attribute__((aligned(16))) float low[kChunk][kRankStep];
  __shared__ float total[4][64];
  const Chunk ck(p.chunks, blockIdx.x);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int c = blockIdx.y * 64 + lane, C = p.heads * p.dim, cc = min(c, C - 1), t0 = wave * kSeg;
  float acc[kSeg];
  const float b = p.decay_b[cc];
#pragma unroll
  for (int t = 0; t < kSeg; ++t) acc[t] = b;
  for (int j0 = 0; j0 < p.rank; j0 += kRankStep) {
    __syncthreads();
    for (int i = threadIdx.x; i < kChunk * kRankStep; i += 256) {
      const int t = i / kRankStep, j = i % kRankStep;
      low[t][j] = t < ck.n && j0 + j < p.rank ? p.low[(size_t)(ck.row + t) * p.ldlow + j0 + j] : 0.f;
    }
    __syncthreads();
    float w[kRankStep];
#pragma unroll
    for (int j = 0; j < kRankStep; ++j) w[j] = j0 + j < p.rank ? p.decay_w[(size_t)(j0 + j) * C + cc] : 0.f;
#pragma unroll
    for (int t = 0; t < kSeg; ++t)
#pragma unroll
      for (int j = 0; j < kRankStep; j += 4) {
        const floatx4 l = *reinterpret_cast<const floatx4*>(&low[t0 + t][j]);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t] = fmaf(w[j + e], l[e], acc[t]);
      }
  }
  const float scale = p.inv_tau * kLog2e;
  float sum = 0.f;
#pragma unroll
  for (int t = 0; t < kSeg; ++t) {
    sum -= softplus(-acc[t]) * scale;
    acc[t] = sum;
  }
  total[wave][lane] = sum;
  __syncthreads();
  float base = 0.f;
  for (int w = 0; w < wave; ++w) base += total[w][lane];
  if (c >= C) return;
#pragma unroll
  for (int t = 0; t < kSeg; ++t)
    if (t0 + t < ck.n) p.cum[(size_t)(ck.row + t0 + t) * p.ldcum + c] = base + acc[t];
}

// c and dt per head: a wave per head, a lane per token
__device__ __forceinline__ void prep_heads(const Rec& p, const Chunk& ck, int h) {
  const int lane = threadIdx.x & 63;
  if (h >= p.heads) return;
  const bool on = lane < ck.n;
  const size_t row = (size_t)ck.row + min(lane, ck.n - 1);
  const float dt = softplus(p.dt_raw[row * p.lddt + h] + p.dt_bias[h]);
  float s = on ? -p.decay_rate[h] * dt * kLog2e : 0.f;
#pragma unroll
  for (int o = 1; o < 64; o *= 2) {
    const float u = __shfl_up(s, o, 64);
    if (lane >= o) s += u;
  }
  if (on) {
    p.cum[(size_t)h * p.ldcum + row] = s;
    p.dt[(size_t)h * p.ldcum + row] = dt;
  }
}

// causal convolution per channel and silu, 16 tokens per thread; the last rows of workgroups: prep_heads
constexpr int kConvTokens = 16;

template <typename T, int TM>
__global__ __launch_bounds__(256) void recur_conv_kernel(const Rec p) {
  const Chunk ck(p.chunks, blockIdx.x / (kChunk / kConvTokens));
  const int part = blockIdx.x % (kChunk / kConvTokens), t0 = part * kConvTokens, c = blockIdx.y * 256 + threadIdx.x;
  const int conv_rows = (p.channels + 255) / 256;
  if ((int)blockIdx.y >= conv_rows) {
    prep_heads(p, ck, (((int)blockIdx.y - conv_rows) * (kChunk / kConvTokens) + part) * 4 + (threadIdx.x >> 6));
    return;
  }
  if (t0 >= ck.n || c >= p.channels) return;
  float w[TM], x[TM];  // the latest TM inputs, oldest first (taps < TM: zero weights in front)
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int tap = i - (TM - p.taps);
    w[i] = tap >= 0 ? p.conv_w[(size_t)tap * p.channels + c] : 0.f;
  }
  const float b = p.conv_b[c];
  const T* raw = as<T>(p.raw) + (size_t)ck.row * p.ldraw + c;
  const T* ring = as<T>(p.ring) + (size_t)p.map[ck.crow] * p.taps * p.channels + c;
#pragma unroll
  for (int i = 0; i < TM - 1; ++i) {
    const int back = TM - 1 - i, at = ck.pos + t0 - back;  // position of that input
    x[i] = 0.f;
    if (back < p.taps && at >= 0)
      x[i] = at >= ck.pos0 ? Elem<T>::load(raw[(ptrdiff_t)(t0 - back) * p.ldraw])
                           : Elem<T>::load(ring[(size_t)(at % p.taps) * p.channels]);
  }
  T in[kConvTokens];
#pragma unroll
  for (int t = 0; t < kConvTokens; ++t) in[t] = raw[(size_t)min(t0 + t, ck.n - 1) * p.ldraw];
  T* out = reinterpret_cast<T*>(p.act) + (size_t)ck.row * p.ldact + c;
#pragma unroll
  for (int t = 0; t < kConvTokens; ++t) {
    x[TM - 1] = Elem<T>::load(in[t]);
    float y = b;
#pragma unroll
    for (int i = 0; i < TM; ++i) y = fmaf(w[i], x[i], y);
    if (t0 + t < ck.n) out[(size_t)(t0 + t) * p.ldact] = Elem<T>::make(y * sigmoidf(y));
#pragma unroll
    for (int i = 0; i < TM - 1; ++i) x[i] = x[i + 1];
  }
}

// ---- exponential gates
__device__ __forceinline__ float capped(float z, float cap) { return cap * tanhf(z / cap); }
// logarithms of the input and the forget gate
__device__ __forceinline__ float2 log_gates(const Rec& p, size_t row, int h) {
  const float i = capped(p.gate_i[row * p.ldgate + h], p.gate_cap), f = capped(p.gate_f[row * p.ldgate + h], p.gate_cap);
  return float2{i, -softplus(-f)};
}
__device__ __forceinline__ double* peak_at(const Rec& p, int slot, int pos, int h) {
  return p.peak + ((size_t)slot * 2 + (pos & 1)) * p.heads + h;
}

// c, dt and the running maximum along a portion, one head per workgroup, a chunk per wave and pass.  A step
// takes m to max(F + m, M), F = f and M = i; two steps one after the other are such a step again.
constexpr int kGateWaves = 16;

__global__ __launch_bounds__(64 * kGateWaves) void recur_gates_kernel(const Rec p) {
  __shared__ double2 total[kGateWaves];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), h = blockIdx.x;
  const int32_t* seq = p.seqs + 4 * (size_t)blockIdx.y;
  const int first = seq[0], count = seq[1];
  const Chunk c0(p.chunks, first), last(p.chunks, first + count - 1);
  const int slot = p.map[c0.crow];
  double m = c0.pos0 > 0 ? *peak_at(p, slot, c0.pos0 - 1, h) : 0.;  // ahead of the pass
  for (int i0 = 0; i0 < count; i0 += kGateWaves) {
    const bool mine = i0 + wave < count;
    const Chunk ck(p.chunks, first + min(i0 + wave, count - 1));
    const bool on = mine && lane < ck.n;
    const size_t row = (size_t)ck.row + min(lane, ck.n - 1);
    const float2 g = log_gates(p, row, h);  // i, f
    double F = on ? g.y : 0., M = on ? (double)g.x : -INFINITY;
#pragma unroll
    for (int o = 1; o < 64; o *= 2) {  // up to and with this lane
      const double f1 = __shfl_up(F, o, 64), m1 = __shfl_up(M, o, 64);
      if (lane >= o) {
        M = fmax(F + m1, M);
        F += f1;
      }
    }
    if (lane == 63) total[wave] = double2{F, M};
    __syncthreads();
    double ahead = m;
#pragma unroll
    for (int w = 0; w < kGateWaves; ++w) {
      if (w == wave) ahead = m;
      m = fmax(total[w].x + m, total[w].y);  // (the step of a chunk past the last: nothing)
    }
    const double mt = fmax(F + ahead, M);
    if (on) {
      p.cum[(size_t)h * p.ldcum + row] = (float)(F + ahead - mt) * kLog2e;
      p.dt[(size_t)h * p.ldcum + row] = expf((float)(g.x - mt));
      p.peaks[row * p.ldpeaks + h] = (float)mt;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) *peak_at(p, slot, last.pos + last.n - 1, h) = m;
}

// ------------------------------------------------------------------------------ chunks
// the value columns [e0, e0 + 64) of a chunk, transposed: vt[column][token], zero past n and E
template <typename T>
constexpr int kVStride = kChunk + 16 / (int)sizeof(T);

// one element, as the bits of the low half or of a whole register
template <typename T>
__device__ __forceinline__ uint32_t raw_one(__amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff) {
  if constexpr (sizeof(T) == 2)
    return __builtin_amdgcn_raw_buffer_load_b16(rs, voff, soff, 0);
  else
    return __builtin_amdgcn_raw_buffer_load_b32(rs, voff, soff, 0);
}
// four value (or key) columns of a token on their way to LDS.  VEC: whole 8- or 16-byte loads through a range-
// checked buffer, so that nothing branches and nothing is waited for before the columns are used.
template <typename T, bool VEC>
struct Quad4 {
  uint32_t w[VEC ? (int)sizeof(T) : 4];
  // voff: the thread's place (kPastEnd: none), soff: the same for all
  __device__ __forceinline__ void request(__amdgpu_buffer_rsrc_t rv, uint32_t voff, uint32_t soff, int left) {
    if constexpr (VEC) {
      if constexpr (sizeof(T) == 2) {
        const uint2 v = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rv, voff, soff, 0));
        w[0] = v.x, w[1] = v.y;
      } else {
        const uint4 v = buf_load16(rv, voff, soff);
        w[0] = v.x, w[1] = v.y, w[2] = v.z, w[3] = v.w;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = raw_one<T>(rv, e < left ? voff + e * (uint32_t)sizeof(T) : kPastEnd, soff);
    }
  }
  __device__ __forceinline__ T at(int e) const {
    if constexpr (VEC && sizeof(T) == 2)
      return T(w[e / 2] >> (16 * (e & 1)));
    else if constexpr (sizeof(T) == 2)
      return T(w[e]);
    else
      return __builtin_bit_cast(T, w[e]);
  }
};

// scores of a chunk, decay per head: the plain products of a group's queries and keys
template <typename T>
__global__ __launch_bounds__(256) void recur_scores_head_kernel(const Rec p) {
  constexpr int KV = Elem<T>::kVec;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const Chunk ck(p.chunks, blockIdx.x);
  const int grp = blockIdx.y, i0 = wave * 16;
  if (i0 >= ck.n) return;
  const T* qp = as<T>(p.q) + (size_t)(ck.row + min(i0 + r, ck.n - 1)) * p.ldq + grp * p.dim;
  const T* kp[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) kp[j] = as<T>(p.k) + (size_t)(ck.row + min(j * 16 + r, ck.n - 1)) * p.ldk + grp * p.dim;
  floatx4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < p.dim; s += 4 * KV) {
    const int d = s + g * KV, left = p.dim - d;
    struct alignas(16) Vec {
      T e[KV];
    } a, b[4];
    load_n<T, KV>(qp + d, a.e, p.qk_vec != 0, left);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j <= wave) load_n<T, KV>(kp[j] + d, b[j].e, p.qk_vec != 0, left);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j <= wave) acc[j] = Elem<T>::mma16(__builtin_bit_cast(uint4, a), __builtin_bit_cast(uint4, b[j]), acc[j]);
  }
  float* out = p.scores + ((size_t)blockIdx.x * p.groups + grp) * kChunk * kChunk;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (j <= wave) {
#pragma unroll
      for (int e = 0; e < 4; ++e) out[(i0 + 4 * g + e) * kChunk + j * 16 + r] = acc[j][e] * p.q_scale;
    }
}

// scores of 16 queries of a chunk, decay per key channel (queries and keys per head); 64 channels at a
// time in LDS.  Wave j takes the keys of block j ahead of the queries' own.  Of that one, wave 3 takes the
// later eight queries with the earlier eight keys like an earlier block; the two squares of eight are
// dealt out over the waves by channels.
template <typename T>
__global__ __launch_bounds__(256) void recur_scores_channel_kernel(const Rec p) {
  constexpr int KV = Elem<T>::kVec, ST = 68;
  __shared__ __attribute__((aligned(16))) float qs[16][ST], ks[kChunk][ST], cs[kChunk][ST];
  __shared__ float part[4][128], cross[256];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int sk = (lane >> 5) * 8 + (lane & 7), sq = (lane >> 5) * 8 + ((lane >> 3) & 3) * 2;  // a square's key, two queries
  const Chunk ck(p.chunks, blockIdx.x);
  const int h = blockIdx.y, block = 3 - (int)blockIdx.z, i0 = block * 16;  // (the longest first)
  if (i0 >= ck.n) return;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  float own[2] = {0.f, 0.f};
  T kr[16], qr[4];
  float cr[16];
  auto request = [&](int d) {
    const int dc = h * p.dim + min(d, p.dim - 1);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const size_t row = (size_t)ck.row + min(min(wave + 4 * j, i0 + 15), ck.n - 1);
      kr[j] = as<T>(p.k)[row * p.ldk + dc];
      cr[j] = p.cum[row * p.ldcum + dc];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) qr[j] = as<T>(p.q)[((size_t)ck.row + min(i0 + wave + 4 * j, ck.n - 1)) * p.ldq + dc];
  };
  request(lane);
  for (int d0 = 0; d0 < p.dim; d0 += 64) {
    const bool on = d0 + lane < p.dim;
    __syncthreads();  // (the channels before have been read)
#pragma unroll
    for (int j = 0; j < 16; ++j)
    {
      ks[wave + 4 * j][lane] = on ? Elem<T>::load(kr[j]) : 0.f;
      cs[wave + 4 * j][lane] = on ? cr[j] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) qs[wave + 4 * j][lane] = on ? Elem<T>::load(qr[j]) * p.q_scale : 0.f;
    __syncthreads();
    request(min(d0 + 64, p.dim - 1) + lane);
    {
      const int i = tid >> 4, c = (tid & 15) * 4;
      float f[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) f[e] = qs[i][c + e] * pow2(cs[i0 + i][c + e]);
      split_store<T>(p.qhat, (((size_t)blockIdx.x * p.heads + h) * kChunk + i0 + i) * p.dp + d0 + c, p.nhat, f);
    }
    if (i0 + 16 >= ck.n) {  // (the last block has all the keys)
      const int c = tid >> 2, t0 = (tid & 3) * 16;
      const float cend = cs[ck.n - 1][c];
#pragma unroll
      for (int tk = 0; tk < 16; tk += KV) {
        float f[KV];
#pragma unroll
        for (int e = 0; e < KV; ++e) {
          const int t = t0 + tk + e;
          f[e] = t < ck.n ? ks[t][c] * pow2(cend - cs[t][c]) : 0.f;
        }
        Split<T> out;
        out.set(f);
        T* dst = reinterpret_cast<T*>(p.khat) + (((size_t)blockIdx.x * p.heads + h) * p.dp + d0 + c) * kChunk + t0 + tk;
        *reinterpret_cast<uint4*>(dst) = out.hi;
        if constexpr (sizeof(T) == 2) *reinterpret_cast<uint4*>(dst + p.nhat) = out.lo;
      }
    }
    const int db = min(64, p.dim - d0);
    // earlier keys: both factors relative to the last token ahead of the queries
    if (wave < block || wave == 3) {
      const int ref = wave < block ? i0 - 1 : i0 + 7, key = wave < block ? wave * 16 + r : i0 + r;
      const float qon = wave < block || r >= 8 ? 1.f : 0.f, kon = wave < block || r < 8 ? 1.f : 0.f;
      for (int s = 0; s < db; s += 4 * KV) {
        const int dd = s + g * KV;
        float fa[KV], fb[KV];
#pragma unroll
        for (int e = 0; e < KV; ++e) {
          const float base = cs[ref][dd + e];
          fa[e] = qon * qs[r][dd + e] * pow2(fminf(cs[i0 + r][dd + e] - base, 0.f));
          fb[e] = kon * ks[key][dd + e] * pow2(fminf(base - cs[key][dd + e], 0.f));
        }
        Split<T> a, b;
        a.set(fa);
        b.set(fb);
        acc = mma<T>(a, b, acc);
      }
    }
    // the squares, pair by pair
    for (int dd = wave * 16; dd < min(db, wave * 16 + 16); dd += 4) {
      const floatx4 k = *reinterpret_cast<const floatx4*>(&ks[i0 + sk][dd]), c = *reinterpret_cast<const floatx4*>(&cs[i0 + sk][dd]);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const floatx4 q = *reinterpret_cast<const floatx4*>(&qs[sq + e][dd]), b = *reinterpret_cast<const floatx4*>(&cs[i0 + sq + e][dd]);
#pragma unroll
        for (int i = 0; i < 4; ++i) own[e] = fmaf(q[i] * k[i], pow2(fminf(b[i] - c[i], 0.f)), own[e]);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < 2; ++e) part[wave][(sq + e) * 8 + (sk & 7)] = own[e];
  float* out = p.scores + (((size_t)blockIdx.x * p.heads + h) * kChunk + i0) * kChunk;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (wave < block)
      out[(4 * g + e) * kChunk + wave * 16 + r] = acc[e];
    else if (wave == 3)
      cross[(4 * g + e) * 16 + r] = acc[e];
  }
  __syncthreads();
  const int qi = tid >> 4, kj = tid & 15, at = qi * 8 + (kj & 7);
  out[qi * kChunk + i0 + kj] = (qi ^ kj) & 8 ? cross[tid] : part[0][at] + part[1][at] + part[2][at] + part[3][at];
}

template <typename T, bool CHANNEL, int NE>
constexpr int carry_lds() {
  constexpr int tile = 16 * NE * kVStride<T> * (int)sizeof(T);
  return 2 * tile + 2 * tile * (sizeof(T) == 2 ? 2 : 1) + (CHANNEL ? 0 : 2 * 64 * kVStride<T> * (int)sizeof(T)) + 2 * kChunk * 4;
}

// Along a portion's chunks with a tile of the state, 64 keys x (16 NE) value columns, in registers.  One
// workgroup per CU at most, so the loop is kept short: every address is a thread's fixed offset plus a
// scalar that steps with the chunk, and the ends of rows and of the portion are the buffers' ends.
// blockIdx.y == heads: the convolution's ring takes the portion's last inputs.
template <typename T, bool CHANNEL, int NE, bool VEC>
__global__ __launch_bounds__(256) void recur_carry_kernel(const Rec p) {
  constexpr int KV = Elem<T>::kVec, KS = kChunk / (4 * KV), VS = kVStride<T>, EB = sizeof(T), NT = sizeof(T) == 2 ? 2 : 1;
  // two buffers each: values [column][token], keys [key][token] (decay per head), the state on its way
  // out [term][column][key], weights of the tokens (decay per head)
  extern __shared__ __attribute__((aligned(16))) char lds_raw[];
  constexpr int TILE = 16 * NE * VS;
  T(*vt)[TILE] = reinterpret_cast<T(*)[TILE]>(lds_raw);
  T(*sv)[NT][TILE] = reinterpret_cast<T(*)[NT][TILE]>(vt + 2);
  T(*kt)[64 * VS] = reinterpret_cast<T(*)[64 * VS]>(sv + 2);
  float(*wt)[kChunk] = reinterpret_cast<float(*)[kChunk]>(kt + (CHANNEL ? 0 : 2));
  const int32_t* seq = p.seqs + 4 * (size_t)blockIdx.z;
  const int first = seq[0], count = seq[1];
  const Chunk c0(p.chunks, first), cl(p.chunks, first + count - 1);
  const int slot = p.map[c0.crow];
  if ((int)blockIdx.y == p.heads) {
    const int end = cl.pos + cl.n;  // one past the last position
    for (int c = blockIdx.x * 256 + threadIdx.x; c < p.channels; c += gridDim.x * 256) {
      T* ring = reinterpret_cast<T*>(p.ring) + (size_t)slot * p.taps * p.channels + c;
      for (int at = max(end - p.taps, c0.pos0); at < end; ++at)
        ring[(size_t)(at % p.taps) * p.channels] = as<T>(p.raw)[(size_t)(c0.row + at - c0.pos0) * p.ldraw + c];
    }
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int h = blockIdx.y, gk = h / (p.heads / p.groups), ne = (p.lds + 16 * NE - 1) / (16 * NE);
  const int e0 = ((int)blockIdx.x % ne) * 16 * NE, d0 = ((int)blockIdx.x / ne) * 64 + wave * 16;
  const int total = cl.row + cl.n - c0.row;  // tokens: a portion's chunks lie one behind the other
  // the state tile: lane (g, r) has keys d0 + 4g .. + 3 of column r
  floatx4 s[NE];
  float* st = p.state + ((size_t)slot * p.heads + h) * p.dim * p.lds;
#pragma unroll
  for (int j = 0; j < NE; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d = d0 + 4 * g + e, col = e0 + j * 16 + r;
      s[j][e] = c0.pos0 > 0 && d < p.dim && col < p.lds ? st[(size_t)d * p.lds + col] : 0.f;
    }
  // ---- where a chunk's parts lie
  constexpr int CQ = 4 * NE, TP = kChunk * CQ / 256;  // quads of columns, tokens per thread
  const int q = (tid % CQ) * 4, t0 = (tid / CQ) * TP;
  auto rows = [&](const void* base, int ld, int bytes) {  // the portion's rows of a matrix, from its first
    return buf_of(reinterpret_cast<const char*>(base) + (size_t)c0.row * ld * bytes, (uint32_t)total * ld * bytes);
  };
  const __amdgpu_buffer_rsrc_t rv = rows(p.v, p.ldv, EB), rk = rows(p.k, p.ldk, EB);
  const size_t mine = (size_t)h * p.ldcum + c0.row;  // decay per head: a head's tokens in a run
  const __amdgpu_buffer_rsrc_t rc = CHANNEL ? rows(p.cum, p.ldcum, 4) : buf_of(p.cum + mine, total * 4u),
                               rd = CHANNEL ? rc : buf_of(p.dt + mine, total * 4u);
  uint32_t voff[TP], koff[4];
#pragma unroll
  for (int k = 0; k < TP; ++k)
    voff[k] = e0 + q < p.vdim ? ((uint32_t)(t0 + k) * p.ldv + h * p.vdim + e0 + q) * EB : kPastEnd;
  const int kq = (tid & 15) * 4, kt0 = (tid >> 4) * 4, dq = ((int)blockIdx.x / ne) * 64 + kq;  // decay per head: the keys
#pragma unroll
  for (int k = 0; k < 4; ++k) koff[k] = dq < p.dim ? ((uint32_t)(kt0 + k) * p.ldk + gk * p.dim + dq) * EB : kPastEnd;
  const uint32_t cstep = (uint32_t)p.heads * p.dp * kChunk * EB;  // khat, per chunk
  const __amdgpu_buffer_rsrc_t rh = buf_of(as<T>(p.khat) + ((size_t)first * p.heads + h) * p.dp * kChunk, CHANNEL ? count * cstep : 0u);
  const __amdgpu_buffer_rsrc_t rl =
      buf_of(as<T>(p.khat) + p.nhat + ((size_t)first * p.heads + h) * p.dp * kChunk, CHANNEL ? count * cstep : 0u);
  const uint32_t hoff = ((uint32_t)(d0 + r) * kChunk + g * KV) * EB;
  const uint32_t eoff = (h * p.dim + d0 + 4 * g) * 4u, woff = lane * 4u;
  const uint32_t sstep = (uint32_t)p.heads * p.lds * p.dp * EB;  // states, per chunk
  const __amdgpu_buffer_rsrc_t sh = buf_of(as<T>(p.states) + ((size_t)first * p.heads + h) * p.lds * p.dp, count * sstep);
  const __amdgpu_buffer_rsrc_t sl = buf_of(as<T>(p.states) + p.nstates + ((size_t)first * p.heads + h) * p.lds * p.dp, count * sstep);
  // 16-byte pieces of the tile's columns, 64 keys each: whole lines
  constexpr int PIECES = kChunk / KV, SP = 16 * NE * PIECES / 256;  // per column, per thread
  uint32_t soff[SP];
#pragma unroll
  for (int k = 0; k < SP; ++k) {
    const int col = (tid + 256 * k) / PIECES, piece = (tid + 256 * k) % PIECES;
    soff[k] = e0 + col < p.lds ? ((uint32_t)(e0 + col) * p.dp + ((int)blockIdx.x / ne) * 64 + piece * KV) * EB : kPastEnd;
  }

  struct Request {
    Quad4<T, VEC> vin[TP];
    Split<T> kh[CHANNEL ? KS : 1];
    Quad4<T, VEC> kin[CHANNEL ? 1 : 4];
    floatx4 end;
    float w_c, w_end, w_dt;
  };
  constexpr int AHEAD = !VEC || NE > 2 ? 2 : 4;  // (at most 63 loads and stores can be told apart)
  Request rq[AHEAD];
  // Requests past the last chunk re-read it: every load is unconditional, so the waits count exactly
  // the loads in front of the ones they are for.
  auto request = [&](Request& q_, int i_) {
    const int i = min(i_, count - 1);
    const uint32_t row = i * kChunk, last = min(row + kChunk, (uint32_t)total) - 1;
#pragma unroll
    for (int k = 0; k < TP; ++k) q_.vin[k].request(rv, voff[k], row * p.ldv * EB, p.vdim - e0 - q);
    if constexpr (CHANNEL) {
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        q_.kh[k].hi = buf_load16(rh, hoff + k * 4 * KV * EB, i * cstep);
        if constexpr (sizeof(T) == 2) q_.kh[k].lo = buf_load16(rl, hoff + k * 4 * KV * EB, i * cstep);
      }
      q_.end = __builtin_bit_cast(floatx4, buf_load16(rc, eoff, last * p.ldcum * 4));
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) q_.kin[k].request(rk, koff[k], row * p.ldk * EB, p.dim - dq);
      q_.w_end = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rc, 0u, last * 4, 0));
      q_.w_c = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rc, woff, row * 4, 0));
      q_.w_dt = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, woff, row * 4, 0));  // zero past the end
    }
  };
  auto chunk = [&](Request& q_, int i) {
    const int b = i & 1;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      struct alignas(TP * sizeof(T)) Run {
        T t[TP];
      } out;
#pragma unroll
      for (int k = 0; k < TP; ++k) out.t[k] = q_.vin[k].at(e);
      *reinterpret_cast<Run*>(&vt[b][(q + e) * VS + t0]) = out;
    }
    if constexpr (!CHANNEL) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        struct alignas(4 * sizeof(T)) Run {
          T t[4];
        } out;
#pragma unroll
        for (int k = 0; k < 4; ++k) out.t[k] = q_.kin[k].at(e);
        *reinterpret_cast<Run*>(&kt[b][(kq + e) * VS + kt0]) = out;
      }
      wt[b][lane] = pow2(q_.w_end - q_.w_c) * q_.w_dt;  // (every wave the same)
    }
    float f[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = pow2(CHANNEL ? q_.end[e] : q_.w_end);
#pragma unroll
    for (int j = 0; j < NE; ++j) {
      const float x[4] = {s[j][0], s[j][1], s[j][2], s[j][3]};
      split_store<T>(&sv[b][0][0], (j * 16 + r) * VS + wave * 16 + 4 * g, 16 * NE * VS, x);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[j][e] *= f[e];
    }
    __syncthreads();  // this chunk is complete in its buffer; the other one has been read
#pragma unroll
    for (int k = 0; k < SP; ++k) {
      const int at = (tid + 256 * k) / PIECES * VS + (tid + 256 * k) % PIECES * KV;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(int4v, *reinterpret_cast<const uint4*>(&sv[b][0][at])), sh, soff[k], i * sstep, 0);
      if constexpr (sizeof(T) == 2)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(int4v, *reinterpret_cast<const uint4*>(&sv[b][NT - 1][at])), sl, soff[k],
                                               i * sstep, 0);
    }
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const int t = k * 4 * KV + g * KV;
      Split<T> a;
      if constexpr (CHANNEL) {
        a = q_.kh[k];
      } else {
        float x[KV];
        unpack_vec<T>(*reinterpret_cast<const uint4*>(&kt[b][(wave * 16 + r) * VS + t]), x);
#pragma unroll
        for (int e = 0; e < KV; ++e) x[e] *= wt[b][t + e];
        a.set(x);
      }
#pragma unroll
      for (int j = 0; j < NE; ++j) s[j] = mma<T>(a, *reinterpret_cast<const uint4*>(&vt[b][(j * 16 + r) * VS + t]), s[j]);
    }
  };
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) {
    request(rq[u], u);
    __builtin_amdgcn_sched_barrier(0);  // (in this order: the first wait is for the first of them only)
  }
  int i = 0;
  for (; i + AHEAD <= count; i += AHEAD) {  // (no way out in between: a set's registers stay where they are)
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      chunk(rq[u], i + u);
      request(rq[u], i + u + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int u = 0; u < AHEAD - 1; ++u)
    if (i + u < count) chunk(rq[u], i + u);
#pragma unroll
  for (int j = 0; j < NE; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d = d0 + 4 * g + e, col = e0 + j * 16 + r;
      if (d < p.dim && col < p.lds) st[(size_t)d * p.lds + col] = s[j][e];
    }
}

// 64 value columns of a chunk's outputs
template <typename T, bool CHANNEL, bool VEC>
__global__ __launch_bounds__(256) void recur_out_kernel(const Rec p) {
  constexpr int KV = Elem<T>::kVec, NT = sizeof(T) == 2 ? 2 : 1;
  __shared__ __attribute__((aligned(16))) T vt[64 * kVStride<T>];
  __shared__ __attribute__((aligned(16))) T st[NT][64 * 9 * KV];  // [column][keys], value and remainder
  __shared__ float cl[kChunk], dl[kChunk];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const Chunk ck(p.chunks, blockIdx.x);
  const int h = blockIdx.y, grp = h / (p.heads / p.groups), e0 = (int)blockIdx.z * 64, i0 = wave * 16;
  // the values, scores and step sizes are requested ahead of the product with the state
  const int q4 = (tid & 15) * 4, t0 = (tid >> 4) * 4;
  const __amdgpu_buffer_rsrc_t rv = buf_of(as<T>(p.v) + (size_t)ck.row * p.ldv, (uint32_t)ck.n * p.ldv * (uint32_t)sizeof(T));
  Quad4<T, VEC> values[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    values[i].request(rv, e0 + q4 < p.vdim ? ((uint32_t)(t0 + i) * p.ldv + h * p.vdim + e0 + q4) * (uint32_t)sizeof(T) : kPastEnd, 0,
                      p.vdim - e0 - q4);
  constexpr int SQ = kChunk / 16;  // quads of scores per lane
  const float* A = p.scores + ((size_t)blockIdx.x * p.groups + grp) * kChunk * kChunk + (i0 + r) * kChunk;
  floatx4 sc[SQ];
#pragma unroll
  for (int i = 0; i < SQ; ++i) {
    const int j = (i * 4 / KV) * 4 * KV + g * KV + (i * 4) % KV;
    sc[i] = *reinterpret_cast<const floatx4*>(A + j);  // (those of later keys are not written: any values)
  }
  float c_own = 0.f, dt_own = 0.f;
  if (!CHANNEL) {
    const size_t at = (size_t)h * p.ldcum + ck.row + min(lane, ck.n - 1);
    c_own = p.cum[at];
    dt_own = p.dt[at];
  }
  floatx4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const size_t head = (size_t)blockIdx.x * p.heads + h;
  // ---- from the state ahead of the chunk (nothing is ahead of the sequence's first token); 128 bytes of
  // keys per column at a time through LDS
  if (ck.pos > 0) {
    constexpr int DB = 8 * KV, SS = DB + KV;
    const T* qp = as<T>(p.q) + (size_t)(ck.row + min(i0 + r, ck.n - 1)) * p.ldq + grp * p.dim;
    const size_t qh = (head * kChunk + i0 + r) * p.dp + g * KV;
    const int piece = tid & 7, col = tid >> 3;  // 16-byte pieces of columns col and col + 32
    const T* src[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) src[k] = as<T>(p.states) + (head * p.lds + min(e0 + col + 32 * k, p.lds - 1)) * p.dp + piece * KV;
    Split<T> in[2];
    auto load_state = [&](int s) {
#pragma unroll
      for (int k = 0; k < 2; ++k) in[k] = split_at<T>(src[k], s, p.nstates);
    };
    load_state(0);
    for (int s0 = 0; s0 < p.dim; s0 += DB) {
      __syncthreads();  // (the keys before have been read)
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        *reinterpret_cast<uint4*>(&st[0][(col + 32 * k) * SS + piece * KV]) = in[k].hi;
        if constexpr (sizeof(T) == 2) *reinterpret_cast<uint4*>(&st[NT - 1][(col + 32 * k) * SS + piece * KV]) = in[k].lo;
      }
      Split<T> a[2];
      struct alignas(16) Vec {
        T e[KV];
      } raw[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int su = s0 + u * 4 * KV;
        if constexpr (CHANNEL)
          a[u] = split_at<T>(p.qhat, qh + su, p.nhat);
        else
          load_n<T, KV>(qp + su + g * KV, raw[u].e, VEC, p.dim - su - g * KV);
      }
      load_state(min(s0 + DB, p.dp - DB));
      __syncthreads();
      if (i0 >= ck.n) continue;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int at = (j * 16 + r) * SS + u * 4 * KV + g * KV;
          Split<T> b;
          b.hi = *reinterpret_cast<const uint4*>(&st[0][at]);
          if constexpr (sizeof(T) == 2) b.lo = *reinterpret_cast<const uint4*>(&st[NT - 1][at]);
          if constexpr (CHANNEL)
            acc[j] = mma<T>(a[u], b, acc[j]);
          else
            acc[j] = mma<T>(__builtin_bit_cast(uint4, raw[u]), b, acc[j]);
        }
    }
    if (!CHANNEL) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float f = pow2(__shfl(c_own, i0 + 4 * g + e, 64)) * p.q_scale;
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j][e] *= f;
      }
    }
  }
  // ---- from the chunk's own tokens
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    struct alignas(4 * sizeof(T)) Run {
      T t[4];
    } out;
#pragma unroll
    for (int i = 0; i < 4; ++i) out.t[i] = values[i].at(e);
    *reinterpret_cast<Run*>(vt + (q4 + e) * kVStride<T> + t0) = out;
  }
  if (!CHANNEL && wave == 0) cl[lane] = c_own, dl[lane] = dt_own;
  __syncthreads();
  if (i0 >= ck.n) return;
#pragma unroll
  for (int s = 0; s < kChunk; s += 4 * KV) {
    if (s > i0 + 15) break;
    float f[KV];
#pragma unroll
    for (int e4 = 0; e4 < KV; e4 += 4) {
      const int j = s + g * KV + e4;
      const floatx4 v = sc[(s / (4 * KV)) * (KV / 4) + e4 / 4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int jj = j + e;
        const float w = CHANNEL ? 1.f : pow2(fminf(cl[i0 + r] - cl[jj], 0.f)) * dl[jj];
        f[e4 + e] = jj <= i0 + r && jj < ck.n ? v[e] * w : 0.f;
      }
    }
    Split<T> a;
    a.set(f);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      acc[j] = mma<T>(a, *reinterpret_cast<const uint4*>(vt + (j * 16 + r) * kVStride<T> + s + g * KV), acc[j]);
  }
  const float skip = p.skip ? p.skip[h] : 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int col = e0 + j * 16 + r;
    if (col >= p.vdim) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = i0 + 4 * g + e;
      if (t >= ck.n) continue;
      float y = acc[j][e];
      if (p.skip) y = fmaf(skip, Elem<T>::load(vt[(j * 16 + r) * kVStride<T> + t]), y);
      p.y[(size_t)(ck.row + t) * p.ldy + h * p.vdim + col] = y;
    }
  }
}

// ------------------------------------------------------------------------------ single tokens
// One convolved input: the current one from its row, the others from the ring; `keep`: the current one
// takes its place in the ring (`here` = pos % taps).
template <typename T>
__device__ __forceinline__ float conv_one(const Rec& p, int row, int slot, int pos, int here, int c, bool keep) {
  T* ring = reinterpret_cast<T*>(p.ring) + (size_t)slot * p.taps * p.channels + c;
  const T cur = as<T>(p.raw)[(size_t)row * p.ldraw + c];
  float y = p.conv_b[c];
  for (int b0 = 1; b0 < p.taps; b0 += 4) {  // four requests together
    float w[4], x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int back = b0 + i, bc = min(back, p.taps - 1), at = here - bc;
      x[i] = Elem<T>::load(ring[(size_t)(at < 0 ? at + p.taps : at) * p.channels]);
      w[i] = back < p.taps && pos >= back ? p.conv_w[(size_t)(p.taps - 1 - bc) * p.channels + c] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) y = fmaf(w[i], x[i], y);
  }
  y = fmaf(p.conv_w[(size_t)(p.taps - 1) * p.channels + c], Elem<T>::load(cur), y);
  if (keep) ring[(size_t)here * p.channels] = cur;
  return Elem<T>::load(Elem<T>::make(y * sigmoidf(y)));
}

enum Kind { kSteps = 0, kChannel = 1, kGates = 2 };  // what the decay comes from

template <typename T, int KIND>
__global__ __launch_bounds__(256) void recur_step_kernel(const Rec p, int cols) {
  request_arguments(p);  // (64 heads under 4 rows 8.4 -> 8.1 us, in float32 32 heads under 2 rows 7.9 -> 7.4)
  constexpr bool CHANNEL = KIND == kChannel;
  extern __shared__ __attribute__((aligned(16))) float lds[];  // q, k, decay [dim]; values [64]; partials [4][cols]
  const int tid = threadIdx.x, D = p.dim, h = blockIdx.y, e0 = blockIdx.x * cols;
  const int Dp = (D + 3) / 4 * 4;
  float *qs = lds, *ks = qs + Dp, *as_ = ks + Dp, *vs = as_ + Dp, *red = vs + 64;
  const int row = p.list ? p.list[blockIdx.z] : (int)blockIdx.z;
  const int crow = p.slot[row], pos = p.pos[row], slot = p.map[crow];
  const int hpg = p.heads / p.groups, grp = h / hpg;
  // this thread's part of the state is requested ahead of everything it depends on
  const int lpr = cols / 4, cq = (tid % lpr) * 4, dr = tid / lpr, rpp = 256 / lpr;
  const bool on = e0 + cq < p.lds;
  float* st = p.state + ((size_t)slot * p.heads + h) * D * p.lds + e0 + cq;
  constexpr int kAhead = 8;
  floatx4 s[kAhead];
  auto load_state = [&](int d0) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      s[i] = floatx4{0.f, 0.f, 0.f, 0.f};
      const int d = d0 + i * rpp;
      if (on && pos > 0 && d < D) s[i] = *reinterpret_cast<const floatx4*>(st + (size_t)d * p.lds);
    }
  };
  load_state(dr);
  float vscale = 1.f, skip = 0.f;
  if (KIND == kGates) {
    const float2 g = log_gates(p, row, h);
    const double m = pos > 0 ? *peak_at(p, slot, pos - 1, h) : 0., mt = fmax(g.y + m, (double)g.x);
    const float a = expf((float)(g.y + m - mt));
    vscale = expf((float)(g.x - mt));
    for (int d = tid; d < D; d += 256) {
      as_[d] = a;
      qs[d] = Elem<T>::load(as<T>(p.q)[(size_t)row * p.ldq + grp * D + d]) * p.q_scale;
      ks[d] = Elem<T>::load(as<T>(p.k)[(size_t)row * p.ldk + grp * D + d]);
    }
    if (tid < cols) vs[tid] = e0 + tid < p.vdim ? Elem<T>::load(as<T>(p.v)[(size_t)row * p.ldv + h * p.vdim + e0 + tid]) : 0.f;
    if (blockIdx.x == 0 && tid == 0) {
      *peak_at(p, slot, pos, h) = mt;  // (the other workgroups read the other entry)
      p.peaks[(size_t)row * p.ldpeaks + h] = (float)mt;
    }
  } else if (CHANNEL) {
    const int C = p.heads * D;
    const float* low = p.low + (size_t)row * p.ldlow;
    for (int d = tid; d < D; d += 256) {
      const int c = h * D + d;
      float z = p.decay_b[c];
      for (int j0 = 0; j0 < p.rank; j0 += 16) {  // (16 requests together)
        float w[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) w[j] = p.decay_w[(size_t)min(j0 + j, p.rank - 1) * C + c];
#pragma unroll
        for (int j = 0; j < 16; ++j) z = fmaf(w[j], j0 + j < p.rank ? low[j0 + j] : 0.f, z);
      }
      as_[d] = expf(-softplus(-z) * p.inv_tau);
      qs[d] = Elem<T>::load(as<T>(p.q)[(size_t)row * p.ldq + grp * D + d]) * p.q_scale;
      ks[d] = Elem<T>::load(as<T>(p.k)[(size_t)row * p.ldk + grp * D + d]);
    }
    if (tid < cols) vs[tid] = e0 + tid < p.vdim ? Elem<T>::load(as<T>(p.v)[(size_t)row * p.ldv + h * p.vdim + e0 + tid]) : 0.f;
  } else {
    const bool keep = blockIdx.x == 0 && h == grp * hpg;  // a group's keys and queries: one workgroup's to keep
    const int here = pos % p.taps;
    for (int i = tid; i < 2 * D + cols; i += 256) {  // keys, queries, values
      if (i < 2 * D) {
        const bool key = i < D;
        const int d = key ? i : i - D;
        const float f = conv_one<T>(p, row, slot, pos, here, (key ? p.k_channel : p.q_channel) + grp * D + d, keep);
        if (key)
          ks[d] = f;
        else
          qs[d] = f * p.q_scale;
      } else {
        const int e = i - 2 * D;
        vs[e] = e0 + e < p.vdim ? conv_one<T>(p, row, slot, pos, here, p.v_channel + h * p.vdim + e0 + e, true) : 0.f;
      }
    }
    vscale = softplus(p.dt_raw[(size_t)row * p.lddt + h] + p.dt_bias[h]);
    const float a = expf(-p.decay_rate[h] * vscale);
    for (int d = tid; d < D; d += 256) as_[d] = a;
    if (p.skip) skip = p.skip[h];
  }
  __syncthreads();
  floatx4 v, o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = vs[cq + e] * vscale;
  for (int d0 = dr; d0 < D; d0 += kAhead * rpp) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int d = d0 + i * rpp;
      if (d >= D) break;
      const float a = as_[d], k = ks[d], q = qs[d];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[i][e] = fmaf(a, s[i][e], k * v[e]);
        o[e] = fmaf(q, s[i][e], o[e]);
      }
      if (on) *reinterpret_cast<floatx4*>(st + (size_t)d * p.lds) = s[i];
    }
    if (d0 + kAhead * rpp < D) load_state(d0 + kAhead * rpp);
  }
  // over the wave's rows (lanes with the same columns), then over the waves
  auto rows = [&](auto step) __attribute__((always_inline)) {
    constexpr int S = decltype(step)::value;
    if (lpr > S) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float v = o[e];
      o[e] = add_across<S>(v);
    }
  };
  rows(std::integral_constant<int, 1>{});
  rows(std::integral_constant<int, 2>{});
  rows(std::integral_constant<int, 4>{});
  rows(std::integral_constant<int, 8>{});
  rows(std::integral_constant<int, 16>{});
  rows(std::integral_constant<int, 32>{});
  if ((tid & 63) < lpr) *reinterpret_cast<floatx4*>(red + (tid >> 6) * cols + cq) = o;
  __syncthreads();
  if (tid < cols && e0 + tid < p.vdim) {
    float y = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) y += red[i * cols + tid];
    p.y[(size_t)row * p.ldy + h * p.vdim + e0 + tid] = fmaf(skip, vs[tid], y);
  }
}

// ------------------------------------------------------------------------------ gated norm
// out = norm of equal parts of y, with the gate silu(z) or sigmoid(z) ahead of the norm or behind it; the
// gain repeats with `period`.  With peaks a part is first divided by max(|its entry `den`|, exp(-peak)) + 1e-6.
// (DIVIDE: with peaks, or with a sigmoid.)  TEAM threads per part, each with PASSES runs of VEC columns.
template <typename T, int TEAM, int BLOCK, int VEC, int PASSES, bool DIVIDE>
__global__ __launch_bounds__(BLOCK) void gated_norm_kernel(const exo_gated_norm p, const int32_t* __restrict__ rows) {
  __shared__ float part[BLOCK / 64];
  const int tid = threadIdx.x, team = tid / TEAM, l = tid % TEAM;
  const int gi = blockIdx.x * (BLOCK / TEAM) + team;
  const int row = rows ? rows[blockIdx.y] : (int)blockIdx.y;
  const int size = p.width / p.groups;
  const size_t at = (size_t)min(gi, p.groups - 1) * size;
  const float* y = p.y + (size_t)row * p.ldy + (DIVIDE ? (size_t)min(gi, p.groups - 1) * p.ldpart : at);
  float scale = 1.f;
  if (DIVIDE && p.peaks) {
    const float peak = p.peaks[(size_t)row * p.ldpeaks + min(gi, p.groups - 1)];
    scale = 1.f / (fmaxf(fabsf(y[p.den]), expf(-peak)) + 1e-6f);
  }
  const T* z = as<T>(p.gate) + (size_t)row * p.ldg + at;
  // Inputs, gates and gains are requested together and without a branch (past the part: its first columns, as zeros): the gains behind the sum
  // were a memory latency of their own.  Gains in L2, bf16: 4 rows of 4 parts of 512 3.1 -> 2.8 us, of 64 of 64 2.8 -> 2.7, one of 4096 3.5 | 3.6; decode
  // passes of six mixed layers of 2048, whose gains come from memory, 1 % (two such norms a layer).  Parts of 1024 in one pass
  // instead of a half-empty second: 1004 rows of 8 19.9 -> 15.0.
  constexpr bool AHEAD = PASSES <= 2;
  const int g0 = (int)((uint32_t)at % (uint32_t)p.period);
  auto gain_at = [&](int c) {
    const uint32_t gc = g0 + c;
    return p.gain + (gc >= (uint32_t)p.period ? gc % (uint32_t)p.period : gc);  // (VEC divides the period)
  };
  float v[PASSES][VEC], gate[PASSES][VEC], gain[PASSES][VEC], ss = 0.f;
  T zz[PASSES][VEC];
#pragma unroll
  for (int i = 0; i < PASSES; ++i) {
    const int c = (l + i * TEAM) * VEC, from = c < size ? c : 0;
    if constexpr (VEC == 4) {
      const floatx4 f = *reinterpret_cast<const floatx4*>(y + from);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i][e] = f[e];
      load_n<T, 4>(z + from, zz[i], true, 4);
    } else {
      v[i][0] = y[from];
      zz[i][0] = z[from];
    }
    if (AHEAD) {
      const float* const w = gain_at(from);
#pragma unroll
      for (int e = 0; e < VEC; ++e) gain[i][e] = w[e];
    }
  }
#pragma unroll
  for (int i = 0; i < PASSES; ++i) {
    const int c = (l + i * TEAM) * VEC;
#pragma unroll
    for (int e = 0; e < VEC; ++e) v[i][e] = c >= size ? 0.f : DIVIDE ? v[i][e] * scale : v[i][e];
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float f = c < size ? Elem<T>::load(zz[i][e]) : 0.f;
      gate[i][e] = (DIVIDE && p.sigmoid ? 1.f : f) * sigmoidf(f);
      if (p.gate_first) v[i][e] *= gate[i][e];
      ss += v[i][e] * v[i][e];
    }
  }
  ss = wave_total(ss);
  if (TEAM > 64) {
    if ((tid & 63) == 0) part[tid >> 6] = ss;
    __syncthreads();
    ss = 0.f;
#pragma unroll
    for (int w = 0; w < TEAM / 64; ++w) ss += part[w];
  }
  if (gi >= p.groups) return;
  const float inv = 1.f / sqrtf(ss / size + p.eps);
  T* out = reinterpret_cast<T*>(p.out) + (size_t)row * p.ldo + at;
#pragma unroll
  for (int i = 0; i < PASSES; ++i) {
    const int c = (l + i * TEAM) * VEC;
    if (c >= size) break;
    const float* const gw = AHEAD ? nullptr : gain_at(c);
    T o[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float w = v[i][e] * inv * (AHEAD ? gain[i][e] : gw[e]);
      o[e] = Elem<T>::make(p.gate_first ? w : w * gate[i][e]);
    }
    if constexpr (VEC == 4 && sizeof(T) == 2)
      *reinterpret_cast<uint2*>(out + c) = uint2{(uint32_t)o[0] | (uint32_t)o[1] << 16, (uint32_t)o[2] | (uint32_t)o[3] << 16};
    else
#pragma unroll
      for (int e = 0; e < VEC; ++e) out[c + e] = o[e];
  }
}

template <typename T, int VEC, bool DIVIDE>
int launch_gated_norm(const exo_gated_norm& a, const int32_t* rows, int n, hipStream_t st) {
  const int size = a.width / a.groups, per = exo_ceil_div(size, VEC);  // runs of VEC columns per part
  const dim3 small(exo_ceil_div(a.groups, 4), n), wide(a.groups, n);
  if (per <= 64)
    gated_norm_kernel<T, 64, 256, VEC, 1, DIVIDE><<<small, 256, 0, st>>>(a, rows);
  else if (per <= 128)
    gated_norm_kernel<T, 64, 256, VEC, 2, DIVIDE><<<small, 256, 0, st>>>(a, rows);
  else if (per <= 256)
    gated_norm_kernel<T, 256, 256, VEC, 1, DIVIDE><<<wide, 256, 0, st>>>(a, rows);
  else if (per <= 512)
    gated_norm_kernel<T, 256, 256, VEC, 2, DIVIDE><<<wide, 256, 0, st>>>(a, rows);
  else if (per <= 1024)
    gated_norm_kernel<T, 1024, 1024, VEC, 1, DIVIDE><<<wide, 1024, 0, st>>>(a, rows);
  else if (per <= 2048)
    gated_norm_kernel<T, 1024, 1024, VEC, 2, DIVIDE><<<wide, 1024, 0, st>>>(a, rows);
  else if (per <= 8192)
    gated_norm_kernel<T, 1024, 1024, VEC, 8, DIVIDE><<<wide, 1024, 0, st>>>(a, rows);
  else {
    exo_set_error("exo_gated_norm_rows: parts of %d columns are too long", size);
    return EXO_ERR_ARG;
  }
  return EXO_OK;
}

int check(const exo_recurrence* a, const char* what) {
  EXO_REQUIRE(a && (a->dtype == 0 || a->dtype == 1), "%s: bad dtype", what);
  EXO_REQUIRE(a->heads > 0 && a->groups > 0 && a->heads % a->groups == 0 && a->dim > 0 && a->dim <= 1024 && a->vdim > 0 &&
                  a->lds >= a->vdim && a->lds % 4 == 0,
              "%s: bad sizes (heads=%d groups=%d dim=%d vdim=%d stride=%d)", what, a->heads, a->groups, a->dim, a->vdim, a->lds);
  EXO_REQUIRE(a->heads <= 65534, "%s: %d heads", what, a->heads);
  EXO_REQUIRE(a->state && a->map && a->y && a->ldy >= a->heads * a->vdim && ((uintptr_t)a->state & 15) == 0, "%s: bad state or output", what);
  if (a->gate_i) {
    EXO_REQUIRE(!a->per_channel && a->groups == a->heads && a->taps == 0 && !a->skip,
                "%s: exponential gates go with queries and keys per head, no convolution", what);
    EXO_REQUIRE(a->gate_f && a->peak && a->peaks && a->ldgate >= a->heads && a->ldpeaks >= a->heads && a->gate_cap > 0.f,
                "%s: incomplete gates", what);
  } else if (a->per_channel) {
    EXO_REQUIRE(a->groups == a->heads && a->taps == 0 && !a->skip, "%s: a decay per channel goes with queries and keys per head, no convolution", what);
    EXO_REQUIRE(a->low && a->decay_w && a->decay_b && a->rank > 0 && a->ldlow >= a->rank, "%s: incomplete decay", what);
  } else {
    EXO_REQUIRE(a->dt_raw && a->dt_bias && a->decay_rate && a->lddt >= a->heads, "%s: incomplete step sizes", what);
    EXO_REQUIRE(a->taps > 0 && a->taps <= 16 && a->raw && a->ring && a->conv_w && a->conv_b && a->ldraw >= a->channels,
                "%s: incomplete convolution (%d taps, at most 16)", what, a->taps);
    EXO_REQUIRE(a->v_channel >= 0 && a->v_channel + a->heads * a->vdim <= a->channels && a->k_channel >= 0 &&
                    a->k_channel + a->groups * a->dim <= a->channels && a->q_channel >= 0 &&
                    a->q_channel + a->groups * a->dim <= a->channels,
                "%s: values, keys and queries do not lie inside the %d channels", what, a->channels);
  }
  return EXO_OK;
}

template <typename T>
bool vec_ok(const void* p, int ld, int part, int n) {
  return part % n == 0 && ld % n == 0 && (uintptr_t)p % (n * sizeof(T)) == 0;
}

int64_t chunk_bytes(const exo_recurrence* a, int n_chunks, Rec* out, char* ws) {
  const int dp = exo_ceil_div(a->dim, 64) * 64, terms = a->dtype == 0 ? 2 : 1, esz = a->dtype == 0 ? 2 : 4;
  const int64_t scores = (int64_t)n_chunks * a->groups * kChunk * kChunk * 4;
  const int64_t nstates = (int64_t)n_chunks * a->heads * a->lds * dp, nhat = a->per_channel ? (int64_t)n_chunks * a->heads * kChunk * dp : 0;
  const int64_t states = nstates * terms * esz, hat = nhat * terms * esz;
  if (out) {
    out->scores = reinterpret_cast<float*>(ws);
    out->states = ws + scores;
    out->qhat = ws + scores + states;
    out->khat = ws + scores + states + hat;
    out->nstates = nstates;
    out->nhat = nhat;
    out->dp = dp;
  }
  return scores + states + 2 * hat;
}

template <typename T, bool CHANNEL, int NE, bool VEC>
int launch_carry(const Rec& p, hipStream_t st) {
  constexpr int lds = carry_lds<T, CHANNEL, NE>();
  const auto fn = recur_carry_kernel<T, CHANNEL, NE, VEC>;
  static bool done = false;
  if (!done && lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      exo_set_error("exo_recur_chunks: cannot raise the dynamic LDS limit: %s", hipGetErrorString(e));
      return EXO_ERR_HIP;
    }
  }
  done = true;
  fn<<<dim3(exo_ceil_div(p.lds, 16 * NE) * (p.dp / 64), p.heads + (p.taps > 0 ? 1 : 0), p.n_seqs), 256, lds, st>>>(p);
  return EXO_OK;
}

template <typename T, bool CHANNEL>
int launch_chunks(Rec p, hipStream_t st) {
  constexpr int KV = Elem<T>::kVec;
  p.qk_vec = vec_ok<T>(p.q, p.ldq, p.dim, KV) && vec_ok<T>(p.k, p.ldk, p.dim, KV);
  p.v_vec = vec_ok<T>(p.v, p.ldv, p.vdim, 4);
  if constexpr (CHANNEL) {
    recur_prep_channel_kernel<<<dim3(p.n_chunks, exo_ceil_div(p.heads * p.dim, 64)), 256, 0, st>>>(p);
    recur_scores_channel_kernel<T><<<dim3(p.n_chunks, p.heads, 4), 256, 0, st>>>(p);
  } else if (p.gate_i) {
    recur_gates_kernel<<<dim3(p.heads, p.n_seqs), 64 * kGateWaves, 0, st>>>(p);
    recur_scores_head_kernel<T><<<dim3(p.n_chunks, p.groups), 256, 0, st>>>(p);
  } else {
    const int parts = kChunk / kConvTokens;
    const dim3 grid(p.n_chunks * parts, exo_ceil_div(p.channels, 256) + exo_ceil_div(p.heads, 4 * parts));
    if (p.taps <= 4)
      recur_conv_kernel<T, 4><<<grid, 256, 0, st>>>(p);
    else if (p.taps <= 8)
      recur_conv_kernel<T, 8><<<grid, 256, 0, st>>>(p);
    else
      recur_conv_kernel<T, 16><<<grid, 256, 0, st>>>(p);
    recur_scores_head_kernel<T><<<dim3(p.n_chunks, p.groups), 256, 0, st>>>(p);
  }
  const dim3 out_grid(p.n_chunks, p.heads, exo_ceil_div(p.vdim, 64));
  // wide tiles of the state (a key tile is read by fewer workgroups) once they leave a workgroup per CU
  const bool wide = (int64_t)exo_ceil_div(p.lds, 64) * (p.dp / 64) * p.heads * p.n_seqs >= 256;
  int rc;
  if (p.v_vec && p.qk_vec) {
    rc = wide ? launch_carry<T, CHANNEL, 4, true>(p, st) : launch_carry<T, CHANNEL, 2, true>(p, st);
    if (rc) return rc;
    recur_out_kernel<T, CHANNEL, true><<<out_grid, 256, 0, st>>>(p);
  } else {
    rc = launch_carry<T, CHANNEL, 2, false>(p, st);
    if (rc) return rc;
    recur_out_kernel<T, CHANNEL, false><<<out_grid, 256, 0, st>>>(p);
  }
  return EXO_OK;
}

template <typename T, int KIND>
void launch_step_kind(const Rec& p, hipStream_t st) {
  int cols = 64;
  while (cols > 16 && (int64_t)p.n * p.heads * exo_ceil_div(p.lds, cols) < 256) cols /= 2;
  const int lds = (3 * ((p.dim + 3) / 4 * 4) + 64 + 4 * cols) * 4;
  recur_step_kernel<T, KIND><<<dim3(exo_ceil_div(p.lds, cols), p.heads, p.n), 256, lds, st>>>(p, cols);
}
template <typename T>
void launch_step(const Rec& p, hipStream_t st) {
  p.per_channel ? launch_step_kind<T, kChannel>(p, st) : p.gate_i ? launch_step_kind<T, kGates>(p, st) : launch_step_kind<T, kSteps>(p, st);
}

}  // namespace

extern "C" int exo_recur_chunk(void) { return kChunk; }
extern "C" int64_t exo_recur_workspace(const exo_recurrence* a) {
  return a && a->n_chunks > 0 && a->dim > 0 ? chunk_bytes(a, a->n_chunks, nullptr, nullptr) : 0;
}

extern "C" int exo_recur_chunks(const exo_recurrence* a, void* workspace, int64_t workspace_bytes, exo_stream_t stream) {
  const int rc = check(a, "exo_recur_chunks");
  if (rc) return rc;
  EXO_REQUIRE(a->n_chunks > 0 && a->n_chunks <= 65535 && a->n_seqs > 0 && a->n_seqs <= 65535 && a->chunks && a->seqs,
              "exo_recur_chunks: bad lists (%d chunks, %d portions)", a->n_chunks, a->n_seqs);
  EXO_REQUIRE(a->q && a->k && a->v && a->cum && a->ldcum >= (a->per_channel ? a->heads * a->dim : 1) &&
                  a->ldq >= a->groups * a->dim && a->ldk >= a->groups * a->dim && a->ldv >= a->heads * a->vdim,
              "exo_recur_chunks: bad inputs");
  EXO_REQUIRE(a->per_channel || (a->dt && (a->gate_i || (a->act && a->ldact >= a->channels))), "exo_recur_chunks: no place for the convolved inputs");
  EXO_REQUIRE((int64_t)a->n_chunks * a->heads * (a->lds > kChunk ? a->lds : kChunk) * exo_ceil_div(a->dim, 64) * 256 < (1ll << 31) &&
                  (int64_t)a->n_chunks * kChunk * (a->per_channel && a->ldcum > a->ldv ? a->ldcum : a->ldv) * 4 < (1ll << 31) &&
                  (int64_t)a->n_chunks * kChunk * a->ldk * 4 < (1ll << 31),
              "exo_recur_chunks: %d chunks exceed 31-bit byte offsets", a->n_chunks);
  EXO_REQUIRE(workspace && (uintptr_t)workspace % 16 == 0 && workspace_bytes >= exo_recur_workspace(a), "exo_recur_chunks: workspace too small");
  Rec p{*a};
  chunk_bytes(a, a->n_chunks, &p, reinterpret_cast<char*>(workspace));
  const hipStream_t st = (hipStream_t)stream;
  int rc2;
  if (a->dtype == 0)
    rc2 = a->per_channel ? launch_chunks<bf16_t, true>(p, st) : launch_chunks<bf16_t, false>(p, st);
  else
    rc2 = a->per_channel ? launch_chunks<float, true>(p, st) : launch_chunks<float, false>(p, st);
  if (rc2) return rc2;
  EXO_CHECK_LAUNCH("exo_recur_chunks");
  return EXO_OK;
}

extern "C" int exo_recur_step(const exo_recurrence* a, exo_stream_t stream) {
  const int rc = check(a, "exo_recur_step");
  if (rc) return rc;
  EXO_REQUIRE(a->n > 0 && a->n <= 65535 && a->slot && a->pos, "exo_recur_step: bad rows (n=%d)", a->n);
  EXO_REQUIRE(!(a->per_channel || a->gate_i) || (a->q && a->k && a->v && a->ldq >= a->heads * a->dim && a->ldk >= a->heads * a->dim && a->ldv >= a->heads * a->vdim),
              "exo_recur_step: bad inputs");
  const Rec p{*a};
  if (a->dtype == 0)
    launch_step<bf16_t>(p, (hipStream_t)stream);
  else
    launch_step<float>(p, (hipStream_t)stream);
  EXO_CHECK_LAUNCH("exo_recur_step");
  return EXO_OK;
}

extern "C" int exo_gated_norm_rows(const exo_gated_norm* a, const int32_t* rows, int n, exo_stream_t stream) {
  EXO_REQUIRE(a && (a->dtype == 0 || a->dtype == 1) && a->y && a->gate && a->gain && a->out && n >= 0 && n <= 65535,
              "exo_gated_norm_rows: bad argument");
  EXO_REQUIRE(a->width > 0 && a->groups > 0 && a->width % a->groups == 0 && a->period > 0 && a->width % a->period == 0 &&
                  a->ldpart >= a->width / a->groups && a->ldy >= a->groups * a->ldpart && a->ldg >= a->width && a->ldo >= a->width,
              "exo_gated_norm_rows: bad sizes (width=%d groups=%d period=%d)", a->width, a->groups, a->period);
  EXO_REQUIRE(!a->peaks || (a->ldpeaks >= a->groups && a->den >= 0 && a->den < a->ldpart), "exo_gated_norm_rows: bad divisor (entry %d)", a->den);
  if (n == 0) return EXO_OK;
  const int esz = a->dtype == 0 ? 2 : 4;
  const bool vec = (a->width / a->groups) % 4 == 0 && a->period % 4 == 0 && a->ldy % 4 == 0 && a->ldpart % 4 == 0 && a->ldg % 4 == 0 && a->ldo % 4 == 0 &&
                   (uintptr_t)a->y % 16 == 0 && (uintptr_t)a->gate % (4 * esz) == 0 && (uintptr_t)a->out % (4 * esz) == 0;
  const hipStream_t st = (hipStream_t)stream;
  const auto launch = [&](auto divide) {
    constexpr bool DIVIDE = decltype(divide)::value;
    if (a->dtype == 0) return vec ? launch_gated_norm<bf16_t, 4, DIVIDE>(*a, rows, n, st) : launch_gated_norm<bf16_t, 1, DIVIDE>(*a, rows, n, st);
    return vec ? launch_gated_norm<float, 4, DIVIDE>(*a, rows, n, st) : launch_gated_norm<float, 1, DIVIDE>(*a, rows, n, st);
  };
  const int rc = a->peaks || a->sigmoid || a->ldpart != a->width / a->groups ? launch(std::true_type{}) : launch(std::false_type{});
  if (rc) return rc;
  EXO_CHECK_LAUNCH("exo_gated_norm_rows");
  return EXO_OK;
}
