// Small operators of a layer-list decoder with a float32 residual stream: embedding rows,
// normalisation of a sublayer's OUTPUT before it is added and of the sum as the next one's input, routing with a choice correction and
// identity experts, and the expert products of a decode step.  Element type bf16 or float
// (dense.h); every norm, router and sum here is float32.
#include "../../include/exo_mi355x.h"
#include "dense.h"
#include "route.h"

namespace {

constexpr int kRowThreads = 256;

// sum over a workgroup of TH threads, in every thread.  tmp: 2 x TH / 64 floats; a call leaves its own half alone until the
// one after the next, so that one barrier is enough (at most 32 waves' worth of sums through the crossbar, two barriers and
// sixteen dependent additions before: post_norm_add of 4 rows of 2048 columns 3.5 -> 3.1 us, of two branches 4.9 -> 3.9)
template <int TH = kRowThreads>
__device__ __forceinline__ float block_sum(float v, float* tmp, int& phase) {
  v = wave_total(v);
  float* const mine = tmp + (phase ^= 1) * (TH / 64);
  if ((threadIdx.x & 63) == 0) mine[threadIdx.x >> 6] = v;
  __syncthreads();
  return total_of<TH / 64>(mine);
}

// ------------------------------------------------------------------------------ embedding
template <typename T>
__global__ void embed_rows_kernel(const int32_t* __restrict__ ids, const T* __restrict__ table, float* __restrict__ x,
                                  T* __restrict__ xb, int V, int H, int ldt, int ldx, float scale) {
  const int row = blockIdx.x;
  const int id = min(max(ids[row], 0), V - 1);
  for (int c = threadIdx.x; c < H; c += blockDim.x) {
    const float v = Elem<T>::load(table[(size_t)id * ldt + c]) * scale;
    x[(size_t)row * H + c] = v;
    xb[(size_t)row * ldx + c] = Elem<T>::make(v);
  }
}

// ------------------------------------------------------------------------------ norms
// y = x / rms(x) * gain (center: the mean is taken off x first), rows given by an index list (null: row i)
template <typename T, int TH>
__global__ __launch_bounds__(TH) void norm_rows_kernel(const float* __restrict__ x, const int32_t* __restrict__ rows,
                                                       const float* __restrict__ gain, T* __restrict__ y, int H, int ldx,
                                                       int ldy, float eps, int center) {
  __shared__ float tmp[2 * (TH / 64)];
  int phase = 0;
  const float* xr = x + (size_t)(rows ? rows[blockIdx.x] : (int)blockIdx.x) * ldx;
  float mean = 0.f, ss = 0.f;
  if (center) {
    for (int c = threadIdx.x; c < H; c += TH) mean += xr[c];
    mean = block_sum<TH>(mean, tmp, phase) / H;
  }
  for (int c = threadIdx.x; c < H; c += TH) ss += (xr[c] - mean) * (xr[c] - mean);
  const float inv = 1.f / sqrtf(block_sum<TH>(ss, tmp, phase) / H + eps);
  for (int c = threadIdx.x; c < H; c += TH) y[(size_t)blockIdx.x * ldy + c] = Elem<T>::make((xr[c] - mean) * inv * gain[c]);
}

struct MoeSum {        // the feed-forward's output as a sum over a token's experts
  const void* y;       // T [R][top][ldy] expert outputs (null: `branch` holds the sum already)
  const int32_t* idx;  // [R][top]
  const float* wt;     // [R][top]
  const void* shared;  // T [R][lds] output of the shared expert, or null
  const float* logits; // router logits; column E + identity is the shared expert's gate
  int top, experts, ldy, lds, ldl, gate_col;  // gate_col < 0: the shared expert as it is
};

// x += mult * gain * v / rms(v), v = the branch row, half the sum of two branches normed each with a
// gain of its own, or the weighted sum over the experts (without `gain`: x += mult * v); or (sum) x = gain * norm(keep * x + v); xb = x,
// or x / rms(x) * pre.
// Four columns per thread and pass (VEC: rows of four columns are aligned), v in registers.
constexpr int kCols = 4;  // at most 16 passes: H <= 16384

template <typename T>
__device__ __forceinline__ void load_cols(const T* p, float (&f)[kCols], bool vec, int left) {
  if (vec) {
    if (sizeof(T) == 2) {
      const uint2 v = *reinterpret_cast<const uint2*>(p);
      f[0] = bf_lo(v.x), f[1] = bf_hi(v.x), f[2] = bf_lo(v.y), f[3] = bf_hi(v.y);
    } else {
      const floatx4 v = *reinterpret_cast<const floatx4*>(p);
#pragma unroll
      for (int i = 0; i < kCols; ++i) f[i] = v[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < kCols; ++i) f[i] = i < left ? Elem<T>::load(p[i]) : 0.f;
  }
}

template <typename T, int TH, int PASSES>
__global__ __launch_bounds__(TH) void post_norm_add_kernel(const exo_post_norm q, const MoeSum m,
                                                                    float* __restrict__ x, T* __restrict__ xb, int ldx) {
  __shared__ float tmp[2 * (TH / 64)];
  int phase = 0;
  const int row = blockIdx.x, H = q.H;
  float* xr = x + (size_t)row * H;
  const bool vec = H % kCols == 0 && (m.y ? m.ldy % kCols == 0 && m.lds % kCols == 0 : q.ldb % kCols == 0);
  const bool gvec = H % kCols == 0;
  float v[PASSES][kCols], xv[PASSES][kCols];
  // The gains with the inputs where a row's chain counts and it pays: requested between one sum and the next
  // they are a memory latency each (4 rows, one branch / two: 1024 columns 3.35 -> 3.25 / 4.5 -> 4.2 us, 5120 4.4 ->
  // 4.2 / 6.4 -> 6.4), but 2048 to 4096 columns in one pass of 1024 threads lose or are level (2048 3.57 -> 3.66 / 5.15).
  constexpr bool AHEAD = TH == 256 ? PASSES == 1 : PASSES == 2;
  float ga[PASSES][kCols], gb[PASSES][kCols], gn[PASSES][kCols], gp[PASSES][kCols];
  auto load_gains = [&](int i, int c, int left, bool branches, bool sum, bool pre) {
    if (q.branch2 && branches) load_cols<float>(q.gain_a + c, ga[i], gvec, left), load_cols<float>(q.gain_b + c, gb[i], gvec, left);
    if (q.gain && sum) load_cols<float>(q.gain + c, gn[i], gvec, left);
    if (q.pre && pre) load_cols<float>(q.pre + c, gp[i], gvec, left);
  };
  float pass = 0.f, sg = 0.f;  // weight of the input itself; gate of the shared expert
  const T *y = nullptr, *sh = nullptr;
  if (m.y) {
    y = reinterpret_cast<const T*>(m.y) + (size_t)row * m.top * m.ldy;
    if (m.shared) {
      sh = reinterpret_cast<const T*>(m.shared) + (size_t)row * m.lds;
      sg = m.gate_col < 0 ? 1.f : 1.f / (1.f + expf(-m.logits[(size_t)row * m.ldl + m.gate_col]));
    }
    for (int j = 0; j < m.top; ++j)
      if (m.idx[row * m.top + j] >= m.experts) pass += m.wt[row * m.top + j];
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < PASSES; ++i) {
    const int c = (threadIdx.x + i * TH) * kCols, left = H - c;
    if (left <= 0) break;
    load_cols<float>(xr + c, xv[i], vec, left);
    if (AHEAD) load_gains(i, c, left, true, true, true);
    if (m.y) {
#pragma unroll
      for (int e = 0; e < kCols; ++e) v[i][e] = pass * xv[i][e];
      for (int j = 0; j < m.top; ++j) {
        if (m.idx[row * m.top + j] >= m.experts) continue;
        const float w = m.wt[row * m.top + j];
        float f[kCols];
        load_cols<T>(y + (size_t)j * m.ldy + c, f, vec, left);
#pragma unroll
        for (int e = 0; e < kCols; ++e) v[i][e] = fmaf(w, f[e], v[i][e]);
      }
      if (sh) {
        float f[kCols];
        load_cols<T>(sh + c, f, vec, left);
#pragma unroll
        for (int e = 0; e < kCols; ++e) v[i][e] = fmaf(sg, f[e], v[i][e]);
      }
    } else {
      load_cols<float>(q.branch + (size_t)row * q.ldb + c, v[i], vec, left);
    }
#pragma unroll
    for (int e = 0; e < kCols; ++e) ss += e < left ? v[i][e] * v[i][e] : 0.f;
  }
  if (q.branch2) {
    float u[PASSES][kCols], su = 0.f;
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      const int c = (threadIdx.x + i * TH) * kCols, left = H - c;
      if (left <= 0) break;
      load_cols<float>(q.branch2 + (size_t)row * q.ldb + c, u[i], vec, left);
#pragma unroll
      for (int e = 0; e < kCols; ++e) su += e < left ? u[i][e] * u[i][e] : 0.f;
    }
    const float ia = 0.5f / sqrtf(block_sum<TH>(ss, tmp, phase) / H + q.eps), ib = 0.5f / sqrtf(block_sum<TH>(su, tmp, phase) / H + q.eps);
    ss = 0.f;
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      const int c = (threadIdx.x + i * TH) * kCols, left = H - c;
      if (left <= 0) break;
      if (!AHEAD) load_gains(i, c, left, true, false, false);
#pragma unroll
      for (int e = 0; e < kCols; ++e) {
        v[i][e] = v[i][e] * ia * ga[i][e] + u[i][e] * ib * gb[i][e];
        ss += e < left ? v[i][e] * v[i][e] : 0.f;
      }
    }
  }
  if (q.sum) {  // the sum itself is normed
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      const int c = (threadIdx.x + i * TH) * kCols, left = H - c;
      if (left <= 0) break;
#pragma unroll
      for (int e = 0; e < kCols; ++e) {
        v[i][e] = fmaf(q.keep, xv[i][e], v[i][e]);
        xv[i][e] = 0.f;
        s += e < left ? v[i][e] : 0.f;
      }
    }
    const float mean = q.center ? block_sum<TH>(s, tmp, phase) / H : 0.f;
    ss = 0.f;
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      const int c = (threadIdx.x + i * TH) * kCols, left = H - c;
      if (left <= 0) break;
#pragma unroll
      for (int e = 0; e < kCols; ++e) {
        v[i][e] -= mean;
        ss += e < left ? v[i][e] * v[i][e] : 0.f;
      }
    }
  }
  const float inv = q.gain ? (q.sum ? 1.f : q.mult) / sqrtf(block_sum<TH>(ss, tmp, phase) / H + q.eps) : q.mult;
  ss = 0.f;
#pragma unroll
  for (int i = 0; i < PASSES; ++i) {
    const int c = (threadIdx.x + i * TH) * kCols, left = H - c;
    if (left <= 0) break;
    if (!AHEAD) load_gains(i, c, left, false, true, false);
#pragma unroll
    for (int e = 0; e < kCols; ++e) {
      xv[i][e] += v[i][e] * inv * (q.gain ? gn[i][e] : 1.f);
      ss += e < left ? xv[i][e] * xv[i][e] : 0.f;
    }
  }
  const float pinv = q.pre ? 1.f / sqrtf(block_sum<TH>(ss, tmp, phase) / H + q.eps) : 1.f;
#pragma unroll
  for (int i = 0; i < PASSES; ++i) {
    const int c = (threadIdx.x + i * TH) * kCols, left = H - c;
    if (left <= 0) break;
    float y[kCols];
#pragma unroll
    for (int e = 0; e < kCols; ++e) y[e] = xv[i][e];
    if (q.pre) {
      if (!AHEAD) load_gains(i, c, left, false, false, true);
#pragma unroll
      for (int e = 0; e < kCols; ++e) y[e] = y[e] * pinv * gp[i][e];
    }
    T* bo = xb + (size_t)row * ldx + c;
    if (vec && ldx % kCols == 0) {
      *reinterpret_cast<floatx4*>(xr + c) = floatx4{xv[i][0], xv[i][1], xv[i][2], xv[i][3]};
      if (sizeof(T) == 2)
        *reinterpret_cast<uint2*>(bo) = uint2{pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3])};
      else
        *reinterpret_cast<floatx4*>(bo) = floatx4{y[0], y[1], y[2], y[3]};
    } else {
#pragma unroll
      for (int e = 0; e < kCols; ++e)
        if (e < left) xr[c + e] = xv[i][e], bo[e] = Elem<T>::make(y[e]);
    }
  }
}

// ------------------------------------------------------------------------------ routing
// One wave per token: softmax over all N <= 64 NR outputs, the `top` largest of score + correction
// (equals: the lower index), weight = score * scale.  renorm: the largest of logit + correction instead,
// weights = softmax over the chosen logits alone, times scale.  On return lane j < top holds the j-th choice.
// Reductions on the DPP path; the winner's lane comes from a ballot, so a choice costs about a
// hundred cycles.
template <int NR>
__device__ __forceinline__ void route_choose(const float* __restrict__ logits, const float* __restrict__ corr, int N,
                                             int top, float scale, int renorm, int lane, int& my_id, float& my_wt) {
  float s[NR], c[NR];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < NR; ++i) {  // unconditional: all requests go out before the first wait
    const int e = min(lane + 64 * i, N - 1);
    s[i] = logits[e];
    c[i] = corr[e];
  }
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    if (lane + 64 * i >= N) s[i] = c[i] = -INFINITY;
    if (renorm) c[i] += s[i];
    mx = fmaxf(mx, s[i]);
  }
  mx = wave_max_f32_uniform(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    s[i] = expf(s[i] - mx);
    sum += s[i];
  }
  sum = wave_sum_uniform(sum);
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    if (renorm) continue;
    s[i] = s[i] / sum;
    c[i] += s[i];
  }
  my_id = 0;
  my_wt = 0.f;
  for (int j = 0; j < top; ++j) {
    float best = c[0];
#pragma unroll
    for (int i = 1; i < NR; ++i) best = fmaxf(best, c[i]);
    best = wave_max_f32_uniform(best);
    bool found = false;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const uint64_t who = __ballot(c[i] == best);
      if (!found && who) {
        found = true;
        const int owner = __builtin_ctzll(who);
        const float sv = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, s[i]), owner));
        if (lane == owner) c[i] = -INFINITY;
        if (lane == j) my_id = owner + 64 * i, my_wt = sv * scale;
      }
    }
  }
  if (renorm) my_wt = my_wt * scale / wave_sum_uniform(my_wt);
}

template <int NR>
__global__ __launch_bounds__(64) void moe_route_kernel(const float* __restrict__ logits, const float* __restrict__ corr,
                                                       int32_t* __restrict__ idx, float* __restrict__ wt, int N, int ldl,
                                                       int top, float scale, int renorm) {
  const int row = blockIdx.x, lane = threadIdx.x;
  int id;
  float w;
  route_choose<NR>(logits + (size_t)row * ldl, corr, N, top, scale, renorm, lane, id, w);
  if (lane < top) {
    idx[(size_t)row * top + lane] = id;
    wt[(size_t)row * top + lane] = w;
  }
}

// ------------------------------------------------------------------------------ experts, decode
// A decode step's (token, expert) pairs, weights streamed once per pair: 16 output rows per
// workgroup, K over its waves, as dense_gemv_kernel.
struct MoeRows {
  const void* x;       // T [R][ldx]
  const void *gate, *up, *down;     // experts: [E][ff][ldx], [E][H][lda]
  const void *sgate, *sup, *sdown;  // the shared expert, or null
  void* act;           // T [R][top][lda]
  void* sact;          // T [R][ldsa]
  float* out;          // [R][H]
  const float* xres;   // [R][H] the sublayer's input (identity experts)
  int32_t* idx;        // [R][top]
  float* wt;
  const float* logits; // [R][ldl]
  const float* corr;   // routing inside the gated launch (null: idx and wt are given)
  float rscale;
  int outputs, renorm;
  int R, top, experts, ff, sff, H, ldx, lda, ldsa, ldl, gate_col;
  GluConst glu, sglu;
};

constexpr int kBatch = 4;
constexpr int kGuWaves = 4;

// NR > 0: every wave chooses its token's experts itself from the router's logits (no barrier, one
// launch fewer); the first tile of a token's first pair leaves idx and wt for the launch behind.
template <typename T, int NR>
__global__ __launch_bounds__(64 * kGuWaves) void moe_glu_rows_kernel(const MoeRows p) {
  __shared__ float red[kGuWaves][2][256];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int tiles = (p.ff + 15) / 16, pairs = p.R * p.top;
  int b = blockIdx.x, rows, N, ldo, tok0;
  const char *wg, *wu;
  T* out;
  GluConst glu;
  const uint32_t row_b = (uint32_t)p.ldx * sizeof(T);
  if (b < pairs * tiles) {
    const int pair = b / tiles;
    const int t = pair / p.top, slot = pair - t * p.top;
    b -= pair * tiles;
    int e;
    if constexpr (NR > 0) {
      int id;
      float w;
      route_choose<NR>(p.logits + (size_t)t * p.ldl, p.corr, p.outputs, p.top, p.rscale, p.renorm, lane, id, w);
      if (b == 0 && slot == 0 && wave == 0 && lane < p.top) {
        p.idx[pair + lane] = id;
        p.wt[pair + lane] = w;
      }
      e = __builtin_amdgcn_readlane(id, slot);
    } else {
      e = __builtin_amdgcn_readfirstlane(p.idx[pair]);
    }
    if (e >= p.experts) return;  // whole workgroup: the input itself, nothing to multiply
    const size_t off = (size_t)e * p.ff * row_b;
    wg = reinterpret_cast<const char*>(p.gate) + off;
    wu = reinterpret_cast<const char*>(p.up) + off;
    tok0 = pair / p.top;
    rows = 1;
    N = p.ff;
    out = reinterpret_cast<T*>(p.act) + (size_t)pair * p.lda;
    ldo = p.lda;
    glu = p.glu;
  } else {
    b -= pairs * tiles;
    wg = reinterpret_cast<const char*>(p.sgate);
    wu = reinterpret_cast<const char*>(p.sup);
    tok0 = 0;
    rows = p.R;
    N = p.sff;
    out = reinterpret_cast<T*>(p.sact);
    ldo = p.ldsa;
    glu = p.sglu;
  }
  const int n0 = b * 16, nrows = min(16, N - n0);
  const __amdgpu_buffer_rsrc_t rg = buf_of(wg + (size_t)n0 * row_b, (uint32_t)nrows * row_b);
  const __amdgpu_buffer_rsrc_t ru = buf_of(wu + (size_t)n0 * row_b, (uint32_t)nrows * row_b);
  const __amdgpu_buffer_rsrc_t rx =
      buf_of(reinterpret_cast<const char*>(p.x) + (size_t)tok0 * row_b, (uint32_t)rows * row_b);
  const int steps = (int)(row_b >> 6), per = (steps + kGuWaves - 1) / kGuWaves;
  const int s0 = min(steps, wave * per), s1 = min(steps, s0 + per);
  const uint32_t off = r * row_b + g * 16;
  floatx4 ag = {0.f, 0.f, 0.f, 0.f}, au = {0.f, 0.f, 0.f, 0.f};
  for (int s = s0; s < s1; s += kBatch) {
    uint4 gv[kBatch], uv[kBatch], xv[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const uint32_t o = s + i < s1 ? off + (s + i) * 64 : kPastEnd;
      gv[i] = buf_load16(rg, o, 0);
      uv[i] = buf_load16(ru, o, 0);
      xv[i] = buf_load16(rx, o, 0);
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      ag = Elem<T>::mma16(gv[i], xv[i], ag);
      au = Elem<T>::mma16(uv[i], xv[i], au);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    red[wave][0][r * 16 + 4 * g + e] = ag[e];
    red[wave][1][r * 16 + 4 * g + e] = au[e];
  }
  __syncthreads();
  for (int o = threadIdx.x; o < 16 * rows; o += 64 * kGuWaves) {
    const int m = o >> 4, n = o & 15;
    if (n >= nrows) continue;
    float gs = 0.f, us = 0.f;
#pragma unroll
    for (int w = 0; w < kGuWaves; ++w) gs += red[w][0][o], us += red[w][1][o];
    out[(size_t)m * ldo + n0 + n] = Elem<T>::make(clamped_glu(gs, us, glu));
  }
}

constexpr int kDnWaves = 16, kDnBatch = 8;

// out[t] = sum of weight * (down @ act) over the token's experts, + gate * shared, + weight * input
template <typename T>
__global__ __launch_bounds__(64 * kDnWaves) void moe_down_rows_kernel(const MoeRows p) {
  __shared__ float red[kDnWaves][16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int t = blockIdx.y, n0 = blockIdx.x * 16, nrows = min(16, p.H - n0);
  const uint32_t arow = (uint32_t)p.lda * sizeof(T), srow = (uint32_t)p.ldsa * sizeof(T);
  const int es = (int)(arow >> 6), ss = p.sdown ? (int)(srow >> 6) : 0;  // steps per expert, shared
  const int units = p.top * es + ss, per = (units + kDnWaves - 1) / kDnWaves;
  int u = min(units, wave * per);
  const int u1 = min(units, u + per);
  // the token's choice in lanes 0 .. top - 1
  const int my_id = p.idx[t * p.top + min(lane, p.top - 1)];
  const float my_wt = p.wt[t * p.top + min(lane, p.top - 1)];
  float tot[4] = {0.f, 0.f, 0.f, 0.f};
  while (u < u1) {  // the part of one expert's K range that falls into this wave's share
    const int slot = min(u / es, p.top);
    const bool sh = slot == p.top;
    const int base = slot * es, lim = sh ? ss : es;
    const int s0 = u - base, s1 = min(lim, u1 - base);
    u = base + s1;
    float wt;
    const char *w, *a;
    uint32_t rowb;
    if (sh) {
      wt = p.gate_col < 0 ? 1.f : 1.f / (1.f + expf(-p.logits[(size_t)t * p.ldl + p.gate_col]));
      w = reinterpret_cast<const char*>(p.sdown);
      a = reinterpret_cast<const char*>(p.sact) + (size_t)t * srow;
      rowb = srow;
    } else {
      const int e = __builtin_amdgcn_readlane(my_id, slot);
      if (e >= p.experts) continue;
      wt = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, my_wt), slot));
      w = reinterpret_cast<const char*>(p.down) + (size_t)e * p.H * arow;
      a = reinterpret_cast<const char*>(p.act) + (size_t)(t * p.top + slot) * arow;
      rowb = arow;
    }
    const __amdgpu_buffer_rsrc_t rw = buf_of(w + (size_t)n0 * rowb, (uint32_t)nrows * rowb);
    const __amdgpu_buffer_rsrc_t rx = buf_of(a, rowb);
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s = s0; s < s1; s += kDnBatch) {
      uint4 wv[kDnBatch], xv[kDnBatch];
#pragma unroll
      for (int i = 0; i < kDnBatch; ++i) {
        const bool ok = s + i < s1;
        wv[i] = buf_load16(rw, ok ? r * rowb + g * 16 + (s + i) * 64 : kPastEnd, 0);
        xv[i] = buf_load16(rx, ok ? g * 16 + (s + i) * 64 : kPastEnd, 0);  // every column: the one row
      }
#pragma unroll
      for (int i = 0; i < kDnBatch; ++i) acc = Elem<T>::mma16(wv[i], xv[i], acc);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) tot[e] = fmaf(wt, acc[e], tot[e]);
  }
  if (r == 0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) red[wave][4 * g + e] = tot[e];
  }
  const float pass = wave_sum_uniform(lane < p.top && my_id >= p.experts ? my_wt : 0.f);  // the input's own weight
  __syncthreads();
  if (threadIdx.x < (unsigned)nrows) {
    const int n = threadIdx.x;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < kDnWaves; ++w) v += red[w][n];
    if (pass != 0.f) v += pass * p.xres[(size_t)t * p.H + n0 + n];
    p.out[(size_t)t * p.H + n0 + n] = v;
  }
}

}  // namespace

#define EXO_TYPE_OK(what) EXO_REQUIRE(dtype == 0 || dtype == 1, what ": dtype must be 0 (bf16) or 1 (float32)")
#define EXO_LAUNCH_T(kernel, grid, block, lds, ...)                                  \
  do {                                                                               \
    if (dtype == 0)                                                                  \
      kernel<bf16_t><<<grid, block, lds, (hipStream_t)stream>>>(__VA_ARGS__);        \
    else                                                                             \
      kernel<float><<<grid, block, lds, (hipStream_t)stream>>>(__VA_ARGS__);         \
  } while (0)

extern "C" int exo_embed_rows(const int32_t* ids, const void* table, float* x, void* xb, int n, int V, int H, int ldt,
                              int ldx, float scale, int dtype, exo_stream_t stream) {
  EXO_TYPE_OK("exo_embed_rows");
  EXO_REQUIRE(ids && table && x && xb && n >= 0 && V > 0 && H > 0 && ldt >= H && ldx >= H, "exo_embed_rows: bad argument");
  if (n == 0) return EXO_OK;
  if (dtype == 0)
    embed_rows_kernel<bf16_t><<<n, 256, 0, (hipStream_t)stream>>>(ids, (const bf16_t*)table, x, (bf16_t*)xb, V, H, ldt, ldx, scale);
  else
    embed_rows_kernel<float><<<n, 256, 0, (hipStream_t)stream>>>(ids, (const float*)table, x, (float*)xb, V, H, ldt, ldx, scale);
  EXO_CHECK_LAUNCH("exo_embed_rows");
  return EXO_OK;
}

extern "C" int exo_norm_rows(const float* x, const int32_t* rows, const float* gain, void* y, int n, int H, int ldx,
                             int ldy, float eps, int center, int dtype, exo_stream_t stream) {
  EXO_TYPE_OK("exo_norm_rows");
  EXO_REQUIRE(x && gain && y && n >= 0 && H > 0 && ldx >= H && ldy >= H, "exo_norm_rows: bad argument");
  if (n == 0) return EXO_OK;
  const hipStream_t st = (hipStream_t)stream;
  if (n <= 256 && H > 1024) {
    if (dtype == 0)
      norm_rows_kernel<bf16_t, 1024><<<n, 1024, 0, st>>>(x, rows, gain, (bf16_t*)y, H, ldx, ldy, eps, center);
    else
      norm_rows_kernel<float, 1024><<<n, 1024, 0, st>>>(x, rows, gain, (float*)y, H, ldx, ldy, eps, center);
  } else if (dtype == 0)
    norm_rows_kernel<bf16_t, 256><<<n, 256, 0, st>>>(x, rows, gain, (bf16_t*)y, H, ldx, ldy, eps, center);
  else
    norm_rows_kernel<float, 256><<<n, 256, 0, st>>>(x, rows, gain, (float*)y, H, ldx, ldy, eps, center);
  EXO_CHECK_LAUNCH("exo_norm_rows");
  return EXO_OK;
}

static int post_norm(const exo_post_norm* q, const MoeSum& m, int n, int ldx, int dtype, exo_stream_t stream) {
  EXO_TYPE_OK("exo_post_norm_add");
  EXO_REQUIRE(q && q->x && q->x == q->x_out && q->operand && n >= 0 && q->H > 0 && q->H <= 16384 && ldx >= q->H,
              "exo_post_norm_add: bad argument (H=%d, x in place)", q ? q->H : 0);
  EXO_REQUIRE(!(q->sum && q->branch2) && (q->sum || !q->center), "exo_post_norm_add: a norm of the sum takes one branch");
  EXO_REQUIRE(q->gain || !(q->sum || q->branch2), "exo_post_norm_add: a branch without a norm is one, added as it is");
  EXO_REQUIRE(!q->branch2 || (q->gain_a && q->gain_b && !m.y), "exo_post_norm_add: two branches need a gain each");
  if (n == 0) return EXO_OK;
#define EXO_POST(TH, P)                                                                                          \
  do {                                                                                                           \
    if (dtype == 0)                                                                                              \
      post_norm_add_kernel<bf16_t, TH, P><<<n, TH, 0, (hipStream_t)stream>>>(*q, m, q->x_out, (bf16_t*)q->operand, ldx); \
    else                                                                                                         \
      post_norm_add_kernel<float, TH, P><<<n, TH, 0, (hipStream_t)stream>>>(*q, m, q->x_out, (float*)q->operand, ldx);   \
  } while (0)
  const int passes = exo_ceil_div(q->H, kRowThreads * kCols);
  if (n <= 256 && passes > 1) {  // few rows: the length of a row's chain counts, not the workgroups per CU
    if (passes <= 4) EXO_POST(1024, 1);
    else if (passes <= 8) EXO_POST(1024, 2);
    else EXO_POST(1024, 4);
  } else if (passes <= 1) EXO_POST(256, 1);
  else if (passes <= 2) EXO_POST(256, 2);
  else if (passes <= 4) EXO_POST(256, 4);
  else if (passes <= 8) EXO_POST(256, 8);
  else EXO_POST(256, 16);
#undef EXO_POST
  EXO_CHECK_LAUNCH("exo_post_norm_add");
  return EXO_OK;
}

extern "C" int exo_post_norm_add(const exo_post_norm* q, int n, int ldx, int dtype, exo_stream_t stream) {
  EXO_REQUIRE(q && q->branch && q->ldb >= q->H, "exo_post_norm_add: bad branch");
  return post_norm(q, MoeSum{}, n, ldx, dtype, stream);
}

extern "C" int exo_moe_sum_post_norm(const void* y, const int32_t* idx, const float* wt, const void* shared,
                                     const float* logits, int top, int experts, int ldy, int lds, int ldl, int gate_col,
                                     const exo_post_norm* q, int n, int ldx, int dtype, exo_stream_t stream) {
  EXO_REQUIRE(q && y && idx && wt && top > 0 && experts > 0 && ldy >= q->H && (!shared || (lds >= q->H && (gate_col < 0 || (logits && gate_col < ldl)))),
              "exo_moe_sum_post_norm: bad argument");
  return post_norm(q, MoeSum{y, idx, wt, shared, logits, top, experts, ldy, lds, ldl, gate_col}, n, ldx, dtype, stream);
}

extern "C" int exo_moe_route(const float* logits, const float* correction, int32_t* idx, float* wt, int rows, int n,
                             int ldl, int top, float scale, int renorm, exo_stream_t stream) {
  EXO_REQUIRE(logits && correction && idx && wt, "exo_moe_route: null pointer");
  EXO_REQUIRE(rows >= 0 && n > 0 && n <= 512 && ldl >= n && top > 0 && top <= 64 && top <= n,
              "exo_moe_route: need 0 < n <= %d and 0 < top <= min(64, n); got n=%d top=%d", 512, n, top);
  if (rows == 0) return EXO_OK;
  const auto fn = n <= 64 ? moe_route_kernel<1> : n <= 128 ? moe_route_kernel<2> : n <= 256 ? moe_route_kernel<4> : moe_route_kernel<8>;
  fn<<<rows, 64, 0, (hipStream_t)stream>>>(logits, correction, idx, wt, n, ldl, top, scale, renorm);
  EXO_CHECK_LAUNCH("exo_moe_route");
  return EXO_OK;
}

static MoeRows moe_rows_of(const exo_moe_rows* a) {
  MoeRows p{};
  p.x = a->x, p.gate = a->gate, p.up = a->up, p.down = a->down;
  p.sgate = a->shared_gate, p.sup = a->shared_up, p.sdown = a->shared_down;
  p.act = a->act, p.sact = a->shared_act, p.out = a->out, p.xres = a->x_res;
  p.idx = a->idx, p.wt = a->wt, p.logits = a->logits, p.corr = a->correction, p.rscale = a->router_scale;
  p.outputs = a->outputs, p.renorm = a->renorm;
  p.R = a->rows, p.top = a->top, p.experts = a->experts, p.ff = a->ff, p.sff = a->shared_ff, p.H = a->H;
  p.ldx = a->ldx, p.lda = a->lda, p.ldsa = a->ldsa, p.ldl = a->ldl, p.gate_col = a->gate_col;
  p.glu = GluConst{a->limit, a->alpha, a->shift, 0.f};
  p.sglu = GluConst{a->shared_limit, a->shared_alpha, a->shared_shift, 0.f};
  return p;
}
static int moe_rows_check(const exo_moe_rows* a) {
  EXO_REQUIRE(a && (a->dtype == 0 || a->dtype == 1), "exo_moe_rows: bad dtype");
  EXO_REQUIRE(a->rows > 0 && a->rows <= 16 && a->top > 0 && a->experts > 0 && a->ff > 0 && a->H > 0 && a->top <= 64,
              "exo_moe_rows: need 1..16 rows, top <= 64 and positive sizes (rows=%d top=%d)", a->rows, a->top);
  EXO_REQUIRE(!a->correction || (a->logits && a->outputs >= a->top && a->outputs <= 512 && a->ldl >= a->outputs),
              "exo_moe_rows: bad router (%d outputs)", a->outputs);
  EXO_REQUIRE(a->ldx % 64 == 0 && a->lda % 64 == 0 && a->ldx >= a->H && a->lda >= a->ff,
              "exo_moe_rows: row strides must be multiples of 64 (ldx=%d lda=%d)", a->ldx, a->lda);
  EXO_REQUIRE(a->x && a->gate && a->up && a->down && a->act && a->out && a->x_res && a->idx && a->wt,
              "exo_moe_rows: null pointer");
  EXO_REQUIRE(!a->shared_gate || (a->shared_up && a->shared_down && a->shared_act && (a->gate_col < 0 || a->logits) && a->shared_ff > 0 &&
                                  a->ldsa % 64 == 0 && a->ldsa >= a->shared_ff && a->gate_col < a->ldl),
              "exo_moe_rows: incomplete shared expert");
  return EXO_OK;
}

extern "C" int exo_moe_glu_rows(const exo_moe_rows* a, exo_stream_t stream) {
  const int rc = moe_rows_check(a);
  if (rc) return rc;
  const int dtype = a->dtype;
  const MoeRows p = moe_rows_of(a);
  const int grid = p.R * p.top * exo_ceil_div(p.ff, 16) + (p.sgate ? exo_ceil_div(p.sff, 16) : 0);
  const int n = p.corr ? p.outputs : 0;
#define EXO_GLU(NR)                                                                                   \
  do {                                                                                                \
    if (dtype == 0)                                                                                   \
      moe_glu_rows_kernel<bf16_t, NR><<<grid, 64 * kGuWaves, 0, (hipStream_t)stream>>>(p);            \
    else                                                                                              \
      moe_glu_rows_kernel<float, NR><<<grid, 64 * kGuWaves, 0, (hipStream_t)stream>>>(p);             \
  } while (0)
  if (n == 0) EXO_GLU(0);
  else if (n <= 64) EXO_GLU(1);
  else if (n <= 128) EXO_GLU(2);
  else if (n <= 256) EXO_GLU(4);
  else EXO_GLU(8);
#undef EXO_GLU
  EXO_CHECK_LAUNCH("exo_moe_glu_rows");
  return EXO_OK;
}

extern "C" int exo_moe_down_rows(const exo_moe_rows* a, exo_stream_t stream) {
  const int rc = moe_rows_check(a);
  if (rc) return rc;
  const int dtype = a->dtype;
  const MoeRows p = moe_rows_of(a);
  EXO_LAUNCH_T(moe_down_rows_kernel, dim3(exo_ceil_div(p.H, 16), p.R), 64 * kDnWaves, 0, p);
  EXO_CHECK_LAUNCH("exo_moe_down_rows");
  return EXO_OK;
}
