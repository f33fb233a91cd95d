// The sampling step of decode on the device: logits processors (token bans, repetition /
// presence / frequency penalties), log-normaliser, temperature / top-p / min-p / top-k
// filtering, a seeded draw, and the 20 most likely tokens with their log-probabilities -
// everything `_patched_step` of the reference does between the model call and the next
// token (src/exo/worker/engines/mlx/patches/opt_batch_gen.py:67-107), as a fixed sequence
// of launches that can sit at the end of a captured decode graph.
//
// The row of logits ([V] bf16, 250-300 KB, L2 resident: the lm_head GEMV has just written
// it) is cut into 64 slices, one workgroup each; every pass streams it once:
//   edits    one workgroup per row lists the few tokens the processors touch (banned ids
//            and the tokens of the penalty contexts, <= 264) with their edited values; the
//            streaming passes patch those positions through a slice bitmap, so the logits
//            themselves are never rewritten;
//   stats    per slice (max, argmax, sum exp(x - max));
//   coarse   (only with top-p / top-k / top-logprobs) every value is a bf16, i.e. a 16-bit
//   fine     order-preserving key.  Count and probability mass (2^-40 fixed point: integer sums
//            are exact, so nothing depends on arrival order) are first accumulated per BUCKET
//            of 128 keys (sign and exponent: 512 buckets) - in LDS per slice, then the few
//            non-empty buckets with global atomics.  Values that cannot matter to what the row asks
//            for are left out (`smallest_key`).  A scan of the 512 buckets from the top
//            finds the bucket in which the running count reaches k (and 20), and the one in
//            which the running mass reaches top_p; a second pass histograms only the values of
//            those buckets by their low 7 key bits, and a scan of those 128 entries, continued
//            from the totals above the bucket, gives the exact keys: the k-th largest value,
//            the nucleus edge, the 20th largest value.  (A flat 65536-entry table took 85 us to
//            fill with 2 atomics per logit and 115 us to scan and clear; the two levels take four
//            microseconds each.)
//   weights  per slice the sum of exp((x - max) / T) over the kept tokens (x >= threshold);
//            tokens at or above the 20th largest key are appended to a candidate list;
//   select   one workgroup per row: uniform from Philox-4x32-10 (key = request seed,
//            counter = draws so far), the slice in which the running sum crosses u * total,
//            then the token inside it (inverse CDF in vocabulary order); ranks the
//            candidates; appends the token to the history ring; advances the cache position.
//   greedy   in place of both where no row is drawn or listed: a wave per row (greedy steps 0.95 of the time, 1 to 64 rows).
// (Weights and select in one launch, whose last slice of a row to arrive finishes it: what the slices hand over costs as much as a launch; one to
// sixteen rows 0.97 to 1.07 of the time, and the 4096 workgroups of 64 rows wait for their stores where others could run, drawn rows 19.8 -> 26 us.)
// What bounds a step is latency: up to five dependent launches of 64 workgroups per row, each the way of its operands from
// memory and then a chain of reductions.  One row of 128256, top-p, min-p and top-logprobs: 30.8 -> 19.9 us (four rows
// of 151936: 35.3 -> 23.6) with everything requested up front, reductions through lane permutes, one word per table
// entry and only the values counted that matter; no filter but top-logprobs 44.4 -> 19.5 (an LDS maximum that all kept tokens
// took one by one), penalties over 64 tokens 76.3 -> 29.4 (edits found by position, not by a walk over the list).
// All filters compose to one value threshold: token i is kept iff x_i >= max(t_top_p,
// t_min_p, t_top_k).
#include "../../include/exo_mi355x.h"
#include "common.h"

namespace {

constexpr int kBlocks = 64;      // slices per row
constexpr int kMaxSlice = 4096;  // elements per slice (one or two 8-element chunks per thread)
constexpr int kMaxEdits = EXO_SAMPLER_MAX_CONTEXT + EXO_SAMPLER_MAX_BANNED;
constexpr int kTop = EXO_SAMPLER_TOP_LOGPROBS;
constexpr int kMaxCand = 32;    // values strictly above the 20th largest: 19 at most
constexpr int kBuckets = 512;  // key >> 7: sign and exponent
constexpr int kFine = 128;     // key & 127: mantissa, in value order inside a bucket
constexpr int kTargets = 3;    // 0: k-th largest (top-k), 1: nucleus edge (top-p), 2: 20th largest
constexpr float kBan = -1e9f;

typedef unsigned long long u64;

// Count and mass of a table entry in one word, so that one integer addition carries both: the mass in 2^-40 below, the
// count above.  A row has at most 2^18 tokens.  Its probabilities sum up to 1 but for the rounding of the log-normaliser lse = max + log
// sum: less than 2 where |max| is below 2^23 (lse off by 1/2 at most).  Beyond that the logarithm may be lost whole, each of n equal
// maxima then has a probability of 1, and masses count in 2^-26 (mass_shift): 2^18 of those still fit below the count.
constexpr int kCountShift = 45;
constexpr u64 kMassMask = (1ull << kCountShift) - 1;
constexpr float kMassOne = 0x1p40f;
constexpr int kMassShift = 14;
__device__ __forceinline__ int mass_shift(float mx) { return fabsf(mx) < 0x1p23f ? 0 : kMassShift; }

struct RowWs {
  float part[kBlocks][4];  // max, argmax (int bits), sum exp(x - max), kept weight
  int n_edit;
  float thr;    // value threshold from top-p / top-k (-inf: none)
  int key_top;  // key of the 20th largest value
  int cand_n;
  // per target: the bucket in which the running count / mass from the top crosses it (-1:
  // never), and the count and mass of the buckets above it
  int bkt[4];
  u64 above[4];
  int edit_idx[kMaxEdits];
  float edit_val[kMaxEdits];
  u64 cand[kMaxCand];  // key << 32 | index, values strictly above the 20th largest
  // tokens whose value EQUALS the 20th largest, per slice: the first kTop of them in
  // vocabulary order (a flat row has thousands; which of them make the list must not depend
  // on the order in which workgroups arrive)
  int tie_n[kBlocks];
  int tie_idx[kBlocks][kTop];
};
constexpr size_t kRowWsBytes = (sizeof(RowWs) + 255) / 256 * 256;

// count and mass per bucket, and per low key of each target's bucket; zero between steps
struct Tables {
  u64 coarse[kBuckets];
  u64 fine[kTargets][kFine];
};
constexpr size_t kTablesBytes = (sizeof(Tables) + 255) / 256 * 256;

// Workspace: one self-contained region per row (the row's RowWs, then its tables), so
// launches of different row counts can share one workspace.
constexpr size_t kRowStride = kRowWsBytes + kTablesBytes;
__device__ __forceinline__ RowWs* row_ws(void* ws, int row) {
  return reinterpret_cast<RowWs*>(static_cast<char*>(ws) + (size_t)row * kRowStride);
}
__device__ __forceinline__ Tables* row_tables(void* ws, int row) {
  return reinterpret_cast<Tables*>(static_cast<char*>(ws) + (size_t)row * kRowStride + kRowWsBytes);
}

// order-preserving 16-bit key of a bf16 value and back
__device__ __forceinline__ int key_of(float x) {
  const uint32_t b = __builtin_bit_cast(uint32_t, x) >> 16;
  return (b & 0x8000u) ? (~b & 0xffffu) : (b | 0x8000u);
}
__device__ __forceinline__ float value_of(int key) {
  const uint32_t b = (key & 0x8000) ? (key & 0x7fff) : (~key & 0xffff);
  return __builtin_bit_cast(float, b << 16);
}
__device__ __forceinline__ float bf16r(float v) { return bf2f(f2bf(v)); }

// ---- slices -------------------------------------------------------------------
// What a launch waits for is the way of its operands from memory (the logits and the tables lie in the other dies' caches:
// a microsecond a request).  So every kernel requests all it needs, the edit list's length among it, before it
// uses any of it.
struct SliceGeom {
  int per, lo, hi;
  bool vec;
};
__host__ __device__ __forceinline__ int slice_elements(int V) { return ((((V + 7) >> 3) + kBlocks - 1) / kBlocks) << 3; }
__device__ __forceinline__ SliceGeom slice_geom(const bf16_t* logits, int V, int block) {
  SliceGeom g;
  g.vec = (V & 7) == 0 && ((uintptr_t)logits & 15) == 0;
  g.per = slice_elements(V);
  g.lo = min(block * g.per, V);
  g.hi = min(g.lo + g.per, V);
  return g;
}

// This thread's share of the slice as it was requested: chunk u < NU holds the 8 elements from index i0[u].  Slices of up
// to 2048 elements (rows of up to 131072) are one chunk per thread.
template <int NU>
struct Share {
  uint32_t w[4 * NU];
  int i0[NU];
  int chunks;  // that hold elements for some lane of this wave (its values past them are all -inf)
};
template <int NU>
__device__ __forceinline__ void request_share(const bf16_t* src, const SliceGeom& g, Share<NU>& s) {
#pragma unroll
  for (int u = 0; u < NU; ++u) s.i0[u] = g.lo + ((int)threadIdx.x + 256 * u) * 8;
  s.chunks = NU == 1 || g.lo + 2048 + 8 * __builtin_amdgcn_readfirstlane((int)threadIdx.x & ~63) >= g.hi ? 1 : NU;
  if (g.vec) {
#pragma unroll
    for (int u = 0; u < NU; ++u) {  // (past the slice: the row's first chunk, dropped afterwards)
      const uint4 v = *reinterpret_cast<const uint4*>(src + (s.i0[u] < g.hi ? s.i0[u] : 0));
      s.w[4 * u] = v.x, s.w[4 * u + 1] = v.y, s.w[4 * u + 2] = v.z, s.w[4 * u + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = s.i0[u] + 2 * k;
        const uint32_t lo = i < g.hi ? src[i] : 0xff80u, hi = i + 1 < g.hi ? src[i + 1] : 0xff80u;  // (-inf)
        s.w[4 * u + k] = lo | hi << 16;
      }
  }
}

// The slice's edited positions as a bitmap in LDS, and their values by position.
struct EditLds {
  uint32_t bm[kMaxSlice / 32];
  bf16_t val[kMaxSlice];
};
// (n: the row's number of edits, the same in every thread; ends in a barrier where there are any)
__device__ __forceinline__ void stage_edits(const RowWs* w, const SliceGeom& g, int n, EditLds& e) {
  if (n <= 0) return;
  for (int i = threadIdx.x; i < kMaxSlice / 32; i += blockDim.x) e.bm[i] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int t = w->edit_idx[i] - g.lo;
    if (t >= 0 && t < g.hi - g.lo) {
      e.val[t] = f2bf(w->edit_val[i]);  // (rounded already)
      atomicOr(&e.bm[t >> 5], 1u << (t & 31));
    }
  }
  __syncthreads();
}

// The share's values; positions outside the slice read -inf.  Edits are applied.
template <int NU>
__device__ __forceinline__ void expand_share(const Share<NU>& s, const SliceGeom& g, int n_edit, const EditLds& e,
                                             float (&xv)[8 * NU]) {
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const bool in = s.i0[u] < g.hi;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t w = in ? s.w[4 * u + k] : 0xff80ff80u;  // (-inf)
      xv[8 * u + 2 * k] = bf_lo(w);
      xv[8 * u + 2 * k + 1] = bf_hi(w);
    }
    if (n_edit > 0 && in) {
      const int o = s.i0[u] - g.lo;  // multiple of 8: the chunk's bits sit in one byte
      const uint32_t bits = (e.bm[o >> 5] >> (o & 31)) & 0xffu;
      if (bits) {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (bits & (1u << k)) xv[8 * u + k] = bf2f(e.val[o + k]);
      }
    }
  }
}

// (max, lowest index holding it, sum exp(x - max)) over the row from the slice partials;
// every wave computes it for itself (64 partials = one per lane).
struct Partial {
  float mx, sum;
  int at;
};
__device__ __forceinline__ Partial request_partial(const RowWs* w) {
  const int lane = threadIdx.x & 63;
  const float2 a = *reinterpret_cast<const float2*>(&w->part[lane][0]);
  return {a.x, w->part[lane][2], __float_as_int(a.y)};
}
// the largest of the lanes' values and the lowest index among the lanes that hold it
__device__ __forceinline__ void wave_argmax(float v, int i, float& mx, int& mi) {
  mx = wave_max_f32_uniform(v);
  mi = (int)~wave_max_u32(~(uint32_t)(v == mx ? i : 0x7fffffff));
}
__device__ __forceinline__ void merge_stats(const Partial& p, float& mx, int& mi, float& lse) {
  wave_argmax(p.mx, p.at, mx, mi);
  const float se = wave_sum((p.mx > -INFINITY) ? p.sum * expf(p.mx - mx) : 0.f);
  lse = mx + logf(se);
}

// ---- edits --------------------------------------------------------------------
__global__ __launch_bounds__(512) void sampler_edits_kernel(
    const bf16_t* __restrict__ logits, const exo_sampler_params* __restrict__ params,
    const int32_t* __restrict__ history, const int32_t* __restrict__ hist_len, void* ws, int V,
    int hist_cap) {
  static_assert(kMaxEdits % 4 == 0 && kMaxEdits <= 512, "a candidate per thread, read four at a time");
  __shared__ __align__(16) int s_tok[kMaxEdits];
  __shared__ int s_n;
  const int row = blockIdx.x, c = threadIdx.x;
  const exo_sampler_params& p = params[row];
  RowWs* w = row_ws(ws, row);
  const bool rep_on = p.repetition_penalty != 0.f && p.repetition_penalty != 1.f;
  const bool pres_on = p.presence_penalty != 0.f;
  const bool freq_on = p.frequency_penalty != 0.f;
  const int len = hist_len[row];
  const int n_hist = min(len, hist_cap);
  const int rep_ctx = rep_on ? min(max(p.repetition_context, 0), n_hist) : 0;
  const int pres_ctx = pres_on ? min(max(p.presence_context, 0), n_hist) : 0;
  const int freq_ctx = freq_on ? min(max(p.frequency_context, 0), n_hist) : 0;
  const int max_ctx = max(rep_ctx, max(pres_ctx, freq_ctx));
  const int nb = min(max(p.n_banned, 0), EXO_SAMPLER_MAX_BANNED);
  const int32_t* hrow = history + (size_t)row * hist_cap;
  // candidate c: banned id c, or the token j = c - MAX_BANNED positions back in the history
  int tok = -1;
  if (c < nb) {
    tok = p.banned[c];
  } else if (c >= EXO_SAMPLER_MAX_BANNED && c - EXO_SAMPLER_MAX_BANNED < max_ctx) {
    const int j = c - EXO_SAMPLER_MAX_BANNED;
    tok = hrow[(len - 1 - j) % hist_cap];
  }
  if (tok >= V) tok = -1;
  if (c < kMaxEdits) s_tok[c] = tok;
  if (c == 0) s_n = 0;
  float v = tok >= 0 ? bf2f(logits[(size_t)row * V + tok]) : 0.f;
  __syncthreads();
  if (c < kMaxEdits && tok >= 0) {
    // one walk over all candidates, four a step (a step at a time its latency was the launch: 64 tokens of history 8 us)
    bool first = true, banned = false, in_rep = false, in_pres = false;
    int cf = 0;
    const int steps = (EXO_SAMPLER_MAX_BANNED + max_ctx + 3) / 4;
#pragma unroll 4
    for (int i = 0; i < steps; ++i) {
      const int4 four = reinterpret_cast<const int4*>(s_tok)[i];
      const int t[4] = {four.x, four.y, four.z, four.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int o = 4 * i + k, j = o - EXO_SAMPLER_MAX_BANNED;
        const bool hit = t[k] == tok, past = hit && j >= 0;
        first = first && !(hit && o < c);
        banned = banned || (hit && j < 0);  // (places past the last banned id hold none)
        in_rep = in_rep || (past && j < rep_ctx);
        in_pres = in_pres || (past && j < pres_ctx);
        cf += past && j < freq_ctx ? 1 : 0;
      }
    }
    if (first) {
      if (banned) v = bf16r(kBan);
      if (in_rep) v = bf16r(v < 0.f ? __fmul_rn(v, p.repetition_penalty) : __fdiv_rn(v, p.repetition_penalty));
      if (in_pres) v = bf16r(__fsub_rn(v, p.presence_penalty));
      if (cf > 0) v = bf16r(__fsub_rn(v, __fmul_rn(p.frequency_penalty, (float)cf)));
      const int slot = atomicAdd(&s_n, 1);
      w->edit_idx[slot] = tok;
      w->edit_val[slot] = v;
    }
  }
  __syncthreads();
  if (c == 0) w->n_edit = s_n;
}

// ---- stats --------------------------------------------------------------------
template <int NU>
__global__ __launch_bounds__(256) void sample_stats_kernel(const bf16_t* __restrict__ logits,
                                                           void* ws, int V, int has_edits) {
  __shared__ EditLds ed;
  __shared__ float smax[4], ssum[4];
  __shared__ int sidx[4];
  const int row = blockIdx.y;
  RowWs* w = row_ws(ws, row);
  const SliceGeom g = slice_geom(logits, V, blockIdx.x);
  Share<NU> sh;
  request_share(logits + (size_t)row * V, g, sh);
  const int n_edit = has_edits ? w->n_edit : 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {  // per-step fields of the row
    w->thr = -INFINITY;
    w->key_top = 0;
    w->cand_n = 0;
  }
  stage_edits(w, g, n_edit, ed);
  float xv[8 * NU];
  expand_share(sh, g, n_edit, ed, xv);
  float mx = -INFINITY;
  int mi = 0x7fffffff;
#pragma unroll
  for (int u = 0; u < NU; ++u)
    if (u < sh.chunks) {
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (xv[8 * u + k] > mx) {
          mx = xv[8 * u + k];
          mi = sh.i0[u] + k;
        }
    }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  wave_argmax(mx, mi, mx, mi);
  if (lane == 0) {
    smax[wave] = mx;
    sidx[wave] = mi;
  }
  __syncthreads();
  float bm = smax[0];
  int bi = sidx[0];
#pragma unroll
  for (int wv = 1; wv < 4; ++wv)
    if (smax[wv] > bm || (smax[wv] == bm && sidx[wv] < bi)) {
      bm = smax[wv];
      bi = sidx[wv];
    }
  float se = 0.f;
  if (bm > -INFINITY) {
#pragma unroll
    for (int u = 0; u < NU; ++u)
      if (u < sh.chunks) {
#pragma unroll
        for (int k = 0; k < 8; ++k) se += expf(xv[8 * u + k] - bm);  // padding is -inf: exp = 0
      }
  }
  se = wave_sum(se);
  if (lane == 0) ssum[wave] = se;
  __syncthreads();
  if (threadIdx.x == 0)
    *reinterpret_cast<float4*>(&w->part[blockIdx.x][0]) =
        make_float4(bm, __int_as_float(bi), ssum[0] + ssum[1] + ssum[2] + ssum[3], 0.f);
}

// ---- key table ----------------------------------------------------------------
__device__ __forceinline__ bool row_needs_table(const exo_sampler_params& p, bool want_top) {
  const bool sampling = p.temperature != 0.f;
  return want_top || (sampling && (p.top_k > 0 || (p.top_p > 0.f && p.top_p < 1.f)));
}

// what a row asks of the tables
struct Wanted {
  unsigned int kk;  // top-k (0: none)
  bool use_p;       // top-p
  u64 target;       // top_p of the mass, fixed point
  float one;        // a probability of 1 in the same
  bool top;         // the 20 most likely
};
__device__ __forceinline__ Wanted wanted_of(const exo_sampler_params& p, bool want_top, float mx) {
  const bool sampling = p.temperature != 0.f;
  Wanted q;
  q.kk = (sampling && p.top_k > 0) ? (unsigned int)p.top_k : 0u;
  q.use_p = sampling && p.top_p > 0.f && p.top_p < 1.f;
  const int shift = mass_shift(mx);
  q.one = shift ? kMassOne / (float)(1 << kMassShift) : kMassOne;
  q.target = q.use_p ? ((u64)((double)p.top_p * (double)kMassOne) + (1u << shift) - 1) >> shift : 0ull;
  q.top = want_top;
  return q;
}
__device__ __forceinline__ float keep_threshold(const exo_sampler_params& p, float table_thr,
                                                float mx) {
  float thr = table_thr;
  if (p.min_p > 0.f) thr = fmaxf(thr, mx + logf(p.min_p));
  return thr;
}

// The smallest key that can matter to what the row asks of the tables; values below it are not counted.
//   20th (k-th) largest: 32 pairs of slices hold a maximum each, so 32 values lie at or above the smallest of these (64
//   at or above the smallest maximum of a slice), and the 20th largest is none below it;
//   nucleus edge: below the threshold of min_p it changes nothing.
// A row of 128256 normally distributed logits keeps some 100 values for the 20 largest, and 3 % for a min_p of 0.05.
__device__ __forceinline__ int smallest_key(const exo_sampler_params& p, const Wanted& q, float slice_max, float mx) {
  const float pair = fmaxf(slice_max, dpp_get<0xB1, 0xf>(slice_max));  // (quad_perm [1,0,3,2])
  const float of_pairs = -wave_max_f32_uniform(-pair), of_slices = -wave_max_f32_uniform(-slice_max);
  const int k32 = of_pairs > -INFINITY ? key_of(of_pairs) : 0, k64 = of_slices > -INFINITY ? key_of(of_slices) : 0;
  int lo = 0x10000;
  static_assert(kTop <= 32, "as many values at least lie above the pairs' bound");
  if (q.top) lo = min(lo, k32);
  if (q.kk) lo = min(lo, q.kk <= 32 ? k32 : q.kk <= 64 ? k64 : 0);
  // (key_of cuts towards zero: the values at or above a negative bound are those from its key on, and for a positive
  // one a value below it may be counted too)
  if (q.use_p) lo = min(lo, p.min_p > 0.f ? key_of(keep_threshold(p, -INFINITY, mx)) : 0);
  return lo;
}

__device__ __forceinline__ u64 readlane_u64(u64 v, int src) {
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)v, src), hi = __builtin_amdgcn_readlane((int)(v >> 32), src);
  return ((u64)hi << 32) | lo;
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ u64 dpp_get_u64(u64 v) {  // (0 from lanes outside)
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, ROW_MASK, 0xf, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROW_MASK, 0xf, false);
  return ((u64)hi << 32) | lo;
}
// inclusive sums over the lanes, in lane order
__device__ __forceinline__ int wave_scan_i32(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1, 2, 4, 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}
__device__ __forceinline__ u64 wave_scan_u64(u64 v) {
  v += dpp_get_u64<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
  v += dpp_get_u64<0x112, 0xf>(v);
  v += dpp_get_u64<0x114, 0xf>(v);
  v += dpp_get_u64<0x118, 0xf>(v);
  v += dpp_get_u64<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v += dpp_get_u64<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}

// One wave walks N = 64 * PER entries from the highest index down (lane t holds entries
// N-1 - PER*t .. downwards in v), the running (count, mass) starting at above[j].  For each target:
// the entry at which the running count reaches kk / 20 (count before it below, count with it
// at or above), or the running mass reaches `target`; found[] = entry index or -1, and
// above[] = the totals strictly above that entry.  Every lane returns the same values.
template <int PER>
__device__ __forceinline__ void request_table(const u64* __restrict__ t, u64 (&v)[PER]) {
  const int hi = 64 * PER - 1 - PER * (int)(threadIdx.x & 63);
#pragma unroll
  for (int i = 0; i < PER; ++i) v[i] = t[hi - i];
}
template <int PER>
__device__ __forceinline__ void scan_down(const u64 (&v)[PER], const Wanted& q, const bool (&active)[kTargets],
                                          int (&found)[kTargets], u64 (&above)[kTargets]) {
  const int lane = threadIdx.x & 63;
  const int hi = 64 * PER - 1 - PER * lane;
  u64 sum = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) sum += v[i];
  const u64 ahead = wave_scan_u64(sum) - sum;  // totals of the lanes above (higher entries)
#pragma unroll
  for (int j = 0; j < kTargets; ++j) {
    int f = -1;
    u64 fa = 0;
    if (active[j]) {
      u64 run = above[j] + ahead;
      const unsigned int want_c = j == 0 ? q.kk : (unsigned int)kTop;
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const u64 next = run + v[i];
        const bool hit = (j == 1) ? ((run & kMassMask) < q.target && (next & kMassMask) >= q.target)
                                  : ((unsigned int)(run >> kCountShift) < want_c && (unsigned int)(next >> kCountShift) >= want_c);
        if (hit) {
          f = hi - i;
          fa = run;
        }
        run = next;
      }
    }
    const u64 mask = __ballot(f >= 0);
    if (mask) {
      const int src = __ffsll((long long)mask) - 1;
      found[j] = __builtin_amdgcn_readlane(f, src);
      above[j] = readlane_u64(fa, src);
    } else {
      found[j] = -1;
      above[j] = 0;
    }
  }
}

// ---- coarse: count and mass per bucket ------------------------------------------------
// Logits fall into a handful of buckets: additions of a wave to one word of LDS go one by one, so every eighth
// lane has a table of its own.
constexpr int kCopies = 8;
template <int NU>
__global__ __launch_bounds__(256) void sample_coarse_kernel(
    const bf16_t* __restrict__ logits, const exo_sampler_params* __restrict__ params, void* ws,
    int V, int has_edits, int want_top) {
  __shared__ EditLds ed;
  __shared__ __align__(16) u64 hist[kBuckets * kCopies];
  const int row = blockIdx.y;
  RowWs* w = row_ws(ws, row);
  const SliceGeom g = slice_geom(logits, V, blockIdx.x);
  Share<NU> sh;
  request_share(logits + (size_t)row * V, g, sh);
  const Partial part = request_partial(w);
  const int n_edit = has_edits ? w->n_edit : 0;
  const exo_sampler_params p = params[row];
  if (!row_needs_table(p, want_top != 0)) return;
  for (int i = threadIdx.x; i < kBuckets * kCopies / 2; i += 256) reinterpret_cast<uint4*>(hist)[i] = make_uint4(0, 0, 0, 0);
  stage_edits(w, g, n_edit, ed);
  float xv[8 * NU];
  expand_share(sh, g, n_edit, ed, xv);
  float mx, lse;
  int mi;
  merge_stats(part, mx, mi, lse);
  const Wanted q = wanted_of(p, want_top != 0, mx);
  const int lo = smallest_key(p, q, part.mx, mx);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NU; ++u)
    if (u < sh.chunks) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float x = xv[8 * u + k];
        const int key = key_of(x);
        if (sh.i0[u] + k < g.hi && key >= lo) {  // (-inf logits are real values too: key 0x007f)
          u64 v = 1ull << kCountShift;
          if (q.use_p) v += (u64)(expf(x - lse) * q.one);
          atomicAdd(&hist[(key >> 7) * kCopies + (threadIdx.x & (kCopies - 1))], v);
        }
      }
    }
  __syncthreads();
  Tables* T = row_tables(ws, row);
  for (int b = threadIdx.x; b < kBuckets; b += 256) {
    u64 v = 0;
#pragma unroll
    for (int c = 0; c < kCopies; ++c) v += hist[b * kCopies + c];
    if (v) atomicAdd(&T->coarse[b], v);
  }
}

// ---- fine: the buckets that hold a target, by their low key bits ----------------------
template <int NU>
__global__ __launch_bounds__(256) void sample_fine_kernel(
    const bf16_t* __restrict__ logits, const exo_sampler_params* __restrict__ params, void* ws,
    int V, int has_edits, int want_top) {
  __shared__ EditLds ed;
  __shared__ u64 hist[kTargets][kFine];
  const int row = blockIdx.y;
  RowWs* w = row_ws(ws, row);
  Tables* T = row_tables(ws, row);
  const SliceGeom g = slice_geom(logits, V, blockIdx.x);
  // every wave finds the target buckets for itself (512 entries, L2 resident)
  u64 entry[kBuckets / 64];
  request_table(T->coarse, entry);
  Share<NU> sh;
  request_share(logits + (size_t)row * V, g, sh);
  const Partial part = request_partial(w);
  const int n_edit = has_edits ? w->n_edit : 0;
  const exo_sampler_params p = params[row];
  if (!row_needs_table(p, want_top != 0)) return;
  for (int i = threadIdx.x; i < kTargets * kFine; i += 256) (&hist[0][0])[i] = 0;
  stage_edits(w, g, n_edit, ed);
  float mx, lse;
  int mi;
  merge_stats(part, mx, mi, lse);
  const Wanted q = wanted_of(p, want_top != 0, mx);
  int bkt[kTargets];
  u64 above[kTargets] = {0ull, 0ull, 0ull};
  {
    const bool active[kTargets] = {q.kk != 0, q.use_p, q.top};
    scan_down(entry, q, active, bkt, above);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
#pragma unroll
    for (int j = 0; j < kTargets; ++j) {
      w->bkt[j] = bkt[j];
      w->above[j] = above[j];
    }
  }
  if (bkt[0] < 0 && bkt[1] < 0 && bkt[2] < 0) return;  // (uniform over the workgroup)
  float xv[8 * NU];
  expand_share(sh, g, n_edit, ed, xv);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NU; ++u)
    if (u < sh.chunks) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float x = xv[8 * u + k];
        const int key = key_of(x), b = key >> 7, f = key & (kFine - 1);
        if (sh.i0[u] + k < g.hi && (b == bkt[0] || b == bkt[1] || b == bkt[2])) {
          const u64 one = 1ull << kCountShift;
          if (b == bkt[0]) atomicAdd(&hist[0][f], one);
          if (b == bkt[1]) atomicAdd(&hist[1][f], one + (u64)(expf(x - lse) * q.one));
          if (b == bkt[2]) atomicAdd(&hist[2][f], one);
        }
      }
    }
  __syncthreads();
  for (int i = threadIdx.x; i < kTargets * kFine; i += 256) {
    const u64 v = (&hist[0][0])[i];
    if (v) atomicAdd(&T->fine[0][0] + i, v);
  }
}

// The exact keys from the fine tables, a target per wave (left in `keys`; the caller's barrier): the keys of
// the k-th largest value, of the nucleus edge and of the 20th largest value, -1 for none.
struct FineRequest {
  u64 entry[kFine / 64], above;
  int bkt;
};
__device__ __forceinline__ FineRequest request_fine(const RowWs* w, const Tables* T) {
  FineRequest r;
  const int j = min(__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), kTargets - 1);
  request_table(T->fine[j], r.entry);
  r.bkt = w->bkt[j];
  r.above = w->above[j];
  return r;
}
__device__ __forceinline__ void fine_keys(const FineRequest& r, const Wanted& q, int (&keys)[kTargets]) {
  const int j = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  if (j >= kTargets) return;
  // (-1: fewer than k (20) tokens in all, or the mass never reaches top_p above min_p's threshold)
  const bool have[kTargets] = {j == 0 && q.kk != 0, j == 1 && q.use_p, j == 2 && q.top};
  int f[kTargets];
  u64 above[kTargets] = {r.above, r.above, r.above};
  scan_down(r.entry, q, have, f, above);
  const int at = j == 0 ? f[0] : j == 1 ? f[1] : f[2];
  if ((threadIdx.x & 63) == 0) keys[j] = r.bkt >= 0 && at >= 0 ? (r.bkt << 7) | at : -1;
}

// ---- weights ------------------------------------------------------------------
template <int NU>
__global__ __launch_bounds__(256) void sample_weights_kernel(
    const bf16_t* __restrict__ logits, const exo_sampler_params* __restrict__ params, void* ws,
    int V, int has_edits, int has_tables, int want_top) {
  __shared__ EditLds ed;
  __shared__ float ssum[4];
  __shared__ int s_keys[kTargets], s_ties[4];
  const int row = blockIdx.y;
  RowWs* w = row_ws(ws, row);
  Tables* T = row_tables(ws, row);
  const SliceGeom g = slice_geom(logits, V, blockIdx.x);
  FineRequest fine = {};
  if (has_tables) fine = request_fine(w, T);
  Share<NU> sh;
  request_share(logits + (size_t)row * V, g, sh);
  const Partial part = request_partial(w);
  const int n_edit = has_edits ? w->n_edit : 0;
  const exo_sampler_params p = params[row];
  const bool sampling = p.temperature != 0.f;
  if (!sampling && !want_top) return;
  // the exact keys of this step from the fine tables; the first workgroup leaves them for the select
  // launch and clears the bucket table, whose last reader was the previous launch
  float table_thr = -INFINITY;
  int kt = 0;
  const bool table = has_tables && row_needs_table(p, want_top != 0);  // (uniform over the workgroup)
  float mx, lse;
  int mi;
  merge_stats(part, mx, mi, lse);
  if (table) {
    fine_keys(fine, wanted_of(p, want_top != 0, mx), s_keys);
    if (blockIdx.x == 0)
      for (int b = threadIdx.x; b < kBuckets; b += 256) T->coarse[b] = 0;
  }
  stage_edits(w, g, n_edit, ed);
  float xv[8 * NU];
  expand_share(sh, g, n_edit, ed, xv);
  if (table) {
    __syncthreads();
    if (s_keys[0] >= 0) table_thr = value_of(s_keys[0]);
    if (s_keys[1] >= 0) table_thr = fmaxf(table_thr, value_of(s_keys[1]));
    if (s_keys[2] >= 0) kt = s_keys[2];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      w->thr = table_thr;
      w->key_top = kt;
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int mine[NU];  // of this thread's chunks, the values equal to the 20th largest
  if (want_top) {
    // strictly above the 20th largest value: at most 19 tokens in the whole row, any order
    // (the select launch ranks them)
    int all = 0;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      mine[u] = 0;
      if (u < sh.chunks) {
        uint32_t larger = 0;  // (a bit per value: without branches, since hardly any thread has one)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int key = sh.i0[u] + k < g.hi ? key_of(xv[8 * u + k]) : -1;
          larger |= key > kt ? 1u << k : 0u;
          mine[u] += key == kt ? 1 : 0;
        }
        if (larger) {
#pragma unroll
          for (int k = 0; k < 8; ++k)
            if (larger & (1u << k)) {
              const int slot = atomicAdd(&w->cand_n, 1);
              if (slot < kMaxCand) w->cand[slot] = ((u64)key_of(xv[8 * u + k]) << 32) | (unsigned int)(sh.i0[u] + k);
            }
        }
      }
      all += mine[u];
    }
    const u64 any = __ballot(all > 0);
    if (lane == 0) s_ties[wave] = any != 0;
  }
  if (sampling) {
    const float thr = keep_threshold(p, table_thr, mx);
    const float inv_t = 1.f / p.temperature;
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < NU; ++u)
      if (u < sh.chunks) {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (xv[8 * u + k] >= thr) s += expf((xv[8 * u + k] - mx) * inv_t);
      }
    s = wave_sum(s);
    if (lane == 0) ssum[wave] = s;
  }
  __syncthreads();
  if (sampling && threadIdx.x == 0) w->part[blockIdx.x][3] = ssum[0] + ssum[1] + ssum[2] + ssum[3];
  if (!want_top) return;
  if (!(s_ties[0] | s_ties[1] | s_ties[2] | s_ties[3])) {  // (most slices; uniform over the workgroup)
    if (threadIdx.x == 0) w->tie_n[blockIdx.x] = 0;
    return;
  }
  // equal to the 20th largest: this slice's first kTop in vocabulary order, by a scan over the
  // threads (chunk 0 of every thread precedes chunk 1 of any)
  int base = 0;
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int inc = wave_scan_i32(mine[u]);
    __syncthreads();  // (the words are read above and in the round before)
    if (lane == 63) s_ties[wave] = inc;
    __syncthreads();
    int before = base;
    for (int q = 0; q < wave; ++q) before += s_ties[q];
    int at = before + inc - mine[u];  // ties of this slice in front of this thread's chunk
    if (mine[u] > 0 && at < kTop) {
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (sh.i0[u] + k < g.hi && key_of(xv[8 * u + k]) == kt) {
          if (at < kTop) w->tie_idx[blockIdx.x][at] = sh.i0[u] + k;
          ++at;
        }
    }
    base += s_ties[0] + s_ties[1] + s_ties[2] + s_ties[3];
  }
  if (threadIdx.x == 0) w->tie_n[blockIdx.x] = min(base, kTop);
}

// ---- select -------------------------------------------------------------------
__device__ __forceinline__ void philox4x32_10(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const unsigned long long p0 = 0xD2511F53ull * c[0], p1 = 0xCD9E8D57ull * c[2];
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0, n1 = (uint32_t)p1;
    const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1, n3 = (uint32_t)p0;
    c[0] = n0;
    c[1] = n1;
    c[2] = n2;
    c[3] = n3;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

// What a step writes, and what of the sequence it reads for that (requested up front).
struct StepOut {
  int32_t *history, *hist_len;
  uint32_t* draws;
  int32_t* token;
  float *logprob, *lse;
  int32_t* top_idx;
  float* top_val;
  int32_t *feedback, *pos_inc;
  int hist_cap;
};
struct Sequence {
  int len, pos;
  uint32_t drawn;
};
__device__ __forceinline__ Sequence request_sequence(const StepOut& o, int row) {
  return {o.history && o.hist_len ? o.hist_len[row] : 0, o.pos_inc ? o.pos_inc[row] : 0, o.draws ? o.draws[row] : 0u};
}
// (one thread)
__device__ __forceinline__ void write_step(const StepOut& o, const Sequence& seq, int row, int tok, float x, float lse, bool draw) {
  o.token[row] = tok;
  if (o.logprob) o.logprob[row] = x - lse;
  if (o.lse) o.lse[row] = lse;
  if (o.feedback) o.feedback[row] = tok;
  if (o.history && o.hist_len) {
    o.history[(size_t)row * o.hist_cap + seq.len % o.hist_cap] = tok;
    o.hist_len[row] = seq.len + 1;
  }
  if (o.draws && draw) o.draws[row] = seq.drawn + 1;
  if (o.pos_inc) o.pos_inc[row] = seq.pos + 1;
}

// Rows that are neither drawn nor listed: the largest value.
__global__ __launch_bounds__(64) void sample_greedy_kernel(const StepOut o, const void* ws, int V) {
  const int row = blockIdx.x;
  const Partial part = request_partial(row_ws(const_cast<void*>(ws), row));
  const Sequence seq = request_sequence(o, row);
  float mx, lse;
  int mi;
  merge_stats(part, mx, mi, lse);
  if (threadIdx.x == 0) write_step(o, seq, row, min(max(mi, 0), V - 1), mx, lse, false);
}

template <int NU>
__global__ __launch_bounds__(256) void sample_select_kernel(
    const bf16_t* __restrict__ logits, const exo_sampler_params* __restrict__ params, const StepOut out, void* ws, int V,
    int has_edits, int has_tables, int want_top) {
  __shared__ EditLds ed;
  __shared__ float s_wsum[4], s_rem;
  __shared__ int s_block, s_tok, s_last[4];
  __shared__ float s_x;
  const int row = blockIdx.x, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  RowWs* w = row_ws(ws, row);
  // everything that does not depend on the slice of the draw is requested here
  const float4 stat = *reinterpret_cast<const float4*>(&w->part[lane][0]);
  const int n_edit = has_edits ? w->n_edit : 0;
  const float table_thr = w->thr;
  const int key_top = w->key_top, cand_n = w->cand_n;
  const u64 my_cand = lane < kMaxCand ? w->cand[lane] : 0ull;
  const int my_ties = w->tie_n[lane];
  const Sequence seq = request_sequence(out, row);
  const exo_sampler_params p = params[row];
  if (has_tables && row_needs_table(p, want_top != 0)) {  // the weights launch was the fine tables' last reader
    Tables* T = row_tables(ws, row);
    for (int i = tid; i < kTargets * kFine; i += 256) (&T->fine[0][0])[i] = 0;
  }
  float mx, lse;
  int mi;
  merge_stats({stat.x, stat.z, __float_as_int(stat.y)}, mx, mi, lse);
  const bool draw = p.temperature != 0.f;
  SliceGeom g = {};
  Share<NU> sh;
  if (draw) {
    if (wave == 0) {
      // the slice in which the running sum of kept weights crosses u * total (slices in order, sums in float32,
      // the same order every time): a lane holds its slice's sum and what runs up to it
      const float wb = stat.w;
      float total = 0.f, run = 0.f;
#pragma unroll
      for (int b = 0; b < kBlocks; ++b) {
        if (lane == b) run = total;
        total += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wb), b));
      }
      uint32_t c[4] = {seq.drawn, 0u, 0u, 0u};
      philox4x32_10(c, p.seed_lo, p.seed_hi);
      const float u = (float)(c[0] >> 8) * 0x1p-24f;
      const float target = u * total;
      const u64 kept = __ballot(wb > 0.f), hit = __ballot(wb > 0.f && run + wb > target);
      // (no slice: rounding at the very end of the distribution)
      const int blk = hit ? __ffsll((long long)hit) - 1 : kept ? 63 - __clzll((long long)kept) : 0;
      if (lane == blk) {
        s_block = blk;
        s_rem = hit ? target - run : INFINITY;
        s_tok = -1;
      }
    }
    __syncthreads();
    g = slice_geom(logits, V, s_block);
    request_share(logits + (size_t)row * V, g, sh);
  }
  if (want_top) {
    // (while the slice is on its way) the tokens strictly above the 20th largest value, ranked: higher key first,
    // lower index first among equals; then the tokens equal to it, lowest ids first (slices in order)
    const int n = min(cand_n, kTop - 1);
    if (wave == 2) {
      const u64 me = lane < n ? my_cand : 0ull;
      const unsigned int mk = (unsigned int)(me >> 32), mi2 = (unsigned int)me;
      int rank = 0;
#pragma unroll
      for (int o = 0; o < kTop - 1; ++o) {
        const unsigned int ok = (unsigned int)__builtin_amdgcn_readlane((int)mk, o);
        const unsigned int oi = (unsigned int)__builtin_amdgcn_readlane((int)mi2, o);
        rank += o < n && (ok > mk || (ok == mk && oi < mi2)) ? 1 : 0;
      }
      if (lane < n) {
        out.top_idx[(size_t)row * kTop + rank] = (int)mi2;
        out.top_val[(size_t)row * kTop + rank] = value_of((int)mk) - lse;
      }
    }
    if (wave == 3) {  // a lane per slice: its ties go behind those of the slices before it
      const int inc = wave_scan_i32(my_ties);
      const float tv = value_of(key_top) - lse;
      const int first = n + inc - my_ties;
      for (int j = 0; j < my_ties && first + j < kTop; ++j) {
        out.top_idx[(size_t)row * kTop + first + j] = w->tie_idx[lane][j];
        out.top_val[(size_t)row * kTop + first + j] = tv;
      }
      // vocabularies of fewer than 20 tokens
      const int all = n + __builtin_amdgcn_readlane(inc, 63);
      if (lane >= all && lane < kTop) {
        out.top_idx[(size_t)row * kTop + lane] = -1;
        out.top_val[(size_t)row * kTop + lane] = -INFINITY;
      }
    }
  }
  int tok = mi;
  float x_tok = mx;
  if (draw) {
    stage_edits(w, g, n_edit, ed);
    float xv[8 * NU];
    expand_share(sh, g, n_edit, ed, xv);
    const float thr = keep_threshold(p, table_thr, mx);
    const float inv_t = 1.f / p.temperature;
    float rem = s_rem;
    int last_kept = -1;  // of this thread's tokens
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      // chunk u of every thread, in thread order = vocabulary order
      float wk[8], local = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        wk[k] = (xv[8 * u + k] >= thr) ? expf((xv[8 * u + k] - mx) * inv_t) : 0.f;
        local += wk[k];
        if (wk[k] > 0.f) last_kept = sh.i0[u] + k;
      }
      // inclusive scan of `local` over the 256 threads; the intervals [excl, incl) of
      // consecutive threads tile the line exactly (excl is the neighbour's incl, bit for bit)
      float inc = local;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const float up = __shfl_up(inc, o, 64);
        if (lane >= o) inc += up;
      }
      const float prev = __shfl_up(inc, 1, 64);
      if (lane == 63) s_wsum[wave] = inc;
      __syncthreads();
      float before = 0.f;
      for (int wv = 0; wv < wave; ++wv) before += s_wsum[wv];
      const float round_total = ((s_wsum[0] + s_wsum[1]) + s_wsum[2]) + s_wsum[3];
      const float excl = lane > 0 ? before + prev : before;
      const float incl = before + inc;
      if (excl <= rem && rem < incl) {  // exactly one thread
        float run = excl;
        int sel = -1, last = -1;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          if (wk[k] > 0.f) {
            last = k;
            if (sel < 0 && run + wk[k] > rem) sel = k;
          }
          run += wk[k];
        }
        if (sel < 0) sel = last;  // the in-thread sum rounds differently from the scan
        if (sel >= 0) {
          s_tok = sh.i0[u] + sel;
          float xs = 0.f;
#pragma unroll
          for (int k = 0; k < 8; ++k)
            if (k == sel) xs = xv[8 * u + k];
          s_x = xs;
        }
      }
      __syncthreads();
      if (s_tok >= 0) break;
      rem -= round_total;
    }
    if (s_tok < 0) {  // float32 rounding put the target past the last kept token (uniform over the workgroup)
      const int last = (int)wave_max_u32((uint32_t)(last_kept + 1)) - 1;
      if (lane == 0) s_last[wave] = last;
      __syncthreads();
      const int lk = max(max(s_last[0], s_last[1]), max(s_last[2], s_last[3]));
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (sh.i0[u] + k == lk) {
            s_tok = lk;
            s_x = xv[8 * u + k];
          }
      __syncthreads();
    }
    tok = s_tok;
    x_tok = s_x;
    if (tok < 0 || tok >= V) {  // no token was kept (min_p above 1, logits that are not numbers)
      tok = mi;
      x_tok = mx;
    }
  }
  if (tid == 0) write_step(out, seq, row, min(max(tok, 0), V - 1), x_tok, lse, draw);
}

// The launches of a step, for slices of one or two chunks a thread.
template <int NU>
void launch_sample(const bf16_t* lg, const exo_sampler_params* params, const StepOut& out, void* ws, int rows, int V, int mode, hipStream_t st) {
  const int edits = mode & EXO_SAMPLE_EDITS ? 1 : 0, top = mode & EXO_SAMPLE_TOP ? 1 : 0;
  const int tables = mode & (EXO_SAMPLE_TABLE | EXO_SAMPLE_TOP) ? 1 : 0;
  const dim3 slices(kBlocks, rows);
  if (edits) sampler_edits_kernel<<<dim3(rows), 512, 0, st>>>(lg, params, out.history, out.hist_len, ws, V, out.hist_cap);
  sample_stats_kernel<NU><<<slices, 256, 0, st>>>(lg, ws, V, edits);
  if (tables) {
    sample_coarse_kernel<NU><<<slices, 256, 0, st>>>(lg, params, ws, V, edits, top);
    sample_fine_kernel<NU><<<slices, 256, 0, st>>>(lg, params, ws, V, edits, top);
  }
  // (the weights launch also resolves and clears the tables: it runs whenever they were filled)
  if (tables || (mode & EXO_SAMPLE_DRAW)) {
    sample_weights_kernel<NU><<<slices, 256, 0, st>>>(lg, params, ws, V, edits, tables, top);
    sample_select_kernel<NU><<<dim3(rows), 256, 0, st>>>(lg, params, out, ws, V, edits, tables, top);
  } else {
    sample_greedy_kernel<<<dim3(rows), 64, 0, st>>>(out, ws, V);
  }
}

}  // namespace

extern "C" int64_t exo_sample_workspace(int rows) {
  if (rows <= 0) return 0;
  return (int64_t)rows * (int64_t)kRowStride;
}

extern "C" int exo_sample(const uint16_t* logits, const exo_sampler_params* params,
                          int32_t* history, int32_t* hist_len, uint32_t* draws, int32_t* token,
                          float* logprob, float* lse, int32_t* top_idx, float* top_val,
                          int32_t* feedback, int32_t* pos_inc, void* workspace,
                          int64_t workspace_bytes, int rows, int V, int hist_cap, int mode,
                          exo_stream_t stream) {
  EXO_REQUIRE(rows >= 0 && rows <= 65535 && V > 0, "exo_sample: bad size rows=%d V=%d", rows, V);
  EXO_REQUIRE(V <= kBlocks * kMaxSlice, "exo_sample: V=%d exceeds %d", V, kBlocks * kMaxSlice);
  EXO_REQUIRE(hist_cap >= 0 && hist_cap <= EXO_SAMPLER_MAX_CONTEXT,
              "exo_sample: hist_cap=%d outside [0,%d]", hist_cap, EXO_SAMPLER_MAX_CONTEXT);
  EXO_REQUIRE((mode & ~(EXO_SAMPLE_EDITS | EXO_SAMPLE_DRAW | EXO_SAMPLE_TABLE | EXO_SAMPLE_TOP)) == 0,
              "exo_sample: unknown mode bits 0x%x", mode);
  EXO_REQUIRE(logits && params && token && workspace, "exo_sample: null pointer");
  EXO_REQUIRE(workspace_bytes >= exo_sample_workspace(rows) && ((uintptr_t)workspace & 255) == 0,
              "exo_sample: workspace of %lld bytes, need %lld (256-byte aligned)",
              (long long)workspace_bytes, (long long)exo_sample_workspace(rows));
  const bool edits = mode & EXO_SAMPLE_EDITS, want_top = mode & EXO_SAMPLE_TOP;
  EXO_REQUIRE(!edits || hist_cap == 0 || (history && hist_len),
              "exo_sample: the penalty processors need the history ring");
  EXO_REQUIRE(!history || hist_cap > 0, "exo_sample: a history ring of zero entries (hist_cap=0)");
  EXO_REQUIRE(!want_top || (top_idx && top_val), "exo_sample: top-logprob outputs missing");
  EXO_REQUIRE(!(mode & EXO_SAMPLE_DRAW) || draws, "exo_sample: draw counters missing");
  if (rows == 0) return EXO_OK;
  const auto launch = slice_elements(V) <= 2048 ? launch_sample<1> : launch_sample<2>;
  const StepOut out = {history, hist_len, draws, token, logprob, lse, top_idx, top_val, feedback, pos_inc, hist_cap > 0 ? hist_cap : 1};
  launch(logits, params, out, workspace, rows, V, mode, (hipStream_t)stream);
  EXO_CHECK_LAUNCH("exo_sample");
  return EXO_OK;
}
