// Attention over a paged KV pool, for batches that mix portions of prompts with single decoded
// tokens.  Options, each a parameter of the layer: unit-RMS queries and keys (with a gain per
// channel), per head or over the whole projection, rotary positions (interleaved pairs), scores bent
// to cap * tanh(score / cap), values mixed with another layer's values of the token, a gate per head on
// the output (sigmoid of a given number) or per channel, a per-head linear distance penalty, a sliding window
// with kept first tokens or with the means of whole blocks of positions past it, a softmax with one more in its
// sum, sigmoid weights that are not divided by their sum, a causal convolution over projected queries and keys,
// values that are the keys ahead of their rotation, value size other than key size, keys and values of another layer.
// Scores, penalty, weights and sums are float32; where the weights enter a bf16 matrix product they go in as two bf16 terms (high and remainder), so that they keep
// 16 bits.
//
// Pool layout (page = 64 positions of one sequence, all kv heads):
//   keys    [page][G][64][ldk]   a position's key, already normalised
//   values  [page][G][ldv][64]   TRANSPOSED: a value column's 64 positions in one run
// With the values transposed both operands of both products are rows of memory in matrix-core
// operand order; nothing is transposed on the way.  ldk, ldv are multiples of 32 and the padding is
// zero, so any key / value size is taken.
// Means of blocks lie in pools of the same layout (a page: 64 blocks) behind a table of their own.  They are
// tiles like any other in front of the window's; a block's mean is formed from the pool when its last position
// has been stored (paged_rows_kernel for a step of single tokens, else paged_means_kernel).
//
// paged_rows_kernel: one query position per workgroup row (decode; also the 32-bit mode's prompts).
//   The up to 16 query heads of a kv head are the 16 columns of 16x16 products:
//     S^T[key][head] = K . Q^T,   O^T[d][head] += V^T . P^T
//   Each wave walks tiles of 32 keys, dealt out round robin over the waves of all splits; only the
//   tiles that hold a visible key are dealt (kept first tokens, then the window).  Splits meet
//   through device-scope partials and an arrival counter.  FUSE: the launch also normalises and
//   stores the row's own key and value (the workgroup that owns the last tile does).
//   What bounds a launch of short contexts is a chain of ways through memory by a few waves: the arguments, position and slot, the page, the
//   tile, the partials, their counter and the partials again.  So the arguments come in one way, a row's channels with its position (plain
//   ones 16 bytes a thread, not element by element), the page of a wave's first tile behind that, and partials in requests of up to
//   16 bytes, a thread to every run of columns.  Launches of a graph, four rows of 32 / 4 heads of 128 with normed queries: 17 | 150 | 700 keys 8.1 | 10.8 | 11.7 ->
//   6.9 | 10.1 | 11.2 us (48 keys of 64 in float32, one split: 6.55 -> 6.45).
// paged_prepare_kernel: norm over whole projections, rotation and value mixing of all rows of a step
//   ahead of the other two (queries in place, keys and values into the pool); a step of single tokens
//   does the same inside paged_rows_kernel.  Convolved queries go to a buffer of their own, since other rows
//   still read the projected ones; a sequence's latest projections stay in a ring (position p at p % taps), which
//   paged_keep_kernel writes behind that launch.
// paged_prompt_kernel: 32 query positions of one head per wave, four such units of one kv head and
//   one sequence per workgroup sharing page-sized key tiles through LDS (two buffers, the next tile
//   in registers meanwhile); 32x32 products, transposed like above so that running maximum, sum and
//   rescale factor are per-lane scalars.
#include <type_traits>

#include "../../include/exo_mi355x.h"
#include "dense.h"
#include "rotary.h"

namespace {

constexpr int kPage = 64;
constexpr int kCounters = 16384;  // arrival counters at the start of the workspace
constexpr float kLog2e = 1.4426950408889634f;

struct Params {
  const void* qkv;      // T [R][ldq]: q heads, then (own keys) k heads, v heads
  void* kpool;
  void* vpool;
  const int32_t* table; // [slots][max_pages]
  const int32_t* slot;  // [R]
  const int32_t* pos;   // [R]
  const int32_t* list;  // rows: row indices (null: all); prompt: blocks of {row, slot, pos, n}
  const float* slopes;  // [H], or null
  const float* qgain;   // [D] (whole: [H * D]), or null
  const float* kgain;   // [D] (whole: [G * D]), or null
  const double* freq;   // [rot / 2] turns per position
  const void* vmix;     // T [R][ldmix] values mixed in, or null
  const float* gate;    // [R][ldg] a number per head, or null
  const void* ogate;    // T [R][ldog] a number per output, or null
  const float* wbias;   // [H] added to the score of sigmoid weights, or null
  void* mkpool;         // means of blocks of `pool` positions
  void* mvpool;
  const int32_t* mtable;  // [slots][mpages]
  const float* convw;   // [taps][(H + G) * D], or null
  void* ring;           // T [states][taps][(H + G) * D]
  const int32_t* map;   // slot -> state
  void* qout;           // T [R][ldqo] prepared queries (null: in place)
  void* out;            // T [R][ldo]
  float* ws;
  int* counters;
  float scale, eps, cap, mix;  // cap 0: none
  int n, H, G, D, E, ldq, ldk, ldv, ldo, ldg, ldmix, max_pages, size, keep, unit, whole, rot, nsplit, gsz, hgroups, group;  // (the last four: of the rows' launch)
  int ldog, ldqo, mpages, pool, one, half, taps, vkeys;  // pool 0, taps 0: none; vkeys: values are keys
  float amp;
};
// expanded latent keys and values (latent_attn.hip) in place of the pool: rows of a sequence from its
// block's second entry on
struct Expanded {
  const bf16_t* k;      // [keys][ldk]: head h's d8 entries at h * d8
  const bf16_t* kr;     // [keys][r8]: shared by the heads
  const bf16_t* v;      // [heads * E][ldv]: positions in a run
  int ldk, ldv, d8, r8, qs, rot_col;  // queries: head h's at h * qs, its rotated part at rot_col + h * r8
};
constexpr int kMaxRot = 256;

// Which options an instance of the attention kernels has: kPlain leaves out what few designs need (means of
// blocks, convolution, gates per channel, one more in the sum, rotation by halves, values that are keys).
enum Mode { kPlain, kMore, kSigmoid };
int mode_of(const Params& p) {
  return p.wbias ? kSigmoid : p.pool || p.taps || p.ogate || p.one || p.half || p.vkeys || p.amp != 1.f ? kMore : kPlain;
}
template <int MODE>
__device__ __forceinline__ Params only(Params p) {
  if (MODE == kPlain) p.pool = p.taps = p.one = p.half = p.vkeys = 0, p.ogate = nullptr, p.amp = 1.f;
  return p;
}

// W floats at a multiple of four bytes, written and read at device scope in one request
constexpr int kDeviceScope = 16;  // (the sc1 bit)
template <int W>
struct alignas(W * 4) Run {
  float v[W];
};
template <int W>
__device__ __forceinline__ void st_dev(__amdgpu_buffer_rsrc_t to, uint32_t voff, uint32_t soff, const Run<W>& r) {
  if constexpr (W == 4)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, r), to, voff, soff, kDeviceScope);
  else if constexpr (W == 2)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, r), to, voff, soff, kDeviceScope);
  else
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, r), to, voff, soff, kDeviceScope);
}
template <int W>
__device__ __forceinline__ Run<W> ld_dev(__amdgpu_buffer_rsrc_t from, uint32_t voff, uint32_t soff) {
  if constexpr (W == 4)
    return __builtin_bit_cast(Run<W>, __builtin_amdgcn_raw_buffer_load_b128(from, voff, soff, kDeviceScope));
  else if constexpr (W == 2)
    return __builtin_bit_cast(Run<W>, __builtin_amdgcn_raw_buffer_load_b64(from, voff, soff, kDeviceScope));
  else
    return __builtin_bit_cast(Run<W>, __builtin_amdgcn_raw_buffer_load_b32(from, voff, soff, kDeviceScope));
}

// whole blocks that lie before the window of a query at pos
__device__ __forceinline__ int blocks_seen(const Params& p, int pos) { return p.pool ? max(0, pos - p.size + 1) / p.pool : 0; }

// key tiles of `tile` positions that hold a key visible to a query in [first, last]: means of blocks, tiles
// 0 .. means - 1 of their own pool; then the kept ones, then those from w0 on
struct Tiles {
  int means, sink, w0, n;
  __device__ __forceinline__ bool mean(int j) const { return means > 0 && j < means; }
  __device__ __forceinline__ int at(int j) const {
    const int i = j - means;
    return mean(j) ? j : i < sink ? i : w0 + (i - sink);
  }
};
__device__ __forceinline__ Tiles tiles_of(const Params& p, int first, int last, int tile) {
  Tiles t;
  t.means = (blocks_seen(p, last) + tile - 1) / tile;
  t.sink = (min(p.keep, last + 1) + tile - 1) / tile;
  const int lo = max(0, first - p.size + 1);
  t.w0 = max(lo / tile, t.sink);
  t.n = t.means + t.sink + max(0, last / tile + 1 - t.w0);
  return t;
}

// what a head's output is multiplied with
__device__ __forceinline__ float head_gate(const Params& p, int row, int h) {
  return p.gate ? 1.f / (1.f + expf(-p.gate[(size_t)row * p.ldg + h])) : 1.f;
}
// ... and one of its columns
template <typename T>
__device__ __forceinline__ float column_gate(const Params& p, int row, int c) {
  return p.ogate ? 1.f / (1.f + expf(-Elem<T>::load(reinterpret_cast<const T*>(p.ogate)[(size_t)row * p.ldog + c]))) : 1.f;
}

// one wave: src[0..D) / rms * gain -> dst (element type T, float32 arithmetic), in two steps: what it needs is requested, and much later
// turned into the row
template <typename T, int DMAX>
struct UnitRow {
  T x[DMAX / 64];
  __device__ __forceinline__ void request(const T* __restrict__ src, int D, int lane) {
#pragma unroll
    for (int i = 0; i < DMAX / 64; ++i)
      if (lane + 64 * i < D) x[i] = src[lane + 64 * i];
  }
  __device__ __forceinline__ void put(T* dst, int D, int unit, float eps, const float* __restrict__ gain, int lane) const {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < DMAX / 64; ++i)
      if (lane + 64 * i < D) {
        const float v = Elem<T>::load(x[i]);
        ss += v * v;
      }
    const float inv = unit ? 1.f / sqrtf(wave_total(ss) / D + eps) : 1.f;
#pragma unroll
    for (int i = 0; i < DMAX / 64; ++i)
      if (lane + 64 * i < D) dst[lane + 64 * i] = Elem<T>::make(Elem<T>::load(x[i]) * inv * (gain ? gain[lane + 64 * i] : 1.f));
  }
};

// this thread's share (of `threads`) of the sum of squares of src[0..n); vec: in vectors
template <typename T>
__device__ __forceinline__ float square_sum(const T* src, int n, bool vec, int thread, int threads) {
  constexpr int VEC = Elem<T>::kVec;
  float ss = 0.f;
  if (vec) {
    for (int c = thread * VEC; c < n; c += threads * VEC) {
      float f[VEC];
      unpack_vec<T>(load16(src + c), f);
#pragma unroll
      for (int e = 0; e < VEC; ++e) ss += f[e] * f[e];
    }
  } else {
    for (int c = thread; c < n; c += threads) ss += Elem<T>::load(src[c]) * Elem<T>::load(src[c]);
  }
  return ss;
}
// cap * tanh(x) as 1 - 2 / (e^2x + 1): an absolute error of some 1e-7 cap, for scores of bf16 operands
__device__ __forceinline__ float bent(float x, float cap) {
  return cap - 2.f * cap * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x * (2.f * kLog2e)) + 1.f);
}

// A row's projected queries and keys, channel by channel, behind the convolution if there is one.  The inputs
// of the `run` rows ahead belong to the same sequence; what lies before them is in the ring.
template <typename T>
struct Channels {
  static constexpr int VEC = Elem<T>::kVec;
  const T *raw, *ring;
  const float* w;
  int ldq, taps, channels, run, pos;
  __device__ __forceinline__ Channels(const Params& p, int row, int pos_, int slot, int run_) : run(run_), pos(pos_) {
    raw = reinterpret_cast<const T*>(p.qkv) + (size_t)row * p.ldq;
    taps = p.taps, channels = (p.H + p.G) * p.D, ldq = p.ldq, w = p.convw;
    ring = taps ? reinterpret_cast<const T*>(p.ring) + (size_t)p.map[slot] * taps * channels : nullptr;
  }
  // the input `back` positions earlier (one that exists)
  __device__ __forceinline__ const T* input(int back) const {
    return back <= run ? raw - (ptrdiff_t)back * ldq : ring + (size_t)((pos - back) % taps) * channels;
  }
  __device__ __forceinline__ float at(int c) const {
    if (!taps) return Elem<T>::load(raw[c]);
    float y = 0.f;
    const int last = min(taps - 1, pos);
    for (int b0 = 0; b0 <= last; b0 += 4) {  // four requests together
      float x[4], u[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int b = min(b0 + i, last);
        x[i] = Elem<T>::load(input(b)[c]);
        u[i] = w[(size_t)(taps - 1 - b) * channels + c];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) y = b0 + i <= last ? fmaf(u[i], x[i], y) : y;
    }
    return y;
  }
  __device__ __forceinline__ void vec(int c, float (&f)[VEC]) const {
    if (!taps) {
      unpack_vec<T>(load16(raw + c), f);
      return;
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) f[e] = 0.f;
    const int last = min(taps - 1, pos);
    for (int b0 = 0; b0 <= last; b0 += 4) {  // four requests together
      uint4 in[4];
      floatx4 u[4][VEC / 4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int b = min(b0 + i, last);
        in[i] = load16(input(b) + c);
        const float* wc = w + (size_t)(taps - 1 - b) * channels + c;
#pragma unroll
        for (int e = 0; e < VEC / 4; ++e) u[i][e] = *reinterpret_cast<const floatx4*>(wc + 4 * e);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (b0 + i > last) break;
        float x[VEC];
        unpack_vec<T>(in[i], x);
#pragma unroll
        for (int e = 0; e < VEC; ++e) f[e] = fmaf(u[i][e / 4][e % 4], x[e], f[e]);
      }
    }
  }
};
// this thread's share of the channels [c0, c0 + n) into the ring (a step of single tokens)
template <typename T>
__device__ __forceinline__ void keep_channels(const Channels<T>& x, int c0, int n, int thread, int threads) {
  T* dst = const_cast<T*>(x.ring) + (size_t)(x.pos % x.taps) * x.channels;
  for (int c = c0 + thread; c < c0 + n; c += threads) dst[c] = x.raw[c];
}

// one wave: the channels [c0, c0 + D) times inv and gain, the first p.rot of them turned -> dst (may be their place);
// the channels themselves -> plain, if it is given
template <typename T>
__device__ __forceinline__ void turn_row(const Params& p, const Channels<T>& x, int c0, T* dst, float inv,
                                         const float* __restrict__ gain, const float2* cs, int lane, T* plain = nullptr) {
  const int D = p.D, half = p.half ? p.rot / 2 : 0;  // pairs (i, i + half) below 2 half, pairs (2i, 2i + 1) behind them
  for (int i = lane; 2 * i < D; i += 64) {
    const int a = i < half ? i : 2 * i, b = i < half ? i + half : 2 * i + 1;
    const bool two = b < D;
    float2 v{x.at(c0 + a) * inv, two ? x.at(c0 + b) * inv : 0.f};
    if (plain) {
      plain[a] = Elem<T>::make(v.x);
      if (two) plain[b] = Elem<T>::make(v.y);
    }
    if (gain) v.x *= gain[a], v.y *= two ? gain[b] : 0.f;
    if (2 * i < p.rot) v = turn_pair(v.x, v.y, cs[i]);
    dst[a] = Elem<T>::make(v.x);
    if (two) dst[b] = Elem<T>::make(v.y);
  }
}
// the token's value column, mixed with the other layer's
template <typename T>
__device__ __forceinline__ T mixed_value(const Params& p, T v, int row, int c) {
  if (!p.vmix) return v;
  const float o = Elem<T>::load(reinterpret_cast<const T*>(p.vmix)[(size_t)row * p.ldmix + c]);
  return Elem<T>::make((1.f - p.mix) * Elem<T>::load(v) + p.mix * o);
}

// key (turned) and value of one (row, kv head) to their places in the pool, by one wave each
template <typename T>
__device__ __forceinline__ void put_key(const Params& p, const Channels<T>& x, int g, T* dst, int lane, float inv, const float2* cs) {
  const int c0 = (p.H + g) * p.D;
  turn_row<T>(p, x, c0, dst, inv, p.kgain ? p.kgain + g * p.D : nullptr, cs, lane);
  if (p.taps) keep_channels<T>(x, c0, p.D, lane, 64);
}
template <typename T>
__device__ __forceinline__ void put_value(const Params& p, const Channels<T>& x, int row, int g, T* dst, int lane) {
  if (p.vkeys) {
    for (int d = lane; d < p.E; d += 64) dst[(size_t)d * kPage] = Elem<T>::make(x.at((p.H + g) * p.D + d));
    return;
  }
  const T* src = x.raw + (p.H + p.G) * p.D + g * p.E;
  for (int d = lane; d < p.E; d += 64) dst[(size_t)d * kPage] = mixed_value<T>(p, src[d], row, g * p.E + d);
}

// means of the keys and values of one kv head over a block whose positions are all stored, by `threads` threads
template <typename T>
__device__ __forceinline__ void put_means(const Params& p, int slot, int block, int g, int thread, int threads) {
  const int32_t* table = p.table + (size_t)slot * p.max_pages;
  const size_t page = p.mtable[(size_t)slot * p.mpages + block / kPage];
  const int at = block % kPage, first = block * p.pool;
  const float inv = 1.f / p.pool;
  for (int c = thread; c < p.D + p.E; c += threads) {
    const bool key = c < p.D;
    const int d = key ? c : c - p.D;
    float sum = 0.f;
    for (int t0 = 0; t0 < p.pool; t0 += 8) {  // eight requests together
      T v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int t = first + min(t0 + i, p.pool - 1), in = t % kPage;
        const size_t head = (size_t)table[t / kPage] * p.G + g;
        v[i] = key ? reinterpret_cast<const T*>(p.kpool)[(head * kPage + in) * p.ldk + d]
                   : reinterpret_cast<const T*>(p.vpool)[(head * p.ldv + d) * kPage + in];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) sum += t0 + i < p.pool ? Elem<T>::load(v[i]) : 0.f;
    }
    const size_t head = page * p.G + g;
    if (key)
      reinterpret_cast<T*>(p.mkpool)[(head * kPage + at) * p.ldk + d] = Elem<T>::make(sum * inv);
    else
      reinterpret_cast<T*>(p.mvpool)[(head * p.ldv + d) * kPage + at] = Elem<T>::make(sum * inv);
  }
}
// list: {slot, block}
template <typename T>
__global__ __launch_bounds__(256) void paged_means_kernel(const Params p) {
  const int32_t* b = p.list + 2 * (size_t)blockIdx.x;
  put_means<T>(p, b[0], b[1], blockIdx.y, threadIdx.x, 256);
}

// the last `taps` rows of each sequence of a step into its ring; the workgroups of blockIdx.x look through 64 rows
// and share those that they find, blockIdx.z their channels
constexpr int kKeepers = 4, kKept = 1024;
template <typename T>
__global__ __launch_bounds__(256) void paged_keep_kernel(const Params p) {
  const int row0 = blockIdx.x * 64, row = row0 + (threadIdx.x & 63), behind = row + p.taps;
  const bool tail = row < p.n && (behind >= p.n || p.slot[min(behind, p.n - 1)] != p.slot[min(row, p.n - 1)]);
  int i = 0;
  for (uint64_t left = __ballot(tail); left; left &= left - 1, ++i) {
    if (i % kKeepers != (int)blockIdx.y) continue;
    const int r = row0 + __builtin_ctzll(left);
    const Channels<T> x(p, r, p.pos[r], p.slot[r], 0);
    const int c0 = blockIdx.z * kKept;
    keep_channels<T>(x, c0, min(kKept, x.channels - c0), threadIdx.x, 256);
  }
}

// A wave takes eight rows of one head: the keys' loads go out together, and the values of eight
// consecutive positions of one page leave as one 16-byte (bf16) store per column - element by
// element they would be eight stores that touch a line each.
constexpr int kAppendRows = 8;

template <typename T>
__global__ __launch_bounds__(256) void paged_append_kernel(const Params p) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int row0 = blockIdx.x * kAppendRows, unit = blockIdx.y * 4 + wave;  // units: keys of G heads, values of G heads
  if (unit >= 2 * p.G) return;
  const int n = min(kAppendRows, p.n - row0);
  const int lr = row0 + min(lane, n - 1);  // lane i < n: row i's place
  const int my_pos = p.pos[lr], my_slot = p.slot[lr];
  const int my_page = p.table[(size_t)my_slot * p.max_pages + my_pos / kPage];
  if (unit < p.G) {
    const T* src = reinterpret_cast<const T*>(p.qkv) + (size_t)row0 * p.ldq + p.H * p.D + unit * p.D;
    constexpr int VEC = Elem<T>::kVec;
    if (p.D % VEC == 0 && p.ldq % VEC == 0) {  // 16 bytes per lane, several rows per pass
      int lpr = 1;  // lanes per row
      while (lpr * VEC < p.D) lpr *= 2;
      const int c = lane % lpr;
      for (int i0 = 0; i0 < n; i0 += 64 / lpr) {
        const int i = i0 + lane / lpr, ic = min(i, n - 1);
        const bool on = c * VEC < p.D;
        const uint4 raw = on ? *reinterpret_cast<const uint4*>(src + (size_t)ic * p.ldq + c * VEC) : uint4{0, 0, 0, 0};
        float f[VEC], ss = 0.f;
        unpack_vec<T>(raw, f);
#pragma unroll
        for (int e = 0; e < VEC; ++e) ss += f[e] * f[e];
        const float inv = p.unit ? 1.f / sqrtf(group_sum(ss, lpr) / p.D + p.eps) : 1.f;
        const int page = __shfl(my_page, ic, 64), at = __shfl(my_pos, ic, 64) % kPage;
        struct alignas(16) Vec {
          T e[VEC];
        } w;
#pragma unroll
        for (int e = 0; e < VEC; ++e) w.e[e] = Elem<T>::make(f[e] * inv * (p.kgain && on ? p.kgain[c * VEC + e] : 1.f));
        if (on && i < n)
          *reinterpret_cast<uint4*>(reinterpret_cast<T*>(p.kpool) + (((size_t)page * p.G + unit) * kPage + at) * p.ldk +
                                    c * VEC) = __builtin_bit_cast(uint4, w);
      }
      return;
    }
    float v[kAppendRows][4];  // D <= 256
#pragma unroll
    for (int i = 0; i < kAppendRows; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = lane + 64 * j;
        v[i][j] = d < p.D ? Elem<T>::load(src[(size_t)min(i, n - 1) * p.ldq + d]) : 0.f;
      }
#pragma unroll
    for (int i = 0; i < kAppendRows; ++i) {
      if (i >= n) break;
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) ss += v[i][j] * v[i][j];
      const float inv = p.unit ? 1.f / sqrtf(wave_sum(ss) / p.D + p.eps) : 1.f;
      const int page = __builtin_amdgcn_readlane(my_page, i), at = __builtin_amdgcn_readlane(my_pos, i) % kPage;
      T* dst = reinterpret_cast<T*>(p.kpool) + (((size_t)page * p.G + unit) * kPage + at) * p.ldk;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (lane + 64 * j < p.D) dst[lane + 64 * j] = Elem<T>::make(v[i][j] * inv * (p.kgain ? p.kgain[lane + 64 * j] : 1.f));
    }
    return;
  }
  const int g = unit - p.G;
  const T* src = reinterpret_cast<const T*>(p.qkv) + (size_t)row0 * p.ldq + (p.H + p.G) * p.D + g * p.E;
  const int pos0 = __builtin_amdgcn_readfirstlane(my_pos), page0 = __builtin_amdgcn_readfirstlane(my_page);
  const bool run = n == kAppendRows && pos0 % kAppendRows == 0 &&
                   __ballot(lane < kAppendRows && (my_page != page0 || my_pos != pos0 + lane)) == 0;
  for (int d = lane; d < p.E; d += 64) {
    T v[kAppendRows];
#pragma unroll
    for (int i = 0; i < kAppendRows; ++i) v[i] = src[(size_t)min(i, n - 1) * p.ldq + d];
    if (run) {
      T* dst = reinterpret_cast<T*>(p.vpool) + (((size_t)page0 * p.G + g) * p.ldv + d) * kPage + pos0 % kPage;
      constexpr int per = 16 / (int)sizeof(T);
#pragma unroll
      for (int k = 0; k < kAppendRows; k += per) {
        struct alignas(16) Vec {
          T e[per];
        } w;
#pragma unroll
        for (int i = 0; i < per; ++i) w.e[i] = v[k + i];
        *reinterpret_cast<uint4*>(dst + k) = __builtin_bit_cast(uint4, w);
      }
    } else {
#pragma unroll
      for (int i = 0; i < kAppendRows; ++i) {
        if (i >= n) break;
        const int page = __builtin_amdgcn_readlane(my_page, i), at = __builtin_amdgcn_readlane(my_pos, i) % kPage;
        reinterpret_cast<T*>(p.vpool)[(((size_t)page * p.G + g) * p.ldv + d) * kPage + at] = v[i];
      }
    }
  }
}

// Norm over whole projections, rotation and value mixing of eight rows, a wave each.  blockIdx.y 0: the keys, then
// the values of all kv heads, eight positions of a column per store where they lie in one run; the others: the
// queries, dealt out by heads, which stay in qkv or go to qout.
// c0: the first channel of a run of heads; plain: turn_row.
template <typename T>
__device__ __forceinline__ void prepare_run(const Params& p, const Channels<T>& x, int c0, T* dst, int ldd, int heads, float inv,
                                            const float* gain, const float2* cs, bool vec, int lane, T* plain = nullptr) {
  constexpr int VEC = Elem<T>::kVec;
  const int D = p.D, half = p.half ? p.rot / 2 : 0;
  struct alignas(16) Vec {
    T e[VEC];
  };
  if (vec && half % VEC == 0) {
    const int per = (D - half) / VEC;  // vectors of a head, partners in one
    for (int i = lane; i < heads * per; i += 64) {
      const int h = i / per, j = (i - h * per) * VEC, d = j < half ? j : j + half, c = h * D + d;
      float f[VEC];
      x.vec(c0 + c, f);
      Vec w;
      if (d < half) {
        float u[VEC];
        x.vec(c0 + c + half, u);
        Vec z;
        if (plain) {
#pragma unroll
          for (int e = 0; e < VEC; ++e) w.e[e] = Elem<T>::make(f[e]), z.e[e] = Elem<T>::make(u[e]);
          *reinterpret_cast<uint4*>(plain + c) = __builtin_bit_cast(uint4, w);
          *reinterpret_cast<uint4*>(plain + c + half) = __builtin_bit_cast(uint4, z);
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          float2 v{f[e] * inv, u[e] * inv};
          if (gain) v.x *= gain[c + e], v.y *= gain[c + half + e];
          v = turn_pair(v.x, v.y, cs[d + e]);
          w.e[e] = Elem<T>::make(v.x), z.e[e] = Elem<T>::make(v.y);
        }
        *reinterpret_cast<uint4*>(dst + (size_t)h * ldd + d + half) = __builtin_bit_cast(uint4, z);
      } else {
        if (plain) {
#pragma unroll
          for (int e = 0; e < VEC; ++e) w.e[e] = Elem<T>::make(f[e]);
          *reinterpret_cast<uint4*>(plain + c) = __builtin_bit_cast(uint4, w);
        }
#pragma unroll
        for (int e = 0; e < VEC; e += 2) {
          float2 v{f[e] * inv, f[e + 1] * inv};
          if (gain) v.x *= gain[c + e], v.y *= gain[c + e + 1];
          if (d + e < p.rot) v = turn_pair(v.x, v.y, cs[(d + e) / 2]);
          w.e[e] = Elem<T>::make(v.x), w.e[e + 1] = Elem<T>::make(v.y);
        }
      }
      *reinterpret_cast<uint4*>(dst + (size_t)h * ldd + d) = __builtin_bit_cast(uint4, w);
    }
  } else {
    for (int h = 0; h < heads; ++h)
      turn_row<T>(p, x, c0 + h * D, dst + (size_t)h * ldd, inv, gain ? gain + h * D : nullptr, cs, lane, plain ? plain + h * D : nullptr);
  }
}
// rows ahead of `row` in the step that belong to its sequence, as far as a convolution reaches
__device__ __forceinline__ int rows_ahead(const Params& p, int row, int slot) {
  int run = 0;
  while (run < p.taps - 1 && row - run > 0 && p.slot[row - run - 1] == slot) ++run;
  return run;
}
__device__ __forceinline__ float2 turn_at(const Params& p, int pos, int i) {
  float2 cs = turn_of(pos, p.freq[i]);
  cs.x *= p.amp, cs.y *= p.amp;
  return cs;
}
// staged: a row's keys ahead of their rotation go through LDS to become its values
template <typename T>
__global__ __launch_bounds__(64 * kAppendRows) void paged_prepare_kernel(const Params p, int staged) {
  extern __shared__ __attribute__((aligned(16))) char lds_raw[];  // staged: T [rows][G * D up to 8]
  __shared__ float2 cs[kAppendRows][kMaxRot / 2];
  __shared__ int s_page[kAppendRows], s_pos[kAppendRows], s_slot[kAppendRows], s_run[kAppendRows];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int row0 = blockIdx.x * kAppendRows, n = min(kAppendRows, p.n - row0);
  constexpr int VEC = Elem<T>::kVec;
  const int ldp = (p.G * p.D + 7) & ~7;
  T* plain = reinterpret_cast<T*>(lds_raw);
  const int part = blockIdx.y - 1, parts = gridDim.y - 1;
  if (wave < n) {
    const int row = row0 + wave, pos = p.pos[row], slot = p.slot[row], ahead = rows_ahead(p, row, slot);
    const int page = p.table[(size_t)slot * p.max_pages + pos / kPage];
    if (lane == 0) s_page[wave] = page, s_pos[wave] = pos, s_slot[wave] = slot, s_run[wave] = ahead;
    for (int i = lane; 2 * i < p.rot; i += 64) cs[wave][i] = turn_at(p, pos, i);  // (read by this wave only)
    const Channels<T> x(p, row, pos, slot, ahead);
    const T *q = x.raw, *k = q + p.H * p.D;
    const bool vec = p.D % VEC == 0 && p.ldq % VEC == 0 && p.ldqo % VEC == 0;
    if (part >= 0) {
      const float iq = p.whole ? 1.f / sqrtf(wave_sum(square_sum<T>(q, p.H * p.D, vec, lane, 64)) / (p.H * p.D) + p.eps) : 1.f;
      const int h0 = p.H * part / parts, h1 = p.H * (part + 1) / parts;
      T* qo = p.qout ? reinterpret_cast<T*>(p.qout) + (size_t)row * p.ldqo : const_cast<T*>(q);
      prepare_run<T>(p, x, h0 * p.D, qo + h0 * p.D, p.D, h1 - h0, iq, p.qgain ? p.qgain + h0 * p.D : nullptr, cs[wave], vec, lane);
      return;
    }
    const float ik = p.whole ? 1.f / sqrtf(wave_sum(square_sum<T>(k, p.G * p.D, vec, lane, 64)) / (p.G * p.D) + p.eps) : 1.f;
    T* dst = reinterpret_cast<T*>(p.kpool) + ((size_t)page * p.G * kPage + pos % kPage) * p.ldk;
    prepare_run<T>(p, x, p.H * p.D, dst, kPage * p.ldk, p.G, ik, p.kgain, cs[wave], vec, lane, staged ? plain + wave * ldp : nullptr);
  }
  if (part >= 0) return;
  __syncthreads();
  bool run = n == kAppendRows && s_pos[0] % kAppendRows == 0;
#pragma unroll
  for (int i = 1; i < kAppendRows; ++i)
    if (i < n) run = run && s_page[i] == s_page[0] && s_pos[i] == s_pos[0] + i;
  for (int c = threadIdx.x; c < p.G * p.E; c += 64 * kAppendRows) {
    const int g = c / p.E, d = c - g * p.E;
    T v[kAppendRows];
#pragma unroll
    for (int i = 0; i < kAppendRows; ++i) {
      const int ic = min(i, n - 1), row = row0 + ic;
      if (staged)
        v[i] = plain[ic * ldp + c];
      else if (p.vkeys)
        v[i] = Elem<T>::make(Channels<T>(p, row, s_pos[ic], s_slot[ic], s_run[ic]).at(p.H * p.D + c));
      else
        v[i] = mixed_value<T>(p, reinterpret_cast<const T*>(p.qkv)[(size_t)row * p.ldq + (p.H + p.G) * p.D + c], row, c);
    }
    if (run) {
      T* dst = reinterpret_cast<T*>(p.vpool) + (((size_t)s_page[0] * p.G + g) * p.ldv + d) * kPage + s_pos[0] % kPage;
      constexpr int per = 16 / (int)sizeof(T);
#pragma unroll
      for (int k = 0; k < kAppendRows; k += per) {
        struct alignas(16) Vec {
          T e[per];
        } w;
#pragma unroll
        for (int i = 0; i < per; ++i) w.e[i] = v[k + i];
        *reinterpret_cast<uint4*>(dst + k) = __builtin_bit_cast(uint4, w);
      }
    } else {
#pragma unroll
      for (int i = 0; i < kAppendRows; ++i)
        if (i < n) reinterpret_cast<T*>(p.vpool)[(((size_t)s_page[i] * p.G + g) * p.ldv + d) * kPage + s_pos[i] % kPage] = v[i];
    }
  }
}

template <typename T>
struct PTerms;  // softmax weights of 32 keys as B operands
template <>
struct PTerms<bf16_t> {
  uint4 hi, lo;
  __device__ __forceinline__ void set(const float (&a)[4], const float (&b)[4]) {
    float ra[4], rb[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ra[i] = a[i] - bf2f(f2bf(a[i])), rb[i] = b[i] - bf2f(f2bf(b[i]));
    hi = uint4{pack_bf2(a[0], a[1]), pack_bf2(a[2], a[3]), pack_bf2(b[0], b[1]), pack_bf2(b[2], b[3])};
    lo = uint4{pack_bf2(ra[0], ra[1]), pack_bf2(ra[2], ra[3]), pack_bf2(rb[0], rb[1]), pack_bf2(rb[2], rb[3])};
  }
};
template <>
struct PTerms<float> {
  uint4 hi, lo;
  __device__ __forceinline__ void set(const float (&a)[4], const float (&b)[4]) {
    hi = __builtin_bit_cast(uint4, floatx4{a[0], a[1], a[2], a[3]});
    lo = __builtin_bit_cast(uint4, floatx4{b[0], b[1], b[2], b[3]});
  }
};
// a value column's entries of this lane's keys: 4g.. and 16 + 4g.. of the 32-key tile at v.  (Keys dealt to the two operands in runs
// of four, so that the eight of a bf16 column are one request of 16 bytes, meet in other sums, and a decoder's outputs change: four rows of 32 / 4 heads of 128,
// 700 keys 10.6 us for 11.2.)
template <typename T>
struct VTerms;
template <>
struct VTerms<bf16_t> {
  uint2 a, b;
  __device__ __forceinline__ void load(const bf16_t* v, int g) {
    a = *reinterpret_cast<const uint2*>(v + 4 * g);
    b = *reinterpret_cast<const uint2*>(v + 16 + 4 * g);
  }
  __device__ __forceinline__ floatx4 mma(const PTerms<bf16_t>& p, floatx4 c) const {
    const uint4 x{a.x, a.y, b.x, b.y};
    return Elem<bf16_t>::mma16(x, p.lo, Elem<bf16_t>::mma16(x, p.hi, c));
  }
};
template <>
struct VTerms<float> {
  uint4 a, b;
  __device__ __forceinline__ void load(const float* v, int g) {
    a = *reinterpret_cast<const uint4*>(v + 4 * g);
    b = *reinterpret_cast<const uint4*>(v + 16 + 4 * g);
  }
  __device__ __forceinline__ floatx4 mma(const PTerms<float>& p, floatx4 c) const {
    return Elem<float>::mma16(b, p.lo, Elem<float>::mma16(a, p.hi, c));
  }
};

constexpr int kRowWaves = 4;

template <typename T, int DMAX, bool FUSE, int MODE>
__global__ __launch_bounds__(64 * kRowWaves) void paged_rows_kernel(const Params all) {
  constexpr bool SIGMOID = MODE == kSigmoid;
  if (MODE == kPlain) request_arguments(all);  // (the other modes' registers do not hold what it makes the compiler keep)
  const Params p = only<MODE>(all);
  constexpr int KST = DMAX * (int)sizeof(T) / 64;  // 64-byte steps over a key
  constexpr int VT = DMAX / 16;                    // 16-row tiles of O^T
  constexpr int QS = DMAX + 16 / (int)sizeof(T);   // LDS row stride of q
  extern __shared__ __attribute__((aligned(16))) char lds_raw[];
  T* qs = reinterpret_cast<T*>(lds_raw);                          // [16][QS]
  float* os = reinterpret_cast<float*>(lds_raw);                  // later: [waves][gsz][ldv + 4]
  __shared__ float ms[kRowWaves][16], ls[kRowWaves][16];
  __shared__ float2 cs[kMaxRot / 2];
  __shared__ int s_last;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int split = blockIdx.x, kvh = p.hgroups == 1 ? (int)blockIdx.y : (int)blockIdx.y / p.hgroups, hg = blockIdx.y - kvh * p.hgroups;
  const int row = p.list ? p.list[blockIdx.z] : (int)blockIdx.z;
  const int group = p.group;
  const int h0 = kvh * group + hg * p.gsz, gs = min(p.gsz, (kvh + 1) * group - h0);
  // The row's channels are requested before its position is known, so that they come with it (each is a way through memory): as they are
  // (plain: 16 bytes per thread), or to be divided by their RMS.
  const bool turned = p.whole || p.rot || p.taps;
  const T* const raw = reinterpret_cast<const T*>(p.qkv) + (size_t)row * p.ldq;
  constexpr int EPV = 16 / (int)sizeof(T), VPR = DMAX / EPV, NQ = (16 * VPR + 64 * kRowWaves - 1) / (64 * kRowWaves);
  const bool plain = !turned && !p.unit && p.D % EPV == 0 && ((uintptr_t)raw & 15) == 0;
  u32x4_t qv[NQ], kv = {0, 0, 0, 0};
  UnitRow<T, DMAX> qin[16 / kRowWaves], kvin;
  if (plain) {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int at = threadIdx.x + 64 * kRowWaves * i, h = at / VPR, c = at % VPR * EPV;
      qv[i] = u32x4_t{0, 0, 0, 0};
      if (h < gs && c < p.D) qv[i] = *reinterpret_cast<const u32x4_t*>(raw + (h0 + h) * p.D + c);
    }
    if (FUSE && wave == kRowWaves - 1 && lane * EPV < p.D) kv = *reinterpret_cast<const u32x4_t*>(raw + (p.H + kvh) * p.D + lane * EPV);
  } else if (!turned) {
#pragma unroll
    for (int i = 0; i < 16 / kRowWaves; ++i)
      if (wave + kRowWaves * i < gs) qin[i].request(raw + (h0 + wave + kRowWaves * i) * p.D, p.D, lane);
    if (FUSE && wave == kRowWaves - 1) kvin.request(raw + (p.H + kvh) * p.D, p.D, lane);
  }
  if (FUSE && !turned && wave == kRowWaves - 2 && !p.vkeys) kvin.request(raw + (p.H + p.G) * p.D + kvh * p.E, p.E, lane);
  const int pos = p.pos[row], slot = p.slot[row];
  const int32_t* table = p.table + (size_t)slot * p.max_pages;
  const Tiles tl = tiles_of(p, pos, pos, 32);
  const int seen = blocks_seen(p, pos);
  // The launch is laid out for the longest context that the host allows for: splits without a tile leave at
  // once and take no part in the merge, and a single one writes the result itself (48 keys of 64, 16 heads, 2 rows
  // laid out for 3 splits: 10.7 -> 8.6 us).
  const int used = max(1, min(p.nsplit, (tl.n + kRowWaves - 1) / kRowWaves));
  if (split >= used) return;

  const int ksteps = p.ldk * (int)sizeof(T) / 64, vtiles = p.ldv / 16;
  struct Tile {
    uint4 ka[KST], kb[KST];
    VTerms<T> v[VT];
  };
  auto page_of = [&](int j) { return (tl.mean(j) ? p.mtable + (size_t)slot * p.mpages : table)[tl.at(j) * 32 / kPage]; };
  auto load_tile = [&](Tile& t, int j, int page) {
    const bool mean = tl.mean(j);
    const int key0 = tl.at(j) * 32;
    const size_t head = (size_t)page * p.G + kvh;
    const char* kp = reinterpret_cast<const char*>(reinterpret_cast<const T*>(mean ? p.mkpool : p.kpool) +
                                                   (head * kPage + (key0 % kPage) + r) * p.ldk) + g * 16;
    const T* vp = reinterpret_cast<const T*>(mean ? p.mvpool : p.vpool) + (head * p.ldv + r) * kPage + (key0 % kPage);
#pragma unroll
    for (int s = 0; s < KST; ++s)
      if (s < ksteps) {
        t.ka[s] = *reinterpret_cast<const uint4*>(kp + s * 64);
        t.kb[s] = *reinterpret_cast<const uint4*>(kp + (size_t)16 * p.ldk * sizeof(T) + s * 64);
      }
#pragma unroll
    for (int i = 0; i < VT; ++i)
      if (i < vtiles) t.v[i].load(vp + (size_t)i * 16 * kPage, g);
  };
  // The page of a wave's first tile is on its way while the queries are normalised, and the tile while the row's key is stored - unless it
  // is the one that this key goes into.  Where one split holds all tiles the tile goes out ahead of the queries' arithmetic (us, normed
  // queries, 48 keys: 16 / 8 heads of 64 float 6.60 -> 6.40, bf16 5.64 -> 5.55, 32 / 4 of 128 bf16 7.40 -> 7.14); with several it is the slower order (4 rows of
  // 32 / 4 of 128, 3000 keys 17.1 -> 17.7, 150 10.1 -> 10.5).
  const int stride = p.nsplit * kRowWaves;
  int j = split * kRowWaves + wave;
  Tile tile;
  const bool early = j < tl.n && !(FUSE && j == tl.n - 1);
  const bool owner = FUSE && split == ((tl.n - 1) % stride) / kRowWaves;
  const int page0 = j < tl.n ? page_of(j) : 0, own_page = owner ? table[pos / kPage] : 0;

  // ---- queries (and the row's own key and value) through float32 norms
  float iq = 1.f, ik = 1.f;
  if (early && used == 1) load_tile(tile, j, page0);
  const Channels<T> x(p, row, pos, slot, 0);
  if (turned) {  // angles, and the RMS of the whole projections, once per workgroup
    const T* src = raw;
    for (int i = threadIdx.x; 2 * i < p.rot; i += 64 * kRowWaves) cs[i] = turn_at(p, pos, i);
    if (p.whole) {
      const bool vec = p.D % Elem<T>::kVec == 0 && p.ldq % Elem<T>::kVec == 0;
      float sq = square_sum<T>(src, p.H * p.D, vec, threadIdx.x, 64 * kRowWaves);
      float sk = FUSE ? square_sum<T>(src + p.H * p.D, p.G * p.D, vec, threadIdx.x, 64 * kRowWaves) : 0.f;
      sq = wave_sum(sq), sk = wave_sum(sk);
      if (lane == 0) ms[wave][0] = sq, ms[wave][1] = sk;
    }
    __syncthreads();
    if (p.whole) {
      float sq = 0.f, sk = 0.f;
#pragma unroll
      for (int w = 0; w < kRowWaves; ++w) sq += ms[w][0], sk += ms[w][1];
      iq = 1.f / sqrtf(sq / (p.H * p.D) + p.eps), ik = 1.f / sqrtf(sk / (p.G * p.D) + p.eps);
    }
  }
  if (plain) {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int at = threadIdx.x + 64 * kRowWaves * i, h = at / VPR, c = at % VPR * EPV;
      if (16 * VPR % (64 * kRowWaves) == 0 || h < 16) *reinterpret_cast<u32x4_t*>(qs + h * QS + c) = qv[i];
    }
  } else if (turned) {
    for (int h = wave; h < 16; h += kRowWaves) {
      T* dst = qs + h * QS;
      if (h < gs) turn_row<T>(p, x, (h0 + h) * p.D, dst, iq, p.qgain ? p.qgain + (h0 + h) * p.D : nullptr, cs, lane);
      for (int d = (h < gs ? p.D : 0) + lane; d < QS; d += 64) dst[d] = Elem<T>::make(0.f);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16 / kRowWaves; ++i) {
      const int h = wave + kRowWaves * i;
      T* dst = qs + h * QS;
      if (h < gs) qin[i].put(dst, p.D, p.unit, p.eps, p.qgain, lane);
      for (int d = (h < gs ? p.D : 0) + lane; d < QS; d += 64) dst[d] = Elem<T>::make(0.f);
    }
  }
  if (early && used > 1) load_tile(tile, j, page0);
  if (owner) {
    const size_t head = (size_t)own_page * p.G + kvh;
    if (wave == kRowWaves - 1) {
      T* const dst = reinterpret_cast<T*>(p.kpool) + (head * kPage + pos % kPage) * p.ldk;
      if (plain) {
        if (lane * EPV < p.D) *reinterpret_cast<u32x4_t*>(dst + lane * EPV) = kv;
      } else if (turned) {
        put_key<T>(p, x, kvh, dst, lane, ik, cs);
      } else {
        kvin.put(dst, p.D, p.unit, p.eps, p.kgain, lane);
      }
    } else if (wave == kRowWaves - 2) {
      T* const dst = reinterpret_cast<T*>(p.vpool) + head * p.ldv * kPage + pos % kPage;
      if (turned || p.vkeys) {
        put_value<T>(p, x, row, kvh, dst, lane);
      } else {
#pragma unroll
        for (int i = 0; i < DMAX / 64; ++i)
          if (lane + 64 * i < p.E) dst[(size_t)(lane + 64 * i) * kPage] = mixed_value<T>(p, kvin.x[i], row, kvh * p.E + lane + 64 * i);
      }
    }
    wait_own_stores_done();
  }
  if (FUSE && p.taps && split == 0) keep_channels<T>(x, h0 * p.D, gs * p.D, threadIdx.x, 64 * kRowWaves);
  __syncthreads();
  if (!early && j < tl.n) load_tile(tile, j, page0);
  uint4 q[KST];
#pragma unroll
  for (int s = 0; s < KST; ++s)
    q[s] = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(qs + r * QS) + s * 64 + g * 16);

  const float sc = p.cap > 0.f ? p.scale / p.cap : p.scale * kLog2e, cap2 = p.cap * kLog2e;
  const float slope = p.slopes && r < gs ? p.slopes[h0 + r] * kLog2e : 0.f;
  floatx4 o[VT];
#pragma unroll
  for (int t = 0; t < VT; ++t) o[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  if (!SIGMOID && p.one && split == 0 && wave == 0) m = 0.f, l = 1.f;  // (a score of 0 without a value)
  const float wb = SIGMOID && r < gs ? p.wbias[h0 + r] * kLog2e : 0.f;

  while (j < tl.n) {
    const int key0 = tl.at(j) * 32;
    const int lim = tl.mean(j) ? seen - 1 : pos, size = tl.mean(j) ? 0x3FFFFFFF : p.size;
    floatx4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KST; ++s)
      if (s < ksteps) {
        s0 = Elem<T>::mma16(tile.ka[s], q[s], s0);
        s1 = Elem<T>::mma16(tile.kb[s], q[s], s1);
      }
    float x0[4], x1[4], mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 4; ++e) s0[e] *= sc, s1[e] *= sc;
    if (p.cap > 0.f) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s0[e] = sizeof(T) == 2 ? bent(s0[e], cap2) : cap2 * tanhf(s0[e]);
        s1[e] = sizeof(T) == 2 ? bent(s1[e], cap2) : cap2 * tanhf(s1[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int ja = key0 + 4 * g + e, jb = ja + 16;
      const bool va = ja <= lim && (pos - ja < size || ja < p.keep);
      const bool vb = jb <= lim && (pos - jb < size || jb < p.keep);
      if (SIGMOID) {
        x0[e] = va ? 1.f / (1.f + __builtin_amdgcn_exp2f(-(s0[e] + wb))) : 0.f;
        x1[e] = vb ? 1.f / (1.f + __builtin_amdgcn_exp2f(-(s1[e] + wb))) : 0.f;
        continue;
      }
      x0[e] = va ? s0[e] - slope * (float)(pos - ja) : -INFINITY;
      x1[e] = vb ? s1[e] - slope * (float)(pos - jb) : -INFINITY;
      mx = fmaxf(mx, fmaxf(x0[e], x1[e]));
    }
    float a = 1.f;
    if (!SIGMOID) {
      mx = max_across<32>(max_across<16>(mx));
      const float mn = fmaxf(m, mx);  // finite: a dealt tile holds a visible key
      a = __builtin_amdgcn_exp2f(m - mn);
      float sum = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x0[e] = __builtin_amdgcn_exp2f(x0[e] - mn);
        x1[e] = __builtin_amdgcn_exp2f(x1[e] - mn);
        sum += x0[e] + x1[e];
      }
      sum = add_across<32>(add_across<16>(sum));
      l = l * a + sum;
      m = mn;
    }
    PTerms<T> pt;
    pt.set(x0, x1);
#pragma unroll
    for (int t = 0; t < VT; ++t)
      if (t < vtiles) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (!SIGMOID) o[t][e] *= a;
        o[t] = tile.v[t].mma(pt, o[t]);
      }
    j += stride;
    if (j < tl.n) load_tile(tile, j, page_of(j));
  }

  if (owner && p.pool && hg == 0 && (pos + 1) % p.pool == 0) put_means<T>(p, slot, pos / p.pool, kvh, threadIdx.x, 64 * kRowWaves);

  // ---- the waves of the workgroup
  if (SIGMOID) m = 0.f, l = split == 0 && wave == 0 ? 1.f : 0.f;  // (factors of 1 from here on)
  if (g == 0) ms[wave][r] = m, ls[wave][r] = l;
  __syncthreads();  // (also: q in LDS is no longer read)
  float mw = ms[0][r];
#pragma unroll
  for (int w = 1; w < kRowWaves; ++w) mw = fmaxf(mw, ms[w][r]);
  const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mw);
  const int osl = p.ldv + 4;  // (rows a bank group apart)
  if (r < gs) {
#pragma unroll
    for (int t = 0; t < VT; ++t)
      if (t < vtiles) {
        floatx4 v = o[t];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= f;
        *reinterpret_cast<floatx4*>(&os[(wave * p.gsz + r) * osl + t * 16 + 4 * g]) = v;
      }
  }
  __syncthreads();
  T* out = reinterpret_cast<T*>(p.out) + (size_t)row * p.ldo;
  const size_t wsrow = (size_t)blockIdx.z * p.H;
  const int stride_ws = p.E + 2;
  const auto ws = buf_of(p.ws + (wsrow + h0) * p.nsplit * stride_ws, used > 1 ? (uint32_t)(gs * p.nsplit * stride_ws) * 4 : 0);
  const uint32_t head_ws = (uint32_t)(p.nsplit * stride_ws) * 4;
  // W neighbouring columns per thread, as many as give every column a thread
  const int columns = p.E % 4 == 0 && gs * p.E > 2 * 64 * kRowWaves ? 4 : p.E % 2 == 0 && gs * p.E > 64 * kRowWaves ? 2 : 1;
  auto finished = [&](int h, int d, auto& a, float l) __attribute__((always_inline)) {
    constexpr int W = sizeof(a.v) / 4;
    const float hgate = head_gate(p, row, h0 + h);
    T* const to = out + (h0 + h) * p.E + d;
    float f[W];
#pragma unroll
    for (int c = 0; c < W; ++c) f[c] = a.v[c] / l * hgate;
    if (p.ogate) {
#pragma unroll
      for (int c = 0; c < W; ++c) f[c] *= column_gate<T>(p, row, (h0 + h) * p.E + d + c);
    }
    struct alignas(W * sizeof(T)) {
      T v[W];
    } t;
#pragma unroll
    for (int c = 0; c < W; ++c) t.v[c] = Elem<T>::make(f[c]);
    if (((uintptr_t)to & (W * sizeof(T) - 1)) == 0) {
      *reinterpret_cast<decltype(t)*>(to) = t;
    } else {
#pragma unroll
      for (int c = 0; c < W; ++c) to[c] = t.v[c];
    }
  };
  auto combine = [&](auto run) __attribute__((always_inline)) {
    constexpr int W = decltype(run)::value;
    const int per = p.E / W;
    for (int i = threadIdx.x; i < gs * per; i += 64 * kRowWaves) {
      const int h = i / per, d = (i - h * per) * W;
      Run<W> a = {};
      float lw = 0.f, mm = -INFINITY;
#pragma unroll
      for (int w = 0; w < kRowWaves; ++w) mm = fmaxf(mm, ms[w][h]);
#pragma unroll
      for (int w = 0; w < kRowWaves; ++w) {
        const Run<W> v = *reinterpret_cast<const Run<W>*>(&os[(w * p.gsz + h) * osl + d]);
#pragma unroll
        for (int c = 0; c < W; ++c) a.v[c] += v.v[c];
        lw += ms[w][h] == -INFINITY ? 0.f : ls[w][h] * __builtin_amdgcn_exp2f(ms[w][h] - mm);
      }
      if (used == 1) {
        finished(h, d, a, lw);
      } else {
        const uint32_t at = h * head_ws, part = (uint32_t)(split * stride_ws) * 4;
        st_dev<W>(ws, at + d * 4, part, a);
        if (d == 0) st_dev<2>(ws, at + p.E * 4, part, Run<2>{{mm, lw}});
      }
    }
  };
  if (columns == 4)
    combine(std::integral_constant<int, 4>());
  else if (columns == 2)
    combine(std::integral_constant<int, 2>());
  else
    combine(std::integral_constant<int, 1>());
  if (used == 1) return;

  // ---- the splits: the last workgroup to arrive merges them (values at device scope, every
  // wave's stores complete before the barrier, then one counter increment; it returns to zero)
  wait_own_stores_done();
  __syncthreads();
  if (threadIdx.x == 0) {
    int* cnt = p.counters + (size_t)blockIdx.z * gridDim.y + blockIdx.y;
    const int old = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = old == used - 1;
    if (s_last) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!s_last) return;
  // A batch of splits at a time, all its requests ahead of their use, in a running (maximum, sum, weighted sum).  (First every
  // split's factor, then sixteen values of one column at a time whatever the number of splits, the waves one column at a
  // time through conflicting banks: 4 rows of 32 / 4 heads, 700 keys 19.8 us against 16.3, then.)
  auto merge = [&](auto run) __attribute__((always_inline)) {
    constexpr int MS = 8, W = decltype(run)::value;
    const int per = p.E / W;
    for (int i = threadIdx.x; i < gs * per; i += 64 * kRowWaves) {
      const int h = i / per, d = (i - h * per) * W;
      const uint32_t at = h * head_ws;
      Run<W> a = {};
      float lsum = 0.f, mw = -INFINITY;
      for (int s0 = 0; s0 < used; s0 += MS) {
        Run<2> ml[MS];
        Run<W> v[MS];
#pragma unroll
        for (int s = 0; s < MS; ++s) {
          const uint32_t part = (uint32_t)(min(s0 + s, used - 1) * stride_ws) * 4;
          ml[s] = ld_dev<2>(ws, at + p.E * 4, part);
          v[s] = ld_dev<W>(ws, at + d * 4, part);
        }
        float mc = mw;
#pragma unroll
        for (int s = 0; s < MS; ++s) mc = s0 + s < used ? fmaxf(mc, ml[s].v[0]) : mc;
        const float back = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - mc);
#pragma unroll
        for (int c = 0; c < W; ++c) a.v[c] *= back;
        lsum *= back;
#pragma unroll
        for (int s = 0; s < MS; ++s) {
          const float w1 = s0 + s >= used || ml[s].v[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml[s].v[0] - mc);
#pragma unroll
          for (int c = 0; c < W; ++c) a.v[c] += v[s].v[c] * w1;
          lsum += ml[s].v[1] * w1;
        }
        mw = mc;
      }
      finished(h, d, a, lsum);
    }
  };
  if (columns == 4)
    merge(std::integral_constant<int, 4>());
  else if (columns == 2)
    merge(std::integral_constant<int, 2>());
  else
    merge(std::integral_constant<int, 1>());
}

// ------------------------------------------------------------------------------ prompts
constexpr int kPadK = 8;

template <int DK, int DV>
constexpr int prompt_lds() {
  return 2 * (kPage * (DK + kPadK) + DV * (kPage + kPadK)) * 2;
}

// DK, DV: key and value size at most; HW: query heads per workgroup (4, 2, 1), its other factor is token
// tiles of 32; ROWS: expanded keys and values instead of the pool's (HW 1); MODE kSigmoid: weights that are no softmax
template <int DK, int DV, int HW, bool ROWS, int MODE>
__global__ __launch_bounds__(256, DK > 128 ? 1 : 2) void paged_prompt_kernel(const Params all, const Expanded x) {
  constexpr bool SIGMOID = MODE == kSigmoid;
  const Params p = only<MODE>(all);
  constexpr int STEPS = DK / 16, DT = DV / 32, KS = DK + kPadK, VS = kPage + kPadK;
  constexpr int VEC = DK / 8, LOADS = kPage * VEC / 256, VLOADS = DV / 32;
  constexpr int BUF = kPage * KS + DV * VS;
  constexpr int TT = 4 / HW;  // token tiles per workgroup
  extern __shared__ __attribute__((aligned(16))) bf16_t lds[];  // [2][BUF]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, kq = lane >> 5;
  const int group = p.H / p.G, hgroups = (group + HW - 1) / HW;
  const int kvh = blockIdx.y / hgroups, hg = blockIdx.y % hgroups;
  const int4 blk = reinterpret_cast<const int4*>(p.list)[gridDim.x - 1 - blockIdx.x];  // row, slot, pos, n
  const int hi = hg * HW + wave % HW, tt = wave / HW;
  const bool active = hi < group && tt * 32 < blk.w;
  const int hq = kvh * group + min(hi, group - 1);
  const int t_lane = min(tt * 32 + n, blk.w - 1);  // this lane's token of the block
  const int row = blk.x + t_lane, qpos = blk.z + t_lane;
  const int wfirst = blk.z + min(tt * 32, blk.w - 1), wlast = blk.z + min(tt * 32 + 31, blk.w - 1);
  const int32_t* table = ROWS ? nullptr : p.table + (size_t)blk.y * p.max_pages;
  const Tiles tl = tiles_of(p, blk.z, blk.z + blk.w - 1, kPage);
  const int seen = blocks_seen(p, qpos), seen_first = blocks_seen(p, wfirst), seen_last = blocks_seen(p, wlast);

  // Q^T operand: lane (query n, half kq) holds d = 16 step + 8 kq .. + 8, normalised in float32
  uint4 q[STEPS];
  {
    const bf16_t* qp = reinterpret_cast<const bf16_t*>(p.qkv) + (size_t)row * p.ldq + (size_t)hq * (ROWS ? x.qs : p.D);
    float ss = 0.f;
    const bool vec = p.D % 8 == 0 && p.ldq % 8 == 0;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int d0 = 16 * s + 8 * kq;
      uint32_t w[4];
      if (ROWS) {
        const bf16_t* at = d0 < x.d8 ? qp + d0
                                     : reinterpret_cast<const bf16_t*>(p.qkv) + (size_t)row * p.ldq + x.rot_col + hq * x.r8 + (d0 - x.d8);
        const uint4 v = d0 < x.d8 + x.r8 ? *reinterpret_cast<const uint4*>(at) : uint4{0, 0, 0, 0};
        w[0] = v.x, w[1] = v.y, w[2] = v.z, w[3] = v.w;
      } else if (vec) {
        const uint4 v = d0 < p.D ? *reinterpret_cast<const uint4*>(qp + d0) : uint4{0, 0, 0, 0};
        w[0] = v.x, w[1] = v.y, w[2] = v.z, w[3] = v.w;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t a = d0 + 2 * i < p.D ? qp[d0 + 2 * i] : 0, b = d0 + 2 * i + 1 < p.D ? qp[d0 + 2 * i + 1] : 0;
          w[i] = a | b << 16;
        }
      }
      q[s] = uint4{w[0], w[1], w[2], w[3]};
#pragma unroll
      for (int i = 0; i < 4; ++i) ss += bf_lo(w[i]) * bf_lo(w[i]) + bf_hi(w[i]) * bf_hi(w[i]);
    }
    ss = add_across<32>(ss);
    if (p.unit) {
      const float inv = 1.f / sqrtf(ss / p.D + p.eps);
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        const uint32_t w[4] = {q[s].x, q[s].y, q[s].z, q[s].w};
        uint32_t u[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int d = 16 * s + 8 * kq + 2 * i;  // (past D the queries are zero)
          const float ga = p.qgain ? p.qgain[min(d, p.D - 1)] * inv : inv, gb = p.qgain ? p.qgain[min(d + 1, p.D - 1)] * inv : inv;
          u[i] = pack_bf2(bf_lo(w[i]) * ga, bf_hi(w[i]) * gb);
        }
        q[s] = uint4{u[0], u[1], u[2], u[3]};
      }
    }
  }

  uint4 kreg[LOADS], vreg[VLOADS];
  const uint32_t kbytes = kPage * (uint32_t)p.ldk * 2, vbytes = (uint32_t)p.ldv * kPage * 2;
  auto load_tile = [&](int j) __attribute__((always_inline)) {
    if (ROWS) {  // (columns past a key's and rows past the values': any finite ones)
      const int key = blk.y + tl.at(j) * kPage;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const int vi = tid + i * 256, kr = key + vi / VEC, kc = vi % VEC * 8;
        const bf16_t* at = kc < x.d8 ? x.k + (size_t)kr * x.ldk + hq * x.d8 + kc : x.kr + (size_t)kr * x.r8 + min(kc - x.d8, x.r8 - 8);
        kreg[i] = load16(at);
      }
#pragma unroll
      for (int i = 0; i < VLOADS; ++i) {
        const int vi = tid + i * 256;
        vreg[i] = load16(x.v + (size_t)(hq * p.E + min(vi >> 3, p.E - 1)) * x.ldv + key + (vi & 7) * 8);
      }
      return;
    }
    const bool mean = tl.mean(j);
    const size_t head = (size_t)(mean ? p.mtable + (size_t)blk.y * p.mpages : table)[tl.at(j)] * p.G + kvh;
    const __amdgpu_buffer_rsrc_t rk = buf_of(reinterpret_cast<const bf16_t*>(mean ? p.mkpool : p.kpool) + head * kPage * p.ldk, kbytes);
    const __amdgpu_buffer_rsrc_t rv = buf_of(reinterpret_cast<const bf16_t*>(mean ? p.mvpool : p.vpool) + head * p.ldv * kPage, vbytes);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int vi = tid + i * 256, kr = vi / VEC, kc = vi % VEC;
      kreg[i] = buf_load16(rk, kc * 8 < p.ldk ? (kr * p.ldk + kc * 8) * 2 : kPastEnd, 0);
    }
#pragma unroll
    for (int i = 0; i < VLOADS; ++i) vreg[i] = buf_load16(rv, (tid + i * 256) * 16, 0);  // rows of 64 positions; rows past ldv read as zero
  };
  auto store_tile = [&](int b) {
    bf16_t* kl = lds + b * BUF;
    bf16_t* vl = kl + kPage * KS;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int vi = tid + i * 256;
      *reinterpret_cast<uint4*>(&kl[(vi / VEC) * KS + (vi % VEC) * 8]) = kreg[i];
    }
#pragma unroll
    for (int i = 0; i < VLOADS; ++i) {
      const int vi = tid + i * 256;
      *reinterpret_cast<uint4*>(&vl[(vi >> 3) * VS + (vi & 7) * 8]) = vreg[i];
    }
  };
  // A-operand row n of a 32-key sub-tile holds this key, so that result registers 8s..8s+7 of
  // lane half kq are keys 16s + 8kq .. + 8 (the B operand order of the second product)
  const int jr = n >> 3;
  const int key_of_row = 16 * (jr >> 1) + 8 * ((n >> 2) & 1) + 4 * (jr & 1) + (n & 3);
  const float sc = p.scale * kLog2e, cap2 = p.cap * kLog2e, icap = p.cap > 0.f ? p.scale / p.cap : 0.f;
  const float slope = p.slopes ? p.slopes[hq] * kLog2e : 0.f;

  floatx16 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
  float m = -INFINITY, l = 0.f;
  if (SIGMOID || p.one) m = 0.f, l = 1.f;  // (a score of 0 without a value; weights that are no softmax end with 1)
  const float wb = SIGMOID ? p.wbias[hq] * kLog2e : 0.f;

  load_tile(0);
  store_tile(0);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): no wait for the queries inside the loop
  if (tl.n > 1) load_tile(1);
  for (int j = 0; j < tl.n; ++j) {
    __syncthreads();  // tile j is complete in its buffer, the other buffer is no longer read
    if (j + 1 < tl.n) {
      store_tile((j + 1) & 1);
      if (j + 2 < tl.n) load_tile(j + 2);
    }
    const int key0 = tl.at(j) * kPage, key1 = key0 + kPage - 1;
    // wave-uniform: nothing of the tile is visible to the wave's queries
    const bool mean = tl.mean(j);
    if (!active || (mean ? key0 >= seen_last : key0 > wlast || (wfirst - key1 >= p.size && key0 >= p.keep))) continue;
    const bf16_t* kl = lds + (j & 1) * BUF;
    const bf16_t* vl = kl + kPage * KS;
    floatx16 s[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int e = 0; e < 16; ++e) s[ks][e] = 0.f;
      const bf16_t* kr = &kl[(ks * 32 + key_of_row) * KS + kq * 8];
#pragma unroll
      for (int st = 0; st < STEPS; ++st)
        s[ks] = Elem<bf16_t>::mma32(*reinterpret_cast<const uint4*>(kr + st * 16), q[st], s[ks]);
    }
    const bool partial = mean ? key1 >= seen_first : key1 > wfirst || (wlast - key0 >= p.size && key1 >= p.keep);
    const int rel = (mean ? seen - 1 : qpos) - key0 - 8 * kq;  // distance to the lane's first key
    const int size = mean ? 0x3FFFFFFF : p.size;
    const float base = -slope * (float)rel;
    float mx = -INFINITY;
    if (p.cap > 0.f) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          s[ks][e] = bent(s[ks][e] * icap, cap2);
    }
    const float scl = p.cap > 0.f ? 1.f : sc;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int k = ks * 32 + 16 * (e >> 3) + (e & 7);
        float sv = SIGMOID ? fmaf(s[ks][e], sc, wb) : fmaf(s[ks][e], scl, fmaf(slope, (float)k, base));
        if (partial && (k > rel || (rel - k >= size && key0 + 8 * kq + k >= p.keep))) sv = -INFINITY;
        s[ks][e] = sv;
        mx = fmaxf(mx, sv);
      }
    float mr = 0.f, mn = 0.f, al = 1.f;
    if (!SIGMOID) {
      mx = max_across<32>(mx);
      mn = fmaxf(m, mx), mr = mn == -INFINITY ? 0.f : mn;  // (a query may see none of the tile)
      al = __builtin_amdgcn_exp2f(m - mr);
    }
    float sum = 0.f;
    uint4 ph[2][2], pl[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        float a[8], b[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (SIGMOID) {
            a[e] = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-s[ks][8 * st + e]));
          } else {
            a[e] = __builtin_amdgcn_exp2f(s[ks][8 * st + e] - mr);
            sum += a[e];
          }
        }
        ph[ks][st] = uint4{pack_bf2(a[0], a[1]), pack_bf2(a[2], a[3]), pack_bf2(a[4], a[5]), pack_bf2(a[6], a[7])};
        const uint32_t w[4] = {ph[ks][st].x, ph[ks][st].y, ph[ks][st].z, ph[ks][st].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) b[2 * e] = a[2 * e] - bf_lo(w[e]), b[2 * e + 1] = a[2 * e + 1] - bf_hi(w[e]);
        pl[ks][st] = uint4{pack_bf2(b[0], b[1]), pack_bf2(b[2], b[3]), pack_bf2(b[4], b[5]), pack_bf2(b[6], b[7])};
      }
    if (!SIGMOID) {
      sum = add_across<32>(sum);
      l = l * al + sum;
      m = mn;
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (!SIGMOID) o[t][e] *= al;
      const bf16_t* vr = &vl[(t * 32 + n) * VS + kq * 8];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          const uint4 a = *reinterpret_cast<const uint4*>(vr + ks * 32 + st * 16);
          o[t] = Elem<bf16_t>::mma32(a, ph[ks][st], o[t]);
          o[t] = Elem<bf16_t>::mma32(a, pl[ks][st], o[t]);
        }
    }
  }
  if (!active || tt * 32 + n >= blk.w) return;
  const float inv = head_gate(p, row, hq) / l;
  bf16_t* op = reinterpret_cast<bf16_t*>(p.out) + (size_t)row * p.ldo + (size_t)hq * p.E;
  const bool pairs = p.E % 4 == 0;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = t * 32 + 8 * i + 4 * kq;
      if (p.ogate && d < p.E) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[t][4 * i + e] *= column_gate<bf16_t>(p, row, hq * p.E + min(d + e, p.E - 1));
      }
      if (pairs) {
        if (d < p.E)
          *reinterpret_cast<uint2*>(op + d) = uint2{pack_bf2(o[t][4 * i] * inv, o[t][4 * i + 1] * inv),
                                                    pack_bf2(o[t][4 * i + 2] * inv, o[t][4 * i + 3] * inv)};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < p.E) op[d + e] = f2bf(o[t][4 * i + e] * inv);
      }
    }
}

Params params_of(const exo_paged_attn* a) {
  Params p{};
  p.qkv = a->qkv, p.kpool = a->k_pool, p.vpool = a->v_pool, p.table = a->table, p.slot = a->slot, p.pos = a->pos;
  p.list = a->list, p.slopes = a->slopes, p.out = a->out;
  p.qgain = a->q_gain, p.kgain = a->k_gain, p.gate = a->gate, p.ldg = a->ldg;
  p.scale = a->scale, p.eps = a->eps, p.n = a->n, p.H = a->heads, p.G = a->kv_heads, p.D = a->dim, p.E = a->vdim;
  p.ldq = a->ldq, p.ldk = a->ldk, p.ldv = a->ldv, p.ldo = a->ldo, p.max_pages = a->max_pages;
  p.size = a->window > 0 ? a->window : 0x3FFFFFFF;
  p.keep = a->keep_first, p.unit = a->unit_qk;
  p.freq = a->freq, p.vmix = a->v_mix, p.ldmix = a->ldmix, p.mix = a->mix, p.cap = a->softcap, p.whole = a->whole_norm, p.rot = a->rot;
  p.ogate = a->out_gate, p.ldog = a->ldog, p.wbias = a->weight_bias, p.one = a->plus_one, p.half = a->rot_half, p.amp = a->rot ? a->rot_amp : 1.f;
  p.mkpool = a->mean_k, p.mvpool = a->mean_v, p.mtable = a->mean_table, p.mpages = a->mean_pages, p.pool = a->pool;
  p.convw = a->conv_w, p.ring = a->ring, p.map = a->map, p.taps = a->taps, p.qout = a->q_out, p.ldqo = a->ldqo, p.vkeys = a->shared_kv;
  if (a->prepared) p.unit = p.whole = p.rot = p.taps = p.half = 0, p.amp = 1.f, p.qgain = p.kgain = nullptr;
  p.nsplit = 1;
  return p;
}

int check(const exo_paged_attn* a, const char* what) {
  EXO_REQUIRE(a && (a->dtype == 0 || a->dtype == 1), "%s: bad dtype", what);
  EXO_REQUIRE(a->n > 0 && a->n <= 65535 && a->heads > 0 && a->kv_heads > 0 && a->heads % a->kv_heads == 0,
              "%s: bad counts (n=%d heads=%d kv_heads=%d)", what, a->n, a->heads, a->kv_heads);
  EXO_REQUIRE(a->dim > 0 && a->vdim > 0 && a->dim <= 256 && a->vdim <= 256, "%s: head sizes %d / %d not in 1..256", what,
              a->dim, a->vdim);
  EXO_REQUIRE(a->ldk % 32 == 0 && a->ldk >= a->dim && a->ldk <= 256 && a->ldv % 32 == 0 && a->ldv >= a->vdim && a->ldv <= 256,
              "%s: pool strides %d / %d do not fit head sizes %d / %d", what, a->ldk, a->ldv, a->dim, a->vdim);
  EXO_REQUIRE(a->qkv && a->k_pool && a->v_pool && a->table && a->max_pages > 0, "%s: null pointer", what);
  EXO_REQUIRE(!a->gate || a->ldg >= a->heads, "%s: %d gates per row for %d heads", what, a->ldg, a->heads);
  EXO_REQUIRE(a->rot >= 0 && a->rot % 2 == 0 && a->rot <= a->dim && a->rot <= kMaxRot && (!a->rot || a->freq) && !(a->rot && a->unit_qk),
              "%s: %d rotated dimensions of %d (an even number, angles given, no norm per head)", what, a->rot, a->dim);
  EXO_REQUIRE(!a->whole_norm || (!a->unit_qk && a->q_gain && a->k_gain), "%s: one norm, with gains over the whole projections", what);
  EXO_REQUIRE(a->softcap >= 0.f && (!a->v_mix || a->ldmix >= a->kv_heads * a->vdim), "%s: bad cap or mixed values", what);
  EXO_REQUIRE(a->unit_qk || a->whole_norm || (!a->q_gain && !a->k_gain), "%s: a query / key gain belongs to the norm", what);
  EXO_REQUIRE(a->keep_first >= 0 && a->window >= 0, "%s: negative window", what);
  EXO_REQUIRE(!a->out_gate || a->ldog >= a->heads * a->vdim, "%s: %d gates per row for %d outputs", what, a->ldog, a->heads * a->vdim);
  EXO_REQUIRE(a->pool >= 0 && (!a->pool || (a->window > 0 && !a->keep_first && !a->slopes && a->mean_k && a->mean_v && a->mean_table && a->mean_pages > 0)),
              "%s: means of blocks of %d positions need a window, no kept positions and no slopes, and their pools", what, a->pool);
  EXO_REQUIRE(!a->weight_bias || (!a->plus_one && a->softcap == 0.f && !a->slopes), "%s: weights that are no softmax go without its options", what);
  EXO_REQUIRE(a->taps >= 0 && (!a->taps || (a->conv_w && a->ring && a->map && !a->unit_qk && !a->whole_norm)), "%s: incomplete convolution of %d taps", what, a->taps);
  EXO_REQUIRE(!a->shared_kv || (a->dim == a->vdim && !a->v_mix && !a->unit_qk && !a->whole_norm), "%s: values of size %d cannot be keys of size %d", what, a->vdim, a->dim);
  return EXO_OK;
}

int row_columns(const exo_paged_attn* a) {  // of queries, keys and values
  return (a->heads + a->kv_heads) * a->dim + (a->shared_kv ? 0 : a->kv_heads * a->vdim);
}

template <typename T, int DMAX, bool FUSE, int MODE>
int launch_rows(const Params& p, hipStream_t st) {
  constexpr int qbytes = 16 * (DMAX + 16 / (int)sizeof(T)) * (int)sizeof(T);
  const int obytes = kRowWaves * p.gsz * (p.ldv + 4) * 4;
  const int lds = qbytes > obytes ? qbytes : obytes;  // at most 65 KiB (16 heads x 256 values x 4 waves)
  exo_note_variant("paged_rows<%s,%d,%s,%s> splits=%d rows=%d", sizeof(T) == 2 ? "bf16" : "f32", DMAX, FUSE ? "fused" : "plain",
                   MODE == kSigmoid ? "sigmoid" : MODE == kMore ? "more" : "softmax", p.nsplit, p.n);
  static bool done = false;
  const auto fn = paged_rows_kernel<T, DMAX, FUSE, MODE>;
  if (!done) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
    if (e != hipSuccess) {
      exo_set_error("exo_paged_attn_rows: cannot raise the dynamic LDS limit: %s", hipGetErrorString(e));
      return EXO_ERR_HIP;
    }
    done = true;
  }
  fn<<<dim3(p.nsplit, p.G * p.hgroups, p.n), 64 * kRowWaves, lds, st>>>(p);
  return EXO_OK;
}

template <typename T, int DMAX>
int launch_rows_f(const Params& p, bool fuse, hipStream_t st) {
  const int mode = mode_of(p);
  if (mode == kSigmoid) return fuse ? launch_rows<T, DMAX, true, kSigmoid>(p, st) : launch_rows<T, DMAX, false, kSigmoid>(p, st);
  if (mode == kMore) return fuse ? launch_rows<T, DMAX, true, kMore>(p, st) : launch_rows<T, DMAX, false, kMore>(p, st);
  return fuse ? launch_rows<T, DMAX, true, kPlain>(p, st) : launch_rows<T, DMAX, false, kPlain>(p, st);
}
template <typename T>
int launch_rows_d(const Params& p, int d, bool fuse, hipStream_t st) {
  return d <= 64 ? launch_rows_f<T, 64>(p, fuse, st) : d <= 128 ? launch_rows_f<T, 128>(p, fuse, st) : launch_rows_f<T, 256>(p, fuse, st);
}

template <int DK, int DV, int HW, bool ROWS = false, int MODE = kPlain>
int launch_prompt(const Params& p, hipStream_t st, const Expanded& x = Expanded{}) {
  constexpr int lds = prompt_lds<DK, DV>();
  static bool done = false;
  const auto fn = paged_prompt_kernel<DK, DV, HW, ROWS, MODE>;
  if (!done && lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      exo_set_error("exo_paged_attn_prompt: cannot raise the dynamic LDS limit: %s", hipGetErrorString(e));
      return EXO_ERR_HIP;
    }
  }
  done = true;
  const int group = p.H / p.G;
  const dim3 grid(p.n, p.G * ((group + HW - 1) / HW));
  exo_note_variant("paged_prompt<%d,%d,%d,%s,%s> grid=%dx%d", DK, DV, HW, ROWS ? "rows" : "pool", MODE == kSigmoid ? "sigmoid" : MODE == kMore ? "more" : "softmax",
                   (int)grid.x, (int)grid.y);
  fn<<<grid, 256, lds, st>>>(p, x);
  return EXO_OK;
}
template <int D, int MODE>
int launch_prompt_w(const Params& p, hipStream_t st) {
  const int group = p.H / p.G;
  return group >= 3 ? launch_prompt<D, D, 4, false, MODE>(p, st)
                    : group == 2 ? launch_prompt<D, D, 2, false, MODE>(p, st) : launch_prompt<D, D, 1, false, MODE>(p, st);
}
template <int D>
int launch_prompt_h(const Params& p, hipStream_t st) {
  const int mode = mode_of(p);
  return mode == kSigmoid ? launch_prompt_w<D, kSigmoid>(p, st) : mode == kMore ? launch_prompt_w<D, kMore>(p, st) : launch_prompt_w<D, kPlain>(p, st);
}

}  // namespace

extern "C" int exo_paged_append(const exo_paged_attn* a, exo_stream_t stream) {
  const int rc = check(a, "exo_paged_append");
  if (rc) return rc;
  EXO_REQUIRE(a->slot && a->pos && a->ldq >= row_columns(a),
              "exo_paged_append: rows of %d elements do not hold q, k and v", a->ldq);
  EXO_REQUIRE(!a->whole_norm && !a->rot && !a->v_mix && !a->taps && !a->shared_kv,
              "exo_paged_append: a norm over whole projections, rotations, convolutions and values of other kinds need exo_paged_prepare");
  const Params p = params_of(a);
  const dim3 grid((p.n + kAppendRows - 1) / kAppendRows, (2 * p.G + 3) / 4);
  if (a->dtype == 0)
    paged_append_kernel<bf16_t><<<grid, 256, 0, (hipStream_t)stream>>>(p);
  else
    paged_append_kernel<float><<<grid, 256, 0, (hipStream_t)stream>>>(p);
  EXO_CHECK_LAUNCH("exo_paged_append");
  return EXO_OK;
}

extern "C" int exo_paged_prepare(const exo_paged_attn* a, exo_stream_t stream) {
  const int rc = check(a, "exo_paged_prepare");
  if (rc) return rc;
  EXO_REQUIRE(a->slot && a->pos && !a->prepared && !a->unit_qk && a->ldq >= row_columns(a),
              "exo_paged_prepare: rows of %d elements do not hold q, k and v, or a norm per head", a->ldq);
  EXO_REQUIRE(a->taps ? a->q_out && a->q_out != a->qkv && a->ldqo >= a->heads * a->dim : !a->q_out,
              "exo_paged_prepare: convolved queries (and no others) need a place of their own");
  const Params p = params_of(a);
  // (a norm over whole rows reads all heads: one part, since the queries are written in place)
  const int qparts = p.whole ? 1 : max(1, min(min(p.H, 8), p.H * p.D / 1024));
  const dim3 grid((p.n + kAppendRows - 1) / kAppendRows, 1 + qparts);
  const int64_t lds = (int64_t)kAppendRows * (p.G * p.D + 8) * (a->dtype == 0 ? 2 : 4);
  const bool staged = p.vkeys && lds <= 32 * 1024;
  if (a->dtype == 0)
    paged_prepare_kernel<bf16_t><<<grid, 64 * kAppendRows, staged ? lds : 0, (hipStream_t)stream>>>(p, staged);
  else
    paged_prepare_kernel<float><<<grid, 64 * kAppendRows, staged ? lds : 0, (hipStream_t)stream>>>(p, staged);
  const dim3 keepers(exo_ceil_div(p.n, 64), kKeepers, exo_ceil_div((p.H + p.G) * p.D, kKept));
  if (p.taps && a->dtype == 0)
    paged_keep_kernel<bf16_t><<<keepers, 256, 0, (hipStream_t)stream>>>(p);
  else if (p.taps)
    paged_keep_kernel<float><<<keepers, 256, 0, (hipStream_t)stream>>>(p);
  EXO_CHECK_LAUNCH("exo_paged_prepare");
  return EXO_OK;
}

extern "C" int exo_paged_means(const exo_paged_attn* a, exo_stream_t stream) {
  const int rc = check(a, "exo_paged_means");
  if (rc) return rc;
  EXO_REQUIRE(a->pool && a->list, "exo_paged_means: no blocks");
  const Params p = params_of(a);
  if (a->dtype == 0)
    paged_means_kernel<bf16_t><<<dim3(p.n, p.G), 256, 0, (hipStream_t)stream>>>(p);
  else
    paged_means_kernel<float><<<dim3(p.n, p.G), 256, 0, (hipStream_t)stream>>>(p);
  EXO_CHECK_LAUNCH("exo_paged_means");
  return EXO_OK;
}

extern "C" int64_t exo_paged_attn_workspace(int n, int heads, int vdim, int nsplit) {
  return ((int64_t)n * heads * nsplit * (vdim + 2) + kCounters) * 4;
}

extern "C" int exo_paged_attn_rows(const exo_paged_attn* a, int nsplit, int append, void* workspace,
                                   int64_t workspace_bytes, exo_stream_t stream) {
  const int rc = check(a, "exo_paged_attn_rows");
  if (rc) return rc;
  EXO_REQUIRE(a->slot && a->pos && a->out && a->ldo >= a->heads * a->vdim && a->ldq >= a->heads * a->dim,
              "exo_paged_attn_rows: bad rows or output");
  EXO_REQUIRE(!append || a->ldq >= row_columns(a),
              "exo_paged_attn_rows: rows of %d elements do not hold q, k and v", a->ldq);
  EXO_REQUIRE(nsplit >= 1 && nsplit <= 64 &&
                  (nsplit == 1 || (workspace && (int64_t)a->n * a->heads <= kCounters && workspace_bytes >= exo_paged_attn_workspace(a->n, a->heads, a->vdim, nsplit))),
              "exo_paged_attn_rows: workspace too small for %d splits", nsplit);
  Params p = params_of(a);
  p.nsplit = nsplit;
  const int group = p.H / p.G;
  // few (sequence, kv head) pairs: fewer query heads per workgroup, whose keys then come from the
  // L2 again, but whose merge is shorter
  p.hgroups = (group + 15) / 16;
  while (nsplit > 1 && p.hgroups < group && p.hgroups < 16 && (int64_t)a->n * p.G * p.hgroups * nsplit * 2 <= 256) p.hgroups *= 2;
  if (p.hgroups > group) p.hgroups = group;
  p.gsz = (group + p.hgroups - 1) / p.hgroups, p.group = group;
  p.hgroups = (group + p.gsz - 1) / p.gsz;  // (none without a head)
  p.counters = reinterpret_cast<int*>(workspace);
  p.ws = nsplit > 1 ? reinterpret_cast<float*>(workspace) + kCounters : nullptr;
  const int d = p.ldk > p.ldv ? p.ldk : p.ldv;
  const hipStream_t st = (hipStream_t)stream;
  const int rc2 = a->dtype == 0 ? launch_rows_d<bf16_t>(p, d, append != 0, st) : launch_rows_d<float>(p, d, append != 0, st);
  if (rc2) return rc2;
  EXO_CHECK_LAUNCH("exo_paged_attn_rows");
  return EXO_OK;
}

extern "C" int exo_paged_prompt_block(int heads, int kv_heads) {
  const int group = kv_heads > 0 ? heads / kv_heads : 0;
  return group >= 3 ? 32 : group == 2 ? 64 : 128;
}

extern "C" int exo_paged_attn_prompt(const exo_paged_attn* a, exo_stream_t stream) {
  const int rc = check(a, "exo_paged_attn_prompt");
  if (rc) return rc;
  EXO_REQUIRE(a->dtype == 0, "exo_paged_attn_prompt: bf16 only");
  EXO_REQUIRE(a->prepared || !(a->whole_norm || a->rot || a->taps), "exo_paged_attn_prompt: queries must be prepared (exo_paged_prepare)");
  EXO_REQUIRE(a->list && a->out && a->ldo >= a->heads * a->vdim && a->ldq >= a->heads * a->dim && a->ldo % 4 == 0 &&
                  a->ldk % 8 == 0,
              "exo_paged_attn_prompt: bad rows or output");
  const Params p = params_of(a);
  const int d = p.ldk > p.ldv ? p.ldk : p.ldv;
  const hipStream_t st = (hipStream_t)stream;
  const int rc2 = d <= 64 ? launch_prompt_h<64>(p, st) : d <= 128 ? launch_prompt_h<128>(p, st) : launch_prompt_h<256>(p, st);
  if (rc2) return rc2;
  EXO_CHECK_LAUNCH("exo_paged_attn_prompt");
  return EXO_OK;
}

extern "C" int exo_latent_prompt(const exo_latent_prompt_args* a, exo_stream_t stream) {
  EXO_REQUIRE(a && a->q && a->k && a->k_rot && a->v && a->list && a->out && a->n > 0 && a->heads > 0 && a->heads <= 65535 && a->vdim > 0,
              "exo_latent_prompt: null pointer or bad counts");
  EXO_REQUIRE(a->d8 > 0 && a->d8 % 8 == 0 && a->r8 >= 8 && a->r8 % 8 == 0 && a->d8 + a->r8 <= 256 && a->vdim <= 256,
              "exo_latent_prompt: key parts %d and %d (multiples of 8, at most 256 together), values %d", a->d8, a->r8, a->vdim);
  EXO_REQUIRE(a->ldk >= a->heads * a->d8 && a->ldk % 8 == 0 && a->ldv % 64 == 0 && a->ldq % 8 == 0 && a->q_head % 8 == 0 &&
                  a->q_head >= a->d8 && a->rot_col % 8 == 0 && a->rot_col >= a->heads * a->q_head &&
                  a->ldq >= a->rot_col + a->heads * a->r8 && a->ldo >= a->heads * a->vdim && a->ldo % 4 == 0,
              "exo_latent_prompt: bad row strides");
  Params p{};
  p.qkv = a->q, p.list = a->list, p.out = a->out, p.scale = a->scale, p.n = a->n, p.H = p.G = a->heads, p.D = a->d8, p.E = a->vdim;
  p.ldq = a->ldq, p.ldo = a->ldo, p.size = 0x3FFFFFFF, p.nsplit = 1;
  const Expanded x{(const bf16_t*)a->k, (const bf16_t*)a->k_rot, (const bf16_t*)a->v, a->ldk, a->ldv, a->d8, a->r8, a->q_head, a->rot_col};
  const int dk = a->d8 + a->r8;
  const hipStream_t st = (hipStream_t)stream;
  const int rc = dk <= 128 && a->vdim <= 128   ? launch_prompt<128, 128, 1, true>(p, st, x)
                 : dk <= 192 && a->vdim <= 128 ? launch_prompt<192, 128, 1, true>(p, st, x)
                                               : launch_prompt<256, 256, 1, true>(p, st, x);
  if (rc) return rc;
  EXO_CHECK_LAUNCH("exo_latent_prompt");
  return EXO_OK;
}
