// Quantised matmul of 9 to 64 rows (short prompts, batches of an 8-bit model): y[M,N] = x[M,K] @ dq(W)[N,K]^T, or the gate / up pair
// with its SwiGLU.
//
// A launch of so few rows streams its weights once and has little arithmetic per weight, so what
// counts is that every CU has weights on their way all the time and that nothing but the result leaves.
// One workgroup of eight waves per CU owns NT tiles of 16 weight rows (pair: 8 rows of each matrix per
// tile) over the WHOLE of K; its waves take the K steps of 64 in turn, each for itself: a wave loads its
// step's activations (64 rows of 128 bytes) straight into LDS slots of its own and its weights into
// registers, two steps ahead, without a barrier, and multiplies 16 x 16 x 32 products.  The waves' float32
// sums meet in LDS once, at the end, in a fixed order.
//  * scales and biases of the workgroup's rows go to LDS first, as pairs: loaded per lane and step they
//    are 2 bytes out of a line each.
//  * rows of an activation slot are 128 bytes; chunk c of row r sits at c ^ (r / 2 % 8), so that an
//    operand read of 16 rows touches all 64 banks.
//  * the activations of a step are in registers before the products start, so its slot is refilled at once.
//  * every workgroup reads all activations (64 rows x 4096: 512 KB, as much as 228 rows of 4-bit weights and
//    scales); where K is long and the columns are few, one tile of columns per CU, that is most of the launch.  Such
//    launches give a workgroup four tiles and a quarter of K, and a reduce launch adds the quarters.
// 4-bit under 61 rows: pair of 14336x4096 52 -> 34 us (two products of 21, their reduce launches and the SwiGLU before:
// 57), 6144x4096 23 -> 14, 4096x4096 17 -> 11, 4096x14336 30 -> 25; under 20 rows the pair 49 -> 26.
// What bounds it: the dequantisation alone is 11 us of the pair's vector issue and a plain read of
// its weights 12; the rest is the start (scales, first steps: two memory latencies), the
// activations through L2 (3.4 us at a CU's 64 bytes per cycle) and the sums' way through LDS.
// Where a launch is one round of such workgroups it replaces tiles of 32 or 64 x 256 with K split over
// workgroups, whose partial sums (up to 16 times the output in float32) go to memory and come back through a
// second launch; where not, those stay (exo_qmm_short_beats_split, exo_qmm_short_fits).
#include "dequant.h"
#include "qmm_short.h"

#include "../../include/exo_mi355x.h"

#include <algorithm>

namespace {

constexpr int kWaves = 8;
constexpr int kCUs = 256;

struct ShortParams {
  const bf16_t* x;
  const uint32_t *w, *w2;
  const bf16_t *s, *b, *s2, *b2;
  const bf16_t* residual;
  bf16_t* y;
  int M, N, K, tiles;  // tiles of columns
  int groups;          // of 64 elements of K that a workgroup takes: all, or a part whose float32 sums go to `part`
  float* part;         // [parts][part_stride]
  size_t part_stride;
  int vec;                         // rows of scales and biases are whole, aligned 16-byte pieces
};

template <int N>
__device__ __forceinline__ void wait_vm() {
  __builtin_amdgcn_s_waitcnt((N & 15) | 0x0F70 | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// 16 bytes per lane from a buffer straight into LDS: lane l of the wave writes lds_base + 16*l; counted by vmcnt
__device__ __forceinline__ void load_to_lds16(__amdgpu_buffer_rsrc_t rsrc, void* lds_base, uint32_t voffset,
                                              uint32_t soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)lds_base, 16, voffset, soffset,
                                           0, 0);
}

template <int BITS, bool PAIR, int MT, int NT>
__global__ __launch_bounds__(64 * kWaves) void qmm_short_kernel(const ShortParams p) {
  constexpr int SLOT = MT * 16 * 128;              // bytes of a step's activations
  constexpr int XR = MT * 2;                       // 1 KB loads of a step's activations
  constexpr int COLS = PAIR ? 8 : 16;              // output columns of a tile
  constexpr int WORDS = BITS / 2;                  // 32-bit words of a lane's 16 codes
  constexpr int XBYTES = kWaves * 2 * SLOT;
  __shared__ __attribute__((aligned(1024))) char lds[XBYTES + kQmmShortMaxK * 4 / 64 * 16];
  static_assert(NT * MT * 1024 * (kWaves / 2) <= XBYTES, "half of the waves' sums in the activation slots");

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile0 = (int)blockIdx.x * NT;
  const int GA = p.K >> 6, g0 = (int)blockIdx.y * p.groups, G = min(p.groups, GA - g0);  // this workgroup's groups

  // scales and biases of the workgroup's rows: [tile][group][row] as (scale, bias)
  uint32_t* const sb = reinterpret_cast<uint32_t*>(lds + XBYTES);
  const int n16 = lane & 15, g4 = lane >> 4;

  // activations: lane l of load j takes row 8 j + l / 8, chunk (l % 8) ^ (row / 2 % 8)
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.x), 0, -1, 0x00020000);
  uint32_t xoff[XR];
#pragma unroll
  for (int j = 0; j < XR; ++j) {
    const int row = 8 * j + (lane >> 3), chunk = (lane & 7) ^ ((row >> 1) & 7);
    xoff[j] = ((uint32_t)min(row, p.M - 1) * (uint32_t)p.K + g0 * 64) * 2 + chunk * 16;
  }
  char* const mine = lds + wave * (2 * SLOT);
  auto load_x = [&](int slot, int j, int k0) {
      load_to_lds16(rx, mine + slot * SLOT + j * 1024, xoff[j], k0 * 2);
  };
  // weights: lane (row n16, quarter g4) takes the 16 codes k0 + 16 g4 ..
  const size_t wpr = (size_t)p.K * BITS / 32;
  const bool up = PAIR && n16 >= 8;
  const uint32_t* const wm = (up ? p.w2 : p.w) + g0 * (BITS * 2) + g4 * WORDS;
  struct Codes {
    uint32_t q[WORDS];
  };
  const uint32_t* wrow[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
    wrow[i] = wm + (size_t)min((tile0 + i) * COLS + (PAIR ? n16 & 7 : n16), p.N - 1) * wpr;
  auto load_w = [&](Codes(&c)[NT], int i, int k0) {
      const uint32_t* at = wrow[i] + (k0 >> 6) * (BITS * 2);
      if (BITS == 4) {
        const uint2 v = *reinterpret_cast<const uint2*>(at);
        c[i].q[0] = v.x, c[i].q[1] = v.y;
      } else {
        const uint4 v = *reinterpret_cast<const uint4*>(at);
        c[i].q[0] = v.x, c[i].q[1] = v.y, c[i].q[WORDS - 2] = v.z, c[i].q[WORDS - 1] = v.w;
      }
  };

  floatx4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[i][m] = floatx4{0.f, 0.f, 0.f, 0.f};

  // scales and biases of eight groups of a row at a time (rows of whole 16-byte pieces), all requested before
  // anything else; piece e = (tile row, eight groups)
  constexpr int PIECES = kQmmShortMaxK / 64 * 16 / 8 / (64 * kWaves);
  const int G8 = G >> 3, pieces = NT * 16 * G8;
  auto row_at = [&](int row) {
    const int n = row & 15;
    return (size_t)min((tile0 + (row >> 4)) * COLS + (PAIR ? n & 7 : n), p.N - 1) * GA + g0;
  };
  uint4 vs[PIECES], vb[PIECES];
  if (p.vec) {
#pragma unroll
    for (int q = 0; q < PIECES; ++q) {
      const int e = min(tid + q * 64 * kWaves, pieces - 1), row = e / G8;
      const bool second = PAIR && (row & 15) >= 8;
      const size_t at = row_at(row) + (e - row * G8) * 8;
      vs[q] = *reinterpret_cast<const uint4*>((second ? p.s2 : p.s) + at);
      vb[q] = *reinterpret_cast<const uint4*>((second ? p.b2 : p.b) + at);
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  // steps of this wave: wave, wave + 8, ...; requests past the last one repeat it and are never used
  const int steps = (G - wave + kWaves - 1) / kWaves;
  auto k_of = [&](int i) { return (wave + kWaves * min(i, steps - 1)) * 64; };
  Codes w0[NT], w1[NT];
  if (steps > 0) {
#pragma unroll
    for (int j = 0; j < NT; ++j) load_w(w0, j, k_of(0));
#pragma unroll
    for (int j = 0; j < XR; ++j) load_x(0, j, k_of(0));
    // (step 0 waits by count for all but the last XR + NT requests: none of step 1 may be sent ahead of these)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NT; ++j) load_w(w1, j, k_of(1));
#pragma unroll
    for (int j = 0; j < XR; ++j) load_x(1, j, k_of(1));
  }
  __builtin_amdgcn_sched_barrier(0);
  if (p.vec) {
#pragma unroll
    for (int q = 0; q < PIECES; ++q) {
      const int e = tid + q * 64 * kWaves, row = e / G8, g = (e - row * G8) * 8;
      if (e >= pieces) break;
      const uint32_t sw[4] = {vs[q].x, vs[q].y, vs[q].z, vs[q].w}, bw[4] = {vb[q].x, vb[q].y, vb[q].z, vb[q].w};
      uint32_t* to = sb + ((row >> 4) * G + g) * 16 + (row & 15);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        to[(2 * c) * 16] = (sw[c] & 0xffffu) | bw[c] << 16;
        to[(2 * c + 1) * 16] = sw[c] >> 16 | (bw[c] & 0xffff0000u);
      }
    }
  } else {
    for (int e = tid; e < NT * 16 * G; e += 64 * kWaves) {
      const int row = e / G, g = e - row * G;
      const bool second = PAIR && (row & 15) >= 8;
      const size_t at = row_at(row) + g;
      const uint32_t s = (second ? p.s2 : p.s)[at], b = (second ? p.b2 : p.b)[at];
      sb[((row >> 4) * G + g) * 16 + (row & 15)] = s | b << 16;
    }
  }
  // (No fence.  The first two steps have landed here all the same: the requests stand in branches, across which the
  // compiler cannot count, so that its waits for the scales are waits for everything.)
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);

  float most = 0.f;  // 4 bits: the largest scale so far (from 2^104 on the steps do not make operands right)
  auto step = [&](Codes(&w)[NT], int slot, int i) {
    // x(i) and w(i) are here; those of step i + 1 may still be out
    wait_vm<XR + NT>();
    bf16x8_t a[2][MT];
    const char* xs = mine + slot * SLOT;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int row = m * 16 + n16;
        a[t][m] = *reinterpret_cast<const bf16x8_t*>(xs + row * 128 + ((2 * g4 + t) ^ ((row >> 1) & 7)) * 16);
      }
    uint32_t sc[NT];
    const int g = wave + kWaves * i;
#pragma unroll
    for (int j = 0; j < NT; ++j) sc[j] = sb[(j * G + g) * 16 + n16];
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the slot has been read
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    // Products of one operand (tile q / 2, half q % 2 of the step), the next operand made between them; behind
    // a tile its codes of step i + 2 are requested and a share of that step's activations.
    const int kn = k_of(i + 2);
    u32x4 bw[2];
    PieceCodes pc{};
    GroupScale<BITS> gs{};
    if (BITS == 4) {
#pragma unroll
      for (int j = 0; j < NT; j += 2) note_scales(most, bf_lo(sc[j]), bf_lo(sc[min(j + 1, NT - 1)]));
    }
    auto piece = [&](int q, int d) {  // two of an operand's eight values
      const int j = q >> 1, t = q & 1;
      if (d == 0 && t == 0) gs = group_scale<BITS>(bf_lo(sc[j]), bf_hi(sc[j]));
      piece_codes<BITS>(pc, d, w[j].q[BITS == 4 ? t : (2 * t) & (WORDS - 1)], w[j].q[BITS == 4 ? t : (2 * t + 1) & (WORDS - 1)]);
      bw[q & 1][piece_reg<BITS>(d)] = piece_value<BITS>(d, pc, gs);
    };
#pragma unroll
    for (int d = 0; d < 4; ++d) piece(0, d);
#pragma unroll
    for (int q = 0; q < 2 * NT; ++q) {
      const int j = q >> 1, t = q & 1;
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        acc[j][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t][m], __builtin_bit_cast(bf16x8_t, bw[q & 1]), acc[j][m], 0, 0, 0);
        if (q + 1 < 2 * NT) {
#pragma unroll
          for (int d = m * 4 / MT; d < (m + 1) * 4 / MT; ++d) piece(q + 1, d);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (t == 0) continue;
      load_w(w, j, kn);
#pragma unroll
      for (int c = j * XR / NT; c < (j + 1) * XR / NT; ++c) load_x(slot, c, kn);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int i = 0;
  for (; i + 2 <= steps; i += 2) {
    step(w0, 0, i);
    step(w1, 1, i + 1);
  }
  if (i < steps) step(w0, 0, i);

  // Weights of large scales (dequant.h): the wave's sums once more, in the same order, one step at a time and without the
  // activations' slots
  if constexpr (BITS == 4) {
    if (__builtin_expect(any_large(most), 0)) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[j][m] = floatx4{0.f, 0.f, 0.f, 0.f};
      for (int n = 0; n < steps; ++n) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          load_w(w0, j, k_of(n));
          const uint32_t sc = sb[(j * G + wave + kWaves * n) * 16 + n16];
          const GroupScale<BITS> gs = group_scale<BITS>(bf_lo(sc), bf_hi(sc));
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            bf16x8_t w = dequant_words8<BITS>(w0[j].q[t], 0, gs);
            large_scales<BITS>(w, w0[j].q[t], bf_lo(sc), gs.b);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
              const uint32_t at = ((uint32_t)min(m * 16 + n16, p.M - 1) * (uint32_t)p.K + g0 * 64 + (2 * g4 + t) * 8) * 2;
              const bf16x8_t a = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rx, at, k_of(n) * 2, 0));
              acc[j][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w, acc[j][m], 0, 0, 0);
              __builtin_amdgcn_sched_barrier(0);  // (no registers for this)
            }
          }
        }
      }
    }
  }

  // the waves' sums: four of them through LDS into the other four, then all eight waves add the four
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the repeated requests have landed
  __syncthreads();
  float* const ex = reinterpret_cast<float*>(lds);
  constexpr int PER = NT * MT * 256;  // floats of a wave's sums
  if (wave >= 4) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) ex[(wave - 4) * PER + ((j * MT + m) * 4 + r) * 64 + lane] = acc[j][m][r];
  }
  __syncthreads();
  if (wave < 4) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float* at = &ex[wave * PER + ((j * MT + m) * 4 + r) * 64 + lane];
          *at = acc[j][m][r] + *at;
        }
  }
  __syncthreads();
  for (int e = tid; e < PER; e += 64 * kWaves) {
    const int l = e & 63, c = l & 15, r = (e >> 6) & 3, jm = e >> 8, j = jm / MT, m = jm - j * MT;
    if (PAIR && c >= 8) continue;
    const int row = m * 16 + 4 * (l >> 4) + r, col = (tile0 + j) * COLS + c;
    if (row >= p.M || col >= p.N) continue;
    auto sum = [&](int at) { return ((ex[at] + ex[PER + at]) + ex[2 * PER + at]) + ex[3 * PER + at]; };
    const size_t o = (size_t)row * p.N + col;
    if (!PAIR && p.part) {
      p.part[(size_t)blockIdx.y * p.part_stride + o] = sum(e);
      continue;
    }
    float v = bf2f(f2bf(sum(e)));
    if (PAIR) {  // (the projections rounded to bf16 as two launches would leave them)
      const float u = bf2f(f2bf(sum(e + 8)));
      v = v / (1.f + __expf(-v)) * u;
    } else if (p.residual) {
      v += bf2f(p.residual[o]);
    }
    p.y[o] = f2bf(v);
  }
}

template <int BITS, bool PAIR, int MT, int NT>
void launch_tiles(const ShortParams& p, int parts, hipStream_t st) {
  exo_note_variant("qmm_short<%d,%s,%d,%d> parts=%d", BITS, PAIR ? "pair" : "one", MT, NT, parts);
  qmm_short_kernel<BITS, PAIR, MT, NT><<<dim3(exo_ceil_div(p.tiles, NT), parts), 64 * kWaves, 0, st>>>(p);
}

// Tiles per workgroup: one workgroup per CU, as many tiles each as that takes - as far as the scales of K elements
// per row fit into LDS.  (Five and six run as seven, on fewer CUs: pair of K = 4096 under 33 rows, 10240 columns
// 30.7 us, 12288 32.1, 14336 33.4.)
int tiles_per_wg(int wanted, int K) {
  const int fit = kQmmShortMaxK / K, nt = std::min(wanted, fit);
  return nt >= 5 && fit >= 7 ? 7 : nt >= 4 ? 4 : std::max(nt, 1);
}

template <int BITS, bool PAIR, int MT>
void launch(const ShortParams& p, int parts, hipStream_t st) {
  switch (tiles_per_wg(parts > 1 ? parts : exo_ceil_div(p.tiles, kCUs), p.groups * 64)) {
    case 7: return launch_tiles<BITS, PAIR, MT, 7>(p, parts, st);
    case 4: return launch_tiles<BITS, PAIR, MT, 4>(p, parts, st);
    case 3: return launch_tiles<BITS, PAIR, MT, 3>(p, parts, st);
    case 2: return launch_tiles<BITS, PAIR, MT, 2>(p, parts, st);
    default: return launch_tiles<BITS, PAIR, MT, 1>(p, parts, st);
  }
}

template <int BITS, bool PAIR>
void launch_rows(const ShortParams& p, int parts, hipStream_t st) {
  if (p.M <= 32)
    launch<BITS, PAIR, 2>(p, parts, st);
  else
    launch<BITS, PAIR, 4>(p, parts, st);
}

}  // namespace

// Four quarters of K where one tile per CU would make every CU read 1 MB of activations and more: 4096x14336 4-bit
// under 61 rows 37 -> 25 us, 2048x8192 16.8 -> 15.8 (4096x4096, whole: 11 us).
// (Under up to 32 rows the tile that splits K is ahead beyond K = 16384, 4096x28672 28.3 us against 29.6, and
// on narrow matrices, 128x8192 10.7 against 11.6, 1024x12288 0.92 of its speed.)
int exo_qmm_short_parts(int M, int N, int K) {
  return exo_ceil_div(N, 16) <= kCUs && K >= 8192 && (M > 32 || (N >= 2048 && K <= 16384)) && K % (4 * 512) == 0 ? 4 : 1;
}

// Up to 8192 rows of weights a CU has four tiles at most, and the 128-row tile half of the chip: ahead by a third and
// more, until K is so long that the activations of every workgroup outweigh it (8192x11008 under 64 rows 0.88 of the
// other's speed, under 32 rows 1.13).  Beyond that the two are rounds of workgroups against rounds of workgroups,
// and the times below (us) hold within 7 % (here) and 12 % over 512 <= K <= 28672 and up to 53248 rows.  Pairs, 4-bit,
// us, 128-row tile -> here: 14336x4096 33 rows 51 -> 33, 16384x2048 (a round against two) 33 rows 0.69 of
// the speed, 16384x8192 1.33, 28672x1024 17 rows 1.03, 64 rows 0.78, 14336x768 17 rows 1.05, 64 rows 0.80.
// Products of more than 32768 rows are the matrices of a vocabulary, alone: 65536x4096 17 rows 82 -> 74, 33
// rows 82 -> 91; 128256x4096 17 rows 161 -> 126, 64 rows 171 -> 170; 128256x2048 17 rows 79 -> 83, 64 rows 85 -> 113.
bool exo_qmm_short_fits(int M, int N, int K, int bits) {
  if (!exo_qmm_short_can(M, K)) return false;
  if (N <= 8192) return K <= 8192 || (M <= 32 && K <= 16384);
  if (N > 32768 && (M > 32 || K < 3072)) return false;
  const int tiles = exo_ceil_div(N, 8), nt = tiles_per_wg(exo_ceil_div(tiles, kCUs), K);
  const int rounds = exo_ceil_div(exo_ceil_div(tiles, nt), kCUs), rounds128 = exo_ceil_div(exo_ceil_div(N, 64), kCUs);
  const double k = K / 1000., per_tile = bits == 4 ? 0.58 : 0.85;
  const double whole = M <= 32 ? 7.3 + k * (per_tile * nt + 0.4) : 10.5 + k * (per_tile * nt + 0.9);
  const double here = K % 512 == 0 ? whole : 1.2 * whole;  // (scales that are no whole 16-byte pieces)
  const double other = bits == 4 ? 3.7 + 9.75 * k : 2.6 + 12 * k;
  return rounds * here <= (M > 32 && K > 8192 ? 0.9 : 0.95) * (rounds128 * other);
}

// One round of workgroups, each with the whole of a K of up to 8192 or with a quarter of it.  A second round does not
// overlap the first one's end, and every workgroup reads all activations, which over a long K is more than its
// weights.  4-bit under 64 rows, us, split tile -> here: 16384x8192 (four tiles each) 47 -> 42, 24576x8192 (two
// rounds) 64 -> 78, 8192x14336 41 -> 48, 8192x28672 66 -> 139, 4096x11008 27 -> 32, 32768x2048 (two rounds) 29 -> 45;
// under 17 rows 24576x8192 52.5 -> 54, 8192x28672 53 -> 73, 32768x768 14.5 -> 23.
bool exo_qmm_short_beats_split(int M, int N, int K) {
  if (exo_qmm_short_parts(M, N, K) > 1) return true;
  const int tiles = exo_ceil_div(N, 16);
  return K <= (tiles <= kCUs ? 8191 : 8192) && exo_ceil_div(tiles, tiles_per_wg(exo_ceil_div(tiles, kCUs), K)) <= kCUs;
}

void exo_qmm_short(const bf16_t* x, const uint32_t* w, const bf16_t* s, const bf16_t* b, const uint32_t* w2,
                   const bf16_t* s2, const bf16_t* b2, const bf16_t* residual, bf16_t* y, int M, int N, int K, int bits,
                   int parts, float* part, size_t part_stride, hipStream_t stream) {
  const bool pair = w2 != nullptr;
  const ShortParams p{x, w, w2, s, b, s2, b2, residual, y, M, N, K, exo_ceil_div(N, pair ? 8 : 16), K / 64 / parts,
                      parts > 1 ? part : nullptr, part_stride,
                      K / parts % 512 == 0 && (((uintptr_t)s | (uintptr_t)b | (uintptr_t)s2 | (uintptr_t)b2) & 15) == 0};
  if (bits == 4 && pair) launch_rows<4, true>(p, parts, stream);
  if (bits == 4 && !pair) launch_rows<4, false>(p, parts, stream);
  if (bits == 8 && pair) launch_rows<8, true>(p, parts, stream);
  if (bits == 8 && !pair) launch_rows<8, false>(p, parts, stream);
}
