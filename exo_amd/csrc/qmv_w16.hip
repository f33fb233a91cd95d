// Fused dequant-GEMV for up to 16 activation rows on v_mfma_f32_16x16x32_bf16 (4-bit codes).
//
// The instruction multiplies A[16][32] by B[32][16]: lane l holds A[l%16][8*(l/16) .. +8],
// B[8*(l/16) .. +8][l%16], and D[4*(l/16) + r][l%16] in register r.  Here A is the activations,
// B a block of 16 weight rows (column = weight row j), so a lane's four results belong to ONE
// weight row: scale and bias of a quantisation group are one value per lane.
//  * a wave instruction loads 16 rows x 64 contiguous bytes (128 codes = two groups of a row):
//    lane (lane/4, lane%4) takes 16-byte chunk lane%4 of row lane/4, so that the four lanes of
//    a quad read 64 contiguous bytes.  A product wants words of row j in the lanes (j, kg): they
//    change lanes through 1 KB of the wave's own LDS, one 16-byte write and one or two reads per
//    lane (chunk c of row r at c ^ r/4 % 4: all 64 banks in each).  (Through the crossbar, two
//    ds_bpermute_b32 and a select per product, the same took 1.5 us of the pair's 20.)
//  * more than eight rows (WIDE): lane (j, kg) takes 8 bytes of each of the slice's two groups, so
//    that a product's four K slots belong to one group.
//  * up to eight rows: lane (j, kg) takes chunk kg, of whose words K slots 0 and 1 belong to the
//    first group and 2 and 3 to the second.  The operand A keeps them apart: its rows 0..7 are the
//    activation rows with zeros in slots 2 and 3, its rows 8..15 the same with zeros in slots 0 and 1.
//    Lanes kg < 2 get the first group's sums and the others the second's: no lane scales rows that
//    do not exist.  The halves of the wave are added once per row block.
//  * a wave owns SL such 64-byte slices of every row block of its workgroup; the matching
//    activations stay in registers in operand order for the whole launch.  They are loaded as
//    whole runs of a row, normalised there, and change lanes through the same LDS region.  The waves of
//    a workgroup together cover K; their partial sums meet in LDS once, at the end.
//  * codes become (128+nibble) bf16 pairs with one v_and_or_b32 each (exact; up to four rows: 16+nibble).  Per group, float32:
//      up to 8 rows   acc += s * D + (b / -128) * C      C = -128 sum x,  D = C + sum (128+q) x
//      up to 16       acc += s * D + (b - 128 s) * Sx    Sx = sum x,  D = sum (128+q) x
//    C | Sx comes out of products with a column of -128 | 1, in the lanes and registers of D.  Where D's sum starts at C the offset
//    leaves in the matrix core and not between two scaled sums: 0.7 outputs in 1000 of 14336x4096 under 8 rows are not the exact result's
//    rounding, against 1.7, at the same time.  (9 to 16 rows keep their sums, 1.6 in 1000: prompts of up to 16 tokens go through them,
//    and which of two tied tokens follows hangs on their bits.)
//  * DEPTH row blocks of weights are in flight per wave (register buffers in rotation), all of
//    them requested right behind the activations.  Every refill is issued whether or not a block is
//    left (past the end all lanes read the same 16 bytes), so that the number of loads in flight at
//    each wait is a constant.
// At 8 | 16 rows, behind a norm, up to 12 matrices in turn, before the operands came this way -> now: pair of 14336x4096 18.5 | 21.0 -> 15.7 | 18.7
// us, 6144x4096 11.0 | 12.2 -> 8.4 | 10.3, 4096x4096 9.9 | 11.2 -> 6.9 | 8.7, 128256x4096 69 | 83 -> 56 | 73, pair of 8192x2048 9.6 | 10.7 -> 7.8 |
// 9.0, 2048x4096 9.8 | 11.0 -> 6.4 | 8.1; 4096x14336 without one 15.5 | 17.4 -> 13.4 | 15.5.
// What bounds it: the way to the first product (activations, norm, lane changes: 3 us), after which the pair
// streams at 5 TB/s; with K split, 3 us of hand-over; at 16 rows vector issue (two epilogues per slice).
#include "../../include/exo_mi355x.h"
#include "common.h"
#include "qmv_internal.h"

namespace {

struct W16Params {
  const bf16_t* x;       // [M, K]
  const bf16_t* norm_w;  // [K] or null: fused RMSNorm of x
  float eps;
  const uint32_t* w[2];  // packed [N, K/8]   ([1]: the up matrix of a (gate, up) pair)
  const bf16_t* s[2];    // [N, K/64]
  const bf16_t* b[2];
  const bf16_t* residual;  // [M, N] or null
  bf16_t* y;               // [M, N]
  int M, N, K;
  int row_bytes;  // K / 2
  int G;          // K / 64
  int blocks;     // N / 16 (pair: N / 8)
  int wave_bytes; // LDS of a wave: lane changes, partial sums
  int wide_pieces;  // a row's scales are whole pieces of eight groups, else a piece may begin in one row and end in the next
  int piece_mul;    // 65536 / pieces of a row + 1, else 2^20 / pairs of groups of a row + 1
  int pairs_log2;   // else: pairs of groups of a piece: 1, where there are threads for all of them, or 4
  // K split over `kparts` workgroups per group of row blocks (long rows: the activations of
  // a whole row would not fit the registers): workgroup i takes part i % kparts, Gp groups
  // of every row; float32 partial results meet in `part`, the last workgroup of a group to
  // arrive adds them in part order
  int kparts, Gp;
  float* part;    // [kparts][M][N]
  int* counters;  // [block groups], zero between launches
};

constexpr int kLdsMax = 160 * 1024 - 2048 - 64, kLdsHalf = 80 * 1024 - 2048 - 64;  // (beside the sums of squares)
constexpr int kRowPad = 16;                      // bytes between rows of staged scales: 16 rows, 64 banks

// bytes through which a wave's chunks change lanes: all slices at once where the LDS allows it
constexpr int turn_bytes(bool wide, int sl) { return (wide ? 1 : sl) * 1024; }
// staged activation rows: 16, or eight and one of zeros
constexpr int x_bytes(bool wide, int sl) { return (wide ? 16 : 9) * (sl * 256); }
// partial sums of a row block
constexpr int sum_bytes(bool wide) { return wide ? 1024 : 512; }

__device__ __forceinline__ void st_dev(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_dev(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ float sumsq8(const uint4& v) {
  return bf_lo(v.x) * bf_lo(v.x) + bf_hi(v.x) * bf_hi(v.x) + bf_lo(v.y) * bf_lo(v.y) +
         bf_hi(v.y) * bf_hi(v.y) + bf_lo(v.z) * bf_lo(v.z) + bf_hi(v.z) * bf_hi(v.z) +
         bf_lo(v.w) * bf_lo(v.w) + bf_hi(v.w) * bf_hi(v.w);
}
__device__ __forceinline__ void norm8(uint4& xv, const uint4& wv, float inv) {
  xv.x = pack_bf2(bf_lo(xv.x) * inv * bf_lo(wv.x), bf_hi(xv.x) * inv * bf_hi(wv.x));
  xv.y = pack_bf2(bf_lo(xv.y) * inv * bf_lo(wv.y), bf_hi(xv.y) * inv * bf_hi(wv.y));
  xv.z = pack_bf2(bf_lo(xv.z) * inv * bf_lo(wv.z), bf_hi(xv.z) * inv * bf_hi(wv.z));
  xv.w = pack_bf2(bf_lo(xv.w) * inv * bf_lo(wv.w), bf_hi(xv.w) * inv * bf_hi(wv.w));
}
// the 8 activations of one packed word in the order of the unpacked nibble pairs:
// (x0,x4),(x1,x5),(x2,x6),(x3,x7)
__device__ __forceinline__ uint4 pair_order(const uint4& xv) {
  uint4 o;
  o.x = __builtin_amdgcn_perm(xv.z, xv.x, 0x05040100u);
  o.y = __builtin_amdgcn_perm(xv.z, xv.x, 0x07060302u);
  o.z = __builtin_amdgcn_perm(xv.w, xv.y, 0x05040100u);
  o.w = __builtin_amdgcn_perm(xv.w, xv.y, 0x07060302u);
  return o;
}
__device__ __forceinline__ floatx4 mfma(const uint4& a, const uint4& b, const floatx4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
// a of lanes l and l + 32 added in lane l, b of both in lane l + 32
__device__ __forceinline__ float fold_halves(float a, float b) {
  const auto t = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
  const uint32_t lo = t[0], hi = t[1];
  return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
// what the lanes of a wave wrote to LDS is read by others of its lanes behind this (its LDS operations complete in order)
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
// a workgroup's LDS writes before it are visible behind it; requests to memory stay in flight
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// WIDE: more than eight activation rows.  SL: 64-byte slices of K per wave.  DEPTH: row blocks in
// flight per wave (1: the launch gives a workgroup no more than one).  NORM: fused RMSNorm of the activations.
// KSPLIT: K split over several workgroups (single matrix, no fused norm).  An instance of its
// own: compiled into the others, the hand-over code costs them 0.5 us per launch untaken.
// PAIR: a (gate, up) pair with SwiGLU; the 16 columns of a product are 8 rows of the gate matrix and the
// same 8 rows of the up matrix.  A workgroup's share is then counted in blocks of 8 rows of both -
// 14336 rows are 1792 blocks, seven for each of 256 workgroups, where blocks of 16 rows leave
// half the workgroups with four and half with three.
// The scales and biases of ALL the workgroup's rows are staged in LDS in front of the loop, as pairs
// and with whole-line loads (one piece per thread and array).  Loaded per block by the lanes
// that need them - 8 bytes each out of 16 different lines per instruction, every line touched again
// by each of the 16 waves - they cost 4.5 of 24 us of the 14336x4096 pair (measured with the loads
// taken out).  Rows that are not whole pieces of eight groups follow one another all the same, so that a piece begins in one row
// and ends in the next; up to four pieces per thread.  (With pieces of two groups, one per thread, a workgroup held two blocks of K = 2304:
// 8 rows, 9216 columns 9.0 -> 6.6 us, 256000 119 -> 73, pair of 9216 15.9 -> 9.7.)
// FEW: up to four rows.  A code c goes into the products as 16 + c instead of 128 + c - the sums that the offset leaves behind are
// an eighth - for one shift more per four words (1 % of a launch where it was taken for 8 rows).  The 4x4x4 kernel, which takes
// the other launches of up to four rows, rounds 0.4 to 0.5 outputs in 1000 the other way than the exact result, 128 + c 0.6 to 0.7
// and 16 + c 0.1 to 0.15.
template <bool WIDE, int SL, int DEPTH, bool NORM, bool KSPLIT, bool PAIR, bool FEW>
__global__ __launch_bounds__(1024) void qmv_w16_kernel(const W16Params p) {
  static_assert(!KSPLIT || (!NORM && !PAIR), "split K: one matrix, activations as they are");
  static_assert(!FEW || (!KSPLIT && !WIDE), "up to four rows: K is not split");
  constexpr uint32_t COLUMN = WIDE ? 0x3F803F80u : FEW ? 0xC180C180u : 0xC300C300u;  // 1, -16, -128
  constexpr int RPB = PAIR ? 8 : 16;       // rows of a matrix per block
  constexpr int TURN = turn_bytes(WIDE, SL), SUMS = sum_bytes(WIDE);
  constexpr int LPR = 16 * SL;             // lanes that load a wave's run of an activation row
  constexpr int RPL = 64 / LPR;            // rows of a load
  constexpr int NX = (WIDE ? 16 : 8) / RPL;
  constexpr int XROW = SL * 256;
  constexpr int NG = WIDE ? 2 : 1;         // groups of a slice whose sums a lane holds
  extern __shared__ __attribute__((aligned(16))) char lds[];  // [nw][wave_bytes], scales [rows][Gp (s, b) pairs + pad]
  __shared__ __attribute__((aligned(16))) float s_part[16][32];
  __shared__ int s_last;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nw = blockDim.x >> 6;
  const int j = lane & 15, kg = lane >> 4;  // operand layout: weight row (or activation row), K slot
  const int lr = lane >> 2, lc = lane & 3;  // load layout: row of the block, chunk of the slice

  // contiguous, balanced range of row blocks of this workgroup
  const int kparts = KSPLIT ? p.kparts : 1;
  const int kpart = KSPLIT ? (int)blockIdx.x % kparts : 0, bgroup = KSPLIT ? (int)blockIdx.x / kparts : (int)blockIdx.x;
  const int ngroups = KSPLIT ? (int)gridDim.x / kparts : (int)gridDim.x;
  const int qbase = p.blocks / ngroups, qrem = p.blocks - qbase * ngroups;
  const int q0 = bgroup * qbase + min(bgroup, qrem);
  const int nq = qbase + (bgroup < qrem ? 1 : 0);
  if (nq <= 0) return;
  const int g_first = kpart * p.Gp;  // first quantisation group of this workgroup's part of K

  char* const mine = lds + wave * p.wave_bytes;
  char* const red = mine + TURN;  // this wave's partial sums: [block][64 lanes][4 or 2]
  char* const sb_lds = lds + nw * p.wave_bytes;
  const int sb_row = p.Gp * 4 + kRowPad;

  // ---- requests: the wave's runs of the activation rows (rows past M: out of range, zeros), norm weights,
  // this thread's piece of the scales and biases, the first row blocks of weights, in this order
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.x), 0, p.M * p.K * 2, 0x00020000);
  const int run_ofs = g_first * 128 + wave * (SL * 256);  // bytes of activations in front of the wave's
  const int xrow = lane / LPR, xchunk = lane % LPR;
  uint4 xr[NX], gain = make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < NX; ++i)
    xr[i] = __builtin_bit_cast(
        uint4, __builtin_amdgcn_raw_buffer_load_b128(rx, (i * RPL + xrow) * (p.K * 2) + xchunk * 16, run_ofs, 0));
  if (NORM) gain = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(p.norm_w) + run_ofs + xchunk * 16);
  const int prow = (tid * p.piece_mul) >> 16, pcol = tid - prow * (p.Gp >> 3);  // (whole pieces)
  const int of_one = nq * RPB * p.Gp >> 1 >> p.pairs_log2;  // (else: pieces of a matrix, whose rows follow one another - K is not split then)
  u32x4 ps = {}, pb = {};
  auto piece_of = [&](int e) {  // (a matrix may begin at any row of a larger one)
    typedef u32x4 __attribute__((aligned(4))) four;
    const bool a = PAIR && e >= of_one;
    const size_t at = (size_t)(q0 * RPB) * p.G + ((a ? e - of_one : e) << p.pairs_log2) * 2;
    const bf16_t *s = (a ? p.s[1] : p.s[0]) + at, *b = (a ? p.b[1] : p.b[0]) + at;
    if (p.pairs_log2) {
      ps = *reinterpret_cast<const four*>(s);
      pb = *reinterpret_cast<const four*>(b);
    } else {
      ps[0] = *reinterpret_cast<const uint32_t*>(s);
      pb[0] = *reinterpret_cast<const uint32_t*>(b);
    }
  };
  if (p.wide_pieces) {
    const int row = min(prow, nq * 16 - 1), a = PAIR ? (row >> 3) & 1 : 0;
    const int r = PAIR ? (row >> 4) * 8 + (row & 7) : row;
    const size_t at = (size_t)(q0 * RPB + r) * p.G + g_first + pcol * 8;
    ps = *reinterpret_cast<const u32x4*>((a ? p.s[1] : p.s[0]) + at);
    pb = *reinterpret_cast<const u32x4*>((a ? p.b[1] : p.b[0]) + at);
  } else {
    piece_of(min(tid, (PAIR ? 2 : 1) * of_one - 1));
  }
  __builtin_amdgcn_sched_barrier(0);
  struct Block {
    u32x4 w[SL];
  } b0, b1;
  const uint32_t* const w_mine = (PAIR && lr >= 8) ? p.w[1] : p.w[0];
  const char* const w_lane = reinterpret_cast<const char*>(w_mine) + (size_t)(q0 * RPB + (lr & (RPB - 1))) * p.row_bytes +
                             g_first * 32 + wave * (SL * 64) + lc * 16;
  auto issue = [&](Block& to, int q) {
    const char* src = q < nq ? w_lane + (size_t)(q * RPB) * p.row_bytes : reinterpret_cast<const char*>(p.w[0]);
#pragma unroll
    for (int sl = 0; sl < SL; ++sl) to.w[sl] = *reinterpret_cast<const u32x4*>(src + sl * 64);
  };
  issue(b0, 0);
  __builtin_amdgcn_sched_barrier(0);
  if (DEPTH == 2) issue(b1, 1);
  __builtin_amdgcn_sched_barrier(0);

  // ---- activations into operand order
  auto stage_sb = [&]() {
    if (p.wide_pieces) {
      if (prow >= nq * 16) return;
      uint2* to = reinterpret_cast<uint2*>(sb_lds + prow * sb_row + pcol * 32);
#pragma unroll
      for (int c = 0; c < 4; ++c) to[c] = make_uint2((ps[c] & 0xffffu) | pb[c] << 16, ps[c] >> 16 | (pb[c] & 0xffff0000u));
      return;
    }
    const int row_pairs = p.Gp >> 1;
    for (int e = tid; e < (PAIR ? 2 : 1) * of_one; e += (int)blockDim.x) {
      const int a = PAIR && e >= of_one;
      if (e != tid) piece_of(e);
#pragma unroll
      for (int c = 0; c < 4; ++c) {  // two groups of a row at a time
        if (c > 0 && p.pairs_log2 == 0) break;
        const uint32_t at = ((e - a * of_one) << p.pairs_log2) + c, r = at * (uint32_t)p.piece_mul >> 20, col = at - r * row_pairs;
        const uint32_t row = PAIR ? (r >> 3) * 16 + a * 8 + (r & 7) : r;
        *reinterpret_cast<uint2*>(sb_lds + row * sb_row + col * 8) =
            make_uint2((ps[c] & 0xffffu) | pb[c] << 16, ps[c] >> 16 | (pb[c] & 0xffff0000u));
      }
    }
  };
  if (NORM) {
    // sums of squares: of a row by runs of 16 lanes, [row][slice of the row]
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const float ss = run_sum<16>(sumsq8(xr[i]));
      if ((lane & 15) == 0) s_part[i * RPL + xrow][wave * SL + (xchunk >> 4)] = ss;
    }
  }
  stage_sb();
  lds_barrier();
  if (NORM) {
    // lane (row lane/8, four slices from 4 (lane%8) on); a row's total in each of its eight lanes
    const int slices = nw * SL, c0 = (lane & 7) * 4;
#pragma unroll
    for (int h = 0; h < (WIDE ? 2 : 1); ++h) {
      const floatx4 v = *reinterpret_cast<const floatx4*>(&s_part[h * 8 + (lane >> 3)][c0]);
      float t = ((c0 < slices ? v[0] : 0.f) + (c0 + 1 < slices ? v[1] : 0.f)) +
                ((c0 + 2 < slices ? v[2] : 0.f) + (c0 + 3 < slices ? v[3] : 0.f));
      t = run_sum<8>(t);
      const float inv = rsqrtf(t / (float)p.K + p.eps);
#pragma unroll
      for (int i = 0; i < 8 / RPL; ++i) norm8(xr[h * (8 / RPL) + i], gain, __shfl(inv, (i * RPL + xrow) * 8, 64));
    }
  }
  uint4 xa[SL][4];      // operands of the products of a slice
  floatx4 sx[SL][NG];   // Sx or C of a group, where D has them
  {
    // chunk c of row r sits at c ^ r (in 256 bytes): an operand read touches all 64 banks
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int r = i * RPL + xrow;
      *reinterpret_cast<uint4*>(mine + r * XROW + (xchunk ^ r) * 16) = pair_order(xr[i]);
    }
    if (!WIDE && lane < LPR) *reinterpret_cast<uint4*>(mine + 8 * XROW + lane * 16) = make_uint4(0, 0, 0, 0);
    wave_lds_order();
    // (up to eight rows: row 8 of the staged ones, zeros, in the slots of the other group)
    const int r = WIDE ? j : (j >> 3) == (kg >> 1) ? j & 7 : 8;
    const char* from = mine + r * XROW;
    const uint4 column = make_uint4(COLUMN, COLUMN, COLUMN, COLUMN);
#pragma unroll
    for (int sl = 0; sl < SL; ++sl)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int c = WIDE ? (t >> 1) * 8 + kg * 2 + (t & 1) : kg * 4 + t;
        xa[sl][t] = *reinterpret_cast<const uint4*>(from + sl * 256 + (c ^ r) * 16);
      }
    wave_lds_order();
#pragma unroll
    for (int sl = 0; sl < SL; ++sl)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        floatx4& to = sx[sl][WIDE ? t >> 1 : 0];
        if (t % (4 / NG) == 0) to = floatx4{0.f, 0.f, 0.f, 0.f};
        to = mfma(xa[sl][t], column, to);
      }
  }

  uint32_t kmask = FEW ? 0x00780078u : 0x000F000Fu, kmagic = FEW ? 0x41804180u : 0x43004300u;
  asm volatile("" : "+s"(kmask));
  asm volatile("" : "+v"(kmagic));
  char* const turn_to = mine + lr * 64 + ((lc ^ (lr >> 2)) & 3) * 16;
  const char* const turn_from = mine + j * 64 + (WIDE ? (((kg >> 1) ^ (j >> 2)) & 3) * 16 + (kg & 1) * 8 : ((kg ^ (j >> 2)) & 3) * 16);
  const int turn_group = (((2 + (kg >> 1)) ^ (j >> 2)) & 3) * 16 - (((kg >> 1) ^ (j >> 2)) & 3) * 16;  // WIDE: to the second group
  const char* const sb_lane = sb_lds + j * sb_row + (wave * (SL * 2) + (WIDE ? 0 : kg >> 1)) * 4;

  // one row block of this wave's slices; leaves the wave's partial sums in LDS.  The block's registers are
  // free, and the next one requested into them, as soon as its words change lanes.
  auto consume = [&](Block& block, int slot) {
    uint4 c[SL];
    uint32_t sb[SL][NG];
#pragma unroll
    for (int sl = 0; sl < SL; ++sl) {
      char* const to = turn_to + (WIDE ? 0 : sl * 1024);
      if (WIDE) wave_lds_order();
      *reinterpret_cast<u32x4*>(to) = block.w[sl];
      if (!WIDE) continue;
      wave_lds_order();
      const uint2 g0 = *reinterpret_cast<const uint2*>(turn_from), g1 = *reinterpret_cast<const uint2*>(turn_from + turn_group);
      c[sl] = make_uint4(g0.x, g0.y, g1.x, g1.y);
    }
    wave_lds_order();
#pragma unroll
    for (int sl = 0; sl < SL; ++sl) {
      if (!WIDE) c[sl] = *reinterpret_cast<const uint4*>(turn_from + sl * 1024);
#pragma unroll
      for (int g = 0; g < NG; ++g) sb[sl][g] = *reinterpret_cast<const uint32_t*>(sb_lane + slot * 16 * sb_row + sl * 8 + g * 4);
    }
    wave_lds_order();
    if (DEPTH == 2) issue(block, slot + 2);
    __builtin_amdgcn_sched_barrier(0);
    floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int sl = 0; sl < SL; ++sl) {
      const uint32_t word[4] = {c[sl].x, c[sl].y, c[sl].z, c[sl].w};
      floatx4 dq[NG];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        uint4 bw;
        bw.x = ((FEW ? word[t] << 3 : word[t]) & kmask) | kmagic;
        bw.y = ((word[t] >> (FEW ? 1 : 4)) & kmask) | kmagic;
        bw.z = ((word[t] >> (FEW ? 5 : 8)) & kmask) | kmagic;
        bw.w = ((word[t] >> (FEW ? 9 : 12)) & kmask) | kmagic;
        const int g = WIDE ? t >> 1 : 0;
        dq[g] = mfma(xa[sl][t], bw, t % (4 / NG) ? dq[g] : WIDE ? floatx4{0.f, 0.f, 0.f, 0.f} : sx[sl][g]);
      }
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const float sc = bf_lo(sb[sl][g]), b = bf_hi(sb[sl][g]), tb = WIDE ? fmaf(-128.f, sc, b) : b * (FEW ? -0x1p-4f : -0x1p-7f);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = fmaf(tb, sx[sl][g][r], fmaf(sc, dq[g][r], acc[r]));
      }
    }
    if (WIDE) {
      *reinterpret_cast<floatx4*>(red + slot * SUMS + lane * 16) = acc;
    } else {
      // the two groups' halves of the wave: lanes 0..31 get results r = 0 and 2 of rows 4 (kg%2) + r, the others 1 and 3
      const float2 v = make_float2(fold_halves(acc[0], acc[1]), fold_halves(acc[2], acc[3]));
      *reinterpret_cast<float2*>(red + slot * SUMS + lane * 8) = v;
    }
  };

  if constexpr (DEPTH == 2) {
    // (a workgroup of one block multiplies what its second request brought as well, for nobody)
    int q = 0;
    do {
      consume(b0, q);
      consume(b1, q + 1);
      q += 2;
    } while (q + 1 < nq);
    if (q < nq) consume(b0, q);
  } else {
    consume(b0, 0);
  }

  // ---- the workgroup's results: sum over the waves in a fixed order, epilogue, store
  lds_barrier();
  // result (column jj, row m) of a block: where consume() has left it
  auto total = [&](int slot, int jj, int m) {
    const int at = WIDE ? ((m >> 2) * 16 + jj) * 4 + (m & 3) : ((m & 1) * 32 + (m >> 2) * 16 + jj) * 2 + ((m >> 1) & 1);
    const char* src = lds + TURN + slot * SUMS + at * 4;
    float t = 0.f;
    for (int w = 0; w < nw; ++w) t += *reinterpret_cast<const float*>(src + w * p.wave_bytes);
    return t;
  };
  if constexpr (PAIR) {
    for (int idx = tid; idx < nq * p.M * 8; idx += (int)blockDim.x) {
      const int jj = idx & 7, m = (idx >> 3) % p.M, slot = (idx >> 3) / p.M;
      // SwiGLU on the bf16-rounded projections
      const float g = bf2f(f2bf(total(slot, jj, m))), up = bf2f(f2bf(total(slot, jj + 8, m)));
      p.y[(size_t)m * p.N + (q0 + slot) * 8 + jj] = f2bf(g / (1.f + __expf(-g)) * up);
    }
    return;
  }
  for (int idx = tid; idx < nq * p.M * 16; idx += (int)blockDim.x) {
    const int jj = idx & 15, m = (idx >> 4) % p.M, slot = (idx >> 4) / p.M;
    const size_t o = (size_t)m * p.N + (q0 + slot) * 16 + jj;
    float out = total(slot, jj, m);
    if (KSPLIT) {  // this part's share of the sum
      st_dev(&p.part[(size_t)kpart * p.M * p.N + o], out);
      continue;
    }
    if (p.residual) out = bf2f(f2bf(out)) + bf2f(p.residual[o]);
    p.y[o] = f2bf(out);
  }
  if constexpr (KSPLIT) {
    // The last of a group's workgroups to arrive adds the parts in part order (the result does not
    // depend on arrival order) and writes y; the counter returns to zero.
    wait_own_stores_done();  // this wave's device-scope partial stores have completed
    __syncthreads();
    if (tid == 0) {
      int* cnt = &p.counters[bgroup];
      const int old = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_last = (old == p.kparts - 1);
      if (s_last) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!s_last) return;
    for (int idx = tid; idx < nq * p.M * 16; idx += (int)blockDim.x) {
      const int jj = idx & 15, m = (idx >> 4) % p.M, slot = (idx >> 4) / p.M;
      const size_t o = (size_t)m * p.N + (q0 + slot) * 16 + jj;
      float t = 0.f;
      for (int kp = 0; kp < p.kparts; ++kp) t += ld_dev(&p.part[(size_t)kp * p.M * p.N + o]);
      if (p.residual) t = bf2f(f2bf(t)) + bf2f(p.residual[o]);
      p.y[o] = f2bf(t);
    }
  }
}

template <bool WIDE, int SL, int DEPTH, bool NORM, bool KSPLIT, bool PAIR, bool FEW>
int launch_instance(const W16Params& p, int grid, int nq, int nw, size_t bytes, hipStream_t st) {
  auto kern = qmv_w16_kernel<WIDE, SL, DEPTH, NORM, KSPLIT, PAIR, FEW>;
  static bool attr_done = false;
  if (!attr_done && bytes > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax);
    if (e != hipSuccess) {
      exo_set_error("exo_qmv: cannot raise dynamic LDS limit: %s", hipGetErrorString(e));
      return EXO_ERR_HIP;
    }
    attr_done = true;
  }
  exo_note_variant("qmv_w16<%d,%d,%d,%s,%s> grid=%d waves=%d blocks=%d kparts=%d", PAIR ? 2 : 1, SL, DEPTH,
                   NORM ? "norm" : "plain", PAIR ? "pair8" : "staged", grid, nw, nq, p.kparts);
  kern<<<dim3(grid), dim3(64 * nw), bytes, st>>>(p);
  return EXO_OK;
}

template <bool WIDE, int SL, bool NORM, bool KSPLIT, bool PAIR, bool FEW = false>
int launch_w16s(W16Params p, int nw, hipStream_t st) {
  if constexpr (!WIDE && !KSPLIT && !FEW)
    if (p.M <= 4) return launch_w16s<WIDE, SL, NORM, KSPLIT, PAIR, true>(p, nw, st);
  p.blocks = p.N / (PAIR ? 8 : 16);
  // a wave's region: its activations on their way into operand order, later the lane changes and the partial sums
  const int scales = 16 * (p.Gp * 4 + kRowPad);
  auto wave_bytes = [&](int nq) {
    const int stream = turn_bytes(WIDE, SL) + nq * sum_bytes(WIDE);
    return stream > x_bytes(WIDE, SL) ? stream : x_bytes(WIDE, SL);
  };
  auto lds_bytes = [&](int nq) { return nw * wave_bytes(nq) + nq * scales; };
  p.wide_pieces = p.Gp % 8 == 0;
  p.piece_mul = p.wide_pieces ? 65536 / (p.Gp / 8) + 1 : (1 << 20) / (p.Gp / 2) + 1;
  // row blocks that a workgroup can hold: partial sums, scales (pieces per thread and array)
  const int pieces = p.wide_pieces ? 1 : 4;
  auto fits = [&](int nq) { return lds_bytes(nq) <= kLdsMax && nq * 2 * p.Gp <= 64 * nw * pieces; };
  if (!fits(1)) {
    exo_set_error("exo_qmv: internal: no LDS for one row block (M=%d K=%d)", p.M, p.K);
    return EXO_ERR_ARG;
  }
  // one workgroup per CU (kparts workgroups per group of row blocks); more rounds where a
  // workgroup's share would not fit
  const int round = 256 / p.kparts;
  int groups = round;
  auto share = [&]() { return (p.blocks + groups - 1) / groups; };
  while (!fits(share())) groups += round;
  // Rows of few waves (rows of broken pieces; whole ones have eight waves or sixteen): two workgroups per CU beside each other where one
  // round of one has up to six waves, or where there are several rounds of up to nine.  Behind a norm, one per CU -> two, 8 | 16 rows, us:
  // 262144x1152 41 | 50 -> 35 | 54 (without the norm 39 | 46 -> 33 | 39), 151936x896 31 | 32 -> 21 | 27, 40000x640 8.3 | 10.0 -> 7.5 | 9.0; but
  // of ten waves and more 128000x1280 22.8 | 30.1 -> 22.4 | 38.2, 151936x1664 36 -> 41.
  if (!p.wide_pieces && ((nw <= 6 && share() > 4) || (nw <= 9 && SL == 1 && groups > round))) {
    if (groups == round) groups = 2 * round;
    while (share() > 8 || lds_bytes(share()) > kLdsHalf) groups += round;
  }
  if (groups > p.blocks) groups = p.blocks;
  const int nq = (p.blocks + groups - 1) / groups;
  p.wave_bytes = wave_bytes(nq);
  p.pairs_log2 = nq * 8 * p.Gp <= 64 * nw ? 0 : 2;
  const int grid = groups * p.kparts;
  const size_t bytes = (size_t)lds_bytes(nq);
  if (nq == 1) return launch_instance<WIDE, SL, 1, NORM, KSPLIT, PAIR, FEW>(p, grid, nq, nw, bytes, st);
  return launch_instance<WIDE, SL, 2, NORM, KSPLIT, PAIR, FEW>(p, grid, nq, nw, bytes, st);
}
template <bool WIDE, int SL>
int launch_w16(const W16Params& p, bool pair, int nw, hipStream_t st) {
  if (p.kparts > 1) {
    if (!pair && !p.norm_w) return launch_w16s<WIDE, SL, false, true, false>(p, nw, st);
    exo_set_error("exo_qmv: internal: split K with a matrix pair or a norm");
    return EXO_ERR_ARG;
  }
  if (pair)
    return p.norm_w ? launch_w16s<WIDE, SL, true, false, true>(p, nw, st) : launch_w16s<WIDE, SL, false, false, true>(p, nw, st);
  return p.norm_w ? launch_w16s<WIDE, SL, true, false, false>(p, nw, st) : launch_w16s<WIDE, SL, false, false, false>(p, nw, st);
}

// 64-byte slices per wave and waves per workgroup for rows of `row_bytes`
bool w16_shape(int row_bytes, int* sl_out, int* nw_out) {
  if (row_bytes % 64) return false;
  const int slices = row_bytes / 64;
  for (int sl = 1; sl <= 2; sl *= 2) {
    if (slices % sl) continue;
    const int nw = slices / sl;
    if (nw > 16 || nw < 4) continue;
    *sl_out = sl;
    *nw_out = nw;
    return true;
  }
  return false;
}

// parts of K (workgroups per group of row blocks) for rows of `row_bytes`: 1 where a row's
// activations fit the registers of one workgroup, else - with a workspace, without a fused norm
// or a second matrix - the smallest split into equal parts of whole 16-byte scale chunks
int w16_parts(int row_bytes, bool can_split, int* sl_out, int* nw_out) {
  if (w16_shape(row_bytes, sl_out, nw_out)) return 1;
  if (!can_split || row_bytes % 64) return 0;
  const int slices = row_bytes / 64;  // one slice = two quantisation groups
  for (int kp = 2; kp <= 8; ++kp)
    if (slices % kp == 0 && (2 * slices / kp) % 8 == 0 && w16_shape(row_bytes / kp, sl_out, nw_out))
      return kp;
  return 0;
}

}  // namespace

bool exo_qmv_w16_ok(int M, int N, int K, int bits, bool norm, bool pair, bool has_workspace) {
  int sl, nw;
  if (M < 1 || M > 16 || N % 16 || N < 16 || bits != 4 || K % 128) return false;
  if ((int64_t)N * K / 2 >= (1ll << 31)) return false;
  const int kp = w16_parts(K / 2, has_workspace && !norm && !pair, &sl, &nw);
  if (kp == 0) return false;
  if (kp > 1 && (N / 16) * 4 > 64 * 1024) return false;  // counters: one per group of row blocks
  return true;
}

int exo_qmv_w16_launch(const bf16_t* x, const bf16_t* norm_w, float eps, const uint32_t* w,
                       const bf16_t* s, const bf16_t* b, const uint32_t* w2, const bf16_t* s2,
                       const bf16_t* b2, const bf16_t* residual, bf16_t* y, int M, int N, int K,
                       void* workspace, hipStream_t st) {
  W16Params p;
  p.x = x;
  p.norm_w = norm_w;
  p.eps = eps;
  p.w[0] = w;
  p.s[0] = s;
  p.b[0] = b;
  p.w[1] = w2 ? w2 : w;
  p.s[1] = s2 ? s2 : s;
  p.b[1] = b2 ? b2 : b;
  p.residual = residual;
  p.y = y;
  p.M = M;
  p.N = N;
  p.K = K;
  p.row_bytes = K / 2;
  p.G = K / 64;
  p.blocks = N / 16;  // (the launcher sets the count for its block size)
  p.wave_bytes = p.wide_pieces = p.piece_mul = p.pairs_log2 = 0;
  const bool pair = w2 != nullptr;
  int sl = 0, nw = 0;
  const int kp = exo_qmv_w16_ok(M, N, K, 4, norm_w != nullptr, pair, workspace != nullptr)
                     ? w16_parts(p.row_bytes, workspace && !norm_w && !pair, &sl, &nw)
                     : 0;
  if (kp == 0) {
    exo_set_error("exo_qmv: shape M=%d N=%d K=%d not covered by the 16x16x32 kernel", M, N, K);
    return EXO_ERR_ARG;
  }
  p.kparts = kp;
  p.Gp = p.G / kp;
  // the workspace of the split-K GEMV: counters (64 KiB), then the float32 partial results
  p.counters = reinterpret_cast<int*>(workspace);
  p.part = workspace ? reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + 64 * 1024) : nullptr;
  if (sl == 1) return M > 8 ? launch_w16<true, 1>(p, pair, nw, st) : launch_w16<false, 1>(p, pair, nw, st);
  return M > 8 ? launch_w16<true, 2>(p, pair, nw, st) : launch_w16<false, 2>(p, pair, nw, st);
}
