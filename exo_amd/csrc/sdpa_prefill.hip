// Causal attention for a chunk of T new tokens (prefill) on the matrix cores.
//
// Flash-attention recurrence with both products on v_mfma_f32_32x32x16_bf16, written
// transposed so that every per-query quantity (running max, sum, rescale factor) is a
// per-LANE scalar:
//   S^T[key][query] = K . Q^T          A = K rows from LDS,      B = Q^T from registers
//   O^T[d][query]  += V^T . P^T        A = V^T rows from LDS,    B = P^T = the S^T registers
// The D-operand layout of the first product puts, in lane (query, half), registers that
// are 8 consecutive keys per 16-key step once the K rows are fed in a permuted order;
// they are rounded to bf16 and used as the B operand of the second product without any
// data movement; the V^T operand comes out of the row-major V tile through the transposing LDS read.
//
// Work split: a wave owns 32 query tokens of ONE query head; the four waves of a
// workgroup take four consecutive (token tile, head) units of one kv head, so with GQA
// (4, 8, 16 query heads per kv head) they share every K/V tile they stage.  Key tiles of
// 64, straight from the cache into LDS, two buffers each for K and V; one barrier per tile.
//
// What bounds it: a tile is 32 matrix instructions (1024 cycles) and about as many cycles of vector work
// for its 32 weights per lane (each a multiply-add, a power at a quarter of the rate, a sum, half a
// rounding and half a maximum).  So the two are written into each other: a wave multiplies the NEXT
// tile's scores between this tile's weights, and takes the next scores' maxima between this
// tile's V products; the output is rescaled only where some query of the wave has a new maximum.
// 32 / 8 heads of 128, 4096 tokens behind 12288: 1230 -> 935 us (1029 TFLOP/s), 2047 tokens 67 -> 49 us,
// 4096 behind 12288 with heads of 64 807 -> 580 us.
//
// SPLIT (launches of at most one workgroup per CU, i.e. prompts of about a thousand tokens):
// eight waves, two teams of four that take the first and the second half of the
// workgroup's key tiles for the same four units, each with tile buffers of its own; at the end
// the second team's (O^T, max, sum) pass through LDS and are merged into the first's.  The
// causal triangle gives a launch of one round workgroups of 1 to N tiles; without the split
// the heavy ones run on alone, one wave per SIMD, for most of the launch.
#include "../../include/exo_mi355x.h"
#include "common.h"
#include "sdpa_internal.h"

namespace {

constexpr int kBN = 64;   // keys per tile
constexpr int kBM = 32;   // query tokens per wave

struct FaParams {
  const bf16_t* q;    // [B*T, Hq*D] (already rotated)
  const bf16_t* k;    // [B, Hkv, S_max, D]
  const bf16_t* v;
  const int32_t* pos;  // [B] tokens in the cache before this chunk
  bf16_t* out;         // [B*T, Hq*D]
  float scale_log2e;  // > 0 (a negative scale is in q_sign)
  uint32_t q_sign;    // flips the queries of a negative scale
  int T, Hq, Hkv, S_max, G, units;  // units = token tiles * G
};

template <int D>
constexpr int fa_lds_bytes() {
  return 4 * kBN * D * 2;  // two K tiles, two V tiles
}

typedef short short4_t __attribute__((ext_vector_type(4)));

// ds_read_b64_tr_b16: four consecutive rows of one column out of a row-major bf16 tile
__device__ __forceinline__ uint2 read_tr16(lds_char at) {
  const short4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4_t __attribute__((address_space(3)))*)at);
  return __builtin_bit_cast(uint2, v);
}

// keeps the computation of a value in the slot where it is written
template <typename T>
__device__ __forceinline__ void hold(T& v) {
  asm volatile("" : "+v"(v));
}

template <int D, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 512 : 256, SPLIT ? 1 : 2) void fa_prefill_kernel(const FaParams p) {
  constexpr int STEPS = D / 16;  // MFMA steps over d for S^T
  constexpr int DT = D / 32;     // 32-row tiles of O^T
  constexpr int ROW = D * 2;     // bytes of a K or V row in LDS
  constexpr int TILE = kBN * ROW;
  constexpr int VEC = D / 8;     // 16-byte chunks of a row
  constexpr int LOADS = kBN * VEC / 256;
  extern __shared__ __attribute__((aligned(16))) char fa_lds[];  // per team: K tiles 0, 1, V tiles 0, 1

  const int tid = threadIdx.x & 255, lane = tid & 63;  // within the team
  const int team = SPLIT ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) : 0;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const lds_char lds = (lds_char)fa_lds + team * (4 * TILE);
  const int n = lane & 31, kq = lane >> 5;
  const int kvh = blockIdx.y, b = blockIdx.z;
  // Heavy (late) token tiles first - but a launch of up to two workgroups per CU is one round
  // with nothing left to balance it, and the dispatcher hands a CU its second workgroup 256
  // positions after its first: every other run of 256 then takes the light tiles first, so
  // that the two workgroups of a CU are a heavy and a light one (2046 tokens, 32 / 8 heads:
  // 129 -> 109 us; with 2048 launches the same order lost 10 %).
  const int row = (int)blockIdx.y + (int)gridDim.y * (int)blockIdx.z;
  const int rows_per_run = max(1, 256 / (int)gridDim.x);
  const bool one_round = !SPLIT && gridDim.x * gridDim.y * gridDim.z <= 512;  // (longer launches balance
  const bool light_first = one_round && ((row / rows_per_run) & 1);  //  themselves, heavy first)
  const int u0 = (light_first ? (int)blockIdx.x : (int)gridDim.x - 1 - (int)blockIdx.x) * 4;
  const int u = u0 + wave;
  const bool active = u < p.units;
  const int uc = active ? u : p.units - 1;
  const int tt = uc / p.G, g = uc % p.G;
  const int hq = kvh * p.G + g;
  const int pos = p.pos[b];
  const int t_lane = min(tt * kBM + n, p.T - 1);            // this lane's query token
  const int last_w = pos + min(tt * kBM + kBM - 1, p.T - 1);  // last key any row of the wave sees
  const int tt_max = min(u0 + 3, p.units - 1) / p.G;
  const int last_wg = min(pos + min(tt_max * kBM + kBM - 1, p.T - 1), p.S_max - 1);
  const int n_all = last_wg / kBN + 1;  // key tiles of the workgroup
  // SPLIT: team 0 takes tiles [0, n_all / 2), team 1 the rest - at least as many, and the
  // ones with the causal edge; the workgroup's barriers are counted by team 1's tiles
  const int t_first = (SPLIT && team) ? n_all / 2 : 0;
  const int n_tiles = !SPLIT ? n_all : team ? n_all - n_all / 2 : n_all / 2;
  const int n_iter = SPLIT ? n_all - n_all / 2 : n_all;

  // Q^T operand: lane (query n, half kq) holds d = step*16 + kq*8 .. +8 for every step
  uint4 qreg[STEPS];
  {
    const bf16_t* qp = p.q + ((size_t)b * p.T + t_lane) * ((size_t)p.Hq * D) + (size_t)hq * D + kq * 8;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      qreg[s] = *reinterpret_cast<const uint4*>(qp + s * 16);
      qreg[s].x ^= p.q_sign;
      qreg[s].y ^= p.q_sign;
      qreg[s].z ^= p.q_sign;
      qreg[s].w ^= p.q_sign;
    }
  }

  // K and V tiles go from the cache straight into LDS, row by row as they are (by the instruction: the compiler
  // makes every transposing LDS read wait for all such loads that it knows of; the wait and the barrier
  // at the end of a tile are theirs): one descriptor per
  // (sequence, kv head), a lane offset that never changes and the tile as the scalar offset.  A wave's
  // load writes its 64 chunks of 16 bytes in lane order, so the order of the chunks inside a row is
  // chosen by what a lane requests: chunk c of K row r sits at c ^ (r % 16) (128-byte rows: c ^ (r / 2 % 8)),
  // so that the 16 rows of an operand read touch all 64 banks; chunk c of V row r at c ^ (4 * (r % 4))
  // (c ^ (4 * (r / 2 % 2))), so that the four rows of a transposing read do.
  const size_t head_off = ((size_t)b * p.Hkv + kvh) * (size_t)p.S_max * D;
  auto rsrc = [&](const bf16_t* base) {
    const uint64_t at = (uint64_t)base;
    return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)at), (uint32_t)__builtin_amdgcn_readfirstlane((int)(at >> 32)) & 0xffffu,
                 0xffffffffu, 0x00020000u};
  };
  const u32x4 rk = rsrc(p.k + head_off), rv = rsrc(p.v + head_off);
  const int lrow = tid / VEC, lslot = tid % VEC;  // (row of load i: lrow + i * 256 / VEC, a multiple of 16 further)
  const uint32_t koff = (lslot ^ (D == 128 ? lrow & 15 : (lrow >> 1) & 7)) * 16;
  const uint32_t voff = (lslot ^ (D == 128 ? (lrow & 3) << 2 : ((lrow >> 1) & 1) << 2)) * 16;
  // piece i of a wave's share of key tile kt (past the last one: that one again); rows past the end of the cache: its last
  // row again (they are masked).  Rows are clamped before they are multiplied: a piece may begin past the end, and the bytes of a
  // whole cache need not fit 31 bits; both offsets of the instruction are unsigned.
  auto load_piece = [&](u32x4 r, uint32_t off, int tile, int kt, int i) {
    const int row0 = (t_first + min(kt, max(n_tiles, 1) - 1)) * kBN;
    const int first = min(row0 + i * (256 / VEC), p.S_max - 1);
    const uint32_t at = (uint32_t)min(lrow, p.S_max - 1 - first) * ROW + off;
    load_to_lds16_untracked(r, lds + tile * TILE + wave * 1024 + i * 4096, at, (uint32_t)first * ROW);
  };
  auto load_tile = [&](u32x4 r, uint32_t off, int tile, int kt) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) load_piece(r, off, tile, kt, i);
  };

  // A-operand row r of a 32-key sub-tile holds this key, so that D registers 8s..8s+7
  // of lane half kq are keys 16s + 8kq .. +8
  const int jr = n >> 3;
  const int key_of_row = 16 * (jr >> 1) + 8 * ((n >> 2) & 1) + 4 * (jr & 1) + (n & 3);
  const int k_at = key_of_row * ROW, k_x = kq ^ (D == 128 ? key_of_row & 15 : (key_of_row >> 1) & 7);
  // V^T operand: lane (d = 32*dt + n, half kq) takes keys 16*st + 8*kq .. +8 of that d, four at
  // a time: a block of 16 lanes whose lane r points at V[key0 + r/4][d0 + 4*(r%4) ..+4] gets
  // V[key0 .. key0+4][d0 + i] in lane i
  const int v_row = kq * 8 + ((lane & 15) >> 2);
  const int v_at = v_row * ROW + ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
  const int v_x = D == 128 ? v_row & 3 : (v_row >> 1) & 1;  // (the same for every key block: they are 4 rows apart)

  floatx16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[dt][e] = 0.f;
  // running maximum, the same scaled; this half's sums
  float m_run = -INFINITY, m_ref = 0.f, l0 = 0.f, l1 = 0.f;

  auto read_k = [&](lds_char tile, int slot) {  // operand of product `slot` of S^T: step slot / 2, sub-tile slot % 2
    return *reinterpret_cast<__attribute__((address_space(3))) const u32x4*>(
        tile + (slot & 1) * (32 * ROW) + k_at + (((slot >> 1) * 2) ^ k_x) * 16);
  };
  auto read_v = [&](lds_char tile, int slot) {  // of O^T: 16 keys slot / DT, columns slot % DT
    const lds_char at = tile + (slot / DT) * (16 * ROW) + v_at + ((slot % DT) ^ v_x) * 64;
    const uint2 lo = read_tr16(at), hi = read_tr16(at + 4 * ROW);
    return u32x4{lo.x, lo.y, hi.x, hi.y};
  };
  // what the scores of tile kt need before they become weights: the causal edge
  auto mask = [&](floatx16(&s)[2], int kt) {
    const int key0 = (t_first + kt) * kBN;
    if (key0 + kBN - 1 > pos + tt * kBM) {  // some (query, key) pair of the wave is masked
      const int vis = pos + t_lane - key0;  // keys 0..vis of the tile are visible
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (ks * 32 + 16 * (e >> 3) + 8 * kq + (e & 7) > vis) s[ks][e] = -INFINITY;
    }
  };
  // The rescaling, and the exchange between the halves of a query, is left out where no query of the wave
  // has a new maximum.  The weights refer to the maximum itself: the largest is 1, which bf16 holds.  (Left
  // behind until a score lay 2^8 above it, the largest weight was rounded while its sum was not:
  // error 2.2e-3 -> 2.35e-3 under scores of unit width, 1.9e-3 -> 2.4e-3 under twice that.)
  auto settle = [&](float mx) {
    if (__builtin_amdgcn_ballot_w64(mx > m_run) == 0) return;  // (at the first tile: -infinity)
    mx = max_across<32>(mx);
    const float m_new = fmaxf(m_run, mx);
    // (a query that has seen no key yet keeps -infinity as its maximum and 0 as its reference)
    const float ref = m_new == -INFINITY ? 0.f : m_new * p.scale_log2e;
    const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_ref - ref);
    l0 *= alpha;
    l1 *= alpha;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[dt][e] *= alpha;
    m_run = m_new;
    m_ref = ref;
  };
  constexpr int AHEAD = 3;  // operands in flight from LDS

  // One tile: the products of the NEXT tile's scores, the weights of this one between them; then
  // this tile's V products, the next scores' maximum between them.  Tile kt's scores are in `s`
  // (masked, the maximum settled), K of kt + 1 and V of kt in LDS.
  auto tile_step = [&](floatx16(&s)[2], floatx16(&sn)[2], int kt, int par) {
    const lds_char kt_lds = lds + (par ^ 1) * TILE, vt_lds = lds + (2 + par) * TILE;
    u32x4 a[4];
    float x[32], w[32];
    uint32_t pb[16];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) a[i] = read_k(kt_lds, i);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int e = 0; e < 16; ++e) sn[ks][e] = 0.f;
    // weights in three stages, a stage per slot: exponent; power; sum and rounding
    constexpr int PER = 32 / (2 * STEPS);  // scores per slot
    auto stage = [&](int i) {
#pragma unroll
      for (int e = i * PER; e < (i + 1) * PER; ++e)
        if (e < 32) {
          x[e] = fmaf(s[e >> 4][e & 15], p.scale_log2e, -m_ref);
          hold(x[e]);
        }
#pragma unroll
      for (int e = (i - 1) * PER; e < i * PER; ++e)
        if (e >= 0 && e < 32) {
          w[e] = __builtin_amdgcn_exp2f(x[e]);
          hold(w[e]);
        }
#pragma unroll
      for (int e = (i - 2) * PER; e < (i - 1) * PER; e += 2)
        if (e >= 0 && e < 32) {
          l0 += w[e];
          l1 += w[e + 1];
          pb[e >> 1] = pack_bf2(w[e], w[e + 1]);
          hold(pb[e >> 1]);
          hold(l0);
          hold(l1);
        }
    };
#pragma unroll
    for (int i = 0; i < 2 * STEPS; ++i) {
      sn[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[i & 3]),
                                                          __builtin_bit_cast(bf16x8_t, qreg[i >> 1]), sn[i & 1], 0, 0, 0);
      a[(i + AHEAD) & 3] = i + AHEAD < 2 * STEPS ? read_k(kt_lds, i + AHEAD) : read_v(vt_lds, i + AHEAD - 2 * STEPS);
      stage(i);
      if (SPLIT && i % (STEPS / LOADS) == 0) {
        const int l = i / (STEPS / LOADS);
        if (l & 1) load_piece(rv, voff, 2 + (par ^ 1), kt + 1, l >> 1);
        else load_piece(rk, koff, par, kt + 2, l >> 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    stage(2 * STEPS);
    stage(2 * STEPS + 1);
    mask(sn, kt + 1);
    float mx = fmaxf(sn[0][0], sn[1][0]);
    constexpr int VS = 4 * DT, MPER = 16 / VS;  // V products; pairs of scores per slot
#pragma unroll
    for (int i = 0; i < VS; ++i) {
      const int g = i / DT, dt = i % DT;  // 16 keys: registers 4g .. 4g+3 of the weights
      const uint4 bw = make_uint4(pb[4 * g], pb[4 * g + 1], pb[4 * g + 2], pb[4 * g + 3]);
      o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[(i + 2 * STEPS) & 3]),
                                                      __builtin_bit_cast(bf16x8_t, bw), o[dt], 0, 0, 0);
      if (i + AHEAD < VS) a[(i + AHEAD + 2 * STEPS) & 3] = read_v(vt_lds, i + AHEAD);
#pragma unroll
      for (int e = i * MPER; e < (i + 1) * MPER; ++e) mx = fmaxf(fmaxf(mx, sn[0][e]), sn[1][e]);
      hold(mx);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (kt + 1 < n_tiles) settle(mx);
  };

  // A context of one tile (prompts of up to 64 tokens) has nothing to be written into each other: no second K
  // tile, no next scores, no barriers of the loop (61 tokens, 32 / 8 heads of 128: 7.4 -> 6.5 us, of 64 5.4 -> 4.5;
  // plain tiles without the interleaving 6.6 and 5.0)
  const bool one_tile = !SPLIT && n_all == 1;
  const int n_mine = last_w / kBN + 1 - t_first;  // tiles that this wave's rows see (<= 0: none)
  load_tile(rk, koff, 0, 0);
  load_tile(rv, voff, 2, 0);
  if (!one_tile) load_tile(rk, koff, 1, 1);
  // Every load so far (the Q operand among them) has landed before the loop is entered: left
  // to itself the compiler waits, in EVERY iteration, for as many loads as were issued after Q.
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
  floatx16 s0[2], s1[2];
  if (n_mine > 0) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int e = 0; e < 16; ++e) s0[ks][e] = 0.f;
#pragma unroll
    for (int i = 0; i < 2 * STEPS; ++i)
      s0[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, read_k(lds, i)),
                                                          __builtin_bit_cast(bf16x8_t, qreg[i >> 1]), s0[i & 1], 0, 0, 0);
    mask(s0, 0);
    float mx = fmaxf(s0[0][0], s0[1][0]);
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(fmaxf(mx, s0[0][e]), s0[1][e]);
    settle(mx);
  }
  if (one_tile) {
    const lds_char vt_lds = lds + 2 * TILE;
#pragma unroll
    for (int g = 0; g < 4; ++g) {  // 16 keys
      uint32_t pb[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float w0 = __builtin_amdgcn_exp2f(fmaf(s0[g >> 1][(g & 1) * 8 + e], p.scale_log2e, -m_ref));
        const float w1 = __builtin_amdgcn_exp2f(fmaf(s0[g >> 1][(g & 1) * 8 + e + 1], p.scale_log2e, -m_ref));
        l0 += w0;
        l1 += w1;
        pb[e >> 1] = pack_bf2(w0, w1);
      }
      const bf16x8_t bw = __builtin_bit_cast(bf16x8_t, make_uint4(pb[0], pb[1], pb[2], pb[3]));
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, read_v(vt_lds, g * DT + dt)), bw, o[dt], 0, 0, 0);
    }
  }
  // K of tile kt + 2 goes where K of kt was, V of kt + 1 where V of kt - 1 was: both last read before the barrier
  // that ended the previous tile, both complete at the one that ends this tile.  (A step past the wave's
  // or the workgroup's last tile multiplies what lies in LDS and uses none of it.)
  // SPLIT: the requests of a tile stand one by one between its products; together at its start they fill the CU's address
  // unit (16 cycles per KB) and the wave stands (1023 tokens of 32 / 4 heads 25.3 -> 24.3 us, 300 behind 2000 of 64 / 4
  // 42.8 -> 40.2, 512 behind 9000 with heads of 64 97.7 -> 90.7).  Of two workgroups per CU one goes on meanwhile: the same
  // there is 1 to 3 % on some shapes, but 1500 tokens of 64 / 4 heads take 64 -> 66, with two tiles requested past the last.
  for (int kt = 0; !one_tile && kt < n_iter; kt += 2) {
    auto turn = [&](floatx16(&s)[2], floatx16(&sn)[2], int kt, int par) {
      const bool mine = kt < n_mine && kt < n_tiles;
      __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
      if (!SPLIT || !mine) {
        if (SPLIT || kt + 2 < n_tiles) load_tile(rk, koff, par, kt + 2);
        if (SPLIT || kt + 1 < n_tiles) load_tile(rv, voff, 2 + (par ^ 1), kt + 1);
      }
      if (mine) tile_step(s, sn, kt, par);
    };
    turn(s0, s1, kt, 0);
    turn(s1, s0, kt + 1, 1);
  }
  if (SPLIT) __builtin_amdgcn_s_waitcnt(0x0F70);  // the repeats requested past the end
  float l_run = l0 + l1;
  l_run = add_across<32>(l_run);
  if (SPLIT) {
    // the second team's sums: through LDS (lane-contiguous floats per register), merged into
    // the first team's, which goes on alone
    float* ex = reinterpret_cast<float*>(fa_lds) + wave * ((DT * 16 + 2) * 64);
    __syncthreads();  // both teams have finished with their tile buffers
    if (team == 1) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) ex[(dt * 16 + e) * 64 + lane] = o[dt][e];
      ex[(DT * 16) * 64 + lane] = m_run;
      ex[(DT * 16 + 1) * 64 + lane] = l_run;
    }
    __syncthreads();
    if (team == 1) return;  // (no workgroup barrier after this point)
    const float m1 = ex[(DT * 16) * 64 + lane], l1 = ex[(DT * 16 + 1) * 64 + lane];
    const float m = fmaxf(m_run, m1);  // finite: key 0 is visible to one of the teams
    const float a0 = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_run - m) * p.scale_log2e);
    const float a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m1 - m) * p.scale_log2e);
    l_run = l_run * a0 + l1 * a1;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[dt][e] = o[dt][e] * a0 + ex[(dt * 16 + e) * 64 + lane] * a1;
  }

  // ---- out[token][hq*D + d] = O^T[d][token] / l
  if (!active || tt * kBM + n >= p.T) return;
  const float inv = 1.f / l_run;
  bf16_t* op = p.out + ((size_t)b * p.T + t_lane) * ((size_t)p.Hq * D) + (size_t)hq * D;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint2 w;
      w.x = pack_bf2(o[dt][4 * j + 0] * inv, o[dt][4 * j + 1] * inv);
      w.y = pack_bf2(o[dt][4 * j + 2] * inv, o[dt][4 * j + 3] * inv);
      *reinterpret_cast<uint2*>(op + dt * 32 + 8 * j + 4 * kq) = w;
    }
}

}  // namespace

int exo_sdpa_prefill_mfma(const bf16_t* q, const bf16_t* k_cache, const bf16_t* v_cache,
                          const int32_t* pos, bf16_t* out, float scale, int B, int T, int Hq,
                          int Hkv, int D, int S_max, hipStream_t stream) {
  FaParams p;
  p.q = q;
  p.k = k_cache;
  p.v = v_cache;
  p.pos = pos;
  p.out = out;
  // (a scale of zero: one that rounds every score to zero, so that masked ones stay minus infinity; not fmaxf,
  // which would make a number of NaN)
  p.scale_log2e = fabsf(scale) * 1.4426950408889634f;
  if (p.scale_log2e < 1e-30f) p.scale_log2e = 1e-30f;
  p.q_sign = scale < 0.f ? 0x80008000u : 0u;
  p.T = T;
  p.Hq = Hq;
  p.Hkv = Hkv;
  p.S_max = S_max;
  p.G = Hq / Hkv;
  p.units = ((T + kBM - 1) / kBM) * p.G;
  const dim3 grid((p.units + 3) / 4, Hkv, B);
  // the split variant where its eight-wave workgroups are one round of one per CU (their two
  // teams' tile buffers leave room for one) and the heaviest has enough tiles to share out:
  // 1022 tokens of 32 / 4 heads (256 workgroups) 34.9 -> 30.3 us; with 512 workgroups it is
  // two rounds and loses to two four-wave workgroups per CU (2046 tokens, 32 / 8: 75 -> 106 us)
  const bool split = (int64_t)grid.x * grid.y * grid.z <= 256 && T >= 256;
  // more than 64 KiB of LDS per workgroup: raised once per kernel instance
  auto raise = [](const void* fn, int bytes, bool* done) {
    if (*done || bytes <= 64 * 1024) return EXO_OK;
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) {
      exo_set_error("exo_sdpa_prefill: cannot raise dynamic LDS limit: %s", hipGetErrorString(e));
      return EXO_ERR_HIP;
    }
    *done = true;
    return EXO_OK;
  };
  static bool done[4] = {false, false, false, false};
  const int lds = (D == 64 ? fa_lds_bytes<64>() : fa_lds_bytes<128>()) * (split ? 2 : 1);
  int rc;
  exo_note_variant("fa_prefill<%d,%s> grid=%dx%dx%d", D, split ? "true" : "false", (int)grid.x, (int)grid.y,
                   (int)grid.z);
  if (D == 64 && !split) {
    if ((rc = raise(reinterpret_cast<const void*>(fa_prefill_kernel<64, false>), lds, &done[0]))) return rc;
    fa_prefill_kernel<64, false><<<grid, 256, lds, stream>>>(p);
  } else if (D == 64) {
    if ((rc = raise(reinterpret_cast<const void*>(fa_prefill_kernel<64, true>), lds, &done[1]))) return rc;
    fa_prefill_kernel<64, true><<<grid, 512, lds, stream>>>(p);
  } else if (!split) {
    if ((rc = raise(reinterpret_cast<const void*>(fa_prefill_kernel<128, false>), lds, &done[2]))) return rc;
    fa_prefill_kernel<128, false><<<grid, 256, lds, stream>>>(p);
  } else {
    if ((rc = raise(reinterpret_cast<const void*>(fa_prefill_kernel<128, true>), lds, &done[3]))) return rc;
    fa_prefill_kernel<128, true><<<grid, 512, lds, stream>>>(p);
  }
  return EXO_OK;
}
