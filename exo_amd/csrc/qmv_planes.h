// One activation row against packed codes on the integer matrix cores (part of qmv.hip).
//
// The dot-product kernel spends 44 vector instructions on 32 codes of a lane, half of them at half rate: masks, shifts and
// dot products, 70 ns of a SIMD per KiB of 4-bit codes, and 15 to 20 more for scales and the sum over the wave.  Here codes enter
// v_mfma_i32_16x16x64_i8 as they are (4 bits: two masks and a shift per word; 8 bits: less 128) and the row enters as
// 32-bit whole numbers in units of 2^(E-29), E the exponent of the largest element of a group of 64, cut into four
// signed bytes ("planes") that are rows of the A operand.  Products and sums over a group are whole numbers, without
// rounding; a lane puts a group's four plane sums together (exact but for the conversions), scales them, and adds
// float32.  An element more than 22 binades below the largest of its group is rounded to that unit, which is at most 2^-30 of the
// largest; float32 sums of products with 128 + c lose 2^-17 of it.  (A unit per group and not per row: an element
// far larger than all others leaves the other groups as they are.)
//
// A workgroup's four waves split K.  A tile is 8 weight rows (a pair: 4 of each matrix): columns 0..7 of the B operand are the
// first half of a wave's share of K, columns 8..15 the second, and a wave instruction loads 16 x 64 bytes.  The planes of the
// halves are different rows of A.  With 4 bits the slots of lanes q = 0, 1 and of q = 2, 3 belong to two groups: their planes
// are different rows too, with zeros in the other group's slots, so that one accumulator keeps them apart.  Lanes that
// hold the other half's accumulator rows add the groups' biases instead.
// What it measured beside the dot products, us (norm ahead of the product): 128256x2048 36.6 -> 29.1, 14336x2048 7.3 -> 5.6, pair
// of 8192x2048 7.5 -> 6.2, 2048x8192 5.5 -> 4.9, 128256x4096 64.6 -> 56.9; 8 bits: 9216x4096 12.7 -> 10.3, pair of 14336x4096 29.3 -> 24.8, of
// 4096x8192 22.2 -> 15.9.  Of 16 rows without halves: 0.97 to 1.24 of that time.  Conditional requests cost what the arithmetic had won: the
// waits behind them cover everything in flight (pair of 8192x2048 1.5 us).
// Wrongly rounded outputs in a million: 0 to 1000 where the dot products had 250 to 4000 (2048 to 4096 rows, elements normal, with
// outliers of 300 times, or spread over e^3).
#pragma once

typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int kPlaneRows = 8;  // weight rows of a tile
// A product's planes in LDS: four lanes' 16 codes, four planes, 16 bytes each, and 16 zeros for the operand rows that a lane does
// not hold
constexpr int kPlaneBlock = 272;
// A group of the row beside its planes
struct GroupSum {
  float sum;
  int unit;  // its whole numbers count in 2^unit
};
// LDS of a wave: the planes of K / 4 codes and their groups' sums
__host__ __device__ constexpr int planes_wave_bytes(int K) { return K / 256 * kPlaneBlock + K / 256 * (int)sizeof(GroupSum); }

// What a lane does for its rows of a tile and half of a row's share (see above): the groups' products, from the four accumulator rows
// that it holds, or the biases.
struct PlaneLane {
  int row, half, group;  // of the tile; of the share; of a unit (4 bits)
  bool products, bias;
  float offset;          // of the codes in the products
};
template <int BITS>
__device__ __forceinline__ PlaneLane plane_lane(int lane) {
  const int n = lane & 15, q = lane >> 4;
  PlaneLane l;
  l.row = n & 7;
  l.half = n >> 3;
  l.group = BITS == 4 ? q & 1 : 0;
  l.products = BITS == 4 ? (q >> 1) == l.half : q == l.half;
  l.bias = BITS == 4 ? !l.products : q == 2 + l.half;
  l.offset = l.products ? (BITS == 8 ? 128.f : 0.f) : 1.f;
  return l;
}
// where the lane's row of the A operand begins: plane n & 3 of a half and (4 bits) a group of the units; zeros in the other group's
// slots.  `units`: of a half
template <int BITS>
__device__ __forceinline__ const char* plane_operand(const char* planes, int lane, int units) {
  const int n = lane & 15, q = lane >> 4, half = BITS == 4 ? n >> 3 : n >> 2;
  const bool mine = half < 2 && (BITS == 8 || ((n >> 2) & 1) == q >> 1);
  return planes + (mine ? half * (units * (BITS == 4 ? 2 : 1) * kPlaneBlock) + q * 64 + (n & 3) * 16 : 256);
}

// to the nearest whole number (of halves the larger)
__device__ __forceinline__ int nearest(float v) {
  int r;
  asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}
// the largest of eight lanes' runs, as the bits of its absolute value
__device__ __forceinline__ uint32_t group_most(const uint4& x) {
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  auto larger = [](uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
  };
  constexpr uint32_t kAbs = 0x7fff7fffu;
  uint32_t m = larger(larger(x.x & kAbs, x.y & kAbs), larger(x.z & kAbs, x.w & kAbs));
  m = larger(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0xB1, 0xf, 0xf, false));   // quad_perm [1,0,3,2]
  m = larger(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x4E, 0xf, 0xf, false));   // quad_perm [2,3,0,1]
  m = larger(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x141, 0xf, 0xf, false));  // row_half_mirror
  return max(m & 0xffffu, m >> 16);
}

// A wave's elements as planes: `runs` runs of 8, lane l holding the runs l, l + 64 ...
// `place`: where the 16-byte pieces of 16 elements begin, their four planes 16 bytes apart.
// `bad`: an element is infinite or not a number, which makes every result one that is
// not a number, as its products with 128 + c would.
template <int BITS, int XS, typename Place>
__device__ __forceinline__ void store_planes(const uint4 (&xr)[XS], int runs, Place place, GroupSum* sums, bool& bad) {
  const int lane = threadIdx.x & 63;
  uint32_t largest = 0;
#pragma unroll
  for (int i = 0; i < XS; ++i) {
    const int run = lane + 64 * i;
    const uint32_t x4[4] = {xr[i].x, xr[i].y, xr[i].z, xr[i].w};
    const uint32_t most = group_most(xr[i]);
    largest = max(largest, most);
    const int shift = 29 + 127 - (int)(most >> 7);  // |x| * 2^shift < 2^30
    uint32_t d[8];
    float gs = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      gs += bf_lo(x4[k]) + bf_hi(x4[k]);
      // byte i of X + 0x808080 less 128 (the top one as it is): the signed digits of X
      d[2 * k] = (uint32_t)nearest(__builtin_ldexpf(bf_lo(x4[k]), shift)) + 0x00808080u;
      d[2 * k + 1] = (uint32_t)nearest(__builtin_ldexpf(bf_hi(x4[k]), shift)) + 0x00808080u;
    }
    // operand words: the codes of a word's even places, then of its odd ones (8 bits: as they come)
    uint32_t out[4][2];  // [plane][operand word]
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      uint32_t e[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) e[k] = d[BITS == 4 ? 2 * k + o : 4 * o + k];
      const uint32_t a01 = __builtin_amdgcn_perm(e[1], e[0], 0x05010400u);  // e0.0 e1.0 e0.1 e1.1
      const uint32_t a23 = __builtin_amdgcn_perm(e[3], e[2], 0x05010400u);
      const uint32_t b01 = __builtin_amdgcn_perm(e[1], e[0], 0x07030602u);  // e0.2 e1.2 e0.3 e1.3
      const uint32_t b23 = __builtin_amdgcn_perm(e[3], e[2], 0x07030602u);
      out[0][o] = __builtin_amdgcn_perm(a23, a01, 0x05040100u) ^ 0x80808080u;
      out[1][o] = __builtin_amdgcn_perm(a23, a01, 0x07060302u) ^ 0x80808080u;
      out[2][o] = __builtin_amdgcn_perm(b23, b01, 0x05040100u) ^ 0x80808080u;
      out[3][o] = __builtin_amdgcn_perm(b23, b01, 0x07060302u);
    }
    gs = run_sum<8>(gs);
    if (XS * 64 == runs || run < runs) {
#pragma unroll
      for (int pl = 0; pl < 4; ++pl) *reinterpret_cast<uint2*>(place(run >> 1) + pl * 16 + (run & 1) * 8) = make_uint2(out[pl][0], out[pl][1]);
      if ((run & 7) == 0) sums[run >> 3] = {gs, -shift};
    }
  }
  bad = __ballot(largest >= 0x7f80u) != 0;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();  // (what a wave reads below it has written itself)
}
// of one row: [unit][product] blocks of [q][plane] x 16 bytes
template <int BITS>
__device__ __forceinline__ char* plane_piece(char* planes, int piece) {
  return planes + (BITS == 4 ? ((piece >> 3) * 2 + (piece & 1)) * kPlaneBlock + ((piece >> 1) & 3) * 64 : (piece >> 2) * kPlaneBlock + (piece & 3) * 64);
}
// zeros of the `blocks` product blocks at `planes`
__device__ __forceinline__ void clear_planes(char* planes, int blocks) {
  for (int i = threadIdx.x & 63; i < blocks; i += 64) *reinterpret_cast<uint4*>(planes + i * kPlaneBlock + 256) = make_uint4(0, 0, 0, 0);
}

// acc += a batch's groups: UB units of codes w and their scales s, the operands from a and the groups' sums from sr on
template <int BITS, int UB, int SW>
__device__ __forceinline__ void plane_products(const uint4 (&w)[UB], const uint32_t (&s)[SW], const char* a, const GroupSum* sr, const PlaneLane& l,
                                               uint32_t kmask, float& acc) {
  constexpr int GU = BITS == 4 ? 2 : 1;
  i32x4 d[UB];
#pragma unroll
  for (int u = 0; u < UB; ++u) {
    const uint32_t w4[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
    const i32x4 zero = {0, 0, 0, 0};
    if constexpr (BITS == 4) {
      i32x4 c[2];
#pragma unroll
      for (int h = 0; h < 2; ++h)
        c[h] = i32x4{(int)(w4[2 * h] & kmask), (int)((w4[2 * h] >> 4) & kmask), (int)(w4[2 * h + 1] & kmask), (int)((w4[2 * h + 1] >> 4) & kmask)};
      d[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const i32x4*>(a + 2 * u * kPlaneBlock), c[0], zero, 0, 0, 0);
      d[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const i32x4*>(a + (2 * u + 1) * kPlaneBlock), c[1], d[u], 0, 0, 0);
    } else {
      const i32x4 c = {(int)(w4[0] ^ 0x80808080u), (int)(w4[1] ^ 0x80808080u), (int)(w4[2] ^ 0x80808080u), (int)(w4[3] ^ 0x80808080u)};
      d[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const i32x4*>(a + u * kPlaneBlock), c, zero, 0, 0, 0);
    }
  }
#pragma unroll
  for (int u = 0; u < UB; ++u) {
    const GroupSum g = sr[u * GU];
    // (the unit is put in ahead of the scales, which may be as large as their type holds)
    float f = __builtin_ldexpf(fmaf((float)((d[u][3] << 8) + d[u][2]), 65536.f, (float)((d[u][1] << 8) + d[u][0])), g.unit);
    if (!l.products) f = 0.f;  // (the other half's codes)
    const float v = fmaf(l.offset, g.sum, f);
    float sc;
    if constexpr (BITS == 4)
      sc = l.group ? bf_hi(s[u]) : bf_lo(s[u]);
    else
      sc = (u & 1) ? bf_hi(s[u >> 1]) : bf_lo(s[u >> 1]);
    acc = fmaf(sc, v, acc);
  }
}
// the tile's row sums of the wave, in the lanes below kPlaneRows
__device__ __forceinline__ float plane_row_sum(float acc, const PlaneLane& l) {
  float v = l.products || l.bias ? acc : 0.f;
  v += dpp_get<0x128, 0xf>(v);  // row_ror:8
  const auto e = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
  const uint32_t e0 = e[0], e1 = e[1];
  v = __builtin_bit_cast(float, e0) + __builtin_bit_cast(float, e1);
  const auto g = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
  const uint32_t g0 = g[0], g1 = g[1];
  v = __builtin_bit_cast(float, g0) + __builtin_bit_cast(float, g1);
  return v;
}

// units (64 lanes x 16 bytes) per batch of requests: four, or two where half a wave's share is no multiple of four
template <int BITS, int XS>
constexpr int plane_units = BITS == 4 && XS % 2 == 1 ? 2 : 4;

// K = 2048 * XS; p.slots: tiles
template <int BITS, int NMAT, int XS, bool ROUTE>
__global__ __launch_bounds__(256) void qmv_planes_kernel(const QmvParams p) {
  extern __shared__ uint4 smem[];
  constexpr int K = 2048 * XS, G = K / 64;
  constexpr int UB = plane_units<BITS, XS>;
  constexpr int CODES = 64 * 8 / BITS;         // codes of 64 bytes: a unit's, of one half
  constexpr int GU = CODES / 64;               // groups of those
  constexpr int H = BITS == 4 ? 2 : 1;         // products per unit
  constexpr int RPT = kPlaneRows / NMAT;       // rows per tile and matrix
  constexpr int SW = UB * GU * 2 / 4;          // words of a batch's scales
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int UW = K / 8 / CODES, ITERS = UW / UB;  // units and batches of a wave per tile

  // LDS, of each wave by itself: the planes, the groups' sums; then the tiles' partial sums
  char* const planes = reinterpret_cast<char*>(smem) + wave * planes_wave_bytes(K);
  GroupSum* const sums = reinterpret_cast<GroupSum*>(planes + (K / 256) * kPlaneBlock);
  float (*const red)[4][kPlaneRows] = reinterpret_cast<float (*)[4][kPlaneRows]>(reinterpret_cast<char*>(smem) + 4 * planes_wave_bytes(K));
  __shared__ float s_ss[4];

  // balanced contiguous tiles of this workgroup
  const int tiles = p.slots;
  const int base = tiles / (int)gridDim.x, rem = tiles - base * (int)gridDim.x;
  const int t0 = (int)blockIdx.x * base + min((int)blockIdx.x, rem);
  const int t1 = t0 + base + ((int)blockIdx.x < rem ? 1 : 0);

  const bf16_t* xin = p.x;
  bf16_t* yout = p.y;
  const int pair = blockIdx.y;
  if (p.idx || p.each_row || (ROUTE && p.route)) {
    xin += (size_t)(p.x_rows == 1 ? pair / p.topk : pair) * p.K;
    yout += (size_t)pair * p.N;
  }
  clear_planes(planes, K / 256);

  uint32_t route_raw[4] = {0, 0, 0, 0};
  if (ROUTE && p.route) route_load(p.route + (size_t)(pair / p.topk) * p.E, p.E, lane, route_raw);
  // the wave's share of the row, 8 elements a run
  uint4 xr[XS], nw[XS];
  {
    const bf16_t* xs = xin + (size_t)wave * (K / 4);
    const bf16_t* ns = p.norm_w + (size_t)wave * (K / 4);
#pragma unroll
    for (int i = 0; i < XS; ++i) {
      const int run = lane + 64 * i;
      xr[i] = *reinterpret_cast<const uint4*>(xs + run * 8);
      if (p.norm_w) nw[i] = *reinterpret_cast<const uint4*>(ns + run * 8);
    }
  }
  size_t ew = 0, eg = 0;
  if (ROUTE && p.route) {
    const int t = pair / p.topk, slot = pair - t * p.topk;
    int my_id;
    float my_p, tot;
    const bool record = blockIdx.x == 0 && slot == 0 && wave == 0;
    route_topk_regs(route_raw, p.E, record ? p.topk : slot + 1, lane, my_id, my_p, tot);
    if (record && lane < p.topk) {
      p.route_idx[(size_t)t * p.topk + lane] = my_id;
      p.route_scores[(size_t)t * p.topk + lane] = route_score(my_p, tot, p.route_renorm);
    }
    const int e = __builtin_amdgcn_readlane(my_id, slot);
    ew = (size_t)e * p.N * p.wpr;
    eg = (size_t)e * p.N * G;
  } else if (p.idx) {
    int e = p.idx[pair];
    e = e < 0 ? 0 : (e >= p.E ? p.E - 1 : e);  // memory safety only: the host rejects such ids
    ew = (size_t)e * p.N * p.wpr;
    eg = (size_t)e * p.N * G;
  }

  const PlaneLane l = plane_lane<BITS>(lane);
  const int mat = NMAT == 2 ? l.row / RPT : 0, r_of = l.row % RPT;
  const size_t row_bytes = (size_t)p.wpr * 4;
  const char* const wm = reinterpret_cast<const char*>((mat ? p.w[NMAT - 1] : p.w[0]) + ew) + (wave * 2 + l.half) * (UW * 64) + (lane >> 4) * 16;
  const bf16_t* const sm = mat ? (l.bias ? p.b[NMAT - 1] : p.s[NMAT - 1]) : (l.bias ? p.b[0] : p.s[0]);
  const char* const sc = reinterpret_cast<const char*>(sm + eg) + (wave * 2 + l.half) * (UW * GU * 2);

  struct Batch {
    uint4 w[UB];
    uint32_t s[SW];
  };
  const int nb = (t1 - t0) * ITERS;
  int it = t0, ib = 0;  // tile and batch that are requested next
  auto issue = [&](Batch& b) {
    const int row = min(min(it, t1 - 1) * RPT + r_of, p.N - 1);  // (rows and tiles past the end: the last one's, dropped)
    const char* w = wm + (size_t)row * row_bytes + ib * (UB * 64);
    const char* s = sc + (size_t)row * (G * 2) + ib * (SW * 4);
#pragma unroll
    for (int u = 0; u < UB; ++u) b.w[u] = *reinterpret_cast<const uint4*>(w + u * 64);
    if constexpr (SW == 4) {
      const uint4 v = *reinterpret_cast<const uint4*>(s);
      b.s[0] = v.x, b.s[1] = v.y, b.s[2] = v.z, b.s[3] = v.w;
    } else if constexpr (SW == 2) {
      const uint2 v = *reinterpret_cast<const uint2*>(s);
      b.s[0] = v.x, b.s[1] = v.y;
    } else {
      b.s[0] = *reinterpret_cast<const uint32_t*>(s);
    }
    if (++ib == ITERS) {
      ib = 0;
      ++it;
    }
  };

  // No request sits behind a branch, so that every wait leaves those behind it in flight.
  Batch buf[2];
  issue(buf[0]);
  __builtin_amdgcn_sched_barrier(0);
  issue(buf[1]);
  __builtin_amdgcn_sched_barrier(0);

  // ---- the row: norm, whole numbers, planes
  if (p.norm_w) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < XS; ++i) ss += sumsq_word<4>(xr[i]);
    ss = wave_total(ss);
    if (lane == 0) s_ss[wave] = ss;
    __syncthreads();
    const float inv = rsqrtf((s_ss[0] + s_ss[1] + s_ss[2] + s_ss[3]) / (float)K + p.eps);
#pragma unroll
    for (int i = 0; i < XS; ++i) norm_word<4>(xr[i], nw[i], inv);
  }
  bool bad;
  store_planes<BITS, XS>(xr, XS * 64, [&](int piece) { return plane_piece<BITS>(planes, piece); }, sums, bad);
  const char* const a_row = plane_operand<BITS>(planes, lane, UW);
  const GroupSum* const s_row = sums + l.half * (UW * GU) + l.group;
  uint32_t kmask = 0x0F0F0F0Fu;
  asm volatile("" : "+s"(kmask));

  float acc = 0.f;
  int tile = t0, batch = 0;
  auto compute = [&](const Batch& b) {
    const char* a = a_row + batch * (UB * H * kPlaneBlock);
    const GroupSum* sr = s_row + batch * (UB * GU);
    plane_products<BITS>(b.w, b.s, a, sr, l, kmask, acc);
    if (++batch == ITERS) {  // the tile's row sums of this wave
      batch = 0;
      const float v = plane_row_sum(acc, l);
      acc = 0.f;
      if (lane < kPlaneRows) red[tile - t0][wave][lane] = bad ? __builtin_nanf("") : v;
      ++tile;
    }
  };
  int left = nb;
  for (; left > 3; left -= 2) {
    compute(buf[0]);
    issue(buf[0]);
    compute(buf[1]);
    issue(buf[1]);
  }
  if (left == 3) {
    compute(buf[0]);
    issue(buf[0]);
    compute(buf[1]);
    compute(buf[0]);
  } else if (left == 2) {
    compute(buf[0]);
    compute(buf[1]);
  } else {
    compute(buf[0]);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < (t1 - t0) * RPT; i += 256) {
    const int t = i / RPT, r = i % RPT, row = (t0 + t) * RPT + r;
    if (row >= p.N) continue;
    float v[NMAT];
#pragma unroll
    for (int a = 0; a < NMAT; ++a) v[a] = ((red[t][0][a * RPT + r] + red[t][1][a * RPT + r]) + red[t][2][a * RPT + r]) + red[t][3][a * RPT + r];
    float out;
    if (NMAT == 2) {
      const float g = bf2f(f2bf(v[0])), up = bf2f(f2bf(v[NMAT - 1]));
      out = g / (1.f + __expf(-g)) * up;
    } else {
      out = v[0];
      if (p.residual) out = bf2f(f2bf(out)) + bf2f(p.residual[row]);
    }
    yout[row] = f2bf(out);
  }
}
