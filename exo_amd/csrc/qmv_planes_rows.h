// Two to eight activation rows against packed codes on the integer matrix cores (part of qmv.hip; the planes are those of
// qmv_planes.h).
//
// The four planes of four rows of x are the sixteen rows of the A operand, sixteen weight rows the columns of B: a lane holds one weight row's
// products with one row of x, all four planes of them, so that nothing changes lanes.  A group of 64 codes is one product (two of
// them for five to eight rows of x, whose planes are two operands).  4 bits: a lane's 16 bytes are half a group; its words change
// places with the lanes 32 further (v_permlane32_swap), so that a product's slots belong to one group.
// Eight waves split K; each prepares one row of x, or half of one, for all of them.  Their sums of a tile meet in LDS, double-buffered, at one
// barrier for every one or two tiles, which the requests in flight cross.
// What bounds it: from some 50 MB of weights the memory (8 bits, 128256 rows of 2048 under four rows of x 52 us, 5.4 TB/s; the 4x4x4 kernel 63); below, the way
// of the rows of x to planes (a norm, 18 instructions an element and two barriers, 2 to 4 us), which every workgroup goes.  us before | now, 8
// bits: pair of 14336x4096 under 4 | 8 rows 33.6 | 46.9 -> 28.1 | 30.8, 4096x4096 8.8 | 11.8 -> 7.1 | 8.5, 3072x2048 behind a norm 7.7 | 10.4 -> 5.8 | 7.0; 4
// bits: pair of 8192x2048 under 4 rows 8.9 -> 7.4, 5120x2048 behind a norm 6.4 -> 5.6.
// Wrongly rounded outputs in a million 0 to 790 where the 4x4x4 and the 16x16x32 kernel have 0 to 3500 (normal elements, one of a row 300 times as
// large).
#pragma once

constexpr int kRowsWaves = 8;
// LDS of a group's planes: 4 quarters of the product's slots, each 16 rows of 16 bytes and 16 bytes more, so that the 64 lanes that write
// eight groups' meet every bank twice
constexpr int kPlaneQuarter = 272, kPlaneGroup = 4 * kPlaneQuarter;
template <int TOK>
constexpr int kRowsTiles = TOK == 4 ? 2 : 1;  // tiles between barriers
template <int TOK>
constexpr int rows_lds(int K) {
  return K / 64 * kPlaneGroup * (TOK / 4) + TOK * (K / 64 + 4) * (int)sizeof(GroupSum) + 2 * kRowsTiles<TOK> * kRowsWaves * TOK * 16 * 4;
}

// K = 2048 * XS; p.slots: tiles of 16 rows (a pair: 8 of each matrix), 8 bits: of p.spw, where the product's other columns repeat the
// last one
template <int BITS, int NMAT, int XS, int TOK>
__global__ __launch_bounds__(64 * kRowsWaves) void qmv_planes_rows_kernel(const QmvParams p) {
  extern __shared__ uint4 smem[];
  constexpr int K = 2048 * XS, G = K / 64, GW = G / kRowsWaves;  // groups; of a wave
  constexpr int GB = BITS == 4 && XS % 2 == 0 ? 8 : 4, ITERS = GW / GB;  // groups of a batch of requests; batches of a wave per tile
  constexpr int UB = GB * BITS / 8;                              // requests of 16 bytes per lane for them
  constexpr int SW = GB / 2;                                     // words of scales
  constexpr int SETS = TOK / 4, WPT = kRowsWaves / TOK;          // operands of planes; waves per row of x
  constexpr int XR = K / WPT / 512;                              // runs of 8 elements per lane
  constexpr int RPT = 16 / NMAT, C = kRowsTiles<TOK>;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, q = lane >> 4;

  char* const planes = reinterpret_cast<char*>(smem);
  GroupSum* const sums = reinterpret_cast<GroupSum*>(planes + SETS * G * kPlaneGroup);  // [TOK][G + 4]
  float (*const red)[C][kRowsWaves][SETS * 64] = reinterpret_cast<float (*)[C][kRowsWaves][SETS * 64]>(sums + TOK * (G + 4));
  __shared__ float s_ss[kRowsWaves];
  __shared__ int s_bad[kRowsWaves];

  const int tiles = p.slots, rows = BITS == 8 ? p.spw : RPT;
  const int base = tiles / (int)gridDim.x, rem = tiles - base * (int)gridDim.x;
  const int t0 = (int)blockIdx.x * base + min((int)blockIdx.x, rem);
  const int t1 = t0 + base + ((int)blockIdx.x < rem ? 1 : 0);

  // this wave's part of the rows of x (past the last one: that one again, never stored)
  const int tok = wave % TOK, part = wave / TOK;
  uint4 xr[XR], nw[XR];
  {
    const bf16_t* xs = p.x + (size_t)min(tok, p.M - 1) * K + part * (K / WPT);
    const bf16_t* ns = p.norm_w + part * (K / WPT);
#pragma unroll
    for (int i = 0; i < XR; ++i) {
      xr[i] = *reinterpret_cast<const uint4*>(xs + (lane + 64 * i) * 8);
      if (p.norm_w) nw[i] = *reinterpret_cast<const uint4*>(ns + (lane + 64 * i) * 8);
    }
  }

  const int mat = NMAT == 2 ? n >> 3 : 0, r_in = BITS == 8 ? min(n % RPT, p.spw - 1) : n % RPT;
  const size_t row_bytes = (size_t)p.wpr * 4;
  const char* const wm = reinterpret_cast<const char*>(mat ? p.w[NMAT - 1] : p.w[0]) + wave * (GW * 8 * BITS) + q * 16;
  const bf16_t* const sm = (mat ? p.s[NMAT - 1] : p.s[0]) + wave * GW;
  const bf16_t* const bm = (mat ? p.b[NMAT - 1] : p.b[0]) + wave * GW;
  struct Batch {
    uint4 w[UB];
    uint32_t s[SW], b[SW];
  };
  auto words = [](const bf16_t* at, uint32_t(&o)[SW]) __attribute__((always_inline)) {
    if constexpr (SW == 4) {
      const uint4 v = *reinterpret_cast<const uint4*>(at);
      o[0] = v.x, o[1] = v.y, o[2] = v.z, o[3] = v.w;
    } else {
      const uint2 v = *reinterpret_cast<const uint2*>(at);
      o[0] = v.x, o[1] = v.y;
    }
  };
  const int nb = (t1 - t0) * ITERS;
  int it = t0, ib = 0;  // tile and batch that are requested next
  auto issue = [&](Batch& b) {
    const int row = min(min(it, t1 - 1) * rows + r_in, p.N - 1);  // (rows and tiles past the end: the last one's, dropped)
    const char* w = wm + (size_t)row * row_bytes + ib * (UB * 64);
#pragma unroll
    for (int u = 0; u < UB; ++u) b.w[u] = *reinterpret_cast<const uint4*>(w + u * 64);
    words(sm + (size_t)row * G + ib * GB, b.s);
    words(bm + (size_t)row * G + ib * GB, b.b);
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

  // ---- the rows of x: norm, whole numbers, planes
  auto lds_barrier = [] {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  if (p.norm_w) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < XR; ++i) ss += sumsq_word<4>(xr[i]);
    ss = wave_total(ss);
    if (lane == 0) s_ss[wave] = ss;
    lds_barrier();
    ss = s_ss[tok];
#pragma unroll
    for (int w = 1; w < WPT; ++w) ss += s_ss[tok + w * TOK];
    const float inv = rsqrtf(ss / (float)K + p.eps);
#pragma unroll
    for (int i = 0; i < XR; ++i) norm_word<4>(xr[i], nw[i], inv);
  }
  bool bad;
  {
    char* const mine = planes + ((tok >> 2) * G + part * (G / WPT)) * kPlaneGroup + (tok & 3) * 64;
    GroupSum* const ms = sums + tok * (G + 4) + part * (G / WPT);
    store_planes<BITS, XR>(xr, XR * 64, [&](int piece) {
      const int pc = piece & 3, slot = BITS == 4 ? (pc & 1) << 1 | pc >> 1 : pc;
      return mine + (piece >> 2) * kPlaneGroup + slot * kPlaneQuarter;
    }, ms, bad);
  }
  if (lane == 0) s_bad[wave] = bad;
  lds_barrier();

  float poison[SETS];
#pragma unroll
  for (int s = 0; s < SETS; ++s) {
    const int t = s * 4 + q;
    int any = s_bad[t];
#pragma unroll
    for (int w = 1; w < WPT; ++w) any |= s_bad[t + w * TOK];
    poison[s] = any ? __builtin_nanf("") : 0.f;
  }
  const char* const a_row = planes + wave * GW * kPlaneGroup + q * kPlaneQuarter + n * 16;
  const GroupSum* const s_row = sums + q * (G + 4) + wave * GW;
  uint32_t kmask = 0x0F0F0F0Fu;
  asm volatile("" : "+s"(kmask));

  float acc[SETS];
#pragma unroll
  for (int s = 0; s < SETS; ++s) acc[s] = poison[s];
  int tile = t0, batch = 0;
  // the waves' sums of the tiles since the last call, their last one before tile `end`
  auto finish = [&](int end) {
    const int first = t0 + (end - 1 - t0) / C * C;
    const auto& from = red[(first - t0) / C & 1];
    lds_barrier();
    for (int e = threadIdx.x; e < C * TOK * RPT; e += 64 * kRowsWaves) {
      const int c = e / (TOK * RPT), t = e / RPT % TOK, r = e % RPT, row = (first + c) * rows + r;
      if (r >= rows || first + c >= end || t >= p.M || row >= p.N) continue;
      const int at = t * 16 + r;
      auto sum = [&](int at) {
        float v = from[c][0][at];
#pragma unroll
        for (int w = 1; w < kRowsWaves; ++w) v += from[c][w][at];
        return v;
      };
      float out = sum(at);
      if (NMAT == 2) {
        const float g = bf2f(f2bf(out)), up = bf2f(f2bf(sum(at + 8)));
        out = g / (1.f + __expf(-g)) * up;
      } else if (p.residual) {
        out = bf2f(f2bf(out)) + bf2f(p.residual[(size_t)t * p.N + row]);
      }
      p.y[(size_t)t * p.N + row] = f2bf(out);
    }
  };
  auto compute = [&](Batch& b) {
    const char* a = a_row + batch * (GB * kPlaneGroup);
    int at = batch * GB;
    if (SETS == 2) asm volatile("" : "+v"(at));  // (eight groups' sums held across tiles would leave one workgroup per CU)
    const GroupSum* sr = s_row + at;
#pragma unroll
    for (int j = 0; j < GB; ++j) {
      i32x4 c;
      if constexpr (BITS == 4) {
        uint4& w = b.w[j / 2];
        if (j % 2 == 0) {  // words of the lanes 32 further for the group that this product leaves
          const auto x = __builtin_amdgcn_permlane32_swap(w.x, w.z, false, false);
          const auto y = __builtin_amdgcn_permlane32_swap(w.y, w.w, false, false);
          w = make_uint4(x[0], y[0], x[1], y[1]);
        }
        const uint32_t w0 = j % 2 ? w.z : w.x, w1 = j % 2 ? w.w : w.y;
        c = i32x4{(int)(w0 & kmask), (int)((w0 >> 4) & kmask), (int)(w1 & kmask), (int)((w1 >> 4) & kmask)};
      } else {
        const uint4 w = b.w[j];
        c = i32x4{(int)(w.x ^ 0x80808080u), (int)(w.y ^ 0x80808080u), (int)(w.z ^ 0x80808080u), (int)(w.w ^ 0x80808080u)};
      }
      const float sc = j % 2 ? bf_hi(b.s[j / 2]) : bf_lo(b.s[j / 2]), bi = j % 2 ? bf_hi(b.b[j / 2]) : bf_lo(b.b[j / 2]);
#pragma unroll
      for (int s = 0; s < SETS; ++s) {
        const i32x4 zero = {0, 0, 0, 0};
        const i32x4 d = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const i32x4*>(a + (s * G + j) * kPlaneGroup), c, zero, 0, 0, 0);
        const GroupSum x = sr[s * 4 * (G + 4) + j];
        float f = __builtin_ldexpf(fmaf((float)((d[3] << 8) + d[2]), 65536.f, (float)((d[1] << 8) + d[0])), x.unit);
        if (BITS == 8) f = fmaf(128.f, x.sum, f);
        acc[s] = fmaf(bi, x.sum, fmaf(sc, f, acc[s]));
      }
    }
    if (++batch == ITERS) {  // the tile's sums of this wave
      batch = 0;
#pragma unroll
      for (int s = 0; s < SETS; ++s) {
        red[(tile - t0) / C & 1][(tile - t0) % C][wave][s * 64 + lane] = acc[s];
        acc[s] = poison[s];
      }
      ++tile;
      if ((tile - t0) % C == 0 || tile == t1) finish(tile);
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
}
