// Shared device helpers and host-side error plumbing for the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

typedef uint16_t bf16_t;  // raw bfloat16 bit pattern

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;
typedef __attribute__((address_space(3))) char* lds_char;

#define EXO_WAVE 64

// 16 bytes per lane from a buffer into LDS at `to` + 16 * lane, counted by vmcnt.  Written as the instruction (it
// has no register result): the compiler makes the first LDS read behind such a request of its own wait for
// it, whichever tile it fills.  It knows nothing of this one: the waits are the caller's.
__device__ __forceinline__ void load_to_lds16_untracked(u32x4 rsrc, lds_char to, uint32_t voffset, uint32_t soffset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"((uint32_t)(uintptr_t)to), "v"(voffset), "s"(rsrc), "s"(soffset)
               : "memory", "m0");
}

__device__ __forceinline__ float bf2f(bf16_t b) {
  return __builtin_bit_cast(float, (uint32_t)b << 16);
}
// round-to-nearest-even (v_cvt_pk_bf16_f32 on gfx950)
__device__ __forceinline__ bf16_t f2bf(float f) {
  __bf16 b = (__bf16)f;
  return __builtin_bit_cast(bf16_t, b);
}
__device__ __forceinline__ uint32_t pack_bf2(float lo, float hi) {
  bf16x2_t r;
  r[0] = (__bf16)lo;
  r[1] = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ float bf_lo(uint32_t v) {
  return __builtin_bit_cast(float, v << 16);
}
__device__ __forceinline__ float bf_hi(uint32_t v) {
  return __builtin_bit_cast(float, v & 0xffff0000u);
}
__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a),
                                         __builtin_bit_cast(bf16x2_t, b), acc, false);
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
// sum over aligned sub-groups of `width` lanes (power of two <= 64)
__device__ __forceinline__ float group_sum(float v, int width) {
  for (int o = width >> 1; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// ---- cross-lane sums on the DPP path (no LDS traffic) ----
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_get(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xf, false));
}
// sum over the wave, in every lane (all 64 active): what lies 32, 16, 8, 4, 2 and 1 lanes away is added in turn.  Swaps of
// halves and rotations of rows stand for the exchanges (from the third on a value depends on the low lane bits alone), so
// no step goes through the LDS crossbar.
__device__ __forceinline__ float wave_sum(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
  const uint32_t a0 = a[0], a1 = a[1];
  v = __builtin_bit_cast(float, a0) + __builtin_bit_cast(float, a1);
  const auto b = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
  const uint32_t b0 = b[0], b1 = b[1];
  v = __builtin_bit_cast(float, b0) + __builtin_bit_cast(float, b1);
  v += dpp_get<0x128, 0xf>(v);  // row_ror:8
  v += dpp_get<0x124, 0xf>(v);  // row_ror:4
  v += dpp_get<0x4E, 0xf>(v);   // quad_perm [2,3,0,1]
  v += dpp_get<0xB1, 0xf>(v);   // quad_perm [1,0,3,2]
  return v;
}
// ---- exchanges between lanes whose numbers differ in one bit, without the LDS crossbar (the same values, and for two lanes' sum the same
// bits, as with __shfl_xor, which is one or two hundred cycles to the result where these are ten)
template <int BIT>
__device__ __forceinline__ uint32_t lane_xor_bits(uint32_t v) {
  static_assert(BIT == 1 || BIT == 2 || BIT == 4 || BIT == 8 || BIT == 16 || BIT == 32, "one bit of the lane's number");
  auto dpp = [](uint32_t x, auto ctrl) __attribute__((always_inline)) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, 0xf, 0xf, false);
  };
  if constexpr (BIT == 1) return dpp(v, std::integral_constant<int, 0xB1>{});
  if constexpr (BIT == 2) return dpp(v, std::integral_constant<int, 0x4E>{});
  if constexpr (BIT == 4) return dpp(dpp(v, std::integral_constant<int, 0x141>{}), std::integral_constant<int, 0x1B>{});  // 7 - i, then i ^ 3
  if constexpr (BIT == 8) return dpp(v, std::integral_constant<int, 0x128>{});                                             // row_ror:8
  if constexpr (BIT >= 16) {
    const auto t = BIT == 16 ? __builtin_amdgcn_permlane16_swap(v, v, false, false) : __builtin_amdgcn_permlane32_swap(v, v, false, false);
    const uint32_t low = t[0], high = t[1];  // of the lanes with the bit clear, and set, in both
    return threadIdx.x & BIT ? low : high;
  }
}
template <int BIT>
__device__ __forceinline__ float lane_xor(float v) {
  return __builtin_bit_cast(float, lane_xor_bits<BIT>(__builtin_bit_cast(uint32_t, v)));
}
// a lane's value and the other's: {with the bit clear, with it set}, or the other way round
template <int BIT>
__device__ __forceinline__ void lane_pair(float v, float& a, float& b) {
  if constexpr (BIT >= 16) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const auto t = BIT == 16 ? __builtin_amdgcn_permlane16_swap(u, u, false, false) : __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const uint32_t low = t[0], high = t[1];
    a = __builtin_bit_cast(float, low), b = __builtin_bit_cast(float, high);
  } else {
    a = v, b = lane_xor<BIT>(v);
  }
}
template <int BIT>
__device__ __forceinline__ float add_across(float v) {
  float a, b;
  lane_pair<BIT>(v, a, b);
  return a + b;
}
template <int BIT>
__device__ __forceinline__ float max_across(float v) {
  float a, b;
  lane_pair<BIT>(v, a, b);
  return fmaxf(a, b);
}

// sum over the wave; the total lands in lane 63
__device__ __forceinline__ float wave_sum_to_lane63(float v) {
  v += dpp_get<0xB1, 0xf>(v);   // quad_perm [1,0,3,2]
  v += dpp_get<0x4E, 0xf>(v);   // quad_perm [2,3,0,1]
  v += dpp_get<0x141, 0xf>(v);  // row_half_mirror
  v += dpp_get<0x140, 0xf>(v);  // row_mirror: every lane holds its row-of-16 total
  v += dpp_get<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v += dpp_get<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}

// sum over aligned runs of W (8 or 16) lanes, in every lane of the run
template <int W>
__device__ __forceinline__ float run_sum(float v) {
  v += dpp_get<0xB1, 0xf>(v);   // quad_perm [1,0,3,2]
  v += dpp_get<0x4E, 0xf>(v);   // quad_perm [2,3,0,1]
  v += dpp_get<0x141, 0xf>(v);  // row_half_mirror
  if (W == 16) v += dpp_get<0x140, 0xf>(v);  // row_mirror
  return v;
}

// sum over the wave, in every lane (all 64 active), without the LDS crossbar: rows of 16 by DPP, the four rows by swaps
__device__ __forceinline__ float wave_total(float v) {
  v = run_sum<16>(v);
  const auto a = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
  const uint32_t a0 = a[0], a1 = a[1];
  v = __builtin_bit_cast(float, a0) + __builtin_bit_cast(float, a1);
  const auto b = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
  const uint32_t b0 = b[0], b1 = b[1];
  return __builtin_bit_cast(float, b0) + __builtin_bit_cast(float, b1);
}
// sum of the NW values (a power of two up to 16) that a workgroup's waves have left at `part`, in every lane
template <int NW>
__device__ __forceinline__ float total_of(const float* part) {
  float v = part[threadIdx.x & (NW - 1)];
  if (NW >= 2) v += dpp_get<0xB1, 0xf>(v);
  if (NW >= 4) v += dpp_get<0x4E, 0xf>(v);
  if (NW >= 8) v += dpp_get<0x141, 0xf>(v);
  if (NW >= 16) v += dpp_get<0x140, 0xf>(v);
  return v;
}

// ---- maxima over the wave, as wave-uniform values ----
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_max_u32(uint32_t v) {
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, ROW_MASK, 0xf, false);
  return o > v ? o : v;
}
// maximum over the wave, as a wave-uniform value (a six-step DPP reduction into lane 63)
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = dpp_max_u32<0xB1, 0xf>(v);   // quad_perm [1,0,3,2]
  v = dpp_max_u32<0x4E, 0xf>(v);   // quad_perm [2,3,0,1]
  v = dpp_max_u32<0x141, 0xf>(v);  // row_half_mirror
  v = dpp_max_u32<0x140, 0xf>(v);  // row_mirror: every lane holds its row-of-16 maximum
  v = dpp_max_u32<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_max_u32<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_max_f32(float v) {
  const int o = __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), CTRL,
                                            ROW_MASK, 0xf, false);
  return fmaxf(__builtin_bit_cast(float, o), v);
}
__device__ __forceinline__ float wave_max_f32_uniform(float v) {
  v = dpp_max_f32<0xB1, 0xf>(v);
  v = dpp_max_f32<0x4E, 0xf>(v);
  v = dpp_max_f32<0x141, 0xf>(v);
  v = dpp_max_f32<0x140, 0xf>(v);
  v = dpp_max_f32<0x142, 0xa>(v);
  v = dpp_max_f32<0x143, 0xc>(v);
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// Hand-over of results to another workgroup without a device-wide fence: the producer
// writes its values with device-scope stores, then every storing wave waits here until all
// of its outstanding vector-memory operations have completed (on gfx9 stores count in
// vmcnt and are acknowledged once they are visible at the scope they were issued with),
// then the workgroup barrier, then ONE thread bumps the arrival counter with a
// device-scope read-modify-write.  A consumer that saw the counter value loads the values
// at device scope.  The chain  store(sc1) -> vmcnt(0) -> s_barrier -> RMW(agent) ->
// load(sc1)  orders the values before the counter without writing the L2 back.
__device__ __forceinline__ void wait_own_stores_done() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// A kernel's arguments, a word of every 64 bytes: the scalar cache then holds them all after one way through memory.  (The compiler loads a
// field where it is used, and the first field of each line waits again, some 0.3 us.)
template <typename P>
__device__ __forceinline__ void request_arguments(const P& p) {
  const int* const at = reinterpret_cast<const int*>(&p);
#pragma unroll
  for (int i = 0; i < (int)(sizeof(P) / 4); i += 16) {
    const int word = at[i];
    asm volatile("" ::"s"(word));
  }
}

// ---- host side -------------------------------------------------------------
#define EXO_OK 0
#define EXO_ERR_ARG (-1)
#define EXO_ERR_HIP (-2)

void exo_set_error(const char* fmt, ...);
// records the kernel instance a launcher chose (read back with exo_last_variant())
void exo_note_variant(const char* fmt, ...);

#define EXO_REQUIRE(cond, ...)      \
  do {                              \
    if (!(cond)) {                  \
      exo_set_error(__VA_ARGS__);   \
      return EXO_ERR_ARG;           \
    }                               \
  } while (0)

#define EXO_CHECK_LAUNCH(name)                                               \
  do {                                                                       \
    hipError_t e__ = hipGetLastError();                                      \
    if (e__ != hipSuccess) {                                                 \
      exo_set_error("%s: launch failed: %s", name, hipGetErrorString(e__));  \
      return EXO_ERR_HIP;                                                    \
    }                                                                        \
  } while (0)

static inline int exo_ceil_div(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }
