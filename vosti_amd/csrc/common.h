// Shared definitions of the gfx950 kernel library.
//
// The library is compiled twice from the same sources: once with -DVK_BF16
// (elements are bfloat16, the serving precision) and once with -DVK_F32
// (elements are float: the true 32-bit path, which uses fp32 MFMA and rounds
// nothing to a shorter type).  Both builds export the same C symbols.
//
// Every reduction in these kernels has an order that is a function of the
// model's sizes only, never of the number of rows in a launch or of which rows
// share a tile, so a row of a batch is bit-identical to the same row alone.
// All sources are compiled with -ffp-contract=off: a fused multiply-add
// appears only where __builtin_fmaf is written.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#if defined(VK_F32) == defined(VK_BF16)
#error "compile with exactly one of -DVK_BF16 or -DVK_F32"
#endif

#ifdef VK_F32
typedef float elem_t;
#define VK_ELEM_BYTES 4
#else
typedef __bf16 elem_t;
#define VK_ELEM_BYTES 2
#endif

#define VK_WAVE 64
#define EXPERT_PART_ROWS 192   // the most rows of one expert that a workgroup of the experts' product takes (gemm_experts_kernel)

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(__bf16 x) { return (float)x; }

template <typename T> __device__ __forceinline__ T from_f32(float x);
template <> __device__ __forceinline__ float from_f32<float>(float x) { return x; }
// Round to nearest even (v_cvt_pk_bf16_f32 on gfx950).
template <> __device__ __forceinline__ __bf16 from_f32<__bf16>(float x) { return (__bf16)x; }

// The value an element-typed store would hold, as a float.
__device__ __forceinline__ float round_to_elem(float x) { return to_f32(from_f32<elem_t>(x)); }

// The values of lanes l ^ 16 and l ^ 32 (what __shfl_xor gives), through the row and half swaps of
// gfx950, which stay in the vector unit instead of going through LDS.
__device__ __forceinline__ float lane_xor16(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  // Rows of 16 lanes r0 r1 r2 r3: the swap leaves (r0 r0 r2 r2, r1 r1 r3 r3).
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return __builtin_bit_cast(float, (threadIdx.x & 16) ? r[0] : r[1]);
}
__device__ __forceinline__ float lane_xor32(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  // Halves h0 h1: the swap leaves (h0 h0, h1 h1).
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (threadIdx.x & 32) ? r[0] : r[1]);
}

// The sum over the R neighbouring lanes of an aligned group, in every lane of the group: a butterfly whose steps stay
// in the vector unit (quad permutes, the mirrors of a half row and of a row, the swaps of rows and halves).  The order
// of the additions is fixed by R.
// (All lanes of a group are active where these are called, so that no lane keeps an old value and the compiler folds the permute into
// the addition: one instruction a step instead of four.)
__device__ __forceinline__ float dpp_f(float v, int ctrl_tag) {
  const int x = __builtin_bit_cast(int, v);
  int y;
  switch (ctrl_tag) {
    case 0: y = __builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, true); break;    // quad_perm [1, 0, 3, 2]
    case 1: y = __builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, true); break;    // quad_perm [2, 3, 0, 1]
    case 2: y = __builtin_amdgcn_mov_dpp(x, 0x141, 0xF, 0xF, true); break;   // row_half_mirror
    default: y = __builtin_amdgcn_mov_dpp(x, 0x140, 0xF, 0xF, true); break;  // row_mirror
  }
  return __builtin_bit_cast(float, y);
}
// The sum of a swap's two results.  (Each is copied first: a bit cast of a vector's element reads the vector's first one.)
template <typename PAIR>
__device__ __forceinline__ float pair_sum(const PAIR& r) {
  const unsigned a = r[0], b = r[1];
  return __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
}
template <int R>
__device__ __forceinline__ float group_sum(float v) {
  if (R >= 2) v = v + dpp_f(v, 0);
  if (R >= 4) v = v + dpp_f(v, 1);
  if (R >= 8) v = v + dpp_f(v, 2);
  if (R >= 16) v = v + dpp_f(v, 3);
  // A swap of a number with itself leaves the two rows' (halves') numbers in every lane of both, whichever was its own.
  if (R >= 32) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    v = pair_sum(__builtin_amdgcn_permlane16_swap(u, u, false, false));
  }
  if (R >= 64) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    v = pair_sum(__builtin_amdgcn_permlane32_swap(u, u, false, false));
  }
  return v;
}

// Sixteen of group_sum<16>'s sums at once (a recurrence's read-outs of 16 tokens): lane r of the 16 ends with the one of token
// walk_token(r).  Each step of the butterfly leaves a lane half as many; whether it goes on with the first or the second of two is chosen
// so that the partner of every later step has gone on with the same ones.
__device__ __forceinline__ int walk_token(int r) {
  const int b0 = r & 1, b1 = (r >> 1) & 1, b2 = (r >> 2) & 1, b3 = (r >> 3) & 1;
  return (b0 ^ b2) | (b1 ^ b2) << 1 | (b2 ^ b3) << 2 | b3 << 3;
}
__device__ __forceinline__ float walk_sums(float (&p)[16], int token) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float a = p[2 * i] + dpp_f(p[2 * i], 0), b = p[2 * i + 1] + dpp_f(p[2 * i + 1], 0);
    p[i] = token & 1 ? b : a;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = p[2 * i] + dpp_f(p[2 * i], 1), b = p[2 * i + 1] + dpp_f(p[2 * i + 1], 1);
    p[i] = token & 2 ? b : a;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float a = p[2 * i] + dpp_f(p[2 * i], 2), b = p[2 * i + 1] + dpp_f(p[2 * i + 1], 2);
    p[i] = token & 4 ? b : a;
  }
  const float a = p[0] + dpp_f(p[0], 3), b = p[1] + dpp_f(p[1], 3);
  return token & 8 ? b : a;
}

// The value of lane l ^ OFF where the steps 32, 16, 8, 4, 2, 1 of a butterfly over the whole wave are taken in this order, so that at
// step 4 lanes 8 apart hold the same value and a rotation of their row brings either: all in the vector unit (a shuffle through LDS
// is several times as long, and a norm of a few rows waits for six of them).  All lanes are active.
template <int OFF>
__device__ __forceinline__ float wave_partner(float v) {
  if (OFF == 32) return lane_xor32(v);
  if (OFF == 16) return lane_xor16(v);
  const int x = __builtin_bit_cast(int, v);
  const int y = OFF == 8   ? __builtin_amdgcn_mov_dpp(x, 0x128, 0xF, 0xF, true)      // row_ror:8
                : OFF == 4 ? __builtin_amdgcn_mov_dpp(x, 0x124, 0xF, 0xF, true)      // row_ror:4
                : OFF == 2 ? __builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, true)       // quad_perm [2, 3, 0, 1]
                           : __builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, true);      // quad_perm [1, 0, 3, 2]
  return __builtin_bit_cast(float, y);
}

// Butterflies over a wave: every lane ends with the same value; the order of the additions is fixed by the lane pattern (lanes 32
// apart first).
__device__ __forceinline__ float wave_sum_xor(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  v = pair_sum(__builtin_amdgcn_permlane32_swap(u, u, false, false));
  const unsigned w = __builtin_bit_cast(unsigned, v);
  v = pair_sum(__builtin_amdgcn_permlane16_swap(w, w, false, false));
  v = v + wave_partner<8>(v);
  v = v + wave_partner<4>(v);
  v = v + wave_partner<2>(v);
  return v + wave_partner<1>(v);
}
__device__ __forceinline__ float wave_max_xor(float v) {
  v = fmaxf(v, wave_partner<32>(v));
  v = fmaxf(v, wave_partner<16>(v));
  v = fmaxf(v, wave_partner<8>(v));
  v = fmaxf(v, wave_partner<4>(v));
  v = fmaxf(v, wave_partner<2>(v));
  return fmaxf(v, wave_partner<1>(v));
}

// Host side -----------------------------------------------------------------
#ifdef __cplusplus
extern "C" {
#endif
// Text of the last error on this thread ("" if none).
const char* vk_last_error(void);
#ifdef __cplusplus
}
#endif

int vk_fail(const char* fmt, ...) __attribute__((format(printf, 1, 2)));
int vk_check_launch(const char* what);

#define VK_REQUIRE(cond, ...)             \
  do {                                    \
    if (!(cond)) return vk_fail(__VA_ARGS__); \
  } while (0)

// Compute units of the current device.
static inline int vk_device_cus() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0, n = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
    cus = n > 0 ? n : 256;
  }
  return cus;
}
