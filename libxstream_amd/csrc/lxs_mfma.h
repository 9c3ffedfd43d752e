/*
 * Matrix-core helpers shared by the stack kernels (HIP device code, gfx950).
 *
 * MFMA 16x16x4 with one operand element per lane: lane l holds A[l % 16][l / 16] of a 16x4 A
 * fragment and B[l / 16][l % 16] of a 4x16 B fragment. Output tile 16x16, lane l, register r,
 * column l % 16: FP64 row = l/16 + 4r, FP32 row = 4(l/16) + r (checked on gfx950 with a probe).
 */
#ifndef LXS_MFMA_H
#define LXS_MFMA_H

#include <hip/hip_runtime.h>

namespace lxs {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

template <typename T>
struct mfma;
template <>
struct mfma<double> {
  typedef d4_t acc_t;
  static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <>
struct mfma<float> {
  typedef f4_t acc_t;
  static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

/* 4x4-block MFMA (checked on gfx950 with probes). FP64 v_mfma_f64_4x4x4_4b: four blocks of 4x4x4; lane l feeds
   k = l / 16 of block (l / 4) % 4, A row l % 4 and B column l % 4, and holds the block's result for A row l / 16
   and B column l % 4 (one register). FP32 v_mfma_f32_4x4x1_16b: sixteen blocks of 4x4x1; lane l feeds block
   l / 4 (its one k), A row l % 4 and B column l % 4, and holds the block's column l % 4 in its four registers
   (register r: row r). klane: the k within 16 that lane l feeds when the blocks of one instruction take
   consecutive k of the same C block. */
template <typename T>
struct mfma4;
template <>
struct mfma4<double> {
  typedef double acc_t;
  static constexpr bool FP32 = false;
  static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int klane(int lane) { return 4 * ((lane >> 2) & 3) + (lane >> 4); }
};
template <>
struct mfma4<float> {
  typedef f4_t acc_t;
  static constexpr bool FP32 = true;
  static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int klane(int lane) { return lane >> 2; }
};

/* zero operands for fragment lanes past k (read-only) */
__device__ const double zeros_f64[2] = {0.0, 0.0};
__device__ const float zeros_f32[4] = {0.0f, 0.0f, 0.0f, 0.0f};
template <typename T>
__device__ __forceinline__ const T* zeros();
template <>
__device__ __forceinline__ const double* zeros<double>() {
  return zeros_f64;
}
template <>
__device__ __forceinline__ const float* zeros<float>() {
  return zeros_f32;
}

/* load through the global address space: fragment pointers may point at the operand blocks or at
   the zero array, and a generic (flat) load would force the compiler to wait for all loads */
template <typename T>
__device__ __forceinline__ T gload(const T* p) {
  return *(const __attribute__((address_space(1))) T*)p;
}

/* two consecutive elements at the element type's alignment (one 16-byte load for FP64, 8-byte for FP32;
   the operand blocks only guarantee the element alignment) */
typedef double d2u_t __attribute__((ext_vector_type(2), aligned(8)));
typedef float f2u_t __attribute__((ext_vector_type(2), aligned(4)));
template <typename T>
struct pair_of;
template <>
struct pair_of<double> {
  typedef d2u_t type;
};
template <>
struct pair_of<float> {
  typedef f2u_t type;
};
template <typename T>
__device__ __forceinline__ typename pair_of<T>::type gload2(const T* p) {
  return *(const __attribute__((address_space(1))) typename pair_of<T>::type*)p;
}

/* Grouped tiles: up to V = 16 bytes / element size tiles of one dimension form a group whose rows (or columns)
   are interleaved, so that one load of up to 16 bytes per lane feeds all of them. Lane l of the group of G tiles from base on
   loads the G elements at s = min(base + G l, extent - G) (clamped so all stay inside the extent, which has at least G)
   for the group's tiles 0 .. G - 1. Output row l of its tile x is then element s + x; it is written by the one lane with
   s + x >= base + G l. */
template <typename T>
constexpr int group_max = 16 / (int)sizeof(T);
template <typename T>
__host__ __device__ constexpr int group_of(int c, int ntiles) { /* tiles of group c */
  return (ntiles - c * group_max<T> < group_max<T> ? ntiles - c * group_max<T> : group_max<T>);
}
template <typename T>
__device__ __forceinline__ int group_base(int c, int g, int l) { return 16 * group_max<T> * c + g * l; }
template <typename T>
__device__ __forceinline__ int group_start(int c, int g, int l, int extent) { return min(group_base<T>(c, g, l), extent - g); }

/* G consecutive elements at the element type's alignment */
typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));
struct f3u_t { float x, y, z; }; /* a vector of three would be loaded as four */
template <int G, typename T>
__device__ __forceinline__ void gload_group(T* v, const T* p) {
  if constexpr (1 == G) {
    v[0] = gload(p);
  }
  else if constexpr (2 == G) {
    const typename pair_of<T>::type w = gload2(p);
    v[0] = w[0];
    v[1] = w[1];
  }
  else if constexpr (3 == G) {
    const auto* const q = (const __attribute__((address_space(1))) f3u_t*)p;
    v[0] = q->x;
    v[1] = q->y;
    v[2] = q->z;
  }
  else {
    const f4u_t w = *(const __attribute__((address_space(1))) f4u_t*)p;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = w[i];
  }
}

/* this lane's elements of NTILE tiles, group by group */
template <int NTILE, int C, typename T>
__device__ __forceinline__ void gload_tiles(T* v, const T* p, const int* off) {
  constexpr int V = group_max<T>;
  gload_group<group_of<T>(C, NTILE)>(v + C * V, p + off[C]);
  if constexpr ((C + 1) * V < NTILE) gload_tiles<NTILE, C + 1>(v, p, off);
}

/* Sums over lanes without the LDS (DPP and the lane swaps of gfx950). Every lane l gets the sum over its row of 16
   of the lanes with the same l % 4 (sum_row), or over all rows as well (sum_blocks); lanes 0 .. 3 of a row add
   (x0 + x4) + (x8 + x12), then rows (0 + 1) + (2 + 3), the order that shuffles by 4, 8, 16, 32 give. */
template <int N> /* the value of lane (l - N) mod 16 of the row */
__device__ __forceinline__ float row_ror(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + N, 0xf, 0xf, true));
}
template <int N>
__device__ __forceinline__ double row_ror(double v) {
  typedef int i2_t __attribute__((ext_vector_type(2)));
  i2_t w = __builtin_bit_cast(i2_t, v);
  w.x = __builtin_amdgcn_update_dpp(0, w.x, 0x120 + N, 0xf, 0xf, true);
  w.y = __builtin_amdgcn_update_dpp(0, w.y, 0x120 + N, 0xf, 0xf, true);
  return __builtin_bit_cast(double, w);
}
template <typename T>
__device__ __forceinline__ T sum_row(T v) {
  v += row_ror<12>(v);
  return v + row_ror<8>(v);
}
__device__ __forceinline__ float sum_blocks(float v) {
  const unsigned int x = __builtin_bit_cast(unsigned int, sum_row(v));
  const auto rows = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  const unsigned int r0 = rows[0], r1 = rows[1];
  const unsigned int y = __builtin_bit_cast(unsigned int, __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1));
  const auto halves = __builtin_amdgcn_permlane32_swap(y, y, false, false);
  const unsigned int h0 = halves[0], h1 = halves[1];
  return __builtin_bit_cast(float, h0) + __builtin_bit_cast(float, h1);
}

/* Long C-runs are cut into pieces at the segment boundaries of the stack (multiples of the
   segment size bs, where one work-group's entries begin). Boundary entry i starts a new piece
   when the entry tsplit places earlier has the same C block ci: in a stack sorted by C, the run
   through i has then gone on for more than tsplit entries. The two owners that meet at i both
   evaluate this function of the stack alone, so each piece has exactly one owner; pieces of a cut
   run update their C block with atomic adds. tsplit <= 0: runs are never cut. */
__device__ __forceinline__ bool lxs_cut(const int* stack, int ps, int i, int ci, int tsplit) {
  return 0 < tsplit && tsplit <= i && stack[ps * (i - tsplit) + 2] == ci;
}

} /* namespace lxs */

#endif /*LXS_MFMA_H*/
