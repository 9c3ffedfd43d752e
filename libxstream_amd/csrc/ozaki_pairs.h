/*
 * Ozaki scheme I, the whole product of a call in one kernel (gfx950): every slice pair (p, q) with p + q <= cutoff,
 * all levels of an output tile in registers, recombined and stored without int32 partials in memory.
 * The digits and planes are those of oz_slice (ozaki.hip), the result bit for bit that of oz_level_gemm followed by
 * oz_recombine: S_L exact in int32, cd = sum over L = cutoff .. 0 of 2^(-7(L+2)) S_L in FP64,
 * C = fma(alpha, 2^(ea + eb) cd, beta C).
 */
#ifndef LXS_OZAKI_PAIRS_H
#define LXS_OZAKI_PAIRS_H

#include <hip/hip_runtime.h>
#include <stdint.h>
#include "lxs_kernels.h"

namespace {

typedef int i4_t __attribute__((ext_vector_type(4)));
typedef int i16_t __attribute__((ext_vector_type(16)));

constexpr int PT = 64;                 /* columns (j) of a work-group's tile, k of a block */
constexpr int PROWS = 256;             /* rows of a plane tile (oz_plane_off: 256 rows x 64 k, 16 KB contiguous) */
constexpr int PNONE = -(1 << 30);      /* exponent of a row without a nonzero element */

__device__ __forceinline__ void ozp_dma16(const int8_t* src, int8_t* lds_dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
    (__attribute__((address_space(3))) void*)lds_dst, 16, 0, 0);
}

/* one bit per plane that holds a nonzero digit (one load for all of them) */
__device__ __forceinline__ unsigned int oz_occupied(const int* occ, int s) {
  const int lane = threadIdx.x & 63;
  return (unsigned int)__ballot(lane < s && 0 != occ[lane < s ? lane : 0]);
}
/* the pairs p + q <= cutoff with digits in both planes; levels: one bit per level p + q that has any */
__device__ __forceinline__ int oz_some_pairs(unsigned int oa, unsigned int ob, int s, int cutoff, unsigned int& levels) {
  int some = 0;
  levels = 0;
  for (int p = 0; p < s && p <= cutoff; ++p) {
    const unsigned int q = (0 != ((oa >> p) & 1u) ? ob & ((2u << (cutoff - p)) - 1u) : 0u);
    some += __popc(q);
    levels |= q << p;
  }
  return some;
}
/* all pairs up to the cutoff s - 1 or 2 (s - 1) */
__host__ __device__ constexpr int oz_all_pairs(int s, int cutoff) { return (2 * (s - 1) == cutoff ? s * s : s * (s + 1) / 2); }
/* products without branches, of zero planes and all: faster than branches above 0.65 of the pairs (4096^3, ms: 8 slices,
   triangle, 24 of 36 pairs 2.29 with branches, 2.16 without; all pairs, 36 of 64 2.77 and 3.06), for 3 slices above 0.7
   (4 of 6 pairs 0.594 with, 0.641 without) */
__device__ __forceinline__ bool oz_branch_free(int some, int s, int cutoff) {
  return 20 * some > (3 < s ? 13 : 14) * oz_all_pairs(s, cutoff);
}
/*
 * 1 when oz_level_gemm and oz_recombine, which move and multiply only the planes with digits, are faster than oz_pairs,
 * which moves every plane of a tile: the products of the pairs with digits, and int32 partials per level that cost about
 * as much as 3000 k of a pair, against the products of all pairs. ms a call by the bits of whole numbers in FP64 (one
 * plane per 7), oz_pairs / the other two: 8192^3, 8 slices, triangle: 7 bits 11.5 / 1.6, 21 13.2 / 5.6, 35 16.0 / 12.3, 42
 * 15.7 / 14.9; 4096^3 all pairs 7 1.64 / 0.42, 28 2.2 / 1.47, 42 2.8 / 2.66; 8192x8192x1024 all pairs 28 2.34 / 2.23, 35
 * 2.58 / 2.97, 6 slices 28 1.79 / 2.15. The partials cost more where all pairs share a tile's loads.
 * A triangle of few slices has few products for the planes that oz_pairs moves for a tile of 128 x 64 (3 slices: 2 pairs a
 * plane, 8: 4.5), 1.5 times the time of 8 slices per pair, and the other two win with all planes from K = 4000 on (3 slices)
 * and 6000 (4): 3 slices 8192^3 4.32 / 3.51, 3000x3000x16000 1.60 / 1.35, 5000^3 1.14 / 1.14, 8192x8192x2048 1.36 / 1.40;
 * 4 slices 8192^3 6.46 / 5.43, 5500x5500x8192 2.94 / 2.89, 6000x6000x3000 1.26 / 1.48; 5 slices with 4 planes 8192^3 8.0 /
 * 7.2, with all 7.91 / 7.85.
 */
__device__ __forceinline__ bool oz_few_pairs(unsigned int oa, unsigned int ob, int s, int cutoff, int Kp) {
  unsigned int levels;
  const int some = oz_some_pairs(oa, ob, s, cutoff, levels), all = oz_all_pairs(s, cutoff);
  long cost = (2 * (s - 1) == cutoff ? 75L : 92L); /* of a pair in oz_pairs, in hundredths */
  if (s - 1 == cutoff && 5 >= s && 20 * some > 13 * all) cost = (3 >= s ? 138L : (4 == s ? 120L : 103L));
  /* whole numbers: the three kernels of a call have to agree */
  return 100L * ((long)some * Kp + 3000L * __popc(levels)) <= cost * all * Kp;
}

/*
 * A work-group of 4 wavefronts (2 x 2) computes 64 WI x 64 elements of C, a wavefront 32 WI x 32 (v_mfma_i32_32x32x32_i8,
 * the B planes as first operand as in oz_level_gemm): CUT + 1 level sums of 16 WI registers each. Per block of 64 k the
 * NS planes of its A rows and B columns move into LDS by DMA once (64 KB for 8 slices) and serve every pair: 128
 * matrix instructions per wavefront and block for 8 slices over all pairs, where a kernel that takes the pairs one by
 * one moves both operands again for each of them.
 * LDS rows of 64 bytes, chunk c of row r at c ^ ((r >> 2) & 3). Two buffers, alternating by block; the fragments of
 * a half block (32 k) are read while the other half is multiplied: at mid-block a wavefront has read all of the
 * block and its DMA of the next has landed, so after the barrier there the buffer is refilled with the block after
 * next, a whole block of matrix work ahead of its use.
 * Where the tiles would leave CUs idle, gridDim.y work-groups share a tile's k and write their level sums (int32) for
 * oz_recombine.
 * Bound: the matrix cores, busy 0.81 of the time at 4096^3 with 8 slices over all pairs, at the clock the card holds under
 * int8 products (1.73 GHz): 4336 -> 3307 us a call; 1000x1100x900 267 -> 141 (the level GEMM wrote and oz_recombine
 * read 57 planes of int32 partials, 300 MB), 4000x3000x70 506 -> 175, FP32 2500x2600x1111 438 -> 276. With k shared:
 * 64x64x4096 168 -> 111 (one work-group alone: 184), 512x512x4096 408 -> 239. int32 sums are exact for NS Kp / 64 <= 2080 (2080 * 64 * 127^2 < 2^31).
 */
template <int NS, int CUT, int WI>
__global__ void __launch_bounds__(256) oz_pairs(const int8_t* __restrict__ pa, const int8_t* __restrict__ pb,
  const int* __restrict__ occa, const int* __restrict__ occb, int Mp, int Np, int Kp, int tiles_m, int tiles_n,
  const int* __restrict__ ea, const int* __restrict__ eb, int M, int N, double alpha, double beta, int dtype,
  void* __restrict__ c, long ldc, int* __restrict__ part, int gate) {
  constexpr int RA = 64 * WI, BUF = NS * (RA + PT) * 64, NDMA = NS * (WI + 1);
  __shared__ __attribute__((aligned(1024))) int8_t lds0[BUF], lds1[BUF];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wi = wave & 1, wj = wave >> 1;
  /* work-groups go to the 8 XCDs in turn: each takes one contiguous part of the tiles, in bands of 8 tile rows, so
     that the operands of its resident work-groups meet in its L2 */
  int t = blockIdx.x;
  {
    const int per = tiles_m * tiles_n / 8;
    if (t < 8 * per) t = (t & 7) * per + (t >> 3);
  }
  const int band = t / (8 * tiles_n), rows = min(8, tiles_m - 8 * band), tb = t - 8 * tiles_n * band;
  const int i0 = (8 * band + tb % rows) * RA, j0 = (tb / rows) * PT;
  const int nkb = Kp / 64; /* even: planes are padded to 128 k */
  /* this work-group's blocks of k (all of them, or part blockIdx.y of gridDim.y, a multiple of two) */
  const int kb0 = 2 * (int)((long)(nkb / 2) * blockIdx.y / gridDim.y);
  const int kb1 = 2 * (int)((long)(nkb / 2) * (blockIdx.y + 1) / gridDim.y);
  constexpr unsigned int EVERY = (1u << NS) - 1u;
  unsigned int oa = oz_occupied(occa, NS), ob = oz_occupied(occb, NS); /* the planes to move and multiply */
  if (0 != gate && oz_few_pairs(oa, ob, NS, CUT, Kp)) return; /* oz_level_gemm's */
  {
    unsigned int levels;
    if (oz_branch_free(oz_some_pairs(oa, ob, NS, CUT, levels), NS, CUT)) oa = ob = EVERY;
  }
  i16_t acc[CUT + 1][WI];
#pragma unroll
  for (int L = 0; L <= CUT; ++L) {
#pragma unroll
    for (int x = 0; x < WI; ++x) acc[L][x] = i16_t{0};
  }
  /* wavefront w moves rows 16 w .. + 15 of every 64 rows of every plane: lane l writes position l % 4 of row l / 4 */
  const unsigned int doff = (unsigned int)(16 * wave + (lane >> 2)) * 64 + 16u * ((lane & 3) ^ ((lane >> 4) & 3));
  const int8_t* const ga = pa + ((long)(i0 / PROWS) * nkb * PROWS + i0 % PROWS) * 64;
  const int8_t* const gb = pb + ((long)(j0 / PROWS) * nkb * PROWS + j0 % PROWS) * 64;
  const long sa = (long)Mp * Kp, sb = (long)Np * Kp; /* bytes of a plane */
  const auto dma = [&](int8_t* buf, int kb, unsigned int ma, unsigned int mb) { /* ma, mb: the planes of A and B to move */
    const int8_t* const ka = ga + (long)kb * (PROWS * 64);
    const int8_t* const kbp = gb + (long)kb * (PROWS * 64);
#pragma unroll
    for (int p = 0; p < NS; ++p) {
      if (0 != ((ma >> p) & 1u)) {
#pragma unroll
        for (int x = 0; x < WI; ++x) ozp_dma16(ka + p * sa + x * 4096 + doff, buf + p * RA * 64 + x * 4096 + wave * 1024);
      }
      if (0 != ((mb >> p) & 1u)) ozp_dma16(kbp + p * sb + doff, buf + NS * RA * 64 + p * 4096 + wave * 1024);
    }
  };
  const int frow = lane & 31, fswz = (frow >> 2) & 3;
  const int fpos[2] = {((lane >> 5) ^ fswz) * 16, ((2 + (lane >> 5)) ^ fswz) * 16};
  i4_t fa[2][NS][WI], fb[2][NS];
  const auto frags = [&](const int8_t* buf, int half, int set) {
#pragma unroll
    for (int p = 0; p < NS; ++p) {
      fb[set][p] = *(const i4_t*)(buf + NS * RA * 64 + p * 4096 + (32 * wj + frow) * 64 + fpos[half]);
#pragma unroll
      for (int x = 0; x < WI; ++x) {
        fa[set][p][x] = *(const i4_t*)(buf + p * RA * 64 + (32 * (WI * wi + x) + frow) * 64 + fpos[half]);
      }
    }
  };
  constexpr int NM = [] {
    int n = 0;
    for (int p = 0; p < NS; ++p) {
      for (int q = 0; q < NS; ++q) n += (p + q <= CUT ? WI : 0);
    }
    return n;
  }();
  const auto mfmas = [&](int set) {
#pragma unroll
    for (int p = 0; p < NS; ++p) {
#pragma unroll
      for (int q = 0; q < NS; ++q) {
        if (p + q <= CUT) {
#pragma unroll
          for (int x = 0; x < WI; ++x) {
            acc[p + q][x] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[set][q], fa[set][p][x], acc[p + q][x], 0, 0, 0);
          }
        }
      }
    }
  };
#define OZP_MIDSYNC() \
  do { \
    __builtin_amdgcn_s_waitcnt(0); /* own reads of this block, own DMA of the next (the one in flight) */ \
    __asm__ __volatile__("" ::: "memory"); \
    __builtin_amdgcn_s_barrier(); /* no fence: DMA and reads are counted above */ \
    __asm__ __volatile__("" ::: "memory"); \
  } while (0)
  dma(lds0, kb0, oa, ob);
  OZP_MIDSYNC();
  dma(lds1, kb0 + 1, oa, ob);
  frags(lds0, 0, 0);
  if (EVERY == (oa & ob)) { /* no branches */
    /* a block: its second half's fragments while the first half is multiplied; then the DMA of the block after next
       and the next block's first fragments while the second half is multiplied */
#define OZP_BLOCK(CUR, NXT, KB) \
  do { \
    frags(CUR, 1, 1); \
    mfmas(0); \
    _Pragma("unroll") for (int i_ = 0; i_ < NS * (WI + 1); ++i_) { \
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); /* DS read */ \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); /* MFMA */ \
    } \
    if constexpr (NM > NS * (WI + 1)) __builtin_amdgcn_sched_group_barrier(0x008, NM - NS * (WI + 1), 0); \
    OZP_MIDSYNC(); \
    dma(CUR, min((KB) + 2, kb1 - 1), EVERY, EVERY); \
    frags(NXT, 0, 0); \
    mfmas(1); \
    _Pragma("unroll") for (int i_ = 0; i_ < NS * (WI + 1); ++i_) { \
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); \
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0); /* VMEM read (DMA) */ \
    } \
    if constexpr (NM > NS * (WI + 1)) __builtin_amdgcn_sched_group_barrier(0x008, NM - NS * (WI + 1), 0); \
  } while (0)
    for (int kb = kb0; kb < kb1; kb += 2) {
      OZP_BLOCK(lds0, lds1, kb);
      OZP_BLOCK(lds1, lds0, kb + 1);
    }
#undef OZP_BLOCK
  }
  else { /* products of planes without a nonzero digit are skipped */
    const auto some = [&](int set) {
#pragma unroll
      for (int p = 0; p < NS; ++p) {
        if (0 == ((oa >> p) & 1u)) continue;
#pragma unroll
        for (int q = 0; q < NS; ++q) {
          if (p + q <= CUT && 0 != ((ob >> q) & 1u)) {
#pragma unroll
            for (int x = 0; x < WI; ++x) {
              acc[p + q][x] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[set][q], fa[set][p][x], acc[p + q][x], 0, 0, 0);
            }
          }
        }
      }
    };
    for (int kb = kb0; kb < kb1; kb += 2) {
      frags(lds0, 1, 1);
      some(0);
      OZP_MIDSYNC();
      dma(lds0, min(kb + 2, kb1 - 1), oa, ob);
      frags(lds1, 0, 0);
      some(1);
      frags(lds1, 1, 1);
      some(0);
      OZP_MIDSYNC();
      dma(lds1, min(kb + 3, kb1 - 1), oa, ob);
      frags(lds0, 0, 0);
      some(1);
    }
  }
#undef OZP_MIDSYNC
  __builtin_amdgcn_s_waitcnt(0); /* the last DMA lands before the work-group ends */
  if (NULL != part) { /* the level sums of this part of k: level L at plane L gridDim.y + blockIdx.y */
#pragma unroll
    for (int L = 0; L <= CUT; ++L) {
      int* const o = part + (long)(L * gridDim.y + blockIdx.y) * Mp * Np;
#pragma unroll
      for (int x = 0; x < WI; ++x) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int j = j0 + 32 * wj + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          o[(long)j * Mp + i0 + 32 * (WI * wi + x) + (lane & 31)] = acc[L][x][r];
        }
      }
    }
    return;
  }
#pragma unroll
  for (int x = 0; x < WI; ++x) {
    const int i = i0 + 32 * (WI * wi + x) + (lane & 31);
    const int ex = ea[i]; /* rows up to the padding have an exponent (none) */
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int j = j0 + 32 * wj + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
      const int ey = eb[j];
      double cd = 0;
#pragma unroll
      for (int L = CUT; L >= 0; --L) cd = fma(ldexp(1.0, -7 * (L + 2)), (double)acc[L][x][r], cd);
      const double v = (PNONE != ex && PNONE != ey) ? ldexp(cd, ex + ey) : 0.0;
      if (i < M && j < N) {
        if (3 == dtype) {
          double* const pc = (double*)c + i + (long)j * ldc;
          *pc = (0 != beta ? fma(alpha, v, beta * *pc) : alpha * v);
        }
        else {
          float* const pc = (float*)c + i + (long)j * ldc;
          *pc = (float)(0 != beta ? fma(alpha, v, beta * (double)*pc) : alpha * v);
        }
      }
    }
  }
}

template <int NS, int CUT>
int oz_pairs_launch(const int8_t* pa, const int8_t* pb, const int* occa, const int* occb, int Mp, int Np, int Kp, const int* ea,
  const int* eb, int M, int N, double alpha, double beta, int dtype, void* c, int ldc, int ks, int* part, int gate, hipStream_t st) {
  /* 128 rows of A per tile where the level sums fit 256 registers and two buffers the LDS */
  constexpr int WI = (32 * (CUT + 1) <= 256 && NS <= 6 ? 2 : 1);
  const int tm = (M + 64 * WI - 1) / (64 * WI), tn = (N + PT - 1) / PT;
  if ((double)tm * tn > 2147483647.0) return LXS_ELIMIT;
  oz_pairs<NS, CUT, WI><<<dim3((unsigned int)(tm * tn), (unsigned int)ks), 256, 0, st>>>(pa, pb, occa, occb, Mp, Np, Kp, tm,
    tn, ea, eb, M, N, alpha, beta, dtype, c, (long)ldc, part, gate);
  return (int)hipGetLastError();
}

} /* namespace */

extern "C" int lxs_oz_pairs_fits(int s, int cutoff, int Kp) {
  return (1 <= s && s <= 8 && (s - 1 == cutoff || 2 * (s - 1) == cutoff) && 0 < Kp && s * (Kp / 64) <= 2080) ? 1 : 0;
}

extern "C" int lxs_oz_pairs_split(int s, int cutoff, int M, int N, int Kp, int nitems) {
  const int wi = (32 * (cutoff + 1) <= 256 && s <= 6 ? 2 : 1);
  const long tiles = (long)((M + 64 * wi - 1) / (64 * wi)) * ((N + PT - 1) / PT);
  long ks = (0 < tiles ? 256 / tiles : 1);
  if (nitems / (cutoff + 1) < ks) ks = nitems / (cutoff + 1);
  if (Kp / 512 < ks) ks = Kp / 512; /* at least 8 blocks each */
  return (2 <= ks ? (int)ks : 1);
}

/* from this much work on (pairs x M x N x K; 0.6 ms of products) a call launches oz_pairs and oz_level_gemm, of which one
   leaves the work to the other by the planes that hold digits */
constexpr double OZP_GATE_WORK = 5e11;

extern "C" int lxs_oz_pairs_gate(int s, int cutoff, int M, int N, int Kp, int ks) {
  return (1 == ks && 2 < s && OZP_GATE_WORK <= (double)oz_all_pairs(s, cutoff) * M * N * Kp) ? 1 : 0;
}

extern "C" int lxs_oz_pairs(int dtype, const signed char* pa, const signed char* pb, const int* occa, const int* occb, int s,
  int cutoff, int Mp, int Np, int Kp, const int* ea, const int* eb, int M, int N, double alpha, double beta, void* c, int ldc,
  int ks, int* part, int gate, void* hip_stream) {
  const hipStream_t st = (hipStream_t)hip_stream;
  const int8_t *a8 = (const int8_t*)pa, *b8 = (const int8_t*)pb;
  int result;
  if (0 == lxs_oz_pairs_fits(s, cutoff, Kp) || 0 != Mp % 256 || 0 != Np % 256 || 0 != Kp % 128 || Mp < M || Np < N ||
      1 > ks || Kp / 128 < ks || (1 < ks && (NULL == part || 0 != gate))) {
    return LXS_ELIMIT;
  }
  if (3 != dtype && 1 != dtype) return LXS_ENOVARIANT;
  if (0 >= M || 0 >= N) return 0;
  if (1 == ks) part = NULL;
#define OZP_CASE(NS) \
  case NS: \
    result = (NS - 1 == cutoff) ? oz_pairs_launch<NS, NS - 1>(a8, b8, occa, occb, Mp, Np, Kp, ea, eb, M, N, alpha, beta, \
                                    dtype, c, ldc, ks, part, gate, st) \
                                : oz_pairs_launch<NS, 2 * (NS - 1)>(a8, b8, occa, occb, Mp, Np, Kp, ea, eb, M, N, alpha, \
                                    beta, dtype, c, ldc, ks, part, gate, st); \
    break;
  switch (s) {
    OZP_CASE(1)
    OZP_CASE(2)
    OZP_CASE(3)
    OZP_CASE(4)
    OZP_CASE(5)
    OZP_CASE(6)
    OZP_CASE(7)
    OZP_CASE(8)
    default: return LXS_ELIMIT;
  }
#undef OZP_CASE
  if (0 == result && 1 < ks) { /* level L: the ks partials from L ks on */
    int zb[17], L;
    for (L = 0; L <= cutoff + 1; ++L) zb[L] = L * ks;
    result = lxs_oz_recombine(dtype, part, zb, cutoff, Mp, Np, ea, eb, M, N, alpha, beta, c, ldc, NULL, NULL, s, 0,
      hip_stream);
  }
  return result;
}

#endif /* LXS_OZAKI_PAIRS_H */
