/*
 * Ozaki scheme I over a DBCSR parameter stack (gfx950): C[c] += A[a] B[b] for every stack entry, the
 * products emulated with int8 matrix cores. No counterpart in the reference (its Ozaki sample,
 * samples/ozaki/, multiplies whole matrices); the stack semantics are those of libsmm_acc_process
 * (samples/smm/kernels/multiply.cl:12-20, 1-based element offsets in triplets, A column-major m x k,
 * B in the kernel layout k x n row-major, C column-major m x n) and the digits those of ozaki_gemm
 * (per-row exponent, 7-bit signed digits, levels recombined in FP64).
 *
 *   ozs_slice   every block of a pool -> s digit planes of 64 x 64 int8 (rows of A, columns of B;
 *               k contiguous) and the 64 row exponents; padding rows and k are zero.
 *   ozs_check   whether C offsets ever decrease (the stack is then not grouped by C).
 *   ozs_stack   persistent: work-group g owns the runs (entries of one C offset) that start in its equal
 *               share of the stack and walks each to its end; a run's C block stays in registers
 *               (FP64, or FP32 updated through FP64); per entry the 2s digit planes of its A and B
 *               blocks move into LDS by DMA (double-buffered across entries), every level sum
 *               S_L = sum over pairs p + q = L of A_p B_q^T (64 x 64 x 64) accumulates exactly in its own
 *               int32 tile (v_mfma_i32_16x16x64_i8, 8 wavefronts of 32 x 16), then
 *               cd = sum over L = cutoff .. 0 of 2^(-7(L+2)) S_L in FP64 and C += 2^(ea_i + eb_j) cd.
 *               A stack that is not sorted by C is processed by one work-group, run after run, in order.
 * Every element of C is therefore updated entry by entry in stack order, reproducibly.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "lxs_kernels.h"

namespace {

typedef int i4_t __attribute__((ext_vector_type(4)));
typedef int i16_t __attribute__((ext_vector_type(16)));

constexpr int SB = 64;           /* block rows, columns and k, padded */
constexpr int SPL = SB * SB;     /* bytes of one digit plane */
constexpr int SNONE = -(1 << 30);

__device__ __forceinline__ int ozs_expo(double v) { /* |v| < 2^ex for a normal finite v */
  const long long bits = __double_as_longlong(v);
  const int be = (int)((bits >> 52) & 0x7FF);
  return (0 == be || 0x7FF == be) ? SNONE : be - 1022;
}
__device__ __forceinline__ int ozs_expo(float v) {
  const int bits = __float_as_int(v);
  const int be = (bits >> 23) & 0xFF;
  return (0 == be || 0xFF == be) ? SNONE : be - 126;
}

/*
 * Pool slicing: block b of the pool, element (r, kk) at p[b * bsz + r * rs + kk * ks] for r < R, kk < K.
 * Thread t owns row t / 4 and k = 16 (t % 4) .. +15; the row exponent is the maximum over 4 lanes.
 * Planes at planes[((b * s + pl) * 64 + r) * 64 + kk]; exponents at ex[b * 64 + r].
 */
template <typename T>
__global__ void __launch_bounds__(256) ozs_slice(const T* __restrict__ p, long bsz, int rs, int ks, int R, int K, int s,
  int8_t* __restrict__ planes, int* __restrict__ ex) {
  const long blk = blockIdx.x;
  const int t = threadIdx.x, r = t >> 2, kq = (t & 3) * 16;
  const T* const src = p + blk * bsz;
  double v[16];
  int e = SNONE;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const T x = (r < R && kq + i < K) ? src[(long)r * rs + (long)(kq + i) * ks] : T(0);
    const int ev = ozs_expo(x);
    v[i] = (SNONE != ev ? (double)x : 0.0);
    e = max(e, ev);
  }
  e = max(e, __shfl_xor(e, 1));
  e = max(e, __shfl_xor(e, 2));
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = (SNONE != e ? ldexp(v[i], -e) : 0.0); /* |x| < 1, exact */
  for (int pl = 0; pl < s; ++pl) {
    union {
      int8_t b[16];
      i4_t w;
    } d;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const double y = v[i] * 128.0;
      const double q = trunc(y); /* |q| <= 127 */
      d.b[i] = (int8_t)q;
      v[i] = y - q; /* exact */
    }
    *(i4_t*)(planes + ((blk * s + pl) * SB + r) * SB + kq) = d.w;
  }
  if (0 == (t & 3)) ex[blk * SB + r] = e;
}

__global__ void ozs_clear(int* __restrict__ info) { info[threadIdx.x] = 0; }

/* info[0] = 1 when some C offset is smaller than its predecessor's */
__global__ void __launch_bounds__(256) ozs_check(const int* __restrict__ stack, int S, int* __restrict__ info) {
  int bad = 0;
  for (int i = blockIdx.x * 256 + threadIdx.x + 1; i < S; i += gridDim.x * 256) {
    bad |= (stack[3 * i + 2] < stack[3 * (i - 1) + 2]) ? 1 : 0;
  }
  if (0 != __syncthreads_or(bad) && 0 == threadIdx.x) atomicOr(info, 1);
}

__device__ __forceinline__ void ozs_dma16(const int8_t* src, int8_t* lds_dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
    (__attribute__((address_space(3))) void*)lds_dst, 16, 0, 0);
}
__device__ __forceinline__ void ozs_dma4(const int* src, int8_t* lds_dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
    (__attribute__((address_space(3))) void*)lds_dst, 4, 0, 0);
}
constexpr int SEX = 2 * SB * 4; /* LDS bytes of an entry's exponent rows (A rows, then B columns) */

/*
 * LDS: two entry buffers of 2 NS planes (A planes, then B planes), 4 KB each, and the entry's exponent rows; row r of a
 * plane holds its 4 chunks of 16 bytes with chunk c at position c ^ ((r >> 2) & 3). Wavefronts 0..3 move the planes
 * of A, 4..7 those of B, wavefront w rows 16 (w & 3) .. + 15 (one DMA instruction per plane: lane l writes position
 * l % 4 of row 16 (w & 3) + l / 4); rows past m or n are not moved, what they leave in the tile is not stored.
 *
 * 8 wavefronts, two per SIMD, each 32 x 16 elements of the block (v_mfma_i32_16x16x64_i8: all 64 k in one instruction,
 * the B planes as first operand): 15 level sums of 8 registers each for 8 slices over all pairs. Wavefronts 4..7 cross the
 * barrier of an entry between its products and its recombination, 0..3 before its products: on every SIMD one
 * wavefront's FP64 recombination (120 conversions and 120 FMA) runs beside the other's products. The entries of a
 * work-group follow each other without a break from run to run, and the records of 64 of them are one lane each
 * (chains of dependent scalar loads before an entry's DMA: 1791 -> 1976 us below).
 * Bound: 8 slices over all pairs, the products (4096 cycles an entry and SIMD) and what of the DMA (64 KB an entry, 3.7 TB/s
 * over the device) and the barrier they do not cover. With 4 wavefronts of 32 x 32, one per SIMD, products and
 * recombination took turns. us a call, before -> now: FP64 64x64x64, 100000 entries, 8 slices 2583 -> 1791, 20000 entries, 7
 * slices 584 -> 326; 23x23x23, 50000, 8 slices 1379 -> 517; 33x13x50, 5000, 6 slices 175 -> 76; FP32 64x30x64, 100000, 3 slices
 * 603 -> 354. Work-groups as many as are resident: 256 (5 to 8 slices) 517 us and 512 625 us for 23x23x23 above, two per
 * CU for 3 and 4 slices (FP32 45x45x13, 60000, 4 slices: 512 353 us, 256 488, 1024 401).
 */
template <typename T, int NS, int CUT>
__global__ void __launch_bounds__(512, (4 >= NS ? 4 : 2)) ozs_stack(const int* __restrict__ stack, int S,
  const int* __restrict__ info, const int8_t* __restrict__ pa, const int* __restrict__ ea, const int8_t* __restrict__ pb,
  const int* __restrict__ eb, int cutoff_rt, int m, int n, int k, int na, int nb, T* __restrict__ c) {
  /* the level cutoff: compiled in (CUT >= 0), so the pair loop below has no conditional matrix-core work,
     or taken at run time (CUT < 0) */
  const int cutoff = (0 <= CUT ? CUT : cutoff_rt);
  __shared__ __attribute__((aligned(1024))) int8_t lds0[2 * NS * SPL + SEX], lds1[2 * NS * SPL + SEX];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int late = wave >> 2; /* 1: recombines an entry after the next barrier */
  const int wi = wave & 1, wj = ((wave >> 1) & 1) + 2 * late;
  const int unsorted = info[0];
  const unsigned int mk = (unsigned int)(m * k), kn = (unsigned int)(k * n);
  /* this work-group's share of the stack (all of it for work-group 0 when the stack is not grouped by C) */
  const int share = (S + (int)gridDim.x - 1) / (int)gridDim.x;
  const int lo = (0 != unsorted ? 0 : (int)blockIdx.x * share);
  const int hi = (0 != unsorted ? S : (lo + share < S ? lo + share : S));
  if (0 != unsorted && 0 != blockIdx.x) return;
  /* run boundaries found 64 entries at a time (one lane each, then a ballot): from the first run that starts in
     [lo, hi) to the end of the last one */
  const auto first_start = [&](int x0, int x1) {
    for (; x0 < x1; x0 += 64) {
      const int x = x0 + lane;
      const unsigned long long bal = __ballot(x < x1 && (0 == x || stack[3 * x + 2] != stack[3 * (x - 1) + 2]));
      if (0 != bal) return x0 + __ffsll((long long)bal) - 1;
    }
    return x1;
  };
  const int e0 = __builtin_amdgcn_readfirstlane(first_start(lo, hi));
  if (e0 >= hi) return;
  const int e1 = __builtin_amdgcn_readfirstlane(first_start(hi, S));
  /* the DMA of this wavefront: planes of one operand, 16 of their rows */
  const int dr = 16 * (wave & 3), drow = dr + (lane >> 2), dchunk = (lane & 3) ^ ((lane >> 4) & 3);
  const bool dma_any = (dr < (0 == late ? m : n));
  const int8_t* const dsrc = (0 == late ? pa : pb) + drow * SB + 16 * dchunk;
  const int* const dex = (0 == late ? ea : eb) + lane;
  /* the tile: columns i (A rows) 32 wi + 16 x + lane % 16, rows j (B columns) 16 wj + 4 (lane / 16) + r per register */
  const bool active = (32 * wi < m && 16 * wj < n);
  const int frow = lane & 15, fpos = 16 * ((lane >> 4) ^ ((frow >> 2) & 3));
  const int i0 = 32 * wi + frow, j0 = 16 * wj + 4 * (lane >> 4);
  double creg[2][4];
  i4_t acc[2 * NS - 1][2];
  int exi[2];
  i4_t exj;
  /* entries base .. base + 63, one per lane: the blocks of A and B (-1 when an offset is not a block start inside the
     pool) and the C offset; first, last: bit l set when entry base + l begins or ends a run */
  int base, wa, wb, wc;
  unsigned long long firsts, lasts;
  const auto block_of = [](int ofs, unsigned int sz, int cnt) {
    const unsigned int q = (unsigned int)ofs / sz;
    return (0 <= ofs && (unsigned int)ofs == q * sz && q < (unsigned int)cnt) ? (int)q : -1;
  };
  const auto window = [&](int x0) {
    const int x = min(x0 + lane, S - 1);
    const int ra = stack[3 * x], rb = stack[3 * x + 1], rc = stack[3 * x + 2];
    const int before = stack[3 * max(x - 1, 0) + 2], after = stack[3 * min(x + 1, S - 1) + 2];
    wa = block_of(ra - 1, mk, na);
    wb = block_of(rb - 1, kn, nb);
    wc = rc;
    firsts = __ballot(x == e0 || before != rc);
    lasts = __ballot(x + 1 >= e1 || after != rc);
    base = x0;
  };
  /* entry e into buffer e % 2; an entry without valid blocks loads block 0, unused */
  const auto dma = [&](int8_t* buf, int e) {
    const int blk = max(__builtin_amdgcn_readlane(0 == late ? wa : wb, e - base), 0);
    if (dma_any) {
#pragma unroll
      for (int pl = 0; pl < NS; ++pl) {
        ozs_dma16(dsrc + ((long)blk * NS + pl) * SPL, buf + (late * NS + pl) * SPL + (wave & 3) * 1024);
      }
    }
    if (0 == (wave & 3)) ozs_dma4(dex + (long)blk * SB, buf + 2 * NS * SPL + late * SB * 4);
  };
  bool valid = false, last = false; /* of the entry whose level sums are in acc */
  T* cblk = c;
  const auto recombine = [&]() {
    if (valid) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          double cd = 0.0;
#pragma unroll
          for (int L = 2 * NS - 2; 0 <= L; --L) {
            if (L <= cutoff) cd = fma(ldexp(1.0, -7 * (L + 2)), (double)acc[L][x][r], cd);
          }
          const double v = (SNONE != exi[x] && SNONE != exj[r]) ? ldexp(cd, exi[x] + exj[r]) : 0.0;
          creg[x][r] = (double)(T)(creg[x][r] + v);
        }
      }
    }
    if (last && active) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (i0 + 16 * x < m && j0 + r < n) cblk[i0 + 16 * x + (long)(j0 + r) * m] = (T)creg[x][r];
        }
      }
    }
  };
  window(e0);
  dma(lds0, e0);
  for (int e = e0; e < e1; ++e) {
    int8_t* const cur = (0 == ((e - e0) & 1) ? lds0 : lds1);
    int8_t* const nxt = (0 == ((e - e0) & 1) ? lds1 : lds0);
    __builtin_amdgcn_s_waitcnt(0); /* own DMA of entry e, own reads of entry e - 1 */
    __syncthreads();              /* every wave's DMA of e has landed, every wave is done with e - 1 */
    if (e + 1 - base >= 64) window(e);
    dma(nxt, min(e + 1, e1 - 1)); /* the last entry loads itself again, unused */
    if (0 != late && e != e0) recombine();
    {
      const int l = e - base;
      const bool first = (0 != ((firsts >> l) & 1));
      last = (0 != ((lasts >> l) & 1));
      cblk = c + ((long)__builtin_amdgcn_readlane(wc, l) - 1);
      valid = active && 0 <= __builtin_amdgcn_readlane(wa, l) && 0 <= __builtin_amdgcn_readlane(wb, l);
      if (first && active) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            creg[x][r] = (i0 + 16 * x < m && j0 + r < n) ? (double)cblk[i0 + 16 * x + (long)(j0 + r) * m] : 0.0;
          }
        }
        __builtin_amdgcn_s_waitcnt(0xF70); /* once per run, so that no recombination waits for the DMA of the next entry */
      }
    }
    if (valid) {
      /* exponents from LDS: rows of A, columns of B */
      const int* const lex = (const int*)(cur + 2 * NS * SPL);
      exi[0] = lex[i0];
      exi[1] = lex[i0 + 16];
      exj = *(const i4_t*)(lex + SB + j0);
      i4_t fb[NS];
#pragma unroll
      for (int q = 0; q < NS; ++q) fb[q] = *(const i4_t*)(cur + (NS + q) * SPL + (16 * wj + frow) * SB + fpos);
#pragma unroll
      for (int L = 0; L < 2 * NS - 1; ++L) acc[L][0] = acc[L][1] = i4_t{0};
#pragma unroll
      for (int p = 0; p < NS; ++p) {
        i4_t fa[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) fa[x] = *(const i4_t*)(cur + p * SPL + (32 * wi + 16 * x + frow) * SB + fpos);
#pragma unroll
        for (int q = 0; q < NS; ++q) {
          if (p + q <= cutoff) {
#pragma unroll
            for (int x = 0; x < 2; ++x) acc[p + q][x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[q], fa[x], acc[p + q][x], 0, 0, 0);
          }
        }
      }
    }
    if (0 == late) recombine();
  }
  if (0 != late) recombine();
  __builtin_amdgcn_s_waitcnt(0); /* no DMA in flight at the end */
}

/* NS slices with the level cutoff compiled in for the triangle (NS - 1) and all pairs (2 NS - 2) */
template <typename T, int NS>
void ozs_launch_ns(dim3 grid, hipStream_t st, const int* stack, int S, const int* info, const int8_t* pa,
  const int* ea, const int8_t* pb, const int* eb, int cutoff, int m, int n, int k, int na, int nb, T* c) {
  if (NS - 1 == cutoff) {
    ozs_stack<T, NS, NS - 1><<<grid, 512, 0, st>>>(stack, S, info, pa, ea, pb, eb, cutoff, m, n, k, na, nb, c);
  }
  else if (2 * (NS - 1) == cutoff) {
    ozs_stack<T, NS, 2 * (NS - 1)><<<grid, 512, 0, st>>>(stack, S, info, pa, ea, pb, eb, cutoff, m, n, k, na, nb, c);
  }
  else {
    ozs_stack<T, NS, -1><<<grid, 512, 0, st>>>(stack, S, info, pa, ea, pb, eb, cutoff, m, n, k, na, nb, c);
  }
}

template <typename T>
int ozs_launch_stack(int s, dim3 grid, hipStream_t st, const int* stack, int S, const int* info,
  const int8_t* pa, const int* ea, const int8_t* pb, const int* eb, int cutoff, int m, int n, int k, int na, int nb, T* c) {
  switch (s) {
    case 1: ozs_launch_ns<T, 1>(grid, st, stack, S, info, pa, ea, pb, eb, cutoff, m, n, k, na, nb, c); break;
    case 2: ozs_launch_ns<T, 2>(grid, st, stack, S, info, pa, ea, pb, eb, cutoff, m, n, k, na, nb, c); break;
    case 3: ozs_launch_ns<T, 3>(grid, st, stack, S, info, pa, ea, pb, eb, cutoff, m, n, k, na, nb, c); break;
    case 4: ozs_launch_ns<T, 4>(grid, st, stack, S, info, pa, ea, pb, eb, cutoff, m, n, k, na, nb, c); break;
    case 5: ozs_launch_ns<T, 5>(grid, st, stack, S, info, pa, ea, pb, eb, cutoff, m, n, k, na, nb, c); break;
    case 6: ozs_launch_ns<T, 6>(grid, st, stack, S, info, pa, ea, pb, eb, cutoff, m, n, k, na, nb, c); break;
    case 7: ozs_launch_ns<T, 7>(grid, st, stack, S, info, pa, ea, pb, eb, cutoff, m, n, k, na, nb, c); break;
    case 8: ozs_launch_ns<T, 8>(grid, st, stack, S, info, pa, ea, pb, eb, cutoff, m, n, k, na, nb, c); break;
    default: return LXS_ELIMIT;
  }
  return 0;
}

} /* namespace */

/*
 * A pool of na blocks m x k (column-major), B pool of nb blocks in the kernel layout (k x n row-major);
 * planes_a: na * s * 4 KB, planes_b: nb * s * 4 KB, ea: na * 64 ints, eb: nb * 64 ints, info: 1 int (all
 * device memory).
 */
extern "C" int lxs_ozs_process(int dtype, const int* stack, int S, int m, int n, int k, const void* a, int na,
  const void* b, int nb, void* c, int s, int cutoff, signed char* planes_a, int* ea, signed char* planes_b, int* eb,
  int* info, int ncus, void* hip_stream) {
  const hipStream_t st = (hipStream_t)hip_stream;
  if (1 > m || SB < m || 1 > n || SB < n || 1 > k || SB < k || 1 > s || 8 < s || 0 > cutoff || 2 * (s - 1) < cutoff) {
    return LXS_ELIMIT;
  }
  if (0 >= S) return 0;
  if (0 >= na || 0 >= nb) return LXS_ELIMIT;
  /* as many work-groups as are resident (LDS: one per CU above 4 slices, else two), each with one share of the stack */
  const int wgs = (4 < s ? 1 : 2) * (0 < ncus ? ncus : 256);
  const dim3 grid((unsigned int)(S < wgs ? S : wgs));
  const unsigned int cgrid = (unsigned int)((S + 255) / 256 < 256 ? (S + 255) / 256 : 256);
  int result = 0;
  if (3 == dtype) { /* A rows: (r, kk) at r + kk m; B columns: (j, kk) at j + kk n */
    ozs_slice<double><<<na, 256, 0, st>>>((const double*)a, (long)m * k, 1, m, m, k, s, (int8_t*)planes_a, ea);
    ozs_slice<double><<<nb, 256, 0, st>>>((const double*)b, (long)k * n, 1, n, n, k, s, (int8_t*)planes_b, eb);
    ozs_clear<<<1, 1, 0, st>>>(info);
    ozs_check<<<cgrid, 256, 0, st>>>(stack, S, info);
    result = ozs_launch_stack<double>(s, grid, st, stack, S, info, (const int8_t*)planes_a, ea, (const int8_t*)planes_b,
      eb, cutoff, m, n, k, na, nb, (double*)c);
  }
  else if (1 == dtype) {
    ozs_slice<float><<<na, 256, 0, st>>>((const float*)a, (long)m * k, 1, m, m, k, s, (int8_t*)planes_a, ea);
    ozs_slice<float><<<nb, 256, 0, st>>>((const float*)b, (long)k * n, 1, n, n, k, s, (int8_t*)planes_b, eb);
    ozs_clear<<<1, 1, 0, st>>>(info);
    ozs_check<<<cgrid, 256, 0, st>>>(stack, S, info);
    result = ozs_launch_stack<float>(s, grid, st, stack, S, info, (const int8_t*)planes_a, ea, (const int8_t*)planes_b,
      eb, cutoff, m, n, k, na, nb, (float*)c);
  }
  else {
    return LXS_ENOVARIANT;
  }
  return (0 != result ? result : (int)hipGetLastError());
}
