// FP32 grouped GEMM on gfx950 matrix cores: C += A*B for a list of independent row-major FP32
// GEMMs of any shapes, one launch. Two families: the direct kernels (gemm_rm.h,
// v_mfma_f32_16x16x4f32), and the register-staged ones below (v_mfma_f32_32x32x2f32), for tuning
// and for rows of B too far apart and rows of A too long for the direct kernels' 32-bit offsets. Both sum
// each output as one FMA chain in k order: the same bits.
//
// The register-staged kernels: a BM x BN macro tile per workgroup, 4 waves in a
// 2 x 2 arrangement, operands staged HBM -> registers (raw buffer loads, out-of-range
// lanes read zero) -> LDS (A transposed, At[k][m]; B as Bs[k][n]) in 16-deep slabs with
// double buffering, and a persistent workgroup loop over the flat tile list of all GEMMs.
// MFMA 32x32x2: lane l holds A[row l%32][k l/32] and B[k l/32][col l%32]; the 16
// accumulators of lane l are rows 8(r/4) + 4(l/32) + r%4, column l%32.
#include "gemm_rm.h"
#include "phpc_internal.h"
#include "phpc_split.h"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float __attribute__((address_space(1))) gfloat;

constexpr int BK = 16;

struct F32Batch {
  const F32Desc *descs;
  int ndesc;
  int total_tiles;
  F32Desc d0;
};

__device__ __forceinline__ F32Desc f32_desc(const F32Batch &b, int t) {
  const F32Desc *d = &b.d0;
  if (b.ndesc > 1) {
    int lo = 0, hi = b.ndesc - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (b.descs[mid].tile_start <= t)
        lo = mid;
      else
        hi = mid - 1;
    }
    d = &b.descs[lo];
  }
  F32Desc u;
  u.A = uni(d->A);
  u.B = uni(d->B);
  u.C = uni(d->C);
  u.lda = uni(d->lda);
  u.ldb = uni(d->ldb);
  u.ldc = uni(d->ldc);
  u.m = uni(d->m);
  u.n = uni(d->n);
  u.k = uni(d->k);
  u.tiles_n = uni(d->tiles_n);
  u.tile_start = uni(d->tile_start);
  return u;
}

template <int BM, int BN, int VEC>
__global__ __launch_bounds__(256) void f32_gemm_kernel(F32Batch batch) {
  constexpr int WTM = BM / 2, WTN = BN / 2;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  constexpr int APITCH = BM + 4, BPITCH = BN + 4;
  constexpr int STAGE = BK * APITCH + BK * BPITCH;
  constexpr int CA = BM * BK / VEC / 256, CB = BN * BK / VEC / 256;
  static_assert(CA * VEC * 256 == BM * BK && CB * VEC * 256 == BN * BK, "slab split");
  static_assert(TM >= 1 && TN >= 1, "wave tile");
  __shared__ float lds[2 * STAGE];

  const int tid = threadIdx.x;
  const int wave = uni(tid >> 6);
  const int lane = tid & 63;
  const int wm = wave >> 1, wn = wave & 1;
  const int G = gridDim.x, bid = blockIdx.x;
  const int slot = uni((G % 8) == 0 ? (bid % 8) * (G / 8) + bid / 8 : bid);

  for (int round = 0;; ++round) {
    const int t = round * G + slot;
    if (t >= batch.total_tiles) break;
    const F32Desc d = f32_desc(batch, uni(t));
    const int lt = t - d.tile_start;
    const int row0 = uni((lt / d.tiles_n) * BM);
    const int col0 = uni((lt % d.tiles_n) * BN);
    const int m_rem = d.m - row0, n_rem = d.n - col0;
    const long lda = d.lda, ldb = d.ldb, ldc = d.ldc;
    const float *Ag = d.A + (long)row0 * lda;
    const float *Bg = d.B + col0;
    gfloat *Cg = (gfloat *)(d.C + (long)row0 * ldc + col0);
    const rsrc_t rA = make_rsrc(Ag, (long)min(m_rem, BM) * lda * 4);

    f16v acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f16v{};

    float ra[CA][VEC], rb[CB][VEC];
    auto load = [&](int kb) {
      const int krem = d.k - kb;
#pragma unroll
      for (int i = 0; i < CA; ++i) {
        const int q = tid + i * 256;
        const int row = q / (BK / VEC), kc = (q % (BK / VEC)) * VEC;
        const uint32_t off = (row < m_rem && kc < krem) ? (uint32_t)(((long)row * lda + kb + kc) * 4) : kOOB;
        if constexpr (VEC == 4) {
          // bit-cast the whole 128-bit result (element-wise extraction from the builtin's
          // integer vector is lowered to a single-dword load)
          const f4v v = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(rA, off, 0, 0));
#pragma unroll
          for (int e = 0; e < 4; ++e) ra[i][e] = v[e];
        } else {
          ra[i][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rA, off, 0, 0));
        }
      }
      const rsrc_t rB = make_rsrc(Bg + (long)kb * ldb, (long)krem * ldb * 4);
#pragma unroll
      for (int i = 0; i < CB; ++i) {
        const int q = tid + i * 256;
        const int kr = q / (BN / VEC), cc = (q % (BN / VEC)) * VEC;
        const uint32_t off = (kr < krem && cc < n_rem) ? (uint32_t)(((long)kr * ldb + cc) * 4) : kOOB;
        if constexpr (VEC == 4) {
          const f4v v = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(rB, off, 0, 0));
#pragma unroll
          for (int e = 0; e < 4; ++e) rb[i][e] = v[e];
        } else {
          rb[i][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rB, off, 0, 0));
        }
      }
    };
    auto store = [&](int buf) {
      float *At = lds + buf * STAGE;
      float *Bs = At + BK * APITCH;
#pragma unroll
      for (int i = 0; i < CA; ++i) {
        const int q = tid + i * 256;
        const int row = q / (BK / VEC), kc = (q % (BK / VEC)) * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) At[(kc + e) * APITCH + row] = ra[i][e];
      }
#pragma unroll
      for (int i = 0; i < CB; ++i) {
        const int q = tid + i * 256;
        const int kr = q / (BN / VEC), cc = (q % (BN / VEC)) * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) Bs[kr * BPITCH + cc + e] = rb[i][e];
      }
    };

    __syncthreads();
    const int nslab = (d.k + BK - 1) / BK;
    load(0);
    store(0);
    __syncthreads();
    for (int sidx = 0; sidx < nslab; ++sidx) {
      const int buf = sidx & 1;
      if (sidx + 1 < nslab) load((sidx + 1) * BK);
      const float *At = lds + buf * STAGE;
      const float *Bs = At + BK * APITCH;
#pragma unroll
      for (int kk = 0; kk < BK / 2; ++kk) {
        const int k = kk * 2 + (lane >> 5);
        float a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = At[k * APITCH + wm * WTM + i * 32 + (lane & 31)];
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = Bs[k * BPITCH + wn * WTN + j * 32 + (lane & 31)];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
      }
      if (sidx + 1 < nslab) {
        store(buf ^ 1);
        __syncthreads();
      }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int cc = wn * WTN + j * 32 + (lane & 31);
        if (cc >= n_rem) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int rr = wm * WTM + i * 32 + 8 * (r / 4) + 4 * (lane >> 5) + (r % 4);
          if (rr < m_rem) {
            gfloat *pc = Cg + (long)rr * ldc + cc;
            *pc = *pc + acc[i][j][r];
          }
        }
      }
  }
}


// ---------------------------------------------------------------------------
// FP32-accurate GEMM from three BF16 slices (v_mfma_f32_32x32x16_bf16)
// ---------------------------------------------------------------------------
// Every FP32 operand is cut exactly into x = hi + mid + lo, each a BF16 value: hi is x
// rounded to nearest BF16, mid the rounded remainder, lo the rest (|mid| <= 2^-8|x|,
// |lo| <= 2^-16|x|; with round-to-nearest the remainder after two slices has at most 8
// significant bits, so lo is exact for finite inputs whose slices stay normal). The six
// products with slice indices summing to at most 2 (hi.hi, hi.mid, mid.hi, hi.lo,
// mid.mid, lo.hi) run on the BF16 matrix cores, hi.hi into one FP32 accumulator, the five
// small ones into a second, both added to C in 64 bits at the end; the dropped
// mid.lo, lo.mid and lo.lo terms are below 2^-23 |a||b|. The result carries the error
// of an FP32 dot product: |C - exact| <= ((k + 2) 2^-24 + 2^-23) (|C0| + |A||B|).
//
// Operands are loaded as FP32 from HBM (raw buffer loads, zero outside the matrix),
// split in registers and stored to LDS as three BF16 planes with k contiguous: A as
// [plane][row][k], B transposed as [plane][col][k], so each MFMA operand is one 16-byte
// LDS read (lane l: row / column l % 32, k = 8 (l / 32) .. + 7 of the 16-deep step).
// The next slab's FP32 values are loaded into registers while the current one computes.
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));
typedef unsigned short us8v __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t bf16_rne(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ float bf16_val(uint32_t h) { return __uint_as_float(h << 16); }

// For products too small for the slice planes of gemm_bf3.hip, and where these cannot be had (a
// stream being captured, no memory): the same products in the same order, so the same sums.
// Bound by the cut in registers and the barriers of a slab: 1500^3 87 us, 57 on planes; 8192 x 64 x 8192 144 us, C alone 112 at a copy's rate. Tiles of 128x128 in
// 8 waves (in 4 the two accumulators spill: 4096 x 128 x 4096 81 us against 52). waves_per_eu(2)
// keeps the accumulators where the MFMAs take them.
template <int BM, int BN, int WN, int VEC>
__global__ __launch_bounds__(128 * WN) __attribute__((amdgpu_waves_per_eu(2))) void f32x3_gemm_kernel(F32Batch batch) {
  constexpr int NT = 128 * WN;  // 2 x WN waves
  constexpr int BK = 32;
  constexpr int KP = BK + 8;  // bf16 per LDS row (80 bytes: 16-byte aligned, staggered banks)
  constexpr int WTM = BM / 2, WTN = BN / WN;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  constexpr int AE = BM * BK / NT;  // A floats per thread
  constexpr int BE = BN * BK / NT;  // B floats per thread
  static_assert(BM == BN && AE % 8 == 0 && TM >= 1 && TN >= 1, "thread mapping");
  __shared__ __attribute__((aligned(16))) unsigned short lds[3 * BM * KP + 3 * BN * KP];
  unsigned short *Al = lds;
  unsigned short *Bl = lds + 3 * BM * KP;

  const int tid = threadIdx.x;
  const int wave = uni(tid >> 6);
  const int lane = tid & 63;
  const int wm = wave / WN, wn = wave % WN;
  const int G = gridDim.x, bid = blockIdx.x;
  const int slot = uni((G % 8) == 0 ? (bid % 8) * (G / 8) + bid / 8 : bid);
  // AE consecutive k of one row of A, BE of one column of B per thread
  const int a_row = tid / (BK / AE), a_k = tid % (BK / AE) * AE;
  const int b_col = tid % BN, b_k = tid / BN * BE;

  for (int round = 0;; ++round) {
    const int t = round * G + slot;
    if (t >= batch.total_tiles) break;
    const F32Desc d = f32_desc(batch, uni(t));
    const int lt = t - d.tile_start;
    const int row0 = uni((lt / d.tiles_n) * BM);
    const int col0 = uni((lt % d.tiles_n) * BN);
    const int m_rem = d.m - row0, n_rem = d.n - col0;
    const long lda = d.lda, ldb = d.ldb, ldc = d.ldc;
    const float *Ag = d.A + (long)row0 * lda;
    const float *Bg = d.B + col0;
    const rsrc_t rA = make_rsrc(Ag, (long)min(m_rem, BM) * lda * 4);

    f16v big[TM][TN], small[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) big[i][j] = small[i][j] = f16v{};

    float ra[AE], rb[BE];
    auto load = [&](int kb) {
      const int krem = d.k - kb;
      if constexpr (VEC == 4) {
#pragma unroll
        for (int q = 0; q < AE / 4; ++q) {
          const int kc = a_k + 4 * q;
          const uint32_t off = (a_row < m_rem && kc < krem) ? (uint32_t)(((long)a_row * lda + kb + kc) * 4) : kOOB;
          const f4v v = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(rA, off, 0, 0));
#pragma unroll
          for (int e = 0; e < 4; ++e) ra[4 * q + e] = v[e];
        }
      } else {
#pragma unroll
        for (int e = 0; e < AE; ++e) {
          const int kc = a_k + e;
          const uint32_t off = (a_row < m_rem && kc < krem) ? (uint32_t)(((long)a_row * lda + kb + kc) * 4) : kOOB;
          ra[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rA, off, 0, 0));
        }
      }
      const rsrc_t rB = make_rsrc(Bg + (long)kb * ldb, (long)krem * ldb * 4);
#pragma unroll
      for (int e = 0; e < BE; ++e) {
        const int kr = b_k + e;
        const uint32_t off = (kr < krem && b_col < n_rem) ? (uint32_t)(((long)kr * ldb + b_col) * 4) : kOOB;
        rb[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rB, off, 0, 0));
      }
    };
    // split AE consecutive-k values into three BF16 runs at dst + plane * pstride
    auto split_store = [&](const float *x, unsigned short *dst, int pstride) {
      us8v h[AE / 8], m[AE / 8], l[AE / 8];
#pragma unroll
      for (int e = 0; e < AE; ++e) {
        const uint32_t hb = bf16_rne(x[e]);
        const float r1 = x[e] - bf16_val(hb);
        const uint32_t mb = bf16_rne(r1);
        const float r2 = r1 - bf16_val(mb);
        h[e >> 3][e & 7] = (unsigned short)hb;
        m[e >> 3][e & 7] = (unsigned short)mb;
        l[e >> 3][e & 7] = (unsigned short)bf16_rne(r2);
      }
#pragma unroll
      for (int hlf = 0; hlf < AE / 8; ++hlf) {
        *(us8v *)(dst + 8 * hlf) = h[hlf];
        *(us8v *)(dst + pstride + 8 * hlf) = m[hlf];
        *(us8v *)(dst + 2 * pstride + 8 * hlf) = l[hlf];
      }
    };

    const int nslab = (d.k + BK - 1) / BK;
    load(0);
    for (int sidx = 0; sidx < nslab; ++sidx) {
      __syncthreads();  // the previous slab's MFMA reads are done
      split_store(ra, Al + a_row * KP + a_k, BM * KP);
      split_store(rb, Bl + b_col * KP + b_k, BN * KP);
      __syncthreads();
      if (sidx + 1 < nslab) load((sidx + 1) * BK);
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk) {
        const int ko = kk * 16 + 8 * (lane >> 5);
        bf8v a[TM][3], b[TN][3];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int p = 0; p < 3; ++p)
            a[i][p] = __builtin_bit_cast(
                bf8v, *(const us8v *)(Al + p * BM * KP + (wm * WTM + i * 32 + (lane & 31)) * KP + ko));
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int p = 0; p < 3; ++p)
            b[j][p] = __builtin_bit_cast(
                bf8v, *(const us8v *)(Bl + p * BN * KP + (wn * WTN + j * 32 + (lane & 31)) * KP + ko));
        // each accumulator's order is that of the planes' kernel
        auto product = [&](f16v(&acc)[TM][TN], int p, int r) {
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][p], b[j][r], acc[i][j], 0, 0, 0);
        };
        product(small, 0, 2);
        product(small, 1, 1);
        product(small, 2, 0);
        product(big, 0, 0);
        product(small, 0, 1);
        product(small, 1, 0);
      }
    }
    const int wrow = wm * WTM, wcol = wn * WTN;
    if (wrow < m_rem && wcol < n_rem) {
      const CTile<float, f16v, TM, TN, 32, 16> ct(d.C + (long)(row0 + wrow) * ldc + col0 + wcol, ldc, m_rem - wrow,
                                                  n_rem - wcol, lane);
      ct.update([&](float c, int i, int j, int r) {
        return (float)((double)c + ((double)big[i][j][r] + (double)small[i][j][r]));
      });
    }
    __syncthreads();  // LDS is rewritten by the next tile
  }
}

typedef void (*F32Fn)(F32Batch);
struct F32Cfg {
  int bm, bn;
  F32Fn fn[2];  // [vec4]
};
const F32Cfg kF32[] = {
    {64, 64, {f32_gemm_kernel<64, 64, 1>, f32_gemm_kernel<64, 64, 4>}},
    {128, 64, {f32_gemm_kernel<128, 64, 1>, f32_gemm_kernel<128, 64, 4>}},
    {128, 128, {f32_gemm_kernel<128, 128, 1>, f32_gemm_kernel<128, 128, 4>}},
};
constexpr int kNumF32 = sizeof(kF32) / sizeof(kF32[0]);

std::mutex g_mu;
bool g_ready = false;
int g_occ[kNumF32][2];

int occ(int c, int v) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (!g_ready) {
    for (int i = 0; i < kNumF32; ++i)
      for (int j = 0; j < 2; ++j) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void *>(kF32[i].fn[j]), 256, 0) !=
                hipSuccess ||
            n < 1)
          n = 1;
        g_occ[i][j] = n;
      }
    g_ready = true;
  }
  return g_occ[c][v];
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int g_f32_direct = 1;  // FP32 products through the direct kernels
int g_f32_plan_cfg = -1;  // FP32 plans' configuration without autotuning (-1: by work)

// The direct kernels (gemm_rm.h) by tile shape: head T, tail U (the same type: no tail).
struct F32RmConfig {
  int bm, bn, threads;
  int a_rows, b_rows;  // rows of A, rows of B under one 32-bit buffer offset
  size_t lds_bytes;
  void (*fn)(RmBatch<F32Desc>);
  int tail_bm, tail_bn;  // 0: no tail
};
template <class T, class U>
constexpr F32RmConfig f32_rm_config() {
  constexpr bool same = std::is_same<T, U>::value;
  return {T::BM, T::BN, T::THREADS, std::max(T::A_ROWS, U::A_ROWS), std::max(T::B_ROWS, U::B_ROWS),
          (size_t)std::max(T::LDS, U::LDS), rm_kernel<T, U>, same ? 0 : U::BM, same ? 0 : U::BN};
}
using G32 = RmTile<float, 32, 32, 2, 2, 32, 4, false>;
using G32K64 = RmTile<float, 32, 32, 2, 2, 64, 4, false>;
using G64 = RmTile<float, 64, 64, 2, 2, 32, 4, false>;
using G64K64 = RmTile<float, 64, 64, 4, 2, 64, 4, false>;
using G64W8 = RmTile<float, 64, 64, 4, 2, 32, 4, false>;
using G128 = RmTile<float, 128, 64, 4, 2, 32, 3, false>;
// The tile shapes of the planner's rule. Measured (device time): 256^3 5.4 us on 32x32 against
// 9.5 on 64x64; 1500x1000x700 28.1 on 64x64 with the tail against 40 without it and 54.4 on the
// register-staged 64x64 tiles before; 4096^3 949 us (145 TF/s) on 128x64 with two workgroups to
// a CU, 966 on 64x64, 966 on 256x128 with one; 512 products log-uniform in [64, 4096] 9.25 ms
// on 128x64, 9.45 on 64x64, 9.9 on 256x128, 11.6 before (128x128, operands staged).
enum { kF32Small = 0, kF32Mid = 1, kF32Big = 2, kF32One = 3 };
const F32RmConfig kF32Rm[] = {
    f32_rm_config<G32, G32>(),
    f32_rm_config<G64, G32K64>(),
    f32_rm_config<G128, G64W8>(),
    f32_rm_config<G64K64, G64K64>(),
};
std::once_flag g_rm_once;

// The planes of 3 x BF16 products. Large products share one workspace, which a captured one refers
// to from then on. Smaller ones must not move it: they have four of their own, each stream keeping
// to one while there are no more than four, so that products on different streams run side by
// side. Planes of more than kWayBytes an operand go to the first, so that the others together
// stay below 3 GiB.
struct X3Workspaces {
  static constexpr int kWays = 4;
  static constexpr size_t kWayBytes = 512u << 20;
  SharedWorkspace large, way[kWays];
  SharedWorkspace &of(hipStream_t s, size_t bytes) {
    if (bytes > kWayBytes) return way[0];
    std::lock_guard<std::mutex> lk(mu);
    for (int i = 0; i < used; ++i)
      if (user[i] == s) return way[i];
    const int i = next;
    next = (next + 1) % kWays;
    used = std::max(used, i + 1);
    user[i] = s;
    return way[i];
  }

 private:
  std::mutex mu;
  hipStream_t user[kWays] = {};
  int used = 0, next = 0;
};

}  // namespace

static_assert(kF32DirectConfig == kNumF32, "the direct kernels follow the register-staged ones");

int phpc_f32_num_configs() { return kNumF32 + 1; }

void phpc_f32_config_tile(int id, int *bm, int *bn) {
  *bm = kF32[id].bm;
  *bn = kF32[id].bn;
}

// Fills tiles_n / tile_start of descs for register-staged config `id`; returns the total tile
// count.
int phpc_f32_plan_tiles(F32Desc *descs, int ndesc, int id) {
  int bm, bn;
  phpc_f32_config_tile(id, &bm, &bn);
  int start = 0;
  for (int i = 0; i < ndesc; ++i) {
    F32Desc &d = descs[i];
    d.tiles_n = (d.n + bn - 1) / bn;
    d.tile_start = start;
    start += ((d.m + bm - 1) / bm) * d.tiles_n;
  }
  return start;
}

// A load spans a_rows rows of A and b_rows of B. Rows of A that lie too far apart become products
// of one row, lda = k (rm_split_rows), so of A it is k that has to fit.
bool phpc_f32_direct_ok(const F32Desc *descs, int ndesc) {
  for (int i = 0; i < ndesc; ++i)
    for (const F32RmConfig &c : kF32Rm)
      if ((long)c.a_rows * descs[i].k * 4 >= 0x7fffffffL || (long)c.b_rows * descs[i].ldb * 4 >= 0x7fffffffL)
        return false;
  return true;
}

int phpc_f32_prepare(const F32Desc *descs, int ndesc, F32Work *w) {
  w->descs.clear();
  w->total = w->tail_start = 0;
  long t64 = 0, t128 = 0;
  int kmax = 0;
  for (int i = 0; i < ndesc; ++i) {
    if (descs[i].m <= 0 || descs[i].n <= 0 || descs[i].k <= 0) continue;
    w->descs.push_back(descs[i]);
    t64 += rm_tiles(descs[i], 64, 64);
    t128 += rm_tiles(descs[i], 128, 64);
    kmax = std::max(kmax, descs[i].k);
  }
  const long cus = phpc_device().cus;
  // 128x64 tiles from four a CU on (two rounds of the two resident ones): 3000^3, 4.4 a CU, 404
  // us against 416 on 64x64, but 2500^3, 3.1 a CU, 265 against 249. 64x64 in 4 waves above one a CU
  // (1.06 a CU, k = 1000: 27 us against 30 on 32x32). Up to one 64x64 tile a CU 32x32 tiles, which
  // leave no CU empty (256^3 5.4 us against 9.5); but more than three quarters of one and k >= 1000,
  // 64x64 in 8 waves on 64-deep slabs (0.76, 0.88 and 1.0 a CU: k = 3000 53 us each against 58, 59
  // and 60 on 32x32; k = 1500 30.8, 30.9 and 31.5 against 32.2, 33.3 and 33.5; k = 700 19.8, 19.9 and 20.2
  // against 18.0, 18.9 and 18.6; 0.70, k = 3000: 53 against 47).
  w->config = t128 >= 4 * cus                     ? kF32Big
              : t64 > cus                         ? kF32Mid
              : 4 * t64 > 3 * cus && kmax >= 1000 ? kF32One
                                                  : kF32Small;
  const F32RmConfig &c = kF32Rm[w->config];
  if (!phpc_f32_direct_ok(w->descs.data(), (int)w->descs.size()))
    return phpc_set_error(PHPC_ERR_ARG, "leading dimension too large");
  rm_split_rows(w->descs, c.a_rows);
  std::vector<F32Desc> tail;
  if (c.tail_bm) rm_split_tail(w->descs, c.bm, c.bn, cus, tail);
  long t = 0;
  bool fits = rm_number(w->descs, c.bm, c.bn, &t);
  w->tail_start = (int)t;
  fits = fits && rm_number(tail, c.tail_bm, c.tail_bn, &t);
  if (!fits) return phpc_set_error(PHPC_ERR_ARG, "too many tiles");
  w->total = (int)t;
  w->descs.insert(w->descs.end(), tail.begin(), tail.end());
  w->list.clear();
  if (w->descs.size() > 2) w->list = rm_list(w->descs, w->total);
  return PHPC_OK;
}

int phpc_f32_launch_direct(const F32Work &w, const void *list_dev, int grid, hipStream_t stream) {
  if (w.total <= 0) return PHPC_OK;
  std::call_once(g_rm_once, [] {
    for (const F32RmConfig &c : kF32Rm)
      (void)hipFuncSetAttribute(reinterpret_cast<const void *>(c.fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)c.lds_bytes);
  });
  const F32RmConfig &c = kF32Rm[w.config];
  RmBatch<F32Desc> b{};
  b.descs = static_cast<const F32Desc *>(list_dev);
  b.ndesc = (int)w.descs.size();
  b.total_tiles = w.total;
  b.group_m = 8;
  b.xcd_remap = 1;
  b.window = rm_window(!w.list.empty(), w.total, phpc_device().cus);
  b.tail_start = w.tail_start;
  b.d0 = w.descs[0];
  if (b.ndesc == 2) b.d1 = w.descs[1];
  const int G = rm_grid(grid, w.total, c.threads);
  const int kt = phpc_ktime_begin(stream);
  hipLaunchKernelGGL(c.fn, dim3(G), dim3(c.threads), c.lds_bytes, stream, b);
  phpc_ktime_end(kt, stream);
  PHPC_HIP(hipGetLastError());
  return PHPC_OK;
}

bool phpc_f32_vec4_ok(const F32Desc *descs, int ndesc) {
  for (int i = 0; i < ndesc; ++i) {
    const F32Desc &d = descs[i];
    if (!aligned16(d.A) || !aligned16(d.B) || d.lda % 4 || d.ldb % 4 || d.k % 4 || d.n % 4) return false;
  }
  return true;
}

namespace {
// The in-register 3 x BF16 kernel's tiles: configuration 0's (64x64) or 2's (128x128). A CU holds
// four workgroups of 64x64 or one of 128x128. Measured at k = 512, by tiles a CU: 64x64 24 us for
// one, 29 for two, 36 for three, 46 for four, 80 for five; 128x128 36 for one (as for fewer), 67
// for two, 100 for three. So 128x128 from more than three 64x64 tiles a CU on, where it does not
// take more than 4 / 3 of the rounds (64 x 512 x 100000, four rounds of 128x128 for two of 64x64:
// 123 us against 86; 100 x 512 x 40000, two each: 68 against 82).
int x3_tile(const std::vector<F32Desc> &descs) {
  long t64 = 0, t128 = 0;
  for (const F32Desc &d : descs) {
    t64 += rm_tiles(d, 64, 64);
    t128 += rm_tiles(d, 128, 128);
  }
  const long cus = phpc_device().cus;
  return t64 > 3 * cus && 3 * ((t128 + cus - 1) / cus) <= 4 * ((t64 + 4 * cus - 1) / (4 * cus)) ? 2 : 0;
}
}  // namespace

// 128x128 tiles in whole rounds, and what would leave their last round nearly empty in a second
// launch of its own tiles (100 x 4096 x 40000, 313 tiles of 128x128: 445 us, 380 so).
void phpc_f32x3_prepare(const F32Desc *descs, int ndesc, F32X3Work *w) {
  w->descs.assign(descs, descs + ndesc);
  w->vec4 = phpc_f32_vec4_ok(descs, ndesc);
  std::vector<F32Desc> tail;
  w->config[0] = x3_tile(w->descs);
  if (w->config[0] == 2) rm_split_tail(w->descs, 128, 128, phpc_device().cus, tail, 3);
  w->config[1] = x3_tile(tail);
  w->head = (int)w->descs.size();
  w->tiles[0] = phpc_f32_plan_tiles(w->descs.data(), w->head, w->config[0]);
  w->tiles[1] = phpc_f32_plan_tiles(tail.data(), (int)tail.size(), w->config[1]);
  w->descs.insert(w->descs.end(), tail.begin(), tail.end());
}

bool phpc_f32x3_in_register_ok(const F32Desc &d) { return 128L * d.lda * 4 < 0x7fffffffL && 32L * d.ldb * 4 < 0x7fffffffL; }

// Whether a 3 x BF16 product that could take either is faster on slice planes, which cost 16 bytes
// of traffic an element of A and B where the in-register kernel reads 4 once a tile: from k = 512
// on with more than 256 rows and columns (1000 x 512 x 1000 23 us against 24, 512 x 4096 x 2000 77
// against 141; at k = 256 18 against 16), and on narrower ones from k = 1024 on while the planes
// stay in the last-level cache (128 x 1024 x 8192 37 us against 42; 128 x 512 x 8192 28 against 25,
// 128 x 4096 x 8192 164 against 138, 32 x 4096 x 40000 590 against 275).
bool phpc_f32x3_planes_pay(const F32Desc &d) {
  return std::min(d.m, d.n) > 256 ? d.k >= 512 : d.k >= 1024 && ((long)d.m + d.n) * d.k <= 16L << 20;
}

namespace {
int x3_launch(const F32Desc *descs_dev, const F32Desc *descs_host, int ndesc, int total_tiles, int config, bool vec4,
              int grid, hipStream_t stream) {
  if (ndesc <= 0 || total_tiles <= 0) return PHPC_OK;
  for (int i = 0; i < ndesc; ++i)
    if (!phpc_f32x3_in_register_ok(descs_host[i])) return phpc_set_error(PHPC_ERR_ARG, "leading dimension too large");
  static void (*const kernels[2][2])(F32Batch) = {{f32x3_gemm_kernel<64, 64, 2, 1>, f32x3_gemm_kernel<64, 64, 2, 4>},
                                                  {f32x3_gemm_kernel<128, 128, 4, 1>, f32x3_gemm_kernel<128, 128, 4, 4>}};
  void (*fn)(F32Batch) = kernels[config == 2][vec4];
  const int threads = config == 2 ? 512 : 256;
  int occ;
  {
    static int occ_cache[2][2] = {};
    std::lock_guard<std::mutex> lk(g_mu);
    int &cached = occ_cache[config == 2][vec4];
    if (cached == 0) {
      int n = 0;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void *>(fn), threads, 0) != hipSuccess ||
          n < 1)
        n = 1;
      cached = n;
    }
    occ = cached;
  }
  F32Batch b{};
  b.descs = descs_dev;
  b.ndesc = ndesc;
  b.total_tiles = total_tiles;
  b.d0 = descs_host[0];
  int G = grid > 0 ? grid : occ * phpc_device().cus;
  if (G > total_tiles) G = total_tiles;
  if (G < 1) G = 1;
  hipLaunchKernelGGL(fn, dim3(G), dim3(threads), 0, stream, b);
  PHPC_HIP(hipGetLastError());
  return PHPC_OK;
}
}  // namespace

int phpc_f32x3_launch(const F32X3Work &w, const F32Desc *descs_dev, int grid, hipStream_t stream) {
  const int n = (int)w.descs.size();
  if (int rc = x3_launch(descs_dev, w.descs.data(), w.head, w.tiles[0], w.config[0], w.vec4, grid, stream)) return rc;
  return x3_launch(descs_dev ? descs_dev + w.head : nullptr, w.descs.data() + w.head, n - w.head, w.tiles[1], w.config[1],
                   w.vec4, grid, stream);
}

// Launch the grouped kernel over device-resident descriptors (planned for config id).
int phpc_f32_launch(const F32Desc *descs_dev, const F32Desc *descs_host, int ndesc, int total_tiles, int id, bool vec4,
                    int grid, hipStream_t stream) {
  if (ndesc <= 0 || total_tiles <= 0) return PHPC_OK;
  if (id < 0 || id >= kNumF32) return phpc_set_error(PHPC_ERR_ARG, "FP32 config %d is not register-staged", id);
  for (int i = 0; i < ndesc; ++i) {
    const F32Desc &d = descs_host[i];
    if ((long)kF32[id].bm * d.lda * 4 >= 0x7fffffffL || 16L * d.ldb * 4 >= 0x7fffffffL)
      return phpc_set_error(PHPC_ERR_ARG, "leading dimension too large");
  }
  F32Batch b{};
  b.descs = descs_dev;
  b.ndesc = ndesc;
  b.total_tiles = total_tiles;
  b.d0 = descs_host[0];
  int G = grid > 0 ? grid : occ(id, vec4) * phpc_device().cus;
  if (G > total_tiles) G = total_tiles;
  if (G < 1) G = 1;
  const int kt = phpc_ktime_begin(stream);
  hipLaunchKernelGGL(kF32[id].fn[vec4 ? 1 : 0], dim3(G), dim3(256), 0, stream, b);
  phpc_ktime_end(kt, stream);
  PHPC_HIP(hipGetLastError());
  return PHPC_OK;
}

// Single FP32 GEMM on device pointers: FP32 matrix cores or the 3 x BF16 kernel.
extern "C" int phpc_sgemm_device(const float *dA, long lda, const float *dB, long ldb, float *dC, long ldc, int m, int k,
                                 int n, int method, void *stream) {
  if (phpc_init()) return phpc_last_error();
  if (method != PHPC_SGEMM_FP32 && method != PHPC_SGEMM_BF16X3) return phpc_set_error(PHPC_ERR_ARG, "bad method");
  if (m < 0 || k < 0 || n < 0) return phpc_set_error(PHPC_ERR_ARG, "negative size");
  if ((m > 0 && k > 0 && (!dA || lda < k)) || (k > 0 && n > 0 && (!dB || ldb < n)) || (m > 0 && n > 0 && (!dC || ldc < n)))
    return phpc_set_error(PHPC_ERR_ARG, "bad pointers or leading dimensions");
  if (m == 0 || n == 0 || k == 0) return phpc_set_error(PHPC_OK, nullptr);
  F32Desc d{};
  d.A = dA;
  d.B = dB;
  d.C = dC;
  d.lda = lda;
  d.ldb = ldb;
  d.ldc = ldc;
  d.m = m;
  d.n = n;
  d.k = k;
  int rc = PHPC_OK;
  bool planes = false;
  const bool large = (long)m * n >= 2048L * 2048 && k >= 256;
  if (method == PHPC_SGEMM_BF16X3) {
    // Slice planes from one 64x64 tile per CU on, where they pay or rows lie too far apart for the
    // in-register kernel; at 512^3, 18 us against 23, the one launch that needs no workspace is the
    // simpler. A stream being captured takes a workspace (which may grow, and waits for its last
    // user) only where it always did.
    planes = large;
    if (!large && rm_tiles(d, 64, 64) >= phpc_device().cus && (phpc_f32x3_planes_pay(d) || !phpc_f32x3_in_register_ok(d)) &&
        phpc_bf3_fits(k)) {
      hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
      const hipError_t e = hipStreamIsCapturing((hipStream_t)stream, &st);
      if (e != hipSuccess) (void)hipGetLastError();
      planes = e == hipSuccess && st == hipStreamCaptureStatusNone;
    }
  }
  if (planes) {
    // slice planes cut once, then multiplied on the direct-to-LDS pipeline
    static X3Workspaces all;
    SharedWorkspace &ws =
        large ? all.large : all.of((hipStream_t)stream, std::max(phpc_bf3_plane_bytes(m, k), phpc_bf3_plane_bytes(n, k)));
    std::lock_guard<std::mutex> lk(ws.mu);
    ws.after_previous((hipStream_t)stream);
    rc = phpc_sgemm_bf16x3_planes(dA, lda, dB, ldb, dC, ldc, m, k, n, (hipStream_t)stream, &ws.ws);
    ws.mark_used((hipStream_t)stream);
    planes = large || rc != PHPC_ERR_MEM;
    if (!planes) (void)hipGetLastError();  // the allocation's, before the launch below asks for its own
  }
  if (method == PHPC_SGEMM_BF16X3 && !planes) {
    F32X3Work w;
    phpc_f32x3_prepare(&d, 1, &w);
    rc = phpc_f32x3_launch(w, nullptr, 0, (hipStream_t)stream);
  } else if (method != PHPC_SGEMM_BF16X3) {
    if (g_f32_direct && phpc_f32_direct_ok(&d, 1)) {
      F32Work w;
      rc = phpc_f32_prepare(&d, 1, &w);
      if (!rc && w.list.empty()) {
        rc = phpc_f32_launch_direct(w, nullptr, 0, (hipStream_t)stream);
      } else if (!rc) {
        // rows too far apart for one launch's offsets (rm_split_rows): one by one, without a list
        for (int r = 0; r < m && !rc; ++r) {
          F32Desc row = d;
          row.A += (long)r * lda;
          row.C += (long)r * ldc;
          row.m = 1;
          row.lda = k;
          rc = phpc_f32_prepare(&row, 1, &w);
          if (!rc) rc = phpc_f32_launch_direct(w, nullptr, 0, (hipStream_t)stream);
        }
      }
    } else {
      const long work = (long)((m + 127) / 128) * ((n + 127) / 128);
      const int cfg = work >= 2L * phpc_device().cus ? 2 : 0;
      const int tiles = phpc_f32_plan_tiles(&d, 1, cfg);
      rc = phpc_f32_launch(nullptr, &d, 1, tiles, cfg, phpc_f32_vec4_ok(&d, 1), 0, (hipStream_t)stream);
    }
  }
  return rc ? rc : phpc_set_error(PHPC_OK, nullptr);
}

void phpc_f32_set_direct(int on) { g_f32_direct = on ? 1 : 0; }

int phpc_f32_set_plan_config(int id) {
  if (id < -1 || id > kF32DirectConfig) return phpc_set_error(PHPC_ERR_ARG, "FP32 config %d out of range", id);
  g_f32_plan_cfg = id;
  return phpc_set_error(PHPC_OK, nullptr);
}

int phpc_f32_pick_plan_config(const F32Desc *descs, int ndesc) {
  if (g_f32_plan_cfg >= 0 && (g_f32_plan_cfg != kF32DirectConfig || phpc_f32_direct_ok(descs, ndesc))) return g_f32_plan_cfg;
  if (g_f32_direct && phpc_f32_direct_ok(descs, ndesc)) return kF32DirectConfig;
  long work = 0;
  for (int i = 0; i < ndesc; ++i) work += (long)((descs[i].m + 127) / 128) * ((descs[i].n + 127) / 128);
  return work < 2L * phpc_device().cus ? 0 : 2;
}
