// FP32-accurate GEMM on the BF16 matrix cores (3 x BF16), one product or a list of them.
//
// Every FP32 operand is cut exactly into x = hi + mid + lo, each a BF16 value: hi is x rounded
// to nearest BF16, mid the rounded remainder, lo the rest. The six products with slice indices
// summing to at most 2 run on the BF16 matrix cores: hi.hi into one FP32 accumulator, the five
// small ones into a second, both added to C in 64 bits at the end; the dropped ones are below
// 2^-23 |a||b|. One kernel cuts every operand into planes; one launch then multiplies. Error
// against 64 bits (2-norm, uniform inputs): 4096^3 3.75e-7 (3.74e-7 with one accumulator over
// all six), 1500^3 2.1e-7 (5.9e-7 with one in the in-register kernel before).
#include "gemm_rm.h"
#include "phpc_internal.h"
#include "phpc_split.h"

#include <algorithm>
#include <mutex>
#include <vector>

namespace {

typedef int i4v __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned int u4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));

// Planes are stored as the product kernel's MFMA operands: a block is kMI plane rows (rows of A,
// columns of B) x kFK k of one slice, 1 KiB, lane l's 16 bytes (row l % kMI, the 8 k from 8 (l /
// kMI)) at 16 l; [row block][k block][slice] in memory. A load to LDS then moves one contiguous
// KiB, and an operand read of LDS is linear in the lane: no swizzle, no bank conflicts.
constexpr int kMI = 32, kFK = 16;
constexpr int kBlock = 1024, kSlab = 3 * kBlock;

__device__ __forceinline__ uint32_t bf16_rne(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ void split3(float x, uint32_t &h, uint32_t &mi, uint32_t &lo) {
  h = bf16_rne(x);
  const float r1 = x - __uint_as_float(h << 16);
  mi = bf16_rne(r1);
  const float r2 = r1 - __uint_as_float(mi << 16);
  lo = bf16_rne(r2);
}

// ---------------------------------------------------------------------------
// the cut: bound by memory (4 bytes read, 6 written per element: 5.0 TB/s over the operands of
// 512 products, where a large copy makes 4.8). A wave takes kCutK k blocks of one row block: all
// its loads are in flight before the first cut, and every store is a contiguous KiB.
// ---------------------------------------------------------------------------
constexpr int kCutK = 4;  // k blocks per wave
struct Bf3CutArgs {
  const Bf3Cut *cuts;    // device list and the cut of every workgroup; nullptr: c0, then c1
  const int *block_cut;
  Bf3Cut c0, c1;
};

__global__ __launch_bounds__(256) void bf3_cut_kernel(Bf3CutArgs args) {
  const int b = blockIdx.x;
  const Bf3Cut c = args.cuts ? args.cuts[uni(args.block_cut[b])] : b < args.c1.block_start ? args.c0 : args.c1;
  const int lb = b - c.block_start;
  const int lane = threadIdx.x & 63;
  const int rb = uni((lb / c.tiles_k) * 4 + (int)(threadIdx.x >> 6));
  const int kb0 = uni((lb % c.tiles_k) * kCutK);
  const int nrows = c.is_b ? c.cols : c.rows, kk = c.is_b ? c.rows : c.cols;
  const int nkb = (kk + kFK - 1) / kFK;
  if (rb * kMI >= nrows) return;
  const int row = rb * kMI + lane % kMI, k0 = kb0 * kFK + lane / kMI * 8;
  float x[kCutK][8];
  const bool full = rb * kMI + kMI <= nrows && (kb0 + kCutK) * kFK <= kk;
  if (!c.is_b) {
    const float *src = c.src + (long)row * c.ld + k0;
    if (full) {
#pragma unroll
      for (int j = 0; j < kCutK; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f4u v = *reinterpret_cast<const f4u *>(src + j * kFK + 4 * h);
#pragma unroll
          for (int e = 0; e < 4; ++e) x[j][4 * h + e] = v[e];
        }
    } else {
#pragma unroll
      for (int j = 0; j < kCutK; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) x[j][e] = row < nrows && k0 + j * kFK + e < kk ? src[j * kFK + e] : 0.0f;
    }
  } else {
    const float *src = c.src + (long)k0 * c.ld + row;
    if (full) {
#pragma unroll
      for (int j = 0; j < kCutK; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) x[j][e] = src[(long)(j * kFK + e) * c.ld];
    } else {
#pragma unroll
      for (int j = 0; j < kCutK; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          x[j][e] = row < nrows && k0 + j * kFK + e < kk ? src[(long)(j * kFK + e) * c.ld] : 0.0f;
    }
  }
  char *dst = c.dst + ((long)rb * nkb + kb0) * kSlab + lane * 16;
#pragma unroll
  for (int j = 0; j < kCutK; ++j) {
    if (kb0 + j >= nkb) break;
    uint32_t s[3][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) split3(x[j][e], s[0][e], s[1][e], s[2][e]);
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      u4v v;
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = s[p][2 * q] | (s[p][2 * q + 1] << 16);
      *reinterpret_cast<u4v *>(dst + j * kSlab + p * kBlock) = v;
    }
  }
}

// ---------------------------------------------------------------------------
// The product. Bound by the matrix cores where it fills the GPU: 4096^3 at 247 TFLOP/s is 1482
// of BF16, more than a plain library product of BF16 matrices reaches on this card (1379). A
// slab (16 k of all three slices) is loaded once for six products (in three passes over k, one
// per level, each plane was loaded up to three times: 205 TFLOP/s, with LDS reads as long as
// the MFMAs: one per MFMA of 32x32x16 in a 64x64 wave tile, now a half). The loop over full
// slabs holds MFMAs, LDS reads at a constant address, loads at a constant offset plus a scalar
// one, and no vector arithmetic; a slab's operands are read behind the MFMAs of the one before.
// Three stages are enough (a slab of a 128x128 tile takes 0.4 us) and leave room for two
// workgroups of 128x128 on a CU, so that one's C passes under the other's MFMAs.
// ---------------------------------------------------------------------------
template <int BM, int BN, int WM, int WN, int STAGES_>
struct Bf3Shape {
  static constexpr int STAGES = STAGES_;
  static constexpr int NW = WM * WN;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int TM = WTM / kMI, TN = WTN / kMI;
  static constexpr int RA = BM / kMI, RB = BN / kMI;  // row blocks
  static constexpr int A_BYTES = RA * kSlab, B_BYTES = RB * kSlab;
  static constexpr int B_BASE = STAGES * A_BYTES;
  static constexpr int LDS_BYTES = STAGES * (A_BYTES + B_BYTES);
  static constexpr int NB = (RA + RB) * 3;
  static constexpr int PER = NB / NW, REST = NB % NW;  // blocks per wave; waves with one more
  static constexpr int UNROLL = STAGES % 2 ? 2 * STAGES : STAGES;
  static_assert(TM >= 1 && TN >= 1 && STAGES >= 3 && LDS_BYTES <= 160 * 1024, "shape");
};

template <int BM, int BN, int WM, int WN, int STAGES>
__device__ __forceinline__ void bf3_tile(const Bf3Desc &d, int row0, int col0) {
  using K = Bf3Shape<BM, BN, WM, WN, STAGES>;
  constexpr int TM = K::TM, TN = K::TN;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int wave = uni((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const int wm = wave / WN, wn = wave % WN;
  const int nslab = d.k;

  // block u of this wave: its source, and where it lies in stage 0
  rsrc_t src[K::PER + 1];
  int lds[K::PER + 1], lds_step[K::PER + 1];
  const int last_a = (d.m - 1) / kMI, last_b = (d.n - 1) / kMI;
#pragma unroll
  for (int u = 0; u < K::PER + 1; ++u) {
    const int b = wave + u * K::NW;
    const bool is_a = b < K::RA * 3;
    const int bb = is_a ? b : b - K::RA * 3;
    // row blocks past the matrix edge: the last one again, whose outputs are not written
    const long rb = is_a ? min(row0 / kMI + bb / 3, last_a) : min(col0 / kMI + bb / 3, last_b);
    src[u] = make_rsrc((is_a ? d.A + rb * kMI * d.lda : d.B + rb * kMI * d.ldb) + bb % 3 * kBlock, 0x7fffffffL);
    lds[u] = is_a ? bb * kBlock : K::B_BASE + bb * kBlock;
    lds_step[u] = is_a ? K::A_BYTES : K::B_BYTES;
  }
  auto issue = [&](int stage, int slab) {
#pragma unroll
    for (int u = 0; u < K::PER + 1; ++u)
      if (u < K::PER || (K::REST && wave < K::REST))
        __builtin_amdgcn_raw_ptr_buffer_load_lds(src[u], (lds_void *)(smem + lds[u] + stage * lds_step[u]), 16,
                                                 lane * 16, slab * kSlab, 0, 0);
  };
  // until at most N slabs of this wave's loads are outstanding
  auto wait_slabs = [&](auto n) {
    constexpr int N = decltype(n)::value;
    if (K::REST && wave < K::REST)
      wait_vm_c<N * (K::PER + 1)>();
    else
      wait_vm_c<N * K::PER>();
  };
  // walk the slabs: step t waits for slab t + 1, refills the stage of slab t (whose operands are
  // in registers by then) with slab t + STAGES, reads the operands of slab t + 1 and multiplies
  auto walk = [&](auto read, auto mul) {
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
      if (s < nslab) issue(s, s);
    if (nslab >= STAGES)
      wait_slabs(std::integral_constant<int, STAGES - 1>{});
    else
      wait_vm_c<0>();
    slab_barrier();
    read(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
    int t = 0;
#pragma unroll 1
    while (t < nslab) {
#pragma unroll 1
      for (; t + K::UNROLL + STAGES <= nslab; t += K::UNROLL)
        for_stages<K::UNROLL>([&](auto qc) {
          constexpr int q = decltype(qc)::value;
          wait_slabs(std::integral_constant<int, STAGES - 2>{});
          __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave has its operands
          slab_barrier();
          issue(q % STAGES, t + q + STAGES);
          read(std::integral_constant<int, (q + 1) % STAGES>{}, std::integral_constant<int, (q + 1) % 2>{});
          mul(std::integral_constant<int, q % 2>{}, std::true_type{});
        });
      for_stages<K::UNROLL>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if (t < nslab) {
          if (t + STAGES <= nslab)
            wait_slabs(std::integral_constant<int, STAGES - 2>{});
          else
            wait_vm_c<0>();
          __builtin_amdgcn_s_waitcnt(0xC07F);
          slab_barrier();
          if (t + STAGES < nslab) issue(q % STAGES, t + STAGES);
          if (t + 1 < nslab)
            read(std::integral_constant<int, (q + 1) % STAGES>{}, std::integral_constant<int, (q + 1) % 2>{});
          mul(std::integral_constant<int, q % 2>{}, std::false_type{});
          ++t;
        }
      });
    }
  };
  const int wrow = row0 + wm * K::WTM, wcol = col0 + wn * K::WTN;
  if (wrow >= d.m || wcol >= d.n) {
    // all of this wave's outputs lie past the matrix edge: it only loads its share
    walk([](auto, auto) {}, [](auto, auto) {});
    return;
  }

  f16v big[TM][TN], small[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) big[i][j] = small[i][j] = f16v{};
  i4v a[2][TM][3], b[2][TN][3];
  const int a0 = wm * TM * kSlab + lane * 16, b0 = K::B_BASE + wn * TN * kSlab + lane * 16;
  auto read = [&](auto stage, auto set) {
    constexpr int q = decltype(stage)::value, x = decltype(set)::value;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
        a[x][i][p] = *reinterpret_cast<const i4v *>(smem + a0 + (q * K::A_BYTES + i * kSlab + p * kBlock));
#pragma unroll
      for (int j = 0; j < TN; ++j)
        b[x][j][p] = *reinterpret_cast<const i4v *>(smem + b0 + (q * K::B_BYTES + j * kSlab + p * kBlock));
    }
  };
  auto product = [&](f16v(&acc)[TM][TN], const i4v(&x)[TM][3], const i4v(&y)[TN][3], int p, int r) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8v, x[i][p]),
                                                            __builtin_bit_cast(bf8v, y[j][r]), acc[i][j], 0, 0, 0);
  };
  auto mul = [&](auto set, auto steady) {
    constexpr int x = decltype(set)::value;
    product(small, a[x], b[x], 0, 2);
    product(small, a[x], b[x], 1, 1);
    product(small, a[x], b[x], 2, 0);
    product(big, a[x], b[x], 0, 0);
    product(small, a[x], b[x], 0, 1);
    product(small, a[x], b[x], 1, 0);
    if constexpr (decltype(steady)::value) {
      // the next slab's operand reads evenly between the MFMAs
      constexpr int NRD = 3 * (TM + TN), NMF = 6 * TM * TN, EACH = NMF / NRD;
      static_assert(EACH >= 1, "an MFMA for every read");
#pragma unroll
      for (int r = 0; r < NRD; ++r) {
        __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, NMF, 0);
    }
  };
  walk(read, mul);

  const CTile<float, f16v, TM, TN, kMI, 16> ct(d.C + (long)wrow * d.ldc + wcol, d.ldc, d.m - wrow, d.n - wcol, lane);
  // in 64 bits, so that the two sums and C are rounded once
  ct.update([&](float c, int i, int j, int r) {
    return (float)((double)c + ((double)big[i][j][r] + (double)small[i][j][r]));
  });
}

template <int BM_, int BN_, int WM, int WN, int STAGES>
struct Bf3Tile {
  using Desc = Bf3Desc;
  static constexpr int BM = BM_, BN = BN_, THREADS = WM * WN * 64, LDS = Bf3Shape<BM, BN, WM, WN, STAGES>::LDS_BYTES;
  static __device__ __forceinline__ void run(const Desc &d, int row0, int col0) {
    bf3_tile<BM, BN, WM, WN, STAGES>(d, row0, col0);
  }
};

struct Bf3Config {
  int bm, bn, threads;
  size_t lds;
  void (*fn)(RmBatch<Bf3Desc>);
  int tail_bm, tail_bn;
};
template <class T, class U>
constexpr Bf3Config bf3_config() {
  constexpr bool same = std::is_same<T, U>::value;
  return {T::BM, T::BN, T::THREADS, (size_t)std::max(T::LDS, U::LDS), rm_kernel<T, U>, same ? 0 : U::BM, same ? 0 : U::BN};
}
using T64 = Bf3Tile<64, 64, 2, 2, 3>;        // four workgroups per CU
using T128x64 = Bf3Tile<128, 64, 2, 2, 3>;   // two
using T128 = Bf3Tile<128, 128, 2, 2, 3>;     // two
using T256 = Bf3Tile<256, 128, 4, 2, 3>;     // one, of 8 waves
// The first kNumGroup are the plans' configurations kF32X3PlanesConfig + id.
enum { kT64 = 0, kT256 = 1, kT128 = 2, kT128x64 = 3 };
const Bf3Config kBf3[] = {
    bf3_config<T64, T64>(),
    bf3_config<T256, T256>(),
    bf3_config<T128, T64>(),
    bf3_config<T128x64, T64>(),
};
constexpr int kNumGroup = 3;
std::once_flag g_bf3_once;
int g_f32x3_plan_cfg = -1;

// bytes of an operand's planes
size_t plane_bytes(long rows, long k) { return (size_t)((rows + kMI - 1) / kMI) * ((k + kFK - 1) / kFK) * kSlab; }
// a tile's plane rows are read through 32-bit buffer offsets, k among them
bool planes_fit(long k) { return 256L * 6 * ((k + 63) / 64 * 64) < 0x7fffffffL; }

Bf3Cut make_cut(const float *src, long ld, int rows, int cols, int is_b, int block_start) {
  Bf3Cut c{};
  c.src = src;
  c.ld = ld;
  c.rows = rows;
  c.cols = cols;
  c.is_b = is_b;
  c.block_start = block_start;
  const int nkb = ((is_b ? rows : cols) + kFK - 1) / kFK;
  c.tiles_k = (nkb + kCutK - 1) / kCutK;
  return c;
}
// workgroups of a cut: four row blocks x kCutK k blocks each
long cut_blocks(const Bf3Cut &c) { return (long)c.tiles_k * (((c.is_b ? c.cols : c.rows) + 4 * kMI - 1) / (4 * kMI)); }

Bf3Desc make_desc(const F32Desc &f) {
  Bf3Desc d{};
  d.C = f.C;
  d.ldc = f.ldc;
  d.m = f.m;
  d.n = f.n;
  d.k = (f.k + kFK - 1) / kFK;
  d.lda = d.ldb = (long)d.k * (kSlab / kMI);
  return d;
}

// Tiles of one product, by how many it gives the CUs (device time of the launch, us):
//   256x128 where they fill at least 95% of their rounds: 4096^3 556 (247 TFLOP/s, 1482 of
//     BF16) against 600 on 128x128, 8192^3 4503 against 4653; but 3000^3, 82% full, 353
//     against 235;
//   128x128 with a 64x64 tail from one and a half a CU on: 3000^3 235 against 255 on 128x64;
//     2048^3, one a CU, 87 against 83;
//   128x64 with a 64x64 tail from one a CU on: 1500^3 46 against 48 on 64x64 and 59 on 128x128;
//     1250^3, 0.8 a CU, 33 against 31;
//   else 64x64: 1000^3 21 against 27 on 128x64.
int pick(const Bf3Desc &d) {
  const long cus = phpc_device().cus, t256 = rm_tiles(d, 256, 128);
  if (100 * t256 >= 95 * cus * ((t256 + cus - 1) / cus)) return kT256;
  if (2 * rm_tiles(d, 128, 128) >= 3 * cus) return kT128;
  return rm_tiles(d, 128, 64) >= cus ? kT128x64 : kT64;
}

int number(Bf3Work *w, int config) {
  w->config = config;
  const Bf3Config &c = kBf3[config];
  std::vector<Bf3Desc> tail;
  if (c.tail_bm) rm_split_tail(w->descs, c.bm, c.bn, phpc_device().cus, tail, 2);
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

int launch(const Bf3Work &w, const void *list_dev, int grid, hipStream_t s) {
  std::call_once(g_bf3_once, [] {
    for (const Bf3Config &c : kBf3)
      (void)hipFuncSetAttribute(reinterpret_cast<const void *>(c.fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)c.lds);
  });
  const Bf3Config &c = kBf3[w.config];
  RmBatch<Bf3Desc> b{};
  b.descs = static_cast<const Bf3Desc *>(list_dev);
  b.ndesc = (int)w.descs.size();
  b.total_tiles = w.total;
  b.group_m = 8;
  b.xcd_remap = 1;
  b.window = rm_window(!w.list.empty(), w.total, phpc_device().cus);
  b.tail_start = w.tail_start;
  b.d0 = w.descs[0];
  if (b.ndesc == 2) b.d1 = w.descs[1];
  const int G = rm_grid(grid, w.total, c.threads);
  const int kt = phpc_ktime_begin(s);
  hipLaunchKernelGGL(c.fn, dim3((unsigned)G), dim3(c.threads), c.lds, s, b);
  phpc_ktime_end(kt, s);
  PHPC_HIP(hipGetLastError());
  return PHPC_OK;
}

size_t align256(size_t b) { return (b + 255) / 256 * 256; }

}  // namespace

int phpc_sgemm_bf16x3_planes(const float *dA, long lda, const float *dB, long ldb, float *dC, long ldc, int m, int k,
                             int n, hipStream_t s, Workspace *ws) {
  if (!planes_fit(k)) return phpc_set_error(PHPC_ERR_ARG, "k = %d too large for the slice planes", k);
  char *A3 = (char *)ws->get(plane_bytes(m, k), 0, s);
  char *B3 = (char *)ws->get(plane_bytes(n, k), 1, s);
  if (!A3 || !B3) return phpc_set_error(PHPC_ERR_MEM, "slice plane allocation failed");
  Bf3CutArgs ca{};
  ca.c0 = make_cut(dA, lda, m, k, 0, 0);
  ca.c0.dst = A3;
  ca.c1 = make_cut(dB, ldb, k, n, 1, (int)cut_blocks(ca.c0));
  ca.c1.dst = B3;
  hipLaunchKernelGGL(bf3_cut_kernel, dim3((unsigned)(cut_blocks(ca.c0) + cut_blocks(ca.c1))), dim3(256), 0, s, ca);
  PHPC_HIP(hipGetLastError());
  F32Desc f{};
  f.C = dC;
  f.ldc = ldc;
  f.m = m;
  f.n = n;
  f.k = k;
  Bf3Work w;
  w.descs.push_back(make_desc(f));
  w.descs[0].A = A3;
  w.descs[0].B = B3;
  if (int rc = number(&w, pick(w.descs[0]))) return rc;
  return launch(w, nullptr, 0, s);
}

// ---------------------------------------------------------------------------
// Grouped plans on slice planes (declared in phpc_internal.h)
// ---------------------------------------------------------------------------
int phpc_bf3_num_configs() { return kNumGroup; }
bool phpc_bf3_fits(long k) { return planes_fit(k); }
size_t phpc_bf3_plane_bytes(long rows, long k) { return plane_bytes(rows, k); }

int phpc_f32x3_set_plan_config(int id) {
  if (id != -1 && id != 2 && (id < kF32X3PlanesConfig || id >= kF32X3PlanesConfig + kNumGroup))
    return phpc_set_error(PHPC_ERR_ARG, "3 x BF16 plan config %d out of range", id);
  g_f32x3_plan_cfg = id;
  return phpc_set_error(PHPC_OK, nullptr);
}

int phpc_f32x3_pick_plan_config(const F32Desc *descs, int ndesc) {
  if (g_f32x3_plan_cfg >= 0) return g_f32x3_plan_cfg;
  // The in-register kernel where the items give fewer 64x64 tiles than CUs (one launch instead
  // of two), and where most of the work is in items of no more than 256 rows or columns, whose
  // planes are little used (512 of 256 x 128 x 256 123 us against 174, 24 of 100 x 1024 x 8192 408
  // against 693; 100 of [64, 1024] 186 against 143, 64 of 1000 x 256 x 1000 344 against 308); else
  // planes, on 128x128 tiles with a 64x64 tail from two a CU on: 512 products log-uniform in [64,
  // 4096] 7.4 ms, 8.3 on 64x64 tiles, 7.8 on 256x128.
  long t64 = 0, t128 = 0;
  double all = 0, narrow = 0;
  bool ok = true;
  for (int i = 0; i < ndesc; ++i) {
    const F32Desc &d = descs[i];
    t64 += rm_tiles(d, 64, 64);
    t128 += rm_tiles(d, 128, 128);
    all += (double)d.m * d.n * d.k;
    if (std::min(d.m, d.n) <= 256) narrow += (double)d.m * d.n * d.k;
    ok &= phpc_f32x3_in_register_ok(d);
  }
  const long cus = phpc_device().cus;
  return t64 < cus || (ok && 2 * narrow > all) ? 2 : kF32X3PlanesConfig + (t128 >= 2 * cus ? kT128 : kT64);
}

int Bf3Planes::build(const F32Desc *descs, int ndesc, int gcfg) {
  release();
  cuts.clear();
  block_cut.clear();
  work = Bf3Work{};
  if (gcfg < 0 || gcfg >= kNumGroup) return phpc_set_error(PHPC_ERR_ARG, "slice-plane tile %d out of range", gcfg);
  size_t ws_bytes = 0;
  long blocks = 0;
  std::vector<size_t> off;  // bytes into the workspace, per cut
  // one cut per distinct operand (an A or B shared by several items is cut once)
  auto find_or_add = [&](const float *src, long ld, int rows, int cols, int is_b) {
    for (size_t j = 0; j < cuts.size(); ++j) {
      const Bf3Cut &c = cuts[j];
      if (c.src == src && c.ld == ld && c.rows == rows && c.cols == cols && c.is_b == is_b) return (int)j;
    }
    const Bf3Cut c = make_cut(src, ld, rows, cols, is_b, (int)blocks);
    block_cut.insert(block_cut.end(), cut_blocks(c), (int)cuts.size());
    blocks += cut_blocks(c);
    cuts.push_back(c);
    off.push_back(ws_bytes);
    ws_bytes += align256(is_b ? plane_bytes(cols, rows) : plane_bytes(rows, cols));
    return (int)cuts.size() - 1;
  };
  std::vector<int> ca, cb;
  for (int i = 0; i < ndesc; ++i) {
    const F32Desc &d = descs[i];
    if (d.m <= 0 || d.n <= 0 || d.k <= 0) continue;
    if (!planes_fit(d.k)) return phpc_set_error(PHPC_ERR_ARG, "k = %d too large for the slice planes", d.k);
    ca.push_back(find_or_add(d.A, d.lda, d.m, d.k, 0));
    cb.push_back(find_or_add(d.B, d.ldb, d.k, d.n, 1));
    work.descs.push_back(make_desc(d));
  }
  if (work.descs.empty()) return PHPC_OK;
  if (hipMalloc(&ws, ws_bytes) != hipSuccess) {
    ws = nullptr;
    (void)hipGetLastError();  // the caller may go on without planes
    return phpc_set_error(PHPC_ERR_MEM, "slice-plane workspace allocation failed (%zu bytes)", ws_bytes);
  }
  for (size_t j = 0; j < cuts.size(); ++j) cuts[j].dst = static_cast<char *>(ws) + off[j];
  for (size_t i = 0; i < work.descs.size(); ++i) {
    work.descs[i].A = cuts[ca[i]].dst;
    work.descs[i].B = cuts[cb[i]].dst;
  }
  if (int rc = number(&work, gcfg)) return rc;
  const size_t cuts_b = align256(cuts.size() * sizeof(Bf3Cut)), bc_b = align256(block_cut.size() * sizeof(int));
  if (hipMalloc(&list, cuts_b + bc_b + work.list.size()) != hipSuccess) {
    list = nullptr;
    (void)hipGetLastError();
    release();
    return phpc_set_error(PHPC_ERR_MEM, "slice-plane list allocation failed");
  }
  char *l = static_cast<char *>(list);
  PHPC_HIP(hipMemcpy(l, cuts.data(), cuts.size() * sizeof(Bf3Cut), hipMemcpyHostToDevice));
  PHPC_HIP(hipMemcpy(l + cuts_b, block_cut.data(), block_cut.size() * sizeof(int), hipMemcpyHostToDevice));
  if (!work.list.empty())
    PHPC_HIP(hipMemcpy(l + cuts_b + bc_b, work.list.data(), work.list.size(), hipMemcpyHostToDevice));
  return PHPC_OK;
}

int Bf3Planes::run(hipStream_t s, int grid) const {
  if (work.total <= 0) return PHPC_OK;
  const char *l = static_cast<const char *>(list);
  const size_t cuts_b = align256(cuts.size() * sizeof(Bf3Cut)), bc_b = align256(block_cut.size() * sizeof(int));
  Bf3CutArgs ca{};
  ca.cuts = reinterpret_cast<const Bf3Cut *>(l);
  ca.block_cut = reinterpret_cast<const int *>(l + cuts_b);
  hipLaunchKernelGGL(bf3_cut_kernel, dim3((unsigned)block_cut.size()), dim3(256), 0, s, ca);
  PHPC_HIP(hipGetLastError());
  return launch(work, l + cuts_b + bc_b, grid, s);
}

void Bf3Planes::release() {
  if (list) (void)hipFree(list);
  if (ws) (void)hipFree(ws);
  list = nullptr;
  ws = nullptr;
}
