// FP64 GEMM on gfx950 matrix cores: C += A*B, one launch for any number of GEMMs.
//
// Replaces the reference's gemm_kernel (src/phpc_gemm.cu:6-57). The reference gives
// each thread one output and walks the K dimension in T-wide shared-memory phases.
// Here a workgroup owns a BM x BN macro tile, its waves own 16x16 MFMA sub-tiles
// (v_mfma_f64_16x16x4f64), operands are staged through LDS in slabs of k, and the
// workgroups share a flat list of tiles covering any number of GEMMs (one launch for all
// SUMMA ranks, or for a batch of unrelated GEMMs). Two kernels: rm_kernel (gemm_rm.h) copies
// slabs HBM -> LDS directly and runs everything the planner picks; f64_gemm_kernel stages them
// through registers and is kept as the fixed configurations that it is compared with.
//
// Arithmetic. v_mfma_f64_16x16x4f64 computes, per output, the FMA chain
// d = fma(a3,b3, fma(a2,b2, fma(a1,b1, fma(a0,b0,c)))) in k order (measured on the
// device against 10^6 random cases). With the accumulator started at zero for each
// panel, k visited in ascending order and the panel sum added to C afterwards, every
// output equals the reference kernel's `c = 0; c += a*b (contracted to FMA); C += c`
// (src/phpc_gemm.cu:32,50-51,55). Zero padding of partial slabs adds fma(0,0,c) = c,
// as the reference's own tile padding does (:38-46).
//
// Layout. Row-major, arbitrary leading dimensions. The register-staged kernel's LDS holds A
// transposed (At[k][m]) and B as is (Bs[k][n]) so each MFMA operand fetch is 16 consecutive
// doubles per lane group; the direct kernel's layout is described with it.
#include "gemm_rm.h"
#include "phpc_internal.h"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <type_traits>
#include <vector>

typedef double d4 __attribute__((ext_vector_type(4)));

namespace {

using GemmBatch = RmBatch<GemmDesc>;
typedef double __attribute__((address_space(1))) gdouble;

template <int VEC>
struct Chunk;
template <>
struct Chunk<1> {
  double x;
};
template <>
struct Chunk<2> {
  double x, y;
};

template <int VEC>
__device__ __forceinline__ Chunk<VEC> buf_load(rsrc_t r, uint32_t off) {
  Chunk<VEC> c;
  if constexpr (VEC == 2) {
    const double2 v = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    c.x = v.x;
    c.y = v.y;
  } else {
    c.x = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
  }
  return c;
}

template <int BM, int BN, int WM, int WN, int BK, bool MP, int VEC>
struct F64Gemm {
  static constexpr int NT = WM * WN * 64;
  static constexpr int WTM = BM / WM;
  static constexpr int WTN = BN / WN;
  static constexpr int TM = WTM / 16;
  static constexpr int TN = WTN / 16;
  static constexpr int APITCH = BM + 4;
  static constexpr int BPITCH = BN + 4;
  static constexpr int STAGE = BK * APITCH + BK * BPITCH;  // doubles per LDS stage
  // global->register chunks per thread (VEC doubles per chunk)
  static constexpr int CA = BM * BK / VEC / NT;
  static constexpr int CB = BN * BK / VEC / NT;
  static_assert(CA * VEC * NT == BM * BK, "A slab must split evenly over threads");
  static_assert(CB * VEC * NT == BN * BK, "B slab must split evenly over threads");
  static_assert(TM >= 1 && TN >= 1, "wave tile must hold at least one 16x16 block");
};

template <int BM, int BN, int WM, int WN, int BK, bool MP, int VEC>
// two waves per SIMD at least: a 4-wave workgroup then fits twice on a CU
__global__ __launch_bounds__(WM *WN * 64) __attribute__((amdgpu_waves_per_eu(2))) void f64_gemm_kernel(
    GemmBatch batch) {
  using K = F64Gemm<BM, BN, WM, WN, BK, MP, VEC>;
  __shared__ double lds[2 * K::STAGE];

  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int g = lane >> 4;   // k index inside an MFMA (0..3)
  const int li = lane & 15;  // row (A) / column (B) inside a 16-block
  const int wm = wave / WN;
  const int wn = wave % WN;

  const int G = gridDim.x;
  const int bid = blockIdx.x;
  // XCD-aware order: workgroup bid runs on XCD bid % 8; give each XCD a contiguous
  // run of the tiles processed in the same round so neighbouring tiles share its L2.
  const bool xcd_remap = batch.xcd_remap && (G % 8) == 0;
  const int slot = uni(xcd_remap ? (bid % 8) * (G / 8) + bid / 8 : bid);

  for (int round = 0;; ++round) {
    const int t = round * G + slot;
    if (t >= batch.total_tiles) break;
    const GemmDesc d = uniform_desc(batch, uni(t));
    const int lt = t - d.tile_start;
    const int tiles_n = d.tiles_n;
    const int tiles_m = (d.m + BM - 1) / BM;
    // group-M swizzle
    const int gm = batch.group_m;
    const int grp = lt / (gm * tiles_n);
    const int first_m = grp * gm;
    const int gsz = min(tiles_m - first_m, gm);
    const int in_grp = lt - grp * gm * tiles_n;
    const int tm_idx = first_m + in_grp % gsz;
    const int tn_idx = in_grp / gsz;
    const int row0 = tm_idx * BM;
    const int col0 = tn_idx * BN;
    const int m_rem = uni(d.m - row0);
    const int n_rem = uni(d.n - col0);
    const long lda = uni(d.lda), ldb = uni(d.ldb), ldc = uni(d.ldc);
    const double *Ag = uni(d.A) + (long)row0 * lda;
    const double *Bg = uni(d.B) + col0;
    gdouble *Cg = (gdouble *)(uni(d.C) + (long)row0 * ldc + col0);
    const rsrc_t rA = make_rsrc(Ag, (long)min(m_rem, BM) * lda * 8);
    const int Kdim = uni(d.k);
    const int dpanel = uni(d.panel);
    const int w = dpanel > 0 && dpanel < Kdim ? dpanel : Kdim;

    d4 acc[K::TM][K::TN];
    d4 creg[MP ? K::TM : 1][MP ? K::TN : 1];
#pragma unroll
    for (int i = 0; i < K::TM; ++i)
#pragma unroll
      for (int j = 0; j < K::TN; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};

    if constexpr (MP) {
#pragma unroll
      for (int i = 0; i < K::TM; ++i)
#pragma unroll
        for (int j = 0; j < K::TN; ++j) {
          const int cc = wn * K::WTN + j * 16 + li;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int rr = wm * K::WTM + i * 16 + 4 * r + g;
            creg[i][j][r] = (rr < m_rem && cc < n_rem) ? Cg[(long)rr * ldc + cc] : 0.0;
          }
        }
    }

    Chunk<VEC> ra[K::CA];
    Chunk<VEC> rb[K::CB];

    auto load_slab = [&](int kb, int ke) {
      const int krem = ke - kb;
#pragma unroll
      for (int i = 0; i < K::CA; ++i) {
        const int q = tid + i * K::NT;
        const int row = q / (BK / VEC);
        const int kc = (q % (BK / VEC)) * VEC;
        const uint32_t off = (row < m_rem && kc < krem) ? (uint32_t)(((long)row * lda + kb + kc) * 8) : kOOB;
        ra[i] = buf_load<VEC>(rA, off);
      }
      const rsrc_t rB = make_rsrc(Bg + (long)kb * ldb, (long)krem * ldb * 8);
#pragma unroll
      for (int i = 0; i < K::CB; ++i) {
        const int q = tid + i * K::NT;
        const int kr = q / (BN / VEC);
        const int cc = (q % (BN / VEC)) * VEC;
        const uint32_t off = (kr < krem && cc < n_rem) ? (uint32_t)(((long)kr * ldb + cc) * 8) : kOOB;
        rb[i] = buf_load<VEC>(rB, off);
      }
    };

    auto store_slab = [&](int buf) {
      double *At = lds + buf * K::STAGE;
      double *Bs = At + BK * K::APITCH;
#pragma unroll
      for (int i = 0; i < K::CA; ++i) {
        const int q = tid + i * K::NT;
        const int row = q / (BK / VEC);
        const int kc = (q % (BK / VEC)) * VEC;
        At[kc * K::APITCH + row] = ra[i].x;
        if constexpr (VEC == 2) At[(kc + 1) * K::APITCH + row] = ra[i].y;
      }
#pragma unroll
      for (int i = 0; i < K::CB; ++i) {
        const int q = tid + i * K::NT;
        const int kr = q / (BN / VEC);
        const int cc = (q % (BN / VEC)) * VEC;
        if constexpr (VEC == 2) {
          *reinterpret_cast<double2 *>(&Bs[kr * K::BPITCH + cc]) = double2{rb[i].x, rb[i].y};
        } else {
          Bs[kr * K::BPITCH + cc] = rb[i].x;
        }
      }
    };

    auto mfma_step = [&](const double *At, const double *Bs, int kk) {
      double a[K::TM], b[K::TN];
#pragma unroll
      for (int i = 0; i < K::TM; ++i) a[i] = At[(kk * 4 + g) * K::APITCH + wm * K::WTM + i * 16 + li];
#pragma unroll
      for (int j = 0; j < K::TN; ++j) b[j] = Bs[(kk * 4 + g) * K::BPITCH + wn * K::WTN + j * 16 + li];
#pragma unroll
      for (int i = 0; i < K::TM; ++i)
#pragma unroll
        for (int j = 0; j < K::TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
    };

    auto compute = [&](int buf, int klen) {
      const double *At = lds + buf * K::STAGE;
      const double *Bs = At + BK * K::APITCH;
      // k beyond the slab was loaded as zero, so a partial slab adds fma(0, 0, c) = c
      // terms only (the reference kernel pads its own T-wide phases the same way)
      (void)klen;
#pragma unroll
      for (int kk = 0; kk < BK / 4; ++kk) mfma_step(At, Bs, kk);
    };

    // All waves must be done with the previous tile's last slab before the prologue
    // overwrites LDS.
    __syncthreads();
    int kb = 0;
    int pe = min(w, Kdim);
    load_slab(kb, min(kb + BK, pe));
    store_slab(0);
    __syncthreads();
    int buf = 0;
    while (true) {
      const int ke = min(kb + BK, pe);
      const bool panel_end = (ke == pe);
      const int nkb = panel_end ? pe : kb + BK;
      const int npe = panel_end ? min(pe + w, Kdim) : pe;
      const bool has_next = nkb < Kdim;
      if (has_next) load_slab(nkb, min(nkb + BK, npe));
      compute(buf, ke - kb);
      if constexpr (MP) {
        if (panel_end) {
#pragma unroll
          for (int i = 0; i < K::TM; ++i)
#pragma unroll
            for (int j = 0; j < K::TN; ++j) {
              creg[i][j] = creg[i][j] + acc[i][j];
              acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
            }
        }
      }
      if (!has_next) break;
      store_slab(buf ^ 1);
      __syncthreads();
      buf ^= 1;
      kb = nkb;
      pe = npe;
    }

    // epilogue: C = C + (panel sum) ; or store the carried C
#pragma unroll
    for (int i = 0; i < K::TM; ++i)
#pragma unroll
      for (int j = 0; j < K::TN; ++j) {
        const int cc = wn * K::WTN + j * 16 + li;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int rr = wm * K::WTM + i * 16 + 4 * r + g;
          if (rr < m_rem && cc < n_rem) {
            gdouble *pc = Cg + (long)rr * ldc + cc;
            if constexpr (MP)
              *pc = creg[i][j][r];
            else
              *pc = *pc + acc[i][j][r];
          }
        }
      }
  }
}

typedef void (*KernelFn)(GemmBatch);

// One tile configuration: kernels for [panel grouping][16-byte loads]. The row-major kernels
// take any alignment, so both slots hold the same one.
struct ConfigEntry {
  int bm, bn, threads;
  int a_rows, b_rows;   // rows of A, rows of B under one 32-bit buffer offset
  size_t lds_bytes;     // dynamic LDS
  bool panels;          // panel-grouped variants fit without spills
  KernelFn fn[2][2];
  int tail_bm, tail_bn;  // the tail's tile; 0: none
};

#define PHPC_V1(BM_, BN_, WM_, WN_, BK_, MP_, VEC_) f64_gemm_kernel<BM_, BN_, WM_, WN_, BK_, MP_, VEC_>

// a row-major configuration: head tile T, tail tile U (the same type: no tail); SP: single
// panel only
template <template <bool> class T, template <bool> class U, bool SP = false>
constexpr ConfigEntry rm_config() {
  using T0 = T<false>;
  using U0 = U<false>;
  constexpr bool same = std::is_same<T0, U0>::value;
  KernelFn one = rm_kernel<T<false>, U<false>>;
  KernelFn mp = rm_kernel<T<!SP>, U<!SP>>;
  return {T0::BM, T0::BN, T0::THREADS, std::max(T0::A_ROWS, U0::A_ROWS), std::max(T0::B_ROWS, U0::B_ROWS),
          (size_t)std::max(T0::LDS, U0::LDS), !SP, {{one, one}, {mp, mp}}, same ? 0 : U0::BM, same ? 0 : U0::BN};
}
// waves x 16-deep slabs unless named otherwise
template <bool MP> using T32 = RmTile<double, 32, 32, 2, 2, 16, 4, MP>;         // 4 waves, 32 KiB: five workgroups per CU
template <bool MP> using T32K32 = RmTile<double, 32, 32, 2, 2, 32, 4, MP>;      // 4 waves, 32-deep slabs
template <bool MP> using T64x32 = RmTile<double, 64, 32, 2, 2, 16, 5, MP>;      // 4 waves
template <bool MP> using T64 = RmTile<double, 64, 64, 2, 2, 16, 4, MP>;         // 4 waves, 64 KiB: two workgroups per CU
template <bool MP> using T64W8 = RmTile<double, 64, 64, 2, 4, 16, 4, MP>;       // 8 waves
template <bool MP> using T64W16 = RmTile<double, 64, 64, 4, 4, 32, 4, MP>;      // 16 waves, 32-deep slabs
template <bool MP> using T128x64 = RmTile<double, 128, 64, 4, 2, 16, 3, MP>;    // 8 waves
template <bool MP> using T128W8 = RmTile<double, 128, 128, 2, 4, 16, 4, MP>;    // 8 waves
template <bool MP> using T128K32 = RmTile<double, 128, 128, 4, 4, 32, 2, MP>;   // 16 waves, two 32-deep stages
template <bool MP> using T128 = RmTile<double, 128, 128, 4, 4, 16, 4, MP>;      // 16 waves
template <bool MP> using T192 = RmTile<double, 192, 128, 4, 2, 16, 4, MP>;      // 8 waves, all of LDS
template <bool MP> using T256W8 = RmTile<double, 256, 128, 4, 2, 16, 3, MP>;    // 8 waves
template <bool MP> using T256 = RmTile<double, 256, 128, 4, 4, 16, 3, MP>;      // 16 waves

// a register-staged configuration
#define V1_CONFIG(BM_, BN_, WM_, WN_, BK_)                                                                     \
  {BM_, BN_, WM_ *WN_ * 64, BM_, BK_, 0, true,                                                                 \
   {{PHPC_V1(BM_, BN_, WM_, WN_, BK_, false, 1), PHPC_V1(BM_, BN_, WM_, WN_, BK_, false, 2)},                  \
    {PHPC_V1(BM_, BN_, WM_, WN_, BK_, true, 1), PHPC_V1(BM_, BN_, WM_, WN_, BK_, true, 2)}}, 0, 0}
#define V1_CONFIG_SP(BM_, BN_, WM_, WN_, BK_)                                                                  \
  {BM_, BN_, WM_ *WN_ * 64, BM_, BK_, 0, false,                                                                \
   {{PHPC_V1(BM_, BN_, WM_, WN_, BK_, false, 1), PHPC_V1(BM_, BN_, WM_, WN_, BK_, false, 2)},                  \
    {PHPC_V1(BM_, BN_, WM_, WN_, BK_, false, 1), PHPC_V1(BM_, BN_, WM_, WN_, BK_, false, 2)}}, 0, 0}

constexpr int kSmall = 13, kMid = 5, kBig = 11, kBigPanels = 16, kOne = 10;  // the planner's
const ConfigEntry kConfigs[] = {
    V1_CONFIG(128, 128, 2, 4, 16),             // 0: register-staged, 8 waves (wave tile 64x32)
    V1_CONFIG(128, 128, 2, 4, 32),             // 1: register-staged, 8 waves, 32-deep slabs
    V1_CONFIG(64, 64, 2, 2, 16),               // 2: register-staged, 4 waves (wave tile 32x32)
    rm_config<T128W8, T128W8>(),               // 3
    rm_config<T64W8, T64W8, true>(),           // 4: single panel only
    rm_config<T64, T32K32>(),                  // 5: the planner's for middle sizes
    V1_CONFIG_SP(256, 128, 4, 2, 16),          // 6: register-staged, 8 waves (wave tile 64x64); single panel only
    rm_config<T256W8, T256W8, true>(),         // 7: single panel only
    V1_CONFIG_SP(128, 128, 2, 2, 16),          // 8: register-staged, 4 waves (wave tile 64x64); single panel only
    rm_config<T64x32, T64x32, true>(),         // 9: single panel only
    rm_config<T64W16, T64W16, true>(),         // 10: the planner's for about one 64x64 tile per CU; single panel only
    rm_config<T256, T64W16, true>(),           // 11: the planner's for large single-panel work; single panel only
    rm_config<T128x64, T128x64>(),             // 12
    rm_config<T32, T32>(),                     // 13: the planner's for small work
    rm_config<T128, T128>(),                   // 14
    rm_config<T128K32, T128K32>(),             // 15
    rm_config<T192, T64W8>(),                  // 16: the planner's for large panel-grouped work
};
constexpr int kNumConfigs = sizeof(kConfigs) / sizeof(kConfigs[0]);

std::mutex g_mu;
bool g_occ_ready = false;
int g_occ[kNumConfigs][2][2];
void *g_desc_dev = nullptr;
size_t g_desc_cap = 0;
void *g_desc_pinned = nullptr;
size_t g_pinned_cap = 0;
std::mutex g_desc_mu;  // guards the descriptor buffers below (never held with g_mu)
hipEvent_t g_desc_done = nullptr;  // recorded after the last launch that read g_desc_dev

void init_kernels_locked() {
  if (g_occ_ready) return;
  for (int c = 0; c < kNumConfigs; ++c)
    for (int a = 0; a < 2; ++a)
      for (int b = 0; b < 2; ++b) {
        const void *fn = reinterpret_cast<const void *>(kConfigs[c].fn[a][b]);
        const size_t lds = kConfigs[c].lds_bytes;
        if (lds > 0) (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, kConfigs[c].threads, lds) != hipSuccess || n < 1)
          n = 1;
        g_occ[c][a][b] = n;
      }
  g_occ_ready = true;
}

int occupancy(int cfg, int mp, int vec2) {
  std::lock_guard<std::mutex> lk(g_mu);
  init_kernels_locked();
  return g_occ[cfg][mp][vec2];
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
bool has_panels(const GemmDesc &d) { return d.panel > 0 && d.panel < d.k; }

// the planner's configurations for large work, replaceable through phpc_set_tuning
int g_big_config = kBigPanels;  // panel-grouped, on device-resident lists
int g_big_single = kBig;        // single-panel, on device-resident lists
int g_big_single_host = kBig;
int g_big_config_host = kBigPanels;
int g_group_m = 8;
int g_xcd_remap = 1;

}  // namespace

int phpc_f64_num_configs() { return kNumConfigs; }

F64Config phpc_f64_config(int id) {
  F64Config c{};
  if (id < 0 || id >= kNumConfigs) return c;
  c.id = id;
  c.bm = kConfigs[id].bm;
  c.bn = kConfigs[id].bn;
  c.threads = kConfigs[id].threads;
  c.wg_per_cu = occupancy(id, 0, 1);
  return c;
}

namespace {

// Planner: by how many tiles the work gives the CUs. Measured on MI355X, with the neighbouring
// choices:
//   up to one 64x64 tile per CU: 32x32 tiles (512^3: 8.6 us against 20.4 on 64x64, N = 256:
//     6.2 against 12.7), whose workgroups share a CU five at a time; but more than three quarters
//     of a tile per CU and k >= 900, those in 16 waves on 32-deep slabs, which hide each other's
//     barriers where no second workgroup does (0.76, 0.88 and 1.0 a CU: k = 3000 92, 92 and 94 us
//     against 98, 100 and 103 on 32x32; k = 1300 45.7, 46.2 and 46.5 against 48.1, 48.4 and 49.6; k =
//     400 21.5, 20.8 and 21.2 against 19.9, 19.2 and 19.4; 0.70, k = 3000: 92 against 79);
//   then 64x64 tiles in 4 waves with a 32x32 tail (1.06 a CU, k = 3000: 120 us, 128 on 32x32 alone;
//     2048^3: 68 TFLOP/s against 54); with panels from one a CU (1024^3 in panels of 256: 46 us
//     against 54);
//   from two 256x128 tiles per CU on, those (4096^3: 73.2 against 68; 16384^3: 74.8 against 65
//     on 64x64);
//   with panels, from six 192x128 tiles per CU on, those: the largest whose waves have room for
//     accumulators and the carried C (16384^3 in panels of 256 122.9 ms against 127.8 on 128x128 in
//     16 waves and 126.4 on 64x64; 6000^3, 5.9 a CU, 6.26 against 6.47 and 6.28; 5000^3, 4.2 a CU,
//     3.81 against 3.83 and 3.69);
//   lists with panels take them from four 128x128 tiles per CU on. Alone, 64x64 tiles are faster
//     up to some ten of 192x128 a CU, but a plan's launches meet others on the GPU, where tiles
//     that load less of L2 per output lose less (ranks of N = 4000, 4800, 7000, 8000 and 10000, 2.7 to
//     17 a CU, three plans in turn: 1.92, 3.28, 10.7, 14.5, 29.5 ms a launch against 2.09, 3.45,
//     11.3, 16.9 and 34.4 on 64x64; alone 2.05, 3.50, 10.9, 14.7 and 29.5 against 1.94, 3.19, 10.2, 14.9
//     and 30.1).
int config_for(const GemmDesc *descs, int ndesc, bool device_list) {
  long t64 = 0, t128 = 0, t192 = 0, t256 = 0;
  int k = 0;
  bool mp = false;
  for (int i = 0; i < ndesc; ++i) {
    t64 += rm_tiles(descs[i], 64, 64);
    t128 += rm_tiles(descs[i], 128, 128);
    t192 += rm_tiles(descs[i], 192, 128);
    t256 += rm_tiles(descs[i], 256, 128);
    k = std::max(k, descs[i].k);
    mp |= has_panels(descs[i]);
  }
  const long cus = phpc_device().cus;
  if (mp && (device_list ? t128 >= 4 * cus : t192 >= 6 * cus))
    // key 0 may hold a configuration without panel-grouped variants
    return !device_list ? g_big_config_host : kConfigs[g_big_config].panels ? g_big_config : kBigPanels;
  if (!mp && t256 >= 2 * cus) return device_list ? g_big_single : g_big_single_host;
  if (t64 > cus || (mp && t64 == cus)) return kMid;
  return !mp && 4 * t64 > 3 * cus && k >= 900 ? kOne : kSmall;
}

}  // namespace

int phpc_f64_prepare(const GemmDesc *descs, int ndesc, int config_id, bool device_list, F64Work *w) {
  w->descs.clear();
  w->total = w->tail_start = 0;
  // drop empty GEMMs; k == 0 leaves C unchanged (C += 0 adds +0.0 only to tiles we skip)
  for (int i = 0; i < ndesc; ++i) {
    const GemmDesc &d = descs[i];
    if (d.m < 0 || d.n < 0 || d.k < 0) return phpc_set_error(PHPC_ERR_ARG, "negative GEMM size");
    if (d.m > 0 && d.n > 0 && d.k > 0) w->descs.push_back(d);
  }
  if (config_id < 0) config_id = config_for(w->descs.data(), (int)w->descs.size(), device_list);
  if (config_id >= kNumConfigs) return phpc_set_error(PHPC_ERR_ARG, "bad FP64 config id %d", config_id);
  const ConfigEntry &ce = kConfigs[config_id];
  w->config = config_id;
  w->mp = false;
  w->vec2 = true;
  if (ce.lds_bytes) rm_split_rows(w->descs, ce.a_rows);
  for (const GemmDesc &d : w->descs) {
    w->mp |= has_panels(d);
    if ((long)ce.a_rows * d.lda * 8 >= 0x7fffffffL || (long)ce.b_rows * d.ldb * 8 >= 0x7fffffffL)
      return phpc_set_error(PHPC_ERR_ARG, "leading dimension too large (lda=%ld, ldb=%ld)", d.lda, d.ldb);
    // the register-staged kernels' 16-byte loads need 16-byte aligned rows and even k / n
    // boundaries
    const bool a_ok = aligned16(d.A) && d.lda % 2 == 0 && d.k % 2 == 0 && (!has_panels(d) || d.panel % 2 == 0);
    if (!a_ok || !aligned16(d.B) || d.ldb % 2 || d.n % 2) w->vec2 = false;
  }
  if (w->mp && !ce.panels)
    return phpc_set_error(PHPC_ERR_ARG, "FP64 config %d does not support panel grouping", config_id);
  std::vector<GemmDesc> tail;
  if (ce.tail_bm) rm_split_tail(w->descs, ce.bm, ce.bn, phpc_device().cus, tail);
  long t = 0;
  bool fits = rm_number(w->descs, ce.bm, ce.bn, &t);
  w->tail_start = (int)t;
  fits = fits && rm_number(tail, ce.tail_bm, ce.tail_bn, &t);
  if (!fits) return phpc_set_error(PHPC_ERR_ARG, "too many tiles");
  w->total = (int)t;
  w->descs.insert(w->descs.end(), tail.begin(), tail.end());
  w->list.clear();
  if (w->descs.size() > 2) w->list = rm_list(w->descs, w->total);
  return PHPC_OK;
}

int phpc_f64_launch(const F64Work &w, const void *list_dev, int grid, hipStream_t stream) {
  if (w.total <= 0) return PHPC_OK;
  const ConfigEntry &ce = kConfigs[w.config];
  GemmBatch b{};
  b.descs = static_cast<const GemmDesc *>(list_dev);
  b.ndesc = (int)w.descs.size();
  b.total_tiles = w.total;
  b.group_m = g_group_m;
  b.xcd_remap = g_xcd_remap;
  b.window = rm_window(!w.list.empty(), w.total, phpc_device().cus);
  b.tail_start = w.tail_start;
  b.d0 = w.descs[0];
  if (b.ndesc == 2) b.d1 = w.descs[1];
  // the row-major kernels leave it to the dispatcher to hand out tiles, so that a CU whose
  // tiles end early takes the next one; the register-staged ones walk a persistent grid
  if (grid <= 0) grid = ce.lds_bytes ? 0 : occupancy(w.config, w.mp, w.vec2) * phpc_device().cus;
  const int G = rm_grid(grid, w.total, ce.threads);
  {
    std::lock_guard<std::mutex> lk(g_mu);
    init_kernels_locked();
  }
  const int kt = phpc_ktime_begin(stream);
  hipLaunchKernelGGL(ce.fn[w.mp][w.vec2], dim3(G), dim3(ce.threads), ce.lds_bytes, stream, b);
  phpc_ktime_end(kt, stream);
  PHPC_HIP(hipGetLastError());
  return PHPC_OK;
}

int phpc_f64_grouped(const GemmDesc *descs, int ndesc, int grid, int config_id, hipStream_t stream) {
  F64Work w;
  if (int rc = phpc_f64_prepare(descs, ndesc, config_id, false, &w)) return rc;
  if (w.list.empty()) return phpc_f64_launch(w, nullptr, grid, stream);
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capture) != hipSuccess) (void)hipGetLastError();
  if (capture == hipStreamCaptureStatusActive) {
    // A replay would read what the buffer below holds by then: as many GEMMs a launch as it carries.
    const std::vector<GemmDesc> all = w.descs;
    for (size_t i = 0, n; i < all.size(); i += n) {
      n = std::min<size_t>(2, all.size() - i);
      if (int rc = phpc_f64_prepare(&all[i], (int)n, w.config, false, &w)) return rc;
      if (!w.list.empty()) {  // two and their tails
        n = 1;
        if (int rc = phpc_f64_prepare(&all[i], 1, w.config, false, &w)) return rc;
      }
      if (int rc = phpc_f64_launch(w, nullptr, grid, stream)) return rc;
    }
    return PHPC_OK;
  }
  // More GEMMs than travel with the launch: their list goes through one process-wide device
  // buffer. Callers on other streams may still have a launch queued that reads it, so the
  // buffer is rewritten only after the previous user's launch has finished (g_desc_done).
  std::lock_guard<std::mutex> lk(g_desc_mu);
  const size_t bytes = w.list.size();
  if (g_desc_done) PHPC_HIP(hipEventSynchronize(g_desc_done));
  if (bytes > g_desc_cap) {
    if (g_desc_dev) PHPC_HIP(hipFree(g_desc_dev));
    g_desc_dev = nullptr;
    g_desc_cap = 0;
    const size_t cap = std::max(bytes, (size_t)64 * sizeof(GemmDesc));
    PHPC_HIP(hipMalloc(&g_desc_dev, cap));
    g_desc_cap = cap;
  }
  if (bytes > g_pinned_cap) {
    if (g_desc_pinned) PHPC_HIP(hipHostFree(g_desc_pinned));
    g_desc_pinned = nullptr;
    g_pinned_cap = 0;
    const size_t cap = std::max(bytes, (size_t)64 * sizeof(GemmDesc));
    PHPC_HIP(hipHostMalloc(&g_desc_pinned, cap, hipHostMallocDefault));
    g_pinned_cap = cap;
  }
  if (!g_desc_done) PHPC_HIP(hipEventCreateWithFlags(&g_desc_done, hipEventDisableTiming));
  memcpy(g_desc_pinned, w.list.data(), bytes);
  PHPC_HIP(hipMemcpyAsync(g_desc_dev, g_desc_pinned, bytes, hipMemcpyHostToDevice, stream));
  const int rc = phpc_f64_launch(w, g_desc_dev, grid, stream);
  PHPC_HIP(hipEventRecord(g_desc_done, stream));
  return rc;
}

// Tuning knobs for the autotuner: 0 = config for large panel-grouped problems on device
// descriptors (one without panel-grouped variants leaves the default), 1 = tile-row swizzle
// width, 2 = XCD-contiguous tile order on/off, 3 = config for large single-panel problems on
// device descriptors, 4 = the same through host descriptors, 5 = large panel-grouped problems
// through host descriptors.
extern "C" int phpc_set_tuning(int key, int value) {
  switch (key) {
    case 0:
    case 3:
      if (value < 0 || value >= kNumConfigs) return phpc_set_error(PHPC_ERR_ARG, "config %d out of range", value);
      (key == 0 ? g_big_config : g_big_single) = value;
      break;
    case 1:
      if (value < 1 || value > 64) return phpc_set_error(PHPC_ERR_ARG, "group width %d out of range", value);
      g_group_m = value;
      break;
    case 2:
      g_xcd_remap = value ? 1 : 0;
      break;
    case 4:
      if (value < 0 || value >= kNumConfigs) return phpc_set_error(PHPC_ERR_ARG, "config %d out of range", value);
      g_big_single_host = value;
      break;
    case 5:
      if (value < 0 || value >= kNumConfigs || !kConfigs[value].panels)
        return phpc_set_error(PHPC_ERR_ARG, "config %d out of range", value);
      g_big_config_host = value;
      break;
    case 6:
      phpc_f32_set_direct(value);
      break;
    case 7:
      return phpc_f32_set_plan_config(value);
    case 8:
      return phpc_f32x3_set_plan_config(value);

    default:
      return phpc_set_error(PHPC_ERR_ARG, "unknown tuning key %d", key);
  }
  return phpc_set_error(PHPC_OK, nullptr);
}

bool phpc_f64_config_panels(int id) { return id >= 0 && id < kNumConfigs && kConfigs[id].panels; }
