// FP64 GEMM on gfx950 matrix cores: C += A*B, one launch for any number of GEMMs.
//
// Replaces the reference's gemm_kernel (src/phpc_gemm.cu:6-57). The reference gives
// each thread one output and walks the K dimension in T-wide shared-memory phases.
// Here a workgroup owns a BM x BN macro tile, its waves own 16x16 MFMA sub-tiles
// (v_mfma_f64_16x16x4f64), operands are staged through LDS in slabs of k, and the
// workgroups share a flat list of tiles covering any number of GEMMs (one launch for all
// SUMMA ranks, or for a batch of unrelated GEMMs). Two kernels: f64_rm_kernel copies slabs
// HBM -> LDS directly and runs everything the planner picks; f64_gemm_kernel stages them
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
#include "phpc_internal.h"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <type_traits>
#include <vector>

typedef double d4 __attribute__((ext_vector_type(4)));

namespace {

struct GemmBatch {
  const GemmDesc *descs;  // device array (ndesc > 2)
  int ndesc;
  int total_tiles;
  int group_m;            // tile-row swizzle width
  int xcd_remap;          // 1: contiguous tile runs per XCD
  int tail_start;         // row-major kernels: tiles from here on have the tail's shape
  GemmDesc d0, d1;        // inline copies when there are at most two (ndesc <= 2)
};

typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef double __attribute__((address_space(1))) gdouble;

// Out-of-range offset: raw buffer loads past num_records return zero, which is the
// zero padding of partial tiles (rows >= m, columns >= n, k beyond the panel).
constexpr uint32_t kOOB = 0x80000000u;

__device__ __forceinline__ rsrc_t make_rsrc(const double *base, long bytes) {
  const uint32_t nb = bytes > 0x7fffffffL ? 0x7fffffffu : (uint32_t)(bytes < 0 ? 0 : bytes);
  // 0x00020000: gfx9-family buffer descriptor word 3 (32-bit data format, raw access)
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(base), (short)0, (int)nb, 0x00020000);
}

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

// Values that are the same for every lane of the workgroup (tile descriptors), moved to
// scalar registers so that buffer descriptors built from them need no per-lane loop.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ long uni(long v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)(uint64_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
  return (long)(((uint64_t)hi << 32) | lo);
}
template <typename T>
__device__ __forceinline__ T *uni(T *p) {
  return reinterpret_cast<T *>(uni((long)reinterpret_cast<uintptr_t>(p)));
}

// Decode global tile id -> (descriptor, tile row, tile col).
__device__ __forceinline__ const GemmDesc *find_desc(const GemmBatch &b, int t) {
  if (b.ndesc <= 2) return b.ndesc == 2 && t >= b.d1.tile_start ? &b.d1 : &b.d0;
  int lo = 0, hi = b.ndesc - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (b.descs[mid].tile_start <= t)
      lo = mid;
    else
      hi = mid - 1;
  }
  return &b.descs[lo];
}

// Descriptor of tile t with every field moved to scalar registers (the tile id and
// hence the descriptor are the same for the whole workgroup).
__device__ __forceinline__ GemmDesc uniform_desc(const GemmBatch &b, int t) {
  const GemmDesc &d = *find_desc(b, t);
  GemmDesc u;
  u.A = uni(d.A);
  u.B = uni(d.B);
  u.C = uni(d.C);
  u.lda = uni(d.lda);
  u.ldb = uni(d.ldb);
  u.ldc = uni(d.ldc);
  u.m = uni(d.m);
  u.n = uni(d.n);
  u.k = uni(d.k);
  u.panel = uni(d.panel);
  u.tiles_n = uni(d.tiles_n);
  u.tile_start = uni(d.tile_start);
  return u;
}

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

typedef __attribute__((address_space(3))) void lds_void;

// s_waitcnt vmcnt(N) leaving expcnt and lgkmcnt unconstrained (gfx9 encoding: vmcnt
// bits [3:0] and [15:14], expcnt [6:4], lgkmcnt [11:8])
template <int N>
__device__ __forceinline__ void wait_vm_c() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 0xF) | (((N >> 4) & 3) << 14));
}
// Workgroup barrier of the slab rings. __syncthreads() brackets s_barrier with
// workgroup-scope fences, and the release fence makes the compiler wait for every
// outstanding vector-memory operation (vmcnt(0)) first: that drains the direct-to-LDS
// loads of the slabs still in flight and leaves a ring one slab deep whatever its number
// of stages. The rings wait for the loads they need themselves (wait_vm_c) and write no
// LDS with ordinary stores, so the barrier only has to keep each wave's LDS reads of a
// slab ahead of the loads that refill its buffer; the memory clobber keeps the compiler
// from moving memory operations across it.
__device__ __forceinline__ void slab_barrier() { asm volatile("s_barrier" ::: "memory"); }

// ---------------------------------------------------------------------------
// Row-major direct-to-LDS kernels: A and B are read where they lie, any leading dimension
// and any (8-byte) alignment. Slabs are copied HBM -> LDS by 16-byte buffer loads, which
// need 4-byte aligned addresses only: each wave instruction fills one contiguous 1 KiB LDS
// block, lane p writing bytes [16p, 16p+16), and the lane -> address map sets the layout.
//
// LDS layout of one stage, in 16-byte chunks:
//   A: BM rows x BK doubles, CPR = BK/2 chunks per row, chunk c of row r at slot
//      c ^ sw(r), sw(r) = (r * CPR / 16) mod CPR: the 32 lanes of a half-wave of an MFMA
//      operand read (16 rows, one chunk, both halves) cover all 64 banks once.
//   B: BK rows x BN doubles, chunk c of row k at slot c ^ ((k & 1) << 3), so the two
//      16-lane groups of a half-wave (rows k, k+1) use opposite bank halves.
// A slab with fewer than BK k rows (the end of a panel) takes 4-byte loads into the same
// layout, each checked against k, rows and columns, so padding is exact zeros in both
// operands. So does the last slab of a GEMM with an odd n whose B rows are not 16-byte
// aligned: there a 16-byte load of the last column would read past the last row's end.
//
// What bounds it. An FP64 MFMA holds its SIMD's vector pipe for 64 cycles, and a vector
// instruction of any kind waits for the MFMA before it to leave: one address addition per
// MFMA makes 64 cycles 99 (measured on one wave), while LDS reads, loads to LDS and scalar
// instructions issue beside it for nothing. So the loop over full slabs holds MFMAs, LDS
// reads at a lane's constant address plus an immediate, loads at a lane's constant offset
// plus a scalar one, and nothing vector: every stage of the ring has its own copy of the code.
// Operands are read ahead of their MFMAs and across the slab barrier (the barrier of slab s
// waits for slab s + 1), since in a small problem one wave per SIMD has nothing else to hide
// LDS latency with. At the full MFMA rate a CU on 256x128 tiles loads 14 GB/s, one on 32x32
// tiles 74, half of what its loads to LDS reach from L2 (150): hence large tiles where there
// are enough of them.
//
// Measured (MI355X, whole call, before -> after; before: A staged transposed by a kernel of
// its own, or the address arithmetic in the loop):
//   N = 256     16.0 -> 6.2 us          N = 1024     68 -> 41 us
//   N = 2048     277 -> 240 us          N = 4096   2.05 -> 1.88 ms (73 TFLOP/s)
//   N = 16384  123.8 -> 117.5 ms (74.8 TFLOP/s, 95% of the FP64 peak)
// ---------------------------------------------------------------------------
template <int BM, int BN, int WM, int WN, int BK_, int STAGES_>
struct F64Rm {
  static constexpr int BK = BK_;
  static constexpr int STAGES = STAGES_;
  static constexpr int NW = WM * WN;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int TM = WTM / 16, TN = WTN / 16;
  static constexpr int CPR = BK / 2, CPB = BN / 2;       // chunks per A row, per B row
  static constexpr int ARB = 64 / CPR, BRB = 64 / CPB;   // A rows, B rows per 1 KiB block
  static constexpr int A_BYTES = BM * BK * 8, B_BYTES = BK * BN * 8;  // of a stage; A's stages, then B's
  static constexpr int B_BASE = STAGES * A_BYTES;
  static constexpr int LDS_BYTES = STAGES * (A_BYTES + B_BYTES);
  static constexpr int PA = A_BYTES / 1024 / NW, PB = B_BYTES / 1024 / NW;  // 1 KiB blocks per wave
  static constexpr int PER = PA + PB;
  static constexpr int KSTEPS = BK / 4;
  static_assert(CPR == 8 || CPR == 16, "slab depth");
  static_assert(CPB >= 16 && CPB <= 64 && BM % (NW * ARB) == 0 && BK % (NW * BRB) == 0, "blocks split evenly");
  static_assert((NW * ARB) % 16 == 0 && (NW * BRB) % 2 == 0, "a wave's blocks share their swizzle");
  static_assert(TM >= 1 && TN >= 1, "wave tile");
  // Operand sets in registers: set kk % RING holds k step kk, and behind step kk's MFMAs the
  // set of step kk - 1 is refilled with step kk + RING - 1. The fewer MFMAs a k step has, the
  // further ahead its operands are read. Two stages leave no slab to read ahead from: the
  // operands of a slab are read after its own barrier.
  static constexpr bool AHEAD = STAGES >= 3;
  static constexpr int RING = TM * TN >= 4 ? 2 : TM * TN == 2 ? 4 : KSTEPS;
  static_assert(KSTEPS % RING == 0, "operand ring");
  static_assert(STAGES >= 2 && (STAGES + 1) * PER < 64 && LDS_BYTES <= 160 * 1024, "pipeline depth");
};

// wait until at most `units` * PER vector-memory operations are outstanding (units <= MAX)
template <int PER, int MAX>
__device__ __forceinline__ void wait_units(int units) {
  if constexpr (MAX == 0) {
    wait_vm_c<0>();
  } else {
    if (units >= MAX)
      wait_vm_c<MAX * PER>();
    else
      wait_units<PER, MAX - 1>(units);
  }
}

// f(integral_constant 0), ..., f(integral_constant N - 1)
template <int N, class F>
__device__ __forceinline__ void for_stages(const F &f) {
  if constexpr (N > 0) {
    for_stages<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// One BM x BN tile at (row0, col0) of GEMM d, all of them uniform.
template <int BM, int BN, int WM, int WN, int BK, int STAGES, bool MP>
__device__ __forceinline__ void f64_rm_tile(const GemmDesc &d, int row0, int col0) {
  using K = F64Rm<BM, BN, WM, WN, BK, STAGES>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x;
  const int wave = uni(tid >> 6);
  const int lane = tid & 63;
  const int g = lane >> 4;
  const int li = lane & 15;
  // waves 0, 4, 8, ... share a SIMD: the column index is rotated so that the waves of one tile
  // row or column, all that is left of a tile at the matrix edge, lie on different SIMDs
  const int wm = wave / WN;
  const int wn = (wave + (WN % 4 == 0 ? wm : wave / 4)) % WN;
  auto swz = [](int r) { return (r * K::CPR / 16) & (K::CPR - 1); };

  // LDS operand offsets of this lane (stage-relative bytes); blocks of 16 rows, and the k
  // steps of B, add constants
  int a_off[K::KSTEPS], b_off[K::TN];
#pragma unroll
  for (int kk = 0; kk < K::KSTEPS; ++kk)
    a_off[kk] = (wm * K::WTM + li) * BK * 8 + (((2 * kk + (g >> 1)) ^ swz(li)) << 4) + (g & 1) * 8;
#pragma unroll
  for (int j = 0; j < K::TN; ++j) {
    const int col = wn * K::WTN + j * 16 + li;
    b_off[j] = K::B_BASE + g * BN * 8 + (((col >> 1) ^ ((g & 1) << 3)) << 4) + (col & 1) * 8;
  }
  // this lane's row and chunk in the wave's first A block and first B block
  const int ar = wave * K::ARB + lane / K::CPR, ac = (lane % K::CPR) ^ swz(ar);
  const int br = wave * K::BRB + lane / K::CPB, bc = (lane % K::CPB) ^ ((br & 1) << 3);
  {
    const int m_rem = uni(d.m - row0);
    const int n_rem = uni(d.n - col0);
    const long lda = uni(d.lda), ldb = uni(d.ldb), ldc = uni(d.ldc);
    const double *Ag = uni(d.A) + (long)row0 * lda;
    const double *Bg = uni(d.B) + col0;
    gdouble *Cg = (gdouble *)(uni(d.C) + (long)row0 * ldc + col0);
    const int Kdim = uni(d.k);
    const int dpanel = uni(d.panel);
    const int w = MP && dpanel > 0 && dpanel < Kdim ? dpanel : Kdim;
    const int spp = (w + BK - 1) / BK;  // slabs per full panel
    const int full_panels = MP ? Kdim / w : 1;
    const int nslab = MP ? uni(full_panels * spp + (Kdim - full_panels * w + BK - 1) / BK) : spp;
    const int last_panel = MP && Kdim % w ? Kdim % w : w;
    const bool exact_last = (d.n & 1) && (((reinterpret_cast<uintptr_t>(Bg) >> 3) | ldb) & 1);

    // Every 1 KiB block is addressed from its own first row (ARB or BRB rows, uniform), so one
    // lane offset serves all of an operand's blocks. A rows past m_rem lie at or beyond
    // num_records and read zero (k rides in the scalar offset, which the range check leaves
    // out); B chunks past n_rem go out of range here.
    rsrc_t rA[K::PA];
#pragma unroll
    for (int u = 0; u < K::PA; ++u) {
      const int r0 = (wave + u * K::NW) * K::ARB;
      rA[u] = make_rsrc(Ag + (long)r0 * lda, (long)min(m_rem - r0, K::ARB) * lda * 8);
    }
    const uint32_t ga = (uint32_t)(((long)(lane / K::CPR) * lda + 2 * ac) * 8);
    const uint32_t gb = 2 * bc < n_rem ? (uint32_t)(((long)(lane / K::CPB) * ldb + 2 * bc) * 8) : kOOB;

    // the next slab to issue: its first k row, the end of its panel, its stage
    int ikb = 0, ipe = min(w, Kdim), istage = 0;
    const double *iB = Bg;
    auto rsrc_b = [&](int u) {
      return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(iB + (long)(wave + u * K::NW) * K::BRB * ldb),
                                               (short)0, 0x7fffffff, 0x00020000);
    };
    // block u of a full slab: A's, then B's
    auto load_block = [&](int u, int q) {
      if (u < K::PA)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rA[u], (lds_void *)(smem + q * K::A_BYTES + (wave + u * K::NW) * 1024), 16, ga,
                                                  ikb * 8, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rsrc_b(u - K::PA), (lds_void *)(smem + K::B_BASE + q * K::B_BYTES + (wave + (u - K::PA) * K::NW) * 1024),
            16, gb, 0, 0, 0);
    };
    auto advance = [&](int rows) {
      ikb += rows;
      iB += rows * ldb;
    };
    auto issue = [&]() {
      const int krem = min(BK, ipe - ikb);
      if (krem == BK && !(exact_last && ikb + BK >= Kdim)) {
#pragma unroll
        for (int u = 0; u < K::PER; ++u) load_block(u, istage);
      } else {
#pragma unroll
        for (int u = 0; u < K::PA; ++u)
#pragma unroll 1
          for (int v = 0; v < 4; ++v) {
            const int pos = v * 16 + (lane >> 2), r0 = (wave + u * K::NW) * K::ARB, r = pos / K::CPR;
            const int c = (pos % K::CPR) ^ swz(r0 + r);
            const uint32_t off = r0 + r < m_rem && 2 * c + ((lane >> 1) & 1) < krem
                                     ? (uint32_t)((long)r * lda * 8 + c * 16 + (lane & 3) * 4)
                                     : kOOB;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rA[u], (lds_void *)(smem + istage * K::A_BYTES + (wave + u * K::NW) * 1024 + v * 256), 4, off,
                ikb * 8, 0, 0);
          }
#pragma unroll
        for (int u = 0; u < K::PB; ++u)
#pragma unroll 1
          for (int v = 0; v < 4; ++v) {
            const int pos = v * 16 + (lane >> 2), r0 = (wave + u * K::NW) * K::BRB, r = pos / K::CPB;
            const int c = (pos % K::CPB) ^ (((r0 + r) & 1) << 3);
            const uint32_t off = r0 + r < krem && 2 * c + ((lane >> 1) & 1) < n_rem
                                     ? (uint32_t)((long)r * ldb * 8 + c * 16 + (lane & 3) * 4)
                                     : kOOB;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rsrc_b(u), (lds_void *)(smem + K::B_BASE + istage * K::B_BYTES + (wave + u * K::NW) * 1024 + v * 256), 4,
                off, 0, 0, 0);
          }
      }
      advance(krem);
      istage = istage + 1 == STAGES ? 0 : istage + 1;
      if (MP && ikb == ipe) ipe = min(ipe + w, Kdim);
    };

    // every wave must be done reading the previous tile's stages before refilling them
    slab_barrier();
    const int last_units = last_panel % BK || exact_last ? 3 : 0;  // extra loads of a last slab in 4-byte pieces
#pragma unroll 1
    for (int s0 = 0; s0 < STAGES - 1 && s0 < nslab; ++s0) issue();

    int issued = min(STAGES - 1, nslab);
    // slab t has landed once the slabs issued after it are all that is outstanding
    auto wait_slab = [&](int t) {
      const int later = issued - 1 - t;
      wait_units<K::PER, STAGES + 1>(later > 0 && issued == nslab ? later + last_units : later);
    };
    const int k16 = Kdim - (exact_last ? 1 : 0);  // a slab that ends past it takes 4-byte loads
    // walk the slabs, STAGES at a time while the slabs that they issue are full ones of one
    // panel; compute(stage, steady) is a slab's work behind its barrier
    auto walk = [&](auto compute) {
      int t = 0;  // the slab, in stage 0 at the head of this loop
#pragma unroll 1
      while (t < nslab) {
#pragma unroll 1
        while (ikb + STAGES * BK <= min(ipe, k16)) {
          for_stages<STAGES>([&](auto qc) { compute(qc, std::true_type{}); });
          t += STAGES;
          if (MP && ikb == ipe) ipe = min(ipe + w, Kdim);
        }
        istage = STAGES - 1;  // slab t + STAGES - 1's
        for_stages<STAGES>([&](auto qc) {
          if (t < nslab) {
            if (!K::AHEAD || t + 1 < nslab) wait_slab(K::AHEAD ? t + 1 : t);
            slab_barrier();
            if (issued < nslab) {
              issue();
              ++issued;
            }
            compute(qc, std::false_type{});
            ++t;
          }
        });
      }
    };
    // a full slab's turn: its successor has landed (two stages: it has itself), and every
    // wave is done with the stage that is filled next
    auto turn = [&]() {
      wait_vm_c<(K::AHEAD ? STAGES - 3 : 0) * K::PER>();
      slab_barrier();
    };
    if (wm * K::WTM >= m_rem || wn * K::WTN >= n_rem) {
      // all of this wave's rows or columns lie past the matrix edge: it only loads its share
      // of the slabs and keeps the barriers
      if constexpr (K::AHEAD) {
        wait_slab(0);
        slab_barrier();
      }
      walk([&](auto stage, auto steady) {
        if constexpr (decltype(steady)::value) {
          turn();
#pragma unroll
          for (int u = 0; u < K::PER; ++u) load_block(u, (decltype(stage)::value + STAGES - 1) % STAGES);
          advance(BK);
          ++issued;
        }
      });
      return;
    }

    // a small wave tile (and a panel kernel, which carries it) reads C first, so that its
    // latency passes under the slabs'
    constexpr bool CFIRST = MP || (K::TM * K::TN <= 4 && K::NW <= 8);
    d4 acc[K::TM][K::TN], creg[CFIRST ? K::TM : 1][CFIRST ? K::TN : 1];
#pragma unroll
    for (int i = 0; i < K::TM; ++i)
#pragma unroll
      for (int j = 0; j < K::TN; ++j) {
        acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
        if constexpr (CFIRST) {
          const int cc = wn * K::WTN + j * 16 + li;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int rr = wm * K::WTM + i * 16 + 4 * r + g;
            creg[i][j][r] = (rr < m_rem && cc < n_rem) ? Cg[(long)rr * ldc + cc] : 0.0;
          }
        }
      }

    auto read_ops = [&](int q, int kk, double(&x)[K::TM], double(&y)[K::TN]) {
#pragma unroll
      for (int i = 0; i < K::TM; ++i)
        x[i] = *reinterpret_cast<const double *>(smem + a_off[kk] + (q * K::A_BYTES + i * 16 * BK * 8));
#pragma unroll
      for (int j = 0; j < K::TN; ++j)
        y[j] = *reinterpret_cast<const double *>(smem + b_off[j] + (q * K::B_BYTES + kk * 4 * BN * 8));
    };
    auto mfmas = [&](const double(&x)[K::TM], const double(&y)[K::TN]) {
#pragma unroll
      for (int i = 0; i < K::TM; ++i)
#pragma unroll
        for (int j = 0; j < K::TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i], y[j], acc[i][j], 0, 0, 0);
    };
    double a[K::RING][K::TM], b[K::RING][K::TN];
    if constexpr (K::AHEAD) {
      wait_slab(0);
      slab_barrier();
#pragma unroll
      for (int q = 0; q < K::RING - 1; ++q) {
        read_ops(0, q, a[q], b[q]);
        __builtin_amdgcn_sched_barrier(0);  // in the order of their use
      }
    }
    int kend = min(w, Kdim), kb = 0;  // MP: the panel end that the slab works towards
    walk([&](auto stage, auto steady) {
      constexpr int Q = decltype(stage)::value;
      constexpr bool STEADY = decltype(steady)::value;
      constexpr int R = K::RING, D = R - 1;
      if constexpr (STEADY && !K::AHEAD) turn();
#pragma unroll
      for (int kk = 0; kk < K::KSTEPS; ++kk) {
        if (!K::AHEAD && kk == 0) {
#pragma unroll
          for (int q = 0; q < D; ++q) read_ops(Q, q, a[q], b[q]);
        }
        mfmas(a[kk % R], b[kk % R]);
        if constexpr (STEADY) {
          if (K::AHEAD && kk == 0) turn();
          // the loads are spread behind the k steps' MFMAs (two stages: all behind the first,
          // since the next slab waits for them)
#pragma unroll
          for (int u = 0; u < K::PER; ++u)
            if ((K::AHEAD ? u * K::KSTEPS / K::PER : 0) == kk)
              load_block(u, (Q + STAGES - 1) % STAGES);
          if (kk + 1 == K::KSTEPS) {
            advance(BK);
            ++issued;
          }
        }
        // keep the reads behind these MFMAs and ahead of the next (the scheduler would sink
        // them to their use)
        __builtin_amdgcn_sched_barrier(0);
        if (kk + D < K::KSTEPS)
          read_ops(Q, kk + D, a[(kk + D) % R], b[(kk + D) % R]);
        else if constexpr (K::AHEAD)  // past the last slab: read, not used
          read_ops((Q + 1) % STAGES, kk + D - K::KSTEPS, a[(kk + D) % R], b[(kk + D) % R]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (MP) {
        kb = min(kb + BK, kend);
        if (kb == kend) {
          kend = min(kend + w, Kdim);
#pragma unroll
          for (int i = 0; i < K::TM; ++i)
#pragma unroll
            for (int j = 0; j < K::TN; ++j) {
              creg[i][j] = creg[i][j] + acc[i][j];
              acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
            }
        }
      }
    });
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
            else if constexpr (CFIRST)
              *pc = creg[i][j][r] + acc[i][j][r];
            else
              *pc = *pc + acc[i][j][r];
          }
        }
      }
  }
}

template <int BM, int BN>
__device__ __forceinline__ void tile_origin(const GemmDesc &d, int lt, int group_m, int &row0, int &col0) {
  const int tiles_n = d.tiles_n;
  const int tiles_m = (d.m + BM - 1) / BM;
  const int grp = lt / (group_m * tiles_n);
  const int first_m = grp * group_m;
  const int gsz = min(tiles_m - first_m, group_m);
  const int in_grp = lt - grp * group_m * tiles_n;
  row0 = uni((first_m + in_grp % gsz) * BM);
  col0 = uni((in_grp / gsz) * BN);
}

// A contiguous run of the `total` tiles per XCD (workgroup bid runs on XCD bid % 8)
__device__ __forceinline__ int xcd_run(int bid, int total) {
  return (bid % 8) * (total / 8) + min(bid % 8, total % 8) + bid / 8;
}

// Tiles of shape T, and, from tile batch.tail_start on, the smaller tiles of shape U: the part
// of the work that would leave the last round of T tiles nearly empty.
template <class T, class U>
__device__ __forceinline__ void f64_rm_body(const GemmBatch &batch) {
  const int G = gridDim.x;
  const int bid = blockIdx.x;
  const int total = batch.total_tiles, head = batch.tail_start;
  int slot = bid;
  if (batch.xcd_remap) {
    if (G == total)
      slot = bid < head ? xcd_run(bid, head) : head + xcd_run(bid - head, total - head);
    else if (G % 8 == 0)
      slot = (bid % 8) * (G / 8) + bid / 8;
  }
  slot = uni(slot);
  for (int t = slot; t < total; t += G) {
    int row0, col0;
    const GemmDesc d = uniform_desc(batch, uni(t));
    if (t < head) {
      tile_origin<T::BM, T::BN>(d, t - d.tile_start, batch.group_m, row0, col0);
      T::run(d, row0, col0);
    } else {
      tile_origin<U::BM, U::BN>(d, t - d.tile_start, batch.group_m, row0, col0);
      U::run(d, row0, col0);
    }
  }
}

template <int BM_, int BN_, int WM, int WN, int BK, int STAGES, bool MP>
struct RmTile {
  using K = F64Rm<BM_, BN_, WM, WN, BK, STAGES>;
  static constexpr int BM = BM_, BN = BN_, THREADS = WM * WN * 64;
  static constexpr int LDS = K::LDS_BYTES, A_ROWS = K::ARB, B_ROWS = K::BRB;
  static __device__ __forceinline__ void run(const GemmDesc &d, int row0, int col0) {
    f64_rm_tile<BM, BN, WM, WN, BK, STAGES, MP>(d, row0, col0);
  }
};

template <class T, class U>
__global__ __launch_bounds__(T::THREADS) __attribute__((amdgpu_waves_per_eu(2))) void f64_rm_kernel(GemmBatch batch) {
  static_assert(T::THREADS == U::THREADS, "one workgroup shape");
  f64_rm_body<T, U>(batch);
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
  KernelFn one = f64_rm_kernel<T<false>, U<false>>;
  KernelFn mp = f64_rm_kernel<T<!SP>, U<!SP>>;
  return {T0::BM, T0::BN, T0::THREADS, std::max(T0::A_ROWS, U0::A_ROWS), std::max(T0::B_ROWS, U0::B_ROWS),
          (size_t)std::max(T0::LDS, U0::LDS), !SP, {{one, one}, {mp, mp}}, same ? 0 : U0::BM, same ? 0 : U0::BN};
}
// waves x 16-deep slabs unless named otherwise
template <bool MP> using T32 = RmTile<32, 32, 2, 2, 16, 4, MP>;         // 4 waves, 32 KiB: five workgroups per CU
template <bool MP> using T32K32 = RmTile<32, 32, 2, 2, 32, 4, MP>;      // 4 waves, 32-deep slabs
template <bool MP> using T64x32 = RmTile<64, 32, 2, 2, 16, 5, MP>;      // 4 waves
template <bool MP> using T64 = RmTile<64, 64, 2, 2, 16, 4, MP>;         // 4 waves, 64 KiB: two workgroups per CU
template <bool MP> using T64W8 = RmTile<64, 64, 2, 4, 16, 4, MP>;       // 8 waves
template <bool MP> using T64W16 = RmTile<64, 64, 4, 4, 32, 4, MP>;      // 16 waves, 32-deep slabs
template <bool MP> using T128x64 = RmTile<128, 64, 4, 2, 16, 3, MP>;    // 8 waves
template <bool MP> using T128W8 = RmTile<128, 128, 2, 4, 16, 4, MP>;    // 8 waves
template <bool MP> using T128K32 = RmTile<128, 128, 4, 4, 32, 2, MP>;   // 16 waves, two 32-deep stages
template <bool MP> using T128 = RmTile<128, 128, 4, 4, 16, 4, MP>;      // 16 waves
template <bool MP> using T256W8 = RmTile<256, 128, 4, 2, 16, 3, MP>;    // 8 waves
template <bool MP> using T256 = RmTile<256, 128, 4, 4, 16, 3, MP>;      // 16 waves

// a register-staged configuration
#define V1_CONFIG(BM_, BN_, WM_, WN_, BK_)                                                                     \
  {BM_, BN_, WM_ *WN_ * 64, BM_, BK_, 0, true,                                                                 \
   {{PHPC_V1(BM_, BN_, WM_, WN_, BK_, false, 1), PHPC_V1(BM_, BN_, WM_, WN_, BK_, false, 2)},                  \
    {PHPC_V1(BM_, BN_, WM_, WN_, BK_, true, 1), PHPC_V1(BM_, BN_, WM_, WN_, BK_, true, 2)}}, 0, 0}
#define V1_CONFIG_SP(BM_, BN_, WM_, WN_, BK_)                                                                  \
  {BM_, BN_, WM_ *WN_ * 64, BM_, BK_, 0, false,                                                                \
   {{PHPC_V1(BM_, BN_, WM_, WN_, BK_, false, 1), PHPC_V1(BM_, BN_, WM_, WN_, BK_, false, 2)},                  \
    {PHPC_V1(BM_, BN_, WM_, WN_, BK_, false, 1), PHPC_V1(BM_, BN_, WM_, WN_, BK_, false, 2)}}, 0, 0}

constexpr int kSmall = 13, kMid = 5, kBig = 11, kBigPanels = 16;  // the planner's
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
    rm_config<T64W16, T64W16, true>(),         // 10: single panel only
    rm_config<T256, T64W16, true>(),           // 11: the planner's for large single-panel work; single panel only
    rm_config<T128x64, T128x64>(),             // 12
    rm_config<T32, T32>(),                     // 13: the planner's for small work
    rm_config<T128, T128>(),                   // 14
    rm_config<T128K32, T128K32>(),             // 15
    rm_config<T128, T64W16>(),                 // 16: the planner's for large panel-grouped work
};
constexpr int kNumConfigs = sizeof(kConfigs) / sizeof(kConfigs[0]);

std::mutex g_mu;
bool g_occ_ready = false;
int g_occ[kNumConfigs][2][2];
GemmDesc *g_desc_dev = nullptr;
size_t g_desc_cap = 0;
GemmDesc *g_desc_pinned = nullptr;
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
long tiles_of(const GemmDesc &d, int bm, int bn) { return (long)((d.m + bm - 1) / bm) * ((d.n + bn - 1) / bn); }

// the planner's configurations, replaceable through phpc_set_tuning; -1: the planner's own
// choice (config_for)
int g_big_config = -1;       // large panel-grouped work on device-resident lists
int g_big_single = -1;       // large single-panel work on device-resident lists
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

// Planner: by how many tiles the work gives the CUs. Measured on MI355X in TFLOP/s, with the
// neighbouring choices:
//   fewer 64x64 tiles than CUs: 32x32 tiles (512^3: 8.6 us against 20.4 on 64x64, N = 256:
//     6.2 against 12.7), whose workgroups share a CU five at a time;
//   then 64x64 tiles with a 32x32 tail (2048^3: 68 TFLOP/s against 54 on 32x32 alone);
//   from two 256x128 tiles per CU on, those (4096^3: 73.2 against 68; 16384^3: 74.8 against 65
//     on 64x64), or, with panels, 128x128 tiles, whose waves have room for the carried C.
int config_for(const GemmDesc *descs, int ndesc, bool device_list) {
  long t64 = 0, t128 = 0, t256 = 0;
  bool mp = false;
  for (int i = 0; i < ndesc; ++i) {
    t64 += tiles_of(descs[i], 64, 64);
    t128 += tiles_of(descs[i], 128, 128);
    t256 += tiles_of(descs[i], 256, 128);
    mp |= has_panels(descs[i]);
  }
  const long cus = phpc_device().cus;
  if (mp && t128 >= 4 * cus) return device_list && g_big_config >= 0 ? g_big_config : g_big_config_host;
  if (!mp && t256 >= 2 * cus) return device_list && g_big_single >= 0 ? g_big_single : g_big_single_host;
  return t64 >= cus ? kMid : kSmall;
}

// Split `live` (tiles planned for head tiles of ce) so that the head fills whole rounds of the
// CUs and the rest runs on the smaller tail tiles: a last round of head tiles that is nearly
// empty costs as much as a full one (1777 x 1999 x 1235: 560 tiles of 64x64 on 256 CUs take
// three rounds, 187 us; 500 of them and the rest as 32x32 take 2.25). Every output's
// arithmetic is its own, so where the line runs does not change a result. The cut takes rows
// or columns of tiles, whichever step is finer, off the last GEMMs.
void split_tail(std::vector<GemmDesc> &live, const ConfigEntry &ce, std::vector<GemmDesc> &tail) {
  const long cus = phpc_device().cus;
  long total = 0;
  for (const GemmDesc &d : live) total += tiles_of(d, ce.bm, ce.bn);
  const long rounds = total / cus, rest = total % cus;
  if (rounds == 0 || rest == 0 || 5 * rest > 4 * cus) return;
  long excess = rest;
  for (int i = (int)live.size() - 1; i >= 0 && excess > 0; --i) {
    GemmDesc &d = live[i];
    const long tm = (d.m + ce.bm - 1) / ce.bm, tn = (d.n + ce.bn - 1) / ce.bn;
    GemmDesc t = d;
    if (tn <= tm) {  // whole rows of tn tiles
      const long cut = std::min(tm, (excess + tn - 1) / tn), keep = (tm - cut) * ce.bm;
      t.A += keep * t.lda;
      t.C += keep * t.ldc;
      t.m -= (int)keep;
      d.m = (int)keep;
      excess -= cut * tn;
    } else {
      const long cut = std::min(tn, (excess + tm - 1) / tm), keep = (tn - cut) * ce.bn;
      t.B += keep;
      t.C += keep;
      t.n -= (int)keep;
      d.n = (int)keep;
      excess -= cut * tm;
    }
    tail.insert(tail.begin(), t);
    if (d.m == 0 || d.n == 0) live.erase(live.begin() + i);
  }
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
  if (ce.tail_bm) split_tail(w->descs, ce, tail);
  long t = 0;
  auto number = [&t](std::vector<GemmDesc> &v, int bm, int bn) {
    for (GemmDesc &d : v) {
      d.tiles_n = (d.n + bn - 1) / bn;
      d.tile_start = (int)t;
      t += tiles_of(d, bm, bn);
    }
  };
  number(w->descs, ce.bm, ce.bn);
  w->tail_start = (int)t;
  number(tail, ce.tail_bm, ce.tail_bn);
  if (t > 0x7fffffffL) return phpc_set_error(PHPC_ERR_ARG, "too many tiles");
  w->total = (int)t;
  w->descs.insert(w->descs.end(), tail.begin(), tail.end());
  return PHPC_OK;
}

int phpc_f64_launch(const F64Work &w, const GemmDesc *descs_dev, int grid, hipStream_t stream) {
  if (w.total <= 0) return PHPC_OK;
  const ConfigEntry &ce = kConfigs[w.config];
  GemmBatch b{};
  b.descs = descs_dev;
  b.ndesc = (int)w.descs.size();
  b.total_tiles = w.total;
  b.group_m = g_group_m;
  b.xcd_remap = g_xcd_remap;
  b.tail_start = w.tail_start;
  b.d0 = w.descs[0];
  if (b.ndesc == 2) b.d1 = w.descs[1];
  int G = grid;
  if (G <= 0) {
    // the row-major kernels leave it to the dispatcher to hand out tiles, so that a CU whose
    // tiles end early takes the next one; the register-staged ones walk a persistent grid
    G = ce.lds_bytes ? w.total : occupancy(w.config, w.mp, w.vec2) * phpc_device().cus;
    if (G > w.total) G = w.total;
  }
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
  if (w.descs.size() <= 2) return phpc_f64_launch(w, nullptr, grid, stream);
  // More GEMMs than travel with the launch: descriptors go through one process-wide device
  // buffer. Callers on other streams may still have a launch queued that reads it, so the
  // buffer is rewritten only after the previous user's launch has finished (g_desc_done).
  std::lock_guard<std::mutex> lk(g_desc_mu);
  const size_t bytes = w.descs.size() * sizeof(GemmDesc);
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
  memcpy(g_desc_pinned, w.descs.data(), bytes);
  PHPC_HIP(hipMemcpyAsync(g_desc_dev, g_desc_pinned, bytes, hipMemcpyHostToDevice, stream));
  const int rc = phpc_f64_launch(w, g_desc_dev, grid, stream);
  PHPC_HIP(hipEventRecord(g_desc_done, stream));
  return rc;
}

// Tuning knobs for the autotuner: 0 = config for large panel-grouped problems on device
// descriptors, 1 = tile-row swizzle width, 2 = XCD-contiguous tile order on/off, 3 = config
// for large single-panel problems on device descriptors, 4 = the same through host
// descriptors, 5 = large panel-grouped problems through host descriptors.
extern "C" int phpc_set_tuning(int key, int value) {
  switch (key) {
    case 0:
    case 3:
      if (value < 0 || value >= 10) return phpc_set_error(PHPC_ERR_ARG, "config %d out of range", value);
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
      phpc_f32_set_transposed_a(value);
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
