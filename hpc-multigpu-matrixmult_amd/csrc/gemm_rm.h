// Row-major GEMM tiles on gfx950 matrix cores, FP64 and FP32, shared by the FP64 and FP32
// sources: C += A*B for any number of GEMMs in one launch.
#pragma once

#include "phpc_internal.h"
#include "rm_edges.h"

#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

namespace {

// A launch over the tiles of several GEMMs, numbered through (Desc::tile_start).
template <class Desc>
struct RmBatch {
  const Desc *descs;      // device list (ndesc > 2): the descriptors, then their index
  int ndesc;
  int total_tiles;
  int group_m;            // tile-row swizzle width
  int xcd_remap;          // 1: contiguous tile runs per XCD
  int window;             // tiles over which the XCDs' runs extend
  int tail_start;         // tiles from here on have the tail's shape
  Desc d0, d1;            // inline copies when there are at most two (ndesc <= 2)
};

typedef __amdgpu_buffer_rsrc_t rsrc_t;

// Out-of-range offset: raw buffer loads past num_records return zero, which is the
// zero padding of partial tiles (rows >= m, columns >= n, k beyond the panel).
constexpr uint32_t kOOB = 0x80000000u;

__device__ __forceinline__ rsrc_t make_rsrc(const void *base, long bytes) {
  const uint32_t nb = bytes > 0x7fffffffL ? 0x7fffffffu : (uint32_t)(bytes < 0 ? 0 : bytes);
  // 0x00020000: gfx9-family buffer descriptor word 3 (32-bit data format, raw access)
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)nb, 0x00020000);
}

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

// Index of a device list: entry c is the descriptor that holds tile c * kIndexTiles, so the
// search for a tile's descriptor is a load and a step or two, not a chain of log2(ndesc) loads
// at the head of every tile (512 FP32 GEMMs: 9.4 -> 9.2 ms, those with k < 256 13% faster).
constexpr int kIndexTiles = 64;
inline size_t rm_index_entries(int total_tiles) { return (size_t)total_tiles / kIndexTiles + 2; }

// Lists are read through the constant address space: nothing writes them while a launch reads
// them, and scalar loads then serve the whole wave.
template <class T>
__device__ __forceinline__ T list_load(const T *p, int i) {
  return ((const __attribute__((address_space(4))) T *)(uintptr_t)p)[i];
}

// The descriptor that holds tile t
template <class Desc>
__device__ __forceinline__ int find_desc(const RmBatch<Desc> &b, int t) {
  const int *index = reinterpret_cast<const int *>(b.descs + b.ndesc);
  int lo = uni(list_load(index, t / kIndexTiles)), hi = uni(list_load(index, t / kIndexTiles + 1));
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (uni(list_load(&b.descs[mid].tile_start, 0)) <= t)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// Descriptor of tile t with every field moved to scalar registers (the tile id and
// hence the descriptor are the same for the whole workgroup).
template <class Desc>
__device__ __forceinline__ Desc uniform_desc(const RmBatch<Desc> &b, int t) {
  if (b.ndesc <= 2) return b.ndesc == 2 && t >= b.d1.tile_start ? b.d1 : b.d0;
  const Desc *d = b.descs + find_desc(b, t);
  Desc u;
  u.A = uni(list_load(&d->A, 0));
  u.B = uni(list_load(&d->B, 0));
  u.C = uni(list_load(&d->C, 0));
  u.lda = uni(list_load(&d->lda, 0));
  u.ldb = uni(list_load(&d->ldb, 0));
  u.ldc = uni(list_load(&d->ldc, 0));
  u.m = uni(list_load(&d->m, 0));
  u.n = uni(list_load(&d->n, 0));
  u.k = uni(list_load(&d->k, 0));
  if constexpr (std::is_same<Desc, GemmDesc>::value) u.panel = uni(list_load(&d->panel, 0));
  u.tiles_n = uni(list_load(&d->tiles_n, 0));
  u.tile_start = uni(list_load(&d->tile_start, 0));
  return u;
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

// C at a wave's tile: TM x TN MFMA blocks of MI x MI outputs, NR registers a lane each. Blocks
// are read ahead and written, by buffer accesses whose lanes past the matrix edge are out
// of range, so that nothing branches and several blocks' loads are in flight: element by
// element (load, wait, add, store), 64 memory latencies in a row ended a 256x128 tile (FP64
// 7187^3 in SUMMA steps 11.29 ms, 10.96 now).
// Where a tile's rows span 2 GiB or more, lanes check and use full addresses.
template <class E, class Acc, int TM, int TN, int MI, int NR>
struct CTile {
  typedef E __attribute__((address_space(1))) global_t;
  static constexpr int SZ = sizeof(E);
  static constexpr int kAhead = NR * SZ > 32 ? 2 : 128 / (NR * SZ);  // blocks in flight, 32 registers
  rsrc_t rs;
  global_t *C;
  long ldc;
  int m_rem, n_rem, lrow, lcol;
  bool near;
  uint32_t off[TN];
  // C: the tile's first output; m_rem x n_rem outputs are the matrix's
  __device__ __forceinline__ CTile(E *c, long ldc_, int m_rem_, int n_rem_, int lane)
      : C((global_t *)c), ldc(ldc_), m_rem(m_rem_), n_rem(n_rem_) {
    lrow = MI == 32 ? 4 * (lane >> 5) : SZ == 8 ? lane >> 4 : 4 * (lane >> 4);
    lcol = lane % MI;
    near = (long)TM * MI * ldc * SZ < 0x7fffffffL;
    rs = make_rsrc(c, 0x7fffffffL);
#pragma unroll
    for (int j = 0; j < TN; ++j)
      off[j] = lcol + j * MI < n_rem ? (uint32_t)(((long)lrow * ldc + lcol + j * MI) * SZ) : kOOB;
  }
  // row of register r of block row i: a part of its own and the lane's
  static __device__ __forceinline__ constexpr int row(int i, int r) {
    return i * MI + (MI == 32 ? 8 * (r / 4) + r % 4 : SZ == 8 ? 4 * r : r);
  }
  __device__ __forceinline__ bool inside(int i, int j, int r, int lrow) const {
    return row(i, r) + lrow < m_rem && lcol + j * MI < n_rem;
  }
  __device__ __forceinline__ global_t *at(int i, int j, int r, int lrow) const {
    return C + (long)(row(i, r) + lrow) * ldc + lcol + j * MI;
  }
  template <bool NEAR>
  __device__ __forceinline__ Acc load(int i, int j) const {
    Acc c;
    int lrow = this->lrow;
    asm volatile("" : "+v"(lrow));  // its row tests are made again for the stores, not kept
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if constexpr (NEAR) {
        const uint32_t o = row(i, r) + lrow < m_rem ? off[j] : kOOB;
        const int so = (int)(row(i, r) * ldc * SZ);
        if constexpr (SZ == 8)
          c[r] = __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b64(rs, o, so, 0));
        else
          c[r] = __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b32(rs, o, so, 0));
      } else {
        c[r] = inside(i, j, r, lrow) ? *at(i, j, r, lrow) : E(0);
      }
    }
    return c;
  }
  template <bool NEAR>
  __device__ __forceinline__ void store(int i, int j, const Acc &v) const {
    int lrow = this->lrow;
    asm volatile("" : "+v"(lrow));
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if constexpr (NEAR) {
        typedef uint32_t __attribute__((ext_vector_type(2))) u2v;
        const uint32_t o = row(i, r) + lrow < m_rem ? off[j] : kOOB;
        const int so = (int)(row(i, r) * ldc * SZ);
        if constexpr (SZ == 8)
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2v, (E)v[r]), rs, o, so, 0);
        else
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, (E)v[r]), rs, o, so, 0);
      } else if (inside(i, j, r, lrow)) {
        *at(i, j, r, lrow) = v[r];
      }
    }
  }
  __device__ __forceinline__ void load_all(Acc (&c)[TM][TN]) const {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) c[i][j] = near ? load<true>(i, j) : load<false>(i, j);
  }
  __device__ __forceinline__ void store_all(const Acc (&c)[TM][TN]) const {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if (near)
          store<true>(i, j, c[i][j]);
        else
          store<false>(i, j, c[i][j]);
      }
  }
  // C = f(C, i, j, r)
  template <class F>
  __device__ __forceinline__ void update(const F &f) const {
    if (near)
      walk<true>(f);
    else
      walk<false>(f);
  }
  template <bool NEAR, class F>
  __device__ __forceinline__ void walk(const F &f) const {
    constexpr int N = TM * TN, D = N < kAhead ? N : kAhead;
    Acc c[D];
#pragma unroll
    for (int q = 0; q < D; ++q) c[q] = load<NEAR>(q / TN, q % TN);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < N; ++q) {
      Acc v;
#pragma unroll
      for (int r = 0; r < NR; ++r) v[r] = f(c[q % D][r], q / TN, q % TN, r);
      if (q + D < N) c[q % D] = load<NEAR>((q + D) / TN, (q + D) % TN);
      store<NEAR>(q / TN, q % TN, v);
      __builtin_amdgcn_sched_barrier(0);  // no more of C in registers at once
    }
  }
};

// What differs between the element types. Both products keep a lane's operands at A[row l %
// 16][k l / 16] and B[k l / 16][column l % 16] and add four k to each output as an FMA chain in
// k order (checked on the device against 10^6 chains of each type, infinities, NaNs, signed
// zeros and subnormals among them), so the order of k alone fixes a result's bits.
template <class E>
struct RmElem;
template <>
struct RmElem<double> {
  typedef double acc_t __attribute__((ext_vector_type(4)));
  static constexpr int CYCLES = 64;  // of a SIMD per MFMA
  static __device__ __forceinline__ acc_t mfma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // B slot rotation of k row k (chunks per row cpb): see the LDS layout below
  static constexpr __device__ __forceinline__ int swz_b(int k, int) { return (k & 1) << 3; }
};
template <>
struct RmElem<float> {
  typedef float acc_t __attribute__((ext_vector_type(4)));
  static constexpr int CYCLES = 32;
  static __device__ __forceinline__ acc_t mfma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static constexpr __device__ __forceinline__ int swz_b(int k, int cpb) {
    return cpb >= 16 ? (k & 3) << 2 : ((k >> 1) & 1) << 2;
  }
};

// ---------------------------------------------------------------------------
// Row-major direct-to-LDS kernels: A and B are read where they lie, any leading dimension
// and any alignment of the element type. Slabs are copied HBM -> LDS by 16-byte buffer loads,
// which need 4-byte aligned addresses only: each wave instruction fills one contiguous 1 KiB
// LDS block, lane p writing bytes [16p, 16p+16), and the lane -> address map sets the layout.
//
// LDS layout of one stage, in 16-byte chunks (CH elements: 2 doubles or 4 floats):
//   A: BM rows x BK elements, CPR = BK/CH chunks per row, chunk c of row r at slot
//      c ^ sw(r), sw(r) = (r * CPR / 16) mod CPR: the lanes of an MFMA operand read (16 rows,
//      neighbouring k) cover all 64 banks evenly.
//   B: BK rows x BN elements, chunk c of row k at slot c ^ swz_b(k), so the 16-lane groups of
//      an operand read (rows k, k+1, ...) use different banks.
// A slab with fewer than BK k rows (the end of a panel) takes 4-byte loads into the same
// layout, each checked against k, rows and columns, so padding is exact zeros in both
// operands. So do the slabs that hold the last rows of B where a 16-byte load of the last columns
// would read past the last row's end (rm_checked_rows).
//
// What bounds it. An FP64 MFMA holds its SIMD's vector pipe for 64 cycles, an FP32 one for 32,
// and a vector instruction of any kind waits for the MFMA before it to leave: one address
// addition per FP64 MFMA makes 64 cycles 99 (measured on one wave), while LDS reads, loads to
// LDS and scalar instructions issue beside it for nothing. So the loop over full slabs holds
// MFMAs, LDS reads at a lane's constant address plus an immediate, loads at a lane's constant
// offset plus a scalar one, and nothing vector: every stage of the ring has its own copy of the
// code. Operands are read ahead of their MFMAs and across the slab barrier (the barrier of slab
// s waits for slab s + 1), since in a small problem one wave per SIMD has nothing else to hide
// LDS latency with. At the full MFMA rate a CU on 256x128 tiles loads 14 GB/s, one on 32x32
// tiles 74, half of what its loads to LDS reach from L2 (150): hence large tiles where there
// are enough of them.
// ---------------------------------------------------------------------------
template <class E, int BM, int BN, int WM, int WN, int BK_, int STAGES_>
struct RmShape {
  static constexpr int SZ = sizeof(E), CH = 16 / SZ;  // bytes per element, elements per chunk
  static constexpr int BK = BK_;
  static constexpr int STAGES = STAGES_;
  static constexpr int NW = WM * WN;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int TM = WTM / 16, TN = WTN / 16;
  static constexpr int CPR = BK / CH, CPB = BN / CH;     // chunks per A row, per B row
  static constexpr int ARB = 64 / CPR, BRB = 64 / CPB;   // A rows, B rows per 1 KiB block
  static constexpr int A_BYTES = BM * BK * SZ, B_BYTES = BK * BN * SZ;  // of a stage; A's stages, then B's
  static constexpr int B_BASE = STAGES * A_BYTES;
  static constexpr int LDS_BYTES = STAGES * (A_BYTES + B_BYTES);
  static constexpr int PA = A_BYTES / 1024 / NW, PB = B_BYTES / 1024 / NW;  // 1 KiB blocks per wave
  static constexpr int PER = PA + PB;
  static constexpr int KSTEPS = BK / 4;
  static_assert(CPR == 8 || CPR == 16, "slab depth");
  static_assert(CPB >= 8 && CPB <= 64 && BM % (NW * ARB) == 0 && BK % (NW * BRB) == 0, "blocks split evenly");
  static_assert((NW * ARB) % 16 == 0 && (NW * BRB) % 4 == 0, "a wave's blocks share their swizzle");
  static_assert(TM >= 1 && TN >= 1, "wave tile");
  // Operand sets in registers: set kk % RING holds k step kk, and behind step kk's MFMAs the
  // set of step kk - 1 is refilled with step kk + RING - 1. The fewer MFMAs a k step has, the
  // further ahead its operands are read. Two stages leave no slab to read ahead from: the
  // operands of a slab are read after its own barrier.
  static constexpr bool AHEAD = STAGES >= 3;
  static constexpr int STEP = TM * TN * RmElem<E>::CYCLES;  // cycles of a k step's MFMAs
  static constexpr int RING = STEP >= 256 ? 2 : STEP >= 128 ? 4 : KSTEPS < 8 ? KSTEPS : 8;
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
template <class E, int BM, int BN, int WM, int WN, int BK, int STAGES, bool MP, class Desc>
__device__ __forceinline__ void rm_tile(const Desc &d, int row0, int col0) {
  using K = RmShape<E, BM, BN, WM, WN, BK, STAGES>;
  using X = RmElem<E>;
  using acc_t = typename X::acc_t;
  constexpr int SZ = K::SZ, CH = K::CH;
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
    a_off[kk] = (wm * K::WTM + li) * BK * SZ + ((((4 * kk + g) / CH) ^ swz(li)) << 4) + (4 * kk + g) % CH * SZ;
#pragma unroll
  for (int j = 0; j < K::TN; ++j) {
    const int col = wn * K::WTN + j * 16 + li;
    b_off[j] = K::B_BASE + g * BN * SZ + (((col / CH) ^ X::swz_b(g, K::CPB)) << 4) + col % CH * SZ;
  }
  // this lane's row and chunk in the wave's first A block and first B block
  const int ar = wave * K::ARB + lane / K::CPR, ac = (lane % K::CPR) ^ swz(ar);
  const int br = wave * K::BRB + lane / K::CPB, bc = (lane % K::CPB) ^ X::swz_b(br, K::CPB);
  {
    const int m_rem = uni(d.m - row0);
    const int n_rem = uni(d.n - col0);
    const long lda = uni(d.lda), ldb = uni(d.ldb), ldc = uni(d.ldc);
    const E *Ag = uni(d.A) + (long)row0 * lda;
    const E *Bg = uni(d.B) + col0;
    const int Kdim = uni(d.k);
    int w = Kdim;
    if constexpr (MP) {
      const int dpanel = uni(d.panel);
      if (dpanel > 0 && dpanel < Kdim) w = dpanel;
    }
    const int spp = (w + BK - 1) / BK;  // slabs per full panel
    const int full_panels = MP ? Kdim / w : 1;
    const int nslab = MP ? uni(full_panels * spp + (Kdim - full_panels * w + BK - 1) / BK) : spp;
    const int last_panel = MP && Kdim % w ? Kdim % w : w;
    // slabs that end past k16 take 4-byte loads
    const int checked =
        rm_checked_rows<CH>(d.n, ldb, !((reinterpret_cast<uintptr_t>(Bg) / SZ | (uintptr_t)ldb) & (CH - 1)));
    const int k16 = Kdim - checked;

    // Every 1 KiB block is addressed from its own first row (ARB or BRB rows, uniform), so one
    // lane offset serves all of an operand's blocks. A rows past m_rem lie at or beyond
    // num_records and read zero (k rides in the scalar offset, which the range check adds: within
    // a row of lda >= k it stays below); B chunks past n_rem go out of range here.
    rsrc_t rA[K::PA];
#pragma unroll
    for (int u = 0; u < K::PA; ++u) {
      const int r0 = (wave + u * K::NW) * K::ARB;
      rA[u] = make_rsrc(Ag + (long)r0 * lda, (long)min(m_rem - r0, K::ARB) * lda * SZ);
    }
    const uint32_t ga = (uint32_t)(((long)(lane / K::CPR) * lda + CH * ac) * SZ);
    const uint32_t gb = CH * bc < n_rem ? (uint32_t)(((long)(lane / K::CPB) * ldb + CH * bc) * SZ) : kOOB;

    // the next slab to issue: its first k row, the end of its panel, its stage
    int ikb = 0, ipe = min(w, Kdim), istage = 0;
    const E *iB = Bg;
    auto rsrc_b = [&](int u) {
      return __builtin_amdgcn_make_buffer_rsrc(const_cast<E *>(iB + (long)(wave + u * K::NW) * K::BRB * ldb),
                                               (short)0, 0x7fffffff, 0x00020000);
    };
    // block u of a full slab: A's, then B's
    auto load_block = [&](int u, int q) {
      if (u < K::PA)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rA[u], (lds_void *)(smem + q * K::A_BYTES + (wave + u * K::NW) * 1024),
                                                  16, ga, ikb * SZ, 0, 0);
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
      if (krem == BK && ikb + BK <= k16) {
#pragma unroll
        for (int u = 0; u < K::PER; ++u) load_block(u, istage);
      } else {
#pragma unroll
        for (int u = 0; u < K::PA; ++u)
#pragma unroll 1
          for (int v = 0; v < 4; ++v) {
            const int pos = v * 16 + (lane >> 2), r0 = (wave + u * K::NW) * K::ARB, r = pos / K::CPR;
            const int c = (pos % K::CPR) ^ swz(r0 + r);
            const uint32_t off = r0 + r < m_rem && CH * c + (lane & 3) * 4 / SZ < krem
                                     ? (uint32_t)((long)r * lda * SZ + c * 16 + (lane & 3) * 4)
                                     : kOOB;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rA[u], (lds_void *)(smem + istage * K::A_BYTES + (wave + u * K::NW) * 1024 + v * 256), 4, off,
                ikb * SZ, 0, 0);
          }
#pragma unroll
        for (int u = 0; u < K::PB; ++u)
#pragma unroll 1
          for (int v = 0; v < 4; ++v) {
            const int pos = v * 16 + (lane >> 2), r0 = (wave + u * K::NW) * K::BRB, r = pos / K::CPB;
            const int c = (pos % K::CPB) ^ X::swz_b(r0 + r, K::CPB);
            const uint32_t off = r0 + r < krem && CH * c + (lane & 3) * 4 / SZ < n_rem
                                     ? (uint32_t)((long)r * ldb * SZ + c * 16 + (lane & 3) * 4)
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
    // extra loads of a last slab in 4-byte pieces (one before it, with ldb < CH, is waited for longer)
    const int last_units = last_panel % BK || checked ? 3 : 0;
#pragma unroll 1
    for (int s0 = 0; s0 < STAGES - 1 && s0 < nslab; ++s0) issue();

    int issued = min(STAGES - 1, nslab);
    // slab t has landed once the slabs issued after it are all that is outstanding
    auto wait_slab = [&](int t) {
      const int later = issued - 1 - t;
      wait_units<K::PER, STAGES + 1>(later > 0 && issued == nslab ? later + last_units : later);
    };
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
    constexpr bool CFIRST = MP || (K::TM * K::TN * SZ <= 32 && K::NW <= 8);
    acc_t acc[K::TM][K::TN], creg[CFIRST ? K::TM : 1][CFIRST ? K::TN : 1];
#pragma unroll
    for (int i = 0; i < K::TM; ++i)
#pragma unroll
      for (int j = 0; j < K::TN; ++j) {
        acc[i][j] = acc_t{};
      }
    const CTile<E, acc_t, K::TM, K::TN, 16, 4> ct(uni(d.C) + (long)(row0 + wm * K::WTM) * ldc + col0 + wn * K::WTN, ldc,
                                                  m_rem - wm * K::WTM, n_rem - wn * K::WTN, lane);
    if constexpr (CFIRST) ct.load_all(creg);

    auto read_ops = [&](int q, int kk, E(&x)[K::TM], E(&y)[K::TN]) {
#pragma unroll
      for (int i = 0; i < K::TM; ++i)
        x[i] = *reinterpret_cast<const E *>(smem + a_off[kk] + (q * K::A_BYTES + i * 16 * BK * SZ));
#pragma unroll
      for (int j = 0; j < K::TN; ++j)
        y[j] = *reinterpret_cast<const E *>(smem + b_off[j] + (q * K::B_BYTES + kk * 4 * BN * SZ));
    };
    auto mfmas = [&](const E(&x)[K::TM], const E(&y)[K::TN]) {
#pragma unroll
      for (int i = 0; i < K::TM; ++i)
#pragma unroll
        for (int j = 0; j < K::TN; ++j)
          acc[i][j] = X::mfma(x[i], y[j], acc[i][j]);
    };
    E a[K::RING][K::TM], b[K::RING][K::TN];
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
              acc[i][j] = acc_t{};
            }
        }
      }
    });
    if constexpr (CFIRST) {
      if constexpr (!MP)
#pragma unroll
        for (int i = 0; i < K::TM; ++i)
#pragma unroll
          for (int j = 0; j < K::TN; ++j) creg[i][j] = creg[i][j] + acc[i][j];
      ct.store_all(creg);
    } else {
      ct.update([&](E c, int i, int j, int r) { return c + acc[i][j][r]; });
    }
  }
}

template <int BM, int BN, class Desc>
__device__ __forceinline__ void tile_origin(const Desc &d, int lt, int group_m, int &row0, int &col0) {
  const int tiles_n = d.tiles_n;
  const int tiles_m = (d.m + BM - 1) / BM;
  const int grp = lt / (group_m * tiles_n);
  const int first_m = grp * group_m;
  const int gsz = min(tiles_m - first_m, group_m);
  const int in_grp = lt - grp * group_m * tiles_n;
  row0 = uni((first_m + in_grp % gsz) * BM);
  col0 = uni((in_grp / gsz) * BN);
}

// Tile of workgroup bid, which runs on XCD bid % 8: of every `window` tiles each XCD takes a
// contiguous run, so that neighbouring tiles share its L2
__device__ __forceinline__ int xcd_run(int bid, int total, int window) {
  const int w0 = bid / window * window, r = bid - w0;
  const int n = min(window, total - w0);
  return w0 + (r % 8) * (n / 8) + min(r % 8, n % 8) + r / 8;
}

// Tiles of shape T, and, from tile batch.tail_start on, the smaller tiles of shape U: the part
// of the work that would leave the last round of T tiles nearly empty.
template <class T, class U>
__device__ __forceinline__ void rm_body(const RmBatch<typename T::Desc> &batch) {
  const int G = gridDim.x;
  const int bid = blockIdx.x;
  const int total = batch.total_tiles, head = batch.tail_start;
  int slot = bid;
  if (batch.xcd_remap) {
    if (G == total)
      slot = bid < head ? xcd_run(bid, head, batch.window) : head + xcd_run(bid - head, total - head, batch.window);
    else if (G % 8 == 0)
      slot = (bid % 8) * (G / 8) + bid / 8;
  }
  slot = uni(slot);
  for (int t = slot; t < total; t += G) {
    int row0, col0;
    const typename T::Desc d = uniform_desc(batch, uni(t));
    if (std::is_same<T, U>::value || t < head) {
      tile_origin<T::BM, T::BN>(d, t - d.tile_start, batch.group_m, row0, col0);
      T::run(d, row0, col0);
    } else if constexpr (!std::is_same<T, U>::value) {
      tile_origin<U::BM, U::BN>(d, t - d.tile_start, batch.group_m, row0, col0);
      U::run(d, row0, col0);
    }
  }
}

// A tile shape: BM x BN outputs, WM x WN waves, STAGES slabs of BK k
template <class E, int BM_, int BN_, int WM, int WN, int BK, int STAGES, bool MP>
struct RmTile {
  using K = RmShape<E, BM_, BN_, WM, WN, BK, STAGES>;
  using Desc = typename std::conditional<std::is_same<E, double>::value, GemmDesc, F32Desc>::type;
  static constexpr int BM = BM_, BN = BN_, THREADS = WM * WN * 64;
  static constexpr int LDS = K::LDS_BYTES, A_ROWS = K::ARB, B_ROWS = K::BRB;
  static __device__ __forceinline__ void run(const Desc &d, int row0, int col0) {
    rm_tile<E, BM, BN, WM, WN, BK, STAGES, MP>(d, row0, col0);
  }
};

// waves_per_eu(2): with the whole register file of a SIMD for one wave, the compiler keeps the
// accumulators in one half of it and copies them through the other on every slab
template <class T, class U>
__global__ __launch_bounds__(T::THREADS) __attribute__((amdgpu_waves_per_eu(2))) void rm_kernel(
    RmBatch<typename T::Desc> batch) {
  static_assert(T::THREADS == U::THREADS, "one workgroup shape");
  rm_body<T, U>(batch);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
template <class Desc>
long rm_tiles(const Desc &d, int bm, int bn) {
  return (long)((d.m + bm - 1) / bm) * ((d.n + bn - 1) / bn);
}

// GEMMs whose rows of A lie so far apart that `rows` of them span 2 GiB or more, a load's 32-bit
// offset, become GEMMs of one row each
template <class Desc>
void rm_split_rows(std::vector<Desc> &v, long rows) {
  auto far = [&](const Desc &d) { return rows * d.lda * (long)sizeof(*d.C) >= 0x7fffffffL; };
  if (std::none_of(v.begin(), v.end(), far)) return;
  std::vector<Desc> split;
  for (const Desc &d : v) {
    if (!far(d)) {
      split.push_back(d);
      continue;
    }
    for (int r = 0; r < d.m; ++r) {
      Desc t = d;
      t.A += (long)r * d.lda;
      t.C += (long)r * d.ldc;
      t.m = 1;
      t.lda = d.k;
      split.push_back(t);
    }
  }
  v.swap(split);
}

// elements of B from one column to the next
inline long rm_col_step(const GemmDesc &) { return 1; }
inline long rm_col_step(const F32Desc &) { return 1; }
inline long rm_col_step(const Bf3Desc &d) { return d.ldb; }

// Split `live` so that its bm x bn head tiles fill whole rounds of the CUs and the rest, moved
// to `tail`, runs on smaller tiles: a last round of head tiles that is nearly empty costs as
// much as a full one (FP64 1777 x 1999 x 1235: 560 tiles of 64x64 on 256 CUs take three
// rounds, 181 us; 500 of them and the rest as 32x32 take 2.25, 138 us). Every output's
// arithmetic is its own, so where the line runs does not change a result. The cut takes rows
// or columns of tiles, whichever step is finer, off the last GEMMs; a last round that is more
// than `most` fifths full stays.
template <class Desc>
void rm_split_tail(std::vector<Desc> &live, int bm, int bn, long cus, std::vector<Desc> &tail, int most = 4) {
  long total = 0;
  for (const Desc &d : live) total += rm_tiles(d, bm, bn);
  const long rounds = total / cus, rest = total % cus;
  if (rounds == 0 || rest == 0 || 5 * rest > most * cus) return;
  long excess = rest;
  for (int i = (int)live.size() - 1; i >= 0 && excess > 0; --i) {
    Desc &d = live[i];
    const long tm = (d.m + bm - 1) / bm, tn = (d.n + bn - 1) / bn;
    Desc t = d;
    if (tn <= tm) {  // whole rows of tn tiles
      const long cut = std::min(tm, (excess + tn - 1) / tn), keep = (tm - cut) * bm;
      t.A += keep * t.lda;
      t.C += keep * t.ldc;
      t.m -= (int)keep;
      d.m = (int)keep;
      excess -= cut * tn;
    } else {
      const long cut = std::min(tn, (excess + tm - 1) / tm), keep = (tn - cut) * bn;
      t.B += keep * rm_col_step(t);
      t.C += keep;
      t.n -= (int)keep;
      d.n = (int)keep;
      excess -= cut * tm;
    }
    tail.insert(tail.begin(), t);
    if (d.m == 0 || d.n == 0) live.erase(live.begin() + i);
  }
}

// Tiles over which an XCD's runs extend: all of a launch's own tiles where its descriptors travel
// with it (16384^3 FP64 117.8 ms, 118.4 with runs over a round of CUs), a round of CUs for a list,
// whose tiles take unequal times (512 FP32 GEMMs of k from 64 to 4096: 24.5 ms with eight runs
// over the whole list, 9.25 with runs over a round).
inline int rm_window(bool list, int total, int cus) { return list ? cus : total; }

// Number the tiles of v from *t on; false if there are too many for an int
template <class Desc>
bool rm_number(std::vector<Desc> &v, int bm, int bn, long *t) {
  for (Desc &d : v) {
    d.tiles_n = (d.n + bn - 1) / bn;
    d.tile_start = (int)*t;
    *t += rm_tiles(d, bm, bn);
    if (*t > 0x7fffffffL) return false;
  }
  return true;
}

// The device list of a launch of `total` tiles: its descriptors, then their index
template <class Desc>
std::vector<char> rm_list(const std::vector<Desc> &descs, int total) {
  const size_t n = descs.size() * sizeof(Desc);
  std::vector<char> list(n + rm_index_entries(total) * sizeof(int));
  memcpy(list.data(), descs.data(), n);
  int *index = reinterpret_cast<int *>(list.data() + n);
  int d = 0;
  for (size_t c = 0; c < rm_index_entries(total); ++c) {
    while (d + 1 < (int)descs.size() && (long)descs[d + 1].tile_start <= (long)c * kIndexTiles) ++d;
    index[c] = d;
  }
  return list;
}

}  // namespace
