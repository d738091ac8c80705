// The residue products of the CRT split GEMM: for every modulus m_t, R_t = A_t B_t mod m_t on
// int8 operands, all moduli in one launch.
//
// What bounds it: the matrix cores, at the rate that the card sustains on dense int8 operands
// (16384^3 with 13 moduli 44.8 ms, 2550 TOP/s at the 1.83 GHz that its power leaves; a plain
// library int8 product makes 2230), then the reduction of each tile's sums. In 64x64 wave
// tiles, 16-byte LDS reads took as long as the
// MFMAs; a wave of 8 now has 128x64 outputs (three quarters), reads a slab's operands behind the
// MFMAs of the slab before, and does no vector arithmetic in the loop over slabs. One launch for
// all moduli fills the last round once, not once per modulus: 1105x3061x7548 (150 tiles of
// 256x256 a modulus) 715 -> 366 us, 2000^3 306 -> 116, 4096^3 960 -> 795, 8192^3 5.97 -> 5.7 ms,
// 16384^3 46.1 -> 44.8 (the rate that the card holds).
// Runs of tiles per XCD extend over two rounds, so that all eight work on a modulus or two and
// operands come from memory about once (a run of whole moduli per XCD: 16384^3 47.6 ms;
// 1105x3061x7548 is 366 us with two rounds, 425 with one).
#include "gemm_rm.h"
#include "phpc_internal.h"

#include <algorithm>
#include <mutex>

namespace {

typedef int i4v __attribute__((ext_vector_type(4)));
typedef uint32_t __attribute__((aligned(1))) u1u;

// |residues| <= 128: 128^2 * 130944 + 128 < 2^31, and 130944 is a whole number of slabs
constexpr int kMaxExactTerms = 130944;
constexpr int kBK = 64;  // bytes of k per slab

struct CrtLevelArgs {
  const int8_t *A8, *B8;  // crt_offset()
  int8_t *res;            // plane t at t * m * n, row-major
  int kp, m, n, L;
  int tiles_m, tiles_n, window;
  int mods[20];
  int c19[20];  // 2^19 mod m, symmetric
};

// v mod an odd m <= 255 in the symmetric range (|r| <= (m - 1) / 2), m wave-uniform: v = h 2^19 + l
// with -4096 <= h < 4096, so h c + l with c = 2^19 mod m (|c| <= 127) is v mod m and below 2^20,
// exact in FP32. Over m it is below 6100, where rounding 1 / m and the product moves it by less
// than 0.001, while it lies at least 1 / (2 m) from a half-integer: the nearest integer is the
// exact quotient. (Two rounds on |v|, with twice the instructions: 4096^3 with 13 moduli 840 us,
// 795 now.)
__device__ __forceinline__ int smod_odd(int v, int c, float m, float rm) {
  const float f = (float)(__mul24(v >> 19, c) + (v & 0x7ffff));
  return (int)fmaf(-rintf(f * rm), m, f);
}

// LDS slots of a 64-byte row. A 16-byte read serves lanes 0-3, 12-15 and 20-27 together, then
// 4-11, 16-19 and 28-31 (the upper lanes likewise): with lane l on row l % 16, chunk l / 16, the
// rows 8-15 two slots on, these cover all 64 banks once. (r / 4 % 4 covers them once for 16
// neighbouring lanes, and cost a conflict on every read: 16384^3 47.1 ms, 44.8 now.)
__device__ __forceinline__ int swizzle(int r) { return (r >> 3 & 1) << 1; }

template <int BM, int BN, int WM, int WN, int STAGES>
struct CrtShape {
  static constexpr int NW = WM * WN;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int TM = WTM / 16, TN = WTN / 16;
  static constexpr int A_BYTES = BM * kBK, B_BYTES = BN * kBK;
  static constexpr int B_BASE = STAGES * A_BYTES;
  static constexpr int LDS_BYTES = STAGES * (A_BYTES + B_BYTES);
  static constexpr int PA = A_BYTES / 1024 / NW, PB = B_BYTES / 1024 / NW, PER = PA + PB;
  static constexpr int UNROLL = STAGES % 2 ? 2 * STAGES : STAGES;
  static_assert(PA * NW * 1024 == A_BYTES && PB * NW * 1024 == B_BYTES, "blocks split evenly");
  static_assert(STAGES >= 3 && LDS_BYTES <= 160 * 1024, "pipeline");
};

template <int BM, int BN, int WM, int WN, int STAGES>
__device__ __forceinline__ void crt_tile(const CrtLevelArgs &g, int mod, int row0, int col0) {
  using K = CrtShape<BM, BN, WM, WN, STAGES>;
  constexpr int TM = K::TM, TN = K::TN;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int wave = uni((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const int wm = wave / WN, wn = wave % WN;
  const int m = g.m, n = g.n;

  // crt_offset() keeps 16 rows' 64 bytes together, so a load takes one KiB (rows of one modulus
  // 64 bytes at a time: 16384^3 59.7 ms against 50.2 on the same tiles).
  // A stage holds rows of 64 bytes, 16-byte chunk c of row r at slot c ^ swizzle(r). A wave's
  // load fills 16 rows; rows past the matrix edge read the last one, whose outputs are not
  // written.
  rsrc_t src[K::PER];
  uint32_t off[K::PER];
  int step[K::PER];  // bytes from one slab to the next
#pragma unroll
  for (int u = 0; u < K::PER; ++u) {
    const bool is_a = u < K::PA;
    const int rows = is_a ? m : n, r = lane >> 2;
    const int r0 = min(is_a ? row0 + (wave + u * K::NW) * 16 : col0 + (wave + (u - K::PA) * K::NW) * 16,
                       (rows - 1) / 16 * 16);
    const int held = min(16, rows - r0);
    src[u] = make_rsrc((is_a ? g.A8 : g.B8) + ((long)mod * rows + r0) * g.kp, 0x7fffffffL);
    off[u] = (uint32_t)(min(r, held - 1) * kBK + (((lane & 3) ^ swizzle(r)) << 4));
    step[u] = held * kBK;
  }
  auto issue = [&](int stage, int slab) {
#pragma unroll
    for (int u = 0; u < K::PER; ++u) {
      const int at = u < K::PA ? stage * K::A_BYTES + (wave + u * K::NW) * 1024
                               : K::B_BASE + stage * K::B_BYTES + (wave + (u - K::PA) * K::NW) * 1024;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(src[u], (lds_void *)(smem + at), 16, off[u], slab * step[u], 0, 0);
    }
  };
  // walk slabs s0 .. s1: step t waits for slab t + 1, refills the stage of slab t (whose operands
  // are in registers by then) with slab t + STAGES, reads the operands of t + 1 and multiplies
  auto walk = [&](int s0, int s1, auto read, auto mul) {
    const int nslab = s1 - s0;
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
      if (s < nslab) issue(s, s0 + s);
    if (nslab >= STAGES)
      wait_vm_c<(STAGES - 1) * K::PER>();
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
          wait_vm_c<(STAGES - 2) * K::PER>();
          __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave has its operands
          slab_barrier();
          issue(q % STAGES, s0 + t + q + STAGES);
          read(std::integral_constant<int, (q + 1) % STAGES>{}, std::integral_constant<int, (q + 1) % 2>{});
          mul(std::integral_constant<int, q % 2>{}, std::true_type{});
        });
      for_stages<K::UNROLL>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if (t < nslab) {
          if (t + STAGES <= nslab)
            wait_vm_c<(STAGES - 2) * K::PER>();
          else
            wait_vm_c<0>();
          __builtin_amdgcn_s_waitcnt(0xC07F);
          slab_barrier();
          if (t + STAGES < nslab) issue(q % STAGES, s0 + t + STAGES);
          if (t + 1 < nslab)
            read(std::integral_constant<int, (q + 1) % STAGES>{}, std::integral_constant<int, (q + 1) % 2>{});
          mul(std::integral_constant<int, q % 2>{}, std::false_type{});
          ++t;
        }
      });
    }
  };
  const int nslab = g.kp / kBK;
  constexpr int kPiece = kMaxExactTerms / kBK;
  const int wrow = row0 + wm * K::WTM, wcol = col0 + wn * K::WTN;
  if (wrow >= m || wcol >= n) {
    // all of this wave's outputs lie past the matrix edge: it only loads its share
#pragma unroll 1
    for (int s0 = 0; s0 < nslab; s0 += kPiece)
      walk(s0, min(s0 + kPiece, nslab), [](auto, auto) {}, [](auto, auto) {});
    return;
  }

  i4v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = i4v{};
  i4v a[2][TM], b[2][TN];
  const int slot = ((lane >> 4) ^ swizzle(lane % 16)) << 4;
  const int a0 = (wm * K::WTM + lane % 16) * kBK + slot, b0 = K::B_BASE + (wn * K::WTN + lane % 16) * kBK + slot;
  auto read = [&](auto stage, auto set) {
    constexpr int q = decltype(stage)::value, x = decltype(set)::value;
#pragma unroll
    for (int i = 0; i < TM; ++i)
      a[x][i] = *reinterpret_cast<const i4v *>(smem + a0 + (q * K::A_BYTES + i * 16 * kBK));
#pragma unroll
    for (int j = 0; j < TN; ++j)
      b[x][j] = *reinterpret_cast<const i4v *>(smem + b0 + (q * K::B_BYTES + j * 16 * kBK));
  };
  auto mul = [&](auto set, auto steady) {
    constexpr int x = decltype(set)::value;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)  // operands swapped: a lane's registers run along a row of the result
        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b[x][j], a[x][i], acc[i][j], 0, 0, 0);
    if constexpr (decltype(steady)::value) {
      // the next slab's operand reads evenly between the MFMAs
      constexpr int NRD = TM + TN, NMF = TM * TN;
      constexpr int EACH = NMF / NRD > 0 ? NMF / NRD : 1;
#pragma unroll
      for (int r = 0; r < NRD; ++r) {
        __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, NMF, 0);
    }
  };
  const int mod_m = g.mods[mod];
  const int c19 = g.c19[mod];
  const float mf = (float)mod_m, rmf = 1.0f / mf;
  // m = 256 takes the low byte
  auto smod = [&](int v) { return mod_m == 256 ? (int)(int8_t)v : smod_odd(v, c19, mf, rmf); };
  auto reduce = [&]() {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] = smod(acc[i][j][r]);
  };
  walk(0, min(kPiece, nslab), read, mul);
#pragma unroll 1
  for (int s0 = kPiece; s0 < nslab; s0 += kPiece) {
    reduce();
    walk(s0, min(s0 + kPiece, nslab), read, mul);
  }

  int8_t *out = g.res + (long)mod * m * n + (long)wrow * n + wcol;
  const int m_rem = m - wrow, n_rem = n - wcol;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int row = i * 16 + lane % 16, col = j * 16 + 4 * (lane >> 4);
      uint32_t b[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) b[r] = mod_m == 256 ? acc[i][j][r] : smod_odd(acc[i][j][r], c19, mf, rmf);
      // their low bytes in order
      const uint32_t w = __builtin_amdgcn_perm(__builtin_amdgcn_perm(b[3], b[2], 0x0c0c0400),
                                               __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400), 0x05040100);
      int8_t *o = out + (long)row * n + col;
      if (row < m_rem) {
        if (col + 3 < n_rem) {
          *reinterpret_cast<u1u *>(o) = w;
        } else {
#pragma unroll
          for (int e = 0; e < 3; ++e)
            if (col + e < n_rem) o[e] = (int8_t)(w >> (8 * e));
        }
      }
    }
}

template <int BM, int BN, int WM, int WN, int STAGES>
__global__ __launch_bounds__(WM *WN * 64) __attribute__((amdgpu_waves_per_eu(2))) void crt_level_kernel(CrtLevelArgs g) {
  const int tiles = g.tiles_m * g.tiles_n;
  const int t = uni(xcd_run(blockIdx.x, tiles * g.L, g.window));
  const int mod = t / tiles, lt = t - mod * tiles;
  const int gm = 8, grp = lt / (gm * g.tiles_n), first_m = grp * gm;
  const int gsz = min(g.tiles_m - first_m, gm), in_grp = lt - grp * gm * g.tiles_n;
  crt_tile<BM, BN, WM, WN, STAGES>(g, mod, uni((first_m + in_grp % gsz) * BM), uni((in_grp / gsz) * BN));
}

struct CrtConfig {
  int bm, bn, threads;
  size_t lds;
  void (*fn)(CrtLevelArgs);
};
template <int BM, int BN, int WM, int WN, int STAGES>
constexpr CrtConfig crt_config() {
  return {BM, BN, WM * WN * 64, (size_t)CrtShape<BM, BN, WM, WN, STAGES>::LDS_BYTES,
          crt_level_kernel<BM, BN, WM, WN, STAGES>};
}
const CrtConfig kCrt[] = {
    crt_config<256, 256, 2, 4, 4>(),
    crt_config<128, 128, 2, 2, 3>(),
    crt_config<64, 64, 2, 2, 3>(),
};
// By how many tiles all moduli give the CUs (13 moduli, device time): 256x256 from six a CU on
// (4096^3, 13 a CU: 795 us against 854 on 128x128; 2000^3, 3.3 a CU: 143 against 116); 64x64 for
// fewer than two 128x128 tiles a CU (100x130x70: 7.6 us against 12.5).
int pick(long m, long n, int L) {
  const long cus = phpc_device().cus;
  if (L * ((m + 255) / 256) * ((n + 255) / 256) >= 6 * cus) return 0;
  return L * ((m + 127) / 128) * ((n + 127) / 128) >= 2 * cus ? 1 : 2;
}
std::once_flag g_crt_once;

}  // namespace

int phpc_crt_level(const int8_t *A8, const int8_t *B8, long kp, int m, int n, int L, const int *mods, int8_t *res,
                   hipStream_t s) {
  // 16 rows' k is read through a 32-bit buffer offset
  if (16 * kp >= 0x7fffffffL || kp % kBK)
    return phpc_set_error(PHPC_ERR_ARG, "operand rows of %ld bytes too long for the residue products", kp);
  std::call_once(g_crt_once, [] {
    for (const CrtConfig &c : kCrt)
      (void)hipFuncSetAttribute(reinterpret_cast<const void *>(c.fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)c.lds);
  });
  const CrtConfig &c = kCrt[pick(m, n, L)];
  CrtLevelArgs g{};
  g.A8 = A8;
  g.B8 = B8;
  g.res = res;
  g.kp = (int)kp;
  g.m = m;
  g.n = n;
  g.L = L;
  g.tiles_m = (m + c.bm - 1) / c.bm;
  g.tiles_n = (n + c.bn - 1) / c.bn;
  for (int t = 0; t < L; ++t) {
    g.mods[t] = mods[t];
    const int c = (1 << 19) % mods[t];
    g.c19[t] = 2 * c > mods[t] ? c - mods[t] : c;
  }
  const long total = (long)g.tiles_m * g.tiles_n * L;
  if (total > 0x7fffffffL) return phpc_set_error(PHPC_ERR_ARG, "too many tiles");
  g.window = 2 * phpc_device().cus;
  const int kt = phpc_ktime_begin(s);
  hipLaunchKernelGGL(c.fn, dim3((unsigned)total), dim3(c.threads), c.lds, s, g);
  phpc_ktime_end(kt, s);
  PHPC_HIP(hipGetLastError());
  return PHPC_OK;
}
