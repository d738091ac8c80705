// Internal declarations shared by the HIP sources of libphpc (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <vector>
#include <stdint.h>
#include <stddef.h>

#include "phpc_gemm.h"

// An event destroyed when its scope ends, error returns included.
struct ScopedEvent {
  hipEvent_t e = nullptr;
  explicit ScopedEvent(unsigned flags = hipEventDefault) {
    if (hipEventCreateWithFlags(&e, flags) != hipSuccess) e = nullptr;
  }
  ~ScopedEvent() {
    if (e) (void)hipEventDestroy(e);
  }
  ScopedEvent(const ScopedEvent &) = delete;
  ScopedEvent &operator=(const ScopedEvent &) = delete;
  ScopedEvent(ScopedEvent &&o) noexcept : e(o.e) { o.e = nullptr; }
};

// p[idx] where ok, else 0, through a load that always happens (from p[0] where !ok; p[0]
// must be readable). A guarded load compiles to a branch with a wait for the load inside
// it, so a thread's guarded loads go out one at a time; these all go out before the first
// wait.
template <class T>
__device__ __forceinline__ T load_or_zero(const T *p, long idx, bool ok) {
  const T v = p[ok ? idx : 0];
  return ok ? v : T(0);
}

// ---------------------------------------------------------------------------
// Error handling: every entry point records its status in a thread-local slot
// (phpc_last_error) and returns it where the signature allows.
// ---------------------------------------------------------------------------
extern "C" int phpc_set_error(int code, const char *fmt, ...);
#define PHPC_HIP(call)                                                                   \
  do {                                                                                   \
    hipError_t e_ = (call);                                                              \
    if (e_ != hipSuccess)                                                                \
      return phpc_set_error(PHPC_ERR_HIP, "%s failed: %s (%s:%d)", #call,                \
                            hipGetErrorString(e_), __FILE__, __LINE__);                  \
  } while (0)

// ---------------------------------------------------------------------------
// One GEMM of a grouped launch: C[m x n] (ldc) += A[m x k] (lda) * B[k x n] (ldb),
// row-major FP64. The k range is walked in panels of `panel` columns; each panel's
// product is summed from zero and then added to the C value carried from the
// previous panel, i.e. C = ((C0 + s_0) + s_1) + ... (the grouping produced by one
// local-GEMM call per SUMMA step, src/phpc_summa.c:63-95 with src/phpc_gemm.cu:32,55).
// ---------------------------------------------------------------------------
struct GemmDesc {
  const double *A;
  const double *B;
  double *C;
  long lda, ldb, ldc;
  int m, n, k;
  int panel;       // >= k: one panel
  int tiles_n;     // tiles along n for this GEMM (filled by the planner)
  int tile_start;  // first global tile id of this GEMM (prefix sum)
};

// One FP32 GEMM of a grouped launch (row-major, C += A*B).
struct F32Desc {
  const float *A;
  const float *B;
  float *C;
  long lda, ldb, ldc;
  int m, n, k;
  int tiles_n;
  int tile_start;
};
int phpc_f32_num_configs();
void phpc_f32_config_tile(int id, int *bm, int *bn);
int phpc_f32_plan_tiles(F32Desc *descs, int ndesc, int id);
void phpc_f32_set_direct(int on);
// configuration of FP32 plans created without autotuning: -1 = the direct kernels
// (configuration 3), or by work 0 (64x64) or 2 (128x128) where a leading dimension does not fit
// their 32-bit offsets or tuning key 6 is off; 0-3 = that configuration (3 where it applies)
int phpc_f32_set_plan_config(int id);
int phpc_f32_pick_plan_config(const struct F32Desc *descs, int ndesc);
// FP32 configuration ids: 0-2 register-staged (64x64, 128x64, 128x128); kF32DirectConfig the
// direct kernels, whose tile shape follows from the work.
constexpr int kF32DirectConfig = 3;
// the descriptors fit the direct kernels' 32-bit buffer offsets
bool phpc_f32_direct_ok(const F32Desc *descs, int ndesc);
// A launch of the direct FP32 kernels: as F64Work
struct F32Work {
  int config = 0;
  int total = 0, tail_start = 0;
  std::vector<F32Desc> descs;
  std::vector<char> list;
};
int phpc_f32_prepare(const F32Desc *descs, int ndesc, F32Work *w);
int phpc_f32_launch_direct(const F32Work &w, const void *list_dev, int grid, hipStream_t stream);
bool phpc_f32_vec4_ok(const F32Desc *descs, int ndesc);

// FP32-accurate products on BF16 slice planes (3 x BF16, gemm_bf3.hip): one kernel cuts every
// distinct operand into planes, one launch multiplies. Every output is summed in the same order
// whatever the tile and whether alone or in a plan, so results are the same bits. Plan
// configurations kF32X3PlanesConfig + g, g < phpc_bf3_num_configs(), select the tile.
constexpr int kF32X3PlanesConfig = 4;
int phpc_bf3_num_configs();
bool phpc_bf3_fits(long k);  // a plane row of k fits the kernel's 32-bit offsets
size_t phpc_bf3_plane_bytes(long rows, long k);  // of one operand's planes
// configuration of 3 x BF16 plans created without autotuning: -1 = by work, 2 (the in-register
// kernel) or kF32X3PlanesConfig + g
int phpc_f32x3_set_plan_config(int id);
int phpc_f32x3_pick_plan_config(const F32Desc *descs, int ndesc);
struct Bf3Cut {  // one operand's planes
  const float *src;
  long ld;
  int rows, cols;  // source shape: A is m x k, B is k x n
  char *dst;
  int is_b;        // B: plane rows are its columns
  int tiles_k;     // workgroups across k
  int block_start; // first workgroup of the batched kernel on this cut
};
struct Bf3Desc {  // one GEMM on planes
  const char *A;
  const char *B;
  float *C;
  long lda, ldb, ldc;  // planes: bytes per plane row
  int m, n, k;         // k: in blocks
  int tiles_n;
  int tile_start;
};
struct Bf3Work {  // as F64Work
  int config = 0;
  int total = 0, tail_start = 0;
  std::vector<Bf3Desc> descs;
  std::vector<char> list;
};
struct Bf3Planes {
  std::vector<Bf3Cut> cuts;
  std::vector<int> block_cut;   // the cut of each workgroup of the batched kernel
  Bf3Work work;
  void *ws = nullptr;   // the planes
  void *list = nullptr; // cuts, block_cut and the launch's list on the device
  // plans the cuts and tiles of descs for tile g, allocates the planes and uploads the
  // lists (synchronously); PHPC_ERR_ARG when a plane row is too long for the kernel's
  // 32-bit offsets
  int build(const F32Desc *descs, int ndesc, int g);
  // the cut kernel, then the product kernel; grid 0 = a workgroup per tile
  int run(hipStream_t stream, int grid) const;
  void release();
  Bf3Planes() = default;
  Bf3Planes(const Bf3Planes &) = delete;
  Bf3Planes &operator=(const Bf3Planes &) = delete;
  ~Bf3Planes() { release(); }
};

bool phpc_f32x3_planes_pay(const F32Desc &d);
bool phpc_f32x3_in_register_ok(const F32Desc &d);  // its 32-bit buffer offsets reach A's and B's rows
// Launches of the in-register 3 x BF16 kernel: the first `head` GEMMs on the tiles of config[0] (0:
// 64x64, 2: 128x128), the rest in a second launch on those of config[1]. One GEMM travels with its
// launch; otherwise the caller holds a copy of descs on the device.
struct F32X3Work {
  std::vector<F32Desc> descs;
  int head = 0;
  int config[2] = {}, tiles[2] = {};
  bool vec4 = false;
};
void phpc_f32x3_prepare(const F32Desc *descs, int ndesc, F32X3Work *w);
int phpc_f32x3_launch(const F32X3Work &w, const F32Desc *descs_dev, int grid, hipStream_t stream);
int phpc_f32_launch(const F32Desc *descs_dev, const F32Desc *descs_host, int ndesc, int total_tiles, int id, bool vec4,
                    int grid, hipStream_t stream);

bool phpc_f64_config_panels(int id);

// Kernel-level tile configuration chosen by the planner / autotuner.
struct F64Config {
  int id;         // index into the instantiated kernel table
  int bm, bn;     // macro tile
  int threads;    // workgroup size
  int wg_per_cu;  // resident workgroups per CU the config is built for
};

// Launch policy knobs (see phpc_set_launch_policy in phpc_gemm.h).
struct LaunchPolicy {
  int honor_grid;     // 1: persistent grid = caller's grid_width * grid_height
  int config_id;      // -1: autotuned
  int grid_override;  // >0: persistent grid size
};
LaunchPolicy &phpc_policy();

// Device properties cached per process (one GPU).
struct DeviceInfo {
  int device;
  int cus;
  int xcds;
  size_t lds_per_cu;
};
const DeviceInfo &phpc_device();

// Grouped FP64 launch. Descriptors that do not travel with the launch are copied into a
// library-owned device buffer (stream-ordered). `grid` <= 0 selects the configuration's own
// workgroup count, config_id < 0 the planner's. Returns PHPC_OK or an error code.
int phpc_f64_grouped(const GemmDesc *descs_host, int ndesc, int grid, int config_id, hipStream_t stream);

// A grouped FP64 launch prepared for one configuration: the GEMMs that hold work, numbered in
// tiles, the ones cut off for the tail's smaller tiles (from tile tail_start on) last; at most
// twice the GEMMs passed in. Where there are more than two, they do not travel with the launch:
// the caller of phpc_f64_launch holds a copy of `list` on the device. device_list: the work
// comes from a caller that keeps it there (a plan, the serving loop), which two tuning knobs
// set apart.
struct F64Work {
  int config = 0;
  bool mp = false, vec2 = false;
  int total = 0, tail_start = 0;
  std::vector<GemmDesc> descs;
  std::vector<char> list;  // empty where the descriptors travel with the launch
};
int phpc_f64_prepare(const GemmDesc *descs, int ndesc, int config_id, bool device_list, F64Work *w);
int phpc_f64_launch(const F64Work &w, const void *list_dev, int grid, hipStream_t stream);
int phpc_f64_num_configs();
F64Config phpc_f64_config(int id);

// Strided block pack: dst[r*ldd + c] = src[r*lds + c] for r < rows, c < cols.
// Host <-> device copies through pinned staging buffers (rows x width bytes, strided).
// h2d returns once the source may be reused (transfers complete in stream order); d2h
// returns once the destination holds the data.
struct StageCopy {
  void *dst;
  size_t dpitch;
  const void *src;
  size_t spitch;
  size_t width, rows;  // bytes per row, rows
};
int phpc_stage_h2d(const StageCopy *copies, int count, hipStream_t stream);
int phpc_stage_d2h(const StageCopy *copies, int count, hipStream_t stream);
inline int phpc_stage_h2d(void *dst, size_t dpitch, const void *src, size_t spitch, size_t width, size_t rows,
                          hipStream_t stream) {
  const StageCopy c{dst, dpitch, src, spitch, width, rows};
  return phpc_stage_h2d(&c, 1, stream);
}
inline int phpc_stage_d2h(void *dst, size_t dpitch, const void *src, size_t spitch, size_t width, size_t rows,
                          hipStream_t stream) {
  const StageCopy c{dst, dpitch, src, spitch, width, rows};
  return phpc_stage_d2h(&c, 1, stream);
}
// Process-wide copy and compute streams of the host-pointer entry points.
int phpc_host_streams(hipStream_t *copy, hipStream_t *compute);
int phpc_pack_launch(const double *src, long lds, double *dst, long ldd, int rows, int cols,
                     hipStream_t stream);

// Scratch device buffer owned by the library (grows; stream-ordered use only).
void *phpc_scratch(size_t bytes, int slot);
// Kernel event timing (phpc_kernel_timing): begin returns a token (-1 when timing is off
// or the stream is capturing); end records the closing event for that token.
int phpc_ktime_begin(hipStream_t stream);
void phpc_ktime_end(int token, hipStream_t stream);

// A set of growable device buffers for one caller at a time (the split path needs four).
// Growing synchronises `stream` before the old buffer is freed.
struct Workspace {
  static constexpr int kSlots = 8;
  void *p[kSlots] = {};
  size_t cap[kSlots] = {};
  // Fixed region (set by use_fixed): get() allocates nothing and instead carves each
  // slot, in call order, out of [fixed, fixed + fixed_size) at 256-byte aligned offsets,
  // returning nullptr once the region is exhausted; release() frees nothing.
  char *fixed = nullptr;
  size_t fixed_size = 0, fixed_used = 0;
  void use_fixed(void *base, size_t size);
  void *get(size_t bytes, int slot, hipStream_t stream);
  size_t total() const;
  void release();
  ~Workspace() { release(); }
};

// A workspace shared by calls that may come on different streams: the holder of the
// lock orders its stream after the previous holder's last use (device-side wait), and
// marks its own last use before unlocking.
struct SharedWorkspace {
  std::mutex mu;
  Workspace ws;
  hipEvent_t last = nullptr;
  void after_previous(hipStream_t stream) {
    if (last) (void)hipStreamWaitEvent(stream, last, 0);
  }
  void mark_used(hipStream_t stream) {
    if (!last) (void)hipEventCreateWithFlags(&last, hipEventDisableTiming);
    if (last) (void)hipEventRecord(last, stream);
  }
};

// Bytes of k per residue / slice plane row of the split GEMM: k rounded up to 128, so
// that every level range is a whole number of the level kernels' k slabs (64 or 128
// bytes) and the 16-byte direct-to-LDS loads never straddle a plane.
inline long phpc_split_kp(long k) { return (k + 127) / 128 * 128; }

#include "phpc_split.h"
// Split-precision GEMM with an explicit workspace and method (the public entry point
// uses a process-wide workspace and the method set by phpc_split_set_method).
// FP32-accurate 3 x BF16 GEMM through BF16 slice planes (workspace slots 0 and 1).
int phpc_sgemm_bf16x3_planes(const float *dA, long lda, const float *dB, long ldb, float *dC, long ldc, int m, int k,
                             int n, hipStream_t s, Workspace *ws);
// Residue operands of the CRT split GEMM, rows x kp bytes per modulus (kp a multiple of 64, rows
// those of A or the columns of B): 16 rows at a time, and of these 64 k at a time, so that a load
// of the product's is one contiguous KiB. The last rows lie as close together as there are of
// them: no padding, modulus t's operand is rows * kp bytes.
__host__ __device__ inline long crt_offset(int t, int rows, long kp, int r, long k) {
  const int r0 = r / 16 * 16, held = rows - r0 < 16 ? rows - r0 : 16;
  return ((long)t * rows + r0) * kp + k / 64 * (held * 64) + (r - r0) * 64 + k % 64;
}
// Residue products: res plane t (m x n bytes, row-major) = A_t B_t mod mods[t].
int phpc_crt_level(const int8_t *A8, const int8_t *B8, long kp, int m, int n, int L, const int *mods, int8_t *res,
                   hipStream_t s);
int phpc_dgemm_split_ws(const double *dA, long lda, const double *dB, long ldb, double *dC, long ldc, int m, int k,
                        int n, int slices, double target_err, int method, hipStream_t stream, Workspace *ws,
                        phpc_split_info *info);
