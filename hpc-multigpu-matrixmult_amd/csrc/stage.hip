// Host <-> device staging through pinned memory.
//
// The drop-in entry points take pageable host pointers, as the reference's do
// (src/phpc_gemm.cu:59-156). A pageable hipMemcpy goes through the runtime's own
// staging at a fraction of the link rate. Here a small pool of host threads copies
// pieces of rows between the caller's memory and a ring of pinned slots while the DMA
// engine moves the pieces before, so host copies, PCIe transfers and (in the callers)
// kernels overlap. All operands of a call go through in one turn of the pool: 1024^3 from
// host matrices (25 MB in, 8 MB out, 590 us at the link's rate) 1115 us with one 32 MiB chunk
// per operand, copied whole before its transfer, 960 now (512^3 510 -> 355, 2048^3 3.9 -> 3.4 ms).
#include "phpc_internal.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

namespace {

// Parallel for over [0, n) with a fixed set of worker threads; the caller participates.
class CopyPool {
 public:
  explicit CopyPool(int nthreads) {
    for (int i = 0; i < nthreads; ++i) th_.emplace_back([this] { work(); });
  }
  ~CopyPool() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_ = true;
    }
    cv_.notify_all();
    for (auto &t : th_) t.join();
  }
  void run(int n, const std::function<void(int)> &fn) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      fn_ = &fn;
      n_ = n;
      next_ = 0;
      left_ = n;
      ++gen_;
    }
    cv_.notify_all();
    drain();
    std::unique_lock<std::mutex> lk(mu_);
    done_.wait(lk, [&] { return left_ == 0; });
    fn_ = nullptr;
  }

 private:
  void drain() {
    for (;;) {
      int i;
      const std::function<void(int)> *fn;
      {
        std::lock_guard<std::mutex> lk(mu_);
        if (!fn_ || next_ >= n_) return;
        i = next_++;
        fn = fn_;
      }
      (*fn)(i);
      std::lock_guard<std::mutex> lk(mu_);
      if (--left_ == 0) done_.notify_all();
    }
  }
  void work() {
    uint64_t seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> lk(mu_);
        cv_.wait(lk, [&] { return stop_ || gen_ != seen; });
        if (stop_) return;
        seen = gen_;
      }
      drain();
    }
  }
  std::vector<std::thread> th_;
  std::mutex mu_;
  std::condition_variable cv_, done_;
  const std::function<void(int)> *fn_ = nullptr;
  int n_ = 0, next_ = 0, left_ = 0;
  uint64_t gen_ = 0;
  bool stop_ = false;
};

// Pinned memory: kBuffers buffers, cut into slots of a piece each. A piece is about kPieceBytes
// of whole rows, kLargePieceBytes from kLarge bytes on: one transfer (each costs some 15 us
// beside its bytes: 1024^3 in pieces of 1 MiB 1120 us, of 2 MiB 940, of 8 MiB 1070). The host
// copies it in parts of about kPartBytes, so that all threads work on the first piece and its
// transfer starts after a part's time, not a piece's. Transfers alternate between kLanes streams,
// so that one starts under another (940 us, 1030 on one stream, 1020 on four); copies of a
// piece's size in all stay on the caller's stream, which takes no events.
constexpr int kBuffers = 4;
constexpr size_t kBufferBytes = 32u << 20;
constexpr size_t kPieceBytes = 2u << 20, kPartBytes = 256u << 10;
constexpr size_t kLarge = 64u << 20, kLargePieceBytes = 32u << 20;
constexpr int kMaxSlots = (int)(kBuffers * (kBufferBytes / kPieceBytes));

constexpr int kLanes = 2;

struct Stager {
  std::mutex mu;  // one staged copy at a time
  bool ready = false;
  char *buffer[kBuffers] = {};
  hipEvent_t done[kMaxSlots] = {};
  hipStream_t lane[kLanes] = {};
  hipEvent_t before = nullptr, after[kLanes] = {};
  size_t slot_bytes = 0;  // of the transfers that may still be under way
  CopyPool *pool = nullptr;

  int init() {
    if (ready) return PHPC_OK;
    for (char *&b : buffer)
      if (!b && hipHostMalloc((void **)&b, kBufferBytes, hipHostMallocDefault) != hipSuccess) {
        b = nullptr;
        return phpc_set_error(PHPC_ERR_MEM, "pinned staging allocation failed");
      }
    for (hipEvent_t &e : done)
      if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        e = nullptr;
        return phpc_set_error(PHPC_ERR_HIP, "staging event creation failed");
      }
    for (hipStream_t &l : lane)
      if (!l && hipStreamCreateWithFlags(&l, hipStreamNonBlocking) != hipSuccess) {
        l = nullptr;
        return phpc_set_error(PHPC_ERR_HIP, "staging stream creation failed");
      }
    for (hipEvent_t *e : {&before, &after[0], &after[1]})
      if (!*e && hipEventCreateWithFlags(e, hipEventDisableTiming) != hipSuccess) {
        *e = nullptr;
        return phpc_set_error(PHPC_ERR_HIP, "staging event creation failed");
      }
    if (!pool) {
      const unsigned hw = std::thread::hardware_concurrency();
      pool = new CopyPool((int)std::min(7u, hw > 1 ? hw - 1 : 1u));
    }
    ready = true;
    return PHPC_OK;
  }
  // slots of `bytes` from here on, once no transfer uses the old ones
  int use_slots(size_t bytes) {
    if (bytes == slot_bytes) return PHPC_OK;
    for (hipEvent_t e : done) PHPC_HIP(hipEventSynchronize(e));
    slot_bytes = bytes;
    return PHPC_OK;
  }
  int slots() const { return (int)std::min<size_t>(kMaxSlots, kBuffers * (kBufferBytes / slot_bytes)); }
  char *slot(int i) const {
    const int per = (int)(kBufferBytes / slot_bytes);
    return buffer[i / per] + (size_t)(i % per) * slot_bytes;
  }
};
Stager g_stage;

// A piece: rows [r0, r0 + rows) of a copy
struct Piece {
  const StageCopy *c;
  size_t r0, rows;
};

void copy_rows(char *dst, size_t dpitch, const char *src, size_t spitch, size_t width, size_t rows) {
  if (dpitch == width && spitch == width) {
    memcpy(dst, src, width * rows);
    return;
  }
  for (size_t r = 0; r < rows; ++r) memcpy(dst + r * dpitch, src + r * spitch, width);
}

// one piece's transfer between its slot and the device
hipError_t transfer(const Piece &p, char *slot, bool in, hipStream_t s) {
  const StageCopy &c = *p.c;
  char *dev = in ? (char *)c.dst + p.r0 * c.dpitch : (char *)c.src + p.r0 * c.spitch;
  const size_t pitch = in ? c.dpitch : c.spitch;
  const hipMemcpyKind kind = in ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost;
  void *dst = in ? dev : slot, *src = in ? slot : dev;
  if (pitch == c.width) return hipMemcpyAsync(dst, src, c.width * p.rows, kind, s);
  return hipMemcpy2DAsync(dst, in ? pitch : c.width, src, in ? c.width : pitch, c.width, p.rows, kind, s);
}

// The copies' pieces through the slots in order: into the device (in) the host fills a slot and
// its last part's thread starts the transfer; out of it a part waits for its piece's transfer,
// and the last part out of a slot starts the transfer of the piece that takes it next.
int stage(const StageCopy *copies, int count, bool in, hipStream_t stream) {
  std::lock_guard<std::mutex> lk(g_stage.mu);
  if (int rc = g_stage.init()) return rc;
  size_t widest = 1, total = 0;
  for (int i = 0; i < count; ++i) total += copies[i].width * copies[i].rows;
  const size_t piece_bytes = total >= kLarge ? kLargePieceBytes : kPieceBytes;
  const bool lanes = total > kPieceBytes;
  std::vector<Piece> pieces;
  for (int i = 0; i < count; ++i) {
    const StageCopy &c = copies[i];
    if (c.rows == 0 || c.width == 0) continue;
    if (c.width > kBufferBytes) {  // a row longer than a buffer: let the runtime stage it
      PHPC_HIP(hipMemcpy2DAsync(c.dst, c.dpitch, c.src, c.spitch, c.width, c.rows,
                                in ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, stream));
      PHPC_HIP(hipStreamSynchronize(stream));
      continue;
    }
    widest = std::max(widest, c.width);
    const size_t per = std::max<size_t>(1, piece_bytes / c.width);
    for (size_t r = 0; r < c.rows; r += per) pieces.push_back({&c, r, std::min(per, c.rows - r)});
  }
  if (pieces.empty()) return PHPC_OK;
  if (int rc = g_stage.use_slots(std::max(piece_bytes, (widest + 4095) / 4096 * 4096))) return rc;
  const int np = (int)pieces.size(), ns = g_stage.slots();

  std::vector<int> part_piece, first_part(np);
  std::vector<std::pair<size_t, size_t>> part_rows;
  for (int p = 0; p < np; ++p) {
    first_part[p] = (int)part_piece.size();
    const size_t per = std::max<size_t>(1, (total >= kLarge ? 4 : 1) * kPartBytes / pieces[p].c->width);
    for (size_t r = 0; r < pieces[p].rows; r += per) {
      part_piece.push_back(p);
      part_rows.push_back({r, std::min(per, pieces[p].rows - r)});
    }
  }
  const int nparts = (int)part_piece.size();
  std::vector<std::atomic<int>> left(np), started(np);
  for (int p = 0; p < np; ++p) {
    left[p] = (p + 1 < np ? first_part[p + 1] : nparts) - first_part[p];
    started[p] = 0;
  }
  std::atomic<int> failed{(int)hipSuccess};
  auto note = [&](hipError_t e) {
    int none = (int)hipSuccess;
    if (e != hipSuccess) failed.compare_exchange_strong(none, (int)e);
  };
  auto start = [&](int p) {
    hipStream_t s = lanes ? g_stage.lane[p % kLanes] : stream;
    hipError_t e = transfer(pieces[p], g_stage.slot(p % ns), in, s);
    if (e == hipSuccess) e = hipEventRecord(g_stage.done[p % ns], s);
    note(e);
    started[p].store(1, std::memory_order_release);
  };
  // once the transfer of piece p has been started and is done
  auto wait = [&](int p) {
    while (!started[p].load(std::memory_order_acquire)) std::this_thread::yield();
    note(hipEventSynchronize(g_stage.done[p % ns]));
  };
  if (lanes) {  // they follow what is queued on stream
    PHPC_HIP(hipEventRecord(g_stage.before, stream));
    for (hipStream_t l : g_stage.lane) PHPC_HIP(hipStreamWaitEvent(l, g_stage.before, 0));
  }
  if (!in) {
    for (int p = 0; p < std::min(np, ns); ++p) {
      // the slot's last transfer, of an earlier call, is done before it is overwritten
      note(hipEventSynchronize(g_stage.done[p % ns]));
      start(p);
    }
  }
  const std::function<void(int)> part = [&](int i) {
    const int p = part_piece[i];
    const StageCopy &c = *pieces[p].c;
    const size_t r = part_rows[i].first, n = part_rows[i].second, at = pieces[p].r0 + r;
    char *slot = g_stage.slot(p % ns) + r * c.width;
    if (in) {
      if (p >= ns)
        wait(p - ns);
      else
        note(hipEventSynchronize(g_stage.done[p]));
      copy_rows(slot, c.width, (const char *)c.src + at * c.spitch, c.spitch, c.width, n);
      if (left[p].fetch_sub(1) == 1) start(p);
    } else {
      wait(p);
      copy_rows((char *)c.dst + at * c.dpitch, c.dpitch, slot, c.width, c.width, n);
      if (left[p].fetch_sub(1) == 1 && p + ns < np) start(p + ns);
    }
  };
  if (nparts == 1)
    part(0);
  else
    g_stage.pool->run(nparts, part);
  for (int l = 0; l < (lanes ? kLanes : 0); ++l) {
    note(hipEventRecord(g_stage.after[l], g_stage.lane[l]));
    note(hipStreamWaitEvent(stream, g_stage.after[l], 0));
  }
  if (failed.load() != (int)hipSuccess)
    return phpc_set_error(PHPC_ERR_HIP, "staged copy failed: %s", hipGetErrorString((hipError_t)failed.load()));
  return PHPC_OK;
}

}  // namespace

// Host -> device copies, on stream. Returns once the sources may be reused; the transfers
// complete in stream order.
int phpc_stage_h2d(const StageCopy *copies, int count, hipStream_t stream) { return stage(copies, count, true, stream); }

// Device -> host copies, after the work already queued on stream. Returns once the
// destinations hold the data.
int phpc_stage_d2h(const StageCopy *copies, int count, hipStream_t stream) {
  return stage(copies, count, false, stream);
}
