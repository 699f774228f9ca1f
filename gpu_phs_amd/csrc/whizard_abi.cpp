// The Whizard-facing C ABI (include/gpu_phs.h group 1): the reference's 14 c_whizard_* entry
// points with the same signatures and index conventions (whizard_gpu_phs.cpp:12-249), on top
// of the process/plan machinery of phs_api.cpp.  The reference keeps its state in process
// globals (global_phs.cpp:6-27, phs.cu:27-41); this file keeps the equivalent in one static
// module object, so the calls keep their order-dependent semantics.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "phs_state.h"

namespace gphs {
namespace {

// Host copies go through a ring of pinned slots in chunks of one slot, to the host on two streams in turn.
// Large chunks keep the link busy (32 MiB to the host, one stream and two: 2 MiB chunks 41 and 46 GB/s, 4 MiB 48
// and 50, 8 MiB 52 and 53), small ones start the first DMA and end the last host copy early (a call of
// 10^5 2 -> 4 events on one stream: 1.40 ms at 2 MiB, 1.27 at 4, 1.40 at 8).  A second stream for the smaller
// transfers to the device gained another 0.04 ms, but cost two more calls of 7-14 ms at the start of a process.
//
// From kOneStream bytes on, transfers to the host take one stream and chunks of two slots: in a process that has
// used other streams the copy engines that the runtime gives to two streams made every second of the first ten
// calls of 10^6 events take 13.4 ms, the others 9.7, before they settled at 9.0; one stream takes 9.4 from the
// first.  (Below, two streams take 208 us for 1,818 2 -> 6 events, 1.06 and 2.85 ms for 10^5 and 3 x 10^5 of
// 2 -> 4, also beside others; one stream with chunks of two slots 226 us, 1.13 and 2.92.)
constexpr int kPinSlots = 8;
constexpr size_t kPinChunk = (size_t)4 << 20;
constexpr size_t kOneStream = (size_t)128 << 20;

struct WhizardModule {
  int n_channels = 0, n_in = 0, n_out = 0, n_x = 0;
  bool sized = false, maps_ready = false, trees_ready = false, initialized = false;
  ProcessSpec spec;                 // trees and maps as filled
  // from c_whizard_init_channel_ids: the channel of events [end of the previous run, end)
  struct Run { int channel; int64_t end; };
  std::vector<Run> runs;
  int block = 256;
  // compiled process for the current beams
  int process = -1;
  double E1 = -1, E2 = -1;
  // device buffers kept between calls (grow-only)
  double* x_d = nullptr; double* p_d = nullptr; double* f_d = nullptr; double* v_d = nullptr;
  double* e_d = nullptr;             // beam energies of the last call: E1 [n], then E2 [n] (phs.cu:1361-1363)
  size_t last_n = 0;                 // events of the last generate call
  uint8_t* ok_d = nullptr;
  size_t cap = 0;                   // events the buffers hold
  int cap_nx = 0, cap_nout = 0;
  // inverse mapping outputs: factors [n][n_channels], randoms [n_channels][n][n_x]
  double* fa_d = nullptr; double* xo_d = nullptr;
  size_t inv_cap = 0;               // doubles of xo_d
  double* last_p = nullptr;         // device momenta of the last generate call
  // the plan of the last call, reused (tables, inverse tables) while its segments repeat
  std::unique_ptr<PlanObj> plan;
  std::vector<gpu_phs_segment> plan_segs;
  bool plan_varying = false;
  // the module's own streams (non-blocking, default priority): kernels and most chunks, and odd chunks to the host
  hipStream_t stream = nullptr, stream2 = nullptr;
  hipEvent_t kernels_ev = nullptr;
  // pinned staging of the host copies: a ring of slots, one chunk each (transfer below)
  char* pin = nullptr;
  hipEvent_t pin_ev[kPinSlots] = {};   // the slot's last DMA
};

WhizardModule& W() {
  static WhizardModule w;
  return w;
}

void free_buffers(WhizardModule& w) {
  w.plan.reset();   // its segments point into the buffers
  w.plan_segs.clear();
  (void)hipFree(w.x_d); (void)hipFree(w.p_d); (void)hipFree(w.f_d); (void)hipFree(w.v_d); (void)hipFree(w.ok_d);
  (void)hipFree(w.fa_d); (void)hipFree(w.xo_d); (void)hipFree(w.e_d);
  w.x_d = w.p_d = w.f_d = w.v_d = nullptr;
  w.fa_d = w.xo_d = w.e_d = nullptr;
  w.last_n = 0;
  w.ok_d = nullptr;
  w.cap = 0;
  w.inv_cap = 0;
  w.last_p = nullptr;
}

int ensure_buffers(WhizardModule& w, size_t n) {
  if (n <= w.cap && w.cap_nx == w.n_x && w.cap_nout == w.n_out) return GPU_PHS_OK;
  free_buffers(w);
  hipError_t e;
  if ((e = hipMalloc(&w.x_d, n * w.n_x * sizeof(double))) != hipSuccess ||
      (e = hipMalloc(&w.p_d, n * w.n_out * 4 * sizeof(double))) != hipSuccess ||
      (e = hipMalloc(&w.f_d, n * sizeof(double))) != hipSuccess ||
      (e = hipMalloc(&w.v_d, n * sizeof(double))) != hipSuccess ||
      (e = hipMalloc(&w.e_d, 2 * n * sizeof(double))) != hipSuccess ||
      (e = hipMalloc(&w.ok_d, n)) != hipSuccess) {
    free_buffers(w);
    return hip_error(e, "hipMalloc(event buffers)");
  }
  w.cap = n; w.cap_nx = w.n_x; w.cap_nout = w.n_out;
  return GPU_PHS_OK;
}

int ensure_inverse_buffers(WhizardModule& w, size_t n) {
  const size_t need = n * w.n_channels * w.n_x;
  if (need <= w.inv_cap && w.fa_d) return GPU_PHS_OK;
  (void)hipFree(w.fa_d); (void)hipFree(w.xo_d);
  w.fa_d = w.xo_d = nullptr;
  w.inv_cap = 0;
  hipError_t e;
  if ((e = hipMalloc(&w.fa_d, n * w.n_channels * sizeof(double))) != hipSuccess ||
      (e = hipMalloc(&w.xo_d, std::max<size_t>(need, 1) * sizeof(double))) != hipSuccess) {
    (void)hipFree(w.fa_d); w.fa_d = nullptr;
    return hip_error(e, "hipMalloc(inverse buffers)");
  }
  w.inv_cap = need;
  return GPU_PHS_OK;
}

void free_staging(WhizardModule& w) {
  // both streams copy from and to the ring
  if (w.stream) (void)hipStreamSynchronize(w.stream);
  if (w.stream2) (void)hipStreamSynchronize(w.stream2);
  for (hipEvent_t& ev : w.pin_ev) {
    if (ev) (void)hipEventDestroy(ev);
    ev = nullptr;
  }
  if (w.pin) (void)hipHostFree(w.pin);
  w.pin = nullptr;
  if (w.kernels_ev) (void)hipEventDestroy(w.kernels_ev);
  if (w.stream2) (void)hipStreamDestroy(w.stream2);
  if (w.stream) (void)hipStreamDestroy(w.stream);
  w.stream = w.stream2 = nullptr;
  w.kernels_ev = nullptr;
}

// The transfers of a few calls, so that the runtime sets up here, in c_whizard_init_gpu_phs, what it otherwise does
// in the middle of the first calls: the streams' queues (3 ms each), and a copy engine (5-7 ms) whenever one
// is first used, by the second stream or because the ones in use are busy.  A process's first call of
// 10^5 2 -> 4 events takes 13 ms, as before the second stream (32 without this), and the ones after it 1.1 (one
// of the first ten 7 ms without this).
hipError_t warm_up(WhizardModule& w) {
  char* dev = nullptr;
  hipError_t e = hipMalloc(&dev, kPinChunk);
  for (int call = 0; call < 3 && e == hipSuccess; call++) {
    for (int k = 0; k < 2 && e == hipSuccess; k++)
      e = hipMemcpyAsync(dev, w.pin + k * kPinChunk, kPinChunk, hipMemcpyHostToDevice, w.stream);
    if (e == hipSuccess) e = hipEventRecord(w.kernels_ev, w.stream);
    if (e == hipSuccess) e = hipStreamWaitEvent(w.stream2, w.kernels_ev, 0);
    for (int k = 0; k < kPinSlots && e == hipSuccess; k++) {
      hipStream_t st = k % 2 ? w.stream2 : w.stream;
      if ((e = hipMemcpyAsync(w.pin + k * kPinChunk, dev, kPinChunk, hipMemcpyDeviceToHost, st)) == hipSuccess)
        e = hipEventRecord(w.pin_ev[k], st);
    }
    const hipError_t e1 = hipStreamSynchronize(w.stream), e2 = hipStreamSynchronize(w.stream2);
    if (e == hipSuccess) e = e1 != hipSuccess ? e1 : e2;
  }
  (void)hipFree(dev);
  return e;
}

int ensure_staging(WhizardModule& w) {
  if (w.stream) return GPU_PHS_OK;
  hipError_t e = hipStreamCreateWithFlags(&w.stream, hipStreamNonBlocking);
  if (e != hipSuccess) { w.stream = nullptr; return hip_error(e, "hipStreamCreate"); }
  if ((e = hipStreamCreateWithFlags(&w.stream2, hipStreamNonBlocking)) == hipSuccess &&
      (e = hipEventCreateWithFlags(&w.kernels_ev, hipEventDisableTiming)) == hipSuccess)
    e = hipHostMalloc((void**)&w.pin, kPinSlots * kPinChunk, hipHostMallocDefault);
  for (int k = 0; k < kPinSlots && e == hipSuccess; k++)
    e = hipEventCreateWithFlags(&w.pin_ev[k], hipEventDisableTiming);
  if (e == hipSuccess) e = warm_up(w);
  if (e != hipSuccess) {
    free_staging(w);
    return hip_error(e, "pinned staging buffers");
  }
  return GPU_PHS_OK;
}

// Threads that copy between pinned and pageable memory beside the calling one: started at the first large
// transfer and kept until the library is unloaded.  One thread copies some 10-15 GB/s, well below what
// PCIe moves (a call of 10^5 2 -> 4 events with four threads 1.10 ms, with five 1.07, with seven 1.06 and a quarter
// more processor time).
constexpr int kCopyThreads = 5;
class CopyPool {
 public:
  // Runs `job` on every thread, until wait(); the number of threads (0 if none can be started).
  int start(const std::function<void()>& job) {
    std::lock_guard<std::mutex> lk(m_);
    try {
      while ((int)th_.size() < kCopyThreads) th_.emplace_back([this, seen = gen_] { worker(seen); });
    } catch (const std::system_error&) {   // with as many as there are
    }
    job_ = &job;
    pending_ = (int)th_.size();
    gen_++;
    work_.notify_all();
    return (int)th_.size();
  }
  void wait() {
    std::unique_lock<std::mutex> lk(m_);
    done_.wait(lk, [&] { return pending_ == 0; });
  }
  ~CopyPool() {
    {
      std::lock_guard<std::mutex> lk(m_);
      stop_ = true;
    }
    work_.notify_all();
    for (auto& t : th_) t.join();
  }

 private:
  void worker(uint64_t seen) {
    for (;;) {
      const std::function<void()>* job;
      {
        std::unique_lock<std::mutex> lk(m_);
        work_.wait(lk, [&] { return stop_ || gen_ != seen; });
        if (stop_) return;
        seen = gen_;
        job = job_;
      }
      (*job)();
      std::lock_guard<std::mutex> lk(m_);
      if (--pending_ == 0) done_.notify_one();
    }
  }
  std::vector<std::thread> th_;
  std::mutex m_;
  std::condition_variable work_, done_;
  const std::function<void()>* job_ = nullptr;
  int pending_ = 0;
  uint64_t gen_ = 0;
  bool stop_ = false;
};

CopyPool& copy_pool() {
  static CopyPool pool;
  return pool;
}

// A condition that other threads bring about and announce with changed(): waited for asleep after kAwake, about the
// time from one chunk to the next, so that the copy threads take nothing from the host program while the
// kernels run or the link is slow.  Calls of 1,818 2 -> 6, 10^5 and 10^6 2 -> 4 events, time and processor time:
// 208 us and 0.82 ms, 1.07 and 4.9 ms, 8.9 and 48 ms; with seven threads that only wait actively 209 us and 1.2 ms,
// 1.07 and 7.9 ms, 9.0 and 68 ms; asleep after 20 us 218 us and 0.74 ms, 1.06 and 4.7 ms, 9.2 and 50 ms.
constexpr std::chrono::microseconds kAwake{100};
class Waiting {
 public:
  template <class Done>
  void until(Done done) {
    const auto end = std::chrono::steady_clock::now() + kAwake;
    do {
      for (int k = 0; k < 32; k++) {
        if (done()) return;
        __builtin_ia32_pause();
      }
    } while (std::chrono::steady_clock::now() < end);
    std::unique_lock<std::mutex> lk(m_);
    cv_.wait(lk, done);
  }
  void changed() {
    { std::lock_guard<std::mutex> lk(m_); }   // whoever has found the condition false sleeps by now
    cv_.notify_all();
  }

 private:
  std::mutex m_;
  std::condition_variable cv_;
};

struct Transfer {
  void* host;
  void* dev;
  size_t n;
};

// Copies the list between the caller's arrays and the device, on the module's stream.  The calling thread
// issues the DMAs, ahead as far as the ring allows, while the pool copies in pieces between the slots and
// the caller's memory: a call of 10^5 2 -> 4 events (8 MB in, 35 MB out) takes 1.10 ms, 1.47 array by array
// with two slots of 16 MiB, whose copies waited for one another wherever an array was a single chunk.
// To the device: returns when every DMA is queued.  To the host: when all has arrived.
int transfer(WhizardModule& w, const std::vector<Transfer>& list, bool to_device) {
  constexpr size_t kPiece = (size_t)256 << 10, kPoolBytes = (size_t)1 << 20;
  struct Chunk {
    char* host;
    char* dev;
    size_t n;
  };
  std::vector<Chunk> chunks;
  size_t total = 0;
  for (const Transfer& t : list) total += t.n;
  const bool large = !to_device && total >= kOneStream, one_stream = to_device || large;
  const size_t chunk = large ? 2 * kPinChunk : kPinChunk;
  const int slots = (int)(kPinSlots * kPinChunk / chunk), pieces_of = (int)(chunk / kPiece);
  for (const Transfer& t : list)
    for (size_t off = 0; off < t.n; off += chunk)
      chunks.push_back(Chunk{(char*)t.host + off, (char*)t.dev + off, std::min(chunk, t.n - off)});
  const int n = (int)chunks.size();
  auto slot = [&](int c) { return w.pin + (size_t)(c % slots) * chunk; };
  auto host_copy = [&](int c, size_t off, size_t bytes) {
    char* pinned = slot(c) + off;
    char* user = chunks[c].host + off;
    if (to_device) std::memcpy(pinned, user, bytes);
    else std::memcpy(user, pinned, bytes);
  };
  auto dma = [&](int c) -> hipError_t {
    const Chunk& k = chunks[c];
    hipStream_t st = c % 2 && !one_stream ? w.stream2 : w.stream;
    hipError_t e = to_device ? hipMemcpyAsync(k.dev, slot(c), k.n, hipMemcpyHostToDevice, st)
                             : hipMemcpyAsync(slot(c), k.dev, k.n, hipMemcpyDeviceToHost, st);
    return e != hipSuccess ? e : hipEventRecord(w.pin_ev[c % slots], st);
  };
  auto arrived = [&](int c) { return hipEventSynchronize(w.pin_ev[c % slots]); };
  // no DMA on the slots or the device arrays goes on after a transfer that failed
  auto failed = [&](hipError_t e, const char* what) {
    (void)hipStreamSynchronize(w.stream);
    (void)hipStreamSynchronize(w.stream2);
    return hip_error(e, what);
  };

  // pieces [pieces_of c, pieces_of (c + 1)) are chunk c's (those past its end are empty); `open` chunks may be
  // copied so far: arrived from the device, or with a free slot
  std::unique_ptr<std::atomic<int>[]> left(new std::atomic<int>[n > 0 ? n : 1]);
  for (int c = 0; c < n; c++) left[c].store(pieces_of, std::memory_order_relaxed);
  std::atomic<int> next{0}, open{to_device ? std::min(n, slots) : 0};
  std::atomic<bool> abort{false};
  Waiting for_open, for_copied;
  auto open_to = [&](int c) {
    open.store(c, std::memory_order_release);
    for_open.changed();
  };
  const std::function<void()> pieces = [&] {
    for (;;) {
      const int q = next.fetch_add(1, std::memory_order_relaxed), c = q / pieces_of;
      if (c >= n) return;
      for_open.until([&] { return open.load(std::memory_order_acquire) > c || abort.load(std::memory_order_relaxed); });
      if (abort.load(std::memory_order_relaxed)) return;
      const size_t off = (size_t)(q % pieces_of) * kPiece;
      if (off < chunks[c].n) host_copy(c, off, std::min(kPiece, chunks[c].n - off));
      if (left[c].fetch_sub(1, std::memory_order_release) == 1) for_copied.changed();
    }
  };
  auto copied = [&](int c) { return left[c].load(std::memory_order_acquire) == 0; };

  hipError_t e = hipSuccess;
  // the slots' DMAs of the previous transfer; to the host, the other stream follows the kernels
  for (int c = 0; to_device && c < std::min(n, slots) && e == hipSuccess; c++) e = arrived(c);
  if (!to_device && (e = hipEventRecord(w.kernels_ev, w.stream)) == hipSuccess && !one_stream)
    e = hipStreamWaitEvent(w.stream2, w.kernels_ev, 0);
  if (e != hipSuccess) return failed(e, "staging events");
  int threads = 0;
  auto start = [&] { threads = total >= kPoolBytes ? copy_pool().start(pieces) : 0; };
  auto copy_whole = [&](int c) {   // without threads
    if (threads > 0) return;
    host_copy(c, 0, chunks[c].n);
    left[c].store(0, std::memory_order_relaxed);
  };
  if (to_device) {
    start();
    for (int c = 0, freed = 0; c < n && e == hipSuccess; c++) {
      copy_whole(c);
      for_copied.until([&] { return copied(c); });
      e = dma(c);
      // half the ring stays in flight
      for (; e == hipSuccess && freed + slots < n && c - freed >= slots / 2; freed++)
        if ((e = arrived(freed)) == hipSuccess) open_to(freed + slots + 1);
    }
  } else {
    for (int c = 0, issued = 0; c < n && e == hipSuccess; c++) {
      // every chunk whose slot has been copied out; at least this one
      for (; issued < n && issued < c + slots && e == hipSuccess; issued++) {
        if (issued >= slots) {
          if (issued > c && !copied(issued - slots)) break;
          for_copied.until([&] { return copied(issued - slots); });
        }
        e = dma(issued);
      }
      // the threads sleep through the kernels and wake up during the first DMA
      if (c == 0 && e == hipSuccess && (e = hipEventSynchronize(w.kernels_ev)) == hipSuccess) start();
      if (e == hipSuccess) e = arrived(c);
      if (e == hipSuccess) open_to(c + 1);
      if (e == hipSuccess) copy_whole(c);
    }
  }
  if (e != hipSuccess) {
    abort.store(true);
    for_open.changed();
  } else if (threads > 0) {
    pieces();   // of the last chunk, while the threads wake up
  }
  if (threads > 0) copy_pool().wait();
  return e == hipSuccess ? GPU_PHS_OK : failed(e, to_device ? "host to device copy" : "device to host copy");
}

int compile_for_beams(WhizardModule& w, double E1, double E2) {
  if (w.process >= 0 && E1 == w.E1 && E2 == w.E2) return GPU_PHS_OK;
  if (w.process >= 0) { drop_process(w.process); w.process = -1; }
  ProcessSpec sp = w.spec;
  sp.E1 = E1; sp.E2 = E2;
  auto po = std::make_unique<ProcessObj>();
  std::string err = compile_process(sp, po->cp);
  if (!err.empty()) return set_error(GPU_PHS_E_TREE, err);
  w.process = register_process(std::move(po));
  w.E1 = E1; w.E2 = E2;
  return GPU_PHS_OK;
}

}  // namespace
}  // namespace gphs

using namespace gphs;

extern "C" {

void c_whizard_set_particle_structure(int* n_channels, int* n_trees, int* n_groves, int* n_x, int* n_in, int* n_out) {
  std::lock_guard<std::mutex> lk(api_mutex());
  (void)n_trees; (void)n_groves;
  WhizardModule& w = W();
  if (!n_channels || !n_x || !n_in || !n_out || *n_channels < 1 || *n_in != 2 || *n_out < 2 || *n_out > kMaxOut) {
    set_error(GPU_PHS_E_ARG, "set_particle_structure: need n_channels >= 1, n_in = 2, 2 <= n_out <= 12");
    return;
  }
  w.n_channels = *n_channels; w.n_in = *n_in; w.n_out = *n_out; w.n_x = *n_x;
  w.spec = ProcessSpec();
  w.spec.n_in = w.n_in; w.spec.n_out = w.n_out; w.spec.n_channels = w.n_channels;
  w.spec.flv_masses.assign(w.n_in + w.n_out, 0.0);
  w.spec.flv_widths.assign(w.n_in + w.n_out, 0.0);
  w.sized = true; w.maps_ready = w.trees_ready = w.initialized = false;
  if (w.n_x != w.spec.n_x()) {
    set_error(GPU_PHS_E_ARG, "set_particle_structure: n_x must be 3 n_out - 4");
    return;
  }
  ok_status();
}

void c_whizard_set_flavors(double* masses, double* widths) {
  std::lock_guard<std::mutex> lk(api_mutex());
  WhizardModule& w = W();
  if (!w.sized) { set_error(GPU_PHS_E_STATE, "set_flavors before set_particle_structure"); return; }
  for (int i = 0; i < w.n_in + w.n_out; i++) {
    w.spec.flv_masses[i] = masses[i];
    w.spec.flv_widths[i] = widths ? widths[i] : 0.0;
  }
  if (w.process >= 0) { drop_process(w.process); w.process = -1; }
  ok_status();
}

void c_whizard_init_mappings(void) {
  std::lock_guard<std::mutex> lk(api_mutex());
  WhizardModule& w = W();
  if (!w.sized) { set_error(GPU_PHS_E_STATE, "init_mappings before set_particle_structure"); return; }
  size_t n = (size_t)w.n_channels * w.spec.n_prt_out();
  w.spec.map_ids.assign(n, 0);
  w.spec.map_masses.assign(n, 0.0);
  w.spec.map_widths.assign(n, 0.0);
  w.maps_ready = true;
  ok_status();
}

void c_whizard_fill_mapping(int* channel, int* map_ids, double* masses, double* widths) {
  std::lock_guard<std::mutex> lk(api_mutex());
  WhizardModule& w = W();
  if (!w.maps_ready) { set_error(GPU_PHS_E_STATE, "fill_mapping before init_mappings"); return; }
  int c = *channel - 1;  // Fortran -> C index
  if (c < 0 || c >= w.n_channels) { set_error(GPU_PHS_E_ARG, "fill_mapping: channel out of range"); return; }
  const int n = w.spec.n_prt_out();
  for (int i = 0; i < n; i++) {
    w.spec.map_ids[c * n + i] = map_ids[i];
    w.spec.map_masses[c * n + i] = masses[i];
    w.spec.map_widths[c * n + i] = widths[i];
  }
  ok_status();
}

void c_whizard_init_tree_structures(void) {
  std::lock_guard<std::mutex> lk(api_mutex());
  WhizardModule& w = W();
  if (!w.sized) { set_error(GPU_PHS_E_STATE, "init_tree_structures before set_particle_structure"); return; }
  size_t n = (size_t)w.n_channels * w.spec.n_prt();
  w.spec.d1.assign(n, 0); w.spec.d2.assign(n, 0); w.spec.has_children.assign(n, 0); w.spec.friends.assign(n, 0);
  w.trees_ready = true;
  ok_status();
}

void c_whizard_fill_tree_structure(int* channel, int* daughters1, int* daughters2, int* has_children, int* friends) {
  std::lock_guard<std::mutex> lk(api_mutex());
  WhizardModule& w = W();
  if (!w.trees_ready) { set_error(GPU_PHS_E_STATE, "fill_tree_structure before init_tree_structures"); return; }
  int c = *channel - 1;
  if (c < 0 || c >= w.n_channels) { set_error(GPU_PHS_E_ARG, "fill_tree_structure: channel out of range"); return; }
  const int n = w.spec.n_prt();
  for (int i = 0; i < n; i++) {
    w.spec.d1[c * n + i] = daughters1[i];
    w.spec.d2[c * n + i] = daughters2[i];
    w.spec.has_children[c * n + i] = has_children[i];
    w.spec.friends[c * n + i] = friends ? friends[i] : 0;
  }
  ok_status();
}

void c_whizard_init_channel_ids(int* batch_size, int* n_channels, int* channel_limits) {
  std::lock_guard<std::mutex> lk(api_mutex());
  WhizardModule& w = W();
  if (!batch_size || !n_channels || !channel_limits || *batch_size < 0 || *n_channels < 1) {
    set_error(GPU_PHS_E_ARG, "init_channel_ids: invalid arguments");
    return;
  }
  // Event i belongs to the first channel c with i < channel_limits[c] (cumulative ends).
  // The reference skips only leading empty channels (whizard_gpu_phs.cpp:93-97); every empty
  // channel is skipped here.
  w.runs.clear();
  int64_t done = 0;
  for (int c = 0; c < *n_channels && done < *batch_size; c++)
    if (channel_limits[c] > done) {
      done = std::min(channel_limits[c], *batch_size);
      w.runs.push_back({c, done});
    }
  if (done < *batch_size) {
    set_error(GPU_PHS_E_ARG, "init_channel_ids: channel_limits end before batch_size");
    w.runs.clear();
    return;
  }
  ok_status();
}

void c_whizard_set_threads(int* msq_threads, int* cb_threads, int* ab_threads) {
  std::lock_guard<std::mutex> lk(api_mutex());
  (void)cb_threads; (void)ab_threads;
  int t = msq_threads ? *msq_threads : 256;
  t = (t / 64) * 64;
  if (t < 64) t = 64;
  if (t > 256) t = 256;
  W().block = t;
  ok_status();
}

void c_whizard_init_gpu_phs(void) {
  std::lock_guard<std::mutex> lk(api_mutex());
  WhizardModule& w = W();
  if (!w.sized || !w.maps_ready || !w.trees_ready) {
    set_error(GPU_PHS_E_STATE, "init_gpu_phs before the structure, mappings and trees were set");
    return;
  }
  // validate the trees now (constants are recompiled for the beams of each generate call)
  ProcessSpec sp = w.spec;
  sp.E1 = sp.E2 = 0.5 * 1e3;
  CompiledProcess cp;
  std::string err = compile_process(sp, cp);
  if (!err.empty()) { set_error(GPU_PHS_E_TREE, err); return; }
  if (require_device()) return;
  w.initialized = true;
  (void)ensure_staging(w);   // (a failure is the next generate call's, which tries again)
  ok_status();
}

void c_whizard_finalize_gpu_phs(void) {
  std::lock_guard<std::mutex> lk(api_mutex());
  WhizardModule& w = W();
  free_buffers(w);
  free_staging(w);
  if (w.process >= 0) drop_process(w.process);
  w = WhizardModule();
  ok_status();
}

void c_whizard_gen_phs_from_x_gpu(double* E1_in, double* E2_in, bool* requires_boost_to_lab, int* n_events,
                                  int* n_channels, int* n_x, double* x, double* factors, double* volumes, bool* oks,
                                  double* p, double* x_out) {
  std::lock_guard<std::mutex> lk(api_mutex());
  (void)requires_boost_to_lab;
  WhizardModule& w = W();
  if (!w.initialized) { set_error(GPU_PHS_E_STATE, "gen_phs_from_x_gpu before init_gpu_phs"); return; }
  const int64_t n = *n_events;
  if (n <= 0) { ok_status(); return; }
  if (*n_x != w.n_x || *n_channels != w.n_channels) {
    set_error(GPU_PHS_E_ARG, "gen_phs_from_x_gpu: n_x / n_channels differ from set_particle_structure");
    return;
  }
  if (w.runs.empty() || w.runs.back().end < n) {
    set_error(GPU_PHS_E_STATE, "gen_phs_from_x_gpu: init_channel_ids covers fewer events");
    return;
  }
  // beams: fixed, or per event (phs.cu:1313-1317); the trees are compiled for the first
  // event's, and with per-event beams the kernels recompute what depends on them
  const double E1 = E1_in[0], E2 = E2_in[0];
  bool varying = false, positive = true;
  for (int64_t i = 0; i < n; i++) {   // (no branches: vector instructions)
    positive &= (E1_in[i] > 0) & (E2_in[i] > 0);
    varying |= (E1_in[i] != E1) | (E2_in[i] != E2);
  }
  if (!positive) {
    set_error(GPU_PHS_E_ARG, "gen_phs_from_x_gpu: beam energies must be positive");
    return;
  }
  if (compile_for_beams(w, E1, E2)) return;
  if (w.plan && !w.plan_segs.empty() && w.plan_segs[0].process != w.process) { w.plan.reset(); w.plan_segs.clear(); }
  if (ensure_buffers(w, (size_t)n)) return;
  if (ensure_staging(w)) return;
  // the beam energies stay on the device, E1 then E2, as the reference keeps them
  // (get_in_momentum_device_pointer, phs.cu:1361-1363); per-event beams read them from there
  const size_t row = (size_t)n * sizeof(double);
  if (transfer(w, {{x, w.x_d, row * w.n_x}, {E1_in, w.e_d, row}, {E2_in, w.e_d + n, row}}, true)) return;

  // segments = runs of equal channel id
  std::vector<gpu_phs_segment> segs;
  for (int64_t i = 0, r = 0; i < n; r++) {
    const int64_t j = std::min<int64_t>(n, w.runs[r].end);
    gpu_phs_segment s{};
    s.process = w.process;
    s.channel = w.runs[r].channel;
    s.n_events = j - i;
    s.x = w.x_d + i * w.n_x;
    s.p = w.p_d + i * w.n_out * 4;
    s.factors = w.f_d + i;
    s.volumes = w.v_d + i;
    s.oks = w.ok_d + i;
    segs.push_back(s);
    i = j;
  }
  // the plan (and its inverse tables) is kept while the segments and the beam mode repeat
  const bool same = w.plan && w.plan_varying == varying && w.plan_segs.size() == segs.size() &&
                    std::memcmp(w.plan_segs.data(), segs.data(), segs.size() * sizeof(gpu_phs_segment)) == 0;
  if (!same) {
    if (!w.plan) w.plan = std::make_unique<PlanObj>();
    PlanObj& pl = *w.plan;
    pl.user = segs;
    pl.beam_e1.clear();
    pl.beam_e2.clear();
    if (varying) {
      for (size_t k = 0, r = 0; k < segs.size(); r += segs[k].n_events, k++) {
        pl.beam_e1.push_back(w.e_d + r);
        pl.beam_e2.push_back(w.e_d + n + r);
      }
    }
    // each tile class keeps its default shape with the block capped at set_threads' value,
    // and smaller where the LDS tables of the deepest trees would not fit
    const PlanObj defaults;
    for (int c = 0; c < kTileClasses; c++) pl.lcs[c].block = std::min(defaults.lcs[c].block, w.block);
    if (plan_build(pl)) { w.plan.reset(); return; }
    for (int c = 0; c < kTileClasses; c++)
      while (pl.lcs[c].block > 64 && forward_lds_bytes(pl.dps[c], pl.lcs[c]) > forward_lds_limit()) {
        pl.lcs[c].block -= 64;
        if (plan_build(pl)) { w.plan.reset(); return; }
      }
    w.plan_segs = segs;
    w.plan_varying = varying;
  }
  PlanObj& pl = *w.plan;
  if (plan_run(pl, w.stream)) return;
  // the inverse mapping of every event into every channel (the reference always asks for it,
  // whizard_gpu_phs.cpp:118): factors [n][n_channels] at [n_channels i + c] (phs.cu:207) and
  // x_out channel-major [n_x n c + n_x i + k] (phs.cu:222), own channel included
  if (ensure_inverse_buffers(w, (size_t)n)) return;
  std::vector<int64_t> rows(segs.size());
  for (size_t k = 0, r = 0; k < segs.size(); r += segs[k].n_events, k++) rows[k] = (int64_t)r;
  if (plan_inverse(pl, rows.data(), n, w.fa_d, w.xo_d, 0, w.stream)) return;
  const int nc = w.n_channels;
  if (transfer(w, {{p, w.p_d, row * w.n_out * 4}, {factors, w.fa_d, row * nc}, {volumes, w.v_d, row},
                   {oks, w.ok_d, (size_t)n}, {x_out, w.xo_d, x_out ? row * nc * w.n_x : 0}}, false))
    return;
  w.last_p = w.p_d;
  w.last_n = (size_t)n;
  ok_status();
}

void c_whizard_get_momentum_device_pointer(double* p) {
  std::lock_guard<std::mutex> lk(api_mutex());
  if (p) {
    uint64_t addr = (uint64_t)(uintptr_t)W().last_p;
    std::memcpy(p, &addr, sizeof addr);
  }
  ok_status();
}

}  // extern "C"

// transfer_to_whizard.h:1-3 (C++ linkage, as the reference declares them): device pointers of
// the last generate call's momenta ([n_events][n_out][4], the Whizard layout: the reference
// returns its internal per-branch array and gathers on the host, phs.cu:1566-1575), beam
// energies (E1 [n_events], then E2 [n_events]) and ok flags ([n_events] bool).  NULL before
// the first call.
double* get_momentum_device_pointer() {
  std::lock_guard<std::mutex> lk(api_mutex());
  return W().last_p;
}
double* get_in_momentum_device_pointer() {
  std::lock_guard<std::mutex> lk(api_mutex());
  return W().last_n ? W().e_d : nullptr;
}
bool* get_ok_device_pointer() {
  std::lock_guard<std::mutex> lk(api_mutex());
  return W().last_n ? reinterpret_cast<bool*>(W().ok_d) : nullptr;
}

extern "C" {

void c_whizard_reset_generator(void) {
  std::lock_guard<std::mutex> lk(api_mutex());
  WhizardModule& w = W();
  free_buffers(w);
  free_staging(w);
  std::fill(w.spec.flv_masses.begin(), w.spec.flv_masses.end(), 0.0);
  std::fill(w.spec.flv_widths.begin(), w.spec.flv_widths.end(), 0.0);
  if (w.process >= 0) { drop_process(w.process); w.process = -1; }
  ok_status();
}

void c_whizard_show_module(void) {
  std::lock_guard<std::mutex> lk(api_mutex());
  WhizardModule& w = W();
  const ProcessSpec& sp = w.spec;
  printf("n_channels: %d\nn_ext_in: %d\nn_ext_out: %d\nn_ext_tot: %d\n", w.n_channels, w.n_in, w.n_out, w.n_in + w.n_out);
  if (!w.sized) { printf(" STRUCTURE NOT SET UP!\n"); ok_status(); return; }
  printf("n_prt: %d\nn_prt_out: %d\nroot_branch: %d\nn_branches: %d\nn_x: %d\n", sp.n_prt(), sp.n_prt_out(), sp.root(),
         2 * w.n_out - 1, w.n_x);
  printf("flv_masses:");
  for (double m : sp.flv_masses) printf(" %lf", m);
  printf("\nMappings:\n");
  if (!w.maps_ready) printf(" MAPPINGS NOT SET UP!\n");
  else
    for (int c = 0; c < w.n_channels; c++) {
      printf(" c: %d\n ids:", c);
      for (int i = 0; i < sp.n_prt_out(); i++) printf(" %d", sp.map_ids[c * sp.n_prt_out() + i]);
      printf("\n masses:");
      for (int i = 0; i < sp.n_prt_out(); i++) printf(" %lf", sp.map_masses[c * sp.n_prt_out() + i]);
      printf("\n widths:");
      for (int i = 0; i < sp.n_prt_out(); i++) printf(" %lf", sp.map_widths[c * sp.n_prt_out() + i]);
      printf("\n");
    }
  printf("Trees:\n");
  if (!w.trees_ready) printf(" TREES NOT SET UP!\n");
  else
    for (int c = 0; c < w.n_channels; c++) {
      printf(" channel %d:", c);
      for (int i = 0; i < sp.n_prt(); i++)
        if (sp.has_children[c * sp.n_prt() + i])
          printf(" %d->(%d,%d)", i + 1, sp.d1[c * sp.n_prt() + i], sp.d2[c * sp.n_prt() + i]);
      printf("\n");
    }
  if (w.initialized && w.process >= 0) {
    ProcessObj* po = find_process(w.process);
    if (po) {
      printf("Programs (visit order: branch, phi random, daughters, next):\n");
      for (size_t c = 0; c < po->cp.channels.size(); c++) {
        const ChannelDesc& cd = po->cp.channels[c];
        printf(" channel %zu:", c);
        for (int i = 0; i < cd.n_nodes; i++) {
          const NodeCmd& nd = po->cp.nodes[cd.node0 + i];
          printf(" [%d x%d desc=%d push=%d]", po->cp.node_branch[cd.node0 + i] + 1, nd.x_phi, nd.desc, nd.push);
        }
        printf("\n");
      }
    }
  }
  printf("END OF MODULE\n");
  fflush(stdout);
  ok_status();
}

}  // extern "C"
