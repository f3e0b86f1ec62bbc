// Staging of host buffers: device mirrors that outlive a call, and copies between
// pageable host memory and the device that run at the speed of the link.
//
// A call with host arrays (device id -1) used to allocate and free a device buffer per
// array and leave the copies to hipMemcpy.  Two passes over 2 x 256 x 64 x 64 with 512
// boxes move 68 MB, 1.2 ms of a 56 GB/s link, and took 3.6-4.7 ms: hipMemcpy reaches
// 38 GB/s to the device and 17 GB/s back, where one thread copies out of the runtime's
// buffer into memory that is being touched for the first time.  Here a copy goes in
// pieces through a ring of pinned slots: the calling thread issues the transfers, helper
// threads (and the calling thread while it waits) move pieces between the slots and the
// caller's memory, and take the page faults in parallel: the same two passes in 1.9 ms.
#include "runtime.h"

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>

#include <pthread.h>

namespace mobula_hip {
namespace {

// A transfer is one slot.  A transfer and its event cost some 20 us beside the time on the link, in which nothing moves if
// the next one stands in the same queue: transfers take turns in two lanes, streams of the copier that follow the
// caller's and that the caller's then follows.  Threads copy in smaller pieces, so that a slot is emptied by all of them.
// (Both passes of the shape above, one lane: 2293 us with transfers of 2 MB, 2068 with 4, 2189 with 8; two lanes: 1880 with
// 2 MB, 1900 with 4; three lanes of 2 MB 1890 to 2550, four of 1 MB 1940.)  Below some seven megabytes one lane, the caller's
// stream, with transfers of 4 MB is faster (a forward pass with a map of 2.4 MB: 150 us, two lanes 178; 6.5: 259 and 274; 9: 354 and
// 323; 20: 603 and 540).
constexpr size_t kTransfer = 2u << 20;
constexpr size_t kPiece = 256u << 10;
constexpr int kSlots = 12;
constexpr int kLanes = 2;
constexpr size_t kLanesAbove = 7u << 20;
// Below this hipMemcpy is as fast: waking the helpers costs some twenty microseconds.
constexpr size_t kPipelinedBytes = 2u << 20;
constexpr int kMostHelpers = 7;
// Device mirrors above this are allocated for the call alone.
constexpr size_t kMostKept = 1ull << 30;

inline void relax() { __builtin_ia32_pause(); }

// One copy in flight.  Pieces are claimed in order; `open` is how many may be claimed (to the
// device: their slot is free; from the device: they have arrived).
struct Job {
  char* host = nullptr;
  size_t bytes = 0;
  bool to_device = false;
  size_t transfer = kTransfer;   // bytes of one, and of a slot
  int ring = kSlots, per_transfer = 0, pieces = 0, transfers = 0;
  char* slots = nullptr;
  std::atomic<int> next{0}, open{0}, finished{0};
  std::atomic<int> copied[kSlots];   // pieces of the slot's transfer that have been copied

  size_t transfer_bytes(int t) const { return std::min(transfer, bytes - static_cast<size_t>(t) * transfer); }
  int pieces_of(int t) const { return std::min(per_transfer, pieces - t * per_transfer); }
  bool is_copied(int t) const { return copied[t % ring].load(std::memory_order_acquire) == pieces_of(t); }
  char* slot(int t) const { return slots + static_cast<size_t>(t % ring) * transfer; }
  // Claims and copies one piece; false: none is open.
  bool help() {
    int i = next.load(std::memory_order_relaxed);
    do {
      if (i >= open.load(std::memory_order_acquire) || i >= pieces) return false;
    } while (!next.compare_exchange_weak(i, i + 1, std::memory_order_acq_rel));
    const int t = i / per_transfer;
    char* const there = slot(t) + static_cast<size_t>(i % per_transfer) * kPiece;
    char* const mine = host + static_cast<size_t>(i) * kPiece;
    const size_t size = std::min(kPiece, bytes - static_cast<size_t>(i) * kPiece);
    if (to_device) std::memcpy(there, mine, size);
    else std::memcpy(mine, there, size);
    copied[t % ring].fetch_add(1, std::memory_order_acq_rel);
    finished.fetch_add(1, std::memory_order_acq_rel);
    return true;
  }
};

// The pinned ring and the helper threads, shared by all calling threads: a copy that finds them
// taken goes through hipMemcpy instead.  Helpers end after two idle seconds; after a fork the
// child starts with none.
class Copier {
 public:
  static Copier& get() {
    static Copier* const one = new Copier;   // (never destroyed: helpers may outlive static objects)
    return *one;
  }

  // True if the copy was made (or has failed, with the error set); false: use hipMemcpy.  On return
  // from a copy to the device its last transfers may still be in flight; `stream` waits for them.
  bool copy(void* dev, void* host, size_t bytes, bool to_device, hipStream_t stream) {
    if (bytes < kPipelinedBytes) return false;
    std::unique_lock<std::mutex> mine(busy_, std::try_to_lock);
    if (!mine.owns_lock() || !ready()) return false;
    job_.host = static_cast<char*>(host); job_.bytes = bytes; job_.to_device = to_device;
    const int wide = bytes > kLanesAbove ? 1 : kLanes;   // (as many bytes in the ring)
    job_.transfer = wide * kTransfer; job_.ring = kSlots / wide; job_.per_transfer = static_cast<int>(job_.transfer / kPiece);
    job_.pieces = static_cast<int>((bytes + kPiece - 1) / kPiece);
    job_.transfers = static_cast<int>((bytes + job_.transfer - 1) / job_.transfer);
    job_.slots = slots_;
    for (auto& c : job_.copied) c.store(0, std::memory_order_relaxed);
    for (int k = 0; k < kSlots; ++k)   // slots that a previous copy to the device still reads
      if (pending_[k]) { MOBULA_HIP_TRY(hipEventSynchronize(events_[k])); pending_[k] = false; }
    if (failed()) return true;
    job_.next.store(0); job_.finished.store(0);
    job_.open.store(to_device ? std::min(job_.ring * job_.per_transfer, job_.pieces) : 0);
    wake();
    if (to_device) send(static_cast<char*>(dev), stream);
    else receive(static_cast<const char*>(dev), stream);
    if (!failed()) (void)hipGetLastError();   // (a query that found an event not ready is no error of the call)
    // nobody may look at the job any more (a helper that came late finds nothing open)
    job_.next.store(job_.pieces);
    {
      std::lock_guard<std::mutex> lock(state_);
      working_ = false;
    }
    while (inside_.load(std::memory_order_acquire) != 0) relax();
    return true;
  }

  // Gives the pinned ring back (unless a copy is using it).
  void release() {
    std::unique_lock<std::mutex> mine(busy_, std::try_to_lock);
    if (!mine.owns_lock() || slots_ == nullptr) return;
    for (int k = 0; k < kSlots; ++k) {
      if (pending_[k]) (void)hipEventSynchronize(events_[k]);
      pending_[k] = false;
    }
    drop_events();
    (void)hipHostFree(slots_);
    slots_ = nullptr;
  }

 private:
  Copier() { pthread_atfork(nullptr, nullptr, [] { get().after_fork(); }); }

  // (the child of a fork has no helpers, and must not wait for locks its parent's threads held)
  void after_fork() {
    new (&busy_) std::mutex;
    new (&state_) std::mutex;
    new (&wake_) std::condition_variable;
    helpers_ = 0;
    inside_.store(0);
    working_ = false;
  }

  // The ring, its events and lanes for the current device.
  bool ready() {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return false;
    if (slots_ == nullptr) {
      void* p = nullptr;
      if (hipHostMalloc(&p, kTransfer * kSlots, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
      slots_ = static_cast<char*>(p);
    }
    if (device != events_device_) {
      for (int k = 0; k < kSlots; ++k) {
        if (pending_[k]) (void)hipEventSynchronize(events_[k]);
        pending_[k] = false;
      }
      drop_events();
      bool made = hipEventCreateWithFlags(&ordered_, hipEventDisableTiming) == hipSuccess;
      for (auto& e : events_) made = made && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
      for (auto& lane : lanes_) made = made && hipStreamCreateWithFlags(&lane, hipStreamNonBlocking) == hipSuccess;
      if (!made) {
        (void)hipGetLastError();
        drop_events();
        return false;
      }
      events_device_ = device;
    }
    return true;
  }
  void drop_events() {
    for (auto& e : events_) {
      if (e != nullptr) (void)hipEventDestroy(e);
      e = nullptr;
    }
    if (ordered_ != nullptr) (void)hipEventDestroy(ordered_);
    ordered_ = nullptr;
    for (auto& lane : lanes_) {
      if (lane != nullptr) (void)hipStreamDestroy(lane);
      lane = nullptr;
    }
    events_device_ = -1;
  }

  void wake() {
    std::lock_guard<std::mutex> lock(state_);
    working_ = true;
    ++jobs_;
    const int wanted = std::min({kMostHelpers, processors() - 1, job_.pieces / 2});
    while (helpers_ < wanted) {
      try {
        std::thread([this] { help_with_jobs(); }).detach();
      } catch (...) {
        break;   // (as many as the system gives; the calling thread copies as well)
      }
      ++helpers_;
    }
    wake_.notify_all();
  }
  static int processors() {   // half of those the process may use: the others are the caller's
    cpu_set_t set;
    CPU_ZERO(&set);
    const int n = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 2;
    return std::max(1, (n + 1) / 2);
  }

  void help_with_jobs() {
    unsigned long long seen = 0;
    std::unique_lock<std::mutex> lock(state_);
    for (;;) {
      if (!wake_.wait_for(lock, std::chrono::seconds(2), [&] { return working_ && jobs_ != seen; })) {
        --helpers_;
        return;
      }
      seen = jobs_;
      inside_.fetch_add(1, std::memory_order_acq_rel);
      lock.unlock();
      int idle = 0;
      while (job_.next.load(std::memory_order_acquire) < job_.pieces) {
        if (job_.help()) idle = 0;
        else if (++idle < 256) relax();
        else sched_yield();
      }
      inside_.fetch_sub(1, std::memory_order_acq_rel);
      lock.lock();
    }
  }

  bool in_lanes() const { return job_.transfer == kTransfer; }
  // The lanes follow what the caller's stream has been given: it may use the memory that a transfer writes, or
  // write what one reads.
  void follow(hipStream_t stream) {
    if (!in_lanes()) return;
    MOBULA_HIP_TRY(hipEventRecord(ordered_, stream));
    for (const hipStream_t lane : lanes_)
      if (!failed()) MOBULA_HIP_TRY(hipStreamWaitEvent(lane, ordered_, 0));
  }

  void send(char* dev, hipStream_t stream) {
    int issued = 0, sent = 0;
    follow(stream);
    while (issued < job_.transfers && !failed()) {
      bool moved = false;
      if (issued < sent + job_.ring && job_.is_copied(issued)) {   // (beyond: the slot still counts the round before)
        const hipStream_t lane = in_lanes() ? lanes_[issued % kLanes] : stream;
        MOBULA_HIP_TRY(hipMemcpyAsync(dev + static_cast<size_t>(issued) * job_.transfer, job_.slot(issued),
                                      job_.transfer_bytes(issued), hipMemcpyHostToDevice, lane));
        MOBULA_HIP_TRY(hipEventRecord(events_[issued % job_.ring], lane));
        pending_[issued % job_.ring] = true;
        ++issued;
        moved = true;
      }
      // a slot whose transfer has ended is free for the transfer a round later
      if (sent < issued && sent + job_.ring < job_.transfers && hipEventQuery(events_[sent % job_.ring]) == hipSuccess) {
        job_.copied[sent % job_.ring].store(0, std::memory_order_relaxed);
        ++sent;
        job_.open.store(std::min(job_.pieces, (sent + job_.ring) * job_.per_transfer), std::memory_order_release);
        moved = true;
      }
      if (!moved && !job_.help()) relax();
    }
    if (failed()) finish_claimed();
    // the caller's stream goes on when the last transfer of every lane has ended
    for (int t = std::max(0, issued - kLanes); t < issued && in_lanes() && !failed(); ++t)
      MOBULA_HIP_TRY(hipStreamWaitEvent(stream, events_[t % job_.ring], 0));
    if (failed()) wait_for_lanes(stream);
  }

  void receive(const char* dev, hipStream_t stream) {
    int issued = 0, arrived = 0;
    follow(stream);
    while (job_.finished.load(std::memory_order_acquire) < job_.pieces && !failed()) {
      bool moved = false;
      if (issued < job_.transfers && (issued < job_.ring || job_.is_copied(issued - job_.ring))) {
        if (issued >= job_.ring) job_.copied[issued % job_.ring].store(0, std::memory_order_relaxed);
        const hipStream_t lane = in_lanes() ? lanes_[issued % kLanes] : stream;
        MOBULA_HIP_TRY(hipMemcpyAsync(job_.slot(issued), dev + static_cast<size_t>(issued) * job_.transfer,
                                      job_.transfer_bytes(issued), hipMemcpyDeviceToHost, lane));
        MOBULA_HIP_TRY(hipEventRecord(events_[issued % job_.ring], lane));
        ++issued;
        moved = true;
      }
      if (arrived < issued) {
        const hipError_t state = hipEventQuery(events_[arrived % job_.ring]);
        if (state == hipSuccess) {
          ++arrived;
          job_.open.store(std::min(job_.pieces, arrived * job_.per_transfer), std::memory_order_release);
          moved = true;
        } else if (state != hipErrorNotReady) {
          MOBULA_HIP_TRY(state);
        }
      }
      if (!moved && !job_.help()) relax();
    }
    if (failed()) {
      wait_for_lanes(stream);
      finish_claimed();
    }
  }
  void wait_for_lanes(hipStream_t stream) {
    if (!in_lanes()) (void)hipStreamSynchronize(stream);
    for (const hipStream_t lane : lanes_) (void)hipStreamSynchronize(lane);
  }
  // After an error: nothing more is claimed, and what was claimed is finished.
  void finish_claimed() {
    const int claimed = job_.next.exchange(job_.pieces);
    while (job_.finished.load(std::memory_order_acquire) < std::min(claimed, job_.pieces)) relax();
  }

  std::mutex busy_;    // held for a copy
  std::mutex state_;   // helpers_, working_, jobs_
  std::condition_variable wake_;
  int helpers_ = 0;
  bool working_ = false;
  unsigned long long jobs_ = 0;
  std::atomic<int> inside_{0};   // helpers looking at the job
  Job job_;
  char* slots_ = nullptr;
  hipEvent_t events_[kSlots] = {};
  hipEvent_t ordered_ = nullptr;
  hipStream_t lanes_[kLanes] = {};
  bool pending_[kSlots] = {};    // a transfer out of the slot may be in flight
  int events_device_ = -1;
};

// Device memory for mirrors, one block per calling thread and device, used like a stack by the
// HostStaging objects of a call.
struct Arena {
  char* base = nullptr;
  size_t bytes = 0, used = 0;
};
struct ArenasOfThread {
  std::map<int, Arena> per_device;
  ~ArenasOfThread() {
    for (auto& it : per_device)
      if (it.second.base != nullptr) (void)hipFree(it.second.base);
  }
};
Arena* arena_of_current_device() {
  static thread_local ArenasOfThread mine;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return nullptr;
  return &mine.per_device[device];
}
size_t mirror_bytes(size_t bytes) { return (std::max<size_t>(bytes, 1) + 255) / 256 * 256; }

}  // namespace

HostStaging::HostStaging() {
  Arena* const a = arena_of_current_device();
  mark_ = a == nullptr ? 0 : a->used;
}

HostStaging::~HostStaging() {
  if (unfinished_) (void)hipStreamSynchronize(nullptr);   // (left early: transfers may still use the mirrors)
  for (auto& it : items_)
    if (it.own) (void)hipFree(it.dev);
  Arena* const a = arena_of_current_device();
  if (a != nullptr) a->used = mark_;
}

void HostStaging::reserve(std::initializer_list<size_t> sizes) {
  size_t total = 0;
  for (const size_t s : sizes) total += mirror_bytes(s);
  Arena* const a = arena_of_current_device();
  if (a == nullptr || a->used != 0 || total <= a->bytes || total > kMostKept) return;
  if (a->base != nullptr) (void)hipFree(a->base);
  a->base = nullptr;
  a->bytes = 0;
  void* p = nullptr;
  const size_t want = std::min(kMostKept, total + total / 8);
  if (hipMalloc(&p, want) != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  a->base = static_cast<char*>(p);
  a->bytes = want;
}

void* HostStaging::in(const void* host, size_t bytes, bool upload) {
  void* dev = inout(const_cast<void*>(host), bytes, upload);
  items_.back().download = false;
  return dev;
}

void* HostStaging::inout(void* host, size_t bytes, bool upload) {
  Item item{nullptr, host, bytes, true, false};
  if (items_.empty()) reserve({bytes});
  Arena* const a = arena_of_current_device();
  if (a != nullptr && a->used + mirror_bytes(bytes) <= a->bytes) {
    item.dev = a->base + a->used;
    a->used += mirror_bytes(bytes);
  } else {
    MOBULA_HIP_TRY(hipMalloc(&item.dev, bytes > 0 ? bytes : 1));
    item.own = true;
  }
  items_.push_back(item);
  if (!failed() && upload && bytes > 0) {
    if (Copier::get().copy(item.dev, host, bytes, /*to_device=*/true, nullptr)) unfinished_ = true;
    else MOBULA_HIP_TRY(hipMemcpy(item.dev, host, bytes, hipMemcpyHostToDevice));
  }
  return item.dev;
}

bool HostStaging::flush(hipStream_t stream) {
  bool waited = false;
  for (auto& it : items_) {
    if (failed()) break;
    if (!it.download || it.bytes == 0) continue;
    if (Copier::get().copy(it.dev, it.host, it.bytes, /*to_device=*/false, stream)) continue;
    if (!waited) MOBULA_HIP_TRY(hipStreamSynchronize(stream));
    waited = true;
    if (!failed()) MOBULA_HIP_TRY(hipMemcpy(it.host, it.dev, it.bytes, hipMemcpyDeviceToHost));
  }
  if (!waited) MOBULA_HIP_TRY(hipStreamSynchronize(stream));
  if (!failed()) unfinished_ = false;
  return !failed();
}

long long staging_bytes() {
  const Arena* const a = arena_of_current_device();
  return a == nullptr ? 0 : static_cast<long long>(a->bytes);
}

long long release_staging() {
  Copier::get().release();
  Arena* const a = arena_of_current_device();
  if (a == nullptr || a->base == nullptr || a->used != 0) return 0;
  const long long bytes = static_cast<long long>(a->bytes);
  (void)hipFree(a->base);
  *a = Arena();
  return bytes;
}

}  // namespace mobula_hip
