// transfer.cpp -- copies between pageable host memory and the device.
//
// The runtime moves pageable memory through a staging buffer of its own with
// one thread: bound by that thread's copy.  Copies of kStagedCopyMin bytes or
// more go through a ring of pinned slots here instead: the DMA engine moves
// some slots while a few threads move others between the ring and the caller's
// memory.  Measured (us, the runtime's copy -> this one; the DMA alone reaches
// 57 GB/s, 4700 us for 256 MB):
//     bytes      down            up
//     16 MB      943 ->  940     492 ->  515   waking the helpers costs the gain
//     64 MB     3689 -> 2780    2350 -> 1850
//    256 MB    15039 -> 7230    9344 -> 6910
// Memory that HIP knows (pinned, managed, device) and smaller copies take the
// runtime's path, and so does a process that was forked from the one whose
// helper threads these are.
#include <pthread.h>
#include <sched.h>
#include <signal.h>
#include <unistd.h>

#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

#include "lc_internal.hpp"

namespace lchip {

namespace {

constexpr int kSlots = 8;
constexpr std::size_t kSlotBytes = std::size_t{2} << 20;
constexpr std::size_t kMinChunk = std::size_t{256} << 10;

// One copy: chunks 0 .. n - 1, chunk i in slot i % kSlots.  Each thread owns
// some slots and runs their chunks by itself, so nobody waits for another
// thread on the way:
//   down: wait for the slot's DMA, move the chunk out, enqueue the slot's next;
//   up:   wait for the slot's last DMA (of this copy or an earlier one), move
//         the chunk in, enqueue its DMA.
// Waits on events spin, so the other threads join only once the stream has
// reached the copy.
struct Transfer {
  HipContext* ctx = nullptr;
  bool down = false;
  char* host = nullptr;
  char* dev = nullptr;
  std::size_t bytes = 0, chunk = 0;
  int n = 0;
  int threads = 1;             // that share the slots: thread w has slots w, w + threads, ...
  int first = 0, end = 0;      // the chunks they move
  std::atomic<int> error{0};   // first hipError_t; everyone stops

  std::size_t size(int i) const { return i + 1 < n ? chunk : bytes - static_cast<std::size_t>(i) * chunk; }
  bool failed() const { return error.load(std::memory_order_acquire) != 0; }
  void fail(hipError_t e) {
    int none = 0;
    error.compare_exchange_strong(none, static_cast<int>(e));
  }
};

class Engine {
 public:
  static Engine* get() {
    static Engine* e = new (std::nothrow) Engine();  // process lifetime: its threads are never joined
    return e != nullptr && e->helpers_ > 0 && e->pid_ == getpid() ? e : nullptr;
  }

  // hipSuccess, or the error of the first call that failed.
  hipError_t run(HipContext* ctx, bool down, void* host, void* dev, std::size_t bytes) {
    std::lock_guard<std::mutex> one(run_mu_);
    Transfer t;
    t.ctx = ctx;
    t.down = down;
    t.host = static_cast<char*>(host);
    t.dev = static_cast<char*>(dev);
    t.bytes = bytes;
    t.chunk = kMinChunk;
    while (t.chunk < kSlotBytes && t.chunk * 2 * kSlots <= bytes) {
      t.chunk *= 2;  // a ring's worth of chunks, or more
    }
    t.n = t.end = static_cast<int>((bytes + t.chunk - 1) / t.chunk);
    if (down) {
      for (int i = 0; i < kSlots && i < t.n && !t.failed(); ++i) {
        enqueue(t, i);
      }
      // The helpers are woken once the first chunk is here.
      const hipError_t e = t.failed() ? hipSuccess : hipEventSynchronize(events_[0]);
      if (e != hipSuccess) {
        t.fail(e);
      }
    } else {
      // While the stream is busy with earlier work the caller fills the ring
      // alone, and the helpers are woken once the stream has come this far.  An
      // event tells: after a hipStreamQuery that finds the stream busy, the copies
      // that follow run at half the rate (2 x 256 MB 28.7 against 14.2 ms).
      hipError_t e = hipEventRecord(reached_, ctx->stream);
      bool busy = e == hipSuccess && hipEventQuery(reached_) == hipErrorNotReady;
      t.end = 0;
      while (busy && t.end < kSlots && t.end < t.n && !t.failed()) {
        t.first = t.end++;
        work(t, 0);
        busy = hipEventQuery(reached_) == hipErrorNotReady;
      }
      (void)hipGetLastError();
      if (busy) {
        e = hipEventSynchronize(reached_);
      }
      if (e != hipSuccess) {
        t.fail(e);
      }
      t.first = t.end;
      t.end = t.n;
    }
    if (t.failed()) {
      return static_cast<hipError_t>(t.error.load());
    }
    t.threads = helpers_ + 1;
    {
      std::lock_guard<std::mutex> lock(mu_);
      current_ = &t;
      ++generation_;
      working_ = helpers_;
    }
    wake_.notify_all();
    work(t, 0);
    {
      std::unique_lock<std::mutex> lock(mu_);
      idle_.wait(lock, [&] { return working_ == 0; });
      current_ = nullptr;
    }
    return static_cast<hipError_t>(t.error.load());
  }

 private:
  Engine() {
    // Three helpers, or half of the CPUs this process may use; the caller
    // moves chunks too.
    cpu_set_t set;
    CPU_ZERO(&set);
    const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
    const int want = cpus / 2 < 3 ? cpus / 2 : 3;
    if (want < 1 || ring_.ensure(kSlots * kSlotBytes) != Status::kSuccess) {
      return;
    }
    for (hipEvent_t& e : events_) {
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        return;
      }
    }
    if (hipEventCreateWithFlags(&reached_, hipEventDisableTiming) != hipSuccess) {
      return;
    }
    // Helpers take no signals: those stay with the program's own threads.
    sigset_t all, before;
    sigfillset(&all);
    pthread_sigmask(SIG_SETMASK, &all, &before);
    for (int i = 0; i < want; ++i) {
      try {
        std::thread([this, i] { help(i + 1); }).detach();
        ++helpers_;
      } catch (...) {
        break;  // as many as the process may have
      }
    }
    pthread_sigmask(SIG_SETMASK, &before, nullptr);
  }

  char* slot(int i) const {
    return static_cast<char*>(ring_.get()) + static_cast<std::size_t>(i % kSlots) * kSlotBytes;
  }

  void enqueue(Transfer& t, int i) {
    char* dev = t.dev + static_cast<std::size_t>(i) * t.chunk;
    hipError_t e = t.down ? hipMemcpyAsync(slot(i), dev, t.size(i), hipMemcpyDeviceToHost, t.ctx->stream)
                          : hipMemcpyAsync(dev, slot(i), t.size(i), hipMemcpyHostToDevice, t.ctx->stream);
    if (e == hipSuccess) {
      e = hipEventRecord(events_[i % kSlots], t.ctx->stream);
    }
    if (e != hipSuccess) {
      t.fail(e);
    }
  }

  void work(Transfer& t, int w) {
    for (int i = t.first; i < t.end; ++i) {
      const int s = i % kSlots;
      if (s % t.threads != w) {
        continue;
      }
      if (t.failed()) {
        return;
      }
      const hipError_t e = hipEventSynchronize(events_[s]);
      if (e != hipSuccess) {
        t.fail(e);
        return;
      }
      char* host = t.host + static_cast<std::size_t>(i) * t.chunk;
      if (t.down) {
        std::memcpy(host, slot(i), t.size(i));
        if (i + kSlots < t.n) {
          enqueue(t, i + kSlots);
        }
      } else {
        std::memcpy(slot(i), host, t.size(i));
        enqueue(t, i);
      }
    }
  }

  void help(int w) {
    unsigned long long seen = 0;  // the copy this thread joined last
    std::unique_lock<std::mutex> lock(mu_);
    for (;;) {
      wake_.wait(lock, [&] { return generation_ != seen; });
      seen = generation_;
      Transfer* t = current_;
      lock.unlock();
      const hipError_t e = hipSetDevice(t->ctx->device);
      if (e != hipSuccess) {
        t->fail(e);
      }
      work(*t, w);
      lock.lock();
      if (--working_ == 0) {
        idle_.notify_one();
      }
    }
  }

  PinnedBuffer ring_;
  hipEvent_t events_[kSlots] = {};
  hipEvent_t reached_ = nullptr;  // recorded before an upload
  int helpers_ = 0;
  const pid_t pid_ = getpid();
  std::mutex run_mu_;  // one copy at a time
  std::mutex mu_;      // the members below
  std::condition_variable wake_, idle_;
  Transfer* current_ = nullptr;
  unsigned long long generation_ = 0;
  int working_ = 0;  // helpers that have not finished current_
};

// A pointer HIP has an allocation for is copied by the runtime directly.
bool pageable(const void* p) {
  hipPointerAttribute_t attr{};
  if (hipPointerGetAttributes(&attr, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return attr.type == hipMemoryTypeUnregistered;
}

Status transfer(HipContext* ctx, bool down, void* host, void* dev, std::size_t bytes, bool* done) {
  *done = false;
  if (bytes < kStagedCopyMin || !pageable(host)) {
    return Status::kSuccess;
  }
  Engine* engine = Engine::get();
  if (engine == nullptr) {
    return Status::kSuccess;
  }
  *done = true;
  const hipError_t e = engine->run(ctx, down, host, dev, bytes);
  return e == hipSuccess ? Status::kSuccess : failHip(e, down ? "download" : "upload");
}

}  // namespace

Status upload(HipContext* ctx, void* dst, const void* src, std::size_t bytes) {
  bool done = false;
  LC_TRY(transfer(ctx, false, const_cast<void*>(src), dst, bytes, &done));
  if (!done) {
    LC_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
  }
  return Status::kSuccess;
}

Status download(HipContext* ctx, void* dst, const void* src, std::size_t bytes) {
  bool done = false;
  LC_TRY(transfer(ctx, true, dst, const_cast<void*>(src), bytes, &done));
  if (!done) {
    LC_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
  }
  return Status::kSuccess;
}

}  // namespace lchip
