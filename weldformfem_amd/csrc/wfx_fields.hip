// Field transfer between the host's layout ([items][components], the
// reference's element order, double) and the device's ([components][items],
// stored element order, double or float).
//
// The kernels read and write pinned host memory directly, so that the
// transposition, the element permutation and the float conversion happen on
// the device, in the same pass that crosses the host link.  Before, the host
// did them in one thread over a pageable copy: the stress of the 4M-element
// block (192 MB) took 92 ms to read, now 12; a nodal vector of one element 22
// us, now 14 (where that way is still the shorter one it is taken: kCopyFrom).  What bounds it: the host link (57 GB/s pinned) and, for the
// fresh pages of a new array, the host's page faults, which is why several
// threads copy from the pinned ring to the caller's memory.
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "../../include/wfx.h"
#include "wfx_internal.hpp"
#include "wfx_launch.hpp"

namespace wfx {

// The pinned ring: kSlots chunks of kChunkBytes.  Measured on the stress of
// the 4M-element block (192 MB), read into the same array again / a new one /
// set: 1 MiB chunks 9.7 / 15.8 / 4.7 ms, 2 MiB 7.3 / 14.6 / 4.1, 4 MiB 5.7 /
// 11.9 / 4.0 (the link alone: 3.4); 12 or 16 threads instead of 8 gain nothing
// at 4 MiB.  Transfers of one chunk use a buffer of their own.
constexpr size_t kChunkBytes = (size_t)4 << 20;
constexpr int kSlots = 16, kCopyThreads = 8;

struct Staging {
  int device = -1;        // the events'
  char *small = nullptr;  // one chunk
  char *ring = nullptr;   // kSlots chunks, allocated by the first transfer that needs them
  hipEvent_t ev[kSlots] = {};
  ~Staging() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    if (small) (void)hipHostFree(small);
    if (ring) (void)hipHostFree(ring);
  }
};

// The staging belongs to a transfer, not to a context: a transfer takes one that
// is idle, or makes one, and leaves it for the next.  Many contexts in turn then
// hold one (68 MiB of pinned memory), not one each; transfers at the same time
// have their own.  At most kIdle stay, for as many threads that read fields all
// the time, and none after the last context.
constexpr int kIdle = 4;
static std::mutex g_stage_mu;
static Staging *g_idle[kIdle] = {};
static long g_contexts = 0;

void staging_open() {
  std::lock_guard<std::mutex> l(g_stage_mu);
  ++g_contexts;
}
void staging_close() {
  Staging *drop[kIdle] = {};
  {
    std::lock_guard<std::mutex> l(g_stage_mu);
    if (--g_contexts == 0) std::swap(drop, g_idle);
  }
  for (Staging *s : drop) delete s;
}

// The current device is the transfer's.
class StagingLease {
 public:
  explicit StagingLease(int device) {
    {
      std::lock_guard<std::mutex> l(g_stage_mu);
      for (Staging *&q : g_idle)
        if (!s_ && q && q->device == device) std::swap(s_, q);
    }
    if (!s_) s_ = new Staging();
    s_->device = device;
  }
  ~StagingLease() {
    {
      std::lock_guard<std::mutex> l(g_stage_mu);
      for (Staging *&q : g_idle)
        if (s_ && !q) std::swap(s_, q);
    }
    delete s_;
  }
  StagingLease(const StagingLease &) = delete;
  StagingLease &operator=(const StagingLease &) = delete;
  Staging &operator*() const { return *s_; }

 private:
  Staging *s_ = nullptr;
};

// Allocates what is not there yet.  Without memory for a ring the transfer goes
// chunk by chunk.
static int staging_ready(Staging &s, bool ring) {
  if (ring && !s.ring) {
    for (hipEvent_t &e : s.ev)
      if (!e) WFX_CHECK_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    if (hipHostMalloc((void **)&s.ring, kChunkBytes * kSlots, hipHostMallocPortable) != hipSuccess) {
      s.ring = nullptr;
      (void)hipGetLastError();  // or the next launch would report it
    }
  }
  if (!(ring && s.ring) && !s.small) {
    const hipError_t e = hipHostMalloc((void **)&s.small, kChunkBytes, hipHostMallocPortable);
    if (e != hipSuccess) {
      s.small = nullptr;
      (void)hipGetLastError();
    }
    WFX_CHECK_HIP(e);
  }
  return WFX_OK;
}

namespace {

constexpr int kB = 256;

// one row of blocks per buffer, 16 bytes a thread and turn (hipMalloc aligns to
// 256; the words past the last whole 16 bytes one by one)
__global__ __launch_bounds__(kB) void k_fill(FillList f) {
  const auto b = f.buf[blockIdx.y];
  const size_t n4 = b.words / 4;
  const uint4 v = make_uint4(b.lo, b.hi, b.lo, b.hi);
  const size_t t = (size_t)blockIdx.x * kB + threadIdx.x, step = (size_t)gridDim.x * kB;
  for (size_t i = t; i < n4; i += step) static_cast<uint4 *>(b.p)[i] = v;
  for (size_t i = 4 * n4 + t; i < b.words; i += step) static_cast<unsigned *>(b.p)[i] = i & 1 ? b.hi : b.lo;
}

// device row of host component r, or -1 (the spin's zero diagonal: host
// columns 0..2 of 6, device rows 0..2 for columns 3..5)
template <bool SPIN>
__device__ __forceinline__ int device_row(int r) {
  return SPIN ? r - 3 : r;
}

// host values [k0, k0 + n) of the flat [items][rows] array, one per thread:
// consecutive threads write consecutive host addresses (full link packets);
// the scattered device reads stay in L2, which outruns the link by far
template <typename T, bool SPIN>
__global__ __launch_bounds__(kB) void k_field_out(long k0, long n, int rows, long cnt, const int *__restrict__ perm,
                                                  const T *__restrict__ dev, double *__restrict__ host) {
  const long t = (long)blockIdx.x * kB + threadIdx.x;
  if (t >= n) return;
  const long k = k0 + t, i = k / rows;
  const int r = device_row<SPIN>((int)(k - i * rows));
  double v = 0.0;
  if (r >= 0) v = (double)dev[(long)r * cnt + (perm ? (long)perm[i] : i)];
  host[t] = v;
}
template <typename T, bool SPIN>
__global__ __launch_bounds__(kB) void k_field_in(long k0, long n, int rows, long cnt, const int *__restrict__ perm,
                                                 const double *__restrict__ host, T *__restrict__ dev) {
  const long t = (long)blockIdx.x * kB + threadIdx.x;
  if (t >= n) return;
  const long k = k0 + t, i = k / rows;
  const int r = device_row<SPIN>((int)(k - i * rows));
  if (r >= 0) dev[(long)r * cnt + (perm ? (long)perm[i] : i)] = (T)host[t];
}

template <bool OUT>
hipError_t launch_chunk(const FieldMove &f, long k0, long n, double *pinned) {
  const dim3 grid((unsigned)((n + kB - 1) / kB)), block(kB);
  auto go = [&](auto *dev, auto spin) {
    using T = std::remove_pointer_t<decltype(dev)>;
    constexpr bool S = decltype(spin)::value;
    if constexpr (OUT)
      hipLaunchKernelGGL((k_field_out<T, S>), grid, block, 0, nullptr, k0, n, f.rows, f.cnt, f.perm,
                         (const T *)dev, pinned);
    else
      hipLaunchKernelGGL((k_field_in<T, S>), grid, block, 0, nullptr, k0, n, f.rows, f.cnt, f.perm,
                         (const double *)pinned, dev);
  };
  if (f.f32) {
    if (f.spin) go((float *)f.dev, std::true_type());
    else go((float *)f.dev, std::false_type());
  } else {
    if (f.spin) go((double *)f.dev, std::true_type());
    else go((double *)f.dev, std::false_type());
  }
  return hipGetLastError();
}

// Threads that copy chunks between the ring and the caller's array: chunk c
// is handed out once ready exceeds c, and done[c] is set when its copy ended.
// Host memory only; every GPU call stays in the calling thread.
class Copiers {
 public:
  Copiers(long chunks, int threads, void (*copy)(void *, long), void *arg)
      : done_(chunks, 0), copy_(copy), arg_(arg) {
    try {
      for (int t = 0; t < threads; ++t) th_.emplace_back([this] { work(); });
    } catch (const std::exception &) {  // fewer threads (or none: the caller copies)
    }
  }
  ~Copiers() {
    {
      std::lock_guard<std::mutex> l(mu_);
      stop_ = true;
    }
    cv_.notify_all();
    for (auto &t : th_) t.join();
  }
  void hand_out(long upto) {  // chunks below upto may be copied
    if (th_.empty()) {
      for (; ready_ < upto; ++ready_) {
        copy_(arg_, ready_);
        done_[ready_] = 1;
      }
      return;
    }
    {
      std::lock_guard<std::mutex> l(mu_);
      ready_ = upto;
    }
    cv_.notify_all();
  }
  void wait(long c) {  // until chunk c (handed out before) is copied
    std::unique_lock<std::mutex> l(mu_);
    cv_done_.wait(l, [&] { return done_[c] != 0; });
  }

 private:
  void work() {
    for (;;) {
      long c;
      {
        std::unique_lock<std::mutex> l(mu_);
        cv_.wait(l, [&] { return stop_ || next_ < ready_; });
        if (next_ >= ready_) return;  // stopping, nothing handed out is left
        c = next_++;
      }
      copy_(arg_, c);
      {
        std::lock_guard<std::mutex> l(mu_);
        done_[c] = 1;
      }
      cv_done_.notify_one();
    }
  }
  std::vector<char> done_;
  long ready_ = 0, next_ = 0;
  void (*copy_)(void *, long);
  void *arg_;
  bool stop_ = false;
  std::mutex mu_;
  std::condition_variable cv_, cv_done_;
  std::vector<std::thread> th_;
};

struct CopyJob {
  char *ring, *user;
  long total;  // bytes
  bool out;
  static void run(void *p, long c) {
    const CopyJob &j = *static_cast<CopyJob *>(p);
    char *a = j.ring + (size_t)(c % kSlots) * kChunkBytes, *b = j.user + (size_t)c * kChunkBytes;
    const size_t n = std::min<size_t>(kChunkBytes, (size_t)j.total - (size_t)c * kChunkBytes);
    if (j.out) std::memcpy(b, a, n);
    else std::memcpy(a, b, n);
  }
};

// Fields of more than kCopyFrom and up to kCopyTo bytes on the device, of at most
// kCopyItems items: one hipMemcpy, the transposition, permutation and conversion
// on the host.  The runtime copies up to 16 KiB by a way that takes 20 us, more in
// 8; above the other two lines the host's loop takes longer than a kernel and the
// wait for it.  us to read / set, this way and by the kernels: three components,
// 12,288 B 23.1 / 22.2 and 15.5 / 15.2, 17,496 B 11.9 / 11.5 and 15.6 / 15.3,
// 31,944 B 13.0 / 12.8 and 15.8 / 15.5, 52,728 B 15.0 / 14.7 and 16.5 / 15.9,
// 81,000 B 17.6 / 17.2 and 17.7 / 16.8; one component, 4096 items 14.8 / 14.4 and
// 16.2 / 15.7, 4913 items 15.9 / 16.4 and 16.3 / 15.6.
constexpr size_t kCopyFrom = 16 << 10, kCopyTo = 64 << 10;
constexpr long kCopyItems = 4500;
template <bool OUT, typename T>
int move_by_copy(const FieldMove &f, double *user) {
  const int skip = f.spin ? 3 : 0, dr = f.rows - skip;  // the spin's zero diagonal
  std::vector<T> t((size_t)dr * f.cnt);
  if (OUT) WFX_CHECK_HIP(hipMemcpy(t.data(), f.dev, t.size() * sizeof(T), hipMemcpyDeviceToHost));
  for (long i = 0; i < f.cnt; ++i) {
    double *u = user + i * f.rows;
    T *d = t.data() + (f.perm_h ? (long)f.perm_h[i] : i);
    for (int r = 0; OUT && r < skip; ++r) u[r] = 0.0;
    for (int r = 0; r < dr; ++r) {
      if (OUT) u[skip + r] = (double)d[r * f.cnt];
      else d[r * f.cnt] = (T)u[skip + r];
    }
  }
  if (!OUT) WFX_CHECK_HIP(hipMemcpy(f.dev, t.data(), t.size() * sizeof(T), hipMemcpyHostToDevice));
  return WFX_OK;
}

// The caller has synchronised the device and made it current.  Returns when the
// transfer is over.
template <bool OUT>
int move_field(wfx_ctx *c, const FieldMove &f, double *user) {
  const long values = f.cnt * f.rows, per = (long)(kChunkBytes / sizeof(double));
  if (values == 0) return WFX_OK;
  const size_t bytes = (size_t)f.cnt * (f.rows - (f.spin ? 3 : 0)) * (f.f32 ? sizeof(float) : sizeof(double));
  if (bytes > kCopyFrom && bytes <= kCopyTo && f.cnt <= kCopyItems)
    return f.f32 ? move_by_copy<OUT, float>(f, user) : move_by_copy<OUT, double>(f, user);
  const long chunks = (values + per - 1) / per;
  const StagingLease lease(c->device);
  Staging &s = *lease;
  int rc = staging_ready(s, chunks > 1);
  if (rc) return rc;
  if (chunks == 1 || !s.ring) {
    double *pin = (double *)s.small;
    for (long k = 0; k < chunks; ++k) {
      const long n = std::min(per, values - k * per);
      if (!OUT) std::memcpy(pin, user + k * per, n * sizeof(double));
      WFX_CHECK_HIP(launch_chunk<OUT>(f, k * per, n, pin));
      WFX_CHECK_HIP(hipStreamSynchronize(nullptr));
      if (OUT) std::memcpy(user + k * per, pin, n * sizeof(double));
    }
    return WFX_OK;
  }
  auto slot = [&](long k) { return (double *)(s.ring + (size_t)(k % kSlots) * kChunkBytes); };
  auto launch = [&](long k) {
    hipError_t e = launch_chunk<OUT>(f, k * per, std::min(per, values - k * per), slot(k));
    return e == hipSuccess ? hipEventRecord(s.ev[k % kSlots], nullptr) : e;
  };
  CopyJob job{s.ring, (char *)user, values * (long)sizeof(double), OUT};
  hipError_t err = hipSuccess;
  {
    Copiers cp(chunks, (int)std::min<long>(kCopyThreads, chunks), CopyJob::run, &job);
    if (OUT) {
      long sent = 0;
      for (long k = 0; k < chunks && err == hipSuccess; ++k) {
        for (; sent < chunks && sent < k + kSlots && err == hipSuccess; ++sent) {
          if (sent >= kSlots) cp.wait(sent - kSlots);  // handed out: sent - kSlots < k
          err = launch(sent);
        }
        if (err == hipSuccess) err = hipEventSynchronize(s.ev[k % kSlots]);
        if (err == hipSuccess) cp.hand_out(k + 1);
      }
    } else {
      cp.hand_out(std::min<long>(kSlots, chunks));
      for (long k = 0; k < chunks && err == hipSuccess; ++k) {
        cp.wait(k);
        err = launch(k);
        // the slot of chunk k takes chunk k + kSlots once the kernel has read
        // it; freed half a ring late, so that the copies stay ahead
        const long f0 = k - kSlots / 2;
        if (err == hipSuccess && f0 >= 0 && f0 + kSlots < chunks) {
          err = hipEventSynchronize(s.ev[f0 % kSlots]);
          if (err == hipSuccess) cp.hand_out(f0 + kSlots + 1);
        }
      }
    }
  }  // the copies handed out end here
  const hipError_t end = hipStreamSynchronize(nullptr);  // no kernel uses the ring any more
  WFX_CHECK_HIP(err);
  WFX_CHECK_HIP(end);
  return WFX_OK;
}

}  // namespace

// A restart clears 14 arrays and more: as memsets of their own they took
// 60 of the 130 us of a small mesh's wfx_init.
hipError_t launch_fill(const FillList &f, hipStream_t s) {
  if (f.count == 0) return hipSuccess;
  size_t most = 1;
  for (int k = 0; k < f.count; ++k) most = std::max(most, f.buf[k].words);
  const size_t blocks = std::min<size_t>((most / 4 + kB - 1) / kB + 1, 2048);
  hipLaunchKernelGGL(k_fill, dim3((unsigned)blocks, (unsigned)f.count), dim3(kB), 0, s, f);
  return hipGetLastError();
}

int field_to_host(wfx_ctx *c, const FieldMove &f, double *host) { return move_field<true>(c, f, host); }
int field_from_host(wfx_ctx *c, const FieldMove &f, const double *host) {
  return move_field<false>(c, f, const_cast<double *>(host));
}

}  // namespace wfx
