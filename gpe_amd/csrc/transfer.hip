// transfer.hip -- fields between host arrays and device storage.
//
// A field crosses PCIe through page-locked staging buffers: the device
// converts between its storage form and the host array's type as it reads or
// writes them, and a few host threads move the data between them and the
// caller's array, each part while the next ones are on the bus.  The bus
// moves 57 GB/s each way on this machine; one hipMemcpy to or from a pageable
// array moves 18 to 28 GB/s once the array's pages exist, and 4 GB/s into an
// array that is written for the first time, because one host thread then also
// takes every page fault (eight threads reach 22 GB/s with small pages, 72 with
// huge ones).
#include <hip/hip_runtime.h>

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "host_common.h"

namespace gpe {
namespace {

// ---- conversions -------------------------------------------------------------
// Storage form to host type: complex128 gets hi + lo in double, complex64
// fl32(hi + lo); and back: hi = fl32(v), lo = fl32(v - hi) of the compensated
// form (0 from complex64).  One real word per step; n counts them.

__global__ void __launch_bounds__(256) f32_to_f64(const float *__restrict__ hi, const float *__restrict__ lo,
                                                  double *__restrict__ out, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    out[i] = (double)hi[i] + (double)(lo ? lo[i] : 0.0f);
}
__global__ void __launch_bounds__(256) pair_to_f32(const float *__restrict__ hi, const float *__restrict__ lo,
                                                   float *__restrict__ out, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    out[i] = (float)((double)hi[i] + (double)lo[i]);
}
__global__ void __launch_bounds__(256) f64_to_f32(const double *__restrict__ v, float *__restrict__ out, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) out[i] = (float)v[i];
}
__global__ void __launch_bounds__(256) f64_to_pair(const double *__restrict__ v, float *__restrict__ hi,
                                                   float *__restrict__ lo, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const double s = v[i];
    const float h = (float)s;
    hi[i] = h;
    if (lo) lo[i] = (float)(s - (double)h);
  }
}
__global__ void __launch_bounds__(256) fill_zero(float *__restrict__ p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = 0.0f;
}
int blocks_for(size_t n) { return (int)std::min<size_t>((n + 255) / 256, 1024); }

// ---- staging -----------------------------------------------------------------
constexpr size_t kChunk = (size_t)8 << 20;  // bytes of one staging buffer
constexpr int kSlots = 4;
constexpr int kThreads = 8;                   // that move host data, the caller's among them
constexpr size_t kShare = (size_t)256 << 10;  // least bytes worth a thread

// Helper threads of one transfer at a time.
class Team {
 public:
  ~Team() {
    {
      std::lock_guard<std::mutex> l(m_);
      quit_ = true;
      ++round_;
    }
    cv_.notify_all();
    for (std::thread &t : th_) t.join();
  }
  // f(part, parts) for every part, the caller's part 0 included
  void run(int parts, const std::function<void(int, int)> &f) {
    if (parts > 1 && !started_) start();
    parts = std::min(parts, (int)th_.size() + 1);
    if (parts > 1) {
      std::lock_guard<std::mutex> l(m_);
      f_ = &f;
      parts_ = parts;
      left_.store(parts - 1, std::memory_order_relaxed);
      round_.store(round_.load(std::memory_order_relaxed) + 1, std::memory_order_release);
    }
    if (parts > 1) cv_.notify_all();
    f(0, parts);
    while (parts > 1 && left_.load(std::memory_order_acquire) > 0) __builtin_ia32_pause();
  }

 private:
  // the first transfer that shares its bytes out starts the helpers
  void start() {
    started_ = true;
    cpu_set_t set;
    int cpus = kThreads;
    if (sched_getaffinity(0, sizeof set, &set) == 0) cpus = CPU_COUNT(&set);
    try {
      for (int i = 1; i < std::min(kThreads, cpus); ++i) th_.emplace_back([this, i] { work(i); });
    } catch (const std::system_error &) {
      // fewer helpers
    }
  }
  void work(int me) {
    uint64_t seen = 0;
    for (;;) {
      // a transfer's chunks follow one another within some 100 us
      for (int i = 0; i < 4000 && round_.load(std::memory_order_acquire) == seen; ++i) __builtin_ia32_pause();
      const std::function<void(int, int)> *f = nullptr;
      int parts = 0;
      {
        std::unique_lock<std::mutex> l(m_);
        cv_.wait(l, [&] { return round_.load(std::memory_order_relaxed) != seen; });
        seen = round_.load(std::memory_order_relaxed);
        if (quit_) return;
        f = f_;
        parts = parts_;
      }
      if (me < parts) {
        (*f)(me, parts);
        left_.fetch_sub(1, std::memory_order_release);
      }
    }
  }
  std::vector<std::thread> th_;
  std::mutex m_;
  std::condition_variable cv_;
  std::atomic<uint64_t> round_{0};
  std::atomic<int> left_{0};
  const std::function<void(int, int)> *f_ = nullptr;
  int parts_ = 0;
  bool quit_ = false, started_ = false;
};

struct Stage {
  int device = 0;
  hipStream_t s = nullptr;
  char *buf[kSlots] = {};
  size_t room[kSlots] = {};
  hipEvent_t done[kSlots] = {};
  Team team;
  bool ok = false;
  Stage() {
    ok = hipGetDevice(&device) == hipSuccess && hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess;
    for (int i = 0; i < kSlots && ok; ++i) ok = hipEventCreateWithFlags(&done[i], hipEventDisableTiming) == hipSuccess;
  }
  // Buffers for a transfer of `bytes`, no more than it fills: 32 MiB of locked
  // pages take 10 ms to get, a small field moves in a fraction of that.  Called
  // with the stream idle.
  bool reserve(size_t bytes) {
    for (int i = 0; i < kSlots && (size_t)i * kChunk < bytes; ++i) {
      size_t want = (size_t)256 << 10;
      while (want < std::min(kChunk, bytes - (size_t)i * kChunk)) want *= 2;
      if (room[i] >= want) continue;
      if (buf[i]) (void)hipHostFree(buf[i]);
      buf[i] = nullptr;
      room[i] = 0;
      if (hipHostMalloc((void **)&buf[i], want, hipHostMallocDefault) != hipSuccess) return false;
      room[i] = want;
    }
    return true;
  }
  ~Stage() {
    if (s) (void)hipStreamSynchronize(s);
    for (int i = 0; i < kSlots; ++i) {
      if (buf[i]) (void)hipHostFree(buf[i]);
      if (done[i]) (void)hipEventDestroy(done[i]);
    }
    if (s) (void)hipStreamDestroy(s);
  }
};

// Stages wait here between transfers (two at most; a transfer that finds none
// makes its own) while contexts or batches live, and go with the last of them.
std::mutex g_mu;
std::vector<Stage *> g_idle;
int g_users = 0;

Stage *take_stage() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  {
    std::lock_guard<std::mutex> l(g_mu);
    for (size_t i = 0; i < g_idle.size(); ++i)
      if (g_idle[i]->device == dev) {
        Stage *st = g_idle[i];
        g_idle.erase(g_idle.begin() + i);
        return st;
      }
  }
  Stage *st = new (std::nothrow) Stage();
  if (st && !st->ok) {
    delete st;
    st = nullptr;
  }
  return st;
}

void give_stage(Stage *st) {
  {
    std::lock_guard<std::mutex> l(g_mu);
    if (st->ok && g_users > 0 && g_idle.size() < 2) {
      g_idle.push_back(st);
      return;
    }
  }
  delete st;
}

struct Lease {
  Stage *st;
  explicit Lease(bool wanted = true) : st(wanted ? take_stage() : nullptr) {}
  ~Lease() {
    if (st) give_stage(st);
  }
};

// Parts of a host array's bytes, to as many threads as its size is worth.
int parts_of(size_t bytes) { return (int)std::min<size_t>(kThreads, std::max<size_t>(1, bytes / kShare)); }
size_t part_begin(size_t bytes, int p, int n) { return p == n ? bytes : (bytes / n * p) & ~(size_t)63; }

// Host side of a transfer: bytes [at, at + len) of the host array's field,
// planes of `plane` bytes that lie `pitch` bytes apart.
struct HostField {
  char *base;
  size_t plane, pitch;
  void piece(char *buf, size_t at, size_t len, bool out) const {
    while (len) {
      const size_t k = at / plane, r = at - k * plane, m = std::min(len, plane - r);
      char *h = base + k * pitch + r;
      out ? std::memcpy(h, buf, m) : std::memcpy(buf, h, m);
      buf += m;
      at += m;
      len -= m;
    }
  }
  void move(Team &team, char *buf, size_t at, size_t len, bool out) const {
    team.run(parts_of(len), [&](int p, int n) {
      const size_t a = part_begin(len, p, n), b = part_begin(len, p + 1, n);
      piece(buf + a, at + a, b - a, out);
    });
  }
};

// Move `bytes` of a field through the reserved staging buffers.  bus(buf, at,
// len) puts the device work of bytes [at, at + len) on the stage's stream.
template <typename Bus>
int through(Stage &st, const HostField &h, size_t bytes, bool out, Bus bus) {
  const size_t n = (bytes + kChunk - 1) / kChunk;
  auto put = [&](size_t i) {
    const size_t at = i * kChunk;
    hipError_t e = bus(st.buf[i % kSlots], at, std::min(kChunk, bytes - at));
    return e != hipSuccess ? e : hipEventRecord(st.done[i % kSlots], st.s);
  };
  hipError_t e = hipSuccess;
  if (out)
    for (size_t i = 0; i < std::min<size_t>(n, kSlots) && e == hipSuccess; ++i) e = put(i);
  for (size_t i = 0; i < n && e == hipSuccess; ++i) {
    const size_t at = i * kChunk, len = std::min(kChunk, bytes - at);
    if (out || i >= kSlots) e = hipEventSynchronize(st.done[i % kSlots]);
    if (e != hipSuccess) break;
    h.move(st.team, st.buf[i % kSlots], at, len, out);
    if (!out)
      e = put(i);
    else if (i + kSlots < n)
      e = put(i + kSlots);
  }
  const hipError_t w = hipStreamSynchronize(st.s);
  if (e == hipSuccess) e = w;
  if (e != hipSuccess) {
    st.ok = false;
    return fail(GPE_EHIP, "field transfer: %s", hipGetErrorString(e));
  }
  return GPE_OK;
}

// ---- without page-locked memory ----------------------------------------------
// Where none is to be had (a limit on locked pages, a host short of memory), a
// field moves by synchronous copies of the caller's pages, converted here in
// pieces of kPlainWords.
constexpr size_t kPlainWords = (size_t)1 << 18;

int plain_upload(const HostField &h, size_t bytes, bool split, void *hi, void *lo) {
  constexpr size_t word = 8;  // of a value that is split
  const size_t piece = split ? kPlainWords * word : h.plane == h.pitch ? bytes : h.plane;
  std::vector<double> v;
  std::vector<float> w;
  if (split) {
    v.resize(kPlainWords);
    w.resize(2 * kPlainWords);
  }
  for (size_t at = 0; at < bytes; at += piece) {
    const size_t len = std::min(piece, bytes - at);
    if (!split) {
      const size_t k = at / h.plane;
      GPE_HIPCHK(hipMemcpy((char *)hi + at, h.base + k * h.pitch, len, hipMemcpyHostToDevice));
      continue;
    }
    const size_t n = len / word;
    h.piece((char *)v.data(), at, len, false);
    float *whi = w.data(), *wlo = whi + kPlainWords;
    for (size_t i = 0; i < n; ++i) {
      whi[i] = (float)v[i];
      wlo[i] = (float)(v[i] - (double)whi[i]);
    }
    GPE_HIPCHK(hipMemcpy((float *)hi + at / word, whi, n * 4, hipMemcpyHostToDevice));
    if (lo) GPE_HIPCHK(hipMemcpy((float *)lo + at / word, wlo, n * 4, hipMemcpyHostToDevice));
  }
  if (lo && !split) {
    GPE_HIPCHK(hipMemset(lo, 0, bytes));
    GPE_HIPCHK(hipStreamSynchronize(nullptr));
  }
  return GPE_OK;
}

// stored: bytes of a stored word (hi's; lo: the compensated form's, or null);
// word: of a host word.
int plain_download(size_t stored, size_t word, size_t words, const void *hi, const void *lo, void *dst) {
  if (stored == word && !lo) {
    GPE_HIPCHK(hipMemcpy(dst, hi, words * word, hipMemcpyDeviceToHost));
    return GPE_OK;
  }
  std::vector<double> v(kPlainWords);
  std::vector<float> w(kPlainWords), l(kPlainWords, 0.0f);
  for (size_t at = 0; at < words; at += kPlainWords) {
    const size_t n = std::min(kPlainWords, words - at);
    if (stored == 8) {
      GPE_HIPCHK(hipMemcpy(v.data(), (const double *)hi + at, n * 8, hipMemcpyDeviceToHost));
    } else {
      GPE_HIPCHK(hipMemcpy(w.data(), (const float *)hi + at, n * 4, hipMemcpyDeviceToHost));
      if (lo) GPE_HIPCHK(hipMemcpy(l.data(), (const float *)lo + at, n * 4, hipMemcpyDeviceToHost));
      for (size_t i = 0; i < n; ++i) v[i] = (double)w[i] + (double)l[i];
    }
    if (word == 8)
      std::memcpy((double *)dst + at, v.data(), n * 8);
    else
      for (size_t i = 0; i < n; ++i) ((float *)dst)[at + i] = (float)v[i];
  }
  return GPE_OK;
}

template <typename F>
int plainly(F f) {
  (void)hipGetLastError();  // the refusal is not the next launch's error
  try {
    return f();
  } catch (const std::bad_alloc &) {
    return fail(GPE_ENOMEM, "host memory of a field transfer");
  }
}

// A conversion kernel over n words on the stage's stream.
template <typename K, typename... V>
hipError_t launch(Stage &st, size_t n, K kernel, V... v) {
  hipLaunchKernelGGL(kernel, dim3(blocks_for(n)), dim3(256), 0, st.s, v..., n);
  return hipGetLastError();
}

}  // namespace

void transfers_retain() {
  std::lock_guard<std::mutex> l(g_mu);
  ++g_users;
}

void transfers_release() {
  std::vector<Stage *> gone;
  {
    std::lock_guard<std::mutex> l(g_mu);
    if (--g_users == 0) gone.swap(g_idle);
  }
  for (Stage *st : gone) delete st;
}

void host_parts(size_t bytes, const std::function<void(size_t, size_t)> &f) {
  const int parts = parts_of(bytes);
  Lease lease(parts > 1);
  if (!lease.st) return f(0, bytes);
  lease.st->team.run(parts, [&](int p, int n) { f(part_begin(bytes, p, n), part_begin(bytes, p + 1, n)); });
}

// Host array -> device storage.  src_pitch_planes: elements between
// z-planes of the host array; row_off: element offset of the interior's
// (0, 0, 0).  FP32 forms from complex128 split each value into hi = fl32(v)
// and lo = fl32(v - hi); complex64 into a compensated form sets lo = 0.
int field_upload(int prec, size_t plane, int nz, const void *src, int host_type, size_t src_pitch_planes,
                 size_t row_off, void *hi, void *lo) {
  if (host_type != GPE_HOST_C128 && host_type != GPE_HOST_C64) return fail(GPE_EINVAL, "unsupported host type");
  if (prec == GPE_FP64 && host_type != GPE_HOST_C128)
    return fail(GPE_EINVAL, "FP64 storage takes complex128 host data");
  const size_t esz = host_type == GPE_HOST_C128 ? 16 : 8, bytes = plane * (size_t)nz * esz;
  const bool comp = prec == GPE_FP32C, split = prec != GPE_FP64 && host_type == GPE_HOST_C128;
  const HostField h{(char *)const_cast<void *>(src) + row_off * esz, plane * esz, src_pitch_planes * esz};
  Lease lease;
  if (!lease.st || !lease.st->reserve(bytes))
    return plainly([&] { return plain_upload(h, bytes, split, hi, comp ? lo : nullptr); });
  Stage &st = *lease.st;
  if (comp && !split) {
    const size_t n = 2 * plane * (size_t)nz;
    GPE_HIPCHK(launch(st, n, fill_zero, (float *)lo));
  }
  return through(st, h, bytes, false, [&](char *buf, size_t at, size_t len) -> hipError_t {
    if (!split) return hipMemcpyAsync((char *)hi + at, buf, len, hipMemcpyHostToDevice, st.s);
    const size_t w = at / 8, n = len / 8;
    return launch(st, n, f64_to_pair, (const double *)buf, (float *)hi + w, comp ? (float *)lo + w : nullptr);
  });
}

// Device storage -> contiguous host array (complex128 gets hi + lo in
// double; complex64 gets fl32(hi + lo)).  The caller orders this after the
// kernels that wrote the field.
int field_download(int prec, size_t plane, int nz, const void *hi, const void *lo, void *dst, int host_type) {
  if (host_type != GPE_HOST_C128 && host_type != GPE_HOST_C64) return fail(GPE_EINVAL, "unsupported host type");
  if (prec == GPE_FP64 && host_type != GPE_HOST_C128)
    return fail(GPE_EINVAL, "FP64 storage returns complex128 host data");
  return words_download(prec == GPE_FP64 ? 16 : 8, plane * (size_t)nz, hi, prec == GPE_FP32C ? lo : nullptr, dst,
                        host_type);
}

int words_download(int stored, size_t sites, const void *hi, const void *lo, void *dst, int host_type) {
  const size_t esz = host_type == GPE_HOST_C128 ? 16 : 8, bytes = sites * esz;
  Lease lease;
  if (!lease.st || !lease.st->reserve(bytes))
    return plainly([&] { return plain_download(stored / 2, esz / 2, 2 * sites, hi, lo, dst); });
  Stage &st = *lease.st;
  const HostField h{(char *)dst, bytes, bytes};
  return through(st, h, bytes, true, [&](char *buf, size_t at, size_t len) -> hipError_t {
    if (stored == (int)esz && !lo) return hipMemcpyAsync(buf, (const char *)hi + at, len, hipMemcpyDeviceToHost, st.s);
    const size_t word = esz / 2, w = at / word, n = len / word;
    const float *l = lo ? (const float *)lo + w : nullptr;
    if (stored == 16) return launch(st, n, f64_to_f32, (const double *)hi + w, (float *)buf);
    if (esz == 16) return launch(st, n, f32_to_f64, (const float *)hi + w, l, (double *)buf);
    return launch(st, n, pair_to_f32, (const float *)hi + w, l, (float *)buf);
  });
}

}  // namespace gpe
