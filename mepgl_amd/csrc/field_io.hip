// Transfers between the host's field arrays, (F, N, N, 2) doubles with x
// fastest, and a string's device planes (common.hpp).
//
// The host arrays are cut into chunks of sites.  A worker takes a chunk at a
// time: on the way out, a kernel gathers the chunk's planes into the worker's
// pinned buffer in the host order and the storage type, and the worker copies
// (widens, in mixed precision) it to the caller's array; on the way in, the
// worker copies (rounds) the caller's values to its pinned buffer and a kernel
// scatters them to the planes.  The kernels read and write the pinned buffer
// across the bus themselves, so a chunk costs one launch and no device
// staging, and the bus carries the storage type.
//
// What bounds a transfer is the host: the caller's pages are touched for the
// first time, and one thread moves a few GB/s; hence several workers.  With
// the planes converted by one host thread and copied through pageable
// memory, 64 images of 256 x 256 sites took 73 ms in and 54 ms out in FP64
// (39 and 33 ms in mixed precision); this way 4-5 and 3.6 ms (3-4 and 3.2
// ms), 24 images of 160 x 160 7.0 and 5.4 ms against 0.9 and 0.8.  One worker
// per 16 MB of host arrays: beside a program whose own threads spin on every
// CPU, eight workers for 10 to 30 MB took 19 ms, mostly waiting for one of
// them to be scheduled, and two take 9.
#include "field_io.hpp"

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>
#include <vector>

namespace mepgl {

namespace {

constexpr int kIoBlock = 256;

struct SiteRange {
  int N;               // grid side
  unsigned r0;         // first site of the range within image n0, j * N + i
  int n0;
  unsigned count;      // sites
  long long pitch, ps, is;
};

__device__ __forceinline__ long long site_offset(const SiteRange& s, unsigned t) {
  const unsigned nn = (unsigned)s.N * (unsigned)s.N, r = s.r0 + t;
  const unsigned n = r / nn, q = r - n * nn, j = q / (unsigned)s.N, i = q - j * (unsigned)s.N;
  return (long long)(s.n0 + (int)n) * s.is + (long long)j * s.pitch + i;
}

template <class T, int C>
struct alignas(sizeof(T) * C) SiteValues {
  T v[C];
};

// Planes to the host order: one site per lane, its C values in one store.
template <class T, int C>
__global__ __launch_bounds__(kIoBlock) void k_gather_sites(SiteRange s, const T* src, T* out) {
  const unsigned t = blockIdx.x * kIoBlock + threadIdx.x;
  if (t >= s.count) return;
  const long long o = site_offset(s, t);
  SiteValues<T, C> w;
#pragma unroll
  for (int c = 0; c < C; ++c) w.v[c] = src[o + c * s.ps];
  ((SiteValues<T, C>*)out)[t] = w;
}

// Host order to the planes of one or two field sets.
template <class T, int C>
__global__ __launch_bounds__(kIoBlock) void k_scatter_sites(SiteRange s, const T* in, T* a, T* b) {
  const unsigned t = blockIdx.x * kIoBlock + threadIdx.x;
  if (t >= s.count) return;
  const long long o = site_offset(s, t);
  const SiteValues<T, C> w = ((const SiteValues<T, C>*)in)[t];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    a[o + c * s.ps] = w.v[c];
    if (b) b[o + c * s.ps] = w.v[c];
  }
}

// One chunk of one host array.
struct Chunk {
  int field;
  size_t first, count;  // sites, in the order (n, j, i)
};

std::vector<Chunk> chunks_of(const DevString& d, const HostField* f, int nf, size_t bytes) {
  const size_t sites = (size_t)d.F * d.N * d.N;
  std::vector<Chunk> out;
  for (int k = 0; k < nf; ++k) {
    const size_t per = std::max<size_t>(bytes / (f[k].count * sizeof(double)), 1);
    for (size_t s = 0; s < sites; s += per) out.push_back({k, s, std::min(per, sites - s)});
  }
  return out;
}

SiteRange range_of(const DevString& d, const Chunk& c) {
  const size_t nn = (size_t)d.N * d.N;
  SiteRange s;
  s.N = d.N;
  s.n0 = (int)(c.first / nn);
  s.r0 = (unsigned)(c.first % nn);
  s.count = (unsigned)c.count;
  s.pitch = d.pitch;
  s.ps = d.plane_stride;
  s.is = d.image_stride;
  return s;
}

int host_threads() {
  cpu_set_t set;
  CPU_ZERO(&set);
  return sched_getaffinity(0, sizeof set, &set) == 0 ? std::max(CPU_COUNT(&set), 1) : 1;
}

// Runs work(w) on up to `want` workers, the calling thread among them; a
// worker that cannot be started leaves its share to the others (they take
// chunks from a common counter).
template <class W>
void on_workers(int want, const W& work) {
  std::vector<std::thread> team;
  try {
    team.reserve((size_t)std::max(want - 1, 0));
    for (int w = 1; w < want; ++w) team.emplace_back([&work, w] { work(w); });
  } catch (...) {
  }
  work(0);
  for (auto& t : team) t.join();
}

hipError_t ensure_slot(FieldIo::Slot& s, size_t bytes) {
  for (auto& ev : s.done)
    if (!ev) {
      const hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
      if (e != hipSuccess) {
        ev = nullptr;
        return e;
      }
    }
  if (s.bytes >= bytes) return hipSuccess;
  if (s.host) (void)hipHostFree(s.host);
  s.host = nullptr;
  s.bytes = 0;
  const hipError_t e = hipHostMalloc(&s.host, 2 * bytes, hipHostMallocDefault);
  if (e != hipSuccess) {
    s.host = nullptr;
    return e;
  }
  s.bytes = bytes;
  return hipSuccess;
}

// Runs one worker(slot, w, take) per worker, take(chunk&) giving it the next
// chunk.  A string whose fields fit one small chunk gets buffers of that
// size; the chunks of a larger one are kSlotBytes.  Workers beyond the first
// are started for large transfers only, and dropped when their buffers cannot
// be had.
template <class F>
hipError_t transfer(FieldIo& io, const DevString& d, const HostField* f, int nf, int device,
                    const F& worker) {
  size_t most = 0, total = 0;
  for (int k = 0; k < nf; ++k) {
    const size_t n = (size_t)d.F * d.N * d.N * f[k].count * sizeof(double);
    most = std::max(most, n);
    total += n;
  }
  const size_t bytes = std::min(FieldIo::kSlotBytes, (most + 4095) / 4096 * 4096);
  const std::vector<Chunk> chunks = chunks_of(d, f, nf, bytes);
  const int want = (int)std::min<size_t>(
      {(size_t)FieldIo::kMaxWorkers, (size_t)host_threads(), total / FieldIo::kWorkerBytes + 1});
  int have = 0;
  hipError_t e = hipSuccess;
  while (have < want && (e = ensure_slot(io.slot[have], bytes)) == hipSuccess) ++have;
  if (have == 0) return e;
  if (have < want) (void)hipGetLastError();
  std::atomic<size_t> next{0};
  std::atomic<int> bad{(int)hipSuccess};
  on_workers(have, [&](int w) {
    auto take = [&](Chunk& c) {
      const size_t k = next.fetch_add(1);
      if (k < chunks.size()) c = chunks[k];
      return k < chunks.size();
    };
    hipError_t r = hipSetDevice(device);
    if (r == hipSuccess) r = worker(io.slot[w], w, take);
    if (r != hipSuccess) {
      bad.store((int)r);
      next.store(chunks.size());
    }
  });
  return (hipError_t)bad.load();
}

template <class T>
hipError_t gather(const SiteRange& s, const T* src, int count, T* out, hipStream_t st) {
  const dim3 g((s.count + kIoBlock - 1) / kIoBlock), b(kIoBlock);
  if (count == 2)
    hipLaunchKernelGGL((k_gather_sites<T, 2>), g, b, 0, st, s, src, out);
  else
    hipLaunchKernelGGL((k_gather_sites<T, 1>), g, b, 0, st, s, src, out);
  return hipGetLastError();
}

template <class T>
hipError_t scatter(const SiteRange& s, const T* in, int count, T* a, T* b2, hipStream_t st) {
  const dim3 g((s.count + kIoBlock - 1) / kIoBlock), b(kIoBlock);
  if (count == 2)
    hipLaunchKernelGGL((k_scatter_sites<T, 2>), g, b, 0, st, s, in, a, b2);
  else
    hipLaunchKernelGGL((k_scatter_sites<T, 1>), g, b, 0, st, s, in, a, b2);
  return hipGetLastError();
}

void copy_values(double* dst, const double* src, size_t n) { std::memcpy(dst, src, n * sizeof(double)); }
void copy_values(double* dst, const float* src, size_t n) {
  for (size_t k = 0; k < n; ++k) dst[k] = (double)src[k];
}
void copy_values(float* dst, const double* src, size_t n) {
  for (size_t k = 0; k < n; ++k) dst[k] = (float)src[k];
}

// Each worker has two buffers: while the kernel of one chunk runs, the worker
// copies the other's values.
template <class T>
hipError_t download_impl(FieldIo& io, const DevString& d, const T* dev, const HostField* f, int nf,
                         const hipStream_t* streams, int nstreams, int device) {
  return transfer(io, d, f, nf, device, [&](FieldIo::Slot& s, int w, auto& take) {
    const hipStream_t st = streams[w % nstreams];
    auto issue = [&](const Chunk& c, int b) {
      const HostField& h = f[c.field];
      const hipError_t e = gather<T>(range_of(d, c), dev + h.plane * d.plane_stride, h.count,
                                     (T*)s.buffer(b), st);
      return e == hipSuccess ? hipEventRecord(s.done[b], st) : e;
    };
    Chunk c[2];
    hipError_t e = hipSuccess;
    bool more = take(c[0]);
    if (more) e = issue(c[0], 0);
    for (int b = 0; more && e == hipSuccess; b ^= 1) {
      more = take(c[b ^ 1]);
      if (more) e = issue(c[b ^ 1], b ^ 1);
      const hipError_t w0 = hipEventSynchronize(s.done[b]);
      if (w0 != hipSuccess) return w0;
      const HostField& h = f[c[b].field];
      copy_values(h.host + c[b].first * h.count, (const T*)s.buffer(b), c[b].count * h.count);
    }
    return e;
  });
}

template <class T>
hipError_t upload_impl(FieldIo& io, const DevString& d, T* a, T* b2, const HostField* f, int nf,
                       const hipStream_t* streams, int nstreams, int device) {
  return transfer(io, d, f, nf, device, [&](FieldIo::Slot& s, int w, auto& take) {
    const hipStream_t st = streams[w % nstreams];
    Chunk c;
    hipError_t e = hipSuccess;
    bool busy[2] = {false, false};
    for (int b = 0; e == hipSuccess && take(c); b ^= 1) {
      if (busy[b] && (e = hipEventSynchronize(s.done[b])) != hipSuccess) break;
      const HostField& h = f[c.field];
      const long long o = h.plane * d.plane_stride;
      copy_values((T*)s.buffer(b), h.host + c.first * h.count, c.count * h.count);
      e = scatter<T>(range_of(d, c), (const T*)s.buffer(b), h.count, a + o, b2 ? b2 + o : nullptr, st);
      if (e == hipSuccess) e = hipEventRecord(s.done[b], st);
      busy[b] = true;
    }
    for (int b = 0; b < 2; ++b)
      if (busy[b]) {
        const hipError_t w0 = hipEventSynchronize(s.done[b]);
        if (e == hipSuccess) e = w0;
      }
    return e;
  });
}

}  // namespace

void FieldIo::release() {
  for (auto& s : slot) {
    if (s.host) (void)hipHostFree(s.host);
    for (auto ev : s.done)
      if (ev) (void)hipEventDestroy(ev);
    s = Slot();
  }
}

hipError_t download_fields(FieldIo& io, const DevString& d, const void* dev, bool fp32,
                           const HostField* f, int nf, const hipStream_t* streams, int nstreams,
                           int device) {
  return fp32 ? download_impl<float>(io, d, (const float*)dev, f, nf, streams, nstreams, device)
              : download_impl<double>(io, d, (const double*)dev, f, nf, streams, nstreams, device);
}

hipError_t upload_fields(FieldIo& io, const DevString& d, void* const* dev, int ndev, bool fp32,
                         const HostField* f, int nf, const hipStream_t* streams, int nstreams,
                         int device) {
  void* b = ndev > 1 ? dev[1] : nullptr;
  return fp32 ? upload_impl<float>(io, d, (float*)dev[0], (float*)b, f, nf, streams, nstreams, device)
              : upload_impl<double>(io, d, (double*)dev[0], (double*)b, f, nf, streams, nstreams,
                                    device);
}

bool images_equal(const double* a, int F, size_t image) {
  std::atomic<int> next{1};
  std::atomic<bool> same{true};
  const size_t total = (size_t)F * image * sizeof(double);
  const int want = (int)std::min<size_t>({(size_t)FieldIo::kMaxWorkers, (size_t)host_threads(),
                                          total / FieldIo::kWorkerBytes + 1});
  on_workers(want, [&](int) {
    for (int n; same.load() && (n = next.fetch_add(1)) < F;)
      if (std::memcmp(a, a + (size_t)n * image, image * sizeof(double)) != 0) same.store(false);
  });
  return same.load();
}

}  // namespace mepgl
