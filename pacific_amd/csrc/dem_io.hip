// Row transfers of the state (dem_io.hpp).
//
// One kernel turns the structure of arrays into rows by id (or back) in a
// device buffer, and the rows cross PCIe as one block.  A copy and a host loop
// per component, the way before, cost a synchronisation each: 395 us for the
// state of 500 bodies (now about 75), 34 ms for 1,000,000 (now 7: 176 MB, of
// which the bus takes 4 ms; one thread writing the caller's fresh pages took
// the rest), 146 ms for 512 batch members one by one (now 34).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

#include "dem_io.hpp"
#include "dem_math.hpp"

namespace dem {

__global__ __launch_bounds__(256) void k_rows_out(RowMap m, const int* __restrict__ id, int n,
                                                  double* __restrict__ out) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const unsigned i = (unsigned)(id[s] - 1);
  if (i >= (unsigned)n) return;
  for (int c = 0; c < m.nc; ++c) out[m.base[c] + (size_t)m.stride[c] * i] = m.comp[c][s];
}

__global__ __launch_bounds__(256) void k_rows_in(RowMap m, const int* __restrict__ id, int n,
                                                 const double* __restrict__ in) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const unsigned i = (unsigned)(id[s] - 1);
  if (i >= (unsigned)n) return;
  for (int c = 0; c < m.nc; ++c) m.comp[c][s] = in[m.base[c] + (size_t)m.stride[c] * i];
}

__global__ __launch_bounds__(256) void k_body_spin(Particles P, int n, int cv) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const quat q{d3{P.q[0][s], P.q[1][s], P.q[2][s]}, P.q[3][s]};
  const d3 wb = to_body(q, d3{P.w[cv][0][s], P.w[cv][1][s], P.w[cv][2][s]});
  P.wb[0][s] = wb.x;
  P.wb[1][s] = wb.y;
  P.wb[2][s] = wb.z;
}

hipError_t launch_rows_out(const RowMap& m, const int* id, int n, double* out, hipStream_t stream) {
  if (n == 0 || m.nc == 0) return hipSuccess;
  hipLaunchKernelGGL(k_rows_out, dim3((n + 255) / 256), dim3(256), 0, stream, m, id, n, out);
  return hipGetLastError();
}
hipError_t launch_rows_in(const RowMap& m, const int* id, int n, const double* in, hipStream_t stream) {
  if (n == 0 || m.nc == 0) return hipSuccess;
  hipLaunchKernelGGL(k_rows_in, dim3((n + 255) / 256), dim3(256), 0, stream, m, id, n, in);
  return hipGetLastError();
}
hipError_t launch_body_spin(const Particles& P, int n, int cv, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_body_spin, dim3((n + 255) / 256), dim3(256), 0, stream, P, n, cv);
  return hipGetLastError();
}

template <class T>
struct ArrayGroup {
  T* a[kPermuteGroup];
};
// blockIdx.y selects the array; gather into tmp, then back
template <class T>
__global__ __launch_bounds__(256) void k_permute(ArrayGroup<T> g, const int* __restrict__ order, int n,
                                                 T* __restrict__ tmp, bool back) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  T* const t = tmp + (size_t)blockIdx.y * n;
  if (back) {
    g.a[blockIdx.y][i] = t[i];
  } else {
    const int o = order[i];
    t[i] = g.a[blockIdx.y][(unsigned)o < (unsigned)n ? o : i];
  }
}
template <class T>
static hipError_t permute_arrays(const std::vector<T*>& a, const int* order, int n, T* tmp, hipStream_t stream) {
  for (size_t k = 0; k < a.size(); k += kPermuteGroup) {
    ArrayGroup<T> g{};
    const int m = (int)std::min<size_t>(kPermuteGroup, a.size() - k);
    for (int j = 0; j < m; ++j) g.a[j] = a[k + j];
    for (int back = 0; back < 2; ++back)
      hipLaunchKernelGGL(k_permute<T>, dim3((n + 255) / 256, m), dim3(256), 0, stream, g, order, n, tmp, back != 0);
  }
  return hipGetLastError();
}
hipError_t launch_permute(const std::vector<double*>& a8, const std::vector<int*>& a4, const int* order, int n,
                          double* tmp, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipError_t e = permute_arrays(a8, order, n, tmp, stream);
  return e == hipSuccess ? permute_arrays(a4, order, n, (int*)tmp, stream) : e;
}

namespace {

// Up to kSingle bytes cross as one copy through one pinned slice; more is cut
// into chunks that up to kThreads threads copy, each with two pinned slices
// and a stream of its own: writing the caller's (often fresh) pages is what
// takes the time, and threads share it.
constexpr size_t kSingle = (size_t)2 << 20;
constexpr size_t kChunk = (size_t)1 << 20;
constexpr int kThreads = 8;

struct Chunk {
  char* host;
  size_t off, bytes;  // offset in the row buffer
};

}  // namespace

void RowBuffers::release() {
  if (dev_) (void)hipFree(dev_);
  if (pin_) (void)hipHostFree(pin_);
  for (auto s : lanes_) (void)hipStreamDestroy(s);
  dev_ = nullptr;
  pin_ = nullptr;
  dev_cap_ = pin_cap_ = 0;
  lanes_.clear();
}

// How many threads copy a part, and the pinned bytes it needs.
static int copy_threads(size_t total) {
  if (total <= kSingle) return 0;
  return (int)std::min<size_t>({(size_t)kThreads, total / kChunk,
                                (size_t)std::max(1u, std::thread::hardware_concurrency() / 2)});
}

hipError_t RowBuffers::reserve(const RowIO& io, size_t first, size_t last, hipStream_t stream) {
  size_t total = 0;
  for (size_t k = first; k < last; ++k) total += io.segs()[k].count * sizeof(double);
  const int nthreads = copy_threads(total);
  const size_t pinned = nthreads ? (size_t)nthreads * 2 * kChunk : std::max<size_t>(total, 4096);
  if (total <= dev_cap_ && pinned <= pin_cap_) return hipSuccess;
  // what was enqueued before may still use the buffers
  hipError_t e = hipStreamSynchronize(stream);
  if (e != hipSuccess) return e;
  if (total > dev_cap_) {
    if (dev_) (void)hipFree(dev_);
    dev_ = nullptr;
    dev_cap_ = 0;
    if ((e = hipMalloc((void**)&dev_, total)) != hipSuccess) return e;
    dev_cap_ = total;
  }
  if (pinned > pin_cap_) {
    if (pin_) (void)hipHostFree(pin_);
    pin_ = nullptr;
    pin_cap_ = 0;
    if ((e = hipHostMalloc((void**)&pin_, pinned, hipHostMallocDefault)) != hipSuccess) return e;
    pin_cap_ = pinned;
  }
  return e;
}

hipError_t RowBuffers::copy(const RowIO& io, size_t first, size_t last, bool to_host, int device, hipStream_t stream) {
  size_t total = 0;
  for (size_t k = first; k < last; ++k) total += io.segs()[k].count * sizeof(double);
  const int nthreads = copy_threads(total);
  if (!nthreads) {
    if (to_host) {
      hipError_t e = hipMemcpyAsync(pin_, dev_, total, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipStreamSynchronize(stream);
      if (e != hipSuccess) return e;
      const char* from = pin_;
      for (size_t k = first; k < last; from += io.segs()[k++].count * sizeof(double))
        std::memcpy(io.segs()[k].host, from, io.segs()[k].count * sizeof(double));
      return hipSuccess;
    }
    char* to = pin_;
    for (size_t k = first; k < last; to += io.segs()[k++].count * sizeof(double))
      std::memcpy(to, io.segs()[k].host, io.segs()[k].count * sizeof(double));
    return hipMemcpyAsync(dev_, pin_, total, hipMemcpyHostToDevice, stream);
  }
  while ((int)lanes_.size() < nthreads) {
    hipStream_t st;
    hipError_t e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
    if (e != hipSuccess) return e;
    lanes_.push_back(st);
  }
  const hipError_t drained = hipStreamSynchronize(stream);
  if (drained != hipSuccess) return drained;
  std::vector<Chunk> chunks;
  size_t off = 0;
  for (size_t k = first; k < last; ++k) {
    const size_t bytes = io.segs()[k].count * sizeof(double);
    for (size_t o = 0; o < bytes; o += kChunk)
      chunks.push_back(Chunk{(char*)io.segs()[k].host + o, off + o, std::min(kChunk, bytes - o)});
    off += bytes;
  }
  std::atomic<int> next{0};
  std::atomic<int> error{(int)hipSuccess};
  const int nc = (int)chunks.size();
  auto work = [&](int t) {
    hipError_t e = hipSetDevice(device);
    char* slice[2] = {pin_ + (size_t)(2 * t) * kChunk, pin_ + (size_t)(2 * t + 1) * kChunk};
    char* const d = (char*)dev_;
    int held = -1, h = 0;  // to_host: the chunk on its way into slice[h ^ 1]
    for (;;) {
      const int c = e == hipSuccess ? next.fetch_add(1) : nc;
      if (to_host) {
        // the copy of the next chunk runs while this thread empties the last
        if (held >= 0) e = hipStreamSynchronize(lanes_[t]);
        if (c < nc && e == hipSuccess)
          e = hipMemcpyAsync(slice[h], d + chunks[c].off, chunks[c].bytes, hipMemcpyDeviceToHost, lanes_[t]);
        if (held >= 0 && e == hipSuccess) std::memcpy(chunks[held].host, slice[h ^ 1], chunks[held].bytes);
        held = c < nc ? c : -1;
      } else if (c < nc) {
        std::memcpy(slice[h], chunks[c].host, chunks[c].bytes);
        // the other slice is free once its copy, enqueued before, is done
        if (e == hipSuccess) e = hipStreamSynchronize(lanes_[t]);
        if (e == hipSuccess)
          e = hipMemcpyAsync(d + chunks[c].off, slice[h], chunks[c].bytes, hipMemcpyHostToDevice, lanes_[t]);
      }
      h ^= 1;
      if (c >= nc) break;
    }
    const hipError_t es = hipStreamSynchronize(lanes_[t]);
    if (e == hipSuccess) e = es;
    if (e != hipSuccess) error.store((int)e);
  };
  std::vector<std::thread> pool;
  for (int t = 1; t < nthreads; ++t) {
    try {
      pool.emplace_back(work, t);
    } catch (...) {
      break;  // no more threads: the others take its chunks
    }
  }
  work(0);
  for (auto& p : pool) p.join();
  return (hipError_t)error.load();
}

hipError_t RowBuffers::plain(const RowIO& io, size_t first, bool to_host, const int* id, int n, hipStream_t stream) {
  (void)hipGetLastError();  // the allocation that failed
  hipError_t e = hipStreamSynchronize(stream);
  std::vector<int> ids((size_t)n);
  std::vector<double> buf((size_t)n);
  if (e == hipSuccess) e = hipMemcpy(ids.data(), id, sizeof(int) * n, hipMemcpyDeviceToHost);
  for (size_t k = first; e == hipSuccess && k < io.segs().size(); ++k) {
    const RowIO::Seg& s = io.segs()[k];
    for (int c = 0; c < s.width && e == hipSuccess; ++c) {
      auto row = [&](int i) -> double& { return s.host[(size_t)s.width * (ids[i] - 1) + c]; };
      if (to_host) {
        e = hipMemcpy(buf.data(), s.comp[c], sizeof(double) * n, hipMemcpyDeviceToHost);
        if (e == hipSuccess)
          for (int i = 0; i < n; ++i) row(i) = buf[i];
      } else {
        for (int i = 0; i < n; ++i) buf[i] = row(i);
        e = hipMemcpy(s.comp[c], buf.data(), sizeof(double) * n, hipMemcpyHostToDevice);
      }
    }
  }
  return e;
}

hipError_t RowBuffers::down(const RowIO& io, const int* id, int n, int device, hipStream_t stream) {
  if (io.segs().empty()) return hipStreamSynchronize(stream);
  hipError_t e = hipSuccess;
  for (size_t k = 0, l; k < io.segs().size() && e == hipSuccess; k = l) {
    l = io.part(k);
    e = reserve(io, k, l, stream);
    if (e == hipErrorOutOfMemory) return plain(io, k, true, id, n, stream);
    if (e == hipSuccess) e = launch_rows_out(io.map(k, l), id, n, dev_, stream);
    if (e == hipSuccess) e = copy(io, k, l, true, device, stream);
  }
  return e;
}

hipError_t RowBuffers::up(const RowIO& io, const int* id, int n, int device, hipStream_t stream) {
  hipError_t e = hipSuccess;
  for (size_t k = 0, l; k < io.segs().size() && e == hipSuccess; k = l) {
    l = io.part(k);
    // the buffers may still be read by what an earlier call or part enqueued
    e = hipStreamSynchronize(stream);
    if (e == hipSuccess) e = reserve(io, k, l, stream);
    if (e == hipErrorOutOfMemory) return plain(io, k, false, id, n, stream);
    if (e == hipSuccess) e = copy(io, k, l, false, device, stream);
    if (e == hipSuccess) e = launch_rows_in(io.map(k, l), id, n, dev_, stream);
  }
  return e;
}

}  // namespace dem
