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
#include <map>
#include <thread>

#include "dem_io.hpp"
#include "dem_math.hpp"

namespace dem {

std::mutex& capture_lock() {
  static std::mutex m;
  return m;
}
hipError_t copy_sync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind) {
  std::lock_guard<std::mutex> hold(capture_lock());
  return hipMemcpy(dst, src, bytes, kind);
}
hipError_t fill_sync(void* dst, int value, size_t bytes) {
  std::lock_guard<std::mutex> hold(capture_lock());
  return hipMemset(dst, value, bytes);
}

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
// into chunks that up to kThreads threads copy, each with two pinned slices:
// writing the caller's (often fresh) pages is what takes the time, and threads
// share it.  The copies go through the system's stream and kLanes of the
// buffers' own, which the first calls make one by one: a stream costs 0.7 ms
// until its first copy is done, 3 early in a process, against 0.35 ms for a
// whole state of 27,000 (a state of 1M: 5.5 ms through the system's stream
// alone, 4.8 with four; one stream and chunks of 2 MB are as fast there, but 3 %
// of a pass of 200,000 slower).
constexpr size_t kSingle = (size_t)2 << 20;
constexpr size_t kChunk = (size_t)1 << 20;
constexpr int kThreads = 8;
constexpr int kLanes = 4;
constexpr int kStatusBlocks = 128;  // per page

struct Chunk {
  char* host;
  size_t off, bytes;  // offset in the row buffer
};

size_t part_bytes(const RowIO& io, size_t first, size_t last) {
  size_t total = 0;
  for (size_t k = first; k < last; ++k) total += io.segs()[k].count * sizeof(double);
  return total;
}

// How many threads copy a part of so many bytes (0: one copy).
int copy_threads(size_t total) {
  if (total <= kSingle) return 0;
  return (int)std::min<size_t>({(size_t)kThreads, total / kChunk,
                                (size_t)std::max(1u, std::thread::hardware_concurrency() / 2)});
}

}  // namespace

std::shared_ptr<RowBuffers> RowBuffers::of(int device) {
  static std::mutex m;
  static std::map<int, std::weak_ptr<RowBuffers>> made;
  std::lock_guard<std::mutex> hold(m);
  auto& w = made[device];
  std::shared_ptr<RowBuffers> p = w.lock();
  if (!p) w = p = std::make_shared<RowBuffers>(device);
  return p;
}

RowBuffers::~RowBuffers() {
  if (dev_) (void)hipFree(dev_);
  if (pin_) (void)hipHostFree(pin_);
  for (auto p : pages_) (void)hipHostFree(p);
  for (auto e : copied_) (void)hipEventDestroy(e);
  for (auto s : lanes_) (void)hipStreamDestroy(s);
  if (read_) (void)hipEventDestroy(read_);
}

DevStatus* RowBuffers::status_block() {
  std::lock_guard<std::mutex> hold(blocks_);
  if (free_.empty()) {
    DevStatus* page = nullptr;
    if (hipHostMalloc((void**)&page, kStatusBlocks * sizeof(DevStatus), hipHostMallocDefault) == hipSuccess) {
      pages_.push_back(page);
    } else {  // ordinary memory: copies to it are staged
      (void)hipGetLastError();
      plain_.emplace_back(new DevStatus[kStatusBlocks]);
      page = plain_.back().get();
    }
    for (int i = kStatusBlocks; i-- > 0;) free_.push_back(page + i);
  }
  DevStatus* p = free_.back();
  free_.pop_back();
  return p;
}

void RowBuffers::give_back(DevStatus* p) {
  std::lock_guard<std::mutex> hold(blocks_);
  free_.push_back(p);
}

hipError_t RowBuffers::reserve(const RowIO& io, size_t first, size_t last) {
  const size_t total = part_bytes(io, first, last);
  const int nthreads = copy_threads(total);
  const size_t pinned =
      nthreads ? (size_t)nthreads * 2 * kChunk : (total <= kSingle / 8 ? kSingle / 8 : kSingle);
  // what an earlier call or part put into the buffers has to have been read
  hipError_t e = in_use_ ? hipEventSynchronize(read_) : hipSuccess;
  if (e != hipSuccess) return e;
  in_use_ = false;
  if (!read_ && (e = hipEventCreateWithFlags(&read_, hipEventDisableTiming)) != hipSuccess) return e;
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
  if (nthreads && copied_.empty()) {
    for (int t = 0; t < kThreads; ++t) {
      hipEvent_t ev;
      if ((e = hipEventCreateWithFlags(&ev, hipEventDisableTiming)) != hipSuccess) return e;
      copied_.push_back(ev);
    }
  } else if (nthreads && lanes_.size() < kLanes) {
    hipStream_t st;
    if ((e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking)) != hipSuccess) return e;
    lanes_.push_back(st);
  }
  return hipSuccess;
}

hipError_t RowBuffers::copy(const RowIO& io, size_t first, size_t last, bool to_host, hipStream_t stream) {
  const size_t total = part_bytes(io, first, last);
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
  // the lanes follow what the stream holds; rows that go to the device, the
  // stream follows the lanes, each thread having waited for its last copy
  if (!lanes_.empty()) {
    const hipError_t e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return e;
  }
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
    hipError_t e = hipSetDevice(device_);
    const size_t l = t % (lanes_.size() + 1);
    const hipStream_t lane = l ? lanes_[l - 1] : stream;
    char* slice[2] = {pin_ + (size_t)(2 * t) * kChunk, pin_ + (size_t)(2 * t + 1) * kChunk};
    char* const d = (char*)dev_;
    int held = -1, h = 0;  // held: the chunk whose copy, in slice[h ^ 1], was enqueued last
    for (;;) {
      const int c = e == hipSuccess ? next.fetch_add(1) : nc;
      if (!to_host && c < nc) std::memcpy(slice[h], chunks[c].host, chunks[c].bytes);
      if (held >= 0 && e == hipSuccess) e = hipEventSynchronize(copied_[t]);
      if (c < nc && e == hipSuccess) {
        e = to_host ? hipMemcpyAsync(slice[h], d + chunks[c].off, chunks[c].bytes, hipMemcpyDeviceToHost, lane)
                    : hipMemcpyAsync(d + chunks[c].off, slice[h], chunks[c].bytes, hipMemcpyHostToDevice, lane);
        if (e == hipSuccess) e = hipEventRecord(copied_[t], lane);
      }
      // to the host: while that copy runs, this thread empties the one before
      if (to_host && held >= 0 && e == hipSuccess)
        std::memcpy(chunks[held].host, slice[h ^ 1], chunks[held].bytes);
      held = c < nc ? c : -1;
      h ^= 1;
      if (c >= nc) break;
    }
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
  if (error.load() != (int)hipSuccess)  // a copy may have been left under way
    for (auto l : lanes_) (void)hipStreamSynchronize(l);
  return (hipError_t)error.load();
}

hipError_t RowBuffers::plain(const RowIO& io, size_t first, bool to_host, const int* id, int n, hipStream_t stream) {
  (void)hipGetLastError();  // the allocation that failed
  std::vector<int> ids((size_t)n);
  std::vector<double> buf((size_t)n);
  hipError_t e = hipStreamSynchronize(stream);
  if (e == hipSuccess) e = dem::copy_sync(ids.data(), id, sizeof(int) * n, hipMemcpyDeviceToHost);
  for (size_t k = first; e == hipSuccess && k < io.segs().size(); ++k) {
    const RowIO::Seg& s = io.segs()[k];
    for (int c = 0; c < s.width && e == hipSuccess; ++c) {
      auto row = [&](int i) -> double& { return s.host[(size_t)s.width * (ids[i] - 1) + c]; };
      if (to_host) {
        e = dem::copy_sync(buf.data(), s.comp[c], sizeof(double) * n, hipMemcpyDeviceToHost);
        if (e == hipSuccess)
          for (int i = 0; i < n; ++i) row(i) = buf[i];
      } else {
        for (int i = 0; i < n; ++i) buf[i] = row(i);
        e = dem::copy_sync(s.comp[c], buf.data(), sizeof(double) * n, hipMemcpyHostToDevice);
      }
    }
  }
  return e;
}

hipError_t RowBuffers::down(const RowIO& io, const int* id, int n, hipStream_t stream) {
  if (io.segs().empty()) return hipStreamSynchronize(stream);
  std::lock_guard<std::mutex> hold(use_);
  hipError_t e = hipSuccess;
  for (size_t k = 0, l; k < io.segs().size() && e == hipSuccess; k = l) {
    l = io.part(k);
    e = reserve(io, k, l);
    if (e == hipErrorOutOfMemory) return plain(io, k, true, id, n, stream);
    if (e == hipSuccess) e = launch_rows_out(io.map(k, l), id, n, dev_, stream);
    if (e == hipSuccess) e = copy(io, k, l, true, stream);
    if (e != hipSuccess) (void)hipStreamSynchronize(stream);
  }
  return e;
}

hipError_t RowBuffers::up(const RowIO& io, const int* id, int n, hipStream_t stream) {
  std::lock_guard<std::mutex> hold(use_);
  hipError_t e = hipSuccess;
  for (size_t k = 0, l; k < io.segs().size() && e == hipSuccess; k = l) {
    l = io.part(k);
    e = reserve(io, k, l);
    if (e == hipErrorOutOfMemory) return plain(io, k, false, id, n, stream);
    if (e == hipSuccess) e = copy(io, k, l, false, stream);
    if (e == hipSuccess) e = launch_rows_in(io.map(k, l), id, n, dev_, stream);
    if (e == hipSuccess) e = hipEventRecord(read_, stream);
    if (e == hipSuccess) in_use_ = true;
    else (void)hipStreamSynchronize(stream);
  }
  return e;
}

}  // namespace dem
