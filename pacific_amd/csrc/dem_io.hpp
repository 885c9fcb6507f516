// Transfers between the library's structure-of-arrays device state and the
// caller's host arrays of rows by particle id (x, y, z of particle 1, of
// particle 2, ...).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <memory>
#include <mutex>
#include <vector>

#include "dem_types.hpp"

namespace dem {

// Synchronous copies and fills go through the legacy stream, which ends the
// capture that another thread has under way on a stream of its own, and fails
// itself: captures hold this lock, and so does each of these.
std::mutex& capture_lock();
hipError_t copy_sync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind);
hipError_t fill_sync(void* dst, int value, size_t bytes);

// Component c of the particle in storage index s <-> element
// base[c] + stride[c] * (id[s] - 1) of one buffer of rows.
struct RowMap {
  static constexpr int kMax = 24;
  double* comp[kMax];
  size_t base[kMax];
  int stride[kMax];
  int nc = 0;
};
hipError_t launch_rows_out(const RowMap& m, const int* id, int n, double* out, hipStream_t stream);
hipError_t launch_rows_in(const RowMap& m, const int* id, int n, const double* in, hipStream_t stream);
// body-fixed angular velocity from w and q (ParticleKinematics::setAngularVelocity)
hipError_t launch_body_spin(const Particles& P, int n, int cv, hipStream_t stream);

// a[k][i] <- a[k][order[i]] for every array (8- and 4-byte elements); tmp
// holds kPermuteGroup * n doubles
constexpr int kPermuteGroup = 4;
hipError_t launch_permute(const std::vector<double*>& a8, const std::vector<int*>& a4, const int* order, int n,
                          double* tmp, hipStream_t stream);

// The rows of one call: rows of `width` doubles per particle in the caller's
// array (a null array is left out).  They pass through the buffers below in
// parts of whole arrays, each as long as fits in kPart bytes (one array at
// least), so that what is kept on the device stays small beside a large state
// (64 MB, three parts, cost 2 % of a pass of the 1M gas).
class RowIO {
 public:
  static constexpr size_t kPart = (size_t)192 << 20;
  explicit RowIO(int n) : n_((size_t)n) {}
  void add(double* host, double* const* comps, int width) {
    if (!host || n_ == 0) return;
    Seg s{host, (size_t)width * n_, {}, width};
    for (int c = 0; c < width; ++c) s.comp[c] = comps[c];
    segs_.push_back(s);
  }
  void add(const double* host, double* const* comps, int width) { add(const_cast<double*>(host), comps, width); }
  struct Seg {
    double* host;
    size_t count;  // doubles
    double* comp[9];
    int width;
  };
  const std::vector<Seg>& segs() const { return segs_; }
  // the part that begins with array `first` ends before the one returned
  size_t part(size_t first) const {
    size_t last = first, bytes = 0;
    int nc = 0;
    while (last < segs_.size()) {
      bytes += segs_[last].count * sizeof(double);
      nc += segs_[last].width;
      if (last > first && (bytes > kPart || nc > RowMap::kMax)) break;
      ++last;
    }
    return last;
  }
  // its rows one array after the other, from 0
  RowMap map(size_t first, size_t last) const {
    RowMap m;
    size_t at = 0;
    for (size_t k = first; k < last; ++k) {
      for (int c = 0; c < segs_[k].width; ++c) {
        m.comp[m.nc] = segs_[k].comp[c];
        m.base[m.nc] = at + c;
        m.stride[m.nc] = segs_[k].width;
        ++m.nc;
      }
      at += segs_[k].count;
    }
    return m;
  }

 private:
  size_t n_;
  std::vector<Seg> segs_;
};

// What the transfers of one device pass through, shared by its systems and
// batches: a device buffer in row layout and pinned host slices, each as large
// as the largest part so far, and pinned blocks that a status block comes back
// to.  Made with the first system and freed with the last: allocating them
// costs 0.3 ms each above 2 MB, as long as a state of 27,000 takes.  A call holds
// the lock while it uses the buffers, and therefore comes with a stream that
// has little left to do.  Where the card or the host has no room for
// them, the components cross one by one and are put in their rows here on the
// host (plain).
class RowBuffers {
 public:
  static std::shared_ptr<RowBuffers> of(int device);
  explicit RowBuffers(int device) : device_(device) {}
  RowBuffers(const RowBuffers&) = delete;
  ~RowBuffers();
  // device state (storage order, ids at id) -> the host arrays of io; the
  // stream has drained on return
  hipError_t down(const RowIO& io, const int* id, int n, hipStream_t stream);
  // the host arrays of io -> device state; enqueued on the stream after the
  // rows have left the host arrays
  hipError_t up(const RowIO& io, const int* id, int n, hipStream_t stream);
  // a block for a DevStatus, to be given back
  DevStatus* status_block();
  void give_back(DevStatus* p);

 private:
  hipError_t reserve(const RowIO& io, size_t first, size_t last);
  hipError_t copy(const RowIO& io, size_t first, size_t last, bool to_host, hipStream_t stream);
  hipError_t plain(const RowIO& io, size_t first, bool to_host, const int* id, int n, hipStream_t stream);
  const int device_;
  std::mutex use_;  // the buffers
  double* dev_ = nullptr;
  size_t dev_cap_ = 0;  // bytes
  char* pin_ = nullptr;
  size_t pin_cap_ = 0;
  std::vector<hipEvent_t> copied_;  // one per copying thread
  std::vector<hipStream_t> lanes_;
  hipEvent_t read_ = nullptr;  // after the kernel that last read rows from the device buffer
  bool in_use_ = false;
  std::mutex blocks_;
  std::vector<DevStatus*> pages_, free_;
  std::vector<std::unique_ptr<DevStatus[]>> plain_;
};

}  // namespace dem
