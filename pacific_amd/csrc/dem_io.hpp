// Transfers between the library's structure-of-arrays device state and the
// caller's host arrays of rows by particle id (x, y, z of particle 1, of
// particle 2, ...).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <vector>

#include "dem_types.hpp"

namespace dem {

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

// The rows of one call (rows of `width` doubles per particle in the caller's
// array; a null array is left out) and the buffers they pass through: a device
// buffer in row layout and pinned host slices, both kept for the next call
// and freed with the system.
class RowIO {
 public:
  explicit RowIO(int n) : n_(n) {}
  void add(double* host, double* const* comps, int width) {
    if (!host || n_ == 0) return;
    for (int c = 0; c < width; ++c) {
      map_.comp[map_.nc] = comps[c];
      map_.base[map_.nc] = off_ + c;
      map_.stride[map_.nc] = width;
      ++map_.nc;
    }
    segs_.push_back(Seg{host, off_, (size_t)width * n_});
    off_ += (size_t)width * n_;
  }
  void add(const double* host, double* const* comps, int width) { add(const_cast<double*>(host), comps, width); }
  const RowMap& map() const { return map_; }
  size_t doubles() const { return off_; }
  struct Seg {
    double* host;
    size_t off, count;
  };
  const std::vector<Seg>& segs() const { return segs_; }

 private:
  int n_;
  size_t off_ = 0;
  RowMap map_;
  std::vector<Seg> segs_;
};

class RowBuffers {
 public:
  ~RowBuffers() { release(); }
  void release();
  // device state (storage order, ids at id) -> the host arrays of io; the
  // stream has drained on return
  hipError_t down(const RowIO& io, const int* id, int n, int device, hipStream_t stream);
  // the host arrays of io -> device state; enqueued on the stream after the
  // rows have left the host arrays
  hipError_t up(const RowIO& io, const int* id, int n, int device, hipStream_t stream);

 private:
  hipError_t reserve(size_t doubles);
  hipError_t copy(const RowIO& io, bool to_host, int device, hipStream_t stream);
  double* dev_ = nullptr;
  size_t dev_cap_ = 0;
  char* pin_ = nullptr;
  size_t pin_cap_ = 0;
  std::vector<hipStream_t> lanes_;  // one per copying thread
};

}  // namespace dem
