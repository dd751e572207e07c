// Transfers between the host's field arrays and a string's device planes.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

#include "common.hpp"

namespace mepgl {

// One host array (F, N, N, count) and the first of the `count` (1 or 2)
// device planes it holds.
struct HostField {
  double* host;
  int plane;
  int count;
};

// Workspace of the transfers: two pinned host buffers and their events per
// worker, made on first use and kept by the context.
struct FieldIo {
  static constexpr int kMaxWorkers = 8;
  static constexpr size_t kSlotBytes = 1u << 20;     // one buffer
  static constexpr size_t kWorkerBytes = 16u << 20;  // host bytes per worker
  struct Slot {
    void* host = nullptr;  // both buffers
    size_t bytes = 0;      // of one
    hipEvent_t done[2] = {nullptr, nullptr};
    void* buffer(int b) const { return (char*)host + (size_t)b * bytes; }
  };
  Slot slot[kMaxWorkers];
  void release();
};

// Copies the device planes at `dev` (stored in float when fp32, else in
// double) to the host arrays.  Work already queued on `streams` is waited
// for by the caller; the call returns once the host arrays are written.
hipError_t download_fields(FieldIo& io, const DevString& d, const void* dev, bool fp32,
                           const HostField* f, int nf, const hipStream_t* streams, int nstreams,
                           int device);

// Copies the host arrays to the planes of `ndev` (1 or 2) device field sets.
hipError_t upload_fields(FieldIo& io, const DevString& d, void* const* dev, int ndev, bool fp32,
                         const HostField* f, int nf, const hipStream_t* streams, int nstreams,
                         int device);

// Whether images 1 .. F-1 of a host array of `image` doubles each hold the
// bytes of image 0.
bool images_equal(const double* a, int F, size_t image);

}  // namespace mepgl
