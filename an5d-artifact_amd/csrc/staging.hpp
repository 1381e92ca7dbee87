// Host arrays to and from the device, through a ring of pinned buffers.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

#include "internal.hpp"

namespace an5d {

// A device's ring of pinned buffers with the stream and the events that order
// its copies.  One host call at a time uses it (the staging grid's lock).
struct Staging {
  static constexpr int kSlots = 4;
  static constexpr size_t kSlotBytes = 4ull << 20;
  void* slot[kSlots] = {};
  hipEvent_t ev[kSlots] = {};
  hipStream_t st = nullptr;
  bool ready = false;
};
int staging_init(Staging& s);
void staging_free(Staging& s);
// Enqueues the copies on s.st and returns when the host array may be used
// again; an upload may still be on its way from the ring.
int staging_upload(Staging& s, void* dev, const void* host, size_t bytes);
int staging_download(Staging& s, void* host, const void* dev, size_t bytes);
// The halo cells of one grid (reference layout) only.
int staging_upload_halo(Staging& s, void* dev, const void* host, const Geom& g, size_t esz);

// cpu_path.cpp: memcpy over the OpenMP threads; the halo cells of the interior
// planes [i0, i1) of a grid, plane by plane, as halo_scatter_kernel takes them
void parallel_copy(void* dst, const void* src, size_t bytes);
void pack_side_halo(char* dst, const char* grid, int dim, long long r, long long D1, long long D2, size_t esz,
                    long long i0, long long i1);

}  // namespace an5d
