// Host arrays to and from the device.
//
// A pitched copy of a pageable array runs row by row (9 us a row here: 143 ms
// for the four transfers of a 4096^2 FP32 call whose kernels take 1.4 ms), and
// a plain pageable copy is bound by one thread's memcpy.  So the device grid
// keeps the caller's layout, and the bytes go through a ring of four pinned
// 4 MiB buffers: every OpenMP thread copies a share of a buffer while the DMA
// engine moves the one before.  The ring (16 MiB a device) stays until
// an5d_release.
#include "staging.hpp"

#include <string.h>

namespace an5d {

int staging_init(Staging& s) {
  if (s.ready) return AN5D_OK;
  hipError_t e = hipStreamCreateWithFlags(&s.st, hipStreamNonBlocking);
  for (int i = 0; i < Staging::kSlots && e == hipSuccess; i++) {
    e = hipHostMalloc(&s.slot[i], Staging::kSlotBytes, hipHostMallocDefault);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&s.ev[i], hipEventDisableTiming);
  }
  if (e != hipSuccess) {
    staging_free(s);
    return fail(AN5D_E_ALLOC, std::string("pinned staging buffers: ") + hipGetErrorString(e));
  }
  s.ready = true;
  return AN5D_OK;
}

void staging_free(Staging& s) {
  if (s.st) (void)hipStreamSynchronize(s.st);
  for (int i = 0; i < Staging::kSlots; i++) {
    if (s.ev[i]) (void)hipEventDestroy(s.ev[i]);
    if (s.slot[i]) (void)hipHostFree(s.slot[i]);
  }
  if (s.st) (void)hipStreamDestroy(s.st);
  s = Staging();
}

int staging_upload(Staging& s, void* dev, const void* host, size_t bytes) {
  size_t at = 0;
  for (int c = 0; at < bytes; c++) {
    const int k = c % Staging::kSlots;
    const size_t n = bytes - at < Staging::kSlotBytes ? bytes - at : Staging::kSlotBytes;
    // the slot's last use (of this or an earlier transfer) is over; an event
    // never recorded counts as done
    hipError_t e = hipEventSynchronize(s.ev[k]);
    if (e != hipSuccess) return hip_fail(e, "staging event");
    parallel_copy(s.slot[k], static_cast<const char*>(host) + at, n);
    e = hipMemcpyAsync(static_cast<char*>(dev) + at, s.slot[k], n, hipMemcpyHostToDevice, s.st);
    if (e == hipSuccess) e = hipEventRecord(s.ev[k], s.st);
    if (e != hipSuccess) return hip_fail(e, "staged H2D copy");
    at += n;
  }
  return AN5D_OK;
}

int staging_download(Staging& s, void* host, const void* dev, size_t bytes) {
  const long long chunks = (long long)((bytes + Staging::kSlotBytes - 1) / Staging::kSlotBytes);
  auto size = [&](long long c) {
    const size_t at = (size_t)c * Staging::kSlotBytes;
    return bytes - at < Staging::kSlotBytes ? bytes - at : Staging::kSlotBytes;
  };
  // chunk c is requested kSlots - 1 chunks before it is copied out of its slot;
  // a slot is refilled after that copy, and the stream keeps the order with
  // earlier uploads from it
  for (long long c = 0; c < chunks + Staging::kSlots - 1; c++) {
    if (c < chunks) {
      const int k = (int)(c % Staging::kSlots);
      hipError_t e = hipMemcpyAsync(s.slot[k], static_cast<const char*>(dev) + (size_t)c * Staging::kSlotBytes, size(c),
                                    hipMemcpyDeviceToHost, s.st);
      if (e == hipSuccess) e = hipEventRecord(s.ev[k], s.st);
      if (e != hipSuccess) return hip_fail(e, "staged D2H copy");
    }
    const long long o = c - (Staging::kSlots - 1);
    if (o >= 0) {
      const int k = (int)(o % Staging::kSlots);
      const hipError_t e = hipEventSynchronize(s.ev[k]);
      if (e != hipSuccess) return hip_fail(e, "staged D2H copy");
      parallel_copy(static_cast<char*>(host) + (size_t)o * Staging::kSlotBytes, s.slot[k], size(o));
    }
  }
  return AN5D_OK;
}

// Cells of one interior plane's halo: 2D the R cells at both ends of the row;
// 3D R whole rows at both sides, and the row ends between them.
static long long side_cells(const Geom& g) {
  return g.dim == 3 ? 2 * g.r * g.D2 + (g.D1 - 2 * g.r) * 2 * g.r : 2 * g.r;
}

// Packed halo cells of interior planes (pack_side_halo's order) to their
// places; `src` is pinned host memory, read once.
template <typename T>
__global__ __launch_bounds__(256) void halo_scatter_kernel(const T* __restrict__ src, T* __restrict__ dst,
                                                           long long planes, int R, int dim3, long long D1,
                                                           long long D2, long long side) {
  const long long total = planes * side;
  for (long long x = (long long)blockIdx.x * blockDim.x + threadIdx.x; x < total;
       x += (long long)gridDim.x * blockDim.x) {
    const long long p = x / side;
    long long o = x - p * side, j = 0, k;
    if (dim3) {
      const long long rows = R * D2;  // the whole rows above, then below
      if (o < rows) {
        j = o / D2;
        k = o - j * D2;
      } else if (o < 2 * rows) {
        o -= rows;
        j = o / D2;
        k = o - j * D2;
        j += D1 - R;
      } else {
        o -= 2 * rows;
        j = o / (2 * R);
        k = o - j * (2 * R);
        j += R;
        k = k < R ? k : D2 - 2 * R + k;
      }
    } else {
      k = o < R ? o : D2 - 2 * R + o;
    }
    dst[p * D1 * D2 + j * D2 + k] = src[x];
  }
}

int staging_upload_halo(Staging& s, void* dev, const void* host, const Geom& g, size_t esz) {
  const size_t plane = (size_t)g.D1 * g.D2 * esz;
  const long long side = side_cells(g);
  const long long per = (long long)(Staging::kSlotBytes / ((size_t)side * esz));  // interior planes per slot
  if (per < 1) return staging_upload(s, dev, host, (size_t)g.area * esz);
  int rc = staging_upload(s, dev, host, (size_t)g.r * plane);
  if (rc) return rc;
  const size_t bot = (size_t)(g.D0 - g.r) * plane;
  rc = staging_upload(s, static_cast<char*>(dev) + bot, static_cast<const char*>(host) + bot, (size_t)g.r * plane);
  if (rc) return rc;
  int c = 0;
  for (long long i0 = g.r; i0 < g.D0 - g.r; i0 += per, c++) {
    const int k = c % Staging::kSlots;
    const long long i1 = i0 + per < g.D0 - g.r ? i0 + per : g.D0 - g.r;
    hipError_t e = hipEventSynchronize(s.ev[k]);
    if (e != hipSuccess) return hip_fail(e, "staging event");
    pack_side_halo(static_cast<char*>(s.slot[k]), static_cast<const char*>(host), g.dim, g.r, g.D1, g.D2, esz, i0, i1);
    const long long total = (i1 - i0) * side;
    const long long blocks = (total + 255) / 256;
    const dim3 grid((unsigned)(blocks < 1024 ? blocks : 1024));
    char* d = static_cast<char*>(dev) + (size_t)i0 * plane;
    if (esz == 8)
      hipLaunchKernelGGL((halo_scatter_kernel<double>), grid, dim3(256), 0, s.st, static_cast<const double*>(s.slot[k]),
                         reinterpret_cast<double*>(d), i1 - i0, g.r, g.dim == 3, g.D1, g.D2, side);
    else
      hipLaunchKernelGGL((halo_scatter_kernel<float>), grid, dim3(256), 0, s.st, static_cast<const float*>(s.slot[k]),
                         reinterpret_cast<float*>(d), i1 - i0, g.r, g.dim == 3, g.D1, g.D2, side);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipEventRecord(s.ev[k], s.st);
    if (e != hipSuccess) return hip_fail(e, "halo upload");
  }
  return AN5D_OK;
}

}  // namespace an5d
