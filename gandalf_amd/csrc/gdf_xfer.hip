// Transfers between the caller's memory and the device, and whole-column fills and copies.
//
// Results are written by the device to a pinned staging buffer of the context, a megabyte at a
// time, while the host copies the megabyte before it to the caller's pageable memory.  Every
// particle column of a new run is written from the interleaved arrays once they have arrived, where
// each column used to be gathered on the host and copied by itself.  (us, before and after)
//   particles              4096       100003        1048576
//   all set             360   80    1340  333    13660   2610
//   a vector read        64   21     157  138     1340   1244
// Only the calling thread and stream synchronisation are used: with helper threads, or with events
// to wait for, a program that computes with its own threads between calls (sixteen on sixteen CPUs)
// had them descheduled for 4 ms at a time.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "gdf_internal.h"

namespace gdf {
namespace {

constexpr int BS = 256;
constexpr size_t kChunk = 1 << 17;          // doubles a staging slot
// Up to here arrays go to the device through the staging buffer: 4096 doubles set in 19 us against
// 60 plainly; from 100003 vectors on the runtime's copy from the caller's own pages is faster (99 us
// against 108, 0.69 ms against 0.78 at a million).
constexpr size_t kStagedIn = 1 << 16;
static_assert(kStagedIn <= 2*kChunk, "an array staged in one piece");

__global__ void k_copy_out(int n, const double* __restrict__ src, double* __restrict__ dst) {
  const int i = 2*(blockIdx.x*BS + threadIdx.x);
  if (i + 1 < n) *reinterpret_cast<double2*>(dst + i) = *reinterpret_cast<const double2*>(src + i);
  else if (i < n) dst[i] = src[i];
}

// an array of w interleaved components, n doubles in all, to up to two sets of columns
__global__ void k_unpack(size_t n, XferCols to, const double* __restrict__ src) {
  const size_t e = (size_t) blockIdx.x*BS + threadIdx.x;
  if (e >= n) return;
  const size_t i = to.w == 1 ? e : e/3;
  const int k = to.w == 1 ? 0 : (int) (e - 3*i);
  const double v = src[e];
  to.a[k][i] = v;
  if (to.b[k]) to.b[k][i] = v;
}

__global__ void k_zero_cols(int n, ColSet s) {
  const int i = blockIdx.x*BS + threadIdx.x, k = blockIdx.y;
  if (i >= n) return;
  if (k < s.nd) s.d[k][i] = 0.0;
  else s.i[k - s.nd][i] = 0;
}

__global__ void k_copy_cols(int n, ColSet s, ColSet from) {
  const int i = blockIdx.x*BS + threadIdx.x, k = blockIdx.y;
  if (i >= n) return;
  if (k < s.nd) s.d[k][i] = from.d[k][i];
  else s.i[k - s.nd][i] = from.i[k - s.nd][i];
}

// the two staging slots; false: none to be had (the caller copies plainly)
bool stage_ensure(gdf_ctx* c) {
  if (c->xfer) return true;
  if (hipHostMalloc(&c->xfer, sizeof(double)*2*kChunk) == hipSuccess) return true;
  (void) hipGetLastError();
  c->xfer = nullptr;
  return false;
}

}  // namespace

int xfer_out(gdf_ctx* c, double* out, const double* dev, size_t n) {
  hipStream_t s = c->stream;
  if (!stage_ensure(c)) {
    GDF_HIP(c, hipMemcpyAsync(out, dev, sizeof(double)*n, hipMemcpyDeviceToHost, s));
    GDF_HIP(c, hipStreamSynchronize(s));
    return GDF_OK;
  }
  auto issue = [&](size_t e0) {
    const int m = (int) std::min(kChunk, n - e0);
    k_copy_out<<<(m + 2*BS - 1)/(2*BS), BS, 0, s>>>(m, dev + e0, c->xfer + e0 % (2*kChunk));
    return hipGetLastError();
  };
  GDF_HIP(c, issue(0));
  for (size_t e0 = 0; e0 < n; e0 += kChunk) {
    GDF_HIP(c, hipStreamSynchronize(s));
    if (e0 + kChunk < n) GDF_HIP(c, issue(e0 + kChunk));
    memcpy(out + e0, c->xfer + e0 % (2*kChunk), sizeof(double)*std::min(kChunk, n - e0));
  }
  return GDF_OK;
}

int xfer_in(gdf_ctx* c, const double* in, size_t n, const XferCols& to, bool wait) {
  hipStream_t s = c->stream;
  const bool staged = n <= kStagedIn && stage_ensure(c);
  double* src = staged ? c->xfer : c->tmpd;      // tmpd: room for three components a particle
  if (staged) memcpy(src, in, sizeof(double)*n);
  else GDF_HIP(c, hipMemcpyAsync(src, in, sizeof(double)*n, hipMemcpyHostToDevice, s));
  if (to.a[0] != src) {
    k_unpack<<<(unsigned) ((n + BS - 1)/BS), BS, 0, s>>>(n, to, src);
    GDF_HIP(c, hipGetLastError());
  }
  if (wait) GDF_HIP(c, hipStreamSynchronize(s));
  return GDF_OK;
}

int cols_zero(gdf_ctx* c, const ColSet& s, int n) {
  if (n <= 0 || s.nd + s.ni == 0) return GDF_OK;
  k_zero_cols<<<dim3((n + BS - 1)/BS, s.nd + s.ni), BS, 0, c->stream>>>(n, s);
  GDF_HIP(c, hipGetLastError());
  return GDF_OK;
}

int cols_copy(gdf_ctx* c, const ColSet& to, const ColSet& from, int n) {
  if (n <= 0 || to.nd + to.ni == 0) return GDF_OK;
  k_copy_cols<<<dim3((n + BS - 1)/BS, to.nd + to.ni), BS, 0, c->stream>>>(n, to, from);
  GDF_HIP(c, hipGetLastError());
  return GDF_OK;
}

}  // namespace gdf
