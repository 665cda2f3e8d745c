// Device tree: Morton keys, radix sort, LBVH topology, bottom-up cell moments, walk groups.
//
// Replaces KDTree::BuildTree / StockTree (src/Tree/KDTree.cpp:220-313, :760-1083) behind
// HydroTree::BuildTree (src/Tree/HydroTree.cpp:310-372).  Instead of median QuickSelect splits
// the particles are sorted along a 63-bit Morton curve and the binary radix tree over the sorted
// keys (Karras 2012) supplies the cells.  Cell moments follow the reference's bottom-up stock:
// mass, centre of mass, traceless quadrupole with the parallel-axis merge (KDTree.cpp:950-1051),
// bounding box, hmax and the geometric-MAC distance cdistsqd = max(rmax^2, hmax^2)/theta^2
// (KDTree.cpp:917,997).  The particle arrays are physically permuted into key order so every
// later pass streams coalesced SoA data.
#include <hip/hip_runtime.h>
#include <cstring>
#include <rocprim/device/device_radix_sort.hpp>

#include "gdf_internal.h"
#include "gdf_device.h"
#include "gdf_filter.h"

namespace gdf {
namespace {

constexpr int BS = 256;

__global__ void k_bounds_partial(int N, const double* __restrict__ x, const double* __restrict__ y,
                                 const double* __restrict__ z, double* __restrict__ part) {
  __shared__ double s[6][BS];
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  for (int i = blockIdx.x*BS + threadIdx.x; i < N; i += gridDim.x*BS) {
    const double v[3] = {x[i], y[i], z[i]};
    for (int k = 0; k < 3; k++) { lo[k] = fmin(lo[k], v[k]); hi[k] = fmax(hi[k], v[k]); }
  }
  for (int k = 0; k < 3; k++) { s[k][threadIdx.x] = lo[k]; s[3+k][threadIdx.x] = hi[k]; }
  __syncthreads();
  for (int w = BS/2; w > 0; w >>= 1) {
    if (threadIdx.x < w)
      for (int k = 0; k < 3; k++) {
        s[k][threadIdx.x] = fmin(s[k][threadIdx.x], s[k][threadIdx.x + w]);
        s[3+k][threadIdx.x] = fmax(s[3+k][threadIdx.x], s[3+k][threadIdx.x + w]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 6) part[blockIdx.x*6 + threadIdx.x] = s[threadIdx.x][0];
}

// out: lo[3], scale; one block of BS threads folds the per-block partials
__global__ __launch_bounds__(BS) void k_bounds_final(int nb, const double* __restrict__ part,
                                                     double* __restrict__ out) {
  __shared__ double s[6][BS];
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  for (int b = threadIdx.x; b < nb; b += BS)
    for (int k = 0; k < 3; k++) {
      lo[k] = fmin(lo[k], part[b*6 + k]);
      hi[k] = fmax(hi[k], part[b*6 + 3 + k]);
    }
  for (int k = 0; k < 3; k++) { s[k][threadIdx.x] = lo[k]; s[3+k][threadIdx.x] = hi[k]; }
  __syncthreads();
  for (int w = BS/2; w > 0; w >>= 1) {
    if (threadIdx.x < w)
      for (int k = 0; k < 3; k++) {
        s[k][threadIdx.x] = fmin(s[k][threadIdx.x], s[k][threadIdx.x + w]);
        s[3+k][threadIdx.x] = fmax(s[3+k][threadIdx.x], s[3+k][threadIdx.x + w]);
      }
    __syncthreads();
  }
  if (threadIdx.x != 0) return;
  double span = s[3][0] - s[0][0];
  if (s[4][0] - s[1][0] > span) span = s[4][0] - s[1][0];
  if (s[5][0] - s[2][0] > span) span = s[5][0] - s[2][0];
  if (!(span > 0.0)) span = 1.0;
  out[0] = s[0][0]; out[1] = s[1][0]; out[2] = s[2][0];
  out[3] = 2097152.0/span;
}

// ---- serving batches: per-segment bounds and segment-prefixed keys ----
// partial-reduction blocks per segment: kMaxSeg x 16 x 6 partials fit the reduction buffer
constexpr int kSegBlocks = 16;
constexpr int kSegShift = 57;       // the segment id's place in a key
constexpr int kSelBlock = 256;      // workgroup of the group selection

// grid (kSegBlocks, nseg): block (b, s) folds a strided share of segment s
__global__ void k_seg_bounds_partial(const int* __restrict__ off, const double* __restrict__ x,
                                     const double* __restrict__ y, const double* __restrict__ z,
                                     double* __restrict__ part) {
  __shared__ double sh[6][BS];
  const int sg = blockIdx.y, b = blockIdx.x;
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  for (int i = off[sg] + b*BS + threadIdx.x; i < off[sg + 1]; i += kSegBlocks*BS) {
    const double v[3] = {x[i], y[i], z[i]};
    for (int k = 0; k < 3; k++) { lo[k] = fmin(lo[k], v[k]); hi[k] = fmax(hi[k], v[k]); }
  }
  for (int k = 0; k < 3; k++) { sh[k][threadIdx.x] = lo[k]; sh[3+k][threadIdx.x] = hi[k]; }
  __syncthreads();
  for (int w = BS/2; w > 0; w >>= 1) {
    if (threadIdx.x < w)
      for (int k = 0; k < 3; k++) {
        sh[k][threadIdx.x] = fmin(sh[k][threadIdx.x], sh[k][threadIdx.x + w]);
        sh[3+k][threadIdx.x] = fmax(sh[3+k][threadIdx.x], sh[3+k][threadIdx.x + w]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 6) part[(sg*kSegBlocks + b)*6 + threadIdx.x] = sh[threadIdx.x][0];
}

// one 64-thread block per segment: lower corner and scale of a 2^19 grid per axis
__global__ void k_seg_bounds_final(const double* __restrict__ part, double* __restrict__ bnd) {
  const int sg = blockIdx.x, t = threadIdx.x;
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  if (t < kSegBlocks)
    for (int k = 0; k < 3; k++) {
      lo[k] = part[(sg*kSegBlocks + t)*6 + k];
      hi[k] = part[(sg*kSegBlocks + t)*6 + 3 + k];
    }
  for (int k = 0; k < 3; k++)
    for (int d = 32; d >= 1; d >>= 1) {
      lo[k] = fmin(lo[k], __shfl_xor(lo[k], d, 64));
      hi[k] = fmax(hi[k], __shfl_xor(hi[k], d, 64));
    }
  if (t != 0) return;
  double span = fmax(fmax(hi[0] - lo[0], hi[1] - lo[1]), hi[2] - lo[2]);
  if (!(span > 0.0)) span = 1.0;
  bnd[4*sg] = lo[0]; bnd[4*sg + 1] = lo[1]; bnd[4*sg + 2] = lo[2];
  bnd[4*sg + 3] = 524288.0/span;
}

__device__ __forceinline__ uint64_t spread3(uint64_t x) {
  x &= 0x1fffffULL;
  x = (x | (x << 32)) & 0x1f00000000ffffULL;
  x = (x | (x << 16)) & 0x1f0000ff0000ffULL;
  x = (x | (x << 8))  & 0x100f00f00f00f00fULL;
  x = (x | (x << 4))  & 0x10c30c30c30c30c3ULL;
  x = (x | (x << 2))  & 0x1249249249249249ULL;
  return x;
}

__global__ void k_morton(int N, const double* __restrict__ x, const double* __restrict__ y,
                         const double* __restrict__ z, const double* __restrict__ bnd,
                         uint64_t* __restrict__ keys, int* __restrict__ vals,
                         int* __restrict__ gstart) {
  const int i = blockIdx.x*BS + threadIdx.x;
  if (i >= N) return;
  gstart[i] = -1;                       // k_lbvh marks the group starts
  const double scale = bnd[3];
  const double v[3] = {x[i], y[i], z[i]};
  uint64_t q[3];
  for (int k = 0; k < 3; k++) {
    const double f = __dmul_rn(__dadd_rn(v[k], -bnd[k]), scale);
    q[k] = f >= 2097151.0 ? 2097151ULL : (uint64_t) f;
  }
  keys[i] = (spread3(q[0]) << 2) | (spread3(q[1]) << 1) | spread3(q[2]);
  vals[i] = i;
}

struct PermArgs {
  const double* src[F_NPERSIST]; double* dst[F_NPERSIST];
  const int* isrc[I_NINT]; int* idst[I_NINT];
};

__global__ void k_permute(int N, const int* __restrict__ vals, PermArgs a,
                          const int* __restrict__ io, int* __restrict__ io_alt) {
  const int s = blockIdx.x*BS + threadIdx.x;
  if (s >= N) return;
  const int o = vals[s];
  #pragma unroll
  for (int f = 0; f < F_NPERSIST; f++) a.dst[f][s] = a.src[f][o];
  #pragma unroll
  for (int f = 0; f < I_NINT; f++) a.idst[f][s] = a.isrc[f][o];
  io_alt[s] = io[o];
}

// block timesteps: the derived fields an inactive particle keeps until its step ends (its
// neighbours read rho, P, Omega, zeta, c_s, hfactor; diagnostics read gpot; a, atree, du/dt and
// div v are its visible state); the search radius, the timestep criterion, the N-body jerk and
// the gravity walk's partial sums are rewritten before every use and are not moved
constexpr int kPermD[] = {D_AX, D_AY, D_AZ, D_ATX, D_ATY, D_ATZ, D_RHO, D_DUDT, D_DIVV, D_GPOT,
                          D_INVOMEGA, D_ZETA, D_SOUND, D_PRESSURE, D_HFACTOR};
constexpr int kNPermD = sizeof(kPermD)/sizeof(kPermD[0]);
struct PermDArgs { const double* src[kNPermD]; double* dst[kNPermD]; };

__global__ void k_permute_d(int N, const int* __restrict__ vals, PermDArgs a) {
  const int s = blockIdx.x*BS + threadIdx.x;
  if (s >= N) return;
  const int o = vals[s];
  #pragma unroll
  for (int f = 0; f < kNPermD; f++) a.dst[f][s] = a.src[f][o];
}

__device__ __forceinline__ int delta(const uint64_t* __restrict__ key, int N, int i, long long j) {
  if (j < 0 || j > N - 1) return -1;
  const uint64_t a = key[i], b = key[j];
  if (a != b) return __clzll((long long) (a ^ b));
  return 64 + __clz((int) (i ^ (int) j));
}

// segment-prefixed key: segment id from bit kSegShift (57) on, 19 bits per axis below
__global__ void k_morton_seg(int N, const double* __restrict__ x, const double* __restrict__ y,
                             const double* __restrict__ z, const int* __restrict__ seg,
                             const double* __restrict__ bnd, uint64_t* __restrict__ keys,
                             int* __restrict__ vals, int* __restrict__ gstart) {
  const int i = blockIdx.x*BS + threadIdx.x;
  if (i >= N) return;
  gstart[i] = -1;                       // k_lbvh marks the group starts
  const int sg = seg[i];
  const double scale = bnd[4*sg + 3];
  const double v[3] = {x[i], y[i], z[i]};
  uint64_t q[3];
  for (int k = 0; k < 3; k++) {
    const double f = __dmul_rn(__dadd_rn(v[k], -bnd[4*sg + k]), scale);
    q[k] = f >= 524287.0 ? 524287ULL : (uint64_t) f;
  }
  keys[i] = ((uint64_t) sg << kSegShift) | (spread3(q[0]) << 2) | (spread3(q[1]) << 1) | spread3(q[2]);
  vals[i] = i;
}

// the node spanning exactly segment s is its subtree root (the keys of a segment share the
// segment prefix and no other key does)
__global__ void k_seg_roots(int N, int nseg, const int* __restrict__ off,
                            const int* __restrict__ first, const int* __restrict__ last,
                            const int* __restrict__ seg, int* __restrict__ root) {
  const int n = blockIdx.x*BS + threadIdx.x;
  if (n < N - 1) {
    const int f = first[n], l = last[n], sg = seg[f];
    if (f == off[sg] && l == off[sg + 1] - 1) root[sg] = n;
  } else if (n < 2*N - 1) {
    const int leaf = n - (N - 1), sg = seg[leaf];
    if (off[sg + 1] - off[sg] == 1) root[sg] = n;
  }
}

// The walking group's factor of the gadget2 / eigenmac opening criterion (the reference's
// walking leaf cell's amin / macfactor, stocked from its particles, KDTree.cpp:900-903):
// gadget2 the smallest |atree|, eigenmac the largest gpot^(-2/3).  One wavefront per group;
// perm (non-NULL) maps a group's sorted slots to the force arrays' order when the build did not
// permute them.
__global__ __launch_bounds__(BS) void k_group_mac(int ngroups, const int* __restrict__ grp_first,
                                                  const int* __restrict__ grp_count,
                                                  const int* __restrict__ perm,
                                                  const double* __restrict__ ax,
                                                  const double* __restrict__ ay,
                                                  const double* __restrict__ az,
                                                  const double* __restrict__ gpot, int mode,
                                                  double* __restrict__ out) {
#pragma clang fp contract(off)
  const int g = blockIdx.x*(BS/kWave) + (int) threadIdx.x/kWave;
  const int lane = threadIdx.x & (kWave - 1);
  if (g >= ngroups) return;
  const bool gadget = mode == GDF_MAC_GADGET2;
  double v = gadget ? 9.9e30 : 0.0;
  if (lane < grp_count[g]) {
    int i = grp_first[g] + lane;
    if (perm) i = perm[i];
    v = gadget ? sqrt(ax[i]*ax[i] + ay[i]*ay[i] + az[i]*az[i])
               : pow(gpot[i], -0.66666666666666666666666);
  }
  for (int o = 32; o > 0; o >>= 1) {
    const double w = __shfl_xor(v, o, kWave);
    v = gadget ? fmin(v, w) : fmax(v, w);
  }
  if (lane == 0) out[g] = v;
}

int group_mac(gdf_ctx* c, const int* perm) {
  if (c->phys.gravity_mac == GDF_MAC_GEOMETRIC || c->ngroups <= 0) return GDF_OK;
  constexpr int gpb = BS/kWave;
  k_group_mac<<<(c->ngroups + gpb - 1)/gpb, BS, 0, c->stream>>>(
      c->ngroups, c->grp_first, c->grp_count, perm, c->df[D_ATX], c->df[D_ATY], c->df[D_ATZ],
      c->df[D_GPOT], c->phys.gravity_mac, c->grp_gmac);
  GDF_HIP(c, hipGetLastError());
  return GDF_OK;
}

__global__ void k_grp_roots(int ngroups, const int* __restrict__ grp_first,
                            const int* __restrict__ seg, const int* __restrict__ root,
                            int* __restrict__ grp_root) {
  const int g = blockIdx.x*BS + threadIdx.x;
  if (g < ngroups) grp_root[g] = root[seg[grp_first[g]]];
}

// Karras 2012, "Maximizing parallelism in the construction of BVHs, octrees, and k-d trees".  The
// walk groups are the maximal nodes of at most gmax particles, in a serving batch (segs) of one
// request alone (a group walks from its request's subtree): a node that is more marks those of its
// children that are groups, with their sizes, at their first particles.
__global__ void k_lbvh(int N, int gmax, bool segs, int* __restrict__ gstart, int* __restrict__ gsize, const uint64_t* __restrict__ key, int* __restrict__ left,
                       int* __restrict__ right, int* __restrict__ first, int* __restrict__ last,
                       int* __restrict__ parent, int4* __restrict__ lnk) {
  const int i = blockIdx.x*BS + threadIdx.x;
  if (i >= N - 1) return;
  const int d = (delta(key, N, i, (long long) i + 1) - delta(key, N, i, (long long) i - 1)) >= 0 ? 1 : -1;
  const int dmin = delta(key, N, i, (long long) i - d);
  long long lmax = 2;
  while (delta(key, N, i, (long long) i + lmax*d) > dmin) lmax *= 2;
  long long l = 0;
  for (long long t = lmax/2; t >= 1; t /= 2)
    if (delta(key, N, i, (long long) i + (l + t)*d) > dmin) l += t;
  const long long j = (long long) i + l*d;
  const int dnode = delta(key, N, i, j);
  long long s = 0, div = 2, step;
  do {
    step = (l + div - 1)/div;
    if (delta(key, N, i, (long long) i + (s + step)*d) > dnode) s += step;
    div *= 2;
  } while (step > 1);
  const int gamma = (int) ((long long) i + s*d + (d < 0 ? d : 0));
  const int f = (int) (i < j ? i : j), la = (int) (i < j ? j : i);
  first[i] = f; last[i] = la;
  const int L = (f == gamma) ? (N - 1 + gamma) : gamma;
  const int R = (la == gamma + 1) ? (N - 1 + gamma + 1) : gamma + 1;
  left[i] = L; right[i] = R;
  lnk[i] = make_int4(f, la, L, R);
  parent[L] = i; parent[R] = i;
  if (i == 0) parent[0] = -1;
  auto group = [&](int a, int b) {
    return b - a + 1 <= gmax && !(segs && key[a] >> kSegShift != key[b] >> kSegShift);
  };
  if (!group(f, la)) {
    if (group(f, gamma)) { gstart[f] = L; gsize[f] = gamma - f + 1; }
    if (group(gamma + 1, la)) { gstart[gamma + 1] = R; gsize[gamma + 1] = la - gamma; }
  } else if (i == 0) {
    gstart[0] = 0;
    gsize[0] = N;
  }
}

struct NodeArgs {
  double4* geo_c; double4* geo_h; double* mp;
};

__global__ void k_leaves(int N, const double* __restrict__ x, const double* __restrict__ y,
                         const double* __restrict__ z, const double* __restrict__ m,
                         const double* __restrict__ h, double theta2, NodeArgs a,
                         int* __restrict__ parent, int* __restrict__ gstart,
                         int* __restrict__ gsize) {
  const int l = blockIdx.x*BS + threadIdx.x;
  if (l >= N) return;
  if (N == 1) { parent[0] = -1; gstart[0] = 0; gsize[0] = 1; }
  const int n = N - 1 + l;
  const double r[3] = {x[l], y[l], z[l]};
  const double hh = h[l];
  double* mp = a.mp + (size_t) kMom*n;
  for (int k = 0; k < 3; k++) mp[k] = mp[10 + k] = mp[13 + k] = r[k];
  mp[3] = m[l];
  for (int k = 4; k < 9; k++) mp[k] = 0.0;
  mp[9] = hh;
  a.geo_c[n] = make_double4(r[0], r[1], r[2], hh);
  a.geo_h[n] = make_double4(0.0, 0.0, 0.0, __ddiv_rn(__dmul_rn(hh, hh), theta2));
}

// Moments of one node as a refit climb carries them: bounding box, centre of mass, mass,
// quadrupole moment and the largest smoothing length below the node.
struct NodeD {
  double lo[3], hi[3], com[3], m, q[5], hmax;
};

// merge children L (left) and R (right) into o; operation order of KDTree.cpp:950-1051
__device__ __forceinline__ void merge_d(const NodeD& L, const NodeD& R, NodeD& o) {
#pragma clang fp contract(off)
  const double m = L.m + R.m;
  for (int k = 0; k < 3; k++) {
    o.com[k] = m > 0 ? (L.m*L.com[k] + R.m*R.com[k])/m : 0.0;
    o.lo[k] = fmin(L.lo[k], R.lo[k]);
    o.hi[k] = fmax(L.hi[k], R.hi[k]);
  }
  o.m = m;
  o.hmax = fmax(L.hmax, R.hmax);
  for (int k = 0; k < 5; k++) o.q[k] = 0.0;
  for (int c = 0; c < 2; c++) {
    const NodeD& C = c == 0 ? L : R;
    const double mi = C.m;
    if (!(mi > 0)) continue;
    double dr[3];
    for (int k = 0; k < 3; k++) dr[k] = C.com[k] - o.com[k];
    const double drsqd = dr[0]*dr[0] + dr[1]*dr[1] + dr[2]*dr[2];
    for (int k = 0; k < 5; k++) o.q[k] += C.q[k];
    o.q[0] += mi*(3.0*dr[0]*dr[0] - drsqd);
    o.q[1] += mi*3.0*dr[0]*dr[1];
    o.q[2] += mi*(3.0*dr[1]*dr[1] - drsqd);
    o.q[3] += mi*3.0*dr[2]*dr[0];
    o.q[4] += mi*3.0*dr[2]*dr[1];
  }
}

// box centre and half-widths with the bound on h and the opening distance
__device__ __forceinline__ void store_geo(int n, const NodeD& d, double theta2, const NodeArgs& a) {
#pragma clang fp contract(off)
  double c[3], hf[3];
  for (int k = 0; k < 3; k++) { c[k] = 0.5*(d.lo[k] + d.hi[k]); hf[k] = 0.5*(d.hi[k] - d.lo[k]); }
  const double rmaxsqd = hf[0]*hf[0] + hf[1]*hf[1] + hf[2]*hf[2];
  a.geo_c[n] = make_double4(c[0], c[1], c[2], d.hmax);
  a.geo_h[n] = make_double4(hf[0], hf[1], hf[2], fmax(rmaxsqd, d.hmax*d.hmax)/theta2);
}

// Bottom-up refit.  A workgroup takes a contiguous run of finished nodes and merges the nodes whose
// leaf range lies inside the run, level by level: the second child to finish puts its parent on the
// next level's list, and the list's nodes are merged one a lane, so that the lanes of a wavefront
// stay together however uneven the tree is.  The moments stay in LDS, each node's in the place of
// its left child's.  Phase 1 runs over chunks of RB leaves; what it leaves (the maximal nodes inside
// each chunk, in leaf order) is the input of the next phase, RS runs a workgroup, until one
// workgroup reaches the root.  Every node is merged exactly once from finished children in the fixed
// (left, right) operand order, and no two workgroups touch the same node, so there are no atomics
// beyond LDS (device-scope ones would write back the per-XCD L2 on every level).
//
// Bound by the chain of levels at small runs and by vector issue before this: with a thread climbing
// from every leaf each wavefront carried the whole merge through every level for a few lanes.  (us,
// before and after, phase 1 and the rest)
//   particles                4096     20011    131072   262144   1048576
//   all moments, phase 1     37 23    58 29    54 36    65 39    240 148
//   all moments, the rest     7  7    36 30   122 88   101 62    167  80
//   h alone, phase 1         10  9    13 13             19 17     63  59
//   h alone, the rest         5  6    18 18             42 38     61  47
constexpr int RB = 1024;   // leaves per phase-1 workgroup
constexpr int RS = 32;     // runs per workgroup of the later phases
constexpr int RF = 768;    // nodes a workgroup of the later phases holds at a time
constexpr int RT = 512;    // its threads (a level merges at most half of the nodes)

// The moments in LDS, component by component in the order of a node's record in memory: one spare
// slot in 32, as the slots of higher levels are multiples of ever higher powers of two, and an odd
// stride, as a record's components are read together.  A record is one line, written and read by
// eight lanes together: a lane writing its own node's would touch a line with every store.
template <bool HONLY, int CAP> struct RefitSlots {
  static constexpr int ND = HONLY ? 1 : kMom, STRIDE = CAP + CAP/32 + (CAP/32 & 1 ? 0 : 1);
  double v[ND*STRIDE];
  __device__ __forceinline__ static int at(int s) { return s + (s >> 5); }
  __device__ __forceinline__ void put(int s, const NodeD& d) {
    double* p = v + at(s);
    if (HONLY) { p[0] = d.hmax; return; }
    for (int k = 0; k < 3; k++) {
      p[k*STRIDE] = d.com[k]; p[(10 + k)*STRIDE] = d.lo[k]; p[(13 + k)*STRIDE] = d.hi[k];
    }
    p[3*STRIDE] = d.m;
    for (int k = 0; k < 5; k++) p[(4 + k)*STRIDE] = d.q[k];
    p[9*STRIDE] = d.hmax;
  }
  __device__ __forceinline__ void get(int s, NodeD& d) const {
    const double* p = v + at(s);
    if (HONLY) { d.hmax = p[0]; return; }
    for (int k = 0; k < 3; k++) {
      d.com[k] = p[k*STRIDE]; d.lo[k] = p[(10 + k)*STRIDE]; d.hi[k] = p[(13 + k)*STRIDE];
    }
    d.m = p[3*STRIDE];
    for (int k = 0; k < 5; k++) d.q[k] = p[(4 + k)*STRIDE];
    d.hmax = p[9*STRIDE];
  }
  // record part k (two components of sixteen) of slot s, from or to node n's in memory
  __device__ __forceinline__ void part_out(int s, int n, int k, const NodeArgs& a) const {
    const double* p = v + at(s) + 2*k*STRIDE;
    reinterpret_cast<double2*>(a.mp)[(size_t) n*(kMom/2) + k] = make_double2(p[0], p[STRIDE]);
  }
  __device__ __forceinline__ void part_in(int s, int n, int k, const NodeArgs& a) {
    const double2 x = reinterpret_cast<const double2*>(a.mp)[(size_t) n*(kMom/2) + k];
    double* p = v + at(s) + 2*k*STRIDE;
    p[0] = x.x; p[STRIDE] = x.y;
  }
  // merge slots l and r into l as node n; rmax2: the squared half-diagonal of its box (HONLY).
  // The record is left to part_out.
  __device__ __forceinline__ void merge(int l, int r, int n, double rmax2, double theta2,
                                        const NodeArgs& a) {
#pragma clang fp contract(off)
    NodeD L, R, o;
    get(l, L);
    get(r, R);
    if (HONLY) {
      o.hmax = fmax(L.hmax, R.hmax);
      a.geo_c[n].w = o.hmax;
      a.geo_h[n].w = fmax(rmax2, o.hmax*o.hmax)/theta2;
    } else {
      merge_d(L, R, o);
      store_geo(n, o, theta2, a);
    }
    put(l, o);
  }
  // the records of a wavefront's merged nodes, the first `count` of which are node(j), slot(j)
  template <class A, class B>
  __device__ __forceinline__ void records_out(int count, A node, B slot, const NodeArgs& a) const {
    if (HONLY) return;
    wave_lds_order();
    for (int j = lane_id()/(kMom/2); j < count; j += kWave/(kMom/2))
      part_out(slot(j), node(j), lane_id() & (kMom/2 - 1), a);
    wave_lds_order();
  }
};

__device__ __forceinline__ double box_rmax2(const NodeArgs& a, int n) {
#pragma clang fp contract(off)
  const double4 gh = a.geo_h[n];
  return gh.x*gh.x + gh.y*gh.y + gh.z*gh.z;
}

// Phase 1, fused with the leaf moments.
template <bool HONLY>
__global__ __launch_bounds__(RB) void k_refit_chunks(
    int N, const double* __restrict__ x, const double* __restrict__ y,
    const double* __restrict__ z, const double* __restrict__ mass, const double* __restrict__ h,
    const int* __restrict__ parent, const int4* __restrict__ lnk, double theta2, NodeArgs a,
    int* __restrict__ front, int* __restrict__ nfront) {
#pragma clang fp contract(off)
  __shared__ RefitSlots<HONLY, RB> sd;
  __shared__ int arr[RB];               // arrivals at internal node c0 + t
  __shared__ int ipar[RB];              // its parent
  __shared__ int lr[RB];                // its children's slots, left | right << 16; -1 if not inside
  __shared__ int fr[RB];                // the maximal node that starts at leaf c0 + t, or -1
  __shared__ short list[2][RB/2];       // nodes to merge
  __shared__ int cnt[3];
  __shared__ int wsum[RB/kWave];
  const int t = threadIdx.x;
  const int c0 = blockIdx.x*RB;
  const int c1 = min(c0 + RB, N) - 1;
  const int l = c0 + t;
  arr[t] = 0;
  fr[t] = -1;
  lr[t] = -1;
  if (t < 3) cnt[t] = 0;
  int up = -1;
  double rmax2 = 0.0;                   // HONLY: of internal node c0 + t
  if (l <= c1) {
    up = parent[N - 1 + l];
    if (l < N - 1) {
      ipar[t] = parent[l];
      const int4 k = lnk[l];            // (first, last, left, right)
      if (k.x >= c0 && k.y <= c1) {
        const int split = k.z >= N - 1 ? k.z - (N - 1) : k.z;      // last leaf of the left child
        lr[t] = (k.x - c0) | (split + 1 - c0) << 16;
      }
      if (HONLY) rmax2 = box_rmax2(a, l);
    }
    const int n = N - 1 + l;
    const double hh = h[l];
    NodeD d;
    d.hmax = hh;
    if (HONLY) {
      a.geo_c[n].w = hh;
      a.geo_h[n].w = hh*hh/theta2;
    } else {
      const double r[3] = {x[l], y[l], z[l]};
      for (int k = 0; k < 3; k++) { d.lo[k] = r[k]; d.hi[k] = r[k]; d.com[k] = r[k]; }
      d.m = mass[l];
      for (int k = 0; k < 5; k++) d.q[k] = 0.0;
      a.geo_c[n] = make_double4(r[0], r[1], r[2], hh);
      a.geo_h[n] = make_double4(0.0, 0.0, 0.0, hh*hh/theta2);
    }
    sd.put(t, d);
  }
  // HONLY: the half-diagonals wait for their merge in LDS
  __shared__ double rm[HONLY ? RB : 1];
  if (HONLY) rm[t] = rmax2;
  __syncthreads();
  // node n with parent p, starting at slot s, is finished
  auto arrive = [&](int n, int p, int s, int b) {
    if (p < 0) return;
    if (p < c0 || p > c1 || lr[p - c0] < 0) fr[s] = n;
    else if (atomicAdd(&arr[p - c0], 1) == 1) list[b & 1][atomicAdd(&cnt[b % 3], 1)] = (short) (p - c0);
  };
  if (l <= c1) arrive(N - 1 + l, up, t, 0);
  if (!HONLY)
    for (int k = t; k <= (c1 - c0)*(kMom/2) + kMom/2 - 1; k += RB)
      sd.part_out(k/(kMom/2), N - 1 + c0 + k/(kMom/2), k & (kMom/2 - 1), a);
  __syncthreads();
  for (int b = 0; ; b++) {
    const int n = cnt[b % 3];
    if (n == 0) break;
    if (t == 0) cnt[(b + 2) % 3] = 0;
    if (t < n) {
      const int q = list[b & 1][t], w = lr[q], L = w & 0xffff;
      sd.merge(L, w >> 16, c0 + q, HONLY ? rm[q] : 0.0, theta2, a);
      arrive(c0 + q, ipar[q], L, b + 1);
    }
    const short* w = list[b & 1] + t/kWave*kWave;
    sd.records_out(min(n - t/kWave*kWave, kWave), [&](int j) { return c0 + w[j]; },
                   [&](int j) { return lr[w[j]] & 0xffff; }, a);
    __syncthreads();
  }
  // the maximal nodes in leaf order
  const int node = fr[t];
  const unsigned long long m = __ballot(node >= 0);
  if (lane_id() == 0) wsum[t/kWave] = __popcll(m);
  __syncthreads();
  int o = 0, total = 0;
  for (int w = 0; w < RB/kWave; w++) {
    if (w < t/kWave) o += wsum[w];
    total += wsum[w];
  }
  if (node >= 0) front[c0 + o + lanes_below(m)] = node;
  if (t == 0) nfront[blockIdx.x] = total;
}

// Later phases: runs [blk RS, blk RS + RS) of `span` leaves each, the run starting at leaf f having
// its maximal nodes at in[f ...], nin of them; their merge leaves out[lo ...] and nout.  More nodes
// than the workgroup holds are merged a window at a time until they fit (a window of RF adjacent
// nodes leaves at most two a level of the tree).
template <bool HONLY>
__global__ __launch_bounds__(RT) void k_refit_runs(
    int N, int nruns, long long span, const int* __restrict__ parent, const int4* __restrict__ lnk,
    double theta2, NodeArgs a, const int* __restrict__ in, const int* __restrict__ nin,
    int* __restrict__ out, int* __restrict__ nout) {
#pragma clang fp contract(off)
  struct Ready { int node, parent; short left, right; };
  __shared__ RefitSlots<HONLY, RF> sd;
  __shared__ int nd[RF];                // the node starting at slot s, or -1
  __shared__ short en[RF];              // one past its last slot
  __shared__ int arr[RF + 1];           // arrivals at the node whose right child starts at slot s
  __shared__ short lft[RF + 1];         // ... and the slot of its left child, once that arrived
  __shared__ Ready list[2][RF/2];
  __shared__ double rm[HONLY ? RF + 1 : 1];      // ... and its box's squared half-diagonal
  __shared__ int cnt[3];
  __shared__ int pre[RS + 1];
  const int t = threadIdx.x;
  const int k0 = blockIdx.x*RS, k1 = min(k0 + RS, nruns);
  const int lo = (int) (k0*span), hi = (int) min(k1*span, (long long) N) - 1;
  if (t == 0) {
    pre[0] = 0;
    for (int c = 0; c < RS; c++) pre[c + 1] = pre[c] + (k0 + c < k1 ? nin[k0 + c] : 0);
  }
  __syncthreads();
  int total = pre[RS];
  bool first = true;                    // nodes still in `in`, run by run; else in out[lo ...]
  for (;;) {
    int done = 0;                       // nodes left by the windows so far
    for (int w0 = 0; w0 < total; w0 += RF) {
      const int F = min(RF, total - w0);
      if (t < 3) cnt[t] = 0;
      for (int s = t; s < F; s += RT) {
        int n;
        if (first) {
          int c = 0;
          while (pre[c + 1] <= w0 + s) c++;
          n = in[(size_t) ((k0 + c)*span) + (w0 + s - pre[c])];
        } else {
          n = out[lo + w0 + s];
        }
        nd[s] = n;
        en[s] = (short) (s + 1);
        if (HONLY) sd.v[sd.at(s)] = a.geo_c[n].w;
      }
      for (int s = t; s <= F; s += RT) arr[s] = 0;
      __syncthreads();
      if (!HONLY) {
        for (int k = t; k < F*(kMom/2); k += RT)
          sd.part_in(k/(kMom/2), nd[k/(kMom/2)], k & (kMom/2 - 1), a);
      }
      // node n with parent p and its topology, slots [s, e), is finished
      struct Up { int4 k; int parent; double rmax2; };
      auto above = [&](int p) {
        Up u = {make_int4(0, 0, 0, 0), -1, 0.0};
        if (p < 0) return u;
        u.k = lnk[p];                   // (first, last, left, right)
        u.parent = parent[p];
        if (HONLY) u.rmax2 = box_rmax2(a, p);
        return u;
      };
      auto arrive = [&](int n, int p, const Up& u, int s, int e, int b) {
        if (p < 0 || u.k.x < lo || u.k.y > hi) return;
        const bool isleft = u.k.z == n;
        const int r = isleft ? e : s;
        if (isleft) lft[r] = (short) s;
        if (__hip_atomic_fetch_add(&arr[r], 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP) == 0)
          return;
        if (HONLY) rm[r] = u.rmax2;
        list[b & 1][atomicAdd(&cnt[b % 3], 1)] = {p, u.parent, lft[r], (short) r};
      };
      for (int s = t; s < F; s += RT) {
        const int p = parent[nd[s]];
        arrive(nd[s], p, above(p), s, s + 1, 0);
      }
      __syncthreads();
      for (int b = 0; ; b++) {
        const int n = cnt[b % 3];
        if (n == 0) break;
        if (t == 0) cnt[(b + 2) % 3] = 0;
        if (t < n) {
          const Ready q = list[b & 1][t];
          const Up u = above(q.parent);    // in flight during the merge
          sd.merge(q.left, q.right, q.node, HONLY ? rm[q.right] : 0.0, theta2, a);
          const int e = en[q.right];
          nd[q.right] = -1;
          nd[q.left] = q.node;
          en[q.left] = (short) e;
          arrive(q.node, q.parent, u, q.left, e, b + 1);
        }
        const Ready* w = list[b & 1] + t/kWave*kWave;
        sd.records_out(min(n - t/kWave*kWave, kWave), [&](int j) { return w[j].node; },
                       [&](int j) { return (int) w[j].left; }, a);
        __syncthreads();
      }
      // what is left, in leaf order, by the first wavefront
      int left = 0;
      for (int s0 = 0; s0 < F; s0 += kWave) {
        const int s = s0 + (t & (kWave - 1));
        const int n = s < F ? nd[s] : -1;
        const unsigned long long m = __ballot(n >= 0);
        if (t < kWave && n >= 0) out[lo + done + left + lanes_below(m)] = n;
        left += __popcll(m);
      }
      done += left;
      __syncthreads();
    }
    const bool more = total > RF && done < total;
    total = done;
    first = false;
    if (!more) break;
  }
  if (t == 0) nout[blockIdx.x] = total;
}

template <bool HONLY>
void launch_refit(gdf_ctx* c, const NodeArgs& na, double theta2) {
  const int N = c->N;
  hipStream_t s = c->stream;
  int nrun = (N + RB - 1)/RB;
  int* from = c->front;                            // N entries a buffer, and a count a run
  int* to = from + N;
  int* nfrom = to + N;
  int* nto = nfrom + nrun;
  k_refit_chunks<HONLY><<<nrun, RB, 0, s>>>(N, c->pf[F_X], c->pf[F_Y], c->pf[F_Z], c->pf[F_M],
                                            c->pf[F_H], c->parent, c->lnk, theta2, na, from,
                                            nfrom);
  for (long long span = RB; nrun > 1; span *= RS) {
    const int nb = (nrun + RS - 1)/RS;
    k_refit_runs<HONLY><<<nb, RT, 0, s>>>(N, nrun, span, c->parent, c->lnk, theta2, na, from, nfrom,
                                          to, nto);
    std::swap(from, to);
    std::swap(nfrom, nto);
    nrun = nb;
  }
}

__global__ void k_hleaves(int N, const double* __restrict__ h, double theta2, NodeArgs a) {
  const int l = blockIdx.x*BS + threadIdx.x;
  if (l >= N) return;
  const int n = N - 1 + l;
  const double hh = h[l];
  double4 gc = a.geo_c[n]; gc.w = hh; a.geo_c[n] = gc;
  double4 gh = a.geo_h[n]; gh.w = __ddiv_rn(__dmul_rn(hh, hh), theta2); a.geo_h[n] = gh;
}

// Order-preserving compaction of n byte flags (0 or 1; zero-padded to a multiple of 16) into the
// indices of the set ones, their count at out[cap]: a workgroup takes 1024 flags, 16 a lane, and
// counts the flags before its own by itself, so that it waits for no other.  It may run while
// another stream's kernels fill the device: a look-back scan then stalls until its predecessors find
// a compute unit, and any workgroup that needs LDS waits until enough LDS is free on one CU (both
// measured at up to 2-4 ms beside the gravity walk); a wavefront without LDS starts at once.  Bound
// by the latency of two loads: 23600 flags of a million particles in 5.5 us, where one wavefront alone
// for all of them took 24.
__device__ __forceinline__ int flag_count(uint4 x) {                // bytes are 0 or 1
  return __popc(x.x) + __popc(x.y) + __popc(x.z) + __popc(x.w);
}

__global__ __launch_bounds__(64) void k_compact_flags(int n, const uint4* __restrict__ blocks,
                                                      int* __restrict__ out, int cap) {
  const int lane = threadIdx.x, nblk = (n + 15)/16;
  const int first = blockIdx.x*kWave, own = first + lane;
  const uint4 x = own < nblk ? blocks[own] : make_uint4(0, 0, 0, 0);
  int before = 0;
  #pragma unroll 8
  for (int b = 0; b < first; b += kWave) before += flag_count(blocks[b + lane]);
  for (int d = 32; d >= 1; d >>= 1) before += __shfl_xor(before, d, kWave);
  const int cnt = flag_count(x), incl = wave_incl_scan(cnt);
  int o = before + incl - cnt;
  const unsigned wd[4] = {x.x, x.y, x.z, x.w};
  for (int k = 0; k < 4; k++) {
    if (!wd[k]) continue;
    for (int q = 0; q < 4; q++)
      if ((wd[k] >> (8*q)) & 1u) out[o++] = 16*own + 4*k + q;
  }
  if (blockIdx.x == gridDim.x - 1 && lane == kWave - 1) out[cap] = before + incl;
}

// one wavefront per walk group: does any of its particles have status 1?
__global__ void k_group_flags(int ngroups, const int* __restrict__ grp_first,
                              const int* __restrict__ grp_count, const int* __restrict__ status,
                              unsigned char* __restrict__ flags, int* __restrict__ ncand,
                              int* __restrict__ gnc, int* __restrict__ gnn,
                              int* __restrict__ zero, int nzero) {
  const int g = blockIdx.x*(BS/kWave) + threadIdx.x/kWave;
  const int lane = threadIdx.x % kWave;
  if (blockIdx.x == 0 && (int) threadIdx.x < nzero) zero[threadIdx.x] = 0;
  if (g >= ngroups) return;
  const bool on = lane < grp_count[g] && status[grp_first[g] + lane] == 1;
  const bool any = __ballot(on) != 0;
  if (lane == 0) {
    flags[g] = any ? 1 : 0;
    // the compaction reads whole 16-byte blocks: the bytes after the last flag read 0
    if (g == ngroups - 1)
      for (int k = ngroups; k & 15; k++) flags[k] = 0;
    if (!any) {
      if (ncand) ncand[g] = 0;
      if (gnc) { gnc[g] = 0; gnn[g] = 0; }
    }
  }
}

}  // namespace

TreeView tree_view(const gdf_ctx* c) {
  TreeView v;
  v.N = c->N; v.left = c->left; v.right = c->right; v.first = c->first; v.last = c->last;
  v.geo_c = c->geo_c; v.geo_h = c->geo_h; v.mp = c->mp;
  return v;
}

static NodeArgs node_args(gdf_ctx* c) {
  NodeArgs a; a.geo_c = c->geo_c; a.geo_h = c->geo_h;
  a.mp = c->mp;
  return a;
}

int seg_alloc(gdf_ctx* c) {
  if (c->d_seg_off) return GDF_OK;
  GDF_HIP(c, hipMalloc(&c->d_seg_off, sizeof(int)*(kMaxSeg + 1)));
  GDF_HIP(c, hipMalloc(&c->seg_root, sizeof(int)*kMaxSeg));
  GDF_HIP(c, hipMalloc(&c->seg_dt, sizeof(double)*kMaxSeg));
  GDF_HIP(c, hipMalloc(&c->seg_bnd, sizeof(double)*4*kMaxSeg));
  GDF_HIP(c, hipMalloc(&c->seg_bad, sizeof(int)*kMaxSeg));
  return GDF_OK;
}

// segment offsets to the device and the per-particle segment ids
__global__ void k_fill_seg(int n0, int n1, int sg, int* __restrict__ seg) {
  const int i = n0 + blockIdx.x*BS + threadIdx.x;
  if (i < n1) seg[i] = sg;
}

int seg_upload(gdf_ctx* c) {
  GDF_TRY(seg_alloc(c));
  if (c->nseg < 1 || c->nseg > kMaxSeg || (int) c->seg_off.size() != c->nseg + 1)
    return fail(c, GDF_ERR_INVALID, "bad segment table");
  GDF_HIP(c, hipMemcpyAsync(c->d_seg_off, c->seg_off.data(), sizeof(int)*(c->nseg + 1),
                            hipMemcpyHostToDevice, c->stream));
  for (int sg = 0; sg < c->nseg; sg++) {
    const int n0 = c->seg_off[sg], n1 = c->seg_off[sg + 1];
    if (n1 > n0) k_fill_seg<<<nblocks(n1 - n0, BS), BS, 0, c->stream>>>(n0, n1, sg, c->pi[I_SEG]);
  }
  GDF_HIP(c, hipGetLastError());
  c->tree_valid = false;
  c->topo_valid = false;
  return GDF_OK;
}

int tree_alloc(gdf_ctx* c) {
  const size_t N = (size_t) c->Ncap;
  const size_t nn = 2*N;  // >= 2N-1
  GDF_HIP(c, hipMalloc(&c->keys, sizeof(uint64_t)*N));
  GDF_HIP(c, hipMalloc(&c->keys_alt, sizeof(uint64_t)*N));
  GDF_HIP(c, hipMalloc(&c->vals, sizeof(int)*N));
  GDF_HIP(c, hipMalloc(&c->vals_alt, sizeof(int)*N));
  GDF_HIP(c, hipMalloc(&c->left, sizeof(int)*N));
  GDF_HIP(c, hipMalloc(&c->right, sizeof(int)*N));
  GDF_HIP(c, hipMalloc(&c->first, sizeof(int)*N));
  GDF_HIP(c, hipMalloc(&c->last, sizeof(int)*N));
  GDF_HIP(c, hipMalloc(&c->parent, sizeof(int)*nn));
  GDF_HIP(c, hipMalloc(&c->lnk, sizeof(int4)*N));
  GDF_HIP(c, hipMalloc(&c->visit, sizeof(int)*(N + 16)));   // 16-byte-padded byte flags
  // refit frontiers: two buffers of N nodes that the phases use in turn, and a count a run for each
  GDF_HIP(c, hipMalloc(&c->front, sizeof(int)*(2*N + 2*(N/1024 + 16))));
  GDF_HIP(c, hipMalloc(&c->geo_c, sizeof(double4)*nn));
  GDF_HIP(c, hipMalloc(&c->geo_h, sizeof(double4)*nn));
  GDF_HIP(c, hipMalloc(&c->mp, sizeof(double)*kMom*nn));
  GDF_HIP(c, hipMalloc(&c->gstart, sizeof(int)*N));
  GDF_HIP(c, hipMalloc(&c->grp_first, sizeof(int)*N));
  GDF_HIP(c, hipMalloc(&c->grp_count, sizeof(int)*N));
  GDF_HIP(c, hipMalloc(&c->grp_node, sizeof(int)*N));
  GDF_HIP(c, hipMalloc(&c->grp_root, sizeof(int)*N));
  GDF_HIP(c, hipMalloc(&c->grp_gmac, sizeof(double)*N));
  GDF_HIP(c, hipMalloc(&c->nsel, sizeof(int)*4));
  // temporary storage of the sort and the group compaction
  size_t b1 = 0, b2 = 0;
  GDF_HIP(c, rocprim::radix_sort_pairs(nullptr, b1, c->keys, c->keys_alt, c->vals, c->vals_alt,
                                       (unsigned int) N, 0, 64, c->stream));
  b2 = sizeof(int)*((size_t) nblocks(nblocks((long long) N, 16), kSelBlock) + 16);
  c->sort_tmp_bytes = b1;
  c->sel_tmp_bytes = b2;
  GDF_HIP(c, hipMalloc(&c->sort_tmp, b1 > 0 ? b1 : 16));
  GDF_HIP(c, hipMalloc(&c->sel_tmp, b2 > 0 ? b2 : 16));
  return GDF_OK;
}

namespace {

// The marked group starts (gstart[i] >= 0: the group's node) in ascending order: per-block counts,
// an exclusive scan of them by one workgroup, and a scatter of the groups' first particles, nodes
// and sizes; up to kSelSmall particles all in one workgroup.  No memset and no library call, so the
// tree build's launches capture into a graph of kernel nodes only.  (Marked by a pass over all
// nodes into cleared byte flags, with a pass over the groups for their nodes, it was six launches, 21
// to 28 us and the gaps between them; now 4 us for 4096 particles, 14 for 20011, 17 in three launches
// for 131072.)
constexpr int kSelPer = 16;                // particles a thread
constexpr int kSelSmall = 32768;

struct SelOut { int* first; int* node; int* count; };

// marks i .. i + 3 of N (unmarked past the end)
__device__ __forceinline__ int4 sel_marks(int N, int i, const int* __restrict__ gstart) {
  if (i + 3 < N) return *reinterpret_cast<const int4*>(gstart + i);
  return make_int4(i < N ? gstart[i] : -1, i + 1 < N ? gstart[i + 1] : -1,
                   i + 2 < N ? gstart[i + 2] : -1, -1);
}
__device__ __forceinline__ int sel_count(int4 m) {
  return (m.x >= 0) + (m.y >= 0) + (m.z >= 0) + (m.w >= 0);
}
__device__ __forceinline__ int sel_write(int4 m, int i, int o, const int* __restrict__ gsize,
                                         const SelOut& out) {
  const int n[4] = {m.x, m.y, m.z, m.w};
  #pragma unroll
  for (int k = 0; k < 4; k++)
    if (n[k] >= 0) {
      out.first[o] = i + k; out.node[o] = n[k]; out.count[o] = gsize[i + k];
      o++;
    }
  return o;
}

// exclusive scan over a workgroup of up to 16 wavefronts, its sum into total
__device__ __forceinline__ int block_scan(int v, int& total) {
  __shared__ int sum[16];
  const int w = threadIdx.x/kWave;
  const int incl = wave_incl_scan(v);
  if ((threadIdx.x & (kWave - 1)) == kWave - 1) sum[w] = incl;
  __syncthreads();
  int before = 0;
  total = 0;
  for (int k = 0; k < (int) blockDim.x/kWave; k++) {
    if (k < w) before += sum[k];
    total += sum[k];
  }
  __syncthreads();
  return before + incl - v;
}

__global__ __launch_bounds__(1024) void k_sel_small(int N, const int* __restrict__ gstart,
                                                    const int* __restrict__ gsize,
                                                    int* __restrict__ ngroups, SelOut out) {
  int run = 0;
  int4 next = sel_marks(N, 4*threadIdx.x, gstart);
  for (int base = 0; base < N; base += 4096) {
    const int i = base + 4*threadIdx.x;
    const int4 m = next;
    next = sel_marks(N, i + 4096, gstart);
    int total;
    const int o = run + block_scan(sel_count(m), total);
    sel_write(m, i, o, gsize, out);
    run += total;
  }
  if (threadIdx.x == 0) *ngroups = run;
}

__global__ __launch_bounds__(kSelBlock) void k_sel_count(int N, const int* __restrict__ gstart,
                                                         int* __restrict__ bcount) {
  const int i0 = (blockIdx.x*kSelBlock + threadIdx.x)*kSelPer;
  int c = 0, total;
  for (int i = i0; i < i0 + kSelPer; i += 4) c += sel_count(sel_marks(N, i, gstart));
  (void) block_scan(c, total);
  if (threadIdx.x == 0) bcount[blockIdx.x] = total;
}

// exclusive scan of nb block counts in place, the total into *ngroups; one workgroup
__global__ __launch_bounds__(1024) void k_sel_scan(int nb, int* __restrict__ bcount,
                                                   int* __restrict__ ngroups) {
  const int per = (nb + 1023)/1024;
  const int b0 = min((int) threadIdx.x*per, nb), b1 = min(b0 + per, nb);
  int sum = 0, total;
  for (int b = b0; b < b1; b++) sum += bcount[b];
  int run = block_scan(sum, total);
  for (int b = b0; b < b1; b++) { const int v = bcount[b]; bcount[b] = run; run += v; }
  if (threadIdx.x == 0) *ngroups = total;
}

__global__ __launch_bounds__(kSelBlock) void k_sel_scatter(int N, const int* __restrict__ gstart,
                                                           const int* __restrict__ gsize,
                                                           const int* __restrict__ boff,
                                                           SelOut out) {
  const int i0 = (blockIdx.x*kSelBlock + threadIdx.x)*kSelPer;
  int4 m[kSelPer/4];
  int c = 0, total;
  #pragma unroll
  for (int k = 0; k < kSelPer/4; k++) {
    m[k] = sel_marks(N, i0 + 4*k, gstart);
    c += sel_count(m[k]);
  }
  int o = boff[blockIdx.x] + block_scan(c, total);
  #pragma unroll
  for (int k = 0; k < kSelPer/4; k++) o = sel_write(m[k], i0 + 4*k, o, gsize, out);
}

// Steps 1-6 of a tree build: every launch that needs no value back on the host.  The host's
// buffer swaps (double-buffered keys, indices and particle state) run with launch == false
// too, so a replayed graph of these launches leaves the host state as the launches themselves
// would.
int build_body(gdf_ctx* c, hipStream_t s, bool launch) {
  const int N = c->N;
  const int nbp = std::min(nblocks(N, BS), 1024);
  // 1. bounds and Morton keys
  if (launch) {
    if (c->nseg > 0) {
      k_seg_bounds_partial<<<dim3(kSegBlocks, c->nseg), BS, 0, s>>>(c->d_seg_off, c->pf[F_X],
                                                                    c->pf[F_Y], c->pf[F_Z],
                                                                    c->red);
      k_seg_bounds_final<<<c->nseg, 64, 0, s>>>(c->red, c->seg_bnd);
      k_morton_seg<<<nblocks(N, BS), BS, 0, s>>>(N, c->pf[F_X], c->pf[F_Y], c->pf[F_Z],
                                                 c->pi[I_SEG], c->seg_bnd, c->keys, c->vals, c->gstart);
    } else {
      k_bounds_partial<<<nbp, BS, 0, s>>>(N, c->pf[F_X], c->pf[F_Y], c->pf[F_Z], c->red);
      k_bounds_final<<<1, BS, 0, s>>>(nbp, c->red, c->red + 6*1024);
      k_morton<<<nblocks(N, BS), BS, 0, s>>>(N, c->pf[F_X], c->pf[F_Y], c->pf[F_Z],
                                             c->red + 6*1024, c->keys, c->vals, c->gstart);
    }
    // 2. stable radix sort of (key, index)
    size_t bytes = c->sort_tmp_bytes;
    GDF_HIP(c, rocprim::radix_sort_pairs(c->sort_tmp, bytes, c->keys, c->keys_alt, c->vals,
                                         c->vals_alt, (unsigned int) N, 0,
                                         c->nseg > 0 ? 64 : 63, s));
  }
  std::swap(c->keys, c->keys_alt);
  std::swap(c->vals, c->vals_alt);
  // 3. permute persistent particle state into key order
  if (launch) {
    PermArgs pa;
    for (int f = 0; f < F_NPERSIST; f++) { pa.src[f] = c->pf[f]; pa.dst[f] = c->pf_alt[f]; }
    for (int f = 0; f < I_NINT; f++) { pa.isrc[f] = c->pi[f]; pa.idst[f] = c->pi_alt[f]; }
    k_permute<<<nblocks(N, BS), BS, 0, s>>>(N, c->vals, pa, c->iorig, c->iorig_alt);
  }
  for (int f = 0; f < F_NPERSIST; f++) std::swap(c->pf[f], c->pf_alt[f]);
  for (int f = 0; f < I_NINT; f++) std::swap(c->pi[f], c->pi_alt[f]);
  std::swap(c->iorig, c->iorig_alt);
  if (c->df_alt[0]) {
    if (launch) {
      PermDArgs pd;
      for (int k = 0; k < kNPermD; k++) {
        pd.src[k] = c->df[kPermD[k]]; pd.dst[k] = c->df_alt[kPermD[k]];
      }
      k_permute_d<<<nblocks(N, BS), BS, 0, s>>>(N, c->vals, pd);
    }
    for (int k = 0; k < kNPermD; k++) std::swap(c->df[kPermD[k]], c->df_alt[kPermD[k]]);
  }
  if (!launch) return GDF_OK;
  // 4. topology
  if (N > 1)
    k_lbvh<<<nblocks(N - 1, BS), BS, 0, s>>>(N, c->cfg.group_max, c->nseg > 0, c->gstart, c->visit, c->keys, c->left, c->right, c->first, c->last,
                                             c->parent, c->lnk);
  // 5. moments, bottom-up
  NodeArgs na = node_args(c);
  const double theta2 = c->phys.thetamaxsqd;
  if (N > 1)
    launch_refit<false>(c, na, theta2);
  else
    k_leaves<<<1, BS, 0, s>>>(N, c->pf[F_X], c->pf[F_Y], c->pf[F_Z], c->pf[F_M], c->pf[F_H],
                              theta2, na, c->parent, c->gstart, c->visit);
  // 6. walk groups in ascending first-particle order
  const SelOut out = {c->grp_first, c->grp_node, c->grp_count};
  if (N <= kSelSmall) {
    k_sel_small<<<1, 1024, 0, s>>>(N, c->gstart, c->visit, c->nsel, out);
  } else {
    const int nsb = nblocks(nblocks(N, kSelPer), kSelBlock);
    int* bcount = reinterpret_cast<int*>(c->sel_tmp);
    k_sel_count<<<nsb, kSelBlock, 0, s>>>(N, c->gstart, bcount);
    k_sel_scan<<<1, 1024, 0, s>>>(nsb, bcount, c->nsel);
    k_sel_scatter<<<nsb, kSelBlock, 0, s>>>(N, c->gstart, c->visit, bcount, out);
  }
  GDF_HIP(c, hipGetLastError());
  return GDF_OK;
}

// every buffer pointer the build swaps, in a fixed order: with the particle count, segment
// count and configuration of the context it keys a captured graph
std::vector<const void*> build_key(const gdf_ctx* c) {
  std::vector<const void*> k = {c->keys, c->keys_alt, c->vals, c->vals_alt, c->iorig,
                                c->iorig_alt, c->df_alt[0]};
  for (int f = 0; f < F_NPERSIST; f++) { k.push_back(c->pf[f]); k.push_back(c->pf_alt[f]); }
  for (int f = 0; f < I_NINT; f++) { k.push_back(c->pi[f]); k.push_back(c->pi_alt[f]); }
  for (int i = 0; i < kNPermD; i++) {
    k.push_back(c->df[kPermD[i]]); k.push_back(c->df_alt[kPermD[i]]);
  }
  // every other buffer and value the launches take
  const void* other[] = {c->d_seg_off, c->seg_bnd, c->red, c->sort_tmp, c->sel_tmp, c->nsel,
                         c->left, c->right, c->first, c->last, c->parent, c->lnk, c->visit, c->front,
                         c->geo_c, c->geo_h, c->mp, c->gstart, c->grp_first,
                         c->grp_count, c->grp_node};
  for (const void* q : other) k.push_back(q);
  uint64_t theta_bits;
  std::memcpy(&theta_bits, &c->phys.thetamaxsqd, sizeof(theta_bits));
  const uint64_t vals[] = {(uint64_t) c->N, (uint64_t) c->nseg, (uint64_t) c->sort_tmp_bytes,
                           (uint64_t) c->sel_tmp_bytes, (uint64_t) c->cfg.group_max, theta_bits};
  for (uint64_t v : vals) k.push_back(reinterpret_cast<const void*>((uintptr_t) v));
  return k;
}

// a captured graph is used only if it holds kernel and copy nodes (no memset nodes, whose
// replays are not trusted here)
// returns 0, or 100 + the type of the first node of another kind
int graph_nodes_check(hipGraph_t g) {
  size_t n = 0;
  if (hipGraphGetNodes(g, nullptr, &n) != hipSuccess) return 99;
  std::vector<hipGraphNode_t> nodes(n);
  if (n > 0 && hipGraphGetNodes(g, nodes.data(), &n) != hipSuccess) return 99;
  for (hipGraphNode_t nd : nodes) {
    hipGraphNodeType t;
    if (hipGraphNodeGetType(nd, &t) != hipSuccess) return 99;
    if (t != hipGraphNodeTypeKernel && t != hipGraphNodeTypeMemcpy &&
        t != hipGraphNodeTypeEmpty)
      return 100 + (int) t;
  }
  return 0;
}

// the build's launches through a graph captured at the first build of each buffer
// arrangement (the swaps alternate between two) and replayed after; a capture that fails or
// holds other nodes leaves the context building eagerly
int build_launches(gdf_ctx* c, hipStream_t s) {
  if (!c->cfg.graph_capture || c->graph_failed) return build_body(c, s, true);
  const std::vector<const void*> key = build_key(c);
  for (int e = 0; e < gdf_ctx::kBuildGraphs; e++)
    if (c->bg_exec[e] && c->bg_key[e] == key) {
      GDF_HIP(c, hipGraphLaunch(c->bg_exec[e], s));
      c->graph_replays++;
      return build_body(c, s, false);
    }
  // capture: the host swaps happen during the capture, so they are undone afterwards (the
  // replay below redoes them)
  struct Saved {
    double* pf[F_NPERSIST]; double* pf_alt[F_NPERSIST];
    int* pi[I_NINT]; int* pi_alt[I_NINT];
    double* df[D_NDERIVED]; double* df_alt[D_NDERIVED];
    uint64_t* keys; uint64_t* keys_alt; int* vals; int* vals_alt; int* iorig; int* iorig_alt;
  } sv;
  std::copy(std::begin(c->pf), std::end(c->pf), sv.pf);
  std::copy(std::begin(c->pf_alt), std::end(c->pf_alt), sv.pf_alt);
  std::copy(std::begin(c->pi), std::end(c->pi), sv.pi);
  std::copy(std::begin(c->pi_alt), std::end(c->pi_alt), sv.pi_alt);
  std::copy(std::begin(c->df), std::end(c->df), sv.df);
  std::copy(std::begin(c->df_alt), std::end(c->df_alt), sv.df_alt);
  sv.keys = c->keys; sv.keys_alt = c->keys_alt; sv.vals = c->vals; sv.vals_alt = c->vals_alt;
  sv.iorig = c->iorig; sv.iorig_alt = c->iorig_alt;
  auto restore = [&]() {
    std::copy(sv.pf, sv.pf + F_NPERSIST, c->pf);
    std::copy(sv.pf_alt, sv.pf_alt + F_NPERSIST, c->pf_alt);
    std::copy(sv.pi, sv.pi + I_NINT, c->pi);
    std::copy(sv.pi_alt, sv.pi_alt + I_NINT, c->pi_alt);
    std::copy(sv.df, sv.df + D_NDERIVED, c->df);
    std::copy(sv.df_alt, sv.df_alt + D_NDERIVED, c->df_alt);
    c->keys = sv.keys; c->keys_alt = sv.keys_alt; c->vals = sv.vals; c->vals_alt = sv.vals_alt;
    c->iorig = sv.iorig; c->iorig_alt = sv.iorig_alt;
  };
  hipGraph_t g = nullptr;
  hipGraphExec_t ex = nullptr;
  // why a capture was given up, kept for gdf_graph_state: 1 begin, 2 a launch, 3 end,
  // 100 + node type of a node that is not a kernel or copy, 4 instantiation
  int why = 0;
  if (hipStreamBeginCapture(s, hipStreamCaptureModeRelaxed) != hipSuccess) {
    why = 1;
  } else {
    const int rc = build_body(c, s, true);
    const hipError_t ee = hipStreamEndCapture(s, &g);
    if (rc != GDF_OK) why = 2;
    else if (ee != hipSuccess || !g) why = 3;
    else if (const int nt = graph_nodes_check(g)) why = nt;
    else if (hipGraphInstantiate(&ex, g, nullptr, nullptr, 0) != hipSuccess) why = 4;
  }
  const bool ok = why == 0;
  c->graph_why = why;
  if (g) (void) hipGraphDestroy(g);
  // a capture invalidated part way (by another thread's call on the device, say) may leave the
  // stream capturing: end it, and clear the error it left, before building eagerly
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone) {
    hipGraph_t g2 = nullptr;
    (void) hipStreamEndCapture(s, &g2);
    if (g2) (void) hipGraphDestroy(g2);
  }
  (void) hipGetLastError();
  restore();
  if (!ok) {
    if (ex) (void) hipGraphExecDestroy(ex);
    c->graph_failed = true;
    return build_body(c, s, true);
  }
  const int e = c->bg_next;
  c->bg_next = (c->bg_next + 1)%gdf_ctx::kBuildGraphs;
  if (c->bg_exec[e]) (void) hipGraphExecDestroy(c->bg_exec[e]);
  c->bg_exec[e] = ex;
  c->bg_key[e] = key;
  GDF_HIP(c, hipGraphLaunch(ex, s));
  return build_body(c, s, false);
}

}  // namespace

void build_graphs_free(gdf_ctx* c) {
  for (int e = 0; e < gdf_ctx::kBuildGraphs; e++) {
    if (c->bg_exec[e]) (void) hipGraphExecDestroy(c->bg_exec[e]);
    c->bg_exec[e] = nullptr;
    c->bg_key[e].clear();
  }
}

int tree_build(gdf_ctx* c) {
  const int N = c->N;
  hipStream_t s = c->stream;
  if (N <= 0) return fail(c, GDF_ERR_INVALID, "tree build without particles");
  GDF_TRY(build_launches(c, s));
  GDF_HIP(c, hipMemcpyAsync(c->h_counters, c->nsel, sizeof(int), hipMemcpyDeviceToHost, s));
  GDF_HIP(c, hipStreamSynchronize(s));
  c->ngroups = c->h_counters[0];
  if (c->ngroups <= 0 || c->ngroups > N) return fail(c, GDF_ERR_INVALID, "walk group build failed");
  if (c->nseg > 0) {
    k_seg_roots<<<nblocks(2*N - 1, BS), BS, 0, s>>>(N, c->nseg, c->d_seg_off, c->first, c->last,
                                                    c->pi[I_SEG], c->seg_root);
    k_grp_roots<<<nblocks(c->ngroups, BS), BS, 0, s>>>(c->ngroups, c->grp_first, c->pi[I_SEG],
                                                       c->seg_root, c->grp_root);
  }
  // the force arrays follow the new order only when the build permuted them
  GDF_TRY(group_mac(c, c->df_alt[0] ? nullptr : c->vals));
  c->tree_valid = true;
  c->topo_valid = true;
  sph_drop_lists(c);
  GDF_HIP(c, hipGetLastError());
  return integ_pack_posm(c);
}

// The kept topology and walk groups with every node's box, moments and hmax recomputed from the
// particles' current state: the bottom-up pass of a build without the sort, the permutation and
// the group selection.  Synchronises the stream, as a build does.
int tree_restock(gdf_ctx* c) {
  const int N = c->N;
  hipStream_t s = c->stream;
  if (!c->topo_valid) return fail(c, GDF_ERR_INVALID, "tree refit without a built tree");
  NodeArgs na = node_args(c);
  const double theta2 = c->phys.thetamaxsqd;
  if (N > 1)
    launch_refit<false>(c, na, theta2);
  else
    k_leaves<<<1, BS, 0, s>>>(N, c->pf[F_X], c->pf[F_Y], c->pf[F_Z], c->pf[F_M], c->pf[F_H],
                              theta2, na, c->parent, c->gstart, c->visit);
  GDF_HIP(c, hipGetLastError());
  GDF_TRY(group_mac(c, nullptr));
  GDF_TRY(integ_pack_posm(c));
  GDF_HIP(c, hipStreamSynchronize(s));
  c->tree_valid = true;
  sph_drop_lists(c);
  return GDF_OK;
}

int group_list(gdf_ctx* c, const int* status, int* list, int* ncand, int* gnc, int* gnn,
               int* zero, int nzero) {
  const int ng = c->ngroups;
  hipStream_t s = c->stream;
  unsigned char* flags = reinterpret_cast<unsigned char*>(c->visit);
  constexpr int gpb = BS/kWave;   // groups per block
  k_group_flags<<<(ng + gpb - 1)/gpb, BS, 0, s>>>(ng, c->grp_first, c->grp_count, status, flags,
                                                  ncand, gnc, gnn, zero, nzero);
  k_compact_flags<<<(ng + 16*kWave - 1)/(16*kWave), kWave, 0, s>>>(
      ng, reinterpret_cast<const uint4*>(flags), list, c->Ncap);
  GDF_HIP(c, hipGetLastError());
  return GDF_OK;
}

int tree_refit_h(gdf_ctx* c) {
  const int N = c->N;
  hipStream_t s = c->stream;
  NodeArgs na = node_args(c);
  const double theta2 = c->phys.thetamaxsqd;
  if (N > 1)
    launch_refit<true>(c, na, theta2);
  else
    k_hleaves<<<1, BS, 0, s>>>(N, c->pf[F_H], theta2, na);
  GDF_HIP(c, hipGetLastError());
  return GDF_OK;
}

}  // namespace gdf
