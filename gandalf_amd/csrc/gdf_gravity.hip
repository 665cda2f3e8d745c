// Tree-gravity walk with per-wavefront interaction lists.
//
// Replaces the gravity half of GradhSphTree::UpdateAllSphForces
// (src/GradhSph/GradhSphTree.cpp:444-657): the walk of Tree::ComputeGravityInteractionAndGhostList
// (src/Tree/Tree.cpp:628-735), the kernel-softened neighbour gravity of
// GradhSph::ComputeSphHydroGravForces (src/GradhSph/GradhSph.cpp:555-565), the direct sum of
// GradhSphBase::ComputeDirectGravForces (:657-690) and the quadrupole cell terms of
// ComputeQuadropole (src/Headers/NeighbourSearch.h:423-449).
//
// One workgroup of W wavefronts per walk group, which share its node stack: a round tests up to 64
// nodes a wavefront.  Acceptance per node, with the group's bounding box G:
//   * kernel-range test (as the reference's neighbour-cell test, Tree.cpp:662-663): if the
//     minimum box-box distance is below k*max(hmax_G, hmax_cell) (with a 1e-4 relative slack
//     on the squared distance) the node is resolved to particles (bucket of <= Nleafmax
//     particles) or opened;
//   * geometric MAC (Tree.h:413-432) evaluated from the nearest point of G: accept the
//     multipole iff dist(G, centre_cell)^2 >= cdistsqd = max(rmax^2, hmax^2)/theta^2, a
//     conservative form of the reference's centre-to-centre test; the gadget2 and eigenmac
//     criteria then open more cells, from the same distance (mac_opens);
//   * otherwise open, or send the bucket's particles to the direct list.
// As in the reference, the kernel-softened gravity of the scatter-gather neighbours is summed by
// the hydro pass (GradhSph::ComputeSphHydroGravForces); the walk adds the direct 1/r^2 terms of
// every other particle and the multipole terms, masking the neighbour pairs with the same range
// test.  Without a hydro pass the walk evaluates the softened pairs itself.  Accepted cells and
// direct particles are staged 64 at a time in LDS, a batch a wavefront, and every lane (one target
// particle) sweeps the batch; the FP32 path sums each batch in registers and carries
// Kahan-compensated totals across batches.  The wavefronts' sums are added in order at the end.
//
// Bound by latency where the groups do not fill the device (each round and each batch waits for
// its scattered node, cell or particle loads), and by vector issue beside the hydro pass where they
// do.  20011 particles, FP64: 98 us with four wavefronts a group against 295 with one and the cell
// term's products written out; a million, FP64, beside the hydro pass: 4.4 against 5.5 ms.  Groups
// cost unequally, so they are fetched one by one (dealt out beforehand they took 3.4 ms instead of
// 2.65, FP32), from counters a line apart (on one line: 560 us at 262144 particles instead of 455).
#include <hip/hip_runtime.h>

#include <cstdlib>

#include "gdf_internal.h"
#include "gdf_device.h"
#include "gdf_filter.h"

namespace gdf {
namespace {

// Wavefronts that share a walk group, and the group's ring buffers (powers of two): a round adds
// at most 64 W cells or 64 W buckets to what is left of the last one, less than 64 W of either
template <int W> struct GravRings {
  static constexpr int cells = 2*kWave*W;
  static constexpr int parts = W == 1 ? 1024 : 512*W;
  static constexpr int wide = 4096;      // stack entries beyond which a round takes 64 nodes
};

static_assert(kGravQueue + (kXcds - 1)*kQueueStride < 16 + kGravZero, "range counters are cleared");

struct GravArgs {
  int N, ngroups, nleaf;
  const int* grp_node; const int* grp_first; const int* grp_count;
  const int4* lnk;
  const double4* geo_c; const double4* geo_h; const double* mp;
  const double4* posm; const double4* grec;     // grec: (h, zeta, hfactor, 0)
  double* atx; double* aty; double* atz; double* gpot;
  int* stacks; int* queue; int* flags; long long* icount;
  const int* glist; int ncap;   // groups to walk (count at glist[ncap]); NULL = all groups
  int32_t* gnc; int32_t* gnn;
  const int* act;         // block timesteps: only active targets (NULL = all)
  const int* grp_root;    // serving batches: walk from the group's segment subtree (NULL = root)
  const double* gmac;     // per group: factor of the gadget2 / eigenmac criterion
  // non-NULL: the walk runs beside the hydro pass and writes its own sums here (acceleration,
  // potential, self term) instead of adding to the hydro pass's atx/gpot
  double* gwx; double* gwy; double* gwz; double* gwp; double* gwp0;
  PhysParams p;
};

// Unified FP64 pair term for walks that also own the neighbour pairs (no hydro pass): the
// kernel-softened form of GradhSph.cpp:555-565 inside either smoothing range, the direct form
// of GradhSphBase::ComputeDirectGravForces (:657-690) outside
__device__ __forceinline__ void pair_fp64(const KernelDesc& k, double krsqd, double dx, double dy,
                                          double dz, double mj, double hi, double hj, double zi,
                                          double zj, double hfi, double hfj, double& ax,
                                          double& ay, double& az, double& pot) {
  const double d2 = dx*dx + dy*dy + dz*dz;
  if (d2 < krsqd*hi*hi || d2 < krsqd*hj*hj) {
    const double invh_i = 1/hi, invh_j = 1/hj;
    const double drmag = sqrt(d2 + 1.0e-20);
    const double inv = 1.0/drmag;
    dx *= inv; dy *= inv; dz *= inv;
    const double si = drmag*invh_i, sj = drmag*invh_j;
    const double wkerni = hfi*kw1<double>(k, si);
    const double wkernj = hfj*kw1<double>(k, sj);
    const double paux = 0.5*(invh_i*invh_i*kwgrav<double>(k, si) + zi*wkerni +
                             invh_j*invh_j*kwgrav<double>(k, sj) + zj*wkernj);
    ax += mj*dx*paux; ay += mj*dy*paux; az += mj*dz*paux;
    pot += 0.5*mj*(invh_i*kwpot<double>(k, si) + invh_j*kwpot<double>(k, sj));
  } else {
    const double inv = rsq_d(d2 + 1.0e-20);
    const double inv3 = inv*inv*inv;
    ax += mj*dx*inv3; ay += mj*dy*inv3; az += mj*dz*inv3;
    pot += mj*inv;
  }
}

__device__ __forceinline__ void pair_fp32(const KernelDesc& k, float d2, bool soft, float dx,
                                          float dy, float dz, float mj, float hi, float hj,
                                          float zi, float zj, float hfi, float hfj, float& ax,
                                          float& ay, float& az, float& pot) {
  if (soft) {
    const float invh_i = rcp_f(hi), invh_j = rcp_f(hj);
    const float drmag = sqrt_f(d2 + 1.0e-20f);
    const float inv = rcp_f(drmag);
    dx *= inv; dy *= inv; dz *= inv;
    const float si = drmag*invh_i, sj = drmag*invh_j;
    const float wkerni = hfi*kw1<float>(k, si);
    const float wkernj = hfj*kw1<float>(k, sj);
    const float paux = 0.5f*(invh_i*invh_i*kwgrav<float>(k, si) + zi*wkerni +
                             invh_j*invh_j*kwgrav<float>(k, sj) + zj*wkernj);
    ax += mj*dx*paux; ay += mj*dy*paux; az += mj*dz*paux;
    pot += 0.5f*mj*(invh_i*kwpot<float>(k, si) + invh_j*kwpot<float>(k, sj));
  } else {
    const float inv = rsq_f(d2 + 1.0e-20f);
    const float inv3 = inv*inv*inv;
    ax += mj*dx*inv3; ay += mj*dy*inv3; az += mj*dz*inv3;
    pot += mj*inv;
  }
}

// quadrupole cell term with dr = rp - com (NeighbourSearch.h:423-449), q = (xx, xy, yy, xz, yz,
// zz): Q dr once for the field and the scalar dr Q dr; 1/|dr| from the reciprocal square root
// instead of a division and a square root
template <typename T>
__device__ __forceinline__ void quad_term(T dx, T dy, T dz, T mc, const T* q, T& ax, T& ay,
                                          T& az, T& pot, T soft2 = T(1.0e-20)) {
  const T drsqd = dx*dx + dy*dy + dz*dz + soft2;
  T invdrmag;
  if (sizeof(T) == 4) invdrmag = (T) rsq_f((float) drsqd);
  else invdrmag = (T) rsq_d((double) drsqd);
  const T invdrsqd = invdrmag*invdrmag;
  const T invdr5 = invdrsqd*invdrsqd*invdrmag;
  const T qx = q[0]*dx + q[1]*dy + q[3]*dz;
  const T qy = q[1]*dx + q[2]*dy + q[4]*dz;
  const T qz = q[3]*dx + q[4]*dy + q[5]*dz;
  const T qs5 = (qx*dx + qy*dy + qz*dz)*invdr5;
  const T m1 = mc*invdrmag;
  const T c = (m1 + T(2.5)*qs5)*invdrsqd;
  ax += qx*invdr5 - c*dx;
  ay += qy*invdr5 - c*dy;
  az += qz*invdr5 - c*dz;
  pot += m1 + T(0.5)*qs5;
}

// Tree::open_cell_for_gravity (Tree.h:413-432) past its geometric test, for a cell at squared
// distance d2 from the walk group's box: gadget2 opens a cell whose m rmax^2 / d^4 exceeds
// macerror times the group's smallest |atree| (gfac); eigenmac one nearer than
// (0.5 lambda / macerror)^(2/3) (KDTree.cpp:1058-1079, lambda = 2 sqrt(-p/3) bounding the
// quadrupole's largest eigenvalue) times the group's largest gpot^(-2/3) (gfac)
__device__ __forceinline__ bool mac_opens(const PhysParams& p, const double4& nh, const double* mp,
                                          double d2, double gfac) {
#pragma clang fp contract(off)
  if (p.gravity_mac == GDF_MAC_GADGET2) {
    const double rmax = sqrt(nh.x*nh.x + nh.y*nh.y + nh.z*nh.z);
    return d2*d2*gfac*p.macerror < rmax*rmax*mp[3];
  }
  const double* q = mp + 4;
  const double pq = q[0]*q[2] - (q[0] + q[2])*(q[0] + q[2]) - q[1]*q[1] - q[3]*q[3] - q[4]*q[4];
  const double lambda = pq >= 0.0 ? 0.0 : 2.0*sqrt(-pq/3.0);
  const double mac = pow(0.5*lambda/p.macerror, 0.66666666666666);
  return d2 < mac*gfac;
}

// FastMultipoleForces::AddMonopoleContribution / AddQuadrupoleContribution
// (NeighbourSearch.h:564-597, 675-723) with the second-order terms off: one accepted cell's
// potential, acceleration and tidal tensor at the walk group's expansion point, added to
// f = (pot, ax, ay, az, txx, txy, tyy, txz, tyz, tzz).  dr = cell - expansion point; the
// reference's dphi takes the same increments as its ac, so one vector serves both.
__device__ __forceinline__ void fast_add(double* f, double dx, double dy, double dz, double mc,
                                         const double* q, bool quad) {
  {
    const double invdrmag = sqrt(1.0/(dx*dx + dy*dy + dz*dz));
    const double invdrsqd = invdrmag*invdrmag;
    const double mc3 = mc*invdrsqd*invdrmag;
    f[0] += mc*invdrmag;
    f[1] += mc3*dx; f[2] += mc3*dy; f[3] += mc3*dz;
    f[4] += mc3*(3.0*dx*dx*invdrsqd - 1.0);
    f[5] += mc3*(3.0*dx*dy*invdrsqd);
    f[6] += mc3*(3.0*dy*dy*invdrsqd - 1.0);
    f[7] += mc3*(3.0*dz*dx*invdrsqd);
    f[8] += mc3*(3.0*dz*dy*invdrsqd);
    f[9] += mc3*(3.0*dz*dz*invdrsqd - 1.0);
  }
  if (!quad) return;
  // the quadrupole part is written with d = expansion point - cell
  const double ex = -dx, ey = -dy, ez = -dz;
  const double invdrsqd = 1.0/(ex*ex + ey*ey + ez*ez + 1.0e-20);
  const double invdrmag = sqrt(invdrsqd);
  const double invdr5 = invdrsqd*invdrsqd*invdrmag;
  const double qzz = -(q[0] + q[2]);
  const double qscalar = q[0]*ex*ex + q[2]*ey*ey + qzz*ez*ez +
                         2.0*(q[1]*ex*ey + q[3]*ex*ez + q[4]*ey*ez);
  const double qfactor = 2.5*qscalar*invdr5*invdrsqd;
  double qx = (q[0]*ex + q[1]*ey + q[3]*ez)*invdr5;
  double qy = (q[1]*ex + q[2]*ey + q[4]*ez)*invdr5;
  double qz = (q[3]*ex + q[4]*ey + qzz*ez)*invdr5;
  f[0] += 0.5*qscalar*invdr5;
  f[1] += qx - qfactor*ex; f[2] += qy - qfactor*ey; f[3] += qz - qfactor*ez;
  const double s5 = 5.0*invdrsqd;
  qx *= s5; qy *= s5; qz *= s5;
  f[4] += qfactor*(7.0*ex*ex*invdrsqd - 1.0) - (2.0*qx*ex - q[0]*invdr5);
  f[5] += qfactor*(7.0*ex*ey*invdrsqd) - (qx*ey + qy*ex - q[1]*invdr5);
  f[6] += qfactor*(7.0*ey*ey*invdrsqd - 1.0) - (2.0*qy*ey - q[2]*invdr5);
  f[7] += qfactor*(7.0*ex*ez*invdrsqd) - (qx*ez + qz*ex - q[3]*invdr5);
  f[8] += qfactor*(7.0*ey*ez*invdrsqd) - (qy*ez + qz*ey - q[4]*invdr5);
  f[9] += qfactor*(7.0*ez*ez*invdrsqd - 1.0) - (2.0*qz*ez - qzz*invdr5);
}

// A lane's share of a batch of nb, U terms at a time.  (With one target a lane the terms' LDS
// addresses are constants apart: kept by itself, 6 % of a million particles' walk.)
template <int U, class F>
__device__ __forceinline__ void over_batch(const TargetLanes& tl, int nb, F term) {
  if (tl.copies == 1) {
    #pragma unroll U
    for (int q = 0; q < nb; q++) term(q);
  } else {
    const int trips = (nb + tl.copies - 1)/tl.copies;
    #pragma unroll 2
    for (int k = 0; k < trips; k++) term(k*tl.copies + tl.copy);
  }
}

// SOFT: the walk also evaluates the kernel-softened neighbour pairs (no hydro pass ran).
// Otherwise the hydro pass has already written the softened gravity of every scatter-gather
// pair into atree/gpot (GradhSph::ComputeSphHydroGravForces), the walk masks exactly those pairs
// (same squared distance, same range test, so each pair lands in one of the two sums) and adds
// the direct and multipole terms.  PLUMMER (pure N-body stars): every particle pair and every
// multipole term is softened with the Plummer length eps, the star itself is skipped and
// there is no self potential.  EWALD (periodic box with self-gravity): every particle of the
// walk's buckets (the hydro pass's neighbours and the target itself included) and every accepted
// cell adds its periodic correction at its separation, as GradhSphTree::UpdateAllSphForces does
// for all its neighbours and cells (GradhSphTree.cpp:558-578).  FAST (multipole fast_monopole or
// fast_quadrupole, gas walks): the accepted cells are summed once per group into the Taylor
// coefficients about the group's centre of mass (each lane takes the cells of its batch slot,
// the lanes' sums are reduced at the end of the walk) and every target applies the first-order
// series (ComputeFastMonopoleForces / ComputeFastQuadrupoleForces, NeighbourSearch.h:769-830).
// A cell is then accepted only if its centre of mass also lies beyond the group's extent about
// that point divided by theta, so that the series converges for every target.  multipole
// monopole: the cells' moments are staged as zeros (the quadrupole term reduces to
// ComputeCellMonopoleForces, NeighbourSearch.h:350-377).
template <bool MIXED, bool SOFT, bool PLUMMER, bool EWALD = false, bool FAST = false, int W = 4>
__global__ __launch_bounds__(64*W, EWALD || FAST || (SOFT && !PLUMMER) ? 2 : 3) void k_gravity(GravArgs a) {
  typedef GravRings<W> R;
  __shared__ int pbuf[R::parts];
  __shared__ int cbuf[R::cells];
  __shared__ int sidx[W][kWave];
  // a wavefront's staged batch.  FP64: particles (x, y), (z, m), r2, (h, zeta), (hfactor, -) or
  // cells (com x, y), (com z, m), (q0, q1), (q2, q3), (q4, q5).  FP32: two float4 records and a
  // float2: particles (dx, dy, dz, m), (h, zeta, hfactor, -), (r2, -); cells (dx, dy, dz, m),
  // (q0, q1, q2, q3), (q4, q5).  Each is read back with broadcast LDS loads.
  __shared__ __align__(16) double stage[W][(MIXED ? 5 : 10)*kWave];
  __shared__ int lstk[kLdsStack];    // node stack; deeper entries go to the global region
  __shared__ int count[W][3];        // a round's opened nodes, cells and particles
  const int lane = threadIdx.x & (kWave - 1), wv = W == 1 ? 0 : (int) threadIdx.x/kWave;
  double2 (*sd)[kWave] = reinterpret_cast<double2 (*)[kWave]>(stage[wv]);
  double* sr = stage[wv] + 8*kWave;
  float4* s4a = reinterpret_cast<float4*>(stage[wv]);
  float4* s4b = s4a + kWave;
  float2* s2 = reinterpret_cast<float2*>(s4b + kWave);
  int* sj = sidx[wv];
  int* stk = a.stacks + (size_t) blockIdx.x*kStackCap;
  const int N = a.N;
  const KernelDesc& K = a.p.kern;
  const double kr = K.range, krsqd = K.rangesqd;
  __shared__ int next;
  const int nq = a.glist ? a.glist[a.ncap] : a.ngroups;
  int range = blockIdx.x % kXcds;
  for (bool once = nq <= (int) gridDim.x; ; ) {
    if (once) {
      if (range < 0 || (int) blockIdx.x >= nq) break;
      range = -1;
    }
    // one lane alone fetches: in a divergent branch every active lane's part is an atomic
    else if (threadIdx.x == 0) next = group_fetch(a.queue, nq, range);
    __syncthreads();
    const int k = once ? (int) blockIdx.x : __builtin_amdgcn_readfirstlane(next);
    __syncthreads();
    if (k >= nq) break;
    const int g = a.glist ? a.glist[k] : k;
    const int G = a.grp_node[g], gfirst = a.grp_first[g], gcnt = a.grp_count[g];
    const unsigned long long on = __ballot(lane < gcnt && (!a.act || a.act[gfirst + lane]));
    const int nact = __popcll(on);
    if (nact == 0) {                 // no active target in this group
      if (threadIdx.x == 0) { a.gnc[g] = 0; a.gnn[g] = 0; }
      continue;
    }
    const TargetLanes tl(on);
    const bool has = tl.has;
    const int i = gfirst + tl.member;
    const double4 gc = a.geo_c[G], gh = a.geo_h[G];
    const double hmaxG = gc.w;
    // fast multipoles: expansion point (group centre of mass, relative to the group centre), the
    // squared distance beyond which a cell's series converges for the whole group, and this
    // lane's share of the coefficients
    double rcx = 0.0, rcy = 0.0, rcz = 0.0, rg2t = 0.0;
    double fc[10];
    if (FAST) {
#pragma clang fp contract(off)
      const double* mG = a.mp + kMom*(size_t) G;
      rcx = mG[0] - gc.x; rcy = mG[1] - gc.y; rcz = mG[2] - gc.z;
      const double ex = fabs(rcx) + gh.x, ey = fabs(rcy) + gh.y, ez = fabs(rcz) + gh.z;
      rg2t = (ex*ex + ey*ey + ez*ez)/a.p.thetamaxsqd;
      for (int k = 0; k < 10; k++) fc[k] = 0.0;
    }
    const bool mono = !PLUMMER && a.p.multipole == GDF_MULTIPOLE_MONOPOLE;
    const bool gmac = !PLUMMER && a.p.gravity_mac != GDF_MAC_GEOMETRIC;
    const double gfac = gmac ? a.gmac[g] : 0.0;
    double4 me = make_double4(0, 0, 0, 0), mr = make_double4(1, 0, 0, 0);
    if (has) { me = a.posm[i]; mr = a.grec[i]; }
    const double r2i = range2_rn(krsqd, mr.x);
    const float r2if = (float) r2i;
    double ax = 0.0, ay = 0.0, az = 0.0, pot = 0.0;
    KahanF fx, fy, fz, fp;
    const double eps2 = a.p.eps2;
    const float eps2f = (float) eps2;
    // target position relative to the group centre (cell-relative frame of the FP32 path)
    const float rxi = (float) (me.x - gc.x), ryi = (float) (me.y - gc.y), rzi = (float) (me.z - gc.z);

    // a batch of nb accepted cells from ring position c0.  The copies' last trip goes past the batch:
    // the slots there hold its last cell again without mass and moments.  (A fixed place can be a
    // target's, where the term overflows in FP32 and is 0 times infinity: massless cells one code unit
    // from the centre left NaN in the forces of lattices of unit spacing.)
    auto eval_cells = [&](int c0, int nb) {
      const bool fill = lane >= nb;
      const int c = cbuf[(c0 + min(lane, nb - 1)) & (R::cells - 1)];
      const double* m = a.mp + kMom*(size_t) c;
      double cx = m[0], cy = m[1], cz = m[2];
      const double mc = fill ? 0.0 : m[3];
      if (FAST && !fill) {
#pragma clang fp contract(off)
        // the cell relative to the expansion point, with the node test's replica
        double dx = cx - gc.x, dy = cy - gc.y, dz = cz - gc.z;
        nearest_image<double>(a.p, dx, dy, dz);
        fast_add(fc, dx - rcx, dy - rcy, dz - rcz, mc, m + 4,
                 a.p.multipole == GDF_MULTIPOLE_FAST_QUADRUPOLE);
      }
      if (a.p.periodic) {
        // nearest periodic replica of the cell relative to the group centre
        double dx = cx - gc.x, dy = cy - gc.y, dz = cz - gc.z;
        nearest_image<double>(a.p, dx, dy, dz);
        cx = gc.x + dx; cy = gc.y + dy; cz = gc.z + dz;
      }
      const double qs = mono || fill ? 0.0 : 1.0;      // monopole: no quadrupole moments
      const double q0 = qs*m[4], q2 = qs*m[6];
      if (MIXED) {
        s4a[lane] = make_float4((float) (cx - gc.x), (float) (cy - gc.y),
                                (float) (cz - gc.z), (float) mc);
        s4b[lane] = make_float4((float) q0, (float) (qs*m[5]), (float) q2, (float) (qs*m[7]));
        s2[lane] = make_float2((float) (qs*m[8]), -((float) q0 + (float) q2));
      } else {
        sd[0][lane] = make_double2(cx, cy); sd[1][lane] = make_double2(cz, mc);
        sd[2][lane] = make_double2(q0, qs*m[5]); sd[3][lane] = make_double2(q2, qs*m[7]);
        sd[4][lane] = make_double2(qs*m[8], -(q0 + q2));
      }
      wave_lds_order();
      // fast multipoles leave only the periodic corrections to the per-target sweep
      if (has && (!FAST || EWALD)) {
        if (MIXED) {
          float bx = 0.f, by = 0.f, bz = 0.f, bp = 0.f;
          auto term = [&](int q) {
            const float4 c = s4a[q], qa = s4b[q];
            const float2 qb = s2[q];
            const float qq[6] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y};
            if (!FAST)
              quad_term<float>(rxi - c.x, ryi - c.y, rzi - c.z, c.w, qq, bx, by, bz, bp,
                               PLUMMER ? eps2f : 1.0e-20f);
            if (EWALD) ewald_corr<float>(a.p, c.x - rxi, c.y - ryi, c.z - rzi, c.w, bx, by, bz,
                                         bp);
          };
          over_batch<4>(tl, nb, term);
          fx.add(bx); fy.add(by); fz.add(bz); fp.add(bp);
        } else {
          auto term = [&](int q) {
            const double2 xy = sd[0][q], zm = sd[1][q], qa = sd[2][q], qb = sd[3][q], qc = sd[4][q];
            const double qq[6] = {qa.x, qa.y, qb.x, qb.y, qc.x, qc.y};
            if (!FAST)
              quad_term<double>(me.x - xy.x, me.y - xy.y, me.z - zm.x, zm.y, qq, ax, ay, az, pot,
                                PLUMMER ? eps2 : 1.0e-20);
            if (EWALD) ewald_corr<double>(a.p, xy.x - me.x, xy.y - me.y, zm.x - me.z, zm.y, ax,
                                          ay, az, pot);
          };
          over_batch<2>(tl, nb, term);
        }
      }
      wave_lds_order();
    };
    // a batch of nb direct particles from ring position p0, massless ones up to the copies' last
    auto eval_parts = [&](int p0, int nb) {
      if (lane >= nb) {
        sj[lane] = -1;
        if (MIXED) {
          s4a[lane] = make_float4(1.f, 0.f, 0.f, 0.f);
          s2[lane] = make_float2(0.f, 0.f);
          if (SOFT) s4b[lane] = make_float4(1.f, 0.f, 0.f, 0.f);
        } else {
          sd[0][lane] = make_double2(gc.x, gc.y); sd[1][lane] = make_double2(gc.z, 0.0);
          if (SOFT) { sd[2][lane] = make_double2(1.0, 0.0); sd[3][lane].x = 0.0; }
          sr[lane] = 0.0;
        }
      } else {
        const int j = pbuf[(p0 + lane) & (R::parts - 1)];
        const double4 pj = a.posm[j];
        const double4 rj = a.grec[j];
        sj[lane] = j;
        if (MIXED) {
          double dx = pj.x - gc.x, dy = pj.y - gc.y, dz = pj.z - gc.z;
          nearest_image<double>(a.p, dx, dy, dz);
          s4a[lane] = make_float4((float) dx, (float) dy, (float) dz, (float) pj.w);
          s2[lane] = make_float2((float) range2_rn(krsqd, rj.x), 0.f);
          if (SOFT) s4b[lane] = make_float4((float) rj.x, (float) rj.y, (float) rj.z, 0.f);
        } else {
          sd[0][lane] = make_double2(pj.x, pj.y); sd[1][lane] = make_double2(pj.z, pj.w);
          if (SOFT) { sd[2][lane] = make_double2(rj.x, rj.y); sd[3][lane].x = rj.z; }
          sr[lane] = range2_rn(krsqd, rj.x);
        }
      }
      wave_lds_order();
      if (has) {
        if (MIXED) {
          const float hi = (float) mr.x, zi = (float) mr.y, hfi = (float) mr.z;
          float bx = 0.f, by = 0.f, bz = 0.f, bp = 0.f;
          // unrolled so that several LDS reads are in flight (same summation order)
          auto term = [&](int q) {
            // every record is loaded whatever the pair's branch: no LDS read under a mask
            const float4 s = s4a[q];
            const float r2j = s2[q].x;
            const float dx = s.x - rxi, dy = s.y - ryi, dz = s.z - rzi;
            const float d2 = dot3_f(dx, dy, dz);
            const bool soft = (d2 < r2if) | (d2 < r2j);
            if (PLUMMER) {
              const float inv = rsq_f(d2 + eps2f);
              const float mj = sj[q] == i ? 0.f : s.w;
              const float minv3 = mj*inv*inv*inv;
              bx += minv3*dx; by += minv3*dy; bz += minv3*dz; bp += mj*inv;
            } else if (SOFT) {
              const float4 hq = s4b[q];
              pair_fp32(K, d2, soft, dx, dy, dz, s.w, hi, hq.x, zi, hq.y, hfi, hq.z, bx, by,
                        bz, bp);
            } else {
              const float inv = rsq_f(d2 + 1.0e-20f);
              const float mj = soft ? 0.f : s.w;
              const float minv3 = mj*inv*inv*inv;
              bx += minv3*dx; by += minv3*dy; bz += minv3*dz; bp += mj*inv;
            }
            if (EWALD) ewald_corr<float>(a.p, dx, dy, dz, s.w, bx, by, bz, bp);
          };
          over_batch<8>(tl, nb, term);
          fx.add(bx); fy.add(by); fz.add(bz); fp.add(bp);
        } else {
          auto term = [&](int q) {
            const double2 xy = sd[0][q], zm = sd[1][q];
            double dx = xy.x - me.x, dy = xy.y - me.y, dz = zm.x - me.z;
            nearest_image<double>(a.p, dx, dy, dz);
            if (PLUMMER) {
              const double inv = rsq_d(dot3_rn(dx, dy, dz) + eps2);
              const double mj = sj[q] == i ? 0.0 : zm.y;
              const double minv3 = mj*inv*inv*inv;
              ax += minv3*dx; ay += minv3*dy; az += minv3*dz; pot += mj*inv;
            } else if (SOFT) {
              const double2 hq = sd[2][q];
              pair_fp64(K, krsqd, dx, dy, dz, zm.y, mr.x, hq.x, mr.y, hq.y, mr.z, sd[3][q].x, ax,
                        ay, az, pot);
            } else {
              const double d2 = dot3_rn(dx, dy, dz);
              const bool soft = (d2 < r2i) | (d2 < sr[q]);
              const double inv = rsq_d(d2 + 1.0e-20);
              const double mj = soft ? 0.0 : zm.y;
              const double minv3 = mj*inv*inv*inv;
              ax += minv3*dx; ay += minv3*dy; az += minv3*dz; pot += mj*inv;
            }
            if (EWALD) ewald_corr<double>(a.p, dx, dy, dz, zm.y, ax, ay, az, pot);
          };
          over_batch<2>(tl, nb, term);
        }
      }
      wave_lds_order();
    };

    int sp = 1, phead = 0, ptail = 0, chead = 0, ctail = 0;
    bool overflow = false;
    // nodes a round may take: what the particle ring holds at the largest bucket
    const int most = min(kWave*W, (R::parts - kWave*W)/max(a.nleaf, 1));
    if (threadIdx.x == 0) lstk[0] = a.grp_root ? a.grp_root[g] : 0;  // the group's segment subtree
    __syncthreads();
    while (sp > 0) {
      const int b = min(sp, sp > R::wide ? min(most, kWave) : most);
      const int slot = wv*kWave + lane;
      int node = -1;
      if (slot < b) node = stack_get(lstk, stk, sp - 1 - slot);
      sp -= b;
      bool open = false, near = false, cell = false;
      int ef = 0, ec = 0, cl = 0, cr = 0;
      if (node >= 0) {
#pragma clang fp contract(off)
        // box, range and children in one round of loads
        const double4 nc = a.geo_c[node], nh = a.geo_h[node];
        NodeLinks nl;
        load_links(node, N, a.lnk, nl);
        double dx = nc.x - gc.x, dy = nc.y - gc.y, dz = nc.z - gc.z;
        nearest_image<double>(a.p, dx, dy, dz);
        const double gx = fmax(fabs(dx) - nh.x - gh.x, 0.0);
        const double gy = fmax(fabs(dy) - nh.y - gh.y, 0.0);
        const double gz = fmax(fabs(dz) - nh.z - gh.z, 0.0);
        const double dbox2 = gx*gx + gy*gy + gz*gz;
        const double hr = kr*fmax(hmaxG, nc.w);
        ef = nl.first; ec = nl.count;
        const bool bucket = ec <= a.nleaf || node >= N - 1;
        if (dbox2 < hr*hr*kGravNeibSlack) {
          if (bucket) near = true; else open = true;
        } else {
          const double ex = fmax(fabs(dx) - gh.x, 0.0);
          const double ey = fmax(fabs(dy) - gh.y, 0.0);
          const double ez = fmax(fabs(dz) - gh.z, 0.0);
          const double dmac2 = ex*ex + ey*ey + ez*ez;
          bool accept = dmac2 >= nh.w;
          if (gmac && accept) accept = !mac_opens(a.p, nh, a.mp + kMom*(size_t) node, dmac2, gfac);
          if (FAST && accept) {
            const double* mc = a.mp + kMom*(size_t) node;
            double cx = mc[0] - gc.x, cy = mc[1] - gc.y, cz = mc[2] - gc.z;
            nearest_image<double>(a.p, cx, cy, cz);
            cx -= rcx; cy -= rcy; cz -= rcz;
            accept = cx*cx + cy*cy + cz*cz >= rg2t;
          }
          if (accept) {
            if (ec == 1) near = true; else cell = true;
          } else {
            if (bucket) near = true; else open = true;
          }
        }
        if (open) { cl = nl.left; cr = nl.right; }
      }
      // places of the round's opened nodes, cells and particles, wavefront by wavefront
      const unsigned long long om = __ballot(open), cm = __ballot(cell);
      const int ecount = near ? ec : 0;
      const int incl = wave_incl_scan(ecount);
      int o0 = 0, c0 = ctail, p0 = ptail, nopen = __popcll(om);
      if (W == 1) {
        ctail += __popcll(cm);
        ptail += __shfl(incl, 63, 64);
      } else {
        if (lane == 63) { count[wv][0] = nopen; count[wv][1] = __popcll(cm); count[wv][2] = incl; }
        __syncthreads();
        nopen = 0;
        #pragma unroll
        for (int w = 0; w < W; w++) {
          if (w == wv) { o0 = nopen; c0 = ctail; p0 = ptail; }
          nopen += count[w][0]; ctail += count[w][1]; ptail += count[w][2];
        }
      }
      if (sp + 2*nopen > kLdsStack + kStackCap) { overflow = true; break; }
      if (open) {
        const int o = sp + 2*(o0 + lanes_below(om));
        stack_put(lstk, stk, o, cr);
        stack_put(lstk, stk, o + 1, cl);
      }
      sp += 2*nopen;
      if (sp > kLdsStack) __threadfence_block();   // entries in the global overflow region
      if (cell) cbuf[(c0 + lanes_below(cm)) & (R::cells - 1)] = node;
      for (int k = 0; k < ecount; k++) pbuf[(p0 + incl - ecount + k) & (R::parts - 1)] = ef + k;
      __syncthreads();
      // full batches, as many as the wavefronts share evenly; all that is left after the last
      // round
      const int cells = ctail - chead, parts = ptail - phead;
      const int jc = sp == 0 ? (cells + kWave - 1)/kWave : cells/kWave;
      int jobs = jc + (sp == 0 ? (parts + kWave - 1)/kWave : parts/kWave);
      if (sp > 0) jobs -= jobs % W;
      for (int j = wv; j < jobs; j += W) {
        if (j < jc) eval_cells(chead + kWave*j, min(cells - kWave*j, kWave));
        else eval_parts(phead + kWave*(j - jc), min(parts - kWave*(j - jc), kWave));
      }
      chead += min(cells, kWave*min(jobs, jc));
      phead += min(parts, kWave*max(jobs - jc, 0));
    }
    if (overflow) {
      if (threadIdx.x == 0) atomicOr(&a.flags[2], 1);
      if (W > 1) __syncthreads();
      continue;
    }
    if (MIXED) { ax = (double) fx.s; ay = (double) fy.s; az = (double) fz.s; pot = (double) fp.s; }
    ax = tl.over_copies(ax); ay = tl.over_copies(ay); az = tl.over_copies(az);
    pot = tl.over_copies(pot);
    if (FAST) {
      // the lanes' coefficient sums, reduced by a butterfly (every lane ends with the same sums)
      for (int k = 0; k < 10; k++) {
        double v = fc[k];
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        fc[k] = v;
      }
    }
    if (W > 1) {
      // the wavefronts' sums, added in order by the first
      double* red = &stage[0][0];
      __syncthreads();
      red[(4*wv + 0)*kWave + lane] = ax; red[(4*wv + 1)*kWave + lane] = ay;
      red[(4*wv + 2)*kWave + lane] = az; red[(4*wv + 3)*kWave + lane] = pot;
      double* redf = red + 4*kWave*W;
      if (FAST && lane < 10) {
        double v = 0.0;
        for (int k = 0; k < 10; k++) v = lane == k ? fc[k] : v;
        redf[10*wv + lane] = v;
      }
      __syncthreads();
      if (wv == 0) {
        for (int w = 1; w < W; w++) {
          ax += red[(4*w + 0)*kWave + lane]; ay += red[(4*w + 1)*kWave + lane];
          az += red[(4*w + 2)*kWave + lane]; pot += red[(4*w + 3)*kWave + lane];
          if (FAST) for (int k = 0; k < 10; k++) fc[k] += redf[10*w + k];
        }
      }
    }
    if (has && wv == 0 && tl.copy == 0) {
      if (FAST) {
        // ApplyForcesTaylor (NeighbourSearch.h:735-760), first order about the expansion point
        const double* mG = a.mp + kMom*(size_t) G;
        const double d0 = me.x - mG[0], d1 = me.y - mG[1], d2 = me.z - mG[2];
        ax += fc[1] + fc[4]*d0 + fc[5]*d1 + fc[7]*d2;
        ay += fc[2] + fc[5]*d0 + fc[6]*d1 + fc[8]*d2;
        az += fc[3] + fc[7]*d0 + fc[8]*d1 + fc[9]*d2;
        pot += fc[0] + fc[1]*d0 + fc[2]*d1 + fc[3]*d2;
      }
      // the self term (m/h) wpot(0) (GradhSphTree.cpp:512)
      const double pot0 = PLUMMER ? 0.0 : (me.w/mr.x)*kwpot<double>(K, 0.0);
      if (SOFT) {
        a.atx[i] = ax; a.aty[i] = ay; a.atz[i] = az;
        a.gpot[i] = pot0 + pot;
      } else if (a.gwx) {
        a.gwx[i] = ax; a.gwy[i] = ay; a.gwz[i] = az;
        a.gwp[i] = pot; a.gwp0[i] = pot0;
      } else {
        a.atx[i] += ax; a.aty[i] += ay; a.atz[i] += az;
        a.gpot[i] = pot0 + a.gpot[i] + pot;
      }
    }
    if (threadIdx.x == 0) {
      a.gnc[g] = ctail;
      a.gnn[g] = ptail;
      atomicAdd((unsigned long long*) &a.icount[2], (unsigned long long) ptail*nact);
      atomicAdd((unsigned long long*) &a.icount[3], (unsigned long long) ctail*(FAST ? 1 : nact));
    }
  }
}

struct NbDirectArgs {
  int N;
  const double* x; const double* y; const double* z;
  const double* vx; const double* vy; const double* vz;
  const double* m; const double* h;
  double* ax; double* ay; double* az; double* adx; double* ady; double* adz; double* gpot;
  KernelDesc kern;
  int add;          // add to a, adot and gpot (after the stars' gas terms) instead of writing
};

// Star-star direct sums.  SMOOTH = false: Nbody::CalculateDirectGravForces
// (src/Nbody/Nbody.cpp:233-293), point masses with jerk; SMOOTH = true:
// NbodyLeapfrogKDK::CalculateDirectSmoothedGravForces (src/Nbody/NbodyLeapfrogKDK.cpp:78-150),
// kernel softening over the mean smoothing length, whose (2/(h_i+h_j))^3 factor the reference
// forms in single precision (powf).
//
// A block of 256 threads takes T targets; the 256/T threads of a target take every (256/T)-th
// source of the tiles staged in LDS (the next tile is in flight meanwhile) and their sums are
// added in a fixed order.  Bound by FP64 issue, about 45 instructions a pair.  T small enough that
// the blocks fill the device: one thread a target put 6007 stars on 24 of the 256 CUs, and a
// division and a square root cost more than the rest of the pair.  6007 stars, softened: 99 us
// against 3690.
template <bool SMOOTH, int T>
__global__ __launch_bounds__(256) void k_nbody_direct(NbDirectArgs a) {
  constexpr int BT = 256, S = BT/T;
  __shared__ double2 sxy[BT], szm[BT], suv[BT], swh[BT];
  __shared__ double red[BT/kWave][7][T];
  const int tid = threadIdx.x, t = tid % T;
  const int i = blockIdx.x*T + t;
  const int ii = min(i, a.N - 1);
  const double xi = a.x[ii], yi = a.y[ii], zi = a.z[ii];
  const double vxi = a.vx[ii], vyi = a.vy[ii], vzi = a.vz[ii];
  const double hi = SMOOTH ? a.h[ii] : 1.0;
  const double hrange = 0.5*a.kern.range*(1.0 + 1.0e-12);
  double sum[7] = {0, 0, 0, 0, 0, 0, 0};      // a, adot, gpot
  double2 nxy, nzm, nuv, nwh;
  auto fetch = [&](int j0) {
    const int j = min(j0 + tid, a.N - 1);
    nxy = make_double2(a.x[j], a.y[j]);
    nzm = make_double2(a.z[j], a.m[j]);
    nuv = make_double2(a.vx[j], a.vy[j]);
    nwh = make_double2(a.vz[j], SMOOTH ? a.h[j] : 0.0);
  };
  fetch(0);
  for (int j0 = 0; j0 < a.N; j0 += BT) {
    sxy[tid] = nxy; szm[tid] = nzm; suv[tid] = nuv; swh[tid] = nwh;
    __syncthreads();
    if (j0 + BT < a.N) fetch(j0 + BT);
    const int nb = min(BT, a.N - j0);
    for (int q = tid/T; q < nb; q += S) {
      if (j0 + q == i) continue;
      const double2 xy = sxy[q], zm = szm[q], uv = suv[q], wh = swh[q];
      const double dx = xy.x - xi, dy = xy.y - yi, dz = zm.x - zi;
      const double dvx = uv.x - vxi, dvy = uv.y - vyi, dvz = wh.x - vzi;
      const double drsqd = dx*dx + dy*dy + dz*dz;
      const double mj = zm.y;
      // 1/|dr| from the estimate; coincident stars and separations at the ends of the exponent
      // range keep the division
      const bool easy = drsqd > (SMOOTH ? 1.0e-30 : 1.0e-280) && drsqd < 1.0e280;
      double invdrmag, drmag;
      if (easy) {
        const double y = rsq_d(drsqd);
        if (SMOOTH) {
          // drmag = sqrt(drsqd) + 1e-20 and its reciprocal: the shift is below 1e-5 of either
          drmag = fma(drsqd, y, 1.0e-20);
          const double e = 1.0e-20*y;
          invdrmag = fma(-e*(1.0 - e), y, y);
        } else {
          invdrmag = y;
          drmag = 0.0;
        }
      } else {
        drmag = sqrt(drsqd) + (SMOOTH ? 1.0e-20 : 0.0);
        invdrmag = 1.0/drmag;
      }
      const double inv2 = invdrmag*invdrmag;
      const double c = 3.0*(dvx*dx + dvy*dy + dvz*dz)*inv2;      // 3 drdt/|dr|
      double paux = mj*(inv2*invdrmag), p = mj*invdrmag, cw = 0.0;
      if (SMOOTH && drmag < hrange*(hi + wh.y)) {     // at or inside the kernel's range
        const double invhmean = 2.0/(hi + wh.y);
        const double s = drmag*invhmean;
        paux = mj*invhmean*invhmean*kwgrav<double>(a.kern, s)*invdrmag;
        p = mj*invhmean*kwpot<double>(a.kern, s);
        // the reference's single-precision powf(invhmean, 3): the correctly rounded cube
        // (exact in double before the one rounding to float), which is what glibc's powf
        // returns for all but ~0.07% of arguments (those differ by one float ulp)
        const float hmf = (float) invhmean;
        const double wmean = kw0<double>(a.kern, s)*
                             (double) (float) ((double) hmf*(double) hmf*(double) hmf);
        cw = 2.0*6.28318530717959*(1.0/3.0)*mj*c*wmean;
      }
      const double cj = cw - paux*c;
      sum[0] += paux*dx; sum[1] += paux*dy; sum[2] += paux*dz;
      sum[3] += paux*dvx + cj*dx; sum[4] += paux*dvy + cj*dy; sum[5] += paux*dvz + cj*dz;
      sum[6] += p;
    }
    __syncthreads();
  }
  for (int k = 0; k < 7; k++) {
    #pragma unroll
    for (int o = T; o < kWave; o *= 2) sum[k] += __shfl_xor(sum[k], o, kWave);
    if (tid % kWave < T) red[tid/kWave][k][t] = sum[k];
  }
  __syncthreads();
  if (tid >= T || i >= a.N) return;
  for (int k = 0; k < 7; k++)
    sum[k] = (red[0][k][t] + red[1][k][t]) + (red[2][k][t] + red[3][k][t]);
  double* out[7] = {a.ax, a.ay, a.az, a.adx, a.ady, a.adz, a.gpot};
  for (int k = 0; k < 7; k++) out[k][i] = a.add ? out[k][i] + sum[k] : sum[k];
}

// Four targets a block while eight leave CUs idle: 500 stars 7.1 against 8.6 us, 2000 19.4 against
// 22.7, 4000 50 against 53; then eight, which read half the source tiles: 6007 99 against 102 us,
// 16000 576 against 622.  (Sixteen: 68 us at 4000, 132 at 6007, 589 at 16000.)
void launch_nbody_direct(const NbDirectArgs& a, int smoothed, hipStream_t s) {
  if (a.N < 8*512) {
    const int nb = (a.N + 3)/4;
    if (smoothed) k_nbody_direct<true, 4><<<nb, 256, 0, s>>>(a);
    else k_nbody_direct<false, 4><<<nb, 256, 0, s>>>(a);
  } else {
    const int nb = (a.N + 7)/8;
    if (smoothed) k_nbody_direct<true, 8><<<nb, 256, 0, s>>>(a);
    else k_nbody_direct<false, 8><<<nb, 256, 0, s>>>(a);
  }
}

__global__ void k_pack_grav(int N, const double* __restrict__ h, const double* __restrict__ zeta,
                            const double* __restrict__ hf, double4* __restrict__ g) {
  const int i = blockIdx.x*256 + threadIdx.x;
  if (i < N) g[i] = make_double4(h[i], zeta[i], hf[i], 0.0);
}

__global__ void k_zero_ints(int* p) { p[threadIdx.x] = 0; }

// the walk's sums joined to the hydro pass's in the order of the single-stream update
// (atx += walk; gpot = self + gpot + walk), then a += atree (GradhSphTree.cpp:615-617)
struct JoinArgs {
  int N;
  const int* act;
  const double* gw[3]; const double* gwp; const double* gwp0;
  double* at[3]; double* gpot; double* a[3];
};
__global__ void k_grav_join(JoinArgs j) {
  const int i = blockIdx.x*256 + threadIdx.x;
  if (i >= j.N || (j.act && !j.act[i])) return;
  for (int k = 0; k < 3; k++) {
    const double t = j.at[k][i] + j.gw[k][i];
    j.at[k][i] = t;
    j.a[k][i] += t;
  }
  j.gpot[i] = j.gwp0[i] + j.gpot[i] + j.gwp[i];
}

}  // namespace

int nbody_direct(gdf_ctx* c, int smoothed) {
  const int N = c->N;
  if (N <= 0) return fail(c, GDF_ERR_INVALID, "no particles");
  NbDirectArgs a;
  a.N = N;
  a.x = c->pf[F_X]; a.y = c->pf[F_Y]; a.z = c->pf[F_Z];
  a.vx = c->pf[F_VX]; a.vy = c->pf[F_VY]; a.vz = c->pf[F_VZ];
  a.m = c->pf[F_M]; a.h = c->pf[F_H];
  a.ax = c->df[D_AX]; a.ay = c->df[D_AY]; a.az = c->df[D_AZ];
  a.adx = c->df[D_ADOTX]; a.ady = c->df[D_ADOTY]; a.adz = c->df[D_ADOTZ];
  a.gpot = c->df[D_GPOT];
  a.kern = c->phys.kern;
  a.add = 0;
  launch_nbody_direct(a, smoothed, c->stream);
  GDF_HIP(c, hipGetLastError());
  return GDF_OK;
}

int nbody_direct_stars(gdf_ctx* c, int smoothed) {
  const int N = c->Nstar;
  if (N <= 0) return GDF_OK;
  NbDirectArgs a;
  a.N = N;
  a.x = c->sv[S_X]; a.y = c->sv[S_Y]; a.z = c->sv[S_Z];
  a.vx = c->sv[S_VX]; a.vy = c->sv[S_VY]; a.vz = c->sv[S_VZ];
  a.m = c->sv[S_M]; a.h = c->sv[S_H];
  a.ax = c->sv[S_AX]; a.ay = c->sv[S_AY]; a.az = c->sv[S_AZ];
  a.adx = c->sv[S_ADX]; a.ady = c->sv[S_ADY]; a.adz = c->sv[S_ADZ];
  a.gpot = c->sv[S_GPOT];
  a.kern = c->phys.kern;
  a.add = 1;
  launch_nbody_direct(a, smoothed, c->stream);
  GDF_HIP(c, hipGetLastError());
  return GDF_OK;
}

namespace {

// Wavefronts that share a walk group.  A group's walk is a chain of dependent loads, so while one
// wavefront a group leaves SIMDs idle more of them finish sooner; with the device full they only
// add barriers and partly filled rounds.  Walk (us) with 1, 2 and 4 wavefronts: 512 groups (20011
// particles, FP64) 230 147 100, 1024 (FP64) 253 183 200, 2048 (FP32) 320 283 300, 2700 of stars
// 397 390 450; the whole force pass (ms): 4096 groups 2.16 2.15 2.26, 16384 9.38 9.57 9.99 (FP32),
// 11.6 12.1 12.3 (FP64).  A serving batch keeps to two: a request's sums must not depend on what
// else is resident.
int grav_waves(const gdf_ctx* c) {
  if (c->nseg > 0) return 2;
  return c->ngroups <= 1024 ? 4 : c->ngroups <= 8192 ? 2 : 1;
}

template <bool MIXED, bool SOFT, bool PLUMMER, bool EWALD, bool FAST, int W>
void launch_walk_w(const GravArgs& a, bool beside, hipStream_t s) {
  // beside the hydro pass half the persistent wavefronts of a lone walk: at the full count they
  // fill the CUs' LDS and the hydro pass waits for the walk to drain
  const int most = (beside ? kGravSlots/2 : kGravSlots)/(W == 4 ? 2 : 1);
  const int grid = std::min(a.ngroups, most);
  k_gravity<MIXED, SOFT, PLUMMER, EWALD, FAST, W><<<grid, kWave*W, 0, s>>>(a);
}

// The walk's variant: stars, gas beside or after a hydro pass, or gas alone (SOFT); the options
// off the main path (periodic corrections, fast multipoles, gas alone) take two wavefronts a group
template <bool MIXED, bool SOFT>
void launch_gas(const GravArgs& a, bool ewald, bool beside, int waves, hipStream_t s) {
  const bool fast = a.p.multipole >= GDF_MULTIPOLE_FAST_MONOPOLE;
  if (ewald) {
    if (fast) launch_walk_w<MIXED, SOFT, false, true, true, 2>(a, beside, s);
    else launch_walk_w<MIXED, SOFT, false, true, false, 2>(a, beside, s);
  } else if (fast) {
    launch_walk_w<MIXED, SOFT, false, false, true, 2>(a, beside, s);
  } else if (SOFT || waves == 2) {
    launch_walk_w<MIXED, SOFT, false, false, false, 2>(a, beside, s);
  } else if (waves == 4) {
    launch_walk_w<MIXED, SOFT, false, false, false, SOFT ? 2 : 4>(a, beside, s);
  } else {
    launch_walk_w<MIXED, SOFT, false, false, false, SOFT ? 2 : 1>(a, beside, s);
  }
}

template <bool MIXED>
void launch_grav(const gdf_ctx* c, const GravArgs& a, bool beside, hipStream_t s) {
  const int waves = grav_waves(c);
  if (c->phys.nbody) {
    if (waves == 4) launch_walk_w<MIXED, true, true, false, false, 4>(a, beside, s);
    else if (waves == 2) launch_walk_w<MIXED, true, true, false, false, 2>(a, beside, s);
    else launch_walk_w<MIXED, true, true, false, false, 1>(a, beside, s);
  } else if (c->phys.hydro_forces) {
    launch_gas<MIXED, false>(a, c->phys.ewald, beside, waves, s);
  } else {
    launch_gas<MIXED, true>(a, c->phys.ewald, beside, waves, s);
  }
}

GravArgs grav_args(gdf_ctx* c) {
  GravArgs a;
  a.N = c->N; a.ngroups = c->ngroups; a.nleaf = c->phys.nleaf;
  a.grp_node = c->grp_node; a.grp_first = c->grp_first; a.grp_count = c->grp_count;
  a.lnk = c->lnk;
  a.geo_c = c->geo_c; a.geo_h = c->geo_h; a.mp = c->mp;
  a.posm = c->posm; a.grec = c->grec;
  a.atx = c->df[D_ATX]; a.aty = c->df[D_ATY]; a.atz = c->df[D_ATZ]; a.gpot = c->df[D_GPOT];
  a.stacks = c->stacks; a.flags = c->counters + 16; a.queue = c->counters + kGravQueue;
  a.icount = c->icount; a.gnc = c->grav_nc; a.gnn = c->grav_nn;
  a.act = c->nlevels > 1 ? c->pi[I_ACT] : nullptr;
  a.grp_root = c->nseg > 0 ? c->grp_root : nullptr;
  a.gmac = c->grp_gmac;
  a.gwx = a.gwy = a.gwz = a.gwp = a.gwp0 = nullptr;
  a.glist = nullptr; a.ncap = c->Ncap;
  a.p = c->phys;
  return a;
}

// in a block step, the compacted list of groups with active particles (built on the main stream)
// zero[0, nzero): the flags of the walk, cleared with the list (or by the
// caller when there is no list: returns false)
bool grav_group_list(gdf_ctx* c, GravArgs& a, int* zero, int nzero, int& rc) {
  rc = GDF_OK;
  if (!a.act || !c->glist) return false;
  int* gl = c->glist + 2*((size_t) c->Ncap + 1);
  rc = group_list(c, a.act, gl, nullptr, c->grav_nc, c->grav_nn, zero, nzero);
  a.glist = gl;
  return true;
}

}  // namespace

int gravity_launch(gdf_ctx* c) {
  if (!c->tree_valid) return fail(c, GDF_ERR_INVALID, "gravity pass before tree build");
  if (!c->stacks2 || !c->phys.hydro_forces || c->phys.nbody)
    return fail(c, GDF_ERR_INVALID, "gravity walk beside the hydro pass needs hydro + self-gravity");
  const int N = c->N;
  // on the second stream beside the scatter-gather walk and the hydro pass: measured faster
  // than running them in turn, both at 1M active particles and in sparse block steps
  hipStream_t s2 = c->stream2;
  GravArgs a = grav_args(c);
  int rc = GDF_OK;
  const bool listed = grav_group_list(c, a, c->counters + 16, kGravZero, rc);
  GDF_TRY(rc);
  GDF_HIP(c, hipEventRecord(c->ev_dens, c->stream));        // h, zeta, tree, posm are ready
  GDF_HIP(c, hipStreamWaitEvent(s2, c->ev_dens, 0));
  k_pack_grav<<<nblocks(N, 256), 256, 0, s2>>>(N, c->pf[F_H], c->df[D_ZETA], c->df[D_HFACTOR],
                                                 c->grec);
  a.stacks = c->stacks2;
  a.gwx = c->df[D_GWX]; a.gwy = c->df[D_GWY]; a.gwz = c->df[D_GWZ];
  a.gwp = c->df[D_GWP]; a.gwp0 = c->df[D_GWP0];
  if (!listed) {
    k_zero_ints<<<1, kGravZero, 0, s2>>>(c->counters + 16);
  }
  const int kt = ktime_begin(c, s2, 5);
  const bool mixed = c->cfg.precision == GDF_PREC_MIXED;
  if (mixed) launch_grav<true>(c, a, true, s2);
  else launch_grav<false>(c, a, true, s2);
  GDF_HIP(c, hipGetLastError());
  ktime_end(c, s2, kt);
  GDF_HIP(c, hipMemcpyAsync(c->h_counters + 16, c->counters + 16, sizeof(int)*8,
                            hipMemcpyDeviceToHost, s2));
  GDF_HIP(c, hipEventRecord(c->ev_grav, s2));
  return GDF_OK;
}

// Fault injection for the failure-path tests: with GDF_FAULT_HYDRO=1 in the environment the hydro
// pass beside the gravity walk reports a failure.
static bool hydro_fault_injected() {
  const char* e = std::getenv("GDF_FAULT_HYDRO");
  return e && e[0] == '1';
}

int gravity_beside_hydro(gdf_ctx* c) {
  int rc = hydro_fault_injected() ? fail(c, GDF_ERR_NOMEM, "injected failure of the hydro pass")
                                  : sph_build_sg(c);
  if (rc == GDF_OK) rc = sph_hydro(c, 1);
  if (rc != GDF_OK) (void) hipStreamSynchronize(c->stream2);
  return rc;
}

int gravity_join(gdf_ctx* c) {
  GDF_HIP(c, hipStreamWaitEvent(c->stream, c->ev_grav, 0));
  JoinArgs j;
  j.N = c->N; j.act = c->nlevels > 1 ? c->pi[I_ACT] : nullptr;
  for (int k = 0; k < 3; k++) {
    j.gw[k] = c->df[D_GWX + k]; j.at[k] = c->df[D_ATX + k]; j.a[k] = c->df[D_AX + k];
  }
  j.gwp = c->df[D_GWP]; j.gwp0 = c->df[D_GWP0]; j.gpot = c->df[D_GPOT];
  k_grav_join<<<nblocks(c->N, 256), 256, 0, c->stream>>>(j);
  GDF_HIP(c, hipGetLastError());
  GDF_HIP(c, hipEventSynchronize(c->ev_grav));
  if (c->h_counters[16 + 2]) return fail(c, GDF_ERR_CAPACITY, "tree walk stack overflow in gravity pass");
  return GDF_OK;
}

int gravity_walk(gdf_ctx* c) {
  const int N = c->N;
  hipStream_t s = c->stream;
  if (!c->tree_valid) return fail(c, GDF_ERR_INVALID, "gravity pass before tree build");
  k_pack_grav<<<nblocks(N, 256), 256, 0, s>>>(N, c->pf[F_H], c->df[D_ZETA], c->df[D_HFACTOR],
                                                c->grec);
  GravArgs a = grav_args(c);
  int rc = GDF_OK;
  if (!grav_group_list(c, a, c->counters + 16, kGravZero, rc)) {
    k_zero_ints<<<1, kGravZero, 0, s>>>(c->counters + 16);
  }
  GDF_TRY(rc);
  const int kt = ktime_begin(c, s, 5);
  const bool mixed = c->cfg.precision == GDF_PREC_MIXED;
  if (mixed) launch_grav<true>(c, a, false, s);
  else launch_grav<false>(c, a, false, s);
  GDF_HIP(c, hipGetLastError());
  ktime_end(c, s, kt);
  GDF_HIP(c, hipMemcpyAsync(c->h_counters + 16, c->counters + 16, sizeof(int)*8,
                            hipMemcpyDeviceToHost, s));
  GDF_HIP(c, hipStreamSynchronize(s));
  if (c->h_counters[16 + 2]) return fail(c, GDF_ERR_CAPACITY, "tree walk stack overflow in gravity pass");
  return GDF_OK;
}

}  // namespace gdf
