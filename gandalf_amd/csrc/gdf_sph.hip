// grad-h SPH passes: candidate walks, h-rho iteration and hydro forces.
//
// Replaces the OpenMP cell loops of GradhSphTree::UpdateAllSphProperties
// (src/GradhSph/GradhSphTree.cpp:83-271) and UpdateAllSphHydroForces (:280-435) with the
// per-particle physics of GradhSph::ComputeH (src/GradhSph/GradhSph.cpp:142-326) and
// ComputeSphHydroForces / ComputeSphHydroGravForces (:361-460, :474-585).
//
// Work mapping: a walk pass (two wavefronts per walk group, a tree node of up to 64
// Morton-consecutive particles) resolves the group's candidate particles from the tree: the
// members of every bucket that come within the group's search range.  The h-rho pass walks with bounds that also hold the scatter-gather sets of the converged smoothing
// lengths, so the force pass reads the same lists.  A pair pass takes one walk group per
// workgroup, one target a lane, and its wavefronts share the group's candidates: each stages its
// own in LDS batch by batch, filters them against the 64 targets on the matrix cores
// (gdf_filter.h) and lets every lane take its own target's hits, deciding each pair by the path's
// own range test.  The h-rho pass re-sweeps the same candidates until every target of the group
// has converged.
//
// The lists hold no masks: exact 64-bit masks per batch and target, made by the walk with 64
// distance tests a candidate and read back by the pair passes, cost 12 to 19 VALU instructions a
// test and 640 bytes a batch, and the FP64 force pass a walk of its own.  Without them one FP64
// force evaluation of a million particles (quintic, 64-particle groups) went from 17.2 to 13.2 ms
// (11.3 with the later changes described at each kernel).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gdf_internal.h"
#include "gdf_device.h"
#include "gdf_filter.h"

namespace gdf {
namespace {

constexpr int BS = 256;
constexpr double NODE_SLACK = 1.0 + 1e-12; // node tests err on the inclusive side
// the per-member filter of the candidate walks errs further on the inclusive side than any
// target's own test (FP32 tests of the mixed path included)
constexpr double KEEP_SLACK = 1.0 + 1e-4;
constexpr int kInitBatches = 16;           // initial candidate capacity per group, in batches
constexpr int kMaxLeaf = 14;               // largest bucket (Nleafmax)
constexpr int kWideStack = 4096;           // stack entries beyond which a round takes 64 nodes
constexpr int kMaxRounds = 64;             // search radii tried for a particle's h
constexpr double kMaxGrowth = 23.26;       // between 1.05^64 and 1.05^65: beyond the last of them

struct CandWalk {
  int N, ngroups, nleaf, capb;
  const int* grp_node; const int* grp_first; const int* grp_count;
  const int4* lnk;
  const double4* geo_c; const double4* geo_h;
  const double* x; const double* y; const double* z; const double* hcand; const double* htarget;
  const int* status;                 // only targets with status 1 take part (NULL = every member)
  const int* grp_root;               // serving batches: the group's segment subtree (NULL = root)
  const int* glist;                  // groups to walk (count at glist[Ncap]); NULL = all groups
  int ncap;
  int* idx; unsigned long long* mask; int* ncand;
  int* stacks; int* flags;
  PhysParams p;
};

// Candidate lists.  MODE 0: the gather search, every particle within k hs_i of a target (hs the
// search radii); MODE 1, 2: scatter-gather, within k h_i of a target i or k h_j of its own.
// UNION (MODE 0): the gather search's candidates also include every particle whose own search
// radius reaches the targets' box (hcand = the search radii hs_j = 1.05 h_j; a node's hs bound is
// 1.05 times its h maximum), so that while no smoothing length outgrows its search radius the
// list holds the scatter-gather set of the converged smoothing lengths as well.  The lists err on
// the inclusive side; the pair passes test every pair.  W wavefronts share a group: a round tests up
// to 64 W nodes of the group's stack, each wavefront the members of its own buckets.  Bound by the
// chain of rounds (stack, node, member loads), so wavefronts in flight count: one a group and 3072
// in all, fetching groups from eight counters on one line, took 870 us at a million particles, 405
// at 262144 (M4) and 97 at 100003; two a group and 6144 in all take 570, 108 and 67 (20011: 42 and
// 37; one a group and 4096: 567, 108, 79, 42; four and 8192: 975, 205, 88, 35).  MASKS (the parity
// tap): also each target's exact scatter-gather set as masks over the list, MODE 1 in FP64 with the
// oracle's operation order, MODE 2 in FP32 in the frame of the mixed path's pair kernels with their
// expression.  PER: periodic nearest images.
template <int MODE, bool PER, int W, bool MASKS = false, bool UNION = false>
__global__ __launch_bounds__(64*W) void k_walk_cand(CandWalk a) {
  static_assert(!MASKS || W == 1, "the masks' tests are a lone wavefront's");
  constexpr bool F32 = MODE == 2;      // group-frame FP32 tests
  constexpr bool GATHER = MODE == 0;
  __shared__ double4 sc[MASKS && !F32 ? kWave : 1];   // MODE 1: (x, y, z, (k h_j)^2)
  __shared__ float4 fc[MASKS && F32 ? kWave : 1];     // MODE 2: the same in the FP32 frame
  __shared__ int lstk[kLdsStack];    // node stack; deeper entries go to the global region
  __shared__ int kept[W > 1 ? W : 1][W > 1 ? kWave*kMaxLeaf : 1];    // a round's candidates
  __shared__ int count[W][2];        // a round's opened nodes and candidates
  const int lane = threadIdx.x & (kWave - 1), wv = W == 1 ? 0 : (int) threadIdx.x/kWave;
  int* stk = a.stacks + (size_t) blockIdx.x*kStackCap;
  const int N = a.N;
  const double krsqd = a.p.kern.rangesqd, kr = a.p.kern.range;
  PhysParams pp = a.p;
  pp.periodic = PER ? 1 : 0;
  const GroupQueue q = group_queue(a.glist ? a.glist[a.ncap] : a.ngroups);
  for (int k = q.first; k < q.end; k += q.step) {
    __syncthreads();                 // the last group's stack is done with
    const int g = a.glist ? a.glist[k] : k;
    const int G = a.grp_node[g], gfirst = a.grp_first[g], gcnt = a.grp_count[g];
    // tc, th: the box the walk tests nodes and members against, that of the group's targets
    // alone; a block step's sparse groups hold a few targets each and reach far fewer buckets
    // with it.  hG: their largest search radius
    double lox = HUGE_VAL, loy = HUGE_VAL, loz = HUGE_VAL, hG = 0.0;
    double hix = -HUGE_VAL, hiy = -HUGE_VAL, hiz = -HUGE_VAL;
    const int i = gfirst + lane;
    const bool has = lane < gcnt && (!a.status || a.status[i] == 1);
    double xi = 0.0, yi = 0.0, zi = 0.0, r2i = 0.0;
    if (has) {
      lox = hix = xi = a.x[i]; loy = hiy = yi = a.y[i]; loz = hiz = zi = a.z[i];
      hG = a.htarget[i];
      r2i = range2_rn(krsqd, hG);
    }
    if (__ballot(has) == 0) {        // nothing left to do in this group
      if (threadIdx.x == 0) a.ncand[g] = 0;
      continue;
    }
    hG = wave_max_d(hG);
    double4 tc, th;
    {
#pragma clang fp contract(off)
      lox = -wave_max_d(-lox); hix = wave_max_d(hix);
      loy = -wave_max_d(-loy); hiy = wave_max_d(hiy);
      loz = -wave_max_d(-loz); hiz = wave_max_d(hiz);
      tc = make_double4(0.5*(lox + hix), 0.5*(loy + hiy), 0.5*(loz + hiz), 0.0);
      th = make_double4(0.5*(hix - lox), 0.5*(hiy - loy), 0.5*(hiz - loz), 0.0);
    }
    int* idx = a.idx + (size_t) g*a.capb*kWave;
    const int cap = a.capb*kWave;
    int sp = 1, tail = 0;
    bool overflow = false;
    if (threadIdx.x == 0) lstk[0] = a.grp_root ? a.grp_root[g] : 0;  // the group's segment subtree
    __syncthreads();
    // 1. traversal: the particles of every bucket within range, round by round and wavefront by
    // wavefront, into idx
    while (sp > 0) {
      const int b = min(sp, sp > kWideStack ? kWave : kWave*W);
      const int slot = wv*kWave + lane;
      int node = -1;
      if (slot < b) node = stack_get(lstk, stk, sp - 1 - slot);
      sp -= b;
      bool open = false, emit = false;
      int ef = 0, ec = 0, cl = 0, cr = 0;
      if (node >= 0) {
        // box, range and children in one round of loads
        const double4 nc = a.geo_c[node], nh = a.geo_h[node];
        NodeLinks nl;
        load_links(node, N, a.lnk, nl);
        double dx = nc.x - tc.x, dy = nc.y - tc.y, dz = nc.z - tc.z;
        nearest_image<double>(pp, dx, dy, dz);
        const double gx = fmax(fabs(dx) - nh.x - th.x, 0.0);
        const double gy = fmax(fabs(dy) - nh.y - th.y, 0.0);
        const double gz = fmax(fabs(dz) - nh.z - th.z, 0.0);
        const double dbox2 = gx*gx + gy*gy + gz*gz;
        const double rr = UNION ? kr*fmax(hG, 1.05*nc.w) : GATHER ? kr*hG : kr*fmax(hG, nc.w);
        if (dbox2 <= rr*rr*NODE_SLACK) {
          ef = nl.first; ec = nl.count;
          if (ec <= a.nleaf) emit = true;
          else { open = true; cl = nl.left; cr = nl.right; }
        }
      }
      const unsigned long long om = __ballot(open);
      // a bucket's members that lie beyond the largest range from the group box fail every
      // target's test below: they are dropped here, once per member, instead of being tested
      // on all 64 lanes and staged by every pair pass (about a quarter of the members of the
      // buckets a group reaches).  The round's members are dealt one per lane, so that their
      // loads go out together, and the kept ones are recorded in bucket order.
      const int mcount = emit ? ec : 0;
      const int mincl = wave_incl_scan(mcount);
      const int mtot = __shfl(mincl, 63, 64);
      int nkept = 0;
      for (int base = 0; base < mtot; base += kWave) {
        const int s = base + lane;
        // the lane whose bucket holds member s: the first with an inclusive count above s
        int L = 0;
        #pragma unroll
        for (int step = 32; step >= 1; step >>= 1)
          if (__shfl(mincl, L + step - 1, 64) <= s) L += step;
        const int fL = __shfl(ef, L, 64), xL = __shfl(mincl - mcount, L, 64);
        bool kp = false;
        const int j = fL + (s - xL);
        if (s < mtot) {
          double dx = a.x[j] - tc.x, dy = a.y[j] - tc.y, dz = a.z[j] - tc.z;
          nearest_image<double>(pp, dx, dy, dz);
          const double ex = fmax(fabs(dx) - th.x, 0.0);
          const double ey = fmax(fabs(dy) - th.y, 0.0);
          const double ez = fmax(fabs(dz) - th.z, 0.0);
          const double rr = (GATHER && !UNION) ? kr*hG : kr*fmax(hG, a.hcand[j]);
          kp = ex*ex + ey*ey + ez*ez <= rr*rr*KEEP_SLACK;
        }
        const unsigned long long km = __ballot(kp);
        if (kp) {
          const int o = nkept + lanes_below(km);
          if (W > 1) kept[wv][o] = j;
          else if (tail + o < cap) idx[tail + o] = j;
        }
        nkept += __popcll(km);
      }
      // places of the round's opened nodes and candidates, wavefront by wavefront
      int nopen = __popcll(om), o0 = 0;
      if (W == 1) {
        tail += nkept;
      } else {
        if (lane == 0) { count[wv][0] = nopen; count[wv][1] = nkept; }
        __syncthreads();
        int t0 = 0;
        nopen = 0;
        #pragma unroll
        for (int w = 0; w < W; w++) {
          if (w == wv) { o0 = nopen; t0 = tail; }
          nopen += count[w][0]; tail += count[w][1];
        }
        for (int o = lane; o < nkept; o += kWave)
          if (t0 + o < cap) idx[t0 + o] = kept[wv][o];
      }
      if (sp + 2*nopen > kLdsStack + kStackCap) { overflow = true; break; }
      if (open) {
        const int o = sp + 2*(o0 + lanes_below(om));
        stack_put(lstk, stk, o, cr);
        stack_put(lstk, stk, o + 1, cl);
      }
      sp += 2*nopen;
      if (sp > kLdsStack) __threadfence_block();   // entries in the global overflow region
      __syncthreads();
    }
    if (overflow) {
      if (threadIdx.x == 0) atomicOr(&a.flags[2], 1);
      continue;
    }
    const int nbat = (tail + kWave - 1)/kWave;
    if (tail > cap) {                // candidates beyond the set's capacity: grow and repeat
      if (threadIdx.x == 0) { a.ncand[g] = tail; atomicMax(&a.flags[1], nbat); }
      continue;
    }
    if (!MASKS) {
      if (threadIdx.x == 0) a.ncand[g] = tail;
      continue;
    }
    __threadfence_block();
    unsigned long long* msk = a.mask + (size_t) g*a.capb*kWave;
    const double4 gc = a.geo_c[G];
    const float rxi = (float) (xi - gc.x), ryi = (float) (yi - gc.y), rzi = (float) (zi - gc.z);
    const float r2if = (float) r2i;
    // 2. masks: batch b holds the candidates at walk positions b, b + nbat, b + 2 nbat, ...,
    // so every batch samples the whole candidate region and each target's neighbours spread
    // evenly over the batches (fewer idle lanes in the per-target mask loops of the pair passes)
    // The candidate records of batch b + 1 are loaded while batch b is tested, and the
    // candidate indices of batch b + 2 with them.
    auto nbat_of = [&](int bb) { return (tail - bb + nbat - 1)/nbat; };
    auto record = [&](int j) {
      return make_double4(a.x[j], a.y[j], a.z[j], a.hcand[j]);
    };
    double4 cur = make_double4(0.0, 0.0, 0.0, 0.0), nxt = cur;
    int jn = 0;
    if (lane < nbat_of(0)) cur = record(idx[lane*nbat]);
    if (nbat > 1 && lane < nbat_of(1)) jn = idx[1 + lane*nbat];
    for (int b = 0; b < nbat; b++) {
      const int nb = nbat_of(b);
      if (lane < nb) {
        const double r2j = range2_rn(krsqd, cur.w);
        if (F32) {
          double dx = cur.x - gc.x, dy = cur.y - gc.y, dz = cur.z - gc.z;
          nearest_image<double>(pp, dx, dy, dz);
          fc[lane] = make_float4((float) dx, (float) dy, (float) dz, (float) r2j);
        } else {
          sc[lane] = make_double4(cur.x, cur.y, cur.z, r2j);
        }
      }
      int jn2 = 0;
      if (b + 1 < nbat && lane < nbat_of(b + 1)) nxt = record(jn);
      if (b + 2 < nbat && lane < nbat_of(b + 2)) jn2 = idx[b + 2 + lane*nbat];
      __syncthreads();
      unsigned long long m = 0;
      if (has) {
        // all 64 slots in a fixed-count unrolled loop, so several LDS reads are in flight (a
        // loop over the nb filled slots waited on one read per test); slots past nb are
        // masked off after the loop
        #pragma unroll 16
        for (int q = 0; q < kWave; q++) {
          bool in;
          if (F32) {
            const float4 c = fc[q];
            const float d2 = dot3_f(c.x - rxi, c.y - ryi, c.z - rzi);
            in = (d2 < r2if) | (d2 < c.w);
          } else {
            const double4 c = sc[q];
            double dx = c.x - xi, dy = c.y - yi, dz = c.z - zi;
            nearest_image<double>(pp, dx, dy, dz);
            const double d2 = dot3_rn(dx, dy, dz);
            in = (d2 < r2i) | (d2 < c.w);
          }
          m |= (unsigned long long) in << q;
        }
        if (nb < kWave) m &= (1ULL << nb) - 1ULL;
      }
      msk[b*kWave + lane] = m;
      __syncthreads();
      cur = nxt;
      jn = jn2;
    }
    if (lane == 0) a.ncand[g] = tail;
  }
}

struct DensArgs {
  int N, ngroups, capb, nopbc;
  const int* grp_node; const int* grp_first; const int* grp_count; const double4* geo_c;
  const double4* geo_h;
  const int* idx; const int* ncand;
  const double4* posm;
  double* h; double* hsearch; double* rho; double* invomega; double* zeta; double* hfactor;
  double* u; double* sound; double* pressure;
  int* status; int* flags; long long* icount;
  // stars of a gas + star run for their zeta terms (nstar = 0: none, or the terms are off)
  int nstar, star_soft;
  int ordered;             // tabulated FP32 kernels: see k_density
  // serving batches: a particle's request, and the requests whose lists do not bound their
  // scatter-gather sets (NULL otherwise)
  const int* seg; int* seg_bad;
  const double* sx; const double* sy; const double* sz; const double* sm; const double* sh;
  PhysParams p;
};

// One step of the grad-h iteration after the sums at h (GradhSph.cpp:219-256): the fixed point
// h <- h_fac (m/rho)^(1/3), bisection on [h_lower, h_upper] after hrho_itmax (30) iterations,
// failure after five times as many; cbrt differs from the reference's pow(., 1/3), which the final h
// takes, in the last bit.  Returns 2 to iterate again, 1 done (converged, or the bracket closed), 0
// retry with a larger search radius, -1 no convergence.
__device__ __forceinline__ int hrho_step(const PhysParams& p, double m, double hmax, int iteration,
                                         double rho, double& h, double& h_lower,
                                         double& h_upper) {
  const double invh = 1.0/h;
  const double hrho = rho > 0.0 ? p.h_fac*cbrt(m/rho) : 0.0;
  if (rho > 0.0 && h > h_lower && fabs(h - hrho)*invh < p.h_converge) return 1;
  if (iteration < p.hrho_itmax) h = hrho;
  else if (iteration == p.hrho_itmax) h = 0.5*(h_lower + h_upper);
  else if (iteration < 5*p.hrho_itmax) {
    if (rho < 1.0e-20 || h > hrho) h_upper = h; else h_lower = h;
    h = 0.5*(h_lower + h_upper);
  } else return -1;
  if (h > hmax) return 0;
  return (h > h_lower && h < h_upper) ? 2 : 1;
}

// Final h from rho, grad-h terms and EOS (GradhSph.cpp:260-317)
__device__ void hrho_finish(const DensArgs& a, const PhysParams& p, int i, double m, double rho,
                            double invomega, double zeta, double h_lower) {
  const double hrho = p.h_fac*pow(m/rho, 1.0/3);
  const double h = fmax(hrho, h_lower);
  const double invh = 1/h;
  const double hfac4 = invh*invh*invh*invh;
  const double deriv = -(1.0/3)*h/rho;
  double iom = 1.0 - deriv*invomega;
  iom = 1.0/iom;
  // the stars' conservative-gravity zeta terms (Hubber et al. 2013) at the final h, over the
  // pair's mean smoothing length or the particle's own (GradhSph.cpp:282-303)
  if (a.nstar > 0) {
#pragma clang fp contract(off)
    const double4 me = a.posm[i];
    for (int j = 0; j < a.nstar; j++) {
      double invhsqd;
      if (a.star_soft) { const double t = 2.0/(h + a.sh[j]); invhsqd = t*t; }
      else invhsqd = 4.0*invh*invh;
      const double dx = a.sx[j] - me.x, dy = a.sy[j] - me.y, dz = a.sz[j] - me.z;
      const double ssqd = (dx*dx + dy*dy + dz*dz)*invhsqd;
      zeta += a.sm[j]*invhsqd*kwzeta_s2(p.kern, ssqd);
    }
  }
  const double zt = deriv*zeta*iom;
  a.h[i] = h; a.rho[i] = rho; a.invomega[i] = iom; a.zeta[i] = zt; a.hfactor[i] = hfac4;
  double u = a.u[i], snd, press;
  eos_state(p, rho, u, snd, press);
  a.u[i] = u; a.sound[i] = snd; a.pressure[i] = press;
}

// h-rho pass, one walk group per workgroup, its W wavefronts sharing the candidates.  A sweep
// stages the candidates' positions batch by batch, filters them against the targets' current
// ranges and sums the hits; every wavefront adds the W partial sums in the same order and takes
// the same step of the iteration.  T = double: FP64 throughout; T = float: FP32 pair terms in the
// group-centred frame, the density's added up in FP64, the other sums batch by batch (the
// convergence test and the final h are always FP64).  KT: DensSums' kernel.
// Tabulated FP32 kernels take the nearest lower entry, so that an h rounded otherwise moves one pair
// in 10^4 to the next entry, 1 % of a particle's acceleration where it nearly cancels.  These
// passes keep to one order of summation, whatever the group: every batch of a lone wavefront's list
// by itself in FP32, batch after batch compensated, one lane a target (ORDER).  A force evaluation
// of 72^3 particles, ms, with masks, in this order and in any order: M4 3.20, 2.41, 2.44, quintic
// 3.79, 3.29, 2.83; of 14^3, M4, 0.57, 0.36, 0.33.
// Bound by vector issue where the device is full (1M particles, quintic: 0.25 VALU instructions
// a cycle and SIMD), by the latency of the dependent loads and of each sweep's reduction below;
// 3 wavefronts a SIMD, as 4 spill.  1M, quintic: 0.95 ms against 1.20 with masks (FP32), 1.51
// against 1.59 (FP64).
template <typename T, int KT, int W>
__global__ __launch_bounds__(64*W, 3) void k_density(DensArgs a) {
  constexpr bool F64 = sizeof(T) == 8, ORDER = !F64 && KT == 2;
  static_assert(!ORDER || W == 1, "one wavefront's order");
  typedef typename std::conditional<F64, double4, float4>::type Rec;
  __shared__ Rec stage[W][kPairSlots];
  __shared__ double red[W > 1 ? W : 1][3][W > 1 ? kWave : 1];
  const int g = xcd_block(blockIdx.x, gridDim.x);
  const int lane = threadIdx.x & (kWave - 1), wv = W == 1 ? 0 : (int) threadIdx.x/kWave;
  const int nc = a.ncand[g];
  if (nc <= 0 || nc > a.capb*kWave) return;   // no active target, or the walk overflowed
  const int gfirst = a.grp_first[g], gcnt = a.grp_count[g];
  Rec* const st = stage[wv];
  const unsigned long long on = __ballot(lane < gcnt && a.status[gfirst + lane] == 1);
  if (on == 0) return;
  const TargetLanes tl(on, ORDER);
  const bool has = tl.has, writes = wv == 0 && tl.copy == 0;
  const int i = has ? gfirst + tl.member : 0;
  const unsigned mine = tl.share();
  int state = has ? 2 : 3;                    // 2 iterating, 3 not a target
  PhysParams p = a.p;
  if (a.nopbc) p.periodic = 0;
  const double4 gc = a.geo_c[a.grp_node[g]], gh = a.geo_h[a.grp_node[g]];
  double4 me = make_double4(gc.x, gc.y, gc.z, 1.0);
  double h = 1.0, hmax = 1.0;
  if (has) { me = a.posm[i]; h = a.h[i]; hmax = a.hsearch[i]; }
  const double m = me.w;
  double h_lower = 0.0, h_upper = hmax;
  int iteration = 0, ngather = 0, evals = 0;
  const float rxi = (float) (me.x - gc.x), ryi = (float) (me.y - gc.y), rzi = (float) (me.z - gc.z);
  const double rsq = p.kern.rangesqd;
  // the filter's frame: the group's half-diagonal plus the targets' largest search range below one
  const double rG = p.kern.range*wave_max_d(has ? hmax : 0.0);
  const T fs = filter_scale<T>(sqrt(gh.x*gh.x + gh.y*gh.y + gh.z*gh.z) + rG);
  const float fx = (float) ((T) (me.x - gc.x)*fs), fy = (float) ((T) (me.y - gc.y)*fs),
              fz = (float) ((T) (me.z - gc.z)*fs);
  // FP64 separations take the nearest image target by target: where a candidate's image about
  // the group's centre need not be its image about every target, all candidates are taken
  const bool all = F64 && p.periodic && (gh.x + rG >= p.boxhalf[0] || gh.y + rG >= p.boxhalf[1] ||
                                         gh.z + rG >= p.boxhalf[2]);
  FiltTargets ft;
  ft.position(fx, fy, fz);
  const PairBatches pb((nc - wv + W - 1)/W);
  const int* idx = a.idx + (size_t) g*a.capb*kWave + wv;
  while (__ballot(state == 2)) {
    const bool run = state == 2;
    if (run) iteration++;
    const double invh = 1.0/h;
    const double invhsqd = invh*invh;
    const float invhsqdf = (float) invhsqd, hs = (float) ((T) h*fs);
    ft.range(fx, fy, fz, run ? (float) rsq*hs*hs : -1.f);
    int inside = 0;
    DensSums<double, KT> sum;
    KahanF kr, kom, kz;
    const float invhf = (float) invh;
    HitQueue hq;
    Rec rec{};
    // the next batch's record and the indices of the one after it are in flight
    double4 nx = make_double4(0.0, 0.0, 0.0, 0.0);
    if (pb.filled(0, lane)) nx = a.posm[idx[pb.index(0, lane)*W]];
    int jn = pb.filled(1, lane) ? idx[pb.index(1, lane)*W] : -1;
    for (int b = 0; b < pb.nb; b++) {
      const int s0 = kWave*(b & 1);
      if constexpr (F64) {
        st[s0 + lane] = nx;
      } else {
        double dx = nx.x - gc.x, dy = nx.y - gc.y, dz = nx.z - gc.z;
        nearest_image<double>(p, dx, dy, dz);
        st[s0 + lane] = make_float4((float) dx, (float) dy, (float) dz, (float) nx.w);
      }
      wave_lds_order();
      if (jn >= 0) nx = a.posm[jn];
      jn = pb.filled(b + 2, lane) ? idx[pb.index(b + 2, lane)*W] : -1;
      const uint2 hit = filter64<false>(ft, [&](int l) {
        FiltCand f;
        const Rec r = st[s0 + l];
        if (F64) {
          double dx = r.x - gc.x, dy = r.y - gc.y, dz = r.z - gc.z;
          nearest_image<double>(p, dx, dy, dz);
          f.x = (float) (dx*fs); f.y = (float) (dy*fs); f.z = (float) (dz*fs);
        } else {
          f.x = (float) (r.x*fs); f.y = (float) (r.y*fs); f.z = (float) (r.z*fs);
        }
        f.thr = 0.f;
        f.state = !pb.filled(b, l) ? 1 : all ? -1 : 0;
        return f;
      });
      hq.stage(b == 0, run ? make_uint2(hit.x & mine, hit.y & mine) : make_uint2(0u, 0u));
      const int need = b + 1 < pb.nb && !ORDER ? hq.older : hq.staged;
      if constexpr (F64) {
        hq.run(need, rec, [&](int q) { return st[q]; }, [&](const Rec& pj, bool take) {
          double dx = pj.x - me.x, dy = pj.y - me.y, dz = pj.z - me.z;
          nearest_image<double>(p, dx, dy, dz);
          const double ssqd = invhsqd*(dx*dx + dy*dy + dz*dz);
          inside += take & (ssqd < rsq);
          sum.add(p.kern, ssqd, take ? pj.w : 0.0);
        });
      } else if constexpr (ORDER) {
        float br = 0.f, bom = 0.f, bz = 0.f;
        hq.run(need, rec, [&](int q) { return st[q]; }, [&](const Rec& pj, bool take) {
          const float dx = pj.x - rxi, dy = pj.y - ryi, dz = pj.z - rzi;
          const float ssqd = invhsqdf*(dx*dx + dy*dy + dz*dz);
          if (take && ssqd < (float) rsq) {
            inside++;
            const float* t = ktab<float>(p.kern) + (int) (ssqd*(float) p.kern.resinvsqd);
            const int res = p.kern.res;
            br += pj.w*t[KW0S2*res];
            bom += pj.w*invhf*t[KWOMEGAS2*res];
            bz += pj.w*t[KWZETAS2*res];
          }
        });
        kr.add(br); kom.add(bom); kz.add(bz);
      } else {
        DensSums<float, KT> part;
        hq.run(need, rec, [&](int q) { return st[q]; }, [&](const Rec& pj, bool take) {
          const float dx = pj.x - rxi, dy = pj.y - ryi, dz = pj.z - rzi;
          const float ssqd = invhsqdf*(dx*dx + dy*dy + dz*dz);
          inside += take & (ssqd < (float) rsq);
          part.add(p.kern, ssqd, take ? pj.w : 0.f);
        });
        sum.r += part.r; sum.o += (double) part.o; sum.z += (double) part.z;
      }
      wave_lds_order();
    }
    if (ORDER) { sum.r = (double) kr.s; sum.o = (double) kom.s; sum.z = (double) kz.s; }
    evals += hq.staged;
    double r_ = tl.over_copies(sum.r), om_ = tl.over_copies(sum.o), z_ = tl.over_copies(sum.z);
    inside = tl.over_copies(inside);
    if (W > 1) {
      red[wv][0][lane] = r_; red[wv][1][lane] = om_; red[wv][2][lane] = z_;
      __syncthreads();
      r_ = om_ = z_ = 0.0;
      for (int w = 0; w < W; w++) {
        r_ += red[w][0][lane]; om_ += red[w][1][lane]; z_ += red[w][2][lane];
      }
      __syncthreads();
    }
    if (run) {
      const double hfac3 = invh*invhsqd;
      DensSums<T, KT>::finish(p.kern, r_, om_, z_);
      const double rho = r_*hfac3, invomega = (ORDER ? om_ : om_*invh)*hfac3, zeta = z_*invhsqd;
      const int rc = hrho_step(p, m, hmax, iteration, rho, h, h_lower, h_upper);
      if (rc == 1) {
        // converged: the sums and the bracket go to k_hrho_finish (status 2), which keeps
        // the final h, grad-h terms and EOS out of this kernel's register budget
        if (writes) {
          a.rho[i] = rho; a.invomega[i] = invomega; a.zeta[i] = zeta; a.hfactor[i] = h_lower;
          a.status[i] = 2;
        }
        ngather = tl.copy == 0 ? inside : 0;
        state = 1;
      } else if (rc == 0) {
        if (writes) {
          // a larger search radius (k_hrho_finish, status 3) for an h past this one's
          a.hfactor[i] = h;
          a.status[i] = 3;
          atomicAdd(&a.flags[0], 1);
        }
        state = 0;
      } else if (rc < 0) {
        if (writes) {
          a.status[i] = 0;
          atomicOr(&a.flags[3], 1);
        }
        state = -1;
      }
    }
  }
  wave_add_ll(&a.icount[0], ngather);
  wave_add_ll(&a.icount[4], evals);
}

template <typename T, int KT>
void launch_density_k(const DensArgs& d, int waves, hipStream_t s) {
  constexpr int many = sizeof(T) == 4 && KT == 2 ? 1 : 4;     // (waves is then 1)
  if (waves == 4) k_density<T, KT, many><<<d.ngroups, many*kWave, 0, s>>>(d);
  else k_density<T, KT, 1><<<d.ngroups, kWave, 0, s>>>(d);
}

template <typename T>
void launch_density(const DensArgs& d, int waves, hipStream_t s) {
  if (d.p.kern.tabulated) launch_density_k<T, 2>(d, waves, s);
  else if (d.p.kern.type == 0) launch_density_k<T, 0>(d, waves, s);
  else launch_density_k<T, 1>(d, waves, s);
}

// Final h, grad-h terms and EOS of the particles the h-rho pass has just converged (status 2:
// rho, invomega and zeta hold the sums at the converged h, hfactor the bracket's lower end), and
// the next search radius of those that need one (status 3: hfactor holds the h that was past it)
__global__ void k_hrho_finish(DensArgs a) {
  const int i = blockIdx.x*BS + threadIdx.x;
  if (i >= a.N || a.status[i] < 2) return;
  if (a.status[i] == 3) {
    // GradhSphTree.cpp:154: hmax = 1.05 hmax per retry, here at once as often as it takes to reach
    // the h that was past it: the iteration starts again from the same h and comes back to it, so
    // the retries on the way would end where the last one did.  (An h of a first guess takes two
    // or three instead of up to ten: six spheres set up and served 38.4 -> 36.8 ms.)  One step at a
    // time where the order of the sums counts (ordered): it follows the targets' common search.
    const double h = a.hfactor[i];
    double hs = a.hsearch[i]*1.05;
    for (int k = 0; k < kMaxRounds && hs < h && !a.ordered; k++) hs *= 1.05;
    a.hsearch[i] = hs;
    a.status[i] = 1;
    if (a.seg_bad) a.seg_bad[a.seg[i]] = 1;
    // past the last radius that a round each would try
    if (hs > kMaxGrowth*a.h[i]) atomicOr(&a.flags[3], 4);
    return;
  }
  hrho_finish(a, a.p, i, a.posm[i].w, a.rho[i], a.invomega[i], a.zeta[i], a.hfactor[i]);
  a.status[i] = 0;
  // a final h past the search radius (h from rho after the convergence test can exceed it by
  // up to h_converge): the walk's union lists no longer bound the scatter-gather set
  if (a.h[i] > a.hsearch[i]) {
    atomicOr(&a.flags[3], 2);
    if (a.seg_bad) a.seg_bad[a.seg[i]] = 1;
  }
}

// act (block timesteps): only the active particles iterate; NULL = all.  seg_bad[0, nseg) is cleared
// (a batch's requests have two particles or more each)
__global__ void k_init_density(int N, const double* __restrict__ h, double* __restrict__ hs,
                               int* __restrict__ status, const int* __restrict__ act, int nseg,
                               int* __restrict__ seg_bad) {
  const int i = blockIdx.x*BS + threadIdx.x;
  if (i >= N) return;
  if (i < nseg) seg_bad[i] = 0;
  hs[i] = 1.05*h[i];      // the search radius and bisection bracket, as GradhSphTree.cpp:154
  status[i] = act ? act[i] : 1;
}

// status 1 for the particles of the requests that seg_bad marks (or, bad = 0, does not), 0 for the rest
__global__ void k_seg_status(int N, const int* __restrict__ seg, const int* __restrict__ seg_bad,
                             int bad, int* __restrict__ status) {
  const int i = blockIdx.x*BS + threadIdx.x;
  if (i < N) status[i] = seg_bad[seg[i]] == bad;
}

__global__ void k_zero_ints(int n, int* __restrict__ p) {
  const int i = blockIdx.x*BS + threadIdx.x;
  if (i < n) p[i] = 0;
}

// hydro neighbour records: A = (v, 1/h), B = (1/rho, P invomega/rho^2, sound, hfactor); tgt (block
// steps): the pass's targets, kept for the parity tap
__global__ void k_pack_hydro(int N, const double* __restrict__ vx, const double* __restrict__ vy,
                             const double* __restrict__ vz, const double* __restrict__ h,
                             const double* __restrict__ rho, const double* __restrict__ pres,
                             const double* __restrict__ iom, const double* __restrict__ snd,
                             const double* __restrict__ hf, double4* __restrict__ A,
                             double4* __restrict__ B, const int* __restrict__ act,
                             int* __restrict__ tgt) {
  const int i = blockIdx.x*BS + threadIdx.x;
  if (i >= N) return;
  if (tgt) tgt[i] = act[i];
  A[i] = make_double4(vx[i], vy[i], vz[i], 1/h[i]);
  const double r = rho[i];
  B[i] = make_double4(1/r, (pres[i]*iom[i])/(r*r), snd[i], hf[i]);
}

struct HydroArgs {
  int N, ngroups, capb;
  const int* grp_node; const int* grp_first; const int* grp_count;
  const double4* geo_c; const double4* geo_h;
  const int* idx; const int* ncand;
  // serving batches: the lists of the groups that walked again (ncand2 > 0), in place of idx's
  int capb2; const int* idx2; const int* ncand2;
  const double4* posm; const double4* A; const double4* B;
  const double* h;
  const double* invomega; const double* pressure; const double* zeta;
  double* ax; double* ay; double* az; double* dudt; double* div_v;
  double* gx; double* gy; double* gz; double* gpot;    // softened neighbour gravity (VAR 1)
  long long* icount;
  // block timesteps (BLK): active flags, levels and neighbour levels
  const int* act; const int* level; int* levelneib;
  PhysParams p;
};

// Neighbour levels of a block step (GradhSph.cpp:445-446, merged as GradhSphTree.cpp:375-417):
// an active i takes the largest level of its scatter-gather set (itself included), and every
// inactive j of that set takes max(levelneib_j, level_i).  The set relation is symmetric, so an
// active j gets level_i from its own pass; records carry level_j and the bound below which an
// update of j is needed (255 for an active j: never).
__device__ __forceinline__ int blk_record(const HydroArgs& a, int j) {
  return a.level[j] | ((a.act[j] ? 255 : a.levelneib[j]) << 8);
}

// The nine sums of a hydro pass
template <typename T> struct HydroSums {
  T ax = T(0), ay = T(0), az = T(0), du = T(0), dv = T(0);
  T gx = T(0), gy = T(0), gz = T(0), gp = T(0);
  template <typename U> __device__ __forceinline__ void add(const HydroSums<U>& o) {
    ax += (T) o.ax; ay += (T) o.ay; az += (T) o.az; du += (T) o.du; dv += (T) o.dv;
    gx += (T) o.gx; gy += (T) o.gy; gz += (T) o.gz; gp += (T) o.gp;
  }
  template <typename U> __device__ __forceinline__ void to(HydroSums<U>& o) const {
    o.ax = (U) ax; o.ay = (U) ay; o.az = (U) az; o.du = (U) du; o.dv = (U) dv;
    o.gx = (U) gx; o.gy = (U) gy; o.gz = (U) gz; o.gp = (U) gp;
  }
};

template <typename T> struct Vec4 { T x, y, z, w; };
// A wavefront's staged candidates of the hydro passes: position and mass, velocity and 1/h,
// (1/rho, P Omega^-1/rho^2, c_s, hfactor), zeta, the squared range, and a block step's particle
// and level record
template <typename T, int VAR, bool BLK> struct HydroStage {
  Vec4<T> P[kPairSlots], V[kPairSlots], B[kPairSlots];
  T Z[VAR == 1 ? kPairSlots : 1], R[kPairSlots];
  int J[BLK ? kPairSlots : 1], L[BLK ? kPairSlots : 1];
};

// VAR 0: ComputeSphHydroForces (GradhSph.cpp:361-460); VAR 1: ComputeSphHydroGravForces
// (:474-585), the hydro terms plus the kernel-softened gravity of the pair (into gx, gy, gz,
// gpot; the tree walk adds the direct and multipole terms afterwards).  One walk group per
// workgroup, its W wavefronts sharing the candidates.  T = double: FP64
// throughout, separations target by target.  T = float: records in FP32 in the group's frame
// (positions relative to its centre, velocities to its first particle), pair terms in FP32 summed
// batch by batch, FP64 totals.  A hit of the filter is a pair if the path's own test says so, the
// one its gravity walk masks with.
// Bound by vector issue (1M particles, quintic: 0.27 VALU instructions a cycle and SIMD in FP32,
// 0.18 in FP64); the launch bounds are the most wavefronts a SIMD without spills (one more cost
// 24 % in FP32).  1M, quintic, with gravity, alone on the device: 2.02 ms against 2.25 (FP32) and
// 3.45 against 5.06 (FP64) with masks.
template <typename T, int KT, int VAR, bool BLK, int W>
__global__ __launch_bounds__(64*W, sizeof(T) == 8 ? 2 : 3) void k_hydro(HydroArgs a) {
  constexpr bool F64 = sizeof(T) == 8, ORDER = !F64 && KT == 2;       // see k_density
  static_assert(!ORDER || W == 1, "one wavefront's order");
  constexpr int NS = VAR == 1 ? 9 : 5;
  __shared__ HydroStage<T, VAR, BLK> stage[W];
  const int g = xcd_block(blockIdx.x, gridDim.x);
  const int lane = threadIdx.x & (kWave - 1), wv = W == 1 ? 0 : (int) threadIdx.x/kWave;
  const int n2 = a.ncand2 ? a.ncand2[g] : 0;
  const int nc = n2 > 0 ? n2 : a.ncand[g];
  if (nc <= 0) return;                        // no target in this group
  const int gfirst = a.grp_first[g], gcnt = a.grp_count[g];
  HydroStage<T, VAR, BLK>& st = stage[wv];
  const unsigned long long on = __ballot(lane < gcnt && (!BLK || a.act[gfirst + lane] != 0));
  if (on == 0) return;
  const TargetLanes tl(on, ORDER);
  const bool has = tl.has, writes = wv == 0 && tl.copy == 0;
  const int i = has ? gfirst + tl.member : 0;
  const unsigned mine = tl.share();
  const PhysParams& p = a.p;
  const double krsqd = p.kern.rangesqd;
  const double4 gc = a.geo_c[a.grp_node[g]], gh = a.geo_h[a.grp_node[g]];
  const double4 vref = a.A[gfirst];
  int lmax = 0, npairs = 0;
  const int level_i = BLK && has ? a.level[i] : 0;
  double4 me = make_double4(gc.x, gc.y, gc.z, 1.0), mA = make_double4(vref.x, vref.y, vref.z, 1.0);
  double4 mB = make_double4(1.0, 0.0, 0.0, 0.0);
  T zeta_i = T(0), r2i = T(-1);
  double h_i = 0.0;
  if (has) {
    me = a.posm[i]; mA = a.A[i]; mB = a.B[i];
    if (VAR == 1) zeta_i = (T) a.zeta[i];
    h_i = a.h[i];
    r2i = (T) range2_rn(krsqd, h_i);
  }
  const T rxi = (T) (F64 ? me.x : me.x - gc.x), ryi = (T) (F64 ? me.y : me.y - gc.y),
          rzi = (T) (F64 ? me.z : me.z - gc.z);
  const T vxi = F64 ? (T) mA.x : (T) (mA.x - vref.x), vyi = F64 ? (T) mA.y : (T) (mA.y - vref.y),
          vzi = F64 ? (T) mA.z : (T) (mA.z - vref.z);
  const T invh_i = (T) mA.w, invrho_i = (T) mB.x, pterm_i = (T) mB.y, snd_i = (T) mB.z;
  const T hf_i = (T) (mB.w*HydroKern<T, KT>::w1_factor(p.kern));
  const T alpha = (T) p.alpha_visc, beta = (T) p.beta_visc;
  // the filter's frame: the group's half-diagonal plus the targets' largest range below one
  const double rG = p.kern.range*wave_max_d(h_i);
  const double diag = sqrt(gh.x*gh.x + gh.y*gh.y + gh.z*gh.z);
  const T fs = filter_scale<T>(diag + rG);
  const float fx = (float) ((T) (me.x - gc.x)*fs), fy = (float) ((T) (me.y - gc.y)*fs),
              fz = (float) ((T) (me.z - gc.z)*fs);
  FiltTargets ft;
  ft.position(fx, fy, fz);
  ft.range(fx, fy, fz, has ? (float) ((double) r2i*fs*fs) : -1.f);
  HydroSums<double> sum;
  KahanF kx, ky, kz, ku, kv;
  const PairBatches pb((nc - wv + W - 1)/W);
  const int* idx = (n2 > 0 ? a.idx2 + (size_t) g*a.capb2*kWave : a.idx + (size_t) g*a.capb*kWave) + wv;
  const double w1f = HydroKern<T, KT>::w1_factor(p.kern);
  HitQueue hq;
  int rec = 0;
  int jn = pb.filled(0, lane) ? idx[pb.index(0, lane)*W] : -1;
  for (int b = 0; b < pb.nb; b++) {
    const int s0 = kWave*(b & 1);
    if (jn >= 0) {
      const int j = jn, s = s0 + lane;
      const double4 pj = a.posm[j], Aj = a.A[j], Bj = a.B[j];
      if (F64) {
        st.P[s] = {(T) pj.x, (T) pj.y, (T) pj.z, (T) pj.w};
        st.V[s] = {(T) Aj.x, (T) Aj.y, (T) Aj.z, (T) Aj.w};
      } else {
        double dx = pj.x - gc.x, dy = pj.y - gc.y, dz = pj.z - gc.z;
        nearest_image<double>(p, dx, dy, dz);
        st.P[s] = {(T) dx, (T) dy, (T) dz, (T) pj.w};
        st.V[s] = {(T) (Aj.x - vref.x), (T) (Aj.y - vref.y), (T) (Aj.z - vref.z), (T) Aj.w};
      }
      st.B[s] = {(T) Bj.x, (T) Bj.y, (T) Bj.z, (T) (Bj.w*w1f)};
      if (VAR == 1) st.Z[s] = (T) a.zeta[j];
      st.R[s] = (T) range2_rn(krsqd, a.h[j]);
      if (BLK) { st.J[s] = j; st.L[s] = blk_record(a, j); }
    }
    jn = pb.filled(b + 1, lane) ? idx[pb.index(b + 1, lane)*W] : -1;
    wave_lds_order();
    const uint2 hit = filter64<true>(ft, [&](int l) {
      FiltCand f = {0.f, 0.f, 0.f, 0.f, 1};
      if (!pb.filled(b, l)) return f;
      const Vec4<T> r = st.P[s0 + l];
      const T r2 = st.R[s0 + l];
      f.state = 0;
      if (F64) {
        double dx = r.x - gc.x, dy = r.y - gc.y, dz = r.z - gc.z;
        nearest_image<double>(p, dx, dy, dz);
        f.x = (float) (dx*fs); f.y = (float) (dy*fs); f.z = (float) (dz*fs);
        if (p.periodic) {
          // taken unless its image about the centre is its image about every target in range
          const double R = fmax(rG, sqrt((double) r2));
          if (gh.x + R >= p.boxhalf[0] || gh.y + R >= p.boxhalf[1] || gh.z + R >= p.boxhalf[2])
            f.state = -1;
        }
      } else {
        f.x = (float) (r.x*fs); f.y = (float) (r.y*fs); f.z = (float) (r.z*fs);
      }
      f.thr = filter_thr((float) ((double) r2*fs*fs));
      return f;
    });
    hq.stage(b == 0, has ? make_uint2(hit.x & mine, hit.y & mine) : make_uint2(0u, 0u));
    const int need = b + 1 < pb.nb && !ORDER ? hq.older : hq.staged;
    HydroSums<T> part;
    if (F64) sum.to(part);
    hq.run(need, rec, [&](int q) { return q; }, [&](int q, bool take) {
      const Vec4<T> P = st.P[q], V = st.V[q], B = st.B[q];
      T dx = P.x - rxi, dy = P.y - ryi, dz = P.z - rzi;
      if (F64) nearest_image<T>(p, dx, dy, dz);
      const T d2 = dot3_t(dx, dy, dz);
      const bool in = take & ((d2 < r2i) | (d2 < st.R[q]));
      const T mj = in ? P.w : T(0);
      npairs += in;
      if (BLK) {
        const int lj = st.L[q];
        if (in) lmax = max(lmax, lj & 255);
        if (in && level_i > (lj >> 8)) atomicMax(&a.levelneib[st.J[q]], level_i);
      }
      // unit separation; the particle itself has none
      const T tiny = F64 ? T(1.0e-280) : T(1.0e-36);
      const T d2e = VAR == 1 ? d2 + T(1.0e-20) : (d2 > tiny ? d2 : tiny);
      T inv = rsq_t(d2e), drmag = d2e*inv;
      if constexpr (ORDER) {
        // a fixed rounding: it decides the table's entry
        const float s2 = fmaf(dz, dz, fmaf(dx, dx, dy*dy));
        drmag = sqrt_f(VAR == 1 ? s2 + 1.0e-20f : s2);
        inv = drmag > 0.f ? rcp_f(drmag) : 0.f;
      }
      dx *= inv; dy *= inv; dz *= inv;
      const T invh_j = V.w;
      HydroKern<T, KT> ki, kj;
      ki.set(p.kern, drmag*invh_i);
      kj.set(p.kern, drmag*invh_j);
      const T wkerni = hf_i*ki.w1, wkernj = B.w*kj.w1;
      const T dvdr = (V.x - vxi)*dx + (V.y - vyi)*dy + (V.z - vzi)*dz;
      part.dv -= mj*dvdr*wkerni;
      T paux = pterm_i*wkerni + B.y*wkernj;
      if (dvdr < T(0)) {
        const T winvrho = T(0.25)*(wkerni + wkernj)*(invrho_i + B.x);
        if constexpr (ORDER) {
          const float vsignal = snd_i + B.z - beta*alpha*dvdr;
          paux -= alpha*vsignal*dvdr*winvrho;
          part.du -= 0.5f*mj*alpha*vsignal*dvdr*dvdr*winvrho;
        } else {
          const T q2 = alpha*(snd_i + B.z - beta*alpha*dvdr)*dvdr*winvrho;
          paux -= q2;
          part.du -= T(0.5)*mj*q2*dvdr;
        }
      }
      if constexpr (ORDER) {
        part.ax += mj*dx*paux; part.ay += mj*dy*paux; part.az += mj*dz*paux;
      } else {
        const T ma = mj*paux;
        part.ax += ma*dx; part.ay += ma*dy; part.az += ma*dz;
      }
      if (VAR == 1) {
        T mi, poti, mjj, potj;
        ki.grav(p.kern, mi, poti);
        kj.grav(p.kern, mjj, potj);
        // wgrav/h^2 = M/d^2 and wpot/h = M/d + P/h (enclosed mass M, outer integral P); the
        // factor 1/2 of the pair mean is applied to the sums
        const T M = mi + mjj;
        const T mg = mj*(M*(inv*inv) + zeta_i*wkerni + st.Z[q]*wkernj);
        part.gx += mg*dx; part.gy += mg*dy; part.gz += mg*dz;
        part.gp += mj*(M*inv + (invh_i*poti + invh_j*potj));
      }
    });
    if (ORDER) {
      kx.add((float) part.ax); ky.add((float) part.ay); kz.add((float) part.az);
      ku.add((float) part.du); kv.add((float) part.dv);
    }
    if (F64) part.to(sum);
    else sum.add(part);
    wave_lds_order();
  }
  if (ORDER) {
    sum.ax = (double) kx.s; sum.ay = (double) ky.s; sum.az = (double) kz.s;
    sum.du = (double) ku.s; sum.dv = (double) kv.s;
  }
  if (tl.copies > 1) {
    sum.ax = tl.over_copies(sum.ax); sum.ay = tl.over_copies(sum.ay); sum.az = tl.over_copies(sum.az);
    sum.du = tl.over_copies(sum.du); sum.dv = tl.over_copies(sum.dv);
    if (VAR == 1) {
      sum.gx = tl.over_copies(sum.gx); sum.gy = tl.over_copies(sum.gy);
      sum.gz = tl.over_copies(sum.gz); sum.gp = tl.over_copies(sum.gp);
    }
    if (BLK) for (int o = tl.span; o < kWave; o <<= 1) lmax = max(lmax, __shfl_xor(lmax, o, kWave));
  }
  if (W > 1) {
    // the wavefronts' sums, added in order by the first
    double v[NS] = {sum.ax, sum.ay, sum.az, sum.du, sum.dv};
    if (VAR == 1) { v[NS - 4] = sum.gx; v[NS - 3] = sum.gy; v[NS - 2] = sum.gz; v[NS - 1] = sum.gp; }
    static_assert(sizeof(stage) >= sizeof(double)*64*W, "a row of sums per wavefront");
    double* red = reinterpret_cast<double*>(&stage[0]);     // one sum at a time
    for (int k = 0; k < NS; k++) {
      __syncthreads();
      red[threadIdx.x] = v[k];
      __syncthreads();
      if (wv == 0)
        for (int w = 1; w < W; w++) v[k] += red[w*kWave + lane];
    }
    sum.ax = v[0]; sum.ay = v[1]; sum.az = v[2]; sum.du = v[3]; sum.dv = v[4];
    if (VAR == 1) { sum.gx = v[NS - 4]; sum.gy = v[NS - 3]; sum.gz = v[NS - 2]; sum.gp = v[NS - 1]; }
    if (BLK) {
      int* ri = reinterpret_cast<int*>(&stage[0]);
      __syncthreads();
      ri[threadIdx.x] = lmax;
      __syncthreads();
      if (wv == 0)
        for (int w = 1; w < W; w++) lmax = max(lmax, ri[w*kWave + lane]);
    }
  }
  wave_add_ll(&a.icount[1], npairs);
  // the filter's candidate-target tests (counted for the mixed path)
  if (!F64) wave_add_ll(&a.icount[5], has && writes ? nc : 0);
  if (!has || !writes) return;
  if (BLK) a.levelneib[i] = lmax;
  const double dvd = sum.dv*mB.x;
  const double dud = sum.du - a.pressure[i]*dvd*mB.x*a.invomega[i];
  a.ax[i] = sum.ax; a.ay[i] = sum.ay; a.az[i] = sum.az;
  a.dudt[i] = dud; a.div_v[i] = dvd;
  if (VAR == 1) {
    a.gx[i] = 0.5*sum.gx; a.gy[i] = 0.5*sum.gy; a.gz[i] = 0.5*sum.gz;
    a.gpot[i] = 0.5*sum.gp;
  }
}

template <typename T, int KT, int W>
void launch_hydro_w(const HydroArgs& h, int variant, bool blk, hipStream_t s) {
  const int grid = h.ngroups;
  if (variant == 0) {
    if (blk) k_hydro<T, KT, 0, true, W><<<grid, W*kWave, 0, s>>>(h);
    else k_hydro<T, KT, 0, false, W><<<grid, W*kWave, 0, s>>>(h);
  } else {
    if (blk) k_hydro<T, KT, 1, true, W><<<grid, W*kWave, 0, s>>>(h);
    else k_hydro<T, KT, 1, false, W><<<grid, W*kWave, 0, s>>>(h);
  }
}

template <typename T, int KT>
void launch_hydro_k(const HydroArgs& h, int variant, bool blk, int waves, hipStream_t s) {
  constexpr bool ordered = sizeof(T) == 4 && KT == 2;         // waves is 1
  if (waves == 4) launch_hydro_w<T, KT, ordered ? 1 : 4>(h, variant, blk, s);
  else if (waves == 2) launch_hydro_w<T, KT, ordered ? 1 : 2>(h, variant, blk, s);
  else launch_hydro_w<T, KT, 1>(h, variant, blk, s);
}

template <typename T>
void launch_hydro(const HydroArgs& h, int variant, bool blk, int waves, hipStream_t s) {
  if (h.p.kern.tabulated) launch_hydro_k<T, 2>(h, variant, blk, waves, s);
  else if (h.p.kern.type == 0) launch_hydro_k<T, 0>(h, variant, blk, waves, s);
  else launch_hydro_k<T, 1>(h, variant, blk, waves, s);
}

// Wavefronts that share a walk group's candidates in the pair passes.  A group's pass is a chain
// of dependent loads, sums and reductions, so while one wavefront a group leaves most of the 1024
// SIMDs idle more of them finish sooner; once the device is full every further wavefront only
// adds partly filled batches and, in the h-rho pass, barriers between sweeps.  Times (us) with 1,
// 2 and 4 wavefronts, by groups (FP64 below 2048, FP32 from there on):
//   groups      128          512          1024          2048          4096
//   h-rho    36 24 20     46 43 61     91  89 133    164 183 257   198 319 589
//   hydro    48 32 22     94 63 70    159 153 177    575 474 456   547 560 668
// A serving batch keeps to one: a request's sums must not depend on what else is resident.
// Nor may a tabulated FP32 kernel's passes depend on the number (see k_density).
bool ordered_sums(const gdf_ctx* c) {
  return c->cfg.precision == GDF_PREC_MIXED && c->phys.kern.tabulated;
}
int density_waves(const gdf_ctx* c) {
  return c->ngroups <= 256 && c->nseg == 0 && !ordered_sums(c) ? 4 : 1;
}
int hydro_waves(const gdf_ctx* c) {
  if (c->nseg > 0 || c->ngroups > 2048 || ordered_sums(c)) return 1;
  return c->ngroups <= 256 ? 4 : 2;
}

int read_flags(gdf_ctx* c) {
  GDF_HIP(c, hipMemcpyAsync(c->h_counters, c->counters, sizeof(int)*8, hipMemcpyDeviceToHost,
                            c->stream));
  GDF_HIP(c, hipStreamSynchronize(c->stream));
  return GDF_OK;
}

void free_cand(CandSet& cs) {
  if (cs.idx) (void) hipFree(cs.idx);
  if (cs.mask) (void) hipFree(cs.mask);
  if (cs.ncand) (void) hipFree(cs.ncand);
  cs.idx = nullptr; cs.mask = nullptr; cs.ncand = nullptr;
  cs.capb = 0; cs.gcap = 0;
}

// (Re)allocate a candidate set for at least ng groups and capb batches; masks: with room for
// the parity tap's masks.
int alloc_cand(gdf_ctx* c, CandSet& cs, int ng, int capb, bool masks) {
  const int gcap = ng <= cs.gcap ? cs.gcap : ng + ng/4 + 64;
  if (cs.idx && gcap == cs.gcap && capb == cs.capb && (cs.mask || !masks)) return GDF_OK;
  GDF_HIP(c, hipStreamSynchronize(c->stream));
  free_cand(cs);
  const size_t n = (size_t) gcap*(size_t) capb*kWave;
  if (hipMalloc(&cs.idx, sizeof(int)*n) != hipSuccess ||
      (masks && hipMalloc(&cs.mask, sizeof(unsigned long long)*n) != hipSuccess) ||
      hipMalloc(&cs.ncand, sizeof(int)*(size_t) gcap) != hipSuccess) {
    free_cand(cs);
    return fail(c, GDF_ERR_NOMEM, "candidate set allocation failed");
  }
  cs.gcap = gcap;
  cs.capb = capb;
  return GDF_OK;
}

int ensure_cand(gdf_ctx* c, CandSet& cs, int ng, bool masks) {
  const int capb = cs.capb > 0 ? cs.capb : c->cfg.cand_batches_init > 0 ? c->cfg.cand_batches_init
                                                                       : kInitBatches;
  return alloc_cand(c, cs, ng, capb, masks);
}

int grow_cand(gdf_ctx* c, CandSet& cs, int ng, int need, bool masks) {
  return alloc_cand(c, cs, ng, std::max(need + need/4 + 1, cs.capb + 1), masks);
}

// The candidate walks of the h-rho pass (gather; uni: with the scatter-gather bounds) and of the
// force pass (scatter-gather); masks: the parity tap's sets.
enum WalkKind { WALK_GATHER, WALK_UNION, WALK_SG, WALK_MASKS };

// glist: the groups holding targets (from group_list), or NULL to walk every group
int launch_walk(gdf_ctx* c, WalkKind kind, int nopbc, CandSet& cs, const int* status,
                const int* glist) {
  CandWalk w;
  const int ng = c->ngroups;
  w.N = c->N; w.ngroups = ng; w.nleaf = c->phys.nleaf; w.capb = cs.capb;
  w.grp_node = c->grp_node; w.grp_first = c->grp_first; w.grp_count = c->grp_count;
  w.lnk = c->lnk;
  w.geo_c = c->geo_c; w.geo_h = c->geo_h;
  w.x = c->pf[F_X]; w.y = c->pf[F_Y]; w.z = c->pf[F_Z];
  w.hcand = kind == WALK_UNION ? c->df[D_HSEARCH] : c->pf[F_H];
  w.htarget = kind == WALK_GATHER || kind == WALK_UNION ? c->df[D_HSEARCH] : c->pf[F_H];
  w.status = status;
  w.grp_root = c->nseg > 0 ? c->grp_root : nullptr;
  w.glist = glist; w.ncap = c->Ncap;
  w.idx = cs.idx; w.mask = cs.mask; w.ncand = cs.ncand;
  w.stacks = c->stacks; w.flags = c->counters;
  w.p = c->phys;
  if (nopbc) w.p.periodic = 0;
  const int grid = std::min(ng, kWalkSlots);
  constexpr int W = kWalkWaves;
  // (lists in the order of a lone wavefront's rounds where the order of the sums counts)
  const bool lone = ordered_sums(c) && kind != WALK_MASKS;
  const int nt = kind == WALK_MASKS || lone ? kWave : kWave*W;
  const bool mixed = c->cfg.precision == GDF_PREC_MIXED;
  hipStream_t st = c->stream;
  if (lone) {
    if (kind == WALK_GATHER && w.p.periodic) k_walk_cand<0, true, 1><<<grid, nt, 0, st>>>(w);
    else if (kind == WALK_GATHER) k_walk_cand<0, false, 1><<<grid, nt, 0, st>>>(w);
    else if (kind == WALK_SG && w.p.periodic) k_walk_cand<1, true, 1><<<grid, nt, 0, st>>>(w);
    else if (kind == WALK_SG) k_walk_cand<1, false, 1><<<grid, nt, 0, st>>>(w);
    else if (w.p.periodic) k_walk_cand<0, true, 1, false, true><<<grid, nt, 0, st>>>(w);
    else k_walk_cand<0, false, 1, false, true><<<grid, nt, 0, st>>>(w);
  } else if (w.p.periodic) {
    if (kind == WALK_GATHER) k_walk_cand<0, true, W><<<grid, nt, 0, st>>>(w);
    else if (kind == WALK_UNION) k_walk_cand<0, true, W, false, true><<<grid, nt, 0, st>>>(w);
    else if (kind == WALK_SG) k_walk_cand<1, true, W><<<grid, nt, 0, st>>>(w);
    else if (mixed) k_walk_cand<2, true, 1, true><<<grid, nt, 0, st>>>(w);
    else k_walk_cand<1, true, 1, true><<<grid, nt, 0, st>>>(w);
  } else {
    if (kind == WALK_GATHER) k_walk_cand<0, false, W><<<grid, nt, 0, st>>>(w);
    else if (kind == WALK_UNION) k_walk_cand<0, false, W, false, true><<<grid, nt, 0, st>>>(w);
    else if (kind == WALK_SG) k_walk_cand<1, false, W><<<grid, nt, 0, st>>>(w);
    else if (mixed) k_walk_cand<2, false, 1, true><<<grid, nt, 0, st>>>(w);
    else k_walk_cand<1, false, 1, true><<<grid, nt, 0, st>>>(w);
  }
  GDF_HIP(c, hipGetLastError());
  return GDF_OK;
}

}  // namespace

int sph_alloc_lists(gdf_ctx* c) {
  GDF_HIP(c, hipMalloc(&c->status, sizeof(int)*(size_t) c->Ncap));
  GDF_HIP(c, hipMalloc(&c->hrecA, sizeof(double4)*(size_t) c->Ncap));
  GDF_HIP(c, hipMalloc(&c->hrecB, sizeof(double4)*(size_t) c->Ncap));
  GDF_HIP(c, hipMalloc(&c->stacks, sizeof(int)*(size_t) kStackSlots*kStackCap));
  GDF_HIP(c, hipMalloc(&c->glist, sizeof(int)*3*((size_t) c->Ncap + 1)));
  if (c->phys.self_gravity && c->phys.hydro_forces && !c->phys.nbody)
    GDF_HIP(c, hipMalloc(&c->stacks2, sizeof(int)*(size_t) kStackSlots*kStackCap));
  return GDF_OK;
}

void sph_free_lists(gdf_ctx* c) {
  free_cand(c->cs_g);
  free_cand(c->cs_s);
  if (c->sg_tgt) (void) hipFree(c->sg_tgt);
  c->sg_tgt = nullptr;
  c->sg_tgt_cap = 0;
  c->sg_tgt_all = true;
  c->sg_tgt_now = false;
}

int sph_density(gdf_ctx* c, int nopbc) {
  const int N = c->N;
  hipStream_t s = c->stream;
  if (!c->tree_valid) return fail(c, GDF_ERR_INVALID, "density pass before tree build");
  GDF_TRY(ensure_cand(c, c->cs_g, c->ngroups, false));
  const int* act = c->nlevels > 1 ? c->pi[I_ACT] : nullptr;
  k_init_density<<<nblocks(N, BS), BS, 0, s>>>(N, c->pf[F_H], c->df[D_HSEARCH], c->status, act,
                                               c->nseg, c->seg_bad);
  DensArgs d;
  d.N = N; d.ngroups = c->ngroups; d.nopbc = nopbc;
  d.grp_node = c->grp_node; d.grp_first = c->grp_first; d.grp_count = c->grp_count;
  d.geo_c = c->geo_c; d.geo_h = c->geo_h;
  d.posm = c->posm;
  d.h = c->pf[F_H]; d.hsearch = c->df[D_HSEARCH]; d.rho = c->df[D_RHO];
  d.invomega = c->df[D_INVOMEGA]; d.zeta = c->df[D_ZETA]; d.hfactor = c->df[D_HFACTOR];
  d.u = c->pf[F_U]; d.sound = c->df[D_SOUND]; d.pressure = c->df[D_PRESSURE];
  d.status = c->status; d.flags = c->counters; d.icount = c->icount;
  d.nstar = c->cfg.conservative_sph_star_gravity ? c->Nstar : 0;
  d.star_soft = c->cfg.nbody_softening;
  d.sx = c->sv[S_X]; d.sy = c->sv[S_Y]; d.sz = c->sv[S_Z]; d.sm = c->sv[S_M]; d.sh = c->sv[S_H];
  d.p = c->phys;
  d.seg = c->pi[I_SEG]; d.seg_bad = c->nseg > 0 ? c->seg_bad : nullptr;
  c->sg_union = c->sg_part = false;
  const bool mixed = c->cfg.precision == GDF_PREC_MIXED;
  d.ordered = ordered_sums(c);
  const int waves = density_waves(c);
  // with periodic images the walk makes the union lists, which the force pass reads if they
  // still bound its set: no search radius may have grown (a retry) or been outgrown, in a batch of
  // several requests none of the request's own
  const bool uni = !nopbc;
  const bool several = c->nseg > 1;
  const WalkKind kind = uni ? WALK_UNION : WALK_GATHER;
  bool grown = false, retried = false, outgrown = false;
  for (int round = 0; round < kMaxRounds; round++) {
    // also clears the round's flags (and, where they are not read any more, the settled groups' lists)
    GDF_TRY(group_list(c, c->status, c->glist, round > 0 && several ? nullptr : c->cs_g.ncand,
                       nullptr, nullptr, c->counters, 4));
    GDF_TRY(launch_walk(c, kind, nopbc, c->cs_g, c->status, c->glist));
    d.capb = c->cs_g.capb; d.idx = c->cs_g.idx; d.ncand = c->cs_g.ncand;
    if (mixed) launch_density<float>(d, waves, s);
    else launch_density<double>(d, waves, s);
    k_hrho_finish<<<nblocks(N, BS), BS, 0, s>>>(d);
    GDF_HIP(c, hipGetLastError());
    GDF_TRY(read_flags(c));
    const int* f = c->h_counters;
    if (f[2]) return fail(c, GDF_ERR_CAPACITY, "tree walk stack overflow in gather pass");
    if (f[3] & 1) return fail(c, GDF_ERR_NOCONV, "Problem with convergence of h-rho iteration");
    if (f[3] & 4) break;
    outgrown = outgrown || (f[3] & 2);
    retried = retried || f[0] > 0;
    // groups whose candidates overflowed skipped the density kernel and keep status 1
    if (f[1] > 0) {
      GDF_TRY(grow_cand(c, c->cs_g, c->ngroups, f[1], false));
      grown = true;
      continue;
    }
    if (f[0] != 0) continue;
    c->sg_valid = false;
    c->sg_union = uni && !retried && !outgrown;
    c->sg_part = uni && !c->sg_union && several;
    if ((c->sg_union || c->sg_part) && grown) {
      // growing dropped the lists of the groups settled before: every group's again (of the
      // requests whose lists are read), as the first round would have made them with room enough
      // (the radii and the nodes' bounds are still those of its start)
      const int* on = act;
      if (c->sg_part) {
        k_seg_status<<<nblocks(N, BS), BS, 0, s>>>(N, c->pi[I_SEG], c->seg_bad, 0, c->status);
        on = c->status;
      }
      if (on) GDF_TRY(group_list(c, on, c->glist, c->cs_g.ncand, nullptr, nullptr,
                                 c->counters, 4));
      else k_zero_ints<<<1, BS, 0, s>>>(4, c->counters);
      GDF_TRY(launch_walk(c, kind, nopbc, c->cs_g, on, on ? c->glist : nullptr));
      GDF_TRY(read_flags(c));
      if (c->h_counters[2]) return fail(c, GDF_ERR_CAPACITY, "tree walk stack overflow in gather pass");
      if (c->h_counters[1] > 0) c->sg_union = c->sg_part = false;
    }
    return tree_refit_h(c);
  }
  return fail(c, GDF_ERR_CAPACITY, "h-rho neighbour search did not settle after 64 rounds");
}

int sph_build_sg(gdf_ctx* c, bool masks) {
  c->sg_from_union = false;
  if (!masks && c->sg_union) {      // the density pass's union lists hold the set
    c->sg_from_union = true;
    c->sg_valid = true;
    c->sg_masks = false;
    return GDF_OK;
  }
  const int ng = c->ngroups;
  GDF_TRY(ensure_cand(c, c->cs_s, ng, masks));
  const int* act = c->nlevels > 1 ? c->pi[I_ACT] : nullptr;
  // the FP64 path's tap after a force pass: that pass's targets, whose flags the step's end clears
  if (masks && act && c->cfg.precision != GDF_PREC_MIXED && c->sg_valid && c->sg_tgt_now) act = c->sg_tgt;
  if (!masks && c->sg_part) {       // the marked requests' groups alone
    k_seg_status<<<nblocks(c->N, BS), BS, 0, c->stream>>>(c->N, c->pi[I_SEG], c->seg_bad, 1, c->status);
    act = c->status;
  }
  for (int round = 0; round < 8; round++) {
    int* sl = c->glist + (c->Ncap + 1);
    if (act) GDF_TRY(group_list(c, act, sl, c->cs_s.ncand, nullptr, nullptr, c->counters, 4));
    else k_zero_ints<<<1, BS, 0, c->stream>>>(4, c->counters);
    GDF_TRY(launch_walk(c, masks ? WALK_MASKS : WALK_SG, 0, c->cs_s, act, act ? sl : nullptr));
    GDF_TRY(read_flags(c));
    if (c->h_counters[2]) return fail(c, GDF_ERR_CAPACITY, "tree walk stack overflow in force pass");
    if (c->h_counters[1] > 0) {
      GDF_TRY(grow_cand(c, c->cs_s, ng, c->h_counters[1], masks));
      continue;
    }
    c->sg_from_union = !masks && c->sg_part;
    c->sg_valid = true;
    c->sg_masks = masks;
    return GDF_OK;
  }
  return fail(c, GDF_ERR_CAPACITY, "scatter-gather candidate capacity");
}

int sph_hydro(gdf_ctx* c, int variant) {
  const int N = c->N;
  hipStream_t s = c->stream;
  if (!c->sg_valid || c->sg_masks) GDF_TRY(sph_build_sg(c));
  const bool blk = c->nlevels > 1;
  // the pass's targets, for the sets it evaluates (its lists cover those alone)
  c->sg_tgt_all = !blk;
  c->sg_tgt_now = blk;
  if (blk && c->sg_tgt_cap < N) {
    if (c->sg_tgt) (void) hipFree(c->sg_tgt);
    c->sg_tgt = nullptr;
    c->sg_tgt_cap = 0;
    GDF_HIP(c, hipMalloc(&c->sg_tgt, sizeof(int)*(size_t) c->Ncap));
    c->sg_tgt_cap = c->Ncap;
  }
  k_pack_hydro<<<nblocks(N, BS), BS, 0, s>>>(N, c->pf[F_VX], c->pf[F_VY], c->pf[F_VZ],
                                             c->pf[F_H], c->df[D_RHO], c->df[D_PRESSURE],
                                             c->df[D_INVOMEGA], c->df[D_SOUND],
                                             c->df[D_HFACTOR], c->hrecA, c->hrecB,
                                             c->pi[I_ACT], blk ? c->sg_tgt : nullptr);
  HydroArgs h;
  const CandSet& cs = c->sg_from_union ? c->cs_g : c->cs_s;
  h.N = N; h.ngroups = c->ngroups; h.capb = cs.capb;
  h.grp_node = c->grp_node; h.grp_first = c->grp_first; h.grp_count = c->grp_count;
  h.geo_c = c->geo_c; h.geo_h = c->geo_h;
  h.idx = cs.idx; h.ncand = cs.ncand;
  const bool part = c->sg_from_union && c->sg_part;
  h.capb2 = c->cs_s.capb; h.idx2 = c->cs_s.idx; h.ncand2 = part ? c->cs_s.ncand : nullptr;
  h.posm = c->posm; h.A = c->hrecA; h.B = c->hrecB; h.h = c->pf[F_H];
  h.invomega = c->df[D_INVOMEGA]; h.pressure = c->df[D_PRESSURE]; h.zeta = c->df[D_ZETA];
  h.ax = c->df[D_AX]; h.ay = c->df[D_AY]; h.az = c->df[D_AZ];
  h.gx = c->df[D_ATX]; h.gy = c->df[D_ATY]; h.gz = c->df[D_ATZ]; h.gpot = c->df[D_GPOT];
  h.dudt = c->df[D_DUDT]; h.div_v = c->df[D_DIVV]; h.p = c->phys;
  h.icount = c->icount;
  h.act = c->pi[I_ACT]; h.level = c->pi[I_LEVEL]; h.levelneib = c->pi[I_LEVELNEIB];
  const bool mixed = c->cfg.precision == GDF_PREC_MIXED;
  const int kt = ktime_begin(c, s, 6);
  if (mixed) launch_hydro<float>(h, variant, blk, hydro_waves(c), s);
  else launch_hydro<double>(h, variant, blk, hydro_waves(c), s);
  GDF_HIP(c, hipGetLastError());
  ktime_end(c, s, kt);
  return GDF_OK;
}

int sph_copy_sg(gdf_ctx* c, std::vector<int>& idx, std::vector<unsigned long long>& mask,
                std::vector<int>& ncand, int& capb) {
  // the force passes leave no masks: the set is walked again with them (same tests)
  if (!c->sg_valid || !c->sg_masks) GDF_TRY(sph_build_sg(c, true));
  GDF_HIP(c, hipStreamSynchronize(c->stream));
  const CandSet& cs = c->cs_s;
  const size_t n = (size_t) c->ngroups*(size_t) cs.capb*kWave;
  idx.resize(n); mask.resize(n); ncand.resize(c->ngroups);
  capb = cs.capb;
  GDF_HIP(c, hipMemcpy(idx.data(), cs.idx, sizeof(int)*n, hipMemcpyDeviceToHost));
  GDF_HIP(c, hipMemcpy(mask.data(), cs.mask, sizeof(unsigned long long)*n, hipMemcpyDeviceToHost));
  GDF_HIP(c, hipMemcpy(ncand.data(), cs.ncand, sizeof(int)*c->ngroups, hipMemcpyDeviceToHost));
  return GDF_OK;
}

}  // namespace gdf
