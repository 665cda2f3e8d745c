// Candidate filter of the SPH pair passes: which of a batch of 64 candidates can lie inside the
// range of which of a walk group's 64 targets, on the matrix cores.
//
// The squared distances of 64 x 64 (candidate, target) pairs minus the squared range are a
// product of six-element feature vectors,
//   |c - r|^2 - R^2 = x (-2 rx) + y (-2 ry) + z (-2 rz) + |c|^2 1 + 1 (|r|^2 - R_i^2),
// so v_mfma_f32_32x32x2_f32 forms them and only the sign bits are kept: one v_alignbit per 64
// pairs, against eleven vector instructions for a test written out per pair.  The result is a
// superset of the pairs inside the range (the thresholds are widened by the rounding of the
// expanded form); the pair loops decide each pair themselves.
//
// The features are single precision in the group's frame, scaled by a power of two so that the
// group's extent plus its largest search range is below one: the error bounds below are then
// independent of the units.
#pragma once

#include <hip/hip_runtime.h>

#include "gdf_device.h"

namespace gdf {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// Rounding of the expanded form: the features carry 2^-24 of their size (at most 1 + R for a
// candidate whose own range R reaches the group), which moves the squared distance by at most
// 4e-7 (1 + R)^2, and the products and sums of the six terms round to within 1e-6 (1 + R)^2.
constexpr float kFilterSlack = 8.0e-6f;
constexpr float kFilterFar = 1.0e30f;     // |c|^2 of an empty slot (and, negated, of a sure hit)

// power of two that brings the length `ext` (> 0) below one; T: the precision of the frame, so that
// FP64 lengths outside the range of single precision are scaled before they are rounded to it
template <typename T> __device__ __forceinline__ T filter_scale(double ext) {
  constexpr int most = sizeof(T) == 8 ? 1000 : 120;
  int e;
  (void) frexp(ext, &e);
  return (T) ldexp(1.0, max(-most, min(most, -e)));
}

// One candidate's features: scaled position and the square of its own scaled range (widened;
// read by the scatter-gather filter only).  state: 0 a candidate, 1 an empty slot, -1 a
// candidate that every target is to take.
struct FiltCand { float x, y, z, thr; int state; };

__device__ __forceinline__ float filter_thr(float r2) {
  const float m = 1.f + sqrt_f(r2);
  return fmaf(kFilterSlack*m, m, r2);
}

// The targets' side, one target per lane, spread as the B operands of two blocks of 32 targets:
// lanes 0-31 hold the even feature of their column, lanes 32-63 the odd one.
struct FiltTargets {
  float xy[2], z1[2], base[2], rr[2];
  __device__ __forceinline__ static float at(float lo, float hi, int tb) {
    const int lane = lane_id(), src = 32*tb + (lane & 31);
    const float a = __shfl(lo, src, 64), b = __shfl(hi, src, 64);
    return lane < 32 ? a : b;
  }
  // rx, ry, rz: the lane's target in the scaled frame
  __device__ __forceinline__ void position(float rx, float ry, float rz) {
    #pragma unroll
    for (int tb = 0; tb < 2; tb++) {
      xy[tb] = at(-2.f*rx, -2.f*ry, tb);
      z1[tb] = at(-2.f*rz, 1.f, tb);
      rr[tb] = at(dot3_f(rx, ry, rz), 1.f, tb);
    }
  }
  // r2: the squared scaled range (widened here); a negative r2 takes no candidate
  __device__ __forceinline__ void range(float rx, float ry, float rz, float r2) {
    const float b = r2 < 0.f ? kFilterFar : dot3_f(rx, ry, rz) - (r2 + kFilterSlack);
    #pragma unroll
    for (int tb = 0; tb < 2; tb++) base[tb] = at(b, 0.f, tb);
  }
};

// 64 slots against 64 targets: bit p of word h says that slot 32 h + p can lie inside the lane's
// target's range (or, SG, its own range reaches the target).  cand(slot) gives a slot's
// features.  D = A B: A's rows are slots, in the order that puts row r of block cb into the bit
// the sign extraction below leaves it in; B's columns are targets.  Lane l of a 32x32 product
// holds column l % 32 and, for l / 32 = h, the rows 8 (v / 4) + 4 h + v % 4 of its 16 registers.
template <bool SG, class F>
__device__ __forceinline__ uint2 filter64(const FiltTargets& t, F cand) {
  const int lane = lane_id(), row = lane & 31;
  const bool hi = lane >= 32;
  const int slot = 32*((row >> 2) & 1) + 15 - (4*(row >> 3) + (row & 3));
  unsigned w0 = 0, w1 = 0;
  #pragma unroll
  for (int cb = 0; cb < 2; cb++) {
    const FiltCand c = cand(slot + 16*(1 - cb));
    float q = dot3_f(c.x, c.y, c.z);
    float x = c.x, y = c.y, z = c.z, thr = c.thr;
    if (c.state != 0) {
      x = y = z = thr = 0.f;
      q = c.state > 0 ? kFilterFar : -kFilterFar;
    }
    const float axy = hi ? y : x, az1 = hi ? q : z;
    #pragma unroll
    for (int tb = 0; tb < 2; tb++) {
      f32x16 d = {};
      d = __builtin_amdgcn_mfma_f32_32x32x2f32(axy, t.xy[tb], d, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_32x32x2f32(az1, t.z1[tb], d, 0, 0, 0);
      const f32x16 own = __builtin_amdgcn_mfma_f32_32x32x2f32(hi ? 0.f : 1.f, t.base[tb], d, 0, 0, 0);
      if (SG) d = __builtin_amdgcn_mfma_f32_32x32x2f32(hi ? -thr : 1.f, t.rr[tb], d, 0, 0, 0);
      unsigned w = tb ? w1 : w0;
      #pragma unroll
      for (int v = 0; v < 16; v++) {
        unsigned b = __float_as_uint(own[v]);
        if (SG) b |= __float_as_uint(d[v]);
        w = __builtin_amdgcn_alignbit(w, b, 31);       // w = 2 w + sign
      }
      if (tb) w1 = w; else w0 = w;
      __builtin_amdgcn_sched_barrier(0);      // one product's registers at a time
    }
  }
  // lanes 0-31 hold targets 0-31 in w0 and 32-63 in w1 (rows of half 0), lanes 32-63 the same
  // targets (rows of half 1): swapped so that every lane holds both halves of its own target
  const auto s = __builtin_amdgcn_permlane32_swap(w0, w1, false, false);
  return make_uint2(s[0], s[1]);
}

// LDS traffic within one wavefront: the hardware keeps it in order, the compiler must too
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// ---- a pair pass's work items ----
// A workgroup takes one walk group, one lane a target; its W wavefronts share the group's
// candidates (wavefront w takes candidates w, w + W, ...), their sums added in that order at the
// end.  Every wavefront stages its own candidates, so the candidate loop has no barriers.

// A wavefront's candidates in nb batches of up to 64, one a lane: lane l of batch b stages the
// wavefront's candidate b + nb l, so that every batch samples the whole list and each target's
// neighbours spread evenly over the batches.
struct PairBatches {
  int nw, nb;
  __device__ __forceinline__ PairBatches(int n) : nw(n), nb((n + kWave - 1)/kWave) {}
  __device__ __forceinline__ int count(int b) const { return (nw - b + nb - 1)/nb; }
  __device__ __forceinline__ bool filled(int b, int l) const { return b < nb && b + nb*l < nw; }
  __device__ __forceinline__ int index(int b, int l) const { return b + nb*l; }
};

// The hits of a lane in the two batches held in LDS (slots 64 (b & 1) + l of batch b), as four
// words of 32 slots in registers, taken one at a time.  A lane that has taken its hits of the
// older batch goes on with the newer one while others are still in the older, which is replaced
// once every lane is through it: a wavefront's trips follow the lanes' totals, which are alike,
// rather than the busiest lane of each batch.
constexpr int kPairSlots = 2*kWave;
struct HitQueue {
  unsigned cur = 0, n0 = 0, n1 = 0, n2 = 0;      // the word being taken and the rem after it
  int rem = 0, base = 0;                         // base: slot of bit 0 of cur
  int done = 0, staged = 0, older = 0;           // hits taken; staged, and without the newest
  bool take = false;
  // the next batch's words (bit p of word h: slot 32 h + p); the batch it replaces is all taken
  __device__ __forceinline__ void stage(bool first, uint2 w) {
    older = staged;
    staged += __popc(w.x) + __popc(w.y);
    if (first) { cur = w.x; n0 = w.y; rem = 1; return; }
    if (rem > 1) {              // at a word of the replaced batch, taken: on to the kept one's first
      const bool far = rem == 3;
      cur = far ? n1 : n0;
      n0 = far ? n2 : n1;
      base = (base + (far ? 64 : 32)) & (kPairSlots - 1);
      rem = 1;
    }
    n0 = rem ? n0 : w.x;
    n1 = rem ? w.x : w.y;
    n2 = w.y;
    rem += 2;
  }
  __device__ __forceinline__ int pop() {
    if (cur == 0 && rem > 0) {
      cur = n0; n0 = n1; n1 = n2;
      rem--;
      base = (base + 32) & (kPairSlots - 1);
    }
    take = cur != 0;
    const int slot = take ? base + __builtin_ctz(cur) : 0;
    cur &= cur - 1;
    return slot;
  }
  // pair(record, take) until every lane has taken `need` hits; rec: the record of the hit popped
  // last, read while the one before it is evaluated.  Every lane runs every trip (no execution
  // mask changes): with !take the record is slot 0's.  The test stands at the loop's end: with it
  // at the head the compiler kept the sums before and after a pair apart, 32 of a hydro trip's
  // 204 vector instructions more (1M particles, quintic, FP32: 9.34 against 9.09 ms a
  // force evaluation; FP64 11.57 against 11.33).
  template <class R, class L, class P>
  __device__ __forceinline__ void run(int need, R& rec, L load, P pair) {
    if (!take) rec = load(pop());
    if (!__ballot(done < need)) return;
    do {
      const bool now = take;
      const R next = load(pop());
      pair(rec, now);
      done += now;
      rec = next;
    } while (__ballot(done < need));
  }
};

}  // namespace gdf
