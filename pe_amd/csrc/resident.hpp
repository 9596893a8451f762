// Sweeps of up to one workgroup's contacts with everything they touch on the chip: one lane holds one
// contact's record, its bodies' records and its impulse in registers for all sweeps, the bodies' velocity
// corrections are in LDS, and a sweep is one workgroup barrier per colour.  Shared by the batched and the
// single-world kernels.
//
// What bounds it is the latency of a colour: a lane's relaxation (about 1k cycles) and, for the models
// with a search, the sliding contacts, which a wavefront relaxes one after the other as a whole (three
// thousand cycles a search instead of a lane's twelve).  The records read from memory at every visit, as
// the sweeps over global arrays do, cost 6k to 8k cycles a colour more, most of it two dependent round
// trips.
#pragma once

#include "step_ops.hpp"

namespace pe_amd {

constexpr uint32_t kResidentThreads = 256;                     // contacts a workgroup can hold
constexpr uint32_t kResidentBodies = 2 * kResidentThreads;     // their non-fixed bodies
// ... and a workgroup of models without a search that reads the bodies' records at every visit
constexpr uint32_t kResidentWide = 768;
constexpr uint32_t kNoBody = 0xFFFFFFFFu;

// A contact's fields held in registers (a reader for relax_update).
struct HeldFields {
  double v[CF_COUNT];
  __device__ __forceinline__ double operator()(int k) const { return v[k]; }
};

// HOLD: the bodies' records in registers too (else they are read from s1, s2 at every visit).
template <bool HOLD>
struct ResidentBodies {
  RelaxBody b1, b2;
};
template <>
struct ResidentBodies<false> {
  const double *s1, *s2;
};
template <bool HOLD = true>
struct ResidentContact {
  HeldFields cf;
  ResidentBodies<HOLD> b;
  uint32_t l1, l2;     // the bodies' places in LDS, kNoBody for fixed ones
  d3 p;
};

// Slot s of C; local(body) is a non-fixed body's place in LDS.
template <bool HOLD, class Local>
__device__ __forceinline__ void resident_load(ResidentContact<HOLD>& r, const SolverContacts& C, size_t s, const double* sb,
                                              const Local& local) {
#pragma unroll
  for (int k = 0; k < CF_COUNT; ++k) r.cf.v[k] = C.f[(size_t)k * C.cap + s];
  const uint32_t e1 = C.b1[s], e2 = C.b2[s];
  const uint32_t i1 = e1 & ~kFixedBit, i2 = e2 & ~kFixedBit;
  if constexpr (HOLD) {
    r.b.b1 = relax_body(sb + (size_t)kSB * i1);
    r.b.b2 = relax_body(sb + (size_t)kSB * i2);
  } else {
    r.b.s1 = sb + (size_t)kSB * i1;
    r.b.s2 = sb + (size_t)kSB * i2;
  }
  r.l1 = (e1 & kFixedBit) ? kNoBody : local(i1);
  r.l2 = (e2 & kFixedBit) ? kNoBody : local(i2);
  r.p = mk3(r.cf.v[CF_P], r.cf.v[CF_P + 1], r.cf.v[CF_P + 2]);
}

// A body's velocity corrections in LDS (six doubles).
__device__ __forceinline__ void lds_dvw(const double* dvw, uint32_t l, d3& dv, d3& dw) {
  dv = dw = mk3(0, 0, 0);
  if (l != kNoBody) {
    const double* q = dvw + 6 * l;
    dv = mk3(q[0], q[1], q[2]);
    dw = mk3(q[3], q[4], q[5]);
  }
}
__device__ __forceinline__ void lds_dvw_store(double* dvw, uint32_t l, d3 dv, d3 dw) {
  if (l != kNoBody) {
    double* q = dvw + 6 * l;
    q[0] = dv.x; q[1] = dv.y; q[2] = dv.z;
    q[3] = dw.x; q[4] = dw.y; q[5] = dw.z;
  }
}

__device__ __forceinline__ d3 wave_read_lane3(d3 x, int lane) {
  return mk3(wave_read_lane(x.x, lane), wave_read_lane(x.y, lane), wave_read_lane(x.z, lane));
}
__device__ __forceinline__ RelaxBody wave_read_body(const RelaxBody& b, int lane) {
  RelaxBody o;
  o.v = wave_read_lane3(b.v, lane);
  o.w = wave_read_lane3(b.w, lane);
  o.im = wave_read_lane(b.im, lane);
#pragma unroll
  for (int k = 0; k < 9; ++k) o.I.a[k] = wave_read_lane(b.I.a[k], lane);
  return o;
}

// The lanes with `mine` relax their contacts, which share no non-fixed body (one colour).  Called by whole
// wavefronts.  Returns the lane's impulse change (0 without one).
template <int MODEL, class Trig, bool HOLD>
__device__ __forceinline__ double resident_relax(ResidentContact<HOLD>& r, bool mine, double* dvw, int maxSub) {
  constexpr bool kSearches = MODEL == 3 || MODEL == 5;
  static_assert(HOLD || !kSearches, "a wavefront's search takes the bodies' records from the lane's registers");
  double delta = 0.0;
  bool slides = false;
  if (mine) {
    d3 dv1, dw1, dv2, dw2, p = r.p;
    lds_dvw(dvw, r.l1, dv1, dw1);
    lds_dvw(dvw, r.l2, dv2, dw2);
    if constexpr (HOLD)
      delta = relax_update<MODEL, Trig, 0, kSearches>(r.cf, r.b.b1, r.b.b2, dv1, dw1, dv2, dw2, p, maxSub);
    else
      delta = relax_update<MODEL, Trig, 0>(r.cf, relax_body(r.b.s1), relax_body(r.b.s2), dv1, dw1, dv2, dw2, p, maxSub);
    slides = kSearches && delta == kDeferred;
    if (!slides) {
      r.p = p;
      lds_dvw_store(dvw, r.l1, dv1, dw1);
      lds_dvw_store(dvw, r.l2, dv2, dw2);
    } else {
      delta = 0.0;
    }
  }
  if constexpr (kSearches) {
    const int lane = (int)(threadIdx.x & 63u);
    unsigned long long left = __ballot(slides);
    while (left) {
      const int l = __builtin_amdgcn_readfirstlane(__builtin_ctzll(left));
      left &= left - 1ull;
      HeldFields cf;
#pragma unroll
      for (int k = 0; k < CF_COUNT; ++k) cf.v[k] = wave_read_lane(r.cf.v[k], l);
      const RelaxBody b1 = wave_read_body(r.b.b1, l), b2 = wave_read_body(r.b.b2, l);
      const uint32_t l1 = (uint32_t)__builtin_amdgcn_readlane((int)r.l1, l);
      const uint32_t l2 = (uint32_t)__builtin_amdgcn_readlane((int)r.l2, l);
      d3 p = wave_read_lane3(r.p, l);
      d3 dv1, dw1, dv2, dw2;
      lds_dvw(dvw, l1, dv1, dw1);
      lds_dvw(dvw, l2, dv2, dw2);
      const double d = relax_update<MODEL, Trig, 6>(cf, b1, b2, dv1, dw1, dv2, dw2, p, maxSub);
      if (lane == l) {
        r.p = p;
        delta = d;
        lds_dvw_store(dvw, l1, dv1, dw1);
        lds_dvw_store(dvw, l2, dv2, dw2);
      }
    }
  }
  return delta;
}

}  // namespace pe_amd
