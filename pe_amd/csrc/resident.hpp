// Sweeps of up to one workgroup's contacts with everything they touch on the chip, for the relaxation models
// without a search: one lane holds one contact's record, its bodies' records and its impulse in registers for
// all sweeps, the bodies' velocity corrections are in LDS, and a sweep is one workgroup barrier per colour.
// Shared by the batched and the single-world kernels.
//
// What bounds it is the latency of a colour, about 2k cycles, most of it a lane's relaxation.  The records
// read from memory at every visit, as the sweeps over global arrays do, cost 6k to 8k cycles a colour more,
// most of it two dependent round trips.
#pragma once

#include "step_ops.hpp"

namespace pe_amd {

constexpr uint32_t kResidentThreads = 256;                     // contacts a workgroup can hold
constexpr uint32_t kResidentBodies = 2 * kResidentThreads;     // their non-fixed bodies
// ... and a workgroup that reads the bodies' records at every visit
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

// One contact's relaxation (no other thread may touch its bodies meanwhile).  Returns its impulse change.
template <int MODEL, class Trig, bool HOLD>
__device__ __forceinline__ double resident_relax(ResidentContact<HOLD>& r, double* dvw, int maxSub) {
  static_assert(MODEL != 3 && MODEL != 5, "a lane's search takes four times a wavefront's");
  d3 dv1, dw1, dv2, dw2;
  lds_dvw(dvw, r.l1, dv1, dw1);
  lds_dvw(dvw, r.l2, dv2, dw2);
  double delta;
  if constexpr (HOLD)
    delta = relax_update<MODEL, Trig, 0>(r.cf, r.b.b1, r.b.b2, dv1, dw1, dv2, dw2, r.p, maxSub);
  else
    delta = relax_update<MODEL, Trig, 0>(r.cf, relax_body(r.b.s1), relax_body(r.b.s2), dv1, dw1, dv2, dw2, r.p, maxSub);
  lds_dvw_store(dvw, r.l1, dv1, dw1);
  lds_dvw_store(dvw, r.l2, dv2, dw2);
  return delta;
}

}  // namespace pe_amd
