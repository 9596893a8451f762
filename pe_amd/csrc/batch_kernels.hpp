// Batched scenes: one workgroup advances one scene through whole time steps, and a
// persistent grid of workgroups pulls scenes from a queue (largest first).  Per scene
// and step, as CollisionSystem<HCSITS>::simulationStep (HCSITS.h:1472-1531):
//   detection    counting sort of the grid bodies into an LDS bucket table (one periodic
//                grid level whose cell edge bounds every AABB), 27-bucket neighbourhood
//                and plane tests, narrowphase -- every pair that is not both fixed and
//                whose closed AABBs overlap is handed to the narrowphase once
//                (HashGrids.h:1121-1358 semantics); count pass, scan, write pass, so the
//                contact order is deterministic;
//   body caching predicted velocities and solver body records;
//   colouring    Jones-Plassmann rounds with LDS claims (a contact whose priority is the
//                smallest among the uncoloured contacts of both its non-fixed bodies takes
//                the round's colour), then a stable colour-major ordering;
//   caching      contact records in sweep order (HCSITS.h:1741-1818);
//   sweeps       K sweeps, one workgroup barrier per colour (HCSITS.h:1891-1947);
//   integration  HCSITS.h:1954-2004, 4135-4184.
// Colours, sweep order and results do not depend on the workgroup size or grid.
#pragma once

#include "batch.hpp"
#include "resident.hpp"
#include "step_ops.hpp"

namespace pe_amd {

namespace {

constexpr uint32_t kEmptyKey = 0xFFFFFFFFu;
constexpr double kBatchSpanFill = 0.999999;
// LDS for the velocity corrections of the bodies (two a contact) of as many contacts as threads; for 64 threads
// it is taken from tab's end.
constexpr uint32_t batch_ldvw_bytes(uint32_t threads) { return 2 * threads * 6 * (uint32_t)sizeof(double); }
constexpr uint32_t kBatchTailFree = kBatchTable - batch_ldvw_bytes(64) / 4;
static_assert(kBatchTailFree % 2 == 0, "the corrections are aligned");
static_assert(kBatchWideThreads == kResidentThreads, "a workgroup holds a contact a thread");

// Inclusive/exclusive scan of one value per thread over the workgroup (blockDim.x a
// multiple of 64, at most 512).  red needs 8 words.
__device__ __forceinline__ uint32_t wg_exclusive_scan(uint32_t x, uint32_t* red, uint32_t* total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  uint32_t v = x;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t t = __shfl_up(v, d, 64);
    if (lane >= d) v += t;
  }
  if (lane == 63) red[wid] = v;
  __syncthreads();
  uint32_t pre = 0, tot = 0;
  for (int k = 0; k < nw; ++k) {
    const uint32_t s = red[k];
    if (k < wid) pre += s;
    tot += s;
  }
  __syncthreads();
  *total = tot;
  return v - x + pre;
}

__device__ __forceinline__ uint32_t wg_sum(uint32_t x, uint32_t* red) {
  uint32_t tot;
  wg_exclusive_scan(x, red, &tot);
  return tot;
}

// Workgroup max of non-negative doubles (wavefront shuffles, then one LDS word per wave).
__device__ __forceinline__ double wg_max(double x, unsigned long long* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  unsigned long long u = (unsigned long long)__double_as_longlong(x);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const unsigned long long o = __shfl_xor(u, d, 64);
    u = o > u ? o : u;
  }
  if (lane == 0) red[wid] = u;
  __syncthreads();
  unsigned long long m = 0;
  for (int k = 0; k < nw; ++k) m = red[k] > m ? red[k] : m;
  __syncthreads();
  return __longlong_as_double((long long)m);
}

// Bijective mix of a contact's scene-local index: distinct, well-spread colouring priorities.
__device__ __forceinline__ uint32_t colour_priority(uint32_t c) {
  uint32_t h = c * 0x9E3779B1u;
  h ^= h >> 16;
  h *= 0x85EBCA6Bu;
  h ^= h >> 13;
  return h;
}

struct SceneCountEmit {
  uint32_t n = 0;
  __device__ void operator()(uint32_t, uint32_t, d3, d3, double) { ++n; }
};

struct SceneWriteEmit {
  const Bodies* B;
  const RawContacts* R;
  const BatchArgs* A;
  const SceneInfo* S;
  uint32_t at;
  __device__ void operator()(uint32_t b1, uint32_t b2, d3 gpos, d3 n, double dist) {
    double mu;
    if (A->scene_mu) mu = contact_is_dynamic(*B, b1, b2, gpos, n) ? S->mu_d : S->mu_s;
    else mu = contact_friction(*B, A->csf, A->cdf, A->nmat, b1, b2, gpos, n);
    R->b1[at] = b1;
    R->b2[at] = b2;
    st3(R->pos, at, gpos);
    st3(R->nrm, at, n);
    R->dist[at] = dist;
    R->mu[at] = mu;
    ++at;
  }
};

__device__ __forceinline__ uint32_t scene_bucket(const SceneInfo& S, const double* a) {
  const long long cx = (long long)floor(a[0] * S.inv);
  const long long cy = (long long)floor(a[1] * S.inv);
  const long long cz = (long long)floor(a[2] * S.inv);
  const uint32_t mx = (1u << S.lx) - 1, my = (1u << S.ly) - 1, mz = (1u << S.lz) - 1;
  return (((uint32_t)cz & mz) << (S.lx + S.ly)) | (((uint32_t)cy & my) << S.lx) | ((uint32_t)cx & mx);
}

// Pairs of grid body a (same rules as the single-world broadphase): bodies of the 27
// neighbouring buckets with a larger index, then the scene's planes.
template <class Emit>
__device__ void scene_pairs(const Bodies& B, const BatchArgs& A, const SceneInfo& S, const uint32_t* tab,
                            uint32_t a, Emit& emit) {
  const double* aa = B.aabb + 6 * (size_t)a;
  double abox[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) abox[k] = aa[k];
  const bool fa = B.fixed[a] != 0;
  const long long cx = (long long)floor(abox[0] * S.inv);
  const long long cy = (long long)floor(abox[1] * S.inv);
  const long long cz = (long long)floor(abox[2] * S.inv);
  const uint32_t mx = (1u << S.lx) - 1, my = (1u << S.ly) - 1, mz = (1u << S.lz) - 1;
  for (int dz = -1; dz <= 1; ++dz)
    for (int dy = -1; dy <= 1; ++dy)
      for (int dx = -1; dx <= 1; ++dx) {
        const uint32_t key = (((uint32_t)(cz + dz) & mz) << (S.lx + S.ly)) |
                             (((uint32_t)(cy + dy) & my) << S.lx) | ((uint32_t)(cx + dx) & mx);
        const uint32_t st = tab[key], en = tab[key + 1];
        for (uint32_t t = st; t < en; ++t) {
          const uint32_t b = A.sorted[S.body0 + t];
          if (b <= a) continue;
          if (fa && B.fixed[b]) continue;
          if (!aabb_overlap(abox, B.aabb + 6 * (size_t)b)) continue;
          narrowphase(B, a, b, emit);
        }
      }
  if (fa) return;  // planes are fixed
  for (uint32_t k = 0; k < S.nplane; ++k) {
    const uint32_t p = A.plane_idx[S.plane0 + k];
    if (!aabb_overlap(abox, B.aabb + 6 * (size_t)p)) continue;
    narrowphase(B, a, p, emit);
  }
}

// A sliding contact by one lane: a function of its own, so that its search does not stand beside the
// wavefront's in the kernel's registers.
template <int MODEL, class Trig>
__device__ __attribute__((noinline)) double relax_slide_lane(const SolverContacts& C, uint32_t i, const double* sb,
                                                             double* dvw, double dtinv, int max_sub) {
  return relax_contact<MODEL, Trig>(C, i, sb, dvw, dtinv, max_sub);
}

// One time step of scene sc.  Returns false (uniformly) if the scene hit an error; its
// flags are then set and it does not advance.
template <int MODEL, class Trig, bool WIDE>
__device__ bool scene_step(const Bodies& B, const RawContacts& R, const SolverContacts& C, const BatchArgs& A,
                           const SceneInfo& S, uint32_t sc, uint32_t* tab, uint32_t* coff, uint32_t* red,
                           unsigned long long* red64, uint32_t* lflag, double* ldvw) {
  const uint32_t T = blockDim.x, tid = threadIdx.x;
  const uint32_t b0 = S.body0, b1 = S.body0 + S.nbody;
  const uint32_t table = 1u << (S.lx + S.ly + S.lz);
  SceneOut& O = A.out[sc];

  // ---- detection: bucket counts
  for (uint32_t t = tid; t <= table; t += T) tab[t] = 0;
  if (tid == 0) {
    *lflag = 0;
    O.counters[0] = 0;
    O.counters[1] = 0;
  }
  __syncthreads();
  uint32_t ngrid_local = 0;
  for (uint32_t i = b0 + tid; i < b1; i += T) {
    if (B.shape[i] == kShapePlane) { A.bucket[i] = kEmptyKey; continue; }
    const double* a = B.aabb + 6 * (size_t)i;
    const double size = aabb_size(a);
    bool finite = true;
#pragma unroll
    for (int k = 0; k < 6; ++k) finite = finite && isfinite(a[k]);
    if (!finite) { atomicOr(lflag, ERR_NONFINITE); A.bucket[i] = kEmptyKey; continue; }
    if (size > S.span * kBatchSpanFill) atomicOr(lflag, ERR_LEVEL_OVERFLOW);
    const uint32_t key = scene_bucket(S, a);
    A.bucket[i] = key;
    atomicAdd(&tab[key], 1u);
    ++ngrid_local;
  }
  const uint32_t ngrid = wg_sum(ngrid_local, red);  // (barriers inside)
  if (*lflag) {
    if (tid == 0) { O.flags |= *lflag; atomicOr(A.any_flags, *lflag); }
    return false;
  }
  // inclusive bucket ends, each thread a contiguous run of the table
  {
    const uint32_t per = (table + T - 1) / T;
    const uint32_t lo = tid * per, hi = min(lo + per, table);
    uint32_t sum = 0;
    for (uint32_t t = lo; t < hi; ++t) sum += tab[t];
    uint32_t tot;
    uint32_t run = wg_exclusive_scan(sum, red, &tot);
    for (uint32_t t = lo; t < hi; ++t) {
      run += tab[t];
      tab[t] = run;
    }
  }
  __syncthreads();
  for (uint32_t i = b0 + tid; i < b1; i += T) {
    const uint32_t key = A.bucket[i];
    if (key == kEmptyKey) continue;
    const uint32_t pos = atomicSub(&tab[key], 1u) - 1u;
    A.sorted[b0 + pos] = i;
  }
  if (tid == 0) tab[table] = ngrid;
  __syncthreads();
  // bucket lists in body order (the placement above is in arrival order)
  for (uint32_t t = tid; t < table; t += T) {
    const uint32_t st = tab[t], en = tab[t + 1];
    for (uint32_t x = st + 1; x < en; ++x) {
      const uint32_t v = A.sorted[b0 + x];
      uint32_t y = x;
      while (y > st && A.sorted[b0 + y - 1] > v) {
        A.sorted[b0 + y] = A.sorted[b0 + y - 1];
        --y;
      }
      A.sorted[b0 + y] = v;
    }
  }
  __syncthreads();

  // ---- detection: count, scan, write
  for (uint32_t i = b0 + tid; i < b1; i += T) {
    uint32_t n = 0;
    if (A.bucket[i] != kEmptyKey) {
      SceneCountEmit e;
      scene_pairs(B, A, S, tab, i, e);
      n = e.n;
    }
    A.count[i] = n;
  }
  __syncthreads();
  uint32_t nc = 0;
  for (uint32_t base = b0; base < b1; base += T) {
    const uint32_t i = base + tid;
    const uint32_t x = i < b1 ? A.count[i] : 0u;
    uint32_t tot;
    const uint32_t ex = wg_exclusive_scan(x, red, &tot);
    if (i < b1) A.count[i] = nc + ex;
    nc += tot;
  }
  if (nc > S.ccap) {
    if (tid == 0) { O.flags |= ERR_CAPACITY; atomicOr(A.any_flags, ERR_CAPACITY); }
    return false;
  }
  for (uint32_t i = b0 + tid; i < b1; i += T) {
    if (A.bucket[i] == kEmptyKey) continue;
    SceneWriteEmit e{&B, &R, &A, &S, S.c0 + A.count[i]};
    scene_pairs(B, A, S, tab, i, e);
  }
  // ---- body caching
  for (uint32_t i = b0 + tid; i < b1; i += T) predict_body(B, i, A.gravity, A.dt);
  __syncthreads();

  // ---- colouring (claims in LDS, indexed by the scene-local body)
  const uint32_t c0 = S.c0;
  for (uint32_t c = tid; c < nc; c += T) A.colour[c0 + c] = kUncoloured;
  uint32_t ncol = 0;
  for (;;) {
    for (uint32_t i = tid; i < S.nbody; i += T) tab[i] = 0xFFFFFFFFu;
    __syncthreads();
    for (uint32_t c = tid; c < nc; c += T) {
      if (A.colour[c0 + c] != kUncoloured) continue;
      const uint32_t p = colour_priority(c);
      const uint32_t e1 = R.b1[c0 + c], e2 = R.b2[c0 + c];
      if (!B.fixed[e1]) atomicMin(&tab[e1 - b0], p);
      if (!B.fixed[e2]) atomicMin(&tab[e2 - b0], p);
    }
    __syncthreads();
    uint32_t left = 0;
    for (uint32_t c = tid; c < nc; c += T) {
      if (A.colour[c0 + c] != kUncoloured) continue;
      const uint32_t p = colour_priority(c);
      const uint32_t e1 = R.b1[c0 + c], e2 = R.b2[c0 + c];
      const bool win = (B.fixed[e1] || tab[e1 - b0] == p) && (B.fixed[e2] || tab[e2 - b0] == p);
      if (win) A.colour[c0 + c] = ncol;
      else ++left;
    }
    ++ncol;
    const uint32_t remaining = wg_sum(left, red);
    if (remaining == 0) break;
    if (ncol >= kMaxColours) {
      if (tid == 0) { O.flags |= ERR_COLOURS; atomicOr(A.any_flags, ERR_COLOURS); }
      return false;
    }
  }
  if (nc == 0) ncol = 0;
  // colour offsets
  for (uint32_t k = tid; k <= kMaxColours; k += T) coff[k] = 0;
  __syncthreads();
  for (uint32_t c = tid; c < nc; c += T) atomicAdd(&coff[A.colour[c0 + c] + 1], 1u);
  __syncthreads();
  if (tid == 0)
    for (uint32_t k = 1; k <= ncol; ++k) coff[k] += coff[k - 1];
  __syncthreads();
  // stable colour-major order: per chunk of T contacts, rank within the wave by colour
  // (7 ballots), per-wave counts in LDS, running cursors per colour
  {
    const uint32_t nw = T >> 6, lane = tid & 63, wid = tid >> 6;
    uint32_t* wc = tab;                        // nw x kMaxColours
    uint32_t* cursor = tab + nw * kMaxColours; // kMaxColours
    for (uint32_t k = tid; k < kMaxColours; k += T) cursor[k] = 0;
    for (uint32_t base = 0; base < nc; base += T) {
      for (uint32_t k = tid; k < nw * kMaxColours; k += T) wc[k] = 0;
      __syncthreads();
      const uint32_t c = base + tid;
      const bool valid = c < nc;
      const uint32_t col = valid ? A.colour[c0 + c] : 0u;
      unsigned long long mask = __ballot(valid);
#pragma unroll
      for (int bit = 0; bit < 7; ++bit) {
        const unsigned long long bb = __ballot(((col >> bit) & 1u) != 0);
        mask &= ((col >> bit) & 1u) ? bb : ~bb;
      }
      const uint32_t rank = (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
      if (valid && rank == 0) wc[wid * kMaxColours + col] = (uint32_t)__popcll(mask);
      __syncthreads();
      for (uint32_t k = tid; k < ncol; k += T) {
        uint32_t run = cursor[k];
        for (uint32_t w = 0; w < nw; ++w) {
          const uint32_t x = wc[w * kMaxColours + k];
          wc[w * kMaxColours + k] = run;
          run += x;
        }
        cursor[k] = run;
      }
      __syncthreads();
      if (valid) A.perm[c0 + coff[col] + wc[wid * kMaxColours + col] + rank] = c0 + c;
      __syncthreads();
    }
  }
  if (tid == 0)
    for (uint32_t k = 0; k <= ncol; ++k) A.colour_off[(size_t)sc * (kMaxColours + 1) + k] = coff[k];

  // ---- contact caching in sweep order (a slot whose contact index is out of range -- an
  // internal error -- stops the scene before any sweep reads it)
  for (uint32_t s = tid; s < nc; s += T) {
    const uint32_t c = A.perm[c0 + s];
    if (c - c0 >= nc) { atomicOr(lflag, ERR_INTERNAL); continue; }
    setup_contact(B, R, c, c0 + s, C, A.erp, A.dtinv, O.counters);
  }
  __syncthreads();
  if (*lflag) {
    if (tid == 0) { O.flags |= *lflag; atomicOr(A.any_flags, *lflag); }
    return false;
  }

  // ---- sweeps.  Models without a search, scenes of at most as many contacts as threads (256 at most): everything
  // on the chip, see resident.hpp.  Model 3's WIDE kernel, in two parts a colour: every contact by one lane,
  // except that the sliding ones go on a list (in tab: a colour's contacts share no non-fixed body, so it holds
  // them), which the wavefronts then take one contact at a time.  A colour of a scene holds few contacts, of which
  // up to a third slide; a lane's search takes 12.6k cycles a pass however few of its wavefront's lanes search, a
  // wavefront's 3.0k to 3.7k.  (Measured for this model too: the contacts on the chip, each wavefront relaxing its
  // own sliding ones: 100 against 89 ms for ten steps of 640 scenes of 50 to 2,000 spheres, because the sliding
  // contacts of a colour, five on average, fall unevenly on the wavefronts.)  Model 5 stays with one lane a
  // contact and the narrow kernel: its tree search takes a wavefront so long that lists made its batches up to 2.2
  // times slower (10 steps of 1,500 settled scenes of 200 to 600 spheres: 239 ms by lanes, 527 with lists; of 640
  // scenes of 50 to 2,000, still falling: 59 and 86).
  constexpr bool kSearches = WIDE && MODEL == 3, kResident = MODEL != 3 && MODEL != 5;
  // Three counts in turn: the one of the colour before is cleared between this colour's first barrier,
  // when every thread has read it, and the next colour's, behind which it is used again.
  uint32_t* slide_count = red + 13;    // (the scans use the first eight words)
  uint32_t turn = 0;
  if (kSearches) {
    if (tid < 3) slide_count[tid] = 0;
    __syncthreads();
  }
  uint32_t iters = 0;
  double last = 0;
  bool resident = false;
  if constexpr (kResident) {
    resident = nc != 0 && nc <= T && T <= kResidentThreads && (T > 64 || S.nbody <= kBatchTailFree);
    if (resident) {
      // places in LDS for the contacts' non-fixed bodies, in arrival order
      for (uint32_t i = tid; i < S.nbody; i += T) tab[i] = kNoBody;
      if (tid == 0) red[13] = 0;
      __syncthreads();
      const uint32_t slot = tid;
      const bool have = slot < nc;
      uint32_t colour = kMaxColours;
      if (have) {
        const uint32_t ends[2] = {C.b1[c0 + slot], C.b2[c0 + slot]};
#pragma unroll
        for (int e = 0; e < 2; ++e)
          if (!(ends[e] & kFixedBit) && atomicCAS(&tab[ends[e] - b0], kNoBody, kNoBody - 1u) == kNoBody)
            tab[ends[e] - b0] = atomicAdd(&red[13], 1u);
        colour = A.colour[A.perm[c0 + slot]];
      }
      __syncthreads();
      for (uint32_t i = tid; i < S.nbody; i += T)
        if (tab[i] != kNoBody)
          for (uint32_t k = 0; k < 6; ++k) ldvw[6 * tab[i] + k] = B.dvw[(size_t)kDVW * (b0 + i) + k];
      ResidentContact<> r;
      if (have) resident_load(r, C, c0 + slot, B.sb, [&](uint32_t b) { return tab[b - b0]; });
      __syncthreads();
      for (int it = 0; it < A.iters; ++it) {
        double dmax = 0;
        for (uint32_t k = 0; k < ncol; ++k) {
          if (colour == k) dmax = smax(dmax, resident_relax<MODEL, Trig>(r, ldvw, A.max_sub));
          __syncthreads();
        }
        iters = it + 1;
        if (A.thr > 0 || it + 1 == A.iters) {
          last = wg_max(dmax, red64);
          if (A.thr > 0 && last < A.thr) break;
        }
      }
      if (have) {
        C.f[CF_P * C.cap + c0 + slot] = r.p.x;
        C.f[(CF_P + 1) * C.cap + c0 + slot] = r.p.y;
        C.f[(CF_P + 2) * C.cap + c0 + slot] = r.p.z;
      }
      for (uint32_t i = tid; i < S.nbody; i += T)
        if (tab[i] != kNoBody)
          for (uint32_t k = 0; k < 6; ++k) B.dvw[(size_t)kDVW * (b0 + i) + k] = ldvw[6 * tab[i] + k];
      __syncthreads();
    }
  }
  if (nc && !resident) {
    for (int it = 0; it < A.iters; ++it) {
      double dmax = 0;
      for (uint32_t k = 0; k < ncol; ++k) {
        const uint32_t en = coff[k + 1];
        if constexpr (kSearches) {
          for (uint32_t s = coff[k] + tid; s < en; s += T) {
            const double d = relax_contact<MODEL, Trig, 0, false, true>(C, c0 + s, B.sb, B.dvw, A.dtinv, A.max_sub);
            if (d == kDeferred) tab[atomicAdd(&slide_count[turn], 1u)] = s;
            else dmax = smax(dmax, d);
          }
          __syncthreads();
          const uint32_t slides = __builtin_amdgcn_readfirstlane(slide_count[turn]);
          if (tid == 0) slide_count[turn == 0 ? 2 : turn - 1] = 0;
          turn = turn == 2 ? 0 : turn + 1;
          if (slides > 5 * (T >> 6)) {       // a wavefront takes 14k cycles for one, the lanes 70k for all
            for (uint32_t x = tid; x < slides; x += T)
              dmax = smax(dmax, relax_slide_lane<MODEL, Trig>(C, c0 + tab[x], B.sb, B.dvw, A.dtinv, A.max_sub));
            __syncthreads();
          } else if (slides) {
            for (uint32_t x = __builtin_amdgcn_readfirstlane(tid >> 6); x < slides; x += T >> 6) {
              const uint32_t s = __builtin_amdgcn_readfirstlane(tab[x]);
              dmax = smax(dmax, relax_contact<MODEL, Trig, 6>(C, c0 + s, B.sb, B.dvw, A.dtinv, A.max_sub));
            }
            __syncthreads();
          }
        } else {
          for (uint32_t s = coff[k] + tid; s < en; s += T)
            dmax = smax(dmax, relax_contact<MODEL, Trig>(C, c0 + s, B.sb, B.dvw, A.dtinv, A.max_sub));
          __syncthreads();
        }
      }
      iters = it + 1;
      if (A.thr > 0 || it + 1 == A.iters) {
        last = wg_max(dmax, red64);
        if (A.thr > 0 && last < A.thr) break;
      }
    }
  }

  // ---- integration
  for (uint32_t i = b0 + tid; i < b1; i += T) integrate_body<Trig>(B, i, A.dt, A.damping);
  __syncthreads();
  if (tid == 0) {
    O.nc = nc;
    O.ncol = ncol;
    O.iters = iters;
    O.delta = last;
  }
  return true;
}

}  // namespace

// Two kernels a model; batch_wide() in batch.hip chooses.  WIDE: workgroups of at most 256 threads, bounded for
// them, so that a wavefront has its SIMD's whole register file and one 256-thread workgroup fills a CU; model 3's
// search spills 16 registers instead of 186, which makes it twice as fast.  Otherwise up to 512 threads within half
// of the file, two wavefronts a SIMD.  Corrections on the chip: 96 bytes a thread of dynamic LDS; one
// wavefront's lie behind the bodies' places in tab (scenes of up to kBatchTailFree bodies), so that eight of
// its workgroups still share a CU's 160 KB.
template <int MODEL, class Trig, bool WIDE>
__global__ void __launch_bounds__(WIDE ? kBatchWideThreads : kBatchMaxThreads) k_batch(Bodies B, RawContacts R,
                                                                                       SolverContacts C, BatchArgs A) {
  extern __shared__ double dyn[];
  __shared__ alignas(8) uint32_t tab[kBatchTable + 1];
  double* ldvw = blockDim.x == 64 ? reinterpret_cast<double*>(tab + kBatchTailFree) : dyn;
  __shared__ uint32_t coff[kMaxColours + 1];
  __shared__ uint32_t red[16];
  __shared__ unsigned long long red64[8];
  __shared__ uint32_t lflag;
  __shared__ uint32_t lscene;
  const uint32_t target = A.queue[1];
  for (;;) {
    if (threadIdx.x == 0) lscene = atomicAdd(&A.queue[0], 1u);
    __syncthreads();
    const uint32_t q = lscene;
    __syncthreads();
    if (q >= A.nscenes) break;
    const uint32_t sc = A.order[q];
    const SceneInfo S = A.info[sc];
    uint32_t done = A.out[sc].steps;
    if (A.out[sc].flags & ~ERR_CAPACITY) continue;  // a failed scene stays where it failed
    __syncthreads();
    if (threadIdx.x == 0) A.out[sc].flags = 0;
    while (done < target) {
      if (!scene_step<MODEL, Trig, WIDE>(B, R, C, A, S, sc, tab, coff, red, red64, &lflag, ldvw)) break;
      ++done;
      if (threadIdx.x == 0) A.out[sc].steps = done;
    }
    __syncthreads();
  }
}

template <class Trig>
static void batch_dispatch(int model, const Bodies& B, const RawContacts& R, const SolverContacts& C,
                           const BatchArgs& A, uint32_t grid, uint32_t threads, bool wide, hipStream_t s) {
  const dim3 g(grid), b(threads);
  const bool resident = model != 3 && model != 5 && threads > 64 && threads <= kResidentThreads;
  const uint32_t lds = resident ? batch_ldvw_bytes(threads) : 0;
#define PE_BATCH(model, wide) hipLaunchKernelGGL((k_batch<model, Trig, wide>), g, b, lds, s, B, R, C, A)
  switch (model) {
    case 0: if (wide) PE_BATCH(0, true); else PE_BATCH(0, false); break;
    case 1: if (wide) PE_BATCH(1, true); else PE_BATCH(1, false); break;
    case 2: if (wide) PE_BATCH(2, true); else PE_BATCH(2, false); break;
    case 4: if (wide) PE_BATCH(4, true); else PE_BATCH(4, false); break;
    case 5: PE_BATCH(5, false); break;
    default: if (wide) PE_BATCH(3, true); else PE_BATCH(3, false); break;
  }
#undef PE_BATCH
}

}  // namespace pe_amd
