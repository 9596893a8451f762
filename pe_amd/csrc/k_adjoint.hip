// Kernels of the adjoint time step (spheres and planes, relaxation models 0, 1 and 3).
//
// For one recorded step (contacts in sweep order with their converged impulses, positions at
// the start of the step, solver body records, post-solve velocities):
//   k_adj_jacobian  one thread per (contact, input direction): contact_map() in dual numbers
//                   gives one column of the contact's 15 x 22 Jacobian;
//   k_adj_prepare   per contact, what a sweep reads: the Jacobian's velocity and impulse blocks and the
//                   inverse of the transposed local system's 3 x 3 matrix, field-major;
//   k_adj_init      body adjoints alpha = adjoint of the post-solve velocities;
//   k_adj_sweep     one colour of a Gauss-Seidel sweep on the transposed (adjoint) system;
//   k_adj_block     all sweeps of a step in one workgroup, for few contacts;
//   k_adj_assemble  position and friction adjoints from the converged (alpha, lambda).
#include "adjoint.hpp"
#include "kernels.hpp"

namespace pe_amd {

using ad::ContactConst;
using ad::Dual;
using ad::kAdjIn;
using ad::kAdjOut;

__device__ __forceinline__ ContactConst make_const(const AdjTape& T, const AdjConsts& A, uint32_t s, uint32_t& i1,
                                                   uint32_t& i2, bool& f1, bool& f2) {
  const uint32_t e1 = T.b1[s], e2 = T.b2[s];
  i1 = e1 & ~kFixedBit;
  i2 = e2 & ~kFixedBit;
  f1 = (e1 & kFixedBit) != 0;
  f2 = (e2 & kFixedBit) != 0;
  ContactConst K;
  K.rad1 = A.param[3 * (size_t)i1];
  K.rad2 = A.param[3 * (size_t)i2];
  const double* s1 = T.sb + (size_t)kSB * i1;
  const double* s2 = T.sb + (size_t)kSB * i2;
  K.im1 = s1[SB_IM];
  K.im2 = s2[SB_IM];
#pragma unroll
  for (int k = 0; k < 9; ++k) { K.I1[k] = s1[SB_IW + k]; K.I2[k] = s2[SB_IW + k]; }
  K.plane = A.shape[i2] == kShapePlane ? 1 : 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    K.pn[k] = A.pnormal[3 * (size_t)i2 + k];
    K.xp[k] = A.ppos[3 * (size_t)i2 + k];
  }
  K.pd = A.pd[i2];
  K.erp = A.erp;
  K.dtinv = A.dtinv;
  return K;
}

template <int MODEL>
__global__ void k_adj_jacobian(AdjTape T, AdjConsts A, double* jac) {
  const size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t s = (uint32_t)(g / kAdjIn), j = (uint32_t)(g % kAdjIn);
  if (s >= T.nc) return;
  uint32_t i1, i2;
  bool f1, f2;
  const ContactConst K = make_const(T, A, s, i1, i2, f1, f2);
  Dual z[kAdjIn];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    z[k] = ad::mkd(T.pos[3 * (size_t)i1 + k]);
    z[3 + k] = ad::mkd(T.pos[3 * (size_t)i2 + k]);
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    z[6 + k] = ad::mkd(f1 ? 0.0 : T.vel[6 * (size_t)i1 + k]);
    z[12 + k] = ad::mkd(f2 ? 0.0 : T.vel[6 * (size_t)i2 + k]);
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) z[18 + k] = ad::mkd(T.p[3 * (size_t)s + k]);
  z[21] = ad::mkd(T.mu[s]);
  z[j].d = 1.0;
  Dual out[kAdjOut];
  ad::contact_map<Dual, MODEL>(K, z, out);
  double* J = jac + ((size_t)s * kAdjIn + j) * kAdjOut;
#pragma unroll
  for (int k = 0; k < kAdjOut; ++k) J[k] = out[k].d;
}

// Jacobian entry d out[k] / d z[j] of contact s.
__device__ __forceinline__ double jget(const double* jac, uint32_t s, int j, int k) {
  return jac[((size_t)s * kAdjIn + j) * kAdjOut + k];
}

// Mc = P_p^T - Q_p^T P_U^T (P_p = dE2/dp, Q_p = d(-contrib)/dp, P_U = dE2/dU), inverted.
// Fields of a contact in `pk` (field f of contact s at pk[f * nc + s]): P_U^T, 12 x 3; Q_p^T, 3 x 12; Mc^-1.
constexpr int AK_PU = 0, AK_QP = 36, AK_MI = 72;
static_assert(AK_MI + 9 == kAdjSweepFields, "fields of a contact in an adjoint sweep");
__global__ void k_adj_prepare(uint32_t nc, const double* jac, double* pk) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nc) return;
  m33 M;
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      double v = jget(jac, s, 18 + a, b);                    // P_p[b][a]
      for (int m = 0; m < 12; ++m) v -= jget(jac, s, 18 + a, 3 + m) * jget(jac, s, 6 + m, b);
      M.a[3 * a + b] = v;
    }
  const m33 Mi = mat_inv(M);
  for (int m = 0; m < 12; ++m)
    for (int c = 0; c < 3; ++c) {
      pk[(size_t)(AK_PU + 3 * m + c) * nc + s] = jget(jac, s, 6 + m, c);
      pk[(size_t)(AK_QP + 12 * c + m) * nc + s] = jget(jac, s, 18 + c, 3 + m);
    }
#pragma unroll
  for (int k = 0; k < 9; ++k) pk[(size_t)(AK_MI + k) * nc + s] = Mi.a[k];
}

// alpha_b = (vbar + dt * xbar, wbar) for non-fixed bodies, 0 for fixed ones.
__global__ void k_adj_init(uint32_t n, const uint8_t* fixed, const double* xbar, const double* vbar,
                           const double* wbar, double dt, double* alpha) {
  const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n) return;
  double* a = alpha + 6 * (size_t)b;
  if (fixed[b]) {
#pragma unroll
    for (int k = 0; k < 6; ++k) a[k] = 0.0;
    return;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    a[k] = vbar[3 * (size_t)b + k] + dt * xbar[3 * (size_t)b + k];
    a[3 + k] = wbar[3 * (size_t)b + k];
  }
}

__device__ __forceinline__ void wave_max_u64(double v, unsigned long long* out) {
  unsigned long long u = (unsigned long long)__double_as_longlong(v);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const unsigned long long o = __shfl_xor(u, d, 64);
    u = o > u ? o : u;
  }
  if ((threadIdx.x & 63) == 0 && u) atomicMax(out, u);
}

// One contact's update of an adjoint sweep: f(k) reads its fields, a1 / a2 are its non-fixed bodies'
// adjoints (null for fixed ones) and l its lambda, updated in place.  Returns the largest change of lambda.
template <class F>
__device__ __forceinline__ double adj_relax(const F& f, double* a1, double* a2, double* l) {
  double a[12];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    a[k] = a1 ? a1[k] : 0.0;
    a[6 + k] = a2 ? a2[k] : 0.0;
  }
  double ln[3];
  // remove the contact's own term: a += P_U^T lambda_old
#pragma unroll
  for (int m = 0; m < 12; ++m)
    a[m] += f(AK_PU + 3 * m) * l[0] + f(AK_PU + 3 * m + 1) * l[1] + f(AK_PU + 3 * m + 2) * l[2];
  double rhs[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double v = 0.0;
#pragma unroll
    for (int m = 0; m < 12; ++m) v -= f(AK_QP + 12 * c + m) * a[m];
    rhs[c] = v;
  }
#pragma unroll
  for (int c = 0; c < 3; ++c)
    ln[c] = f(AK_MI + 3 * c) * rhs[0] + f(AK_MI + 3 * c + 1) * rhs[1] + f(AK_MI + 3 * c + 2) * rhs[2];
#pragma unroll
  for (int m = 0; m < 12; ++m)
    a[m] -= f(AK_PU + 3 * m) * ln[0] + f(AK_PU + 3 * m + 1) * ln[1] + f(AK_PU + 3 * m + 2) * ln[2];
  if (a1)
#pragma unroll
    for (int k = 0; k < 6; ++k) a1[k] = a[k];
  if (a2)
#pragma unroll
    for (int k = 0; k < 6; ++k) a2[k] = a[6 + k];
  double d = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    d = fmax(d, fabs(ln[k] - l[k]));
    l[k] = ln[k];
  }
  return d;
}

struct AdjFields {
  const double* pk;
  size_t nc, s;
  __device__ __forceinline__ double operator()(int k) const { return pk[(size_t)k * nc + s]; }
};
struct AdjHeldFields {
  double v[kAdjSweepFields];
  __device__ __forceinline__ double operator()(int k) const { return v[k]; }
};

// One colour of the adjoint sweep: contacts [begin, end) share no non-fixed body.
__global__ void k_adj_sweep(AdjTape T, uint32_t begin, uint32_t end, const double* pk, double* alpha, double* lambda,
                            unsigned long long* delta) {
  const uint32_t s = begin + blockIdx.x * blockDim.x + threadIdx.x;
  double d = 0.0;
  if (s < end) {
    const uint32_t e1 = T.b1[s], e2 = T.b2[s];
    double l[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) l[k] = lambda[3 * (size_t)s + k];
    d = adj_relax(AdjFields{pk, T.nc, s}, (e1 & kFixedBit) ? nullptr : alpha + 6 * (size_t)e1,
                  (e2 & kFixedBit) ? nullptr : alpha + 6 * (size_t)e2, l);
#pragma unroll
    for (int k = 0; k < 3; ++k) lambda[3 * (size_t)s + k] = l[k];
  }
  wave_max_u64(d, delta);
}

// All sweeps of a step in one workgroup, a barrier between colours (the contacts of one share no non-fixed
// body, so these are the colour launches' updates in their order) and the host's test for the end -- the
// change of every eighth sweep and of the last against tol, if tol > 0.  out[0]: sweeps done, out[1]: the
// change last looked at (the last sweep's without tol).
//
// What bounds it is the latency of a colour.  HOLD: one contact a thread with its 81 fields in registers for
// all sweeps and the adjoints of all bodies in LDS (kAdjHeldBodies); otherwise fields and adjoints come from
// L2.  576 contacts in 8 colours, 2,000 sweeps: 45 to 50 ms from L2 against 130 by colour launches (1,024
// threads, whose 128 registers do not hold a contact's fields at once: 117); up to 180 contacts in 2 or 3
// colours, held: 2.2 us a sweep against 12.
//   From L2 a colour costs about 3.6 us and 14 ns a contact, a colour launch 11 to 13 us: kAdjBlockColour contacts a
// colour on average.  Reverse pass of two steps of 400 sweeps, one workgroup against colour launches: blocks of
// 931 contacts in 8 colours 38 against 66 ms, 1,408 in 9: 42 and 71, 2,025 in 8: 50 and 74; in 2 colours 1,000
// contacts 16.5 and 20.7, 1,100: 19.7 and 20.7, 1,200: 21.0 and 20.5, 2,000: 28 and 21.
template <bool HOLD, uint32_t THREADS>
__global__ void __launch_bounds__(THREADS) k_adj_block(AdjTape T, ColourOffsets O, uint32_t n, const double* pk,
                                                       double* alpha, double* lambda, uint32_t sweeps, double tol,
                                                       unsigned long long* out) {
  __shared__ double la[HOLD ? 6 * kAdjHeldBodies : 1];
  __shared__ unsigned long long wmax[THREADS / 64];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  AdjHeldFields held;
  double hl[3];
  double *h1 = nullptr, *h2 = nullptr;
  uint32_t colour = kMaxColours;
  if constexpr (HOLD) {
    for (uint32_t i = tid; i < 6 * n; i += THREADS) la[i] = alpha[i];
    if (tid < T.nc) {
#pragma unroll
      for (int k = 0; k < kAdjSweepFields; ++k) held.v[k] = pk[(size_t)k * T.nc + tid];
#pragma unroll
      for (int k = 0; k < 3; ++k) hl[k] = lambda[3 * (size_t)tid + k];
      const uint32_t e1 = T.b1[tid], e2 = T.b2[tid];
      h1 = (e1 & kFixedBit) ? nullptr : la + 6 * e1;
      h2 = (e2 & kFixedBit) ? nullptr : la + 6 * e2;
      for (colour = 0; tid >= O.off[colour + 1]; ++colour) {}
    }
    __syncthreads();
  }
  uint32_t it = 0;
  unsigned long long seen = 0;
  while (it < sweeps) {
    // non-negative doubles order like their bit patterns
    unsigned long long u = 0;
    for (uint32_t k = 0; k < O.ncol; ++k) {
      if constexpr (HOLD) {
        if (colour == k) u = (unsigned long long)__double_as_longlong(adj_relax(held, h1, h2, hl));
      } else {
        for (uint32_t s = O.off[k] + tid; s < O.off[k + 1]; s += THREADS) {
          const uint32_t e1 = T.b1[s], e2 = T.b2[s];
          double l[3];
#pragma unroll
          for (int c = 0; c < 3; ++c) l[c] = lambda[3 * (size_t)s + c];
          const unsigned long long d = (unsigned long long)__double_as_longlong(
              adj_relax(AdjFields{pk, T.nc, s}, (e1 & kFixedBit) ? nullptr : alpha + 6 * (size_t)e1,
                        (e2 & kFixedBit) ? nullptr : alpha + 6 * (size_t)e2, l));
#pragma unroll
          for (int c = 0; c < 3; ++c) lambda[3 * (size_t)s + c] = l[c];
          u = d > u ? d : u;
        }
      }
      __syncthreads();
    }
    ++it;
    if (it == sweeps || (tol > 0 && it % 8 == 0)) {
#pragma unroll
      for (int x = 32; x > 0; x >>= 1) {
        const unsigned long long o = __shfl_xor(u, x, 64);
        u = o > u ? o : u;
      }
      if (lane == 0) wmax[wave] = u;
      __syncthreads();
      seen = 0;
      for (uint32_t w = 0; w < THREADS / 64; ++w) seen = wmax[w] > seen ? wmax[w] : seen;
      __syncthreads();
      if (tol > 0 && __longlong_as_double((long long)seen) < tol) break;
    }
  }
  if constexpr (HOLD) {
    for (uint32_t i = tid; i < 6 * n; i += THREADS) alpha[i] = la[i];
    if (tid < T.nc)
#pragma unroll
      for (int k = 0; k < 3; ++k) lambda[3 * (size_t)tid + k] = hl[k];
  }
  if (tid == 0) {
    out[0] = it;
    out[1] = seen;
  }
}

// xbar += -(Q_x^T alpha_c + P_x^T lambda_c) per contact; mubar += -P_mu . lambda.
__global__ void k_adj_assemble(AdjTape T, const double* jac, const double* alpha, const double* lambda, double* xbar,
                               double* mubar) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  double mg = 0.0;
  if (s < T.nc) {
    const uint32_t e1 = T.b1[s], e2 = T.b2[s];
    const uint32_t i1 = e1 & ~kFixedBit, i2 = e2 & ~kFixedBit;
    const bool f1 = (e1 & kFixedBit) != 0, f2 = (e2 & kFixedBit) != 0;
    double a[12];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      a[k] = f1 ? 0.0 : alpha[6 * (size_t)i1 + k];
      a[6 + k] = f2 ? 0.0 : alpha[6 * (size_t)i2 + k];
    }
    const double l0 = lambda[3 * (size_t)s], l1 = lambda[3 * (size_t)s + 1], l2 = lambda[3 * (size_t)s + 2];
    double xg[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      double v = jget(jac, s, j, 0) * l0 + jget(jac, s, j, 1) * l1 + jget(jac, s, j, 2) * l2;
      for (int m = 0; m < 12; ++m) v += jget(jac, s, j, 3 + m) * a[m];
      xg[j] = -v;
    }
    if (!f1)
      for (int k = 0; k < 3; ++k) atomicAdd(&xbar[3 * (size_t)i1 + k], xg[k]);
    if (!f2)
      for (int k = 0; k < 3; ++k) atomicAdd(&xbar[3 * (size_t)i2 + k], xg[3 + k]);
    mg = -(jget(jac, s, 21, 0) * l0 + jget(jac, s, 21, 1) * l1 + jget(jac, s, 21, 2) * l2);
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) mg += __shfl_xor(mg, d, 64);
  if ((threadIdx.x & 63) == 0 && mg != 0.0) atomicAdd(mubar, mg);
}

// vbar = alpha_v, wbar = alpha_w (the predictor passes velocities through for spheres).
__global__ void k_adj_finish(uint32_t n, const double* alpha, double* vbar, double* wbar) {
  const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n) return;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    vbar[3 * (size_t)b + k] = alpha[6 * (size_t)b + k];
    wbar[3 * (size_t)b + k] = alpha[6 * (size_t)b + 3 + k];
  }
}

// Body-major copy of (v, w) into 6 doubles per body.
__global__ void k_adj_pack_vel(uint32_t n, const double* v, const double* w, double* vel) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    vel[6 * (size_t)i + k] = v[3 * (size_t)i + k];
    vel[6 * (size_t)i + 3 + k] = w[3 * (size_t)i + k];
  }
}

// Impulses of solver slots as 3 doubles per contact (from the field-major solver arrays).
__global__ void k_adj_pack_p(uint32_t nc, const double* f, size_t cap, double* p, double* mu) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nc) return;
#pragma unroll
  for (int k = 0; k < 3; ++k) p[3 * (size_t)s + k] = f[(CF_P + k) * cap + s];
  mu[s] = f[CF_MU * cap + s];
}

// ---------------------------------------------------------------------------------------------
// Launchers.
// ---------------------------------------------------------------------------------------------
static inline dim3 blocks(size_t n) { return dim3((unsigned)((n + 255) / 256)); }

void adj_jacobian(int model, const AdjTape& T, const AdjConsts& A, double* jac, hipStream_t s) {
  if (!T.nc) return;
  const size_t n = (size_t)T.nc * kAdjIn;
  if (model == 0) hipLaunchKernelGGL(k_adj_jacobian<0>, blocks(n), dim3(256), 0, s, T, A, jac);
  else if (model == 1) hipLaunchKernelGGL(k_adj_jacobian<1>, blocks(n), dim3(256), 0, s, T, A, jac);
  else hipLaunchKernelGGL(k_adj_jacobian<3>, blocks(n), dim3(256), 0, s, T, A, jac);
}
void adj_prepare(uint32_t nc, const double* jac, double* pk, hipStream_t s) {
  if (nc) hipLaunchKernelGGL(k_adj_prepare, blocks(nc), dim3(256), 0, s, nc, jac, pk);
}
void adj_init(uint32_t n, const uint8_t* fixed, const double* xbar, const double* vbar, const double* wbar, double dt,
              double* alpha, hipStream_t s) {
  hipLaunchKernelGGL(k_adj_init, blocks(n), dim3(256), 0, s, n, fixed, xbar, vbar, wbar, dt, alpha);
}
void adj_sweep(const AdjTape& T, uint32_t begin, uint32_t end, const double* pk, double* alpha, double* lambda,
               unsigned long long* delta, hipStream_t s) {
  if (end > begin)
    hipLaunchKernelGGL(k_adj_sweep, blocks(end - begin), dim3(256), 0, s, T, begin, end, pk, alpha, lambda, delta);
}
bool adj_block(const AdjTape& T, const ColourOffsets& O, uint32_t n, const double* pk, double* alpha, double* lambda,
               uint32_t sweeps, double tol, unsigned long long* out, hipStream_t s) {
  if (T.nc <= kAdjHeldContacts && n <= kAdjHeldBodies)
    hipLaunchKernelGGL((k_adj_block<true, kAdjHeldContacts>), dim3(1), dim3(kAdjHeldContacts), 0, s, T, O, n, pk,
                       alpha, lambda, sweeps, tol, out);
  else if (T.nc <= kAdjBlockContacts && T.nc <= kAdjBlockColour * O.ncol)
    hipLaunchKernelGGL((k_adj_block<false, 512>), dim3(1), dim3(512), 0, s, T, O, n, pk, alpha, lambda, sweeps, tol,
                       out);
  else return false;
  return true;
}
void adj_assemble(const AdjTape& T, const double* jac, const double* alpha, const double* lambda, double* xbar,
                  double* mubar, hipStream_t s) {
  if (T.nc) hipLaunchKernelGGL(k_adj_assemble, blocks(T.nc), dim3(256), 0, s, T, jac, alpha, lambda, xbar, mubar);
}
void adj_finish(uint32_t n, const double* alpha, double* vbar, double* wbar, hipStream_t s) {
  hipLaunchKernelGGL(k_adj_finish, blocks(n), dim3(256), 0, s, n, alpha, vbar, wbar);
}
void adj_pack_vel(uint32_t n, const double* v, const double* w, double* vel, hipStream_t s) {
  hipLaunchKernelGGL(k_adj_pack_vel, blocks(n), dim3(256), 0, s, n, v, w, vel);
}
void adj_pack_p(uint32_t nc, const double* f, size_t cap, double* p, double* mu, hipStream_t s) {
  if (nc) hipLaunchKernelGGL(k_adj_pack_p, blocks(nc), dim3(256), 0, s, nc, f, cap, p, mu);
}

}  // namespace pe_amd
