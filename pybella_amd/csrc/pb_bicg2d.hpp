// The scalar steps of BiCGStab on the 2D nodal operator and the tile order of
// its launches, shared by the launch-per-phase iteration and the resident one.
#pragma once
#include "pb_op2d.hpp"

namespace pb2d {

__device__ __forceinline__ double eps2() { return 4.930380657631324e-32; }   // DBL_EPSILON^2

__device__ __forceinline__ int block_id() { return blockIdx.x + blockIdx.y * gridDim.x; }
__device__ __forceinline__ int nblocks() { return gridDim.x * gridDim.y; }

// XCD-aware tile order.  Hardware block h is dispatched to XCD h mod 8 (8
// XCDs, each with its own L2).  Giving XCD x the contiguous tile range
// [start(x), start(x) + count(x)) keeps vertically adjacent tiles, which share
// halo rows, in one L2.  Bijective on [0, n); partial records stay indexed by
// the tile number, so sums and iterates do not depend on the mapping.
__device__ __forceinline__ int xcd_tile(int h, int n) {
  constexpr int NX = 8;
  const int x = h % NX, k = h / NX, base = n / NX, rem = n % NX;
  return x < rem ? x * (base + 1) + k : rem * (base + 1) + (x - rem) * base + k;
}

// ---------------------------------------------------------------------------
// scalar steps shared by every block
// ---------------------------------------------------------------------------
__device__ __forceinline__ KState scalars_after_init(KState st, double rr, double bb) {
  st.bnrm2 = sqrt(bb);
  st.rnorm0 = sqrt(rr);
  st.resid = st.rnorm0;
  st.iter = 0;
  st.half = 0;
  st.alpha = 0.0;
  st.omega = 0.0;
  st.beta = 0.0;
  st.x_upd = 0;
  st.rho = rr;
  st.atol = st.tol * st.bnrm2;
  if (st.legacy ? (st.rnorm0 <= st.tol) : (st.rnorm0 <= st.atol)) {
    st.status = ST_CONV;
  } else if (fabs(rr) < eps2()) {
    st.status = ST_BRK_RHO;
  } else {
    st.status = ST_RUN;
  }
  return st;
}

__device__ __forceinline__ KState scalars_after_b(KState st, const double (&tot)[5]) {
  const double ss = tot[0], ts = tot[1], tt = tot[2], rts = tot[3], rtt = tot[4];
  const double snrm = sqrt(ss);
  st.x_upd = 1;
  if (snrm <= st.atol) {
    st.status = ST_P_HALF;
    st.resid = snrm;
    return st;
  }
  const double om = ts / tt;
  if (!isfinite(om) || !isfinite(snrm)) {
    st.status = ST_BRK_OMEGA;
    return st;
  }
  st.omega = om;
  const double rr = ss - 2.0 * om * ts + om * om * tt;
  const double rho_new = rts - om * rtt;
  st.iter += 1;
  st.resid = sqrt(fmax(rr, 0.0));
  if (st.resid <= st.atol) {
    st.status = ST_P_CONV;
  } else if (fabs(om) < eps2()) {
    st.status = ST_P_BRK_OMEGA;
  } else if (st.iter >= st.maxiter) {
    st.status = ST_P_MAXIT;
  } else {
    const double beta = (rho_new / st.rho) * (st.alpha / om);
    st.rho = rho_new;
    if (fabs(rho_new) < eps2() || !isfinite(beta)) {
      st.status = ST_P_BRK_RHO;
    } else {
      st.beta = beta;
      st.status = ST_RUN;
    }
  }
  return st;
}

__device__ __forceinline__ KState scalars_after_l3(KState st, double rtr, double rr) {
  const double rnrm = sqrt(rr);
  st.iter += 1;
  st.resid = rnrm;
  if (!isfinite(rnrm) || !isfinite(rtr)) {
    st.status = ST_BRK_RHO;
  } else if (rnrm <= st.atol) {
    st.status = ST_CONV;
  } else if (fabs(st.omega) < eps2()) {
    st.status = ST_BRK_OMEGA;
  } else if (st.iter >= st.maxiter) {
    st.status = ST_MAXIT;
  } else if (fabs(rtr) < eps2()) {
    st.status = ST_BRK_RHO;
  } else {
    st.beta = (rtr / st.rho) * (st.alpha / st.omega);
    st.rho = rtr;
    st.status = ST_RUN;
  }
  return st;
}

__device__ __forceinline__ int finalize(int pending) {
  switch (pending) {
    case ST_P_CONV: return ST_CONV;
    case ST_P_HALF: return ST_CONV;
    case ST_P_MAXIT: return ST_MAXIT;
    case ST_P_BRK_RHO: return ST_BRK_RHO;
    case ST_P_BRK_OMEGA: return ST_BRK_OMEGA;
    default: return pending;
  }
}

}  // namespace pb2d
