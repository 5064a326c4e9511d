// LETKF local analysis with grid-point localisation (gfx950).
//
// For every grid point of one grid type (cells or nodes), the analysis of
// Hunt et al. (2007) over the obs_x x obs_y window around it, as the
// reference's r-localised LETKF computes it (src/data_assimilation/letkf.py:
// analysis.analyse :120-166 on the windows of prepare_rloc :288-426):
//   Y   the members' values at the window's observed locations minus their
//       ensemble mean (the window wraps periodically over the inner grid);
//   w   localisation weight / observation variance per observation (the
//       weight is zero outside a wall);
//   Pa  = (k-1)/rho I + Y^T diag(w) Y      (k x k, in the ensemble space)
//   Wa  = sqrt(k-1) Pa^-1/2 + 1 wa^T,   wa = Pa^-1 Y^T diag(w) (y_obs - y_mean)
//   x_a^(i) = x_mean + sum_j Wa[i][j] (x^(j) - x_mean)  at the grid point.
//
// Every contraction is on the FP64 matrix unit (v_mfma_f64_16x16x4: lane l
// supplies A[l%16][l/16] and B[l/16][l%16] and holds D[l/16 + 4r][l%16], r =
// 0..3).  A block analyses 8 x 4 points (2 x 4 above 16 members), a wave one
// row of them, and stages the observation space of their windows attribute by
// attribute in LDS, [position][member], the members' mean taken out once per
// position instead of once per point and position.  Pa of a point is then one
// matrix product per four observations, both operands from one LDS word per
// lane; its inverse square root follows from scaled coupled Newton-Schulz
// iterations (Higham, Functions of Matrices, 2008, sec. 6.7 and 8.3):
//   X = Z Y, T = sqrt(s) (3 I - s X) / 2, Y <- Y T, Z <- T Z,
// from Y = Pa / c, Z = I with c the largest column sum, Z -> sqrt(c) Pa^-1/2.
// All spectra lie in [l, 1], l = (k-1) / (rho c) at first, so the scaling s =
// 3 / (1 + sqrt(l) + l), which maps both ends of the interval to the same
// value, is known in advance; l grows ~6x per iteration while it is small, and
// 7 to 10 iterations reach rounding.  The registers of D are the right operand
// of the next product as they stand and the left operand of its transpose, so
// every iterate is kept with its transpose, at twice the products and without
// a word through LDS.  (Taking a symmetric iterate's own registers for its
// transpose's loses the iteration's stability: the error grows to 1e-3 at a
// condition number of 1e4 instead of 2e-12.)
//
// Bound by the matrix unit: per point 2 * 16 * 16 flops per observation and
// ~50 products of 16 x 16 matrices, 9 Gflop at 160 x 80 points, 4
// attributes, 11 x 11 windows, 16 members (0.13 ms at the 73 Tflop/s of a large
// product).  Both grid types of 161 x 81
// (cells with 4 attributes, nodes with 1) take 0.50 ms; one wave per point with a
// cyclic Jacobi eigendecomposition in LDS, 120 dependent rotations a sweep, took
// 7.6 ms.
// Layout: state and analysis (members, attrs, ny, nx), obs and mask
// (attrs, ny, nx), x fastest; loc (obs_x, obs_y) row-major.
#include "pb_common.hpp"

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;   // waves of a block, one per row of points

struct LetkfArgs {
  int k, attrs, nx, ny, ox, oy, px, py, wall_x, wall_y;
  double rho;
};

// KT 16-member tiles; P points of a wave; CAP window positions staged at once
template <int KT>
struct LetkfShape {
  static constexpr int P = KT == 1 ? 8 : 2;
  static constexpr int CAP = KT == 1 ? 288 : 192;
  static constexpr int S = 16 * KT + 1;   // members of a position, padded to an odd stride
};

__device__ __forceinline__ double over_groups(double v) {   // sum over the four 16-lane groups
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}

// A matrix of KT x KT register tiles, block (I, J) as the matrix unit's D
template <int KT>
struct Mat {
  d4 b[KT][KT];
};

// A B from the registers of A^T and B.  As (A B)^T = B^T A^T, the transpose of
// the product is mul(B, At), bit for bit.
template <int KT>
__device__ __forceinline__ Mat<KT> mul(const Mat<KT>& At, const Mat<KT>& B) {
  Mat<KT> C;
#pragma unroll
  for (int I = 0; I < KT; ++I)
#pragma unroll
    for (int J = 0; J < KT; ++J) {
      d4 c = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int K = 0; K < KT; ++K)
#pragma unroll
        for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f64_16x16x4f64(At.b[K][I][r], B.b[K][J][r], c, 0, 0, 0);
      C.b[I][J] = c;
    }
  return C;
}

// A v, v and the result as member J 16 + lane % 16 in every group
template <int KT>
__device__ __forceinline__ void mul_vec(const Mat<KT>& A, const double (&v)[KT], double (&w)[KT]) {   // A symmetric
  const int row = threadIdx.x / 16;
#pragma unroll
  for (int J = 0; J < KT; ++J) w[J] = 0.0;
#pragma unroll
  for (int I = 0; I < KT; ++I)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double x = __shfl(v[I], row + 4 * r);
#pragma unroll
      for (int J = 0; J < KT; ++J) w[J] += A.b[I][J][r] * x;
    }
#pragma unroll
  for (int J = 0; J < KT; ++J) w[J] = over_groups(w[J]);
}

template <int KT>
__global__ __launch_bounds__(64 * kWaves) void k_letkf(LetkfArgs a, int chunk_w, int chunk_h,
                                                       const double* __restrict__ state,
                                                       const double* __restrict__ obs, const double* __restrict__ mask,
                                                       const double* __restrict__ covar, const double* __restrict__ loc,
                                                       double* __restrict__ out) {
  using H = LetkfShape<KT>;
  constexpr int P = H::P, S = H::S;
  __shared__ double Ys[H::CAP * S];          // observation anomalies [position][member]
  __shared__ double wv[H::CAP], dv[H::CAP];  // 1 / deviation (root of the variance's size; 0: not observed, outside a wall); innovation
  const int lane = threadIdx.x, wave = threadIdx.y, tid = lane + 64 * wave;
  const int m = lane % 16, grp = lane / 16;
  const int tiles_x = (a.nx + P - 1) / P;
  const int i0 = (blockIdx.x % tiles_x) * P, j0 = (blockIdx.x / tiles_x) * kWaves;
  const int k = a.k;
  const long plane = (long)a.nx * a.ny;
  Mat<KT> acc[P];
  double dacc[P][KT];
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int I = 0; I < KT; ++I) {
      dacc[p][I] = 0.0;
#pragma unroll
      for (int J = 0; J < KT; ++J) acc[p].b[I][J] = d4{0.0, 0.0, 0.0, 0.0};
    }

  // Y^T W Y and Y^T W d over the windows, by attribute, by chunks of
  // chunk_w window columns and of chunk_h rows of the block's window union
  for (int at = 0; at < a.attrs; ++at) {
    const double var = covar ? covar[at] : 1.0, idev = 1.0 / sqrt(fabs(var));
    for (int c0 = 0; c0 < a.ox; c0 += chunk_w) {
      const int cw = min(chunk_w, a.ox - c0), RW = P + cw - 1;
      for (int r0 = 0; r0 < kWaves + a.oy - 1; r0 += chunk_h) {
        const int rh = min(chunk_h, kWaves + a.oy - 1 - r0);
        __syncthreads();
        for (int s = tid; s < RW * rh; s += 64 * kWaves) {
          const int ux = i0 + c0 + s % RW - a.px, uy = j0 + r0 + s / RW - a.py;
          const int gx = ((ux % a.nx) + a.nx) % a.nx, gy = ((uy % a.ny) + a.ny) % a.ny;
          const long g = at * plane + (long)gy * a.nx + gx;
          double* y = Ys + s * S;
          const bool seen = mask[g] == 0.0;
          double sum = 0.0;
          if (seen) {
            const double* f = state + g;
#pragma unroll 8
            for (int q = 0; q < k; ++q) {
              const double v = f[q * a.attrs * plane];
              y[q] = v;
              sum += v;
            }
          }
          const double ym = sum / k;
          for (int q = 0; q < 16 * KT; ++q) y[q] = (seen && q < k) ? y[q] - ym : 0.0;
          const bool outside = (a.wall_x && (ux < 0 || ux >= a.nx)) || (a.wall_y && (uy < 0 || uy >= a.ny));
          wv[s] = (seen && !outside) ? idev : 0.0;
          dv[s] = seen ? obs[g] - ym : 0.0;
        }
        __syncthreads();
        if (j0 + wave >= a.ny) continue;
        // this row's window rows in the chunk, four observations at a time
        const int w0 = max(0, r0 - wave), w1 = min(a.oy, r0 + rh - wave);
        const int n = (w1 - w0) * cw;
        int q = 0, c = grp;
        while (c >= cw) {
          c -= cw;
          ++q;
        }
        auto weight = [&](int s) { return s < n ? loc[(c0 + c) * a.oy + w0 + q] : 0.0; };
        double L = weight(grp);
        for (int s = grp; s < n + grp; s += 4) {   // the same number of steps in every group
          const bool ok = s < n;
          const int pos = ok ? (wave + w0 + q - r0) * RW + c : 0;
          // both operands carry the root of the weight, so Pa is exactly
          // symmetric; the sign of a negative weight / variance goes with one of them
          const double rl = sqrt(fabs(L));
          const bool neg = (L < 0.0) != (var < 0.0);
          c += 4;
          while (c >= cw) {
            c -= cw;
            ++q;
          }
          L = weight(s + 4);   // in flight during this step's products
#pragma unroll
          for (int p = 0; p < P; ++p) {
            const double w = rl * wv[pos + p], wd = ok ? w * dv[pos + p] : 0.0;
            double y[KT], wy[KT];
#pragma unroll
            for (int I = 0; I < KT; ++I) {
              y[I] = ok ? w * Ys[(pos + p) * S + 16 * I + m] : 0.0;
              wy[I] = neg ? -y[I] : y[I];
              dacc[p][I] += wy[I] * wd;
            }
#pragma unroll
            for (int I = 0; I < KT; ++I)
#pragma unroll
              for (int J = 0; J < KT; ++J)
                acc[p].b[I][J] = __builtin_amdgcn_mfma_f64_16x16x4f64(wy[I], y[J], acc[p].b[I][J], 0, 0, 0);
          }
        }
      }
    }
  }
  if (j0 + wave >= a.ny) return;

  const double diag = (k - 1.0) / a.rho;
#pragma unroll 1
  for (int p = 0; p < P && i0 + p < a.nx; ++p) {
    // Pa; the rows past the members are those of diag I
    Mat<KT> Y, Yt, Z, Zt, T, Tt;   // with their transposes
    double d[KT], big = 0.0;
#pragma unroll
    for (int q = 0; q < P; ++q) {   // acc[p] by a constant index
      if (q == p) {
        Y = acc[q];
#pragma unroll
        for (int I = 0; I < KT; ++I) d[I] = dacc[q][I];
      }
    }
#pragma unroll
    for (int J = 0; J < KT; ++J) {
      double col = 0.0;
#pragma unroll
      for (int I = 0; I < KT; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (I == J && grp + 4 * r == m) Y.b[I][J][r] += diag;
          col += fabs(Y.b[I][J][r]);
        }
      big = fmax(big, over_groups(col));
      d[J] = over_groups(d[J]);
    }
    for (int o = 1; o < 16; o <<= 1) big = fmax(big, __shfl_xor(big, o));
    const double ic = 1.0 / big;
    double low = fmin(diag * ic, 1.0), dev0 = 1e300;
#pragma unroll
    for (int I = 0; I < KT; ++I)
#pragma unroll
      for (int J = 0; J < KT; ++J) Y.b[I][J] *= ic;
    Yt = Y;
    for (int it = 0; it < 80; ++it) {
      T = it == 0 ? Y : mul<KT>(Zt, Y);
      Tt = it == 0 ? Y : mul<KT>(Y, Zt);
      // the planned iterations leave X within ~1e-9 of I; then on to where
      // it no longer improves
      const bool planned = 1.0 - low > 1e-9;
      bool last = false;
      if (!planned) {
        double dev = 0.0;
#pragma unroll
        for (int I = 0; I < KT; ++I)
#pragma unroll
          for (int J = 0; J < KT; ++J)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              dev = fmax(dev, fabs(T.b[I][J][r] - ((I == J && grp + 4 * r == m) ? 1.0 : 0.0)));
        for (int o = 1; o < 64; o <<= 1) dev = fmax(dev, __shfl_xor(dev, o));
        last = dev < 1e-8 || (dev < 1e-2 && dev > 0.5 * dev0);
        dev0 = dev;
      }
      const double sc = planned ? 3.0 / (1.0 + sqrt(low) + low) : 1.0, rs = sqrt(sc), hs = 0.5 * rs * sc;
#pragma unroll
      for (int I = 0; I < KT; ++I)
#pragma unroll
        for (int J = 0; J < KT; ++J)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const double e = (I == J && grp + 4 * r == m) ? 1.5 * rs : 0.0;
            T.b[I][J][r] = e - hs * T.b[I][J][r];
            Tt.b[I][J][r] = e - hs * Tt.b[I][J][r];
          }
      if (it == 0) {
        Z = T;
        Zt = Tt;
      } else {
        const Mat<KT> Zn = mul<KT>(Tt, Z);
        Zt = mul<KT>(Z, Tt);
        Z = Zn;
      }
      if (last) break;
      const Mat<KT> Yn = mul<KT>(Yt, T);
      Yt = mul<KT>(T, Yt);
      Y = Yn;
      low = fmin(0.25 * sc * low * (3.0 - sc * low) * (3.0 - sc * low), 1.0);
    }
    // Z = Pa^-1/2; wa = Pa^-1 d
    const double rc = sqrt(ic);
#pragma unroll
    for (int I = 0; I < KT; ++I)
#pragma unroll
      for (int J = 0; J < KT; ++J) Z.b[I][J] *= rc;
    double z[KT], wa[KT];
    mul_vec<KT>(Z, d, z);
    mul_vec<KT>(Z, z, wa);
    // Wa as the left operand: row J 16 + m, column I 16 + grp + 4 r
    const double sk = sqrt(k - 1.0);
#pragma unroll
    for (int I = 0; I < KT; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double w = __shfl(wa[I], grp + 4 * r);
#pragma unroll
        for (int J = 0; J < KT; ++J) Z.b[I][J][r] = sk * Z.b[I][J][r] + w;
      }
    // the analysis of up to 16 attributes at once: attribute a0 + m in column m
    const long g = (long)(j0 + wave) * a.nx + i0 + p;
    for (int a0 = 0; a0 < a.attrs; a0 += 16) {
      const bool has = a0 + m < a.attrs;
      const double* f = state + (has ? a0 + m : 0) * plane + g;
      double x[KT][4], sum = 0.0;
#pragma unroll
      for (int I = 0; I < KT; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int mem = 16 * I + grp + 4 * r;
          x[I][r] = (has && mem < k) ? f[(long)mem * a.attrs * plane] : 0.0;
          sum += x[I][r];
        }
      const double xm = over_groups(sum) / k;
#pragma unroll
      for (int I = 0; I < KT; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) x[I][r] = (has && 16 * I + grp + 4 * r < k) ? x[I][r] - xm : 0.0;
#pragma unroll
      for (int J = 0; J < KT; ++J) {
        d4 o = {xm, xm, xm, xm};
#pragma unroll
        for (int I = 0; I < KT; ++I)
#pragma unroll
          for (int r = 0; r < 4; ++r) o = __builtin_amdgcn_mfma_f64_16x16x4f64(Z.b[I][J][r], x[I][r], o, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int mem = 16 * J + grp + 4 * r;
          if (has && mem < k) out[((long)mem * a.attrs + a0 + m) * plane + g] = o[r];
        }
      }
    }
  }
}

template <int KT>
void launch_letkf(const LetkfArgs& a, hipStream_t s, const double* state, const double* obs, const double* mask,
                  const double* covar, const double* loc, double* out) {
  using H = LetkfShape<KT>;
  // the window union of the block, whole where it fits the staging area, else
  // in chunks of whole rows, else of parts of rows
  const int rows = kWaves + a.oy - 1;
  int cw = a.ox, ch = H::CAP / (H::P + cw - 1);
  if (ch < 1) {
    ch = 1;
    cw = H::CAP - H::P + 1;
  }
  if (ch > rows) ch = rows;
  const dim3 grid((unsigned)ceil_div(a.nx, H::P) * (unsigned)ceil_div(a.ny, kWaves));
  hipLaunchKernelGGL(k_letkf<KT>, grid, dim3(64, kWaves), 0, s, a, cw, ch, state, obs, mask, covar, loc, out);
}

}  // namespace

extern "C" int pb_letkf_analyse(pb_ctx* ctx, const pb_letkf_cfg* cfg, const double* state, const double* obs,
                                const double* mask, const double* covar, const double* loc, double* analysis) {
  if (!ctx || !cfg || !state || !obs || !mask || !loc || !analysis)
    return pb_fail(ctx, PB_ERR_ARG, "pb_letkf_analyse: null argument");
  const int k = cfg->members;
  if (k < 2 || k > 32) return pb_fail(ctx, PB_ERR_ARG, "pb_letkf_analyse: members %d (2..32)", k);
  if (cfg->attrs < 1 || cfg->nx < 1 || cfg->ny < 1)
    return pb_fail(ctx, PB_ERR_ARG, "pb_letkf_analyse: empty grid or no attribute");
  if (cfg->obs_x < 1 || cfg->obs_y < 1 || cfg->obs_x % 2 == 0 || cfg->obs_y % 2 == 0 || cfg->obs_x >= cfg->nx ||
      cfg->obs_y >= cfg->ny)
    return pb_fail(ctx, PB_ERR_ARG, "pb_letkf_analyse: window %d x %d must be odd and smaller than the grid",
                   cfg->obs_x, cfg->obs_y);
  if (!(cfg->inflation > 0.0)) return pb_fail(ctx, PB_ERR_ARG, "pb_letkf_analyse: inflation must be > 0");
  if ((long)cfg->nx * cfg->ny > (1L << 31) - 1) return pb_fail(ctx, PB_ERR_ARG, "pb_letkf_analyse: grid too large");
  LetkfArgs a{k, cfg->attrs, cfg->nx, cfg->ny, cfg->obs_x, cfg->obs_y, (cfg->obs_x - 1) / 2, (cfg->obs_y - 1) / 2,
              !cfg->periodic_x, !cfg->periodic_y, cfg->inflation};
  if (k <= 16) launch_letkf<1>(a, ctx->stream, state, obs, mask, covar, loc, analysis);
  else launch_letkf<2>(a, ctx->stream, state, obs, mask, covar, loc, analysis);
  PB_LAUNCH_CHECK(ctx);
  return PB_OK;
}
