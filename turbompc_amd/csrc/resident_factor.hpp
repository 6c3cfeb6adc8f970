// Factorization for the on-chip ADMM kernel (resident.hpp): the block-tridiagonal
// Schur matrix of the explicit-integrator structure with diagonal costs,
//   S_tt      = theta_t = D_t + sigma I + rho G_t^T G_t + rho_f (A_t^T A_t [t < N]
//               + diag(I_nx, 0) [t > 0] + A0^T A0 [t = 0])
//   S_{t+1,t} = phi_t = -rho_f [A_t; 0]            (rows x_{t+1}, columns z_t = [x_t; u_t])
// (compute_S_Phiinv's blocks, turbompc/solvers/admm/admm.py:71-154), eliminated in
// an order that halves the serial chain and keeps it in the states:
//   1. the controls of every stage (they couple to their own stage and to x_{t+1}
//      only):  Kx = Suu^-1 S_ux, Kn = Suu^-1 phi_u^T, which leaves the state system
//      X_t = S_xx - S_xu Kx - phi_u,t-1 Kn_{t-1},  P_t = phi_x - phi_u Kx;
//   2. the states from both ends towards the middle stage m = T / 2:
//        t < m:  Theta_t = X_t - P_{t-1} Theta_{t-1}^-1 P_{t-1}^T,  V_t = -P_t Theta_t^-1
//        t > m:  Theta_t = X_t - P_t^T Theta_{t+1}^-1 P_t,          V_t = -P_{t-1}^T Theta_t^-1
//        Theta_m = X_m minus both sides' terms.
// fp64 throughout, rounded on store.
//
// The steps' serial chain bounds small batches.  With SPLIT a workgroup has two
// wavefronts: one prepares step s + 1 (what does not follow from other stages: gram,
// control elimination) while the other eliminates step s; the blocks pass through LDS.
// One problem of T = 41, NX = 13: 117 -> 80 us; a launch that fills the SIMDs anyway
// loses (16384 problems of T = 61, NX = 6: 844 -> 1080 us).
//
// A wavefront holds two problems, each in two 16-lane rows, one per direction: lane
// i of a row owns row i of every nx x nx block, and everything that crosses lanes
// goes by DPP row broadcasts (row_dpp.hpp).  A row's step handles the stage p it
// prepares (gram of [A_p; G_p], control elimination) and the stage it eliminates:
// p = t towards higher t, p = t - 1 towards lower t (whose X_t needs stage t - 1).
//
// Output per problem and stage:
//   V  [VW]       row i of V_t (Theta_m^-1 at t = m) in 16-byte chunks, chunk q of
//                 lane i at (q NX + i) W
//   L  [NX+2NU][NX+NU]  lane-minor: word k of lane i;  state lanes i < NX: row i of
//                 Theta_t^-1, -Kx^T, -Kn^T;  control lanes NX + k: row k of -Kx, Suu^-1
#pragma once
#include "factor_rows.hpp"
#include "resident_args.hpp"
#include "row_dpp.hpp"

namespace tmpc {

template <typename R, int NX, int NU>
struct ResGeom {
  static constexpr int W = 16 / (int)sizeof(R);
  static constexpr int NQ = (NX + W - 1) / W;  // 16-byte chunks of a V row
  static constexpr int VW = NQ * W * NX;
  static constexpr int NL = NX + NU;
  static constexpr int LK = NX + 2 * NU;
  static constexpr int LW = LK * NL;
};

__device__ __forceinline__ float buf_load1(__amdgpu_buffer_rsrc_t rs, int off, float) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
}
__device__ __forceinline__ double buf_load1(__amdgpu_buffer_rsrc_t rs, int off, double) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0));
}

// minus-free inverse of the SPD block whose row i is lane i's a[] (symmetric
// sweep, Goodnight; a pivot row is scaled at the end), then its symmetric part
// through sym[16][NX + 1] of the row
template <int NX>
__device__ __forceinline__ void row_inverse(double (&a)[NX], int i, double (*sym)[NX + 1]) {
  double myip = 1.0;
  static_for_pivots<0, NX>([&](auto kc) __attribute__((always_inline)) {
    constexpr int KP = decltype(kc)::value;
    const double ip = recip(row_bcast<KP>(a[KP]));
    const bool me = i == KP;
    const double f = a[KP];
    const double g = me ? 0.0 : -f * ip;
    const double fk = me ? -1.0 : f * ip;
    myip = me ? ip : myip;
    row_sweep<KP>(a, g);
    a[KP] = fk;
  });
#pragma unroll
  for (int k = 0; k < NX; ++k) a[k] *= -myip;
#pragma unroll
  for (int k = 0; k < NX; ++k) sym[i][k] = a[k];
  lds_order();
  const int ic = min(i, NX - 1);
#pragma unroll
  for (int k = 0; k < NX; ++k) a[k] = 0.5 * (a[k] + sym[k][ic]);
  lds_order();
}

// CG: G_t is the same for every stage and problem (its gram is formed once)
template <typename R, int NX, int NU, int MM, bool CG, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 2 * kWave : kWave) void resident_factor_kernel(ResFactorArgs<R> a) {
  using Ge = ResGeom<R, NX, NU>;
  constexpr int W = Ge::W;
  __shared__ double sym_all[4][16][NX + 1];
  __shared__ double prep[SPLIT ? 2 : 1][3][SPLIT ? NX : 1][kWave];  // own, xn, qq of a step, by turns
  const Dims d = a.d;
  const int T = d.T, N = d.N, n = d.n, nx = d.nx, nu = d.n - d.nx, m = d.m, B = d.B;
  const bool chain = SPLIT && threadIdx.x < kWave;  // wavefront 0 eliminates, wavefront 1 prepares
  const int lane = threadIdx.x & (kWave - 1), q4 = lane >> 4, i = lane & 15;
  const bool bwd = (q4 & 1) != 0;
  const int b0 = blockIdx.x * 2;
  const int np = min(2, B - b0);
  const int pr = min(q4 >> 1, np - 1), b = b0 + pr;
  const bool real = (q4 >> 1) < np;
  if (a.ctl != nullptr && __ballot(real && a.ctl[b * 4 + 2] != 0) == 0) return;
  double(*sym)[NX + 1] = sym_all[q4];
  const double rho = (double)a.rho[b], rf = rho * (double)a.rho_f_factor, sig = (double)a.sigma;
  const int mid = T / 2, nf = mid, nb = T - 1 - mid, S = max(nf, nb);
  const bool ix = i < nx, iu = i < nu;

  // this wavefront's dynamics and inequality blocks; masked lanes take an offset
  // past the range and read zero
  const int sa = N * nx * n, sg = T * m * n;  // elements per problem
  const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<R*>(a.Am + (size_t)b0 * sa), (short)0, (int)((size_t)np * sa * sizeof(R)), kBufferFlags);
  const __amdgpu_buffer_rsrc_t rsg = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<R*>(CG ? a.G : a.G + (size_t)b0 * sg), (short)0,
      (int)((size_t)(CG ? m * n : np * sg) * sizeof(R)), kBufferFlags);
  constexpr int kOff = (int)0x80000000u;
  auto lda = [&](bool ok, int e) { return buf_load1(rsa, ok ? e * (int)sizeof(R) : kOff, R()); };
  auto ldg = [&](bool ok, int e) { return buf_load1(rsg, ok ? e * (int)sizeof(R) : kOff, R()); };

  struct Regs {
    R col[NX], row[NX], au[NU], uc[NX], dx, du;
    R gc[CG ? 1 : MM], gu[CG ? 1 : MM], gr[CG ? 1 : NU];
  } nx_;
  auto stage_of = [&](int s) { return bwd ? T - 1 - s : s - 1; };
  auto load = [&](int s) {
    const int p = stage_of(s);
    const bool dyn = p >= 0 && p < N;
    const int ba = pr * sa + p * nx * n;
#pragma unroll
    for (int r = 0; r < NX; ++r) {
      nx_.col[r] = lda(dyn && ix && r < nx, ba + r * n + i);
      nx_.row[r] = lda(dyn && ix && r < nx, ba + i * n + r);
      nx_.uc[r] = lda(dyn && iu && r < nx, ba + r * n + nx + i);
    }
#pragma unroll
    for (int k = 0; k < NU; ++k) nx_.au[k] = lda(dyn && ix && k < nu, ba + i * n + nx + k);
    const int pc = min(max(p, 0), T - 1);
    const R* Dp = a.D + ((size_t)b * T + pc) * n * n;
    nx_.dx = ix ? Dp[i * n + i] : R(1);
    nx_.du = iu ? Dp[(nx + i) * n + nx + i] : R(1);
    if constexpr (!CG) {
      const int bg = pr * sg + pc * m * n;
#pragma unroll
      for (int j = 0; j < MM; ++j) {
        nx_.gc[j] = ldg(ix && j < m, bg + j * n + i);
        nx_.gu[j] = ldg(iu && j < m, bg + j * n + nx + i);
      }
#pragma unroll
      for (int k = 0; k < NU; ++k) nx_.gr[k] = ldg(i < m && k < nu, bg + i * n + nx + k);
    }
  };

  // rho G^T G: row i of the xx and xu blocks, row i of the uu block (lanes < NU)
  auto gram_g = [&](const double (&gc)[MM], const double (&gu)[MM], const double (&gr)[NU], double (&xx)[NX],
                    double (&xu)[NU], double (&uu)[NU]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < MM; ++j)
      if (j < m) row_axpy(xx, gc[j], rho * gc[j]);
#pragma unroll
    for (int k = 0; k < NU; ++k) {
      double sx = 0.0, su = 0.0;
#pragma unroll
      for (int j = 0; j < MM; ++j)
        if (j < m) {
          const double gk = row_bcast_at(gr[k], j);
          sx += gc[j] * gk;
          su += gu[j] * gk;
        }
      xu[k] += rho * sx;
      uu[k] += rho * su;
    }
  };
  double gxx[NX], gxu[NU], guu[NU];
  auto clear_g = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < NX; ++k) gxx[k] = 0.0;
#pragma unroll
    for (int k = 0; k < NU; ++k) gxu[k] = guu[k] = 0.0;
  };
  if (CG && !chain) {
    double gc[MM], gu[MM], gr[NU];
#pragma unroll
    for (int j = 0; j < MM; ++j) {
      gc[j] = (double)ldg(ix && j < m, j * n + i);
      gu[j] = (double)ldg(iu && j < m, j * n + nx + i);
    }
#pragma unroll
    for (int k = 0; k < NU; ++k) gr[k] = (double)ldg(i < m && k < nu, i * n + nx + k);
    clear_g();
    gram_g(gc, gu, gr, gxx, gxu, guu);
  }

  R* Vb = a.V + (size_t)b * T * Ge::VW;
  R* Lb = a.L + (size_t)b * T * Ge::LW;
  const bool st_lane = real && i < NX;
  auto store_v = [&](bool on, int t, const double (&v)[NX], double sgn) __attribute__((always_inline)) {
    if (on && st_lane) {
      R* o = Vb + (size_t)t * Ge::VW + i * W;
#pragma unroll
      for (int k = 0; k < Ge::NQ * W; ++k) o[(k / W) * NX * W + k % W] = k < NX ? (R)(sgn * v[k < NX ? k : 0]) : R(0);
    }
  };

  auto valid_step = [&](int s) { return bwd ? s <= nb : (s >= 1 && s <= nf); };
  auto prepare = [&](int s, double (&own)[NX], double (&xn)[NX], double (&qq)[NX]) __attribute__((always_inline)) {
    const int p = stage_of(s);
    const bool valid = valid_step(s);
    double col[NX], au[NU], xu[NU], uu[NU];
#pragma unroll
    for (int r = 0; r < NX; ++r) col[r] = (double)nx_.col[r];
#pragma unroll
    for (int r = 0; r < NX; ++r) qq[r] = -rf * (double)(bwd ? nx_.col[r] : nx_.row[r]);
#pragma unroll
    for (int k = 0; k < NU; ++k) au[k] = (double)nx_.au[k];
    if constexpr (!CG) {
      double gc[MM], gu[MM], gr[NU];
#pragma unroll
      for (int j = 0; j < MM; ++j) {
        gc[j] = (double)nx_.gc[j];
        gu[j] = (double)nx_.gu[j];
      }
#pragma unroll
      for (int k = 0; k < NU; ++k) gr[k] = (double)nx_.gr[k];
      clear_g();
      gram_g(gc, gu, gr, gxx, gxu, guu);
    }
    // row i of S_xx (without the elimination terms), S_xu and, lanes < NU, S_uu
    const double dgx = (double)nx_.dx + (ix ? sig : 0.0) + (p > 0 && ix ? rf : 0.0);
    const double dgu = (double)nx_.du + (iu ? sig : 0.0);
#pragma unroll
    for (int k = 0; k < NX; ++k) own[k] = gxx[k] + (k == i ? dgx : 0.0);
#pragma unroll
    for (int k = 0; k < NU; ++k) {
      xu[k] = row_fma<0>(col, au[k], 0.0) * rf + gxu[k];
      uu[k] = guu[k] + (k == i ? dgu : 0.0);
    }
    {
      double uc[NX];
#pragma unroll
      for (int r = 0; r < NX; ++r) uc[r] = (double)nx_.uc[r];
#pragma unroll
      for (int k = 0; k < NU; ++k) uu[k] += rf * row_fma<0>(uc, au[k], 0.0);
    }
    if (s < S) load(s + 1);
#pragma unroll
    for (int r = 0; r < NX; ++r) row_axpy(own, col[r], rf * col[r]);
    if (s == 1) {  // stage 0's initial rows (the rows towards lower t never reach it)
      const R* A0b = a.A0 + (size_t)b * d.n0 * n;
      const double w0 = bwd ? 0.0 : rf;
      for (int r = 0; r < d.n0; ++r) {
        const double c = ix ? (double)A0b[r * n + i] : 0.0;
        const double cu = iu ? (double)A0b[r * n + nx + i] : 0.0;
        row_axpy(own, c, w0 * c);
#pragma unroll
        for (int k = 0; k < NU; ++k) {
          const double g = k < nu ? (double)A0b[r * n + nx + k] : 0.0;
          xu[k] += w0 * c * g;
          uu[k] += w0 * cu * g;
        }
      }
    }
    // Suu^-1, the same in every lane
    double si[NU][NU];
#pragma unroll
    for (int r = 0; r < NU; ++r)
#pragma unroll
      for (int k = 0; k <= r; ++k) si[r][k] = si[k][r] = row_bcast_at(uu[r], k);
#pragma unroll
    for (int k = 0; k < NU; ++k) {
      const double ip = recip(si[k][k]);
      double rk[NU];
#pragma unroll
      for (int c = 0; c < NU; ++c) rk[c] = si[k][c] * ip;
#pragma unroll
      for (int r = 0; r < NU; ++r) {
        if (r == k) continue;
        const double f = si[r][k];
#pragma unroll
        for (int c = 0; c < NU; ++c) si[r][c] = c == k ? -f * ip : si[r][c] - f * rk[c];
      }
#pragma unroll
      for (int c = 0; c < NU; ++c) si[k][c] = c == k ? ip : rk[c];
    }
    double kx[NU], kn[NU];
#pragma unroll
    for (int k = 0; k < NU; ++k) {
      kx[k] = kn[k] = 0.0;
#pragma unroll
      for (int c = 0; c < NU; ++c) {
        const double sv = 0.5 * (si[k][c] + si[c][k]);
        kx[k] += sv * xu[c];
        kn[k] -= sv * (rf * au[c]);
      }
    }
    if (valid && st_lane) {
      R* o = Lb + (size_t)p * Ge::LW;
#pragma unroll
      for (int k = 0; k < NU; ++k) {
        o[(NX + k) * Ge::NL + i] = (R)-kx[k];
        o[(NX + NU + k) * Ge::NL + i] = (R)-kn[k];
        o[i * Ge::NL + NX + k] = (R)-kx[k];
      }
      if (i < NU) {
#pragma unroll
        for (int k = 0; k < NU; ++k) {
          double v = 0.5 * (si[0][k] + si[k][0]);
#pragma unroll
          for (int c = 1; c < NU; ++c) v = i == c ? 0.5 * (si[c][k] + si[k][c]) : v;
          o[(NX + k) * Ge::NL + NX + i] = (R)v;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < NX; ++k) xn[k] = 0.0;
#pragma unroll
    for (int k = 0; k < NU; ++k) {
      row_axpy(own, kx[k], -xu[k]);
      row_axpy(xn, kn[k], rf * au[k]);
      row_axpy(qq, bwd ? au[k] : kx[k], rf * (bwd ? kx[k] : au[k]));
    }
  };
  double part[NX];
#pragma unroll
  for (int k = 0; k < NX; ++k) part[k] = 0.0;
  auto eliminate = [&](int s, const double (&own)[NX], const double (&xn)[NX], const double (&qq)[NX])
                       __attribute__((always_inline)) {
    const int p = stage_of(s), t = bwd ? p + 1 : p;
    const bool valid = valid_step(s);
    const bool step = valid && s >= 1;
    if (s == 0) {  // only the last stage's own block (towards lower t)
#pragma unroll
      for (int k = 0; k < NX; ++k) part[k] = valid ? own[k] : part[k];
      return;
    }
    double th[NX];
#pragma unroll
    for (int k = 0; k < NX; ++k) th[k] = part[k] + (bwd ? xn[k] : own[k]);
    row_inverse<NX>(th, i, sym);
    if (step && st_lane) {
      R* o = Lb + (size_t)t * Ge::LW + i;
#pragma unroll
      for (int k = 0; k < NX; ++k) o[k * Ge::NL] = (R)th[k];
    }
    double y[NX];
#pragma unroll
    for (int k = 0; k < NX; ++k) y[k] = row_fma<0>(qq, th[k], 0.0);
    store_v(step, t, y, -1.0);
#pragma unroll
    for (int k = 0; k < NX; ++k) th[k] = 0.0;
#pragma unroll
    for (int k = 0; k < NX; ++k) row_axpy(th, qq[k], y[k]);
#pragma unroll
    for (int k = 0; k < NX; ++k) part[k] = valid ? (bwd ? own[k] : xn[k]) - th[k] : part[k];
  };
  if (!chain) load(0);
  double own[NX], xn[NX], qq[NX];
  if constexpr (SPLIT) {
    for (int s = 0; s <= S + 1; ++s) {  // step s prepared while step s - 1 is eliminated
      auto& buf = prep[chain ? (s + 1) & 1 : s & 1];
      if (chain) {
        if (s >= 1) {
#pragma unroll
          for (int k = 0; k < NX; ++k) {
            own[k] = buf[0][k][lane];
            xn[k] = buf[1][k][lane];
            qq[k] = buf[2][k][lane];
          }
          eliminate(s - 1, own, xn, qq);
        }
      } else if (s <= S) {
        prepare(s, own, xn, qq);
#pragma unroll
        for (int k = 0; k < NX; ++k) {
          buf[0][k][lane] = own[k];
          buf[1][k][lane] = xn[k];
          buf[2][k][lane] = qq[k];
        }
      }
      __syncthreads();
    }
    if (!chain) return;
  } else {
    for (int s = 0; s <= S; ++s) {
      prepare(s, own, xn, qq);
      eliminate(s, own, xn, qq);
    }
  }
  // the middle stage: both directions' terms
#pragma unroll
  for (int k = 0; k < NX; ++k) {
    const RowPair<double> v = row_pair(part[k]);
    part[k] = v.x + v.y;
  }
  row_inverse<NX>(part, i, sym);
  store_v(!bwd, mid, part, 1.0);
  if (a.ctl != nullptr && real && !bwd && i == 0) a.ctl[b * 4 + 2] = 0;
}

}  // namespace tmpc
