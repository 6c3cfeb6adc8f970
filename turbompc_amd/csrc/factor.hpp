// Batched block-tridiagonal factorization of the ADMM Schur matrix
//
//   S = P + sigma I + rho_f C^T C + rho G^T G         (SPD, block tridiagonal)
//
// with diagonal blocks theta_t and sub-diagonal blocks phi_{t-1}
// (turbompc/solvers/admm/admm.py:88-101).  This replaces the cuDSS
// ANALYSIS/FACTORIZATION calls of the reference's direct path
// (turbompc/solvers/admm/csrc/admm_cudss.cu:1046-1053,
// turbompc/solvers/linear_systems_solvers/csrc/cudss_blktridi.cu:59-184).
//
// Factor form (block LDL^T with the stage Schur complements kept inverted):
//   Theta_0 = theta_0
//   Theta_t = theta_t - phi_{t-1} Theta_{t-1}^{-1} phi_{t-1}^T
// and the kernel stores Theta_t^{-1} (symmetric, packed lower) per stage.  The
// solves then need only matrix-vector products (admm_direct.hpp):
//   forward   w_t = Theta_t^{-1} (g_t - phi_{t-1} w_{t-1})
//   backward  x_t = w_t - Theta_t^{-1} phi_t^T x_{t+1}.
//
// One workgroup per problem, G x G threads: thread (ty, tx) keeps the entries
// (ty + G a, tx + G c), a, c < NB, of the stage block in registers; G = 8 (one
// wavefront, no barriers) up to n = 16, else G = 16.  The chain over the stages
// bounds it, and in a stage the n pivots: Gauss-Jordan elimination in place without
// pivoting, which is stable for SPD input (and, eliminating the primal block first,
// for the quasi-definite adjoint KKT blocks of adjoint.hpp), two pivots per trip
// through LDS (their rows and columns; every thread replays both steps).  The next
// stage's blocks of S are fetched while a stage is eliminated.
// Measured (fp64, SRC_S) against one wavefront with the blocks in LDS and a pivot per
// trip: n = 16, T = 51 1290 -> 237 us for 512 problems, 1738 -> 590 for 4096; n = 34,
// T = 41, 128 problems 7898 -> 528; n = 64, T = 20, 64 problems 24289 -> 692.  G = 16
// for n = 16 is the faster at one problem (162 us against 222), even at 512 (223
// against 237) and half as fast at 4096 (1178 against 590).
//
// The recursion is computed in double precision for every storage type: in
// fp32 the update theta_t - phi Theta^{-1} phi^T cancels terms of size rho_f
// |A|^2 down to the curvature of the control directions, and the factor
// would lose most of its digits.  Only the stored Theta_t^{-1} is rounded to
// the storage type; the kernel runs once per QP solve (and per rho change).
#pragma once
#include "common.hpp"

namespace tmpc {

// SRC_QP: assemble theta/phi from QP blocks.  SRC_S: read them from S blocks
// (T, n, 3n) laid out [phi_{t-1} | theta_t | phi_t^T] per block row.
enum FactorSource { SRC_QP = 0, SRC_S = 1 };

using Cmp = double;  // compute type of the factorization

// 1/p of a pivot as a division gives it, zeros and infinities included: S comes from the
// caller (tmpc_blktri_*), and an infinite pivot (a pinned variable) inverts to a zero
// row, where recip's Newton steps alone make NaN of it.  n = 16, T = 51, 512 problems,
// factor and solve: 305 us without, 309 with the fixup (one instruction), 330 with a
// branch to the division outside a range.
__device__ __forceinline__ double pivot_recip(double p) { return __builtin_amdgcn_div_fixup(recip(p), p, 1.0); }

// kc: phi's nonzeros lie in its first kc columns
template <typename R, int SRC, int G, int NB>
__global__ __launch_bounds__(G * G) void factor_kernel(Dims d, int kc, QPDev<R> qp, const R* __restrict__ S,
                                                       const R* __restrict__ rho, R sigma, R rho_f_factor,
                                                       int32_t* __restrict__ ctl, R* __restrict__ thinv) {
  constexpr int TPB = G * G, NP = G * NB;
  const int b = blockIdx.x;
  if (ctl != nullptr && ctl[b * 4 + 2] == 0) return;  // refactor only when flagged
  const int tid = threadIdx.x, ty = tid / G, tx = tid % G;
  const int T = d.T, N = d.N, n = d.n, nx = d.nx, n0 = d.n0, m = d.m;
  const int nn = n * n, pk = th_pitch(n), P = n | 1;  // odd row pitch
  extern __shared__ unsigned char smem_raw[];
  Cmp* Z = reinterpret_cast<Cmp*>(smem_raw);  // Theta_{t-1}^{-1}
  Cmp* F = Z + n * P;                         // phi_{t-1}
  Cmp* U = F + n * P;                         // phi Theta^{-1}; the inverse, for its symmetric part
  Cmp* piv = U + n * P;                       // [2][4][NP] rows k, k + 1, columns k, k + 1, used by turns
  Cmp* sG = piv + 8 * NP;                     // G_t        (m x n)
  Cmp* sAm = sG + m * n;                      // A_minus_t  (nx x n)
  Cmp* sAp = sAm + nx * n;                    // A_plus_t   (nx x n)
  Cmp* sApp = sAp + nx * n;                   // A_plus_{t-1}
  Cmp* sA0 = sApp + nx * n;                   // A0         (n0 x n)

  // the thread's rows and columns; past n: unit rows, decoupled (reads clamped)
  int ri[NB], cj[NB];
#pragma unroll
  for (int a = 0; a < NB; ++a) {
    ri[a] = min(ty + G * a, n - 1);
    cj[a] = min(tx + G * a, n - 1);
  }
  auto in = [&](int a, int c) { return ty + G * a < n && tx + G * c < n; };
  Cmp rho_i = 0, rho_f = 0;
  const Cmp sig = (Cmp)sigma;
  R th[NB][NB], ph[NB][NB];  // SRC_S: theta_t and phi_{t-1} on their way
  auto fetch = [&](int t) {
    const R* Sb = S + ((size_t)b * T + t) * n * (3 * n);
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        const R* row = Sb + ri[a] * (3 * n) + cj[c];
        ph[a][c] = row[0];
        th[a][c] = row[n];
      }
  };
  if constexpr (SRC == SRC_QP) {
    rho_i = (Cmp)rho[b];
    rho_f = rho_i * (Cmp)rho_f_factor;
    for (int e = tid; e < n0 * n; e += TPB) sA0[e] = (Cmp)qp.A0[(size_t)b * n0 * n + e];
  } else {
    fetch(0);
  }

  Cmp A[NB][NB];
  for (int t = 0; t < T; ++t) {
    // ---- theta_t, and phi_{t-1} into F ---------------------------------------
    if constexpr (SRC == SRC_QP) {
      for (int e = tid; e < m * n; e += TPB) sG[e] = (Cmp)qp.G[((size_t)b * T + t) * m * n + e];
      if (t > 0)  // phi_{t-1} = E + rho_f A_plus^T A_minus, from the stage before
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
          for (int c = 0; c < NB; ++c) {
            Cmp s = 0;
            for (int r = 0; r < nx; ++r) s += sAp[r * n + ri[a]] * sAm[r * n + cj[c]];
            s = (Cmp)qp.E[((size_t)b * N + t - 1) * nn + ri[a] * n + cj[c]] + rho_f * s;
            if (in(a, c)) F[ri[a] * P + cj[c]] = s;
          }
      for (int e = tid; e < nx * n; e += TPB) sApp[e] = sAp[e];
      wsync();
      if (t < N)
        for (int e = tid; e < nx * n; e += TPB) {
          sAm[e] = (Cmp)qp.Am[((size_t)b * N + t) * nx * n + e];
          sAp[e] = (Cmp)qp.Ap[((size_t)b * N + t) * nx * n + e];
        }
      wsync();
#pragma unroll
      for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int c = 0; c < NB; ++c) {
          const int i = ri[a], j = cj[c];
          const Cmp v = (Cmp)qp.D[((size_t)b * T + t) * nn + i * n + j] + (i == j ? sig : Cmp(0));
          Cmp gg = 0;
          for (int r = 0; r < m; ++r) gg += sG[r * n + i] * sG[r * n + j];
          Cmp cc = 0;
          if (t == 0)
            for (int r = 0; r < n0; ++r) cc += sA0[r * n + i] * sA0[r * n + j];
          if (t < N)
            for (int r = 0; r < nx; ++r) cc += sAm[r * n + i] * sAm[r * n + j];
          if (t > 0)
            for (int r = 0; r < nx; ++r) cc += sApp[r * n + i] * sApp[r * n + j];
          A[a][c] = v + rho_i * gg + rho_f * cc;
        }
    } else {
#pragma unroll
      for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int c = 0; c < NB; ++c) {
          A[a][c] = (Cmp)th[a][c];
          if (t > 0 && in(a, c)) F[ri[a] * P + cj[c]] = (Cmp)ph[a][c];
        }
      if (t + 1 < T) fetch(t + 1);
      wsync();
    }
    // ---- Theta_t = theta_t - phi_{t-1} Theta_{t-1}^{-1} phi_{t-1}^T ---------
    if (t > 0) {
      Cmp u[NB][NB] = {};
#pragma unroll 8  // (LDS reads in flight)
      for (int q = 0; q < kc; ++q) {
        Cmp f[NB], z[NB];
#pragma unroll
        for (int a = 0; a < NB; ++a) {
          f[a] = F[ri[a] * P + q];
          z[a] = Z[q * P + cj[a]];
        }
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
          for (int c = 0; c < NB; ++c) u[a][c] += f[a] * z[c];
      }
#pragma unroll
      for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int c = 0; c < NB; ++c)
          if (in(a, c)) U[ri[a] * P + cj[c]] = u[a][c];
      wsync();
      Cmp s[NB][NB] = {};
#pragma unroll 8
      for (int l = 0; l < kc; ++l) {
        Cmp f[NB], w[NB];
#pragma unroll
        for (int a = 0; a < NB; ++a) {
          w[a] = U[ri[a] * P + l];
          f[a] = F[cj[a] * P + l];
        }
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
          for (int c = 0; c < NB; ++c) s[a][c] += w[a] * f[c];
      }
#pragma unroll
      for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int c = 0; c < NB; ++c) A[a][c] -= s[a][c];
    }
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int c = 0; c < NB; ++c)
        if (!in(a, c)) A[a][c] = ty + G * a == tx + G * c ? Cmp(1) : Cmp(0);
    // ---- invert -----------------------------------------------------------------
#pragma unroll
    for (int kb = 0; kb < NB; ++kb)
      for (int kk = 0; kk < G; kk += 2) {
        const int k = kb * G + kk;
        if (k >= n) break;
        Cmp* buf = piv + (kk & 2 ? 4 * NP : 0);
#pragma unroll
        for (int c = 0; c < NB; ++c) {
          if (ty == kk) buf[tx + G * c] = A[kb][c];
          if (ty == kk + 1) buf[NP + tx + G * c] = A[kb][c];
          if (tx == kk) buf[2 * NP + ty + G * c] = A[c][kb];
          if (tx == kk + 1) buf[3 * NP + ty + G * c] = A[c][kb];
        }
        wsync();
        const Cmp p11 = buf[k], p12 = buf[k + 1], p21 = buf[NP + k], p22 = buf[NP + k + 1];
        Cmp r1[NB], r2[NB], c1[NB], c2[NB];
#pragma unroll
        for (int c = 0; c < NB; ++c) {
          r1[c] = buf[tx + G * c];
          r2[c] = buf[NP + tx + G * c];
          c1[c] = buf[2 * NP + ty + G * c];
          c2[c] = buf[3 * NP + ty + G * c];
        }
        const bool ik = ty == kk, ik1 = ty == kk + 1, jk = tx == kk, jk1 = tx == kk + 1;
        const Cmp ip = pivot_recip(p11), g21 = p21 * ip, ip2 = pivot_recip(p22 - g21 * p12);
#pragma unroll
        for (int a = 0; a < NB; ++a) {
          const bool i1 = ik && a == kb, i2 = ik1 && a == kb;
          const Cmp g1 = i1 ? -ip : c1[a] * ip;
          const Cmp cc = (i1 ? Cmp(0) : c2[a]) - g1 * p12;  // column k + 1 after the step with pivot k
          const Cmp g2 = i2 ? -ip2 : cc * ip2;
#pragma unroll
          for (int c = 0; c < NB; ++c) {
            const bool j1 = jk && c == kb, j2 = jk1 && c == kb;
            const Cmp q1 = j1 ? Cmp(1) : r1[c];
            const Cmp q2 = j2 ? Cmp(1) : (j1 ? Cmp(0) : r2[c]) - g21 * q1;  // row k + 1 after that step
            const Cmp v = (i1 || j1 ? Cmp(0) : A[a][c]) - g1 * q1;
            A[a][c] = (i2 || j2 ? Cmp(0) : v) - g2 * q2;
          }
        }
      }
    // ---- store packed -----------------------------------------------------------
    // the computed inverse is slightly asymmetric; its symmetric part (not one
    // triangle mirrored, which at cond(Theta) ~ 1e9 breaks the inverse's small
    // residual and makes the ADMM iteration diverge) is what the solves and
    // the next Schur complement use
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int c = 0; c < NB; ++c)
        if (in(a, c)) U[ri[a] * P + cj[c]] = A[a][c];
    wsync();
    R* out = thinv + ((size_t)t * d.B + b) * pk;
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        const int i = ri[a], j = cj[c];
        const Cmp v = Cmp(0.5) * (A[a][c] + U[j * P + i]);
        if (!in(a, c)) continue;
        if (j <= i) out[((i * (i + 1)) >> 1) + j] = (R)v;
        Z[i * P + j] = v;
      }
  }
  if (ctl != nullptr && tid == 0) ctl[b * 4 + 2] = 0;
}

inline size_t factor_smem_bytes(const Dims& d) {
  const size_t n = d.n, np = n <= 16 ? (n + 7) / 8 * 8 : (n + 15) / 16 * 16;
  return sizeof(Cmp) *
         (3 * n * (n | 1) + 8 * np + (size_t)d.m * n + 3 * (size_t)d.nx * n + (size_t)d.n0 * n);
}

}  // namespace tmpc
