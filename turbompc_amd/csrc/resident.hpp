// On-chip ADMM for the explicit-integrator structure with diagonal costs: one
// problem per workgroup, its blocks resident in LDS and registers for a whole
// chunk of iterations, so that no iteration touches HBM.  Same iteration as
// admm_stream_kernel (admm_stream.hpp: ADMMSolver._solve_jax_loop,
// turbompc/solvers/admm/admm.py:795-1049) on the factorization of
// resident_factor.hpp, which eliminates the controls and meets in the middle of
// the horizon.
//
// What bounds it: the two serial passes over the states (T / 2 steps each, one
// NX-term product per step, by one wavefront, both directions of the horizon side
// by side in two 16-lane rows) and, between them, vector instructions: the
// constraint products, updates and the next right-hand side of all stages run
// stage-parallel over the workgroup's wavefronts.  An iteration is
//   C1  r_t = gx_t + h_{t-1} + V r (inwards);  x_m = Theta_m^-1 r_m
//   P1  w_t = Theta_t^-1 r_t                                   (all stages)
//   C2  x_t = w_t + V_t^T x (outwards)
//   P2  u_t = Suu^-1 (gu_t + rho_f A_u^T x_{t+1}) - Kx x_t, products, relaxation,
//       projection, duals, gamma_t -> gx_t = gamma_x - Kx^T gu, h_t  (all stages)
// with a workgroup barrier after each.  Cycles of an iteration seen by wavefront 0 (C1,
// P1, C2, P2, barriers and the rest): fp32, T = 41, NX = 13, alone on its CU 4190 + 960 +
// 3990 + 4500 + 1780, two workgroups on each 4610 + 2000 + 3730 + 8490 + 2410; fp64, T =
// 101, NX = 6 6810 + 1430 + 6170 + 8480 + 1530.  QP solves against the streaming kernel,
// which reads every record twice per iteration and walks all T stages in turn, are listed
// at the shape classes (resident.hip): 1412 -> 319 us for 20 iterations of 256 problems of
// T = 41, NX = 13 in fp32.
//
// A stage is a group of GL lanes: GL = 32 has the states (and dynamics rows) in the
// first 16-lane row, the controls at lanes 16 .. 16 + NU - 1 and the inequality
// rows in the lanes left over (row 1 first); GL = 16 has all in one row.  A stage's
// lane keeps its words of the factor and of the iterate in registers (KS stages per
// group), A_t, G_t and V_t lie in LDS.  NX, NU, MM bound the shape: smaller problems
// run with zero rows and columns (their factor keeps the padding decoupled).
#pragma once
#include "resident_factor.hpp"

namespace tmpc {

// LDS in elements of R.  C: a record per stage for the chains,
//   V_t [VW] | gx_t [NX] | the terms stage t gets from stage t - 1 (h_{t-1}; zero at
//   t = 0) [NX] | r_t, then w_t, then x_t [16] (lanes past NX write throwaway values),
// at the position in which the chains visit it, ascending for both: stage t <= mid at
// t, stage t > mid at end + mid - t, where end = T (+ 1 for even T, whose position
// mid + 1 is an empty record: the outer chain has a step less).  Position end is the
// middle seen from the outer chain: V_mid again, no terms, and x = 0 (x_T).
struct ResLds {
  int C, A, G, a0, red, total;
};

template <typename R, int NX, int NU>
struct ResRec {
  using Ge = ResGeom<R, NX, NU>;
  static constexpr int gx = Ge::VW, h = gx + NX, x = h + NX;
  static constexpr int size = (x + 16 + Ge::W - 1) / Ge::W * Ge::W;
};

template <typename R, int NX, int NU, int MM>
__host__ __device__ inline ResLds res_lds(int T, bool const_g, int nw) {
  using Ge = ResGeom<R, NX, NU>;
  constexpr int P = (NX + NU) | 1;  // odd row pitch
  const int end = T + 1 - T % 2;
  ResLds L;
  L.C = 0;
  L.A = (end + 1) * ResRec<R, NX, NU>::size;
  L.G = L.A + (T - 1) * NX * P;
  L.a0 = L.G + (const_g ? 1 : T) * MM * P;
  L.red = L.a0 + (NX + NU) * P;
  L.total = L.red + 12 * nw;
  return L;
}

// A group vector seen from both of its 16-lane rows: a has row 0's lanes, b row 1's
// (GL = 16: one row, itself).
template <int GL, typename R>
__device__ __forceinline__ RowPair<R> res_pair(R v) {
  if constexpr (GL == 32)
    return row_pair(v);
  else
    return {v, v};
}

// acc + sum over the MM inequality rows of w[j] s(lane of row j)
template <int NX, int NU, int MM, int GL, typename R>
__device__ __forceinline__ R res_ineq_dot(const R (&w)[MM], const RowPair<R>& s, R acc) {
  if constexpr (GL == 16) {
    return row_fma<NX + NU>(w, s.y, acc);
  } else if constexpr (MM <= 16 - NU) {
    return row_fma<NU>(w, s.y, acc);
  } else {
    R w1[16 - NU], w0[MM - (16 - NU)];
#pragma unroll
    for (int j = 0; j < 16 - NU; ++j) w1[j] = w[j];
#pragma unroll
    for (int j = 16 - NU; j < MM; ++j) w0[j - (16 - NU)] = w[j];
    return row_fma<NX>(w0, s.x, row_fma<NU>(w1, s.y, acc));
  }
}

template <typename R, int NX, int NU, int MM, int GL, int KS, int TPB, int WPE>
__global__ __launch_bounds__(TPB, WPE) void admm_resident_kernel(ResArgs<R> a) {
  using Ge = ResGeom<R, NX, NU>;
  using Rp = RowPair<R>;
  using V16 = typename Vec16<R>::T;
  constexpr int W = Ge::W, NQ = Ge::NQ, VW = Ge::VW, NL = Ge::NL, P = NL | 1, AW = NX * P, GW = MM * P;
  using Rec = ResRec<R, NX, NU>;
  constexpr int CW = Rec::size, CX = Rec::x;
  constexpr int GPW = kWave / GL;
  constexpr int OU = GL == 16 ? NX : 0;  // lane of control 0 in its row
  extern __shared__ __align__(16) unsigned char smem_raw[];
  R* lds = reinterpret_cast<R*>(smem_raw);
  const Dims d = a.d;
  const int T = d.T, N = d.N, n = d.n, nx = d.nx, nu = d.n - d.nx, n0 = d.n0, m = d.m;
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, nth = blockDim.x, nw = nth >> 6;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool cg = a.const_g != 0;
  const ResLds L = res_lds<R, NX, NU, MM>(T, cg, nw);
  R *sC = lds + L.C, *sA = lds + L.A, *sG = lds + L.G, *sA0 = lds + L.a0, *sRed = lds + L.red;

  // lane roles in its stage group
  const int g = lane / GL, i = lane % GL, lr = lane & 15, lc = min(lr, NX - 1);
  const bool row1 = GL == 32 && i >= 16;
  const bool xl = !row1 && lr < NX;
  const int ku = GL == 32 ? (row1 ? lr : -1) : i - NX;
  const bool ul = ku >= 0 && ku < NU;
  const int jq = GL == 32 ? (row1 ? lr - NU : (lr >= NX ? 16 - NU + lr - NX : -1)) : i - NX - NU;
  const bool ix = xl && lr < nx, iu = ul && ku < nu, iz = ix || iu, iq = jq >= 0 && jq < m;
  const int zc = xl ? lr : (ul ? NX + ku : 0);  // padded column of A, G
  const int zr = ix ? lr : nx + ku;             // element of z_t (iz)
  const int mid = T / 2, end = T + 1 - T % 2;
  // offset of stage t's record, t <= T
  auto rec = [&](int t) __attribute__((always_inline)) {
    return __mul24(t <= mid ? t : (t < T ? end + mid - t : end), CW);
  };
  // The stage of slot s: stage 0 is wavefront 0's, which also runs the chains; the
  // other slots go to the wavefronts from the last one down, so that wavefront 0 is
  // the last to get one of the stages left over.  Opaque, so that the addresses and
  // masks that follow from it are formed where they are used and not kept in
  // registers over the iterations.
  auto stage = [&](int s) __attribute__((always_inline)) {
    int t = (s * nw + (s == 0 ? wv : nw - 1 - wv)) * GPW + g;
    __asm__ volatile("" : "+v"(t));
    return t;
  };
  // slots of this wavefront that hold a stage
  const int ns = max((T + (wv + 1) * GPW - 1) / (nw * GPW), 1);

  // ---- control state ----------------------------------------------------------
  int it;
  bool done;
  R res[6];
  if (a.first_chunk) {
    it = 0;
    done = (a.chk_conv == nullptr && a.act_in) ? a.act_in[b] == 0 : false;
    res[0] = res[1] = res[4] = res[5] = rinf<R>();
    res[2] = res[3] = R(1);
  } else {
    it = a.ctl[b * 4 + 0];
    done = a.ctl[b * 4 + 1] != 0;
#pragma unroll
    for (int k = 0; k < 6; ++k) res[k] = a.res[b * 8 + k];
  }
  R rho = a.rho[b];
  const R rho_in = rho;
  const bool slack = a.use_slack && m > 0;
  const R gs = (slack && a.slack_w) ? a.slack_w[b] : R(0);
  const R alpha = a.alpha, oma = R(1) - a.alpha, sigma = a.sigma;

  // ---- the iterate and the QP vectors into registers ----------------------------
  // vz: x, u or z_g;  vy: y_f or y_g;  vc: c or l;  vq: q or the upper bound.  The
  // slack stays in memory, written where a later test or the caller reads it.
  R vz[KS], vy[KS], vc[KS], vq[KS], ge[KS];
  R RA[KS][NX], RB[KS][NU], RC[KS][NU];
  R y0 = R(0), c0 = R(0);
  const bool r0l = iz && zr < n0 && wv == 0 && g == 0;  // a row of A0 (stage 0's group)
  if (r0l) {
    y0 = a.y_f0[(size_t)b * n0 + zr];
    c0 = a.c0[(size_t)b * n0 + zr];
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    vz[s] = vy[s] = vc[s] = vq[s] = ge[s] = R(0);
    const int t = stage(s);
    if (t < T) {
      const size_t bt = (size_t)b * T + t, bn = (size_t)b * N + t;
      if (iz) {
        vz[s] = a.x[bt * n + zr];
        vq[s] = a.q[bt * n + zr];
      }
      if (ix && t < N) {
        vy[s] = a.y_f[bn * nx + lr];
        vc[s] = a.c[bn * nx + lr];
      }
      if (iq) {
        vz[s] = a.z[bt * m + jq];
        vy[s] = a.y_g[bt * m + jq];
        vc[s] = a.l[bt * m + jq];
        vq[s] = a.u[bt * m + jq];
      }
    }
  }
  auto finish = [&](bool wrote) {
    // the state back, the iteration word and the control words
    bool bad = !__builtin_isfinite(rho) || (r0l && !__builtin_isfinite(y0));
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int t = stage(s);
      if (t < T) {
        const size_t bt = (size_t)b * T + t, bn = (size_t)b * N + t;
        bad |= !__builtin_isfinite(vz[s]) || !__builtin_isfinite(vy[s]);
        if (wrote) {
          if (iz) a.x[bt * n + zr] = vz[s];
          if (ix && t < N) a.y_f[bn * nx + lr] = vy[s];
          if (iq) {
            a.z[bt * m + jq] = vz[s];
            a.y_g[bt * m + jq] = vy[s];
            if (!slack) a.xi[bt * m + jq] = R(0);
          }
        }
        if (iq) bad |= !__builtin_isfinite(a.xi[bt * m + jq]);
      }
    }
    if (wrote && r0l) a.y_f0[(size_t)b * n0 + zr] = y0;
    const bool any = __syncthreads_or(bad ? 1 : 0) != 0;
    if (tid == 0) {
      if (b == 0) a.ctl[kRecordsWord] = 0;
      a.ctl[b * 4 + 0] = it;
      a.ctl[b * 4 + 1] = done ? 1 : 0;
      const bool turned = rho != rho_in;
      a.ctl[b * 4 + 2] = turned ? 1 : 0;
      if (turned) a.rho[b] = rho;
#pragma unroll
      for (int k = 0; k < 6; ++k) a.res[b * 8 + k] = res[k];
      a.iters_out[b] = (uint32_t)it | (a.last_chunk && any ? 0x80000000u : 0u);
    }
  };
  // cond_fun (admm.py:843-851)
  auto goes_on = [&](int iter) {
    const bool sc = mod_zero(iter, a.check_every);
    const bool tl = (res[0] > a.eps_abs + a.eps_rel * res[2]) || (res[1] > a.eps_abs + a.eps_rel * res[3]);
    return ((iter < a.max_iter) && (!sc || tl)) || iter < 1;
  };
  if (!done && !goes_on(a.it_lo)) done = true;
  if (done) {  // (uniform over the workgroup)
    finish(false);
    return;
  }

  // ---- resident blocks: U loads in flight per thread, then their LDS stores --------
  {
    auto copy = [&](auto un, int cnt, auto&& get, auto&& put) __attribute__((always_inline)) {
      constexpr int U = decltype(un)::value;
      for (int e0 = tid; e0 < cnt; e0 += U * nth) {
        decltype(get(0)) v[U];
#pragma unroll
        for (int k = 0; k < U; ++k) v[k] = get(min(e0 + k * nth, cnt - 1));
#pragma unroll
        for (int k = 0; k < U; ++k)
          if (e0 + k * nth < cnt) put(e0 + k * nth, v[k]);
      }
    };
    using U8 = std::integral_constant<int, 8>;
    constexpr int VC = VW / W;
    const V16* gv = reinterpret_cast<const V16*>(a.V + (size_t)b * T * VW);
    copy(U8{}, T * VC, [&](int e) { return gv[e]; },
         [&](int e, V16 v) {
           const int t = e / VC, k = e - t * VC;
           reinterpret_cast<V16*>(sC + rec(t))[k] = v;
           if (t == mid) reinterpret_cast<V16*>(sC + rec(T))[k] = v;
         });
    // a block of padded rows: row e / NL (of per rows a stage), column e % NL
    auto rows = [&](const R* src, R* dst, int stages, int per, int live) __attribute__((always_inline)) {
      copy(std::integral_constant<int, 12>{}, stages * per * NL,
           [&](int e) {
             const int row = e / NL, c = e - row * NL, t = row / per, r = row - t * per;
             const bool cx = c < nx, cu = c >= NX && c - NX < nu, on = r < live && (cx || cu);
             const R v = src[on ? (t * live + r) * n + (cx ? c : nx + c - NX) : 0];
             return on ? v : R(0);
           },
           [&](int e, R v) { dst[(e / NL) * P + e % NL] = v; });
    };
    rows(a.Am + (size_t)b * N * nx * n, sA, N, NX, nx);
    if (m > 0)
      rows(cg ? a.G : a.G + (size_t)b * T * m * n, sG, cg ? 1 : T, MM, m);
    else
      for (int e = tid; e < (cg ? 1 : T) * MM * P; e += nth) sG[e] = R(0);
    for (int e = tid; e < NL * NL; e += nth) {
      const int r = e / NL, c = e - r * NL;
      const bool cx = c < nx, cu = c >= NX && c - NX < nu;
      const bool rx = r < nx, ru = r >= NX && r - NX < nu;
      const int rr = rx ? r : nx + r - NX;
      sA0[r * P + c] = ((rx || ru) && rr < n0 && (cx || cu))
                           ? a.A0[((size_t)b * n0 + rr) * n + (cx ? c : nx + c - NX)] : R(0);
    }
    if (tid < NX) sC[Rec::h + tid] = R(0);  // nothing reaches stage 0
    for (int e = VW + tid; e < CW; e += nth) sC[end * CW + e] = R(0);
    if (end > T)  // the empty record
      for (int e = tid; e < CW; e += nth) sC[(mid + 1) * CW + e] = R(0);
    // the factor's words of this lane
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const R* gl = a.L + ((size_t)b * T + min(stage(s), T - 1)) * Ge::LW + zc;
#pragma unroll
      for (int k = 0; k < NX; ++k) RA[s][k] = gl[k * NL];
#pragma unroll
      for (int k = 0; k < NU; ++k) RB[s][k] = gl[(NX + k) * NL];
#pragma unroll
      for (int k = 0; k < NU; ++k) RC[s][k] = xl ? gl[(NX + NU + k) * NL] : R(0);
    }
  }
  __syncthreads();

  // row of [A_t; G_t] (state and inequality lanes), column of A_t and of G_t; t < T
  const int rstride = xl ? AW : (cg ? 0 : GW);
  const R* rbase = xl ? sA + lr * P : sG + (jq >= 0 && jq < MM ? jq * P : 0);
  auto get_row = [&](R (&w)[NX], R (&wu)[NU], int t) __attribute__((always_inline)) {
    const R* p = rbase + __umul24(xl ? min(t, N - 1) : t, rstride);
#pragma unroll
    for (int k = 0; k < NX; ++k) w[k] = p[k];
#pragma unroll
    for (int k = 0; k < NU; ++k) wu[k] = p[NX + k];
  };
  auto get_col = [&](R (&w)[NX], int t) __attribute__((always_inline)) {
    const R* p = sA + zc + __umul24(min(t, N - 1), AW);
#pragma unroll
    for (int r = 0; r < NX; ++r) w[r] = p[r * P];
  };
  auto get_gcol = [&](R (&w)[MM], int t) __attribute__((always_inline)) {
    const R* p = sG + zc + (cg ? 0 : __umul24(t, GW));
#pragma unroll
    for (int r = 0; r < MM; ++r) w[r] = p[r * P];
  };
  // row / column products with A0 (stage 0's group; every lane computes)
  auto a0_row = [&](const Rp& z) __attribute__((always_inline)) {
    R w[NX], wu[NU];
    const R* p = sA0 + zc * P;
#pragma unroll
    for (int k = 0; k < NX; ++k) w[k] = p[k];
#pragma unroll
    for (int k = 0; k < NU; ++k) wu[k] = p[NX + k];
    return row_fma<OU>(wu, z.y, row_fma<0>(w, z.x, R(0)));
  };
  auto a0_col = [&](const Rp& z) __attribute__((always_inline)) {
    R w[NX], wu[NU];
    const R* p = sA0 + zc;
#pragma unroll
    for (int k = 0; k < NX; ++k) w[k] = p[k * P];
#pragma unroll
    for (int k = 0; k < NU; ++k) wu[k] = p[(NX + k) * P];
    return row_fma<OU>(wu, z.y, row_fma<0>(w, z.x, R(0)));
  };

  // gamma_t from the updated iterate (compute_gamma, admm.py:157-174), its controls
  // eliminated: gx_t = gamma_x - Kx^T gamma_u, and the terms stage t + 1 gets
  // (A_plus^T = [-I; 0], and the controls' coupling).  Inequality lanes compute
  // throwaway values.
  auto emit = [&](int s, int t, R tgt, R t0, const R (&ac)[NX], const R (&gc)[MM]) __attribute__((always_inline)) {
    const Rp bt = res_pair<GL>(tgt);
    R gam = sigma * vz[s] - vq[s];
    gam = row_fma<0>(ac, bt.x, gam);
    gam = res_ineq_dot<NX, NU, MM, GL>(gc, bt, gam);
    if (s == 0 && wv == 0) {  // (uniform per wavefront)
      const R g0 = a0_col(res_pair<GL>(t0));
      gam += g == 0 ? g0 : R(0);
    }
    ge[s] = gam;
    // gamma_x and -tgt are as large as the duals and nearly cancel (stationarity), so
    // the controls' terms are summed before they meet them: one rounding at that size
    const Rp bg = res_pair<GL>(gam);
    R gx = R(0), hh = R(0);
    row_fma_x2<OU>(bg.y, RB[s], gx, RC[s], hh);
    if (xl && t < T) {
      sC[rec(t) + Rec::gx + lr] = gam + gx;
      if (t < N) sC[rec(t + 1) + Rec::h + lr] = hh - tgt;
    }
  };
  // residual ingredients of the iterate in vz, vy (and y0): exchanged with the
  // neighbouring stages through the x entries of C, which are free outside C1 .. P2.
  // f(s, t, mz, cx, px, aty, a0x): row product [A; G] z, A z - x_{t+1}, D z,
  // C^T y_f + G^T y_g, A0 z (stage 0)
  auto residual_pass = [&](auto&& f) __attribute__((always_inline)) {
    R xn[KS], yp[KS];
    R* sx = sC + CX + lc;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int t = stage(s);
      if (xl && t < T) sx[rec(t)] = vz[s];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int t = stage(s);
      xn[s] = (xl && t < N) ? sx[rec(t + 1)] : R(0);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int t = stage(s);
      if (xl && t < T) sx[rec(t)] = t < N ? vy[s] : R(0);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int t = stage(s);
      yp[s] = (xl && t > 0 && t < T) ? sx[rec(t - 1)] : R(0);
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (s >= ns) break;
      __builtin_amdgcn_sched_barrier(0);  // one slot's working set at a time
      const int t = stage(s), tc = min(t, T - 1);
      R ac[NX], gc[MM], ar[NX], au[NU];
      get_col(ac, tc);
      get_gcol(gc, tc);
      get_row(ar, au, tc);
      const R zv = (xl || ul) ? vz[s] : R(0);
      const R yv = ((xl && t < N) || iq) ? vy[s] : R(0);
      const Rp bz = res_pair<GL>(zv), by = res_pair<GL>(yv);
      const R mz = row_fma<OU>(au, bz.y, row_fma<0>(ar, bz.x, R(0)));
      R aty = res_ineq_dot<NX, NU, MM, GL>(gc, by, row_fma<0>(ac, by.x, R(0))) - yp[s];
      R a0x = R(0);
      if (s == 0 && wv == 0) {
        a0x = a0_row(bz);
        const R ay = a0_col(res_pair<GL>(r0l ? y0 : R(0)));
        aty += g == 0 ? ay : R(0);
      }
      R dd = R(0);
      if (iz && t < T) dd = a.D[(((size_t)b * T + t) * n + zr) * n + zr];
      f(s, t, mz, mz - xn[s], dd * zv, aty, a0x);
    }
  };
  // maxima over the workgroup, the same in every thread
  auto wg_max = [&](auto& v, int cnt) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < cnt; ++k) v[k] = wave_max(v[k]);
    if (lane == 0)
#pragma unroll
      for (int k = 0; k < cnt; ++k) sRed[wv * 12 + k] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < cnt; ++k) v[k] = R(0);
    for (int w = 0; w < nw; ++w)
#pragma unroll
      for (int k = 0; k < cnt; ++k) v[k] = rmax(v[k], sRed[w * 12 + k]);
    __syncthreads();
  };

  // ---- first-order check of the input iterate (admm_stream_kernel's) ---------------
  if (a.first_chunk && a.chk_conv != nullptr) {
    R v[4] = {R(0), R(0), R(0), R(0)};
    residual_pass([&](int s, int t, R mz, R cx, R px, R aty, R a0x) __attribute__((always_inline)) {
      const bool on = t < T;
      v[0] = rmax(v[0], on && iz ? rabs(px + vq[s] + aty) : R(0));
      v[1] = rmax(v[1], ix && t < N ? rabs(cx - vc[s]) : R(0));
      v[1] = rmax(v[1], s == 0 && r0l ? rabs(a0x - c0) : R(0));
      if (on && iq) {
        const R xi = slack ? a.xi[((size_t)b * T + t) * m + jq] : R(0);
        const R gv = mz + xi;
        v[2] = rmax(v[2], rmax(rmax(vc[s] - gv, gv - vq[s]), R(0)));
        if (slack) v[3] = rmax(v[3], rabs(gs * xi + vy[s]));
        if (a.chk_g) a.chk_g[((size_t)b * T + t) * m + jq] = gv;
      }
    });
    __syncthreads();
    wg_max(v, 4);
    const R conv = rmax(rmax(v[0], v[1]), rmax(v[2], v[3]));
    const bool act = (a.act_in ? a.act_in[b] != 0 : true) && conv > a.chk_tol;
    if (tid == 0) {
      a.chk_conv[b] = conv;
      if (a.chk_eq) a.chk_eq[b] = v[1];
      if (a.chk_iq) a.chk_iq[b] = v[2];
      if (a.act_out) a.act_out[b] = act ? 1 : 0;
    }
    if (!act) {  // a stopped problem keeps its input iterate (zero iterations)
      done = true;
      finish(false);
      return;
    }
  }

  // ---- gamma of the input iterate -------------------------------------------------
  {
    const R rho_f = rho * a.rho_f_factor;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (s >= ns) break;
      __builtin_amdgcn_sched_barrier(0);
      const int t = stage(s), tc = min(t, T - 1);
      R ac[NX], gc[MM];
      get_col(ac, tc);
      get_gcol(gc, tc);
      const R tgt = xl ? rho_f * vc[s] - vy[s] : (iq ? rho * vz[s] - vy[s] : R(0));
      emit(s, t, tgt, r0l ? rho_f * c0 - y0 : R(0), ac, gc);
    }
  }
  __syncthreads();

  // The chains, in the first 32 lanes: row 0 from position 0 to mid, row 1 from mid + 1
  // to end, mid steps each.  Records are fetched CB - 1 positions ahead, in CB register
  // sets used by turns: an LDS read of a record takes longer than a step of NX <= 6
  // (fp64, NX = 6: 178 cycles a step with two sets, 141 with three; fp32, NX = 12: 190 and
  // 158); where wide blocks and many stages per group fill the registers, a third set
  // costs spills (fp32, NX = 13, 4096 problems: 2173 us with two sets, 2496 with three).
  constexpr int CB = (NX <= 6 || TPB == 512) ? 3 : 2;
  const bool bw = (lane & 16) != 0;
  R* const cb = sC + (bw ? (mid + 1) * CW : 0);
  struct CBuf {
    R w[NX], g, h;
  };
  auto ld_row = [&](CBuf& c, const R* q) __attribute__((always_inline)) {  // gx, h and V's row
    c.g = q[Rec::gx + lc];
    c.h = q[Rec::h + lc];
    const R* p = q + lc * W;
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      if (k * W + W <= NX) {
        const V16 v = *reinterpret_cast<const V16*>(p + k * NX * W);
#pragma unroll
        for (int e = 0; e < W; ++e) c.w[k * W + e] = v[e];
      } else {  // the last entries alone: the registers of a whole chunk's rest would be
                // given to other values, which then wait for the load (fp32, NX = 13: 210
                // cycles a step, 170 like this)
#pragma unroll
        for (int e = 0; k * W + e < NX; ++e) c.w[k * W + e] = p[k * NX * W + e];
      }
    }
  };
  const int vcol = (lc / W) * NX * W + lc % W;
  auto ld_col = [&](CBuf& c, const R* q) __attribute__((always_inline)) {  // w_t and V's column
    c.g = q[CX + lc];
#pragma unroll
    for (int k = 0; k < NX; ++k) c.w[k] = q[vcol + k * W];
  };

  for (int iter = a.it_lo; iter < a.it_hi; ++iter) {
    if (iter > a.it_lo && !goes_on(iter)) {
      done = true;
      break;
    }
    const R rho_f = rho * a.rho_f_factor;
    R xc = R(0);
    // C1
    if (tid < 32) {
      __builtin_amdgcn_s_setprio(3);
      CBuf c[CB];
      R* q = cb;
#pragma unroll
      for (int k = 0; k < CB - 1; ++k) ld_row(c[k], q + k * CW);
      R r = c[0].g + c[0].h;
      // step k of a turn: (the records past the last one, CB - 2 at most, are fetched in vain)
      auto step = [&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        ld_row(c[(k + CB - 1) % CB], q + (k + CB - 1) * CW);
        q[k * CW + CX + lr] = r;
        // (gx and h first: each alone is as large as the duals, and would be rounded so with
        // every term: fp32, T = 51, NX = 12 states 1.29e-6 off 64 bits, 7.1e-7 like this.
        // With two sets they were fetched in this step, and the wait for them is better
        // not tied to the chain's first instruction: fp64, NX = 13 5080 cycles against 5703)
        const CBuf& e = c[(k + 1) % CB];
        if constexpr (CB > 2)
          r = row_fma_sum(c[k].w, r, e.g, e.h);
        else
          r = row_fma<0>(c[k].w, r, e.g + e.h);
      };
      int p = mid;
      for (; p > CB; p -= CB, q += CB * CW) {
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        if constexpr (CB > 2) step(std::integral_constant<int, 2>{});
      }
      step(std::integral_constant<int, 0>{});
      if (p > 1) step(std::integral_constant<int, 1>{});
      if constexpr (CB > 2)
        if (p > 2) step(std::integral_constant<int, 2>{});
      // the middle: both rows' terms
      const Rp vp = row_pair(r);
      CBuf e;
      ld_row(e, sC + rec(mid));
      xc = row_fma<0>(e.w, vp.x + vp.y, R(0));
      if (!bw) sC[rec(mid) + CX + lr] = xc;
      __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();
    // P1, two slots at a time
#pragma unroll
    for (int s = 0; s < KS; s += 2) {
      if (s >= ns) break;
      constexpr int last = KS - 1;
      const int s2 = s + 1 < KS ? s + 1 : last;
      const int t = stage(s), t2 = stage(s2);
      R* p = sC + rec(min(t, T - 1)) + CX + lc;
      R* p2 = sC + rec(min(t2, T - 1)) + CX + lc;
      R w = R(0), w2 = R(0);
      row_fma_2(RA[s], *p, w, RA[s2], *p2, w2);
      if (xl && t < T && t != mid) *p = w;
      if (s2 != s && xl && t2 < T && t2 != mid) *p2 = w2;
    }
    __syncthreads();
    // C2
    if (tid < 32) {
      __builtin_amdgcn_s_setprio(3);
      CBuf c[CB];
      // a turn's steps are at positions q + CB - 1 .. q; the fetches below position 0,
      // CB - 1 at most, go to position 0
      int q = (mid - CB) * CW;
#pragma unroll
      for (int k = 0; k < CB - 1; ++k) ld_col(c[k], cb + max(q + (CB - 1 - k) * CW, 0));
      auto step = [&](auto kc, auto guard) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        const int f = q - k * CW;
        ld_col(c[(k + CB - 1) % CB], cb + (decltype(guard)::value ? max(f, 0) : f));
        xc = row_fma<0>(c[k].w, xc, c[k].g);
        cb[q + (CB - 1 - k) * CW + CX + lr] = xc;
      };
      int p = mid;
      for (; p >= 2 * CB; p -= CB, q -= CB * CW) {
        step(std::integral_constant<int, 0>{}, std::false_type{});
        step(std::integral_constant<int, 1>{}, std::false_type{});
        if constexpr (CB > 2) step(std::integral_constant<int, 2>{}, std::false_type{});
      }
      for (; p > 0; p -= CB, q -= CB * CW) {
        step(std::integral_constant<int, 0>{}, std::true_type{});
        if (p > 1) step(std::integral_constant<int, 1>{}, std::true_type{});
        if constexpr (CB > 2)
          if (p > 2) step(std::integral_constant<int, 2>{}, std::true_type{});
      }
      __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();
    // P2
    const bool chk = mod_zero(iter, a.check_every);
    // the last iteration (of the chunk, or where the next test may end the solve) and
    // one whose residuals are taken
    const bool keep_xi = chk || iter + 1 == a.it_hi || mod_zero(iter + 1, a.check_every);
    const R inv_rho = R(1) / rho;
    const R frac = slack ? gs / (gs + rho) : R(0), xi_f = slack ? rho / (gs + rho) : R(0);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (s >= ns) break;
      __builtin_amdgcn_sched_barrier(0);
      const int t = stage(s), tc = min(t, T - 1);
      R ac[NX], gc[MM], ar[NX], au[NU];
      const R* px = sC + CX + lc;  // x in both rows of the group
      const R xv = px[rec(tc)], xn = px[rec(tc + 1)];
      get_col(ac, tc);
      get_row(ar, au, tc);
      get_gcol(gc, tc);
      // the controls (their lanes; the others compute throwaway values), and the
      // states' part of the row products
      R d1 = R(0), d2 = R(0), d3 = R(0);
      row_fma_3(ac, xn, d1, ar, xv, d2, RA[s], xv, d3);
      const R uv = row_fma<OU>(RB[s], ge[s] + rho_f * d1, d3);
      const R zv = ul ? uv : xv;
      const Rp bz = res_pair<GL>(zv);
      const R mx = row_fma<OU>(au, bz.y, d2);
      R cx0 = R(0);
      if (s == 0 && wv == 0) cx0 = a0_row(bz);
      // over-relaxation, duals, projection / slack; the last stage has no dynamics
      // row (its c and y_f are zero)
      const R rft = t < N ? rho_f : R(0);
      const R zo = vz[s], yo = vy[s];
      const R xnew = alpha * zv + oma * zo;
      const R yf = yo + rft * (alpha * (mx - xn) + oma * vc[s] - vc[s]);
      const R zt = alpha * mx + oma * zo + yo * inv_rho;
      const R proj = rmin(rmax(zt, vc[s]), vq[s]);
      R zn = proj;
      if (slack) {
        zn = (R(1) - frac) * zt + frac * proj;
        if (keep_xi && iq && t < T) a.xi[((size_t)b * T + t) * m + jq] = xi_f * (proj - zt);
      }
      const R ygn = yo + rho * (alpha * mx + oma * zo - zn);
      const R tgt = xl ? rft * vc[s] - yf : (iq ? rho * zn - ygn : R(0));
      vz[s] = (xl || ul) ? xnew : zn;
      vy[s] = xl ? yf : (iq ? ygn : R(0));
      R t0 = R(0);
      if (s == 0 && r0l) {
        y0 = y0 + rho_f * (alpha * cx0 + oma * c0 - c0);
        t0 = rho_f * c0 - y0;
      }
      emit(s, t, tgt, t0, ac, gc);
    }
    __syncthreads();
    it = iter + 1;
    // ---- residuals and adaptive rho (admm.py:392-556), where a later test or rho
    // reads them
    if (chk && ((a.check_every > 0 && iter + a.check_every < a.max_iter) ||
                (iter >= 2 && mod_zero(iter, a.adapt_every)))) {
      R v[11] = {};
      residual_pass([&](int s, int t, R mz, R cx, R px, R aty, R a0x) __attribute__((always_inline)) {
        const bool on = t < T, dr = ix && t < N, q = iq && on, zl = iz && on;
        v[0] = rmax(v[0], dr ? rabs(cx - vc[s]) : (q ? rabs(mz - vz[s]) : R(0)));
        v[1] = rmax(v[1], dr ? rabs(cx) : R(0));
        v[2] = rmax(v[2], dr ? rabs(vc[s]) : R(0));
        v[3] = rmax(v[3], q ? rabs(mz) : R(0));
        v[4] = rmax(v[4], q ? rabs(vz[s]) : R(0));
        v[5] = rmax(v[5], zl ? rabs(px + vq[s] + aty) : R(0));
        v[6] = rmax(v[6], zl ? rabs(px) : R(0));
        v[7] = rmax(v[7], zl ? rabs(aty) : R(0));
        v[8] = rmax(v[8], zl ? rabs(vq[s]) : R(0));
        if (slack) {
          const R xi = q ? a.xi[((size_t)b * T + t) * m + jq] : R(0);
          v[5] = rmax(v[5], q ? rabs(gs * xi + vy[s]) : R(0));
          v[9] = rmax(v[9], rabs(xi));
          v[10] = rmax(v[10], q ? rabs(vy[s]) : R(0));
        }
        if (s == 0 && r0l) {
          v[0] = rmax(v[0], rabs(a0x - c0));
          v[1] = rmax(v[1], rabs(a0x));
          v[2] = rmax(v[2], rabs(c0));
        }
      });
      __syncthreads();
      wg_max(v, 11);
      const R np = rmax(rmax(v[1], v[3]), rmax(v[2], v[4]));
      R nd = rmax(rmax(v[6], v[7]), v[8]);
      if (slack) nd = rmax(nd, rmax(gs * v[9], v[10]));
      res[0] = v[0];
      res[1] = v[5];
      res[2] = np;
      res[3] = nd;
      res[4] = v[0] / (R(1e-10) + np);
      res[5] = v[5] / (R(1e-10) + nd);
      const R cand = rmin(rmax(rho * r_sqrt(res[4] / res[5]), a.rho_min), a.rho_max);
      const R ratio = rmax(cand / rho, rho / cand);
      const bool conv = !((res[0] > a.eps_abs + a.eps_rel * res[2]) || (res[1] > a.eps_abs + a.eps_rel * res[3]));
      bool keep = iter < 2 || !mod_zero(iter, a.adapt_every);
      keep = keep || conv;
      keep = keep || ratio < a.rho_tol;
      if (!keep) rho = cand;  // (a chunk ends after an iteration that can change rho)
    }
  }
  finish(true);
}

}  // namespace tmpc
