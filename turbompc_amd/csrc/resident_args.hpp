// Kernel arguments of the on-chip ADMM path (resident_factor.hpp, resident.hpp).
#pragma once
#include "common.hpp"

namespace tmpc {

template <typename R>
struct ResFactorArgs {
  Dims d;  // n = nq: the QP's own widths
  const R *D, *Am, *G, *A0, *rho;
  R sigma, rho_f_factor;
  int32_t* ctl;  // not null: only problems whose refactor flag is set
  R *V, *L;
};

template <typename R>
struct ResArgs {
  Dims d;  // n = nq: the QP's own widths
  const R *V, *L;
  const R *D, *q, *A0, *Am, *G, *l, *u, *c0, *c, *slack_w;
  R *x, *z, *y_g, *y_f0, *y_f, *xi, *rho;
  int32_t* ctl;
  R* res;
  uint32_t* iters_out;
  R sigma, alpha, rho_f_factor, eps_abs, eps_rel, rho_min, rho_max, rho_tol;
  int max_iter, check_every, adapt_every, use_slack;
  int it_lo, it_hi, first_chunk, last_chunk, const_g;
  R *chk_conv, *chk_eq, *chk_iq, *chk_g;  // as in StreamArgs
  const uint8_t* act_in;
  uint8_t* act_out;
  R chk_tol;
};

}  // namespace tmpc
