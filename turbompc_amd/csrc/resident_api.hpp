// Host interface of the on-chip ADMM path (resident.hip), a translation unit of
// its own so that it compiles beside capi.hip.
#pragma once
#include <stddef.h>

#include "resident_args.hpp"

namespace tmpc {

// How a problem runs on the on-chip path: the shape class, wavefronts per
// workgroup, workgroups a CU holds and LDS bytes; cls < 0: it does not.
struct ResPlan {
  int cls = -1, nw = 0, per_cu = 0;
  bool dense = false;  // the form of which two workgroups share a CU
  size_t lds = 0;
};

// The shape class of d (its block widths alone; -1: none).
int resident_class(const Dims& d);
// The plan for elements of elem bytes; const_g: one G for all stages and problems.
ResPlan resident_plan(const Dims& d, size_t elem, bool const_g);
// Whether the path beats the streaming kernel at d.B problems: iters iterations in
// chunks chunks (a refactorization between them).
bool resident_pays(const ResPlan& p, const Dims& d, size_t elem, int iters, int chunks);
// Bytes of the factor arrays V and L of resident_factor.hpp.
size_t resident_v_bytes(const Dims& d, size_t elem, int cls);
size_t resident_l_bytes(const Dims& d, size_t elem, int cls);

template <typename R>
hipError_t resident_factor(hipStream_t s, int cls, bool const_g, const ResFactorArgs<R>& a);
template <typename R>
hipError_t resident_iterate(hipStream_t s, const ResPlan& p, const ResArgs<R>& a);

}  // namespace tmpc
