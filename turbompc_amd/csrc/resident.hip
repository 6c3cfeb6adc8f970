// Launches of the on-chip ADMM path: the shape classes it is built for and the
// choice of workgroup (resident.hpp, resident_factor.hpp).
#include "resident_api.hpp"

#include <algorithm>

#include "resident.hpp"

namespace tmpc {
namespace {

constexpr size_t kLdsBytes = 160 * 1024;

// A shape class: at most NX states, NU controls, MM inequality rows per stage, in
// groups of GL lanes (NX + NU + MM <= GL).  Forms of the kernel:
//   fp32, KF stages per group, up to eight wavefronts, two per SIMD (256 registers);
//   fp32, KD stages per group, up to four wavefronts, so that two workgroups share a
//     CU (KD = 0: not built);
//   fp64, K64 stages per group, up to four wavefronts, one per SIMD (512 registers).
// BF, B64: the problems per CU up to which the path is taken (0: at any B): where it is
// the faster one, but for C2 in fp32.  There the two paths' rounding differs, and about
// one obstacle problem in ten thousand amplifies it to 1e-3 .. 1e-2 of its controls (8 SQP
// steps of 16384 problems against fp64, twelve draws: worst control 1e-4 .. 5e-3 off
// on-chip, 4e-4 .. 6e-3 off streaming, relative norm 2.0e-6 and 3.6e-6), so batches large
// enough to hold such problems keep the results that they had.
// A CU works on one or two problems at a time, each for as long as its chains take,
// so the time grows with B from 256 on; the streaming kernel leaves the chip idle up
// to about 2048 problems and then runs at its rate over memory.  QP solves of 20
// iterations, on-chip / streaming in us:
//   C4 fp32, T = 41: 319 / 1412 at B = 256, 1029 / 1696 at 2048, 1534 / 1909 at 3072,
//     1951 / 2081 at 4096 (there the streaming kernel's records, which an SQP step
//     relinearizes in place, decide: 5 steps 10222 / 10038); T = 21: 626 / 912 at 2048,
//     1179 / 1110 at 4096
//   C4 fp64, T = 41: 399 / 1629 at 256, 2053 / 2171 at 2048, 4060 / 4171 at 4096
//   C1 fp32, T = 101: 925 / 5285 at 512, 3275 / 5495 at 2048, 6772 / 6778 at 4096 (50
//     iterations; 2840 / 3181 of 20); fp64: 1175 / 6259 at 512, 4267 / 6663 at 2048,
//     8384 / 14317 at 4096
//   C2 fp32, T = 61: 1385 / 2675 at 2048, 2582 / 3377 at 4096, 9950 / 12842 at 16384; fp64, T = 48:
//     2542 / 2657 at 2048, 4901 / 5118 at 4096
//   C3, T = 51: 660 / 2758 at 512, 4060 / 10603 at 4096; fp64 908 / 3353 at 512
//   C0 fp64, T = 21: 169 / 778 at 64, 944 / 964 at 4096, 3598 / 3572 at 16384; fp32:
//     556 / 836 at 4096, 1761 / 2460 at 16384
template <int NX_, int NU_, int MM_, int GL_, int KF_, int KD_, int K64_, int BF_, int B64_>
struct Cls {
  static constexpr int NX = NX_, NU = NU_, MM = MM_, GL = GL_, KF = KF_, KD = KD_, K64 = K64_, BF = BF_, B64 = B64_;
};
using C0 = Cls<4, 2, 4, 16, 4, 0, 4, 0, 16>;
using C1 = Cls<6, 3, 4, 16, 4, 0, 7, 16, 0>;
using C2 = Cls<6, 3, 12, 32, 4, 8, 8, 8, 0>;
using C3 = Cls<12, 4, 16, 32, 4, 0, 7, 0, 0>;
using C4 = Cls<13, 4, 4, 32, 4, 6, 6, 12, 16>;
constexpr int kClasses = 5;

template <typename F>
auto with_class(int cls, F&& f) {
  switch (cls) {
    case 0: return f(C0{});
    case 1: return f(C1{});
    case 2: return f(C2{});
    case 3: return f(C3{});
    default: return f(C4{});
  }
}

constexpr int kCUs = 256;
constexpr int kSplitProblems = 4 * kCUs;

template <typename R>
ResPlan plan(const Dims& d, int cls, bool const_g) {
  return with_class(cls, [&](auto c) {
    using C = decltype(c);
    ResPlan p;
    auto fit = [&](int ks, int max_nw, size_t lds_max, bool dense) {
      const int per = (kWave / C::GL) * ks;  // stages per wavefront
      const int nw = (d.T + per - 1) / per;
      if (nw > max_nw) return false;
      const size_t lds = (size_t)res_lds<R, C::NX, C::NU, C::MM>(d.T, const_g, nw).total * sizeof(R);
      if (lds > lds_max) return false;
      p.cls = cls;
      p.nw = nw;
      p.lds = lds;
      p.dense = dense;
      return true;
    };
    if (sizeof(R) == 8) {
      fit(C::K64, 4, kLdsBytes, false);
      return p;
    }
    if (C::KD > 0 && d.B > kCUs && fit(C::KD, 4, kLdsBytes / 2, true)) return p;
    fit(C::KF, 8, kLdsBytes, false);
    return p;
  });
}

}  // namespace

int resident_class(const Dims& d) {
  const int nx = d.nx, nu = d.n - d.nx, m = d.m;
  for (int c = 0; c < kClasses; ++c)
    if (with_class(c, [&](auto k) {
          using C = decltype(k);
          return nu >= 1 && nx <= C::NX && nu <= C::NU && m <= C::MM;
        }))
      return c;
  return -1;
}

ResPlan resident_plan(const Dims& d, size_t elem, bool const_g) {
  const int cls = resident_class(d);
  if (cls < 0) return ResPlan{};
  return elem == 4 ? plan<float>(d, cls, const_g) : plan<double>(d, cls, const_g);
}

bool resident_pays(int cls, int B, size_t elem) {
  return with_class(cls, [&](auto c) {
    using C = decltype(c);
    const int per_cu = elem == 4 ? C::BF : C::B64;
    return per_cu == 0 || B <= per_cu * kCUs;
  });
}

size_t resident_v_bytes(const Dims& d, size_t elem, int cls) {
  return with_class(cls, [&](auto c) {
    using C = decltype(c);
    const size_t vw = elem == 4 ? ResGeom<float, C::NX, C::NU>::VW : ResGeom<double, C::NX, C::NU>::VW;
    return (size_t)d.B * d.T * vw * elem;
  });
}

size_t resident_l_bytes(const Dims& d, size_t elem, int cls) {
  return with_class(cls, [&](auto c) {
    using C = decltype(c);
    return (size_t)d.B * d.T * ResGeom<float, C::NX, C::NU>::LW * elem;
  });
}

template <typename R>
hipError_t resident_factor(hipStream_t s, int cls, bool const_g, const ResFactorArgs<R>& a) {
  with_class(cls, [&](auto c) {
    using C = decltype(c);
    const dim3 grid((unsigned)((a.d.B + 1) / 2));
    auto launch = [&](auto split) {
      constexpr bool SP = decltype(split)::value;
      const dim3 block(SP ? 2 * kWave : kWave);
      if (const_g)
        hipLaunchKernelGGL((resident_factor_kernel<R, C::NX, C::NU, C::MM, true, SP>), grid, block, 0, s, a);
      else
        hipLaunchKernelGGL((resident_factor_kernel<R, C::NX, C::NU, C::MM, false, SP>), grid, block, 0, s, a);
    };
    // Two wavefronts for two problems while that leaves a SIMD to each.  Factorization and
    // one iteration, one wavefront / two, us: C4 fp32, T = 41 176 / 139 for one problem,
    // 241 / 208 for 1024, 359 / 395 for 2048; C2, T = 61 230 / 210 for 1024, 530 / 583 for
    // 4096; C3, T = 51 273 / 236 for 1024, 406 / 436 for 2048; C0 (blocks too small to pay
    // for the exchange) fp64, T = 21 87.4 / 90.6 for 64.
    if constexpr (C::NX > 4)
      if (a.d.B <= kSplitProblems) {
        launch(std::true_type{});
        return 0;
      }
    launch(std::false_type{});
    return 0;
  });
  return hipGetLastError();
}

template <typename R>
hipError_t resident_iterate(hipStream_t s, const ResPlan& p, const ResArgs<R>& a) {
  with_class(p.cls, [&](auto c) {
    using C = decltype(c);
    auto launch = [&](auto k) {
      if (p.lds > 65536)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)p.lds);
      hipLaunchKernelGGL(k, dim3((unsigned)a.d.B), dim3((unsigned)(p.nw * kWave)), p.lds, s, a);
    };
    if constexpr (sizeof(R) == 8) {
      launch(admm_resident_kernel<R, C::NX, C::NU, C::MM, C::GL, C::K64, 256, 1>);
    } else {
      if constexpr (C::KD > 0)
        if (p.dense) {
          launch(admm_resident_kernel<R, C::NX, C::NU, C::MM, C::GL, C::KD, 256, 2>);
          return 0;
        }
      launch(admm_resident_kernel<R, C::NX, C::NU, C::MM, C::GL, C::KF, 512, 2>);
    }
    return 0;
  });
  return hipGetLastError();
}

template hipError_t resident_factor<float>(hipStream_t, int, bool, const ResFactorArgs<float>&);
template hipError_t resident_factor<double>(hipStream_t, int, bool, const ResFactorArgs<double>&);
template hipError_t resident_iterate<float>(hipStream_t, const ResPlan&, const ResArgs<float>&);
template hipError_t resident_iterate<double>(hipStream_t, const ResPlan&, const ResArgs<double>&);

}  // namespace tmpc
