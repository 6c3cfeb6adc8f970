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
// takes: whether the path takes B problems, where it is the faster one, but for C2 in fp32
// (below).  A CU works on k problems at a time (k: the workgroups it holds, which follows
// from T), each for as long as its chains take, so the time grows with B from 256 k on;
// the streaming kernel leaves the chip idle up to about 2048 problems and then runs at its
// rate over memory, or, in fp64 with one wavefront per SIMD (C2, C4), in rounds of 2048.
// Between two chunks (adaptive rho) a workgroup gives its iterate up and fetches its blocks
// again, which the streaming kernel does in every iteration anyway, and an SQP step's
// records (C2, C4) are packed already: below few iterations per chunk, and again below 4,
// the line lies lower.  Measured, on-chip over streaming time; QP solves of 20 iterations
// where nothing else stands, "chunks of 5": rho adapted every 5 of 20:
//   C4 fp32, 3 SQP steps: T = 41 (k = 2) 0.87 at B = 3072 (4096, 5 steps: 10222 us against
//     10038); of one iteration 0.80 at 2048, 1.10 at 3072; T = 42 (k = 1) 0.96 at 2560,
//     1.06 at 3072
//   C4 fp64, 3 SQP steps: T = 21 (k = 2) 0.86 at 2048, 0.89 at 4096, of 5 iterations 0.91
//     and 0.99, of one 0.96 and 1.10; T = 25 (k = 1) 0.60 at 1792, 1.05 at 2048, 1.10 at
//     4096, T = 36 0.72 at 2412, 0.85 at 3229; a chunk per iteration T = 21 0.73 at 1536,
//     1.12 at 2048, T = 41 1.14 at 3072
//   C1 fp32: T = 65 (k = 1) 0.84 at 3072, 1.07 at 4096; T = 57 (k = 2) 0.67 at 4096
//   C1 fp64: T = 57 (k = 1) 0.95 at 4096, 1.01 at 16384, but in chunks of 25 (of 100) 1.05
//     and 1.11, of 5 0.90 at 2048, 1.13 at 3072; T = 85, chunks of 25 0.64 and 0.84 (past
//     T = 60 the streaming kernel's LDS holds fewer wavefronts)
//   C2 fp32, T = 61: 1385 us against 2675 at 2048, 2582 against 3377 at 4096, 9950 against
//     12842 at 16384.  The streaming kernel keeps the batches past 2048 all the same: the
//     two paths round differently, and about one problem in ten thousand amplifies that to
//     1e-3 .. 1e-2 of its controls (on either path), so moving the line changes results of
//     large batches beyond rounding.  On-chip is no further from 64 bits there.
//   C2 fp64, 3 SQP steps of 30 iterations: T = 33 (k = 1) 0.99 at 2048, 1.01 at 8192, 1.15
//     at 16384 (three problems per wavefront there), T = 61 0.85, 0.86, 0.93; of 3
//     iterations T = 33 1.07 at 2048; T = 32 (k = 2) 0.74 at 8192; a chunk per iteration
//     1.28 at 3072
//   C3: T = 51 0.24 at 512, 0.38 at 4096; fp64 0.27 at 512; a chunk per iteration fp64, T =
//     31 0.95 at 4096, 1.03 at 8192
//   C0 fp64: T = 17 (k = 2) 0.77 at 2048, 1.06 at 4096, T = 32 0.83 at 4096; T = 33 (k = 1)
//     0.85 at 2048; with the solver's defaults T = 33 1.20 at 3072, T = 61 0.92; chunks of
//     5 T = 17 0.95 at 2048, 1.36 at 4096; fp32: T = 33 (k = 2) 0.88 at 4096, 1.10 at
//     16384, T = 17 (k = 4) 0.80 at 16384, in chunks of 5 1.12
enum class Chunks { kLong, kShort, kTiny };  // iterations between refactorizations

constexpr int kCUs = 256;
// at most p problems per CU (0: any number)
constexpr bool per_cu_at_most(int B, int p) { return p == 0 || B <= p * kCUs; }
// Against a streaming kernel with one wavefront per SIMD: below 2048 problems a wavefront
// holds one of them, and past 1024 the SIMDs hold two in turn; from 2048 on it holds two.
// r rounds of the CUs take as long as 2048 problems there.
constexpr bool within_rounds(int B, int r) { return B < 2048 || (B + kCUs - 1) / kCUs <= r * ((B + 2047) / 2048); }

template <int NX_, int NU_, int MM_, int GL_, int KF_, int KD_, int K64_>
struct Cls {
  static constexpr int NX = NX_, NU = NU_, MM = MM_, GL = GL_, KF = KF_, KD = KD_, K64 = K64_;
};
struct C0 : Cls<4, 2, 4, 16, 4, 0, 4> {
  static constexpr int few(bool, int, bool chunked) { return chunked ? 16 : 0; }
  static constexpr int most(bool f64, int k, int T, Chunks c) {
    if (c == Chunks::kTiny) return f64 ? (k >= 4 ? 8 : (k >= 2 ? 5 : 4)) : (k >= 8 ? 16 : (k >= 2 ? 8 : 4));
    if (!f64) return k >= 4 ? (c == Chunks::kShort && k < 8 ? 32 : 0) : (k >= 2 && c == Chunks::kLong ? 16 : 8);
    if (c == Chunks::kShort) return k >= 4 ? 16 : (k >= 2 ? 8 : 6);
    return k >= 4 ? 16 : (k >= 2 ? std::min(16, 4 * T / 5) : std::min(12, T / 4));
  }
  static constexpr bool takes(int B, bool f64, int k, int T, Chunks c) { return per_cu_at_most(B, most(f64, k, T, c)); }
};
struct C1 : Cls<6, 3, 4, 16, 4, 0, 7> {
  static constexpr int few(bool, int, bool chunked) { return chunked ? 16 : 0; }
  static constexpr int most(bool f64, int k, int T, Chunks c) {
    if (c == Chunks::kTiny) return f64 ? (k >= 4 ? 8 : (k >= 2 ? 7 : 5)) : (k == 2 || k == 3 ? 12 : 8);
    if (!f64) return k >= 2 ? 16 : 12;
    if (c == Chunks::kShort) return k >= 4 ? 16 : (k >= 2 ? 12 : 8);
    return k < 2 && T <= 60 ? 12 : 0;
  }
  static constexpr bool takes(int B, bool f64, int k, int T, Chunks c) { return per_cu_at_most(B, most(f64, k, T, c)); }
};
struct C2 : Cls<6, 3, 12, 32, 4, 8, 8> {
  static constexpr int few(bool, int T, bool chunked) { return T >= 56 && !chunked ? 4 : 16; }
  static constexpr bool takes(int B, bool f64, int k, int T, Chunks c) {
    if (!f64) return per_cu_at_most(B, 8);
    if (c == Chunks::kLong) return k >= 2 || T >= 56 || (B < 12288 && within_rounds(B, 8));
    return B < 12288 && within_rounds(B, c == Chunks::kTiny ? 0 : (k >= 4 ? 8 : 7));
  }
};
struct C3 : Cls<12, 4, 16, 32, 4, 0, 7> {
  static constexpr int few(bool, int, bool chunked) { return chunked ? 16 : 0; }
  static constexpr bool takes(int B, bool f64, int, int, Chunks c) {
    return per_cu_at_most(B, f64 && c == Chunks::kTiny ? 16 : 0);
  }
};
struct C4 : Cls<13, 4, 4, 32, 4, 6, 6> {
  static constexpr int few(bool f64, int, bool chunked) { return f64 || chunked ? 8 : 5; }
  static constexpr bool takes(int B, bool f64, int k, int, Chunks c) {
    if (!f64) return per_cu_at_most(B, c != Chunks::kLong ? 8 : (k < 2 ? 10 : 12));
    return per_cu_at_most(B, 16) && within_rounds(B, c == Chunks::kTiny ? 0 : (c == Chunks::kShort || k < 2 ? 7 : 8));
  }
};
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

constexpr int kSplitProblems = 4 * kCUs;

template <typename R>
ResPlan plan(const Dims& d, int cls, bool const_g) {
  return with_class(cls, [&](auto c) {
    using C = decltype(c);
    ResPlan p;
    // ks stages per group, at most max_nw wavefronts and lds_max bytes; cu_nw wavefronts
    // fill a CU.  The fewest wavefronts that hold T, and more where each then has fewer
    // stages and the CU no fewer workgroups (or its SIMDs would idle).  Three SQP steps of
    // 20 iterations, 4096 problems, fp64, NX = 13: T = 24 on 2 wavefronts 11136 us, on 4
    // 7876; T = 31 on 3 11522, on 4 9578.
    auto fit = [&](int ks, int max_nw, int cu_nw, size_t lds_max, bool dense) {
      constexpr int GPW = kWave / C::GL;  // stages a wavefront holds at once
      auto lds = [&](int nw) {
        return (size_t)res_lds<R, C::NX, C::NU, C::MM>(d.T, const_g, nw).total * sizeof(R);
      };
      auto per_cu = [&](int nw) { return std::min<size_t>(cu_nw / nw, kLdsBytes / lds(nw)); };
      auto passes = [&](int nw) { return (d.T + GPW * nw - 1) / (GPW * nw); };
      int nw = passes(ks);  // the least with passes(nw) <= ks
      if (nw > max_nw || lds(nw) > lds_max) return false;
      for (int w = nw + 1; w <= max_nw; ++w)
        if (lds(w) <= lds_max && passes(w) < passes(nw) &&
            (per_cu(w) == per_cu(nw) || (per_cu(nw) * nw < 4 && per_cu(w) * w > per_cu(nw) * nw)))
          nw = w;
      p.cls = cls;
      p.nw = nw;
      p.per_cu = (int)per_cu(nw);
      p.lds = lds(nw);
      p.dense = dense;
      return true;
    };
    if (sizeof(R) == 8) {
      fit(C::K64, 4, 4, kLdsBytes, false);
      return p;
    }
    if (C::KD > 0 && d.B > kCUs && fit(C::KD, 4, 8, kLdsBytes / 2, true)) return p;
    fit(C::KF, 8, 8, kLdsBytes, false);
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

bool resident_pays(const ResPlan& p, const Dims& d, size_t elem, int iters, int chunks) {
  return with_class(p.cls, [&](auto c) {
    using C = decltype(c);
    const bool f64 = elem == 8, chunked = chunks > 1;
    const bool few = iters < (int64_t)C::few(f64, d.T, chunked) * chunks;
    const Chunks how = !few ? Chunks::kLong : (chunked && iters < (int64_t)4 * chunks ? Chunks::kTiny : Chunks::kShort);
    return C::takes(d.B, f64, p.per_cu, d.T, how);
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
