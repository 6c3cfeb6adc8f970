"""The row products' inline assembly (csrc/row_dpp.hpp, stream_dpp.hpp, factor_rows.hpp,
common.hpp) where an accumulator starts from the same value as a source: the source
lives on after the block's first instruction, so the two may not share a register."""
import re
import subprocess

import pytest

from turbompc_amd import build

SOURCE = """
#include "factor_rows.hpp"
#include "row_dpp.hpp"
using namespace tmpc;
template <typename R, int N>
struct Row { R w[N]; };
template <typename R, int N>
__device__ Row<R, N> row(const R* p) {
  Row<R, N> r;
  for (int k = 0; k < N; ++k) r.w[k] = p[64 * (k + 1) + threadIdx.x];
  return r;
}
// the accumulator is the broadcast source (dead afterwards)
template <typename R, int N>
__global__ void source_fma(const R* p, R* o) {
  const R g = p[threadIdx.x];
  o[threadIdx.x] = row_fma<0>(row<R, N>(p).w, g, g);
}
template <typename R, int N>
__global__ void source_sum(const R* p, R* o) {
  const R g = p[threadIdx.x];
  o[threadIdx.x] = row_fma_sum(row<R, N>(p).w, g, g, p[threadIdx.x + 8192]);
}
template <typename R, int N>
__global__ void source_x2(const R* p, R* o) {
  R g = p[threadIdx.x], a = g, b = R(1);
  row_fma_x2<0>(g, row<R, N>(p).w, a, row<R, N>(p + 4096).w, b);
  o[threadIdx.x] = a * b;
}
template <typename R, int N>
__global__ void source_2(const R* p, R* o) {
  R g = p[threadIdx.x], h = p[threadIdx.x + 8192], a = g, b = h;
  row_fma_2(row<R, N>(p).w, g, a, row<R, N>(p + 4096).w, h, b);
  o[threadIdx.x] = a * b;
}
template <typename R, int N>
__global__ void source_3(const R* p, R* o) {
  R g = p[threadIdx.x], h = p[threadIdx.x + 8192], a = g, b = h, c = R(1);
  row_fma_3(row<R, N>(p).w, g, a, row<R, N>(p + 4096).w, h, b, row<R, N>(p + 4096).w, h, c);
  o[threadIdx.x] = a * b * c;
}
template <int N>
__global__ void source_axpy(const double* p, double* o) {
  auto r = row<double, N>(p);
  const double g = p[threadIdx.x], s = p[threadIdx.x + 8192];
  r.w[0] = g, r.w[1] = s;
  row_axpy(r.w, g, s);
  for (int k = 0; k < N; ++k) o[64 * k + threadIdx.x] = r.w[k];
}
template <int N>
__global__ void source_fac_axpy(const double* p, double* o) {
  auto r = row<double, N>(p);
  const double g = p[threadIdx.x], s = p[threadIdx.x + 8192];
  r.w[0] = g, r.w[1] = s;
  fac_axpy<N>(r.w, g, s);
  for (int k = 0; k < N; ++k) o[64 * k + threadIdx.x] = r.w[k];
}
// a zero accumulator and a zero source
__global__ void source_dot(const double* p, double* o) {
  auto r = row<double, 6>(p);
  r.w[2] = 0.0;
  o[threadIdx.x] = row_dot_dpp(r.w, p[threadIdx.x]) + dot_pair(r.w, RowPair<double>{p[threadIdx.x + 64], 0.0});
}
template __global__ void source_fma<float, 4>(const float*, float*);
template __global__ void source_fma<float, 13>(const float*, float*);
template __global__ void source_fma<double, 6>(const double*, double*);
template __global__ void source_sum<float, 13>(const float*, float*);
template __global__ void source_sum<double, 6>(const double*, double*);
template __global__ void source_x2<float, 3>(const float*, float*);
template __global__ void source_x2<double, 4>(const double*, double*);
template __global__ void source_2<float, 12>(const float*, float*);
template __global__ void source_2<double, 4>(const double*, double*);
template __global__ void source_3<float, 6>(const float*, float*);
template __global__ void source_3<double, 4>(const double*, double*);
template __global__ void source_axpy<6>(const double*, double*);
template __global__ void source_fac_axpy<9>(const double*, double*);
"""


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    d = tmp_path_factory.mktemp("asm")
    (d / "probe.hip").write_text(SOURCE)
    subprocess.run([build.hipcc(), f"--offload-arch={build.ARCH}", "-O3", "-std=c++17", "-S", "--cuda-device-only",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", str(build.PKG / "csrc"),
                    str(d / "probe.hip"), "-o", str(d / "probe.s")], check=True, capture_output=True, timeout=300)
    return (d / "probe.s").read_text()


def test_accumulators_share_no_register_with_a_later_source(assembly):
    kernel, blocks, bad = None, 0, []
    for block in re.findall(r"^(_Z\w+):|;;#ASMSTART\n(.*?);;#ASMEND", assembly, flags=re.S | re.M):
        if block[0]:
            kernel = block[0]
            continue
        written = set()
        for op in re.findall(r"v_(?:fmac|mul|add)_f(?:32|64)(?:_dpp)? ([^\s,]+), ([^\s,]+), ([^\s,]+)", block[1]):
            bad += [(kernel, op)] if written & set(op[1:]) or op[0] in op[1:] else []
            written.add(op[0])
        blocks += bool(written)
    assert blocks >= 14
    assert not bad, bad
