"""BiCGSTAB's early exit does not depend on the order in which workgroups start.

The update kernels' own source (tfg_nonsym.hip, tfg_ir_ns.hip) runs on the CPU
with one thread per workgroup and the workgroups one after the other, in every
order: a workgroup that starts after workgroup 0 has finished still takes its
rows' last step, and the next iteration's update leaves them alone."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "t-flows_amd", "csrc")
CLANG = "/opt/rocm/llvm/bin/clang++"

RUNTIME = """
#include <cmath>
#include <type_traits>
#define __device__
#define __host__
#define __global__
#define __shared__ static
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __builtin_amdgcn_sched_barrier(x)
struct dim3 { unsigned x, y, z; };
static dim3 blockIdx, gridDim, threadIdx;
static inline void __syncthreads() {}
typedef int hipError_t;
typedef void* hipStream_t;
typedef void* hipEvent_t;
static inline int min(int a, int b) { return a < b ? a : b; }
using std::fmax; using std::fmin; using std::isfinite;
"""

MAIN = """
namespace tfg {
typedef float f32;
template <int NV>
void publish(double (&v)[NV], const int (&)[NV], double* part, int stride, double*, double*) {
  for (int k = 0; k < NV; ++k) part[k * stride + blockIdx.x] = v[k];
}
template <int NV>
void block_reduce(double (&v)[NV], const int (&)[NV], double*, double* out) {
  for (int k = 0; k < NV; ++k) out[k] = v[k];
}
%s
}
#include <algorithm>
#include <cstdio>
using namespace tfg;
template <class T> int check() {
  constexpr int N = 7, G = 3, K = 4;   // workgroup 0 has three rows, the others two
  int bad = 0, order[G] = {0, 1, 2};
  do {
    double part[64] = {};
    T x[N], r[N], ad[N], v1[N], v2[N], v3[N], v4[N], rt[N];
    for (int i = 0; i < N; ++i) {
      x[i] = T(i); r[i] = T(-1); ad[i] = T(2); v1[i] = T(100 + i); v2[i] = T(10 * i);
      v3[i] = v4[i] = rt[i] = T(1000);
    }
    State st{};
    st.tol = 1e-3; st.bnorm = 1.0; st.criterion = TFG_CRIT_RELRES; st.alpha = 0.5;
    CgArgs a{};
    a.n = N; a.st = &st;
    a.pt.ext = part; a.pt.upd = part + 32; a.pt.pstride = 4; a.pt.g_vec = a.pt.g_spmv = G;
    for (int g = 0; g < G; ++g) part[3 * 4 + g] = 1e-9;   // ||s||^2, below tol^2
    gridDim = dim3{G, 1, 1};
    for (int k = K; k <= K + 2; ++k)     // the step, and launches after the stop
      for (int g : order) {
        blockIdx.x = g;
        RUN
      }
    for (int i = 0; i < N; ++i) bad += x[i] != T(i) + T(0.5) * T(10 * i) || r[i] != T(100 + i);
    bad += !st.done || st.niter != K || st.iter != K || st.status != TFG_OK;
  } while (std::next_permutation(order, order + G));
  return bad;
}
int main() { return check<REAL>() ? 1 : 0; }
"""

SHARED = [r"double red_apply\(", r"double red_identity\(", r"void gather\(", r"struct Sweep",
          r"void stream_items\(", r"void first_items\("]
RUN64 = """
        a.x = x; a.r = r; a.ad = ad;
        NsArgs s{};
        s.v1 = v1; s.v2 = v2; s.v3 = v3; s.v4 = v4; s.rt = rt;
        k_bcgs_update<PREC_JACOBI>(a, s, k);
"""
RUN32 = """
        IrArgs f{};
        f.e32 = x; f.r32 = r; f.rd32 = ad;
        NsArgs32 s{};
        s.v1 = v1; s.v2 = v2; s.v3 = v3; s.v4 = v4; s.rt = rt;
        k_bcgs32_update<PREC_JACOBI>(a, f, s, &st, k);
"""


def _source(name):
    with open(os.path.join(CSRC, name)) as f:
        return f.read()


def _entity(text, head):
    """The definition whose first lines match `head`, with its template line."""
    m = re.search(r"(?:^template[^\n]*\n)?^[^\n;]*" + head, text, re.M)
    assert m, head
    depth, i = 0, text.index("{", m.end())
    while True:
        depth += {"{": 1, "}": -1}.get(text[i], 0)
        i += 1
        if depth == 0:
            return text[m.start():i] + (";\n" if "struct" in head else "\n")


@pytest.mark.parametrize("source,helpers,kernel,run,real", [
    ("tfg_nonsym.hip", [r"bool lead1\(", r"double measure1\(", r"void stop_at\(", r"double mprec\("],
     "k_bcgs_update", RUN64, "double"),
    ("tfg_ir_ns.hip", [r"bool lead2\(", r"void stop2\(", r"f32 mp\("], "k_bcgs32_update", RUN32, "float"),
], ids=["fp64", "fp32"])
def test_every_order(tmp_path, source, helpers, kernel, run, real):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    internal, reduce_h, text = _source("tfg_internal.h"), _source("tfg_reduce.h"), _source(source)
    block = "constexpr int kBlock = 256;"
    assert internal.count(block) == 1
    (tmp_path / "tfg_internal.h").write_text(internal.replace(block, "constexpr int kBlock = 1;"))
    body = "".join(_entity(reduce_h, h) for h in SHARED)
    body += "".join(c + "\n" for c in re.findall(r"^constexpr int kNsItems = .*$", text, re.M))
    body += "".join(_entity(text, h) for h in helpers + [rf"void {kernel}\("])
    main = MAIN.replace("%s", body).replace("RUN", run).replace("REAL", real)
    (tmp_path / "order.cpp").write_text('#include "tfg_internal.h"\n' + main)
    inc = os.path.join(os.path.dirname(os.path.dirname(CSRC)), "include")
    exe = str(tmp_path / "order")
    build = subprocess.run([CLANG, "-std=c++17", "-O1", "-w", "-I", str(tmp_path), "-I", inc, "-o", exe,
                            str(tmp_path / "order.cpp")], capture_output=True, text=True)
    assert build.returncode == 0, build.stderr
    assert subprocess.run([exe]).returncode == 0
