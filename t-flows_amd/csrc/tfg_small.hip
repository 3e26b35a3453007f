// FP64 Jacobi / unpreconditioned CG of a small system in one launch.
//
// Below some ten thousand rows an iteration of the three-kernel form
// (tfg_kernels.hip) moves almost nothing and costs three launches, each with
// its own chain of state, partials, reduction and first loads: 14 us per
// iteration at 960 rows and at 40^3, as a replayed graph.  Here the whole loop
// runs in one kernel, with the rows' scaled values, x, r, p and the diagonal in
// registers:
//   k_tiny_cg   up to 2048 rows: one workgroup, everything handed over in LDS;
//               2.8 us per iteration at 960 rows.
//   k_small_cg  up to 65536 rows: workgroups that stay resident on ONE XCD, so
//               that they share an L2; 6.1 us per iteration at 6120 rows, 9.6 at 40^3, of
//               which the five hand-overs of an iteration are some 6.
//
// Same bits as the three-kernel form.  A thread group of 256 does what
// workgroups of that form do: the row blocks of one or two (VW) product
// workgroups (XcdWalk) and the pairs of one element-wise workgroup; every sum
// runs through the same trees (wavefront butterfly, the four wavefronts in
// order, then the butterfly over the workgroups' partials).
#include <algorithm>

#include "tfg_spmv.h"

namespace tfg {

namespace {

constexpr int kSmallRow = 8;   // entries of a row, at most
constexpr int kTinyGroups = 4; // thread groups of the one-workgroup kernel

typedef unsigned long long u64;

// What the stopping test needs (MODE): 0 the relative residual, 1 NRMS with
// norm, 2 NRMS over the x range; the sums of the update, in order.
template <int MODE>
struct Sums {
  static constexpr int NV = MODE == 2 ? 4 : 2;
  __device__ __forceinline__ static constexpr int op(int c) {
    return MODE == 2 && c == 1 ? OP_MIN : (MODE == 2 && c == 2 ? OP_MAX : OP_SUM);
  }
  __device__ __forceinline__ static double start(int c) {
    return op(c) == OP_MIN ? kHuge : (op(c) == OP_MAX ? -kHuge : 0.0);
  }
  __device__ __forceinline__ static double measure(const State* st, const double* s) {
    if (MODE == 0) return sqrt(s[0]) / st->bnorm;
    const double range = MODE == 1 ? fmax(st->norm - 0.0, kTiny) : fmax(s[2] - s[1], kTiny);
    return sqrt(s[0]) / range;
  }
};

// One row's update (Cg.f90:204-209) and its terms of the sums.  d: 1 / a_ii in
// mode 0, a_ii otherwise.
template <int PREC, int MODE>
__device__ __forceinline__ void update_row(double alpha, double& x, double& r, double p, double q,
                                           double d, double* s) {
  x = x + alpha * p;
  r = r - alpha * q;
  const double z = PREC == PREC_JACOBI ? r * (MODE == 0 ? d : 1.0 / d) : r;
  s[0] = s[0] + (MODE == 0 ? r * r : (r * r) / (d * d));
  if (MODE == 2) {
    s[1] = fmin(s[1], x);
    s[2] = fmax(s[2], x);
  }
  s[Sums<MODE>::NV - 1] = s[Sums<MODE>::NV - 1] + z * r;
}

// p = z + beta p (p = z in the first iteration)                Cg.f90:145-171
template <int PREC, int MODE>
__device__ __forceinline__ double direction(int k, double beta, double r, double d, double p) {
  const double z = PREC == PREC_JACOBI ? r * (MODE == 0 ? d : 1.0 / d) : r;
  return k == 1 ? z : z + beta * p;
}

// A row of the product: its length and where its columns' offsets are.
struct Row {
  int i, len, po, rs;
  bool own;
  __device__ __forceinline__ void find(const SmallArgs& a, int lb, int lt) {
    const int r0 = a.blk[lb], nr = a.blk[lb + 1] - r0;
    own = lt < nr;
    i = r0 + min(lt, nr - 1);
    const int pat = a.pat[i];
    rs = a.row[i];
    len = a.plen[pat];
    po = pat * kPatMax;
  }
  // the scaled values
  __device__ __forceinline__ void values(const SmallArgs& a, double fn, double (&v)[kSmallRow]) const {
#pragma unroll
    for (int u = 0; u < kSmallRow; ++u) v[u] = a.val[rs + min(u, len - 1)] * fn;
  }
  __device__ __forceinline__ double sum(const double (&v)[kSmallRow],
                                        const double (&x)[kSmallRow]) const {
    double acc = 0.0;
#pragma unroll
    for (int u = 0; u < kSmallRow; ++u)
      if (u < len) acc = acc + v[u] * x[u];
    return acc;
  }
};

// Butterfly inside the wavefront (block_reduce's first part).
template <int NV>
__device__ __forceinline__ void wave_reduce(double (&w)[NV], const int (&ops)[NV]) {
  butterfly_step<32>(w, ops);
  butterfly_step<16>(w, ops);
  butterfly_step<8>(w, ops);
  butterfly_step<4>(w, ops);
  butterfly_step<2>(w, ops);
  butterfly_step<1>(w, ops);
}
// The four wavefronts of a group in order (its second part).
__device__ __forceinline__ double group_total(int op, const double* s) {
  double t = s[0];
  for (int w = 1; w < kBlock / 64; ++w) t = red_apply(op, t, s[w]);
  return t;
}

}  // namespace

// One workgroup.  Three barriers per iteration: p, the product's sums, the
// update's sums; every thread adds up the (at most eight) partials itself, in
// gather()'s order.
template <int PREC, int MODE, int VW>
__global__ __launch_bounds__(kTinyGroups* kBlock) void k_tiny_cg(SmallArgs a) {
  using S = Sums<MODE>;
  constexpr int NV = S::NV, kParts = kTinyGroups * VW, W = kBlock / 64;
  __shared__ double s_p[kParts * kBlock], s_q[kParts * kBlock];
  __shared__ double s_pq[kParts][W], s_up[kTinyGroups][NV][W], s_odd[4];
  __shared__ int s_off[kPatCount * kPatMax];
  State* st = a.st;
  if (st->done) return;
  const int tid = threadIdx.x, tg = tid / kBlock, lt = tid % kBlock, wv = lt / 64;
  const bool lane0 = (tid & 63) == 0;
  for (int t = tid; t < kPatCount * kPatMax; t += kTinyGroups * kBlock) s_off[t] = a.poff[t];
  const double fn = st->fn;
  Row row[VW];
  double val[VW][kSmallRow];
#pragma unroll
  for (int j = 0; j < VW; ++j) {
    const int g = tg * VW + j;
    row[j].find(a, min(g, a.g_spmv - 1), lt);
    row[j].values(a, fn, val[j]);
    row[j].own = row[j].own && g < a.g_spmv;
  }
  const int npair = a.n >> 1, k0 = st->kcur;
  const bool pair = tg < a.g_vec && tid < npair, odd = (a.n & 1) && tid == 0;
  dbl2 r{0.0, 0.0}, x{0.0, 0.0}, d{1.0, 1.0}, p{0.0, 0.0};
  if (pair) {
    r = reinterpret_cast<const dbl2*>(a.r)[tid];
    x = reinterpret_cast<const dbl2*>(a.x)[tid];
    d = reinterpret_cast<const dbl2*>(a.ad)[tid];
    if (k0 > 1) p = reinterpret_cast<const dbl2*>(a.p)[tid];
  }
  if (odd) {
    s_odd[0] = a.r[a.n - 1];
    s_odd[1] = a.x[a.n - 1];
    s_odd[2] = a.ad[a.n - 1];
    s_odd[3] = k0 > 1 ? a.p[a.n - 1] : 0.0;
  }
  // gather()'s butterfly over at most eight partials: lanes 4, 2, 1 apart
  auto over = [](int op, const double (&w)[8]) {
    const double a04 = red_apply(op, w[0], w[4]), a26 = red_apply(op, w[2], w[6]);
    const double a15 = red_apply(op, w[1], w[5]), a37 = red_apply(op, w[3], w[7]);
    return red_apply(op, red_apply(op, a04, a26), red_apply(op, a15, a37));
  };
  double rho = st->rho[k0 & 1], beta = k0 > 1 ? st->beta : 0.0, res = st->res;
  const double tol = st->tol;
  int k = k0, stop = 0, status = TFG_OK;
  for (; k <= a.kend; ++k) {
    if (pair) {
      p.x = direction<PREC, MODE>(k, beta, r.x, d.x, p.x);
      p.y = direction<PREC, MODE>(k, beta, r.y, d.y, p.y);
      s_p[2 * tid] = p.x;
      s_p[2 * tid + 1] = p.y;
    }
    if (odd) {
      s_odd[3] = direction<PREC, MODE>(k, beta, s_odd[0], s_odd[2], s_odd[3]);
      s_p[a.n - 1] = s_odd[3];
    }
    __syncthreads();
    // q = (A fn) p and (p, q)                                 Cg.f90:176-195
    double v1[VW];
    int sum[VW];
#pragma unroll
    for (int j = 0; j < VW; ++j) {
      int po = row[j].po;
      asm volatile("" : "+v"(po));  // not eight columns kept per row: they would spill
      double xv[kSmallRow];
#pragma unroll
      for (int u = 0; u < kSmallRow; ++u)
        xv[u] = s_p[row[j].i + s_off[po + min(u, row[j].len - 1)]];
      const double q = row[j].sum(val[j], xv);
      v1[j] = 0.0;
      sum[j] = OP_SUM;
      if (row[j].own) {
        s_q[row[j].i] = q;
        v1[j] = v1[j] + xv[0] * q;
      }
    }
    wave_reduce<VW>(v1, sum);
    if (lane0) {
#pragma unroll
      for (int j = 0; j < VW; ++j) s_pq[tg * VW + j][wv] = v1[j];
    }
    __syncthreads();
    double w8[8];
#pragma unroll
    for (int g = 0; g < 8; ++g)
      w8[g] = g < kParts && g < a.g_spmv ? group_total(OP_SUM, s_pq[min(g, kParts - 1)]) : 0.0;
    const double pq = over(OP_SUM, w8);
    if (pq == 0.0 || !isfinite(pq)) {
      status = TFG_EBREAKDOWN;
      stop = 1;
      break;
    }
    const double alpha = rho / pq;                          // Cg.f90:198
    double v[NV];
    int ops[NV];
#pragma unroll
    for (int c = 0; c < NV; ++c) {
      ops[c] = S::op(c);
      v[c] = S::start(c);
    }
    if (pair) {
      double x0 = x.x, x1 = x.y, r0 = r.x, r1 = r.y;
      update_row<PREC, MODE>(alpha, x0, r0, p.x, s_q[2 * tid], d.x, v);
      update_row<PREC, MODE>(alpha, x1, r1, p.y, s_q[2 * tid + 1], d.y, v);
      x = dbl2{x0, x1};
      r = dbl2{r0, r1};
    }
    if (odd) {
      double xv = s_odd[1], rv = s_odd[0];
      update_row<PREC, MODE>(alpha, xv, rv, s_odd[3], s_q[a.n - 1], s_odd[2], v);
      s_odd[0] = rv;
      s_odd[1] = xv;
    }
    wave_reduce<NV>(v, ops);
    if (lane0) {
#pragma unroll
      for (int c = 0; c < NV; ++c) s_up[tg][c][wv] = v[c];
    }
    __syncthreads();
    double tot[NV];
#pragma unroll
    for (int c = 0; c < NV; ++c) {
#pragma unroll
      for (int g = 0; g < 8; ++g)
        w8[g] = g < kTinyGroups && g < a.g_vec ? group_total(ops[c], s_up[min(g, kTinyGroups - 1)][c])
                                               : red_identity(ops[c]);
      tot[c] = over(ops[c], w8);
    }
    // the stopping test (Cg.f90:214-222), the next rho and beta
    res = S::measure(st, tot);
    const bool fail = !isfinite(res);
    if (fail || res < tol) {
      status = fail ? TFG_EBREAKDOWN : TFG_OK;
      stop = 2;
      break;
    }
    beta = tot[NV - 1] / rho;
    rho = tot[NV - 1];
  }
  if (pair) {
    reinterpret_cast<dbl2*>(a.r)[tid] = r;
    reinterpret_cast<dbl2*>(a.x)[tid] = x;
    reinterpret_cast<dbl2*>(a.p)[tid] = p;
  }
  if (odd) {
    a.r[a.n - 1] = s_odd[0];
    a.x[a.n - 1] = s_odd[1];
    a.p[a.n - 1] = s_odd[3];
  }
  if (tid == 0) {
    st->res = res;
    st->status = status;
    if (stop) {
      st->niter = k;
      st->iter = stop == 2 ? k : k - 1;
      st->done = 1;
    } else {
      st->iter = k - 1;
      st->kcur = k;
      st->rho[k & 1] = rho;
      st->beta = beta;
    }
  }
}

// ---------------------------------------------------------------------------
// Several workgroups on one XCD.  What they hand each other is stored through
// to the shared L2 and read past the L1 (agent-scope loads); no L2 write-back
// or invalidation is needed, which is what a grid barrier across XCDs spends
// its 9 us (64 workgroups) to 50 us (512) on, and what one invalidation per
// hand-over would cost here too (29 us with 128 workgroups).
//
// Hand-over.  A partial sum goes out as two words, each half of the value with
// the iteration's tag in the other half: a reader that sees both tags has the
// value, whatever the order in which the words arrive.  Workgroup 0 polls the
// partials, forms the totals and sends them back the same way, in kSmallCopies
// copies on lines of their own; with every workgroup polling every partial the
// polls held up the stores (22 us per iteration with 128 workgroups).  p is handed over by one flag per workgroup, on a line of
// its own (stores to one line take turns, 33 ns each), stored after the
// workgroup's stores of p have been acknowledged.  Each slot is written again
// only after every reader has shown, by a later hand-over, that it has read it.
// Tags grow from launch to launch, so slots are never cleared.
//
// The workgroups have to be resident together.  They fit on the idle XCD
// (small_plan), one process runs one such launch per device at a time
// (XcdLease), and other kernels end.  Where another process's launch is in the
// way all the same, every wait is bounded (kSmallPolls): a workgroup whose wait
// ends without the tag, or that finds itself on another XCD than the others,
// raises State::refine and leaves, the others follow by their own bounds, and
// the host runs the solve again with the three-kernel form.  A cooperative
// launch would not do better: its queue is one process's at a time, and a second
// process's launch fails.
namespace {

constexpr int kGroups = 2;          // thread groups of a workgroup
constexpr int kLine = 16;           // words of a 128-byte line

__device__ __forceinline__ u64 load_shared(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_shared(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// element i of a workgroup-uniform array (32-bit byte offset)
__device__ __forceinline__ double load_shared(const double* p, int i) {
  typedef __attribute__((address_space(1))) const char gB;
  gB* base = (gB*)p;
  const u64* q = (const u64*)(base + 8u * (unsigned)i);
  return __longlong_as_double((long long)load_shared(q));
}
// this wave's stores have reached the L2
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ void store_slot(u64* slot, double v, unsigned tag) {
  const u64 b = (u64)__double_as_longlong(v);
  store_shared(slot, (b & 0xffffffff00000000ull) | tag);
  store_shared(slot + 1, (b << 32) | tag);
}
// NV slots `apart` words apart; false when a wait ends without the tag
template <int NV>
__device__ __forceinline__ bool poll_slots(const u64* slot, int apart, unsigned tag,
                                           double (&v)[NV]) {
#pragma unroll 1
  for (int n = 0; n < kSmallPolls; ++n) {
    bool all = true;
    u64 hi[NV], lo[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      hi[k] = load_shared(slot + k * apart);
      lo[k] = load_shared(slot + k * apart + 1);
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      v[k] = __longlong_as_double((long long)((hi[k] & 0xffffffff00000000ull) | (lo[k] >> 32)));
      all = all && (unsigned)hi[k] == tag && (unsigned)lo[k] == tag;
    }
    if (all) return true;
  }
  return false;
}

// Which row block slot j (of VW) of thread group u takes, and the product
// workgroup g it stands for: the walk of XcdWalk, in which a few of the first
// kXcds workgroups may have a second block (a.twice).  Those take both slots of
// the first thread groups, the others follow one to a slot.
struct Slot {
  int g, block;
  bool used, both;
  __device__ __forceinline__ Slot(const SmallArgs& a, int VW, int u, int j) {
    const int D = __popc(a.twice), G = a.g_spmv;
    both = u < D;
    if (both) {
      unsigned m = a.twice;
      for (int t = 0; t < u; ++t) m &= m - 1;
      g = __ffs(m) - 1;
    } else {
      g = VW * (u - D) + j;
      for (unsigned m = a.twice; m; m &= m - 1) g += g >= __ffs(m) - 1;
    }
    used = g < G;
    g = min(g, G - 1);
    if (G >= kXcds && G % kXcds == 0) {
      const int x = g % kXcds, l = g / kXcds;
      block = (int)(((long long)a.nblk * x) / kXcds) + l + (both ? j * (G / kXcds) : 0);
    } else {
      block = g;
    }
  }
};

}  // namespace

template <int PREC, int MODE, int VW>
__global__ __launch_bounds__(kGroups* kBlock, 4) void k_small_cg(SmallArgs a) {
  using S = Sums<MODE>;
  constexpr int NV = S::NV, W = kBlock / 64;
  __shared__ double s_w[kGroups * (VW > NV ? VW : NV) * W], s_t[NV * W], s_in[2], s_odd[4];
  __shared__ double s_v[VW][kSmallRow][kGroups * kBlock];  // in registers they would spill
  __shared__ int s_off[kPatCount * kPatMax], s_g[kGroups * VW], s_bad;
  if (blockIdx.x % kXcds) return;               // one XCD's workgroups only
  State* st = a.st;
  if (st->done) return;
  const int w = blockIdx.x / kXcds, tid = threadIdx.x;
  const int tg = tid / kBlock, lt = tid % kBlock, wv = lt / 64;
  const int G = a.g_spmv, GV = a.g_vec;
  const int NW = gridDim.x / kXcds, NWV = (GV + kGroups - 1) / kGroups;  // NWV: with pairs
  const bool lane0 = (tid & 63) == 0, lead = w == 0 && tid == 0, vec = w < NWV;
  for (int t = tid; t < kPatCount * kPatMax; t += kGroups * kBlock) s_off[t] = a.poff[t];
  // the XCD this workgroup runs on (hardware register XCC_ID), the same for all
  const unsigned xcc = __builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11));
  const u64 here = ((u64)xcc << 32) | a.tag;
  if (tid == 0) {
    s_bad = 0;
    store_shared(a.xcd + w, here);
  }
  __syncthreads();
  if (tid < NW) {
    u64 f = 0;
#pragma unroll 1
    for (int n = 0; n < a.polls && (unsigned)f != a.tag; ++n) f = load_shared(a.xcd + tid);
    if (f != here) s_bad = 1;
  }
  __syncthreads();
  if (s_bad) {
    if (tid == 0) st->refine = 1;
    return;
  }
  const int k0 = st->kcur;
  const double fn = st->fn;
  // this thread's rows: one of each slot's block
  Row row[VW];
  bool both = false;
#pragma unroll
  for (int j = 0; j < VW; ++j) {
    const Slot s(a, VW, w * kGroups + tg, j);
    double v[kSmallRow];
    row[j].find(a, s.block, lt);
    row[j].own = row[j].own && s.used;
    row[j].values(a, fn, v);
    both = s.both;
#pragma unroll
    for (int u = 0; u < kSmallRow; ++u) s_v[j][u][tid] = v[u];
    if (lt == 0) s_g[tg * VW + j] = s.used && !(s.both && j) ? s.g : -1;
  }
  // its pair of rows, and the last row of an odd number (thread 0 of
  // workgroup 0, in LDS: r, x, diagonal, p)
  const int npair = a.n >> 1, gv = w * kGroups + tg, t0 = gv * kBlock + lt;
  const bool pair = gv < GV && t0 < npair, odd = (a.n & 1) && lead;
  dbl2 r{0.0, 0.0}, x{0.0, 0.0}, d{1.0, 1.0}, p{0.0, 0.0};
  if (pair) {
    r = reinterpret_cast<const dbl2*>(a.r)[t0];
    x = reinterpret_cast<const dbl2*>(a.x)[t0];
    d = reinterpret_cast<const dbl2*>(a.ad)[t0];
    if (k0 > 1) p = reinterpret_cast<const dbl2*>(a.p)[t0];
  }
  if (odd) {
    s_odd[0] = a.r[a.n - 1];
    s_odd[1] = a.x[a.n - 1];
    s_odd[2] = a.ad[a.n - 1];
    s_odd[3] = k0 > 1 ? a.p[a.n - 1] : 0.0;
  }
  double rho = st->rho[k0 & 1], beta = k0 > 1 ? st->beta : 0.0, res = st->res;
  const double tol = st->tol;
  const u64* in = a.out + (w % kSmallCopies) * kLine;
  int k = k0, stop = 0, status = TFG_OK;
  for (; k <= a.kend; ++k) {
    const unsigned tag = a.tag + (unsigned)(k - k0) + 1u;
    if (vec) {
      if (pair) {
        p.x = direction<PREC, MODE>(k, beta, r.x, d.x, p.x);
        p.y = direction<PREC, MODE>(k, beta, r.y, d.y, p.y);
        reinterpret_cast<dbl2*>(a.p)[t0] = p;
      }
      if (odd) {
        s_odd[3] = direction<PREC, MODE>(k, beta, s_odd[0], s_odd[2], s_odd[3]);
        a.p[a.n - 1] = s_odd[3];
      }
      stores_done();
    }
    __syncthreads();  // every wave's stores are done; s_bad has been read
    if (vec && tid == 0) store_shared(a.flag + w * kLine, tag);
    if (tid < NWV) {
      bool ok = false;
#pragma unroll 1
      for (int n = 0; n < kSmallPolls && !ok; ++n)
        ok = (unsigned)load_shared(a.flag + tid * kLine) == tag;
      if (!ok) s_bad = 1;
    }
    __syncthreads();
    if (s_bad) break;
    // q = (A fn) p and (p, q)                                 Cg.f90:176-195
    double v1[VW];
    int sum[VW];
#pragma unroll
    for (int j = 0; j < VW; ++j) {
      double xv[kSmallRow];
      int po = row[j].po;
      asm volatile("" : "+v"(po));  // not eight addresses kept per row: they would spill
#pragma unroll
      for (int u = 0; u < kSmallRow; ++u)
        xv[u] = load_shared(a.p, row[j].i + s_off[po + min(u, row[j].len - 1)]);
      double v[kSmallRow];
#pragma unroll
      for (int u = 0; u < kSmallRow; ++u) v[u] = s_v[j][u][tid];
      const double q = row[j].sum(v, xv);
      v1[j] = 0.0;
      sum[j] = OP_SUM;
      if (row[j].own) {
        a.q[row[j].i] = q;
        v1[j] = v1[j] + xv[0] * q;
      }
    }
    if (VW == 2 && both) v1[0] = v1[0] + v1[VW - 1];
    wave_reduce<VW>(v1, sum);
    stores_done();
    if (lane0) {
#pragma unroll
      for (int j = 0; j < VW; ++j) s_w[(tg * VW + j) * W + wv] = v1[j];
    }
    __syncthreads();
    if (tid < kGroups * VW && s_g[tid] >= 0)
      store_slot(a.pq + 2 * s_g[tid], group_total(OP_SUM, s_w + tid * W), tag);
    if (w == 0) {
      if (tid < kBlock) {   // the partials, as gather() adds them up
        double t[1] = {0.0}, v[1] = {0.0};
        const int ops[1] = {OP_SUM};
        if (tid < G && !poll_slots<1>(a.pq + 2 * tid, 0, tag, t)) s_bad = 1;
        v[0] = v[0] + t[0];
        wave_reduce<1>(v, ops);
        if (lane0) s_t[wv] = v[0];
      }
    } else if (tid == 0) {
      double v[1];
      if (!poll_slots<1>(in, 0, tag, v)) s_bad = 1;
      s_in[0] = v[0];
    }
    __syncthreads();
    if (s_bad) break;
    const double pq = w == 0 ? group_total(OP_SUM, s_t) : s_in[0];
    if (w == 0 && tid < kSmallCopies) store_slot(a.out + tid * kLine, pq, tag);
    if (pq == 0.0 || !isfinite(pq)) {
      status = TFG_EBREAKDOWN;
      stop = 1;
      break;
    }
    const double alpha = rho / pq;                          // Cg.f90:198
    if (vec) {
      double v[NV];
      int ops[NV];
#pragma unroll
      for (int c = 0; c < NV; ++c) {
        ops[c] = S::op(c);
        v[c] = S::start(c);
      }
      if (pair) {
        const double q0 = load_shared(a.q, 2 * t0), q1 = load_shared(a.q, 2 * t0 + 1);
        double x0 = x.x, x1 = x.y, r0 = r.x, r1 = r.y;
        update_row<PREC, MODE>(alpha, x0, r0, p.x, q0, d.x, v);
        update_row<PREC, MODE>(alpha, x1, r1, p.y, q1, d.y, v);
        x = dbl2{x0, x1};
        r = dbl2{r0, r1};
      }
      if (odd) {
        double xl = s_odd[1], rl = s_odd[0];
        update_row<PREC, MODE>(alpha, xl, rl, s_odd[3], load_shared(a.q, a.n - 1), s_odd[2], v);
        s_odd[0] = rl;
        s_odd[1] = xl;
      }
      wave_reduce<NV>(v, ops);
      if (lane0) {
#pragma unroll
        for (int c = 0; c < NV; ++c) s_w[(tg * NV + c) * W + wv] = v[c];
      }
    }
    __syncthreads();  // also: s_in and s_bad have been read by every thread
    if (vec && tid < kGroups * NV) {
      const int g = tid / NV, c = tid % NV;
      if (w * kGroups + g < GV)
        store_slot(a.upd + 2 * (c * kBlock + w * kGroups + g), group_total(S::op(c), s_w + tid * W),
                   tag);
    }
    // the stopping test (Cg.f90:214-222), the next rho and beta
    if (w == 0) {
      if (tid < kBlock) {
        double t[NV], v[NV];
        int ops[NV];
#pragma unroll
        for (int c = 0; c < NV; ++c) {
          ops[c] = S::op(c);
          v[c] = red_identity(ops[c]);
        }
        if (tid < GV) {
          if (!poll_slots<NV>(a.upd + 2 * tid, 2 * kBlock, tag, t)) s_bad = 1;
#pragma unroll
          for (int c = 0; c < NV; ++c) v[c] = red_apply(ops[c], v[c], t[c]);
        }
        wave_reduce<NV>(v, ops);
        if (lane0) {
#pragma unroll
          for (int c = 0; c < NV; ++c) s_t[c * W + wv] = v[c];
        }
      }
    } else if (tid == 0) {
      double v[2];
      if (!poll_slots<2>(in + 2, 2, tag, v)) s_bad = 1;
      s_in[0] = v[0];
      s_in[1] = v[1];
    }
    __syncthreads();
    if (s_bad) break;
    double next;
    if (w == 0) {
      double tot[NV];
#pragma unroll
      for (int c = 0; c < NV; ++c) tot[c] = group_total(S::op(c), s_t + c * W);
      res = S::measure(st, tot);
      next = tot[NV - 1];
      if (tid < kSmallCopies) {
        store_slot(a.out + tid * kLine + 2, res, tag);
        store_slot(a.out + tid * kLine + 4, next, tag);
      }
    } else {
      res = s_in[0];
      next = s_in[1];
    }
    const bool fail = !isfinite(res);
    if (fail || res < tol) {
      status = fail ? TFG_EBREAKDOWN : TFG_OK;
      stop = 2;
      break;
    }
    beta = next / rho;
    rho = next;
  }
  if (s_bad) {
    if (tid == 0) st->refine = 1;
    return;
  }
  if (pair) {
    reinterpret_cast<dbl2*>(a.r)[t0] = r;
    reinterpret_cast<dbl2*>(a.x)[t0] = x;
  }
  if (odd) {
    a.r[a.n - 1] = s_odd[0];
    a.x[a.n - 1] = s_odd[1];
  }
  if (lead) {
    st->res = res;
    st->status = status;
    if (stop) {
      st->niter = k;
      st->iter = stop == 2 ? k : k - 1;
      st->done = 1;
    } else {
      st->iter = k - 1;
      st->kcur = k;
      st->rho[k & 1] = rho;
      st->beta = beta;
    }
  }
}

namespace {
template <int PREC, int VW, typename F>
void small_modes(bool tiny, int mode, F f) {
  if (tiny) {
    if (mode == 0) f(k_tiny_cg<PREC, 0, VW>);
    else if (mode == 1) f(k_tiny_cg<PREC, 1, VW>);
    else f(k_tiny_cg<PREC, 2, VW>);
  } else {
    if (mode == 0) f(k_small_cg<PREC, 0, VW>);
    else if (mode == 1) f(k_small_cg<PREC, 1, VW>);
    else f(k_small_cg<PREC, 2, VW>);
  }
}
template <typename F>
void small_dispatch(const SmallPlan& s, int prec, int mode, F f) {
  const bool tiny = s.workgroups == 1;
  if (prec == PREC_JACOBI) {
    if (s.share == 1) small_modes<PREC_JACOBI, 1>(tiny, mode, f);
    else small_modes<PREC_JACOBI, 2>(tiny, mode, f);
  } else {
    if (s.share == 1) small_modes<PREC_NONE, 1>(tiny, mode, f);
    else small_modes<PREC_NONE, 2>(tiny, mode, f);
  }
}
}  // namespace

// One workgroup where its thread groups hold every block and pair, else
// workgroups of kGroups thread groups.  Two slots per thread group where some
// product workgroup has two blocks, and above 64 blocks: fewer workgroups to
// wait for (us per iteration with one slot and two: 24 blocks 6.1 and 7.2,
// 128 blocks 8.2 and 7.5; 129 and more do not fit with one).
SmallPlan small_plan(int nblk, int g_spmv, int g_vec, int cu_per_xcd) {
  SmallPlan s{};
  if (nblk == g_spmv && g_spmv <= 2 * kTinyGroups && g_vec <= kTinyGroups) {
    s.workgroups = 1;
    s.share = g_spmv <= kTinyGroups ? 1 : 2;
    return s;
  }
  if (g_spmv > kBlock || g_vec > kBlock) return s;
  // product workgroups with a second block (XcdWalk); none may have a third
  if (g_spmv >= kXcds && g_spmv % kXcds == 0) {
    const int step = g_spmv / kXcds;
    for (int x = 0; x < kXcds; ++x) {
      const int count = (int)(((long long)nblk * (x + 1)) / kXcds - ((long long)nblk * x) / kXcds);
      if (count > step + 1) return s;
      if (count > step) s.twice |= 1u << x;
    }
  } else if (nblk != g_spmv) {
    return s;
  }
  const int two = __builtin_popcount(s.twice);
  for (s.share = two || g_spmv > 64 ? 2 : 1; s.share <= 2; ++s.share) {
    const int groups = two + (g_spmv - two + s.share - 1) / s.share;
    s.workgroups = (std::max(groups, g_vec) + kGroups - 1) / kGroups;
    int least = 1 << 30;
    for (int prec : {PREC_NONE, PREC_JACOBI})
      for (int mode = 0; mode < 3; ++mode)
        small_dispatch(s, prec, mode, [&](auto kernel) {
          int nb = 0;
          if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, kGroups * kBlock, 0) != hipSuccess)
            nb = 0;
          least = std::min(least, nb);
        });
    if (s.workgroups > 1 && s.workgroups <= std::min(least * cu_per_xcd, 64)) return s;
  }
  return SmallPlan{};
}

hipError_t launch_small_cg(hipStream_t stream, const SmallArgs& a, const SmallPlan& s, int prec,
                           int mode) {
  SmallArgs q = a;
  q.twice = s.twice;
  hipError_t e = hipErrorInvalidValue;
  small_dispatch(s, prec, mode, [&](auto kernel) {
    if (s.workgroups == 1)
      kernel<<<1, kTinyGroups * kBlock, 0, stream>>>(q);
    else
      kernel<<<kXcds * s.workgroups, kGroups * kBlock, 0, stream>>>(q);
    e = hipGetLastError();
  });
  return e;
}

}  // namespace tfg
