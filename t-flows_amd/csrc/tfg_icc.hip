// Incomplete Cholesky (DIC) preconditioner of Native_Mod on the GPU:
// Prec_Form.f90:68-78 and Prec_Solve.f90:64-92 (the reference's default
// "icc"), exact to the bit.
//
// Both recurrences run over rows in increasing order (form, forward
// substitution) or decreasing order (backward substitution), and row i needs
// the finished values of its lower (upper) neighbours only.  Rows are
// therefore grouped in dependency levels computed once per structure
// (level(i) = 1 + the largest level among the neighbours it reads), and one
// launch processes one level, one row per thread.  Every row performs the
// reference's operations in the reference's order on the same operands, so
// d, d_inv and z = M^-1 r are bit-identical to the serial sweeps.  A
// structured N^3 grid has 3N-2 levels per sweep.
//
// The scaled matrix of the solve is used (a_ij * fn rounded like the
// reference's in-place scaling, Cg.f90:77-84); the stand-alone building
// block passes fn = 1.
#include "tfg_spmv.h"

namespace tfg {

// d_inv_i = a_ii - sum_{k<i} d_k a_ik^2, d_i = 1 / d_inv_i     Prec_Form.f90:68-78
__global__ __launch_bounds__(kBlock) void k_icc_form(IccArgs c, const double* __restrict__ val,
                                                     const State* st, int lo, int hi) {
  const int t = lo + blockIdx.x * kBlock + threadIdx.x;
  if (t >= hi) return;
  const double fn = st ? st->fn : 1.0;
  const int i = c.rows_f[t];
  const int rs = c.row[i], re = c.row[i + 1];
  double sum = val[rs] * fn;
  for (int j = rs + 1; j < re; ++j) {
    const int k = c.col[j];
    if (k > i) break;
    const double a = val[j] * fn;
    sum = sum - c.d[k] * a * a;
  }
  c.dinv[i] = sum;
  c.d[i] = 1.0 / sum;
}

// forward substitution y_i = (r_i - sum_{k<i} a_ik y_k) d_i  Prec_Solve.f90:64-75
__global__ __launch_bounds__(kBlock) void k_icc_fwd(IccArgs c, const double* __restrict__ val,
                                                    const State* st, const double* __restrict__ r,
                                                    int lo, int hi) {
  if (st && st->done) return;
  const int t = lo + blockIdx.x * kBlock + threadIdx.x;
  if (t >= hi) return;
  const double fn = st ? st->fn : 1.0;
  const int i = c.rows_f[t];
  const int rs = c.row[i], re = c.row[i + 1];
  double sum = r[i];
  for (int j = rs + 1; j < re; ++j) {
    const int k = c.col[j];
    if (k > i) break;
    sum = sum - (val[j] * fn) * c.y[k];
  }
  c.y[i] = sum * c.d[i];
}

// z_i = (y_i d_inv_i - sum_{k>i} a_ik z_k) d_i, the upper terms taken from
// the end of the row down                                Prec_Solve.f90:77-92
__global__ __launch_bounds__(kBlock) void k_icc_bwd(IccArgs c, const double* __restrict__ val,
                                                    const State* st, double* __restrict__ z,
                                                    int lo, int hi) {
  if (st && st->done) return;
  const int t = lo + blockIdx.x * kBlock + threadIdx.x;
  if (t >= hi) return;
  const double fn = st ? st->fn : 1.0;
  const int i = c.rows_b[t];
  const int rs = c.row[i], re = c.row[i + 1];
  double sum = c.y[i] * c.dinv[i];
  for (int j = re - 1; j > rs; --j) {
    const int k = c.col[j];
    if (k < i) break;
    if (k < c.n) sum = sum - (val[j] * fn) * z[k];
  }
  z[i] = sum * c.d[i];
}

// ---------------------------------------------------------------------------
// Box grids: tiled sweeps
// ---------------------------------------------------------------------------
// On a box grid (rows (x, y, z), x slowest; every entry a box neighbour) row
// i's lower entries are, in CSR order, (x-1), (y-1), (z-1), and its upper
// entries from the end of the row down (x+1), (y+1), (z+1).  In sweep
// coordinates (u, v, w) = (x, y, z) for the form and the forward sweep and
// (nx-1-x, ny-1-y, nz-1-z) for the backward sweep, a row reads the finished
// values at u-1, v-1, w-1, in that order.  The grid is cut into tiles of at
// most kBoxTX x kBoxTY x kBoxTZ cells; a tile needs the tiles before it along
// u, v and w, so the tiles of one level X + Y + Z run in one launch, one
// workgroup each (61 launches per sweep at 200^3 instead of 598 row levels).
// A workgroup loads the three finished faces next to its tile and its cells'
// values, one thread per cell; one wave then runs the tile's own levels
// lu + lv + lw, a lane per (u, v) pencil, with no barrier between them.
// Every row does the reference's operations in the reference's order; an
// entry the row lacks is a zero in the diagonals and takes a zero product
// away, so for finite values the results are the same bits as the
// row-level sweeps'.

// the seven diagonals of val (entries a row lacks stay zero from the
// allocation)
__global__ __launch_bounds__(kBlock) void k_box_pack(IccArgs c, const double* __restrict__ val) {
  const BoxIcc& b = c.bx;
  const int nyz = b.ny * b.nz;
  const int stride = gridDim.x * kBlock;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < c.n; i += stride) {
    const int rs = c.row[i], re = c.row[i + 1];
    b.dg[i] = val[rs];
    for (int j = rs + 1; j < re; ++j) {
      const int off = c.col[j] - i;
      const double v = val[j];
      if (off == -nyz) b.lo[0][i] = v;
      else if (off == -b.nz) b.lo[1][i] = v;
      else if (off == -1) b.lo[2][i] = v;
      else if (off == 1) b.up[2][i] = v;
      else if (off == b.nz) b.up[1][i] = v;
      else if (off == nyz) b.up[0][i] = v;
    }
  }
}

// The tiles of level X + Y + Z = l: X = first + x, Y from lo(X) on.
struct TileLevel {
  int l, first, rows, span;  // X values, and the most Y values of one of them
  __host__ __device__ TileLevel(const BoxIcc& b, int level) : l(level) {
    first = max0(l - (b.nty - 1) - (b.ntz - 1));
    rows = (l < b.ntx - 1 ? l : b.ntx - 1) - first + 1;
    span = b.nty < b.ntz ? b.nty : b.ntz;
  }
  __host__ __device__ static int max0(int v) { return v > 0 ? v : 0; }
  __host__ __device__ int lo(const BoxIcc& b, int X) const { return max0(l - X - (b.ntz - 1)); }
  __host__ __device__ int hi(const BoxIcc& b, int X) const {
    return l - X < b.nty - 1 ? l - X : b.nty - 1;
  }
};

// v of the lane N below in the same 16 lanes; `other` for the first N lanes
template <int N>
__device__ __forceinline__ double row_shift(double other, double v) {
  const long long o = __double_as_longlong(other), b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)o, (int)b, 0x110 + N, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(b >> 32), 0x110 + N, 0xf, 0xf,
                                             false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// MODE 0 form: d_inv, d from a_ii and the lower entries   Prec_Form.f90:68-78
// MODE 1 forward: y from r                                Prec_Solve.f90:64-75
// MODE 2 backward: z from y                               Prec_Solve.f90:77-92
// The value the neighbours read (d, y, z) is `out`.
//
// A launch is a chain: its loads, the tile's levels, its stores, and each was
// cut to what it needs.  All loads leave together, before the stop flag is
// looked at.  The levels run on one wave, a lane per (u, v) pencil, each lane
// going up its pencil, and a step is bound by the instructions of that wave:
// - w - 1 is the lane's own last result, u - 1 and every other v - 1 a shift
//   inside 16 lanes;
// - the other v - 1 (across the rows of 16 lanes) is read back from LDS, where
//   the results go anyway: each row of lanes runs one step behind the row
//   before it, so the value was stored two steps ago; for v = 0 the same read
//   fetches the face;
// - the u face is taken off when the values are staged (its entry is the first
//   of the row; the entry is then zero);
// - what a step needs leaves LDS two steps before.
// 100^3, per launch of a sweep: 8.1 us with three loads in turn and the
// neighbours handed over in LDS, 5.9 now (an empty launch 1.7, loads and
// stores 1.5, the steps 2.1).
template <int MODE>
__global__ __launch_bounds__(kBoxThreads) void k_box_sweep(IccArgs c, const State* st,
                                                           const double* __restrict__ in,
                                                           double* __restrict__ out,
                                                           TileLevel level) {
  constexpr int TX = kBoxTX, TY = kBoxTY, TZ = kBoxTZ;
  static_assert(TX == 8 && TY == 8, "a lane per pencil, the v pencils two to 16 lanes");
  static_assert(TX * TY * TZ == kBoxThreads, "one thread per cell when staging");
  // Pencil (u, v) starts at P u + S v + v / 2: the lanes of a step, whose w
  // differ by u + v + v / 2, fall on different banks.  Reads run past a
  // pencil's ends by up to kPad, where nothing is used.
  constexpr int P = TZ + 2, S = 169, kPad = 24, kFace = TZ + 3;
  constexpr int kCells = 7 * S + 3 + 7 * P + TZ + 2 * kPad, kFaces = 7 * kFace + TZ + 2 * kPad;
  constexpr int kSink = kCells - 1;
  __shared__ dbl2 m01[kCells], m2d[kCells];  // scaled c0 and c1, c2 and d
  __shared__ double m[kCells + kFaces];      // r or y, then the result; the v face
  __shared__ double mw[64];                  // the w face
  const BoxIcc& b = c.bx;
  const int X = level.first + blockIdx.y, Y = level.lo(b, X) + blockIdx.x;
  if (Y > level.hi(b, X)) return;
  const int u0 = X * b.tx, v0 = Y * b.ty, w0 = (level.l - X - Y) * b.tz;
  const int tid = threadIdx.x;
  auto row_of = [&](int u, int v, int w) {
    const int x = MODE == 2 ? b.nx - 1 - u : u;
    const int y = MODE == 2 ? b.ny - 1 - v : v;
    const int z = MODE == 2 ? b.nz - 1 - w : w;
    return (x * b.ny + y) * b.nz + z;
  };
  auto in_tile = [&](int lu, int lv, int lw) {
    return lu < b.tx && lv < b.ty && lw < b.tz && u0 + lu < b.nx && v0 + lv < b.ny &&
           w0 + lw < b.nz;
  };
  // this thread's cell (w fastest: the loads coalesce) and its value of the
  // three finished faces next to the tile (zero outside the grid)
  const int su = tid / (TY * TZ), sv = (tid / TZ) % TY, sw = tid % TZ;
  const bool mine = in_tile(su, sv, sw);
  const int si = mine ? row_of(u0 + su, v0 + sv, w0 + sw) : 0;
  const int sq = kPad + su * P + sv * S + sv / 2 + sw;
  double c0 = 0.0, c1 = 0.0, c2 = 0.0, a0 = 0.0, d0 = 0.0, f0 = 0.0;
  if (mine) {
    const double* const* cf = MODE == 2 ? b.up : b.lo;
    c0 = cf[0][si];
    c1 = cf[1][si];
    c2 = cf[2][si];
    a0 = MODE == 0 ? b.dg[si] : in[si];
    if (MODE != 0) d0 = c.d[si];
    if (MODE == 2) f0 = c.dinv[si];
  }
  const int side = tid / (TY * TZ), fa = (tid / TZ) % TY, fb = tid % TZ;  // side 2: (u, v) in a row
  double face = 0.0;
  {
    const int lu = side == 0 ? 0 : side == 1 ? fa : (tid / TY) % TX;
    const int lv = side == 0 ? fa : side == 1 ? 0 : tid % TY;
    const int lw = side == 2 ? 0 : fb;
    const bool edge = side == 0 ? u0 > 0 : side == 1 ? v0 > 0 : side == 2 && tid < 2 * TY * TZ + 64 && w0 > 0;
    if (edge && in_tile(lu, lv, lw))
      face = out[row_of(u0 + lu - (side == 0), v0 + lv - (side == 1), w0 + lw - (side == 2))];
  }
  const double fn = st ? st->fn : 1.0;
  const int done = MODE != 0 && st ? st->done : 0;
  asm volatile("" : "+v"(c0), "+v"(c1), "+v"(c2), "+v"(a0), "+v"(d0), "+v"(f0), "+v"(face));
  if (done) return;
  c0 = c0 * fn;
  a0 = MODE == 0 ? a0 * fn : MODE == 2 ? a0 * f0 : a0;
  if (side == 0) {  // su = 0, and `face` is this cell's u - 1
    a0 = a0 - (MODE == 0 ? face * c0 * c0 : c0 * face);
    c0 = 0.0;
  }
  m01[sq] = dbl2{c0, c1 * fn};
  m2d[sq] = dbl2{c2 * fn, d0};
  m[sq] = a0;
  if (side == 1) m[kCells + kPad + fa * kFace + fb] = face;
  else if (side == 2 && tid < 2 * TY * TZ + 64) mw[tid - 2 * TY * TZ] = face;  // [u][v]
  __syncthreads();
  if (tid < 64) {
    const int pu = tid & 7, pv = ((tid >> 4) << 1) | ((tid >> 3) & 1), late = tid >> 4;
    const int steps = b.tx + b.ty + b.tz - 2 + (b.ty - 1) / 2;
    const unsigned wend = in_tile(pu, pv, 0) ? min(b.tz, b.nz - w0) : 0;
    int lw = -(pu + pv + late);
    const int at = kPad + pu * P + pv * S + pv / 2;
    const int across = pv == 0 ? kCells + kPad + pu * kFace : (pv & 1) ? at : at - S - 1;
    struct Ahead { dbl2 c01, c2d; double a, x; };
    Ahead v[3];
    double prev = mw[pu * TY + pv];
    // the compiler may not move these reads: LDS answers in order
    auto ahead = [&](int w, Ahead& g) {
      __builtin_amdgcn_sched_barrier(0);
      g.x = m[across + w];
      g.a = m[at + w];
      g.c01 = m01[at + w];
      g.c2d = m2d[at + w];
      __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](const Ahead& g, Ahead& next) {
      const double n0 = row_shift<1>(0.0, prev), n1 = row_shift<8>(g.x, prev), n2 = prev;
      double sum = g.a, r;
      if (MODE == 0) {
        sum = sum - n0 * g.c01.x * g.c01.x;
        sum = sum - n1 * g.c01.y * g.c01.y;
        sum = sum - n2 * g.c2d.x * g.c2d.x;
        r = 1.0 / sum;
      } else {
        sum = sum - g.c01.x * n0;
        sum = sum - g.c01.y * n1;
        sum = sum - g.c2d.x * n2;
        r = sum * g.c2d.y;
      }
      const bool in = (unsigned)lw < wend;
      prev = in ? r : prev;
      const int q = in ? at + lw : kSink;   // a store without a branch around it
      m[q] = r;
      if (MODE == 0) m2d[q].y = sum;
      ahead(lw + 2, next);
      ++lw;
    };
    ahead(lw, v[0]);
    ahead(lw + 1, v[1]);
    for (int t = 0; t < steps; t += 3) {  // a step more than needed does nothing
      step(v[0], v[2]);
      step(v[1], v[0]);
      step(v[2], v[1]);
    }
  }
  __syncthreads();
  if (mine) {
    out[si] = m[sq];
    if (MODE == 0) c.dinv[si] = m2d[sq].y;
  }
}

hipError_t launch_box_sweep(hipStream_t s, const IccArgs& c, int mode, const State* st,
                            const double* in, double* out) {
  // the level loop hands cells between the lanes of one wave of 64
  static const int wave = [] {
    int dev = 0, w = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&w, hipDeviceAttributeWarpSize, dev) != hipSuccess)
      return 0;
    return w;
  }();
  if (wave != 64) return hipErrorInvalidDeviceFunction;
  const int nl = c.bx.ntx + c.bx.nty + c.bx.ntz - 2;
  for (int l = 0; l < nl; ++l) {
    const TileLevel t(c.bx, l);
    const dim3 grid(t.span, t.rows);
    if (mode == 0) k_box_sweep<0><<<grid, kBoxThreads, 0, s>>>(c, st, in, out, t);
    else if (mode == 1) k_box_sweep<1><<<grid, kBoxThreads, 0, s>>>(c, st, in, out, t);
    else k_box_sweep<2><<<grid, kBoxThreads, 0, s>>>(c, st, in, out, t);
  }
  return hipGetLastError();
}

// CG with ICC, iteration k: the stopping test of iteration k-1 on the update
// partials (one workgroup), before the sweeps (Cg.f90:214-222).
__global__ __launch_bounds__(kBlock) void k_icc_check(CgArgs a, int k) {
  __shared__ double s_tmp[5 * 4], s_out[5];
  State* st = a.st;
  if (st->done) return;
  const int ops[5] = {OP_SUM, OP_MIN, OP_MAX, OP_SUM, OP_SUM};
  gather<5>(a.pt.upd, a.pt.pstride, a.pt.g_upd, ops, s_tmp, s_out);
  if (threadIdx.x != 0) return;
  double res;
  if (st->criterion == TFG_CRIT_RELRES) {
    res = sqrt(s_out[4]) / st->bnorm;
  } else {
    const double range = st->has_norm ? fmax(st->norm - 0.0, kTiny) : fmax(s_out[2] - s_out[1], kTiny);
    res = sqrt(s_out[0]) / range;
  }
  st->res = res;
  st->iter = k - 1;
  if (!isfinite(res)) {
    st->status = TFG_EBREAKDOWN;
    st->niter = k - 1;
    st->done = 1;
  } else if (res < st->tol) {
    st->niter = k - 1;
    st->done = 1;
  }
}

// partials of rho = (z, r)                                  Cg.f90:150-156
__global__ __launch_bounds__(kBlock) void k_icc_rho(CgArgs a, const double* __restrict__ z) {
  __shared__ double s_tmp[4], s_out[1];
  if (a.st->done) return;
  double v[1] = {0.0};
  const int stride = gridDim.x * kBlock;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < a.n; i += stride) v[0] = v[0] + z[i] * a.r[i];
  const int ops[1] = {OP_SUM};
  publish<1>(v, ops, a.pt.ext, a.pt.pstride, s_tmp, s_out);
}

// beta = rho_k / rho_{k-1}; p = z + beta p (p = z when k = 1)  Cg.f90:158-171
__global__ __launch_bounds__(kBlock) void k_icc_pupdate(CgArgs a, const double* __restrict__ z,
                                                        int k) {
  __shared__ double s_tmp[4], s_out[1];
  State* st = a.st;
  if (st->done) return;
  const int ops[1] = {OP_SUM};
  gather<1>(a.pt.ext, a.pt.pstride, a.pt.g_vec, ops, s_tmp, s_out);
  const double rho = s_out[0];
  const double beta = k > 1 ? rho / st->rho[(k - 1) & 1] : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) st->rho[k & 1] = rho;
  const int stride = gridDim.x * kBlock;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < a.n; i += stride)
    a.p[i] = k == 1 ? z[i] : z[i] + beta * a.p[i];
}

// z = r * (1 / a_ii) on the unscaled matrix (the building block)
__global__ __launch_bounds__(kBlock) void k_jacobi_apply(int n, const int* __restrict__ row,
                                                         const double* __restrict__ val,
                                                         const double* __restrict__ r,
                                                         double* __restrict__ z) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) z[i] = r[i] * (1.0 / val[row[i]]);
}

hipError_t launch_jacobi_apply(hipStream_t s, int n, const int* row, const double* val,
                               const double* r, double* z) {
  k_jacobi_apply<<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(n, row, val, r, z);
  return hipGetLastError();
}

hipError_t launch_icc_form(hipStream_t s, const IccArgs& c, const double* val, const State* st) {
  if (c.box) {
    const int grid = std::max(1, std::min((c.n + kBlock - 1) / kBlock, 4096));
    k_box_pack<<<grid, kBlock, 0, s>>>(c, val);
    return launch_box_sweep(s, c, 0, st, nullptr, c.d);
  }
  for (int l = 0; l < c.nlev_f; ++l) {
    const int lo = c.off_f_host[l], hi = c.off_f_host[l + 1];
    k_icc_form<<<(hi - lo + kBlock - 1) / kBlock, kBlock, 0, s>>>(c, val, st, lo, hi);
  }
  return hipGetLastError();
}

hipError_t launch_icc_apply(hipStream_t s, const IccArgs& c, const double* val, const State* st,
                            const double* r, double* z) {
  if (c.box) {  // the diagonals were packed from val by launch_icc_form
    const hipError_t e = launch_box_sweep(s, c, 1, st, r, c.y);
    if (e != hipSuccess) return e;
    return launch_box_sweep(s, c, 2, st, c.y, z);
  }
  for (int l = 0; l < c.nlev_f; ++l) {
    const int lo = c.off_f_host[l], hi = c.off_f_host[l + 1];
    k_icc_fwd<<<(hi - lo + kBlock - 1) / kBlock, kBlock, 0, s>>>(c, val, st, r, lo, hi);
  }
  for (int l = 0; l < c.nlev_b; ++l) {
    const int lo = c.off_b_host[l], hi = c.off_b_host[l + 1];
    k_icc_bwd<<<(hi - lo + kBlock - 1) / kBlock, kBlock, 0, s>>>(c, val, st, z, lo, hi);
  }
  return hipGetLastError();
}

hipError_t launch_icc_check(const Launch& L, const CgArgs& a, int k) {
  k_icc_check<<<1, kBlock, 0, L.stream>>>(a, k);
  return hipGetLastError();
}

hipError_t launch_icc_rho(const Launch& L, const CgArgs& a, const double* z) {
  k_icc_rho<<<L.grid_vec, kBlock, 0, L.stream>>>(a, z);
  return hipGetLastError();
}

hipError_t launch_icc_pupdate(const Launch& L, const CgArgs& a, const double* z, int k) {
  k_icc_pupdate<<<L.grid_vec, kBlock, 0, L.stream>>>(a, z, k);
  return hipGetLastError();
}

}  // namespace tfg
