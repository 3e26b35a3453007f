// Pressure-system assembly on the device from face data, so that a pressure
// solve needs no host-to-device copy of A % val and b.  What it computes is
// the reference's, in the reference's order:
//   A % val = 0, b = 0                          Compute_Pressure.f90:121-122
//   internal faces s (in order): a12 = fc(s) (f(s) v_m(c1) + (1 - f(s)) v_m(c2)),
//     val(pos(1,s)) = val(pos(2,s)) = -a12, val(dia(c1)) += a12,
//     val(dia(c2)) += a12                          Rhie_And_Chow.f90:184-205
//   all faces s (in order): b(c1) -= flux(s), b(c2) += flux(s) (internal);
//     boundary faces with a pressure / ambient condition:
//     val(dia(c1)) += fc(s) v_m(c1)             Compute_Pressure.f90:147-169
//   boundary regions: b(c1) = 0 in pressure regions, b(c1) = fc(s) v_m(c1)
//     pp(c2) in ambient regions, assigned region by region and face by
//     face                                        Compute_Pressure.f90:173-188
//   optionally a_ii *= (1 + MICRO)              Solver_Mod/Set_Singular.f90:28-31
// The face loop scatters into the diagonal and b, so it is turned around:
// one thread per row walks, in increasing face order, the faces of its cell
// (a list built once per structure) and forms its diagonal and b entry as
// the serial loop would; each off-diagonal entry takes -a12 of the last face
// that sets it.  The region assignments of b follow face order, which is the
// region loop's order when each region's faces are one range and the ranges
// ascend with the region number (Faces_In_Region, as T-Flows numbers its
// boundary faces).  Every value is bit-identical to the serial assembly.
#include <algorithm>

#include "tflows_gpu.h"
#include "tfg_spmv.h"

namespace tfg {

// The row block of this workgroup: kBlock consecutive cells, consecutive
// blocks on one XCD (workgroup g runs on XCD g % 8), so that the faces and
// neighbours two blocks share are in one L2.  -1: no block.
__device__ __forceinline__ int cell_block(int nblk) {
  const int x = (int)blockIdx.x % kXcds, l = (int)blockIdx.x / kXcds;
  const int first = (int)(((long long)nblk * x) / kXcds);
  const int end = (int)(((long long)nblk * (x + 1)) / kXcds);
  return first + l < end ? first + l : -1;
}
int cell_grid(int n) {
  const int nblk = (n + kBlock - 1) / kBlock;
  return kXcds * ((nblk + kXcds - 1) / kXcds);
}

// The matrix rows of a workgroup's cells, staged in LDS and written with
// whole cache lines (a thread's own row is 7 scattered 8-byte stores on a
// hex grid); rows of more than kStage entries in all are written directly.
struct RowStage {
  static constexpr int kStage = 8 * kBlock;
  double* lds;
  double* val;
  int base, count;
  bool staged;
  __device__ __forceinline__ RowStage(const CellFaces& t, double* s_val, double* v, int c0, int c1,
                                      int c, bool live)
      : lds(s_val), val(v) {
    base = t.row[c0];
    count = t.row[c1] - base;
    staged = count <= kStage;
    if (t.unset) {   // entries that no face sets are zero
      if (staged) {
        for (int j = threadIdx.x; j < count; j += kBlock) lds[j] = 0.0;
        __syncthreads();
      } else if (live) {
        for (int j = t.row[c]; j < t.row[c + 1]; ++j) val[j] = 0.0;
      }
    }
  }
  __device__ __forceinline__ void put(int j, double v) const {
    if (staged) lds[j - base] = v;
    else val[j] = v;
  }
  // every thread of the workgroup calls it
  __device__ __forceinline__ void flush() const {
    if (!staged) return;
    __syncthreads();
    for (int j = threadIdx.x; j < count; j += kBlock) val[base + j] = lds[j];
  }
};

// One pass over a cell's faces forms its diagonal, b entry and off-diagonal
// entries; a boundary face's diagonal term waits for the internal ones (the
// second loop of Compute_Pressure).  Bound by the memory behind the L2 and the
// latency of the list -> face data chain, so each face is read once per cell
// and three faces' loads are in flight together: 128^3 in grid order 333 us
// with a pass for the diagonal, one for b and one over the entries (each
// fetching the face data again, one load at a time), 111 us now.
constexpr int kFaces = 3;

template <class S>
__global__ __launch_bounds__(kBlock) void k_assemble(AsmArgs g) {
  __shared__ double s_val[RowStage::kStage];
  const CellFaces& t = g.t;
  const int blk = cell_block((t.n + kBlock - 1) / kBlock);
  if (blk < 0) return;
  const int c0 = blk * kBlock, c1 = min(t.n, c0 + kBlock), c = c0 + (int)threadIdx.x;
  const bool live = c < c1;
  const RowStage row(t, s_val, g.val, c0, c1, c, live);
  if (live) {
    const S* slot = static_cast<const S*>(t.slot);
    const int fs0 = t.off[c], fs1 = t.off[c + 1], rs = t.row[c];
    const double vm = g.vm[c];
    double diag = 0.0, bc = 0.0, bset = 0.0;
    bool set = false, bnd = false;
    // kFaces faces at a time, their loads in flight together (the last face
    // repeated past the end)
    for (int f0 = fs0; f0 < fs1; f0 += kFaces) {
      int e[kFaces], nb[kFaces], sl[kFaces];
      double flux[kFaces], fs[kFaces], fc[kFaces], vn[kFaces];
#pragma unroll
      for (int k = 0; k < kFaces; ++k) {
        const int f = min(f0 + k, fs1 - 1);
        e[k] = t.face[f];
        nb[k] = t.nbr[f];
        sl[k] = slot[f];
      }
#pragma unroll
      for (int k = 0; k < kFaces; ++k) {
        const int s = e[k] >> 1;
        flux[k] = g.vflux[s];
        fs[k] = g.fw[s];
        fc[k] = g.fc[s];
        vn[k] = g.vm[nb[k] > 0 ? nb[k] - 1 : c];
      }
#pragma unroll
      for (int k = 0; k < kFaces; ++k) {
        if (f0 + k >= fs1) continue;
        const bool second = e[k] & 1;
        if (nb[k] > 0) {
          const double v1 = second ? vn[k] : vm, v2 = second ? vm : vn[k];
          const double a12 = fc[k] * (fs[k] * v1 + (1.0 - fs[k]) * v2);  // Rhie_And_Chow.f90:200
          diag = diag + a12;
          bc = second ? bc + flux[k] : bc - flux[k];
          row.put(rs + sl[k], -a12);
        } else {
          bc = bc - flux[k];
          bnd = true;
        }
      }
    }
    if (bnd) {
      for (int f = fs0; f < fs1; ++f) {
        const int nb = t.nbr[f];
        if (nb > 0) continue;
        const int s = t.face[f] >> 1, fl = g.flags[s];
        if (fl & 1) diag = diag + g.fc[s] * vm;
        if (fl & 2) {
          bset = 0.0;
          set = true;
        } else if (fl & 4) {
          const double a12 = g.fc[s] * vm;
          bset = a12 * g.pp[nb - 1];
          set = true;
        }
      }
    }
    if (g.singular) diag = diag * (1.0 + 1.0e-6);
    row.put(rs, diag);
    g.b[c] = set ? bset : bc;
  }
  row.flush();
}

hipError_t launch_assemble(hipStream_t stream, const AsmArgs& g) {
  if (g.t.wide) k_assemble<int><<<cell_grid(g.t.n), kBlock, 0, stream>>>(g);
  else k_assemble<uint8_t><<<cell_grid(g.t.n), kBlock, 0, stream>>>(g);
  return hipGetLastError();
}

// vel_max = max(MICRO, max_c sqrt(u_c^2 + v_c^2 + w_c^2))  Compute_Momentum.f90:201-204
// (a maximum: the same bits in any order).  One workgroup per chunk of
// cells, the chunk maxima combined by the second kernel.
__global__ __launch_bounds__(kBlock) void k_vel_max(int n, const double* __restrict__ u,
                                                    const double* __restrict__ v,
                                                    const double* __restrict__ w,
                                                    double* __restrict__ part) {
  __shared__ double s_tmp[4], s_out[1];
  double m[1] = {1.0e-6};
  const int stride = gridDim.x * kBlock;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += stride)
    m[0] = fmax(m[0], sqrt(u[i] * u[i] + v[i] * v[i] + w[i] * w[i]));
  const int ops[1] = {OP_MAX};
  publish<1>(m, ops, part, 1, s_tmp, s_out);
}

__global__ __launch_bounds__(kBlock) void k_vel_max_final(const double* __restrict__ part,
                                                          int G, double* out) {
  __shared__ double s_tmp[4], s_out[1];
  const int ops[1] = {OP_MAX};
  gather<1>(part, 1, G, ops, s_tmp, s_out);
  if (threadIdx.x == 0) out[0] = s_out[0];
}

// p_min, p_max over the cells (Compute_Pressure.f90:104-109; HUGE
// starts, which a finite field always replaces)
__global__ __launch_bounds__(kBlock) void k_range(int n, const double* __restrict__ v,
                                                 double* __restrict__ part) {
  __shared__ double s_tmp[2 * 4], s_out[2];
  double m[2] = {kHuge, -kHuge};
  const int stride = gridDim.x * kBlock;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
    m[0] = fmin(m[0], v[i]);
    m[1] = fmax(m[1], v[i]);
  }
  const int ops[2] = {OP_MIN, OP_MAX};
  publish<2>(m, ops, part, 1024, s_tmp, s_out);
}

__global__ __launch_bounds__(kBlock) void k_range_final(const double* __restrict__ part, int G,
                                                       double* out) {
  __shared__ double s_tmp[2 * 4], s_out[2];
  const int ops[2] = {OP_MIN, OP_MAX};
  gather<2>(part, 1024, G, ops, s_tmp, s_out);
  if (threadIdx.x < 2) out[threadIdx.x] = s_out[threadIdx.x];
}

hipError_t launch_range(hipStream_t stream, int n, const double* v, double* part, int G,
                        double* out) {
  if (G > 1024) return hipErrorInvalidValue;
  k_range<<<G, kBlock, 0, stream>>>(n, v, part);
  k_range_final<<<1, kBlock, 0, stream>>>(part, G, out);
  return hipGetLastError();
}

hipError_t launch_vel_max(hipStream_t stream, int n, const double* u, const double* v,
                          const double* w, double* part, int G, double* out) {
  k_vel_max<<<G, kBlock, 0, stream>>>(n, u, v, w, part);
  k_vel_max_final<<<1, kBlock, 0, stream>>>(part, G, out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Momentum assembly of one velocity component (Compute_Momentum.f90:119-366
// with Numerics_Mod).  As for the pressure, every face loop of the reference
// is turned around: one thread per cell walks its faces and sums its own
// entries in the reference's order.  That order is increasing face index in
// every loop except the advection loops, which take the boundary faces first
// and then the domain faces (Advection_Term.f90:35-102: boundary regions,
// then Faces_In_Domain_And_At_Buffers).  The two coincide for T-Flows' face
// numbering (boundary regions first); a cell where they do not (CellFaces::
// late) sums its boundary faces' advection in a pass of its own first.
// A face's value is computed by both of its cells with the same arithmetic,
// so both see the same bits.
// ---------------------------------------------------------------------------

namespace {

__device__ __forceinline__ double cell(const double* a, int c) { return a[c - 1]; }
__device__ __forceinline__ double dmin(double a, double b) { return b < a ? b : a; }
__device__ __forceinline__ double dmax(double a, double b) { return b > a ? b : a; }

// Advection schemes that bound the face value by the range of phi around the
// upwind cell (k_mom_minmax).
constexpr bool needs_range(int adv) {
  return adv != TFG_ADV_CENTRAL && adv != TFG_ADV_UPWIND && adv != TFG_ADV_BLENDED &&
         adv != TFG_ADV_GAMMA;
}

// What a face's value needs of one of its cells; of the face.
struct MomCell {
  double phi, g[3], mn, mx;
};
struct MomFace {
  double F, f, d[3];
};

// Face value (Numerics_Mod/Advection_Scheme.f90:22-183) from the face's two
// cells P1 (c1) and P2 (c2).
template <int ADV>
__device__ __forceinline__ double face_value(const MomArgs& m, const MomFace& q, const MomCell& P1,
                                             const MomCell& P2) {
  const double fs = q.f;
  if (ADV == TFG_ADV_CENTRAL) return fs * P1.phi + (1.0 - fs) * P2.phi;
  const bool pos = q.F > 0.0;
  const double fj = pos ? 1.0 - fs : fs, sgn = pos ? +1.0 : -1.0;
  const double phi_c = pos ? P1.phi : P2.phi, phi_d = pos ? P2.phi : P1.phi;
  if (ADV == TFG_ADV_UPWIND) return phi_c;
  if (ADV == TFG_ADV_BLENDED) {
    const double phi_f_c = phi_c + fj * sgn * (P2.phi - P1.phi);
    const double phi_f_u = phi_c;
    return m.blend * phi_f_c + (1.0 - m.blend) * phi_f_u;
  }
  const double gd = (pos ? P1.g[0] : P2.g[0]) * q.d[0] + (pos ? P1.g[1] : P2.g[1]) * q.d[1] +
                    (pos ? P1.g[2] : P2.g[2]) * q.d[2];
  if (ADV == TFG_ADV_GAMMA) {
    const double beta = 0.1;
    const double phi_star = pos ? 1.0 - (phi_d - phi_c) / (2.0 * gd)
                                : 1.0 + (phi_d - phi_c) / (2.0 * gd);
    const double gamma_c = phi_star / beta;
    if (phi_star < beta && phi_star > 0.0)
      return (1.0 - gamma_c * (1.0 - fs)) * phi_c + gamma_c * (1.0 - fs) * phi_d;
    if (phi_star < 1.0 && phi_star >= beta) return fs * phi_c + (1.0 - fs) * phi_d;
    return phi_c;
  }
  const double phi_star = pos ? phi_d - 2.0 * gd : phi_d + 2.0 * gd;
  const double mn = pos ? P1.mn : P2.mn, mx = pos ? P1.mx : P2.mx;
  const double phi_u = dmax(mn, dmin(phi_star, mx));
  double denom = phi_d - phi_c;
  if (fabs(denom) < 1.0e-15) denom = denom + copysign(1.0e-15, denom);
  const double rj = (phi_c - phi_u) / denom;
  const double g_d = 0.5 * fj * (1.0 + fj), g_u = 0.5 * fj * (1.0 - fj);
  double phij = fj;
  if (ADV == TFG_ADV_QUICK) {
    const double alfa = 0.0;
    phij = (g_d - alfa) + (g_u + alfa) * rj;
  } else if (ADV == TFG_ADV_LUDS) {
    const double alfa = 0.5 * fj * (1 + fj);
    phij = (g_d - alfa) + (g_u + alfa) * rj;
  } else if (ADV == TFG_ADV_MINMOD) {
    phij = fj * dmax(0.0, dmin(rj, 1.0));
  } else if (ADV == TFG_ADV_SMART) {
    const double beta1 = 3.0, beta2 = 1.0;
    phij = dmax(0.0, dmin(dmin((beta1 - 1.0) * rj, g_d + g_u * rj), beta2));
  } else if (ADV == TFG_ADV_AVL_SMART) {
    const double beta1 = 1.0 + fj * (2.0 + fj), beta2 = fj * (2.0 - fj);
    phij = dmax(0.0, dmin(dmin((beta1 - 1.0) * rj, g_d + g_u * rj), beta2));
  } else if (ADV == TFG_ADV_SUPERBEE) {
    phij = 0.5 * dmax(dmax(0.0, dmin(2.0 * rj, 1.0)), dmin(rj, 2.0));
  }
  return phi_c + phij * sgn * (P2.phi - P1.phi);
}

// Cell C (0-based own: the cell whose face leads there, whose range stands in
// for a boundary cell's until the caller knows phi: Min_Max.f90:19-34 gives a
// boundary cell the range of itself and its one neighbour).
template <int ADV>
__device__ __forceinline__ MomCell mom_cell(const MomArgs& m, int C, int own) {
  MomCell q{cell(m.phi, C), {cell(m.g[0], C), cell(m.g[1], C), cell(m.g[2], C)}, 0.0, 0.0};
  if (needs_range(ADV)) {
    const dbl2 r = m.mm[C > 0 ? C - 1 : own];
    q.mn = r.x;
    q.mx = r.y;
  }
  return q;
}
template <int ADV>
__device__ __forceinline__ void boundary_range(int C, double phi_own, MomCell& q) {
  if (needs_range(ADV)) {
    q.mn = C > 0 ? q.mn : dmin(q.phi, phi_own);
    q.mx = C > 0 ? q.mx : dmax(q.phi, phi_own);
  }
}

}  // namespace

__global__ __launch_bounds__(kBlock) void k_mom_minmax(MomArgs m) {
  const CellFaces& t = m.t;
  const int blk = cell_block((t.n + kBlock - 1) / kBlock);
  if (blk < 0) return;
  const int c = blk * kBlock + (int)threadIdx.x;
  if (c >= t.n) return;
  double mn = cell(m.phi, c + 1), mx = mn;
  const int f1 = t.off[c + 1];
  for (int f = t.off[c]; f < f1; ++f) {
    const double o = cell(m.phi, t.nbr[f]);
    mn = dmin(mn, o);
    mx = dmax(mx, o);
  }
  m.mm[c] = dbl2{mn, mx};
}

// One pass over the cell's faces: advection, diffusion, the diagonal and the
// off-diagonal entries.  Bound by the latency of the list -> face and
// neighbour loads at the four waves per SIMD that ~110 registers leave, and
// by the memory behind the L2 (0.87 GB fetched at 110x100x90, MINMOD).  So the
// loop body has no load under a condition (all of a face's loads and the next
// face's indices are issued before any is waited for), the scheme is a
// template argument, and the cell's own values stay in registers: 454 us with
// four passes over the faces and both cells gathered in each, 254 us in one
// pass with the loads where they are used, 194 us now.
template <int ADV, class S>
__global__ __launch_bounds__(kBlock) void k_momentum(MomArgs m) {
  __shared__ double s_val[RowStage::kStage];
  const CellFaces& t = m.t;
  const int blk = cell_block((t.n + kBlock - 1) / kBlock);
  if (blk < 0) return;
  const int c0 = blk * kBlock, c1 = min(t.n, c0 + kBlock), c = c0 + (int)threadIdx.x;
  const bool live = c < c1;
  const RowStage row(t, s_val, m.val, c0, c1, c, live);
  if (live) {
    const S* slot = static_cast<const S*>(t.slot);
    const int C = c + 1, t0 = t.off[c], t1 = t.off[c + 1], rs = t.row[c];
    const double rho_c = cell(m.rho, C);
    const MomCell P = mom_cell<ADV>(m, C, c);
    // advection, b = fi (Advection_Term.f90:35-120)
    double adv = 0.0, upw = 0.0;
    auto advect = [&](bool second, const MomFace& q, const MomCell& N, bool skip) {
      const MomCell P1 = second ? N : P, P2 = second ? P : N;
      const double phif = face_value<ADV>(m, q, P1, P2);
      const double a = q.F * phif * rho_c;
      adv = skip ? adv : (second ? adv + a : adv - a);
      if (m.blend_matrix) {
        const double u = q.F * (q.F < 0 ? P2.phi : P1.phi) * rho_c;
        upw = skip ? upw : (second ? upw + u : upw - u);
      }
    };
    const bool late = t.late[c];
    if (late) {
      for (int f = t0; f < t1; ++f) {
        const int nb = t.nbr[f];
        if (nb >= 0) continue;
        const int s = t.face[f] >> 1;
        const MomFace q{m.v_flux[s], m.f[s], {m.dv[0][s], m.dv[1][s], m.dv[2][s]}};
        MomCell N = mom_cell<ADV>(m, nb, c);
        boundary_range<ADV>(nb, P.phi, N);
        advect(false, q, N, false);
      }
    }
    // diffusion (Compute_Momentum.f90:238-301)
    const int ki = (m.comp - 1) % 3, kj = m.comp % 3, kk = (m.comp + 1) % 3;
    auto part = [](const double (&v)[3], int k) { return k == 0 ? v[0] : (k == 1 ? v[1] : v[2]); };
    const double *si = m.sv[ki], *sj = m.sv[kj], *sk = m.sv[kk];
    const double* stress = m.f_stress ? m.f_stress : m.vis_eff;
    const double uj_c = cell(m.uj_i, C), uk_c = cell(m.uk_i, C);
    double cross = 0.0, diag = 0.0;
    bool wall = false;
    int e = t0 < t1 ? t.face[t0] : 0, nb = t0 < t1 ? t.nbr[t0] : 0;
    for (int f = t0; f < t1; ++f) {
      // every load of this face and the next one's indices before any use
      const int s = e >> 1, fn = min(f + 1, t1 - 1);
      const bool second = e & 1;
      const MomFace q{m.v_flux[s], m.f[s], {m.dv[0][s], m.dv[1][s], m.dv[2][s]}};
      const double w = m.fw[s], vis_eff = m.vis_eff[s], fc = m.fc[s], st = stress[s];
      const double siv = si[s], sjv = sj[s], skv = sk[s];
      MomCell N = mom_cell<ADV>(m, nb, c);
      const double ujn = cell(m.uj_i, nb), ukn = cell(m.uk_i, nb);
      const int place = slot[f], e_next = t.face[fn], nb_next = t.nbr[fn], at_wall = m.wall[s];
      boundary_range<ADV>(nb, P.phi, N);
      advect(second, q, N, late && nb < 0);
      const double f_stress = m.f_stress ? st : 0.0;
      auto at_face = [&](double own, double other) {
        return w * (second ? other : own) + (1.0 - w) * (second ? own : other);
      };
      const double ui_i_f = at_face(part(P.g, ki), part(N.g, ki));
      const double ui_j_f = at_face(part(P.g, kj), part(N.g, kj));
      const double ui_k_f = at_face(part(P.g, kk), part(N.g, kk));
      const double uj_i_f = at_face(uj_c, ujn);
      const double uk_i_f = at_face(uk_c, ukn);
      const double ui_si = (ui_i_f + ui_i_f) * siv + (ui_j_f + uj_i_f) * sjv + (ui_k_f + uk_i_f) * skv;
      const double ui_di = ui_i_f * part(q.d, ki) + ui_j_f * part(q.d, kj) + ui_k_f * part(q.d, kk);
      const double f_ex = vis_eff * ui_si;
      const double m0 = vis_eff * fc;
      const double f_im = ui_di * m0;
      cross = second ? cross - f_ex + f_im - f_stress * rho_c : cross + f_ex - f_im + f_stress * rho_c;
      // the cell's side of the face: m12 for c1, m21 for c2 (:271-282)
      double mc = m0;
      if (m.blend_matrix)
        mc = second ? mc + dmax(q.F, 0.0) * rho_c : mc - dmin(q.F, 0.0) * rho_c;
      if (nb > 0) {
        diag = diag + mc;
        row.put(rs + place, 0.0 - mc);
      } else if (at_wall) {
        diag = diag + mc;
        wall = true;
      }
      e = e_next;
      nb = nb_next;
    }
    double fi = 0.0;
    fi = fi + adv - upw;
    if (wall) {
      for (int f = t0; f < t1; ++f) {
        const int nb = t.nbr[f], s = t.face[f] >> 1;
        if (nb > 0 || !m.wall[s]) continue;
        double m12 = m.vis_eff[s] * m.fc[s];
        if (m.blend_matrix) m12 = m12 - dmin(m.v_flux[s], 0.0) * rho_c;
        fi = fi + m12 * cell(m.phi, nb);
      }
    }
    fi = fi + cross;                                        // :306-308
    const double vol = cell(m.vol, C);
    const double a0 = rho_c * vol / m.dt;                   // Inertial_Term.f90:27-41
    if (m.td == TFG_TD_LINEAR) {
      diag = diag + a0;
      fi = fi + a0 * cell(m.phi_o, C);
    } else if (m.td == TFG_TD_PARABOLIC) {
      diag = diag + 1.5 * a0;
      fi = fi + 2.0 * a0 * cell(m.phi_o, C) - 0.5 * a0 * cell(m.phi_oo, C);
    }
    fi = fi + m.p_drop * vol;                               // :322-326
    const double cf = m.cell_f ? cell(m.cell_f, C) : 0.0;
    fi = fi + cf * vol;                                     // :328-331
    double bb = fi - cell(m.p_i, C) * vol;                  // :337-340
    if (m.st) bb = bb + cell(m.st, C) * vol;                // :345-350
    m.v_m[c] = vol / diag;                                  // :361-363
    diag = diag / m.urf;                                    // Under_Relax.f90:18-24
    bb = bb + diag * (1.0 - m.urf) * P.phi;
    row.put(rs, diag);
    m.b[c] = bb;
  }
  row.flush();
}

// ---------------------------------------------------------------------------
// Rhie-Chow volume fluxes (Rhie_And_Chow.f90:86-259).  The cell quantities
// (the corrected velocities u_c, the pressure terms pst) are formed for each
// of a face's two cells with the serial loop's operations, so both faces of a
// cell see the same bits.
// ---------------------------------------------------------------------------
namespace {

struct RcCell {
  double p, vm, u, v, w, px, py, pz, tm, curv, col;
};

template <bool VOF, bool CHOI, bool GU>
__device__ __forceinline__ RcCell rc_cell(const tfg_rhie_chow& r, int c) {
  RcCell o;
  o.p = r.p[c];
  o.vm = r.v_m[c];
  o.px = r.px[c];
  o.py = r.py[c];
  o.pz = r.pz[c];
  o.curv = VOF ? r.curv[c] : 0.0;
  o.col = VOF ? r.col[c] : 0.0;
  if (VOF) {                                              // :107-112
    o.px = o.px - r.sigma * o.curv * r.col_x[c];
    o.py = o.py - r.sigma * o.curv * r.col_y[c];
    o.pz = o.pz - r.sigma * o.curv * r.col_z[c];
  }
  o.u = r.u[c];                                           // :130-134
  o.v = r.v[c];
  o.w = r.w[c];
  o.tm = 0.0;
  if (CHOI) {                                             // :139-163
    o.tm = o.vm * r.density[c] / r.dt;
    o.u = o.u - (r.w_o * r.u_o[c] + r.w_oo * r.u_oo[c]) * o.tm;
    o.v = o.v - (r.w_o * r.v_o[c] + r.w_oo * r.v_oo[c]) * o.tm;
    o.w = o.w - (r.w_o * r.w_o_[c] + r.w_oo * r.w_oo_[c]) * o.tm;
  }
  if (GU) {                                               // :169-179
    o.u = o.u - o.vm * r.cell_fx[c];
    o.v = o.v - o.vm * r.cell_fy[c];
    o.w = o.w - o.vm * r.cell_fz[c];
  }
  return o;
}

}  // namespace

// One thread per cell takes the domain faces it is c1 of (a list of their own:
// with a cell's whole list walked for them, half the indices were read for
// nothing and each face waited for its own), so a cell's 8 to 18 values are read
// once for its faces, and its neighbours' from the lines that nearby threads read
// as their own; in face order the three directions of a grid's faces swept all
// cell arrays once each.  Bound by the memory behind the L2.  The corrections are
// template arguments, so that their loads are issued with the others.  us a call
// in face order, by the cells' whole lists, by this list: 120^3 with Choi's and
// Gu's corrections 312, 262, 221; without 134, 155, 131; 80^3 without 53, 52, 40.
// On small grids a thread's three faces in turn are all the time there is, so
// there they are dealt to up to three threads (SPLIT: gridDim.y) while the chip
// has room for them: 12^3 15.5, 18.5, 15.3; from 64^3 on that only costs.
template <bool VOF, bool CHOI, bool GU, bool SPLIT>
__global__ __launch_bounds__(kBlock) void k_rhie_chow(RcArgs a) {
  const int blk = cell_block((a.n + kBlock - 1) / kBlock);
  if (blk < 0) return;
  const int c1 = blk * kBlock + (int)threadIdx.x;
  if (c1 >= a.n) return;
  const tfg_rhie_chow& r = a.r;
  const RcCell A = rc_cell<VOF, CHOI, GU>(r, c1);
  // kIndex faces' indices together, then each face
  constexpr int kIndex = SPLIT ? 1 : 3;
  const int f1 = a.off[c1 + 1];
  const int first = SPLIT ? (int)blockIdx.y : 0, step = SPLIT ? (int)gridDim.y : kIndex;
  for (int f0 = a.off[c1] + first; f0 < f1; f0 += step) {
    int face[kIndex], nbr[kIndex];
#pragma unroll
    for (int k = 0; k < kIndex; ++k) {
      const int f = min(f0 + k, f1 - 1);
      face[k] = a.face[f];
      nbr[k] = a.nbr[f];
    }
#pragma unroll
    for (int k = 0; k < kIndex; ++k) {
      if (f0 + k >= f1) continue;
      const int s = face[k], c2 = nbr[k];
      const RcCell B = rc_cell<VOF, CHOI, GU>(r, c2);
      const double fs = r.f[s], fc = r.fc[s], sx = r.sx[s], sy = r.sy[s], sz = r.sz[s];
      const double dx = r.dx[s], dy = r.dy[s], dz = r.dz[s];
      const double fo = CHOI ? r.flux_o[s] : 0.0, foo = CHOI ? r.flux_oo[s] : 0.0;
      const double fx = GU ? r.face_fx[s] : 0.0, fy = GU ? r.face_fy[s] : 0.0;
      const double fz = GU ? r.face_fz[s] : 0.0;
      double pst_d = A.p - B.p;                               // :94-98
      if (VOF) {                                              // :115-123
        const double curv_f = fs * A.curv + (1.0 - fs) * B.curv;
        pst_d = pst_d - r.sigma * curv_f * (A.col - B.col);
      }
      const double u_f = fs * A.u + (1.0 - fs) * B.u;
      const double v_f = fs * A.v + (1.0 - fs) * B.v;
      const double w_f = fs * A.w + (1.0 - fs) * B.w;
      const double a12 = fc * (fs * A.vm + (1.0 - fs) * B.vm);
      const double px_f = (fs * (A.px * A.vm) + (1.0 - fs) * (B.px * B.vm)) * dx;
      const double py_f = (fs * (A.py * A.vm) + (1.0 - fs) * (B.py * B.vm)) * dy;
      const double pz_f = (fs * (A.pz * A.vm) + (1.0 - fs) * (B.pz * B.vm)) * dz;
      double fl = (u_f * sx + v_f * sy + w_f * sz) + a12 * pst_d +
                  fc * (px_f + py_f + pz_f);                  // :226-230
      if (CHOI)                                               // :235-246
        fl = fl + (fs * A.tm + (1.0 - fs) * B.tm) * (r.w_o * fo + r.w_oo * foo);
      if (GU)                                                 // :250-256
        fl = fl + (fs * A.vm + (1.0 - fs) * B.vm) * (fx * sx + fy * sy + fz * sz);
      a.v_flux[s] = fl;
    }
  }
}

template <bool VOF, bool CHOI, bool GU>
void run_rhie_chow(hipStream_t stream, const RcArgs& a) {
  // two workgroups for each of the 256 CUs, and three faces for a hexahedron
  const int nblk = std::max(1, (a.n + kBlock - 1) / kBlock);
  const int split = std::min(3, 512 / nblk), grid = cell_grid(a.n);
  if (split > 1) k_rhie_chow<VOF, CHOI, GU, true><<<dim3(grid, split), kBlock, 0, stream>>>(a);
  else k_rhie_chow<VOF, CHOI, GU, false><<<grid, kBlock, 0, stream>>>(a);
}

hipError_t launch_rhie_chow(hipStream_t stream, const RcArgs& a) {
  const int terms = (a.vof ? 4 : 0) | (a.r.choi ? 2 : 0) | (a.r.gu ? 1 : 0);
  switch (terms) {
    case 0: run_rhie_chow<false, false, false>(stream, a); break;
    case 1: run_rhie_chow<false, false, true>(stream, a); break;
    case 2: run_rhie_chow<false, true, false>(stream, a); break;
    case 3: run_rhie_chow<false, true, true>(stream, a); break;
    case 4: run_rhie_chow<true, false, false>(stream, a); break;
    case 5: run_rhie_chow<true, false, true>(stream, a); break;
    case 6: run_rhie_chow<true, true, false>(stream, a); break;
    default: run_rhie_chow<true, true, true>(stream, a); break;
  }
  return hipGetLastError();
}

template <int ADV>
hipError_t run_momentum(hipStream_t stream, const MomArgs& m) {
  const int grid = cell_grid(m.t.n);
  if (needs_range(ADV)) {
    k_mom_minmax<<<grid, kBlock, 0, stream>>>(m);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (m.t.wide) k_momentum<ADV, int><<<grid, kBlock, 0, stream>>>(m);
  else k_momentum<ADV, uint8_t><<<grid, kBlock, 0, stream>>>(m);
  return hipGetLastError();
}

hipError_t launch_momentum(hipStream_t stream, const MomArgs& m) {
  switch (m.adv) {
    case TFG_ADV_CENTRAL: return run_momentum<TFG_ADV_CENTRAL>(stream, m);
    case TFG_ADV_UPWIND: return run_momentum<TFG_ADV_UPWIND>(stream, m);
    case TFG_ADV_LUDS: return run_momentum<TFG_ADV_LUDS>(stream, m);
    case TFG_ADV_QUICK: return run_momentum<TFG_ADV_QUICK>(stream, m);
    case TFG_ADV_SMART: return run_momentum<TFG_ADV_SMART>(stream, m);
    case TFG_ADV_GAMMA: return run_momentum<TFG_ADV_GAMMA>(stream, m);
    case TFG_ADV_MINMOD: return run_momentum<TFG_ADV_MINMOD>(stream, m);
    case TFG_ADV_BLENDED: return run_momentum<TFG_ADV_BLENDED>(stream, m);
    case TFG_ADV_SUPERBEE: return run_momentum<TFG_ADV_SUPERBEE>(stream, m);
    case TFG_ADV_AVL_SMART: return run_momentum<TFG_ADV_AVL_SMART>(stream, m);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace tfg
