// The viscous kernels: nodal systems, scatter terms and their gather.
//
// At a vertex, sub-element p (cell p, volume vol_p) has sub-faces l with
// outward area vectors A_l.  The reference forms dense matrices N, S, S~^T for
// the face values v = N^-1 (S V + B) and reads its scatter terms from their
// products (ns_vectorial_diffusion_module.F90:200-320, ns_diffusion_module.F90:
// 112-184).  Every one of those terms is a function of the sub-element's
// H = sum_l w_l A_l^T over w_l = v_l - V_p:
//   flux through a sub-face     sigma(H) A_l,
//     sigma(H) = (mu H + (mu - mu0) H^T + (mu0 - 2/3 mu) tr(H) I) / vol_p,
//   momentum rhs                sigma(H) A_p,   A_p = sum_l A_l,
//   viscous stress              S = mu (H + H^T - 2/3 tr(H) I) / vol_p,
//   viscous work                sum_l (S v_l).A_l = S : (H + V_p A_p^T),
//   diagonal block              the same with V_p = e_j and all other cells 0,
// and likewise for the heat system with h = sum_l (T_l - T_p) A_l.  So the only
// thing worth keeping per vertex is N^-1; S, S~^T and the diagonal blocks come
// from the area vectors, which the vertex reads anyway.
//
// Two properties make N^-1 small:
// - a default-wall face that is the only one of its sub-element has no unknown
//   of its own: its row is N_bb w_b = -sum N_bi w_i with N_bb = a^2/vol (I +
//   nn^T/3), whose inverse is vol/a^2 (I - nn^T/4).  Such faces are derived, the
//   others stored.  On a one-layer prism mesh that halves the unknowns.
// - with a constant viscosity and no tagged boundary face N is symmetric (and
//   positive definite: it is the sum of the sub-elements' energy forms; wall
//   rows are scaled by mu), so its 3x3 blocks on and below the diagonal are
//   stored: 189 + 21 doubles for an interior prism vertex (6 stored faces)
//   where the products took 1,128.  Other vertices store all blocks.
// With a viscosity per cell the inverse is formed by the wavefront that applies
// it, in LDS, and never stored, except in the large class: 0.92 ms per residual
// on tri 255^2 (130k prisms) where one LDS-resident LU and unblocked inverse per
// wavefront took 42.7 ms.  The constant-viscosity set-up of tri 1024^2 went from
// 680 to 14 ms, tets 15^3 from 20.8 to 1.9 ms (k_visc_tile).
#include "kernels_diff.hpp"

namespace sfv {

namespace {

// fpos: bits 0-5 place (stored faces first, then derived), bit 6 boundary
// face, bit 7 tagged boundary face.  scode: per face a byte with bits 0-5 its
// place, bit 6 the slot is on its right side, bit 7 derived; stored faces
// first, 0xFF ends the list.
constexpr int kPosMask = 63, kPosBound = 64, kPosTag = 128;
constexpr int kCodeRight = 64, kCodeDerived = 128;
// type of a stored face: low two bits 0 interior, 1 neumann, 2 dirichlet for
// the momentum system, bits 2-3 the same for the heat system, then the BC index
constexpr int kTyV = 3, kTyTShift = 2, kTyBc = 4;

SFV_DEV void wsync_d() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

SFV_DEV int tri(int k) { return k * (k + 1) / 2; }

// One thread per vertex: which faces are derived, every face's place and
// every slot's code; once per mesh.  vstat: stored faces, << 8 tagged, << 9 skewed.
//
// Skewed: a stored face is not perpendicular to its sub-element's derived one.
// With a viscosity per cell the reduced rows are positive definite only where it
// is (t = tr(H) over the stored faces, H_2 the part of H across the derived face's
// normal, r the row of H along it): the sub-element's form is then
//   mu0 (|H|^2 + tr(H)^2 / 3) + (mu - mu0) (2 |sym H_2|^2 - t^2 / 2 + |r|^2) > 0.
// Elsewhere a pivot can vanish in a well-conditioned system (a skewed fan of three
// prisms with viscosities 8 : 1), so such vertices are pivoted then.  On extruded
// meshes the faces are perpendicular to rounding.
__global__ __launch_bounds__(256) void k_diff_tables(DevMesh m, int *vstat, uint8_t *fpos, uint32_t *scode,
                                                     double *sivol) {
  const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= m.V) return;
  const int sf0 = m.sf_off[v], nf = m.sf_off[v + 1] - sf0;
  const int se0 = m.se_off[v], se1 = m.se_off[v + 1];
  uint64_t der = 0;
  int skew = 0;
  for (int q = se0; q < se1; q++) {
    const int se = m.v_seid[q];
    sivol[q] = 1.0 / m.se_vol[se];
    int walls = 0, l = 0;
    for (int p = m.se_sfoff[se]; p < m.se_sfoff[se + 1]; p++)
      if (m.sf_re[m.se_sf[p]] == -1) {
        walls++;
        l = m.se_sf[p] - sf0;
      }
    if (walls == 1) {
      der |= 1ull << l;
      for (int p = m.se_sfoff[se]; p < m.se_sfoff[se + 1]; p++) {
        double d = 0.0;
        for (int k = 0; k < 3; k++) d += m.sfn[k * m.SF + m.se_sf[p]] * m.sfn[k * m.SF + sf0 + l];
        if (m.se_sf[p] != sf0 + l && !(fabs(d) <= 1e-8)) skew = 1;
      }
    }
  }
  const int nd = __popcll(der), ni = nf - nd;
  int tag = 0;
  for (int l = 0; l < nf; l++) {
    const uint64_t below = (1ull << l) - 1;
    const bool d = der >> l & 1;
    const int re = m.sf_re[sf0 + l];
    if (re <= -2) tag = 1;
    const int pos = d ? ni + __popcll(der & below) : __popcll(~der & below);
    fpos[sf0 + l] = (uint8_t)(pos | (re < 0 ? kPosBound : 0) | (re <= -2 ? kPosTag : 0));
  }
  for (int q = se0; q < se1; q++) {
    const int se = m.v_seid[q], cell = m.se_cell[q];
    uint32_t code = 0xFFFFFFFFu;
    int cnt = 0;
    for (int round = 0; round < 2; round++)
      for (int p = m.se_sfoff[se]; p < m.se_sfoff[se + 1]; p++) {
        const int l = m.se_sf[p] - sf0;
        if ((int)(der >> l & 1) != round || cnt == kSlotSrc) continue;
        uint32_t b = fpos[sf0 + l] & kPosMask;
        if (m.sf_le[sf0 + l] != cell) b |= kCodeRight;
        if (round) b |= kCodeDerived;
        code = (code & ~(0xFFu << (8 * cnt))) | b << (8 * cnt);
        cnt++;
      }
    scode[q] = code;
  }
  vstat[v] = ni | tag << 8 | skew << 9;
}

// ------------------------------------------------------------- LDS layout
// Per vertex, in doubles: the inverses (or the matrices they are formed from),
// the area vectors in place order, each stored face's flux from either side,
// the right-hand side and the face values, and for the forming kernels the
// slots' data and a broadcast buffer.
struct Lay {
  int A, fL, fh, fv, fhv, ty, sl, sivol, smu, scode, buf, total;
};
SFV_DEV __host__ Lay lds_layout(int lmat, int nim, int nfm, int nsm, bool form) {
  Lay o;
  int p = lmat;
  o.A = p; p += 3 * nfm;
  o.fL = p; p += 6 * nim;
  o.fh = p; p += 2 * nim;
  o.fv = p; p += 3 * nim;
  o.fhv = p; p += nim;
  o.ty = p; p += (nim + 1) / 2;
  o.sl = o.sivol = o.smu = o.scode = o.buf = p;
  if (form) {
    o.sl = p; p += nim;
    o.sivol = p; p += nsm;
    o.smu = p; p += nsm;
    o.scode = p; p += (nsm + 1) / 2;
    o.buf = p; p += 64;
  }
  o.total = p | 1;  // odd: the vertices of a wavefront start on different banks
  return o;
}

// 3x3 block (pe, po) of a vertex's momentum inverse: offset and strides.
// sym: the blocks on and below the diagonal; otherwise all of them.
struct Blk {
  int base, si, sj;
};
SFV_DEV Blk block_at(bool sym, int ni, int pe, int po) {
  Blk b;
  if (sym) {
    const bool up = pe < po;
    const int hi = up ? po : pe, lo = up ? pe : po;
    b.base = 9 * (tri(hi) + lo);
    b.si = up ? 1 : 3;
    b.sj = up ? 3 : 1;
  } else {
    b.base = 9 * (pe * ni + po);
    b.si = 3;
    b.sj = 1;
  }
  return b;
}
SFV_DEV int heat_at(bool sym, int ni, int pe, int po) {
  if (!sym) return pe * ni + po;
  return pe < po ? tri(po) + pe : tri(pe) + po;
}
SFV_DEV int mom_size(bool sym, int ni) { return 9 * (sym ? tri(ni) : ni * ni); }

SFV_DEV void load3(const double *A, int pos, double s, double *o) {
  o[0] = s * A[3 * pos];
  o[1] = s * A[3 * pos + 1];
  o[2] = s * A[3 * pos + 2];
}
SFV_DEV double dot3(const double *a, const double *b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }

// H += w_b A_b^T for the derived face b of H = sum over the stored faces:
// w_b = -(H A_b + A_b (tr(H) - A_b.H A_b / a^2) / 4) / a^2, the solution of b's
// own row
SFV_DEV void add_derived(double H[3][3], const double *Ab, double ia2) {
  double h[3];
  for (int i = 0; i < 3; i++) h[i] = dot3(H[i], Ab);
  const double q = dot3(Ab, h) * ia2, tr = H[0][0] + H[1][1] + H[2][2];
  const double c = 0.25 * (tr - q);
  for (int i = 0; i < 3; i++) {
    const double wb = -ia2 * (h[i] + Ab[i] * c);
    for (int j = 0; j < 3; j++) H[i][j] = H[i][j] + wb * Ab[j];
  }
}

// one slot lane's data: sub-element p, field f (0: the cell's own values, 1..3:
// the unit velocity along axis f; the unit temperature for f = 1)
struct SlotReg {
  int code, ms, posb;
  double V[3], th, mu, ivol, kv, c2, c3, ia2;
  double Ab[3], Q[3];
  double g[kSlotSrc][3], gh[kSlotSrc];
};

template <bool VAR>
SFV_DEV void slot_load(const DiffArgs &a, int q, SlotReg &r, double mu0) {
  const long cell = a.m.se_cell[q];
  r.code = (int)a.scode[q];
  r.ivol = a.sivol[q];
  r.mu = VAR && a.mu_cell ? a.mu_cell[cell] : a.p.mu;
  // kappa (ns_diffusion_module.F90:186-194)
  r.kv = (VAR && a.mu_cell ? r.mu * a.p.cv * kGamma / a.p.pr : a.p.kap) * r.ivol;
  r.c2 = r.mu - mu0;
  r.c3 = mu0 - (2.0 / 3.0) * r.mu;
  double u[5];
  for (int k = 0; k < 5; k++) u[k] = a.U[5 * cell + k];
  const double tau = 1.0 / u[0];
  for (int k = 0; k < 3; k++) r.V[k] = u[k + 1] * tau;
  // temp_u (ns_euler_primitives_module.F90:52-63)
  r.th = (u[4] * tau - 0.5 * (r.V[0] * r.V[0] + r.V[1] * r.V[1] + r.V[2] * r.V[2])) / a.p.cv;
}

// stored count, derived face and Q = sum of the stored area vectors
SFV_DEV void slot_faces(const double *A, SlotReg &r) {
  r.ms = 0;
  r.posb = -1;
  r.ia2 = 0.0;
  for (int d = 0; d < 3; d++) r.Q[d] = r.Ab[d] = 0.0;
#pragma unroll
  for (int e = 0; e < kSlotSrc; e++) {
    const int b = (r.code >> (8 * e)) & 0xFF;
    if (b != 0xFF) {
      double Ae[3];
      load3(A, b & kPosMask, b & kCodeRight ? -1.0 : 1.0, Ae);
      if (b & kCodeDerived) {
        r.posb = b & kPosMask;
        for (int d = 0; d < 3; d++) r.Ab[d] = Ae[d];
        r.ia2 = 1.0 / dot3(Ae, Ae);
      } else {
        r.ms++;
        for (int d = 0; d < 3; d++) r.Q[d] = r.Q[d] + Ae[d];
      }
    }
  }
}

// sigma = (c1 H + c2 H^T + c3 tr(H) I) ivol
SFV_DEV void stress(const double H[3][3], double c1, double c2, double c3, double ivol, double S[3][3]) {
  const double d = c3 * (H[0][0] + H[1][1] + H[2][2]);
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++) S[i][j] = ivol * (c1 * H[i][j] + c2 * H[j][i] + (i == j ? d : 0.0));
}

// g_l = column of S(l, p) V (f = 0) or S(l, p) e_f (f > 0) for the slot's
// stored faces; gh the heat system's.
SFV_DEV void slot_fluxes(const double *A, const int *ty, int f, SlotReg &r) {
  double H[3][3], S[3][3], Sn[3][3];
  for (int i = 0; i < 3; i++) {
    const double u = f == 0 ? r.V[i] : (f == i + 1 ? 1.0 : 0.0);
    for (int j = 0; j < 3; j++) H[i][j] = u * r.Q[j];
  }
  if (r.posb >= 0) add_derived(H, r.Ab, r.ia2);
  stress(H, r.mu, r.c2, r.c3, r.ivol, S);
  // boundary rows take the constant-viscosity form, scaled by the cell's mu
  stress(H, r.mu, 0.0, r.mu / 3.0, r.ivol, Sn);
  double q[3];
  const double qb = r.posb >= 0 ? dot3(r.Ab, r.Q) * r.ia2 : 0.0;
  for (int d = 0; d < 3; d++) q[d] = r.kv * (r.Q[d] - r.Ab[d] * qb);
  const double tf = f == 0 ? r.th : 1.0;
#pragma unroll
  for (int e = 0; e < kSlotSrc; e++)
    if (e < r.ms) {
      const int b = (r.code >> (8 * e)) & 0xFF, pos = b & kPosMask;
      const int t = ty[pos];
      double Ae[3];
      load3(A, pos, b & kCodeRight ? -1.0 : 1.0, Ae);
      for (int i = 0; i < 3; i++) {
        double x = dot3(S[i], Ae);
        if ((t & kTyV) == 1) x = dot3(Sn[i], Ae);
        r.g[e][i] = (t & kTyV) == 2 ? 0.0 : x;
      }
      r.gh[e] = (t >> kTyTShift & 3) == 2 ? 0.0 : tf * dot3(q, Ae);
    }
}

// ------------------------------------------------ inverses, row per lane
// A := A^-1 of each lane group's vertex: lane `row` holds row `row` (NR
// registers), padded with unit rows.  Gauss-Jordan on the transpose: the
// pivot lane's row is broadcast through LDS and every lane eliminates one
// entry of its own row; the registers rotate by one per step, so the pivot is
// always register 0 and the loop stays rolled.  PIV: partial pivoting over
// the not yet eliminated entries of the pivot lane's row.  Returns the row of
// the inverse that the lane holds in the end.
template <int NR, int LPV, bool PIV>
SFV_DEV int lane_inverse(double (&a)[NR], double *buf, int row) {
  int mine = row;
  for (int k = 0; k < NR; k++) {
    if (row == k) {
#pragma unroll
      for (int i = 0; i < NR; i++) buf[i] = a[i];
    }
    wsync_d();
    int p = 0;
    if (PIV) {
      double best = -1.0;
#pragma unroll
      for (int i = 0; i < NR; i++) {
        const double x = fabs(buf[i]);
        if (i < NR - k && x > best) {
          best = x;
          p = i;
        }
      }
      const double a0 = a[0];
      double ap = a0;
#pragma unroll
      for (int i = 1; i < NR; i++)
        if (i == p) {
          ap = a[i];
          a[i] = a0;
        }
      a[0] = ap;
      const int mk = __shfl(mine, k, LPV), mp = __shfl(mine, k + p, LPV);
      if (row == k) mine = mp;
      if (row == k + p && p != 0) mine = mk;
    }
    if (row == k) {
      a[0] = 1.0;
#pragma unroll
      for (int i = 1; i < NR; i++) a[i] = 0.0;
    }
    const double t = a[0] * (1.0 / buf[p]);
#pragma unroll
    for (int i = 1; i < NR; i++) {
      const double c = PIV ? (i == p ? buf[0] : buf[i]) : buf[i];
      a[i - 1] = __builtin_fma(-c, t, a[i]);
    }
    a[NR - 1] = t;
    wsync_d();
  }
  return mine;
}

template <int NR, int LPV>
SFV_DEV void momentum_inverse(double *Lm, double *buf, int ni, int row, bool piv) {
  double a[NR];
  const int l = row / 3, i = row - 3 * l;
  const bool in = row < 3 * ni;
#pragma unroll
  for (int c = 0; c < NR; c++)
    a[c] = in && c < 3 * ni ? Lm[9 * (l * ni + c / 3) + 3 * i + c % 3] : (row == c ? 1.0 : 0.0);
  wsync_d();
  const int mine = piv ? lane_inverse<NR, LPV, true>(a, buf, row) : lane_inverse<NR, LPV, false>(a, buf, row);
  const int ml = mine / 3, mi = mine - 3 * ml;
  if (in) {
#pragma unroll
    for (int c = 0; c < NR; c++)
      if (c < 3 * ni) Lm[9 * (ml * ni + c / 3) + 3 * mi + c % 3] = a[c];
  }
  wsync_d();
}

template <int NR, int LPV>
SFV_DEV void heat_inverse(double *Lh, double *buf, int ni, int row, bool piv) {
  double a[NR];
  const bool in = row < ni;
#pragma unroll
  for (int c = 0; c < NR; c++) a[c] = in && c < ni ? Lh[row * ni + c] : (row == c ? 1.0 : 0.0);
  wsync_d();
  const int mine = piv ? lane_inverse<NR, LPV, true>(a, buf, row) : lane_inverse<NR, LPV, false>(a, buf, row);
  if (in) {
#pragma unroll
    for (int c = 0; c < NR; c++)
      if (c < ni) Lh[mine * ni + c] = a[c];
  }
  wsync_d();
}

// Row i, columns j = 0..2 of the coupling of stored face l with stored face po
// of the same sub-element, the derived face eliminated; heat: its scalar.
struct Pair {
  double Al[3], Ab[3], ivol, c1, c2, c3, kv, ia2, AlAb;
  bool hasb;
};
SFV_DEV void coupling_row(const Pair &w, const double *Ae, int i, double *o) {
  const double d = dot3(w.Al, Ae);
  const double Aei = i == 0 ? Ae[0] : (i == 1 ? Ae[1] : Ae[2]);
  const double Ali = i == 0 ? w.Al[0] : (i == 1 ? w.Al[1] : w.Al[2]);
  const double Abi = i == 0 ? w.Ab[0] : (i == 1 ? w.Ab[1] : w.Ab[2]);
  const double k = w.hasb ? dot3(w.Ab, Ae) : 0.0;
  for (int j = 0; j < 3; j++) {
    const double dl = i == j ? 1.0 : 0.0;
    double t1 = d * dl, t2 = Aei * w.Al[j], t3 = Ae[j];
    if (w.hasb) {
      const double P = w.ia2 * (k * (dl - 0.25 * w.ia2 * Abi * w.Ab[j]) + 0.25 * Abi * Ae[j]);
      t1 = t1 - w.AlAb * P;
      t2 = t2 - Abi * w.ia2 * (k * (w.Al[j] - 0.25 * w.ia2 * w.AlAb * w.Ab[j]) + 0.25 * w.AlAb * Ae[j]);
      t3 = t3 - (0.75 * k * w.ia2 * w.Ab[j] + 0.25 * Ae[j]);
    }
    o[j] = w.ivol * (w.c1 * t1 + w.c2 * t2 + w.c3 * Ali * t3);
  }
}
SFV_DEV double coupling_heat(const Pair &w, const double *Ae) {
  double d = dot3(w.Al, Ae);
  if (w.hasb) d = d - w.AlAb * dot3(w.Ab, Ae) * w.ia2;
  return w.kv * d;
}

// a slot as the forming code sees it: its code, volume and viscosity
SFV_DEV void pair_slot(const DiffArgs &a, const double *A, int code, double ivol, double mu, double mu0, bool boundary,
                       Pair &w) {
  w.ivol = ivol;
  w.c1 = mu;
  w.c2 = boundary ? 0.0 : mu - mu0;
  w.c3 = boundary ? mu / 3.0 : mu0 - (2.0 / 3.0) * mu;
  w.kv = (a.mu_cell ? mu * a.p.cv * kGamma / a.p.pr : a.p.kap) * w.ivol;
  w.hasb = false;
  w.ia2 = 0.0;
  for (int d = 0; d < 3; d++) w.Ab[d] = 0.0;
  for (int e = 0; e < kSlotSrc; e++) {
    const int b = (code >> (8 * e)) & 0xFF;
    if (b != 0xFF && (b & kCodeDerived)) {
      w.hasb = true;
      load3(A, b & kPosMask, 1.0, w.Ab);
      w.ia2 = 1.0 / dot3(w.Ab, w.Ab);
    }
  }
}

struct Group {
  const double *A;
  const int *ty, *sl, *scode;
  const double *sivol, *smu;
};

// rows of N (momentum: row r = 3 l + i; heat: row l) into the full block layout
SFV_DEV void form_rows(const DiffArgs &a, const Group &g, int ni, int lane, int lpv, double mu0, double *Lm, double *Lh) {
  for (int r = lane; r < 3 * ni; r += lpv) {
    const int l = r / 3, i = r - 3 * l;
    const int t = g.ty[l] & kTyV;
    for (int po = 0; po < ni; po++)
      for (int j = 0; j < 3; j++) Lm[9 * (l * ni + po) + 3 * i + j] = 0.0;
    if (t == 2) {
      Lm[9 * (l * ni + l) + 4 * i] = 1.0;
      continue;
    }
    for (int side = 0; side < 2; side++) {
      const int p = g.sl[2 * l + side];
      if (p < 0) continue;
      Pair w;
      const int code = g.scode[p];
      pair_slot(a, g.A, code, g.sivol[p], g.smu[p], mu0, t == 1, w);
      load3(g.A, l, side ? -1.0 : 1.0, w.Al);
      w.AlAb = dot3(w.Al, w.Ab);
      for (int e = 0; e < kSlotSrc; e++) {
        const int b = (code >> (8 * e)) & 0xFF;
        if (b & kCodeDerived) break;  // the derived face or the end of the list
        double Ae[3], o[3];
        load3(g.A, b & kPosMask, b & kCodeRight ? -1.0 : 1.0, Ae);
        coupling_row(w, Ae, i, o);
        double *dst = Lm + 9 * (l * ni + (b & kPosMask)) + 3 * i;
        for (int j = 0; j < 3; j++) dst[j] = dst[j] + o[j];
      }
    }
  }
  for (int l = lane; l < ni; l += lpv) {
    const int t = g.ty[l] >> kTyTShift & 3;
    for (int po = 0; po < ni; po++) Lh[l * ni + po] = 0.0;
    if (t == 2) {
      Lh[l * ni + l] = 1.0;
      continue;
    }
    for (int side = 0; side < 2; side++) {
      const int p = g.sl[2 * l + side];
      if (p < 0) continue;
      Pair w;
      const int code = g.scode[p];
      pair_slot(a, g.A, code, g.sivol[p], g.smu[p], mu0, false, w);
      load3(g.A, l, side ? -1.0 : 1.0, w.Al);
      w.AlAb = dot3(w.Al, w.Ab);
      for (int e = 0; e < kSlotSrc; e++) {
        const int b = (code >> (8 * e)) & 0xFF;
        if (b & kCodeDerived) break;
        double Ae[3];
        load3(g.A, b & kPosMask, b & kCodeRight ? -1.0 : 1.0, Ae);
        double *dst = Lh + l * ni + (b & kPosMask);
        *dst = *dst + coupling_heat(w, Ae);
      }
    }
  }
}

// S : (H + V A_p^T) with the viscous stress S = mu (H + H^T - 2/3 tr(H) I) / vol
SFV_DEV double viscous_work(const double H[3][3], const SlotReg &r, const double *Ap) {
  const double tr = (2.0 / 3.0) * (H[0][0] + H[1][1] + H[2][2]);
  double work = 0.0;
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++)
      work = work + (H[i][j] + H[j][i] - (i == j ? tr : 0.0)) * (H[i][j] + r.V[i] * Ap[j]);
  return work * (r.mu * r.ivol);
}

// type of a stored face from its flags (and, tagged, its right code)
SFV_DEV int face_type(const DiffArgs &a, int fp, long s) {
  if (!(fp & kPosBound)) return 0;
  if (!(fp & kPosTag)) return 1 | 1 << kTyTShift;
  const int ib = -a.m.sf_re[s] - 1;
  return (a.p.bc_V_id[ib] == 2 ? 2 : 1) | (a.p.bc_T_id[ib] == 2 ? 2 : 1) << kTyTShift | ib << kTyBc;
}

// Modes of k_visc: form the inverses and apply them (kForm), store them too
// (kStore), or read stored ones in place (kGlobal, the large class).
enum { kForm = 0, kStore = 1, kGlobal = 2 };

// The scatter terms of every slot of a vertex with its diagonal block, LPV
// lanes per vertex: every residual with a viscosity per cell; once per mesh
// with a constant one, whose blocks depend on the mesh only (k_visc_apply then
// gives the residual's terms).
// (a) faces (area vectors, types) and the inverse into LDS; four lanes per
//     slot (fields f = 0..3 of SlotReg) load the cell;
// (b) f = 0 lanes put S V of each stored face into LDS, rows sum both sides;
// (c) rows: v = N^-1 f from LDS;
// (d) the lanes of a slot rebuild H for their field, f > 0 from the slot's own
//     blocks of N^-1, and write one row of kDiffSlot partials: rhs, and minus
//     the columns of the momentum block and the heat factor.
template <int LPV, int MODE>
__global__ __launch_bounds__(64) void k_visc(DiffArgs a) {
  constexpr bool FORM = MODE != kGlobal;
  extern __shared__ double lds_all[];
  const DevMesh &m = a.m;
  const int lb = xcd_block(a.vper_xcd);  // neighbouring vertices share cells
  if (lb >= a.vblocks) return;
  const int grp = threadIdx.x / LPV, lane = threadIdx.x % LPV;
  const long v_ = (long)lb * (blockDim.x / LPV) + grp;
  const bool live = v_ < m.V;
  const long v = live ? v_ : m.V - 1;  // spare lanes mirror the last vertex and store nothing
  double *const L = lds_all + (long)grp * a.lds_stride;
  const Lay o = lds_layout(a.lmat, a.nim, a.nfm, a.nsm, FORM);
  double *const A = L + o.A, *const fL = L + o.fL, *const fh = L + o.fh, *const fv = L + o.fv, *const fhv = L + o.fhv;
  int *const ty = (int *)(L + o.ty);
  const int sf0 = m.sf_off[v], nf = m.sf_off[v + 1] - sf0;
  const int se0 = m.se_off[v], ns = m.se_off[v + 1] - se0;
  const uint64_t dd = a.doff[v];
  const int ni = (int)(dd >> 48 & 0xFF);
  const bool tag = dd >> 56 & 1, skew = dd >> 57 & 1;
  double *const pre = a.pre + (dd & 0xFFFFFFFFFFFFull);
  const bool sym = MODE == kGlobal && !tag && !a.mu_cell;  // formed here: all blocks, in LDS
  const double mu0 = a.mu_cell ? *a.mu_min : a.p.mu0;
  // ---- (a)
  SlotReg r;
  bool walls = false;
  for (int l = lane; l < nf; l += LPV) {
    const long s = sf0 + l;
    const int fp = a.fpos[s], pos = fp & kPosMask;
    const double ar = m.sfn[3 * m.SF + s];
    for (int d = 0; d < 3; d++) A[3 * pos + d] = m.sfn[d * m.SF + s] * ar;
    if (pos < ni) {
      ty[pos] = face_type(a, fp, s);
      if (fp & kPosBound) {
        walls = true;
        for (int d = 0; d < 3; d++) fL[6 * pos + 3 + d] = 0.0;
        fh[2 * pos + 1] = 0.0;
      }
      if (FORM && (fp & kPosBound)) ((int *)(L + o.sl))[2 * pos + 1] = -1;
    }
  }
  if (FORM) {
    int *sl = (int *)(L + o.sl), *sc = (int *)(L + o.scode);
    for (int p = lane; p < ns; p += LPV) {
      const int code = (int)a.scode[se0 + p];
      sc[p] = code;
      L[o.sivol + p] = a.sivol[se0 + p];
      L[o.smu + p] = a.mu_cell ? a.mu_cell[m.se_cell[se0 + p]] : a.p.mu;
      for (int e = 0; e < kSlotSrc; e++) {
        const int b = (code >> (8 * e)) & 0xFF;
        if (b & kCodeDerived) break;
        sl[2 * (b & kPosMask) + (b & kCodeRight ? 1 : 0)] = p;
      }
    }
  }
  wsync_d();
  double *const Lm = L, *const Lh = L + 9 * ni * ni;
  if (FORM) {
    const Group g = {A, ty, (const int *)(L + o.sl), (const int *)(L + o.scode), L + o.sivol, L + o.smu};
    form_rows(a, g, ni, lane, LPV, mu0, Lm, Lh);
    wsync_d();
    // uniform over the wavefront: the larger vertex's size, and pivoting where
    // the matrix need not be positive definite
    const int big = LPV == 32 ? max(ni, __shfl_xor(ni, 32)) : ni;
    const int nw = __builtin_amdgcn_readfirstlane(big);
    const bool piv = a.pivot || __any(tag || (a.mu_cell && (walls || skew)));
    double *buf = L + o.buf;
    if (LPV == 32) {
      if (nw <= 4) momentum_inverse<12, LPV>(Lm, buf, ni, lane, piv);
      else if (nw <= 5) momentum_inverse<15, LPV>(Lm, buf, ni, lane, piv);
      else if (nw <= 6) momentum_inverse<18, LPV>(Lm, buf, ni, lane, piv);
      else if (nw <= 7) momentum_inverse<21, LPV>(Lm, buf, ni, lane, piv);
      else if (nw <= 8) momentum_inverse<24, LPV>(Lm, buf, ni, lane, piv);
      else momentum_inverse<30, LPV>(Lm, buf, ni, lane, piv);
      if (nw <= 6) heat_inverse<6, LPV>(Lh, buf, ni, lane, piv);
      else heat_inverse<10, LPV>(Lh, buf, ni, lane, piv);
    } else {
      if (nw <= 6) momentum_inverse<18, LPV>(Lm, buf, ni, lane, piv);
      else if (nw <= 12) momentum_inverse<36, LPV>(Lm, buf, ni, lane, piv);
      else if (nw <= 16) momentum_inverse<48, LPV>(Lm, buf, ni, lane, piv);
      else momentum_inverse<63, LPV>(Lm, buf, ni, lane, piv);
      if (nw <= 12) heat_inverse<12, LPV>(Lh, buf, ni, lane, piv);
      else heat_inverse<21, LPV>(Lh, buf, ni, lane, piv);
    }
  }
  if (MODE == kStore && live) {
    // value k of block q at pre[k nb + q], k = 9 the heat system's entry
    const bool half = !tag;
    const int nb = half ? tri(ni) : ni * ni;
    for (int q = lane; q < ni * ni; q += LPV) {
      const int pe = q / ni, po = q - pe * ni;
      if (half && po > pe) continue;
      double *out = pre + (half ? tri(pe) + po : q);
      for (int k = 0; k < 9; k++) out[k * nb] = Lm[9 * q + k];
      out[9 * nb] = Lh[q];
    }
  }
  const double *const Gm = MODE == kGlobal ? pre : Lm;
  const double *const Gh = MODE == kGlobal ? pre + mom_size(sym, ni) : Lh;
  // ---- (b)
  const int rounds = (4 * ns + LPV - 1) / LPV;
  for (int t = lane; t < 4 * ns; t += LPV) {
    slot_load<true>(a, se0 + (t >> 2), r, mu0);
    slot_faces(A, r);
    slot_fluxes(A, ty, t & 3, r);
    if ((t & 3) == 0)
#pragma unroll
      for (int e = 0; e < kSlotSrc; e++)
        if (e < r.ms) {
          const int b = (r.code >> (8 * e)) & 0xFF, pos = b & kPosMask, side = b & kCodeRight ? 1 : 0;
          for (int d = 0; d < 3; d++) fL[6 * pos + 3 * side + d] = r.g[e][d];
          fh[2 * pos + side] = r.gh[e];
        }
  }
  wsync_d();
  for (int q = lane; q < 3 * ni; q += LPV) {
    const int l = q / 3, i = q - 3 * l;
    double x = fL[6 * l + i] + fL[6 * l + 3 + i];
    if (tag && (ty[l] & kTyV) == 2) x = a.p.bc_val_V[ty[l] >> kTyBc][i];
    fv[q] = x;
  }
  for (int l = lane; l < ni; l += LPV) {
    double x = fh[2 * l] + fh[2 * l + 1];
    if (tag && (ty[l] >> kTyTShift & 3) == 2) x = a.p.bc_val_T[ty[l] >> kTyBc];
    fhv[l] = x;
  }
  wsync_d();
  // ---- (c): the face values take the places of the one-sided fluxes
  double *const Vf = fL, *const Tf = fh;
  for (int q = lane; q < 3 * ni; q += LPV) {
    const int l = q / 3, i = q - 3 * l;
    double acc = 0.0;
    for (int po = 0; po < ni; po++) {
      const Blk b = block_at(sym, ni, l, po);
      const double *x = Gm + b.base + b.si * i;
      for (int j = 0; j < 3; j++) acc = acc + x[b.sj * j] * fv[3 * po + j];
    }
    Vf[q] = acc;
  }
  for (int l = lane; l < ni; l += LPV) {
    double acc = 0.0;
    for (int po = 0; po < ni; po++) acc = acc + Gh[heat_at(sym, ni, l, po)] * fhv[po];
    Tf[l] = acc;
  }
  wsync_d();
  // ---- (d)
  const bool mom = a.parts & 1, heat = a.parts & 2;
  for (int t = lane; t < 4 * ns; t += LPV) {
    const int f = t & 3;
    if (rounds > 1) {
      slot_load<true>(a, se0 + (t >> 2), r, mu0);
      slot_faces(A, r);
      slot_fluxes(A, ty, f, r);
    }
    double H[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, h[3] = {0, 0, 0};
#pragma unroll
    for (int e = 0; e < kSlotSrc; e++)
      if (e < r.ms) {
        const int be = (r.code >> (8 * e)) & 0xFF, pe = be & kPosMask;
        double w[3], wt;
        if (f == 0) {
          for (int i = 0; i < 3; i++) w[i] = Vf[3 * pe + i] - r.V[i];
          wt = Tf[pe] - r.th;
        } else {
          for (int i = 0; i < 3; i++) w[i] = f == i + 1 ? -1.0 : 0.0;
          wt = -1.0;
#pragma unroll
          for (int e2 = 0; e2 < kSlotSrc; e2++)
            if (e2 < r.ms) {
              const int po = (r.code >> (8 * e2)) & kPosMask;
              const Blk b = block_at(sym, ni, pe, po);
              const double *x = Gm + b.base;
              for (int i = 0; i < 3; i++)
                for (int j = 0; j < 3; j++) w[i] = w[i] + x[b.si * i + b.sj * j] * r.g[e2][j];
              if (f == 1) wt = wt + Gh[heat_at(sym, ni, pe, po)] * r.gh[e2];
            }
        }
        double Ae[3];
        load3(A, pe, be & kCodeRight ? -1.0 : 1.0, Ae);
        for (int j = 0; j < 3; j++) {
          for (int i = 0; i < 3; i++) H[i][j] = H[i][j] + w[i] * Ae[j];
          h[j] = h[j] + wt * Ae[j];
        }
      }
    if (r.posb >= 0) {
      add_derived(H, r.Ab, r.ia2);
      const double hb = dot3(h, r.Ab) * r.ia2;
      for (int j = 0; j < 3; j++) h[j] = h[j] - hb * r.Ab[j];
    }
    double Ap[3], S[3][3], out[4];
    for (int d = 0; d < 3; d++) Ap[d] = r.Q[d] + r.Ab[d];
    stress(H, r.mu, r.c2, r.c3, r.ivol, S);
    for (int i = 0; i < 3; i++) out[i] = dot3(S[i], Ap);
    // f = 0: the heat rhs; f = 1: S~^T N^-1 S - (row sum of S~^T) of the slot's
    // own cell.  The reference's remaining rhs terms multiply dtheta_dU . U, which
    // is zero: the temperature is homogeneous of degree 0 in the state.
    const double hq = r.kv * dot3(h, Ap);
    // rhs = sigma(H) A_p - D V_p, summed over the slot's four lanes
    double sum[3];
    for (int i = 0; i < 3; i++) {
      const double Vf_ = f == 1 ? r.V[0] : (f == 2 ? r.V[1] : r.V[2]);
      double x = f == 0 ? out[i] : -(out[i] * Vf_);
      x = x + __shfl_xor(x, 1);
      sum[i] = x + __shfl_xor(x, 2);
    }
    if (f == 0) {
      const double work = viscous_work(H, r, Ap);
      for (int i = 0; i < 3; i++) out[i] = mom ? sum[i] : 0.0;
      out[3] = (mom ? work : 0.0) + (heat ? hq : 0.0);
    } else {
      for (int i = 0; i < 3; i++) out[i] = mom ? -out[i] : 0.0;
      out[3] = f == 1 && heat ? -hq : 0.0;
    }
    if (live) {
      double2 *row = (double2 *)(a.PD + (long)kDiffSlot * (se0 + (t >> 2)) + 4 * f);
      row[0] = make_double2(out[0], out[1]);
      row[1] = make_double2(out[2], out[3]);
    }
  }
}

// The scatter terms of every slot with a constant viscosity: rhs rows of four
// partials (rho u, rho v, rho w without the block's own-cell part; E), one lane
// per slot.  16 lanes per vertex (four vertices per wavefront) on prism and quad
// meshes: a prism vertex has 6 slots, 12 faces and 21 blocks.
// The face values v = N^-1 f: a lane owns whole blocks (the first kHold of them
// loaded at the start, in flight while the slots are read), forms their products
// with the two faces they couple, and the products meet in LDS, where each row
// sums its own in face order.  LDS holds the products only, sized per wavefront
// for the vertices it has.
// GLOBAL (large class): one lane per row reads its blocks in place (a workgroup
// per vertex, two lanes per row: 81 us instead of 60 on tets 15^3).
// On tri 1024^2 (2.1M prisms and vertices) the stored products of the dense
// matrices took 4.88 ms per residual (19 GB, 4.6 TB/s); the inverses (4 GB)
// staged in LDS, 9 wavefronts per CU, 2.66 ms; like this 1.46 ms, bound by
// instruction issue (0.8 ms of it) and latency, 3.4 TB/s.
SFV_DEV void put4(double *p, double a, double b, double c, double d) {
  ((double2 *)p)[0] = make_double2(a, b);
  ((double2 *)p)[1] = make_double2(c, d);
}
SFV_DEV void get4(const double *p, double *o) {
  const double2 a = ((const double2 *)p)[0], b = ((const double2 *)p)[1];
  o[0] = a.x;
  o[1] = a.y;
  o[2] = b.x;
  o[3] = b.y;
}

template <int LPV, bool GLOBAL>
__global__ __launch_bounds__(256, 3) void k_visc_apply(DiffArgs a) {
  extern __shared__ double lds_all[];
  constexpr int kHold = GLOBAL ? 0 : 2;
  const DevMesh &m = a.m;
  const int lb = xcd_block(a.vper_xcd);  // neighbouring vertices share cells
  if (lb >= a.vblocks) return;
  constexpr int per = 64 / LPV;
  const int lane = threadIdx.x % LPV, wave = threadIdx.x >> 6, grp = (threadIdx.x & 63) / LPV;
  const long w = (long)lb * (blockDim.x >> 6) + wave;
  const long v = apply_vertex(w, per, grp, m.V);
  if (v < 0) return;  // uniform over the wavefront, which shares no barrier with the others
  const bool live = w * per + grp < m.V;  // spare lanes mirror the last vertex and store nothing
  const int sf0 = m.sf_off[v], nf = m.sf_off[v + 1] - sf0;
  const int se0 = m.se_off[v], ns = m.se_off[v + 1] - se0;
  const uint64_t dd = a.doff[v];
  const int ni = (int)(dd >> 48 & 0xFF);
  const bool tag = dd >> 56 & 1, sym = !tag;
  const double *const pre = a.pre + (dd & 0xFFFFFFFFFFFFull);
  const double mu0 = a.p.mu0;
  const int nb = sym ? tri(ni) : ni * ni;
  double x[kHold ? kHold : 1][10];
#pragma unroll
  for (int h = 0; h < kHold; h++)
    if (lane + h * LPV < nb)
#pragma unroll
      for (int k = 0; k < 10; k++) x[h][k] = pre[k * nb + lane + h * LPV];
  SlotReg r;
  if (lane < ns) slot_load<false>(a, se0 + lane, r, mu0);
  // this vertex's LDS, behind those of the wavefront's earlier vertices
  double *L = lds_all + (long)wave * a.lds_stride;
  {
    const int size = apply_lds<GLOBAL>(ni, nf);
    for (int q = 0; q < per - 1; q++) {
      const int sq = __shfl(size, q * LPV);
      if (q < grp) L += sq;
    }
  }
  double *const fL = L;  // [ni][2][4] one-sided fluxes, then the block products [ni][ni][4]
  double *const fv = L + (GLOBAL ? 8 * ni : (ni > 2 ? 4 * ni * ni : 8 * ni));  // [ni][4] rhs, then the face values
  double *const A = fv + 4 * ni;
  int *const ty = (int *)(A + 3 * nf);
  for (int l = lane; l < nf; l += LPV) {
    const long s = sf0 + l;
    const int fp = a.fpos[s], pos = fp & kPosMask;
    const double ar = m.sfn[3 * m.SF + s];
    for (int d = 0; d < 3; d++) A[3 * pos + d] = m.sfn[d * m.SF + s] * ar;
    if (pos < ni) {
      ty[pos] = face_type(a, fp, s);
      if (fp & kPosBound)
        for (int d = 0; d < 4; d++) fL[8 * pos + 4 + d] = 0.0;
    }
  }
  wsync_d();
  const int rounds = (ns + LPV - 1) / LPV;
  for (int t = lane; t < ns; t += LPV) {
    if (t != lane) slot_load<false>(a, se0 + t, r, mu0);
    slot_faces(A, r);
    double S[3][3], q[3];
    {
      double H[3][3];
      for (int i = 0; i < 3; i++)
        for (int j = 0; j < 3; j++) H[i][j] = r.V[i] * r.Q[j];
      if (r.posb >= 0) add_derived(H, r.Ab, r.ia2);
      stress(H, r.mu, r.c2, r.c3, r.ivol, S);
      const double qb = r.posb >= 0 ? dot3(r.Ab, r.Q) * r.ia2 : 0.0, kt = r.kv * r.th;
      for (int d = 0; d < 3; d++) q[d] = kt * (r.Q[d] - r.Ab[d] * qb);
    }
#pragma unroll
    for (int e = 0; e < kSlotSrc; e++)
      if (e < r.ms) {
        const int b = (r.code >> (8 * e)) & 0xFF;
        double Ae[3];
        load3(A, b & kPosMask, b & kCodeRight ? -1.0 : 1.0, Ae);
        put4(fL + 8 * (b & kPosMask) + (b & kCodeRight ? 4 : 0), dot3(S[0], Ae), dot3(S[1], Ae), dot3(S[2], Ae),
             dot3(q, Ae));
      }
  }
  wsync_d();
  for (int q = lane; q < 4 * ni; q += LPV) {
    const int l = q >> 2, i = q & 3;
    double f = fL[8 * l + i] + fL[8 * l + 4 + i];
    if (tag) {
      const int t = ty[l], ib = t >> kTyBc;
      if (i < 3 ? (t & kTyV) == 2 : (t >> kTyTShift & 3) == 2) f = i < 3 ? a.p.bc_val_V[ib][i] : a.p.bc_val_T[ib];
    }
    fv[q] = f;
  }
  wsync_d();
  if (GLOBAL) {
    double *const vf = fL;
    for (int q = lane; q < 3 * ni; q += LPV) {
      const int l = q / 3, i = q - 3 * l;
      double acc = 0.0;
      for (int po = 0; po < ni; po++) {
        const Blk b = block_at(sym, ni, l, po);
        const double *y = pre + b.base + b.si * i;
        for (int j = 0; j < 3; j++) acc = acc + y[b.sj * j] * fv[4 * po + j];
      }
      vf[4 * l + i] = acc;
    }
    const double *const ph = pre + mom_size(sym, ni);
    for (int l = lane; l < ni; l += LPV) {
      double acc = 0.0;
      for (int po = 0; po < ni; po++) acc = acc + ph[heat_at(sym, ni, l, po)] * fv[4 * po + 3];
      vf[4 * l + 3] = acc;
    }
  } else {
    auto products = [&](int b, const double *y) {
      int hi, lo;
      if (sym) {
        hi = (int)((sqrtf(8.0f * b + 1.0f) - 1.0f) * 0.5f);
        lo = b - tri(hi);
      } else {
        hi = b / ni;
        lo = b - hi * ni;
      }
      double f[4], g[4];
      get4(fv + 4 * lo, f);
      get4(fv + 4 * hi, g);
      put4(fL + 4 * (hi * ni + lo), dot3(y, f), dot3(y + 3, f), dot3(y + 6, f), y[9] * f[3]);
      if (sym && hi != lo)
        put4(fL + 4 * (lo * ni + hi), y[0] * g[0] + y[3] * g[1] + y[6] * g[2], y[1] * g[0] + y[4] * g[1] + y[7] * g[2],
             y[2] * g[0] + y[5] * g[1] + y[8] * g[2], y[9] * g[3]);
    };
#pragma unroll
    for (int h = 0; h < kHold; h++)
      if (lane + h * LPV < nb) products(lane + h * LPV, x[h]);
    for (int b = lane + kHold * LPV; b < nb; b += LPV) {
      double y[10];
#pragma unroll
      for (int k = 0; k < 10; k++) y[k] = pre[k * nb + b];
      products(b, y);
    }
    wsync_d();
    for (int q = lane; q < 4 * ni; q += LPV) {
      const double *row = fL + 4 * ni * (q >> 2) + (q & 3);
      double acc = 0.0;
      for (int po = 0; po < ni; po++) acc = acc + row[4 * po];
      fv[q] = acc;
    }
  }
  wsync_d();
  const double *const Vf = GLOBAL ? fL : fv;
  for (int t = lane; t < ns; t += LPV) {
    if (rounds > 1) {
      slot_load<false>(a, se0 + t, r, mu0);
      slot_faces(A, r);
    }
    double H[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, h[3] = {0, 0, 0};
#pragma unroll
    for (int e = 0; e < kSlotSrc; e++)
      if (e < r.ms) {
        const int be = (r.code >> (8 * e)) & 0xFF, pe = be & kPosMask;
        double w[4], Ae[3];
        get4(Vf + 4 * pe, w);
        for (int i = 0; i < 3; i++) w[i] = w[i] - r.V[i];
        const double wt = w[3] - r.th;
        load3(A, pe, be & kCodeRight ? -1.0 : 1.0, Ae);
        for (int j = 0; j < 3; j++) {
          for (int i = 0; i < 3; i++) H[i][j] = H[i][j] + w[i] * Ae[j];
          h[j] = h[j] + wt * Ae[j];
        }
      }
    if (r.posb >= 0) {
      add_derived(H, r.Ab, r.ia2);
      const double hb = dot3(h, r.Ab) * r.ia2;
      for (int j = 0; j < 3; j++) h[j] = h[j] - hb * r.Ab[j];
    }
    double Ap[3], S[3][3], out[4];
    for (int d = 0; d < 3; d++) Ap[d] = r.Q[d] + r.Ab[d];
    stress(H, r.mu, r.c2, r.c3, r.ivol, S);
    for (int i = 0; i < 3; i++) out[i] = dot3(S[i], Ap);
    out[3] = viscous_work(H, r, Ap) + r.kv * dot3(h, Ap);
    if (live) {
      double2 *row = (double2 *)(a.PD + (long)kDiffRow * (se0 + t));
      row[0] = make_double2(out[0], out[1]);
      row[1] = make_double2(out[2], out[3]);
    }
  }
}

// -------------------------------------- inverses of the large class
// One 256-thread workgroup per vertex: thread (ri, cj) of a 16 x 16 grid holds
// the entries (ri + 16 i, cj + 16 j), i, j < T, in registers, formed from the
// area vectors in place.  A Gauss-Jordan step broadcasts the pivot's column
// and row through LDS (two buffers, one barrier per step); PIV picks the
// pivot row among the unused ones and permutes on the way out.
template <int T>
SFV_DEV void tile_inverse(double (&x)[T][T], int n, double (*col)[16 * T], double (*rw)[16 * T], int *prow, bool piv) {
  const int ri = threadIdx.x & 15, cj = threadIdx.x >> 4, lane = threadIdx.x & 63;
  uint64_t used[3] = {0, 0, 0};
#pragma unroll
  for (int q = 0; q < T; q++)
    for (int kr = 0; kr < 16; kr++) {
      const int k = 16 * q + kr;
      if (k >= n) break;  // uniform
      double *cb = col[k & 1], *rb = rw[k & 1];
      if (cj == kr)
#pragma unroll
        for (int i = 0; i < T; i++) cb[ri + 16 * i] = x[i][q];
      int p = k;
      if (piv) {
        __syncthreads();
        double best = -1.0;
        p = n;
        for (int i = lane; i < n; i += 64)
          if (!(used[i >> 6] >> (i & 63) & 1) && fabs(cb[i]) > best) {
            best = fabs(cb[i]);
            p = i;
          }
        for (int off = 32; off > 0; off >>= 1) {
          const double ob = __shfl_xor(best, off);
          const int op = __shfl_xor(p, off);
          if (ob > best || (ob == best && op < p)) {
            best = ob;
            p = op;
          }
        }
        if (p >= n) {  // no comparable entry (NaN): the first unused row
          p = 0;
          while (used[p >> 6] >> (p & 63) & 1) p++;
        }
        p = __builtin_amdgcn_readfirstlane(p);
        used[p >> 6] |= 1ull << (p & 63);
      }
      if (threadIdx.x == 0) prow[k] = p;
      const int pr = p & 15, pi = p >> 4;
      if (ri == pr)
#pragma unroll
        for (int i = 0; i < T; i++)
          if (i == pi)
#pragma unroll
            for (int j = 0; j < T; j++) rb[cj + 16 * j] = x[i][j];
      __syncthreads();
      const double rp = 1.0 / cb[p];
      if (cj == kr)
#pragma unroll
        for (int i = 0; i < T; i++) x[i][q] = 0.0;
      double t[T];
#pragma unroll
      for (int j = 0; j < T; j++) t[j] = (j == q && cj == kr) ? rp : rb[cj + 16 * j] * rp;
#pragma unroll
      for (int i = 0; i < T; i++) {
        const double c = cb[ri + 16 * i];
        const bool prw = ri == pr && i == pi;
#pragma unroll
        for (int j = 0; j < T; j++) x[i][j] = prw ? t[j] : __builtin_fma(-c, t[j], x[i][j]);
      }
    }
  __syncthreads();
}

template <int T>
__global__ __launch_bounds__(256) void k_visc_tile(DiffArgs a) {
  __shared__ double A[3 * kDiffMaxSub], sivol[kDiffMaxSub], smu[kDiffMaxSub];
  __shared__ int ty[kDiffMaxSub], sl[2 * kDiffMaxSub], sc[kDiffMaxSub];
  __shared__ double col[2][16 * T], rw[2][16 * T];
  __shared__ int prow[16 * T], inv[16 * T];
  __shared__ int any_wall;
  const DevMesh &m = a.m;
  const long v = blockIdx.x;
  const int tid = threadIdx.x;
  const int sf0 = m.sf_off[v], nf = m.sf_off[v + 1] - sf0;
  const int se0 = m.se_off[v], ns = m.se_off[v + 1] - se0;
  const uint64_t dd = a.doff[v];
  const int ni = (int)(dd >> 48 & 0xFF);
  const bool tag = dd >> 56 & 1, sym = !tag && !a.mu_cell;
  double *const pre = a.pre + (dd & 0xFFFFFFFFFFFFull);
  const double mu0 = a.mu_cell ? *a.mu_min : a.p.mu0;
  if (tid == 0) any_wall = 0;
  if (tid < 2 * kDiffMaxSub) sl[tid] = -1;
  __syncthreads();
  if (tid < nf) {
    const long s = sf0 + tid;
    const int fp = a.fpos[s], pos = fp & kPosMask;
    const double ar = m.sfn[3 * m.SF + s];
    for (int d = 0; d < 3; d++) A[3 * pos + d] = m.sfn[d * m.SF + s] * ar;
    if (pos < ni) {
      ty[pos] = face_type(a, fp, s);
      if (fp & kPosBound) any_wall = 1;
    }
  }
  if (tid < ns) {
    const int code = (int)a.scode[se0 + tid];
    sc[tid] = code;
    sivol[tid] = a.sivol[se0 + tid];
    smu[tid] = a.mu_cell ? a.mu_cell[m.se_cell[se0 + tid]] : a.p.mu;
    for (int e = 0; e < kSlotSrc; e++) {
      const int b = (code >> (8 * e)) & 0xFF;
      if (b & kCodeDerived) break;
      sl[2 * (b & kPosMask) + (b & kCodeRight ? 1 : 0)] = tid;
    }
  }
  __syncthreads();
  const bool piv = a.pivot || tag || (a.mu_cell && (any_wall || (dd >> 57 & 1)));
  const int ri = tid & 15, cj = tid >> 4;
  // entry (l, po) of a system: the sub-elements the two faces share
  auto shared_slots = [&](int l, int po, int side) -> int {
    const int p = sl[2 * l + side];
    return p >= 0 && (p == sl[2 * po] || p == sl[2 * po + 1]) ? p : -1;
  };
  auto pair_of = [&](int l, int po, int side, int p, bool boundary, Pair &w, double *Ae) {
    pair_slot(a, A, sc[p], sivol[p], smu[p], mu0, boundary, w);
    load3(A, l, side ? -1.0 : 1.0, w.Al);
    w.AlAb = dot3(w.Al, w.Ab);
    load3(A, po, p == sl[2 * po] ? 1.0 : -1.0, Ae);
  };
  {  // momentum
    const int n = 3 * ni;
    double x[T][T];
#pragma unroll
    for (int i = 0; i < T; i++)
#pragma unroll
      for (int j = 0; j < T; j++) {
        const int rr = ri + 16 * i, cc = cj + 16 * j;
        double val = rr == cc ? 1.0 : 0.0;
        if (rr < n && cc < n) {
          const int l = rr / 3, po = cc / 3, t = ty[l] & kTyV;
          if (t != 2) {
            val = 0.0;
            for (int side = 0; side < 2; side++) {
              const int p = shared_slots(l, po, side);
              if (p >= 0) {
                Pair w;
                double Ae[3], o[3];
                pair_of(l, po, side, p, t == 1, w, Ae);
                coupling_row(w, Ae, rr - 3 * l, o);
                const int jj = cc - 3 * po;
                val = val + (jj == 0 ? o[0] : (jj == 1 ? o[1] : o[2]));
              }
            }
          }
        }
        x[i][j] = val;
      }
    tile_inverse<T>(x, n, col, rw, prow, piv);
    if (tid < n) inv[prow[tid]] = tid;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < T; i++)
#pragma unroll
      for (int j = 0; j < T; j++) {
        const int rr = ri + 16 * i, cc = cj + 16 * j;
        if (rr < n && cc < n) {
          const int orow = inv[rr], ocol = prow[cc];
          const int pe = orow / 3, po = ocol / 3;
          if (!sym || pe >= po) {
            const Blk b = block_at(sym, ni, pe, po);
            pre[b.base + b.si * (orow - 3 * pe) + b.sj * (ocol - 3 * po)] = x[i][j];
          }
        }
      }
    __syncthreads();
  }
  {  // heat: at most 64 unknowns
    constexpr int TH = 4;
    double x[TH][TH];
#pragma unroll
    for (int i = 0; i < TH; i++)
#pragma unroll
      for (int j = 0; j < TH; j++) {
        const int l = ri + 16 * i, po = cj + 16 * j;
        double val = l == po ? 1.0 : 0.0;
        if (l < ni && po < ni && (ty[l] >> kTyTShift & 3) != 2) {
          val = 0.0;
          for (int side = 0; side < 2; side++) {
            const int p = shared_slots(l, po, side);
            if (p >= 0) {
              Pair w;
              double Ae[3];
              pair_of(l, po, side, p, false, w, Ae);
              val = val + coupling_heat(w, Ae);
            }
          }
        }
        x[i][j] = val;
      }
    tile_inverse<TH>(x, ni, (double(*)[16 * TH])col, (double(*)[16 * TH])rw, prow, piv);
    if (tid < ni) inv[prow[tid]] = tid;
    __syncthreads();
    double *const ph = pre + mom_size(sym, ni);
#pragma unroll
    for (int i = 0; i < TH; i++)
#pragma unroll
      for (int j = 0; j < TH; j++) {
        const int rr = ri + 16 * i, cc = cj + 16 * j;
        if (rr < ni && cc < ni) {
          const int pe = inv[rr], po = prow[cc];
          if (!sym || pe >= po) ph[heat_at(sym, ni, pe, po)] = x[i][j];
        }
      }
  }
}

// The cells' sums of their slots' rows in increasing vertex id.  ROW values per
// row, one lane per (cell, value), so a row is read by consecutive lanes and up
// to kDgBatch rows are in flight per lane.
// ROW = kDiffSlot: rdiff and, with BLOCKS, the blocks dblk (nine entries of the
// momentum block by column, the heat factor, all negated) from full rows.
// ROW = kDiffRow: rdiff from rows without the own-cell part, which the cell's
// block adds: rhs += dblk V.
constexpr int kDgBatch = 8;
template <int ROW>
__global__ __launch_bounds__(256) void k_diff_gather(DiffArgs a, int rhs, int blocks) {
  constexpr int kCells = 256 / ROW;
  const DevMesh &m = a.m;
  const int lb = xcd_block(a.cper_xcd);
  if (lb >= a.cblocks) return;  // uniform over the workgroup
  const int t = threadIdx.x, cl = t / ROW, k = t - cl * ROW;
  const long c = (long)lb * kCells + cl;
  if (c >= m.C) return;
  const int b = m.e_voff[c], nv = m.e_voff[c + 1] - b;
  double own = 0.0;
  if (ROW == kDiffRow && k < 3) {
    const double *u = a.U + 5 * c, *D = a.dblk + (long)kDiffBlk * c;
    const double tau = 1.0 / u[0];
    own = (D[k] * u[1] + D[3 + k] * u[2] + D[6 + k] * u[3]) * tau;
  }
  double acc = 0.0;
  for (int j0 = 0; j0 < nv; j0 += kDgBatch) {
    int sl[kDgBatch];
#pragma unroll
    for (int u = 0; u < kDgBatch; u++) sl[u] = j0 + u < nv ? m.c_slot[b + j0 + u] : 0;
    double x[kDgBatch];
#pragma unroll
    for (int u = 0; u < kDgBatch; u++) x[u] = a.PD[(long)ROW * sl[u] + k];
#pragma unroll
    for (int u = 0; u < kDgBatch; u++)
      if (j0 + u < nv) acc = acc + x[u];
  }
  const int f = k >> 2, i = k & 3;
  if (f == 0) {
    if (rhs) a.rdiff[4 * c + i] = acc + own;
  } else if (blocks) {
    if (i < 3) a.dblk[(long)kDiffBlk * c + 3 * (f - 1) + i] = acc;
    if (k == 7) a.dblk[(long)kDiffBlk * c + 9] = acc;
  }
}

// diag(5, 5, C) of the state's blocks (diff_block)
__global__ __launch_bounds__(256) void k_diff_expand(long C, const double *U, const double *dblk, double cv,
                                                     double *diag) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= C) return;
  double D[25];
  diff_block(U + 5 * c, dblk + (long)kDiffBlk * c, cv, D);
  for (int q = 0; q < 25; q++) diag[25 * c + q] = D[q];
}

hipError_t launch_lds(void (*fn)(DiffArgs), unsigned threads, int per, size_t lds, DiffArgs a, hipStream_t s) {
  if (lds > (64u << 10)) {
    hipError_t e = hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  a.vblocks = (int)((a.m.V + per - 1) / per);
  a.vper_xcd = (a.vblocks + 7) / 8;
  hipLaunchKernelGGL(fn, dim3(8 * a.vper_xcd), dim3(threads), lds, s, a);
  return hipGetLastError();
}

template <int LPV, int MODE>
hipError_t launch_visc(DiffArgs a, hipStream_t s) {
  constexpr bool FORM = MODE != kGlobal;
  a.lmat = FORM ? 10 * a.nim * a.nim : 0;
  a.lds_stride = lds_layout(a.lmat, a.nim, a.nfm, a.nsm, FORM).total;
  return launch_lds(k_visc<LPV, MODE>, 64, 64 / LPV, sizeof(double) * (64 / LPV) * a.lds_stride, a, s);
}

template <int LPV, bool GLOBAL>
hipError_t launch_apply(DiffArgs a, hipStream_t s) {
  // doubles of LDS per wavefront: of the fullest one, or of the largest vertices
  a.lds_stride = GLOBAL ? apply_lds<true>(a.nim, a.nfm) : a.lds_wave;
  // four wavefronts per workgroup where their LDS fits in 64 KB, else one
  const unsigned threads = sizeof(double) * 4 * a.lds_stride <= (64u << 10) ? 256 : 64;
  const size_t lds = sizeof(double) * (threads / 64) * a.lds_stride;
  return launch_lds(k_visc_apply<LPV, GLOBAL>, threads, threads / LPV, lds, a, s);
}

}  // namespace

void launch_diff_tables(const DevMesh &m, int *vstat, uint8_t *fpos, uint32_t *scode, double *sivol, hipStream_t s) {
  hipLaunchKernelGGL(k_diff_tables, dim3((unsigned)((m.V + 255) / 256)), dim3(256), 0, s, m, vstat, fpos, scode, sivol);
}

template <int ROW>
static hipError_t launch_gather(DiffArgs a, int rhs, int blocks, hipStream_t s) {
  a.cblocks = (int)((a.m.C + 256 / ROW - 1) / (256 / ROW));
  a.cper_xcd = (a.cblocks + 7) / 8;
  hipLaunchKernelGGL(k_diff_gather<ROW>, dim3(8 * a.cper_xcd), dim3(256), 0, s, a, rhs, blocks);
  return hipGetLastError();
}

static hipError_t launch_tile(DiffArgs a, hipStream_t s) {
  const int n = 3 * a.nim;
  const dim3 g((unsigned)a.m.V), b(256);
  if (n <= 112)
    hipLaunchKernelGGL(k_visc_tile<7>, g, b, 0, s, a);
  else
    hipLaunchKernelGGL(k_visc_tile<12>, g, b, 0, s, a);
  return hipGetLastError();
}

hipError_t launch_diff_setup(int cls, DiffArgs a, hipStream_t s) {
  hipError_t e;
  if (cls == kDiffHalf) {
    e = launch_visc<32, kStore>(a, s);
  } else if (cls == kDiffWave) {
    e = launch_visc<64, kStore>(a, s);
  } else {
    if ((e = launch_tile(a, s)) != hipSuccess) return e;
    e = launch_visc<64, kGlobal>(a, s);
  }
  if (e != hipSuccess) return e;
  return launch_gather<kDiffSlot>(a, 0, 1, s);
}

hipError_t launch_diff_terms(int cls, DiffArgs a, hipStream_t s) {
  if (a.mu_cell) {
    if (cls == kDiffHalf) return launch_visc<32, kForm>(a, s);
    if (cls == kDiffWave) return launch_visc<64, kForm>(a, s);
    hipError_t e = launch_tile(a, s);
    return e != hipSuccess ? e : launch_visc<64, kGlobal>(a, s);
  }
  if (cls == kDiffHalf) return launch_apply<16, false>(a, s);
  if (cls == kDiffWave) return launch_apply<32, false>(a, s);
  return launch_apply<64, true>(a, s);
}

hipError_t launch_diff_gather(DiffArgs a, hipStream_t s) {
  return a.mu_cell ? launch_gather<kDiffSlot>(a, 1, 1, s) : launch_gather<kDiffRow>(a, 1, 0, s);
}

hipError_t launch_diff_expand(long C, const double *U, const double *dblk, double cv, double *diag, hipStream_t s) {
  hipLaunchKernelGGL(k_diff_expand, dim3((unsigned)((C + 255) / 256)), dim3(256), 0, s, C, U, dblk, cv, diag);
  return hipGetLastError();
}

}  // namespace sfv
