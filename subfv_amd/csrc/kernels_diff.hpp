// Viscous terms of compute_rhs_ns (src/ns/ns_main.F90:170-175): the nodal
// momentum system of ns_vectorial_diffusion_module.F90:7-320 and the nodal heat
// system of ns_diffusion_module.F90:7-206, with a constant viscosity or one per
// cell (Sutherland's law, compute_mu, :322-359; caller-given viscosities).
// Parameters, arguments and launchers; the kernels are in diffusion.hip.
#pragma once
#include "device_mesh.hpp"
#include "diff_plan.hpp"
#include "kernels_flux.hpp"
#include "physics.hpp"

namespace sfv {

constexpr int kDiffMaxSub = 64;  // sub-faces (and sub-elements) per vertex at most
// partials per slot with their blocks, one 128-byte line: four groups f = 0..3 of
// four doubles, f = 0 the rhs of rho u, rho v, rho w, E; f = 1..3 column f of the
// 3x3 momentum block, with the heat row's factor behind column 1
constexpr int kDiffSlot = 16;
constexpr int kDiffRow = 4;   // partials per slot of the rhs alone
constexpr int kDiffBlk = 10;  // per cell: the summed momentum block (by column) and heat factor

struct DiffParams {
  double mu, mu0, kap, cv;
  double pr;                  // Prandtl number
  double suth_mu0, suth_T0;   // Sutherland reference viscosity and temperature
  int suth, pad_;             // use_sutherland: mu per cell from mu_cell, mu0corr from mu_min
  int bc_V_id[11], bc_T_id[11];  // 1 neumann, 2 dirichlet, by BC index (1-based)
  double bc_val_V[11][3], bc_val_T[11];
};

// How a mesh's vertices are processed: 32 lanes per vertex, 64, or 64 with the
// inverses left in HBM and formed by a whole workgroup (tetrahedra)
enum DiffClass : int { kDiffHalf = 0, kDiffWave = 1, kDiffLarge = 2 };

struct DiffArgs {
  DevMesh m;
  DiffParams p;
  const uint64_t *doff;    // [V] offset of the vertex's inverses, stored faces << 48, tagged << 56, skewed << 57
  double *pre;             // inverses of the nodal systems
  const double *U;         // [C][5]
  double *PD;              // [SE][kDiffSlot or kDiffRow] node-sorted slot partials
  double *rdiff;           // [C][4]
  double *dblk;            // [C][kDiffBlk]; with a constant viscosity of the mesh only
  const double *mu_cell;   // [C] viscosity of each cell, or null (constant)
  const double *mu_min;    // mu0corr (with mu_cell)
  const uint32_t *scode;   // [SE] node-sorted slot: its sub-element's faces, a byte each (diffusion.hip)
  const double *sivol;     // [SE] node-sorted slot: one over its sub-element's volume
  const uint8_t *fpos;     // [SF] a sub-face's place among its vertex's faces, with boundary flags
  int nim, nfm, nsm;       // largest stored faces, sub-faces and sub-elements of a vertex
  int lmat;                // doubles of LDS for the matrices a vertex forms (set by the launchers)
  int lds_wave;            // doubles of LDS of the apply's fullest wavefront (apply_lds_wave)
  int vper_xcd, vblocks;   // XCD slices of the vertex blocks (apply)
  int cper_xcd, cblocks;   // and of the cell blocks (gather)
  int parts;               // apply: 1 momentum system, 2 heat system, 3 both
  int pivot;               // form the inverses with partial pivoting throughout
  int lds_stride;          // doubles of LDS per vertex, per wavefront in the apply (set by the launchers)
};

// stored faces and tags of every vertex, the faces' places and the slots' codes
void launch_diff_tables(const DevMesh &m, int *vstat, uint8_t *fpos, uint32_t *scode, double *sivol, hipStream_t s);
// constant viscosity, once per mesh and parameters: every vertex's inverses and
// the cells' blocks (a.U: any allocated state)
hipError_t launch_diff_setup(int cls, DiffArgs a, hipStream_t s);
// the slots' terms of the state a.U, and their sums over the cells: rdiff, with
// mu_cell the cells' blocks too
hipError_t launch_diff_terms(int cls, DiffArgs a, hipStream_t s);
hipError_t launch_diff_gather(DiffArgs a, hipStream_t s);
// diag(5, 5, C) from the cells' blocks and the residual's state
hipError_t launch_diff_expand(long C, const double *U, const double *dblk, double cv, double *diag, hipStream_t s);

// temp_u and dtheta_dU (ns_euler_primitives_module.F90:52-63, ns_diffusion_module.F90:196-206)
SFV_DEV double temp_u(const double *u, double cv) {
  const double tau = 1.0 / u[0];
  return (u[4] * tau - 0.5 * (u[1] * u[1] + u[2] * u[2] + u[3] * u[3]) * (tau * tau)) / cv;
}
SFV_DEV void dtheta_du(const double *u, double cv, double *P) {
  const double v1 = u[1] / u[0], v2 = u[2] / u[0], v3 = u[3] / u[0];
  const double nrm = sqrt(v1 * v1 + v2 * v2 + v3 * v3);
  P[0] = (nrm * nrm - u[4] / u[0]) / (u[0] * cv);
  for (int k = 1; k < 4; k++) P[k] = -u[k] / ((u[0] * u[0]) * cv);
  P[4] = 1.0 / (u[0] * cv);
}

// The viscous part of a cell's 5x5 diagonal block (column-major) from its
// summed blocks and the residual's state: momentum block over rho, heat factor
// times dtheta_dU.
SFV_DEV void diff_block(const double *U, const double *blk, double cv, double *D) {
  double u[5], P[5];
  for (int k = 0; k < 5; k++) u[k] = U[k];
  dtheta_du(u, cv, P);
  const double tau = 1.0 / u[0], h = blk[9];
  for (int k = 0; k < 25; k++) D[k] = 0.0;
  for (int j = 0; j < 3; j++)
    for (int i = 0; i < 3; i++) D[1 + i + 5 * (1 + j)] = blk[3 * j + i] * tau;
  for (int k = 0; k < 5; k++) D[4 + 5 * k] = h * P[k];
}

}  // namespace sfv
