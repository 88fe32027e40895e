// kernels.h -- host-side launchers of the gfx950 kernels (implemented in *.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "common.h"
#include "mmo_ff.h"

namespace mmo {

struct InterLaunch {
  int mode;            // MMO_SHIFTED / MMO_GLOBAL
  int k;               // ligand atoms per lane (1, 2, 4, 8)
  int waves;           // wavefronts per block
  int rtile;           // receptor atoms per LDS tile
  int rslice;          // receptor atoms per block row (gridDim.y > 1 splits the receptor)
  int cull;            // culled shifted form: 1 receptor cell list in LDS, 2 in global memory,
                       // 3 positions in LDS; 4 row lists (k_scan_rows), receptor in place,
                       // 5 row lists with the receptor in LDS
  int cull_waves;      // wavefronts per block of the culled kernel
  int cull_k;          // ligand atoms per lane in the culled kernel (1, 2, 4)
  int row_chunk;       // k_scan_rows: receptor atoms fetched at once (4 or 8)
  int row_filter;      // k_scan_rows: far rows' atoms tested against the box first (0 / 1)
  // k_scan_rows: atoms of the scan's ligand; with `part` (n_atoms x 64 x tiles doubles) one
  // of them per wavefront
  int n_atoms;
  double* part;
  CellGrid cg;
  Frame fr;
  const RecPos* rpos;
  const RecAB* rab;
  const RecRes* rres;
  int nrec;
  const LigInfo* ligs;
  const LigAtom* latoms;
  const double* lig_xyz;
};

struct GridDev {
  const float* data;   // ntypes * nvox
  int nx, ny, nz;
  size_t nvox;
  double step, ods;    // step and 1/step
  double ox, oy, oz;   // position of node (0,0,0)
  // nullable: the same values by cell, the 8 corners of cell (i, j, k) (i < nx - 1, ...)
  // contiguous in the trilinear corner order a..h, 32 B per cell and type:
  // cells[((t * (nz-1) + k) * (ny-1) + j) * (nx-1) + i) * 8 + corner]
  const float* cells;
};
hipError_t launch_pack_cells(const GridDev& g, int ntypes, float* cells, hipStream_t s);

struct InterpLaunch {
  GridDev g;
  const LigInfo* ligs;
  const LigAtom* latoms;
  const double* lig_xyz;
};

// interpolated rigid scan over translations X x Y x Z (k_interp_lattice)
struct LatticeArgs {
  const double* rots;          // nrot x 9
  const double* axes;          // the n[0] x, n[1] y and n[2] z values
  int nrot, ntrans, n[3], stride[3];   // translation of (i, j, k) = i stride[0] + ...
  int ztile;                   // z positions of one wavefront, at most
  GridDev g;
  uint32_t grid_bytes;         // of all types' grids together (below 2 GiB)
  const LigInfo* ligs;
  const LigAtom* latoms;
  const double* lig_xyz;
  int lig;
  double* e_out;
};
// z positions of one wavefront, at most: 12 leave 7 wavefronts on a SIMD.  Against the general
// kernel at steps of 0.375, 0.5, 0.75 and 1 A (8 to 40 z, 23 to 131 atoms, mean): 10 2.71, 2.14, 1.92,
// 1.32 times its speed, 12 2.77, 2.17, 1.93, 1.31, 13 2.77, 2.16, 1.91, 1.31, 16 (5 wavefronts)
// 2.67, 2.08, 1.84, 1.26, 20 2.62, 2.02, 1.81, 1.25, 24 (4 wavefronts) 2.81, 2.10, 1.84, 1.25
// Up to 20 (5 wavefronts) instead where that saves tiles, the z are at most 2.25 layers apart, so
// that the two layers read again at each border count, and the wavefronts are at least 20,480 (four
// rounds of the chip) or one round in these tiles (5,120) but more or nearly so in the others
// (6,000 of 7,168): 4,608 rotations of 20^3 at 0.5 A 3.94 -> 3.85 ms; 5,120 to 16,000 rotations of
// 16 x 16 columns, 23 to 131 atoms, 13 z 9 to 24 % less time at 0.375, 0.5 and 0.56 A, 4 to 12 % at 0.75,
// 20 z 0 to 12 % and -5 to 4 %, 28 to 40 z 4 to 16 %; in one round 9 to 29 %.  With other numbers of
// wavefronts the shorter chain counts: 13 to 20 z of 200 rotations take 0.55 to 0.65 times as long in
// two tiles; at 1 A and 3,000 rotations 0.85 to 0.98.
constexpr int kLatticeZ = 12, kLatticeLongZ = 20;
constexpr size_t kLatticeLongUnits = 20480;
// The z axis in as few tiles as that allows, of equal length but for one: tile t's first z and
// their number
__host__ __device__ inline int lattice_tiles(int nz, int ztile) { return (nz + ztile - 1) / ztile; }
__host__ __device__ inline void lattice_tile(int nz, int ztile, int t, int& z0, int& zn) {
  const int tiles = lattice_tiles(nz, ztile), len = nz / tiles, longer = nz - len * tiles;
  z0 = t * len + (t < longer ? t : longer);
  zn = len + (t < longer ? 1 : 0);
}
inline size_t lattice_units(const LatticeArgs& a) {
  return (size_t)a.nrot * (((size_t)a.n[0] * a.n[1] + kWave - 1) / kWave) * lattice_tiles(a.n[2], a.ztile);
}
hipError_t launch_interp_lattice(const LatticeArgs& a, hipStream_t s);

struct IntraArgs {
  const LigInfo* ligs;
  const uint32_t* pair_ij;
  const double4* pair_par;
  const double* xyz;
  const int* atom_off;
  const int* pose_lig;
  int npose;
  int max_atoms;
  double* e_out;
  int e_stride;
  double* grad;
  int grad_accumulate;
};

struct GridArgs {
  Frame fr;
  const RecPos* rpos;
  const RecAB* rab;
  const RecRes* rres;
  int nrec;
  int nx, ny, nz;
  size_t nvox;
  double ox, oy, oz, step;       // node (0,0,0) and spacing, caller frame
  double roi_x, roi_y, roi_z;    // mask: points with |p - roi| < sqrt(roi_r2); roi_r2 <= 0: all
  double roi_r2;
  const double4* probe;          // per type: ke q, A, B
  int ntypes;
  double max_e;                  // clamp (Params.max_E = 1e5, src/params.ml:26)
  float* out;                    // ntypes * nvox, index i + j nx + k nx ny
  int brick0, brick1;   // the launch's bricks
};

struct DofArgs {
  const LigInfo* ligs;
  const double* lig_xyz;        // centred conformers
  const int* rb_left;           // per ligand at rb_base
  const int* rb_right;
  const int* rg_off;            // per ligand at rb_base + lig (nrb+1 entries)
  const int* rg_atoms;
  const int* pose_lig;
  const int* atom_off;
  const int* dof_off;
  int npose, max_atoms;
  int max_rb, max_rg;           // most rbonds and rotation-group atoms of a ligand in the batch
  const double* dofs;
  double* xyz_out;
  double* radius_out;           // nullable
  double* conf;                 // nullable: the posed conformers before the rigid-body motion
                                // (rows), written by apply_config and read by the adjoint
  const double* grad_xyz;       // dE/dxyz (for the adjoint)
  double* gdof;                 // dE/dDOF
  // nullable: the adjoint also evaluates E_intra and its gradient (pair list below) and
  // writes E_intra to e_intra[pose * e_stride]
  double* e_intra;
  int e_stride;
  const uint32_t* pair_ij;
  const double4* pair_par;      // ke qi qj, Ai Aj, 2 Bi Bj
  // the first n_free of `poses` (nullptr: of all, in order) have ligands whose torsions are free
  // (LigHost), of at most max_free_atoms: their adjoint needs no serial pass
  const int* poses;
  int n_free, max_free_atoms;
  const LigAtom* latoms;
  const uint64_t* intra_bits;   // per ligand at bit_base: each atom's pairs (intra_ring)
  const int64_t* bit_base;
  // nullable: the adjoint also sums the poses' units (launch_pose_sum's GRAD form) into
  // e_sum[4 * pose] and clears the rest of the row (E_intra only with clear_intra)
  const double* part;
  const int* unit_off;
  double* e_sum;
  int clear_intra;
};

// part: scratch of (nslices * npose * e_stride) doubles when the receptor is split
hipError_t launch_inter_coords(const InterLaunch& L, const Tile* tiles, const int* perm,
                               int ntiles, int npose, const double* xyz, const int* atom_off,
                               double* e_out, int e_stride, bool comp, double* grad, int write_e,
                               double* part, hipStream_t s);
hipError_t launch_inter_scan(const InterLaunch& L, int lig, const double* rots, int nrot,
                             const double* trans, const int* tperm, int ntrans, double* e_out,
                             hipStream_t s);
hipError_t launch_intra(const IntraArgs& a, bool grad, hipStream_t s);
hipError_t launch_interp_coords(const InterpLaunch& L, const Tile* tiles, const int* perm,
                                int ntiles, const double* xyz, const int* atom_off,
                                const int* type_override, double* e_out, int e_stride,
                                double* grad, int grad_accumulate, hipStream_t s);
hipError_t launch_interp_scan(const InterpLaunch& L, int lig, const double* rots, int nrot,
                              const double* trans, const int* tperm, int ntrans, double* e_out,
                              hipStream_t s);
// filtered scan: score only the listed slots of the scan's pose order (the culled kernel)
hipError_t launch_inter_scan_list(const InterLaunch& L, int lig, const double* rots,
                                  const double* trans, const int* tperm, int ntrans,
                                  const int* list, int nlist, double* e_out, hipStream_t s);
hipError_t launch_interp_scan_list(const InterpLaunch& L, int lig, const double* rots,
                                   const double* trans, const int* tperm, int ntrans,
                                   const int* list, int nlist, double* e_out, hipStream_t s);
// desolvation sums (src/lds.ml:201-267): per listed node v (index i + j nx + k nx ny of
// the grid origin + (i, j, k) step), sum over atoms (x, y, z, q) within 12 A of (q / d^2)^2
struct DesolvArgs {
  const int* vox;             // nodes
  int nvox;
  const double4* atoms;       // x, y, z, q
  int natoms;
  double ox, oy, oz, step;
  int nx, ny;
  double scale;               // nodes: out[v] = scale * sum
  double* out;                // nodes: per grid node
  const double* prot;         // pose: the protein contributions per grid node
  double* part;               // pose: per workgroup (sum, sum of prot[v])
};
// k_desolv_pose writes part[2b], part[2b+1] for workgroup b of kDesolvNodes nodes
constexpr int kDesolvNodes = 256;
hipError_t launch_desolv(const DesolvArgs& a, bool pose, hipStream_t s);
hipError_t launch_fill(double* p, size_t n, double v, hipStream_t s);
hipError_t launch_fill_int(int* p, size_t n, int v, hipStream_t s);
// the bricks (4^3 nodes) of rows kb0 .. kb1 - 1 in z
hipError_t launch_grid(GridArgs a, const CellGrid& cg, bool in_lds, int kb0, int kb1, hipStream_t s);
// one pose per wavefront, shifted form, receptor culled per 8-atom sub-block
struct PoseCullArgs {
  const double* xyz;        // rows (x, y, z), pose-major
  const int* atom_off;
  const int* pose_lig;
  int npose;
  const LigInfo* ligs;
  const LigAtom* latoms;
  double* e_out;            // e_out[pose * e_stride] = E_inter
  int e_stride;
  double* e_comp;           // nullable: [pose*e_stride + 2] elec, [+3] vdW
  double* grad;             // GRAD: dE/dxyz rows (each atom's row is written once)
  int write_e;
  const RecRes* rres;       // receptor quantisation residuals
  // nullable: the pose of each launch slot (slot = workgroup * waves + wavefront), a
  // permutation of 0..npose-1
  const int* order;
};
hipError_t launch_pose_cull(const InterLaunch& L, const PoseCullArgs& a, bool grad, int waves,
                            hipStream_t s);

// shifted form per unit of kUnitAtoms ligand atoms (consecutive in the sweep order)
constexpr int kUnitAtoms = 4;
struct UnitAtom { int row, latom; };   // coordinate row, ligand-atom index; row < 0: none
// the units of a batch, from its poses' ligands: atoms, first ligand atom, place in `sweep`
struct UnitLig { int n_atoms, atom_base, sweep_at; };
hipError_t launch_unit_list(const int* pose_lig, const int* atom_off, const int* unit_off, int npose,
                            const UnitLig* ligs, const int* sweep, UnitAtom* units, hipStream_t s);
struct PoseUnitArgs {
  const double* xyz;        // rows (x, y, z)
  const UnitAtom* units;    // kUnitAtoms per unit, pose-major
  int nunits;
  const LigAtom* latoms;
  const RecRes* rres;
  double* part;             // per unit: E, or with `pairs` (energy form) elec and vdW; nullable (GRAD)
  int pairs;
  double* grad;             // GRAD: each atom's row written once
  int block;                // units a wavefront takes (set by the launch)
};
hipError_t launch_pose_units(const InterLaunch& L, const PoseUnitArgs& a, bool grad, int ncu,
                             hipStream_t s);
// e_out[4p ..] = E_inter, 0, elec, vdW (comp) or E_inter, 0, 0, 0 from the poses' units
// [unit_off[p], unit_off[p + 1]); pairs: part holds (elec, vdW), else E
hipError_t launch_pose_sum(const double* part, const int* unit_off, int npose, bool pairs, bool comp,
                           double* e_out, hipStream_t s);

// LDS a workgroup may hold on gfx950
constexpr size_t kMaxLds = 160 * 1024;
// LDS bytes of one pose of the DOF kernels (coordinates plus the staged torsion tree)
size_t dof_lds_bytes(const DofArgs& a, bool grad);
hipError_t launch_apply_config(const DofArgs& a, hipStream_t s);
hipError_t launch_dof_grad(const DofArgs& a, hipStream_t s);
// total[p] = e[4 p] + e[4 p + 1]; beyond max_radius +inf, and gdof (nullable) 0
hipError_t launch_dof_totals(const double* e, const double* radius, double max_radius,
                             const int* dof_off, int npose, double* gdof, double* total, hipStream_t s);

// -------------------------------------------------- rigid-scan filters, top-k
struct ScanFilterArgs {
  const double* rots;         // nrot x 9
  const double* trans;        // ntrans x 3
  int nrot, ntrans;
  const double* lig;          // centred conformer rows (x, y, z)
  int n_atoms;
  const int* order;           // the order in which its atoms are tested
  const uint32_t* cells;      // protein vdW volume by cell (launch_mask_cells), i + j*nx + k*nx*ny
  double ox, oy, oz, inv_step;
  int nx, ny, nz;
  const uint8_t* skip;        // per translation: 1 = skipped (ROI / centre clash)
  int atom_clash;             // test every atom's 8 corners
  int tiles;                  // scan_keep_tiles (set by the launch)
  double* e;                  // scan energies, set to +inf for skipped poses (all, before scoring)
};
hipError_t launch_scan_filter(const ScanFilterArgs& a, hipStream_t s);
// the bitmask's cells: bit (i, j, k) set when one of the cell's 8 corners is
hipError_t launch_mask_cells(const uint32_t* mask, uint32_t* cells, int nx, int ny, int nz,
                             hipStream_t s);
// Filter before scoring: list[0 .. *total) = the slots of the scan's pose order (rotation r,
// translation tperm[slot - r * ntrans]) that the filters keep, in order; every a.e = +inf.
int scan_keep_tiles(int nrot, int ntrans);       // of 64 slots each: a workgroup's
size_t scan_keep_groups(int nrot, int ntrans);   // workgroups
struct KeepScratch {
  uint64_t* words;            // scan_keep_tiles per workgroup: keep flags
  unsigned* count;            // per workgroup
  unsigned* total;
  int* list;
};
hipError_t launch_scan_keep(const ScanFilterArgs& a, const int* tperm, const KeepScratch& w,
                            hipStream_t s);

constexpr int kTopkMax = 2048;
constexpr int kTopkCand = 4096;   // keys the select leaves to the final sort, at most (>= kTopkMax)
constexpr int kTopkPasses = 5;       // digits of the select
constexpr int kTopkHist = kTopkPasses * 8192;
struct TopkState {
  uint64_t prefix, mask;      // the selected high bits and which they are
  uint64_t rem, k;            // keys still to be taken among those matching the prefix; of k
  unsigned limit;             // candidates to end at (topk_limit)
  unsigned done;              // no more keys than that are at or below the prefix
};
struct TopkScratch {
  TopkState* st;              // kTopkPasses + 1
  unsigned* count;            // candidates gathered
  unsigned* hist;             // kTopkHist: the counts of each pass
  unsigned* bcnt;             // one per chunk
  double* cand_e;             // kTopkCand
  int64_t* cand_i;            // kTopkCand
  size_t chunk;
};
hipError_t launch_topk(const double* e, size_t n, int k, double* out_e, int64_t* out_i,
                       TopkScratch w, hipStream_t s);

// ------------------------------------------------------------ L-BFGS minimiser
constexpr int kMinMaxHist = 16;
enum { kMinRunning = 0, kMinConverged = 1, kMinFailed = 2 };
struct MinPose {
  double f, f0, alpha, gamma;   // energy at x, at the start, step length, H0 scale
  int init, hist, head, status;
  int n_eval, n_acc, n_reset, pad;
};
struct MinArgs {
  int npose, m, ndof_total;
  const int* dof_off;
  double* x;            // accepted point (the best point)
  double* g;            // gradient at x
  double* d;            // search direction
  double* xt;           // trial point: the input of the next evaluation
  const double* gt;     // gradient at the trial point
  const double* et;     // energies at the trial point (npose x 4: inter, intra, ...)
  const double* rad;    // enclosing radius after the torsions
  double* S;            // history (m x ndof_total)
  double* Y;
  double* rho;          // m x npose
  MinPose* st;
  const double* lo;     // box bounds (ndof_total) or null
  const double* hi;
  double max_step, min_step, gtol, c1;
};
hipError_t launch_lbfgs(const MinArgs& a, hipStream_t s);

// energy forms of the DOF evaluator (dofmin.h; the Monte Carlo kernel's numbering)
enum { kDofInterGrid = 0, kDofInterAtom = 1, kDofInterF64 = 3 };

// The whole minimisation of a batch in one persistent launch: each wavefront takes poses
// from a queue and runs all iterations of one pose (evaluation and update) without
// leaving the kernel.  inter: kDofInterAtom (shifted, FP32 per-atom sweep), kDofInterF64
// or kDofInterGrid (dofmin.h); the batch's DOF vectors apply to the registered conformers.
struct MinPersistArgs {
  const LigInfo* ligs;
  const LigAtom* latoms;
  const double* lig_xyz;        // registered centred conformers (the base of every pose)
  const int* atom_order;
  const int* rb_left;
  const int* rb_right;
  const int* rg_off;
  const int* rg_atoms;
  const uint32_t* pair_ij;
  const double4* pair_par;
  int npose, max_atoms, max_rb, max_rg, ndof_total, iters, m;
  const int* pose_lig;
  const int* dof_off;
  const int* order;             // nullable: queue position -> pose (largest ligands first)
  double* x;                    // DOF vectors: start in, best point out
  const double* lo;             // box bounds (ndof_total) or null
  const double* hi;
  double* S;                    // history: S[slot * ndof_total + dof], rho[slot * npose + pose]
  double* Y;
  double* rho;
  MinPose* st;
  double* e_out;                // nullable: best energy per pose
  int* queue;
  int slots;                    // pooled form: poses per workgroup and their units' energies,
  float4* fe;                   // 64 per unit of 4 atoms, min_units(max_atoms) a slot
  int intra;
  double max_step, min_step, gtol, c1;
  Frame fr;
  const RecPos* rpos;
  const RecAB* rab;
  const RecRes* rres;
  int nrec;
  CellGrid cg;
  GridDev g;
};
size_t min_persist_lds_bytes(const MinPersistArgs& a, int waves, bool rec_lds);
// sweep units of a pose of n atoms (dof_sweep_unit)
__host__ __device__ inline int min_units(int n) { return (n + 3) / 4; }
// poses a workgroup of the pooled form may hold, and its LDS with `slots` of them
constexpr int kMinSlots = 8;
size_t min_pooled_lds_bytes(const MinPersistArgs& a);
hipError_t launch_min_pooled(const MinPersistArgs& a, int nblocks, hipStream_t s);
hipError_t launch_min_persist(const MinPersistArgs& a, int inter, int nblocks, int waves,
                              bool rec_lds, hipStream_t s);
hipError_t launch_min_reset(MinPose* st, int npose, hipStream_t s);
hipError_t launch_min_energy(const MinPose* st, int npose, double* e_out, hipStream_t s);

}  // namespace mmo
