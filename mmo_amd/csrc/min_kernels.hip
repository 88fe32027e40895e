// min_kernels.hip -- batched L-BFGS over DOF vectors, one wavefront per pose.
//
// The reference minimises E_intra + E_inter over the DOF vector
// [x, y, z, alpha, beta, gamma, tau_0..] of Optim.apply_config with NLopt inside box
// bounds (ROI cube for the position, [-pi, pi] for angles), with gradients from
// central differences (Lds.minimize_ligand / nlopt_minimize / approx_local_gradient,
// src/lds.ml:1014-1036, :1118-1297, src/optim.ml:34-80).  Here every pose of a batch
// runs limited-memory BFGS on the analytic adjoint gradient:
//
//   iteration = one energy + gradient evaluation of every pose's trial point (the
//   batched DOF kernels) followed by k_lbfgs, which per pose either accepts the trial
//   (Armijo sufficient decrease), updates the (s, y) history and computes the next
//   direction with the two-loop recursion, or halves the step (backtracking);
//   trial points are projected onto the box bounds.  Poses whose torsions make the
//   ligand longer than 12 A (Mol.Too_long, src/optim.ml:75) or whose energy is not
//   finite count as failed trials.
//
// Lanes hold the DOF components (at most 64 per pose); dot products are wavefront
// reductions in FP64.
#include "common.h"
#include "dofmin.h"
#include "kernels.h"

namespace mmo {

__global__ void __launch_bounds__(256) k_lbfgs(MinArgs a) {
  const int lane = threadIdx.x & (kWave - 1);
  const int p = blockIdx.x * (blockDim.x / kWave) + (threadIdx.x / kWave);
  if (p >= a.npose) return;
  MinPose s = a.st[p];
  if (s.status != kMinRunning) return;
  const int o = a.dof_off[p];
  const int n = a.dof_off[p + 1] - o;
  const bool act = lane < n;
  const size_t i = (size_t)o + (act ? lane : 0);
  const double ft = a.et[4 * (size_t)p] + a.et[4 * (size_t)p + 1];
  const double gti = act ? a.gt[i] : 0.0;
  const double xti = act ? a.xt[i] : 0.0;
  const double lo = (act && a.lo) ? a.lo[i] : -__builtin_inf();
  const double hi = (act && a.hi) ? a.hi[i] : __builtin_inf();
  double x = 0.0, g = 0.0, d = 0.0;
  if (s.init && act) {
    x = a.x[i];
    g = a.g[i];
    d = a.d[i];
  }
  const MinCfg cfg{a.m, a.max_step, a.min_step, a.gtol, a.c1};
  const double xn = lbfgs_wave(s, x, g, d, xti, ft, gti, a.rad[p], lo, hi, act, a.S + i,
                               a.Y + i, (size_t)a.ndof_total, a.rho + p, (size_t)a.npose, cfg);
  if (act) {
    a.x[i] = x;
    a.g[i] = g;
    a.d[i] = d;
    a.xt[i] = xn;
  }
  if (lane == 0) a.st[p] = s;
}

// best energies out (the accepted point is the best point: accepted steps decrease E)
__global__ void k_min_energy(const MinPose* st, int npose, double* e_out) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < npose) e_out[p] = st[p].f;
}

__global__ void k_min_reset(MinPose* st, int npose) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < npose) {
    MinPose z{};
    st[p] = z;
  }
}

// ---------------------------------------------------------- persistent minimiser
// LDS per wavefront: the conformer and the adjoint (6 x max_atoms FP64) and the
// atom-sweep scratch; before them, with REC_LDS, the receptor and its cell table.
__host__ __device__ inline size_t min_wave_lds_bytes(int max_atoms) {
  return ((size_t)6 * max_atoms * sizeof(double) + kAtomSweepInts * sizeof(int) + 15) & ~(size_t)15;
}

constexpr int kMinPersistWaves = 16;
// Wavefronts per workgroup each form is compiled for.  With the receptor in LDS at most
// 8-9 wavefronts fit in a workgroup's LDS anyway, so that form is compiled for 8 (up to
// 256 VGPRs, 2 wavefronts per SIMD): at 16 (128 VGPRs) it spilled 236 B per lane.
__host__ __device__ constexpr int min_persist_waves(bool rec_lds) {
  return rec_lds ? 8 : kMinPersistWaves;
}

template <bool REC_LDS, int INTER>
__global__ void __launch_bounds__(min_persist_waves(REC_LDS) * 64) k_min_persist(MinPersistArgs a) {
  extern __shared__ __align__(16) char smem[];
  const RecPos* s_pos;
  const RecAB* s_ab;
  const int* s_cell;
  load_receptor<REC_LDS>(a.rpos, a.rab, a.nrec, a.cg, s_pos, s_ab, s_cell, smem);
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x / kWave;
  char* mine = smem + receptor_lds_bytes<REC_LDS>(a.nrec, a.cg) + wv * min_wave_lds_bytes(a.max_atoms);
  double* tx = reinterpret_cast<double*>(mine);
  double* ty = tx + a.max_atoms;
  double* tz = ty + a.max_atoms;
  double* hx = tz + a.max_atoms;
  double* hy = hx + a.max_atoms;
  double* hz = hy + a.max_atoms;
  int* wl = reinterpret_cast<int*>(hz + a.max_atoms);
  const MinCfg cfg{a.m, a.max_step, a.min_step, a.gtol, a.c1};
  for (;;) {
    // the next pose: lane 0 takes it from the queue, readlane makes it a scalar, so the
    // loop exit is uniform (with a vector broadcast the compiler treats the exit as
    // divergent and may send the other lanes round the loop without lane 0's atomic)
    int qv = 0;
    if (lane == 0) qv = atomicAdd(a.queue, 1);
    const int q = __builtin_amdgcn_readlane(qv, 0);
    if (q >= a.npose) break;
    const int p = a.order ? a.order[q] : q;
    const LigInfo li = a.ligs[a.pose_lig[p]];
    const int o = a.dof_off[p];
    const int n = a.dof_off[p + 1] - o;
    const bool act = lane < n;
    const size_t i = (size_t)o + (act ? lane : 0);
    DofEval ev;
    ev.li = li; ev.latoms = a.latoms; ev.atom_order = a.atom_order; ev.rb_left = a.rb_left;
    ev.rb_right = a.rb_right; ev.rg_off = a.rg_off; ev.rg_atoms = a.rg_atoms;
    ev.pair_ij = a.pair_ij; ev.pair_par = a.pair_par; ev.ntors = n - 6; ev.intra = a.intra != 0;
    ev.fr = a.fr; ev.s_pos = s_pos; ev.s_ab = s_ab; ev.s_cell = s_cell; ev.rres = a.rres;
    ev.cg = a.cg; ev.wl = wl; ev.g = a.g;
    const double* base = a.lig_xyz + 3 * (size_t)li.atom_base;
    const double lo = (act && a.lo) ? a.lo[i] : -__builtin_inf();
    const double hi = (act && a.hi) ? a.hi[i] : __builtin_inf();
    MinPose s{};
    double xt = act ? a.x[i] : 0.0, x = 0.0, g = 0.0, d = 0.0;
    for (int it = 0; it < a.iters && __builtin_amdgcn_readfirstlane(s.status) == kMinRunning; ++it) {
      double gt, ei, ea, rad;
      const double f = dof_eval<INTER>(ev, base, xt, tx, ty, tz, hx, hy, hz, gt, ei, ea, rad);
      xt = lbfgs_wave(s, x, g, d, xt, f, act ? gt : 0.0, rad, lo, hi, act, a.S + i, a.Y + i,
                      (size_t)a.ndof_total, a.rho + p, (size_t)a.npose, cfg);
    }
    if (a.iters > 0) {
      if (act) a.x[i] = x;
      if (lane == 0) {
        a.st[p] = s;
        if (a.e_out) a.e_out[p] = s.f;
      }
    }
    // all lanes meet here before the next pose (a convergent point: without it the
    // compiler joins this lane-0 block to the next queue fetch, and the other lanes
    // would start the next pose without lane 0)
    wave_lds_sync();
  }
}

// ------------------------------------------------------------------- pooled form
// Few poses per CU leave k_min_persist waiting: a pose is one wavefront's chain of
// evaluations (1,000 poses: 125 workgroups of 8, and 21 ms however many there are, the time
// of the largest ligand).  Here a workgroup keeps `slots` poses, one wavefront each, and all
// its wavefronts share the receptor sweeps of these poses, a unit of 4 atoms at a time, as
// they become free; the units leave FP32 energies per lane in memory for the pose's
// wavefront to add up in its atoms' order, so every sum has k_min_persist's bits.  Sweeps and
// the rest alternate between workgroup barriers.
// 100 iterations, ligands of 26 to 94 atoms, 3,000-atom receptor: 64 poses 16.3 -> 8.4 ms,
// 500 21.4 -> 9.5, 1,000 21.4 -> 11.5, 1,500 22.3 -> 13.4, 2,000 22.0 -> 17.0 (4 slots, the
// other half from the queue).  Of an evaluation's 260,000 cycles at 1,000 poses E_intra's
// chain of FP64 LDS additions takes 95,000, the sweeps 94,000, the torsions and their adjoint
// 43,000.  The additions as reads and writes of one diagonal at a time took 199,000.
constexpr int kMinPooledWaves = 8;

// per slot: the atoms' parameters and order, the conformer and the adjoint (FP64), the rigid
// motion, the torsions (rg_off relative to the pose); then the wavefronts' sweep scratch
__host__ __device__ inline size_t min_slot_lds_bytes(int max_atoms, int max_rb, int max_rg) {
  return ((size_t)max_atoms * (6 * sizeof(double) + sizeof(float4)) + 12 * sizeof(double) +
          (3 * (size_t)max_rb + 1 + max_rg) * sizeof(int) + 15) & ~(size_t)15;
}

__global__ void __launch_bounds__(kMinPooledWaves * 64) k_min_pooled(MinPersistArgs a) {
  extern __shared__ __align__(16) char smem[];
  __shared__ int s_atoms[kMinSlots];   // atoms to sweep (0: none), kept until the next round
  __shared__ int s_live[kMinSlots];    // the slot holds a pose
  __shared__ int s_next;               // the next unit of this round
  const RecPos* s_pos;
  const RecAB* s_ab;
  const int* s_cell;
  load_receptor<true>(a.rpos, a.rab, a.nrec, a.cg, s_pos, s_ab, s_cell, smem);
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  char* slots = smem + receptor_lds_bytes<true>(a.nrec, a.cg);
  const size_t slot_bytes = min_slot_lds_bytes(a.max_atoms, a.max_rb, a.max_rg);
  const size_t units = min_units(a.max_atoms);
  float4* fe = a.fe + (size_t)blockIdx.x * a.slots * units * kWave;
  auto slot_at = [&](int s) { return reinterpret_cast<float4*>(slots + s * slot_bytes); };
  auto slot_xyz = [&](int s) { return reinterpret_cast<double*>(slot_at(s) + a.max_atoms); };
  auto slot_rt = [&](int s) { return slot_xyz(s) + 6 * (size_t)a.max_atoms; };
  const MinCfg cfg{a.m, a.max_step, a.min_step, a.gtol, a.c1};
  DofEval ev;
  ev.latoms = a.latoms; ev.atom_order = a.atom_order;
  ev.pair_ij = a.pair_ij; ev.pair_par = a.pair_par; ev.intra = a.intra != 0;
  ev.fr = a.fr; ev.s_pos = s_pos; ev.s_ab = s_ab; ev.s_cell = s_cell; ev.rres = a.rres; ev.cg = a.cg;
  ev.wl = reinterpret_cast<int*>(slots + a.slots * slot_bytes) + wv * kAtomSweepInts;
  // wavefront w < slots keeps slot w's pose: its DOFs in the lanes, as in k_min_persist
  const bool keeper = wv < a.slots;
  float4* at = slot_at(keeper ? wv : 0);
  double* tx = slot_xyz(keeper ? wv : 0);
  double *ty = tx + a.max_atoms, *tz = ty + a.max_atoms;
  double *hx = tz + a.max_atoms, *hy = hx + a.max_atoms, *hz = hy + a.max_atoms;
  int* const rb_left = reinterpret_cast<int*>(slot_rt(keeper ? wv : 0) + 12);
  int* const rb_right = rb_left + a.max_rb;
  int* const rg_off = rb_right + a.max_rb;
  int* const rg_atoms = rg_off + a.max_rb + 1;
  ev.rb_left = rb_left; ev.rb_right = rb_right; ev.rg_off = rg_off; ev.rg_atoms = rg_atoms;
  // a pose per slot dealt by size, to and fro over the workgroups; then from the queue
  const int nb = gridDim.x, b = blockIdx.x;
  int q = keeper ? wv * nb + ((wv & 1) ? nb - 1 - b : b) : a.npose;
  bool live = false;
  int p = 0, it = 0;
  size_t i = 0;
  bool act = false;
  double lo = 0.0, hi = 0.0, xt = 0.0, x = 0.0, g = 0.0, d = 0.0;
  const double* base = nullptr;
  MinPose s{};
  for (;;) {
    double M[9], T[3], sn = 0.0, cs = 0.0, rad = 0.0;
    if (keeper) {
      if (!live && q < a.npose) {
        live = true;
        p = a.order ? a.order[q] : q;
        ev.li = a.ligs[a.pose_lig[p]];
        const int o = a.dof_off[p];
        const int n = a.dof_off[p + 1] - o;
        ev.ntors = n - 6;
        act = lane < n;
        i = (size_t)o + (act ? lane : 0);
        base = a.lig_xyz + 3 * (size_t)ev.li.atom_base;
        lo = (act && a.lo) ? a.lo[i] : -__builtin_inf();
        hi = (act && a.hi) ? a.hi[i] : __builtin_inf();
        s = MinPose{};
        xt = act ? a.x[i] : 0.0;
        x = g = d = 0.0;
        it = 0;
        for (int j = lane; j < ev.li.n_atoms; j += kWave) {
          const int ja = a.atom_order ? a.atom_order[ev.li.atom_base + j] : j;
          const LigAtom la = a.latoms[ev.li.atom_base + ja];
          at[j] = make_float4((float)la.keq, (float)la.a, (float)la.b, __int_as_float(ja));
        }
        const int* off = a.rg_off + ev.li.rg_base;
        const int g0 = off[0], ng = off[ev.ntors] - g0;
        if (lane < ev.ntors) {
          rb_left[lane] = a.rb_left[ev.li.rb_base + lane];
          rb_right[lane] = a.rb_right[ev.li.rb_base + lane];
        }
        if (lane <= ev.ntors) rg_off[lane] = off[lane] - g0;
        for (int m = lane; m < ng; m += kWave) rg_atoms[m] = a.rg_atoms[g0 + m];
        ev.li.rb_base = ev.li.rg_base = 0;   // the staged torsions
        wave_lds_sync();
      }
      if (live) {
        rad = dof_pose(ev, base, xt, tx, ty, tz, M, nullptr, nullptr, nullptr, T, sn, cs);
        double* rt = slot_rt(wv);
        if (lane == 0) {
          for (int k = 0; k < 9; ++k) rt[k] = M[k];
          for (int k = 0; k < 3; ++k) rt[9 + k] = T[k];
        }
      }
      if (lane == 0) {
        s_live[wv] = live;
        s_atoms[wv] = live && rad <= 12.0 ? ev.li.n_atoms : 0;   // Mol.Too_long
      }
    }
    if (threadIdx.x == 0) s_next = 0;
    __syncthreads();
    bool any = false;
    for (int k = 0; k < a.slots; ++k) any |= s_live[k] != 0;
    if (!__builtin_amdgcn_readfirstlane((int)any)) break;   // the same for all wavefronts
    for (;;) {
      int u = 0;
      if (lane == 0) u = atomicAdd(&s_next, 1);
      u = __builtin_amdgcn_readlane(u, 0);
      int sl = 0, n = 0;
      for (; sl < a.slots; ++sl) {
        n = __builtin_amdgcn_readfirstlane(s_atoms[sl]);
        if (u < min_units(n)) break;
        u -= min_units(n);
      }
      if (sl == a.slots) break;
      const double* rt = slot_rt(sl);
      double* sx = slot_xyz(sl);
      const int A = a.max_atoms;
      auto posed = [&](int j, double& x0, double& y0, double& z0) {
        const double c0 = sx[j], c1 = sx[A + j], c2 = sx[2 * A + j];
        x0 = (rt[0] * c0 + rt[1] * c1 + rt[2] * c2) + rt[9];
        y0 = (rt[3] * c0 + rt[4] * c1 + rt[5] * c2) + rt[10];
        z0 = (rt[6] * c0 + rt[7] * c1 + rt[8] * c2) + rt[11];
      };
      dof_sweep_unit(ev, n, u, posed, slot_at(sl), sx + 3 * A, sx + 4 * A, sx + 5 * A,
                     fe + ((size_t)sl * units + u) * kWave);
    }
    __syncthreads();
    if (live) {
      double gt = 0.0, f = __builtin_inf();
      if (rad <= 12.0) {
        double e = 0.0;   // per lane, in the order of the atoms (as atom_sweep adds them)
        const int L = ev.li.n_atoms;
        const float4* mine = fe + (size_t)wv * units * kWave + lane;
        constexpr int kAhead = 8;   // loads in flight
        for (int u0 = 0; u0 < min_units(L); u0 += kAhead) {
          float4 v[kAhead];
#pragma unroll
          for (int k = 0; k < kAhead; ++k)
            if (u0 + k < min_units(L)) v[k] = mine[(size_t)(u0 + k) * kWave];
#pragma unroll
          for (int k = 0; k < kAhead; ++k) {
            const int j = 4 * (u0 + k);
            if (j < L) e += (double)v[k].x;
            if (j + 1 < L) e += (double)v[k].y;
            if (j + 2 < L) e += (double)v[k].z;
            if (j + 3 < L) e += (double)v[k].w;
          }
        }
        const double e_inter = wave_sum(e);
        const double e_intra = dof_adjoint(ev, M, sn, cs, tx, ty, tz, hx, hy, hz, gt);
        f = e_inter + e_intra;
      }
      xt = lbfgs_wave(s, x, g, d, xt, f, act ? gt : 0.0, rad, lo, hi, act, a.S + i, a.Y + i,
                      (size_t)a.ndof_total, a.rho + p, (size_t)a.npose, cfg);
      ++it;
      if (it >= a.iters || __builtin_amdgcn_readfirstlane(s.status) != kMinRunning) {
        if (act) a.x[i] = x;
        int qv = 0;
        if (lane == 0) {
          a.st[p] = s;
          if (a.e_out) a.e_out[p] = s.f;
          qv = atomicAdd(a.queue, 1);
        }
        wave_lds_sync();   // all lanes meet here
        q = a.slots * nb + __builtin_amdgcn_readlane(qv, 0);
        live = false;
      }
    }
  }
}

size_t min_pooled_lds_bytes(const MinPersistArgs& a) {
  return receptor_lds_bytes<true>(a.nrec, a.cg) + a.slots * min_slot_lds_bytes(a.max_atoms, a.max_rb, a.max_rg) +
         kMinPooledWaves * kAtomSweepInts * sizeof(int);
}

hipError_t launch_min_pooled(const MinPersistArgs& a, int nblocks, hipStream_t s) {
  if (a.npose == 0) return hipSuccess;
  const size_t lds = min_pooled_lds_bytes(a);
  if (a.slots < 1 || a.slots > kMinSlots || a.slots > kMinPooledWaves || lds > kMaxLds)
    return hipErrorInvalidValue;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_min_pooled),
                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)(kMaxLds - 128));
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_min_pooled, dim3(nblocks), dim3(kMinPooledWaves * kWave), lds, s, a);
  return hipGetLastError();
}

size_t min_persist_lds_bytes(const MinPersistArgs& a, int waves, bool rec_lds) {
  return (rec_lds ? receptor_lds_bytes<true>(a.nrec, a.cg) : 0) +
         (size_t)waves * min_wave_lds_bytes(a.max_atoms);
}

template <bool R, int I>
static hipError_t min_persist_go(const MinPersistArgs& a, int nblocks, int waves, hipStream_t s) {
  const size_t lds = min_persist_lds_bytes(a, waves, R);
  if (lds > kMaxLds) return hipErrorInvalidConfiguration;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_min_persist<R, I>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_min_persist<R, I>), dim3(nblocks), dim3(waves * kWave), lds, s, a);
  return hipGetLastError();
}

hipError_t launch_min_persist(const MinPersistArgs& a, int inter, int nblocks, int waves,
                              bool rec_lds, hipStream_t s) {
  if (a.npose == 0) return hipSuccess;
  if (waves < 1 || waves > min_persist_waves(rec_lds)) return hipErrorInvalidValue;
  switch (inter + (rec_lds ? 8 : 0)) {
    case kDofInterAtom + 8: return min_persist_go<true, kDofInterAtom>(a, nblocks, waves, s);
    case kDofInterF64 + 8: return min_persist_go<true, kDofInterF64>(a, nblocks, waves, s);
    case kDofInterAtom: return min_persist_go<false, kDofInterAtom>(a, nblocks, waves, s);
    case kDofInterF64: return min_persist_go<false, kDofInterF64>(a, nblocks, waves, s);
    case kDofInterGrid: return min_persist_go<false, kDofInterGrid>(a, nblocks, waves, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_lbfgs(const MinArgs& a, hipStream_t s) {
  if (a.npose == 0) return hipSuccess;
  constexpr int kWaves = 4;
  hipLaunchKernelGGL(k_lbfgs, dim3((a.npose + kWaves - 1) / kWaves), dim3(kWaves * kWave), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_min_reset(MinPose* st, int npose, hipStream_t s) {
  if (npose == 0) return hipSuccess;
  hipLaunchKernelGGL(k_min_reset, dim3((npose + 255) / 256), dim3(256), 0, s, st, npose);
  return hipGetLastError();
}

hipError_t launch_min_energy(const MinPose* st, int npose, double* e_out, hipStream_t s) {
  if (npose == 0) return hipSuccess;
  hipLaunchKernelGGL(k_min_energy, dim3((npose + 255) / 256), dim3(256), 0, s, st, npose, e_out);
  return hipGetLastError();
}

}  // namespace mmo
