// mc_kernels.hip -- batched Monte Carlo chains on gfx950, one wavefront per chain.
//
// Restates Lds.simulate_lig (src/lds.ml:741-1000) for many ligands and chains in one
// persistent launch: wavefronts take chains from a work queue (most expensive first)
// and advance each by `nsteps` frames; the chain state lives in HBM between launches,
// so a launch (or a hipGraph replay of it) continues where the last one stopped.
//
// Per frame (src/lds.ml:882-995):
//   even frames: rigid move, rot' = R_axis(theta) rot (Move.rand_rot src/move.ml:20-31,
//     passive axis matrices src/rot.ml:22-46), pos' = pos + dt U(-1,1)^3 (src/move.ml:46-54);
//   odd frames: torsion move of the conformer (turned in place, the moved atoms restored
//     from the chain's undo rows unless the move is kept), tweak U(-dr_i, dr_i) or, every
//     100th conformer step, flip U(-pi, pi) (src/lds.ml:781-798, src/mol.ml:635-647);
//     enclosing radius > 12 A (Mol.check_elongation_exn) ends the chain (the exception
//     leaves the frame loop, src/lds.ml:996-998);
//   pose x = rot' (conf' - centre(conf')) + pos' (src/mol.ml:705-710);
//   E_intra (odd frames) and E_inter are stored before the acceptance test
//   (src/lds.ml:900-904);
//   hard ROI: a pose centre beyond the ROI radius resets the chain; otherwise
//   E_inter == 0 resets it and Metropolis at beta = 1/(kB T) decides (src/lds.ml:906-954).
//   OCaml attaches the `else` of src/lds.ml:917 to the inner `if dist_roi > out_radius`,
//   so without hard ROI no move is ever accepted; MMO_MC_METROPOLIS_ALWAYS runs the
//   E == 0 / Metropolis branch in that case as well (not the reference's behaviour).
//   Best pose, adaptive steps (x0.95 / x1.05 outside the [0.45, 0.55] acceptance band
//   over 100-event windows, src/lds.ml:586-621, :971-988).
// Random numbers: Philox4x32-10 keyed by the seed, counter (chain, frame, draw).
#include "common.h"
#include "cull.h"
#include "dofmin.h"
#include "kernels.h"
#include "mc.h"

namespace mmo {

// the chains' atom sweep fetches its ligand atoms 64 at a time (one per lane) and
// broadcasts them, rather than one dependent fetch per atom
constexpr bool kMcPreload = true;
// ligand atoms per pass of the chains' per-atom sweep
constexpr int kMcSweepAtoms = 4;

// ------------------------------------------------------------------ Philox4x32-10
// Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as easy as 1, 2, 3" (SC 2011).
__device__ __forceinline__ uint4 philox(uint4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint32_t hi0 = __umulhi(0xD2511F53u, c.x), lo0 = 0xD2511F53u * c.x;
    const uint32_t hi1 = __umulhi(0xCD9E8D57u, c.z), lo1 = 0xCD9E8D57u * c.z;
    c = make_uint4(hi1 ^ c.y ^ k0, lo1, hi0 ^ c.w ^ k1, lo0);
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return c;
}
// two uniform doubles in [0, 1) with 53 random bits each
__device__ __forceinline__ void uniform2(uint4 r, double& a, double& b) {
  a = ((double)(r.x >> 5) * 67108864.0 + (double)(r.y >> 6)) * (1.0 / 9007199254740992.0);
  b = ((double)(r.z >> 5) * 67108864.0 + (double)(r.w >> 6)) * (1.0 / 9007199254740992.0);
}

// ------------------------------------------------------------------ sliding window
// SW.t (src/SW.ml:7-42): last 100 accept/reject events; ratio = accepts / events.
__device__ __forceinline__ void sw_process(SwState& w, bool ev) {
  const int word = w.head >> 5, bit = w.head & 31;
  if (w.count == kMcBlock) {
    if ((w.bits[word] >> bit) & 1u) --w.acc;
  } else {
    ++w.count;
  }
  if (ev) { w.bits[word] |= 1u << bit; ++w.acc; }
  else w.bits[word] &= ~(1u << bit);
  w.head = (w.head + 1 == kMcBlock) ? 0 : w.head + 1;
}
__device__ __forceinline__ double sw_ratio(const SwState& w) {
  return (double)w.acc / (double)w.count;   // 0/0 = NaN: no adaptation (comparisons false)
}
__device__ __forceinline__ void sw_reset(SwState& w) {
  w.bits[0] = w.bits[1] = w.bits[2] = w.bits[3] = 0u;
  w.head = w.count = w.acc = 0;
}

// --------------------------------------------------------------- energies of a pose
// The pose being scored (rotation, conformer centre, position) and the frame's Metropolis
// uniform, in the chain's LDS slot: the energy sweeps read it from there, so none of it
// is held in registers (and spilled to scratch) while a sweep runs.
struct McPose {
  double m[9], c[3], p[3], u;
};
static_assert(sizeof(McPose) % 16 == 0, "McPose slots keep 16-byte alignment");

// pose atom j: rot (conf_j - centre) + pos
struct PoseView {
  const double* sx;
  const double* sy;
  const double* sz;
  const McPose* q;
  __device__ void at(int j, double& x, double& y, double& z) const {
    const double a = sx[j] - q->c[0], b = sy[j] - q->c[1], c = sz[j] - q->c[2];
    x = (q->m[0] * a + q->m[1] * b + q->m[2] * c) + q->p[0];
    y = (q->m[3] * a + q->m[4] * b + q->m[5] * c) + q->p[1];
    z = (q->m[6] * a + q->m[7] * b + q->m[8] * c) + q->p[2];
  }
};

__device__ double mc_inter_interp(const McArgs& a, const LigInfo& li, const PoseView& v) {
  const int lane = threadIdx.x & (kWave - 1);
  double e = 0.0;
  int bad = 0;
  const GridDev& g = a.g;
  for (int j = lane; j < li.n_atoms; j += kWave) {
    double x, y, z;
    v.at(j, x, y, z);
    const double px = x - g.ox, py = y - g.oy, pz = z - g.oz;
    const double fx = px * g.ods, fy = py * g.ods, fz = pz * g.ods;
    if (!(px >= 0.0 && py >= 0.0 && pz >= 0.0 && fx < (double)(g.nx - 1) &&
          fy < (double)(g.ny - 1) && fz < (double)(g.nz - 1))) {
      bad = 1;
      continue;
    }
    const int i0 = (int)fx, j0 = (int)fy, k0 = (int)fz;
    float cv[8];
    grid_corners(g, a.latoms[li.atom_base + j].type, i0, j0, k0, cv);
    const double wlx = (px - i0 * g.step) * g.ods, wly = (py - j0 * g.step) * g.ods,
                 wlz = (pz - k0 * g.step) * g.ods;
    const double whx = 1.0 - wlx, why = 1.0 - wly, whz = 1.0 - wlz;
    // corner order of G3D.trilin, src/G3D.ml:144-151
    e += (double)cv[0] * (whx * why * whz) + (double)cv[1] * (wlx * why * whz) +
         (double)cv[2] * (wlx * wly * whz) + (double)cv[3] * (whx * wly * whz) +
         (double)cv[4] * (whx * why * wlz) + (double)cv[5] * (wlx * why * wlz) +
         (double)cv[6] * (wlx * wly * wlz) + (double)cv[7] * (whx * wly * wlz);
  }
  e = wave_sum(e);
  return __ballot(bad) != 0ull ? __builtin_nan("") : e;
}

// shifted direct sum of the pose: FP32 pairs swept per 8-atom sub-block (pose_sweep);
// the FP64 parity mode sweeps with FP64 pair arithmetic, two atoms per lane
// INTER: kMcInterAtom / kMcInterSub (FP32, atom_sweep / pose_sweep) or kMcInterF64
template <int INTER>
__device__ double mc_inter_direct(const McArgs& a, const LigInfo& li, const PoseView& v,
                                  const RecPos* s_pos, const RecAB* s_ab, const int* s_cell,
                                  int* wl) {
  const Frame fr = a.fr;
  int sat = 0;
  if (INTER != kMcInterF64) {
    double e_el = 0.0, e_vd = 0.0;
    auto atom = [&](int j, LigPt& l, double& cq, double& ca, double& cb) {
      // sweep position j -> ligand atom (the per-atom sweep's order, if given)
      const int ja = (INTER == kMcInterAtom && a.atom_order) ? a.atom_order[li.atom_base + j] : j;
      double x, y, z;
      v.at(ja, x, y, z);
      l = lig_pt(x, y, z, fr, &sat);
      const LigAtom la = a.latoms[li.atom_base + ja];
      cq = la.keq; ca = la.a; cb = la.b;
    };
    auto none = [](int, double, double, double) {};
    if (INTER == kMcInterAtom)
      // pairs closer than 0.5 A add both atoms' quantisation residuals (without them a
      // clashing pose's energy, above 1e7 kcal/mol, is off by up to ~2e-5 relative)
      atom_sweep<false, decltype(atom)&, decltype(none)&, true, kMcPreload, kMcSweepAtoms>(
          a.cg, s_cell, s_pos, s_ab, a.rres, fr, li.n_atoms, wl, atom, none, e_el, e_vd);
    else
      pose_sweep<false>(a.cg, s_cell, s_pos, s_ab, a.rres, fr, li.n_atoms, atom, none, e_el, e_vd);
    return wave_sum(e_el + e_vd);
  }
  constexpr int K = 2;
  const int lane = threadIdx.x & (kWave - 1);
  double e_vd = 0.0;
  const int nblk = (li.n_atoms + kWave * K - 1) / (kWave * K);
  for (int blk = 0; blk < nblk; ++blk) {
    int lx[K], ly[K], lz[K];
    bool valid[K];
    double cq[K], ca[K], cb[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int j = lane + kWave * (blk * K + k);
      valid[k] = j < li.n_atoms;
      if (valid[k]) {
        double x, y, z;
        v.at(j, x, y, z);
        lx[k] = to_fixed(x, fr.ox, fr.scale, fr.lim, &sat);
        ly[k] = to_fixed(y, fr.oy, fr.scale, fr.lim, &sat);
        lz[k] = to_fixed(z, fr.oz, fr.scale, fr.lim, &sat);
        const LigAtom la = a.latoms[li.atom_base + j];
        cq[k] = la.keq; ca[k] = la.a; cb[k] = la.b;
      } else {
        lx[k] = ly[k] = lz[k] = 0;
        cq[k] = ca[k] = cb[k] = 0.0;
      }
    }
    float qx, qy, qz, R;
    if (!wave_query<K>(lx, ly, lz, valid, fr.inv_s, qx, qy, qz, R)) continue;
    e_vd += cull_sweep_f64<K>(a.cg, s_cell, s_pos, s_ab, 1.0 / fr.scale, qx, qy, qz, R, lx, ly,
                              lz, cq, ca, cb);
  }
  return wave_sum(e_vd);
}

// E_intra of the conformer in LDS (rigid-motion invariant, so the pose is not needed);
// src/mol.ml:881-903 over the precomputed pair list, FP64
__device__ double mc_intra(const McArgs& a, const LigInfo& li, const double* sx, const double* sy,
                           const double* sz) {
  const int lane = threadIdx.x & (kWave - 1);
  const int n = li.n_pairs;
  const uint32_t* pij = a.pair_ij + li.pair_base;
  const double4* ppar = a.pair_par + li.pair_base;
  double e = 0.0;
  // four pairs per lane per pass, their loads issued together (one memory latency per
  // four pairs); each lane still sums its pairs lane, lane + 64, ... in that order
  for (int p0 = lane; p0 < n; p0 += 4 * kWave) {
    uint32_t ij[4];
    double4 pp[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int p = p0 + u * kWave;
      ij[u] = p < n ? pij[p] : 0u;
      pp[u] = p < n ? ppar[p] : make_double4(0.0, 0.0, 0.0, 0.0);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (p0 + u * kWave >= n) break;
      const int i = ij[u] & 0xffff, j = ij[u] >> 16;
      const double dx = sx[i] - sx[j], dy = sy[i] - sy[j], dz = sz[i] - sz[j];
      const double r2 = dx * dx + dy * dy + dz * dz;
      const double irr = rsqrt(fmax(r2, 1.0e-4));   // no branch around the refinement
      const double ir = r2 >= 1.0e-4 ? irr : 100.0;   // 1 / max(r, 0.01)
      const double uu = ir * ir, u3 = uu * uu * uu, u6 = u3 * u3;
      e += pp[u].x * ir + pp[u].y * u6 - pp[u].z * u3;
    }
  }
  return wave_sum(e);
}

// LDS writes of one wavefront made visible to its other lanes (the chain's conformer
// buffers belong to one wavefront; the workgroup's other wavefronts run other chains)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// E_intra of a chain that turns one torsion at a time: only pairs with one atom in the turned
// group change, so the energy of every round (64 pairs) is kept per chain and a proposal
// evaluates the rounds that hold such pairs.  The pairs are listed by the torsions they feel
// (McPairs, api.hip), which leaves 41 % of the rounds of ligands of 26 to 132 atoms to a
// torsion (26 % for the largest; 25 % of the pairs).  A round's energy has two places: the
// proposal's goes to the one that sel does not name, and accepting it flips the rounds' bits.
// The sum is over all rounds in their order, whichever were evaluated.
// A frame's latency bounds this form up to some 6,000 chains (96 chains alone take 60 % of
// their time), and the pair sum was half of it: 8,100 pairs of a 132-atom ligand 28,000 cycles
// alone and 57,000 with four wavefronts on a SIMD, now 8,000 to 20,000 and 24,000.  6,144
// chains on the grids, 1,000 frames: 25.4 -> 17.8 ms (12,288: 38.9 -> 30.5).  Energies kept
// per pair, not per round, were 22.9 ms (every frame reads them all back); the whole list with
// the parameters formed from the atoms' in LDS 27.6.
struct PairLoad {
  uint32_t ij;
  double2 qa;   // ke qi qj, Ai Aj
  double b;     // 2 Bi Bj
};
__device__ __forceinline__ PairLoad load_pair(const McArgs& a, int64_t p) {
  return {a.pe_ij[p], a.pe_qa[p], a.pe_b[p]};
}
__device__ __forceinline__ double mc_pair(const PairLoad& p, const double* sx, const double* sy,
                                          const double* sz) {
  const int i = p.ij & 0xffff, j = p.ij >> 16;
  const double dx = sx[i] - sx[j], dy = sy[i] - sy[j], dz = sz[i] - sz[j];
  const double r2 = dx * dx + dy * dy + dz * dz;
  const double irr = rsqrt(fmax(r2, 1.0e-4));   // no branch around the refinement
  const double ir = r2 >= 1.0e-4 ? irr : 100.0;   // 1 / max(r, 0.01)
  const double uu = ir * ir, u3 = uu * uu * uu, u6 = u3 * u3;
  return p.qa.x * ir + p.qa.y * u6 - p.b * u3;
}

// Sums of two rounds at once: the halves of the wavefront are exchanged first, so that the
// other five steps of a wavefront sum serve both; lane 31 gets round 0's, lane 63 round 1's.
__device__ __forceinline__ double two_round_sums(double v0, double v1) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v0), __double2loint(v1), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v0), __double2hiint(v1), false, false);
  double v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
  v += dpp_d<0x111>(v, 0.0);
  v += dpp_d<0x112>(v, 0.0);
  v += dpp_d<0x114>(v, 0.0);
  v += dpp_d<0x118>(v, 0.0);
  v += dpp_d<0x142, 0xa>(v, 0.0);
  return v;
}

// a 64-bit word that all lanes hold, as a scalar
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (uint64_t)hi << 32 | lo;
}

// mask (nullable): the rounds to evaluate, per word of 64 rounds; sel: the rounds' places
__device__ double mc_intra_table(const McArgs& a, const McPairs& mp, double* E, const uint64_t* sel,
                                 const uint64_t* mask, const double* sx, const double* sy,
                                 const double* sz) {
  const int lane = threadIdx.x & (kWave - 1);
  double e = 0.0;
  for (int w = 0; w < mp.words; ++w) {
    const uint64_t s = uniform64(sel[w]), m = mask ? uniform64(mask[w]) : 0ull;
    const int r0 = 64 * w;
    // the next two rounds' pairs are fetched while two are evaluated
    PairLoad next[2];
    int nq[2];
    uint64_t todo = m;
    auto fetch = [&]() {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        // an odd last round is evaluated twice, to the same place
        if (u == 0 || todo) nq[u] = __builtin_ctzll(todo);
        else nq[u] = nq[0];
        todo &= todo - 1;
        next[u] = load_pair(a, mp.base + (int64_t)(r0 + nq[u]) * kWave + lane);
      }
    };
    bool more = todo != 0;
    if (more) fetch();
    while (more) {
      const PairLoad cur[2] = {next[0], next[1]};
      const int q = lane < 32 ? nq[0] : nq[1];
      more = todo != 0;
      if (more) fetch();
      const double v0 = mc_pair(cur[0], sx, sy, sz), v1 = mc_pair(cur[1], sx, sy, sz);
      const double v = two_round_sums(v0, v1);
      if ((lane & 31) == 31) E[((s >> q) & 1 ? 0 : mp.rounds) + r0 + q] = v;
    }
    wave_sync();
    const uint64_t at = s ^ m;
    if (r0 + lane < mp.rounds) e += E[((at >> lane) & 1 ? mp.rounds : 0) + r0 + lane];
  }
  return wave_sum(e);
}

// All rounds of every chain, to the places sel names: before a run's first launch, and when
// the parameters have changed.  One wavefront per chain.
__global__ void __launch_bounds__(64) k_mc_pairs(McArgs a) {
  extern __shared__ __align__(16) char smem[];
  const int chain = blockIdx.x, lane = threadIdx.x;
  const McPairs mp = a.pe_lig[a.chain_lig[chain]];
  if (mp.rounds == 0) return;
  double* sx = reinterpret_cast<double*>(smem);
  double* sy = sx + a.max_atoms;
  double* sz = sy + a.max_atoms;
  const int L = a.ligs[a.chain_lig[chain]].n_atoms;
  const double* conf = a.conf + 3 * (size_t)a.chain_atom[chain];
  for (int j = lane; j < L; j += kWave) {
    sx[j] = conf[3 * j]; sy[j] = conf[3 * j + 1]; sz[j] = conf[3 * j + 2];
  }
  __syncthreads();
  double* E = a.pe + a.pe_off[chain];
  const uint64_t* sel = a.pe_sel + (size_t)chain * a.pe_words;
  for (int q0 = 0; q0 < mp.rounds; q0 += 2) {
    const int q1 = min(q0 + 1, mp.rounds - 1);
    const double v0 = mc_pair(load_pair(a, mp.base + (int64_t)q0 * kWave + lane), sx, sy, sz);
    const double v1 = mc_pair(load_pair(a, mp.base + (int64_t)q1 * kWave + lane), sx, sy, sz);
    const double v = two_round_sums(v0, v1);
    const int q = lane < 32 ? q0 : q1;
    if ((lane & 31) == 31) E[((sel[q / 64] >> (q % 64)) & 1 ? mp.rounds : 0) + q] = v;
  }
}

struct RecView {
  const RecPos* pos;
  const RecAB* ab;
  const int* cell;
  int* wl;                        // this wavefront's atom_sweep scratch (LDS)
};

template <int INTER>
__device__ double mc_inter(const McArgs& a, const LigInfo& li, const PoseView& v, const RecView& r) {
  if (INTER == kMcInterGrid) return mc_inter_interp(a, li, v);
  return mc_inter_direct<INTER>(a, li, v, r.pos, r.ab, r.cell, r.wl);
}

// ---------------------------------------------------------------- pooled sweeps
// With few chains per CU a chain's frame is one wavefront's sweep after another (96 chains of
// 26 to 132 atoms: 225,000 of 240,000 cycles a frame) while the CU's other wavefronts have
// none.  POOL: the first `slots` wavefronts of a workgroup run chains and all of them share the
// sweeps, a unit of four atoms at a time from an LDS counter, between two barriers a frame.  A
// unit leaves its FP32 sums per lane in memory (3 KiB) and the chain's wavefront adds them in
// the atoms' order, as atom_sweep does: every energy keeps its bits.
// 100 frames in the direct form, 3,000-atom receptor: 5 chains 7.9 -> 2.6 ms, 96 17.0 -> 3.9, 1,000
// 14.8 -> 6.5, 2,000 14.8 -> 9.7, 3,000 15.4 -> 12.8.
struct PoolLds {
  int atoms[kMcPoolSlots], base[kMcPoolSlots];   // of the pose to sweep, 0: none
  int live[kMcPoolSlots];
  int next;
};

// One unit: atoms 4 u .. 4 u + 3 (in the sweep's order) of a pose of n atoms.
__device__ __forceinline__ void pool_unit(const McArgs& a, const PoseView& v, int n, int atom_base, int u,
                                          const RecView& rv, float4* out) {
  constexpr int NA = 4;
  const int lane = threadIdx.x & (kWave - 1);
  const Frame& fr = a.fr;
  const PairK pk = pair_k(fr.inv_s2, fr.inv_s, a.rres);
  const int j0 = NA * u;
  LigPt l = lig_pt_zero();
  int sat = 0;
  if (lane < NA && j0 + lane < n) {
    const int ja = a.atom_order ? a.atom_order[atom_base + j0 + lane] : j0 + lane;
    double x, y, z;
    v.at(ja, x, y, z);
    l = lig_pt(x, y, z, fr, &sat);
  }
  (void)sat;   // saturated atoms stay beyond the cutoff of every receptor atom
  LigPt lu[NA];
  float c1[NA] = {}, fa[NA] = {}, fb[NA] = {};
  float sq[NA], s12[NA], s6[NA], fe[NA], fx[NA], fy[NA], fz[NA];
#pragma unroll
  for (int k = 0; k < NA; ++k) {
    const int s = j0 + k < n ? k : 0;   // a short last unit repeats its first atom
    lu[k].x = __builtin_amdgcn_readlane(l.x, s);
    lu[k].y = __builtin_amdgcn_readlane(l.y, s);
    lu[k].z = __builtin_amdgcn_readlane(l.z, s);
    lu[k].rx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(l.rx), s));
    lu[k].ry = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(l.ry), s));
    lu[k].rz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(l.rz), s));
  }
  sweep_pass<false, true, NA, false>(a.cg, rv.cell, rv.pos, rv.ab, fr.inv_s, pk, rv.wl, lu, c1, fa, fb,
                                     sq, s12, s6, fe, fx, fy, fz);
  out[lane] = make_float4(sq[0], sq[1], sq[2], sq[3]);
  out[kWave + lane] = make_float4(s12[0], s12[1], s12[2], s12[3]);
  out[2 * kWave + lane] = make_float4(s6[0], s6[1], s6[2], s6[3]);
}

// The pose's energy from its units, in atom_sweep's order.
__device__ __forceinline__ double pool_energy(const McArgs& a, const LigInfo& li, const float4* units) {
  const int lane = threadIdx.x & (kWave - 1);
  double e_el = 0.0, e_vd = 0.0;
  for (int jb = 0; jb < li.n_atoms; jb += kWave) {
    double mq = 0.0, ma = 0.0, mb = 0.0;
    if (jb + lane < li.n_atoms) {
      const int ja = a.atom_order ? a.atom_order[li.atom_base + jb + lane] : jb + lane;
      const LigAtom la = a.latoms[li.atom_base + ja];
      mq = la.keq; ma = la.a; mb = la.b;
    }
    const int nj = min(kWave, li.n_atoms - jb);
    const float4* p = units + (size_t)(jb / 4) * 3 * kWave + lane;
#pragma unroll 2
    for (int jj = 0; jj < nj; jj += 4, p += 3 * kWave) {
      const float4 q = p[0], t12 = p[kWave], t6 = p[2 * kWave];
      const float sq[4] = {q.x, q.y, q.z, q.w}, s12[4] = {t12.x, t12.y, t12.z, t12.w},
                  s6[4] = {t6.x, t6.y, t6.z, t6.w};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (jj + u >= nj) break;
        e_el = fma((double)sq[u], readlane_d(mq, jj + u), e_el);
        e_vd = fma((double)s12[u], readlane_d(ma, jj + u), e_vd);
        e_vd = fma(-2.0 * (double)s6[u], readlane_d(mb, jj + u), e_vd);
      }
    }
  }
  return wave_sum(e_el + e_vd);
}

// ------------------------------------------------- Monte Carlo-plus-minimisation
// LDS of one chain's minimiser (after the chain slots): the minimised conformer and the
// adjoint, 6 x max_atoms FP64
struct MinLds {
  double *tx, *ty, *tz, *hx, *hy, *hz;
};

// Local minimisation of the proposal (conformer sx.. with centre c, rotation nrot,
// position npos): the base rows are the proposal pose centred at the origin,
// b_j = nrot (x_j - c), so that the DOF vector [npos, 0, 0, 0, 0..] is the proposal
// itself; min_iters L-BFGS evaluations of E_inter + E_intra (the chain's energy form)
// over [t, alpha, beta, gamma, tau_0..] (torsions only for flexible ligands).  Returns
// the energy of the best point and leaves its conformer (before the rigid motion) in
// m.tx.., its rigid motion in M, T and the pose centre (M mean(conformer) + T) in cpos;
// E_inter / E_intra of that point go to the chain state.
template <int INTER>
__device__ double mc_minimize(const McArgs& a, const LigInfo& li, int chain, bool flex,
                              bool use_intra, const PoseView& v, const RecView& rv, const MinLds& m,
                              McState& st, double* M, double* T, double* cpos) {
  const int lane = threadIdx.x & (kWave - 1);
  const int L = li.n_atoms;
  double* gbase = a.min_base + 3 * (size_t)a.chain_atom[chain];
  for (int j = lane; j < L; j += kWave) {   // lane j later reads back the rows it wrote
    double x, y, z;
    v.at(j, x, y, z);
    gbase[3 * j] = x - v.q->p[0]; gbase[3 * j + 1] = y - v.q->p[1]; gbase[3 * j + 2] = z - v.q->p[2];
  }
  DofEval ev;
  ev.li = li; ev.latoms = a.latoms; ev.atom_order = a.atom_order; ev.rb_left = a.rb_left;
  ev.rb_right = a.rb_right; ev.rg_off = a.rg_off; ev.rg_atoms = a.rg_atoms;
  ev.pair_ij = a.pair_ij; ev.pair_par = a.pair_par; ev.ntors = flex ? li.nrb : 0;
  ev.intra = use_intra; ev.fr = a.fr; ev.s_pos = rv.pos; ev.s_ab = rv.ab; ev.s_cell = rv.cell;
  ev.rres = a.rres; ev.cg = a.cg; ev.wl = rv.wl; ev.g = a.g;
  const int n = 6 + ev.ntors;
  const bool act = lane < n;
  const MinCfg cfg{a.min_m, a.min_max_step, a.min_min_step, a.min_gtol, a.min_c1};
  double* S = a.min_S + (size_t)chain * a.min_m * kWave + lane;
  double* Y = a.min_Y + (size_t)chain * a.min_m * kWave + lane;
  double* rho = a.min_rho + (size_t)chain * a.min_m;
  MinPose s{};
  double xt = lane == 0 ? v.q->p[0] : lane == 1 ? v.q->p[1] : lane == 2 ? v.q->p[2] : 0.0;
  double x = 0.0, g = 0.0, d = 0.0, e_inter = 0.0, e_intra = 0.0;
  for (int it = 0; it < a.min_iters && __builtin_amdgcn_readfirstlane(s.status) == kMinRunning; ++it) {
    double gt, ei, ea, rad;
    const double f = dof_eval<INTER>(ev, gbase, xt, m.tx, m.ty, m.tz, m.hx, m.hy, m.hz, gt, ei, ea, rad);
    const int acc0 = s.n_acc, init0 = s.init;
    xt = lbfgs_wave(s, x, g, d, xt, f, act ? gt : 0.0, rad, -__builtin_inf(), __builtin_inf(), act,
                    S, Y, (size_t)kWave, rho, 1, cfg);
    if (!init0 || s.n_acc != acc0) { e_inter = ei; e_intra = ea; }   // the accepted point
  }
  st.min_evals += s.n_eval;
  st.prev_e_inter = e_inter;
  st.prev_e_intra = e_intra;
  // the best point's conformer and rigid motion
  double sn, cs;
  dof_pose(ev, gbase, x, m.tx, m.ty, m.tz, M, nullptr, nullptr, nullptr, T, sn, cs);
  double s0 = 0.0, s1 = 0.0, s2 = 0.0;
  for (int j = lane; j < L; j += kWave) { s0 += m.tx[j]; s1 += m.ty[j]; s2 += m.tz[j]; }
  const double cx = wave_sum(s0) / L, cy = wave_sum(s1) / L, cz = wave_sum(s2) / L;
  cpos[0] = (M[0] * cx + M[1] * cy + M[2] * cz) + T[0];
  cpos[1] = (M[3] * cx + M[4] * cy + M[5] * cz) + T[1];
  cpos[2] = (M[6] * cx + M[7] * cy + M[8] * cz) + T[2];
  return s.f;
}

// --------------------------------------------------------------------- the kernel
// A workgroup of `waves` wavefronts, each running its own chains; with REC_LDS the
// workgroup first stages the receptor and its cell table in LDS, shared by all chains.
// one instantiation per energy form, so that each carries only its own registers
// Wavefronts per workgroup each form is compiled for.  16 caps every form at 128 VGPRs
// (4 wavefronts per SIMD; the chain's control code then spills ~260-340 B per lane to
// scratch): measured faster than 8 (about 200 VGPRs, 2 per SIMD) for the direct forms
// (15.4 M against 14.2 M steps/s) and for the grid form (225 M against 203 M).
__host__ __device__ constexpr int mc_form_waves(int, bool min) { return min ? 8 : 16; }

template <bool REC_LDS, int INTER, bool MIN, bool POOL = false>
__global__ void __launch_bounds__(mc_form_waves(INTER, MIN) * 64) k_mc(McArgs a, int rec_bytes) {
  extern __shared__ __align__(16) char mc_lds[];
  RecView rv;
  load_receptor<REC_LDS>(a.rpos, a.rab, a.nrec, a.cg, rv.pos, rv.ab, rv.cell, mc_lds);
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x / kWave;
  // the chain's conformer; a torsion proposal turns it in place, with the moved atoms'
  // previous coordinates in the chain's undo rows (HBM) until the decision
  double* cx_ = reinterpret_cast<double*>(mc_lds + rec_bytes) + (size_t)wv * 3 * a.max_atoms;
  double* cy_ = cx_ + a.max_atoms;
  double* cz_ = cy_ + a.max_atoms;
  const int nwv = blockDim.x / kWave;
  McState* s_st = reinterpret_cast<McState*>(
      mc_lds + rec_bytes + (((size_t)nwv * 3 * a.max_atoms * sizeof(double) + 15) & ~(size_t)15));
  McPose* pose = reinterpret_cast<McPose*>(s_st + nwv) + wv;   // this chain's pose slot
  rv.wl = reinterpret_cast<int*>(reinterpret_cast<McPose*>(s_st + nwv) + nwv) + wv * kAtomSweepInts;
  MinLds ml{};
  if (MIN) {
    // after the scratch of every wavefront: 6 x max_atoms FP64 per wavefront
    double* b = reinterpret_cast<double*>(
                    reinterpret_cast<int*>(reinterpret_cast<McPose*>(s_st + nwv) + nwv) +
                    nwv * kAtomSweepInts) +
                (size_t)wv * 6 * a.max_atoms;
    ml = MinLds{b, b + a.max_atoms, b + 2 * a.max_atoms, b + 3 * a.max_atoms,
                b + 4 * a.max_atoms, b + 5 * a.max_atoms};
  }
  const double pi = 3.14159265358979311600;       // 4 atan 1 (src/math.ml:13)

  // POOL: shared by the workgroup; a round = the units of every published pose.  False once no
  // wavefront runs a chain: the same for all of them, and the last time any of them asks.
  PoolLds& pl = *reinterpret_cast<PoolLds*>(
      reinterpret_cast<int*>(reinterpret_cast<McPose*>(s_st + nwv) + nwv) + nwv * kAtomSweepInts);
  const size_t pool_units = (a.max_atoms + 3) / 4;
  float4* const pool = POOL ? a.pool + (size_t)blockIdx.x * a.pool_slots * pool_units * 3 * kWave : nullptr;
  auto pool_round = [&]() __attribute__((always_inline)) {
    if (threadIdx.x == 0) pl.next = 0;
    __syncthreads();
    int any = 0;
    for (int k = 0; k < a.pool_slots; ++k) any |= pl.live[k];
    if (!__builtin_amdgcn_readfirstlane(any)) return false;
    for (;;) {
      int u = 0;
      if (lane == 0) u = atomicAdd(&pl.next, 1);
      u = __builtin_amdgcn_readlane(u, 0);
      int sl = 0, n = 0;
      for (; sl < a.pool_slots; ++sl) {
        n = __builtin_amdgcn_readfirstlane(pl.atoms[sl]);
        if (u < (n + 3) / 4) break;
        u -= (n + 3) / 4;
      }
      if (sl == a.pool_slots) break;
      const double* c = reinterpret_cast<const double*>(mc_lds + rec_bytes) + (size_t)sl * 3 * a.max_atoms;
      const PoseView v{c, c + a.max_atoms, c + 2 * a.max_atoms, reinterpret_cast<McPose*>(s_st + nwv) + sl};
      pool_unit(a, v, n, __builtin_amdgcn_readfirstlane(pl.base[sl]), u, rv,
                pool + ((size_t)sl * pool_units + u) * 3 * kWave);
    }
    __syncthreads();
    return true;
  };
  auto inter = [&](const LigInfo& li, const PoseView& v) __attribute__((always_inline)) {
    if constexpr (!POOL) {
      return mc_inter<INTER>(a, li, v, rv);
    } else {
      if (lane == 0) { pl.atoms[wv] = li.n_atoms; pl.base[wv] = li.atom_base; }
      (void)pool_round();
      return pool_energy(a, li, pool + (size_t)wv * pool_units * 3 * kWave);
    }
  };
  bool first = true;   // POOL: the first chains are dealt, to and fro over the workgroups
  const bool keeper = !POOL || wv < a.pool_slots;
  if (POOL && keeper && lane == 0) pl.live[wv] = 1;

  for (; keeper;) {
    // the next chain: lane 0 takes it from the queue; readlane makes it a scalar, so the
    // loop exit is uniform
    int qv = 0;
    if (lane == 0 && !(POOL && first)) qv = atomicAdd(a.queue, 1);
    int q = __builtin_amdgcn_readlane(qv, 0);
    if (POOL) {
      const int nb = gridDim.x, b = blockIdx.x, w = __builtin_amdgcn_readfirstlane(wv);
      q = first ? w * nb + ((w & 1) ? nb - 1 - b : b) : a.pool_slots * nb + q;
      first = false;
    }
    if (q >= a.nwork) break;
    const int chain = a.work[q];
    // the chain's state in this wavefront's LDS slot (wave-uniform values)
    McState& st = s_st[wv];
    {
      const int* src = reinterpret_cast<const int*>(a.st + chain);
      int* dst = reinterpret_cast<int*>(&st);
      for (int k = lane; k < (int)(sizeof(McState) / 4); k += kWave) dst[k] = src[k];
    }
    wave_sync();
    if (st.status != kMcRunning) continue;
    const int lig = a.chain_lig[chain];
    const LigInfo li = a.ligs[lig];
    const int L = li.n_atoms, nrb = li.nrb;
    double* gconf = a.conf + 3 * (size_t)a.chain_atom[chain];
    double* gbest = a.best_xyz + 3 * (size_t)a.chain_atom[chain];
    double* gundo = a.undo + 3 * (size_t)a.chain_atom[chain];
    // group [g0, g1) of a torsion back to the coordinates saved in the undo rows (each
    // lane restores the atoms it saved)
    auto restore = [&](int g0, int g1) {
      for (int m = g0 + lane; m < g1; m += kWave) {
        const int at = a.rg_atoms[m];
        const double* u = gundo + 3 * (size_t)(m - g0);
        cx_[at] = u[0]; cy_[at] = u[1]; cz_[at] = u[2];
      }
      wave_sync();
    };
    double* dr = a.rb_dr + a.chain_rb[chain];
    SwState* rsw = a.rb_sw + a.chain_rb[chain];
    for (int j = lane; j < L; j += kWave) {
      cx_[j] = gconf[3 * j]; cy_[j] = gconf[3 * j + 1]; cz_[j] = gconf[3 * j + 2];
    }
    wave_sync();
    const bool flex = (a.flags & kMcTweak) && nrb > 0;
    const bool use_intra = (a.flags & kMcIntraUff) != 0;
    // the chain's pair energies, if it keeps them
    McPairs mp{};
    if (!MIN && a.pe && use_intra && flex) mp = a.pe_lig[lig];
    double* const pe = mp.rounds ? a.pe + a.pe_off[chain] : nullptr;
    uint64_t* const sel = a.pe_sel + (size_t)chain * a.pe_words;
    const uint64_t* mask = nullptr;   // rounds of the proposal's torsion

    if (!st.initialized) {
      // start pose: Mol.rotate_then_translate_copy centered_lig rot0 pos0, no
      // re-centring (src/lds.ml:759, src/mol.ml:669-672); E of the start pose
      if (lane == 0) {
        for (int k = 0; k < 9; ++k) pose->m[k] = st.rot0[k];
        for (int k = 0; k < 3; ++k) { pose->c[k] = 0.0; pose->p[k] = st.pos0[k]; }
      }
      wave_sync();
      const PoseView v{cx_, cy_, cz_, pose};
      st.prev_e_intra = mp.rounds ? mc_intra_table(a, mp, pe, sel, nullptr, cx_, cy_, cz_)
                        : use_intra ? mc_intra(a, li, cx_, cy_, cz_) : 0.0;
      st.prev_e_inter = inter(li, v);
      st.prev_e = st.prev_e_inter + st.prev_e_intra;
      st.best_e = st.prev_e;
      for (int k = 0; k < 9; ++k) { st.rot[k] = st.rot0[k]; st.best_rot[k] = st.rot0[k]; }
      for (int k = 0; k < 3; ++k) { st.pos[k] = st.pos0[k]; st.best_pos[k] = st.pos0[k]; }
      for (int j = lane; j < L; j += kWave) {
        double x, y, z;
        v.at(j, x, y, z);
        gbest[3 * j] = x; gbest[3 * j + 1] = y; gbest[3 * j + 2] = z;
      }
      st.initialized = 1;
    }

    // the draws of frames draws_at .. draws_end - 1, in the lanes
    constexpr int kDraws = kWave / 3;
    double draw_a = 0.0, draw_b = 0.0, draw_s = 0.0, draw_c = 0.0;
    int draws_at = 0, draws_end = 0;
    const int frame_end = min(st.frame + a.nsteps, a.total_frames);
    for (; st.frame < frame_end; ++st.frame) {
      const bool rigid = (st.frame & 1) == 0;
      const int frame = __builtin_amdgcn_readfirstlane(st.frame);
      if (frame >= draws_end) {
        // the numbers of the next kDraws frames (one draw for all of them where every frame had
        // its three generator calls and a sincos in all lanes: a fifth of the vector
        // instructions of a frame on the grids): lane 3 f + c draws pair c of frame f; lanes
        // of pair 0 also take the frame's angle (rigid: Move.rand_rot, torsion:
        // Move.rand_angle, src/move.ml:14-31) with the step sizes as they are now
        const int f = frame + lane / 3;
        const uint4 r = philox(make_uint4((uint32_t)chain, (uint32_t)f, (uint32_t)(lane % 3), 0x4D4D4F31u),
                               a.seed_lo, a.seed_hi);
        uniform2(r, draw_a, draw_b);
        double u = draw_a, amp = st.max_rot;
        if (f & 1) {
          u = draw_b;
          const int step = st.conf_step + ((f >> 1) - (frame >> 1));
          const bool flip = step > 0 && step % kMcBlock == 0 && !(a.flags & kMcNoFlip);
          amp = pi;
          if (flex && !flip) {
            const int i = (int)(draw_a * nrb);
            amp = dr[i < nrb ? i : nrb - 1];
          }
        }
        sincos(u * (2.0 * amp) - amp, &draw_s, &draw_c);
        draws_at = frame;
        draws_end = frame + kDraws;
      }
      const int dl = 3 * (frame - draws_at);
      const double u0 = readlane_d(draw_a, dl), u1 = readlane_d(draw_b, dl);
      const double ds = readlane_d(draw_s, dl), dc = readlane_d(draw_c, dl);

      // ---- proposal
      double nrot[9], npos[3], ccx, ccy, ccz;
      const double* sx = cx_;
      const double* sy = cy_;
      const double* sz = cz_;
      int just_rotated = -1;
      int mg0 = 0, mg1 = 0;   // torsion group turned in place by this proposal
      ccx = st.center[0]; ccy = st.center[1]; ccz = st.center[2];
      if (!rigid) {
        for (int k = 0; k < 9; ++k) nrot[k] = st.rot[k];
        for (int k = 0; k < 3; ++k) npos[k] = st.pos[k];
        if (flex) {
          // Mol.flip_rbond / tweak_rbond on a copy (src/lds.ml:784-795, src/mol.ml:635-647)
          int i = (int)(u0 * nrb);
          i = i < nrb ? i : nrb - 1;
          const int left = a.rb_left[li.rb_base + i], right = a.rb_right[li.rb_base + i];
          const double ox = cx_[right], oy = cy_[right], oz = cz_[right];
          const double vx = ox - cx_[left], vy = oy - cy_[left], vz = oz - cz_[left];
          const double mag = sqrt(vx * vx + vy * vy + vz * vz);
          const Rod rod = rodrigues(vx / mag, vy / mag, vz / mag, ds, dc);
          const double* Rm = rod.m;
          wave_sync();
          const int g0 = a.rg_off[li.rg_base + i], g1 = a.rg_off[li.rg_base + i + 1];
          for (int m = g0 + lane; m < g1; m += kWave) {
            const int at = a.rg_atoms[m];
            const double x0 = cx_[at], y0 = cy_[at], z0 = cz_[at];
            double* u = gundo + 3 * (size_t)(m - g0);
            u[0] = x0; u[1] = y0; u[2] = z0;
            const double zx = x0 - ox, zy = y0 - oy, zz = z0 - oz;
            cx_[at] = (Rm[0] * zx + Rm[1] * zy + Rm[2] * zz) + ox;
            cy_[at] = (Rm[3] * zx + Rm[4] * zy + Rm[5] * zz) + oy;
            cz_[at] = (Rm[6] * zx + Rm[7] * zy + Rm[8] * zz) + oz;
          }
          wave_sync();
          // update_center (A.favg) and enclosing radius (src/mol.ml:353-356, :576-591)
          double s0 = 0.0, s1 = 0.0, s2 = 0.0;
          for (int j = lane; j < L; j += kWave) { s0 += cx_[j]; s1 += cy_[j]; s2 += cz_[j]; }
          ccx = wave_sum(s0) / L; ccy = wave_sum(s1) / L; ccz = wave_sum(s2) / L;
          double rmax = 0.0;
          for (int j = lane; j < L; j += kWave) {
            const double dx = ccx - cx_[j], dy = ccy - cy_[j], dz = ccz - cz_[j];
            rmax = fmax(rmax, 0.01 + sqrt(dx * dx + dy * dy + dz * dz));
          }
          rmax = wave_max(rmax);
          if (rmax > 12.0) {   // Mol.Too_long: the chain ends (src/lds.ml:794, :997)
            restore(g0, g1);   // with its last accepted conformer
            st.status = kMcTooLong;
            break;
          }
          mg0 = g0;
          mg1 = g1;
          just_rotated = i;
          mask = a.pe_mask + mp.mask_base + (size_t)i * mp.words;
        }
      } else {
        // Move.rand_rot: left-multiply the passive axis rotation Rot.rx / ry / rz
        // (src/move.ml:20-31, src/rot.ml:22-46).  Two rows of rot mix,
        // p' = c p + s q and q' = c q - s p, with (p, q) = rows (1, 2) for x, (2, 0) for y,
        // (0, 1) for z.  Written with selects: a switch that built the 3x3 matrix per axis
        // was mis-lowered by hipcc (the -s entry of the z matrix came out 0).
        int ax = (int)(u1 * 3.0);
        ax = ax < 3 ? ax : 2;
        const double s = ds, c = dc;
        const bool ax0 = ax == 0, ax1 = ax == 1;
        for (int cc = 0; cc < 3; ++cc) {
          const double r0 = st.rot[cc], r1 = st.rot[3 + cc], r2 = st.rot[6 + cc];
          const double p = ax0 ? r1 : (ax1 ? r2 : r0);
          const double q = ax0 ? r2 : (ax1 ? r0 : r1);
          const double pn = c * p + s * q, qn = c * q - s * p;
          nrot[cc] = ax0 ? r0 : (ax1 ? qn : pn);
          nrot[3 + cc] = ax0 ? pn : (ax1 ? r1 : qn);
          nrot[6 + cc] = ax0 ? qn : (ax1 ? pn : r2);
        }
        // Move.rand_trans (src/move.ml:46-54)
        const double u2 = readlane_d(draw_a, dl + 1), u3 = readlane_d(draw_b, dl + 1),
                     u4 = readlane_d(draw_a, dl + 2);
        npos[0] = st.pos[0] + (u2 * 2.0 - 1.0) * st.max_trans;
        npos[1] = st.pos[1] + (u3 * 2.0 - 1.0) * st.max_trans;
        npos[2] = st.pos[2] + (u4 * 2.0 - 1.0) * st.max_trans;
      }

      // the proposal's pose and the frame's Metropolis uniform go to the chain's LDS slot;
      // from here on they are read from there (the memory clobber below keeps the
      // compiler from carrying them in registers across the energy sweep)
      if (lane == 0) {
        for (int k = 0; k < 9; ++k) pose->m[k] = nrot[k];
        pose->c[0] = ccx; pose->c[1] = ccy; pose->c[2] = ccz;
        for (int k = 0; k < 3; ++k) pose->p[k] = npos[k];
        pose->u = readlane_d(draw_b, dl + 2);
      }
      wave_sync();
      asm volatile("" ::: "memory");

      // ---- energies (stored before the acceptance test, src/lds.ml:900-904)
      const PoseView v{sx, sy, sz, pose};
      double curr_e, cpos[3];
      double mM[9], mT[3];   // MIN: rigid motion of the minimised pose
      if constexpr (MIN) {
        // the proposal, locally minimised; its centre is the pose centre of the ROI test
        curr_e = mc_minimize<INTER>(a, li, chain, flex, use_intra, v, rv, ml, st, mM, mT, cpos);
      } else {
        if (!rigid && use_intra && flex)
          st.prev_e_intra = mp.rounds ? mc_intra_table(a, mp, pe, sel, mask, sx, sy, sz)
                                      : mc_intra(a, li, sx, sy, sz);
        st.prev_e_inter = inter(li, v);
        curr_e = st.prev_e_inter + st.prev_e_intra;
      }
      asm volatile("" ::: "memory");
      const McPose& P = *pose;
      if constexpr (!MIN)
        for (int k = 0; k < 3; ++k) cpos[k] = P.p[k];
      const double dxr = a.roi_x - cpos[0], dyr = a.roi_y - cpos[1], dzr = a.roi_z - cpos[2];
      const double dist_roi = sqrt(dxr * dxr + dyr * dyr + dzr * dzr);
      const bool hard = (a.flags & kMcHardRoi) != 0;
      bool reset = false, metropolis = false;
      if (hard) {
        if (dist_roi > a.roi_r) { reset = true; ++st.ooroi; }
        else metropolis = true;
      } else {
        metropolis = (a.flags & kMcMetropolisAlways) != 0;
      }
      if (metropolis && st.prev_e_inter == 0.0) { reset = true; metropolis = false; }
      if (reset) {
        // reset_run_params (src/lds.ml:632-648): the conformer is kept; the best pose
        // becomes the registered conformer at the start pose (best_lig := prev_lig :=
        // rotate_then_translate_copy centered_lig rot0 pos0, src/lds.ml:645-646)
        if (st.max_rot != a.max_rot0) draws_end = 0;   // drawn with the old step size
        st.max_rot = a.max_rot0;
        st.max_trans = a.max_trans0;
        for (int k = 0; k < 9; ++k) { st.rot[k] = st.rot0[k]; st.best_rot[k] = (k % 4 == 0) ? 1.0 : 0.0; }
        for (int k = 0; k < 3; ++k) { st.pos[k] = st.pos0[k]; st.best_pos[k] = 0.0; }
        {
          const double* c0 = a.lig_xyz + 3 * (size_t)li.atom_base;
          const double* R0 = st.rot0;
          const double* p0 = st.pos0;
          for (int j = lane; j < L; j += kWave) {
            const double x0 = c0[3 * j], y0 = c0[3 * j + 1], z0 = c0[3 * j + 2];
            gbest[3 * j] = (R0[0] * x0 + R0[1] * y0 + R0[2] * z0) + p0[0];
            gbest[3 * j + 1] = (R0[3] * x0 + R0[4] * y0 + R0[5] * z0) + p0[1];
            gbest[3 * j + 2] = (R0[6] * x0 + R0[7] * y0 + R0[8] * z0) + p0[2];
          }
        }
        st.prev_e = __builtin_inf();
        st.best_e = __builtin_inf();
        sw_reset(st.sw);
        ++st.resets;
      } else if (metropolis) {
        // u5 is a multiple of 2^-53, so once positive it exceeds exp(-x) for every x >= 40
        // (exp(-40) < 2^-53): those proposals are rejected without evaluating exp
        const double x = (curr_e - st.prev_e) * a.beta;
        const double u5p = P.u;
        const bool accept =
            (curr_e <= st.prev_e) || (!(x >= 40.0 && u5p > 0.0) && u5p < exp(-x));
        if (rigid) sw_process(st.sw, accept);
        else if (just_rotated > -1) sw_process(rsw[just_rotated], accept);
        if (accept) {
          ++st.accepted;
          st.prev_e = curr_e;
          if constexpr (MIN) {
            // the minimised pose: conformer nrot^T c* (the chain's frame), centre nrot^T
            // mean(c*), rotation M* nrot, position its pose centre
            double cm[3] = {0.0, 0.0, 0.0};
            for (int j = lane; j < L; j += kWave) {
              const double x0 = ml.tx[j], y0 = ml.ty[j], z0 = ml.tz[j];
              cx_[j] = P.m[0] * x0 + P.m[3] * y0 + P.m[6] * z0;
              cy_[j] = P.m[1] * x0 + P.m[4] * y0 + P.m[7] * z0;
              cz_[j] = P.m[2] * x0 + P.m[5] * y0 + P.m[8] * z0;
              cm[0] += x0; cm[1] += y0; cm[2] += z0;
            }
            for (int k = 0; k < 3; ++k) cm[k] = wave_sum(cm[k]) / L;
            for (int k = 0; k < 3; ++k)
              st.center[k] = P.m[k] * cm[0] + P.m[3 + k] * cm[1] + P.m[6 + k] * cm[2];
            for (int r = 0; r < 3; ++r)
              for (int cc = 0; cc < 3; ++cc)
                st.rot[3 * r + cc] = mM[3 * r] * P.m[cc] + mM[3 * r + 1] * P.m[3 + cc] +
                                     mM[3 * r + 2] * P.m[6 + cc];
            for (int k = 0; k < 3; ++k) st.pos[k] = cpos[k];
            mg0 = mg1 = 0;   // conf holds the minimised conformer: nothing to restore
            wave_sync();
          } else {
            for (int k = 0; k < 9; ++k) st.rot[k] = P.m[k];
            for (int k = 0; k < 3; ++k) st.pos[k] = P.p[k];
            if (mg1 > mg0) {   // conf := conf' (already in place): keep it
              for (int k = 0; k < 3; ++k) st.center[k] = P.c[k];
              mg0 = mg1 = 0;
              for (int w = lane; w < mp.words; w += kWave) sel[w] ^= mask[w];
            }
          }
        }
        if (curr_e < st.best_e) {   // best pose, accepted or not (src/lds.ml:959-969)
          st.best_e = curr_e;
          if constexpr (MIN) {
            for (int r = 0; r < 3; ++r)
              for (int cc = 0; cc < 3; ++cc)
                st.best_rot[3 * r + cc] = mM[3 * r] * P.m[cc] + mM[3 * r + 1] * P.m[3 + cc] +
                                          mM[3 * r + 2] * P.m[6 + cc];
            for (int k = 0; k < 3; ++k) st.best_pos[k] = cpos[k];
            for (int j = lane; j < L; j += kWave) {
              const double x0 = ml.tx[j], y0 = ml.ty[j], z0 = ml.tz[j];
              gbest[3 * j] = (mM[0] * x0 + mM[1] * y0 + mM[2] * z0) + mT[0];
              gbest[3 * j + 1] = (mM[3] * x0 + mM[4] * y0 + mM[5] * z0) + mT[1];
              gbest[3 * j + 2] = (mM[6] * x0 + mM[7] * y0 + mM[8] * z0) + mT[2];
            }
          } else {
            for (int k = 0; k < 9; ++k) st.best_rot[k] = P.m[k];
            for (int k = 0; k < 3; ++k) st.best_pos[k] = P.p[k];
            for (int j = lane; j < L; j += kWave) {
              double x, y, z;
              v.at(j, x, y, z);
              gbest[3 * j] = x; gbest[3 * j + 1] = y; gbest[3 * j + 2] = z;
            }
          }
        }
        // adaptive rigid steps every 100 rigid frames (src/lds.ml:971-974, :586-600)
        if (rigid && st.rigid_step > 0 && st.rigid_step % kMcBlock == 0) {
          const double ar = sw_ratio(st.sw);
          draws_end = 0;
          if (ar <= 0.45) { st.max_trans *= 0.95; st.max_rot *= 0.95; }
          else if (ar >= 0.55) { st.max_trans *= 1.05; st.max_rot = fmin(pi, 1.05 * st.max_rot); }
        }
        // adaptive torsion steps on the proposal's copy (src/lds.ml:976-979, :603-621):
        // kept only when the proposal was accepted (conf := conf')
        if (accept && flex && !rigid && st.conf_step > 0 && st.conf_step % (kMcBlock * nrb) == 0) {
          draws_end = 0;
          for (int k = 0; k < nrb; ++k) {
            const double ar = sw_ratio(rsw[k]);
            if (ar <= 0.45) dr[k] = 0.95 * dr[k];
            else if (ar >= 0.55) dr[k] = fmin(pi, 1.05 * dr[k]);
          }
        }
      }
      if (mg1 > mg0) restore(mg0, mg1);   // the proposal was not taken: conf stays
      if (rigid) ++st.rigid_step;
      else ++st.conf_step;
    }
    if (st.status == kMcRunning && st.frame >= a.total_frames) st.status = kMcDone;
    // write the chain back (lane 0 for the scalars, all lanes for the conformer)
    for (int j = lane; j < L; j += kWave) {
      gconf[3 * j] = cx_[j]; gconf[3 * j + 1] = cy_[j]; gconf[3 * j + 2] = cz_[j];
    }
    wave_sync();
    {
      const int* src = reinterpret_cast<const int*>(&st);
      int* dst = reinterpret_cast<int*>(a.st + chain);
      for (int k = lane; k < (int)(sizeof(McState) / 4); k += kWave) dst[k] = src[k];
    }
    wave_sync();
  }
  if constexpr (POOL) {
    if (keeper && lane == 0) { pl.live[wv] = 0; pl.atoms[wv] = 0; }
    while (pool_round()) {
    }
  }
}

__global__ void k_mc_reset_queue(int* q) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *q = 0;
}

size_t mc_lds_bytes(const McArgs& a, int waves, bool rec_lds) {
  size_t rec = 0;
  if (rec_lds)
    rec = ((size_t)a.nrec * (sizeof(RecPos) + sizeof(RecAB)) +
           (size_t)(a.cg.nx * a.cg.ny * a.cg.nz + 1) * sizeof(int) + 15) & ~(size_t)15;
  const size_t conf = ((size_t)waves * 3 * a.max_atoms * sizeof(double) + 15) & ~(size_t)15;
  const size_t mins = a.min_iters > 0 ? (size_t)waves * 6 * a.max_atoms * sizeof(double) : 0;
  return rec + conf + (size_t)waves * (sizeof(McState) + sizeof(McPose) + kAtomSweepInts * sizeof(int)) +
         mins + (a.pool_slots > 0 ? (sizeof(PoolLds) + 15) & ~(size_t)15 : 0);
}

template <bool R, int I>
static hipError_t mc_allow_lds(int cap) {
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_mc<R, I, false>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, cap);
  if (e == hipSuccess && I != kMcInterSub)
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_mc<R, I, I != kMcInterSub>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, cap);
  return e;
}

hipError_t mc_prepare() {
  // dynamic LDS above 64 KiB must be allowed per kernel (gfx950: 160 KiB per CU); set
  // once, outside any stream capture
  const int cap = 160 * 1024;
  hipError_t e = hipSuccess;
  if (e == hipSuccess) e = mc_allow_lds<true, kMcInterAtom>(cap);
  if (e == hipSuccess) e = mc_allow_lds<true, kMcInterSub>(cap);
  if (e == hipSuccess) e = mc_allow_lds<true, kMcInterF64>(cap);
  if (e == hipSuccess) e = mc_allow_lds<false, kMcInterAtom>(cap);
  if (e == hipSuccess) e = mc_allow_lds<false, kMcInterSub>(cap);
  if (e == hipSuccess) e = mc_allow_lds<false, kMcInterF64>(cap);
  if (e == hipSuccess) e = mc_allow_lds<false, kMcInterGrid>(cap);
  if (e == hipSuccess)
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_mc<true, kMcInterAtom, false, true>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, cap);
  return e;
}

int mc_inter_kind(const McArgs& a) {
  if (a.inter_mode == MMO_INTERP) return kMcInterGrid;
  if (a.flags & kMcFp64) return kMcInterF64;
  // the minimiser's gradients come from the per-atom sweep
  return (a.sweep == 1 || a.min_iters > 0) ? kMcInterAtom : kMcInterSub;
}

bool mc_can_pool(const McArgs& a) { return mc_inter_kind(a) == kMcInterAtom && a.min_iters == 0; }

int mc_max_waves(const McArgs& a) { return mc_form_waves(mc_inter_kind(a), a.min_iters > 0); }

__global__ void __launch_bounds__(64) k_mc_start(McArgs a) {
  const int chain = blockIdx.x;
  const LigInfo li = a.ligs[a.chain_lig[chain]];
  const double* from = a.lig_xyz + 3 * (size_t)li.atom_base;
  const size_t to = 3 * (size_t)a.chain_atom[chain];
  for (int k = threadIdx.x; k < 3 * li.n_atoms; k += blockDim.x) a.conf[to + k] = a.best_xyz[to + k] = from[k];
}

__global__ void __launch_bounds__(256) k_mc_pair_list(const uint32_t* index, size_t n, const uint32_t* pair_ij,
                                                      const double4* pair_par, uint32_t* ij, double2* qa,
                                                      double* b) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint32_t p = index[k];
  const double4 v = p == kNoPair ? make_double4(0.0, 0.0, 0.0, 0.0) : pair_par[p];
  ij[k] = p == kNoPair ? 0u : pair_ij[p];
  qa[k] = make_double2(v.x, v.y);
  b[k] = v.z;
}

hipError_t launch_mc_pair_list(const uint32_t* index, size_t n, const uint32_t* pair_ij, const double4* pair_par,
                               uint32_t* ij, double2* qa, double* b, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_mc_pair_list, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, index, n, pair_ij, pair_par,
                     ij, qa, b);
  return hipGetLastError();
}

hipError_t launch_mc_start(const McArgs& a, int nchain, hipStream_t s) {
  hipLaunchKernelGGL(k_mc_start, dim3(nchain), dim3(kWave), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_mc_pairs(const McArgs& a, int nchain, hipStream_t s) {
  hipLaunchKernelGGL(k_mc_pairs, dim3(nchain), dim3(kWave), 3 * (size_t)a.max_atoms * sizeof(double), s, a);
  return hipGetLastError();
}

hipError_t launch_mc(const McArgs& a, int nblocks, int waves, bool rec_lds, hipStream_t s) {
  if (waves < 1 || waves > mc_max_waves(a)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_mc_reset_queue, dim3(1), dim3(1), 0, s, a.queue);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const size_t lds = mc_lds_bytes(a, waves, rec_lds);
  const int rec_bytes = (int)(mc_lds_bytes(a, waves, rec_lds) - mc_lds_bytes(a, waves, false));
  const dim3 g(nblocks), b(waves * kWave);
  const int key = mc_inter_kind(a) + (rec_lds ? 8 : 0) + (a.min_iters > 0 ? 16 : 0);
  switch (key) {
    case kMcInterAtom + 8:
      if (a.pool_slots > 0) hipLaunchKernelGGL((k_mc<true, kMcInterAtom, false, true>), g, b, lds, s, a, rec_bytes);
      else hipLaunchKernelGGL((k_mc<true, kMcInterAtom, false>), g, b, lds, s, a, rec_bytes);
      break;
    case kMcInterSub + 8: hipLaunchKernelGGL((k_mc<true, kMcInterSub, false>), g, b, lds, s, a, rec_bytes); break;
    case kMcInterF64 + 8: hipLaunchKernelGGL((k_mc<true, kMcInterF64, false>), g, b, lds, s, a, rec_bytes); break;
    case kMcInterAtom: hipLaunchKernelGGL((k_mc<false, kMcInterAtom, false>), g, b, lds, s, a, 0); break;
    case kMcInterSub: hipLaunchKernelGGL((k_mc<false, kMcInterSub, false>), g, b, lds, s, a, 0); break;
    case kMcInterF64: hipLaunchKernelGGL((k_mc<false, kMcInterF64, false>), g, b, lds, s, a, 0); break;
    case kMcInterGrid: hipLaunchKernelGGL((k_mc<false, kMcInterGrid, false>), g, b, lds, s, a, 0); break;
    // with local minimisation after every proposal
    case kMcInterAtom + 24: hipLaunchKernelGGL((k_mc<true, kMcInterAtom, true>), g, b, lds, s, a, rec_bytes); break;
    case kMcInterF64 + 24: hipLaunchKernelGGL((k_mc<true, kMcInterF64, true>), g, b, lds, s, a, rec_bytes); break;
    case kMcInterAtom + 16: hipLaunchKernelGGL((k_mc<false, kMcInterAtom, true>), g, b, lds, s, a, 0); break;
    case kMcInterF64 + 16: hipLaunchKernelGGL((k_mc<false, kMcInterF64, true>), g, b, lds, s, a, 0); break;
    case kMcInterGrid + 16: hipLaunchKernelGGL((k_mc<false, kMcInterGrid, true>), g, b, lds, s, a, 0); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace mmo
