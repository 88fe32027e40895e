// select_kernels.hip -- rigid-scan clash filters and top-k selection of scan energies.
//
// Clash filters (Lds.exhaustive_rigid_ligand_docking, src/lds.ml:1040-1114): a pose is
// skipped when its translation lies outside the ROI sphere or, for ligands whose
// centre is inside one of their atoms, on a voxel whose 8 corners are all protein vdW
// volume (G3D.vdW_clash_AND, src/G3D.ml:188-213), or when any atom has a protein-volume
// voxel among its 8 corners (Mol.protein_ligand_clash + G3D.vdW_clash_OR,
// src/mol.ml:1195-1206, src/G3D.ml:159-185).  Skipped poses get +inf.
//
// Top-k (the TopKeeper of src/lds.ml:1055-1064, :1110-1113, lowest energies first):
// an MSB-first radix select over order-preserving 64-bit keys of the energies narrows the
// k-th smallest key down by 13 bits a pass (at most 5 passes) until no more than
// topk_limit keys are at or below the prefix; those are gathered, and one workgroup sorts
// them by (energy, index) and keeps the first k.  Where more than that many keys are equal
// to the k-th, the passes resolve all 64 bits and the equal keys are taken in index order
// (so ties resolve to the lowest pose indices).  NaN sorts as the largest value.
//
// Bound: reading the energies (8 bytes each) once per pass and once to gather.  Measured,
// 36,864,000 energies and k = 100, against the byte-wise select (8 passes, 21 launches)
// before it: all but 500 +inf 732 -> 131 us, normally distributed 700 -> 169, in one
// thousandth of a binade 921 -> 248, seven distinct values 876 -> 530; 20,000 energies 118 ->
// 36 us and 1,000 energies 85 -> 26 us, where launches are all of it.
#include <cstdint>

#include "common.h"
#include "kernels.h"

namespace mmo {

// exclusive prefix sums of n counts in place, their total to *total: each thread scans a
// contiguous run, the run totals are scanned across the workgroup (st: the top-k's state,
// nothing to do once it is done)
__global__ void __launch_bounds__(1024) k_scan_counts(const TopkState* st, unsigned* cnt, int n,
                                                      unsigned* total) {
  __shared__ unsigned part[1024];
  if (st && st->done) return;
  const int t = threadIdx.x;
  const int per = (n + 1023) / 1024;
  const int b0 = min(n, t * per), b1 = min(n, b0 + per);
  unsigned sum = 0;
  for (int b = b0; b < b1; ++b) sum += cnt[b];
  part[t] = sum;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const unsigned v = t >= off ? part[t - off] : 0u;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  unsigned run = part[t] - sum;
  for (int b = b0; b < b1; ++b) {
    const unsigned c = cnt[b];
    cnt[b] = run;
    run += c;
  }
  if (total && t == 1023) *total = part[1023];
}

// ------------------------------------------------------------------ clash filter
// Both filters (energies of a finished scan; keep flags before scoring) are bound by the FP64
// position and cell test of each atom until all 64 poses of a wavefront have clashed; the
// +inf for every pose (8 bytes each) is written in their shade.  36.9 M poses of a 38-atom
// ligand, 71,000 kept: 381 us, against 1,774 us with 8 corner reads an atom, the rotation
// applied for every pose and the atoms in file order, and 417 us more for rocPRIM's flagged
// selection of the slots and the fill, now 25 us of counting and listing.

// The cells of the mask: bit v = (i, j, k) set when one of the 8 corners (i..i+1, j..j+1,
// k..k+1) is protein volume, so that an atom's 8-corner test (G3D.vdW_clash_OR) is one read.
// One thread per word; cells on the grid's upper faces are not asked for and stay 0.
__global__ void __launch_bounds__(256) k_mask_cells(const uint32_t* mask, uint32_t* cells, int nx,
                                                    int ny, int nz) {
  const size_t nvox = (size_t)nx * ny * nz;
  const size_t w = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= (nvox + 31) / 32) return;
  uint32_t out = 0;
  for (int b = 0; b < 32; ++b) {
    const size_t v = 32 * w + b;
    if (v >= nvox) break;
    const int i = (int)(v % nx), j = (int)((v / nx) % ny), k = (int)(v / ((size_t)nx * ny));
    if (i + 1 >= nx || j + 1 >= ny || k + 1 >= nz) continue;
    for (int c = 0; c < 8; ++c) {
      const size_t u = v + (c & 1) + (size_t)((c >> 1) & 1) * nx + (size_t)(c >> 2) * nx * ny;
      out |= ((mask[u >> 5] >> (u & 31)) & 1u) << b;
    }
  }
  cells[w] = out;
}

hipError_t launch_mask_cells(const uint32_t* mask, uint32_t* cells, int nx, int ny, int nz,
                             hipStream_t s) {
  const size_t words = ((size_t)nx * ny * nz + 31) / 32;
  hipLaunchKernelGGL(k_mask_cells, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, s, mask, cells,
                     nx, ny, nz);
  return hipGetLastError();
}

// Whether an atom at (x, y, z) has a protein-volume voxel among its 8 corners.  Corners
// outside the grid count as free: the conversion truncates as int_of_float and saturates,
// so 0 <= i < nx - 1 is the cell test (coordinates are finite, see clash_coord).
__device__ __forceinline__ uint32_t trunc_sat(double v) {
  int i;   // the instruction: a conversion out of int's range is undefined in C++
  asm("v_cvt_i32_f64 %0, %1" : "=v"(i) : "v"(v));
  return (uint32_t)i;
}
__device__ __forceinline__ uint32_t atom_cell(const ScanFilterArgs& a, double x, double y, double z) {
  const uint32_t i = trunc_sat((x - a.ox) * a.inv_step), j = trunc_sat((y - a.oy) * a.inv_step),
                 k = trunc_sat((z - a.oz) * a.inv_step);
  if (!(i < (uint32_t)a.nx - 1u && j < (uint32_t)a.ny - 1u && k < (uint32_t)a.nz - 1u)) return ~0u;
  return i + (uint32_t)a.nx * (j + (uint32_t)a.ny * k);   // fewer than 2^31 voxels
}
__device__ __forceinline__ bool cell_clash(const ScanFilterArgs& a, uint32_t v) {
  return v != ~0u && ((a.cells[v >> 5] >> (v & 31u)) & 1u) != 0u;
}
// a coordinate of the clash test: one that is not finite is outside every grid
__device__ __forceinline__ double clash_coord(double v) { return fabs(v) <= 1e300 ? v : 1e300; }

// A workgroup takes a.tiles x 64 slots of the scan's pose order, 64 per wavefront at a time
// (one 64-bit word of keep flags).  TILED (at least 64 translations): the slots of one
// rotation (workgroup = rotation, then its share of the translations), whose rotated atoms
// R c are formed once in LDS, so that a pose's atom costs three additions instead of the
// whole transform; else consecutive slots of any rotations, each lane forming its own.
// 32 tiles share the rotated atoms; scans that would fill fewer than 2,048 workgroups (8 a CU) so
// take fewer, down to one a wavefront: 40,000 poses of a 5-atom ligand 79 us with 32, 53 now, of 38
// atoms 94 and 63.
constexpr int kKeepTiles = 32;

template <bool TILED>
struct KeepSlots {
  int nrot, ntrans, size, per_rot;   // slots of a workgroup; workgroups per rotation (TILED)
  __device__ KeepSlots(const ScanFilterArgs& a)
      : nrot(a.nrot), ntrans(a.ntrans), size(64 * a.tiles), per_rot((a.ntrans + size - 1) / size) {}
  // slot `lane` of the workgroup's tile q: its rotation and translation slot; false: none
  __device__ bool at(int q, int lane, int& r, int& ts) const {
    if (TILED) {
      r = blockIdx.x / per_rot;
      ts = (blockIdx.x - r * per_rot) * size + q * 64 + lane;
      return ts < ntrans;
    }
    const size_t slot = (size_t)blockIdx.x * size + q * 64 + lane;
    if (slot >= (size_t)nrot * ntrans) return false;
    r = (int)(slot / ntrans);
    ts = (int)(slot - (size_t)r * ntrans);
    return true;
  }
};

// tperm: translation of each slot (nullptr: the slots are the poses themselves).  KEEP: one
// word of keep flags per tile to `words`, their number per workgroup to `count`, and every
// energy of the workgroup's linear share of e set to +inf; else +inf for the skipped poses.
template <bool TILED, bool KEEP>
__global__ void __launch_bounds__(256) k_scan_filter(ScanFilterArgs a, const int* tperm, uint64_t* words,
                                                     unsigned* count) {
  extern __shared__ double s_lig[];
  __shared__ unsigned s_count;
  const KeepSlots<TILED> slots(a);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t npose = (size_t)a.nrot * a.ntrans;
  if (KEEP) {
    if (threadIdx.x == 0) s_count = 0u;
    const size_t share = (npose + gridDim.x - 1) / gridDim.x;
    const size_t p1 = min(npose, (blockIdx.x + 1) * share);
    for (size_t p = blockIdx.x * share + threadIdx.x; p < p1; p += blockDim.x) a.e[p] = __builtin_inf();
  }
  if (a.atom_clash) {
    const double* R = a.rots + 9 * (size_t)(TILED ? blockIdx.x / slots.per_rot : 0);
    for (int j = threadIdx.x; j < a.n_atoms; j += blockDim.x) {
      const double* c = a.lig + 3 * (size_t)a.order[j];
      const double c0 = c[0], c1 = c[1], c2 = c[2];
      s_lig[3 * j] = TILED ? clash_coord(R[0] * c0 + R[1] * c1 + R[2] * c2) : c0;
      s_lig[3 * j + 1] = TILED ? clash_coord(R[3] * c0 + R[4] * c1 + R[5] * c2) : c1;
      s_lig[3 * j + 2] = TILED ? clash_coord(R[6] * c0 + R[7] * c1 + R[8] * c2) : c2;
    }
  }
  __syncthreads();
  for (int q = wave; q < a.tiles; q += 4) {
    int r = 0, ts = 0;
    const bool in = slots.at(q, lane, r, ts);
    if (__ballot(in) == 0ull) {
      if (KEEP && lane == 0) words[(size_t)blockIdx.x * a.tiles + q] = 0ull;
      continue;
    }
    const int t = in ? (tperm ? tperm[ts] : ts) : 0;
    bool keep = in && !a.skip[t];
    if (a.atom_clash && __ballot(keep) != 0ull) {
      const double* T = a.trans + 3 * (size_t)t;
      const double tx = clash_coord(T[0]), ty = clash_coord(T[1]), tz = clash_coord(T[2]);
      const double* R = a.rots + 9 * (size_t)r;
      // the pose's atom position as the scan kernel computes it
      auto cell = [&](int j) {
        const double c0 = s_lig[3 * j], c1 = s_lig[3 * j + 1], c2 = s_lig[3 * j + 2];
        if (TILED) return atom_cell(a, c0 + tx, c1 + ty, c2 + tz);
        return atom_cell(a, clash_coord(R[0] * c0 + R[1] * c1 + R[2] * c2) + tx,
                         clash_coord(R[3] * c0 + R[4] * c1 + R[5] * c2) + ty,
                         clash_coord(R[6] * c0 + R[7] * c1 + R[8] * c2) + tz);
      };
      // two atoms at a time: their reads of the mask overlap
      for (int j = 0; j < a.n_atoms; j += 2) {
        if (keep) {
          const uint32_t v0 = cell(j), v1 = j + 1 < a.n_atoms ? cell(j + 1) : ~0u;
          const bool h0 = cell_clash(a, v0), h1 = cell_clash(a, v1);
          keep = !(h0 || h1);
        }
        if (__ballot(keep) == 0ull) break;
      }
    }
    if (KEEP) {
      const uint64_t w = __ballot(keep);
      if (lane == 0) {
        words[(size_t)blockIdx.x * a.tiles + q] = w;
        if (w) atomicAdd(&s_count, (unsigned)__popcll(w));
      }
    } else if (in && !keep) {
      a.e[(size_t)r * a.ntrans + t] = __builtin_inf();
    }
  }
  if (KEEP) {
    __syncthreads();
    if (threadIdx.x == 0) count[blockIdx.x] = s_count;
  }
}

// the kept slots in the scan's order (consecutive kept poses stay in the scan's bricks):
// one wavefront per workgroup of k_scan_filter, from its first place `start`
template <bool TILED>
__global__ void __launch_bounds__(64) k_keep_list(ScanFilterArgs a, const uint64_t* words,
                                                  const unsigned* start, const unsigned* total, int* list) {
  const KeepSlots<TILED> slots(a);
  const int lane = threadIdx.x;
  const unsigned first = start[blockIdx.x];
  // nothing kept here: the next workgroup (or the end of the list) starts at the same place
  if ((blockIdx.x + 1 < gridDim.x ? start[blockIdx.x + 1] : *total) == first) return;
  unsigned base = first;
  const uint64_t mine = lane < a.tiles ? words[(size_t)blockIdx.x * a.tiles + lane] : 0ull;
  for (uint64_t any = __ballot(mine != 0ull); any; any &= any - 1) {
    const int q = __builtin_ctzll(any);
    const uint64_t w = __shfl((unsigned long long)mine, q, 64);
    int r, ts;
    const bool in = slots.at(q, lane, r, ts);
    if (in && ((w >> lane) & 1ull))
      list[base + __popcll(w & ((1ull << lane) - 1ull))] = r * a.ntrans + ts;
    base += (unsigned)__popcll(w);
  }
}

static size_t keep_groups(int nrot, int ntrans, int tiles) {
  const int size = 64 * tiles;
  return ntrans >= 64 ? (size_t)nrot * ((ntrans + size - 1) / size)
                      : ((size_t)nrot * ntrans + size - 1) / size;
}
int scan_keep_tiles(int nrot, int ntrans) {
  int tiles = kKeepTiles;
  while (tiles > 4 && keep_groups(nrot, ntrans, tiles) < 2048) tiles /= 2;
  return tiles;
}
size_t scan_keep_groups(int nrot, int ntrans) {
  return keep_groups(nrot, ntrans, scan_keep_tiles(nrot, ntrans));
}

template <bool TILED>
static hipError_t scan_filter_t(ScanFilterArgs a, const int* tperm, const KeepScratch* w, hipStream_t s) {
  a.tiles = scan_keep_tiles(a.nrot, a.ntrans);
  const size_t groups = scan_keep_groups(a.nrot, a.ntrans);
  const size_t lds = a.atom_clash ? (size_t)3 * a.n_atoms * sizeof(double) : 0;
  if (!w) {
    hipLaunchKernelGGL((k_scan_filter<TILED, false>), dim3((unsigned)groups), dim3(256), lds, s, a, tperm,
                       (uint64_t*)nullptr, (unsigned*)nullptr);
    return hipGetLastError();
  }
  hipLaunchKernelGGL((k_scan_filter<TILED, true>), dim3((unsigned)groups), dim3(256), lds, s, a, tperm,
                     w->words, w->count);
  hipLaunchKernelGGL(k_scan_counts, dim3(1), dim3(1024), 0, s, (const TopkState*)nullptr, w->count,
                     (int)groups, w->total);
  hipLaunchKernelGGL((k_keep_list<TILED>), dim3((unsigned)groups), dim3(64), 0, s, a, w->words, w->count,
                     w->total, w->list);
  return hipGetLastError();
}

hipError_t launch_scan_keep(const ScanFilterArgs& a, const int* tperm, const KeepScratch& w,
                            hipStream_t s) {
  if ((size_t)a.nrot * a.ntrans == 0) return hipSuccess;
  return a.ntrans >= 64 ? scan_filter_t<true>(a, tperm, &w, s) : scan_filter_t<false>(a, tperm, &w, s);
}

hipError_t launch_scan_filter(const ScanFilterArgs& a, hipStream_t s) {
  if ((size_t)a.nrot * a.ntrans == 0) return hipSuccess;
  return a.ntrans >= 64 ? scan_filter_t<true>(a, nullptr, nullptr, s)
                        : scan_filter_t<false>(a, nullptr, nullptr, s);
}

// -------------------------------------------------------------------- top-k
__device__ __forceinline__ uint64_t order_key(double v) {
  if (v != v) return ~0ull;
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

constexpr int kTopkThreads = 1024;
// digit widths: sign, exponent and the first bit of the mantissa, then the mantissa
constexpr int kTopkBits[kTopkPasses] = {13, 13, 13, 13, 12};
constexpr int kTopkBins = kTopkHist / kTopkPasses;

// f(energy, valid, index) for every energy, each lane a stride apart, four reads in flight;
// all lanes of a wavefront call f together
template <class F>
__device__ __forceinline__ void topk_walk(const double* e, size_t n, F&& f) {
  constexpr int U = 4;
  const size_t stride = (size_t)gridDim.x * kTopkThreads;
  size_t b = (size_t)blockIdx.x * kTopkThreads;   // the workgroup's first index of a round
  size_t i0 = b + threadIdx.x;
  for (; b + (U - 1) * stride + kTopkThreads <= n; b += U * stride, i0 += U * stride) {
    double v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = e[i0 + u * stride];
#pragma unroll
    for (int u = 0; u < U; ++u) f(v[u], true, i0 + u * stride);
  }
  for (; b < n; b += stride, i0 += stride) f(i0 < n ? e[i0] : 0.0, i0 < n, i0);
}

// The select's state after the digit counted in `hist` (bits wide, at shift): that of the
// k-th smallest key appended to the prefix.  Every workgroup of the next kernel computes it
// for itself, so no launch waits for a single workgroup in between and no kernel fences (a
// release to the whole device in every workgroup, with the last one picking the digit, cost
// 40 us a pass).  s: LDS for kTopkThreads / 64 + 8 words of 64 bits.
__device__ TopkState topk_next(const TopkState& p, const unsigned* hist, int shift, int bits,
                               uint64_t* s) {
  if (p.done) return p;
  constexpr int per = kTopkBins / kTopkThreads, nw = kTopkThreads / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint4* h4 = reinterpret_cast<const uint4*>(hist + tid * per);
  static_assert(per == 8, "two 16-byte reads of counts per thread");
  const uint4 lo = h4[0], hi = h4[1];
  const unsigned cnt[per] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  uint64_t mine = 0;
#pragma unroll
  for (int q = 0; q < per; ++q) mine += cnt[q];
  uint64_t incl = mine;
  for (int off = 1; off < 64; off <<= 1) {
    const uint64_t v = __shfl_up((unsigned long long)incl, off, 64);
    if (lane >= off) incl += v;
  }
  if (lane == 63) s[wave] = incl;
  __syncthreads();
  uint64_t cum = incl - mine;
  for (int w = 0; w < wave; ++w) cum += s[w];
  if (cum < p.rem && p.rem <= cum + mine) {   // one thread: 1 <= rem <= matching keys
    for (int q = 0; q < per; ++q) {
      if (p.rem <= cum + cnt[q]) {
        s[nw] = (uint64_t)(tid * per + q);
        s[nw + 1] = p.rem - cum;
        s[nw + 2] = cnt[q];
        break;
      }
      cum += cnt[q];
    }
  }
  __syncthreads();
  TopkState r = p;
  r.prefix |= s[nw] << shift;
  r.mask |= (uint64_t)((1 << bits) - 1) << shift;
  r.rem = s[nw + 1];
  // keys below the prefix: k - rem
  r.done = p.k - r.rem + s[nw + 2] <= (uint64_t)p.limit ? 1u : 0u;
  return r;
}

__global__ void k_topk_init(TopkState* st, unsigned* hist, unsigned* count, uint64_t k, unsigned limit) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    st[0] = TopkState{0ull, 0ull, k, k, limit, 0u};
    *count = 0u;
  }
  if (i < kTopkHist) hist[i] = 0u;
}

// One digit of the select: the digits at `shift` of the keys that match the prefix so far
// are counted in LDS, then added to this pass's counts.  Nothing is done once the keys at or
// below the prefix fit the candidate list.
__global__ void __launch_bounds__(kTopkThreads) k_topk_pass(const double* e, size_t n, TopkState* st,
                                                            unsigned* hist, int pass, int shift,
                                                            int bits, int prev_shift, int prev_bits) {
  __shared__ unsigned h[kTopkBins];
  __shared__ uint64_t s[kTopkThreads / 64 + 8];
  const int tid = threadIdx.x, lane = tid & 63, nb = 1 << bits;
  TopkState cur = st[pass > 0 ? pass - 1 : 0];
  if (pass > 0) {
    cur = topk_next(cur, hist + (pass - 1) * kTopkBins, prev_shift, prev_bits, s);
    if (blockIdx.x == 0 && tid == 0) st[pass] = cur;
  }
  if (cur.done) return;
  for (int i = tid; i < nb; i += kTopkThreads) h[i] = 0u;
  __syncthreads();
  topk_walk(e, n, [&](double v, bool in, size_t) {
    const uint64_t key = order_key(v);
    const int d = (int)(key >> shift) & (nb - 1);
    uint64_t act = __ballot(in && (key & cur.mask) == cur.prefix);
    // a digit that many lanes share (filtered scans are nearly all +inf) is added once
    while (act) {
      const int first = __builtin_ctzll(act), d0 = __builtin_amdgcn_readlane(d, first);
      const uint64_t same = __ballot(d == d0) & act;
      if (__popcll(same) < 8) break;
      if (lane == first) atomicAdd(&h[d0], (unsigned)__popcll(same));
      act &= ~same;
    }
    if ((act >> lane) & 1ull) atomicAdd(&h[d], 1u);
  });
  __syncthreads();
  unsigned* mine = hist + pass * kTopkBins;
  for (int i = tid; i < nb; i += kTopkThreads)
    if (h[i]) atomicAdd(&mine[i], h[i]);
}

// the candidates, in any order: every key at or below the prefix, or (ties beyond the list)
// the k - rem keys below the fully resolved one
__global__ void __launch_bounds__(kTopkThreads) k_topk_gather(const double* e, size_t n, TopkState* st,
                                                              const unsigned* hist, int prev_bits,
                                                              unsigned* count, double* cand_e,
                                                              int64_t* cand_i) {
  __shared__ uint64_t s[kTopkThreads / 64 + 8];
  const TopkState cur = topk_next(st[kTopkPasses - 1], hist + (kTopkPasses - 1) * kTopkBins, 0,
                                  prev_bits, s);
  if (blockIdx.x == 0 && threadIdx.x == 0) st[kTopkPasses] = cur;
  const bool done = cur.done != 0u;
  const uint64_t T = done ? (cur.prefix | ~cur.mask) : cur.prefix;
  topk_walk(e, n, [&](double v, bool in, size_t i) {
    const uint64_t key = order_key(v);
    if (in && (done ? key <= T : key < T)) {
      const unsigned p = atomicAdd(count, 1u);
      if (p < (unsigned)kTopkCand) {
        cand_e[p] = v;
        cand_i[p] = (int64_t)i;
      }
    }
  });
}

// ties beyond the candidate list: keys equal to the threshold, counted per chunk of `chunk`
// consecutive indices
__global__ void __launch_bounds__(64) k_topk_eq_count(const double* e, size_t n, size_t chunk, int nb,
                                                      const TopkState* st, unsigned* bcnt) {
  if (st->done) return;
  const uint64_t T = st->prefix;
  for (int b = blockIdx.x; b < nb; b += gridDim.x) {
    const size_t b0 = (size_t)b * chunk, b1 = min(n, b0 + chunk);
    unsigned c = 0;
    for (size_t i = b0 + threadIdx.x; i < b1; i += 64) c += order_key(e[i]) == T ? 1u : 0u;
    for (int off = 1; off < 64; off <<= 1) c += __shfl_xor(c, off, 64);
    if (threadIdx.x == 0) bcnt[b] = c;
  }
}

// the first st->rem equal keys in index order go after the k - st->rem smaller ones
__global__ void __launch_bounds__(64) k_topk_eq_write(const double* e, size_t n, size_t chunk, int nb,
                                                      const TopkState* st, const unsigned* bcnt,
                                                      double* cand_e, int64_t* cand_i) {
  if (st->done) return;
  const uint64_t T = st->prefix, take = st->rem, k = st->k;
  const int lane = threadIdx.x;
  for (int b = blockIdx.x; b < nb; b += gridDim.x) {
    const size_t b0 = (size_t)b * chunk, b1 = min(n, b0 + chunk);
    uint64_t base = bcnt[b];
    for (size_t s0 = b0; s0 < b1 && base < take; s0 += 64) {
      const size_t i = s0 + lane;
      const bool f = i < b1 && order_key(e[i]) == T;
      const uint64_t m = __ballot(f);
      const uint64_t below = lane ? (m & ((1ull << lane) - 1ull)) : 0ull;
      const uint64_t rank = base + (uint64_t)__popcll(below);
      if (f && rank < take) {
        const uint64_t p = (k - take) + rank;
        cand_e[p] = e[i];
        cand_i[p] = (int64_t)i;
      }
      base += (uint64_t)__popcll(m);
    }
  }
}

// one workgroup: bitonic sort of the candidates by (energy key, index), the first k out.
// With `e` (n <= kTopkCand) the candidates are the energies themselves.
__global__ void __launch_bounds__(1024) k_topk_sort(const TopkState* st, const unsigned* count,
                                                    const double* cand_e, const int64_t* cand_i,
                                                    const double* e, int n, int k, double* out_e,
                                                    int64_t* out_i) {
  extern __shared__ __align__(16) uint64_t s_topk[];
  const int c = e ? n : st->done ? (int)min(*count, (unsigned)kTopkCand) : k;
  int n2 = 1;
  while (n2 < c) n2 <<= 1;
  uint64_t* sk = s_topk;
  int64_t* si = reinterpret_cast<int64_t*>(sk + n2);
  for (int i = threadIdx.x; i < n2; i += blockDim.x) {
    sk[i] = i < c ? order_key(e ? e[i] : cand_e[i]) : ~0ull;
    si[i] = i < c ? (e ? (int64_t)i : cand_i[i]) : INT64_MAX;
  }
  __syncthreads();
  for (int size = 2; size <= n2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = threadIdx.x; i < n2; i += blockDim.x) {
        const int j = i ^ stride;
        if (j > i) {
          const bool up = (i & size) == 0;
          const bool gt = sk[i] > sk[j] || (sk[i] == sk[j] && si[i] > si[j]);
          if (gt == up) {
            const uint64_t tk = sk[i]; sk[i] = sk[j]; sk[j] = tk;
            const int64_t ti = si[i]; si[i] = si[j]; si[j] = ti;
          }
        }
      }
      __syncthreads();
    }
  }
  for (int i = threadIdx.x; i < k; i += blockDim.x) {
    const uint64_t kk = sk[i];
    const uint64_t b = (kk >> 63) ? (kk & 0x7FFFFFFFFFFFFFFFull) : ~kk;
    out_e[i] = kk == ~0ull ? __builtin_nan("") : __longlong_as_double((long long)b);
    out_i[i] = si[i];
  }
}

// The sort of the candidates takes 25, 45 and 91 us for 1,024, 2,048 and 4,096 of them, a pass 6
// us up to some 4 M energies and 60 us for 36.9 M: few energies (or, for large k, as many as the
// list holds) are sorted at once, and up to 4 M the passes go on until they have left 1,024 (or
// k) candidates, beyond until the list holds them.  20,000 energies of seven values, k = 1 or 100:
// 159 us with 4,096, 75 and 84 now; 4,096 energies, k = 1, sorted at once 112 to 121, 75 to 80
// by passes; 3,000,000 normally distributed, k = 100, 196 and 75.
constexpr int kTopkSort = 2048;
static unsigned topk_limit(size_t n, int k) {
  return n <= ((size_t)1 << 22) ? std::max(1024, k) : kTopkCand;
}

hipError_t launch_topk(const double* e, size_t n, int k, double* out_e, int64_t* out_i,
                       TopkScratch w, hipStream_t s) {
  if (k <= 0 || n == 0) return hipSuccess;
  // LDS: kTopkCand keys and indices (64 KiB, the most a launch may ask for without the
  // kernel's limit being raised)
  constexpr size_t lds = (size_t)kTopkCand * (sizeof(uint64_t) + sizeof(int64_t));
  if (n <= (size_t)kTopkSort || (n <= (size_t)kTopkCand && k > kTopkSort / 2)) {
    hipLaunchKernelGGL(k_topk_sort, dim3(1), dim3(1024), lds, s, w.st, w.count, w.cand_e, w.cand_i, e,
                       (int)n, k, out_e, out_i);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_topk_init, dim3(kTopkHist / 1024), dim3(1024), 0, s, w.st, w.hist, w.count,
                     (uint64_t)k, topk_limit(n, k));
  const int blocks = (int)std::min<size_t>(512, (n + 4 * kTopkThreads - 1) / (4 * kTopkThreads));
  int shift = 64;
  for (int p = 0; p < kTopkPasses; ++p) {
    const int prev = shift;
    shift -= kTopkBits[p];
    hipLaunchKernelGGL(k_topk_pass, dim3(blocks), dim3(kTopkThreads), 0, s, e, n, w.st, w.hist, p, shift,
                       kTopkBits[p], prev, p > 0 ? kTopkBits[p - 1] : 0);
  }
  hipLaunchKernelGGL(k_topk_gather, dim3(blocks), dim3(kTopkThreads), 0, s, e, n, w.st, w.hist,
                     kTopkBits[kTopkPasses - 1], w.count, w.cand_e, w.cand_i);
  const TopkState* fin = w.st + kTopkPasses;
  const int nb = (int)((n + w.chunk - 1) / w.chunk);
  const int eq_blocks = std::min(nb, 2048);
  hipLaunchKernelGGL(k_topk_eq_count, dim3(eq_blocks), dim3(64), 0, s, e, n, w.chunk, nb, fin, w.bcnt);
  hipLaunchKernelGGL(k_scan_counts, dim3(1), dim3(1024), 0, s, fin, w.bcnt, nb, (unsigned*)nullptr);
  hipLaunchKernelGGL(k_topk_eq_write, dim3(eq_blocks), dim3(64), 0, s, e, n, w.chunk, nb, fin, w.bcnt,
                     w.cand_e, w.cand_i);
  hipLaunchKernelGGL(k_topk_sort, dim3(1), dim3(1024), lds, s, fin, w.count, w.cand_e, w.cand_i,
                     (const double*)nullptr, 0, k, out_e, out_i);
  return hipGetLastError();
}

}  // namespace mmo
