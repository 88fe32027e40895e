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
// kTopkCand keys are at or below the prefix; those are gathered, and one workgroup sorts
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

#include <hipcub/hipcub.hpp>

#include "common.h"
#include "kernels.h"

namespace mmo {

// ------------------------------------------------------------------ clash filter
// whether an atom of pose (rotation r, translation t) has a protein-volume voxel among its
// 8 corners (Mol.protein_ligand_clash); s_lig: the centred conformer rows
__device__ bool pose_atom_clash(const ScanFilterArgs& a, const double* s_lig, int r, int t) {
  const double* R = a.rots + 9 * (size_t)r;
  const double* T = a.trans + 3 * (size_t)t;
  const size_t nxy = (size_t)a.nx * a.ny;
  for (int j = 0; j < a.n_atoms; ++j) {
    const double* c = s_lig + 3 * j;
    // the pose's atom position as the scan kernel computes it
    const double x = R[0] * c[0] + R[1] * c[1] + R[2] * c[2] + T[0];
    const double y = R[3] * c[0] + R[4] * c[1] + R[5] * c[2] + T[1];
    const double z = R[6] * c[0] + R[7] * c[1] + R[8] * c[2] + T[2];
    const double fx = (x - a.ox) * a.inv_step, fy = (y - a.oy) * a.inv_step,
                 fz = (z - a.oz) * a.inv_step;
    // corners outside the grid count as free (bounds checked in floating point first)
    if (!(fx > -1.0 && fy > -1.0 && fz > -1.0 && fx < (double)(a.nx - 1) &&
          fy < (double)(a.ny - 1) && fz < (double)(a.nz - 1)))
      continue;
    const int i0 = (int)fx, j0 = (int)fy, k0 = (int)fz;   // truncation, as int_of_float
    bool hit = false;
#pragma unroll
    for (int cidx = 0; cidx < 8; ++cidx) {
      const size_t v = (size_t)(i0 + (cidx & 1)) + (size_t)(j0 + ((cidx >> 1) & 1)) * a.nx +
                       (size_t)(k0 + (cidx >> 2)) * nxy;
      hit |= ((a.mask[v >> 5] >> (v & 31)) & 1u) != 0u;
    }
    if (hit) return true;
  }
  return false;
}

__global__ void __launch_bounds__(256) k_scan_filter(ScanFilterArgs a) {
  extern __shared__ double s_lig[];
  for (int i = threadIdx.x; i < 3 * a.n_atoms; i += blockDim.x) s_lig[i] = a.lig[i];
  __syncthreads();
  const size_t pose = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (pose >= (size_t)a.nrot * a.ntrans) return;
  const int r = (int)(pose / a.ntrans), t = (int)(pose - (size_t)r * a.ntrans);
  if (a.skip[t] || (a.atom_clash && pose_atom_clash(a, s_lig, r, t))) a.e[pose] = __builtin_inf();
}

// filter before scoring: the same tests, as keep flags over the scan's pose order
__global__ void __launch_bounds__(256) k_scan_keep(ScanFilterArgs a, const int* tperm, uint8_t* keep) {
  extern __shared__ double s_lig[];
  for (int i = threadIdx.x; i < 3 * a.n_atoms; i += blockDim.x) s_lig[i] = a.lig[i];
  __syncthreads();
  const size_t slot = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (slot >= (size_t)a.nrot * a.ntrans) return;
  const int r = (int)(slot / a.ntrans);
  const int t = tperm[slot - (size_t)r * a.ntrans];
  keep[slot] = (a.skip[t] || (a.atom_clash && pose_atom_clash(a, s_lig, r, t))) ? 0 : 1;
}

hipError_t launch_scan_keep(const ScanFilterArgs& a, const int* tperm, uint8_t* keep, hipStream_t s) {
  const size_t n = (size_t)a.nrot * a.ntrans;
  if (n == 0) return hipSuccess;
  const size_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(k_scan_keep, dim3((unsigned)blocks), dim3(256),
                     (size_t)3 * a.n_atoms * sizeof(double), s, a, tperm, keep);
  return hipGetLastError();
}

hipError_t select_flagged_slots(const uint8_t* flags, int n, int* out, int* n_out, void* temp,
                                size_t* temp_bytes, hipStream_t s) {
  return hipcub::DeviceSelect::Flagged(temp, *temp_bytes, hipcub::CountingInputIterator<int>(0),
                                       flags, out, n_out, n, s);
}

hipError_t launch_scan_filter(const ScanFilterArgs& a, hipStream_t s) {
  const size_t n = (size_t)a.nrot * a.ntrans;
  if (n == 0) return hipSuccess;
  const size_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(k_scan_filter, dim3((unsigned)blocks), dim3(256),
                     (size_t)3 * a.n_atoms * sizeof(double), s, a);
  return hipGetLastError();
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
  r.done = p.k - r.rem + s[nw + 2] <= (uint64_t)kTopkCand ? 1u : 0u;
  return r;
}

__global__ void k_topk_init(TopkState* st, unsigned* hist, unsigned* count, uint64_t k) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    st[0] = TopkState{0ull, 0ull, k, k, 0u, 0u};
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

// exclusive prefix sum of the per-chunk counts: each thread scans a contiguous run of
// chunks, the run totals are scanned across the workgroup
__global__ void __launch_bounds__(1024) k_topk_eq_scan(const TopkState* st, unsigned* bcnt, int nb) {
  __shared__ unsigned part[1024];
  if (st->done) return;
  const int t = threadIdx.x;
  const int per = (nb + 1023) / 1024;
  const int b0 = min(nb, t * per), b1 = min(nb, b0 + per);
  unsigned sum = 0;
  for (int b = b0; b < b1; ++b) sum += bcnt[b];
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
    const unsigned c = bcnt[b];
    bcnt[b] = run;
    run += c;
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

hipError_t launch_topk(const double* e, size_t n, int k, double* out_e, int64_t* out_i,
                       TopkScratch w, hipStream_t s) {
  if (k <= 0 || n == 0) return hipSuccess;
  // LDS: kTopkCand keys and indices (64 KiB, the most a launch may ask for without the
  // kernel's limit being raised)
  constexpr size_t lds = (size_t)kTopkCand * (sizeof(uint64_t) + sizeof(int64_t));
  if (n <= (size_t)kTopkCand) {
    hipLaunchKernelGGL(k_topk_sort, dim3(1), dim3(1024), lds, s, w.st, w.count, w.cand_e, w.cand_i, e,
                       (int)n, k, out_e, out_i);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_topk_init, dim3(kTopkHist / 1024), dim3(1024), 0, s, w.st, w.hist, w.count,
                     (uint64_t)k);
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
  hipLaunchKernelGGL(k_topk_eq_scan, dim3(1), dim3(1024), 0, s, fin, w.bcnt, nb);
  hipLaunchKernelGGL(k_topk_eq_write, dim3(eq_blocks), dim3(64), 0, s, e, n, w.chunk, nb, fin, w.bcnt,
                     w.cand_e, w.cand_i);
  hipLaunchKernelGGL(k_topk_sort, dim3(1), dim3(1024), lds, s, fin, w.count, w.cand_e, w.cand_i,
                     (const double*)nullptr, 0, k, out_e, out_i);
  return hipGetLastError();
}

}  // namespace mmo
