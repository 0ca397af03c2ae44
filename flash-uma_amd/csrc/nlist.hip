// Capped periodic radius graph on the GPU (the FAIRChem a2g graph the reference takes as
// input, readme.md:34), with the exact definition of the host builder in systems.py:
//
//   for receiver j, candidates (i, o), o an integer cell offset (0 on non-periodic axes),
//   (i, o) != (j, 0);  d = (pos_i - pos_j) + ((o0 c0 + o1 c1) + o2 c2) in float64 from the
//   float32 inputs;  |d|^2 = (dx dx + dy dy) + dz dz < cutoff^2;  ordered by
//   (|d|^2, i, o0, o1, o2);  the first max_neighbors kept;  edges grouped by receiver.
//
// Every float64 operation is written out in that order with contraction disabled, so the
// graph is bit-identical to the host one (same edges, same order, same offsets).
//
// Pipeline: (1) fu_nlist_bin: fractional coordinates -> wrapped cell-list bin + wrap count
// per atom; atoms are then sorted by bin (fu_sort_pairs_i64) and bin ranges found
// (fu_csr_row_ptr).  Bins are at least cutoff + 1e-3 wide, so with `reach` bins searched
// per side every neighbour is visited exactly once per periodic image.  (2) fu_nlist_search:
// one wave per receiver reads the ranges of the neighbouring bins, one a lane, tests the atoms in them
// 64 at a time across bins, appends hits to an LDS list (ballot + prefix count), then ranks the list
// by the ordering key (each entry's rank = number of smaller keys; keys are unique) and writes the
// first max_neighbors.  Bound by latency: bin by bin, a receiver of 27 bins of about ten atoms waited
// for three dependent loads at each, 233 us for 20,000 atoms; 64 candidates at a time 137, and 107
// with an entry of the list in one LDS read and no branch where distances are equal.
// (3) fu_nlist_scan: exclusive scan of the per-receiver counts (20,000 of them: 8 us, 28 by one
// workgroup).
// (4) fu_nlist_emit: edge_index (2, E) int64 and cell_offsets (E, 3) float32.
#include "fu_common.h"

namespace fu {

constexpr int NL_CAP = 512;  // hits held per receiver (the host checks the counts against it)

struct NLGeom {
  double cell[9];   // lattice vectors as rows, float64 copies of the float32 cell
  double inv[9];    // inverse of cell (fractional coordinates s = pos inv)
  int nb[3];        // bins per axis
  int reach[3];     // bins searched on each side (0 on non-periodic axes)
  int pbc[3];
  double cut2;      // cutoff * cutoff
};

__device__ __forceinline__ int floor_div(int a, int n) { return a >= 0 ? a / n : -((-a + n - 1) / n); }

__global__ __launch_bounds__(256) void nlist_bin_kernel(const float* __restrict__ pos, NLGeom g, int64_t N,
                                                        int64_t* __restrict__ bin_key, int32_t* __restrict__ wrap) {
  for (int64_t a = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; a < N; a += (int64_t)gridDim.x * blockDim.x) {
    const double p[3] = {(double)pos[3 * a], (double)pos[3 * a + 1], (double)pos[3 * a + 2]};
    int b[3];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
      double s = p[0] * g.inv[ax] + p[1] * g.inv[3 + ax] + p[2] * g.inv[6 + ax];
      int w = 0;
      if (g.pbc[ax]) {
        const double f = floor(s);
        w = (int)f;
        s -= f;
        int bb = (int)floor(s * g.nb[ax]);
        b[ax] = bb < 0 ? 0 : (bb >= g.nb[ax] ? g.nb[ax] - 1 : bb);
      } else {
        b[ax] = 0;
      }
      wrap[3 * a + ax] = w;
    }
    bin_key[a] = ((int64_t)b[0] * g.nb[1] + b[1]) * g.nb[2] + b[2];
  }
}

// d and |d|^2 in the host's operation order, each operation rounded separately.
__device__ __forceinline__ double pair_d2(const double* pi, const double* pj, const int* o, const double* cell) {
#pragma clang fp contract(off)
  double d[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double sh = ((double)o[0] * cell[a] + (double)o[1] * cell[3 + a]) + (double)o[2] * cell[6 + a];
    d[a] = (pi[a] - pj[a]) + sh;
  }
  return (d[0] * d[0] + d[1] * d[1]) + d[2] * d[2];
}

__global__ __launch_bounds__(256) void nlist_search_kernel(
    const float* __restrict__ pos, const int64_t* __restrict__ sorted_atoms, const int32_t* __restrict__ bin_ptr,
    const int32_t* __restrict__ wrap, const int64_t* __restrict__ bin_key, NLGeom g, int64_t N, int32_t K,
    int32_t* __restrict__ out_sender, int32_t* __restrict__ out_off, int32_t* __restrict__ count,
    int32_t* __restrict__ nout) {
  // hits: d^2 and (i << 24) | (o0 + 128) << 16 | (o1 + 128) << 8 | (o2 + 128), side by side so that an
  // entry is one LDS read
  struct __attribute__((aligned(16))) Hit {
    double d2;
    uint64_t key;
  };
  __shared__ Hit s_hit[4][NL_CAP];
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int64_t j = (int64_t)blockIdx.x * 4 + w;
  const bool active = j < N;
  int cnt = 0;  // wave-uniform
  if (active) {
    const double pj[3] = {(double)pos[3 * j], (double)pos[3 * j + 1], (double)pos[3 * j + 2]};
    const int wj[3] = {wrap[3 * j], wrap[3 * j + 1], wrap[3 * j + 2]};
    const int64_t kj = bin_key[j];
    const int bj[3] = {(int)(kj / ((int64_t)g.nb[1] * g.nb[2])), (int)((kj / g.nb[2]) % g.nb[1]), (int)(kj % g.nb[2])};
    const int ny = 2 * g.reach[1] + 1, nz = 2 * g.reach[2] + 1, total = (2 * g.reach[0] + 1) * ny * nz;
    const int per = N < (1 << 25) ? 64 : 1;   // bins a time: their candidates are counted in 32 bits
    for (int q0 = 0; q0 < total; q0 += per) {
      // a bin per lane: its image, its first atom and, summed over the lanes before, its first
      // candidate; the candidates of the 64 bins are then taken 64 at a time whatever bin they are
      // in, so one receiver waits for its loads about every 64 candidates and not at every bin
      const int q = q0 + lane;
      int kk[3] = {0, 0, 0}, lo = 0, len = 0;
      if (lane < per && q < total) {
        const int u[3] = {bj[0] + q / (ny * nz) - g.reach[0], bj[1] + (q / nz) % ny - g.reach[1], bj[2] + q % nz - g.reach[2]};
        int nbn[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          kk[a] = floor_div(u[a], g.nb[a]);
          nbn[a] = u[a] - kk[a] * g.nb[a];
        }
        const int64_t bin = ((int64_t)nbn[0] * g.nb[1] + nbn[1]) * g.nb[2] + nbn[2];
        lo = bin_ptr[bin];
        len = bin_ptr[bin + 1] - lo;
      }
      int first = len;
#pragma unroll
      for (int s = 1; s < 64; s <<= 1) {
        const int v = __shfl_up(first, s, 64);
        if (lane >= s) first += v;
      }
      const int cands = __shfl(first, 63, 64);
      first -= len;
      // candidate c: the last bin whose first candidate is at or before c (empty bins share theirs with
      // the next one, which is later)
      auto bin_of = [&](int64_t c) {
        int p = 0;
#pragma unroll
        for (int s = 32; s > 0; s >>= 1)
          if (__shfl(first, p + s, 64) <= c) p += s;
        return p;
      };
      auto atom_of = [&](int64_t c, int p) {
        const int64_t at = __shfl(lo, p, 64) + c - __shfl(first, p, 64);
        return c < cands ? sorted_atoms[at] : (int64_t)0;
      };
      int p = bin_of(lane);
      int64_t i = atom_of(lane, p);
      for (int64_t c0 = 0; c0 < cands; c0 += 64) {
        const int pn = bin_of(c0 + 64 + lane);
        const int64_t in = atom_of(c0 + 64 + lane, pn);   // the next candidates' atoms, one step ahead
        const int kc[3] = {__shfl(kk[0], p, 64), __shfl(kk[1], p, 64), __shfl(kk[2], p, 64)};
        bool hit = false;
        double d2 = 0.0;
        uint64_t key = 0;
        if (c0 + lane < cands) {
          int o[3];
#pragma unroll
          for (int a = 0; a < 3; ++a) o[a] = g.pbc[a] ? kc[a] - wrap[3 * i + a] + wj[a] : 0;
          const bool self = (i == j) && o[0] == 0 && o[1] == 0 && o[2] == 0;
          const double pi[3] = {(double)pos[3 * i], (double)pos[3 * i + 1], (double)pos[3 * i + 2]};
          d2 = pair_d2(pi, pj, o, g.cell);
          hit = !self && d2 < g.cut2;
          key = ((uint64_t)i << 24) | ((uint64_t)(o[0] + 128) << 16) | ((uint64_t)(o[1] + 128) << 8) |
                (uint64_t)(o[2] + 128);
        }
        const uint64_t mask = __ballot(hit);
        const int slot = cnt + __popcll(mask & ((1ull << lane) - 1ull));
        if (hit && slot < NL_CAP) s_hit[w][slot] = Hit{d2, key};
        cnt += __popcll(mask);
        p = pn;
        i = in;
      }
    }
  }
  __syncthreads();
  if (!active) return;
  const int n = cnt < NL_CAP ? cnt : NL_CAP;
  // two entries per lane and walk of the list
  for (int e0 = 0; e0 < n; e0 += 128) {
    double de[2];
    uint64_t ke[2];
    int rank[2] = {0, 0};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int e = e0 + 64 * h + lane;
      const Hit x = s_hit[w][e < n ? e : 0];
      de[h] = x.d2;
      ke[h] = x.key;
    }
    // no branch on equal distances: an entry always meets itself, and lattices are full of them
#pragma unroll 4
    for (int f = 0; f < n; ++f) {
      const Hit x = s_hit[w][f];
#pragma unroll
      for (int h = 0; h < 2; ++h) rank[h] += (int)(x.d2 < de[h]) | ((int)(x.d2 == de[h]) & (int)(x.key < ke[h]));
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (e0 + 64 * h + lane < n && rank[h] < K) {
        const int64_t slot = j * K + rank[h];
        out_sender[slot] = (int32_t)(ke[h] >> 24);
        out_off[3 * slot + 0] = (int)((ke[h] >> 16) & 0xff) - 128;
        out_off[3 * slot + 1] = (int)((ke[h] >> 8) & 0xff) - 128;
        out_off[3 * slot + 2] = (int)(ke[h] & 0xff) - 128;
      }
    }
  }
  if (lane == 0) {
    count[j] = cnt;
    nout[j] = n < K ? n : K;
  }
}

// Exclusive scan of nout into row_ptr (N + 1 entries, row_ptr[N] = E).  Up to 256 workgroups, each with
// a span of whole 1,024s: a workgroup sums the counts before its span (coalesced, from the L2)
// instead of waiting for the workgroups before it, then scans its span 1,024 at a time.
__global__ __launch_bounds__(1024) void nlist_scan_kernel(const int32_t* __restrict__ nout, int64_t* __restrict__ row_ptr,
                                                          int64_t N, int64_t span) {
  __shared__ int64_t s_base[16], s_sum[2][16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t b0 = (int64_t)blockIdx.x * span, b1 = b0 + span < N ? b0 + span : N;
  int64_t base = 0;
  for (int64_t m = t; m < b0; m += 1024) base += nout[m];
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) base += __shfl_xor(base, s, 64);
  if (lane == 0) s_base[wave] = base;
  __syncthreads();
  int64_t before = 0;
#pragma unroll
  for (int v = 0; v < 16; ++v) before += s_base[v];
  int buf = 0;
  for (int64_t k0 = b0; k0 < b1; k0 += 1024, buf ^= 1) {
    const int64_t k = k0 + t, own = k < b1 ? nout[k] : 0;
    int64_t run = own;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
      const int64_t v = __shfl_up(run, s, 64);
      if (lane >= s) run += v;
    }
    if (lane == 63) s_sum[buf][wave] = run;
    __syncthreads();   // the other buffer's readers are past the previous tile's barrier
    int64_t prior = 0, all = 0;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      prior += v < wave ? s_sum[buf][v] : 0;
      all += s_sum[buf][v];
    }
    if (k < b1) row_ptr[k] = before + prior + run - own;
    before += all;
  }
  if (b1 == N && t == 0) row_ptr[N] = before;
}

// limits[0], limits[1] (zeroed by the caller) = the largest |wrap| and the largest count.  Unsigned: a
// coordinate 2^31 cells or more below the origin has the wrap -2^31, whose magnitude no int holds.
__global__ __launch_bounds__(256) void nlist_limits_kernel(const int32_t* __restrict__ wrap,
                                                           const int32_t* __restrict__ count, int64_t N,
                                                           int64_t* __restrict__ limits) {
  unsigned m[2] = {0u, 0u};
  for (int64_t a = (int64_t)blockIdx.x * 256 + threadIdx.x; a < 3 * N; a += (int64_t)gridDim.x * 256) {
    const int32_t v = wrap[a];
    const unsigned u = v < 0 ? 0u - (unsigned)v : (unsigned)v;
    m[0] = u > m[0] ? u : m[0];
    if (a < N) m[1] = (unsigned)count[a] > m[1] ? (unsigned)count[a] : m[1];
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
      const unsigned v = (unsigned)__shfl_xor((int)m[h], s, 64);
      m[h] = v > m[h] ? v : m[h];
    }
    if ((threadIdx.x & 63) == 0 && m[h] > 0)
      atomicMax(reinterpret_cast<unsigned long long*>(limits + h), (unsigned long long)m[h]);
  }
}

__global__ __launch_bounds__(256) void nlist_emit_kernel(const int32_t* __restrict__ sender,
                                                         const int32_t* __restrict__ off,
                                                         const int32_t* __restrict__ nout,
                                                         const int64_t* __restrict__ row_ptr, int64_t N, int32_t K,
                                                         int64_t* __restrict__ edge_index,
                                                         float* __restrict__ cell_offsets, int64_t E) {
  const int64_t total = N * K;
  for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < total; s += (int64_t)gridDim.x * blockDim.x) {
    const int64_t j = s / K;
    const int r = (int)(s - j * K);
    if (r >= nout[j]) continue;
    const int64_t e = row_ptr[j] + r;
    edge_index[e] = sender[s];
    edge_index[E + e] = j;
#pragma unroll
    for (int a = 0; a < 3; ++a) cell_offsets[3 * e + a] = (float)off[3 * s + a];
  }
}

static NLGeom nl_geom(const double* cell, const double* inv, const int32_t* nbins, const int32_t* reach,
                      const int32_t* pbc, double cutoff) {
  NLGeom g;
  for (int k = 0; k < 9; ++k) {
    g.cell[k] = cell[k];
    g.inv[k] = inv[k];
  }
  for (int a = 0; a < 3; ++a) {
    g.nb[a] = nbins[a];
    g.reach[a] = reach[a];
    g.pbc[a] = pbc[a] ? 1 : 0;
  }
  g.cut2 = cutoff * cutoff;
  return g;
}

static int nl_check_geom(const double* cell, const double* inv, const int32_t* nbins, const int32_t* reach,
                         const int32_t* pbc, const char* who) {
  if (!cell || !inv || !nbins || !reach || !pbc) return set_error(FU_ERR_NULL, "%s: NULL geometry", who);
  int64_t total = 1;
  for (int a = 0; a < 3; ++a) {
    if (nbins[a] < 1 || reach[a] < 0 || reach[a] > 64 || (!pbc[a] && (nbins[a] != 1 || reach[a] != 0)))
      return set_error(FU_ERR_SHAPE, "%s: bad bins/reach on axis %d", who, a);
    total *= nbins[a];
  }
  if (total > 0x7fffffffLL) return set_error(FU_ERR_SHAPE, "%s: too many bins", who);
  return FU_OK;
}

}  // namespace fu

using namespace fu;

extern "C" int fu_nlist_bin(const float* pos, int64_t N, const double* cell, const double* inv_cell,
                            const int32_t* nbins, const int32_t* reach, const int32_t* pbc, int64_t* bin_key,
                            int32_t* wrap, void* stream) {
  if (N < 0) return set_error(FU_ERR_SHAPE, "fu_nlist_bin: bad shape");
  int st = nl_check_geom(cell, inv_cell, nbins, reach, pbc, "fu_nlist_bin");
  if (st != FU_OK) return st;
  if (N == 0) return FU_OK;
  if (!pos || !bin_key || !wrap) return set_error(FU_ERR_NULL, "fu_nlist_bin: NULL argument");
  const NLGeom g = nl_geom(cell, inv_cell, nbins, reach, pbc, 0.0);
  hipLaunchKernelGGL(nlist_bin_kernel, dim3((unsigned)std::min<int64_t>(cdiv(N, 256), 65536)), dim3(256), 0,
                     as_stream(stream), pos, g, N, bin_key, wrap);
  return check_launch("fu_nlist_bin");
}

extern "C" int fu_nlist_search(const float* pos, const int64_t* sorted_atoms, const int32_t* bin_ptr,
                               const int32_t* wrap, const int64_t* bin_key, int64_t N, const double* cell,
                               const double* inv_cell, const int32_t* nbins, const int32_t* reach,
                               const int32_t* pbc, double cutoff, int32_t max_neighbors, int32_t* out_sender,
                               int32_t* out_off, int32_t* count, int32_t* nout, void* stream) {
  if (N < 0 || max_neighbors < 1 || !(cutoff > 0.0)) return set_error(FU_ERR_SHAPE, "fu_nlist_search: bad arguments");
  if (N > 0x7fffffffLL) return set_error(FU_ERR_SHAPE, "fu_nlist_search: N too large");
  int st = nl_check_geom(cell, inv_cell, nbins, reach, pbc, "fu_nlist_search");
  if (st != FU_OK) return st;
  if (N == 0) return FU_OK;
  if (!pos || !sorted_atoms || !bin_ptr || !wrap || !bin_key || !out_sender || !out_off || !count || !nout)
    return set_error(FU_ERR_NULL, "fu_nlist_search: NULL argument");
  const NLGeom g = nl_geom(cell, inv_cell, nbins, reach, pbc, cutoff);
  hipLaunchKernelGGL(nlist_search_kernel, dim3((unsigned)cdiv(N, 4)), dim3(256), 0, as_stream(stream), pos,
                     sorted_atoms, bin_ptr, wrap, bin_key, g, N, max_neighbors, out_sender, out_off, count, nout);
  return check_launch("fu_nlist_search");
}

extern "C" int fu_nlist_scan(const int32_t* nout, int64_t* row_ptr, int64_t N, void* stream) {
  if (N < 0) return set_error(FU_ERR_SHAPE, "fu_nlist_scan: bad shape");
  if (!row_ptr || (N > 0 && !nout)) return set_error(FU_ERR_NULL, "fu_nlist_scan: NULL argument");
  const int64_t span = 1024 * std::max<int64_t>(1, (N + 256 * 1024 - 1) / (256 * 1024));
  hipLaunchKernelGGL(nlist_scan_kernel, dim3(std::max(1u, cdiv(N, span))), dim3(1024), 0, as_stream(stream), nout, row_ptr,
                     N, span);
  return check_launch("fu_nlist_scan");
}

extern "C" int fu_nlist_limits(const int32_t* wrap, const int32_t* count, int64_t N, int64_t* limits, void* stream) {
  if (N < 0) return set_error(FU_ERR_SHAPE, "fu_nlist_limits: bad shape");
  if (N == 0) return FU_OK;
  if (!wrap || !count || !limits) return set_error(FU_ERR_NULL, "fu_nlist_limits: NULL argument");
  hipLaunchKernelGGL(nlist_limits_kernel, dim3((unsigned)std::min<int64_t>(cdiv(3 * N, 256), 256)), dim3(256), 0,
                     as_stream(stream), wrap, count, N, limits);
  return check_launch("fu_nlist_limits");
}

extern "C" int fu_nlist_emit(const int32_t* sender, const int32_t* off, const int32_t* nout, const int64_t* row_ptr,
                             int64_t N, int32_t max_neighbors, int64_t* edge_index, float* cell_offsets, int64_t E,
                             void* stream) {
  if (N < 0 || E < 0 || max_neighbors < 1) return set_error(FU_ERR_SHAPE, "fu_nlist_emit: bad shape");
  if (N == 0 || E == 0) return FU_OK;
  if (!sender || !off || !nout || !row_ptr || !edge_index || !cell_offsets)
    return set_error(FU_ERR_NULL, "fu_nlist_emit: NULL argument");
  hipLaunchKernelGGL(nlist_emit_kernel, dim3((unsigned)std::min<int64_t>(cdiv(N * max_neighbors, 256), 65536)),
                     dim3(256), 0, as_stream(stream), sender, off, nout, row_ptr, N, max_neighbors, edge_index,
                     cell_offsets, E);
  return check_launch("fu_nlist_emit");
}
