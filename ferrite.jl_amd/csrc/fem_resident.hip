// Resident CG: the Chronopoulos–Gear recurrence of fem_solve.hip (same scalars, same hand-over
// rule, same reseed) in one cooperative launch per solve, hand-overs included.
//
// What bounds the separate kernels on systems of up to a few hundred thousand rows is not their
// bytes but two launches per iteration.  Here every block (one per CU) owns a compact part of
// the mesh and keeps on chip, for the whole stretch, its rows' operator entries (registers and
// LDS, with 16-bit positions into the block's part of r̂), r̂ for its rows and for the rows they
// couple to (LDS), and p, ŝ = Âp, x̂ (registers).  One exchange per iteration is left: a block publishes
// w = Âr̂ of its rows and its partials of γ = r̂·r̂ and δ = r̂·w, and reads the others' partials
// and the w of its coupled rows; with those it also moves the coupled rows' ŝ and r̂ itself
// (the same operations on the same values as their owner, so they stay equal bit for bit), and
// the next product needs no second exchange.  A hand-over folds x̂ into the FP64 u, publishes the u
// other blocks read, forms the FP64 residual f − K u from K's own entries and publishes the new r̂:
// two more exchanges instead of half a dozen launches and a host round trip (301×227 Q1 quads in
// FP32, 13 hand-overs: whole assembly and solve 5.78 → 5.14 ms; 47×53×61 hexes, 10: 2.68 → 2.29).
//
// Several independent systems can share a launch, their rows cut into separate parts: sums and
// waits stay inside a system's own blocks, which leave when their system is done.
//
// The exchange has no barrier and no fence.  Every published value travels in 8-byte words of
// 32 data bits and the exchange's 32-bit number, written and read with agent-scope accesses
// (which reach the memory all XCDs share); a reader polls the words it needs until
// they carry the number.  Two buffers alternate: a block writes exchange e + 2 only after it
// holds every block's partials of e + 1, which they publish after reading all of e.  Partials
// are summed in block order, so every block holds the same scalars and results are bitwise
// reproducible.  Waits are bounded (kResPolls): a block that gives up reports it and stops
// publishing, so every other block gives up too, and the host runs the separate kernels.
//
// Measured, µs per iteration, separate kernels → here: 100×100 Q1 quads FP64 11.7 → 3.0 (21
// blocks); 24×20×17 distorted hexes FP64 17.4 → 3.6 (24); 64³ hexes FP64 33 → 6.3 (216); 512×256
// Q1² quads FP64 26.5 → 4.0 (180); 301×227 Q1 quads FP32 cell form 13.3 → 3.6 (140) and 47×53×61
// hexes FP32 planes 16.2 → 5.9 (both with their hand-overs).  Vector units busy 25% (64³) to 34%
// (301×227), LDS 25% and 9%: the exchange's latency is what is left.  At 100×100 an iteration is about 0.25 µs of
// products, 0.3 µs of sums inside the block, 1.3 µs until the other blocks' values are there and
// 0.5 µs of scalars and vector moves.
#include <algorithm>
#include <cmath>

#include "fem_resident_dev.h"

namespace fem {

constexpr int kResRows = 256;           // least rows per block when there are several
constexpr int kMaxStallRes = 6;         // hand-overs in a row without progress (kMaxStall of fem_solve.hip)

struct ResOp {
  int state = 0;                        // 1 usable, −1 does not fit
  // parts: one block each; own rows (those other parts read first, each class ascending),
  // coupled rows (ascending), published slots
  int nb = 0, ng = 0, Rmax = 0, Rp = 0, nz = 0, nlocmax = 0, nhmax = 0, nslots = 0;
  int4* grp = nullptr;                  // [nb] system of each part, its first part, how many, its largest
  int32_t* oofs = nullptr;              // [nb + 1] ranges of orow
  int32_t* orow = nullptr;              // own rows of each part
  int32_t* pofs = nullptr;              // [nb + 1] published slots: one per row other parts read
  int32_t* hoff = nullptr;              // [nb + 1] ranges of hrow, hslot
  int32_t* hrow = nullptr;              // coupled rows of each part
  int32_t* hslot = nullptr;             // ... and their published slots
  uint32_t* ai = nullptr;               // [nb][nz2][Rp] positions of two entries each
  // values per precision: [nb][nz][Rp]
  float* val32 = nullptr;
  double* val64 = nullptr;
  double* raw = nullptr;                // [nb][nz][Rp] unscaled FP64 entries (FP32 solver: residuals)
  uint64_t ver[2] = {0, 0}, aux[2] = {0, 0};
  int jac[2] = {-1, -1}, vsrc[2] = {-1, -1};
  // exchange buffers and the number of the last exchange handed out
  uint32_t* wx = nullptr;               // [2][nslots] values (8 or 16 bytes each)
  uint32_t* wu = nullptr;               // [nslots] FP64 values: u of a hand-over
  ResState* st = nullptr;               // [ng] pinned host memory, written by the launch
  uint32_t* rec = nullptr;              // [2][kResCopies][2][kResMaxBlocks] values of 16 bytes
  uint32_t epoch = 0;
};

void resident_free(ResOp** op) {
  if (!*op) return;
  ResOp* o = *op;
  dev_free(&o->grp); dev_free(&o->oofs); dev_free(&o->orow); dev_free(&o->pofs); dev_free(&o->hoff); dev_free(&o->hrow);
  dev_free(&o->hslot); dev_free(&o->ai); dev_free(&o->val32); dev_free(&o->val64); dev_free(&o->raw);
  dev_free(&o->wx); dev_free(&o->wu);
  if (o->st) (void)hipHostFree(o->st); dev_free(&o->rec);
  delete o;
  *op = nullptr;
}

// ---- row access ---------------------------------------------------------------------------
struct ResRows {
  int src, dim;
  int64_t n, npad;
  int32_t px, pxy;
  const int32_t *colptr, *rowval, *dofp, *map;
  const double *nzval, *sc, *kc;
  const void *val, *t;
  double f[8];
};

// Row of entry k of a row in the order of K's column, −1 when the column has no such entry.
__device__ __forceinline__ int32_t res_col(const ResRows& a, int32_t row, int k) {
  const int32_t j = a.src == 0 ? row : a.dofp[row];
  if (j < 0) return -1;
  const int32_t p = a.colptr[j] + k;
  if (p >= a.colptr[j + 1]) return -1;
  return a.src == 0 ? a.rowval[p] : a.map[a.rowval[p]];
}

// ---- parts --------------------------------------------------------------------------------
// The rows are cut into sx × sy × sz compact parts of nearly equal size by nested quantiles of
// their positions: slabs along x, each slab along y, each of those along z.  Compact parts read
// few rows of others (a part of 1,000 rows of a 2D grid about 130, where a range of consecutive
// rows reads 1,000): what the parts publish and read per iteration is what bounds it.
constexpr int kResBins = 4096;

// Position of a row: its lattice index, or that of a node of its first cell.
struct ResPos {
  int src, dim;                      // dim: of the lattice / of the coordinates
  int32_t px, pxy;
  const int32_t *dofp, *node;        // node: [n]
  const double* x[3];
};
__device__ __forceinline__ bool res_pos(const ResPos& a, int32_t row, double (&x)[3]) {
  x[1] = x[2] = 0.0;
  if (a.src != 0) {
    if (a.dofp[row] < 0) return false;
    const int32_t z = a.dim == 3 ? row / a.pxy : 0, r = row - z * a.pxy, y = r / a.px;
    x[0] = r - y * a.px;
    x[1] = y;
    x[2] = z;
    return true;
  }
  const int32_t nd = a.node[row];
  for (int d = 0; d < a.dim; ++d) x[d] = a.x[d][nd];
  return true;
}

// A system of the launch: its rows, and (x − lo) inv in [0, kResBins) along each axis.
struct ResSystem {
  int32_t row0, row1;
  double lo[3], inv[3];
};
__device__ __forceinline__ int res_bin(const ResSystem& g, const double (&x)[3], int d) {
  return max(0, min(kResBins - 1, (int)((x[d] - g.lo[d]) * g.inv[d])));
}

// One block per system: bounding box of its rows (out[0..2], out[3..5]), their number (out[9]),
// and per axis the mean over sampled rows of the largest distance to a row they couple to
// (out[6..8]): the spacing of the rows.
__global__ __launch_bounds__(1024) void k_res_geom(ResPos g, ResRows a, const ResSystem* __restrict__ sys, int nz,
                                                   double* __restrict__ out) {
  __shared__ double sh[10][16];
  __shared__ double hsum[16];
  const int32_t row0 = sys[blockIdx.x].row0, row1 = sys[blockIdx.x].row1;
  double v[10] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300, 0.0, 0.0, 0.0, 0.0};
  for (int32_t row = row0 + (int32_t)threadIdx.x; row < row1; row += 1024) {
    double x[3];
    if (!res_pos(g, row, x)) continue;
    for (int d = 0; d < 3; ++d) {
      v[d] = fmin(v[d], x[d]);
      v[3 + d] = fmax(v[3 + d], x[d]);
    }
    v[9] += 1.0;
  }
  const int32_t s = row0 + (int32_t)(((int64_t)threadIdx.x * (row1 - row0)) / 1024);
  double xs[3], hs = 0.0;
  if (res_pos(g, s, xs)) {
    double far[3] = {0.0, 0.0, 0.0};
    for (int k = 0; k < nz; ++k) {
      const int32_t q = res_col(a, s, k);
      double x[3];
      if (q < 0 || !res_pos(g, q, x)) continue;
      for (int d = 0; d < 3; ++d) far[d] = fmax(far[d], fabs(x[d] - xs[d]));
    }
    for (int d = 0; d < 3; ++d) v[6 + d] = far[d];
    hs = 1.0;
  }
  for (int i = 0; i < 10; ++i)
    for (int o = 32; o > 0; o >>= 1) {
      const double u = __shfl_down(v[i], o, 64);
      v[i] = i < 3 ? fmin(v[i], u) : i < 6 ? fmax(v[i], u) : v[i] + u;
    }
  for (int o = 32; o > 0; o >>= 1) hs += __shfl_down(hs, o, 64);
  if ((threadIdx.x & 63) == 0) {
    for (int i = 0; i < 10; ++i) sh[i][threadIdx.x >> 6] = v[i];
    hsum[threadIdx.x >> 6] = hs;
  }
  __syncthreads();
  if (threadIdx.x < 10) {
    const int i = threadIdx.x;
    double r = sh[i][0], h = hsum[0];
    for (int w = 1; w < 16; ++w) {
      const double u = sh[i][w];
      r = i < 3 ? fmin(r, u) : i < 6 ? fmax(r, u) : r + u;
      h += hsum[w];
    }
    out[10 * blockIdx.x + i] = i >= 6 && i < 9 ? r / fmax(h, 1.0) : r;
  }
}

// part = the system of each row that has a place, −1 elsewhere.
__global__ __launch_bounds__(256) void k_res_start(ResPos g, const ResSystem* __restrict__ sys,
                                                   int32_t* __restrict__ part) {
  const int32_t row0 = sys[blockIdx.y].row0, row1 = sys[blockIdx.y].row1;
  for (int32_t row = row0 + (int32_t)(blockIdx.x * 256 + threadIdx.x); row < row1; row += gridDim.x * 256) {
    double x[3];
    part[row] = res_pos(g, row, x) ? (int32_t)blockIdx.y : -1;
  }
}

// One level of the cut along axis d: rows per (slab, bin), the finer slab of each (slab, bin),
// the rows' finer slabs.  A slab: its system, how many slabs it is cut into, the first of them.
__global__ __launch_bounds__(256) void k_res_hist(ResPos g, const ResSystem* __restrict__ sys,
                                                  const int4* __restrict__ slab, int64_t n, int d,
                                                  const int32_t* __restrict__ part, int32_t* __restrict__ hist) {
  for (int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x; row < n; row += (int64_t)gridDim.x * 256) {
    const int32_t p = part[row];
    double x[3];
    if (p >= 0 && res_pos(g, (int32_t)row, x))
      atomicAdd(&hist[(int64_t)p * kResBins + res_bin(sys[slab[p].x], x, d)], 1);
  }
}
__global__ __launch_bounds__(256) void k_res_cut(const int4* __restrict__ slab, int32_t* __restrict__ hist) {   // one block per slab
  __shared__ int32_t sum[256];
  const int s = slab[blockIdx.x].y, first = slab[blockIdx.x].z;
  int32_t* h = hist + (int64_t)blockIdx.x * kResBins;
  constexpr int PER = kResBins / 256;
  int32_t c[PER], all = 0;
  for (int i = 0; i < PER; ++i) all += c[i] = h[threadIdx.x * PER + i];
  sum[threadIdx.x] = all;
  __syncthreads();
  for (int o = 1; o < 256; o <<= 1) {
    const int32_t v = (int)threadIdx.x >= o ? sum[threadIdx.x - o] : 0;
    __syncthreads();
    sum[threadIdx.x] += v;
    __syncthreads();
  }
  const int64_t total = sum[255];
  int64_t before = sum[threadIdx.x] - all;
  for (int i = 0; i < PER; ++i) {   // the slab that holds the bin's middle row
    const int64_t f = total > 0 ? (2 * before + c[i]) * s / (2 * total) : 0;
    before += c[i];
    h[threadIdx.x * PER + i] = first + (int32_t)min<int64_t>(f, s - 1);
  }
}
__global__ __launch_bounds__(256) void k_res_split(ResPos g, const ResSystem* __restrict__ sys,
                                                   const int4* __restrict__ slab, int64_t n, int d,
                                                   const int32_t* __restrict__ hist, int32_t* __restrict__ part) {
  for (int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x; row < n; row += (int64_t)gridDim.x * 256) {
    const int32_t p = part[row];
    double x[3];
    if (p >= 0 && res_pos(g, (int32_t)row, x)) part[row] = hist[(int64_t)p * kResBins + res_bin(sys[slab[p].x], x, d)];
  }
}

// Rows that another part's rows name; the size of each part.
__global__ __launch_bounds__(256) void k_res_shared(ResRows a, int nz, const int32_t* __restrict__ part,
                                                    uint8_t* __restrict__ flag, int32_t* __restrict__ size) {
  for (int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x; row < a.n; row += (int64_t)gridDim.x * 256) {
    const int32_t p = part[row];
    if (p < 0) continue;
    atomicAdd(&size[p], 1);
    for (int k = 0; k < nz; ++k) {
      const int32_t q = res_col(a, (int32_t)row, k);
      if (q >= 0 && part[q] != p) flag[q] = 1;
    }
  }
}

// The rows of each part, then (one block per part) sorted: rows other parts read first, each
// class ascending; rank[row] = the row's place, shared[b] = how many other parts read.
__global__ __launch_bounds__(256) void k_res_gather(int64_t n, const int32_t* __restrict__ part,
                                                    const uint8_t* __restrict__ flag, const int32_t* __restrict__ oofs,
                                                    int32_t* __restrict__ fill, int32_t* __restrict__ orow) {
  for (int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x; row < n; row += (int64_t)gridDim.x * 256) {
    const int32_t p = part[row];
    if (p >= 0) orow[oofs[p] + atomicAdd(&fill[p], 1)] = (int32_t)row | (flag[row] ? 0 : 1 << 30);
  }
}
__global__ __launch_bounds__(1024) void k_res_sort(int pow2, const int32_t* __restrict__ oofs,
                                                   int32_t* __restrict__ orow, int32_t* __restrict__ rank,
                                                   int32_t* __restrict__ shared) {
  extern __shared__ int32_t res_key[];
  __shared__ int ns;
  const int32_t o0 = oofs[blockIdx.x], m = oofs[blockIdx.x + 1] - o0;
  if (threadIdx.x == 0) ns = 0;
  for (int i = threadIdx.x; i < pow2; i += 1024) res_key[i] = i < m ? orow[o0 + i] : INT_MAX;
  __syncthreads();
  for (int k = 2; k <= pow2; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < pow2; i += 1024) {
        const int l = i ^ j;
        if (l > i) {
          const int32_t x = res_key[i], y = res_key[l];
          if ((x > y) == ((i & k) == 0)) {
            res_key[i] = y;
            res_key[l] = x;
          }
        }
      }
      __syncthreads();
    }
  int mine = 0;
  for (int i = threadIdx.x; i < m; i += 1024) {
    const int32_t v = res_key[i], row = v & ~(1 << 30);
    mine += !(v & (1 << 30));
    orow[o0 + i] = row;
    rank[row] = i;
  }
  atomicAdd(&ns, mine);
  __syncthreads();
  if (threadIdx.x == 0) shared[blockIdx.x] = ns;
}

// A part's bitmap of the rows of other parts that its rows name, in LDS: of the rows of its
// system, which start at row0.
__device__ __forceinline__ void res_mark(const ResRows& a, int nz, int32_t row0, const int32_t* __restrict__ part,
                                         const int32_t* __restrict__ own, int m, uint32_t* bm, int words) {
  for (int i = threadIdx.x; i < words; i += blockDim.x) bm[i] = 0u;
  __syncthreads();
  for (int i = threadIdx.x; i < m; i += blockDim.x)
    for (int k = 0; k < nz; ++k) {
      const int32_t q = res_col(a, own[i], k);
      if (q >= 0 && part[q] != (int32_t)blockIdx.x) atomicOr(&bm[(q - row0) >> 5], 1u << ((q - row0) & 31));
    }
  __syncthreads();
}

__global__ __launch_bounds__(256) void k_res_count(ResRows a, int nz, int words, const ResSystem* __restrict__ sys,
                                                   const int4* __restrict__ grp, const int32_t* __restrict__ part,
                                                   const int32_t* __restrict__ oofs,
                                                   const int32_t* __restrict__ orow, int32_t* __restrict__ cnt) {
  extern __shared__ uint32_t res_bm[];
  __shared__ int tot;
  if (threadIdx.x == 0) tot = 0;
  res_mark(a, nz, sys[grp[blockIdx.x].x].row0, part, orow + oofs[blockIdx.x], oofs[blockIdx.x + 1] - oofs[blockIdx.x], res_bm, words);
  int all = 0;
  for (int i = threadIdx.x; i < words; i += blockDim.x) all += __popc(res_bm[i]);
  atomicAdd(&tot, all);
  __syncthreads();
  if (threadIdx.x == 0) cnt[blockIdx.x] = tot;
}

// The coupled rows of each part with their slots, and the entries' positions in its local
// numbering: own rows by rank, then the coupled rows.
__global__ __launch_bounds__(256) void k_res_fill(ResRows a, int nz, int Rp, int words, const ResSystem* __restrict__ sys,
                                                  const int4* __restrict__ grp, const int32_t* __restrict__ part,
                                                  const int32_t* __restrict__ rank, const int32_t* __restrict__ oofs,
                                                  const int32_t* __restrict__ orow, const int32_t* __restrict__ pofs,
                                                  const int32_t* __restrict__ hoff, int32_t* __restrict__ hrow,
                                                  int32_t* __restrict__ hslot, uint32_t* __restrict__ ai) {
  extern __shared__ uint32_t res_bm[];
  const int ng = (words + 7) / 8;
  const int32_t row0 = sys[grp[blockIdx.x].x].row0;
  uint32_t* pre = res_bm + words;    // [ng] rows before each group of 8 words
  const int32_t o0 = oofs[blockIdx.x], m = oofs[blockIdx.x + 1] - o0, h0 = hoff[blockIdx.x];
  res_mark(a, nz, row0, part, orow + o0, m, res_bm, words);
  for (int g = threadIdx.x; g < ng; g += blockDim.x) {
    uint32_t c = 0;
    for (int i = 8 * g; i < min(words, 8 * g + 8); ++i) c += __popc(res_bm[i]);
    pre[g] = c;
  }
  __syncthreads();
  if (threadIdx.x < 64) {            // exclusive scan by one wave
    uint32_t base = 0;
    for (int g0 = 0; g0 < ng; g0 += 64) {
      const int g = g0 + (int)threadIdx.x;
      const uint32_t v = g < ng ? pre[g] : 0u;
      uint32_t s = v;
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t up = __shfl_up(s, o, 64);
        if ((int)threadIdx.x >= o) s += up;
      }
      if (g < ng) pre[g] = base + s - v;
      base += __shfl(s, 63, 64);
    }
  }
  __syncthreads();
  auto coupled = [&](int32_t q) {    // place of a marked row
    q -= row0;
    const int w = q >> 5, g = w >> 3;
    uint32_t l = pre[g];
    for (int i = 8 * g; i < w; ++i) l += __popc(res_bm[i]);
    return l + __popc(res_bm[w] & ((1u << (q & 31)) - 1u));
  };
  for (int i = threadIdx.x; i < words; i += blockDim.x) {
    uint32_t bits = res_bm[i];
    while (bits) {
      const int32_t q = row0 + i * 32 + __ffs(bits) - 1;
      bits &= bits - 1;
      const int32_t h = h0 + (int32_t)coupled(q);
      hrow[h] = q;
      hslot[h] = pofs[part[q]] + rank[q];
    }
  }
  const int nz2 = (nz + 1) / 2;
  for (int32_t i = threadIdx.x; i < Rp; i += blockDim.x) {
    const int32_t row = i < m ? orow[o0 + i] : -1;
    for (int k2 = 0; k2 < nz2; ++k2) {
      uint32_t pk = 0;
      for (int h = 0; h < 2; ++h) {
        const int32_t q = row >= 0 && 2 * k2 + h < nz ? res_col(a, row, 2 * k2 + h) : -1;
        if (q >= 0) pk |= (part[q] == (int32_t)blockIdx.x ? (uint32_t)rank[q] : (uint32_t)m + coupled(q)) << (16 * h);
      }
      ai[((int64_t)blockIdx.x * nz2 + k2) * Rp + i] = pk;
    }
  }
}

// Values of the rows' entries in X precision (0 where an entry is missing), and unscaled in raw.
template <typename X>
__global__ __launch_bounds__(256) void k_res_vals(ResRows a, int nz, int Rp, int nb, const int32_t* __restrict__ oofs,
                                                  const int32_t* __restrict__ orow, X* __restrict__ val,
                                                  double* __restrict__ raw) {
  for (int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x; g < (int64_t)nb * Rp; g += (int64_t)gridDim.x * 256) {
    const int b = (int)(g / Rp), i = (int)(g - (int64_t)b * Rp);
    const int32_t o0 = oofs[b];
    const bool in = i < oofs[b + 1] - o0;
    const int32_t row = in ? orow[o0 + i] : 0, j = a.src == 0 ? row : a.dofp[row];
    const int64_t out = (int64_t)b * nz * Rp + i;
    const int32_t p0 = in ? a.colptr[j] : 0, len = in ? a.colptr[j + 1] - p0 : 0;
    const double sr = in ? a.sc[j] : 0.0;
    // cell form: the coefficients around the row; a prescribed row (t = 0) keeps its unit diagonal
    const X* tt = static_cast<const X*>(a.t);
    const bool free_p = a.src == 2 && in && tt[row] != X(0);
    double k8[8] = {};
    if (a.src == 2)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (in && (a.dim == 3 || e < 4))
          k8[e] = a.kc[row - (e & 1) - (int64_t)a.px * ((e >> 1) & 1) - (int64_t)a.pxy * (e >> 2)];
    for (int k0 = 0; k0 < nz; k0 += 9) {   // nz is a multiple of 9; nine entries in flight
      double v[9], sj[9];
      int32_t q[9];
#pragma unroll
      for (int u = 0; u < 9; ++u) {
        const bool real = k0 + u < len;
        v[u] = real ? a.nzval[p0 + k0 + u] : 0.0;
        q[u] = real ? a.rowval[p0 + k0 + u] : -1;
      }
#pragma unroll
      for (int u = 0; u < 9; ++u) sj[u] = q[u] >= 0 ? a.sc[q[u]] : 0.0;
#pragma unroll
      for (int u = 0; u < 9; ++u) {
        const int64_t at = out + (int64_t)(k0 + u) * Rp;
        if (raw) raw[at] = v[u];
        X x = X(0);
        if (a.src == 0) {
          x = (X)(v[u] * (sr * sj[u]));
        } else if (q[u] >= 0) {
          const int32_t Q = a.map[q[u]], off = Q - row, shift = 1 + a.px + (a.dim == 3 ? a.pxy : 0);
          // lattice offsets as digits of off + shift (fem_solve.hip lat_code; the pattern is checked there)
          const int32_t t = off + shift, rz = a.dim == 3 ? t % a.pxy : t;
          const int dz = a.dim == 3 ? t / a.pxy - 1 : 0, dy = rz / a.px - 1, dx = rz % a.px - 1;
          const bool near = t >= 0 && dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1 && dz >= -1 && dz <= 1;
          if (near && a.src == 1) {
            const int code = (dx + 1) + 3 * (dy + 1) + 9 * (dz + 1);
            const X* val0 = static_cast<const X*>(a.val);
            x = code >= 13 ? val0[(int64_t)(code - 13) * a.npad + row] : val0[(int64_t)(13 - code) * a.npad + Q];
          } else if (near) {
            // s_P s_Q f[class] Σ k over the cells that hold both corners, in FP64 and rounded once
            double ks = 0.0;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const bool both = (dx == 0 || (e & 1) == (dx < 0)) && (dy == 0 || ((e >> 1) & 1) == (dy < 0)) &&
                                (dz == 0 || (e >> 2) == (dz < 0));
              ks += both ? k8[e] : 0.0;
            }
            if (free_p && tt[Q] != X(0)) x = (X)(a.f[(dx != 0) + 2 * (dy != 0) + 4 * (dz != 0)] * ks * (sr * sj[u]));
            if (!free_p && Q == row) x = X(1);
          }
        }
        val[at] = x;
      }
    }
  }
}

// ---- the recurrence -----------------------------------------------------------------------
// Σ a[e] r[position e] of a row whose entries are in registers; pos[m]: the byte offsets of entries
// 2 m and 2 m + 1.  The LDS reads of a group of entries are under way while the group before is
// summed: left to itself the compiler, short of registers, waits for each (FP64, 18 entries, three
// rows a thread: a product 1.55 → 0.60 µs, an iteration at 512×256 Q1² quads 4.8 → 4.0 µs).
template <typename X, int NZ>
__device__ __forceinline__ X gather_dot(const X* r, const X (&a)[NZ], const uint32_t (&pos)[(NZ + 1) / 2]) {
  constexpr int G = sizeof(X) == 4 ? 6 : 4, NG = (NZ + G - 1) / G;   // G even
  X v[2][G];
  auto load = [&](int g) {
#pragma unroll
    for (int i = 0; i < G; i += 2) {
      const int e = g * G + i;
      if (e >= NZ) break;
      const uint32_t q = pos[e / 2];
      v[g & 1][i] = at_lds(r, q & 0xffffu);
      if (e + 1 < NZ) v[g & 1][i + 1] = at_lds(r, q >> 16);
    }
  };
  X acc = X(0);
  load(0);
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    if (g + 1 < NG) load(g + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < G; ++i)
      if (g * G + i < NZ) acc += a[g * G + i] * v[g & 1][i];
  }
  return acc;
}

template <typename X>
struct ResArgs {
  int Rp, nslots;
  int nl, rl0, nhmax;            // rows whose entries LDS holds; elements of r̂, and of ŝ and w, there
  const int4* grp;
  const int32_t *oofs, *orow, *pofs, *hoff, *hrow, *hslot;
  const uint32_t* ai;
  const X* val;
  const double* raw;             // unscaled entries, or null: read from nzval
  const int32_t* colptr;
  const double* nzval;
  const int32_t* dofp;           // dof of a row (lattice rows), or null: the same index
  const double *f, *sc;
  double* u;
  const double* in;              // [ng][2] squares of the initial residual and the tolerance, or null: in0
  ResState* st;
  uint32_t *wx, *wu, *rec;
  double in0[2], hold2;
  uint32_t epoch, polls;
  int lim, time;
};

// Rows per thread RT; the entries (NZ per row) of the first RRES stay in registers, those of the
// block's other rows (a.nl of them) in LDS.  LDS: r̂ of the rows the block reads (own, coupled,
// and a zero slot for the threads' unused rows), at a hand-over their u in its place; ŝ, w and the
// slots of the coupled rows; the entries of a.nl rows.
template <typename X, int NZ, int RRES, int RT>
__global__ __launch_bounds__(kResT) void k_resident(ResArgs<X> a) {
  constexpr int NZ2 = (NZ + 1) / 2;
  constexpr int QS = NZ2 | 1;                 // a row's words in LDS (odd: no bank conflicts)
  constexpr int H = sizeof(X) == 4 ? 8 : 4;   // coupled rows a thread polls at once
  // reads ahead of the sums, but not where the entries fill the registers (FP64, 27 entries: 64³
  // hexes 6.4 µs per iteration without, 6.8 with)
  constexpr bool AHEAD = sizeof(X) * NZ < 8 * 27;
  extern __shared__ __align__(16) unsigned char res_lds[];
  __shared__ double red[2][2][kResWaves];    // wave sums, alternating
  __shared__ double tot[2][2][4];            // sums of 64 blocks' partials each
  __shared__ int gaveup;
  __shared__ uint32_t polls;                 // what a wait may take (in LDS: scalar registers are short)
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int b = blockIdx.x;
  const int4 gr = a.grp[b];
  const int b0 = gr.y, nb = gr.z;            // the system's blocks
  const long long begin = wall_clock64();
  const int32_t o0 = a.oofs[b], nown = a.oofs[b + 1] - o0;
  const int32_t p0 = a.pofs[b], npub = a.pofs[b + 1] - p0;
  const int32_t h0 = a.hoff[b], nh = a.hoff[b + 1] - h0;
  X* rl = reinterpret_cast<X*>(res_lds);
  X* sl = rl + a.rl0;
  X* wl = sl + a.nhmax;
  X* lv = wl + a.nhmax;
  uint32_t* lq = reinterpret_cast<uint32_t*>(lv + (size_t)NZ * a.nl);
  int32_t* hl = reinterpret_cast<int32_t*>(lq + (size_t)QS * a.nl);
  const int zero = nown + nh;
  double rrt = a.in ? a.in[2 * gr.x] : a.in0[0];   // the true residual's square
  const double tol2 = a.in ? a.in[2 * gr.x + 1] : a.in0[1];
  if (t == 0) {
    gaveup = 0;
    polls = a.polls;
    rl[zero] = X(0);
  }

  // operator rows
  X av[RRES][NZ];
  uint32_t ai[RRES][NZ2];
  const X* vb = a.val + (int64_t)b * NZ * a.Rp;
  const uint32_t* ib = a.ai + (int64_t)b * NZ2 * a.Rp;
#pragma unroll
  for (int k = 0; k < RRES; ++k) {
    const int i = t + k * kResT;
    const bool in = i < nown;
#pragma unroll
    for (int j = 0; j < NZ; ++j) av[k][j] = in ? vb[(int64_t)j * a.Rp + i] : X(0);
#pragma unroll
    for (int j = 0; j < NZ2; ++j) ai[k][j] = in ? ib[(int64_t)j * a.Rp + i] * (uint32_t)sizeof(X) : 0u;   // byte offsets
  }
  // the first residual is f: r̂ = S f
  auto seed = [&](int32_t q) {
    const int32_t d = a.dofp ? a.dofp[q] : q;
    return d >= 0 ? (X)(a.sc[d] * a.f[d]) : X(0);
  };
  X p[RT], sv[RT], x[RT], w[RT];
  int il[RT];                                // this thread's rows in rl
#pragma unroll
  for (int k = 0; k < RT; ++k) {
    const int i = t + k * kResT;
    const bool in = i < nown;
    il[k] = in ? i : zero;
    p[k] = sv[k] = x[k] = X(0);
    if (in) rl[i] = seed(a.orow[o0 + i]);
  }
  for (int h = t; h < nh; h += kResT) {
    hl[h] = a.hslot[h0 + h];
    sl[h] = X(0);
    rl[nown + h] = seed(a.hrow[h0 + h]);
  }
  for (int i = t; i < a.nl; i += kResT) {
    const int row = RRES * kResT + i;
    const bool in = row < nown;
    for (int j = 0; j < NZ; ++j) lv[i * NZ + j] = in ? vb[(int64_t)j * a.Rp + row] : X(0);
    for (int j = 0; j < NZ2; ++j) lq[i * QS + j] = in ? ib[(int64_t)j * a.Rp + row] * (uint32_t)sizeof(X) : 0u;
  }
  res_barrier();

  uint32_t ep = a.epoch;
  const __amdgpu_buffer_rsrc_t rw = buf_rsrc(a.wx, (uint32_t)(2 * sizeof(typename LL<X>::W)) * (uint32_t)a.nslots);
  const __amdgpu_buffer_rsrc_t rr = buf_rsrc(a.rec, (uint32_t)(2 * kResCopies * 2 * 16) * kResMaxBlocks);
  // Publishes w of the rows other parts read: the first npub of the part, whose slots are
  // consecutive; the resource ends there, so the stores of the other rows are dropped.
  auto publish = [&]() {
    typedef typename LL<X>::W W;
    const __amdgpu_buffer_rsrc_t ro =
        buf_rsrc(reinterpret_cast<const W*>(a.wx) + ((size_t)(ep & 1u) * a.nslots + p0), (uint32_t)(sizeof(W) * npub));
#pragma unroll
    for (int k = 0; k < RT; ++k)
      if (k * kResT < npub) ll_put(ro, (uint32_t)(t + k * kResT), w[k], ep);
  };
  double rzp = 0.0, alpha = 0.0, irz = 0.0, ira = 0.0;   // γ and α of the last step; 1 / γ, 1 / (γ α)
  // Sums g0, g1 over the system's blocks; with `halo`, reads the coupled rows' w into wl.  Every
  // thread returns the same sums; false when a wait was given up.
  auto exchange = [&](double& g0, double& g1, bool halo) {
    const int par = (int)(ep & 1u);
    const double v0 = wave_sum63(g0), v1 = wave_sum63(g1);
    if (lane == 63) {
      red[par][0][wave] = v0;
      red[par][1][wave] = v1;
    }
    const uint32_t in_lds = polls;                  // (read before the barrier, which waits for it anyway)
    res_barrier();
    if (nb == 1) {
      irz = 1.0 / rzp;
      ira = 1.0 / (rzp * alpha);
      g0 = g1 = 0.0;
#pragma unroll
      for (int i = 0; i < kResWaves; ++i) {
        g0 += red[par][0][i];
        g1 += red[par][1][i];
      }
      ++ep;
      return true;
    }
    // the block's record: its two sums, one copy per group of readers (blocks ≡ b mod 8), so
    // that the reads of all blocks spread over the memory channels
    const uint32_t most = (uint32_t)uniform((int)in_lds);
    const uint32_t rec = (uint32_t)(par * kResCopies * 2 * kResMaxBlocks);
    if (t < 2 * kResCopies) {
      double sum = 0.0;
#pragma unroll
      for (int i = 0; i < kResWaves; ++i) sum += red[par][t & 1][i];
      ll_put(rr, rec + (uint32_t)(t * kResMaxBlocks + b), sum, ep);
    }
    const uint32_t rin = rec + (uint32_t)((b % kResCopies) * 2 * kResMaxBlocks + b0 + t);
    if (halo) {   // reciprocals of the last step's scalars, while the values travel
      irz = 1.0 / rzp;
      ira = 1.0 / (rzp * alpha);
    }
    const bool reader = t < nb;        // thread t reads the record of the system's block t
    bool lost = false, need = reader;
    U4 q0 = {}, q1 = {};
    if (halo) {                        // the coupled rows' w, and the records along with them
      const uint32_t wi = (ep & 1u) * (uint32_t)a.nslots;
      for (int base = 0; base < nh; base += H * kResT) {
        typename LL<X>::W hv[H];
        uint32_t at[H];
#pragma unroll
        for (int k = 0; k < H; ++k) {
          at[k] = wi + (uint32_t)hl[min(base + k * kResT + t, nh - 1)];   // (spare threads repeat the last row)
        }
        for (uint32_t left = most;; --left) {
          asm volatile("" ::: "memory");
          bool ok = true;
          if (need) {
            q0 = LL<double>::get(rr, rin);
            q1 = LL<double>::get(rr, rin + kResMaxBlocks);
          }
#pragma unroll
          for (int k = 0; k < H; ++k)
            if (base + k * kResT < nh) hv[k] = LL<X>::get(rw, at[k]);
#pragma unroll
          for (int k = 0; k < H; ++k)
            if (base + k * kResT < nh) ok = ok && LL<X>::ok(hv[k], ep);
          if (need) need = !(LL<double>::ok(q0, ep) && LL<double>::ok(q1, ep));
          if (ok) break;
          if (left == 0) { lost = true; break; }
        }
#pragma unroll
        for (int k = 0; k < H; ++k)
          if (base + k * kResT + t < nh) wl[base + k * kResT + t] = LL<X>::val(hv[k]);
      }
    }
    if (wave < (kResMaxBlocks + 63) / 64) {
      for (uint32_t left = most; need; --left) {
        asm volatile("" ::: "memory");
        q0 = LL<double>::get(rr, rin);
        q1 = LL<double>::get(rr, rin + kResMaxBlocks);
        need = !(LL<double>::ok(q0, ep) && LL<double>::ok(q1, ep));
        if (left == 0) { lost = true; break; }
      }
      const double s0 = wave_sum63(reader ? LL<double>::val(q0) : 0.0);
      const double s1 = wave_sum63(reader ? LL<double>::val(q1) : 0.0);
      if (lane == 63) {
        tot[par][0][wave] = s0;
        tot[par][1][wave] = s1;
      }
    }
    if (lost) gaveup = 1;
    res_barrier();
    g0 = (tot[par][0][0] + tot[par][0][1]) + (tot[par][0][2] + tot[par][0][3]);
    g1 = (tot[par][1][0] + tot[par][1][1]) + (tot[par][1][2] + tot[par][1][3]);
    ++ep;
    return gaveup == 0;
  };

  // w = S (f − K u) on the block's rows after u += S x̂, and the partial sum of its square unscaled:
  // from the unscaled entries, in FP64, u of the coupled rows by their own slots (whose tag no
  // other hand-over has; the waits of the iterations in between keep a slot until it was read).
  // The arguments are read again: kept in scalar registers they would crowd the iteration.
  bool fresh = true;                         // u is still to be written
  auto true_residual = [&](double& sum) {
    const ResArgs<X>& z = *reinterpret_cast<const ResArgs<X>*>(res_kernargs());
    double* ul = reinterpret_cast<double*>(res_lds);
    int tt = t;
    asm volatile("" : "+v"(tt));             // no addresses made ahead of the loop
    const int32_t* own = z.orow + o0;
    const __amdgpu_buffer_rsrc_t ru = buf_rsrc(z.wu, 16u * (uint32_t)z.nslots);
    const __amdgpu_buffer_rsrc_t ro = buf_rsrc(reinterpret_cast<const U4*>(z.wu) + p0, 16u * (uint32_t)npub);
    res_barrier();                           // r̂ was read
#pragma unroll
    for (int k = 0; k < RT; ++k) {
      const int i = tt + k * kResT;
      if (i < nown) {
        const int32_t row = own[i], d = z.dofp ? z.dofp[row] : row;
        const double un = (fresh ? 0.0 : z.u[d]) + z.sc[d] * (double)x[k];
        z.u[d] = un;
        ul[i] = un;
        if (nb > 1) ll_put(ro, (uint32_t)i, un, ep);   // (dropped past the published rows)
      }
      x[k] = X(0);
      asm volatile("" ::: "memory");
    }
    fresh = false;
    for (int h = tt; h < nh; h += kResT) {
      const uint32_t at = (uint32_t)hl[h];
      U4 q = {};
      for (uint32_t left = (uint32_t)uniform((int)polls);; --left) {
        asm volatile("" ::: "memory");
        q = LL<double>::get(ru, at);
        if (LL<double>::ok(q, ep)) break;
        if (left == 0) { gaveup = 1; break; }
      }
      ul[nown + h] = LL<double>::val(q);
    }
    res_barrier();
    const uint32_t* iz = z.ai + (int64_t)b * NZ2 * z.Rp;
    const double* raw = z.raw + (int64_t)b * NZ * z.Rp;
#pragma unroll
    for (int k = 0; k < RT; ++k) {
      const int i = tt + k * kResT;
      w[k] = X(0);
      if (i < nown) {
        const int32_t row = own[i], d = z.dofp ? z.dofp[row] : row;
        double acc = z.f[d];
        if (z.raw) {
#pragma unroll 3
          for (int m = 0; m < NZ2; ++m) {
            const uint32_t q = iz[(int64_t)m * z.Rp + i];
            acc -= raw[(int64_t)(2 * m) * z.Rp + i] * ul[q & 0xffffu];
            if (2 * m + 1 < NZ) acc -= raw[(int64_t)(2 * m + 1) * z.Rp + i] * ul[q >> 16];
          }
        } else {
          const int32_t c0 = z.colptr[d], len = z.colptr[d + 1] - c0;
#pragma unroll 1
          for (int m = 0; m < len; ++m)
            acc -= z.nzval[c0 + m] * ul[(iz[(int64_t)(m >> 1) * z.Rp + i] >> (16 * (m & 1))) & 0xffffu];
        }
        sum += acc * acc;
        w[k] = (X)(z.sc[d] * acc);
      }
      asm volatile("" ::: "memory");         // one row's entries in flight
    }
    res_barrier();                           // u was read
  };

  double gstop = 0.0, prev = rrt, rzp0 = 0.0;   // rzp0: γ that the kept p belongs to, 0: p starts anew
  long long ticks = 0;
  int prods = 0, it = 0, handovers = 0, stall = 0, status = 0, done = 0, restart = 0;
  bool first = true, ok = true;
  for (;;) {
    for (;;) {                    // a stretch of the recurrence
      double g0 = 0.0, g1 = 0.0;
      // w = Â r̂ on the block's rows; γ = r̂·r̂ and δ = r̂·w (in a reseed r̂·p instead)
      const long long c0 = a.time ? wall_clock64() : 0;
#pragma unroll
      for (int k = 0; k < RT; ++k) {
        w[k] = X(0);
        if (k * kResT < nown) {
          if constexpr (RRES > 0)
            if (k < RRES) {
              const int kk = k < RRES ? k : 0;
              if constexpr (AHEAD) {
#pragma unroll
                for (int m = 0; m < NZ2; ++m)
                  asm volatile("" : "+v"(ai[kk][m]));   // keeps packed positions, not LDS addresses, in registers
                w[k] = gather_dot<X, NZ>(rl, av[kk], ai[kk]);
              } else {
                X acc = X(0);
#pragma unroll
                for (int m = 0; m < NZ2; ++m) {
                  asm volatile("" : "+v"(ai[kk][m]));
                  const uint32_t q = ai[kk][m];
                  acc += av[kk][2 * m] * at_lds(rl, q & 0xffffu);
                  if (2 * m + 1 < NZ) acc += av[kk][2 * m + 1 < NZ ? 2 * m + 1 : 0] * at_lds(rl, q >> 16);
                }
                w[k] = acc;
              }
            }
          if (k >= RRES) {
            const int rest = t + (k - RRES) * kResT;
            if (rest < a.nl) {
              X acc = X(0);
#pragma unroll
              for (int m = 0; m < NZ2; ++m) {
                const uint32_t q = lq[rest * QS + m];
                acc += lv[rest * NZ + 2 * m] * at_lds(rl, q & 0xffffu);
                if (2 * m + 1 < NZ) acc += lv[rest * NZ + 2 * m + 1] * at_lds(rl, q >> 16);
              }
              w[k] = acc;
            }
          }
        }                  // 0 on unused rows: their entries are 0
      }
      if (a.time) ticks += wall_clock64() - c0;
      ++prods;
      if (nb > 1) publish();
#pragma unroll
      for (int k = 0; k < RT; ++k)
        if (k * kResT < nown) {
          const X r = rl[il[k]];
          g0 += (double)r * (double)r;
          g1 += (double)r * (double)(first ? p[k] : w[k]);
        }
      ok = exchange(g0, g1, true);
      if (!ok) break;
      if (first) {
        // reseed: p made orthogonal to the new residual and extended, α = γ / p·ŝ
        const bool keep = rzp0 > 0.0 && g0 > 0.0;
        const double gam = g0 > 0.0 ? g1 / g0 : 0.0;
        const double conv = rrt > 0.0 ? tol2 / rrt : 0.0;
        gstop = uniform(g0 * (a.hold2 > conv ? a.hold2 : conv));
        const X be = (X)(keep ? g0 / rzp0 : 0.0), ga = (X)gam;
        double pq = 0.0, none = 0.0;
#pragma unroll
        for (int k = 0; k < RT; ++k) {
          const X r = rl[il[k]];
          p[k] = keep ? r + be * (p[k] - ga * r) : r;
          sv[k] = keep ? w[k] + be * (sv[k] - ga * w[k]) : w[k];
          pq += (double)p[k] * (double)sv[k];
        }
        for (int h = t; h < nh; h += kResT) sl[h] = keep ? wl[h] + be * (sl[h] - ga * wl[h]) : wl[h];
        ok = exchange(pq, none, false);
        if (!ok) break;
        alpha = pq > 0.0 ? g0 / pq : 0.0;
        if (!(pq > 0.0)) {          // p vanished (r̂ already zero): nothing to step
          done = restart = 1;
          break;
        }
        rzp = g0;                   // the first step moves x̂ and r̂ along the reseed's p, ŝ
      }
      double be = 0.0;
      if (!first) {
        be = g0 * irz;
        const double den = g1 - g0 * g0 * ira;
        const bool stop = g0 <= gstop;
        const bool brk = !(rzp > 0.0) || !(alpha != 0.0) || !(den > 0.0);
        if (stop || brk || it >= a.lim) {   // hand over: x̂, p and ŝ of the last step
          done = uniform(stop || brk ? 1 : 0);
          restart = uniform(!stop && brk ? 1 : 0);
          break;
        }
        alpha = g0 / den;
        rzp = g0;
      }
      ++it;
      const X al = (X)alpha, bx = (X)be;
#pragma unroll
      for (int k = 0; k < RT; ++k)
        if (k * kResT < nown) {
          const X r = rl[il[k]];
          if (!first) {
            p[k] = r + bx * p[k];
            sv[k] = w[k] + bx * sv[k];
          }
          x[k] += al * p[k];
          rl[il[k]] = r - al * sv[k];
        }
      for (int base = t; base < nh; base += 4 * kResT) {   // four rows' LDS reads in flight
        X sn[4], rn[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int h = base + k * kResT;
          if (h < nh) {
            sn[k] = first ? sl[h] : wl[h] + bx * sl[h];
            rn[k] = rl[nown + h];
          }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int h = base + k * kResT;
          if (h < nh) {
            sl[h] = sn[k];
            rl[nown + h] = rn[k] - al * sn[k];
          }
        }
      }
      first = false;
      res_barrier();
    }
    if (!ok) break;
    double g0 = 0.0, none = 0.0;
    true_residual(g0);
    if (nb > 1) publish();
    ok = exchange(g0, none, true);
    if (!ok) break;
    // the true residual: finished, or the next stretch starts from it
    rrt = uniform(g0);
    handovers += done;
    status = uniform(rrt <= tol2 ? 1 : 0);
    stall = uniform(rrt <= 0.81 * prev ? 0 : stall + 1);   // (a NaN stalls)
    prev = uniform(fmin(prev, rrt));
    if (status || it >= a.lim || stall >= kMaxStallRes) break;
#pragma unroll
    for (int k = 0; k < RT; ++k) {
      const int i = t + k * kResT;
      if (i < nown) rl[i] = w[k];
    }
    for (int h = t; h < nh; h += kResT) rl[nown + h] = wl[h];
    if (t == 0) rl[zero] = X(0);
    rzp0 = uniform(restart || !(rzp > 0.0) ? 0.0 : rzp);
    first = true;
    done = restart = 0;
    res_barrier();
  }
  const ResArgs<X>& z = *reinterpret_cast<const ResArgs<X>*>(res_kernargs());
  ResState* o = z.st + gr.x;
  if (!ok) {
    if (t == 0) o->lost = 1;
    return;
  }
  if (b == b0 && t == 0) {
    o->rr = rrt;
    o->iters = it;
    o->handovers = handovers;
    o->status = status;
    o->prods = prods;
    o->begin = begin;
    o->end = wall_clock64();
    o->epoch = ep;
  }
  if (b == z.grp[b].w && t == 0) o->ticks = ticks;
}

// ---- host ---------------------------------------------------------------------------------
// Most rows per block of the instantiated kernels (FP64 with 27 entries: LDS holds fewer, about 1,400).
static int res_most_rows(int nz, bool fp32) {
  return fp32 ? (nz == 9 ? 4096 : nz == 18 ? 2560 : 2048) : (nz == 9 ? 2048 : 1536);
}

static int res_entries(int widest) { return widest <= 9 ? 9 : widest <= 18 ? 18 : 27; }

// (several systems: their parts are less even, and a part's largest must fit)
static double res_fill_rows(int nz, bool fp32) { return 0.85 * res_most_rows(nz, fp32); }

int resident_blocks(int64_t rows, int widest, bool fp32) {
  return widest > 27 ? 0 : (int)std::max<double>(1.0, std::ceil((double)rows / res_fill_rows(res_entries(widest), fp32)));
}

int resident_most_blocks(const fem_ctx* c) {
  int ncu = 0;
  (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device);
  return std::min(ncu, kResMaxBlocks);
}

// The instantiated kernel for nz entries per row and R rows per block (null: too many).
// Resident rows are what the 256 VGPRs of a thread hold beside the vectors (512 threads, two
// waves per SIMD); the entries of further rows are in LDS.
template <typename X>
static const void* res_kernel(int nz, int R) {
  const int need = (R + kResT - 1) / kResT;
#define FEM_RES(NZ, RRES, RT) \
  if (nz == NZ && need <= RT) return (const void*)k_resident<X, NZ, RRES, RT>
  if constexpr (sizeof(X) == 4) {
    FEM_RES(9, 8, 8);
    FEM_RES(18, 5, 5);
    FEM_RES(27, 3, 4);
  } else {
    FEM_RES(9, 4, 4);
    FEM_RES(18, 3, 3);
    FEM_RES(27, 2, 3);
  }
#undef FEM_RES
  return nullptr;
}

// Elements of r̂ in LDS: its rows and a zero slot, or their u in FP64.
static int res_lds_r(const ResOp* o, size_t xb) { return xb == 4 ? 2 * o->nlocmax + 2 : o->nlocmax + 1; }

// LDS of a block with nl rows' entries in it: r̂, ŝ, w and the slots of the coupled rows, the entries
static size_t res_lds_bytes(const ResOp* o, size_t xb, int nl) {
  const size_t nz2 = (size_t)((o->nz + 1) / 2 | 1);
  return ((size_t)res_lds_r(o, xb) + 2 * (size_t)o->nhmax + (size_t)o->nz * nl) * xb + 4 * (nz2 * nl + (size_t)o->nhmax);
}

// Register rows of the instantiated kernels (kResT threads).
static int res_register_rows(int nz, bool fp32) {
  return kResT * (fp32 ? (nz == 9 ? 8 : nz == 18 ? 5 : 3) : (nz == 9 ? 4 : nz == 18 ? 3 : 2));
}

// Parts along each axis for nx × ny × nz positions of `per` rows each and at most `most` parts.
// An iteration's cost in cycles, fitted to timed stretches (2D and 3D, 18 to 256 parts): every
// kResT rows of the largest part begun (more where their entries are in LDS), its coupled rows,
// and every part's record read by all; parts too large for FP64 values only where nothing else
// is left.
struct ResCut {
  double cost = 1e300;
  int n[3] = {1, 1, 1};
};
// cuts[m]: the best with at most m parts.
static std::vector<ResCut> res_cuts(const double* ext, int dim, double per, int nz, int most) {
  std::vector<ResCut> cuts(most + 1);
  const double regs = kResT * (nz == 9 ? 4 : nz == 18 ? 3 : 2), cap = nz == 27 ? regs + 360.0 : regs;
  for (int x = 1; x <= most; ++x)
    for (int y = 1; x * y <= most; ++y) {
      if (dim < 2 && y > 1) break;
      for (int z = 1; x * y * z <= most; ++z) {
        if (dim < 3 && z > 1) break;
        const double bx = std::ceil(ext[0] / x - 1e-9), by = std::ceil(ext[1] / y - 1e-9),
                     bz = std::ceil(ext[2] / z - 1e-9);
        if (bx < 1 || by < 1 || bz < 1) continue;
        const double own = bx * by * bz;
        const double all = (x > 1 ? bx + 2 : bx) * (y > 1 ? by + 2 : by) * (z > 1 ? bz + 2 : bz);
        const double rounds = std::ceil(per * own / kResT);
        const double cost = rounds * (250.0 + 30.0 * nz) + (per * own > regs ? 1500.0 : 0.0) +
                            0.5 * per * (all - own) + 0.1 * per * own + 8.0 * x * y * z +
                            1e4 * std::max(0.0, per * own - cap);
        ResCut& c = cuts[x * y * z];
        if (cost < c.cost) c = ResCut{cost, {x, y, z}};
      }
    }
  for (int m = 1; m <= most; ++m)
    if (cuts[m - 1].cost <= cuts[m].cost) cuts[m] = cuts[m - 1];
  return cuts;
}

// Blocks per system, at most `total` of them: each the fewest that hold its rows, the others one by
// one to the system that is expected to take longest (its extent in rows, times an iteration's
// cost) as long as it gains.  cut: [ng][3].  false: they do not fit.
struct ResExtent {
  double ext[3], per, count;
  int dim;
};
static bool res_share(const std::vector<ResExtent>& e, int nz, int total, int most_rows, std::vector<int>* cut) {
  const int ng = (int)e.size();
  std::vector<int> m(ng), cap(ng);
  std::vector<double> its(ng);
  std::vector<std::vector<ResCut>> cuts(ng);
  int used = 0;
  for (int i = 0; i < ng; ++i) {
    cap[i] = (int)std::max<double>(1.0, std::min<double>(total, std::ceil(e[i].count / kResRows)));
    m[i] = (int)std::max<double>(1.0, std::ceil(e[i].count / (ng > 1 ? res_fill_rows(nz, true) : most_rows)));
    if (m[i] > cap[i]) return false;
    if (ng == 1) m[i] = cap[i];
    its[i] = e[i].ext[0] + e[i].ext[1] + e[i].ext[2];
    used += m[i];
    cuts[i] = res_cuts(e[i].ext, e[i].dim, e[i].per, nz, cap[i]);
  }
  if (used > total) return false;
  std::vector<bool> last(ng, false);
  for (;;) {
    int at = -1;
    for (int i = 0; i < ng; ++i)
      if (!last[i] && (at < 0 || its[i] * cuts[i][m[i]].cost > its[at] * cuts[at][m[at]].cost)) at = i;
    if (at < 0) break;
    const int most = std::min(cap[at], m[at] + total - used);
    int k = m[at] + 1;
    while (k <= most && !(cuts[at][k].cost < cuts[at][m[at]].cost)) ++k;
    if (k <= most) {
      used += k - m[at];
      m[at] = k;
    } else {
      last[at] = true;
    }
  }
  cut->clear();
  for (int i = 0; i < ng; ++i)
    for (int d = 0; d < 3; ++d) cut->push_back(cuts[i][m[i]].n[d]);
  return true;
}

static int res_build(fem_ctx* c, ResOp* o, const ResSource& s, const ResRows& rows, int nz, int most_rows) {
  int maxlds = 0, coop = 0;
  (void)hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device);
  (void)hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, c->device);
  const int64_t n = rows.n;
  const int ng = s.nsys > 0 ? s.nsys : 1;
  o->state = -1;
  o->nz = nz;
  o->ng = ng;
  std::vector<ResSystem> sys(ng);
  int64_t longest = 0;
  for (int i = 0; i < ng; ++i) {
    sys[i] = ResSystem{s.nsys > 0 ? s.sys[2 * i] : 0, s.nsys > 0 ? s.sys[2 * i + 1] : (int32_t)n, {}, {}};
    longest = std::max<int64_t>(longest, sys[i].row1 - sys[i].row0);
  }
  const int words = (int)((longest + 31) / 32);
  const int lds = 4 * (words + (words + 7) / 8);
  if (lds > maxlds - kStaticLds) return FEM_OK;   // a bitmap of the rows (more than a million): far too many anyway

  struct Scratch {                          // freed on every way out
    int32_t *node = nullptr, *part = nullptr, *hist = nullptr, *size = nullptr, *rank = nullptr, *cnt = nullptr;
    int4* slab = nullptr;
    ResSystem* sys = nullptr;
    uint8_t* flag = nullptr;
    double* geom = nullptr;
    ~Scratch() {
      dev_free(&node); dev_free(&part); dev_free(&hist); dev_free(&size); dev_free(&rank); dev_free(&cnt);
      dev_free(&slab); dev_free(&sys); dev_free(&flag); dev_free(&geom);
    }
  } w;
  int rc;
  ResPos g{};
  g.src = s.src;
  g.px = s.px;
  g.pxy = s.pxy;
  g.dofp = s.dofp;
  g.dim = s.dim;
  g.node = s.node;
  for (int d = 0; d < 3; ++d) g.x[d] = s.x[d];
  if (s.src == 0 && !s.node) {   // a node of each dof's first cell (its own node for a Q1 field)
    const int64_t nc = c->ncells, nd = c->ndpc, npc = c->npc;
    if (nd <= 0 || npc <= 0 || (int64_t)c->h_cell_dofs.size() != nc * nd || (int64_t)c->h_cell_nodes.size() != nc * npc)
      return FEM_OK;
    if (c->ndofs != n) return FEM_OK;         // dofs uploaded after the pattern: not those of its rows
    std::vector<int32_t> node(n, 0), at(nd);
    std::vector<uint8_t> seen(n, 0);
    for (int64_t a = 0; a < nd; ++a) at[a] = (int32_t)(a * npc / nd);
    for (int64_t e = 0; e < nc; ++e)
      for (int64_t a = 0; a < nd; ++a) {
        const int32_t d = c->h_cell_dofs[e * nd + a];
        if (!seen[d]) {
          seen[d] = 1;
          node[d] = c->h_cell_nodes[e * npc + at[a]];
        }
      }
    if ((rc = copy_alloc(c, &w.node, n))) return rc;
    FEM_HIP(c, hipMemcpy(w.node, node.data(), 4 * n, hipMemcpyHostToDevice));
    g.node = w.node;
    g.dim = c->sdim;
    for (int d = 0; d < 3; ++d) g.x[d] = c->d_x[d];
  }
  std::vector<double> geom(10 * ng);
  if ((rc = copy_alloc(c, &w.geom, 10 * ng)) || (rc = copy_alloc(c, &w.sys, ng))) return rc;
  FEM_HIP(c, hipMemcpyAsync(w.sys, sys.data(), sizeof(ResSystem) * ng, hipMemcpyHostToDevice, c->stream));
  k_res_geom<<<ng, 1024, 0, c->stream>>>(g, rows, w.sys, nz, w.geom);
  FEM_HIP(c, hipGetLastError());
  FEM_HIP(c, hipMemcpyAsync(geom.data(), w.geom, sizeof(double) * 10 * ng, hipMemcpyDeviceToHost, c->stream));
  FEM_HIP(c, hipStreamSynchronize(c->stream));
  std::vector<ResExtent> ext(ng);
  for (int i = 0; i < ng; ++i) {
    const double* e = &geom[10 * i];
    double cells = 1.0;
    for (int d = 0; d < 3; ++d) {
      const double len = e[3 + d] - e[d];
      const bool flat = d >= g.dim || !(len > 0.0);
      sys[i].lo[d] = e[d];
      sys[i].inv[d] = flat ? 0.0 : (kResBins - 0.5) / len;
      ext[i].ext[d] = !flat && e[6 + d] > 0.0 ? std::max(1.0, std::floor(len / e[6 + d] + 1.5)) : 1.0;
      cells *= ext[i].ext[d];
    }
    ext[i].count = e[9];
    ext[i].per = e[9] / cells;
    ext[i].dim = g.dim;
  }
  std::vector<int> cut;
  if (!res_share(ext, nz, resident_most_blocks(c), most_rows, &cut)) return FEM_OK;
  int nb = 0;
  std::vector<int4> grp;
  for (int i = 0; i < ng; ++i) {
    const int m = cut[3 * i] * cut[3 * i + 1] * cut[3 * i + 2];
    for (int k = 0; k < m; ++k) grp.push_back(make_int4(i, nb, m, nb));
    if (m > 1 && !coop) return FEM_OK;
    nb += m;
  }
  o->nb = nb;
  const int grid = (int)std::min<int64_t>(2048, (n + 255) / 256);
  const int gridy = (int)std::max<int64_t>(1, std::min<int64_t>(2048 / ng, (longest + 255) / 256));
  if ((rc = copy_alloc(c, &w.part, n)) || (rc = copy_alloc(c, &w.hist, (size_t)kResBins * nb)) ||
      (rc = copy_alloc(c, &w.flag, n)) || (rc = copy_alloc(c, &w.size, 2 * nb)) || (rc = copy_alloc(c, &w.rank, n)) ||
      (rc = copy_alloc(c, &w.cnt, nb)) || (rc = copy_alloc(c, &w.slab, nb)) || (rc = copy_alloc(c, &o->grp, nb)) ||
      (rc = copy_alloc(c, &o->oofs, nb + 1)) || (rc = copy_alloc(c, &o->pofs, nb + 1)) ||
      (rc = copy_alloc(c, &o->hoff, nb + 1)))
    return rc;
  FEM_HIP(c, hipMemcpyAsync(w.sys, sys.data(), sizeof(ResSystem) * ng, hipMemcpyHostToDevice, c->stream));
  FEM_HIP(c, hipMemsetAsync(w.part, 0xff, 4 * n, c->stream));
  FEM_HIP(c, hipMemsetAsync(w.flag, 0, n, c->stream));
  FEM_HIP(c, hipMemsetAsync(w.size, 0, 8 * nb, c->stream));
  k_res_start<<<dim3(gridy, ng), 256, 0, c->stream>>>(g, w.sys, w.part);
  std::vector<int> per(ng, 1);              // slabs of each system so far
  for (int d = 0; d < 3; ++d) {
    std::vector<int4> slab;
    int next = 0;
    bool any = false;
    for (int i = 0; i < ng; ++i) {
      any = any || cut[3 * i + d] > 1;
      for (int k = 0; k < per[i]; ++k) {
        slab.push_back(make_int4(i, cut[3 * i + d], next, 0));
        next += cut[3 * i + d];
      }
    }
    if (!any) continue;
    for (int i = 0; i < ng; ++i) per[i] *= cut[3 * i + d];
    const int ns = (int)slab.size();
    FEM_HIP(c, hipMemcpyAsync(w.slab, slab.data(), sizeof(int4) * ns, hipMemcpyHostToDevice, c->stream));
    FEM_HIP(c, hipMemsetAsync(w.hist, 0, (size_t)4 * kResBins * ns, c->stream));
    k_res_hist<<<grid, 256, 0, c->stream>>>(g, w.sys, w.slab, n, d, w.part, w.hist);
    k_res_cut<<<ns, 256, 0, c->stream>>>(w.slab, w.hist);
    k_res_split<<<grid, 256, 0, c->stream>>>(g, w.sys, w.slab, n, d, w.hist, w.part);
    FEM_HIP(c, hipStreamSynchronize(c->stream));   // slab goes
  }
  k_res_shared<<<grid, 256, 0, c->stream>>>(rows, nz, w.part, w.flag, w.size);
  FEM_HIP(c, hipGetLastError());
  std::vector<int32_t> h(nb), off(nb + 1, 0);
  FEM_HIP(c, hipMemcpyAsync(h.data(), w.size, 4 * nb, hipMemcpyDeviceToHost, c->stream));
  FEM_HIP(c, hipStreamSynchronize(c->stream));
  o->Rmax = 0;
  for (int b = 0; b < nb; ++b) {
    off[b + 1] = off[b] + h[b];
    o->Rmax = std::max(o->Rmax, h[b]);
    if (h[b] > h[grp[grp[b].y].w]) grp[grp[b].y].w = b;
  }
  for (int b = 0; b < nb; ++b) grp[b].w = grp[grp[b].y].w;
  FEM_HIP(c, hipMemcpyAsync(o->grp, grp.data(), sizeof(int4) * nb, hipMemcpyHostToDevice, c->stream));
  if (o->Rmax > 8192) return FEM_OK;
  int pow2 = 2;
  while (pow2 < o->Rmax) pow2 *= 2;
  o->Rp = (o->Rmax + 63) / 64 * 64;
  FEM_HIP(c, hipMemcpyAsync(o->oofs, off.data(), 4 * (nb + 1), hipMemcpyHostToDevice, c->stream));
  if ((rc = copy_alloc(c, &o->orow, off[nb]))) return rc;
  k_res_gather<<<grid, 256, 0, c->stream>>>(n, w.part, w.flag, o->oofs, w.size + nb, o->orow);
  k_res_sort<<<nb, 1024, 4 * pow2, c->stream>>>(pow2, o->oofs, o->orow, w.rank, w.cnt);
  FEM_HIP(c, hipGetLastError());
  std::vector<int32_t> pub(nb + 1, 0), hof(nb + 1, 0);
  FEM_HIP(c, hipMemcpyAsync(h.data(), w.cnt, 4 * nb, hipMemcpyDeviceToHost, c->stream));
  FEM_HIP(c, hipStreamSynchronize(c->stream));
  for (int b = 0; b < nb; ++b) pub[b + 1] = pub[b] + h[b];
  o->nslots = pub[nb];
  (void)res_dynamic_lds((const void*)k_res_count, maxlds);
  (void)res_dynamic_lds((const void*)k_res_fill, maxlds);
  k_res_count<<<nb, 256, 4 * words, c->stream>>>(rows, nz, words, w.sys, o->grp, w.part, o->oofs, o->orow, w.cnt);
  FEM_HIP(c, hipGetLastError());
  FEM_HIP(c, hipMemcpyAsync(h.data(), w.cnt, 4 * nb, hipMemcpyDeviceToHost, c->stream));
  FEM_HIP(c, hipStreamSynchronize(c->stream));
  o->nlocmax = o->nhmax = 0;
  for (int b = 0; b < nb; ++b) {
    hof[b + 1] = hof[b] + h[b];
    o->nhmax = std::max(o->nhmax, h[b]);
    o->nlocmax = std::max(o->nlocmax, off[b + 1] - off[b] + h[b]);
  }
  o->nlocmax += o->nlocmax & 1;             // keeps what follows r̂ and its zero slot apart
  if (o->nlocmax > 65535) return FEM_OK;    // positions are 16 bits (and byte offsets: res_lds_rows)
  const int nz2 = (nz + 1) / 2;
  if ((rc = copy_alloc(c, &o->hrow, hof[nb])) || (rc = copy_alloc(c, &o->hslot, hof[nb])) ||
      (rc = copy_alloc(c, &o->ai, (size_t)nb * nz2 * o->Rp)) || (rc = copy_alloc(c, &o->wx, (size_t)8 * o->nslots)) ||
      (rc = copy_alloc(c, &o->wu, (size_t)4 * o->nslots)) || (rc = copy_alloc(c, &o->rec, kRecWords)))
    return rc;
  FEM_HIP(c, hipMemcpyAsync(o->pofs, pub.data(), 4 * (nb + 1), hipMemcpyHostToDevice, c->stream));
  FEM_HIP(c, hipMemcpyAsync(o->hoff, hof.data(), 4 * (nb + 1), hipMemcpyHostToDevice, c->stream));
  FEM_HIP(c, hipMemsetAsync(o->wx, 0, (size_t)32 * o->nslots, c->stream));
  FEM_HIP(c, hipMemsetAsync(o->wu, 0, (size_t)16 * o->nslots, c->stream));
  FEM_HIP(c, hipMemsetAsync(o->rec, 0, 4 * kRecWords, c->stream));
  if (hipHostMalloc((void**)&o->st, sizeof(ResState) * ng, hipHostMallocDefault) != hipSuccess)
    return set_error(c, FEM_ERR_OOM, "hipHostMalloc failed");
  k_res_fill<<<nb, 256, lds, c->stream>>>(rows, nz, o->Rp, words, w.sys, o->grp, w.part, w.rank, o->oofs, o->orow,
                                          o->pofs, o->hoff, o->hrow, o->hslot, o->ai);
  FEM_HIP(c, hipGetLastError());
  FEM_HIP(c, hipStreamSynchronize(c->stream));   // host vectors and scratch go
  o->epoch = 0;
  o->state = 1;
  return FEM_OK;
}

// Rows whose entries LDS holds: those beyond the register rows; −1 when they do not fit.
static int res_lds_rows(const ResOp* o, bool fp32, int maxlds) {
  const size_t xb = fp32 ? 4 : 8, base = res_lds_bytes(o, xb, 0), per = o->nz * xb + 4 * ((o->nz + 1) / 2 | 1);
  const size_t cap = (size_t)maxlds - kStaticLds;
  if (base > cap || (o->nlocmax + 1) * xb > 65536) return -1;   // 16-bit byte offsets into r̂
  const int rest = std::max(0, o->Rmax - res_register_rows(o->nz, fp32));
  return base + rest * per > cap ? -1 : rest;
}

// Whether `rows` rows may fit in this precision: the fullest block has at least its share of them,
// and, in a mesh with little boundary (26 of 27 entries per row on average), no fewer coupled rows than
// a cube.
static bool res_may_fit(const fem_ctx* c, int64_t rows, int nz, bool fp32, bool one) {
  const int blocks = resident_most_blocks(c);
  if (rows > (int64_t)blocks * res_most_rows(nz, fp32)) return false;
  if (!one || nz != 27 || c->nnz < 26 * rows) return true;
  int maxlds = 0;
  (void)hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device);
  ResOp e;
  e.nz = nz;
  e.Rmax = (int)((rows + blocks - 1) / blocks);
  e.nhmax = (int)(std::pow(std::cbrt((double)e.Rmax) + 2.0, 3.0) - e.Rmax);
  e.nlocmax = e.Rmax + e.nhmax;
  return res_lds_rows(&e, fp32, maxlds) >= 0;
}

static int res_prepare(fem_ctx* c, ResOp* o, const ResSource& s, const double* sc, int jacobi, bool fp32, bool* ok) {
  if (o->state == -1) return FEM_OK;
  ResRows rows{s.src, s.dim, s.n, s.npad, s.px, s.pxy, c->d_colptr, c->d_rowval, s.dofp, s.map, c->d_nzval, sc, s.kc, s.val,
               s.t, {}};
  for (int i = 0; i < 8; ++i) rows.f[i] = s.f[i];
  int rc;
  if (o->state == 0) {
    const int widest = s.widest;
    const int nz = res_entries(widest);
    int64_t all = s.nsys > 0 ? 0 : c->n;    // (s.n counts a lattice's padding too)
    for (int i = 0; i < s.nsys; ++i) all += s.sys[2 * i + 1] - s.sys[2 * i];
    // too large in this precision: nothing is built, which would take about 5 ms at 0.4 M rows (first
    // FP64 solves that then took the separate kernels: 72³ hexes 10.8 → 6.2 ms, 724² quads 33.4 → 28.6)
    if (widest > 27 || all < 1 || !res_may_fit(c, all, nz, fp32, s.nsys == 0)) return FEM_OK;
    o->state = -1;
    if ((rc = res_build(c, o, s, rows, nz, res_most_rows(nz, true)))) return rc;
    if (o->state == -1) return FEM_OK;
  }
  int maxlds = 0;
  (void)hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device);
  if (!(fp32 ? res_kernel<float>(o->nz, o->Rmax) : res_kernel<double>(o->nz, o->Rmax)) ||
      res_lds_rows(o, fp32, maxlds) < 0)
    return FEM_OK;
  const int pi = fp32 ? 0 : 1;
  const size_t len = (size_t)o->nb * o->nz * o->Rp;
  if (fp32 && !o->val32 && ((rc = copy_alloc(c, &o->val32, len)) || (rc = copy_alloc(c, &o->raw, len)))) return rc;
  if (!fp32 && !o->val64 && (rc = copy_alloc(c, &o->val64, len))) return rc;
  if (o->ver[pi] != c->nzval_version + 1 || o->aux[pi] != c->aux_version + 1 || o->jac[pi] != jacobi ||
      o->vsrc[pi] != s.src) {
    const int g = (int)std::min<int64_t>(8192, ((int64_t)o->nb * o->Rp + 255) / 256);
    if (fp32) k_res_vals<float><<<g, 256, 0, c->stream>>>(rows, o->nz, o->Rp, o->nb, o->oofs, o->orow, o->val32,
                                                        o->raw);
    else k_res_vals<double><<<g, 256, 0, c->stream>>>(rows, o->nz, o->Rp, o->nb, o->oofs, o->orow, o->val64,
                                                    nullptr);
    FEM_HIP(c, hipGetLastError());
    o->ver[pi] = c->nzval_version + 1;
    o->aux[pi] = c->aux_version + 1;
    o->jac[pi] = jacobi;
    o->vsrc[pi] = s.src;
  }
  *ok = true;
  return FEM_OK;
}

int resident_prepare(fem_ctx* c, ResOp** op, const ResSource& s, const double* sc, int jacobi, bool fp32, bool* ok) {
  *ok = false;
  if (!*op) *op = new ResOp();
  const int rc = res_prepare(c, *op, s, sc, jacobi, fp32, ok);
  if (!no_memory(c, rc)) return rc;
  resident_free(op);
  *op = new ResOp();
  (*op)->state = -1;
  return FEM_OK;
}

template <typename X>
int resident_run(fem_ctx* c, ResOp* o, const ResSource& s, const double* sc, const double* f, double* u,
                 const double* in, double bnorm2, double tol2, double hold_factor2, int lim, const ResState** out,
                 bool* launched) {
  *launched = false;
  // exchange numbers: one per product and two more per hand-over, of which seven in a row may
  // do without a product; started over before lim of those could reach 2³²
  lim = std::min(lim, 1 << 25);
  if (o->epoch > 0xffffffffu - 32u * (uint32_t)lim - 64u) {
    FEM_HIP(c, hipMemsetAsync(o->wx, 0, (size_t)32 * o->nslots, c->stream));
    FEM_HIP(c, hipMemsetAsync(o->wu, 0, (size_t)16 * o->nslots, c->stream));
    FEM_HIP(c, hipMemsetAsync(o->rec, 0, 4 * kRecWords, c->stream));
    o->epoch = 0;
  }
  int maxlds = 0;
  FEM_HIP(c, hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device));
  constexpr bool fp32 = sizeof(X) == 4;
  const int nl = res_lds_rows(o, fp32, maxlds);
  ResArgs<X> a{};
  a.Rp = o->Rp;
  a.nslots = o->nslots;
  a.nl = nl;
  a.rl0 = res_lds_r(o, sizeof(X));
  a.nhmax = o->nhmax;
  a.grp = o->grp;
  a.oofs = o->oofs;
  a.orow = o->orow;
  a.pofs = o->pofs;
  a.hoff = o->hoff;
  a.hrow = o->hrow;
  a.hslot = o->hslot;
  a.ai = o->ai;
  a.val = fp32 ? reinterpret_cast<const X*>(o->val32) : reinterpret_cast<const X*>(o->val64);
  a.raw = fp32 ? o->raw : nullptr;
  a.colptr = c->d_colptr;
  a.nzval = c->d_nzval;
  a.dofp = s.dofp;
  a.f = f;
  a.sc = sc;
  a.u = u;
  a.in = in;
  a.st = o->st;
  a.wx = o->wx;
  a.wu = o->wu;
  a.rec = o->rec;
  a.in0[0] = bnorm2;
  a.in0[1] = tol2;
  a.hold2 = hold_factor2;
  a.epoch = o->epoch + 1u;
  a.polls = c->res_polls;
  a.lim = lim;
  a.time = c->tune.time_kernels;
  std::fill(o->st, o->st + o->ng, ResState{});
  const void* k = res_kernel<X>(o->nz, o->Rmax);
  const size_t lds = res_lds_bytes(o, sizeof(X), nl);
  FEM_HIP(c, res_dynamic_lds(k, maxlds));
  void* args[] = {&a};
  const hipError_t e = o->nb == o->ng ? hipLaunchKernel(k, dim3(o->nb), dim3(kResT), args, lds, c->stream)
                                      : hipLaunchCooperativeKernel(k, dim3(o->nb), dim3(kResT), args, (unsigned)lds,
                                                                   c->stream);
  if (e != hipSuccess) {   // not as many blocks at once as the device should hold
    (void)hipGetLastError();
    return FEM_OK;
  }
  *launched = true;
  FEM_HIP(c, hipStreamSynchronize(c->stream));
  for (int i = 0; i < o->ng; ++i) o->epoch = std::max(o->epoch, o->st[i].epoch);
  *out = o->st;
  return FEM_OK;
}

template int resident_run<float>(fem_ctx*, ResOp*, const ResSource&, const double*, const double*, double*,
                                 const double*, double, double, double, int, const ResState**, bool*);
template int resident_run<double>(fem_ctx*, ResOp*, const ResSource&, const double*, const double*, double*,
                                  const double*, double, double, double, int, const ResState**, bool*);

}  // namespace fem
