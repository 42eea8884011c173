// Resident CG on the stored Q2 hex³ element matrices (81 × 81 per cell): the stretches of
// fem_resident_cells.hip (one cooperative launch between two hand-overs, the fold and the
// exchange as there) for meshes of up to kElMost × 256 cells, straight or distorted.
//
// What bounds the separate kernels there is not the element matrices (28 MB in FP32 at 12×10×9
// cells, read in about 6 µs) but three dependent launches per iteration: 26 µs.  Here a block
// owns up to kElMost neighbouring cells and keeps their scaled matrices S Ke S in registers, one
// row of one cell per thread; a thread also holds p, ŝ, x̂, r̂ of one dof of the block's cells.
// Dofs that several blocks have are held by each of them.  One exchange per iteration: a block
// publishes its cells' sum for every dof that others have too, with its partials of γ = r̂·r̂ (dofs
// it has first) and δ = r̂·w (over cells, before anything is exchanged: Σ r̂ₑ·Âₑr̂ₑ), and reads all
// blocks' sums of its own dofs.  Those are added in block order by everyone, so the copies of a dof
// stay equal bit for bit.
//
// Measured, µs per iteration with the hand-overs, separate kernels → here: mixed solver, 12×10×9
// cells (29,925 dofs) 28.1 → 5.3, 8×8×7 22.8 → 4.8, 5×4×4 23.7 → 4.4; FP64 solver, 12×11×10 28.7 → 6.0,
// 8×8×7 21.6 → 5.2.  Of an iteration in FP32 0.5 µs are products (FP64: 1.0), the rest is the
// exchange and, once per hand-over, the FP64 residual and the host.
#include <algorithm>
#include <cmath>
#include <numeric>

#include "fem_resident_dev.h"

namespace fem {

constexpr int kElMost = 6;             // cells per block: 6 · 81 rows of 512 threads
constexpr int kElAim = 5;              // cells per block when there are enough blocks (3 to 6: within 5%)
constexpr int kElShare = 8;            // blocks that may have one dof

struct ElemsOp {
  int state = 0;                       // 1 usable, −1 does not fit
  int nb = 0, nslots = 0;
  int32_t* cell = nullptr;             // [nb][kElMost] cells, −1: none
  int32_t* dof = nullptr;              // [nb][kResT] dof of each thread (bit 30: first block that has it), −1: none
  int32_t* pos = nullptr;              // [nb][kElMost][kResT] rows (cell, row of the cell) of a thread's dof
  int32_t* slot = nullptr;             // [nb][kResT] published slot of a thread's dof, −1: no other block has it
  int32_t* from = nullptr;             // [nb][kElShare][kResT] slots of a dof, in block order
  int32_t* nfrom = nullptr;            // [nb][kResT] their number, 0: no other block has it
  float* val32 = nullptr;              // [nb][81][kResT] rows of the scaled matrices
  double* val64 = nullptr;
  uint32_t *wx = nullptr, *rec = nullptr;
  uint32_t epoch = 0;
};

void elems_free(ElemsOp** op) {
  if (!*op) return;
  ElemsOp* o = *op;
  dev_free(&o->cell); dev_free(&o->dof); dev_free(&o->pos); dev_free(&o->slot); dev_free(&o->from);
  dev_free(&o->nfrom); dev_free(&o->val32); dev_free(&o->val64); dev_free(&o->wx); dev_free(&o->rec);
  delete o;
  *op = nullptr;
}

// Row r of a cell in LDS: cell · stride + r (16-byte aligned rows of r̂).
template <typename X>
constexpr int kElStride = sizeof(X) == 4 ? 84 : 82;

// Rows of S Ke S of each block's cells (0 in rows and columns of prescribed dofs), rounded once.
template <typename X, typename P>
__global__ __launch_bounds__(kResT) void k_elems_vals(const int32_t* __restrict__ cell,
                                                      const int32_t* __restrict__ cnode, const P* __restrict__ ke,
                                                      const double* __restrict__ sc, const uint8_t* __restrict__ isc,
                                                      X* __restrict__ val) {
  const int b = blockIdx.x, t = threadIdx.x, e = t / 81, r = t - 81 * e, a = r / 3, i = r - 3 * a;
  const int32_t c = e < kElMost ? cell[b * kElMost + e] : -1;
  const int32_t row = c >= 0 ? 3 * cnode[c * 27 + a] + i : 0;
  const double sr = c >= 0 && !(isc && isc[row]) ? sc[row] : 0.0;
  X* out = val + (int64_t)b * 81 * kResT + t;
  for (int n = blockIdx.y * 9; n < blockIdx.y * 9 + 9; ++n) {   // 27 nodes in three blocks
    const int64_t node = c >= 0 ? cnode[c * 27 + n] : 0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int64_t col = 3 * node + j;
      const double sj = c >= 0 && !(isc && isc[col]) ? sc[col] : 0.0;
      const double k = c >= 0 ? (double)ke[(int64_t)c * (27 * 252) + n * 252 + (3 * i + j) * 28 + a] : 0.0;
      out[(int64_t)(3 * n + j) * kResT] = (X)(k * (sr * sj));
    }
  }
}

template <typename X>
struct ElemsArgs {
  int nb, nslots;
  const int32_t *cell, *dof, *pos, *slot, *from, *nfrom;
  const X* val;
  const uint8_t* isc;
  const int32_t* diag;
  const double *nzval, *res, *sc;
  X *p, *sv;
  double* u;
  Scal* s;
  uint32_t *wx, *rec;
  double hold2, tol2;
  uint32_t epoch, polls;
  int restart, lim, time;
};

template <typename X>
__global__ __launch_bounds__(kResT) void k_resident_elems(ElemsArgs<X> a) {
  constexpr int ST = kElStride<X>, V = 16 / sizeof(X);
  typedef X XV __attribute__((ext_vector_type(V)));
  __shared__ __align__(16) X re[kElMost * ST + V];   // r̂ by cell rows; the last: of no row
  __shared__ X yl[kElMost * ST + V];                 // Âₑ r̂ₑ; the last: 0
  __shared__ double red[2][2][kResWaves];
  __shared__ double tot[2][2][4];
  __shared__ int gaveup;
  __shared__ uint32_t polls;                 // what a wait may take (in LDS: scalar registers are short)
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int b = blockIdx.x;
  const double rzp0 = a.s->rzp, rr0 = a.s->rr;
  const bool keep0 = !a.restart && !a.s->restart && rzp0 > 0.0;
  const int e = t / 81, er = t - 81 * e;
  const bool row = e < kElMost && a.cell[b * kElMost + min(e, kElMost - 1)] >= 0;
  const int at = row ? e * ST + er : 0;
  X av[81];
#pragma unroll
  for (int j = 0; j < 81; ++j) av[j] = a.val[((int64_t)b * 81 + j) * kResT + t];
  const int32_t dw = a.dof[b * kResT + t];
  const bool own = dw >= 0 && (dw & (1 << 30));
  const int32_t d = dw >= 0 ? dw & ~(1 << 30) : 0;
  const int32_t slot = a.slot[b * kResT + t], nfrom = a.nfrom[b * kResT + t];
  int pos[kElMost], from[kElShare];
#pragma unroll
  for (int k = 0; k < kElMost; ++k) {
    const int32_t q = a.pos[(b * kElMost + k) * kResT + t];
    pos[k] = q < 0 ? kElMost * ST : (q / 81) * ST + q % 81;
  }
#pragma unroll
  for (int k = 0; k < kElShare; ++k) from[k] = a.from[(b * kElShare + k) * kResT + t];
  int widest = nfrom;                        // of the wave
  for (int o = 32; o > 0; o >>= 1) widest = max(widest, __shfl_xor(widest, o, 64));
  widest = uniform(widest);
  X r = X(0), p = X(0), sv = X(0), x = X(0), w = X(0), pd = X(0);
  if (dw >= 0) {
    r = (X)(a.sc[d] * a.res[d]);
    if (keep0) {
      p = a.p[d];
      sv = a.sv[d];
    }
    if (a.isc && a.isc[d]) pd = (X)(a.sc[d] * a.sc[d] * a.nzval[a.diag[d]]);
  }
  for (int i = t; i < kElMost * ST + V; i += kResT) re[i] = yl[i] = X(0);
  if (t == 0) {
    gaveup = 0;
    polls = a.polls;
  }
  res_barrier();
  auto spread = [&]() {                      // r̂ to the rows of the cells
#pragma unroll
    for (int k = 0; k < kElMost; ++k)
      if (pos[k] < kElMost * ST) re[pos[k]] = r;
  };
  spread();
  res_barrier();

  uint32_t ep = a.epoch;
  const __amdgpu_buffer_rsrc_t rw = buf_rsrc(a.wx, (uint32_t)(2 * sizeof(typename LL<X>::W)) * (uint32_t)a.nslots);
  const __amdgpu_buffer_rsrc_t rr = buf_rsrc(a.rec, (uint32_t)(2 * kResCopies * 2 * 16) * kResMaxBlocks);
  double rzp = 0.0, alpha = 0.0, irz = 0.0, ira = 0.0;   // γ and α of the last step; 1 / γ, 1 / (γ α)
  // Sums g0, g1 over all blocks; with `halo`, completes w by the sums of the other blocks.  Every
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
    if (a.nb == 1) {
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
    const uint32_t most = (uint32_t)uniform((int)in_lds);
    const uint32_t rec = (uint32_t)(par * kResCopies * 2 * kResMaxBlocks);
    if (t < 2 * kResCopies) {
      double sum = 0.0;
#pragma unroll
      for (int i = 0; i < kResWaves; ++i) sum += red[par][t & 1][i];
      ll_put(rr, rec + (uint32_t)(t * kResMaxBlocks + b), sum, ep);
    }
    const uint32_t rin = rec + (uint32_t)((b % kResCopies) * 2 * kResMaxBlocks + t);
    if (halo) {   // reciprocals of the last step's scalars, while the values travel
      irz = 1.0 / rzp;
      ira = 1.0 / (rzp * alpha);
    }
    const bool reader = t < a.nb;      // thread t reads block t's record
    bool lost = false, need = reader;
    U4 q0 = {}, q1 = {};
    if (halo && widest > 0) {          // (spare reads repeat a slot that is published)
      const uint32_t wi = (ep & 1u) * (uint32_t)a.nslots;
      typename LL<X>::W hv[kElShare];
      for (uint32_t left = most;; --left) {
        asm volatile("" ::: "memory");
        bool ok = true;
        if (need) {
          q0 = LL<double>::get(rr, rin);
          q1 = LL<double>::get(rr, rin + kResMaxBlocks);
        }
#pragma unroll
        for (int k = 0; k < kElShare; ++k)
          if (k < widest) hv[k] = LL<X>::get(rw, wi + (uint32_t)from[k]);
#pragma unroll
        for (int k = 0; k < kElShare; ++k)
          if (k < widest) ok = ok && LL<X>::ok(hv[k], ep);
        if (need) need = !(LL<double>::ok(q0, ep) && LL<double>::ok(q1, ep));
        if (ok) break;
        if (left == 0) { lost = true; break; }
      }
      X sum = X(0);
#pragma unroll
      for (int k = 0; k < kElShare; ++k)
        if (k < widest && k < nfrom) sum += LL<X>::val(hv[k]);
      if (nfrom > 0) w = sum;
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

  double rz = 0.0, rz0 = 0.0, gstop = 0.0, beta = 0.0, gam = 0.0, pq = 0.0;
  long long ticks = 0;
  int done = 0, restart = 0, prods = 0, it = 0;
  bool first = true, ok = true;
  for (;;) {
    const long long c0 = a.time ? wall_clock64() : 0;
    // the cells' products (all threads of a cell read the same r̂)
    X acc = X(0);
    {
      const XV* rv = reinterpret_cast<const XV*>(re + (row ? e * ST : 0));
#pragma unroll
      for (int q = 0; q < (81 + V - 1) / V; ++q) {
        const XV v = rv[q];
#pragma unroll
        for (int k = 0; k < V; ++k)
          if (q * V + k < 81) acc += av[q * V + k] * v[k];
      }
    }
    double g0 = 0.0, g1 = 0.0;
    if (row) {
      yl[at] = acc;
      if (!first) g1 = (double)re[at] * (double)acc;
    }
    res_barrier();
    w = X(0);
#pragma unroll
    for (int k = 0; k < kElMost; ++k) w += yl[pos[k]];
    if (a.time) ticks += wall_clock64() - c0;
    ++prods;
    if (slot >= 0) ll_put(rw, (ep & 1u) * (uint32_t)a.nslots + (uint32_t)slot, w, ep);
    if (own) {
      g0 = (double)r * (double)r;
      g1 += first ? (double)r * (double)p : (double)pd * (double)r * (double)r;
    }
    ok = exchange(g0, g1, true);
    if (!ok) break;
    w += pd * r;
    if (first) {
      // reseed: p made orthogonal to the new residual and extended, α = γ / p·ŝ
      const bool keep = keep0 && g0 > 0.0;
      gam = g0 > 0.0 ? g1 / g0 : 0.0;
      rz = rz0 = g0;
      const double conv = rr0 > 0.0 ? a.tol2 / rr0 : 0.0;
      gstop = g0 * (a.hold2 > conv ? a.hold2 : conv);
      const X be = (X)(keep ? g0 / rzp0 : 0.0), ga = (X)gam;
      p = keep ? r + be * (p - ga * r) : r;
      sv = keep ? w + be * (sv - ga * w) : w;
      double none = 0.0;
      pq = own ? (double)p * (double)sv : 0.0;
      ok = exchange(pq, none, false);
      if (!ok) break;
      alpha = pq > 0.0 ? rz / pq : 0.0;
      if (!(pq > 0.0)) {          // p vanished (r̂ already zero): nothing to step
        done = restart = 1;
        break;
      }
      rzp = rz;                   // the first step moves x̂ and r̂ along the reseed's p, ŝ
    } else {
      const double be = g0 * irz;
      const double den = g1 - g0 * g0 * ira;
      const bool stop = g0 <= gstop;
      const bool brk = !(rzp > 0.0) || !(alpha != 0.0) || !(den > 0.0);
      rz = g0;
      if (stop || brk) {          // hand over: x̂, p and ŝ of the last step
        done = 1;
        restart = stop ? 0 : 1;
        break;
      }
      if (it >= a.lim) break;
      alpha = g0 / den;
      beta = be;
      rzp = g0;
      p = r + (X)be * p;
      sv = w + (X)be * sv;
    }
    ++it;
    x += (X)alpha * p;
    r -= (X)alpha * sv;
    first = false;
    spread();
    res_barrier();
  }
  if (!ok) {
    if (t == 0) a.s->gave_up = 1;
    return;
  }
  if (own) {
    a.p[d] = p;
    a.sv[d] = sv;
    a.u[d] += a.sc[d] * (double)x;
  }
  if (b == 0 && t == 0) {
    Scal* o = a.s;                // all but gave_up
    o->rz = rz;
    o->rz0 = rz0;
    o->rzp = rzp;
    o->gstop = gstop;
    o->alpha = alpha;
    o->beta = beta;
    o->gam = gam;
    o->pq = pq;
    o->done = done;
    o->restart = restart;
    o->fresh = 0;
    o->pend = 0.0;
    o->iters += it;
    o->prods += prods;
    o->prod_ticks += ticks;
  }
}

// ---- host ---------------------------------------------------------------------------------
// Cells of [lo, hi) of `order` into parts [b, b + m): cut across the longest axis in proportion.
static void elems_cut(const std::vector<double>& ctr, std::vector<int32_t>& order, int lo, int hi, int b, int m,
                      std::vector<int32_t>& part) {
  if (m == 1) {
    for (int i = lo; i < hi; ++i) part[order[i]] = b;
    return;
  }
  int axis = 0;
  double widest = -1.0;
  for (int d = 0; d < 3; ++d) {
    double l = 1e300, h = -1e300;
    for (int i = lo; i < hi; ++i) {
      l = std::min(l, ctr[3 * order[i] + d]);
      h = std::max(h, ctr[3 * order[i] + d]);
    }
    if (h - l > widest) {
      widest = h - l;
      axis = d;
    }
  }
  std::stable_sort(order.begin() + lo, order.begin() + hi,
                   [&](int32_t p, int32_t q) { return ctr[3 * p + axis] < ctr[3 * q + axis]; });
  const int ml = m / 2, mid = lo + (int)((int64_t)(hi - lo) * ml / m);
  elems_cut(ctr, order, lo, mid, b, ml, part);
  elems_cut(ctr, order, mid, hi, b + ml, m - ml, part);
}

static int elems_build(fem_ctx* c, ElemsOp* o) {
  o->state = -1;
  int ncu = 0, coop = 0;
  (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device);
  (void)hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, c->device);
  const int64_t nc = c->ncells, n = c->n;
  const int most = std::min(ncu, kResMaxBlocks);
  if (nc < 1 || nc > (int64_t)kElMost * most || n >= (1 << 30) || c->npc < 8 ||
      (int64_t)c->h_cell_nodes.size() != nc * c->npc)
    return FEM_OK;
  const int nb = (int)std::min<int64_t>(most, (nc + kElAim - 1) / kElAim);
  if (nb > 1 && !coop) return FEM_OK;
  std::vector<int32_t> cnode(27 * nc);
  FEM_HIP(c, hipMemcpy(cnode.data(), c->d_q2cnode, 4 * cnode.size(), hipMemcpyDeviceToHost));
  std::vector<double> xyz(c->nnodes), ctr(3 * nc, 0.0);
  for (int d = 0; d < 3; ++d) {
    FEM_HIP(c, hipMemcpy(xyz.data(), c->d_x[d], 8 * c->nnodes, hipMemcpyDeviceToHost));
    for (int64_t e = 0; e < nc; ++e)
      for (int k = 0; k < 8; ++k) ctr[3 * e + d] += xyz[c->h_cell_nodes[e * c->npc + k]];
  }
  std::vector<int32_t> order(nc), part(nc), cell((size_t)nb * kElMost, -1), count(nb, 0);
  std::iota(order.begin(), order.end(), 0);
  elems_cut(ctr, order, 0, (int)nc, 0, nb, part);
  for (int64_t e = 0; e < nc; ++e) {
    if (count[part[e]] == kElMost) return FEM_OK;
    cell[part[e] * kElMost + count[part[e]]++] = (int32_t)e;
  }
  // dofs of each block in order of first appearance, with their rows
  const size_t len = (size_t)nb * kResT;
  std::vector<int32_t> dof(len, -1), pos(len * kElMost, -1), slot(len, -1), from(len * kElShare, 0), nfrom(len, 0);
  std::vector<std::vector<int32_t>> has(n);   // places (block, thread) of each dof, blocks ascending
  for (int b = 0; b < nb; ++b) {
    int used = 0;
    for (int e = 0; e < count[b]; ++e)
      for (int r = 0; r < 81; ++r) {
        const int32_t d = 3 * cnode[27 * (int64_t)cell[b * kElMost + e] + r / 3] + r % 3;
        if (d < 0 || d >= n) return FEM_OK;
        if (has[d].empty() || has[d].back() / kResT != b) has[d].push_back(b * kResT + used++);
        const int32_t at = has[d].back();
        const int tt = at % kResT;
        dof[at] = d | (has[d].size() == 1 ? 1 << 30 : 0);
        int k = 0;
        while (k < kElMost && pos[((size_t)b * kElMost + k) * kResT + tt] >= 0) ++k;
        if (k == kElMost) return FEM_OK;      // a dof twice in a cell
        pos[((size_t)b * kElMost + k) * kResT + tt] = e * 81 + r;
      }
  }
  int nslots = 0;
  for (int b = 0; b < nb; ++b)
    for (int tt = 0; tt < kResT; ++tt) {
      const int32_t at = b * kResT + tt;
      if (dof[at] >= 0 && has[dof[at] & ~(1 << 30)].size() > 1) slot[at] = nslots++;
    }
  for (int64_t d = 0; d < n; ++d) {
    const std::vector<int32_t>& h = has[d];
    if (h.empty() || h.size() > (size_t)kElShare) return FEM_OK;   // a dof of no cell; too many blocks
    if (h.size() == 1) continue;
    for (int32_t at : h) {
      nfrom[at] = (int32_t)h.size();
      for (int k = 0; k < kElShare; ++k)
        from[((size_t)(at / kResT) * kElShare + k) * kResT + at % kResT] = slot[h[std::min<size_t>(k, h.size() - 1)]];
    }
  }
  // dofs of one block only: their wave's reads repeat a slot of that block (one it publishes itself)
  for (int b = 0; b < nb; ++b) {
    int32_t any = -1;
    for (int tt = 0; tt < kResT && any < 0; ++tt) any = slot[b * kResT + tt];
    for (int tt = 0; tt < kResT; ++tt)
      if (nfrom[b * kResT + tt] == 0)
        for (int k = 0; k < kElShare; ++k) from[((size_t)b * kElShare + k) * kResT + tt] = std::max(any, 0);
  }
  int rc;
  if ((rc = copy_alloc(c, &o->cell, cell.size())) || (rc = copy_alloc(c, &o->dof, len)) ||
      (rc = copy_alloc(c, &o->pos, pos.size())) || (rc = copy_alloc(c, &o->slot, len)) ||
      (rc = copy_alloc(c, &o->from, from.size())) || (rc = copy_alloc(c, &o->nfrom, len)) ||
      (rc = copy_alloc(c, &o->wx, (size_t)8 * nslots + 8)) || (rc = copy_alloc(c, &o->rec, kRecWords)))
    return rc;
  FEM_HIP(c, hipMemcpy(o->cell, cell.data(), 4 * cell.size(), hipMemcpyHostToDevice));
  FEM_HIP(c, hipMemcpy(o->dof, dof.data(), 4 * len, hipMemcpyHostToDevice));
  FEM_HIP(c, hipMemcpy(o->pos, pos.data(), 4 * pos.size(), hipMemcpyHostToDevice));
  FEM_HIP(c, hipMemcpy(o->slot, slot.data(), 4 * len, hipMemcpyHostToDevice));
  FEM_HIP(c, hipMemcpy(o->from, from.data(), 4 * from.size(), hipMemcpyHostToDevice));
  FEM_HIP(c, hipMemcpy(o->nfrom, nfrom.data(), 4 * len, hipMemcpyHostToDevice));
  FEM_HIP(c, hipMemset(o->wx, 0, (size_t)32 * nslots + 32));
  FEM_HIP(c, hipMemset(o->rec, 0, 4 * kRecWords));
  o->nb = nb;
  o->nslots = nslots;
  o->epoch = 0;
  o->state = 1;
  return FEM_OK;
}

static int elems_values(fem_ctx* c, ElemsOp* o, const double* sc, bool fp32, bool* ok) {
  int rc;
  if (o->state == 0 && (rc = elems_build(c, o))) return rc;
  if (o->state != 1) return FEM_OK;
  const size_t len = (size_t)o->nb * 81 * kResT;
  if (fp32 && !o->val32 && (rc = copy_alloc(c, &o->val32, len))) return rc;
  if (!fp32 && !o->val64 && (rc = copy_alloc(c, &o->val64, len))) return rc;
  const uint8_t* isc = c->ea_constrained ? c->d_isc : nullptr;
  const dim3 g(o->nb, 3);
  if (fp32 && c->ea_fp64)
    k_elems_vals<float, double><<<g, kResT, 0, c->stream>>>(o->cell, c->d_q2cnode, c->d_keq64, sc, isc, o->val32);
  else if (fp32)
    k_elems_vals<float, float><<<g, kResT, 0, c->stream>>>(o->cell, c->d_q2cnode, c->d_keq32, sc, isc, o->val32);
  else if (c->ea_fp64)
    k_elems_vals<double, double><<<g, kResT, 0, c->stream>>>(o->cell, c->d_q2cnode, c->d_keq64, sc, isc, o->val64);
  else
    k_elems_vals<double, float><<<g, kResT, 0, c->stream>>>(o->cell, c->d_q2cnode, c->d_keq32, sc, isc, o->val64);
  FEM_HIP(c, hipGetLastError());
  *ok = true;
  return FEM_OK;
}

int elems_prepare(fem_ctx* c, ElemsOp** op, const double* sc, bool fp32, bool* ok) {
  *ok = false;
  if (!*op) *op = new ElemsOp();
  const int rc = elems_values(c, *op, sc, fp32, ok);
  if (!no_memory(c, rc)) return rc;
  elems_free(op);
  *op = new ElemsOp();
  (*op)->state = -1;
  return FEM_OK;
}

template <typename X>
int elems_run(fem_ctx* c, ElemsOp* o, const double* res, const double* sc, X* p, X* sv, double* u, Scal* s,
              double hold_factor2, double tol2, int restart, int lim, bool* launched) {
  const uint32_t need = (uint32_t)lim + 8u;   // exchanges: one per product, one more per reseed
  if (o->epoch > 0xf0000000u - need) {
    FEM_HIP(c, hipMemsetAsync(o->wx, 0, (size_t)32 * o->nslots + 32, c->stream));
    FEM_HIP(c, hipMemsetAsync(o->rec, 0, 4 * kRecWords, c->stream));
    o->epoch = 0;
  }
  const X* val = sizeof(X) == 4 ? reinterpret_cast<const X*>(o->val32) : reinterpret_cast<const X*>(o->val64);
  ElemsArgs<X> a{o->nb, std::max(1, o->nslots), o->cell, o->dof, o->pos, o->slot, o->from, o->nfrom, val,
                 c->ea_constrained ? c->d_isc : nullptr, c->d_diag, c->d_nzval, res, sc, p, sv, u, s, o->wx, o->rec,
                 hold_factor2, tol2, o->epoch + 1u, c->res_polls, restart, lim, c->tune.time_kernels};
  o->epoch += need;
  const void* k = (const void*)k_resident_elems<X>;
  void* args[] = {&a};
  const hipError_t e = o->nb == 1 ? hipLaunchKernel(k, dim3(1), dim3(kResT), args, 0, c->stream)
                                  : hipLaunchCooperativeKernel(k, dim3(o->nb), dim3(kResT), args, 0, c->stream);
  *launched = e == hipSuccess;
  if (e != hipSuccess) (void)hipGetLastError();   // not as many blocks at once as the device should hold
  return FEM_OK;
}

template int elems_run<float>(fem_ctx*, ElemsOp*, const double*, const double*, float*, float*, double*, Scal*, double,
                              double, int, int, bool*);
template int elems_run<double>(fem_ctx*, ElemsOp*, const double*, const double*, double*, double*, double*, Scal*,
                               double, double, int, int, bool*);

}  // namespace fem
