// Resident CG on the 3D cell form of the scaled operator, FP32: the recurrence and the exchange
// of fem_resident.hip for lattices whose 27 entries per row no longer fit on chip (more than about
// 0.5 M rows).  The cell form needs one coefficient per cell, so up to 2.6 M rows do: a block owns
// a brick of the lattice and keeps on chip
//   * z = t r̂ of the brick and the nodes around it, and the coefficients of the cells around its
//     nodes, x̂, and where the nodes around are published, in LDS;
//   * r̂, p, ŝ, w and t of its nodes in registers, one thread per (x, y) column of the brick;
//   * r̂, ŝ and t of the nodes around the brick in registers, a few per thread.
// The product marches up the columns: 9 LDS reads of z and 4 of the coefficients per node, the
// planes below carried in registers, as in k_cell_spmv_z.  A node on the brick's surface is
// published as soon as the march has it, so most values have arrived when the march ends.
//
// What bounds it: at 128³ (252 bricks of up to 22 × 22 × 19 nodes) an iteration takes 11 µs, 4.4 of
// them the march (four cycles a vector instruction without packed FP32, on two waves per SIMD; 13
// LDS words a node, with bank conflicts where a wave's columns wrap to the next row of the brick),
// about 4 until the values of the other blocks are there (2,900 published values of 8 bytes a
// block), the rest sums, scalars and vector moves.  Counters over a solve: 104 vector instructions per
// 64 nodes and iteration in all, vector units busy 58%, LDS 42% (42% of that bank conflicts).  No vector or coefficient is read
// from memory between two hand-overs.  The separate kernels (k_cell_spmv_z and k_cg_move_scal)
// took 24–27 µs; whole mixed solve at 128³ 17.4 → 7.1 ms, at 90×84×80 8.9 → 3.85 ms.
// Measured on the way: plane loads issued in the step that uses them 18.6 µs an iteration, one step
// ahead and no branch around a prescribed row's sum 12.9; 54 operations a node (cell_row) instead of
// 39, 12.6 against 12.3 µs (with the hand-overs); x̂ moved in the update instead of while the exchange
// is under way, 0.4 µs more.
#include <algorithm>
#include <cmath>

#include "fem_resident_dev.h"

namespace fem {

constexpr int kBrickZ = 20;             // most nodes of a brick along z (register rows)
constexpr int kBrickX = 24;             // ... along x
constexpr int kBrickSX = kBrickX + 2;   // LDS row lengths of z and of the coefficients
constexpr int kBrickKX = kBrickX + 1;
constexpr int kBrickH = 7;              // most nodes around a brick, per thread

struct BrickOp {
  int state = 0;                        // 1 usable, −1 does not fit
  int n[3] = {}, cut[3] = {}, most[3] = {};   // nodes, bricks, largest brick per axis
  int nb = 0, slots = 0, lds = 0;
  uint32_t* wx = nullptr;               // [2][nb][slots] published values
  uint32_t* rec = nullptr;
  uint32_t epoch = 0;
};

void brick_free(BrickOp** op) {
  if (!*op) return;
  dev_free(&(*op)->wx);
  dev_free(&(*op)->rec);
  delete *op;
  *op = nullptr;
}

struct BrickArgs {
  int nx, ny, nz, sx, sy, sz, slots;
  int zplane, kplane, mz;   // LDS: largest plane of z and of the coefficients, planes of a brick
  int32_t px, pxy;
  const float *t, *kc;
  const int32_t* dofp;
  const double *res, *sc;
  float *p, *sv;
  double* u;
  Scal* s;
  uint32_t *wx, *rec;
  double hold2, tol2;
  uint32_t epoch, polls;
  int restart, lim, time;
  CellKrefT<float> kr;
};

// First node of brick i of s along an axis of n nodes; the brick that owns node x.
__device__ __forceinline__ int brick_lo(int i, int s, int n) { return i * n / s; }
__device__ __forceinline__ int brick_of(int x, int s, int n) { return ((x + 1) * s - 1) / n; }

// Published slot of a surface node of a bx × by × bz brick: the lowest plane, the highest, then
// the rings between (the two y sides, then the two x sides), so that a wave writes and reads runs.
__device__ __forceinline__ int brick_ring(int cx, int cy, int bx, int by) {
  return cy == 0 ? cx : cy == by - 1 ? bx + cx : cx == 0 ? 2 * bx + cy - 1 : cx == bx - 1 ? 2 * bx + by - 3 + cy : -1;
}
__device__ __forceinline__ int brick_slot(int cx, int cy, int cz, int bx, int by, int bz) {
  if (cz == 0) return cy * bx + cx;
  if (cz == bz - 1) return bx * by + cy * bx + cx;
  return 2 * bx * by + (cz - 1) * (2 * bx + 2 * by - 4) + brick_ring(cx, cy, bx, by);
}

__global__ __launch_bounds__(kResT) void k_resident_cells(BrickArgs a) {
  constexpr int BZ = kBrickZ, H = kBrickH, SX = kBrickSX, KX = kBrickKX;
  extern __shared__ __align__(16) unsigned char brick_lds[];
  __shared__ double red[2][2][kResWaves];
  __shared__ double tot[2][2][4];
  __shared__ int gaveup;
  __shared__ uint32_t polls;                 // what a wait may take (in LDS: scalar registers are short)
  float* zl = reinterpret_cast<float*>(brick_lds);     // [bz + 2][by + 2][SX]
  float* kl = zl + a.zplane * (a.mz + 2);              // [bz + 1][by + 1][KX]
  float* xl = kl + a.kplane * (a.mz + 1);              // [BZ][kResT] x̂
  uint32_t* hq = reinterpret_cast<uint32_t*>(xl + kResT * BZ);     // per node around: its published slot
  uint16_t* hp = reinterpret_cast<uint16_t*>(hq + kBrickH * kResT);  // ... and its place in zl
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int b = blockIdx.x, nb = gridDim.x;
  const int ix = b % a.sx, iy = (b / a.sx) % a.sy, iz = b / (a.sx * a.sy);
  const int x0 = brick_lo(ix, a.sx, a.nx), y0 = brick_lo(iy, a.sy, a.ny), z0 = brick_lo(iz, a.sz, a.nz);
  const int bx = brick_lo(ix + 1, a.sx, a.nx) - x0, by = brick_lo(iy + 1, a.sy, a.ny) - y0,
            bz = brick_lo(iz + 1, a.sz, a.nz) - z0;
  const int zp = SX * (by + 2), kp = KX * (by + 1);    // plane strides in LDS
  const bool mine = t < bx * by;
  const int cx = t % bx, cy = t / bx;
  const double rzp0 = a.s->rzp, rr0 = a.s->rr;
  const bool keep0 = !a.restart && !a.s->restart && rzp0 > 0.0;
  if (t == 0) {
    gaveup = 0;
    polls = a.polls;
  }
  auto row_of = [&](int x, int y, int z) { return (x + 1) + a.px * (y + 1) + a.pxy * (z + 1); };   // padded row

  // coefficients of the cells whose first corner is one of (x0 − 1 .., y0 − 1 .., z0 − 1 ..)
  for (int i = t; i < (bx + 1) * (by + 1) * (bz + 1); i += kResT) {
    const int kx = i % (bx + 1), ky = (i / (bx + 1)) % (by + 1), kz = i / ((bx + 1) * (by + 1));
    kl[kz * kp + ky * KX + kx] = a.kc[row_of(x0 - 1 + kx, y0 - 1 + ky, z0 - 1 + kz)];
  }
  for (int i = t; i < zp * (bz + 2); i += kResT) zl[i] = 0.f;   // (nodes outside the lattice stay 0)
  res_barrier();
  float r[BZ], p[BZ], sv[BZ], w[BZ], tt[BZ];
  const int zi0 = cx + 1 + SX * (cy + 1) + zp;         // this column's first node in zl
#pragma unroll
  for (int k = 0; k < BZ; ++k) {
    r[k] = p[k] = sv[k] = w[k] = tt[k] = 0.f;
    xl[k * kResT + t] = 0.f;
    if (mine && k < bz) {
      const int row = row_of(x0 + cx, y0 + cy, z0 + k);
      const int32_t d = a.dofp[row];
      tt[k] = a.t[row];
      r[k] = (float)(a.sc[d] * a.res[d]);
      if (keep0) {
        p[k] = a.p[row];
        sv[k] = a.sv[row];
      }
      zl[zi0 + k * zp] = tt[k] * r[k];
    }
  }
  // the nodes around the brick: their place in zl, published slot, r̂, ŝ, t
  const int plane = (bx + 2) * (by + 2), ring = 2 * (bx + 2) + 2 * by;
  const int around = 2 * plane + ring * bz;
  float hr[H], hs[H], ht[H], hw[H];
  uint32_t there = 0;                                  // bit k: the thread's node k exists
#pragma unroll
  for (int k = 0; k < H; ++k) {
    const int i = t + k * kResT;
    hr[k] = hs[k] = ht[k] = hw[k] = 0.f;
    int gx, gy, gz;                                    // from the brick's first node
    if (i < 2 * plane) {
      const int j = i < plane ? i : i - plane;
      gx = j % (bx + 2) - 1;
      gy = j / (bx + 2) - 1;
      gz = i < plane ? -1 : bz;
    } else {
      const int j = (i - 2 * plane) % ring;
      gz = (i - 2 * plane) / ring;
      gx = j < 2 * (bx + 2) ? j % (bx + 2) - 1 : j < 2 * (bx + 2) + by ? -1 : bx;
      gy = j < bx + 2 ? -1 : j < 2 * (bx + 2) ? by : (j - 2 * (bx + 2)) % by;
    }
    const int X = x0 + gx, Y = y0 + gy, Z = z0 + gz;
    const bool in = i < around && X >= 0 && X < a.nx && Y >= 0 && Y < a.ny && Z >= 0 && Z < a.nz;
    there |= in ? 1u << k : 0u;
    if (in) {
      const int ox = brick_of(X, a.sx, a.nx), oy = brick_of(Y, a.sy, a.ny), oz = brick_of(Z, a.sz, a.nz);
      const int qx = brick_lo(ox, a.sx, a.nx), qy = brick_lo(oy, a.sy, a.ny), qz = brick_lo(oz, a.sz, a.nz);
      hq[i] = (uint32_t)((ox + a.sx * (oy + a.sy * oz)) * a.slots +
                         brick_slot(X - qx, Y - qy, Z - qz, brick_lo(ox + 1, a.sx, a.nx) - qx,
                                    brick_lo(oy + 1, a.sy, a.ny) - qy, brick_lo(oz + 1, a.sz, a.nz) - qz));
      const int at = gx + 1 + SX * (gy + 1) + zp * (gz + 1);
      hp[i] = (uint16_t)at;
      const int row = row_of(X, Y, Z);
      const int32_t d = a.dofp[row];
      ht[k] = a.t[row];
      hr[k] = (float)(a.sc[d] * a.res[d]);
      if (keep0) hs[k] = a.sv[row];
      zl[at] = ht[k] * hr[k];
    }
  }
  res_barrier();

  const uint32_t nall = (uint32_t)(nb * a.slots);
  const __amdgpu_buffer_rsrc_t rw = buf_rsrc(a.wx, 2u * 8u * nall);
  const __amdgpu_buffer_rsrc_t rr = buf_rsrc(a.rec, (uint32_t)(4 * kRecWords));
  const int my_ring = mine ? brick_ring(cx, cy, bx, by) : -1;
  uint32_t ep = a.epoch;
  int nk = bz;
  double rzp = 0.0, alpha = 0.0, irz = 0.0, ira = 0.0;
  float pend = 0.f;                                    // α of the last step: α p is not in x̂ yet
  // Sums g0, g1 over all blocks; with `halo`, the w of the nodes around into hw.
  auto exchange = [&](double& g0, double& g1, bool halo) {
    const int par = (int)(ep & 1u);
    const double v0 = wave_sum63(g0), v1 = wave_sum63(g1);
    if (lane == 63) {
      red[par][0][wave] = v0;
      red[par][1][wave] = v1;
    }
    const uint32_t in_lds = polls;                  // (read before the barrier, which waits for it anyway)
    res_barrier();
    const uint32_t most = (uint32_t)uniform((int)in_lds);
    const uint32_t rec = (uint32_t)(par * kResCopies * 2 * kResMaxBlocks);
    if (t < 2 * kResCopies) {
      double sum = 0.0;
#pragma unroll
      for (int i = 0; i < kResWaves; ++i) sum += red[par][t & 1][i];
      ll_put(rr, rec + (uint32_t)(t * kResMaxBlocks + b), sum, ep);
    }
    const uint32_t rin = rec + (uint32_t)((b % kResCopies) * 2 * kResMaxBlocks + t);
    if (halo) {   // while the values travel: the last step's x̂ move, reciprocals of its scalars
#pragma unroll
      for (int k0 = 0; k0 < BZ; k0 += 4) {
        float xv[4];
        const uint32_t xo = (uint32_t)(k0 * kResT + t);
#pragma unroll
        for (int k = 0; k < 4; ++k)
          xv[k] = xl[xo + (uint32_t)(k * kResT)];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          xl[xo + (uint32_t)(k * kResT)] = xv[k] + pend * p[k0 + k];
      }
      irz = 1.0 / rzp;
      ira = 1.0 / (rzp * alpha);
    }
    const bool reader = t < nb;
    bool lost = false, need = reader;
    U4 q0 = {}, q1 = {};
    if (halo) {
      const uint32_t at = (ep & 1u) * nall;
      LL<float>::W hv[H];
      uint32_t q[H];
#pragma unroll
      for (int k = 0; k < H; ++k) q[k] = at + hq[t + k * kResT];
      for (uint32_t left = most;; --left) {
        asm volatile("" ::: "memory");
        bool ok = true;
        if (need) {
          q0 = LL<double>::get(rr, rin);
          q1 = LL<double>::get(rr, rin + kResMaxBlocks);
        }
#pragma unroll
        for (int k = 0; k < H; ++k)
          if (there >> k & 1u) hv[k] = LL<float>::get(rw, q[k]);
#pragma unroll
        for (int k = 0; k < H; ++k)
          if (there >> k & 1u) ok = ok && LL<float>::ok(hv[k], ep);
        if (need) need = !(LL<double>::ok(q0, ep) && LL<double>::ok(q1, ep));
        if (ok) break;
        if (left == 0) { lost = true; break; }
      }
#pragma unroll
      for (int k = 0; k < H; ++k)
        if (there >> k & 1u) hw[k] = LL<float>::val(hv[k]);
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
    // w = Â r̂ up the columns, the surface published on the way; γ = r̂·r̂ and δ = r̂·w (in a
    // reseed r̂·p instead)
    const long long c0 = a.time ? wall_clock64() : 0;
    double g0 = 0.0, g1 = 0.0;
    asm volatile("" : "+s"(nk));                       // (compared afresh: kept results would fill the scalar registers)
    if (mine) {
      const uint32_t out = (ep & 1u) * nall + (uint32_t)(b * a.slots);
      const int ringlen = 2 * bx + 2 * by - 4;
      // corner (−1, −1) of the column in the plane below, cell (−1, −1) of the layer below, the
      // ring's slot; advanced a plane at a time (opaque, or every plane's offset gets a register)
      uint32_t zc = (uint32_t)(cx + SX * cy), kk = (uint32_t)(cx + KX * cy);
      uint32_t rs = out + (uint32_t)(2 * bx * by + my_ring - ringlen);
      float zr[3][9], kq[2][4];                        // plane k in slot (k + 1) mod 3, layer k in (k + 1) mod 2
      auto plane9 = [&](float* v) {
#pragma unroll
        for (int dy = 0; dy < 3; ++dy)
#pragma unroll
          for (int dx = 0; dx < 3; ++dx) v[dy * 3 + dx] = zl[zc + (uint32_t)(dx + SX * dy)];
        zc += (uint32_t)zp;
        asm volatile("" : "+v"(zc));
      };
      auto layer4 = [&](float* v) {                    // origin P − e, e = ex + 2 ey
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = kl[kk + (uint32_t)((1 - (e & 1)) + KX * (1 - (e >> 1)))];
        kk += (uint32_t)kp;
        asm volatile("" : "+v"(kk));
      };
      // A layer of cells couples two planes.  In each, the neighbours of a node weighted with the
      // layer's coefficients and grouped by |dx| + 2 |dy| give four sums u; the four values f[0..3]
      // of them belong to the plane's own node, f[4..7] to the node of the other plane.  So a node
      // costs 39 operations: nine for u in each of the two planes of the layer above it, five
      // coefficient sums, eight each for its own node and the next one up.
      auto sums = [&](const float* v, const float* k, float* u) {
        const float x0s = k[0] + k[1], x1s = k[2] + k[3], y0s = k[0] + k[2], y1s = k[1] + k[3];
        u[0] = (x0s + x1s) * v[4];
        u[1] = y0s * v[5] + y1s * v[3];
        u[2] = x0s * v[7] + x1s * v[1];
        u[3] = k[0] * v[8] + k[1] * v[6] + k[2] * v[2] + k[3] * v[0];
      };
      auto own = [&](float y, const float* u) {
        return a.kr.f[3] * u[3] + (a.kr.f[2] * u[2] + (a.kr.f[1] * u[1] + (a.kr.f[0] * u[0] + y)));
      };
      auto other = [&](float y, const float* u) {
        return a.kr.f[7] * u[3] + (a.kr.f[6] * u[2] + (a.kr.f[5] * u[1] + (a.kr.f[4] * u[0] + y)));
      };
      plane9(zr[0]);
      plane9(zr[1]);
      layer4(kq[0]);
      plane9(zr[2]);
      layer4(kq[1]);
      float lower[4], upper[4];
      sums(zr[0], kq[0], lower);
      sums(zr[1], kq[0], upper);
      float next = other(own(0.f, upper), lower);      // the layer below node 0
#pragma unroll
      for (int k = 0; k < BZ; ++k) {
        if (k >= nk) continue;
        plane9(zr[k % 3]);                             // for the next step (past the last plane: not used)
        layer4(kq[k % 2]);
        sums(zr[(k + 1) % 3], kq[(k + 1) % 2], lower);
        sums(zr[(k + 2) % 3], kq[(k + 1) % 2], upper);
        float acc = other(own(next, lower), upper);
        next = other(own(0.f, upper), lower);
        asm volatile("" : "+v"(acc), "+v"(tt[k]));     // no branch around the sum, no kept comparison
        const float wv = tt[k] != 0.f ? tt[k] * acc : r[k];
        w[k] = wv;
        if (k == 0) ll_put(rw, out + (uint32_t)t, wv, ep);
        else if (k == nk - 1) ll_put(rw, out + (uint32_t)(bx * by + t), wv, ep);
        else if (my_ring >= 0) ll_put(rw, rs, wv, ep);
        rs += (uint32_t)ringlen;
        asm volatile("" : "+v"(rs));
        g0 += (double)r[k] * (double)r[k];
        g1 += (double)r[k] * (double)(first ? p[k] : wv);
      }
    }
    if (a.time) ticks += wall_clock64() - c0;
    ++prods;
    ok = exchange(g0, g1, true);
    if (!ok) break;
    if (first) {
      const bool keep = keep0 && g0 > 0.0;
      gam = g0 > 0.0 ? g1 / g0 : 0.0;
      rz = rz0 = g0;
      const double conv = rr0 > 0.0 ? a.tol2 / rr0 : 0.0;
      gstop = g0 * (a.hold2 > conv ? a.hold2 : conv);
      const float be = (float)(keep ? g0 / rzp0 : 0.0), ga = (float)gam;
      double none = 0.0;
      pq = 0.0;
#pragma unroll
      for (int k = 0; k < BZ; ++k) {
        p[k] = keep ? r[k] + be * (p[k] - ga * r[k]) : r[k];
        sv[k] = keep ? w[k] + be * (sv[k] - ga * w[k]) : w[k];
        pq += (double)p[k] * (double)sv[k];
      }
#pragma unroll
      for (int k = 0; k < H; ++k) hs[k] = keep ? hw[k] + be * (hs[k] - ga * hw[k]) : hw[k];
      ok = exchange(pq, none, false);
      if (!ok) break;
      alpha = pq > 0.0 ? rz / pq : 0.0;
      if (!(pq > 0.0)) {
        done = restart = 1;
        break;
      }
      rzp = rz;
    } else {
      const double be = g0 * irz;
      const double den = g1 - g0 * g0 * ira;
      const bool stop = g0 <= gstop;
      const bool brk = !(rzp > 0.0) || !(alpha != 0.0) || !(den > 0.0);
      rz = g0;
      if (stop || brk) {
        done = 1;
        restart = stop ? 0 : 1;
        break;
      }
      if (it >= a.lim) break;
      // p, ŝ need no α: their moves fill the division's latency (unused rows stay 0)
      alpha = g0 / den;
      beta = be;
      rzp = g0;
      const float bf = (float)be;
#pragma unroll
      for (int k = 0; k < BZ; ++k) {
        p[k] = r[k] + bf * p[k];
        sv[k] = w[k] + bf * sv[k];
      }
#pragma unroll
      for (int k = 0; k < H; ++k) hs[k] = hw[k] + bf * hs[k];
    }
    ++it;
    const float al = (float)alpha;
    pend = al;
    asm volatile("" : "+s"(nk));
#pragma unroll
    for (int k = 0; k < BZ; ++k) r[k] -= al * sv[k];
#pragma unroll
    for (int k = 0; k < H; ++k) hr[k] -= al * hs[k];
    if (mine) {
      uint32_t zo = (uint32_t)zi0;
#pragma unroll
      for (int k = 0; k < BZ; ++k) {
        if (k >= nk) continue;
        zl[zo] = tt[k] * r[k];
        zo += (uint32_t)zp;
        asm volatile("" : "+v"(zo));
      }
    }
#pragma unroll
    for (int k = 0; k < H; ++k)
      if (there >> k & 1u) zl[hp[t + k * kResT]] = ht[k] * hr[k];
    first = false;
    res_barrier();
  }
  const BrickArgs& z = *reinterpret_cast<const BrickArgs*>(res_kernargs());
  if (!ok) {
    if (t == 0) z.s->gave_up = 1;
    return;
  }
  if (mine) {
#pragma unroll
    for (int k = 0; k < BZ; ++k) {
      if (k >= bz) continue;
      const int row = (x0 + cx + 1) + z.px * (y0 + cy + 1) + z.pxy * (z0 + k + 1);
      z.p[row] = p[k];
      z.sv[row] = sv[k];
      const int32_t d = z.dofp[row];
      z.u[d] += z.sc[d] * (double)xl[k * kResT + t];
    }
  }
  if (b == 0 && t == 0) {
    Scal* o = z.s;                // all but gave_up
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
  }
  if (b == nb - 1 && t == 0) z.s->prod_ticks += ticks;   // of the largest brick: the last along each axis
}

// LDS of bricks of at most by nodes along y and bz along z.
static int brick_lds_bytes(int by, int bz) {
  return 4 * (kBrickSX * (by + 2) * (bz + 2) + kBrickKX * (by + 1) * (bz + 1) + kResT * kBrickZ + kBrickH * kResT) +
         2 * kBrickH * kResT;
}

// Bricks for an nx × ny × nz lattice: the cut with the fewest waves times planes per block, then
// the fewest nodes around.  False when no cut keeps a brick within the kernel's limits.
bool brick_cut(int nx, int ny, int nz, int most, int maxlds, int* cut) {
  const int n[3] = {nx, ny, nz};
  double best = 1e300;
  for (int sx = 1; sx <= most; ++sx)
    for (int sy = 1; sx * sy <= most; ++sy)
      for (int sz = 1; sx * sy * sz <= most; ++sz) {
        const int s[3] = {sx, sy, sz};
        int hi[3], lo[3];
        for (int d = 0; d < 3; ++d) {
          hi[d] = (n[d] + s[d] - 1) / s[d];
          lo[d] = n[d] / s[d];
        }
        if (lo[0] < 2 || lo[1] < 2 || lo[2] < 2) continue;
        if (hi[0] > kBrickX || hi[0] * hi[1] > kResT || hi[2] > kBrickZ) continue;
        const int around = 2 * (hi[0] + 2) * (hi[1] + 2) + (2 * (hi[0] + 2) + 2 * hi[1]) * hi[2];
        if (around > kBrickH * kResT || brick_lds_bytes(hi[1], hi[2]) > maxlds - kStaticLds) continue;
        const double cost = (double)((hi[0] * hi[1] + 63) / 64) * hi[2] * 1e4 + around;
        if (cost < best) {
          best = cost;
          for (int d = 0; d < 3; ++d) cut[d] = s[d];
        }
      }
  return best < 1e300;
}

static int brick_build(fem_ctx* c, BrickOp* o, int nx, int ny, int nz, bool* ok) {
  if (o->state == 0) {
    o->state = -1;
    int ncu = 0, maxlds = 0, coop = 0;
    (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device);
    (void)hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device);
    (void)hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, c->device);
    if (!coop || !brick_cut(nx, ny, nz, std::min(ncu, kResMaxBlocks), maxlds, o->cut)) return FEM_OK;
    const int n[3] = {nx, ny, nz};
    for (int d = 0; d < 3; ++d) {
      o->n[d] = n[d];
      o->most[d] = (n[d] + o->cut[d] - 1) / o->cut[d];
    }
    o->nb = o->cut[0] * o->cut[1] * o->cut[2];
    const int bx = o->most[0], by = o->most[1], bz = o->most[2];
    o->slots = 2 * bx * by + bz * (2 * bx + 2 * by);
    o->lds = brick_lds_bytes(by, bz);
    int rc;
    if ((rc = copy_alloc(c, &o->wx, (size_t)4 * o->nb * o->slots)) || (rc = copy_alloc(c, &o->rec, kRecWords))) return rc;
    FEM_HIP(c, hipMemsetAsync(o->wx, 0, (size_t)16 * o->nb * o->slots, c->stream));
    FEM_HIP(c, hipMemsetAsync(o->rec, 0, 4 * kRecWords, c->stream));
    o->epoch = 0;
    o->state = 1;
  }
  *ok = o->state == 1;
  return FEM_OK;
}

int brick_prepare(fem_ctx* c, BrickOp** op, int nx, int ny, int nz, bool* ok) {
  *ok = false;
  if (!*op) *op = new BrickOp();
  const int rc = brick_build(c, *op, nx, ny, nz, ok);
  if (!no_memory(c, rc)) return rc;
  brick_free(op);
  *op = new BrickOp();
  (*op)->state = -1;
  return FEM_OK;
}

int brick_run(fem_ctx* c, BrickOp* o, const BrickSource& s, const double* res, const double* sc, float* p, float* sv,
              double* u, Scal* scal, double hold_factor2, double tol2, int restart, int lim, bool* launched) {
  const uint32_t need = (uint32_t)lim + 8u;
  if (o->epoch > 0xf0000000u - need) {
    FEM_HIP(c, hipMemsetAsync(o->wx, 0, (size_t)16 * o->nb * o->slots, c->stream));
    FEM_HIP(c, hipMemsetAsync(o->rec, 0, 4 * kRecWords, c->stream));
    o->epoch = 0;
  }
  BrickArgs a{o->n[0], o->n[1], o->n[2], o->cut[0], o->cut[1], o->cut[2], o->slots,
              kBrickSX * (o->most[1] + 2), kBrickKX * (o->most[1] + 1), o->most[2], s.px, s.pxy,
              s.t, s.kc, s.dofp, res, sc, p, sv, u, scal, o->wx, o->rec, hold_factor2, tol2, o->epoch + 1u, c->res_polls, restart,
              lim, c->tune.time_kernels, {}};
  for (int i = 0; i < 8; ++i) a.kr.f[i] = (float)s.f[i];
  o->epoch += need;
  const void* k = (const void*)k_resident_cells;
  int maxlds = 0;
  FEM_HIP(c, hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device));
  FEM_HIP(c, res_dynamic_lds(k, maxlds));
  void* args[] = {&a};
  const hipError_t e =
      hipLaunchCooperativeKernel(k, dim3(o->nb), dim3(kResT), args, (unsigned)o->lds, c->stream);
  *launched = e == hipSuccess;
  if (e != hipSuccess) (void)hipGetLastError();
  return FEM_OK;
}

}  // namespace fem
