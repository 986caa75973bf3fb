// pepsmg_block.h -- NIT red/black iterations on small levels in one launch
// (gfx950): from x, from x = 0 or from x plus the prolongation of the coarser
// level, out of place; REST: then the residual restricted into the coarser
// level's b.
//
// Bound: latency.  On levels of 128^3 cells and fewer a z-march waits for a
// memory round trip at each of its few plane steps (k_rb_fused takes 6 to 8
// us on levels of 16^3 to 64^3, 3 of it such waits), and every iteration and
// the prolongation is a launch of its own.  Here a block holds a BX x BY x BZ
// tile and a ring of 2 NIT cells in LDS: all loads are issued at the start
// (one round trip), the half-sweeps follow with a barrier each, every one on
// a region one cell smaller, and the tile is stored.  Levels this small are
// served from the caches, so the ring (8 times the tile's cells for 16 x 8
// x 4 and two iterations) costs little beside the launches it saves.
//
// Threads own pairs (i odd, i + 1) of the region through the whole launch;
// LDS keeps the first and the second cells of the pairs apart, so lanes touch
// consecutive words.  Values are those of the separate kernels bit for bit.
#pragma once
#include "pepsmg_coarse.h"
#include "pepsmg_sweep.h"

namespace pepsmg {

template <typename T>
struct BlockArgs {
  T* xo;
  const T* xi;
  const T* b;
  const T* xc;               // SW_PROLONG: the coarser level's x
  Lvl<T> L, C;
  ProlongW<T> W;
  T omega;
  int gx, gy;                // tiles along x and y
  double* partial;           // NORM: per-block sums of (b - A x_in)^2
  T* bc;                     // REST: the coarser level's b (C and RW: its layout and the weights)
  RestrictW<T> RW;
  T* ext;                    // FP64: the caller's array that also receives x_out (layout U), or null
  Lvl<T> U;
};

template <int BX_, int BY_, int BZ_, int NT_>
struct BlockTile {
  static constexpr int BX = BX_, BY = BY_, BZ = BZ_, NT = NT_;
};
using BlockSmall = BlockTile<16, 8, 4, 512>;
using BlockLarge = BlockTile<32, 8, 8, 1024>;
// (Its 8 pairs a thread take 127 registers.  One word of state per pair instead
// of four brings BlockLarge to 64, for two blocks on a CU, but unpacking costs
// what that gains: the half-sweeps are short of instruction slots.)
using BlockTall = BlockTile<32, 16, 8, 1024>;

template <typename T, typename B, int NIT, int PRE, bool REST = false>
struct BlockShape {
  // ring along y and z, and along x (even, so that pairs keep their parity)
  static constexpr int H = 2 * NIT + (REST ? 1 : 0), HX = 2 * NIT + (REST ? 2 : 0);
  static constexpr int PX = (B::BX + 2 * HX) / 2, RY = B::BY + 2 * H, RZ = B::BZ + 2 * H;
  static constexpr int NPAIR = PX * RY * RZ, PP = (NPAIR + B::NT - 1) / B::NT;
  // coarse cells the region interpolates from
  static constexpr int CX = PX + 2, CY = RY / 2 + 2, CZ = RZ / 2 + 2, NC = CX * CY * CZ;
  static constexpr int PC = (NC + B::NT - 1) / B::NT;
  static constexpr int NW = 2 * (2 * PX + RY + RZ);        // coefficients (or weights) of the region's lines
  static constexpr int LDS = 2 * NPAIR + NW + (PRE == SW_PROLONG ? NW + NC : 0);   // elements
};

// tile `bid` of the level
template <typename T, typename B, int NIT, int PRE, bool NORM, bool REST = false>
__device__ __forceinline__ void block_tile(const BlockArgs<T>& A, int bid) {
  using S = BlockShape<T, B, NIT, PRE, REST>;
  using V2 = typename SwPair<T>::type;
  constexpr bool F64 = sizeof(T) == 8;
  constexpr int H = S::H, HX = S::HX, PX = S::PX, RY = S::RY, RZ = S::RZ, NP = S::NPAIR, PP = S::PP, NT = B::NT;
  extern __shared__ __align__(16) unsigned char bl_smem[];
  T* const xs = reinterpret_cast<T*>(bl_smem);       // first cells of the pairs, then the second ones
  T* const cx = xs + 2 * NP;                         // cwx, cex of the region's columns (0 outside the level)
  T* const cy = cx + 4 * PX;                         // cwy, cey of its rows
  T* const cz = cy + 2 * RY;                         // cwz, cez of its planes
  T* const pw = cx + S::NW;                          // SW_PROLONG: weights of parent and neighbour, as cx, cy, cz
  T* const cs = pw + S::NW;                          // SW_PROLONG: coarse cells

  const Lvl<T>& L = A.L;
  const int t = threadIdx.x;
  const int bx = bid % A.gx, byz = bid / A.gx;
  const int i0 = 1 + bx * B::BX - HX, j0 = 1 + (byz % A.gy) * B::BY - H, k0 = 1 + (byz / A.gy) * B::BZ - H;   // i0 odd

  // ---- all loads ----
  V2 xv[PP], bv[PP];
  int id[PP], dist[PP][2], at[PP];                   // at: pair, row and plane in the region
  bool tile[PP], first[PP];                          // first: the pair's first cell is red (i + j + k odd)
#pragma unroll
  for (int p = 0; p < PP; p++) {
    const int e = min(t + p * NT, NP - 1);
    const int row = e / PX, px = e - row * PX, rz = row / RY, ry = row - rz * RY;
    const int i = i0 + 2 * px, j = j0 + ry, k = k0 + rz;
    const bool on = t + p * NT < NP;
    const bool vr = on && j >= 1 && j <= L.ny && k >= 1 && k <= L.nz;
    const bool v0 = vr && i >= 1 && i <= L.nx, v1 = vr && i + 1 >= 1 && i + 1 <= L.nx;
    id[p] = e;
    at[p] = px | ry << 8 | rz << 16;
    // distance to the region's face (-1: outside the level), which half-sweeps count down
    const int dyz = min(min(ry, RY - 1 - ry), min(rz, RZ - 1 - rz));
    dist[p][0] = v0 ? min(dyz, min(2 * px, 2 * PX - 1 - 2 * px)) : -1;
    dist[p][1] = v1 ? min(dyz, min(2 * px + 1, 2 * PX - 2 - 2 * px)) : -1;
    first[p] = ((j + k) & 1) == 0;
    tile[p] = v0 && px >= HX / 2 && px < PX - HX / 2 && ry >= H && ry < RY - H && rz >= H && rz < RZ - H;
    // an odd column <= nx keeps the pair inside the padded row
    const int ic = v0 ? i : 1, jc = min(max(j, 1), L.ny), kc = min(max(k, 1), L.nz);
    const long g = lidx(L, ic, jc, kc);
    if (PRE != SW_ZERO) xv[p] = *reinterpret_cast<const V2*>(A.xi + g);
    bv[p] = *reinterpret_cast<const V2*>(A.b + g);
  }
  if (t < 2 * PX + RY + RZ) {
    const int q = t - 2 * PX;
    T w, e;
    if (q < 0) {
      const int i = i0 + t;
      const bool in = i >= 1 && i <= L.nx;
      w = in ? L.cwx[in ? i : 1] : T(0);
      e = in ? L.cex[in ? i : 1] : T(0);
    } else if (q < RY) {
      const int j = min(max(j0 + q, 1), L.ny);
      w = L.cwy[j];
      e = L.cey[j];
    } else {
      const int k = min(max(k0 + q - RY, 1), L.nz);
      w = L.cwz[k];
      e = L.cez[k];
    }
    cx[2 * t] = w;
    cx[2 * t + 1] = e;
    if constexpr (PRE == SW_PROLONG) {
      // odd cell: p(f), p(f + 1); even cell: n(f), n(f - 1)
      const int axis = q < 0 ? 0 : q < RY ? 1 : 2;
      const int f = axis == 0 ? i0 + t : axis == 1 ? j0 + q : k0 + q - RY;
      const int n = axis == 0 ? L.nx : axis == 1 ? L.ny : L.nz;
      const T* p = axis == 0 ? A.W.px_ : axis == 1 ? A.W.py_ : A.W.pz_;
      const T* m = axis == 0 ? A.W.nx_ : axis == 1 ? A.W.ny_ : A.W.nz_;
      const int g = min(max(f, 1), n);
      T ws = g & 1 ? p[g] : m[g], wn = g & 1 ? p[g + 1] : m[g - 1];
      if constexpr (!F64) interp_norm(ws, wn);
      pw[2 * t] = ws;
      pw[2 * t + 1] = wn;
    }
  }
  // REST: the thread's coarse cell and its weights
  constexpr int QX = B::BX / 2, QY = B::BY / 2, QZ = B::BZ / 2;
  const int qx = t % QX, qy = t / QX % QY, qz = t / (QX * QY);
  const int ic = bx * QX + qx + 1, jc = (byz % A.gy) * QY + qy + 1, kc = (byz / A.gy) * QZ + qz + 1;
  const bool rest = REST && t < QX * QY * QZ && ic <= A.C.nx && jc <= A.C.ny && kc <= A.C.nz;
  T ax1 = T(0), ax2 = T(0), ay1 = T(0), ay2 = T(0), az1 = T(0), az2 = T(0);
  if (REST && rest) {
    ax1 = A.RW.wx[2 * ic - 1], ax2 = A.RW.wx[2 * ic];
    ay1 = A.RW.wy[2 * jc - 1], ay2 = A.RW.wy[2 * jc];
    az1 = A.RW.wz[2 * kc - 1], az2 = A.RW.wz[2 * kc];
  }
  if constexpr (PRE == SW_PROLONG) {
    // coarse region: the parents of the fine region and one cell around
    // (i0, j0 and k0 are odd: exact divisions)
    const int ci = (i0 + 1) / 2 - 1, cj0 = (j0 + 1) / 2 - 1, ck0 = (k0 + 1) / 2 - 1;
    T v[S::PC];
#pragma unroll
    for (int q = 0; q < S::PC; q++) {
      const int e = min(t + q * NT, S::NC - 1);
      const int row = e / S::CX, x = e - row * S::CX, z = row / S::CY, y = row - z * S::CY;
      const int ic = ci + x, jc = cj0 + y, kc = ck0 + z;
      const bool in = ic >= 1 && ic <= A.C.nx && jc >= 1 && jc <= A.C.ny && kc >= 1 && kc <= A.C.nz;
      const T u = A.xc[lidx(A.C, min(max(ic, 1), A.C.nx), min(max(jc, 1), A.C.ny), min(max(kc, 1), A.C.nz))];
      v[q] = in ? u : T(0);
    }
#pragma unroll
    for (int q = 0; q < S::PC; q++)
      if (t + q * NT < S::NC) cs[t + q * NT] = v[q];
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PP; p++) {
      const int px = at[p] & 255, ry = at[p] >> 8 & 255, rz = at[p] >> 16;
      const int j = j0 + ry, k = k0 + rz;
      if (dist[p][0] < 0) continue;                  // a halving level: both cells of a pair are in or out
      const bool jo = j & 1, ko = k & 1;
      const T *wx = pw + 4 * px, *wy = pw + 4 * PX + 2 * ry, *wz = pw + 4 * PX + 2 * RY + 2 * rz;
      const T sy = wy[0], ny = wy[1], sz = wz[0], nz = wz[1];
      const int jc = (j + 1) / 2 - cj0, kc = (k + 1) / 2 - ck0;
      const T* P = cs + (kc * S::CY + jc) * S::CX + px + 1;        // the parent's row, at the pair's column
      const int dy = jo ? -S::CX : S::CX, dz = (ko ? -S::CY : S::CY) * S::CX;
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const T sx = wx[2 * c], nx = wx[2 * c + 1];
        const int dx = c ? 1 : -1;
        T add;
        if constexpr (F64) {
          const T num = sx * sy * sz * P[0] + nx * sy * sz * P[dx] + sx * ny * sz * P[dy] + sx * sy * nz * P[dz] +
                        nx * ny * sz * P[dx + dy] + nx * sy * nz * P[dx + dz] + sx * ny * nz * P[dy + dz] +
                        nx * ny * nz * P[dx + dy + dz];
          add = num / ((sx + nx) * (sy + ny) * (sz + nz));
        } else {
          add = interp_zxy(sz, nz, sx, nx, sy, ny, P[0], P[dx], P[dy], P[dx + dy], P[dz], P[dz + dx], P[dz + dy],
                           P[dz + dx + dy]);
        }
        if (c) xv[p].y = xv[p].y + add;
        else xv[p].x = xv[p].x + add;
      }
    }
  }
#pragma unroll
  for (int p = 0; p < PP; p++) {
    if (t + p * NT < NP) {
      xs[id[p]] = PRE != SW_ZERO && dist[p][0] >= 0 ? xv[p].x : T(0);
      xs[NP + id[p]] = PRE != SW_ZERO && dist[p][1] >= 0 ? xv[p].y : T(0);
    }
  }
  __syncthreads();

  if constexpr (NORM) {
    double acc = 0.0;
#pragma unroll
    for (int p = 0; p < PP; p++) {
      if (!tile[p]) continue;
      const T *ky = cy + 2 * (at[p] >> 8 & 255), *kz = cz + 2 * (at[p] >> 16);
      const T c3 = ky[0], c4 = ky[1], c5 = kz[0], c6 = kz[1];
#pragma unroll
      for (int c = 0; c < 2; c++) {
        if (dist[p][c] < 0) continue;
        const T* kx = cx + 2 * (2 * (at[p] & 255) + c);
        const T c0 = diag(kx[0], kx[1], c3, c4, c5, c6);
        const T* o = xs + c * NP + id[p];
        const T* w = xs + (1 - c) * NP + id[p] - (1 - c);
        const T ax = c0 * o[0] + kx[0] * w[0] + kx[1] * w[1] + c3 * o[-PX] + c4 * o[PX] + c5 * o[-PX * RY] +
                     c6 * o[PX * RY];
        const T r = (c ? bv[p].y : bv[p].x) - ax;
        acc += (double)r * (double)r;
      }
    }
    __shared__ double sh[NT / 64];
    const double s = block_sum(acc, sh);             // (its barriers also close the reads of x_in)
    if (t == 0) A.partial[bid] = s;
  }
#pragma unroll
  for (int s = 1; s <= 2 * NIT; s++) {
#pragma unroll
    for (int p = 0; p < PP; p++) {
      const bool c = first[p] == ((s & 1) == 0);     // the cell of this colour is the pair's second
      if ((c ? dist[p][1] : dist[p][0]) < s) continue;
      const T *ky = cy + 2 * (at[p] >> 8 & 255), *kz = cz + 2 * (at[p] >> 16);
      const T c3 = ky[0], c4 = ky[1], c5 = kz[0], c6 = kz[1];
      const T* kx = cx + 2 * (2 * (at[p] & 255) + c);
      const T a1 = kx[0], a2 = kx[1], bb = c ? bv[p].y : bv[p].x;
      T* o = xs + (c ? NP : 0) + id[p];
      // neighbours: own array at +- a row or plane, the other array at the pair and beside it
      const T* w = xs + (c ? 0 : NP) + id[p] - (c ? 0 : 1);
      if (PRE == SW_ZERO && s == 1) {
        o[0] = sor_zero(A.omega, bb, diag(a1, a2, c3, c4, c5, c6));
      } else if constexpr (F64) {
        const T tm = a1 * w[0] + a2 * w[1] + c3 * o[-PX] + c4 * o[PX] + c5 * o[-PX * RY] + c6 * o[PX * RY];
        o[0] = sor_update(A.omega, bb, tm, diag(a1, a2, c3, c4, c5, c6), o[0]);
      } else {
        const T tm = sor_temp(SorC<T>{a1, a2, c3, c4, c5, c6}, w[0], w[1], o[-PX], o[PX], o[-PX * RY], o[PX * RY]);
        o[0] = sor_next(A.omega, bb, tm, sor_factor(A.omega, diag(a1, a2, c3, c4, c5, c6)), o[0]);
      }
    }
    if (s < 2 * NIT) __syncthreads();
  }
  // the owner of a pair updated both of its cells last
#pragma unroll
  for (int p = 0; p < PP; p++) {
    if (!tile[p]) continue;
    const int i = i0 + 2 * (at[p] & 255), j = j0 + (at[p] >> 8 & 255), k = k0 + (at[p] >> 16);
    const V2 o = {xs[id[p]], xs[NP + id[p]]};        // (a second cell beyond nx is 0 and lies in the row's padding)
    *reinterpret_cast<V2*>(A.xo + lidx(L, i, j, k)) = o;
    if (F64 && A.ext) {
      T* u = A.ext + lidx(A.U, i, j, k);
      if (dist[p][1] >= 0) st_pair_unal(u, o.x, o.y);
      else u[0] = o.x;
    }
  }
  if constexpr (REST) {
    // the residual of the tile (the last half-sweep also covered one cell
    // around it), in place of x, and the restriction from there
    // (restrict_axis's weights, k_restrict's terms and order)
    static_assert(QX * QY * QZ <= NT, "a coarse cell per thread");
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PP; p++) {
      if (!tile[p]) continue;
      const T *ky = cy + 2 * (at[p] >> 8 & 255), *kz = cz + 2 * (at[p] >> 16);
      const T c3 = ky[0], c4 = ky[1], c5 = kz[0], c6 = kz[1];
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const T* kx = cx + 2 * (2 * (at[p] & 255) + c);
        const T c0 = diag(kx[0], kx[1], c3, c4, c5, c6);
        const T* o = xs + c * NP + id[p];
        const T* w = xs + (1 - c) * NP + id[p] - (1 - c);
        const T ax = c0 * o[0] + kx[0] * w[0] + kx[1] * w[1] + c3 * o[-PX] + c4 * o[PX] + c5 * o[-PX * RY] +
                     c6 * o[PX * RY];
        if (c) bv[p].y = bv[p].y - ax;
        else bv[p].x = bv[p].x - ax;
      }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PP; p++) {
      if (!tile[p]) continue;
      xs[id[p]] = bv[p].x;
      xs[NP + id[p]] = bv[p].y;
    }
    __syncthreads();
    if (rest) {
      const T v111 = ax1 * ay1 * az1, v211 = ax2 * ay1 * az1, v121 = ax1 * ay2 * az1, v221 = ax2 * ay2 * az1;
      const T v112 = ax1 * ay1 * az2, v212 = ax2 * ay1 * az2, v122 = ax1 * ay2 * az2, v222 = ax2 * ay2 * az2;
      const T vol = v111 + v211 + v121 + v221 + v112 + v212 + v122 + v222;
      // z, p: the odd and the even child along an axis
      auto R = [&](int a, int bb, int cc) {
        return xs[a * NP + ((H + 2 * qz + cc) * RY + H + 2 * qy + bb) * PX + HX / 2 + qx];
      };
      const T sum = v111 * R(1, 1, 1) + v211 * R(0, 1, 1) + v121 * R(1, 0, 1) + v221 * R(0, 0, 1) +
                    v112 * R(1, 1, 0) + v212 * R(0, 1, 0) + v122 * R(1, 0, 0) + v222 * R(0, 0, 0);
      A.bc[lidx(A.C, ic, jc, kc)] = sum / vol;
    }
  }
}

template <typename T, typename B, int NIT, int PRE, bool NORM, bool REST>
__global__ void __launch_bounds__(B::NT) k_block(BlockArgs<T> A) {
  block_tile<T, B, NIT, PRE, NORM, REST>(A, blockIdx.x);
}

}  // namespace pepsmg
