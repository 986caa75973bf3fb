// pepsmg_sweep.h -- NIT = 2 red/black iterations in one pass over a level
// (gfx950), from x, from x = 0 (src/multigrid.f90:1937) or from x plus the
// prolongation of the coarser level (:1958-1959 with :1676-1754), out of
// place.
//
// Bound: HBM bytes.  A launch reads x and b once and writes x once for all
// NIT iterations (k_rb_fused does so for each of them), so what limits it is
// whether the arithmetic of 2 NIT half-sweeps hides behind one pass:
// * A wave owns 128 columns (one pair (i odd, i+1) per lane) x 4 rows of a
//   tile and marches up through a z-chunk.  The planes in flight stay in
//   registers, updated in place: z neighbours are the thread's own values,
//   x neighbours the pair's other cell or one lane away (a DPP move), y
//   neighbours the thread's own rows.  Only the rows at the edge of a wave
//   come from the neighbouring wave, through LDS.
// * Step m loads x of plane m and runs half-sweep s (1 .. 2 NIT, red first)
//   on plane m - s.  It reads planes m - s -+ 1 and its own as half-sweep
//   s - 1 left them, and what it needs of other waves was written a step
//   ago: one barrier per plane step.
// * Each colour's b is used by NIT half-sweeps, up to 2 NIT steps after it
//   was loaded; it waits in LDS in slots private to the thread.
// * Blocks overlap by a ring of 2 NIT cells (each half-sweep needs one less),
//   so blocks never read each other's output.
// * Loads run one (FP64) or two (FP32) planes ahead: 347 against 262 us for
//   the FP32 zero start at 512^3.
// Registers are what the shape is cut to: 4 rows x 6 planes of pairs are 96
// (FP64) or 48 (FP32), and 8 waves leave 256 per thread.  Taller waves,
// more waves or several blocks per CU measured the same or spilled (FP32
// 512^3, two iterations: 4 rows x 8 waves 400 us, 8 x 8 387 us but the
// variant with the prolongation spills, 4 x 12 404 us).
// At 512^3, two iterations: FP64 0.85 ms against 2 x 0.55 ms for k_rb_fused;
// FP32 from x 0.38 against 2 x 0.28, from 0 0.26 against 0.49, with the
// prolongation 0.42 against 0.75 ms for its three launches.  FP32 reads
// 1.10x and writes 1.00x the bytes of one pass.  FP64 is held back by its
// arithmetic (about 500 vector operations a wave and step), FP32 by the
// latency of a step (its vector units are busy for 40 % of the time).
// FP64 values are those of the separate kernels bit for bit: same expression
// and operand order, divisions included.
#pragma once
#include "pepsmg_fused.h"
#include "pepsmg_march.h"

namespace pepsmg {

constexpr int SW_COLS = 128;                       // columns of a tile, ring included

enum { SW_X = 0, SW_ZERO = 1, SW_PROLONG = 2 };    // where x_in comes from

constexpr int SW_ROWS = 4;                         // rows of a wave
constexpr int SW_WAVES = 8;                        // waves of a block

struct SweepGrid {
  int gx, gy, nch, kchunk;   // tiles and z-chunks (kchunk even)
  int uw, uh;                // columns / rows a tile stores (even)
};

template <typename T>
struct SweepArgs {
  T* xo;
  const T* xi;
  const T* b;
  const T* xc;               // SW_PROLONG: the coarser level's x
  Lvl<T> L, C;
  ProlongW<T> W;
  T omega;
  SweepGrid G;
  int zlo, zhi;              // planes with the z coefficients c5u, c6u
  T c5u, c6u;
  T* ext;                    // FP64: the caller's array that also receives x_out (layout U), or null
  Lvl<T> U;
};

// value of the lane to the west (lane - 1) / east (lane + 1), 0 beyond the wave
template <int CTRL>
__device__ __forceinline__ float sw_shift(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double sw_shift(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ float sw_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double sw_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }
// a f, rounded like the ordinary product, but 0 for f = 0 whatever a is
__device__ __forceinline__ float sw_mul0(float a, float f) {
  float r;
  asm("v_mul_legacy_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(f));
  return r;
}
template <typename T>
__device__ __forceinline__ T sw_west(T v) { return sw_shift<0x138>(v); }   // wave_shr:1
template <typename T>
__device__ __forceinline__ T sw_east(T v) { return sw_shift<0x130>(v); }   // wave_shl:1

// A plane's address as one scalar in the global address space: the accesses
// of its rows add a 32-bit lane offset to it (without this the compiler
// keeps a 64-bit address per array and row in vector registers).
typedef __attribute__((address_space(1))) char* sw_ptr;
__device__ __forceinline__ sw_ptr sw_base(const void* p, long off) {
  sw_ptr q = (sw_ptr)p + off;
  asm("" : "+s"(q));
  return q;
}
template <typename T>
struct SwPair {
  typedef T type __attribute__((ext_vector_type(2)));
};
// v as a value the compiler cannot know or keep: what is formed from it is
// formed again in each step instead of being held in registers across steps
template <typename V>
__device__ __forceinline__ V sw_fresh_v(V v) {
  asm volatile("" : "+v"(v));
  return v;
}
__device__ __forceinline__ int sw_fresh_s(int v) {
  asm volatile("" : "+s"(v));
  return v;
}
template <typename T>
__device__ __forceinline__ typename SwPair<T>::type sw_load(sw_ptr base, unsigned off) {
  return *(const __attribute__((address_space(1))) typename SwPair<T>::type*)(base + sw_fresh_v(off));
}

template <typename T, int W, int NIT, int PRE>
struct SweepShape {
  static constexpr int R = SW_ROWS, WAVES = W, THREADS = 64 * W, ROWS = R * W;
  static constexpr int RING = 2 * NIT;
  // SW_PROLONG: the outermost pair only feeds the interpolation of the next
  static constexpr int RINGX = RING + (PRE == SW_PROLONG ? 2 : 0);
  static_assert(NIT == 2, "the march runs four half-sweeps in groups of six plane steps");
  static constexpr int NS = 2 * NIT + 2;            // planes in registers
  static constexpr int NBR = 2 * NIT - 2, NBB = 2 * NIT - 1;   // red / black half planes of b waiting in LDS
  static constexpr int EDGE = 2 * (WAVES + 1) * 64;      // one kind of edge rows of one plane
  static constexpr int LDS = 2 * RING * EDGE + (NBR + NBB) * R * THREADS;   // elements
};

// Block number of the level, or of all levels of a launch, that blockIdx
// stands for: contiguous eighths of the tiles (x fastest, then y, then
// chunks) per XCD, so that neighbouring tiles re-read each other's rings from
// the XCD's L2.  The grid is rounded up to a multiple of 8.
__device__ __forceinline__ int sweep_block() { return (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3); }

// block `lin` of the level
template <typename T, int W, int NIT, int PRE>
__device__ __forceinline__ void sweep_tile(const SweepArgs<T>& A, int lin) {
  using S = SweepShape<T, W, NIT, PRE>;
  using V2 = typename SwPair<T>::type;
  constexpr bool F64 = sizeof(T) == 8;
  constexpr int NW = S::WAVES, NT = S::THREADS;
  constexpr int R = S::R, RING = S::RING, NS = S::NS, NST = 2 * NIT;
  constexpr int CR = R / 2 + 2;                      // coarse rows a wave interpolates from
  extern __shared__ __align__(16) unsigned char sw_smem[];
  T* const edge = reinterpret_cast<T*>(sw_smem);     // [buffer][kind][side][wave + 1][lane]
  T* const bred = edge + 2 * RING * S::EDGE;         // red b, two planes
  T* const bblk = bred + S::NBR * R * NT;    // black b, NBB planes

  const Lvl<T>& L = A.L;
  const SweepGrid& G = A.G;
  const int ntile = G.gx * G.gy;
  const int bz = lin / ntile, tile = lin - bz * ntile;
  const int ty = tile / G.gx, tx = tile - ty * G.gx;
  const int us = 1 + tx * G.uw, ue = min(us + G.uw - 1, L.nx);   // columns / rows stored
  const int vs = 1 + ty * G.uh, ve = min(vs + G.uh - 1, L.ny);
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ia = (tx == 0 ? 1 : us - S::RINGX) + 2 * lane;       // odd
  const int j0 = (ty == 0 ? 1 : vs - RING) + w * R;              // odd
  const int k0 = 1 + bz * G.kchunk, k1 = min(k0 + G.kchunk, L.nz + 1);   // k0 odd
  const int ct = threadIdx.x;

  const bool in0 = ia <= L.nx, in1 = ia + 1 <= L.nx;
  // every cell of the wave inside the level
  const bool full = L.nx >= (tx == 0 ? 1 : us - S::RINGX) + SW_COLS - 1 && L.ny >= j0 + R - 1;
  const bool st = ia >= us && ia <= ue;              // the pair is stored, in rows rlo .. rhi
  const int rlo = vs - j0, rhi = ve - j0;
  // byte offset in a plane of this lane's pair in row r: an odd column <= nx
  // keeps the pair inside the padded row, rows clamped to the level
  unsigned voff[R];
#pragma unroll
  for (int r = 0; r < R; r++)
    voff[r] = (unsigned)(((long)(min(j0 + r, L.ny) - 1) * L.px + (in0 ? ia - 1 : 0)) * (long)sizeof(T));

  T c1[2], c2[2], c3[R], c4[R];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const bool in = c ? in1 : in0;
    c1[c] = in ? L.cwx[ia + c] : T(0);
    c2[c] = in ? L.cex[ia + c] : T(0);
  }
#pragma unroll
  for (int r = 0; r < R; r++) {
    c3[r] = ldc(L.cwy, min(j0 + r, L.ny));
    c4[r] = ldc(L.cey, min(j0 + r, L.ny));
  }
  // Planes zlo .. zhi share their z coefficients: there the divisors are
  // kept.  FP64: c0 and 1 / c0; FP32: omega / c0 alone.  Cells outside the
  // level get the factor 0, which leaves them 0 (in FP32 also beside an
  // infinity or a NaN: sw_mul0).
  T dv[F64 ? R : 1][2], rv[R][2];
  bool kept = A.zhi >= A.zlo;
#pragma unroll
  for (int r = 0; r < R; r++) {
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const bool in = (c ? in1 : in0) && j0 + r <= L.ny;
      const T c0 = -(c1[c] + c2[c] + c3[r] + c4[r] + A.c5u + A.c6u);
      if constexpr (F64) {
        dv[r][c] = c0;
        rv[r][c] = in ? 1.0 / c0 : 0.0;
        kept = kept && (!in || kd_divisor(c0));
      } else {
        rv[r][c] = in ? sor_factor(A.omega, c0) : T(0);
      }
    }
  }
  // Steps flo .. fhi: every half-sweep is on a plane of the level with kept
  // divisors.  They run all of them, also on planes outside the chunk's ring
  // (the first steps of a chunk, and those that fill its last group of NS):
  // what those get never reaches a plane that is stored.
  // (FP64 keeps to the chunk's ring at its start: the quotients of planes
  // that hold zeros would take the division.)
  const int flo = (F64 ? max(k0, A.zlo) : A.zlo) + NST;
  const int fhi = __syncthreads_and(kept) ? min(A.zhi + 1, L.nz) : flo - 1;
  const T om1 = T(1) - A.omega;

  // interpolation weights, each pair of an axis divided by its sum, and
  // coarse planes (SW_PROLONG): the lane's coarse column is (ia + 1) / 2,
  // the wave's coarse rows jc0 - 1 .. jc0 + R / 2
  T wxs[2], wxn[2], wys[R], wyn[R], cp[3][CR], cnew[CR];
  const int jc0 = (j0 + 1) / 2, icl = (ia + 1) / 2;
  const bool cin = icl <= A.C.nx;
  const unsigned coff = (unsigned)((cin ? icl - 1 : 0) * sizeof(T));
  if (PRE == SW_PROLONG) {
    const int ic = in0 ? ia : 1;                     // a halving level: nx is even
    const T sa = A.W.px_[ic], na = A.W.px_[ic + 1], sb = A.W.nx_[ic + 1], nb2 = A.W.nx_[ic];
    wxs[0] = sa / (sa + na);
    wxn[0] = na / (sa + na);
    wxs[1] = sb / (sb + nb2);
    wxn[1] = nb2 / (sb + nb2);
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int j = min(j0 + r, L.ny);
      const bool odd = j & 1;
      const T sy = odd ? ldc(A.W.py_, j) : ldc(A.W.ny_, j), ny = odd ? ldc(A.W.py_, j + 1) : ldc(A.W.ny_, j - 1);
      wys[r] = sy / (sy + ny);
      wyn[r] = ny / (sy + ny);
    }
  }
  auto issue_c = [&](T* dst, int kc) {
    const char* base = (const char*)(A.xc + (long)(min(max(kc, 1), A.C.nz) - 1) * A.C.pxy);
#pragma unroll
    for (int q = 0; q < CR; q++) {
      const int jc = min(max(jc0 - 1 + q, 1), A.C.ny);
      dst[q] = *reinterpret_cast<const T*>(base + (long)(jc - 1) * A.C.px * (long)sizeof(T) + coff);
    }
  };
  auto take_c = [&](T* dst, const T* src, int kc) {
    const bool vz = kc >= 1 && kc <= A.C.nz;
#pragma unroll
    for (int q = 0; q < CR; q++) {
      const int jc = jc0 - 1 + q;
      dst[q] = vz && jc >= 1 && jc <= A.C.ny && cin ? src[q] : T(0);
    }
  };

  // edge rows: value of wave w's row 0 (side 1) and row R - 1 (side 0)
  auto epos = [&](int buf, int kind, int side, int wv) {
    return edge + ((((buf * RING + kind) * 2 + side) * (NW + 1) + wv) << 6);
  };
  if (ct < 64) {   // beyond the tile: 0 (the ghost value at a domain face; ring cells elsewhere)
#pragma unroll
    for (int q = 0; q < 2 * RING; q++) {
      epos(q & 1, q >> 1, 0, 0)[lane] = T(0);
      epos(q & 1, q >> 1, 1, NW)[lane] = T(0);
    }
  }

  T X[NS][R][2];
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int r = 0; r < R; r++) X[s][r][0] = X[s][r][1] = T(0);
  constexpr int PF = F64 ? 1 : 2;                    // planes of look-ahead of the loads
  V2 xpre[PF][PRE == SW_ZERO ? 1 : R], bpre[PF][R];
  auto issue_x = [&](V2* xp, long po) {
    if (PRE == SW_ZERO) return;
    const sw_ptr base = sw_base(A.xi, po);
#pragma unroll
    for (int r = 0; r < R; r++) xp[r] = sw_load<T>(base, voff[r]);
  };
  auto issue_b = [&](V2* bp, long po) {
    const sw_ptr base = sw_base(A.b, po);
#pragma unroll
    for (int r = 0; r < R; r++) bp[r] = sw_load<T>(base, voff[r]);
  };

  const int mstart = k0 - RING, mend = k1 + NST;     // mstart odd
  const long pl = L.pxy * (long)sizeof(T);
  // byte offset of plane m, clamped to the level
  auto next = [&](long o, int m) { return o + (m >= 1 && m < L.nz ? pl : 0); };   // plane m + 1 from plane m's
  long po = (long)(max(mstart, 1) - 1) * pl;         // of the plane x was last issued for
  issue_x(xpre[0], po);
  issue_b(bpre[0], po);                              // (plane mstart - 1 is not needed)
  if (PF == 2) {
    issue_b(bpre[PF - 1], po);
    po = next(po, mstart);
    issue_x(xpre[PF - 1], po);
  }
  if (PRE == SW_PROLONG) {
    const int q = (mstart + 1) / 2;                  // mstart is odd: exact
    T t0[CR], t1[CR];
    issue_c(t0, q - 1);
    issue_c(t1, q);
    take_c(cp[0], t0, q - 1);
    take_c(cp[1], t1, q);
  }

  // one plane step; U = (m - mstart) mod NS, so plane m - d is in slot
  // (U - d) mod NS and m is odd iff U is even
  auto step = [&](int m, auto Uc, auto Fc) {
    constexpr int U = decltype(Uc)::value;
    constexpr bool FAST = decltype(Fc)::value;       // m in flo .. fhi
    constexpr int buf = U & 1;                       // edges published this step; the other buffer is read
    constexpr bool ODD = (U & 1) == 0;
    constexpr int PB = PF == 2 ? (U & 1) : 0;
    const long pn = next(po, m + PF - 1);            // plane m + PF
    lds_barrier();
    // ---- x_in of plane m ----
    {
      const bool vz = FAST || (m >= 1 && m <= L.nz);
      constexpr int s = U;
      if (PRE == SW_PROLONG && !ODD) take_c(cp[2], cnew, m / 2 + 1);
#pragma unroll
      for (int r = 0; r < R; r++) {
        X[s][r][0] = PRE != SW_ZERO ? xpre[PB][r].x : T(0);
        X[s][r][1] = PRE != SW_ZERO ? xpre[PB][r].y : T(0);
      }
      issue_x(xpre[PB], pn);
      if (PRE == SW_PROLONG) {
        if (ODD) issue_c(cnew, (m + 1) / 2 + 1);
        if (vz) {
          T sz = ODD ? ldc(A.W.pz_, m) : ldc(A.W.nz_, m), nz = ODD ? ldc(A.W.pz_, m + 1) : ldc(A.W.nz_, m - 1);
          const T fz = sz / (sz + nz), gz = nz / (sz + nz);
          // parent plane and its neighbour below (odd m) or above
          const T(&P)[CR] = cp[1];
          const T(&N)[CR] = ODD ? cp[0] : cp[2];
          T z[CR];
#pragma unroll
          for (int q = 0; q < CR; q++) z[q] = sw_fma(gz, N[q], fz * P[q]);
#pragma unroll
          for (int c = 0; c < 2; c++) {
            T h[CR];
#pragma unroll
            for (int q = 0; q < CR; q++) h[q] = sw_fma(wxn[c], c ? sw_east(z[q]) : sw_west(z[q]), wxs[c] * z[q]);
#pragma unroll
            for (int r = 0; r < R; r++) {
              const int cj = r / 2 + 1, nj = (r & 1) ? cj + 1 : cj - 1;
              X[s][r][c] = X[s][r][c] + sw_fma(wyn[r], h[nj], wys[r] * h[cj]);
            }
          }
        }
        if (!ODD) {
#pragma unroll
          for (int q = 0; q < CR; q++) {
            cp[0][q] = cp[1][q];
            cp[1][q] = cp[2][q];
          }
        }
      }
      if (PRE != SW_ZERO && !(vz && full)) {
        const int rows = vz ? sw_fresh_s(L.ny) - j0 + 1 : 0;   // rows of the wave inside the level
        const int left = L.nx - sw_fresh_v(ia);                // < 0: the pair lies outside, 0: its second cell
#pragma unroll
        for (int r = 0; r < R; r++) {
          X[s][r][0] = r < rows && left >= 0 ? X[s][r][0] : T(0);
          X[s][r][1] = r < rows && left > 0 ? X[s][r][1] : T(0);
        }
      }
    }
    // ---- b of plane m - 1 (loaded a step ago) ----
    V2 bc[R];
#pragma unroll
    for (int r = 0; r < R; r++) bc[r] = bpre[PB][r];
    issue_b(bpre[PB], po);
    po = pn;
    // ---- plane m - NST - 1 is final ----
    if (m - NST - 1 >= k0 && m - NST - 1 < k1) {
      constexpr int s = (U + 2 * NS - NST - 1) % NS;
      const sw_ptr out = sw_base(A.xo, (long)(m - NST - 2) * pl);
#pragma unroll
      for (int r = 0; r < R; r++) {
        if (st && r >= rlo && r <= rhi) {
          // (a second cell beyond nx lies in the row's padding and is 0)
          const V2 o = {X[s][r][0], X[s][r][1]};
          __builtin_nontemporal_store(o, (__attribute__((address_space(1))) V2*)(out + sw_fresh_v(voff[r])));
        }
      }
      if (F64 && A.ext) {
        T* u = A.ext + (long)(m - NST - 2) * A.U.pxy;
#pragma unroll
        for (int r = 0; r < R; r++) {
          if (st && r >= rlo && r <= rhi) {
            T* q = u + (long)(j0 + r - 1) * A.U.px + (ia - 1);
            if (in1) st_pair_unal(q, X[s][r][0], X[s][r][1]);
            else q[0] = X[s][r][0];
          }
        }
      }
    }
    // ---- half-sweeps ----
    auto half = [&](auto Dc) {
      constexpr int D = decltype(Dc)::value;         // half-sweep number; plane m - D
      constexpr bool RED = (D & 1) == 1;
      constexpr bool Z = PRE == SW_ZERO && D == 1;   // x = 0: the products sum to +0
      constexpr int s = (U + 2 * NS - D) % NS, sm = (s + NS - 1) % NS, sp = (s + 1) % NS;
      constexpr int KP = (ODD ? 1 + D : D) & 1;      // parity of the plane
      // the red cell of a pair is its first iff j + k is even
      auto cell = [](int r) { return (((r + 1 + KP) & 1) != 0) == RED ? 1 : 0; };
      const int k = m - D;
      if (FAST || (k >= max(1, k0 - RING + D) && k <= min(L.nz, k1 - 1 + RING - D))) {
        T ea = T(0), eb = T(0), bv[R];
        if (!Z) {
          ea = epos(buf ^ 1, D - 1, 0, w)[lane];
          eb = epos(buf ^ 1, D - 1, 1, w + 1)[lane];
        }
        if (D == 1) {
#pragma unroll
          for (int r = 0; r < R; r++) bv[r] = cell(r) ? bc[r].y : bc[r].x;
        } else {
          // plane k's half plane was stored at step k + 1
          constexpr int slot = RED ? (U + 2 * NS - D + 1) % 2 : (U + 6 * NS - D + 1) % S::NBB;
          const T* src = (RED ? bred : bblk) + slot * R * NT + ct;
#pragma unroll
          for (int r = 0; r < R; r++) bv[r] = src[r * NT];
        }
        // b - (c1 xw + c2 xe + c3 xs + c4 xn + c5 xb + c6 xt): the reference's
        // order in FP64; FP32 as sor_temp
        auto diff = [&](int r, T c5, T c6) -> T {
          const int c = cell(r);
          if (Z) return bv[r] - T(0);
          const T xw = c == 0 ? sw_west(X[s][r][1]) : X[s][r][0];
          const T xe = c == 0 ? X[s][r][1] : sw_east(X[s][r][0]);
          const T xs = r > 0 ? X[s][r > 0 ? r - 1 : 0][c] : ea;
          const T xn = r < R - 1 ? X[s][r < R - 1 ? r + 1 : r][c] : eb;
          const T xb = X[sm][r][c], xt = X[sp][r][c];
          if constexpr (F64) {
            return bv[r] - (c1[c] * xw + c2[c] * xe + c3[r] * xs + c4[r] * xn + c5 * xb + c6 * xt);
          } else {
            return bv[r] - sor_temp(SorC<T>{c1[c], c2[c], c3[r], c4[r], c5, c6}, xw, xe, xs, xn, xb, xt);
          }
        };
        auto put = [&](int r, T q) {                 // q: omega (b - ...) / c0
          const int c = cell(r);
          if (F64) X[s][r][c] = q + om1 * (Z ? T(0) : X[s][r][c]);
          else X[s][r][c] = Z ? q : sw_fma(om1, X[s][r][c], q);
        };
        if constexpr (FAST && F64) {
          T a[R], q[R];
          unsigned far = 0;
#pragma unroll
          for (int r = 0; r < R; r++) {
            a[r] = A.omega * diff(r, A.c5u, A.c6u);
            far = max(far, kd_range(a[r]));
            q[r] = kd_quotient(a[r], dv[r][cell(r)], rv[r][cell(r)]);
          }
          if (__builtin_amdgcn_ballot_w64(far > KD_SPAN)) {
#pragma unroll
            for (int r = 0; r < R; r++) q[r] = sw_fresh_v(rv[r][cell(r)]) != T(0) ? a[r] / dv[r][cell(r)] : T(0);
          }
#pragma unroll
          for (int r = 0; r < R; r++) put(r, q[r]);
        } else if constexpr (FAST) {
#pragma unroll
          for (int r = 0; r < R; r++) put(r, sw_mul0(diff(r, A.c5u, A.c6u), rv[r][cell(r)]));
        } else {
          const T c5 = ldc(L.cwz, k), c6 = ldc(L.cez, k);
#pragma unroll
          for (int r = 0; r < R; r++) {
            const int c = cell(r);
            const T c0 = -(sw_fresh_v(c1[c]) + c2[c] + c3[r] + c4[r] + c5 + c6);
            T q;
            if constexpr (F64) q = A.omega * diff(r, c5, c6) / c0;
            else q = diff(r, c5, c6) * sor_factor(A.omega, c0);
            put(r, sw_fresh_v(rv[r][c]) != T(0) ? q : T(0));
          }
        }
      }
      if (D < NST) {                                 // edges for half-sweep D + 1 of this plane, next step
        epos(buf, D, 1, w)[lane] = X[s][0][cell(0)];
        epos(buf, D, 0, w + 1)[lane] = X[s][R - 1][cell(R - 1)];
      }
    };
    half(std::integral_constant<int, 1>());
    half(std::integral_constant<int, 2>());
    half(std::integral_constant<int, 3>());
    half(std::integral_constant<int, 4>());
    // ---- b of plane m - 1 into its slots, black cells of plane m to the neighbours ----
    {
      constexpr int KP = ODD ? 0 : 1;                // parity of plane m - 1
      constexpr int sb = (U + 6 * NS) % S::NBB;
#pragma unroll
      for (int r = 0; r < R; r++) {
        const bool rf = ((r + 1 + KP) & 1) == 0;     // red is the first cell
        bblk[(sb * R + r) * NT + ct] = rf ? bc[r].y : bc[r].x;
        bred[((U & 1) * R + r) * NT + ct] = rf ? bc[r].x : bc[r].y;
      }
      if (PRE != SW_ZERO) {
        constexpr int KM = ODD ? 1 : 0;              // parity of plane m
        constexpr int red0 = (1 + KM) & 1, redR = (R + KM) & 1;
        epos(buf, 0, 1, w)[lane] = X[U][0][1 - red0];
        epos(buf, 0, 0, w + 1)[lane] = X[U][R - 1][1 - redR];
      }
    }
  };
  // groups of NS steps: a loop of its own for the fast ones, so that no
  // value has to sit in the same register on two paths through a step
  for (int m = mstart; m <= mend;) {
    while (m <= mend && m >= flo && m + NS - 1 <= fhi) {
      step(m, std::integral_constant<int, 0>(), std::true_type());
      step(m + 1, std::integral_constant<int, 1>(), std::true_type());
      step(m + 2, std::integral_constant<int, 2>(), std::true_type());
      step(m + 3, std::integral_constant<int, 3>(), std::true_type());
      step(m + 4, std::integral_constant<int, 4>(), std::true_type());
      step(m + 5, std::integral_constant<int, 5>(), std::true_type());
      m += NS;
    }
    auto run = [&](auto Uc) {
      constexpr int U = decltype(Uc)::value;
      if (m + U <= mend) step(m + U, Uc, std::false_type());
    };
    run(std::integral_constant<int, 0>());
    run(std::integral_constant<int, 1>());
    run(std::integral_constant<int, 2>());
    run(std::integral_constant<int, 3>());
    run(std::integral_constant<int, 4>());
    run(std::integral_constant<int, 5>());
    m += NS;
  }
}

template <typename T, int W, int NIT, int PRE>
__global__ void __launch_bounds__(64 * W) k_sweep(SweepArgs<T> A) {
  const int lin = sweep_block();
  if (lin < A.G.gx * A.G.gy * A.G.nch) sweep_tile<T, W, NIT, PRE>(A, lin);
}

}  // namespace pepsmg
