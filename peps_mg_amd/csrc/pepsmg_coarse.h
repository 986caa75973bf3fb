// pepsmg_coarse.h -- prolongation+correction z-march kernel and the
// persistent coarse-level kernel (gfx950).
#pragma once
#include "pepsmg_march.h"

namespace pepsmg {

// ---------------------------------------------------------------------------
// x_f += P x_c for a level that halves every axis
// (src/multigrid.f90:1958-1959 / :1965-1966 with
// multigrid_prolongation_linear_on_nonuniform_grid :1676-1754).  A block
// owns a TX x 16 fine tile (a TX/2 x 8 coarse tile; TX = 64, or 128 for
// FP32, with 4 TX threads); coarse planes with a
// one-cell ring are staged in LDS (4 slots), fine x planes stream through
// registers with the next plane's loads in flight.  Per axis the fine cell f
// takes its parent c with weight ws and the neighbour nb with weight wn
// (f odd: dxp(f), dxp(f+1), c-1; f even: dxn(f), dxn(f-1), c+1); the eight
// terms are summed in the reference order.
template <typename T, int TX>
__device__ __forceinline__ void prolong_march_block(int bid, T* __restrict__ xf, const T* __restrict__ xc,
                                                    const Lvl<T>& F, const Lvl<T>& Cc, const ProlongW<T>& W,
                                                    const MarchGrid& G) {
  constexpr int TP = TX / 2, NT = march_threads<TX>();
  constexpr int CX = TP + 2, CY = 10;                // coarse tile TX/2 x 8 + ring 1
  constexpr int NCL = (CX * CY + NT - 1) / NT;
  constexpr int NP = 2;                              // fine pairs per thread
  using V2 = typename Vec2<T>::type;
  __shared__ T sc[4][CY][CX];

  const int t = threadIdx.x;
  const int bz = bid % G.nch;
  const int rxy = bid / G.nch;
  const int i0 = 1 + (rxy % G.gx) * TX;              // fine tile origin
  const int j0 = 1 + (rxy / G.gx) * 16;
  const int ic0 = (i0 + 1) / 2, jc0 = (j0 + 1) / 2;  // coarse tile origin
  const int kc0 = 1 + bz * G.kchunk;                 // coarse planes of this chunk
  const int kc1 = min(kc0 + G.kchunk, Cc.nz + 1);

  // fine pairs: rows ly = t/TP + 8q, pair lp = t%TP -> cells i0+2lp (odd), i0+2lp+1
  int ly[NP];
  bool act[NP], two[NP];
  T wsa[NP], wna[NP], wsb[NP], wnb[NP], wsy[NP], wny[NP];
  int cjr[NP], njr[NP];   // coarse row (LDS) of parent / neighbour in y
  const int lp = t % TP;
  const int ia = i0 + 2 * lp;
  // x: cell ia (odd): parent ic, neighbour ic-1; cell ia+1 (even): parent ic, neighbour ic+1
  const int ic = (ia + 1) / 2;
  const int lcx = ic - ic0 + 1;                      // LDS column of the parent
#pragma unroll
  for (int q = 0; q < NP; q++) {
    ly[q] = t / TP + 8 * q;
    int gj = j0 + ly[q];
    act[q] = gj <= F.ny && ia <= F.nx;
    two[q] = act[q] && ia + 1 <= F.nx;
    wsa[q] = act[q] ? W.px_[ia] : T(0);
    wna[q] = act[q] ? W.px_[ia + 1] : T(0);
    wsb[q] = two[q] ? W.nx_[ia + 1] : T(0);
    wnb[q] = two[q] ? W.nx_[ia] : T(0);
    int jc = (gj + 1) / 2;
    bool jodd = gj & 1;
    wsy[q] = act[q] ? (jodd ? W.py_[gj] : W.ny_[gj]) : T(0);
    wny[q] = act[q] ? (jodd ? W.py_[gj + 1] : W.ny_[gj - 1]) : T(0);
    cjr[q] = jc - jc0 + 1;
    njr[q] = (jodd ? jc - 1 : jc + 1) - jc0 + 1;
    if constexpr (sizeof(T) == 4) {
      interp_norm(wsa[q], wna[q]);
      interp_norm(wsb[q], wnb[q]);
      interp_norm(wsy[q], wny[q]);
    }
  }

  // Coarse and fine planes load from clamped in-bounds addresses with no
  // branch around the loads; coarse values outside the domain are zeroed
  // when staged, fine values of cells outside are never stored.
  T cpre[NCL];
  auto issue_c = [&](T* dst, int kc) {
    const int kcc = min(max(kc, 1), Cc.nz);
#pragma unroll
    for (int q = 0; q < NCL; q++) {
      int e = min(t + q * NT, CX * CY - 1);
      int cy = e / CX, cx = e - cy * CX;
      int gi = min(max(ic0 - 1 + cx, 1), Cc.nx), gj = min(max(jc0 - 1 + cy, 1), Cc.ny);
      dst[q] = xc[lidx(Cc, gi, gj, kcc)];
    }
  };
  // src: the values issue_c loaded for coarse plane kc
  auto stage_c = [&](const T* src, int kc) {
    const bool vz = kc >= 1 && kc <= Cc.nz;
#pragma unroll
    for (int q = 0; q < NCL; q++) {
      int e = t + q * NT;
      if (e < CX * CY) {
        int cy = e / CX, cx = e - cy * CX;
        int gi = ic0 - 1 + cx, gj = jc0 - 1 + cy;
        bool v = vz && gi >= 1 && gi <= Cc.nx && gj >= 1 && gj <= Cc.ny;
        (&sc[kc & 3][0][0])[e] = v ? src[q] : T(0);
      }
    }
  };
  // fine planes are loaded two planes ahead: xpre[h] holds the next fine
  // plane of parity h (h = 0: odd, 1: even)
  V2 xpre[2][NP];
  auto issue_f = [&](V2* dst, int f) {
    const int fc = min(max(f, 1), F.nz);
#pragma unroll
    for (int q = 0; q < NP; q++) {
      // an odd column <= nx keeps the 2-element load inside the padded row
      int gi = act[q] ? ia : 1, gj = act[q] ? j0 + ly[q] : 1;
      dst[q] = ld_stream_v2(xf + lidx(F, gi, gj, fc));
    }
  };

  {   // the three staged planes' loads in flight before the first is staged
    T ca[NCL], cb[NCL];
    issue_c(cpre, kc0 - 1);
    issue_c(ca, kc0);
    issue_c(cb, kc0 + 1);
    stage_c(cpre, kc0 - 1);
    stage_c(ca, kc0);
    stage_c(cb, kc0 + 1);
  }
  issue_c(cpre, kc0 + 2);
  issue_f(xpre[0], 2 * kc0 - 1);
  issue_f(xpre[1], 2 * kc0);
  // coarse-plane step, run twice per iteration so the compiler's wait
  // counts across the back edge stay exact
  auto step = [&](int kc) {
    lds_barrier();
#pragma unroll
    for (int h = 0; h < 2; h++) {
      int f = 2 * kc - 1 + h;                        // h = 0: odd fine plane, 1: even (F.nz = 2 Cc.nz)
      V2 xv[NP];
#pragma unroll
      for (int q = 0; q < NP; q++) xv[q] = xpre[h][q];
      issue_f(xpre[h], f + 2);
      T wsz = (h == 0) ? ldc(W.pz_, f) : ldc(W.nz_, f);
      T wnz = (h == 0) ? ldc(W.pz_, f + 1) : ldc(W.nz_, f - 1);
      if constexpr (sizeof(T) == 4) interp_norm(wsz, wnz);
      T(*P)[CX] = sc[kc & 3];
      T(*N)[CX] = sc[(h == 0 ? kc - 1 : kc + 1) & 3];
#pragma unroll
      for (int q = 0; q < NP; q++) {
        if (!act[q]) continue;
        int cj = cjr[q], nj = njr[q];
        T sy = wsy[q], ny = wny[q];
        // first cell (odd i): parent column lcx, neighbour lcx-1
        {
          T sx = wsa[q], nx = wna[q];
          int ci = lcx, ni = lcx - 1;
          if constexpr (sizeof(T) == 4) {
            xv[q].x = xv[q].x + interp_zxy(wsz, wnz, sx, nx, sy, ny, P[cj][ci], P[cj][ni], P[nj][ci], P[nj][ni],
                                           N[cj][ci], N[cj][ni], N[nj][ci], N[nj][ni]);
          } else {
            T num = sx * sy * wsz * P[cj][ci] + nx * sy * wsz * P[cj][ni] + sx * ny * wsz * P[nj][ci] +
                    sx * sy * wnz * N[cj][ci] + nx * ny * wsz * P[nj][ni] + nx * sy * wnz * N[cj][ni] +
                    sx * ny * wnz * N[nj][ci] + nx * ny * wnz * N[nj][ni];
            xv[q].x = xv[q].x + num / ((sx + nx) * (sy + ny) * (wsz + wnz));
          }
        }
        if (two[q]) {   // second cell (even i): parent lcx, neighbour lcx+1
          T sx = wsb[q], nx = wnb[q];
          int ci = lcx, ni = lcx + 1;
          if constexpr (sizeof(T) == 4) {
            xv[q].y = xv[q].y + interp_zxy(wsz, wnz, sx, nx, sy, ny, P[cj][ci], P[cj][ni], P[nj][ci], P[nj][ni],
                                           N[cj][ci], N[cj][ni], N[nj][ci], N[nj][ni]);
          } else {
            T num = sx * sy * wsz * P[cj][ci] + nx * sy * wsz * P[cj][ni] + sx * ny * wsz * P[nj][ci] +
                    sx * sy * wnz * N[cj][ci] + nx * ny * wsz * P[nj][ni] + nx * sy * wnz * N[cj][ni] +
                    sx * ny * wnz * N[nj][ci] + nx * ny * wnz * N[nj][ni];
            xv[q].y = xv[q].y + num / ((sx + nx) * (sy + ny) * (wsz + wnz));
          }
        }
        long q0 = lidx(F, ia, j0 + ly[q], f);
        if (two[q]) st_stream_pair(xf + q0, xv[q].x, xv[q].y);
        else xf[q0] = xv[q].x;
      }
    }
    stage_c(cpre, kc + 2);
    issue_c(cpre, kc + 3);
  };
  int kc = kc0;
  for (; kc + 1 < kc1; kc += 2) {
    step(kc);
    step(kc + 1);
  }
  if (kc < kc1) step(kc);
}

template <typename T, int TX>
__global__ void __launch_bounds__(march_threads<TX>())
k_prolong_march(T* __restrict__ xf, const T* __restrict__ xc, Lvl<T> F, Lvl<T> Cc, ProlongW<T> W, MarchGrid G) {
  prolong_march_block<T, TX>(blockIdx.x, xf, xc, F, Cc, W, G);
}

// ---------------------------------------------------------------------------
// Persistent coarse-level kernel: one workgroup runs the part of the
// V-cycle below a switch level s entirely in LDS (src/multigrid.f90:1936-1962
// restricted to levels s..L): for each level down to L-1, nu red/black
// iterations from x = 0, residual and restriction; the coarsest solve
// (rbgs_solver, <= 1000 iterations, stop at sqrt(|r|^2/|r0|^2) <= tol, a
// single cell directly); then up again: prolongation + correction and nu
// iterations.  It reads b_s from global memory and writes x_s back.  The
// coarsest level is solved in FP64 whatever T is (T = float in the
// mixed-precision inner cycles).  Operations run in the reference order and
// the coarsest norm of up to 64 cells is summed sequentially, so FP64
// results are bit-identical to the per-level kernels and to the reference.
// The 1-D coefficient and transfer-weight arrays of every level are staged
// into LDS at the start, so no phase waits on a global load.
constexpr int PC_MAXLEV = 8;
constexpr int PC_THREADS = 1024;
constexpr int PC_CINV_MAX = 128;   // largest coarsest level solved by its inverse (FP32 inner cycles)

template <typename T>
struct PCArgs {
  int nlev;                       // levels s..L handled: nlev = L - s + 1
  int nu, nu_post;                // smoothing steps on the way down, on the way up
  T omega;
  double tol;
  int maxit;
  Lvl<T> lv[PC_MAXLEV];           // compact LDS geometry (px = nx, pxy = nx*ny)
  Lvl<double> lc;                 // coarsest level, FP64 coefficients
  RestrictW<T> rw[PC_MAXLEV];     // level q -> q+1
  ProlongW<T> pw[PC_MAXLEV];      // level q <- q+1
  int xoff[PC_MAXLEV], boff[PC_MAXLEV];   // LDS offsets (elements of T)
  int coff[PC_MAXLEV];            // staged coefficients and weights of levels 0..nlev-2 (T)
  int roff;                       // residual of the level being restricted (T, level 0's size)
  int xcoff, bcoff, xctoff;       // coarsest: FP64 x, b (in doubles), T copy of x (in T)
  int xslots;                     // room for the two x slots of pc_coarsest_block at xcoff
  int ccoff;                      // staged coarsest coefficients (doubles)
  Lvl<T> gl;                      // global geometry of level s
  T* gxs;                         // global x_s (output)
  const T* gbs;                   // global b_s (input)
  int* iters_slot;
  // FP32 inner cycles of the mixed-precision solve: the coarsest level's
  // inverse operator, transposed (n x n doubles, entry k n + l = (A^-1)_lk),
  // for an exact coarsest solve in place of the red/black iterations; null
  // otherwise (the FP64 solve keeps the reference's iterations)
  const double* cinv;
};


// Staged arrays of one level in LDS (axis lengths ex = nx+2, ey, ez):
// cwx cex | cwy cey | cwz cez, then for levels with a coarser one the
// restriction weights wx | wy | wz and the prolongation weights
// px nx | py ny | pz nz.  pc_stage_elems gives the length of the block.
__host__ __device__ inline int pc_stage_elems(int nx, int ny, int nz, bool transfer) {
  return (transfer ? 5 : 2) * (nx + ny + nz + 6);
}

// copies level G's arrays (and transfer weights when R, P are given) to s.
// Every load of a thread is issued before its first LDS store (clamped
// indices, no branch next to a load), so staging costs one load latency;
// threads from `first` on begin, and first moves to the next wave behind
// them, so that the levels' latencies overlap (a 16^3 level and three below
// it, with b: 5.7 us one level after the other).
template <typename T>
__device__ void pc_stage(T* s, const Lvl<T>& G, const RestrictW<T>* R, const ProlongW<T>* P, int& first) {
  const int ex = G.nx + 2, ey = G.ny + 2, ez = G.nz + 2;
  const int em = max(ex, max(ey, ez));
  const int t = ((int)threadIdx.x - first) & (PC_THREADS - 1);
  first = (first + em + 63) & ~63 & (PC_THREADS - 1);
  for (int c = t; c < em; c += PC_THREADS) {
    const int cx = min(c, ex - 1), cy = min(c, ey - 1), cz = min(c, ez - 1);
    T v[15];
    v[0] = G.cwx[cx];
    v[1] = G.cex[cx];
    v[2] = G.cwy[cy];
    v[3] = G.cey[cy];
    v[4] = G.cwz[cz];
    v[5] = G.cez[cz];
    if (R) {
      v[6] = R->wx[cx];
      v[7] = R->wy[cy];
      v[8] = R->wz[cz];
      v[9] = P->px_[cx];
      v[10] = P->nx_[cx];
      v[11] = P->py_[cy];
      v[12] = P->ny_[cy];
      v[13] = P->pz_[cz];
      v[14] = P->nz_[cz];
    }
    if (c < ex) {
      s[c] = v[0];
      s[ex + c] = v[1];
    }
    if (c < ey) {
      s[2 * ex + c] = v[2];
      s[2 * ex + ey + c] = v[3];
    }
    if (c < ez) {
      s[2 * (ex + ey) + c] = v[4];
      s[2 * (ex + ey) + ez + c] = v[5];
    }
    if (R) {
      T* w = s + 2 * (ex + ey + ez);
      T* p = w + (ex + ey + ez);
      if (c < ex) {
        w[c] = v[6];
        p[c] = v[9];
        p[ex + c] = v[10];
      }
      if (c < ey) {
        w[ex + c] = v[7];
        p[2 * ex + c] = v[11];
        p[2 * ex + ey + c] = v[12];
      }
      if (c < ez) {
        w[ex + ey + c] = v[8];
        p[2 * (ex + ey) + c] = v[13];
        p[2 * (ex + ey) + ez + c] = v[14];
      }
    }
  }
}

// level geometry G with its coefficient pointers moved to the staged copy s
template <typename T>
__device__ __forceinline__ Lvl<T> pc_lvl(const Lvl<T>& G, const T* s) {
  const int ex = G.nx + 2, ey = G.ny + 2, ez = G.nz + 2;
  Lvl<T> L = G;
  L.cwx = s;
  L.cex = s + ex;
  L.cwy = s + 2 * ex;
  L.cey = s + 2 * ex + ey;
  L.cwz = s + 2 * (ex + ey);
  L.cez = s + 2 * (ex + ey) + ez;
  return L;
}
template <typename T>
__device__ __forceinline__ RestrictW<T> pc_rw(const RestrictW<T>& W, const Lvl<T>& G, const T* s) {
  const int ex = G.nx + 2, ey = G.ny + 2, ez = G.nz + 2;
  RestrictW<T> R = W;
  const T* w = s + 2 * (ex + ey + ez);
  R.wx = w;
  R.wy = w + ex;
  R.wz = w + ex + ey;
  return R;
}
template <typename T>
__device__ __forceinline__ ProlongW<T> pc_pw(const ProlongW<T>& W, const Lvl<T>& G, const T* s) {
  const int ex = G.nx + 2, ey = G.ny + 2, ez = G.nz + 2;
  ProlongW<T> P = W;
  const T* p = s + 3 * (ex + ey + ez);
  P.px_ = p;
  P.nx_ = p + ex;
  P.py_ = p + 2 * ex;
  P.ny_ = p + 2 * ex + ey;
  P.pz_ = p + 2 * (ex + ey);
  P.nz_ = p + 2 * (ex + ey) + ez;
  return P;
}

// value of lane l of v (l a compile-time lane after unrolling)
__device__ __forceinline__ double pc_readlane(double v, int l) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u & 0xffffffffu), l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// What the coarsest solvers keep of one cell in registers: coefficients, c0
// and its reciprocal (see kd_quotient), b, and the indices of its neighbours
// in an x slot, whose element n is 0 (a neighbour outside the level).
struct PCCell {
  double c1, c2, c3, c4, c5, c6, c0, rc, bv;
  int nw, ne, ns, nn, nb, nt;
  int first;                           // i + j + k odd: the first half-sweep
  bool kept;                           // c0 is in kd_quotient's range

  __device__ __forceinline__ void load(const Lvl<double>& L, const double* b, int c, int n) {
    const int sy = L.nx, sz = L.nx * L.ny;
    const int i = c % L.nx + 1, j = (c / L.nx) % L.ny + 1, k = c / sz + 1;
    c1 = L.cwx[i]; c2 = L.cex[i]; c3 = L.cwy[j]; c4 = L.cey[j]; c5 = L.cwz[k]; c6 = L.cez[k];
    c0 = diag(c1, c2, c3, c4, c5, c6);
    rc = 1.0 / c0;
    kept = kd_divisor(c0);
    bv = b[c];
    nw = i > 1 ? c - 1 : n;
    ne = i < L.nx ? c + 1 : n;
    ns = j > 1 ? c - sy : n;
    nn = j < L.ny ? c + sy : n;
    nb = k > 1 ? c - sz : n;
    nt = k < L.nz ? c + sz : n;
    first = (i + j + k) & 1;
  }
  // the update of sor_at with neighbours from x
  __device__ __forceinline__ double sor(const double* x, double omega, double xold) const {
    const double t = c1 * x[nw] + c2 * x[ne] + c3 * x[ns] + c4 * x[nn] + c5 * x[nb] + c6 * x[nt];
    const double a = omega * (bv - t);
    double q = kd_quotient(a, c0, rc);
    if (kd_range(a) > KD_SPAN || !kept) q = a / c0;
    return q + (1.0 - omega) * xold;
  }
  __device__ __forceinline__ double resid(const double* x, double own) const {
    const double y = c0 * own + c1 * x[nw] + c2 * x[ne] + c3 * x[ns] + c4 * x[nn] + c5 * x[nb] + c6 * x[nt];
    return bv - y;
  }
};

// Coarsest rbgs_solver on up to 64 cells (src/rbgs_poisson_matrix.f90:47-179),
// cell c on lane c.  The stopping test sums the squared residuals in cell
// order (the reference's sequential sum, bit for bit), a chain of n dependent
// additions; on the path of the iterations it made up half of the solve.
// Here wave 0 iterates and waves 1 .. PC_BATCH form the norms of the batch of
// PC_BATCH iterations before, each of its own iteration: every iteration
// writes x into a slot of its own (whose element 64 is 0), so the solution
// at the iteration that passes is still there when the test is known, at most
// two batches later.  The persistent kernel of a 16^3 solve (8^3 and 4^3
// levels) takes 29.1 us against 54.9 us with the norm on the path and a
// division per update.
// All threads of the block (four waves or more) call this.  xs: PC_SMALL_X
// doubles; returns the iteration count (the reference's loop variable), *res
// the slot of x.
constexpr int PC_BATCH = 3, PC_SMALL_X = 2 * PC_BATCH * 65;
static __device__ __forceinline__ int pc_coarsest_small(double* __restrict__ xs, const double* __restrict__ b,
                                                        const Lvl<double>& L, double omega, double tol, int maxit,
                                                        double** res) {
  __shared__ double r0s;
  __shared__ int stop;                 // first iteration that passed (maxit: none yet)
  const int n = L.nx * L.ny * L.nz;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool own = lane < n;
  PCCell C;
  if (wave <= PC_BATCH) C.load(L, b, own ? lane : 0, 64);
  auto slot = [&](int q) { return xs + q * 65; };
  for (int q = threadIdx.x; q < PC_SMALL_X; q += blockDim.x) xs[q] = 0.0;
  if (threadIdx.x == 0) stop = maxit;
  __syncthreads();
  auto wsync = []() {                  // one wavefront orders its own LDS traffic
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  // sum of the lanes' r^2 in cell order (lanes without a cell add +0.0,
  // which leaves the non-negative sum unchanged)
  auto norm = [&](double r) -> double {
    const double r2 = own ? r * r : 0.0;
    double s = 0.0;
#pragma unroll
    for (int g = 0; g < 64; g += 16) {
      if (g >= n) break;
#pragma unroll
      for (int l = 0; l < 16; l++) s = s + pc_readlane(r2, g + l);
    }
    return s;
  };
  double xv = 0.0;                     // the lane's x after the last iteration (wave 0)
  int it0 = 0;                         // first iteration of the batch wave 0 runs
  for (;; it0 += PC_BATCH) {
    const int half = (it0 / PC_BATCH & 1) * PC_BATCH;
    if (wave == 0) {
      for (int u = 0; u < PC_BATCH; u++) {
        const double* prev = slot(u ? half + u - 1 : (PC_BATCH - half) + PC_BATCH - 1);
        double* cur = slot(half + u);
        if (own && C.first) {
          xv = C.sor(prev, omega, xv);
          cur[lane] = xv;
        }
        wsync();
        if (own && !C.first) {
          xv = C.sor(cur, omega, xv);
          cur[lane] = xv;
        }
        wsync();
      }
    } else if (wave <= PC_BATCH) {
      if (it0 == 0) {                  // |b - A 0|^2
        if (wave == 1) {
          const double s = norm(C.bv);
          if (lane == 0) r0s = s;
        }
      } else {
        const int it = it0 - PC_BATCH + wave - 1;
        const double* sl = slot((PC_BATCH - half) + wave - 1);
        const double rn = norm(C.resid(sl, sl[lane]));
        if (lane == 0 && it < maxit && sqrt(rn / r0s) <= tol) atomicMin(&stop, it);
      }
    }
    __syncthreads();
    if (stop < maxit || it0 >= maxit) break;   // (the batch just tested ends at it0 - 1)
    __syncthreads();
  }
  // the batch just tested holds the iteration that passed, or the last permitted one
  const int tested = it0 - PC_BATCH, last = min(stop, maxit - 1);
  *res = slot((tested / PC_BATCH & 1) * PC_BATCH + last - tested);
  return stop;
}

// sum over the wave, the tree of wave_sum (v[l] += v[l + 32], .. + 16, 8, 4,
// 2, 1; valid on lane 0) by lane moves in the vector units instead of LDS
__device__ __forceinline__ double pc_wave_sum(double v) {
  auto swap = [](double u, auto f) -> double {
    return __hiloint2double((int)f((unsigned)__double2hiint(u)), (int)f((unsigned)__double2loint(u)));
  };
  v += swap(v, [](unsigned u) { return __builtin_amdgcn_permlane32_swap(u, u, false, false)[1]; });
  v += swap(v, [](unsigned u) { return __builtin_amdgcn_permlane16_swap(u, u, false, false)[1]; });
  v += swap(v, [](unsigned u) { return (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x108, 0xf, 0xf, true); });
  v += swap(v, [](unsigned u) { return (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x104, 0xf, 0xf, true); });
  v += swap(v, [](unsigned u) { return (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x102, 0xf, 0xf, true); });
  v += swap(v, [](unsigned u) { return (unsigned)__builtin_amdgcn_update_dpp(0, (int)u, 0x101, 0xf, 0xf, true); });
  return v;
}

// Coarsest rbgs_solver on 65 to PC_THREADS cells, cell c on thread c with its
// coefficients in registers.  x lies in two slots (n + 1 doubles each, the
// last 0) that iterations use in turn; the norm of an iteration is formed
// beside the next one's half-sweeps (the squares and their wave sums beside
// the first, the sum over the waves beside the second), in coarse_norm's
// order, so an iteration costs its two barriers.  The persistent kernel of
// an 80 x 48 x 40 solve (coarsest level 10 x 6 x 5): 80.8 us against 163.6 us
// with the norm between the iterations.
// xs: the two slots; returns the iteration count, *res the slot of x.
static __device__ __forceinline__ int pc_coarsest_block(double* __restrict__ xs, const double* __restrict__ b,
                                                        const Lvl<double>& L, double omega, double tol, int maxit,
                                                        double** res) {
  __shared__ double part[2][PC_THREADS / 64];
  __shared__ int passed[2];
  __shared__ double r0s;
  const int n = L.nx * L.ny * L.nz;
  const int c = threadIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nwv = (n + 63) / 64;
  const bool own = c < n;
  PCCell C;
  if (own) C.load(L, b, c, n);
  for (int q = c; q < 2 * (n + 1); q += blockDim.x) xs[q] = 0.0;
  __syncthreads();
  double xv = 0.0;
  int it;
  for (it = 0;; it++) {
    const double* prev = xs + ((it + 1) & 1) * (n + 1);
    double* cur = xs + (it & 1) * (n + 1);
    const int par = it & 1;
    double nx = xv;
    if (own && C.first) {
      nx = C.sor(prev, omega, xv);
      cur[c] = nx;
    }
    if (wave < nwv) {
      const double r = own ? C.resid(prev, xv) : 0.0;
      const double s = pc_wave_sum(r * r);
      if (lane == 0) part[par][wave] = s;
    }
    __syncthreads();
    if (own && !C.first) {
      nx = C.sor(cur, omega, xv);
      cur[c] = nx;
    }
    xv = nx;
    if (c == PC_THREADS - 1) {         // the norm of iteration it - 1 (it = 0: of x = 0)
      double t = 0.0;
      for (int q = 0; q < nwv; q++) t += part[par][q];
      if (it == 0) r0s = t;
      passed[par] = it > 0 && sqrt(t / r0s) <= tol;
    }
    __syncthreads();
    if (passed[par]) {
      *res = const_cast<double*>(prev);
      return it - 1;
    }
    if (it >= maxit) {                 // iteration maxit - 1 did not pass either
      *res = const_cast<double*>(prev);
      return maxit;
    }
  }
}

// floor(n / d) for 0 <= n, d < 2^16 (levels held in LDS are far smaller):
// one 64-bit multiply by m = floor((2^32 - 1) / d) + 1 instead of an integer
// division (the error n * (m - 2^32 / d) / 2^32 < n / 2^32 stays below 1/d)
__device__ __forceinline__ unsigned long long pc_magic(int d) { return 0xFFFFFFFFull / (unsigned)d + 1ull; }
__device__ __forceinline__ int pc_div(int n, unsigned long long m) {
  return (int)(((unsigned long long)(unsigned)n * m) >> 32);
}

// Cells of a compact LDS level (px = nx, pxy = nx ny): cell q = (i-1) +
// nx (j-1) + nx ny (k-1); neighbours outside the level read as 0, the
// homogeneous ghost (ldz).  Values and operation order are those of
// sor_at / apply_at.
template <typename T>
struct PCNb {
  T w, e, s, n, b, t;
};
template <typename T>
__device__ __forceinline__ PCNb<T> pc_nb(const T* x, const Lvl<T>& L, int i, int j, int k, int q) {
  const int sy = L.nx, sz = L.nx * L.ny;
  PCNb<T> v;
  v.w = i > 1 ? x[q - 1] : T(0);
  v.e = i < L.nx ? x[q + 1] : T(0);
  v.s = j > 1 ? x[q - sy] : T(0);
  v.n = j < L.ny ? x[q + sy] : T(0);
  v.b = k > 1 ? x[q - sz] : T(0);
  v.t = k < L.nz ? x[q + sz] : T(0);
  return v;
}

template <typename T>
__device__ void pc_colour(T* x, const T* b, const Lvl<T>& L, T omega, int colour, bool zero) {
  const int hx = (L.nx + 1) / 2;
  const int n = hx * L.ny * L.nz;
  const unsigned long long mh = pc_magic(hx), my = pc_magic(L.ny);
  for (int c = threadIdx.x; c < n; c += blockDim.x) {
    const int row = pc_div(c, mh);                 // (j-1) + ny (k-1)
    const int tt = c - row * hx, kk = pc_div(row, my);
    const int j = row - kk * L.ny + 1, k = kk + 1;
    const int i = 1 + ((j + k + colour) & 1) + 2 * tt;
    if (i <= L.nx) {
      const int q = (i - 1) + L.nx * row;
      const T c1 = L.cwx[i], c2 = L.cex[i], c3 = L.cwy[j], c4 = L.cey[j], c5 = L.cwz[k], c6 = L.cez[k];
      if (zero) {
        T z = T(0);
        T temp = c1 * z + c2 * z + c3 * z + c4 * z + c5 * z + c6 * z;
        x[q] = omega * (b[q] - temp) / diag(c1, c2, c3, c4, c5, c6) + (T(1) - omega) * z;
      } else {
        const T c0 = diag(c1, c2, c3, c4, c5, c6);
        const PCNb<T> v = pc_nb(x, L, i, j, k, q);
        const T temp = c1 * v.w + c2 * v.e + c3 * v.s + c4 * v.n + c5 * v.b + c6 * v.t;
        x[q] = omega * (b[q] - temp) / c0 + (T(1) - omega) * x[q];
      }
    }
  }
  __syncthreads();
}

template <typename T>
__device__ void pc_zero(T* a, int n) {
  for (int c = threadIdx.x; c < n; c += blockDim.x) a[c] = T(0);
  __syncthreads();
}

template <typename T>
__device__ void pc_smooth(T* x, const T* b, const Lvl<T>& L, T omega, int nu, bool zero_start) {
  int n = L.nx * L.ny * L.nz;
  if (zero_start) pc_zero(x, n);   // zero-start colour 0 writes only its own colour
  for (int it = 0; it < nu; it++) {
    pc_colour(x, b, L, omega, 0, zero_start && it == 0);
    pc_colour(x, b, L, omega, 1, false);
  }
}

// Pairs of cells (i odd, i + 1) of a compact level owned by a thread through a
// whole leg, everything they need in registers: coefficients, c0 and its
// reciprocal, b and the LDS indices of their neighbours (outside the level
// the two zeros behind x, elements n and n + 1).  A pair holds one cell of each
// colour; entry h of the arrays is the cell half-sweep h updates.  Setting a
// pair up costs about what one half-sweep over it did when each formed these
// anew; up to two pairs per thread (4096 cells of even rows).
// The FP32 kernel of a 64^3 solve (16^3 level on top): 33.8 against 38.2 us.
constexpr int PC_PAIRS = 2;
template <typename T>
struct PCPair {
  T c1[2], c2[2], c0[2], rc[2], bv[2], c3, c4, c5, c6;
  int q[2], w[2], e[2], o[2];          // cell, its x neighbours, 0 or 1: its place in the pair
  int s, n, b, t;                      // y and z neighbours of the pair's first cell
  bool in[2], kept;

  __device__ __forceinline__ void load(const Lvl<T>& L, const T* bs, int p, unsigned long long mh,
                                       unsigned long long my) {
    const int hx = (L.nx + 1) / 2, np = hx * L.ny * L.nz, nc = L.nx * L.ny * L.nz;
    const bool on = p < np;
    const int pp = on ? p : 0;
    const int row = pc_div(pp, mh), kk = pc_div(row, my);
    const int i = 1 + 2 * (pp - row * hx), j = row - kk * L.ny + 1, k = kk + 1;
    const int q0 = (i - 1) + L.nx * row, sz = L.nx * L.ny;
    const int f = (j + k) & 1;           // the cell of the first half-sweep (i + j + k odd): 0 first, 1 second
    c3 = L.cwy[j]; c4 = L.cey[j]; c5 = L.cwz[k]; c6 = L.cez[k];
    s = j > 1 ? q0 - L.nx : nc;
    n = j < L.ny ? q0 + L.nx : nc;
    b = k > 1 ? q0 - sz : nc;
    t = k < L.nz ? q0 + sz : nc;
    kept = true;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int c = h == 0 ? f : 1 - f, ic = i + c;
      in[h] = on && ic <= L.nx;
      const int is = in[h] ? ic : 1;
      o[h] = c;
      q[h] = in[h] ? q0 + c : 0;
      w[h] = ic > 1 ? q0 + c - 1 : nc;
      e[h] = ic < L.nx ? q0 + c + 1 : nc;
      c1[h] = L.cwx[is];
      c2[h] = L.cex[is];
      c0[h] = diag(c1[h], c2[h], c3, c4, c5, c6);
      rc[h] = T(1) / c0[h];
      bv[h] = bs ? bs[q[h]] : T(0);
      if constexpr (sizeof(T) == 8) kept = kept && kd_divisor(c0[h]);
    }
  }
  __device__ __forceinline__ void half(T* x, T omega, int h) const {
    if (!in[h]) return;
    const int c = o[h];
    const T xv = x[q[h]];
    const T tm = c1[h] * x[w[h]] + c2[h] * x[e[h]] + c3 * x[s + c] + c4 * x[n + c] + c5 * x[b + c] + c6 * x[t + c];
    const T a = omega * (bv[h] - tm);
    T v;
    if constexpr (sizeof(T) == 8) {
      v = kd_quotient(a, c0[h], rc[h]);
      if (kd_range(a) > KD_SPAN || !kept) v = a / c0[h];
    } else {
      v = a * rc[h];
      v = __builtin_fmaf(__builtin_fmaf(-c0[h], v, a), rc[h], v);
    }
    x[q[h]] = v + (T(1) - omega) * xv;
  }
  __device__ __forceinline__ void resid(T* r, const T* x) const {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      if (!in[h]) continue;
      const int c = o[h];
      const T y = c0[h] * x[q[h]] + c1[h] * x[w[h]] + c2[h] * x[e[h]] + c3 * x[s + c] + c4 * x[n + c] +
                  c5 * x[b + c] + c6 * x[t + c];
      r[q[h]] = bv[h] - y;
    }
  }
};

// nu red/black iterations on x by owned pairs, then (r given) the residual
// into r.  Both colours' half-sweeps end with a barrier, as pc_colour's do.
template <typename T>
__device__ __forceinline__ void pc_smooth_pairs(T* x, const T* b, T* r, const Lvl<T>& L, T omega, int nu) {
  const int hx = (L.nx + 1) / 2, np = hx * L.ny * L.nz;
  const unsigned long long mh = pc_magic(hx), my = pc_magic(L.ny);
  const bool two = np > (int)blockDim.x;             // uniform
  PCPair<T> P[PC_PAIRS];
  P[0].load(L, b, threadIdx.x, mh, my);
  if (two) P[1].load(L, b, threadIdx.x + blockDim.x, mh, my);
  for (int it = 0; it < nu; it++) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      P[0].half(x, omega, h);
      if (two) P[1].half(x, omega, h);
      __syncthreads();
    }
  }
  if (r) {
    P[0].resid(r, x);
    if (two) P[1].resid(r, x);
    __syncthreads();
  }
}

// residual of every fine cell into r (compact, one per thread in turn; formed:
// r holds it already), then the restriction from r: the same values and sums
// as the per-level kernels
template <typename T, typename TC>
__device__ void pc_restrict(TC* bc, T* r, const T* x, const T* b, const Lvl<T>& F, int cnx, int cny, int cnz,
                            const RestrictW<T>& W, bool formed) {
  const int nf = formed ? 0 : F.nx * F.ny * F.nz;
  const unsigned long long mx = pc_magic(F.nx), my = pc_magic(F.ny);
  for (int c = threadIdx.x; c < nf; c += blockDim.x) {
    const int row = pc_div(c, mx), kk = pc_div(row, my);
    const int i = c - row * F.nx + 1, j = row - kk * F.ny + 1, k = kk + 1;
    const T c1 = F.cwx[i], c2 = F.cex[i], c3 = F.cwy[j], c4 = F.cey[j], c5 = F.cwz[k], c6 = F.cez[k];
    const T c0 = diag(c1, c2, c3, c4, c5, c6);
    const PCNb<T> v = pc_nb(x, F, i, j, k, c);
    const T y = c0 * x[c] + c1 * v.w + c2 * v.e + c3 * v.s + c4 * v.n + c5 * v.b + c6 * v.t;
    r[c] = b[c] - y;
  }
  if (!formed) __syncthreads();
  const int n = cnx * cny * cnz;
  const unsigned long long mcx = pc_magic(cnx), mcy = pc_magic(cny);
  const int sy = F.nx, sz = F.nx * F.ny;
  for (int c = threadIdx.x; c < n; c += blockDim.x) {
    const int row = pc_div(c, mcx), kk = pc_div(row, mcy);
    const int ic = c - row * cnx + 1, jc = row - kk * cny + 1, kc = kk + 1;
    int iz, ip, jz, jp, kz, kp;
    T ax1, ax2, ay1, ay2, az1, az2;
    restrict_axis(W.wx, W.sx, ic, iz, ip, ax1, ax2);
    restrict_axis(W.wy, W.sy, jc, jz, jp, ay1, ay2);
    restrict_axis(W.wz, W.sz, kc, kz, kp, az1, az2);
    T v111 = ax1 * ay1 * az1, v211 = ax2 * ay1 * az1, v121 = ax1 * ay2 * az1, v221 = ax2 * ay2 * az1;
    T v112 = ax1 * ay1 * az2, v212 = ax2 * ay1 * az2, v122 = ax1 * ay2 * az2, v222 = ax2 * ay2 * az2;
    T vol_c = v111 + v211 + v121 + v221 + v112 + v212 + v122 + v222;
    auto R = [&](int a, int bb, int cc) { return r[(a - 1) + sy * (bb - 1) + sz * (cc - 1)]; };
    T s = v111 * R(ip, jp, kp) + v211 * R(iz, jp, kp) + v121 * R(ip, jz, kp) + v221 * R(iz, jz, kp) +
          v112 * R(ip, jp, kz) + v212 * R(iz, jp, kz) + v122 * R(ip, jz, kz) + v222 * R(iz, jz, kz);
    bc[c] = (TC)(s / vol_c);
  }
  __syncthreads();
}

// x_f += P x_c (prolong_at's weights, terms and order) on a compact level that
// halves every axis, by pairs of fine cells (i odd, i + 1) with one parent:
// they share the rows' indices and weights and the parent's
// values.  What a cell costs is instructions (onto 16^3, cell by cell, 8.4 us
// of a 54 us FP64 kernel; by pairs 49 in all, FP32 36 and 29 us, staging
// included).
template <typename T>
__device__ void pc_prolong_pairs(T* xf, const T* xc, const Lvl<T>& F, const Lvl<T>& C, const ProlongW<T>& W) {
  const int hx = C.nx, np = hx * F.ny * F.nz;
  const unsigned long long mh = pc_magic(hx), my = pc_magic(F.ny);
  for (int p = threadIdx.x; p < np; p += blockDim.x) {
    const int row = pc_div(p, mh), kk = pc_div(row, my);
    const int ci = p - row * hx, j = row - kk * F.ny + 1, k = kk + 1, i = 2 * ci + 1;   // ci from 0
    const bool jo = j & 1, ko = k & 1;
    const T sy = jo ? W.py_[j] : W.ny_[j], ny = jo ? W.py_[j + 1] : W.ny_[j - 1];
    const T sz = ko ? W.pz_[k] : W.nz_[k], nz = ko ? W.pz_[k + 1] : W.nz_[k - 1];
    const int cj = (j - 1) >> 1, ck = (k - 1) >> 1, nj = jo ? cj - 1 : cj + 1, nk = ko ? ck - 1 : ck + 1;   // from 0
    const bool vy = nj >= 0 && nj < C.ny, vz = nk >= 0 && nk < C.nz;
    const bool vw = ci > 0, ve = ci + 1 < hx;
    const int ow = vw ? -1 : 0, oe = ve ? 1 : 0;
    const T* a = xc + ci + hx * (cj + C.ny * ck);
    const T* rows[4] = {a, a + (vy ? hx * (nj - cj) : 0), a + (vz ? hx * C.ny * (nk - ck) : 0),
                        a + (vy && vz ? hx * (nj - cj + C.ny * (nk - ck)) : 0)};
    const bool in[4] = {true, vy, vz, vy && vz};
    T w[4], m[4], e[4];                              // west of the parent's column, in it, east of it
#pragma unroll
    for (int r = 0; r < 4; r++) {
      w[r] = rows[r][ow];
      m[r] = rows[r][0];
      e[r] = rows[r][oe];
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      w[r] = in[r] && vw ? w[r] : T(0);
      m[r] = in[r] ? m[r] : T(0);
      e[r] = in[r] && ve ? e[r] : T(0);
    }
    T* x = xf + 2 * p;
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const T sx = c ? W.nx_[i + 1] : W.px_[i], nx = c ? W.nx_[i] : W.px_[i + 1];
      const T* o = c ? e : w;
      const T num = sx * sy * sz * m[0] + nx * sy * sz * o[0] + sx * ny * sz * m[1] + sx * sy * nz * m[2] +
                    nx * ny * sz * o[1] + nx * sy * nz * o[2] + sx * ny * nz * m[3] + nx * ny * nz * o[3];
      x[c] = x[c] + num / ((sx + nx) * (sy + ny) * (sz + nz));
    }
  }
  __syncthreads();
}

// x_f += P x_c on any compact level
template <typename T>
__device__ void pc_prolong_add(T* xf, const T* xc, const Lvl<T>& F, const Lvl<T>& Cc, const ProlongW<T>& W) {
  if (W.sx == 2 && W.sy == 2 && W.sz == 2 && F.nx == 2 * Cc.nx && F.ny == 2 * Cc.ny && F.nz == 2 * Cc.nz) {
    pc_prolong_pairs(xf, xc, F, Cc, W);
    return;
  }
  const int n = F.nx * F.ny * F.nz;
  const unsigned long long mx = pc_magic(F.nx), my = pc_magic(F.ny);
  auto V = [&](int a, int bb, int cc) -> T {
    return (a >= 1 && a <= Cc.nx && bb >= 1 && bb <= Cc.ny && cc >= 1 && cc <= Cc.nz)
               ? xc[(a - 1) + Cc.nx * ((bb - 1) + Cc.ny * (cc - 1))]
               : T(0);
  };
  for (int c = threadIdx.x; c < n; c += blockDim.x) {
    const int row = pc_div(c, mx), kk = pc_div(row, my);
    const int i = c - row * F.nx + 1, j = row - kk * F.ny + 1, k = kk + 1;
    int ci, ni, cj, nj, ck, nk;
    T wsx, wnx, wsy, wny, wsz, wnz;
    prolong_axis(W.px_, W.nx_, W.sx, i, ci, ni, wsx, wnx);
    prolong_axis(W.py_, W.ny_, W.sy, j, cj, nj, wsy, wny);
    prolong_axis(W.pz_, W.nz_, W.sz, k, ck, nk, wsz, wnz);
    T num = wsx * wsy * wsz * V(ci, cj, ck) + wnx * wsy * wsz * V(ni, cj, ck) + wsx * wny * wsz * V(ci, nj, ck) +
            wsx * wsy * wnz * V(ci, cj, nk) + wnx * wny * wsz * V(ni, nj, ck) + wnx * wsy * wnz * V(ni, cj, nk) +
            wsx * wny * wnz * V(ci, nj, nk) + wnx * wny * wnz * V(ni, nj, nk);
    xf[c] = xf[c] + num / ((wsx + wnx) * (wsy + wny) * (wsz + wnz));
  }
  __syncthreads();
}

// Levels smoothed by owned pairs: those with more than one cell of a colour
// for some threads.  Below, a half-sweep is short of setting the pairs up (a
// V(1,1) cycle over 32 x 2 x 16 cells and five smaller levels: 42.8 us with
// owned pairs throughout, 36.9 us without).
template <typename T>
__device__ __forceinline__ bool pc_owned(const Lvl<T>& L) {
  const int np = ((L.nx + 1) / 2) * L.ny * L.nz;
  return np > PC_THREADS && np <= PC_PAIRS * PC_THREADS;
}

template <typename T>
__device__ __forceinline__ void coarse_vcycle_block(const PCArgs<T>& A) {
  extern __shared__ __align__(16) unsigned char pc_smem[];
  T* sm = reinterpret_cast<T*>(pc_smem);
  double* smd = reinterpret_cast<double*>(pc_smem);
  __shared__ double sh[PC_THREADS / 64];
  __shared__ double seq[64];
  const int top = A.nlev - 1;                     // index of the coarsest level
  // coefficients and transfer weights into LDS, b_s from global
  {
    const Lvl<T>& L = A.lv[0];
    const int n = L.nx * L.ny * L.nz;
    const unsigned long long mx = pc_magic(L.nx), my = pc_magic(L.ny);
    // four loads in flight per thread (clamped cells) before the LDS stores
    T v[4];
    auto load = [&](int c0) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int c = min(c0 + u * PC_THREADS, n - 1);
        const int row = pc_div(c, mx), kk = pc_div(row, my);
        v[u] = A.gbs[lidx(A.gl, c - row * L.nx + 1, row - kk * L.ny + 1, kk + 1)];
      }
    };
    load(threadIdx.x);
    int first = 0;
    for (int q = 0; q < top; q++) pc_stage(sm + A.coff[q], A.lv[q], &A.rw[q], &A.pw[q], first);
    pc_stage(smd + A.ccoff, A.lc, (const RestrictW<double>*)nullptr, (const ProlongW<double>*)nullptr, first);
    for (int c0 = threadIdx.x; c0 < n; c0 += 4 * PC_THREADS) {
      if (c0 >= 4 * PC_THREADS) load(c0);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int c = c0 + u * PC_THREADS;
        if (c < n) {
          if (top == 0) smd[A.bcoff + c] = (double)v[u];
          else sm[A.boff[0] + c] = v[u];
        }
      }
    }
    __syncthreads();
  }
  // down-leg: levels 0 .. top-1 (local numbering)
  for (int q = 0; q < top; q++) {
    const T* st = sm + A.coff[q];
    const Lvl<T> L = pc_lvl(A.lv[q], st);
    const RestrictW<T> W = pc_rw(A.rw[q], A.lv[q], st);
    T* x = sm + A.xoff[q];
    const T* b = sm + A.boff[q];
    const bool pairs = pc_owned(L);
    if (pairs) {
      pc_zero(x, L.nx * L.ny * L.nz + 2);
      pc_smooth_pairs(x, b, sm + A.roff, L, A.omega, A.nu);
    } else {
      pc_smooth(x, b, L, A.omega, A.nu, true);
    }
    if (q + 1 < top) {
      const Lvl<T>& C = A.lv[q + 1];
      pc_restrict<T, T>(sm + A.boff[q + 1], sm + A.roff, x, b, L, C.nx, C.ny, C.nz, W, pairs);
    } else {
      pc_restrict<T, double>(smd + A.bcoff, sm + A.roff, x, b, L, A.lc.nx, A.lc.ny, A.lc.nz, W, pairs);
    }
  }
  // coarsest solve in FP64
  const double* xc;
  {
    const Lvl<double> L = pc_lvl(A.lc, (const double*)(smd + A.ccoff));
    double* x = smd + A.xcoff;
    const double* b = smd + A.bcoff;
    int n = L.nx * L.ny * L.nz;
    if (A.cinv && n <= PC_CINV_MAX) {   // x = A^-1 b, one lane per cell
      if ((int)threadIdx.x < n) {
        double v = 0.0;
#pragma unroll 8
        for (int k = 0; k < n; k++) v += A.cinv[(long)k * n + threadIdx.x] * b[k];
        x[threadIdx.x] = v;
      }
      if (threadIdx.x == 0 && A.iters_slot) *A.iters_slot = 0;
      __syncthreads();
    } else if (n == 1) {
      if (threadIdx.x == 0) {
        x[0] = b[0] / diag(L.cwx[1], L.cex[1], L.cwy[1], L.cey[1], L.cwz[1], L.cez[1]);
        if (A.iters_slot) *A.iters_slot = 0;
      }
      __syncthreads();
    } else if (n <= 64) {
      const int it = pc_coarsest_small(smd + A.xcoff, b, L, (double)A.omega, A.tol, A.maxit, &x);
      if (threadIdx.x == 0 && A.iters_slot) *A.iters_slot = it;
    } else if (A.xslots) {
      const int it = pc_coarsest_block(smd + A.xcoff, b, L, (double)A.omega, A.tol, A.maxit, &x);
      if (threadIdx.x == 0 && A.iters_slot) *A.iters_slot = it;
    } else {
      pc_zero(x, n);
      double r0 = coarse_norm(x, b, L, sh, seq);
      int it;
      for (it = 0; it < A.maxit; it++) {
        pc_colour(x, b, L, (double)A.omega, 0, false);
        pc_colour(x, b, L, (double)A.omega, 1, false);
        double rn = coarse_norm(x, b, L, sh, seq);
        if (sqrt(rn / r0) <= A.tol) break;
      }
      if (threadIdx.x == 0 && A.iters_slot) *A.iters_slot = it;
      __syncthreads();
    }
    xc = x;
    if (top > 0) {
      T* xt = sm + A.xctoff;
      for (int c = threadIdx.x; c < n; c += blockDim.x) xt[c] = (T)x[c];
      __syncthreads();
    }
  }
  // up-leg
  for (int q = top - 1; q >= 0; q--) {
    const T* st = sm + A.coff[q];
    const Lvl<T> L = pc_lvl(A.lv[q], st);
    const ProlongW<T> P = pc_pw(A.pw[q], A.lv[q], st);
    T* x = sm + A.xoff[q];
    const T* b = sm + A.boff[q];
    if (q + 1 < top) pc_prolong_add(x, sm + A.xoff[q + 1], L, A.lv[q + 1], P);
    else {
      Lvl<T> C = A.lv[top];   // geometry of the coarsest in T, compact
      pc_prolong_add(x, sm + A.xctoff, L, C, P);
    }
    if (pc_owned(L)) pc_smooth_pairs(x, b, (T*)nullptr, L, A.omega, A.nu_post);
    else pc_smooth(x, b, L, A.omega, A.nu_post, false);
  }
  // x_s to global
  {
    const Lvl<T>& L = A.lv[0];
    int n = L.nx * L.ny * L.nz;
    for (int c = threadIdx.x; c < n; c += blockDim.x) {
      int i = c % L.nx + 1, j = (c / L.nx) % L.ny + 1, k = c / (L.nx * L.ny) + 1;
      A.gxs[lidx(A.gl, i, j, k)] = (top == 0) ? (T)xc[c] : sm[A.xoff[0] + c];
    }
  }
}

// Coarsest solve of 2 to 64 cells for the per-level path (level arrays in
// global memory): what k_coarse_solve computes, 4^3 in 17 against 124 us.
static __global__ void __launch_bounds__(COARSE_THREADS)
k_coarse_small(double* __restrict__ x, const double* __restrict__ b, Lvl<double> L, double omega, double tol,
               int maxit, int* __restrict__ iters_slot) {
  __shared__ double xs[PC_SMALL_X], bs[64];
  const int n = L.nx * L.ny * L.nz, c = threadIdx.x;
  long q = 0;
  if (c < n) {
    q = lidx(L, c % L.nx + 1, (c / L.nx) % L.ny + 1, c / (L.nx * L.ny) + 1);
    bs[c] = b[q];
  }
  __syncthreads();
  double* xr;
  const int it = pc_coarsest_small(xs, bs, L, omega, tol, maxit, &xr);
  if (c < n) x[q] = xr[c];
  if (c == 0 && iters_slot) *iters_slot = it;
}

template <typename T>
__global__ void __launch_bounds__(PC_THREADS) k_coarse_vcycle(PCArgs<T> A) {
  coarse_vcycle_block<T>(A);
}

}  // namespace pepsmg
