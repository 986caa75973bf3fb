// pepsmg_ops.h -- host-side launch helpers shared by the single-grid and
// batched solvers: block decompositions of the z-march kernels and one
// launcher per operation on one level.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <utility>

#include "pepsmg_coarse.h"
#include "pepsmg_fused.h"
#include "pepsmg_internal.h"
#include "pepsmg_march.h"
#include "pepsmg_block.h"

namespace pepsmg {

// tile height of the fine-level residual kernels (norm, refinement update,
// CG steps)
constexpr int RESID_TY = 16;
// the refinement kernels' tile height on levels of 512 rows or more: 32
// rows halve the share of the one-row y ring re-read per tile (512^3 mixed
// solve 18.75 against 19.1 ms; two 256-thread blocks per CU by LDS either
// way).  Smaller levels keep 16: at about 2048 blocks, 32-row tiles leave
// z-chunks of 4 planes at 256^3, half of them halo.
constexpr int RESID_TY_BIG = 32;

// ---------------------------------------------------------------------------
// Launch helpers
static inline dim3 grid3(int nx, int ny, int nz, int bx, int by) {
  return dim3((unsigned)((nx + bx - 1) / bx), (unsigned)((ny + by - 1) / by), (unsigned)nz);
}

template <typename T>
struct Ops {
  hipStream_t s;
  int tile_y = 0;

  // x tile width of the fused smoother: 64 cells in FP64, 128 in FP32 (same
  // bytes per row)
  static constexpr int FTX = sizeof(T) == 8 ? 64 : 128;

  // Blocks of `kern` (launched with `threads` threads) that are resident on
  // the device at once: blocks per CU from the occupancy calculator times
  // the CU count (cached per kernel and device).
  static int resident(const void* kern, int threads) {
    static std::mutex mu;
    static std::map<std::pair<const void*, int>, int> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    std::lock_guard<std::mutex> lock(mu);
    auto key = std::make_pair(kern, dev);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    int per = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, threads, 0) != hipSuccess) per = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 0;
    return cache[key] = per * cus;
  }

  // nxy tiles split into chunks of at least 4 planes fill the device's
  // resident blocks exactly
  static bool one_wave(const DevLevel<T>& d, long nxy, int resident_blocks) {
    return resident_blocks > 0 && resident_blocks % nxy == 0 && d.nz / (resident_blocks / nxy) >= 4;
  }

  // Block decomposition of the fused smoother: TX x TY tiles marching
  // through z-chunks (even, so every chunk starts on an odd plane).  When
  // the tiles divide the resident block count, one chunk count fills the
  // device with exactly one wave of blocks (512^3: 0.58 against 0.63 ms in
  // FP64; 256^3: 73 against 100 us), chunks of at least 4 planes.
  // Otherwise about 2048 blocks, a multiple of 8 chunks (one z-slab per
  // XCD), chunks of at least 12 planes on levels of 192 or more planes and
  // of 2 below: levels of 128 planes and fewer are bound by the latency of
  // the march, not by bytes (FP32 smoother at 32^3 / 64^3: 6.8 / 7.5 us
  // against 8.2 / 8.7 us with chunks of 4 planes).
  // batched: the launch covers many problems at once, so it is bound by
  // bytes rather than latency and keeps chunks of at least 4 planes (12
  // from 96 planes on), which re-read fewer halo planes.
  static FusedGrid fused_grid(const DevLevel<T>& d, int TX, int TY, int resident_blocks = 0, bool batched = false) {
    FusedGrid G;
    G.gx = (d.nx + TX - 1) / TX;
    G.gy = (d.ny + TY - 1) / TY;
    long nxy = (long)G.gx * G.gy;
    long nch;
    if (one_wave(d, nxy, resident_blocks)) {
      nch = resident_blocks / nxy;
    } else {
      const int min_planes = batched ? 4 : 2, long_from = batched ? 96 : 192;
      nch = std::max(1L, std::min<long>((2048 + nxy - 1) / nxy, (d.nz + min_planes - 1) / min_planes));
      if (nch < 8 && d.nz >= 64) nch = 8;   // one z-slab per XCD: tile rings hit the XCD's own L2
      if (nch >= 8) nch = (nch + 7) / 8 * 8;
      if (d.nz >= long_from) nch = std::min<long>(nch, std::max<long>(8, d.nz / 12 / 8 * 8));
    }
    int kc = (int)((d.nz + nch - 1) / nch);
    if (kc & 1) kc++;                      // even chunks: every chunk starts on an odd plane
    G.kchunk = kc;
    G.nch = (d.nz + G.kchunk - 1) / G.kchunk;
    // XCD-aware order for tiles of 2048 cells or more (512^3, one wave:
    // FP64 64 x 32 0.551 against 0.572 ms, FP32 128 x 32 0.289 against
    // 0.298 ms); 64 x 16 FP64 tiles are faster in chunk-fastest order
    // (0.595 against 0.620 ms)
    G.order = TX * TY >= 2048 ? 1 : 0;
    return G;
  }

  // resident blocks of the tile shape's plain kernel (every mode of a shape
  // uses the same decomposition, so mode 2's partial sums have one slot per
  // block of it)
  template <int TX, int TY, int PF>
  static int fused_resident() {
    return resident((const void*)k_rb_fused<T, TX, TY, 0, PF>, fused_threads(TX, TY));
  }

  // output buffer of the next fused launch (nullptr: d.x2)
  T* fused_out = nullptr;
  // modes 3 and 4 (FP64): the caller's padded arrays (pointers at cell
  // (1,1,1)) and their layout
  const T* caller_x = nullptr;
  const T* caller_b = nullptr;
  T* caller_sol = nullptr;
  Lvl<T> caller_lvl{};

  // DOWN: mode 0 marching each chunk from the top (k_rb_fused_down), same
  // decomposition and values
  template <int TX, int TY, int MODE, int PF, bool DOWN = false>
  void fused_launch(DevLevel<T>& d, T omega, double* partial) {
    FusedGrid G = fused_grid(d, TX, TY, fused_resident<TX, TY, PF>());
    unsigned nb = (unsigned)(G.gx * G.gy * G.nch);
    const T* xi = MODE == 3 ? caller_x : d.x;
    const T* b = MODE == 3 ? caller_b : d.b;
    T* ext = MODE == 3 ? d.b : (MODE == 4 ? caller_sol : nullptr);
    if constexpr (DOWN) {
      static_assert(MODE == 0 && PF == 1, "downward march: plain iterations, one plane of look-ahead");
      hipLaunchKernelGGL((k_rb_fused_down<T, TX, TY, MODE, PF>), dim3(nb), dim3(fused_threads(TX, TY)), 0, s,
                         fused_out ? fused_out : d.x2, xi, b, d.L(), omega, G, partial, d.L(), ext);
    } else {
      hipLaunchKernelGGL((k_rb_fused<T, TX, TY, MODE, PF>), dim3(nb), dim3(fused_threads(TX, TY)), 0, s,
                         fused_out ? fused_out : d.x2, xi, b, d.L(), omega, G, partial,
                         (MODE == 3 || MODE == 4) ? caller_lvl : d.L(), ext);
    }
  }

  template <int TX, int TY, int PF>
  void fused_mode(DevLevel<T>& d, T omega, int mode, double* partial, bool down) {
    if (mode == 1) fused_launch<TX, TY, 1, PF>(d, omega, nullptr);
    else if constexpr (sizeof(T) == 8) {
      if (mode == 2) fused_launch<TX, TY, 2, PF>(d, omega, partial);
      else if (mode == 3) fused_launch<TX, TY, 3, PF>(d, omega, partial);
      else if (mode == 4) fused_launch<TX, TY, 4, PF>(d, omega, nullptr);
      else fused_plain<TX, TY, PF>(d, omega, down);
    } else {
      fused_plain<TX, TY, PF>(d, omega, down);
    }
  }
  // The decomposition is sized by the upward kernel's residency, so a tile
  // shape whose downward kernel holds fewer blocks per CU (FP32 64 x 16: 137
  // against 127 registers) marches up.
  template <int TX, int TY, int PF>
  void fused_plain(DevLevel<T>& d, T omega, bool down) {
    if constexpr (PF == 1) {
      if (down && resident((const void*)k_rb_fused_down<T, TX, TY, 0, 1>, fused_threads(TX, TY)) ==
                      fused_resident<TX, TY, 1>()) {
        fused_launch<TX, TY, 0, 1, true>(d, omega, nullptr);
        return;
      }
    }
    d.fused_up = true;
    fused_launch<TX, TY, 0, PF>(d, omega, nullptr);
  }

  template <int TX>
  void fused_tx(DevLevel<T>& d, T omega, int mode, int ty, double* partial, bool down) {
    if (ty == 32) {
      fused_mode<TX, 32, 1>(d, omega, mode, partial, down);
    } else if (ty == 16) {
      if (prefetch == 2) fused_mode<TX, 16, 2>(d, omega, mode, partial, false);
      else fused_mode<TX, 16, 1>(d, omega, mode, partial, down);
    } else {
      if (prefetch == 2) fused_mode<TX, 8, 2>(d, omega, mode, partial, false);
      else fused_mode<TX, 8, 1>(d, omega, mode, partial, down);
    }
  }
  template <int TX>
  int fused_resident_tx(int ty) const {
    if (ty == 32) return fused_resident<TX, 32, 1>();
    if (ty == 16) return prefetch == 2 ? fused_resident<TX, 16, 2>() : fused_resident<TX, 16, 1>();
    return prefetch == 2 ? fused_resident<TX, 8, 2>() : fused_resident<TX, 8, 1>();
  }
  // blocks of one fused launch on level d (partial sums of mode 2)
  int fused_blocks(const DevLevel<T>& d) const {
    int tx = tx_used(d), ty = ty_used(d);
    int res = (sizeof(T) == 4 && tx == 64) ? fused_resident_tx<64>(ty) : fused_resident_tx<FTX>(ty);
    FusedGrid G = fused_grid(d, tx, ty, res);
    return G.gx * G.gy * G.nch;
  }

  // tile sizes in use: width 64 cells in FP64 and 128 in FP32 (the same
  // bytes per row) unless set
  int tile_x = 0;
  // Unless set, the tile follows the level: 64 x 32 (FP64) and 128 x 32 (FP32)
  // on levels of 256 rows or more (FP64 512^3 solve with 64 x 32 tiles in
  // XCD-aware order: 45.4 against 47.5 ms with 64 x 16).  FP32 levels of 128
  // rows whose width is a multiple of 128 (whole tiles) take 128 x 32 too
  // (13.3 against 17.5 us an iteration at 128^3; with partial tiles, 192^3,
  // 64 x 8 stays faster: 26.7 against 31.4 us).  Otherwise 64 x 8, whose
  // smaller blocks keep more CUs busy, but for FP64 levels where 64 x 32
  // tiles make exactly one wave of blocks and their rows are three quarters
  // full or more: solves at 128^3 2.41 against 2.46 ms, 512 x 32 x 256 2.52
  // against 2.61, 64 x 48 x 1024 2.91 against 2.95, 96 x 240 x 96 3.20
  // against 3.34.  Outside that 64 x 8 is the faster: 144^3 4.23 against
  // 4.86, 160^3 3.72 against 4.05, 192^3 4.38 against 4.69; 1024 x 16 x 128,
  // whose rows fill half of a tile, 1.92 against 1.97.
  static bool big_level(const DevLevel<T>& d) {
    if (d.ny >= 256 || (sizeof(T) == 4 && d.ny >= 128 && d.nx % 128 == 0)) return true;
    const long gy = (d.ny + 31) / 32;
    return sizeof(T) == 8 && 4L * d.ny >= 3 * 32 * gy &&
           one_wave(d, (long)((d.nx + FTX - 1) / FTX) * gy, fused_resident<FTX, 32, 1>());
  }
  static int default_tx(const DevLevel<T>& d) { return (sizeof(T) == 4 && big_level(d)) ? FTX : 64; }
  static int default_ty(const DevLevel<T>& d) { return big_level(d) ? 32 : 8; }
  int tx_used(const DevLevel<T>& d) const {
    if (sizeof(T) == 8) return 64;
    return tile_x ? (tile_x == 64 ? 64 : FTX) : default_tx(d);
  }
  int ty_used(const DevLevel<T>& d) const { return tile_y ? tile_y : default_ty(d); }

  // One fused red+black iteration x -> x2, then swap.  mode 0 plain, 1 zero
  // start (x taken as 0), 2 (FP64) plain with the partial sums of
  // (b - A x)^2 of the x it starts from written to partial[0 .. fused_blocks);
  // FP64 on the caller's arrays (set_caller): 3 as 2 with x and b read from
  // them and b stored into d.b, 4 as 0 with x also stored into the caller's sol.
  // prefetch: planes of look-ahead of the global loads.
  int prefetch = 1;
  // A tile or a look-ahead that is set asks for the kernel that has them:
  // every level then runs one iteration a launch (k_rb_fused).  (FP64 tiles
  // are 64 wide whatever tile_x says.)
  bool single() const { return tile_y > 0 || prefetch == 2 || (sizeof(T) == 4 && tile_x > 0); }
  // the caller's padded (0:nx+1, 0:ny+1, 0:nz+1) arrays on level d, for modes 3 and 4
  void set_caller(const DevLevel<T>& d, T* sol, const T* rhs) {
    caller_lvl = d.L();
    caller_lvl.px = d.nx + 2;
    caller_lvl.pxy = (long)(d.nx + 2) * (d.ny + 2);
    const long o = 1 + caller_lvl.px + caller_lvl.pxy;
    caller_sol = sol + o;
    caller_x = sol + o;
    caller_b = rhs + o;
  }

  // measurement hook: plain launches on the timer's level are bracketed by
  // events: those of the one kernel smoother_name names, nothing else
  KernelTimer* timer = nullptr;
  int timed_nit = 1;             // iterations of such a launch
  void timer_begin(const DevLevel<T>& d, int mode, bool& timed) {
    timed = timer && timer->wants(&d, mode);
    if (timed) hipEventRecord(timer->ev[timer->used], s);
  }
  void timer_end(bool timed, int count = 1) {
    if (!timed) return;
    hipEventRecord(timer->ev[timer->used + 1], s);
    timer->count[timer->used / 2] = count;
    timer->used += 2;
  }
  // A plain iteration that follows an upward launch on the same level
  // marches down, so that it first reads the planes the previous launch
  // touched last; every other fused launch marches up.
  bool alternate = true;
  bool next_down(DevLevel<T>& d, int mode) {
    const bool down = alternate && mode == 0 && d.fused_up && (ty_used(d) == 32 || prefetch == 1);
    d.fused_up = !down;
    return down;
  }
  void fused_iter(DevLevel<T>& d, T omega, int mode, double* partial = nullptr) {
    int ty = ty_used(d);
    const bool down = next_down(d, mode);
    bool timed;
    timer_begin(d, timed_nit == 1 && !(timer && blocks(d)) ? mode : 1, timed);
    if (sizeof(T) == 4 && tx_used(d) == 64) fused_tx<64>(d, omega, mode, ty, partial, down);
    else fused_tx<FTX>(d, omega, mode, ty, partial, down);
    timer_end(timed);
    std::swap(d.x, d.x2);
  }
  // one fused iteration (mode 0) from d.x into out; no swap
  void fused_iter_into(DevLevel<T>& d, T omega, T* out) {
    fused_out = out;
    int ty = ty_used(d);
    const bool down = next_down(d, 0);
    bool timed;
    timer_begin(d, timed_nit == 1 && !(timer && blocks(d)) ? 0 : 1, timed);
    if (sizeof(T) == 4 && tx_used(d) == 64) fused_tx<64>(d, omega, 0, ty, nullptr, down);
    else fused_tx<FTX>(d, omega, 0, ty, nullptr, down);
    timer_end(timed);
    fused_out = nullptr;
  }
  // Tiles of one axis: the fewest that cover n cells when a tile holds `span`
  // cells, ring included (none at the domain's faces); the cells each
  // stores come out even, the first of every tile odd.
  static void sweep_axis(int n, int span, int ring, int& tiles, int& use) {
    auto even = [](int v) { return (v + 1) / 2 * 2; };
    if (n <= span) {
      tiles = 1;
      use = even(n);
      return;
    }
    tiles = 2;
    while (even((n + tiles - 1) / tiles) > span - (tiles > 2 ? 2 * ring : ring)) tiles++;
    use = even((n + tiles - 1) / tiles);
    tiles = (n + use - 1) / use;
  }

  static int cu_count() {
    static std::mutex mu;
    static std::map<int, int> cache;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find(dev);
    if (it != cache.end()) return it->second;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) cus = 256;
    return cache[dev] = cus;
  }

  // One block of the sweep kernels runs per CU.  A chunk of kc planes takes
  // kc + 2 ring + 1 plane steps, in groups of NS; of the chunk sizes with the
  // fewest groups over all waves of blocks the smallest is taken (more than
  // four waves of blocks never pay: every chunk adds its ring).
  // *share: the level's cells over the cells of all block steps.
  template <typename S>
  static SweepGrid sweep_grid(const DevLevel<T>& d, double* share = nullptr) {
    SweepGrid G;
    sweep_axis(d.nx, SW_COLS, S::RINGX, G.gx, G.uw);
    sweep_axis(d.ny, S::ROWS, S::RING, G.gy, G.uh);
    const long tiles = (long)G.gx * G.gy, cus = cu_count();
    long best = -1;
    G.kchunk = 2;
    for (long nch = 1; nch <= std::max(1L, 4 * cus / tiles); nch++) {
      const long kc = (d.nz + 2 * nch - 1) / (2 * nch) * 2;
      const long waves = (tiles * ((d.nz + kc - 1) / kc) + cus - 1) / cus;
      const long cost = waves * ((kc + 2 * S::RING + S::NS) / S::NS);
      if (best < 0 || cost <= best) {
        best = cost;
        G.kchunk = (int)kc;
      }
    }
    G.nch = (d.nz + G.kchunk - 1) / G.kchunk;
    if (share) *share = (double)d.cells() / ((double)best * S::NS * cus * SW_COLS * S::ROWS);
    return G;
  }

  // Whether two iterations on level d run in one pass (k_sweep) rather than
  // in two (k_rb_fused): from 4 M cells on, and where a fair share of the
  // work is on cells of the level (thin levels leave the 128-column tiles or
  // the chunks mostly ring).  Solves, both ways:
  // FP64 128^3 (share 0.11) 3.29 against 3.13 ms, 160^3 (0.16) 4.99 against
  // 5.10, 192^3 5.08 against 5.35, 320^3 13.5 against 15.4, 512^3 39.1
  // against 42.8; mixed 128^3 (0.11) 1.55 against 1.57, 160^3 1.97 against
  // 2.21, 256^3 3.22 against 3.78, 384^3 6.49 against 9.89, 512^3 13.1 against
  // 17.5.  Between 2.5 M and 4 M cells mixed solves would gain (160 x 160 x
  // 128 1.39 against 1.59 ms), FP64 ones a little (2.77 against 2.85).
  // With z stretched no plane has kept divisors (zlo, zhi): a launch takes
  // 0.99 ms in FP64 and 0.55 in FP32 at 512^3, against 1.1 and 0.55 for the
  // two it replaces; solves before and after the sweeps FP64 256^3 7.72 and
  // 7.22, 320^3 16.7 and 13.4, 512^3 42.9 and 41.3; mixed 256^3 3.63 and 3.26,
  // 512^3 17.6 and 16.7.  (A plane's row offsets are 32-bit bytes.)
  bool sweeps(const DevLevel<T>& d) const {
    if (single() || d.cells() < 4000000L || d.pxy * (long)sizeof(T) > 0x7fffffffL) return false;
    double share = 0.0;
    sweep_grid<SweepShape<T, SW_WAVES, 2, SW_X>>(d, &share);
    return share >= 0.15;
  }

  // arguments of a k_sweep launch (x -> x2) but for its grid; c: the coarser
  // level of SW_PROLONG, or null
  static SweepArgs<T> sweep_args(const DevLevel<T>& d, const DevLevel<T>* c, T omega) {
    SweepArgs<T> A;
    std::memset(&A, 0, sizeof A);
    A.xo = d.x2;
    A.xi = d.x;
    A.b = d.b;
    A.L = d.L();
    A.omega = omega;
    A.zlo = d.zlo;
    A.zhi = d.zhi;
    A.c5u = d.c5u;
    A.c6u = d.c6u;
    if (c) {
      A.xc = c->x;
      A.C = c->L();
      A.W = d.PW();
    }
    return A;
  }

  // NIT red/black iterations on level d in one pass, x -> x2, then swap.
  // PRE: from x, from 0, or from x + P x_c (c the next coarser level, every
  // axis halving).  to_caller (FP64): the caller's solution also receives x.
  template <int NIT, int PRE>
  void sweep(DevLevel<T>& d, const DevLevel<T>* c, T omega, bool to_caller = false) {
    using S = SweepShape<T, SW_WAVES, NIT, PRE>;
    SweepArgs<T> A = sweep_args(d, c, omega);
    if (to_caller) {
      A.ext = caller_sol;
      A.U = caller_lvl;
    }
    A.G = sweep_grid<S>(d);
    const unsigned nb = (unsigned)((A.G.gx * A.G.gy * A.G.nch + 7) / 8 * 8);
    bool timed;
    timer_begin(d, PRE == SW_X && !to_caller && timed_nit == NIT ? 0 : 1, timed);
    set_dynamic_lds((const void*)k_sweep<T, SW_WAVES, NIT, PRE>, S::LDS * sizeof(T));   // a failure surfaces at the solve's end
    hipLaunchKernelGGL((k_sweep<T, SW_WAVES, NIT, PRE>), dim3(nb), dim3(S::THREADS), S::LDS * sizeof(T), s, A);
    timer_end(timed, NIT);
    d.fused_up = true;
    std::swap(d.x, d.x2);
  }

  // Whether iterations on level d run by blocks of the level in LDS (k_block),
  // where the launches they save outweigh the rings.  Solves against one
  // launch per iteration: FP64 16^3 0.80 against 0.93 ms, 64^3 1.20 against
  // 1.24, 96 x 64 x 80 1.51 against 1.59; mixed 32^3 0.59 against 0.70 ms,
  // 64^3 0.73 against 0.81, 96^3 0.95 against 1.05, 144 x 128 x 128 1.84
  // against 1.98, 144 x 144 x 128 2.02 against 2.03.
  // FP32: up to 3 M cells.  (From there to the sweeps' 4 M one launch per
  // iteration: 160 x 144 x 144 2.37 against 2.50 ms by blocks; sweeps would
  // take 2.17, and 144^3, 2.28 by blocks, 2.02.)
  // FP64: while the large blocks, one to a CU, all run at once.  A second
  // wave of them costs what single iterations do and more: 64 x 64 x 128 (256
  // blocks) 1.49 against 1.55 ms, 80^3 (300) 1.74 against 1.68, 128 x 64 x 96
  // (384) 1.55 against 1.42, 64 x 128 x 128 (512) 1.63 against 1.56, 112 x 96
  // x 96 (576) 2.47 against 2.32.  Only where that wave is four fifths full
  // and the rows fill three quarters of the single iterations' tiles or less
  // do blocks gain: 96^3 (432) 1.63 against 1.66, 96 x 96 x 112 (504) 2.14
  // against 2.19, but 96 x 96 x 80 (360) 1.88 against 1.83.
  // A batch's launch takes its items' blocks together: there by their cells.
  static bool blocks(long cells) { return cells <= (sizeof(T) == 8 ? 1200000L : 3000000L); }
  bool blocks(const DevLevel<T>& d) const {
    if (single()) return false;
    if (sizeof(T) == 4 || d.cells() <= LARGE_BLOCK) return blocks(d.cells());
    const long n = block_count<BlockLarge>(d), cus = cu_count();
    return n <= cus || (n <= 2 * cus && 5 * n >= 4 * 2 * cus && 4L * d.nx <= 3L * ((d.nx + FTX - 1) / FTX) * FTX);
  }
  // 32 x 8 x 8 blocks of 1024 threads from 300000 cells on in FP64 and 150000
  // in FP32: less ring per cell (96^3 FP64 2.14 against 2.38 ms); below,
  // 16 x 8 x 4 keeps more CUs busy (64^3 FP64 1.56 against 1.69 ms when its
  // fine level, too, takes them)
  static constexpr long LARGE_BLOCK = sizeof(T) == 8 ? 300000 : 150000;
  static bool large_block(long cells) { return cells > LARGE_BLOCK; }
  // FP32 from 400000 cells on: 32 x 16 x 8, where a cell's share of the ring
  // shrinks further (mixed 80^3 0.972 against 0.945 ms, 96^3 1.020 against
  // 0.977, 128^3 1.39 against 1.32, 256^3, on its 128^3 level, 3.12 against
  // 3.03; also on 64^3 levels 128^3 takes 1.37).  64 x 8 x 8 and 32 x 16 x 16
  // are slower (128^3 1.31 and 1.53 when this one took 1.29), and in FP64 no
  // other shape gains.
  static constexpr long TALL_BLOCK = 400000;
  static bool tall_block(long cells) { return sizeof(T) == 4 && cells > TALL_BLOCK; }
  // The prolongation in the launch works on the whole ring: it pays up to
  // 200000 cells (96^3 FP64 2.11 ms with it on the fine level, 2.00 without;
  // mixed 128^3 1.45 and 1.36).
  static constexpr long PROLONG_BLOCK = 200000;
  static bool prolong_in_block(long cells) { return cells <= PROLONG_BLOCK; }
  // whether blocks of this shape start from PRE on some level
  static constexpr bool block_shape(BlockSmall, int) { return true; }
  static constexpr bool block_shape(BlockLarge, int pre) { return pre != SW_PROLONG || LARGE_BLOCK < PROLONG_BLOCK; }
  static constexpr bool block_shape(BlockTall, int pre) {
    return sizeof(T) == 4 && (pre != SW_PROLONG || TALL_BLOCK < PROLONG_BLOCK);
  }

  // arguments of a k_block launch (x -> x2) with blocks B, and their number;
  // c as for sweep_args
  template <typename B>
  static BlockArgs<T> block_args(const DevLevel<T>& d, const DevLevel<T>* c, T omega) {
    BlockArgs<T> A;
    std::memset(&A, 0, sizeof A);
    A.xo = d.x2;
    A.xi = d.x;
    A.b = d.b;
    A.L = d.L();
    A.omega = omega;
    if (c) {
      A.xc = c->x;
      A.C = c->L();
      A.W = d.PW();
    }
    A.gx = (d.nx + B::BX - 1) / B::BX;
    A.gy = (d.ny + B::BY - 1) / B::BY;
    return A;
  }
  template <typename B>
  static int block_count(const DevLevel<T>& d) {
    return (d.nx + B::BX - 1) / B::BX * ((d.ny + B::BY - 1) / B::BY) * ((d.nz + B::BZ - 1) / B::BZ);
  }

  // NIT iterations on level d by blocks, x -> x2, then swap (PRE, c,
  // to_caller as for sweep).  NORM (FP64, from x): the blocks' partial sums of
  // |b - A x_in|^2 go to partial; returns their number.
  template <typename B, int NIT, int PRE, bool NORM = false, bool REST = false>
  int block_launch(DevLevel<T>& d, const DevLevel<T>* c, T omega, bool to_caller, double* partial) {
    using S = BlockShape<T, B, NIT, PRE, REST>;
    BlockArgs<T> A = block_args<B>(d, c, omega);
    if (REST) {
      A.bc = c->b;
      A.RW = d.RW();
    }
    if (to_caller) {
      A.ext = caller_sol;
      A.U = caller_lvl;
    }
    A.partial = partial;
    const int nb = block_count<B>(d);
    bool timed;
    timer_begin(d, PRE == SW_X && !NORM && !REST && timed_nit == NIT ? 0 : 1, timed);
    if (S::LDS * sizeof(T) > 65536)
      set_dynamic_lds((const void*)k_block<T, B, NIT, PRE, NORM, REST>, S::LDS * sizeof(T));
    hipLaunchKernelGGL((k_block<T, B, NIT, PRE, NORM, REST>), dim3((unsigned)nb), dim3(B::NT), S::LDS * sizeof(T), s, A);
    timer_end(timed, NIT);
    d.fused_up = true;
    std::swap(d.x, d.x2);
    return nb;
  }
  template <int NIT, int PRE, bool NORM = false>
  int block(DevLevel<T>& d, const DevLevel<T>* c, T omega, bool to_caller = false, double* partial = nullptr) {
    if constexpr (block_shape(BlockTall(), PRE) && !NORM)
      if (tall_block(d.cells())) return block_launch<BlockTall, NIT, PRE, NORM>(d, c, omega, to_caller, partial);
    if constexpr (block_shape(BlockLarge(), PRE))
      if (large_block(d.cells())) return block_launch<BlockLarge, NIT, PRE, NORM>(d, c, omega, to_caller, partial);
    return block_launch<BlockSmall, NIT, PRE, NORM>(d, c, omega, to_caller, partial);
  }

  // the same, then the residual restricted into c's b
  template <int NIT, int PRE>
  void block_restrict(DevLevel<T>& d, const DevLevel<T>* c, T omega) {
    if constexpr (sizeof(T) == 4) {
      if (large_block(d.cells())) {
        block_launch<BlockLarge, NIT, PRE, false, true>(d, c, omega, false, nullptr);
        return;
      }
    }
    block_launch<BlockSmall, NIT, PRE, false, true>(d, c, omega, false, nullptr);
  }
  // The residual needs a ring one cell wider (two along x), so joining the
  // restriction pays on smaller levels than the iterations do: up to 150000
  // cells in FP64 and 300000 in FP32.  Solves without it, with it up to 150000
  // and up to 300000 cells: FP64 64^3 1.436, 1.377 and 1.410 ms, 128^3 2.40,
  // 2.36 and 2.41; mixed 48^3 0.598, 0.563 and 0.553, 64^3 0.743, 0.722 and
  // 0.703, 80^3 0.916, 0.853 and 0.872.
  static bool restricts(const DevLevel<T>& d, const DevLevel<T>& c) {
    return d.cells() <= (sizeof(T) == 8 ? 150000L : 300000L) && d.rs[0] == 2 && d.rs[1] == 2 && d.rs[2] == 2 &&
           d.nx == 2 * c.nx && d.ny == 2 * c.ny && d.nz == 2 * c.nz;
  }
  // nu iterations on level d by blocks (zero_start: from 0), the last launch
  // also restricting the residual into rc's b
  void iterate_restrict(DevLevel<T>& d, T omega, int nu, bool zero_start, const DevLevel<T>* rc) {
    int it = 0;
    if (nu > 2) {
      if (zero_start) block<2, SW_ZERO>(d, nullptr, omega);
      else block<2, SW_X>(d, nullptr, omega);
      zero_start = false;
      for (it = 2; it + 2 < nu; it += 2) block<2, SW_X>(d, nullptr, omega);
    }
    const bool two = nu - it == 2;
    if (two && zero_start) block_restrict<2, SW_ZERO>(d, rc, omega);
    else if (two) block_restrict<2, SW_X>(d, rc, omega);
    else if (zero_start) block_restrict<1, SW_ZERO>(d, rc, omega);
    else block_restrict<1, SW_X>(d, rc, omega);
  }

  // iterate on a level of blocks
  void iterate_blocks(DevLevel<T>& d, T omega, int nu, bool zero_start, DevLevel<T>* c, int last_mode) {
    int it = 0;
    auto last = [&](int n) { return it + n == nu && last_mode == 4; };
    if (c && !(d.ps[0] == 2 && d.ps[1] == 2 && d.ps[2] == 2 && prolong_in_block(d.cells()))) {
      prolong_add(d, *c, d.x);
      c = nullptr;
    }
    if (c && nu >= 2) block<2, SW_PROLONG>(d, c, omega, last(2)), it = 2;
    else if (c) block<1, SW_PROLONG>(d, c, omega, last(1)), it = 1;
    else if (zero_start && nu >= 2) block<2, SW_ZERO>(d, nullptr, omega), it = 2;
    else if (zero_start) block<1, SW_ZERO>(d, nullptr, omega), it = 1;
    for (; it + 2 <= nu; it += 2) block<2, SW_X>(d, nullptr, omega, last(2));
    if (it < nu) block<1, SW_X>(d, nullptr, omega, last(1));
  }

  // nu red/black iterations on level d (x -> x): by twos where that is the
  // faster way, one by one otherwise.  zero_start: from x = 0; c: from
  // x + P x_c; last_mode: fused-kernel mode of the last iteration (4: it also
  // stores x into the caller's array).
  void iterate(DevLevel<T>& d, T omega, int nu, bool zero_start = false, DevLevel<T>* c = nullptr,
               int last_mode = 0) {
    if (blocks(d) && nu > 0) {
      iterate_blocks(d, omega, nu, zero_start, c, last_mode);
      return;
    }
    const bool two = nu >= 2 && sweeps(d);
    int it = 0;
    if (c) {
      // FP64 keeps the separate prolongation: with the coarse planes beside
      // the fine ones the kernel needs more than the 256 registers there are
      bool done = false;
      if constexpr (sizeof(T) == 4) {
        if (two && d.ps[0] == 2 && d.ps[1] == 2 && d.ps[2] == 2) {
          sweep<2, SW_PROLONG>(d, c, omega);
          it = 2;
          done = true;
        }
      }
      if (!done) prolong_add(d, *c, d.x);
    } else if (zero_start && two) {
      sweep<2, SW_ZERO>(d, nullptr, omega);
      it = 2;
    }
    for (; two && it + 2 <= nu; it += 2) sweep<2, SW_X>(d, nullptr, omega, it + 2 == nu && last_mode == 4);
    for (; it < nu; it++) fused_iter(d, omega, (it == 0 && zero_start) ? 1 : (it == nu - 1 && last_mode ? last_mode : 0));
  }

  // iterations of a plain launch of nu iterations on level d
  int launch_nit(const DevLevel<T>& d, int nu) const { return nu >= 2 && (blocks(d) || sweeps(d)) ? 2 : 1; }
  // symbol of the plain smoother kernel iterate launches on level d for nu iterations
  void smoother_name(const DevLevel<T>& d, int nu, char* buf, size_t n) const {
    const char* t = sizeof(T) == 8 ? "double" : "float";
    const int nit = launch_nit(d, nu);
    if (blocks(d)) {
      auto name = [&](auto b) {
        using B = decltype(b);
        std::snprintf(buf, n, "k_block<%s, pepsmg::BlockTile<%d, %d, %d, %d>, %d, %d, false, false>", t, B::BX, B::BY,
                      B::BZ, B::NT, nit, (int)SW_X);
      };
      if (tall_block(d.cells())) name(BlockTall());
      else if (large_block(d.cells())) name(BlockLarge());
      else name(BlockSmall());
      return;
    }
    if (nit == 2) {
      std::snprintf(buf, n, "k_sweep<%s, %d, 2, %d>", t, SW_WAVES, (int)SW_X);
      return;
    }
    const int ty = ty_used(d);
    std::snprintf(buf, n, "k_rb_fused<%s, %d, %d, 0, %d>", sizeof(T) == 8 ? "double" : "float", tx_used(d), ty,
                  ty == 32 ? 1 : prefetch);   // 32-row tiles load one plane ahead
  }

  void smooth_colour(DevLevel<T>& d, const T* b, T* x, T omega, int colour, bool zero) {
    int hx = (d.nx + 1) / 2;
    dim3 g = grid3(hx, d.ny, d.nz, 64, 4), blk(64, 4, 1);
    if (zero)
      hipLaunchKernelGGL((k_rb_colour<T, true>), g, blk, 0, s, x, b, d.L(), omega, colour);
    else
      hipLaunchKernelGGL((k_rb_colour<T, false>), g, blk, 0, s, x, b, d.L(), omega, colour);
  }

  // nu red/black iterations on (x, b); zero_start: x is taken as 0 on entry
  void rbgs(DevLevel<T>& d, T* x, const T* b, int nu, T omega, bool zero_start) {
    if (nu <= 0) {
      if (zero_start) hipMemsetAsync(x, 0, d.ncell * sizeof(T), s);
      return;
    }
    for (int it = 0; it < nu; it++) {
      smooth_colour(d, b, x, omega, 0, zero_start && it == 0);
      smooth_colour(d, b, x, omega, 1, false);
    }
  }

  void residual(DevLevel<T>& d, T* r, const T* x, const T* b) {
    hipLaunchKernelGGL((k_residual<T>), grid3(d.nx, d.ny, d.nz, 64, 4), dim3(64, 4, 1), 0, s, r, x, b, d.L());
  }

  void apply(DevLevel<T>& d, T* y, const T* x) {
    hipLaunchKernelGGL((k_apply<T>), grid3(d.nx, d.ny, d.nz, 64, 4), dim3(64, 4, 1), 0, s, y, x, d.L());
  }

  // tile width of the restriction and prolongation z-march kernels: 64 cells
  // in FP64; in FP32 128 (512-byte rows either way) on levels where that
  // still leaves z-chunks of 8 or more planes (512^3: 20.8 against 21.0 ms
  // for the mixed solve), 64 below (shorter chunks re-read more halo planes)
  static constexpr int MTX = sizeof(T) == 8 ? 64 : 128;

  // z-march decomposition: TX x TY tiles, about 2048 blocks, chunk count a
  // multiple of 8 when >= 8; even chunks for the restriction kernel.
  static MarchGrid march_grid(const DevLevel<T>& d, int TY, bool even, int TX = 64) {
    MarchGrid G;
    G.gx = (d.nx + TX - 1) / TX;
    G.gy = (d.ny + TY - 1) / TY;
    long nxy = (long)G.gx * G.gy;
    long nch = std::max(1L, std::min<long>((2048 + nxy - 1) / nxy, (d.nz + 3) / 4));
    if (nch < 8 && d.nz >= 64) nch = 8;
    if (nch >= 8) nch = (nch + 7) / 8 * 8;
    int kc = (int)((d.nz + nch - 1) / nch);
    if (even && (kc & 1)) kc++;
    G.kchunk = kc;
    G.nch = (d.nz + kc - 1) / kc;
    return G;
  }

  void residual_restrict(DevLevel<T>& f, DevLevel<T>& c, const T* x, const T* b) {
    if (f.rs[0] == 2 && f.rs[1] == 2 && f.rs[2] == 2) {
      MarchGrid G = march_grid(f, 16, true, MTX);
      if (MTX == 64 || G.kchunk < 8) {
        G = march_grid(f, 16, true, 64);
          hipLaunchKernelGGL((k_restrict_march<T, 64>), dim3((unsigned)(G.gx * G.gy * G.nch)),
                           dim3(march_threads<64>()), 0, s, c.b, x, b, f.L(), c.L(), f.RW(), G);
      } else {
        hipLaunchKernelGGL((k_restrict_march<T, MTX>), dim3((unsigned)(G.gx * G.gy * G.nch)),
                           dim3(march_threads<MTX>()), 0, s, c.b, x, b, f.L(), c.L(), f.RW(), G);
      }
      return;
    }
    hipLaunchKernelGGL((k_restrict<T, true>), grid3(c.nx, c.ny, c.nz, 64, 4), dim3(64, 4, 1), 0, s, c.b, x, b,
                       f.L(), c.L(), f.RW());
  }

  // |b - A x|^2 into out[0] (partial sums per block, then one block); r
  // stored when non-null.
  void resid_norm_march(DevLevel<T>& d, const T* x, const T* b, T* r, double* partial, double* out) {
    MarchGrid G = march_grid(d, RESID_TY, false);
    int nb = G.gx * G.gy * G.nch;
    if (nb > PARTIAL_CAP) {
      resid_norm(d, x, b, r, partial, out);
      return;
    }
    if (r)
      hipLaunchKernelGGL((k_resid_march<T, RESID_TY, 1>), dim3((unsigned)nb), dim3(MARCH_THREADS), 0, s, x,
                         (const float*)nullptr, b, r, (float*)nullptr, (T*)nullptr, d.L(), G, partial);
    else
      hipLaunchKernelGGL((k_resid_march<T, RESID_TY, 0>), dim3((unsigned)nb), dim3(MARCH_THREADS), 0, s, x,
                         (const float*)nullptr, b, (T*)nullptr, (float*)nullptr, (T*)nullptr, d.L(), G, partial);
    hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(RED_THREADS), 0, s, partial, nb, out);
  }

  // prolongation march: TX x 16 fine tiles, chunks of coarse planes
  static MarchGrid prolong_grid(const DevLevel<T>& f, const DevLevel<T>& c, int TX = 64) {
    MarchGrid G;
    G.gx = (f.nx + TX - 1) / TX;
    G.gy = (f.ny + 15) / 16;
    long nxy = (long)G.gx * G.gy;
    long nch = std::max(1L, std::min<long>((2048 + nxy - 1) / nxy, (c.nz + 1) / 2));
    if (nch >= 8) nch = (nch + 7) / 8 * 8;
    G.kchunk = (int)((c.nz + nch - 1) / nch);
    G.nch = (c.nz + G.kchunk - 1) / G.kchunk;
    return G;
  }

  void prolong_add(DevLevel<T>& f, DevLevel<T>& c, T* xf) {
    if (f.ps[0] == 2 && f.ps[1] == 2 && f.ps[2] == 2) {
      MarchGrid G = prolong_grid(f, c, MTX);
      if (MTX == 64 || 2 * G.kchunk < 8) {   // chunks count coarse planes
        G = prolong_grid(f, c, 64);
          hipLaunchKernelGGL((k_prolong_march<T, 64>), dim3((unsigned)(G.gx * G.gy * G.nch)),
                           dim3(march_threads<64>()), 0, s, xf, c.x, f.L(), c.L(), f.PW(), G);
      } else {
        hipLaunchKernelGGL((k_prolong_march<T, MTX>), dim3((unsigned)(G.gx * G.gy * G.nch)),
                           dim3(march_threads<MTX>()), 0, s, xf, c.x, f.L(), c.L(), f.PW(), G);
      }
      return;
    }
    hipLaunchKernelGGL((k_prolong_add<T>), grid3(f.nx, f.ny, f.nz, 64, 4), dim3(64, 4, 1), 0, s, xf, c.x, f.L(),
                       c.L(), f.PW());
  }

  int red_blocks(const DevLevel<T>& d) {
    long n = d.cells();
    long b = (n + RED_THREADS - 1) / RED_THREADS;
    return (int)std::max(1L, std::min<long>(b, RED_BLOCKS));
  }

  // out[0] = sum x*y over the interior
  void dot(DevLevel<T>& d, const T* x, const T* y, double* partial, double* out) {
    int nb = red_blocks(d);
    hipLaunchKernelGGL((k_dot_partial<T, 0, false>), dim3(nb), dim3(RED_THREADS), 0, s, x, y, d.L(), partial,
                       (T*)nullptr);
    hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(RED_THREADS), 0, s, partial, nb, out);
  }

  // out[0] = |b - A x|^2; optionally r = b - A x
  void resid_norm(DevLevel<T>& d, const T* x, const T* b, T* r, double* partial, double* out) {
    int nb = red_blocks(d);
    if (r)
      hipLaunchKernelGGL((k_dot_partial<T, 1, true>), dim3(nb), dim3(RED_THREADS), 0, s, x, b, d.L(), partial, r);
    else
      hipLaunchKernelGGL((k_dot_partial<T, 1, false>), dim3(nb), dim3(RED_THREADS), 0, s, x, b, d.L(), partial,
                         (T*)nullptr);
    hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(RED_THREADS), 0, s, partial, nb, out);
  }
};


// Arguments of the persistent coarse kernel for levels s..L of hierarchy h:
// compact LDS layout of every level's x and b (16-byte aligned), the
// coarsest level in FP64.  Returns false if it does not fit in LDS.
template <typename T>
inline bool pc_build(int L, Hier<double>& h64, size_t lds_max, Hier<T>& h, int s, int nu, int nu_post, T omega,
                     double tol,
                     int* slot, PCArgs<T>& A, size_t& lds) {
  int nlev = L - s + 1;
  if (s < 1 || nlev > PC_MAXLEV) return false;
  std::memset(&A, 0, sizeof A);
  A.nlev = nlev;
  A.nu = nu;
  A.nu_post = nu_post;
  A.omega = omega;
  A.tol = tol;
  A.maxit = 1000;
  A.iters_slot = slot;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    size_t o = off;
    off = (off + bytes + 15) / 16 * 16;
    return o;
  };
  for (int q = 0; q < nlev; q++) {
    DevLevel<T>& d = h.lv[s + q];
    Lvl<T> l = d.L();
    l.px = d.nx;
    l.pxy = (long)d.nx * d.ny;
    A.lv[q] = l;
    if (q < nlev - 1) {
      size_t n = (size_t)d.cells();
      A.xoff[q] = (int)(take((n + 2) * sizeof(T)) / sizeof(T));   // two zeros behind it (pc_smooth_pairs)
      A.boff[q] = (int)(take(n * sizeof(T)) / sizeof(T));
      A.coff[q] = (int)(take((size_t)pc_stage_elems(d.nx, d.ny, d.nz, true) * sizeof(T)) / sizeof(T));
      A.rw[q] = d.RW();
      A.pw[q] = d.PW();
    }
  }
  if (nlev > 1) A.roff = (int)(take((size_t)h.lv[s].cells() * sizeof(T)) / sizeof(T));
  DevLevel<double>& cd = h64.lv[L];
  Lvl<double> lc = cd.L();
  lc.px = cd.nx;
  lc.pxy = (long)cd.nx * cd.ny;
  A.lc = lc;
  size_t nc = (size_t)cd.cells();
  // x slots of pc_coarsest_small / pc_coarsest_block
  A.xslots = nc > 64 && nc <= (size_t)PC_THREADS;
  A.xcoff = (int)(take((nc <= 64 ? (size_t)PC_SMALL_X : A.xslots ? 2 * (nc + 1) : nc) * 8) / 8);
  A.bcoff = (int)(take(nc * 8) / 8);
  A.xctoff = (int)(take(nc * sizeof(T)) / sizeof(T));
  A.ccoff = (int)(take((size_t)pc_stage_elems(cd.nx, cd.ny, cd.nz, false) * 8) / 8);
  A.gl = h.lv[s].L();
  A.gxs = h.lv[s].x;
  A.gbs = h.lv[s].b;
  lds = off;
  return off <= lds_max;
}

}  // namespace pepsmg
