// Stage kernel of small grids: the same stage as stage_kernel.hpp, bit for bit,
// laid out for the time of one workgroup instead of the throughput of many.
//
// On a grid whose tiles do not fill the GPU a stage takes as long as one
// workgroup's chain of work, and with one thread per edge and per cell that chain
// is long code run once: each of its instructions is fetched cold (a launch starts
// with an empty instruction cache) and issued by one or two waves per SIMD.  Here
// every phase is cut into its smallest items, dealt to 4 threads per cell: the
// states of one variable at one edge, the flux of one edge, the update of one
// variable of one cell.  A thread runs a quarter of the code for the states and
// the update, all four SIMDs share it, and what the later phases load is asked for
// at the start.  An 8 x 8 tile keeps a phase near one round of the 256 threads.
// A stage of a 64 x 61 grid, FP64 (launch included, of which 1.7 us is the least
// a launch takes): SLAU + van Leer 12.3 -> 7.1 us, HLLC + MLP5 17.3 -> 8.3 us (7.8
// and 9.8 us with 16 x 8 tiles); FP32 flux 8.9 -> 5.0 and 11.8 -> 5.7 us.  What is
// left is the chain itself, FP64: loads 0.9 us, states 0.5 to 1, flux 1, update and
// primitives 1.3.
#pragma once

#include "stage_kernel.hpp"

namespace cato {

// FP64: the edges as items.
template <int FLUX, int LIMC, typename R, int TX, int TY, int NT> struct LatencySmem {
  static constexpr int H = halo_of<LIMC>();
  static constexpr int RX = TX + 2 * H, RY = TY + 2 * H;
  static constexpr int NIE = (TX + 1) * TY, NE = NIE + TX * (TY + 1);  // i-edges first
  static constexpr int kSets = needs_superbee_states<FLUX>() ? 2 : 1;
  union {
    R sp[4][RY][RX];          // primitives with halo
    double nv[4][TX * TY];    // after the edges: the new state
  };
  R lr[kSets][4][2][NE];      // edge states L, R by variable; the flux takes the place of L
  __device__ R flux_i(int v, int ex, int ey) const { return lr[0][v][0][ey * (TX + 1) + ex]; }
  __device__ R flux_j(int v, int ex, int ey) const { return lr[0][v][0][NIE + ey * TX + ex]; }
};
// Precision form: the edges by the one loop of stage_kernel.hpp (edge_pass), a
// thread to an edge.  Cut into items, the same formulas had their products fused
// into other FMAs, so that a small grid would have rounded unlike the same grid in
// a batch or on an explicit tile.
template <int FLUX, int LIMC, int TX, int TY, int NT>
struct LatencySmem<FLUX, LIMC, f32x, TX, TY, NT> : TileSmem<LIMC, f32x, TX, TY, NT, false> {
  double nv[4][TX * TY];
  __device__ f32x flux_i(int v, int ex, int ey) const { return this->sfi[v][ey][ex]; }
  __device__ f32x flux_j(int v, int ex, int ey) const { return this->sfj[v][ey][ex]; }
};

// Cell left of edge e (0-based tile edge index), in global cells; false outside the domain.
template <int TX, int TY, class Args>
__device__ inline bool latency_edge(Args &a, int i0, int j0, int e, bool &idir, int &ci, int &cj) {
  constexpr int NIE = (TX + 1) * TY;
  idir = e < NIE;
  const int k = idir ? e : e - NIE, w = idir ? TX + 1 : TX;
  const int ey = k / w, ex = k - ey * w;
  ci = idir ? i0 - 1 + ex : i0 + ex;
  cj = idir ? j0 + ey : j0 - 1 + ey;
  return ci <= a.ni && cj <= a.nj;
}

// States, then fluxes, of the tile's edges (phase 2 of stage_kernel.hpp; the
// direction is read at run time, as in its one-loop form).
template <int FLUX, int LIMC, typename R, int TX, int TY, class D, class DF, bool GEOM, int NT, class Args, class Smem>
__device__ inline void latency_edges(Args &a, Smem &sm, int i0, int j0) {
  constexpr int H = Smem::H, RX = Smem::RX, NE = Smem::NE;
  const int tid = threadIdx.x;
  bool idir;
  int ci, cj;
  for (int it = tid; it < 4 * NE; it += NT) {
    const int v = it / NE, e = it - v * NE;
    if (!latency_edge<TX, TY>(a, i0, j0, e, idir, ci, cj)) continue;
    const int sn = idir ? 1 : RX, st = idir ? RX : 1;
    const R *q = &sm.sp[v][cj - (j0 - H)][ci - (i0 - H)];
    R L, Rv;
    recon_var<R, LIMC, D>(q, sn, st, L, Rv);
    sm.lr[0][v][0][e] = L;
    sm.lr[0][v][1][e] = Rv;
    if constexpr (needs_superbee_states<FLUX>()) {
      recon_var<R, LIM_SUPERBEE, D>(q, sn, st, L, Rv);
      sm.lr[1][v][0][e] = L;
      sm.lr[1][v][1][e] = Rv;
    }
  }
  __syncthreads();
  for (int e = tid; e < NE; e += NT) {
    if (!latency_edge<TX, TY>(a, i0, j0, e, idir, ci, cj)) continue;
    auto states = [&](int set) {
      EdgeState<R> s;
      s.rL = sm.lr[set][0][0][e], s.rR = sm.lr[set][0][1][e];
      s.uL = sm.lr[set][1][0][e], s.uR = sm.lr[set][1][1][e];
      s.vL = sm.lr[set][2][0][e], s.vR = sm.lr[set][2][1][e];
      s.pL = sm.lr[set][3][0][e], s.pR = sm.lr[set][3][1][e];
      return s;
    };
    EdgeState<R> s = states(0), sb;
    if constexpr (needs_superbee_states<FLUX>()) sb = states(1);
    const int sn = idir ? 1 : RX, st = idir ? RX : 1;
    PressNbr<R> pn;
    if constexpr (needs_pressure_nbrs<FLUX>()) pn = pressure_nbrs(&sm.sp[3][cj - (j0 - H)][ci - (i0 - H)], sn, st);
    s.ax = idir ? 0 : 1;
    edge_normal<GEOM>(a, idir, ci, cj, s);
    R f[4];
    edge_flux<R, FLUX, 4, DF>(gas_of<R>(a.gamma, a.gas[0], a.gas[1], a.gas[2], a.gas[3]), a.low_mach_fix, s, pn, f, &sb);
#pragma unroll
    for (int v = 0; v < 4; ++v) sm.lr[0][v][0][e] = f[v];
  }
  __syncthreads();
}

template <int FLUX, int LIMC, typename R, int TX, int TY, bool GEOM = false>
__global__ __launch_bounds__(4 * TX * TY) void latency_kernel(StageArgs a) {
  constexpr int NC = TX * TY, NT = 4 * NC, NW = NT / 64;
  static_assert(NC % 64 == 0, "a wave updates one variable");
  constexpr bool kExact = !std::is_same<R, f32x>::value;
  using Smem = LatencySmem<FLUX, LIMC, R, TX, TY, NT>;
  __shared__ Smem sm;
  __shared__ RedSmemT<NW> red;
  const int tid = threadIdx.x, tile = xcd_tile(blockIdx.x, gridDim.x);
  const int tx = tile % a.tiles_x, ty = tile / a.tiles_x;
  const int i0 = tx * TX + 1, j0 = ty * TY + 1;

  // ---- 0. what later phases need is asked for now: the loop state, the partials
  // of the step this one closes (StageArgs::fold_n), the geometry and the state of
  // the thread's cell
  constexpr int kLoopWords = sizeof(LoopState) / sizeof(double);
  __shared__ double loop_words[kLoopWords];
  double loop_word = 0.0;
  if (a.loop && tid < kLoopWords) loop_word = global(reinterpret_cast<const double *>(a.loop))[tid];
  double fold_m = __builtin_inf();
  int fold_e = 0;
  for (int k = tid; k < a.fold_n; k += NT) {
    const double x = global(a.fold_min)[k];
    fold_m = (x < fold_m) ? x : fold_m;
    fold_e |= global(a.fold_err)[k];
  }
  const int v = tid / NC, c = tid - v * NC, cy = c / TX, cx = c - cy * TX;
  const int gi = i0 + cx, gj = j0 + cy;
  const bool cell = gi <= a.ni && gj <= a.nj;
  const size_t fs = (size_t)a.fstride, off = (size_t)(gj - 1) * a.pitch + (size_t)(gi - 1);
  const bool conv = a.last_stage && a.conv_first[0] != nullptr;
  double u0 = 0.0, uk = 0.0, src = 0.0, fst = 0.0;
  CellGeo g{};
  if (cell) {
    if (a.mode == MODE_COMBINE || a.mode == MODE_BASE) u0 = global(a.u0[0])[off + v * fs];
    if (a.mode == MODE_FIRST || a.mode == MODE_COMBINE) uk = global(a.uk[0])[off + v * fs];
    if (v == 3 && a.src_E) src = global(a.src_E)[off];
    if (conv) fst = global(a.conv_first[0])[off + v * fs];
    g = cell_geometry<kExact, GEOM>(a, gi, gj);
  }

  // ---- 1. primitives of the tile + halo
  int err = 0;
  const bool in_range = load_tile<FLUX, LIMC, R, TX, TY, NT, false>(a, i0, j0, sm.sp, err);
  // The FastOps flux of the SLAU family and HLLC only: AUSM+, AUSMPW+ and Roe divide
  // as IEEE does here.  Their FastOps forms shorten no chain (Sod 400 x 4 with AUSM+ 2 %
  // slower) and take Roe from 115 to 159 registers, three workgroups a CU instead of
  // four (301 x 243, rk(2,4), superbee, in this layout: 6.39 -> 6.65 ms a pass).
  constexpr bool kFastFlux = slau_family<FLUX>() || FLUX == FLUX_HLLC;
  constexpr bool kFastScheme = kExact && (kFastFlux || LIMC == LIM_MLP3 || LIMC == LIM_MLP5);
  if constexpr (kFastScheme) {
    const int vote = __all(in_range ? 1 : 0);
    if ((tid & 63) == 0) red.fast[tid >> 6] = vote;
  }
  if (tid < kLoopWords) loop_words[tid] = loop_word;
  if (a.fold_n) {
    const double m = wave_min(fold_m);
    const int e = wave_or(fold_e);
    if ((tid & 63) == 0) {
      red.m[tid >> 6] = m;
      red.e[tid >> 6] = e;
    }
  }
  __syncthreads();
  double dt = a.dt_value;
  if (a.loop) {
    const LoopState &now = *reinterpret_cast<const LoopState *>(loop_words);
    if (a.loop_out) {
      LoopState ls = now;
      if (a.fold_n && !ls.done) {
        double m = red.m[0];
        int e = red.e[0];
#pragma unroll
        for (int k = 1; k < NW; ++k) {
          m = (red.m[k] < m) ? red.m[k] : m;
          e |= red.e[k];
        }
        loop_update(&ls, m, e, 2);
      }
      if (tile == 0 && tid == 0) *a.loop_out = ls;
      if (ls.done) return;
      dt = ls.dt;
    } else {
      if (now.done) return;
      dt = now.dt;
    }
  }

  // ---- 2. edge states, 3. edge fluxes
  if constexpr (kFastScheme) {
    bool fast = a.fast_ops != 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) fast = fast && red.fast[w] != 0;
    using DF = typename std::conditional<kFastFlux, FastOps, IeeeOps>::type;
    if (fast)
      latency_edges<FLUX, LIMC, R, TX, TY, FastOps, DF, GEOM, NT>(a, sm, i0, j0);
    else
      latency_edges<FLUX, LIMC, R, TX, TY, IeeeOps, IeeeOps, GEOM, NT>(a, sm, i0, j0);
  } else if constexpr (kExact) {
    latency_edges<FLUX, LIMC, R, TX, TY, IeeeOps, IeeeOps, GEOM, NT>(a, sm, i0, j0);
  } else {
    R hold[4];  // of the split layout only
    edge_pass<FLUX, LIMC, R, TX, TY, IeeeOps, IeeeOps, GEOM, NT, false>(
        a, static_cast<TileSmem<LIMC, R, TX, TY, NT, false> &>(sm), i0, j0, hold);
    __syncthreads();
  }

  // ---- 4. divergence + stage combination of one variable
  double csq0 = 0.0, csq1 = 0.0;
  if (cell) {
    double L = flux_balance<kExact, GEOM>(g, (double)sm.flux_i(v, cx + 1, cy), (double)sm.flux_i(v, cx, cy),
                                          (double)sm.flux_j(v, cx, cy + 1), (double)sm.flux_j(v, cx, cy));
    if (v == 3 && a.src_E) L = L + src;
    const double r = combine<kExact>(a, L, dt, [&] { return u0; }, [&] { return uk; });
    if (conv) {
      const double d = r - fst;
      csq0 = d * d;
      csq1 = fst * fst;
    }
    st_cell<kExact>(&a.out[0][off + v * fs], r);
    sm.nv[v][c] = r;
  }
  if (conv) {
    csq0 = wave_sum(csq0);
    csq1 = wave_sum(csq1);
    if ((tid & 63) == 0) {
      red.s[tid >> 6][0] = csq0;
      red.s[tid >> 6][1] = csq1;
    }
  }
  if (a.mode == MODE_RESIDUAL) return;
  __syncthreads();
  if (conv && tid < 8) {
    constexpr int WV = NC / 64;  // waves per variable
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < WV; ++k) t = t + red.s[(tid & 3) * WV + k][tid >> 2];
    global(a.block_conv)[(size_t)tid * (size_t)(a.tiles_x * a.tiles_y) + tile] = t;
  }

  // ---- 5. primitives of the new state, its checks and its CFL value
  double lmin = __builtin_inf();
  if (v == 0 && cell && (kExact || a.last_stage)) {
    const double nv[4] = {sm.nv[0][c], sm.nv[1][c], sm.nv[2][c], sm.nv[3][c]};
    lmin = finish_cell<kExact>(a, nv, off, gi, g, err);
  }
  if (a.last_stage || a.block_err) store_tile_result<NT>(a, tile, lmin, err, red);
}

}  // namespace cato
