// fw_multi2d.hpp -- K steps of one 2D sheet per launch, for the light models
// (state all of the arithmetic type, at most three arrays) with uniform
// half-step fields.
//
// What it is for.  A step of a small sheet is all launch: replayed from a
// graph, Aliev-Panfilov on 102 x 102 nodes takes 3.1 us per step for 0.3 us
// of work, and a probe's per-step rows keep a run out of the graphs
// altogether (Fenton-Karma on 66 x 66: 8.4 us).  With K = 8 the two take 0.93
// and 1.6 us per step; bound by a launch's 5 us, then by the issue of a
// region's wavefronts.  A block here takes a
// region of kMultiW x RH nodes, one per work-item, and steps it K times
// before it writes the nodes it owns, those at least K from the region's edge:
// after t steps the values t or more nodes inside the region are exact.
//
// The potential is double-buffered in LDS: step t reads plane t & 1 and
// writes plane 1 - (t & 1), one barrier per step.  A node that is not
// updated holds in each plane what the u / u_new pair holds for it at that
// parity, so frozen nodes read as they do in single steps.  State, node code,
// activation word and, in FP64, the node's weights (formed once per launch
// instead of once per step) stay in registers.
//
// Reads and writes go to different arrays (blocks read their neighbours'
// nodes while those write): the potential from one buffer of the pair to the
// other, the state from the caller's arrays to the plan's second set (phase
// 0) or back (phase 1).  Launches come in pairs of equal K, after which
// everything is where single steps would have it, except u_new, which holds
// the potential of K steps ago: the caller ends a run with a single step.
//
// The arithmetic per node and step is step_node's (exact weights and their
// sum in FP64, flux_iso / flux_aniso in FP32, node_update), so every value is
// bit for bit that of single steps.
#pragma once

#include "fw_batch.hpp"
#include "fw_kernels.hpp"

namespace fw {

constexpr int kMultiW = 32;            // region columns: half a wavefront's lanes per row
constexpr int kMultiThreads = 1024;    // work-items of the largest region

template <typename R>
struct MultiArgs {
  const R* cur;          // the current potential of updated nodes
  const R* even;         // what other nodes hold at even and odd steps of the launch
  const R* odd;
  R* out;                // the buffer of the pair that `cur` is not
  const R* sin[3];
  R* sout[3];
  int32_t K, rows;       // steps; region rows
  int32_t own_w, own_h;  // nodes a block owns: kMultiW - 2 K, rows - 2 K
  int32_t tiles_j;
  int32_t ni, nj;
  int32_t step;          // global step of the launch's first step
  int32_t probe_row;     // probe row of the first step (the next ones follow), -1 closed
};

template <int ST, int MODEL, typename R>
__global__ __launch_bounds__(kMultiThreads) void k_multi2d(const KArgs<R, R> a,
                                                           const MultiArgs<R> g) {
  constexpr int NS = model_n_state(MODEL);
  constexpr bool EXACT = sizeof(R) == 8;
  constexpr int NW = EXACT ? (ST == 0 ? 5 : 9) : 1;
  static_assert(NS >= 1 && NS <= 3, "light models");
  __shared__ R plane[2][kMultiThreads];
  __shared__ uint8_t ctile[kMultiThreads];
  const int me = (int)threadIdx.x;
  const int lx = me & (kMultiW - 1), ly = me / kMultiW;
  const int K = g.K;
  const int tile_i = (int)blockIdx.x / g.tiles_j, tile_j = (int)blockIdx.x - tile_i * g.tiles_j;
  const int gi = tile_i * g.own_h - K + ly, gj = tile_j * g.own_w - K + lx;
  const bool in = gi >= 0 && gi < g.ni && gj >= 0 && gj < g.nj;
  const int c = in ? gi * g.nj + gj : 0;
  const uint8_t code = in ? a.code[c] : (uint8_t)0;
  const bool own = in && lx >= K && lx < K + g.own_w && ly >= K && ly < K + g.own_h;
  const bool upd = (code & 3) == 1 && gi > 0 && gi < g.ni - 1 && gj > 0 && gj < g.nj - 1;
  R uc = R(0), other = R(0);
  RegState<R, NS> s;
#pragma unroll
  for (int k = 0; k < NS; ++k) s.v[k] = R(0);
  if (in) {
    uc = upd ? g.cur[c] : g.even[c];
    other = upd ? uc : g.odd[c];
#pragma unroll
    for (int k = 0; k < NS; ++k) s.v[k] = g.sin[k][c];
  }
  int32_t act = 0, act0 = 0;
  if (a.act_on && own) act = act0 = a.act[c];
  plane[0][me] = uc;
  plane[1][me] = other;
  ctile[me] = code;
  __syncthreads();
  // nodes on the region's edge are never stepped: their neighbours lie outside
  const bool inner = lx > 0 && lx < kMultiW - 1 && ly > 0 && ly < g.rows - 1;
  const bool live = upd && inner;
  Hood2<R> q;
  R W[NW];
  if (live) {
#pragma unroll
    for (int di = -1; di <= 1; ++di)
#pragma unroll
      for (int dj = -1; dj <= 1; ++dj) {
        const int k = (di + 1) * 3 + dj + 1;
        const bool need = (ST == 1 || di == 0 || dj == 0) && k != 4;
        q.m[k] = need ? (ctile[me + di * kMultiW + dj] & 1) : 0;
        q.v[k] = R(0);
      }
    q.m[4] = 1;
    if constexpr (EXACT) {
      if constexpr (ST == 0) {
        const double d0 = a.f[0].value, d1 = a.f[1].value;
        W[0] = iso_comp(d0, q.m[1], q.m[7]);
        W[1] = iso_comp(d1, q.m[3], q.m[5]);
        W[3] = iso_comp(d1, q.m[5], q.m[3]);
        W[4] = iso_comp(d0, q.m[7], q.m[1]);
        W[2] = -(W[0] + W[1] + W[3] + W[4]);
        scale_exact<5>(W, 2, a.D, a.dtd, a.rdr2);
      } else {
        Nbr M;
#pragma unroll
        for (int k = 0; k < 27; ++k) M.m[k] = 0;
#pragma unroll
        for (int k = 0; k < 9; ++k) M.m[3 * k + 1] = q.m[k];
        const double xx = a.f[0].value, xy = a.f[1].value, yx = a.f[2].value, yy = a.f[3].value;
        wts_aniso2d(W, M, xx, xx, xy, xy, yx, yx, yy, yy);
        scale_exact<9>(W, 4, a.D, a.dtd, a.rdr2);
      }
    }
  }
  for (int t = 0; t < K; ++t) {
    const int32_t step = g.step + t;
    if (a.act_on && own && uc > a.act_thr && act < 0) act = step;
    const R pre = uc;
    // exact while t + 1 or more nodes inside the region
    if (live && lx > t && lx < kMultiW - 1 - t && ly > t && ly < g.rows - 1 - t) {
      const R* const p = plane[t & 1] + me;
      if constexpr (EXACT && ST == 0) {
        const R d = p[-kMultiW] * W[0] + p[-1] * W[1] + uc * W[2] + p[1] * W[3] +
                    p[kMultiW] * W[4];
        uc = node_update<MODEL, R>(uc, s, 0, a.dt, a.P, [&] { return d; });
      } else if constexpr (EXACT) {
        const R d = p[-kMultiW - 1] * W[0] + p[-kMultiW] * W[1] + p[-kMultiW + 1] * W[2] +
                    p[-1] * W[3] + uc * W[4] + p[1] * W[5] + p[kMultiW - 1] * W[6] +
                    p[kMultiW] * W[7] + p[kMultiW + 1] * W[8];
        uc = node_update<MODEL, R>(uc, s, 0, a.dt, a.P, [&] { return d; });
      } else {
#pragma unroll
        for (int di = -1; di <= 1; ++di)
#pragma unroll
          for (int dj = -1; dj <= 1; ++dj)
            if (ST == 1 || di == 0 || dj == 0)
              q.v[(di + 1) * 3 + dj + 1] = p[di * kMultiW + dj];
        q.v[4] = uc;
        uc = node_update<MODEL, R>(uc, s, 0, a.dt, a.P, [&] {
          if constexpr (ST == 0) {
            const R dx = funi<R>(a.f[0]), dy = funi<R>(a.f[1]);
            return flux_iso<R>(q, dx, dy, dy, dx, a.s);
          } else {
            const R xx = funi<R>(a.f[0]), xy = funi<R>(a.f[1]), yx = funi<R>(a.f[2]),
                    yy = funi<R>(a.f[3]);
            return flux_aniso<R>(q, xx, xx, xy, xy, yx, yx, yy, yy, a.s);
          }
        });
      }
      plane[1 - (t & 1)][me] = uc;
    } else if (!upd) {
      const R next = other;  // this node's value at the other parity
      other = uc;
      uc = next;
    }
    if ((code & 4) && own && g.probe_row >= 0) {
      for (int p = 0; p < a.n_probe; ++p) {
        if (a.probe_idx[p] != c) continue;
        const int var = a.probe_var[p];
        R val = pre;  // the pre-step potential, or a state after the update
#pragma unroll
        for (int k = 0; k < NS; ++k)
          if (var == k) val = s.v[k];
        a.probe_buf[(int64_t)(g.probe_row + t) * a.n_probe + p] = (double)val;
      }
    }
    __syncthreads();
  }
  if (own) {
    if (upd) g.out[c] = uc;
#pragma unroll
    for (int k = 0; k < NS; ++k) g.sout[k][c] = s.v[k];
    if (act != act0) a.act[c] = act;
  }
}

}  // namespace fw
