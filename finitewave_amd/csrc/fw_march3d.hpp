// fw_march3d.hpp -- the FP32 19-point step of 3D plans whose half-step fields
// are uniform or tables along k (layered fibres), for the two- to
// four-variable models: each face flux and each cross-term square computed
// once instead of by every node that touches it.
//
// The flux form of the anisotropic 19-point stencil (asymmetric_stencil_3d.py
// :163-458 in flux form): the flux into a node c across its upper face along
// axis a is
//   F_a(c) = d_aa * m(c) m(c+a) * (u(c+a) - u(c))
//          + sum over the two other axes b of d_ab * [on] * (Q(S_ab(c)) - Q(S_ab(c-b)))
// where S_ab(n) is the 2x2 square {n, n+a, n+b, n+a+b}, Q its mean over
// conducting nodes, and [on] requires c and c+a to conduct and both squares
// to hold at least three conducting nodes (the reference's minor_component,
// asymmetric_stencil_2d.py:246-259).  The flux across the lower face is
// -F_a(c-a), and the node update is u + s * sum of the six face fluxes.
//
// Work decomposition.  Lanes run along k; a lane owns kMarchRows consecutive
// rows j of its column and keeps one more on either side, and marches along i
// over a chunk of planes, starting one plane early (a halo plane whose results
// are not written).  Along j everything shared is in the lane's registers,
// along i in those of the previous plane, along k in the lanes either side (DPP
// wavefront shifts; lanes 0 and 63 are halo).  Per plane a lane loads plane
// i + 2 at its rows -- one potential and one code byte per row -- while it works on
// i and i + 1.
//
// A kernel with one row per lane issued 189 VALU instructions per node and
// waited for its loads every plane: 83 us per step of Aliev-Panfilov 258^3 with
// fibrosis 0.2, layered fibres.  Two rows share a third of the squares and
// fluxes; masks packed a nibble per row let one addition count the conducting
// nodes of a square for all rows (three or more when bit 2 of count + 1 is set,
// four when bit 2 of the count is), and a term's mask is one sign-extracted bit
// ANDed onto it: 118 instructions per node, 63 us, 4.6 TB/s of the 292 MB it
// moves.  It is now bound by HBM and by what four waves per SIMD hide of it;
// three and four rows per lane need 120 and 147 registers and ran at 66 us, the
// non-temporal hint on the state at 89, five waves with 8 registers spilled at
// 79.  The face fluxes are the reference operator's; their rounding differs
// from the per-node kernel's (k_step) by the order of the sums.
#pragma once

#include "fw_kernels.hpp"

namespace fw {

constexpr int kMarchOwn = 62;   // columns a wavefront owns (lanes 1..62)
constexpr int kMarchWaves = 4;  // wavefronts per block
constexpr int kMarchRows = 2;   // rows a lane owns

struct MarchGeom {
  int32_t plane;     // nj * nk
  int32_t columns;   // row groups * nk: a lane's work items per plane
  int32_t tiles;     // wavefront tiles per plane: ceil(columns / kMarchOwn)
  int32_t groups;    // blocks per plane: ceil(tiles / kMarchWaves)
  int32_t chunk;     // planes a block owns along i
  UDiv div_nk;       // division by nk
  uint32_t nblocks;  // groups * blocks along i
  uint32_t per_xcd;  // logical blocks per XCD
};

// all-ones when bit b of x is set, else 0: one instruction, where the compiler
// would test the bit and select (three for a masked value instead of two)
template <int B>
__device__ __forceinline__ uint32_t bit_mask(uint32_t x) {
  uint32_t m;
  asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(m) : "v"(x), "n"(B));
  return m;
}

// v when bit b of x is set, else +0
template <int B>
__device__ __forceinline__ float keep(uint32_t x, float v) {
  return __builtin_bit_cast(float, bit_mask<B>(x) & __builtin_bit_cast(uint32_t, v));
}

// the mean over a square's conducting nodes from their sum, for 4 (bit B of
// the counts set) or 3 of them
template <int B>
__device__ __forceinline__ float square_mean(uint32_t counts, float sum) {
  const uint32_t m = bit_mask<B>(counts);
  constexpr uint32_t quarter = 0x3e800000u, third = 0x3eaaaaabu;
  return sum * __builtin_bit_cast(float, (m & quarter) | (~m & third));
}

// element `off` of a wave-uniform array: a scalar base and a 32-bit byte
// offset per lane, so the address costs one shift
template <typename T>
__device__ __forceinline__ global_t<T>& at(global_t<T>* p, uint32_t off) {
  typedef std::conditional_t<std::is_const_v<T>, const char, char> B;
  return *(global_t<T>*)((global_t<B>*)p + off * (uint32_t)sizeof(T));
}

template <int N, typename F>
__device__ __forceinline__ void rows_of(F&& f) {
  tb_phases([&](auto r) { f(r); return true; }, std::make_integer_sequence<int, N>{});
}

template <int MODEL, int FL>
__global__ __launch_bounds__(kBlock) void k_step3_march(const KArgs<float, float> a,
                                                        const MarchGeom g) {
#pragma clang fp contract(fast)
  static_assert(kBlock == 64 * kMarchWaves, "one wavefront per 64 lanes");
  constexpr int J = kMarchRows, RL = J + 2;  // own rows; loaded rows (own: 1..J)
  static_assert(RL <= 8, "a nibble per row");
  constexpr uint32_t kOnes = 0x11111111u;
  const uint32_t b = blockIdx.x;
  const uint32_t lb = (b % kXcds) * g.per_xcd + b / kXcds;
  const int32_t step = a.step_in ? *a.step_in : a.step;
  if (a.step_out && b == 0 && threadIdx.x == 0) *a.step_out = step + 1;
  if (lb >= g.nblocks) return;
  const int32_t group = (int32_t)(lb % (uint32_t)g.groups);
  const int32_t chunk = (int32_t)(lb / (uint32_t)g.groups);
  const int lane = threadIdx.x & 63;
  const int32_t tile = group * kMarchWaves + (int32_t)(threadIdx.x >> 6);
  const int32_t p = tile * kMarchOwn + lane - 1;
  const int32_t pc = p < 0 ? 0 : (p >= g.columns ? g.columns - 1 : p);
  const int32_t nk = (int32_t)a.nk, nj = (int32_t)a.nj, ni = (int32_t)a.ni;
  const int32_t rg = (int32_t)udiv((uint32_t)pc, g.div_nk);
  const int32_t k = pc - rg * nk, j0 = rg * J;
  const bool own = p >= 0 && p < g.columns && lane > 0 && lane < 63 && tile < g.tiles;
  // plane offsets of the loaded rows, kept inside the grid (a repeated row
  // reaches only nodes of rows 0 and nj - 1, which are never updated)
  uint32_t off[RL];
  bool mine[J], inner[J];
#pragma unroll
  for (int r = 0; r < RL; ++r) {
    const int32_t j = j0 - 1 + r;
    off[r] = (uint32_t)((j < 0 ? 0 : (j >= nj ? nj - 1 : j)) * nk + k);
    if (r >= 1 && r <= J) {
      mine[r - 1] = own && j < nj;
      inner[r - 1] = mine[r - 1] && j >= 1 && j <= nj - 2 && k >= 1 && k <= nk - 2;
    }
  }
  // the faces' half-step values: along i and j the same on both sides; the
  // upper z face's at k (the lower one is lane - 1's upper one)
  float dxx, dxy, dxz, dyx, dyy, dyz, dzx, dzy, dzz;
  if constexpr (FL == kFieldsUniform) {
    dxx = a.f[0].fvalue, dxy = a.f[1].fvalue, dxz = a.f[2].fvalue;
    dyx = a.f[3].fvalue, dyy = a.f[4].fvalue, dyz = a.f[5].fvalue;
    dzx = a.f[6].fvalue, dzy = a.f[7].fvalue, dzz = a.f[8].fvalue;
  } else {
    auto t = [&](int q) { return ((const global_t<float>*)a.f[q].fdata)[k]; };
    dxx = t(0), dxy = t(1), dxz = t(2), dyx = t(3), dyy = t(4), dyz = t(5);
    dzx = t(6), dzy = t(7), dzz = t(8);
  }
  const bool stim_next = stim_due(a, step + 1);
  const int32_t i0 = chunk * g.chunk;
  const int32_t i1 = i0 + g.chunk < ni ? i0 + g.chunk : ni;
  const int32_t ibeg = i0 > 0 ? i0 - 1 : 0;
  // plane i's potentials and codes at the lane's rows, planes past the last
  // one read as the last (no node of it is updated)
  auto load = [&](int32_t i, float (&u)[RL], uint32_t (&cd)[RL]) {
    const int64_t base = (int64_t)(i < ni ? i : ni - 1) * g.plane;
    const global_t<float>* const up = (const global_t<float>*)a.u + base;
    const global_t<uint8_t>* const cp = (const global_t<uint8_t>*)a.code + base;
#pragma unroll
    for (int r = 0; r < RL; ++r) u[r] = at(up, off[r]);
#pragma unroll
    for (int r = 0; r < RL; ++r) cd[r] = cp[off[r]];
  };
  constexpr int NS = model_n_state(MODEL);
  // planes i, i + 1 and i + 2 live in slots c, n and f of three, a phase of
  // the loop each: nothing moves between registers, so no wait for a load in
  // flight comes before the plane that needs it
  float U[3][RL], W[3][RL];
  uint32_t C[3][RL], M[3];
  // the lower-x quantities of a plane are those the plane before stored
  float FX[3][J], XY[3][J + 1], XZ[3][J];
  uint32_t OKXY[3], OKXZ[3];
  auto mask_plane = [&](auto slot) {
    constexpr int q = decltype(slot)::value;
    uint32_t m = 0;
#pragma unroll
    for (int r = 0; r < RL; ++r) m |= (C[q][r] & 1u) << (4 * r);
    M[q] = m;
    rows_of<RL>([&](auto r) { W[q][r] = keep<4 * decltype(r)::value>(m, U[q][r]); });
  };
  load(ibeg, U[0], C[0]);
  load(ibeg + 1, U[1], C[1]);
  mask_plane(std::integral_constant<int, 0>{});
#pragma unroll
  for (int r = 0; r < J; ++r) FX[2][r] = XZ[2][r] = 0.0f;
#pragma unroll
  for (int r = 0; r <= J; ++r) XY[2][r] = 0.0f;
  OKXY[2] = OKXZ[2] = 0;
  int32_t i = ibeg;
  auto plane = [&](auto ph) -> bool {
    constexpr int cu = decltype(ph)::value, nx = (cu + 1) % 3, lo = (cu + 2) % 3;
    if (i >= i1) return false;
    // the offsets stay 32-bit in each iteration (their 64-bit forms, kept
    // across the loop, would double their registers and cost an addition per
    // access)
#pragma unroll
    for (int r = 0; r < RL; ++r) asm volatile("" : "+v"(off[r]));
    // in flight during this plane: the state of i, then, not waited for until
    // the next, the potentials and codes of i + 2
    const int64_t base = (int64_t)i * g.plane;
    RegState<float, NS> st[J];
#pragma unroll
    for (int r = 0; r < J; ++r)
#pragma unroll
      for (int q = 0; q < NS; ++q)
        st[r].v[q] = at((const global_t<float>*)a.st.p[q] + base, off[r + 1]);
    load(i + 2, U[lo], C[lo]);
    asm volatile("" ::: "memory");  // the loads are issued here, not where they are used
    mask_plane(std::integral_constant<int, nx>{});
    const float(&u)[RL] = U[cu];
    const float(&n)[RL] = U[nx];
    const float(&w)[RL] = W[cu];
    const uint32_t(&cd)[RL] = C[cu];
    const uint32_t m = M[cu], mn = M[nx];
    // conducting nodes of the squares each row starts, and the masks of the
    // faces it starts (bit 2 of the row's nibble)
    const uint32_t cx = m + mn, cy = m + (m >> 4);
    const uint32_t cxy = cx + (cx >> 4);
    const uint32_t cxz = cx + from_east(cx);
    const uint32_t cyz = cy + from_east(cy);
    const uint32_t okxy = cxy + kOnes, okxz = cxz + kOnes, okyz = cyz + kOnes;
    const uint32_t m4 = m << 2;
    const uint32_t mx = m4 & (mn << 2), my = m4 & (m4 >> 4), mz = m4 & from_east(m4);
    const uint32_t x_xy = okxy & (okxy << 4) & mx, x_xz = okxz & from_west(okxz) & mx;
    const uint32_t y_xy = okxy & OKXY[lo] & my, y_yz = okyz & from_west(okyz) & my;
    const uint32_t z_xz = okxz & OKXZ[lo] & mz, z_yz = okyz & (okyz << 4) & mz;
    OKXY[cu] = okxy;
    OKXZ[cu] = okxz;
    // the squares' means: S_xy and S_yz of rows 0..J, S_xz of rows 1..J
    float col[RL], yz[J + 1];
    float(&xy)[J + 1] = XY[cu];
    float(&xz)[J] = XZ[cu];
    rows_of<RL>([&](auto r) { col[r] = w[r] + W[nx][r]; });
    rows_of<J + 1>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      xy[r] = square_mean<4 * r + 2>(cxy, col[r] + col[r + 1]);
      const float row = w[r] + w[r + 1];
      yz[r] = square_mean<4 * r + 2>(cyz, row + from_east(row));
    });
    rows_of<J>([&](auto rr) {
      constexpr int r = decltype(rr)::value + 1;
      xz[r - 1] = square_mean<4 * r + 2>(cxz, col[r] + from_east(col[r]));
    });
    // fluxes across the upper y faces of rows 0..J, the upper x and z faces of
    // rows 1..J
    float fy[J + 1], fz[J];
    float(&fx)[J] = FX[cu];
    rows_of<J + 1>([&](auto rr) {
      constexpr int r = decltype(rr)::value, B = 4 * r + 2;
      float f = dyy * keep<B>(my, u[r + 1] - u[r]);
      f += dyx * keep<B>(y_xy, xy[r] - XY[lo][r]);
      f += dyz * keep<B>(y_yz, yz[r] - from_west(yz[r]));
      fy[r] = f;
    });
    rows_of<J>([&](auto rr) {
      constexpr int r = decltype(rr)::value + 1, B = 4 * r + 2;
      float f = dxx * keep<B>(mx, n[r] - u[r]);
      f += dxy * keep<B>(x_xy, xy[r] - xy[r - 1]);
      f += dxz * keep<B>(x_xz, xz[r - 1] - from_west(xz[r - 1]));
      fx[r - 1] = f;
      float h = dzz * keep<B>(mz, from_east(u[r]) - u[r]);
      h += dzx * keep<B>(z_xz, xz[r - 1] - XZ[lo][r - 1]);
      h += dzy * keep<B>(z_yz, yz[r] - yz[r - 1]);
      fz[r - 1] = h;
    });
    float fl[J];
    rows_of<J>([&](auto rr) {
      constexpr int r = decltype(rr)::value;
      fl[r] = (fx[r] - FX[lo][r]) + (fy[r + 1] - fy[r]) + (fz[r] - from_west(fz[r]));
    });
    // the update of every lane first, the stores under their masks after: no
    // wait stands between the rows
    float v[J];
#pragma unroll
    for (int r = 0; r < J; ++r)
      v[r] = node_update<MODEL, float>(u[r + 1], st[r], 0, a.dt, a.P,
                                       [&] { return u[r + 1] + a.s * fl[r]; });
    const bool ours = i >= i0, in_i = ours && i >= 1 && i <= ni - 2;
    if (a.act_on && ours) {
      // the activation word is read only for a potential above the
      // threshold: below it nothing can be recorded, and a read whose
      // result the loop waits on costs every plane its latency
#pragma unroll
      for (int r = 0; r < J; ++r)
        if (mine[r] && u[r + 1] > a.act_thr && a.act[base + off[r + 1]] < 0)
          a.act[base + off[r + 1]] = step;
    }
    if (stim_next && ours) {
#pragma unroll
      for (int r = 0; r < J; ++r) {
        const int64_t c = base + off[r + 1];
        if (!mine[r] || (cd[r + 1] & 1) == 0) continue;
        if (cd[r + 1] & 2)
          a.u_new[c] = stim_node<float>(a, step + 1, i, j0 + r, k, c, a.u_new[c]);
        else
          v[r] = stim_node<float>(a, step + 1, i, j0 + r, k, c, v[r]);
      }
    }
#pragma unroll
    for (int r = 0; r < J; ++r)
      if ((cd[r + 1] & 3) == 1 && inner[r] && in_i) {
        at((global_t<float>*)a.u_new + base, off[r + 1]) = v[r];
#pragma unroll
        for (int q = 0; q < NS; ++q)
          at((global_t<float>*)a.st.p[q] + base, off[r + 1]) = st[r].v[q];
      }
    if (a.probe_row >= 0 && ours) {
#pragma unroll
      for (int r = 0; r < J; ++r)
        if (mine[r])
          probe_node<float, MODEL, 1>(a, base + off[r + 1], (uint8_t)cd[r + 1],
                                      (double)u[r + 1]);
    }
    ++i;
    return true;
  };
  while (tb_phases(plane, std::make_integer_sequence<int, 3>{})) {
  }
}

// the launch geometry of k_step3_march for an ni x nj x nk grid; false when
// the grid's counts do not fit its 32-bit indexing
inline bool march_geom(int64_t ni, int64_t nj, int64_t nk, MarchGeom& g) {
  const int64_t plane = nj * nk, columns = (nj + kMarchRows - 1) / kMarchRows * nk;
  if (plane > (int64_t)1 << 29 || ni > INT32_MAX) return false;
  const int64_t tiles = (columns + kMarchOwn - 1) / kMarchOwn;
  const int64_t groups = (tiles + kMarchWaves - 1) / kMarchWaves;
  // Planes per block: the fewest that leave every block a place on the chip at
  // once (256 CUs, 4 waves per SIMD), 16 at most.  A block marches its planes
  // one after the other, so a small grid wants short chunks (us per step:
  // 37 x 45 x 67 5.1 with one plane, 14.1 with 16; 100 x 90 x 110 9.4 with 2,
  // 15.6 with 16) and a large one the lesser share of halo planes (258^3: 67.4
  // with 6, 63 from 12 to 20, 73 with 43).
  constexpr int64_t kSlots = 256 * 4;
  int64_t chunk = 1;
  while (chunk < 16 && groups * ((ni + chunk - 1) / chunk) > kSlots) ++chunk;
  const int64_t nb = groups * ((ni + chunk - 1) / chunk);
  if (nb > (int64_t)UINT32_MAX / 2) return false;
  g.plane = (int32_t)plane;
  g.columns = (int32_t)columns;
  g.tiles = (int32_t)tiles;
  g.groups = (int32_t)groups;
  g.chunk = (int32_t)chunk;
  g.div_nk = make_udiv((uint32_t)nk);
  g.nblocks = (uint32_t)nb;
  g.per_xcd = (g.nblocks + kXcds - 1) / kXcds;
  return true;
}

}  // namespace fw
