// Two time steps of a D3Q19 block per pass over HBM.
//
// k_step_march takes a block from one swapped (parity 1) state to the next,
// an odd and an even AA step together, reading one population array and
// writing another. A workgroup owns an x-y tile and walks it along z; the
// state between the two steps only ever lives in LDS and registers:
//   odd step   every thread of the tile and of a one-cell ring around it
//              gathers its column's next cell from HBM and collides it;
//   exchange   the post-collision values that move in x or y (16 of 19) go
//              through a plane of LDS; those along +-z stay in the thread;
//   even step  the tile's cells of the plane below are complete once the
//              plane above them has collided: they collide and are stored
//              where the even step stores them, their own slots.
// The ring is computed by the neighbouring workgroups too (the same bits), so
// workgroups share nothing and need no order. The target must not be the
// source: a workgroup reads ring cells that another one writes.
//
// The one-step kernels are bound by HBM (152 bytes per cell and step in FP32,
// at 88 % of the copy rate on the 256^3 cavity), so the bytes are what can be
// saved: two steps here read 1.45 GB there and write 1.28 GB, against
// 2 x 2.59 GB. Measured per step, FP32 BGK cavities: 256^3 0.444 -> 0.291 ms
// (57.6 GLUPS), 192^3 222 -> 142 us, 100^3 27.1 -> 21.5 us; FP64 256x200x160
// 436 -> 292 us. What bounds it now is the walk of one workgroup of 16
// wavefronts per CU (LDS holds no second one): matrix-free VALU work half the
// time, else waiting for the next plane.
//
// Choices measured at 256^3 FP32 (per step): the next plane's loads issued
// before the first collision instead of after it 0.335 ms (against 0.300
// there); two workgroups of 512 threads per CU 0.340 (their rings are
// larger); scalar offsets formed anew for each plane 0.329 (39 % more
// scalar instructions); stores held back to the next plane 0.332. The ring's
// columns x = -1 and x = w sit behind the rows in the thread order, so that
// wavefronts cover aligned rows: rows and ring columns in one run read 17 %
// more from HBM.
//
// The 16-bit kinds do not take it: they are bound by their conversions and
// collisions rather than by bytes (FP16 shift, 190x161x130: 57.0 us against
// 50.8 us in single steps).
//
// Cells, links, wall terms and collisions are those of the one-step kernels,
// in the same order and rounding: a block's populations do not depend on
// which kernels stepped it. Needed of the block (checked on the host):
// - every link of an updated cell that leads to a cell that is not updated is
//   a halfway wall link (k_open_links), so no step reads or writes the slots
//   of cells that are not updated;
// - one dynamics for all updated cells, and none that writes fields (ring
//   cells would be written twice).
#pragma once

#include "flb_kernels.hpp"

namespace flb {
namespace kern {

// LDS planes of the exchange, one value per thread each: the directions that
// move in x or y. Directions 0, 5 and 6 never leave the thread.
constexpr int kMarchPlanes = 16;
__host__ __device__ constexpr int march_plane(int i) { return i >= 7 ? i - 3 : ((i >= 1 && i <= 4) ? i - 1 : -1); }

// One cell's per-plane data, fetched ahead of its populations: bit 0 of lk is
// set when the cell is updated, bit i when its link i is a halfway wall; lm:
// the links of moving walls among them.
struct MarchCell {
  unsigned lk, lm;
};

// pop_rsrc with its words held to scalar registers (the walk's plane index is
// uniform, which the compiler does not always see).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t march_rsrc(void* pops, uint64_t total, size_t elem, int64_t e0) {
  const int64_t u = (int64_t(__builtin_amdgcn_readfirstlane(int(e0 >> 32))) << 32) |
                    uint32_t(__builtin_amdgcn_readfirstlane(int(e0)));
  return pop_rsrc(pops, total, elem, u);
}

// One ring row and cell of slack at both ends for the shifted reads of ring lanes.
constexpr int kMarchSlack = kMarchMaxRow + 1;
template <class S>
constexpr int kMarchLds = 2 * kMarchPlanes * march_threads(sizeof(typename S::E)) + 2 * kMarchSlack;

// Workgroup wg of a block's march from the populations src to dst.
template <class S, int DYN, bool PER>
__device__ __forceinline__ void march_tile(const KArgs& a, const MarchArgs& m, void* src, void* dst, unsigned wg,
                                           typename S::E* lds) {
  constexpr int Q = 19;
  constexpr int NT = march_threads(sizeof(typename S::E));
  constexpr int FAM = DYN == DYN_BGK ? FAM_BGK : FAM_FULL;
  using R = typename S::R;
  using E = typename S::E;
  constexpr uint32_t el = sizeof(E);
  constexpr int kSlack = kMarchSlack;

  const int tid = int(threadIdx.x);
  const int pw = m.w + 2;
  const int tx = int(wg % unsigned(m.ntx)), wy = int(wg / unsigned(m.ntx));
  const int ty = wy % m.nty, zc = wy / m.nty;
  // place in the tile, -1 and w / h on the ring: the tile's columns of every
  // row first, so that wavefronts cover whole aligned rows, then the ring's
  // two columns
  int lx, ly;
  if (tid < m.w * (m.h + 2)) {
    const int r = tid / m.w;
    lx = tid - r * m.w;
    ly = r - 1;
  } else {
    const int j = tid - m.w * (m.h + 2);
    lx = (j & 1) ? m.w : -1;
    ly = (j >> 1) - 1;
  }
  const int pos = min((ly + 1) * pw + lx + 1, NT - 1);  // LDS slot
  int cx0 = tx * m.w + lx, cy0 = ty * m.h + ly;   // updated-cell coordinates
  const bool core = lx >= 0 && lx < m.w && ly >= 0 && ly < m.h && cx0 < a.ex && cy0 < a.ey;
  bool upd = ly <= m.h;  // threads past the ring idle
  if (PER && a.px) {
    upd = upd && cx0 <= a.ex;
    cx0 = cx0 < 0 ? cx0 + a.ex : (cx0 >= a.ex ? cx0 - a.ex : cx0);
  }
  if (PER && a.py) {
    upd = upd && cy0 <= a.ey;
    cy0 = cy0 < 0 ? cy0 + a.ey : (cy0 >= a.ey ? cy0 - a.ey : cy0);
  }
  upd = upd && cx0 >= 0 && cx0 < a.ex && cy0 >= 0 && cy0 < a.ey;
  const int y = a.ys + cy0;
  const int sxy = cx0 + a.pitch * y;  // flags / fields slot in plane 0

  // Lane byte offsets. No periodic axis: the column's cell from the tile's
  // first updated row, the neighbour in the scalar offset. Periodic blocks
  // wrap per lane: the columns and rows of the x and y neighbours, each one
  // element further on (x - 1 may be slot -1).
  const int yt = PER ? 0 : __builtin_amdgcn_readfirstlane(max(a.ys, a.ys + ty * m.h - 1));
  const uint32_t own = uint32_t(a.ypop * (y - yt) + cx0) * el;
  uint32_t X[3], Y[3];
  if constexpr (PER) {
    int xm = cx0 - 1, xp = cx0 + 1, ym = y - 1, yq = y + 1;
    if (a.px) {
      xm = xm < 0 ? xm + a.nx : xm;
      xp = xp >= a.nx ? xp - a.nx : xp;
    }
    if (a.py) {
      ym = ym < 0 ? ym + a.ny : ym;
      yq = yq >= a.ny ? yq - a.ny : yq;
    }
    X[0] = uint32_t(xm + 1) * el;
    X[1] = uint32_t(cx0 + 1) * el;
    X[2] = uint32_t(xp + 1) * el;
    Y[0] = uint32_t(ym * a.ypop) * el;
    Y[1] = uint32_t(y * a.ypop) * el;
    Y[2] = uint32_t(yq * a.ypop) * el;
  }
  const int32_t dp = int32_t(a.dpop), yp = a.ypop, zp = int32_t(a.zpop);
  const int32_t B = zp + yp + 1;

  const int za = __builtin_amdgcn_readfirstlane(a.zs + zc * m.zchunk);
  const int zb = min(za + m.zchunk, a.zs + a.ez);
  // updated planes are zs .. zs + ez - 1; on a periodic axis the planes beyond wrap
  auto live = [&](int z) { return (PER && a.pz) || (z >= a.zs && z < a.zs + a.ez); };
  auto wrap = [&](int z) {
    if (PER && a.pz) z = z < 0 ? z + a.nz : (z >= a.nz ? z - a.nz : z);
    return z;
  };
  auto cell_flag = [&](int z) -> unsigned {
    unsigned fl = 0;
    if (z <= zb && live(z) && upd) fl = in_global(a.flags)[sxy + int(a.plane) * wrap(z)];
    return fl;
  };
  auto cell_info = [&](int z, unsigned fl) {
    MarchCell c{0u, 0u};
    if (z > zb || !live(z) || !(fl & m.mask)) return c;
    c.lk = 1u;
    if (fl & a.bcany) {
      const uint64_t l = in_global(a.links)[sxy + int(a.plane) * wrap(z)];
      c.lm = uint32_t(l >> 32);
      c.lk = 1u | uint32_t(l) | c.lm;
    }
    return c;
  };
  // Gather of the odd step for the column's cell in plane z; a lane whose
  // upstream neighbour is a wall takes its own slot. The descriptor starts B
  // elements before row yt of the plane (as odd_buf's), that of a periodic
  // block one element before plane 0.
  auto gather = [&](int z, const MarchCell& c, E (&f)[Q]) {
    const unsigned lk = c.lk;
    if (!lk) return;
    if constexpr (PER) {
      const auto rs = march_rsrc(src, a.pop_total, el, int64_t(kFrontPad) - 1);
      const uint32_t zo[3] = {uint32_t(wrap(z - 1) * zp) * el, uint32_t(wrap(z) * zp) * el,
                              uint32_t(wrap(z + 1) * zp) * el};
#pragma unroll
      for (int i = 0; i < Q; ++i)
        f[i] = bld_pop_s<1, E>(rs, X[1 - Lat<Q>::cx(i)] + Y[1 - Lat<Q>::cy(i)],
                               uint32_t(opp(i) * dp) * el + zo[1 - Lat<Q>::cz(i)]);
      if (__ballot(lk > 1u) != 0) {
#pragma unroll
        for (int i = 1; i < Q; ++i)
          if ((lk >> opp(i)) & 1u) f[i] = bld_pop_s<1, E>(rs, X[1] + Y[1], uint32_t(i * dp) * el + zo[1]);
      }
    } else {
      const auto rs = march_rsrc(src, a.pop_total, el, int64_t(kFrontPad) + a.zpop * z + int64_t(a.ypop) * yt - B);
      if (__ballot(lk > 1u) == 0) {
#pragma unroll
        for (int i = 0; i < Q; ++i)
          f[i] = bld_pop_s<1, E>(rs, own, uint32_t(B + opp(i) * dp + nb_rel<Q>(opp(i), yp, zp)) * el);
      } else {
#pragma unroll
        for (int i = 0; i < Q; ++i) {
          const uint32_t so = uint32_t(B + opp(i) * dp + nb_rel<Q>(opp(i), yp, zp)) * el;
          const uint32_t sw = uint32_t(B + i * dp) * el;
          f[i] = bld_pop_s<1, E>(rs, own + (i != 0 && ((lk >> opp(i)) & 1u) ? sw : so), 0u);
        }
        // keeps the two forms apart: merged, their scalar offsets become lane values
        asm volatile("; links");
      }
    }
  };

  const R om = R(a.omega), _om = R(1) - om;

  MarchCell cur = cell_info(za - 1, cell_flag(za - 1));
  MarchCell next = cell_info(za, cell_flag(za));
  unsigned fl2 = cell_flag(za + 1);
  unsigned blk = 0u;  // links of the cell below
  E P[Q];             // its streamed-in values of the upward and in-plane directions
  E N[5];             // those moving up into the plane above: directions 5, 9, 11, 16, 18
  constexpr int kUp[5] = {5, 9, 11, 16, 18};
  E g[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) g[i] = P[i] = E(0);
#pragma unroll
  for (int k = 0; k < 5; ++k) N[k] = E(0);
  gather(za - 1, cur, g);
  for (int z = za - 1; z <= zb; ++z) {
    const int k = z - (za - 1);
    E* const L = lds + kSlack + (k & 1) * (kMarchPlanes * NT) + pos;
    const E* const Lb = lds + kSlack + ((k & 1) ^ 1) * (kMarchPlanes * NT) + pos;
    E h[Q];  // post-collision values, unset in lanes that update no cell
    if (cur.lk) {
      const int s0 = sxy + int(a.plane) * wrap(z);
      R f[Q];
#pragma unroll
      for (int i = 0; i < Q; ++i) f[i] = pop_dec<Q, S>(g[i], i);
      wall_terms_in<Q>(a, s0, cur.lm, f);
      collide<Q, R, FAM, kDev<Q, S>>(a, s0, DYN, m.cs, f, om, _om);
      wall_terms_out<Q>(a, s0, cur.lm, f);
#pragma unroll
      for (int i = 0; i < Q; ++i) h[i] = pop_enc<Q, S>(f[i], i);
    }
#pragma unroll
    for (int i = 1; i < Q; ++i)
      if (march_plane(i) >= 0) L[march_plane(i) * NT] = h[i];
    const E h0 = h[0], h5 = h[5], h6 = h[6];
    MarchCell after{0u, 0u};
    {
      E v[Q];  // unset in lanes that gather nothing; their values are never used
      if (z < zb) {
        gather(z + 1, next, v);
        after = cell_info(z + 2, fl2);
        fl2 = cell_flag(z + 3);
      }
#pragma unroll
      for (int i = 0; i < Q; ++i) g[i] = v[i];
    }
    // LDS only: the loads above stay in flight across the barrier
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    auto from = [&](int i) { return L[march_plane(i) * NT - Lat<Q>::cx(i) - Lat<Q>::cy(i) * pw]; };
    if (z > za && core && blk) {
      P[6] = h6;
#pragma unroll
      for (int i = 1; i < Q; ++i)
        if (march_plane(i) >= 0 && Lat<Q>::cz(i) < 0) P[i] = from(i);
      if (blk > 1u) {
#pragma unroll
        for (int i = 1; i < Q; ++i) {
          const int o = opp(i);
          if (Lat<Q>::cz(i) < 0 && ((blk >> o) & 1u)) P[i] = o == 5 ? N[0] : Lb[march_plane(o) * NT];
        }
      }
      R f[Q];
#pragma unroll
      for (int i = 0; i < Q; ++i) f[i] = pop_dec<Q, S>(P[i], i);
      collide<Q, R, FAM, kDev<Q, S>>(a, sxy + int(a.plane) * (z - 1), DYN, m.cs, f, om, _om);
      const auto rd = march_rsrc(dst, a.pop_total, el, int64_t(kFrontPad) + a.zpop * (z - 1) + int64_t(a.ypop) * yt);
#pragma unroll
      for (int i = 0; i < Q; ++i) bst_pop_s<2, E>(rd, own, uint32_t(opp(i) * dp) * el, pop_enc<Q, S>(f[i], i));
    }
    // streamed-in values of this plane, and those moving up into the next
    blk = cur.lk;
    P[0] = h0;
#pragma unroll
    for (int i = 1; i < Q; ++i)
      if (Lat<Q>::cz(i) == 0) P[i] = from(i);
#pragma unroll
    for (int k5 = 0; k5 < 5; ++k5) P[kUp[k5]] = N[k5];
    if (blk > 1u) {
#pragma unroll
      for (int i = 1; i < Q; ++i) {
        const int o = opp(i);
        if (Lat<Q>::cz(i) >= 0 && ((blk >> o) & 1u)) P[i] = o == 6 ? h6 : L[march_plane(o) * NT];
      }
    }
    N[0] = h5;
#pragma unroll
    for (int k5 = 1; k5 < 5; ++k5) N[k5] = from(kUp[k5]);
    cur = next;
    next = after;
  }
}

template <class S, int DYN, bool PER>
__global__ __launch_bounds__(march_threads(sizeof(typename S::E))) void k_step_march(KArgs a, MarchArgs m) {
  __shared__ typename S::E lds[kMarchLds<S>];
  march_tile<S, DYN, PER>(a, m, a.pops, m.dst, xcd_block(blockIdx.x, gridDim.x), lds);
}

// The march of many blocks in one launch, a block and its workgroup for every
// workgroup. back: from the second arrays to the blocks' own. The table's
// order is that of dispatch, longest workgroup first: as contiguous runs per
// XCD, in the blocks' order, 256 cavities of 43.2 M cells take 1.195 ms per
// step against 1.093, 40 of 6.3 M 176 us against 170.
template <class S, int DYN, bool PER>
__global__ __launch_bounds__(march_threads(sizeof(typename S::E))) void k_march_batch(
    const KArgs* __restrict__ tab, const MarchArgs* __restrict__ mt, const MarchWg* __restrict__ wgs, int back) {
  __shared__ typename S::E lds[kMarchLds<S>];
  wgs = in_const(wgs);
  const int e = __builtin_amdgcn_readfirstlane(wgs[blockIdx.x].block);
  const unsigned wg = unsigned(__builtin_amdgcn_readfirstlane(wgs[blockIdx.x].wg));
  const KArgs& a = in_const(tab)[e];
  const MarchArgs& m = in_const(mt)[e];
  march_tile<S, DYN, PER>(a, m, back ? m.dst : a.pops, back ? a.pops : m.dst, wg, lds);
}

// Counts the links of updated cells that lead to a cell that is not updated
// (no task, or beyond a non-periodic face) and are no halfway wall links.
template <int Q, bool PER>
__global__ __launch_bounds__(kMaxThreads) void k_open_links(KArgs a, unsigned mask, uint32_t* open) {
  const int64_t k = int64_t(blockIdx.x) * kMaxThreads + threadIdx.x;
  const int64_t n = int64_t(a.ex) * a.ey * a.ez;
  bool bad = false;
  if (k < n) {
    const int c0 = int(k % a.ex);
    const int64_t r = k / a.ex;
    const int x = a.xs + c0, y = a.ys + int(r % a.ey), z = a.zs + int(r / a.ey);
    const int s0 = c0 + a.pitch * y + int(a.plane) * z;
    const unsigned fl = a.flags[s0];
    if (fl & mask) {
      const uint64_t l = (fl & a.bcany) ? a.links[s0] : 0u;
      const unsigned lk = uint32_t(l) | uint32_t(l >> 32);
#pragma unroll
      for (int i = 1; i < Q; ++i) {
        const int xn = x + Lat<Q>::cx(i), yn = y + Lat<Q>::cy(i), zn = z + Lat<Q>::cz(i);
        const bool in = ((PER && a.px) || (xn >= a.xs && xn < a.xs + a.ex)) &&
                        ((PER && a.py) || (yn >= a.ys && yn < a.ys + a.ey)) &&
                        ((PER && a.pz) || (zn >= a.zs && zn < a.zs + a.ez));
        const bool goes = in && (a.flags[s0 + nb_off<Q, PER, false>(a, i, x, y, z)] & mask);
        bad = bad || (!goes && !((lk >> i) & 1u));
      }
    }
  }
  if (__ballot(bad) != 0 && (threadIdx.x & 63) == 0) *open = 1u;
}

template <class S, int DYN>
hipError_t march_dyn(const KArgs& a, const MarchArgs& m, hipStream_t s) {
  const dim3 grid(unsigned(m.ntx) * unsigned(m.nty) * unsigned(m.nz)), block(march_threads(sizeof(typename S::E)));
  if (a.px || a.py || a.pz) hipLaunchKernelGGL((k_step_march<S, DYN, true>), grid, block, 0, s, a, m);
  else hipLaunchKernelGGL((k_step_march<S, DYN, false>), grid, block, 0, s, a, m);
  return hipGetLastError();
}

template <class S>
hipError_t launch_march(const KArgs& a, const MarchArgs& m, hipStream_t s) {
  switch (m.dyn) {
    case DYN_BGK: return march_dyn<S, DYN_BGK>(a, m, s);
    case DYN_BGK_FORCE: return march_dyn<S, DYN_BGK_FORCE>(a, m, s);
    case DYN_SMAG_MRT:
      if constexpr (sizeof(typename S::E) == 8) return march_dyn<S, DYN_SMAG_MRT>(a, m, s);
      else return hipErrorInvalidValue;  // single steps (march_pays)
    default: return hipErrorInvalidValue;
  }
}

template <class S, int DYN>
hipError_t march_batch_dyn(bool per, const KArgs* tab, const MarchArgs* mt, const MarchWg* wgs, unsigned n, int back,
                           hipStream_t s) {
  const dim3 grid(n), block(march_threads(sizeof(typename S::E)));
  if (per) hipLaunchKernelGGL((k_march_batch<S, DYN, true>), grid, block, 0, s, tab, mt, wgs, back);
  else hipLaunchKernelGGL((k_march_batch<S, DYN, false>), grid, block, 0, s, tab, mt, wgs, back);
  return hipGetLastError();
}

template <class S>
hipError_t launch_march_batch(int dyn, bool per, const KArgs* tab, const MarchArgs* mt, const MarchWg* wgs, unsigned n,
                              int back, hipStream_t s) {
  switch (dyn) {
    case DYN_BGK: return march_batch_dyn<S, DYN_BGK>(per, tab, mt, wgs, n, back, s);
    case DYN_BGK_FORCE: return march_batch_dyn<S, DYN_BGK_FORCE>(per, tab, mt, wgs, n, back, s);
    case DYN_SMAG_MRT: return march_batch_dyn<S, DYN_SMAG_MRT>(per, tab, mt, wgs, n, back, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace kern
}  // namespace flb

// Defines the march launchers of flb_internal.hpp for one storage kind.
#define FLB_DEFINE_MARCH(SUFFIX, STORE)                                                            \
  namespace flb {                                                                                  \
  hipError_t launch_march_##SUFFIX(const KArgs& a, const MarchArgs& m, hipStream_t s) {            \
    return kern::launch_march<STORE>(a, m, s);                                                     \
  }                                                                                                \
  hipError_t launch_march_batch_##SUFFIX(int dyn, bool per, const KArgs* tab, const MarchArgs* mt, \
                                         const MarchWg* wgs, unsigned n, int back, hipStream_t s) { \
    return kern::launch_march_batch<STORE>(dyn, per, tab, mt, wgs, n, back, s);                 \
  }                                                                                                \
  }
