// Host side of the two-step march (flb_march.hpp): which blocks take it, the
// tiles of a block, and the passes of a run of steps.

#include <hip/hip_runtime.h>

#include <algorithm>

#include "flb_host.hpp"
#include "flb_internal.hpp"

namespace flbh {

namespace {

// Estimated time of one plane of a tile of w x h cells (ntx tiles along x).
double plane_time(int w, int h, int ntx, int elem) {
  const int line = 128 / elem;
  const double reads = (h + 2) * (double(w) / line + (ntx > 1 ? 2.0 : 1.0));
  return 2.0 + 0.06 * reads + 0.005 * double((w + 2) * (h + 2)) * (elem == 8 ? 2.0 : 1.0);
}

// Calls f(w, h, ntx, nty) for the tile extents worth considering.
template <class F>
void each_tile(const KArgs& a, int elem, F&& f) {
  const int threads = flb::march_threads(size_t(elem)), line = 128 / elem;
  for (int n = 1; n <= a.ex; ++n) {
    int w = (a.ex + n - 1) / n;
    if (a.pitch >= 256) w = (w + line - 1) / line * line;
    if (w + 2 > flb::kMarchMaxRow) continue;
    if (w < 8 && n > 1) break;
    const int hmax = std::min(a.ey, threads / (w + 2) - 2), first = (a.ey + hmax - 1) / hmax;
    for (int nty = first; nty <= first + 1 && nty <= a.ey; ++nty) {
      const int h = (a.ey + nty - 1) / nty;
      f(w, h, (a.ex + w - 1) / w, (a.ey + h - 1) / h);
    }
  }
}

// Tiles and z chunks of the block: the split with the least estimated time,
// rounds of the device's workgroup slots (one per CU) times the planes each
// workgroup collides times the time of a plane. A plane's time grows with the
// 128-byte lines its gathers touch (per row and direction the tile's own, and
// one for each side of the ring) and with its threads; the weights were
// fitted to 25 blocks of 40^2 x 400 to 256^3 cells with 10 to 60 splits
// each, where the split chosen takes 1.02 times the best one's time in the
// mean (1.14 at worst). Rows of 256 slots and more start on line boundaries:
// their tiles do too.
flb::MarchArgs plan(const KArgs& a, int elem, int cus) {
  flb::MarchArgs best{};
  double best_cost = 1e300;
  each_tile(a, elem, [&](int w, int h, int ntx, int nty) {
    const double plane = plane_time(w, h, ntx, elem);
    const int64_t tiles = int64_t(ntx) * nty;
    for (int rounds = 1; rounds <= 4; ++rounds) {
      const int64_t chunks = std::min<int64_t>(std::max<int64_t>(1, int64_t(rounds) * cus / tiles), a.ez);
      const int zc = int((a.ez + chunks - 1) / chunks), nz = (a.ez + zc - 1) / zc;
      const double cost = double((tiles * nz + cus - 1) / cus) * (zc + 2) * plane;
      if (cost < best_cost) {
        best_cost = cost;
        best.w = w;
        best.h = h;
        best.ntx = ntx;
        best.nty = nty;
        best.zchunk = zc;
        best.nz = nz;
      }
    }
  });
  return best;
}

// The flags and the dynamics of the block's updated cells when one dynamics
// that the march is built for serves them all.
bool one_dynamics(const flb_block_s* b, flb::MarchArgs* m) {
  m->mask = 0;
  for (int t = 0; t < b->ntasks; ++t) {
    const flb_task& k = b->tasks[t];
    if (k.dynamics != b->tasks[0].dynamics || k.smagorinsky != b->tasks[0].smagorinsky) return false;
    m->mask |= k.mask;
  }
  if (!m->mask) return false;
  m->dyn = b->tasks[0].dynamics;
  m->cs = b->tasks[0].smagorinsky;
  return m->dyn == FLB_DYN_BGK || m->dyn == FLB_DYN_BGK_FORCE || m->dyn == FLB_DYN_SMAG_MRT;
}

// Whether the block's links are closed (flb_block_s::closed).
int check_closed(flb_block_s* b, const KArgs& a, unsigned mask) {
  if (b->closed >= 0) return FLB_OK;
  uint32_t* open = reinterpret_cast<uint32_t*>(b->d_red);
  uint32_t h = 1;
  HIP_TRY(hipMemsetAsync(open, 0, sizeof h, b->stream));
  HIP_TRY(flb::launch_open_links(a, mask, open, b->stream));
  HIP_TRY(hipMemcpyAsync(&h, open, sizeof h, hipMemcpyDeviceToHost, b->stream));
  HIP_TRY(hipStreamSynchronize(b->stream));
  b->closed = h == 0 ? 1 : 0;
  return FLB_OK;
}

}  // namespace

// Dynamics, layout and walls; not in a capture (the first check of a block
// waits for the device).
int march_form(flb_block_s* b, flb::MarchArgs* m, bool* ok) {
  *ok = false;
  *m = flb::MarchArgs{};
  if (!b->flags_set || b->desc.q != FLB_D3Q19 || b->elem < 4 || b->ghost_overlap || b->vec != 0 || !one_dynamics(b, m))
    return FLB_OK;
  int rc = ensure_links(b);
  if (rc) return rc;
  const KArgs a = make_args(b);
  if (a.ez < 4) return FLB_OK;
  // the kernel's offsets, from the start of the allocation (periodic blocks)
  // or of a tile's first row, stay below 2 GiB
  const uint64_t tile = uint64_t(flb::march_threads(b->elem)) / 3 * uint64_t(b->ypop);
  const uint64_t span = 3 * uint64_t(b->zpop) + 37 * uint64_t(b->dpop) + tile;
  const bool per = a.px || a.py || a.pz;
  if ((per ? a.pop_total + 37 * uint64_t(b->dpop) * b->elem : span * b->elem) >= (uint64_t(1) << 31)) return FLB_OK;
  if (!per && !a.buf) return FLB_OK;
  rc = check_closed(b, a, m->mask);
  *ok = rc == FLB_OK && b->closed == 1;
  return rc;
}

double march_tiles(const KArgs& a, int elem, int zchunk, flb::MarchArgs* m) {
  double best = 1e300, plane = 0.0;
  each_tile(a, elem, [&](int w, int h, int ntx, int nty) {
    const double t = plane_time(w, h, ntx, elem), cost = t * ntx * nty;
    if (cost < best) {
      best = cost;
      plane = t;
      m->w = w;
      m->h = h;
      m->ntx = ntx;
      m->nty = nty;
    }
  });
  m->nz = (a.ez + zchunk - 1) / zchunk;
  m->zchunk = (a.ez + m->nz - 1) / m->nz;
  m->nz = (a.ez + m->zchunk - 1) / m->zchunk;
  return plane * (m->zchunk + 2);
}

// Second arrays take at most a sixteenth of the device's memory and leave
// half of it free.
bool march_fits(size_t bytes) {
  size_t free_b = 0, total = 0;
  return hipMemGetInfo(&free_b, &total) == hipSuccess && bytes <= total / 16 && free_b >= total / 2 + bytes;
}

bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return st != hipStreamCaptureStatusNone;
}

// The second array is taken at the first run of steps and kept with the block
// (so a captured run stays valid while the block lives). It is scratch: runs
// begin and end in d_pops. Blocks do without it, and step singly, where it
// does not fit (march_fits), and in a capture that comes before the first run.
bool march_ready(flb_block_s* b) {
  if (!b->flags_set || b->march == 0) return false;
  if (b->march == 1 && (b->nbc == 0 || !b->links_dirty) && b->d_alt) return true;
  if (capturing(b->stream)) return false;
  if (b->march < 0) {
    flb::MarchArgs m;
    bool ok = false;
    const int64_t cells = int64_t(axis_ext(b, 0)) * axis_ext(b, 1) * axis_ext(b, 2);
    if (size_t(19 * cells) * b->elem >= kMarchMinBytes && march_form(b, &m, &ok) != FLB_OK) return false;
    b->march = ok ? 1 : 0;
    if (!ok) return false;
  }
  if (ensure_links(b) != FLB_OK) return false;
  if (!b->d_alt) {
    const size_t bytes = size_t(b->pop_elems) * b->elem;
    if (!march_fits(bytes)) return false;
    if (hipMalloc(&b->d_alt, bytes) != hipSuccess) {
      (void)hipGetLastError();
      b->d_alt = nullptr;
      return false;
    }
  }
  return true;
}

int march_run(flb_block_s* b, int n) {
  int cus = 0;
  HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, b->device));
  KArgs a = make_args(b);
  flb::MarchArgs m = plan(a, int(b->elem), cus);
  one_dynamics(b, &m);
  char* const pops = static_cast<char*>(b->d_pops) + flb::kFrontPad * b->elem;
  char* const alt = static_cast<char*>(b->d_alt) + flb::kFrontPad * b->elem;
  for (int k = 0; k < n; k += 2) {
    a.pops = k % 4 == 0 ? pops : alt;
    m.dst = k % 4 == 0 ? alt : pops;
    HIP_TRY(b->elem == 8 ? flb::launch_march_f64(a, m, b->stream) : flb::launch_march_f32(a, m, b->stream));
  }
  return FLB_OK;
}

}  // namespace flbh
