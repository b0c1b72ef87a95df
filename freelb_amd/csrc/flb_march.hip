// Host side of the two-step march (flb_march.hpp): which blocks take it, the
// tiles of a block, and the passes of a run of steps.

#include <hip/hip_runtime.h>

#include <algorithm>

#include "flb_host.hpp"
#include "flb_internal.hpp"

namespace flbh {

namespace {

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
  const int threads = flb::march_threads(size_t(elem)), line = 128 / elem;
  for (int n = 1; n <= a.ex; ++n) {
    int w = (a.ex + n - 1) / n;
    if (a.pitch >= 256) w = (w + line - 1) / line * line;
    if (w + 2 > flb::kMarchMaxRow) continue;
    if (w < 8 && n > 1) break;
    const int ntx = (a.ex + w - 1) / w, hmax = std::min(a.ey, threads / (w + 2) - 2);
    for (int nty = (a.ey + hmax - 1) / hmax; nty <= (a.ey + hmax - 1) / hmax + 1 && nty <= a.ey; ++nty) {
      const int h = (a.ey + nty - 1) / nty;
      const double reads = (h + 2) * (double(w) / line + (ntx > 1 ? 2.0 : 1.0));
      const double plane = 2.0 + 0.06 * reads + 0.005 * double((w + 2) * (h + 2)) * (elem == 8 ? 2.0 : 1.0);
      const int64_t tiles = int64_t(ntx) * ((a.ey + h - 1) / h);
      for (int rounds = 1; rounds <= 4; ++rounds) {
        const int64_t chunks = std::max<int64_t>(1, int64_t(rounds) * cus / tiles);
        const int zc = int((a.ez + std::min<int64_t>(chunks, a.ez) - 1) / std::min<int64_t>(chunks, a.ez));
        const int nz = (a.ez + zc - 1) / zc;
        const double cost = double((tiles * nz + cus - 1) / cus) * (zc + 2) * plane;
        if (cost < best_cost) {
          best_cost = cost;
          best.w = w;
          best.h = h;
          best.ntx = ntx;
          best.nty = (a.ey + h - 1) / h;
          best.zchunk = zc;
          best.nz = nz;
        }
      }
    }
  }
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

// Populations of 32 MiB and more, what the eight L2 caches hold together: the
// one-step kernels run smaller blocks out of the caches (FP32 64^3: 8.8 us a
// step against 9.8 us here, 80^3: 15.9 against 13.8; FP64 32^3: 5.7 against
// 7.7, 64^3: 15.3 against 14.4).
constexpr size_t kMarchMinBytes = size_t(32) << 20;

// Whether the block's dynamics, layout and walls are those the march takes.
int check_block(flb_block_s* b, bool* ok) {
  *ok = false;
  flb::MarchArgs m{};
  if (b->desc.q != FLB_D3Q19 || b->elem < 4 || b->ghost_overlap || b->vec != 0 || !one_dynamics(b, &m)) return FLB_OK;
  const KArgs a = make_args(b);
  if (a.ez < 4 || size_t(19) * size_t(a.ex) * size_t(a.ey) * size_t(a.ez) * b->elem < kMarchMinBytes) return FLB_OK;
  // the kernel's offsets, from the start of the allocation (periodic blocks)
  // or of a tile's first row, stay below 2 GiB
  const uint64_t tile = uint64_t(flb::march_threads(b->elem)) / 3 * uint64_t(b->ypop);
  const uint64_t span = 3 * uint64_t(b->zpop) + 37 * uint64_t(b->dpop) + tile;
  const bool per = a.px || a.py || a.pz;
  if ((per ? a.pop_total + 37 * uint64_t(b->dpop) * b->elem : span * b->elem) >= (uint64_t(1) << 31)) return FLB_OK;
  if (!per && !a.buf) return FLB_OK;
  uint32_t* open = reinterpret_cast<uint32_t*>(b->d_red);
  uint32_t h = 1;
  HIP_TRY(hipMemsetAsync(open, 0, sizeof h, b->stream));
  HIP_TRY(flb::launch_open_links(a, m.mask, open, b->stream));
  HIP_TRY(hipMemcpyAsync(&h, open, sizeof h, hipMemcpyDeviceToHost, b->stream));
  HIP_TRY(hipStreamSynchronize(b->stream));
  *ok = h == 0;
  return FLB_OK;
}

bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return st != hipStreamCaptureStatusNone;
}

}  // namespace

// The second array is taken at the first run of steps and kept with the block
// (so a captured run stays valid while the block lives). It is scratch: runs
// begin and end in d_pops. Blocks do without it, and step singly, where it
// would take more than a sixteenth of the device's memory or leave less than
// half of it free, and in a capture that comes before the first run.
bool march_ready(flb_block_s* b) {
  if (!b->flags_set || b->march == 0) return false;
  if (b->march == 1 && (b->nbc == 0 || !b->links_dirty) && b->d_alt) return true;
  if (capturing(b->stream)) return false;
  if (ensure_links(b) != FLB_OK) return false;
  if (b->march < 0) {
    bool ok = false;
    if (check_block(b, &ok) != FLB_OK) return false;
    b->march = ok ? 1 : 0;
    if (!ok) return false;
  }
  if (!b->d_alt) {
    size_t free_b = 0, total = 0;
    const size_t bytes = size_t(b->pop_elems) * b->elem;
    if (hipMemGetInfo(&free_b, &total) != hipSuccess || bytes > total / 16 || free_b < total / 2 + bytes) return false;
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
