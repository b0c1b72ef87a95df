// Host side of the two-step march (flb_march.hpp): which blocks take it, the
// tiles of a block, and the passes of a run of steps.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <functional>
#include <mutex>
#include <queue>
#include <utility>
#include <vector>

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
void each_tile(const MarchBox& a, int elem, int threads, F&& f) {
  const int line = 128 / elem, least = a.pitch >= 256 ? line : 8;
  for (int n = 1, last = 0; n <= a.ex && last != line; ++n) {
    int w = (a.ex + n - 1) / n;
    if (a.pitch >= 256) w = (w + line - 1) / line * line;
    if (w + 2 > flb::kMarchMaxRow || w == last) continue;
    if (w < least && n > 1) break;
    if (a.pitch >= 256) last = w;
    const int hmax = std::min(a.ey, threads / (w + 2) - 2), first = (a.ey + hmax - 1) / hmax;
    for (int nty = first; nty <= first + 1 && nty <= a.ey; ++nty) {
      const int h = (a.ey + nty - 1) / nty;
      f(w, h, (a.ex + w - 1) / w, (a.ey + h - 1) / h);
    }
  }
}

}  // namespace

// Tiles and z chunks of the block: the split with the least estimated time,
// rounds of the device's workgroup slots (one per CU) times the planes each
// workgroup collides times the time of a plane. A plane's time grows with the
// 128-byte lines its gathers touch (per row and direction the tile's own, and
// one for each side of the ring) and with its threads; the weights were
// fitted to 25 blocks of 40^2 x 400 to 256^3 cells with 10 to 60 splits
// each, where the split chosen takes 1.02 times the best one's time in the
// mean (1.14 at worst). Rows of 256 slots and more start on line boundaries:
// their tiles do too. Made once per block or box, as a run may be four steps:
// in each run, and with every aligned width tried over and over, it cost 36 us
// at 256^3 and 140 us at 1000x60x12 (1 us in the mean now).
flb::MarchArgs march_plan(const MarchBox& a, int elem, int cus, int threads, double* cost_out) {
  flb::MarchArgs best{};
  double best_cost = 1e300;
  each_tile(a, elem, threads, [&](int w, int h, int ntx, int nty) {
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
  if (cost_out) *cost_out = best_cost;
  return best;
}

namespace {

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

namespace {

// Tiles of at most zchunk planes for a box of a batch; returns the estimated
// time of one of its workgroups.
double march_tiles(const MarchBox& a, int elem, int threads, int zchunk, flb::MarchArgs* m) {
  double best = 1e300, plane = 0.0;
  each_tile(a, elem, threads, [&](int w, int h, int ntx, int nty) {
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

// The last end of work given longest first to the device's workgroup slots
// (one per CU); `work` holds estimated times and how many workgroups take
// them, longest first. Long lists end evenly.
double march_span(const std::vector<std::pair<double, int64_t>>& work, int cus) {
  double total = 0.0;
  int64_t wgs = 0;
  for (const auto& w : work) {
    total += w.first * double(w.second);
    wgs += w.second;
  }
  if (wgs > int64_t(16) * cus) return total / cus + 0.5 * work.front().first;
  std::priority_queue<double, std::vector<double>, std::greater<double>> ends;
  for (int k = 0; k < cus; ++k) ends.push(0.0);
  double span = 0.0;
  for (const auto& w : work)
    for (int64_t k = 0; k < w.second; ++k) {
      const double e = ends.top() + w.first;
      ends.pop();
      ends.push(e);
      span = std::max(span, e);
    }
  return span;
}

}  // namespace

// Tiles of every box and the order of all workgroups, for the chunk length
// with the least estimated time. The order is longest workgroup first, so the
// uneven end of a launch is one of the short ones.
double march_plan_batch(const std::vector<MarchBox>& boxes, int elem, int cus, int threads, std::vector<flb::MarchArgs>& mt,
                        std::vector<flb::MarchWg>& wgs) {
  const size_t nb = boxes.size();
  mt.assign(nb, flb::MarchArgs{});
  double best_span = 1e300;
  int best = 8;
  std::vector<double> one(nb);
  std::vector<size_t> order(nb);
  const auto tiles = [&](int len) {
    for (size_t k = 0; k < nb; ++k) {
      one[k] = march_tiles(boxes[k], elem, threads, len, &mt[k]);
      order[k] = k;
    }
    std::sort(order.begin(), order.end(), [&](size_t x, size_t y) { return one[x] > one[y] || (one[x] == one[y] && x < y); });
  };
  std::vector<std::pair<double, int64_t>> work;
  for (int len : {4, 6, 8, 10, 12, 14, 16, 20, 24, 28, 32, 40, 48, 64, 96}) {
    tiles(len);
    work.clear();
    for (size_t k : order) work.emplace_back(one[k], int64_t(mt[k].ntx) * mt[k].nty * mt[k].nz);
    const double span = march_span(work, cus);
    if (span < best_span) {
      best_span = span;
      best = len;
    }
  }
  tiles(best);
  wgs.clear();
  for (size_t k : order) {
    const int n = mt[k].ntx * mt[k].nty * mt[k].nz;
    for (int w = 0; w < n; ++w) wgs.push_back({int(k), w});
  }
  return best_span;
}

// Whether one block marches: from 42 MiB on (kMarchMinBytes), but not where
// single steps gain more from the memory-side cache. Lines drawn by march and
// single steps of 2700 blocks of 44 to 266 MiB, BGK and with a force, FP32 and
// FP64, rows of 12 to 1000 cells, walled and periodic in x, in y and z and in
// all (times of the march over single steps):
// - rows of less than 256 slots: FP32 loses from 160 MiB (periodic in x only or
//   also in one more axis, where single steps lose least: 142) to 215 where rows
//   are split or have at most 64 cells (1.0 to 1.19), from 165 and only if so
//   periodic where a tile holds rows of 65 to 128 (1.02 to 1.07); with a force
//   from 140 (x periodic 122) to 222 (1.0 to 1.23). Rows of at most 24 cells,
//   whose rings are widest, lose with a force and x periodic at any smaller
//   size too (0.96 to 1.16). FP64 from 160 (split rows 180) to 212 (228), with a
//   force from 132 (1.0 to 1.23). Below these bands 0.72 to 1.0, above 0.65 to
//   0.97.
// - rows of 256 slots and more hold a quarter to half of padding, which fills
//   the cache for single steps as well: BGK 0.64 to 0.98 throughout, also with
//   a force where rows leave a tenth of their wavefronts' lanes idle (230, 400
//   cells: 0.72 to 0.99) and on walled boxes. Periodic ones with a force and
//   fuller rows lose from 120 to 270 MiB in FP32 (1.0 to 1.13; all axes 140 to
//   205, to 1.07), from 145 to 230 in FP64, not with all axes (0.8 to 1.0). Thin
//   boxes whose tiles fit badly (700x20 FP64, 1000x30x21: 1.02 to 1.28) are told
//   by the estimate per MiB.
// On 330 other blocks of 43 to 285 MiB, drawn over the same ranges, blocks take
// 0.902 of their single steps' time in the mean so (0.913 if all marched, 0.900
// the better of both for each), the worst march 1.07.
bool march_pays(int dyn, size_t elem, size_t bytes, const MarchRows& r) {
  const bool f64 = elem == 8, force = dyn == FLB_DYN_BGK_FORCE;
  if (dyn == FLB_DYN_SMAG_MRT) return f64 && bytes >= size_t(400) * 1000 * 1000;
  if (bytes < kMarchMinBytes) return false;
  const size_t mib = bytes >> 20;
  size_t lo = 0, hi = 0;
  if (r.pitch >= 256) {
    if (!linear_form(r.ex) && force) {
      if (mib < 56 && r.cost >= 1.25 * double(mib)) return false;
      if (r.per && !r.all) {
        lo = f64 ? 145 : 120;
        hi = f64 ? 230 : 270;
      } else if (r.all && !f64) {
        lo = 140;
        hi = 205;
      }
    }
    if (f64 && mib >= 125 && r.cost >= (mib < 210 ? 1.0 : 0.94) * double(mib)) return false;
  } else if (f64) {
    lo = force ? 132 : (r.split ? 180 : 160);
    hi = r.split ? 228 : 212;
  } else if (force) {
    lo = !r.px ? 140 : (r.ex <= 24 ? 0 : 122);
    hi = 222;
  } else if (r.split || r.ex <= 64) {
    lo = r.px && !r.all ? 142 : 160;
    hi = 215;
  } else if (r.px && !r.all) {
    lo = 165;
    hi = 215;
  }
  if (r.ex < 16 && !f64) hi = std::min<size_t>(hi, 195);  // their padding ends the band earlier
  return !(mib >= lo && mib < hi);
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

namespace {

// Every second array there is; mu guards the list and the arrays' fields.
struct Twins {
  std::mutex mu;
  std::vector<Twin*> list;
};
Twins& twins() {
  static Twins* t = new Twins();  // never destroyed: blocks may outlive static objects
  return *t;
}

// Frees the second arrays of the current device that no run is using and no
// capture has recorded; true if there was one.
bool twins_give_back() {
  Twins& all = twins();
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  std::lock_guard<std::mutex> l(all.mu);
  bool any = false;
  for (size_t k = all.list.size(); k-- > 0;) {
    Twin& t = *all.list[k];
    if (t.users > 0 || t.held || t.device != dev || capturing(t.stream)) continue;
    if (hipStreamSynchronize(t.stream) != hipSuccess || hipFree(t.p) != hipSuccess) continue;
    t.p = nullptr;
    all.list.erase(all.list.begin() + std::ptrdiff_t(k));
    any = true;
  }
  return any;
}

}  // namespace

bool twin_take(Twin& t, size_t bytes, int device, hipStream_t s) {
  Twins& all = twins();
  std::lock_guard<std::mutex> l(all.mu);
  if (t.p) return true;
  if (!march_fits(bytes)) return false;
  if (hipMalloc(reinterpret_cast<void**>(&t.p), bytes) != hipSuccess) {
    (void)hipGetLastError();
    t.p = nullptr;
    return false;
  }
  t.device = device;
  t.stream = s;
  all.list.push_back(&t);
  return true;
}

void twin_drop(Twin& t) {
  Twins& all = twins();
  std::lock_guard<std::mutex> l(all.mu);
  if (!t.p) return;
  all.list.erase(std::find(all.list.begin(), all.list.end(), &t));
  (void)hipFree(t.p);
  t.p = nullptr;
}

TwinUse::TwinUse(Twin& twin) : t(twin) {
  std::lock_guard<std::mutex> l(twins().mu);
  ++t.users;
}
TwinUse::~TwinUse() {
  std::lock_guard<std::mutex> l(twins().mu);
  --t.users;
}

hipError_t dev_alloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    if (e == hipErrorOutOfMemory && twins_give_back()) e = hipMalloc(p, bytes);
  }
  if (e != hipSuccess) {
    (void)hipGetLastError();
    *p = nullptr;
  }
  return e;
}

// The second array is taken at the first run of steps and kept with the block
// until memory is short (twins_give_back; one that a captured run holds, while
// the block lives). It is scratch: runs begin and end in d_pops. Blocks do
// without it, and step singly, where it does not fit (march_fits), and in a
// capture that comes before the first run. The caller holds a TwinUse.
bool march_ready(flb_block_s* b) {
  if (!b->flags_set || b->march == 0) return false;
  if (b->march == 1 && (b->nbc == 0 || !b->links_dirty) && b->twin.p) return true;
  if (capturing(b->stream)) return false;
  if (b->march < 0) {
    flb::MarchArgs m;
    bool ok = false;
    const int64_t cells = int64_t(axis_ext(b, 0)) * axis_ext(b, 1) * axis_ext(b, 2);
    const size_t bytes = size_t(19 * cells) * b->elem;
    if (bytes >= kMarchMinBytes && march_form(b, &m, &ok) != FLB_OK) return false;
    if (ok) {
      const KArgs a = make_args(b);
      if (b->tiles.ntx == 0) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, b->device) != hipSuccess) return false;
        b->tiles = march_plan({a.ex, a.ey, a.ez, a.pitch}, int(b->elem), cus, flb::march_threads(b->elem),
                              &b->tiles_cost);
        b->paths[FLB_PATH_PLANS] += 1;
      }
      ok = march_pays(m.dyn, b->elem, bytes, {a.ex, a.pitch, b->tiles.ntx > 1, a.px != 0, a.px || a.py || a.pz,
                                              a.px && a.py && a.pz, b->tiles_cost});
    }
    b->march = ok ? 1 : 0;
    if (!ok) return false;
  }
  if (ensure_links(b) != FLB_OK) return false;
  return twin_take(b->twin, size_t(b->pop_elems) * b->elem, b->device, b->stream);
}

int march_run(flb_block_s* b, int n) {
  KArgs a = make_args(b);
  flb::MarchArgs m = b->tiles;
  one_dynamics(b, &m);
  char* const pops = static_cast<char*>(b->d_pops) + flb::kFrontPad * b->elem;
  char* const alt = b->twin.p + flb::kFrontPad * b->elem;
  b->twin.held = b->twin.held || capturing(b->stream);
  for (int k = 0; k < n; k += 2) {
    a.pops = k % 4 == 0 ? pops : alt;
    m.dst = k % 4 == 0 ? alt : pops;
    HIP_TRY(b->elem == 8 ? flb::launch_march_f64(a, m, b->stream) : flb::launch_march_f32(a, m, b->stream));
  }
  return FLB_OK;
}

}  // namespace flbh
