// Host-side internals shared by the C-ABI translation units: the block
// object behind flb_block and the helpers that build kernel arguments.
#pragma once

#include <hip/hip_runtime.h>
#include <rocprofiler-sdk-roctx/roctx.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/flb_abi.h"
#include "flb_internal.hpp"

namespace flbh {

// The second population array of a block's or a batch's two-step runs: scratch
// between calls. The library gives those of other objects back where it runs
// out of device memory (dev_alloc); a later run takes one again if it fits.
struct Twin {
  char* p = nullptr;
  int device = 0;
  hipStream_t stream = nullptr;  // of the runs that use it
  int users = 0;                 // runs being enqueued now
  bool held = false;             // a capture recorded it: it stays while its owner lives
};
// Takes the array, if there is none, where march_fits allows it.
bool twin_take(Twin& t, size_t bytes, int device, hipStream_t s);
void twin_drop(Twin& t);
// Keeps the array, if there is one, from being given back while it lives.
struct TwinUse {
  Twin& t;
  explicit TwinUse(Twin& twin);
  ~TwinUse();
  TwinUse(const TwinUse&) = delete;
  TwinUse& operator=(const TwinUse&) = delete;
};
// hipMalloc; out of memory, once more after second arrays were given back. A
// failure leaves *p null and no error for the next launch's check to find.
hipError_t dev_alloc(void** p, size_t bytes);
template <class T>
hipError_t dev_alloc(T** p, size_t bytes) {
  return dev_alloc(reinterpret_cast<void**>(p), bytes);
}

}  // namespace flbh

struct flb_block_s {
  int device = 0;
  hipStream_t stream = nullptr;
  flb_block_desc desc{};
  int d = 3;
  int64_t N = 0;        // host cells nx*ny*nz
  int64_t stride = 0;   // slots between two per-cell arrays (pads included)
  int pitch = 0;        // slots per row
  int64_t plane = 0;    // slots per plane
  int64_t dpop = 0, zpop = 0;  // population strides (see flb_internal.hpp)
  int ypop = 0;
  int64_t pop_elems = 0;       // elements allocated for the populations
  size_t elem = 4;   // bytes per stored population
  size_t real = 4;   // bytes of the compute type
  void* d_pops = nullptr;
  uint8_t* d_flags = nullptr;
  void* d_rho = nullptr;
  void* d_u = nullptr;
  double* d_partials = nullptr;
  double* d_red = nullptr;
  void* d_stage = nullptr;
  size_t stage_bytes = 0;
  std::vector<uint8_t> h_flags;
  bool flags_set = false;
  flb_task tasks[flb::kMaxTasks]{};
  int ntasks = 0;
  flb_hwbc bcs[flb::kMaxBc]{};
  int nbc = 0;
  double rates[19]{};
  double force[3]{};
  int64_t step = 0;
  int parity = 0;
  int pending = 0;  // 1: cell dynamics applied, stream not yet called
  // refinement level of the block and the hierarchy's finest level: the
  // count-gated calls step the block when count % 2^(max_level - level) == 0
  int level = 0, max_level = 0;
  int watchdog = 0;  // flb_step checks mass / momentum every `watchdog` steps (0: off)
  int vec = 0;  // step kernel form: 0 automatic cell form, -1 row segments, -3 linear runs,
                // 1/2/4 row form with that many cells per thread
  int wpb = 4;   // wavefronts per workgroup
  flbh::Twin twin;         // second population array of the two-step march (flb_march.hip)
  int march = -1;          // 1: the march may step the block, 0: not, -1: to be checked (flags, tasks or walls changed)
  flb::MarchArgs tiles{};  // its tiles, planned once (ntx 0: not yet), and their estimated time
  double tiles_cost = 0.0;
  int closed = -1;         // 1: no link of an updated cell leads to a cell that is not updated but wall links, 0, -1 likewise
  bool retained = false;   // holds the read-out buffers (readout_retain)
  int64_t paths[FLB_PATHS] = {};  // flb_block_paths
  uint64_t version = 0;  // bumped by every change a batch table must see
  uint64_t* d_links = nullptr;  // precomputed halfway wall links (slot layout)
  bool links_dirty = true;      // flags or halfway managers changed since d_links was built
  bool ghost_overlap = false;   // the overlap layer mirrors neighbouring blocks (flb_halo)
  void* d_rho_old = nullptr;    // RhoOld / UOld of the convergence residual (field slot layout)
  void* d_u_old = nullptr;
  unsigned long long* d_res = nullptr;  // residual as the bits of a non-negative double
  // Coupled lattices (flb_share_velocity, flb_add_buoyancy). A scalar block
  // advects with vel_src's VELOCITY field; a flow block's DYN_BGK_SCALAR_FORCE
  // cells take the buoyancy of each entry of buoy. users lists the blocks that
  // hold a reference to this one, so destroying either side detaches it.
  struct Buoyancy {
    flb_block src;
    uint8_t mask;
    double gbeta, rho0;
  };
  flb_block vel_src = nullptr;
  std::vector<Buoyancy> buoy;
  std::vector<flb_block> users;
};

struct flb_halo_s {
  int device = 0;
  hipStream_t stream = nullptr;
  std::vector<flb_block> blocks;
  std::vector<uint64_t> versions;
  int q = 19;
  size_t elem = 4;
  std::vector<flb::KArgs> h_tab;
  std::vector<flb::HaloItem> h_items;
  int64_t cells = 0;  // of all items
  unsigned wgs = 0;
  flb::KArgs* d_tab = nullptr;
  flb::HaloItem* d_items = nullptr;
  flb::HaloWg* d_wg = nullptr;
};

namespace flbh {

using flb::KArgs;

// Records the message for flb_last_error() (thread-local) and returns code.
int fail(int code, const char* fmt, ...);

#define HIP_TRY(expr)                                                                 \
  do {                                                                                \
    hipError_t e_ = (expr);                                                           \
    if (e_ != hipSuccess)                                                             \
      return fail(FLB_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(e_));        \
  } while (0)

// A roctx range over a host call (its kernels and waits show under it in
// rocprofv3 traces with --marker-trace; a no-op without a profiler).
struct Range {
  explicit Range(const char* name) { roctxRangePushA(name); }
  ~Range() { roctxRangePop(); }
  Range(const Range&) = delete;
  Range& operator=(const Range&) = delete;
};

struct DeviceGuard {
  int prev = -1;
  explicit DeviceGuard(int dev) {
    if (hipGetDevice(&prev) == hipSuccess && prev != dev) {
      (void)hipSetDevice(dev);
    } else {
      prev = -1;
    }
  }
  ~DeviceGuard() {
    if (prev >= 0) (void)hipSetDevice(prev);
  }
};

KArgs make_args(const flb_block_s* b);
int axis_ext(const flb_block_s* b, int ax);
uint32_t buffer_form_ok(const KArgs& a, int elem, int dims);
// Copies the first n of `have` counts to out; FLB_ERR_ARG for a bad n or a null out.
int copy_paths(const int64_t* from, int have, int64_t* out, int n);
// True when a count-gated call acts on a block of `level` in a hierarchy whose
// finest level is max_level (BlockLatticeManager's 2^(maxlevel - level) rule).
inline bool level_due(int64_t count, int level, int max_level) {
  return count % (int64_t(1) << (max_level - level)) == 0;
}
// Builds the block's wall-link words when flags or halfway managers changed
// (enqueued on the block's stream); a no-op without halfway managers.
int ensure_links(flb_block_s* b);

// Two steps per pass (flb_march.hip): march_ready tells whether a run of
// steps of the block may take it now, march_run advances a block at parity 1
// by n steps (a multiple of 4).
bool march_ready(flb_block_s* b);
int march_run(flb_block_s* b, int n);
// Bytes of populations from which on a block takes it; smaller ones run out of
// the caches. BGK over 110 blocks of 34 MB to 300 MB: 0.95 to 1.06 times the
// single steps' time up to 43 MB, 0.78 to 0.92 beyond. MRT with LES is bound by
// its instructions, those of the ring's cells included: FP32 takes single
// steps (1.0 to 1.4 times their time in the march up to 256^3), FP64 marches
// from 400 MB on (140^3 180 -> 156 us, 200x160x150 303 -> 261; below 320 MB 1.0
// to 1.5 times). In batches, whose single steps run at 4.5 TB/s, both take it
// from there on (40 blocks of 481 MB: 234 -> 197 us), all blocks counted.
//
// In between lies a band where single steps, on one array, still run out of
// the 256 MB memory-side cache and the march, on two, no longer does
// (march_pays for a block). Batches behave as blocks of split rows do: BGK FP32
// 158 to 218 MiB, FP64 150 to 230, with a force from 140 and 135 on (1.0 to
// 1.16 times the single steps' time in it, 0.9 to 0.97 just outside).
constexpr size_t kMarchMinBytes = size_t(42) << 20;
inline bool batch_march_pays(int dyn, size_t elem, size_t bytes) {
  if (dyn == FLB_DYN_SMAG_MRT) return bytes >= size_t(400) * 1000 * 1000;
  const size_t mib = bytes >> 20;
  const bool f64 = elem == 8, force = dyn == FLB_DYN_BGK_FORCE;
  const size_t lo = force ? (f64 ? 135 : 140) : (f64 ? 150 : 158), hi = f64 ? 230 : 218;
  return bytes >= kMarchMinBytes && !(mib >= lo && mib < hi);
}
// The rows of one block, its periodic axes, and march_plan's estimate.
struct MarchRows {
  int ex, pitch;
  bool split;  // into tiles
  bool px, per, all;  // x periodic, any axis, every axis
  double cost;
};
bool march_pays(int dyn, size_t elem, size_t bytes, const MarchRows& rows);
// march_form sets *ok where a block of any size is of the form the march
// takes, with its flags and dynamics in m (not its tiles). march_plan: tiles
// of one box of cells (rows of `pitch` slots) for
// workgroups of `threads`; march_plan_batch: those of
// several in one launch and the order of its workgroups, returns the estimated
// time of a pass in units of 0.75 to 0.94 us. march_fits: whether second
// arrays of `bytes` leave the device enough memory.
struct MarchBox {
  int ex, ey, ez, pitch;
  bool operator==(const MarchBox& o) const { return ex == o.ex && ey == o.ey && ez == o.ez && pitch == o.pitch; }
};
int march_form(flb_block_s* b, flb::MarchArgs* m, bool* ok);
flb::MarchArgs march_plan(const MarchBox& box, int elem, int cus, int threads, double* cost = nullptr);
double march_plan_batch(const std::vector<MarchBox>& boxes, int elem, int cus, int threads,
                        std::vector<flb::MarchArgs>& mt, std::vector<flb::MarchWg>& wgs);
bool march_fits(size_t bytes);
bool capturing(hipStream_t s);

// Read-out to host memory (flb_readout.hip). readout: bytes of device memory
// to the caller's array once the work enqueued on s is done, or several arrays
// at once; widen: FP32 on the device, FP64 at the caller. Each block and
// adjoint box retains the pinned buffers while it lives.
struct ReadPart {
  void* host;
  const void* dev;
  size_t bytes;  // on the device
};
void readout_retain();
void readout_release();
hipError_t readout(void* host, const void* dev, size_t bytes, bool widen, hipStream_t s);
hipError_t readout(const ReadPart* parts, size_t n, bool widen, hipStream_t s);
constexpr size_t kDirect = size_t(256) << 10;
struct DirectOut {
  void* ptr = nullptr;
  explicit DirectOut(size_t bytes);
  ~DirectOut();
  DirectOut(const DirectOut&) = delete;
  DirectOut& operator=(const DirectOut&) = delete;
};

// Block halo (flb_halo.hip): enqueue the exchange that follows a step leaving
// the blocks at `parity`; refresh the device copy of the blocks' arguments;
// the common parity of the blocks.
hipError_t halo_launch(const flb_halo_s* h, int parity, hipStream_t s);
int halo_refresh(flb_halo_s* h);
int halo_parity(const flb_halo_s* h, int* parity);
// True when rows of ex cells fill less than 90 % of their wavefronts' lanes.
bool linear_form(int ex);
int family_of(const flb_block_s* b);

}  // namespace flbh

#define CHECK_BLOCK(b) \
  if (!(b)) return fail(FLB_ERR_ARG, "null block handle")
