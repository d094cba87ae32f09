// C ABI of librhllc_hip.so (declarations and the reference interfaces each
// entry point replaces: include/rhllc_hip.h).
//
// A handle owns the mesh and state in device memory (SoA, Hilbert-relabelled
// when asked), one HIP stream, and optionally a captured hipGraph of the step.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "../../../include/rhllc_hip.h"
#include "../mesh/mesh_common.h"
#include "mlp_internal.h"
#include "rhllc_internal.h"
#include "flux_ext.h"
#include "rhllc_layout.h"
#include "rhllc_records.h"

using namespace rhllc_dev;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg) {
  g_err = msg;
  return code;
}
int hip_fail(hipError_t e, const char *what) {
  return fail(RHLLC_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

#define HIP_TRY(expr)                                   \
  do {                                                  \
    hipError_t e_ = (expr);                             \
    if (e_ != hipSuccess) return hip_fail(e_, #expr);   \
  } while (0)

// Cells per tile of a handle's tiled step: 256, or 64 on a mesh too small to
// fill the chip.  A workgroup of 256 threads takes a 64-cell tile's ~180 faces
// in one pass where a 256-cell tile needs three, so a step that waits for one
// workgroup's chain of loads and divides is shorter; but only one of its four
// waves has cells, and 37% of the faces are shared with another tile (23% at
// 256), so it loses once every CU has several workgroups.  With 256-cell tiles
// the time jumps wherever some CUs get a tile more than the others, at every
// whole round (one tile on each CU: 65,536 cells on 256 CUs); with 64 it grows
// more evenly, so just past a whole round 64 is ahead again, less each time.
// Time of a step with 64 cells over that with 256 on both sides of each line,
// least and most of an early and a developed blast and a shear layer on two
// numberings of a mesh:
//   FP64, rounds        .73      .77       .97   |   1.02     1.49 |    1.55      1.80   |   2.01     2.23 |    2.31      2.73
//     ideal           .88-.96  .94-1.05  .96-1.07| .92-.96  .94-.96|  .99-1.02 1.02-1.10 | .97-.99  .94-.96| .99-1.00  1.02-1.06
//     ideal, source   .91-.98  .95-1.02  .98-1.07| .94-.96  .97-1.0| 1.03-1.06 1.13-1.17 | .99-1.03 .98-1.0|1.01-1.03  1.13-1.15
//     TAUB            .95-.97 1.05-1.08 1.07-1.09| .92-.94  .94-.95| 1.01-1.03 1.07-1.10 | .97-.99  .92-.93| .97-.98  1.02-1.03
//   mixed, rounds      1.49      1.80      2.01      2.23     2.47   |   2.55      2.73      3.00
//     ideal           .90-.90  .99-1.01 1.02-1.05  .90-.92  .94-.95 |  .96-.99   .95-.99 1.04-1.07
//     ideal, source   .91-.94 1.03-1.06 1.03-1.06  .98-.99 1.02-1.04| 1.05-1.07 1.08-1.10 1.14-1.15
//     TAUB            .90-.91 1.01-1.04  .99-1.01  .90-.94  .94-.96 |  .97-.99   .97-.99 1.06-1.09
//     surrogate start .86-.91  .89-1.00  .90-1.02  .88-.93  .92-.94 |  .93-.97   .95-.98  .97-1.04
// (The source is not known yet when the tiles are made.)
int32_t tile_cells_for(int64_t n, bool mixed, int cus) {
  const double rounds = (double)n / ((double)cus * kTileCells);
  const bool small = mixed ? rounds <= 2.5
                           : rounds <= 0.75 || (rounds > 1.0 && rounds <= 1.5) || (rounds > 2.0 && rounds <= 2.25);
  return small ? kSmallTileCells : kTileCells;
}

}  // namespace

namespace rhllc_capi_detail {
int set_error(int code, const std::string &msg) { return fail(code, msg); }

// Compute units of a device (256, or fewer where the GPU is partitioned).
// Without a device 256: the calls after this one report that.
int compute_units(int32_t device) {
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && cus > 0) return cus;
  (void)hipGetLastError();
  return 256;
}
}  // namespace rhllc_capi_detail

// Two pinned chunks that the transfers of a handle go through in turn: the
// host fills (or drains) one while the device works on the other.  One thread
// uses a handle, and everything runs on its stream.
struct Staging {
  // Largest chunk: 8 MB take 150 us over the link, so a transfer of many is
  // pipelined and the launch and wait of each are small beside it.  A 480 MB
  // snapshot measured 15.0 ms with 1 MB chunks, 13.3 with 2, 10.5 with 4 and 8
  // and 9.5 with 16 (173 ms as whole-array copies and serial host loops).
  static constexpr size_t kMaxBytes = (size_t)8 << 20;
  uint8_t *host[2] = {nullptr, nullptr};
  void *dev[2] = {nullptr, nullptr};
  hipEvent_t done[2] = {nullptr, nullptr};
  bool busy[2] = {false, false};  // the device may still use the chunk (done records its end)
  size_t bytes = 0;

  hipError_t alloc(size_t want) {
    bytes = ((want < kMaxBytes ? want : kMaxBytes) + 63) & ~(size_t)63;
    for (int b = 0; b < 2; ++b) {
      hipError_t e = hipHostMalloc((void **)&host[b], bytes, hipHostMallocDefault);
      if (e == hipSuccess) e = hipHostGetDevicePointer(&dev[b], host[b], 0);
      if (e == hipSuccess) e = hipEventCreateWithFlags(&done[b], hipEventDisableTiming);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  ~Staging() {
    for (int b = 0; b < 2; ++b) {
      if (host[b]) (void)hipHostFree(host[b]);
      if (done[b]) (void)hipEventDestroy(done[b]);
    }
  }
  hipError_t wait(int b) {
    if (!busy[b]) return hipSuccess;
    busy[b] = false;
    return hipEventSynchronize(done[b]);
  }
  hipError_t mark(int b, hipStream_t s) {
    busy[b] = true;
    return hipEventRecord(done[b], s);
  }
  // n entries of `each` bytes to the device: fill(first, count, host chunk),
  // then launch(first, count, device address of the chunk).
  template <typename Fill, typename Launch>
  hipError_t send(int64_t n, size_t each, hipStream_t s, Fill fill, Launch launch) {
    const int64_t per = (int64_t)(bytes / each);
    int b = 0;
    for (int64_t i = 0; i < n; i += per, b ^= 1) {
      const int64_t c = n - i < per ? n - i : per;
      hipError_t e = wait(b);
      if (e == hipSuccess) fill(i, c, host[b]), e = launch((int)i, (int)c, dev[b]);
      if (e == hipSuccess) e = mark(b, s);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  // n entries of `each` bytes from the device: launch, then drain(first, count,
  // host chunk).  Everything queued on s before is done when it returns.
  template <typename Launch, typename Drain>
  hipError_t receive(int64_t n, size_t each, hipStream_t s, Launch launch, Drain drain) {
    const int64_t per = (int64_t)(bytes / each), chunks = (n + per - 1) / per;
    for (int64_t k = 0; k <= chunks; ++k) {
      if (k < chunks) {
        const int64_t i = k * per;
        hipError_t e = launch((int)i, (int)(n - i < per ? n - i : per), dev[k & 1]);
        if (e == hipSuccess) e = mark((int)(k & 1), s);
        if (e != hipSuccess) return e;
      }
      if (k > 0) {
        const int64_t i = (k - 1) * per;
        if (const hipError_t e = wait((int)((k - 1) & 1)); e != hipSuccess) return e;
        drain(i, n - i < per ? n - i : per, host[(k - 1) & 1]);
      }
    }
    return hipSuccess;
  }
};

struct rhllc_solver {
  rhllc_params prm{};
  int32_t n_cells = 0, n_faces = 0;
  bool mixed = false;
  bool tiled = true;
  int variant = kFp64Ref;
  bool has_state = false;
  bool rad = false;
  bool rad_kappa = false;  // rhllc_set_radiation was given kappa_a / kappa_s
  hipStream_t stream = nullptr;
  Dev d{};
  // Buffers of the state.  [cur] holds the state at the start of the next
  // step.  The tiled step reads [cur] and writes [cur ^ 1] for whatever the
  // face work gathers (FP64: U, W; mixed: the cell records); arrays a cell
  // only updates in place have [1] == [0], and so has every array of the
  // two-kernel step.
  int cur = 0;
  int last_in = -1;  // buffer the last step read (the tiled step's face fluxes are recomputed from it)
  double4 *U4b[2] = {nullptr, nullptr};
  double *UEb[2] = {nullptr, nullptr};
  double4 *W4b[2] = {nullptr, nullptr};
  double *Wpb[2] = {nullptr, nullptr};
  float4 *Wvab[2] = {nullptr, nullptr};
  double2 *Wsgb[2] = {nullptr, nullptr};
  int32_t n_tiles = 0, tile_slots = 0;
  std::vector<void *> allocs;
  int32_t *cell_old_to_new = nullptr;  // device
  int32_t *face_old_to_new = nullptr;  // device, from the first download of face fluxes on
  rhllc_mesh::RawVec<int32_t> face_old_to_new_host;
  Staging staging;
  Scalars *host_sc = nullptr;   // pinned copy of the device scalars, written by the device
  Scalars *host_sc_dev = nullptr;  // its device address
  unsigned long long fix_fail_seen = 0;  // fix_fail already reported by rhllc_step / rhllc_sync
  float4 *rad_FU = nullptr;
  float4 *rad_FU_add = nullptr;  // moments of rhllc_add_rad_flux
  float *rad_T = nullptr;        // pressure tensor of the fused source (rhllc_set_radiation_tensor)
  float *rad_T_add = nullptr;    // pressure tensor of rhllc_add_rad_flux_tensor
  float2 *rad_k = nullptr;
  double *tab = nullptr;  // opacity table (nx*ny), owned
  // The tiled steps of one rhllc_run rotate through the slot buffers of the
  // speed maximum: `slot` is the next step's, and `open` says that the last
  // step's maximum is still in its buffer (fold_speed of the next step takes
  // it, or close_steps).  Between calls nothing is open and slot is 0; on
  // meshes of more than kFoldMaxTiles tiles every step is closed at once.
  int slot = 0;
  bool open = false;
  // Captured graphs of kGraphSteps steps: the tiled step's starting from state
  // buffer k in [k] (folding: from slot 1 and an open step), the two-kernel
  // step's in [0]; a replay leaves buffer and slot as they were.
  hipGraphExec_t graph[2] = {nullptr, nullptr};
  hipGraph_t graph_src[2] = {nullptr, nullptr};
  int singles = 0;  // steps that rhllc_run launched singly for want of a graph
  int64_t replays = 0;
  unsigned int upload = 1;  // number of the last state upload (Scalars::upload; 1: none yet)
  float *mlp_P = nullptr;
  short *mlp_W2b = nullptr;

  template <typename T>
  hipError_t alloc(T **p, size_t count) {
    void *q = nullptr;
    hipError_t e = hipMalloc(&q, count * sizeof(T) + 64);
    if (e == hipSuccess) allocs.push_back(q);
    *p = static_cast<T *>(q);
    return e;
  }

  void drop_graph() {
    singles = 0;
    for (int k = 0; k < 2; ++k) {
      if (graph[k]) (void)hipGraphExecDestroy(graph[k]);
      if (graph_src[k]) (void)hipGraphDestroy(graph_src[k]);
      graph[k] = nullptr;
      graph_src[k] = nullptr;
    }
  }

  ~rhllc_solver() {
    drop_graph();
    if (stream) (void)hipStreamSynchronize(stream);
    for (void *p : allocs) (void)hipFree(p);
    if (face_old_to_new) (void)hipFree(face_old_to_new);
    if (rad_FU) (void)hipFree(rad_FU);
    if (rad_FU_add) (void)hipFree(rad_FU_add);
    if (rad_T) (void)hipFree(rad_T);
    if (rad_T_add) (void)hipFree(rad_T_add);
    if (rad_k) (void)hipFree(rad_k);
    if (tab) (void)hipFree(tab);
    if (mlp_P) (void)hipFree(mlp_P);
    if (mlp_W2b) (void)hipFree(mlp_W2b);
    if (host_sc) (void)hipHostFree(host_sc);
    if (stream) (void)hipStreamDestroy(stream);
  }

  bool ready() const { return has_state && (variant != kMixedMlp || mlp_P != nullptr); }

  // The kernel arguments with input buffers [in] and output buffers [out].
  Dev dev(int in, int out) const {
    Dev e = d;
    e.U4 = U4b[in], e.UE = UEb[in], e.W4 = W4b[in], e.Wp = Wpb[in], e.Wva = Wvab[in], e.Wsg = Wsgb[in];
    e.U4o = U4b[out], e.UEo = UEb[out], e.W4o = W4b[out], e.Wpo = Wpb[out], e.Wvao = Wvab[out], e.Wsgo = Wsgb[out];
    e.tile_reverse = in;
    return e;
  }
  // The current state, updated in place.
  Dev now() const { return dev(cur, cur); }

  // State and slot buffers both return after kCycle steps.  Between two graphs
  // the GPU idles longer than between two kernels of one, so a graph holds
  // several cycles; more would leave more steps of a run to single launches and
  // take longer to capture.  us a step with 6 / 12 / 24 steps a graph: 5.8 / 5.4 /
  // 5.2 at 162 cells, 6.8 / 6.4 / 6.2 at 6,000, 17.8 / 17.4 / 17.1 at 118,098 (FP64),
  // 32.2 / 31.8 / 31.8 at 663,552 (mixed).  A first run of 20 steps of 162 cells,
  // which then captures nothing, takes 122 us with 24 and 188 with 6.
  static constexpr int kCycle = 2 * kSpeedBufs;
  static constexpr int kGraphSteps = 4 * kCycle;
  static constexpr int kGraphWorth = 3 * kGraphSteps;

  bool folds() const { return tiled && n_tiles <= kFoldMaxTiles; }

  // The tiled step's kernel from buffer cur, at *tau or the device's own; it flips
  // cur and leaves the step open.  With a tau nothing is open before.
  hipError_t enqueue_tile(const double *tau = nullptr) {
    Dev x = dev(cur, cur ^ 1);
    x.slot = slot;
    x.fold = open;
    if (tau) x.use_tau = 1, x.tau = *tau;
    const hipError_t e = launch_tile(x, mixed, variant, rad, prm.collect_stats != 0, n_tiles, tile_slots, stream);
    if (e == hipSuccess) {
      last_in = cur;
      cur ^= 1;
      slot = (slot + 1) % kSpeedBufs;
      open = true;
    }
    return e;
  }
  // One step, closed unless it folds or is at the caller's tau.
  hipError_t enqueue_step(const double *tau = nullptr) {
    hipError_t e;
    if (tiled) {
      e = enqueue_tile(tau);
      if (e == hipSuccess && !tau && !folds()) e = close_steps();
      return e;
    }
    Dev x = now();
    if (tau) x.use_tau = 1, x.tau = *tau;
    e = launch_face(x, mixed, stream);
    x.use_tau = 0;  // the cell kernels read it from the scalars
    if (e == hipSuccess) e = launch_cell(x, variant, rad, prm.collect_stats != 0, stream);
    if (e == hipSuccess) {
      last_in = cur;
      open = true;
      if (!tau) e = close_steps();
    }
    return e;
  }
  // Takes the open step's maximum into the device scalars (tau, t, max_speed),
  // and into host_sc what rhllc_step reports.
  hipError_t close_steps(bool to_host = false) {
    if (!open) return hipSuccess;
    Dev x = now();
    x.slot = tiled ? (slot + kSpeedBufs - 1) % kSpeedBufs : 0;
    slot = 0;
    open = false;
    return launch_dt(x, to_host ? host_sc_dev : nullptr, stream);
  }
  // The device scalars into host_sc, after everything queued so far.
  hipError_t fetch_scalars() {
    const hipError_t e = launch_report(d, host_sc_dev, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
  }
  // Captures graph[cur].
  hipError_t capture() {
    const int k = cur, saved_in = last_in, saved_slot = slot;
    const bool saved_open = open;
    hipError_t e = hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) return e;
    for (int s = 0; s < kGraphSteps && e == hipSuccess; ++s) e = enqueue_step();
    hipGraph_t g = nullptr;
    const hipError_t e2 = hipStreamEndCapture(stream, &g);
    cur = k;  // capture enqueues nothing; replays leave these as they find them
    last_in = saved_in;
    slot = saved_slot;
    open = saved_open;
    if (e == hipSuccess) e = e2;
    if (e == hipSuccess) e = hipGraphInstantiate(&graph[k], g, nullptr, nullptr, 0);
    if (e != hipSuccess) {
      if (g) (void)hipGraphDestroy(g);
      graph[k] = nullptr;
      return e;
    }
    graph_src[k] = g;
    return hipSuccess;
  }
};

extern "C" const char *rhllc_last_error(void) { return g_err.c_str(); }

extern "C" int rhllc_create(const rhllc_params *params, int64_t n_cells, const void *geo_cells, int64_t n_faces,
                            const void *geo_faces, rhllc_solver **out) {
  if (!params || !out || !geo_cells || !geo_faces) return fail(RHLLC_ERR_ARG, "null argument");
  *out = nullptr;
  if (n_cells < 1 || n_cells >= ((int64_t)1 << 25))
    return fail(RHLLC_ERR_ARG, "n_cells must be in [1, 2^25) (geo_face_t::id_l is 25 bits)");
  // Faces below 2^27 (a mesh of 2^25 tets has at most 4 * 2^25 faces): the
  // kernels address the face arrays (at most 32 bytes an element) with 32-bit
  // byte offsets.
  if (n_faces < 1 || n_faces > ((int64_t)1 << 27)) return fail(RHLLC_ERR_ARG, "n_faces out of range [1, 2^27]");
  const rhllc_params &p = *params;
  if (p.eos != RHLLC_EOS_IDEAL && p.eos != RHLLC_EOS_TAUB) return fail(RHLLC_ERR_ARG, "unknown eos");
  if (p.eos == RHLLC_EOS_IDEAL && !(p.gamma > 1.0)) return fail(RHLLC_ERR_ARG, "gamma must be > 1");
  if (p.eos == RHLLC_EOS_TAUB && p.c2p_guess == RHLLC_GUESS_MLP)
    return fail(RHLLC_ERR_ARG, "the surrogate start is trained for the ideal gas; use RHLLC_EOS_IDEAL");
  if (!(p.cfl > 0.0) || !(p.h_min > 0.0)) return fail(RHLLC_ERR_ARG, "CFL and h_min must be > 0");
  if (p.precision != RHLLC_PREC_FP64 && p.precision != RHLLC_PREC_MIXED)
    return fail(RHLLC_ERR_ARG, "unknown precision");
  if (p.schedule != RHLLC_SCHED_TILED && p.schedule != RHLLC_SCHED_TWO_KERNEL)
    return fail(RHLLC_ERR_ARG, "unknown schedule");
  int variant;
  if (p.precision == RHLLC_PREC_FP64) {
    if (p.c2p_guess == RHLLC_GUESS_REFERENCE)
      variant = kFp64Ref;
    else if (p.c2p_guess == RHLLC_GUESS_PREVIOUS)
      variant = kFp64Prev;
    else
      return fail(RHLLC_ERR_ARG, "the FP64 path supports the reference and previous-pressure starts");
  } else {
    if (p.c2p_guess == RHLLC_GUESS_PREVIOUS)
      variant = kMixedPrev;
    else if (p.c2p_guess == RHLLC_GUESS_MLP)
      variant = kMixedMlp;
    else
      return fail(RHLLC_ERR_ARG, "the mixed path supports the previous-pressure and MLP starts");
  }
  const bool mixed = p.precision == RHLLC_PREC_MIXED, tiled = p.schedule == RHLLC_SCHED_TILED;

  // Host layout (validation, relabelling, SoA arrays, tiles) before the device is touched.
  rhllc_layout::Options opt;
  opt.mixed = mixed;
  opt.reorder = p.reorder != 0;
  opt.tiled = tiled;
  opt.has_out_source = p.has_out_source != 0;
  opt.has_inner_source = p.has_inner_source != 0;
  opt.lock_wall = p.lock_wall != 0;
  opt.reject_outer_surface = p.reject_outer_surface != 0;
  opt.out_source_copy = p.out_source_copy != 0;
  opt.tile_cells = tile_cells_for(n_cells, mixed, rhllc_capi_detail::compute_units(p.device));
  rhllc_layout::Layout L;
  {
    std::string err;
    if (!rhllc_layout::build(opt, n_cells, geo_cells, n_faces, geo_faces, L, err)) return fail(RHLLC_ERR_ARG, err);
  }
  // The kernels address the face arrays with 32-bit byte offsets (32-byte
  // FP64 entries).
  if (n_faces + (int64_t)L.tile_extra.size() > ((int64_t)1 << 27))
    return fail(RHLLC_ERR_ARG, "faces plus the tiles' extra faces exceed 2^27; use RHLLC_SCHED_TWO_KERNEL");
  const int32_t N = (int32_t)n_cells, F = (int32_t)n_faces;

  std::unique_ptr<rhllc_solver> h(new rhllc_solver());
  h->prm = p;
  h->n_cells = N;
  h->n_faces = F;
  h->mixed = mixed;
  h->tiled = tiled;
  h->variant = variant;
  HIP_TRY(hipSetDevice(p.device));
  HIP_TRY(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
  HIP_TRY(hipHostMalloc((void **)&h->host_sc, sizeof(Scalars), hipHostMallocDefault));
  HIP_TRY(hipHostGetDevicePointer((void **)&h->host_sc_dev, h->host_sc, 0));
  // Large enough for a pass over all faces or cells, up to the chunk limit.
  HIP_TRY(h->staging.alloc(std::max((size_t)N * 80, (size_t)F * 40)));

  Dev &d = h->d;
  d.n_cells = N;
  d.n_faces = F;
  d.eos = p.eos;
  d.gamma = p.eos == RHLLC_EOS_IDEAL ? p.gamma : 0.0;
  d.Gg = p.eos == RHLLC_EOS_IDEAL ? p.gamma / (p.gamma - 1.0) : 0.0;
  d.cfl_hmin = p.cfl * p.h_min;
  for (int k = 0; k < 5; ++k) {
    d.ghostW[k] = p.out_source_W[k], d.ghostU[k] = p.out_source_U[k];
    d.ghost2W[k] = p.inner_source_W[k], d.ghost2U[k] = p.inner_source_U[k];
  }

  // Uploads count elements of a host array into a new device array (at least
  // one element is allocated; an empty array copies nothing).
  auto upload = [&](auto **dst, const void *src, size_t count) -> hipError_t {
    hipError_t e = h->alloc(dst, count ? count : 1);
    if (e == hipSuccess && count) e = hipMemcpy(*dst, src, sizeof(**dst) * count, hipMemcpyHostToDevice);
    return e;
  };
  HIP_TRY(upload(&h->cell_old_to_new, L.cell_old_to_new.data(), N));
  h->face_old_to_new_host = std::move(L.face_old_to_new);
  // The face arrays, followed on the tiled step by the extra faces' copies
  // (the tiled mixed step reads face_far and the tile-local cells in face_Sn
  // in place of face_lr, which keeps the F faces for the flux download).
  const size_t nfe = (size_t)F + L.tile_extra.size();
  int2 *lr_d;
  HIP_TRY(upload(&lr_d, L.lr.data(), mixed && tiled ? (size_t)F : nfe));
  d.face_lr = lr_d;
  if (mixed && tiled) {
    int32_t *far_d;
    HIP_TRY(upload(&far_d, L.far.data(), nfe));
    d.face_far = far_d;
  }
  if (!mixed) {
    double *V_d;
    double4 *nS_d;
    HIP_TRY(upload(&V_d, L.V.data(), N));
    HIP_TRY(upload(&nS_d, L.nS.data(), nfe));
    d.cell_V = V_d;
    d.face_nS = nS_d;
  } else {
    double *vi_d;
    float4 *sn_d;
    HIP_TRY(upload(&vi_d, L.Vinv.data(), N));
    HIP_TRY(upload(&sn_d, L.Sn.data(), nfe));
    d.cell_Vinv = vi_d;
    d.face_Sn = sn_d;
  }
  if (tiled) {
    int4 *tm;
    uint2 *cs;
    HIP_TRY(upload(&tm, L.tile_meta.data(), L.n_tiles));
    HIP_TRY(upload(&cs, L.cell_slots.data(), N));
    d.tile_cells = opt.tile_cells;
    d.tile_meta = tm;
    d.cell_slots = cs;
    h->n_tiles = L.n_tiles;
    h->tile_slots = L.max_slots > 0 ? L.max_slots : 1;
  } else {
    int4 *cf_d;
    HIP_TRY(upload(&cf_d, L.cf.data(), N));
    d.cell_faces = cf_d;
    if (mixed) {
      HIP_TRY(h->alloc(&d.F4f, F));
      HIP_TRY(h->alloc(&d.FXf, F));
    } else {
      HIP_TRY(h->alloc(&d.F4, F));
      HIP_TRY(h->alloc(&d.FE, F));
    }
  }
  // State buffers: double-buffered where the tiled step gathers them.
  // Two entries more than the cells: N and N + 1 hold the ghost states of
  // codes -3 and -4.
  const bool twoU = tiled && !mixed, twoRec = tiled && mixed;
  for (int k = 0; k < 2; ++k) {
    if (k == 0 || twoU) {
      HIP_TRY(h->alloc(&h->U4b[k], N + 2));
      HIP_TRY(h->alloc(&h->UEb[k], N + 2));
      if (!mixed) {
        HIP_TRY(h->alloc(&h->W4b[k], N + 2));
        HIP_TRY(h->alloc(&h->Wpb[k], N + 2));
      }
    } else {
      h->U4b[k] = h->U4b[0], h->UEb[k] = h->UEb[0], h->W4b[k] = h->W4b[0], h->Wpb[k] = h->Wpb[0];
    }
    if (mixed && (k == 0 || twoRec)) {
      HIP_TRY(h->alloc(&h->Wvab[k], N + 2));
      HIP_TRY(h->alloc(&h->Wsgb[k], N + 2));
    } else {
      h->Wvab[k] = h->Wvab[0], h->Wsgb[k] = h->Wsgb[0];
    }
  }
  HIP_TRY(h->alloc(&d.sc, 1));
  HIP_TRY(h->alloc(&d.speed_slots, (size_t)kSpeedBufs * kSpeedSlots * kSlotStride));
  std::memset(h->host_sc, 0, sizeof(Scalars));
  h->host_sc->tau = d.cfl_hmin / 1.0;
  h->host_sc->last_speed = 1.0;
  h->host_sc->upload = h->upload;
  HIP_TRY(hipMemcpy(d.sc, h->host_sc, sizeof(Scalars), hipMemcpyHostToDevice));
  HIP_TRY(launch_clear_scalars(h->now(), h->stream));
  HIP_TRY(launch_ghost_cell(h->dev(0, 1), mixed, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  *out = h.release();
  return RHLLC_OK;
}

extern "C" int rhllc_destroy(rhllc_solver *h) {
  delete h;
  return RHLLC_OK;
}

extern "C" int rhllc_upload_state(rhllc_solver *h, const void *recs, int64_t stride, int64_t off_phys,
                                  int64_t off_conv) {
  if (!h || !recs) return fail(RHLLC_ERR_ARG, "null argument");
  if (off_phys < 0 || stride < 40 || off_phys + 40 > stride || (off_conv >= 0 && off_conv + 40 > stride))
    return fail(RHLLC_ERR_ARG, "bad record stride/offsets");
  HIP_TRY(hipSetDevice(h->prm.device));
  // On the handle's stream, so after what rhllc_run left in flight.
  const Dev d = h->now();
  const bool conv = off_conv >= 0;
  h->has_state = false;  // until all of it is on its way
  ++h->upload;
  HIP_TRY(h->staging.send(
      h->n_cells, conv ? 80 : 40, h->stream,
      [&](int64_t i, int64_t n, void *chunk) {
        rhllc_records::gather(static_cast<const uint8_t *>(recs) + i * stride, stride, off_phys, off_conv, n, chunk);
      },
      [&](int i, int n, void *chunk) {
        return launch_unpack_state(d, h->mixed, h->cell_old_to_new, i, n, conv, !conv, h->upload,
                                   static_cast<double *>(chunk), h->stream);
      }));
  h->has_state = true;
  h->last_in = -1;
  return RHLLC_OK;
}

extern "C" int rhllc_download_state(rhllc_solver *h, void *recs, int64_t stride, int64_t off_phys,
                                    int64_t off_conv) {
  if (!h || !recs) return fail(RHLLC_ERR_ARG, "null argument");
  if (stride < 40 || (off_phys >= 0 && off_phys + 40 > stride) || (off_conv >= 0 && off_conv + 40 > stride))
    return fail(RHLLC_ERR_ARG, "bad record stride/offsets");
  if (!h->has_state) return fail(RHLLC_ERR_STATE, "no state uploaded");
  HIP_TRY(hipSetDevice(h->prm.device));
  const Dev d = h->now();
  const bool phys = off_phys >= 0, conv = off_conv >= 0;
  if (!phys && !conv) {  // the wait alone
    HIP_TRY(hipStreamSynchronize(h->stream));
    return RHLLC_OK;
  }
  HIP_TRY(h->staging.receive(
      h->n_cells, phys && conv ? 80 : 40, h->stream,
      [&](int i, int n, void *chunk) {
        return launch_pack_state(d, h->mixed, h->cell_old_to_new, i, n, phys, conv, static_cast<double *>(chunk),
                                 h->stream);
      },
      [&](int64_t i, int64_t n, const void *chunk) {
        rhllc_records::scatter(static_cast<uint8_t *>(recs) + i * stride, stride, off_phys, off_conv, n, chunk);
      }));
  return RHLLC_OK;
}

// PhysPressureFix failures and a non-finite speed since the last report.
static int report_step_errors(rhllc_solver *h) {
  const unsigned long long ff = h->host_sc->fix_fail;
  const unsigned long long before = h->fix_fail_seen;
  h->fix_fail_seen = ff;
  if (ff > before)
    return fail(RHLLC_ERR_C2P, std::to_string(ff - before) + " cells failed PhysPressureFix");
  if (!std::isfinite(h->host_sc->last_speed) || !std::isfinite(h->host_sc->tau))
    return fail(RHLLC_ERR_NUMERIC, "non-finite max signal speed");
  return RHLLC_OK;
}

extern "C" int rhllc_step(rhllc_solver *h, double tau, double *max_speed) {
  if (!h) return fail(RHLLC_ERR_ARG, "null handle");
  if (!h->ready()) return fail(RHLLC_ERR_STATE, "no state uploaded (or no MLP model set for RHLLC_GUESS_MLP)");
  HIP_TRY(hipSetDevice(h->prm.device));
  // Two launches and a wait: tau goes in as an argument, and the speed, the
  // next tau and the failures come back through pinned memory.
  HIP_TRY(h->enqueue_step(&tau));
  HIP_TRY(h->close_steps(true));
  HIP_TRY(hipStreamSynchronize(h->stream));
  const double s = h->host_sc->last_speed;
  if (max_speed) *max_speed = s;
  return report_step_errors(h);
}

extern "C" int rhllc_run(rhllc_solver *h, int32_t nsteps, int32_t use_graph) {
  if (!h) return fail(RHLLC_ERR_ARG, "null handle");
  if (!h->ready()) return fail(RHLLC_ERR_STATE, "no state uploaded (or no MLP model set for RHLLC_GUESS_MLP)");
  if (nsteps < 0) return fail(RHLLC_ERR_ARG, "nsteps < 0");
  HIP_TRY(hipSetDevice(h->prm.device));
  int32_t k = 0;
  hipError_t e = hipSuccess;
  if (use_graph) {
    // A folding step's graph continues from an open step, so the first step goes
    // out by itself.  So do the steps that fill no graph, first (folding, in
    // whole cycles: the slot has to be the graph's), so that the GPU has work
    // while one is captured.  A graph is captured once its replays would have
    // served kGraphWorth steps of this and earlier runs: a capture takes as long
    // as about two replays save (first runs of 30 steps were 10% slower with a
    // capture each).
    constexpr int per = rhllc_solver::kGraphSteps, cycle = rhllc_solver::kCycle;
    const int open = h->folds() ? 1 : 0, whole = nsteps < open ? 0 : (nsteps - open) / per * per;
    const int rest = nsteps - whole, lead = open ? open + (rest - open) / cycle * cycle : rest;
    const int first = h->tiled ? h->cur ^ (lead & 1) : 0;
    if (whole > 0 && !h->graph[first] && h->singles + whole < rhllc_solver::kGraphWorth) {
      h->singles += whole;
    } else if (whole > 0) {
      for (; k < lead && e == hipSuccess; ++k) e = h->enqueue_step();
      if (e == hipSuccess && !h->graph[h->cur]) e = h->capture();
      for (; k + per <= nsteps && e == hipSuccess; k += per)
        if ((e = hipGraphLaunch(h->graph[h->cur], h->stream)) == hipSuccess) ++h->replays;
      h->last_in = h->tiled ? h->cur ^ 1 : h->cur;
    }
  }
  for (; k < nsteps && e == hipSuccess; ++k) e = h->enqueue_step();
  const hipError_t e2 = h->close_steps();
  if (e == hipSuccess) e = e2;
  if (e != hipSuccess) return hip_fail(e, "step");
  return RHLLC_OK;
}

extern "C" int rhllc_sync(rhllc_solver *h) {
  if (!h) return fail(RHLLC_ERR_ARG, "null handle");
  HIP_TRY(hipSetDevice(h->prm.device));
  HIP_TRY(h->fetch_scalars());
  return report_step_errors(h);
}

extern "C" int rhllc_set_collect_stats(rhllc_solver *h, int32_t on) {
  if (!h) return fail(RHLLC_ERR_ARG, "null handle");
  HIP_TRY(hipSetDevice(h->prm.device));
  HIP_TRY(hipStreamSynchronize(h->stream));
  if ((h->prm.collect_stats != 0) != (on != 0)) h->drop_graph();  // other kernels
  h->prm.collect_stats = on != 0;
  return RHLLC_OK;
}

extern "C" int rhllc_set_time(rhllc_solver *h, double tau, double t) {
  if (!h) return fail(RHLLC_ERR_ARG, "null handle");
  HIP_TRY(hipSetDevice(h->prm.device));
  HIP_TRY(hipStreamSynchronize(h->stream));
  h->host_sc->tau = tau;
  h->host_sc->t = t;
  HIP_TRY(hipMemcpy(&h->d.sc->tau, &h->host_sc->tau, 2 * sizeof(double), hipMemcpyHostToDevice));
  return RHLLC_OK;
}

extern "C" int rhllc_get_stats(rhllc_solver *h, rhllc_stats *out) {
  if (!h || !out) return fail(RHLLC_ERR_ARG, "null argument");
  HIP_TRY(hipSetDevice(h->prm.device));
  HIP_TRY(h->fetch_scalars());
  const Scalars &s = *h->host_sc;
  std::memset(out, 0, sizeof(*out));
  out->steps = (int64_t)s.steps;
  for (int k = 0; k < 6; ++k) out->c2p_fail[k] = (int64_t)s.c2p_fail[k];
  out->fix_calls = (int64_t)s.fix_calls;
  out->fix_fail = (int64_t)s.fix_fail;
  out->fallback_cells = (int64_t)s.fallback;
  out->mlp_starts = (int64_t)s.mlp_starts;
  out->newton_iters = (int64_t)s.newton_iters;
  for (int k = 0; k < RHLLC_HIST_BINS; ++k) out->newton_hist[k] = (int64_t)s.hist[k];
  out->max_speed = s.last_speed;
  out->tau = s.tau;
  out->t = s.t;
  double r;
  std::memcpy(&r, &s.max_residual_bits, 8);
  out->max_residual = r;
  return RHLLC_OK;
}

extern "C" int rhllc_reset_stats(rhllc_solver *h) {
  if (!h) return fail(RHLLC_ERR_ARG, "null handle");
  HIP_TRY(hipSetDevice(h->prm.device));
  HIP_TRY(launch_clear_scalars(h->now(), h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  h->fix_fail_seen = 0;
  return RHLLC_OK;
}

extern "C" int rhllc_download_face_flux(rhllc_solver *h, double *F) {
  if (!h || !F) return fail(RHLLC_ERR_ARG, "null argument");
  HIP_TRY(hipSetDevice(h->prm.device));
  const int32_t nf = h->n_faces;
  if (h->last_in < 0) {  // no step since the state was set
    std::memset(F, 0, sizeof(double) * 5 * (size_t)nf);
    return RHLLC_OK;
  }
  HIP_TRY(rhllc_records::fill_once(
      h->face_old_to_new, [&](int32_t **p) { return hipMalloc((void **)p, sizeof(int32_t) * nf); },
      [&](int32_t *p) {
        return hipMemcpy(p, h->face_old_to_new_host.data(), sizeof(int32_t) * nf, hipMemcpyHostToDevice);
      },
      [](int32_t *p) { (void)hipFree(p); }));
  rhllc_mesh::RawVec<int32_t>().swap(h->face_old_to_new_host);
  // The tiled step keeps its fluxes in LDS; they are recomputed, to the same
  // bits, from the state the last step read (its input buffer is intact).
  const Dev d = h->tiled ? h->dev(h->last_in, h->last_in) : h->now();
  HIP_TRY(h->staging.receive(
      nf, 40, h->stream,
      [&](int i, int n, void *chunk) {
        return launch_face_out(d, h->mixed, !h->tiled, h->face_old_to_new, i, n, static_cast<double *>(chunk),
                               h->stream);
      },
      [&](int64_t i, int64_t n, const void *chunk) { rhllc_records::copy(F + 5 * i, chunk, sizeof(double) * 5 * n); }));
  return RHLLC_OK;
}

// Per-cell FP32 fields of the caller (moments, opacities, pressure tensor;
// null: not given) into the device arrays, through the staging chunks in the
// order launch_unpack_fields reads them.
static hipError_t send_fields(rhllc_solver *h, const float *Ur, const float *Fr3, const float *ka, const float *ks,
                              const float *Tr9, float4 *FU, float2 *k, float *T, bool mark = false) {
  const size_t each = sizeof(float) * ((FU ? 4 : 0) + (ka ? 2 : 0) + (T ? 9 : 0));
  return h->staging.send(
      h->n_cells, each, h->stream,
      [&](int64_t i, int64_t n, void *chunk) {
        float *o = static_cast<float *>(chunk);
        auto put = [&](const float *src, int w) {
          rhllc_records::copy(o, src + w * i, sizeof(float) * w * n);
          o += w * n;
        };
        if (FU) put(Ur, 1), put(Fr3, 3);
        if (ka) put(ka, 1), put(ks, 1);
        if (T) put(Tr9, 9);
      },
      [&](int i, int n, void *chunk) {
        return launch_unpack_fields(h->cell_old_to_new, i, n, static_cast<const float *>(chunk), FU, k, ka != nullptr,
                                    T, mark && i == 0 ? h->d.sc : nullptr, h->stream);
      });
}

extern "C" int rhllc_set_radiation(rhllc_solver *h, const float *Ur, const float *Fr3, const float *kappa_a,
                                   const float *kappa_s) {
  if (!h) return fail(RHLLC_ERR_ARG, "null handle");
  HIP_TRY(hipSetDevice(h->prm.device));
  HIP_TRY(hipStreamSynchronize(h->stream));
  h->drop_graph();
  if (!Ur) {
    h->rad = false;
    return RHLLC_OK;
  }
  if (!Fr3) return fail(RHLLC_ERR_ARG, "null radiation array");
  if (!kappa_a != !kappa_s) return fail(RHLLC_ERR_ARG, "kappa_a and kappa_s must both be given or both be NULL");
  if (!kappa_a && !h->tab) return fail(RHLLC_ERR_ARG, "no opacities: give kappa_a/kappa_s or set an opacity table");
  const int32_t N = h->n_cells;
  if (!h->rad_FU) HIP_TRY(hipMalloc((void **)&h->rad_FU, sizeof(float4) * N));
  if (!h->rad_k) HIP_TRY(hipMalloc((void **)&h->rad_k, sizeof(float2) * N));
  HIP_TRY(send_fields(h, Ur, Fr3, kappa_a, kappa_s, nullptr, h->rad_FU, h->rad_k, nullptr));
  h->d.rad_FU = h->rad_FU;
  h->d.rad_k = h->rad_k;
  h->rad = true;
  h->rad_kappa = kappa_a != nullptr;
  return RHLLC_OK;
}

extern "C" int rhllc_set_radiation_tensor(rhllc_solver *h, const float *Tr9) {
  if (!h) return fail(RHLLC_ERR_ARG, "null handle");
  HIP_TRY(hipSetDevice(h->prm.device));
  HIP_TRY(hipStreamSynchronize(h->stream));
  h->drop_graph();  // the graph holds the kernel arguments by value
  if (!Tr9) {
    h->d.rad_T = nullptr;
    return RHLLC_OK;
  }
  if (!h->rad_T) HIP_TRY(hipMalloc((void **)&h->rad_T, sizeof(float) * 9 * (size_t)h->n_cells));
  HIP_TRY(send_fields(h, nullptr, nullptr, nullptr, nullptr, Tr9, nullptr, nullptr, h->rad_T));
  h->d.rad_T = h->rad_T;
  return RHLLC_OK;
}

static int add_rad_flux(rhllc_solver *h, double tau, const float *Ur, const float *Fr3, const float *Tr9) {
  if (!h) return fail(RHLLC_ERR_ARG, "null handle");
  if (!Ur || !Fr3) return fail(RHLLC_ERR_ARG, "null radiation array");
  if (!(tau >= 0.0) || !std::isfinite(tau)) return fail(RHLLC_ERR_ARG, "tau must be finite and >= 0");
  if (!h->tab) return fail(RHLLC_ERR_STATE, "no opacity table set (rhllc_set_opacity_table)");
  if (!h->ready()) return fail(RHLLC_ERR_STATE, "no state uploaded");
  HIP_TRY(hipSetDevice(h->prm.device));
  const size_t N = (size_t)h->n_cells;
  // Its own buffers: the moments of rhllc_set_radiation (the step's fused
  // source, also held by a captured graph) stay as they were.
  if (!h->rad_FU_add) HIP_TRY(hipMalloc((void **)&h->rad_FU_add, sizeof(float4) * N));
  if (Tr9 && !h->rad_T_add) HIP_TRY(hipMalloc((void **)&h->rad_T_add, sizeof(float) * 9 * N));
  HIP_TRY(send_fields(h, Ur, Fr3, nullptr, nullptr, Tr9, h->rad_FU_add, nullptr, Tr9 ? h->rad_T_add : nullptr,
                      true));
  Dev x = h->now();
  x.rad_FU = h->rad_FU_add;
  x.rad_T = Tr9 ? h->rad_T_add : nullptr;
  HIP_TRY(launch_add_rad(x, h->mixed, tau, h->stream));
  HIP_TRY(h->fetch_scalars());
  const unsigned long long now_failed = h->host_sc->fix_fail - h->host_sc->fix_mark;  // the source's own
  h->fix_fail_seen += now_failed;  // reported here; earlier steps' failures stay for rhllc_sync
  if (now_failed)
    return fail(RHLLC_ERR_C2P, std::to_string(now_failed) + " cells failed PhysPressureFix after the radiation source");
  return RHLLC_OK;
}

extern "C" int rhllc_add_rad_flux(rhllc_solver *h, double tau, const float *Ur, const float *Fr3) {
  return add_rad_flux(h, tau, Ur, Fr3, nullptr);
}

extern "C" int rhllc_add_rad_flux_tensor(rhllc_solver *h, double tau, const float *Ur, const float *Fr3,
                                         const float *Tr9) {
  if (!Tr9) return fail(RHLLC_ERR_ARG, "null pressure tensor");
  return add_rad_flux(h, tau, Ur, Fr3, Tr9);
}

extern "C" int rhllc_set_radiation_emission(rhllc_solver *h, int32_t on) {
  if (!h) return fail(RHLLC_ERR_ARG, "null handle");
  HIP_TRY(hipSetDevice(h->prm.device));
  HIP_TRY(hipStreamSynchronize(h->stream));
  h->drop_graph();  // the graph holds the kernel arguments by value
  h->d.rad_emission = on != 0;
  return RHLLC_OK;
}

// Table axes as the lookup uses them: finite, min <= max, positive steps.
static int check_table(int32_t nx, int32_t ny, const double *hdr) {
  if (nx < 1 || ny < 2 || (int64_t)nx * ny > (int64_t)1 << 26) return fail(RHLLC_ERR_ARG, "bad table size");
  for (int k = 0; k < 6; ++k)
    if (!std::isfinite(hdr[k])) return fail(RHLLC_ERR_ARG, "non-finite table header");
  if (!(hdr[0] <= hdr[1]) || !(hdr[2] > 0) || !(hdr[3] <= hdr[4]) || !(hdr[5] > 0))
    return fail(RHLLC_ERR_ARG, "table header needs min <= max and step > 0 on both axes");
  return RHLLC_OK;
}

extern "C" int rhllc_set_opacity_table(rhllc_solver *h, int32_t nx, int32_t ny, const double header[6],
                                       const double *data) {
  if (!h) return fail(RHLLC_ERR_ARG, "null handle");
  HIP_TRY(hipSetDevice(h->prm.device));
  HIP_TRY(hipStreamSynchronize(h->stream));
  h->drop_graph();
  if (!data) {
    if (h->rad && !h->rad_kappa)
      return fail(RHLLC_ERR_STATE, "the radiation source has no other opacities: remove it (rhllc_set_radiation "
                                   "with Ur = NULL) or give kappa_a/kappa_s first");
    if (h->tab) HIP_TRY(hipFree(h->tab));
    h->tab = nullptr;
    h->d.tab = nullptr;
    return RHLLC_OK;
  }
  if (!header) return fail(RHLLC_ERR_ARG, "null table header");
  if (int e = check_table(nx, ny, header)) return e;
  double *t = nullptr;
  HIP_TRY(hipMalloc((void **)&t, sizeof(double) * nx * ny));
  const hipError_t e = hipMemcpy(t, data, sizeof(double) * nx * ny, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    (void)hipFree(t);
    HIP_TRY(e);
  }
  if (h->tab) HIP_TRY(hipFree(h->tab));
  h->tab = t;
  Dev &d = h->d;
  d.tab = t;
  d.tab_nx = nx, d.tab_ny = ny;
  d.tab_min_x = header[0], d.tab_max_x = header[1], d.tab_step_x = header[2];
  d.tab_min_y = header[3], d.tab_max_y = header[4], d.tab_step_y = header[5];
  return RHLLC_OK;
}

extern "C" int rhllc_set_mlp(rhllc_solver *h, const float *model) {
  if (!h || !model) return fail(RHLLC_ERR_ARG, "null argument");
  const double mg = model[RHLLC_MLP_MODEL - 1];
  if (!(std::fabs(mg - h->prm.gamma) <= 1e-6 * h->prm.gamma))
    return fail(RHLLC_ERR_ARG, "model was trained for gamma " + std::to_string(mg) + ", the handle uses " +
                                   std::to_string(h->prm.gamma));
  HIP_TRY(hipSetDevice(h->prm.device));
  HIP_TRY(hipStreamSynchronize(h->stream));
  h->drop_graph();
  if (!h->mlp_P) HIP_TRY(hipMalloc((void **)&h->mlp_P, sizeof(float) * RHLLC_MLP_MODEL));
  if (!h->mlp_W2b) HIP_TRY(hipMalloc((void **)&h->mlp_W2b, sizeof(short) * 64 * 64 * 2));
  HIP_TRY(hipMemcpy(h->mlp_P, model, sizeof(float) * RHLLC_MLP_MODEL, hipMemcpyHostToDevice));
  HIP_TRY(rhllc_mlp::launch_pack(h->mlp_P, h->mlp_W2b, h->mlp_W2b + 64 * 64, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  h->d.mlpP = h->mlp_P;
  h->d.mlpW2b = h->mlp_W2b;
  return RHLLC_OK;
}

extern "C" int rhllc_time_kernels(rhllc_solver *h, int32_t nsteps, double out[4]) {
  if (!h || !out) return fail(RHLLC_ERR_ARG, "null argument");
  if (!h->ready()) return fail(RHLLC_ERR_STATE, "no state uploaded (or no MLP model set)");
  if (nsteps < 1 || nsteps > 4096) return fail(RHLLC_ERR_ARG, "nsteps must be in 1..4096");
  HIP_TRY(hipSetDevice(h->prm.device));
  HIP_TRY(hipStreamSynchronize(h->stream));
  // Twenty untimed lead-in steps, then nsteps steps with four events each, all
  // enqueued back to back: the device runs them without the idle gaps that a
  // host wait per step would leave, as it runs the graph-replayed steps.  After
  // an idle period the device clock takes some fifteen steps to settle (the
  // first kernel runs fast, the next few up to 30% slower than steady state).
  constexpr int kLead = 20;
  std::vector<hipEvent_t> ev(4 * (size_t)nsteps, nullptr);
  int rc = RHLLC_OK;
  for (auto &e : ev)
    if (hipError_t err = hipEventCreate(&e); err != hipSuccess) {
      rc = hip_fail(err, "kernel timing");
      break;
    }
  const bool stats = h->prm.collect_stats != 0, folds = h->folds();
  for (int32_t k = 0; k < kLead + nsteps && rc == RHLLC_OK; ++k) {
    hipEvent_t *e4 = k >= kLead ? &ev[4 * (size_t)(k - kLead)] : nullptr;
    hipError_t e = e4 ? hipEventRecord(e4[0], h->stream) : hipSuccess;
    if (h->tiled) {
      if (e == hipSuccess) e = h->enqueue_tile();
    } else {
      if (e == hipSuccess) e = launch_face(h->now(), h->mixed, h->stream);
      if (e == hipSuccess) h->last_in = h->cur, h->open = true;
    }
    if (e == hipSuccess && e4) e = hipEventRecord(e4[1], h->stream);
    if (!folds) {  // a folding step is the tile kernel alone
      if (e == hipSuccess && !h->tiled) e = launch_cell(h->now(), h->variant, h->rad, stats, h->stream);
      if (e == hipSuccess && e4) e = hipEventRecord(e4[2], h->stream);
      if (e == hipSuccess) e = h->close_steps();
      if (e == hipSuccess && e4) e = hipEventRecord(e4[3], h->stream);
    }
    if (e != hipSuccess) rc = hip_fail(e, "kernel timing");
  }
  if (hipError_t e = h->close_steps(); e != hipSuccess && rc == RHLLC_OK) rc = hip_fail(e, "kernel timing");
  double acc[4] = {0, 0, 0, 0};
  if (rc == RHLLC_OK) {
    if (hipError_t e = hipStreamSynchronize(h->stream); e != hipSuccess) rc = hip_fail(e, "kernel timing");
  }
  const auto add = [&](int i, hipEvent_t from, hipEvent_t to) {
    float ms = 0;
    if (hipError_t e = hipEventElapsedTime(&ms, from, to); e != hipSuccess && rc == RHLLC_OK)
      rc = hip_fail(e, "kernel timing");
    acc[i] += ms;
  };
  for (int32_t k = 0; k < nsteps && rc == RHLLC_OK; ++k) {
    const hipEvent_t *e4 = &ev[4 * (size_t)k];
    add(0, e4[0], e4[1]);
    if (folds) continue;
    add(1, e4[1], e4[2]);
    add(2, e4[2], e4[3]);
    add(3, e4[0], e4[3]);
  }
  if (folds && rc == RHLLC_OK) add(3, ev[0], ev[4 * (size_t)(nsteps - 1) + 1]);
  for (auto &e : ev)
    if (e) (void)hipEventDestroy(e);
  if (rc != RHLLC_OK) return rc;
  for (int i = 0; i < 4; ++i) out[i] = acc[i] / nsteps;
  return RHLLC_OK;
}

extern "C" int rhllc_info(rhllc_solver *h, int64_t *n_cells, int64_t *n_faces, int64_t *device_bytes) {
  if (!h) return fail(RHLLC_ERR_ARG, "null handle");
  if (n_cells) *n_cells = h->n_cells;
  if (n_faces) *n_faces = h->n_faces;
  if (device_bytes) {
    const int64_t N = h->n_cells, F = h->n_faces;
    // The two-kernel structure's compulsory bytes at the variant's storage
    // precision: FP64 face 80 N + 80 F, cell 153 N + 40 F; mixed face
    // 20 N + 44 F, cell 141 N + 20 F; the radiation fields 24 N.
    *device_bytes = h->mixed ? 161 * N + 64 * F : 233 * N + 120 * F;
    if (h->rad) *device_bytes += 24 * N;
  }
  return RHLLC_OK;
}

extern "C" int rhllc_step_form(rhllc_solver *h, int64_t out[4]) {
  if (!h || !out) return fail(RHLLC_ERR_ARG, "null argument");
  HIP_TRY(hipSetDevice(h->prm.device));
  HIP_TRY(h->fetch_scalars());
  out[0] = h->tiled ? h->d.tile_cells : 0;
  out[1] = h->folds();
  out[2] = h->replays;
  out[3] = h->tiled && !h->mixed && h->host_sc->unusual != h->host_sc->upload;
  return RHLLC_OK;
}

extern "C" int rhllc_tile_layout(int64_t n_cells, const void *geo_cells, int64_t n_faces, const void *geo_faces,
                                 int32_t reorder, int32_t *n_tiles, int64_t *n_extra, int32_t *max_slots,
                                 int32_t *cell_new_to_old, int32_t *face_new_to_old, int32_t *tile_meta,
                                 int32_t *tile_extra, uint32_t *cell_slots) {
  return rhllc_tile_layout_of(n_cells, geo_cells, n_faces, geo_faces, reorder, kTileCells, n_tiles, n_extra, max_slots,
                              cell_new_to_old, face_new_to_old, tile_meta, tile_extra, cell_slots);
}

extern "C" int rhllc_tile_layout_of(int64_t n_cells, const void *geo_cells, int64_t n_faces, const void *geo_faces,
                                    int32_t reorder, int32_t tile_cells, int32_t *n_tiles, int64_t *n_extra,
                                    int32_t *max_slots, int32_t *cell_new_to_old, int32_t *face_new_to_old,
                                    int32_t *tile_meta, int32_t *tile_extra, uint32_t *cell_slots) {
  if (!geo_cells || !geo_faces || !n_tiles || !n_extra || !max_slots) return fail(RHLLC_ERR_ARG, "null argument");
  if (n_cells < 1 || n_cells >= ((int64_t)1 << 25) || n_faces < 1 || n_faces > 0x7FFFFFFF)
    return fail(RHLLC_ERR_ARG, "mesh size out of range");
  if (tile_cells != kTileCells && tile_cells != kSmallTileCells)
    return fail(RHLLC_ERR_ARG, "tile_cells must be 64 or 256");
  rhllc_layout::Options opt;
  opt.reorder = reorder != 0;
  opt.tiled = true;
  opt.has_out_source = true;
  opt.tile_cells = tile_cells;
  rhllc_layout::Layout L;
  std::string err;
  if (!rhllc_layout::build(opt, n_cells, geo_cells, n_faces, geo_faces, L, err)) return fail(RHLLC_ERR_ARG, err);
  *n_tiles = L.n_tiles;
  *n_extra = (int64_t)L.tile_extra.size();
  *max_slots = L.max_slots;
  if (cell_new_to_old) std::memcpy(cell_new_to_old, L.cell_new_to_old.data(), sizeof(int32_t) * n_cells);
  if (face_new_to_old) std::memcpy(face_new_to_old, L.face_new_to_old.data(), sizeof(int32_t) * n_faces);
  if (tile_meta) std::memcpy(tile_meta, L.tile_meta.data(), sizeof(int32_t) * L.tile_meta.size());
  if (tile_extra && !L.tile_extra.empty())
    std::memcpy(tile_extra, L.tile_extra.data(), sizeof(int32_t) * L.tile_extra.size());
  if (cell_slots) std::memcpy(cell_slots, L.cell_slots.data(), sizeof(uint32_t) * L.cell_slots.size());
  return RHLLC_OK;
}

extern "C" int rhllc_pack_face_vectors(int64_t n, const double *Sn, float *out) {
  if (n < 0) return fail(RHLLC_ERR_ARG, "n < 0");
  if (n > 0 && (!Sn || !out)) return fail(RHLLC_ERR_ARG, "null argument");
  for (int64_t i = 0; i < n; ++i) rhllc_layout::pack_sn(Sn + 3 * i, out + 4 * i);
  return RHLLC_OK;
}

// ------------------------------------------------------------ pointwise evals
namespace {
struct DevBuf {
  void *p = nullptr;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
};
hipError_t to_dev(DevBuf &b, const void *src, size_t bytes) {
  hipError_t e = hipMalloc(&b.p, bytes + 64);
  if (e == hipSuccess && src) e = hipMemcpy(b.p, src, bytes, hipMemcpyHostToDevice);
  return e;
}
}  // namespace

namespace {
bool bad_eos(int32_t eos, double gamma) {
  return !(eos == RHLLC_EOS_TAUB || (eos == RHLLC_EOS_IDEAL && gamma > 1.0));
}
}  // namespace

extern "C" int rhllc_eval_flux(int32_t precision, int32_t eos, double gamma, int64_t n, const double *UL,
                               const double *UR, const double *WL, const double *WR, const double *nS4, double *F,
                               double *speed) {
  if (n < 0 || !UL || !UR || !WL || !WR || !nS4 || !F || !speed) return fail(RHLLC_ERR_ARG, "bad argument");
  if (bad_eos(eos, gamma)) return fail(RHLLC_ERR_ARG, "unknown eos, or gamma <= 1 for the ideal gas");
  DevBuf a, b, c, dd, e, f, g;
  const size_t s5 = sizeof(double) * 5 * n;
  HIP_TRY(to_dev(a, UL, s5));
  HIP_TRY(to_dev(b, UR, s5));
  HIP_TRY(to_dev(c, WL, s5));
  HIP_TRY(to_dev(dd, WR, s5));
  HIP_TRY(to_dev(e, nS4, sizeof(double) * 4 * n));
  HIP_TRY(to_dev(f, nullptr, s5));
  HIP_TRY(to_dev(g, nullptr, sizeof(double) * n));
  HIP_TRY(launch_eval_flux(precision == RHLLC_PREC_MIXED, eos, gamma, n, (double *)a.p, (double *)b.p, (double *)c.p,
                           (double *)dd.p, (double *)e.p, (double *)f.p, (double *)g.p, nullptr));
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(F, f.p, s5, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(speed, g.p, sizeof(double) * n, hipMemcpyDeviceToHost));
  return RHLLC_OK;
}

extern "C" int rhllc_eval_c2p(int32_t precision, int32_t eos, double gamma, int64_t n, const double *U,
                              const double *guess, double *W, int32_t *codes, int32_t *iters) {
  if (n < 0 || !U || !W || !codes || !iters) return fail(RHLLC_ERR_ARG, "bad argument");
  if (bad_eos(eos, gamma)) return fail(RHLLC_ERR_ARG, "unknown eos, or gamma <= 1 for the ideal gas");
  if (precision != RHLLC_PREC_FP64 && precision != RHLLC_PREC_MIXED) return fail(RHLLC_ERR_ARG, "bad precision");
  DevBuf a, b, c, dd, e;
  HIP_TRY(to_dev(a, U, sizeof(double) * 5 * n));
  HIP_TRY(to_dev(c, W, sizeof(double) * 5 * n));
  if (guess) HIP_TRY(to_dev(b, guess, sizeof(double) * n));
  HIP_TRY(to_dev(dd, nullptr, sizeof(int32_t) * n));
  HIP_TRY(to_dev(e, nullptr, sizeof(int32_t) * n));
  HIP_TRY(launch_eval_c2p(precision == RHLLC_PREC_MIXED, eos, gamma, n, (double *)a.p, (double *)b.p, (double *)c.p, (int32_t *)dd.p, (int32_t *)e.p,
                          nullptr));
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(W, c.p, sizeof(double) * 5 * n, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(codes, dd.p, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(iters, e.p, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
  return RHLLC_OK;
}

extern "C" int rhllc_eval_p2c(int32_t eos, double gamma, int64_t n, double *W, double *U) {
  if (n < 0 || !W || !U) return fail(RHLLC_ERR_ARG, "bad argument");
  if (bad_eos(eos, gamma)) return fail(RHLLC_ERR_ARG, "unknown eos, or gamma <= 1 for the ideal gas");
  DevBuf a, b;
  HIP_TRY(to_dev(a, W, sizeof(double) * 5 * n));
  HIP_TRY(to_dev(b, nullptr, sizeof(double) * 5 * n));
  HIP_TRY(launch_eval_p2c(eos, gamma, n, (double *)a.p, (double *)b.p, nullptr));
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(W, a.p, sizeof(double) * 5 * n, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(U, b.p, sizeof(double) * 5 * n, hipMemcpyDeviceToHost));
  return RHLLC_OK;
}

extern "C" int rhllc_eval_pressure_fix(int32_t eos, double gamma, int64_t n, double *U, double *W, int32_t *codes) {
  if (n < 0 || !U || !W || !codes) return fail(RHLLC_ERR_ARG, "bad argument");
  if (bad_eos(eos, gamma)) return fail(RHLLC_ERR_ARG, "unknown eos, or gamma <= 1 for the ideal gas");
  DevBuf a, b, c;
  HIP_TRY(to_dev(a, U, sizeof(double) * 5 * n));
  HIP_TRY(to_dev(b, W, sizeof(double) * 5 * n));
  HIP_TRY(to_dev(c, nullptr, sizeof(int32_t) * n));
  HIP_TRY(launch_eval_fix(eos, gamma, n, (double *)a.p, (double *)b.p, (int32_t *)c.p, nullptr));
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(U, a.p, sizeof(double) * 5 * n, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(W, b.p, sizeof(double) * 5 * n, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(codes, c.p, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
  return RHLLC_OK;
}

extern "C" int rhllc_eval_rad_source(int32_t precision, int64_t n, const double *W, const double *Ur,
                                     const double *Fr3, const double *ka, const double *ks, int32_t emission,
                                     const float *Tr9, double *G) {
  if (n < 0 || !W || !Ur || !Fr3 || !ka || !ks || !G) return fail(RHLLC_ERR_ARG, "bad argument");
  if (precision != RHLLC_PREC_FP64 && precision != RHLLC_PREC_MIXED) return fail(RHLLC_ERR_ARG, "bad precision");
  DevBuf a, b, c, dd, e, f, t;
  if (Tr9) HIP_TRY(to_dev(t, Tr9, sizeof(float) * 9 * n));
  HIP_TRY(to_dev(a, W, sizeof(double) * 5 * n));
  HIP_TRY(to_dev(b, Ur, sizeof(double) * n));
  HIP_TRY(to_dev(c, Fr3, sizeof(double) * 3 * n));
  HIP_TRY(to_dev(dd, ka, sizeof(double) * n));
  HIP_TRY(to_dev(e, ks, sizeof(double) * n));
  HIP_TRY(to_dev(f, nullptr, sizeof(double) * 4 * n));
  HIP_TRY(launch_eval_rad(precision == RHLLC_PREC_MIXED, n, (double *)a.p, (double *)b.p, (double *)c.p,
                          (double *)dd.p, (double *)e.p, emission, (const float *)t.p, (double *)f.p, nullptr));
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(G, f.p, sizeof(double) * 4 * n, hipMemcpyDeviceToHost));
  return RHLLC_OK;
}

extern "C" int rhllc_eval_rad_source_opt(int32_t nx, int32_t ny, const double header[6], const double *table,
                                         int64_t n, const double *W, const double *Ur, const double *Fr3,
                                         const float *Tr9, double *G, double *cell) {
  if (n < 0 || !header || !table || !W || !Ur || !Fr3 || !G || !cell) return fail(RHLLC_ERR_ARG, "bad argument");
  if (int e = check_table(nx, ny, header)) return e;
  DevBuf t, a, b, c, g, o, tt;
  if (Tr9) HIP_TRY(to_dev(tt, Tr9, sizeof(float) * 9 * n));
  HIP_TRY(to_dev(t, table, sizeof(double) * nx * ny));
  HIP_TRY(to_dev(a, W, sizeof(double) * 5 * n));
  HIP_TRY(to_dev(b, Ur, sizeof(double) * n));
  HIP_TRY(to_dev(c, Fr3, sizeof(double) * 3 * n));
  HIP_TRY(to_dev(g, nullptr, sizeof(double) * 4 * n));
  HIP_TRY(to_dev(o, nullptr, sizeof(double) * 5 * n));
  HIP_TRY(launch_eval_rad_opt(nx, ny, header, (double *)t.p, n, (double *)a.p, (double *)b.p, (double *)c.p,
                              (const float *)tt.p, (double *)g.p, (double *)o.p, nullptr));
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(G, g.p, sizeof(double) * 4 * n, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(cell, o.p, sizeof(double) * 5 * n, hipMemcpyDeviceToHost));
  return RHLLC_OK;
}

extern "C" int rhllc_copy_probe(int32_t device, int64_t nbytes, int32_t reps, double *gbps) {
  if (nbytes < 16 || reps < 1 || !gbps) return fail(RHLLC_ERR_ARG, "bad argument");
  HIP_TRY(hipSetDevice(device));
  const int64_t n16 = nbytes / 16;
  DevBuf a, b;
  HIP_TRY(to_dev(a, nullptr, (size_t)n16 * 16));
  HIP_TRY(to_dev(b, nullptr, (size_t)n16 * 16));
  HIP_TRY(hipMemset(a.p, 0, (size_t)n16 * 16));
  HIP_TRY(launch_copy(a.p, b.p, n16, nullptr));
  HIP_TRY(hipDeviceSynchronize());
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  HIP_TRY(hipEventRecord(e0, nullptr));
  for (int32_t r = 0; r < reps; ++r) HIP_TRY(launch_copy(a.p, b.p, n16, nullptr));
  HIP_TRY(hipEventRecord(e1, nullptr));
  HIP_TRY(hipEventSynchronize(e1));
  float ms = 0;
  HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  *gbps = 2.0 * (double)n16 * 16.0 * reps / (ms * 1e-3) / 1e9;
  return RHLLC_OK;
}

extern "C" int rhllc_device_query(int32_t device, char *name, int32_t name_len, int32_t *cus, double *hbm_gb) {
  hipDeviceProp_t prop;
  HIP_TRY(hipGetDeviceProperties(&prop, device));
  if (name && name_len > 0) {
    std::strncpy(name, prop.gcnArchName, (size_t)name_len - 1);
    name[name_len - 1] = 0;
  }
  if (cus) *cus = prop.multiProcessorCount;
  if (hbm_gb) *hbm_gb = (double)prop.totalGlobalMem / 1e9;
  return RHLLC_OK;
}
