// jfc_api.hip -- host driver and C-ABI of libjfcut (include/jfcut.h).
//
// The solve driver replaces QGCWidget::slotCutClicked
// (src/QVisualizer/Graph Cut/QGCWidget.cpp:2364-2558).  Differences by design:
//   - the loop stays on the device: tile lists are rebuilt by ballot
//     compaction kernels and consumed by persistent workgroups, and the host
//     reads one counter every `check_every` sweeps instead of several
//     blocking readbacks per iteration;
//   - convergence is decided by the active-tile count, which is exact because
//     heights stay a valid distance labelling (global relabel is an exact
//     BFS, colour classes never touch each other's nodes); the canonical-cut
//     search then doubles as the certificate (QGCWidget.cpp:3237-3273);
//   - the max-flow value is an int64 reduction of the absorbed deficit
//     (reduce_flow in the reference accumulates int32, reduce.cl:17-42).
#include "jfcut.h"
#include "jfcut_debug.h"
#include "jfc_internal.h"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <numeric>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

using namespace jfc;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg) {
  g_err = msg;
  return code;
}

}  // namespace

// Host-only parts of the library (graph files) report through the same
// thread-local message.
void jfc::set_last_error(const std::string &msg) { g_err = msg; }

namespace {

#define JFC_HIP(call)                                                        \
  do {                                                                       \
    hipError_t e_ = (call);                                                  \
    if (e_ != hipSuccess)                                                    \
      return fail(JFC_ERR_DEVICE, std::string(#call) + ": " +               \
                                      hipGetErrorString(e_));                \
  } while (0)

template <class T>
int dalloc(T **p, size_t n, const char *what) {
  *p = nullptr;
  if (n == 0) n = 1;
  hipError_t e = hipMalloc((void **)p, n * sizeof(T));
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
    return fail(JFC_ERR_OOM, std::string("device allocation failed: ") + what +
                                 " (" + std::to_string(n * sizeof(T)) + " bytes)");
  }
  return JFC_OK;
}

template <class T>
void dfree(T *&p) {
  if (p) (void)hipFree((void *)p);
  p = nullptr;
}

int default_shape(int dim) { return dim == 3 ? SH_8x8x4 : SH_32x8; }

int shape_from_option(int opt, int dim) {
  switch (opt) {
    case JFC_TILE_32x8: return dim == 2 ? SH_32x8 : 0;
    case JFC_TILE_64x4: return dim == 2 ? SH_64x4 : 0;
    case JFC_TILE_16x16: return dim == 2 ? SH_16x16 : 0;
    case JFC_TILE_8x8x4: return dim == 3 ? SH_8x8x4 : 0;
    case JFC_TILE_32x4x2: return dim == 3 ? SH_32x4x2 : 0;
    default: return default_shape(dim);
  }
}

// Process-wide autotuning table: size class -> JFC_TILE_* shape.
// Autotuned choices per size class: tile shape, local-iteration cap and the
// relabel before the first sweep.
struct Tuned {
  int shape = 0;
  int mli = 0;
  int ir = -1;  // initial relabel (-1: not tuned)
  int sc = -1;  // certify first on a stall (-1: not tuned)
  int sp = 0;   // cap of sparse launches (0: not tuned)
};

// Default cap on the local iterations of a launch whose list fits its grid,
// reached by doubling the dense cap once a sweep.  A launch lasts as long as
// its longest visit, which flow that goes nowhere keeps at the cap: over four
// inputs each, 12 / 16 / 24 / 32 iterations took 47 / 39 / 40 / 42 ms for
// 3750x2500 strokes and 3.08 / 3.25 / 3.20 / 3.5 ms for a 181x217x181 scan.
// At 16 from the eighth sweep on, from the first, and doubling: a 640x480
// grid 1.25 / 0.83 / 0.95 ms, a 600x450 widget cut 1.43 / 1.20 / 1.03, a
// 512x512 cut, done after four sweeps, 0.63 / 0.69 / 0.64.
constexpr int kSparseIters = 16;

// Cost of a relabel in ns: its launches, the passes over every region, a chain of
// visits as long as its longest distance, and the cut search that was tried
// before it (stall_certify).  Fitted so that stalls relabel about as often as
// they best do, at 0.7 to 1.2 of what relabels take; this and measured, in us:
// 3750x2500 strokes 750 and 960, 1500x1100 random 510 and 450, 1023x767 105 and
// 150, 4000x3000 60 and 90; 100^3 random 220 and 300, 181x217x181 scan 210 and
// 340, 256x192x176 random 360 and 520, 512^3 volume 1180 and 1560,
// 2560x1440x50 video with its cut search 4250 and 3560.
struct RelabelCost {
  long long launch, region, level, certify;
};
constexpr RelabelCost kCost2D{15000, 16, 500, 20}, kCost3D{15000, 26, 1600, 20};
// And of a sweep: its push launches, each as long as its longest visit (8 us at
// 2 iterations and 22 at 16 with 8 directions, else 6 and 18), and its tile
// visits, by the length of a tile's rows.
constexpr long long kPushNs = 5000, kIterNs8 = 1060, kIterNs = 810, kVisitNs2D = 7,
                    kVisitNs8x8x4 = 11, kVisitNs32x4x2 = 5;
constexpr int kCostIters = 64;  // visits of higher caps end before them
std::mutex g_tune_mu;
std::map<std::string, Tuned> g_tune;

int log2_round(double v) { return v <= 1.0 ? 0 : (int)std::lround(std::log2(v)); }

// Device counters (int64): [0] push tile visits, [kIterSlots, +64) local
// iterations of the push kernel, [kRegionSlots, +64) / [kFloodSlots, +64) region
// visits of the relabel / cut passes, [kDefSlots, +64) the remaining deficit of
// a one-instance graph (workgroup b adds to slot b % 64, so no single address
// takes one atomic per workgroup).
constexpr int kIterSlots = 1, kRegionSlots = kIterSlots + 64, kFloodSlots = kRegionSlots + 64,
              kDefSlots = kFloodSlots + 64, kTotals = kDefSlots + 64;
// Colour classes of at most this many tiles: a push launch gives every tile a
// workgroup of its own or nearly (a device of 256 compute units keeps
// several tile visits per unit resident), so it takes its tiles from the
// flags (no compaction launch).  The reference's fixtures (1083-1200 tiles of
// 32x8 or 16x16) solve 5-15% faster at 2048 than at 1024.
constexpr int kSmallTiles = 2048;
// words of the results block besides the per-instance ones: the counters,
// the sweep state (kSweepState ints) and 4 flag words
constexpr size_t kResFixed = kTotals + (kSweepState + 4) / 2;

// Sweeps whose stop words can be in flight at once (pinned words and events).
constexpr int kStopRing = 8;
constexpr int kQuitWord = kStopRing + 4;

// algorithmic HBM bytes per node of one push-relabel visit: read and write
// e, h and K residual planes (int32)
long long push_bytes_per_node(int K) { return 2LL * 4 * (2 + K); }

}  // namespace

struct jfc_graph {
  int dim = 2;
  int tuned = 0;           // JFC_TILE_* chosen by jfc_autotune (0 = none)
  int tuned_mli = 0;       // local-iteration cap chosen by jfc_autotune (0 = none)
  int tuned_ir = -1;       // initial relabel chosen by jfc_autotune (-1 = none)
  int tuned_sc = -1;       // stall_certify chosen by jfc_autotune (-1 = none)
  int tuned_sp = 0;        // sparse_local_iters chosen by jfc_autotune (0 = none)
  std::string size_class;  // key of the process-wide autotuning table
  int Kg = 4;  // planes stored (max K over instances)
  int shape = 0;
  long long Ntot = 0;   // nodes stored, rows padded (plane stride)
  long long Nuser = 0;  // nodes of the instances as callers number them
  void *stage = nullptr;  // device staging of caller arrays (rows of nx)
  size_t stage_bytes = 0;
  void *model_scratch = nullptr;  // data-term scratch (histograms, centres, sums)
  size_t model_scratch_bytes = 0;
  std::vector<InstDesc> inst;
  std::vector<int> caps_set;  // per instance: bit 0 terminals, bit 1 + d neighbour planes
  std::vector<int> caps_failed;  // per instance: the same bits, for a setter that failed
                                 // (its planes are zeroed; solves refuse the instance)
  // tile tables for the current shape
  int ntiles = 0, ncolors = 2, max_tile_dim = 1, nbins = 2;
  std::vector<int> color_off;
  // device planes
  int *node_block = nullptr;  // cs, ct, e, h, mask0 and rmask
  int *cs = nullptr, *ct = nullptr, *c0 = nullptr, *cap = nullptr;
  int *e = nullptr, *h = nullptr;
  unsigned char *lab = nullptr;
  unsigned char *tag = nullptr;  // tag post-process output (allocated on first use)
  // device tables / work space
  InstDesc *d_inst = nullptr;
  int *d_tile_inst = nullptr, *d_color_tiles = nullptr;
  int *d_list[2] = {nullptr, nullptr};
  int *d_ctr = nullptr;
  unsigned char *d_flag = nullptr, *d_seed = nullptr;
  unsigned char *d_mat = nullptr;  // per tile: residual planes written this solve
  unsigned char *d_hmat = nullptr; // per tile: heights stored this solve
  unsigned char *d_touched = nullptr;  // per tile: planes or masks written by a flush
  // The regions of the global relabel and of the cut and tag floods
  // (jfc_region.hip, jfc_flood.hip), the same for every push tile shape:
  // descriptors and tables like the push tiling's, the marks of two passes,
  // the packed bit planes, the borders' distances and labels.
  struct Regions {
    unsigned char *block = nullptr;  // holds every array below
    std::vector<InstDesc> inst;
    InstDesc *d_inst = nullptr;
    int *d_tile_inst = nullptr;
    int n = 0;
    unsigned char *d_dirty[2] = {nullptr, nullptr};
    int *d_any = nullptr;  // 4 words: a mark is set for pass p (slot p % 4)
    RegionBuf buf{nullptr, nullptr, nullptr, 0};
    unsigned long long *d_out = nullptr;  // floods: labels sent across borders
    unsigned char *d_open = nullptr;      // floods: regions with packed arcs
    int tag = 1;           // of the last relabel
    int seq = 0;           // passes run, the number their posted words carry
    int *d_marks = nullptr;  // words of a one-launch relabel
    int *d_far = nullptr;    // largest distances of the last relabel
    size_t mark_words() const { return (size_t)kSettleLine * (2 * kSettleSlots + n); }
    // time without progress after which a one-launch search leaves the rest to
    // passes: far above the ~50 us of a visit
    long long wait_ticks = 2000000;  // 20 ms
    bool by_passes = false;  // every search takes a launch per pass
  } rg;
  // One device block holds every word a solve reads back at its end (one
  // copy): the per-instance sums, the remaining deficits, the counters, the
  // sweep state and the flag words, in this order (res_words long longs).
  long long *d_res = nullptr;
  size_t res_words = 0;
  long long *d_red = nullptr, *d_total = nullptr;  // in d_res
  long long *d_def = nullptr;  // in d_res; per instance: remaining deficit after the cut
  long long *d_energy = nullptr;  // per instance: cut energy (jfc_get_energy)
  int *d_row_off = nullptr;    // per instance: first row; [count] = rows
  int nrows = 0;
  int *d_sweep = nullptr;
  int sweep_cap = 0;
  int last_sweeps = 0;
  int *d_flagword = nullptr;  // in d_res; [0] certificate, [1] validation
  unsigned *mask0 = nullptr;  // residual-arc bits of the input planes
  unsigned *rmask = nullptr;  // residual-arc bits of the current residual
  bool mask_dirty = true;     // inputs changed since the last solve started
  bool mask0_ok = false;      // mask0 holds the bits of the current inputs
  int slot = 0;
  bool solved = false;
  std::vector<long long> flows;
  std::vector<hipEvent_t> ev_pool;
  int nwg = 2048;
  int *d_sweep_state = nullptr;     // in d_res; {active tiles of the running sweep, sweep index}
  hipStream_t priv_stream = nullptr;  // solve stream when the caller passes NULL
  hipEvent_t priv_event = nullptr;
  // Second stream of the data term (its pair sums and pairwise weights run
  // beside the k-means and the unary terms), with the fork and join events.
  hipStream_t aux_stream = nullptr;
  hipEvent_t aux_fork = nullptr, aux_join = nullptr, aux_ready = nullptr;
  void *aux_pin = nullptr;  // pinned host words the second stream's copies use
  // The caller's stream for every call of the graph (jfc_set_stream): the
  // setters, the data term, the outputs and the backward issue their work
  // on it and wait for that stream alone.  NULL: the legacy default stream.
  hipStream_t ustream = nullptr;
  long long *pin = nullptr;  // pinned word for jfc_get_energy's sum
  // Pinned copy of d_res (the solve's results).
  long long *pin_res = nullptr;
  // Stop words the sweeps post (k_sweep_end), then the words of two groups of
  // search passes, of a setter's range check, and of a flood that gave up
  // waiting, in fine-grained pinned memory the device writes through to; d_ring
  // is its device address.
  int *ring = nullptr, *d_ring = nullptr;
  hipEvent_t cnt_ev[2] = {nullptr, nullptr};
  int ensure_pin() {
    if (pin) return JFC_OK;
    for (hipEvent_t &ev : cnt_ev)
      if (!ev && hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) {
        ev = nullptr;
        return fail(JFC_ERR_DEVICE, "event creation failed");
      }
    if (hipHostMalloc((void **)&pin, sizeof(long long), hipHostMallocDefault) != hipSuccess ||
        hipHostMalloc((void **)&pin_res, res_words * sizeof(long long), hipHostMallocDefault) !=
            hipSuccess ||
        hipHostMalloc((void **)&ring, (kStopRing + 5) * sizeof(int), hipHostMallocCoherent) !=
            hipSuccess ||
        hipHostGetDevicePointer((void **)&d_ring, ring, 0) != hipSuccess) {
      (void)hipGetLastError();
      if (pin) (void)hipHostFree(pin);
      if (pin_res) (void)hipHostFree(pin_res);
      if (ring) (void)hipHostFree(ring);
      pin = nullptr;
      pin_res = nullptr;
      ring = d_ring = nullptr;
      return fail(JFC_ERR_OOM, "pinned host words");
    }
    return JFC_OK;
  }
  ~jfc_graph() { release(); }

  void release_tiles() {
    dfree(d_tile_inst); dfree(d_color_tiles); dfree(d_list[0]); dfree(d_list[1]);
    dfree(d_flag); dfree(d_seed); dfree(d_inst); dfree(d_mat);
    dfree(d_hmat);
    dfree(d_touched);
  }
  void release_aux() {
    if (aux_fork) (void)hipEventDestroy(aux_fork);
    if (aux_join) (void)hipEventDestroy(aux_join);
    if (aux_ready) (void)hipEventDestroy(aux_ready);
    if (aux_stream) (void)hipStreamDestroy(aux_stream);
    if (aux_pin) (void)hipHostFree(aux_pin);
    aux_fork = aux_join = aux_ready = nullptr;
    aux_stream = nullptr;
    aux_pin = nullptr;
  }
  void release() {
    release_tiles();
    dfree(rg.block);
    rg = Regions{};
    dfree(node_block);
    cs = ct = e = h = nullptr;
    mask0 = rmask = nullptr;
    dfree(c0); dfree(cap); dfree(lab); dfree(tag);
    dfree(d_ctr); dfree(d_res); dfree(d_sweep); dfree(d_energy); dfree(d_row_off);
    d_red = d_total = d_def = nullptr;
    d_sweep_state = d_flagword = nullptr;
    if (stage) (void)hipFree(stage);
    stage = nullptr;
    stage_bytes = 0;
    if (model_scratch) (void)hipFree(model_scratch);
    model_scratch = nullptr;
    model_scratch_bytes = 0;
    if (priv_event) (void)hipEventDestroy(priv_event);
    if (priv_stream) (void)hipStreamDestroy(priv_stream);
    priv_event = nullptr;
    priv_stream = nullptr;
    release_aux();
    for (hipEvent_t &ev : cnt_ev) {
      if (ev) (void)hipEventDestroy(ev);
      ev = nullptr;
    }
    if (pin) (void)hipHostFree(pin);
    if (pin_res) (void)hipHostFree(pin_res);
    if (ring) (void)hipHostFree(ring);
    pin = nullptr;
    pin_res = nullptr;
    ring = d_ring = nullptr;
    for (hipEvent_t ev : ev_pool) (void)hipEventDestroy(ev);
    ev_pool.clear();
  }

  Tiles tiles() const {
    // the whole-graph passes stream 4-node groups, 1024 per workgroup step:
    // a one-instance graph with short rows takes several rows per step
    int step = 1;
    if (inst.size() == 1) step = std::max(1, 1024 / ((inst[0].nx + 3) / 4));
    return Tiles{d_inst, d_tile_inst, ntiles, d_row_off, (int)inst.size(), nrows, step,
                 inst.empty() ? InstDesc{} : inst[0]};
  }
  Planes planes() const { return Planes{e, h, cap, c0, cs, ct, lab, Ntot, rmask}; }
  int max_nx() const {
    int m = 1;
    for (const InstDesc &I : inst) m = std::max(m, I.nx);
    return m;
  }
  int first_row(int i) const {
    int r = 0;
    for (int k = 0; k < i; ++k) r += inst[k].ny * inst[k].nz;
    return r;
  }
  long long inst_nodes(int i) const {
    return (long long)inst[i].nx * inst[i].ny * inst[i].nz;
  }
  long long inst_stored(int i) const {
    return (long long)inst[i].px * inst[i].ny * inst[i].nz;
  }

  // Build tile tables, colour classes and instance descriptors for `sh`.
  int set_shape(int sh) {
    if (sh == shape && d_tile_inst) return JFC_OK;
    release_tiles();
    shape = sh;
    int tw, th, td;
    shape_dims(sh, &tw, &th, &td);
    bool all4 = true;
    long long off = 0;
    max_tile_dim = 1;
    int maxsum = 0;
    for (auto &I : inst) {
      I.tx = (I.nx + tw - 1) / tw;
      I.ty = (I.ny + th - 1) / th;
      I.tz = (I.nz + td - 1) / td;
      const long long nt = (long long)I.tx * I.ty * I.tz;
      if (off + nt >= kEntryTile) return fail(JFC_ERR_INVALID, "graph too large for the tile queue");
      I.tile_off = (int)off;
      I.ntiles = (int)nt;
      off += nt;
      if (I.K != 4) all4 = false;
      max_tile_dim = std::max(max_tile_dim, std::max(I.tx, std::max(I.ty, I.tz)));
      maxsum = std::max(maxsum, I.tx + I.ty + I.tz);
    }
    ntiles = (int)off;
    // distance bins of the tile ordering (the last bin holds tiles of
    // instances without seed tiles); farther tiles share the last finite bin
    nbins = std::min(maxsum + 2, 4096);
    // colour classes: tiles of one class are never adjacent through an arc,
    // so no node is in one tile of the class and in the halo of another it
    // pushes across.  2D 4C and 3D 6C: checkerboard; 2D 8C: 2x2 pattern.
    ncolors = (dim == 2 && !all4) ? 4 : 2;
    const bool one = inst.size() == 1;  // (its tiles' instance is 0)
    std::vector<int> tile_inst(one ? 0 : ntiles);
    std::vector<std::vector<int>> cls(ncolors);
    for (size_t i = 0; i < inst.size(); ++i) {
      const InstDesc &I = inst[i];
      for (int z = 0; z < I.tz; ++z)
        for (int y = 0; y < I.ty; ++y)
          for (int x = 0; x < I.tx; ++x) {
            const int t = I.tile_off + x + I.tx * (y + I.ty * z);
            if (!one) tile_inst[t] = (int)i;
            const int c = ncolors == 4 ? ((x & 1) | ((y & 1) << 1)) : ((x + y + z) & 1);
            cls[c].push_back(t);
          }
    }
    std::vector<int> flat;
    color_off.assign(ncolors + 1, 0);
    for (int c = 0; c < ncolors; ++c) {
      color_off[c] = (int)flat.size();
      flat.insert(flat.end(), cls[c].begin(), cls[c].end());
    }
    color_off[ncolors] = (int)flat.size();
    int rc;
    if ((rc = dalloc(&d_inst, inst.size(), "instances")) ||
        (rc = dalloc(&d_tile_inst, ntiles, "tile table")) ||
        (rc = dalloc(&d_color_tiles, ntiles, "colour classes")) ||
        (rc = dalloc(&d_list[0], ntiles, "tile list")) ||
        (rc = dalloc(&d_list[1], ntiles, "tile list")) ||
        (rc = dalloc(&d_flag, ntiles, "tile flags")) ||
        (rc = dalloc(&d_seed, ntiles, "tile seeds")) ||
        (rc = dalloc(&d_mat, ntiles, "tile states")) ||
        (rc = dalloc(&d_hmat, ntiles, "tile states")) ||
        (rc = dalloc(&d_touched, ntiles, "tile states")))
      return rc;
    JFC_HIP(hipMemcpy(d_inst, inst.data(), inst.size() * sizeof(InstDesc), hipMemcpyHostToDevice));
    if (one) launch_fill_i32(d_tile_inst, ntiles, 0, 0);  // (done before the copy behind it)
    else JFC_HIP(hipMemcpy(d_tile_inst, tile_inst.data(), ntiles * sizeof(int), hipMemcpyHostToDevice));
    JFC_HIP(hipMemcpy(d_color_tiles, flat.data(), ntiles * sizeof(int), hipMemcpyHostToDevice));
    return JFC_OK;
  }

  // The relabel's region tables and buffers (once per graph).
  int build_regions() {
    const bool d3 = dim == 3;
    int tw, th, td;
    region_dims(d3, &tw, &th, &td);
    rg.inst = inst;
    long long off = 0;
    for (auto &I : rg.inst) {
      I.tx = (I.nx + tw - 1) / tw;
      I.ty = (I.ny + th - 1) / th;
      I.tz = (I.nz + td - 1) / td;
      const long long nt = (long long)I.tx * I.ty * I.tz;
      if (off + nt >= kEntryTile) return fail(JFC_ERR_INVALID, "graph too large for the tile queue");
      I.tile_off = (int)off;
      I.ntiles = (int)nt;
      off += nt;
    }
    rg.n = (int)off;
    rg.buf.planes = Kg + region_state_planes();
    const size_t border = (size_t)rg.n * region_border_words(d3);
    // one allocation, carved in 256-byte steps (the first walk sizes it)
    const size_t n = rg.n;
    unsigned char *base = nullptr;
    for (size_t total = 0;;) {
      size_t off2 = 0;
      auto carve = [&](auto *&p, size_t count) {
        p = (std::remove_reference_t<decltype(p)>)(base ? base + off2 : nullptr);
        off2 += (count * sizeof(*p) + 255) / 256 * 256;
      };
      carve(rg.buf.packed, n * rg.buf.planes * 64);
      carve(rg.buf.border, border);
      carve(rg.d_out, n * flood_out_words(d3));
      carve(rg.buf.base, n);
      carve(rg.d_inst, rg.inst.size());
      carve(rg.d_tile_inst, n);
      carve(rg.d_any, 4);
      carve(rg.d_far, kFarSlots * kFarLine);
      carve(rg.d_marks, rg.mark_words());
      carve(rg.d_dirty[0], n);
      carve(rg.d_dirty[1], n);
      carve(rg.d_open, n);
      if (total) break;
      total = off2;
      if (int rc = dalloc(&rg.block, total, "regions")) return rc;
      base = rg.block;
    }
    launch_fill_i32(rg.buf.border, (long long)border, 0, 0);
    JFC_HIP(hipMemcpy(rg.d_inst, rg.inst.data(), rg.inst.size() * sizeof(InstDesc),
                      hipMemcpyHostToDevice));
    if (rg.inst.size() == 1) {
      launch_fill_i32(rg.d_tile_inst, rg.n, 0, 0);
      return JFC_OK;
    }
    std::vector<int> tile_inst(rg.n);
    for (size_t i = 0; i < rg.inst.size(); ++i) {
      const InstDesc &I = rg.inst[i];
      std::fill(tile_inst.begin() + I.tile_off, tile_inst.begin() + I.tile_off + I.ntiles, (int)i);
    }
    JFC_HIP(hipMemcpy(rg.d_tile_inst, tile_inst.data(), rg.n * sizeof(int),
                      hipMemcpyHostToDevice));
    return JFC_OK;
  }
  Tiles region_tiles() const {
    Tiles T = tiles();
    T.inst = rg.d_inst;
    T.tile_inst = rg.d_tile_inst;
    T.ntiles = rg.n;
    T.one = rg.inst.empty() ? InstDesc{} : rg.inst[0];
    return T;
  }
};

// ---- accessors for the data-term file ---------------------------------------------

namespace jfc {
int model_fail(int code, const std::string &msg) { return fail(code, msg); }

int graph_instance(jfc_graph *g, int inst, InstDesc *I, int **cs, int **ct, int **c0,
                   long long *stride) {
  if (!g) return fail(JFC_ERR_INVALID, "null graph");
  if (inst < 0 || inst >= (int)g->inst.size())
    return fail(JFC_ERR_INVALID, "instance index out of range");
  *I = g->inst[inst];
  *cs = g->cs;
  *ct = g->ct;
  *c0 = g->c0;
  *stride = g->Ntot;
  return JFC_OK;
}

void graph_mark_inputs(jfc_graph *g, int inst) {
  g->caps_set[inst] = ~0;
  g->caps_failed[inst] = 0;
  g->mask_dirty = true;
  g->solved = false;
}

// A data-term call that failed after writing some of the instance's planes.
void graph_inputs_failed(jfc_graph *g, int inst) {
  g->caps_set[inst] = 0;
  g->caps_failed[inst] = ~0;
  g->mask_dirty = true;
  g->solved = false;
}

hipStream_t graph_stream(jfc_graph *g) { return g->ustream; }

int graph_stage(jfc_graph *g, size_t bytes, void **p);

// The graph's scratch block for the data-term paths, allocated on first use
// and grown when a call needs more.
int graph_scratch(jfc_graph *g, size_t bytes, void **p) {
  if (g->model_scratch_bytes < bytes) {
    if (g->model_scratch) (void)hipFree(g->model_scratch);
    g->model_scratch = nullptr;
    g->model_scratch_bytes = 0;
    if (hipMalloc(&g->model_scratch, bytes) != hipSuccess) {
      (void)hipGetLastError();
      return fail(JFC_ERR_OOM, "out of device memory: data-term scratch");
    }
    g->model_scratch_bytes = bytes;
  }
  *p = g->model_scratch;
  return JFC_OK;
}

// The data term's second stream, its fork / join / ready events and its
// pinned host words (`pin_bytes`): created on first use when `create` is
// set; otherwise null until then (the caller then runs on one stream).
int graph_aux(jfc_graph *g, bool create, size_t pin_bytes, GraphAux *a) {
  if (!g->aux_stream && create) {
    if (hipStreamCreateWithFlags(&g->aux_stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&g->aux_fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&g->aux_join, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&g->aux_ready, hipEventDisableTiming) != hipSuccess ||
        hipHostMalloc(&g->aux_pin, pin_bytes, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      g->release_aux();
      return fail(JFC_ERR_DEVICE, "cannot create the data term's second stream");
    }
  }
  a->st = g->aux_stream;
  a->fork = g->aux_fork;
  a->join = g->aux_join;
  a->ready = g->aux_ready;
  a->pin = g->aux_pin;
  return JFC_OK;
}

// The instance's slice of the excess plane (stored nodes), free between
// solves: every solve rewrites it from the inputs before reading it.
int graph_work_plane(jfc_graph *g, int inst, int **plane, long long *n) {
  *plane = g->e + g->inst[inst].node_off;
  *n = g->inst_stored(inst);
  return JFC_OK;
}
// The instance's slice of the height plane, free between solves as well.
int graph_work_plane2(jfc_graph *g, int inst, int **plane) {
  *plane = g->h + g->inst[inst].node_off;
  return JFC_OK;
}
}  // namespace jfc

// ---- lifetime -------------------------------------------------------------------

extern "C" const char *jfc_last_error(void) { return g_err.c_str(); }

extern "C" void jfc_default_options(jfc_options *o) {
  if (!o) return;
  std::memset(o, 0, sizeof(*o));
  o->max_sweeps = 1 << 20;
  o->check_every = 2;
  o->relabel_work = 2.0;
  o->max_local_iters = 0;
  o->tile_shape = JFC_TILE_DEFAULT;
  o->profile = 0;
  o->stream = nullptr;
  o->initial_relabel = -1;
  o->stall_ratio = 0.99;
  o->graph_sweeps = 1;
  o->tile_order = 0;
  o->method = JFC_METHOD_JFCUT;
  o->sparse_local_iters = 0;
  o->stall_certify = -1;
}

static int create_impl(jfc_graph **out, int count, const int32_t *shapes) {
  if (!out) return fail(JFC_ERR_INVALID, "null graph pointer");
  *out = nullptr;
  if (count <= 0 || !shapes) return fail(JFC_ERR_INVALID, "empty batch");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
    (void)hipGetLastError();
    return fail(JFC_ERR_DEVICE, "no HIP device available");
  }
  jfc_graph *g = new jfc_graph();
  long long off = 0, uoff = 0;
  g->dim = shapes[2] > 1 ? 3 : 2;
  g->Kg = 0;
  for (int i = 0; i < count; ++i) {
    const int nx = shapes[4 * i], ny = shapes[4 * i + 1], nz = shapes[4 * i + 2],
              conn = shapes[4 * i + 3];
    const int dim = nz > 1 ? 3 : 2;
    bool ok = nx > 0 && ny > 0 && nz > 0 && dim == g->dim &&
              ((dim == 2 && (conn == 4 || conn == 8)) || (dim == 3 && conn == 6));
    if (dim == 3 && conn != 6) ok = false;
    if (!ok) {
      delete g;
      return fail(JFC_ERR_INVALID, "instance " + std::to_string(i) +
                                       ": unsupported shape/connectivity (2D: 4 or 8, 3D: 6; "
                                       "all instances of one graph share the dimensionality)");
    }
    InstDesc I{};
    I.nx = nx; I.ny = ny; I.nz = nz; I.conn = conn; I.K = conn;
    I.px = (int)(((long long)nx + 31) / 32 * 32);
    I.node_off = off;
    I.user_off = uoff;
    off += (long long)I.px * ny * nz;
    uoff += (long long)nx * ny * nz;
    g->inst.push_back(I);
    g->Kg = std::max(g->Kg, conn);
  }
  if (off >= (1LL << 40)) { delete g; return fail(JFC_ERR_INVALID, "graph too large"); }
  g->Ntot = off;
  g->Nuser = uoff;
  g->caps_set.assign(count, 0);
  g->caps_failed.assign(count, 0);
  g->flows.assign(count, 0);
  int rc;
  const size_t N = (size_t)off;
  // the planes of one word per node in one block: an allocation of megabytes
  // takes 20 to 30 us, and freeing it more
  if ((rc = dalloc(&g->node_block, 6 * N, "node planes")) ||
      (rc = dalloc(&g->c0, N * g->Kg, "neighbour capacities")) ||
      (rc = dalloc(&g->cap, N * g->Kg, "residual capacities")) ||
      (rc = dalloc(&g->lab, N, "labels")) || (rc = dalloc(&g->d_ctr, 2 * QSLOT, "queues")) ||
      (rc = dalloc(&g->d_res, kResFixed + (size_t)count * (RED_SLOTS + 1), "results")) ||
      (rc = dalloc(&g->d_energy, (size_t)count, "reductions")) ||
      (rc = dalloc(&g->d_row_off, (size_t)count + 1, "row table"))) {
    delete g;
    return rc;
  }
  // (rows are padded to 32 nodes, so every plane starts at a multiple of 128 bytes)
  int *const plane[6] = {g->node_block,         g->node_block + N,     g->node_block + 2 * N,
                         g->node_block + 3 * N, g->node_block + 4 * N, g->node_block + 5 * N};
  g->cs = plane[0];
  g->ct = plane[1];
  g->e = plane[2];
  g->h = plane[3];
  g->mask0 = (unsigned *)plane[4];
  g->rmask = (unsigned *)plane[5];
  g->res_words = kResFixed + (size_t)count * (RED_SLOTS + 1);
  g->d_red = g->d_res;
  g->d_def = g->d_red + (size_t)count * RED_SLOTS;
  g->d_total = g->d_def + count;
  g->d_sweep_state = (int *)(g->d_total + kTotals);
  g->d_flagword = g->d_sweep_state + kSweepState;
  {
    std::vector<int> row_off(count + 1, 0);
    long long rows = 0;
    for (int i = 0; i < count; ++i) {
      row_off[i] = (int)rows;
      rows += (long long)g->inst[i].ny * g->inst[i].nz;
    }
    if (rows >= (1LL << 31)) { delete g; return fail(JFC_ERR_INVALID, "graph too large"); }
    row_off[count] = (int)rows;
    g->nrows = (int)rows;
    if (hipMemcpy(g->d_row_off, row_off.data(), row_off.size() * sizeof(int),
                  hipMemcpyHostToDevice) != hipSuccess) {
      delete g;
      return fail(JFC_ERR_DEVICE, "row table upload failed");
    }
  }
  // everything zero, so the pad nodes of the rows stay isolated and empty
  launch_fill_i32(g->node_block, 6 * off, 0, 0);
  launch_fill_i32(g->c0, off * g->Kg, 0, 0);
  launch_fill_i32(g->cap, off * g->Kg, 0, 0);
  launch_fill_u8(g->lab, off, 0, 0);
  int dev = 0;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
    g->nwg = std::max(64, prop.multiProcessorCount * 8);
  {
    unsigned conns = 0;
    for (const auto &I : g->inst) conns |= 1u << I.conn;
    const double mean = (double)uoff / count;
    g->size_class = std::to_string(g->dim) + ":" + std::to_string(conns) + ":" +
                    std::to_string(log2_round(count)) + ":" + std::to_string(log2_round(mean));
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tune.find(g->size_class);
    if (it != g_tune.end()) {
      g->tuned = it->second.shape;
      g->tuned_mli = it->second.mli;
      g->tuned_ir = it->second.ir;
      g->tuned_sc = it->second.sc;
      g->tuned_sp = it->second.sp;
    }
  }
  if ((rc = g->set_shape(default_shape(g->dim))) || (rc = g->build_regions())) {
    delete g;
    return rc;
  }
  if (hipDeviceSynchronize() != hipSuccess) {
    delete g;
    return fail(JFC_ERR_DEVICE, "device initialisation failed");
  }
  *out = g;
  return JFC_OK;
}

extern "C" int jfc_create(jfc_graph **g, int dims, int nx, int ny, int nz,
                          int connectivity) {
  if (dims == 2 && nz != 1) return fail(JFC_ERR_INVALID, "2D graph needs nz == 1");
  if (dims == 3 && nz < 2) return fail(JFC_ERR_INVALID, "3D graph needs nz >= 2");
  if (dims != 2 && dims != 3) return fail(JFC_ERR_INVALID, "dims must be 2 or 3");
  const int32_t s[4] = {nx, ny, nz, connectivity};
  return create_impl(g, 1, s);
}

extern "C" int jfc_create_batch(jfc_graph **g, int count, const int32_t *shapes) {
  return create_impl(g, count, shapes);
}

extern "C" void jfc_destroy(jfc_graph *g) {
  if (!g) return;
  (void)hipDeviceSynchronize();
  delete g;
}

extern "C" int jfc_num_instances(const jfc_graph *g) {
  return g ? (int)g->inst.size() : 0;
}

// ---- inputs ------------------------------------------------------------------------

static int check_inst(jfc_graph *g, int inst) {
  if (!g) return fail(JFC_ERR_INVALID, "null graph");
  if (inst < 0 || inst >= (int)g->inst.size())
    return fail(JFC_ERR_INVALID, "instance index out of range");
  return JFC_OK;
}

// Caller arrays (rows of nx) <-> stored planes (rows of px); pad entries of
// the stored side are left as they are (zero from creation).  Host arrays
// cross PCIe in one contiguous copy through the graph's device staging
// buffer; the row scatter / gather is a device-to-device 2D copy.  Every copy
// and kernel of an entry point is issued on the graph's stream (ustream), and
// the entry point waits for that stream alone before it returns (sync_user).
static int stage_for(jfc_graph *g, size_t bytes, void **p) {
  if (g->stage_bytes < bytes) {
    if (g->stage) (void)hipFree(g->stage);
    g->stage = nullptr;
    g->stage_bytes = 0;
    if (hipMalloc(&g->stage, bytes) != hipSuccess) {
      (void)hipGetLastError();
      return fail(JFC_ERR_OOM, "out of device memory: staging buffer");
    }
    g->stage_bytes = bytes;
  }
  *p = g->stage;
  return JFC_OK;
}
int jfc::graph_stage(jfc_graph *g, size_t bytes, void **p) { return stage_for(g, bytes, p); }

static int sync_user(jfc_graph *g) {
  JFC_HIP(hipStreamSynchronize(g->ustream));
  return JFC_OK;
}
static int put_rows(jfc_graph *g, const InstDesc &I, void *dst, const void *src, size_t elem,
                    int on_device) {
  const size_t row = (size_t)I.nx * elem, rows = (size_t)I.ny * I.nz;
  hipStream_t st = g->ustream;
  if (I.px == I.nx) {
    JFC_HIP(hipMemcpyAsync(dst, src, row * rows,
                           on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, st));
    return JFC_OK;
  }
  if (!on_device) {
    void *tmp = nullptr;
    if (int rc = stage_for(g, row * rows, &tmp)) return rc;
    JFC_HIP(hipMemcpyAsync(tmp, src, row * rows, hipMemcpyHostToDevice, st));
    src = tmp;
  }
  JFC_HIP(hipMemcpy2DAsync(dst, (size_t)I.px * elem, src, row, row, rows,
                           hipMemcpyDeviceToDevice, st));
  return JFC_OK;
}
static int get_rows(jfc_graph *g, const InstDesc &I, void *dst, const void *src, size_t elem,
                    int on_device) {
  const size_t row = (size_t)I.nx * elem, rows = (size_t)I.ny * I.nz;
  hipStream_t st = g->ustream;
  if (I.px == I.nx) {
    JFC_HIP(hipMemcpyAsync(dst, src, row * rows,
                           on_device ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, st));
    return JFC_OK;
  }
  if (on_device) {
    JFC_HIP(hipMemcpy2DAsync(dst, row, src, (size_t)I.px * elem, row, rows,
                             hipMemcpyDeviceToDevice, st));
    return JFC_OK;
  }
  void *tmp = nullptr;
  if (int rc = stage_for(g, row * rows, &tmp)) return rc;
  JFC_HIP(hipMemcpy2DAsync(tmp, row, src, (size_t)I.px * elem, row, rows,
                           hipMemcpyDeviceToDevice, st));
  JFC_HIP(hipMemcpyAsync(dst, tmp, row * rows, hipMemcpyDeviceToHost, st));
  return JFC_OK;
}
// A kernel may read the bytes at p in place: within one allocation, on the
// device that holds `own`.  Anything else is left to a copy, which takes it (another
// device's memory) or refuses it.
static bool readable_in_place(const void *p, size_t bytes, const void *own) {
  hipPointerAttribute_t at{}, mine{};
  hipDeviceptr_t base = nullptr;
  size_t size = 0;
  if (hipPointerGetAttributes(&at, p) != hipSuccess || at.type != hipMemoryTypeDevice ||
      hipPointerGetAttributes(&mine, own) != hipSuccess || at.device != mine.device ||
      hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return (const char *)p + bytes <= (const char *)base + size;
}

// Capacity planes of the caller onto the stored ones with their range check,
// on the graph's stream; waits for the stream.  Device arrays are read in
// place; others cross in one copy each, to the stored plane itself where its
// rows have no padding (signed values: to the instance's slice of the excess
// plane, which every solve rewrites before reading it), else through the
// staging buffer.  Returns JFC_ERR_OVERFLOW naming the first plane with a
// value outside [lo, hi].
static int put_caps(jfc_graph *g, int inst, const PutPlanes &planes, int on_device, bool excess,
                    int dir, int lo, int hi, const char *const *what) {
  if (int rc = g->ensure_pin()) return rc;
  const InstDesc &I = g->inst[inst];
  const size_t bytes = (size_t)I.nx * I.ny * I.nz * sizeof(int32_t);
  volatile int *const bad = g->ring + kStopRing + 2;
  int *const d_bad = g->d_ring + kStopRing + 2;
  bad[0] = bad[1] = 0;
  const bool direct = on_device && readable_in_place(planes.src[0], bytes, g->cs) &&
                      (!planes.src[1] || readable_in_place(planes.src[1], bytes, g->cs));
  if (direct) {
    launch_put(I, planes, excess, dir, lo, hi, d_bad, g->ustream);
  } else {
    for (int k = 0; k < 2 && planes.src[k]; ++k) {
      void *at = excess ? g->e + I.node_off : planes.dst[k];
      if (I.px != I.nx)
        if (int rc = stage_for(g, bytes, &at)) return rc;
      JFC_HIP(hipMemcpyAsync(at, planes.src[k], bytes,
                             on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice,
                             g->ustream));
      launch_put(I, {{(const int *)at, nullptr}, {planes.dst[k], planes.dst[1]}}, excess, dir, lo, hi,
                 d_bad + k, g->ustream);
    }
  }
  JFC_HIP(hipGetLastError());
  if (int rc = sync_user(g)) return rc;
  const int out = bad[0] ? 0 : bad[1] ? 1 : -1;
  if (out >= 0)
    return fail(JFC_ERR_OVERFLOW, std::string(what[out]) + " outside [" + std::to_string(lo) +
                                      ", " + std::to_string(hi) + "]");
  return JFC_OK;
}

// A setter that failed leaves the plane(s) it wrote zeroed and the instance
// marked incomplete: the solve refuses it until the inputs are set again.
static void input_failed(jfc_graph *g, int inst, int bits) {
  g->caps_set[inst] &= ~bits;
  g->caps_failed[inst] |= bits;
  g->mask_dirty = true;
  g->solved = false;
}

extern "C" int jfc_set_stream(jfc_graph *g, void *stream) {
  if (!g) return fail(JFC_ERR_INVALID, "null graph");
  g->ustream = (hipStream_t)stream;
  return JFC_OK;
}

extern "C" int jfc_set_terminal_caps(jfc_graph *g, int inst, const int32_t *cap_source,
                                     const int32_t *cap_sink, int on_device) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  if (!cap_source || !cap_sink) return fail(JFC_ERR_INVALID, "null capacity pointer");
  const long long n = g->inst_stored(inst);
  const long long o = g->inst[inst].node_off;
  static const char *const what[2] = {"source capacity", "sink capacity"};
  rc = put_caps(g, inst, {{cap_source, cap_sink}, {g->cs + o, g->ct + o}}, on_device, false, -1, 0,
                JFC_MAX_TERMINAL_CAP, what);
  if (rc) {
    launch_fill_i32(g->cs + o, n, 0, g->ustream);
    launch_fill_i32(g->ct + o, n, 0, g->ustream);
    (void)hipStreamSynchronize(g->ustream);
    input_failed(g, inst, 1);
    return rc;
  }
  g->caps_set[inst] |= 1;
  g->caps_failed[inst] &= ~1;
  g->solved = false;
  return JFC_OK;
}

extern "C" int jfc_set_excess(jfc_graph *g, int inst, const int32_t *ef, int on_device) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  if (!ef) return fail(JFC_ERR_INVALID, "null excess pointer");
  const long long n = g->inst_stored(inst);
  const long long o = g->inst[inst].node_off;
  static const char *const what[1] = {"excess"};
  rc = put_caps(g, inst, {{ef, nullptr}, {g->cs + o, g->ct + o}}, on_device, true, -1,
                -JFC_MAX_TERMINAL_CAP, JFC_MAX_TERMINAL_CAP, what);
  if (rc) {
    launch_fill_i32(g->cs + o, n, 0, g->ustream);
    launch_fill_i32(g->ct + o, n, 0, g->ustream);
    (void)hipStreamSynchronize(g->ustream);
    input_failed(g, inst, 1);
    return rc;
  }
  g->caps_set[inst] |= 1;
  g->caps_failed[inst] &= ~1;
  g->solved = false;
  return JFC_OK;
}

extern "C" int jfc_set_neighbor_caps(jfc_graph *g, int inst, int arc, const int32_t *cap,
                                     int on_device) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  if (!cap) return fail(JFC_ERR_INVALID, "null capacity pointer");
  if (arc < 0 || arc >= g->inst[inst].K)
    return fail(JFC_ERR_INVALID, "arc index outside the instance's connectivity");
  const long long n = g->inst_stored(inst);
  int *dst = g->c0 + (long long)arc * g->Ntot + g->inst[inst].node_off;
  static const char *const what[1] = {"neighbour capacity"};
  rc = put_caps(g, inst, {{cap, nullptr}, {dst, nullptr}}, on_device, false, arc, 0,
                JFC_MAX_NEIGHBOR_CAP, what);
  // on failure the plane is zeroed and the mask of the inputs is rebuilt
  // before the next solve, so no stale residual bit of the old arcs survives
  g->mask_dirty = true;
  g->solved = false;
  if (rc) {
    launch_fill_i32(dst, n, 0, g->ustream);
    (void)hipStreamSynchronize(g->ustream);
    input_failed(g, inst, 2 << arc);
    return rc;
  }
  g->caps_set[inst] |= 2 << arc;
  g->caps_failed[inst] &= ~(2 << arc);
  return JFC_OK;
}

extern "C" int jfc_set_seeds(jfc_graph *g, int inst, const uint8_t *fg, const uint8_t *bg,
                             int on_device) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  const InstDesc &I = g->inst[inst];
  const long long o = I.node_off;
  const long long rows = (long long)I.ny * I.nz, n = rows * I.nx;
  // the kernel reads the caller's unpadded seed bytes; host bytes are staged
  // in one contiguous copy each
  const unsigned char *dfg = fg, *dbg = bg;
  if (!on_device && (fg || bg)) {
    void *tmp = nullptr;
    if ((rc = stage_for(g, 2 * (size_t)n, &tmp))) return rc;
    unsigned char *s = (unsigned char *)tmp;
    if (fg) JFC_HIP(hipMemcpyAsync(s, fg, n, hipMemcpyHostToDevice, g->ustream));
    if (bg) JFC_HIP(hipMemcpyAsync(s + n, bg, n, hipMemcpyHostToDevice, g->ustream));
    dfg = fg ? s : nullptr;
    dbg = bg ? s + n : nullptr;
  }
  launch_seeds(g->cs + o, g->ct + o, dfg, dbg, I.nx, I.px, rows, g->ustream);
  if ((rc = sync_user(g))) return rc;
  g->caps_set[inst] |= 1;
  g->solved = false;
  return JFC_OK;
}

extern "C" int jfc_input_planes(jfc_graph *g, int inst, int32_t **cap_source,
                                int32_t **cap_sink, int32_t **neighbor, int64_t *row_pitch,
                                int64_t *plane_stride) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  const long long o = g->inst[inst].node_off;
  if (cap_source) *cap_source = g->cs + o;
  if (cap_sink) *cap_sink = g->ct + o;
  if (neighbor) *neighbor = g->c0 + o;
  if (row_pitch) *row_pitch = g->inst[inst].px;
  if (plane_stride) *plane_stride = g->Ntot;
  return JFC_OK;
}

extern "C" int jfc_inputs_written(jfc_graph *g, int inst) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  graph_mark_inputs(g, inst);
  return JFC_OK;
}

// ---- solve -------------------------------------------------------------------------------

namespace {

struct Timer {
  std::vector<hipEvent_t> *pool;
  size_t used = 0;
  hipStream_t st;
  hipEvent_t next() {
    if (used == pool->size()) {
      hipEvent_t ev;
      if (hipEventCreate(&ev) != hipSuccess) return nullptr;
      pool->push_back(ev);
    }
    return (*pool)[used++];
  }
  hipEvent_t mark() {
    hipEvent_t ev = next();
    if (ev) (void)hipEventRecord(ev, st);
    return ev;
  }
  static double ms(hipEvent_t a, hipEvent_t b) {
    float f = 0.f;
    if (a && b && hipEventElapsedTime(&f, a, b) == hipSuccess) return f;
    return 0.0;
  }
};

struct Solver {
  jfc_graph *g;
  jfc_options o;
  jfc_stats s;
  hipStream_t st;
  Timer tm;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> push_ev, gr_ev, cut_ev;

  SweepCtl sweep_ctl() const {
    SweepCtl c;
    c.hist = g->d_sweep;
    c.state = g->d_sweep_state;
    c.total = g->d_total;
    c.cap = g->sweep_cap;
    c.max_sweeps = o.max_sweeps;
    c.stall_ratio = o.stall_ratio;
    c.budget = o.relabel_work > 0 ? (long long)std::floor(o.relabel_work * g->ntiles) : 0;
    c.ring = g->d_ring;
    c.ring_n = kStopRing;
    const int cap = std::min(std::max(o.max_local_iters, o.sparse_local_iters), kCostIters);
    c.sweep_ns = (kPushNs + cap * (g->Kg == 8 ? kIterNs8 : kIterNs)) *
                 (o.method == JFC_METHOD_FASTCUT ? 2 + 2 * g->dim : g->ncolors);
    c.visit_ns = g->dim == 2 ? kVisitNs2D : g->shape == SH_8x8x4 ? kVisitNs8x8x4 : kVisitNs32x4x2;
    const RelabelCost &cost = g->dim == 3 ? kCost3D : kCost2D;
    c.relabel_ns = cost.launch + (cost.region + (o.stall_certify > 0 ? cost.certify : 0)) * g->rg.n;
    c.level_ns = cost.level;
    c.far = g->rg.d_far;
    return c;
  }

  Queue queue_from_list() {
    Queue q{g->d_list[g->slot], g->d_ctr, g->slot, -1};
    return q;
  }
  void advance() { g->slot ^= 1; }

  // Passes over the regions until no region is marked: `issue(kind, ctl)`
  // launches one.  Passes go out in groups, one group ahead of the host's
  // check, so the device is not idle during it.  A pass with no mark returns at
  // once and says so in its group's word.  The first groups are short, as
  // most searches of dense graphs settle within them; later ones grow, as
  // each check costs a gap of about 6 us between two passes.
  // packed: the regions are packed, and every one is marked for the first pass.
  template <class Issue>
  int region_passes(int slots, int *passes, bool packed, Issue issue) {
    if (int rc = g->ensure_pin()) return rc;
    auto &rg = g->rg;
    int pass = 0;
    auto next = [&](int kind, int group) {
      PassCtl c;
      c.dirty_in = rg.d_dirty[pass & 1];
      c.dirty_out = rg.d_dirty[(pass + 1) & 1];
      c.any_in = rg.d_any + (pass & 3);
      c.any_out = rg.d_any + ((pass + 1) & 3);
      c.any_clear = rg.d_any + ((pass + 2) & 3);
      c.post = g->d_ring + kStopRing + group;
      c.seq = rg.seq = (rg.seq + 1) & 0xffffff;
      c.visits = g->d_total + slots;
      issue(kind, c);
      ++pass;
    };
    if (!packed) next(kPack, 0);
    int want[2] = {0, 0};
    auto issue_group = [&](int k) -> int {
      const int size = k < 2 ? 2 : k < 4 ? 4 : 8;
      for (int j = 0; j < size; ++j) next(kBorders, k & 1);
      want[k & 1] = rg.seq;
      JFC_HIP(hipEventRecord(g->cnt_ev[k & 1], st));
      return JFC_OK;
    };
    if (int rc = issue_group(0)) return rc;
    for (int k = 0;; ++k) {
      if (int rc = issue_group(k + 1)) return rc;
      JFC_HIP(hipEventSynchronize(g->cnt_ev[k & 1]));
      const volatile int *word = g->ring + kStopRing + (k & 1);
      int w = *word;
      for (int spin = 0; (w >> 1) != want[k & 1] && spin < (1 << 20); ++spin) w = *word;
      if ((w >> 1) != want[k & 1])
        return fail(JFC_ERR_DEVICE, "a search pass's word did not reach the host");
      if (!(w & 1)) break;
      if (pass > 1000000) return fail(JFC_ERR_STATE, "search did not settle");
    }
    next(kFinal, 0);
    *passes += pass;
    return JFC_OK;
  }

  // The zeroing region passes need, to go into their caller's fill launch.
  void region_fills(FillSet &f) const {
    f.add(g->rg.d_dirty[0], g->rg.n, 0, 1);
    f.add(g->rg.d_dirty[1], g->rg.n, 0, 1);
    f.add(g->rg.d_any, 4, 0, 4);
  }

  // Every region marked for the first of the passes that finish a search.
  void mark_all_regions() {
    FillSet f;
    region_fills(f);
    f.seg[0].v = 1;
    f.seg[2].v = 1;
    launch_fill_multi(f, st);
  }

  // The searches go by passes: one gave up waiting, as something else holds places
  // on the device, or the graph has it so.
  bool by_passes = false;

  // A cut or tag flood over the regions (jfc_flood.hip).  fills: zeroing of the
  // caller's, done in the same launch.  Where one launch takes every pass the
  // stream has to be waited for and finish_flood() asked afterwards.
  int flood(bool tag, bool stop, FillSet fills, int *passes) {
    auto &rg = g->rg;
    const bool d3 = g->dim == 3;
    region_fills(fills);
    fills.add(rg.d_out, 2LL * rg.n * flood_out_words(d3), 0, 4);
    fills.add(rg.d_marks, (long long)rg.mark_words(), 0, 4);
    if (int rc = g->ensure_pin()) return rc;
    g->ring[kQuitWord] = 0;
    launch_fill_multi(fills, st);
    FloodPass A = flood_pass(stop);
    Planes P = g->planes();
    if (tag) P.lab = g->tag;
    if (!by_passes && launch_flood_all(d3, tag, g->region_tiles(), P, flood_buf(), A, st)) {
      ++*passes;
      return JFC_OK;
    }
    return flood_passes(tag, A, passes, false);
  }

  // After a wait for the flood: one that gave up waiting is finished by passes
  // over its packed regions (true in *again), to be waited for once more.
  int finish_flood(bool tag, bool stop, int *passes, bool *again) {
    *again = *(const volatile int *)(g->ring + kQuitWord) != 0;
    if (!*again) return JFC_OK;
    by_passes = true;
    g->ring[kQuitWord] = 0;
    mark_all_regions();
    return flood_passes(tag, flood_pass(stop), passes, true);
  }

  FloodBuf flood_buf() const {
    auto &rg = g->rg;
    return FloodBuf{rg.buf.packed, rg.d_out, rg.d_open, rg.buf.planes};
  }

  FloodPass flood_pass(bool stop) const {
    FloodPass A{};
    A.w = settle_words();
    A.w.quit_host = g->d_ring + kQuitWord;
    A.c.visits = g->d_total + kFloodSlots;
    A.cert = g->d_flagword;
    A.stop = stop;
    A.def = g->inst.size() == 1 ? g->d_total + kDefSlots : g->d_def;
    A.object = g->lab;
    return A;
  }

  int flood_passes(bool tag, FloodPass A, int *passes, bool packed) {
    A.w.sums = nullptr;
    const Tiles T = g->region_tiles();
    const FloodBuf R = flood_buf();
    Planes P = g->planes();
    if (tag) P.lab = g->tag;
    return region_passes(kFloodSlots, passes, packed, [&](int kind, const PassCtl &c) {
      A.c = c;
      launch_flood(g->dim == 3, tag, T, P, R, A, kind, 2 * g->nwg, st);
    });
  }

  // Exact relabel (graphcut_init_global_relabel + graphcut_global_relabel,
  // graphcut_global_relabel.cl:19-124) on the graph's regions
  // (jfc_region.hip): every region once, then the marked ones until no mark
  // is left, then every region again to write the heights.  Where one launch
  // takes every pass, nothing waits for it here: should its waves have given
  // up waiting, the sweeps queued behind it do nothing and post stop word 5,
  // and finish_relabel() does it by passes.  resume: sweeping goes on after a
  // stop.
  int global_relabel(bool resume) {
    relabel_start = tm.mark();
    first_relabel = !resume;
    if (int rc = g->ensure_pin()) return rc;
    auto &rg = g->rg;
    rg.tag = 3 - rg.tag;
    {
      FillSet f;
      region_fills(f);
      f.add(g->d_flag, g->ntiles, 0, 1);  // kFinal sets the active tiles' flags
      f.add(rg.d_far, kFarSlots * kFarLine, 0, 4);
      f.add(rg.d_marks, (long long)rg.mark_words(), 0, 4);
      launch_fill_multi(f, st);
    }
    RegionPass A = relabel_pass();
    if (!by_passes && launch_relabel(g->dim == 3, g->region_tiles(), g->planes(), rg.buf, A, st)) {
      s.relabel_passes++;
      relabelled(A.w.quit, resume);
    } else {
      if (int rc = relabel_passes(A, false)) return rc;
      relabelled(nullptr, resume);
    }
    return JFC_OK;
  }

  // The relabel whose waves gave up waiting, by passes over its packed regions.
  int finish_relabel() {
    by_passes = true;
    mark_all_regions();
    if (int rc = relabel_passes(relabel_pass(), true)) return rc;
    gr_ev.pop_back();
    s.global_relabels--;
    relabelled(nullptr, true);
    return JFC_OK;
  }

  hipEvent_t relabel_start = nullptr;
  bool first_relabel = false;  // the last relabel came before the first sweep

  SettleWords settle_words() const {
    SettleWords w;
    w.sums = g->rg.d_marks;
    w.state = w.sums + kSettleLine * kSettleSlots;
    w.marks = w.state + kSettleLine * kSettleSlots;
    w.quit = w.state + 1;
    w.quit_host = nullptr;
    w.wait_ticks = g->rg.wait_ticks;
    return w;
  }

  RegionPass relabel_pass() const {
    auto &rg = g->rg;
    int tw, th, td;
    shape_dims(g->shape, &tw, &th, &td);
    RegionPass A{};
    A.tag = rg.tag;
    A.active = g->d_flag;
    A.pinst = g->d_inst;
    A.pone = g->inst[0];
    A.pdims = __builtin_ctz(tw) | __builtin_ctz(th) << 4 | __builtin_ctz(td) << 8;
    A.w = settle_words();
    A.c.visits = g->d_total + kRegionSlots;
    A.far = rg.d_far;
    return A;
  }

  int relabel_passes(RegionPass A, bool packed) {
    A.w.sums = nullptr;
    const Tiles T = g->region_tiles();
    const Planes P = g->planes();
    return region_passes(kRegionSlots, &s.relabel_passes, packed, [&](int kind, const PassCtl &c) {
      A.c = c;
      launch_region(g->dim == 3, T, P, g->rg.buf, A, kind, 2 * g->nwg, st);
    });
  }

  // after a relabel: every height is stored now, sweeping resumes
  void relabelled(const int *quit, bool resume) {
    launch_relabel_end(sweep_ctl(), g->d_hmat, g->ntiles, quit, resume, !first_relabel, st);
    gr_ev.push_back({relabel_start, tm.mark()});
    s.global_relabels++;
  }

  int cuts = 0;  // canonical-cut searches run

  hipEvent_t last_cut_end = nullptr;

  // Returns 1 in *found when an augmenting path still exists.  The search is
  // the solve's last step when it finds none, so the certificate word comes
  // back with every result of the solve, in one copy of the results block.
  // stop: a search that finds a path may end there, without labels.
  int canonical_cut(int *found, bool stop) {
    hipEvent_t a = tm.mark();
    ++cuts;
    FillSet f;
    f.add(g->d_flagword, 1, 0, 4);
    f.add(g->d_def, 2LL * (long long)g->inst.size(), 0, 4);
    f.add(g->d_total + kDefSlots, 2 * 64, 0, 4);
    if (int rc = flood(false, stop, f, &s.cut_passes)) return rc;
    for (bool again = true; again;) {
      last_cut_end = tm.mark();
      JFC_HIP(hipMemcpyAsync(g->pin_res, g->d_res, g->res_words * sizeof(long long),
                             hipMemcpyDeviceToHost, st));
      JFC_HIP(hipEventRecord(g->cnt_ev[0], st));
      JFC_HIP(hipEventSynchronize(g->cnt_ev[0]));
      if (int rc = finish_flood(false, stop, &s.cut_passes, &again)) return rc;
    }
    cut_ev.push_back({a, last_cut_end});
    *found = *((const int *)g->pin_res + ((const int *)g->d_flagword - (const int *)g->d_res));
    return JFC_OK;
  }

  // One push-relabel sweep: per colour class, compact the flagged tiles and
  // discharge them; then file the sweep's active-tile count.  Each kernel is
  // launched by itself: a sweep is 3 or 5 launches, issued while the sweeps
  // before it run, and a captured graph of them started later than the
  // launches did (a solve of 512x512: 321 us replayed, 280 us launched;
  // 4000x3000: 829 against 780; 15000x10000: 3861 against 3850).
  void issue_sweep() {
    const Tiles T = g->tiles();
    const Planes P = g->planes();
    for (int c = 0; c < g->ncolors; ++c) {
      Queue q = queue_from_list();
      const int n = g->color_off[c + 1] - g->color_off[c];
      if (n <= kSmallTiles) {
        // a colour class of a small graph: the push workgroups pick their
        // flagged tiles from the class's list themselves (one per workgroup)
        q = Queue{g->d_color_tiles + g->color_off[c], g->d_ctr, g->slot, n};
        q.pick = g->d_flag;
        q.mat = g->d_mat;
        q.touched = g->d_touched;
        q.hmat = g->d_hmat;
        q.cnt = g->d_sweep_state;
        q.total = g->d_total;
        q.stop = g->d_sweep_state + 2;
      } else {
        launch_compact(g->d_color_tiles + g->color_off[c], n, g->d_flag, g->d_mat,
                       g->d_touched, q, g->d_sweep_state, g->d_total, g->d_sweep_state + 2, st,
                       g->d_hmat);
      }
      hipEvent_t a = o.profile ? tm.mark() : nullptr;
      launch_push(g->shape, g->Kg, std::min(g->nwg, std::max(1, n)), T, P, q, g->d_flag, g->d_mat,
                  g->d_touched, g->d_hmat, o.max_local_iters, o.sparse_local_iters,
                  g->d_sweep_state, g->d_total + kIterSlots, st);
      if (o.profile) push_ev.push_back({a, tm.mark()});
      advance();
    }
    launch_sweep_end(sweep_ctl(), st);
  }

  // Waits for the stop word of sweep `seq` of the solve, which its end kernel
  // writes through to the ring.  An event per sweep to wait for put 5.5 us
  // between the sweeps (600x450 widget, a sweep of 22-40 us); the word itself
  // costs nothing there.  The stream is looked at once a millisecond, for an
  // error or an end without the word.
  int await_stop(int seq, int *stopw) {
    const volatile int *at = g->ring + seq % kStopRing;
    auto here = [&]() {
      const int w = *at;
      *stopw = w & 7;
      return (w >> 3) == seq;
    };
    auto looked = std::chrono::steady_clock::now();
    const auto begin = looked;
    for (;;) {
      for (int spin = 0; spin < 64; ++spin) {
        if (here()) return JFC_OK;
        __builtin_ia32_pause();
      }
      const auto now = std::chrono::steady_clock::now();
      if (now - begin > std::chrono::microseconds(100)) std::this_thread::yield();
      if (now - looked < std::chrono::milliseconds(1)) continue;
      looked = now;
      const hipError_t e = hipStreamQuery(st);
      if (e == hipErrorNotReady) {
        // no error for the caller to find; one that was there stays
        if (hipPeekAtLastError() == hipErrorNotReady) (void)hipGetLastError();
        continue;
      }
      JFC_HIP(e);
      // every kernel has completed, so the word is in the ring; re-read a few
      // times before giving up on it
      for (int spin = 0; spin < (1 << 20); ++spin)
        if (here()) return JFC_OK;
      return fail(JFC_ERR_DEVICE, "sweep " + std::to_string(seq) +
                                      ": its stop word did not reach the host");
    }
  }

  // One Fast-Cut sweep (QGCWidget::relabelPushFast, QGCW:2156-2205): every
  // active tile in one list, Jacobi relabel, line pushes, active flags.
  void issue_fast_sweep() {
    Queue q = queue_from_list();
    launch_compact(g->d_color_tiles, g->ntiles, g->d_flag, nullptr, nullptr, q,
                   g->d_sweep_state, g->d_total, g->d_sweep_state + 2, st);
    hipEvent_t a = o.profile ? tm.mark() : nullptr;
    launch_fc_sweep(g->shape, std::min(g->nwg, g->ntiles), g->tiles(), g->planes(), q,
                    g->d_flag, st);
    if (o.profile) push_ev.push_back({a, tm.mark()});
    advance();
    launch_sweep_end(sweep_ctl(), st);
  }

  int run() {
    const Tiles T = g->tiles();
    const Planes P = g->planes();
    const int nI = (int)g->inst.size();
    // reset the residual state from the inputs
    if (g->sweep_cap < o.max_sweeps + 1) {
      dfree(g->d_sweep);
      int rc = dalloc(&g->d_sweep, (size_t)o.max_sweeps + 1, "sweep counters");
      if (rc) return rc;
      g->sweep_cap = o.max_sweeps + 1;
    }
    hipEvent_t t0 = tm.mark();
    // counters and per-tile states in one launch (the sweep history needs no
    // clearing: each sweep files its entry before any read of it); no
    // heights stored yet, so the push kernel reads them as 0 (the Fast-Cut
    // kernels read every height, and the fold writes the zeros for them)
    {
      FillSet f;
      f.add(g->d_ctr, 2 * QSLOT, 0, 4);
      f.add(g->d_red, 2LL * nI * RED_SLOTS, 0, 4);
      f.add(g->d_total, 2 * kTotals, 0, 4);
      f.add(g->d_sweep_state, kSweepState, 0, 4);
      f.add(g->d_mat, g->ntiles, 0, 1);
      f.add(g->d_hmat, g->ntiles, 0, 1);
      f.add(g->d_touched, g->ntiles, 0, 1);
      // the fold's tile flags
      if (!o.initial_relabel) f.add(g->d_flag, g->ntiles, 0, 1);
      launch_fill_multi(f, st);
    }
    g->slot = 0;
    // the residual-arc masks restart from the inputs' with every plane
    // marked fresh: k_push reads fresh planes from c0 and writes them to cap
    const long long K = g->Kg, nodes = g->Nuser;
    // one pass over the nodes folds the terminal arcs (read cs, ct, write e)
    // and starts the masks: built from the input planes after an input
    // change (read K planes, write rmask), else copied from mask0 (read
    // mask0, write rmask).  mask0 is written by the first solve that can
    // reuse it -- the second solve of the same inputs -- so a solve of new
    // inputs, the common case, skips that write (Fast-Cut reads mask0 at
    // once and always has it written).
    const bool fast = o.method == JFC_METHOD_FASTCUT;
    int masks;
    if (g->mask_dirty) {
      g->mask_dirty = false;
      s.inputs_fresh = 1;
      masks = fast ? 2 : 3;
      g->mask0_ok = fast;
    } else {
      masks = g->mask0_ok ? 1 : 2;
      g->mask0_ok = true;
    }
    s.solve_bytes += nodes * (12 + (masks == 2 ? 4 * K + 8 : masks == 3 ? 4 * K + 4 : 8));
    if (int rc0 = g->ensure_pin()) return rc0;
    launch_fold(g->shape, T, P, g->d_red, o.initial_relabel ? nullptr : g->d_flag, nullptr,
                o.method == JFC_METHOD_FASTCUT && !o.initial_relabel, g->mask0, masks, st, true);
    // Fast-Cut reads and writes the residual planes directly
    if (o.method == JFC_METHOD_FASTCUT) launch_fc_materialize(P, g->mask0, g->Kg, st);
    // the fold's sums are read with the results (no host wait here): an
    // instance without terminal capacity has no excess, so the solve passes
    // over it, and the error is reported at the end
    std::vector<long long> red((size_t)nI * RED_SLOTS);
    int rc;
    if (o.initial_relabel) {
      if ((rc = global_relabel(false))) return rc;
    }  // else the zero heights (a valid labelling) and the fold's flags
    // Sweeps go out up to `ahead` beyond the last one whose stop word the
    // host has read.  The device decides after every sweep whether to go on
    // (k_sweep_end: no active tile, relabel due, budget spent), and a sweep
    // queued after a stop compacts nothing, so the host's wait for a stop
    // word overlaps the sweeps queued behind it.
    const int ahead = std::min(std::max(1, o.check_every), kStopRing - 1);
    int cert_rounds = 0;
    bool done = false;
    // sweeps issued in this solve (no-ops included; the device numbers them
    // the same way), and the stop words the host has read or skipped
    int sent = 0, known = 0;
    // no word of an earlier solve matches a sequence number of this one
    for (int k = 0; k < kStopRing; ++k) g->ring[k] = -1;
    for (;;) {
      int stopw = 0;
      for (;;) {
        while (sent < known + ahead) {
          if (o.method == JFC_METHOD_FASTCUT) {
            issue_fast_sweep();
            s.push_launches += 2 + 2 * g->dim;
          } else {
            issue_sweep();
            s.push_launches += g->ncolors;
          }
          ++sent;
        }
        if ((rc = await_stop(known, &stopw))) return rc;
        ++known;
        if (stopw) break;
      }
      // the sweeps queued behind the stop are no-ops: skip their words
      known = sent;
      // the sweeps queued behind the stop were no-ops
      if (stopw == 3) break;  // sweep budget spent
      if (stopw == 2 && o.stall_certify > 0) {
        // a stalled active set is often excess cut off from every deficit:
        // the canonical-cut search proves that (and is the solve's last
        // step) at less cost than the relabel that would show it
        int found = 0;
        if ((rc = canonical_cut(&found, true))) return rc;
        if (!found) {
          done = true;
          break;
        }
      }
      if (stopw == 2 || stopw == 4) {
        if ((rc = global_relabel(true))) return rc;
        continue;
      }
      if (stopw == 5) {  // the last relabel is not done
        if ((rc = finish_relabel())) return rc;
        continue;
      }
      // no active tile: the canonical cut doubles as the certificate
      int found = 0;
      if ((rc = canonical_cut(&found, true))) return rc;
      if (!found) {
        done = true;
        break;
      }
      // an augmenting path survived: relabel exactly and continue
      s.certificate_failures++;
      if (++cert_rounds > 16) return fail(JFC_ERR_STATE, "certificate kept failing");
      if ((rc = global_relabel(true))) return rc;
    }
    if (!done) {
      // labels of the current preflow are still useful to callers
      int found = 0;
      if ((rc = canonical_cut(&found, false))) return rc;
    }
    // the last cut search ran on the final excess, left the remaining deficit
    // of every instance in d_def and copied the results block back (the
    // solve's device work ends there)
    hipEvent_t t1 = last_cut_end;
    const long long *pred = g->pin_res, *pdef = pred + red.size(), *totals = pdef + nI;
    s.sweeps = ((const int *)(totals + kTotals))[1];
    std::copy(pred, pred + red.size(), red.begin());
    std::vector<long long> def(pdef, pdef + nI);
    if (nI == 1) def[0] = std::accumulate(totals + kDefSlots, totals + kDefSlots + 64, 0LL);
    for (int i = 0; i < nI; ++i)
      if (red[i * RED_SLOTS + RED_DEF0] == 0 && red[i * RED_SLOTS + RED_SUP0] == 0 &&
          red[i * RED_SLOTS + RED_CONST] == 0)
        return fail(JFC_ERR_NO_SEEDS, "instance " + std::to_string(i) +
                                          " has no terminal capacity (no labels)");
    for (int i = 0; i < nI; ++i)
      g->flows[i] = red[i * RED_SLOTS + RED_CONST] + red[i * RED_SLOTS + RED_DEF0] - def[i];
    s.flow = g->flows[0];
    s.converged = done ? 1 : 0;
    s.push_tiles = totals[0];
    s.local_iters = 0;
    for (int k = 0; k < 64; ++k) s.local_iters += totals[kIterSlots + k];
    g->last_sweeps = s.sweeps;
    // region visits: every region in a relabel's first and last pass, the
    // marked ones between
    long long marked = 0;
    for (int k = 0; k < 64; ++k) marked += totals[kRegionSlots + k];
    s.relabel_tiles = marked + 2LL * g->rg.n * s.global_relabels;
    // cut floods: every region in the first and last pass, the marked between
    long long sent_to = 0;
    for (int k = 0; k < 64; ++k) sent_to += totals[kFloodSlots + k];
    s.cut_tiles = sent_to + 2LL * g->rg.n * cuts;
    s.push_bytes = totals[0] * 256LL * push_bytes_per_node(g->Kg);
    // relabels: the first pass reads e and the mask and writes the bit planes
    // and borders, the last reads the bit planes and writes h, a marked
    // region reads its bit planes and borders; cut searches: the first pass
    // reads e, the last writes the labels, a visited region reads its mask or
    // bit planes
    const long long rplanes = 512LL * g->rg.buf.planes;  // bytes per region
    const long long rborder = 4LL * region_border_words(g->dim == 3);
    s.solve_bytes += s.push_bytes +
                     (12LL * nodes + g->rg.n * (2 * rplanes + 2 * rborder)) * s.global_relabels +
                     marked * (rplanes + 2 * rborder) + 5LL * nodes * cuts +
                     sent_to * 512LL * (g->Kg + 2);
    s.ms_total = Timer::ms(t0, t1);
    for (auto &p : push_ev) s.ms_push += Timer::ms(p.first, p.second);
    for (auto &p : gr_ev) s.ms_relabel += Timer::ms(p.first, p.second);
    for (auto &p : cut_ev) s.ms_cut += Timer::ms(p.first, p.second);
    g->solved = true;
    return done ? JFC_OK : JFC_NOT_CONVERGED;
  }
};

}  // namespace

extern "C" int jfc_solve(jfc_graph *g, const jfc_options *opt, jfc_stats *stats) {
  if (!g) return fail(JFC_ERR_INVALID, "null graph");
  Solver S{};
  S.g = g;
  S.by_passes = g->rg.by_passes;
  if (opt) S.o = *opt;
  else jfc_default_options(&S.o);
  if (S.o.max_sweeps <= 0) S.o.max_sweeps = 1 << 20;
  if (S.o.max_sweeps > (1 << 24)) S.o.max_sweeps = 1 << 24;
  if (S.o.check_every <= 0) S.o.check_every = 1;
  // 0: the cap jfc_autotune chose for the graph's size class, else 2
  if (S.o.max_local_iters <= 0) S.o.max_local_iters = g->tuned_mli > 0 ? g->tuned_mli : 2;
  // 0: the tuned cap, else kSparseIters; negative: the dense cap
  if (S.o.sparse_local_iters == 0) S.o.sparse_local_iters = g->tuned_sp ? g->tuned_sp : kSparseIters;
  if (S.o.sparse_local_iters < 0) S.o.sparse_local_iters = S.o.max_local_iters;
  // -1: the choice jfc_autotune made for the size class, else none
  if (S.o.initial_relabel < 0) S.o.initial_relabel = g->tuned_ir > 0 ? 1 : 0;
  if (S.o.stall_certify < 0) S.o.stall_certify = g->tuned_sc > 0 ? 1 : 0;
  if (S.o.tile_order != 0 && S.o.tile_order != 1)
    return fail(JFC_ERR_INVALID, "tile_order must be 0 (distance transform) or 1 (jump flooding)");
  if (S.o.method != JFC_METHOD_JFCUT && S.o.method != JFC_METHOD_FASTCUT)
    return fail(JFC_ERR_INVALID, "unknown method");
  if (S.o.method == JFC_METHOD_FASTCUT)
    for (const InstDesc &I : g->inst)
      if (I.K == 8)
        return fail(JFC_ERR_INVALID, "Fast-Cut runs on 4- and 6-connected graphs only");
  const int sh = shape_from_option(
      S.o.tile_shape == JFC_TILE_DEFAULT && g->tuned ? g->tuned : S.o.tile_shape, g->dim);
  if (!sh) return fail(JFC_ERR_INVALID, "tile shape does not match the graph's dimensionality");
  int rc = g->set_shape(sh);
  if (rc) return rc;
  for (size_t i = 0; i < g->inst.size(); ++i)
    if (g->caps_failed[i])
      return fail(JFC_ERR_STATE, "instance " + std::to_string(i) +
                                     ": an input setter failed and zeroed its plane; set the "
                                     "capacities again before solving");
  std::memset(&S.s, 0, sizeof(S.s));
  // the options' stream, else the graph's stream (jfc_set_stream)
  S.st = S.o.stream ? (hipStream_t)S.o.stream : g->ustream;
  if (!S.st) {
    // the legacy default stream cannot be captured: solve on a stream of the
    // graph's own, ordered after the work already queued on the default one
    if (!g->priv_stream) {
      if (hipStreamCreateWithFlags(&g->priv_stream, hipStreamNonBlocking) != hipSuccess ||
          hipEventCreateWithFlags(&g->priv_event, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        return fail(JFC_ERR_DEVICE, "cannot create the solve stream");
      }
    }
    JFC_HIP(hipEventRecord(g->priv_event, nullptr));
    JFC_HIP(hipStreamWaitEvent(g->priv_stream, g->priv_event, 0));
    S.st = g->priv_stream;
  }
  S.tm.pool = &g->ev_pool;
  S.tm.st = S.st;
  g->solved = false;
  rc = S.run();
  if (stats) *stats = S.s;
  return rc;
}

// ---- outputs -----------------------------------------------------------------------------

extern "C" int jfc_get_flow(jfc_graph *g, int inst, int64_t *flow) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  if (!flow) return fail(JFC_ERR_INVALID, "null output");
  if (!g->solved) return fail(JFC_ERR_STATE, "graph not solved");
  *flow = g->flows[inst];
  return JFC_OK;
}

extern "C" int jfc_get_flows(jfc_graph *g, int64_t *flows) {
  if (!g || !flows) return fail(JFC_ERR_INVALID, "null argument");
  if (!g->solved) return fail(JFC_ERR_STATE, "graph not solved");
  for (size_t i = 0; i < g->flows.size(); ++i) flows[i] = g->flows[i];
  return JFC_OK;
}

extern "C" int jfc_get_labels(jfc_graph *g, int inst, uint8_t *labels, int on_device) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  if (!labels) return fail(JFC_ERR_INVALID, "null output");
  if (!g->solved) return fail(JFC_ERR_STATE, "graph not solved");
  if ((rc = get_rows(g, g->inst[inst], labels, g->lab + g->inst[inst].node_off, 1, on_device)))
    return rc;
  return sync_user(g);
}

extern "C" int jfc_get_tags(jfc_graph *g, int inst, const uint8_t *fg, uint8_t *tags,
                            int on_device) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  if (!fg || !tags) return fail(JFC_ERR_INVALID, "null foreground or output");
  if (!g->solved) return fail(JFC_ERR_STATE, "graph not solved");
  if (!g->tag && (rc = dalloc(&g->tag, (size_t)g->Ntot, "tag plane"))) return rc;
  const long long o = g->inst[inst].node_off;
  launch_fill_u8(g->tag, g->Ntot, 0, g->ustream);
  if ((rc = put_rows(g, g->inst[inst], g->tag + o, fg, 1, on_device))) return rc;
  Solver S{};
  S.g = g;
  S.by_passes = g->rg.by_passes;
  jfc_default_options(&S.o);
  S.st = g->ustream;
  S.tm.pool = &g->ev_pool;
  S.tm.st = g->ustream;
  int passes = 0;
  if ((rc = S.flood(true, false, FillSet{}, &passes))) return rc;
  for (bool again = true; again;) {
    if ((rc = get_rows(g, g->inst[inst], tags, g->tag + o, 1, on_device))) return rc;
    if ((rc = sync_user(g))) return rc;
    if ((rc = S.finish_flood(true, false, &passes, &again))) return rc;
  }
  return JFC_OK;
}

extern "C" int jfc_get_energy(jfc_graph *g, int inst, int64_t *energy) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  if (!energy) return fail(JFC_ERR_INVALID, "null output");
  if (!g->solved) return fail(JFC_ERR_STATE, "graph not solved");
  if ((rc = g->ensure_pin())) return rc;
  const int nI = (int)g->inst.size();
  launch_fill_i32((int *)g->d_energy, 2LL * nI, 0, g->ustream);
  launch_energy(g->shape, g->tiles(), g->planes(), g->d_energy, g->ustream);
  JFC_HIP(hipMemcpyAsync(g->pin, g->d_energy + inst, sizeof(long long),
                         hipMemcpyDeviceToHost, g->ustream));
  if ((rc = sync_user(g))) return rc;
  *energy = *g->pin;
  return JFC_OK;
}

extern "C" int jfc_get_terminal_caps(jfc_graph *g, int inst, int32_t *cap_source,
                                     int32_t *cap_sink, int on_device) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  const InstDesc &I = g->inst[inst];
  if (cap_source && (rc = get_rows(g, I, cap_source, g->cs + I.node_off, 4, on_device))) return rc;
  if (cap_sink && (rc = get_rows(g, I, cap_sink, g->ct + I.node_off, 4, on_device))) return rc;
  return sync_user(g);
}

extern "C" int jfc_get_neighbor_caps(jfc_graph *g, int inst, int arc, int32_t *cap,
                                     int on_device) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  if (!cap) return fail(JFC_ERR_INVALID, "null output");
  if (arc < 0 || arc >= g->inst[inst].K)
    return fail(JFC_ERR_INVALID, "arc index outside the instance's connectivity");
  if ((rc = get_rows(g, g->inst[inst], cap,
                     g->c0 + (long long)arc * g->Ntot + g->inst[inst].node_off, 4, on_device)))
    return rc;
  return sync_user(g);
}

extern "C" int jfc_debug_tiles(jfc_graph *g, int inst, int32_t *ntiles, int32_t *tile_dims,
                               int32_t *grid_dims, int32_t *tile_off) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  int tw, th, td;
  shape_dims(g->shape, &tw, &th, &td);
  if (ntiles) *ntiles = g->ntiles;
  if (tile_dims) { tile_dims[0] = tw; tile_dims[1] = th; tile_dims[2] = td; }
  const InstDesc &I = g->inst[inst];
  if (grid_dims) { grid_dims[0] = I.tx; grid_dims[1] = I.ty; grid_dims[2] = I.tz; }
  if (tile_off) *tile_off = I.tile_off;
  return JFC_OK;
}

extern "C" int jfc_debug_tile_order(jfc_graph *g, int method, const uint8_t *tile_seed,
                                    int32_t *tile_dist, int32_t *order, int32_t *max_dist) {
  if (!g || !tile_seed) return fail(JFC_ERR_INVALID, "null argument");
  if (method != 0 && method != 1) return fail(JFC_ERR_INVALID, "method must be 0 or 1");
  // tile lines along x, y, z per instance (separable distance transform)
  const int n1 = (int)g->inst.size() + 1;
  std::vector<int> lines(3 * n1, 0);
  for (size_t i = 0; i < g->inst.size(); ++i) {
    const InstDesc &I = g->inst[i];
    const int per[3] = {I.ty * I.tz, I.tx * I.tz, I.tx * I.ty};
    for (int a = 0; a < 3; ++a) lines[a * n1 + i + 1] = lines[a * n1 + i] + per[a];
  }
  // work space of the ordering: four words per tile, the bins and the lines
  const size_t nt = g->ntiles;
  int *w = nullptr;
  if (int rc = dalloc(&w, 4 * nt + g->nbins + lines.size(), "tile ordering")) return rc;
  int *jf0 = w, *jf1 = w + nt, *tdist = w + 2 * nt, *d_order = w + 3 * nt, *hist = w + 4 * nt,
      *d_lines = hist + g->nbins;
  auto run = [&]() -> int {
    JFC_HIP(hipMemcpy(g->d_seed, tile_seed, nt, hipMemcpyHostToDevice));
    JFC_HIP(hipMemcpy(d_lines, lines.data(), lines.size() * sizeof(int), hipMemcpyHostToDevice));
    const TileLines L{{d_lines, d_lines + n1, d_lines + 2 * n1},
                      {lines[n1 - 1], lines[2 * n1 - 1], lines[3 * n1 - 1]}};
    launch_tile_order(g->shape, g->tiles(), g->d_seed, jf0, jf1, tdist, hist, g->nbins, d_order,
                      g->max_tile_dim, g->d_flagword + 2, L, method, 0);
    JFC_HIP(hipDeviceSynchronize());
    if (tile_dist) JFC_HIP(hipMemcpy(tile_dist, tdist, nt * 4, hipMemcpyDeviceToHost));
    if (order) JFC_HIP(hipMemcpy(order, d_order, nt * 4, hipMemcpyDeviceToHost));
    if (max_dist) JFC_HIP(hipMemcpy(max_dist, g->d_flagword + 2, 4, hipMemcpyDeviceToHost));
    return JFC_OK;
  };
  const int rc = run();
  dfree(w);
  return rc;
}

extern "C" int jfc_debug_tile_flags(jfc_graph *g, int which, uint8_t *flags) {
  if (!g || !flags || which < 0 || which > 2) return fail(JFC_ERR_INVALID, "bad argument");
  const int nI = (int)g->inst.size();
  launch_fill_i32((int *)g->d_red, 2LL * nI * RED_SLOTS, 0, 0);
  launch_fold(g->shape, g->tiles(), g->planes(), g->d_red, which ? g->d_flag : nullptr,
              which == 0 ? g->d_seed : nullptr, false, nullptr, 0, 0);
  unsigned char *src = which == 0 ? g->d_seed : g->d_flag;
  JFC_HIP(hipDeviceSynchronize());
  JFC_HIP(hipMemcpy(flags, src, g->ntiles, hipMemcpyDeviceToHost));
  g->solved = false;
  return JFC_OK;
}

extern "C" int jfc_autotune(jfc_graph *g, const jfc_options *opt, int reps, int *chosen) {
  if (!g) return fail(JFC_ERR_INVALID, "null graph");
  if (reps < 1) reps = 1;
  jfc_options o;
  if (opt) o = *opt;
  else jfc_default_options(&o);
  const int cand2[3] = {JFC_TILE_32x8, JFC_TILE_64x4, JFC_TILE_16x16};
  const int cand3[2] = {JFC_TILE_8x8x4, JFC_TILE_32x4x2};
  const int *cand = g->dim == 3 ? cand3 : cand2;
  const int nc = g->dim == 3 ? 2 : 3;
  // the local-iteration cap is tuned too unless the caller fixed it: fronts
  // that cross tiles in few visits favour more iterations per visit
  // (the 512^3 volume: 21.6 -> 14.3 ms at 4), others favour 2 (the
  // 2560x1440x50 video volume)
  const int mli_fixed = o.max_local_iters > 0 ? o.max_local_iters : 0;
  const int mcand[3] = {2, 3, 4};
  const int nm = mli_fixed ? 1 : 3;
  // so is the relabel before the first sweep: it pays where zero heights
  // let flow slosh for sweeps (the 2560x1440x50 video volume: 12.2 -> 9.4
  // ms) and costs where the push sweeps settle most of the flow first (the
  // 15000x10000 8-connected cut: 4.8 -> 8.5 ms)
  const int ir_fixed = o.initial_relabel >= 0 ? o.initial_relabel : -1;
  const int ni = ir_fixed >= 0 ? 1 : 2;
  // and whether a stalled active set first tries the certificate (it pays
  // where the last relabel would only prove the remaining excess cut off):
  // it changes how many sweeps and relabels a shape needs, so it is tried
  // with every shape rather than after the shape is chosen.  Then, on the
  // best of those, the cap of sparse launches (large where flow must cross
  // whole tiles, small where visits of a few tiles would iterate without
  // effect).
  const int sc_fixed = o.stall_certify >= 0 ? o.stall_certify : -1;
  const int ns = sc_fixed >= 0 ? 1 : 2;
  const int sp_fixed = o.sparse_local_iters != 0 ? o.sparse_local_iters : 0;
  auto time_it = [&](const jfc_options &t, double *med) -> int {
    std::vector<double> ms;
    for (int r = 0; r <= reps; ++r) {
      jfc_stats st;
      const int rc = jfc_solve(g, &t, &st);
      if (rc < 0) return rc;
      if (r > 0) ms.push_back(st.ms_total);  // the first run warms the shape's tables
    }
    std::sort(ms.begin(), ms.end());
    *med = ms[ms.size() / 2];
    return JFC_OK;
  };
  jfc_options best_o = o;
  double best_ms = 0.0;
  bool have = false;
  auto consider = [&](const jfc_options &t) -> int {
    double med = 0.0;
    if (int rc = time_it(t, &med)) return rc;
    if (!have || med < best_ms) {
      best_o = t;
      best_ms = med;
      have = true;
    }
    return JFC_OK;
  };
  o.sparse_local_iters = sp_fixed ? sp_fixed : kSparseIters;
  for (int c = 0; c < nc; ++c)
    for (int m = 0; m < nm; ++m)
      for (int i = 0; i < ni; ++i)
        for (int k = 0; k < ns; ++k) {
          o.tile_shape = cand[c];
          o.max_local_iters = mli_fixed ? mli_fixed : mcand[m];
          o.initial_relabel = ir_fixed >= 0 ? ir_fixed : i;
          o.stall_certify = sc_fixed >= 0 ? sc_fixed : k;
          if (int rc = consider(o)) return rc;
        }
  if (!sp_fixed) {
    const int spc[3] = {-1, 8, 64};
    const jfc_options base = best_o;
    for (int v : spc) {
      jfc_options t = base;
      t.sparse_local_iters = v;
      if (int rc = consider(t)) return rc;
    }
  }
  g->tuned = best_o.tile_shape;
  g->tuned_mli = mli_fixed ? 0 : best_o.max_local_iters;
  g->tuned_ir = ir_fixed >= 0 ? -1 : best_o.initial_relabel;
  g->tuned_sc = sc_fixed >= 0 ? -1 : best_o.stall_certify;
  g->tuned_sp = sp_fixed ? 0 : best_o.sparse_local_iters;
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tune[g->size_class] = Tuned{g->tuned, g->tuned_mli, g->tuned_ir, g->tuned_sc, g->tuned_sp};
  }
  if (chosen) *chosen = g->tuned;
  return JFC_OK;
}

extern "C" int jfc_get_tuning(const jfc_graph *g, jfc_options *opt) {
  if (!g || !opt) return fail(JFC_ERR_INVALID, "null argument");
  opt->tile_shape = g->tuned ? g->tuned : (g->dim == 3 ? JFC_TILE_8x8x4 : JFC_TILE_32x8);
  opt->max_local_iters = g->tuned_mli > 0 ? g->tuned_mli : 2;
  opt->initial_relabel = g->tuned_ir > 0 ? 1 : 0;
  opt->stall_certify = g->tuned_sc > 0 ? 1 : 0;
  opt->sparse_local_iters = g->tuned_sp ? g->tuned_sp : kSparseIters;
  return JFC_OK;
}

extern "C" int jfc_get_tile_shape(const jfc_graph *g, int *shape) {
  if (!g || !shape) return fail(JFC_ERR_INVALID, "null argument");
  *shape = g->tuned ? g->tuned : (g->dim == 3 ? JFC_TILE_8x8x4 : JFC_TILE_32x8);
  return JFC_OK;
}

extern "C" int jfc_get_local_iters(const jfc_graph *g, int *max_local_iters) {
  if (!g || !max_local_iters) return fail(JFC_ERR_INVALID, "null argument");
  *max_local_iters = g->tuned_mli > 0 ? g->tuned_mli : 2;
  return JFC_OK;
}

extern "C" int jfc_get_initial_relabel(const jfc_graph *g, int *initial_relabel) {
  if (!g || !initial_relabel) return fail(JFC_ERR_INVALID, "null argument");
  *initial_relabel = g->tuned_ir > 0 ? 1 : 0;
  return JFC_OK;
}

extern "C" int jfc_graph_size(const jfc_graph *g, int64_t *nodes, int32_t *kmax) {
  if (!g) return fail(JFC_ERR_INVALID, "null graph");
  if (nodes) *nodes = g->Nuser;
  if (kmax) *kmax = g->Kg;
  return JFC_OK;
}

// Gradients into device outputs directly, or into host outputs through the
// staging buffer (n floats per terminal output, K*n for the neighbour planes).
extern "C" int jfc_backward_all(jfc_graph *g, float *d_cap_source, float *d_cap_sink,
                                float *d_neighbor, int on_device) {
  if (!g) return fail(JFC_ERR_INVALID, "null graph");
  if (!g->solved) return fail(JFC_ERR_STATE, "graph not solved");
  const long long n = g->Nuser;
  hipStream_t st = g->ustream;
  if (on_device) {
    launch_backward_all(g->shape, g->tiles(), g->planes(), g->max_nx(), d_cap_source, d_cap_sink,
                        d_neighbor, n, st);
    return sync_user(g);
  }
  int rc;
  void *tmp = nullptr;
  if ((rc = stage_for(g, (size_t)n * (2 + g->Kg) * sizeof(float), &tmp))) return rc;
  float *a = d_cap_source ? (float *)tmp : nullptr;
  float *b = d_cap_sink ? (float *)tmp + n : nullptr;
  float *c = d_neighbor ? (float *)tmp + 2 * n : nullptr;
  // planes beyond an instance's connectivity keep the caller's values
  if (c) JFC_HIP(hipMemcpyAsync(c, d_neighbor, n * g->Kg * 4, hipMemcpyHostToDevice, st));
  launch_backward_all(g->shape, g->tiles(), g->planes(), g->max_nx(), a, b, c, n, st);
  if (a) JFC_HIP(hipMemcpyAsync(d_cap_source, a, n * 4, hipMemcpyDeviceToHost, st));
  if (b) JFC_HIP(hipMemcpyAsync(d_cap_sink, b, n * 4, hipMemcpyDeviceToHost, st));
  if (c) JFC_HIP(hipMemcpyAsync(d_neighbor, c, n * g->Kg * 4, hipMemcpyDeviceToHost, st));
  return sync_user(g);
}

extern "C" int jfc_debug_relabel_wait(jfc_graph *g, int64_t ticks) {
  if (!g || ticks < 0) return fail(JFC_ERR_INVALID, "bad argument");
  g->rg.wait_ticks = ticks;
  return JFC_OK;
}

extern "C" int jfc_debug_search_passes(jfc_graph *g, int on) {
  if (!g) return fail(JFC_ERR_INVALID, "null graph");
  g->rg.by_passes = on != 0;
  return JFC_OK;
}

extern "C" int jfc_debug_sweep_counts(jfc_graph *g, int32_t *counts, int32_t n) {
  if (!g || !counts) return fail(JFC_ERR_INVALID, "null argument");
  const int m = std::min(n, g->last_sweeps);
  if (m > 0) JFC_HIP(hipMemcpy(counts, g->d_sweep, m * 4, hipMemcpyDeviceToHost));
  return g->last_sweeps;
}

extern "C" int jfc_backward(jfc_graph *g, int inst, float *d_cap_source, float *d_cap_sink,
                            float *d_neighbor, int on_device) {
  int rc;
  if ((rc = check_inst(g, inst))) return rc;
  if (!g->solved) return fail(JFC_ERR_STATE, "graph not solved");
  const InstDesc &I = g->inst[inst];
  const long long n = g->inst_nodes(inst);
  hipStream_t st = g->ustream;
  if (on_device) {
    launch_backward(g->shape, g->tiles(), g->planes(), I, g->first_row(inst), d_cap_source,
                    d_cap_sink, d_neighbor, st);
    return sync_user(g);
  }
  void *tmp = nullptr;
  if ((rc = stage_for(g, (size_t)n * (2 + I.K) * sizeof(float), &tmp))) return rc;
  float *a = d_cap_source ? (float *)tmp : nullptr;
  float *b = d_cap_sink ? (float *)tmp + n : nullptr;
  float *c = d_neighbor ? (float *)tmp + 2 * n : nullptr;
  launch_backward(g->shape, g->tiles(), g->planes(), I, g->first_row(inst), a, b, c, st);
  if (a) JFC_HIP(hipMemcpyAsync(d_cap_source, a, n * 4, hipMemcpyDeviceToHost, st));
  if (b) JFC_HIP(hipMemcpyAsync(d_cap_sink, b, n * 4, hipMemcpyDeviceToHost, st));
  if (c) JFC_HIP(hipMemcpyAsync(d_neighbor, c, n * I.K * 4, hipMemcpyDeviceToHost, st));
  return sync_user(g);
}
