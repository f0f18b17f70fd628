// jfc_internal.h -- structures shared by the host driver and the gfx950
// kernels of libjfcut.  Nothing here is part of the C-ABI (include/jfcut.h).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <string>
#include <vector>

namespace jfc {

// Height of a node proven unable to reach any deficit node.
constexpr int HINF = 0x3fffffff;
// Per-instance reduction slots (int64): folded constant, initial deficit,
// energy, initial supply.  (The final deficit has an array of its own.)
constexpr int RED_CONST = 0, RED_DEF0 = 1, RED_ENERGY = 3, RED_SUP0 = 4,
              RED_SLOTS = 5;

// One grid instance inside a graph.  All instances share the plane arrays;
// instance i owns nodes [node_off, node_off + nx*ny*nz) and tiles
// [tile_off, tile_off + tx*ty*tz).
// Node v of an instance lives at node_off + x + px * (y + ny * z): rows are
// padded to px, a multiple of 32 nodes, so every 32-node tile row is one
// 128-byte line.  Pad nodes have no arcs and no terminal capacity.  Arrays
// exchanged with callers use the unpadded numbering x + nx * (y + ny * z)
// (user_off: the instance's first node in the graph's concatenation).
struct InstDesc {
  int nx, ny, nz;
  int conn, K;
  int tx, ty, tz;
  int tile_off;
  int ntiles;
  long long node_off;
  int px;
  long long user_off;
};

// The data term's second stream of a graph (null members: not created).
struct GraphAux {
  hipStream_t st;
  hipEvent_t fork, join, ready;
  void *pin;  // pinned host words
};

struct Planes {
  int *e;            // excess (> 0) / deficit (< 0), folded terminal arcs
  int *h;            // height; HINF = cannot reach a deficit
  int *cap;          // K residual planes, plane d at cap + d * stride
  const int *c0;     // input neighbour planes (same layout)
  const int *cs;     // input source capacities
  const int *ct;     // input sink capacities
  unsigned char *lab;// canonical labels (1 = source side)
  long long stride;  // nodes per plane (all instances)
  unsigned *rmask;   // bit d: residual of arc d > 0; bit 8+d: plane d still
                     // equals c0 (cap not yet written in this solve)
};

struct Tiles {
  const InstDesc *inst;
  const int *tile_inst;  // instance of every tile
  int ntiles;
  const int *row_off;    // first grid row (y, z) of every instance, + total
  int ninst;
  int nrows;             // rows of nx nodes over all instances
  int row_step;          // rows a workgroup streams at once in the whole-graph
                         // passes (several short rows of a one-instance graph)
  InstDesc one;          // the descriptor of instance 0 (kernel argument: a
                         // one-instance visit reads it with scalar loads)
};

// Tile shapes (256 nodes each, one node per lane).
enum ShapeId {
  SH_32x8 = 1,
  SH_64x4 = 2,
  SH_16x16 = 3,
  SH_8x8x4 = 4,
  SH_32x4x2 = 5
};
bool shape_is_3d(int shape);
void shape_dims(int shape, int *tw, int *th, int *td);

// Persistent work queues.  Slot s of ctr (QSLOT ints) holds the list count at
// [QSLOT*s] and claim head h at [QSLOT*s + QWORD*(1+h)], h < 8; every consumer
// zeroes the other slot's words, so producer/consumer launches alternate slots
// without any memset.  The words sit 256 bytes apart: device atomics on one
// cache line serialize, and with the eight heads in one line the claims of a
// launch queued behind each other (the 15000x10000 8-connected cut 5.64 ->
// 5.22 ms, the 2560x1440x50 video volume 16.9 -> 14.1 ms once they were
// split).
constexpr int QWORD = 64;
constexpr int QSLOT = 9 * QWORD;
struct Queue {
  int *list;
  int *ctr;
  int slot;
  int fixed_count;  // >= 0: consume list[0..fixed_count) instead of ctr count
  // Direct list (pick set): list[0..fixed_count) holds every tile of the
  // launch unfiltered, and the consumer does the compaction's work itself --
  // a tile is visited only if pick[t] is set (and pick[t] is cleared), its
  // entry bits come from mat / touched / hmat, and each visit adds 1 to
  // *cnt and *total; nothing is visited once *stop is nonzero.  For lists
  // no longer than the launch's grid, it saves the compaction launch.
  unsigned char *pick = nullptr;
  const unsigned char *mat = nullptr, *touched = nullptr, *hmat = nullptr;
  int *cnt = nullptr;
  long long *total = nullptr;
  const int *stop = nullptr;
};

// Sets the thread-local message returned by jfc_last_error().
void set_last_error(const std::string &msg);

// ---- launchers (all asynchronous on `st`) --------------------------------
void launch_fill_i32(int *p, long long n, int v, hipStream_t st);
void launch_fill_u8(unsigned char *p, long long n, unsigned char v, hipStream_t st);
// Fills in one launch, up to kMax of them, else in several (bytes = 1 or 4 per
// element).
struct FillSeg {
  void *p;
  long long n;
  int v;
  int bytes;
};
struct FillSet {
  static constexpr int kMax = 8;
  std::vector<FillSeg> seg;
  void add(void *p, long long count, int v, int bytes) {
    if (count > 0) seg.push_back(FillSeg{p, count, v, bytes});
  }
};
void launch_fill_multi(const FillSet &f, hipStream_t st);

// active, defi (either may be null): tiles holding an excess / a deficit node.
// Both zeroed here.
// zero_h: also write h = 0 over all nodes (the Fast-Cut kernels read every
// height; the push kernel instead treats the heights of tiles it has not
// visited in the solve as 0, see launch_push).
// masks: 0 = rmask untouched; 1 = rmask = mask0; 2 = build mask0 from the
// input planes and write it to rmask too (all in the same pass).
// cleared: the caller has zeroed active and defi already.
void launch_fold(int shape, const Tiles &T, const Planes &P, long long *red,
                 unsigned char *active, unsigned char *defi, bool zero_h, unsigned *mask0,
                 int masks, hipStream_t st, bool cleared = false);
// Capacities in the caller's numbering (rows of nx) onto stored planes (rows of
// px): src[1] may be null; excess: src[0] holds signed values, dst both
// terminals.  dir: the arcs' direction (-1: none leaves the grid).  bad: two
// host words, 1 where src[k] has a value outside [lo, hi].
struct PutPlanes {
  const int *src[2];
  int *dst[2];
};
void launch_put(const InstDesc &I, const PutPlanes &p, bool excess, int dir, int lo, int hi,
                int *bad, hipStream_t st);
// fg / bg: rows of nx bytes (the caller's numbering); cs / ct: rows of px.
void launch_seeds(int *cs, int *ct, const unsigned char *fg, const unsigned char *bg, int nx,
                  int px, long long rows, hipStream_t st);

// Jump-flooding tile distance + counting sort of tiles by distance.
// Lines of the tile grids along each axis: prefix[a][i] = lines along axis a
// in the instances before i, total[a] = all of them.
struct TileLines {
  const int *prefix[3];
  int total[3];
};
void launch_tile_order(int shape, const Tiles &T, const unsigned char *seed,
                       int *jf0, int *jf1, int *tdist, int *hist, int nbins,
                       int *order, int max_tile_dim, int *max_dist,
                       const TileLines &lines, int jump_flooding, hipStream_t st);

// Sweep bookkeeping on the device.  state (kSweepState ints): [0] active tiles of the
// running sweep, [1] sweep index, [2] stop word (0 sweep on, 1 no active
// tile, 2 active set stalled, 3 sweep budget spent, 4 relabel budget
// spent, 5 the last relabel is unfinished), [3] sweep index of the last
// relabel, [4..5] tile visits (int64) at the last relabel, [6] sweeps ended
// (no-ops included) in the solve, [8..9] the sweeps' cost (int64, ns) since the
// last relabel, [10..11] that relabel's.
struct SweepCtl {
  int *hist;             // active tiles per sweep
  int *state;
  const long long *total;  // tile visits of the push kernel so far
  int cap;               // entries of hist
  int max_sweeps;
  double stall_ratio;
  long long budget;      // tile visits between relabels (0 = no budget)
  // Pinned host ring the end of sweep s posts s * 8 + stop into, at slot
  // s % ring_n (null: no posting).
  int *ring;
  int ring_n;
  long long sweep_ns;    // cost of a sweep's launches
  long long visit_ns;    // and of each of its tile visits
  long long relabel_ns;  // cost of a relabel of no depth
  long long level_ns;    // and of each level of its longest distance
  const int *far;        // largest distances of the last relabel: kFarSlots, kFarLine apart
};
constexpr int kFarSlots = 64, kFarLine = 16;
constexpr int kSweepState = 12;
void launch_sweep_end(const SweepCtl &c, hipStream_t st);
void launch_relabel_end(const SweepCtl &c, unsigned char *hmat, int n, const int *quit, bool resume,
                        bool charge, hipStream_t st);

// Queue list entries: tile index, plus, when compacted with `mat`, kEntryMat
// if mat[t] is set, else kEntryClean if touched[t] is clear (no visit and no
// flush has written the tile's planes or mask words in this solve); when
// compacted with `hmat`, kEntryHeights if hmat[t] is set (the tile's heights
// are stored in this solve).
constexpr int kEntryMat = 1 << 30;
constexpr int kEntryClean = 1 << 29;
constexpr int kEntryHeights = 1 << 28;
constexpr int kEntryTile = kEntryHeights - 1;
// stop (or null): a nonzero word makes the compaction a no-op.
void launch_compact(const int *src, int n, unsigned char *flag,
                    const unsigned char *mat, const unsigned char *touched, const Queue &q,
                    int *sweep_cnt, long long *total, const int *stop, hipStream_t st,
                    const unsigned char *hmat = nullptr);
// mat: per tile, 1 once every residual plane of the tile was written in
// this solve (cleared when a solve starts).  hmat: per tile, 1 once its heights are stored in
// this solve (by a push visit, which then writes all of them, or by a global
// relabel); heights of a tile with hmat 0 read as 0, the labelling a solve
// starts from.  max_iters caps the local iterations of a visit, sparse_iters
// those of a launch whose list fits its grid, max_iters << sweep until then.
// iter_total: 64 int64 counters of local iterations (or null).
// touched: per tile, 1 once a flush wrote into the tile's planes or mask
// words (cleared when a solve starts).
// sweep_state: the solve's SweepCtl state ([1] = sweep index).
void launch_push(int shape, int kmax, int nwg, const Tiles &T, const Planes &P,
                 const Queue &q, unsigned char *flag, unsigned char *mat,
                 unsigned char *touched, unsigned char *hmat,
                 int max_iters, int sparse_iters, const int *sweep_state,
                 long long *iter_total, hipStream_t st);
// Fast-Cut comparator (jfc_fastcut.hip)
void launch_fc_materialize(const Planes &P, const unsigned *mask0, int K, hipStream_t st);
void launch_fc_sweep(int shape, int nwg, const Tiles &T, const Planes &P, const Queue &q,
                     unsigned char *flag, hipStream_t st);
// Global relabel on bit-parallel regions (jfc_region.hip): regions of 64 x 64
// nodes in 2D, 64 x 8 x 8 in 3D.  T is the region tiling (descriptors with
// the regions' counts and offsets).
struct RegionBuf {
  unsigned long long *packed;  // bit planes: (region * planes + plane) * 64 + row
  int *border;                 // region_border_words() distances per region, zero at first
  int *base;                   // per region: distance its counting planes start at
  int planes;                  // directions stored + region_state_planes()
};
enum RegionPassKind { kPack = 0, kBorders = 1, kFinal = 2 };
// What every pass over the regions (relabel, cut or tag) shares.
struct PassCtl {
  unsigned char *dirty_in, *dirty_out;  // marks this pass takes / sets for the next
  int *any_in, *any_out, *any_clear;  // whether a mark is set; the slot after next is cleared
  int *post;                          // pinned word: seq * 2 + (any mark was set for this pass)
  int seq;
  long long *visits;                  // 64 counters of kBorders visits
};
// A search in one launch (settle): the words its waves share, zeroed by the
// caller, kSettleLine ints apart.
constexpr int kSettleSlots = 64, kSettleLine = 32;
struct SettleWords {
  int *sums = nullptr;   // kSettleSlots times: marks served, marks made, workgroups begun
  int *state;            // kSettleSlots
  int *marks;            // per region: marks made so far
  int *quit;             // set when it gave up waiting
  int *quit_host;        // (or null) pinned word set then, too
  long long wait_ticks;  // time without progress before it gives up (100 MHz clock)
};
struct RegionPass {
  PassCtl c;
  int tag;                            // of this relabel, 1 or 2, alternating
  unsigned char *active;              // push tiles' active flags, cleared by the caller
  const InstDesc *pinst;              // push tiling
  InstDesc pone;                      // its instance 0
  int pdims;                          // push tile dimensions, log2 (x | y << 4 | z << 8)
  int *far;                           // kFarSlots, zeroed by the caller: largest distances
  SettleWords w;                      // launch_relabel (else w.sums null)
};
// Cut and tag floods on the same regions (jfc_flood.hip).
struct FloodBuf {
  unsigned long long *packed;  // the relabel's planes, free between relabels
  unsigned long long *out;     // flood_out_words() per region: labels sent to the
                               // neighbours; zeroed by the caller
  unsigned char *open;         // per region: its direction planes are packed
  int planes;
};
struct FloodPass {
  PassCtl c;
  SettleWords w;         // launch_flood_all (else w.sums null)
  int *cert;             // cut: set when a labelled node has a deficit
  bool stop;             // cut: end the search once *cert is set
  long long *def;        // cut: remaining deficit, per instance, or (one
                         // instance) 64 partial sums; zeroed by the caller
  const unsigned char *object;  // tag: the labels the flood stays in; P.lab then holds the
                                // foreground seeds on entry, the tags at the end
};
int flood_out_words(bool d3);
// The whole flood; *A.w.quit becomes 1 if it gave up waiting (every region is
// packed, no label written).  false: the graph has too many regions for it.
bool launch_flood_all(bool d3, bool tag, const Tiles &T, const Planes &P, const FloodBuf &R,
                      const FloodPass &A, hipStream_t st);
void launch_flood(bool d3, bool tag, const Tiles &T, const Planes &P, const FloodBuf &R,
                  const FloodPass &A, int pass, int nwg, hipStream_t st);
// The whole relabel; *A.w.quit becomes 1 if it gave up waiting (every region is
// packed, no height written).  false: the graph has too many regions for it.
bool launch_relabel(bool d3, const Tiles &T, const Planes &P, const RegionBuf &R,
                    const RegionPass &A, hipStream_t st);
int region_border_words(bool d3);
int region_state_planes();
void region_dims(bool d3, int *tw, int *th, int *td);
void launch_region(bool d3, const Tiles &T, const Planes &P, const RegionBuf &R,
                   const RegionPass &A, int pass, int nwg, hipStream_t st);
// energy: one int64 per instance, zeroed by the caller.
void launch_energy(int shape, const Tiles &T, const Planes &P, long long *energy,
                   hipStream_t st);
// row0: the instance's first row.  max_nx: the longest row of the graph.
void launch_backward(int shape, const Tiles &T, const Planes &P, const InstDesc &I, int row0,
                     float *dcs, float *dct, float *dnb, hipStream_t st);
void launch_backward_all(int shape, const Tiles &T, const Planes &P, int max_nx, float *dcs,
                         float *dct, float *dnb, long long user_total, hipStream_t st);

}  // namespace jfc
