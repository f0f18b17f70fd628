// jfc_solver.hip -- gfx950 kernels of the grid max-flow solve.
//
// Reference counterparts (paths relative to src/QVisualizer/):
//   k_push     graphcut_relabel_push   cl/GraphCut/graphcut_push_relabel.cl:25-203 (2D), :215-439 (3D)
//   k_compact  graphcut_count_node + clogs scan + graphcut_scatter_node
//                               cl/GraphCut/graphcut_count_block.cl:19-65
//
// Layout: every graph stores int32 planes (e, h, K residual planes) in
// structure-of-arrays order over all instances.  Kernels work on tiles of
// 256 nodes (one node per lane) staged in LDS with a one-node halo.  Tiles of
// one colour class never share a node; a halo node shared by two of them is
// reached through different arcs, so within a push-relabel launch every
// residual plane entry has one writer and only excess and mask words need
// atomics.
#include "jfc_rows.h"

#include <algorithm>
#include <atomic>
#include <climits>

namespace jfc {

bool shape_is_3d(int s) { return s == SH_8x8x4 || s == SH_32x4x2; }

void shape_dims(int s, int *tw, int *th, int *td) {
  int a = 0, b = 0, c = 0;
  JFC_DISPATCH(s, { a = S::TW; b = S::TH; c = S::TD; });
  *tw = a; *th = b; *td = c;
}

// ---- small utilities --------------------------------------------------------

__global__ void k_fill_i32(int *p, long long n, int v) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ void k_fill_u8(unsigned char *p, long long n, unsigned char v) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}

static int grid_for(long long n, int per_block = 256, int cap = 8192) {
  long long g = (n + per_block - 1) / per_block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (int)g;
}

void launch_fill_i32(int *p, long long n, int v, hipStream_t st) {
  if (n > 0) k_fill_i32<<<grid_for(n), 256, 0, st>>>(p, n, v);
}
void launch_fill_u8(unsigned char *p, long long n, unsigned char v, hipStream_t st) {
  if (n > 0) k_fill_u8<<<grid_for(n), 256, 0, st>>>(p, n, v);
}

// Several fills in one launch: blockIdx.y picks the segment.
struct FillArgs {
  FillSeg seg[FillSet::kMax];
};

__global__ void k_fill_multi(FillArgs f) {
  const FillSeg s = f.seg[blockIdx.y];
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < s.n;
       i += (long long)gridDim.x * blockDim.x) {
    if (s.bytes == 1) static_cast<unsigned char *>(s.p)[i] = (unsigned char)s.v;
    else static_cast<int *>(s.p)[i] = s.v;
  }
}

void launch_fill_multi(const FillSet &f, hipStream_t st) {
  for (size_t k0 = 0; k0 < f.seg.size(); k0 += FillSet::kMax) {
    const int n = (int)std::min<size_t>(FillSet::kMax, f.seg.size() - k0);
    FillArgs a{};
    long long most = 1;
    for (int k = 0; k < n; ++k) {
      a.seg[k] = f.seg[k0 + k];
      most = std::max(most, a.seg[k].n);
    }
    k_fill_multi<<<dim3(grid_for(most, 256, 1024), n), 256, 0, st>>>(a);
  }
}

// Hard seeds from the caller's unpadded seed bytes (row r of nx bytes) onto
// the stored planes (row r at r * px): fg wins where both are set, the rule
// of graphcut_compute_excessflow.cl:71-74.
__global__ void k_seeds(int *cs, int *ct, const unsigned char *fg, const unsigned char *bg,
                        int nx, int px, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const long long v = (i / nx) * px + i % nx;
    if (fg && fg[i]) { cs[v] = 1 << 30; ct[v] = 0; }
    else if (bg && bg[i]) { cs[v] = 0; ct[v] = 1 << 30; }
  }
}

void launch_seeds(int *cs, int *ct, const unsigned char *fg, const unsigned char *bg, int nx,
                  int px, long long rows, hipStream_t st) {
  const long long n = rows * nx;
  if (n > 0 && (fg || bg)) k_seeds<<<grid_for(n), 256, 0, st>>>(cs, ct, fg, bg, nx, px, n);
}

// A caller's capacities onto the stored planes in one pass: rows of nx read,
// rows of px written, every value checked against [lo, hi] (a plane with one
// outside is named in `bad`, pinned words of the host), and the arcs of
// direction (dx, dy, dz) that leave the grid stored as 0.  EXCESS: one source
// plane of signed values, split into its source and sink capacities.  Bound by
// one read and one write of the plane, and on small ones by its launch and
// the host's wait.  An arc plane from device memory, call to return: 15 us at
// 1023x767 and 220 us at 15000x10000 (5.4 TB/s); a copy, a check and a border
// pass with two waits took 39 and 645.
template <bool EXCESS>
__global__ __launch_bounds__(256) void k_put(PutPlanes p, int nx, int px, int ny, int nz, int lo,
                                             int hi, int dx, int dy, int dz, int *bad) {
  const int x0 = blockIdx.x * 256 + (threadIdx.x & 63);
  const int rows = ny * nz;
  int out = 0;
  for (int row = blockIdx.y * 4 + (threadIdx.x >> 6); row < rows; row += gridDim.y * 4) {
    const int y = row % ny + dy, z = row / ny + dz;
    const bool in = y >= 0 && y < ny && z >= 0 && z < nz;
    const long long s = (long long)row * nx, d = (long long)row * px;
    int v[2][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int x = x0 + 64 * u;
      v[0][u] = x < nx ? p.src[0][s + x] : 0;
      v[1][u] = !EXCESS && p.src[1] && x < nx ? p.src[1][s + x] : 0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int x = x0 + 64 * u;
      if (x >= nx) continue;
      out |= (v[0][u] < lo || v[0][u] > hi) | (v[1][u] < lo || v[1][u] > hi) << 1;
      if (EXCESS) {
        p.dst[0][d + x] = max(v[0][u], 0);
        p.dst[1][d + x] = max(-v[0][u], 0);
      } else {
        p.dst[0][d + x] = in && x + dx >= 0 && x + dx < nx ? v[0][u] : 0;
        if (p.src[1]) p.dst[1][d + x] = v[1][u];
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 2; ++k)
    if (__ballot((out >> k) & 1) && lane_id() == 0)
      __hip_atomic_store(bad + k, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

void launch_put(const InstDesc &I, const PutPlanes &p, bool excess, int dir, int lo, int hi,
                int *bad, hipStream_t st) {
  int dx = 0, dy = 0, dz = 0;
  if (dir >= 0) {
    if (I.K == 6) dir_of<true>(dir, dx, dy, dz);
    else dir_of<false>(dir, dx, dy, dz);
  }
  const long long rows = (long long)I.ny * I.nz;
  const dim3 grid((I.nx + 255) / 256, (unsigned)std::min<long long>((rows + 3) / 4, 16384));
  if (excess) k_put<true><<<grid, 256, 0, st>>>(p, I.nx, I.px, I.ny, I.nz, lo, hi, dx, dy, dz, bad);
  else k_put<false><<<grid, 256, 0, st>>>(p, I.nx, I.px, I.ny, I.nz, lo, hi, dx, dy, dz, bad);
}

// ---- block reductions --------------------------------------------------------

__device__ __forceinline__ long long block_sum_ll(long long v, long long *buf) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if (lane_id() == 0) buf[w] = v;
  __syncthreads();
  long long r = 0;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) r += buf[i];
  return r;
}

// Tile-parallel kernels: workgroup b walks a contiguous chunk of tiles so that
// per-instance sums are flushed once per instance change.
struct Chunk {
  int t0, t1;
  __device__ __forceinline__ Chunk(int ntiles) {
    const int per = (ntiles + gridDim.x - 1) / gridDim.x;
    t0 = blockIdx.x * per;
    t1 = min(ntiles, t0 + per);
  }
};

static int tile_grid(int ntiles) { return ntiles < 4096 ? (ntiles > 0 ? ntiles : 1) : 4096; }

// Any lane of the 256-lane workgroup with pred set: one ballot per wave, one
// LDS word per wave, one barrier.  The buffer half alternates with `parity`,
// so a second barrier is not needed before reuse.
// The barrier also orders the workgroup's LDS accesses like __syncthreads.
__device__ __forceinline__ int block_any(int pred, int *s_w, int &parity) {
  const int w = __ballot(pred) != 0;
  int *buf = s_w + 4 * parity;
  parity ^= 1;
  if (lane_id() == 0) buf[threadIdx.x >> 6] = w;
  __syncthreads();
  return buf[0] | buf[1] | buf[2] | buf[3];
}

// ---- row-streaming passes ----------------------------------------------------
//
// The fold walks grid rows, not tiles (but for the new masks of 2D batches,
// k_fold_tiles): row r of the graph (the rows of all instances concatenated) is
// nx consecutive nodes, so a workgroup streams it with 16-byte loads and
// stores, several in flight per lane.  A lane handles a group of 4 consecutive
// nodes (rows start at multiples of 32 nodes).  A workgroup step takes one row,
// or several short rows of a one-instance graph (RowStep), so that every lane
// has groups to stream.  Per-tile flags are derived from the column and the
// row's tile row; per-instance sums are flushed when a workgroup's step changes
// instance and at its end.

// Groups in flight per lane.
constexpr int RS_U = 4;

template <class S>
struct RowRef {
  int inst, nx;
  long long v0;  // first node of the row
  int tile0;     // tile of column 0
};

template <class S>
__device__ __forceinline__ RowRef<S> row_ref(const Tiles &T, int r) {
  int lo = 0, hi = T.ninst - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (T.row_off[mid] <= r) lo = mid;
    else hi = mid - 1;
  }
  const InstDesc &I = T.inst[lo];
  const int rr = r - T.row_off[lo];
  const int y = rr % I.ny, z = rr / I.ny;
  RowRef<S> R;
  R.inst = lo;
  R.nx = I.nx;
  R.v0 = I.node_off + (long long)rr * I.px;
  R.tile0 = I.tile_off + I.tx * (y / S::TH + I.ty * (z / S::TD));
  return R;
}

// Row r of a one-instance graph (no search over the instances).
template <class S>
__device__ __forceinline__ RowRef<S> row_ref_one(const Tiles &T, int r) {
  const InstDesc &I = T.inst[0];
  const int y = r % I.ny, z = r / I.ny;
  RowRef<S> R;
  R.inst = 0;
  R.nx = I.nx;
  R.v0 = I.node_off + (long long)r * I.px;
  R.tile0 = I.tile_off + I.tx * (y / S::TH + I.ty * (z / S::TD));
  return R;
}

// Group k of a row: first column x and node count n (0 past the end).
struct Group {
  int x, n;
};

// A workgroup step of a whole-graph pass: T.row_step rows from row r0 (one
// instance), seen as slots of 4-node groups, ng per row.  Slot k is group
// k % ng of row r0 + k / ng.  Rows start at multiples of 32 nodes, so a row's
// groups are 4-aligned.
template <class S>
struct RowStep {
  RowRef<S> R0;  // first row of the step
  int r0, ng, slots;
  __device__ __forceinline__ RowStep(const Tiles &T, int step) {
    r0 = step * T.row_step;
    R0 = row_ref<S>(T, r0);
    ng = (R0.nx + 3) / 4;
    slots = min(T.row_step, T.nrows - r0) * ng;
  }
  // The row and group of slot k (k < slots).
  __device__ __forceinline__ void at(const Tiles &T, int k, RowRef<S> &R, Group &g) const {
    const int dr = T.row_step > 1 ? k / ng : 0;
    const int gk = T.row_step > 1 ? k - dr * ng : k;
    R = dr ? row_ref_one<S>(T, r0 + dr) : R0;
    g.x = 4 * gk;
    g.n = min(4, R.nx - g.x);
  }
};

__device__ __forceinline__ int row_steps(const Tiles &T) {
  return (T.nrows + T.row_step - 1) / T.row_step;
}

// Load / store up to 4 consecutive ints (16-byte access when the group is
// full and aligned).
__device__ __forceinline__ int4 load4(const int *p, long long v, int n) {
  int4 r = make_int4(0, 0, 0, 0);
  if (n == 4 && (((size_t)(p + v)) & 15) == 0) return *(const int4 *)(p + v);
  if (n > 0) r.x = p[v];
  if (n > 1) r.y = p[v + 1];
  if (n > 2) r.z = p[v + 2];
  if (n > 3) r.w = p[v + 3];
  return r;
}

__device__ __forceinline__ void store4(int *p, long long v, int n, int4 a) {
  if (n == 4 && (((size_t)(p + v)) & 15) == 0) { *(int4 *)(p + v) = a; return; }
  if (n > 0) p[v] = a.x;
  if (n > 1) p[v + 1] = a.y;
  if (n > 2) p[v + 2] = a.z;
  if (n > 3) p[v + 3] = a.w;
}

__device__ __forceinline__ int comp(const int4 &a, int i) {
  return i == 0 ? a.x : i == 1 ? a.y : i == 2 ? a.z : a.w;
}

// Set flag[tile] = 1 for the tiles of the nodes of a group with a set bit.
template <class S>
__device__ __forceinline__ void flag_group(unsigned char *flag, int tile0, Group g,
                                           unsigned bits) {
  if (!bits) return;
  const int t0 = tile0 + g.x / S::TW, t1 = tile0 + (g.x + g.n - 1) / S::TW;
  if (t0 == t1) {
    flag[t0] = 1;
    return;
  }
  for (int i = 0; i < g.n; ++i)
    if ((bits >> i) & 1u) flag[tile0 + (g.x + i) / S::TW] = 1;
}

// Per-instance int64 sums of a workgroup: accumulated per lane, flushed with
// one atomic per workgroup and instance.
template <int NS>
struct InstSums {
  long long a[NS];
  int cur = -1;
  __device__ __forceinline__ void reset() {
#pragma unroll
    for (int k = 0; k < NS; ++k) a[k] = 0;
  }
  __device__ __forceinline__ void flush(long long *const *dst, const int *stride,
                                        long long *buf) {
    if (cur < 0) return;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const long long A = block_sum_ll(a[k], buf);
      if (threadIdx.x == 0 && A != 0)
        atomicAdd((unsigned long long *)&dst[k][(long long)cur * stride[k]], (unsigned long long)A);
    }
  }
  // Called with the (uniform) instance of the next row.
  __device__ __forceinline__ void enter(int inst, long long *const *dst, const int *stride,
                                        long long *buf) {
    if (inst == cur) return;
    flush(dst, stride, buf);
    cur = inst;
    reset();
  }
};

// Grid of a persistent (queue-consuming) launch: every workgroup must be
// resident from the start -- one dispatched late finds the queue drained but
// still runs its static first run after the others are done, stretching the
// launch -- so the grid is capped at what the device holds at once for this
// kernel (occupancy per CU, from its register and LDS use, times CUs).
// Compute units of the current device, queried once per device (every
// persistent launch sizes its grid with it).
int device_cus() {
  static std::atomic<int> cache[16];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = 0;
  if (dev >= 0 && dev < 16) {
    const int c = cache[dev].load(std::memory_order_relaxed);
    if (c > 0) return c;
  }
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus < 1)
    cus = 1;
  if (dev >= 0 && dev < 16) cache[dev].store(cus, std::memory_order_relaxed);
  return cus;
}

template <auto Kernel>
static int resident_grid(int want) {
  return resident_grid_b<Kernel, 256>(want);
}

// Grid of a pass over the rows (nsteps row steps): one workgroup per step at
// most, and no more than the device holds at once -- a second, partial round
// of workgroups would run with most of the device idle.
template <auto Kernel>
static int row_grid(int nsteps) {
  return resident_grid<Kernel>(std::max(1, nsteps));
}

// Fold terminal arcs: e = cs - ct; const += min(cs, ct);
// deficit0 += max(ct - cs, 0); supply0 += max(cs - ct, 0).
// With `active` set it flags the tiles holding excess (`active` zeroed by the
// launcher); with `zero_h` it starts the labelling at zero heights over all
// nodes (the reference clears h, QGCWidget.cpp:2400; the push kernel reads
// the heights of tiles it has not visited in the solve as 0 instead); with
// `defi` it flags the tiles holding a deficit node (the seed flags of
// graphcut_init_global_relabel, graphcut_global_relabel.cl:19-48).
//
// The same pass starts the residual-arc masks of the solve (MASKS): 0 leaves
// them alone, 1 copies mask0 to rmask, 2 builds mask0 from the input planes
// (residual bit d = c0[d] > 0, every plane fresh) and writes it to both, 3
// builds it into rmask only (mask0 is then built by the next solve of the
// same inputs, if there is one).  One pass instead of a fold, a mask build
// and a copy: the mask words are written once and the terminal planes read
// once.
template <class S, int MASKS>
__global__ __launch_bounds__(256) void k_fold(Tiles T, Planes P, long long *red,
                                              unsigned char *active, unsigned char *defi,
                                              int zero_h, unsigned *mask0) {
  // planes of eight directions in flight per group: one group per lane
  constexpr int U = MASKS >= 2 ? 1 : RS_U;
  __shared__ long long buf[4];
  long long *dst[3] = {red + RED_CONST, red + RED_DEF0, red + RED_SUP0};
  const int stride[3] = {RED_SLOTS, RED_SLOTS, RED_SLOTS};
  InstSums<3> sums;
  sums.reset();
  const int nsteps = row_steps(T);
  for (int step = blockIdx.x; step < nsteps; step += gridDim.x) {
    const RowStep<S> RS(T, step);
    sums.enter(RS.R0.inst, dst, stride, buf);
    const int K = MASKS >= 2 ? T.inst[RS.R0.inst].K : 0;
    for (int k0 = threadIdx.x; k0 < RS.slots; k0 += U * 256) {
      Group g[U];
      RowRef<S> R[U];
      int4 a[U], b[U], m[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * 256;
        if (k < RS.slots) RS.at(T, k, R[u], g[u]);
        else { R[u] = RS.R0; g[u] = Group{0, 0}; }
        a[u] = load4(P.cs, R[u].v0 + g[u].x, g[u].n);
        b[u] = load4(P.ct, R[u].v0 + g[u].x, g[u].n);
        if (MASKS == 1) m[u] = load4((const int *)mask0, R[u].v0 + g[u].x, g[u].n);
        if (MASKS >= 2) {
          int4 c[S::KMAX];
#pragma unroll
          for (int d = 0; d < S::KMAX; ++d)
            c[d] = d < K ? load4(P.c0 + d * P.stride, R[u].v0 + g[u].x, g[u].n) : make_int4(0, 0, 0, 0);
          m[u] = make_int4(0, 0, 0, 0);
#pragma unroll
          for (int d = 0; d < S::KMAX; ++d) {
            if (d >= K) break;
            const int fresh = 1 << (8 + d);
            m[u].x |= (c[d].x > 0 ? 1 << d : 0) | fresh; m[u].y |= (c[d].y > 0 ? 1 << d : 0) | fresh;
            m[u].z |= (c[d].z > 0 ? 1 << d : 0) | fresh; m[u].w |= (c[d].w > 0 ? 1 << d : 0) | fresh;
          }
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (g[u].n == 0) continue;
        const long long v = R[u].v0 + g[u].x;
        int4 e;
        e.x = a[u].x - b[u].x; e.y = a[u].y - b[u].y;
        e.z = a[u].z - b[u].z; e.w = a[u].w - b[u].w;
        store4(P.e, v, g[u].n, e);
        if (zero_h) store4(P.h, v, g[u].n, make_int4(0, 0, 0, 0));
        if (MASKS) store4((int *)P.rmask, v, g[u].n, m[u]);
        if (MASKS == 2) store4((int *)mask0, v, g[u].n, m[u]);
        unsigned bits = 0, dbits = 0;
        for (int i = 0; i < g[u].n; ++i) {
          const int s = comp(a[u], i), t = comp(b[u], i);
          sums.a[0] += min(s, t);
          sums.a[1] += max(t - s, 0);
          sums.a[2] += max(s - t, 0);
          bits |= (unsigned)(s > t) << i;
          dbits |= (unsigned)(s < t) << i;
        }
        if (active) flag_group<S>(active, R[u].tile0, g[u], bits);
        if (defi) flag_group<S>(defi, R[u].tile0, g[u], dbits);
      }
    }
  }
  sums.flush(dst, stride, buf);
}

// The fold of a 2D graph of several instances with new masks: a wave takes a
// tile at a time, 4 nodes per lane, so that every lane has work whatever the
// instances' row lengths are, and consecutive waves take neighbouring tiles.
// Bound by its reads and writes.  Row by row, each step a search for the
// instance and half of the lanes idle on rows of 400, 256 uneven images (171,000
// tiles) took 708 us; this takes 444.
constexpr int kFoldTiles = 8;  // tiles per wave

template <class S, int MASKS>
__global__ __launch_bounds__(256) void k_fold_tiles(Tiles T, Planes P, long long *red,
                                                    unsigned char *active, unsigned char *defi,
                                                    int zero_h, unsigned *mask0) {
  const int lane = threadIdx.x & 63;
  const int lx = lane % (S::TW / 4) * 4, ly = lane / (S::TW / 4);
  const int t0 = blockIdx.x * (4 * kFoldTiles) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  long long sum[3] = {0, 0, 0};
  int cur = -1;
  auto flush = [&]() {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      for (int o = 32; o > 0; o >>= 1) sum[k] += __shfl_xor(sum[k], o);
      const int slot = k == 0 ? RED_CONST : k == 1 ? RED_DEF0 : RED_SUP0;
      if (lane == 0 && sum[k])
        atomicAdd((unsigned long long *)&red[(long long)cur * RED_SLOTS + slot],
                  (unsigned long long)sum[k]);
      sum[k] = 0;
    }
  };
  for (int i = 0; i < kFoldTiles; ++i) {
    const int t = t0 + 4 * i;
    if (t >= T.ntiles) break;
    const int inst = T.tile_inst[t];
    if (inst != cur) {
      if (cur >= 0) flush();
      cur = inst;
    }
    const TileRef r = tile_ref_of<S>(T.inst[inst], t);
    const int K = r.I.K, y = r.oy + ly;
    // rows start at multiples of 32 nodes, so a lane's 4 nodes are aligned and
    // its loads past the row's end stay in its padding
    const int n = y < r.I.ny ? min(4, r.I.nx - (r.ox + lx)) : 0;
    const bool in = n > 0;
    const long long v = in ? node_index(r.I, r.ox + lx, y, 0) : 0;
    const int4 a = *(const int4 *)(P.cs + v), b = *(const int4 *)(P.ct + v);
    int4 c[S::KMAX];
#pragma unroll
    for (int d = 0; d < S::KMAX; ++d)
      c[d] = d < K ? *(const int4 *)(P.c0 + d * P.stride + v) : make_int4(0, 0, 0, 0);
    int4 m = make_int4(0, 0, 0, 0);
#pragma unroll
    for (int d = 0; d < S::KMAX; ++d) {
      const int fresh = d < K ? 1 << (8 + d) : 0;
      m.x |= (c[d].x > 0 ? 1 << d : 0) | fresh; m.y |= (c[d].y > 0 ? 1 << d : 0) | fresh;
      m.z |= (c[d].z > 0 ? 1 << d : 0) | fresh; m.w |= (c[d].w > 0 ? 1 << d : 0) | fresh;
    }
    bool excess = false, deficit = false;
    if (in) {
      int4 e;
      e.x = a.x - b.x; e.y = a.y - b.y; e.z = a.z - b.z; e.w = a.w - b.w;
      store4(P.e, v, n, e);
      if (zero_h) store4(P.h, v, n, make_int4(0, 0, 0, 0));
      store4((int *)P.rmask, v, n, m);
      if (MASKS == 2) store4((int *)mask0, v, n, m);
      for (int j = 0; j < n; ++j) {
        const int s = comp(a, j), u = comp(b, j);
        sum[0] += min(s, u);
        sum[1] += max(u - s, 0);
        sum[2] += max(s - u, 0);
        excess |= s > u;
        deficit |= s < u;
      }
    }
    const bool any_excess = __ballot(excess) != 0, any_deficit = __ballot(deficit) != 0;
    if (lane == 0) {
      if (active && any_excess) active[t] = 1;
      if (defi && any_deficit) defi[t] = 1;
    }
  }
  if (cur >= 0) flush();
}

void launch_fold(int shape, const Tiles &T, const Planes &P, long long *red,
                 unsigned char *active, unsigned char *defi, bool zero_h, unsigned *mask0,
                 int masks, hipStream_t st, bool cleared) {
  if (!cleared) {
    if (active) launch_fill_u8(active, T.ntiles, 0, st);
    if (defi) launch_fill_u8(defi, T.ntiles, 0, st);
  }
  const int z = zero_h ? 1 : 0;
  const int n = (T.nrows + T.row_step - 1) / T.row_step;
  if (masks >= 2 && T.ninst > 1 && !shape_is_3d(shape)) {
    const int grid = (T.ntiles + 4 * kFoldTiles - 1) / (4 * kFoldTiles);
    const auto go = [&](auto *kernel) {
      kernel<<<grid, 256, 0, st>>>(T, P, red, active, defi, z, mask0);
    };
    JFC_DISPATCH_2D(shape, go(masks == 3 ? &k_fold_tiles<S, 3> : &k_fold_tiles<S, 2>));
  } else if (masks == 3) {
    JFC_DISPATCH(shape, (k_fold<S, 3><<<row_grid<&k_fold<S, 3>>(n), 256, 0, st>>>(
                            T, P, red, active, defi, z, mask0)));
  } else if (masks == 2) {
    JFC_DISPATCH(shape, (k_fold<S, 2><<<row_grid<&k_fold<S, 2>>(n), 256, 0, st>>>(
                            T, P, red, active, defi, z, mask0)));
  } else if (masks == 1) {
    JFC_DISPATCH(shape, (k_fold<S, 1><<<row_grid<&k_fold<S, 1>>(n), 256, 0, st>>>(
                            T, P, red, active, defi, z, mask0)));
  } else {
    JFC_DISPATCH(shape, (k_fold<S, 0><<<row_grid<&k_fold<S, 0>>(n), 256, 0, st>>>(
                            T, P, red, active, defi, z, mask0)));
  }
}

// Cut energy on the input capacities (QGCWidget.cpp:2452-2520), summed per
// instance into energy[inst] (zeroed by the caller).
template <class S>
__global__ __launch_bounds__(256) void k_energy(Tiles T, Planes P, long long *energy) {
  __shared__ long long buf[4];
  const Lane<S> L(threadIdx.x);
  const Chunk C(T.ntiles);
  int cur = -1;
  long long a = 0;
  for (int t = C.t0; t < C.t1; ++t) {
    const int inst = T.tile_inst[t];
    if (inst != cur) {
      if (cur >= 0) {
        const long long A = block_sum_ll(a, buf);
        if (threadIdx.x == 0) atomicAdd((unsigned long long *)&energy[cur], (unsigned long long)A);
      }
      cur = inst;
      a = 0;
    }
    const TileRef r = tile_ref<S>(T, t);
    const InstDesc &I = r.I;
    const int gx = r.ox + L.lx, gy = r.oy + L.ly, gz = r.oz + L.lz;
    if (gx < I.nx && gy < I.ny && gz < I.nz) {
      const long long v = node_index(I, gx, gy, gz);
      if (P.lab[v]) {
        a += P.ct[v];
#pragma unroll
        for (int d = 0; d < S::KMAX; ++d) {
          if (d >= I.K) break;
          int dx, dy, dz;
          dir_of<S::D3>(d, dx, dy, dz);
          const int X = gx + dx, Y = gy + dy, Z = gz + dz;
          if (X < 0 || X >= I.nx || Y < 0 || Y >= I.ny || Z < 0 || Z >= I.nz) continue;
          if (!P.lab[node_index(I, X, Y, Z)]) a += P.c0[d * P.stride + v];
        }
      } else {
        a += P.cs[v];
      }
    }
  }
  if (cur >= 0) {
    const long long A = block_sum_ll(a, buf);
    if (threadIdx.x == 0) atomicAdd((unsigned long long *)&energy[cur], (unsigned long long)A);
  }
}

void launch_energy(int shape, const Tiles &T, const Planes &P, long long *energy,
                   hipStream_t st) {
  JFC_DISPATCH(shape, (k_energy<S><<<tile_grid(T.ntiles), 256, 0, st>>>(T, P, energy)));
}

// Subgradient of the cut energy for instance `inst` (outputs in the
// instance's own node numbering).
// Bound by its writes, a float per node and output plane.  A wave takes chunks of
// 256 nodes of consecutive rows, 4 nodes per lane, or as many whole rows of up to
// 128 nodes at once as its lanes hold: the callers' rows have no padding, so what
// a wave writes to a plane is one run that shares only its end lines with the
// next (rows of 32-node tiles, of which every line was shared, took 807 us for
// 256 uneven images; this takes 446), and a lane reads the labels around its
// nodes as words.  With a row at a time whatever its length, and a binary search
// for its instance, a call over 1x2000000 took 996 us, over 8x256x256 49 and over
// 2000 grids of 16x16 42; they take 44,
// 23 and 25.
struct alignas(4) Float4 {
  float v[4];
};
constexpr int kShortRow = 32;  // groups of 4 nodes in a row that is taken with others

template <bool D3>
__global__ __launch_bounds__(256) void k_backward(Tiles T, Planes P, int row0, int nrows,
                                                  int rows_per_wave, float *dcs, float *dct,
                                                  float *dnb, long long user_total) {
  constexpr int KMAX = D3 ? 6 : 8;
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int row = row0 + wave * rows_per_wave;
  const int end = min(row0 + nrows, row + rows_per_wave);
  if (row >= end) return;
  // the row's instance: the last that begins at or before it, a lane per candidate
  int inst = 0;
  for (int n = T.ninst; n > 1;) {
    const int step = (n + 63) / 64, mine = lane * step;
    const bool begun = mine < n && T.row_off[inst + mine] <= row;
    const int k = __popcll(__ballot(begun)) - 1;
    inst += k * step;
    n = min(step, n - k * step);
  }
  InstDesc I = T.inst[inst];
  int first = T.row_off[inst], last = T.row_off[inst + 1];
  // the 4 nodes from column x of row rr (y, z) of the instance
  auto group = [&](int rr, int y, int z, int x) {
    // outputs in the callers' numbering: one instance (user_total = 0) its
    // own, with plane stride = its node count; all instances the graph's
    // concatenation, with plane stride = all their nodes
    const long long n = user_total ? user_total : (long long)I.nx * I.ny * I.nz;
    const long long out0 = (user_total ? I.user_off : 0) + (long long)rr * I.nx;
    const long long base = I.node_off + (long long)rr * I.px, slice = (long long)I.px * I.ny;
    // bit i of the labels around the 4 nodes: column x - 1 + i of a row, set
    // off the grid
    auto nonzero = [](unsigned w) {
      w |= w >> 4;
      w |= w >> 2;
      w |= w >> 1;
      return ((w & 0x01010101u) * 0x01020408u) >> 24;
    };
    auto around = [&](bool have, long long step, bool wide) {
      if (!have) return 63u;
      const unsigned char *p = P.lab + base + step + x;
      const int left = I.nx - x;  // columns x ... of the row
      unsigned m = nonzero(*(const unsigned *)p) << 1;
      if (wide && x > 0) m |= p[-1] ? 1u : 0u;
      else m |= 1u;
      if (wide && left > 4) m |= p[4] ? 32u : 0u;
      else m |= 32u;
      if (left < 4) m |= 63u << (left + 1) & 63u;
      return m;
    };
    const unsigned own = around(true, 0, true);
    const unsigned s = own >> 1 & 15u;
    const int cnt = min(4, I.nx - x);
    auto put = [&](float *plane, unsigned bits) {
      float *q = plane + out0 + x;
      if (cnt == 4) {
        Float4 f;
#pragma unroll
        for (int i = 0; i < 4; ++i) f.v[i] = (bits >> i) & 1u ? 1.f : 0.f;
        *(Float4 *)q = f;
      } else {
        for (int i = 0; i < cnt; ++i) q[i] = (bits >> i) & 1u ? 1.f : 0.f;
      }
    };
    if (dcs) put(dcs, ~s);
    if (dct) put(dct, s);
    if (!dnb) return;
    const bool diag = !D3 && I.K > 4;
    const unsigned up = around(y + 1 < I.ny, I.px, diag), dn = around(y > 0, -I.px, diag);
    unsigned front = 0, back = 0;
    if constexpr (D3) {
      back = around(z + 1 < I.nz, slice, false);
      front = around(z > 0, -slice, false);
    }
#pragma unroll
    for (int d = 0; d < KMAX; ++d) {
      if (d >= I.K) break;
      int dx, dy, dz;
      dir_of<D3>(d, dx, dy, dz);
      const unsigned m = dz > 0 ? back : dz < 0 ? front : dy > 0 ? up : dy < 0 ? dn : own;
      put(dnb + d * n, s & ~(m >> (1 + dx)));
    }
  };
  while (row < end) {
    if (row == last) {
      I = T.inst[++inst];
      first = last;
      last = T.row_off[inst + 1];
    }
    const int stop = min(end, last), ng = (I.nx + 3) / 4;
    if (ng <= kShortRow) {
      const int r = lane / ng, rows = 64 / ng;
      if (blockIdx.y == 0 && r < rows)
        for (int mine = row + r; mine < stop; mine += rows) {
          const int rr = mine - first;
          group(rr, rr % I.ny, rr / I.ny, 4 * (lane - r * ng));
        }
      row = stop;
    } else {
      int rr = row - first, y = rr % I.ny, z = rr / I.ny;
      for (; row < stop; ++row, ++rr) {
        for (int x = (blockIdx.y * 64 + lane) * 4; x < I.nx; x += gridDim.y * 256)
          group(rr, y, z, x);
        if (++y == I.ny) {
          y = 0;
          ++z;
        }
      }
    }
  }
}

// Rows [row0, row0 + nrows) of the graph; nx: the longest of them.  About 16,000
// waves: of few rows each its own chunks, of many short ones several each.
static void backward_rows(int shape, const Tiles &T, const Planes &P, int row0, int nrows, int nx,
                          float *dcs, float *dct, float *dnb, long long user_total,
                          hipStream_t st) {
  const int chunks = std::min((nx + 255) / 256, std::max(64, 16384 / nrows));
  const int ng = (nx + 3) / 4, together = ng <= kShortRow ? 64 / ng : 1;
  const int per_wave = (int)std::max<long long>(together, (long long)nrows * chunks / 16384);
  const dim3 grid((nrows + 4LL * per_wave - 1) / (4LL * per_wave), chunks);
  if (shape_is_3d(shape))
    k_backward<true><<<grid, 256, 0, st>>>(T, P, row0, nrows, per_wave, dcs, dct, dnb, user_total);
  else
    k_backward<false><<<grid, 256, 0, st>>>(T, P, row0, nrows, per_wave, dcs, dct, dnb, user_total);
}

void launch_backward(int shape, const Tiles &T, const Planes &P, const InstDesc &I, int row0,
                     float *dcs, float *dct, float *dnb, hipStream_t st) {
  backward_rows(shape, T, P, row0, I.ny * I.nz, I.nx, dcs, dct, dnb, 0, st);
}
void launch_backward_all(int shape, const Tiles &T, const Planes &P, int max_nx, float *dcs,
                         float *dct, float *dnb, long long user_total, hipStream_t st) {
  backward_rows(shape, T, P, 0, T.nrows, max_nx, dcs, dct, dnb, user_total, st);
}

// ---- list compaction (ballots + one atomic per 1024-lane block) ------------------
//
// Flagged entries of `src` are appended to the queue
// list and their flags cleared; with `mat`, entries of tiles whose residual
// planes are already written carry kEntryMat, so the push kernel knows it
// without a dependent load.  Each wave counts its hits with a ballot; the
// block adds its total to the list count (and to the sweep and run totals)
// with one atomic each, so a pass over 10^5..10^6 tiles costs a few hundred
// same-address atomics.
constexpr int kCompactBlock = 1024;

__global__ __launch_bounds__(kCompactBlock) void k_compact(const int *src, int n,
                                                           unsigned char *flag,
                                                           const unsigned char *mat,
                                                           const unsigned char *touched,
                                                           const unsigned char *hmat, Queue q,
                                                           int *sweep_cnt, long long *total,
                                                           const int *stop) {
  __shared__ int s_cnt[kCompactBlock / 64];
  __shared__ int s_base;
  // a sweep issued after the solve's decision to stop sweeping (a relabel is
  // due, no tile is active, or the sweep budget is spent) compacts nothing
  // and leaves the flags for the sweeps after the host has acted
  if (stop && *stop) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  int t = -1;
  bool f = false;
  if (i < n) {
    t = src[i];
    f = flag[t] != 0;
    if (f) flag[t] = 0;
  }
  const unsigned long long m = __ballot(f);
  const int w = threadIdx.x >> 6, lane = lane_id();
  if (lane == 0) s_cnt[w] = __popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    int sum = 0;
    for (int k = 0; k < kCompactBlock / 64; ++k) sum += s_cnt[k];
    int base = 0;
    if (sum) {
      base = atomicAdd(q.ctr + QSLOT * q.slot, sum);
      if (sweep_cnt) atomicAdd(sweep_cnt, sum);
      if (total) atomicAdd((unsigned long long *)total, (unsigned long long)sum);
    }
    s_base = base;
  }
  __syncthreads();
  if (f) {
    int base = s_base;
    for (int k = 0; k < w; ++k) base += s_cnt[k];
    int ent = t;
    if (mat) ent |= mat[t] ? kEntryMat : (touched && !touched[t] ? kEntryClean : 0);
    if (hmat && hmat[t]) ent |= kEntryHeights;
    q.list[base + __popcll(m & ((1ull << lane) - 1ull))] = ent;
  }
}

// End of a sweep: file the sweep's active-tile count (accumulated by the
// compactions in c.state[0]) under the sweep index c.state[1], start the next
// sweep, and decide on the device what the host would decide after reading
// the count, so that the host can queue sweeps ahead of its checks:
//   stop = 1: no tile was active (converged, or the certificate decides);
//   stop = 2: the active set neither shrank nor grew by more than
//             (1 - stall_ratio) over the last sweep since the last relabel, whose
//             cost the sweeps since have reached (a global relabel is due, or the
//             remaining excess is cut off from every deficit);
//   stop = 3: the sweep budget is spent;
//   stop = 4: the tile visits since the last relabel exceed the budget (the
//             work of relabel_work visits per tile), or the sweeps since have
//             cost kPatience times the last: a relabel is due.
// A sweep that starts with stop set compacts nothing and files nothing.
// Every sweep, no-op or not, posts its stop word to the host ring tagged with
// its sequence number in the solve, so that the host reads it with no copy
// and tells it from an older word in the same slot.
__device__ __forceinline__ void post_stop(const SweepCtl &c, int seq, int stop) {
  if (c.ring)
    __hip_atomic_store(c.ring + seq % c.ring_n, seq * 8 + stop, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

constexpr long long kPatience = 16;

__global__ void k_sweep_end(SweepCtl c) {
  // every word is loaded before any is stored: one lane's chain of round trips
  // is what the kernel takes
  int *st = c.state;
  const int seq = st[6], stopped = st[2], i = st[1], cnt = st[0], last = st[3];
  const long long visits = c.total[0], from = *(const long long *)(st + 4);
  const long long work = *(const long long *)(st + 8) + c.sweep_ns + c.visit_ns * cnt;
  const long long cost = *(const long long *)(st + 10);
  const int since = i - last;  // sweeps since the last relabel, before this one
  const bool filed = c.stall_ratio > 0.0 && i < c.cap;
  const int one = filed && since >= 1 ? c.hist[i - 1] : 0;
  const int two = filed && since >= 3 ? c.hist[i - 2] : 0;
  const int three = filed && since >= 3 ? c.hist[i - 3] : 0;
  st[6] = seq + 1;
  if (stopped) {
    post_stop(c, seq, stopped);
    return;
  }
  if (i < c.cap) c.hist[i] = cnt;
  st[0] = 0;
  st[1] = i + 1;
  *(long long *)(st + 8) = work;
  int stop = 0;
  if (cnt == 0) {
    stop = 1;
  } else if (i + 1 >= c.max_sweeps) {
    stop = 3;
  } else {
    // stalled: the active count repeats that of the sweep before, or two
    // sweeps running repeat the two before them (excess trading places
    // between two sets of tiles, sweep after sweep)
    auto near = [&](int a, int b) {
      return (double)a >= c.stall_ratio * b && a * c.stall_ratio <= (double)b;
    };
    bool stalled = false;
    // A stall counts once the sweeps since the last relabel have cost as much as
    // that relabel: a steady active set is often flow on its way, and a relabel
    // costs many sweeps on large graphs and less than one on small ones.  Costs
    // are those of the work (SweepCtl), not times: a host that looks late, or a
    // device that others use, changes nothing.  By the clock, geometric means
    // over seeds without this, at half, once, twice and four times the relabel's
    // time: 3750x2500 strokes 78.7, 71.3, 68.3, 65.0, 67.3 ms; 2560x1440x50 video
    // 60.5, 46.5, 39.9, 40.9, 38.0; 512^3 volume 27.0, 20.5, 19.7, 22.1, 26.7;
    // 181x217x181 scan 2.94, 3.07, 3.00, 3.36, 3.88; 1023x767 2.59, 2.73, 2.33,
    // 2.03, 2.05; 600x450 widget 1.90, 1.89, 1.78, 1.70, 1.56: once is a compromise.
    // Over other seeds, once by the clock and by cost: strokes 51.1 and 51.3, video
    // 8.87 and 8.92, volume 11.2 and 11.2, scan 1.71 and 1.70, 1023x767 0.95 and
    // 0.98, widget 0.53 and 0.53.
    if (filed && since >= 1 && work >= cost) {
      stalled = near(cnt, one);
      if (!stalled && since >= 3) stalled = near(cnt, two) && near(one, three);
    }
    // Few tiles that hand the same excess around count next to nothing as visits,
    // so a relabel is due, too, once the sweeps have cost as much as kPatience of
    // the last (stall_ratio = 0 has no other end of that than heights that climb
    // to the node count: 1000x1000 images 40-160 ms, 0.7 with it).
    const bool budget = c.budget > 0 && ((double)(visits - from) > (double)c.budget ||
                                         (cost > 0 && work > kPatience * cost));
    if (stalled) stop = 2;
    else if (budget) stop = 4;
  }
  st[2] = stop;
  post_stop(c, seq, stop);
}

void launch_sweep_end(const SweepCtl &c, hipStream_t st) { k_sweep_end<<<1, 1, 0, st>>>(c); }

// After a global relabel: every height is stored (hmat); with resume, sweeping
// goes on, and the relabel's sweep index and visit total are the base of the
// next stall and budget tests, its cost what the sweeps have to reach (charge; the
// relabel before the first sweep costs nothing here).  *quit (or null): the
// relabel's waves gave up waiting, so sweeping stops until the host has finished it.
__global__ void k_relabel_end(SweepCtl c, unsigned char *hmat, int n, const int *quit, int resume,
                              int charge) {
  int *st = c.state;
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  int far = tid < kFarSlots ? c.far[kFarLine * tid] : 0;
  const long long total = c.total[0];
  const int sweep = st[1];
  const bool unfinished = quit && *quit;
  if (tid < kFarSlots && (unfinished || resume)) {
    for (int o = 32; o > 0; o >>= 1) far = max(far, __shfl_xor(far, o));
    if (tid == 0) {
      st[2] = unfinished ? 5 : 0;
      if (!unfinished) {
        st[3] = sweep;
        *(long long *)(st + 4) = total;
        *(long long *)(st + 8) = 0;
        *(long long *)(st + 10) = charge ? c.relabel_ns + c.level_ns * far : 0;
      }
    }
  }
  if (unfinished) return;
  for (int i = tid; i < n; i += gridDim.x * blockDim.x) hmat[i] = 1;
}

void launch_relabel_end(const SweepCtl &c, unsigned char *hmat, int n, const int *quit, bool resume,
                        bool charge, hipStream_t st) {
  k_relabel_end<<<grid_for(n, 256, 1024), 256, 0, st>>>(c, hmat, n, quit, resume, charge);
}

void launch_compact(const int *src, int n, unsigned char *flag,
                    const unsigned char *mat, const unsigned char *touched, const Queue &q,
                    int *sweep_cnt, long long *total, const int *stop, hipStream_t st,
                    const unsigned char *hmat) {
  if (n <= 0) return;
  k_compact<<<(n + kCompactBlock - 1) / kCompactBlock, kCompactBlock, 0, st>>>(
      src, n, flag, mat, touched, hmat, q, sweep_cnt, total, stop);
}

// ---- persistent tile queue ----------------------------------------------------------

// Workgroups claim runs of `chunk` consecutive list entries (16 for long
// lists, down to 1 for short ones).  Each workgroup's first run is static
// (group b takes run first(b) < G, G = grid size), so short or empty lists
// cost no atomics.  Later runs are claimed dynamically, which balances tiles
// of very different cost.
// Workgroups are dispatched to the 8 XCDs round-robin (b % 8), so with 8
// heads, head x serves the workgroups of XCD x: runs >= G form groups of 8
// consecutive runs, group q belongs to head q % nheads, and a head hands out
// its groups' runs in order.  Neighbouring tiles of a jump-flooding band
// thus stay on one XCD's L2, and claims spread over 8 addresses in 8
// different cache lines.  Every run
// belongs to one head and every head has workgroups, so the list is always
// drained.  When the static first runs already cover the list (G * chunk >=
// count, the short lists of late sweeps) no claim is
// issued at all: thousands of workgroups claiming on 8 addresses would
// serialise there.  Slot s of `ctr` holds the list count at [QSLOT*s] and
// head h at [QSLOT*s + QWORD*(1+h)]; the consumer of slot s zeroes the other
// slot's words for the next producer.
//
// VisitCursor walks a queue that way for the push kernel.  A workgroup learns its next list entry while it discharges
// the current tile, so that a visit starts with neither a global load nor a
// barrier of its own: thread 0 works out the next position during the local
// iterations (the rest of the current run, else the run its claim obtained,
// in which case it claims the run after that at once) and loads its entry;
// it publishes position and entry in LDS before the visit's last barrier,
// after which every thread reads them.  A direct list (Queue::pick) is
// walked in strides of the grid instead, workgroup b from position b, each
// workgroup taking the next position whose tile is picked.
struct VisitCursor {
  Queue q;
  int count, chunk, head_id, nheads;
  int *heads;
  const int *list;
  int ahead;             // (thread 0) claim for the run after the current one
  int nidx, nend, nent;  // (thread 0) the next position, its run's end, its entry
  int *s;                // LDS: next position, run end, entry
  int idx, end, ent;     // current position (uniform; idx < 0: drained)
  __device__ __forceinline__ VisitCursor(const Queue &q_, int *lds3) : q(q_) {
    if (blockIdx.x == 0 && threadIdx.x < 9) q.ctr[QSLOT * (q.slot ^ 1) + QWORD * threadIdx.x] = 0;
    count = q.fixed_count >= 0 ? q.fixed_count : q.ctr[QSLOT * q.slot];
    chunk = min(16, max(1, count / (int)(gridDim.x * 4)));
    heads = q.ctr + QSLOT * q.slot + QWORD;
    list = q.list;
    s = lds3;
    const int b = blockIdx.x;
    if (q.pick) {
      chunk = 1;
      ahead = -1;
      if (threadIdx.x == 0) {
        find(b);
        publish();
      }
      __syncthreads();
      advance();
      return;
    }
    nheads = (gridDim.x % 8 == 0) ? 8 : 1;
    head_id = b % nheads;
    int first = b;
    if (gridDim.x % 64 == 0) {
      const int w = b >> 3;
      first = (((w >> 3) << 3) + (b & 7)) * 8 + (w & 7);
    }
    idx = first * chunk;
    end = min(idx + chunk, count);
    ahead = -1;
    nidx = -1;
    nend = nent = 0;
    if (idx < count) {
      ent = __builtin_amdgcn_readfirstlane(list[idx]);
      if (threadIdx.x == 0 && (long long)gridDim.x * chunk < count)
        ahead = atomicAdd(&heads[QWORD * head_id], 1);
    } else {
      idx = -1;
      ent = 0;
    }
  }
  // thread 0, direct list: take position i's tile if it is picked (and the
  // solve has not stopped sweeping); its entry, or -1
  __device__ __forceinline__ int take(int i) const {
    const int t = list[i];
    if (!q.pick[t]) return -1;
    q.pick[t] = 0;
    int e = t;
    if (q.mat) e |= q.mat[t] ? kEntryMat : (q.touched && !q.touched[t] ? kEntryClean : 0);
    if (q.hmat && q.hmat[t]) e |= kEntryHeights;
    if (q.cnt) atomicAdd(q.cnt, 1);
    if (q.total) atomicAdd((unsigned long long *)q.total, 1ull);
    return e;
  }
  // thread 0, direct list: the first taken position from i on, in strides of
  // the grid
  __device__ __forceinline__ void find(int i) {
    nidx = -1;
    nend = nent = 0;
    if (q.stop && *q.stop) return;
    for (; i < count; i += (int)gridDim.x) {
      const int e = take(i);
      if (e >= 0) {
        nidx = i;
        nend = i + 1;
        nent = e;
        return;
      }
    }
  }
  // thread 0, during a visit: the position after the current one, and its entry
  __device__ __forceinline__ void prefetch() {
    if (q.pick) {
      find(idx + (int)gridDim.x);
      return;
    }
    nidx = -1;
    if (idx + 1 < end) {
      nidx = idx + 1;
      nend = end;
    } else if (ahead >= 0) {
      const int k = ahead;  // k-th run handed out by this head
      const int run = (int)gridDim.x + 8 * (head_id + nheads * (k >> 3)) + (k & 7);
      if ((long long)run * chunk < count) {
        nidx = run * chunk;
        nend = min(nidx + chunk, count);
        ahead = (long long)gridDim.x * chunk < count ? atomicAdd(&heads[QWORD * head_id], 1) : -1;
      }
    }
    if (nidx >= 0) nent = list[nidx];
  }
  // thread 0, after prefetch() and before the visit's last barrier
  __device__ __forceinline__ void publish() const {
    s[0] = nidx;
    s[1] = nend;
    s[2] = nent;
  }
  // every thread, after the visit's last barrier
  __device__ __forceinline__ void advance() {
    idx = __builtin_amdgcn_readfirstlane(s[0]);
    end = __builtin_amdgcn_readfirstlane(s[1]);
    ent = __builtin_amdgcn_readfirstlane(s[2]);
  }
};

// ---- residual-arc masks and lazy residual planes ----------------------------------
//
// rmask[v] bit d = (residual of arc d of v > 0); bit 8 + d = "fresh": the
// residual still equals the input c0[d][v] and cap[d][v] has not been
// written in this solve.  The relabel and cut searches only need the low
// bits, so they read 4 bytes per node instead of K planes.  mask0 holds the
// bits of the input planes (every plane fresh), built once per change of the
// inputs and copied to rmask when a solve starts, both inside the fold pass
// (k_fold); k_push reads fresh planes
// from c0 and writes them to cap, so no separate reset copy of the residual
// planes is needed.
// Cells of the padded tile a connectivity reads outside the tile: the sides
// and corners in 2D, the faces in 3D.  (The edges and corners of a 3D padded
// tile are never read: 6-connected arcs only cross faces.)
template <class S>
struct Ring {
  static constexpr int N = S::D3 ? 2 * (S::TW * S::TH + S::TW * S::TD + S::TH * S::TD)
                                 : 2 * S::PW + 2 * S::TH;
  static __device__ __forceinline__ int pos(int k) {
    if constexpr (!S::D3) {
      if (k < S::PW) return k;
      k -= S::PW;
      if (k < S::PW) return (S::PH - 1) * S::PW + k;
      k -= S::PW;
      if (k < S::TH) return (k + 1) * S::PW;
      k -= S::TH;
      return (k + 1) * S::PW + S::PW - 1;
    } else {
      constexpr int XY = S::TW * S::TH, XZ = S::TW * S::TD, YZ = S::TH * S::TD;
      int x, y, z;
      if (k < 2 * XY) {
        const int q = k % XY;
        x = q % S::TW + 1;
        y = q / S::TW + 1;
        z = k < XY ? 0 : S::PD - 1;
      } else if (k < 2 * XY + 2 * XZ) {
        k -= 2 * XY;
        const int q = k % XZ;
        x = q % S::TW + 1;
        z = q / S::TW + 1;
        y = k < XZ ? 0 : S::PH - 1;
      } else {
        k -= 2 * XY + 2 * XZ;
        const int q = k % YZ;
        y = q % S::TH + 1;
        z = q / S::TH + 1;
        x = k < YZ ? 0 : S::PW - 1;
      }
      return x + S::PW * (y + S::PH * z);
    }
  }
};

// The ring split over the four waves of a 256-lane workgroup: wave w owns the
// kRingQ consecutive cells from w * kRingQ (consecutive cells are neighbours
// along a row or face, so a wave's loads stay on few lines), its lanes
// taking kRingPerLane of them each.
template <class S>
constexpr int kRingQ = (Ring<S>::N + 3) / 4;
template <class S>
constexpr int kRingPerLane = (kRingQ<S> + 63) / 64;

// A ring cell by its place: the padded cell, its coordinates in the tile and
// the arcs it has into the tile, which are the planes of the cell that flow
// out of the tile changes -- one across a face, three from a side of an
// 8-connected tile (a corner has one of the three).
template <class S, int KK>
struct RingCell {
  static constexpr int ARCS = !S::D3 && KK == 8 ? 3 : 1;
  int p, xyz;  // padded cell; x, y, z (a byte each), side, corner
  __device__ __forceinline__ explicit RingCell(int k) {
    p = Ring<S>::pos(k);
    int x, y, z, nout;
    bool inter;
    pad_coords<S>(p, x, y, z, inter, nout);
    const int side = x < 0 ? 0 : x >= S::TW ? 1 : y < 0 ? 2 : y >= S::TH ? 3 : z < 0 ? 4 : 5;
    xyz = (x & 255) | (y & 255) << 8 | (z & 255) << 16 | side << 24 | (nout > 1 ? 1 << 30 : 0);
  }
  // The cell as a value of its own: what a phase of the visit derives from it is
  // computed there, instead of being kept in registers from the launch's start.
  __device__ __forceinline__ RingCell again() const {
    RingCell q = *this;
    asm volatile("" : "+v"(q.p), "+v"(q.xyz));
    return q;
  }
  __device__ __forceinline__ int x() const { return __builtin_amdgcn_sbfe(xyz, 0, 8); }
  __device__ __forceinline__ int y() const { return __builtin_amdgcn_sbfe(xyz, 8, 8); }
  __device__ __forceinline__ int z() const { return S::D3 ? __builtin_amdgcn_sbfe(xyz, 16, 8) : 0; }
  // 0 / 1 left / right side, 2 / 3 low / high y, 4 / 5 low / high z
  __device__ __forceinline__ int side() const { return xyz >> 24 & 7; }
  // direction of arc i
  __device__ __forceinline__ int arc(int i) const {
    const int q = side();
    return i == 0 ? q : i == 1 ? 4 + (q & 1) : 0x7667 >> 4 * q & 15;
  }
  // the tile it lies in, relative to this one
  __device__ __forceinline__ int tile_step(const InstDesc &I) const {
    const int x_ = x(), y_ = y(), z_ = z();
    return (x_ >= S::TW) - (x_ < 0) +
           I.tx * ((y_ >= S::TH) - (y_ < 0) + (S::D3 ? I.ty * ((z_ >= S::TD) - (z_ < 0)) : 0));
  }
};

// ---- block-wise push-relabel -------------------------------------------------------
//
// One workgroup discharges one tile at a time: e, h and the K residual planes
// of the tile go to LDS with a halo of neighbour heights.  Each local
// iteration relabels every active node (e > 0, finite h) to
// min over residual arcs of h_nb + 1 when it has no admissible arc, then
// pushes min(e, c) along arcs with h == h_nb + 1 in direction order.  Heights
// are not written during the push phase, so an arc is never pushed both ways
// at once and the reverse residual of an arc is touched by one lane only;
// only excess needs LDS atomics.  Flow pushed into halo cells accumulates in
// their LDS slots and is flushed to HBM once per visit.  The loop ends when a
// whole iteration pushes nothing (graphcut_push_relabel.cl:77-182) or after
// max_iters iterations -- up to sparse_iters when the launch's list is no
// longer than its grid (every workgroup holds at most one tile, so a visit
// that keeps iterating delays no other tile, and the flow crosses the tile in
// one visit instead of one sweep per step).
// ONE: a one-instance graph, whose descriptor every visit reads from the
// kernel arguments instead of loading it behind the tile index.
template <class S, bool ONE, int KK>
// KK: directions of the arrays (4 in a 2D graph without 8-connected
// instances).  A visit is bound by its chain of LDS round trips and, with
// several tiles on a CU, by VALU issue: heights and residuals kept in
// registers through an iteration and 4 directions instead of 8 took a
// 600x450 widget cut from 1.08 to 0.87 ms and a 181x217x181 scan from 2.5 to
// 2.1; with 8 directions 3750x2500 strokes from 46 to 42.
// Dense launches visit 121 tiles a microsecond at any shape and K (15000x10000,
// 256 images, the 2560x1440x50 video), with 20 KB moved per visit at 2.3 TB/s,
// the VALU busy 38% of the time; 6, 7 or 8 waves per SIMD and plain stores
// instead of half of the atomics change it by 1%: bound by the scattered 64-byte
// requests of borders.  What a visit derives per plane and per ring cell it
// derives in its phase, from one lane offset and two words a cell: 77 VGPRs
// for 8 directions (24 spilled otherwise, 4.77 ms against 4.40), and 4000x3000
// 1.349 -> 1.322 ms, the video's launches 1.36 -> 1.28.
__global__ __launch_bounds__(256, kRingPerLane<S> > 1 || KK == 8 ? 6 : 7) void k_push(
    Tiles T, Planes P, Queue q, unsigned char *flag, unsigned char *mat, unsigned char *touched,
    unsigned char *hmat, int max_iters, int sparse_iters,
    const int *sweep_state, long long *iter_total) {
  __shared__ int s_h[S::PADN];
  __shared__ int s_e[S::PADN];
  __shared__ int s_c[KK][S::PADN];
  const int tid = threadIdx.x;
  const Lane<S> L(tid);
  __shared__ int s_next[3];
  __shared__ int s_w[8];
  int par = 0;
  VisitCursor Qc(q, s_next);
  // a sparse launch's cap doubles with every sweep up to sparse_iters: a solve
  // that ends within a few sweeps has nothing to gain from long visits
  const int sweep = min(sweep_state[1], 30);
  // (a direct list is of at most a few thousand tiles and counts those that are not
  // active, too: never dense)
  const int cap_iters = Qc.count > (int)gridDim.x && !q.pick ? max_iters
                        : (sparse_iters >> sweep) < max_iters ? sparse_iters
                                                              : max_iters << sweep;
  long long my_iters = 0;
  // a wave's lanes cover RW rows of one slice of the tile from row wy, slice wz
  constexpr int RW = 64 / S::TW, RPL = kRingPerLane<S>;
  using Cell = RingCell<S, KK>;
  // Four colour classes (2D graphs with 8-connected instances): no two tiles of
  // a class touch one node, so a ring cell's excess and mask word are stored
  // plainly.  With two classes a node at the corner of its tile is in the ring
  // of two tiles of the other class.
  constexpr bool kAlone = !S::D3 && KK == 8;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wy = wave * RW % S::TH, wz = wave * RW / S::TH;
  // the ring, split evenly over the four waves so that each wave loads, clears
  // and flushes the same number of cells; the workgroup barrier after the flush
  // then waits for no straggling wave
  const int k0 = wave * kRingQ<S> + lane;
  const Cell cell0(min(k0, Ring<S>::N - 1)), cell1(min(k0 + 64, Ring<S>::N - 1));
  auto ring_cell = [&](int c) { return (c ? cell1 : cell0).again(); };
  auto has_cell = [&](int c) {
    return c * 64 + lane < kRingQ<S> && wave * kRingQ<S> + c * 64 + lane < Ring<S>::N;
  };
  while (Qc.idx >= 0) {
    const int ent = Qc.ent;
    const int t = ent & kEntryTile;
    const TileRef r = ONE ? tile_ref_of<S>(T.one, t) : tile_ref<S>(T, t);
    const InstDesc &I = r.I;
    const int K = ONE || KK < 8 ? KK : I.K;  // (a compile-time count but in mixed batches)
    const int gx = r.ox + L.lx, gy = r.oy + L.ly, gz = r.oz + wz;
    const bool valid = gx < I.nx && gy < I.ny && gz < I.nz;
    // A valid label never exceeds the distance to a deficit node, which is
    // below the node count; a label that reaches it proves the node cut off
    // (the role of cl_max_height in graphcut_push_relabel.cl, made exact).
    const long long nn = (long long)I.nx * I.ny * I.nz;
    const int hcap = nn < HINF ? (int)nn : HINF;
    // A tile whose every plane is already written in this solve (kEntryMat,
    // from mat[t]) loads cap directly; a tile no visit or flush has written
    // yet (kEntryClean) loads c0 directly, and its mask words are those of
    // the inputs (every plane fresh, residual bits c0 > 0), so neither needs
    // its mask word before its plane loads; otherwise the per-plane fresh
    // bits pick c0 or cap.
    const bool fresh_tile = (ent & kEntryMat) == 0;
    const bool clean = (ent & kEntryClean) != 0;

    // ---- loads: every global load of the visit is issued before any is
    // used; lanes off the grid, planes d >= K and dead halo cells read a
    // valid dummy address and discard the value.  Addresses are a uniform
    // base per plane and one lane offset for all planes.
    const bool wave_in = r.oy + wy < I.ny && gz < I.nz;
    const long long wb = wave_in ? node_index(I, r.ox, r.oy + wy, gz) : I.node_off;
    const long long off = valid ? L.lx + (long long)I.px * (lane / S::TW) : 0;
    // (the stride as a value of the phase, so that its multiples are not kept)
    auto phase_stride = [&]() {
      long long v = P.stride;
      asm volatile("" : "+s"(v));
      return v;
    };
    long long st = phase_stride();
    auto plane = [&](int d) { return (d < K ? d * st : 0) + wb; };
    // the node of a live ring cell, relative to the tile's first
    const long long tb = node_index(I, r.ox, r.oy, r.oz);
    auto ring_node = [&](const Cell &q) {
      return q.x() + (long long)I.px * (q.y() + (S::D3 ? I.ny * q.z() : 0));
    };
    bool live[RPL];
    int hh[RPL], he[RPL];
    unsigned hm[RPL];
#pragma unroll
    for (int c = 0; c < RPL; ++c) {
      const Cell q = ring_cell(c);
      live[c] = has_cell(c) && (unsigned)(r.ox + q.x()) < (unsigned)I.nx &&
                (unsigned)(r.oy + q.y()) < (unsigned)I.ny &&
                (!S::D3 || (unsigned)(r.oz + q.z()) < (unsigned)I.nz) &&
                (S::D3 || K > 4 || !(q.xyz >> 30));
      const long long g = tb + (live[c] ? ring_node(q) : 0);
      // a neighbour tile without stored heights in this solve reads as 0
      const int hw = P.h[g];
      hh[c] = hmat[live[c] ? t + q.tile_step(I) : t] ? hw : 0;
      hm[c] = P.rmask[g];
      he[c] = kAlone ? P.e[g] : 0;
    }
    // heights not yet stored in this solve read as 0 (the start labelling);
    // the visit then stores all of them.  The compaction read hmat[t] into
    // the entry, so no load stands between the entry and the plane loads.
    const bool h_stored = (ent & kEntryHeights) != 0;
    const int hw0 = (P.h + wb)[off];
    int e0 = (P.e + wb)[off], h0 = h_stored ? hw0 : 0;
    unsigned rm = 0;
    int c0r[KK];
    if (!fresh_tile) {
#pragma unroll
      for (int d = 0; d < KK; ++d) c0r[d] = (P.cap + plane(d))[off];
    } else if (clean) {
#pragma unroll
      for (int d = 0; d < KK; ++d) c0r[d] = (P.c0 + plane(d))[off];
      rm = ((1u << K) - 1) << 8;
#pragma unroll
      for (int d = 0; d < KK; ++d)
        if (d < K) rm |= min((unsigned)c0r[d], 1u) << d;
    } else {
      rm = (P.rmask + wb)[off];
#pragma unroll
      for (int d = 0; d < KK; ++d)
        c0r[d] = (((rm >> (8 + d)) & 1u ? P.c0 : P.cap) + plane(d))[off];
    }
    if (!valid) {
      e0 = 0;
      h0 = HINF;
      rm = 0;
    }
#pragma unroll
    for (int d = 0; d < KK; ++d)
      if (!(valid && d < K)) c0r[d] = 0;

    s_e[L.me] = e0;
    s_h[L.me] = h0;
#pragma unroll
    for (int d = 0; d < KK; ++d) s_c[d][L.me] = c0r[d];
#pragma unroll
    for (int c = 0; c < RPL; ++c) {
      if (!has_cell(c)) continue;
      const Cell q = ring_cell(c);
      s_h[q.p] = live[c] ? hh[c] : HINF;
      s_e[q.p] = 0;
#pragma unroll
      for (int i = 0; i < Cell::ARCS; ++i) s_c[q.arc(i)][q.p] = 0;
    }
    __syncthreads();
    // the next entry loads while the tile iterates
    if (tid == 0) Qc.prefetch();

    // The iterations.  A node's height is written by its own lane alone and
    // stays in a register, as do its residuals from the relabel to the push.
    // Every LDS word a phase needs is read before any is used, so a phase
    // waits on LDS once instead of once per direction.
    int it = 0, any, e = e0, h = h0;
    do {
      // relabel (monotone; neighbours may be read before or after their own
      // relabel in this iteration, which keeps the labelling valid)
      const bool live = valid && e > 0 && h < HINF;
      int cv[KK], hv[KK];
      if (live) {
#pragma unroll
        for (int d = 0; d < KK; ++d) {
          cv[d] = s_c[d][L.me];
          hv[d] = s_h[L.me + lds_off<S>(d)];
        }
        // planes d >= K hold 0, so their arcs drop out like saturated ones
        int m = HINF;
#pragma unroll
        for (int d = 0; d < KK; d += 2)
          m = min(m, min(cv[d] > 0 ? hv[d] : HINF, cv[d + 1] > 0 ? hv[d + 1] : HINF));
        m = m + 1 < hcap ? m + 1 : HINF;
        if (m > h) s_h[L.me] = h = m;
      }
      __syncthreads();
      // push.  The reverse residual s_c[d^1][nb] is written only by this
      // lane during the phase (its owner nb cannot push back along an arc
      // this lane pushes on: heights are frozen).
      int pushed = 0;
      if (live && h < HINF) {
#pragma unroll
        for (int d = 0; d < KK; ++d) hv[d] = s_h[L.me + lds_off<S>(d)];
        int rem = e;
        int f[KK];
#pragma unroll
        for (int d = 0; d < KK; ++d) f[d] = hv[d] == h - 1 ? cv[d] : 0;
#pragma unroll
        for (int d = 0; d < KK; ++d) {
          f[d] = min(rem, f[d]);
          rem -= f[d];
        }
#pragma unroll
        for (int d = 0; d < KK; ++d)
          if (f[d] > 0) {
            const int nb = L.me + lds_off<S>(d);
            s_c[d][L.me] = cv[d] - f[d];
            atomicAdd(&s_c[d ^ 1][nb], f[d]);
            atomicAdd(&s_e[nb], f[d]);
          }
        if (rem != e) {
          atomicAdd(&s_e[L.me], rem - e);
          pushed = 1;
        }
      }
      any = block_any(pushed, s_w, par);
      e = s_e[L.me];
    } while (any && ++it < cap_iters);
    my_iters += it + (any ? 0 : 1);
    if (tid == 0) Qc.publish();

    // ---- the flush's reads first: the flow that crossed into each ring cell
    // and the reverse-residual increments (LDS), and for increments into a
    // plane that is still fresh (its value lives in c0) the c0 value they add
    // to, loaded before the interior write-back so that its stores cover the
    // load latency.
    int fl[RPL], dc[RPL][Cell::ARCS], cf[RPL][Cell::ARCS];
    st = phase_stride();
#pragma unroll
    for (int c = 0; c < RPL; ++c) {
      const Cell q = ring_cell(c);
      fl[c] = live[c] ? s_e[q.p] : 0;
#pragma unroll
      for (int i = 0; i < Cell::ARCS; ++i) dc[c][i] = cf[c][i] = 0;
      if (fl[c] == 0) continue;
#pragma unroll
      for (int i = 0; i < Cell::ARCS; ++i) {
        const int d = q.arc(i);
        dc[c][i] = s_c[d][q.p];
        if (dc[c][i] != 0 && ((hm[c] >> (8 + d)) & 1u)) cf[c][i] = P.c0[d * st + tb + ring_node(q)];
      }
    }

    // ---- write back what changed (stores only)
    int act = 0;
    if (valid) {
      const int e1 = e, h1 = h;
      if (e1 != e0) (P.e + wb)[off] = e1;
      if (h1 != h0 || !h_stored) (P.h + wb)[off] = h1;
      // fresh planes are written whether or not they changed; the mask word
      // of a written tile holds residual bits only (exact, no fresh bits)
      unsigned m0 = 0, m1 = 0;
#pragma unroll
      for (int d = 0; d < KK; ++d)
        if (d < K) {
          const int c1 = s_c[d][L.me];
          if (clean || c1 != c0r[d] || ((rm >> (8 + d)) & 1u)) (P.cap + plane(d))[off] = c1;
          m0 |= min((unsigned)c0r[d], 1u) << d;
          m1 |= min((unsigned)c1, 1u) << d;
        }
      if (m1 != (fresh_tile ? rm : m0)) (P.rmask + wb)[off] = m1;
      act = e1 > 0 && h1 < HINF;
    }
    // ---- flush flow that crossed into the halo: excess and the reverse
    // residual of each crossing arc (graphcut_push_relabel.cl:184-195).
    // Plane d of halo node g is the arc from g into this tile, so no other
    // tile of this colour class touches plane d of g or its two mask bits in
    // this launch; other tiles may update other bits of the same mask word,
    // hence atomics.  A plane that is still fresh is written as c0 + dc; the
    // others take a fire-and-forget atomic add.
#pragma unroll
    for (int c = 0; c < RPL; ++c) {
      if (fl[c] == 0) continue;
      const Cell q = ring_cell(c);
      const long long g = tb + ring_node(q);
      // flow entered g, so some plane of g changes below: g's tile is no
      // longer clean
      if (kAlone) P.e[g] = he[c] + fl[c];
      else atomicAdd(&P.e[g], fl[c]);
      const int ht = t + q.tile_step(I);
      flag[ht] = 1;
      touched[ht] = 1;
      unsigned flip = 0;
#pragma unroll
      for (int i = 0; i < Cell::ARCS; ++i) {
        const int d = q.arc(i);
        if (dc[c][i] == 0) continue;
        if ((hm[c] >> (8 + d)) & 1u) {
          P.cap[d * st + g] = cf[c][i] + dc[c][i];
          flip |= 256u << d;
        } else {
          atomicAdd(&P.cap[d * st + g], dc[c][i]);
        }
        if (!((hm[c] >> d) & 1u)) flip |= 1u << d;
      }
      if (kAlone) {
        if (flip) P.rmask[g] = hm[c] ^ flip;
      } else if (flip) {
        atomicXor(&P.rmask[g], flip);
      }
    }
    act = block_any(act, s_w, par);
    if (act && tid == 0) flag[t] = 1;
    if (fresh_tile && tid == 0) mat[t] = 1;
    if (!h_stored && tid == 0) hmat[t] = 1;
    Qc.advance();
  }
  // one atomic per workgroup, spread over 64 counters
  if (tid == 0 && iter_total && my_iters)
    atomicAdd((unsigned long long *)&iter_total[blockIdx.x & 63], (unsigned long long)my_iters);
}

// kmax: the most directions of any instance (a 2D graph of 4-connected
// instances iterates over 4: half the LDS reads of 8).
void launch_push(int shape, int kmax, int nwg, const Tiles &T, const Planes &P,
                 const Queue &q, unsigned char *flag, unsigned char *mat,
                 unsigned char *touched, unsigned char *hmat,
                 int max_iters, int sparse_iters, const int *sweep_state,
                 long long *iter_total, hipStream_t st) {
  const auto go = [&](auto *kernel, int grid) {
    kernel<<<grid, 256, 0, st>>>(T, P, q, flag, mat, touched, hmat, max_iters, sparse_iters,
                                 sweep_state, iter_total);
  };
#define JFC_PUSH(ONE, KK) go(&k_push<S, ONE, KK>, resident_grid<&k_push<S, ONE, KK>>(nwg))
  JFC_DISPATCH(shape, {
    constexpr int k0 = S::D3 ? 6 : 4;
    if (T.ninst == 1 && kmax <= k0) JFC_PUSH(true, k0);
    else if (T.ninst == 1) JFC_PUSH(true, S::KMAX);
    else if (kmax <= k0) JFC_PUSH(false, k0);
    else JFC_PUSH(false, S::KMAX);
  });
#undef JFC_PUSH
}

}  // namespace jfc
