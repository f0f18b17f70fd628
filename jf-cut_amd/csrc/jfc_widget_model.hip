// jfc_widget_model.hip -- the widget's own data terms on the device: the
// "Model" button of QGCWidget (slotModelClicked,
// src/QVisualizer/Graph Cut/QGCWidget.cpp:2560-2606) with lazy snapping
// (k-means unary, inverse-distance pairwise) or BK (histogram unary,
// Gaussian pairwise).
//
// Reference counterparts (src/QVisualizer/cl/GraphCut/):
//   k_wm_scan        graphcut_count_cut / graphcut_scatter_cut   graphcut_count_block.cl:67-104
//                    + graphcut_cut_histogram, _distribution     graphcut_histogram.cl:19-60
//   k_wm_lloyd       the whole k-means                           graphcut_kmeans.cl:21-159,
//                                                                QGCWidget.cpp:2011-2102
//   k_wm_assign      graphcut_kmeans                             graphcut_kmeans.cl:21-159
//   k_wm_unary<lazy> graphcut_compute_excessflow_lazy / _bk      graphcut_compute_excessflow.cl:19-139
//   k_wm_pairwise    graphcut_compute_capacity_lazy / _bk        graphcut_compute_capacity.cl:21-254
//
// Float semantics.  Every float operation is the reference's, in its order,
// IEEE-rounded: no contraction into fused multiply-adds (the pragma below),
// correctly rounded division and square root, and exp / log evaluated in
// double and rounded once to float.  A CPU restatement with the same
// operation order therefore reproduces every integer output.
//
// Readings fixed here where the reference is undefined or racy:
//   - the k-means initial centroid of a seeded level is the pixel with the
//     highest node index at that level (graphcut_cut_distribution lets any
//     writer win);
//   - k-means centroid sums are exact (per-byte counts, summed in double in
//     byte order) before the division, instead of float partial sums in
//     tile order; a cluster with no member becomes 0 as in QGCW:2085-2096;
//   - the BK unary clamps its histogram level to 0..255 (the reference reads
//     past the table when the weighted dot product exceeds 1), a NaN unary
//     (0 * inf, inf - inf) becomes 0, and unaries saturate at +-2^30, the
//     library's capacity bound.
#pragma clang fp contract(off)

#include "jfcut.h"
#include "jfc_device.h"

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

namespace jfc {
int model_fail(int code, const std::string &msg);
int graph_instance(jfc_graph *g, int inst, InstDesc *I, int **cs, int **ct, int **c0,
                   long long *stride);
void graph_mark_inputs(jfc_graph *g, int inst);
void graph_inputs_failed(jfc_graph *g, int inst);
hipStream_t graph_stream(jfc_graph *g);
int graph_stage(jfc_graph *g, size_t bytes, void **p);
int graph_scratch(jfc_graph *g, size_t bytes, void **p);
int graph_work_plane(jfc_graph *g, int inst, int **plane, long long *n);
int graph_work_plane2(jfc_graph *g, int inst, int **plane);
}  // namespace jfc

using namespace jfc;

namespace {

constexpr int kMaxFlow = 32767;  // QGCSetting::cl_max_flow (QGCSetting.cpp:36)
constexpr int kLevels = 256;     // QGCSetting::sizeCutHistogram (QGCSetting.cpp:20)
constexpr int kMaxK = 32;        // spinBoxK maximum (QGCPanel.ui)
constexpr int kSat = 1 << 30;    // library capacity bound

struct W4 {
  float v[4];
};

// read_imagef of a CL_UNORM_INT8 texel: byte / 255
__device__ __host__ __forceinline__ float unorm8(unsigned b) { return (float)b / 255.0f; }

__device__ __forceinline__ void texel(const uchar4 *img, long long v, unsigned t[4]) {
  const uchar4 p = img[v];
  t[0] = p.x;
  t[1] = p.y;
  t[2] = p.z;
  t[3] = p.w;
}

// OpenCL dot(a, b), left to right
__device__ __forceinline__ float dot4(const float a[4], const W4 &w) {
  return ((a[0] * w.v[0] + a[1] * w.v[1]) + a[2] * w.v[2]) + a[3] * w.v[3];
}

// The square under OpenCL distance(c, p) = length(c - p).  Rounded square
// roots keep the order of their arguments, so the nearest distance is the
// root of the least square, and only near ties need the roots themselves.
__device__ __forceinline__ float dist4_sq(const float *c, const float p[4]) {
  const float d0 = c[0] - p[0], d1 = c[1] - p[1], d2 = c[2] - p[2], d3 = c[3] - p[3];
  return ((d0 * d0 + d1 * d1) + d2 * d2) + d3 * d3;
}

// The nearest of k centroids, first on ties of the rounded distances
// (graphcut_kmeans.cl:37-47).  s < best (1 - 2^-20) makes the roots differ by
// more than their rounding; s >= best makes them equal or larger.
__device__ __forceinline__ int nearest4(const float *c, int k, const float p[4]) {
  float best = dist4_sq(c, p);
  int idx = 0;
  for (int j = 1; j < k; ++j) {
    const float s = dist4_sq(c + 4 * j, p);
    if (s >= best) continue;
    if (s < best * (1.0f - 0x1p-20f) || sqrtf(s) < sqrtf(best)) {
      best = s;
      idx = j;
    }
  }
  return idx;
}

// nearest4 for up to KB centroids held in registers (c), whose copy in memory
// is m.  The squares are compared without branches; a centroid whose square is
// alone within 2^-18 of the least has the least rounded distance, and anything
// else (near ties, squares next to or at zero, values that are not finite) is
// nearest4's.
template <int KB>
__device__ __forceinline__ int nearest4_of(const float (&c)[4 * KB], const float *m, int k,
                                           const float p[4]) {
  float s[KB];
  s[0] = dist4_sq(c, p);
  float least = s[0];
#pragma unroll
  for (int j = 1; j < KB; ++j) {
    if (j >= k) break;
    s[j] = dist4_sq(c + 4 * j, p);
    least = fminf(least, s[j]);
  }
  const float near = least * (1.0f + 0x1p-18f);
  int idx = 0, within = 0;
#pragma unroll
  for (int j = 0; j < KB; ++j) {
    if (j >= k) break;
    const bool in = s[j] <= near;
    idx = in ? j : idx;
    within += in;
  }
  if (within != 1 || !(least >= 1e-30f) || !(s[0] == s[0])) return nearest4(m, k, p);
  return idx;
}

// the wave's sum of v, in lane 63
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_update_dpp(0u, (unsigned)b, CTRL, ROWS, 0xf, ROWS == 0xf);
  const unsigned hi =
      __builtin_amdgcn_update_dpp(0u, (unsigned)(b >> 32), CTRL, ROWS, 0xf, ROWS == 0xf);
  return v + __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}
__device__ __forceinline__ double wave_sum(double v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr:1
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);  // row_bcast:15
  return dpp_add<0x143, 0xc>(v);  // row_bcast:31
}

// histogram level of a seeded pixel: clamp(dot, 0, 1) * (size - 1) + 0.5,
// truncated (graphcut_histogram.cl:33-35)
__device__ __forceinline__ int level_clamped(float data) {
  data = fminf(fmaxf(data, 0.0f), 1.0f);
  return (int)(data * (float)(kLevels - 1) + 0.5f);
}

// float unary -> int: round half away from zero, NaN -> 0, saturate
__device__ __forceinline__ int unary_int(float v) {
  if (v != v) return 0;
  const float r = roundf(v);
  if (r >= (float)kSat) return kSat;
  if (r <= -(float)kSat) return -kSat;
  return (int)r;
}

// Scratch of one call.  Everything up to rep is copied back at the end.
struct WmScratch {
  int *ctl;          // [0,1] seeded pixels per side, [2] a side has more than k_wm_lloyd takes,
                     // [3,4] k-means iterations
  unsigned *hist;    // [2][kLevels] seeded pixels per level
  float *cent;       // [2][kMaxK * 4] the centroids of the unary, side 1 from k * 4 on
  unsigned *rep;     // [2][kLevels] highest node index + 1 per seeded level
  unsigned *acc;     // [kMaxK * 4][kLevels] byte counts of an assignment (k_wm_assign)
  uchar4 *list[2];   // the seeded pixels
  unsigned char *owner;  // [2][kLloydSeeds] their clusters (k_wm_lloyd)
};
constexpr int kLloydSeeds = 65536;
// ... and seeds times clusters: one compute unit a side takes the time of their
// product, the host's iterations (an assignment over the whole device, a wait, the
// update) little more for more of either.  32 clusters: 6.0 ms on the device and 6.6
// by the host for 40,000 seeds, 7.1 and 7.2 for 48,000, 9.4 and 8.0 for 65,000; 24
// clusters, 65,000: 7.1 and 8.4.
constexpr int kLloydWork = 49152 * 32;
constexpr size_t kCtlBytes = 64, kHistBytes = 2 * kLevels * 4, kCentBytes = 2 * kMaxK * 4 * 4,
                 kRepBytes = kHistBytes, kAccBytes = (size_t)kMaxK * 4 * kLevels * 4,
                 kOwnerBytes = 2 * kLloydSeeds;
constexpr size_t kBackBytes = kCtlBytes + kHistBytes + kCentBytes;

// One pass over the seed bytes: per side the seeded pixels in a list, their
// level histogram (graphcut_cut_histogram) and the highest node index + 1 per
// level (graphcut_cut_distribution).  Four pixels per lane; a workgroup's
// histograms meet in LDS.
__global__ __launch_bounds__(256) void k_wm_scan(const uchar4 *img, const unsigned char *fg,
                                                 const unsigned char *bg, long long n, W4 w,
                                                 WmScratch S) {
  __shared__ unsigned s_h[2][kLevels], s_r[2][kLevels];
  __shared__ int s_any;
  for (int i = threadIdx.x; i < 2 * kLevels; i += 256) (&s_h[0][0])[i] = (&s_r[0][0])[i] = 0;
  if (threadIdx.x == 0) s_any = 0;
  __syncthreads();
  const bool al = (((size_t)fg | (size_t)bg) & 3) == 0;
  const long long groups = (n + 3) / 4;
  for (long long base = (long long)blockIdx.x * 256; base < groups;
       base += (long long)gridDim.x * 256) {
    const long long g = base + threadIdx.x, v0 = 4 * g;
    unsigned m[2] = {0u, 0u};
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const unsigned char *p = side ? bg : fg;
      if (g < groups) {
        if (al && v0 + 4 <= n) {
          m[side] = *(const unsigned *)(p + v0);
        } else {
          for (int j = 0; j < 4; ++j)
            if (v0 + j < n) m[side] |= (unsigned)p[v0 + j] << (8 * j);
        }
      }
    }
    if (!__ballot((m[0] | m[1]) != 0)) continue;
    s_any = 1;
#pragma unroll
    for (int side = 0; side < 2; ++side)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool on = ((m[side] >> (8 * j)) & 255u) != 0;
        const unsigned long long b = __ballot(on);
        if (!b) continue;
        int at = 0;
        if (lane_id() == 0) at = atomicAdd(&S.ctl[side], __popcll(b));
        at = __builtin_amdgcn_readfirstlane(at);
        if (!on) continue;
        const uchar4 t = img[v0 + j];
        S.list[side][at + __popcll(b & ((1ull << lane_id()) - 1ull))] = t;
        const float f[4] = {unorm8(t.x), unorm8(t.y), unorm8(t.z), unorm8(t.w)};
        const int lv = level_clamped(dot4(f, w));
        atomicAdd(&s_h[side][lv], 1u);
        atomicMax(&s_r[side][lv], (unsigned)(v0 + j) + 1u);
      }
  }
  __syncthreads();
  if (!s_any) return;
  for (int i = threadIdx.x; i < 2 * kLevels; i += 256) {
    const unsigned h = (&s_h[0][0])[i];
    if (!h) continue;
    atomicAdd(&S.hist[i], h);
    atomicMax(&S.rep[i], (&s_r[0][0])[i]);
  }
}

// The k-means of a side (blockIdx.x) with up to `limit` seeded pixels, one
// workgroup of 1024 lanes: initial centroids from the seeded levels'
// representatives, picked at (count - 1) * i / (k - 1) and scaled by weight /
// 255 (QGCW:2011-2039), then Lloyd iterations (QGCW:2073-2102) until the
// centroids move by less than 1 / 1024.  The centroids of the last assignment
// are the ones the unary uses.  An assignment counts bytes per cluster and
// channel; a mean is the exact sum of count * value, which float64 holds in
// any order (a term is a multiple of the smallest value's last bit, and
// 2^16 of them span under 53 bits), divided and rounded once.
// Bound by the vector and LDS instructions of one compute unit, an iteration a
// chain of them: the k-means of a 600x450 image, 8 clusters, takes 140 us; with
// every pixel counted anew in each iteration (an opaque image counts one alpha
// value: 64 lanes on one LDS word), a branch per centroid and sums over lane
// shifts it took 208.  The counts are kept from iteration to iteration, only
// the pixels that change cluster touch them, and up to 8 centroids stay in
// scalar registers.
template <int KB>
__global__ __launch_bounds__(1024) void k_wm_lloyd(const uchar4 *img, W4 w, W4 scale, int k,
                                                   int iterations, int limit, WmScratch S) {
  __shared__ unsigned s_acc[KB * 4][kLevels];
  __shared__ float s_val[4][kLevels];  // weighted feature of a byte per channel
  __shared__ float s_cent[2][KB * 4];  // the centroids, and those of the next iteration
  __shared__ int s_lv[kLevels];        // seeded levels in order
  __shared__ int s_levels;
  const int side = blockIdx.x, tid = threadIdx.x;
  const int n = S.ctl[side];
  if (n == 0) return;
  if (n > limit) {
    if (tid == 0) S.ctl[2] = 1;
    return;
  }
  (&s_val[0][0])[tid] = unorm8(tid & 255) * w.v[tid >> 8];
  if (tid < 64) {
    int c = 0;
#pragma unroll
    for (int q = 0; q < kLevels / 64; ++q) {
      const unsigned rp = S.rep[side * kLevels + 64 * q + tid];
      const unsigned long long b = __ballot(rp != 0);
      if (rp) s_lv[c + __popcll(b & ((1ull << tid) - 1ull))] = (int)(rp - 1u);
      c += __popcll(b);
    }
    if (tid == 0) s_levels = c;
  }
  __syncthreads();
  if (tid < k * 4) {
    const unsigned dsize = (unsigned)s_levels - 1u;
    const uchar4 t = img[s_lv[dsize * (unsigned)(tid >> 2) / (unsigned)(k - 1)]];
    const int c = tid & 3;
    s_cent[0][tid] = (float)(c == 0 ? t.x : c == 1 ? t.y : c == 2 ? t.z : t.w) * scale.v[c];
  }
  for (int i = tid; i < k * 4 * kLevels; i += 1024) (&s_acc[0][0])[i] = 0;
  __syncthreads();
  const uchar4 *list = S.list[side];
  unsigned char *owner = S.owner + side * kLloydSeeds;
  constexpr int kNone = 255;
  int it = 0, cur = 0;
  for (;; cur ^= 1) {
    const float *m = s_cent[cur];
    constexpr bool kRegs = KB <= 8;  // (more centroids don't fit the scalar registers)
    float c[kRegs ? 4 * KB : 1];
    if constexpr (kRegs) {
#pragma unroll
      for (int q = 0; q < 4 * KB; ++q)
        c[q] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(m[q])));
    }
    uchar4 t = make_uchar4(0, 0, 0, 0);
    int old = kNone;
    if (tid < n) {
      t = list[tid];
      if (it) old = owner[tid];
    }
    for (int i = tid; i < n; i += 1024) {
      const uchar4 now = t;
      const int was = old;
      if (i + 1024 < n) {  // the next pixel loads meanwhile
        t = list[i + 1024];
        if (it) old = owner[i + 1024];
      }
      const float p[4] = {s_val[0][now.x], s_val[1][now.y], s_val[2][now.z], s_val[3][now.w]};
      int j;
      if constexpr (kRegs) j = nearest4_of<KB>(c, m, k, p);
      else j = nearest4(m, k, p);
      if (j == was) continue;
      owner[i] = (unsigned char)j;
      const int v[4] = {now.x, now.y, now.z, now.w};
#pragma unroll
      for (int q = 0; q < 4; ++q) atomicAdd(&s_acc[j * 4 + q][v[q]], 1u);
      if (was != kNone) {
#pragma unroll
        for (int q = 0; q < 4; ++q) atomicSub(&s_acc[was * 4 + q][v[q]], 1u);
      }
    }
    __syncthreads();
    // one wave per cluster and channel, four byte values per lane
    float *next = s_cent[cur ^ 1];
    for (int r = tid >> 6; r < k * 4; r += 16) {
      double sum = 0.0;
      unsigned members = 0;
#pragma unroll
      for (int q = 0; q < kLevels / 64; ++q) {
        const int b = 64 * q + (tid & 63);
        const unsigned count = s_acc[r][b];
        sum += (double)count * (double)s_val[r & 3][b];
        members += count;
      }
      sum = wave_sum(sum);
      const double all = wave_sum((double)members);
      if ((tid & 63) == 63) next[r] = all > 0.0 ? (float)(sum / all) : 0.0f;
    }
    __syncthreads();
    ++it;
    // every wave for itself, from the same words
    bool moved = false;
    if ((tid & 63) < k) {
      // glm::length(centroid - previous)
      const int at = (tid & 63) * 4;
      float d[4];
      for (int q = 0; q < 4; ++q) d[q] = next[at + q] - m[at + q];
      const float len = sqrtf((d[0] * d[0] + d[1] * d[1]) + (d[2] * d[2] + d[3] * d[3]));
      moved = !(len < 1.0f / 1024);
    }
    if (!__ballot(moved) || it >= iterations) break;
  }
  if (tid < k * 4) S.cent[side * k * 4 + tid] = s_cent[cur][tid];
  if (tid == 0) S.ctl[3 + side] = it;
}

// One Lloyd assignment over more seeded pixels of a side than k_wm_lloyd
// takes: per cluster and channel, a count per byte value, from which the
// host forms exact sums.
__global__ void k_wm_assign(const uchar4 *list, int n, W4 w, const float *cent, int k,
                            unsigned *acc) {
  __shared__ float s_c[kMaxK * 4];
  for (int i = threadIdx.x; i < k * 4; i += blockDim.x) s_c[i] = cent[i];
  __syncthreads();
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const uchar4 u = list[i];
    const unsigned t[4] = {u.x, u.y, u.z, u.w};
    float p[4];
    for (int c = 0; c < 4; ++c) p[c] = unorm8(t[c]) * w.v[c];
    const int idx = nearest4(s_c, k, p);
    for (int c = 0; c < 4; ++c) atomicAdd(&acc[(idx * 4 + c) * kLevels + t[c]], 1u);
  }
}

// Unary terms, one row of an instance per loop step.  LAZY: distance to the
// nearest centroid of each side (graphcut_compute_excessflow.cl:47-77,
// 109-139); BK: negative log-likelihood from the seeded level histograms
// (graphcut_compute_excessflow.cl:19-45, 79-107).  Seeds: +-cl_max_flow,
// foreground first.  Nothing is written when a side has no seeds, or too many
// for k_wm_lloyd (the host then runs the k-means and launches again).
template <bool LAZY>
__global__ __launch_bounds__(256) void k_wm_unary(
    const uchar4 *img, const unsigned char *fg, const unsigned char *bg, int n, W4 w,
    WmScratch S, int k, int shift, float lambda, int nx, int px, int *cs, int *ct) {
  __shared__ float s_c[2 * kMaxK * 4];
  __shared__ float s_val[4][kLevels];
  __shared__ unsigned s_h[2 * kLevels], s_sum[2];
  if (S.ctl[0] == 0 || S.ctl[1] == 0 || S.ctl[2]) return;
  if (threadIdx.x < 2) s_sum[threadIdx.x] = 0;
  __syncthreads();
  if (LAZY) {
    for (int i = threadIdx.x; i < 2 * k * 4; i += blockDim.x) s_c[i] = S.cent[i];
    for (int c = 0; c < 4; ++c) s_val[c][threadIdx.x] = unorm8(threadIdx.x) * w.v[c];
  } else {
    for (int i = threadIdx.x; i < 2 * kLevels; i += blockDim.x) {
      s_h[i] = S.hist[i];
      if (s_h[i]) atomicAdd(&s_sum[i / kLevels], s_h[i]);
    }
  }
  __syncthreads();
  const unsigned sum_f = s_sum[0], sum_b = s_sum[1];
  const float gain = (float)(kMaxFlow >> shift) * lambda;
  for (unsigned v = blockIdx.x * blockDim.x + threadIdx.x; v < (unsigned)n;
       v += gridDim.x * blockDim.x) {
    int ef;
    if (fg[v]) {
      ef = kMaxFlow;
    } else if (bg[v]) {
      ef = -kMaxFlow;
    } else {
      unsigned t[4];
      texel(img, v, t);
      float val;
      if (LAZY) {
        float p[4];
        for (int c = 0; c < 4; ++c) p[c] = s_val[c][t[c]];
        float dx = 3.402823466e38f, dy = 3.402823466e38f;
        for (int j = 0; j < k; ++j) {
          dx = fminf(dx, dist4_sq(s_c + 4 * j, p));
          dy = fminf(dy, dist4_sq(s_c + 4 * (k + j), p));
        }
        dx = sqrtf(dx);
        dy = sqrtf(dy);
        const float r = (dx + dy == 0.0f) ? 0.0f : (dy - dx) / (dx + dy);
        val = gain * r;
      } else {
        float f[4];
        for (int c = 0; c < 4; ++c) f[c] = unorm8(t[c]);
        int lv = (int)(dot4(f, w) * (float)(kLevels - 1) + 0.5f);
        lv = lv < 0 ? 0 : (lv > kLevels - 1 ? kLevels - 1 : lv);
        const float qf = (float)s_h[lv] / (float)sum_f;
        const float qb = (float)s_h[kLevels + lv] / (float)sum_b;
        const float df = -(float)log((double)qf), db = -(float)log((double)qb);
        val = gain * (db - df);
      }
      ef = unary_int(val);
    }
    // the planes store row r at r * px
    const unsigned row = v / (unsigned)nx;
    const long long sv = (long long)row * px + (v - row * (unsigned)nx);
    cs[sv] = ef > 0 ? ef : 0;
    ct[sv] = ef < 0 ? -ef : 0;
  }
}

// convert_int4(read_imagef(.) * weight * SHRT_MAX): truncation toward zero
__device__ __forceinline__ void scaled_texel(const uchar4 *img, long long v, const W4 &w,
                                             int d[4]) {
  unsigned t[4];
  texel(img, v, t);
  for (int c = 0; c < 4; ++c) d[c] = (int)((unorm8(t[c]) * w.v[c]) * (float)SHRT_MAX);
}

// One arc of graphcut_compute_capacity_lazy / _bk: the squared distance in
// unsigned arithmetic, then top / (1 + dist) or top * exp(-t^2 / 2), + 0.5,
// truncated; top = SHRT_MAX in 2D, CHAR_MAX in 3D.
template <bool LAZY, bool D3>
__device__ __forceinline__ int wm_arc(const int a[4], const int b[4], float scale) {
  unsigned s = 0;
  for (int c = 0; c < 4; ++c) {
    const unsigned d = (unsigned)(a[c] > b[c] ? a[c] - b[c] : b[c] - a[c]);
    s += d * d;
  }
  const float top = D3 ? 127.0f : (float)SHRT_MAX;
  const float x = sqrtf((float)s) * scale;
  if (LAZY) return (int)(top / (1.0f + x) + 0.5f);
  const float e = (float)exp((double)((-0.5f * x) * x));
  return (int)(top * e + 0.5f);
}

// Planes of one instance; plane d of node v is the arc toward v + dir(d)
// (0 +x, 1 -x, 2 +y, 3 -y, 4 +z, 5 -z); border arcs are 0.  The reference's
// c1 / c2 pairs are the same values (c1 = (+x, +y[, +z]), c2 = (-y, -x) in 2D
// and (-z, -y, -x) in 3D).
template <bool LAZY, bool D3>
__global__ __launch_bounds__(256) void k_wm_pairwise(InstDesc I, const uchar4 *img, W4 w,
                                                     float scale, const int *ctl, int *c0,
                                                     long long stride) {
  if (ctl[0] == 0 || ctl[1] == 0) return;
  const long long rows = (long long)I.ny * I.nz;
  for (long long row = blockIdx.x; row < rows; row += gridDim.x) {
    const int y = (int)(row % I.ny), z = (int)(row / I.ny);
    for (int x = threadIdx.x; x < I.nx; x += blockDim.x) {
      const long long v = x + (long long)I.nx * row;
      int a[4];
      scaled_texel(img, v, w, a);
      for (int d = 0; d < (D3 ? 6 : 4); ++d) {
        int dx, dy, dz;
        dir_of<D3>(d, dx, dy, dz);
        const int X = x + dx, Y = y + dy, Z = z + dz;
        int cap = 0;
        if (X >= 0 && X < I.nx && Y >= 0 && Y < I.ny && Z >= 0 && Z < I.nz) {
          int b[4];
          scaled_texel(img, X + (long long)I.nx * (Y + (long long)I.ny * Z), w, b);
          cap = wm_arc<LAZY, D3>(a, b, scale);
        }
        c0[d * stride + I.node_off + x + (long long)I.px * row] = cap;
      }
    }
  }
}

int grid1(long long n) {
  long long g = (n + 255) / 256;
  return (int)(g < 1 ? 1 : (g > 8192 ? 8192 : g));
}

// glm::normalize(vec4): v * (1 / sqrt(dot(v, v))), dot as (xx + yy) + (zz + ww)
W4 normalize_weight(const float in[4]) {
  const float s = (in[0] * in[0] + in[1] * in[1]) + (in[2] * in[2] + in[3] * in[3]);
  const float inv = 1.0f / std::sqrt(s);
  W4 w;
  for (int c = 0; c < 4; ++c) w.v[c] = in[c] * inv;
  return w;
}

}  // namespace

#define WM_RET(call)                                                                    \
  do {                                                                                  \
    hipError_t e_ = (call);                                                             \
    if (e_ != hipSuccess)                                                               \
      return model_fail(JFC_ERR_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

// The k-means of the sides with more seeds than k_wm_lloyd takes, an
// assignment per launch and the update here; ctl and cent of `back` (the host
// copy of the scratch) and of the scratch are completed, the unary's guard
// lifted.
static int lloyd_on_host(const uchar4 *img, const W4 &w, int k, int iterations, int limit,
                         const WmScratch &S, unsigned char *back, hipStream_t st) {
  int *ctl = (int *)back;
  float *cent_used = (float *)(back + kCtlBytes + kHistBytes);
  // weighted feature value of each byte per channel: unorm8(b) * w
  float val[4][kLevels];
  for (int c = 0; c < 4; ++c)
    for (int b = 0; b < kLevels; ++b) val[c][b] = unorm8(b) * w.v[c];
  for (int side = 0; side < 2; ++side) {
    const int cnt = ctl[side];
    if (cnt <= limit) continue;
    // initial centroids: the representatives of the seeded levels, picked at
    // (count - 1) * i / (k - 1) (QGCW:2011-2039), scaled by weight / 255
    std::vector<unsigned> rep(kLevels);
    WM_RET(hipMemcpyAsync(rep.data(), S.rep + side * kLevels, kLevels * sizeof(unsigned),
                          hipMemcpyDeviceToHost, st));
    WM_RET(hipStreamSynchronize(st));
    std::vector<unsigned> dist;
    for (int l = 0; l < kLevels; ++l)
      if (rep[l]) dist.push_back(rep[l]);
    const unsigned dsize = (unsigned)dist.size() - 1u;
    float scale[4];
    for (int c = 0; c < 4; ++c) scale[c] = w.v[c] / 255.0f;
    std::vector<float> cent(k * 4), prev(k * 4);
    std::vector<uchar4> picked(k);
    for (int i = 0; i < k; ++i) {
      const long long idx = (long long)dist[dsize * (unsigned)i / (unsigned)(k - 1)] - 1;
      WM_RET(hipMemcpyAsync(&picked[i], img + idx, sizeof(uchar4), hipMemcpyDeviceToHost, st));
    }
    WM_RET(hipStreamSynchronize(st));
    for (int i = 0; i < k; ++i) {
      const uchar4 t = picked[i];
      const unsigned tb[4] = {t.x, t.y, t.z, t.w};
      for (int c = 0; c < 4; ++c) cent[i * 4 + c] = (float)tb[c] * scale[c];
    }
    // Lloyd iterations (QGCW:2073-2102): the centroids of the last
    // assignment are the ones the unary uses
    std::vector<unsigned> acc((size_t)k * 4 * kLevels);
    float *d_cent = S.cent + side * k * 4;
    int it = 0;
    while (it < iterations) {
      prev = cent;
      WM_RET(hipMemcpyAsync(d_cent, prev.data(), k * 4 * sizeof(float), hipMemcpyHostToDevice, st));
      launch_fill_i32((int *)S.acc, (long long)acc.size(), 0, st);
      k_wm_assign<<<std::min(grid1(cnt), 1024), 256, 0, st>>>(S.list[side], cnt, w, d_cent, k, S.acc);
      WM_RET(hipGetLastError());
      WM_RET(hipMemcpyAsync(acc.data(), S.acc, acc.size() * sizeof(unsigned), hipMemcpyDeviceToHost, st));
      WM_RET(hipStreamSynchronize(st));
      ++it;
      float err = 0.0f;
      for (int i = 0; i < k; ++i) {
        long long members = 0;
        for (int b = 0; b < kLevels; ++b) members += acc[(i * 4) * kLevels + b];
        for (int c = 0; c < 4; ++c) {
          if (!members) {
            cent[i * 4 + c] = 0.0f;
            continue;
          }
          double sum = 0.0;
          for (int b = 0; b < kLevels; ++b) {
            const unsigned m = acc[(i * 4 + c) * kLevels + b];
            if (m) sum += (double)m * (double)val[c][b];
          }
          cent[i * 4 + c] = (float)(sum / (double)members);
        }
        // glm::length(centroid - previous)
        float d[4];
        for (int c = 0; c < 4; ++c) d[c] = cent[i * 4 + c] - prev[i * 4 + c];
        const float len = std::sqrt((d[0] * d[0] + d[1] * d[1]) + (d[2] * d[2] + d[3] * d[3]));
        err = std::max(err, len);
      }
      if (err < 1.0f / 1024) break;
    }
    ctl[3 + side] = it;
    for (int i = 0; i < k * 4; ++i) cent_used[side * k * 4 + i] = prev[i];
  }
  ctl[2] = 0;
  WM_RET(hipMemcpyAsync(S.ctl, back, kBackBytes, hipMemcpyHostToDevice, st));
  return JFC_OK;
}

extern "C" void jfc_default_widget_model_params(jfc_widget_model_params *p) {
  if (!p) return;
  p->lazy = 1;
  p->weight[0] = 0.2126f;
  p->weight[1] = 0.7152f;
  p->weight[2] = 0.0722f;
  p->weight[3] = 0.0f;
  p->lazy_neighbor = 1.0f;
  p->lazy_terminal = 1.0f;
  p->bk_neighbor = 0.002f;
  p->bk_terminal = 0.0f;
  p->k = 8;
  p->kmeans_iterations = 32;
}

#define WM_HIP(call)                                                                  \
  do {                                                                                \
    hipError_t e_ = (call);                                                           \
    if (e_ != hipSuccess) {                                                           \
      rc = model_fail(JFC_ERR_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
      goto done;                                                                      \
    }                                                                                 \
  } while (0)

extern "C" int jfc_model_widget(jfc_graph *g, int inst, const uint8_t *rgba, const uint8_t *fg,
                                const uint8_t *bg, int on_device,
                                const jfc_widget_model_params *prm,
                                jfc_widget_model_stats *stats) {
  InstDesc I;
  int *cs = nullptr, *ct = nullptr, *c0 = nullptr;
  long long stride = 0;
  int rc = graph_instance(g, inst, &I, &cs, &ct, &c0, &stride);
  if (rc) return rc;
  if (!rgba || !fg || !bg || !prm) return model_fail(JFC_ERR_INVALID, "null argument");
  const bool d3 = I.conn == 6;
  if (!(I.conn == 4 || I.conn == 6))
    return model_fail(JFC_ERR_INVALID,
                      "the widget's data terms are 4-connected in 2D and 6-connected in 3D");
  if (prm->k < 2 || prm->k > kMaxK || prm->kmeans_iterations < 1 || prm->kmeans_iterations > 256)
    return model_fail(JFC_ERR_INVALID, "k must be 2..32 and kmeans_iterations 1..256");
  for (int c = 0; c < 4; ++c)
    if (!(prm->weight[c] >= 0.0f) || !std::isfinite(prm->weight[c]))
      return model_fail(JFC_ERR_INVALID, "weights must be finite and >= 0");
  if (!(prm->weight[0] + prm->weight[1] + prm->weight[2] + prm->weight[3] > 0.0f))
    return model_fail(JFC_ERR_INVALID, "at least one weight must be positive");
  if (prm->lazy ? !(prm->lazy_neighbor >= 0.0f && prm->lazy_terminal >= 0.0f &&
                    std::isfinite(prm->lazy_neighbor) && std::isfinite(prm->lazy_terminal))
                : !(prm->bk_neighbor > 0.0f && prm->bk_terminal >= 0.0f &&
                    std::isfinite(prm->bk_neighbor) && std::isfinite(prm->bk_terminal)))
    return model_fail(JFC_ERR_INVALID, "invalid lambda / sigma");
  const long long n = (long long)I.nx * I.ny * I.nz;
  if (n >= (1LL << 31) - 1) return model_fail(JFC_ERR_INVALID, "instance too large for the model path");

  // Everything runs on the graph's stream.  Host inputs cross in one copy
  // each through the graph's staging buffer; the small scratch (WmScratch) is the
  // graph's data-term block.
  const hipStream_t st = graph_stream(g);
  const W4 w = normalize_weight(prm->weight);
  const int k = prm->k;
  const uchar4 *img = reinterpret_cast<const uchar4 *>(rgba);
  const unsigned char *dfg = fg, *dbg = bg;
  WmScratch S{};
  // Seeds a side that k_wm_lloyd takes: none where a weight has no finite norm,
  // whose sums and movements (infinite, or no number) are the host's.
  int limit = std::min(kLloydSeeds, kLloydWork / k);
  for (int c = 0; c < 4; ++c)
    if (!std::isfinite(w.v[c])) limit = 0;
  bool written = false;
  jfc_widget_model_stats st_local;
  jfc_widget_model_stats &ST = stats ? *stats : st_local;
  unsigned char back[kBackBytes];
  const int *ctl = (const int *)back;
  memset(&ST, 0, sizeof(ST));

  if (!on_device) {
    void *stage = nullptr;
    if ((rc = graph_stage(g, (size_t)n * 6 + 256, &stage))) return rc;
    unsigned char *sp = (unsigned char *)stage;
    WM_HIP(hipMemcpyAsync(sp, rgba, n * sizeof(uchar4), hipMemcpyHostToDevice, st));
    WM_HIP(hipMemcpyAsync(sp + n * 4, fg, n, hipMemcpyHostToDevice, st));
    WM_HIP(hipMemcpyAsync(sp + n * 5, bg, n, hipMemcpyHostToDevice, st));
    img = reinterpret_cast<const uchar4 *>(sp);
    dfg = sp + n * 4;
    dbg = sp + n * 5;
  }
  {
    void *sc = nullptr;
    if ((rc = graph_scratch(g, kBackBytes + kRepBytes + kAccBytes + kOwnerBytes, &sc))) return rc;
    unsigned char *b = (unsigned char *)sc;
    S.ctl = (int *)b;
    S.hist = (unsigned *)(b + kCtlBytes);
    S.cent = (float *)(b + kCtlBytes + kHistBytes);
    S.rep = (unsigned *)(b + kBackBytes);
    S.acc = (unsigned *)(b + kBackBytes + kRepBytes);
    S.owner = b + kBackBytes + kRepBytes + kAccBytes;
    // the seed lists borrow the instance's slices of the excess and height
    // planes, which every solve rewrites before reading them
    int *l0 = nullptr, *l1 = nullptr;
    long long cap = 0;
    if ((rc = graph_work_plane(g, inst, &l0, &cap)) || (rc = graph_work_plane2(g, inst, &l1)))
      return rc;
    S.list[0] = (uchar4 *)l0;
    S.list[1] = (uchar4 *)l1;
  }
  {
    // everything is queued without a look at the counts: with a side without
    // seeds the kernels write no plane
    launch_fill_i32(S.ctl, (kBackBytes + kRepBytes) / 4, 0, st);
    k_wm_scan<<<std::min(grid1((n + 3) / 4), 1024), 256, 0, st>>>(img, dfg, dbg, n, w, S);
    if (prm->lazy) {
      W4 scale;
      for (int c = 0; c < 4; ++c) scale.v[c] = w.v[c] / 255.0f;
      const int iters = prm->kmeans_iterations;
      if (k <= 8) k_wm_lloyd<8><<<2, 1024, 0, st>>>(img, w, scale, k, iters, limit, S);
      else if (k <= 16) k_wm_lloyd<16><<<2, 1024, 0, st>>>(img, w, scale, k, iters, limit, S);
      else k_wm_lloyd<32><<<2, 1024, 0, st>>>(img, w, scale, k, iters, limit, S);
    }
    WM_HIP(hipGetLastError());
    const int shift = d3 ? 3 : 2;
    auto unary = [&]() {
      if (prm->lazy)
        k_wm_unary<true><<<grid1(n), 256, 0, st>>>(img, dfg, dbg, (int)n, w, S, k, shift,
                                                   prm->lazy_terminal, I.nx, I.px,
                                                   cs + I.node_off, ct + I.node_off);
      else
        k_wm_unary<false><<<grid1(n), 256, 0, st>>>(img, dfg, dbg, (int)n, w, S, 0, shift,
                                                    prm->bk_terminal, I.nx, I.px,
                                                    cs + I.node_off, ct + I.node_off);
    };
    unary();
    WM_HIP(hipGetLastError());
    const int grid = (int)std::min<long long>((long long)I.ny * I.nz, 65536);
    if (prm->lazy) {
      // lambda / SHRT_MAX (graphcut_compute_capacity.cl:82)
      const float scale = prm->lazy_neighbor / (float)SHRT_MAX;
      if (d3) k_wm_pairwise<true, true><<<grid, 256, 0, st>>>(I, img, w, scale, S.ctl, c0, stride);
      else k_wm_pairwise<true, false><<<grid, 256, 0, st>>>(I, img, w, scale, S.ctl, c0, stride);
    } else {
      // 1 / (SHRT_MAX * sigma) (graphcut_compute_capacity.cl:29)
      const float scale = 1.0f / ((float)SHRT_MAX * prm->bk_neighbor);
      if (d3) k_wm_pairwise<false, true><<<grid, 256, 0, st>>>(I, img, w, scale, S.ctl, c0, stride);
      else k_wm_pairwise<false, false><<<grid, 256, 0, st>>>(I, img, w, scale, S.ctl, c0, stride);
    }
    written = true;
    WM_HIP(hipGetLastError());
    WM_HIP(hipMemcpyAsync(back, S.ctl, kBackBytes, hipMemcpyDeviceToHost, st));
    WM_HIP(hipStreamSynchronize(st));
    for (int side = 0; side < 2; ++side) {
      ST.seeds[side] = ctl[side];
      if (ctl[side] == 0) {
        // computeBFS / kmeans "no labels." (QGCW:2015-2016); no plane was written
        written = false;
        rc = model_fail(JFC_ERR_NO_SEEDS, side ? "no background seeds" : "no foreground seeds");
        goto done;
      }
    }
    if (prm->lazy && ctl[2]) {
      if ((rc = lloyd_on_host(img, w, k, prm->kmeans_iterations, limit, S, back, st))) goto done;
      unary();
      WM_HIP(hipGetLastError());
      WM_HIP(hipStreamSynchronize(st));
    }
    const unsigned *hist = (const unsigned *)(back + kCtlBytes);
    const float *cent = (const float *)(back + kCtlBytes + kHistBytes);
    for (int side = 0; side < 2; ++side) {
      for (int l = 0; l < kLevels; ++l) ST.hist_sum[side] += hist[side * kLevels + l];
      if (!prm->lazy) continue;
      ST.iterations[side] = ctl[3 + side];
      for (int i = 0; i < k * 4; ++i) ST.centroids[side][i / 4][i % 4] = cent[side * k * 4 + i];
    }
    graph_mark_inputs(g, inst);
  }
done:
  if (rc && written) graph_inputs_failed(g, inst);
  return rc;
}
