// jfc_region.hip -- exact global relabel on bit-parallel regions.
//
// Reference counterpart: graphcut_global_relabel
// (src/QVisualizer/cl/GraphCut/graphcut_global_relabel.cl:50-124, :128-249)
// and its back-and-forth tile passes (QGCWidget.cpp:2221-2240).
//
// A region is 4096 nodes owned by one wavefront: 64 x 64 in 2D, 64 x 8 x 8 in
// 3D.  Lane r holds row r of the region as 64-bit words, bit x = column x: one
// word per direction with the nodes whose residual arc in that direction is
// open, one with the deficit nodes.  A breadth-first level of the whole region
// is then a handful of shifts and ANDs per direction in registers -- the
// neighbours in x are the word shifted by one, those in y and z the
// neighbouring lanes' words -- instead of one LDS read per node, direction and
// iteration.
//
// Why regions of this size and shape: a relabel front crosses at least one
// region per pass, and a pass costs its launch and the load latency of a visit
// whatever the region holds, so the pass count decides long searches.  Rows of
// 64 nodes are whole 256-byte lines of every plane, and a 64-bit word is the
// ballot of a wavefront, so planes are packed with one ballot per row and
// direction.
//
// Passes exchange distances over the regions' borders only (an array of the
// border nodes' distances per region, contiguous):
//   kPack     every region: masks and excess signs packed into bit planes
//             (kept for the later passes, 1 bit per direction and node),
//             searched from its own deficits and the borders already written;
//   kBorders  regions whose neighbours' borders fell: searched again, borders
//             updated, neighbours marked;
//   kFinal    every region, once no region is marked: the heights written,
//             with the push tiles' active flags.
// A region's distances are kept as counting planes too (distance minus the
// region's base, bit-sliced), so a later visit resumes at the smallest border
// distance that improves a border node: nodes nearer than that are settled, the
// others are searched again from there.  A visit where none improves ends
// before its search.  No height word is touched before kFinal.
//
// What bounds it, and what it measured.  Long searches are a chain of visits: on
// the 3750x2500 8-connected cut from strokes alone a relabel of 55-73 passes takes
// 1.05 ms in one launch (settle) and 1.6 with a launch per pass; tiles of 32x8
// relaxed node by node in LDS took ~300 passes, 9 ms.  A level costs ~50 vector
// instructions for 4096 nodes; written as one loop with every counting plane
// per level it cost 85.  The first and last step over every region are bound by
// memory and packing: on the 512^3 volume kPack takes 425 us (8 bytes per node
// read: 226 us at the rate of a large copy), kFinal 156 us (134 us).  A relabel
// there takes 1.65 ms in one launch, 1.78 by passes (1.8 on 8x8x4 tiles), of the
// 2560x1440x50 video volume 1.8-2.0 and 2.5-3.0 (2.9-3.0).
#include "jfc_rows.h"

#include <algorithm>
#include <type_traits>

namespace jfc {

namespace {

// Border array of a region: columns x = 0 and x = 63 by row, then the border
// rows by x.
constexpr int kLeft = 0, kRight = 64, kRows = 128;

// The search runs in blocks of kBlock levels, unrolled: the low bits of a
// level's count are then constants, and the high ones are added once per
// block.  The border distances that fall into a block are kept as bits, one
// 64-bit word per level and row; a level's 64 words are padded by one so that
// lanes with different levels fall on different LDS banks.
constexpr int kBlock = 16, kWinPitch = 130;
// distances relative to the epoch's base are counted in this many bit planes
constexpr int kCntBits = 12, kCntMax = 1 << kCntBits;
// planes of a region after its directions': deficits, excess, visited, counts
constexpr int kStatePlanes = 3 + kCntBits;
// a region's base when its distances span more than kCntMax (kept by none of
// the planes: its visits search from scratch)
constexpr int kNoBase = -1;

__device__ __forceinline__ unsigned wave_or(unsigned v) {
  v |= __builtin_amdgcn_update_dpp(0u, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v |= __builtin_amdgcn_update_dpp(0u, v, 0x112, 0xf, 0xf, false);
  v |= __builtin_amdgcn_update_dpp(0u, v, 0x114, 0xf, 0xf, false);
  v |= __builtin_amdgcn_update_dpp(0u, v, 0x118, 0xf, 0xf, false);
  v |= __builtin_amdgcn_update_dpp(0u, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v |= __builtin_amdgcn_update_dpp(0u, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return __builtin_amdgcn_readlane(v, 63);
}
// minimum over the wave, uniform
__device__ __forceinline__ int wave_min(int v) {
  v = min(v, __builtin_amdgcn_update_dpp(HINF, v, 0x111, 0xf, 0xf, false));  // row_shr:1
  v = min(v, __builtin_amdgcn_update_dpp(HINF, v, 0x112, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(HINF, v, 0x114, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(HINF, v, 0x118, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(HINF, v, 0x142, 0xa, 0xf, false));  // row_bcast:15
  v = min(v, __builtin_amdgcn_update_dpp(HINF, v, 0x143, 0xc, 0xf, false));  // row_bcast:31
  return __builtin_amdgcn_readlane(v, 63);
}

__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Border words carry the tag of the relabel that wrote them; a word of an
// earlier relabel reads as unreached.  kPack writes every word of every
// region, so a word can only carry this tag or the one before it.
__device__ __forceinline__ int border_word(const int *p) {
  // device-coherent: a neighbour searched earlier in the same pass, possibly
  // on another XCD, is seen at once.  Every value read is a bound from above.
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// a region's own word, written by its visits of earlier passes only
__device__ __forceinline__ int own_word(const int *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int border_dist(int w, int tag) {
  return (int)((unsigned)w >> 30) == tag ? w & HINF : HINF;
}
__device__ __forceinline__ void border_store(int *p, int v, int tag) {
  __hip_atomic_store(p, (int)((unsigned)v | (unsigned)tag << 30), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

// Visits region t.  W: waves of the workgroup that share a region's packing
// and its heights, 64 / W rows each; the search is the first wave's alone.
template <bool D3, int PASS, bool ONE, int W>
__device__ __forceinline__ void region_visit(const Tiles &T, const Planes &P,
                                             const RegionBuf &R, const RegionPass &A, int t,
                                             unsigned *inj, Marks &marks) {
  using G = Reg<D3>;
  constexpr int KM = G::K, NV = G::NV;
  constexpr int BN = kRows + 64 * NV;
  const int lane = threadIdx.x & 63;
  const int wv0 = W > 1 ? 64 / W * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;  // first row
  const InstDesc &I = ONE ? T.one : T.inst[T.tile_inst[t]];
  const int K = I.K;
  const RegionRef r = region_ref<D3>(I, t, lane);
  const int ox = r.ox, oy = r.oy, oz = r.oz, wx = r.wx;
  const int ly = D3 ? lane & 7 : lane, lz = D3 ? lane >> 3 : 0;
  const u64 valid = r.valid;

  // ---- bit planes: open arcs per direction, deficits, excess
  u64 M[KM], D = 0, X = 0;
  u64 *pk = R.packed + (long long)t * R.planes * 64 + lane;
  u64 *ps = pk + 64 * (R.planes - kStatePlanes);  // deficits, excess, visited, counts
  u64 vis = ~valid, cnt[kCntBits];  // visited (off-grid nodes count); distance - ebase
  int ebase = kNoBase;  // block 0's first level
#pragma unroll
  for (int j = 0; j < kCntBits; ++j) cnt[j] = 0;
  if (PASS != kPack) ebase = R.base[t];
  auto load_state = [&]() {
    vis = ps[128];
#pragma unroll
    for (int j = 0; j < kCntBits; ++j) cnt[j] = ps[64 * (3 + j)];
  };
  // distance of row r's nodes by lane, from the `planes` lowest counts
  auto row_dist = [&](int r, int top) {
    int v = 0;
    if (top > 256) {
#pragma unroll
      for (int j = kCntBits - 1; j >= 8; --j) v = v + v + (bit_of_lane(row_word(cnt[j], r)) ? 1 : 0);
    }
    if (top > 16) {
#pragma unroll
      for (int j = 7; j >= 4; --j) v = v + v + (bit_of_lane(row_word(cnt[j], r)) ? 1 : 0);
    }
#pragma unroll
    for (int j = 3; j >= 0; --j) v = v + v + (bit_of_lane(row_word(cnt[j], r)) ? 1 : 0);
    return v + ebase;
  };
  // the heights of the nodes in `found` and, with `rest`, of the nodes not
  // visited at all (unreachable)
  auto write_heights = [&](u64 found, u64 rest, int top, int begin, int end) {
    for (int r0 = begin; r0 < end; r0 += 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int r = r0 + u;
        const int y = oy + (D3 ? u : r), z = D3 ? oz + (r0 >> 3) : 0;
        if (y >= I.ny || z >= I.nz) continue;
        const bool hit = bit_of_lane(row_word(found, r));
        const int d = row_dist(r, top);
        if (hit || bit_of_lane(row_word(rest, r))) P.h[node_index(I, ox + lane, y, z)] = hit ? d : HINF;
      }
    }
  };
  // the active flags of the push tiles: nodes with excess and a finite height
  auto write_active = [&](u64 excess) {
    const u64 act = excess & vis & valid;
    if (!act) return;
    const InstDesc &PI = ONE ? A.pone : A.pinst[T.tile_inst[t]];
    const int lw = A.pdims & 15;
    const int row = PI.tile_off + PI.tx * (((oy + ly) >> ((A.pdims >> 4) & 15)) +
                                           PI.ty * ((oz + lz) >> (A.pdims >> 8)));
    const u64 seg = lw == 6 ? ~0ull : (1ull << (1 << lw)) - 1;
    for (int x = 0; x < 64; x += 1 << lw)
      if ((act >> x) & seg) A.active[row + ((ox + x) >> lw)] = 1;
  };
  // the largest distance among `found`: the highest count bit that any of them
  // has, then the next among those that have it
  auto note_farthest = [&](u64 found, int top) {
    if (!__ballot(found != 0)) return;
    int d = 0;
#pragma unroll
    for (int j = kCntBits - 1; j >= 0; --j) {
      if ((1 << j) >= top) continue;
      const u64 t = found & cnt[j];
      if (__ballot(t != 0)) d |= 1 << j, found = t;
    }
    if (lane == 0) atomicMax(A.far + kFarLine * (t & (kFarSlots - 1)), ebase + d);
  };
  // 2D visits load their state with everything else; a 3D visit's borders are
  // as large as its planes, and half of them end before the search, so it
  // loads its state after they are compared
  constexpr bool kEarlyState = !D3;
  if (PASS == kBorders && kEarlyState) load_state(), D = ps[0];
  if (PASS == kFinal && ebase != kNoBase) {
    load_state();
    const u64 high = cnt[8] | cnt[9] | cnt[10] | cnt[11], mid = cnt[4] | cnt[5] | cnt[6] | cnt[7];
    const int top = __ballot(high != 0) ? kCntMax : __ballot(mid != 0) ? 256 : 16;
    write_heights(vis & valid, valid & ~vis, top, wv0, wv0 + 64 / W);
    if (wv0 == 0) write_active(ps[64]), note_farthest(vis & valid, top);
    return;
  }
  if (PASS == kFinal && wv0 > 0) return;

  if (PASS == kPack) {
    int mlo[KM], mhi[KM], dlo = 0, dhi = 0, xlo = 0, xhi = 0;
#pragma unroll
    for (int d = 0; d < KM; ++d) mlo[d] = mhi[d] = 0;
    // the next RB rows' loads are in flight while RB rows are packed; rows and
    // columns off the grid read a valid dummy address
    constexpr int RB = 16;
    unsigned w[2][RB];
    int e[2][RB];
    auto row_in = [&](int r) {
      return oy + (D3 ? r & 7 : r) < I.ny && oz + (D3 ? r >> 3 : 0) < I.nz && lane < wx;
    };
    auto load = [&](unsigned *wb, int *eb, int r0) {
#pragma unroll
      for (int u = 0; u < RB; ++u) {
        const int r = r0 + u;
        const long long v =
            row_in(r) ? node_index(I, ox + lane, oy + (D3 ? r & 7 : r), oz + (D3 ? r >> 3 : 0)) : 0;
        wb[u] = P.rmask[v];
        eb[u] = P.e[v];
      }
    };
    load(w[0], e[0], wv0);
#pragma unroll
    for (int b = 0; b < 64 / RB / W; ++b) {
      if (b + 1 < 64 / RB / W) load(w[(b + 1) & 1], e[(b + 1) & 1], RB * (b + 1));
#pragma unroll
      for (int u = 0; u < RB; ++u) {
        const int r = wv0 + RB * b + u;
        const unsigned m = row_in(r) ? w[b & 1][u] : 0u;
        const int ee = row_in(r) ? e[b & 1][u] : 0;
#pragma unroll
        for (int d = 0; d < KM; ++d)
          if (D3 || d < 4 || K == 8) set_row(mlo[d], mhi[d], r, __ballot(m & (1u << d)));
        set_row(dlo, dhi, r, __ballot(ee < 0));
        set_row(xlo, xhi, r, __ballot(ee > 0));
      }
    }
#pragma unroll
    for (int d = 0; d < KM; ++d) M[d] = (u64)(unsigned)mhi[d] << 32 | (unsigned)mlo[d];
    D = (u64)(unsigned)dhi << 32 | (unsigned)dlo;
    X = (u64)(unsigned)xhi << 32 | (unsigned)xlo;
    if constexpr (W > 1) {
      // the waves' rows gathered by the first wave
      __shared__ u64 s_rows[KM + 2][64];
      if ((unsigned)(lane - wv0) < 64u / W) {
#pragma unroll
        for (int d = 0; d < KM; ++d) s_rows[d][lane] = M[d];
        s_rows[KM][lane] = D;
        s_rows[KM + 1][lane] = X;
      }
      __syncthreads();
      if (wv0 > 0) return;
#pragma unroll
      for (int d = 0; d < KM; ++d) M[d] = s_rows[d][lane];
      D = s_rows[KM][lane];
      X = s_rows[KM + 1][lane];
    }
#pragma unroll
    for (int d = 0; d < KM; ++d)
      if (d < K) pk[64 * d] = M[d];
    ps[0] = D;
    ps[64] = X;
  } else {
#pragma unroll
    for (int d = 0; d < KM; ++d) M[d] = pk[64 * min(d, K - 1)];
    if (PASS == kFinal) D = ps[0], X = ps[64];
#pragma unroll
    for (int d = 0; d < KM; ++d)
      if (d >= K) M[d] = 0;
  }

  // ---- distances of the border nodes through the neighbours' borders
  const bool hasl = r.hasl, hasr = r.hasr, hasd = r.hasd, hasu = r.hasu;
  const bool diag = !D3 && K == 8;
  const long long b0 = (long long)t * BN;
  const long long by = (long long)r.sy * BN, bz = (long long)r.sz * BN;
  // every word is loaded before any is used; a missing neighbour's is the
  // region's own, and discarded
  auto word = [&](bool have, long long off, int idx) {
    return border_word(R.border + b0 + (have ? off : 0) + idx);
  };
  auto dist = [&](bool have, int w) { return have ? border_dist(w, A.tag) : HINF; };
  int sl, sr, sv[NV];     // left and right column by row, border rows by x
  int lo = HINF;          // the smallest that improves a border node
  {
    const int wl = word(hasl, -BN, kRight + lane), wr = word(hasr, BN, kLeft + lane);
    int wc[4], wv[NV];
    const bool hc[4] = {hasl && hasd, hasl && hasu, hasr && hasd, hasr && hasu};
    if constexpr (!D3) {
      wc[0] = word(hc[0], -BN - by, kRight + 63);
      wc[1] = word(hc[1], -BN + by, kRight);
      wc[2] = word(hc[2], BN - by, kLeft + 63);
      wc[3] = word(hc[3], BN + by, kLeft);
    }
    const bool has[4] = {hasd, hasu, r.hasf, r.hasb};
    const long long off[4] = {-by, by, -bz, bz};
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int f = D3 ? j >> 3 : j;
      wv[j] = word(has[f], off[f], kRows + 64 * (D3 ? j ^ 8 : j ^ 1) + lane);
    }
    int ow[NV + 2];  // the region's own words so far
    if (PASS == kBorders) {
      const int *bw = R.border + b0;
      ow[NV] = own_word(bw + kLeft + lane);
      ow[NV + 1] = own_word(bw + kRight + lane);
#pragma unroll
      for (int j = 0; j < NV; ++j) ow[j] = own_word(bw + kRows + 64 * j + lane);
    }
    const int hl = dist(hasl, wl), hr = dist(hasr, wr);
    sl = M[1] & 1 ? hl : HINF;
    sr = M[0] >> 63 ? hr : HINF;
    if (diag) {
      int q = __shfl_up(hl, 1);
      if (lane == 0) q = dist(hc[0], wc[0]);
      if (M[5] & 1) sl = min(sl, q);
      q = __shfl_down(hl, 1);
      if (lane == 63) q = dist(hc[1], wc[1]);
      if (M[6] & 1) sl = min(sl, q);
      q = __shfl_up(hr, 1);
      if (lane == 0) q = dist(hc[2], wc[2]);
      if (M[7] >> 63) sr = min(sr, q);
      q = __shfl_down(hr, 1);
      if (lane == 63) q = dist(hc[3], wc[3]);
      if (M[4] >> 63) sr = min(sr, q);
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int h = dist(has[D3 ? j >> 3 : j], wv[j]);
      wv[j] = h;
      sv[j] = bit_of_lane(row_word(M[G::dir(j)], G::row(j))) ? h : HINF;
    }
    if constexpr (!D3) {
      if (diag) {
        int q = __shfl_up(wv[0], 1);
        if (lane > 0 && bit_of_lane(row_word(M[5], 0))) sv[0] = min(sv[0], q);
        q = __shfl_down(wv[0], 1);
        if (lane < 63 && bit_of_lane(row_word(M[7], 0))) sv[0] = min(sv[0], q);
        q = __shfl_down(wv[1], 1);
        if (lane < 63 && bit_of_lane(row_word(M[4], 63))) sv[1] = min(sv[1], q);
        q = __shfl_up(wv[1], 1);
        if (lane > 0 && bit_of_lane(row_word(M[6], 63))) sv[1] = min(sv[1], q);
      }
    } else {
      // arcs through the faces have done their part; what is left stays
      // inside the region, so the lane shifts below need no edge tests
      if (ly == 7) M[2] = 0;
      if (ly == 0) M[3] = 0;
      if (lz == 7) M[4] = 0;
      if (lz == 0) M[5] = 0;
    }
    auto enter = [&](int &v, int k) {
      v = min(v + 1, HINF);
      lo = min(lo, PASS != kBorders || v < border_dist(ow[k], A.tag) ? v : HINF);
    };
    enter(sl, NV);
    enter(sr, NV + 1);
#pragma unroll
    for (int j = 0; j < NV; ++j) enter(sv[j], j);
    lo = wave_min(lo);
  }

  // ---- breadth-first search, level by level
  // Border distances enter through the block's bits.  fill() sets the bits of
  // the block from `base` on, the levels that have any (levels), and the
  // smallest distance beyond the block (beyond).
  unsigned levels = 0;
  int beyond = HINF;
  auto fill = [&](int base) {
    unsigned lv = 0;
    int far = HINF;
    auto put = [&](int v, int row, int half, unsigned bit) {
      const unsigned l = (unsigned)(v - base);
      if (l < (unsigned)kBlock) {
        atomicOr(&inj[l * kWinPitch + 2 * row + half], bit);
        lv |= 1u << l;
      } else if (v > base) {
        far = min(far, v);
      }
    };
    put(sl, lane, 0, 1u);
    put(sr, lane, 1, 1u << 31);
#pragma unroll
    for (int j = 0; j < NV; ++j) put(sv[j], G::row(j), lane >> 5, 1u << (lane & 31));
    lds_order();
    beyond = wave_min(far);
    levels = wave_or(lv);
  };
  const int addr_up = ((lane + 8) & 63) * 4, addr_dn = ((lane - 8) & 63) * 4;
  auto expand = [&](u64 f) {
    u64 up8 = 0, dn8 = 0;
    if constexpr (D3) up8 = from_lane(f, addr_up), dn8 = from_lane(f, addr_dn);
    u64 n = (M[0] & shr1(f)) | (M[1] & shl1(f));
    const u64 up = from_next(f), dn = from_prev(f);
    n |= (M[2] & up) | (M[3] & dn);
    if constexpr (D3) n |= (M[4] & up8) | (M[5] & dn8);
    else if (diag)
      n |= (M[4] & shr1(up)) | (M[5] & shl1(dn)) | (M[6] & shl1(up)) | (M[7] & shr1(dn));
    return n;
  };

  // Where the search starts.  From scratch: the region's deficits, or the
  // smallest border distance.  Resumed (kBorders): the block holding the
  // smallest border distance that improves a border node, with the nodes
  // nearer than the block settled and those at the level before it as the
  // frontier.
  int L = 0;  // first level of the block
  u64 nw = 0;
  bool scratch = true;
  if (PASS == kBorders) {
    if (lo >= HINF && ebase != kNoBase) return;
    if (!kEarlyState) load_state(), D = ps[0];
  }
  if (PASS == kBorders && ebase != kNoBase) {
    L = lo;
    scratch = ebase < HINF && L - ebase >= kCntMax;
    if (!scratch) {
      if (L <= ebase) {
        vis = ~valid;
        ebase = L;
#pragma unroll
        for (int j = 0; j < kCntBits; ++j) cnt[j] = 0;
      } else {
        const int r0 = (L - ebase) & -kBlock, r1 = r0 - 1;
        L = ebase + r0;
        u64 lt = 0, eq = vis & valid;
#pragma unroll
        for (int j = 0; j < kCntBits; ++j) {
          lt = (r0 >> j) & 1 ? lt | ~cnt[j] : lt & ~cnt[j];
          eq &= (r1 >> j) & 1 ? cnt[j] : ~cnt[j];
        }
        vis = (vis & valid & lt) | ~valid;
        nw = r0 ? expand(eq) & ~vis : D;  // block 0 starts from the deficits
#pragma unroll
        for (int j = 0; j < kCntBits; ++j) cnt[j] &= vis;
      }
    }
  }
  if (scratch) {
    if (PASS == kBorders) {
      lo = min(sl, sr);
#pragma unroll
      for (int j = 0; j < NV; ++j) lo = min(lo, sv[j]);
      lo = wave_min(lo);
    }
    L = __ballot(D != 0) ? 0 : lo;
    vis = ~valid;
    ebase = L;
    nw = D;
#pragma unroll
    for (int j = 0; j < kCntBits; ++j) cnt[j] = 0;
  }
  u64 vis0 = vis;  // visited when the epoch began
  bool wrote = false;

  int top = 0;  // the largest count of the epoch is below this
  // The nodes found in the epoch: their border words (kPack, kBorders) or
  // heights (kFinal).  The first flush of kPack writes every border word, the
  // last of kFinal every height that is left.
  auto flush = [&](bool last) {
    const u64 found = vis & ~vis0;
    if (PASS == kFinal) {
      write_heights(found, last ? valid & ~vis : 0, top, 0, 64);
      note_farthest(found, kCntMax);
    } else {
      int *bw = R.border + b0;
      const bool all = PASS == kPack && !wrote;
      int ow[NV + 2];
      if (PASS == kBorders) {
        ow[NV] = own_word(bw + kLeft + lane);
        ow[NV + 1] = own_word(bw + kRight + lane);
#pragma unroll
        for (int j = 0; j < NV; ++j) ow[j] = own_word(bw + kRows + 64 * j + lane);
      }
      auto update = [&](int idx, int old, bool hit, int d) -> u64 {
        const int v = hit ? d : HINF;
        const bool ch = hit && (PASS == kPack || v < border_dist(old, A.tag));
        if (ch || all) border_store(bw + idx, v, A.tag);
        return __ballot(ch);
      };
      auto col_dist = [&](int s) {
        int v = 0;
#pragma unroll
        for (int j = kCntBits - 1; j >= 0; --j) v = v + v + (int)((cnt[j] >> s) & 1);
        return v + ebase;
      };
      const u64 cl = update(kLeft + lane, ow[NV], found & 1, col_dist(0));
      const u64 cr = update(kRight + lane, ow[NV + 1], found >> 63, col_dist(63));
      u64 face[D3 ? 4 : 2];
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const int r = G::row(j);
        const u64 c =
            update(kRows + 64 * j + lane, ow[j], bit_of_lane(row_word(found, r)), row_dist(r, top));
        const int f = D3 ? j >> 3 : j;
        if (!D3 || (j & 7) == 0) face[f] = c;
        else face[f] |= c;
      }
      marks.add(0, hasl && cl);
      marks.add(1, hasr && cr);
      marks.add(2, hasd && face[0]);
      marks.add(3, hasu && face[1]);
      if constexpr (D3) {
        marks.add(4, r.hasf && face[2]);
        marks.add(5, r.hasb && face[3]);
      } else if (diag) {
        marks.add(4, hasl && hasd && (cl & 1));
        marks.add(5, hasl && hasu && cl >> 63);
        marks.add(6, hasr && hasd && (cr & 1));
        marks.add(7, hasr && hasu && cr >> 63);
      }
      marks.at = t + neighbour_step<D3>(r, lane);
    }
  };

  if (L < HINF) fill(L);
  // An epoch ends when its distances no longer fit the counting planes.
  for (bool done = L >= HINF;;) {
    while (!done) {
      const u64 before = vis;
      bool live = true;
#pragma unroll
      for (int i = 0; i < kBlock; ++i) {
        if ((levels >> i) & 1u) {
          u64 *word = (u64 *)&inj[i * kWinPitch + 2 * lane];
          nw |= *word & ~vis;
          *word = 0;  // every bit is taken by the end of its block
        }
        vis |= nw;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if ((i >> j) & 1) cnt[j] |= nw;
        nw = expand(nw) & ~vis;
        live = __ballot(nw != 0) != 0;
        if (!live && (levels >> i) <= 1u) break;
      }
      const u64 found = vis & ~before;
      const int rel = L - ebase;
      top = rel + kBlock;
      auto count = [&](int j) { cnt[j] |= found & (u64)(long long)-((rel >> j) & 1); };
      if (rel >= 16) {
#pragma unroll
        for (int j = 4; j < 8; ++j) count(j);
        if (rel >= 256) {
#pragma unroll
          for (int j = 8; j < kCntBits; ++j) count(j);
        }
      }
      L += kBlock;
      if (!live) {
        // only border distances are left, if any, and nodes to reach
        done = beyond >= HINF || !__ballot(~vis != 0);
        if (done) break;
        L = ebase + ((beyond - ebase) & -kBlock);
      }
      lds_order();
      levels = 0;
      if (beyond < L + kBlock) fill(L);
      if (L - ebase >= kCntMax) break;
    }
    flush(done);
    if (done) break;
    wrote = true;
    vis0 = vis;
    ebase = L;
#pragma unroll
    for (int j = 0; j < kCntBits; ++j) cnt[j] = 0;
  }
  lds_order();
  if (PASS == kFinal) {
    write_active(X);
  } else {
    if (!wrote) {
      ps[128] = vis;
#pragma unroll
      for (int j = 0; j < kCntBits; ++j) ps[64 * (3 + j)] = cnt[j];
    }
    if (lane == 0) R.base[t] = wrote ? kNoBase : ebase;
  }
}

// One pass.  With A.w.sums, kPack and kFinal are the first and last step around
// k_settle: kPack counts its marks for it, kFinal runs if it finished.
template <bool D3, int PASS, bool ONE, int W>
__global__ __launch_bounds__(64 * W) void k_region(Tiles T, Planes P, RegionBuf R, RegionPass A) {
  __shared__ __attribute__((aligned(8))) unsigned inj[kBlock * kWinPitch];
  const int lane = threadIdx.x & 63;
  bool marked = false;
  auto visit = [&](int t, auto w) {
    Marks marks;
    region_visit<D3, PASS, ONE, decltype(w)::value>(T, P, R, A, t, inj, marks);
    if (PASS == kPack && A.w.sums) {
      if (threadIdx.x < 64) publish(A.w, marks, 0, lane);
      return;
    }
    if (marks.on(lane)) A.c.dirty_out[marks.at] = 1;
    marked |= marks.set != 0;
  };
  if (PASS == kFinal && A.w.sums && shared_word(A.w.state) != kDone) return;
  if (PASS == kBorders) {
    // some region was marked for this pass; the host learns it from here
    const int work = *A.c.any_in;
    if (blockIdx.x == 0 && lane == 0) {
      *A.c.any_clear = 0;
      __hip_atomic_store(A.c.post, A.c.seq * 2 + (work != 0), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (!work) return;
  }
  if (threadIdx.x < 64) {
    for (int l = 0; l < kBlock; ++l) *(u64 *)&inj[l * kWinPitch + 2 * lane] = 0;
    lds_order();
  }
  if (PASS != kBorders) {
    visit(blockIdx.x, std::integral_constant<int, W>());
  } else {
    // a wave looks at 64 regions' marks at once, strided by the grid so that
    // a front's neighbouring regions go to different waves
    int visits = 0;
    const int G = gridDim.x;
    for (int base = blockIdx.x; base < T.ntiles; base += 64 * G) {
      const long long mine = base + (long long)lane * G;
      const bool f = mine < T.ntiles && A.c.dirty_in[mine];
      if (f) A.c.dirty_in[mine] = 0;
      u64 m = __ballot(f);
      visits += __popcll(m);
      while (m) {
        const int i = __builtin_ctzll(m);
        m &= m - 1;
        visit(base + i * G, std::integral_constant<int, 1>());
      }
    }
    if (visits && lane == 0)
      atomicAdd((u64 *)&A.c.visits[blockIdx.x & 63], (u64)visits);
  }
  if (PASS != kFinal && marked && threadIdx.x == 0) *A.c.any_out = 1;
}

// The passes between kPack and kFinal in one launch (settle).  W = 4 (one
// region per workgroup): kPack and kFinal too, whose rows the workgroup's other
// waves share.  A pass costs its slowest visit, its launch and, every few
// passes, the host's check; here a front moves on as soon as one region is
// searched.
template <bool D3, bool ONE, int W>
__global__ __launch_bounds__(64 * W) void k_settle(Tiles T, Planes P, RegionBuf R, RegionPass A) {
  __shared__ __attribute__((aligned(8))) unsigned inj[kBlock * kWinPitch];
  __shared__ int s_done;
  constexpr bool kAll = W > 1;
  const int lane = threadIdx.x & 63;
  begin(A.w);
  if (threadIdx.x < 64) {
    for (int l = 0; l < kBlock; ++l) *(u64 *)&inj[l * kWinPitch + 2 * lane] = 0;
    lds_order();
  }
  if (kAll) {
    Marks marks;
    region_visit<D3, kPack, ONE, W>(T, P, R, A, blockIdx.x, inj, marks);
    // served: the packing, which counts as a mark made before the launch
    if (threadIdx.x < 64) publish(A.w, marks, 1, lane);
  }
  bool done = false;
  if (threadIdx.x < 64)
    done = settle(A.w, T.ntiles, kAll, A.c.visits, [&](int t, int served) {
      Marks marks;
      region_visit<D3, kBorders, ONE, 1>(T, P, R, A, t, inj, marks);
      publish(A.w, marks, served, lane);
      return false;
    });
  if constexpr (!kAll) return;
  if (threadIdx.x == 0) s_done = done;
  __syncthreads();
  if (!s_done) return;
  Marks marks;
  region_visit<D3, kFinal, ONE, W>(T, P, R, A, blockIdx.x, inj, marks);
}

template <bool D3, bool ONE>
void launch(const Tiles &T, const Planes &P, const RegionBuf &R, const RegionPass &A, int pass,
            int nwg, hipStream_t st) {
  const int n = T.ntiles;
  const bool shared = n <= kSharedRegions;
  if (pass == kBorders) {
    k_region<D3, kBorders, ONE, 1><<<std::min(n, nwg), 64, 0, st>>>(T, P, R, A);
  } else if (pass == kPack) {
    if (shared) k_region<D3, kPack, ONE, 4><<<n, 256, 0, st>>>(T, P, R, A);
    else k_region<D3, kPack, ONE, 1><<<n, 64, 0, st>>>(T, P, R, A);
  } else {
    if (shared) k_region<D3, kFinal, ONE, 4><<<n, 256, 0, st>>>(T, P, R, A);
    else k_region<D3, kFinal, ONE, 1><<<n, 64, 0, st>>>(T, P, R, A);
  }
}

// A workgroup of k_settle looks after at most 64 regions (W = 4: after one).
template <bool D3, bool ONE>
bool launch_all(const Tiles &T, const Planes &P, const RegionBuf &R, const RegionPass &A,
                hipStream_t st) {
  const int n = T.ntiles;
  if (n <= kSharedRegions && resident_grid_b<&k_settle<D3, ONE, 4>, 256>(n) == n) {
    k_settle<D3, ONE, 4><<<n, 256, 0, st>>>(T, P, R, A);
    return true;
  }
  const int grid = resident_grid_b<&k_settle<D3, ONE, 1>, 64>(n);
  if (64LL * grid < n) return false;
  launch<D3, ONE>(T, P, R, A, kPack, 0, st);
  k_settle<D3, ONE, 1><<<grid, 64, 0, st>>>(T, P, R, A);
  launch<D3, ONE>(T, P, R, A, kFinal, 0, st);
  return true;
}

}  // namespace

bool launch_relabel(bool d3, const Tiles &T, const Planes &P, const RegionBuf &R,
                    const RegionPass &A, hipStream_t st) {
  if (d3) return T.ninst == 1 ? launch_all<true, true>(T, P, R, A, st) : launch_all<true, false>(T, P, R, A, st);
  return T.ninst == 1 ? launch_all<false, true>(T, P, R, A, st) : launch_all<false, false>(T, P, R, A, st);
}

int region_state_planes() { return kStatePlanes; }

int region_border_words(bool d3) { return d3 ? kRows + 64 * Reg<true>::NV : kRows + 64 * Reg<false>::NV; }

void region_dims(bool d3, int *tw, int *th, int *td) {
  *tw = 64;
  *th = d3 ? Reg<true>::TH : Reg<false>::TH;
  *td = d3 ? Reg<true>::TD : Reg<false>::TD;
}

void launch_region(bool d3, const Tiles &T, const Planes &P, const RegionBuf &R,
                   const RegionPass &A, int pass, int nwg, hipStream_t st) {
  if (d3) {
    if (T.ninst == 1) launch<true, true>(T, P, R, A, pass, nwg, st);
    else launch<true, false>(T, P, R, A, pass, nwg, st);
  } else {
    if (T.ninst == 1) launch<false, true>(T, P, R, A, pass, nwg, st);
    else launch<false, false>(T, P, R, A, pass, nwg, st);
  }
}

}  // namespace jfc
