// jfc_flood.hip -- the canonical cut and the tag post-process as floods over
// bit-parallel regions (jfc_rows.h).
//
// Reference counterparts (src/QVisualizer/cl/GraphCut/):
//   cut  graphcut_init_cut, graphcut_compute_cut  graphcut_compute_cut.cl:19-49, :51-140, :182-282
//   tag  graphcut_init_tag, graphcut_compute_tag  graphcut_compute_tag.cl:19-49, :51-242
//   kPack also reduce_flow  bin/x64/cl/Infrastructures/reduce.cl:17-42 (int64 here)
//
// Cut: the nodes with excess are labelled, and a labelled node labels every
// neighbour it has residual capacity toward.  A labelled node with a deficit
// means that an augmenting path is left: *cert is set
// (graphcut_compute_cut.cl:135-139).  Tag: the foreground seeds are tagged, and
// a tagged node tags its axis neighbours on the source side of the cut.
//
// A step of a region's flood is a shift and an AND per direction on 64-bit row
// words.  Passes exchange what crosses a region's border as bits: each region
// keeps the labels it sends to each neighbour, the neighbours read them.
//   kPack     every region: the seeds (cut: excess signs and the remaining
//             deficit) packed; regions holding one are flooded;
//   kBorders  the regions sent new labels: flooded from them;
//   kFinal    every region, once no region is sent any: the labels written.
// One launch takes every pass of graphs of up to 512 regions, and the passes
// between the first and the last of the others (k_flood_all).
// A region's arcs are packed when a label first reaches it, so regions off
// the source side read their excess and nothing else.  Once *cert is set the
// labels of a search that only proves the cut (FloodPass::stop) are not
// needed: its later passes return at once.
//
// What bounds it and what it measured (against a flood of 32x8, 8x8x4 and
// 32x4x2 tiles node by node in LDS after a pass over the nodes that wrote
// their labels): the first and the last pass are bound by their 4 and 1 bytes
// per node, the passes between by their launches.  The cut of the 15000x10000
// 8-connected graph takes 0.30 instead of 0.48 ms, of the 2560x1440x50 video
// volume 0.36 instead of 0.62, of 256 uneven images 0.24 instead of 0.46; the
// tags of a 181x217x181 scan 35 passes fewer.  On a video volume that
// certifies 31 times before its last cut, searches that stop at the first
// deficit take 8.8 instead of 226 ms.
#include "jfc_rows.h"

#include <algorithm>

namespace jfc {

namespace {

// Labels a region sends: 0 / 1 to its left / right neighbour (bit = row); 2D:
// 2 / 3 up from row 0 / down from row 63 (bit = column), 4 corners (bit 0
// (-x,-y), 1 (-x,+y), 2 (+x,-y), 3 (+x,+y)); 3D: 2 + 8 f + k for row k of face f
// (0 low y, 1 high y, 2 low z, 3 high z).
template <bool D3>
constexpr int kOut = D3 ? 2 + 32 : 5;

__device__ __forceinline__ u64 sent(const u64 *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void send(u64 *p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Visits region t.  W: waves of the workgroup that share a region's packing
// and its labels, 64 / W rows each; the flood is the first wave's alone.
template <bool D3, bool TAG, int PASS, bool ONE, int W>
__device__ __forceinline__ void flood_visit(const Tiles &T, const Planes &P, const FloodBuf &R,
                                            const FloodPass &A, int t, Marks &marks) {
  constexpr int KM = D3 ? 6 : TAG ? 4 : 8;
  const int lane = threadIdx.x & 63;
  const int wv0 = W > 1 ? 64 / W * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;  // first row
  const InstDesc &I = ONE ? T.one : T.inst[T.tile_inst[t]];
  const int K = TAG ? KM : I.K;
  const RegionRef r = region_ref<D3>(I, t, lane);
  const int ly = D3 ? lane & 7 : lane, lz = D3 ? lane >> 3 : 0;
  const bool diag = !D3 && !TAG && K == 8;
  u64 *pk = R.packed + (long long)t * R.planes * 64 + lane;  // K direction planes
  u64 *ps = pk + 64 * (R.planes - 2);  // cut: deficits; tag: source side.  Then the labels
  auto row_y = [&](int q) { return r.oy + (D3 ? q & 7 : q); };
  auto row_z = [&](int q) { return r.oz + (D3 ? q >> 3 : 0); };

  if (PASS == kFinal) {
    // four rows at a time, four nodes per lane
    const u64 s = ps[64];
    const int x = 4 * (lane & 15);
#pragma unroll
    for (int u = 0; u < 16 / W; ++u) {
      const int q = wv0 + 4 * u + (lane >> 4);
      const u64 w = from_lane(s, 4 * q);
      const unsigned nib = (unsigned)(w >> x) & 15u;
      if (x < r.wx && row_y(q) < I.ny && row_z(q) < I.nz)
        *(unsigned *)(P.lab + node_index(I, r.ox + x, row_y(q), row_z(q))) =
            (nib * 0x00204081u) & 0x01010101u;
    }
    return;
  }

  // the next RB rows' loads are in flight while RB rows are used; rows and
  // columns off the grid read a valid dummy address
  constexpr int RB = 16;
  auto rows = [&](auto load, auto use) {
    decltype(load(0ll)) w[2][RB];
    auto fetch = [&](decltype(load(0ll)) *wb, int r0) {
#pragma unroll
      for (int u = 0; u < RB; ++u) {
        const int q = r0 + u;
        const bool ok = row_y(q) < I.ny && row_z(q) < I.nz && lane < r.wx;
        wb[u] = load(ok ? node_index(I, r.ox + lane, row_y(q), row_z(q)) : 0);
      }
    };
    fetch(w[0], wv0);
#pragma unroll
    for (int b = 0; b < 64 / RB / W; ++b) {
      if (b + 1 < 64 / RB / W) fetch(w[(b + 1) & 1], RB * (b + 1));
#pragma unroll
      for (int u = 0; u < RB; ++u) {
        const int q = wv0 + RB * b + u;
        const bool ok = row_y(q) < I.ny && row_z(q) < I.nz && lane < r.wx;
        use(q, ok, w[b & 1][u]);
      }
    }
  };
  // the waves' rows of N words gathered in every wave's registers
  __shared__ u64 s_rows[W > 1 ? 8 : 1][64];
  auto gather = [&](u64 *w, int n) {
    if constexpr (W > 1) {
      __syncthreads();
      if ((unsigned)(lane - wv0) < 64u / W)
        for (int d = 0; d < n; ++d) s_rows[d][lane] = w[d];
      __syncthreads();
      for (int d = 0; d < n; ++d) w[d] = s_rows[d][lane];
    }
  };
  u64 M[KM];
  auto pack_arcs = [&]() {
    if constexpr (!TAG) {
      int lo[KM], hi[KM];
#pragma unroll
      for (int d = 0; d < KM; ++d) lo[d] = hi[d] = 0;
      rows([&](long long v) { return P.rmask[v]; },
           [&](int q, bool ok, unsigned m) {
             m = ok ? m : 0u;
#pragma unroll
             for (int d = 0; d < KM; ++d)
               if (D3 || d < 4 || K == 8) set_row(lo[d], hi[d], q, __ballot(m & (1u << d)));
           });
#pragma unroll
      for (int d = 0; d < KM; ++d) M[d] = (u64)(unsigned)hi[d] << 32 | (unsigned)lo[d];
      gather(M, KM);
      if (wv0 == 0) {
#pragma unroll
        for (int d = 0; d < KM; ++d)
          if (d < K) pk[64 * d] = M[d];
      }
    }
  };

  u64 D, S, F;  // deficits (tag: source side), labels, the labels of the last step
  const long long o0 = (long long)t * kOut<D3>;
  u64 own = 0, owny = 0, ownz = 0;  // what the region has sent so far
  const int iy = 2 + (ly == 7 ? 8 : 0) + lz, iz = 18 + (lz == 7 ? 8 : 0) + ly;  // 3D: its words
  if (PASS == kPack) {
    u64 w[2];
    int alo = 0, ahi = 0, blo = 0, bhi = 0;
    if constexpr (TAG) {
      rows([&](long long v) { return (unsigned short)(P.lab[v] | A.object[v] << 8); },
           [&](int q, bool ok, unsigned short b) {
             set_row(alo, ahi, q, __ballot(ok && (b & 255) != 0));
             set_row(blo, bhi, q, __ballot(ok && (b >> 8) != 0));
           });
    } else {
      long long deficit = 0;
      rows([&](long long v) { return P.e[v]; },
           [&](int q, bool ok, int e) {
             e = ok ? e : 0;
             deficit += max(-e, 0);
             set_row(alo, ahi, q, __ballot(e > 0));
             set_row(blo, bhi, q, __ballot(e < 0));
           });
      // one atomic per wave, spread over 64 sums where one instance takes all
      for (int o = 32; o > 0; o >>= 1) deficit += __shfl_xor(deficit, o);
      if (lane == 0 && deficit)
        atomicAdd((u64 *)&A.def[ONE ? t & 63 : T.tile_inst[t]], (u64)deficit);
    }
    w[0] = (u64)(unsigned)ahi << 32 | (unsigned)alo;
    w[1] = (u64)(unsigned)bhi << 32 | (unsigned)blo;
    gather(w, 2);
    F = w[0];
    D = w[1];
    S = 0;
    const bool seeded = __ballot(F != 0) != 0;
    if (seeded) pack_arcs();
    if (wv0 > 0) return;
    ps[0] = D;
    if (lane == 0) R.open[t] = seeded;
    if (!seeded) {
      ps[64] = 0;
      return;
    }
  } else {
    // the labels sent here
    auto word = [&](bool have, int nb, int idx) {
      return have ? sent(R.out + (long long)(t + nb) * kOut<D3> + idx) : 0;
    };
    const u64 wl = word(r.hasl, -1, 1), wr = word(r.hasr, 1, 0);
    u64 in = 0, wy = 0, wz = 0;
    if constexpr (D3) {
      wy = word(ly == 0 ? r.hasd : ly == 7 && r.hasu, ly == 0 ? -r.sy : r.sy, ly == 0 ? 10 + lz : 2 + lz);
      wz = word(lz == 0 ? r.hasf : lz == 7 && r.hasb, lz == 0 ? -r.sz : r.sz,
                lz == 0 ? 26 + ly : 18 + ly);
      if (ly == 0 || ly == 7) owny = sent(R.out + o0 + iy);
      if (lz == 0 || lz == 7) ownz = sent(R.out + o0 + iz);
      if (lane < 2) own = sent(R.out + o0 + lane);
    } else {
      wy = word(lane == 0 ? r.hasd : lane == 63 && r.hasu, lane == 0 ? -r.sy : r.sy, lane == 0 ? 3 : 2);
      if (diag) {
        const u64 c0 = word(r.hasl && r.hasd, -1 - r.sy, 4), c1 = word(r.hasl && r.hasu, -1 + r.sy, 4);
        const u64 c2 = word(r.hasr && r.hasd, 1 - r.sy, 4), c3 = word(r.hasr && r.hasu, 1 + r.sy, 4);
        const u64 bits = lane == 0 ? (c0 >> 3 & 1) | (c2 >> 1 & 1) << 63
                                   : (c1 >> 2 & 1) | (c3 & 1) << 63;
        if (lane == 0 || lane == 63) in = bits;
      }
      if (lane < kOut<D3>) own = sent(R.out + o0 + lane);
    }
    S = ps[64];
    D = ps[0];
    const bool open = TAG || R.open[t];
    if (open) {
#pragma unroll
      for (int d = 0; d < KM; ++d) M[d] = TAG ? 0 : pk[64 * min(d, K - 1)];
#pragma unroll
      for (int d = 0; d < KM; ++d)
        if (d >= K) M[d] = 0;
    }
    in |= wy | wz | (bit_of_lane(wl) ? 1ull : 0ull) | (bit_of_lane(wr) ? 1ull << 63 : 0ull);
    F = in & ~S;
    if (TAG) F &= D;
    if (!__ballot(F != 0)) return;
    if (!open) {
      pack_arcs();
      if (lane == 0) R.open[t] = 1;
    }
  }

  if constexpr (TAG) {
#pragma unroll
    for (int d = 0; d < KM; ++d) M[d] = ~0ull;
  }
  // 3D: what leaves through the faces in y and z, kept apart, so that the
  // lane shifts below need no edge tests
  u64 ey = 0, ez = 0;
  if constexpr (D3) {
    if (ly == 7) ey = M[2], M[2] = 0;
    if (ly == 0) ey = M[3], M[3] = 0;
    if (lz == 7) ez = M[4], M[4] = 0;
    if (lz == 0) ez = M[5], M[5] = 0;
  }
  const int addr_up = ((lane + 8) & 63) * 4, addr_dn = ((lane - 8) & 63) * 4;
  S |= F;
  for (;;) {
    u64 up = F & M[2], dn = F & M[3];  // toward lane + 1, lane - 1
    u64 n = shl1(F & M[0]) | shr1(F & M[1]);
    if constexpr (D3) {
      n |= from_lane(F & M[4], addr_dn) | from_lane(F & M[5], addr_up);
    } else if constexpr (!TAG) {
      if (diag) {
        up |= shl1(F & M[4]) | shr1(F & M[6]);
        dn |= shr1(F & M[5]) | shl1(F & M[7]);
      }
    }
    n |= from_prev(up) | from_next(dn);
    F = n & ~S;
    if (TAG) F &= D;
    S |= F;
    if (!__ballot(F != 0)) break;
  }
  ps[64] = S;
  if (!TAG && __ballot((S & D) != 0)) {
    marks.found = true;
    if (lane == 0) *A.cert = 1;
  }

  // ---- what the region sends, and the marks of the neighbours sent more
  u64 lw = __ballot((S & M[1] & 1) != 0), rw = __ballot((S & M[0]) >> 63 != 0);
  marks.at = t + neighbour_step<D3>(r, lane);
  if constexpr (D3) {
    const u64 vy = S & ey & ~owny, vz = S & ez & ~ownz;
    const u64 vx = (lane == 0 ? lw : lane == 1 ? rw : 0) & ~own;
    if (vx) send(R.out + o0 + lane, own | vx);
    if (vy) send(R.out + o0 + iy, owny | vy);
    if (vz) send(R.out + o0 + iz, ownz | vz);
    const u64 cx = __ballot(vx != 0), cy = __ballot(vy != 0), cz = __ballot(vz != 0);
    constexpr u64 low_y = 0x0101010101010101ull;
    marks.add(0, r.hasl && (cx & 1));
    marks.add(1, r.hasr && (cx & 2));
    marks.add(2, r.hasd && (cy & low_y));
    marks.add(3, r.hasu && (cy & ~low_y));
    marks.add(4, r.hasf && (cz & 0xffull));
    marks.add(5, r.hasb && (cz & ~0xffull));
  } else {
    u64 bw = S & M[2], tw = S & M[3], corners = 0;
    if constexpr (!TAG) {
      if (diag) {
        const u64 r4 = __ballot((S & M[4]) >> 63 != 0), r7 = __ballot((S & M[7]) >> 63 != 0);
        const u64 l5 = __ballot((S & M[5] & 1) != 0), l6 = __ballot((S & M[6] & 1) != 0);
        rw |= r4 << 1 | r7 >> 1;
        lw |= l6 << 1 | l5 >> 1;
        bw |= shl1(S & M[4]) | shr1(S & M[6]);
        tw |= shr1(S & M[5]) | shl1(S & M[7]);
        corners = (l5 & 1) | (l6 >> 63) << 1 | (r7 & 1) << 2 | (r4 >> 63) << 3;
      }
    }
    const u64 top = row_word(tw, 0), bottom = row_word(bw, 63);
    const u64 w = lane == 0 ? lw : lane == 1 ? rw : lane == 2 ? top : lane == 3 ? bottom
                                                                  : lane == 4 ? corners : 0;
    const u64 v = w & ~own;
    if (v) send(R.out + o0 + lane, own | v);
    const u64 ch = __ballot(v != 0);
    const u64 cc = row_word(v, 4);
    marks.add(0, r.hasl && (ch & 1));
    marks.add(1, r.hasr && (ch & 2));
    marks.add(2, r.hasd && (ch & 4));
    marks.add(3, r.hasu && (ch & 8));
    marks.add(4, r.hasl && r.hasd && (cc & 1));
    marks.add(5, r.hasl && r.hasu && (cc & 2));
    marks.add(6, r.hasr && r.hasd && (cc & 4));
    marks.add(7, r.hasr && r.hasu && (cc & 8));
  }
}

template <bool D3, bool TAG, int PASS, bool ONE, int W>
__global__ __launch_bounds__(64 * W) void k_flood(Tiles T, Planes P, FloodBuf R, FloodPass A) {
  const int lane = threadIdx.x & 63;
  bool marked = false;
  const bool found = !TAG && PASS != kPack && A.stop && *A.cert;
  auto mark = [&](const Marks &marks) {
    if (marks.on(lane)) A.c.dirty_out[marks.at] = 1;
    marked |= marks.set != 0;
  };
  if (PASS == kBorders) {
    // some region was marked for this pass; the host learns it from here
    const bool work = *A.c.any_in && !found;
    if (blockIdx.x == 0 && lane == 0) {
      *A.c.any_clear = 0;
      __hip_atomic_store(A.c.post, A.c.seq * 2 + (work ? 1 : 0), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (!work) return;
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
        Marks marks;
        flood_visit<D3, TAG, PASS, ONE, 1>(T, P, R, A, base + i * G, marks);
        mark(marks);
      }
    }
    if (visits && lane == 0) atomicAdd((u64 *)&A.c.visits[blockIdx.x & 63], (u64)visits);
  } else {
    if (found || (PASS == kFinal && A.w.sums && shared_word(A.w.state) != kDone)) return;
    Marks marks;
    flood_visit<D3, TAG, PASS, ONE, W>(T, P, R, A, blockIdx.x, marks);
    if (PASS == kPack && A.w.sums) {
      if (threadIdx.x < 64) publish(A.w, marks, 0, lane);
      return;
    }
    mark(marks);
  }
  if (PASS != kFinal && marked && lane == 0) *A.c.any_out = 1;
}

// The passes between kPack and kFinal in one launch (settle); W = 4 (one region
// per workgroup): kPack and kFinal too.  A search that only proves the cut ends
// for every wave with the first labelled deficit.  Launches, gaps and the
// host's checks of the passes cost small graphs more than the visits: solves of
// 512x512 0.57 -> 0.54 ms, 600x450 with tags 1.08 -> 1.01, 96x80 0.69 -> 0.64,
// 181x217x181 with tags 2.64 -> 2.53; 15000x10000 4.43 -> 4.40.
template <bool D3, bool TAG, bool ONE, int W>
__global__ __launch_bounds__(64 * W) void k_flood_all(Tiles T, Planes P, FloodBuf R, FloodPass A) {
  __shared__ int s_done;
  constexpr bool kAll = W > 1;
  const int lane = threadIdx.x & 63;
  if (!kAll && !TAG && A.stop && *A.cert) return;  // found while packing
  begin(A.w);
  bool done = false, found = false;
  if (kAll) {
    Marks marks;
    flood_visit<D3, TAG, kPack, ONE, W>(T, P, R, A, blockIdx.x, marks);
    if (threadIdx.x < 64) {
      publish(A.w, marks, 1, lane);
      found = !TAG && A.stop && marks.found;
      if (found) tell(A.w, kStop, lane);
    }
  }
  if (threadIdx.x < 64 && !found)
    done = settle(A.w, T.ntiles, kAll, A.c.visits, [&](int t, int served) {
      Marks marks;
      flood_visit<D3, TAG, kBorders, ONE, 1>(T, P, R, A, t, marks);
      publish(A.w, marks, served, lane);
      return !TAG && A.stop && marks.found;
    });
  if constexpr (!kAll) return;
  if (threadIdx.x == 0) s_done = done;
  __syncthreads();
  if (!s_done) return;
  Marks marks;
  flood_visit<D3, TAG, kFinal, ONE, W>(T, P, R, A, blockIdx.x, marks);
}

template <bool D3, bool TAG, bool ONE>
void launch(const Tiles &T, const Planes &P, const FloodBuf &R, const FloodPass &A, int pass,
            int nwg, hipStream_t st) {
  const int n = T.ntiles;
  const bool shared = n <= kSharedRegions;
  if (pass == kBorders) {
    k_flood<D3, TAG, kBorders, ONE, 1><<<std::min(n, nwg), 64, 0, st>>>(T, P, R, A);
  } else if (pass == kPack) {
    if (shared) k_flood<D3, TAG, kPack, ONE, 4><<<n, 256, 0, st>>>(T, P, R, A);
    else k_flood<D3, TAG, kPack, ONE, 1><<<n, 64, 0, st>>>(T, P, R, A);
  } else {
    if (shared) k_flood<D3, TAG, kFinal, ONE, 4><<<n, 256, 0, st>>>(T, P, R, A);
    else k_flood<D3, TAG, kFinal, ONE, 1><<<n, 64, 0, st>>>(T, P, R, A);
  }
}

// A workgroup of k_flood_all looks after at most 64 regions (W = 4: after one).
template <bool D3, bool TAG, bool ONE>
bool launch_all(const Tiles &T, const Planes &P, const FloodBuf &R, const FloodPass &A,
                hipStream_t st) {
  const int n = T.ntiles;
  if (n <= kSharedRegions && resident_grid_b<&k_flood_all<D3, TAG, ONE, 4>, 256>(n) == n) {
    k_flood_all<D3, TAG, ONE, 4><<<n, 256, 0, st>>>(T, P, R, A);
    return true;
  }
  const int grid = resident_grid_b<&k_flood_all<D3, TAG, ONE, 1>, 64>(n);
  if (64LL * grid < n) return false;
  launch<D3, TAG, ONE>(T, P, R, A, kPack, 0, st);
  k_flood_all<D3, TAG, ONE, 1><<<grid, 64, 0, st>>>(T, P, R, A);
  launch<D3, TAG, ONE>(T, P, R, A, kFinal, 0, st);
  return true;
}

template <bool D3, bool TAG>
bool launch_all(const Tiles &T, const Planes &P, const FloodBuf &R, const FloodPass &A,
                hipStream_t st) {
  return T.ninst == 1 ? launch_all<D3, TAG, true>(T, P, R, A, st)
                      : launch_all<D3, TAG, false>(T, P, R, A, st);
}

template <bool D3, bool TAG>
void launch(const Tiles &T, const Planes &P, const FloodBuf &R, const FloodPass &A, int pass,
            int nwg, hipStream_t st) {
  if (T.ninst == 1) launch<D3, TAG, true>(T, P, R, A, pass, nwg, st);
  else launch<D3, TAG, false>(T, P, R, A, pass, nwg, st);
}

}  // namespace

int flood_out_words(bool d3) { return d3 ? kOut<true> : kOut<false>; }

void launch_flood(bool d3, bool tag, const Tiles &T, const Planes &P, const FloodBuf &R,
                  const FloodPass &A, int pass, int nwg, hipStream_t st) {
  if (d3) {
    if (tag) launch<true, true>(T, P, R, A, pass, nwg, st);
    else launch<true, false>(T, P, R, A, pass, nwg, st);
  } else {
    if (tag) launch<false, true>(T, P, R, A, pass, nwg, st);
    else launch<false, false>(T, P, R, A, pass, nwg, st);
  }
}

bool launch_flood_all(bool d3, bool tag, const Tiles &T, const Planes &P, const FloodBuf &R,
                      const FloodPass &A, hipStream_t st) {
  if (d3) return tag ? launch_all<true, true>(T, P, R, A, st) : launch_all<true, false>(T, P, R, A, st);
  return tag ? launch_all<false, true>(T, P, R, A, st) : launch_all<false, false>(T, P, R, A, st);
}

}  // namespace jfc
