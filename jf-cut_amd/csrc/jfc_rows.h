// jfc_rows.h -- regions of 4096 nodes as 64-bit row words, shared by the global
// relabel (jfc_region.hip) and the cut and tag floods (jfc_flood.hip).
//
// One wavefront owns a region: 64 x 64 nodes in 2D, 64 x 8 x 8 in 3D.  Lane r
// holds row r (2D: y = r; 3D: y = r & 7, z = r >> 3), bit x = column x.
#pragma once

#include "jfc_device.h"

namespace jfc {

typedef unsigned long long u64;

// v_writelane: `old` with lane `lane` replaced by the uniform `v`
extern "C" __device__ int jfc_llvm_writelane(int v, int lane, int old) __asm(
    "llvm.amdgcn.writelane.i32");

template <bool D3>
struct Reg {
  static constexpr int TH = D3 ? 8 : 64, TD = D3 ? 8 : 1;
  static constexpr int K = D3 ? 6 : 8;
  // border rows along x: 2D rows 0 and 63; 3D the four faces in y and z, 8
  // rows each (faces: 0 low y, 1 high y, 2 low z, 3 high z)
  static constexpr int NV = D3 ? 32 : 2;
  static __device__ __forceinline__ constexpr int row(int j) {
    if (!D3) return j ? 63 : 0;
    const int k = j & 7;
    switch (j >> 3) {
      case 0: return 8 * k;
      case 1: return 8 * k + 7;
      case 2: return k;
      default: return 56 + k;
    }
  }
  // the direction that leaves the region through border row j
  static __device__ __forceinline__ constexpr int dir(int j) {
    if (!D3) return j ? 2 : 3;
    switch (j >> 3) {
      case 0: return 3;
      case 1: return 2;
      case 2: return 5;
      default: return 4;
    }
  }
};

// one-bit shifts of a row's word as two full-rate 32-bit instructions
__device__ __forceinline__ u64 shr1(u64 f) {
  const unsigned lo = (unsigned)f, hi = (unsigned)(f >> 32);
  return (u64)(hi >> 1) << 32 | __builtin_amdgcn_alignbit(hi, lo, 1);
}
__device__ __forceinline__ u64 shl1(u64 f) {
  const unsigned lo = (unsigned)f, hi = (unsigned)(f >> 32);
  return (u64)__builtin_amdgcn_alignbit(hi, lo, 31) << 32 | lo << 1;
}
__device__ __forceinline__ u64 from_next(u64 f) {  // lane r: lane r + 1's word, 0 in lane 63
  const unsigned lo = __builtin_amdgcn_update_dpp(0u, (unsigned)f, 0x130, 0xf, 0xf, true);
  const unsigned hi = __builtin_amdgcn_update_dpp(0u, (unsigned)(f >> 32), 0x130, 0xf, 0xf, true);
  return (u64)hi << 32 | lo;
}
__device__ __forceinline__ u64 from_prev(u64 f) {  // lane r: lane r - 1's word, 0 in lane 0
  const unsigned lo = __builtin_amdgcn_update_dpp(0u, (unsigned)f, 0x138, 0xf, 0xf, true);
  const unsigned hi = __builtin_amdgcn_update_dpp(0u, (unsigned)(f >> 32), 0x138, 0xf, 0xf, true);
  return (u64)hi << 32 | lo;
}
__device__ __forceinline__ u64 from_lane(u64 f, int addr) {  // lane addr / 4's word
  const unsigned lo = __builtin_amdgcn_ds_bpermute(addr, (int)(unsigned)f);
  const unsigned hi = __builtin_amdgcn_ds_bpermute(addr, (int)(unsigned)(f >> 32));
  return (u64)hi << 32 | lo;
}
// row r's word as a uniform value
__device__ __forceinline__ u64 row_word(u64 w, int r) {
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)w, r);
  const unsigned hi = __builtin_amdgcn_readlane((int)(unsigned)(w >> 32), r);
  return (u64)hi << 32 | lo;
}
__device__ __forceinline__ void set_row(int &lo, int &hi, int r, u64 w) {
  lo = jfc_llvm_writelane((int)(unsigned)w, r, lo);
  hi = jfc_llvm_writelane((int)(unsigned)(w >> 32), r, hi);
}
__device__ __forceinline__ bool bit_of_lane(u64 uniform) {
  return __builtin_amdgcn_inverse_ballot_w64(uniform);
}

// Graphs of up to this many regions leave most of the device's 1024 SIMDs with
// one wave or none in a pass over every region: there four waves share the
// rows of a region.  Above it a wave per region fills the device and the
// exchange through LDS would only add to its work.
constexpr int kSharedRegions = 512;

// A region's place in its instance.
struct RegionRef {
  int ox, oy, oz, wx;       // origin; columns inside the grid
  bool hasl, hasr;          // neighbours at x - 1, x + 1
  bool hasd, hasu;          // at y - 1, y + 1
  bool hasf, hasb;          // at z - 1, z + 1
  int sy, sz;               // region index steps in y and z
  u64 valid;                // the lane's row inside the grid
};

template <bool D3>
__device__ __forceinline__ RegionRef region_ref(const InstDesc &I, int t, int lane) {
  using G = Reg<D3>;
  RegionRef r;
  const int lt = t - I.tile_off;
  const int ltx = lt % I.tx, lq = lt / I.tx;
  const int lty = lq % I.ty, ltz = lq / I.ty;
  r.ox = ltx * 64;
  r.oy = lty * G::TH;
  r.oz = ltz * G::TD;
  r.wx = min(64, I.nx - r.ox);
  r.hasl = ltx > 0;
  r.hasr = ltx + 1 < I.tx;
  r.hasd = lty > 0;
  r.hasu = lty + 1 < I.ty;
  r.hasf = ltz > 0;
  r.hasb = ltz + 1 < I.tz;
  r.sy = I.tx;
  r.sz = I.tx * I.ty;
  const int y = r.oy + (D3 ? lane & 7 : lane), z = r.oz + (D3 ? lane >> 3 : 0);
  r.valid = y < I.ny && z < I.nz ? (r.wx == 64 ? ~0ull : (1ull << r.wx) - 1) : 0;
  return r;
}

// Step from a region to its neighbour b: 0 / 1 left / right, 2 / 3 low / high y,
// 4 / 5 low / high z; 2D 4-7 the corners (-x,-y), (-x,+y), (+x,-y), (+x,+y).
template <bool D3>
__device__ __forceinline__ int neighbour_step(const RegionRef &r, int b) {
  switch (b) {
    case 0: return -1;
    case 1: return 1;
    case 2: return -r.sy;
    case 3: return r.sy;
    case 4: return D3 ? -r.sz : -1 - r.sy;
    case 5: return D3 ? r.sz : -1 + r.sy;
    case 6: return 1 - r.sy;
    default: return 1 + r.sy;
  }
}

// The neighbours a visit marks: bit b of the uniform set, whose region index
// lane b holds.
struct Marks {
  unsigned set = 0;
  bool found = false;  // (cut flood) the visit labelled a deficit
  int at = 0;
  __device__ __forceinline__ void add(int b, bool on) { set |= on ? 1u << b : 0u; }
  __device__ __forceinline__ bool on(int lane) const { return lane < 8 && ((set >> lane) & 1u); }
};

// ---- a search in one launch ----
//
// A wave owns the regions t = blockIdx.x + i gridDim.x, at most 64, and visits
// those its neighbours mark until no mark is left anywhere.
//
// Marks are counts: a wave that changed a border adds 1 to the neighbour's
// count, the owner remembers the count it has served.  Each wave's marks made
// (high half) and marks served (low half) are summed in one of kSlots words; a
// visit adds the marks it is about to make, with those it served, before it
// makes them.  The first workgroup, when idle, reads every word for the marks
// served and then again for the marks made: equal sums mean that nothing was
// left to do between the two readings, and nothing will be (a mark is only made
// while one is being served).  It then tells the others through kSlots words of
// their own.  Every polled word has a cache line to itself: one word for all
// took 1.9 ms for a relabel of the 3750x2500 cut, its polling waves holding back
// the visits.  What a region's neighbours read and the sums are written through
// at device scope and have arrived (s_waitcnt) before a mark is made, and the
// owner reads them at device scope after it has seen the mark; a region's
// planes are touched by its owner only.
//
// The launcher caps the grid at what the device holds, but other kernels (a search
// of another graph, say) may hold places back, so every wait is bounded.  What is
// bounded is the time without progress, not a wave's own idleness: the marks
// made and served and the workgroups begun are looked at before a wave gives up.
//   - Once every workgroup has begun, nothing can hold the search up;
//     wait_ticks without progress is a way out only.
//   - Until then the marks of a workgroup without a place stay unserved, and two
//     searches that hold each other's places would wait for each other, so the
//     first workgroup gives up after kPlaceTicks without progress.
// It tells the others to quit and sets *quit, and the search is finished with
// passes over every region, as the solve's later searches are (a launch per pass
// takes 1.1 to 1.6 times as long).  Three threads that solve 128^3 volumes of
// their own: 57 ms a solve where workgroups without a place were waited for 20
// ms, 31 now; 256x192x176: 138 and 83.
constexpr int kSlots = kSettleSlots, kLine = kSettleLine;
static_assert(kSlots == 64, "a lane per slot");
constexpr int kServed = 0, kMade = 1, kBegun = 2;  // the words of a slot's line of sums
constexpr long long kPlaceTicks = 20000;           // 200 us: a visit takes 10 to 50
enum { kGo = 0, kDone = 1, kQuit = 2, kStop = 3 };

// Counts a workgroup that has begun, at its start.
__device__ __forceinline__ void begin(const SettleWords &A) {
  if (threadIdx.x == 0)
    (void)__hip_atomic_fetch_add(A.sums + kLine * (blockIdx.x & (kSlots - 1)) + kBegun, 1,
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Counts the marks of a visit that served `served` marks, then makes them.
__device__ __forceinline__ void publish(const SettleWords &A, const Marks &marks, int served,
                                        int lane) {
  if (lane == 0)
    (void)__hip_atomic_fetch_add((u64 *)(A.sums + kLine * (blockIdx.x & (kSlots - 1))),
                                 (u64)__popc(marks.set) << 32 | (unsigned)served,
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (marks.set) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (marks.on(lane))
      (void)__hip_atomic_fetch_add(A.marks + kLine * (long long)marks.at, 1, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
  }
}
__device__ __forceinline__ int shared_word(const int *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// the state every wave waits for, a word per slot
__device__ __forceinline__ void tell(const SettleWords &A, int what, int lane) {
  __hip_atomic_store(A.state + kLine * lane, what, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One wave's part.  all: the n regions' packing in this launch counts as
// served marks that nobody made.  visit(t, served) searches region t and
// publishes its marks; it returns true to end the search for every wave.
// Returns whether the search was finished.
template <class Visit>
__device__ __forceinline__ bool settle(const SettleWords &A, int n, bool all, long long *visits_out,
                                       Visit visit) {
  const int lane = threadIdx.x & 63;
  const int slot = blockIdx.x & (kSlots - 1);
  const int G = gridDim.x;
  const int mine = blockIdx.x + lane * G;  // the lane's region of up to 64
  const bool own = mine < n;
  bool done = false;
  int seen = 0, visits = 0, turn = 0;
  long long since = 0;  // idle, and without progress as far as known, since then
  int progress = 0;     // the sums at the last look
  int begun = 0;        // (first workgroup) the workgroups begun, at the last look
  auto sum = [&](int word) {
    int v = shared_word(A.sums + kLine * lane + word);
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
  };
  for (;;) {
    const int now = own ? shared_word(A.marks + kLine * (long long)mine) : 0;
    const int state = shared_word(A.state + kLine * slot);
    const u64 m = __ballot(now != seen);
    if (state == kStop) break;
    if (m) {
      since = 0;
      // one region per poll, in turn: marks made meanwhile for the others are
      // served by one visit each
      const u64 ahead = m & (~0ull << turn);
      const int i = __builtin_ctzll(ahead ? ahead : m);
      turn = (i + 1) & 63;
      const int served = __builtin_amdgcn_readlane(now - seen, i);
      if (lane == i) seen = now;
      ++visits;
      if (visit(blockIdx.x + i * G, served)) {
        tell(A, kStop, lane);
        break;
      }
      continue;
    }
    done = state == kDone;
    if (state != kGo) break;
    const long long tick = wall_clock64();
    if (since == 0) since = tick;
    long long limit = A.wait_ticks;
    int now_at = progress;
    if (blockIdx.x == 0) {
      const int served = sum(kServed);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const int made = sum(kMade);
      if (made + (all ? n : 0) == served) {
        tell(A, kDone, lane);
        continue;
      }
      if (begun < G) {
        limit = min(limit, kPlaceTicks);
        if (tick - since >= limit) begun = sum(kBegun);
        if (begun == G) limit = A.wait_ticks;
      }
      now_at = served + made + begun;
    } else if (limit > 0 && tick - since >= limit) {
      now_at = sum(kBegun) + sum(kServed) + sum(kMade);
    }
    if (now_at != progress) {
      progress = now_at;
      since = tick;
    }
    if (tick - since >= limit) {
      tell(A, kQuit, lane);
      if (lane == 0) {
        __hip_atomic_store(A.quit, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (A.quit_host)
          __hip_atomic_store(A.quit_host, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
      break;
    }
    __builtin_amdgcn_s_sleep(8);
  }
  if (visits && lane == 0) atomicAdd((u64 *)&visits_out[blockIdx.x & 63], (u64)visits);
  return done;
}

// Workgroups of a persistent launch that the device holds at once.
int device_cus();
template <auto Kernel, int Block = 256>
int resident_grid_b(int want) {
  static const int per_cu = [] {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, Kernel, Block, 0) != hipSuccess || n < 1)
      n = 1;
    return n;
  }();
  const int cap = per_cu * device_cus();
  return want < 1 ? 1 : want < cap ? want : cap;
}

}  // namespace jfc
