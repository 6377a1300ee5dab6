// Long bags taken out of the teams' hands (optional part of the fused embedding kernel, for data
// whose bag lengths are skewed).
//
// A bag far longer than its feature's schedule was chosen for keeps one team -- at best one
// wavefront (rfx::wave_bag) -- busy long after the rest of the grid has finished, and the
// wavefront that meets it in the middle of its tiles falls behind the others of its workgroup.
// A library emitted with outliers=True deals with such bags at two levels.
//   * Outliers: find_outliers, launched ahead of the fused kernel, walks all offsets of the
//     batch, and every bag longer than its feature's outlier threshold (beyond its schedule's
//     reach, rfx::long_bag_threshold, and at least 128 KiB of traffic) becomes an entry
//     {feature, bag, first part, parts} of a list in the caller's workspace, parts = its
//     traffic / kOutlierUnit (1..kOutlierMaxParts; 128, 256 and 512 KiB per part give 227, 219
//     and 234 us on a 100-feature model with lognormal bag lengths).  The teams of the fused
//     kernel leave those bags alone.  When a workgroup has run its share of the regular tiles it
//     draws parts from a ticket counter until none is left, so that the workgroups whose
//     regular tiles were cheap take more of them (dealt out like the regular tiles, three parts
//     of 10-30 us to one workgroup and one to another, the same model spent a third of the
//     kernel in its tail: 224 us against 192 with the parts drawn).  A part runs like a part of
//     a split bag (rfx::split_part: the workgroup sums its share, partial sums in a slot,
//     arrival counter, the last one adds the slots in part order and writes the output).  If
//     the list overflows (more than CAP bags or 4 * CAP parts) the launch does without it.
//     The workgroup that holds the last ticket of a counter puts it back to zero, and the last
//     counter to get there the list header, for the next launch.
//   * Mid-size bags (beyond the schedule's reach, below the outlier threshold) are summed by one
//     wavefront, but not necessarily the one that met them: it puts them on a list of its
//     workgroup in LDS (MidQueue), and every wavefront of the workgroup takes bags from that
//     list between its tiles, so that the four wavefronts of a workgroup finish together.
//
// Reference counterpart: the role of rbk::SparseSegmentReduce
// (examples/csrc/include/reduce_by_key_kernel.cuh), load balance under skewed bag lengths.
#pragma once
#include "rfx_binding.hip.h"

namespace rfx {

// The list holds CAP entries and 4 * CAP parts; the emitter sizes it by the model (4 096 entries
// up to 128 features, 16 384 beyond).
constexpr int kOutlierUnit = 256 * 1024;     // traffic of one part
constexpr int kOutlierMaxParts = 64;

struct OutlierHeader {
  unsigned long long pack;                   // entries << 32 | parts, both as reserved so far
  int finished;                              // ticket counters whose last ticket has been drawn
  int last_entries, last_parts;              // what the previous launch found (for the caller)
  int pad[27];
};
// The ticket counters of the parts, in the workspace right ahead of the OutlierSpace, each on a
// cache line of its own.  A device-scope add to one address takes 11 ns, one after the other, so
// where there are fewer parts than workgroups -- most draws only learn that nothing is left, and
// the launch is short -- the workgroups of each XCD draw from a counter of their own (100
// features, 37 samples with lognormal bag lengths: FusedKnl 27.8 us, and some 14 us more with
// 1 280 draws from one counter).  Where parts abound one counter serves the device, because it
// also evens out the XCDs (2 048 samples, 2 050 parts: 171.4 us, 175.3 with a counter per XCD).
struct OutlierTickets {
  int next[8][32];
};
struct OutlierEntry {
  int feat, bag, first, parts;
};

// MAXD: largest embedding dimension among the features that can have outliers, rounded up to 4
template <int MAXD, int CAP> struct OutlierSpace {
  static constexpr int kCap = CAP;           // entries
  static constexpr int kPartCap = 4 * CAP;   // parts of all entries together
  OutlierHeader hdr;
  OutlierEntry entries[kCap];
  int counters[kCap];                        // arrival counters, zero between launches
  int partmap[kPartCap];                     // part -> entry
  unsigned int slots[kPartCap][MAXD];        // partial sums
};

// Bags a workgroup of the finding kernel looks at per round: kFindBags per thread, 256 threads.
constexpr int kFindBags = 8;
constexpr int kFindThreads = 256;

// Grid (x: bags, y: features), any size.  A kernel of a few microseconds: a launch, the feature's
// address, its offsets, one reservation.  The workgroup adds up what its bags need and reserves
// entries and parts for all of them with one atomic add, so that a model of 100 features and
// 2 048 bags makes at most 100 adds to the one word that hands them out (a thousand, one per
// outlier, took 8.5 us in all; 5.1 us this way).
template <int F, typename Space>
__device__ __forceinline__ void
find_outliers(Space *__restrict__ sp, const IoView &io,
              const int *__restrict__ long_thr, const int *__restrict__ lookup_bytes) {
  __shared__ int wave_need[kFindThreads / 64];
  __shared__ unsigned long long base_pack;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int f = blockIdx.y; f < F; f += gridDim.y) {
    const int thr = long_thr[f];
    if (thr <= 0) continue;                  // a schedule that handles long bags itself
    const int *offs = io.offsets(f);
    const int per_lookup = lookup_bytes[f];
    for (int b0 = blockIdx.x * kFindThreads * kFindBags; b0 < io.batch;
         b0 += gridDim.x * kFindThreads * kFindBags) {
      int first[kFindBags], parts[kFindBags];
#pragma unroll
      for (int k = 0; k < kFindBags; ++k) {
        const int b = min(b0 + k * kFindThreads + tid, io.batch - 1);
        first[k] = offs[b];
        parts[k] = offs[b + 1];
      }
      // this thread's entries << kNeedShift | parts, added up over the workgroup in one scan
      constexpr int kNeedShift = 18;
      static_assert(kFindThreads * kFindBags * kOutlierMaxParts < 1 << kNeedShift &&
                    kFindThreads * kFindBags < 1 << (31 - kNeedShift), "fields of the packed need");
      int need = 0;
#pragma unroll
      for (int k = 0; k < kFindBags; ++k) {
        const int len = parts[k] - first[k];
        const bool listed = b0 + k * kFindThreads + tid < io.batch && len > thr;
        const long long cost = static_cast<long long>(len) * per_lookup;
        const long long want = (cost + kOutlierUnit - 1) / kOutlierUnit;
        parts[k] = listed ? static_cast<int>(want > kOutlierMaxParts ? kOutlierMaxParts : want) : 0;
        if (listed) need += (1 << kNeedShift) | parts[k];
      }
      const int upto = wave_inclusive_scan(need, lane);
      if (lane == 63) wave_need[wave] = upto;
      __syncthreads();
      int before = upto - need, total = 0;
#pragma unroll
      for (int w = 0; w < kFindThreads / 64; ++w) {
        if (w < wave) before += wave_need[w];
        total += wave_need[w];
      }
      if (tid == 0 && total)
        base_pack = atomicAdd(&sp->hdr.pack, (static_cast<unsigned long long>(total >> kNeedShift) << 32) |
                                                 static_cast<unsigned long long>(total & ((1 << kNeedShift) - 1)));
      __syncthreads();
      if (need) {
        long long q = static_cast<long long>(base_pack >> 32) + (before >> kNeedShift);
        long long p0 = static_cast<long long>(base_pack & 0xffffffffull) + (before & ((1 << kNeedShift) - 1));
#pragma unroll
        for (int k = 0; k < kFindBags; ++k) {
          if (!parts[k]) continue;
          if (q < Space::kCap && p0 + parts[k] <= Space::kPartCap) {
            sp->entries[q] = OutlierEntry{f, b0 + k * kFindThreads + tid, static_cast<int>(p0), parts[k]};
            for (int p = 0; p < parts[k]; ++p) sp->partmap[p0 + p] = static_cast<int>(q);
          }
          ++q;
          p0 += parts[k];
        }
      }
      __syncthreads();                       // wave_need and base_pack are free again
    }
  }
}

// What a workgroup of the fused kernel knows about the list: the parts to draw (0 if there are
// none or the list overflowed: then the teams sum every bag themselves), and the ticket counter
// it draws from.  Counter c of C (C = 8, one per XCD, or 1: see OutlierTickets) hands out the parts
// c, c + C, c + 2C, ...
struct OutlierDraw {
  int *next;                                 // this workgroup's counter
  int parts;                                 // all parts of the launch
  int counter, counters;
  int sharers;                               // workgroups that draw from it
  bool listed;                               // the header has to be put back to zero

  __device__ __forceinline__ int part_of(const int ticket) const { return counter + ticket * counters; }
  // every workgroup draws until its part lies beyond the last: the tickets handed out are
  // 0 .. (parts of this counter) + sharers - 1
  __device__ __forceinline__ bool is_last(const int ticket) const {
    const int mine = parts > counter ? (parts - counter + counters - 1) / counters : 0;
    return ticket == mine + sharers - 1;
  }
};

template <typename Space>
__device__ __forceinline__ OutlierDraw outlier_draw(Space *sp) {
  const unsigned long long pack =
      __hip_atomic_load(&sp->hdr.pack, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const unsigned long long entries = pack >> 32, parts = pack & 0xffffffffull;
  OutlierDraw d;
  d.parts = entries <= Space::kCap && parts <= Space::kPartCap ? static_cast<int>(parts) : 0;
  d.counters = gridDim.x >= 8 && d.parts < static_cast<int>(gridDim.x) ? 8 : 1;
  d.counter = blockIdx.x % d.counters;
  d.next = &(reinterpret_cast<OutlierTickets *>(sp) - 1)->next[d.counter][0];
  d.sharers = (gridDim.x - d.counter + d.counters - 1) / d.counters;
  d.listed = pack != 0;
  return d;
}

// The next ticket for the calling workgroup (one thread draws).
__device__ __forceinline__ int draw_outlier_ticket(const OutlierDraw &d) {
  return __hip_atomic_fetch_add(d.next, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// By one thread of the workgroup that holds the last ticket of its counter: puts the counter back
// to zero.  True for the last counter of the launch to get there; every workgroup has read the
// header by then, since each of them has drawn.
template <typename Space>
__device__ __forceinline__ bool outlier_counter_done(Space *sp, const OutlierDraw &d) {
  __hip_atomic_store(d.next, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return __hip_atomic_fetch_add(&sp->hdr.finished, 1, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT) == d.counters - 1;
}

// ... which then puts the header back to zero and leaves what the launch found.
template <typename Space> __device__ __forceinline__ void outliers_done(Space *sp) {
  const unsigned long long pack =
      __hip_atomic_load(&sp->hdr.pack, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  sp->hdr.last_entries = static_cast<int>(pack >> 32);
  sp->hdr.last_parts = static_cast<int>(pack & 0xffffffffull);
  __hip_atomic_store(&sp->hdr.finished, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&sp->hdr.pack, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// a launch without outliers: what the caller may read about it (by one thread of the grid)
template <typename Space> __device__ __forceinline__ void no_outliers(Space *sp) {
  sp->hdr.last_entries = 0;
  sp->hdr.last_parts = 0;
}

// ---------------------------------------------------------------------------------------------
// The drawn end of the tile walk (emit option drawn_tail = N): the last N passes of a workgroup
// over the tile space are not dealt out by the stride; the workgroups of an XCD draw them from a
// ticket counter of that XCD (one cache line each), so that a workgroup whose tiles were cheap
// takes over from one whose tiles were dear.  It pays together with a tile order that puts the
// cheap tiles last (a model of a thousand small features, five tiles per workgroup: 70.2 ->
// 67.8 us; alone, or on a model of 100 features with ten tiles per workgroup, nothing).  One
// thread draws, the next ticket is requested before the current tile runs, the workgroup agrees
// through LDS.
//
// Who puts a counter back to zero for the next launch: every workgroup draws until a ticket lies
// beyond the last tile, and exactly one of its tickets does.  A counter that W workgroups share
// over N tiles therefore hands out the tickets 0 .. N + W - 1 and no others, and whoever holds
// N + W - 1 knows that nobody draws any more.  (A counter of finished workgroups told the same
// before: one device-scope add per workgroup to a single address, 11 ns each one after the
// other, 14 us for 1 280 workgroups -- most of a small batch's kernel: 100 features, 8 samples
// 22.7 us with it, 11.1 us without.  A full batch does not show it: its workgroups end at different
// times, 2 048 samples 121.9 and 121.3 us.)
// ---------------------------------------------------------------------------------------------
struct TailTickets {
  int next[8][32];                           // per XCD, each on a cache line of its own
};

__device__ __forceinline__ int draw_tail_ticket(TailTickets *t, const int xcd) {
  return __hip_atomic_fetch_add(&t->next[xcd][0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the tickets as one workgroup sees them: it draws from one counter only
struct TailDraw {
  TailTickets *tickets;
  int counter;
};

__device__ __forceinline__ int draw_tail_ticket(const TailDraw &d, const int xcd) {
  return draw_tail_ticket(d.tickets, xcd);
}

// by one thread of the workgroup that holds the last ticket of its counter
__device__ __forceinline__ void tail_tickets_done(const TailDraw &d) {
  __hip_atomic_store(&d.tickets->next[d.counter][0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

} // namespace rfx
