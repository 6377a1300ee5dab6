// The sizes that the run-time binding cuts a batch into: the traffic of a tile, and the parts of bags
// that several workgroups share.  Arithmetic only, for the device (rfx_binding.hip.h) and for the CPU.
#pragma once

#if defined(__HIPCC__)
#define RFX_SIZES_FN __host__ __device__ __forceinline__
#else
#define RFX_SIZES_FN inline
#endif

namespace rfx {

// Automatic tile size (tile_bytes <= 0): the batch's traffic divided by kAutoTilesPerWorkgroup
// tiles for each workgroup of the grid, within [kAutoTileMin, kAutoTileMax], in steps of 4 KiB.
// Small batches keep 64 KiB tiles; a batch of tens of GB with bags of hundreds of wide rows gets
// 256 KiB, several bags per tile instead of one (measured on the 400-feature fp16 model with its
// default schedules: 7.1 ms with 64 KiB tiles, 5.0 ms with 256 KiB).
// A batch too small for that (less than kAutoTileMin of traffic per workgroup of the grid) gets
// about two tiles per workgroup instead, down to kAutoTileFloor: its launch is a matter of
// latencies -- every pass of a workgroup over a tile is a chain of dependent round trips to
// memory -- so the passes are spread over all workgroups as evenly as their number allows
// (measured on 26 features x 4 096 one-lookup bags, 1 024 workgroups: 9.0 us with 54 KiB tiles
// of two passes each, 8.3 us with 32 KiB tiles of one).
constexpr int kAutoTilesPerWorkgroup = 64;
constexpr int kAutoTileMin = 64 * 1024;
constexpr int kAutoTileMax = 256 * 1024;
constexpr int kAutoTileFloor = 4 * 1024;

RFX_SIZES_FN int auto_tile_size(const long long total, const int grid_blocks) {
  const long long grid = grid_blocks > 0 ? grid_blocks : 1;
  long long t = total / (grid * kAutoTilesPerWorkgroup);
  if (t >= kAutoTileMin) return static_cast<int>(t > kAutoTileMax ? kAutoTileMax : t) & ~4095;
  t = total / (2 * grid);
  t = t < kAutoTileFloor ? kAutoTileFloor : (t > kAutoTileMin ? kAutoTileMin : t);
  return static_cast<int>(t) & ~1023;
}

// The tile size of a library that was built with one beyond kAutoTileMin (tile_bytes = -size): it was
// chosen on full batches, and a batch of less than kCappedTilesPerWorkgroup such tiles per workgroup
// gets smaller ones, so that its end is not a matter of whole tiles, down to kAutoTileMin.  (Below that
// tiles come apart into less than a workgroup's pass and teams idle: 400 fp16 features, 16 samples, 43
// us with 64 KiB, 61 with 32.  A size of 64 KiB or less stays: cut in half it gave 100 and 1 000
// features 3 % at some batches and cost 3 % at others.)  Measured, in us, with the size as built and
// this one: 200 int8 features (128 KiB) 64 / 300 / 1 000 samples 24.5 / 66.6 / 138 and 20.8 / 55.4 /
// 133; 400 fp16 features (256 KiB) 4 / 16 / 64 samples 39.3 / 51.0 / 105 and 36.5 / 47.6 / 100.
constexpr int kCappedTilesPerWorkgroup = 5;

RFX_SIZES_FN int capped_tile_size(const int built, const long long total, const int grid_blocks) {
  const long long t = total / ((grid_blocks > 0 ? grid_blocks : 1) * static_cast<long long>(kCappedTilesPerWorkgroup));
  if (t >= built || kAutoTileMin >= built) return built;
  return t > kAutoTileMin ? static_cast<int>(t) & ~1023 : kAutoTileMin;
}

// Schedules that split a bag over several workgroups (rfx::split_bags) announce themselves with
// a granularity of kSplitGran.  A bag is worth splitting when it alone would keep its workgroup
// busy for a good part of the kernel: the unit is a quarter of a workgroup's fair share of the
// batch's traffic (total / grid), at least one tile and kSplitMinUnit; when the mean bag of such a feature
// carries more than 1.25 units, the feature gets batch * parts tiles, parts = bag / unit, tile t
// being part t % parts of bag t / parts, and bags_per_tile holds -parts.  (A part costs some
// 6 us of dependent memory round trips besides its rows, and with two to five tiles per
// workgroup the time moves in steps of whole tiles: a unit of half a share gave 150 / 162 /
// 161 us where a quarter gives 177 / 109 / 160 us on 16 x 20 000, 64 x 4 000 and 128 x 2 500
// lookups; the finer one is kept, it also evens out bags of unequal length.)
// Always parts <= kBindMaxParts and batch * parts <= kBindMaxSplitTiles (the slots of the feature's
// workspace region).  Otherwise -- many bags, or a small grid -- the feature is bound like any
// other with one bag per workgroup pass.  (Measured on 8 features of 16 bags of 20 000 lookups:
// 968 us unsplit, 177 us split; 64 bags of 4 000: 204 and 109 us; 512 bags of 1 000 stay
// unsplit at 185 us.)
// Smallest part: 256 KiB of traffic (with 128 KiB parts the three shapes above take 175 / 108 /
// 161 us at four workgroups per CU, with 256 KiB parts 142 / 103 / 122 us; at eight workgroups
// per CU, which these light kernels allow, 138 / 76 / 83 us and 107 / 83 / 96 us.  All of these with a
// branch around every row load; without it a part's rows come faster, its round trips stay:
// block_sum_range).
constexpr int kSplitMinUnit = 256 * 1024;
// ... unless the batch is so small that parts of that size leave the workgroups with one or two
// tiles each: then the part size is chosen so that the tiles come out as a whole number per
// workgroup, down to kSplitFloorUnit (16 x 20 000 lookups on 2 048 workgroups: 2 880 parts of
// 256 KiB are 1.4 tiles per workgroup, i.e. two rounds with the second a third full, 94 us;
// 3 872 parts of 199 KiB are 1.9, 88 us).
constexpr int kSplitFloorUnit = 128 * 1024;
// Models of up to kSplitSearchFeats features go by more than that rule: they count the tiles that a part
// size would give, the rule's among 64 of them, and take the size whose rounds of the grid, each as
// long as the longest tile, are over first.  (16 x 20 000 lookups, 2 048 workgroups, in us: 3 712
// parts of 200 KiB 85, 2 176 of 340 KiB 104, 1 984 of 384 KiB 74, 1 696 of 440 KiB 80; 128 x 2 500:
// 2 304 tiles 99, 2 048 of them 77.)  Counting takes a few instructions per feature in every
// workgroup, hence the limit.
constexpr int kSplitSearchFeats = 16;
constexpr int kSplitPartCost = 35 * 1024;      // a part's round trips, in traffic
constexpr int kSplitGran = -1;
constexpr int kBindMaxParts = 64;
constexpr int kBindMaxSplitTiles = 2048;

// Parts a bag of bag_cost bytes (the feature's mean) is cut into at part size 1 / inv_unit; 1: left
// whole.  A bag is split from 1.25 units on (128 x 2 500 lookups: 102.8 us with bags of 1.7 units left
// whole beside split ones, 89.3 us with those in two parts).  most: split_parts_most of the batch.
RFX_SIZES_FN float parts_of_bag(const float bag_cost, const float inv_unit, const float most) {
  const float units = bag_cost * inv_unit;
  return units > 1.25f ? __builtin_fmaxf(__builtin_fminf(__builtin_ceilf(units), most), 1.f) : 1.f;
}
// the most parts a bag may have in a batch of this size
RFX_SIZES_FN float split_parts_most(const int batch) {
  const int slots = kBindMaxSplitTiles / (batch > 0 ? batch : 1);
  return static_cast<float>(slots < kBindMaxParts ? slots : kBindMaxParts);
}

// The part size that follows from the batch's traffic alone: see kSplitMinUnit and kSplitFloorUnit.
RFX_SIZES_FN long long split_unit_rule(const long long total, const int grid, const int tile_size) {
  long long unit = total / (4ll * grid);
  if (unit < tile_size) unit = tile_size;
  if (unit < kSplitMinUnit) {
    // whole tiles per workgroup at about the minimum part size, and 6 % of slack for the
    // rounding up of every feature's parts per bag
    const long long share = static_cast<long long>(grid) * kSplitMinUnit;
    const long long per_workgroup = (total + share - 1) / share;
    unit = total / (grid * (per_workgroup > 0 ? per_workgroup : 1));
    unit += unit >> 4;
    if (unit > kSplitMinUnit) unit = kSplitMinUnit;
    if (unit < kSplitFloorUnit) unit = kSplitFloorUnit;
    if (unit < tile_size) unit = tile_size;
  }
  return unit;
}
// Whether other sizes are looked at: not where a quarter of a workgroup's share, or a tile, is
// kSplitMinUnit already, nor where one round of parts of that size or less is what the rule gives by itself.
RFX_SIZES_FN bool search_is_due(const long long total, const int grid, const int tile_size) {
  return total > static_cast<long long>(grid) * kSplitMinUnit && total / (4ll * grid) < kSplitMinUnit &&
         tile_size < kSplitMinUnit;
}

// The part size that lane 0 .. 63 looks at: a workgroup's share of the batch in 1 to 4 rounds, enlarged
// by 0 to 15 sixteenths -- and the rule's, so that nothing is chosen that is dearer by the same count
// (8 features of 878 bags of 600 / 900 lookups, 2 048 workgroups: 128.6 / 186.8 us where any size that
// filled one to four rounds was taken, 116.7 / 168.8 us where the rule's more and shorter rounds count).
// A whole number, since what is counted with it has to be what the tiles are made with, and beyond the
// share by at least one byte, more than the figures' rounding errors of a few 2^-24 come to at shares
// of up to 1 MiB: bags of equal cost come out at the number of parts that fills the round, not at one
// more (8 features of 16 x 20 000 lookups, dim 64: 2 048 tiles on 2 048 workgroups, 63.7 us, where a size
// cut off to the byte below made 2 176, two rounds, 86.4 us; 4 of dim 128 64.3 and 86.3, 16 of dim 64
// 127.1 and 170.5).
template <typename M>
RFX_SIZES_FN int split_unit_candidate(const int lane, const float total, const int grid, const int rule) {
  if (lane == 63) return rule;
  const float share = total * M::rcp(static_cast<float>(1 + (lane >> 4)) * static_cast<float>(grid));
  return static_cast<int>(share * (1.f + 0.0625f * static_cast<float>(lane & 15))) + 2;
}

// What a part size comes to, feature by feature.
struct SplitTally {
  int tiles = 0;
  float longest = 0.f;                          // traffic of the longest tile

  // bag: mean traffic of one of the feature's bags (0: its schedule does not split); whole_tiles and
  // whole_tile: its tiles with the bags left whole, and the traffic of one
  template <typename M>
  RFX_SIZES_FN void add(const float bag, const int whole_tiles, const float whole_tile, const int batch,
                        const float inv_unit, const float most) {
    const float parts = parts_of_bag(bag, inv_unit, most);
    const bool split = parts > 1.f;
    tiles += split ? batch * static_cast<int>(parts) : whole_tiles;
    longest = __builtin_fmaxf(longest, split ? bag * M::rcp(parts) : whole_tile);
  }
  RFX_SIZES_FN float price(const int unit, const int tile_size, const int grid) const {
    if (unit < kSplitFloorUnit || unit < tile_size) return 3.4e38f;
    const int rounds = (tiles + grid - 1) / grid;
    return static_cast<float>(rounds) * (longest + static_cast<float>(kSplitPartCost));
  }
};

} // namespace rfx
