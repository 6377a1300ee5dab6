// The sizes the run-time binding cuts a batch into (recflex_amd/csrc/include/rfx_tile_sizes.h: the
// functions the device code runs), and around them the binding of a model of up to 16 features with
// its 64 candidates one after the other.
#include "rfx_tile_sizes.h"

struct Rcp {
  static float rcp(const float x) { return 1.f / x; }
};

extern "C" {

int model_auto_tile_size(long long total, int grid) { return rfx::auto_tile_size(total, grid); }
int model_capped_tile_size(int built, long long total, int grid) { return rfx::capped_tile_size(built, total, grid); }

// tiles[f], longest tile and rounds at part size `unit`; the features' tiles with whole bags come
// from the binding's rule for schedules of one bag per workgroup pass (gran -1) or `gran` of them
static void apply(int F, int B, int grid, int tile_size, const float *cost, const int *gran, float unit,
                  int *tiles, float *longest) {
  *longest = 0.f;
  for (int f = 0; f < F; ++f) {
    const float bag = cost[f] * (1.f / static_cast<float>(B));
    const int parts = gran[f] == rfx::kSplitGran
        ? static_cast<int>(rfx::parts_of_bag(bag, 1.f / unit, rfx::split_parts_most(B))) : 1;
    float tile = 0.f;
    if (parts > 1) {
      tiles[f] = B * parts;
      tile = bag / static_cast<float>(parts);
    } else {
      const int g = gran[f] == rfx::kSplitGran ? 1 : gran[f];
      const float want = __builtin_ceilf(cost[f] * (1.f / static_cast<float>(tile_size)));
      int t = want < 1.f ? 1 : (want > static_cast<float>(B) ? B : static_cast<int>(want));
      int bpt = (B + t - 1) / t;
      const int whole = (bpt + g - 1) / g * g;
      const int need = (2 * grid + F - 1) / F;
      if (bpt >= g || B >= g * need || static_cast<float>(whole) * bag <= 8.f * static_cast<float>(tile_size)) bpt = whole;
      tiles[f] = (B + bpt - 1) / bpt;
      tile = static_cast<float>(bpt) * bag;
    }
    if (tile > *longest) *longest = tile;
  }
}

// out: {part size chosen, tiles it was counted with (-1: no search), the rule's part size}; tiles[f]
// and longest as they are bound, rule_tiles / rule_longest as the rule alone would
void model_bind(int F, int B, int grid, int tile_size, const float *cost, const int *gran, int *tiles,
                float *longest, int *rule_tiles, float *rule_longest, long long *out) {
  float total = 0.f;
  for (int f = 0; f < F; ++f) total += cost[f];
  long long unit = rfx::split_unit_rule(static_cast<long long>(total), grid, tile_size);
  out[1] = -1;
  out[2] = unit;
  apply(F, B, grid, tile_size, cost, gran, static_cast<float>(unit), rule_tiles, rule_longest);
  if (F <= rfx::kSplitSearchFeats && rfx::search_is_due(static_cast<long long>(total), grid, tile_size)) {
    int whole[rfx::kSplitSearchFeats];
    float ignored, best = 0.f;
    apply(F, B, grid, tile_size, cost, gran, 3e38f, whole, &ignored);        // no bag is worth splitting
    const int rule = static_cast<int>(unit);
    for (int lane = 0; lane < 64; ++lane) {
      const int candidate = rfx::split_unit_candidate<Rcp>(lane, total, grid, rule);
      rfx::SplitTally tally;
      for (int f = 0; f < F; ++f) {
        const float bag = cost[f] * (1.f / static_cast<float>(B));
        const int bpt = (B + whole[f] - 1) / whole[f];
        tally.add<Rcp>(gran[f] == rfx::kSplitGran ? bag : 0.f, whole[f], static_cast<float>(bpt) * bag, B,
                       1.f / static_cast<float>(candidate), rfx::split_parts_most(B));
      }
      const float price = tally.price(candidate, tile_size, grid);
      if (lane == 0 || price < best) {
        best = price;
        unit = candidate;
        out[1] = tally.tiles;
      }
    }
  }
  out[0] = unit;
  apply(F, B, grid, tile_size, cost, gran, static_cast<float>(unit), tiles, longest);
}

} // extern "C"
