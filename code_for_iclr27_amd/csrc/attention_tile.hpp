// Prefill attention on tiles of query rows (attention_tile.hip): its plan, partial-state bytes, launch.
#pragma once

#include "attention_common.hpp"

namespace lr {

struct AttnTilePlan {
  int64_t segments, rows, tiles, splits, chunk;  // rows of a tile, keys of one split
  double us;  // the estimate it was chosen by (bf16, launches not counted)
};

// `scratch_bytes` bounds the partial states of a call that splits its keys.
AttnTilePlan plan_attention_tiles(int64_t segments, int64_t groups, int64_t length,
                                  int64_t max_keys, int64_t dim, int64_t scratch_bytes);
size_t attention_tiles_bytes(const AttnTilePlan& plan, int64_t dim);
// args.tiles, splits and the partial-state pointers follow the plan.
int launch_attention_tiles(const AttnArgs& args, const AttnTilePlan& plan, int64_t dim, int dtype,
                           hipStream_t stream);

}  // namespace lr
