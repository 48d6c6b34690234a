// Mixture of experts: every row uses ``top`` of ``experts`` feed-forwards.
//
//   route    router logits -> chosen experts and their weights, per (row, choice) pair
//   group    pairs sorted by expert and cut into tiles of at most tile_rows pairs of one expert
//   up       act[i] = silu(gate . h) * (up . h), or relu(up . h)^2, of sorted pair i
//   down     y[i] = down . act[i]
//   (join    the weighted sum over a row's pairs joins the stream: stream_ops.hip)
#pragma once
#include "elem.h"

struct MoeTile {  // pairs [start, start + count) of the sorted list, all of one expert; expert < 0: none (after all others)
  int expert, start, count, used;  // used: how many of the table's tiles there are, in each of them; from MOE_HEIGHT on: MoePick
};
constexpr int MOE_HEIGHT = 24;

// Tiles of the height, of these four, whose rounds on 256 CUs take least in both products, chosen when the experts' pairs are
// counted. nt: columns of tiles of a product; step, own: us of a round's K steps, of its start and end. nt[0] = 0: the height is given.
// Mirrored by llm_sharding_amd/ops/moe.py::Pick.
constexpr int MOE_ROWS[4] = {128, 192, 256, 320};
struct MoePick {
  int nt[2];
  float step[4][2], own[4];
};

// How experts are chosen. Mirrored by llm_sharding_amd/ops/moe.py::RouteArgs.
struct RouteArgs {
  const float* correction;  // [experts] added to a score when choosing, or null
  int sigmoid;              // 0: scores are the logits, weights the softmax over the chosen ones; 1: scores are their
                            // sigmoids, weights those over their sum, times scale
  int groups, keep;         // the keep best of groups equal groups of neighbours can be chosen from (sum of the
                            // two largest choice scores)
  float scale;
};

enum MoeUp { MOE_DOWN = 0, MOE_GLU = 1, MOE_RELU2 = 2 };  // what a product is: down, or up of which kind
