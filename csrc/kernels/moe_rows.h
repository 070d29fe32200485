// Weights of a routed (row, slot) pair, shared by the grouped expert kernels (moe.hip, moe_pipe.hip).
//
// By default a routed expert's weight multiplies its output.  weight_in moves it to the expert's input; the gate and up
// products are linear in it, so it multiplies their fp32 sums.  The shared expert's weight, when topk_w has a column for
// it, always multiplies its output.
#pragma once
#include "api_layers.h"
#include "common.h"

namespace dsse {
namespace {

constexpr int kMoeRows = 64;  // rows of one expert per tile of the work list (moe_align)

DEV float slot_weight(const MoeGroupedParams& p, int row, int k) {
  return k < p.ldw ? p.topk_w[(int64_t)row * p.ldw + k] : 1.0f;
}
DEV float out_weight(const MoeGroupedParams& p, int row, int k) {
  return p.weight_in && k < p.top ? 1.0f : slot_weight(p, row, k);
}
DEV float in_weight(const MoeGroupedParams& p, int id) {
  if (!p.weight_in) return 1.0f;
  const int row = id / p.S, k = id - row * p.S;
  return k < p.top ? slot_weight(p, row, k) : 1.0f;
}

}  // namespace
}  // namespace dsse
