// Rows of B left-padded prompts of T columns without the padding (tnx_packed_rows): position t of prompt b, t >= starts[b], is row base[b] + t of
// every activation; caches, ids and positions stay [B, T].  base null: row b T + t, no padding left out.
#pragma once
#include "common.h"

namespace {
struct PackedRows {
  const int32_t* base;
  const int32_t* starts;
  int64_t rows;   // of all prompts together
};
constexpr PackedRows kAllRows{nullptr, nullptr, 0};

inline int packed_args(const tnx_packed_rows* p, int64_t B, int64_t T, PackedRows& out) {
  TNX_REQUIRE(p && p->row_base && p->starts, "packed rows: null pointer");
  TNX_REQUIRE(p->rows > 0 && p->rows <= B * T, "packed rows: %lld rows of %lld prompts of %lld", (long long)p->rows, (long long)B, (long long)T);
  out = PackedRows{p->row_base, p->starts, p->rows};
  return TNX_OK;
}
}  // namespace
