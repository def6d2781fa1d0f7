// The scratch of short full-attention calls: no larger than the cache it serves, never a reason to refuse an engine or a call, and
// which kernel serves a call where it is missing or too small.
#include "gqa_plan.h"
#include "fake_hip.h"

using ha::gqa_rows_bytes;

static ha::GqaArgs args(int B, int HK, int P, int L, int LT, size_t rows, size_t marks) {
  ha::GqaArgs a{};
  a.B = B; a.HK = HK; a.HQ = 4 * HK; a.HD = 256; a.RD = 64; a.stride = 5120; a.LT = LT; a.P = P; a.L = L; a.dtype = 1;
  a.rows = &a; a.row_marks = (unsigned*)&a; a.rows_bytes = rows; a.marks_bytes = marks;
  return a;
}

int main() {
  const size_t big = ~(size_t)0;
  for (int pairs : {1, 2, 4, 8, 16, 32, 64})
    for (int ctx : {64, 4096, 32768, 262144, 1 << 20})
      CHECK(gqa_rows_bytes(pairs, ctx) <= std::max((size_t)64 << 20, (size_t)pairs * ctx * 256 * 4));
  // every short call on any context of up to 2048 positions fits, and a decode step on any context
  for (int B : {1, 2, 8, 16})
    for (int ctx : {2048, 4096, 32768}) {
      const size_t n = gqa_rows_bytes(2 * B, ctx), m = ha::gqa_rows_marks(2 * B, ctx) * 4;
      const int L = ha::gqa_rows_max(2 * B);
      CHECK(ha::gqa_rows_takes(args(B, 2, 2048 - L, L, ctx, n, m)) && ha::gqa_rows_takes(args(B, 2, ctx - 1, 1, ctx, n, m)));
    }
  // the launch's limits are known before it: 32-bit offsets of maxima and of rows, scratch, rows, context
  CHECK(ha::gqa_rows_takes(args(2, 16, 0, 64, 1 << 20, big, big)));
  CHECK(!ha::gqa_rows_takes(args(2, 16, (1 << 22) - 64, 64, 1 << 22, big, big)));
  ha::GqaArgs a = args(1, 2, 0, 64, 4096, big, big);
  a.stride = 1 << 25;
  CHECK(!ha::gqa_rows_takes(a));
  CHECK(!ha::gqa_rows_takes(args(1, 2, 0, 257, 4096, big, big)) && ha::gqa_rows_takes(args(1, 2, 0, 256, 4096, big, big)));
  CHECK(!ha::gqa_rows_takes(args(1, 2, 4000, 97, 4096, big, big)));
  const ha::gqa_rows::RowsLayout r = ha::gqa_rows::rows_layout(args(1, 2, 1000, 100, 4096, 0, 0));
  const size_t need = (size_t)r.units * ha::gqa_rows::kUnitBytes, marks = (size_t)2 * r.ngrp * r.nt * 4;
  CHECK(ha::gqa_rows_takes(args(1, 2, 1000, 100, 4096, need, marks)));
  CHECK(!ha::gqa_rows_takes(args(1, 2, 1000, 100, 4096, need - 1, marks)) && !ha::gqa_rows_takes(args(1, 2, 1000, 100, 4096, need, marks - 1)));

  // an engine is made where its caches fit and the scratch does not; its short calls then run the general kernel
  const unsigned char kinds[1] = {HA_FULL_ATTENTION};
  const ha_config c = config(kinds, 1, 1, 4096);
  static char in[64], out[64];
  const void* ins[1] = {in};
  void* outs[1] = {out};
  ha_engine *e = nullptr, *f = nullptr;
  limit = gqa_rows_bytes(2, 4096) - 1;  // (21 MiB; the cache is 8)
  CHECK(ha_create(&c, 0, &e) == HA_OK);
  CHECK(ha_forward(e, 64, ins, outs, nullptr, nullptr, nullptr) == HA_OK && calls.back() == "gqa");
  // joining another engine's set, and leaving it, likewise
  limit = ~(size_t)0;
  CHECK(ha_create(&c, 0, &f) == HA_OK);
  CHECK(ha_forward(f, 64, ins, outs, nullptr, nullptr, nullptr) == HA_OK && calls.back() == "gqa_rows");
  void* st = nullptr;
  CHECK(ha_get_stream(f, &st) == HA_OK && ha_set_stream(e, st) == HA_OK);
  limit = gqa_rows_bytes(2, 4096) - 1;
  CHECK(ha_share_scratch(e, f) == HA_OK);
  CHECK(ha_forward(e, 64, ins, outs, nullptr, nullptr, nullptr) == HA_OK && calls.back() == "gqa_rows");
  CHECK(ha_set_stream(e, nullptr) == HA_OK);
  CHECK(ha_forward(e, 64, ins, outs, nullptr, nullptr, nullptr) == HA_OK && calls.back() == "gqa");
  CHECK(ha_destroy(e) == HA_OK && ha_destroy(f) == HA_OK);
  printf("%d failures\n", fails);
  return fails != 0;
}
