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
      CHECK(gqa_rows_bytes(pairs, ctx, pairs <= 2, false) <= std::max((size_t)24 << 20, (size_t)pairs * ctx * 256 * 5));
  // every call that the short-call kernels are expected to be the faster for fits the engine's scratch
  for (int f16 = 0; f16 < 2; f16++)
   for (int B : {1, 2, 3, 5, 8, 16})
    for (int ctx : {64, 2048, 4096, 32768, 131072}) {
      const size_t n = gqa_rows_bytes(2 * B, ctx, B == 1, !f16), m = ha::gqa_rows_marks(2 * B, ctx) * 4;
      for (int L = 1; L <= ha::gqa_rows_max(2 * B) && L <= ctx; L++)
        for (int P = 0; P + L <= ctx; P += 63 + (P >> 5)) {
          ha::GqaArgs x = args(B, 2, P, L, ctx, n, m);
          x.dtype = f16;
          x.split = B == 1 ? std::max(8, (ctx / 64 + 7) / 8) : 0;
          if (ha::gqa_rows_faster(x)) CHECK(ha::gqa_rows_takes(x));
        }
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

  // calls of many pairs, rows and tiles are the general kernel's: lines between measured cases on either side
  auto faster = [&](int B, int P, int L, int split) {
    ha::GqaArgs x = args(B, 2, P, L, 1 << 20, big, big);
    x.split = split;
    return ha::gqa_rows_faster(x);
  };
  CHECK(faster(8, 12000, 1, 0) && faster(8, 48000, 1, 0) && faster(8, 24000, 64, 0) && !faster(8, 64000, 64, 0));
  CHECK(faster(8, 1500, 128, 0) && !faster(8, 12000, 128, 0) && faster(16, 12000, 1, 0) && !faster(16, 12000, 32, 0) && !faster(16, 24000, 1, 0));
  CHECK(faster(16, 1500, 64, 0) && !faster(16, 6000, 64, 0) && faster(2, 96000, 128, 0) && faster(3, 48000, 128, 0));
  CHECK(faster(1, 48000, 1, 100) && !faster(1, 96000, 64, 200) && faster(1, 12000, 128, 25) && !faster(1, 24000, 128, 50));
  auto faster32 = [&](int B, int P, int L, int split) {
    ha::GqaArgs x = args(B, 2, P, L, 1 << 20, big, big);
    x.split = split; x.dtype = 0;
    return ha::gqa_rows_faster(x);
  };
  CHECK(faster32(8, 3000, 64, 0) && !faster32(8, 3000, 96, 0) && !faster32(16, 3000, 32, 0) && faster32(16, 3000, 1, 0));
  CHECK(!faster32(8, 0, 32, 0) && faster32(8, 300, 32, 0) && !faster32(1, 0, 16, 8) && faster32(1, 300, 16, 8));
  CHECK(faster32(1, 3000, 128, 8) && !faster32(1, 12000, 128, 25) && !faster32(1, 3000, 256, 8) && faster32(1, 300, 256, 8));
  CHECK(faster(1, 1500, 256, 8) && faster(1, 3000, 256, 8) && !faster(1, 6000, 256, 13) && !faster(1, 6000, 192, 13));

  // an engine is made where its caches fit and the scratch does not; its short calls then run the general kernel
  const unsigned char kinds[1] = {HA_FULL_ATTENTION};
  const ha_config c = config(kinds, 1, 1, 4096);
  static char in[64], out[64];
  const void* ins[1] = {in};
  void* outs[1] = {out};
  ha_engine *e = nullptr, *f = nullptr;
  limit = gqa_rows_bytes(2, 4096, true, false) - 1;  // (18 MB; the cache is 8)
  CHECK(ha_create(&c, 0, &e) == HA_OK);
  CHECK(ha_forward(e, 64, ins, outs, nullptr, nullptr, nullptr) == HA_OK && calls.back() == "gqa");
  // joining another engine's set, and leaving it, likewise
  limit = ~(size_t)0;
  CHECK(ha_create(&c, 0, &f) == HA_OK);
  CHECK(ha_forward(f, 64, ins, outs, nullptr, nullptr, nullptr) == HA_OK && calls.back() == "gqa_rows");
  void* st = nullptr;
  CHECK(ha_get_stream(f, &st) == HA_OK && ha_set_stream(e, st) == HA_OK);
  limit = gqa_rows_bytes(2, 4096, true, false) - 1;
  CHECK(ha_share_scratch(e, f) == HA_OK);
  CHECK(ha_forward(e, 64, ins, outs, nullptr, nullptr, nullptr) == HA_OK && calls.back() == "gqa_rows");
  CHECK(ha_set_stream(e, nullptr) == HA_OK);
  CHECK(ha_forward(e, 64, ins, outs, nullptr, nullptr, nullptr) == HA_OK && calls.back() == "gqa");
  CHECK(ha_destroy(e) == HA_OK && ha_destroy(f) == HA_OK);
  printf("%d failures\n", fails);
  return fails != 0;
}
