// A call that keeps a snapshot: no allocation in front of its launches, whichever memory the snapshot gets, and the snapshot holds
// the call's state and raw rows.
#include "fake_hip.h"

int main() {
  const unsigned char kinds[4] = {HA_LINEAR_ATTENTION, HA_ADAPTER, HA_LINEAR_ATTENTION, HA_FULL_ATTENTION};
  const ha_config c = config(kinds, 4, 1, 512);
  ha_engine* e = nullptr;
  CHECK(ha_create(&c, 0, &e) == HA_OK);
  static char in[64], out[64];
  const void* ins[4] = {in, in, in, in};
  void* outs[4] = {out, out, out, out};
  const size_t n = 16 * 128 * 128;
  std::vector<float> got(n);
  for (int timed = 0; timed < 2; timed++)
    for (int round = 0; round < 3; round++) {  // new memory, the block that snapshot gave back, untimed new memory again
      calls.clear(); state_out.clear();
      ha_forward_opts o;
      memset(&o, 0, sizeof o);
      o.timestamps = timed;
      ha_snapshot* s = nullptr;
      CHECK(ha_forward(e, 192, ins, outs, nullptr, &s, &o) == HA_OK && s);
      const bool fresh = where("malloc") >= 0;
      CHECK(fresh == (round == 0 || (round == 2 && !timed)));
      if (fresh && !timed) {  // behind the last mixer, in front of what needs the memory
        CHECK(where("malloc") > where("gqa_rows") && where("gqa_rows") >= 0 && where("malloc") < where("tails") && where("malloc") < where("copy2d"));
        CHECK(where("launch", where("malloc")) < 0);
      }
      if (fresh && timed) CHECK(where("malloc") < where("event"));  // the times hold no allocation
      if (!fresh) CHECK(where("copy") < 0);  // the layers wrote the snapshot's block themselves
      for (int k = 0; k < 2; k++) {
        CHECK(ha_snapshot_read(s, k ? 2 : 0, "state", got.data(), n * 4) == HA_OK);
        CHECK(got[0] == 300.0f + 1 + k && got[n - 1] == 300.0f + 1 + k);
        std::vector<char> tail(3 * 8256 * 4);
        CHECK(ha_snapshot_read(s, k ? 2 : 0, "tail", tail.data(), tail.size()) == HA_OK && tail[0] == 7);
      }
      if (round == 0 || timed) CHECK(ha_snapshot_destroy(s) == HA_OK);  // its block becomes the spare
    }
  // no memory: reported, nothing kept, and the next call runs
  const unsigned char one[1] = {HA_LINEAR_ATTENTION};
  const ha_config c1 = config(one, 1, 1, 512);
  ha_engine* f = nullptr;
  CHECK(ha_create(&c1, 0, &f) == HA_OK);
  limit = 1 << 20;
  ha_snapshot* s = nullptr;
  CHECK(ha_forward(f, 192, ins, outs, nullptr, &s, nullptr) == HA_ERR_NOMEM && !s);
  limit = ~(size_t)0;
  last_error = hipSuccess;
  CHECK(ha_forward(f, 192, ins, outs, nullptr, &s, nullptr) == HA_OK && s);
  CHECK(ha_snapshot_destroy(s) == HA_OK && ha_destroy(f) == HA_OK && ha_destroy(e) == HA_OK);
  printf("%d failures\n", fails);
  return fails != 0;
}
