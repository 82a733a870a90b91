// The block prefill's buffers and copies on the fake HIP runtime: a prompt of several
// blocks runs with the second set of rows on a second stream, without memory for them
// one block after the other on the decoder's stream, and a prompt that failed for lack
// of memory can be repeated.
#include "fake_hip.hpp"

#include <cstdio>
#include <vector>

#include "mtg_verify.h"

static int failures = 0;
static void expect(bool ok, const char* what, long a = 0, long b = 0) {
  if (ok) return;
  std::fprintf(stderr, "%s (%ld, %ld)\n", what, a, b);
  ++failures;
}

constexpr int kRows = 2048, kHidden = 1024;  // rows of a block, and floats of a row
static const mtg_hparams kHp{kHidden, 16, 8, 128, 3072, 1, 256, 1e6f, 1e-6f};

// One prompt: its status, and that the copies bring every row down and up once, in
// order, a block's hidden rows before anything overwrites them.
static void prompt(mtg_ctx* ctx, int S, bool want_hidden, bool two_streams) {
  std::vector<float> in((size_t)S * kHidden), out(want_hidden ? in.size() : 0);
  fake::State& f = fake::state();
  f.launches.clear();
  f.copies.clear();
  f.waits = f.stream_syncs = 0;
  expect(mtg_prefill(ctx, in.data(), S, want_hidden ? out.data() : nullptr) == MTG_OK, "prefill", S, two_streams);
  // one stream keeps its own order: no events to wait for, one wait for its end
  if (!two_streams) expect(f.waits == 0 && f.stream_syncs == 1, "waits on one stream", f.waits, f.stream_syncs);
  size_t up = 0, down = 0;
  void* compute = f.launches.empty() ? nullptr : f.launches[0].stream;
  std::map<const void*, size_t> rows_in;  // device buffer -> the end of what it was last filled with
  for (const fake::Copy& c : f.copies) {
    expect((c.stream != compute) == two_streams, "stream of a copy", S, two_streams);
    if (c.kind == 1) {
      expect(c.src == in.data() + up, "rows down in order", S);
      up += c.bytes / 4;
      if (rows_in.count(c.dst) && want_hidden && !two_streams) expect(down + c.bytes / 4 >= up, "rows of a block still in use", S);
      rows_in[c.dst] = up;
    } else {
      expect(c.dst == out.data() + down, "hidden rows up in order", S);
      down += c.bytes / 4;
      if (!two_streams) expect(down == up, "hidden rows before the next block", S);
    }
  }
  expect(up == in.size() && down == out.size(), "all rows", (long)up, (long)down);
  expect(rows_in.size() == (two_streams ? 2u : 1u), "row buffers", (long)rows_in.size(), two_streams);
  for (const fake::Launch& l : f.launches) expect(l.stream == compute, "stream of a launch", S);
}

int main() {
  const int types[] = {MTG_TYPE_Q8_0, MTG_TYPE_F16, MTG_TYPE_F32, MTG_TYPE_Q4_K};
  for (int type : types) {
    mtg_synth_model* synth = nullptr;
    expect(mtg_synth_create(&kHp, type, 3, 0.02f, 0.0f, &synth) == MTG_OK, "synthetic model", type);
    fake::State& f = fake::state();
    auto context = [&](int max_seq) {
      mtg_ctx* ctx = nullptr;
      expect(mtg_create(mtg_synth_desc(synth), max_seq, MTG_TYPE_F16, &ctx) == MTG_OK, "context", type);
      return ctx;
    };
    {
      mtg_ctx* ctx = context(5000);
      for (bool hidden : {true, false}) {
        prompt(ctx, 5000, hidden, true);
        prompt(ctx, kRows, hidden, false);
        prompt(ctx, kRows + 1, hidden, true);
      }
      mtg_destroy(ctx);
    }
    // no memory beyond the first set: from the first allocation after it on
    for (int set : {0, 1}) {  // 0: neither buffer of the second set, 1: only its first
      mtg_ctx* ctx = context(5000);
      prompt(ctx, 16, true, false);
      int given = 0;
      f.malloc_fails = [&](size_t) { return given++ >= set; };
      for (bool hidden : {true, false}) prompt(ctx, 5000, hidden, false);
      f.malloc_fails = nullptr;
      prompt(ctx, 5000, true, true);  // there is room again
      mtg_destroy(ctx);
    }
    // A prompt that fails at its allocation number `have` launches nothing, and its repeat
    // makes all the buffers that are missing, the failed one first.
    int total = 0;
    for (int have = -1; have < total; ++have) {  // -1: none fails, to count them
      mtg_ctx* ctx = context(64);
      std::vector<float> in((size_t)16 * kHidden);
      int asked = 0;
      f.malloc_fails = [&](size_t) { return asked++ == have; };
      f.launches.clear();
      const int rc = mtg_prefill(ctx, in.data(), 16, nullptr);
      if (have < 0) total = asked;
      expect(rc == (have < 0 ? MTG_OK : MTG_ERR_NOMEM), "prefill without allocation", have, rc);
      expect(have < 0 || f.launches.empty(), "launches without allocation", have);
      const int before = asked - (have >= 0);
      asked = -1000;  // none fails
      expect(mtg_prefill(ctx, in.data(), 16, nullptr) == MTG_OK, "prefill again", have);
      expect(before + asked + 1000 == total, "buffers after the repeat", before + asked + 1000, total);
      f.malloc_fails = nullptr;
      mtg_destroy(ctx);
    }
    expect(total >= 7, "prefill buffers", total);
    std::printf("weights %d: %d failures\n", type, failures);
    mtg_synth_free(synth);
  }
  std::printf("{\"record\": \"prefillBuffers\", \"failures\": %d}\n", failures);
  return failures ? 1 : 0;
}
