// Host-side check of rd::split_plan() (gpu_ragged_dot_amd/csrc/rd_sched.h), by which the host, the scheduling-map kernel and the gmm kernels
// each decide how a launch's last round is cut along K.  For every launch tried:
//   - what is cut is the last, partly filled round, and its pieces have a slot each and run at a time;
//   - no piece is shorter than the core asks for, and the pieces, cut at multiples of 64, cover the contraction;
//   - the caller's own number of pieces is the upper bound, and no slots cut nothing;
//   - halves of the columns are taken whenever all of them run at a time;
//   - by gain: what is cut gains more than it costs, and no other number of pieces more.
// Then the numbers of pieces at sizes on either side of the lines.  Built without GPU code by the library's Makefile; run by
// tests/test_host_checks.py.
#include <stdio.h>
#include "rd_sched.h"

static long long g_checked = 0;

static bool check(int live, const rd::SplitRule& r, int halves) {
  const rd::SplitPlan sp = rd::split_plan(live, r, halves);
  const int first = live / r.num_cus * r.num_cus, tiles = (live - first) * halves;
  auto fail = [&](const char* what) {
    fprintf(stderr, "live=%d k=%d k_cost=%d slots=%d cus=%d max_parts=%d by_gain=%d halves=%d: %s (first=%d parts=%d tiles=%d)\n", live, r.k, r.k_cost, r.slots,
            r.num_cus, r.max_parts, (int)r.by_gain, halves, what, sp.first_tile, sp.parts, sp.tiles);
    return false;
  };
  ++g_checked;
  if (sp.tiles == 0) {
    if (sp.first_tile != live || sp.parts != 1) return fail("uncut, but not from the end of the launch");
    if (halves == 2 && r.slots > 0 && tiles > 0 && tiles <= r.slots && tiles <= r.num_cus) return fail("halves that run at a time are not taken");
    return true;
  }
  if (r.slots <= 0) return fail("cut without slots");
  if (sp.first_tile != first || sp.tiles != tiles) return fail("not the last round");
  if (halves == 1 && sp.parts < 2) return fail("one piece");
  if (sp.parts < 1 || sp.parts > rd::kMaxSplitParts || sp.tiles * sp.parts > r.slots || sp.tiles > r.num_cus) return fail("more pieces than slots");
  if (sp.parts > 1 && r.k / sp.parts < r.min_k) return fail("pieces too short");
  if (r.max_parts > 0 && sp.parts > r.max_parts) return fail("more pieces than asked for");
  const int k64 = (r.k + 63) >> 6;
  int at = 0;
  for (int p = 0; p < sp.parts; ++p) {  // as gmm_kernel() cuts them
    const int k0 = (int)((long long)k64 * p / sp.parts) << 6, end = (int)((long long)k64 * (p + 1) / sp.parts) << 6;
    const int len = (r.k < end ? r.k : end) - k0;
    if (k0 != at || len <= 0) return fail("pieces do not follow one another");
    at = k0 + len;
  }
  if (at != r.k) return fail("pieces do not cover the contraction");
  if (r.by_gain && r.max_parts == 0 && sp.parts > 1) {
    auto gain = [&](int p) { return r.k_cost - r.k_cost / p - p * (100 + 7 * sp.tiles) - (first == 0 ? -200 : 400); };
    if (gain(sp.parts) <= 0) return fail("a cut that does not pay");
    for (int p = 2; p <= rd::kMaxSplitParts && sp.tiles * p <= r.slots && r.k / p >= r.min_k; ++p)
      if (gain(p) > gain(sp.parts)) return fail("another number of pieces pays more");
  }
  return true;
}

int main() {
  for (int cus : {256, 240})
    for (int live = 1; live < 3 * cus; live += live < 40 ? 1 : 7)
      for (int k = 8; k < 40000; k += k < 8000 ? 136 : 1500)
        for (int quarters : {2, 4, 24})
          for (int max_parts : {0, 1, 2, 3, 8, 100})
            for (int slots : {0, 256})
              for (bool by_gain : {false, true})
                for (int halves : {1, 2})
                  if (!check(live, rd::SplitRule{k, (int)((long long)k * quarters / 4), quarters == 24 ? 256 : 512, slots, cus, max_parts, by_gain}, halves)) return 1;
  // tiles, contraction, pieces: the 256 x 256 cores' launches of one round, and of more
  const struct { int live, k, parts; } want[] = {{10, 1023, 1}, {10, 1024, 2}, {10, 2048, 3}, {10, 3000, 4}, {10, 6000, 6}, {50, 1400, 1}, {50, 1536, 2}, {110, 3080, 1}, {110, 3084, 2}, {128, 4096, 2}, {129, 4096, 1},
                                                 {256 + 10, 1480, 1}, {256 + 10, 1484, 2}, {256 + 10, 3000, 4}, {256 + 90, 2800, 1}, {256 + 90, 3800, 2}, {256, 9000, 1}, {512 + 110, 5600, 2}};
  for (const auto& w : want) {
    const int got = rd::split_plan(w.live, rd::SplitRule{w.k, w.k, 512, 256, 256, 0, true}).parts;
    if (got != w.parts) { fprintf(stderr, "live=%d k=%d: %d pieces, not %d\n", w.live, w.k, got, w.parts); return 1; }
  }
  // by the square root: none below four, from k_cost 6400 on
  if (rd::split_plan(10, rd::SplitRule{6399, 6399, 512, 256, 256, 0, false}).parts != 1 || rd::split_plan(10, rd::SplitRule{6400, 6400, 512, 256, 256, 0, false}).parts != 4) return 1;
  printf("split_rule ok %lld\n", g_checked);
  return 0;
}
