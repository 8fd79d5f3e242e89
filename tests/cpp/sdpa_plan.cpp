// Sweeps the packed attention's host plan (csrc/sdq_sdpa_plan.h): every launch
// of a call must lie inside the scratch that is asked for the call, that
// scratch inside 2 GiB (and its records' exponents), and every item's keys must
// be covered once. Prints the first call that breaks a rule. With an argument:
// prints one call's cut.
#include <cmath>
#include <cstdio>
#include <random>

#include "sdq_sdpa_plan.h"

namespace sd = sdq::sdpa;

namespace {

bool check(int64_t Lq, int64_t Lk, int heads, int batch, int cus) {
  if (const int S = sd::few_splits(Lq, Lk, heads, cus); S > 1) {
    const int64_t nkb = sd::div_up(Lk, sd::kKB), b = sd::few_scratch(Lq, heads, S, batch);
    if (S > 32 || sd::div_up(nkb, sd::div_up(nkb, S)) != S || b > sd::kMaxScratch ||
        (b && b < sd::few_bytes(Lq, heads, S))) {
      std::printf("few queries: Lq=%lld Lk=%lld heads=%d: %d ranges, %lld bytes\n", (long long)Lq,
                  (long long)Lk, heads, S, (long long)b);
      return false;
    }
  }
  const int64_t have = sd::scratch_bytes(Lq, Lk, heads, batch, cus);
  if (have == 0) return true;
  auto bad = [&](const char* what, int64_t a, int64_t b) {
    std::printf("Lq=%lld Lk=%lld heads=%d batch=%d cus=%d: %s (%lld, %lld)\n", (long long)Lq,
                (long long)Lk, heads, batch, cus, what, (long long)a, (long long)b);
    return false;
  };
  const sd::Chunk c = sd::chunk(Lq, Lk, heads, batch, cus);
  if (have > (int64_t(1) << 31) + (5 << 20)) return bad("more than 2 GiB", have, c.seqs);
  if (c.heads < 1 || c.seqs < 1) return bad("empty chunk", c.heads, c.seqs);
  if (c.heads < heads && c.seqs != 1) return bad("chunk of heads and sequences", c.heads, c.seqs);
  for (int h : {c.heads, heads % c.heads})
    for (int n : {c.seqs, batch % c.seqs}) {
      if (h == 0 || n == 0) continue;
      const sd::Plan p = sd::launch_plan(Lq, Lk, h, cus);
      const int64_t need = sd::layout(p, h, n).bytes;
      if (need > have) return bad("launch past the scratch (needs, has)", need, have);
      if (p.items != h * p.qgroups || p.nfull < 0 || p.nfull > p.items)
        return bad("items", p.items, p.nfull);
      if ((int64_t)p.splits * p.kbs < p.nkb || (int64_t)(p.splits - 1) * p.kbs >= p.nkb)
        return bad("shares (splits, blocks each)", p.splits, p.kbs);
    }
  return true;
}

}  // namespace

int main(int argc, char**) {
  if (argc > 1) {  // the cut of 157 queries x 768 keys x 24 heads
    const sd::Plan p = sd::launch_plan(157, 768, 24, 256);
    std::printf("%d shares of %d blocks\n", p.splits, p.kbs);
    return 0;
  }
  // shares' outputs beyond the records: 2.7, 3.0 and 49 GiB without a bound of
  // their own; then ragged last chunks of heads
  bool ok = check(27280, 1 << 20, 1, 1, 256) && check(1024, 1024, 24, 64, 256) &&
            check(27280, 4099, 1, 512, 256) && check(1, 1 << 21, 1, 1, 256) &&
            check(9000, 1 << 21, 3, 1, 256) && check(151584, 151584, 24, 1, 256) && check(38688, 262244, 12, 1, 256) &&
            check(278008, 349526, 24, 1, 256) && check(1, 1, 1, 1, 256) &&
            check(40, 1100000, 2, 2, 256);
  std::mt19937_64 g(7);
  auto log = [&](double lo, double hi) {
    return (int64_t)std::exp(std::uniform_real_distribution<>(std::log(lo), std::log(hi))(g));
  };
  for (int i = 0; ok && i < 200000; i++) {
    const int64_t Lq = log(1, 4e5), Lk = log(1, 2.2e6);
    const int heads = (int)log(1, 129), batch = (int)log(1, 600);
    ok = check(Lq, Lk, heads, batch, i % 8 ? 256 : (int)log(1, 400));
  }
  return ok ? 0 : 1;
}
