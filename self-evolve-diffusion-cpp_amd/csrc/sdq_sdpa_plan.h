// Host side of the packed attention (sdq_sdpa.hip): how a call is spread over
// workgroups and what scratch that takes. Plain C++, so that it is checked
// without a GPU.
#pragma once

#include <cstdint>
#include <cstdlib>
#include <initializer_list>

namespace sdq {
namespace sdpa {

constexpr int kHd = 128;     // head dim
constexpr int kKB = 32;      // keys per block
constexpr int kQ = 256;      // queries per workgroup
constexpr int kRec = 32768;  // bytes of a packed block: K parts, V parts

inline int64_t div_up(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline int64_t pad256(int64_t n) { return div_up(n, 256) * 256; }

// How a sequence's items (256 queries of one head, all its key blocks) are
// spread over workgroups. The first nfull items, whole rounds of the CUs, run
// whole. The others, which would fill only part of a round, are cut by keys
// into `splits` shares of kbs blocks (splits = 1: not cut); a share leaves its
// unnormalized output and its (reference, sum) pair in slot (item - nfull) *
// splits + share, and sdpa_combine_kernel adds up an item's shares.
struct Plan {
  int nkb;      // key blocks
  int qgroups;  // items per head
  int items;    // heads * qgroups
  int nfull;
  int splits;
  int kbs;
};
// Scratch of a launch: at most this, whatever the call (a head's 2^21 keys are
// 2 GiB of records; their exponents and shifts come on top).
constexpr int64_t kMaxRecs = int64_t(1) << 31;
constexpr int64_t kMaxScratch = kMaxRecs + (5 << 20);
constexpr int64_t kShareBytes = kQ * (kHd * 4 + 8);  // a share's partial output

// `most`: bytes that the partial outputs of one sequence may take. Depends on
// the sequence only, not on the batch, so stacked and separate calls give the
// same bits.
inline Plan make_plan(int64_t Lq, int64_t Lk, int heads, int cu_count, int64_t most) {
  Plan p{};
  p.nkb = (int)div_up(Lk, kKB);
  p.qgroups = (int)div_up(Lq, kQ);
  p.items = heads * p.qgroups;
  p.splits = 1;
  p.kbs = p.nkb;
  const int cus = cu_count > 0 ? cu_count : 256;
  p.nfull = p.items / cus * cus;
  const int rest = p.items - p.nfull;
  // for comparisons: a factor (2 to 16, where the shares fit), below 2 no cut
  const char* forced = std::getenv("SDQ_SDPA_SPLIT");
  int f = forced ? std::atoi(forced) : 0;
  if (rest == 0 || (forced && f < 2)) {
    p.nfull = p.items;
    return p;
  }
  if (forced) {
    for (f = f < 16 ? f : 16; f > 1 && rest * f * kShareBytes > most;) f--;
    p.kbs = (p.nkb + f - 1) / f;
    p.splits = (p.nkb + p.kbs - 1) / p.kbs;  // no empty share
    return p;
  }
  // The cut that ends first, in key-block times: rounds of shares, each with
  // its own start and end (about 3 blocks), plus the second pass over the
  // partial outputs.
  double best = p.nkb + 3;
  for (int S = 2; S <= 32 && 3 * S <= p.nkb && rest * S * kShareBytes <= most; S++) {
    const int kbs = (p.nkb + S - 1) / S;
    if ((p.nkb + kbs - 1) / kbs != S) continue;  // no empty share
    const double cost = (double)((rest * S + cus - 1) / cus) * (kbs + 3) + 3;
    if (cost < best) best = cost, p.splits = S, p.kbs = kbs;
  }
  return p;
}

// Scratch of one launch over `heads` heads of `batch` sequences.
struct Layout {
  // offsets of its parts (the records lie at 0): the records' exponents, their
  // keys' shifts (V's, K's), the shares' outputs and sums
  int64_t exps, shifts, o, ml, bytes;
};
inline Layout layout(const Plan& p, int64_t heads, int64_t batch) {
  const int64_t recs = batch * heads * p.nkb;
  const int64_t rows =
      p.splits > 1 ? batch * (p.items - p.nfull) * p.splits * (int64_t)kQ : 0;
  Layout l;
  l.exps = recs * kRec;
  l.shifts = l.exps + pad256(recs * 8);
  l.o = l.shifts + pad256(recs * 2 * kKB);
  l.ml = l.o + rows * kHd * 4;
  l.bytes = l.ml + rows * 8;
  return l;
}

// The plan of a launch over `heads` heads, its partial outputs within what the
// records leave of kMaxScratch.
inline Plan launch_plan(int64_t Lq, int64_t Lk, int heads, int cu_count) {
  Plan p{};
  p.nkb = (int)div_up(Lk, kKB);
  p.splits = 1;
  return make_plan(Lq, Lk, heads, cu_count, kMaxScratch - layout(p, heads, 1).bytes);
}

// A call runs in launches of as many sequences, or of equal numbers of heads
// of one sequence, as fit kMaxScratch with the plan they would have without
// that limit (heads: a sequence's own share, so that it does not depend on the
// batch); a single head takes fewer shares instead.
struct Chunk {
  int heads, seqs;
};
inline Chunk chunk(int64_t Lq, int64_t Lk, int heads, int batch, int cu_count) {
  auto bytes = [&](int h) {
    return layout(make_plan(Lq, Lk, h, cu_count, INT64_MAX), h, 1).bytes;
  };
  if (const int64_t b = bytes(heads); b <= kMaxScratch) {
    const int64_t n = kMaxScratch / b;
    return {heads, (int)(n < batch ? n : batch)};
  }
  // (from the fewest launches that the records allow)
  for (int64_t c = div_up(heads * div_up(Lk, kKB) * kRec, kMaxRecs); c < heads; c++) {
    const int h = (int)div_up(heads, c);
    if (bytes(h) <= kMaxScratch && (heads % h == 0 || bytes(heads % h) <= kMaxScratch))
      return {h, 1};
  }
  return {1, 1};
}

// Bytes that every launch of a call fits in; 0: the packed form does not take
// it. A last chunk of fewer heads has a plan of its own, whose shares' outputs
// can outweigh the records that the missing heads leave free.
inline int64_t scratch_bytes(int64_t Lq, int64_t Lk, int heads, int batch, int cu_count) {
  // a head's records are addressed with 32-bit offsets; a grid holds 2^32 threads
  if (Lk > kMaxRecs / kRec * kKB || heads > 65535 || div_up(Lq, kQ) * heads > (1 << 22)) return 0;
  const Chunk c = chunk(Lq, Lk, heads, batch, cu_count);
  int64_t most = 0;
  for (const int h : {c.heads, heads % c.heads}) {
    const int64_t b = h ? layout(launch_plan(Lq, Lk, h, cu_count), h, c.seqs).bytes : 0;
    most = b > most ? b : most;
  }
  return most;
}

// Few queries over many keys (at most 64 over more than kFewKeys): packing K and
// V moves them three times where one pass reads them once, so that pass takes
// less, cut into this many key ranges (1: the packed form). us, 24 heads, 64
// queries, packed / one pass: 4096 keys 64 / 67, 8192 116-126 / 101, 20000 303 /
// 197, 27280 450-470 / 258. More queries need a pass per 64: 157 queries over 8192
// keys 133 / 195.
constexpr int64_t kFewKeys = 4096;
inline int few_splits(int64_t Lq, int64_t Lk, int heads, int cu_count) {
  if (Lq > 64 || Lk <= kFewKeys || heads > 65535) return 1;
  const int64_t nkb = div_up(Lk, kKB);
  if (const char* forced = std::getenv("SDQ_SDPA_SPLIT")) {  // for comparisons
    const int f = std::atoi(forced);
    return f < 2 ? 1 : (int)div_up(nkb, div_up(nkb, f < 16 ? f : 16));
  }
  // the fewest rounds of workgroups (two per CU) per unit of work, no empty range
  const int64_t slots = 2 * (int64_t)(cu_count > 0 ? cu_count : 256);
  int best = 1;
  double best_cost = 0.9 * (double)div_up(heads, slots);
  for (int S = 2; S <= 32; S++) {
    if (div_up(nkb, div_up(nkb, S)) != S) continue;
    const double cost = (double)div_up((int64_t)heads * S, slots) / S;
    if (cost < best_cost) best_cost = cost, best = S;
  }
  return best;
}
// Scratch of one sequence's partial outputs, and of a call's: sequences run in
// turns of as many as fit kMaxScratch.
inline int64_t few_bytes(int64_t Lq, int heads, int splits) {
  return splits * Lq * heads * (kHd + 2) * 4;
}
inline int64_t few_scratch(int64_t Lq, int heads, int splits, int batch) {
  const int64_t one = few_bytes(Lq, heads, splits);
  if (one > kMaxScratch) return 0;
  const int64_t n = kMaxScratch / one;
  return one * (n < batch ? n : batch);
}

}  // namespace sdpa
}  // namespace sdq
