// Host-side check of the prefill split (PrefillSched in prefill_split.h) with
// the settings of the kernel whose source is included before this file, run on
// the CPU (no GPU call). Over random batches (ragged, mixed, equal, a few long
// items, empty sequences, chunks longer than max_query_len): the bounds never
// decrease, every workgroup in use has a group of its own, every tile of every
// item is taken exactly once, and the merge can find the pieces of a cut item
// from the descriptors alone: in consecutive groups, in order, the first begun
// and the others continued by their group, at most one of each in a group, the
// last one marked as the end.
#pragma once

#include <algorithm>
#include <cstdio>
#include <map>
#include <random>
#include <tuple>
#include <vector>

// The included file's host launcher references this; nothing here launches.
namespace clv {
hipError_t launch_prefill_valu(const PrefillParams &, DType, hipStream_t) {
  return hipErrorInvalidValue;
}
}  // namespace clv

template <class Cfg>
struct SplitCheck {
  typedef clv::PrefillSched<Cfg> Sched;
  long cases = 0, bad = 0, cut = 0, uncut = 0, most = 0;
  std::mt19937_64 rng{5};
  int upto(int n) { return (int)(rng() % (uint64_t)(n + 1)); }

  struct Piece {
    int item[3], t0, t1, nt;
    bool is(const Piece &o) const { return std::equal(item, item + 3, o.item); }
  };

  bool batch(int rows, int groups) {
    clv::PrefillParams p{};
    p.group = 1 + upto(upto(1) ? 7 : 63);
    p.num_kv_heads = 1 + upto(upto(1) ? 7 : 31);
    p.block_shift = 4;
    const int bq = rows / p.group;
    const int kind = upto(4), seqs = 1 + upto(kind == 0 ? 200 : 30);
    const int hi = 1 << upto(16), chunk = 1 + upto(kind == 3 ? 2000 : 300), cached = upto(hi);
    std::vector<int> ctx(seqs), qsl(seqs + 1, 0);
    for (int s = 0; s < seqs; ++s) {
      int n = kind == 1 ? chunk : 1 + upto(chunk - 1);
      if (kind == 0 && upto(9)) n = 1;
      if (kind == 2 && upto(3) == 0) n = 0;
      ctx[s] = (kind == 1 ? cached : upto(hi)) + n - (upto(19) == 0 ? std::min(n, 7) : 0);
      qsl[s + 1] = qsl[s] + n;
    }
    int longest = 0;
    for (int s = 0; s < seqs; ++s) longest = std::max(longest, qsl[s + 1] - qsl[s]);
    if (upto(9) == 0) longest = std::max(1, longest / 2);  // a caller's error: rows past it
    const int nq = std::max(1, (longest + bq - 1) / bq);
    if (seqs * nq > clv::kPrefillSplitItems) return true;
    p.num_seqs = seqs;
    p.max_query_len = longest;
    p.context_lens = ctx.data();
    p.query_start_loc = qsl.data();
    p.max_blocks_per_seq = *std::max_element(ctx.begin(), ctx.end()) / 16 + 1 + upto(3);

    Sched sc;
    sc.nq = nq;
    sc.n = seqs * nq;
    std::vector<int> pre(sc.n + 1);
    int units = 0, items = 0, longest_item = 0;
    for (int i = 0; i < sc.n; ++i) {
      pre[i] = sc.entry_units(p, bq, i);
      units += pre[i];
      items += pre[i] > 0;
      longest_item = std::max(longest_item, pre[i]);
    }
    sc.set_totals(p.num_kv_heads, groups, units, items, longest_item);
    int run = 0;
    for (int i = 0; i < sc.n; ++i) {
      const int u = pre[i];
      pre[i] = run;
      run += sc.whole ? (u > 0) : u;
    }
    pre[sc.n] = run;
    sc.pre = pre.data();
    ++cases;

    bool ok = sc.W >= 1 && sc.W <= groups && run == sc.C;
    std::vector<int> owner(groups, 0);
    int used = 0;
    for (int b = 0; b < groups; ++b) {
      const int w = sc.group_of(b);
      if (w >= sc.W || (w >= 0 && owner[w]++)) ok = false;
      used += w >= 0;
    }
    ok = ok && used == sc.W;
    for (int w = 0; w < sc.W; ++w) ok = ok && sc.bound(w) <= sc.bound(w + 1);
    ok = ok && sc.bound(0) == 0 && sc.bound(sc.W) == sc.N;

    std::map<std::tuple<int, int, int>, std::vector<std::pair<int, int>>> taken;
    std::vector<Piece> begun(groups, Piece{{-1, -1, -1}, 0, 0, 0}), cont = begun;
    for (int w = 0; w < sc.W && ok; ++w) {
      int cur[Sched::kCursorInts];
      sc.start(w, cur);
      clv::PrefillItem it;
      Piece x;
      while (Sched::next(p, bq, nq, pre.data(), cur, it, x.t0, x.t1, x.nt)) {
        x.item[0] = it.s, x.item[1] = it.kvh, x.item[2] = it.qt;
        taken[{it.s, it.kvh, it.qt}].push_back({x.t0, x.t1});
        if (it.q0 >= it.q_hi || x.t1 > x.nt || x.nt != Sched::tiles(it.kv_end)) ok = false;
        if (x.t0 == 0 && x.t1 == x.nt) continue;
        Piece &slot = x.t0 == 0 ? begun[w] : cont[w];
        if (slot.item[0] >= 0 || sc.whole) ok = false;
        slot = x;
      }
    }
    // Every tile of every item once, in the order of the groups.
    size_t want = 0;
    for (int s = 0; s < seqs; ++s)
      want += (size_t)std::min(nq, (qsl[s + 1] - qsl[s] + bq - 1) / bq) * p.num_kv_heads;
    ok = ok && taken.size() == want;
    for (auto &kv : taken) {
      clv::PrefillItem it;
      it.set(p, bq, std::get<0>(kv.first), std::get<1>(kv.first), std::get<2>(kv.first));
      int at = 0;
      for (auto &r : kv.second) {
        if (r.first != at || r.second <= r.first) ok = false;
        at = r.second;
      }
      ok = ok && at == Sched::tiles(it.kv_end);
    }
    // As the merge reads the descriptors.
    for (int w = 0; w < groups && ok; ++w) {
      if (begun[w].item[0] < 0) continue;
      ++cut;
      int at = begun[w].t1, n = 1;
      for (int b = w + 1;; ++b) {
        if (b >= groups || !cont[b].is(begun[w]) || cont[b].t0 != at) {
          ok = false;
          break;
        }
        at = cont[b].t1;
        ++n;
        if (at == cont[b].nt) break;
      }
      most = std::max(most, (long)n);
    }
    if (sc.whole) ++uncut;
    if (!ok && bad < 5)
      printf("bad: group %d heads %d seqs %d nq %d kind %d hi %d\n", p.group, p.num_kv_heads, seqs,
             nq, kind, hi);
    return ok;
  }

  int run(int rows, int groups, int batches) {
    for (int it = 0; it < batches; ++it)
      if (!batch(rows, groups)) ++bad;
    if (cut == 0 || uncut == 0 || most < 65) ++bad;  // every kind of schedule was there
    printf("cases %ld uncut %ld cut items %ld most pieces %ld bad %ld\n", cases, uncut, cut, most, bad);
    return bad != 0;
  }
};
