// Short-context plans (planner.hpp: build_plan with short_waves > 0) over
// random batches: where the planner takes that form, its items cover every
// (query row, visible token) once with both masks, their block lists
// name the pages the page table does, split rows have partial slots of
// their own inside the budget and a merge record each, and no other list is
// filled.  Where it does not, the plan is the ordinary one.  Host code only;
// built and run by tests/test_short_plan.py.
#include <stdio.h>

#include <algorithm>
#include <map>
#include <random>
#include <set>
#include <string>
#include <vector>

#include "fe_attn.h"
#include "planner.hpp"

using namespace feattn;

static int g_fail = 0;
#define CHECK(c)                                                   \
  do {                                                             \
    if (!(c)) {                                                    \
      printf("check failed, line %d: %s\n", __LINE__, #c);         \
      if (++g_fail > 20) return false;                             \
    }                                                              \
  } while (0)

struct Case {
  PlanShape sh;
  std::vector<int32_t> qo, kv, pages, last;
  int batch = 0, rows = 0;
};

static Case make(std::mt19937& rng) {
  static const int heads[][2] = {{16, 8}, {32, 8}, {32, 4}, {40, 8}, {64, 8}, {28, 4}, {8, 8}};
  Case c;
  auto pick = [&](int lo, int hi) { return std::uniform_int_distribution<int>(lo, hi)(rng); };
  const auto& h = heads[pick(0, 6)];
  c.sh.hq = h[0];
  c.sh.hkv = h[1];
  c.sh.dim = 128;
  c.sh.page = 16 << pick(0, 2);
  c.batch = pick(1, 24);
  const int kind = pick(0, 3);
  const int hi = pick(1, 3000);
  c.qo.push_back(0);
  c.kv.push_back(0);
  int most = 0;
  for (int b = 0; b < c.batch; ++b) {
    const int q = kind == 0 ? 1 : kind == 1 ? pick(0, 8) : kind == 2 ? 16 : pick(1, 400);
    const int len = q + pick(q ? 0 : 1, hi);
    const int np = (len + c.sh.page - 1) / c.sh.page;
    c.qo.push_back(c.qo.back() + q);
    c.kv.push_back(c.kv.back() + np);
    c.last.push_back(len - (np - 1) * c.sh.page);
    most = std::max(most, np);
  }
  c.rows = c.qo.back();
  c.sh.max_batch = c.batch;
  c.sh.max_pages = most + 1;
  c.sh.blocks = c.kv.back() + 3;
  for (int i = 0; i < c.kv.back(); ++i) c.pages.push_back(pick(0, c.sh.blocks));
  c.sh.partial_cap = 8192;
  return c;
}

static bool check(const Case& c, int waves, int& taken) {
  BuiltPlan bp, plain;
  std::string err;
  CHECK(build_plan(c.sh, c.qo.data(), c.kv.data(), c.pages.data(), c.last.data(), c.batch, c.rows, bp, err,
                   waves) == FE_OK);
  CHECK(build_plan(c.sh, c.qo.data(), c.kv.data(), c.pages.data(), c.last.data(), c.batch, c.rows, plain, err) ==
        FE_OK);
  CHECK(plain.shorts.empty());
  if (bp.shorts.empty()) {
    CHECK(bp.decode.size() == plain.decode.size());
    for (int m = 0; m < 2; ++m)
      CHECK(bp.mode[m].tile.size() == plain.mode[m].tile.size() && bp.mode[m].merge.size() == plain.mode[m].merge.size());
    return true;
  }
  ++taken;
  const int G = c.sh.hq / c.sh.hkv;
  CHECK(bp.decode.empty() && bp.decode_items.empty() && bp.decode_starts.empty() && bp.decode_merge.empty());
  CHECK(bp.decode_nc == 16 || bp.decode_nc == 32);
  for (int causal = 0; causal < 2; ++causal) {
    const ModeLists& ml = bp.mode[causal];
    CHECK(ml.tile.empty() && ml.tile_off.empty());
    CHECK((int64_t)bp.shorts.size() * (int64_t)sizeof(ShortItem) <= (int64_t)c.sh.item_cap * (int64_t)sizeof(WorkItem));
    CHECK(ml.partial_rows <= c.sh.partial_cap && (int)ml.merge.size() <= c.sh.partial_cap);
    // row -> pieces (a record stands for every kv head); partial slot -> owners
    std::map<int, std::vector<const ShortItem*>> cover;
    std::map<int, std::set<int>> slot_rows;
    for (const ShortItem& w : bp.shorts) {
      CHECK(w.nq >= 1 && w.nq * G <= bp.decode_nc);
      CHECK(w.t0 >= 0 && w.t0 % 16 == 0 && w.t1 > w.t0);
      const int b = (int)(std::upper_bound(c.qo.begin(), c.qo.end(), w.q0) - c.qo.begin()) - 1;
      const SeqInfo& s = bp.seqs[b];
      CHECK(w.q0 >= s.qo && w.q0 + w.nq <= s.qo + s.qlen && w.page_off == s.page_off && w.t1 <= s.len);
      CHECK(w.vis == s.len - s.qlen + (w.q0 - s.qo));
      for (int r = 0; r < w.nq; ++r) {
        cover[w.q0 + r].push_back(&w);
        if (w.part >= 0) {
          CHECK(w.part + r < ml.partial_rows);
          slot_rows[w.part + r].insert(w.q0 + r);
        }
      }
      // the wavefronts' blocks, by the kernel's division
      const int nblk = (w.t1 - w.t0 + 15) / 16, nbw = (nblk + waves - 1) / waves;
      for (int v = 0; v < waves; ++v) {
        const int nb = std::min(nblk, (v + 1) * nbw) - v * nbw;
        for (int j = 0; j < 4 && nb > 0; ++j) {
          const int tok = w.t0 + 16 * (v * nbw + std::min(j, nb - 1));
          const int64_t slot = (int64_t)c.pages[w.page_off + tok / c.sh.page] * c.sh.page + tok % c.sh.page;
          CHECK((int64_t)w.block[4 * v + j] * 16 == slot);
        }
      }
    }
    std::map<int, MergeRow> merge;
    for (const MergeRow& r : ml.merge) CHECK(merge.emplace(r.row, r).second);
    for (const auto& s : slot_rows) CHECK(s.second.size() == 1);
    size_t rows = 0;
    for (int b = 0; b < c.batch; ++b)
      for (int i = 0; i < bp.seqs[b].qlen; ++i) {
        const SeqInfo& s = bp.seqs[b];
        const int row = s.qo + i, seen = causal ? s.len - s.qlen + i + 1 : s.len;
        ++rows;
        std::vector<const ShortItem*>& v = cover[row];
        std::sort(v.begin(), v.end(), [](const ShortItem* x, const ShortItem* y) { return x->t0 < y->t0; });
        int at = 0;
        for (size_t p = 0; p < v.size(); ++p) {
          CHECK(v[p]->t0 == at);
          at = v[p]->t1;
          if (v.size() > 1) {
            CHECK(merge.count(row) == 1);
            const MergeRow& m = merge[row];
            CHECK(m.nsplit == (int)v.size() && v[p]->part + (row - v[p]->q0) == m.part + (int)p * m.stride);
          } else {
            CHECK(v[p]->part == -1 && merge.count(row) == 0);
          }
        }
        CHECK(at >= seen && at <= s.len);
      }
    CHECK(rows == cover.size());
  }
  return true;
}

// Plans with small_tiles: where a mode's tile list is not the ordinary one,
// its items are unsplit, at most 64 columns wide, cover every row of the tile
// sequences once per kv head over all the tokens it sees, and its shares
// cover the list.
static bool check_tiles(const Case& c, int& taken) {
  BuiltPlan bp, plain;
  std::string err;
  CHECK(build_plan(c.sh, c.qo.data(), c.kv.data(), c.pages.data(), c.last.data(), c.batch, c.rows, bp, err, 0, true) ==
        FE_OK);
  CHECK(build_plan(c.sh, c.qo.data(), c.kv.data(), c.pages.data(), c.last.data(), c.batch, c.rows, plain, err) ==
        FE_OK);
  const int G = c.sh.hq / c.sh.hkv;
  CHECK(bp.decode.size() == plain.decode.size() && bp.decode_partials == plain.decode_partials);
  for (int causal = 0; causal < 2; ++causal) {
    const ModeLists& ml = bp.mode[causal];
    if (ml.tile.empty()) continue;
    CHECK(ml.tile_rows >= 1 && ml.tile_rows * G <= kTileCols);
    for (const WorkItem& w : ml.tile) CHECK(w.nq <= ml.tile_rows);
    if (ml.tile_rows == plain.mode[causal].tile_rows) {
      CHECK(ml.tile.size() == plain.mode[causal].tile.size() && ml.tile_off == plain.mode[causal].tile_off);
      continue;
    }
    ++taken;
    CHECK(ml.tile_rows == kTileCols / 2 / G && ml.partial_rows == bp.decode_partials);
    CHECK(ml.merge.size() == bp.decode_merge.size());
    CHECK(!ml.tile_off.empty() && ml.tile_off.front() == 0 && ml.tile_off.back() == (int)ml.tile.size());
    CHECK((int)ml.tile_off.size() - 1 <= c.sh.tile_slots);
    std::map<std::pair<int, int>, int> seen;  // (row, kv head) -> end of its tokens
    for (const WorkItem& w : ml.tile) {
      CHECK(w.part == -1 && w.t0 == 0 && w.nq >= 1);
      const SeqInfo& s = bp.seqs[w.seq];
      CHECK(w.q0 >= s.qo && w.q0 + w.nq <= s.qo + s.qlen && w.t1 <= s.len);
      for (int r = 0; r < w.nq; ++r) CHECK(seen.emplace(std::make_pair(w.q0 + r, w.kvh), w.t1).second);
    }
    size_t want = 0;
    for (const SeqInfo& s : bp.seqs) {
      if (s.qlen * G <= kDecodeCols) continue;
      for (int i = 0; i < s.qlen; ++i)
        for (int h = 0; h < c.sh.hkv; ++h, ++want)
          CHECK((seen[{s.qo + i, h}] >= (causal ? s.len - s.qlen + i + 1 : s.len)));
    }
    CHECK(want == seen.size());
  }
  return true;
}

// One causal prompt of growing length, nothing cached: the tile list takes the
// small form from the first length on and changes to the ordinary one at most
// once.  (ordinary: the length from which it does.)
static bool check_prompts(int hq, int hkv, int& ordinary) {
  const int G = hq / hkv, most = 3000;
  Case c;
  c.sh.hq = hq;
  c.sh.hkv = hkv;
  c.sh.dim = 128;
  c.sh.page = 16;
  c.sh.max_batch = 1;
  c.sh.max_pages = most / 16 + 2;
  c.sh.blocks = most;
  c.sh.partial_cap = 8192;
  for (int i = 0; i <= most / 16; ++i) c.pages.push_back(i);
  ordinary = 0;
  for (int n = kDecodeCols / G + 1; n <= most; n += n < 1500 ? 3 : 7) {
    const int np = (n + 15) / 16;
    const int32_t qo[2] = {0, n}, kv[2] = {0, np}, last[1] = {n - 16 * (np - 1)};
    BuiltPlan bp;
    std::string err;
    CHECK(build_plan(c.sh, qo, kv, c.pages.data(), last, 1, n, bp, err, 0, true) == FE_OK);
    const bool small = bp.mode[1].tile_rows == kTileCols / 2 / G;
    if (!small && ordinary == 0) ordinary = n;
    CHECK(!small || ordinary == 0);
  }
  return true;
}

// Decode batches of one length, up to and past the workgroups that run at
// once: beyond them only sequences of at most 64 tokens that the shares would
// have to merge are short-context items.
static bool check_two_sets() {
  for (const int waves : {4, 8})
    for (const int len : {16, 30, 33, 48, 49, 64, 65, 100, 128}) {
      Case c;
      c.sh.hq = 32;
      c.sh.hkv = waves;
      c.sh.dim = 128;
      c.sh.page = 16;
      c.sh.max_pages = 10;
      c.sh.partial_cap = 8192;
      const int slots = c.sh.decode_waves / waves / waves;  // sequences whose workgroups run at once
      for (const int seqs : {slots, slots + 1, 2 * slots, 2 * slots + 1}) {
        const int np = (len + 15) / 16;
        c.sh.max_batch = seqs;
        c.sh.blocks = seqs * np;
        c.qo.assign(1, 0);
        c.kv.assign(1, 0);
        c.pages.clear();
        c.last.assign(seqs, len - 16 * (np - 1));
        for (int b = 0; b < seqs; ++b) {
          c.qo.push_back(b + 1);
          c.kv.push_back((b + 1) * np);
          for (int i = 0; i < np; ++i) c.pages.push_back(b * np + i);
        }
        BuiltPlan bp;
        std::string err;
        CHECK(build_plan(c.sh, c.qo.data(), c.kv.data(), c.pages.data(), c.last.data(), seqs, seqs, bp, err, waves) ==
              FE_OK);
        const bool merged = np == 3;  // 48-token strides cross the shares' 64-token borders
        CHECK(!bp.shorts.empty() == (seqs <= slots || (seqs <= 2 * slots && len <= 64 && merged)));
      }
    }
  return true;
}

int main() {
  if (!check_two_sets()) return 1;
  static const int heads[][2] = {{4, 1},  {8, 2},  {8, 8},  {12, 2}, {16, 2}, {16, 8},
                                 {28, 4}, {32, 4}, {32, 8}, {40, 8}, {64, 4}, {64, 8}};
  for (const auto& h : heads) {
    int at = 0;
    if (!check_prompts(h[0], h[1], at) || at < 300) {
      printf("prompts, %d/%d heads: ordinary from %d tokens\n", h[0], h[1], at);
      return 1;
    }
  }
  std::mt19937 rng(7);
  int taken = 0, n = 0, tiles = 0;
  for (int i = 0; i < 3000; ++i) {
    const Case c = make(rng);
    if (!check_tiles(c, tiles)) {
      printf("batch %d, small tiles\n", i);
      return 1;
    }
    for (int waves : {4, 8}) {
      ++n;
      if (!check(c, waves, taken)) {
        printf("batch %d, %d wavefronts\n", i, waves);
        return 1;
      }
    }
  }
  printf("%d plans, %d short, %d small tile lists\n", n, taken, tiles);
  return g_fail || taken < n / 20 || taken == n || tiles < 100;
}
