// Host planner.  Validation mirrors the reference's checks
// (src/flashinfer_attention.cu:23,30; src/portable_gpu_ops.cpp:28-30) and adds
// the ones a raw-pointer kernel needs to stay in bounds (page ids, `last`).
#include "planner.hpp"

#include <algorithm>
#include <new>

#include "fe_attn.h"

namespace feattn {

namespace {

// Shortest decode share: below this, per-piece start-up and merge cost more
// than the extra wavefronts gain.
constexpr int64_t kMinShareTokens = 64;

bool is_pow2(int v) { return v > 0 && (v & (v - 1)) == 0; }

int round_up(int v, int m) { return (v + m - 1) / m * m; }

int ceil_div(int a, int b) { return (a + b - 1) / b; }

// Share boundaries (token offsets into the decode stream, multiples of 16):
// equal shares of `quota` tokens.
std::vector<int64_t> cut_uniform(int64_t stream, int64_t quota) {
  std::vector<int64_t> cuts;
  for (int64_t c = 0; c < stream; c += quota) cuts.push_back(c);
  cuts.push_back(stream);
  return cuts;
}

}  // namespace

// Assigns items to `slots` shares (one per tile workgroup) by the longest
// processing time rule -- in decreasing cost order, each item goes to the
// least-loaded share -- and regroups them share by share (longest first
// inside a share).  off receives the CSR offsets of the shares in use.
void assign_shares(std::vector<WorkItem>& items, int slots, std::vector<int32_t>& off, int fast) {
  // Stable sort by decreasing cost: a counting sort over the (small,
  // non-negative) costs, else the comparison sort.
  int32_t cmin = 0, cmax = 0;
  for (const WorkItem& w : items) {
    cmin = std::min(cmin, w.cost);
    cmax = std::max(cmax, w.cost);
  }
  if (cmin >= 0 && cmax <= (1 << 16)) {
    std::vector<int32_t> start((size_t)cmax + 2, 0);
    for (const WorkItem& w : items) ++start[(size_t)(cmax - w.cost) + 1];
    for (size_t c = 1; c < start.size(); ++c) start[c] += start[c - 1];
    std::vector<WorkItem> sorted(items.size());
    for (const WorkItem& w : items) sorted[start[(size_t)(cmax - w.cost)]++] = w;
    items.swap(sorted);
  } else {
    std::stable_sort(items.begin(), items.end(),
                     [](const WorkItem& x, const WorkItem& y) { return x.cost > y.cost; });
  }
  const int n = std::max(1, std::min<int>(slots, (int)items.size()));
  if (!items.empty() && (int)items.size() <= slots && items.back().cost > 0) {
    // A share for every item: each goes to the first that is still empty.
    off.resize((size_t)n + 1);
    for (int k = 0; k <= n; ++k) off[k] = k;
    return;
  }
  std::vector<int> share(items.size());
  // Binary min-heap of (load << 20 | share) keys: the root is the least-loaded
  // share, the lowest index among equals.  Each item raises the root's load
  // and sifts it down (one pass instead of a pop and a push).  Shares below
  // `fast` count their load at kFastShareWeight / kSlowShareWeight (2/3): they
  // end up with 3/2 of the others' work.
  constexpr int kShareBits = 20;  // shares (tile workgroups) < 2^20; loads < 2^43
  const bool weighted = fast < n;
  std::vector<uint64_t> heap(n);
  for (int k = 0; k < n; ++k) heap[k] = (uint64_t)k;  // ascending: already a heap
  for (size_t i = 0; i < items.size(); ++i) {
    const int k = (int)(heap[0] & ((uint64_t(1) << kShareBits) - 1));
    share[i] = k;
    const uint64_t w = !weighted ? 1 : (k < fast ? kFastShareWeight : kSlowShareWeight);
    const uint64_t key = heap[0] + (((uint64_t)items[i].cost * w) << kShareBits);
    size_t h = 0;
    for (;;) {
      size_t c = 2 * h + 1;
      if (c >= (size_t)n) break;
      if (c + 1 < (size_t)n && heap[c + 1] < heap[c]) ++c;
      if (heap[c] >= key) break;
      heap[h] = heap[c];
      h = c;
    }
    heap[h] = key;
  }
  off.assign(n + 1, 0);
  for (size_t i = 0; i < items.size(); ++i) ++off[share[i] + 1];
  for (int k = 0; k < n; ++k) off[k + 1] += off[k];
  std::vector<WorkItem> grouped(items.size());
  std::vector<int32_t> pos(off.begin(), off.end() - 1);
  for (size_t i = 0; i < items.size(); ++i) grouped[pos[share[i]]++] = items[i];
  items.swap(grouped);
}

namespace {

// Tile work list by an equal cut of the tile stream: the query-row chunks of
// the tile sequences (qr rows each, over their visible token ranges), in
// batch order, are laid end to end and cut at tile boundaries into `slots /
// hkv` shares of equal cost (tiles x 16-column blocks per wavefront).  Every
// kv head uses the same cut, and share k of kv head h goes to workgroup
// k * hkv + h, so the workgroups of one share read the same pages at the same
// time.  A chunk cut into several pieces gets partial slots and merge rows
// as in the longest-first list.  Returns false, leaving `ml` alone, when the
// cut needs more partial slots or items than `slot_budget` / `item_cap`.
bool cut_tile_stream(const std::vector<SeqInfo>& seqs, int G, int hkv, bool causal, int slots, int partial_base,
                     int slot_budget, int item_cap, ModeLists& ml) {
  const int qr = kTileCols / G;
  const int n_shares = slots / hkv;
  if (n_shares < 1) return false;
  struct Chunk {
    int seq, q0, nq, extent, tiles, c;
  };
  std::vector<Chunk> ch;
  int64_t total = 0;
  for (int b = 0; b < (int)seqs.size(); ++b) {
    const SeqInfo& s = seqs[b];
    if (s.qlen * G <= kDecodeCols) continue;
    for (int i0 = 0; i0 < s.qlen; i0 += qr) {
      const int nq = std::min(qr, s.qlen - i0);
      const int extent = causal ? std::min(s.len, s.len - s.qlen + i0 + nq) : s.len;
      const int tiles = ceil_div(extent, kTileTokens);
      const int c = nq * G > kTileCols / 2 ? 2 : 1;
      ch.push_back(Chunk{b, s.qo + i0, nq, extent, tiles, c});
      total += (int64_t)tiles * c;
    }
  }
  if (ch.empty()) return false;
  // Pieces in stream order: (chunk, first tile, tiles, share).  Share k ends
  // at the first tile boundary where the cumulative cost reaches
  // (k + 1) * total / n_shares, so a tile's granularity never accumulates
  // from share to share; the last share ends with the stream.
  struct Piece {
    int chunk, tile0, ntiles, share;
  };
  std::vector<Piece> pcs;
  std::vector<int> npc(ch.size(), 0);
  int share = 0;
  int64_t cum = 0;
  auto target = [&](int k) { return ((int64_t)(k + 1) * total + n_shares - 1) / n_shares; };
  for (int i = 0; i < (int)ch.size(); ++i) {
    int done = 0;
    while (done < ch[i].tiles) {
      while (share < n_shares - 1 && cum >= target(share)) ++share;
      int take = ch[i].tiles - done;
      if (share < n_shares - 1) {
        const int64_t need = (target(share) - cum + ch[i].c - 1) / ch[i].c;  // >= 1 tile
        take = (int)std::min<int64_t>(need, take);
      }
      pcs.push_back(Piece{i, done, take, share});
      ++npc[i];
      done += take;
      cum += (int64_t)take * ch[i].c;
    }
  }
  if ((int64_t)pcs.size() * hkv > item_cap) return false;
  std::vector<int> base(ch.size(), -1);
  int64_t rows = partial_base;
  for (size_t i = 0; i < ch.size(); ++i)
    if (npc[i] > 1) {
      base[i] = (int)rows;
      rows += (int64_t)npc[i] * ch[i].nq;
    }
  if (rows > slot_budget) return false;

  ModeLists out;
  out.tile_rows = qr;
  out.partial_rows = (int)rows;
  for (size_t i = 0; i < ch.size(); ++i)
    if (base[i] >= 0)
      for (int r = 0; r < ch[i].nq; ++r) out.merge.push_back(MergeRow{ch[i].q0 + r, base[i] + r, npc[i], ch[i].nq});
  // Piece p's index within its chunk (pieces of a chunk are consecutive).
  std::vector<int> sp(pcs.size());
  for (size_t p = 0; p < pcs.size(); ++p) sp[p] = (p > 0 && pcs[p - 1].chunk == pcs[p].chunk) ? sp[p - 1] + 1 : 0;
  const int used = pcs.back().share + 1;
  out.tile.reserve(pcs.size() * (size_t)hkv);
  out.tile_off.assign((size_t)used * hkv + 1, 0);
  size_t p0 = 0;
  for (int k = 0; k < used; ++k) {
    size_t p1 = p0;
    while (p1 < pcs.size() && pcs[p1].share == k) ++p1;
    for (int h = 0; h < hkv; ++h) {
      for (size_t p = p0; p < p1; ++p) {
        const Chunk& c = ch[pcs[p].chunk];
        const int t0 = pcs[p].tile0 * kTileTokens;
        const int t1 = std::min(c.extent, (pcs[p].tile0 + pcs[p].ntiles) * kTileTokens);
        const int part = base[pcs[p].chunk] < 0 ? -1 : base[pcs[p].chunk] + sp[p] * c.nq;
        out.tile.push_back(WorkItem{c.seq, c.q0, c.nq, h, t0, t1, part, pcs[p].ntiles * c.c});
      }
      out.tile_off[(size_t)k * hkv + h + 1] = (int32_t)out.tile.size();
    }
    p0 = p1;
  }
  ml = std::move(out);
  return true;
}

// Plans a batch of decode sequences as short-context items, or returns false
// (leaving `out` alone) where shares are the faster plan.
//
// A workgroup takes W * 64 tokens per round of loads (a "step").  Measured on
// the MI355X, us per call over caches larger than the L2, this plan against
// shares + merge, 8 kv heads (W = 8) and 4 query heads each unless said
// otherwise:
//   * sequences of one step: 9.2 / 14.8 (12 x 200), 10.3 / 15.4 (12 x 512); of
//     two, with W = 4: 10.2 / 14.5 (12 x 512, 4 kv heads).  A second round
//     of 8 wavefronts costs more than merging two pieces: 15.4 / 12.2 for 1
//     x 1001 whole, cut 12.2.
//   * cut into steps: 13.7 / 18.3 (1 x 4001), 13.8 / 17.4 (4 x 1984).
//   * more items than resident workgroups: 17.0 / 15.9 (64 x 200) and, cut,
//     27.9 / 22.3 (12 x 2048); up to twice as many still gain where no sequence
//     is longer than 64 tokens, 11.4 / 15.1 (64 x 41), 13.5 / 15.5 (200 x 33, W =
//     4), in a graph 13.3 / 15.0 and 15.7 / 15.4 -- but only against a merge:
//     where every sequence lies within one share, 12.4 / 9.9 (64 x 64), 15.6 /
//     10.2 (200 x 64, W = 4); and not longer ones, 17.0 / 13.2 (64 x 128), in a
//     graph 18.9 / 13.1.
//   * with more K and V per compute unit, the shares' whole-page streams win
//     when the cache is cold: 188 KB, inside a replayed decode step, 1.6 us a
//     layer slower so.  Two column blocks are slow on the shares (20.3 /
//     26.9 at 182 KB, 5 rows of 5 heads), so the line is higher there.
bool plan_short(const PlanShape& sh, const int32_t* pages, int waves, BuiltPlan& out) {
  const int G = sh.hq / sh.hkv;
  const int64_t slots = sh.decode_waves / waves;  // workgroups that run at once
  const int step = 64 * waves;
  int max_len = 0, max_cols = 0;
  int64_t whole = 0, cut = 0, tokens = 0;  // items of either form
  int64_t off = 0;                         // in the stream of the decode shares
  bool crossing = false;                   // a sequence crosses the border of two (shortest) shares
  for (const SeqInfo& s : out.seqs) {
    if (s.qlen == 0) continue;
    if (s.qlen * G > kDecodeCols) return false;
    max_len = std::max(max_len, s.len);
    max_cols = std::max(max_cols, s.qlen * G);
    whole += sh.hkv;
    cut += (int64_t)sh.hkv * ceil_div(s.len, step);
    tokens += s.len;
    const int64_t end = off + round_up(s.len, 16);
    crossing = crossing || off / kMinShareTokens != (end - 1) / kMinShareTokens;
    off = end;
  }
  if (whole == 0) return false;
  const int64_t per_cu = tokens * sh.hkv * (2 * kHeadDim * 2) / sh.num_cus;
  const int64_t limit = max_cols <= 16 ? 144 << 10 : 256 << 10;
  if (per_cu > limit) return false;
  int piece;
  // (Twice as many workgroups of such sequences: the shares are the shortest.)
  if (max_len <= 512 && (whole <= slots || (max_len <= kMinShareTokens && whole <= 2 * slots && crossing)))
    piece = 512;
  else if (cut <= slots)
    piece = step;
  else
    return false;
  // Longest first: the order in which workgroups start.
  std::vector<int> order;
  for (int b = 0; b < (int)out.seqs.size(); ++b)
    if (out.seqs[b].qlen > 0) order.push_back(b);
  auto longer = [&](int x, int y) { return out.seqs[x].len > out.seqs[y].len; };
  if (!std::is_sorted(order.begin(), order.end(), longer)) std::stable_sort(order.begin(), order.end(), longer);
  int in_page = 0;  // log2 of the 16-token blocks of a page
  while ((16 << in_page) < sh.page) ++in_page;
  const int block_mask = (1 << in_page) - 1;
  ModeLists ml;
  std::vector<ShortItem> items;
  items.reserve((size_t)((max_len <= piece ? whole : cut) / sh.hkv));
  for (int b : order) {
    const SeqInfo& s = out.seqs[b];
    int len = s.len, np = 1;  // of one piece; pieces
    if (s.len > piece) {
      len = round_up(ceil_div(s.len, ceil_div(s.len, piece)), 16);
      np = ceil_div(s.len, len);
    }
    int base = -1;
    if (np > 1) {
      base = ml.partial_rows;
      ml.partial_rows += np * s.qlen;
      for (int r = 0; r < s.qlen; ++r) ml.merge.push_back(MergeRow{s.qo + r, base + r, np, s.qlen});
    }
    for (int p = 0; p < np; ++p) {
      items.emplace_back();  // for every kv head
      ShortItem& it = items.back();
      it.q0 = s.qo;
      it.nq = s.qlen;
      it.vis = s.len - s.qlen;
      it.t0 = p * len;
      it.t1 = std::min(s.len, it.t0 + len);
      it.part = base < 0 ? -1 : base + p * s.qlen;
      it.page_off = s.page_off;
      const int nblk = ceil_div(it.t1 - it.t0, 16);
      const int per = ceil_div(nblk, waves);
      const int32_t* pg = pages + s.page_off;
      int32_t* dst = it.block;
      for (int b0 = it.t0 >> 4, end = b0 + nblk; b0 < end; b0 += per)  // a wavefront's blocks
        for (int j = 0; j < 4; ++j) {
          const int blk = std::min(b0 + j, std::min(end, b0 + per) - 1);
          *dst++ = (int32_t)(((uint32_t)pg[blk >> in_page] << in_page) + (uint32_t)(blk & block_mask));
        }
    }
  }
  if (ml.partial_rows > sh.partial_cap || ml.merge.size() > (size_t)sh.partial_cap) return false;
  out.decode_nc = max_cols <= 16 ? 16 : 32;
  out.shorts = std::move(items);
  out.mode[0] = ml;  // every row's tokens are one sequence's: the mask changes no list
  out.mode[1] = std::move(ml);
  return true;
}

// A small amount of tile work as items of half a tile's columns over their
// whole visible range, or false (leaving `ml` alone) where full-width items,
// split over the tokens and merged, are faster.
//
// While workgroups do not fill the chip an item's time is its chain of tiles:
// about 4.4 us for the launch and the first tile, then 0.93 us a tile of 64
// tokens, and little for the other items (0.2 us per 64 x 64 block of the
// call's whole area on each compute unit).  Splitting the tokens costs the
// merge launch, about 14 us however small the call, and 0.8 us per block of
// area.  So unsplit items win below a line in the longest chain that rises
// with the area, and falls where many sequences' cached K/V, which narrower
// items read twice, stand against it (a tile for every 25 KB on each compute
// unit).  All are taken exactly, not in whole tiles or items, so that
// neighbouring lengths of a prompt get the same plan.  Fitted over 4087 timed
// batches (12 head counts, prompts, chunks over a prefix, 16-row blocks, eager
// and in graphs; MI355X): 13 of them are more than 3 % slower than with
// full-width items, 1.5 us at most.  us a call, this form against those:
//   * no sequence of 512 tokens: the other list does not split either, and
//     half-width items only halve a tile's work.  12.9 / 17.3 (4 x 208 over
//     300, 16/8 heads, area 5.1), 16.0 / 18.5 (32/8, 10.3), 16.4 / 17.0 (16 x
//     48 over 298, 40/8, 9.5); from area 11 on slower, 21.0 / 19.0 (4 x 194
//     over 300, 40/8, 11.8), 30.4 / 25.2 (64 x 16 over 456, 32/4, all visible,
//     14.8).
//   * longer ones at little area: 15.6 / 18.0 (256 over 500, 16/8: 12 tiles,
//     area 2.5), 20.2 / 15.2 (64 over 1000, 16/8: 17 tiles, 1.0).
//   * prompts, 16/8: 15.2 / 18.9 (704 tokens), 17.2 / 19.7 (848), 18.3 / 19.8
//     (896, in a graph 21.9 / 21.7), 20.1 / 20.5 (992, in a graph 23.7 / 22.3),
//     25.8 / 24.9 (1328); 32/8: 23.2 / 27.5 (1024, area 16).
//   * 16-row blocks, all visible: 36.8 / 29.7 (64 over 1146, 12/2 heads, 290 KB
//     of K/V per compute unit), 33.2 / 28.4 (16 over 1043, 40/8, 265 KB).
//   * items that are whole columns already (at most 64 in a sequence) gain
//     only the merge: the line lies 3.5 tiles lower.  17.5 / 21.6 (32 x 16
//     over 250 to 500, 32/8: 8 tiles, area 6), 18.1 / 14.7 (4 x 16 over up to
//     750: 12 tiles, 1.3).
//   * past an area of 40 the chip is full and the form no longer matters or
//     loses: 24.3 / 31.8 at 20 (1024 tokens, 40/8), 52.8 / 51.1 at 51 (912 over
//     1000), 94.2 / 70.1 at 71 (64 x 16 over 2253, 32/4, all visible).
bool plan_small_tiles(const PlanShape& sh, bool causal, const BuiltPlan& bp, ModeLists& ml) {
  constexpr int64_t kMaxItems = 768;  // (a bound on the list; fuller chips are past the area's)
  const int G = sh.hq / sh.hkv;
  const int qr = kTileCols / 2 / G;  // query rows per item
  if (qr < 1) return false;
  int64_t n_items = 0, visible = 0, cached = 0;  // visible: (query row, token) pairs
  int longest = 0;
  bool halved = false;
  for (const SeqInfo& s : bp.seqs) {
    if (s.qlen * G <= kDecodeCols) continue;
    n_items += (int64_t)ceil_div(s.qlen, qr) * sh.hkv;
    const int64_t full = (int64_t)s.qlen * s.len;
    visible += causal ? full - (int64_t)s.qlen * (s.qlen - 1) / 2 : full;
    cached += s.len - s.qlen;
    longest = std::max(longest, s.len);
    halved = halved || s.qlen > qr;
  }
  if (n_items > kMaxItems) return false;
  const double area = (double)visible * sh.hq / ((double)kTileTokens * kTileTokens * sh.num_cus);
  const double cached_kb = (double)cached * sh.hkv * (2 * kHeadDim * 2) / (1024.0 * sh.num_cus);
  if (longest < 512 ? area > 11.0
                    : area > 40.0 || (double)longest / kTileTokens >
                                         (halved ? 10.5 : 7.0) + 0.62 * area - 0.04 * cached_kb)
    return false;
  std::vector<WorkItem> items;
  items.reserve((size_t)n_items);
  for (int b = 0; b < (int)bp.seqs.size(); ++b) {
    const SeqInfo& s = bp.seqs[b];
    if (s.qlen * G <= kDecodeCols) continue;
    for (int i0 = 0; i0 < s.qlen; i0 += qr) {
      const int nq = std::min(qr, s.qlen - i0);
      const int extent = causal ? std::min(s.len, s.len - s.qlen + i0 + nq) : s.len;
      for (int h = 0; h < sh.hkv; ++h)
        items.push_back(WorkItem{b, s.qo + i0, nq, h, 0, extent, -1, ceil_div(extent, kTileTokens)});
    }
  }
  ml.tile = std::move(items);
  ml.tile_rows = qr;
  assign_shares(ml.tile, sh.tile_slots, ml.tile_off, sh.num_cus);
  return true;
}

}  // namespace

int validate_shape(const PlanShape& sh, std::string& err) {
  if (sh.dim != kHeadDim) {
    err = "attention supports head_dim 128 only (got " + std::to_string(sh.dim) + ")";
    return FE_EINVAL;
  }
  if (sh.hq <= 0 || sh.hkv <= 0 || sh.hq % sh.hkv != 0) {
    err = "hq must be a positive multiple of hkv";
    return FE_EINVAL;
  }
  if (sh.hq / sh.hkv > kTileCols) {
    err = "GQA group larger than 128 query heads per kv head";
    return FE_EINVAL;
  }
  if (!is_pow2(sh.page) || sh.page < 16) {
    err = "page size must be a power of two >= 16";
    return FE_EINVAL;
  }
  if (sh.max_batch <= 0 || sh.max_pages <= 0 || sh.blocks < 0) {
    err = "max_batch and max_pages must be positive, blocks non-negative";
    return FE_EINVAL;
  }
  return FE_OK;
}

static int build_plan_impl(const PlanShape& sh, const int32_t* qo, const int32_t* kv, const int32_t* pages,
               const int32_t* last, int batch, int rows, BuiltPlan& out, std::string& err, int short_waves,
               bool small_tiles) {
  int rc = validate_shape(sh, err);
  if (rc != FE_OK) return rc;
  if (batch < 0 || rows < 0) {
    err = "negative batch or rows";
    return FE_EINVAL;
  }
  if (batch > sh.max_batch) {
    err = "attention metadata exceeds capacity: batch " + std::to_string(batch) + " > max_batch " +
          std::to_string(sh.max_batch);
    return FE_ECAPACITY;
  }
  out = BuiltPlan();
  if (batch > 0 && (qo == nullptr || kv == nullptr || last == nullptr)) {
    err = "null metadata pointer";
    return FE_EINVAL;
  }
  const int64_t max_context = (int64_t)(sh.max_pages - 1) * sh.page;
  if (batch > 0) {
    if (qo[0] < 0 || kv[0] < 0) {
      err = "qo[0] and kv[0] must be non-negative";
      return FE_EINVAL;
    }
    if ((int64_t)kv[batch] > (int64_t)sh.max_batch * sh.max_pages) {
      err = "attention metadata exceeds capacity: kv[batch] > max_batch * max_pages";
      return FE_ECAPACITY;
    }
    if (kv[batch] > 0 && pages == nullptr) {
      err = "null page table";
      return FE_EINVAL;
    }
  }
  out.seqs.resize(batch);
  for (int b = 0; b < batch; ++b) {
    const int np = kv[b + 1] - kv[b];
    const int ql = qo[b + 1] - qo[b];
    if (np < 1 || ql < 0) {
      err = "sequence " + std::to_string(b) + ": qo/kv offsets must be non-decreasing with >= 1 page";
      return FE_EINVAL;
    }
    if (last[b] < 1 || last[b] > sh.page) {
      err = "sequence " + std::to_string(b) + ": last must be in [1, page]";
      return FE_EINVAL;
    }
    const int64_t len = (int64_t)(np - 1) * sh.page + last[b];
    if (len < ql || len > max_context) {
      err = "attention context out of range for sequence " + std::to_string(b) + " (len " + std::to_string(len) +
            ", query rows " + std::to_string(ql) + ", max_context " + std::to_string(max_context) + ")";
      return FE_EINVAL;
    }
    for (int i = kv[b]; i < kv[b + 1]; ++i) {
      if (pages[i] < 0 || pages[i] > sh.blocks) {
        err = "page id " + std::to_string(pages[i]) + " outside [0, blocks]";
        return FE_EINVAL;
      }
    }
    out.seqs[b] = SeqInfo{qo[b], ql, (int32_t)len, kv[b]};
  }
  if (batch > 0 && qo[batch] > rows) {
    err = "qo[batch] exceeds rows";
    return FE_EINVAL;
  }

  if (short_waves > 0 && plan_short(sh, pages, short_waves, out)) return FE_OK;

  const int G = sh.hq / sh.hkv;
  const int slot_budget = sh.partial_cap;

  // ---- decode pieces: sequences whose (rows x group) fit one MFMA column
  // block.  Each kv head's token stream -- the decode sequences one after
  // another, each padded to whole 16-token blocks -- is cut into equal
  // shares, one per decode wavefront slot (decode_waves / hkv shares); a
  // share's pieces are its intersections with the sequences.  Every kv head
  // uses the same cut, so the wavefronts of one workgroup (consecutive kv
  // heads of one share) read the same pages at the same time.  A sequence
  // cut into several pieces is merged by log-sum-exp afterwards; when the
  // partials would not fit, shares grow (fewer wavefronts busy).
  int max_cols = 0;
  int64_t stream = 0;
  for (int b = 0; b < batch; ++b) {
    const SeqInfo& s = out.seqs[b];
    if (s.qlen > 0 && s.qlen * G <= kDecodeCols) {
      stream += round_up(s.len, 16);
      max_cols = std::max(max_cols, s.qlen * G);
    }
  }
  // columns per decode item, in 16-column MFMA blocks: 1 or 2 blocks
  out.decode_nc = max_cols <= 16 ? 16 : 32;
  const int n_static = std::max(1, sh.decode_waves / sh.hkv);
  if (stream > 0) {
    // Partial slots and pieces that a cut needs (a sequence overlapping
    // several shares is cut into pieces, each with qlen partial rows).
    auto cost_of = [&](const std::vector<int64_t>& cuts, int64_t& slots, int64_t& pieces) {
      slots = pieces = 0;
      int64_t off = 0;
      size_t k = 0;
      for (int b = 0; b < batch; ++b) {
        const SeqInfo& s = out.seqs[b];
        if (s.qlen == 0 || s.qlen * G > kDecodeCols) continue;
        const int64_t end = off + round_up(s.len, 16);
        while (cuts[k + 1] <= off) ++k;
        size_t k1 = k;
        while (cuts[k1 + 1] < end) ++k1;
        const int64_t np = (int64_t)(k1 - k + 1);
        if (np > 1) slots += np * s.qlen;
        pieces += np;
        off = end;
      }
    };
    auto fits = [&](const std::vector<int64_t>& cuts) {
      int64_t slots, pieces;
      cost_of(cuts, slots, pieces);
      return slots <= slot_budget && pieces <= sh.item_cap;
    };
    std::vector<int64_t> cuts;
    int64_t quota = std::max<int64_t>(kMinShareTokens, round_up((int)((stream + n_static - 1) / n_static), 16));
    for (;;) {
      cuts = cut_uniform(stream, quota);
      if (fits(cuts)) break;
      if (quota >= stream) {
        err = "attention metadata exceeds capacity: decode work list";
        return FE_ECAPACITY;
      }
      quota *= 2;
    }
    const int used = (int)cuts.size() - 1;
    out.decode_share_off.assign(used + 1, 0);
    int64_t off = 0;
    int share = 0;
    size_t k = 0;
    for (int b = 0; b < batch; ++b) {
      const SeqInfo& s = out.seqs[b];
      if (s.qlen == 0 || s.qlen * G > kDecodeCols) continue;
      const int64_t end = off + round_up(s.len, 16);
      while (cuts[k + 1] <= off) ++k;
      size_t k1 = k;
      while (cuts[k1 + 1] < end) ++k1;
      const int np = (int)(k1 - k + 1);
      int base = -1;
      if (np > 1) {
        base = out.decode_partials;
        out.decode_partials += np * s.qlen;
        for (int r = 0; r < s.qlen; ++r) out.decode_merge.push_back(MergeRow{s.qo + r, base + r, np, s.qlen});
      }
      for (size_t j = k; j <= k1; ++j) {
        while (share < (int)j) out.decode_share_off[++share] = (int32_t)out.decode.size();
        const int t0 = (int)(std::max<int64_t>(off, cuts[j]) - off);
        const int t1 = (int)std::min<int64_t>(s.len, std::min<int64_t>(end, cuts[j + 1]) - off);
        out.decode.push_back(
            WorkItem{b, s.qo, s.qlen, 0, t0, t1, base < 0 ? -1 : base + (int)(j - k) * s.qlen, t1 - t0});
      }
      off = end;
    }
    while (share < used) out.decode_share_off[++share] = (int32_t)out.decode.size();
    out.decode_items.resize(out.decode.size());
    for (size_t i = 0; i < out.decode.size(); ++i) {
      const WorkItem& w = out.decode[i];
      const SeqInfo& sq = out.seqs[w.seq];
      out.decode_items[i] = DecodeItem{w.q0, w.nq, sq.len, sq.page_off, w.t0, w.t1, w.part, w.seq};
    }
    auto page_of = [&](const DecodeItem& d, int tok) { return pages[d.page_off + tok / sh.page]; };
    out.decode_starts.assign(used, ShareStart{});
    for (int k = 0; k < used; ++k) {
      ShareStart& ss = out.decode_starts[k];
      ss.it_begin = out.decode_share_off[k];
      ss.it_end = out.decode_share_off[k + 1];
      if (ss.it_begin >= ss.it_end) continue;
      const DecodeItem& d = out.decode_items[ss.it_begin];
      ss.first = d;
      ss.pg0 = page_of(d, d.t0);
      if (d.t0 + 16 < d.t1) ss.pg1 = page_of(d, d.t0 + 16);
      else if (ss.it_begin + 1 < ss.it_end) {
        const DecodeItem& d2 = out.decode_items[ss.it_begin + 1];
        ss.pg1 = page_of(d2, d2.t0);
      }
    }
  }

  // ---- tile items, per mask mode.
  const int qr = kTileCols / G;  // query rows per tile item
  for (int causal = 0; causal < 2; ++causal) {
    ModeLists& ml = out.mode[causal];
    ml.partial_rows = out.decode_partials;
    ml.tile_rows = qr;
    // (q tile, kv head) pairs before splitting, to size the split factor.
    int64_t pairs = 0;
    for (int b = 0; b < batch; ++b) {
      const SeqInfo& s = out.seqs[b];
      if (s.qlen * G > kDecodeCols) pairs += (int64_t)ceil_div(s.qlen, qr) * sh.hkv;
    }
    if (pairs == 0) continue;
    if (small_tiles && plan_small_tiles(sh, causal != 0, out, ml)) continue;
    // Aim for about 8 items per compute unit (2 resident workgroups, several
    // rounds in longest-first order); never split below 256 tokens.
    int want = (int)std::max<int64_t>(1, ((int64_t)sh.num_cus * 8 + pairs - 1) / pairs);
    for (;;) {
      ml.tile.clear();
      ml.tile.reserve((size_t)std::min<int64_t>(pairs * want, sh.item_cap + 1));  // at most want pieces per pair
      ml.merge.clear();
      ml.partial_rows = out.decode_partials;
      for (int b = 0; b < batch; ++b) {
        const SeqInfo& s = out.seqs[b];
        if (s.qlen * G <= kDecodeCols) continue;
        for (int i0 = 0; i0 < s.qlen; i0 += qr) {
          const int nq = std::min(qr, s.qlen - i0);
          const int extent = causal ? std::min(s.len, s.len - s.qlen + i0 + nq) : s.len;
          int ns = std::max(1, std::min(want, extent / 256));
          int chunk = round_up(ceil_div(extent, ns), kTileTokens);
          ns = ceil_div(extent, chunk);
          int base = -1;
          if (ns > 1) {
            base = ml.partial_rows;
            ml.partial_rows += ns * nq;
            for (int r = 0; r < nq; ++r) ml.merge.push_back(MergeRow{s.qo + i0 + r, base + r, ns, nq});
          }
          for (int sp = 0; sp < ns; ++sp) {
            const int t0 = sp * chunk;
            const int t1 = std::min(extent, t0 + chunk);
            // Cost ~ tiles times the 16-column blocks each wavefront
            // computes (1 for items of <= 64 columns, else 2).
            const int cost = ceil_div(t1 - t0, kTileTokens) * (nq * G > kTileCols / 2 ? 2 : 1);
            for (int h = 0; h < sh.hkv; ++h)
              ml.tile.push_back(WorkItem{b, s.qo + i0, nq, h, t0, t1, base < 0 ? -1 : base + sp * nq, cost});
          }
        }
      }
      if (ml.partial_rows <= slot_budget && ml.tile.size() <= (size_t)sh.item_cap) break;
      if (want == 1) {
        err = "attention metadata exceeds capacity: tile work list (" + std::to_string(ml.tile.size()) + " items)";
        return FE_ECAPACITY;
      }
      want = std::max(1, want / 2);
    }
    // Two tile workgroups share each CU; the first of the pair to be
    // dispatched (workgroup b < num_cus) wins the SIMDs' issue arbitration
    // and, at equal work, finished the 8192-token prefill in 184 us against
    // 230 us for the second.  The first ones therefore get more of the work:
    // 3/2 of the second's measured fastest (0.261 against 0.267 ms for equal
    // shares; 4/3 gained 1 %, 2/1 lost), since the second speeds up once its
    // partner has finished.
    assign_shares(ml.tile, sh.tile_slots, ml.tile_off, sh.num_cus);
    // When the longest-first list had to split chunks anyway, an equal cut
    // of the tile stream balances the workgroups to within a tile, usually
    // with fewer pieces; it replaces the list if it needs no more partial rows.
    if (ml.partial_rows > out.decode_partials) {
      ModeLists cut;
      if (cut_tile_stream(out.seqs, G, sh.hkv, causal != 0, sh.tile_slots, out.decode_partials, slot_budget,
                          sh.item_cap, cut) &&
          cut.partial_rows <= ml.partial_rows)
        ml = std::move(cut);
    }
  }
  for (int causal = 0; causal < 2; ++causal) {
    std::vector<MergeRow>& m = out.mode[causal].merge;
    m.insert(m.begin(), out.decode_merge.begin(), out.decode_merge.end());
    if (m.size() > (size_t)slot_budget) {
      err = "attention metadata exceeds capacity: merge rows";
      return FE_ECAPACITY;
    }
  }
  return FE_OK;
}

int build_plan(const PlanShape& sh, const int32_t* qo, const int32_t* kv, const int32_t* pages,
               const int32_t* last, int batch, int rows, BuiltPlan& out, std::string& err, int short_waves,
               bool small_tiles) {
  try {
    return build_plan_impl(sh, qo, kv, pages, last, batch, rows, out, err, short_waves, small_tiles);
  } catch (const std::bad_alloc&) {
    err = "out of host memory while building the work lists";
    return FE_ENOMEM;
  }
}

}  // namespace feattn

