// index_check.cpp - a host-side walk of every thread of the render kernels'
// launches through the same index code the kernels run (sample_index.hpp), with
// every index checked against the length of the buffer it addresses (the
// lengths the engine allocates: prepare_common, render_hw, render_sa).
//
// For a frame set (nframes frames of nr x nc in a sample order) it checks:
//  * the start kernels (plain and series): each (workgroup, tile, j, thread) of
//    the launch grid: the tile's frame span, the sample's frame (and that the
//    one-frame shortcut names the sample's own frame), its position, the column /
//    row table entries, the cardioid-mask word, the tile-skip entry, and the
//    per-sample, per-wave (hand-on word) and per-tile stores;
//  * k_scatter: for hand-on words with pseudo-random bits on the valid sample
//    ids, its word loads, and that the positions it writes are exactly
//    0 .. count - 1, each once, in sample order;
//  * k_emit: every sample's output element of the row-major grids, and that the
//    valid samples cover every pixel of every frame exactly once;
//  * the active-list chunks of both iterate kernels (every run length) for a
//    range of list lengths: every entry read below the length, each entry taken
//    once, the waves' own first chunks each taken once, and the claim ranges
//    partitioning the chunks.
// Test support, not part of the render path: built as its own library and called
// from the CPU tests.
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <limits>
#include <vector>

#include "coords.hpp"
#include "hpfloat.hpp"
#include "orbit_steps.hpp"
#include "sample_index.hpp"
#include "series_chain.hpp"

namespace {

struct Report {
  unsigned long long violations = 0, checked = 0;
  char* msg;
  int cap;
  void fail(const char* fmt, ...) {
    if (violations++ == 0 && msg && cap > 0) {
      va_list ap;
      va_start(ap, fmt);
      std::vsnprintf(msg, (size_t)cap, fmt, ap);
      va_end(ap);
    }
  }
  bool in(uint64_t idx, uint64_t len, const char* what, uint64_t gid) {
    checked++;
    if (idx < len) return true;
    fail("%s index %llu >= length %llu (sample %llu)", what, (unsigned long long)idx, (unsigned long long)len,
         (unsigned long long)gid);
    return false;
  }
};

// the slot caps of the engine's start and iterate launches
constexpr uint64_t kStartSlots = 4096;

}  // namespace

extern "C" {

// Returns the number of violations (0: every index in bounds, every pixel
// covered once); msg gets the first.  mask: frames carry cardioid masks;
// skip_T: tile side of per-tile series skips (0: none).  plant (the checker's
// own negative controls, 0 for none): 1 moves the last frame's column tables
// one entry on, 2 gives the frames one sample more than the sample order has,
// 3 interleaves the plain chunks with one chunk too few, 4 counts a lane's own
// bit into its scatter position, 5 launches the tile scan with one group too few,
// 6 selects the next set bit in the sparse scatter.
long long nm_index_check(int nr, int nc, int nframes, int tile, int num_cu, int mask, int skip_T, int plant,
                         char* msg, int cap, unsigned long long* checked) {
  using namespace nm;
  Report R;
  R.msg = msg;
  R.cap = cap;
  if (msg && cap > 0) msg[0] = 0;
  if (nr <= 0 || nc <= 0 || nframes <= 0 || num_cu <= 0) return -1;
  const uint64_t fs = frame_samples(nr, nc, tile);
  if (fs == 0) return -1;
  const uint64_t total64 = fs * (uint64_t)nframes;
  if (total64 >= 0xFFFFF000ull) return -2;  // the engine refuses it (prepare_common)
  const uint32_t total = (uint32_t)total64;
  // the frame records and buffer lengths as render_hw / render_sa build them
  const uint64_t mask_words = ((uint64_t)nr * nc + 31) / 32;
  std::vector<DevFrame> df;
  for (int k = 0; k < nframes; k++) {
    DevFrame d = make_frame((uint64_t)k, nr, nc, tile, (uint32_t)fs);
    d.tab_c = (uint32_t)((uint64_t)k * nc);
    d.tab_r = (uint32_t)((uint64_t)k * nr);
    d.mask_base = mask ? (uint64_t)k * mask_words * 32 : 0;
    if (plant == 1 && k == nframes - 1) d.tab_c += 1;
    if (plant == 2) d.sample_base = (uint32_t)((uint64_t)k * (fs + 1));
    df.push_back(d);
  }
  const double inv_frame = 1.0 / (double)(plant == 2 ? fs + 1 : fs);
  const uint64_t ncol = (uint64_t)nframes * nc, nrow = (uint64_t)nframes * nr;
  const uint64_t nmask = mask ? (uint64_t)nframes * mask_words : 1;
  const uint64_t nout = (uint64_t)nframes * nr * nc;
  const uint32_t ntiles = start_tiles(total);
  const uint32_t sk_ntc = skip_T ? (uint32_t)((nc + skip_T - 1) / skip_T) : 0;
  const uint32_t sk_tpf = skip_T ? sk_ntc * (uint32_t)((nr + skip_T - 1) / skip_T) : 0;
  const uint64_t nskip = (uint64_t)sk_tpf * nframes;
  std::vector<uint8_t> seen(nout, 0);

  // ---- the start kernels
  const int grid = start_grid(total, num_cu, kStartSlots);
  for (int b = 0; b < grid; b++)
    for (uint32_t t = (uint32_t)b; t < ntiles; t += (uint32_t)grid) {
      for (uint32_t w = 0; w < (uint32_t)kCountsPerTile; w++)
        R.in(count_index(t, w), start_counts(total), "start counts", t);
      uint32_t f0, f1;
      tile_frame_span(t, total, inv_frame, &f0, &f1);
      R.in(f0, (uint64_t)nframes, "frames (tile span)", (uint64_t)t * kTile);
      R.in(f1, (uint64_t)nframes, "frames (tile span)", (uint64_t)t * kTile);
      for (int j = 0; j < kPerThread; j++)
        for (uint32_t tid = 0; tid < (uint32_t)kThreads; tid++) {
          const uint32_t gid = start_gid(t, j, tid);
          if (tid % 64 == 0) {  // lane 0 stores the wave's hand-on word, idle waves too
            if (gid % 64) R.fail("wave of sample %u does not start a hand-on word", gid);
            R.in(hand_word(gid), hand_words(total), "hand-on words", gid);
          }
          if (gid >= total) continue;  // an idle lane: the kernels load and store nothing else for it
          const uint32_t fi = f0 == f1 ? f0 : frame_of(gid, inv_frame);
          if (fi != gid / fs) R.fail("sample %u: frame %u, want %llu", gid, fi, (unsigned long long)(gid / fs));
          if (frame_of(gid, inv_frame) != gid / fs) R.fail("sample %u: frame_of is not the quotient", gid);
          if (!R.in(fi, (uint64_t)nframes, "frames", gid)) continue;
          const DevFrame& f = df[fi];
          if (gid < f.sample_base) {
            R.fail("sample %u below its frame's base %u", gid, f.sample_base);
            continue;
          }
          const uint32_t local = gid - f.sample_base;
          R.in(local, fs, "frame-local sample", gid);
          R.in(gid, total, "out/flag/state/state_i/r2", gid);
          const Loc lc = locate(f, local);
          if (!lc.valid) continue;  // tile padding: only its flag is written
          R.in(lc.r, f.nr, "row", gid);
          R.in(lc.c, f.nc, "column", gid);
          R.in((uint64_t)f.tab_c + lc.c, ncol, "column tables (cre, crelo, epsre)", gid);
          R.in((uint64_t)f.tab_r + lc.r, nrow, "row tables (cim, cimlo, epsim)", gid);
          if (mask) R.in((f.mask_base + (uint64_t)lc.r * f.nc + lc.c) >> 5, nmask, "cardioid mask", gid);
          if (skip_T)
            R.in((uint64_t)fi * sk_tpf + (lc.r / (uint32_t)skip_T) * sk_ntc + lc.c / (uint32_t)skip_T, nskip,
                 "tile skips", gid);
        }
    }

  // ---- k_scatter over hand-on words with pseudo-random bits on valid ids: tiles
  // in turn about 3 in 8, 1 in 16 and 1 in 64 marked, and none (the kernel's
  // dense and sparse paths)
  auto marked = [](uint32_t gid, uint64_t x) {
    static const uint64_t dens[4] = {24, 4, 1, 0};
    return (x & 63) < dens[(gid / kTile) % 4];
  };
  {
    const uint32_t nwords = hand_words(total);
    std::vector<uint64_t> words(nwords, 0);
    uint64_t x = 0x9E3779B97F4A7C15ull ^ total;
    for (uint32_t gid = 0; gid < total; gid++) {
      x ^= x << 13;
      x ^= x >> 7;
      x ^= x << 17;
      if (marked(gid, x)) words[hand_word(gid)] |= 1ull << (gid % 64);
    }
    std::vector<uint32_t> off(ntiles, 0);
    uint64_t count = 0;
    for (uint32_t t = 0; t < ntiles; t++) {
      off[t] = (uint32_t)count;
      for (int k = 0; k < kHandWordsPerTile; k++) count += (uint64_t)__builtin_popcountll(words[t * kHandWordsPerTile + k]);
    }
    std::vector<int64_t> at(count, -1);
    for (uint32_t t = 0; t < ntiles; t++) {
      uint32_t before = 0;
      for (int k = 0; k < kHandWordsPerTile; k++) {
        const uint64_t wi = (uint64_t)t * kHandWordsPerTile + k;
        if (!R.in(wi, nwords, "hand-on words (scatter)", (uint64_t)t * kTile)) continue;
        const uint64_t w = words[wi];
        for (uint32_t l = 0; l < 64; l++) {
          if (!((w >> l) & 1ull)) continue;
          const uint32_t gid = t * kTile + (uint32_t)k * 64 + l;
          const uint32_t pos = hand_position(off[t], before, w, plant == 4 ? l + 1 : l);
          if (!R.in(pos, count, "active (scatter)", gid)) continue;
          if (at[pos] >= 0) R.fail("active position %u written twice (sample %u)", pos, gid);
          at[pos] = gid;
        }
        before += (uint32_t)__builtin_popcountll(w);
      }
    }
    // the sparse-tile path (tiles with at most kScatterSparse marked samples):
    // lane j of batch p0 takes entry p = p0 + j, the last word k whose prefix
    // is <= p (the kernel's 4-step search) and bit select_bit(w_k, p - before_k)
    for (uint32_t t = 0; t < ntiles; t++) {
      uint32_t pre[kHandWordsPerTile], m = 0;
      for (int k = 0; k < kHandWordsPerTile; k++) {
        pre[k] = m;
        m += (uint32_t)__builtin_popcountll(words[(uint64_t)t * kHandWordsPerTile + k]);
      }
      if (m > kScatterSparse) continue;
      for (uint32_t p0 = 0; p0 < m; p0 += 64)
        for (uint32_t j = 0; j < 64; j++) {
          const uint32_t p = p0 + j;
          int k = 0;
          for (int step = kHandWordsPerTile / 2; step >= 1; step >>= 1)
            if (pre[k + step] <= p) k += step;
          if (p >= m) continue;
          const uint64_t wk = words[(uint64_t)t * kHandWordsPerTile + k];
          const uint32_t gid = t * kTile + (uint32_t)k * 64 + select_bit(wk, p - pre[k] + (plant == 6 ? 1u : 0u));
          if (!R.in((uint64_t)off[t] + p, count, "active (sparse scatter)", gid)) continue;
          if (at[off[t] + p] != (int64_t)gid)
            R.fail("sparse scatter: tile %u entry %u takes sample %u, want %lld", t, p, gid, (long long)at[off[t] + p]);
        }
    }
    // select_bit against a bit-by-bit walk
    {
      uint64_t y = 0x2545F4914F6CDD1Dull ^ total;
      for (int trial = 0; trial < 2000; trial++) {
        y ^= y << 13;
        y ^= y >> 7;
        y ^= y << 17;
        const uint64_t w = trial < 3 ? (trial == 0 ? 1ull : trial == 1 ? ~0ull : 1ull << 63) : y & (y >> (trial % 7));
        uint32_t r = 0;
        for (uint32_t b = 0; b < 64; b++)
          if ((w >> b) & 1ull) {
            if (select_bit(w, r) != b) R.fail("select_bit(%llx, %u) = %u, want %u", (unsigned long long)w, r,
                                              select_bit(w, r), b);
            r++;
          }
      }
    }
    for (uint64_t p = 0; p < count; p++) {
      if (at[p] < 0) {
        R.fail("active position %llu written by no sample", (unsigned long long)p);
        break;
      }
      if (p && at[p] <= at[p - 1]) {
        R.fail("active position %llu out of sample order", (unsigned long long)p);
        break;
      }
    }
  }

  // ---- the tile scan (k_tile_sums, then k_scan_tiles) over the scatter's tile
  // counts: every thread's loads and stores, the groups' carries and the total;
  // plant 5 launches one group too few
  {
    std::vector<uint32_t> cnt(ntiles), seq(ntiles);
    uint64_t acc = 0;
    {  // the marked samples of the scatter check's generator, per tile
      uint64_t x = 0x9E3779B97F4A7C15ull ^ total;
      for (uint32_t gid = 0; gid < total; gid++) {
        x ^= x << 13;
        x ^= x >> 7;
        x ^= x << 17;
        if (marked(gid, x)) cnt[gid / kTile]++;
      }
    }
    for (uint32_t t = 0; t < ntiles; t++) {
      seq[t] = (uint32_t)acc;
      acc += cnt[t];
    }
    const ScanSplit sp = scan_split(ntiles);
    const uint32_t groups = plant == 5 ? sp.groups - 1 : sp.groups;
    if (sp.groups < 1 || sp.groups > kScanGroups) R.fail("tile scan of %u counts: %u groups", ntiles, sp.groups);
    std::vector<uint32_t> gsum(groups, 0), out(ntiles, 0);
    std::vector<uint8_t> wrote(ntiles, 0);
    for (int pass = 0; pass < 2; pass++) {  // 0: k_tile_sums, 1: k_scan_tiles
      for (uint32_t g = 0; g < groups; g++) {
        uint32_t lo, hi;
        scan_group_range(ntiles, sp.per, g, lo, hi);
        uint32_t carry = 0;
        for (uint32_t q = 0; q < g; q++) carry += gsum[q];
        for (uint32_t base = lo; base < hi; base += kScanRound) {
          uint32_t before = 0;  // the counts of the round's earlier threads (the wave scans)
          for (uint32_t tid = 0; tid < 1024; tid++) {
            const uint32_t i0 = base + 16 * tid;
            uint32_t mine = 0;
            for (uint32_t k = 0; k < 16; k++) {
              if (i0 + k >= hi) continue;
              if (!R.in(i0 + k, ntiles, "tile counts (scan)", (uint64_t)g)) continue;
              if (pass == 1) {
                if (wrote[i0 + k]++) R.fail("tile offset %u written twice", i0 + k);
                out[i0 + k] = carry + before + mine;
              }
              mine += cnt[i0 + k];
            }
            before += mine;
          }
          carry += before;
          if (pass == 0) gsum[g] += before;
        }
        if (pass == 1 && g + 1 == groups && carry != (uint32_t)acc)
          R.fail("tile scan total %u, want %llu", carry, (unsigned long long)acc);
      }
    }
    for (uint32_t t = 0; t < ntiles; t++)
      if (!wrote[t] || out[t] != seq[t]) {
        R.fail("tile offset %u: %s %u, want %u", t, wrote[t] ? "wrote" : "not written", out[t], seq[t]);
        break;
      }
    // the split at edge sizes: at most kScanGroups groups of consecutive,
    // non-empty count ranges covering [0, ntiles)
    const uint32_t edge[] = {0u, 1u, kScanRound - 1, kScanRound, kScanRound + 1, kScanGroups * kScanRound,
                             kScanGroups * kScanRound + 1, 100 * kScanRound + 7, start_counts(0xFFFFEFFFu), start_counts(total), ntiles};
    for (uint32_t n : edge) {
      const ScanSplit e = scan_split(n);
      if (e.groups < 1 || e.groups > kScanGroups) R.fail("tile scan of %u counts: %u groups", n, e.groups);
      uint32_t next = 0;
      for (uint32_t g = 0; g < e.groups; g++) {
        uint32_t lo, hi;
        scan_group_range(n, e.per, g, lo, hi);
        if (lo != next || hi < lo || (n > 0 && hi == lo))
          R.fail("tile scan of %u counts: group %u covers [%u, %u) after %u", n, g, lo, hi, next);
        next = hi;
      }
      if (next != n) R.fail("tile scan of %u counts: the groups end at %u", n, next);
    }
  }

  // ---- k_emit: sample order -> the row-major grids
  for (uint32_t gid = 0; gid < total; gid++) {
    const uint32_t fi = frame_of(gid, inv_frame);
    if (!R.in(fi, (uint64_t)nframes, "frames (emit)", gid)) continue;
    const DevFrame& f = df[fi];
    const Loc lc = locate(f, gid - f.sample_base);
    if (!lc.valid) continue;
    const uint64_t o = f.out_base + (uint64_t)lc.r * f.nc + lc.c;
    if (!R.in(o, nout, "grid", gid)) continue;
    if (seen[o]++) R.fail("grid element %llu written twice (sample %u)", (unsigned long long)o, gid);
  }
  for (uint64_t o = 0; o < nout; o++)
    if (!seen[o]) {
      R.fail("grid element %llu written by no sample", (unsigned long long)o);
      break;
    }

  // ---- the iterate kernels' chunks of an active list of n entries
  std::vector<uint64_t> lens = {0, 1, 3, 4, 63, 64, 65, 255, 256, 257, 1000, 4095, 4097};
  lens.push_back(total / 3);
  lens.push_back(total > 0 ? total - 1 : 0);
  lens.push_back(total);
  std::vector<uint8_t> took;
  for (uint64_t n64 : lens) {
    if (n64 > total) continue;
    const uint32_t n = (uint32_t)n64, nch = chunk_count(n);
    // claim ranges: a partition of [0, nch)
    uint32_t next = 0;
    for (uint32_t h = 0; h < (uint32_t)kQueues; h++) {
      const uint32_t lo = claim_lo(nch, h), hi = claim_lo(nch, h + 1);
      if (lo != next || hi < lo) R.fail("claim range %u of %u chunks: [%u, %u) after %u", h, nch, lo, hi, next);
      next = hi;
    }
    if (next != nch) R.fail("claim ranges end at %u of %u chunks", next, nch);
    // a launch's waves: their own first chunks and the claimed rest, each chunk once
    for (const uint32_t grid : {1u, 2u, 7u, (uint32_t)num_cu * 4u})
      for (const uint32_t wpw : {4u, 8u}) {
        const uint32_t waves = grid * wpw, base = nch < waves ? nch : waves;
        std::vector<uint8_t> first(nch, 0);
        for (uint32_t b = 0; b < grid; b++)
          for (uint32_t w = 0; w < wpw; w++) {
            const uint32_t c = first_chunk(w, b, grid);
            if (c < base && first[c]++) R.fail("chunk %u of %u is the first of two waves (grid %u)", c, nch, grid);
            if (c < base && b >= base) R.fail("workgroup %u of %u leaves before its chunk %u", b, grid, c);
          }
        for (uint32_t c = 0; c < base; c++)
          if (!first[c]) {
            R.fail("chunk %u of %u is no wave's first (grid %u)", c, nch, grid);
            break;
          }
        R.checked += base;
      }
    // interleaved chunks: runs of 1 (plain), runs of 1 .. 64 (series: 64 is 64
    // consecutive entries); plant 3 interleaves the plain chunks with one too few
    for (uint32_t shift = 0; shift <= 7; shift++) {  // 7: the plain kernel's own chunk_pos
      took.assign(n, 0);
      const uint32_t nchp = plant == 3 && shift == 7 && nch > 1 ? nch - 1 : nch;
      for (uint32_t c = 0; c < nch; c++) {
        uint32_t items = 0;
        auto at = [&](uint32_t l) { return shift == 7 ? chunk_pos(l, c, nchp) : chunk_pos_run(l, c, nchp, shift); };
        for (uint32_t l = 0; l < (uint32_t)kChunk; l++) items += at(l) < n;
        for (uint32_t l = 0; l < (uint32_t)kChunk; l++) {
          const uint32_t p = at(l);
          if ((l < items) != (p < n))
            R.fail("chunk %u of %u entries (shift %u): the lanes with entries are not a prefix", c, n, shift);
          if (l < items && R.in(p, n, "active (chunks)", c) && took[p]++)
            R.fail("active entry %u taken twice (shift %u)", p, shift);
        }
      }
      for (uint32_t p = 0; p < n; p++)
        if (!took[p]) {
          R.fail("active entry %u of %u taken by no chunk (shift %u)", p, n, shift);
          break;
        }
    }
  }
  if (checked) *checked = R.checked;
  return (long long)R.violations;
}


// tree_first_le against a linear scan: `len` thresholds from a seed (some +-inf,
// many equal), every start, values below, at, between and above them.  Returns the
// number of differing answers.
long long nm_tree_check(int len, unsigned seed) {
  if (len <= 0) return -1;
  uint32_t leaves = 1;
  while (leaves < (uint32_t)len) leaves <<= 1;
  const double inf = std::numeric_limits<double>::infinity();
  std::vector<double> tree(2 * (size_t)leaves, inf);
  std::vector<double> vals = {-inf, -1.0, 41.0};
  unsigned s = seed;
  for (int i = 0; i < len; i++) {
    s = s * 1664525u + 1013904223u;
    const unsigned r = s >> 24;
    const double t = r < 8 ? inf : r < 12 ? -inf : (double)(r % 41);
    tree[leaves + (size_t)i] = t;
  }
  for (int v = 0; v < 41; v += 5) vals.push_back(v), vals.push_back(v + 0.5);
  for (size_t k = leaves - 1; k >= 1; k--) tree[k] = std::min(tree[2 * k], tree[2 * k + 1]);
  long long bad = 0;
  for (double v : vals) {
    int want = len;  // first i >= lo with T_i <= v, from the end
    for (int lo = len; lo >= 0; lo--) {
      if (lo < len && tree[leaves + (size_t)lo] <= v) want = lo;
      bad += nm::tree_first_le(tree.data(), leaves, len, lo, v) != want;
    }
  }
  return bad;
}

// The engine's record of whose tables are on the device: a set's are its own after
// they were written whole, and nobody's from the first write of another set's on, also
// where those then fail.  Returns the number of wrong answers.
long long nm_table_key_check() {
  nm::TableKey k;
  long long bad = k.holds(0, -1) + k.holds(0, 0) + k.holds(5, 0);
  k.writing();
  k.written(5, 32);
  bad += !k.holds(5, 32) + k.holds(5, 0) + k.holds(6, 32) + k.holds(0, 32);
  k.writing();  // set 6's records are under way, and fail
  bad += k.holds(5, 32) + k.holds(6, 32) + k.holds(0, 32);
  k.writing();
  k.written(0, 32);  // a set without a serial
  return bad + k.holds(0, 32) + k.holds(5, 32);
}

// The device's coordinate entries against hpfloat.cpp: `n` cases from a seed, with
// random mantissas (some sparse), exponents, signs and offsets, every combination of
// precisions that `ML` limbs hold; the truncated coordinate, its remainder and the
// truncated difference from a reference point near it.  Returns the number of cases
// that differ in a bit.
}  // extern "C"
namespace {
uint64_t next_u64(uint64_t& s) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
nm::HpVal val_of(const nm::hpf& v) {
  nm::HpVal d;
  std::memcpy((void*)&d, (const void*)&v, sizeof d);
  return d;
}
// as mandelbrot.cpp's get_d_nearest
double nearest(const nm::hpf& a) {
  const double t = a.get_d();
  if (a.sign == 0 || !std::isfinite(t)) return t;
  nm::hpf td(2), r(a.L), half(2);
  nm::hp_set_d(td, t);
  nm::hp_sub(r, a, td);
  if (r.sign == 0) return t;
  const double up = std::nextafter(t, a.sign > 0 ? INFINITY : -INFINITY);
  nm::hp_set_d(half, (up - t) * 0.5);
  r.sign = half.sign = 1;
  const int c = nm::hp_cmp(r, half);
  uint64_t bits;
  std::memcpy(&bits, &t, 8);
  return c > 0 || (c == 0 && (bits & 1)) ? up : t;
}
// The orbit tables' arithmetic: sums, differences and products of random values at
// random precisions, and the nearest double, from exponents near 0 to the ends of the
// doubles' range and far past it.
template <int ML>
long long hp_ops_check(unsigned seed, int n) {
  uint64_t s = seed;
  long long bad = 0;
  for (int t = 0; t < n; t++) {
    const int L = 1 + (int)(next_u64(s) % ML);
    const int64_t range = t % 4 == 0 ? 3 : t % 4 == 1 ? 64 * ML + 130 : t % 4 == 2 ? 1100 : 40000;
    auto random_hpf = [&] {
      nm::hpf v(L);
      if (next_u64(s) % 16 == 0) return v;  // zero
      const int kind = (int)(next_u64(s) % 5);
      for (int i = 0; i < v.L; i++) v.m[i] = kind == 0 ? 0 : kind == 1 ? ~0ull : next_u64(s);
      if (kind == 3) v.m[v.L - 1] &= ~0ull << 10;  // a double and half of its last bit, or nearly
      if (kind == 4) v.m[v.L - 1] |= (1ull << 10) - 1;
      v.m[v.L - 1] |= 1ull << 63;
      v.sign = next_u64(s) & 1 ? 1 : -1;
      v.exp = (int64_t)(next_u64(s) % (uint64_t)(2 * range)) - range;
      return v;
    };
    const nm::hpf a = random_hpf();
    nm::hpf b = random_hpf();
    if (a.sign && t % 7 == 0) {  // cancellation down to the last limb
      b = a;
      b.sign = -a.sign;
      b.m[0] ^= next_u64(s) % 3;
    }
    const auto da = nm::hpd_load<ML>(val_of(a)), db = nm::hpd_load<ML>(val_of(b));
    auto differ = [&](const nm::hpd<ML>& x, const nm::hpf& y) {
      const auto z = nm::hpd_load<ML>(val_of(y));
      return x.sign != z.sign || (z.sign && (x.exp != z.exp || std::memcmp(x.m, z.m, sizeof x.m) != 0));
    };
    nm::hpf sum(L), less(L), product(L);
    nm::hp_add(sum, a, b);
    nm::hp_sub(less, a, b);
    nm::hp_mul(product, a, b);
    const double want = nearest(a), got = nm::hpd_nearest(da, L);
    bad += differ(nm::hpd_add(da, db, 1, L), sum) || differ(nm::hpd_add(da, db, -1, L), less) ||
           differ(nm::hpd_mul(da, db, L), product) || std::memcmp(&want, &got, 8) != 0;
  }
  return bad;
}
template <int ML>
long long coords_check(unsigned seed, int n) {
  uint64_t s = seed;
  auto random_hpf = [&](int64_t e) {
    nm::hpf v(1 + (int)(next_u64(s) % ML));
    if (next_u64(s) % 16 == 0) return v;  // zero
    const int kind = (int)(next_u64(s) % 4);
    for (int i = 0; i < v.L; i++) v.m[i] = kind == 0 ? 0 : kind == 1 ? ~0ull : next_u64(s);
    if (kind == 3 && v.L > 2) v.m[1] = 0;
    v.m[v.L - 1] |= 1ull << 63;
    v.sign = next_u64(s) & 1 ? 1 : -1;
    v.exp = e;
    return v;
  };
  auto same = [](double a, double b) { return std::memcmp(&a, &b, 8) == 0 || a == b; };
  long long bad = 0;
  for (int t = 0; t < n; t++) {
    const int L = 1 + (int)(next_u64(s) % ML);
    const nm::hpf c = random_hpf((int64_t)(next_u64(s) % 5) - 2);
    const nm::hpf z = random_hpf(-(int64_t)(next_u64(s) % (next_u64(s) % 2 ? 40 : 64 * ML + 80)));
    const long k = (long)(next_u64(s) % 16385) - 8192;
    nm::hpf step(L), p(L), x0(L), y(L), td(2), rem(L);
    nm::hp_mul_si(step, z, k);
    nm::hp_add(p, c, step);
    if (next_u64(s) % 2) nm::hp_set(x0, c);  // a reference point: the centre, or one step off
    else nm::hp_add(x0, c, z);
    nm::hp_sub(y, p, x0);
    const double hi = p.get_d();
    nm::hp_set_d(td, hi);
    nm::hp_sub(rem, p, td);
    const double lo = nearest(rem);
    const auto q = nm::hpd_pixel<ML>(val_of(c), val_of(z), k, L);
    const double dy = nm::hpd_get_d(nm::hpd_add(q, nm::hpd_load<ML>(val_of(x0)), -1, L));
    // the remainder serves the plain path alone, whose sample size is at least
    // 1.5e-16: it stays far above the subnormal doubles
    const bool rest = rem.sign == 0 || rem.exp > -900;
    bad += !same(nm::hpd_get_d(q), hi) || (rest && !same(nm::hpd_rest(q), lo)) || !same(dy, y.get_d());
  }
  return bad;
}

// The device's passes over an orbit (orbit.hip's sweeps, terms and emission, one value
// after the other) against the host's chain.  out[0]: the bound (orbit_tables_hold)
// accepts; out[1]: doubles, mantissas or exponents that differ; out[2]: the most bits
// that cancelled in one step of A; out[3]: values off from the host's by more than
// their bound; out[4]: the largest such difference in units of the bound, times 2^10.
template <int ML>
long long orbit_check(const std::vector<nm::HPComplex>& X, int len, int L, long long* out) {
  typedef nm::hpd<ML> V;
  const int n = len - 1, c = std::max(1, (int)std::ceil(std::cbrt((double)n)));
  const int n1 = (n + c - 1) / c, n2 = (n1 + c - 1) / c;
  std::vector<V> x(2 * (size_t)(len + 1));
  std::vector<double> Zd(2 * (size_t)(len + 2), 0.0);
  bool real = true;
  for (int k = 0; k <= len; k++)
    for (int p = 0; p < 2; p++) {
      const nm::hpf& v = p ? X[k].im : X[k].re;
      x[2 * (size_t)k + p] = nm::hpd_load<ML>(val_of(v));
      Zd[2 * (size_t)(k + 1) + p] = nm::hpd_nearest(x[2 * (size_t)k + p], L);
      if (p && k < len && v.sign) real = false;
    }
  // chunk q of the elements, v = factor v + terms; as orbit.hip's k_sweep
  auto sweep = [&](const std::vector<V>& f, const V* u1, const V* u2, bool twice, bool one, int count, int chunk,
                   const V* start, int first, V* end, V* before, V* after, V* product) {
    for (int side = 0; side < (product ? 2 : 1); side++)
      for (int q = 0; q * chunk < count; q++) {
        V v[2] = {nm::hpd_small<ML>(side ? 1 : first), nm::hpd_small<ML>(0)};
        if (start && !side) v[0] = start[2 * q], v[1] = start[2 * q + 1];
        for (int e = q * chunk; e < std::min(count, (q + 1) * chunk); e++) {
          V s[2];
          for (int p = 0; p < 2; p++) {
            if (before && !side) before[2 * e + p] = v[p];
            s[p] = nm::sweep_part(p, f[2 * e], f[2 * e + 1], v[p], v[1 - p], twice, one && !side,
                                  u1 && !side ? u1 + 2 * e + p : nullptr, u2 && !side ? u2 + 2 * e + p : nullptr, L);
          }
          for (int p = 0; p < 2; p++) {
            v[p] = s[p];
            if (after && !side) after[2 * e + p] = s[p];
          }
        }
        for (int p = 0; p < 2; p++) {
          if (side) product[2 * q + p] = v[p];
          else if (end) end[2 * q + p] = v[p];
        }
      }
  };
  std::vector<V> P1(2 * n1), E1(2 * n1), S1(2 * n1), P2(2 * n2), E2(2 * n2), S2(2 * n2), y[3], u1(2 * n), u2(2 * n);
  std::vector<V> chain[3];  // the host's chain: one chunk
  std::vector<double> trace(3 * (size_t)len, -1.0);
  std::fill(trace.begin(), trace.begin() + 3 * (c + 1), 0.0);
  std::vector<uint16_t> run[3];
  std::vector<int32_t> gap[3], ex[3];
  nm::SaReferenceHost r;
  nm::series_chain(X.data(), len, L, r);
  const std::vector<double>*hd[3] = {&r.A, &r.B, &r.C}, *hm[3] = {&r.Am, &r.Bm, &r.Cm};
  const std::vector<int32_t>* he[3] = {&r.Ae, &r.Be, &r.Ce};
  out[1] = out[2] = 0;
  for (int k = 0; k < 3; k++) {
    chain[k].assign(2 * (size_t)len, nm::hpd_small<ML>(0));
    chain[k][0] = nm::hpd_small<ML>(k == 0);
    y[k] = chain[k];
    auto terms = [&](const std::vector<V>* v) {
      for (int e = 0; k && e < n; e++)
        for (int p = 0; p < 2; p++)
          nm::terms_part(p, &v[0][2 * (e + 1)], k == 2 ? &v[1][2 * (e + 1)] : nullptr, L, u1[2 * e + p], u2[2 * e + p]);
    };
    const V *t1 = k ? u1.data() : nullptr, *t2 = k ? u2.data() : nullptr;
    terms(chain);
    sweep(x, t1, t2, true, k == 0, n, n, nullptr, k == 0, nullptr, nullptr, chain[k].data() + 2, nullptr);
    terms(y);
    sweep(x, t1, t2, true, k == 0, n, c, nullptr, 0, E1.data(), nullptr, nullptr, k ? nullptr : P1.data());
    sweep(P1, E1.data(), nullptr, false, false, n1, c, nullptr, 0, E2.data(), nullptr, nullptr, k ? nullptr : P2.data());
    sweep(P2, E2.data(), nullptr, false, false, n2, n2, nullptr, k == 0, nullptr, S2.data(), nullptr, nullptr);
    sweep(P1, E1.data(), nullptr, false, false, n1, c, S2.data(), 0, nullptr, S1.data(), nullptr, nullptr);
    sweep(x, t1, t2, true, k == 0, n, c, S1.data(), 0, E1.data(), nullptr, y[k].data() + 2, nullptr);
    for (int t = 0; t < 2 * (n1 - 1); t++) {
      const V g = nm::hpd_add(S1[t + 2], E1[t], -1, L);
      gap[k].push_back(g.sign ? (int32_t)g.exp : nm::kFxZeroExp);
    }
    for (size_t t = 0; t < 2 * (size_t)len; t++) {
      const V& v = y[k][t];
      const double m = v.sign ? v.sign * std::ldexp((double)(v.m[ML - 1] >> 11), -53) : 0.0;
      ex[k].push_back(v.sign ? (int32_t)v.exp : nm::kFxZeroExp);
      run[k].push_back(nm::hpd_run(v, L));
      const double d = nm::hpd_get_d(v);
      out[1] += d != (*hd[k])[t] || m != (*hm[k])[t] || ex[k][t] != (*he[k])[t];
    }
  }
  out[0] = nm::orbit_tables_hold(Zd.data(), len, L, c, real, {ex[0].data(), ex[1].data(), ex[2].data()},
                                 {run[0].data(), run[1].data(), run[2].data()},
                                 {gap[0].data(), gap[1].data(), gap[2].data()}, trace.data());
  int worst = 0;
  out[3] = out[4] = 0;
  for (int k = 0; k < 3; k++)
    for (size_t t = 0; t < 2 * (size_t)len; t++) {
      const double b = trace[3 * (t / 2) + k];
      const V g = nm::hpd_add(y[k][t], chain[k][t], -1, L);
      if (b < 0.0 || g.sign == 0) continue;  // not reached; the same
      const int E = std::max(ex[k][t | 1], ex[k][t & ~(size_t)1]);
      const double off = std::ldexp(0.5 * (1.0 + (double)(g.m[ML - 1] << 1) * 0x1p-64), (int)(g.exp - E) + 64 * L - 1);
      out[3] += off > b;
      out[4] = std::max<long long>(out[4], b > 0.0 ? (long long)(off / b * 1024.0) : 1024);
    }
  for (int i = 1; i < len; i++) {
    const int e0 = std::max(ex[0][2 * (size_t)i - 2], ex[0][2 * (size_t)i - 1]),
              e1 = std::max(ex[0][2 * (size_t)i], ex[0][2 * (size_t)i + 1]);
    const int ez = std::ilogb(std::hypot(Zd[2 * (size_t)i], Zd[2 * (size_t)i + 1]));
    worst = std::max(worst, std::max(e0 + ez + 1, 0) - e1);
  }
  out[2] = worst;
  return 0;
}
}  // namespace
extern "C" {
// An orbit of `len` from (re, im) at L limbs through orbit_check.  out: accepted,
// differing entries, the most bits that cancelled in a step of A.  cancel > 0: not the
// point's own orbit, but after every `cancel` steps an x that all but cancels A's step
// (to a double's last bits).
long long nm_orbit_check(const char* re, const char* im, int L, int len, int cancel, long long* out) {
  std::vector<nm::HPComplex> X;
  nm::HPComplex c, z;
  for (nm::hpf* v : {&c.re, &c.im, &z.re, &z.im}) *v = nm::hpf(L), v->L = L;
  if (!nm::hp_set_str(c.re, re) || !nm::hp_set_str(c.im, im)) return -1;
  nm::hp_copy_prec(z.re, c.re);
  nm::hp_copy_prec(z.im, c.im);
  nm::hpf t1(L), t2(L), ar(L), ai(L), br(L), bi(L), one(L);
  nm::hp_set_d(one, 1.0);
  nm::hp_set_d(ar, 1.0);
  for (int k = 0; k <= len; k++) {
    nm::HPComplex w;
    w.re = nm::hpf(L), w.im = nm::hpf(L);
    nm::hp_copy_prec(w.re, z.re);
    nm::hp_copy_prec(w.im, z.im);
    if (cancel > 0 && k % cancel == cancel - 1) {  // 2 x A = -1: x = -conj(A) / (2 |A|^2)
      long er, ei;
      double mr = ar.get_d_2exp(&er), mi = ai.get_d_2exp(&ei);
      const long e = std::max(ar.sign ? er : -1000000l, ai.sign ? ei : -1000000l);
      mr = ar.sign ? std::ldexp(mr, (int)std::max(-1000l, er - e)) : 0.0;
      mi = ai.sign ? std::ldexp(mi, (int)std::max(-1000l, ei - e)) : 0.0;
      const double q = 2.0 * (mr * mr + mi * mi);
      nm::hp_set_d(w.re, -mr / q);
      nm::hp_set_d(w.im, mi / q);
      if (w.re.sign) w.re.exp -= e;
      if (w.im.sign) w.im.exp -= e;
    }
    X.push_back(w);
    // A's next value, for where to cancel
    nm::hp_mul(br, w.re, ar); nm::hp_mul(t1, w.im, ai); nm::hp_sub(br, br, t1); nm::times2(br); nm::hp_add(br, br, one);
    nm::hp_mul(bi, w.re, ai); nm::hp_mul(t1, w.im, ar); nm::hp_add(bi, bi, t1); nm::times2(bi);
    nm::hp_copy_prec(ar, br);
    nm::hp_copy_prec(ai, bi);
    nm::hp_mul(t1, z.re, z.re); nm::hp_mul(t2, z.im, z.im); nm::hp_sub(t1, t1, t2);
    nm::hp_mul(t2, z.re, z.im); nm::times2(t2);
    nm::hp_add(z.re, t1, c.re);
    nm::hp_add(z.im, t2, c.im);
  }
  if (L <= 4) return orbit_check<4>(X, len, L, out);
  if (L <= 8) return orbit_check<8>(X, len, L, out);
  return L <= 16 ? orbit_check<16>(X, len, L, out) : -1;
}
long long nm_hp_ops_check(int limbs, unsigned seed, int n) {
  switch (limbs) {
    case 4: return hp_ops_check<4>(seed, n);
    case 6: return hp_ops_check<6>(seed, n);
    case 8: return hp_ops_check<8>(seed, n);
    case 16: return hp_ops_check<16>(seed, n);
    default: return -1;
  }
}
long long nm_coords_check(int limbs, unsigned seed, int n) {
  switch (limbs) {
    case 4: return coords_check<4>(seed, n);
    case 8: return coords_check<8>(seed, n);
    case 16: return coords_check<16>(seed, n);
    case 40: return coords_check<40>(seed, n);
    default: return -1;
  }
}
}  // extern "C"
