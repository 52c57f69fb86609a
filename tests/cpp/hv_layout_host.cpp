// Host checks of what the H.v kernels read of a layout (no device).  Each
// check prints "<name> <mismatches> <checked>".
#include <cmath>
#include <cstdio>
#include <random>

#include "ed_layout.hpp"

using namespace alps_ed;

static ModelSpec ring(int N, int n_up) {
  ModelSpec s;
  s.n_sites = N;
  s.n_up = n_up;
  for (int i = 0; i < N; ++i) {
    s.bonds.push_back(make_bond(i, (i + 1) % N, 1.0, 1.0, 0.0));
    s.sites.push_back(make_site(0.0, 0.0));
  }
  return s;
}

static void report(const char* name, long bad, long checked) { std::printf("%s %ld %ld\n", name, bad, checked); }

// The low-low target table is made once for all sectors of a lattice, and an
// operator's layout holds no copy of it.
static void shared_low_table() {
  long bad = 0, n = 0;
  const SectorLayout first = build_layout(ring(23, 8), -1, false);
  for (int k : {8, 9, 7, 15, 8}) {
    const SectorLayout L = build_layout(ring(23, k), -1, false);
    bad += !L.nbp16.empty() || low_flip_table(L) != low_flip_table(first);
    ++n;
  }
  bad += low_flip_table(build_layout(ring(11, 5), -1, false)) == low_flip_table(first);
  report("shared_low_table", bad, n + 1);
}

// Large layouts: the segments of XCD g (positions g, g + 8, ...) are, class by
// class, one of the eight runs of the class ordered by the set bits of the low
// five bits of the high word and then by address (by address alone, in four
// slices, past 16384 segments), in ascending address.
static void segment_order() {
  long bad = 0, n = 0;
  const int cases[][2] = {{21, 10}, {22, 11}, {22, 5}, {23, 15}, {24, 12}, {25, 9}, {26, 13}, {28, 14}, {30, 15}};
  for (const auto& c : cases) {
    const SectorLayout L = build_layout(ring(c[0], c[1]), -1, false);
    size_t at = 0;
    while (at < L.proc_hi.size()) {
      const int pc = __builtin_popcount(L.proc_hi[at]);
      std::vector<uint32_t> v;
      for (uint32_t h : L.seg_hi)
        if (__builtin_popcount(h) == pc) v.push_back(h);
      const bool keyed = v.size() <= 16384;
      if (keyed)
        std::stable_sort(v.begin(), v.end(), [](uint32_t a, uint32_t b) {
          return __builtin_popcount(a & 31u) < __builtin_popcount(b & 31u);
        });
      const size_t slice = keyed ? v.size() : (v.size() + 3) / 4;
      for (size_t s0 = 0; s0 < v.size(); s0 += slice) {
        const size_t cnt = std::min(slice, v.size() - s0), run = cnt / kXcds;
        for (int g = 0; g < kXcds; ++g) {
          std::vector<uint32_t> want(v.begin() + s0 + g * run, v.begin() + s0 + (g + 1) * run), got;
          std::sort(want.begin(), want.end());
          for (size_t p = at; p < at + run * kXcds; ++p)
            if ((int)(p % kXcds) == g) got.push_back(L.proc_hi[p]);
          bad += got != want;
          ++n;
        }
        const std::vector<uint32_t> tail(v.begin() + s0 + run * kXcds, v.begin() + s0 + cnt);
        bad += !std::equal(tail.begin(), tail.end(), L.proc_hi.begin() + at + run * kXcds);
        at += cnt;
      }
    }
  }
  report("segment_order", bad, n);
}

// The first row of the segment of a high word: the rank of its smallest state.
static uint32_t first_row(const SectorLayout& L, uint32_t h) {
  const int kl = L.k - __builtin_popcount(h);
  if (kl < 0 || kl > L.B) return 0xffffffffu;
  const uint32_t st = (h << L.B) | ((1u << kl) - 1u);
  uint64_t r = 0;
  int m = 0;
  for (int p = 0; p < L.N; ++p)
    if (st >> p & 1u) r += binom(p, ++m);
  return (uint32_t)r;
}

// Page positions are linear over xor and distinct for words of one parity.
static void page_positions() {
  long bad = 0, n = 0;
  for (int B = 1; B <= 12; ++B) {
    const uint32_t nlo = 1u << B, np = std::max(1u, nlo / 2);
    std::vector<int> seen(2 * np, 0);
    for (uint32_t a = 0; a < nlo; ++a, ++n) {
      const uint32_t at = page_pos(a);
      bad += at >= np || seen[(__builtin_popcount(a) & 1) * np + at]++ != 0;
      for (int p = 0; p < B; ++p) bad += page_pos(a ^ (1u << p)) != (at ^ page_pos(1u << p));
    }
    const LowTables& T = low_tables(B);
    for (uint32_t i = 0; i < nlo; ++i) bad += T.lo_word[i] != T.lo_state[i] || T.lo_page[i] != 8 * page_pos(T.lo_state[i]);
  }
  report("page_positions", bad, n);
}

// What a segment stages for the cross bonds, and their share of its rows'
// diagonal, against the bonds: one entry per segment, so that sectors of few
// up spins among many high words stay small.
static void cross_stages_of_segments() {
  long bad = 0, n = 0;
  std::mt19937 rng(3);
  std::uniform_real_distribution<double> U(-1, 1);
  const int cases[][2] = {{14, 7}, {16, 8}, {17, 3}, {20, 10}, {20, 2}, {20, 18}, {22, 11}, {24, 2}};
  for (const auto& c : cases) {
    ModelSpec s = ring(c[0], c[1]);
    const int high = c[0] - 12;
    for (int b = 0; b < 8 * high; ++b)
      s.bonds.push_back(make_bond((int)(rng() % high), high + (int)(rng() % 12), U(rng), U(rng), U(rng)));
    const SectorLayout L = build_layout(s, -1, false, true);
    const size_t ng = L.xb_grp.size(), ns = L.seg_hi.size();
    bad += !L.stage || L.xs.size() != ns * ng || L.xw.size() != ns * kXwStride || !L.xb_nb.empty();
    if (bad) break;
    for (size_t q = 0; q < ns; ++q) {
      const uint32_t h = L.seg_hi[q];
      bad += L.seg_hi[L.proc_index[q]] != L.proc_hi[q];
      size_t i = 0;
      for (int set = 1; set >= 0; --set)
        for (uint32_t bit = 1; bit < (1u << L.NH); bit <<= 1) {
          size_t b0 = 0, b1 = 0;
          for (size_t b = 0; b < L.xb.size(); ++b)
            if (L.xb[b].hbit == bit) {
              if (b1 == 0) b0 = b;
              b1 = b + 1;
            }
          const uint32_t nb = first_row(L, h ^ bit);
          if (b1 == 0 || ((h & bit) != 0u) != (set == 1) || nb == 0xffffffffu) continue;
          const XStage st = L.xs[q * ng + i++];
          bad += st.nb != nb || (int)(st.info >> 31) != set || (st.info & 0xffffu) != b0 ||
                 (st.info >> 16 & 0x7fffu) != b1 - b0;
          ++n;
        }
      for (; i < ng; ++i) bad += L.xs[q * ng + i].info != 0u;
      const int kl = L.k - __builtin_popcount(h);
      for (uint32_t r = L.lo_class_off[kl]; r < L.lo_class_off[kl + 1]; r += 1 + rng() % 64) {
        const uint32_t lo = L.low->lo_state[r];
        double want = 0, got = L.xw[q * kXwStride + L.B];
        for (const CrossBond& x : L.xb)
          if (((lo & x.lbit) != 0u) != ((h & x.hbit) != 0u)) want += x.e_anti - x.e_par;
        for (int p = 0; p < L.B; ++p)
          if (lo >> p & 1u) got += L.xw[q * kXwStride + p];
        bad += !(std::abs(got - want) < 1e-11);  // at most 112 terms below 2, added twice
        ++n;
      }
    }
    for (size_t b = 0; b < L.xb.size(); ++b)
      bad += L.xb_p[b].t != L.xb[b].t || L.xb_p[b].m != 8 * page_pos(L.xb[b].lbit);
  }
  report("cross_stages", bad, n);
}

// Any number of cross bonds has a layout; more than a stage can name are
// gathered.
static void many_cross_bonds() {
  long bad = 0, n = 0;
  for (int count : {0x7fff, 0x8000}) {
    ModelSpec s;
    s.n_sites = 14;
    s.n_up = 7;
    for (int i = 0; i < 14; ++i) s.sites.push_back(make_site(0.0, 0.0));
    for (int b = 0; b < count; ++b) s.bonds.push_back(make_bond(b & 1, 2 + b % 12, 1.0, 1.0, 0.0));
    try {
      const SectorLayout L = build_layout(s, -1, false);
      bad += L.stage != (count <= 0x7fff) || L.xb.size() != (size_t)count;
    } catch (const std::exception&) {
      ++bad;
    }
    ++n;
  }
  report("many_cross_bonds", bad, n);
}

int main() {
  many_cross_bonds();
  shared_low_table();
  segment_order();
  page_positions();
  cross_stages_of_segments();
  return 0;
}
