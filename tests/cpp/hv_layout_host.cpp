// Host checks of what the H.v kernels read of a layout (no device).  Each
// check prints "<name> <mismatches> <checked>".
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

int main() {
  shared_low_table();
  segment_order();
  return 0;
}
