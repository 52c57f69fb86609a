// ed_measure.hip -- expectation values of spin operators in a vector of a
// fixed-Sz sector, for the eigenvector measurements of
// DiagMatrix::perform_measurements (applications/diag/diag.h:191-314), which
// evaluates <v| O |v> (SparseDiagMatrix::calculate, sparsediag.h:151-159)
// for site terms, site-pair terms and bond terms built from Sz, S+ and S-.
//
// Every such term is a combination of two families of sums over the rows r
// of the sector (w_r = v_r^2, s_i(r) = +-1/2 the Sz of site i in row r):
//   - diagonal moments: sum w, sum w s_i, sum w s_i s_j for all sites;
//   - flip amplitudes F(i,j) = sum over rows with site j up and site i down
//     of v_r v_r', r' the row with both spins turned (<v|S+_i S-_j|v>).
//
// Each comes from a pass over the vector that leaves one partial per workgroup
// and value, and a launch that adds the partials in a fixed order
// (sum_parts_kernel); the host picks the sites' entries from the sums.
// All sums are FP64 and deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ed_device.hpp"
#include "ed_kernels.hpp"

namespace alps_ed {

namespace {

using namespace dev;

constexpr int kPairChunk = 8;  // site pairs per workgroup of the flip kernel

__device__ __forceinline__ double half_spin(uint32_t word, int bit) { return ((word >> bit) & 1u) ? 0.5 : -0.5; }

typedef double d4 __attribute__((ext_vector_type(4)));

// FP64 matrix product D += A B, 16x16 by 4 deep: lane l holds A[l%16][l/16]
// and B[l/16][l%16], and D[4v + l/16][l%16] in element v.
__device__ __forceinline__ d4 mma16(double a, double b, d4 d) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, d, 0, 0, 0);
}

// The next larger word with as many set bits.
__device__ __forceinline__ uint32_t next_same_popcount(uint32_t h) {
  const uint32_t c = h & (0u - h), r = h + c;
  return r | (((h ^ r) >> 2) >> __builtin_ctz(h));
}

struct Binomials {
  uint32_t c[kMaxHigh + 1][kMaxHigh + 1];
  constexpr Binomials() : c() {
    for (int n = 0; n <= kMaxHigh; ++n) {
      c[n][0] = 1u;
      for (int p = 1; p <= n; ++p) c[n][p] = c[n - 1][p - 1] + (p < n ? c[n - 1][p] : 0u);
    }
  }
};
__constant__ const Binomials kBinom{};

// Word number i, ascending, of the n-bit words with p set bits.
__device__ __forceinline__ uint32_t word_with_popcount(uint32_t i, int p, int n) {
  uint32_t h = 0u;
  for (int b = n - 1; b >= 0 && p > 0; --b) {
    const uint32_t c = p <= b ? kBinom.c[b][p] : 0u;  // words with bit b clear
    if (i >= c) {
      h |= 1u << b;
      i -= c;
      --p;
    }
  }
  return h;
}

// Sum over the lanes, of four values at once: lane l returns the sum of w[l % 4].
__device__ __forceinline__ double wave_sum4(const double (&w)[4], uint32_t lane) {
  const bool o1 = (lane & 1u) != 0u, o2 = (lane & 2u) != 0u;
  const double a = (o1 ? w[1] : w[0]) + __shfl_xor(o1 ? w[0] : w[1], 1, 64);
  const double b = (o1 ? w[3] : w[2]) + __shfl_xor(o1 ? w[2] : w[3], 1, 64);
  double c = (o2 ? b : a) + __shfl_xor(o2 ? a : b, 2, 64);
#pragma unroll
  for (int off = 4; off < 64; off <<= 1) c += __shfl_xor(c, off, 64);
  return c;
}

// Sums over a workgroup's rows: blocks of 256 rows of the segments of one
// class (popcount kl of the low word), whose low words are the same in every
// segment, so each thread keeps one low word and adds over the segments
// w, and w s_b for every high bit b.  The low bits come in at the end, once
// per workgroup, as two products on the matrix cores,
//   M[a][c] = sum_r s_a(r) col_c(r),  P[a][b] = sum_r s_a(r) s_b(r) col_0(r)
// with s_0 = 1 and col_0 = w (index 0: no bit).  Pairs of high bits need only
// the segment's sum of w: lane l adds those of every fourth segment for the
// pairs (b, b + d mod NHX), (d - 1) NHX + b = l / 4 + 16 t.
// At 24 sites (FP64, 21.6 MB of v: 3 us at the rate of a copy of that size)
// 25 us, against 166 us for 79 sums per segment and 2.8 ms for adding them up
// over the segments with a thread per output; bound by the chain first
// segment -> rows -> products -> partial sums of its 4096 waves and by 12
// FP64 multiply-adds and the cross-lane sum per row.
template <class V, int NHX>
__global__ __launch_bounds__(kBlock) void moments_kernel(DevLayout L, MomentPlan P, const V* __restrict__ v,
                                                         double* __restrict__ part) {
  constexpr int kCols = 1 + NHX, kStride = 65, kPairs = (NHX * (NHX / 2) + 15) / 16;
  constexpr int kTiles = kCols > 16 ? 3 : 2, kIdx = moment_values(NHX);
  static_assert(kIdx == kTiles * 256 + 16 * kPairs, "partial layout");
  constexpr int kWaveDoubles = kCols * kStride + 32;
  static_assert(kIdx <= kWaveDoubles, "the results reuse the columns' place");
  extern __shared__ __align__(16) double mom_lds[];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  int kl = 0;
  while (blockIdx.x >= P.first[kl + 1]) ++kl;
  const uint32_t cls0 = ldc(L.lo_class_off + kl), len = ldc(L.lo_class_off + kl + 1) - cls0;
  const uint32_t nrb = (len + kBlock - 1) / kBlock, loc = blockIdx.x - P.first[kl];
  const uint32_t s0 = loc / nrb * P.chunk, s1 = s0 + P.chunk < P.count[kl] ? s0 + P.chunk : P.count[kl];
  const uint32_t r = loc % nrb * kBlock + tid;
  const bool in = r < len;
  const uint32_t off = lane_off((in ? r : len - 1u) * (uint32_t)sizeof(V));
  double col[kCols], hh[kPairs];
  uint32_t pm[kPairs];
#pragma unroll
  for (int c = 0; c < kCols; ++c) col[c] = 0.0;
#pragma unroll
  for (int t = 0; t < kPairs; ++t) {
    const uint32_t p = lane / 4u + 16u * t, b = p % NHX, d = p / NHX + 1u;
    hh[t] = 0.0;
    pm[t] = (1u << b) | (1u << ((b + d) % NHX));
  }
  uint32_t h = word_with_popcount(s0, L.k - kl, L.NH);
  for (uint32_t s = s0; s < s1; s += 4) {
    uint32_t hs[4];
    V x[4];
    double w[4];
    // past the last segment the last one again, with weight 0
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      hs[u] = h;
      if (s + u + 1 < s1) h = next_same_popcount(h);
      x[u] = ld_at<V>(v + ldc(L.hi_base + hs[u]), off);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      w[u] = in && s + u < s1 ? (double)x[u] * (double)x[u] : 0.0;
      col[0] += w[u];
#pragma unroll
      for (int b = 0; b < NHX; ++b) col[1 + b] = fma(w[u], ((hs[u] >> b) & 1u) != 0u ? 0.5 : -0.5, col[1 + b]);
    }
    const double ws = wave_sum4(w, lane);
    const uint32_t hw = (lane & 2u) ? ((lane & 1u) ? hs[3] : hs[2]) : ((lane & 1u) ? hs[1] : hs[0]);
#pragma unroll
    for (int t = 0; t < kPairs; ++t) hh[t] += (__builtin_popcount(hw & pm[t]) & 1) ? -ws : ws;
  }
  double* const wl = mom_lds + wave * kWaveDoubles;
  uint32_t* const lo_s = reinterpret_cast<uint32_t*>(wl + kCols * kStride);
#pragma unroll
  for (int c = 0; c < kCols; ++c) wl[c * kStride + lane] = col[c];
  lo_s[lane] = L.lo_state[cls0 + (in ? r : len - 1u)];
  __syncthreads();
  const int i = (int)(lane & 15u), kq = (int)(lane >> 4);
  d4 m0 = {0.0, 0.0, 0.0, 0.0}, m1 = m0, pp = m0;
  for (int row = kq; row < 64; row += 4) {
    const double a = i == 0 ? 1.0 : i <= L.B ? half_spin(lo_s[row], i - 1) : 0.0;
    m0 = mma16(a, i < kCols ? wl[i * kStride + row] : 0.0, m0);
    pp = mma16(a, a * wl[row], pp);
    if (kCols > 16) m1 = mma16(a, 16 + i < kCols ? wl[(16 + i) * kStride + row] : 0.0, m1);
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int at = (4 * e + kq) * 16 + i;
    wl[at] = m0[e];
    wl[256 + at] = pp[e];
    if (kCols > 16) wl[512 + at] = m1[e];
  }
#pragma unroll
  for (int t = 0; t < kPairs; ++t) {
    hh[t] += __shfl_xor(hh[t], 1, 64);
    hh[t] += __shfl_xor(hh[t], 2, 64);
    if ((lane & 3u) == 0u) wl[kTiles * 256 + lane / 4u + 16u * t] = hh[t];
  }
  __syncthreads();
  for (uint32_t e = tid; e < (uint32_t)kIdx; e += kBlock) {
    double sum = 0.0;
#pragma unroll
    for (int q = 0; q < kBlock / 64; ++q) sum += mom_lds[q * kWaveDoubles + e];
    part[(size_t)blockIdx.x * kIdx + e] = sum;
  }
}

// out[e] = the sum of part[b * n + e] over the nb workgroups of the kernel
// before: 16 entries a workgroup, 64 threads each.
__global__ __launch_bounds__(1024) void sum_parts_kernel(const double* __restrict__ part, uint32_t nb, uint32_t n,
                                                         double* __restrict__ out) {
  __shared__ double red[64][17];
  const uint32_t c = threadIdx.x & 15u, q = threadIdx.x >> 4, e = blockIdx.x * 16u + c;
  double acc = 0.0;
  if (e < n)
#pragma unroll 4
    for (uint32_t b = q; b < nb; b += 64u) acc += part[(size_t)b * n + e];
  red[q][c] = acc;
  __syncthreads();
  if (threadIdx.x < 16u && e < n) {
    double s = 0.0;
    for (int t = 0; t < 64; ++t) s += red[t][threadIdx.x];
    out[e] = s;
  }
}

// Flip amplitudes of all site pairs at once, as the Gram matrix of the states
// with one spin less up: F(i, j) = sum over the words g with k - 1 set bits of
// f_i(g) f_j(g), f_i(g) = v(g with bit i) where g has it clear, 0 where it has
// it set.  A workgroup takes high words h; the rows are the low words of class
// k - 1 - popcount(h).  For a low bit f is an element of the segment of h,
// read from its LDS page at the row's position xor the bit's (words that have
// the bit lead to a place that holds 0); for a high bit it is the same row of
// the segment of h with that bit.  The lanes hold the operand of the FP64
// matrix product as it is, bit lane % 16 of a tile of 16 (tile 0 the low
// bits, the next the high ones) by rows lane / 16; both operands of a product
// have the same form.  G is symmetric: tiles (a, b) with a <= b only.
// The high words are those of the segments, in the order of H.v (longest class
// first: the workgroups' shares are alike), then the n_last ones whose rows
// have all low bits set.
// Bound by the matrix cores: 3 products of 64 clocks per 4 rows, 49 us at 24
// sites (2.5 M words g), where it takes 90 us (the pair kernel, eight pairs a
// pass over v, 810 us for the 276 pairs, and 256 us for a thread per pair to
// add its partials); the rest is filling the pages, one segment after another.
template <class V, int HT>
__global__ __launch_bounds__(kBlock) void flip_gram_kernel(DevLayout L, uint32_t n_last,
                                                           const V* __restrict__ v, double* __restrict__ part) {
  typedef V V4 __attribute__((ext_vector_type(4), aligned(sizeof(V))));
  typedef uint16_t u16x4 __attribute__((ext_vector_type(4), aligned(2)));
  constexpr int NT = gram_tiles(HT);
  const uint32_t tid = threadIdx.x, lane = tid & 63u, i = lane & 15u, kq = lane >> 4;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const bool low = (int)i < L.B;
  const uint32_t bit_pos = 8u * (((1u << i) ^ ((1u << i) >> 1)) >> 1);  // 8 * page_pos(1 << i)
  d4 g[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) g[t] = d4{0.0, 0.0, 0.0, 0.0};
  for (uint32_t n = blockIdx.x; n < L.n_seg + n_last; n += gridDim.x) {
    const uint32_t h = n < L.n_seg ? ldc(L.proc_hi + n) : word_with_popcount(n - L.n_seg, L.k - 1 - L.B, L.NH);
    const int kg = L.k - 1 - __builtin_popcount(h);
    if (kg < 0) continue;  // uniform
    const uint32_t cls = ldc(L.lo_class_off + kg), cls1 = ldc(L.lo_class_off + kg + 1), len = cls1 - cls;
    __syncthreads();  // every wave is done with the page
    clear_page<kBlock>(L.B);
    __syncthreads();
    if (kg < L.B) {
      const uint32_t len1 = ldc(L.lo_class_off + kg + 2) - cls1;
      const V* seg = v + ldc(L.hi_base + h);
      for (uint32_t r = tid; r < len1; r += kBlock) lds_st<double>(L.lo_page[cls1 + r], (double)seg[r]);
    }
    __syncthreads();
    const V* nb[HT];
    bool ok[HT];
#pragma unroll
    for (int t = 0; t < HT; ++t) {
      const uint32_t b = i + 16u * t;
      ok[t] = (int)b < L.NH && ((h >> b) & 1u) == 0u;
      nb[t] = ok[t] ? v + L.hi_base[h | (1u << b)] : v;  // a segment of the rows' class
    }
    for (uint32_t r0 = 16u * wave; r0 < len; r0 += 16u * (kBlock / 64)) {
      const uint32_t r = r0 + 4u * kq;  // this lane's rows r .. r + 3
      double f[1 + HT][4];
      uint32_t pos[4];
      if (r0 + 16u <= len) {  // uniform
        const u16x4 p4 = *reinterpret_cast<const u16x4*>(L.lo_page + cls + r);
#pragma unroll
        for (int t = 0; t < HT; ++t) {
          V4 x = {(V)0, (V)0, (V)0, (V)0};
          if (ok[t]) x = *reinterpret_cast<const V4*>(nb[t] + r);
#pragma unroll
          for (int q = 0; q < 4; ++q) f[1 + t][q] = (double)x[q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) pos[q] = p4[q];
#pragma unroll
        for (int q = 0; q < 4; ++q) f[0][q] = low ? lds_ld<double>(pos[q] ^ bit_pos) : 0.0;
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const bool in = r + q < len;
          pos[q] = in ? L.lo_page[cls + r + q] : 0u;
          f[0][q] = in && low ? lds_ld<double>(pos[q] ^ bit_pos) : 0.0;
#pragma unroll
          for (int t = 0; t < HT; ++t) f[1 + t][q] = in && ok[t] ? (double)nb[t][r + q] : 0.0;
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int b = 0; b <= HT; ++b)
#pragma unroll
          for (int a = 0; a <= b; ++a) g[gram_tiles(b - 1) + a] = mma16(f[a][q], f[b][q], g[gram_tiles(b - 1) + a]);
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    __syncthreads();
#pragma unroll
    for (uint32_t e = 0; e < 4; ++e) lds_st<double>(2048u * wave + 8u * ((4u * e + kq) * 16u + i), g[t][e]);
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (uint32_t q = 0; q < kBlock / 64; ++q) s += lds_ld<double>(2048u * q + 8u * tid);
    part[((size_t)blockIdx.x * NT + t) * 256u + tid] = s;
  }
}

// Flip amplitudes of the pairs [blockIdx.y*8, +8): masks[2p] is the bit of
// site j (must be up), masks[2p+1] the bit of site i (must be down).
template <class V>
__global__ __launch_bounds__(kBlock) void flip_pairs_kernel(DevLayout L, const V* __restrict__ v,
                                                            const uint32_t* __restrict__ masks, int n_pairs,
                                                            double* __restrict__ part) {
  const int p0 = (int)blockIdx.y * kPairChunk;
  const int np = n_pairs - p0 < kPairChunk ? n_pairs - p0 : kPairChunk;
  uint32_t mu[kPairChunk], md[kPairChunk];
#pragma unroll
  for (int q = 0; q < kPairChunk; ++q) {
    mu[q] = q < np ? masks[2 * (p0 + q)] : 0u;
    md[q] = q < np ? masks[2 * (p0 + q) + 1] : 0u;
  }
  const uint32_t lomask = L.B >= 32 ? 0xffffffffu : ((1u << L.B) - 1u);
  double acc[kPairChunk];
#pragma unroll
  for (int q = 0; q < kPairChunk; ++q) acc[q] = 0.0;
  for (uint32_t s = blockIdx.x; s < L.n_seg; s += gridDim.x) {
    const uint32_t h = L.seg_hi[s];
    const int kl = L.k - __builtin_popcount(h);
    const uint32_t cls0 = L.lo_class_off[kl];
    const uint32_t len = L.lo_class_off[kl + 1] - cls0;
    const uint32_t base = L.hi_base[h];
    for (uint32_t r = threadIdx.x; r < len; r += kBlock) {
      const uint32_t st = (L.NH > 0 ? (h << L.B) : 0u) | L.lo_state[cls0 + r];
      const double x = (double)v[base + r];
#pragma unroll
      for (int q = 0; q < kPairChunk; ++q) {
        if (q < np && (st & mu[q]) != 0u && (st & md[q]) == 0u) {
          const uint32_t t = st ^ mu[q] ^ md[q];
          const uint32_t rr = L.hi_base[L.NH > 0 ? (t >> L.B) : 0u] + L.lo_rank[t & lomask];
          acc[q] += x * (double)v[rr];
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < kPairChunk; ++q) {
    const double bs = block_sum_all(acc[q]);
    if (threadIdx.x == 0 && q < np) part[(size_t)(p0 + q) * gridDim.x + blockIdx.x] = bs;
  }
}

// out[p] = the sum of pair p's partials, one workgroup a pair.
__global__ __launch_bounds__(kBlock) void flip_combine_kernel(const double* __restrict__ part, uint32_t nbx,
                                                              double* __restrict__ out) {
  double acc = 0.0;
  for (uint32_t b = threadIdx.x; b < nbx; b += kBlock) acc += part[(size_t)blockIdx.x * nbx + b];
  const double s = block_sum_all(acc);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

uint64_t choose(int n, int p) {
  if (p < 0 || p > n) return 0;
  uint64_t c = 1;
  for (int i = 1; i <= p; ++i) c = c * (uint64_t)(n - p + i) / (uint64_t)i;
  return c;
}

void launch_sum_parts(const double* part, uint32_t nb, uint32_t n, double* out, hipStream_t st) {
  hipLaunchKernelGGL(sum_parts_kernel, dim3((n + 15u) / 16u), dim3(1024), 0, st, part, nb, n, out);
}

}  // namespace

MomentPlan moment_plan(const DevLayout& L) {
  MomentPlan P{};
  uint64_t blocks = 0;  // of 256 rows of a segment
  for (int kl = 0; kl <= L.B; ++kl) {
    P.count[kl] = (uint32_t)choose(L.NH, L.k - kl);
    blocks += P.count[kl] * ((choose(L.B, kl) + kBlock - 1) / kBlock);
  }
  P.chunk = (uint32_t)std::max<uint64_t>(1, (blocks + kMomentBlocks - 1) / kMomentBlocks);
  for (int kl = 0; kl <= L.B; ++kl)
    P.first[kl + 1] = P.first[kl] + (uint32_t)((P.count[kl] + P.chunk - 1) / P.chunk *
                                               ((choose(L.B, kl) + kBlock - 1) / kBlock));
  P.blocks = P.first[L.B + 1];
  return P;
}

template <class V>
hipError_t launch_spin_moments(const DevLayout& L, const MomentPlan& P, const V* v, double* part, double* out,
                               hipStream_t st) {
  const int nhx = moment_high_bits(L.NH);
  const size_t lds = (size_t)(kBlock / 64) * ((1 + nhx) * 65 + 32) * sizeof(double);
  if (nhx == 12)
    hipLaunchKernelGGL((moments_kernel<V, 12>), dim3(P.blocks), dim3(kBlock), lds, st, L, P, v, part);
  else
    hipLaunchKernelGGL((moments_kernel<V, kMaxHigh>), dim3(P.blocks), dim3(kBlock), lds, st, L, P, v, part);
  launch_sum_parts(part, P.blocks, (uint32_t)moment_values(nhx), out, st);
  return hipGetLastError();
}

void read_moments(const DevLayout& L, const double* sums, double* norm2, double* sz, double* szsz) {
  const int N = L.N, B = L.B, nhx = moment_high_bits(L.NH);
  const double* const pp = sums + 256;
  const double* const hh = sums + (nhx > 15 ? 768 : 512);
  auto m = [&](int a, int c) { return c < 16 ? sums[a * 16 + c] : sums[512 + a * 16 + c - 16]; };
  if (norm2) *norm2 = m(0, 0);
  for (int i = 0; i < N; ++i) {
    const int p = N - 1 - i;
    if (sz) sz[i] = p < B ? m(1 + p, 0) : m(0, 1 + p - B);
    for (int j = 0; szsz && j < N; ++j) {
      const int q = N - 1 - j, lo = std::min(p, q), hi = std::max(p, q);
      double e;
      if (i == j) {
        e = 0.25 * m(0, 0);
      } else if (hi < B) {
        e = pp[(1 + lo) * 16 + 1 + hi];
      } else if (lo < B) {
        e = m(1 + lo, 1 + hi - B);
      } else {
        const int d = hi - lo;
        e = 0.25 * (d <= nhx / 2 ? hh[(d - 1) * nhx + lo - B] : hh[(nhx - d - 1) * nhx + hi - B]);
      }
      szsz[i * N + j] = e;
    }
  }
}

uint32_t flip_pair_blocks(const DevLayout& L) { return L.n_seg < 2048u ? L.n_seg : 2048u; }

template <class V>
hipError_t launch_flip_pairs(const DevLayout& L, const V* v, const uint32_t* masks, int n_pairs, double* part,
                             double* out, hipStream_t st) {
  if (n_pairs <= 0) return hipSuccess;
  const uint32_t nbx = flip_pair_blocks(L);
  const uint32_t nby = (uint32_t)((n_pairs + kPairChunk - 1) / kPairChunk);
  hipLaunchKernelGGL((flip_pairs_kernel<V>), dim3(nbx, nby), dim3(kBlock), 0, st, L, v, masks, n_pairs, part);
  hipLaunchKernelGGL(flip_combine_kernel, dim3(n_pairs), dim3(kBlock), 0, st, part, nbx, out);
  return hipGetLastError();
}

uint32_t flip_gram_blocks(const DevLayout& L) { return std::min(1u << L.NH, kGramBlocks); }

template <class V>
hipError_t launch_flip_gram(const DevLayout& L, const V* v, double* part, double* out, hipStream_t st) {
  const uint32_t nb = flip_gram_blocks(L), last = (uint32_t)choose(L.NH, L.k - 1 - L.B);
  const size_t lds = std::max<size_t>(page_bytes(L.B), (kBlock / 64) * 256 * sizeof(double));
  if (L.NH <= 16)
    hipLaunchKernelGGL((flip_gram_kernel<V, 1>), dim3(nb), dim3(kBlock), lds, st, L, last, v, part);
  else
    hipLaunchKernelGGL((flip_gram_kernel<V, 2>), dim3(nb), dim3(kBlock), lds, st, L, last, v, part);
  launch_sum_parts(part, nb, (uint32_t)flip_gram_values(L), out, st);
  return hipGetLastError();
}

double read_flip(const DevLayout& L, const double* sums, int site_i, int site_j) {
  const int p = L.N - 1 - site_i, q = L.N - 1 - site_j;
  auto at = [&](int bit) { return bit < L.B ? bit : 16 + bit - L.B; };
  const int a = std::min(at(p), at(q)), b = std::max(at(p), at(q));
  return sums[(gram_tiles(b / 16 - 1) + a / 16) * 256 + a % 16 * 16 + b % 16];
}

template hipError_t launch_spin_moments<float>(const DevLayout&, const MomentPlan&, const float*, double*, double*,
                                               hipStream_t);
template hipError_t launch_flip_pairs<float>(const DevLayout&, const float*, const uint32_t*, int, double*, double*,
                                             hipStream_t);
template hipError_t launch_flip_gram<float>(const DevLayout&, const float*, double*, double*, hipStream_t);
template hipError_t launch_spin_moments<double>(const DevLayout&, const MomentPlan&, const double*, double*, double*,
                                               hipStream_t);
template hipError_t launch_flip_pairs<double>(const DevLayout&, const double*, const uint32_t*, int, double*, double*,
                                             hipStream_t);
template hipError_t launch_flip_gram<double>(const DevLayout&, const double*, double*, double*, hipStream_t);

}  // namespace alps_ed
