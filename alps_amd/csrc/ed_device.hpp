// ed_device.hpp -- device-side building blocks shared by the single-solve
// and the batched kernels: wave/block reductions, uniform (scalar) table
// reads and the H.v of one row segment.
#pragma once

#include <hip/hip_runtime.h>

#include "ed_kernels.hpp"

namespace alps_ed {
namespace dev {

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Block sum, returned to every thread.
__device__ __forceinline__ double block_sum_all(double v) {
  __shared__ double red_smem[kBlock / 64];
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6;
  __syncthreads();  // red_smem may still be read by a previous call
  if ((threadIdx.x & 63) == 0) red_smem[wave] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) s += red_smem[w];
  return s;
}

// Two block sums through one pair of barriers (each equal to its
// block_sum_all).
__device__ __forceinline__ void block_sum_all2(double& a, double& b) {
  __shared__ double red2_smem[2][kBlock / 64];
  a = wave_sum(a);
  b = wave_sum(b);
  const int wave = threadIdx.x >> 6;
  __syncthreads();  // red2_smem may still be read by a previous call
  if ((threadIdx.x & 63) == 0) {
    red2_smem[0][wave] = a;
    red2_smem[1][wave] = b;
  }
  __syncthreads();
  a = 0.0;
  b = 0.0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) {
    a += red2_smem[0][w];
    b += red2_smem[1][w];
  }
}

// A thread's share of a sum of partials: entries tid, tid + kBlock, ... in
// index order.  The loads of eight terms are issued together before their
// additions (a loop with one load per addition waits for each in turn).
__device__ __forceinline__ double thread_partials(const Partials& P) {
  double v = 0.0;
  for (uint32_t i = threadIdx.x; i < P.n; i += 8u * kBlock) {
    double t[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) t[k] = i + k * kBlock < P.n ? P.p[i + k * kBlock] : 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (i + k * kBlock < P.n) v += t[k];
  }
  return v;
}

__device__ __forceinline__ double sum_partials(const Partials& P) { return block_sum_all(thread_partials(P)); }

// LDS by address.  The kernels that use LDS pages hold all their LDS in the
// dynamic allocation, which then starts at address 0, and xor page addresses:
// none of them may have a __shared__ variable, its own or of a function that
// it calls (tests/test_kernel_resources.py reads their static LDS from the
// built library and names every kernel that these functions are used in).
template <class T>
__device__ __forceinline__ T lds_ld(uint32_t addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) T*>(addr);
}
template <class T>
__device__ __forceinline__ void lds_st(uint32_t addr, T v) {
  *reinterpret_cast<__attribute__((address_space(3))) T*>(addr) = v;
}

// The sum of v over a block of NT threads stored to *out by thread 0, through
// the first NT / 8 bytes of LDS, which no thread may still use.
template <int NT>
__device__ __forceinline__ void store_block_sum_lds(double* out, double v) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) lds_st<double>(threadIdx.x >> 3, v);
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
#pragma unroll
    for (uint32_t w = 0; w < NT / 64; ++w) s += lds_ld<double>(8u * w);
    *out = s;
  }
}

__device__ __forceinline__ void store_partial(double* out, double v) {
  const double s = block_sum_all(v);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}


// Basis state of row i (binary search over the segment starts) and the row
// of state s (D when s is not in the sector): the split ranking
// rank = hi_base[s >> B] + lo_rank[s & (2^B - 1)].
__device__ __forceinline__ uint32_t unrank(const DevLayout& L, uint32_t i) {
  uint32_t lo = 0, hi = L.n_seg - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (L.seg_start[mid] <= i) lo = mid;
    else hi = mid - 1;
  }
  const uint32_t h = L.seg_hi[lo];
  const uint32_t r = i - L.seg_start[lo];
  const int kl = L.k - __builtin_popcount(h);
  return (h << L.B) | L.lo_state[L.lo_class_off[kl] + r];
}

__device__ __forceinline__ uint32_t rank_of(const DevLayout& L, uint32_t s) {
  if (__builtin_popcount(s) != L.k) return L.D;
  if (L.N < 32 && (s >> L.N) != 0u) return L.D;
  const uint32_t h = L.NH > 0 ? (s >> L.B) : 0u;
  const uint32_t lo = L.B >= 32 ? s : (s & ((1u << L.B) - 1u));
  const uint32_t hb = L.hi_base[h];
  if (hb == 0xffffffffu) return L.D;
  return hb + L.lo_rank[lo];
}

// Uniform reads of the layout tables.  The tables are never written while a
// kernel runs, so they are read through the constant address space, which
// lets the compiler use scalar loads for wave-uniform addresses.
template <class T>
__device__ __forceinline__ T ldc(const T* p) {
  return *(const __attribute__((address_space(4))) T*)(p);
}

// Start-vector element i of stream `seed`: uniform on [lo, hi) from the
// splitmix64 output of the counter seed + (i+1) * golden gamma.
__device__ __forceinline__ uint64_t splitmix64_mix(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  return z ^ (z >> 31);
}

__device__ __forceinline__ double start_value(uint64_t seed, uint64_t i, double lo, double hi) {
  const uint64_t z = splitmix64_mix(seed + (i + 1) * 0x9e3779b97f4a7c15ULL);
  const double u = (double)(z >> 11) * (1.0 / 9007199254740992.0);
  return lo + (hi - lo) * u;
}

// Whole struct read through the constant address space (scalar loads when
// the address is wave-uniform); T is plain data of 8-byte multiple size.
template <class T>
__device__ __forceinline__ T ldc_struct(const T* p) {
  static_assert(sizeof(T) % 8 == 0, "ldc_struct needs an 8-byte multiple");
  T out;
  uint64_t* o = reinterpret_cast<uint64_t*>(&out);
  const __attribute__((address_space(4))) uint64_t* s = (const __attribute__((address_space(4))) uint64_t*)(p);
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T) / 8); ++i) o[i] = s[i];
  return out;
}

// A load of T at byte offset `off` (per lane, 32 bits) from a wave-uniform
// global base: the load adds the offset to the base, held in scalar
// registers, in the address unit (global_load with a scalar base), instead
// of a 64-bit vector add per lane and load.  The empty asm keeps the
// compiler from folding the offset into a 64-bit per-lane address.
template <class T>
__device__ __forceinline__ T ld_lane(const void* base, uint32_t off) {
  typedef __attribute__((address_space(1))) const char gchar;
  typedef __attribute__((address_space(1))) const T gT;
  asm volatile("" : "+v"(off));
  return *reinterpret_cast<gT*>(reinterpret_cast<gchar*>(reinterpret_cast<uintptr_t>(base)) + off);
}

// The same for an offset that serves many loads: lane_off() makes it opaque
// once, and ld_at / st_at use it as it is (no register copy per access).
__device__ __forceinline__ uint32_t lane_off(uint32_t off) {
  asm volatile("" : "+v"(off));
  return off;
}

template <class T>
__device__ __forceinline__ T ld_at(const void* base, uint32_t off) {
  typedef __attribute__((address_space(1))) const char gchar;
  typedef __attribute__((address_space(1))) const T gT;
  return *reinterpret_cast<gT*>(reinterpret_cast<gchar*>(reinterpret_cast<uintptr_t>(base)) + off);
}

template <class T>
__device__ __forceinline__ void st_at(void* base, uint32_t off, T v) {
  typedef __attribute__((address_space(1))) char gchar;
  typedef __attribute__((address_space(1))) T gT;
  *reinterpret_cast<gT*>(reinterpret_cast<gchar*>(reinterpret_cast<uintptr_t>(base)) + off) = v;
}

// Workgroup barrier for data exchanged through LDS: waits for this wave's LDS
// accesses only.  __syncthreads() also waits for every global load in flight,
// which here are the reads issued early to overlap the LDS work.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Two sums over a workgroup of NT threads, to every thread, through LDS
// barriers only: the vector elements read before stay in flight.  Once per
// kernel.
template <int NT>
__device__ __forceinline__ void update_sums(double& a, double& b) {
  __shared__ double red[2][NT / 64];
  a = wave_sum(a);
  b = wave_sum(b);
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = a;
    red[1][threadIdx.x >> 6] = b;
  }
  lds_barrier();
  a = 0.0;
  b = 0.0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {
    a += red[0][w];
    b += red[1][w];
  }
}

// The sum of v over a workgroup of NT threads, in wave order, to
// out[blockIdx.x].  Once per kernel.
template <int NT>
__device__ __forceinline__ void store_update_partial(double* out, double v) {
  __shared__ double red_out[NT / 64];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red_out[threadIdx.x >> 6] = v;
  lds_barrier();
  if (threadIdx.x == 0) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < NT / 64; ++q) s += red_out[q];
    out[blockIdx.x] = s;
  }
}

// The workgroup's (NT threads) part of clearing the page of B low bits.
template <int NT>
__device__ __forceinline__ void clear_page(int B) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 zero = {0u, 0u, 0u, 0u};
  if (B == 12) {
#pragma unroll
    for (uint32_t i = 0; i < 4u << 12; i += 16u * NT) lds_st<u32x4>(16u * threadIdx.x + i, zero);
  } else {
    for (uint32_t i = 16u * threadIdx.x; i < page_bytes(B); i += 16u * NT) lds_st<u32x4>(i, zero);
  }
}

// Keeps the instructions before it (the reads of a chunk) ahead of those
// after it: the compiler otherwise pairs every LDS read with its use, one
// wait each, to save registers.
__device__ __forceinline__ void issue_barrier() { __builtin_amdgcn_sched_barrier(0); }

// v where the mask is all ones, 0 where it is 0.
__device__ __forceinline__ float masked(float v, uint32_t m) { return __uint_as_float(__float_as_uint(v) & m); }
__device__ __forceinline__ double masked(double v, uint32_t m) {
  return __hiloint2double((int)((uint32_t)__double2hiint(v) & m), (int)((uint32_t)__double2loint(v) & m));
}

// Every multiply-add of a row is an explicit fma, so that rows and dot
// partials do not depend on what the compiler contracts.
//
// The rows of hv_segment for NQ row slots per thread (rows tid,
// tid + NT, ... of NT threads), NQ fixed at compile time so that the loads of all
// slots are issued together.  Every slot of the wave but the last is full
// (hv_segment gives a wave the slots up to its last row); in the last, rows
// past the segment repeat row 0 and are not stored in y.  A wave without rows (NQ =
// 0) takes part in the staging and the barriers.  The low-low and high-high
// bonds are processed in chunks of CLL and CHH.  Returns the thread's share
// of x.Hx when DOT.
//
// Low-low flips read the segment's LDS page: one FP64 element per low word of
// the segment's parity at its position (page_pos), zero for words outside the
// segment's class.  A flip moves the position by a constant xor, without a
// table; parallel bits lead to a word with two bits more or fewer, which
// reads zero.
//
// Cross bonds with STAGE: the bonds of one high bit read the same neighbour
// segment, which is staged once for all of them in the page, after the
// low-low pass (its words have the other parity; parallel bits lead to the
// class on the other side, zero).  FP32 vectors use the page as two halves of
// FP32 elements in turn, one barrier a stage; FP64 ones have one page, two
// barriers.  The high bits set in h come first (their segments' words have
// one low bit more), then the others; the page is cleared before each kind,
// within a kind every place is overwritten.  The rows of the next AHEAD
// stages are in flight.  Their share of the diagonal is linear in the bits of
// the low word (xw): two sums over six bits each, tabled in the page at the
// end, two reads and additions per row instead of a test, a select and an fma
// per bond.
// Without STAGE each bond gathers: its rank comes from a per-class table.
//
// Addressing: a slot's element of a segment of x (or y) is read at the
// lane offset of slot 0 from a base moved by q * NT elements, or, for
// the last slot, at its own clamped offset; its flip-table records at slot
// 0's lane offset from a base moved by q * NT records.  Rows of the last
// slot past the segment stay inside the class table (padded to groups of
// 64 rows), whose padding entries are in-range offsets.
template <class V, bool DOT, bool STAGE, int NT, int NQ, int CLL, int CHH>
__device__ __forceinline__ double hv_rows(const DevLayout& L, const SegRec& S, const V* __restrict__ x,
                                          V* __restrict__ y) {
  constexpr uint32_t VS = (uint32_t)sizeof(V);
  constexpr int QL = NQ - 1;           // the last slot
  constexpr int NA = NQ > 0 ? NQ : 1;  // array extent
  constexpr int MQ = kMaxSegRows / NT;  // slots of any segment
  const uint32_t tid = threadIdx.x;
  const uint32_t len = S.len, base = S.base, e0 = S.e0, e1 = S.e1;
  const uint32_t rl = tid + QL * NT;
  const bool okl = NQ > 0 && rl < len;
  const uint32_t vo0 = lane_off(VS * tid);               // slot 0 (and every full slot)
  const uint32_t vol = lane_off(okl ? VS * rl : 0u);     // the last slot, clamped
  // element of slot q of the segment starting at p
  auto seg_ld = [&](const V* p, int q) -> V {
    return q < QL ? ld_at<V>(p + q * NT, vo0) : ld_at<V>(p, vol);
  };
  // entry of slot q of a table of 16-bit words in class order
  auto word_ld = [&](const uint16_t* t, int q) -> uint32_t {
    return q < QL ? ld_at<uint16_t>(t + S.cls0 + q * NT, vo0 / (VS / 2u)) : ld_at<uint16_t>(t + S.cls0, vol / (VS / 2u));
  };
  V xo[NA];
  uint32_t pg[NA];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    xo[q] = seg_ld(x + base, q);
    pg[q] = word_ld(L.lo_page, q);
  }
  issue_barrier();  // the page waits for these only, not for what follows
  // high-high flips: a bond flips every row of the segment or none (its two
  // bits lie in h), with a contiguous target run.  The bonds that flip h are
  // listed per high word in bond order (hh_off / hh_ent), padded with
  // weight-0 reads of this segment; slots of a chunk past the list do the
  // same.  Bonds that do not flip would add exact zeros, so the sums are
  // those over all bonds.  The first chunk is read here and used after the
  // low-low pass (lds_barrier does not wait for it).
  V hv[NA][CHH];
  double ht[CHH];
  auto hh_load = [&](uint32_t e) {
    uint32_t xt[CHH];  // neighbour segment starts as element offsets (a select
                       // between pointers would make the loads generic-address ones)
#pragma unroll
    for (int c = 0; c < CHH; ++c) {
      if (c < kHHList || e + c < e1) {
        const HHEntry en = ldc_struct(L.hh_ent + e + c);
        xt[c] = en.nb;
        ht[c] = en.t;
      } else {
        xt[c] = base;
        ht[c] = 0.0;
      }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int c = 0; c < CHH; ++c) hv[q][c] = seg_ld(x + xt[c], q);
  };
  if (NQ > 0 && e0 < e1) hh_load(e0);
  issue_barrier();
  clear_page<NT>(L.B);
  lds_barrier();
#pragma unroll
  for (int q = 0; q < NQ; ++q)
    lds_st<double>(pg[q], (double)xo[q]);
  lds_barrier();
  double d[NA], off[NA];
#pragma unroll
  for (int q = 0; q < NQ; ++q) off[q] = 0.0;
  if (NQ > 0) {
    int b = 0;
    for (; b + CLL <= L.n_ll; b += CLL) {
      PageBond k[CLL];
      double v[CLL][NA];
#pragma unroll
      for (int c = 0; c < CLL; ++c) k[c] = ldc_struct(L.ll_c + b + c);
#pragma unroll
      for (int c = 0; c < CLL; ++c)
#pragma unroll
        for (int q = 0; q < NQ; ++q) v[c][q] = lds_ld<double>(pg[q] ^ k[c].m);
      issue_barrier();
#pragma unroll
      for (int c = 0; c < CLL; ++c)
#pragma unroll
        for (int q = 0; q < NQ; ++q) off[q] = fma(k[c].t, v[c][q], off[q]);
    }
    for (; b < L.n_ll; ++b) {
      const PageBond k = ldc_struct(L.ll_c + b);
#pragma unroll
      for (int q = 0; q < NQ; ++q) off[q] = fma(k.t, lds_ld<double>(pg[q] ^ k.m), off[q]);
    }
  }
  if (NQ > 0)
    for (uint32_t e = e0; e < e1; e += CHH) {
#pragma unroll
      for (int c = 0; c < CHH; ++c)
#pragma unroll
        for (int q = 0; q < NQ; ++q) off[q] = fma(ht[c], (double)hv[q][c], off[q]);
      if (e + CHH < e1) hh_load(e + CHH);
    }
  const double* dlp = L.diag_lo_cls + S.cls0;
  auto diag_ld = [&](int q) -> double {
    return q < QL ? ld_at<double>(dlp + q * NT, vo0 * (8u / VS)) : ld_at<double>(dlp, vol * (8u / VS));
  };
  if constexpr (STAGE) {
    constexpr int AHEAD = NT >= 256 ? 4 : 2;
    constexpr uint32_t kHalf = (4u << 12) / 2u;  // bytes of half a page (staged layouts have 12 low bits)
    constexpr uint32_t PS = 8u / VS;             // FP32 elements are at half the page offset
    const uint32_t w0 = __builtin_amdgcn_readfirstlane(tid & ~63u);
    // entry of slot q of n rows at p (the last row again past the end); a
    // wave's last slot alone takes the clamped offset
    auto ld_rows = [&](auto* p, int q, uint32_t n) {
      using T = std::decay_t<decltype(*p)>;
      constexpr uint32_t TS = (uint32_t)sizeof(T);
      if (w0 + q * NT + 64u <= n) return ld_at<T>(p + q * NT, TS >= VS ? vo0 * (TS / VS) : vo0 / (VS / TS));
      return ld_lane<T>(p, TS * min(tid + q * NT, n - 1u));
    };
    V sv[AHEAD][MQ];
    uint32_t sp[MQ];
    const XStage* xs = L.xs + (size_t)S.h_or_index * L.n_xs;
    auto stage_of = [&](int i) { return i < L.n_xs ? ldc_struct(xs + i) : XStage{0u, 0u}; };
    auto rows_of = [&](uint32_t info) { return (int)info < 0 ? S.len_up : S.len_dn; };
    auto stage_load = [&](V(&v)[MQ], XStage st) {
      const uint32_t n = rows_of(st.info);
      if (st.info == 0u) return;
#pragma unroll
      for (int q = 0; q < MQ; ++q)
        if (w0 + q * NT < n) v[q] = ld_rows(x + st.nb, q, n);
    };
    XStage st[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      st[i] = stage_of(i);
      stage_load(sv[i], st[i]);
    }
    if (VS == 4)
#pragma unroll
      for (int q = 0; q < NQ; ++q) pg[q] /= PS;
    uint32_t kind = 2u;  // the staged kind (info's sign); 2: none yet
    for (int i0 = 0; st[0].info != 0u; i0 += AHEAD) {
#pragma unroll
      for (int s = 0; s < AHEAD; ++s) {
        const XStage cur = st[s];
        if (cur.info == 0u) continue;  // past the last stage; the loop ends
        const uint32_t half = VS == 4 ? (s & 1) * kHalf : 0u;
        const uint32_t n = rows_of(cur.info);
        if ((cur.info >> 31) != kind) {
          kind = cur.info >> 31;
          const uint32_t cls = kind ? S.cls_up : S.cls_dn;
#pragma unroll
          for (int q = 0; q < MQ; ++q)
            if (w0 + q * NT < n) sp[q] = (uint32_t)ld_rows(L.lo_page + cls, q, n) / PS;
          lds_barrier();  // every wave is done with the page
          clear_page<NT>(12);
          lds_barrier();
        } else if (VS == 8) {
          lds_barrier();
        }
#pragma unroll
        for (int q = 0; q < MQ; ++q)
          if (w0 + q * NT < n) lds_st<V>(half + sp[q], sv[s][q]);
        lds_barrier();
        st[s] = stage_of(i0 + s + AHEAD);
        stage_load(sv[s], st[s]);
        if (NQ > 0) {
          const uint32_t b1 = (cur.info & 0xffffu) + ((cur.info >> 16) & 0x7fffu);
          for (uint32_t b = cur.info & 0xffffu; b < b1; ++b) {
            const PageBond k = ldc_struct(L.xb_p + b);
            const uint32_t m = k.m / PS;
            V v[NA];
#pragma unroll
            for (int q = 0; q < NQ; ++q) v[q] = lds_ld<V>(half + (pg[q] ^ m));
            issue_barrier();
#pragma unroll
            for (int q = 0; q < NQ; ++q) off[q] = fma(k.t, (double)v[q], off[q]);
          }
        }
      }
    }
    // the cross bonds' share of the diagonal, six low bits each
    lds_barrier();
    if (tid < 128u) {
      const uint32_t hf = __builtin_amdgcn_readfirstlane(tid >> 6);
      const double* w = L.xw + (size_t)S.h_or_index * kXwStride;
      double s = hf ? S.dh_page : ldc(w + L.B);
#pragma unroll
      for (uint32_t p = 0; p < 6u; ++p) s = fma((tid >> p & 1u) ? 1.0 : 0.0, ldc(w + 6u * hf + p), s);
      lds_st<double>(8u * tid, s);
    }
    uint32_t lo[NA];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      lo[q] = word_ld(L.lo_word, q);
      d[q] = diag_ld(q);
    }
    lds_barrier();
#pragma unroll
    for (int q = 0; q < NQ; ++q) d[q] += lds_ld<double>(8u * (lo[q] & 63u)) + lds_ld<double>(512u + 8u * (lo[q] >> 6));
  } else {
    // gathered cross bonds: flip when the high and low bits differ (bit 15 of
    // the table entry is the row's low bit).  Where the neighbouring high word
    // has no segment no row can flip (its low word would need a set bit more
    // or fewer than it has), and xb_nb points to this segment.  The diagonal
    // already holds every cross bond's parallel value (diag_hi); each
    // antiparallel bond adds its anti - par difference.
    static_assert(kXChunk == 2, "one 4-byte load per row and chunk");
    const uint16_t* xnp = L.xn16 + S.xnp;
    static_assert(NT % 64 == 0, "slots start at groups of 64 rows");
    const uint32_t lo_x = lane_off(2u * ((tid >> 6) * 64u * (uint32_t)L.n_xb_p + (tid & 63u) * kXChunk));
    const uint32_t x_slot = (uint32_t)NT * (uint32_t)L.n_xb_p;  // u16 entries per slot
#pragma unroll
    for (int q = 0; q < NQ; ++q) d[q] = S.dh_page;
    const uint32_t h = S.h_or_index;  // not staged: the high word
    const uint32_t* xnb = L.xb_nb + h * (uint32_t)L.n_xb_p;
    for (int b0 = 0; NQ > 0 && b0 < L.n_xb; b0 += kXChunk) {
      // the two bonds' entries, bits 15 and 31 set where the row flips
      uint32_t e[NA];
#pragma unroll
      for (int q = 0; q < NQ; ++q) e[q] = ld_at<uint32_t>(xnp + q * x_slot + (uint32_t)b0 * 64u, lo_x);
      const XBondConst k0 = ldc_struct(L.xb_c + b0), k1 = ldc_struct(L.xb_c + b0 + 1);
      const uint32_t hx = ((h & k0.hbit) != 0u ? 0x8000u : 0u) | ((h & k1.hbit) != 0u ? 0x80000000u : 0u);
      const V *x0 = x + ldc(xnb + b0), *x1 = x + ldc(xnb + b0 + 1);
      // all ones where the row flips: it masks the gathered offset (to the
      // segment's first row), the value and the 1.0 of the diagonal
      auto mask = [&](int q, int c) { return c == 0 ? (uint32_t)((int)(e[q] << 16) >> 31) : (uint32_t)((int)e[q] >> 31); };
      V v[NA][kXChunk];
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        e[q] ^= hx;
        v[q][0] = ld_lane<V>(x0, (e[q] & 0x7fffu & mask(q, 0)) * (VS / 4u));
        v[q][1] = ld_lane<V>(x1, (e[q] >> 16 & 0x7fffu & mask(q, 1)) * (VS / 4u));
      }
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int c = 0; c < kXChunk; ++c) {
          const uint32_t m = mask(q, c);
          d[q] = fma(__hiloint2double((int)(0x3ff00000u & m), 0), c == 0 ? k0.de : k1.de, d[q]);
          off[q] = fma(c == 0 ? k0.t : k1.t, (double)masked(v[q][c], m), off[q]);
        }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) d[q] += diag_ld(q);
  }
  double dotp = 0.0;
  V* yb = y + base;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if (q < QL || okl) {
      const double xi = (double)xo[q];
      const double yv = fma(d[q], xi, off[q]);
      if (q < QL) st_at<V>(yb + q * NT, vo0, (V)yv);
      else st_at<V>(yb, vol, (V)yv);
      if (DOT) dotp = fma(xi, yv, dotp);  // FP64 value before the storage rounding
    }
  }
  return dotp;
}

// H.v over the row segment of record S (one workgroup of NT threads; dynamic
// LDS of at least page_bytes(L.B)):
//   y[r] = sum_c H[r][c] x[c] for the segment's rows r;
// with DOT, *dot_slot receives the segment's sum of x_r (H x)_r (FP64, before
// y is rounded to the storage type).  STAGE: L.n_xs > 0.
//
// The segment's slice of x is staged in an LDS page in FP64.  Each thread owns
// up to kMaxSegRows / NT rows (r = tid + q*NT); the number of row slots that
// hold rows is uniform over each wave and selects a fixed-size instance of the
// bond loops, so a wave does no work for slots past the segment (the waves of a
// short segment's last slot skip it, those without rows only clear and stage
// their part of the page).  CLL, CHH: chunk sizes of the flip loops (the
// schedule, ed_kernels.hpp).
//
// What bounds it: at 24 sites (2.7 M rows, FP32) 33 MB of neighbour reads that
// miss the XCDs' L2 and 11 MB of y take 5.9 us at the 7.4 TB/s such misses
// reach, the rest is the chain of dependent rounds of a segment (record -> x ->
// page -> list entries -> neighbour rows) with 2 generations of workgroups
// (waves wait for 47 % of their cycles, the address unit is busy for 57 % of
// the 14.7 us); at 25 sites (4.5 M rows, FP64) 104 + 36 MB take 18.9 of 34.5
// us. On the 30-site J1-J2 lattice (155 M rows) 15.3 GB of misses and 0.7 GB of
// writes take 2.2 of 3.3 ms; the address unit is busy for 62 % of it (98 % with
// tables and gathers), LDS for 52 %, half of that bank conflicts, the vector
// ALUs for 46 %.  Measured against flip tables in memory, a page indexed by
// rank and __syncthreads, the earlier segment order on both sides: 15.7 -> 14.3
// us at 24 sites, 4.22 -> 3.32 ms on J1-J2, FP64 38.9 -> 36.5 us (25 sites),
// 5.0 -> 4.4 us (20 sites).
// Of that, the table loads that the xor positions save are the most (a
// quarter of the J1-J2 launch's vector loads), then the staged cross bonds
// (3.93 -> 3.37 ms) and barriers that do not drain the loads in flight.
template <class V, bool DOT, bool STAGE, int NT, int NQ, int CLL, int CHH>
__device__ __forceinline__ double hv_slots(uint32_t nq, const DevLayout& L, const SegRec& S, const V* __restrict__ x,
                                           V* __restrict__ y) {
  if constexpr (NQ > 0) {
    if (nq < (uint32_t)NQ) return hv_slots<V, DOT, STAGE, NT, NQ - 1, CLL, CHH>(nq, L, S, x, y);
  }
  return hv_rows<V, DOT, STAGE, NT, NQ, CLL, CHH>(L, S, x, y);
}

template <class V, bool DOT, bool STAGE, int NT = kBlock, int CLL = 2, int CHH = sizeof(V) == 4 ? 4 : 2>
__device__ __forceinline__ void hv_segment_at(const DevLayout& L, const SegRec& S, const V* __restrict__ x,
                                              V* __restrict__ y, double* __restrict__ dot_slot) {
  // row slots of this wave: slot q holds rows wave*64 + q*NT + lane
  const uint32_t w0 = threadIdx.x & ~63u;
  const uint32_t nq = __builtin_amdgcn_readfirstlane(S.len > w0 ? (S.len - w0 + NT - 1) / NT : 0u);
  // Every wave passes the same workgroup barriers, in the instance of its
  // slots (the branch is uniform over each wave).
  const double dotp = hv_slots<V, DOT, STAGE, NT, kMaxSegRows / NT, CLL, CHH>(nq, L, S, x, y);
  if (DOT) {
    lds_barrier();  // every wave is done with the page
    store_block_sum_lds<NT>(dot_slot, dotp);
  }
}

// H.v over a segment with the low-low targets from tables (nbp16, one LDS
// byte offset per row and bond, the zero slot where the bits are parallel) and
// the slice of x in LDS by rank: nothing to clear and one barrier, at one more
// load per four low-low bonds.  It is the faster one where segments are short
// on average (ranked_rows, ed_layout.hpp), where the fixed part of a segment
// in hv_rows outweighs its rows.  Bound by the chain of dependent loads of a
// segment, so by the waves in flight and by scalar loads: a row's own element
// is read from LDS again at the end rather than kept (FP64: 64 registers, 8
// waves per SIMD instead of 7), the coefficients are contiguous and only
// what it needs of the record is read: 24 sites 8 up 7.84 -> 7.52 us (FP32)
// and 10.68 -> 10.46 (FP64), 22 sites 7 up 4.23 -> 4.14 and 4.68 -> 4.55, 23
// sites 7 up 4.69 -> 4.54 and 5.44 -> 5.30, 27-site J1-J2 9 up 132.5 -> 130.6
// and 181.3 -> 180.2.
template <class V, bool DOT, int NQ, int CLL, int CHH, int CX>
__device__ __forceinline__ double hv_ranked_rows(const DevLayout& L, const SegHead& S, const V* __restrict__ x,
                                                 V* __restrict__ y) {
  const uint32_t h = S.h_or_index, len = S.len, base = S.base, e0 = S.e0, e1 = S.e1;
  const double dh = S.dh;
  const uint16_t* nbp = L.nbp16 + S.nbp;
  const uint16_t* xnp = L.xn16 + S.xnp;
  const double* dlp = L.diag_lo_cls + S.cls0;
  constexpr uint32_t VS = (uint32_t)sizeof(V);
  constexpr int QL = NQ - 1;  // the last slot
  const uint32_t tid = threadIdx.x;
  const V* xb = x + base;
  static_assert(CLL % kLLChunk == 0 && CX % kXChunk == 0, "schedule chunks are multiples of the table chunks");
  typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  const uint32_t rl = tid + QL * kBlock;
  const bool okl = rl < len;
  const uint32_t vo0 = lane_off(VS * tid);               // slot 0 (and every full slot)
  const uint32_t vol = lane_off(okl ? VS * rl : 0u);     // the last slot, clamped
  // flip-table records (flip_index, ed_layout.hpp): bond chunk k of row r
  // starts at rec(r) + k * 64 * chunk
  const uint32_t lo_ll = lane_off(2u * ((tid >> 6) * 64u * (uint32_t)L.n_ll_p + (tid & 63u) * kLLChunk));
  const uint32_t lo_x = lane_off(2u * ((tid >> 6) * 64u * (uint32_t)L.n_xb_p + (tid & 63u) * kXChunk));
  const uint32_t ll_slot = (uint32_t)kBlock * (uint32_t)L.n_ll_p;  // u16 entries per slot
  const uint32_t x_slot = (uint32_t)kBlock * (uint32_t)L.n_xb_p;
  // element of slot q of the segment starting at p
  auto seg_ld = [&](const V* p, int q) -> V {
    return q < QL ? ld_at<V>(p + q * kBlock, vo0) : ld_at<V>(p, vol);
  };
  V xo[NQ];
  double d[NQ], off[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    xo[q] = seg_ld(xb, q);
    d[q] = dh + (q < QL ? ld_at<double>(dlp + q * kBlock, vo0 * (8u / VS)) : ld_at<double>(dlp, vol * (8u / VS)));
    off[q] = 0.0;
  }
  // The cross-bond table entries of the first chunk are loaded now, so that
  // they arrive while the other bonds are processed.
  const int n_xb = (L.n_xb + CX - 1) / CX * CX;
  constexpr int KX = CX / kXChunk;
  u16x2 xr[NQ][KX];
  if (n_xb > 0) {
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int k = 0; k < KX; ++k) xr[q][k] = ld_at<u16x2>(xnp + q * x_slot + k * kXChunk * 64u, lo_x);
  }
  // low-low flips: target rows from the class table, values from LDS.  The
  // table entries of chunk b + CLL are loaded while chunk b is processed,
  // into the other of two register sets (ta, tb).
  const int n_ll = (L.n_ll + CLL - 1) / CLL * CLL;
  constexpr int KL = CLL / kLLChunk;
  u16x4 ta[NQ][KL], tb[NQ][KL];
  auto ll_load = [&](u16x4(&t)[NQ][KL], int b) {
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int k = 0; k < KL; ++k)
        t[q][k] = ld_at<u16x4>(nbp + q * ll_slot + (uint32_t)(b + k * kLLChunk) * 64u, lo_ll);
  };
  auto ll_apply = [&](const u16x4(&t)[NQ][KL], int b) {
    double tc[CLL];
#pragma unroll
    for (int c = 0; c < CLL; ++c) tc[c] = ldc(L.ll_t + b + c);
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int c = 0; c < CLL; ++c) {
        const uint32_t j = t[q][c / kLLChunk][c % kLLChunk];
        off[q] = fma(tc[c], lds_ld<double>(j), off[q]);
      }
  };
  if (n_ll > 0) ll_load(ta, 0);
  // The segment's slice of x into LDS: each thread stores its own rows (the
  // rows of the segment are exactly the rows of the threads' slots), with
  // the table loads above already in flight; then the barrier that every
  // wave of the workgroup passes once (hv_ranked_at).
#pragma unroll
  for (int q = 0; q < QL; ++q) lds_st<double>(8u * (tid + q * kBlock), (double)xo[q]);
  if (okl) lds_st<double>(8u * rl, (double)xo[QL]);
  if (tid == 0) lds_st<double>(8u * len, 0.0);
  lds_barrier();
  for (int b0 = 0; b0 < n_ll; b0 += 2 * CLL) {
    if (b0 + CLL < n_ll) ll_load(tb, b0 + CLL);
    ll_apply(ta, b0);
    if (b0 + CLL >= n_ll) break;
    if (b0 + 2 * CLL < n_ll) ll_load(ta, b0 + 2 * CLL);
    ll_apply(tb, b0 + CLL);
  }
  // high-high flips: a bond flips every row of the segment or none (its two
  // bits lie in h), with a contiguous target run.  The bonds that flip h are
  // listed per high word in bond order (hh_off / hh_ent), padded with
  // weight-0 reads of this segment; slots of a chunk past the list do the
  // same.  Bonds that do not flip would add exact zeros, so the sums are
  // those over all bonds.
  {
    for (uint32_t e = e0; e < e1; e += CHH) {
      // neighbour segment starts as element offsets (a select between
      // pointers would make the loads generic-address ones)
      uint32_t xt[CHH];
      double tt[CHH];
#pragma unroll
      for (int c = 0; c < CHH; ++c) {
        if (c < kHHList || e + c < e1) {
          const HHEntry en = ldc_struct(L.hh_ent + e + c);
          xt[c] = en.nb;
          tt[c] = en.t;
        } else {
          xt[c] = base;
          tt[c] = 0.0;
        }
      }
      V v[NQ][CHH];
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int c = 0; c < CHH; ++c) v[q][c] = seg_ld(x + xt[c], q);
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int c = 0; c < CHH; ++c) off[q] = fma(tt[c], (double)v[q][c], off[q]);
    }
  }
  // cross bonds: diagonal always, flip when the high and low bits differ
  // (bit 15 of the table entry is the row's low bit).  Where the
  // neighbouring high word has no segment no row can flip (its low word
  // would need a set bit more or fewer than it has), and xb_nb points to this
  // segment.  The diagonal already holds every cross bond's parallel value
  // (diag_hi); each antiparallel bond adds its anti - par difference.
  const uint32_t* xnb = L.xb_nb + h * (uint32_t)L.n_xb_p;
  for (int b0 = 0; b0 < n_xb; b0 += CX) {
    uint32_t xt[CX], hx[CX];
    double de[CX], tx[CX];
#pragma unroll
    for (int c = 0; c < CX; ++c) {
      const XBondConst k = ldc_struct(L.xb_c + b0 + c);
      hx[c] = (h & k.hbit) != 0u ? 0x8000u : 0u;
      xt[c] = ldc(xnb + b0 + c);
      de[c] = k.de;
      tx[c] = k.t;
    }
    uint32_t e[NQ][CX];
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int k = 0; k < KX; ++k)
#pragma unroll
        for (int c = 0; c < kXChunk; ++c) e[q][k * kXChunk + c] = xr[q][k][c];
    if (b0 + CX < n_xb) {
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int k = 0; k < KX; ++k)
          xr[q][k] = ld_at<u16x2>(xnp + q * x_slot + (uint32_t)(b0 + CX + k * kXChunk) * 64u, lo_x);
    }
    V v[NQ][CX];
    bool f[NQ][CX];
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int c = 0; c < CX; ++c) {
        f[q][c] = ((e[q][c] ^ hx[c]) & 0x8000u) != 0u;
        v[q][c] = ld_lane<V>(x + xt[c], f[q][c] ? (e[q][c] & 0x7fffu) * (VS / 4u) : 0u);
      }
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int c = 0; c < CX; ++c) {
        // the flag as 1.0 / 0.0 and the value selected in the storage type
        // (one 32-bit select each; the asm keeps the select before the
        // conversion, where selecting the FP64 value takes two)
        V w = f[q][c] ? v[q][c] : (V)0;
        asm volatile("" : "+v"(w));
        d[q] = fma(f[q][c] ? 1.0 : 0.0, de[c], d[q]);
        off[q] = fma(tx[c], (double)w, off[q]);
      }
  }
  double dotp = 0.0;
  V* yb = y + base;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if (q < QL || okl) {
      const double xi = lds_ld<double>(8u * (q < QL ? tid + q * kBlock : rl));
      const double yv = fma(d[q], xi, off[q]);
      if (q < QL) st_at<V>(yb + q * kBlock, vo0, (V)yv);
      else st_at<V>(yb, vol, (V)yv);
      if (DOT) dotp = fma(xi, yv, dotp);  // FP64 value before the storage rounding
    }
  }
  return dotp;
}

// The same workgroup and slots as hv_segment_at; dynamic LDS of max_seg + 1
// doubles.
template <class V, bool DOT, int CLL = 4, int CHH = 4, int CX = 2>
__device__ __forceinline__ void hv_ranked_at(const DevLayout& L, const SegHead& S, const V* __restrict__ x,
                                             V* __restrict__ y, double* __restrict__ dot_slot) {
  const uint32_t w0 = threadIdx.x & ~63u;
  const uint32_t nq = __builtin_amdgcn_readfirstlane(S.len > w0 ? (S.len - w0 + kBlock - 1) / kBlock : 0u);
  static_assert(kMaxSegRows == 4 * kBlock, "one to four row slots");
  double dotp = 0.0;
  if (nq == 0) lds_barrier();
  else if (nq == 1) dotp = hv_ranked_rows<V, DOT, 1, CLL, CHH, CX>(L, S, x, y);
  else if (nq == 2) dotp = hv_ranked_rows<V, DOT, 2, CLL, CHH, CX>(L, S, x, y);
  else if (nq == 3) dotp = hv_ranked_rows<V, DOT, 3, CLL, CHH, CX>(L, S, x, y);
  else dotp = hv_ranked_rows<V, DOT, 4, CLL, CHH, CX>(L, S, x, y);
  if (DOT) {
    lds_barrier();  // every wave is done with the slice
    store_block_sum_lds<kBlock>(dot_slot, dotp);
  }
}

// The record of segment seg of the processing order, looked up in the tables
// (staged: cross bonds staged; tables: low-low target tables).
__device__ __forceinline__ SegRec seg_record(const DevLayout& L, uint32_t seg, bool staged, bool tables) {
  const uint32_t h = ldc(L.proc_hi + seg);
  const int kl = L.k - __builtin_popcount(h);
  SegRec S;
  S.h_or_index = staged ? ldc(L.proc_index + seg) : h;
  S.base = ldc(L.hi_base + h);
  S.cls0 = ldc(L.lo_class_off + kl);
  S.cls_up = ldc(L.lo_class_off + kl + 1);
  S.len = S.cls_up - S.cls0;
  S.len_up = kl < L.B ? ldc(L.lo_class_off + kl + 2) - S.cls_up : 0u;
  S.cls_dn = kl > 0 ? ldc(L.lo_class_off + kl - 1) : 0u;
  S.len_dn = kl > 0 ? S.cls0 - S.cls_dn : 0u;
  S.e0 = ldc(L.hh_off + h);
  S.e1 = ldc(L.hh_off + h + 1);
  S.xnp = ldc(L.xn_off + kl);
  S.nbp = tables ? ldc(L.nbp_off + kl) : 0u;
  S.dh = ldc(L.diag_hi + h);
  S.dh_page = S.dh;
  return S;
}

// Row i of H.v in a momentum sector (vectors of 2 * Bl.dk reals, the real
// and imaginary parts of element i at 2i and 2i + 1); rows i >= Bl.dk do
// nothing.
// The diagonal is the site terms plus each bond's parallel / antiparallel
// value; each antiparallel bond flips to s' = s_i ^ mask, whose rank in the
// fixed-Sz sector (split ranking) gives its representative j and
// translation t, and contributes t_b * phase_t * norm_j / norm_i times x_j
// (hamiltonian_matrix.hpp:308-345 with bloch_basis_states::index_and_phase,
// blochbasisstates.h:47-55).  Returns Re(conj(x_i) (Hx)_i) when DOT.
template <class V, bool DOT>
__device__ __forceinline__ double bloch_row(const DevLayout& L, const DevBloch& Bl, const V* __restrict__ x,
                                            V* __restrict__ y, uint32_t i) {
  const uint32_t dk = Bl.dk;
  if (i >= dk) return 0.0;
  const uint32_t lomask = (1u << L.B) - 1u;
  const uint32_t s = Bl.rep_state[i];
  double d = 0.0;
  for (int site = 0; site < L.N; ++site) d += ((s >> (L.N - 1 - site)) & 1u) ? L.site_up[site] : L.site_dn[site];
  const double xr = (double)x[2 * i], xi = (double)x[2 * i + 1];
  const double ni = Bl.norm[i];
  double ar = 0.0, ai = 0.0;
  for (int b = 0; b < L.n_bonds; ++b) {
    const uint32_t p1 = L.bond_p1[b], p2 = L.bond_p2[b];
    if (((s >> p1) & 1u) == ((s >> p2) & 1u)) {
      d += L.bond_par[b];
      continue;
    }
    d += L.bond_anti[b];
    const double tb = L.bond_t[b];
    if (tb == 0.0) continue;
    const uint32_t t = s ^ ((1u << p1) | (1u << p2));
    const uint32_t rk = L.hi_base[L.NH > 0 ? (t >> L.B) : 0u] + L.lo_rank[t & lomask];
    const uint64_t pk = Bl.full_pk[rk];
    const uint32_t j = (uint32_t)pk;
    if (j == 0xffffffffu) continue;  // an orbit not in this sector
    const uint32_t tr = (uint32_t)(pk >> 32) & 0xffu;
    const double f = tb * (Bl.norm_tab[(uint32_t)(pk >> 40)] / ni);
    const double cr = f * Bl.ph_re[tr], ci = f * Bl.ph_im[tr];
    const double yr = (double)x[2 * j], yi = (double)x[2 * j + 1];
    ar += cr * yr - ci * yi;
    ai += cr * yi + ci * yr;
  }
  const double outr = d * xr + ar, outi = d * xi + ai;
  y[2 * i] = (V)outr;
  y[2 * i + 1] = (V)outi;
  return DOT ? xr * outr + xi * outi : 0.0;
}

}  // namespace dev
}  // namespace alps_ed
