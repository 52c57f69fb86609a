// ed_batch_kernels.hip -- gfx950 kernels that advance many Lanczos solves
// in one launch (see ed_batch.hpp).  Every work item reads its problem's
// descriptor with wave-uniform (scalar) loads, then runs the same per-segment
// H.v and per-chunk vector code as the single-solve kernels.
#include <hip/hip_runtime.h>

#include "ed_batch.hpp"
#include "ed_device.hpp"

namespace alps_ed {

namespace {

using namespace dev;

template <class V>
__device__ __forceinline__ V* slot_ptr(void* vec, uint64_t stride, uint32_t cap, int j) {
  return static_cast<V*>(vec) + (uint64_t)((uint32_t)j % cap) * stride;
}

template <class V>
__global__ __launch_bounds__(kBlock) void batch_start_kernel(const BatchJob* __restrict__ jobs,
                                                             const BatchItem* __restrict__ items) {
  const BatchItem it = ldc_struct(items + blockIdx.x);
  const BatchJob* J = jobs + it.job;
  const uint32_t D = ldc(&J->n);
  const uint64_t seed = ldc(&J->seed);
  V* u = static_cast<V*>(ldc(&J->vec));
  double* part = ldc(&J->part_up);
  const uint32_t r0 = it.idx * kBatchChunk;
  const uint32_t r1 = min(D, r0 + kBatchChunk);
  double acc = 0.0;
  for (uint32_t i = r0 + threadIdx.x; i < r1; i += kBlock) {
    const V v = (V)start_value(seed, i, -1.0, 1.0);
    u[i] = v;
    acc += (double)v * (double)v;
  }
  const double s = block_sum_all(acc);
  if (threadIdx.x == 0) part[it.idx] = s;
}

// Each form has a launch of its own, so that none's code costs the others
// registers.
template <class V, BatchHv FORM>
__global__ __launch_bounds__(kBlock, HvWaves<V>::value) void batch_hv_kernel(const BatchJob* __restrict__ jobs,
                                                          const BatchItem* __restrict__ items, int t) {
  const BatchItem it = ldc_struct(items + blockIdx.x);
  const BatchJob* J = jobs + it.job;
  const int j = ldc(&J->j0) + t;
  if (j >= ldc(&J->jmax)) return;  // uniform over the workgroup
  const DevLayout L = ldc_struct(&J->L);
  void* vec = ldc(&J->vec);
  const uint64_t stride = ldc(&J->stride);
  const uint32_t cap = ldc(&J->cap);
  const V* x = slot_ptr<V>(vec, stride, cap, j);
  V* y = slot_ptr<V>(vec, stride, cap, j + 1);
  double* part = ldc(&J->part_hv);
  if (FORM == kHvGathered && ldc(&J->Bl.dk) != 0u) {  // momentum sector: uniform over the workgroup
    const DevBloch Bl = ldc_struct(&J->Bl);
    const double p = bloch_row<V, true>(L, Bl, x, y, it.idx * kBlock + threadIdx.x);
    store_block_sum_lds<kBlock>(part + it.idx, p);
    return;
  }
  if constexpr (FORM == kHvTables)
    hv_ranked_at<V, true>(L, seg_record(L, it.idx, false, true), x, y, part + it.idx);
  else
    hv_segment_at<V, true, FORM == kHvStaged>(L, seg_record(L, it.idx, FORM == kHvStaged, false), x, y, part + it.idx);
}

// Where stage j (the start for j = 0, the update of step j - 1 otherwise)
// leaves its partials of |u_j|^2: two buffers in turn, as the blocks of an
// update read one while others fill the next.
__device__ __forceinline__ double* norm_part(const BatchJob* J, int j) {
  return ldc(&J->part_up) + ((j & 1) != 0 ? ldc(&J->n_chunks) : 0u);
}

// One row chunk of an update.  A fused job's blocks each form alpha_j, scale_j
// and beta_{j-1} from the partials (in the same order as batch_finish_kernel,
// so the values are the same) while their vector elements, read before, are
// on the way; the first block stores them.  Bound by latency at the sizes of a
// batch: 64 chains of 12 to 20 sites 12.6 us, against 9.8 us and two
// reduction launches of 3.6 us each.
template <class V>
__global__ __launch_bounds__(kBlock) void batch_update_kernel(const BatchJob* __restrict__ jobs,
                                                              const BatchItem* __restrict__ items, int t) {
  typedef V v4 __attribute__((ext_vector_type(4), aligned(sizeof(V))));
  const BatchItem it = ldc_struct(items + blockIdx.x);
  const BatchJob* J = jobs + it.job;
  const int j = ldc(&J->j0) + t;
  if (j >= ldc(&J->jmax)) return;
  const uint32_t D = ldc(&J->n);
  void* vec = ldc(&J->vec);
  const uint64_t stride = ldc(&J->stride);
  const uint32_t cap = ldc(&J->cap);
  const V* u = slot_ptr<V>(vec, stride, cap, j);
  V* w = slot_ptr<V>(vec, stride, cap, j + 1);
  double* alpha = ldc(&J->alpha);
  double* beta = ldc(&J->beta);
  double* scale = ldc(&J->scale);
  const bool has_prev = j > 0;
  const V* up = has_prev ? slot_ptr<V>(vec, stride, cap, j - 1) : u;
  // four consecutive rows per thread (slots are 256-byte aligned, chunks
  // start at multiples of kBatchChunk rows)
  const uint32_t i0 = it.idx * kBatchChunk + 4u * threadIdx.x;
  const bool full = i0 + 4u <= D;
  v4 wv, uv, pv;
  if (full) {
    wv = *reinterpret_cast<const v4*>(w + i0);
    uv = *reinterpret_cast<const v4*>(u + i0);
    pv = *reinterpret_cast<const v4*>(up + i0);
  }
  double sc, a, b = 0.0;
  if (ldc(&J->fuse) != 0u) {  // uniform over the workgroup
    double nsum = thread_partials(Partials{norm_part(J, j), ldc(&J->n_chunks)});
    double hsum = thread_partials(Partials{ldc(&J->part_hv), ldc(&J->n_hv)});
    update_sums<kBlock>(nsum, hsum);
    const double nrm = sqrt(nsum);
    sc = 1.0 / nrm;
    a = sc * sc * hsum;
    if (it.idx == 0u && threadIdx.x == 0u) {
      alpha[j] = a;
      ldc(&J->host_alpha)[j] = a;
      if (t > 0 || j == 0) scale[j] = sc;  // the last launch of a group before stored it
      if (t > 0 && has_prev) {
        beta[j - 1] = nrm;
        ldc(&J->host_beta)[j - 1] = nrm;
      }
    }
    if (has_prev) b = nrm;
  } else {
    sc = ldc(scale + j);
    a = ldc(alpha + j);
    if (has_prev) b = ldc(beta + j - 1);
  }
  const double ca = a * sc;
  double cb = 0.0;
  if (has_prev) {
    // scale_{j-1}: of the step before, which may be of this launch group
    cb = b * scale[j - 1];
  }
  double acc = 0.0;
  if (full) {
    v4 o;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      double r = sc * (double)wv[c] - ca * (double)uv[c];
      if (has_prev) r -= cb * (double)pv[c];
      o[c] = (V)r;
      const double rd = (double)o[c];
      acc += rd * rd;
    }
    *reinterpret_cast<v4*>(w + i0) = o;
  } else {
    for (uint32_t i = i0; i < D && i < i0 + 4u; ++i) {
      double r = sc * (double)w[i] - ca * (double)u[i];
      if (has_prev) r -= cb * (double)up[i];
      const V rs = (V)r;
      w[i] = rs;
      const double rd = (double)rs;
      acc += rd * rd;
    }
  }
  const double s = block_sum_all(acc);
  if (threadIdx.x == 0) norm_part(J, j + 1)[it.idx] = s;
}

__global__ __launch_bounds__(kBlock) void batch_finish_kernel(const BatchJob* __restrict__ jobs,
                                                              const uint32_t* __restrict__ job_list, int t,
                                                              int mode) {
  const BatchJob* J = jobs + ldc(job_list + blockIdx.x);
  const int jmax = ldc(&J->jmax), j0 = ldc(&J->j0);
  int j = j0 + t;
  if (mode == kBatchLast) {  // t: the steps of the group
    j = min(j, jmax) - 1;
    if (j < j0) return;
  } else if (mode != kBatchStart && j >= jmax) {
    return;
  }
  const bool hv = mode == kBatchAlpha;
  const double* part = hv ? ldc(&J->part_hv) : norm_part(J, mode == kBatchStart ? 0 : j + 1);
  const uint32_t n = hv ? ldc(&J->n_hv) : ldc(&J->n_chunks);
  const double s = sum_partials(Partials{part, n});
  if (threadIdx.x != 0) return;
  double* scale = ldc(&J->scale);
  if (mode == kBatchStart) {
    scale[0] = 1.0 / sqrt(s);
  } else if (mode == kBatchAlpha) {
    const double sj = scale[j];
    const double a = sj * sj * s;
    ldc(&J->alpha)[j] = a;
    ldc(&J->host_alpha)[j] = a;
  } else {
    const double b = sqrt(s);
    ldc(&J->beta)[j] = b;
    ldc(&J->host_beta)[j] = b;
    scale[j + 1] = 1.0 / b;
  }
}

// Rows r0 + 4 tid .. + 3 of NV Ritz vectors of a chunk, kRitzAhead basis
// vectors in flight; their squares into acc2.
template <class V, int NV>
__device__ __forceinline__ void ritz_rows(const RitzJob* J, uint32_t r0, int nv, double (&acc2)[NV]) {
  typedef V v4 __attribute__((ext_vector_type(4), aligned(sizeof(V))));
  typedef double o4 __attribute__((ext_vector_type(4), aligned(8)));
  constexpr int kRitzAhead = 8;
  const V* vec = static_cast<const V*>(ldc(&J->vec));
  const uint64_t stride = ldc(&J->stride);
  const uint32_t D = ldc(&J->D);
  const int m = ldc(&J->m);
  const double* scale = ldc(&J->scale);
  const double* coef = ldc(&J->coef);
  double* out = ldc(&J->out);
  const uint32_t r = r0 + 4u * threadIdx.x;
  double acc[NV][4];
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[i][e] = 0.0;
  auto add = [&](int j, const v4& u) {
    const double sj = ldc(scale + j);
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (i < nv) {
        const double c = ldc(coef + (size_t)i * m + j);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][e] += c * (sj * (double)u[e]);
      }
  };
  if (r + 4u <= D) {
    int j = 0;
    for (; j + kRitzAhead <= m; j += kRitzAhead) {
      v4 u[kRitzAhead];
#pragma unroll
      for (int c = 0; c < kRitzAhead; ++c) u[c] = *reinterpret_cast<const v4*>(vec + (uint64_t)(j + c) * stride + r);
      issue_barrier();
#pragma unroll
      for (int c = 0; c < kRitzAhead; ++c) add(j + c, u[c]);
    }
    for (; j < m; ++j) add(j, *reinterpret_cast<const v4*>(vec + (uint64_t)j * stride + r));
  } else if (r < D) {
    for (int j = 0; j < m; ++j) {
      v4 u = {(V)0, (V)0, (V)0, (V)0};
      for (uint32_t e = 0; e < 3u; ++e)
        if (r + e < D) u[e] = vec[(uint64_t)j * stride + r + e];
      add(j, u);
    }
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    acc2[i] = 0.0;
    if (i < nv && r < D) {
      double* o = out + (uint64_t)i * D + r;
      if (r + 4u <= D) *reinterpret_cast<o4*>(o) = o4{acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
#pragma unroll
      for (uint32_t e = 0; e < 4u; ++e)
        if (r + e < D) {
          if (r + 4u > D) o[e] = acc[i][e];
          acc2[i] += acc[i][e] * acc[i][e];
        }
    }
  }
}

// Bound by the read of the kept basis; with a handful of problems in a launch
// by the rounds of dependent waits per row, of which four rows per thread and
// eight vectors at a time leave one in 32: 130 -> 38 us for a tenth of 64
// chains of 12 to 20 sites.
template <class V>
__global__ __launch_bounds__(kBlock) void batch_ritz_kernel(const RitzJob* __restrict__ jobs,
                                                            const BatchItem* __restrict__ items) {
  const BatchItem it = ldc_struct(items + blockIdx.x);
  const RitzJob* J = jobs + it.job;
  const int nv = ldc(&J->nv);
  double acc2[kMaxRitz];
#pragma unroll
  for (int i = 0; i < kMaxRitz; ++i) acc2[i] = 0.0;
  if (nv == 1) {  // uniform
    double one[1];
    ritz_rows<V, 1>(J, it.idx * kBatchChunk, nv, one);
    acc2[0] = one[0];
  } else {
    ritz_rows<V, kMaxRitz>(J, it.idx * kBatchChunk, nv, acc2);
  }
  double* part = ldc(&J->part);
  const uint32_t nc = ldc(&J->n_chunks);
#pragma unroll
  for (int i = 0; i < kMaxRitz; ++i) {
    if (i < nv) {  // uniform: every thread reaches the same barriers
      const double s = block_sum_all(acc2[i]);
      if (threadIdx.x == 0) part[(uint64_t)i * nc + it.idx] = s;
    }
  }
}

// y = H x of a refinement, once per reported level: all forms in one kernel
// (the registers that they cost each other matter in the steps, not here), the
// page also for short segments.
__global__ __launch_bounds__(kBlock) void batch_plain_hv_kernel(const PlainHvJob* __restrict__ jobs,
                                                                const BatchItem* __restrict__ items) {
  const BatchItem it = ldc_struct(items + blockIdx.x);
  const PlainHvJob* J = jobs + it.job;
  const DevLayout L = ldc_struct(&J->L);
  if (ldc(&J->Bl.dk) != 0u) {  // momentum sector: uniform over the workgroup
    const DevBloch Bl = ldc_struct(&J->Bl);
    const double p = bloch_row<double, true>(L, Bl, ldc(&J->x), ldc(&J->y), it.idx * kBlock + threadIdx.x);
    store_block_sum_lds<kBlock>(ldc(&J->part) + it.idx, p);
    return;
  }
  if (L.n_xs > 0)
    hv_segment_at<double, true, true>(L, seg_record(L, it.idx, true, false), ldc(&J->x), ldc(&J->y), ldc(&J->part) + it.idx);
  else
    hv_segment_at<double, true, false>(L, seg_record(L, it.idx, false, false), ldc(&J->x), ldc(&J->y), ldc(&J->part) + it.idx);
}

}  // namespace

template <class V>
hipError_t launch_batch_start(const BatchJob* jobs, const BatchItem* items, uint32_t n_items, hipStream_t st) {
  if (n_items == 0) return hipSuccess;
  hipLaunchKernelGGL((batch_start_kernel<V>), dim3(n_items), dim3(kBlock), 0, st, jobs, items);
  return hipGetLastError();
}

template <class V>
hipError_t launch_batch_hv(const BatchJob* jobs, const BatchItem* items, uint32_t n_items, int t, BatchHv form,
                           uint32_t lds, hipStream_t st) {
  if (n_items == 0) return hipSuccess;
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(n_items), dim3(kBlock), lds, st, jobs, items, t); };
  if (form == kHvTables) launch(batch_hv_kernel<V, kHvTables>);
  else if (form == kHvStaged) launch(batch_hv_kernel<V, kHvStaged>);
  else launch(batch_hv_kernel<V, kHvGathered>);
  return hipGetLastError();
}

template <class V>
hipError_t launch_batch_update(const BatchJob* jobs, const BatchItem* items, uint32_t n_items, int t,
                               hipStream_t st) {
  if (n_items == 0) return hipSuccess;
  hipLaunchKernelGGL((batch_update_kernel<V>), dim3(n_items), dim3(kBlock), 0, st, jobs, items, t);
  return hipGetLastError();
}

hipError_t launch_batch_finish(const BatchJob* jobs, const uint32_t* job_list, uint32_t n_jobs, int t, int mode,
                               hipStream_t st) {
  if (n_jobs == 0) return hipSuccess;
  hipLaunchKernelGGL(batch_finish_kernel, dim3(n_jobs), dim3(kBlock), 0, st, jobs, job_list, t, mode);
  return hipGetLastError();
}

template <class V>
hipError_t launch_batch_ritz(const RitzJob* jobs, const BatchItem* items, uint32_t n_items, hipStream_t st) {
  if (n_items == 0) return hipSuccess;
  hipLaunchKernelGGL((batch_ritz_kernel<V>), dim3(n_items), dim3(kBlock), 0, st, jobs, items);
  return hipGetLastError();
}

hipError_t launch_batch_plain_hv(const PlainHvJob* jobs, const BatchItem* items, uint32_t n_items,
                                 uint32_t lds, hipStream_t st) {
  if (n_items == 0) return hipSuccess;
  hipLaunchKernelGGL(batch_plain_hv_kernel, dim3(n_items), dim3(kBlock), lds, st, jobs, items);
  return hipGetLastError();
}

#define ALPS_ED_BATCH_INSTANTIATE(V)                                                                           \
  template hipError_t launch_batch_start<V>(const BatchJob*, const BatchItem*, uint32_t, hipStream_t);       \
  template hipError_t launch_batch_hv<V>(const BatchJob*, const BatchItem*, uint32_t, int, BatchHv, uint32_t, \
                                         hipStream_t);                                                       \
  template hipError_t launch_batch_update<V>(const BatchJob*, const BatchItem*, uint32_t, int, hipStream_t); \
  template hipError_t launch_batch_ritz<V>(const RitzJob*, const BatchItem*, uint32_t, hipStream_t);

ALPS_ED_BATCH_INSTANTIATE(float)
ALPS_ED_BATCH_INSTANTIATE(double)

}  // namespace alps_ed
