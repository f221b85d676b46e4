// Per-molecule sums of several columns, for the kernels that close an
// evaluation (tm_mol_sums, tm_force_gather_sums).  256 threads per block.
#pragma once

#include "tm_common.h"

namespace {

constexpr int SUMS_MAX_SRC = 4, SUMS_MAX_COL = 16;

// Column c is in[c][a * ld[c]] of atom a (float64 when f64[c], else float32);
// its sum over molecule m goes to out[c][m * old[c]].
struct SumCols {
  const void* in[SUMS_MAX_COL];
  double* out[SUMS_MAX_COL];
  int f64[SUMS_MAX_COL], ld[SUMS_MAX_COL], old[SUMS_MAX_COL];
  int n;
};

__device__ __forceinline__ double col_val(const SumCols& S, int c, long a) {
  return S.f64[c] ? static_cast<const double*>(S.in[c])[a * S.ld[c]]
                  : (double)static_cast<const float*>(S.in[c])[a * S.ld[c]];
}

// Sum over a 256-thread block: butterfly inside each wave, then the wave sums
// in order.  Columns go in groups of 8, whose loads are all issued before the
// first is used; column c's sum ends in thread c.
struct SumsLds {
  double part[SUMS_MAX_COL][16];
};

// Molecule m by one block of NT threads, thread t taking atoms lo + t + NT j.
template <int NT>
__device__ __forceinline__ void sums_of_molecule(const SumCols& S, const int* __restrict__ mol_start,
                                                 int m, SumsLds& L) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int lo = mol_start[m], hi = mol_start[m + 1];
  for (int c0 = 0; c0 < S.n; c0 += 8) {
    double acc[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int a = lo + tid; a < hi; a += NT) {
      double v[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = c0 + c < S.n ? col_val(S, c0 + c, a) : 0.0;
#pragma unroll
      for (int c = 0; c < 8; ++c) acc[c] += v[c];
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if (c0 + c >= S.n) break;
      const double v = tm_wave_sum_d(acc[c]);
      if (lane == 0) L.part[c0 + c][wv] = v;
    }
  }
  __syncthreads();
  if (tid < S.n) {
    double v = 0.0;
    for (int w = 0; w < NT / 64; ++w) v += L.part[tid][w];
    S.out[tid][(long)m * S.old[tid]] = v;
  }
}

// One system of n atoms by nb blocks: block k sums atoms [1024 k, 1024 (k + 1))
// of every column into the partials of work; the last block to finish
// (completion counter in work's first word, agent-scope acquire/release) adds
// the partials in block order and resets the counter to zero.  Deterministic
// whatever the block that finishes last.
__device__ __forceinline__ void sums_by_blocks(const SumCols& S, int n, int k, int nb, double* work,
                                               SumsLds& L) {
  __shared__ double stage[256];
  __shared__ int last;
  unsigned int* counter = reinterpret_cast<unsigned int*>(work);
  double* partial = work + 1;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int lo = k * 1024, hi = min(n, lo + 1024), C = S.n;
  for (int c0 = 0; c0 < C; c0 += 8) {
    double v[8][4];
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int u = 0; u < 4; ++u)   // rows past the end read row n - 1
        v[c][u] = c0 + c < C ? col_val(S, c0 + c, min(lo + u * 256 + tid, n - 1)) : 0.0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if (c0 + c >= C) break;
      double acc = 0.0;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (lo + u * 256 + tid < hi) acc += v[c][u];
      acc = tm_wave_sum_d(acc);
      if (lane == 0) L.part[c0 + c][wv] = acc;
    }
  }
  __syncthreads();
  if (tid < C)
    partial[(long)k * C + tid] = ((L.part[tid][0] + L.part[tid][1]) + L.part[tid][2]) + L.part[tid][3];
  __syncthreads();
  if (tid == 0) {
    const unsigned int done =
        __hip_atomic_fetch_add(counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    last = done == (unsigned)nb - 1u;
  }
  __syncthreads();
  if (!last) return;
  __threadfence();
  // partials [nb][C] staged 256 at a time; thread c < C adds column c in block order
  const int tot_n = nb * C;
  double tot = 0.0;
  for (int e0 = 0; e0 < tot_n; e0 += 256) {
    stage[tid] = e0 + tid < tot_n ? partial[e0 + tid] : 0.0;
    __syncthreads();
    if (tid < C) {
      const int e1 = min(e0 + 256, tot_n);
      for (int e = e0 + ((tid - e0 % C) + C) % C; e < e1; e += C) tot += stage[e - e0];
    }
    __syncthreads();
  }
  if (tid < C) S.out[tid][0] = tot;
  if (tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The columns of nsrc sources (host arrays, as tm_mol_sums takes them).
inline int sum_cols(const char* name, int B, int n_total, int nsrc, const void* const* in,
                    const int* f64, const int* cols, const int* ld, double* const* out, SumCols* S) {
  TM_REQUIRE(B >= 0 && n_total >= 0 && nsrc > 0 && nsrc <= SUMS_MAX_SRC, "%s: bad sizes", name);
  *S = SumCols{};
  for (int k = 0; k < nsrc; ++k) {
    TM_REQUIRE(cols[k] > 0 && ld[k] >= cols[k] && in[k] != nullptr && out[k] != nullptr,
               "%s: bad source %d", name, k);
    TM_REQUIRE(S->n + cols[k] <= SUMS_MAX_COL, "%s: more than %d columns", name, SUMS_MAX_COL);
    for (int c = 0; c < cols[k]; ++c) {
      const int q = S->n++;
      S->in[q] = static_cast<const char*>(in[k]) + (f64[k] ? 8 : 4) * (long)c;
      S->out[q] = out[k] + c;
      S->f64[q] = f64[k];
      S->ld[q] = ld[k];
      S->old[q] = cols[k];
    }
  }
  return TM_OK;
}

}  // namespace
