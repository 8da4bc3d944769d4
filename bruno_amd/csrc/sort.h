/*
 * sort.h -- the order of a few thousand records, by counting.
 *
 * A job's unitig heads, its branch points and a cleaning round's bubble
 * candidates are sorted by wide keys (a k-mer, with the job number or with
 * three more k-mers and a length), and there are mostly few of them.  A radix
 * sort takes a gather, up to nine launches, a copy and a wait for every key
 * of 64 bits, five keys for a bubble candidate, and each launch has less to
 * do than it costs.  Here each record counts the records before it, n^2
 * comparisons of whole keys, which is one launch that fills the device.
 */
#ifndef BRUNO_SORT_H_
#define BRUNO_SORT_H_

#include "kernels.h"

namespace br {

/* k-mers by (job, k-mer); job may be null */
template <typename KT>
struct JobKmer {
  KT key;
  uint32_t job;
  __device__ __forceinline__ bool operator<(const JobKmer& o) const {
    return job != o.job ? job < o.job : key < o.key;
  }
};
template <typename KT>
struct JobKmers {
  typedef JobKmer<KT> Item;
  const KT* key;
  const uint32_t* job;
  __device__ __forceinline__ Item operator()(uint32_t i) const { return Item{key[i], job ? job[i] : 0u}; }
};

/* rank[i] (zeroed) += the records of this workgroup's share that come before
 * record i: the smaller ones, and equal ones before it (a stable order).
 * blockIdx.x: BLOCK records i; blockIdx.y: every gridDim.y-th RANK_TILE
 * records they are compared with, through LDS, all lanes reading the same
 * one.  Bound by instruction issue, a compare and an add with carry per
 * pair; few records by the latency of the reads, so tiles are short. */
constexpr uint32_t RANK_TILE = 64;
template <typename Src>
__global__ __launch_bounds__(BLOCK) void k_rank_count(Src src, uint32_t n, uint32_t* rank) {
  typedef typename Src::Item Item;
  __shared__ Item tile[RANK_TILE];
  const uint32_t i0 = blockIdx.x * BLOCK, i = i0 + threadIdx.x;
  const Item mine = src(i < n ? i : n - 1);
  uint32_t before = 0;
  for (uint32_t j0 = blockIdx.y * RANK_TILE; j0 < n; j0 += gridDim.y * RANK_TILE) {
    const uint32_t m = n - j0 < RANK_TILE ? n - j0 : RANK_TILE;
    __syncthreads();
    if (threadIdx.x < m) tile[threadIdx.x] = src(j0 + threadIdx.x);
    __syncthreads();
    if (j0 + m <= i0) {
#pragma unroll 8
      for (uint32_t q = 0; q < m; ++q) before += !(mine < tile[q]);
    } else if (j0 >= i0 + BLOCK) {
#pragma unroll 8
      for (uint32_t q = 0; q < m; ++q) before += tile[q] < mine;
    } else {
#pragma unroll 8
      for (uint32_t q = 0; q < m; ++q) before += j0 + q < i ? !(mine < tile[q]) : tile[q] < mine;
    }
  }
  if (i < n && before) atomicAdd(&rank[i], before);
}

/* order[rank[i]] = i */
__global__ __launch_bounds__(BLOCK) void k_rank_place(const uint32_t* rank, uint32_t n, uint32_t* order) {
  const uint32_t i = blockIdx.x * BLOCK + threadIdx.x;
  if (i < n) order[rank[i]] = i;
}

}  // namespace br

#endif
