/*
 * partition.h -- grouping a count's instance records by table region.
 *
 * The record parser (k_parse_records, regions.h) leaves one record per k-mer
 * instance, rec = (hash << 5) | biedge index, in buckets picked by the
 * hash's top `beta` bits (up to 512 buckets per job).  A bucket is a list of
 * chunks taken from one pool, so no bucket has a capacity of its own.  The
 * next hash bits (b2 of them) name the region inside the bucket, and one
 * multisplit pass, k_split, groups every bucket's records by region, in
 * pieces of 64 records that a region's build reads with one wave each.
 *
 * One workgroup owns a bucket: it sorts tile after tile by digit in LDS and
 * appends each digit's run to the digit's open piece, taking new pieces from
 * the bucket's own room (its chunks, and one piece per region) with a counter
 * of its own: no global atomic, and no pass over the records to count them
 * first (a region's count cannot be estimated: a k-mer repeated thousands of
 * times puts all its instances in one region).  The pieces' regions, a 64th
 * of the records, are grouped at the end instead.  A tile fills 128 KB of
 * LDS, one 1,024-thread workgroup per CU, so that a run of a tile is still
 * 64 bytes when a bucket has 2,048 regions; 256 buckets are one per CU.
 *
 * The records are read and written once, 2.7 TB/s at 1.6 G records of 8
 * bytes (9.4 ms; LDS work and the barriers between a tile's steps take the
 * rest).  Contiguous regions behind a count pass took 12.9 ms.  Before that, 32
 * coarser buckets and two passes (on small tables, 32 workgroups in the
 * second) took 0.73 ms for 21 M records (now 0.13), 1.84 for 184 M (1.09),
 * 5.5 for 301 M of 16 bytes (3.6).
 *
 * The order of records inside a region is not kept, which nothing
 * downstream depends on (a region's slots come out the same up to the order
 * of keys inside a probe run).
 */
#ifndef BRUNO_PARTITION_H_
#define BRUNO_PARTITION_H_

#include "kernels.h"

namespace br {

/* A record drops the hash's top REC_BUCKET_BITS bits, so every job has at
 * least that many bucket bits. */
constexpr int REC_BUCKET_BITS = 5;
constexpr int MAX_BUCKET_BITS = 9;
constexpr int SPLIT_BS = 1024;
constexpr int SPLIT_BITS = 11, SPLIT_MAX_BITS = 12; /* region bits a bucket is split by: usual, more than 2^19 regions */
constexpr uint32_t REC_CODE_FILL = 31; /* chunk padding, never a biedge index (0..24) */
constexpr uint32_t NO_CHUNK = ~0u;
constexpr int REC_CHUNK_LOG = 10, REC_CHUNK_LOG_MIN = 6; /* log2 records per chunk: at most SPLIT_BS, at least a piece */

/* A record: one word (k <= 31) or the key word and the k-mer's high word
 * (k <= 63).  The key word, (hash << 5) | biedge index, is what the split
 * goes by. */
template <typename KT> struct RecOf;
template <> struct RecOf<uint64_t> { typedef uint64_t T; };
template <> struct RecOf<u128> { typedef ulonglong2 T; };
__device__ __forceinline__ uint64_t rec_key(uint64_t r) { return r; }
__device__ __forceinline__ uint64_t rec_key(const ulonglong2& r) { return r.x; }
template <typename R> __device__ __forceinline__ R rec_zero();
template <> __device__ __forceinline__ uint64_t rec_zero<uint64_t>() { return 0; }
template <> __device__ __forceinline__ ulonglong2 rec_zero<ulonglong2>() { return make_ulonglong2(0, 0); }

/* the job holding bucket / region x: the largest j with first(j) <= x */
template <typename F>
__device__ __forceinline__ uint32_t count_job_of(uint32_t n_jobs, uint32_t x, F first) {
  uint32_t lo = 0, hi = n_jobs;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (first(mid) <= x) lo = mid;
    else hi = mid;
  }
  return lo;
}

/* The chunk pool: chunk c holds records [c << clog, (c + 1) << clog) of one
 * bucket.  A parser workgroup takes numbers ahead, as many as it has
 * buckets at a time. */
struct ChunkPool {
  void* recs;                 /* RecOf<KT>::T */
  uint32_t clog;              /* log2 records per chunk */
  uint32_t n_max;             /* chunks the pool has room for */
  uint32_t* next;             /* chunks taken */
  uint32_t* taken;            /* per bucket: chunks taken */
  uint32_t* owner;            /* per chunk: its bucket (NO_CHUNK: not used) */
  uint32_t* overflow;         /* set when records found no room (the count then starts over with atomics) */
};

/* first[b] = chunks of the buckets from b_lo to b (first[b_hi] = all); a
 * bucket with more than `limit` chunks sets the overflow flag: one k-mer in a large
 * share of all instances would leave one workgroup the work of the whole
 * device.  One workgroup. */
__global__ __launch_bounds__(1024) void k_chunk_first(ChunkPool p, uint32_t b_lo, uint32_t b_hi, uint32_t limit,
                                                      uint32_t* first) {
  typedef hipcub::BlockScan<uint32_t, 1024> Scan;
  __shared__ typename Scan::TempStorage tmp;
  uint32_t before = 0;
  for (uint32_t b0 = b_lo; b0 < b_hi; b0 += 1024) {
    const uint32_t b = b0 + threadIdx.x;
    const uint32_t v = b < b_hi ? p.taken[b] : 0;
    if (v > limit) *p.overflow = 1;
    uint32_t at, total;
    Scan(tmp).ExclusiveSum(v, at, total);
    if (b < b_hi) first[b] = before + at;
    before += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) first[b_hi] = before;
}

/* The chunks in bucket order (in any order within a bucket).  listed counts
 * a bucket's chunks so far, one counter per cache line: with 32 in a line
 * the atomics on it took 0.5 ms for 1.6 M chunks. */
constexpr uint32_t LISTED_STRIDE = 32;
__global__ __launch_bounds__(BLOCK) void k_chunk_list(ChunkPool p, uint32_t b_lo, const uint32_t* first,
                                                      uint32_t* listed, uint32_t* list) {
  if (*p.overflow) return; /* chunks may be missing, or a bucket too large */
  const uint32_t n = min(*p.next, p.n_max);
  for (uint32_t c = blockIdx.x * BLOCK + threadIdx.x; c < n; c += gridDim.x * BLOCK) {
    const uint32_t b = p.owner[c];
    if (b != NO_CHUNK) list[first[b] + atomicAdd(&listed[(uint64_t)(b - b_lo) * LISTED_STRIDE], 1u)] = c;
  }
}

/* The split's output: pieces of 64 records (one per lane of a build's wave).
 * A region's records are the pieces list[region_start ...], all full but
 * the last. */
constexpr int PIECE_LOG = 6;
constexpr uint32_t PIECE = 1u << PIECE_LOG;

/* tile of the split: 128 KB of records, less with twice the digits (both
 * beside the digits' state in the CU's 160 KB) */
template <typename R, int BITS> struct SplitShape {
  static constexpr int FULL = (int)((128 << 10) / sizeof(R) / SPLIT_BS);
  static constexpr int ITEMS = BITS > SPLIT_BITS ? FULL * 13 / 16 : FULL;
  static constexpr int TILE = ITEMS * SPLIT_BS;
};

struct SplitArgs {
  ChunkPool pool;
  const uint32_t* first;      /* by bucket, see k_chunk_first */
  const uint32_t* list;       /* chunks in bucket order */
  const JobLayout* jobs;
  uint32_t n_jobs;
  uint32_t b0, b1;            /* this launch: buckets [b0, b1) */
  uint32_t q_lo;              /* the pass's first region */
  void* out;                  /* pieces; bucket b's from piece_base(b) */
  uint16_t* digit_of;         /* per piece: its region's place in the bucket */
  uint32_t* pieces;           /* per region its pieces, from region_start on */
  uint32_t* region_start;
  uint32_t* region_count;     /* records */
};

template <typename R, int BITS>
__global__ __launch_bounds__(SPLIT_BS) void k_split(SplitArgs a) {
  constexpr int ITEMS = SplitShape<R, BITS>::ITEMS, TILE = SplitShape<R, BITS>::TILE;
  constexpr int MAXD = 1 << BITS, DPT = MAXD / SPLIT_BS; /* digits per thread of the scan */
  __shared__ R buf[TILE];
  __shared__ uint32_t cnt[MAXD + 1]; /* a tile's counts, then first place | first new piece << 16 */
  __shared__ uint32_t nxt[MAXD];     /* next place of each digit in the bucket's pieces (a multiple of PIECE: none open) */
  __shared__ uint32_t tot[MAXD];     /* records so far */
  __shared__ uint32_t part[SPLIT_BS / 64];
  if (*a.pool.overflow) return;
  const R* in = (const R*)a.pool.recs;
  const uint32_t clog = a.pool.clog, cmask = (1u << clog) - 1;
  for (uint32_t b = a.b0 + blockIdx.x; b < a.b1; b += gridDim.x) {
    const uint32_t ji = count_job_of(a.n_jobs, b, [&](uint32_t q) { return a.jobs[q].bucket0; });
    const uint32_t beta = a.jobs[ji].beta, b2 = a.jobs[ji].rbits - beta;
    /* the digit: the b2 hash bits below the bucket's */
    const uint32_t nd = 1u << b2, dmask = nd - 1;
    const int sh = 64 + REC_BUCKET_BITS - (int)beta - (int)b2;
    auto digit = [&](uint64_t x) -> uint32_t { return b2 ? (uint32_t)(x >> sh) & dmask : 0u; };
    const uint32_t l0 = a.first[b];
    const uint64_t n = (uint64_t)(a.first[b + 1] - l0) << clog;
    const uint32_t* list = a.list + l0;
    /* the bucket's pieces: room for its chunks and one more per region */
    const uint32_t g0 = a.jobs[ji].region0 + ((b - a.jobs[ji].bucket0) << b2);
    const uint32_t p0 = (l0 << (clog - PIECE_LOG)) + (g0 - a.q_lo);
    R* out = (R*)a.out + ((uint64_t)p0 << PIECE_LOG);
    uint16_t* digit_of = a.digit_of + p0;
    /* Record slot k of a tile is the tile's record k * SPLIT_BS + thread; m
     * (wave-uniform) is what is left of the bucket, so a slot is filled when
     * thread < m - k * SPLIT_BS.  A chunk holds 64 to SPLIT_BS records, so a
     * wave's record slot has one chunk and a thread one place in it; the
     * chunk numbers are read a tile ahead of the records. */
    const uint32_t in_chunk = threadIdx.x & cmask;
    auto left = [&](uint64_t i0) -> int { return i0 < n ? (int)(n - i0 < (uint64_t)TILE ? n - i0 : TILE) : 0; };
    auto load_list = [&](uint64_t i0, uint32_t (&ln)[ITEMS]) {
      const int m = left(i0);
      const uint32_t* l = list + (i0 >> clog);
      const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)threadIdx.x) >> clog;
#pragma unroll
      for (int k = 0; k < ITEMS; ++k) {
        ln[k] = 0;
        if ((int)threadIdx.x < m - k * SPLIT_BS) ln[k] = l[w + ((uint32_t)(k * SPLIT_BS) >> clog)];
      }
    };
    auto load = [&](uint64_t i0, const uint32_t (&ln)[ITEMS], R (&r)[ITEMS]) {
      const int m = left(i0);
#pragma unroll
      for (int k = 0; k < ITEMS; ++k) {
        r[k] = rec_zero<R>();
        if ((int)threadIdx.x < m - k * SPLIT_BS)
          r[k] = in[((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)ln[k]) << clog) + in_chunk];
      }
    };
    /* exclusive prefix of v over the digits, thread t holding digits
     * t * DPT ...; v is replaced by it, the sum returned.  One barrier (LDS
     * only: records in flight are not waited for). */
    auto scan = [&](uint32_t (&v)[DPT]) -> uint32_t {
      uint32_t mine = 0;
#pragma unroll
      for (int q = 0; q < DPT; ++q) {
        const uint32_t c = v[q];
        v[q] = mine;
        mine += c;
      }
      uint32_t incl = mine;
      const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
      }
      if (lane == 63) part[w] = incl;
      lds_barrier();
      /* the waves' sums: lane l takes wave l's */
      constexpr int NW = SPLIT_BS / 64;
      uint32_t x = part[lane & (NW - 1)];
#pragma unroll
      for (int off = 1; off < NW; off <<= 1) {
        const uint32_t o = __shfl_up(x, off, 64);
        if (lane >= off) x += o;
      }
      const uint32_t sum = (uint32_t)__builtin_amdgcn_readlane((int)x, NW - 1);
      const int wu = __builtin_amdgcn_readfirstlane(w);
      const uint32_t before = incl - mine + (wu ? (uint32_t)__builtin_amdgcn_readlane((int)x, wu - 1) : 0u);
#pragma unroll
      for (int q = 0; q < DPT; ++q) v[q] += before;
      return sum;
    };
    for (uint32_t d = threadIdx.x; d < MAXD; d += SPLIT_BS) cnt[d] = nxt[d] = tot[d] = 0;
    lds_barrier();
    uint32_t n_pieces = 0;
    uint32_t ln[ITEMS];
    R r[ITEMS];
    load_list(0, ln);
    load(0, ln, r);
    load_list(TILE, ln);
    for (uint64_t i0 = 0; i0 < n; i0 += TILE) {
      uint32_t okm = 0;
      const int m = left(i0);
#pragma unroll
      for (int k = 0; k < ITEMS; ++k)
        if ((int)threadIdx.x < m - k * SPLIT_BS && (rec_key(r[k]) & 31) != REC_CODE_FILL) okm |= 1u << k;
      /* digit << 16 | rank among the tile's records of the digit (a tile has
       * at most 2^14 records, a digit 12 bits) */
      uint32_t dr[ITEMS];
#pragma unroll
      for (int k = 0; k < ITEMS; ++k) {
        const uint32_t d = digit(rec_key(r[k]));
        dr[k] = d << 16 | (okm >> k & 1u ? atomicAdd(&cnt[d], 1u) : 0u);
      }
      lds_barrier();
      /* A digit's run fills its open piece (`room` places), then new pieces
       * in a row.  Counts and new pieces are scanned as one word (sums of at
       * most 2^14 and 2^14 / PIECE + 2^12). */
      uint32_t c[DPT], v[DPT];
#pragma unroll
      for (int q = 0; q < DPT; ++q) {
        const uint32_t d = threadIdx.x * DPT + q, room = -nxt[d] & (PIECE - 1);
        c[q] = cnt[d];
        v[q] = c[q] | (c[q] > room ? (c[q] - room + PIECE - 1) >> PIECE_LOG : 0) << 16;
      }
      const uint32_t sum = scan(v), total = sum & 0xFFFF;
#pragma unroll
      for (int q = 0; q < DPT; ++q) cnt[threadIdx.x * DPT + q] = v[q];
      lds_barrier();
#pragma unroll
      for (int k = 0; k < ITEMS; ++k)
        if (okm >> k & 1u) buf[(cnt[dr[k] >> 16] & 0xFFFFu) + (dr[k] & 0xFFFFu)] = r[k];
      lds_barrier();
      /* the next tile's records, ahead of this one's stores (loads and
       * stores complete in order) */
      if (i0 + TILE < n) {
        load(i0 + TILE, ln, r);
        load_list(i0 + 2 * (uint64_t)TILE, ln);
      }
#pragma unroll 1
      for (uint32_t i = threadIdx.x; i < total; i += SPLIT_BS) {
        const R x = buf[i];
        const uint32_t d = digit(rec_key(x)), w = cnt[d], p = nxt[d];
        const uint32_t rank = i - (w & 0xFFFFu), room = -p & (PIECE - 1);
        out[rank < room ? p + rank : ((n_pieces + (w >> 16)) << PIECE_LOG) + (rank - room)] = x;
      }
      lds_barrier();
#pragma unroll
      for (int q = 0; q < DPT; ++q) {
        const uint32_t d = threadIdx.x * DPT + q, p = nxt[d], room = -p & (PIECE - 1);
        const uint32_t np = n_pieces + (v[q] >> 16);
        if (c[q] > room) {
          const uint32_t more = c[q] - room;
#pragma unroll 1
          for (uint32_t i = 0; i << PIECE_LOG < more; ++i) digit_of[np + i] = (uint16_t)d;
          nxt[d] = (np << PIECE_LOG) + more;
        } else {
          nxt[d] = p + c[q];
        }
        tot[d] += c[q];
        cnt[d] = 0;
      }
      n_pieces += sum >> 16;
      lds_barrier();
    }
    /* the regions' pieces in order: the full ones as they come, an open one
     * last */
    {
      uint32_t v[DPT];
#pragma unroll
      for (int q = 0; q < DPT; ++q) v[q] = (tot[threadIdx.x * DPT + q] + PIECE - 1) >> PIECE_LOG;
      scan(v);
#pragma unroll
      for (int q = 0; q < DPT; ++q) {
        const uint32_t d = threadIdx.x * DPT + q;
        cnt[d] = v[q];
        if (d < nd) {
          a.region_start[g0 + d] = p0 + v[q];
          a.region_count[g0 + d] = tot[d];
        }
      }
      __syncthreads();
      for (uint32_t i = threadIdx.x; i < n_pieces; i += SPLIT_BS) {
        const uint32_t d = digit_of[i], p = nxt[d];
        if (p >> PIECE_LOG != i || !(p & (PIECE - 1))) a.pieces[p0 + atomicAdd(&cnt[d], 1u)] = p0 + i;
      }
      __syncthreads();
      for (uint32_t d = threadIdx.x; d < nd; d += SPLIT_BS)
        if (nxt[d] & (PIECE - 1)) a.pieces[p0 + cnt[d]] = p0 + (nxt[d] >> PIECE_LOG);
    }
    __syncthreads();
  }
}

}  // namespace br

#endif
