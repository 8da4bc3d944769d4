/*
 * regions.h -- counting by table region (k <= 63).
 *
 * A job's table is 2^rbits regions of span slots (one region fills a build
 * workgroup's LDS at most); a k-mer's probe window never leaves the region
 * its hash's top rbits bits pick (see Probe in table.h).  Counting then needs
 * no HBM atomics on the table:
 *
 *   1. k_parse_records: one read per lane, k-mer and reverse complement
 *      rolled along the read; each instance becomes a record (8 bytes,
 *      (hash bits 0..58) << 5 | biedge index; k > 31 adds the k-mer's high
 *      word) in one of its job's 2^beta buckets picked by the top hash bits.
 *      A workgroup stages records per bucket in LDS and appends whole cache
 *      lines to chunks of a common pool.
 *   2. k_split (partition.h) groups each bucket's records by region, in
 *      pieces of 64, and lists every region's pieces.
 *   3. k_region_build: a workgroup takes regions one by one; per region it
 *      loads the slots into LDS (or starts from EMPTY when the table holds
 *      nothing yet), adds the region's records with LDS atomics, and writes
 *      the region back with coalesced stores.  Entries beyond a slot's NSUB
 *      sub-entries go to the HBM side table exactly as in the atomic count.
 *
 * A batch's jobs go through the same launches: every parser workgroup reads
 * one job's reads, buckets and regions are numbered through all jobs, and a
 * region's job gives its layout.
 *
 * The table contents equal those of the atomic count up to the order of
 * keys inside a probe run, which no result depends on.
 */
#ifndef BRUNO_REGIONS_H_
#define BRUNO_REGIONS_H_

#include "kernels.h"
#include "partition.h"

namespace br {

/* Region sizes: 2560 slots (80 KB of LDS, two 512-thread builds per CU) or
 * 1280 (40 KB, four 256-thread builds per CU); the region_slots knob picks
 * one when a table is allocated. */
constexpr uint32_t REGION_MAX_SLOTS = 2560;
constexpr uint32_t REGION_SMALL_SLOTS = 1280;
/* the same LDS for 64-byte slots (k > 31) */
constexpr uint32_t REGION_WIDE_SLOTS = 1280;
constexpr uint32_t REGION_WIDE_SMALL_SLOTS = 640;
constexpr uint64_t REGION_BUILD_CU_SLOTS = 512; /* build workgroups resident on the device (x2 for small) */
/* record parser: workgroup size, staged records of all its buckets (128 KB),
 * records parked in LDS that found their bucket's stage full */
constexpr int REC_BS = 1024, REC_PARK = 256;
constexpr uint32_t REC_STAGE_BYTES = 128 << 10;
constexpr uint64_t REC_WG_INSTANCES = 1 << 15; /* enough instances for a parser workgroup */
/* most records between two appends: a workgroup appends every PF positions,
 * or every 16 when its reads have at most so many records in them */
template <typename R> constexpr uint32_t rec_interval() { return REC_STAGE_BYTES / sizeof(R) / 4 * 3; }
constexpr int REGION_ITEMS = 8;              /* records per thread loaded at once by the build */

/* A parser workgroup's share: reads of job `job`, part i of n of them. */
struct ParseShare {
  uint32_t job, i, n, pad;
};

struct RecArgs {
  ChunkPool pool;
  const JobLayout* jobs;
  const uint64_t* first;     /* job q holds reads [first[q], first[q + 1]) */
  const ParseShare* share;   /* per workgroup */
  void* over;                /* per workgroup over_cap records (RecOf<KT>::T) that found the park full, */
  uint32_t* over_at;         /* and their places */
  uint32_t over_cap;
  uint32_t lanes;            /* most lanes that take part in one round */
  unsigned long long* stat;  /* per job: instances, dropped reads */
};

/* Instances of each job's reads (reads with non-ACGT bases included, so an
 * upper bound).  A few workgroups per job: their totals are one atomic each
 * (with a workgroup per 256 reads the atomics took 0.63 ms for 13 M reads,
 * whose offsets are read in 0.03 ms). */
__global__ __launch_bounds__(BLOCK) void k_count_instances(ParseArgs a, const uint64_t* first, const ParseShare* share,
                                                           unsigned long long* out) {
  const ParseShare sh = share[blockIdx.x];
  const uint64_t r0 = first[sh.job], nr = first[sh.job + 1] - r0;
  const uint64_t lo = r0 + nr * sh.i / sh.n, hi = r0 + nr * (sh.i + 1) / sh.n;
  unsigned long long n = 0;
  for (uint64_t r = lo + threadIdx.x; r < hi; r += BLOCK) {
    const uint64_t off = a.starts ? a.starts[r] : a.offsets[r];
    const uint64_t L = (a.starts ? a.ends[r] : a.offsets[r + 1]) - off;
    if (L >= (uint64_t)a.K + 2) n += L - a.K + 1;
  }
  block_add(n, out + sh.job);
}

/* A k-mer instance's record: the key word (hash << 5) | biedge index, and
 * for k > 31 the k-mer's high word (with the hash it gives the low word
 * back, see kmer_unhash_lo). */
template <typename KT> __device__ __forceinline__ typename RecOf<KT>::T make_rec(uint64_t key, KT km);
template <> __device__ __forceinline__ uint64_t make_rec<uint64_t>(uint64_t key, uint64_t) { return key; }
template <> __device__ __forceinline__ ulonglong2 make_rec<u128>(uint64_t key, u128 km) {
  return make_ulonglong2(key, (uint64_t)(km >> 64));
}

/* chunk padding: a record the split drops (code 31) */
template <typename R> __device__ __forceinline__ R rec_filler();
template <> __device__ __forceinline__ uint64_t rec_filler<uint64_t>() { return REC_CODE_FILL; }
template <> __device__ __forceinline__ ulonglong2 rec_filler<ulonglong2>() { return make_ulonglong2(REC_CODE_FILL, 0); }

/* `more` consecutive chunks of the pool for a bucket at once (more than one
 * for a crowded bucket only, so out of line: inlined, these parts cost the
 * parser registers); NO_CHUNK and the overflow flag if there are none. */
__device__ __noinline__ uint32_t take_chunks(uint32_t* next, uint32_t* taken, uint32_t* owner, uint32_t n_max,
                                             uint32_t* overflow, uint32_t bucket, uint32_t more) {
  const uint32_t nid = atomicAdd(next, more);
  atomicAdd(taken, more);
  if (nid > n_max || more > n_max - nid) {
    *overflow = 1;
    return NO_CHUNK;
  }
  for (uint32_t q = 0; q < more; ++q) owner[nid + q] = bucket;
  return nid;
}

/* the parked records that are in HBM to their chunks (see flush) */
template <typename R>
__device__ __noinline__ void place_over(const R* over, const uint32_t* over_at, uint32_t n, R* recs, uint32_t clog,
                                        const uint32_t* fl_n, const uint32_t* fl_n1, const uint32_t* fl_c1,
                                        const uint32_t* fl_f1, const uint32_t* fl_c2) {
  for (uint32_t p = threadIdx.x; p < n; p += REC_BS) {
    const uint32_t b = over_at[p] & 511u, i = over_at[p] >> 9, m1 = fl_n1[b];
    if (fl_n[b] == 0) continue;
    R* d = i < m1 ? recs + ((uint64_t)fl_c1[b] << clog) + fl_f1[b] + i
                  : recs + ((uint64_t)fl_c2[b] << clog) + (i - m1);
    *d = over[p];
  }
}

/* Parse into bucketed instance records, one read per lane.  A lane rolls
 * its read's k-mer and reverse complement along the read one base at a
 * time (a shift and an or each), so an instance costs its hash and its
 * record, not a window extraction and a reverse complement.  The lanes
 * step through their reads in aligned 16-byte blocks, all lanes of the
 * workgroup at the same block index (bases before a read's start or past
 * its end are masked off).  A read with a non-ACGT base is dropped whole
 * (NFilterSequencesIterator, compact_dbg_freq_construct_clean.cpp:210-213),
 * found by a first pass over its blocks.
 *
 * Long reads: a round lasts as long as its longest read, so reads that the
 * others would wait for are left out of it and then taken one by one, each
 * by all lanes, a piece of its instances per lane; where the line lies
 * depends on the round (long_line).  A read of 1 M bases among 50,000 of 150: 266
 * ms by one lane, 78 by atomics (a wave per read), now 1.5; 3,000 reads of 5,000
 * to 15,000: 5.5, 2.3, now 1.1; 60,000 of log-normal length (median 490, up to
 * 20,000) 4.5, 2.8, now 1.9.
 *
 * Staging: the LDS stage is divided among the job's buckets; every PF
 * positions the workgroup appends each bucket's whole 128-byte lines to the
 * bucket's open chunk (the rest moves to the front of its stage), so chunks
 * are written in full lines whatever their number.  A record that finds its
 * stage full is parked, in LDS and past REC_PARK of them in HBM, with its
 * number in the bucket, which is its place in the append: the append takes a
 * crowded bucket's records all, staged and parked (reads of low complexity
 * or of one locus side by side put a whole interval's into one bucket).  The
 * count of 1 M reads of 150 bases, 2.7 ms, takes 3.6 with 2,000 poly-A reads
 * among them in one place and 10.2 with 20 times 1,000; when a record that
 * found a park of 512 full gave the count up, to HBM atomics, 13.3 and 43.  An
 * append without crowded buckets pays for it with 1 to 2% of the kernel (910 for
 * 900 us, 2.47 for 2.42 ms of 16-byte records).
 *
 * One 1,024-thread workgroup per CU with 256 buckets (512 for the largest
 * tables).  Bound by instruction issue.  The appends to 256 buckets cost
 * 5-15% over 32 and the split after it needs one pass instead of two; the
 * bases tested and coded four at a time and read four blocks at a time give
 * it back (1.6 G instances 7.4 ms with 32 buckets, 7.8 with 256, now 7.3; 184
 * M 0.84, 0.96, 0.91; 301 M of k = 63 2.48, 2.59, 2.47).  With the split the
 * count phase as a whole 35.9 -> 30.1, 4.5 -> 3.8, 13.2 -> 10.7 and 1.39 ->
 * 0.81 ms.  A batch of 16 jobs of 0.05 to 2 Mbp (243 M instances), which HBM
 * atomics counted in 18.6 ms, takes 5.9. */
constexpr int LONG_BINS = 40, LONG_LOG = 8; /* bin b: reads of 2^(LONG_LOG + b) + 1 .. 2^(LONG_LOG + b + 1) bases */
constexpr uint64_t LANE_READ_MAX = 1ULL << 30; /* a lane's positions are 32-bit numbers */

/* The length from which a round's reads are taken by all lanes: the power
 * of two 2^b >= 2^LONG_LOG with the fewest steps in all, 2^b for the reads up to
 * it and for every longer one a lane's piece and the k bases before it (~0: none). */
__device__ __noinline__ uint64_t long_line(const uint32_t* hist, uint32_t lanes, int K) {
  uint64_t line = ~0ULL, least = 0, longer = 0;
  for (int b = LONG_BINS - 1; b >= 0; --b) {
    const uint64_t n = hist[b], at = 1ULL << (LONG_LOG + b);
    if (n && least == 0) least = 2 * at;
    longer += n * (2 * at / lanes + (uint64_t)K + 48);
    if (longer && at + longer < least) {
      least = at + longer;
      line = at;
    }
  }
  return line < LANE_READ_MAX ? line : least < LANE_READ_MAX ? line : LANE_READ_MAX;
}

template <typename KT, int MAXB, int PF>
__global__ __launch_bounds__(REC_BS) void k_parse_records(ParseArgs a, RecArgs ra) {
  typedef typename RecOf<KT>::T R;
  constexpr uint32_t LINE = 128 / sizeof(R);
  constexpr uint32_t STAGE = REC_STAGE_BYTES / sizeof(R);
  __shared__ R stg[STAGE];
  __shared__ uint32_t cnt[MAXB];
  __shared__ uint32_t ch_id[MAXB], ch_fill[MAXB];     /* open chunk (NO_CHUNK: none) */
  __shared__ uint32_t fl_n1[MAXB], fl_n[MAXB], fl_c1[MAXB], fl_f1[MAXB], fl_c2[MAXB]; /* an append: see flush */
  /* Parked records are numbered through the whole launch, n_park of them so
   * far, `parked` of them before the last append.  An interval's first
   * REC_PARK are here, by their number, beside as many of the interval
   * before, which are placed meanwhile. */
  __shared__ R park[2 * REC_PARK];
  __shared__ uint32_t park_at[2 * REC_PARK]; /* number in the bucket << 9 | bucket */
  __shared__ uint32_t n_park, blocks_max;
  /* the round's reads of more than 2^LONG_LOG bases by length, those left for all
   * lanes, whether one of these has a byte that is no base */
  __shared__ uint32_t len_hist[LONG_BINS], long_bad;
  __shared__ unsigned long long long_mask[REC_BS / 64];
  /* (kept here for the rare path that uses them, not in registers) */
  __shared__ R* over;
  __shared__ uint32_t* over_at;
  __shared__ uint32_t over_cap;
  /* chunk numbers in hand, at least one per bucket before an append: pl_n0
   * from pl_b0, then up to pl_n from pl_b1; pl_used are given out */
  __shared__ uint32_t pl_b0, pl_n0, pl_b1, pl_n, pl_used;
  static_assert(16 % PF == 0, "flush points split a block evenly");
  static_assert(REC_BS * PF <= rec_interval<R>(), "an interval's records");
  static_assert(MAXB <= 512 && rec_interval<R>() + STAGE < (1u << 23), "park_at");
  const uint32_t tid = threadIdx.x;
  const ParseShare sh = ra.share[blockIdx.x];
  const JobLayout* jb = ra.jobs + sh.job;
  const uint32_t beta = jb->beta, nb_ = 1u << beta, S = STAGE >> beta, bucket0 = jb->bucket0;
  const uint32_t clog = ra.pool.clog, C = 1u << clog;
  const int K = a.K;
  kops<KT> ops(K);
  unsigned long long my_inst = 0, my_drop = 0;
  for (uint32_t b = tid; b < nb_; b += REC_BS) {
    cnt[b] = 0;
    ch_id[b] = NO_CHUNK;
    ch_fill[b] = 0;
  }
  if (tid == 0) {
    over = (R*)ra.over + (uint64_t)blockIdx.x * ra.over_cap;
    over_at = ra.over_at + (uint64_t)blockIdx.x * ra.over_cap;
    over_cap = ra.over_cap;
    n_park = pl_b0 = pl_n0 = pl_used = 0;
    pl_b1 = atomicAdd(ra.pool.next, nb_);
    pl_n = nb_;
  }
  __syncthreads();
  R* const recs = (R*)ra.pool.recs;
  uint32_t parked = 0;
  auto put = [&](uint32_t b, const R& rec) {
    const uint32_t pos = atomicAdd(&cnt[b], 1u);
    if (pos < S) {
      stg[b * S + pos] = rec;
    } else {
      const uint32_t p = atomicAdd(&n_park, 1u), i = p - parked, at = pos << 9 | b;
      if (i < REC_PARK) {
        park[p & (2 * REC_PARK - 1)] = rec;
        park_at[p & (2 * REC_PARK - 1)] = at;
      } else if (i - REC_PARK < over_cap) {
        over[i - REC_PARK] = rec;
        over_at[i - REC_PARK] = at;
      } else {
        *ra.pool.overflow = 1; /* no interval has so many */
      }
    }
  };
  /* append every bucket's whole lines, up to a line's end in its chunk (last,
   * or some of them parked: everything), to its open chunk, the rest to new
   * ones: the first fl_n1 of them to chunk fl_c1 from place fl_f1, the others
   * to the chunks from fl_c2 on, consecutive ones, the last of which is open
   * then; fl_n are staged, the rest is parked.  The number of parked records is read between the two
   * barriers, where nothing is put, so that every wave finds the same. */
  auto flush = [&](bool last) {
    if (tid < nb_) {
      const uint32_t c = cnt[tid];
      const uint32_t id = ch_id[tid], fill = ch_fill[tid], end = (fill + c) & ~(LINE - 1);
      const uint32_t m = last || c > S ? c : end > fill ? end - fill : 0u;
      const uint32_t room = id == NO_CHUNK ? 0u : C - fill;
      const uint32_t m1 = m < room ? m : room, m2 = m - m1, more = (m2 + C - 1) >> clog;
      fl_n[tid] = m < S ? m : S;
      fl_n1[tid] = m1;
      fl_c1[tid] = id;
      fl_f1[tid] = fill;
      cnt[tid] = c - m;
      ch_fill[tid] = m2 ? m2 - ((more - 1) << clog) : fill + m1;
      /* One chunk number per bucket that needs one, from those in hand (an
       * atomic in HBM here would hold up the whole workgroup at the next
       * barrier: 2 of 9 ms). */
      const uint64_t need = __ballot(more == 1);
      if (need) {
        const uint32_t lane = tid & 63;
        uint32_t u = 0;
        if (lane == 0) u = atomicAdd(&pl_used, (uint32_t)__popcll(need));
        u = (uint32_t)__builtin_amdgcn_readfirstlane((int)u) + (uint32_t)__popcll(need & ((1ULL << lane) - 1));
        if (more == 1) {
          const uint32_t nid = u < pl_n0 ? pl_b0 + u : pl_b1 + (u - pl_n0);
          atomicAdd(&ra.pool.taken[bucket0 + tid], 1u);
          if (nid < ra.pool.n_max) ra.pool.owner[nid] = bucket0 + tid;
          else *ra.pool.overflow = 1;
          fl_c2[tid] = ch_id[tid] = nid < ra.pool.n_max ? nid : ra.pool.n_max - 1;
        }
      }
      if (more > 1) {
        const uint32_t nid = take_chunks(ra.pool.next, ra.pool.taken + bucket0 + tid, ra.pool.owner, ra.pool.n_max,
                                         ra.pool.overflow, bucket0 + tid, more);
        if (nid == NO_CHUNK) { /* nothing will be counted, so nothing is written */
          fl_n[tid] = 0;
          ch_id[tid] = ra.pool.n_max - 1;
        } else {
          fl_c2[tid] = nid;
          ch_id[tid] = nid + more - 1;
        }
      }
    }
    lds_barrier();
    const uint32_t n_parked = n_park;
    /* numbers for the next append, while the other waves copy: those left
     * (fewer than nb_, so all of the later range), then nb_ more */
    if (tid == REC_BS - 1 && pl_n - pl_used < nb_) {
      const uint32_t left = pl_n - pl_used;
      pl_b0 = pl_b1 + (pl_used - pl_n0);
      pl_n0 = left;
      pl_b1 = atomicAdd(ra.pool.next, nb_);
      pl_n = left + nb_;
      pl_used = 0;
    }
    /* LINE lanes per bucket */
    const uint32_t gl = tid & (LINE - 1);
    for (uint32_t b = tid / LINE; b < nb_; b += REC_BS / LINE) {
      const uint32_t m = fl_n[b];
      if (m == 0) continue;
      const uint32_t m1 = fl_n1[b];
      R* d1 = recs + ((uint64_t)fl_c1[b] << clog) + fl_f1[b];
      R* d2 = recs + ((uint64_t)fl_c2[b] << clog);
      for (uint32_t i = gl; i < m; i += LINE) {
        R* d = i < m1 ? d1 + i : d2 + (i - m1);
        *d = stg[b * S + i];
      }
      /* fewer than LINE records are left; the lanes read before they write */
      if (gl < cnt[b]) stg[b * S + gl] = stg[b * S + m + gl];
    }
    const uint32_t p0 = parked;
    parked = (uint32_t)__builtin_amdgcn_readfirstlane((int)n_parked);
    const uint32_t np = parked - p0;
    if (np > REC_PARK) {
      __syncthreads(); /* the records in HBM are there */
      place_over<R>(over, over_at, np - REC_PARK < over_cap ? np - REC_PARK : over_cap, recs, clog, fl_n, fl_n1, fl_c1,
                    fl_f1, fl_c2);
    }
    /* The parked records in LDS: behind the barrier, since their reads one
     * after the other would hold up the whole workgroup; fl_* stay as they
     * are until all waves have come to the next append.  (More than the LDS
     * holds: the next interval's may take the same places.) */
    if (np <= REC_PARK) lds_barrier();
    if (np && tid < (np < REC_PARK ? np : (uint32_t)REC_PARK)) {
      const uint32_t q = (p0 + tid) & (2 * REC_PARK - 1), b = park_at[q] & 511u, i = park_at[q] >> 9, m1 = fl_n1[b];
      if (fl_n[b] != 0) {
        R* d = i < m1 ? recs + ((uint64_t)fl_c1[b] << clog) + fl_f1[b] + i
                      : recs + ((uint64_t)fl_c2[b] << clog) + (i - m1);
        *d = park[q];
      }
    }
    if (np > REC_PARK) lds_barrier();
  };
  const int sh2 = 2 * (K - 1);
  const KT kmask = ops.mask;
  /* the share's reads, in as many rounds of up to REC_BS lanes as it takes,
   * evenly filled */
  const uint64_t r_job = ra.first[sh.job], n_job = ra.first[sh.job + 1] - r_job;
  const uint64_t lo_r = r_job + n_job * sh.i / sh.n, hi_r = r_job + n_job * (sh.i + 1) / sh.n;
  const uint64_t rounds = (hi_r - lo_r + REC_BS - 1) / REC_BS;
  for (uint64_t round = 0; round < rounds; ++round) {
    const uint64_t ra0 = lo_r + (hi_r - lo_r) * round / rounds, ra1 = lo_r + (hi_r - lo_r) * (round + 1) / rounds;
    const uint64_t r = ra0 + tid;
    uint64_t lo = 0, L = 0;
    if (r < ra1) {
      lo = a.starts ? a.starts[r] : a.offsets[r];
      L = (a.starts ? a.ends[r] : a.offsets[r + 1]) - lo;
    }
    /* (every thread is past the last round's use of these) */
    __syncthreads();
    if (tid < LONG_BINS) len_hist[tid] = 0;
    if (tid < REC_BS / 64) long_mask[tid] = 0;
    if (tid == 0) blocks_max = 0;
    __syncthreads();
    if (L > (1u << LONG_LOG)) {
      const int b = 63 - __clzll(L - 1) - LONG_LOG;
      atomicAdd(&len_hist[b < LONG_BINS ? b : LONG_BINS - 1], 1u);
      blocks_max = 1;
    }
    __syncthreads();
    uint32_t long_w = REC_BS / 64; /* words of long_mask gone through */
    unsigned long long long_m = 0;
    if (blocks_max) {
      const bool left = L > long_line(len_hist, ra.lanes, K);
      const uint64_t m = __ballot(left);
      if ((tid & 63) == 0) long_mask[tid >> 6] = m;
      if (left) L = 0;
      long_w = 0;
    }
    /* the instances at j_lo .. j_hi of this lane's bases [lo, lo + L) */
    int j_lo = K, j_hi = (int)L;
    uint32_t lanes = (uint32_t)(ra1 - ra0);
    bool piece = false; /* of a read that all lanes share */
    for (;;) {
      const LaneRead rd(a.bases + lo, L);
      const int mis = rd.mis;
      const bool bad = rd.bad(L);
      __syncthreads();
      if (tid == 0) blocks_max = long_bad = 0;
      __syncthreads();
      /* reads shorter than the parser window k + 2 give nothing
       * (debruijn_biedge_loader.hpp:464-465) */
      int Lp = bad || L < (uint64_t)K + 1 + !piece ? 0 : (int)L;
      if (!piece && bad) ++my_drop;
      if (piece && bad) long_bad = 1;
      if (Lp) atomicMax(&blocks_max, (uint32_t)(mis + Lp + 16) / 16); /* through position Lp */
      __syncthreads();
      uint32_t nbw = blocks_max;
      if (piece && long_bad) {
        if (tid == 0) ++my_drop;
        nbw = 0;
      }
      if (Lp == 0) j_hi = -1;
      /* fw: the last k bases read, rv its reverse complement; gone: the base
       * that left fw at the previous step.  At position j >= k the instance
       * starting at j - k is complete: its out base is base j (none at
       * j == L) and its in base the one that left at step j - 1 (none for
       * the first instance). */
      KT fw = 0, rv = 0;
      uint32_t gone = 0;
      /* a round of few reads fills its stages more slowly: an append at every
       * PF-th position, or once a block when a bucket's share of the block's
       * records leaves a quarter of its stage to chance and what stays behind */
      const bool often = lanes * 16 > rec_interval<R>() - nb_ * (LINE / 2);
      uint4 v[4] = {};
      for (uint32_t t = 0; t < nbw; ++t) {
        if (t % 4 == 0) rd.four(t, v);
        const uint4 cur = v[0];
        v[0] = v[1];
        v[1] = v[2];
        v[2] = v[3];
        const uint32_t cw[4] = {codes4(cur.x), codes4(cur.y), codes4(cur.z), codes4(cur.w)};
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const int j = (int)(16 * t) + q - mis;
          if (j >= 0 && j <= j_hi) {
            const uint32_t c = (cw[q >> 2] >> (8 * (q & 3))) & 3u;
            const bool in_read = j < Lp;
            if (j >= j_lo) {
              const bool flip = !(fw < rv);
              const KT km = flip ? rv : fw;
              const uint32_t has_in = j > K, has_out = in_read;
              const uint32_t il = !has_in ? 0u : flip ? 0u : 1u + gone;
              const uint32_t ir = !has_out ? 0u : flip ? 0u : 1u + c;
              /* biedge_rc: the in side becomes the complement of the out
               * base and the other way round */
              const uint32_t il2 = flip && has_out ? 4u - c : il;
              const uint32_t ir2 = flip && has_in ? 4u - gone : ir;
              const uint64_t h = kmer_hash(km);
              const uint64_t key = (h << REC_BUCKET_BITS) | (il2 * 5u + ir2);
              put((uint32_t)(h >> (64 - beta)), make_rec<KT>(key, km));
              ++my_inst;
            }
            if (in_read) {
              gone = (uint32_t)(fw >> sh2) & 3u;
              fw = ((fw << 2) | (KT)c) & kmask;
              rv = (rv >> 2) | ((KT)(3u - c) << sh2);
            }
          }
          if (q % PF == PF - 1 && (often || q == 15)) {
            lds_barrier();
            flush(false);
          }
        }
      }
      /* the next read left for all lanes */
      while (long_m == 0 && long_w < REC_BS / 64) long_m = long_mask[long_w++];
      if (long_m == 0) break;
      const uint64_t rl = ra0 + 64 * (long_w - 1) + __builtin_ctzll(long_m);
      long_m &= long_m - 1;
      const uint64_t l0 = a.starts ? a.starts[rl] : a.offsets[rl], ll = (a.starts ? a.ends[rl] : a.offsets[rl + 1]) - l0;
      /* a piece's instances begin at bases [i0, i1) of the read; its own bases
       * are those and the one on either side */
      piece = true;
      lanes = ra.lanes;
      const uint64_t n = ll - K + 1, per = (n + lanes - 1) / lanes;
      const uint64_t i0 = tid < lanes ? tid * per : n, i1 = i0 + per < n ? i0 + per : n;
      const uint64_t from = i0 ? i0 - 1 : 0, to = i1 + K < ll ? i1 + K : ll;
      lo = l0 + from;
      L = i0 < n ? to - from : 0;
      j_lo = K + (i0 ? 1 : 0);
      j_hi = (int)(i1 == n ? L : L - 1);
    }
  }
  lds_barrier(); /* the last append's parked records are placed */
  flush(true);
  for (uint32_t u = pl_used + tid; u < pl_n; u += REC_BS) {
    const uint32_t nid = u < pl_n0 ? pl_b0 + u : pl_b1 + (u - pl_n0);
    if (nid < ra.pool.n_max) ra.pool.owner[nid] = NO_CHUNK;
  }
  /* pad the open chunks */
  for (uint32_t b = tid / 64; b < nb_; b += REC_BS / 64) {
    if (ch_id[b] == NO_CHUNK) continue;
    R* d = recs + ((uint64_t)ch_id[b] << clog);
    for (uint32_t i = ch_fill[b] + (tid & 63); i < C; i += 64) d[i] = rec_filler<R>();
  }
  const unsigned long long si = wave_sum(my_inst), sd = wave_sum(my_drop);
  if ((tid & 63) == 0) {
    if (si) atomicAdd(&ra.stat[2 * sh.job], si);
    if (sd) atomicAdd(&ra.stat[2 * sh.job + 1], sd);
  }
}

struct RegionArgs {
  void* table;               /* Slot<KT> */
  const JobLayout* jobs;      /* their table layouts; regions are numbered through all of them */
  uint32_t n_jobs;
  uint32_t q0, q1;           /* this launch: regions [q0, q1) */
  const void* recs;          /* pieces of PIECE records (RecOf<KT>::T) */
  const uint32_t* pieces;    /* region q holds region_count[q] records, in the pieces
                                pieces[region_start[q] ...] */
  const uint32_t* region_start;
  const uint32_t* region_count;
  const uint32_t* overflow;  /* set: the records are not complete, nothing is built */
  int valid;                 /* the table holds earlier counts (else start from EMPTY) */
  Spill* spill;
  uint64_t spcap;
  /* side-table entries are queued, not added inline: wave w of the grid
   * appends (slot << 5 | biedge index) to spq[w * spq_cap ...] and leaves
   * its count in spq_n[w]; k_spill_flush adds them after the build (an
   * inline add is a chain of dependent HBM atomics that the whole
   * workgroup waits for at the next barrier) */
  uint64_t* spq;
  uint32_t* spq_n;
  uint32_t spq_cap;
  Counters* ctr;
  /* filter pre-pass (optional): from word q * stride, region q's candidate
   * bits (occupied, no spilled entries, k-mer count >= t1lo when
   * thresholding) and of spilled-slot bits, bit i of word w = slot 64 w + i */
  uint64_t* cbits;
  uint64_t* sbits;
  uint64_t stride;
  int thresholding;
  uint64_t t1lo;
  /* the filter fused into the build (fuse != 0, with the bits): every
   * candidate slot gets local_insert_by_freqencies and its branch / chain
   * class in LDS before the write-back, and its node record; the candidate
   * bits then keep only what a wave could not place (a full node list).
   * List positions come in chunks of FUSE_CHUNK per wave; wave w leaves
   * its open chunks' unused positions marked LIST_HOLE and described in
   * holes[2 w + list] = start << 7 | count. */
  int fuse; /* the kernel's FUSE parameter */
  int K;
  Thresh th;
  NodeLists nl;
  uint64_t* holes;
};

constexpr uint32_t FUSE_CHUNK = 64;
constexpr uint64_t LIST_HOLE = ~0ULL;

__device__ __forceinline__ uint64_t lds_load(const uint64_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_store(uint64_t* p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

/* A region in LDS, one row per slot word (row 0 the key / meta word, then
 * the two-word key's words, then the sub-entries): a wave's lanes touch
 * random slots, and with 32- or 64-byte slots side by side every key word
 * would sit in one of a few banks; in rows, consecutive slots' words are
 * consecutive and random slots spread over all banks.  Set-up and
 * write-back move the region's bytes in table order, 16 per lane, so every
 * load or store instruction covers whole cache lines (lane i takes piece
 * i % P of slot i / P, P = 16-byte pieces per slot). */
template <typename KT, uint32_t SLOTS>
struct LdsRegion {
  static constexpr int W = sizeof(Slot<KT>) / 8;
  static constexpr int P = W / 2;
  static constexpr int SUB0 = sizeof(KT) == 8 ? 1 : 3; /* first sub-entry row */
  uint64_t w[W][SLOTS];
  __device__ __forceinline__ uint64_t* flag(uint32_t s) { return &w[0][s]; }
  __device__ __forceinline__ uint64_t* sub(int j, uint32_t s) { return &w[SUB0 + j][s]; }
  /* slots [0, span) from / to their table copy t, BS threads */
  template <int BS>
  __device__ __forceinline__ void load(uint32_t span, const Slot<KT>* t) {
    const ulonglong2* v = (const ulonglong2*)t;
    for (uint32_t i = threadIdx.x; i < span * P; i += BS) {
      const ulonglong2 x = v[i];
      const uint32_t s = i / P, q = i % P;
      w[2 * q][s] = x.x;
      w[2 * q + 1][s] = x.y;
    }
  }
  template <int BS>
  __device__ __forceinline__ void clear(uint32_t span) {
    for (uint32_t s = threadIdx.x; s < span; s += BS)
#pragma unroll
      for (int q = 0; q < W; ++q) w[q][s] = EMPTY64;
  }
  template <int BS>
  __device__ __forceinline__ void store(uint32_t span, Slot<KT>* t) const {
    typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
    u64x2* v = (u64x2*)t;
    for (uint32_t i = threadIdx.x; i < span * P; i += BS) {
      const uint32_t s = i / P, q = i % P;
      u64x2 x;
      x.x = w[2 * q][s];
      x.y = w[2 * q + 1][s];
      /* streaming: the region is not read again during the count */
      __builtin_nontemporal_store(x, v + i);
    }
  }
};

/* An EMPTY word by its high half: no key, meta or sub-entry word of a
 * region being counted has an all-ones high half (F_PRESENT is never set
 * there, a biedge code is at most 25), so one 32-bit compare decides. */
__device__ __forceinline__ bool lds_empty(uint64_t v) { return (uint32_t)(v >> 32) == ~0u; }

/* v, with what the compiler knows of it forgotten: the word a loop ended
 * with is tested again after the loop (two instructions), where the
 * compiler would carry each test's result through the loop as a lane mask
 * (three scalar instructions a pass, more than the pass itself). */
__device__ __forceinline__ uint64_t opaque(uint64_t v) {
  uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
  asm("" : "+v"(lo), "+v"(hi));
  return ((uint64_t)hi << 32) | lo;
}

/* Find or claim the k-mer of a record in the LDS region L of span slots
 * from home slot s; returns the slot, or ~0u when the region is full.
 * fresh: this call inserted the key.  During the adds a slot's first word
 * holds the record's 59 hash bits (with the region they determine a one-word
 * k-mer), so a record needs no unhashing; lds_finish puts the k-mers in.
 * (One exit and no state but the word read: a wave runs the loop to its
 * longest probe sequence, so what counts is the instructions per probe,
 * vector and scalar.) */
template <uint32_t SLOTS>
__device__ __forceinline__ uint32_t lds_claim(LdsRegion<uint64_t, SLOTS>& L, uint32_t span, const uint32_t home,
                                              const uint64_t& rec, bool& fresh) {
  const uint64_t v = rec >> REC_BUCKET_BITS;
  uint32_t s = home, at;
  uint64_t k0;
  bool miss;
  do {
    at = s;
    k0 = lds_load(L.flag(s));
    if (lds_empty(k0)) k0 = atomicCAS((unsigned long long*)L.flag(s), EMPTY64, (unsigned long long)v);
    miss = !lds_empty(k0) && (k0 & ~F_SPILL) != v;
    s = (s + 1 == span) ? 0 : s + 1;
  } while (miss && s != home);
  k0 = opaque(k0);
  fresh = lds_empty(k0);
  return fresh || (k0 & ~F_SPILL) == v ? at : ~0u;
}
/* Two-word k-mers: the hash word is claimed, then the high word stored
 * (all ones until then, which no k-mer's high word is); a slot whose hash
 * word agrees is read on, waiting (bounded) for its high word.  The claiming
 * lanes of a wave store before any lane of it waits.  A probe that misses
 * costs one LDS read; with the k-mer's own words as the key it was three. */
template <uint32_t SLOTS>
__device__ __forceinline__ uint32_t lds_claim(LdsRegion<u128, SLOTS>& L, uint32_t span, const uint32_t home,
                                              const ulonglong2& rec, bool& fresh) {
  const uint64_t v = rec.x >> REC_BUCKET_BITS, hi = rec.y;
  uint32_t s = home, at;
  uint64_t k0;
  bool miss, same;
  do {
    at = s;
    k0 = lds_load(L.flag(s));
    if (lds_empty(k0)) {
      k0 = atomicCAS((unsigned long long*)L.flag(s), EMPTY64, (unsigned long long)v);
      if (lds_empty(k0)) lds_store(&L.w[2][s], hi);
    }
    same = (k0 & ~F_SPILL) == v;
    if (same) {
      uint64_t h2 = lds_load(&L.w[2][s]);
      for (uint32_t spin = 0; h2 == EMPTY64 && spin < MAX_SPIN; ++spin) h2 = lds_load(&L.w[2][s]);
      same = h2 == hi;
    }
    miss = !(lds_empty(k0) || same);
    s = (s + 1 == span) ? 0 : s + 1;
  } while (miss && s != home);
  k0 = opaque(k0);
  fresh = lds_empty(k0);
  return fresh || same ? at : ~0u;
}

/* Between the adds' slots and the table's: the hash word of slot i made
 * from its k-mer (after a load) and back (before a write-back; h_top: the
 * hash's top bits, the region's bucket). */
template <uint32_t SLOTS>
__device__ __forceinline__ void lds_begin(LdsRegion<uint64_t, SLOTS>& L, uint32_t i) {
  const uint64_t w = L.w[0][i];
  if (!lds_empty(w)) L.w[0][i] = (w & F_SPILL) | (kmer_hash(w & KEY_BITS) << REC_BUCKET_BITS >> REC_BUCKET_BITS);
}
template <uint32_t SLOTS>
__device__ __forceinline__ void lds_begin(LdsRegion<u128, SLOTS>& L, uint32_t i) {
  const uint64_t w = L.w[0][i];
  if (w != EMPTY64)
    L.w[0][i] = (w & F_SPILL) |
                (kmer_hash(((u128)L.w[2][i] << 64) | L.w[1][i]) << REC_BUCKET_BITS >> REC_BUCKET_BITS);
}
template <uint32_t SLOTS>
__device__ __forceinline__ void lds_finish(LdsRegion<uint64_t, SLOTS>& L, uint32_t i, uint64_t h_top) {
  const uint64_t w = L.w[0][i];
  if (!lds_empty(w)) L.w[0][i] = (w & F_SPILL) | kmer_unhash(h_top | (w & ~F_SPILL));
}
template <uint32_t SLOTS>
__device__ __forceinline__ void lds_finish(LdsRegion<u128, SLOTS>& L, uint32_t i, uint64_t h_top) {
  const uint64_t w = L.w[0][i];
  if (!lds_empty(w)) {
    L.w[1][i] = (uint64_t)kmer_unhash(h_top | (w & ~F_SPILL), L.w[2][i]);
    L.w[0][i] = w & F_SPILL;
  }
}

/* add_k2 on LDS slot s (code = biedge index + 1).  Returns 1 for a new k2
 * entry in the slot, 0 for a count added, and LDS_SPILL when the entry
 * belongs in the side table (the slot is marked as having spilled entries;
 * the caller queues the entry).  A loop over the sub-entry rows: almost
 * every record ends at the first or second. */
constexpr int LDS_SPILL = 2;
template <typename KT, uint32_t SLOTS>
__device__ __forceinline__ int lds_add_k2(LdsRegion<KT, SLOTS>& L, uint32_t s, uint32_t code) {
  constexpr int N = Slot<KT>::NSUB;
  uint64_t* q = L.sub(0, s);
  uint64_t* const end = q + (size_t)N * SLOTS;
  const uint64_t first = ((uint64_t)code << 48) | 1;
  uint64_t* at;
  uint64_t v;
  bool more;
  do {
    at = q;
    v = lds_load(q);
    if (lds_empty(v)) v = atomicCAS((unsigned long long*)q, EMPTY64, (unsigned long long)first);
    more = !lds_empty(v) && (uint32_t)(v >> 48) != code;
    q += SLOTS;
  } while (more && q != end);
  v = opaque(v);
  if ((uint32_t)(v >> 48) == code) atomicAdd((unsigned long long*)at, 1ULL);
  else if (!lds_empty(v)) {
    uint64_t* fw = L.flag(s);
    if (!(lds_load(fw) & F_SPILL)) atomicOr((unsigned long long*)fw, (unsigned long long)F_SPILL);
    return LDS_SPILL;
  }
  return lds_empty(v) ? 1 : 0;
}

/* an empty use of a register: the compiler waits for its load here */
__device__ __forceinline__ void consume(uint64_t v) { asm volatile("" ::"v"(v)); }
__device__ __forceinline__ void consume(const ulonglong2& v) {
  asm volatile("" ::"v"(v.x));
  asm volatile("" ::"v"(v.y));
}

/* Add one record to its region in LDS.  Returns the LDS slot of a
 * side-table entry to queue (of the record's biedge index), or NO_SPILL. */
constexpr uint32_t NO_SPILL = ~0u;
template <typename KT, uint32_t SLOTS, typename R>
__device__ __forceinline__ uint32_t region_add(const RegionArgs& g, LdsRegion<KT, SLOTS>& L, uint32_t span,
                                               uint32_t rbits, const R& rec, uint32_t& my_new, uint32_t& my_k2) {
  const uint64_t key = rec_key(rec);
  bool fresh;
  /* the record's hash bits below the region's, as region_home takes them */
  const uint32_t home = region_home(key, rbits - REC_BUCKET_BITS, span);
  const uint32_t s = lds_claim(L, span, home, rec, fresh);
  if (s == ~0u) {
    atomicOr(&g.ctr->err, ERR_TABLE_FULL);
    return NO_SPILL;
  }
  my_new += fresh ? 1 : 0;
  const int r = lds_add_k2<KT, SLOTS>(L, s, (uint32_t)(key & 31) + 1);
  my_k2 += r & 1;
  return r == LDS_SPILL ? s : NO_SPILL;
}

/* a side-table entry added at once: the wave's queue is full (kept out of
 * line: inlined at every record slot it was most of the build's code) */
__device__ __noinline__ int spill_add_now(Spill* sp, uint64_t spcap, uint64_t e, uint32_t* err) {
  return spill_add(sp, spcap, e >> 5, (e & 31) + 1, err);
}

/* Queue side-table entries (table slot << 5 | biedge index) from converged
 * code: one ballot per record slot of the tile; qn (this wave's queue fill)
 * stays wave-uniform.  A full queue adds the entry at once.  s: LDS slot or
 * NO_SPILL; base: the region's first table slot. */
__device__ __forceinline__ void spill_queue(const RegionArgs& g, uint64_t* q, uint32_t& qn, uint32_t s, uint64_t base,
                                            uint32_t code, uint32_t& my_k2) {
  const uint64_t m = __ballot(s != NO_SPILL);
  if (!m) return;
  const uint32_t at = qn + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
  if (s != NO_SPILL) {
    const uint64_t e = ((base + s) << 5) | code;
    if (at < g.spq_cap) q[at] = e;
    else my_k2 += spill_add_now(g.spill, g.spcap, e, &g.ctr->err);
  }
  qn += (uint32_t)__popcll(m);
}

/* ------------------------------------------------------------------ */
/* the filter fused into the build                                      */
/* ------------------------------------------------------------------ */
template <uint32_t SLOTS>
__device__ __forceinline__ uint64_t lds_kmer(LdsRegion<uint64_t, SLOTS>& L, uint32_t s) {
  return *L.flag(s) & KEY_BITS;
}
template <uint32_t SLOTS>
__device__ __forceinline__ u128 lds_kmer(LdsRegion<u128, SLOTS>& L, uint32_t s) {
  return ((u128)L.w[2][s] << 64) | L.w[1][s];
}

/* The filter pre-pass's choice for LDS slot i: a candidate (occupied, no
 * side-table entries, not yet a node, k-mer count >= t1lo when
 * thresholding), or *spilled for a slot with side-table entries. */
template <typename KT, uint32_t SLOTS>
__device__ __forceinline__ bool lds_candidate(const RegionArgs& g, LdsRegion<KT, SLOTS>& L, uint32_t i,
                                              bool& spilled) {
  const uint64_t fw = *L.flag(i);
  spilled = fw != EMPTY64 && (fw & F_SPILL);
  if (fw == EMPTY64 || (fw & (F_SPILL | F_PRESENT))) return false;
  if (!g.thresholding) return true;
  uint64_t tot = 0;
#pragma unroll
  for (int j = 0; j < Slot<KT>::NSUB; ++j) {
    const uint64_t v = *L.sub(j, i);
    tot += v != EMPTY64 ? (v & 0xFFFFFFFFFFFFULL) : 0;
  }
  return tot >= g.t1lo;
}

/* A wave's open chunk of a node list: positions [base, base + size), of
 * which the first `used` are given out.  Wave-uniform. */
struct ListChunk {
  uint64_t base;
  uint32_t used;
};

/* Consecutive list positions for the lanes with take set, called by the
 * whole wave: from the open chunk, then from a new chunk of `size` >= 64
 * (one atomic) when it runs out. */
__device__ __forceinline__ uint64_t chunk_take(ListChunk& ch, bool take, unsigned long long* counter,
                                               uint32_t size = FUSE_CHUNK) {
  const uint64_t m = __ballot(take);
  const uint32_t n = (uint32_t)__popcll(m);
  const uint32_t lane = __lane_id();
  const uint32_t rank = (uint32_t)__popcll(m & ((1ULL << lane) - 1));
  const uint32_t room = size - ch.used;
  uint64_t pos = ch.base + ch.used + rank;
  if (n > room) {
    uint64_t nb = 0;
    if (lane == 0) nb = atomicAdd(counter, (unsigned long long)size);
    nb = readlane64(nb, 0);
    if (rank >= room) pos = nb + (rank - room);
    ch.base = nb;
    ch.used = n - room;
  } else {
    ch.used += n;
  }
  return pos;
}

/* The fused filter for queued slots of the region whose table slots start
 * at base (lane l holds LDS slot qs when active): the slot's k2 entries
 * from LDS, local_insert_by_freqencies (debruijn_graph_map.hpp:1351-1609;
 * the k+1-mer edge filter, or none, as the job asks), IsBranchPoint /
 * IsChainNode (debruijn_graph_filters.hpp:142-220), then the node record
 * with its list position and F_PRESENT written into the LDS slot and the
 * slot appended to its list.  Called by the whole wave; true (for the
 * wave) when a node found its list full: that slot stays a candidate for
 * the filter pass. */
template <typename KT, uint32_t SLOTS>
__device__ __forceinline__ bool fuse_nodes(const RegionArgs& g, LdsRegion<KT, SLOTS>& L, uint64_t base, uint32_t qs,
                                           bool active, ListChunk (&ch)[2]) {
  constexpr int N = Slot<KT>::NSUB;
  const kops<KT> ops(g.K);
  bool kept = false;
  NodeRec rec;
  rec.cls = 0;
  if (active) {
    K2L<N> Lk;
    Lk.n = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const uint64_t v = *L.sub(j, qs);
      const bool ok = v != EMPTY64;
      Lk.e[j] = ok ? biedge_sides((uint32_t)(v >> 48) - 1) : 0;
      Lk.c[j] = ok ? (uint32_t)(v & 0xFFFFFFFFFFFFULL) : 0;
      Lk.n += ok;
    }
    const KT k = lds_kmer(L, qs);
    const KmerFacts f = kmer_facts(ops, k);
    uint16_t c[9];
    if (g.thresholding == 2) {
      kept = edge_counts<KT, N>(ops, k, Lk, g.th, c);
    } else if (g.thresholding) {
      kept = p2_counts_slot<KT, N>(ops, f, Lk, g.th, c);
    } else {
      p1_counts(Lk, c);
      kept = true;
    }
    if (kept) rec = make_node_facts<KT>(ops, f, c);
  }
  const bool chn = kept && rec.cls == CLS_CHAIN, brn = kept && rec.cls == CLS_BRANCH;
  const uint64_t pc = chunk_take(ch[0], chn, &g.ctr->n_chain);
  const uint64_t pb = chunk_take(ch[1], brn, &g.ctr->n_branch);
  bool full = false;
  if (kept) {
    const uint64_t pos = chn ? pc : pb;
    if (pos < g.nl.cap && pos <= 0x7FFFFFFFULL) {
      rec.idx = (uint32_t)pos;
      uint64_t w[3];
      __builtin_memcpy(w, &rec, sizeof(rec));
#pragma unroll
      for (int j = 0; j < 3; ++j) *L.sub(j, qs) = w[j];
      *L.flag(qs) |= F_PRESENT;
      (chn ? g.nl.chain_slot : g.nl.branch_slot)[pos] = base + qs;
    } else {
      full = true;
    }
  }
  return __ballot(full) != 0;
}

/* Side-table entries the region builds queued, a wave per queue (a queue
 * holds tens of entries), in four workgroups per CU at most: their one sum
 * each goes to the same counter, and with a workgroup for each of 8,192
 * queues those atomics were the time (84 us on 21 M records, now
 * 20, on 184 M 113, now 46; the entries themselves are probes and adds in HBM). */
__global__ __launch_bounds__(BLOCK) void k_spill_flush(const uint64_t* spq, const uint32_t* spq_n, uint32_t n_queues,
                                                        uint32_t spq_cap, const uint32_t* overflow, Spill* spill,
                                                        uint64_t spcap, Counters* ctr) {
  if (*overflow) return; /* nothing was built */
  const uint32_t lane = threadIdx.x & 63, step = gridDim.x * (BLOCK / 64);
  unsigned long long mine = 0;
  for (uint32_t w = blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6); w < n_queues; w += step) {
    const uint32_t n = min(spq_n[w], spq_cap);
    const uint64_t* q = spq + (uint64_t)w * spq_cap;
    for (uint32_t i = lane; i < n; i += 64) {
      const uint64_t e = q[i];
      mine += spill_add(spill, spcap, e >> 5, (e & 31) + 1, &ctr->err);
    }
  }
  block_add(mine, &ctr->n_k2);
}

/* Build regions [q0, q1), workgroup i taking every gridDim-th of them (the
 * jobs of a batch differ in records per region, so neighbours in one
 * workgroup would leave some with the work of several).
 * Per region: set up the slots in LDS (EMPTY, or the table's slots when an
 * earlier count wrote them; a region without records is then left as it
 * is), add the region's records (REGION_ITEMS per thread at a time), write
 * the filter pre-pass bits when asked, and write the region back (16-byte
 * stores, a slot per lane).  The next region's first records are loaded
 * before this region's records are added, so their latency hides behind
 * the LDS work; barriers order LDS only, so one region's write-back
 * overlaps the next region's set-up.  Nothing between two write-backs may
 * wait for a load issued after the first one (loads and stores complete in
 * order): piece numbers are read two regions ahead and region bounds three,
 * and a job's layout only when a workgroup comes to it (184 M records: 1.70
 * -> 1.52 ms; 301 M of 16 bytes: 5.13 -> 4.40).
 *
 * Bound by the instructions per record (vector and scalar; LDS is busy a
 * third of the time), so the adds carry no lane masks through their loops,
 * compare one 32-bit half for EMPTY, take the home slot from one 32-bit
 * product and leave the k-mer to the write-back (a record needs no
 * unhashing; one slot in two holds a k-mer).  184 M records into 113 M slots:
 * 1.86 -> 1.56 ms; 301 M 16-byte records (k = 63): 5.5 -> 4.55 ms.  Twice the
 * waves (1,024 threads a workgroup, half the registers) were slower, 2.34 and
 * 6.2 ms. */
template <typename KT, uint32_t SLOTS, int BS, bool FUSE>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(4))) void k_region_build(RegionArgs g) {
  typedef typename RecOf<KT>::T R;
  /* records per thread per tile: a 64-byte-slot region holds half the
   * slots, so half as many (and the registers stay without spills) */
  constexpr int REGION_ITEMS = sizeof(R) == 8 ? br::REGION_ITEMS : br::REGION_ITEMS / 2;
  __shared__ LdsRegion<KT, SLOTS> L;
  if (*g.overflow) return;
  const uint32_t qa = g.q0 + blockIdx.x, step = gridDim.x;
  const R* recs = (const R*)g.recs;
  uint32_t my_new = 0, my_k2 = 0; /* a lane's records of one launch: far below 2^32 */
  constexpr uint32_t TILE = REGION_ITEMS * BS;
  /* first piece and record count of the workgroup's regions, 64 at a
   * time: lane l of every wave holds its region number rs_n + l and the
   * next 64 are loaded ahead, so a region's bounds are lane reads, not
   * dependent loads */
  const int lane = threadIdx.x & 63;
  uint32_t rs_n = 0;
  auto rs_load = [&](uint32_t n, uint32_t& st, uint32_t& c) {
    const uint64_t q = qa + (uint64_t)(n + lane) * step;
    st = q < g.q1 ? g.region_start[q] : 0;
    c = q < g.q1 ? g.region_count[q] : 0;
  };
  uint32_t rs, rs_nx, rc, rc_nx;
  rs_load(0, rs, rc);
  rs_load(64, rs_nx, rc_nx);
  auto bounds = [&](uint32_t n, uint32_t& start, uint32_t& count) { /* n never decreases */
    while (n >= rs_n + 64) {
      rs = rs_nx;
      rc = rc_nx;
      rs_n += 64;
      rs_load(rs_n + 64, rs_nx, rc_nx);
    }
    start = (uint32_t)__builtin_amdgcn_readlane((int)rs, (int)(n - rs_n));
    count = (uint32_t)__builtin_amdgcn_readlane((int)rc, (int)(n - rs_n));
  };
  /* this wave's side-table queue */
  const uint64_t wave_id = (uint64_t)blockIdx.x * (BS / 64) + (threadIdx.x >> 6);
  uint64_t* spq = g.spq + wave_id * g.spq_cap;
  uint32_t qn = 0;
  /* this wave's open chunks of the chain and branch lists (fused filter) */
  ListChunk ch[2] = {{0, FUSE_CHUNK}, {0, FUSE_CHUNK}};
  /* A region's piece numbers, 64 of this wave's at a time: record slot k
   * of tile t is the region's piece (t * REGION_ITEMS + k) * NW + wave, so
   * lane l loads the number of piece l * NW + wave, for 64 / REGION_ITEMS
   * tiles. */
  constexpr uint32_t NW = BS / 64, TILES = 64 / REGION_ITEMS;
  auto numbers = [&](uint32_t start, uint32_t count, uint32_t t) -> uint32_t {
    const uint32_t i = (t * REGION_ITEMS + lane) * NW + (threadIdx.x >> 6);
    /* (no branch: a value of two paths would be copied, and waited for) */
    return g.pieces[i << PIECE_LOG < count ? start + i : 0];
  };
  auto load = [&](uint32_t count, uint32_t nums, uint32_t t, R (&r)[REGION_ITEMS]) {
#pragma unroll
    for (int k = 0; k < REGION_ITEMS; ++k) {
      const uint32_t p = (uint32_t)__builtin_amdgcn_readlane((int)nums, (int)((t % TILES) * REGION_ITEMS + k));
      r[k] = rec_zero<R>();
      if (t * TILE + k * BS + threadIdx.x < count) r[k] = recs[((uint64_t)p << PIECE_LOG) + lane];
    }
  };
  /* Read ahead of the region being built: the next one's first tile, the
   * piece numbers of the one after, and where the pieces of the third are (a
   * region without records in a written table stays as it is and is passed
   * over; past the last one the counts are 0). */
  struct Ahead {
    uint32_t q, start, count;
  };
  Ahead nx, af, th; /* next, after it, third */
  uint32_t th_n = 0; /* number of the third of the workgroup's regions */
  R rn[REGION_ITEMS];
  uint32_t af_nums;
  auto find = [&]() {
    for (;; ++th_n) {
      th.q = qa + th_n * step;
      th.start = th.count = 0;
      if (th.q >= g.q1) return;
      bounds(th_n, th.start, th.count);
      if (!(g.valid && th.count == 0)) break;
    }
    ++th_n;
  };
  auto ahead = [&]() {
    nx = af;
    load(nx.count, af_nums, 0, rn);
    af = th;
    af_nums = numbers(af.start, af.count, 0);
  };
  /* the current region's job (read when a workgroup comes to it: a load at
   * each region would wait for the write-back before it) */
  uint32_t ji = count_job_of(g.n_jobs, qa, [&](uint32_t j) { return g.jobs[j].region0; });
  uint32_t ji_end, span, rbits, region0;
  uint64_t slot0;
  auto uniform = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
  auto job = [&]() {
    ji_end = ji + 1 < g.n_jobs ? uniform(g.jobs[ji + 1].region0) : ~0u;
    span = uniform((uint32_t)g.jobs[ji].span);
    rbits = uniform(g.jobs[ji].rbits);
    region0 = uniform(g.jobs[ji].region0);
    slot0 = readlane64(g.jobs[ji].slot0, 0);
  };
  job();
  find();
  af = th;
  af_nums = numbers(af.start, af.count, 0);
  find();
  uint32_t nums = af_nums;
  ahead();
  find();
  /* nothing read ahead is under way where the loop is entered or repeated:
   * a wait inside it then covers its own loads only */
#pragma unroll
  for (int k = 0; k < REGION_ITEMS; ++k) consume(rn[k]);
  consume((uint64_t)af_nums);
  while (nx.q < g.q1) {
    const uint32_t q = nx.q, count = nx.count, start = nx.start;
    while (q >= ji_end) {
      ++ji;
      job();
    }
    const uint32_t rq = q - region0;
    R rr[REGION_ITEMS];
#pragma unroll
    for (int k = 0; k < REGION_ITEMS; ++k) rr[k] = rn[k];
    const uint64_t base = slot0 + (uint64_t)rq * span;
    Slot<KT>* T = (Slot<KT>*)g.table + base;
    if (g.valid) {
      L.template load<BS>(span, T);
      lds_barrier();
      for (uint32_t i = threadIdx.x; i < span; i += BS) lds_begin(L, i);
    } else {
      L.template clear<BS>(span);
    }
    uint32_t nums_nx = af_nums;
    ahead();
    lds_barrier();
    /* the first tile, loaded ahead; a region longer than one tile loads
     * the rest here (in registers of their own, so the first tile's adds
     * wait for nothing) */
#pragma unroll
    for (int k = 0; k < REGION_ITEMS; ++k) {
      uint32_t e = NO_SPILL;
      if (k * BS + threadIdx.x < count) e = region_add<KT, SLOTS, R>(g, L, span, rbits, rr[k], my_new, my_k2);
      spill_queue(g, spq, qn, e, base, (uint32_t)rec_key(rr[k]) & 31, my_k2);
    }
    for (uint32_t t = 1; t * TILE < count; ++t) {
      if (t % TILES == 0) nums = numbers(start, count, t);
      R rt[REGION_ITEMS];
      load(count, nums, t, rt);
#pragma unroll
      for (int k = 0; k < REGION_ITEMS; ++k) consume(rt[k]);
#pragma unroll
      for (int k = 0; k < REGION_ITEMS; ++k) {
        uint32_t e = NO_SPILL;
        if (t * TILE + k * BS + threadIdx.x < count)
          e = region_add<KT, SLOTS, R>(g, L, span, rbits, rt[k], my_new, my_k2);
        spill_queue(g, spq, qn, e, base, (uint32_t)rec_key(rt[k]) & 31, my_k2);
      }
    }
    /* what was read ahead since this region began is waited for here, before the write-back's stores: stores and loads
     * share one in-order counter, so waiting for them after the stores
     * would wait for the stores too */
#pragma unroll
    for (int k = 0; k < REGION_ITEMS; ++k) consume(rn[k]);
    consume((uint64_t)af_nums);
    find();
    nums = nums_nx;
    lds_barrier();
    /* a slot's words are finished by the thread that reads them below (the
     * fused filter: by a lane of the same wave) */
    const uint64_t h_top = (uint64_t)(rq >> (rbits - REC_BUCKET_BITS)) << (64 - REC_BUCKET_BITS);
    if (FUSE || !g.cbits)
      for (uint32_t i = threadIdx.x; i < span; i += BS) lds_finish(L, i, h_top);
    bool left = false; /* a candidate of this wave's slots found its list full */
    if constexpr (FUSE) {
      /* each wave queues the candidates of its slots (lane l holds the
       * l-th) and filters them 64 at a time, so every lane of a pass has
       * a slot */
      const uint32_t lane = __lane_id();
      uint32_t fs = 0, fn = 0; /* this lane's queued slot, the queue's fill */
      for (uint32_t i0 = 0; i0 < span; i0 += BS) {
        const uint32_t i = i0 + threadIdx.x;
        bool sp = false;
        const bool c = i < span && lds_candidate(g, L, i, sp);
        const uint64_t m = __ballot(c);
        const uint32_t n = (uint32_t)__popcll(m);
        if (n == 0) continue;
        const uint32_t rank = (uint32_t)__popcll(m & ((1ULL << lane) - 1));
        /* a permutation of the lanes: the candidates to lanes fn + rank,
         * the other lanes after them (mod 64) */
        const uint32_t to = (c ? fn + rank : fn + n + lane - rank) & 63;
        const uint32_t v = (uint32_t)__builtin_amdgcn_ds_permute((int)(to << 2), (int)i);
        if (fn + n < 64) {
          if (((lane - fn) & 63) < n) fs = v;
          fn += n;
        } else {
          if (lane >= fn) fs = v;
          left |= fuse_nodes<KT, SLOTS>(g, L, base, fs, true, ch);
          fs = v; /* lanes below the new fill hold the rest */
          fn = fn + n - 64;
        }
      }
      if (fn) left |= fuse_nodes<KT, SLOTS>(g, L, base, fs, lane < fn, ch);
    }
    if (g.cbits) {
      /* the filter scan's choice for every slot of the region, one
       * ballot per 64 slots; with the filter fused, only what a full
       * list left */
      for (uint32_t i0 = 0; i0 < span; i0 += BS) {
        const uint32_t i = i0 + threadIdx.x;
        bool c = false, sp = false;
        if (i < span) {
          c = lds_candidate(g, L, i, sp);
          if (!FUSE) lds_finish(L, i, h_top);
        }
        if (FUSE && !left) c = false;
        const uint64_t bc = __ballot(c), bsp = __ballot(sp);
        const uint32_t w0 = i0 + (threadIdx.x & ~63u);
        if ((threadIdx.x & 63) == 0 && w0 < span) {
          g.cbits[(uint64_t)q * g.stride + w0 / 64] = bc;
          g.sbits[(uint64_t)q * g.stride + w0 / 64] = bsp;
        }
      }
    }
    lds_barrier(); /* the k-mers and node records are in LDS */
    L.template store<BS>(span, T);
    lds_barrier();
  }
  const unsigned long long sn = wave_sum(my_new), sk = wave_sum(my_k2);
  if ((threadIdx.x & 63) == 0) {
    if (sn) atomicAdd(&g.ctr->n_distinct, sn);
    if (sk) atomicAdd(&g.ctr->n_k2, sk);
    g.spq_n[wave_id] = qn;
  }
  if constexpr (FUSE) {
    /* the open chunks' unused positions */
    const uint32_t lane = __lane_id();
#pragma unroll
    for (int l = 0; l < 2; ++l) {
      const uint64_t start = ch[l].base + ch[l].used;
      const uint32_t cnt = FUSE_CHUNK - ch[l].used;
      if (lane < cnt && start + lane < g.nl.cap) (l ? g.nl.branch_slot : g.nl.chain_slot)[start + lane] = LIST_HOLE;
      if (lane == 0) g.holes[2 * wave_id + l] = (start << 7) | cnt;
    }
  }
}

}  // namespace br

#endif
