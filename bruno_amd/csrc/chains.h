/*
 * chains.h -- list ranking by ruler contraction and the placing of its
 * result (well-formed chain graphs).
 *
 * Included by bruno_hip.hip inside its kernel section.  On a chain graph
 * where every end pointing at a chain node is pointed back at, the chain
 * nodes form disjoint paths and cycles, and the end state of bruno's
 * pointer jumping (debruijn_chain_graph.hpp:793-994, :1040-1310) is fixed:
 * every node knows the two chain ends it leads to and their distances, cycle
 * nodes end with both distances 2^T, and the number of rounds T is the
 * largest ceil(log2 L) over paths of L >= 2 nodes, at least 1 when a cycle
 * exists.  So neither the rounds nor the per-node end state are computed:
 *
 *   k_ruler_list  rulers (chain ends and sampled nodes, marked by
 *                 k_chain_init) are numbered
 *   k_lr_walk     a walk from every ruler along each open end to the next
 *                 ruler, reading one pointer per step and writing nothing:
 *                 the contracted list
 *   k_lr_jump     pointer jumping on the contracted list
 *   k_lr_ends     path lengths, T, counts
 *   k_chain_heads, k_units   one record per path (its representative, its
 *                 length, the ruler it starts from), sorted and given its
 *                 place in the output
 *   k_place       every ruler, now knowing its place, walks to the next
 *                 ruler once more and writes the k-mers it passes to
 *                 consecutive places of the output order
 *
 * What bounds it: the walks' random reads, one 32-byte record per step
 * (20-30 G records/s when the records exceed the 256 MB Infinity Cache), and
 * on small graphs the longest walk (ruler period x ln(rulers) steps of one
 * cache miss each).  Before, every node was visited from both sides and
 * written, then read, ranked and scattered by four whole-array passes, and
 * each path's rulers were walked serially from its ends: list ranking and
 * output of 40 M chain nodes took 7.6 + 4.4 ms and take 2.7 + 2.7 ms, of
 * 1 M nodes in 48 paths 2.0 + 0.34 ms and now 0.18 + 0.27 ms.
 */
#ifndef BRUNO_CHAINS_H_
#define BRUNO_CHAINS_H_

constexpr uint32_t NONE32 = 0xFFFFFFFFu;
constexpr uint32_t WALK_MAX = 1u << 16;
constexpr uint32_t ERR_WALK = 32;
constexpr uint32_t ERR_NO_NODE = 64; /* an output k-mer without its filtered-graph record */

/* The numbered rulers: one bit per chain node, the number of the first
 * ruler of every 64 nodes, and the rulers' nodes.  (A ruler's number comes
 * from its word's bits, so nothing is written to the node.) */
struct Rulers {
  const uint64_t* bits;
  const uint32_t* base;
  const uint32_t* node;
  uint64_t n;
};
__device__ __forceinline__ bool is_ruler(const Rulers& R, uint32_t j) { return (R.bits[j >> 6] >> (j & 63)) & 1; }
__device__ __forceinline__ uint32_t ruler_number(const Rulers& R, uint32_t j) {
  return R.base[j >> 6] + (uint32_t)__popcll(R.bits[j >> 6] & ((1ULL << (j & 63)) - 1));
}

/* State of the directed list entry x = 2 * ruler + end ("leaving that ruler
 * through that end"): bits 0-30 the distance covered, bits 31-62 the entry
 * reached, bit 63 set when that entry's end is a chain end (entry 2 r + f:
 * ruler r is the end of the chain, f its open side). */
constexpr uint64_t LS_DONE = 1ULL << 63;
constexpr uint64_t LS_UNSET = ~0ULL;
__device__ __forceinline__ uint64_t ls_pack(bool done, uint32_t next, uint32_t dist) {
  return (done ? LS_DONE : 0ULL) | ((uint64_t)next << 31) | (dist & DIST_MASK);
}
__device__ __forceinline__ uint32_t ls_next(uint64_t s) { return (uint32_t)(s >> 31); }
__device__ __forceinline__ uint32_t ls_dist(uint64_t s) { return (uint32_t)s & DIST_MASK; }
__device__ __forceinline__ uint64_t ls_load(const uint64_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void ls_store(uint64_t* p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

/* totals of a ranking: LRT_* words, then per job the rounds T, and the
 * isolated and cycle nodes */
enum : int { LRT_SUM = 0, LRT_HEADS, LRT_SINGLES, LRT_ISOLATED, LRT_CYCLE, LRT_UNITS, LRT_PLACED, LRT_WORDS };

__device__ __forceinline__ uint32_t ceil_log2(uint32_t L) { return L <= 1 ? 0 : 32 - __clz(L - 1); }

/* Whether chain node t is a sampled ruler (one in mask + 1 on average). */
__device__ __forceinline__ bool sampled_ruler(uint64_t t, uint64_t mask) {
  return (fmix64(t * 0x9e3779b97f4a7c15ULL + 0x1234567ULL) & mask) == 0;
}

/* Numbers the marked rulers: one word of 64 nodes per thread. */
__global__ __launch_bounds__(BLOCK) void k_ruler_list(const uint64_t* bits, uint64_t n_words, uint32_t* base,
                                                      uint32_t* node, Counters* ctr) {
  __shared__ ReserveSmem sm;
  for (uint64_t w0 = (uint64_t)blockIdx.x * BLOCK; w0 < n_words; w0 += (uint64_t)gridDim.x * BLOCK) {
    const uint64_t w = w0 + threadIdx.x;
    const uint64_t m = w < n_words ? bits[w] : 0;
    unsigned long long at = block_reserve((uint32_t)__popcll(m), &ctr->lr_next, sm);
    if (w < n_words) base[w] = (uint32_t)at;
    for (uint64_t b = m; b; b &= b - 1) node[at++] = (uint32_t)(w * 64 + __builtin_ctzll(b));
  }
}

/* From every ruler along each open end to the next ruler.  A walk gives the
 * contracted list's entry for its own direction and for the way back, and a
 * walk whose entry the other side has already written is not made: the ends
 * of one side go first (entries in the order end 0 of all rulers, end 1 of
 * all rulers), which leaves about half of the second half to do when the
 * list is larger than what runs at once.  alive[] loses the isolated nodes
 * (separate_isolated, debruijn_chain_graph.hpp:735-777). */
__global__ __launch_bounds__(BLOCK) void k_lr_walk(const LRNode* lr, Rulers R, uint64_t* S, uint8_t* alive,
                                                   const uint32_t* cjob, unsigned long long* tot,
                                                   unsigned long long* job_isolated, Counters* ctr) {
  const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
  unsigned long long iso = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; i < 2 * R.n; i += stride) {
    const int E = i >= R.n;
    const uint32_t rid = (uint32_t)(i - (E ? R.n : 0)), x = 2 * rid + (uint32_t)E;
    const uint32_t r = R.node[rid];
    const uint32_t d0 = lr[r].d[0], d1 = lr[r].d[1];
    if (is_terminal(E ? d1 : d0)) {
      ls_store(S + x, ls_pack(true, x, 0));
      if (!E && points_to_self(d0) && points_to_self(d1)) {
        alive[r] = 0;
        ++iso;
        if (cjob) atomicAdd(&job_isolated[cjob[r]], 1ULL);
      }
      continue;
    }
    if (__hip_atomic_load(S + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != LS_UNSET) continue;
    uint32_t ptr = lr[r].p[E], dist = 0;
    for (;;) {
      const uint32_t j = ptr & IDX_MASK;
      const uint32_t e = ptr >> 31;
      ++dist;
      if (is_ruler(R, j)) {
        const uint32_t y = 2 * ruler_number(R, j) + (1 - e);
        __hip_atomic_store(S + x, ls_pack(false, y, dist), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(S + (y ^ 1), ls_pack(false, x ^ 1, dist), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
      if (dist >= WALK_MAX) {
        atomicOr(&ctr->err, ERR_WALK);
        break;
      }
      ptr = lr[j].p[1 - e];
    }
  }
  block_add(iso, &tot[LRT_ISOLATED]);
}

/* Pointer jumping on the contracted list, JUMPS hops per entry and launch,
 * in place: an entry only ever grows (the distance and the entry reached
 * are one word, and both an old and a new value of another entry are
 * valid), so after a launch every unfinished entry covers at least JUMPS + 1
 * times what the least advanced entry covered before it.  A launch that
 * follows one that left nothing unfinished does nothing; what is still
 * unfinished after the last one lies on cycles.  (A serial walk of every
 * path's rulers took 1.5 ms of a 4.2 ms job on one 1 Mbp chain.) */
constexpr int LR_JUMPS = 3;
constexpr int LR_JUMP_LAUNCHES = 17; /* 4^17 entries */
__global__ __launch_bounds__(BLOCK) void k_lr_jump(uint64_t* S, uint64_t n, const uint32_t* left_before,
                                                   uint32_t* left_after) {
  if (left_before && *left_before == 0) return;
  const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
  bool left = false;
  for (uint64_t x = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; x < n; x += stride) {
    uint64_t s = ls_load(S + x);
    if (s & LS_DONE) continue;
#pragma unroll
    for (int q = 0; q < LR_JUMPS; ++q) {
      if (s & LS_DONE) break;
      const uint64_t t = ls_load(S + ls_next(s));
      s = ls_pack((t & LS_DONE) != 0, ls_next(t), ls_dist(s) + ls_dist(t));
    }
    ls_store(S + x, s);
    left |= !(s & LS_DONE);
  }
  if (__any(left) && (threadIdx.x & 63) == 0) *left_after = 1;
}

/* Entry x leads into a path from its end (a head), is the one entry kept
 * for a path of one node (through the OUT end), or neither. */
__device__ __forceinline__ int head_kind(const LRNode* lr, uint32_t r, uint32_t E) {
  const uint32_t d0 = lr[r].d[0], d1 = lr[r].d[1];
  const bool here = is_terminal(E ? d1 : d0), other = is_terminal(E ? d0 : d1);
  if (!here && other) return 1;
  if (E && here && other && !(points_to_self(d0) && points_to_self(d1))) return 2;
  return 0;
}

/* Nodes on paths (every path counted from both of its heads), paths, and
 * the rounds T per job.  (Two workgroups per CU: the totals are a few
 * atomics per workgroup on one line, and 4,096 workgroups spent 0.49 ms on
 * them where the entries' reads take 0.03 ms.) */
__global__ __launch_bounds__(BLOCK) void k_lr_ends(const LRNode* lr, Rulers R, const uint64_t* S, const uint32_t* cjob,
                                                   unsigned long long* tot, unsigned long long* jT, Counters* ctr) {
  const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
  unsigned long long sum = 0, heads = 0, singles = 0;
  uint32_t maxr = 0;
  for (uint64_t x = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; x < 2 * R.n; x += stride) {
    const uint32_t r = R.node[x >> 1];
    const int kind = head_kind(lr, r, (uint32_t)(x & 1));
    if (kind == 2) ++singles;
    if (kind != 1) continue;
    const uint64_t s = S[x];
    if (!(s & LS_DONE)) {
      atomicOr(&ctr->err, ERR_WALK);
      continue;
    }
    const uint32_t L = ls_dist(s) + 1, T = ceil_log2(L);
    sum += L;
    ++heads;
    if (cjob) {
      if (T > jT[cjob[r]]) atomicMax(&jT[cjob[r]], (unsigned long long)T);
    } else {
      maxr = T > maxr ? T : maxr;
    }
  }
  block_add(sum, &tot[LRT_SUM]);
  __syncthreads();
  block_add(heads, &tot[LRT_HEADS]);
  __syncthreads();
  block_add(singles, &tot[LRT_SINGLES]);
  if (!cjob) {
    typedef hipcub::BlockReduce<uint32_t, BLOCK> BR;
    __shared__ typename BR::TempStorage tmp;
    const uint32_t m = BR(tmp).Reduce(maxr, hipcub::Max());
    if (threadIdx.x == 0 && m) atomicMax(&jT[0], (unsigned long long)m);
  }
}

/* Only when some nodes lie on cycles (fewer nodes on paths than there are):
 * the nodes of the paths are marked, the rest separated (separate_cycles,
 * debruijn_chain_graph.hpp:670-733). */
__global__ __launch_bounds__(BLOCK) void k_lr_mark_paths(const LRNode* lr, Rulers R, const uint64_t* S, uint8_t* on_path) {
  const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
  for (uint64_t x = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; x < 2 * R.n; x += stride) {
    if (!(S[x] & LS_DONE)) continue;
    const uint32_t r = R.node[x >> 1], E = (uint32_t)(x & 1);
    on_path[r] = 1;
    if (is_terminal(lr[r].d[E])) continue;
    uint32_t ptr = lr[r].p[E];
    for (uint32_t n = 0; n < WALK_MAX; ++n) {
      const uint32_t j = ptr & IDX_MASK;
      if (is_ruler(R, j)) break;
      on_path[j] = 1;
      ptr = lr[j].p[1 - (ptr >> 31)];
    }
  }
}
__global__ __launch_bounds__(BLOCK) void k_lr_drop_cycles(const uint8_t* on_path, uint64_t n_chain, const uint32_t* cjob,
                                                          uint8_t* alive, unsigned long long* job_cycle) {
  const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
  for (uint64_t t = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; t < n_chain; t += stride)
    if (!on_path[t]) {
      alive[t] = 0;
      atomicAdd(&job_cycle[cjob ? cjob[t] : 0u], 1ULL);
    }
}

/* The mailboxes back to empty, for the round-by-round path (k_chain_init
 * leaves the node's k-mer in them). */
__global__ __launch_bounds__(BLOCK) void k_lr_zero_mail(LRNode* lr, uint64_t n_chain) {
  const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
  for (uint64_t t = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; t < n_chain; t += stride) {
    lr[t].mail[0] = 0ULL;
    lr[t].mail[1] = 0ULL;
  }
}

/* a chain node's k-mer as k_chain_init left it in the node's record */
template <typename KT> __device__ __forceinline__ KT lr_kmer(const LRNode& n);
template <> __device__ __forceinline__ uint64_t lr_kmer<uint64_t>(const LRNode& n) { return n.mail[0]; }
template <> __device__ __forceinline__ u128 lr_kmer<u128>(const LRNode& n) {
  return ((u128)n.mail[1] << 64) | n.mail[0];
}

/* Every path once, from the end whose k-mer, on the strand that leads into
 * the path, is the smaller: that k-mer is the representative
 * (to_listranked_chain_node, debruijn_chain_operations.hpp:261-310). */
template <typename KT>
__global__ __launch_bounds__(BLOCK) void k_chain_heads(const LRNode* lr, Rulers R, const uint64_t* S, int K,
                                                       const uint32_t* cjob, uint64_t n_units, KT* key, uint32_t* len,
                                                       uint32_t* entry, uint32_t* job, unsigned long long* tot,
                                                       Counters* ctr) {
  __shared__ ReserveSmem sm;
  kops<KT> ops(K);
  for (uint64_t base = (uint64_t)blockIdx.x * BLOCK; base < 2 * R.n; base += (uint64_t)gridDim.x * BLOCK) {
    const uint64_t x = base + threadIdx.x;
    bool rep = false;
    KT k = 0;
    uint32_t r = 0, L = 1;
    if (x < 2 * R.n) {
      const uint32_t E = (uint32_t)(x & 1);
      r = R.node[x >> 1];
      const int kind = head_kind(lr, r, E);
      if (kind) {
        k = lr_kmer<KT>(lr[r]);
        if (!E) k = ops.rc(k);
        rep = true;
        if (kind == 1) {
          /* the far end: its open side is y & 1, so the way back leaves it
           * through the other */
          const uint64_t s = S[x];
          const uint32_t y = ls_next(s);
          KT o = lr_kmer<KT>(lr[R.node[y >> 1]]);
          if (y & 1) o = ops.rc(o);
          L = ls_dist(s) + 1;
          rep = (s & LS_DONE) && (k < o || (k == o && (uint32_t)x < (y ^ 1)));
        }
      }
    }
    const unsigned long long at = block_reserve(rep, &tot[LRT_UNITS], sm);
    if (!rep) continue;
    if (at >= n_units) {
      atomicOr(&ctr->err, ERR_LIST_FULL);
      continue;
    }
    key[at] = k;
    len[at] = L;
    entry[at] = (uint32_t)x;
    if (job) job[at] = cjob[r];
  }
}

/* the paths in output order: representative, length, and the path's number
 * at the entry it starts from */
template <typename KT>
__global__ void k_units(const uint32_t* perm, const KT* key, const uint32_t* len, const uint32_t* entry,
                        const uint32_t* job, uint64_t n, KT* urep, uint32_t* ulen, uint32_t* ujob, uint32_t* unit_of) {
  const uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u > n) return;
  if (u == n) {
    ulen[n] = 0; /* so the exclusive sum ends with the total */
    return;
  }
  const uint32_t p = perm[u];
  urep[u] = key[p];
  ulen[u] = len[p];
  unit_of[entry[p]] = (uint32_t)u;
  if (ujob) ujob[u] = job[p];
}

/* per job: its first path (q0) and that path's first node (c0) */
__global__ void k_unit_starts(const uint64_t* ustart, uint64_t n, const uint32_t* coff, uint64_t* cstart) {
  const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) cstart[q] = coff[ustart[q]];
}

/* Every ruler finds its path and its place (the path's first place plus the
 * distance from the end the path starts at), writes its k-mer on the
 * representative's strand there, and walks away from that end to the next
 * ruler, writing every node it passes to the next place. */
template <typename KT>
__global__ __launch_bounds__(BLOCK) void k_place(const LRNode* lr, Rulers R, const uint64_t* S, const uint32_t* unit_of,
                                                 const uint32_t* coff, int K, KT* out_k, unsigned long long* tot,
                                                 Counters* ctr) {
  kops<KT> ops(K);
  const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
  unsigned long long placed = 0;
  for (uint64_t rid = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; rid < R.n; rid += stride) {
    const uint64_t s0 = S[2 * rid], s1 = S[2 * rid + 1];
    if (!(s0 & s1 & LS_DONE)) continue; /* on a cycle */
    /* the end reached through E is the path's start when the entry that
     * leads into the path from there has a path number */
    const uint32_t u0 = unit_of[ls_next(s0) ^ 1], u1 = unit_of[ls_next(s1) ^ 1];
    const uint32_t u = u0 != NONE32 ? u0 : u1;
    if (u == NONE32) continue; /* isolated */
    const int F = u0 != NONE32 ? 1 : 0; /* away from the start */
    uint64_t pos = (uint64_t)coff[u] + ls_dist(F ? s0 : s1);
    const uint64_t end = coff[u + 1];
    LRNode st = lr[R.node[rid]];
    int out_end = F;
    for (;;) {
      if (pos >= end) {
        atomicOr(&ctr->err, ERR_WALK);
        break;
      }
      const KT k = lr_kmer<KT>(st);
      out_k[pos++] = out_end ? k : ops.rc(k);
      ++placed;
      if (is_terminal(st.d[out_end])) break;
      const uint32_t ptr = st.p[out_end], j = ptr & IDX_MASK;
      if (is_ruler(R, j)) break;
      st = lr[j];
      out_end = 1 - (int)(ptr >> 31);
    }
  }
  block_add(placed, &tot[LRT_PLACED]);
}

/* The listranked nodes in output order (by job, representative, distance):
 * after a placing by paths the k-mers are stored in that order, with each
 * node's path number, the paths' representatives and first places; after a
 * sort, through a permutation. */
template <typename KT>
struct OutView {
  const KT* k;
  const uint32_t* uid; /* null: sorted */
  const uint32_t* coff;
  const KT* urep;
  const uint32_t* perm;
  const KT* rep;
  const uint32_t* dist;
  __device__ __forceinline__ KT kmer(uint64_t i) const { return uid ? k[i] : k[perm[i]]; }
  __device__ __forceinline__ KT rep_of(uint64_t i) const { return uid ? urep[uid[i]] : rep[perm[i]]; }
  __device__ __forceinline__ uint32_t dist_of(uint64_t i) const { return uid ? (uint32_t)i - coff[uid[i]] : dist[i]; }
};

/* Largest u < n with start[u] <= x (start[0] <= x), by the whole wave: 64
 * probes a step, so three dependent loads for 2^18 entries. */
__device__ __forceinline__ uint32_t wave_find(const uint32_t* start, uint32_t n, uint32_t x) {
  const uint32_t lane = threadIdx.x & 63;
  uint32_t lo = 0, hi = n; /* start[lo] <= x < start[hi] */
  while (hi - lo > 1) {
    const uint32_t step = (hi - lo + 63) / 64;
    const uint32_t at = lo + (lane + 1) * step;
    const uint64_t m = __ballot(at < hi && start[at] <= x);
    const uint32_t c = (uint32_t)__popcll(m);
    lo += c * step;
    hi = lo + step < hi ? lo + step : hi;
  }
  return lo;
}

/* .chain.fasta from the placed k-mers (print_chain_as_fasta,
 * debruijn_chain_operations.hpp:352-385: a path's first node starts a
 * record "\n>" canonical(K) "\n" K, every other node adds its last base),
 * and every node's path number.  A workgroup takes TILE consecutive nodes:
 * the path numbers come from a scan over the path starts inside the tile,
 * a node's byte from its place and path number alone (each record before
 * it adds 2K + 2 bytes beyond one per node), so bytes go out in order, and
 * a wave writes each record's start. */
constexpr int FASTA_ITEMS = 8;
template <typename KT>
__global__ __launch_bounds__(BLOCK) void k_path_fasta(const KT* out_k, const uint32_t* coff, uint64_t n_units,
                                                      uint64_t n, int K, uint32_t* uid, char* buf) {
  constexpr uint32_t TILE = BLOCK * FASTA_ITEMS;
  typedef hipcub::BlockScan<uint32_t, BLOCK> Scan;
  __shared__ typename Scan::TempStorage tmp;
  __shared__ uint32_t mark[TILE];
  kops<KT> ops(K);
  const char A[4] = {'A', 'C', 'G', 'T'};
  const uint64_t extra = 2 * (uint64_t)K + 2;
  for (uint64_t i0 = (uint64_t)blockIdx.x * TILE; i0 < n; i0 += (uint64_t)gridDim.x * TILE) {
    const uint64_t i1 = i0 + TILE < n ? i0 + TILE : n;
    for (uint32_t q = threadIdx.x; q < TILE; q += BLOCK) mark[q] = 0;
    const uint32_t uf = wave_find(coff, (uint32_t)n_units, (uint32_t)i0);
    __syncthreads();
    for (uint64_t u = (uint64_t)uf + 1 + threadIdx.x; u < n_units && coff[u] < i1; u += BLOCK)
      mark[coff[u] - i0] = (uint32_t)(u - uf);
    __syncthreads();
    uint32_t v[FASTA_ITEMS];
#pragma unroll
    for (int q = 0; q < FASTA_ITEMS; ++q) v[q] = mark[threadIdx.x * FASTA_ITEMS + q];
    Scan(tmp).InclusiveScan(v, v, hipcub::Max());
    __syncthreads();
#pragma unroll
    for (int q = 0; q < FASTA_ITEMS; ++q) mark[threadIdx.x * FASTA_ITEMS + q] = v[q];
    __syncthreads();
    for (uint64_t i = i0 + threadIdx.x; i < i1; i += BLOCK) {
      const uint32_t u = uf + mark[i - i0];
      uid[i] = u;
      if (coff[u] != (uint32_t)i) buf[i + (u + 1) * extra] = A[(uint32_t)out_k[i] & 3u];
    }
    /* record starts */
    const uint32_t ul = uf + mark[i1 - 1 - i0];
    const uint32_t lane = threadIdx.x & 63;
    for (uint32_t u = uf + (coff[uf] < i0 ? 1 : 0) + (threadIdx.x >> 6); u <= ul; u += BLOCK / 64) {
      const KT k = out_k[coff[u]], c = ops.canon(k);
      char* o = buf + coff[u] + u * extra;
      for (uint32_t p = lane; p < extra + 1; p += 64) {
        char ch = '\n';
        if (p == 1) ch = '>';
        else if (p >= 2 && p < 2 + (uint32_t)K) ch = A[(int)((c >> (2 * (K + 1 - (int)p))) & 3)];
        else if (p >= 3 + (uint32_t)K) ch = A[(int)((k >> (2 * (2 * K + 2 - (int)p))) & 3)];
        o[p] = ch;
      }
    }
    __syncthreads();
  }
}

#endif
