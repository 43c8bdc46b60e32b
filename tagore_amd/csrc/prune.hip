// prune.hip -- CFS (Collect-Filter-Store) pruning kernels for gfx950.
//
// One wave64 workgroup per node.  The Collect step (path beam search / two-hop list), the
// incremental Filter and the Store of reverse edges follow the deterministic rule spec that
// the CPU oracle restates (oracle/tagore_oracle.cpp), so the adjacency produced here is
// bit-identical to it:
//   collect_path  Tagore_src.cu:1209-1349     collect_2hop      Tagore_src.cu:1352-1396
//   Filter_path   Tagore_src.cu:1399-1485     rules             Tagore_src.cu:1488-1495
//   filter_reverse Tagore_src.cu:1537-1657    cal_ep_gpu        Tagore_src.cu:1889-2058
//   filter_cagra  Tagore_src.cu:1668-1710     filter_dpg        Tagore_src.cu:1713-1785
//   filter_reverse_1hop Tagore_src.cu:1812-1886
// Distances are the canonical FP32 squared L2 on FP32 rows (16 lanes per distance, four
// distances in flight per wave).  The kNN input graph is never modified: pruned rows go to
// separate buffers, so one kNN build can feed several prunings.
#include "common.hpp"
#include "kernels.hpp"
#include "screen.hpp"

namespace tg {

constexpr int RING = 480;

// phase-clock sums of one workgroup (profiling builds of the forward kernels): distance batches,
// and the beam rounds' candidate step, sort, merge and id-set rebuild.  A type, not a flag:
// the sums and the tests of a flag took scalar registers across the whole kernel (95 of them
// spilled in the u8 path kernel).
struct PhaseOff {
  static constexpr bool on = false;
  long long ev, sub[4];
};
struct PhaseOn {
  static constexpr bool on = true;
  long long ev = 0;
  long long sub[4] = {0, 0, 0, 0};
};
template <class Ph>
__device__ __forceinline__ long long pclock(const Ph&) {
  return Ph::on ? clock64() : 0;
}
template <class Ph>
__device__ __forceinline__ void padd(Ph&, long long& sum, long long dt) {
  if (Ph::on) sum += dt;
}
constexpr int POOL_MAX = 1024;  // K + 480 <= 608, padded to a power of two

// Id set in LDS: 2^bits buckets of four ids (INV: empty), each with a 16-bit count, in
// hs_words(bits) words.  An insert takes a place by adding to its bucket's count and moves on to the
// next bucket when this one is full; a look-up reads one bucket and moves on only past a full
// one.  The beam's set holds at most TOPM + K members, less than its places (hs_bits), so both
// end whatever the ids are.  Against open addressing over single slots there is no chain of
// compare-and-swaps, as long as the longest of the wave's 64: the inserts of one round overlap.
// (Path Collect over 1M x 128 u8 rows, K 96, TOPM 64, profiled cycles per node: look-ups and
// compaction 106k with 256 single slots, 43k with 512, 36k with the buckets; inserts 62k / 58k
// with 512 / the buckets.)
// -------------------------------------------------------------------------------------
__host__ __device__ constexpr int hs_words(int bits) { return (4 << bits) + ((1 << bits) >> 1); }
// 64 buckets up to 128 members (W = 1), half of the places, 128 up to 256.  Where the pool's
// filter needs little LDS itself (no matrix filter), 128 leave 21 workgroups per CU instead of
// 24, so more nodes than then run at once take 64 up to 176 members too; fewer nodes only wait
// for the longer chains.  (FP32 rows without a 16-bit copy, forward pass with 128 / 64 buckets:
// 6k x 100, K = 64, TOPM 88 NSG 0.290 / 0.282 ms, Vamana 0.765 / 0.688; 40k x 36, K = 72, TOPM 64
// 1.96 / 1.87 and 4.54 / 4.18; 120k x 100, K = 112 8.82 / 8.67 and 29.0 / 27.9; 2k x 100, K = 96
// 0.222 / 0.243 and 0.610 / 0.624; 600 x 4, K = 100 0.12 / 0.22.  W = 1, 100k x 36, K = 48: NSG 4.15 /
// 3.86, Vamana 10.9 / 9.9).
constexpr uint32_t HS_AT_ONCE = 21 * 256;
__host__ __device__ constexpr int hs_bits(int W, uint32_t nodes, int members, bool mf) {
  return W == 1 ? 6 : (mf || nodes <= HS_AT_ONCE || members > 176) ? 7 : 6;
}
// (the 24-bit product is a full-rate instruction, the 32-bit one a quarter; ids that share
// their low 24 bits share a bucket)
__device__ __forceinline__ uint32_t hbucket(uint32_t id, int bits) {
  return ((id & 0xFFFFFFu) * 0x9E3779u) >> (32 - bits);
}
__device__ __forceinline__ void hset_clear(uint32_t* tab, int bits) {  // tab 16-byte aligned
  for (int i = 4 * threadIdx.x; i < (4 << bits); i += 4 * TG_WAVE)
    *reinterpret_cast<uint4*>(tab + i) = make_uint4(TG_INV, TG_INV, TG_INV, TG_INV);
  // (128 buckets: every lane; the test alone took the u8 path kernel four more spilled scalars,
  // 28.6 -> 28.9 ms for NSG over 1M x 128)
  if (bits == 7 || int(threadIdx.x) < (1 << bits) / 2) tab[(4 << bits) + threadIdx.x] = 0;
}
// inserts one id per lane and list entry (INV: none)
template <int C>
__device__ __forceinline__ void hset_insert(uint32_t* tab, const uint32_t (&id)[C], int bits) {
  uint32_t h[C], old[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    h[c] = hbucket(id[c], bits);
    old[c] = 0;
    if (id[c] != TG_INV)
      old[c] = atomicAdd(&tab[(4 << bits) + (h[c] >> 1)], 1u << ((h[c] & 1) * 16));
  }
#pragma unroll
  for (int c = 0; c < C; ++c) {
    if (id[c] == TG_INV) continue;
    uint32_t at = (old[c] >> ((h[c] & 1) * 16)) & 0xFFFFu;
    while (at >= 4) {
      h[c] = (h[c] + 1) & ((1 << bits) - 1);
      const uint32_t o = atomicAdd(&tab[(4 << bits) + (h[c] >> 1)], 1u << ((h[c] & 1) * 16));
      at = (o >> ((h[c] & 1) * 16)) & 0xFFFFu;
    }
    tab[h[c] * 4 + at] = id[c];
  }
}
__device__ __forceinline__ bool hset_has(const uint32_t* tab, uint32_t id, int bits) {
  uint32_t h = hbucket(id, bits);
  for (;;) {
    const uint4 v = *reinterpret_cast<const uint4*>(tab + h * 4);
    if (v.x == id || v.y == id || v.z == id || v.w == id) return true;
    if (v.w == TG_INV) return false;
    h = (h + 1) & ((1 << bits) - 1);
  }
}
static_assert((1 << 7) / 2 <= TG_WAVE, "one lane clears one word of counts");

// -------------------------------------------------------------------------------------
// Beam search shared by cal_ep and path Collect (spec in the oracle's beam_search).
// The beam lives in registers: position p = b*64 + lane is slot b of lane `lane`
// (b < W, TOPM <= 64*W; positions >= TOPM hold TG_KEY_INF).  A round evaluates the fresh
// candidates of the expanded node, sorts all K candidates in registers (S holds them by
// list position, 64*W >= K slots) and takes the TOPM smallest of beam and candidates with
// one bitonic merge: min(beam[p], cand[64W-1-p]) is bitonic and holds the 64W smallest of
// both, so sorting it gives the first 64W keys of merge(beam, candidates).
// tab: id set of the previous round's beam and candidates (the dedup set).  An entry is
// explored when its id is among the expanded ids (held in a register, one per lane): the
// beam never holds two finite entries with one id, and an expanded node that falls out of
// the beam can never re-enter it (the beam's TOPM-th key only decreases).  `out` (optional)
// receives the final beam (TOPM keys).
// With six waves per SIMD the rounds are bound by instruction issue, not by the loads: the
// profiling sums as a type, the buckets and the next list's early load took the NSG forward
// pass at that size from 31.9 to 29.3 ms.
// -------------------------------------------------------------------------------------
template <int MC, class T, int W, class Ph>
__device__ __forceinline__ void beam_search(const PruneArgs& a, const Row16<MC>& tgt,
                                            uint32_t start,
                                            int max_exp, uint64_t* S, uint32_t* tab, int bits,
                                            uint16_t* cl, uint64_t* ring, uint64_t* out, uint32_t& ring_c,
                                            uint32_t& n_eval, uint32_t& n_adj, Ph& ph) {
  const int lane = threadIdx.x;
  const int K = a.K, TOPM = a.TOPM, D = a.D;
  constexpr int NS = 64 * W;
  const T* X = reinterpret_cast<const T*>(a.rows);
  const uint64_t INFKEY = mk_key(__uint_as_float(0x7F800000u), 0u);
  auto load_adj = [&](uint32_t x, uint32_t (&y)[W]) {
#pragma unroll
    for (int q = 0; q < W; ++q)
      y[q] = q * TG_WAVE + lane < K ? a.G[size_t(x) * K + q * TG_WAVE + lane] : TG_INV;
  };
  // start list S = G[start] with distances (ring slots 0..K-1 in list order)
  for (int j = lane; j < NS; j += TG_WAVE)
    S[j] = j < K ? (INFKEY | a.G[size_t(start) * K + j]) : TG_KEY_INF;
  __syncthreads();
  eval_batch<MC, T, true>(X, D, tgt, K, [&](int q) { return key_id(S[q]); },
                 [&](int q, float d) {
                   const uint64_t k = mk_key(d, key_id(S[q]));
                   S[q] = k;
                   if (ring) ring[q % RING] = k;
                 });
  n_eval += K;
  n_adj += 1;
  ring_c = K;
  hset_clear(tab, bits);
  __syncthreads();
  uint64_t v[W], bk[W];
  {
    uint32_t ids[W];  // the first dedup set is ids(S); padding ids are INV
#pragma unroll
    for (int r = 0; r < W; ++r) {
      v[r] = S[r * 64 + lane];
      ids[r] = key_id(v[r]);
    }
    hset_insert(tab, ids, bits);
  }
  reg_bitonic<W>(v);
#pragma unroll
  for (int b = 0; b < W; ++b) bk[b] = b * 64 + lane < TOPM ? v[b] : TG_KEY_INF;
  __syncthreads();
  // the expanded ids in registers: lane e < nexpl holds the e-th (max_exp <= 64)
  uint32_t ex = TG_INV;
  int nexpl = 0;
  // key of the first explorable beam entry (position order), TG_KEY_INF when there is none
  auto explorable = [&]() {
    uint64_t k = TG_KEY_INF;
#pragma unroll
    for (int b = 0; b < W; ++b) {
      if (k != TG_KEY_INF) break;
      const uint32_t id = key_id(bk[b]);
      bool ok = key_finite(bk[b]);
      for (int e = 0; e < nexpl; ++e)
        ok = ok & (id != uint32_t(__builtin_amdgcn_readlane(int(ex), e)));
      const uint64_t m = ballot(ok);
      if (m) k = readlane64(bk[b], __ffsll((unsigned long long)m) - 1);
    }
    return k;
  };
  uint64_t next = explorable();
  uint32_t y[W];
  if (next != TG_KEY_INF) load_adj(key_id(next), y);
  for (int r = 0; r < max_exp && next != TG_KEY_INF; ++r) {
    const long long s0 = pclock(ph);
    if (lane == nexpl) ex = key_id(next);
    ++nexpl;
    n_adj += 1;
    // new candidates: duplicates of the dedup set get +inf; the rest compacted in j order
    int cnt = 0;
#pragma unroll
    for (int q = 0; q < W; ++q) {
      const int j = q * TG_WAVE + lane;
      bool fresh = false;
      if (j < K) {
        fresh = !hset_has(tab, y[q], bits);
        S[j] = INFKEY | y[q];
      } else {
        S[j] = TG_KEY_INF;
      }
      const uint64_t fm = ballot(fresh);
      if (fresh) cl[cnt + mask_rank(fm)] = uint16_t(j);
      cnt += __popcll(fm);
    }
    __syncthreads();
    const uint32_t c0 = ring_c;
    const long long e0 = pclock(ph);
    padd(ph, ph.sub[0], e0 - s0);
    eval_batch<MC, T, true>(X, D, tgt, cnt, [&](int q) { return key_id(S[cl[q]]); },
                   [&](int q, float d) {
                     const int j = cl[q];
                     const uint64_t k = mk_key(d, key_id(S[j]));
                     S[j] = k;
                     if (ring) ring[(c0 + q) % RING] = k;
                   });
    padd(ph, ph.ev, pclock(ph) - e0);
    ring_c += cnt;
    n_eval += cnt;
    __syncthreads();
    const long long s1 = pclock(ph);
#pragma unroll
    for (int q = 0; q < W; ++q) v[q] = S[q * 64 + lane];
    // Only candidates below the beam's TOPM-th key can enter it (a fresh id is in neither
    // the beam nor the previous candidates, so no key ties one in the beam).  With TOPM <= 64
    // and at most 64 such candidates, they are compacted and merged with one-slot sorts; none
    // leaves the beam as it is.  (One slot per lane: only once the beam is full of finite keys;
    // until then the merge also keeps keys without a distance, which count as seen.)  Either way
    // the beam becomes the TOPM smallest keys of beam and candidates.
    uint64_t worst = TG_KEY_INF;
#pragma unroll
    for (int b = 0; b < W; ++b)
      if (b == (TOPM - 1) >> 6) worst = readlane64(bk[b], (TOPM - 1) & 63);
    int m = 64 * W;
    bool small = false;
    uint64_t c[W];  // the candidates, sorted
#pragma unroll
    for (int q = 0; q < W; ++q) c[q] = v[q];
    if (TOPM <= 64 && (W > 1 || key_finite(worst))) {
      uint64_t qm[W];
      m = 0;
#pragma unroll
      for (int q = 0; q < W; ++q) {
        qm[q] = ballot(key_finite(v[q]) && v[q] < worst);
        m += __popcll(qm[q]);
      }
      small = m <= 64;
      if (small && m > 0) {
        int base = 0;
#pragma unroll
        for (int q = 0; q < W; ++q) {
          if ((qm[q] >> lane) & 1ull) S[base + mask_rank(qm[q])] = v[q];
          base += __popcll(qm[q]);
        }
        if (lane >= m) S[lane] = TG_KEY_INF;
        __syncthreads();
        c[0] = S[lane];
        // keys in lanes 0..m-1, +inf above: sorting blocks of the next power of two is enough
        if (m <= 16) reg_bitonic_upto<16>(c[0]);
        else if (m <= 32) reg_bitonic_upto<32>(c[0]);
        else reg_bitonic_upto<64>(c[0]);
      }
    }
    if (!small) reg_bitonic<W>(c);
    const long long s2 = pclock(ph);
    padd(ph, ph.sub[1], s2 - s1);
    // The next expansion is known before the merge: the smaller of the first explorable entry
    // and the smallest candidate that enters (an entry that the candidates push out of the beam
    // has a smaller candidate before it; an expanded id never comes back as one).  Its list is
    // on its way while the id set is rebuilt and the beam merged.
    next = explorable();
    if (m > 0) {
      const uint64_t cmin = readlane64(c[0], 0);
      if (cmin < worst && key_finite(cmin) && cmin < next) next = cmin;
    }
    if (next != TG_KEY_INF) load_adj(key_id(next), y);
    // next dedup set: ids of this round's beam and candidates
    hset_clear(tab, bits);
    __syncthreads();
    {
      uint32_t ids[2 * W];
#pragma unroll
      for (int q = 0; q < W; ++q) {
        ids[2 * q] = key_id(bk[q]);
        ids[2 * q + 1] = key_id(v[q]);
      }
      hset_insert(tab, ids, bits);
    }
    const long long s3 = pclock(ph);
    padd(ph, ph.sub[3], s3 - s2);
    if (small) {
      if (m > 0) {
        const uint64_t rv = lane_xor64(c[0], 63);
        uint64_t w1[1] = {bk[0] < rv ? bk[0] : rv};
        reg_bitonic_merge<1>(w1);
        bk[0] = lane < TOPM ? w1[0] : TG_KEY_INF;
      }
    } else {
      uint64_t w[W];
#pragma unroll
      for (int b = 0; b < W; ++b) {
        const uint64_t rv = lane_xor64(c[W - 1 - b], 63);  // candidate 64W-1-p
        w[b] = bk[b] < rv ? bk[b] : rv;
      }
      reg_bitonic_merge<W>(w);
#pragma unroll
      for (int b = 0; b < W; ++b) bk[b] = b * 64 + lane < TOPM ? w[b] : TG_KEY_INF;
    }
    __syncthreads();
    padd(ph, ph.sub[2], pclock(ph) - s3);
  }
  if (out) {
#pragma unroll
    for (int b = 0; b < W; ++b)
      if (b * 64 + lane < TOPM) out[b * 64 + lane] = bk[b];
  }
  __syncthreads();
}

// -------------------------------------------------------------------------------------
// The reverse pass's pool: the forward row (deg keys, ascending: selections come in key
// order) and the reverse top (nr keys, ascending) as one sorted sequence of 64 NPL keys,
// +inf after L = deg + nr.  [forward | +inf | reverse, last first] is bitonic, so one
// bitonic merge gives what a sort of the union gives.
// -------------------------------------------------------------------------------------
template <int NPL>
__device__ __forceinline__ void merge_pool(const PruneArgs& a, uint32_t u, int deg,
                                           const uint64_t* rev, int nr, uint64_t* P) {
  const int lane = threadIdx.x;
  constexpr int n = 64 * NPL;
  uint64_t v[NPL];
#pragma unroll
  for (int b = 0; b < NPL; ++b) {
    const int i = b * 64 + lane;
    v[b] = TG_KEY_INF;
    if (i < deg) v[b] = mk_key(a.fwd_d[size_t(u) * a.FD + i], a.fwd_ids[size_t(u) * a.FD + i]);
    else if (i >= n - nr) v[b] = rev[n - 1 - i];
  }
  reg_bitonic_merge<NPL>(v);
#pragma unroll
  for (int b = 0; b < NPL; ++b) P[b * 64 + lane] = v[b];
  __syncthreads();
}

// -------------------------------------------------------------------------------------
// In a sorted pool of n keys, replace the id of every entry whose id equals its
// predecessor's (original values) by INV.
// -------------------------------------------------------------------------------------
__device__ void mark_dups(uint64_t* P, int n) {
  const int lane = threadIdx.x;
  bool dup[POOL_MAX / TG_WAVE];
#pragma unroll
  for (int q = 0; q < POOL_MAX / TG_WAVE; ++q) {
    const int i = q * TG_WAVE + lane;
    dup[q] = (i < n && i > 0) ? (key_id(P[i]) == key_id(P[i - 1])) : false;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < POOL_MAX / TG_WAVE; ++q) {
    const int i = q * TG_WAVE + lane;
    if (dup[q]) P[i] = key_with_id(P[i], TG_INV);
  }
  __syncthreads();
}

// first index >= from, < L, whose id is not INV (and not `skip`); L if none
__device__ int next_valid(const uint64_t* P, int from, int L, uint32_t skip) {
  const int lane = threadIdx.x;
  for (int base = from; base < L; base += TG_WAVE) {
    const int i = base + lane;
    bool ok = false;
    if (i < L) {
      const uint32_t id = key_id(P[i]);
      ok = id != TG_INV && id != skip;
    }
    const uint64_t m = ballot(ok);
    if (m) return base + __ffsll((unsigned long long)m) - 1;
  }
  return L;
}

// -------------------------------------------------------------------------------------
// The next selection and the next round's candidate list, in one pass over the entries
// cl[from..from+n) (pool indices, in pool order): the first entry not invalidated is the
// selection (its pool index goes to pi, -1 when there is none); the entries after it that
// are not invalidated are the candidates, compacted to cl[0..), except those repeating the
// selection's id, which are invalidated uncounted (a round's start rule).  Returns the
// candidates' number.  Each 64-entry chunk is read before any of its entries is written,
// and writes land below the next chunk, so the compaction is in place.
// -------------------------------------------------------------------------------------
__device__ __forceinline__ int advance_cl(uint64_t* P, uint16_t* cl, int from, int n, int& pi) {
  const int lane = threadIdx.x;
  int out = 0;
  uint32_t sid = TG_INV;
  pi = -1;
  for (int base = 0; base < n; base += TG_WAVE) {
    const int j = base + lane;
    const int c = j < n ? int(cl[from + j]) : 0;
    const uint32_t id = j < n ? key_id(P[c]) : TG_INV;
    bool k = id != TG_INV;
    if (pi < 0) {
      const uint64_t m = ballot(k);
      if (m) {
        const int f = __ffsll((unsigned long long)m) - 1;
        pi = __builtin_amdgcn_readlane(c, f);
        sid = uint32_t(__builtin_amdgcn_readlane(int(id), f));
        k = k && lane > f;
      }
    }
    if (k && id == sid) {
      P[c] = key_with_id(P[c], TG_INV);
      k = false;
    }
    const uint64_t m = ballot(k);
    __syncthreads();
    if (k) cl[out + mask_rank(m)] = uint16_t(c);
    out += __popcll(m);
    __syncthreads();
  }
  return out;
}

// -------------------------------------------------------------------------------------
// Incremental Filter over the sorted pool P[0..L) (spec A.4 in the oracle).  Writes the
// kept entries to sel[] and returns their number.  cl holds the round's candidates: the pool
// indices after the current selection p that are not invalidated and do not repeat p's id,
// in pool order, so a round touches only the survivors of the previous round.  For rows that
// filter_pool_mfma does not take: wider than 256 elements, or without an 8-, 16-bit copy.
// -------------------------------------------------------------------------------------
template <int MC, class T, class Ph>
__device__ __forceinline__ int filter_pool(const PruneArgs& a, uint64_t* P, int L, uint32_t u,
                                           int rule, uint64_t* sel, uint16_t* cl,
                                           uint32_t& n_eval, Ph& ph) {
  const int lane = threadIdx.x, t = lane & 15;
  const int D = a.D, FD = a.FD;
  int tix = next_valid(P, 0, L, u);
  if (tix >= L) return 0;
  int nsel = 1;
  if (lane == 0) sel[0] = P[tix];
  float cur = key_d(P[tix]);
  uint32_t pid = key_id(P[tix]);
  ++tix;
  // the first round's candidates; entries repeating p's id are invalidated uncounted
  int nl = 0;
  for (int base = tix; base < L; base += TG_WAVE) {
    const int i = base + lane;
    const uint32_t id = i < L ? key_id(P[i]) : TG_INV;
    bool live = id != TG_INV;
    if (live && id == pid) {
      P[i] = key_with_id(P[i], TG_INV);
      live = false;
    }
    const uint64_t m = ballot(live);
    if (live) cl[nl + mask_rank(m)] = uint16_t(i);
    nl += __popcll(m);
  }
  __syncthreads();
  while (nsel < FD) {
    const int cnt = nl;  // this round's candidates cl[0..cnt)
    Row16<MC> prow;
    const long long e0 = pclock(ph);
    load_row16<MC>(prow, reinterpret_cast<const T*>(a.rows) + size_t(pid) * D, D, t);
    eval_batch<MC>(reinterpret_cast<const T*>(a.rows), D, prow, cnt, [&](int q) { return key_id(P[cl[q]]); },
                   [&](int q, float res) {
                     const int i = cl[q];
                     const uint64_t k = P[i];
                     if (rule_eval(rule, res, key_d(k), cur, a.th) < 0.0f)
                       P[i] = key_with_id(k, TG_INV);
                   });
    padd(ph, ph.ev, pclock(ph) - e0);
    n_eval += cnt;
    __syncthreads();
    // the next selection is the first survivor; the survivors after it are the next round's
    // candidates
    int pi;
    nl = advance_cl(P, cl, 0, cnt, pi);
    if (pi >= 0) {
      if (lane == 0) sel[nsel] = P[pi];
      cur = key_d(P[pi]);
      pid = key_id(P[pi]);
      tix = pi;
    } else {
      tix = L;
    }
    ++nsel;  // an exhausted pool appends a placeholder, dropped below
    ++tix;
    __syncthreads();
    if (tix >= L) break;
  }
  return nsel - 1;  // the last appended entry is never kept (Tagore_src.cu:1462-1477)
}

// -------------------------------------------------------------------------------------
// The same Filter with the distances on the matrix cores, up to 16 rounds at a time: the next
// 16 live candidates are the rows of 16 x 16 products against every live candidate's row,
// which is read once for all of them (one round, or two, per read before: long live lists were
// bound by the row reads).  Whether row i's rule kills column j does not depend on which rows
// are selected, so each column gets a 16-bit mask of its killers; the selections among the 16
// rows follow from their own masks in order, and a column survives when its mask holds no
// selected row.  Rounds, selections and evaluation counts are those of one round at a time: a
// column counts for every selection before it up to its first killer (a killer that repeats
// its id is not an evaluation).
//   u8 rows (int8 MFMA): the distances are exact.
//   16-bit copy (a.Xb): s +- kap (|p|^2 + |c|^2) brackets the canonical distance and the rules
//   are monotone in it, so equal verdicts at both ends are the verdict; other pairs of a
//   selected row are queued and evaluated canonically from a.rows.
// A lane loads 16 bytes of row t = lane & 15 per step of 64 bytes, straight into the operand
// layout; KS steps.
// k_forward / k_reverse, before and after: Vamana (alpha 1.2, 12.8 k evaluations per node) over
// 400k x 128 u8 rows 51.1 -> 18.3 / 4.98 -> 1.36 ms, over 160k x 96 real-valued rows 22.5 -> 5.5 /
// 3.16 -> 0.67 ms; NSG over 1M x 128 u8 rows 34.3 -> 31.9 / 3.29 -> 1.77 ms; two-hop with angles
// over 300k x 96 13.8 -> 8.8 / 3.26 -> 1.06 ms.  Now bound by the chain of a block (its rows, its
// own columns, the tiles' loads), not by the products.
// LDS: cl and km [L + 16] (live pool indices, killer masks), queue [FQ_CAP] (16-bit copy).
// -------------------------------------------------------------------------------------
typedef int i32x4 __attribute__((ext_vector_type(4)));
constexpr int FQ_CAP = 512;

// Verdict of the rule for a distance in [lo, hi]: 1 below zero, 0 not, 2 undecided.  rule 0 is
// evaluated at both ends.  rule 1 (angle): th - ((dis + cur) - res) / 2 / sqrt(dis cur) < 0 where
// res < T = dis + cur - 2 th sqrt(dis cur); its roundings and those of T here move the border by
// less than (1 + |th|)(dis + cur) 2^-20, as long as dis cur is a normal number.
__device__ __forceinline__ int rule_bracket(int rule, float lo, float hi, float dis, float cur,
                                            float th) {
  if (rule == 0) {
    const float a = th * lo - dis, b = th * hi - dis;
    return (a < 0.0f && b < 0.0f) ? 1 : (a >= 0.0f && b >= 0.0f) ? 0 : 2;
  }
  const float dc = dis * cur, sum = dis + cur;
  if (!(dc > 1e-30f && dc < 1e37f)) return 2;
  const float T = __builtin_fmaf(-2.0f * th, __builtin_amdgcn_sqrtf(dc), sum);
  const float sl = (1.0f + fabsf(th)) * sum * 0x1p-20f;
  return hi < T - sl ? 1 : lo > T + sl ? 0 : 2;
}

template <int MC, class T, class Ph>
__device__ __forceinline__ int filter_pool_mfma(const PruneArgs& a, const uint64_t* P, int L,
                                                uint32_t u, int rule, uint64_t* sel,
                                                uint16_t* cl, uint16_t* km, uint16_t* queue,
                                                uint32_t& n_eval, Ph& ph) {
  constexpr bool U8 = std::is_same<T, uint8_t>::value;
  constexpr int KS = U8 ? MC : 2 * MC;  // 64-byte steps of a row
  constexpr int ESZ = U8 ? 1 : 2;
  using Acc = typename std::conditional<U8, i32x4, f32x4>::type;
  const int lane = threadIdx.x, t = lane & 15, g = lane >> 4;
  const int D = a.D;
  const float th = a.th;
  const unsigned char* X8 = U8 ? reinterpret_cast<const unsigned char*>(a.rows)
                               : reinterpret_cast<const unsigned char*>(a.Xb);
  const int tix = next_valid(P, 0, L, u);
  if (tix >= L || a.FD < 2) return 0;
  const int rounds = int(a.FD) - 1;  // the last appended entry is never kept
  // the live list: the first selection and every valid entry after it
  int cnt = 0;
  for (int base = tix; base < L; base += TG_WAVE) {
    const int i = base + lane;
    const bool live = i < L && key_id(P[i]) != TG_INV;
    const uint64_t m = ballot(live);
    if (live) cl[cnt + mask_rank(m)] = uint16_t(i);
    cnt += __popcll(m);
  }
  __syncthreads();

  auto load_row = [&](uint4 (&f)[KS], uint32_t id) {
    const unsigned char* x = X8 + size_t(id) * (D * ESZ);
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      f[k] = make_uint4(0u, 0u, 0u, 0u);
      if constexpr (U8) {
        if (64 * k < D) f[k] = load_u8x16(x, k, D, g);
      } else {
        if (32 * k + 8 * g < D) f[k] = *reinterpret_cast<const uint4*>(x + 64 * k + 16 * g);
      }
    }
  };
  auto product = [&](const uint4 (&x)[KS], const uint4 (&y)[KS]) {
    Acc c = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      if (k * 64 >= D * ESZ) break;
      if constexpr (U8) {
        c = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, x[k]),
                                                  __builtin_bit_cast(i32x4, y[k]), c, 0, 0, 0);
      } else if (a.h_bf16) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x[k]),
                                                    __builtin_bit_cast(bf16x8, y[k]), c, 0, 0, 0);
      } else {
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x[k]),
                                                   __builtin_bit_cast(f16x8, y[k]), c, 0, 0, 0);
      }
    }
    return c;
  };
  // |x|^2 of the lane's row t (u8: of the signed bytes), in every lane of that row
  auto norm_u8 = [&](const uint4 (&f)[KS]) {
    int s = 0;
#pragma unroll
    for (int k = 0; k < KS; ++k) s = dot16_u8(f[k], f[k], s);
    s += int(lane_xor32(uint32_t(s), 16));
    return s + int(lane_xor32(uint32_t(s), 32));
  };
  auto or_groups = [&](uint32_t m) {
    m |= lane_xor32(m, 16);
    return m | lane_xor32(m, 32);
  };

  int kept = 0;
  while (kept < rounds && cnt > 0) {
    const int nb = min(16, cnt);
    const long long e0 = pclock(ph);
    // row t of the block in the lanes t + 16 g; rows past nb repeat row 0, their bits masked
    const uint64_t krow = P[cl[t < nb ? t : 0]];
    const uint32_t idt = key_id(krow);
    uint4 fr[KS];
    load_row(fr, idt);
    float nf = 0.f;  // |x|^2 of row t
    int ni = 0;
    if constexpr (U8) ni = norm_u8(fr);
    else nf = a.nrm2[idt];
    // rows 4g + r, as the products hold them
    uint32_t rid[4];
    float rcur[4], rnf[4];
    int rni[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      rid[r] = uint32_t(__shfl(int(idt), 4 * g + r, TG_WAVE));
      rcur[r] = __shfl(key_d(krow), 4 * g + r, TG_WAVE);
      if constexpr (U8) rni[r] = __shfl(ni, 4 * g + r, TG_WAVE);
      else rnf[r] = __shfl(nf, 4 * g + r, TG_WAVE);
    }
    int qn = 0;  // queued pairs
    // killer bits of column (key kc, norm) from its products; `rows`: the rows that matter;
    // undecided pairs are queued under column number col
    auto kill_bits = [&](const Acc& c, uint64_t kc, float cnf, int cni, uint32_t rows, int col) {
      const float dis = key_d(kc);
      const uint32_t cid = key_id(kc);
      uint32_t nib = 0, und = 0;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (U8) {
          const float res = float(rni[r] + cni - 2 * c[r]);
          if (rule == 0) {
            nib |= (th * res - dis < 0.0f) ? 1u << r : 0u;
          } else {
            const int v = rule_bracket(1, res, res, dis, rcur[r], th);
            nib |= v == 1 ? 1u << r : 0u;
            und |= v == 2 ? 1u << r : 0u;
          }
        } else {
          const float nsum = rnf[r] + cnf;
          const float s = __builtin_fmaf(-a.pscale, c[r], nsum);
          const int v = rule_bracket(rule, __builtin_fmaf(-a.kap, nsum, s),
                                     __builtin_fmaf(a.kap, nsum, s), dis, rcur[r], th);
          nib |= v == 1 ? 1u << r : 0u;
          und |= v == 2 ? 1u << r : 0u;
        }
        if (rid[r] == cid) {  // a repeated id is dropped whatever its distance
          nib |= 1u << r;
          und &= ~(1u << r);
        }
      }
      und &= rows >> (4 * g);
      if (ballot((und & 15u) != 0) != 0) {
        if constexpr (U8) {  // the distances are exact: the rule itself
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float res = float(rni[r] + cni - 2 * c[r]);
            if (((und >> r) & 1u) && rule_eval(rule, res, dis, rcur[r], th) < 0.0f) nib |= 1u << r;
          }
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bool q = (und >> r) & 1u;
            const uint64_t m = ballot(q);
            if (q) queue[qn + mask_rank(m)] = uint16_t((4 * g + r) << 10 | col);
            qn += __popcll(m);
          }
        }
      }
      return or_groups((nib & 15u) << (4 * g)) & rows;
    };
    // canonical distances of the queued pairs, one per 16-lane group (few, and a second pair's
    // registers would cost a wave per SIMD)
    auto flush = [&]() {
      if constexpr (!U8) {
        __syncthreads();
        const T* X = reinterpret_cast<const T*>(a.rows);
        for (int q0 = 0; q0 < qn; q0 += 4) {
          const int q = q0 + g;
          const uint32_t ent = queue[q < qn ? q : 0], i = ent >> 10, col = ent & 1023u;
          const uint64_t ki = P[cl[i]], kcol = P[cl[col]];
          const T* const ra[1] = {X + size_t(key_id(ki)) * D};
          const T* const rb[1] = {X + size_t(key_id(kcol)) * D};
          float dd[1];
          dist16_pairs<MC, 1>(ra, rb, D, t, dd);
          if (t == 0 && q < qn && rule_eval(rule, dd[0], key_d(kcol), key_d(ki), th) < 0.0f)
            atomicOr(reinterpret_cast<uint32_t*>(km) + (col >> 1), (1u << i) << (16 * (col & 1)));
        }
        qn = 0;
        __syncthreads();
      }
    };
    // ---- the block's own columns: row j is selected when no selected row kills it
    const uint32_t before = t < nb ? ((1u << t) - 1u) : 0u;
    uint32_t own = kill_bits(product(fr, fr), krow, nf, ni, before, t);
    if (qn) {
      if (g == 0) km[t] = uint16_t(own);
      flush();
      own = km[t];
    }
    // a selection at the pool's last position ends the filter unkept, but for the first one
    const bool at_end = int(cl[cnt - 1]) == L - 1;
    uint32_t chosen = 0;
    int n = kept;
    bool done = false;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const uint32_t mj = uint32_t(__builtin_amdgcn_readlane(int(own), j));
      if (j < nb && !done && (mj & chosen) == 0) {
        if (n == rounds || (at_end && j == cnt - 1 && n > 0)) done = true;
        else {
          chosen |= 1u << j;
          ++n;
        }
      }
    }
    if (g == 0) {
      km[t] = uint16_t(own);
      if ((chosen >> t) & 1u) sel[kept + __popc(chosen & before)] = krow;
    }
    kept = n;
    // ---- the other columns; u8: two tiles' rows in flight (16-bit rows take the registers)
    constexpr int TI = U8 ? 2 : 1;
    for (int c0 = 16; c0 < cnt; c0 += 16 * TI) {
      uint64_t kc[TI];
      uint4 fc[TI][KS];
      float nc[TI];
#pragma unroll
      for (int x = 0; x < TI; ++x) {
        const int c = c0 + 16 * x + t;
        kc[x] = P[cl[c < cnt ? c : 0]];
        load_row(fc[x], key_id(kc[x]));
        nc[x] = U8 ? 0.f : a.nrm2[key_id(kc[x])];
      }
      if (qn > FQ_CAP - 256) flush();
#pragma unroll
      for (int x = 0; x < TI; ++x) {
        const int c = c0 + 16 * x + t;
        const uint32_t m = kill_bits(product(fr, fc[x]), kc[x], nc[x], U8 ? norm_u8(fc[x]) : 0,
                                     c < cnt ? chosen : 0u, c);
        if (g == 0 && c < cnt) km[c] = uint16_t(m);
      }
    }
    if (qn) flush();
    else __syncthreads();
    padd(ph, ph.ev, pclock(ph) - e0);
    // ---- evaluations and the survivors, in order (in place: a chunk is read before any of
    // its entries is written, and writes land at or below it)
    int live = 0;
    uint32_t ev = 0;
    for (int base = 0; base < cnt; base += TG_WAVE) {
      const int c = base + lane;
      const bool in = c < cnt;
      const uint32_t idx = in ? cl[c] : 0u;
      const uint32_t rows = c < 16 ? chosen & ((1u << c) - 1u) : chosen;
      const uint32_t k = in ? km[c] & rows : 0u;
      const int f = k ? __ffs(k) - 1 : 0;
      const uint32_t fid = uint32_t(__shfl(int(idt), f, TG_WAVE));
      if (in) {
        ev += k ? __popc(rows & ((1u << f) - 1u)) + (fid != key_id(P[idx]) ? 1u : 0u)
                : __popc(rows);
      }
      const bool alive = in && k == 0 && !(c < 16 && ((chosen >> c) & 1u));
      const uint64_t m = ballot(alive);
      __syncthreads();
      if (alive) cl[live + mask_rank(m)] = uint16_t(idx);
      live += __popcll(m);
      __syncthreads();
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ev += uint32_t(__shfl_xor(int(ev), o, TG_WAVE));
    n_eval += ev;
    cnt = live;
    if (done) break;
  }
  return kept;
}

__device__ __forceinline__ void count_add(unsigned long long* c, int idx, uint32_t v) {
  if (c && threadIdx.x == 0 && v) atomicAdd(&cnt_slot(c)[idx], (unsigned long long)v);
}

// -------------------------------------------------------------------------------------
// Forward pass (Collect + Filter + Store reverse pushes).  kind 0: path, 1: two-hop.
//
// LDS (dynamic, sized from K, TOPM and FD so that more workgroups fit a CU):
//   during the beam: the 480-slot ring (its sort pads it to 512 in registers), then S | tab |
//       beam compaction indices;
//   afterwards: the pool (K + 480 keys, over the ring and the dead start of the beam's
//       scratch), then the selected list and the filter's lists.
// The pool is the merge of the sorted own list and the sorted ring, formed in registers as
// one bitonic merge of [own list ascending | +inf | ring descending] (1024 slots); it is
// the sequence a sort of their union gives.
// -------------------------------------------------------------------------------------
constexpr int RING_P = 512;

struct FwdLayout {
  int W, NS, L, HB, offB, offF, bytes;
};
// mf: filter_pool_mfma; queue: its re-score queue (16-bit copy); beam: the path's Collect
__host__ __device__ inline FwdLayout fwd_layout(uint32_t N, int K, int TOPM, int FD, bool mf,
                                                bool queue, bool beam) {
  FwdLayout l;
  l.W = (K <= 64 && TOPM <= 64) ? 1 : 2;
  l.NS = 64 * l.W;
  l.L = K + RING;
  l.HB = hs_bits(l.W, N, TOPM + K, mf);
  l.offB = RING * 8;
  l.offF = ((l.L > RING_P ? l.L : RING_P) * 8 + 15) / 16 * 16;
  const int coll = beam ? l.offB + l.NS * 8 + hs_words(l.HB) * 4 + l.NS * 2 : l.offB;
  // the filter's selection, live list, killer masks and re-score queue
  const int lists = (l.L + 17) * 2;
  const int filt = l.offF + (FD + 1) * 8 + (mf ? 2 * lists : lists) + (queue ? FQ_CAP * 2 : 0);
  l.bytes = ((coll > filt ? coll : filt) + 15) / 16 * 16;
  return l;
}

// mfma: filter_pool_mfma on the 16-bit copy (u8 rows always take it).
// Ph: PhaseOn in profiling runs.
template <int MC, class T, int KIND, int W, bool MF, class Ph>
// Waves per SIMD, chosen at 96 and 128 elements: six (80 VGPRs; 0 to 6 spilled) for u8 rows, five
// for 16-bit rows (11 to 15 spilled).  Rows of 129 to 256 elements took the next step down
// unmeasured: three for 16-bit rows spill nothing, five for u8 rows spill 40 to 55 registers in
// the path's kernels (four: 2 at most, Vamana over 100k x 160 6.09 -> 4.82 ms).
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(MC == 2 ? (std::is_same<T, uint8_t>::value || !MF ? 6 : 5)
                                           : (MC == 4 ? (std::is_same<T, uint8_t>::value ? 5 : 3) : 2))))
void k_forward(PruneArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char dsm[];
  const uint32_t u = row_of_block(a.perm, a.N);
  if (u >= a.N) return;
  const int lane = threadIdx.x, t = lane & 15;
  const int K = a.K, D = a.D;
  const FwdLayout ly = fwd_layout(a.N, K, int(a.TOPM), int(a.FD), MF,
                                  MF && !std::is_same<T, uint8_t>::value, KIND == 0);
  uint64_t* R = reinterpret_cast<uint64_t*>(dsm);
  uint64_t* P = R;  // after the pool is formed
  uint64_t* S = reinterpret_cast<uint64_t*>(dsm + ly.offB);
  uint32_t* tab = reinterpret_cast<uint32_t*>(S + ly.NS);
  const int hb = hs_bits(W, a.N, K + int(a.TOPM), MF);  // ly.HB, a constant in most kernels
  uint16_t* clb = reinterpret_cast<uint16_t*>(tab + hs_words(hb));
  uint64_t* sel = reinterpret_cast<uint64_t*>(dsm + ly.offF);  // after the beam
  uint16_t* cl = reinterpret_cast<uint16_t*>(sel + a.FD + 1);
  uint16_t* km = cl + ((ly.L + 17) & ~1);
  uint16_t* fq = km + ((ly.L + 17) & ~1);
  const int L = ly.L;
  Row16<MC> xu;
  load_row16<MC>(xu, reinterpret_cast<const T*>(a.rows) + size_t(u) * D, D, t);
  for (int i = lane; i < RING; i += TG_WAVE) R[i] = mk_key(__uint_as_float(0x7F800000u), TG_INV);
  __syncthreads();
  uint32_t n_col = 0, n_adj = 0, n_flt = 0;
  Ph ph;
  const long long c0 = pclock(ph);
  if (KIND == 0) {
    uint32_t ring_c = 0;
    const uint32_t ep = a.ep[a.seg_of ? a.seg_of[u] : 0];
    beam_search<MC, T, W>(a, xu, ep, 10, S, tab, hb, clb, R, nullptr, ring_c, n_col,
                          n_adj, ph);
  } else {
    // two-hop ids y_i = G[G[u][i/K]][i%K], i < 480
    for (int i = lane; i < RING; i += TG_WAVE) {
      const uint32_t v = a.G[size_t(u) * K + i / K];
      R[i] = mk_key(0.f, a.G[size_t(v) * K + (i % K)]);
    }
    __syncthreads();
    eval_batch<MC>(reinterpret_cast<const T*>(a.rows), D, xu, RING, [&](int q) { return key_id(R[q]); },
                   [&](int q, float d) { R[q] = mk_key(d, key_id(R[q])); });
    n_col = RING;
    n_adj = (RING + K - 1) / K;
  }
  __syncthreads();
  const long long c1 = pclock(ph);
  // pool = merge(own list, sorted ring), in registers; the own list is a kNN row, sorted by
  // (distance, id) already (builds keep them so, tg_set_knn rejects others)
  uint64_t pv[16];
  {
    uint64_t o[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int j = r * 64 + lane;
      o[r] = j < K ? mk_key(a.GD[size_t(u) * K + j], a.G[size_t(u) * K + j]) : TG_KEY_INF;
    }
    uint64_t rr[RING_P / 64];
#pragma unroll
    for (int q = 0; q < RING_P / 64; ++q)
      rr[q] = q * 64 + lane < RING ? R[q * 64 + lane] : TG_KEY_INF;
    reg_bitonic<RING_P / 64, uint64_t, true>(rr);
    pv[0] = o[0];
    pv[1] = o[1];
#pragma unroll
    for (int q = 2; q < 8; ++q) pv[q] = TG_KEY_INF;
#pragma unroll
    for (int q = 0; q < 8; ++q) pv[8 + q] = rr[q];
  }
  const long long c1s = pclock(ph);
  reg_bitonic_merge<16>(pv);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 16; ++q)
    if (q * 64 + lane < L) P[q * 64 + lane] = pv[q];
  __syncthreads();
  // entries repeating their predecessor's id get id INV
  constexpr int PQ = (128 + RING + TG_WAVE - 1) / TG_WAVE;
  bool dup[PQ];
#pragma unroll
  for (int q = 0; q < PQ; ++q) {
    const int i = q * TG_WAVE + lane;
    dup[q] = (i < L && i > 0) ? (key_id(P[i]) == key_id(P[i - 1])) : false;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PQ; ++q)
    if (dup[q]) P[q * TG_WAVE + lane] = key_with_id(P[q * TG_WAVE + lane], TG_INV);
  __syncthreads();
  const long long c2 = pclock(ph);
  int deg;
  if constexpr (MF) deg = filter_pool_mfma<MC, T>(a, P, L, u, a.fwd_rule, sel, cl, km, fq, n_flt, ph);
  else deg = filter_pool<MC, T>(a, P, L, u, a.fwd_rule, sel, cl, n_flt, ph);
  __syncthreads();
  if (Ph::on && lane == 0 && a.counters) {
    const long long c3 = pclock(ph);
    atomicAdd(&cnt_slot(a.counters)[6], (unsigned long long)(c1 - c0));
    atomicAdd(&cnt_slot(a.counters)[7], (unsigned long long)(c3 - c2));
    atomicAdd(&cnt_slot(a.counters)[8], (unsigned long long)(c2 - c1));
    atomicAdd(&cnt_slot(a.counters)[9], (unsigned long long)ph.ev);
    for (int i = 0; i < 4; ++i) atomicAdd(&cnt_slot(a.counters)[10 + i], (unsigned long long)ph.sub[i]);
    atomicAdd(&cnt_slot(a.counters)[14], (unsigned long long)(c1s - c1));
  }
  for (int k = lane; k < deg; k += TG_WAVE) {
    const uint64_t s = sel[k];
    a.fwd_ids[size_t(u) * a.FD + k] = key_id(s);
    a.fwd_d[size_t(u) * a.FD + k] = key_d(s);
    pb_push(a.rev, key_id(s), mk_key(key_d(s), u));
  }
  if (lane == 0) a.fwd_deg[u] = deg;
  count_add(a.counters, 0, n_col);
  count_add(a.counters, 1, n_flt);
  count_add(a.counters, 3, n_adj);
}

// -------------------------------------------------------------------------------------
// Reverse pass (filter_reverse, spec A.7): forward list plus the K best reverse pushes;
// re-filtered with the reverse rule when more than FD, otherwise their union.
// -------------------------------------------------------------------------------------
template <int MC, class T, bool MF>
__global__ __launch_bounds__(64) void k_reverse(PruneArgs a) {
  __shared__ uint64_t buf[256];
  __shared__ uint64_t P[256];
  __shared__ __attribute__((aligned(4))) uint16_t cl[272], km[MF ? 272 : 2];
  __shared__ uint16_t fq[MF && !std::is_same<T, uint8_t>::value ? FQ_CAP : 1];
  __shared__ uint64_t sel[129];
  const uint32_t u = row_of_block(a.perm, a.N);
  if (u >= a.N) return;
  const int lane = threadIdx.x;
  const int K = a.K, FD = a.FD;
  const int nr = pb_top(a.rev, u, pb_count(a.rev, u), K, false, [](uint64_t) { return true; }, buf);
  const int deg = a.fwd_deg[u];
  const int L = deg + nr;
  uint32_t* row = a.out_ids + size_t(u) * FD;
  uint32_t n_flt = 0;
  if (L > FD) {
    const int n = pow2_at_least(max(L, TG_WAVE));  // L <= FD + K <= 256
    if (n == 64) merge_pool<1>(a, u, deg, buf, nr, P);
    else if (n == 128) merge_pool<2>(a, u, deg, buf, nr, P);
    else merge_pool<4>(a, u, deg, buf, nr, P);
    mark_dups(P, n);
    PhaseOff ph;  // not reported for the reverse pass
    int nd;
    if constexpr (MF) nd = filter_pool_mfma<MC, T>(a, P, L, u, a.rev_rule, sel, cl, km, fq, n_flt, ph);
    else nd = filter_pool<MC, T>(a, P, L, u, a.rev_rule, sel, cl, n_flt, ph);
    __syncthreads();
    for (int k = lane; k < FD; k += TG_WAVE) row[k] = k < nd ? key_id(sel[k]) : TG_INV;
    if (lane == 0) a.out_deg[u] = nd;
  } else {
    // union: forward ids in order, then reverse ids (R order) not already present
    const uint32_t* f = a.fwd_ids + size_t(u) * FD;
    for (int k = lane; k < deg; k += TG_WAVE) row[k] = f[k];
    bool add = false;
    uint32_t w = 0;
    if (lane < nr) {
      w = key_id(buf[lane]);
      add = true;
      for (int j = 0; j < deg; ++j) add = add && (f[j] != w);
    }
    // nr <= L <= FD <= 128; handle lanes 64..127 in a second step
    const uint64_t m0 = ballot(add);
    if (add) row[deg + mask_rank(m0)] = w;
    int n = deg + __popcll(m0);
    if (nr > TG_WAVE) {
      bool add2 = false;
      uint32_t w2 = 0;
      if (TG_WAVE + lane < nr) {
        w2 = key_id(buf[TG_WAVE + lane]);
        add2 = true;
        for (int j = 0; j < deg; ++j) add2 = add2 && (f[j] != w2);
      }
      const uint64_t m1 = ballot(add2);
      if (add2) row[n + mask_rank(m1)] = w2;
      n += __popcll(m1);
    }
    for (int k = n + lane; k < FD; k += TG_WAVE) row[k] = TG_INV;
    if (lane == 0) a.out_deg[u] = n;
  }
  count_add(a.counters, 2, n_flt);
}

// -------------------------------------------------------------------------------------
// One-hop rank (CAGRA: id membership; DPG: occlusion by distance), spec A.8 / A.9.
// -------------------------------------------------------------------------------------
// The d = FD entries of smallest (detour count, id) of node u and their reverse pushes.
// det / nei: the counts and ids by list position; srt: 128 keys of scratch.
__device__ __forceinline__ void rank_select(const PruneArgs& a, uint32_t u, const uint32_t* det,
                                            const uint32_t* nei, uint64_t* srt) {
  const int lane = threadIdx.x, K = a.K, d = a.FD;
  const int n = pow2_at_least(K);
  for (int j = lane; j < n; j += TG_WAVE)
    srt[j] = j < K ? ((uint64_t(det[j]) << 32) | nei[j]) : TG_KEY_INF;
  __syncthreads();
  wave_sort<128>(srt, n);
  for (int i = lane; i < d; i += TG_WAVE) {
    const uint64_t k = srt[i];
    a.fwd_ids[size_t(u) * d + i] = uint32_t(k);
    pb_push(a.rev, uint32_t(k), (k & 0xFFFFFFFF00000000ull) | u);
  }
  if (lane == 0) a.fwd_deg[u] = d;
}

// CAGRA: neighbour j of u gets one detour per earlier neighbour r < j whose list holds j.
// K rows of K ids are looked up per node, so the lookups' instructions set the time.  u's ids
// sit in an LDS hash of 256 buckets of four 32-bit entries: an id is its bucket and the 24
// bits id >> 8 (the bucket adds a function of those bits to the low byte, so the two give
// the id back), and an entry packs these bits and the id's list position.  A lookup is one
// 16-byte read and four subtract-and-compares, which test the id and j > r at once, with no
// loop; ids that find their bucket full (0.01 per node at K = 96) are tested one by one.
// VEC ids per lane and load (16 bytes where rows are 16-byte aligned, K % 4 == 0), the rows'
// id groups dealt to the lanes as one flat sequence, two groups in flight per lane.
// 500k x K = 96: 9.84 -> 2.91 ms (seven-step binary searches of the
// sorted ids before; 75 % of VALU issue now, LDS reads busy 65 %).
constexpr int CAGRA_BUCKETS = 256;
__device__ __forceinline__ uint32_t cagra_bucket(uint32_t id) {
  return (((id >> 8) * 0x9E3779u + (id << 16)) >> 16) & (CAGRA_BUCKETS - 1);
}
__device__ __forceinline__ uint32_t cagra_entry(uint32_t id, uint32_t pos) {
  return (id >> 8) << 7 | pos;
}
template <int VEC>
__global__ __launch_bounds__(64) void k_cagra_forward(PruneArgs a) {
  __shared__ __attribute__((aligned(16))) uint32_t tab[CAGRA_BUCKETS * 4];
  __shared__ uint32_t ovid[128], ovpos[128];  // ids of full buckets
  __shared__ uint32_t novf;
  __shared__ uint64_t srt[128];  // row offsets of the neighbours, then the selection's keys
  __shared__ uint32_t det[128];
  __shared__ uint32_t nei[128];
  const uint32_t u = row_of_block(a.perm, a.N);
  if (u >= a.N) return;
  const int lane = threadIdx.x, K = a.K;
  for (int i = lane; i < CAGRA_BUCKETS * 4; i += TG_WAVE) tab[i] = TG_INV;
  for (int j = lane; j < 128; j += TG_WAVE) {
    det[j] = 0;
    nei[j] = j < K ? a.G[size_t(u) * K + j] : TG_INV;
    srt[j] = uint64_t(nei[j]) * uint32_t(K) * 4;
  }
  if (lane == 0) novf = 0;
  __syncthreads();
  for (int j = lane; j < K; j += TG_WAVE) {
    uint32_t* b = tab + 4 * cagra_bucket(nei[j]);
    const uint32_t e = cagra_entry(nei[j], uint32_t(j));
    int q = 0;
    while (q < 4 && atomicCAS(&b[q], TG_INV, e) != TG_INV) ++q;
    if (q == 4) {
      const uint32_t o = atomicAdd(&novf, 1u);
      ovid[o] = nei[j];
      ovpos[o] = uint32_t(j);
    }
  }
  __syncthreads();
  const int nov = int(novf);
  // an id listed twice counts at its first position only (rows given by a caller may repeat
  // one); a position 0 never counts, so a later copy in the overflow list takes that
  for (int j0 = 0; j0 < K; j0 += TG_WAVE) {
    const int j = j0 + lane;
    bool dup = false;
    if (j < K) {
      const uint32_t id = nei[j], none = cagra_entry(id, 0u);
      const uint4 v = *reinterpret_cast<const uint4*>(tab + 4 * cagra_bucket(id));
      dup = v.x - none < uint32_t(j) || v.y - none < uint32_t(j) || v.z - none < uint32_t(j) ||
            v.w - none < uint32_t(j);
      for (int o = 0; o < nov; ++o) dup = dup || (ovid[o] == id && int(ovpos[o]) < j);
    }
    __syncthreads();
    if (dup) {
      uint32_t* b = tab + 4 * cagra_bucket(nei[j]);
      for (int q = 0; q < 4; ++q)
        if (b[q] == cagra_entry(nei[j], uint32_t(j))) b[q] = TG_INV;
      for (int o = 0; o < nov; ++o)
        if (ovid[o] == nei[j] && int(ovpos[o]) == j) ovpos[o] = 0;
    }
    __syncthreads();
  }
  // groups of VEC ids, row by row; the last row has no later neighbour
  const int per = K / VEC, total = (K - 1) * per;
  const int dr = TG_WAVE / per, dc = TG_WAVE - dr * per;  // TG_WAVE groups further on
  int r = lane / per, c = lane - r * per;
  const char* G = reinterpret_cast<const char*>(a.G);
  auto row_group = [&](uint32_t (&y)[VEC]) {
    const char* p = G + srt[r] + uint32_t(c) * (VEC * 4);
    if constexpr (VEC == 4) {
      const uint4 q = *reinterpret_cast<const uint4*>(p);
      y[0] = q.x; y[1] = q.y; y[2] = q.z; y[3] = q.w;
    } else {
      y[0] = *reinterpret_cast<const uint32_t*>(p);
    }
  };
  auto advance = [&]() {
    r += dr;
    c += dc;
    if (c >= per) {
      c -= per;
      ++r;
    }
  };
  auto look_up = [&](const uint32_t (&y)[VEC], uint32_t r1) {  // r1 = r + 1
    uint4 v[VEC];
#pragma unroll
    for (int q = 0; q < VEC; ++q)
      v[q] = *reinterpret_cast<const uint4*>(tab + 4 * cagra_bucket(y[q]));
#pragma unroll
    for (int q = 0; q < VEC; ++q) {
      // entry - base is pos - (r + 1) when the ids are equal, which is below 127 - r for
      // r < pos <= 127; other ids differ by at least 128 - r - 1 from there (an empty entry
      // too), so the smallest difference of the bucket decides, and gives the position
      const uint32_t base = cagra_entry(y[q], 0u) + r1;
      const uint32_t m = min(min(v[q].x - base, v[q].y - base), min(v[q].z - base, v[q].w - base));
      if (m < 128u - r1) atomicAdd(&det[m + r1], 1u);
    }
    if (nov)
      for (int o = 0; o < nov; ++o)
#pragma unroll
        for (int q = 0; q < VEC; ++q)
          if (ovid[o] == y[q] && ovpos[o] >= r1) atomicAdd(&det[ovpos[o]], 1u);
  };
  for (int e = lane; e < total; e += 2 * TG_WAVE) {
    uint32_t ya[VEC], yb[VEC];
    const uint32_t ra = uint32_t(r) + 1;
    row_group(ya);
    advance();
    const bool second = e + TG_WAVE < total;
    const uint32_t rb = uint32_t(r) + 1;
    if (second) row_group(yb);
    advance();
    look_up(ya, ra);
    if (second) look_up(yb, rb);
  }
  count_add(a.counters, 3, K);
  __syncthreads();
  rank_select(a, u, det, nei, srt);
}

template <int MC, class T>
__global__ __launch_bounds__(64) void k_dpg_forward(PruneArgs a) {
  __shared__ uint64_t srt[128];
  __shared__ uint32_t det[128];
  __shared__ uint32_t nei[128];
  const uint32_t u = row_of_block(a.perm, a.N);
  if (u >= a.N) return;
  const int lane = threadIdx.x, g = lane >> 4, t = lane & 15;
  const int K = a.K, D = a.D;
  for (int j = lane; j < 128; j += TG_WAVE) {
    det[j] = 0;
    nei[j] = j < K ? a.G[size_t(u) * K + j] : TG_INV;
  }
  __syncthreads();
  // pairs r < j, row by row; the four groups take every fourth j of a row
  const int npairs = K * (K - 1) / 2;
  for (int r = 0; r + 1 < K; ++r) {
    const T* xr = reinterpret_cast<const T*>(a.rows) + size_t(nei[r]) * D;
    for (int j = r + 1 + g; j < K; j += 4) {
      const float dd =
          dist16_mm<MC>(xr, reinterpret_cast<const T*>(a.rows) + size_t(nei[j]) * D, D, t);
      if (t == 0 && dd < a.GD[size_t(u) * K + j]) atomicAdd(&det[j], 1u);
    }
  }
  count_add(a.counters, 1, npairs);
  __syncthreads();
  rank_select(a, u, det, nei, srt);
}

// filter_reverse_1hop (spec A.10): half forward, up to half reverse, forward fill.  The
// reverse entries w that the first `lim` forward ids do not name follow the forward half, in
// (detour, id) order.  One reverse entry per lane (two past 64), its membership a scan of the
// forward ids broadcast from LDS; the whole pass was lane 0's serial insertion sorts and
// scans before (500k x FD = 32: 7.37 -> 0.65 ms).
__global__ __launch_bounds__(64) void k_rank_reverse(PruneArgs a) {
  __shared__ uint64_t buf[256];
  __shared__ uint32_t T[128];
  const uint32_t u = blockIdx.x;
  if (u >= a.N) return;
  const int lane = threadIdx.x;
  const int d = a.FD, h = d / 2;
  const uint32_t np = pb_count(a.rev, u);
  for (int i = lane; i < 128; i += TG_WAVE)
    T[i] = i < d ? a.fwd_ids[size_t(u) * d + i] : TG_INV;
  // R1[u]: the d smallest (detour, src) pushes, already sorted by (detour, id)
  const int r = pb_top(a.rev, u, np, d, false, [](uint64_t) { return true; }, buf);
  uint32_t* row = a.out_ids + size_t(u) * d;
  // Later copies of a source get detour INV and go last, by id.  Sources repeat only where a
  // given kNN row lists an id twice.
  bool any = false;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int i = q * TG_WAVE + lane;
    const uint32_t id = uint32_t(buf[i]);
    bool dup = false;
    const int top = min(r, (q + 1) * TG_WAVE);
    if (top > q * TG_WAVE)
      for (int j = 0; j + 1 < top; ++j) dup = dup || (j < i && uint32_t(buf[j]) == id);
    dup = dup && i < r;
    any = any || ballot(dup) != 0;
    if (dup) buf[128 + i] = (uint64_t(TG_INV) << 32) | id;
    else if (i < r) buf[128 + i] = buf[i];
  }
  __syncthreads();
  if (any) {
    const int n = pow2_at_least(r);
    for (int i = lane; i < n; i += TG_WAVE) buf[i] = i < r ? buf[128 + i] : TG_KEY_INF;
    __syncthreads();
    wave_sort<128>(buf, n);
  }
  const int lim = (r < h) ? (d - r) : h;
  int na = 0;
  for (int base = 0; base < r; base += TG_WAVE) {
    const int i = base + lane;
    const uint32_t w = i < r ? uint32_t(buf[i]) : TG_INV;
    bool add = i < r;
    for (int j = 0; j < lim; ++j) add = add && T[j] != w;
    const uint64_t m = ballot(add);
    const int p = na + mask_rank(m);
    if (add && (r < h || p < h)) row[h + p] = w;
    na += int(__popcll(m));
  }
  if (r >= h) na = min(na, h);
  for (int i = lane; i < h; i += TG_WAVE) row[i] = T[i];
  for (int i = lane; h + na + i < d; i += TG_WAVE) row[h + na + i] = T[h + i];
  if (lane == 0) a.out_deg[u] = d;
}

// -------------------------------------------------------------------------------------
// Entry point (cal_ep_gpu, Tagore_src.cu:1889-2058): beam of TOPM from the first node's list
// toward the centroid; one workgroup per segment.
// -------------------------------------------------------------------------------------
template <int MC, class T>
__global__ __launch_bounds__(64) void k_cal_ep(PruneArgs a, const float* centroid, uint32_t* ep) {
  __shared__ uint64_t M0[128], S[128];
  __shared__ __attribute__((aligned(16))) uint32_t tab[hs_words(7)];
  __shared__ uint16_t cl[128];
  const uint32_t seg = blockIdx.x;
  const uint32_t start = a.seg_lo ? a.seg_lo[seg] : 0u;
  Row16<MC> c;
  load_row16<MC>(c, centroid + size_t(seg) * a.D, a.D, threadIdx.x & 15);
  uint32_t rc = 0, ne = 0, na = 0;
  PhaseOff ph;  // not reported for the entry point
  if (a.K <= 64 && a.TOPM <= 64)
    beam_search<MC, T, 1>(a, c, start, 30, S, tab, 7, cl, nullptr, M0, rc, ne, na, ph);
  else
    beam_search<MC, T, 2>(a, c, start, 30, S, tab, 7, cl, nullptr, M0, rc, ne, na, ph);
  if (threadIdx.x == 0) ep[seg] = key_id(M0[0]);
  count_add(a.counters, 4, ne);
}

// Deterministic centroid: FP64 sums over chunks of 1024 rows, then over chunks in order.
// The centroid's FP64 sums in index order (chunks of 1024 rows, then the chunk partials):
// each step loads 16 values together and adds them in order, so 16 loads are in flight per
// lane and the sums are the serial ones.
__global__ void k_centroid_part(const float* X, uint32_t N, uint32_t D, double* part) {
  const uint32_t j = blockIdx.y * blockDim.x + threadIdx.x;
  if (j >= D) return;
  const size_t lo = size_t(blockIdx.x) * 1024, hi = min(size_t(N), lo + 1024);
  double s = 0.0;
  size_t i = lo;
  for (; i + 16 <= hi; i += 16) {
    float v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = X[(i + q) * D + j];
#pragma unroll
    for (int q = 0; q < 16; ++q) s += double(v[q]);
  }
  for (; i < hi; ++i) s += double(X[i * D + j]);
  part[size_t(blockIdx.x) * D + j] = s;
}
__global__ void k_centroid_final(const double* part, uint32_t nch, uint32_t N, uint32_t D,
                                 float* c) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= D) return;
  double s = 0.0;
  uint32_t ch = 0;
  for (; ch + 16 <= nch; ch += 16) {
    double v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = part[size_t(ch + q) * D + j];
#pragma unroll
    for (int q = 0; q < 16; ++q) s += v[q];
  }
  for (; ch < nch; ++ch) s += part[size_t(ch) * D + j];
  c[j] = float(s / double(N));
}

// ------------------------------------------------------------------------- launchers
// The passes with a filter.
template <int MC, class T, bool MF>
static void launch_filter_mc(const PruneArgs& a, int phase, hipStream_t s) {
  const dim3 grid(grid_rows(a.perm, a.N)), block(64);
  const FwdLayout f = fwd_layout(a.N, a.K, a.TOPM, a.FD, MF, MF && !std::is_same<T, uint8_t>::value,
                                 phase == PH_FWD_PATH);
#define FWD(KIND, W)                                                                            \
  do {                                                                                         \
    if (a.phase_clock) k_forward<MC, T, KIND, W, MF, PhaseOn><<<grid, block, f.bytes, s>>>(a); \
    else k_forward<MC, T, KIND, W, MF, PhaseOff><<<grid, block, f.bytes, s>>>(a);              \
  } while (0)
  switch (phase) {
    case PH_FWD_PATH:
      if (f.W == 1) FWD(0, 1);
      else FWD(0, 2);
      break;
    case PH_FWD_2HOP: FWD(1, 1); break;
    default: k_reverse<MC, T, MF><<<grid, block, 0, s>>>(a); break;
  }
#undef FWD
}

template <class T>
static void launch_prune_t(const PruneArgs& a, int phase, const float* centroid, uint32_t* ep,
                           hipStream_t s, uint32_t nseg) {
  const int mc = (a.D + 63) / 64;
#define PR_MC(CALL)                       \
  do {                                    \
    if (mc <= 2) CALL(2);                 \
    else if (mc <= 4) CALL(4);            \
    else CALL(16);                        \
  } while (0)
#define PR_EP(M) k_cal_ep<M, T><<<nseg, 64, 0, s>>>(a, centroid, ep)
#define PR_DPG(M) k_dpg_forward<M, T><<<grid_rows(a.perm, a.N), 64, 0, s>>>(a)
#define PR_FLT(M) launch_filter_mc<M, T, false>(a, phase, s)
  if (phase == PH_EP) PR_MC(PR_EP);
  else if (phase == PH_DPG) PR_MC(PR_DPG);
  // the 16-bit copy, rows up to 256 elements (operands of wider rows do not stay in registers)
  else if (a.Xb && mc <= 2) launch_filter_mc<2, T, true>(a, phase, s);
  else if (a.Xb && mc <= 4) launch_filter_mc<4, T, true>(a, phase, s);
  else PR_MC(PR_FLT);
#undef PR_FLT
#undef PR_DPG
#undef PR_EP
#undef PR_MC
}

void launch_prune(const PruneArgs& a, int phase, const float* centroid, uint32_t* ep,
                  hipStream_t s, uint32_t nseg) {
  if (phase == PH_CAGRA) {  // ids only
    if (a.K % 4 == 0) k_cagra_forward<4><<<grid_rows(a.perm, a.N), 64, 0, s>>>(a);
    else k_cagra_forward<1><<<grid_rows(a.perm, a.N), 64, 0, s>>>(a);
    return;
  }
  if (phase == PH_RANK_REV) {
    k_rank_reverse<<<a.N, 64, 0, s>>>(a);
    return;
  }
  // (rows up to 256 values: wider u8 batches would not stay in registers)
  if (a.rows8 && a.D <= 256 && (phase == PH_FWD_PATH || phase == PH_FWD_2HOP || phase == PH_REV)) {
    PruneArgs b = a;
    b.rows = a.rows8;
    b.rows_bf16 = 0;
    if (a.D <= 128) launch_filter_mc<2, uint8_t, true>(b, phase, s);
    else launch_filter_mc<4, uint8_t, true>(b, phase, s);
    return;
  }
  if (a.rows_bf16) launch_prune_t<uint16_t>(a, phase, centroid, ep, s, nseg);
  else launch_prune_t<float>(a, phase, centroid, ep, s, nseg);
}

void launch_centroid(const float* X, uint32_t N, uint32_t D, double* part, float* c,
                     hipStream_t s) {
  const uint32_t nch = (N + 1023) / 1024;
  k_centroid_part<<<dim3(nch, (D + 63) / 64), 64, 0, s>>>(X, N, D, part);
  k_centroid_final<<<(D + 63) / 64, 64, 0, s>>>(part, nch, N, D, c);
}

}  // namespace tg
