// search.hip -- beam search over a pruned index, the validator of the produced graphs.
//
// Restates get_neighbors (common.cu:65-127, the NSG search the reference carries but never
// runs on its outputs) for the variable-degree rows of a pruned graph, with the same rules
// as the CPU oracle's or_search:
//   * initial ids: the first min(L, deg(ep)) neighbours of the entry point, then draws from a
//     per-query SplitMix64 stream (the reference: rand() % N) that skip visited ids, until
//     min(L, N) ids or 4096 draws; all of them are marked visited;
//   * the pool holds those ids sorted by (canonical distance, id), each with a checked flag;
//   * k = 0; repeat: k = first unchecked position >= k; mark it checked and expand its node:
//     every neighbour not yet visited is marked visited and evaluated, and the pool becomes
//     the L smallest of pool and candidates -- the set the reference's one-at-a-time
//     InsertIntoPool leaves -- with nk = the position of the smallest candidate if it
//     enters (that is the smallest insertion position), else L; k = nk <= k ? nk : k + 1.
// One wave per query, the pool in registers (64*NPL >= L slots, NPL = 1, 2 or 4).  An expansion
// is one serial chain (adjacency row, visited checks, candidate rows, sort, merge), so the
// kernel shortens the chain:
//   * the visited set is an LDS hash, sized by the host for the usual number of visited ids;
//     a query that fills it moves its ids to a bitmap in device memory (exact for any N) and
//     goes on there.  Each workgroup owns a bitmap and a list of the ids it set; it clears those
//     words after the query (or the whole bitmap when the list overflowed), so the bitmap is all
//     zero again.  Bitmap and list are only touched with device-coherent atomics, loads, stores;
//   * a node's degree and row are loaded together, and the next unchecked pool entry's row is
//     requested meanwhile (it is the next expansion unless a candidate beats it);
//   * all candidate rows of an expansion (32 FP32 rows, or 64 u8 rows) are in flight at once;
//     u8 data whose query is integer too takes the exact dot4 distances of a quarter the bytes;
//   * up to 64 candidates are sorted in one register slot, by blocks of the next power of two.
// 100k x 128 u8, L = 64, one query: 207 -> 122 us (some 65 expansions); 10,000 queries over
// 1M x 128: 2.26 -> 0.93 ms.
#include "common.hpp"
#include "kernels.hpp"
#include "rules.hpp"

namespace tg {

namespace {

__device__ __forceinline__ uint32_t ld_dev(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// marks id visited; true when it was not before
__device__ __forceinline__ bool visit(uint32_t* bm, uint32_t id) {
  const uint32_t bit = 1u << (id & 31);
  return (atomicOr(&bm[id >> 5], bit) & bit) == 0;
}

constexpr int FILL_ROUNDS = 64;  // 64 rounds of 64 draws

// LDS hash set of ids (INV: empty): true when id was not a member
__device__ __forceinline__ bool vset_add(uint32_t* tab, int bits, uint32_t id) {
  const uint32_t mask = (1u << bits) - 1;
  uint32_t h = (id * 0x9E3779B1u) >> (32 - bits);
  for (;;) {
    const uint32_t old = atomicCAS(&tab[h], TG_INV, id);
    if (old == TG_INV) return true;
    if (old == id) return false;
    h = (h + 1) & mask;
  }
}
__device__ __forceinline__ bool vset_has(const uint32_t* tab, int bits, uint32_t id) {
  const uint32_t mask = (1u << bits) - 1;
  uint32_t h = (id * 0x9E3779B1u) >> (32 - bits);
  for (;;) {
    const uint32_t v = tab[h];
    if (v == id || v == TG_INV) return v == id;
    h = (h + 1) & mask;
  }
}

// The query as a u8 row (quad layout) when it is integer in [0, 255]; false otherwise.  Every
// distance to a u8 row is then an exact integer below 2^24 (D <= 256), in either arithmetic.
template <int MC>
__device__ __forceinline__ bool query_u8(Row16<MC>& r, const float* q, int D) {
  const int j = threadIdx.x & 3;
  bool ok = true;
  int sq = 0;
#pragma unroll
  for (int m = 0; m < MC; ++m) {
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = m * 64 + 16 * j + 4 * k;
      w[k] = 0;
      if (i < D) {
        const float4 v = load4(q + i);
        const float x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          ok = ok && x[b] >= 0.f && x[b] <= 255.f && rintf(x[b]) == x[b];
          w[k] |= (uint32_t(int(x[b])) & 255u) << (8 * b);
        }
        w[k] ^= 0x80808080u;
      }
    }
    const uint4 u = make_uint4(w[0], w[1], w[2], w[3]);
    r.v[m] = make_float4(__uint_as_float(w[0]), __uint_as_float(w[1]), __uint_as_float(w[2]),
                         __uint_as_float(w[3]));
    sq = dot16_u8(u, u, sq);
  }
  r.n2 = quad_sum(sq);
  return ballot(!ok) == 0;
}

// Distances of the ids nbr[0..n) into keys S[0..n): NB candidates per 16-lane group in flight;
// the group's lane b takes its candidate b from lane 0.
template <int MC>
__device__ __forceinline__ void eval_f32(const float* X, int D, const Row16<MC>& xq, int n,
                                         const uint32_t* nbr, uint64_t* S) {
  constexpr int NB = MC <= 2 ? 8 : 4;
  const int lane = threadIdx.x, g = lane >> 4, t = lane & 15;
  for (int q0 = 0; q0 < n; q0 += 4 * NB) {
    const float* rows[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int q = q0 + g + 4 * b;
      rows[b] = q < n ? X + size_t(nbr[q]) * D : X;  // unused slots read row 0
    }
    float dd[NB];
    dist16_batch<MC, NB>(xq, rows, D, t, dd);
    float d = dd[0];
    const float d1 = row_shr<1>(dd[1]), d2 = row_shr<2>(dd[2]), d3 = row_shr<3>(dd[3]);
    d = t == 1 ? d1 : t == 2 ? d2 : t == 3 ? d3 : d;
    if constexpr (NB == 8) {
      const float d4 = row_shr<4>(dd[4]), d5 = row_shr<5>(dd[5]), d6 = row_shr<6>(dd[6]),
                  d7 = row_shr<7>(dd[7]);
      d = t == 4 ? d4 : t == 5 ? d5 : t == 6 ? d6 : t == 7 ? d7 : d;
    }
    const int q = q0 + g + 4 * t;
    if (t < NB && q < n) S[q] = mk_key(d, nbr[q]);
  }
}

// U8: a.X8 holds the u8 copy of the data.
// WV: waves per SIMD that the registers leave at least.
template <int MC, int NPL, bool U8, int WV>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WV))) void k_search(SearchArgs a) {
  extern __shared__ uint32_t vtab[];  // visited hash, 2^hbits ids
  __shared__ uint64_t S[256];     // candidate keys
  __shared__ uint32_t nbr[256];   // initial ids, then the fresh neighbours of a round
  __shared__ uint32_t firstocc[64];
  static_assert(sizeof(S) + sizeof(nbr) + sizeof(firstocc) == SEARCH_LDS, "search_hash_bits");
  const int lane = threadIdx.x, t = lane & 15;
  const uint32_t N = a.N, D = a.D, FD = a.FD;
  const int L = int(a.L), hb = int(a.hbits);
  // ids the hash may hold: three quarters of its slots (a probe ends at an empty one)
  const uint32_t hcap = (3u << hb) >> 2;
  uint32_t* bm = a.bitmap + size_t(blockIdx.x) * a.words;
  uint32_t* vl = a.vlist + size_t(blockIdx.x) * a.vcap;
  unsigned long long n_eval = 0, n_exp = 0;
  for (uint32_t q = blockIdx.x; q < a.nq; q += gridDim.x) {
    const float* qrow = a.Q + size_t(q) * D;
    Row16<MC> xq, x8;
    load_row16<MC>(xq, qrow, int(D), t);
    bool q8 = false;
    if constexpr (U8) q8 = query_u8<MC>(x8, qrow, int(D));
    auto eval = [&](int n) {
      if constexpr (U8) {
        if (q8) {
          eval_batch<MC, uint8_t, true>(a.X8, int(D), x8, n, [&](int i) { return nbr[i]; },
                                        [&](int i, float d) { S[i] = mk_key(d, nbr[i]); });
          return;
        }
      }
      eval_f32<MC>(a.X, int(D), xq, n, nbr, S);
    };
    for (int i = 4 * lane; i < (1 << hb); i += 4 * TG_WAVE)
      *reinterpret_cast<uint4*>(vtab + i) = make_uint4(TG_INV, TG_INV, TG_INV, TG_INV);
    __syncthreads();
    uint32_t nvis = 0;     // visited ids (counting repeats in the entry point's row)
    bool in_lds = true;    // the visited set is the hash; false: the bitmap
    // moves to the bitmap when `more` further ids may not fit the hash
    auto reserve = [&](uint32_t more) {
      if (!in_lds || nvis + more <= hcap) return;
      in_lds = false;
      nvis = 0;
      for (int i0 = 0; i0 < (1 << hb); i0 += TG_WAVE) {
        const uint32_t y = vtab[i0 + lane];
        const bool have = y != TG_INV;
        const uint64_t m = ballot(have);
        if (have) {
          atomicOr(&bm[y >> 5], 1u << (y & 31));
          const uint32_t o = nvis + uint32_t(mask_rank(m));
          if (o < a.vcap) st_dev(&vl[o], y);
        }
        nvis += uint32_t(__popcll(m));
      }
    };
    // ---- initial ids: the entry point's row, then random draws
    const int target = int(min(uint32_t(L), N));
    const int d0 = int(min(a.deg[a.ep], uint32_t(L)));
    reserve(uint32_t(target) + 128);
    for (int j = lane; j < d0; j += TG_WAVE) {
      const uint32_t y = a.ids[size_t(a.ep) * FD + j];
      nbr[j] = y;
      if (in_lds) {
        (void)vset_add(vtab, hb, y);
      } else {
        atomicOr(&bm[y >> 5], 1u << (y & 31));
        if (uint32_t(j) < a.vcap) st_dev(&vl[j], y);
      }
    }
    int ninit = d0;
    nvis = uint32_t(d0);
    const uint64_t qs = segment_seed(a.seed, q);
    __syncthreads();
    for (int r = 0; r < FILL_ROUNDS && ninit < target; ++r) {
      const uint32_t y = sm_bounded(sm_stream(qs, uint64_t(r) * 64 + lane), N);
      const bool seen = in_lds ? vset_has(vtab, hb, y) : ((ld_dev(&bm[y >> 5]) >> (y & 31)) & 1u) != 0;
      // first occurrence of y among this round's draws (lowest lane)
      uint64_t kv[1] = {(uint64_t(y) << 32) | uint32_t(lane)};
      reg_bitonic<1>(kv);
      const uint64_t prev = uint64_t(__shfl(int(kv[0] >> 32), (lane + 63) & 63, TG_WAVE));
      const bool first = lane == 0 || uint32_t(prev) != uint32_t(kv[0] >> 32);
      firstocc[uint32_t(kv[0])] = first ? 1u : 0u;
      __syncthreads();
      const bool ok = !seen && firstocc[lane] != 0;
      const uint64_t m = ballot(ok);
      const int need = target - ninit;
      const int rank = mask_rank(m);
      if (ok && rank < need) {
        nbr[ninit + rank] = y;
        if (in_lds) {
          (void)vset_add(vtab, hb, y);
        } else {
          atomicOr(&bm[y >> 5], 1u << (y & 31));
          if (nvis + uint32_t(rank) < a.vcap) st_dev(&vl[nvis + rank], y);
        }
      }
      const int got = min(int(__popcll(m)), need);
      ninit += got;
      nvis += uint32_t(got);
      __syncthreads();
    }
    // ---- the pool: initial ids with distances, sorted
    eval(ninit);
    n_eval += uint64_t(ninit);
    __syncthreads();
    uint64_t v[NPL];
    uint32_t f[NPL];
#pragma unroll
    for (int b = 0; b < NPL; ++b) {
      const int p = b * 64 + lane;
      v[b] = p < ninit ? S[p] : TG_KEY_INF;
      f[b] = 0;
    }
    reg_bitonic<NPL>(v);
    __syncthreads();
    // the first unchecked entry at or after position `from`: its position (-1: none) and id
    auto unchecked = [&](int from, uint32_t& id) {
      int pos = -1;
#pragma unroll
      for (int b = 0; b < NPL; ++b) {
        if (pos >= 0) break;
        const int p = b * 64 + lane;
        const uint64_t m = ballot(p >= from && p < L && v[b] != TG_KEY_INF && f[b] == 0);
        if (m) {
          const int fl = __ffsll((unsigned long long)m) - 1;
          pos = b * 64 + fl;
          id = uint32_t(__builtin_amdgcn_readlane(int(key_id(v[b])), fl));
        }
      }
      return pos;
    };
    auto load_adj = [&](uint32_t n, uint32_t& dn, uint32_t (&y)[2]) {
      dn = a.deg[n];
      y[0] = uint32_t(lane) < FD ? a.ids[size_t(n) * FD + lane] : TG_INV;
      y[1] = uint32_t(TG_WAVE + lane) < FD ? a.ids[size_t(n) * FD + TG_WAVE + lane] : TG_INV;
    };
    // ---- expansions
    int kk = 0;
    uint32_t pre = TG_INV, pre_dn = 0, pre_y[2] = {TG_INV, TG_INV};  // the requested row
    for (;;) {
      uint32_t n = 0;
      const int first = unchecked(kk, n);
      if (first < 0) break;
#pragma unroll
      for (int b = 0; b < NPL; ++b)
        if (b * 64 + lane == first) f[b] = 1;
      ++n_exp;
      uint32_t dn = pre_dn, y[2] = {pre_y[0], pre_y[1]};
      if (n != pre) load_adj(n, dn, y);
      uint32_t n2 = TG_INV;
      if (unchecked(first + 1, n2) >= 0) load_adj(n2, pre_dn, pre_y);
      pre = n2;
      // unvisited neighbours of n
      reserve(128);
      int cnt = 0;
#pragma unroll
      for (int base = 0; base < 128; base += TG_WAVE) {
        if (uint32_t(base) >= FD) break;
        const uint32_t w = y[base / TG_WAVE];
        bool fresh = false;
        if (uint32_t(base + lane) < dn) fresh = in_lds ? vset_add(vtab, hb, w) : visit(bm, w);
        const uint64_t fm = ballot(fresh);
        if (fresh) {
          const int pos = cnt + mask_rank(fm);
          nbr[pos] = w;
          if (!in_lds && nvis + uint32_t(pos) < a.vcap) st_dev(&vl[nvis + pos], w);
        }
        cnt += int(__popcll(fm));
      }
      nvis += uint32_t(cnt);
      if (cnt == 0) {
        kk = first + 1;
        continue;
      }
      __syncthreads();
      eval(cnt);
      n_eval += uint64_t(cnt);
      __syncthreads();
      // candidates sorted in registers (at most 128)
      uint64_t c[2] = {lane < cnt ? S[lane] : TG_KEY_INF, TG_KEY_INF};
      if (cnt <= 16) {
        reg_bitonic_upto<16>(c[0]);
      } else if (cnt <= 32) {
        reg_bitonic_upto<32>(c[0]);
      } else if (cnt <= 64) {
        reg_bitonic_upto<64>(c[0]);
      } else {
        c[1] = TG_WAVE + lane < cnt ? S[TG_WAVE + lane] : TG_KEY_INF;
        reg_bitonic<2>(c);
      }
      const uint64_t cmin = uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(c[0] >> 32)))) << 32 |
                            uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(c[0]))));
      // the pool's last slot L-1
      const int lb = (L - 1) >> 6, ll = (L - 1) & 63;
      uint64_t lastk = TG_KEY_INF;
#pragma unroll
      for (int b = 0; b < NPL; ++b)
        if (b == lb)
          lastk = uint64_t(uint32_t(__builtin_amdgcn_readlane(int(v[b] >> 32), ll))) << 32 |
                  uint32_t(__builtin_amdgcn_readlane(int(uint32_t(v[b])), ll));
      if (!(cmin < lastk)) {  // no candidate enters
        kk = first + 1;
        continue;
      }
      int nk = 0;
#pragma unroll
      for (int b = 0; b < NPL; ++b) nk += int(__popcll(ballot(v[b] < cmin)));
      // the L smallest of pool and candidates: min(pool[p], cand[64 NPL - 1 - p]) is
      // bitonic; candidate slots past the first two are +inf
      uint64_t w[NPL];
      uint32_t g[NPL];
#pragma unroll
      for (int b = 0; b < NPL; ++b) {
        const int rs = NPL - 1 - b;
        const uint64_t rv = rs < 2 ? lane_xor64(c[rs < 2 ? rs : 0], 63) : TG_KEY_INF;
        const bool keep = v[b] < rv;
        w[b] = keep ? v[b] : rv;
        g[b] = keep ? f[b] : 0u;
      }
      reg_bitonic_merge_kv<NPL>(w, g);
#pragma unroll
      for (int b = 0; b < NPL; ++b) {
        const bool in = b * 64 + lane < L;
        v[b] = in ? w[b] : TG_KEY_INF;
        f[b] = in ? g[b] : 0u;
      }
      kk = nk <= first ? nk : first + 1;
    }
    // ---- the first k entries
#pragma unroll
    for (int b = 0; b < NPL; ++b) {
      const int p = b * 64 + lane;
      if (p < int(a.k)) {
        const bool valid = v[b] != TG_KEY_INF;
        a.out_ids[size_t(q) * a.k + p] = valid ? key_id(v[b]) : TG_INV;
        a.out_d[size_t(q) * a.k + p] = valid ? key_d(v[b]) : __uint_as_float(0x7F800000u);
      }
    }
    // ---- clear this query's bits
    if (!in_lds) {
      if (nvis <= a.vcap) {
        for (uint32_t i = lane; i < nvis; i += TG_WAVE) st_dev(&bm[ld_dev(&vl[i]) >> 5], 0u);
      } else {
        for (uint32_t i = lane; i < a.words; i += TG_WAVE) st_dev(&bm[i], 0u);
      }
      __threadfence();
    }
    __syncthreads();
  }
  if (a.counters && lane == 0) {
    atomicAdd(&a.counters[0], n_eval);
    atomicAdd(&a.counters[1], n_exp);
  }
}

template <int MC, int NPL, bool U8, int WV>
void launch_search_w(SearchArgs a, uint32_t grid, uint32_t per_cu, hipStream_t s) {
  // workgroups a CU has to hold: those launched, up to what the registers allow (asked for only
  // where it can matter)
  int fit = 0;
  if (per_cu > 4 && hipOccupancyMaxActiveBlocksPerMultiprocessor(&fit, k_search<MC, NPL, U8, WV>, 64,
                                                                 0) == hipSuccess && fit > 0)
    per_cu = std::min(per_cu, uint32_t(fit));
  a.hbits = search_hash_bits(a.L, a.FD, per_cu);
  k_search<MC, NPL, U8, WV><<<grid, 64, size_t(4) << a.hbits, s>>>(a);
}
template <int MC, int NPL, bool U8>
void launch_search_t(const SearchArgs& a, uint32_t grid, hipStream_t s) {
  const uint32_t per_cu = (grid + 255) / 256;
  // u8 rows above 128 elements, pool above 128: two waves per SIMD by themselves, three with 20
  // spilled registers.  More than eight queries per CU need the third (10,000 over 100k x 256, L
  // 256, FD 16 / 32 / 48: 5.5 / 5.4 / 5.3 ms with two, 4.5 / 4.3 / 4.2 with three); one does not
  // (554 us, 576)
  if constexpr (MC == 4 && U8 && NPL == 4)
    if (per_cu > 8) return launch_search_w<MC, NPL, U8, 3>(a, grid, per_cu, s);
  launch_search_w<MC, NPL, U8, 1>(a, grid, per_cu, s);
}

}  // namespace

void launch_search(const SearchArgs& a, uint32_t grid, hipStream_t s) {
  const int mc = (int(a.D) + 63) / 64;
  const int npl = a.L <= 64 ? 1 : (a.L <= 128 ? 2 : 4);
#define SR(M, P, U) launch_search_t<M, P, U>(a, grid, s)
#define SR_P(M, U)                                \
  do {                                            \
    if (npl == 1) SR(M, 1, U);                    \
    else if (npl == 2) SR(M, 2, U);               \
    else SR(M, 4, U);                             \
  } while (0)
  if (a.X8 && mc <= 2) SR_P(2, true);
  else if (a.X8 && mc <= 4) SR_P(4, true);
  else if (mc <= 2) SR_P(2, false);
  else if (mc <= 4) SR_P(4, false);
  else SR_P(16, false);
#undef SR_P
#undef SR
}

}  // namespace tg
