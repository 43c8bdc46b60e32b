// prune_screen.hip -- DPG occlusion counts from an MFMA Gram of each node's neighbours.
//
// DPG (filter_dpg, Tagore_src.cu:1713-1785; rule A.9) counts, for every neighbour j of u,
// the earlier neighbours r < j with d(G[u][r], G[u][j]) < D[u][j].  That is K(K-1)/2
// canonical distances per node (2,016 at K=64), which at dimension 960 makes the plain kernel
// read each pair's two rows: ~15 MB per node.  Here the K rows are staged through LDS once,
// their Gram matrix runs on MFMA (16-bit 16x16x32, or FP8 e4m3 16x16x32 with per-vector scales),
// and each screen distance s comes with the rigorous bound E of the local join's screen:
//   s + E <  D[u][j]  -> occludes (d <= s + E);
//   s - E >= D[u][j]  -> does not (d >= s - E);
//   otherwise the canonical FP32 distance decides.
// The counts, and so the pruned rows, are those of the exact rule.  K <= 64.
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "screen.hpp"

namespace tg {

namespace {

__device__ __forceinline__ float dpg_bound(float na, float qa, float ea, float nb, float qb,
                                           float eb, float eta) {
  return 2.0f * (ea * qb + qa * eb + ea * eb) + eta * (na + nb + 2.0f * qa * qb);
}

// PREC 2: 16-bit rows (q.Xb; BF: BF16, else scaled FP16), PREC 3: FP8 rows
// (q.Xq8, scales q.sc8).  256 threads; wave w owns rows 16w..16w+15 of the 64 x 64 Gram,
// against the column blocks at or after its own (pairs r < j only).
// 100k x 960, K = 64: 15.5 -> 5.5 ms (the FP16 copy leaves 55 of the 2,016 pairs undecided;
// one BF16 product with its eight times wider bound left several times as many, and each reads
// two 3.8 KB rows).
template <int PREC, int MC, class T, bool BF>
__global__ __launch_bounds__(256) void k_dpg_screen(PruneArgs a, DpgScreen q) {
  constexpr int DC = PREC == 3 ? 256 : 128;  // elements staged per round (256 bytes per row)
  static_assert(PREC == 3 || DC == int(DPG_CHAIN), "a chain per round");
  using St = ScreenStage<PREC, DC, 64>;
  constexpr int MROW = 65;
  constexpr int SMEM = St::BYTES > 64 * MROW * 4 ? St::BYTES : 64 * MROW * 4;
  __shared__ __attribute__((aligned(16))) unsigned char smem[SMEM];
  __shared__ uint32_t nei[64], det[64];
  __shared__ float nn[64], nq[64], ne[64], sc[64], thr[64];
  __shared__ uint16_t queue[64 * 63 / 2];
  __shared__ uint32_t nqueue;
  __shared__ uint64_t srt[64];
  float* M = reinterpret_cast<float*>(smem);

  const uint32_t u = row_of_block(a.perm, a.N);
  if (u >= a.N) return;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int K = a.K, D = a.D, d = a.FD;
  if (tid < 64) {
    det[tid] = 0;
    if (tid < K) {
      const uint32_t v = a.G[size_t(u) * K + tid];
      nei[tid] = v;
      nn[tid] = q.nrm2[v];
      if (PREC == 3) {
        nq[tid] = q.nq[v];
        ne[tid] = q.ne[v];
        sc[tid] = q.sc8[v];
      }
      thr[tid] = a.GD[size_t(u) * K + tid];
    }
  }
  if (tid == 0) nqueue = 0;
  __syncthreads();
  f32x4 acc[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  screen_chunks<PREC, DC, 64>(
      PREC == 3 ? static_cast<const void*>(q.Xq8) : static_cast<const void*>(q.Xb), nei, D,
      [&](int r) { return r < K; }, smem, [&]() {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (c >= w) {
            // a sum of its own per round, added up: the chain, and with it the bound, stays
            // short (DPG over
            // 100k x 960: 6.53 -> 6.09 ms a call)
            f32x4 p = {0.f, 0.f, 0.f, 0.f};
            screen_block<PREC, BF, DC>(smem + 16 * w * St::RS, smem + 16 * c * St::RS, l, p);
            acc[c] += p;
          }
      });
  // screen distances (the matrix aliases the staging area, free after the last round)
#pragma unroll
  for (int c = 0; c < 4; ++c) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * w + 4 * (l >> 4) + r, j = 16 * c + (l & 15);
      float s = 0.f;
      if (i < K && j < K)
        s = PREC == 3 ? (nn[i] + nn[j]) - 2.0f * ((sc[i] * sc[j]) * acc[c][r])
                      : __builtin_fmaf(-q.pscale, acc[c][r], nn[i] + nn[j]);
      M[i * MROW + j] = s;  // used where i < j
    }
  }
  __syncthreads();
  // classify every pair r < j
  const int npairs = K * (K - 1) / 2;
  for (int p = tid; p < npairs; p += 256) {
    // p -> (r, j), j = 1..K-1, pairs of column j are r = 0..j-1
    int j = int((1.0f + sqrtf(1.0f + 8.0f * float(p))) * 0.5f);
    while (j * (j - 1) / 2 > p) --j;
    while ((j + 1) * j / 2 <= p) ++j;
    const int r = p - j * (j - 1) / 2;
    const float s = M[r * MROW + j];
    const float E = PREC == 3 ? dpg_bound(nn[r], nq[r], ne[r], nn[j], nq[j], ne[j], q.eta)
                              : q.kap * (nn[r] + nn[j]);
    const float tau = thr[j];
    if (s + E < tau) {
      atomicAdd(&det[j], 1u);
    } else if (!(s - E >= tau)) {
      const uint32_t slot = atomicAdd(&nqueue, 1u);
      queue[slot] = uint16_t((r << 8) | j);
    }
  }
  __syncthreads();
  // canonical distances of the undecided pairs, four per 16-lane group in flight
  const int nqd = int(nqueue);
  const int gg = tid >> 4, t = tid & 15;
  const T* rows = reinterpret_cast<const T*>(a.rows);
  for (int e0 = 0; e0 < nqd; e0 += 64) {
    const T* ra[4];
    const T* rb[4];
    int jj[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int e = e0 + gg + 16 * b;
      ra[b] = rb[b] = rows;  // unused slots read row 0
      jj[b] = -1;
      if (e < nqd) {
        const int r = queue[e] >> 8, j = queue[e] & 255;
        ra[b] = rows + size_t(nei[r]) * D;
        rb[b] = rows + size_t(nei[j]) * D;
        jj[b] = j;
      }
    }
    float dd[4];
    dist16_pairs<MC, 4>(ra, rb, D, t, dd);
    if (t == 0) {
#pragma unroll
      for (int b = 0; b < 4; ++b)
        if (jj[b] >= 0 && dd[b] < thr[jj[b]]) atomicAdd(&det[jj[b]], 1u);
    }
  }
  __syncthreads();
  if (tid == 0 && a.counters) {
    atomicAdd(&cnt_slot(a.counters)[1], (unsigned long long)npairs);
    atomicAdd(&cnt_slot(a.counters)[5], (unsigned long long)nqd);
  }
  // select the d entries of smallest (detour count, id) and push the reverse pairs
  if (tid < 64) srt[tid] = tid < K ? ((uint64_t(det[tid]) << 32) | nei[tid]) : TG_KEY_INF;
  __syncthreads();
  wave_bitonic(srt, 64);  // every thread calls it: 32 compare-exchanges per step, one each
  for (int i = tid; i < d; i += 256) {
    const uint64_t k = srt[i];
    a.fwd_ids[size_t(u) * d + i] = uint32_t(k);
    pb_push(a.rev, uint32_t(k), (k & 0xFFFFFFFF00000000ull) | u);
  }
  if (tid == 0) a.fwd_deg[u] = d;
}

}  // namespace

void launch_dpg_screen(const PruneArgs& a, const DpgScreen& q, int precision, hipStream_t s) {
  const int mc = (int(a.D) + 63) / 64;
#define DS(P, M, T, BF) k_dpg_screen<P, M, T, BF><<<grid_rows(a.perm, a.N), 256, 0, s>>>(a, q)
#define DS_MC(P, T, BF)                                                \
  do {                                                                 \
    if (mc <= 2) DS(P, 2, T, BF);                                      \
    else if (mc <= 4) DS(P, 4, T, BF);                                 \
    else DS(P, 16, T, BF);                                             \
  } while (0)
  if (precision == KP_FP8) {
    if (a.rows_bf16) DS_MC(3, uint16_t, false); else DS_MC(3, float, false);
  } else {
    if (a.rows_bf16) DS_MC(2, uint16_t, true);
    else if (a.h_bf16) DS_MC(2, float, true);
    else DS_MC(2, float, false);
  }
#undef DS_MC
#undef DS
}

}  // namespace tg
