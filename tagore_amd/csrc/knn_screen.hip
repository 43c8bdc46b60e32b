// knn_screen.hip -- screened local join on MFMA (FP32 or BF16) with exact FP32 re-scoring.
//
// The local join of GNN-Descent (nn_descent_opt_cal, Tagore_src.cu:684-1033) needs, for every
// sampled node list A = new'(u) (<= 64 rows) and B = old'(u) (<= 64 rows), the per-16-wide-
// tile minimum of the pair distances A x B, B x A and A x A.  Here the Gram matrices A.B^T and
// A.A^T are contracted on the matrix cores from LDS-staged, coalesced row loads:
//   16-bit: v_mfma_f32_16x16x32_bf16 / _f16 on a 16-bit copy of the vectors (screen.hpp),
//   FP32: v_mfma_f32_16x16x4_f32 on the FP32 vectors,
// and turned into screen distances s = |a|^2 + |b|^2 - 2 a'.b'.  A rigorous bound on
// |s - dist(a,b)| (quantisation + accumulation + canonical-distance rounding) selects, per
// tile, the only candidates that can be the exact (distance, id) minimum and pass the
// destination's worst distance; those are re-scored with the canonical FP32 distance.  The
// pushes are therefore bit-identical to the exact kernel's: graph decisions stay FP32.
#include "common.hpp"
#include "kernels.hpp"
#include "screen.hpp"

namespace tg {

constexpr int HROW_S = 128;


// Maximum / union over the workgroup of one value per thread, in thread 0 (sh: 4 words).
template <class Op>
__device__ __forceinline__ uint32_t wg_reduce(uint32_t v, uint32_t* sh, Op op) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = op(v, uint32_t(__shfl_xor(int(v), o, TG_WAVE)));
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  const uint32_t r = op(op(sh[0], sh[1]), op(sh[2], sh[3]));
  __syncthreads();
  return r;
}
__device__ __forceinline__ uint32_t op_max(uint32_t a, uint32_t b) { return a > b ? a : b; }
__device__ __forceinline__ uint32_t op_or(uint32_t a, uint32_t b) { return a | b; }

// |x|^2 of every row (FP64 sums, rounded once; NaN above 0 and below 2^-96) and the data-set
// certificates:
// flags[0] |= some value is not exactly representable in BF16,
// flags[1] |= some value is not an integer in [-256, 256], flags[2] |= some value is
// negative, flags[3] = max |x|^2 (FP32 bits; exact for integer data below 2^24),
// flags[4] |= some value is above 255, flags[5] = max |value| (FP32 bits).
// A 16-lane group per row with 16-byte loads; the flags leave a workgroup once (an atomic per
// row on one word took 11.3 ms for 1M x 128 rows, all of it the atomics).
__global__ __launch_bounds__(256) void k_screen_prep(const float* X, uint32_t N, uint32_t D,
                                                     float* nrm2, uint32_t* flags) {
  __shared__ uint32_t sh[4];
  const int t = threadIdx.x & 15;
  uint32_t bits = 0, top = 0, big = 0;  // bits: 1 not BF16, 2 not integer, 4 negative, 8 above 255
  for (size_t row = size_t(blockIdx.x) * 16 + (threadIdx.x >> 4); row < N;
       row += size_t(gridDim.x) * 16) {
    const float* x = X + row * D;
    double s2 = 0.0;
    for (uint32_t j = 4 * t; j < D; j += 64) {
      const float4 q = load4(x + j);
      const float v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        bits |= (bf2f(f2bf(v[b])) != v[b]) ? 1u : 0u;
        bits |= !(rintf(v[b]) == v[b] && fabsf(v[b]) <= 256.f) ? 2u : 0u;
        bits |= v[b] < 0.f ? 4u : 0u;
        bits |= v[b] > 255.f ? 8u : 0u;
        big = op_max(big, __float_as_uint(v[b]) & 0x7FFFFFFFu);
        s2 += double(v[b]) * double(v[b]);
      }
    }
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) s2 += __shfl_xor(s2, o, 16);
    top = op_max(top, __float_as_uint(float(s2)));
    // products of rows this small are not normal FP32 numbers, which no bound covers: not a
    // number, so that no screen decides a pair of such a row
    if (t == 0) nrm2[row] = s2 > 0.0 && s2 < 0x1p-96 ? __uint_as_float(0x7FC00000u) : float(s2);
  }
  bits = wg_reduce(bits, sh, op_or);
  top = wg_reduce(top, sh, op_max);
  big = wg_reduce(big, sh, op_max);
  if (threadIdx.x == 0) {
    if (bits & 1u) atomicOr(&flags[0], 1u);
    if (bits & 2u) atomicOr(&flags[1], 1u);
    if (bits & 4u) atomicOr(&flags[2], 1u);
    atomicMax(&flags[3], top);
    if (bits & 8u) atomicOr(&flags[4], 1u);
    atomicMax(&flags[5], big);
  }
}

// 16-bit copy of the rows: BF16 bits (COPY_EXACT: every value exact), FP16 of x * scale (a power
// of two that puts the largest value below 2^15), or BF16 to nearest (scale 1); results below
// the smallest normal value become 0.  The last two: flags[6] = max over the rows of
// |x' / scale - x| / |x|, rounded up (FP32 bits).  Rows whose |x|^2 is no finite FP32 value or
// below 2^-96 are left out: no screen decides a pair of such a row (k_screen_prep).
template <int KIND>
__global__ __launch_bounds__(256) void k_screen_copy(const float* X, uint32_t N, uint32_t D,
                                                     float scale, uint16_t* Xb, uint32_t* flags) {
  __shared__ uint32_t sh[4];
  const int t = threadIdx.x & 15;
  const double inv = 1.0 / double(scale);
  uint32_t worst = 0;
  for (size_t row = size_t(blockIdx.x) * 16 + (threadIdx.x >> 4); row < N;
       row += size_t(gridDim.x) * 16) {
    const float* x = X + row * D;
    double s2 = 0.0, e2 = 0.0;
    for (uint32_t j = 4 * t; j < D; j += 64) {
      const float4 q = load4(x + j);
      const float v[4] = {q.x, q.y, q.z, q.w};
      uint32_t h[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        if (KIND != COPY_EXACT) {
          float x16;
          if (KIND == COPY_FP16) {
            _Float16 f = _Float16(v[b] * scale);
            if (fabsf(float(f)) < 0x1p-14f) f = _Float16(0.f);
            h[b] = __builtin_bit_cast(uint16_t, f);
            x16 = float(f);
          } else {
            h[b] = f2bf(v[b]);
            if (fabsf(bf2f(h[b])) < 0x1p-126f) h[b] = 0;
            x16 = bf2f(h[b]);
          }
          const double w = double(x16) * inv;
          s2 += double(v[b]) * double(v[b]);
          e2 += (w - double(v[b])) * (w - double(v[b]));
        } else {
          h[b] = __float_as_uint(v[b]) >> 16;
        }
      }
      *reinterpret_cast<uint2*>(Xb + row * D + j) = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
    }
    if (KIND != COPY_EXACT) {
#pragma unroll
      for (int o = 8; o >= 1; o >>= 1) {
        s2 += __shfl_xor(s2, o, 16);
        e2 += __shfl_xor(e2, o, 16);
      }
      const bool in = s2 >= 0x1p-96 && s2 <= 3.4028234e38;
      const float r = in ? float(sqrt(e2 / s2) * (1.0 + 1e-6)) : 0.f;
      worst = op_max(worst, __float_as_uint(r));
    }
  }
  if (KIND != COPY_EXACT) {
    worst = wg_reduce(worst, sh, op_max);
    if (threadIdx.x == 0) atomicMax(&flags[6], worst);
  }
}

// u8 copy of X as signed bytes x - 128 (the byte XOR 0x80), four values per thread (every value
// an integer in [0, 255], D % 4 == 0)
__global__ void k_make_u8(const float4* X, size_t n4, uint32_t* X8) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n4;
       i += size_t(gridDim.x) * blockDim.x) {
    const float4 v = X[i];
    X8[i] = (uint32_t(v.x) | uint32_t(v.y) << 8 | uint32_t(v.z) << 16 | uint32_t(v.w) << 24) ^
            0x80808080u;
  }
}

void launch_make_u8(const float* X, size_t n, uint8_t* X8, hipStream_t s) {
  const size_t n4 = n / 4;
  const uint32_t grid = uint32_t(std::min<size_t>((n4 + 255) / 256, 8192));
  k_make_u8<<<grid, 256, 0, s>>>(reinterpret_cast<const float4*>(X), n4,
                                 reinterpret_cast<uint32_t*>(X8));
}

// |x - 128|^2 of every u8 row, one wave per row (an integer below 2^24 for D <= 256, so
// exact as FP32)
__global__ void k_u8_shift_norms(const uint8_t* X8, uint32_t N, uint32_t D, float* n2s) {
  const uint32_t row = blockIdx.x;
  if (row >= N) return;
  const uint8_t* x = X8 + size_t(row) * D;
  int acc = 0;
  for (uint32_t j = threadIdx.x; j < D; j += TG_WAVE) {
    const int v = int(int8_t(x[j]));
    acc += v * v;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, TG_WAVE);
  if (threadIdx.x == 0) n2s[row] = float(acc);
}

void launch_u8_shift_norms(const uint8_t* X8, uint32_t N, uint32_t D, float* n2s, hipStream_t s) {
  k_u8_shift_norms<<<N, 64, 0, s>>>(X8, N, D, n2s);
}

// FP8 e4m3 copy with a per-vector scale: q = e4m3(x / s), s = max|x| / 440 (below the
// format's 448 maximum), and the norms the screen bound needs: |s q| and |x - s q| in FP64,
// rounded up.  One wave per row, four elements per lane per step.
__global__ void k_screen_prep8(const float* X, uint32_t N, uint32_t D, uint8_t* Xq, float* sc,
                               float* nq, float* ne) {
  const uint32_t row = blockIdx.x;
  if (row >= N) return;
  const float* x = X + size_t(row) * D;
  float mx = 0.f;
  for (uint32_t j = threadIdx.x; j < D; j += TG_WAVE) mx = fmaxf(mx, fabsf(x[j]));
  for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, TG_WAVE));
  const float s = mx > 0.f ? mx / 440.f : 1.f;
  double q2 = 0.0, e2 = 0.0;
  for (uint32_t j = 4 * threadIdx.x; j < D; j += 4 * TG_WAVE) {
    const float v0 = x[j], v1 = x[j + 1], v2 = x[j + 2], v3 = x[j + 3];
    int p = __builtin_amdgcn_cvt_pk_fp8_f32(v0 / s, v1 / s, 0, false);
    p = __builtin_amdgcn_cvt_pk_fp8_f32(v2 / s, v3 / s, p, true);
    *reinterpret_cast<int*>(Xq + size_t(row) * D + j) = p;
    typedef float f2 __attribute__((ext_vector_type(2)));
    const f2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(p, false), hi = __builtin_amdgcn_cvt_pk_f32_fp8(p, true);
    const float v[4] = {v0, v1, v2, v3}, dq[4] = {lo.x, lo.y, hi.x, hi.y};
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const double w = double(s) * double(dq[b]);
      q2 += w * w;
      e2 += (double(v[b]) - w) * (double(v[b]) - w);
    }
  }
  for (int o = 32; o >= 1; o >>= 1) {
    q2 += __shfl_xor(q2, o, TG_WAVE);
    e2 += __shfl_xor(e2, o, TG_WAVE);
  }
  if (threadIdx.x == 0) {
    sc[row] = s;
    nq[row] = float(sqrt(q2) * (1.0 + 1e-6));
    ne[row] = float(sqrt(e2) * (1.0 + 1e-6));
  }
}

void launch_screen_prep8(const float* X, uint32_t N, uint32_t D, uint8_t* Xq, float* sc,
                         float* nq, float* ne, hipStream_t s) {
  k_screen_prep8<<<N, TG_WAVE, 0, s>>>(X, N, D, Xq, sc, nq, ne);
}

static uint32_t prep_grid(uint32_t N) { return std::min<uint32_t>((N + 15) / 16, 2048u); }
void launch_screen_prep(const float* X, uint32_t N, uint32_t D, float* nrm2, uint32_t* flags,
                        hipStream_t s) {
  k_screen_prep<<<prep_grid(N), 256, 0, s>>>(X, N, D, nrm2, flags);
}
void launch_screen_copy(const float* X, uint32_t N, uint32_t D, int kind, float scale,
                        uint16_t* Xb, uint32_t* flags, hipStream_t s) {
#define SC(KIND) k_screen_copy<KIND><<<prep_grid(N), 256, 0, s>>>(X, N, D, scale, Xb, flags)
  if (kind == COPY_EXACT) SC(COPY_EXACT);
  else if (kind == COPY_FP16) SC(COPY_FP16);
  else SC(COPY_BF16);
#undef SC
}

// Local join when the screen distances are the canonical distances (integer data): each job's
// answer is the (s, id) minimum of its 16-wide tile, taken from the accumulators by cross-lane
// minima, so the kernel holds only the staging area (and runs more workgroups per CU).  Jobs:
// A rows x B tiles, B columns x A tiles, A rows x A tiles.  Only blocks that hold pairs are
// formed (an iteration from fresh lists has no B), shared evenly by the waves.
// 1M x 128 u8 rows, K = 96, one iteration: 8.7 -> 6.7 ms; 10k x 128, K = 32 with precision FP32
// (u8 products are as exact): 264 -> 62 us per iteration.
// (d, id) minimum over the lanes l ^ x for the masks x in [x0, x1) (powers of two): the
// smallest d, then the smallest id among the lanes holding it.  The exact screen's distances
// are integers >= 0 or +inf, whose FP32 bits order as unsigned integers, so both minima are
// integer minima (no NaN handling), and the result is the minimum of the keys mk_key(d, id).
template <int X0, int X1>
__device__ __forceinline__ uint64_t key_min_lanes(float d, uint32_t id) {
  const uint32_t db = __float_as_uint(d);
  uint32_t m = db;
#pragma unroll
  for (int x = X0; x < X1; x <<= 1) m = min(m, lane_xor32(m, x));
  uint32_t k = db == m ? id : 0xFFFFFFFFu;
#pragma unroll
  for (int x = X0; x < X1; x <<= 1) k = min(k, lane_xor32(k, x));
  return (uint64_t(m) << 32) | k;
}

// Minimum over the 16 lanes of the lane's DPP row, in every lane of it: quad exchanges, then
// row rotations by 4 and 8 (a minimum needs no exact partners).  Each step is one DPP-fused
// v_min_u32.
template <int CTRL>
__device__ __forceinline__ uint32_t min_dpp(uint32_t m) {
  return min(m, uint32_t(__builtin_amdgcn_update_dpp(int(0xFFFFFFFFu), int(m), CTRL, 0xF, 0xF,
                                                     false)));
}
__device__ __forceinline__ uint32_t row_min16(uint32_t m) {
  m = min_dpp<0xB1>(m);   // quad: lane ^ 1
  m = min_dpp<0x4E>(m);   // quad: lane ^ 2
  m = min_dpp<0x124>(m);  // row_ror:4
  return min_dpp<0x128>(m);  // row_ror:8
}
// key_min_lanes<1, 16> with row_min16: the (d, id) minimum over the lane's 16-lane row.
__device__ __forceinline__ uint64_t key_min_row16(float d, uint32_t id) {
  const uint32_t db = __float_as_uint(d);
  const uint32_t m = row_min16(db);
  return (uint64_t(m) << 32) | row_min16(db == m ? id : 0xFFFFFFFFu);
}

// Membership of Q keys in kNN rows (rows sorted by (distance, id), canonical distances):
// found[q] = key[q] is an entry of row v[q], for the searches with on[q], whose keys lie below
// the row's last distance.  Every lane searches a row of its own, so each load is an L2 request of
// its own, and their number and round trips set the push phase's time.  A search runs on
// blocks of four distances: by the blocks' last ones, then one load for the block (any 4-byte
// alignment); the ids are read where a distance is equal.  The searches go in lockstep, so the
// loads of one step are in flight together.  (By single distances, two or three requests and as
// many round trips more: local join 2290 -> 2151 us for 1M x 128 u8 rows, K = 96; 1590 -> 1493 for
// 160k x 96 clusters, K = 64.)
struct __attribute__((packed, aligned(4))) Dist4 {
  float x[4];
};
template <int Q>
__device__ __forceinline__ void rows_have_keys(const uint32_t* G, const float* GD, int K,
                                               const uint32_t (&v)[Q], const uint64_t (&key)[Q],
                                               const bool (&on)[Q], bool (&found)[Q]) {
  int lo[Q], hi[Q];
  const float* row[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    lo[q] = 0;
    hi[q] = on[q] ? (K + 3) / 4 - 1 : 0;
    row[q] = GD + size_t(v[q]) * K;
    found[q] = false;
  }
  // the first block whose last distance is not below the key's (the last block at the latest)
  for (;;) {
    bool any = false;
#pragma unroll
    for (int q = 0; q < Q; ++q) any = any || lo[q] < hi[q];
    if (!any) break;
    float x[Q];
    int mid[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      mid[q] = (lo[q] + hi[q]) >> 1;
      x[q] = lo[q] < hi[q] ? row[q][4 * mid[q] + 3] : 0.f;
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (lo[q] < hi[q]) {
        if (x[q] < key_d(key[q])) lo[q] = mid[q] + 1;
        else hi[q] = mid[q];
      }
    }
  }
  // its first entry of that distance, and that entry's id
  int at[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    at[q] = -1;
    if (!on[q]) continue;
    const float d = key_d(key[q]);
    if (K >= 4) {
      const int s = min(4 * lo[q], K - 4);  // the entries before the block's are below d
      const Dist4 y = *reinterpret_cast<const Dist4*>(row[q] + s);
#pragma unroll
      for (int k = 3; k >= 0; --k) at[q] = y.x[k] == d ? s + k : at[q];
    } else {
      for (int k = K - 1; k >= 0; --k) at[q] = row[q][k] == d ? k : at[q];
    }
  }
  uint32_t id[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) id[q] = at[q] >= 0 ? G[size_t(v[q]) * K + at[q]] : TG_INV;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    if (at[q] < 0) continue;
    found[q] = id[q] == key_id(key[q]);
    for (int p = at[q] + 1; !found[q] && p < K && row[q][p] == key_d(key[q]); ++p)
      found[q] = G[size_t(v[q]) * K + p] == key_id(key[q]);
  }
}

// The 16 x 16 blocks of a node's pairs, A x B and -- A x A being symmetric -- A x A on and above
// the diagonal, dealt to the four waves: block b of wave w is number w + 4b (NBLK of 26 at
// most).  Lane x holds block x's first candidate (an index into ids: B tiles from 64 on) and
// first row << 8, LJ_NONE past the last one; a wave reads its blocks' lanes.  (Scalar loops
// over the tiles for each block issued more instructions than everything else.)
constexpr int NBLK = 7;
constexpr int LJ_NONE = 0xFFFF;
__device__ __forceinline__ int lj_blocks(int RA, int RB) {
  const int x = lane_id();
  if (x < RA * RB) {
    const int rb = (x >= RB ? 1 : 0) + (x >= 2 * RB ? 1 : 0) + (x >= 3 * RB ? 1 : 0);
    return (16 * rb) << 8 | (64 + 16 * (x - rb * RB));
  }
  const int y = x - RA * RB;
  if (y >= RA * (RA + 1) / 2) return LJ_NONE;
  // row tile rb starts at number rb RA - rb (rb - 1) / 2
  const int rb = (y >= RA ? 1 : 0) + (y >= 2 * RA - 1 ? 1 : 0) + (RA > 1 && y >= 3 * RA - 3 ? 1 : 0);
  return (16 * rb) << 8 | 16 * (rb + y - (rb * RA - rb * (rb - 1) / 2));
}

// The jobs of a block of exact distances (s = (n_i + n_j) - 2 acc): the (d, id) minimum of every
// row over the 16 candidates, and of every candidate over the 16 rows.  kb: [64 rows of A][4
// tiles of B], ka: [64 rows of A][4 tiles of A], kc: [4 tiles of A][64 rows of B]; every job is
// one block's, so its key is stored, not merged.  Lane t of group g stores row 4g + t (t < 4),
// group 0 the candidates.
__device__ __forceinline__ void lj_block_minima(int bi, int bj, const f32x4& acc,
                                                const uint32_t* ids, const float* nn, int nA,
                                                int nB, uint64_t* kb, uint64_t* ka,
                                                uint64_t* kc) {
  const int l = threadIdx.x & 63, g = l >> 4, t = l & 15;
  const float INF = __uint_as_float(0x7F800000u);
  const int i0 = bi + 4 * g, jj = bj + t;
  const bool bt = bj >= 64;
  const bool jn = bt ? jj - 64 < nB : jj < nA;
  const float nj = nn[jj];
  const uint32_t idj = ids[jj];
  const float4 ni = *reinterpret_cast<const float4*>(nn + i0);
  const uint4 idi = *reinterpret_cast<const uint4*>(ids + i0);
  const float nv[4] = {ni.x, ni.y, ni.z, ni.w};
  const uint32_t iv[4] = {idi.x, idi.y, idi.z, idi.w};
  float cd = INF;  // the candidate's minimum: this lane's 4 rows, then across the groups
  uint32_t cid = 0xFFFFFFFFu;
  uint64_t mine = TG_KEY_INF;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const bool ok = i0 + r < nA && jn && (bt ? iv[r] != idj : i0 + r != jj);
    const float d = ok ? (nv[r] + nj) - 2.0f * acc[r] : INF;
    const uint64_t k = key_min_row16(d, idj);
    if (t == r) mine = k;
    if (d < cd || (d == cd && iv[r] < cid)) {
      cd = d;
      cid = iv[r];
    }
  }
  // a tile of invalid pairs keeps +inf distances, which no worst distance admits
  if (t < 4) (bt ? kb : ka)[4 * (i0 + t) + ((bt ? bj - 64 : bj) >> 4)] = mine;
  if (bi != bj) {
    const uint64_t kj = key_min_lanes<16, 64>(cd, cid);
    if (g == 0) {
      if (bt) kc[64 * (bi >> 4) + (jj - 64)] = kj;
      else ka[4 * jj + (bi >> 4)] = kj;
    }
  }
}

// The jobs' pushes: a job's minimum enters when it beats the destination's worst entry and
// is not already listed (the merge would drop it); the three row searches run together.
// Keys for one destination take one counter update and consecutive slots, so they share
// cache lines: the row jobs of A row i sit in the four lanes t = (i % 4) + 4c of a 16-lane
// row (up to 8 keys), the column jobs of B row l in lane l of the four waves (up to 4 keys,
// gathered through colk, 4 x 64 keys of LDS that no wave reads any more).  The slot order
// of a list is immaterial (its reduction sorts).
__device__ __forceinline__ void lj_push(const KnnArgs& a, const uint32_t* A, const uint32_t* B,
                                        const float* wA, const float* wB, int nA, int nB,
                                        int w, int g, int t, int l, uint64_t row_b,
                                        uint64_t row_a, uint64_t col_b, uint64_t* colk) {
  const int i = 16 * w + 4 * g + (t & 3);
  const bool inA = i < nA, inB = l < nB;
  const uint32_t destA = inA ? A[i] : 0u, destB = inB ? B[l] : 0u;
  const float worstA = inA ? wA[i] : 0.f, worstB = inB ? wB[l] : 0.f;
  const uint32_t dv[3] = {destA, destA, destB};
  const uint64_t kv[3] = {row_b, row_a, col_b};
  const bool on[3] = {inA && key_d(row_b) < worstA, inA && key_d(row_a) < worstA,
                      inB && key_d(col_b) < worstB};
  bool found[3];
  rows_have_keys<3>(a.G, a.GD, a.K, dv, kv, on, found);
  // row jobs: counts of the four lanes c = t / 4, their prefix in c order, one counter update
  const bool pb = on[0] && !found[0], pa = on[1] && !found[1];
  const int cnt = int(pb) + int(pa), c = t >> 2;
  const int x4 = int(lane_xor32(uint32_t(cnt), 4));
  const int p1 = cnt + x4;
  const int x8 = int(lane_xor32(uint32_t(p1), 8));
  const int total = p1 + x8;
  const int prefix = ((c & 1) ? x4 : 0) + ((c & 2) ? x8 : 0);
  uint32_t base = 0;
  if (c == 0 && total > 0) base = atomicAdd(&a.pc.cnt[destA], uint32_t(total));
  base = uint32_t(__shfl(int(base), (l & ~15) | (t & 3), TG_WAVE));
  if (pb) pb_put(a.pc, destA, base + uint32_t(prefix), row_b);
  if (pa) pb_put(a.pc, destA, base + uint32_t(prefix) + (pb ? 1u : 0u), row_a);
  // column jobs: wave 0 pushes the four waves' keys of B row l together
  __syncthreads();
  colk[w * 64 + l] = (on[2] && !found[2]) ? col_b : TG_KEY_INF;
  __syncthreads();
  if (w == 0 && inB) {
    uint64_t k4[4];
    uint32_t n = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      k4[q] = colk[q * 64 + l];
      n += k4[q] != TG_KEY_INF ? 1u : 0u;
    }
    if (n) {
      uint32_t s = atomicAdd(&a.pc.cnt[destB], n);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (k4[q] != TG_KEY_INF) pb_put(a.pc, destB, s++, k4[q]);
    }
  }
}

// The node's sample lists, their norms (na) and their destinations' worst distances (wl).
__device__ __forceinline__ void lj_lists(const KnnArgs& a, uint32_t u, const float* norms,
                                         int nA, int nB, uint32_t* A, uint32_t* B, float* naA,
                                         float* wA, float* naB, float* wB) {
  const int tid = threadIdx.x, K = a.K;
  if (tid < 64) {
    const bool in = tid < nA;
    const uint32_t v = in ? a.H[size_t(u) * HROW_S + tid] : 0u;
    A[tid] = v;
    naA[tid] = in ? norms[v] : 0.f;
    wA[tid] = in ? a.GD[size_t(v) * K + K - 1] : 0.f;
  } else if (tid < 128) {
    const int j = tid - 64;
    const bool in = j < nB;
    const uint32_t v = in ? a.H[size_t(u) * HROW_S + 64 + j] : 0u;
    B[j] = v;
    naB[j] = in ? norms[v] : 0.f;
    wB[j] = in ? a.GD[size_t(v) * K + K - 1] : 0.f;
  }
}

// Products of the exact kernels.  PREC 0: u8 data on int8 MFMA (every value an integer in
// [0, 255], D <= DC <= 256): rows, stored as x - 128, are staged whole and
// v_mfma_i32_16x16x64_i8 gives a'.b' exactly, so s = |a'|^2 + |b'|^2 - 2 a'.b' = |a - b|^2
// exactly (|a'|^2 from n2s), the canonical distance of this data.  PREC 1 / 2: FP32 / BF16
// MFMA, exact for integers too (values in [-256, 256]).
typedef int i32x4 __attribute__((ext_vector_type(4)));
template <int PREC, int DC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(PREC == 0 && DC == 128 ? 8 : 4)))
void k_localjoin_exact_screen(KnnArgs a) {
  static_assert(PREC <= 2, "u8, FP32 or BF16 products");
  using St = ScreenStage<(PREC == 0 ? 3 : PREC), DC, 128>;
  constexpr int RS = St::RS;
  constexpr int KEYS = 3 * 256 * 8;
  __shared__ __attribute__((aligned(16))) unsigned char smem[St::BYTES > KEYS ? St::BYTES : KEYS];
  __shared__ __attribute__((aligned(16))) uint32_t ids[128];
  __shared__ __attribute__((aligned(16))) float nn[128];
  __shared__ float wd[128];
  const uint32_t u = row_of_block(a.perm, a.N);
  if (u >= a.N) return;
  const int tid = threadIdx.x, l = tid & 63, g = l >> 4, t = l & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int D = a.D;
  const int nA = a.na[u], nB = a.nb[u];
  lj_lists(a, u, PREC == 0 ? a.n2s : a.nrm2, nA, nB, ids, ids + 64, nn, wd, nn + 64, wd + 64);
  __syncthreads();
  const int blocks = lj_blocks((nA + 15) >> 4, (nB + 15) >> 4);
  f32x4 acc[NBLK];
  if constexpr (PREC == 0) {
    // rows of both lists, up to whole tiles: bytes past D and rows past the list ends are 0
    constexpr int CPR = DC / 16;
    for (int e = tid; e < 2 * 64 * CPR; e += 256) {
      const int r = e / CPR, col = (e % CPR) * 16;
      const int n = r < 64 ? nA : nB, x = r & 63;
      if (x >= ((n + 15) & ~15)) continue;
      uint4 v = make_uint4(0u, 0u, 0u, 0u);
      if (x < n && col < D) {
        const uint8_t* src = a.X8 + size_t(ids[r]) * D + col;
        if ((D & 15) == 0) {
          v = *reinterpret_cast<const uint4*>(src);
        } else {
          v.x = *reinterpret_cast<const uint32_t*>(src);
          if (col + 4 < D) v.y = *reinterpret_cast<const uint32_t*>(src + 4);
          if (col + 8 < D) v.z = *reinterpret_cast<const uint32_t*>(src + 8);
          if (col + 12 < D) v.w = *reinterpret_cast<const uint32_t*>(src + 12);
        }
      }
      *reinterpret_cast<uint4*>(smem + r * RS + col) = v;
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < NBLK; ++b) {
      const int d = __builtin_amdgcn_readlane(blocks, w + 4 * b);
      if (d == LJ_NONE) continue;
      const int bi = d >> 8, bj = d & 255;
      i32x4 p = {0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < DC / 64; ++k)
        p = __builtin_amdgcn_mfma_i32_16x16x64_i8(
            *reinterpret_cast<const i32x4*>(smem + (bi + t) * RS + 64 * k + 16 * g),
            *reinterpret_cast<const i32x4*>(smem + (bj + t) * RS + 64 * k + 16 * g), p, 0, 0, 0);
      acc[b] = f32x4{float(p[0]), float(p[1]), float(p[2]), float(p[3])};
    }
    __syncthreads();
  } else {
#pragma unroll
    for (int b = 0; b < NBLK; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    screen_chunks<PREC, DC, 128>(
        PREC == 2 ? static_cast<const void*>(a.Xb) : a.X, ids, D,
        [&](int r) { return r < 64 ? r < nA : r - 64 < nB; }, smem, [&]() {
#pragma unroll
          for (int b = 0; b < NBLK; ++b) {
            const int d = __builtin_amdgcn_readlane(blocks, w + 4 * b);
            if (d != LJ_NONE)
              screen_block<PREC, true, DC>(smem + (d >> 8) * RS, smem + (d & 255) * RS, l, acc[b]);
          }
        });
  }
  // the jobs' keys, in the staging area (free from here on)
  uint64_t* kb = reinterpret_cast<uint64_t*>(smem);
  uint64_t* ka = kb + 256;
  uint64_t* kc = ka + 256;
  kb[tid] = TG_KEY_INF;
  ka[tid] = TG_KEY_INF;
  kc[tid] = TG_KEY_INF;
  __syncthreads();
#pragma unroll
  for (int b = 0; b < NBLK; ++b) {
    const int d = __builtin_amdgcn_readlane(blocks, w + 4 * b);
    if (d != LJ_NONE) lj_block_minima(d >> 8, d & 255, acc[b], ids, nn, nA, nB, kb, ka, kc);
  }
  __syncthreads();
  const int ir = 16 * w + 4 * g + (t & 3), tile = t >> 2;  // this lane's row jobs (lj_push)
  const uint64_t row_b = kb[4 * ir + tile], row_a = ka[4 * ir + tile], col_b = kc[64 * w + l];
  lj_push(a, ids, ids + 64, wd, wd + 64, nA, nB, w, g, t, l, row_b, row_a, col_b, kc);
  if (a.counters && tid == 0)
    atomicAdd(&cnt_slot(a.counters)[0], (unsigned long long)(nA * nB + nA * (nA - 1) / 2));
}

// -------------------------------------------------------------------------------------
// Screened local join of real-valued data.  PREC 1: FP32 MFMA, 2: 16-bit MFMA (BF: BF16 copy,
// else FP16), 3: FP8 MFMA.  T = uint16_t: rows that BF16 holds exactly.  The jobs are those of
// k_localjoin_exact_screen: a row's minimum over a 16-wide tile, for rows of A over the tiles
// of B and of A, and of B over the tiles of A.  Every 16 x 16 block of pairs holds whole jobs
// of its rows and of its columns (A x A is symmetric: blocks on and above the diagonal only),
// so the valid blocks, at most 26, are dealt to the four waves whatever the list lengths.  Per
// job tau = min(worst, smallest s + E) straight from the accumulators; a pair with s - E <= tau
// in its row's or its column's job is queued, once.  An exact minimum below the job's worst
// distance is always among them, and one that a job did not want cannot be its minimum, so
// every queued pair is offered to both jobs.  The queue is worked by all 16 lane groups:
//   * rows up to 256 elements (MC <= 4): straight from global memory, where the block's rows
//     have just been read (L2);
//   * wider rows: 64 elements of every queued row at a time through LDS, 12 pairs per group
//     with their partial sums in registers -- a row is read once more, not once per pair.
// Two iterations of 500k x 96 (K = 64, learned lists, 150 re-scores per node): 48.5 -> 13.0 ms;
// eight of 160k x 96 clusters from random lists 46 -> 12.8 ms; two of 100k x 960 (170 re-scores
// per node) 48 -> 16.1 ms.  Before, one BF16 product left a bound eight times wider, one of the
// four waves formed the masks, and each re-score read both rows from L2.  What is left: half
// of the narrow kernel's cycles issue VALU work, the rest waits on the list, row and push
// round trips; the wide one streams each sampled row twice.  Waves per SIMD were chosen at 96 and
// 960 elements; at 129 to 256 six spill 44 to 49 vector registers (two iterations of
// 100k x 160: 5.99 ms, 4.03 with four waves and no spills).
// -------------------------------------------------------------------------------------
template <int PREC, int MC, class T, int DC, bool BF>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MC <= 4 ? 6 : 3)))
void k_localjoin_screen(KnnArgs a) {
  using St = ScreenStage<PREC, DC, 128>;
  constexpr int QCAP = 1024;  // pairs queued per pass (one pass, but for degenerate data)
  constexpr bool WIDE = MC > 4;
  constexpr int KEYS = 3 * 256 * 8, QBYTES = QCAP * 2;
  constexpr int WRS = 64 * int(sizeof(T)) + 16;  // staged row of the wide re-scores
  constexpr int WORK = KEYS + QBYTES + (WIDE ? 128 * WRS : 0);
  __shared__ __attribute__((aligned(16))) unsigned char smem[St::BYTES > WORK ? St::BYTES : WORK];
  __shared__ __attribute__((aligned(16))) uint32_t ids[128];
  __shared__ __attribute__((aligned(16))) float nn[128];
  __shared__ __attribute__((aligned(16))) float wd[128];
  __shared__ float qn[PREC == 3 ? 128 : 1], en[PREC == 3 ? 128 : 1], sc[PREC == 3 ? 128 : 1];
  __shared__ uint32_t wsum[4];
  const uint32_t u = row_of_block(a.perm, a.N);
  if (u >= a.N) return;
  const int tid = threadIdx.x, l = tid & 63, g = l >> 4, t = l & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int D = a.D;
  const int nA = a.na[u], nB = a.nb[u];
  uint32_t *A = ids, *B = ids + 64;
  lj_lists(a, u, a.nrm2, nA, nB, A, B, nn, wd, nn + 64, wd + 64);
  if (PREC == 3 && tid < 128) {
    const bool in = tid < 64 ? tid < nA : tid - 64 < nB;
    const uint32_t v = in ? a.H[size_t(u) * HROW_S + tid] : 0u;
    qn[tid] = in ? a.nq[v] : 0.f;
    en[tid] = in ? a.ne[v] : 0.f;
    sc[tid] = in ? a.sc8[v] : 0.f;
  }
  __syncthreads();
  // ---- this wave's blocks
  const int blocks = lj_blocks((nA + 15) >> 4, (nB + 15) >> 4);
  int bi[NBLK], bj[NBLK];
#pragma unroll
  for (int b = 0; b < NBLK; ++b) {
    const int d = __builtin_amdgcn_readlane(blocks, w + 4 * b);
    bi[b] = d == LJ_NONE ? -1 : d >> 8;
    bj[b] = d & 255;
  }
  f32x4 acc[NBLK];
#pragma unroll
  for (int b = 0; b < NBLK; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const void* src = PREC == 3   ? static_cast<const void*>(a.Xq8)
                    : PREC == 2 ? static_cast<const void*>(a.Xb)
                                : static_cast<const void*>(a.X);
  screen_chunks<PREC, DC, 128>(
      src, ids, D, [&](int r) { return r < 64 ? r < nA : r - 64 < nB; }, smem, [&]() {
#pragma unroll
        for (int b = 0; b < NBLK; ++b)
          if (bi[b] >= 0)
            screen_block<PREC, BF, DC>(smem + bi[b] * St::RS, smem + bj[b] * St::RS, l, acc[b]);
      });
  // the jobs' keys and the queue, in the staging area (free from here on)
  uint64_t* kb = reinterpret_cast<uint64_t*>(smem);  // [64 rows of A][4 tiles of B]
  uint64_t* ka = kb + 256;                           // [64 rows of A][4 tiles of A]
  uint64_t* kc = ka + 256;                           // [4 tiles of A][64 rows of B]
  uint16_t* queue = reinterpret_cast<uint16_t*>(kc + 256);  // row << 7 | candidate
  kb[tid] = TG_KEY_INF;
  ka[tid] = TG_KEY_INF;
  kc[tid] = TG_KEY_INF;
  // ---- which pairs to evaluate: bit 4b + r, element r of block b
  const float INF = __uint_as_float(0x7F800000u);
  const float kap = a.kap, ps = a.pscale;
  uint32_t want = 0;
#pragma unroll
  for (int b = 0; b < NBLK; ++b) {
    if (bi[b] < 0) continue;
    const int i0 = bi[b] + 4 * g, jj = bj[b] + t;
    const bool bt = bj[b] >= 64;
    const bool jn = bt ? jj - 64 < nB : jj < nA;
    const float4 ni = *reinterpret_cast<const float4*>(nn + i0);
    const float4 wi = *reinterpret_cast<const float4*>(wd + i0);
    const uint4 idi = *reinterpret_cast<const uint4*>(ids + i0);
    const float nv[4] = {ni.x, ni.y, ni.z, ni.w}, wv[4] = {wi.x, wi.y, wi.z, wi.w};
    const uint32_t iv[4] = {idi.x, idi.y, idi.z, idi.w};
    const float nj = nn[jj], wj = wd[jj];
    const uint32_t idj = ids[jj];
    float lo[4];
    uint32_t hi[4];
    bool ok[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      ok[r] = i0 + r < nA && jn && (bt ? iv[r] != idj : i0 + r != jj);
      const float nsum = nv[r] + nj;
      float h;
      if constexpr (PREC == 3) {
        const int i = i0 + r;
        const float s = nsum - 2.0f * ((sc[i] * sc[jj]) * acc[b][r]);
        const float E = 2.0f * (en[i] * qn[jj] + qn[i] * en[jj] + en[i] * en[jj]) +
                        a.eta * (nsum + 2.0f * qn[i] * qn[jj]);
        lo[r] = s - E;
        h = s + E;
      } else {
        const float s = __builtin_fmaf(-ps, acc[b][r], nsum);
        lo[r] = __builtin_fmaf(-kap, nsum, s);
        h = __builtin_fmaf(kap, nsum, s);
      }
      // non-negative bits order as unsigned integers; +inf where there is no bound
      hi[r] = (ok[r] && h < INF) ? __float_as_uint(fmaxf(h, 0.f)) : 0x7F800000u;
    }
    uint32_t mc = min(min(hi[0], hi[1]), min(hi[2], hi[3]));
    mc = min(mc, lane_xor32(mc, 16));
    mc = min(mc, lane_xor32(mc, 32));
    const float tc = fminf(wj, __uint_as_float(mc));
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float tau = fmaxf(fminf(wv[r], __uint_as_float(row_min16(hi[r]))), tc);
      // on the diagonal a pair appears twice: queued above it
      if (ok[r] && !(lo[r] > tau) && (bi[b] != bj[b] || i0 + r < jj)) want |= 1u << (4 * b + r);
    }
  }
  // ---- queue positions
  const int own = __popc(want);
  const int incl = wave_incl_scan(own);
  if (l == 63) wsum[w] = uint32_t(incl);
  __syncthreads();
  int first = incl - own, total = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (q < w) first += int(wsum[q]);
    total += int(wsum[q]);
  }
  const T* X = reinterpret_cast<const T*>(std::is_same<T, uint16_t>::value
                                              ? static_cast<const void*>(a.Xr16)
                                              : static_cast<const void*>(a.X));
  // offers pair (i, x)'s distance to its two jobs
  auto offer = [&](uint32_t e, float d) {
    const int i = int(e >> 7), x = int(e & 127u);
    auto put = [](uint64_t* k, uint64_t v) {
      atomicMin(reinterpret_cast<unsigned long long*>(k), (unsigned long long)v);
    };
    const uint64_t ki = mk_key(d, ids[x]), kx = mk_key(d, ids[i]);
    if (x >= 64) {
      put(&kb[4 * i + ((x - 64) >> 4)], ki);
      put(&kc[64 * (i >> 4) + (x - 64)], kx);
    } else {
      put(&ka[4 * i + (x >> 4)], ki);
      put(&ka[4 * x + (i >> 4)], kx);
    }
  };
  for (int q0 = 0; q0 < total; q0 += QCAP) {
    const int n = min(total - q0, QCAP);
    uint32_t m = want;
    int pos = first - q0;
    while (ballot(m != 0) != 0) {
      const int p = m ? __ffs(m) - 1 : 0;
      const int d = __shfl(blocks, w + (p & ~3), TG_WAVE);  // block of element p
      if (m && pos >= 0 && pos < QCAP)
        queue[pos] = uint16_t(((d >> 8) + 4 * g + (p & 3)) << 7 | ((d & 255) + t));
      pos += m ? 1 : 0;
      m &= m - 1;
    }
    __syncthreads();
    const int gg = tid >> 4;
    if constexpr (!WIDE) {
      constexpr int NB = 2;  // pairs in flight per group: more would cost waves per SIMD
      for (int e0 = 0; e0 < n; e0 += 16 * NB) {
        uint32_t ent[NB];
        const T *ra[NB], *rb[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int e = e0 + gg + 16 * b;
          ent[b] = queue[e < n ? e : 0];
          ra[b] = X + size_t(ids[ent[b] >> 7]) * D;
          rb[b] = X + size_t(ids[ent[b] & 127u]) * D;
        }
        float dd[NB];
        dist16_pairs<MC, NB>(ra, rb, D, t, dd);
        // the group's lane b takes pair b (the distances are in lane 0)
        const float d1 = row_shr<1>(dd[1]);
        if (t < NB && e0 + gg + 16 * t < n) offer(t == 0 ? ent[0] : ent[1], t == 0 ? dd[0] : d1);
      }
    } else {
      // 64 elements of every row at a time; pass p0 holds pairs p0 + gg + 16 k in group gg.  PK:
      // what three waves per SIMD keep in registers; a second pass for nodes with more than 192
      // pairs costs less than spills (learned build of 100k x 960, PK 8 / 10 / 12 / 16 / 20:
      // 32.7 / 32.2 / 32.2 / 33.5 / 44.0 ms; 60k x 288 from random lists, 12 / 16: 16.3 / 19.4)
      constexpr int PK = 12;
      constexpr int PPR = 64 * int(sizeof(T)) / 16, NP = 128 * PPR / 256;
      unsigned char* stage = smem + KEYS + QBYTES;
      for (int p0 = 0; p0 < n; p0 += 16 * PK) {
        uint32_t ent[PK];
        float p[PK][4];
#pragma unroll
        for (int k = 0; k < PK; ++k) {
          const int e = p0 + gg + 16 * k;
          ent[k] = queue[e < n ? e : p0];
          p[k][0] = p[k][1] = p[k][2] = p[k][3] = 0.f;
        }
        const int nk = (min(n - p0, 16 * PK) + 15) >> 4;  // pairs per group in this pass
        uint4 v[NP];
        auto load = [&](int d0) {
#pragma unroll
          for (int q = 0; q < NP; ++q) {
            const int e = tid + 256 * q, r = e / PPR, col = d0 + (e % PPR) * (16 / int(sizeof(T)));
            v[q] = make_uint4(0u, 0u, 0u, 0u);
            if ((r < 64 ? r < nA : r - 64 < nB) && col < D)
              v[q] = *reinterpret_cast<const uint4*>(X + size_t(ids[r]) * D + col);
          }
        };
        load(0);
        for (int d0 = 0; d0 < D; d0 += 64) {
#pragma unroll
          for (int q = 0; q < NP; ++q) {
            const int e = tid + 256 * q;
            *reinterpret_cast<uint4*>(stage + (e / PPR) * WRS + (e % PPR) * 16) = v[q];
          }
          __syncthreads();
          if (d0 + 64 < D) load(d0 + 64);
          const bool in = d0 + 4 * t < D;
#pragma unroll
          for (int k = 0; k < PK; ++k) {
            if (k < nk) {
              const T* xa = reinterpret_cast<const T*>(stage + (ent[k] >> 7) * WRS) + 4 * t;
              const T* xb = reinterpret_cast<const T*>(stage + (ent[k] & 127u) * WRS) + 4 * t;
              const float4 xv = load4(xa), yv = load4(xb);
              if (in) fold4(xv, yv, p[k]);
            }
          }
          __syncthreads();
        }
#pragma unroll
        for (int k = 0; k < PK; ++k) {
          if (k < nk) {
            const float d = tree16(p[k][0], p[k][1], p[k][2], p[k][3]);
            if (t == 0 && p0 + gg + 16 * k < n) offer(ent[k], d);
          }
        }
      }
    }
    __syncthreads();
  }
  const int ir = 16 * w + 4 * g + (t & 3), tile = t >> 2;  // this lane's row jobs (lj_push)
  const uint64_t row_b = kb[4 * ir + tile], row_a = ka[4 * ir + tile], col_b = kc[64 * w + l];
  lj_push(a, A, B, wd, wd + 64, nA, nB, w, g, t, l, row_b, row_a, col_b, kc);
  if (a.counters && tid == 0) {
    // [0] pair evaluations (screen), [1] exact re-scores
    atomicAdd(&cnt_slot(a.counters)[0], (unsigned long long)(nA * nB + nA * (nA - 1) / 2));
    atomicAdd(&cnt_slot(a.counters)[1], (unsigned long long)total);
  }
}

// Staged bytes per row and round, tile 0 / 1: rows up to 256 elements 64 / 128 (little LDS and
// few registers, so eight waves per SIMD, and D = 96 is whole rounds: 500k x 96, two
// iterations, 17.0 / 17.9 ms before the dealt blocks), wider rows 128 / 64 (half the rounds and barriers; their
// re-scores hold the LDS anyway: 100k x 960 15.1 / 18.9 ms; 256 bytes per round 17.0 ms).
void launch_knn_localjoin_screen(const KnnArgs& a, int precision, int tile, hipStream_t s) {
  if (a.exact_screen && (precision == KP_BF16 || precision == KP_FP32)) {
    const dim3 grid(grid_rows(a.perm, a.N));
    if (a.X8 && a.n2s && a.D <= 256) {
      // u8 data: the products on int8 MFMA, exact as the FP32 and BF16 ones are
      if (a.D <= 128) k_localjoin_exact_screen<0, 128><<<grid, 256, 0, s>>>(a);
      else k_localjoin_exact_screen<0, 256><<<grid, 256, 0, s>>>(a);
    } else if (precision == KP_BF16) {
      // 256-byte staged rows (128 BF16 / 64 FP32 elements), 64-byte rows with tile 1
      if (tile == 1) k_localjoin_exact_screen<2, 32><<<grid, 256, 0, s>>>(a);
      else k_localjoin_exact_screen<2, 128><<<grid, 256, 0, s>>>(a);
    } else {
      if (tile == 1) k_localjoin_exact_screen<1, 16><<<grid, 256, 0, s>>>(a);
      else k_localjoin_exact_screen<1, 64><<<grid, 256, 0, s>>>(a);
    }
    return;
  }
  const int mc = (int(a.D) + 63) / 64;
#define LJS(P, M, T, DC, BF) \
  k_localjoin_screen<P, M, T, DC, BF><<<grid_rows(a.perm, a.N), 256, 0, s>>>(a)
#define LJS_DC(P, M, T, BF)                                                  \
  do {                                                                       \
    constexpr int near_ = (P == 3 ? 64 : P == 2 ? 32 : 16);                  \
    if ((tile == 1) == (M > 4)) LJS(P, M, T, near_, BF);                     \
    else LJS(P, M, T, 2 * near_, BF);                                        \
  } while (0)
#define LJS_MC(P, T, BF)                                                   \
  do {                                                                     \
    if (mc <= 2) LJS_DC(P, 2, T, BF);                                      \
    else if (mc <= 4) LJS_DC(P, 4, T, BF);                                 \
    else LJS_DC(P, 16, T, BF);                                             \
  } while (0)
  if (precision == KP_FP8) {
    if (a.Xr16) LJS_MC(3, uint16_t, false); else LJS_MC(3, float, false);
  } else if (precision == KP_BF16) {
    if (a.Xr16) LJS_MC(2, uint16_t, true);
    else if (a.copy_bf16) LJS_MC(2, float, true);
    else LJS_MC(2, float, false);
  } else {
    if (a.Xr16) LJS_MC(1, uint16_t, false); else LJS_MC(1, float, false);
  }
#undef LJS_MC
#undef LJS_DC
#undef LJS
}

}  // namespace tg
