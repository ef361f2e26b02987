// General-index attention kernels with the Metal kernels' semantics, and the
// relative index table.
//
// Reference: FusedKernels.swift:13-81 (fused attention) and :83-123 (relative
// bias), launched at :160-258; the index math DeBERTa.swift:498-551.  These
// take the c2p / p2c index tables as inputs (any indices, bounds-checked) and
// back the FusedKernels-shaped entry points.  The encoder itself runs the
// staged kernel of deberta_attention.hip, which derives the indices from the
// bucket function directly.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <initializer_list>
#include <type_traits>

#include "gd_common.hpp"
#include "gd_kernels.hpp"

namespace gd {
namespace {

// ---------------------------------------------------------------------------
// General-index kernels with the Metal kernels' semantics (API parity).
// One wave64 per (b, h, query); lanes stride over keys (scores) and then over
// the head dimension (context).  fp32 arithmetic throughout, as the reference.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(64) void relative_bias_general_kernel(
    const half_t* __restrict__ q, const half_t* __restrict__ k, const half_t* __restrict__ pos_key,
    const half_t* __restrict__ pos_query, const int32_t* __restrict__ c2p_idx, const int32_t* __restrict__ p2c_idx,
    const half_t* __restrict__ key_mask, float scale, int H, int L, int D, int P, half_t* __restrict__ out,
    int32_t* __restrict__ error_flag) {
  extern __shared__ float qcache[];
  const int row = blockIdx.x;  // (b*H + h)*L + query
  const int query = row % L;
  const int h = (row / L) % H;
  const int b = row / (H * L);
  const int lane = threadIdx.x;
  const half_t* qrow = q + (int64_t)row * D;
  for (int d = lane; d < D; d += 64) qcache[d] = (float)qrow[d];
  __syncthreads();
  for (int key = lane; key < L; key += 64) {
    const half_t* krow = k + (((int64_t)b * H + h) * L + key) * D;
    int ci = c2p_idx[((int64_t)h * L + query) * L + key];
    int pi = p2c_idx[((int64_t)h * L + key) * L + query];
    if (ci < 0 || ci >= P || pi < 0 || pi >= P) {
      if (error_flag) atomicOr(error_flag, 1);
      ci = ci < 0 ? 0 : (ci >= P ? P - 1 : ci);
      pi = pi < 0 ? 0 : (pi >= P ? P - 1 : pi);
    }
    const half_t* pk = pos_key + ((int64_t)h * P + ci) * D;
    const half_t* pq = pos_query + ((int64_t)h * P + pi) * D;
    float c2p = 0.f, p2c = 0.f;
    for (int d = 0; d < D; ++d) {
      const float kd = (float)krow[d];
      c2p += qcache[d] * (float)pk[d];
      p2c += kd * (float)pq[d];
    }
    float score = (c2p + p2c) * scale;
    if ((float)key_mask[(int64_t)b * L + key] < -60000.f) score = -65504.f;
    out[(int64_t)row * L + key] = (half_t)score;
  }
}

__global__ __launch_bounds__(64) void fused_attention_general_kernel(
    const half_t* __restrict__ q, const half_t* __restrict__ k, const half_t* __restrict__ v,
    const half_t* __restrict__ pos_key, const half_t* __restrict__ pos_query, const int32_t* __restrict__ c2p_idx,
    const int32_t* __restrict__ p2c_idx, const half_t* __restrict__ key_mask, float scale, int H, int L, int D, int P,
    half_t* __restrict__ out, int32_t* __restrict__ error_flag) {
  extern __shared__ float shm[];  // D floats of q, then L weights
  float* qcache = shm;
  float* weights = shm + D;
  const int row = blockIdx.x;
  const int query = row % L;
  const int h = (row / L) % H;
  const int b = row / (H * L);
  const int lane = threadIdx.x;
  const half_t* qrow = q + (int64_t)row * D;
  for (int d = lane; d < D; d += 64) qcache[d] = (float)qrow[d];
  __syncthreads();
  float local_max = -65504.f;
  for (int key = lane; key < L; key += 64) {
    const half_t* krow = k + (((int64_t)b * H + h) * L + key) * D;
    int ci = c2p_idx[((int64_t)h * L + query) * L + key];
    int pi = p2c_idx[((int64_t)h * L + key) * L + query];
    if (ci < 0 || ci >= P || pi < 0 || pi >= P) {
      if (error_flag) atomicOr(error_flag, 1);
      ci = ci < 0 ? 0 : (ci >= P ? P - 1 : ci);
      pi = pi < 0 ? 0 : (pi >= P ? P - 1 : pi);
    }
    const half_t* pk = pos_key + ((int64_t)h * P + ci) * D;
    const half_t* pq = pos_query + ((int64_t)h * P + pi) * D;
    float qk = 0.f, c2p = 0.f, p2c = 0.f;
    for (int d = 0; d < D; ++d) {
      const float kd = (float)krow[d];
      qk += qcache[d] * kd;
      c2p += qcache[d] * (float)pk[d];
      p2c += kd * (float)pq[d];
    }
    float score = (qk + c2p + p2c) * scale;
    if ((float)key_mask[(int64_t)b * L + key] < -60000.f) score = -65504.f;
    weights[key] = score;
    local_max = fmaxf(local_max, score);
  }
  const float gmax = wave_max(local_max);
  float local_sum = 0.f;
  for (int key = lane; key < L; key += 64) local_sum += expf(weights[key] - gmax);
  const float gsum = wave_sum(local_sum);
  for (int key = lane; key < L; key += 64) weights[key] = expf(weights[key] - gmax) / gsum;
  __syncthreads();
  for (int d = lane; d < D; d += 64) {
    float acc = 0.f;
    for (int key = 0; key < L; ++key) acc += weights[key] * (float)v[(((int64_t)b * H + h) * L + key) * D + d];
    out[(((int64_t)b * L + query) * H + h) * D + d] = (half_t)acc;
  }
}

// ---------------------------------------------------------------------------
// The relative bias with index tensors on the matrix cores (D = 64, L <= 512,
// any length, P <= 65536).  A workgroup of 4 waves owns 64 queries x 64 keys
// of one head and walks `nb` batch rows: the index tensors and the position
// tables do not depend on the batch row, so a wave reads its indices and its
// table rows once, keeps the rows as MFMA fragments and the scores' table
// offsets in registers, and per batch row brings only Q and K.
//
// Relative-position indices of 16 x 64 positions span at most 79 rows, so
// from exactly the least index on five 16-row tiles of posK serve the c2p
// terms of a wave's 16 queries, and five of posQ the p2c terms of its 16 keys:
// C2P = Q . posK^T and P2C = K . posQ^T (v_mfma_f32_16x16x32_f16, fp32) go
// through LDS tables of 80 columns, and each score takes one term from each at
// its index.  C2P rows are read by the wave that writes them; P2C rows by all
// four, so they alternate between two tables with one barrier per batch row.
// Wider spans (arbitrary index tensors) run windows of 128 or 192 table rows, a
// position outside the window at hand reading a -0 column.  A score is (-0 +
// c2p) + p2c, term by term the reference's fp32 sum.  Indices outside [0, P)
// are clamped, as the per-query kernel does.  Queries and keys past L repeat
// the last one (indices of a valid pair of the tile); their scores are not
// stored.
//
// A workgroup of one batch row uses a table row once, so it takes the rows
// through LDS in whole lines, one window of 128 for all four waves: a fragment
// load from global memory touches 16 half lines for every 16 lanes (64 address
// lookups a wave), which bound that form at 3.3 us per workgroup and CU (B = 1,
// H = 16, L = 512: 18.1 us so, 14.5 through LDS; L = 256: 6.4 and 6.0).
//
// Several batch rows are bound by the batch row's chain (MFMA, table, gather,
// barrier, store) with two waves per SIMD (254 VGPRs).  B = 32, H = 16, L =
// 256: 36 us against 71 us of a kernel that read indices and table rows for
// every batch row and ran 64-row windows of either table, a gather per window;
// at 5 TB/s its 111 MB take 22 us.  Random indices (the whole table for every
// tile): B = 1, L = 64 to 512 13.0 to 32.5 us, B = 32, L = 256 199 us (that
// kernel 18.6 to 33.7 and 184; each wave reading its own windows of 80 rows
// from global memory 27 to 88 and 540).
// ---------------------------------------------------------------------------
constexpr int64_t kGenCus = 256;  // compute units of the device the grids are sized for
constexpr int kGenKeyBlocks = 4;  // 16-key blocks per key block (64 keys)
constexpr int kBiasTiles = 5;     // 16-row tiles of a table window
constexpr int kBiasCols = 16 * kBiasTiles;
// fp32 row stride of the tables: float4 stores of 8 consecutive rows hit 32
// distinct banks; column kBiasCols holds the -0 of a position outside the window.
constexpr int kBiasStride = kBiasCols + 4;

constexpr int kGenWin = 128;  // table rows per window in LDS

// 64-half rows in LDS: 16-byte chunk `chunk` of row `row`.
__device__ __forceinline__ int gen_swz(int row, int chunk) { return row * 64 + ((chunk ^ ((row >> 1) & 7)) << 3); }

// Least of a wave's values (VALU moves, no LDS round trips).
template <int CTRL>
__device__ __forceinline__ int gen_dpp(int v) { return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false); }
__device__ __forceinline__ int gen_wave_min(int v) {
  v = min(v, gen_dpp<0xB1>(v));   // quad_perm [1,0,3,2]
  v = min(v, gen_dpp<0x4E>(v));   // quad_perm [2,3,0,1]
  v = min(v, gen_dpp<0x141>(v));  // row_half_mirror
  v = min(v, gen_dpp<0x140>(v));  // row_mirror
  return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// Workgroups per CU (waves per SIMD) the registers and LDS are held to.
constexpr int bias_waves(bool multi) { return multi ? 2 : 3; }

// W: the largest of 8, 4, 2 and 1 that divides L, the halfs of the output
// pieces (every row starts aligned to one); from 4 on the c2p indices and the
// mask of four consecutive keys are one aligned load.  MULTI: the workgroup
// walks several batch rows.  With one there is nothing to keep: P2C takes the
// C2P rows' place, and three workgroups share a CU.
template <int W, bool MULTI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(bias_waves(MULTI), bias_waves(MULTI)))) void relative_bias_mfma_kernel(
    const half_t* __restrict__ q, const half_t* __restrict__ k, const half_t* __restrict__ pos_key,
    const half_t* __restrict__ pos_query, const int32_t* __restrict__ c2p_idx, const int32_t* __restrict__ p2c_idx,
    const half_t* __restrict__ key_mask, float scale, int B, int H, int L, int P, int nb, half_t* __restrict__ out) {
  constexpr int KB = kGenKeyBlocks;
  constexpr bool VEC = W >= 4;
  // C2P [query][column] and P2C [key][column]: MULTI keeps two tables of the
  // latter, in an array of their own (so that their stores and C2P's reads may
  // pass each other); with one batch row P2C takes C2P's place, and a window
  // of posK rows and one of posQ rows follow.  Wide spans: a window of kWin
  // rows, and one table of kWin columns.
  constexpr int kTab = 64 * kBiasStride, kRows = kGenWin * 64 / 2;  // floats
  constexpr int kWin = MULTI ? 192 : kGenWin, kWideStride = kWin + 4;
  constexpr int kWideRows = kWin * 64 / 2, kWideTab = 64 * kWideStride;
  constexpr int kOneRow = kTab + 2 * kRows > kWideRows + kWideTab ? kTab + 2 * kRows : kWideRows + kWideTab;
  __shared__ __attribute__((aligned(1024))) float ctab[!MULTI ? kOneRow : kTab > kWideRows ? kTab : kWideRows];
  __shared__ __attribute__((aligned(16))) float ptabs[!MULTI ? 4 : 2 * kTab > kWideTab ? 2 * kTab : kWideTab];
  auto ptab = [&](int i) -> float* { return MULTI ? ptabs + i * kTab : ctab; };
  __shared__ int ranges[4][2 + 2 * KB];  // per wave: least c2p, -c2p, then p2c and -p2c of each 16-key block
  // Workgroup -> (h, 64-query block qb, key block ky, batch rows b0 ..).
  // Workgroups go to the 8 XCDs round-robin; with H a multiple of 8, XCD x
  // takes heads x H / 8 .. (x + 1) H / 8 - 1 only, so its L2 holds just those
  // heads' index tensors and position tables.
  const int nq = (L + 63) / 64;
  int h, qb, ky, b0;
  {
    const int w = blockIdx.x;
    int r;
    if (H % 8 == 0) {
      const int hx = H / 8, l = w >> 3;
      h = (w & 7) * hx + l % hx;
      r = l / hx;
    } else {
      h = w % H;
      r = w / H;
    }
    qb = r % nq;
    r /= nq;
    ky = r % nq;
    b0 = r / nq * nb;
  }
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lc = lane & 15, g = lane >> 4;
  const int qw = qb * 64 + 16 * wave;            // the wave's first query
  const int qr = qw + lc < L ? qw + lc : L - 1;  // this lane's query (keys 4 g .. 4 g + 3 of a block)
  const int kw = 64 * ky + 16 * wave + lc;       // this lane's key of the wave's P2C rows
  const int kr = kw < L ? kw : L - 1;
  const half_t* pkh = pos_key + (int64_t)h * P * 64;
  const half_t* pqh = pos_query + (int64_t)h * P * 64;
  const int32_t* c2ph = c2p_idx + (int64_t)h * L * L;
  const int32_t* p2ch = p2c_idx + (int64_t)h * L * L;
  auto clampi = [&](int x) { return x < 0 ? 0 : (x >= P ? P - 1 : x); };
  auto key_of = [&](int kb) { return 64 * ky + 16 * kb + 4 * g; };  // this lane's first key of block kb
  auto row_frags = [&](const half_t* base, int row, half8_t (&f)[2]) {
    f[0] = *reinterpret_cast<const half8_t*>(base + (uint32_t)(row * 64 + 8 * g));
    f[1] = *reinterpret_cast<const half8_t*>(base + (uint32_t)(row * 64 + 32 + 8 * g));
  };
  // Of one batch row: fragments of this wave's queries and of its P2C keys,
  // the mask of this lane's keys.
  struct Row {
    half8_t q[2], k[2];
    half4_t mask[KB];
  };
  auto fetch_mask = [&](int b, half4_t (&mask)[KB]) {
    const half_t* mrow = key_mask + (int64_t)b * L;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int key = key_of(kb);
      if constexpr (VEC) {
        mask[kb] = *reinterpret_cast<const half4_t*>(mrow + (uint32_t)(key < L ? key : L - 4));
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) mask[kb][j] = mrow[(uint32_t)(key + j < L ? key + j : L - 1)];
      }
    }
  };
  auto fetch = [&](int b, Row& x) {
    const int64_t bh = (int64_t)b * H + h;
    row_frags(q + bh * L * 64, qr, x.q);
    row_frags(k + bh * L * 64, kr, x.k);
    fetch_mask(b, x.mask);
  };

  // ---- once: indices, their ranges, table rows ----
  int ci[KB][4], pi[KB][4];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int key = key_of(kb);
    if constexpr (VEC) {
      const int kc = key < L ? key : L - 4;
      const int4 x = *reinterpret_cast<const int4*>(c2ph + (uint32_t)(qr * L + kc));
      ci[kb][0] = x.x, ci[kb][1] = x.y, ci[kb][2] = x.z, ci[kb][3] = x.w;
#pragma unroll
      for (int j = 0; j < 4; ++j) pi[kb][j] = p2ch[(uint32_t)((kc + j) * L + qr)];
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int kc = key + j < L ? key + j : L - 1;
        ci[kb][j] = c2ph[(uint32_t)(qr * L + kc)];
        pi[kb][j] = p2ch[(uint32_t)(kc * L + qr)];
      }
    }
  }
  // Fragments of the 16-row tile of a table from row `row0` on (rows past P
  // repeat row P - 1).
  auto tile_frags = [&](const half_t* table, int row0, half8_t (&f)[2]) {
    row_frags(table, row0 + lc < P ? row0 + lc : P - 1, f);
  };
  // A window of table rows from row `base` on, in whole lines through
  // registers into LDS, and the 16-row tile there from its row r0 on.
  auto fetch_window = [&](const half_t* table, int base, half8_t (&x)[kWin / 32]) {
#pragma unroll
    for (int i = 0; i < kWin / 32; ++i) {
      const int row = base + 32 * i + (int)(threadIdx.x >> 3);
      x[i] = *reinterpret_cast<const half8_t*>(table + (uint32_t)((row < P ? row : P - 1) * 64 + 8 * (threadIdx.x & 7)));
    }
  };
  auto put_window = [&](const half8_t (&x)[kWin / 32], float* rows) {
#pragma unroll
    for (int i = 0; i < kWin / 32; ++i)
      *reinterpret_cast<half8_t*>(reinterpret_cast<half_t*>(rows) + gen_swz(32 * i + (int)(threadIdx.x >> 3), threadIdx.x & 7)) =
          x[i];
  };
  auto window_frags = [&](const float* rows, int r0, half8_t (&f)[2]) {
    f[0] = *reinterpret_cast<const half8_t*>(reinterpret_cast<const half_t*>(rows) + gen_swz(r0 + lc, g));
    f[1] = *reinterpret_cast<const half8_t*>(reinterpret_cast<const half_t*>(rows) + gen_swz(r0 + lc, 4 + g));
  };
  half8_t ct[kBiasTiles][2], pt[kBiasTiles][2];  // MULTI only
  uint32_t cp[KB][4];  // the clamped indices, c2p | p2c << 16
  auto c_of = [](uint32_t x) { return (int)(x & 0xFFFFu); };
  auto p_of = [](uint32_t x) { return (int)(x >> 16); };
  Row cur, nxt;
  if constexpr (MULTI && VEC) fetch(b0, nxt);  // (the others would spill)
  {
    int c_mn = P, c_mx = 0, p_mn[KB], p_mx[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      p_mn[kb] = P, p_mx[kb] = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        ci[kb][j] = clampi(ci[kb][j]), pi[kb][j] = clampi(pi[kb][j]);
        c_mn = min(c_mn, ci[kb][j]), c_mx = max(c_mx, ci[kb][j]);
        p_mn[kb] = min(p_mn[kb], pi[kb][j]), p_mx[kb] = max(p_mx[kb], pi[kb][j]);
        cp[kb][j] = (uint32_t)ci[kb][j] | ((uint32_t)pi[kb][j] << 16);
      }
    }
    int r[2 + 2 * KB];
    r[0] = gen_wave_min(c_mn), r[1] = gen_wave_min(-c_mx);
    // the c2p rows need no other wave's range: in flight from here
#pragma unroll
    for (int tp = 0; MULTI && tp < kBiasTiles; ++tp) tile_frags(pkh, r[0] + 16 * tp, ct[tp]);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) r[2 + 2 * kb] = gen_wave_min(p_mn[kb]), r[3 + 2 * kb] = gen_wave_min(-p_mx[kb]);
    if (lane == 0) {
#pragma unroll
      for (int i = 0; i < 2 + 2 * KB; ++i) ranges[wave][i] = r[i];
    }
  }
  stage_barrier();
  // least index of the wave's c2p, of every wave's and of each block's p2c,
  // and the greatest
  int c_lo = 0, c_all = P, c_end = 0;
  int p_lo[KB], p_all = P, p_end = 0;
  bool narrow = true;  // uniform over the workgroup: every window is one
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const int lo = __builtin_amdgcn_readfirstlane(ranges[w][0]), hi = -__builtin_amdgcn_readfirstlane(ranges[w][1]);
    narrow = narrow && hi - lo < kBiasCols;
    if (w == wave) c_lo = lo;
    c_all = min(c_all, lo), c_end = max(c_end, hi);
  }
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    int lo = P, hi = P;
#pragma unroll
    for (int w = 0; w < 4; ++w) lo = min(lo, ranges[w][2 + 2 * kb]), hi = min(hi, ranges[w][3 + 2 * kb]);
    p_lo[kb] = __builtin_amdgcn_readfirstlane(lo);
    hi = -__builtin_amdgcn_readfirstlane(hi);
    narrow = narrow && hi - p_lo[kb] < kBiasCols;
    p_all = min(p_all, p_lo[kb]), p_end = max(p_end, hi);
  }
  if constexpr (!MULTI) {
    narrow = narrow && c_end - c_all < kGenWin && p_end - p_all < kGenWin;
    // (a wave's tiles stay inside the workgroup's window)
    c_lo = min(c_lo, c_all + kGenWin - kBiasCols);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) p_lo[kb] = min(p_lo[kb], p_all + kGenWin - kBiasCols);
  }
  // One tile's products into a table row's columns.
  auto product = [&](const half8_t (&a)[2], const half8_t (&f)[2], float* row, int tp) {
    float4_t r = {0.f, 0.f, 0.f, 0.f};
    r = mfma16x16x32(a[0], f[0], r);
    r = mfma16x16x32(a[1], f[1], r);  // lane: row lc, columns 16 tp + 4 g + i
    *reinterpret_cast<float4_t*>(row + 16 * tp + 4 * g) = r;
  };
  float* const crow = ctab + (16 * wave + lc) * kBiasStride;
  const int b_end = !MULTI ? b0 + 1 : (b0 + nb < B ? b0 + nb : B);

  auto await_next = [&] {
    asm volatile("" : "+v"(nxt.q[0]), "+v"(nxt.q[1]), "+v"(nxt.k[0]), "+v"(nxt.k[1]));
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) asm volatile("" : "+v"(nxt.mask[kb]));
  };

  // ---- scores: (c2p + p2c) * scale, masked keys -65504, staged through the
  // wave's table rows into row pieces of up to 128 bytes ----
  auto finish = [&](auto prefetched, int b, const float (&acc)[KB][4], const half4_t (&mask)[KB], float* own) {
    half_t* const stage = reinterpret_cast<half_t*>(own);
    wave_lds_sync();
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      half4_t sv;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        sv[j] = (float)mask[kb][j] < -60000.f ? (half_t)-65504.f : (half_t)(acc[kb][j] * scale);
      *reinterpret_cast<half4_t*>(stage + lc * (2 * kBiasStride) + 16 * kb + 4 * g) = sv;
    }
    wave_lds_sync();
    typedef _Float16 piece_t __attribute__((ext_vector_type(W)));
    constexpr int PER = 16 * KB / W, ROWS = 64 / PER;  // pieces per row, rows per store
    const int r = lane / PER, cc = lane % PER * W;
    const uint32_t off = (uint32_t)(r * L + 64 * ky + cc);
    half_t* const orow = out + (((int64_t)b * H + h) * L + qw) * L;  // uniform
    // (the next batch row's loads are waited for here: behind the stores, the
    // wait would be for the stores too)
    if constexpr (decltype(prefetched)::value) await_next();
#pragma unroll
    for (int r0 = 0; r0 < 16; r0 += ROWS)
      if (qw + r0 + r < L && 64 * ky + cc < L)
        *reinterpret_cast<piece_t*>(orow + (int64_t)r0 * L + off) =
            *reinterpret_cast<const piece_t*>(stage + (r0 + r) * (2 * kBiasStride) + cc);
    wave_lds_sync();
  };

  if (narrow) {
    int p_own = p_lo[0];
#pragma unroll
    for (int kb = 1; kb < KB; ++kb) p_own = wave == kb ? p_lo[kb] : p_own;
    if constexpr (!(MULTI && VEC)) fetch(b0, nxt);
    if constexpr (MULTI) {
#pragma unroll
      for (int tp = 0; tp < kBiasTiles; ++tp) tile_frags(pqh, p_own + 16 * tp, pt[tp]);
      // (used here, so that they are waited for here: a wait inside the loop
      // would also wait for the next batch row's loads, issued after them)
#pragma unroll
      for (int tp = 0; tp < kBiasTiles; ++tp)
        asm volatile("" : "+v"(ct[tp][0]), "+v"(ct[tp][1]), "+v"(pt[tp][0]), "+v"(pt[tp][1]));
      await_next();
    } else {
      half8_t x[kWin / 32], y[kWin / 32];
      fetch_window(pkh, c_all, x), fetch_window(pqh, p_all, y);
      put_window(x, ctab + kTab), put_window(y, ctab + kTab + kRows);
      stage_barrier();
    }
    int pbuf = 0;
    for (int b = b0; b < b_end; ++b) {  // uniform
      cur = nxt;
      if (b + 1 < b_end) fetch(b + 1, nxt);
      float* const pt_b = ptab(pbuf);
      float* const prow = pt_b + (16 * wave + lc) * kBiasStride;
      // one table's tiles against the wave's rows: from registers, or from row r0 of a window on
      auto products = [&](const half8_t (&f)[kBiasTiles][2], const float* rows, int r0, const half8_t (&a)[2], float* row) {
#pragma unroll
        for (int tp = 0; tp < kBiasTiles; ++tp) {
          if constexpr (MULTI) {
            product(f[tp], a, row, tp);
          } else {
            half8_t x[2];
            window_frags(rows, r0 + 16 * tp, x);
            product(x, a, row, tp);
          }
        }
      };
      products(ct, ctab + kTab, c_lo - c_all, cur.q, crow);
      if constexpr (MULTI) products(pt, nullptr, 0, cur.k, prow);
      wave_lds_sync();
      float acc[KB][4];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[kb][j] = crow[c_of(cp[kb][j]) - c_lo];
      if constexpr (!MULTI) {
        wave_lds_sync();
        products(pt, ctab + kTab + kRows, p_own - p_all, cur.k, prow);
      }
      stage_barrier();  // P2C rows visible; the last batch row's P2C reads are a barrier back
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[kb][j] += pt_b[(16 * kb + 4 * g + j) * kBiasStride + (p_of(cp[kb][j]) - p_lo[kb])];
      if constexpr (!MULTI) stage_barrier();  // the scores are staged in the rows that were read
      finish(std::bool_constant<MULTI>{}, b, acc, cur.mask, ctab + 16 * wave * kBiasStride);
      pbuf ^= 1;
    }
  } else {
    // Wide spans: windows of kWin rows of either table in turn, a position
    // outside the window at hand reading a -0 column.  Wave w takes the
    // window's tiles w, w + 4, .. against all 64 queries or keys, so that a
    // table row is read once for the workgroup, and the next window comes during
    // the products and the gather.
    float* const wtab = MULTI ? ptabs : ctab + kWideRows;
    half8_t x[kWin / 32];
    auto windows = [&](const half_t* table, int lo, int end, const half_t* base, int row0, auto&& gather) {
      // (opaque: with both tables' fragments and addresses hoisted out of the
      // loops, registers would spill)
      int row = row0 + lc;
      asm volatile("" : "+v"(row));
      half8_t r64[4][2];
#pragma unroll
      for (int u = 0; u < 4; ++u) row_frags(base, row + 16 * u < L ? row + 16 * u : L - 1, r64[u]);
      fetch_window(table, lo, x);
      if (MULTI) put_window(x, ctab);
      for (int w0 = lo; w0 <= end; w0 += kWin) {  // uniform
        if (!MULTI) put_window(x, ctab);
        stage_barrier();  // (and every wave is past the last window's gather)
        if (w0 + kWin <= end) fetch_window(table, w0 + kWin, x);
#pragma unroll
        for (int tp = 0; tp < kWin / 16; tp += 4) {
          if (w0 + 16 * (wave + tp) > end) continue;  // uniform
          half8_t f[2];
          window_frags(ctab, 16 * (wave + tp), f);
#pragma unroll
          for (int u = 0; u < 4; ++u) product(f, r64[u], wtab + (16 * u + lc) * kWideStride, wave + tp);
        }
        stage_barrier();
        // (before the gather where two workgroups share a CU: 199 against 207 us;
        // with three after it: 32 against 34 us)
        if (MULTI && w0 + kWin <= end) put_window(x, ctab);
        gather(w0);
      }
    };
    float* const own = wtab + (16 * wave + lc) * kWideStride;
    for (int b = b0; b < b_end; ++b) {  // uniform
      int zero = 0;  // (opaque, as above)
      asm volatile("" : "+v"(zero));
      zero = __builtin_amdgcn_readfirstlane(zero);
      const int64_t bh = (int64_t)b * H + h;
      float acc[KB][4];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[kb][j] = -0.0f;
      if (lane < 16) own[kWin] = -0.0f;
      windows(pkh, c_all + zero, c_end, q + bh * L * 64, 64 * qb, [&](int w0) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[kb][j] += own[min((uint32_t)(c_of(cp[kb][j]) - w0), (uint32_t)kWin)];
      });
      windows(pqh, p_all + zero, p_end, k + bh * L * 64, 64 * ky, [&](int w0) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[kb][j] += wtab[(16 * kb + 4 * g + j) * kWideStride + min((uint32_t)(p_of(cp[kb][j]) - w0), (uint32_t)kWin)];
      });
      half4_t mask[KB];
      fetch_mask(b, mask);
      stage_barrier();  // the scores are staged in the rows that were read
      finish(std::false_type{}, b, acc, mask, wtab + 16 * wave * kWideStride);
    }
  }
}

// ---------------------------------------------------------------------------
// The fused attention with index tensors on the matrix cores (D = 64, L <=
// 512, any length, P <= 65536).  A workgroup of 4 waves owns (b, h, 64
// queries), wave w queries q0 + 16 w .. + 15, and walks the keys in blocks of
// 64.  C2P and P2C go through an LDS table of 80 columns from the least index
// of the wave's 16 x 64 positions on, as in the bias kernel; here each key
// block needs fresh table rows, so a window of 128 rows of each table (the 64 x
// 64 tile's relative positions span at most 127) comes by DMA for all four
// waves.  Wider spans run windows of 128 rows and columns one after the other,
// the rows in whole lines, the next ones in flight (random indices: B = 1, L =
// 512 97 us, B = 32, L = 256 230 us; 80 columns at a time, each window waited
// for, 153 and 347; 64-row windows in a kernel of four workgroups per CU, 176
// and 249).  Every c2p window precedes every p2c window, so a score accumulates
// (q.k + c2p) + p2c, the reference's fp32 sum, term by term.
//
// Scores (masked keys -65504, keys past L -inf) feed an online softmax per
// query row (running max seeded at -65504, the reference's seed), and P . V
// runs on the matrix cores with the fp32 weights split into fp16 parts (V rows
// in LDS, read transposed by ds_read_b64_tr_b16); the output row is divided by
// the row's sum at the end.  EXACT splits a weight into three parts that hold
// its 24 bits: error against 64 bits beyond the output's rounding, in 2^-24 of
// the sum of |w v|, over lengths 3 to 511 and normal, sharp (4 q), flat and
// cancelling inputs: at most 25, the per-query kernel's 55.  Two parts (22 bits,
// a floor of 2^-25 of the row's largest weight) reach 1,200 on sharp rows.
//
// The next key block's windows, K and V rows come by DMA during the softmax and
// P . V, its indices a block earlier; two barriers per block.
// Bound by the block's chain of LDS round trips with two waves per SIMD (79 KB
// of LDS, 254 VGPRs).  B = 8, H = 16, L = 200 (EXACT): 27.5 us (two
// parts 25.5, P . V in fp32 products 33.6, the per-query kernel 495); B = 32,
// L = 256: 90 us (64-row windows, a gather per window: 97 us).
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(3))) half_t gen_lds_half_t;
typedef short gen_short4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) gen_short4_t gen_lds_short4_t;

// A row of zeros: the V rows of keys past L.
__device__ __attribute__((aligned(16))) const half_t g_zero_row[64] = {};

// VEC: L is a multiple of 4, so the c2p indices and the mask of four
// consecutive keys are one aligned load.  EXACT: P . V takes all 24 bits of
// the weights.
template <bool VEC, bool EXACT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void fused_attention_mfma_kernel(
    const half_t* __restrict__ q, const half_t* __restrict__ k, const half_t* __restrict__ v,
    const half_t* __restrict__ pos_key, const half_t* __restrict__ pos_query, const int32_t* __restrict__ c2p_idx,
    const int32_t* __restrict__ p2c_idx, const half_t* __restrict__ key_mask, float scale, int H, int L, int P,
    half_t* __restrict__ out) {
  constexpr int KB = kGenKeyBlocks;
  // K rows of the key block and windows of posK and posQ rows, whose place the
  // table of kGenWin columns takes with wide spans.
  constexpr int kBlock = 64 * 64, kWideStride = kGenWin + 4;
  __shared__ __attribute__((aligned(1024))) half_t krows[kBlock + 2 * kGenWin * 64];
  half_t* const rk = krows + kBlock;
  half_t* const rq = rk + kGenWin * 64;
  __shared__ __attribute__((aligned(1024))) half_t vrows[2][kBlock];    // V rows of this and the next key block
  static_assert(64 * kWideStride * 2 <= kBlock + 2 * kGenWin * 64 && kGenWin * 64 <= 2 * 64 * kBiasStride, "wide spans fit");
  __shared__ __attribute__((aligned(16))) float tab[64 * kBiasStride];  // C2P [query][col], then P2C [key][col]
  __shared__ int ranges[2][4][2 + 2 * KB];  // per wave: least c2p, -c2p, then p2c and -p2c of each 16-key block
  // Workgroup -> (b, h, query block qb), heads to XCDs as in the bias kernel.
  const int nqb = (L + 63) / 64, nky = nqb;
  int h, qb, b;
  {
    const int w = blockIdx.x;
    int r;
    if (H % 8 == 0) {
      const int hx = H / 8, l = w >> 3;
      h = (w & 7) * hx + l % hx;
      r = l / hx;
    } else {
      h = w % H;
      r = w / H;
    }
    qb = r % nqb;
    b = r / nqb;
  }
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lc = lane & 15, g = lane >> 4;
  const int qw = qb * 64 + 16 * wave;            // the wave's first query
  const int qg = qw + lc;                        // this lane's query in the score tile (keys 4 g .. 4 g + 3 of a block)
  const int qr = qg < L ? qg : L - 1;
  const half_t* pkh = pos_key + (int64_t)h * P * 64;
  const half_t* pqh = pos_query + (int64_t)h * P * 64;
  const int32_t* c2ph = c2p_idx + (int64_t)h * L * L;
  const int32_t* p2ch = p2c_idx + (int64_t)h * L * L;
  const half_t* mrow = key_mask + (int64_t)b * L;
  const int64_t bh = (int64_t)b * H + h;
  const half_t* kbase = k + bh * L * 64;
  const half_t* vbase = v + bh * L * 64;
  auto clampi = [&](int x) { return x < 0 ? 0 : (x >= P ? P - 1 : x); };
  auto key_of = [&](int kyb, int kb) { return 64 * kyb + 16 * kb + 4 * g; };  // this lane's first key of block kb
  const half8_t q0 = *reinterpret_cast<const half8_t*>(q + bh * L * 64 + (uint32_t)(qr * 64 + 8 * g));
  const half8_t q1 = *reinterpret_cast<const half8_t*>(q + bh * L * 64 + (uint32_t)(qr * 64 + 32 + 8 * g));

  // This lane's indices of a key block: c2p of keys key_of + j at query qr,
  // p2c of query qr at those keys (keys past L: the last ones).
  int ci[KB][4], pi[KB][4];
  auto load_indices = [&](int kyb) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int key = key_of(kyb, kb);
      if constexpr (VEC) {
        const int kc = key < L ? key : L - 4;
        const int4 x = *reinterpret_cast<const int4*>(c2ph + (uint32_t)(qr * L + kc));
        ci[kb][0] = x.x, ci[kb][1] = x.y, ci[kb][2] = x.z, ci[kb][3] = x.w;
#pragma unroll
        for (int j = 0; j < 4; ++j) pi[kb][j] = p2ch[(uint32_t)((kc + j) * L + qr)];
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int kc = key + j < L ? key + j : L - 1;
          ci[kb][j] = c2ph[(uint32_t)(qr * L + kc)];
          pi[kb][j] = p2ch[(uint32_t)(kc * L + qr)];
        }
      }
    }
  };
  half4_t mk[KB];
  auto load_mask = [&](int kyb) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int key = key_of(kyb, kb);
      if constexpr (VEC) {
        mk[kb] = *reinterpret_cast<const half4_t*>(mrow + (uint32_t)(key < L ? key : L - 4));
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) mk[kb][j] = mrow[(uint32_t)(key + j < L ? key + j : L - 1)];
      }
    }
  };
  // The clamped indices packed, c2p | p2c << 16, and the wave's index ranges
  // to LDS.
  auto put_ranges = [&](int buf, uint32_t (&cp)[KB][4]) {
    int c_mn = P, c_mx = 0, p_mn[KB], p_mx[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      p_mn[kb] = P, p_mx[kb] = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int c = clampi(ci[kb][j]), p = clampi(pi[kb][j]);
        c_mn = min(c_mn, c), c_mx = max(c_mx, c);
        p_mn[kb] = min(p_mn[kb], p), p_mx[kb] = max(p_mx[kb], p);
        cp[kb][j] = (uint32_t)c | ((uint32_t)p << 16);
      }
    }
    int r[2 + 2 * KB];
    r[0] = gen_wave_min(c_mn), r[1] = gen_wave_min(-c_mx);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) r[2 + 2 * kb] = gen_wave_min(p_mn[kb]), r[3 + 2 * kb] = gen_wave_min(-p_mx[kb]);
    if (lane == 0) {
#pragma unroll
      for (int i = 0; i < 2 + 2 * KB; ++i) ranges[buf][wave][i] = r[i];
    }
  };
  // The tile's ranges (after a barrier): first row and last row of each
  // window, the first c2p row of this wave and p2c row of each key block, and
  // whether one window of each table serves every wave with kBiasTiles tiles.
  struct Range {
    int c_lo, c_hi, p_lo, p_hi, c_wave, p_own, p_block[KB];
    bool single;
  };
  auto get_ranges = [&](int buf) -> Range {
    Range x;
    x.c_lo = P, x.c_hi = 0, x.p_lo = P, x.p_hi = 0, x.single = true;
    x.c_wave = __builtin_amdgcn_readfirstlane(ranges[buf][wave][0]);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int lo = __builtin_amdgcn_readfirstlane(ranges[buf][w][0]);
      const int hi = -__builtin_amdgcn_readfirstlane(ranges[buf][w][1]);
      x.c_lo = min(x.c_lo, lo), x.c_hi = max(x.c_hi, hi);
      x.single = x.single && hi - lo < kBiasCols;
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      int lo = P, hi = P;
#pragma unroll
      for (int w = 0; w < 4; ++w) lo = min(lo, ranges[buf][w][2 + 2 * kb]), hi = min(hi, ranges[buf][w][3 + 2 * kb]);
      lo = __builtin_amdgcn_readfirstlane(lo), hi = -__builtin_amdgcn_readfirstlane(hi);
      x.p_block[kb] = lo;
      x.p_lo = min(x.p_lo, lo), x.p_hi = max(x.p_hi, hi);
      x.single = x.single && hi - lo < kBiasCols;
    }
    x.single = x.single && x.c_hi - x.c_lo < kGenWin && x.p_hi - x.p_lo < kGenWin;
    // the tiles stay inside the window
    x.c_wave = min(x.c_wave, x.c_lo + kGenWin - kBiasCols);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) x.p_block[kb] = min(x.p_block[kb], x.p_lo + kGenWin - kBiasCols);
    x.p_own = x.p_block[0];
#pragma unroll
    for (int kb = 1; kb < KB; ++kb) x.p_own = wave == kb ? x.p_block[kb] : x.p_own;
    return x;
  };
  // DMA of `ROWS` rows, halfs c .. c + 7 of row r from src(r, c): lane l of a 1
  // KiB block brings physical chunk l % 8 of row l / 8.
  auto issue_rows = [&](auto rows_c, half_t* dst, auto&& src) {
    constexpr int BLOCKS = decltype(rows_c)::value / 32;  // 1 KiB blocks per wave
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j) {
      const int blk = wave * BLOCKS + j;
      const int row = 8 * blk + (lane >> 3);
      load_lds16(src(row, ((lane & 7) ^ ((row >> 1) & 7)) << 3), dst + blk * 512);
    }
  };
  // (one 32-bit offset from a uniform base wherever that can be: 64-bit
  // addresses of every block, kept over the key blocks, would spill)
  auto issue_window = [&](const half_t* table, half_t* dst, int base) {  // rows past P repeat row P - 1
    issue_rows(std::integral_constant<int, kGenWin>{}, dst,
               [&](int row, int c) { return table + (uint32_t)((base + row < P ? base + row : P - 1) * 64 + c); });
  };
  auto issue_block = [&](int kyb) {  // K rows (past L: the last one) and V rows (past L: zeros)
    issue_rows(std::integral_constant<int, 64>{}, krows, [&](int row, int c) {
      const int key = 64 * kyb + row;
      return kbase + (uint32_t)((key < L ? key : L - 1) * 64 + c);
    });
    issue_rows(std::integral_constant<int, 64>{}, vrows[kyb & 1], [&](int row, int c) {
      const int key = 64 * kyb + row;
      return key < L ? vbase + (uint32_t)(key * 64 + c) : g_zero_row + c;
    });
  };
  // kBiasTiles tiles of 16 window rows from row `r0` on against the 16 rows
  // whose fragments are f0, f1, into this wave's table rows.
  float* const own = tab + (16 * wave + lc) * kBiasStride;
  auto products = [&](const half_t* win, int r0, half8_t f0, half8_t f1) {
#pragma unroll
    for (int tp = 0; tp < kBiasTiles; ++tp) {
      const half8_t a0 = *reinterpret_cast<const half8_t*>(win + gen_swz(r0 + 16 * tp + lc, g));
      const half8_t a1 = *reinterpret_cast<const half8_t*>(win + gen_swz(r0 + 16 * tp + lc, 4 + g));
      float4_t r = {0.f, 0.f, 0.f, 0.f};
      r = mfma16x16x32(a0, f0, r);
      r = mfma16x16x32(a1, f1, r);  // lane: row lc, columns 16 tp + 4 g + i
      *reinterpret_cast<float4_t*>(own + 16 * tp + 4 * g) = r;
    }
  };
  auto c_of = [](uint32_t cp) { return (int)(cp & 0xFFFFu); };
  auto p_of = [](uint32_t cp) { return (int)(cp >> 16); };

  // Weights are exp(s - m) = 2^(s log2e - log_max(m)), with m log2e rounded
  // once per block (never part of an fma): the rounding scales a row's weights
  // alike, and the rounded value is what carries from block to block, so that
  // it cancels in the normalisation and the rescale is 1 where the max stays.
  constexpr float kLog2e = 1.4426950408889634f;
  auto log_max = [](float m) {
#pragma clang fp contract(off)
    return m * kLog2e;
  };
  // With EXACT, P . V takes weights times 2^15: the largest still fits fp16,
  // and fp16 parts of small ones keep 15 more bits above the subnormal floor.
  constexpr float kScaleP = EXACT ? 32768.f : 1.f;
  // running max (per query row, the same in the row's four lanes), its
  // log_max, this lane's part of the row sum, and O^T (lane: query lc, d 16 dt
  // + 4 g + i)
  float m_run = -65504.f, m_l2 = log_max(m_run), l_run = 0.f;
  float4_t o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = (float4_t){0.f, 0.f, 0.f, 0.f};

  uint32_t cp[KB][4], cpn[KB][4];  // this block's and the next one's indices
  load_indices(0);
  issue_block(0);
  load_mask(0);
  put_ranges(0, cp);
  stage_barrier();
  Range rg = get_ranges(0);
  if (rg.single) {
    issue_window(pkh, rk, rg.c_lo);
    issue_window(pqh, rq, rg.p_lo);
  }
  if (nky > 1) load_indices(1);
  for (int kyi = 0; kyi < nky; ++kyi) {  // uniform
    wait_vmcnt<0>();  // this block's windows, K and V rows
    stage_barrier();  // (and every wave is done with the last block's P2C rows)
    const bool more = kyi + 1 < nky;  // uniform
    if (more) {
      put_ranges((kyi + 1) & 1, cpn);
      if (kyi + 2 < nky) load_indices(kyi + 2);
    }
    float acc[KB][4];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      float4_t r = {0.f, 0.f, 0.f, 0.f};
      r = mfma16x16x32(*reinterpret_cast<const half8_t*>(krows + gen_swz(16 * kb + lc, g)), q0, r);
      r = mfma16x16x32(*reinterpret_cast<const half8_t*>(krows + gen_swz(16 * kb + lc, 4 + g)), q1, r);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[kb][j] = r[j];  // lane: query lc, keys 16 kb + 4 g + j
    }
    const half8_t kp0 = *reinterpret_cast<const half8_t*>(krows + gen_swz(16 * wave + lc, g));
    const half8_t kp1 = *reinterpret_cast<const half8_t*>(krows + gen_swz(16 * wave + lc, 4 + g));
    half4_t mkb[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) mkb[kb] = mk[kb];
    if (rg.single) {
      products(rk, rg.c_wave - rg.c_lo, q0, q1);
      wave_lds_sync();
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[kb][j] += own[c_of(cp[kb][j]) - rg.c_wave];
      wave_lds_sync();
      products(rq, rg.p_own - rg.p_lo, kp0, kp1);
    } else {
      // Tiles wider than one window or one wave's columns: windows of kGenWin
      // rows of each table in turn, through registers into the table's place
      // `tab`, the next one in flight meanwhile; a position outside them reads a
      // -0 column (x + -0 = x for every fp32 x).
      // (opaque: addresses hoisted out of the loop over the key blocks would
      // spill registers there)
      int tw = t;
      asm volatile("" : "+v"(tw));
      const int lw = tw & 15, gw = (tw >> 4) & 3, rw = tw >> 3, cw = tw & 7;
      float* const wtab = reinterpret_cast<float*>(krows);
      float* const wown = wtab + (16 * wave + lw) * kWideStride;
      half_t* const rows = reinterpret_cast<half_t*>(tab);
      half8_t x[kGenWin / 32];
      auto fetch = [&](const half_t* table, int base) {
#pragma unroll
        for (int i = 0; i < kGenWin / 32; ++i) {
          const int row = base + 32 * i + rw;
          x[i] = *reinterpret_cast<const half8_t*>(table + (uint32_t)((row < P ? row : P - 1) * 64 + 8 * cw));
        }
      };
      auto put = [&] {
#pragma unroll
        for (int i = 0; i < kGenWin / 32; ++i) *reinterpret_cast<half8_t*>(rows + gen_swz(32 * i + rw, cw)) = x[i];
      };
      auto wide_products = [&](half8_t f0, half8_t f1) {
#pragma unroll
        for (int tp = 0; tp < kGenWin / 16; ++tp) {
          const half8_t a0 = *reinterpret_cast<const half8_t*>(rows + gen_swz(16 * tp + lw, gw));
          const half8_t a1 = *reinterpret_cast<const half8_t*>(rows + gen_swz(16 * tp + lw, 4 + gw));
          float4_t r = {0.f, 0.f, 0.f, 0.f};
          r = mfma16x16x32(a0, f0, r);
          r = mfma16x16x32(a1, f1, r);
          *reinterpret_cast<float4_t*>(wown + 16 * tp + 4 * gw) = r;
          // (four tiles in flight: with all reads ahead of all products B = 32,
          // L = 256 takes 264 us)
          if (tp % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
      };
      fetch(pkh, rg.c_lo);
      stage_barrier();  // every wave holds its K fragments
      if (lane < 16) wown[kGenWin] = -0.0f;
      for (int w0 = rg.c_lo; w0 <= rg.c_hi; w0 += kGenWin) {  // uniform
        put();
        stage_barrier();
        if (w0 + kGenWin <= rg.c_hi) fetch(pkh, w0 + kGenWin);
        else fetch(pqh, rg.p_lo);
        wide_products(q0, q1);
        stage_barrier();  // every wave is done with the window
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[kb][j] += wown[min((uint32_t)(c_of(cp[kb][j]) - w0), (uint32_t)kGenWin)];
      }
      for (int w0 = rg.p_lo; w0 <= rg.p_hi; w0 += kGenWin) {  // uniform
        put();
        stage_barrier();  // (and every wave is past the last window's gather)
        if (w0 + kGenWin <= rg.p_hi) fetch(pqh, w0 + kGenWin);
        wide_products(kp0, kp1);
        stage_barrier();
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[kb][j] +=
                wtab[(16 * kb + 4 * gw + j) * kWideStride + min((uint32_t)(p_of(cp[kb][j]) - w0), (uint32_t)kGenWin)];
      }
      // (waited for here on every path: else the compiler waits for them, and
      // for whatever was issued since, in the next block's narrow path)
#pragma unroll
      for (int i = 0; i < kGenWin / 32; ++i) asm volatile("" : "+v"(x[i]));
    }
    stage_barrier();  // P2C rows visible; every wave is done with both windows and the K rows
    const Range now = rg;
    if (more) {
      rg = get_ranges((kyi + 1) & 1);
      if (rg.single) {
        issue_window(pkh, rk, rg.c_lo);
        issue_window(pqh, rq, rg.p_lo);
      }
      issue_block(kyi + 1);
      load_mask(kyi + 1);
    }
    if (now.single) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[kb][j] += tab[(16 * kb + 4 * g + j) * kBiasStride + (p_of(cp[kb][j]) - now.p_block[kb])];
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int j = 0; j < 4; ++j) cp[kb][j] = cpn[kb][j];

    // ---- online softmax over this key block, then P . V ----
    float bmax = m_run;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float sc = (float)mkb[kb][j] < -60000.f ? -65504.f : acc[kb][j] * scale;
        if (key_of(kyi, kb) + j >= L) sc = -__builtin_inff();
        acc[kb][j] = sc;
        bmax = fmaxf(bmax, sc);
      }
    bmax = rows_max(bmax);
    const float next_l2 = log_max(bmax);
    const float alpha = __builtin_amdgcn_exp2f(m_l2 - next_l2);
    m_run = bmax, m_l2 = next_l2;
    l_run *= alpha;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float e = __builtin_amdgcn_exp2f(fmaf(acc[kb][j], kLog2e, -m_l2));
        acc[kb][j] = e * kScaleP;
        l_run += e;
      }
    {
      // ds_read_b64_tr_b16: in each 16-lane group, source lane s names 4
      // consecutive halfs and lane j receives element j % 4 of source lanes
      // j / 4, 4 + j / 4, 8 + j / 4, 12 + j / 4.  Source lane lc of group g
      // names V[16 T + 4 g + lc / 4][16 dt + 4 (lc % 4) ..], so lane (g, lc)
      // receives V[16 T + 4 g + i][16 dt + lc], i = 0..3 (from 16 rows on,
      // tile T + 1): with V as the A operand and P^T as the B operand the
      // product lane holds O[query lc][16 dt + 4 g + i].  The swizzle term
      // (row >> 1) & 7 of those rows is (2 g + lc / 8) & 7.
      gen_lds_half_t* const rows3 = (gen_lds_half_t*)(lds_void_t*)vrows[kyi & 1];
      const int tr_sw = (2 * g + (lc >> 3)) & 7;
      const int tr_lane = (4 * g + (lc >> 2)) * 64 + 4 * (lc & 1);
      const int tr_c = (lc >> 1) & 1;
      auto v_tile = [&](int T, int dt) -> half4_t {  // V[16 T + 4 g + i][16 dt + lc]
        gen_lds_half_t* const a = rows3 + 16 * T * 64 + tr_lane + (((2 * dt + tr_c) ^ tr_sw) << 3);
        return __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((gen_lds_short4_t*)a));
      };
      // Two tiles' V fragments against parts of P (registers 4 u + i of a
      // fragment: key 16 (T + u) + 4 g + i).
      auto v_frag = [&](int T, int dt) -> half8_t {
        const half4_t h0 = v_tile(T, dt), h1 = v_tile(T + 1, dt);
        half8_t vb;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          vb[i] = h0[i];
          vb[4 + i] = h1[i];
        }
        return vb;
      };
      if constexpr (!EXACT) {
#pragma unroll
        for (int T = 0; T < KB; T += 2) {
          half8_t pa, pl;
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
              const float x0 = acc[T + u][i], x1 = acc[T + u][i + 1];
              const half2_t hi = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(x0, x1));
              pa[4 * u + i] = hi[0];
              pa[4 * u + i + 1] = hi[1];
              pl[4 * u + i] = (half_t)(x0 - (float)hi[0]);
              pl[4 * u + i + 1] = (half_t)(x1 - (float)hi[1]);
            }
#pragma unroll
          for (int dt = 0; dt < 4; ++dt) {
            const half8_t vb = v_frag(T, dt);
            o[dt] = mfma16x16x32(vb, pa, o[dt]);
            o[dt] = mfma16x16x32(vb, pl, o[dt]);
          }
        }
      } else {
        // All 24 bits of a weight x: hi + (mid + low) 2^-10 in fp16, exact for
        // weights from 2^-25 of the row's largest on, below that to 2^-49 of
        // it (512 of them on V = 65504: one subnormal step of the output).
        float4_t before[4], rest[4];
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) before[dt] = o[dt], rest[dt] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int T = 0; T < KB; T += 2) {
          half8_t pa, pm, pl;
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
              const float x0 = acc[T + u][i], x1 = acc[T + u][i + 1];
              const half2_t hi = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(x0, x1));
              const float r0 = (x0 - (float)hi[0]) * 1024.f, r1 = (x1 - (float)hi[1]) * 1024.f;
              const half2_t mid = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(r0, r1));
              const half2_t low = __builtin_bit_cast(
                  half2_t, __builtin_amdgcn_cvt_pkrtz(r0 - (float)mid[0], r1 - (float)mid[1]));
#pragma unroll
              for (int e = 0; e < 2; ++e)
                pa[4 * u + i + e] = hi[e], pm[4 * u + i + e] = mid[e], pl[4 * u + i + e] = low[e];
            }
#pragma unroll
          for (int dt = 0; dt < 4; ++dt) {
            const half8_t vb = v_frag(T, dt);
            rest[dt] = mfma16x16x32(vb, pl, rest[dt]);
            rest[dt] = mfma16x16x32(vb, pm, rest[dt]);
            o[dt] = mfma16x16x32(vb, pa, o[dt]);
          }
        }
        float sum = 0.f;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            o[dt][i] = fmaf(rest[dt][i], 1.f / 1024.f, o[dt][i]);
            sum += o[dt][i];
          }
        // An infinite V times a part that is 0 is NaN where the whole weight
        // gives an infinity: the block again, in fp32 products (v_mfma_f32_
        // 16x16x4_f32, k = g: key 16 T + 4 g + i).  They take 25% to 30% of the
        // kernel's time, so they are kept for this case.
        if (__builtin_amdgcn_ballot_w64(sum != sum) != 0) {  // uniform
#pragma unroll
          for (int dt = 0; dt < 4; ++dt) o[dt] = before[dt];
#pragma unroll
          for (int T = 0; T < KB; ++T)
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
              const half4_t vt = v_tile(T, dt);
#pragma unroll
              for (int i = 0; i < 4; ++i) o[dt] = mfma16x16x4f32((float)vt[i], acc[T][i], o[dt]);
            }
        }
      }
    }
  }
  if (qg < L) {
    const float inv = 1.0f / (kScaleP * rows_sum(l_run));
    half_t* orow = out + (((int64_t)b * L + qg) * H + h) * 64;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      half4_t ov;
#pragma unroll
      for (int i = 0; i < 4; ++i) ov[i] = (half_t)(o[dt][i] * inv);
      *reinterpret_cast<half4_t*>(orow + 16 * dt + 4 * g) = ov;
    }
  }
}

__global__ void relative_index_table_kernel(int32_t* __restrict__ out, int n, int bucket_size, int max_position) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 2 * n - 1) out[i] = relative_index(i - (n - 1), bucket_size, max_position);
}

// The matrix-core kernels read q, k, v and the table rows in 16-byte pieces
// and, where L allows, the c2p indices and the key mask four at a time, and
// store pieces of up to 16 bytes of the output; both entry points hold every
// operand to 16-byte alignment, as the header states.  A launch holds fewer
// than 2^32 threads: up to three queries in a workgroup of 256 threads reach
// that before the per-query kernels' 64 threads a query do, so `groups` of them
// (at most) that do not fit leave the call to those.
bool general_mfma_ok(int64_t D, int64_t L, int64_t P, int64_t groups, const int32_t* error_flag,
                     std::initializer_list<const void*> ptrs) {
  if (D != 64 || L > 512 || P > 65536 || groups >= (int64_t{1} << 32) / 256 || error_flag != nullptr) return false;
  for (const void* p : ptrs)
    if (reinterpret_cast<uintptr_t>(p) % 16 != 0) return false;
  return true;
}

}  // namespace

int launch_relative_bias_general(const void* q, const void* k, const void* pos_key, const void* pos_query,
                                 const int32_t* c2p, const int32_t* p2c, const void* key_mask, float scale, int64_t B,
                                 int64_t H, int64_t L, int64_t D, int64_t P, void* out, int32_t* error_flag,
                                 hipStream_t stream) {
  if (B * H * L == 0) return GD_OK;
  // Batch rows per workgroup: the fewest that leave one round of the two
  // workgroups a CU holds, all of them at most (B = 32, L = 256, 8,192 tiles: 1,
  // 2, 4, 8, 16 and 32 rows per workgroup take 133, 81, 55, 43, 36 and 45 us).
  // A round takes about 7 us for a workgroup's indices and table rows and 2 us
  // for each batch row; the form for one batch row takes about 3 us and 3 us
  // for each workgroup of a CU (256, 576 and 1,024 of them 6.0, 10.9 and 14.5
  // us), which is less where several rows would need a second round (B = 2, L =
  // 384, 1,152 tiles: 15.5 against 19.0 us).
  const int64_t blocks = (L + 63) / 64, tiles = H * blocks * blocks, slots = 2 * kGenCus;
  const int64_t want = std::min(B, (B * tiles + slots - 1) / slots);
  int64_t nb = (B + (B + want - 1) / want - 1) / ((B + want - 1) / want);  // in even groups
  const int64_t rounds = (tiles * ((B + nb - 1) / nb) + slots - 1) / slots;
  if (3.0 + 3.0 * (double)(B * tiles) / kGenCus < (double)rounds * (7.0 + 2.0 * (double)nb)) nb = 1;
  const int64_t groups = tiles * ((B + nb - 1) / nb);
  if (general_mfma_ok(D, L, P, groups, error_flag, {q, k, pos_key, pos_query, c2p, p2c, key_mask, out})) {
    const dim3 grid((unsigned)groups);
    auto pick = [&](auto multi) {
      constexpr bool M = decltype(multi)::value;
      return L % 8 == 0   ? relative_bias_mfma_kernel<8, M>
             : L % 4 == 0 ? relative_bias_mfma_kernel<4, M>
             : L % 2 == 0 ? relative_bias_mfma_kernel<2, M>
                          : relative_bias_mfma_kernel<1, M>;
    };
    const auto kernel = nb > 1 ? pick(std::true_type{}) : pick(std::false_type{});
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, static_cast<const half_t*>(q),
                       static_cast<const half_t*>(k), static_cast<const half_t*>(pos_key),
                       static_cast<const half_t*>(pos_query), c2p, p2c, static_cast<const half_t*>(key_mask), scale,
                       (int)B, (int)H, (int)L, (int)P, (int)nb, static_cast<half_t*>(out));
    GD_LAUNCH_CHECK();
    return GD_OK;
  }
  hipLaunchKernelGGL(relative_bias_general_kernel, dim3((unsigned)(B * H * L)), dim3(64), (size_t)D * sizeof(float),
                     stream, static_cast<const half_t*>(q), static_cast<const half_t*>(k),
                     static_cast<const half_t*>(pos_key), static_cast<const half_t*>(pos_query), c2p, p2c,
                     static_cast<const half_t*>(key_mask), scale, (int)H, (int)L, (int)D, (int)P,
                     static_cast<half_t*>(out), error_flag);
  GD_LAUNCH_CHECK();
  return GD_OK;
}

int launch_fused_attention_general(const void* q, const void* k, const void* v, const void* pos_key,
                                   const void* pos_query, const int32_t* c2p, const int32_t* p2c, const void* key_mask,
                                   float scale, int64_t B, int64_t H, int64_t L, int64_t D, int64_t P, void* out,
                                   int32_t* error_flag, hipStream_t stream) {
  if (B * H * L == 0) return GD_OK;
  const int64_t groups = B * H * ((L + 63) / 64);
  if (general_mfma_ok(D, L, P, groups, error_flag, {q, k, v, pos_key, pos_query, c2p, p2c, key_mask, out})) {
    const dim3 grid((unsigned)groups);
    // Lengths that are a multiple of 16 take the weights in two parts (4% to 9%
    // faster), as they always have; the others kept fp32 weights on the
    // per-query kernels, so they keep all bits here.
    const auto kernel = L % 16 == 0  ? fused_attention_mfma_kernel<true, false>
                        : L % 4 == 0 ? fused_attention_mfma_kernel<true, true>
                                     : fused_attention_mfma_kernel<false, true>;
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, static_cast<const half_t*>(q),
                       static_cast<const half_t*>(k), static_cast<const half_t*>(v),
                       static_cast<const half_t*>(pos_key), static_cast<const half_t*>(pos_query), c2p, p2c,
                       static_cast<const half_t*>(key_mask), scale, (int)H, (int)L, (int)P,
                       static_cast<half_t*>(out));
    GD_LAUNCH_CHECK();
    return GD_OK;
  }
  hipLaunchKernelGGL(fused_attention_general_kernel, dim3((unsigned)(B * H * L)), dim3(64),
                     (size_t)(D + L) * sizeof(float), stream, static_cast<const half_t*>(q),
                     static_cast<const half_t*>(k), static_cast<const half_t*>(v), static_cast<const half_t*>(pos_key),
                     static_cast<const half_t*>(pos_query), c2p, p2c, static_cast<const half_t*>(key_mask), scale,
                     (int)H, (int)L, (int)D, (int)P, static_cast<half_t*>(out), error_flag);
  GD_LAUNCH_CHECK();
  return GD_OK;
}

int launch_relative_index_table(int32_t* out, int n, int bucket_size, int max_position, hipStream_t stream) {
  const int count = 2 * n - 1;
  hipLaunchKernelGGL(relative_index_table_kernel, dim3((count + 255) / 256), dim3(256), 0, stream, out, n, bucket_size,
                     max_position);
  GD_LAUNCH_CHECK();
  return GD_OK;
}

}  // namespace gd
