// out [M, N] = fp16_rn(a [M, K] @ b [K, N]), fp16 row-major operands, a short and wide output
// (a few hundred rows) contracted over a very long K: the head's hidden gradient, dlogits
// [labelled rows, vocabulary] @ W [vocabulary, hidden] (solution/head.py:113, cuBLAS there).
//
// Measured on MI355X at [n, 151936] @ [151936, 1536], both launches, against hipBLASLt's heuristic:
// 18 rows 92 us (5.1 TB/s) / 326, 130 rows 106 / 466, 420 rows 249 (788 TFLOP/s) / 580, 930 rows 483
// / 842, 1536 rows 686 (1045 TFLOP/s) / 935, 2048 rows 935 / 1060; a large square hipBLASLt product
// reaches 1280 TFLOP/s on the same card and a large copy 6.6 TB/s.  What bounds it: at few rows
// the read of W (467 MB at Qwen2.5-1.5B's vocabulary), at some
// hundred rows the matrix cores.  The output has few tiles (24 rows: one row of tiles), so a GEMM
// that walks all of K per tile leaves most of the 256 CUs idle.  Here K is cut into as many parts
// as fill the chip once (split_plan), each workgroup writes the fp32 partial of its part, and a
// second launch adds the parts in a fixed order and rounds once.
//
// A workgroup is 8 wavefronts over a BM x 256 tile, BM = 16 * MT * WM rows: WM wavefronts down,
// 8 / WM across (WM = 1 up to 64 rows, else 2), 64 of K per step.  The steps' tiles are read
// through registers (buffer loads: rows past M, columns past N and K read zero) into one of two
// LDS buffers, PF steps ahead, one barrier per step.  The product is formed transposed, out^T =
// b^T a^T, on v_mfma_f32_16x16x32_f16: b's fragments (lane: column l%16 of b, 8 consecutive k) come
// from the row-major LDS tile by transpose reads, a's with 16-byte reads, and a lane ends with
// four consecutive columns of one row (one 16-byte store).  Both tiles are XOR-swizzled in
// 16-byte chunks so that every LDS read is free of bank conflicts (256 B per clock).

#include <algorithm>
#include <type_traits>

#include "soupk_common.hpp"

namespace soupk {
namespace {

typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s4 lds_s4;
typedef __attribute__((address_space(3))) unsigned char lds_b;

constexpr int kNnThreads = 512;
constexpr int kNnBN = 256;
constexpr int kNnBK = 64;
constexpr uint32_t kOob = 0x80000000u;   // a byte offset past every operand (< 2^31 bytes)
constexpr int kNnMaxSplits = 128;

__device__ __forceinline__ u32x4 buf_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                       r, static_cast<int>(off), 0, 0));
}

// Workgroup ids go round-robin over the 8 XCDs; consecutive logical ids (the tiles of one K part,
// which read the same rows of b or the same columns of a) are given to one XCD's L2.
__device__ __forceinline__ int xcd_local(int id, int total8) {
  return (id & 7) * (total8 >> 3) + (id >> 3);
}

struct NnPlan {
  int tiles_m, tiles_n, splits, per;
};

// Most rows the 16- to 64-row tiles take; their two workgroups per CU.
constexpr int kSmallRows = 64;

// The row tile and the K parts.  The parts fill the CUs once (twice up to 64 rows, where two
// workgroups fit a CU's LDS); a kernel plans them itself, from the rows that count.  Up to 192 rows one row of tiles, of the fewest rows that cover M;
// above, the tile of 160, 192 or 256 rows with the least work per workgroup (rows x steps: the
// three run at the same rate, 0.91 - 0.94 PFLOP/s where they are full; with 256-row tiles alone 640
// rows took 369 us against 336, 1300 rows 681 against 598).  Two steps of prefetch instead of one
// took the 160- and 192-row tiles from 147 and 152 us to 113 and 124 at one row of tiles; the
// 256-row tile has no registers for the second.  The tile is the host's choice from the most rows;
// the parts follow from the rows that count (420 of 700: 279 us on the tile for 700, 257 on the
// tile for 420).
__host__ __device__ inline NnPlan nn_plan(int bm, int M, int N, int K, int cus) {
  NnPlan p;
  p.tiles_m = (M + bm - 1) / bm;
  p.tiles_n = (N + kNnBN - 1) / kNnBN;
  const int kt = (K + kNnBK - 1) / kNnBK;
  int s = cus * (bm <= kSmallRows ? 2 : 1) / (p.tiles_m * p.tiles_n);
  s = s < 1 ? 1 : (s > kNnMaxSplits ? kNnMaxSplits : s);
  s = s > kt ? kt : s;
  p.per = (kt + s - 1) / s;
  p.splits = (kt + p.per - 1) / p.per;
  return p;
}

// The row tile for up to M rows.
int nn_tile_rows(int M, int N, int K, int cus) {
  if (M <= kSmallRows) return (M + 15) / 16 * 16;
  if (M <= 192) return M <= 96 ? 96 : (M + 31) / 32 * 32;
  int best = 256;
  int64_t best_work = -1;
  for (int bm : {256, 192, 160}) {
    const NnPlan p = nn_plan(bm, M, N, K, cus);
    const int wgs = p.tiles_m * p.tiles_n * p.splits;
    const int64_t work = static_cast<int64_t>((wgs + cus - 1) / cus) * p.per * bm;
    if (best_work < 0 || work < best_work) {
      best = bm;
      best_work = work;
    }
  }
  return best;
}

struct NnArgs {
  const uint16_t* a;
  const uint16_t* b;
  float* part;
  uint16_t* out;
  int64_t ldo;
  uint32_t lda, ldb;
  int M, N, K, cus;
  const int32_t* rows;   // nullable: the rows of a that count (at most M), in device memory
};

__device__ __forceinline__ int nn_rows(const NnArgs& g) {
  // (wave-uniform, and told so: the plan made of it stays in scalar registers)
  return g.rows != nullptr ? __builtin_amdgcn_readfirstlane(max(0, min(*g.rows, g.M))) : g.M;
}

template <int MT, int WM, int PF>
__global__ __launch_bounds__(kNnThreads, 16 * MT * WM <= kSmallRows ? 4 : 2) void gemm_nn_kernel(
    NnArgs g) {
  constexpr int BM = 16 * MT * WM, WN = 8 / WM, NT = kNnBN / WN / 16;
  constexpr int AI = (BM + 63) / 64;          // 64-row groups of a's tile
  constexpr int kABytes = BM * kNnBK * 2, kStage = kABytes + kNnBK * kNnBN * 2;
  __shared__ __align__(16) unsigned char smem[2 * kStage];
  // The plan is made from the row count in device memory (or M), so that a caller need not know the
  // count; workgroups past the plan's exit.
  const int M = nn_rows(g);
  if (M == 0) return;
  NnPlan p = nn_plan(BM, M, g.N, g.K, g.cus);
  p.tiles_m = __builtin_amdgcn_readfirstlane(p.tiles_m);
  p.tiles_n = __builtin_amdgcn_readfirstlane(p.tiles_n);
  p.splits = __builtin_amdgcn_readfirstlane(p.splits);
  p.per = __builtin_amdgcn_readfirstlane(p.per);
  const int total = p.tiles_m * p.tiles_n * p.splits;
  const int total8 = (total + 7) & ~7;
  if (static_cast<int>(blockIdx.x) >= total8) return;
  const int logical = xcd_local(blockIdx.x, total8);
  if (logical >= total) return;
  const uint16_t* const a = g.a;
  const uint16_t* const b = g.b;
  const uint32_t lda = g.lda, ldb = g.ldb;
  const int N = g.N, K = g.K, splits = p.splits;
  const int tiles = p.tiles_m * p.tiles_n;
  const int split = __builtin_amdgcn_readfirstlane(logical / tiles);
  const int tile = logical - split * tiles;
  const int tn = __builtin_amdgcn_readfirstlane(tile / p.tiles_m), tm = tile - tn * p.tiles_m;
  const int m0 = tm * BM, n0 = tn * kNnBN;
  const int kt = (K + kNnBK - 1) / kNnBK;
  const int t0 = split * p.per, steps = min(p.per, kt - t0);

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w / WN, wn = w % WN;
  const int ql = lane & 15, gr = lane >> 4;

  // Global and LDS places of this thread's 16-byte chunks (the swizzles are constant per thread).
  const __amdgpu_buffer_rsrc_t ra =
      buffer_rsrc(a, (static_cast<uint32_t>(M - 1) * lda + static_cast<uint32_t>(K)) * 2u);
  const __amdgpu_buffer_rsrc_t rb = buffer_rsrc(
      b, (static_cast<uint32_t>(K - 1) * ldb + static_cast<uint32_t>(N)) * 2u);
  const int ar = tid >> 3, ac = tid & 7, br = tid >> 5, bc = tid & 31;
  // (rows past M and columns past N read the last row's or column's values: never stored)
  uint32_t aoff[AI];
#pragma unroll
  for (int i = 0; i < AI; ++i)
    aoff[i] = (static_cast<uint32_t>(min(m0 + 64 * i + ar, M - 1)) * lda + 8u * ac +
               static_cast<uint32_t>(t0) * kNnBK) * 2u;
  const uint32_t boff = (static_cast<uint32_t>(t0 * kNnBK + br) * ldb +
                         static_cast<uint32_t>(min(n0 + 8 * bc, N - 8))) * 2u;
  const uint32_t a_st = ar * 128 + ((ac ^ (ar & 7)) << 4);
  const uint32_t b_st = br * 512 + ((bc ^ (2 * ((br & 3) | (((br >> 3) & 1) << 2)))) << 4);

  struct Regs {
    u32x4 av[AI], bv[4];
  } regs[PF];
  auto load = [&](Regs& r, int t) {
    // Past this part's last step, and past K in a's columns, the offset is out of range and the
    // load returns zeros; b's rows past K lie past its end.
    const bool live = t < steps;
    const uint32_t at = static_cast<uint32_t>(t) * (kNnBK * 2u);
    const bool a_in = live && (t0 + t) * kNnBK + 8 * ac < K;
    const uint32_t bt = static_cast<uint32_t>(t) * (kNnBK * 2u) * ldb;
#pragma unroll
    for (int i = 0; i < AI; ++i) r.av[i] = buf_load(ra, a_in ? aoff[i] + at : kOob);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      r.bv[i] = buf_load(rb, live ? boff + bt + static_cast<uint32_t>(i) * 32u * ldb : kOob);
  };
  auto store = [&](const Regs& r, int buf) {
    unsigned char* sa = smem + buf * kStage;
    unsigned char* sb = sa + kABytes;
#pragma unroll
    for (int i = 0; i < AI; ++i)
      if (BM % 64 == 0 || 64 * i + ar < BM)
        *reinterpret_cast<u32x4*>(sa + a_st + i * 64 * 128) = r.av[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(sb + b_st + i * 16 * 512) = r.bv[i];
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // LDS read places.  a: row 16i + ql of the wavefront's rows, chunk 4ks + gr.  b (transpose
  // read): lane kk = l%16 of a group reads row 8gr + kk/4 (+ 4 for the second), columns 4(kk%4)..+3
  // of its 16-column tile, so that lane i of the group gets column i of those four rows.
  const uint32_t a_row = (wm * 16 * MT + ql) * 128;
  const int kk = ql;
  const int brow = 8 * gr + (kk >> 2);
  const uint32_t b_sw = 2 * ((brow & 3) | (((brow >> 3) & 1) << 2));
  auto compute = [&](int buf) {
    const unsigned char* sa = smem + buf * kStage;
    const lds_b* sb = (const lds_b*)(sa + kABytes);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      // (the tallest tiles' registers hold one half step's fragments: no reads ahead of it)
      if constexpr (MT == 8) __asm__ volatile("" ::: "memory");
      h8 bf[NT], af[MT];
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const uint32_t c = (wn * NT + j) * 2 + ((kk & 3) >> 1);
        const uint32_t at = (32 * ks + brow) * 512 + ((c ^ b_sw) << 4) + (kk & 1) * 8;
        const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(sb + at));
        const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(sb + at + 4 * 512));
        bf[j] = __builtin_shufflevector(__builtin_bit_cast(h4, lo), __builtin_bit_cast(h4, hi), 0, 1,
                                        2, 3, 4, 5, 6, 7);
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
        af[i] = *reinterpret_cast<const h8*>(sa + a_row + i * 16 * 128 +
                                             (((4 * ks + gr) ^ (ql & 7)) << 4));
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[j], af[i], acc[i][j], 0, 0, 0);
    }
  };

#pragma unroll
  for (int p = 0; p < PF; ++p) load(regs[p], p);
  store(regs[0], 0);
  __syncthreads();
  auto step = [&](int t, auto parity) {
    constexpr int P = decltype(parity)::value;
    load(regs[P % PF], t + PF);
    compute(P);
    store(regs[(P + 1) % PF], P ^ 1);
    __syncthreads();
  };
  // (an odd last step is followed by one on zeros: a tail of its own made the compiler copy the
  // accumulators every iteration)
  for (int t = 0; t < steps; t += 2) {
    step(t, std::integral_constant<int, 0>{});
    step(t + 1, std::integral_constant<int, 1>{});
  }

  // C: column (lane) = row of out, rows = columns 16j + 4gr .. +3 of the tile
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + (wm * MT + i) * 16 + ql;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = n0 + (wn * NT + j) * 16 + 4 * gr;
      if (n >= N) continue;
      const f32x4 v = acc[i][j];
      if (splits > 1)
        *reinterpret_cast<f32x4*>(g.part + (static_cast<int64_t>(split) * M + m) * N + n) = v;
      else
        *reinterpret_cast<u32x2*>(g.out + m * g.ldo + n) =
            u32x2{pack_h2(v[0], v[1]), pack_h2(v[2], v[3])};
    }
  }
}

// out = fp16_rn of the sum of the parts: a workgroup takes 64 float4 columns-of-row, wavefront w
// adds a quarter of the parts in order, the quarters are added in order.
__global__ __launch_bounds__(256) void gemm_nn_sum_kernel(NnArgs g, int bm) {
  __shared__ f32x4 sums[3][64];
  const int M = nn_rows(g);
  const int n_cols4 = g.N / 4;
  const int64_t n4 = static_cast<int64_t>(M) * n_cols4;
  if (static_cast<int64_t>(blockIdx.x) * 64 >= n4) return;
  const int splits = nn_plan(bm, M, g.N, g.K, g.cus).splits;
  if (splits == 1) return;
  const f32x4* const parts = reinterpret_cast<const f32x4*>(g.part);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 64 + lane;
  const int64_t ic = min(i, n4 - 1);
  const int q = (splits + 3) / 4;
  const int s0 = min(w * q, splits), s1 = min(s0 + q, splits);
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  for (int p = s0; p < s1; p += 8) {
    f32x4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = parts[min(p + u, s1 - 1) * n4 + ic];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (p + u < s1) s = s + v[u];
  }
  if (w > 0) sums[w - 1][lane] = s;
  __syncthreads();
  if (w > 0 || i >= n4) return;
  s = ((s + sums[0][lane]) + sums[1][lane]) + sums[2][lane];
  const int64_t m = i / n_cols4;
  const int64_t n = (i - m * n_cols4) * 4;
  *reinterpret_cast<u32x2*>(g.out + m * g.ldo + n) =
      u32x2{pack_h2(s[0], s[1]), pack_h2(s[2], s[3])};
}

// Workgroups that any row count up to M can need: the CUs filled once (twice), or one part of
// the most tiles.
int64_t nn_grid(int bm, int64_t M, int32_t N, int cus) {
  const int64_t tiles = (M + bm - 1) / bm * ((N + kNnBN - 1) / kNnBN);
  return std::max<int64_t>(bm <= kSmallRows ? 2 * cus : cus, tiles);
}

// Floats of the partials for any row count up to M: with more than one part, tiles x parts fill
// the CUs at most once (twice), so the parts' rows x columns are at most that many whole tiles.
int64_t nn_workspace(int64_t M, int32_t N, int32_t K, int cus) {
  const bool small = M <= kSmallRows;
  const int64_t kt = (K + kNnBK - 1) / kNnBK;
  const int64_t tiles = static_cast<int64_t>(small ? 2 * cus * kSmallRows : cus * 256) * kNnBN;
  return std::min(tiles, std::min<int64_t>(kNnMaxSplits, kt) * M * N);
}

int check_nn(const void* a, int64_t lda, const void* b, int64_t ldb, const void* out, int64_t ldo,
             int64_t M, int32_t N, int32_t K) {
  if (M < 0 || N <= 0 || K <= 0 || N % 8 || K % 8 || lda < K || ldb < N || ldo < N || lda % 8 ||
      ldb % 8 || ldo % 4)
    return kInvalid;
  if (M == 0) return kOk;
  if (M > (1 << 20) || M * lda >= (int64_t{1} << 30) || K * ldb >= (int64_t{1} << 30))
    return kInvalid;
  if (!a || !b || !out || (reinterpret_cast<uintptr_t>(a) & 15) ||
      (reinterpret_cast<uintptr_t>(b) & 15) || (reinterpret_cast<uintptr_t>(out) & 7))
    return kInvalid;
  return kOk;
}

}  // namespace
}  // namespace soupk

using namespace soupk;

extern "C" __attribute__((visibility("default"))) int soupk_gemm_nn_workspace(
    int64_t M, int32_t N, int32_t K, int64_t* floats) {
  if (M < 0 || N <= 0 || K <= 0 || !floats || M > (1 << 20)) return kInvalid;
  *floats = nn_workspace(M, N, K, device_cu_count());
  return kOk;
}

extern "C" __attribute__((visibility("default"))) int soupk_gemm_nn(
    const uint16_t* a, int64_t lda, const uint16_t* b, int64_t ldb, uint16_t* out, int64_t ldo,
    int64_t M, int32_t N, int32_t K, const int32_t* rows, float* workspace,
    int64_t workspace_floats, void* stream) {
  const int rc0 = check_nn(a, lda, b, ldb, out, ldo, M, N, K);
  if (rc0 != kOk) return rc0;
  if (M == 0) return kOk;
  const int cus = device_cu_count();
  if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 15) ||
      workspace_floats < nn_workspace(M, N, K, cus))
    return kInvalid;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int bm = nn_tile_rows(static_cast<int>(M), N, K, cus);
  const int64_t wgs = (nn_grid(bm, M, N, cus) + 7) / 8 * 8;
  const int64_t sums = (M * N / 4 + 63) / 64;
  if (wgs > 0x7fffffff || sums > 0x7fffffff) return kInvalid;
  const NnArgs g{a, b, workspace, out, ldo, static_cast<uint32_t>(lda), static_cast<uint32_t>(ldb),
                 static_cast<int>(M), N, K, cus, rows};
  auto run = [&](auto kernel) {
    return launch_kernel(kernel, dim3(static_cast<unsigned>(wgs)), dim3(kNnThreads), st, g);
  };
  int rc;
  switch (bm) {
    case 16: rc = run(gemm_nn_kernel<1, 1, 2>); break;
    case 32: rc = run(gemm_nn_kernel<2, 1, 2>); break;
    case 48: rc = run(gemm_nn_kernel<3, 1, 2>); break;
    case 64: rc = run(gemm_nn_kernel<4, 1, 1>); break;
    case 96: rc = run(gemm_nn_kernel<3, 2, 2>); break;
    case 128: rc = run(gemm_nn_kernel<4, 2, 2>); break;
    case 160: rc = run(gemm_nn_kernel<5, 2, 2>); break;
    case 192: rc = run(gemm_nn_kernel<6, 2, 2>); break;
    default: rc = run(gemm_nn_kernel<8, 2, 1>); break;
  }
  // (one part whatever the row count: the tiles alone fill the CUs, or K is one step)
  if (rc != kOk ||
      (rows == nullptr && nn_plan(bm, static_cast<int>(M), N, K, cus).splits == 1))
    return rc;
  return launch_kernel(gemm_nn_sum_kernel, dim3(static_cast<unsigned>(sums)), dim3(256), st, g, bm);
}
