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

template <int MT, int WM, int PF>
__global__ __launch_bounds__(kNnThreads, MT * WM <= 4 ? 4 : 2) void gemm_nn_kernel(
    const uint16_t* a, uint32_t lda, const uint16_t* b, uint32_t ldb, float* __restrict__ part,
    uint16_t* __restrict__ out, int64_t ldo, int M, int N, int K, int tiles_m, int tiles_n,
    int splits, int per) {
  constexpr int BM = 16 * MT * WM, WN = 8 / WM, NT = kNnBN / WN / 16;
  constexpr int AI = (BM + 63) / 64;          // 64-row groups of a's tile
  constexpr int kABytes = BM * kNnBK * 2, kBBytes = kNnBK * kNnBN * 2;
  __shared__ __align__(16) unsigned char smem[2][kABytes + kBBytes];
  const int logical = xcd_local(blockIdx.x, gridDim.x);
  const int tiles = tiles_m * tiles_n;
  const int split = logical / tiles;
  if (split >= splits) return;
  const int tile = logical - split * tiles;
  const int tm = tile % tiles_m, tn = tile / tiles_m;
  const int m0 = tm * BM, n0 = tn * kNnBN;
  const int kt = (K + kNnBK - 1) / kNnBK;
  const int t0 = split * per, steps = min(per, kt - t0);

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
    unsigned char* sa = smem[buf];
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
    const unsigned char* sa = smem[buf];
    const lds_b* sb = (const lds_b*)(smem[buf] + kABytes);
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
  int t = 0;
  for (; t + 2 <= steps; t += 2) {
    step(t, std::integral_constant<int, 0>{});
    step(t + 1, std::integral_constant<int, 1>{});
  }
  if (t < steps) compute(0);

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
        *reinterpret_cast<f32x4*>(part + (static_cast<int64_t>(split) * M + m) * N + n) = v;
      else
        *reinterpret_cast<u32x2*>(out + m * ldo + n) =
            u32x2{pack_h2(v[0], v[1]), pack_h2(v[2], v[3])};
    }
  }
}

// out = fp16_rn of the sum of the splits' partials: a workgroup takes 64 float4 columns-of-row,
// wavefront w adds a quarter of the splits in order, the quarters are added in order.
__global__ __launch_bounds__(256) void gemm_nn_sum_kernel(const f32x4* __restrict__ parts,
                                                          int splits, int64_t n4, int n_cols4,
                                                          uint16_t* __restrict__ out, int64_t ldo) {
  __shared__ f32x4 sums[3][64];
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
  *reinterpret_cast<u32x2*>(out + m * ldo + n) = u32x2{pack_h2(s[0], s[1]), pack_h2(s[2], s[3])};
}

struct NnPlan {
  int bm, tiles_m, tiles_n, splits, per;
};

// The row tile and the K parts.  The parts fill the CUs once (twice up to 64 rows, where two
// workgroups fit a CU's LDS).  Up to 192 rows one row of tiles, of the fewest rows that cover M;
// above, the tile of 160, 192 or 256 rows with the least work per workgroup (rows x steps: the
// three run at the same rate, 0.91 - 0.94 PFLOP/s where they are full; with 256-row tiles alone 640
// rows took 369 us against 336, 1300 rows 681 against 598).  Two steps of prefetch instead of one
// took the 160- and 192-row tiles from 147 and 152 us to 113 and 124 at one row of tiles; the
// 256-row tile has no registers for the second.
NnPlan nn_plan(int64_t M, int32_t N, int32_t K) {
  const int tiles_n = (N + kNnBN - 1) / kNnBN;
  const int kt = (K + kNnBK - 1) / kNnBK;
  const int cus = device_cu_count();
  auto plan = [&](int bm) {
    NnPlan p;
    p.bm = bm;
    p.tiles_m = static_cast<int>((M + bm - 1) / bm);
    p.tiles_n = tiles_n;
    const int64_t tiles = static_cast<int64_t>(p.tiles_m) * tiles_n;
    const int64_t fill = std::max<int64_t>(1, cus * (bm <= 64 ? 2 : 1) / tiles);
    const int s = static_cast<int>(std::min<int64_t>(fill, std::min(kNnMaxSplits, kt)));
    p.per = (kt + s - 1) / s;
    p.splits = (kt + p.per - 1) / p.per;
    return p;
  };
  const int rows = static_cast<int>(std::min<int64_t>(M, 1 << 20));
  if (rows <= 64) return plan((rows + 15) / 16 * 16);
  if (rows <= 192) return plan((rows + 31) / 32 * 32);
  NnPlan best = plan(256);
  int64_t best_work = -1;
  for (int bm : {256, 192, 160}) {
    const NnPlan p = plan(bm);
    const int64_t wgs = static_cast<int64_t>(p.tiles_m) * tiles_n * p.splits;
    const int64_t work = (wgs + cus - 1) / cus * p.per * bm;
    if (best_work < 0 || work < best_work) {
      best = p;
      best_work = work;
    }
  }
  return best;
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
  *floats = 0;
  if (M == 0) return kOk;
  const NnPlan p = nn_plan(M, N, K);
  if (p.splits > 1) *floats = static_cast<int64_t>(p.splits) * M * N;
  return kOk;
}

extern "C" __attribute__((visibility("default"))) int soupk_gemm_nn(
    const uint16_t* a, int64_t lda, const uint16_t* b, int64_t ldb, uint16_t* out, int64_t ldo,
    int64_t M, int32_t N, int32_t K, float* workspace, int64_t workspace_floats, void* stream) {
  const int rc0 = check_nn(a, lda, b, ldb, out, ldo, M, N, K);
  if (rc0 != kOk) return rc0;
  if (M == 0) return kOk;
  const NnPlan p = nn_plan(M, N, K);
  const int64_t need = p.splits > 1 ? static_cast<int64_t>(p.splits) * M * N : 0;
  if (need > 0 && (!workspace || workspace_floats < need ||
                   (reinterpret_cast<uintptr_t>(workspace) & 15)))
    return kInvalid;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int total = p.tiles_m * p.tiles_n * p.splits;
  const dim3 grid(static_cast<unsigned>((total + 7) / 8 * 8)), block(kNnThreads);
  auto run = [&](auto kernel) {
    return launch_kernel(kernel, grid, block, st, a, static_cast<uint32_t>(lda), b,
                         static_cast<uint32_t>(ldb), workspace, out, ldo, static_cast<int>(M), N, K,
                         p.tiles_m, p.tiles_n, p.splits, p.per);
  };
  int rc;
  switch (p.bm) {
    case 16: rc = run(gemm_nn_kernel<1, 1, 2>); break;
    case 32: rc = run(gemm_nn_kernel<2, 1, 2>); break;
    case 48: rc = run(gemm_nn_kernel<3, 1, 2>); break;
    case 64: rc = run(gemm_nn_kernel<4, 1, 1>); break;
    case 96: rc = run(gemm_nn_kernel<3, 2, 2>); break;
    case 128: rc = run(gemm_nn_kernel<4, 2, 2>); break;
    case 160: rc = run(gemm_nn_kernel<5, 2, 2>); break;
    case 192: rc = run(gemm_nn_kernel<6, 2, 2>); break;
    case 256: rc = run(gemm_nn_kernel<8, 2, 1>); break;
    default: return kInvalid;
  }
  if (rc != kOk || p.splits == 1) return rc;
  const int64_t n4 = M * N / 4;
  return launch_kernel(gemm_nn_sum_kernel, dim3(static_cast<unsigned>((n4 + 63) / 64)), dim3(256),
                       st, reinterpret_cast<const f32x4*>(workspace), p.splits, n4, N / 4, out, ldo);
}
