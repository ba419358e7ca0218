// matmul.hip -- general f32 GEMMs on MFMA and the host-slice GEMM workspace.
//
// Replaces the cuBLAS fallback of the reference's prichs-core
// (crates/prichs-cuda/src/cublas.rs): GpuWorkspace (46-166), its matmul_at_b
// (170-219) and matmul_a_bt (221-268), and the process-wide workspace with
// matmul_gpu / matmul_at_b_gpu / matmul_a_bt_gpu (283-327) that
// crates/prichs-core/src/ops.rs:3, 24-31 dispatches every large matmul_2d
// to.  Shapes are arbitrary (no multiple-of-tile requirement).
//
// Arithmetic: v_mfma_f32_16x16x4f32 -- full f32 products with f32
// accumulation (the reference's cuBLAS runs TF32 tensor cores,
// engine.rs:370 / cublas.rs:72; this path is at least as precise and stays
// within 1e-4 of the reference's CPU loop, crates/prichs-core/src/ops.rs:
// 33-58, on its shapes).
#include <algorithm>
#include <cmath>
#include <mutex>
#include <new>
#include <type_traits>

#include "common.hpp"
#include "f32_tile.hpp"

struct prichs_gpu_workspace {
  std::mutex mu;  // serialises the calls on this handle (the reference's Mutex<GpuWorkspace>)
  int device = 0;
  void *base = nullptr;
  float *a = nullptr, *b = nullptr, *c = nullptr;  // slabs A, B, C
  size_t cap_a = 0, cap_b = 0, cap_c = 0;          // bytes
};

namespace prichs {
namespace {

using f32t::f32x4;

// C[M, N] = sum_r opA(i, r) opB(r, j), row-major C with ldc = N.
//   OP 0 (A B):    opA(i, r) = A[i R + r],  opB(r, j) = B[r N + j]
//   OP 1 (A^T B):  opA(i, r) = A[r M + i],  opB(r, j) = B[r N + j]
//   OP 2 (A B^T):  opA(i, r) = A[i R + r],  opB(r, j) = B[j R + r]
// Tiles in bands of 4 tile rows, column by column in a band, each XCD taking a
// contiguous run of them.  Rows and columns past the matrix read its last ones
// and are not stored.
template <class T, int OP>
__device__ __forceinline__ void f32_matmul_tile(float *lds, const float *__restrict__ A,
                                                const float *__restrict__ B,
                                                float *__restrict__ C, long long M, long long N,
                                                long long R, long long m0, long long n0,
                                                int vec_c) {
  const int t = threadIdx.x;
  T tile(t);
  typename T::OpA oa;
  typename T::OpB ob;
  if constexpr (OP == 1)
    oa.init_rm(A + m0, M, M - m0, t);
  else
    oa.init_rc([&](int r) { return A + min(m0 + r, M - 1) * R; }, A, t);
  if constexpr (OP == 2)
    ob.init_rc([&](int r) { return B + min(n0 + r, N - 1) * R; }, B, t);
  else
    ob.init_rm(B + n0, N, N - n0, t);
  if (!tile.run(lds, oa, ob, R, OP == 1 ? T::BK * M : T::BK, OP == 2 ? T::BK : T::BK * N, t))
    return;
#pragma unroll
  for (int i = 0; i < T::MI; ++i)
#pragma unroll
    for (int j = 0; j < T::NJ; ++j) {
      const long long row = m0 + tile.wm * T::WM + 16 * i + (tile.lane & 15);
      const long long col = n0 + tile.wn * T::WN + 16 * j + 4 * (tile.lane >> 4);
      if (row >= M || col >= N) continue;
      float *dst = C + row * N + col;
      if (vec_c) {
        *reinterpret_cast<f32x4 *>(dst) = tile.acc[i][j];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < N) dst[e] = tile.acc[i][j][e];
      }
    }
}

// One workgroup per tile.  Tiles n_full .. are computed as two half-height
// tiles (TH) each, on two workgroups: the last partial round of a launch.
// TH = T: no halves (n_full is the number of tiles).
template <class T, class TH, int OP>
__global__ __launch_bounds__(T::kThreads) void f32_matmul_kernel(
    const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C, long long M,
    long long N, long long R, unsigned m_tiles, unsigned n_tiles, unsigned n_full, int vec_c) {
  static_assert(T::kThreads == TH::kThreads && T::BN == TH::BN, "one launch for both");
  __shared__ __attribute__((aligned(16))) float
      lds[T::kLdsFloats > TH::kLdsFloats ? T::kLdsFloats : TH::kLdsFloats];
  const bool half = blockIdx.x >= n_full;
  const unsigned run = half ? n_full + f32t::xcd_run(blockIdx.x - n_full, gridDim.x - n_full) / 2
                            : f32t::xcd_run(blockIdx.x, n_full);
  const unsigned band = run / n_tiles / 4, in = run - band * 4 * n_tiles;
  const unsigned rows = min(4u, m_tiles - band * 4);
  const long long m0 = (long long)(band * 4 + in % rows) * T::BM;
  const long long n0 = (long long)(in / rows) * T::BN;
  if constexpr (!std::is_same<T, TH>::value) {
    if (half) {
      const unsigned u = f32t::xcd_run(blockIdx.x - n_full, gridDim.x - n_full);
      const long long mh = m0 + (u & 1) * TH::BM;
      if (mh < M) f32_matmul_tile<TH, OP>(lds, A, B, C, M, N, R, mh, n0, vec_c);
      return;
    }
  }
  f32_matmul_tile<T, OP>(lds, A, B, C, M, N, R, m0, n0, vec_c);
}

// Short reductions, where a pipelined tile would mostly fill and drain its two
// stages: one workgroup per 64 x 64 tile (tiles numbered row-major over the
// grid), 4 waves of 32 x 32 (2 x 2 MFMA blocks of 16 x 16), steps of 16
// reduction elements through one padded LDS buffer of 8.5 KiB (eight
// workgroups share a CU and hide each other's loads), loaded with bounds
// checks so that consecutive threads read consecutive addresses of whichever
// index is contiguous.
constexpr int kShortTile = 64;  // output tile (rows and columns)
constexpr int kShortStep = 16;  // reduction elements per LDS stage
constexpr int kShortThreads = 256;

template <int OP>
__global__ __launch_bounds__(kShortThreads) void f32_matmul_short_kernel(
    const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C, long long M,
    long long N, long long R, long long n_tiles) {
  __shared__ float As[kShortTile][kShortStep + 1];
  __shared__ float Bs[kShortTile][kShortStep + 1];
  const long long tile = blockIdx.x;
  const long long m0 = (tile / n_tiles) * kShortTile;
  const long long n0 = (tile % n_tiles) * kShortTile;
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  // Loader coordinates: "rc" = the reduction index is the contiguous one.
  constexpr bool a_rc = OP != 1, b_rc = OP == 2;
  const int a_i = a_rc ? t >> 2 : (t & 15) * 4, a_r = a_rc ? (t & 3) * 4 : t >> 4;
  const int b_j = b_rc ? t >> 2 : (t & 15) * 4, b_r = b_rc ? (t & 3) * 4 : t >> 4;

  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  float ra[4], rb[4];
  auto gload = [&](long long r0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const long long i = m0 + a_i + (a_rc ? 0 : q), ar = r0 + a_r + (a_rc ? q : 0);
      ra[q] = (i < M && ar < R) ? (OP == 1 ? A[ar * M + i] : A[i * R + ar]) : 0.f;
      const long long j = n0 + b_j + (b_rc ? 0 : q), br = r0 + b_r + (b_rc ? q : 0);
      rb[q] = (j < N && br < R) ? (OP == 2 ? B[j * R + br] : B[br * N + j]) : 0.f;
    }
  };
  auto lstore = [&]() {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      As[a_i + (a_rc ? 0 : q)][a_r + (a_rc ? q : 0)] = ra[q];
      Bs[b_j + (b_rc ? 0 : q)][b_r + (b_rc ? q : 0)] = rb[q];
    }
  };

  // MFMA operands (v_mfma_f32_16x16x4f32): lane l holds A[row l%16][k l/16]
  // and B[k l/16][col l%16]; the result lane holds rows 4 (l/16) + 0..3 of
  // column l%16.
  const int fr = lane & 15, fk = lane >> 4;
  gload(0);
  for (long long r0 = 0; r0 < R; r0 += kShortStep) {
    __syncthreads();  // the previous stage's reads are done
    lstore();
    __syncthreads();
    if (r0 + kShortStep < R) gload(r0 + kShortStep);
#pragma unroll
    for (int ks = 0; ks < kShortStep / 4; ++ks) {
      const int kk = ks * 4 + fk;
      float af[2], bf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) af[i] = As[wm * 32 + i * 16 + fr][kk];
#pragma unroll
      for (int j = 0; j < 2; ++j) bf[j] = Bs[wn * 32 + j * 16 + fr][kk];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i], bf[j], acc[i][j], 0, 0, 0);
    }
  }

#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const long long col = n0 + wn * 32 + j * 16 + fr;
      if (col >= N) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const long long row = m0 + wm * 32 + i * 16 + 4 * fk + r;
        if (row < M) C[row * N + col] = acc[i][j][r];
      }
    }
}

// The tile shapes, from large outputs to outputs of a few tiles with a long
// reduction (waves m x n x k: the last split the reduction).
template <int CFG, int OP, int W> struct MatmulCfg;
#define PRICHS_MATMUL_CFG(I, BM, BN, BK, WM, WN, WK)                                      \
  template <int OP, int W> struct MatmulCfg<I, OP, W> {                                   \
    typedef f32t::Tile<BM, BN, BK, WM, WN, WK, OP != 1, OP == 2, W> T;                    \
    typedef T TH;                                                                         \
  };
PRICHS_MATMUL_CFG(0, 128, 128, 32, 2, 2, 1)
PRICHS_MATMUL_CFG(1, 64, 64, 64, 2, 2, 2)
PRICHS_MATMUL_CFG(2, 32, 64, 64, 1, 2, 2)
PRICHS_MATMUL_CFG(3, 32, 32, 64, 2, 2, 2)
PRICHS_MATMUL_CFG(4, 16, 16, 256, 1, 1, 8)
#undef PRICHS_MATMUL_CFG
// 64 x 64 tiles with the last partial round as 32 x 64 halves.
template <int OP, int W> struct MatmulCfg<5, OP, W> {
  typedef f32t::Tile<64, 64, 32, 2, 2, 1, OP != 1, OP == 2, W> T;
  typedef f32t::Tile<32, 64, 64, 1, 2, 2, OP != 1, OP == 2, W> TH;
};
constexpr int kMatmulCfgs = 5;

// Nanoseconds per reduction element of one tile on a CU: alone, and each of
// several on the same CU (measured on MI355X at 512 x 512 x 2048, 128 x 128 x
// 4096, 1024^3, 2048 x 1280 x 1536 and 4096 x 4096 x 1024; the single-element
// loads at 145 x 58 x 1895 and 1001 x 777 x 333, where they bound the small
// tiles).  The shape with the least whole rounds x time wins: at 1024^3 64 x
// 64 tiles take 22.0 us against 69.5 (128 x 128, 64 CUs busy) and 25.6 (32 x
// 32), at 4096 x 4096 x 1024 288 against 258 and 356, at 128 x 128 x 4096 72
// against 256 and 26, and 16 x 16 with the reduction over 8 waves 10.2.
struct MatmulTileCost {
  int bm, bn, bk, threads;
  double alone[2], shared[2];  // [0] 16-byte, [1] single-element loads
};
constexpr MatmulTileCost kMatmulCost[kMatmulCfgs] = {
    {128, 128, 32, 256, {63.0, 78.0}, {63.0, 78.0}},
    {64, 64, 64, 512, {18.6, 30.0}, {17.8, 30.0}},
    {32, 64, 64, 256, {12.7, 18.0}, {9.7, 20.0}},
    {32, 32, 64, 512, {7.2, 10.5}, {5.6, 11.0}},
    {16, 16, 256, 512, {2.5, 5.7}, {2.6, 10.0}},
};
// A launch has at most 2^32 - 1 threads in x.
constexpr double kMaxLaunchThreads = 4294967295.0;

// Configuration 5: a last partial round of at most half the CUs in half tiles
// (2048 x 1280 x 1536: 640 tiles are 2.5 rounds, 71.0 us against 75.0 in 32
// x 64 tiles and 83 in whole 64 x 64 ones).
constexpr double kMatmulWhole = 17.6, kMatmulHalf = 9.8;
bool matmul_halves(size_t M, size_t N, int cus, size_t &full) {
  const size_t tiles = cdiv(M, 64) * cdiv(N, 64), tail = tiles % (size_t)cus;
  full = tiles - tail;
  return full > 0 && tail > 0 && 2 * tail <= (size_t)cus;
}

// Configuration 6: the kernel for short reductions.  Before its first products a
// pipelined tile fetches and stores its stages, as long as the products of 98
// reduction elements with 16-byte loads and of 224 with single ones; the short
// kernel has no such start but takes longer per element, 9 ns and 42.5 for each
// 64 x 64 tile on a CU (partly filled rounds count three quarters as whole ones).
// Fitted to 2919 measured sizes; the choice is the slower one by more than 8% on
// 3 of them.  MI355X, us, pipelined -> short: 4096 x 4096 outputs of 16 elements
// 24.5 -> 18.2, 3000 x 3001 of 17 43.2 -> 15.4, 341 x 3005 of 1 13.8 -> 4.7, 1341
// x 1245 of 91 21.0 -> 9.8, 936 x 1140 of 613 31.2 -> 46.6; on small outputs the
// two meet near 40 elements with single-element loads and near 16 with 16-byte
// ones (60 x 84 of 64: 3.9 -> 6.0).
constexpr int kMatmulShort = 6;
constexpr double kShortBase = 9.0, kShortTileCost = 42.5, kFillElems[2] = {98.0, 224.0};

int matmul_cfg(size_t M, size_t N, size_t R, bool vec, int cus) {
  int best = 0, bk = 0;
  double best_t = 0, per = 0;  // per: ns per reduction element
  for (int c = 0; c < kMatmulCfgs; ++c) {
    const MatmulTileCost &k = kMatmulCost[c];
    const double tiles = (double)cdiv(M, k.bm) * (double)cdiv(N, k.bn);
    if (c > 0 && tiles * k.threads > kMaxLaunchThreads) continue;
    const double e = std::max(k.alone[!vec], std::ceil(tiles / cus) * k.shared[!vec]);
    const double t = (double)roundup(R, k.bk) * e;
    if (c == 0 || t < best_t) best = c, best_t = t, per = e, bk = k.bk;
  }
  size_t full = 0;
  if (vec && matmul_halves(M, N, cus, full) && (double)(full + cus) * 256 <= kMaxLaunchThreads) {
    const double e = (double)(full / cus) * kMatmulWhole + kMatmulHalf;
    if ((double)roundup(R, 32) * e < best_t) best = 5, per = e, bk = 32;
  }
  const double tiles = (double)cdiv(M, kShortTile) * (double)cdiv(N, kShortTile);
  const double rounds = std::max(1.0, 0.25 * tiles / cus + 0.75 * std::ceil(tiles / cus));
  if (tiles * kShortThreads <= kMaxLaunchThreads &&
      (double)roundup(R, kShortStep) * (kShortBase + kShortTileCost * rounds) <
          ((double)roundup(R, bk) + kFillElems[!vec]) * per)
    return kMatmulShort;
  return best;
}

// Product of two sizes, or SIZE_MAX when it overflows.
size_t mul_sat(size_t a, size_t b) { return (b != 0 && a > SIZE_MAX / b) ? SIZE_MAX : a * b; }

// Output [M, N] and reduction length R of an op in the reference's (m, k, n)
// naming, and the element counts of a, b, c.
struct MatmulDims {
  size_t M, N, R, a_elems, b_elems, c_elems;
};
MatmulDims matmul_dims(int op, size_t m, size_t k, size_t n) {
  MatmulDims d{};
  if (op == PRICHS_MATMUL_ATB) {
    d = {k, n, m, mul_sat(m, k), mul_sat(m, n), mul_sat(k, n)};
  } else if (op == PRICHS_MATMUL_ABT) {
    d = {m, n, k, mul_sat(m, k), mul_sat(n, k), mul_sat(m, n)};
  } else {
    d = {m, n, k, mul_sat(m, k), mul_sat(k, n), mul_sat(m, n)};
  }
  return d;
}

int check_matmul(int op, size_t m, size_t k, size_t n, const char *who, MatmulDims &d) {
  PRICHS_REQUIRE(op == PRICHS_MATMUL_AB || op == PRICHS_MATMUL_ATB || op == PRICHS_MATMUL_ABT,
                 "%s: unknown op %d", who, op);
  d = matmul_dims(op, m, k, n);
  const size_t lim = (size_t)1 << 46;  // element counts: far past any device, no overflow below
  PRICHS_REQUIRE(d.a_elems < lim && d.b_elems < lim && d.c_elems < lim,
                 "%s: m=%zu, k=%zu, n=%zu too large", who, m, k, n);
  return PRICHS_OK;
}

template <int CFG, int OP, int W>
void launch_matmul_kernel(const float *a, const float *b, float *c, const MatmulDims &d, int vec_c,
                          hipStream_t s) {
  typedef typename MatmulCfg<CFG, OP, W>::T T;
  typedef typename MatmulCfg<CFG, OP, W>::TH TH;
  static_assert(CFG >= kMatmulCfgs || T::kThreads == kMatmulCost[CFG < kMatmulCfgs ? CFG : 0].threads,
                "the cost table's workgroup");
  const unsigned mt = (unsigned)cdiv(d.M, T::BM), nt = (unsigned)cdiv(d.N, T::BN);
  size_t full = (size_t)mt * nt;
  if (!std::is_same<T, TH>::value) matmul_halves(d.M, d.N, device_cu_count(), full);
  const unsigned grid = (unsigned)(full + 2 * ((size_t)mt * nt - full));
  hipLaunchKernelGGL((f32_matmul_kernel<T, TH, OP>), dim3(grid), dim3(T::kThreads), 0, s, a, b, c,
                     (long long)d.M, (long long)d.N, (long long)d.R, mt, nt, (unsigned)full,
                     vec_c);
}

template <int OP>
void launch_matmul_short(const float *a, const float *b, float *c, const MatmulDims &d,
                         hipStream_t s) {
  const size_t nt = cdiv(d.N, kShortTile);
  hipLaunchKernelGGL(f32_matmul_short_kernel<OP>, dim3((unsigned)(cdiv(d.M, kShortTile) * nt)),
                     dim3(kShortThreads), 0, s, a, b, c, (long long)d.M, (long long)d.N,
                     (long long)d.R, (long long)nt);
}

template <int OP, int W>
void launch_matmul_cfg(int cfg, const float *a, const float *b, float *c, const MatmulDims &d,
                       int vec_c, hipStream_t s) {
  switch (cfg) {
    case 0: return launch_matmul_kernel<0, OP, W>(a, b, c, d, vec_c, s);
    case 1: return launch_matmul_kernel<1, OP, W>(a, b, c, d, vec_c, s);
    case 2: return launch_matmul_kernel<2, OP, W>(a, b, c, d, vec_c, s);
    case 3: return launch_matmul_kernel<3, OP, W>(a, b, c, d, vec_c, s);
    case 5: return launch_matmul_kernel<W == 4 ? 5 : 4, OP, W>(a, b, c, d, vec_c, s);
    case kMatmulShort: return launch_matmul_short<OP>(a, b, c, d, s);
    default: return launch_matmul_kernel<4, OP, W>(a, b, c, d, vec_c, s);
  }
}

int launch_matmul(int op, const float *a, const float *b, float *c, const MatmulDims &d,
                  hipStream_t s) {
  if (d.M == 0 || d.N == 0) return PRICHS_OK;
  PRICHS_REQUIRE(cdiv(d.M, 64) * cdiv(d.N, 64) <= (size_t)INT32_MAX,
                 "matmul: %zu x %zu output has too many tiles", d.M, d.N);
  const int cus = device_cu_count();
  if (cus <= 0) return fail(PRICHS_ERR_HIP, "matmul: cannot query the device");
  // 16-byte loads where every row of both operands starts 16-byte aligned,
  // 16-byte stores where every row of C does.
  auto aligned = [](const float *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const size_t lda = op == PRICHS_MATMUL_ATB ? d.M : d.R;
  const size_t ldb = op == PRICHS_MATMUL_ABT ? d.R : d.N;
  const bool vec = lda % 4 == 0 && ldb % 4 == 0 && aligned(a) && aligned(b);
  const int vec_c = d.N % 4 == 0 && aligned(c);
  const int cfg = matmul_cfg(d.M, d.N, d.R, vec, cus);
#define PRICHS_MATMUL_OP(OP)                                     \
  (vec ? launch_matmul_cfg<OP, 4>(cfg, a, b, c, d, vec_c, s)     \
       : launch_matmul_cfg<OP, 1>(cfg, a, b, c, d, vec_c, s))
  if (op == PRICHS_MATMUL_ATB)
    PRICHS_MATMUL_OP(1);
  else if (op == PRICHS_MATMUL_ABT)
    PRICHS_MATMUL_OP(2);
  else
    PRICHS_MATMUL_OP(0);
#undef PRICHS_MATMUL_OP
  PRICHS_LAUNCH_CHECK("matmul launch");
  return PRICHS_OK;
}

// The reference's slab sizes (cublas.rs:77-84): A 16 MB, B 32 MB, C 16 MB.
constexpr size_t kDefaultSlabA = 16u << 20, kDefaultSlabB = 32u << 20, kDefaultSlabC = 16u << 20;

struct Guard {
  int prev = -1;
  bool ok = true;
  explicit Guard(int dev) {
    if (hipGetDevice(&prev) != hipSuccess) {
      ok = false;
      return;
    }
    if (prev != dev && hipSetDevice(dev) != hipSuccess) ok = false;
  }
  ~Guard() {
    int cur = -1;
    if (prev >= 0 && hipGetDevice(&cur) == hipSuccess && cur != prev) (void)hipSetDevice(prev);
  }
};

// H2D of a and b into slabs A and B, the product into slab C, D2H, device
// synchronisation: the sequence of GpuWorkspace::matmul (cublas.rs:117-166).
int workspace_run(prichs_gpu_workspace *ws, int op, const float *a, const float *b, float *c,
                  size_t m, size_t k, size_t n, const char *who) {
  PRICHS_REQUIRE(ws != nullptr, "%s: null workspace", who);
  MatmulDims d;
  if (int rc = check_matmul(op, m, k, n, who, d)) return rc;
  PRICHS_REQUIRE((a || d.a_elems == 0) && (b || d.b_elems == 0) && (c || d.c_elems == 0),
                 "%s: null pointer argument", who);
  if (d.a_elems * 4 > ws->cap_a || d.b_elems * 4 > ws->cap_b || d.c_elems * 4 > ws->cap_c)
    return fail(PRICHS_ERR_CAPACITY,
                "%s: matrix dimensions exceed preallocated GPU workspace slabs (m=%zu, k=%zu, "
                "n=%zu; slabs %zu/%zu/%zu bytes)",
                who, m, k, n, ws->cap_a, ws->cap_b, ws->cap_c);
  if (d.c_elems == 0) return PRICHS_OK;
  Guard g(ws->device);
  if (!g.ok) return fail(PRICHS_ERR_HIP, "%s: cannot select device %d", who, ws->device);
  if (d.a_elems)
    PRICHS_HIP_TRY(hipMemcpy(ws->a, a, d.a_elems * 4, hipMemcpyHostToDevice), "workspace: H2D A");
  if (d.b_elems)
    PRICHS_HIP_TRY(hipMemcpy(ws->b, b, d.b_elems * 4, hipMemcpyHostToDevice), "workspace: H2D B");
  if (int rc = launch_matmul(op, ws->a, ws->b, ws->c, d, nullptr)) return rc;
  PRICHS_HIP_TRY(hipMemcpy(c, ws->c, d.c_elems * 4, hipMemcpyDeviceToHost), "workspace: D2H C");
  PRICHS_HIP_TRY(hipDeviceSynchronize(), "workspace: synchronize");
  return PRICHS_OK;
}

// The process-wide workspace of get_gpu_workspace (cublas.rs:283-300):
// created with the reference's slab sizes on first use, on the device that
// is current then; if that fails it stays absent, as the reference's Lazy
// does.  Its calls are serialised by g_ws_mu (the reference's Mutex).
std::mutex g_ws_mu;
prichs_gpu_workspace *g_ws = nullptr;
bool g_ws_tried = false;
char g_ws_error[512] = {0};

prichs_gpu_workspace *global_workspace_locked() {
  if (!g_ws_tried) {
    g_ws_tried = true;
    if (prichs_gpu_workspace_create(0, 0, 0, &g_ws) != PRICHS_OK) {
      g_ws = nullptr;
      snprintf(g_ws_error, sizeof g_ws_error, "%s", prichs_last_error());
    }
  }
  if (!g_ws) set_error("GPU workspace unavailable: %s", g_ws_error);
  return g_ws;
}

// One call on a handle, under that handle's lock: the slabs are shared by
// every caller of the handle (the process-wide one included).
int locked_run(prichs_gpu_workspace *ws, int op, const float *a, const float *b, float *c,
               size_t m, size_t k, size_t n, const char *who) {
  PRICHS_REQUIRE(ws != nullptr, "%s: null workspace", who);
  std::lock_guard<std::mutex> lock(ws->mu);
  return workspace_run(ws, op, a, b, c, m, k, n, who);
}

int global_run(int op, const float *a, const float *b, float *c, size_t m, size_t k, size_t n,
               const char *who) {
  prichs_gpu_workspace *ws;
  {
    std::lock_guard<std::mutex> lock(g_ws_mu);
    ws = global_workspace_locked();
  }
  if (!ws) return PRICHS_ERR_HIP;
  return locked_run(ws, op, a, b, c, m, k, n, who);
}

}  // namespace
}  // namespace prichs

using namespace prichs;

extern "C" int prichs_matmul_f32(int op, const float *a, const float *b, float *c, size_t m,
                                 size_t k, size_t n, void *stream) {
  MatmulDims d;
  if (int rc = check_matmul(op, m, k, n, "matmul_f32", d)) return rc;
  if (d.c_elems == 0) return PRICHS_OK;
  PRICHS_REQUIRE((a || d.a_elems == 0) && (b || d.b_elems == 0) && c,
                 "matmul_f32: null pointer argument");
  return launch_matmul(op, a, b, c, d, as_stream(stream));
}

extern "C" int prichs_gpu_workspace_create(size_t a_bytes, size_t b_bytes, size_t c_bytes,
                                           prichs_gpu_workspace **out) {
  PRICHS_REQUIRE(out != nullptr, "gpu_workspace_create: null output handle");
  *out = nullptr;
  if (a_bytes == 0) a_bytes = kDefaultSlabA;
  if (b_bytes == 0) b_bytes = kDefaultSlabB;
  if (c_bytes == 0) c_bytes = kDefaultSlabC;
  const size_t ra = roundup(a_bytes, 256), rb = roundup(b_bytes, 256), rc_ = roundup(c_bytes, 256);
  PRICHS_REQUIRE(ra >= a_bytes && rb >= b_bytes && rc_ >= c_bytes && ra <= ((size_t)1 << 44) &&
                     rb <= ((size_t)1 << 44) && rc_ <= ((size_t)1 << 44),
                 "gpu_workspace_create: slab sizes too large");
  prichs_gpu_workspace *ws = new (std::nothrow) prichs_gpu_workspace();
  if (!ws) return fail(PRICHS_ERR_CAPACITY, "gpu_workspace_create: out of host memory");
  if (hipGetDevice(&ws->device) != hipSuccess) {
    delete ws;
    return fail(PRICHS_ERR_HIP, "gpu_workspace_create: no HIP device");
  }
  const hipError_t e = hipMalloc(&ws->base, ra + rb + rc_);
  if (e != hipSuccess) {
    delete ws;
    return fail(PRICHS_ERR_CAPACITY, "gpu_workspace_create: hipMalloc(%zu bytes): %s",
                ra + rb + rc_, hipGetErrorString(e));
  }
  char *p = static_cast<char *>(ws->base);
  ws->a = reinterpret_cast<float *>(p);
  ws->b = reinterpret_cast<float *>(p + ra);
  ws->c = reinterpret_cast<float *>(p + ra + rb);
  ws->cap_a = a_bytes;
  ws->cap_b = b_bytes;
  ws->cap_c = c_bytes;
  *out = ws;
  return PRICHS_OK;
}

extern "C" int prichs_gpu_workspace_destroy(prichs_gpu_workspace *ws) {
  if (!ws) return PRICHS_OK;
  {
    // The process-wide workspace lives until the process ends, as the
    // reference's static does (cublas.rs:283-300).
    std::lock_guard<std::mutex> lock(g_ws_mu);
    PRICHS_REQUIRE(ws != g_ws, "gpu_workspace_destroy: the process-wide workspace "
                               "(get_gpu_workspace) is not destroyed by callers");
  }
  int rc = PRICHS_OK;
  {
    Guard g(ws->device);
    if (ws->base && hipFree(ws->base) != hipSuccess)
      rc = fail(PRICHS_ERR_HIP, "gpu_workspace_destroy: hipFree failed");
  }
  delete ws;
  return rc;
}

extern "C" int prichs_gpu_workspace_slabs(const prichs_gpu_workspace *ws, size_t *a_bytes,
                                          size_t *b_bytes, size_t *c_bytes) {
  PRICHS_REQUIRE(ws != nullptr, "gpu_workspace_slabs: null workspace");
  if (a_bytes) *a_bytes = ws->cap_a;
  if (b_bytes) *b_bytes = ws->cap_b;
  if (c_bytes) *c_bytes = ws->cap_c;
  return PRICHS_OK;
}

extern "C" int prichs_gpu_workspace_matmul(prichs_gpu_workspace *ws, const float *a,
                                           const float *b, float *c, size_t m, size_t k,
                                           size_t n) {
  return locked_run(ws, PRICHS_MATMUL_AB, a, b, c, m, k, n, "gpu_workspace_matmul");
}

extern "C" int prichs_gpu_workspace_matmul_at_b(prichs_gpu_workspace *ws, const float *a,
                                                const float *b, float *dw, size_t m, size_t k,
                                                size_t n) {
  return locked_run(ws, PRICHS_MATMUL_ATB, a, b, dw, m, k, n, "gpu_workspace_matmul_at_b");
}

extern "C" int prichs_gpu_workspace_matmul_a_bt(prichs_gpu_workspace *ws, const float *dy,
                                                const float *w, float *dx, size_t m, size_t k,
                                                size_t n) {
  return locked_run(ws, PRICHS_MATMUL_ABT, dy, w, dx, m, k, n, "gpu_workspace_matmul_a_bt");
}

extern "C" prichs_gpu_workspace *prichs_get_gpu_workspace(void) {
  std::lock_guard<std::mutex> lock(g_ws_mu);
  return global_workspace_locked();
}

extern "C" int prichs_matmul_gpu(const float *a, const float *b, float *c, size_t m, size_t k,
                                 size_t n) {
  return global_run(PRICHS_MATMUL_AB, a, b, c, m, k, n, "matmul_gpu");
}

extern "C" int prichs_matmul_at_b_gpu(const float *a, const float *b, float *dw, size_t m,
                                      size_t k, size_t n) {
  return global_run(PRICHS_MATMUL_ATB, a, b, dw, m, k, n, "matmul_at_b_gpu");
}

extern "C" int prichs_matmul_a_bt_gpu(const float *dy, const float *w, float *dx, size_t m,
                                      size_t k, size_t n) {
  return global_run(PRICHS_MATMUL_ABT, dy, w, dx, m, k, n, "matmul_a_bt_gpu");
}
