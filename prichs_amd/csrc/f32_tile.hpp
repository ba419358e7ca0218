// f32_tile.hpp -- the f32 MFMA tile shared by the general f32 GEMMs, the f32
// grouped GEMMs and the f32 weight gradients.
//
// One workgroup computes a BM x BN tile of C[i][j] = sum_r opA(i, r) opB(r, j)
// on v_mfma_f32_16x16x4f32 (f32 products, f32 accumulation).  Each operand
// comes in one of two storage orders: reduction-contiguous ("RC", rows of
// consecutive r) or reduction-major (rows of consecutive i or j for each r).
//
// Pipeline: global -> registers two stages of BK reduction elements ahead of
// the products, registers -> one of two LDS buffers one stage ahead, one
// barrier per stage; fragments LDS -> registers one 16-element slice ahead.
// Loads are unpredicated (an address past the reduction is replaced by the
// operand's first one and its value by zero at the LDS store), so the
// compiler's waits stay exact and a stage's loads stay in flight behind the
// whole of the previous stage's products.
//
// LDS: an RC operand keeps [row][BK] with 16-byte chunk c of row r at slot
// c ^ (r & 7), so a fragment is read as one ds_read_b128 per lane (rows 0..7
// on distinct banks); lane group q = lane / 16 then holds r = 4q .. 4q + 3 of
// a 16-element slice, which it feeds to four MFMAs.  A reduction-major
// operand keeps [r][rows + 4] and reads the same four r's as ds_read_b32 (the
// pad puts the four lane groups, 4 rows apart, on two bank halves).  Both
// operands use the same r for the same MFMA slot, so the sum only runs over r
// in another order.
//
// The four MFMAs of a 16 x 16 x 16 slice keep a SIMD busy for 128 cycles, so
// what costs is whatever stalls the issuing wave: with the memory instructions
// of a stage in a row, 4096 x 4096 x 1024 took 289-297 us in 128 x 128 tiles;
// with one of them in front of each share of the MFMAs (no branch in a whole
// stage, sched_group_barrier) 253-260 us, 134 of the 154 TFLOP/s that MFMAs
// alone reach.  2048 x 1280 x 1536: 196 us (64 x 64 tiles, 4-byte checked
// loads, one LDS buffer) -> 71 us.
//
// WGK > 1: that many waves share an output block and split each stage's
// 16-element slices; their sums are added in wave order through LDS at the
// end (deterministic).  It is what gives a small output with a long reduction
// enough waves.
#pragma once

#include "common.hpp"

namespace prichs {
namespace f32t {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Wrapper: a builtin called with template-dependent arguments fails silently
// in the host pass.
__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Tile `b` of `n` for workgroup b: workgroups are dealt round-robin to the 8
// XCDs, each of which takes a contiguous run of tiles (any n) so that
// neighbouring tiles share operand panels in its L2.
__device__ __forceinline__ unsigned xcd_run(unsigned b, unsigned n) {
  const unsigned x = b & 7, q = n >> 3, r = n & 7;
  return x * q + (x < r ? x : r) + (b >> 3);
}

// Order of a slice's instructions: each memory instruction in front of a share
// of the MFMAs (in a row they would keep the wave, and with one or two waves
// per SIMD the matrix pipe, waiting for the LDS).
template <class OpA, class OpB, int MFMAS, int READS>
__device__ __forceinline__ void interleave_slice(bool first) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int kMem = OpA::N + OpB::N;
  if (first) {
    constexpr int kShare = MFMAS / (kMem + READS) > 0 ? MFMAS / (kMem + READS) : 1;
#pragma unroll
    for (int i = 0; i < kMem; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // DS write
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // global load
      __builtin_amdgcn_sched_group_barrier(0x008, kShare, 0);
    }
#pragma unroll
    for (int i = 0; i < READS; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
      __builtin_amdgcn_sched_group_barrier(0x008, kShare, 0);
    }
  } else {
    constexpr int kShare = MFMAS / READS > 0 ? MFMAS / READS : 1;
#pragma unroll
    for (int i = 0; i < READS; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, kShare, 0);
    }
  }
#endif
}

// ROWS x BK of one operand, staged by THREADS threads in pieces of W elements:
// 16-byte chunks where the operand's base and row stride allow them (W = 4),
// else single elements, dealt so that a wave still reads whole lines.
template <int ROWS, int BK, bool RC, int W, int THREADS> struct Operand {
  static constexpr int kLd = RC ? BK : ROWS + 4;            // LDS row (floats)
  static constexpr int kElems = RC ? ROWS * BK : BK * kLd;  // one stage
  static constexpr int kPerRow = (RC ? BK : ROWS) / W;      // pieces of a row
  static constexpr int N = ROWS * BK / W / THREADS;         // pieces per thread
  static_assert((W == 4 || W == 1) && ROWS * BK % (W * THREADS) == 0 && (!RC || BK % 32 == 0),
                "whole pieces per thread");
  typedef float piece __attribute__((ext_vector_type(W)));

  const float *p[N];  // this thread's pieces of the next stage
  const float *safe;  // a readable piece of this operand
  piece v[N];
  bool whole;         // the stage in v lies inside the reduction
  int left;           // else: how many of its reduction elements do

  // Position of piece i of thread t: LDS row and place in it, and its (first)
  // reduction element.
  __device__ static int row_of(int i, int t) { return (t + i * THREADS) / kPerRow; }
  __device__ static int col_of(int i, int t) { return (t + i * THREADS) % kPerRow * W; }
  __device__ static int red_of(int i, int t) { return RC ? col_of(i, t) : row_of(i, t); }

  // Reduction-contiguous: row_ptr(row) = element (row, r = 0) of a readable row.
  template <class F> __device__ void init_rc(F row_ptr, const float *first, int t) {
    safe = first;
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = row_ptr(row_of(i, t)) + col_of(i, t);
  }
  // Reduction-major: element (r, c) at base + r * ld + c, n_cols columns from
  // the tile's first one on (columns past them read the last piece; their
  // outputs are dropped).
  __device__ void init_rm(const float *base, long long ld, long long n_cols, int t) {
    safe = base;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const long long c = col_of(i, t), last = n_cols - W;
      p[i] = base + (long long)row_of(i, t) * ld + (c < last ? c : last);
    }
  }

  // Loads the next stage, the reduction elements [r0, r0 + BK) of R, and
  // advances by it (step elements).  Stages past the reduction load nothing
  // of use (a readable address).  WHOLE: the caller knows that the stage lies
  // inside the reduction (no branch).
  template <bool WHOLE> __device__ __forceinline__ void fetch(long long r0, long long R,
                                                              long long step, int t) {
    whole = WHOLE || R - r0 >= BK;
    if (whole) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        v[i] = *reinterpret_cast<const piece *>(p[i]);
        p[i] += step;
      }
    } else {
      left = (int)(R - r0 > 0 ? R - r0 : 0);
#pragma unroll
      for (int i = 0; i < N; ++i)
        v[i] = *reinterpret_cast<const piece *>(red_of(i, t) < left ? p[i] : safe);
    }
  }

  template <bool WHOLE> __device__ __forceinline__ void store(float *lds, int t) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if (!WHOLE && !whole && red_of(i, t) >= left) v[i] = 0.f;
      const int r = row_of(i, t), c = col_of(i, t);
      float *dst = lds + r * kLd + (RC ? (((c >> 2) ^ (r & 7)) << 2) + (c & 3) : c);
      *reinterpret_cast<piece *>(dst) = v[i];
    }
  }

  // Fragment of 16 rows from `row` on, slice sl (16 reduction elements).
  __device__ __forceinline__ static f32x4 frag(const float *lds, int row, int sl, int lane) {
    const int r = row + (lane & 15), q = lane >> 4;
    if (RC) return *reinterpret_cast<const f32x4 *>(lds + r * kLd + (((4 * sl + q) ^ (r & 7)) << 2));
    f32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = lds[(16 * sl + 4 * q + e) * kLd + r];
    return w;
  }
};

template <int BM_, int BN_, int BK_, int WGM_, int WGN_, int WGK_, bool ARC_, bool BRC_, int W_ = 4>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, BK = BK_;
  static constexpr int WGM = WGM_, WGN = WGN_, WGK = WGK_;
  static constexpr int kThreads = 64 * WGM * WGN * WGK;
  static constexpr int WM = BM / WGM, WN = BN / WGN;
  static constexpr int MI = WM / 16, NJ = WN / 16;
  static constexpr int kSlices = BK / 16 / WGK;  // 16-element slices of a wave per stage
  typedef Operand<BM, BK, ARC_, W_, kThreads> OpA;
  typedef Operand<BN, BK, BRC_, W_, kThreads> OpB;
  // LDS read instructions of a slice (two b32 in one for reduction-major).
  static constexpr int kReads = MI * (ARC_ ? 1 : 2) + NJ * (BRC_ ? 1 : 2);
  static constexpr int kStage = OpA::kElems + OpB::kElems;
  static constexpr int kLdsFloats = 2 * kStage;
  static_assert(BK % (16 * WGK) == 0 && BM % (16 * WGM) == 0 && BN % (16 * WGN) == 0, "");
  static_assert((WGK - 1) * BM * BN <= kLdsFloats, "the K split's sums fit the stage buffers");

  int lane, wm, wn, wk;
  // acc[i][j]: lane holds row 16 i + lane % 16 and columns 16 j + 4 (lane / 16)
  // .. + 3 of the wave's block (the B fragment is the MFMA's first operand).
  f32x4 acc[MI][NJ];

  __device__ Tile(int t) {
    lane = t & 63;
    const int w = t >> 6;
    wk = w / (WGM * WGN);
    wm = w % (WGM * WGN) / WGN;
    wn = w % WGN;
  }

  // Fragments of one slice.
  struct Frags {
    f32x4 a[MI], b[NJ];
  };
  __device__ __forceinline__ void read(Frags &f, const float *stage, int s) const {
    const int sl = wk * kSlices + s;
#pragma unroll
    for (int i = 0; i < MI; ++i) f.a[i] = OpA::frag(stage, wm * WM + 16 * i, sl, lane);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      f.b[j] = OpB::frag(stage + OpA::kElems, wn * WN + 16 * j, sl, lane);
  }
  __device__ __forceinline__ void products(const Frags &f) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = mfma_f32(f.b[j][e], f.a[i][e], acc[i][j]);
  }

  // One stage: products of the stage in cur (its first slice's fragments are
  // in f[0]) while the next stage goes to nx and the one after into registers.
  // FAST: both lie inside the reduction, and the block has no branch, so the
  // memory instructions interleave with the MFMAs.
  template <bool FAST>
  __device__ __forceinline__ void stage(Frags (&f)[2], const float *cur, float *nx, OpA &oa,
                                        OpB &ob, long long r0, long long R, long long a_step,
                                        long long b_step, int t) {
    // nx's last readers are past the barrier of the stage before.
    oa.template store<FAST>(nx, t);
    ob.template store<FAST>(nx + OpA::kElems, t);
    oa.template fetch<FAST>(r0 + 2 * BK, R, a_step, t);
    ob.template fetch<FAST>(r0 + 2 * BK, R, b_step, t);
#pragma unroll
    for (int sl = 0; sl < kSlices; ++sl) {
      // Each slice's products cover the reads of the next slice; the barrier
      // of the stage sits before its last slice, whose products cover the
      // first reads of the next stage.
      if (sl + 1 < kSlices) {
        read(f[(sl + 1) & 1], cur, sl + 1);
      } else {
        lds_write_barrier();
        read(f[(sl + 1) & 1], nx, 0);
      }
      products(f[sl & 1]);
      if (FAST) interleave_slice<OpA, OpB, 4 * MI * NJ, kReads>(sl == 0);
    }
    if (kSlices & 1) f[0] = f[1];
  }

  // The whole reduction; a_step / b_step: elements by which one stage advances
  // the operand (BK for RC, BK * ld otherwise).  Returns whether this wave
  // holds the result (wk == 0).
  __device__ __forceinline__ bool run(float *lds, OpA &oa, OpB &ob, long long R, long long a_step,
                                      long long b_step, int t) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (R > 0) {
      oa.template fetch<false>(0, R, a_step, t);
      ob.template fetch<false>(0, R, b_step, t);
      oa.template store<false>(lds, t);
      ob.template store<false>(lds + OpA::kElems, t);
      oa.template fetch<false>(BK, R, a_step, t);
      ob.template fetch<false>(BK, R, b_step, t);
      lds_write_barrier();
      Frags f[2];
      read(f[0], lds, 0);
      long long r0 = 0;
      int buf = 0;
      for (; r0 + 3 * BK <= R; r0 += BK, buf ^= 1)
        stage<true>(f, lds + buf * kStage, lds + (buf ^ 1) * kStage, oa, ob, r0, R, a_step,
                            b_step, t);
      for (; r0 < R; r0 += BK, buf ^= 1)
        stage<false>(f, lds + buf * kStage, lds + (buf ^ 1) * kStage, oa, ob, r0, R,
                             a_step, b_step, t);
    }
    if (WGK == 1) return true;
    lds_write_barrier();  // the last stage's reads ahead are done
    float *part = lds + ((wm * WGN + wn) * 64 + lane) * 4;
    constexpr int kBlock = WGM * WGN * 64 * 4, kWave = MI * NJ * kBlock;
    if (wk > 0) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          *reinterpret_cast<f32x4 *>(part + (wk - 1) * kWave + (i * NJ + j) * kBlock) = acc[i][j];
    }
    lds_write_barrier();
    if (wk > 0) return false;
#pragma unroll
    for (int k = 0; k < WGK - 1; ++k)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          acc[i][j] += *reinterpret_cast<const f32x4 *>(part + k * kWave + (i * NJ + j) * kBlock);
    return true;
  }
};

}  // namespace f32t
}  // namespace prichs
