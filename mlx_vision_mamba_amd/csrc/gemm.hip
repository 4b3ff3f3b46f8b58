// float32 matrix products for the block's projections on the bf16 matrix
// units of gfx950 (in_proj / out_proj and their gradients,
// mamba_block.py:125, :153, :165, :191).
//
// Why not the float32 matrix instructions: they reach 155 TFLOP/s on this
// chip, the bf16 ones 1,700-1,800 from registers.  The method is a published
// one (Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial
// intelligence datatype for higher-precision computations", 2019): every
// float32 x is the exact sum of three bf16 values
//   hi = bf16(x), mid = bf16(x - hi), lo = x - hi - mid    (round to nearest)
// (24 = 8 + 8 + 8 significand bits), and
//   a b = hi hi + (hi mid + mid hi) + (mid mid + hi lo + lo hi) + r,
// |r| <= 2^-25 |a b| at the most and about 2^-28 on average: six bf16 products stand for
// one float32 product, ~290 TFLOP/s at best.  The products of bf16 values
// are exact in float32, and a 32x32x16 MFMA rounds the sum of its 16 less
// often than 16 float32 FMAs do.
//
// hi hi has an accumulator of its own.  The matrix unit cuts off, downwards,
// what lies far below the accumulator: with the small products added to the
// same one, C came out low by 2e-8 of its rms (k = 384) whatever its sign,
// invisible in C's own error but not in later sums over its rows (a block's
// x_proj weight gradient: 4e-5 instead of 3e-6).  Apart, the mean error is
// that of the float32 instructions (3e-10), and the error in the 2-norm
// against float64 1.1e-7 at k = 384 and 2.7e-7 at k = 6144 in 3 parts (normal
// inputs; the BLAS library's float32 matrix instructions: 3.5e-7 and 1.4e-6).
//
// What the split cannot hold, and what is done.  Infinities and NaN (and
// values above the largest bf16, which round to infinity) make a NaN out of
// hi - hi.  Below 2^-110 the low parts are finer than bf16's smallest subnormal
// and lose up to 2^-134, which a result c shows only if it is small beside the
// other operand: len 2^-133 max(|A|, |B|) > 2^-24 |c|.  And products of parts
// below 2^-126 may be lost, which shows in |c| < 6 len 2^-102.  So every thread
// keeps the largest magnitude of its share of the row (or column) it stages,
// one instruction per two values, and a wave computes its part of the tile
// again with the float32 matrix instructions, which have none of these limits,
// when
//   - a result is not finite;
//   - a row or a column it uses is nonzero but below 2^-110 throughout (its
//     results may have lost everything); or
//   - a nonzero result is below one of the two bounds.
// Rows and columns are looked at, through LDS, only in a tile with a thread
// whose share is tiny or holds a value from 2^10 up; elsewhere the second bound
// is the higher one.  (Left out: a result of exactly zero to which, in a row and
// a column that hold normal values, only products with values below 2^-134
// contribute.)  The bookkeeping costs 1-1.5 % (6272 x 6144 x 384: 182-187 us
// without it, 184-188 with it).  The second computation reads its operands from
// global memory value by value: there, 200 us become 385 with one NaN in A, 350
// with A of order 2^-80 and 950 with an infinity in every row; the library's
// float32 kernels stay at 265.
//
// Work split: a 256-thread workgroup computes a BM x BN tile, its 4 waves
// (2 x 2) a quarter each in 32x32x16 MFMA tiles.  Both operands are split
// into their three bf16 planes once per workgroup, on the way from global
// memory (held in registers two steps ahead) into double-buffered LDS; each
// fragment read from LDS then feeds six MFMAs.  A thread holds 8 consecutive
// k of one row, whichever way the operand lies in memory, so both layouts
// arrive in LDS the same way.  The 16-byte chunks of a row are permuted by
// bits of the row so that neither the writes nor the fragment reads of 16
// neighbouring lanes share a bank.
// Bound: with the MFMAs alone the loop runs at 230-240 TFLOP/s; the
// split's VALU work (11 instructions per pair of values), the LDS traffic and
// the global loads take the rest: 135-170 TFLOP/s on in_proj and out_proj of
// 6272-16384 rows, where the BLAS library's float32 kernels reach 95-137 (MFMA
// pipes busy 39-47 % of the cycles, the VALU 29-37 %, LDS 20-24 %; the waves
// wait to issue for half of theirs).
// Scheduling barriers and raised wave priority around the MFMAs were both
// slower (they keep the split's instructions from filling in between).
//
// Order of tiles: workgroups are dealt to the 8 XCDs in turn, so the tile
// index is remapped to give each XCD one contiguous range, walked in groups
// of 8 row tiles, whose operands stay in that XCD's L2.
#include <algorithm>

#include "gemm_kernels.h"
#include "scan_common.h"

namespace mvm {

namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kGroupM = 8;  // row tiles per group of the tile order
constexpr float kLarge = 0x1p10f;  // up to here the second bound below is the higher one

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// max(m, |a|, |b|), NaN if one of them is, in one instruction (from fmaxf or
// the maximum builtins the compiler makes up to three)
__device__ __forceinline__ float max3_abs(float m, float a, float b) {
  asm("v_maximum3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(a), "v"(b));
  return m;
}

// the three bf16 planes of 8 values
__device__ __forceinline__ void split8(const float (&v)[8], uint4 (&pl)[3]) {
  uint32_t w[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = v[2 * i], b = v[2 * i + 1];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      w[q][i] = pack_bf16(a, b);
      if (q < 2) {
        a -= __uint_as_float(w[q][i] << 16);
        b -= __uint_as_float(w[q][i] & 0xffff0000u);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) pl[q] = make_uint4(w[q][0], w[q][1], w[q][2], w[q][3]);
}

// One operand's share of a workgroup: ROWS rows (of A, or columns of B) by
// BK values of k per step.  KM: k is the contiguous index.
template <int ROWS, int BK, bool KM>
struct Operand {
  static constexpr int kChunks = BK / 8;
  static constexpr int kItems = ROWS * kChunks / kThreads;  // 8-value items per thread
  static_assert(kItems * kThreads == ROWS * kChunks, "items divide evenly");
  int row[kItems], chunk[kItems];
  uint32_t off[kItems];  // element offset of the item's first value from the step's base

  // rows past `nrows` read the last row: their results are not stored
  __device__ __forceinline__ void init(int tid, int nrows, int ld) {
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const int x = tid + kThreads * i;
      row[i] = KM ? x / kChunks : x % ROWS;
      chunk[i] = KM ? x % kChunks : x / ROWS;
      const int r = row[i] < nrows ? row[i] : nrows - 1;
      off[i] = KM ? r * ld + chunk[i] * 8 : chunk[i] * 8 * ld + r;
    }
  }
  __device__ __forceinline__ void load(float (&v)[kItems][8], const float* __restrict__ base, int ld) const {
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      if constexpr (KM) {
        const float4 x = *reinterpret_cast<const float4*>(base + off[i]);
        const float4 y = *reinterpret_cast<const float4*>(base + off[i] + 4);
        v[i][0] = x.x; v[i][1] = x.y; v[i][2] = x.z; v[i][3] = x.w;
        v[i][4] = y.x; v[i][5] = y.y; v[i][6] = y.z; v[i][7] = y.w;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = (base + e * ld)[off[i]];
      }
    }
  }
  // the last, partial step: `left` < BK values of k remain; the others are
  // read from the step's first value (in bounds) and replaced by zero
  __device__ __forceinline__ void load_tail(float (&v)[kItems][8], const float* __restrict__ base, int ld,
                                            int left) const {
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const uint32_t r = off[i] - (KM ? chunk[i] * 8 : chunk[i] * 8 * ld);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int p = chunk[i] * 8 + e;
        const float t = base[r + static_cast<uint32_t>(p < left ? (KM ? p : p * ld) : 0)];
        v[i][e] = p < left ? t : 0.f;
      }
    }
  }
  // LDS position of a row's chunk: at one chunk, 16 neighbouring rows cover
  // all the 16-byte columns of 256 bytes (as the reads are served) and 8 rows
  // those of 128 bytes (the writes)
  __device__ static __forceinline__ int swz(int r, int c) {
    return BK == 16 ? (c ^ (((r >> 2) ^ (r >> 3)) & 1)) * 8 : (c ^ (((r >> 1) ^ (r >> 3)) & 3)) * 8;
  }
  // (kItems is 1: the thread's values all belong to one row, whose largest
  // magnitude it keeps in `top`)
  static_assert(kItems == 1, "one row per thread");
  __device__ __forceinline__ void store(uint16_t (*lds)[ROWS][BK], const float (&v)[kItems][8], float& top) const {
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
#pragma unroll
      for (int e = 0; e < 8; e += 2) top = max3_abs(top, v[i][e], v[i][e + 1]);
      uint4 pl[3];
      split8(v[i], pl);
      const int o = swz(row[i], chunk[i]);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<uint4*>(&lds[q][row[i]][o]) = pl[q];
    }
  }
};

template <int BM, int BN, int BK, int OCC, bool AKM, bool BKM>
__global__ void __launch_bounds__(kThreads, OCC)
gemm_kernel(GemmGeom g, const float* __restrict__ A, const float* __restrict__ B,
            const float* add_src, float* C) {
  constexpr int MT = BM / 64, NT = BN / 64;  // 32 x 32 tiles of a wave
  __shared__ __attribute__((aligned(16))) uint16_t sA[2][3][BM][BK];
  __shared__ __attribute__((aligned(16))) uint16_t sB[2][3][BN][BK];
  __shared__ uint32_t sTop[BM + BN];  // largest magnitude of each row of A and column of B, as bits
  __shared__ __attribute__((aligned(16))) uint32_t sLook[kThreads / 64];  // a wave's reason to form them
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntm = (g.M + BM - 1) / BM, ntn = (g.N + BN - 1) / BN;
  int tm, tn;
  {
    const int nt = ntm * ntn, bid = blockIdx.x;
    const int per = nt / 8, rem = nt % 8, x = bid % 8;
    const int t = x * per + min(x, rem) + bid / 8;  // XCD x owns one contiguous range
    const int grp = t / (kGroupM * ntn), r = t % (kGroupM * ntn);
    const int gm = min(kGroupM, ntm - grp * kGroupM);
    tm = grp * kGroupM + r % gm;
    tn = r / gm;
  }
  const int m0 = tm * BM, n0 = tn * BN;
  const int sp = blockIdx.z % g.nsplit, q = blockIdx.z / g.nsplit;
  const int k0 = sp * g.kper, k1 = min(g.K, k0 + g.kper);
  const int len = k1 - k0;  // may be <= 0 in the last parts: a zero product
  const int full = len > 0 ? len / BK : 0;
  // step bases, advanced by one step at a time; B moves to its next segment
  // when it reaches the end of one
  const float* Ab = A + q * g.sa + (AKM ? static_cast<int64_t>(m0) * g.lda + k0
                                        : static_cast<int64_t>(k0) * g.lda + m0);
  const int seg0 = k0 / g.seg;
  int kin = k0 - seg0 * g.seg;
  const float* Bb = B + q * g.sb + seg0 * g.seg_stride +
                    (BKM ? static_cast<int64_t>(n0) * g.ldb + kin : static_cast<int64_t>(kin) * g.ldb + n0);
  const float* const A0 = Ab;
  const float* const B0 = Bb;
  const int64_t astep = AKM ? BK : static_cast<int64_t>(BK) * g.lda;
  const int64_t bstep = BKM ? BK : static_cast<int64_t>(BK) * g.ldb;
  const int64_t bfix = g.seg_stride - (BKM ? g.seg : static_cast<int64_t>(g.seg) * g.ldb);
  int pos = 0;
  Operand<BM, BK, AKM> oa;
  Operand<BN, BK, BKM> ob;
  oa.init(tid, g.M - m0, g.lda);
  ob.init(tid, g.N - n0, g.ldb);
  float pa[2][oa.kItems][8], pb[2][ob.kItems][8];
  // the next full step into register set r; past the last one it is read
  // again (never used), so the main loop has no branches
  auto prefetch = [&](int r) {
    oa.load(pa[r], Ab, g.lda);
    ob.load(pb[r], Bb, g.ldb);
    if (pos + 1 < full) {
      ++pos;
      Ab += astep;
      Bb += bstep;
      kin += BK;
      if (kin == g.seg) {
        kin = 0;
        Bb += bfix;
      }
    }
  };
  float topa = 0.f, topb = 0.f;
  auto stage = [&](int buf, int r) {
    oa.store(sA[buf], pa[r], topa);
    ob.store(sB[buf], pb[r], topb);
  };
  // before the last barrier: whether a thread's share of a row or column is
  // tiny throughout, or any value is large
  auto tiny = [](float t) { return t > 0.f && t < 0x1p-110f; };
  auto note = [&] {
    const bool look = __ballot(tiny(topa) || tiny(topb) || fmaxf(topa, topb) >= kLarge) != 0;
    if (lane == 0) sLook[wave] = look;
  };

  // hi * hi, and the five smaller products (added at the end)
  f32x16 acc[MT][NT] = {}, acs[MT][NT] = {};
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const int fr = lane & 31, fh = lane >> 5;
  auto compute = [&](int buf) {
#pragma unroll
    for (int h = 0; h < BK / 16; ++h) {
      const int fo = Operand<BM, BK, AKM>::swz(fr, 2 * h + fh);
      bf16x8 b[3][NT];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          b[p][j] = *reinterpret_cast<const bf16x8*>(&sB[buf][p][wn + j * 32 + fr][fo]);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        bf16x8 a[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) a[p] = *reinterpret_cast<const bf16x8*>(&sA[buf][p][wm + i * 32 + fr][fo]);
        constexpr int kPa[5] = {2, 0, 1, 1, 0}, kPb[5] = {0, 2, 1, 0, 1};
#pragma unroll
        for (int t = 0; t < 5; ++t)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acs[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kPa[t]], b[kPb[t]][j], acs[i][j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0][j], acc[i][j], 0, 0, 0);
      }
    }
  };
  if (full > 0) {
    prefetch(0);
    prefetch(1);
    stage(0, 0);
    int s = 0;
    for (; s + 1 < full; s += 2) {
      __syncthreads();
      prefetch(0);
      compute(0);
      stage(1, 1);
      __syncthreads();
      prefetch(1);
      compute(1);
      stage(0, 0);
    }
    if (s < full) {
      __syncthreads();
      compute(0);
    }
    note();
    __syncthreads();
  }
  if (len > full * BK) {  // (segments are whole steps: no segment ends in a partial one)
    const int64_t done = full;
    int64_t bo = done * bstep;
    if (g.seg < g.K) bo += ((k0 + full * BK) / g.seg - seg0) * bfix;
    oa.load_tail(pa[0], A0 + done * astep, g.lda, len - full * BK);
    ob.load_tail(pb[0], B0 + bo, g.ldb, len - full * BK);
    stage(0, 0);
    note();
    __syncthreads();
    compute(0);
  }

  // results the split cannot vouch for: again with the float32 instructions
  float most = 0.f;               // the largest magnitude (NaN: one of them is)
  uint32_t least = 0xffffffffu;  // the smallest that is not zero: 2 |bits| - 1
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      acc[i][j] += acs[i][j];
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float x = acc[i][j][r], y = acc[i][j][r + 1];
        most = max3_abs(most, x, y);
        least = min(least, min((__float_as_uint(x) << 1) - 1u, (__float_as_uint(y) << 1) - 1u));
      }
    }
  bool again = __ballot(!(most < __builtin_inff())) != 0;
  // (largest: of the operands' magnitudes)
  auto doubtful = [&](float largest) {
    const float bound = static_cast<float>(len) * fmaxf(largest * 0x1p-109f, 0x1p-99f);
    return __ballot(least < (__float_as_uint(bound) << 1) - 1u) != 0;
  };
  if (len > 0) {
    const uint4 look = *reinterpret_cast<const uint4*>(sLook);
    if ((look.x | look.y | look.z | look.w) == 0u) {
      again |= doubtful(kLarge);
    } else {  // (the same for all waves)
      for (int i = tid; i < BM + BN; i += kThreads) sTop[i] = 0u;
      __syncthreads();
      atomicMax(&sTop[oa.row[0]], __float_as_uint(topa));
      atomicMax(&sTop[BM + ob.row[0]], __float_as_uint(topb));
      __syncthreads();
      // the rows and columns of the wave's quarter of the tile
      const float ta = __uint_as_float(sTop[wm + lane % (BM / 2)]);
      const float tb = __uint_as_float(sTop[BM + wn + lane % (BN / 2)]);
      float m = fmaxf(ta, tb);
#pragma unroll
      for (int d = 32; d > 0; d /= 2) m = fmaxf(m, __shfl_xor(m, d));
      again |= __ballot(tiny(ta) || tiny(tb)) != 0 || doubtful(m);
    }
  }
  // (per wave: no barrier below)
  if (again) {
    int ra[MT], rb[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) ra[i] = min(wm + i * 32 + fr, g.M - 1 - m0);
#pragma unroll
    for (int j = 0; j < NT; ++j) rb[j] = min(wn + j * 32 + fr, g.N - 1 - n0);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = f32x16{};
    for (int p = 0; p < len; p += 2) {  // lane half fh holds k = p + fh
      const bool in = p + fh < len;
      const int64_t pk = in ? p + fh : 0;
      const int64_t bs = g.seg < g.K ? ((k0 + pk) / g.seg - seg0) * bfix : 0;
      float a[MT], b[NT];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const float v = A0[AKM ? static_cast<int64_t>(ra[i]) * g.lda + pk : pk * g.lda + ra[i]];
        a[i] = in ? v : 0.f;
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const float v = B0[bs + (BKM ? static_cast<int64_t>(rb[j]) * g.ldb + pk : pk * g.ldb + rb[j])];
        b[j] = in ? v : 0.f;
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  }

  // split: partial products side by side, (q, part, m, n)
  const bool split = g.nsplit > 1;
  float* Cq = split ? C + static_cast<int64_t>(blockIdx.z) * g.M * g.N : C + q * g.sc;
  const int64_t ldc = split ? g.N : g.ldc;
  const bool add = !split && add_src != nullptr;  // (may be C itself)
  const float* Sq = add_src + (add ? q * g.sc : 0);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int col = n0 + wn + j * 32 + fr;
      const int row0 = m0 + wm + i * 32 + 4 * fh;
      if (add) {
        // all 16 values in flight together, from in-bounds addresses (6272 x
        // 768 x 56 in 4 batches: 84 us with each load behind its own bounds
        // test, 63 like this)
        float old[16];
#pragma unroll
        for (int r = 0; r < 16; ++r)
          old[r] = Sq[min(row0 + 8 * (r / 4) + (r & 3), g.M - 1) * ldc + min(col, g.N - 1)];
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] += old[r];
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = row0 + 8 * (r / 4) + (r & 3);
        if (row < g.M && col < g.N) Cq[row * ldc + col] = acc[i][j][r];
      }
    }
}

// C = the sum of the partial products, left to right (+ add_src)
template <typename V>
__global__ void __launch_bounds__(kThreads)
gemm_reduce_kernel(GemmGeom g, const float* __restrict__ part, const float* add_src, float* C) {
  constexpr int W = sizeof(V) / sizeof(float);
  const int64_t mn = static_cast<int64_t>(g.M) * g.N;
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x) * W;
  if (i >= mn) return;
  const int64_t q = blockIdx.y;
  const float* p = part + q * g.nsplit * mn + i;
  const int64_t row = i / g.N;
  const int64_t at = q * g.sc + row * g.ldc + (i - row * g.N);
  float s[W];
  V v = *reinterpret_cast<const V*>(p);
#pragma unroll
  for (int e = 0; e < W; ++e) s[e] = reinterpret_cast<const float*>(&v)[e];
  for (int z = 1; z < g.nsplit; ++z) {
    v = *reinterpret_cast<const V*>(p + z * mn);
#pragma unroll
    for (int e = 0; e < W; ++e) s[e] += reinterpret_cast<const float*>(&v)[e];
  }
  if (add_src != nullptr) {
    v = *reinterpret_cast<const V*>(add_src + at);
#pragma unroll
    for (int e = 0; e < W; ++e) s[e] += reinterpret_cast<const float*>(&v)[e];
  }
#pragma unroll
  for (int e = 0; e < W; ++e) reinterpret_cast<float*>(&v)[e] = s[e];
  *reinterpret_cast<V*>(C + at) = v;
}

// Tile shapes: 2 workgroups on a CU (by VGPRs), 3 (by LDS).
struct TileCfg {
  int bm, bn, bk, occ;
  // microseconds per step (bk of k) of a workgroup that has a CU to itself,
  // and per step and workgroup of a CU that runs several (measured on the
  // shapes of gemm_plan's comment)
  float alone, shared;
};
constexpr TileCfg kCfg[2] = {{128, 128, 16, 2, 0.80f, 0.68f}, {64, 64, 32, 3, 0.50f, 0.46f}};
constexpr int kCUs = 256;
constexpr float kBytesPerUs = 4.5e6f;  // HBM, streaming
constexpr int kMaxSplit = 24;

template <int CFG, bool AKM, bool BKM>
void launch_cfg(const GemmGeom& g, const float* A, const float* B, const float* add, float* C, hipStream_t s) {
  constexpr TileCfg c = kCfg[CFG];
  const unsigned nt = static_cast<unsigned>((g.M + c.bm - 1) / c.bm) * static_cast<unsigned>((g.N + c.bn - 1) / c.bn);
  hipLaunchKernelGGL((gemm_kernel<c.bm, c.bn, c.bk, c.occ, AKM, BKM>),
                     dim3(nt, 1, static_cast<unsigned>(g.batch * g.nsplit)), dim3(kThreads), 0, s, g, A, B, add, C);
}
template <int CFG>
void launch_layout(const GemmGeom& g, const float* A, const float* B, const float* add, float* C, hipStream_t s) {
  if (g.a_km)
    g.b_km ? launch_cfg<CFG, true, true>(g, A, B, add, C, s) : launch_cfg<CFG, true, false>(g, A, B, add, C, s);
  else
    g.b_km ? launch_cfg<CFG, false, true>(g, A, B, add, C, s) : launch_cfg<CFG, false, false>(g, A, B, add, C, s);
}

}  // namespace

// The tile shape and split with the least estimated time: the steps of the
// busiest CU, writing C, and with a split the partial products (written and
// read) and the second launch.  Measured (estimated) us on MI355X, the BLAS
// library's time last: 6272 x 6144 x 384: 128-tiles unsplit 207 (197), 64-tiles
// 241, library 248-290; 6272 x 384 x 6144: 128-tiles in 3 parts 187 (191), in 4
// (76 workgroups past a full round) 222 (233), unsplit 310, library 262; 196 x
// 1536 x 384: 64-tiles unsplit 10.0 (6.3 + launch), 128-tiles 22.8, library
// 19.6; 196 x 384 x 768: 64-tiles in 4-8 parts 10.3, unsplit 15.9, library 19.2.
void gemm_plan(GemmGeom& g) {
  const int want = g.nsplit;  // > 0: the caller's split
  if (g.K < 32) {  // less than a step of the small tile, which loads it value by value
    g.cfg = 1;
    g.nsplit = want > 0 ? want : 1;
    g.kper = 32;
    return;
  }
  const int64_t mn4 = int64_t{4} * g.batch * g.M * g.N;
  const float write = static_cast<float>(mn4) / kBytesPerUs;
  float best = __builtin_inff();
  for (int c = 0; c < 2; ++c) {
    const TileCfg& t = kCfg[c];
    if (g.seg < g.K && g.seg % t.bk != 0) continue;  // no step straddles two segments
    const int64_t tiles = int64_t{g.batch} * ((g.M + t.bm - 1) / t.bm) * ((g.N + t.bn - 1) / t.bn);
    const int64_t slots = int64_t{kCUs} * t.occ;
    for (int ns = want > 0 ? want : 1; ns <= (want > 0 ? want : kMaxSplit); ++ns) {
      // (at least 64 values of k per part, partial products of at most 1 GiB,
      // and no further split of what fills the chip four times)
      if (want == 0 && ns > 1 &&
          (g.K < 64 * ns || mn4 * ns > (int64_t{1} << 30) || int64_t{g.batch} * ns > 65535 ||
           tiles * (ns - 1) > 4 * slots)) break;
      const int kper = static_cast<int>((int64_t{g.K} + ns - 1) / ns + t.bk - 1) / t.bk * t.bk;
      // whole rounds of t.occ workgroups per CU, then the rest
      const int64_t n = tiles * ns, rounds = n / slots, rest = (n % slots + kCUs - 1) / kCUs;
      float us = static_cast<float>(kper / t.bk) *
                     (t.shared * static_cast<float>(rounds * t.occ + (rest == 1 ? 0 : rest)) +
                      (rest == 1 ? t.alone : 0.f)) + write;
      if (ns > 1) us += 3.f + 3.f * static_cast<float>(ns) * write;
      if (us < best) {
        best = us;
        g.cfg = c;
        g.nsplit = ns;
        g.kper = kper;
      }
    }
  }
}

int64_t gemm_partial_floats(const GemmGeom& g) {
  return g.nsplit > 1 ? static_cast<int64_t>(g.batch) * g.nsplit * g.M * g.N : 0;
}

hipError_t launch_gemm(const GemmGeom& g, const float* A, const float* B, const float* add, float* C,
                       float* part, hipStream_t s) {
  float* out = g.nsplit > 1 ? part : C;
  switch (g.cfg) {
    case 0: launch_layout<0>(g, A, B, add, out, s); break;
    default: launch_layout<1>(g, A, B, add, out, s); break;
  }
  if (g.nsplit > 1) {
    const bool vec = g.N % 4 == 0 && g.ldc % 4 == 0 && g.sc % 4 == 0 &&
                     ((reinterpret_cast<uintptr_t>(C) | reinterpret_cast<uintptr_t>(add)) & 15u) == 0;
    const int64_t n = static_cast<int64_t>(g.M) * g.N / (vec ? 4 : 1);
    const dim3 grid(static_cast<unsigned>((n + kThreads - 1) / kThreads), static_cast<unsigned>(g.batch));
    if (vec)
      hipLaunchKernelGGL((gemm_reduce_kernel<float4>), grid, dim3(kThreads), 0, s, g, part, add, C);
    else
      hipLaunchKernelGGL((gemm_reduce_kernel<float>), grid, dim3(kThreads), 0, s, g, part, add, C);
  }
  return hipGetLastError();
}

}  // namespace mvm
