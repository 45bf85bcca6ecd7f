// f32 projection GEMM on bf16 matrix products (kernel; launched from gemm.hip).
//
// An f32 value is the exact sum of three bf16 values (8 + 8 + 8 significant
// bits, the exponent range of f32), a bf16 product is exact in f32, and
// v_mfma_f32_16x16x32_bf16 accumulates in f32 at 16 times the rate of the f32
// MFMA.  Rounded to nearest, mid is at most 2^-8 of x and lo 2^-17, so of the
// nine products in x w the three dropped ones (mid lo, lo mid, lo lo) reach
// 2^-24 of the term at worst, as much as one f32 rounding, and 2^-26.5 in the
// mean square over all significands.  The six others are formed.  Each
// 32-deep step of K sums its products from zero, small ones first; steps are
// added up in groups of four and the groups in a running sum, so the sum's
// own magnitude is rounded once per 128 columns (the f32 MFMA kernel: once per
// 32, after 16 roundings inside).  Against 64 bits, 2-norm, N(0,1) x N(0,0.02):
// K = 64 0.58e-7 (f32 MFMA kernel 1.31e-7), K = 320 0.67e-7 (1.20e-7), K =
// 2048 1.07e-7 (1.79e-7), K = 6144 1.68e-7 (2.74e-7); without the groups 1.60
// and 2.69e-7 at the last two.  With the significands that drop most in every
// operand, both signs: K = 4 0.60e-7 (0.41e-7), K = 32 0.59e-7 (0.71e-7), K =
// 2048 1.60e-7 (1.64e-7).
// Outputs that the split does not hold (not finite, or where values below
// 2^-100 matter) are formed on the f32 MFMA instead, at the end, their 16 x 16
// blocks dealt to all waves.  At 2048 x 8192 x 2048 (f32 MFMA kernel 654 us,
// here 367): one such weight 382, one such value in every x row 426, one
// infinity 490, a whole x row of such values 556; where every output is one,
// 2.1 ms.
//
// The tile's x and weight rows pass through registers (loaded D stages
// ahead), where they are split, into two LDS buffers of three planes each.
// What bounds it: at 2048 x 8192 x 2048 (655 -> 363 us) the products run at
// 1.14 PFLOP/s in bf16, where a large bf16 product of the vendor library
// reaches 1.29 on this card (the clock drops under random operands); smaller
// launches by the walk of one work-group along K.  Four tile shapes (launch
// rule in gemm.hip); all sum in one order, so a row's result does not depend
// on the shape.  On 256 x 128 and 128 x 128 tiles (FAST) the splitting of the
// next stage is interleaved with the products of this one, three vector
// instructions per product: one after the other leaves the matrix cores idle
// while a wave splits (374 -> 355 us before the groups were added; letting
// half of the waves multiply first while the others split took 414,
// single-buffered tiles with two to four work-groups per CU 377 to 420).
// 256 x 128 as 2 x 4 waves of 128 x 32: as 4 x 2 of 64 x 64 the second set of
// sums spills (426 us).
#pragma once
#include "bf16_split.hpp"
#include "common.hpp"
#include "gemm.hpp"

namespace clef {
namespace {

typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));

// Stores four consecutive columns c .. c + 3 of row r: as a vector (`whole`), or
// one by one those within N and not in the mask `skip`.
__device__ __forceinline__ void store_row4(const GemmParams& p, int r, int c, const float4_t& o, bool whole,
                                           uint32_t skip) {
  const int64_t off = (int64_t)r * p.ldy + c;
  if (p.dtype_out == 1) {
    const half4 h = {static_cast<half_t>(o[0]), static_cast<half_t>(o[1]), static_cast<half_t>(o[2]),
                     static_cast<half_t>(o[3])};
    half_t* dst = static_cast<half_t*>(p.y) + off;
    if (whole) {
      *reinterpret_cast<half4*>(dst) = h;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < p.N && !(skip >> e & 1)) dst[e] = h[e];
    }
  } else {
    float* dst = static_cast<float*>(p.y) + off;
    if (whole) {
      *reinterpret_cast<float4_t*>(dst) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < p.N && !(skip >> e & 1)) dst[e] = o[e];
    }
  }
}

template <int BM, int BN, int VM, int VN, int U, int D, bool FAST, int EPI>
__global__ __launch_bounds__(512, 2) void gemm_f32_split(GemmParams p) {
  constexpr int NT = 512;
  constexpr int WM = BM / VM, WN = BN / VN, TM = WM / 16, TN = WN / 16;
  constexpr int ROWS = BM + BN, CPS = ROWS * 4;  // rows and 8-element chunks of a 32-deep sub-stage
  constexpr int CH = U * CPS / NT;               // chunks per thread per stage
  constexpr int kPlane = ROWS * 32;              // bf16 of one plane of a sub-stage
  constexpr int kSub = 3 * kPlane, kBuf = U * kSub;
  static_assert(VM * VN <= 8 && TM * 16 * VM == BM && TN * 16 * VN == BN, "wave layout");
  static_assert(U * CPS % NT == 0 && (BM * 4) % 64 == 0, "whole chunks per thread, one operand per wave");
  static_assert(EPI != 2 || TN % 2 == 0, "a SwiGLU wave holds gate and up columns of the same outputs");
  static_assert(D == 1 || D == 2, "stages in flight in registers");
  static_assert(!FAST || (U == 1 && D == 1), "the interleaved loop is one sub-stage deep");
  static_assert(2 * kBuf * 2 + 16 <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(16))) __bf16 smem[2 * kBuf];
  // of [x rows | weight rows], formed only if the tile met a value below 2^-100:
  // K 2^-97 if the row holds one, else 0; its largest magnitude
  __shared__ float row_tiny[ROWS], row_max[ROWS];
  __shared__ int any_tiny, any_odd;  // a value below 2^-100, or that or an output that is not finite

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / VN, wn = wave % VN;
  constexpr int ON = EPI == 2 ? BN / 2 : BN;  // output columns of a tile
  // XCD-compact tile order in groups of 4 row tiles, as the f16 kernels'
  const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + ON - 1) / ON;
  const int ntiles = gridDim.x, xcd = blockIdx.x & 7, per = ntiles >> 3, rem = ntiles & 7;
  const int t = xcd * per + min(xcd, rem) + (blockIdx.x >> 3);
  const int gsize = 4 * tiles_n, first_m = (t / gsize) * 4, gm = min(4, tiles_m - first_m);
  const int m0 = (first_m + (t % gsize) % gm) * BM, n0 = ((t % gsize) / gm) * ON;

  const float* X = static_cast<const float*>(p.x);
  const float* W = static_cast<const float*>(p.w);
  const float* W2 = static_cast<const float*>(p.w2);
  // Chunk i of a thread: sub-stage sub[i], row r of [x rows | weight rows],
  // columns 8 (tid % 4) .. + 7.  A SwiGLU tile's 16-row weight blocks
  // alternate gate and up rows of the same 16 outputs.
  const int c4 = tid & 3;
  auto chunk = [&](int i, int& sub, int& row) {
    const int ci = i * NT + wave * 64;  // uniform part
    sub = ci / CPS;
    row = (ci % CPS) / 4 + (lane >> 2);
  };
  // each through a buffer resource over the tile's rows of its operand
  uint32_t voff[CH];  // byte offset of the chunk at stage 0
  __amdgpu_buffer_rsrc_t rs[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    int sub, row;
    chunk(i, sub, row);
    const int first = ((i * NT + wave * 64) % CPS) / 4;  // the wave's first row names the operand
    const bool is_x = first < BM;
    const int64_t ld = is_x ? p.ldx : p.ldw;
    const int base = is_x ? m0 : n0, rows = is_x ? p.M - m0 : p.N - n0;
    const float* op = is_x ? X : EPI == 2 && ((first - BM) & 16) ? W2 : W;
    const int rb = row - BM;
    const int r = min(is_x ? row : EPI == 2 ? (rb >> 5) * 16 + (rb & 15) : rb, rows - 1);
    rs[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(op + base * ld), 0,
                                              static_cast<int>(min(rows, BM + BN) * (int)ld * 4), 0x00020000);
    voff[i] = (uint32_t)(r * (int)ld + sub * 32 + 8 * c4) * 4u;
  }
  const int nsub = (p.K + 31) / 32, nst = (nsub + U - 1) / U;
  float4_t ld[D][CH][2];
  auto load = [&](int st, int d) {
    const bool whole = (st + 1) * U * 32 <= p.K;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      int sub, row;
      chunk(i, sub, row);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t vo = voff[i] + 16 * h;
        const uint32_t so = (uint32_t)st * (U * 128);
        if (!whole) {  // past K: the row's last four elements, zeroed by split()
          const int k = st * U * 32 + sub * 32 + 8 * c4 + 4 * h;
          vo -= k + 4 > p.K ? (uint32_t)(k - (p.K - 4)) * 4u : 0u;
        }
        const uint4_t v = __builtin_amdgcn_raw_buffer_load_b128(rs[i], whole ? vo : vo + so, whole ? so : 0u, 0);
        ld[d][i][h] = __builtin_bit_cast(float4_t, v);
      }
    }
  };
  // LDS: per buffer, sub-stage and plane [x rows | weight rows][32] bf16, the
  // 16-byte chunk c of row r at c ^ ((r >> 2) & 3) (16 consecutive rows of
  // one chunk, and 4 rows of all four, cover the 64 banks once)
  uint32_t smallest = 0xffffffffu;  // of |x| > 0, as 2 * bits - 1
  constexpr uint32_t kTiny = (27u << 24) - 1u;  // of 2^-100
  auto split = [&](int st, int d) {
    const bool whole = (st + 1) * U * 32 <= p.K;
    __bf16* const buf = smem + (st & 1) * kBuf;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      int sub, row;
      chunk(i, sub, row);
      float4_t a = ld[d][i][0], b = ld[d][i][1];
      if (!whole) {
        const int k = st * U * 32 + sub * 32 + 8 * c4;
        if (k >= p.K) a = float4_t{0.f, 0.f, 0.f, 0.f};
        if (k + 4 >= p.K) b = float4_t{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        smallest = min(smallest, 2u * __float_as_uint(a[e]) - 1u);
        smallest = min(smallest, 2u * __float_as_uint(b[e]) - 1u);
      }
      bf16x8 hi, mid, lo;
      split8(a, b, hi, mid, lo);
      __bf16* const dst = buf + sub * kSub + row * 32 + ((c4 ^ ((row >> 2) & 3)) << 3);
      *reinterpret_cast<bf16x8*>(dst) = hi;
      *reinterpret_cast<bf16x8*>(dst + kPlane) = mid;
      *reinterpret_cast<bf16x8*>(dst + 2 * kPlane) = lo;
    }
  };

  // 16 x 16 x 32 products, weights as the A operand (a lane's four results
  // are consecutive columns of one row).  Six products per block: all but
  // mid*lo, lo*mid and lo*lo; the small ones first.
  // Each 32-deep step starts from zero, so the small products are summed
  // among themselves.
  const bool active = wave < VM * VN;
  float4_t sum[TM][TN], tot[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) sum[i][j] = tot[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  const int r16 = lane & 15, c16 = lane >> 4;
  const int goff = r16 * 32 + ((c16 ^ ((r16 >> 2) & 3)) << 3);
  auto product = [&](const __bf16* sub) {
    const __bf16* ab = sub + wm * WM * 32 + goff;
    const __bf16* bb = sub + (BM + wn * WN) * 32 + goff;
    bf16x8 bf[TN][3];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int s = 0; s < 3; ++s) bf[j][s] = *reinterpret_cast<const bf16x8*>(bb + s * kPlane + j * 512);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      bf16x8 af[3];
#pragma unroll
      for (int s = 0; s < 3; ++s) af[s] = *reinterpret_cast<const bf16x8*>(ab + s * kPlane + i * 512);
      constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
      float4_t acc[TN];
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              bf[j][pb[q]], af[pa[q]], q == 0 ? float4_t{0.f, 0.f, 0.f, 0.f} : acc[j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < TN; ++j) sum[i][j] += acc[j];
    }
  };
  constexpr int G = 4;  // steps added up before they join the running sum
  auto fold = [&] {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        tot[i][j] += sum[i][j];
        sum[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
      }
  };
  auto compute = [&](int st) {
    const __bf16* const buf = smem + (st & 1) * kBuf;
    if (!active) return;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      product(buf + u * kSub);  // sub-stages past K are zeros
      if ((st * U + u) % G == G - 1) fold();
    }
  };

  if (tid == 0) any_tiny = any_odd = 0;
  load(0, 0);
  if (D == 2 && nst > 1) load(1, 1);
  split(0, 0);
  if (nst > D) load(D, 0);
  lds_barrier();
  // stage st is multiplied from one buffer while stage st + 1 (in registers
  // since D stages) is split into the other
  auto step = [&](int st, int d) {
    if (st + 1 < nst) {
      split(st + 1, d);
      if (st + 1 + D < nst) load(st + 1 + D, d);
    }
    compute(st);
    lds_barrier();
  };
  int st = 0;
  if constexpr (FAST) {
    // whole stages with two more after them: one basic block, so that the
    // splitting of stage st + 1 runs under the products of stage st
    const int nfast = min(nst - 2, p.K / 32 - 2);
    auto fast = [&](int s, __bf16* cur, __bf16* oth) {
      const __bf16* ab = cur + wm * WM * 32 + goff;
      const __bf16* bb = cur + (BM + wn * WN) * 32 + goff;
      bf16x8 bf[TN][3];
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 3; ++q) bf[j][q] = *reinterpret_cast<const bf16x8*>(bb + q * kPlane + j * 512);
      bf16x8 pl[CH][3];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        bf16x8 af[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) af[q] = *reinterpret_cast<const bf16x8*>(ab + q * kPlane + i * 512);
        constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
        float4_t acc[TN];
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                bf[j][pb[q]], af[pa[q]], q == 0 ? float4_t{0.f, 0.f, 0.f, 0.f} : acc[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < TN; ++j) sum[i][j] += acc[j];
      }
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        int sub, row;
        chunk(i, sub, row);
        const float4_t a = ld[0][i][0], b = ld[0][i][1];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          smallest = min(smallest, 2u * __float_as_uint(a[e]) - 1u);
          smallest = min(smallest, 2u * __float_as_uint(b[e]) - 1u);
        }
        split8(a, b, pl[i][0], pl[i][1], pl[i][2]);
        __bf16* const dst = oth + sub * kSub + row * 32 + ((c4 ^ ((row >> 2) & 3)) << 3);
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8*>(dst + q * kPlane) = pl[i][q];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          ld[0][i][h] = __builtin_bit_cast(
              float4_t, __builtin_amdgcn_raw_buffer_load_b128(rs[i], voff[i] + 16 * h, (uint32_t)(s + 2) * 128u, 0));
        }
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 3 * TN + 3, 0);
#pragma unroll
      for (int q = 0; q < 6 * TM * TN; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        if (q % (2 * TN) == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if (q % 10 == 9) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      lds_barrier();
    };
    for (; st + 1 < nfast; st += 2) {
      fast(st, smem, smem + kBuf);
      fast(st + 1, smem + kBuf, smem);
      if ((st + 1) % G == G - 1) fold();
    }
  }
  if constexpr (D == 1) {
    for (; st < nst; ++st) step(st, 0);
  } else {
    for (; st < nst; st += 2) {
      step(st, 1);
      if (st + 1 < nst) step(st + 1, 0);
    }
  }
  if (active) fold();

  // Values the split does not hold.  Below 2^-100 the low parts leave bf16's
  // range: the term errs by up to 2^-124 of the other factor.  Infinities, NaN
  // and values that round to infinity make every output they meet NaN.  An
  // output that is not finite, or smaller than K 2^-97 of the largest factor
  // that such a small value of its x row or weight row may meet (larger ones
  // err by less than 2^-27), is formed again on f32 products.  That follows
  // from the row, the column and the result alone, so a row's bits do not
  // depend on what shares its tile.
  const bool small = smallest < kTiny;
  float4_t z = {0.f, 0.f, 0.f, 0.f};  // NaN once something is not finite
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) z[e] = fmaf(tot[i][j][e], 0.0f, z[e]);
  if (small) any_tiny = 1;
  if (small || z[0] + z[1] + z[2] + z[3] != 0.0f) any_odd = 1;
  lds_barrier();

  const int esz = (EPI == 1 || p.dtype_out != 1) ? 4 : 2;
  const bool yvec = ((reinterpret_cast<uintptr_t>(p.y) | (uintptr_t)(p.ldy * esz)) & (4 * esz - 1)) == 0;
  constexpr int TO = EPI == 2 ? TN / 2 : TN;
  constexpr int NBLK = TM * TO;  // 16 x 16 output blocks of a wave
  static_assert(NBLK <= 16, "a lane's outputs fit a 64-bit mask");
  // block (i, j) of wave w: the lane's row and its first column
  auto orow = [&](int w, int i) { return m0 + w / VN * WM + 16 * i + r16; };
  auto ocol = [&](int w, int j) { return n0 + w % VN * (EPI == 2 ? WN / 2 : WN) + 16 * j + 4 * c16; };
  // the lane's four outputs from column c of row r, without those in `skip`
  auto finish = [&](int r, int c, float4_t v, const float4_t& up, uint32_t skip) {
    if (r >= p.M) return;
    const bool whole = yvec && c + 3 < p.N && skip == 0;
    if constexpr (EPI == 2) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (p.dtype_out == 1) {
          const float gh = static_cast<float>(to_f16(v[e]));
          const float sh = static_cast<float>(to_f16(silu_hw(gh)));
          v[e] = sh * static_cast<float>(to_f16(up[e]));
        } else {
          v[e] = (v[e] / (1.0f + expf(-v[e]))) * up[e];
        }
      }
    }
    if constexpr (EPI == 1) {
      float* dst = static_cast<float*>(p.y) + (int64_t)r * p.ldy + c;
      auto rd = [&](float x) { return p.dtype_out == 1 ? static_cast<float>(static_cast<half_t>(x)) : x; };
      if (whole) {
        float4_t h = *reinterpret_cast<const float4_t*>(dst);
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] += rd(v[e]);
        *reinterpret_cast<float4_t*>(dst) = h;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < p.N && !(skip >> e & 1)) dst[e] += rd(v[e]);
      }
    } else {
      store_row4(p, r, c, v, whole, skip);
    }
  };
  if (__builtin_expect(any_odd == 0, 1)) {
    if (active)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TO; ++j)
          finish(orow(wave, i), ocol(wave, j), tot[i][EPI == 2 ? 2 * j : j], tot[i][EPI == 2 ? 2 * j + 1 : j], 0);
    return;
  }
  const bool tiny = __builtin_amdgcn_readfirstlane(any_tiny) != 0;
  if (tiny) {
    // the rows once more, four of them a wave at a time
    const int rl = lane >> 4, cl = 4 * (lane & 15);
    for (int row = 4 * wave + rl; row < ROWS; row += 32) {
      const bool is_x = row < BM;
      const int rb = row - BM;
      const float* op = is_x ? X : EPI == 2 && (rb & 16) ? W2 : W;
      const int r = is_x ? min(m0 + row, p.M - 1) : min(n0 + (EPI == 2 ? (rb >> 5) * 16 + (rb & 15) : rb), p.N - 1);
      const float* src = op + (int64_t)r * (is_x ? p.ldx : p.ldw);
      float m = 0.0f;
      uint32_t least = 0xffffffffu;
      for (int k0 = 0; k0 < p.K; k0 += 512) {
        float4_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const float4_t*>(src + min(k0 + 64 * u + cl, p.K - 4));
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            m = fmaxf(m, fabsf(v[u][e]));
            least = min(least, 2u * __float_as_uint(v[u][e]) - 1u);
          }
      }
      m = lane_max<16>(m);
      const float t = lane_max<16>(least < kTiny ? static_cast<float>(p.K) * 0x1p-97f : 0.0f);
      if (cl == 0) row_max[row] = m, row_tiny[row] = t;
    }
    lds_barrier();
  }
  uint64_t redo = 0;  // bit 4 (i TO + j) + e
  if (active) {
    const int xr = wm * WM + r16, wr = BM + wn * WN + 4 * c16;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TO; ++j) {
        const int j0 = EPI == 2 ? 2 * j : j, j1 = EPI == 2 ? 2 * j + 1 : j;
        uint32_t again = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          auto is = [&](int jj) {
            const float a = fabsf(tot[i][jj][e]);
            if (!tiny) return !(a < __builtin_inff());
            const int x = xr + 16 * i, w = wr + 16 * jj + e;
            return !(a < __builtin_inff()) || a < row_tiny[x] * row_max[w] + row_tiny[w] * row_max[x];
          };
          again |= (is(j0) || (EPI == 2 && is(j1)) ? 1u : 0u) << e;
        }
        redo |= (uint64_t)again << (4 * (i * TO + j));
        finish(orow(wave, i), ocol(wave, j), tot[i][j0], tot[i][j1], again);
      }
  }
  uint64_t* const masks = reinterpret_cast<uint64_t*>(smem);  // (no longer read) by wave and lane
  masks[tid] = redo;
  lds_barrier();

  // one 16 x 16 block on v_mfma_f32_16x16x4_f32, operands straight from memory
  // (64 columns of K in registers while the 64 before are multiplied)
  auto exact = [&](const float* w, int xr, int wr) __attribute__((always_inline)) {
    float4_t s = {0.f, 0.f, 0.f, 0.f};
    const float* xp = X + (int64_t)min(xr, p.M - 1) * p.ldx + 4 * c16;
    const float* wp = w + (int64_t)min(wr, p.N - 1) * p.ldw + 4 * c16;
    float4_t xv[2][4], wv[2][4];
    auto fetch = [&](int k0, float4_t* xd, float4_t* wd) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {  // past K: the row's first elements, zeroed by the products
        const int k = k0 + 16 * u + 4 * c16 < p.K ? k0 + 16 * u : -4 * c16;
        xd[u] = *reinterpret_cast<const float4_t*>(xp + k);
        wd[u] = *reinterpret_cast<const float4_t*>(wp + k);
      }
    };
    auto multiply = [&](int k0, float4_t* xd, float4_t* wd) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (k0 + 32 * h >= p.K) break;
        float4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 2 * h; u < 2 * h + 2; ++u) {
          const bool in = k0 + 16 * u + 4 * c16 < p.K;
          const float4_t z = {0.f, 0.f, 0.f, 0.f};
          Mma<float>::mma(a, in ? wd[u] : z, in ? xd[u] : z);
        }
        s += a;
      }
    };
    fetch(0, xv[0], wv[0]);
    for (int k0 = 0; k0 < p.K; k0 += 128) {
      fetch(k0 + 64, xv[1], wv[1]);
      multiply(k0, xv[0], wv[0]);
      fetch(k0 + 128, xv[0], wv[0]);
      multiply(k0 + 64, xv[1], wv[1]);
    }
    return s;
  };
  // the blocks dealt to all eight waves
  for (int b = wave; b < VM * VN * NBLK; b += 8) {
    const int w = b / NBLK, blk = b % NBLK;
    const uint32_t odd = (uint32_t)(masks[w * 64 + lane] >> (4 * blk)) & 15u;
    if (__ballot(odd != 0) == 0) continue;
    const int r = orow(w, blk / TO), c = ocol(w, blk % TO), wr = c - 4 * c16 + r16;
    const float4_t v = exact(W, r, wr);
    const float4_t up = EPI == 2 ? exact(W2, r, wr) : v;
    if (odd) finish(r, c, v, up, odd ^ 15u);
  }
}

}  // namespace
}  // namespace clef
