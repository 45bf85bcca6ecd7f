// f16 projection GEMM on small tiles, for launches whose 128- or 256-row tiles
// would leave most of the CUs idle (short requests, 2048-wide outputs).
//
// What bounds it: such a launch has little to multiply; its time is the
// stream of weights from HBM and the latency of one work-group's walk along
// K.  So the tile is made small enough that a round fills the CUs, and the
// LDS holds as much of K in flight as it can: a ring of S slots, each U
// 64-deep sub-stages of the tile's x and weight rows, filled by DMA S - 1
// stages ahead by all eight waves, with one barrier per stage.  (The general
// kernel's 128 x 128 tiles, register-staged one 64-deep stage ahead, took 108
// us for 33 x 2048 x 6144 on 16 work-groups; 32 x 16 tiles take 12.6.)  K is
// not split: every output is summed by one wave over k in the order of the
// larger kernels, on the same 16 x 16 x 32 products, so the results are
// theirs bit for bit and a row does not depend on how many rows share the
// call.
//
// A sub-stage is [BM + BN][64] halves: x rows, then weight rows, 128-byte
// rows with gemm_f16_dma's chunk swizzle.  VM x VN waves multiply (the rest
// of the eight only move data).  Tiles and rings, time of one round at
// K = 6144 (weights from HBM): 32 x 16 U 4 S 3: 12.6 us, 64 x 32 U 2 S 3: 22
// (both 72 KiB, two work-groups per CU), 64 x 64 U 2 S 5: 30, 128 x 64 U 2 S 3:
// 45.  Deeper rings at one work-group per CU (S 6, S 9) timed 0-8% slower.
#pragma once
#include "common.hpp"
#include "gemm.hpp"
#include "gemm_dma.hpp"

namespace clef {
namespace {

template <int BM, int BN, int VM, int VN, int U, int S, int EPI>
__global__ __launch_bounds__(512, (U * S * (BM + BN) * 128 <= 80 * 1024 ? 4 : 2)) void gemm_f16_ring(GemmParams p) {
  constexpr int kWaves = 8;
  constexpr int WM = BM / VM, WN = BN / VN, TM = WM / 16, TN = WN / 16;
  constexpr int RB = (BM + BN) / 8;        // 8-row DMA blocks of one 64-deep sub-stage
  constexpr int ND = U * RB / kWaves;      // DMA instructions per wave per stage
  constexpr int kSub = (BM + BN) * 64;     // halves of a sub-stage: A rows, then B rows
  constexpr int kSlot = U * kSub;
  static_assert(VM * VN <= kWaves && TM * 16 * VM == BM && TN * 16 * VN == BN, "wave layout");
  static_assert(U * RB % kWaves == 0 && ND * (S - 1) < 64, "whole DMA instructions per wave, vmcnt is 6 bits");
  static_assert(EPI != 2 || TN % 2 == 0, "a SwiGLU wave holds gate and up columns of the same outputs");
  static_assert(S * kSlot * 2 <= 160 * 1024, "LDS");
  typedef half8 frag;
  __shared__ __attribute__((aligned(1024))) half_t smem[S * kSlot];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / VN, wn = wave % VN;
  // tiles in XCD-compact order, row tiles of one column first: the work-groups
  // that share weight rows run side by side on one XCD
  constexpr int ON = EPI == 2 ? BN / 2 : BN;  // output columns of a tile
  const int tiles_m = (p.M + BM - 1) / BM;
  const int ntiles = gridDim.x, xcd = blockIdx.x & 7, per = ntiles >> 3, rem = ntiles & 7;
  const int t = xcd * per + min(xcd, rem) + (blockIdx.x >> 3);
  const int m0 = (t % tiles_m) * BM, n0 = (t / tiles_m) * ON;

  const __amdgpu_buffer_rsrc_t rA = operand_rsrc(static_cast<const half_t*>(p.x), p.M, p.ldx);
  const __amdgpu_buffer_rsrc_t rB = operand_rsrc(static_cast<const half_t*>(p.w), p.N, p.ldw);
  const __amdgpu_buffer_rsrc_t rU = EPI == 2 ? operand_rsrc(static_cast<const half_t*>(p.w2), p.N, p.ldw) : rB;

  // DMA instruction q of this wave: block b = wave * ND + q of the stage's
  // U * RB, i.e. 8 rows of one operand in sub-stage b / RB.  A SwiGLU tile's
  // 16-row weight blocks alternate gate and up rows of the same 16 outputs.
  uint32_t voff[ND];
#pragma unroll
  for (int q = 0; q < ND; ++q) {
    const int r8 = (wave * ND + q) % RB;
    const int lrow = lane >> 3;
    if (r8 < BM / 8) {
      const int col = ((lane & 7) ^ ((4 * r8 + (lane >> 4)) & 7)) << 3;
      voff[q] = (uint32_t)(min(m0 + 8 * r8 + lrow, p.M - 1) * (int)p.ldx + col) * 2u;
    } else {
      const int rb = r8 - BM / 8;
      const int col = ((lane & 7) ^ ((4 * rb + (lane >> 4)) & 7)) << 3;
      const int row = EPI == 2 ? n0 + (rb >> 2) * 16 + (rb & 1) * 8 + lrow : n0 + 8 * rb + lrow;
      voff[q] = (uint32_t)(min(row, p.N - 1) * (int)p.ldw + col) * 2u;
    }
  }
  const int nk = p.K >> 6, nst = (nk + U - 1) / U;
  auto issue = [&](int st) {  // stage st into its slot; past K the last sub-stage again (never read)
    half_t* const slot = smem + (st % S) * kSlot;
#pragma unroll
    for (int q = 0; q < ND; ++q) {
      const int b = wave * ND + q, sub = b / RB, r8 = b % RB;
      const uint32_t k0 = (uint32_t)min(st * U + sub, nk - 1) * 128u;
      if (r8 < BM / 8)
        bdma16(rA, voff[q], k0, slot + b * 512);
      else if (EPI == 2 && ((r8 - BM / 8) & 2))
        bdma16(rU, voff[q], k0, slot + b * 512);
      else
        bdma16(rB, voff[q], k0, slot + b * 512);
    }
  };

  float4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  // fragments as gemm_f16_dma's: row lane % 16 of a 16-row block, chunk
  // 4 ks + lane / 16, at chunk ^ ((row >> 1) & 7)
  const int r16 = lane & 15, c16 = lane >> 4;
  int goff[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) goff[ks] = r16 * 64 + (((4 * ks + c16) ^ ((r16 >> 1) & 7)) << 3);
  auto sub_product = [&](const half_t* sub) {
    const half_t* ab = sub + wm * WM * 64;
    const half_t* bb = sub + (BM + wn * WN) * 64;
    frag af[2][TM], bf[2][TN];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int i = 0; i < TM; ++i) af[ks][i] = *reinterpret_cast<const frag*>(ab + goff[ks] + i * 1024);
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[ks][j] = *reinterpret_cast<const frag*>(bb + goff[ks] + j * 1024);
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[ks][j], af[ks][i], acc[i][j], 0, 0, 0);
  };

  // output block (I, J) of a wave: row 16 I + lane % 16, columns
  // 16 J + 4 (lane / 16) .. + 3
  const bool active = wave < VM * VN;
  constexpr int ON16 = EPI == 2 ? TN / 2 : TN;
  const int orow = m0 + wm * WM + r16, ocol = n0 + wn * (EPI == 2 ? WN / 2 : WN) + 4 * c16;
  const int esz = (EPI == 1 || p.dtype_out != 1) ? 4 : 2;
  const bool yvec = ((reinterpret_cast<uintptr_t>(p.y) | (uintptr_t)(p.ldy * esz)) & (4 * esz - 1)) == 0;
  // the residual tile, read first: it is in by the time the products end
  float4_t res[EPI == 1 ? TM : 1][EPI == 1 ? TN : 1];
  if constexpr (EPI == 1) {
    const float* y = static_cast<const float*>(p.y);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int r = orow + 16 * i, c = ocol + 16 * j;
        res[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
        if (!active || r >= p.M) continue;
        const float* src = y + (int64_t)r * p.ldy + c;
        if (yvec && c + 3 < p.N) {
          res[i][j] = *reinterpret_cast<const float4_t*>(src);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (c + e < p.N) res[i][j][e] = src[e];
        }
      }
  }

#pragma unroll
  for (int st = 0; st < S - 1; ++st)
    if (st < nst) issue(st);
  int slot = 0;
  for (int st = 0; st < nst; ++st) {
    // stage st has landed once only the stages after it are in flight
    const int after = min(nst - 1 - st, S - 2);
#pragma unroll
    for (int a = 0; a <= S - 2; ++a)
      if (after == a) vm_wait_n(a * ND, std::make_integer_sequence<int, 64>{});
    lds_barrier();  // publishes stage st; every wave is past stage st - 1
    if (st + S - 1 < nst) issue(st + S - 1);
    const half_t* const base = smem + slot * kSlot;
    slot = slot + 1 == S ? 0 : slot + 1;
    if (active) {
      if (U == 1 || (st + 1) * U <= nk) {
#pragma unroll
        for (int u = 0; u < U; ++u) sub_product(base + u * kSub);
      } else {
        for (int u = 0; u < nk - st * U; ++u) sub_product(base + u * kSub);
      }
    }
  }

  if (!active) return;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < ON16; ++j) {
      const int r = orow + 16 * i, c = ocol + 16 * j;
      if (r >= p.M) continue;
      float4_t o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (EPI == 2) {  // half roundings of neural.metal:35-42, as gemm_f16_dma's
          const float gh = static_cast<float>(to_f16(acc[i][2 * j][e]));
          const float sh = static_cast<float>(to_f16(silu_hw(gh)));
          o[e] = sh * static_cast<float>(to_f16(acc[i][2 * j + 1][e]));
        } else if constexpr (EPI == 1) {
          const float v = acc[i][j][e];
          o[e] = res[i][j][e] + (p.dtype_out == 1 ? static_cast<float>(static_cast<half_t>(v)) : v);
        } else {
          o[e] = acc[i][j][e];
        }
      }
      const int64_t off = (int64_t)r * p.ldy + c;
      if (esz == 2) {
        const half4 h = {static_cast<half_t>(o[0]), static_cast<half_t>(o[1]), static_cast<half_t>(o[2]),
                         static_cast<half_t>(o[3])};
        half_t* dst = static_cast<half_t*>(p.y) + off;
        if (yvec && c + 3 < p.N) {
          *reinterpret_cast<half4*>(dst) = h;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (c + e < p.N) dst[e] = h[e];
        }
      } else {
        float* dst = static_cast<float*>(p.y) + off;
        if (yvec && c + 3 < p.N) {
          *reinterpret_cast<float4_t*>(dst) = o;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (c + e < p.N) dst[e] = o[e];
        }
      }
    }
}

}  // namespace
}  // namespace clef
