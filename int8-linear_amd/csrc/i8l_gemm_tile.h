// Pieces the macro-tile schedules share (i8l_gemm_prefill.hip, i8l_gemm_phased.hip): the epilogue
// operands of a 32x32-fragment wave tile, the LDS swizzle, the tile order and the explicit waits.
#pragma once

#include "i8l_gemm.h"

namespace i8l {

// The scales and bias of a wave's FA x 4 column quads (column n = nb + 32a + 8q), every load
// issued before any is used: one memory round trip.  BD (the bias dtype) and SBC (per-column
// scale_b) are fixed per specialization, so no branch separates the loads.
template <int FA, int BD, bool SBC>
__device__ __forceinline__ void load_tile_cols_k(const Epi& e, int64_t nb, Cols4 (&cl)[FA][4]) {
  float4 sbv[FA][4];
  float sb0 = 0.0f;
  uint2 bh[FA][4];
  float4 bf[FA][4];
#pragma unroll
  for (int a = 0; a < FA; ++a)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t n = nb + 32 * a + 8 * q;
      if constexpr (SBC) sbv[a][q] = *(const float4*)(e.sb + n);
      if constexpr (BD == I8L_F32) bf[a][q] = *(const float4*)((const float*)e.bias + n);
      if constexpr (BD == I8L_BF16 || BD == I8L_F16)
        bh[a][q] = *(const uint2*)((const uint16_t*)e.bias + n);
    }
  if constexpr (!SBC) sb0 = e.sb[0];
#pragma unroll
  for (int a = 0; a < FA; ++a)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      Cols4& c = cl[a][q];
      if constexpr (SBC) {
        c.sb[0] = sbv[a][q].x, c.sb[1] = sbv[a][q].y, c.sb[2] = sbv[a][q].z, c.sb[3] = sbv[a][q].w;
      } else {
        c.sb[0] = c.sb[1] = c.sb[2] = c.sb[3] = sb0;
      }
      if constexpr (BD == I8L_F32) {
        c.bias[0] = bf[a][q].x, c.bias[1] = bf[a][q].y, c.bias[2] = bf[a][q].z,
        c.bias[3] = bf[a][q].w;
      } else if constexpr (BD == I8L_BF16 || BD == I8L_F16) {
        const uint32_t w[4] = {bh[a][q].x & 0xffffu, bh[a][q].x >> 16, bh[a][q].y & 0xffffu,
                               bh[a][q].y >> 16};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          c.bias[r] = BD == I8L_BF16 ? bf16_bits_to_f32(w[r]) : f16_bits_to_f32(w[r]);
      } else {
        // no bias: -0, the identity of IEEE addition (x + -0 == x for every x, -0 and NaN
        // included), so the epilogue adds the bias without a test
        c.bias[0] = c.bias[1] = c.bias[2] = c.bias[3] = -0.0f;
      }
    }
}

template <int FA, bool SBC>
__device__ __forceinline__ void load_tile_cols_s(const Epi& e, int64_t nb, Cols4 (&cl)[FA][4]) {
  switch (e.bias_dtype) {
    case I8L_DTYPE_NONE: load_tile_cols_k<FA, I8L_DTYPE_NONE, SBC>(e, nb, cl); break;
    case I8L_BF16: load_tile_cols_k<FA, I8L_BF16, SBC>(e, nb, cl); break;
    case I8L_F16: load_tile_cols_k<FA, I8L_F16, SBC>(e, nb, cl); break;
    default: load_tile_cols_k<FA, I8L_F32, SBC>(e, nb, cl); break;
  }
}

// An LDS tile row (one token or one weight row) holds BK bytes as BK/16 chunks of 16 bytes,
// chunk c at slot c ^ swz(row), so that the lanes of an MFMA fragment read hit distinct banks.
template <int BK>
__device__ __forceinline__ int swz(int row) {
  constexpr int NCH = BK / 16;
  constexpr int SH = (BK == 64) ? 2 : (BK == 128 ? 1 : 0);
  return (row >> SH) & (NCH - 1);
}

// Tile order: GROUP_M rows of tiles are walked together so that concurrently running
// workgroups share A rows and B columns in L2, and consecutive positions of that order are
// given to the same XCD (the dispatcher deals workgroups to the 8 XCDs round-robin).
__device__ __forceinline__ void staged_tile(int pid, int npid, int num_pid_m, int num_pid_n,
                                            int group_m, int& pid_m, int& pid_n) {
  if (npid % 8 == 0) pid = (pid % 8) * (npid / 8) + pid / 8;
  const int in_group = group_m * num_pid_n;
  const int first_m = (pid / in_group) * group_m;
  const int gsize = min(num_pid_m - first_m, group_m);
  pid_m = first_m + (pid % in_group) % gsize;
  pid_n = (pid % in_group) / gsize;
}

// Position `pid` of `npid` in the order staged_tile makes of a multiple of 8, for any other count:
// consecutive positions go to one XCD, the first npid % 8 XCDs taking one more.  The phased tiles
// need it: without, an operand's rows are fetched into every XCD's L2, and 222 tiles of 128 x 256
// (331 tokens, 3584 -> 18944) took 42.3 us where the ring of that size takes 38; with it 32.3.
// 1536 -> 8960 at 2500 tokens (128 x 256) 62.9 -> 45.9, 2560 -> 9728 at 300 (128 x 128) 22.6 ->
// 15.9, 1792 -> 9792 at 1543 (128 x 192) 55.8 -> 51.1.
__device__ __forceinline__ int xcd_order(int pid, int npid) {
  const int x = pid % 8;
  return x * (npid / 8) + min(x, npid % 8) + pid / 8;
}

typedef __attribute__((address_space(3))) int8_t lds_i8;

// s_waitcnt with vmcnt = N and the LGKM / EXP counters left unconstrained (gfx9 encoding:
// vmcnt[3:0] in bits 3:0 and vmcnt[5:4] in bits 15:14, expcnt 6:4, lgkmcnt 11:8).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt out of range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// The same with lgkmcnt = 0 as well: this wave's LDS reads (and scalar loads) have returned.
template <int N>
__device__ __forceinline__ void wait_vmcnt_lgkm0() {
  static_assert(N >= 0 && N < 64, "vmcnt out of range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
}

}  // namespace i8l
