// Shared-ring schedule of the W8A8 GEMM for batches of 17 to 128 tokens on long K
// (v_mfma_i32_16x16x64_i8).
#include "i8l_gemm_tile.h"

namespace i8l {

// ------------------------------------------------------------------ shared-ring schedule
// A workgroup of 8 waves computes 16 MT tokens (every token of the batch, so that a weight byte is
// copied into one CU only) x 64 columns over its part of K in 128-byte steps.  The steps of both
// operands go through one ring of S LDS slots, filled by global_load_lds_dwordx4 S - 1 steps ahead:
// a slot holds the 64 weight rows and then the 16 MT token rows of a step (chunk c of row r at slot
// c ^ (r & 7)).  Wave w multiplies columns 16 (w % 4) .. +15 by every token over half w / 4 of each
// step; the two halves' sums meet once, at the end.
//
// What bounds it is the bytes a CU has in flight, LDS-limited to about 140 KiB: 516 KB go through a
// CU in 15.2 us (75 tokens, 14336 -> 4096, 4 parts), so a request takes about 4 us to be used; the
// waves wait for 51% of their cycles, MFMA busy is 8.5%.  gemm_wlds_a keeps a ring per wave (one or
// two steps of it in flight), sums its four waves' K slices through LDS and needs two 64-row blocks
// past 64 tokens, each copying every weight byte.
template <int MT, int EK>
__global__ void __launch_bounds__(512)
gemm_ring(const int8_t* __restrict__ A, int64_t lda, const int8_t* __restrict__ B, int64_t ldb,
          Epi e, int steps, int parts) {
  pin_args(e, A, lda, B, ldb, steps, parts);
  constexpr int BK = 128, NC = 64, W = 8;
  constexpr int ROWS = NC + 16 * MT;
  constexpr int SLOT = ROWS * BK;
  constexpr int S = ring_slots(MT);
  constexpr int NI = ROWS / 8;                 // copies (8 rows each) of a step
  constexpr int CL = NI / W, CX = NI % W;      // a wave issues CL, the first CX waves one more
  extern __shared__ __attribute__((aligned(16))) int8_t lds[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, grp = lane >> 4;
  const int cg = wave & 3, kh = wave >> 2;
  const int64_t n0 = xcd_col_tile() * NC;
  const int64_t m0 = (int64_t)blockIdx.y * (16 * MT);
  const int s0 = (int)((int64_t)blockIdx.z * steps / parts);
  const int ns = (int)((int64_t)(blockIdx.z + 1) * steps / parts) - s0;

  // Copy j of this wave: slot rows [8x, 8x + 8), x = W j + wave; lane l fetches chunk
  // (l % 8) ^ (row & 7) of row 8x + l / 8 (token rows past M: the last row, never stored).
  const int l8 = lane >> 3, chunk = ((lane & 7) ^ l8) * 16;
  const int8_t* gp[CL + 1];
#pragma unroll
  for (int j = 0; j <= CL; ++j) {
    const int row = min(W * j + wave, NI - 1) * 8 + l8;
    gp[j] = (row < NC ? B + (n0 + row) * ldb
                      : A + min(m0 + row - NC, (int64_t)e.M - 1) * lda) + (int64_t)s0 * BK + chunk;
  }
  const bool more = wave < CX;
  auto request = [&](int t, int slot) {
    lds_i8* dst = (lds_i8*)(lds + slot * SLOT + wave * 1024);
    const int64_t ko = (int64_t)t * BK;
#pragma unroll
    for (int j = 0; j < CL; ++j) {
      if ((W * j + W) * 8 <= NC)   // weight rows only: streamed
        __builtin_amdgcn_global_load_lds((const void*)(gp[j] + ko), dst + j * W * 1024, 16, 0,
                                         kWeightCpol);
      else
        __builtin_amdgcn_global_load_lds((const void*)(gp[j] + ko), dst + j * W * 1024, 16, 0, 0);
    }
    if (CX && more)
      __builtin_amdgcn_global_load_lds((const void*)(gp[CL] + ko), dst + CL * W * 1024, 16, 0, 0);
  };
  // All but the newest `D` requested steps have landed (this wave's copies of them).
  auto landed = [&](auto d) {
    constexpr int D = decltype(d)::value;
    if (CX && more) wait_vmcnt_lgkm0<D * (CL + 1)>();
    else wait_vmcnt_lgkm0<D * CL>();
  };

  const int bofs = (16 * cg + r16) * BK + (((4 * kh + grp) ^ (r16 & 7)) * 16);
  const int aofs = (NC + r16) * BK + (((4 * kh + grp) ^ (r16 & 7)) * 16);
  v4i acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = v4i{0, 0, 0, 0};
  auto multiply = [&](int slot) {
    const int8_t* base = lds + slot * SLOT;
    const v4i b = *(const v4i*)(base + bofs);
    v4i a[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) a[i] = *(const v4i*)(base + aofs + i * 16 * BK);
    __builtin_amdgcn_sched_barrier(0);   // every read in flight before the first MFMA waits
#pragma unroll
    for (int i = 0; i < MT; ++i)
      acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, a[i], acc[i], 0, 0, 0);
  };

#pragma unroll
  for (int t = 0; t < S - 1; ++t)
    if (t < ns) request(t, t);
  // Step t: its copies have landed everywhere and every wave is done with step t - 1, whose slot
  // then takes step t + S - 1.
  int t = 0, slot = 0;
  for (; t + S - 1 < ns; ++t) {
    landed(std::integral_constant<int, S - 2>{});
    lds_barrier();
    request(t + S - 1, slot == 0 ? S - 1 : slot - 1);
    multiply(slot);
    slot = slot + 1 == S ? 0 : slot + 1;
  }
  // the last S - 1 steps (fewer on a short K), the waits coarser: half of them, then the rest
  constexpr int H = (S - 1) / 2;
  for (; t < ns; ++t) {
    if (ns - 1 - t >= H) landed(std::integral_constant<int, H>{});
    else landed(std::integral_constant<int, 0>{});
    lds_barrier();
    multiply(slot);
    slot = slot + 1 == S ? 0 : slot + 1;
  }

  // the halves' sums: waves 4-7 hand theirs over, waves 0-3 add and store
  __syncthreads();
  v4i* red = (v4i*)lds;   // [4][MT][64]
  if (kh == 1) {
#pragma unroll
    for (int i = 0; i < MT; ++i) red[(cg * MT + i) * 64 + lane] = acc[i];
  }
  __syncthreads();
  if (kh == 1) return;
  const int64_t n = n0 + 16 * cg + 4 * grp;
  if (parts > 1) {
    int32_t* out = (int32_t*)e.out + (int64_t)blockIdx.z * e.M * e.ldc;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int64_t m = m0 + 16 * i + r16;
      if (m < e.M) *(v4i*)(out + m * e.ldc + n) = acc[i] + red[(cg * MT + i) * 64 + lane];
    }
  } else {
    const Cols4 cl = load_cols4<EK>(e, n);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int64_t m = m0 + 16 * i + r16;
      if (m < e.M)
        store4s<EK>(e, m, n, acc[i] + red[(cg * MT + i) * 64 + lane], cl, load_sa<EK>(e, m));
    }
  }
}

// ------------------------------------------------------------------ host side
bool ring_ok(const i8l_config& c, int64_t K) {
  return c.stages == kRingStages && c.bn == 64 && c.bk == 128 && c.warps == 8 && c.bm >= 32 &&
         c.bm <= 128 && c.bm % 16 == 0 && c.group_m >= 1 && c.group_m <= 8 && K > 0 &&
         K % 128 == 0 && K / 128 >= c.group_m;
}

template <int MT, int EK>
hipError_t launch_ring_k(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb, const Epi& e,
                         int64_t K, int parts, hipStream_t st) {
  auto kern = gemm_ring<MT, EK>;
  constexpr size_t shm = (size_t)ring_slots(MT) * (64 + 16 * MT) * 128;
  static std::atomic<uint64_t> lds_done{0};  // devices this kernel is opted in on
  lds_opt_in((const void*)kern, shm, lds_done);
  const dim3 grid(e.N / 64, (e.M + 16 * MT - 1) / (16 * MT), parts);
  hipLaunchKernelGGL(kern, grid, dim3(512), shm, st, a, lda, b, ldb, e, (int)(K / 128), parts);
  return hipGetLastError();
}

template <int MT>
hipError_t launch_ring_t(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb, const Epi& e,
                         int64_t K, int parts, hipStream_t st) {
  if (parts > 1) return launch_ring_k<MT, EK_ANY>(a, lda, b, ldb, e, K, parts, st);
  switch (epi_kind(e)) {
    case EK_BF16: return launch_ring_k<MT, EK_BF16>(a, lda, b, ldb, e, K, 1, st);
    case EK_BF16_BBF16: return launch_ring_k<MT, EK_BF16_BBF16>(a, lda, b, ldb, e, K, 1, st);
  }
  return launch_ring_k<MT, EK_ANY>(a, lda, b, ldb, e, K, 1, st);
}

// `out`: the output, or the partial planes of a split of K (ws, ldc = N), which splitk_sum adds.
hipError_t launch_ring(const i8l_config& c, const int8_t* a, int64_t lda, const int8_t* b,
                       int64_t ldb, const Epi& e, int64_t K, hipStream_t st) {
  switch (c.bm / 16) {
    case 2: return launch_ring_t<2>(a, lda, b, ldb, e, K, c.group_m, st);
    case 3: return launch_ring_t<3>(a, lda, b, ldb, e, K, c.group_m, st);
    case 4: return launch_ring_t<4>(a, lda, b, ldb, e, K, c.group_m, st);
    case 5: return launch_ring_t<5>(a, lda, b, ldb, e, K, c.group_m, st);
    case 6: return launch_ring_t<6>(a, lda, b, ldb, e, K, c.group_m, st);
    case 7: return launch_ring_t<7>(a, lda, b, ldb, e, K, c.group_m, st);
    case 8: return launch_ring_t<8>(a, lda, b, ldb, e, K, c.group_m, st);
  }
  return hipErrorInvalidValue;
}

}  // namespace i8l
