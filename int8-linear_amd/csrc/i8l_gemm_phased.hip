// Phased prefill schedule of the W8A8 GEMM: persistent macro tiles whose K steps are cut into
// four phases, one per quadrant of a wave's tile (v_mfma_i32_32x32x32_i8).
#include "i8l_gemm_tile.h"

namespace i8l {

// ------------------------------------------------------------------ phased schedule
// A workgroup of 4 waves (2 x 2, one a SIMD) computes BM x BN output tiles in BK-byte K steps.
// A wave's tile is 2 x 2 quadrants of 32 x 32 fragments: its tokens are an A half 0 and 1 of QA
// fragments each, its columns a B half 0 and 1 of QB0 and QB1, and the LDS holds each operand's
// step as those two halves (half h: the h-th part of every wave's rows), in two buffers.
//
// Step t is four phases, with f = t % 2 and s = 1 - f (the order of the B halves alternates):
//   phase 0: MFMAs of (A0, Bf);   reads Bs(t);     requests A0(t+2)
//   phase 1: MFMAs of (A0, Bs);   reads A1(t);     requests Bf(t+2)
//   phase 2: MFMAs of (A1, Bs);   reads A0(t+1);   requests Bs(t+2)
//   phase 3: MFMAs of (A1, Bf);   reads Bs(t+1), which is t+1's first;  requests A1(t+2)
// so every fragment is read from LDS once a step and a phase before its first use, and the copies
// of a step (global_load_lds) go out a quarter a phase, each into the half whose reads ended a
// phase before, six phases before it is read.  Each phase ends with lgkmcnt(0) (this wave's
// reads are done: that half may be refilled), vmcnt (all but the newest five halves have landed:
// the next phase's reads) and one workgroup barrier, which makes both true of every wave.
//
// The workgroups walk the tiles (tile, tile + gridDim.x, ...): the copies of a tile's last two
// steps are the next tile's first two, so they fly during the epilogue, which every wave does
// alone through its own 4 KiB of LDS.
//
// What bounds it: power.  On random operands the clock falls to 1.5-1.6 GHz at 73-77% MFMA busy
// (v_mfma alone reaches 3.45 POP/s at 1.77 GHz); in timing copies, leaving out the barriers gains
// 1%, the LDS reads 8%, the copies 13%.
// So a wave's tile is as large as its registers allow (128 x 128: 256 accumulators), which reads
// LDS least per MFMA.  Llama-3-8B at 4096 tokens, us: down_proj 199 (gemm_dmap 256x256x128) ->
// 181 (8 waves of 128x64) -> 174.5 (4 of 128x128), o_proj 63 -> 57.4 -> 55.4, gate_up 433 -> 380.

// global_load_lds_dwordx4 with a scalar base and a 32-bit lane offset: 16 bytes a lane into 1 KiB of
// LDS from `dst` on.  Written as assembly for that form (the builtin keeps a 64-bit address per
// lane, two registers a copy) and so that the compiler, which cannot count these among other
// requests, places no wait of its own: the phases' explicit waits cover them.
__device__ __forceinline__ void copy_1k(const int8_t* base, uint32_t off, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               ::"v"(off), "s"(base), "s"(dst) : "memory", "m0");
}

// How the epilogue takes its bias: none, of the output's dtype, or of the dtype found at run time
// (the switch over dtypes costs registers that the 256 x 256 tile does not have to spare).
enum { kNoBias = 0, kOwnBias = 1, kAnyBias = 2 };

// The epilogue operands of a wave's 64 columns (2 fragments): per-column scales, and the bias.
template <int OD, int BIAS>
__device__ __forceinline__ void load_phased_cols(const Epi& e, int64_t n, Cols4 (&cl)[2][4]) {
  if constexpr (BIAS == kAnyBias) {
    if (e.sb_per_col) load_tile_cols_s<2, true>(e, n, cl);
    else load_tile_cols_s<2, false>(e, n, cl);
  } else {
    constexpr int BD = BIAS == kNoBias ? I8L_DTYPE_NONE : OD;
    if (e.sb_per_col) load_tile_cols_k<2, BD, true>(e, n, cl);
    else load_tile_cols_k<2, BD, false>(e, n, cl);
  }
}

// OD: the output dtype; BIAS: as above.
template <int QA, int QB0, int QB1, int BK, int OD, int BIAS>
__global__ void __launch_bounds__(256)
gemm_phased(const int8_t* __restrict__ A, int64_t lda, const int8_t* __restrict__ B, int64_t ldb,
            Epi e, int K, int group_m, int tiles) {
  pin_args(e, A, lda, B, ldb, K, group_m, tiles);
  constexpr int W = 4, WN = 2;                       // 2 x 2 waves
  constexpr int QB[2] = {QB0, QB1};
  constexpr int QN = QB0 + QB1;                      // column fragments of a wave
  constexpr int BM = 128 * QA, BN = 64 * QN;
  constexpr int CPR = BK / 16, RPC = 64 / CPR;       // chunks of a row, rows of a copy
  constexpr int KK = BK / 32;                        // MFMA substeps of a step
  constexpr int HA = BM / 2 * BK;                    // bytes of an A half
  constexpr int HB[2] = {64 * QB0 * BK, 64 * QB1 * BK};
  constexpr int JA = HA / 1024 / W, JB[2] = {HB[0] / 1024 / W, HB[1] / 1024 / W};  // copies a wave
  constexpr int B0 = 4 * HA;                         // LDS: A [buffer][half], then B, then staging
  constexpr int SB = HB[0] + HB[1];
  constexpr int STG = B0 + 2 * SB;
  static_assert(QB1 <= QB0 && QB1 >= 1, "the first B half is the larger");
  extern __shared__ __attribute__((aligned(16))) int8_t lds[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int num_pid_m = (e.M + BM - 1) / BM, num_pid_n = e.N / BN;
  const int KT = K / BK;

  // Copies: copy j of a half writes LDS rows [RPC x, RPC x + RPC), x = W j + wave; lane l writes
  // slot l % CPR of row l / CPR.  Half row r lies in wave block r / R of that half (R rows each).
  const int lrow = lane / CPR;
  const int chunk = ((lane % CPR) ^ swz<BK>(wave * RPC + lrow)) * 16;
  static_assert((W * RPC) % 16 == 0, "the swizzle must not depend on j");
  const int lda32 = (int)lda, ldb32 = (int)ldb;
  int arow[2][JA], brow[2][JB[0]];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    constexpr int RA = 32 * QA;
#pragma unroll
    for (int j = 0; j < JA; ++j) {
      const int r = (W * j + wave) * RPC;
      arow[h][j] = (r / RA) * (2 * RA) + h * RA + r % RA;
    }
    const int RB = 32 * QB[h];
#pragma unroll
    for (int j = 0; j < JB[0]; ++j) {
      const int r = (W * j + wave) * RPC;
      brow[h][j] = ((r / RB) * (32 * QN) + h * 32 * QB0 + r % RB) * ldb32;
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_i8*)lds + wave * 1024;
  const uint32_t voffB = (uint32_t)(lrow * ldb32 + chunk);
  uint32_t voffA[2][JA];
  const int8_t *pA, *pB;   // the K position being requested, in the tile being requested
  auto tile_at = [&](int tile, int64_t& mt, int64_t& nt) {
    int pid_m, pid_n;
    staged_tile(tiles % 8 == 0 ? tile : xcd_order(tile, tiles), tiles, num_pid_m, num_pid_n, group_m,
                pid_m, pid_n);
    mt = (int64_t)pid_m * BM;
    nt = (int64_t)pid_n * BN;
  };
  auto request_from = [&](int64_t mt, int64_t nt) {
    pA = A + mt * lda;
    pB = B + nt * ldb;
    const int last = e.M - 1 - (int)mt;   // token rows past M copy the last row, never stored
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < JA; ++j)
        voffA[h][j] = (uint32_t)(min(arow[h][j] + lrow, last) * lda32 + chunk);
  };
  // copy j of A's / B's half h of the step at pA / pB, into buffer buf
  auto copyA = [&](int h, int buf, int j) {
    copy_1k(pA, voffA[h][j], lds0 + (2 * buf + h) * HA + j * 1024 * W);
  };
  auto copyB = [&](int h, int buf, int j) {
    copy_1k(pB + brow[h][j], voffB, lds0 + B0 + buf * SB + h * HB[0] + j * 1024 * W);
  };

  // Fragment reads: lane l reads row l%32 of a 32-row block, chunk 2*kk + l/32.
  const int frow = lane & 31, fhalf = lane >> 5;
  int ofs[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) ofs[kk] = frow * BK + (((2 * kk + fhalf) ^ swz<BK>(frow)) * 16);
  const int8_t* la = lds + wm * 32 * QA * BK;
  const int8_t* lb[2] = {lds + B0 + wn * 32 * QB0 * BK, lds + B0 + HB[0] + wn * 32 * QB1 * BK};
  v4i fa[2][QA][KK], fb[2][QB0][KK];
  auto readA = [&](int h, int buf, int kk) {
#pragma unroll
    for (int i = 0; i < QA; ++i)
      fa[h][i][kk] = *(const v4i*)(la + ofs[kk] + (2 * buf + h) * HA + i * 32 * BK);
  };
  auto readB = [&](int h, int buf, int kk) {
#pragma unroll
    for (int i = 0; i < QB0; ++i)
      if (i < QB[h]) fb[h][i][kk] = *(const v4i*)(lb[h] + ofs[kk] + buf * SB + i * 32 * BK);
  };

  v16i acc[2][2][QA][QB0];
  // A phase's work: per MFMA substep its MFMAs with the next phase's reads of that substep
  // between them, and one in KK of its copies, so that neither the LDS nor the copy path gets a
  // burst that holds up the MFMAs behind it.
  // zero: a tile's first step, whose first substep starts the sums from 0.
  auto body = [&](auto hac, auto hbc, auto zero, auto read, int reads, auto copy, auto copies) {
    constexpr int ha = decltype(hac)::value, hb = decltype(hbc)::value;
    constexpr int NC = decltype(copies)::value;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
#pragma unroll
      for (int i = 0; i < QA; ++i)
#pragma unroll
        for (int j = 0; j < QB[hb]; ++j)
          acc[ha][hb][i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(
              fb[hb][j][kk], fa[ha][i][kk],
              decltype(zero)::value && kk == 0 ? v16i{} : acc[ha][hb][i][j], 0, 0, 0);
      read(kk);
#pragma unroll
      for (int j = kk * NC / KK; j < (kk + 1) * NC / KK; ++j) copy(j);
#pragma unroll
      for (int i = 0; i < QA * QB[hb]; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                 // one MFMA
        if (i < reads) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // One K step of parity `par`.  TAIL: a tile's last (it reads nothing ahead).  HEAD: 4 for a
  // tile's first step and 1 for its second, the phases that `landed` spares the wait for copies
  // (a workgroup's later tiles find them landed).
  auto step = [&](auto par, auto tail, auto headc, bool landed) {
    constexpr int f = decltype(par)::value, s = 1 - f;
    constexpr bool TAIL = decltype(tail)::value;
    constexpr int HEAD = decltype(headc)::value;   // phases whose wait `landed` may skip
    constexpr std::bool_constant<HEAD == 4> zero{};
    typedef std::integral_constant<int, 0> H0;
    typedef std::integral_constant<int, 1> H1;
    typedef std::integral_constant<int, f> HF;
    typedef std::integral_constant<int, s> HS;
    constexpr int NA = 3 * JA + JB[0] + JB[1], NB = 2 * JA + JB[0] + JB[1] + JB[f];
    auto phase_end = [&](auto phasec, auto nc) {
      constexpr int phase = decltype(phasec)::value, N = decltype(nc)::value;
      if constexpr (phase < HEAD) {
        wait_lgkmcnt0();
        if (!landed) wait_vmcnt<N>();
      } else {
        wait_vmcnt_lgkm0<N>();
      }
      lds_barrier();
    };
    // opaque to the compiler, so that it keeps them in scalar registers (and steps no lane
    // addresses)
    asm volatile("" : "+s"(pA), "+s"(pB));
    body(H0{}, HF{}, zero, [&](int kk) { readB(s, f, kk); }, QB[s],
         [&](int j) { copyA(0, f, j); }, std::integral_constant<int, JA>{});
    phase_end(std::integral_constant<int, 0>{}, std::integral_constant<int, NA>{});

    body(H0{}, HS{}, zero, [&](int kk) { readA(1, f, kk); }, QA,
         [&](int j) { copyB(f, f, j); }, std::integral_constant<int, JB[f]>{});
    phase_end(std::integral_constant<int, 1>{}, std::integral_constant<int, NB>{});

    body(H1{}, HS{}, zero, [&](int kk) { if constexpr (!TAIL) readA(0, 1 - f, kk); }, TAIL ? 0 : QA,
         [&](int j) { copyB(s, f, j); }, std::integral_constant<int, JB[s]>{});
    if constexpr (!TAIL) phase_end(std::integral_constant<int, 2>{}, std::integral_constant<int, NB>{});

    body(H1{}, HF{}, zero, [&](int kk) { if constexpr (!TAIL) readB(s, 1 - f, kk); }, TAIL ? 0 : QB[s],
         [&](int j) { copyA(1, f, j); }, std::integral_constant<int, JA>{});
    if constexpr (!TAIL) phase_end(std::integral_constant<int, 3>{}, std::integral_constant<int, NA>{});
    pA += BK;
    pB += BK;
  };
  typedef std::integral_constant<int, 0> P0;
  typedef std::integral_constant<int, 1> P1;
  auto request_step = [&](auto par) {   // a whole step, in the order the phases request it
    constexpr int f = decltype(par)::value, s = 1 - f;
    for (int j = 0; j < JA; ++j) copyA(0, f, j);
    for (int j = 0; j < JB[f]; ++j) copyB(f, f, j);
    for (int j = 0; j < JB[s]; ++j) copyB(s, f, j);
    for (int j = 0; j < JA; ++j) copyA(1, f, j);
    pA += BK;
    pB += BK;
  };

  int tile = blockIdx.x;
  int64_t m0, n0;
  tile_at(tile, m0, n0);
  request_from(m0, n0);
  request_step(P0{});
  request_step(P1{});
  bool landed = false;
  for (;;) {
    // A0(0) and B0(0) into registers, then the steps in pairs, the first and the last apart
    if (!landed) wait_vmcnt<3 * JA + JB[0] + 2 * JB[1]>();
    lds_barrier();
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      readA(0, 0, kk);
      readB(0, 0, kk);
    }
    wait_lgkmcnt0();
    if (!landed) wait_vmcnt<3 * JA + JB[0] + JB[1]>();
    lds_barrier();

    const int next = tile + gridDim.x;   // past the last tile: its own start again, not used
    int64_t m1 = m0, n1 = n0;
    if (next < tiles) tile_at(next, m1, n1);
    // the copies awaited in the first five phases were requested before the previous tile's
    // stores, whose epilogue waited for them
    step(P0{}, std::false_type{}, std::integral_constant<int, 4>{}, landed);
    step(P1{}, std::false_type{}, std::integral_constant<int, 1>{}, landed);
    for (int t = 2; t + 2 < KT; t += 2) {
      step(P0{}, std::false_type{}, P0{}, false);
      step(P1{}, std::false_type{}, P0{}, false);
    }
    request_from(m1, n1);
    step(P0{}, std::false_type{}, P0{}, false);
    step(P1{}, std::true_type{}, P0{}, false);

    // ---- epilogue: acc * scale_a * scale_b (+ bias) in fp32, left to right, then one cast.
    // Each wave takes 32 tokens x 64 columns (16-bit outputs; 32 columns of 4-byte ones) at a
    // time through its 4 KiB: rows of 128 bytes, chunk c at slot c ^ (row & 7), written out in
    // whole 128-byte lines, 8 rows a store.  The lane index is taken anew, opaque, so that what
    // the epilogue derives from it is not kept in registers over the main loop.
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int erow = ln & 31, ehalf = ln >> 5, srow = ln >> 3, sch = ln & 7;
    const int64_t nw = n0 + wn * 32 * QN, mw = m0 + wm * 64 * QA;
    int8_t* stg = lds + STG + wave * 4096;
    float sam[2][QA];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < QA; ++i) {
        const int64_t m = mw + (h * QA + i) * 32 + erow;
        sam[h][i] = OD == I8L_I32 ? 0.0f : load_sa(e, m < e.M ? m : 0);
      }
#pragma unroll
    for (int g = 0; g < (QN + 1) / 2; ++g) {   // fragments 2g and 2g+1 of the wave's columns
      constexpr bool ODD = QN % 2 == 1;
      const int nf = ODD && g == QN / 2 ? 1 : 2;   // (an odd last fragment stands alone)
      Cols4 cl[2][4];
      if constexpr (OD != I8L_I32) {
        const int64_t n = nw + 64 * g + 4 * ehalf;
        if (nf == 2) {
          load_phased_cols<OD, BIAS>(e, n, cl);
        } else {   // the second fragment's columns would lie past the wave's: its first again
          Cols4 c2[2][4];
          load_phased_cols<OD, BIAS>(e, n - 32, c2);
#pragma unroll
          for (int q = 0; q < 4; ++q) cl[0][q] = c2[1][q], cl[1][q] = c2[1][q];
        }
      }
      if (g == 0) {
        // every copy in flight (the next tile's first two steps) has landed past here, so the
        // next tile's first waits need not count past this tile's stores
        wait_vmcnt<0>();
        asm volatile("" ::: "memory");
      }
      auto value = [&](int h, int i, int c, int q, int r) {
        const int x = 2 * g + c, hb = x >= QB0;
        float v = (float)acc[h][hb][i][x - hb * QB0][4 * q + r];
        v = v * sam[h][i];
        v = v * cl[c][q].sb[r];
        if constexpr (BIAS != kNoBias) v = v + cl[c][q].bias[r];
        // the value itself is rounded to fp32 before its cast: opaque, or the product and the
        // cast to fp16 become one v_fma_mixlo_f16, which rounds once
        else if constexpr (OD == I8L_F16) asm volatile("" : "+v"(v));
        return v;
      };
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < QA; ++i) {
          const int64_t mb = mw + (h * QA + i) * 32;
          if constexpr (OD == I8L_I32 || OD == I8L_F32) {
#pragma unroll
            for (int c = 0; c < nf; ++c) {
              const int x = 2 * g + c, hb = x >= QB0;
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                v4i v;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  v[r] = OD == I8L_I32 ? acc[h][hb][i][x - hb * QB0][4 * q + r]
                                       : __float_as_int(value(h, i, c, q, r));
                *(v4i*)(stg + erow * 128 + (((2 * q + ehalf) ^ (erow & 7)) * 16)) = v;
              }
#pragma unroll
              for (int y = 0; y < 4; ++y) {
                const int row = 8 * y + srow;
                const v4i v = *(const v4i*)(stg + row * 128 + ((sch ^ srow) * 16));
                if (mb + row < e.M)
                  __builtin_nontemporal_store(
                      v, (v4i*)((int32_t*)e.out + (mb + row) * e.ldc + nw + 32 * x + 4 * sch));
              }
            }
          } else {
#pragma unroll
            for (int c = 0; c < nf; ++c)
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = value(h, i, c, q, r);
                *(uint2*)(stg + erow * 128 + (((4 * c + q) ^ (erow & 7)) * 16) + 8 * ehalf) =
                    make_uint2(f32x2_to_act2<OD>(v[0], v[1]), f32x2_to_act2<OD>(v[2], v[3]));
              }
#pragma unroll
            for (int y = 0; y < 4; ++y) {
              const int row = 8 * y + srow;
              const v4i v = *(const v4i*)(stg + row * 128 + ((sch ^ srow) * 16));
              if (mb + row < e.M && (nf == 2 || sch < 4))
                __builtin_nontemporal_store(
                    v, (v4i*)((uint16_t*)e.out + (mb + row) * e.ldc + nw + 64 * g + 8 * sch));
            }
          }
        }
      asm volatile("" ::: "memory");   // the next 64 columns' operands load after these
    }
    if (next >= tiles) break;
    tile = next;
    m0 = m1;
    n0 = n1;
    landed = true;
  }
}

// ------------------------------------------------------------------ host side
struct PhasedTile {
  int bm, bn;
};
constexpr PhasedTile kPhased[] = {{256, 256}, {256, 192}, {256, 128},
                                  {128, 256}, {128, 192}, {128, 128}};

int phased_index(const i8l_config& c, int64_t K) {
  if (c.stages != kPhasedStages || c.warps != 4 || c.bk != 128 || c.group_m < 1) return -1;
  for (int i = 0; i < (int)(sizeof(kPhased) / sizeof(kPhased[0])); ++i)
    if (kPhased[i].bm == c.bm && kPhased[i].bn == c.bn)
      // whole pairs of steps, the first and the last apart
      return K % (2 * c.bk) == 0 && K >= 4 * c.bk ? i : -1;
  return -1;
}

template <int QA, int QB0, int QB1, int BK, int OD, int BIAS>
hipError_t launch_phased_k(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                           const Epi& e, int K, int group_m, hipStream_t st) {
  auto kern = gemm_phased<QA, QB0, QB1, BK, OD, BIAS>;
  constexpr int BM = 128 * QA, BN = 64 * (QB0 + QB1);
  constexpr size_t shm = 2 * (size_t)(BM + BN) * BK + 4 * 4096;
  static_assert(shm <= kMaxLds, "two buffers and the staging fit the LDS");
  static std::atomic<uint64_t> lds_done{0};  // devices this kernel is opted in on
  lds_opt_in((const void*)kern, shm, lds_done);
  const int tiles = ((e.M + BM - 1) / BM) * (e.N / BN);
  const int grid = std::min(tiles, cu_count() * (int)(kMaxLds / shm));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), shm, st, a, lda, b, ldb, e, K, group_m, tiles);
  return hipGetLastError();
}

template <int QA, int QB0, int QB1, int BK>
hipError_t launch_phased_t(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                           const Epi& e, int K, int gm, hipStream_t st) {
  auto by_bias = [&](auto odc) {
    constexpr int OD = decltype(odc)::value;
    if (e.bias_dtype == I8L_DTYPE_NONE)
      return launch_phased_k<QA, QB0, QB1, BK, OD, kNoBias>(a, lda, b, ldb, e, K, gm, st);
    if (e.bias_dtype == OD)
      return launch_phased_k<QA, QB0, QB1, BK, OD, kOwnBias>(a, lda, b, ldb, e, K, gm, st);
    return launch_phased_k<QA, QB0, QB1, BK, OD, kAnyBias>(a, lda, b, ldb, e, K, gm, st);
  };
  switch (e.out_dtype) {
    case I8L_BF16: return by_bias(std::integral_constant<int, I8L_BF16>{});
    case I8L_F16: return by_bias(std::integral_constant<int, I8L_F16>{});
    case I8L_F32: return by_bias(std::integral_constant<int, I8L_F32>{});
  }
  return launch_phased_k<QA, QB0, QB1, BK, I8L_I32, kNoBias>(a, lda, b, ldb, e, K, gm, st);
}

hipError_t launch_phased(int idx, const i8l_config& c, const int8_t* a, int64_t lda,
                         const int8_t* b, int64_t ldb, const Epi& e, int K, hipStream_t st) {
  switch (idx) {
    case 0: return launch_phased_t<2, 2, 2, 128>(a, lda, b, ldb, e, K, c.group_m, st);
    case 1: return launch_phased_t<2, 2, 1, 128>(a, lda, b, ldb, e, K, c.group_m, st);
    case 2: return launch_phased_t<2, 1, 1, 128>(a, lda, b, ldb, e, K, c.group_m, st);
    case 3: return launch_phased_t<1, 2, 2, 128>(a, lda, b, ldb, e, K, c.group_m, st);
    case 4: return launch_phased_t<1, 2, 1, 128>(a, lda, b, ldb, e, K, c.group_m, st);
    case 5: return launch_phased_t<1, 1, 1, 128>(a, lda, b, ldb, e, K, c.group_m, st);
  }
  return hipErrorInvalidValue;
}

}  // namespace i8l
