// fp32 GEMM C = epilogue(A * B^T) for B stored [N][K] (Linear / attention projections / FFN,
// PyTorch weight layout; Linear.swift:337-352 computes y = x W^T + b), on v_mfma_f32_32x32x2_f32.
//
// Operand tiles move from HBM to LDS with the CDNA4 LDS-DMA load (global_load_lds_dwordx4): the
// data never passes through VGPRs and no ds_write is issued, so the only per-step work besides
// the matrix cores is one s_barrier and the wave's fragment reads. K advances in 32-deep stages
// held in a ring of S LDS buffers; the loads of stage kt+S are issued once every wave has read
// stage kt into registers, so up to S-1 stages of HBM/L2 latency are in flight behind the
// matrix work.
//
// LDS layout of one stage: A rows [BM][32 floats] then B rows [BN][32 floats], unpadded
// (LDS-DMA writes each wave's 64 x 16 bytes contiguously). A row's 16-byte chunk c is stored at
// slot c ^ f(r), f(r) = (r + r/8) mod 8; the lane that fills slot s of row r fetches chunk s ^ f(r)
// from global memory (the 8 lanes of a row still read one contiguous 128-byte segment). The
// fragment reads (32 rows x one chunk per lane group) then hit distinct banks for 32- and 64-bank
// LDS alike.
//
// The loads are issued by inline asm: the compiler's own tracking of LDS-DMA would make every
// LDS read wait for all outstanding loads (it cannot tell the ring buffers apart), and a
// __syncthreads would wait for them at every barrier. Here the kernel waits itself for exactly the
// stage it is about to read (s_waitcnt vmcnt((S-2) * loads per stage)) before the barrier.
// S = 2 is allowed: the slot of stage kt is refilled as soon as its fragments are in registers.
//
// Within a stage, lane group g = lane/32 owns k in [16g, 16g+16): the MFMA's two k slots are fed
// k = 16g + 4q + s in sub-step (q, s). A and B use the same assignment, so the sum over k is
// unchanged, and each lane reads its 4 consecutive k of a row with one 16-byte LDS read.
#include "device_utils.hpp"
#include "gemm_epilogue.hpp"
#include "kernels.hpp"
#include "lds_dma.hpp"

namespace mnn {
namespace k {

using namespace dev;

namespace {

constexpr int BK = 32;

template <int WMW, int WNW, int WM, int WN, int S>
struct LdsCfg {
  static constexpr int BM = WMW * WM * 32, BN = WNW * WN * 32;
  static constexpr int NW = WMW * WNW, NT = NW * 64;
  static constexpr int A_INS = BM / 8 / NW, B_INS = BN / 8 / NW;  // 8 rows per wave load
  static constexpr int L = A_INS + B_INS;                         // loads per wave per stage
  static constexpr int STAGE = (BM + BN) * BK;                    // floats
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "tile rows must split over waves");
  static_assert((S - 1) * L < 64, "vmcnt range");
};

// EPI: 0 bias / activation / residual (store_tile), 1 GLU (store_glu: an encoder's rewrite GEMM whose
// split weight would pass 4 GiB, from 18919 channels on), 3 K-split partials (store_part); each a
// separate instantiation.
//
// BF: A and B hold bf16 values (lda / ldb / sA / sB count bf16 elements). A stage is still 128
// bytes per row — 64 k — with the same swizzle; a lane's 16-byte fragment read is then 8
// consecutive k, exactly the operand of one v_mfma_f32_32x32x16_bf16 (lane group g supplies k
// slots 8g..8g+7), so chunk c = 4g + q4 of a stage feeds MFMA step q4 for A and B alike.
// The second launch bound asks for two workgroups per CU where two rings fit the 160 KB of LDS.
template <int WMW, int WNW, int WM, int WN, int S, int EPI, bool BF = false>
__global__ __launch_bounds__(WMW* WNW * 64,
                             (2 * S * (WMW * WM + WNW * WN) * 32 * BK * 4 <= 160 * 1024) ? 2 : 1)
void gemm_nk_lds_kernel(GemmArgs a) {
  using Cfg = LdsCfg<WMW, WNW, WM, WN, S>;
  constexpr int BM = Cfg::BM, BN = Cfg::BN, A_INS = Cfg::A_INS, B_INS = Cfg::B_INS;
  constexpr int STAGE = Cfg::STAGE;
  constexpr int ES = BF ? 2 : 4;           // operand element bytes
  constexpr int BKE = BF ? 2 * BK : BK;    // k per 128-byte stage row
  __shared__ __attribute__((aligned(1024))) float smem[S * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WNW, wn = wave % WNW;
  // blockIdx.z = batch * ksplit + K part (ksplit = 1 unless EPI == 3)
  const int ks = EPI == 3 ? a.ksplit : 1;
  const int bz = blockIdx.z / ks;
  // XCD-aware renumbering (workgroups go round robin over the 8 XCDs): consecutive logical tiles,
  // N fastest, land on one XCD and share the A panel in its L2.
  const int gx = gridDim.x;
  const int logical = xcd_logical_tile(blockIdx.x + gx * blockIdx.y, gx * gridDim.y);
  const int tn = logical % gx, tm = logical / gx;
  const int m0 = tm * BM, n0 = tn * BN;
  const int M = a.M, N = a.N, K = a.K;
  const int nk = K / BKE / ks, kt0 = (int)(blockIdx.z % ks) * nk;  // this workgroup's stages
  // a folded LayerNorm's row partials (thread r: row m0 + r % BM)
  LnRow lnr;
  if constexpr (EPI == 0 && !BF) lnr = ln_row_load(a, m0 + tid % BM);
  const char* __restrict__ A = reinterpret_cast<const char*>(a.A) + (int64_t)bz * a.sA * ES;
  const char* __restrict__ B = reinterpret_cast<const char*>(a.B) + (int64_t)bz * a.sB * ES;

  // Per-lane byte offsets of this wave's stage loads from the operand base (rows past M / N are
  // clamped to the last row: they are read but their products are never stored). The base moves
  // by one stage per load round in SGPRs, so the loads need no per-stage VALU address work.
  const int lr = lane >> 3, ls = lane & 7;
  unsigned aoffg[A_INS], boffg[B_INS];
#pragma unroll
  for (int i = 0; i < A_INS; ++i) {
    const int rr = (wave * A_INS + i) * 8 + lr;
    const int gm = min(m0 + rr, M - 1);
    aoffg[i] = (unsigned)(ES * gm * a.lda + 16 * (ls ^ chunk_swizzle(rr)));
  }
#pragma unroll
  for (int i = 0; i < B_INS; ++i) {
    const int rr = (wave * B_INS + i) * 8 + lr;
    const int gn = min(n0 + rr, N - 1);
    boffg[i] = (unsigned)(ES * gn * a.ldb + 16 * (ls ^ chunk_swizzle(rr)));
  }
  const unsigned lds0 = lds_address(smem);
  auto issue = [&](int kt, int slot) {
    const unsigned base = lds0 + 4u * (unsigned)(slot * STAGE);
    const float* ak = reinterpret_cast<const float*>(A + (int64_t)(kt0 + kt) * BKE * ES);
    const float* bk = reinterpret_cast<const float*>(B + (int64_t)(kt0 + kt) * BKE * ES);
#pragma unroll
    for (int i = 0; i < A_INS; ++i)
      lds_dma16_s(ak, aoffg[i],
                  __builtin_amdgcn_readfirstlane(base + 4u * ((wave * A_INS + i) * 8 * BK)));
#pragma unroll
    for (int i = 0; i < B_INS; ++i)
      lds_dma16_s(bk, boffg[i], __builtin_amdgcn_readfirstlane(
                                    base + 4u * (BM * BK + (wave * B_INS + i) * 8 * BK)));
  };

  floatx16 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // LDS word offsets of this lane's fragment rows in slot 0 (other slots: a constant offset)
  const int g = lane >> 5, l32 = lane & 31;
  int aoff[WM], boff[WN], asw[WM], bsw[WN];
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int rr = wm * WM * 32 + 32 * i + l32;
    aoff[i] = rr * BK;
    asw[i] = chunk_swizzle(rr);
  }
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const int rr = wn * WN * 32 + 32 * j + l32;
    boff[j] = BM * BK + rr * BK;
    bsw[j] = chunk_swizzle(rr);
  }

  // Software pipeline: the fragments of stage kt sit in registers while the matrix cores work on
  // them. Halfway through stage kt (after the MFMAs of its first two 8-deep k slices) the waves
  // meet at the barrier that makes stage kt+1 visible and frees the slot of stage kt, issue the
  // loads of stage kt+S into that slot, and read stage kt+1's fragments interleaved with the
  // second half's MFMAs, so neither the barrier nor the LDS latency stalls the matrix pipe.
  // The stage loop is unrolled by U (a multiple of S and of 2), so every ring slot and the two
  // fragment register sets are compile-time choices: no address arithmetic and no register copies
  // between stages.
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < nk) issue(s, s);
  float4 fa[2][4][WM], fb[2][4][WN];
  auto read_frags = [&](int slot, float4 (&xa)[4][WM], float4 (&xb)[4][WN]) {
    const float* base = smem + slot * STAGE;
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int c = 4 * g + q4;
#pragma unroll
      for (int i = 0; i < WM; ++i)
        xa[q4][i] = *reinterpret_cast<const float4*>(base + aoff[i] + 4 * (c ^ asw[i]));
#pragma unroll
      for (int j = 0; j < WN; ++j)
        xb[q4][j] = *reinterpret_cast<const float4*>(base + boff[j] + 4 * (c ^ bsw[j]));
    }
  };
  auto mfma_slice = [&](const float4 (&xa)[4][WM], const float4 (&xb)[4][WN], int q4) {
    if constexpr (BF) {
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              __builtin_bit_cast(bf16x8, xa[q4][i]), __builtin_bit_cast(bf16x8, xb[q4][j]),
              acc[i][j], 0, 0, 0);
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int j = 0; j < WN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xa[q4][i][s], xb[q4][j][s],
                                                             acc[i][j], 0, 0, 0);
    }
  };
  // stage 0: at most the S-1 newer stages may still be in flight
  if (S - 1 < nk) wait_vmcnt<(S - 1) * Cfg::L>();
  else wait_vmcnt<0>();
  stage_barrier();
  read_frags(0, fa[0], fb[0]);
  constexpr int U = S % 2 == 0 ? S : 2 * S;
  for (int kt0 = 0; kt0 + 1 < nk; kt0 += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kt = kt0 + u;
      if (kt + 1 < nk) {
        const int cur = u % 2, nxt = 1 - u % 2;
        mfma_slice(fa[cur], fb[cur], 0);
        mfma_slice(fa[cur], fb[cur], 1);
        __builtin_amdgcn_sched_barrier(0);  // the first half's MFMAs stay ahead of the barrier
        // stage kt+1 is complete for this wave once at most the S-2 newer stages are outstanding
        if (kt + S - 1 < nk) wait_vmcnt<(S - 2) * Cfg::L>();
        else wait_vmcnt<0>();
        stage_barrier();  // ... and for every wave; every wave's reads of stage kt are done
        if (kt + S < nk) issue(kt + S, u % S);  // stage kt+S goes to the slot stage kt frees
        read_frags((u + 1) % S, fa[nxt], fb[nxt]);
        mfma_slice(fa[cur], fb[cur], 2);
        mfma_slice(fa[cur], fb[cur], 3);
        // fragment reads alternate with the first MFMAs of the second half, so the last read has
        // the remaining MFMAs to complete before the next stage needs it
        constexpr int kReads = 4 * (WM + WN), kMfma = 8 * WM * WN;
        if constexpr (BF) {
          // bf16: one MFMA per fragment pair and k step, 2 * WM * WN in the second half; the
          // reads are spread over them
          constexpr int kM = 2 * WM * WN, kR = (kReads + kM - 1) / kM;
#pragma unroll
          for (int r = 0; r < kM; ++r) {
            __builtin_amdgcn_sched_group_barrier(0x100, kR, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          }
        } else {
#pragma unroll
          for (int r = 0; r < kReads; ++r) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
          }
          __builtin_amdgcn_sched_group_barrier(0x008, kMfma, 0);
        }
      }
    }
  }
  // last stage: its fragments are in set (nk - 1) % 2 (moved to set 0 once, so a single copy of
  // the MFMAs owns the accumulators)
  if ((nk - 1) & 1) {
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
#pragma unroll
      for (int i = 0; i < WM; ++i) fa[0][q4][i] = fa[1][q4][i];
#pragma unroll
      for (int j = 0; j < WN; ++j) fb[0][q4][j] = fb[1][q4][j];
    }
  }
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4) mfma_slice(fa[0], fb[0], q4);

  // ---------------------------------------------------------------- epilogue
  // The activation and residual form are uniform: one specialised copy of the store loop each
  // for the forms the transformer uses, a generic one for the rest.
  const bool res = a.R != nullptr, bm = a.bias_mode == BIAS_M;
  // row-ordered stores through LDS where rows are 16-byte aligned (see store_tile_lds)
  const bool rows16 = (a.N % 4 == 0) && (a.ldc % 4 == 0) && (a.sC % 4 == 0) &&
                      ((reinterpret_cast<uintptr_t>(a.C) & 15) == 0) &&
                      (!res || ((a.ldr % 4 == 0) && (a.sR % 4 == 0) &&
                                (reinterpret_cast<uintptr_t>(a.R) & 15) == 0)) &&
                      (a.bias_mode != BIAS_N || (reinterpret_cast<uintptr_t>(a.bias) & 15) == 0) &&
                      (!a.rscale || (reinterpret_cast<uintptr_t>(a.rscale) & 15) == 0);
  if constexpr (EPI == 0) {
    if (rows16 && !bm) {
      __syncthreads();  // every wave's last fragment reads of the LDS ring are done
      const float2 lnc = ln_row_merge(a, lnr);
      if (a.act == 0 && !res)
        store_tile_lds<WMW, WNW, WM, WN, 0, false, S * STAGE>(a, acc, m0, n0, wm, wn, lane, smem,
                                                              lnc);
      else if (a.act == 0)
        store_tile_lds<WMW, WNW, WM, WN, 0, true, S * STAGE>(a, acc, m0, n0, wm, wn, lane, smem,
                                                             lnc);
      else if (a.act == 3 && !res)
        store_tile_lds<WMW, WNW, WM, WN, 3, false, S * STAGE>(a, acc, m0, n0, wm, wn, lane, smem,
                                                              lnc);
      else
        store_tile_lds<WMW, WNW, WM, WN, -1, true, S * STAGE>(a, acc, m0, n0, wm, wn, lane, smem,
                                                              lnc);
      return;
    }
  }
  if constexpr (EPI == 1) store_glu<WMW, WNW, WM, WN>(a, acc, m0, n0, wm, wn, lane);
  else if constexpr (EPI == 3) store_part<WMW, WNW, WM, WN>(a, acc, m0, n0, wm, wn, lane);
  else if (a.act == 0 && !res && !bm)
    store_tile<WMW, WNW, WM, WN, 0, false, true>(a, acc, m0, n0, wm, wn, lane);
  else if (a.act == 0 && !bm)
    store_tile<WMW, WNW, WM, WN, 0, true, false>(a, acc, m0, n0, wm, wn, lane);
  else if (a.act == 3 && !res && !bm)
    store_tile<WMW, WNW, WM, WN, 3, false, true>(a, acc, m0, n0, wm, wn, lane);
  else store_tile<WMW, WNW, WM, WN, -1, true, false>(a, acc, m0, n0, wm, wn, lane);
}

struct LdsTile {
  int id, bm, bn;
  double eff;  // relative matrix-core efficiency of the tile shape (measured)
};
constexpr LdsTile kLdsTiles[] = {
    {0, 128, 128, 1.00},  // <2,2,2,2> S2, 64 KB LDS, 2 workgroups per CU
    {1, 128, 64, 0.93},   // <2,2,2,1> S3
    {2, 64, 128, 0.93},   // <2,2,1,2> S3
    {3, 64, 64, 0.88},    // <2,2,1,1> S4
};

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int forced_lds_tile() {
  static const int v = [] {
    const char* e = std::getenv("MNN_GEMM_LDS_TILE");
    return e ? std::atoi(e) : -1;
  }();
  return v;
}

// Per-CU critical path: the most tiles any CU runs x tile area / shape efficiency. A CU that holds a
// single workgroup runs it at about 0.6 of the rate of two co-resident ones (the issuing wave waits
// for each LDS-DMA load to be accepted, and no other workgroup's MFMAs fill those cycles; measured on
// the transformer shapes), so a grid of at most one tile per CU is charged 1/0.6.
const LdsTile& choose_lds_tile(const GemmArgs& a) {
  const int f = forced_lds_tile();
  if (f >= 0 && f < (int)(sizeof(kLdsTiles) / sizeof(kLdsTiles[0]))) return kLdsTiles[f];
  const LdsTile* best = &kLdsTiles[0];
  double best_cost = 1e300;
  for (const LdsTile& t : kLdsTiles) {
    const int64_t tiles = (int64_t)cdiv(a.M, t.bm) * cdiv(a.N, t.bn) * a.batch * a.ksplit;
    const int64_t per_cu = cdiv(tiles, (int64_t)256);
    const double cost = (double)per_cu * t.bm * t.bn / t.eff / (per_cu == 1 ? 0.6 : 1.0);
    if (cost < best_cost * 0.999) {
      best_cost = cost;
      best = &t;
    }
  }
  return *best;
}

template <int WMW, int WNW, int WM, int WN, int S, bool BF = false>
void launch_lds(const LaunchCtx& c, const GemmArgs& a) {
  using Cfg = LdsCfg<WMW, WNW, WM, WN, S>;
  dim3 grid(cdiv(a.N, Cfg::BN), cdiv(a.M, Cfg::BM), a.batch * a.ksplit), block(Cfg::NT);
  if constexpr (BF) {  // bf16 operands: bias / activation / residual epilogue only
    launch(c, a.name ? a.name : "gemm_bf16_mfma_nk",
           gemm_nk_lds_kernel<WMW, WNW, WM, WN, S, 0, true>, grid, block, 0, a);
  } else {
    const char* name = a.name ? a.name : "gemm_f32_mfma_nk";
    if (a.ksplit > 1)
      launch(c, name, gemm_nk_lds_kernel<WMW, WNW, WM, WN, S, 3>, grid, block, 0, a);
    else if (a.glu) launch(c, name, gemm_nk_lds_kernel<WMW, WNW, WM, WN, S, 1>, grid, block, 0, a);
    else launch(c, name, gemm_nk_lds_kernel<WMW, WNW, WM, WN, S, 0>, grid, block, 0, a);
  }
}

}  // namespace

namespace {
// The folded-LayerNorm and row-statistics epilogue forms exist in the row-ordered store only:
// the conditions under which the kernel takes it (fp32, plain epilogue, 16-byte aligned rows),
// batch 1, and whole 64-column groups.
bool ln_fold_epilogue_ok(const GemmArgs& a) {
  const bool res = a.R != nullptr;
  const bool rows16 = a.N % 4 == 0 && a.ldc % 4 == 0 && aligned16(a.C) &&
                      (!res || (a.ldr % 4 == 0 && aligned16(a.R))) &&
                      (a.bias_mode != BIAS_N || aligned16(a.bias)) &&
                      (!a.rscale || aligned16(a.rscale));
  return rows16 && a.batch == 1 && !a.ab_bf16 && !a.glu && a.ksplit == 1 &&
         a.bias_mode != BIAS_M &&
         (!a.ln_parts || (a.K % 64 == 0 && a.K <= 64 * kLnMaxParts && a.ln_c &&
                          aligned16(a.ln_c) && aligned16(a.ln_parts))) &&
         (!a.row_parts || (a.N % 64 == 0 && (reinterpret_cast<uintptr_t>(a.row_parts) & 7) == 0));
}
}  // namespace

bool gemm_nk_lds_supported(const GemmArgs& a) {
  if (a.ab_bf16) {
    // bf16 operands: 64 k per stage, rows 16-byte aligned (8 elements), plain epilogue
    const bool off32 = ((int64_t)(a.M - 1) * a.lda + a.K) * 2 < ((int64_t)1 << 32) &&
                       ((int64_t)(a.N - 1) * a.ldb + a.K) * 2 < ((int64_t)1 << 32);
    return off32 && a.blayout == B_NK && a.precision == MNN_PRECISION_BF16 &&
           a.K % (2 * BK) == 0 && a.lda % 8 == 0 && a.ldb % 8 == 0 && a.sA % 8 == 0 &&
           a.sB % 8 == 0 && aligned16(a.A) && aligned16(a.B) && a.stats == nullptr &&
           a.pro_coef == nullptr && a.pro_stats == nullptr && !a.glu && a.ct_stride == 0 &&
           a.ksplit == 1 && a.bias_mode != BIAS_M;
  }
  // per-lane load offsets are 32-bit byte offsets from the operand (batch) base
  const bool off32 = ((int64_t)(a.M - 1) * a.lda + a.K) * 4 < ((int64_t)1 << 32) &&
                     ((int64_t)(a.N - 1) * a.ldb + a.K) * 4 < ((int64_t)1 << 32);
  return off32 && a.blayout == B_NK && a.precision == MNN_PRECISION_F32 && a.K % BK == 0 &&
         a.lda % 4 == 0 && a.ldb % 4 == 0 && a.sA % 4 == 0 && a.sB % 4 == 0 && aligned16(a.A) &&
         aligned16(a.B) && a.pro_coef == nullptr && a.pro_stats == nullptr &&
         (!a.glu || (a.M % 32 == 0 && a.bias_mode != BIAS_N && a.R == nullptr && a.act == 0)) &&
         a.ct_stride == 0 && a.stats == nullptr &&
         a.ksplit >= 1 && (a.K / BK) % a.ksplit == 0 &&
         (a.ksplit == 1 || (a.ws != nullptr && !a.glu)) &&
         ((!a.ln_parts && !a.row_parts) || ln_fold_epilogue_ok(a));
}

void gemm_nk_lds(const LaunchCtx& c, const GemmArgs& a) {
  MNN_REQUIRE(gemm_nk_lds_supported(a), MNN_ERR_INVALID_ARGUMENT,
              "gemm_nk_lds: operands outside the LDS-DMA path's contract");
  if (a.ab_bf16) {
    // bf16: a stage holds 64 k, so its matrix work is an eighth of the fp32 kernel's while its
    // loads are as large: four-stage rings keep more load latency in flight. 128x128 tiles where
    // they fill the CUs, 64x64 tiles for grids of fewer than 256 of them.
    const int f = forced_lds_tile();
    const int64_t big = (int64_t)cdiv(a.M, 128) * cdiv(a.N, 128) * a.batch;
    if (f == 3 || (f < 0 && big < 256)) return launch_lds<2, 2, 1, 1, 4, true>(c, a);
    return launch_lds<2, 2, 2, 2, 4, true>(c, a);
  }
  if (gemm_x3_supported(a)) return gemm_x3(c, a);
  switch (choose_lds_tile(a).id) {
    case 0: return launch_lds<2, 2, 2, 2, 2>(c, a);
    case 1: return launch_lds<2, 2, 2, 1, 3>(c, a);
    case 2: return launch_lds<2, 2, 1, 2, 3>(c, a);
    default: return launch_lds<2, 2, 1, 1, 4>(c, a);
  }
}

}  // namespace k
}  // namespace mnn
