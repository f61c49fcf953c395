// fp32 GEMM C = epilogue(A * B^T) with fp32 results from bf16 matrix cores (x3.hpp): one operand
// is a weight, kept as three bf16 planes laid out when it was loaded; the other is fp32 activations,
// taken apart in registers. Everything else is k_gemm_lds.hip's: LDS-DMA staging in a ring of S
// stages of 32 k, XCD-aware tile order, the same epilogues (gemm_epilogue.hpp).
//
// What bounds it: the bf16 MFMAs, 24 per 64x64 wave block and 16 k (768 cycles), with the split of
// the activations (about 11 VALU instructions per pair, 88 per 32x16 fragment) and the LDS reads
// (4 bytes per activation, 6 per weight) underneath. The weights come split because splitting
// both operands would cost as many VALU cycles as there are MFMA cycles, and because a weight
// would be split again by every workgroup of its column. With two workgroups on a CU the loop keeps
// the matrix cores 90 % busy, and the chip then clocks it at 1.47 GHz (2.4 for fp32 MFMAs, 1.73 for
// bf16 MFMAs on registers alone): the energy of the products is the limit. Fp32 kernel -> this one:
// 4096^3 1050 -> 754 us (131 -> 182 TFLOP/s), 10752 x 1536 x 384 117 -> 70 us, 2048 x 2048 x 512
// 42 -> 27 us, 67 x 1536 x 384 9.3 -> 8.1 us.
//
// LDS of one stage: the activation rows [R][32 floats], 16-byte chunk c of row r at slot
// c ^ chunk_swizzle(r), then the weight rows [P][3 planes][32 bf16] of 192 bytes, chunk c of a
// plane at slot c ^ ((r / 4) mod 4): 16 consecutive rows at one chunk then cover the 64 banks once.
// MFMA step s (0, 1) of a stage takes k 16 s + 8 g .. + 7 from lane group g, for both operands.
#include "device_utils.hpp"
#include "gemm_epilogue.hpp"
#include "kernels.hpp"
#include "lds_dma.hpp"
#include "x3.hpp"

#include <type_traits>

namespace mnn {
namespace k {

using namespace dev;

namespace {

constexpr int BK = 32;

template <int WMW, int WNW, int WM, int WN, int S, bool WA>
struct X3Cfg {
  static constexpr int BM = WMW * WM * 32, BN = WNW * WN * 32;
  static constexpr int NW = WMW * WNW, NT = NW * 64;
  static constexpr int RB = WA ? BN : BM, PB = WA ? BM : BN;  // activation / weight rows of a tile
  static constexpr int R_INS = RB * 8 / 64 / NW, P_INS = PB * 12 / 64 / NW;
  static constexpr int L = R_INS + P_INS;  // loads per wave per stage
  static constexpr int STAGE = RB * 32 + PB * 48;  // floats
  static constexpr int OCC =
      NW > 4 ? NW / 4 : (2 * S * STAGE * 4 <= 160 * 1024 ? 2 : 1);  // waves per SIMD
  static_assert(RB * 8 % (64 * NW) == 0 && PB * 12 % (64 * NW) == 0, "loads split over waves");
  static_assert((S - 1) * L < 64, "vmcnt range");
  static_assert(S * STAGE * 4 <= 160 * 1024, "LDS");
};

// EPI as gemm_nk_lds_kernel's. WA: A is the weight (M the weight's rows), else B is.
template <int WMW, int WNW, int WM, int WN, int S, int EPI, bool WA>
__global__ __launch_bounds__(WMW* WNW * 64, (X3Cfg<WMW, WNW, WM, WN, S, WA>::OCC))
void gemm_x3_kernel(GemmArgs a) {
  using Cfg = X3Cfg<WMW, WNW, WM, WN, S, WA>;
  constexpr int BM = Cfg::BM, BN = Cfg::BN, RB = Cfg::RB;
  constexpr int R_INS = Cfg::R_INS, P_INS = Cfg::P_INS, STAGE = Cfg::STAGE, L = Cfg::L;
  constexpr int WR = WA ? WN : WM, WP = WA ? WM : WN;  // 32-row fragments of each operand
  __shared__ __attribute__((aligned(1024))) float smem[S * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WNW, wn = wave % WNW;
  const int wr = WA ? wn : wm, wp = WA ? wm : wn;
  // blockIdx.z = batch * ksplit + K part (ksplit = 1 unless EPI == 3)
  const int ks = EPI == 3 ? a.ksplit : 1;
  const int bz = blockIdx.z / ks;
  const int gx = gridDim.x;
  const int logical = xcd_logical_tile(blockIdx.x + gx * blockIdx.y, gx * gridDim.y);
  const int tn = logical % gx, tm = logical / gx;
  const int m0 = tm * BM, n0 = tn * BN;
  const int M = a.M, N = a.N, K = a.K;
  const int nk = K / BK / ks, kt0 = (int)(blockIdx.z % ks) * nk;
  LnRow lnr;
  if constexpr (EPI == 0) lnr = ln_row_load(a, m0 + tid % BM);
  // activations (fp32, row pitch ldr_) and weight planes (192 bytes per row and 32 k)
  const int64_t ldx = WA ? a.ldb : a.lda;
  const float* __restrict__ X =
      WA ? a.B + (int64_t)bz * a.sB : a.A + (int64_t)bz * a.sA;
  const int xr0 = WA ? n0 : m0, xrows = WA ? N : M, pr0 = WA ? m0 : n0, prows = WA ? M : N;

  // per-lane byte offsets of this wave's loads (rows past the end repeat the last one; their
  // products are never stored)
  unsigned roff[R_INS], poff[P_INS];
#pragma unroll
  for (int i = 0; i < R_INS; ++i) {
    const int rr = (wave * R_INS + i) * 8 + (lane >> 3);
    roff[i] = 4u * (unsigned)(min(xr0 + rr, xrows - 1) * (int)ldx) +
              16u * (unsigned)((lane & 7) ^ chunk_swizzle(rr));
  }
#pragma unroll
  for (int i = 0; i < P_INS; ++i) {
    const int e = (wave * P_INS + i) * 64 + lane, rr = e / 12, slot = e % 12;
    poff[i] = 6u * (unsigned)(min(pr0 + rr, prows - 1) * K) +
              16u * (unsigned)((slot & ~3) | ((slot & 3) ^ ((rr >> 2) & 3)));
  }
  const unsigned lds0 = lds_address(smem);
  auto issue = [&](int kt, int slot) {
    const unsigned base = lds0 + 4u * (unsigned)(slot * STAGE);
    const float* xk = X + (int64_t)(kt0 + kt) * BK;
    const float* pk = reinterpret_cast<const float*>(a.wplanes) + (int64_t)(kt0 + kt) * 48;
#pragma unroll
    for (int i = 0; i < R_INS; ++i)
      lds_dma16_s(xk, roff[i], __builtin_amdgcn_readfirstlane(base + 1024u * (wave * R_INS + i)));
#pragma unroll
    for (int i = 0; i < P_INS; ++i)
      lds_dma16_s(pk, poff[i], __builtin_amdgcn_readfirstlane(base + 4u * (RB * 32) +
                                                              1024u * (wave * P_INS + i)));
  };

  floatx16 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  const int g = lane >> 5, l32 = lane & 31;
  // LDS word offsets of this lane's fragment rows; chunk of step s: raw 4 s + 2 g + {0, 1},
  // planes 2 s + g
  int ro[WR], rsw[WR], po[WP];
#pragma unroll
  for (int i = 0; i < WR; ++i) {
    const int rr = wr * WR * 32 + 32 * i + l32;
    ro[i] = rr * 32;
    rsw[i] = chunk_swizzle(rr);
  }
  // slot of step s: (2 s + g) ^ f = (g ^ f) ^ 2 s
  int psw[WP];
#pragma unroll
  for (int j = 0; j < WP; ++j) {
    const int rr = wp * WP * 32 + 32 * j + l32;
    po[j] = RB * 32 + rr * 48;
    psw[j] = g ^ ((rr >> 2) & 3);
  }
  // Software pipeline over steps of 16 k, two per stage. While the MFMAs of step t run, the wave
  // splits step t+1's activations (read during step t-1), reads step t+1's weight parts and, from
  // the middle of the step on, step t+2's activations. By the middle of a stage's first step every
  // read of that stage has been issued: the one barrier of the stage stands there, makes the next
  // stage visible and frees this one's slot for stage kt + S.
  float4 raw[2][WR][2];
  Split8 xs[2][WR], pl[2][WP];
  auto read_raw = [&](const float* base, int s) {
#pragma unroll
    for (int i = 0; i < WR; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        raw[s][i][h] = *reinterpret_cast<const float4*>(base + ro[i] +
                                                        4 * ((4 * s + 2 * g + h) ^ rsw[i]));
  };
  auto read_planes = [&](const float* base, int s) {
#pragma unroll
    for (int j = 0; j < WP; ++j) {
      const float* p = base + po[j] + 4 * (psw[j] ^ (2 * s));
      pl[s][j].h = *reinterpret_cast<const bf16x8*>(p);
      pl[s][j].m = *reinterpret_cast<const bf16x8*>(p + 16);
      pl[s][j].l = *reinterpret_cast<const bf16x8*>(p + 32);
    }
  };
  auto split = [&](int s) {
#pragma unroll
    for (int i = 0; i < WR; ++i)
      xs[s][i] = split8_trunc(reinterpret_cast<const float*>(&raw[s][i][0]));
  };
  auto products = [&](int s, int p0, int p1) {
#pragma unroll
    for (int p = p0; p < p1; ++p)
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
          acc[i][j] = WA ? mfma_x3(pl[s][i], xs[s][j], acc[i][j], p)
                         : mfma_x3(xs[s][i], pl[s][j], acc[i][j], p);
  };
  // n MFMAs with kV VALU instructions behind each
  auto interleave = [&](auto nc) {
    constexpr int kV = (88 * WR / 2 + 6 * WM * WN - 1) / (6 * WM * WN);
#pragma unroll
    for (int r = 0; r < decltype(nc)::value; ++r) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, kV, 0);
    }
  };
  constexpr std::integral_constant<int, 3 * WM * WN> kHalf{};
  constexpr std::integral_constant<int, 6 * WM * WN> kAll{};

#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < nk) issue(s, s);
  if (S - 1 < nk) wait_vmcnt<(S - 1) * L>();
  else wait_vmcnt<0>();
  stage_barrier();
  read_raw(smem, 0);
  read_planes(smem, 0);
  read_raw(smem, 1);
  split(0);
  for (int kb = 0; kb + 1 < nk; kb += S) {
#pragma unroll
    for (int u = 0; u < S; ++u) {
      const int kt = kb + u;
      if (kt + 1 < nk) {
        const float* here = smem + u * STAGE;
        const float* next = smem + (u + 1) % S * STAGE;
        __builtin_amdgcn_sched_barrier(0);
        read_planes(here, 1);
        split(1);
        products(0, 0, 3);
        interleave(kHalf);
        __builtin_amdgcn_sched_barrier(0);
        wait_lgkmcnt0();  // this wave's reads of stage kt are done
        if (kt + S - 1 < nk) wait_vmcnt<(S - 2) * L>();
        else wait_vmcnt<0>();
        stage_barrier();  // stage kt + 1 is whole, stage kt's slot is free
        if (kt + S < nk) issue(kt + S, u);
        read_raw(next, 0);
        products(0, 3, 6);
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * WR, 0);  // the reads first
        __builtin_amdgcn_sched_group_barrier(0x008, kHalf, 0);
        __builtin_amdgcn_sched_barrier(0);
        read_planes(next, 0);
        split(0);
        products(1, 0, 6);
        read_raw(next, 1);
        interleave(kAll);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  {
    read_planes(smem + (nk - 1) % S * STAGE, 1);
    split(1);
    products(0, 0, 6);
    products(1, 0, 6);
  }

  // Not finite somewhere: this wave's block again in fp32, straight from memory (the parts of a
  // weight sum to it).
  if (any_not_finite(acc)) {
    const unsigned short* W = reinterpret_cast<const unsigned short*>(a.wplanes);
    auto weight = [&](int row, int k) {
      const unsigned short* p = W + ((int64_t)min(row, prows - 1) * (K / 32) + k / 32) * 96 + k % 32;
      auto f = [](unsigned short b) { return __builtin_bit_cast(float, (unsigned)b << 16); };
      return f(p[0]) + (f(p[32]) + f(p[64]));
    };
    auto act = [&](int row, int k) { return X[(int64_t)min(row, xrows - 1) * ldx + k]; };
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    const int rm = m0 + wm * WM * 32 + l32, rn = n0 + wn * WN * 32 + l32;
#pragma unroll 1
    for (int k = kt0 * BK + g; k < (kt0 + nk) * BK; k += 2) {
      float fa[WM], fb[WN];
#pragma unroll
      for (int i = 0; i < WM; ++i) fa[i] = WA ? weight(rm + 32 * i, k) : act(rm + 32 * i, k);
#pragma unroll
      for (int j = 0; j < WN; ++j) fb[j] = WA ? act(rn + 32 * j, k) : weight(rn + 32 * j, k);
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
  }

  // ---------------------------------------------------------------- epilogue
  if constexpr (EPI == 1) {
    store_glu<WMW, WNW, WM, WN>(a, acc, m0, n0, wm, wn, lane);
  } else if constexpr (EPI == 2) {
    __syncthreads();  // every wave's last fragment reads of the LDS ring are done
    store_ct<WMW, WNW, WM, WN>(a, acc, m0, n0, wm, wn, lane, smem);
  } else if constexpr (EPI == 3) {
    store_part<WMW, WNW, WM, WN>(a, acc, m0, n0, wm, wn, lane);
  } else {
    const bool res = a.R != nullptr, bm = a.bias_mode == BIAS_M;
    const bool rows16 = (a.N % 4 == 0) && (a.ldc % 4 == 0) && (a.sC % 4 == 0) &&
                        ((reinterpret_cast<uintptr_t>(a.C) & 15) == 0) &&
                        (!res || ((a.ldr % 4 == 0) && (a.sR % 4 == 0) &&
                                  (reinterpret_cast<uintptr_t>(a.R) & 15) == 0)) &&
                        (a.bias_mode != BIAS_N || (reinterpret_cast<uintptr_t>(a.bias) & 15) == 0) &&
                        (!a.rscale || (reinterpret_cast<uintptr_t>(a.rscale) & 15) == 0);
    if (rows16 && !bm) {
      __syncthreads();  // every wave's last fragment reads of the LDS ring are done
      if (a.act == 0 && !res)
        store_tile_lds<WMW, WNW, WM, WN, 0, false, S * STAGE>(a, acc, m0, n0, wm, wn, lane, smem,
                                                              lnr);
      else if (a.act == 0)
        store_tile_lds<WMW, WNW, WM, WN, 0, true, S * STAGE>(a, acc, m0, n0, wm, wn, lane, smem,
                                                             lnr);
      else if (a.act == 3 && !res)
        store_tile_lds<WMW, WNW, WM, WN, 3, false, S * STAGE>(a, acc, m0, n0, wm, wn, lane, smem,
                                                              lnr);
      else
        store_tile_lds<WMW, WNW, WM, WN, -1, true, S * STAGE>(a, acc, m0, n0, wm, wn, lane, smem,
                                                              lnr);
      return;
    }
    if (a.act == 0 && !res && !bm)
      store_tile<WMW, WNW, WM, WN, 0, false, true>(a, acc, m0, n0, wm, wn, lane);
    else store_tile<WMW, WNW, WM, WN, -1, true, false>(a, acc, m0, n0, wm, wn, lane);
  }
}

// planes[row][k / 32][part][k % 32] of a [rows][K] weight, eight k per thread.
__global__ __launch_bounds__(256) void x3_planes_kernel(const float* __restrict__ w,
                                                        unsigned short* __restrict__ out,
                                                        int64_t n8, int K) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const int64_t row = i / (K / 8);
  const int k = 8 * (int)(i % (K / 8));
  unsigned short* o = out + (row * (K / 32) + k / 32) * 96 + k % 32;
  bf16x8 h, m, l;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    __bf16 a, b, c;
    split_weight(w[row * K + k + e], a, b, c);
    h[e] = a;
    m[e] = b;
    l[e] = c;
  }
  *reinterpret_cast<bf16x8*>(o) = h;
  *reinterpret_cast<bf16x8*>(o + 32) = m;
  *reinterpret_cast<bf16x8*>(o + 64) = l;
}

// Output tiles, named by activation rows x weight rows (M x N where B is the weight, N x M where A
// is). eff: relative matrix-core rate of the shape, measured over the transformer's GEMMs (us,
// 128x128 / 64x128 / 64x64): 10752x1536x384 70 / 76 / 94, 5376x1152x384 34 / 31 / 38,
// 2048x2048x512 29 / 27 / 34, 5376x384x1536 62 / 41 / 43, 1000x384x384 17 / 11 / 8.6 (the fp32
// kernel: 117, 48, 42, 57, 9.9). 128 activation rows by 64 weight rows were behind 64x128 at every
// shape (half the products per split value), 256x128 ahead only from about 4096^3 on.
struct X3Tile {
  int id, rb, pb;
  double eff;
};
constexpr X3Tile kX3Tiles[] = {{0, 128, 128, 1.00}, {1, 64, 128, 0.95}, {2, 64, 64, 0.70}};

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int forced_x3_tile() {
  static const int v = [] {
    const char* e = std::getenv("MNN_GEMM_LDS_TILE");
    return e ? std::atoi(e) : -1;
  }();
  return v;
}

int64_t x3_tiles(const GemmArgs& a, const X3Tile& t) {
  return (int64_t)cdiv(a.wa ? a.N : a.M, t.rb) * cdiv(a.wa ? a.M : a.N, t.pb);
}

// Per-CU critical path as in the fp32 kernel's chooser; a workgroup alone on its CU runs at about
// 0.8 of the rate of two (2450 against 3420 / 2 cycles per stage of a 128x128 tile).
const X3Tile& choose_x3_tile(const GemmArgs& a) {
  const int f = forced_x3_tile();
  if (f >= 0 && f < (int)(sizeof(kX3Tiles) / sizeof(kX3Tiles[0]))) return kX3Tiles[f];
  const X3Tile* best = &kX3Tiles[0];
  double best_cost = 1e300;
  for (const X3Tile& t : kX3Tiles) {
    const int64_t per_cu = cdiv(x3_tiles(a, t) * a.batch * a.ksplit, (int64_t)256);
    const double cost = (double)per_cu * t.rb * t.pb / t.eff / (per_cu == 1 ? 0.8 : 1.0);
    if (cost < best_cost * 0.999) {
      best_cost = cost;
      best = &t;
    }
  }
  return *best;
}

// WR x WP 32-row blocks (activations x weights) per wave, 2 x 2 waves.
template <int WR, int WP, int S>
void launch_x3(const LaunchCtx& c, const GemmArgs& a) {
  const dim3 block(256);
  const char* name = a.name ? a.name : "gemm_f32_mfma_nk";
  if (!a.wa) {
    const dim3 grid(cdiv(a.N, WP * 64), cdiv(a.M, WR * 64), a.batch);
    return launch(c, name, gemm_x3_kernel<2, 2, WR, WP, S, 0, false>, grid, block, 0, a);
  }
  const dim3 grid(cdiv(a.N, WR * 64), cdiv(a.M, WP * 64), a.batch * a.ksplit);
  if (a.ksplit > 1)
    launch(c, name, gemm_x3_kernel<2, 2, WP, WR, S, 3, true>, grid, block, 0, a);
  else if (a.glu) launch(c, name, gemm_x3_kernel<2, 2, WP, WR, S, 1, true>, grid, block, 0, a);
  else launch(c, name, gemm_x3_kernel<2, 2, WP, WR, S, 2, true>, grid, block, 0, a);
}

}  // namespace

int64_t x3_planes_bytes(int64_t rows, int64_t K) { return rows * K * 6; }

void x3_planes(const LaunchCtx& c, const float* w, int64_t rows, int64_t K, void* out) {
  MNN_REQUIRE(K % BK == 0 && K < (1 << 30) && rows > 0, MNN_ERR_INVALID_ARGUMENT,
              "x3_planes: the depth must be a multiple of 32");
  const int64_t n8 = rows * K / 8;
  launch(c, "x3_planes", x3_planes_kernel, dim3(cdiv(n8, 256)), dim3(256), 0, w,
         static_cast<unsigned short*>(out), n8, (int)K);
}

bool gemm_x3_supported(const GemmArgs& a) {
  if (!a.wplanes || a.ab_bf16 || a.blayout != B_NK || !aligned16(a.wplanes)) return false;
  // per-lane load offsets are 32-bit byte offsets
  const int64_t wrows = a.wa ? a.M : a.N;
  const bool off32 = x3_planes_bytes(wrows, a.K) < ((int64_t)1 << 32);
  // the weight is the same for every batch, its rows are K apart
  if ((a.wa ? a.sA : a.sB) != 0 || (a.wa ? a.lda : a.ldb) != a.K) return false;
  // the forms that are built: plain epilogue over activations x weights, GLU / transposed conv /
  // K parts over weights x activations
  const bool rows = a.glu || a.ct_stride > 0 || a.ksplit > 1;
  return off32 && rows == a.wa;
}

int64_t gemm_x3_tiles(const GemmArgs& a) { return x3_tiles(a, choose_x3_tile(a)); }

void gemm_x3(const LaunchCtx& c, const GemmArgs& a) {
  switch (choose_x3_tile(a).id) {
    case 0: return launch_x3<2, 2, 2>(c, a);
    case 1: return launch_x3<1, 2, 2>(c, a);
    default: return launch_x3<1, 1, 3>(c, a);
  }
}

}  // namespace k
}  // namespace mnn
