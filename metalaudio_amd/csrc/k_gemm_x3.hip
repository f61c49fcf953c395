// fp32 GEMM C = epilogue(A * B^T) with fp32 results from bf16 matrix cores (x3.hpp): one operand
// is a weight, kept as three bf16 planes laid out when it was loaded; the other is fp32 activations,
// taken apart in registers. Everything else is k_gemm_lds.hip's: LDS-DMA staging in a ring of S
// stages of 32 k, XCD-aware tile order, the same epilogues (gemm_epilogue.hpp).
//
// What bounds it: the bf16 MFMAs, 24 per 64x64 wave block and 16 k (768 cycles), with the split of
// the activations (11 VALU instructions per pair, 44 per 32x16 fragment) and the LDS reads
// (4 bytes per activation, 6 per weight) underneath. The weights come split because splitting
// both operands would cost as many VALU cycles as there are MFMA cycles, and because a weight
// would be split again by every workgroup of its column. With two workgroups on a CU the 128x128 loop
// keeps the matrix cores 90 % busy, and the chip then clocks it at 1.47 GHz (2.4 for fp32 MFMAs, 1.73 for
// bf16 MFMAs on registers alone): the energy of the products is the limit. Small tiles are bound by the
// split: a wave of a 64x64 tile has 6 MFMAs (192 cycles) and one fragment's 44 instructions (about 200
// cycles, 52 instructions with the taps' masks) per 16 k. Fp32 kernel -> this one: 4096^3 1050 -> 700 us
// (131 -> 196 TFLOP/s), 10752 x 1536 x 384 117 -> 71 us, 2048 x 2048 x 512 42 -> 28.6 us, 67 x 1536 x 384
// 9.3 -> 8.0 us.
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
constexpr int kLongRow = 1 << 25;  // 32 rows of fewer samples lie within 4 GiB

// How the fp32 operand lies in memory (GemmArgs::raw_mode).
//   RAW_ROWS  rows [row][K], K contiguous.
//   RAW_TAPS  [channel][position] rows of length ldb (two matrices: channels below kc1 from B, the
//             others from B2) read at TT taps: k = (block of 32 / TT channels, tap, channel of the block)
//             and element (k, n) is position n - tap of the channel, zero outside [0, ldb): the operand
//             of a transposed conv, with no unfolded copy. A stage is one block of channels with a
//             window of R + TT - 1 positions, whose taps the fragment reads pick by their column (a
//             window per tap was 35 % slower: rows at odd positions make every 16-byte copy two
//             requests). Windows start at the last 16-byte boundary of memory before their first
//             position, w = (alignment of the row - (TT - 1)) mod 4 positions earlier; rows four apart
//             have the same w, so it is four scalars per stage. Row pitch R + 4 (two taps): the two lane
//             groups, 8 rows apart, read opposite halves of the banks. One tap: windows of R positions
//             as they are, chunk c of row r at c ^ 8 * ((r / 8) mod 2) for the same reason.
//   RAW_CONV  [channel][sample] rows of length ldb, k = (channel, 8 taps) of the stride-4 conv: element
//             (k, n) is sample 4 n - conv_pad + tap, reflected or zero outside. A stage holds 4
//             channels' windows of R + 1 chunks of 4 samples; the 8 taps of a column are two chunks.
// Chunks that cross an end of the signal are loaded clamped to its first / last 4 samples and rewritten
// in LDS by the lane that loaded them (tiles at an end only).
template <int WMW, int WNW, int WM, int WN, int S, bool WA, int RAW, int TT>
struct X3Cfg {
  static constexpr int BM = WMW * WM * 32, BN = WNW * WN * 32;
  static constexpr int NW = WMW * WNW, NT = NW * 64;
  static constexpr int RB = WA ? BN : BM, PB = WA ? BM : BN;  // activation / weight rows of a tile
  static constexpr int WCH = RB + 1;                          // RAW_CONV: chunks per channel window
  static constexpr int CR = 32 / TT;                          // RAW_TAPS: channels a stage,
  static constexpr int CPW = RB / 4 + TT / 2;                 //   chunks per channel window
  static constexpr int R_CH = RAW == RAW_CONV ? 4 * WCH : RAW == RAW_TAPS ? CR * CPW : RB * 8;
  static constexpr int R_WL = (R_CH + 63) / 64;               // wave loads a stage
  static constexpr int P_WL = PB * 12 / 64;
  static constexpr int T = R_WL + P_WL;
  static constexpr int L = (T + NW - 1) / NW;  // per wave (waves >= T % NW have one fewer)
  static constexpr int RF = R_WL * 256;        // floats of the activations' part of a stage
  static constexpr int STAGE = RF + PB * 48;   // floats
  static constexpr int OCC = 2 * S * STAGE * 4 <= 160 * 1024 ? 2 : 1;  // workgroups per CU
  static_assert(NW == 4 && PB * 12 % 64 == 0 && RB % 8 == 0, "whole wave loads");
  static_assert(RAW != RAW_TAPS || RB >= 64, "two lane groups on opposite bank halves");
  static_assert((S - 1) * L < 64, "vmcnt range");
  static_assert(S * STAGE * 4 <= 160 * 1024, "LDS");
};

// Value of position p of a signal of L samples from the 4 samples of the clamped chunk at q0.
__device__ __forceinline__ float edge_sample(const float4& v, int p, int q0, int L, bool reflect) {
  int q = p;
  if (reflect) {
    q = q < 0 ? -q : q;
    q = q > L - 1 ? 2 * (L - 1) - q : q;
  } else if (p < 0 || p > L - 1) {
    return 0.f;
  }
  const int i = min(max(q - q0, 0), 3);  // outside 0..3 only for samples no stored column uses
  return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
}

// TM = 2: two teams of four waves, each with a ring of its own and half of the K stages (an even
// number), whose sums the first team adds up and stores.
// EPI as gemm_nk_lds_kernel's, and 4: bias along M and, with a.stats, the GroupNorm(1) partial of the
// tile (store_rows_stats). WA: A is the weight (M the weight's rows), else B is.
template <int WMW, int WNW, int WM, int WN, int S, int EPI, bool WA, int RAW, int TT = 1, int TM = 1>
__global__ __launch_bounds__(WMW* WNW * 64 * TM, (X3Cfg<WMW, WNW, WM, WN, S, WA, RAW, TT>::OCC))
void gemm_x3_kernel(GemmArgs a) {
  using Cfg = X3Cfg<WMW, WNW, WM, WN, S, WA, RAW, TT>;
  constexpr int BM = Cfg::BM, BN = Cfg::BN, RB = Cfg::RB, RF = Cfg::RF, NW = Cfg::NW;
  constexpr int R_WL = Cfg::R_WL, T = Cfg::T, STAGE = Cfg::STAGE, L = Cfg::L, WCH = Cfg::WCH;
  constexpr int CR = Cfg::CR, CPW = Cfg::CPW;
  constexpr int WR = WA ? WN : WM, WP = WA ? WM : WN;  // 32-row fragments of each operand
  static_assert(RAW == RAW_ROWS || WA, "channel-major activations are B");
  __shared__ __attribute__((aligned(1024))) float smem_all[TM * S * STAGE];

  const int tid = threadIdx.x % (NW * 64), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int team = TM == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / (NW * 64));
  float* const smem = smem_all + team * (S * STAGE);
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
  const int nk = K / BK / ks / TM, kt0 = ((int)(blockIdx.z % ks) * TM + team) * nk;
  constexpr bool kFold = EPI == 0 && !WA;  // a folded LayerNorm is one of the activations
  LnRow lnr;
  if constexpr (kFold) lnr = ln_row_load(a, m0 + tid % BM);
  const int64_t ldx = WA ? a.ldb : a.lda;
  const float* __restrict__ X =
      WA ? a.B + (int64_t)bz * a.sB : a.A + (int64_t)bz * a.sA;
  const float* X2 = RAW == RAW_TAPS && a.B2 ? a.B2 + (int64_t)bz * a.sB2 : X;
  const int xr0 = WA ? n0 : m0, xrows = WA ? N : M, pr0 = WA ? m0 : n0, prows = WA ? M : N;
  const int Ls = (int)ldx;  // RAW_TAPS / RAW_CONV: samples per channel

  // Wave load j = i * NW + wave of a stage: activations (j < R_WL), then weights. Per-lane byte
  // offsets from the stage's scalar bases; rows past the end repeat the last one (their products
  // are never stored).
  // (is_raw / is_weight: constant for most i once the loops are unrolled)
  auto is_raw = [&](int i) { return i * NW + NW <= R_WL || (i * NW < R_WL && i * NW + wave < R_WL); };
  auto is_weight = [&](int i) { return i * NW + NW <= T || i * NW + wave < T; };
  unsigned off[L];
  int pos[L], row[L];  // channel-major modes: first position of the lane's chunk, channel of the stage
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int j = i * NW + wave;
    off[i] = 0;
    pos[i] = row[i] = 0;
    if (j < R_WL) {
      if constexpr (RAW == RAW_ROWS) {
        const int rr = j * 8 + (lane >> 3);
        off[i] = 4u * (unsigned)(min(xr0 + rr, xrows - 1) * (int)ldx) +
                 16u * (unsigned)((lane & 7) ^ chunk_swizzle(rr));
      } else if constexpr (RAW == RAW_TAPS) {
        const int e = min(j * 64 + lane, Cfg::R_CH - 1);  // past the windows: the last chunk again
        row[i] = e / CPW;
        const int ch = TT == 1 ? (e % CPW) ^ (8 * ((row[i] >> 3) & 1)) : e % CPW;
        pos[i] = n0 - (TT - 1) + 4 * ch;
        off[i] = (unsigned)row[i] * (unsigned)Ls;  // floats
      } else {
        const int e = min(j * 64 + lane, 4 * WCH - 1);  // past the windows: the last chunk again
        row[i] = e / WCH;
        pos[i] = 4 * n0 - a.conv_pad + 4 * (e % WCH);
        off[i] = 4u * (unsigned)(row[i] * Ls + min(max(pos[i], 0), Ls - 4));
      }
    } else {
      const int e = (j - R_WL) * 64 + lane, rr = e / 12, slot = e % 12;
      off[i] = 6u * (unsigned)(min(pr0 + rr, prows - 1) * K) +
               16u * (unsigned)((slot & ~3) | ((slot & 3) ^ ((rr >> 2) & 3)));
    }
  }
  // RAW_TAPS: a stage's channels come from one matrix (a scalar base) or, across the two or past the
  // last channel (whose weights are zero), from an address per lane. Row r's window starts
  // w = (align0 + r * ldb) mod 4 positions before its first (off holds r * ldb).
  // Whole stages of 16-byte aligned chunks (shifted) may read up to 3 floats before and past a row,
  // within the 16 bytes of its first or last sample: the fragment reads mask those columns. Other
  // stages (one tap: rows that are no whole chunks, or too long for a stage's 32-bit offsets) clamp
  // their chunks into the row and rewrite them in LDS.
  const bool shifted = TT > 1 || (Ls % 4 == 0 && Ls < kLongRow);
  struct Taps {
    int c0;
    bool first, second;
    const float* x;
    int align0;
    __device__ bool whole() const { return first || second; }
  };
  auto taps = [&](int kt) {
    Taps t;
    t.c0 = kt * CR;
    t.first = shifted && t.c0 + CR <= a.kc1;
    t.second = shifted && t.c0 >= a.kc1 && t.c0 + CR <= a.kvalid;
    t.x = t.second ? X2 + (int64_t)(t.c0 - a.kc1) * Ls : X + (int64_t)t.c0 * Ls;
    t.align0 = (int)((unsigned)reinterpret_cast<uintptr_t>(t.x) >> 2) - (TT - 1);
    return t;
  };
  // tiles whose windows cross an end of the signal
  const bool reflect = RAW == RAW_CONV && a.conv_reflect;
  const bool edge = RAW == RAW_CONV   ? 4 * n0 - a.conv_pad < 0 ||
                                            4 * (n0 + RB) - a.conv_pad + 3 > Ls - 1
                    : RAW == RAW_TAPS ? n0 < 8 || n0 + RB + 8 > Ls
                                      : false;
  const unsigned lds0 = lds_address(smem);
  auto issue = [&](int kl, int slot) {
    const int kt = kt0 + kl;
    const unsigned base = lds0 + 4u * (unsigned)(slot * STAGE);
    const float* pk = reinterpret_cast<const float*>(a.wplanes) + (int64_t)kt * 48;
    auto weights = [&](int i, int j) {
      lds_dma16_s(pk, off[i], __builtin_amdgcn_readfirstlane(base + 1024u * j));
    };
    auto each = [&](auto raw_load) {
#pragma unroll
      for (int i = 0; i < L; ++i) {
        const int j = i * NW + wave;
        if (is_raw(i)) raw_load(i, (unsigned)__builtin_amdgcn_readfirstlane(base + 1024u * j));
        else if (is_weight(i)) weights(i, j);
      }
    };
    if constexpr (RAW == RAW_ROWS) {
      const float* xk = X + (int64_t)kt * BK;
      each([&](int i, unsigned dst) { lds_dma16_s(xk, off[i], dst); });
    } else if constexpr (RAW == RAW_TAPS) {
      const Taps tp = taps(kt);
      auto start = [&](int i) {
        return pos[i] - (TT == 1 ? 0 : (tp.align0 + (int)off[i]) & 3);
      };
      if (tp.whole() && !edge) {
        each([&](int i, unsigned dst) { lds_dma16_s(tp.x, 4u * (off[i] + (unsigned)start(i)), dst); });
      } else if (tp.whole()) {
        // chunks with no sample of the row: another one (their columns are masked)
        each([&](int i, unsigned dst) {
          int p = start(i);
          p = p <= -4 ? p + 4 : p;
          p -= max(p - Ls + 4, 0) & ~3;
          lds_dma16_s(tp.x - 4, 4u * (off[i] + (unsigned)(p + 4)), dst);
        });
      } else {
        each([&](int i, unsigned dst) {
          const int p = min(max(start(i), 0), Ls - 4);
          const int c = min(tp.c0 + row[i], a.kvalid - 1);
          lds_dma16((c < a.kc1 ? X + (int64_t)c * Ls : X2 + (int64_t)(c - a.kc1) * Ls) + p, dst);
        });
      }
    } else {
      const float* xk = X + (int64_t)(4 * kt) * Ls;
      if (4 * kt + 4 > a.kvalid)  // padded channels read the last real one
        each([&](int i, unsigned dst) {
          lds_dma16_s(xk,
                      4u * (unsigned)(min(row[i], a.kvalid - 1 - 4 * kt) * Ls +
                                      min(max(pos[i], 0), Ls - 4)),
                      dst);
        });
      else
        each([&](int i, unsigned dst) { lds_dma16_s(xk, off[i], dst); });
    }
  };
  // this lane's landed chunks of stage kl that cross an end of the signal, rewritten
  auto fix_edges = [&](int kl, int slot) {
    if constexpr (RAW != RAW_ROWS) {
      if (RAW == RAW_TAPS && taps(kt0 + kl).whole()) return;
      const int align0 = RAW == RAW_TAPS ? taps(kt0 + kl).align0 : 0;
#pragma unroll
      for (int i = 0; i < L; ++i) {
        const int j = i * NW + wave;
        const int p = pos[i] - (RAW == RAW_TAPS && TT > 1 ? (align0 + (int)off[i]) & 3 : 0);
        if (j < R_WL && (p < 0 || p + 3 > Ls - 1)) {
          float4* cp = reinterpret_cast<float4*>(smem + slot * STAGE + 4 * (j * 64 + lane));
          const float4 v = *cp;
          const int q0 = min(max(p, 0), Ls - 4);
          float4 r;
          r.x = edge_sample(v, p, q0, Ls, reflect);
          r.y = edge_sample(v, p + 1, q0, Ls, reflect);
          r.z = edge_sample(v, p + 2, q0, Ls, reflect);
          r.w = edge_sample(v, p + 3, q0, Ls, reflect);
          *cp = r;
        }
      }
      wait_lgkmcnt0();
    }
  };
  const bool full = T % NW == 0 || wave < T % NW;  // this wave has L loads a stage, else L - 1

  // h * h and the five smaller products apart (x3.hpp); added after the loop
  floatx16 acc[WM][WN], low[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = low[i][j][v] = 0.f;

  const int g = lane >> 5, l32 = lane & 31;
  // LDS word offsets of this lane's fragments. Rows: chunk of step s 4 s + 2 g + {0, 1}; weights:
  // chunk 2 s + g at slot (g ^ f) ^ 2 s
  int ro[WR], rsw[WR], po[WP], psw[WP];
#pragma unroll
  for (int i = 0; i < WR; ++i) {
    const int rr = wr * WR * 32 + 32 * i + l32;
    ro[i] = RAW == RAW_ROWS   ? rr * 32
            : RAW == RAW_TAPS && TT == 1
                ? 8 * g * RB + ((((rr >> 2) ^ (8 * g)) << 2) | (rr & 3))
            : RAW == RAW_TAPS ? (TT == 4 ? -g : 8 * g * 4 * CPW) + rr + (TT - 1)
                              : 4 * rr + g * 4 * WCH;
    rsw[i] = chunk_swizzle(rr);
  }
#pragma unroll
  for (int j = 0; j < WP; ++j) {
    const int rr = wp * WP * 32 + 32 * j + l32;
    po[j] = RF + rr * 48;
    psw[j] = g ^ ((rr >> 2) & 3);
  }
  // Software pipeline over steps of 16 k, two per stage. While the MFMAs of step t run, the wave
  // splits step t+1's activations (read during step t-1), reads step t+1's weight parts and, from
  // the middle of the step on, step t+2's activations. By the middle of a stage's first step every
  // read of that stage has been issued: the one barrier of the stage stands there, makes the next
  // stage visible and frees this one's slot for stage kt + S.
  float4 raw[2][WR][2];
  Split8 xs[2][WR], pl[2][WP];
  // RAW_TAPS: whether step s's element of this lane's column lies in the row
  auto inside = [&](int i, int s) {
    const int p = n0 + wr * WR * 32 + 32 * i + l32 - (TT == 1 ? 0 : TT == 2 ? s : 2 * s + g);
    return p >= 0 && p < Ls;
  };
  auto read_raw = [&](const float* base, int s, int kt) {
    int w[4] = {0, 0, 0, 0};  // positions before the window's first, rows r mod 4
    if constexpr (RAW == RAW_TAPS && TT > 1) {
      const int align0 = taps(kt0 + min(kt, nk - 1)).align0;
#pragma unroll
      for (int r = 0; r < 4; ++r) w[r] = (align0 + r * Ls) & 3;
    }
#pragma unroll
    for (int i = 0; i < WR; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if constexpr (RAW == RAW_ROWS) {
          raw[s][i][h] = *reinterpret_cast<const float4*>(base + ro[i] +
                                                          4 * ((4 * s + 2 * g + h) ^ rsw[i]));
        } else if constexpr (RAW == RAW_TAPS) {  // k = 16 s + 8 g + 4 h ..: tap k / CR, row k % CR
          constexpr int P = 4 * CPW;
          const float* p = base + ro[i] +
                           (TT == 1 ? (16 * s + 4 * h) * P : TT == 2 ? 4 * h * P - s : 4 * h * P - 2 * s);
          raw[s][i][h] = make_float4(p[w[0]], p[P + w[1]], p[2 * P + w[2]], p[3 * P + w[3]]);
        } else {  // channel 2 s + g, taps 4 h ..
          raw[s][i][h] = *reinterpret_cast<const float4*>(base + ro[i] + s * 8 * WCH + 4 * h);
        }
      }
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
    if constexpr (RAW == RAW_TAPS) {  // in every tile: a branch would keep the split apart from the MFMAs
#pragma unroll
      for (int i = 0; i < WR; ++i) {
        const bool in = inside(i, s);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          raw[s][i][h].x = in ? raw[s][i][h].x : 0.f;
          raw[s][i][h].y = in ? raw[s][i][h].y : 0.f;
          raw[s][i][h].z = in ? raw[s][i][h].z : 0.f;
          raw[s][i][h].w = in ? raw[s][i][h].w : 0.f;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < WR; ++i)
      xs[s][i] = split8(reinterpret_cast<const float*>(&raw[s][i][0]));
  };
  auto products = [&](int s, int p0, int p1) {
#pragma unroll
    for (int p = p0; p < p1; ++p)
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) {
          floatx16& c = p == 5 ? acc[i][j] : low[i][j];
          c = WA ? mfma_x3(pl[s][i], xs[s][j], c, p) : mfma_x3(xs[s][i], pl[s][j], c, p);
        }
  };
  // n MFMAs with kV VALU instructions behind each
  auto interleave = [&](auto nc) {
    constexpr int kV = ((RAW == RAW_TAPS ? 104 : 88) * WR / 2 + 6 * WM * WN - 1) / (6 * WM * WN);
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
  if (S - 1 < nk) {
    if (full) wait_vmcnt<(S - 1) * L>();
    else wait_vmcnt<(S - 1) * (L - 1)>();
  } else {
    wait_vmcnt<0>();
  }
  if (edge) fix_edges(0, 0);
  stage_barrier();
  // merged here, where the partials have landed, and not in the epilogue: 2 registers instead of 16
  // beside the accumulators
  float2 lnc = make_float2(0.f, 0.f);
  if constexpr (kFold) {
    lnc = ln_row_merge(a, lnr);
    asm volatile("" : "+v"(lnc.x), "+v"(lnc.y));
  }
  read_raw(smem, 0, 0);
  read_planes(smem, 0);
  read_raw(smem, 1, 0);
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
        if (kt + S - 1 < nk) {
          if (full) wait_vmcnt<(S - 2) * L>();
          else wait_vmcnt<(S - 2) * (L - 1)>();
        } else {
          wait_vmcnt<0>();
        }
        if (edge) fix_edges(kt + 1, (u + 1) % S);
        stage_barrier();  // stage kt + 1 is whole, stage kt's slot is free
        if (kt + S < nk) issue(kt + S, u);
        read_raw(next, 0, kt + 1);
        products(0, 3, 6);
        __builtin_amdgcn_sched_group_barrier(0x100, (RAW == RAW_TAPS ? 8 : 2) * WR, 0);  // reads first
        __builtin_amdgcn_sched_group_barrier(0x008, kHalf, 0);
        __builtin_amdgcn_sched_barrier(0);
        read_planes(next, 0);
        split(0);
        products(1, 0, 6);
        read_raw(next, 1, kt + 1);
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
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] += low[i][j][v];

  if constexpr (TM == 2) {  // the second team hands its sums over and is done
    constexpr int Q = WM * WN * 4;  // float4 per lane
    static_assert(NW * Q * 64 * 4 <= TM * S * STAGE, "the sums fit the rings");
    float4* x = reinterpret_cast<float4*>(smem_all) + wave * Q * 64 + lane;
    __syncthreads();  // the last fragment reads of the rings are done
    if (team == 1) {
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            x[((i * WN + j) * 4 + q) * 64] = make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1],
                                                         acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
    }
    __syncthreads();
    if (team == 1) return;  // barriers wait for the waves that are left
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4 v = x[((i * WN + j) * 4 + q) * 64];
          acc[i][j][4 * q] += v.x;
          acc[i][j][4 * q + 1] += v.y;
          acc[i][j][4 * q + 2] += v.z;
          acc[i][j][4 * q + 3] += v.w;
        }
  }

  // Not finite or tiny somewhere: this wave's block again in fp32, straight from memory (the parts of
  // a weight sum to it).
  if (any_out_of_range(acc)) {
    const unsigned short* W = reinterpret_cast<const unsigned short*>(a.wplanes);
    auto weight = [&](int row, int k) {
      const unsigned short* p = W + ((int64_t)min(row, prows - 1) * (K / 32) + k / 32) * 96 + k % 32;
      auto f = [](unsigned short b) { return __builtin_bit_cast(float, (unsigned)b << 16); };
      return f(p[0]) + (f(p[32]) + f(p[64]));
    };
    auto act = [&](int n, int k) {
      n = min(n, xrows - 1);
      if constexpr (RAW == RAW_ROWS) return X[(int64_t)n * ldx + k];
      int c = k / 8, p = 4 * n - a.conv_pad + k % 8;  // RAW_CONV
      if constexpr (RAW == RAW_TAPS) {
        c = k / 32 * CR + k % 32 % CR;
        p = n - k % 32 / CR;
      }
      if (c >= a.kvalid) return 0.f;
      if (reflect) {
        p = p < 0 ? -p : p;
        p = p > Ls - 1 ? 2 * (Ls - 1) - p : p;
      }
      if (p < 0 || p > Ls - 1) return 0.f;
      return RAW == RAW_TAPS && c >= a.kc1 ? X2[(int64_t)(c - a.kc1) * Ls + p]
                                           : X[(int64_t)c * Ls + p];
    };
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    const int rm = m0 + wm * WM * 32 + l32, rn = n0 + wn * WN * 32 + l32;
#pragma unroll 1
    for (int k = kt0 * BK + g; k < (kt0 + TM * nk) * BK; k += 2) {
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
  } else if constexpr (EPI == 4) {
    __syncthreads();
    store_rows_stats<WMW, WNW, WM, WN>(a, acc, m0, n0, wm, wn, lane, logical, smem);
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
// 128x128 / 64x128 / 64x64): 10752x1536x384 80 / 88 / 103, 5376x1152x384 35 / 33 / 40,
// 2048x2048x512 32 / 29 / 39, 5376x384x1536 61 / 44 / 49, 1000x384x384 17.6 / 11 / 8.4 (the fp32
// kernel: 117, 48, 42, 57, 9.9). Transposed convs read in place, 128x128 / 64x128 / 64x64: 384x768 at
// 5376 columns, two taps 33 / 30 / 32, 864x384 at 10836, one tap 70 / 52 / 58, and over the twelve of a 60 s
// separation 1043 / 955 / 944 against 884 as chosen. 128 activation rows by 64 weight rows were behind 64x128 at every
// shape (half the products per split value), 256x128 ahead only from about 4096^3 on.
// Two teams (tile 3): a lone workgroup of four waves has one wave per SIMD, which runs its split and its
// products one after the other (64x64: 987 cycles a stage, 384 of them MFMAs, some 400 the split's), so two of
// them share a workgroup, each with half of K. 64x64 one team / two (us): 67x1536x384 8.1 / 7.8,
// 67x384x1536 22.5 / 18.7, 1000x384x384 8.4 / 8.2, 2688x384x1536 28.7 / 26.8, the transposed conv 384 -> 96 at
// 5375 positions 32.6 / 30.4. Two teams of 64x128 or 128x128 were behind these everywhere.
struct X3Tile {
  int id, rb, pb, teams;
  double eff, alone;  // alone: part of eff that one workgroup on a CU reaches
};
constexpr X3Tile kX3Tiles[] = {{0, 128, 128, 1, 1.00, 0.80}, {1, 64, 128, 1, 0.95, 0.80},
                               {2, 64, 64, 1, 0.70, 0.80}, {3, 64, 64, 2, 0.74, 0.87}};

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int forced_x3_tile() {
  static const int v = [] {
    const char* e = std::getenv("MNN_GEMM_X3_TILE");
    return e ? std::atoi(e) : -1;
  }();
  return v;
}

int64_t x3_tiles(const GemmArgs& a, const X3Tile& t) {
  return (int64_t)cdiv(a.wa ? a.N : a.M, t.rb) * cdiv(a.wa ? a.M : a.N, t.pb);
}

// Two teams need whole stages for both, four or more each (else the hand-over costs what they gain);
// the encoders' GLU rewrites, whose epilogue is light, were 1 us slower with them (time encoder 146 / 147).
// 128x128 has two accumulators of 64 registers beside its fragments. The forms whose addresses do not fit
// beside them would read them back from scratch memory in the loop, behind every load in flight (strided
// convs over a 60 s separation 1178 -> 1842 us), and have the smaller tiles only: GLU, K parts, strided convs.
bool x3_tile_fits(const GemmArgs& a, const X3Tile& t) {
  if (t.id == 0 && (a.glu || a.ksplit > 1)) return false;
  const int nk = a.K / BK / a.ksplit;
  return t.teams == 1 || (nk % 2 == 0 && nk >= 8 && !a.glu);
}

// Per-CU critical path as in the fp32 kernel's chooser; a workgroup alone on its CU runs at about
// 0.8 of the rate of two (2450 against 3420 / 2 cycles per stage of a 128x128 tile). The taps' longer
// reads (four rows an address each) make two teams worth more: 0.78.
const X3Tile& choose_x3_tile(const GemmArgs& a) {
  const int f = forced_x3_tile();
  if (f >= 0 && f < (int)(sizeof(kX3Tiles) / sizeof(kX3Tiles[0])) && x3_tile_fits(a, kX3Tiles[f]))
    return kX3Tiles[f];
  const X3Tile* best = &kX3Tiles[1];
  double best_cost = 1e300;
  for (const X3Tile& t : kX3Tiles) {
    if (!x3_tile_fits(a, t)) continue;
    const int64_t per_cu = cdiv(x3_tiles(a, t) * a.batch * a.ksplit, (int64_t)256);
    const double eff = t.teams == 2 && a.kn_cp > 0 && a.K > a.kn_cp ? 0.78 : t.eff;
    const double cost = (double)per_cu * t.rb * t.pb / eff / (per_cu == 1 ? t.alone : 1.0);
    if (cost < best_cost * 0.999) {
      best_cost = cost;
      best = &t;
    }
  }
  return *best;
}

// WR x WP 32-row blocks (activations x weights) per wave, 2 x 2 waves (WP = 3: 1 x 4) in each of TM
// teams.
template <int WR, int WP, int S, int RAW, int TT = 1, int TM = 1>
void launch_x3(const LaunchCtx& c, const GemmArgs& a) {
  const dim3 block(256 * TM);
  const char* name = a.name ? a.name : "gemm_f32_mfma_nk";
  if constexpr (RAW == RAW_ROWS) {
    if (!a.wa) {
      const dim3 grid(cdiv(a.N, WP * 64), cdiv(a.M, WR * 64), a.batch);
      return launch(c, name, gemm_x3_kernel<2, 2, WR, WP, S, 0, false, RAW, 1, TM>, grid, block, 0, a);
    }
  }
  constexpr int MW = WP == 3 ? 1 : 2, NWV = WP == 3 ? 4 : 2;
  constexpr bool kBig = WR == 2 && WP == 2;  // x3_tile_fits
  const dim3 grid(cdiv(a.N, WR * 32 * NWV), cdiv(a.M, WP * 32 * MW), a.batch * a.ksplit);
  if constexpr (RAW == RAW_CONV) {
    if (a.ksplit > 1)
      return launch(c, name, gemm_x3_kernel<MW, NWV, WP, WR, S, 3, true, RAW, 1, TM>, grid, block, 0, a);
    return launch(c, name, gemm_x3_kernel<MW, NWV, WP, WR, S, 4, true, RAW, 1, TM>, grid, block, 0, a);
  } else if constexpr (RAW == RAW_TAPS) {
    auto go = [&](auto kern) { launch(c, name, kern, grid, block, 0, a); };
    MNN_REQUIRE(!kBig || a.ksplit == 1, MNN_ERR_INVALID_ARGUMENT, "gemm_x3: no such tile for K parts");
    if constexpr (!kBig)
      if (a.ksplit > 1) return go(gemm_x3_kernel<MW, NWV, WP, WR, S, 3, true, RAW, TT, TM>);
    if (a.ct_stride > 0) return go(gemm_x3_kernel<MW, NWV, WP, WR, S, 2, true, RAW, TT, TM>);
    if constexpr (TT == 1) return go(gemm_x3_kernel<MW, NWV, WP, WR, S, 0, true, RAW, TT, TM>);
    fail(MNN_ERR_INVALID_ARGUMENT, "gemm_x3_taps: the plain epilogue is built for one tap");
  } else {
    if constexpr (TM == 1 && !kBig) {
      if (a.glu)
        return launch(c, name, gemm_x3_kernel<MW, NWV, WP, WR, S, 1, true, RAW>, grid, block, 0, a);
    }
    MNN_REQUIRE(!a.glu, MNN_ERR_INVALID_ARGUMENT, "gemm_x3: no such tile for the GLU form");
    return launch(c, name, gemm_x3_kernel<MW, NWV, WP, WR, S, 0, true, RAW, 1, TM>, grid, block, 0, a);
  }
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
  // the forms that are built: the plain epilogue, and GLU over weights x activations
  return off32 && (a.wa ? !a.ln_parts : !a.glu) && a.ksplit == 1;
}

int64_t gemm_x3_tiles(const GemmArgs& a) { return x3_tiles(a, choose_x3_tile(a)); }

void gemm_x3(const LaunchCtx& c, const GemmArgs& a) {
  switch (choose_x3_tile(a).id) {
    case 0: return launch_x3<2, 2, 2, RAW_ROWS>(c, a);
    case 1: return launch_x3<1, 2, 2, RAW_ROWS>(c, a);
    case 2: return launch_x3<1, 1, 3, RAW_ROWS>(c, a);
    default: return launch_x3<1, 1, 2, RAW_ROWS, 1, 2>(c, a);
  }
}

namespace {
// What both channel-major forms address: signals of 4 samples or more, weights within 4 GiB.
void require_channel_major(const GemmArgs& a) {
  MNN_REQUIRE(a.wplanes && a.wa && a.batch >= 1 && a.K % BK == 0 && a.K > 0 && a.M > 0 && a.N > 0 &&
                  a.lda == a.K && a.sA == 0 && a.ldb >= 4 &&
                  a.kvalid >= 1 && x3_planes_bytes(a.M, a.K) < ((int64_t)1 << 32) &&
                  a.ksplit >= 1 && (a.K / BK) % a.ksplit == 0 && (a.ksplit == 1 || a.ws),
              MNN_ERR_INVALID_ARGUMENT, "gemm_x3: operands outside the channel-major forms");
}
}  // namespace

void gemm_x3_taps(const LaunchCtx& c, const GemmArgs& a) {
  require_channel_major(a);
  MNN_REQUIRE(a.ldb < (a.K == a.kn_cp ? (int64_t)1 << 30 : (int64_t)kLongRow) &&
                  a.kn_cp % BK == 0 && a.kn_cp >= a.kvalid && a.K % a.kn_cp == 0 &&
                  (a.K / a.kn_cp == 1 || a.K / a.kn_cp == 2 || a.K / a.kn_cp == 4) &&
                  a.kc1 >= 0 && a.kc1 <= a.kvalid &&
                  (a.kc1 == a.kvalid || a.B2) && (a.stats == nullptr || a.ct_stride > 0),
              MNN_ERR_INVALID_ARGUMENT, "gemm_x3_taps: unsupported operands");
  auto tile = [&](auto tt) {
    constexpr int TT = decltype(tt)::value;
    switch (choose_x3_tile(a).id) {
      case 0: return launch_x3<2, 2, 2, RAW_TAPS, TT>(c, a);
      case 1: return launch_x3<1, 2, 2, RAW_TAPS, TT>(c, a);
      case 2: return launch_x3<1, 1, 2, RAW_TAPS, TT>(c, a);
      default: return launch_x3<1, 1, 2, RAW_TAPS, TT, 2>(c, a);
    }
  };
  switch (a.K / a.kn_cp) {
    case 1: return tile(std::integral_constant<int, 1>{});
    case 2: return tile(std::integral_constant<int, 2>{});
    default: return tile(std::integral_constant<int, 4>{});
  }
}

void gemm_x3_conv(const LaunchCtx& c, const GemmArgs& a, int tile) {
  require_channel_major(a);
  // the length is bounded as in enc_conv_supported, with the padded channels
  MNN_REQUIRE(a.K % 32 == 0 && a.K >= 8 * a.kvalid && a.conv_pad >= 0 && a.conv_pad < 4 &&
                  a.ldb >= 8 && (int64_t)a.K / 8 * a.ldb < ((int64_t)1 << 29),
              MNN_ERR_INVALID_ARGUMENT, "gemm_x3_conv: unsupported operands");
  switch (tile) {
    case 0: return launch_x3<1, 2, 2, RAW_CONV>(c, a);
    case 1: return launch_x3<1, 1, 3, RAW_CONV>(c, a);
    default: return launch_x3<1, 3, 2, RAW_CONV>(c, a);
  }
}

}  // namespace k
}  // namespace mnn
