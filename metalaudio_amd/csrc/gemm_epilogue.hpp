// Epilogues of the LDS-DMA GEMM kernels (k_gemm_lds.hip, k_gemm_x3.hip): what is done with a
// workgroup's accumulators of 32x32 blocks. Accumulator layout of a block: lane l, register v ->
// row 8*(v/4) + 4*(l/32) + v%4, column l%32.
#pragma once

#include "device_utils.hpp"
#include "kernels.hpp"
#include "lds_dma.hpp"

namespace mnn {
namespace k {
namespace {

using namespace dev;

// C = R + rscale[n] * act(acc + bias) (R, rscale optional). ACT = -1: activation code at run time.
// Accumulator layout of a 32x32 block: lane l, register v -> row 8*(v/4) + 4*(l/32) + v%4,
// column l%32; each store instruction writes two 128-byte row segments.
//
// The values the stores depend on are loaded before the stores, and one explicit wait separates
// them. The vector memory counter counts stores as well as loads, so a load issued between stores
// (or one the compiler cannot track through a branch) makes each later store wait for every
// earlier store, and the epilogue would run at one memory latency per store. R may be C itself
// (in-place residual, element for element); no lane stores an element another lane reads, so
// loading before storing is exact. FAST (no bias along M, no residual): the few loads of the tile
// come first. Otherwise one 32-row block at a time: its loads, a wait, its stores (holding every
// residual of the tile at once would push the kernel past the register budget of two workgroups
// per CU).
template <int WMW, int WNW, int WM, int WN, int ACT, bool RES, bool FAST>
__device__ __forceinline__ void store_tile(const GemmArgs& a, const floatx16 (&acc)[WM][WN], int m0,
                                           int n0, int wm, int wn, int lane) {
  const int g = lane >> 5, l32 = lane & 31;
  const int bz = blockIdx.z;
  float* __restrict__ Cp = a.C + (int64_t)bz * a.sC;
  const float* Rp = RES && a.R ? a.R + (int64_t)bz * a.sR : nullptr;
  const bool full_m = m0 + WMW * WM * 32 <= a.M;
  constexpr int RI = FAST ? WM : 1;  // 32-row blocks whose residuals are held at once
  float bnv[WN], rsv[WN];
  float rv[RES ? RI : 1][RES ? WN : 1][16];
  if (a.bias_mode == BIAS_N) {
#pragma unroll
    for (int j = 0; j < WN; ++j) bnv[j] = a.bias[min(n0 + wn * WN * 32 + j * 32 + l32, a.N - 1)];
  } else {
#pragma unroll
    for (int j = 0; j < WN; ++j) bnv[j] = 0.f;
  }
#pragma unroll
  for (int j = 0; j < WN; ++j)
    rsv[j] = RES && Rp && a.rscale ? a.rscale[min(n0 + wn * WN * 32 + j * 32 + l32, a.N - 1)] : 1.f;
  // residuals of blocks [i0, i0 + RI)
  auto load_res = [&](int i0) {
    if constexpr (RES) {
#pragma unroll
      for (int ii = 0; ii < RI; ++ii)
#pragma unroll
        for (int j = 0; j < WN; ++j) {
          const int gn = min(n0 + wn * WN * 32 + j * 32 + l32, a.N - 1);
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int gm =
                min(m0 + wm * WM * 32 + (i0 + ii) * 32 + 8 * (v / 4) + 4 * g + (v % 4), a.M - 1);
            rv[ii][j][v] = Rp ? Rp[(int64_t)gm * a.ldr + gn] : 0.f;
          }
        }
    }
  };
  if constexpr (FAST) {
    load_res(0);
    wait_vmcnt<0>();
  }
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int mblk = m0 + wm * WM * 32 + i * 32;
    float bmv[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) bmv[v] = 0.f;
    if constexpr (!FAST) {
      if (a.bias_mode == BIAS_M) {
#pragma unroll
        for (int v = 0; v < 16; ++v) bmv[v] = a.bias[min(mblk + 8 * (v / 4) + 4 * g + (v % 4), a.M - 1)];
      }
      load_res(i);
      wait_vmcnt<0>();
    }
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const int gn = n0 + wn * WN * 32 + j * 32 + l32;
      if (gn >= a.N) continue;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int gm = mblk + 8 * (v / 4) + 4 * g + (v % 4);
        if (full_m || gm < a.M) {
          float val = acc[i][j][v] + bnv[j] + bmv[v];
          val = ACT < 0 ? apply_act(val, a.act, a.act_alpha) : apply_act(val, ACT);
          if constexpr (RES) val = rv[FAST ? i : 0][j][v] + rsv[j] * val;
          Cp[(int64_t)gm * a.ldc + gn] = val;
        }
      }
    }
  }
}

// Folded LayerNorm of A's rows: (rstd, -rstd * mean) of row m merged from its K / 64 partials
// (mean, M2) of 64 features each (Chan's formula for equal counts, a fixed order; K <= 64 *
// kLnMaxParts). ln_row_load issues the loads before the main loop (GEMMs without a folded LayerNorm
// read a zero dummy, so no load sits under a branch); ln_row_merge combines them.
constexpr int kLnMaxParts = 8;
struct LnRow {
  float2 q[kLnMaxParts];
};

__device__ float2 ln_dummy_parts[kLnMaxParts];

__device__ __forceinline__ LnRow ln_row_load(const GemmArgs& a, int m) {
  const bool on = a.ln_parts != nullptr;
  const int P = on ? a.K / 64 : 1;
  const float2* pp =
      on ? reinterpret_cast<const float2*>(a.ln_parts) + (int64_t)min(m, a.M - 1) * P
         : ln_dummy_parts;
  LnRow r;
#pragma unroll
  for (int p = 0; p < kLnMaxParts; ++p) r.q[p] = pp[min(p, P - 1)];
  return r;
}

__device__ __forceinline__ float2 ln_row_merge(const GemmArgs& a, const LnRow& r) {
  if (!a.ln_parts) return make_float2(0.f, 0.f);
  const int P = a.K / 64;
  float mean = r.q[0].x, m2 = r.q[0].y;
#pragma unroll
  for (int p = 1; p < kLnMaxParts; ++p) {
    if (p < P) {
      const float d = r.q[p].x - mean;
      mean += d * (1.f / (float)(p + 1));
      m2 += r.q[p].y + d * d * (64.f * (float)p / (float)(p + 1));
    }
  }
  const float rstd = 1.f / sqrtf(m2 / (float)a.K + a.ln_eps);
  return make_float2(rstd, -rstd * mean);
}

// The same epilogue with the tile transposed through LDS into row order, for outputs whose rows
// are 16-byte aligned (N % 4 == 0, ldc % 4 == 0; residual likewise): the accumulators are written
// to LDS ([rows][BN + 8 floats]: rows four apart, which the two lane groups write together, sit 32
// banks apart), read back as float4 along rows and stored so that consecutive lanes cover
// consecutive 16-byte pieces of a row — 512-byte row runs per half-wave for BN = 128 instead of the
// accumulator layout's 128-byte pieces of 32 rows, which the memory system served at about 2 TB/s.
// Bias (along N), activation, residual and LayerScale apply in row order. Tiles whose rows do not
// fit the LDS ring at once go in passes of whole wave rows. The caller has synchronised the
// workgroup after its last LDS read of the main loop.
template <int WMW, int WNW, int WM, int WN, int ACT, bool RES, int LDS_FLOATS>
__device__ __forceinline__ void store_tile_lds(const GemmArgs& a, const floatx16 (&acc)[WM][WN],
                                               int m0, int n0, int wm, int wn, int lane,
                                               float* smem, float2 lnc) {
  constexpr int BM = WMW * WM * 32, BN = WNW * WN * 32, NT = WMW * WNW * 64;
  constexpr int PITCH = BN + 8;
  constexpr int WROWS = WM * 32;  // rows per wave row
  constexpr int PASS_WM = (BM * PITCH <= LDS_FLOATS) ? WMW : 1;  // wave rows per pass
  constexpr int PROWS = PASS_WM * WROWS;                          // rows per pass
  static_assert(PROWS * PITCH <= LDS_FLOATS, "epilogue tile does not fit the LDS ring");
  constexpr int C4 = BN / 4;                  // float4 per row
  constexpr int RPI = NT / C4;                // rows per thread iteration
  constexpr int IT = PROWS / RPI;             // iterations per pass
  static_assert(NT % C4 == 0 && PROWS % RPI == 0, "epilogue thread layout");
  const int g = lane >> 5, l32 = lane & 31;
  const int tid = threadIdx.x;
  const int bz = blockIdx.z;
  float* __restrict__ Cp = a.C + (int64_t)bz * a.sC;
  const float* Rp = RES && a.R ? a.R + (int64_t)bz * a.sR : nullptr;
  const int c4 = tid % C4, rr0 = tid / C4;
  const int gn = n0 + 4 * c4;
  const bool col_ok = gn < a.N;  // N % 4 == 0: a float4 is all in or all out
  float4 bn = make_float4(0.f, 0.f, 0.f, 0.f), rs = make_float4(1.f, 1.f, 1.f, 1.f);
  if (col_ok && a.bias_mode == BIAS_N) bn = *reinterpret_cast<const float4*>(a.bias + gn);
  if (RES && Rp && a.rscale && col_ok) rs = *reinterpret_cast<const float4*>(a.rscale + gn);
  // Folded LayerNorm: thread r < BM holds row m0 + r's (rstd, -rstd * mean), kept at the end of the
  // LDS ring past the rows the passes below write; the first pass's barrier makes them visible.
  static_assert(PROWS * PITCH + 2 * BM <= LDS_FLOATS, "epilogue tile and row coefficients");
  static_assert(BM <= NT, "one row coefficient per thread");
  float2* lnrow = reinterpret_cast<float2*>(smem + LDS_FLOATS - 2 * BM);
  const bool ln = a.ln_parts != nullptr;
  float4 lc = make_float4(0.f, 0.f, 0.f, 0.f);
  if (ln) {
    if (col_ok) lc = *reinterpret_cast<const float4*>(a.ln_c + gn);
    if (tid < BM) lnrow[tid] = lnc;
  }
  const bool rstats = a.row_parts != nullptr;
#pragma unroll
  for (int pass = 0; pass < WMW / PASS_WM; ++pass) {
    if (pass > 0) __syncthreads();  // the previous pass's reads are done
    if (wm / PASS_WM == pass) {
      const int wr0 = (wm % PASS_WM) * WROWS;
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int r = wr0 + 32 * i + 8 * (v / 4) + 4 * g + (v % 4);
            const int c = wn * WN * 32 + 32 * j + l32;
            smem[r * PITCH + c] = acc[i][j][v];
          }
    }
    __syncthreads();
    const int prow0 = m0 + pass * PROWS;
    // residual rows first (loads before any store), then the stores
    float4 rv[RES ? IT : 1];
    if constexpr (RES) {
#pragma unroll
      for (int it = 0; it < IT; ++it) {
        const int gm = min(prow0 + rr0 + it * RPI, a.M - 1);
        rv[it] = (Rp && col_ok) ? *reinterpret_cast<const float4*>(Rp + (int64_t)gm * a.ldr + gn)
                                : make_float4(0.f, 0.f, 0.f, 0.f);
      }
      wait_vmcnt<0>();
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int r = rr0 + it * RPI;
      const int gm = prow0 + r;
      float4 v = *reinterpret_cast<const float4*>(smem + r * PITCH + 4 * c4);
      if (ln) {
        const float2 rc = lnrow[pass * PROWS + r];
        v.x = rc.x * v.x + rc.y * lc.x;
        v.y = rc.x * v.y + rc.y * lc.y;
        v.z = rc.x * v.z + rc.y * lc.z;
        v.w = rc.x * v.w + rc.y * lc.w;
      }
      v.x += bn.x;
      v.y += bn.y;
      v.z += bn.z;
      v.w += bn.w;
      if (ACT < 0) {
        v.x = apply_act(v.x, a.act, a.act_alpha);
        v.y = apply_act(v.y, a.act, a.act_alpha);
        v.z = apply_act(v.z, a.act, a.act_alpha);
        v.w = apply_act(v.w, a.act, a.act_alpha);
      } else if (ACT > 0) {
        v.x = apply_act(v.x, ACT);
        v.y = apply_act(v.y, ACT);
        v.z = apply_act(v.z, ACT);
        v.w = apply_act(v.w, ACT);
      }
      if constexpr (RES) {
        if (Rp) {
          v.x = rv[it].x + rs.x * v.x;
          v.y = rv[it].y + rs.y * v.y;
          v.z = rv[it].z + rs.z * v.z;
          v.w = rv[it].w + rs.w * v.w;
        }
      }
      if (rstats) {
        // (mean, M2) of the row's 64 columns held by this lane's 16-lane group (N % 64 == 0, so
        // col_ok is uniform over the group)
        const bool ok = col_ok && gm < a.M;
        const float mean = row16_sum(ok ? (v.x + v.y) + (v.z + v.w) : 0.f) * (1.f / 64.f);
        const float dx = v.x - mean, dy = v.y - mean, dz = v.z - mean, dw = v.w - mean;
        const float m2 = row16_sum(ok ? (dx * dx + dy * dy) + (dz * dz + dw * dw) : 0.f);
        if (ok && (c4 & 15) == 0)
          *reinterpret_cast<float2*>(a.row_parts + ((int64_t)gm * (a.N / 64) + gn / 64) * 2) =
              make_float2(mean, m2);
      }
      if (col_ok && gm < a.M) *reinterpret_cast<float4*>(Cp + (int64_t)gm * a.ldc + gn) = v;
    }
  }
}

// GLU epilogue: rows come in 32-row blocks [a0..a15 | b0..b15] (weights regrouped by the caller);
// output row 16*blk + r = (a_r + bias) * sigmoid(b_r + bias). In the accumulator layout register v
// (< 8) holds row rr = 8*(v/4) + 4*(l/32) + v%4 < 16 and register v + 8 holds row rr + 16, so every
// lane has both GLU partners.
template <int WMW, int WNW, int WM, int WN>
__device__ __forceinline__ void store_glu(const GemmArgs& a, const floatx16 (&acc)[WM][WN], int m0,
                                          int n0, int wm, int wn, int lane) {
  const int g = lane >> 5, l32 = lane & 31;
  float* __restrict__ Cp = a.C + (int64_t)blockIdx.z * a.sC;
  // bias values first (the compiler may not move these loads past the stores)
  float ba[WM][8], bb[WM][8];
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int mblk = min(m0 + wm * WM * 32 + i * 32, a.M - 32);
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const int rr = 8 * (v / 4) + 4 * g + (v % 4);
      ba[i][v] = a.bias ? a.bias[mblk + rr] : 0.f;
      bb[i][v] = a.bias ? a.bias[mblk + 16 + rr] : 0.f;
    }
  }
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int mblk = m0 + wm * WM * 32 + i * 32;
    if (mblk >= a.M) continue;
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const int gn = n0 + wn * WN * 32 + j * 32 + l32;
      if (gn >= a.N) continue;
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        const int rr = 8 * (v / 4) + 4 * g + (v % 4);
        const float va = acc[i][j][v] + ba[i][v];
        const float vb = acc[i][j][v + 8] + bb[i][v];
        Cp[(int64_t)((mblk >> 5) * 16 + rr) * a.ldc + gn] = va * stable_sigmoid(vb);
      }
    }
  }
}

// Transposed-conv epilogue: row m = s*oc + r (phase r of output channel oc), column n = q; the value
// (+ bias[oc]) belongs at output position o = s*q + r - ct_pad of channel oc:
// C[oc * ldc + o] when 0 <= o < ct_len. A lane holds the s phases of one (oc, q) in registers
// v..v+s-1 (s = 4: rows 4i..4i+3 of a 32-row block), so consecutive lanes cover consecutive
// 4-sample runs of one output row. Bias values are loaded first (see store_tile). Every output
// sample is stored by exactly one (row, column), so with a.stats each workgroup also writes the
// GroupNorm(1) partial (count, mean, M2) of the samples it stored (red: LDS for 3 floats per wave
// that nothing else uses any more) at
// stats[(batch * tiles + blockIdx.y * gridDim.x + blockIdx.x) * 3], tiles = gridDim.x * gridDim.y.
template <int WMW, int WNW, int WM, int WN>
__device__ __forceinline__ void store_ct(const GemmArgs& a, const floatx16 (&acc)[WM][WN], int m0,
                                         int n0, int wm, int wn, int lane, float* red) {
  const int g = lane >> 5, l32 = lane & 31;
  float* __restrict__ Cp = a.C + (int64_t)blockIdx.z * a.sC;
  const int s = a.ct_stride;
  float bmv[WM][16];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int gm = min(m0 + wm * WM * 32 + i * 32 + 8 * (v / 4) + 4 * g + (v % 4), a.M - 1);
      bmv[i][v] = a.bias ? a.bias[gm / s] : 0.f;
    }
  wait_vmcnt<0>();
  // four statistics accumulators, so the per-sample updates are not one dependent chain
  ShiftedStats st[4];
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int mblk = m0 + wm * WM * 32 + i * 32;
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const int q = n0 + wn * WN * 32 + j * 32 + l32;
      if (q >= a.N) continue;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int gm = mblk + 8 * (v / 4) + 4 * g + (v % 4);
        const int oc = gm / s, o = s * q + (gm - oc * s) - a.ct_pad;
        if (gm < a.M && o >= 0 && o < a.ct_len) {
          const float val = acc[i][j][v] + bmv[i][v];
          if (a.stats) st[v & 3].add(val);
          Cp[(int64_t)oc * a.ldc + o] = val;
        }
      }
    }
  }
  if (a.stats) {
    float sn, smean, sm2;
    st[0].finish(sn, smean, sm2);
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      float n2, mean2, m22;
      st[k].finish(n2, mean2, m22);
      welford_combine(sn, smean, sm2, n2, mean2, m22);
    }
    block_welford(sn, smean, sm2, red, WMW * WNW);
    if (threadIdx.x == 0) {
      float* o = a.stats + ((int64_t)blockIdx.z * gridDim.x * gridDim.y + blockIdx.y * gridDim.x +
                            blockIdx.x) * 3;
      o[0] = sn;
      o[1] = smean;
      o[2] = sm2;
    }
  }
}

// C[m][n] = acc + bias[m], with a.stats also the GroupNorm(1) partial (count, mean, M2) of the tile at
// stats[(batch * tiles + tile) * 3], tiles = gridDim.x * gridDim.y (red: LDS for 3 floats per wave).
// Bias rows come first (the compiler may not move these loads past the stores); four statistics
// accumulators keep the per-element updates from being one dependent chain.
template <int WMW, int WNW, int WM, int WN>
__device__ __forceinline__ void store_rows_stats(const GemmArgs& a, const floatx16 (&acc)[WM][WN],
                                                 int m0, int n0, int wm, int wn, int lane,
                                                 int tile, float* red) {
  const int g = lane >> 5, l32 = lane & 31;
  float* __restrict__ Cp = a.C + (int64_t)blockIdx.z * a.sC;
  ShiftedStats st[4];
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int mblk = m0 + wm * WM * 32 + i * 32;
    float bv[16];
#pragma unroll
    for (int v = 0; v < 16; ++v)
      bv[v] = a.bias ? a.bias[min(mblk + 8 * (v / 4) + 4 * g + (v % 4), a.M - 1)] : 0.f;
    wait_vmcnt<0>();
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const int gn = n0 + wn * WN * 32 + j * 32 + l32;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int gm = mblk + 8 * (v / 4) + 4 * g + (v % 4);
        if (gm < a.M && gn < a.N) {
          const float val = acc[i][j][v] + bv[v];
          if (a.stats) st[v & 3].add(val);
          Cp[(int64_t)gm * a.ldc + gn] = val;
        }
      }
    }
  }
  if (a.stats) {
    float sn, smean, sm2;
    st[0].finish(sn, smean, sm2);
#pragma unroll
    for (int q = 1; q < 4; ++q) {
      float n2, mean2, m22;
      st[q].finish(n2, mean2, m22);
      welford_combine(sn, smean, sm2, n2, mean2, m22);
    }
    block_welford(sn, smean, sm2, red, WMW * WNW);
    if (threadIdx.x == 0) {
      float* o = a.stats + ((int64_t)blockIdx.z * gridDim.x * gridDim.y + tile) * 3;
      o[0] = sn;
      o[1] = smean;
      o[2] = sm2;
    }
  }
}

// K-split partial: the raw accumulators of K part p of batch b go to
// ws[((b * ksplit + p) * M + m) * N + n]; the caller reduces the parts (and applies the epilogue).
template <int WMW, int WNW, int WM, int WN>
__device__ __forceinline__ void store_part(const GemmArgs& a, const floatx16 (&acc)[WM][WN], int m0,
                                           int n0, int wm, int wn, int lane) {
  const int g = lane >> 5, l32 = lane & 31;
  float* __restrict__ wp = a.ws + (int64_t)blockIdx.z * a.M * a.N;
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int mblk = m0 + wm * WM * 32 + i * 32;
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const int gn = n0 + wn * WN * 32 + j * 32 + l32;
      if (gn >= a.N) continue;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int gm = mblk + 8 * (v / 4) + 4 * g + (v % 4);
        if (gm < a.M) wp[(int64_t)gm * a.N + gn] = acc[i][j][v];
      }
    }
  }
}

}  // namespace
}  // namespace k
}  // namespace mnn
