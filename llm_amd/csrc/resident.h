// Matrix product of several tokens (prefill) with the activations resident in
// LDS: prologue and product in one launch, the same arithmetic per block and
// the same epilogues as the decode and prefill kernels of gemv_impl.h.
// Included by one translation unit per weight type.
#pragma once

#include "gemv_impl.h"
#include "resident_plan.h"

#include <type_traits>

namespace llmhip {

// The epilogues of a tile's row for four consecutive tokens (tok .. tok + 3) of
// one lane: what row_epilogue does for two, with one pointer per row.  `pre`:
// epi4_load's inputs, loaded under the tile's last unit.
struct Epi4In {
  float bias;
  float c[4], s[4];  // EPI_QKV: RoPE entries; EPI_ACC: the residual in c
};

// The rows of a tile are all of q, of k or of v (head sizes are multiples of
// 16 and row_base too): 0, 1 or 2, uniform over the wave.
__device__ __forceinline__ uint32_t qkv_region(const GemvArgs& a, uint32_t tile) {
  const uint32_t lf = a.row_base + tile * 16;
  return lf < a.nq ? 0 : lf < a.nq + a.nk ? 1 : 2;
}

template <int EPI>
__device__ __forceinline__ void epi4_load(Epi4In& e, const GemvArgs& a, uint32_t tile, int r, bool active, uint32_t tok) {
  const uint32_t lr = min(row_of_pos(tile * 16 + r, a.map, a.map_hd, a.map_seg0, a.map_seg1, a.ff), a.rows - 1);
  if (EPI == EPI_ACC) {
#pragma unroll
    for (int i = 0; i < 4; i++) e.c[i] = a.y[(uint64_t)min(tok + i, a.ntok - 1) * a.ldy + lr];
  }
  if (EPI == EPI_QKV) {
    const uint32_t lf = a.row_base + lr;
    e.bias = a.bias ? a.bias[lf] : 0.f;
    const uint32_t hd = a.hd, hp = hd / 2, w = lf & (hd - 1);  // (q and k start at multiples of hd)
    const float* cs = a.cs + 2 * (a.neox ? w & (hp - 1) : w / 2);
    const uint32_t p0 = state_pos(a.state);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float* p = cs + (uint64_t)(p0 + min(tok + i, a.ntok - 1)) * hd;
      e.c[i] = p[0];
      e.s[i] = p[1];
    }
  }
}

// Every lane of the wave calls it (EPI_QKV and EPI_GATEUP exchange rows).
template <int EPI>
__device__ __forceinline__ void epi4(const GemvArgs& a, uint32_t tile, int r, bool active, uint32_t tok, f4 v,
                                     const Epi4In& e, float* y) {
  const uint32_t lr = row_of_pos(tile * 16 + r, a.map, a.map_hd, a.map_seg0, a.map_seg1, a.ff);
  const bool ok = active && lr < a.rows;
  const uint32_t n = tok < a.ntok ? a.ntok - tok : 0;  // tokens that exist
  if (EPI == EPI_STORE || EPI == EPI_ACC) {
    float* p = y + (uint64_t)tok * a.ldy + lr;
#pragma unroll
    for (uint32_t i = 0; i < 4; i++)
      if (ok && i < n) p[(uint64_t)i * a.ldy] = EPI == EPI_ACC ? e.c[i] + v[i] : v[i];
  }
  if (EPI == EPI_QKV) {
    // bias (qwen2), RoPE of the q and k rows' pairs (cpu.go:284-303, 374-385), K and V into the cache
    const uint32_t reg = qkv_region(a, tile), lf = a.row_base + lr;
    v += e.bias;
    const int pm = a.neox ? 8 : 1;
    f4 o;
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = __shfl_xor(v[i], pm);
    if (reg < 2) {
      const uint32_t w = lf & (a.hd - 1);
      const bool first = a.neox ? w < a.hd / 2 : (w & 1) == 0;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float x = first ? v[i] : o[i], z = first ? o[i] : v[i];
        v[i] = first ? __fsub_rn(__fmul_rn(x, e.c[i]), __fmul_rn(z, e.s[i]))
                     : __fadd_rn(__fmul_rn(x, e.s[i]), __fmul_rn(z, e.c[i]));
      }
    }
    if (reg == 0) {
      float* p = a.y + (uint64_t)tok * a.nq + lf;
#pragma unroll
      for (uint32_t i = 0; i < 4; i++)
        if (ok && i < n) p[i * a.nq] = v[i];
    } else {
      const uint64_t c0 = (uint64_t)(reg == 2 ? a.ctx : 0) * a.kvd + (uint64_t)(state_pos(a.state) + tok) * a.kvd +
                          (lf - a.nq - (reg == 2 ? a.nk : 0));
      if (a.kv16) {
        _Float16* p = (_Float16*)a.kv + c0;
#pragma unroll
        for (uint32_t i = 0; i < 4; i++)
          if (ok && i < n) p[i * a.kvd] = to_f16(v[i]);
      } else {
        float* p = a.kv + c0;
#pragma unroll
        for (uint32_t i = 0; i < 4; i++)
          if (ok && i < n) p[i * a.kvd] = v[i];
      }
    }
  }
  if (EPI == EPI_GATEUP) {
    // act = g / (1 + exp(-g)) * u (cpu.go:345); gate row i at lane r < 8, up row i at r + 8
    const uint32_t c = 8 * tile + (r & 7);
    f4 o;
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = __shfl_xor(v[i], 8);
    const bool gate = r < 8;
    float* p = (gate ? a.y : a.up) + (uint64_t)tok * a.ff + c;
    const bool st = active && c < a.ff && (gate || a.up);
    const uint32_t t0 = gate ? 0 : a.up0;
#pragma unroll
    for (uint32_t i = 0; i < 4; i++)
      if (st && i < n && tok + i >= t0) p[i * a.ff] = gate ? v[i] / (1.f + __expf(-v[i])) * o[i] : v[i];
  }
}

// A workgroup of NW waves holds TT groups of 16 tokens over its part of k
// (all of it, or one of ra.kparts) as MFMA operands in LDS, f16 hi and lo, and
// streams its part of the row tiles past them.
//
// Staging: each lane loads its items (block b, k-group kq of one token: 8
// elements; the four lanes of a block's row share a 128-byte line), for PRO_RMS
// adds up the parts of the row (ra.nparts partial products), then the residual x
// (last, so that its larger magnitude is rounded once: logits of 701 tokens
// 2.5e-7 -> 2.0e-7 off 64-bit ones; the first row part's workgroups store the
// sum), and
// multiplies by the norm weights, the scale 1/rms following after the product
// as in the decode kernel.  Per token the largest magnitude over the part of
// k gives the power of two that puts it in [2^14, 2^15); hi = f16(x 2^e),
// lo = f16(x 2^e - hi).  Two barriers, then none: every wave streams groups of
// GT tiles on its own, units of four blocks through two register sets (the
// next unit's weights are in flight under the current one's MFMAs, across tile
// groups too), so memory latency is hidden by depth and not by barriers.
//
// Per block, tile and token group two v_mfma_f32_16x16x32_f16 chained in one
// accumulator (hi, then lo), then four FMAs by the block's scale; a weight word
// is dequantised once for TT token groups.  The steps (block, tile) are
// software-pipelined: a step's MFMAs with the scaling of the step before and
// the dequantisation of the step after between them.
//
// A tile's block products are summed in chains of two units (eight blocks), the
// chains in `tot`: one chain over 896 inputs was 1.18e-7 off 64-bit sums where
// gemm_kernel, whose waves split k, is 0.95e-7 off; so it is 0.94e-7, for 1% of
// the time (151936x896 for 64 tokens: 50.7 -> 51.4 us).
//
// Bound by VALU issue: at TT = 2 a step is 17 VALU instructions (9 dequantise,
// 8 scale) beside 4 MFMAs, 84 of the 104 busy kcycles of a SIMD in the gate/up
// product of 1024 tokens (9728x896, 50 us, 357 TFLOP/s of f32 products; the
// 16-token kernel: 16 launches of 12 us).  Two groups are what the LDS holds
// of 896 inputs.  Fewer tokens: the staging's round trips (x, the parts, the
// norm weights) and 2 us of launch.
template <uint32_t QT, int PRO, int EPI, int TT, int GT, bool TAIL, int NW>
__global__ __launch_bounds__(64 * NW, NW / 4) void resident_kernel(GemvArgs a, ResArgs ra) {
  extern __shared__ __align__(16) char lds[];
  constexpr int WPT = NW / TT;  // waves staging one token group
  // one tile per group: one copy of the loop body and its epilogue, the next unit's registers copied (few tokens:
  // the instruction fetch of code run once counts; [q; k; v] of 128 tokens 12.8 -> 12.0 us); else two copies, one
  // per register set
  constexpr bool ROLL = GT == 1;
  constexpr bool LATE = GT == 4;  // the residual read in the epilogue: ahead of it, its registers would spill
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int r = lane & 15, q = lane >> 4;
  const uint32_t nb = a.nb, ng = a.ng;
  // (row part, k part, token tile) of the workgroup
  uint32_t wt, col;
  if (!res_place(blockIdx.x, ra.ttiles, ra.rparts * ra.kparts, &wt, &col)) return;
  const uint32_t kp = col / ra.rparts, rp = col % ra.rparts, g0 = wt * TT;
  const uint32_t u0 = kp * ra.kunits, units = min(ng + (a.tail ? 1u : 0u) - u0, ra.kunits), b0 = 4 * u0,
                 nblk = min(nb - b0, 4 * units);
  const uint32_t t0 = rp * a.tiles / ra.rparts, t1 = (rp + 1) * a.tiles / ra.rparts;
  h8* xs = (h8*)lds;                                         // [nblk][TT][2][64]
  float* red = (float*)(lds + (uint64_t)nblk * TT * 2048);   // [16 waves][16] max, [16][16] sums of squares
  float* rw = red + 512;                                     // PRO_RMS: [16] max |nw| per wave
  int* tex = (int*)(rw + 16);                                // [TT * 16] exponents
  float* trs = (float*)(tex + TT * 16);                      // [TT * 16] RMS scales
  float* nws = trs + TT * 16;                                // PRO_RMS: [32 nblk] norm weights
  float* bs = nws + (PRO & PRO_RMS ? 32 * nblk : 0);         // Q4_1: [nblk][TT * 16] block sums

  // ---- the tiles of this wave
  // (GT == 1) kw waves share a tile, wave ks of them the units ks, ks + kw, ..., their sums added in order at the
  // end: with few tiles a workgroup one wave each ran all of k in a chain of dependent steps, 55 ns a block, and the
  // others waited (prefill of 128 tokens, Qwen2.5-0.5B shape: 1389 -> 1329 us).  The plan leaves one round of tiles then.
  const uint32_t lkw = ROLL ? ra.lkw : 0, kw = 1u << lkw, ks = wave & (kw - 1), slot = wave >> lkw;
  const uint32_t ngrp = (t1 - t0 + GT - 1) / GT;
  const uint32_t mine = ngrp > slot ? (ngrp - slot + (NW >> lkw) - 1) / (NW >> lkw) : 0;
  const uint32_t steps_n = units > ks ? mine * ((units - ks + kw - 1) >> lkw) : 0;
  WUnit w[2][GT];
  uint32_t fj = 0, fu = ks;  // the next unit to fetch: tile group fj of the wave's, unit fu of the part
  auto fetch = [&](WUnit (&W)[GT]) {
    const uint32_t ft = t0 + (slot + NW * fj) * GT;
#pragma unroll
    for (int u = 0; u < GT; u++) {
      const uint32_t t = min(ft + u, t1 - 1);
      if (!TAIL || u0 + fu < ng) {
        load_group<QT>(W[u], a.qs, nb, t, u0 + fu, lane, r);
      } else {
        // the tail's blocks in the places of a group's
        WUnit x;
        load_unit<QT>(x, a.qs, nb, t, ng, ng, a.tail, lane, r);
        if (QT == LLMHIP_Q8_0) {
          W[u].w0 = uint4{x.w0.x, x.w1.x, x.w0.y, x.w1.y};
          W[u].w1 = uint4{x.w0.z, x.w1.z, 0, 0};
        } else {
          W[u].w0 = x.w0;
        }
        W[u].sv = QT == LLMHIP_Q4_1 ? x.sv : uint4{x.sv.x | x.sv.y << 16, x.sv.z, 0, 0};
      }
    }
    if ((fu += kw) >= units) {
      fu = ks;
      fj = min(fj + 1, mine - 1);  // past the end: the last group again (not used)
    }
  };

  // ---- staging
  {
    constexpr int NI = (RES_ITEMS * 8 / NW + 1) / 2;
    const uint32_t tg = wave / WPT, ws = wave % WPT, t = lane >> 2, kq = lane & 3;
    const uint32_t tok = (g0 + tg) * 16 + t;
    const bool live = tok < a.ntok, two = nblk > NI * WPT;
    const uint64_t row = (uint64_t)(a.xrow0 + min(tok, a.ntok - 1)) * a.ldx + b0 * 32 + 4 * kq;
    f4 v[2][NI][2];
    auto each = [&](auto&& f) {
#pragma unroll
      for (int i = 0; i < NI; i++) f(0, i, ws + i * WPT);
      if (two)
#pragma unroll
        for (int i = 0; i < NI; i++) f(1, i, ws + (NI + i) * WPT);
    };
    constexpr int NWL = (RES_ITEMS * 8 * 32 + 64 * NW * 4 - 1) / (64 * NW * 4);
    f4 wl[NWL];  // norm weights on their way to LDS
    if (PRO & PRO_RMS)
#pragma unroll
      for (int i = 0; i < NWL; i++) wl[i] = *(const f4*)(a.nw + min((uint32_t)(tid + i * 64 * NW) * 4, nblk * 32 - 4));
    // loads without a condition (a block past the part reads its last one; it
    // takes no part in the maximum, the sum or the operands)
    // (the sum's terms: the parts, then x)
    auto term = [&](uint32_t p) { return (PRO & PRO_RMS) && p < ra.nparts ? ra.parts + p * ra.pstride + row : a.x + row; };
    each([&](int h, int i, uint32_t b) {
      const float* p = term(0) + 32 * min(b, nblk - 1);
      v[h][i][0] = *(const f4*)p;
      v[h][i][1] = *(const f4*)(p + 16);
    });
    if (PRO & PRO_RMS) {
      // parts in one round of loads each, or (rows in one batch of items) PU parts in one
      constexpr int PU = NW == 8 ? 4 : 2;
      uint32_t p = 1;
      if (!two)
        for (; p < ra.nparts; p += PU) {
          f4 y[PU][NI][2];
#pragma unroll
          for (int k = 0; k < PU; k++) {
            const float* xp = term(min(p + k, ra.nparts));
#pragma unroll
            for (int i = 0; i < NI; i++) {
              const uint32_t b = min(ws + i * WPT, nblk - 1);
              y[k][i][0] = *(const f4*)(xp + 32 * b);
              y[k][i][1] = *(const f4*)(xp + 32 * b + 16);
            }
          }
#pragma unroll
          for (int k = 0; k < PU; k++)
            if (p + k <= ra.nparts)
#pragma unroll
              for (int i = 0; i < NI; i++) {
                v[0][i][0] += y[k][i][0];
                v[0][i][1] += y[k][i][1];
              }
        }
      for (; p <= ra.nparts; p++) {
        const float* xp = term(p);
        f4 y[2][NI][2];
        each([&](int h, int i, uint32_t b) {
          y[h][i][0] = *(const f4*)(xp + 32 * min(b, nblk - 1));
          y[h][i][1] = *(const f4*)(xp + 32 * min(b, nblk - 1) + 16);
        });
        each([&](int h, int i, uint32_t) {
          v[h][i][0] += y[h][i][0];
          v[h][i][1] += y[h][i][1];
        });
      }
      if (ra.xout && rp == 0)
        each([&](int h, int i, uint32_t b) {
          if (b < nblk && live) {
            float* o = ra.xout + row + 32 * b;
            *(f4*)o = v[h][i][0];
            *(f4*)(o + 16) = v[h][i][1];
          }
        });
    }
    float mx = 0, ss = 0, mw = 0;
    if (PRO & PRO_RMS) {
#pragma unroll
      for (int i = 0; i < NWL; i++) {
        const uint32_t e = (uint32_t)(tid + i * 64 * NW) * 4;
        if (e < nblk * 32) *(f4*)(nws + e) = wl[i];
        mw = fmaxf(fmaxf(mw, fmaxf(fabsf(wl[i][0]), fabsf(wl[i][1]))), fmaxf(fabsf(wl[i][2]), fabsf(wl[i][3])));
      }
      mw = wave_max_dpp(mw);
      if (lane == 0) rw[wave] = mw;
      each([&](int h, int i, uint32_t b) {
        if (b < nblk)
#pragma unroll
          for (int e = 0; e < 8; e++) ss += v[h][i][e / 4][e % 4] * v[h][i][e / 4][e % 4];
      });
    }
    if (steps_n) {
      fetch(w[0]);
      if (!ROLL) fetch(w[1]);
    }
    each([&](int h, int i, uint32_t b) {
      if (b < nblk)
#pragma unroll
        for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(v[h][i][e / 4][e % 4]));
    });
    mx = fmaxf(mx, dpp_mov<DPP_XOR1>(mx));
    mx = fmaxf(mx, dpp_mov<DPP_XOR2>(mx));
    if (PRO & PRO_RMS) {
      ss += dpp_mov<DPP_XOR1>(ss);
      ss += dpp_mov<DPP_XOR2>(ss);
    }
    if (kq == 0) {
      red[wave * 16 + t] = mx;
      if (PRO & PRO_RMS) red[256 + wave * 16 + t] = ss;
    }
    __syncthreads();
    mx = 0;
    ss = 0;
#pragma unroll
    for (int i = 0; i < WPT; i++) {
      mx = fmaxf(mx, red[(tg * WPT + i) * 16 + t]);
      if (PRO & PRO_RMS) ss += red[256 + (tg * WPT + i) * 16 + t];
    }
    if (PRO & PRO_RMS) {
      // a bound on |x nw|: the split keeps its 22 bits well below the largest
      // magnitude, so a bound some bits above it does as well as the maximum
      mw = 0;
#pragma unroll
      for (int i = 0; i < NW; i++) mw = fmaxf(mw, rw[i]);
      mx *= mw;
    }
    int ex = 0;
    if (live && mx > 0 && mx <= 3.0e38f) {
      int E;
      frexpf(mx, &E);
      ex = 15 - E;
    }
    if (ws == 0 && kq == 0) {
      tex[tg * 16 + t] = ex;
      if (PRO & PRO_RMS) trs[tg * 16 + t] = rms_scale((double)(ss / (float)a.k + a.eps));
    }
    each([&](int h, int i, uint32_t b) {
      if (b >= nblk) return;
      f4 A = v[h][i][0], C = v[h][i][1];
      if (PRO & PRO_RMS) {
        A *= *(const f4*)(nws + 32 * b + 4 * kq);
        C *= *(const f4*)(nws + 32 * b + 4 * kq + 16);
      }
      const float x8[8] = {A[0], A[2], C[0], C[2], A[1], A[3], C[1], C[3]};
      h8 hi, lo;
      float sx = 0;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float sv = live ? ldexpf(x8[e], ex) : 0.f;
        hi[e] = (_Float16)sv;
        lo[e] = (_Float16)(sv - (float)hi[e]);
        sx += sv;
      }
      h8* dst = xs + (b * TT + tg) * 128 + t * 4 + (kq ^ ((t >> 1) & 3));
      dst[0] = hi;
      dst[64] = lo;
      if (QT == LLMHIP_Q4_1) {
        sx += dpp_mov<DPP_XOR1>(sx);
        sx += dpp_mov<DPP_XOR2>(sx);
        if (kq == 0) bs[b * TT * 16 + tg * 16 + t] = sx;
      }
    });
    __syncthreads();
  }

  // ---- the products
  const h8* xl = xs + r * 4 + (q ^ ((r >> 1) & 3));
  f4 acc[GT][TT], tot[GT][TT], D[TT];
  h8 B, Bn;
  float d = 0.f, dn = 0.f, dp = 0.f, m;
#pragma unroll
  for (int u = 0; u < GT; u++)
#pragma unroll
    for (int t = 0; t < TT; t++) acc[u][t] = tot[u][t] = f4{0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < TT; t++) D[t] = f4{0, 0, 0, 0};
  auto operands = [&](h8 (&A)[TT][2], uint32_t b) {
#pragma unroll
    for (int t = 0; t < TT; t++) {
      A[t][0] = xl[(b * TT + t) * 128];
      A[t][1] = xl[(b * TT + t) * 128 + 64];
    }
  };
  uint32_t cj = 0, cu = ks;  // the unit in the MFMAs
  Epi4In ein[GT][TT];
  auto finish = [&]() __attribute__((always_inline)) {
    const uint32_t tile = t0 + (slot + NW * cj) * GT;
    float* yo = a.y + kp * ra.ystride;
#pragma unroll
    for (int t = 0; t < TT; t++) {
      const uint32_t l = t * 16 + 4 * q;
      typedef int i4 __attribute__((ext_vector_type(4)));
      const i4 ex = *(const i4*)(tex + l);
      f4 rs = f4{1, 1, 1, 1};
      if (PRO & PRO_RMS) rs = *(const f4*)(trs + l);
#pragma unroll
      for (int u = 0; u < GT; u++) {
        f4 v;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          v[i] = ldexpf(acc[u][t][i] + tot[u][t][i], -ex[i]);
          if (PRO & PRO_RMS) v[i] *= rs[i];
        }
        if (EPI == EPI_ACC && LATE) epi4_load<EPI>(ein[u][t], a, tile + u, r, tile + u < t1, g0 * 16 + l);
        epi4<EPI>(a, tile + u, r, tile + u < t1, g0 * 16 + l, v, ein[u][t], yo);
      }
    }
  };
  auto process = [&](WUnit (&W)[GT], auto set) {
    constexpr bool FOLD = !ROLL && decltype(set)::value == 0;  // this unit starts chains of two units' blocks
    const bool last = cu + kw >= units;
    if ((EPI == EPI_QKV || (EPI == EPI_ACC && !LATE)) && last && ks == 0) {
      // the epilogue's inputs, under the tile group's last unit
      const uint32_t tile = t0 + (slot + NW * cj) * GT;
#pragma unroll
      for (int u = 0; u < GT; u++)
#pragma unroll
        for (int t = 0; t < TT; t++) epi4_load<EPI>(ein[u][t], a, tile + u, r, tile + u < t1, (g0 + t) * 16 + 4 * q);
    }
    const uint32_t bu = 4 * cu, n = TAIL ? min(nblk - bu, 4u) : 4;
    h8 A[2][TT][2];
    operands(A[0], bu);
    unit_block<QT, false, true>(W[0], 0, B, d, m);
    float S[TT];
    if (QT == LLMHIP_Q4_1)
#pragma unroll
      for (int t = 0; t < TT; t++) S[t] = bs[min(bu + q, nblk - 1) * TT * 16 + t * 16 + r];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (TAIL && (uint32_t)j >= n) break;
      if (j < 3) operands(A[(j + 1) & 1], TAIL ? min(bu + j + 1, nblk - 1) : bu + j + 1);
#pragma unroll
      for (int u = 0; u < GT; u++) {
        __builtin_amdgcn_sched_barrier(0);
        f4 Dn[TT];
#pragma unroll
        for (int t = 0; t < TT; t++)
          Dn[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[j & 1][t][0], B, f4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
        for (int t = 0; t < TT; t++) Dn[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[j & 1][t][1], B, Dn[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < TT; t++) {
          f4& c = acc[(u + GT - 1) % GT][t];
          if (FOLD && j == 0) {
            tot[(u + GT - 1) % GT][t] += c;
            c = dp * D[t];
          } else {
            c += dp * D[t];
          }
        }
        if (u + 1 < GT) unit_block<QT, false, true>(W[u + 1], j, Bn, dn, m);
        else if (j < 3) unit_block<QT, false, true>(W[0], j + 1, Bn, dn, m);
#pragma unroll
        for (int i = 0; i < 2 * TT; i++) {
          __builtin_amdgcn_sched_group_barrier(8, 1, 0);  // an MFMA, then
          __builtin_amdgcn_sched_group_barrier(2, 3, 0);  // three VALU instructions in its shadow
        }
#pragma unroll
        for (int t = 0; t < TT; t++) D[t] = Dn[t];
        dp = d;
        B = Bn;
        d = dn;
      }
    }
    if (QT == LLMHIP_Q4_1) {
      // the unit's sum of m times the block sums, its four blocks as the k of one f32 MFMA; into the chain that the
      // unit's other products are in, which it largely cancels (into the one before: errors 12% larger)
#pragma unroll
      for (int u = 0; u < GT; u++) {
        const uint32_t lo = q & 1 ? W[u].sv.y : W[u].sv.x, hi = q & 1 ? W[u].sv.w : W[u].sv.z;
        const float mm = f16_hw((q & 2 ? hi : lo) >> 16);  // (0 past the tail)
#pragma unroll
        for (int t = 0; t < TT; t++) acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(S[t], mm, acc[u][t], 0, 0, 0);
      }
    }
    if (!ROLL) fetch(W);
    cu += kw;
    if (ROLL && !((cu >> lkw) & 1))
#pragma unroll
      for (int u = 0; u < GT; u++)
#pragma unroll
        for (int t = 0; t < TT; t++) {
          tot[u][t] += acc[u][t];
          acc[u][t] = f4{0, 0, 0, 0};
        }
    if (!last) return;
    // the tile group is complete
#pragma unroll
    for (int t = 0; t < TT; t++) acc[GT - 1][t] += dp * D[t];
    dp = 0.f;
    if (ROLL && kw > 1) return;  // summed over the tile's waves below
    finish();
#pragma unroll
    for (int u = 0; u < GT; u++)
#pragma unroll
      for (int t = 0; t < TT; t++) acc[u][t] = tot[u][t] = f4{0, 0, 0, 0};
    cu = ks;
    cj++;
  };
  if constexpr (ROLL) {
    for (uint32_t i = 0; i < steps_n; i++) {
      WUnit cur[GT];
#pragma unroll
      for (int u = 0; u < GT; u++) cur[u] = w[0][u];
      fetch(w[0]);
      process(cur, std::integral_constant<int, 0>());
    }
    if (kw > 1) {  // uniform over the workgroup
      f4* ps = (f4*)lds;  // [NW][TT][64], in the operands' place (a wave has at least 1 KB of them per token group)
      __syncthreads();
#pragma unroll
      for (int t = 0; t < TT; t++) {
        tot[0][t] += acc[0][t];
        acc[0][t] = f4{0, 0, 0, 0};
        ps[(wave * TT + t) * 64 + lane] = tot[0][t];
      }
      __syncthreads();
      if (ks == 0 && mine) {
        for (uint32_t i = 1; i < kw; i++)
#pragma unroll
          for (int t = 0; t < TT; t++) tot[0][t] += ps[((wave + i) * TT + t) * 64 + lane];
        finish();
      }
    }
  } else {
    uint32_t i = 0;
    for (; i + 1 < steps_n; i += 2) {
      process(w[0], std::integral_constant<int, 0>());
      process(w[1], std::integral_constant<int, 1>());
    }
    if (i < steps_n) process(w[0], std::integral_constant<int, 0>());
  }
}

template <uint32_t QT, int PRO, int EPI, int TT, int GT, bool TAIL, int NW>
static int resident_go(const GemvArgs& a, const ResArgs& ra0, const ResPlan& p, hipStream_t s) {
  auto k = resident_kernel<QT, PRO, EPI, TT, GT, TAIL, NW>;
  LLM_TRY((allow_lds<resident_kernel<QT, PRO, EPI, TT, GT, TAIL, NW>>(RES_LDS)));
  ResArgs ra = ra0;
  ra.ttiles = (a.ntok + 16 * TT - 1) / (16 * TT);
  ra.lkw = p.lkw;
  hipLaunchKernelGGL(k, dim3(res_blocks(ra.ttiles, ra.rparts * ra.kparts)), dim3(64 * NW), p.lds, s, a, ra);
  LLM_HIP(hipGetLastError());
  return 0;
}

template <uint32_t QT, int PRO, int EPI, int TT, int GT, int NW>
static int resident_tail(const GemvArgs& a, const ResArgs& ra, const ResPlan& p, hipStream_t s) {
  return a.tail ? resident_go<QT, PRO, EPI, TT, GT, true, NW>(a, ra, p, s)
                : resident_go<QT, PRO, EPI, TT, GT, false, NW>(a, ra, p, s);
}

// The forms of RES_FORMS.
template <uint32_t QT, int PRO, int EPI>
static int resident_form(const GemvArgs& a, const ResArgs& ra, const ResPlan& p, hipStream_t s) {
  const uint32_t f = p.tt * 1000 + p.gt * 100 + p.nw;
  if (f == 1108) return resident_tail<QT, PRO, EPI, 1, 1, 8>(a, ra, p, s);
  if (f == 1116) return resident_tail<QT, PRO, EPI, 1, 1, 16>(a, ra, p, s);
  if (f == 1216) return resident_tail<QT, PRO, EPI, 1, 2, 16>(a, ra, p, s);
  if (f == 2208) return resident_tail<QT, PRO, EPI, 2, 2, 8>(a, ra, p, s);
  if constexpr (EPI != EPI_QKV)
    if (f == 2408) return resident_tail<QT, PRO, EPI, 2, 4, 8>(a, ra, p, s);
  return set_error(LLMHIP_ERR_ARG, "llm: resident product: no form of %u token groups, %u tiles, %u waves", p.tt, p.gt,
                   p.nw);
}

template <uint32_t QT, int EPI, int TT, int GT, int NW>
static int resident_allow() {
  LLM_TRY((allow_lds<resident_kernel<QT, PRO_PLAIN, EPI, TT, GT, true, NW>>(RES_LDS)));
  return allow_lds<resident_kernel<QT, PRO_PLAIN, EPI, TT, GT, false, NW>>(RES_LDS);
}

template <uint32_t QT, int EPI>
static int resident_allow_epi() {
  LLM_TRY((resident_allow<QT, EPI, 1, 1, 8>()));
  LLM_TRY((resident_allow<QT, EPI, 1, 1, 16>()));
  LLM_TRY((resident_allow<QT, EPI, 1, 2, 16>()));
  LLM_TRY((resident_allow<QT, EPI, 2, 2, 8>()));
  return resident_allow<QT, EPI, 2, 4, 8>();
}

// The current device lets every form of the plain products (EPI_STORE, EPI_ACC)
// have its LDS: a launch after it makes no other runtime call.
template <uint32_t QT>
int resident_ready_qt() {
  LLM_TRY((resident_allow_epi<QT, EPI_STORE>()));
  return resident_allow_epi<QT, EPI_ACC>();
}

template <uint32_t QT>
int resident_launch_qt(const GemvArgs& a, const ResArgs& ra, const ResPlan& p, int pro, int epi, hipStream_t s) {
  switch (pro * 8 + epi) {
    case PRO_PLAIN * 8 + EPI_STORE: return resident_form<QT, PRO_PLAIN, EPI_STORE>(a, ra, p, s);
    case PRO_PLAIN * 8 + EPI_ACC: return resident_form<QT, PRO_PLAIN, EPI_ACC>(a, ra, p, s);
    case PRO_RMS * 8 + EPI_QKV: return resident_form<QT, PRO_RMS, EPI_QKV>(a, ra, p, s);
    case PRO_RMS * 8 + EPI_GATEUP: return resident_form<QT, PRO_RMS, EPI_GATEUP>(a, ra, p, s);
  }
  return set_error(LLMHIP_ERR_ARG, "llm: resident product: unsupported prologue/epilogue %d/%d", pro, epi);
}

}  // namespace llmhip
