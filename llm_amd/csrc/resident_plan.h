// How a many-token product with resident activations (resident.h) is laid out
// on the GPU: host-side plan, plain C++.
#pragma once

#include <algorithm>
#include <cstdint>

#if defined(__HIP__)
#define RES_HD __host__ __device__
#else
#define RES_HD
#endif

namespace llmhip {

constexpr uint32_t RES_LDS = 160 * 1024;  // LDS of a workgroup (one per CU)
constexpr uint32_t RES_ITEMS = 10;        // staged items per lane, at most

// What a resident launch takes beside GemvArgs.
struct ResArgs {
  uint32_t ttiles;  // token tiles
  uint32_t rparts;  // workgroups along the rows, part p tiles [p tiles / rparts, (p + 1) tiles / rparts)
  uint32_t lkw;     // log2 of the waves that share a tile (one tile per group only)
  uint32_t kparts, kunits;  // workgroups along k, each kunits units of four blocks; part p's product goes to y + p * ystride
  uint64_t ystride;
  // PRO_RMS: the row is parts[0] + parts[pstride] + ... + x (nparts of them, added in that order), and xout
  // (null: not) receives it
  const float* parts;
  uint64_t pstride;
  uint32_t nparts;
  float* xout;
};

// The token tile and column (row part and k part) of workgroup b.  Workgroup b
// runs on XCD b % 8; an XCD takes a contiguous range of the (token tile,
// column) pairs, columns within token tiles, so that the columns of a token
// tile read its activations through one XCD's L2 (with the columns dealt round,
// every XCD read every row: the staging of 1024 tokens' rows and four parts
// took 40 us).  false: no work.
RES_HD inline bool res_place(uint32_t b, uint32_t ttiles, uint32_t cols, uint32_t* tile, uint32_t* col) {
  const uint32_t n = ttiles * cols, x = b % 8, s = x * n / 8, l = s + b / 8;
  *tile = l / cols;
  *col = l - *tile * cols;
  return l < (x + 1) * n / 8;
}
inline uint32_t res_blocks(uint32_t ttiles, uint32_t cols) { return (ttiles * cols + 7) / 8 * 8; }

struct ResPlan {
  // token groups, tiles per group and waves of a workgroup; row parts, k parts, units per k part; bytes of LDS
  // (tt = 0: the product does not fit)
  // lkw: log2 of the waves that share a tile
  uint32_t tt = 0, gt = 0, nw = 0, rparts = 0, kparts = 0, kunits = 0, lds = 0, lkw = 0;
};

// LDS of nblk blocks of tt token groups: the operands, the staging's partial
// reductions and the token scalars, and (sums) the block sums of Q4_1.
inline uint32_t res_lds(uint32_t nblk, uint32_t tt, bool rms, bool sums) {
  return nblk * tt * 2048 + 2048 + 64 + tt * 16 * 8 + (rms ? nblk * 128 : 0) + (sums ? nblk * tt * 64 : 0);
}

// Microseconds, as measured on MI355X (res_plan only compares them): a step
// (a block of one tile for 16 tt tokens) of each of `busy` waves at once on a
// SIMD, and a workgroup's staging of nblk blocks with its launch.
struct ResCost {
  static double step(uint32_t tt, uint32_t gt, double busy) {
    const double alone = tt == 2 ? 0.075 : 0.055;  // one wave by itself: latency
    const double full = tt == 2 ? (gt == 4 ? 0.052 : 0.055) : (gt == 2 ? 0.036 : 0.040);
    return std::max(alone, full * busy);
  }
  static double stage(uint32_t tt, uint32_t nblk, uint32_t nw) { return 1.5 + (nw == 16 ? 0.04 : 0.05) * tt * nblk; }
  // a part of k more: its product stored and read again by the next RMSNorm
  static double part(uint32_t ntok) { return 0.4 + 0.0016 * ntok; }
};

// The forms the kernel is built in: token groups, tiles per group, waves.  (Two
// token groups with many tiles spill in the epilogue of the [q; k; v] product,
// whose inputs are the most: not built there.)
struct ResForm {
  uint32_t tt, gt, nw;
  bool qkv;
};
constexpr ResForm RES_FORMS[] = {{1, 1, 8, true},  {1, 1, 16, true},  {1, 2, 16, true},
                                 {2, 2, 8, true},  {2, 4, 8, false}};

// The layout of a product of `tiles` row tiles by nb blocks for ntok tokens
// (rms: PRO_RMS; qkv: EPI_QKV; sums: Q4_1), over at most kmax parts of k: the
// one of least estimated time among the forms and the row splits that give
// every wave whole tile groups or the chip whole rounds of workgroups.
// tt == 0: no part of k in any form fits the staging and the LDS.
inline ResPlan res_plan(uint32_t tiles, uint32_t nb, uint32_t ntok, bool rms, bool qkv, bool sums, uint32_t kmax,
                        uint32_t cus = 256) {
  ResPlan best;
  double least = 0;
  const uint32_t units = (nb + 3) / 4;
  for (const ResForm& f : RES_FORMS) {
    if ((f.tt == 2 && ntok <= 16) || (qkv && !f.qkv)) continue;
    const uint32_t groups = (ntok + 16 * f.tt - 1) / (16 * f.tt);
    for (uint32_t k = 1; k <= kmax && k <= units; k++) {
      const uint32_t kunits = (units + k - 1) / k, nblk = std::min(nb, 4 * kunits), lds = res_lds(nblk, f.tt, rms, sums);
      if ((units + kunits - 1) / kunits != k || nblk > RES_ITEMS * (8 / f.tt) || lds > RES_LDS) continue;
      auto consider = [&](uint32_t rp) {
        if (rp < 1 || rp > tiles) return;
        // the kernel's row split and place are 32-bit
        if ((uint64_t)tiles * rp >> 32 || (uint64_t)groups * rp * k >> 28) return;
        const uint32_t grps = ((tiles + rp - 1) / rp + f.gt - 1) / f.gt, rounds = (groups * rp * k + cus - 1) / cus;
        const uint32_t per = (grps + f.nw - 1) / f.nw;
        const double busy = std::max(1.0, std::min(grps, f.nw) / 4.0);  // waves at work on a SIMD
        const double t = rounds * (ResCost::stage(f.tt, nblk, f.nw) +
                                   per * (f.gt * nblk * ResCost::step(f.tt, f.gt, busy) + 0.3)) +
                         (k - 1) * ResCost::part(ntok);
        if (best.tt && t >= least) return;
        least = t;
        best = ResPlan{f.tt, f.gt, f.nw, rp, k, kunits, lds, 0};
        // waves share a tile where the workgroup has at most one tile per SIMD (each then waits for its own chain of
        // steps: prefill of 128 tokens 1389 -> 1329 us; with five tiles, 4864x896 for 64 tokens, 7.9 -> 8.1), each
        // has a unit, and their sums a place in the operands' LDS (of the last part of k too, the shortest)
        const uint32_t least_blk = nb - (k - 1) * 4 * kunits;
        if (f.gt == 1 && grps <= 4 && least_blk * 2 >= f.nw)
          while (best.lkw < 3 && (grps << (best.lkw + 1)) <= f.nw && kunits >= (2u << best.lkw)) best.lkw++;
      };
      for (uint32_t m = 1; m <= 32; m++) {  // m tile groups for every wave
        const uint32_t rp = (tiles + f.nw * f.gt * m - 1) / (f.nw * f.gt * m);
        consider(rp);
        if (rp == 1) break;
      }
      for (uint32_t r = 1; r <= 3; r++) consider(r * cus / (groups * k));  // r whole rounds of workgroups
    }
  }
  return best;
}

}  // namespace llmhip
