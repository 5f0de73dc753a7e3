// Checks res_plan / res_place (llm_amd/csrc/resident_plan.h) over a range of
// shapes: every (token tile, row part, k part) belongs to one workgroup, the
// row parts and the k parts cover the matrix, and staging and LDS hold what
// the kernel puts there.  Prints "ok <plans>" or the first plan that is wrong.
#include "../llm_amd/csrc/resident_plan.h"

#include <cstdio>
#include <vector>

using namespace llmhip;

int main() {
  unsigned long plans = 0, shared = 0;
  for (uint32_t tiles : {1u, 3u, 7u, 36u, 56u, 72u, 608u, 9496u})
    for (uint32_t nb : {1u, 2u, 4u, 6u, 18u, 28u, 38u, 48u, 78u, 152u, 400u})
      for (uint32_t ntok : {1u, 5u, 16u, 17u, 37u, 64u, 65u, 127u, 128u, 257u, 701u, 1023u, 1024u})
        for (int mode = 0; mode < 16; mode++) {
          const bool rms = mode & 1, qkv = mode & 2, sums = mode & 4;
          const uint32_t kmax = mode & 8 ? 8 : 1, units = (nb + 3) / 4;
          const ResPlan p = res_plan(tiles, nb, ntok, rms, qkv, sums, kmax);
          const bool one = nb <= RES_ITEMS * 8 && res_lds(nb, 1, rms, sums) <= RES_LDS;  // whole rows of 16 tokens
          auto bad = [&](const char* what) {
            printf("%s: tiles %u nb %u ntok %u mode %d -> tt %u gt %u nw %u rparts %u kparts %u kunits %u lds %u\n", what, tiles,
                   nb, ntok, mode, p.tt, p.gt, p.nw, p.rparts, p.kparts, p.kunits, p.lds);
            return 1;
          };
          if (!p.tt) {
            if (one) return bad("no plan");
            continue;
          }
          plans++;
          bool form = false;
          for (const ResForm& f : RES_FORMS) form = form || (f.tt == p.tt && f.gt == p.gt && f.nw == p.nw && (f.qkv || !qkv));
          if (!form) return bad("form");
          if (p.kparts < 1 || p.kparts > kmax || p.kparts * p.kunits < units || (p.kparts - 1) * p.kunits >= units)
            return bad("k parts");
          const uint32_t nblk = nb < 4 * p.kunits ? nb : 4 * p.kunits;
          // what the kernel stages: NI items twice per lane, NW / TT waves per token group
          const uint32_t ni = (RES_ITEMS * 8 / p.nw + 1) / 2;
          if (nblk > 2 * ni * (p.nw / p.tt)) return bad("staged items");
          if (nblk * 32 > ((RES_ITEMS * 8 * 32 + 64 * p.nw * 4 - 1) / (64 * p.nw * 4)) * 64 * p.nw * 4) return bad("norm weights");
          if (p.lds != res_lds(nblk, p.tt, rms, sums) || p.lds > RES_LDS) return bad("lds");
          if (p.rparts < 1 || p.rparts > tiles) return bad("row parts");
          if (p.lkw) {  // waves that share a tile: one round of tiles, a unit each, and room for their sums
            const uint32_t last = nb - (p.kparts - 1) * 4 * p.kunits;
            if (p.gt != 1 || (((tiles + p.rparts - 1) / p.rparts) << p.lkw) > p.nw || p.kunits < (1u << p.lkw) ||
                last * p.tt * 2048 < p.nw * p.tt * 1024)
              return bad("shared tiles");
            shared++;
          }
          uint32_t at = 0;
          for (uint32_t r = 0; r < p.rparts; r++) {
            const uint32_t t0 = r * tiles / p.rparts, t1 = (r + 1) * tiles / p.rparts;
            if (t0 != at || t1 <= t0) return bad("row split");
            at = t1;
          }
          if (at != tiles) return bad("row split end");
          const uint32_t ttiles = (ntok + 16 * p.tt - 1) / (16 * p.tt), cols = p.rparts * p.kparts;
          std::vector<uint8_t> seen((size_t)ttiles * cols, 0);
          for (uint32_t b = 0; b < res_blocks(ttiles, cols); b++) {
            uint32_t t, c;
            if (!res_place(b, ttiles, cols, &t, &c)) continue;
            if (t >= ttiles || c >= cols || seen[(size_t)t * cols + c]++) return bad("place");
          }
          for (uint8_t s : seen)
            if (s != 1) return bad("not placed");
        }
  if (!shared) {
    printf("no plan shares tiles\n");
    return 1;
  }
  printf("ok %lu\n", plans);
  return 0;
}
