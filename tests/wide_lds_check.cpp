// Host replay of fwd_wide_kernel's addressing (htree_amd/csrc/htree_fwd_wide.h)
// against the LDS layout its launch allocates (wide_lds() of htree_common.h, the
// function the kernel, its launch and make_plan call).  For every configuration
// the library accepts on the wide path (top_k > 64 or more than 64 candidate
// tiles; top_k <= 1024, top_k * CR <= 16384, CR in [4, 128], D in {32, 64, 128, 256};
// one part, and the two parts of a KV-head pair where their layout fits
// 160 KB) and every configuration with the four parts of a KV-head quad
// (any level size) where their layout fits 160 KB, and every level shape (np
// parents, child index ct of the query), it forms each LDS index, list slot and
// RoPE row of
//   * the pass-down of a level of at most top_k candidates,
//   * the importance batches (tiles clamped to the last one, the next batch's
//     keys and table rows, the tab rows of D = 32),
//   * the selection's keys (whole runs of C positions, of which only those below
//     nc count), its list and bit writes,
//   * the accumulation's batches in each form (slots past the list, the query
//     turned back from them, the selection words), and the merge,
// and checks it against its region where the value counts, against the
// allocation where it is dropped.  The regions are disjoint and, with the
// static rows, inside 160 KB.  Test infrastructure: built and run by
// tests/test_wide_lds.py on the CPU.
#include <cstdio>
#include <cstdlib>

#include "htree_common.h"

using namespace htree;

static int fails = 0;
#define CHECK(c, ...)                                             \
  do {                                                            \
    if (!(c)) {                                                   \
      if (fails < 20) {                                           \
        std::printf("FAIL %s: ", #c);                             \
        std::printf(__VA_ARGS__);                                 \
        std::printf("\n");                                        \
      }                                                           \
      ++fails;                                                    \
    }                                                             \
  } while (0)

static void check_config(int TK, int CR, int D, int parts) {
  int crlg = 0;
  while ((1 << crlg) < CR) ++crlg;
  const int max_tiles = TK * (CR > 16 ? CR : 16) / 16;  // make_plan
  const int maxpos = TK << crlg;                        // launch: TK << crlg
  const WideLds w = wide_lds(TK, maxpos, max_tiles, D, parts);
  const int NW = kWideWaves / parts;                    // waves per part
  const int C = maxpos > kWideMidPos ? 2 * kWideC : kWideC;  // the launch's choice
  const int U = kWideBatch, UA = D <= 64 ? 4 : 1;       // tiles of a batch
  const bool wide = CR >= 16;
  const int CRU = CR < 16 ? CR : 16, lgt = wide ? 4 : crlg;
  const int rows = maxpos;  // RoPE rows make_plan asks for (and more than CR of them)
  const int words = (maxpos + 31) / 32;
  const long imp_floats = (w.bytes - w.imp) / 4, lds_floats_from_mt = (w.bytes - w.mt) / 4;
  // ---- regions: par | selw | mt | red | imp, the static rows beside them
  CHECK(256 * C >= maxpos, "TK %d CR %d: %d keys per thread", TK, CR, C);
  CHECK(w.par == 0 && 2L * TK * 4 <= w.selw && w.selw + 4L * words <= w.mt, "par / selw / mt");
  CHECK(w.mt + 4L * max_tiles * parts <= w.red && w.red + 256 <= w.imp, "mt / red / imp");
  CHECK(4L * 36 <= 256, "red: counts, scans, maxima");
  CHECK(4L * maxpos * parts <= w.bytes - w.imp, "importance of every part");
  CHECK(w.imp % 16 == 0 && w.mt % 4 == 0 && w.red % 4 == 0, "alignment");
  CHECK(w.total == w.bytes + (D == 32 ? 2048 : 0) && w.total <= 160 * 1024, "total %d", w.total);
  CHECK(CR < rows || maxpos == CR, "row of the angle CR");  // (rope_rows > CR is a rule of its own)
  // ---- tab (D = 32): element lane + 64 k of a wave's rows, read at D j (+ D / 2) + 8 (kg & 1) .. + 7
  if (D == 32) {
    CHECK((63 + 64 * (U * D / 64 - 1)) < wide_tab_floats(D), "tab write");
    CHECK(D * (U - 1) + D / 2 + 8 + 7 < wide_tab_floats(D), "tab read");
    for (int i = 0; i < U * D; ++i) CHECK(i / D < U, "tab row");
  }
  // ---- keys: thread tid reads positions C tid .. C tid + C - 1 of every part in 16-byte runs
  for (int tid = 0; tid < 256; ++tid) {
    if ((long)tid * C < maxpos)  // (the selection words it writes)
      CHECK((tid + 1) * (C / 32) <= words, "selw of thread %d, maxpos %d", tid, maxpos);
    for (int j = 0; j < parts; ++j)
      for (int i4 = 0; i4 < C; i4 += 4) {
        const int pos = tid * C + i4;
        if ((long)tid * C >= maxpos) continue;  // tid * C < nc <= maxpos
        CHECK((j * maxpos + pos) % 4 == 0, "16-byte run at %d", j * maxpos + pos);
        CHECK(j * maxpos + pos + 3 < imp_floats, "TK %d CR %d D %d: imp run %d of part %d past the allocation",
              TK, CR, D, pos, j);
        CHECK(j * max_tiles + (pos >> lgt) < lds_floats_from_mt, "mt of run %d past the allocation", pos);
        if (pos < maxpos) {  // a run with a candidate in it: one tile, this part's regions
          CHECK((pos >> lgt) == ((pos + 3) >> lgt) && (pos >> lgt) < max_tiles, "run %d in one tile", pos);
          CHECK(pos + 3 < maxpos, "run %d in the part's importances", pos);
        }
      }
  }
  // ---- every level shape
  for (int np = 1; np <= TK; ++np)
    for (int ct = 0; ct < CR; ++ct) {
      const int nc = ((np - 1) << crlg) + ct + 1, apos = nc - 1;
      const int nt = wide ? (nc + 15) >> 4 : np;
      CHECK(nc <= maxpos && nt <= max_tiles, "nc %d nt %d", nc, nt);
      auto slot_of = [&](int tau) { return wide ? (tau << 4) >> crlg : tau; };
      auto tile_ok = [&](int tau, const char* what) {
        CHECK(tau >= 0 && tau < nt && slot_of(tau) < np, "%s: tile %d of %d, np %d", what, tau, nt, np);
        // its first candidate exists, so its node's 16-node block does
        CHECK((wide ? tau << 4 : tau << crlg) < nc, "%s: first candidate of tile %d", what, tau);
      };
      // a level passed down: pc[i >> crlg] of nc positions, nc <= TK entries written
      if (nc <= TK) CHECK(((nc - 1) >> crlg) < np, "pass-down");
      // importance
      for (int wvh = 0; wvh < NW; ++wvh)
        for (int i0 = wvh; i0 < nt; i0 += U * NW)
          for (int j = 0; j < U; ++j) {
            const int tau = i0 + NW * j < nt ? i0 + NW * j : nt - 1;
            tile_ok(tau, "importance");
            const int prow = apos - (slot_of(tau) << crlg);
            CHECK(prow >= 0 && prow < rows, "row %d", prow);
            const int nx = i0 + U * NW < nt ? i0 + U * NW : i0;
            tile_ok(nx + NW * j < nt ? nx + NW * j : nt - 1, "next batch");
          }
      for (int tk = 0; tk < nt; ++tk) {  // stores: mt[tk], imp[(tk << lgt) + u] where a candidate
        CHECK(tk < max_tiles, "mt store");
        const int last = (tk << lgt) + CRU - 1 < nc ? (tk << lgt) + CRU - 1 : nc - 1;
        CHECK(last < maxpos, "imp store");
      }
      // the selection: pn[idx] (idx < take), pc[pos >> crlg] (pos < nc)
      CHECK((TK < nc ? TK : nc) <= TK && ((nc - 1) >> crlg) < np, "list");
      // accumulation: batch bi of UA tiles by wave bi mod NW
      const int nb = (nt + UA - 1) / UA;
      for (int bi = 0; bi < nb; ++bi)
        for (int j = 0; j < UA; ++j) {
          const int tau0 = bi * UA, tau = tau0 + j < nt ? tau0 + j : nt - 1;
          tile_ok(tau, "accumulation");
          CHECK((tau << lgt) >> 5 < words, "selection word of tile %d", tau);
          // one word holds the tile's bits (FORM 0 and 2)
          CHECK((((tau << lgt) & 31) + CRU) <= 32, "bits of tile %d", tau);
          // FORM 0 (whole tiles of the top level's nodes 0 .. apos)
          if (UA > 1 && wide) CHECK(16 * tau <= apos, "top-level tile %d", tau);
          // FORM 1 (CR 16, TK >= UA): slots past the list, and the rows turned back from them
          if (UA > 1 && CR == 16 && TK >= UA) {
            CHECK(tau0 + j < TK, "pc[%d] of %d", tau0 + j, TK);
            const int prow = apos - ((tau0 + j) << crlg);
            CHECK((prow < 0 ? -prow : prow) < rows, "row %d", prow);
          }
          // FORM 2
          const int prow = apos - (slot_of(tau) << crlg);
          CHECK(prow >= 0 && prow < rows, "row %d", prow);
        }
    }
  // ---- each part's waves merge in the importance area, part hf from byte
  // merge_part * hf: mw, lw then ow rows of D + 1
  const int DP = D + 1;
  for (int hf = 0; hf < parts; ++hf) {
    const long base = (long)hf * w.merge_part / 4;
    const long last_ow = base + 2L * NW * 16 + (long)((NW - 1) * 16 + 15) * DP + (D - 1);
    CHECK(last_ow < imp_floats, "TK %d CR %d D %d: merge index %ld of %ld", TK, CR, D, last_ow,
          imp_floats);
    CHECK(last_ow < (long)(hf + 1) * w.merge_part / 4, "merge regions of parts %d, %d", hf, hf + 1);
  }
  CHECK(w.merge_part % 4 == 0 && w.merge_part >= 4 * (2 * NW * 16 + NW * 16 * DP), "merge region size");
  // the parent-list rows: part hf's waves (threads 64 NW hf .. 64 NW (hf + 1) - 1)
  // write entries i = tid - 64 NW hf, stride 64 NW
  for (int tid = 0; tid < 256; ++tid) {
    const int hf = (tid >> 6) / NW;
    const int i0 = tid - hf * 64 * NW;
    CHECK(hf < parts && i0 >= 0 && i0 < 64 * NW, "parent-row index of thread %d", tid);
  }
}

int main() {
  int n = 0, refused = 0;
  for (int D : {32, 64, 128, 256})
    for (int CR = 4; CR <= 128; CR *= 2)
      for (int TK = 1; TK <= kWideMaxTK; TK *= 2) {
        if ((long)TK * CR > kWideMaxPos) continue;
        const int max_tiles = TK * (CR > 16 ? CR : 16) / 16;
        const bool wide = max_tiles > kMaxTiles || TK > kMaxTK;  // make_plan
        for (int parts : {1, 2, 4}) {
          if (parts < 4 && !wide) continue;  // (quads: any level size)
          const WideLds w = wide_lds(TK, TK * CR, max_tiles, D, parts);
          // the static rows take no configuration from the wide form
          refused += w.bytes <= 160 * 1024 && w.total > 160 * 1024;
          if (parts > 1 && w.total > 160 * 1024) continue;  // make_plan: the split selection
          check_config(TK, CR, D, parts);
          ++n;
        }
      }
  CHECK(refused == 0, "%d layouts only fit without their static rows", refused);
  std::printf("%d wide configurations checked, %d failures\n", n, fails);
  return fails ? 1 : 0;
}
