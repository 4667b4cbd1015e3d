// Tiled int8-activation GEMM for the engine-signature calls with more than 16 rows: tile
// geometry, coverage and launch (the kernel is in prefill_i8_kernel.h; the weight kinds are
// instantiated in prefill_i8_w8.hip, prefill_i8_w4.hip and prefill_i8_w4z.hip).
#include <stdlib.h>

#include <algorithm>

#include "prefill_i8_kernel.h"

namespace qlin {

void prefill_i8_geometry(int tile, int* bm, int* bn) {
  static const int kBm[I8_TILES] = {128, 64, 96, 128, 160};
  *bm = kBm[tile];
  *bn = tile == I8_128x128 ? 128 : 64;
}

// Whether the tiled kernel covers a call with a tile shape.
bool prefill_i8_ok(const SkArgs& a, int wk, int epi, int tile) {
  if (a.M <= 16 || a.K % 64 != 0 || ((uintptr_t)a.x & 15) != 0) return false;
  // the copies address activations, their scales and each weight matrix with buffer
  // offsets computed in 31 bits
  if ((long long)a.M * a.K >= (1LL << 31) || (long long)a.M * (a.K / 64) * 4 >= (1LL << 31)) return false;
  for (int s = 0; s < a.nseg; ++s)
    if ((long long)a.K * a.seg[s].n >= (1LL << 31)) return false;
  if (wk == WK_W4 && a.group < 64) return false;
  int bm, bn;
  prefill_i8_geometry(tile, &bm, &bn);
  const int nsets = (epi == EPI_STORE) ? a.nseg : 1;  // gate/up: one column range, two weight sets
  for (int s = 0; s < nsets; ++s)
    if (a.seg[s].n % bn != 0) return false;
  return true;
}

hipError_t launch_prefill_i8(SkArgs a, int wk, bool hz, int epi, int tile, hipStream_t st) {
  int BM, bn;
  prefill_i8_geometry(tile, &BM, &bn);
  int tn = 0;
  if (epi == EPI_STORE) {
    for (int s = 0; s < a.nseg; ++s) {
      a.seg[s].tile0 = tn;
      tn += a.seg[s].n / bn;
    }
  } else {
    a.seg[0].tile0 = a.seg[1].tile0 = 0;
    tn = a.seg[0].n / bn;
  }
  a.ntiles = tn;
  if (a.splits < 1) a.splits = 1;
  const int tiles = ((a.M + BM - 1) / BM) * tn * a.splits;
  // Tile order: each XCD runs one contiguous eighth of it, going down gm row tiles
  // before the next column tile; gm minimises what a run reads into its XCD's L2: rows
  // x (BM x K int8 activations) + columns x (the weights of bn columns, every set).
  // QLIN_I8_GM overrides it (0: groups of 8 row tiles, workgroups in launch order).
  const char* eg = getenv("QLIN_I8_GM");
  if (eg && *eg) {
    a.gm = atoi(eg) > 0 ? atoi(eg) : 0;
  } else {
    const long long tm = (a.M + BM - 1) / BM;
    const long long run = std::max<long long>(1, (tm * tn + 7) / 8);
    const double arow = (double)BM * a.K, wcol = (double)a.K * bn * (wk == WK_W4 ? 0.5 : 1.0) * (epi == EPI_STORE ? 1 : 2);
    double best_c = 0.0;
    for (int gm = 1; gm <= 64; gm *= 2) {
      const long long h = std::min<long long>(gm, tm);
      const long long rows = std::min(h, run), cols = (run + h - 1) / h;
      const double c = (double)rows * arow + (double)cols * wcol;
      if (gm == 1 || c < best_c) best_c = c, a.gm = gm;
      if (gm >= tm) break;
    }
  }
  if (wk == WK_W8) return launch_i8_w<WK_W8, false>(a, epi, tile, tiles, st);
  if (hz) return launch_i8_w<WK_W4, true>(a, epi, tile, tiles, st);
  return launch_i8_w<WK_W4, false>(a, epi, tile, tiles, st);
}

}  // namespace qlin
