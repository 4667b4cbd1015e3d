// extern "C" entry points of libqlin.so (declared in include/qlin.h).
//
// Every entry point validates its arguments (shape, group, dtype, alignment) and
// returns a status before anything is launched; the launch plan (column tile width,
// waves per workgroup, split-K) is chosen here from K and N.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>

#include "../../include/qlin.h"
#include "qlin_dev.h"
#include "qlin_internal.h"

using namespace qlin;

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int hip_status(const char* fn, hipError_t e) {
  if (e == hipSuccess) return QLIN_OK;
  return fail(QLIN_ERR_HIP, "%s: HIP error %d (%s)", fn, (int)e, hipGetErrorString(e));
}

// Fill kernel behind clear_counters (a kernel node, not a memset, so a call that clears
// its counters can be captured in a graph).
__global__ void zero_u32(unsigned* p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0u;
}

#define QL_TRY(expr)              \
  do {                            \
    const int rc_ = (expr);       \
    if (rc_ != QLIN_OK) return rc_; \
  } while (0)


// Workspace: [counters | polling-exchange slots | partial sums].  Counters and slots
// must be zero between calls (every kernel leaves them so; the slots are used only by
// the engine decode units' polling exchange).
constexpr size_t kWorkspaceBytes = size_t(256) << 20;
constexpr size_t kCounterBytes = size_t(1) << 20;
constexpr size_t kPollBytes = size_t(4) << 20;
constexpr size_t kPartBase = kCounterBytes + kPollBytes;
constexpr int kWideTiles = 512;          // 256-column tiles at which no K split is needed
// narrow launches: most waves to spread K over, and least K per wave (measured with
// 8-wave workgroups: many short waves keep the most weight bytes in flight)
constexpr long long kTargetWavesW8 = 2048;
constexpr long long kTargetWavesW4 = 1024;
constexpr int kMinWaveKW8 = 64;
// fp16-activation W8 launches of at most this many (column tile x 32-row) units run
// one 32-row step per wave (measured: 2048x2048 and 2048x512 gain 0.4-0.9 us per
// launch; larger launches lose with that many workgroups)
constexpr long long kOneStepUnits = 1024;
constexpr int kMinWaveKW4 = 128;
// largest one-pass tile (weight bytes per set; measured with the weights streaming
// from HBM: 64 KB tiles win, 128 KB tiles lose to split-K)
constexpr long long kOnePassTileBytes = 64 * 1024;

bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }
bool dtype_scale_ok(int dt) { return dt == QLIN_F16 || dt == QLIN_BF16 || dt == QLIN_F32; }
bool dtype_out_ok(int dt) { return dt == QLIN_F16 || dt == QLIN_BF16; }
bool group_ok(int g) { return g == 32 || (g > 0 && g % 64 == 0); }


struct Problem {
  int act, wk, epi;
  bool hz;
  int M, K, group;
  int nsets;  // weight sets per output tile (1, or 2 for gate/up)
  int ncols;  // total output columns
};

// Fills L (kernel variant, grid, LDS) and a.kchunk / a.splits / a.ntiles / seg tiles.
// Launch-plan override for tuning sweeps: QLIN_SKINNY_PLAN="cols,waves,units" (0 keeps
// the default for that field; units = K granules of one wave).  Unset in normal use.
void plan_override(const Problem& P, int& cols, int& waves, int& upw) {
  const char* e = getenv("QLIN_SKINNY_PLAN");
  if (!e || !*e) return;
  int c = 0, w = 0, u = 0;
  if (sscanf(e, "%d,%d,%d", &c, &w, &u) != 3) return;
  if (c == 4 || c == 8 || c == 16) cols = c;
  if (P.epi != EPI_STORE && cols == 16) cols = 8;  // gate/up kernels: 4- and 8-column tiles
  if (w >= 1 && w <= 16) waves = w;  // clamped to the variant's maximum by the caller
  if (u >= 1) upw = u;
}

// ---------------------------------------------------------------------------
// Engine-signature calls with at least kRowsM rows (prefill chunks, chunk remainders)
//
// One K order for every M: the result of a row depends on (K, N) and the call kind,
// never on M, on the chunking of a prompt or on which kernel family runs, so a
// chunked prefill equals an unchunked one bit for bit.  The order is the tiled int8
// kernel's: K/64 blocks in S contiguous splits; within a split, lane 0 folds the
// blocks at even offsets and lane 1 those at odd offsets (acc = fma(float(dot),
// scale, acc) from zero, in increasing K); split value = lane 0 + lane 1; total =
// ((v0 + v1) + v2) + ...; then the W8 column scale (and residual, one rounding).
// The 16-row skinny tiles reproduce it with two waves per split (lanes == 2).
// S is chosen for the engine's 512-row chunk and then held for every M.
// Calls with fewer rows (decode: one sequence, or up to eight best-of candidates,
// engine.py:392) run the engine decode work units (echain.hip), whose results depend
// on (K, N) and the call kind only, so batch rows equal single rows; a chunk remainder
// of 1-8 rows therefore agrees with the unchunked prefill to the tolerance, not bit
// for bit.
constexpr int kRowsM = kDecodeRowsMax + 1;
constexpr int kRefChunkM = 512;

// Column tiles of `tn` over the call's column ranges.
long long col_tiles(const Problem& P, const SkArgs& a, int tn) {
  long long t = 0;
  for (int s = 0; s < (P.epi == EPI_STORE ? a.nseg : 1); ++s) t += (a.seg[s].n + tn - 1) / tn;
  return t;
}

// Time models (microseconds) of the kernel families of an engine call of M rows split S
// ways, for the choice between them (it changes no bits):
//   tiled: t0 + 128-wide K stages x s[q - 1] for each round of q workgroups per CU (`cap` of
//          them are resident at once) + wmb per MB of weights + the split-K exchange, xs per
//          split and xmb per MB of partial tiles
//   rows:  t0 + 64-wide block pairs x (c0 + c1 x workgroups per CU) + the exchange
// Fitted to MI355X measurements of every tile and of the 16-row tiles at the calls' own splits
// (M = 17-4096 at 25 row counts, 41 shapes from 2048x64 to 12288x4096 and 3584x18944, one set
// and gate/up, weights rotated so that they stream from HBM), then moved where that let the
// choice agree with the measurements: over those 4626 calls the chosen kernel is 0.4 % behind
// the fastest.  (A fit over one workgroup count per shape, without the weights' term, chose
// 96x64 tiles for gemm_i8 4096x12288 at 96 rows: 36 us against 28 on 128x128.)
struct TileTime {
  double t0, s[3], xs, xmb, wmb;
  int cap;
};
struct RowsTime {
  double t0, c0, c1, xs, xw;
};
constexpr TileTime kTileTime[3][2][I8_TILES] = {
    // W8: 128x128, 64x64, 96x64, 128x64, 160x64; one weight set, then gate/up
    {{{5.27, {1, 0, 0}, 0.693, 0.477, 0.00798, 1},
      {4.03, {0.527, 0.755, 1.17}, 0.41, 0.355, 0.0985, 3},
      {6.21, {0.604, 0.965, 1.51}, 0.993, 0.32, 0.0599, 3},
      {5.27, {0.868, 1.34, 0}, 0.721, 0.351, 0.0278, 2},
      {5.32, {1.05, 1.69, 0}, 1.49, 0.272, 0.0402, 2}},
     {{8.42, {1.99, 0, 0}, 0.952, 0.407, 0.00836, 1},
      {9.78, {0.791, 1.2, 1.91}, 0.556, 0.281, 0.0284, 3},
      {8.62, {1.04, 1.72, 0}, 1.51, 0.362, 0.0899, 2}}},
    // W4
    {{{3.61, {1.27, 0, 0}, 0.539, 0.423, 0.05, 1},
      {4.38, {0.605, 0.992, 1.23}, 0.67, 0.24, 0.0716, 3},
      {4.77, {0.888, 1.18, 0}, 1.05, 0.384, 0.0926, 2},
      {5.14, {1.08, 1.5, 0}, 0.816, 0.305, 0.047, 2},
      {5.46, {1.39, 2.01, 0}, 1.49, 0.229, 0.00759, 2}},
     {{7.67, {2.53, 0, 0}, 0.833, 0.392, 0, 1},
      {6.41, {0.778, 1.53, 2.06}, 0.965, 0.277, 0.0689, 3},
      {7.89, {1.43, 1.94, 0}, 1.75, 0.352, 0.078, 2}}},
    // W4 with zeros
    {{{3.87, {1.57, 0, 0}, 0.614, 0.418, 0.0639, 1},
      {4.88, {0.694, 1.16, 1.45}, 0.617, 0.224, 0.0565, 3},
      {5.09, {1.12, 1.41, 0}, 0.991, 0.384, 0.0301, 2},
      {5.99, {1.3, 1.61, 0}, 0.68, 0.392, 0.0575, 2},
      {6.79, {1.72, 2.23, 0}, 1.47, 0.284, 0.0386, 2}},
     {{10.6, {2.98, 0, 0}, 1.17, 0.417, 0.00702, 1},
      {6.71, {1.05, 1.97, 0}, 1.02, 0.336, 0.0333, 2},
      {7.96, {1.93, 2.34, 0}, 1.75, 0.441, 0.0158, 2}}}};
constexpr RowsTime kRowsTime[3][2][2] = {  // [W8, W4, W4 with zeros][one set, gate/up][S = 1, S > 1]
    {{{4.3, 0.114, 0.376, 0, 0}, {9.68, 0.0748, 0.644, 0, 1.25}}, {{4.92, 0.601, 0.479, 0, 0}, {14.6, 0, 1.54, 0, 0.497}}},
    {{{5, 0.277, 0.184, 0, 0}, {8.86, 0.441, 0.282, 0.0523, 1.84}}, {{6.59, 0.455, 0.285, 0, 0}, {12, 0.454, 0.783, 0.143, 5.72}}},
    {{{6.07, 0.339, 0.186, 0, 0}, {8.87, 0.525, 0.328, 0.0555, 1.83}}, {{6.14, 0.574, 0.371, 0, 0}, {12.1, 0.689, 0.929, 0.134, 3.85}}}};

// index of a call's weight kind in the tables
int time_kind(const Problem& P) { return P.wk != WK_W4 ? 0 : P.hz ? 2 : 1; }

double tile_time(const Problem& P, const SkArgs& a, int tile, int M, int S) {
  const TileTime& m = kTileTime[time_kind(P)][P.nsets - 1][tile];
  int bm, bn;
  prefill_i8_geometry(tile, &bm, &bn);
  const long long wgs = (long long)((M + bm - 1) / bm) * col_tiles(P, a, bn) * S;
  const int nst = (P.K / 64 / S + 1) / 2;
  const long long full = wgs / (256LL * m.cap), rest = wgs - full * 256LL * m.cap;
  double st = (double)full * m.s[m.cap - 1];
  if (rest > 0) st += m.s[(rest + 255) / 256 - 1];
  const double weights = (double)P.K * P.ncols * P.nsets * (P.wk == WK_W4 ? 0.5e-6 : 1e-6);
  double t = m.t0 + st * nst + m.wmb * weights;
  if (S > 1) t += m.xs * S + m.xmb * 1e-6 * (double)wgs * bm * bn * 4 * P.nsets;
  return t;
}

double rows_time(const Problem& P, const SkArgs& a, int M, int S) {
  const RowsTime& m = kRowsTime[time_kind(P)][P.nsets - 1][S > 1];
  const double w = (double)((M + 15) / 16) * col_tiles(P, a, S > 1 ? 128 : 64) * S / 256.0;
  return m.t0 + (P.K / 64 / S / 2) * (m.c0 + m.c1 * std::max(1.0, w)) + m.xs * S + m.xw * w;
}

// Rows per launch that `cap` bytes of partial tiles and the arrival counters hold, in
// whole tiles of bm rows (every row with one split).
long long rows_that_fit(const Problem& P, const SkArgs& a, int M, int S, int bm, int bn, size_t cap) {
  if (S <= 1) return M;
  const long long nt = col_tiles(P, a, bn);
  const double row_bytes = (double)S * P.nsets * nt * bn * sizeof(float);
  const long long cap_rows = (long long)((double)cap / row_bytes) / bm * bm;
  const long long cnt_rows = (long long)(kCounterBytes / sizeof(unsigned)) / nt * bm;
  return std::min<long long>(M, std::min(cap_rows, cnt_rows));
}

// The tile the model prefers for M rows and S splits among those that cover the call and
// whose partials fit `cap` bytes, -1 if there is none; *t its time.
int best_tile(const Problem& P, const SkArgs& a, int M, int S, size_t cap, double* t, const char* force = nullptr) {
  SkArgs probe = a;
  probe.M = M;
  int best = -1;
  const int n = P.epi == EPI_STORE ? I8_TILES : I8_128x64;  // gate/up: the first three
  for (int k = 0; k < n; ++k) {
    int bm, bn;
    prefill_i8_geometry(k, &bm, &bn);
    if (!prefill_i8_ok(probe, P.wk, P.epi, k) || rows_that_fit(P, a, M, S, bm, bn, cap) < std::min(M, bm)) continue;
    const double tk = tile_time(P, a, k, M, S);
    const bool forced = force && *force && atoi(force) == k;
    if (best < 0 || tk < *t || forced) best = k, *t = tk;
    if (forced) break;
  }
  return best;
}

// Microseconds that split_estimate gives the engine's 512-row chunk with S K splits, on
// 128x128 tiles or on 16-row tiles, whichever is less.  These estimates define the K order
// (S, and so the bits, of every call of kRowsM rows or more): they stay as they are when the
// kernels and the time models below change.
double split_estimate(const Problem& P, const SkArgs& a, int S) {
  const bool w4 = P.wk == WK_W4;
  const double elems = (double)P.K * P.ncols * P.nsets / 1e6;
  const double rows = 5.0 + (w4 ? 0.17 : 0.125) * ((kRefChunkM + 15) / 16) * elems + (S > 1 ? 1.45 * S : 0.0);
  SkArgs probe = a;
  probe.M = kRefChunkM;
  if (!prefill_i8_ok(probe, P.wk, P.epi, I8_128x128)) return rows;
  const long long wgs = (long long)((kRefChunkM + 127) / 128) * col_tiles(P, a, 128) * S;
  const double occ = (double)std::min<long long>(wgs, 256);
  const double stage = (w4 ? 1.8 + 1.6e-3 * occ : 1.05 + 2.5e-3 * occ) * P.nsets;
  double t = 7.0 + (double)((wgs + 255) / 256) * ((P.K / 64 / S + 1) / 2) * stage;
  if (S > 1) t += 1.45 * S + 12e-3 * wgs + 0.1e-6 * (double)wgs * P.nsets * 128 * 128 * sizeof(float);
  return std::min(t, rows);
}

// Split count of the K order: the S (1, 2, 4 or 8, dividing K into ranges of at least two
// 64-wide blocks) with the least estimate.  S picked for 128 rows as well as 512, by the tiles'
// own models, gained at some row counts and lost at others (gemm_i8 12288x4096 at 512 rows
// 69 -> 81 us, at 2048 243 -> 298; W8 gate/up 4096x12288 at 9 rows 37 -> 61).
// QLIN_ENGINE_SPLITS overrides it (tuning; it changes the K order).
int engine_splits(const Problem& P, const SkArgs& a) {
  const int nb = P.K / 64;
  const char* es = getenv("QLIN_ENGINE_SPLITS");
  if (es && *es) return atoi(es);
  double best = 0.0;
  int S = 1;
  SkArgs b = a;
  b.x = nullptr;  // the choice must not depend on where the activations sit
  for (int s = 1; s <= 8; s *= 2) {
    if (nb % s != 0 || (s > 1 && nb / s < 2)) break;
    const double t = split_estimate(P, b, s);
    if (s == 1 || t < best) best = t, S = s;
  }
  return S;
}

// The rows [m0, m0 + rows) of a call as a call of its own (rows are independent).
SkArgs row_block(const SkArgs& a, int m0, int rows) {
  SkArgs b = a;
  b.M = rows;
  b.x = (const int8_t*)a.x + (long long)m0 * a.K;
  b.xs = a.xs + (long long)m0 * (a.K / 64);
  if (a.out) b.out = (uint16_t*)a.out + (long long)m0 * a.ldo;
  if (a.res) b.res = (const uint16_t*)a.res + (long long)m0 * a.ldr;
  if (a.oq) b.oq = a.oq + (long long)m0 * a.ncols;
  if (a.os) b.os = a.os + (long long)m0 * (a.ncols / 64);
  if (a.pro.kind != PRO_NONE) {
    ProArgs& p = b.pro;
    p.x = (const uint16_t*)a.pro.x + (long long)m0 * a.pro.ldx;
    if (a.pro.g) p.g = (const uint16_t*)a.pro.g + (long long)m0 * a.pro.ldg;
    if (a.pro.q) p.q = a.pro.q + (long long)m0 * a.K, p.s = a.pro.s + (long long)m0 * (a.K / 64);
    p.tq = a.pro.tq + (long long)m0 * a.K;
    p.ts = a.pro.ts + (long long)m0 * (a.K / 64);
  }
  return b;
}

// Activation producer of a call (a.pro): run it as a launch of its own, writing the
// codes and scales to a.pro.tq / a.pro.ts, which the call then reads as its
// activations.
int pro_materialize(const char* fn, SkArgs& a, hipStream_t stream) {
  ProArgs p = a.pro;
  p.q = p.tq;
  p.s = p.ts;
  QL_TRY(hip_status(fn, launch_producer(p, a.M, a.K, stream)));
  a.x = p.tq;
  a.xs = p.ts;
  a.pro.kind = PRO_NONE;
  return QLIN_OK;
}

// Fused prologue for a skinny launch plan: places the code block of the workgroup's
// rows and K range after the finish layout in dynamic LDS.  False when the plan has
// no fused instantiation, the block does not fit, or the prologue would hold each
// thread for more than kProItems values (every column tile of a row tile makes the
// same codes: cheap for decode's short K ranges, slower than one producer launch for
// 16-row tiles over long ones); the caller then makes the codes with their own launch.
constexpr long long kProItems = 32;
bool pro_plan(SkLaunch& L, SkArgs& a, int K, int rows) {
  L.pro = 1;
  if (!skinny_pro_ok(L, a.group)) {
    L.pro = 0;
    return false;
  }
  const int kr = (a.lanes == 2) ? a.kchunk : std::min(K, L.waves * a.kchunk);
  const int mt = std::min(16, rows);
  const long long work = (long long)mt * kr + (a.pro.kind == PRO_RMSNORM ? (long long)mt * K : 0);
  if (work > kProItems * 64 * L.waves) {
    L.pro = 0;
    return false;
  }
  const size_t off = (L.lds + 15) & ~(size_t)15;
  const int ldq = kr + 16;  // 16 bytes of padding staggers the rows over the LDS banks
  const size_t bytes = (size_t)mt * ldq + (size_t)mt * (kr / 64) * sizeof(float) + (size_t)mt * sizeof(float);
  if (bytes > kProLdsBytes) {
    L.pro = 0;
    return false;
  }
  a.pro.lds_off = (int)off;
  a.pro.ldq = ldq;
  L.lds = off + bytes;
  return true;
}

int engine_rows(const char* fn, const Problem& P, SkArgs& a, void* workspace, size_t ws_bytes,
                hipStream_t stream, bool clear) {
  const int S = engine_splits(P, a);
  const int nb = P.K / 64;
  if (S < 1 || S > 64 || nb % S != 0 || (S > 1 && nb / S < 2))
    return fail(QLIN_ERR_UNSUPPORTED, "%s: %d K splits do not divide K=%d into ranges of at least 128", fn, S, P.K);
  // family: the tiled int8 kernel where it applies and a time model prefers it to the
  // 16-row tiles; both give the same bits.  QLIN_ENGINE_PREFILL=tiled|skinny forces one.
  const char* e = getenv("QLIN_ENGINE_PREFILL");
  const bool force_rows = e && strcmp(e, "skinny") == 0;
  const bool force_tiled = e && strcmp(e, "tiled") == 0;
  const size_t part_cap = (workspace && ws_bytes > kPartBase) ? ws_bytes - kPartBase : 0;
  int tile = -1;
  if (!force_rows) {
    double t_tile = 0.0;
    // (QLIN_I8_TILE forces one tile where it covers the call: the same bits)
    tile = best_tile(P, a, P.M, S, part_cap, &t_tile, getenv("QLIN_I8_TILE"));
    if (!force_tiled && tile >= 0 && t_tile >= rows_time(P, a, P.M, S)) tile = -1;
  }
  const bool tiled = tile >= 0;
  // the tiled kernel has no producer prologue: make the activations first
  if (tiled && a.pro.kind != PRO_NONE) QL_TRY(pro_materialize(fn, a, stream));
  int rstep = 16, TN = S == 1 ? 64 : 128;
  if (tiled) prefill_i8_geometry(tile, &rstep, &TN);
  const long long ntiles = col_tiles(P, a, TN);
  // rows per launch: the split-K partials and arrival counters of a launch must fit
  // the workspace (rows are independent, so blocks of rows give the same bits)
  const long long mb_rows = rows_that_fit(P, a, P.M, S, rstep, TN, part_cap);
  if (mb_rows < std::min(P.M, rstep))
    return fail(QLIN_ERR_WORKSPACE, "%s: the workspace (%zu bytes) cannot hold %d K splits of %lld columns", fn,
                ws_bytes, S, (long long)ntiles * TN);
  if (clear && S > 1) {
    // one counter per (16-row tile, column tile) at most, for the rows of one launch
    const long long n = ((mb_rows + 15) / 16) * ntiles;
    QL_TRY(hip_status(fn, clear_counters(workspace, std::min<long long>(n, kCounterBytes / sizeof(unsigned)), stream)));
  }
  for (long long m0 = 0; m0 < P.M; m0 += mb_rows) {
    const int rows = (int)std::min<long long>(mb_rows, P.M - m0);
    SkArgs b = row_block(a, (int)m0, rows);
    b.splits = S;
    b.cnt = S > 1 ? (unsigned*)workspace : nullptr;
    b.part = S > 1 ? (float*)((char*)workspace + kPartBase) : nullptr;
    hipError_t err;
    if (tiled) {
      if (!b.x || !b.xs) return fail(QLIN_ERR_INVALID, "%s: internal error: no activations for the tiled kernel", fn);
      err = launch_prefill_i8(b, P.wk, P.hz, P.epi, tile, stream);
    } else {
      SkLaunch L;
      L.act = P.act;
      L.wk = P.wk;
      L.hz = P.hz ? 1 : 0;
      L.epi = P.epi;
      L.cols = TN / 16;
      L.waves = 2;
      L.pro = 0;
      int acc = 0;
      for (int s = 0; s < b.nseg; ++s) {
        b.seg[s].tile0 = (P.epi == EPI_STORE) ? acc : 0;
        if (P.epi == EPI_STORE) acc += (b.seg[s].n + TN - 1) / TN;
      }
      b.ntiles = (int)ntiles;
      b.kchunk = P.K / S;
      b.lanes = 2;
      const int rtiles = (rows + 15) / 16;
      if (ntiles * S > 0x7FFFFFFFLL || rtiles > 65535)
        return fail(QLIN_ERR_UNSUPPORTED, "%s: grid too large (M=%d, N=%d)", fn, P.M, P.ncols);
      L.grid = dim3((unsigned)(ntiles * S), (unsigned)rtiles, 1);
      const int rg0 = ((rows < 16 ? rows : 16) + 3) / 4;
      L.lds = ((size_t)L.waves * P.nsets * rg0 * 4 * (TN + 4) + (size_t)P.nsets * TN) * sizeof(float);
      if (b.pro.kind != PRO_NONE && !pro_plan(L, b, P.K, rows)) QL_TRY(pro_materialize(fn, b, stream));
      if (!L.pro && (!b.x || !b.xs)) return fail(QLIN_ERR_INVALID, "%s: internal error: no activations", fn);
      err = launch_skinny(L, b, stream);
    }
    if (err != hipSuccess) return hip_status(fn, err);
  }
  return QLIN_OK;
}

// Chooses the kernel variant, column tile, waves per workgroup and split-K, then launches.
// Every choice depends on K, N (and whether M > 16), never on M itself, so an output row
// is computed the same way for every M <= 16.  Engine-signature calls with kRowsM rows
// or more take engine_rows (one K order for every M).
// clear: zero the arrival counters the launch can use first (a scratch whose counters
// are not known to be zero).
int plan_and_launch(const char* fn, const Problem& P, SkArgs& a, void* workspace, size_t ws_bytes,
                    hipStream_t stream, bool clear = false) {
  // decode rows (one sequence or up to eight best-of rows) run on the engine decode
  // work units, the units an engine chain runs: a call equals its chain job bit for bit
  // (QLIN_ENGINE_DECODE=skinny keeps such calls on the skinny decode plans below, for
  // comparisons; it changes the K order)
  if (P.act == ACT_I8 && P.M <= kDecodeRowsMax && echain_covers(a, P.wk, P.M)) {
    const char* ed = getenv("QLIN_ENGINE_DECODE");
    if (!(ed && strcmp(ed, "skinny") == 0))
      return echain_engine_call(fn, a, P.wk, P.epi, P.M, workspace, ws_bytes, kCounterBytes, kPollBytes, stream,
                                clear);
  }
  if (P.act == ACT_I8 && P.M >= kRowsM) return engine_rows(fn, P, a, workspace, ws_bytes, stream, clear);
  SkLaunch L;
  L.act = P.act;
  L.wk = P.wk;
  L.hz = P.hz ? 1 : 0;
  L.epi = P.epi;
  L.pro = 0;

  auto count_tiles = [&](int tn) {
    int nt = 0;
    if (P.epi == EPI_STORE) {
      for (int s = 0; s < a.nseg; ++s) nt += (a.seg[s].n + tn - 1) / tn;
    } else {
      nt = (a.seg[0].n + tn - 1) / tn;
    }
    return nt;
  };
  // K granule of one wave's range: the MFMA step, the activation group (int8) and
  // whole W4 weight groups
  int kalign = (P.act == ACT_I8) ? 64 : 32;
  if (P.wk == WK_W4 && P.group > kalign) kalign = P.group;
  const int nunits = P.K / kalign;
  const int rtiles = (P.M + 15) / 16;
  const bool wide = P.M > 16 || count_tiles(256) >= kWideTiles;

  // Measured on MI355X: wide W8 launches stream best as single-wave workgroups over
  // 128-column tiles, wide W4 over 256-column tiles; narrow launches over 128-column
  // tiles with K spread first over the waves of one workgroup (up to 8, reduced in
  // LDS) and only then over workgroups.
  int cols = (wide && P.wk == WK_W4 && P.epi == EPI_STORE && P.M <= 16) ? 16 : 8;
  int waves = (wide && P.M <= 16) ? 1 : (wide ? 4 : (skinny_big(P.act, P.wk, P.epi, cols) ? 8 : 4)), upw = 0;
  // Narrow launches whose whole-K 64-column tile of one weight set is small read it in
  // one pass: 4-column lanes, K over the 8 waves of one workgroup, no split-K exchange
  // (partial store, arrival counter and final read are three memory round trips).
  // Larger tiles keep split-K: a CU moves only 16 bytes per cycle with 4-byte lanes.
  const long long tile_bytes = (long long)P.K * 64 / (P.wk == WK_W4 ? 2 : 1);
  if (!wide && tile_bytes <= kOnePassTileBytes) cols = 4, waves = 8;
  plan_override(P, cols, waves, upw);
  const bool one_pass = cols == 4;
  const int maxw = one_pass ? 8 : (skinny_big(P.act, P.wk, P.epi, cols) ? 8 : 4);
  if (waves > maxw) waves = maxw;
  const int TN = 16 * cols;
  const int ntiles = count_tiles(TN);
  int ntile_acc = 0;
  for (int s = 0; s < a.nseg; ++s) {
    a.seg[s].tile0 = (P.epi == EPI_STORE) ? ntile_acc : 0;
    if (P.epi == EPI_STORE) ntile_acc += (a.seg[s].n + TN - 1) / TN;
  }
  a.ntiles = ntiles;

  int splits;
  if (one_pass) {
    if (waves > nunits) waves = nunits;
    upw = (nunits + waves - 1) / waves;
    splits = 1;
  } else if (wide) {
    if (waves > nunits) waves = nunits;
    if (upw == 0) upw = (nunits + waves - 1) / waves;
    splits = (nunits + upw * waves - 1) / (upw * waves);
    if (P.M > 16) splits = 1, upw = (nunits + waves - 1) / waves;
  } else {
    // narrow N: spread K over up to kTargetWaves waves, each at least kMinWaveK deep
    const long long target = (P.wk == WK_W4) ? kTargetWavesW4 : kTargetWavesW8;
    int min_k = (P.wk == WK_W4) ? kMinWaveKW4 : kMinWaveKW8;
    if (P.act == ACT_F16 && P.wk == WK_W8 && (long long)ntiles * nunits <= kOneStepUnits) min_k = 32;
    const int min_upw = (min_k + kalign - 1) / kalign;
    if (upw == 0) {
      upw = (int)(((long long)ntiles * nunits + target - 1) / target);
      if (upw < min_upw) upw = min_upw;
    }
    if (upw > nunits) upw = nunits;
    const int chunks = (nunits + upw - 1) / upw;  // waves per tile
    if (waves > chunks) waves = chunks;
    splits = (chunks + waves - 1) / waves;
  }
  // partial sums must fit the workspace; without a workspace there is no cross-workgroup split
  const size_t part_cap = (workspace && ws_bytes > kPartBase) ? ws_bytes - kPartBase : 0;
  auto fits = [&](int s) {
    const size_t need = (size_t)s * P.nsets * (size_t)P.M * (size_t)P.ncols * sizeof(float);
    const size_t cnt_need = (size_t)rtiles * ntiles * sizeof(unsigned);
    return need <= part_cap && cnt_need <= kCounterBytes;
  };
  while (splits > 1 && !fits(splits)) {
    upw *= 2;
    splits = (nunits + upw * waves - 1) / (upw * waves);
  }
  if (splits <= 1) {
    splits = 1;
    upw = (nunits + waves - 1) / waves;
  }
  a.kchunk = upw * kalign;
  a.splits = splits;
  if (splits > 1) {
    a.cnt = (unsigned*)workspace;
    a.part = (float*)((char*)workspace + kPartBase);
  } else {
    a.cnt = nullptr;
    a.part = nullptr;
  }
  L.cols = cols;
  L.waves = waves;
  L.grid = dim3((unsigned)(ntiles * splits), (unsigned)rtiles, 1);
  // LDS: one finish-layout slot per wave ([set][row][column], rows of the first row
  // tile rounded up to 4, row stride TN + 4 floats), then the tile's column scales
  const int rg0 = (((P.M < 16) ? P.M : 16) + 3) / 4;
  L.lds = ((size_t)waves * P.nsets * rg0 * 4 * (TN + 4) + (size_t)P.nsets * TN) * sizeof(float);
  if ((long long)ntiles * splits > 0x7FFFFFFFLL || rtiles > 65535)
    return fail(QLIN_ERR_UNSUPPORTED, "%s: grid too large (M=%d, N=%d)", fn, P.M, P.ncols);
  // activation producer: fused into the prologue of narrow plans; wide plans (every
  // workgroup would redo the whole row) make the activations with a launch of their own
  if (a.pro.kind != PRO_NONE && (wide || !pro_plan(L, a, P.K, P.M))) QL_TRY(pro_materialize(fn, a, stream));
  // every launch reads its activations from memory unless its prologue makes them
  if (!L.pro && (!a.x || (P.act == ACT_I8 && !a.xs)))
    return fail(QLIN_ERR_INVALID, "%s: internal error: no activations", fn);
  if (clear && splits > 1) QL_TRY(hip_status(fn, clear_counters(workspace, (long long)rtiles * ntiles, stream)));
  return hip_status(fn, launch_skinny(L, a, stream));
}

int check_common(const char* fn, int M, int K, int N) {
  if (M < 0 || K <= 0 || N < 0) return fail(QLIN_ERR_INVALID, "%s: bad sizes M=%d K=%d N=%d", fn, M, K, N);
  return QLIN_OK;
}

int check_weight(const char* fn, const void* w, const void* s, const uint8_t* z, int n, int wk) {
  if (n == 0) return QLIN_OK;
  if (!w || !s) return fail(QLIN_ERR_INVALID, "%s: null weight or scale", fn);
  if (n % 16 != 0) return fail(QLIN_ERR_UNSUPPORTED, "%s: N=%d is not a multiple of 16", fn, n);
  if (!aligned(w, 16) || !aligned(s, 16) || (z && !aligned(z, 16)))
    return fail(QLIN_ERR_UNSUPPORTED, "%s: weight/scale/zero pointers must be 16-byte aligned", fn);
  (void)wk;
  return QLIN_OK;
}

int check_engine_act(const char* fn, const int8_t* a_q, const float* a_s, int M, int K) {
  if (M > 0 && (!a_q || !a_s)) return fail(QLIN_ERR_INVALID, "%s: null activations", fn);
  if (K % 64 != 0) return fail(QLIN_ERR_UNSUPPORTED, "%s: K=%d is not a multiple of 64", fn, K);
  if (!aligned(a_s, 4)) return fail(QLIN_ERR_UNSUPPORTED, "%s: a_s must be 4-byte aligned", fn);
  return QLIN_OK;
}

// Engine-signature calls take any N and pointers aligned to their element size only
// (the reference's kernels mask every edge, kernels/gemm.py:50-57).  The fast kernels
// need N % 16 == 0, 16-byte aligned weights, scales, zeros and 16-bit rows (row
// strides multiples of 8) and 8-byte aligned codes; a valid call outside those rules
// runs on the edge kernel (edge.hip).
int check_engine_weight(const char* fn, const void* w, const void* s, int n, int sdt) {
  if (n == 0) return QLIN_OK;
  if (!w || !s) return fail(QLIN_ERR_INVALID, "%s: null weight or scale", fn);
  if (!aligned(s, sdt == QLIN_F32 ? 4 : 2))
    return fail(QLIN_ERR_UNSUPPORTED, "%s: scales must be aligned to their element size", fn);
  return QLIN_OK;
}

bool engine_weight_fast(const void* w, const void* s, const uint8_t* z, int n) {
  return n == 0 || (n % 16 == 0 && aligned(w, 16) && aligned(s, 16) && (!z || aligned(z, 16)));
}

int check_engine_out(const char* fn, const void* p, int64_t ld, int N, const char* what) {
  if (!p) return fail(QLIN_ERR_INVALID, "%s: null %s", fn, what);
  if (ld < N) return fail(QLIN_ERR_INVALID, "%s: %s row stride %lld < N=%d", fn, what, (long long)ld, N);
  if (!aligned(p, 2)) return fail(QLIN_ERR_UNSUPPORTED, "%s: %s must be 2-byte aligned", fn, what);
  return QLIN_OK;
}

bool engine_out_fast(const void* p, int64_t ld) { return aligned(p, 16) && ld % 8 == 0; }

// A call on the edge kernel; a producer first runs as a launch of its own into the
// codes setup_pro chose.
int engine_edge(const char* fn, int wk, int epi, const int8_t* a_q, const float* a_s, int M, int K, const Seg* segs,
                int nseg, int ncols, int group, int sdt, void* out, int64_t ldo, const void* res, int64_t ldr,
                int8_t* oq, float* os, const ProArgs* pa, hipStream_t st) {
  if (pa && pa->kind != PRO_NONE) {
    ProArgs p = *pa;
    p.q = p.tq;
    p.s = p.ts;
    QL_TRY(hip_status(fn, launch_producer(p, M, K, st)));
    a_q = p.tq;
    a_s = p.ts;
  }
  EdgeArgs e;
  memset(&e, 0, sizeof(e));
  e.x = a_q;
  e.xs = a_s;
  e.M = M;
  e.K = K;
  for (int i = 0; i < nseg; ++i) e.seg[i] = segs[i];
  e.nseg = nseg;
  e.ncols = ncols;
  e.group = (wk == WK_W4) ? group : 64;
  e.sdt = sdt;
  e.epi = epi;
  e.odt = QLIN_BF16;
  e.out = out;
  e.ldo = ldo;
  e.res = res;
  e.ldr = ldr;
  e.oq = oq;
  e.os = os;
  return hip_status(fn, launch_edge(e, wk, st));
}

// Validates an activation producer (kernels/norm.py:28-57, 95-137, 168-188) for M rows
// of K columns and completes it: norm_gated reads v contiguous (row stride K), and the
// codes go to q / s or, without them, to the end of the workspace, which is taken off
// *wsb so no split-K partial reaches it.
int setup_pro(const char* fn, ProArgs& p, int M, int K, void* ws, size_t* wsb) {
  QL_TRY(check_producer(fn, p, M, K));
  if (p.q) {
    p.tq = p.q;
    p.ts = p.s;
  } else {
    const size_t qb = ((size_t)M * K + 255) & ~(size_t)255;
    const size_t sb = ((size_t)M * (K / 64) * sizeof(float) + 255) & ~(size_t)255;
    if (!ws || *wsb < kPartBase + qb + sb)
      return fail(QLIN_ERR_WORKSPACE, "%s: no room in the workspace for the activation codes", fn);
    *wsb -= qb + sb;
    p.tq = (int8_t*)ws + *wsb;
    p.ts = (float*)((char*)ws + *wsb + qb);
  }
  p.lds_off = 0;
  p.ldq = 0;
  return QLIN_OK;
}

}  // namespace

int qlin::check_producer(const char* fn, ProArgs& p, int M, int K) {
  (void)M;
  if (p.kind != PRO_RMSNORM && p.kind != PRO_GATE_MUL && p.kind != PRO_NORM_GATED)
    return fail(QLIN_ERR_INVALID, "%s: unknown producer kind %d", fn, p.kind);
  if (K % 64 != 0) return fail(QLIN_ERR_UNSUPPORTED, "%s: K=%d is not a multiple of 64", fn, K);
  if (p.xdt != QLIN_BF16 && p.xdt != QLIN_F16)
    return fail(QLIN_ERR_UNSUPPORTED, "%s: activation dtype %d (need bf16 or fp16)", fn, p.xdt);
  if (!p.x) return fail(QLIN_ERR_INVALID, "%s: null producer input", fn);
  if (p.kind == PRO_NORM_GATED) p.ldx = K;
  if (p.ldx < K || p.ldx % 8 != 0 || !aligned(p.x, 16))
    return fail(QLIN_ERR_UNSUPPORTED, "%s: producer input must be 16-byte aligned with a row stride >= K and a "
                "multiple of 8", fn);
  if (p.kind != PRO_GATE_MUL) {
    if (!p.w) return fail(QLIN_ERR_INVALID, "%s: null norm weight", fn);
    if (!dtype_scale_ok(p.wdt)) return fail(QLIN_ERR_UNSUPPORTED, "%s: norm weight dtype %d", fn, p.wdt);
    if (!aligned(p.w, 16)) return fail(QLIN_ERR_UNSUPPORTED, "%s: norm weight must be 16-byte aligned", fn);
  }
  if (p.kind != PRO_RMSNORM) {
    if (!p.g) return fail(QLIN_ERR_INVALID, "%s: null gate input", fn);
    if (p.ldg % 8 != 0 || !aligned(p.g, 16))
      return fail(QLIN_ERR_UNSUPPORTED, "%s: gate input must be 16-byte aligned with a row stride multiple of 8", fn);
  }
  if (p.kind == PRO_GATE_MUL) {
    if (p.hd <= 0 || p.hd % 8 != 0 || K % p.hd != 0)
      return fail(QLIN_ERR_UNSUPPORTED, "%s: head size %d must be a multiple of 8 dividing K=%d", fn, p.hd, K);
    if (p.ldg < 2LL * K) return fail(QLIN_ERR_INVALID, "%s: gate row stride %lld < 2 K", fn, (long long)p.ldg);
  }
  if (p.kind == PRO_NORM_GATED) {
    if ((p.hd != 128 && p.hd != 256 && p.hd != 512) || K % p.hd != 0)
      return fail(QLIN_ERR_UNSUPPORTED, "%s: head size %d (need 128, 256 or 512, dividing K=%d)", fn, p.hd, K);
    if (p.ldg < K) return fail(QLIN_ERR_INVALID, "%s: z row stride %lld < K", fn, (long long)p.ldg);
  }
  if ((p.q == nullptr) != (p.s == nullptr)) return fail(QLIN_ERR_INVALID, "%s: give both q and s, or neither", fn);
  if (p.q && (!aligned(p.q, 8) || !aligned(p.s, 4)))
    return fail(QLIN_ERR_UNSUPPORTED, "%s: q must be 8-byte aligned", fn);
  return QLIN_OK;
}

hipError_t qlin::clear_counters(void* ws, long long n, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(zero_u32, dim3((unsigned)std::min<long long>(256, (n + 255) / 256)), dim3(256), 0, stream,
                     (unsigned*)ws, (int)n);
  return hipGetLastError();
}

namespace {

int check_out16(const char* fn, const void* p, int64_t ld, int N, const char* what) {
  if (!p) return fail(QLIN_ERR_INVALID, "%s: null %s", fn, what);
  if (ld < N) return fail(QLIN_ERR_INVALID, "%s: %s row stride %lld < N=%d", fn, what, (long long)ld, N);
  if (!aligned(p, 16) || ld % 8 != 0)
    return fail(QLIN_ERR_UNSUPPORTED, "%s: %s must be 16-byte aligned with a row stride multiple of 8", fn,
                what);
  return QLIN_OK;
}

int check_group(const char* fn, int group, int K) {
  if (!group_ok(group)) return fail(QLIN_ERR_UNSUPPORTED, "%s: weight group %d (need 32 or a multiple of 64)", fn, group);
  if (K % group != 0) return fail(QLIN_ERR_INVALID, "%s: K=%d not a multiple of the group %d", fn, K, group);
  return QLIN_OK;
}


Seg make_seg(const void* w, const void* s, const uint8_t* z, int n, int col0) {
  Seg g;
  g.w = (const uint8_t*)w;
  g.s = s;
  g.z = z;
  g.n = n;
  g.col0 = col0;
  g.tile0 = 0;
  return g;
}

SkArgs base_args() {
  SkArgs a;
  memset(&a, 0, sizeof(a));
  return a;
}

// Common body of gemm_i8 / gemm_w4.
int engine_gemm(const char* fn, int wk, const int8_t* a_q, const float* a_s, int M, int K, const void* b,
                const void* b_s, int bs_dtype, const uint8_t* b_z, int group, int N, void* out, int64_t ldo,
                const void* residual, int64_t ldr, void* ws, size_t wsb, void* stream, bool clear = false,
                const ProArgs* pro = nullptr) {
  QL_TRY(check_common(fn, M, K, N));
  if (M == 0 || N == 0) return QLIN_OK;
  ProArgs pa{};
  if (pro) {
    pa = *pro;
    QL_TRY(setup_pro(fn, pa, M, K, ws, &wsb));
  } else {
    QL_TRY(check_engine_act(fn, a_q, a_s, M, K));
  }
  if (!dtype_scale_ok(bs_dtype)) return fail(QLIN_ERR_UNSUPPORTED, "%s: scale dtype %d", fn, bs_dtype);
  if (wk == WK_W4) QL_TRY(check_group(fn, group, K));
  QL_TRY(check_engine_weight(fn, b, b_s, N, bs_dtype));
  QL_TRY(check_engine_out(fn, out, ldo, N, "out"));
  if (residual) QL_TRY(check_engine_out(fn, residual, ldr, N, "residual"));
  if (!engine_weight_fast(b, b_s, b_z, N) || !engine_out_fast(out, ldo) ||
      (residual && !engine_out_fast(residual, ldr)) || (!pro && !aligned(a_q, 8))) {
    const Seg s0 = make_seg(b, b_s, b_z, N, 0);
    return engine_edge(fn, wk, EPI_STORE, a_q, a_s, M, K, &s0, 1, N, group, bs_dtype, out, ldo, residual, ldr,
                       nullptr, nullptr, pro ? &pa : nullptr, (hipStream_t)stream);
  }
  SkArgs a = base_args();
  a.x = a_q;
  a.xs = a_s;
  a.M = M;
  a.K = K;
  a.seg[0] = make_seg(b, b_s, b_z, N, 0);
  a.nseg = 1;
  a.ncols = N;
  a.group = (wk == WK_W4) ? group : 64;
  a.sdt = bs_dtype;
  a.out = out;
  a.ldo = ldo;
  a.odt = QLIN_BF16;
  a.res = residual;
  a.ldr = ldr;
  a.pro = pa;
  Problem P{ACT_I8, wk, EPI_STORE, b_z != nullptr, M, K, a.group, 1, N};
  if (clear && (!ws || wsb <= kPartBase)) return fail(QLIN_ERR_WORKSPACE, "%s: no scratch", fn);
  return plan_and_launch(fn, P, a, ws, wsb, (hipStream_t)stream, clear);
}

int engine_proj3(const char* fn, int wk, const int8_t* a_q, const float* a_s, int M, int K, const void* w1,
                 const void* s1, const uint8_t* z1, int n1, const void* w2, const void* s2, const uint8_t* z2,
                 int n2, const void* w3, const void* s3, const uint8_t* z3, int n3, int bs_dtype, int group,
                 void* out, int64_t ldo, void* ws, size_t wsb, void* stream, const ProArgs* pro = nullptr) {
  const int NT = n1 + n2 + n3;
  QL_TRY(check_common(fn, M, K, NT));
  if (n1 < 0 || n2 < 0 || n3 < 0) return fail(QLIN_ERR_INVALID, "%s: negative N", fn);
  if (M == 0 || NT == 0) return QLIN_OK;
  ProArgs pa{};
  if (pro) {
    pa = *pro;
    QL_TRY(setup_pro(fn, pa, M, K, ws, &wsb));
  } else {
    QL_TRY(check_engine_act(fn, a_q, a_s, M, K));
  }
  if (!dtype_scale_ok(bs_dtype)) return fail(QLIN_ERR_UNSUPPORTED, "%s: scale dtype %d", fn, bs_dtype);
  if (wk == WK_W4) QL_TRY(check_group(fn, group, K));
  QL_TRY(check_engine_weight(fn, w1, s1, n1, bs_dtype));
  QL_TRY(check_engine_weight(fn, w2, s2, n2, bs_dtype));
  QL_TRY(check_engine_weight(fn, w3, s3, n3, bs_dtype));
  QL_TRY(check_engine_out(fn, out, ldo, NT, "out"));
  const bool hz = (z1 || z2 || z3);
  if (hz && ((n1 && !z1) || (n2 && !z2) || (n3 && !z3)))
    return fail(QLIN_ERR_INVALID, "%s: zeros must be given for every projection or for none", fn);
  if (!engine_weight_fast(w1, s1, z1, n1) || !engine_weight_fast(w2, s2, z2, n2) ||
      !engine_weight_fast(w3, s3, z3, n3) || !engine_out_fast(out, ldo) || (!pro && !aligned(a_q, 8))) {
    Seg sg[3];
    int ns = 0, col = 0;
    const void* wv[3] = {w1, w2, w3};
    const void* sv[3] = {s1, s2, s3};
    const uint8_t* zv[3] = {z1, z2, z3};
    const int nv[3] = {n1, n2, n3};
    for (int i = 0; i < 3; ++i) {
      if (nv[i] == 0) continue;
      sg[ns++] = make_seg(wv[i], sv[i], zv[i], nv[i], col);
      col += nv[i];
    }
    return engine_edge(fn, wk, EPI_STORE, a_q, a_s, M, K, sg, ns, NT, group, bs_dtype, out, ldo, nullptr, 0,
                       nullptr, nullptr, pro ? &pa : nullptr, (hipStream_t)stream);
  }
  SkArgs a = base_args();
  a.x = a_q;
  a.xs = a_s;
  a.M = M;
  a.K = K;
  int ns = 0, col = 0;
  const void* ws_[3] = {w1, w2, w3};
  const void* ss_[3] = {s1, s2, s3};
  const uint8_t* zs_[3] = {z1, z2, z3};
  const int ns_[3] = {n1, n2, n3};
  for (int i = 0; i < 3; ++i) {
    if (ns_[i] == 0) continue;
    a.seg[ns++] = make_seg(ws_[i], ss_[i], zs_[i], ns_[i], col);
    col += ns_[i];
  }
  a.nseg = ns;
  a.ncols = NT;
  a.group = (wk == WK_W4) ? group : 64;
  a.sdt = bs_dtype;
  a.out = out;
  a.ldo = ldo;
  a.odt = QLIN_BF16;
  a.pro = pa;
  Problem P{ACT_I8, wk, EPI_STORE, hz, M, K, a.group, 1, NT};
  return plan_and_launch(fn, P, a, ws, wsb, (hipStream_t)stream);
}

int engine_gate_up(const char* fn, int wk, int epi, const int8_t* a_q, const float* a_s, int M, int K,
                   const void* wg, const void* sg, const uint8_t* zg, const void* wu, const void* su,
                   const uint8_t* zu, int bs_dtype, int group, int N, void* out, int8_t* out_q, float* out_s,
                   void* ws, size_t wsb, void* stream, const ProArgs* pro = nullptr) {
  QL_TRY(check_common(fn, M, K, N));
  if (M == 0 || N == 0) return QLIN_OK;
  ProArgs pa{};
  if (pro) {
    pa = *pro;
    QL_TRY(setup_pro(fn, pa, M, K, ws, &wsb));
  } else {
    QL_TRY(check_engine_act(fn, a_q, a_s, M, K));
  }
  if (!dtype_scale_ok(bs_dtype)) return fail(QLIN_ERR_UNSUPPORTED, "%s: scale dtype %d", fn, bs_dtype);
  if (wk == WK_W4) QL_TRY(check_group(fn, group, K));
  QL_TRY(check_engine_weight(fn, wg, sg, N, bs_dtype));
  QL_TRY(check_engine_weight(fn, wu, su, N, bs_dtype));
  if ((zg == nullptr) != (zu == nullptr))
    return fail(QLIN_ERR_INVALID, "%s: zeros must be given for both gate and up or for neither", fn);
  bool fast = engine_weight_fast(wg, sg, zg, N) && engine_weight_fast(wu, su, zu, N) && (pro || aligned(a_q, 8));
  if (epi == EPI_GATEUP) {
    QL_TRY(check_engine_out(fn, out, N, N, "out"));
    fast = fast && engine_out_fast(out, N);
  } else {
    if (N % 64 != 0) return fail(QLIN_ERR_UNSUPPORTED, "%s: N=%d is not a multiple of 64", fn, N);
    if (!out_q || !out_s) return fail(QLIN_ERR_INVALID, "%s: null out_q/out_s", fn);
    if (!aligned(out_s, 4)) return fail(QLIN_ERR_UNSUPPORTED, "%s: out_s must be 4-byte aligned", fn);
    fast = fast && aligned(out_q, 16);
  }
  if (!fast) {
    const Seg sgs[2] = {make_seg(wg, sg, zg, N, 0), make_seg(wu, su, zu, N, 0)};
    return engine_edge(fn, wk, epi, a_q, a_s, M, K, sgs, 2, N, group, bs_dtype, out, N, nullptr, 0, out_q, out_s,
                       pro ? &pa : nullptr, (hipStream_t)stream);
  }
  SkArgs a = base_args();
  a.x = a_q;
  a.xs = a_s;
  a.M = M;
  a.K = K;
  a.seg[0] = make_seg(wg, sg, zg, N, 0);
  a.seg[1] = make_seg(wu, su, zu, N, 0);
  a.nseg = 2;
  a.ncols = N;
  a.group = (wk == WK_W4) ? group : 64;
  a.sdt = bs_dtype;
  a.out = out;
  a.ldo = N;
  a.odt = QLIN_BF16;
  a.oq = out_q;
  a.os = out_s;
  a.pro = pa;
  Problem P{ACT_I8, wk, epi, zg != nullptr, M, K, a.group, 2, N};
  return plan_and_launch(fn, P, a, ws, wsb, (hipStream_t)stream);
}

// Prefill plan: the LDS-tiled kernel with a tile shape and a split-K factor or the balanced
// schedule, the short-prompt kernel, or the skinny kernel over row tiles (its 16-row tiles
// re-read the weights from L2), whichever a time model fitted to MI355X measurements prefers.
struct PfPlan {
  bool tiled;
  int shape;
  int splits;
  int sk;  // balanced schedule: K tiles per workgroup (0 = off)
  int kg;  // rows of the short-prompt kernel's tile (32 or 64), with `splits`; 0: not that kernel
};

// Short-prompt kernel (prefill_kg.hip), microseconds: t0 + 32-wide steps of a wave x s[q - 1]
// for each round of q workgroups per CU (`cap` resident at once) + the bytes its tiles read,
// mb per MB + the exchange, x0 + xs per split and xmb per MB of partial tiles.  Fitted to
// MI355X measurements of both tiles with 1, 2, 3, 4, 6 and 8 splits (M = 17-512, shapes
// 1024x1024 to 4096x12288, weights from HBM): 4-7 % rms, choices within 0.3 % of the best.
struct KgTime {
  double t0, s[3], mb, x0, xs, xmb;
  int cap;
};
constexpr KgTime kKgTime[2][2] = {  // [W8, W4][32, 64 rows]
    {{3.8, {0.27, 0.46, 0.73}, 0.0206, 0.36, 0.41, 0.42, 3}, {4.5, {0.30, 0.62, 0}, 0.0243, 0.28, 0.43, 0.37, 2}},
    {{4.0, {0.37, 0.44, 0.65}, 0.0149, 0.11, 0.40, 0.41, 3}, {4.8, {0.46, 0.68, 0}, 0.0133, 0.13, 0.42, 0.41, 2}}};
// (larger grids were measured behind the large tiles, which re-read less; a W4 call that may
// not use those takes them: 80 such calls of up to 4000 workgroups 1.49x the 16-row tiles on
// average, none slower)
constexpr long long kKgWorkgroups = 1024;
// Above the rows of the fit the model is up to a third below what runs (more tiles of few
// steps each).  Measured there at 518 calls of 513-4096 rows against the plans without this
// kernel: W8 takes it where it is 17 % ahead instead of 10 (8 calls were up to 21 % slower for
// it, now 2 of them up to 12; K = 1280, N = 1248 at 1323 rows 16.7 us, 15.0 on 128x128 tiles),
// and a W4 round of two 64-row workgroups to a CU costs what it does with many tiles.
constexpr int kKgRows = 512;
constexpr double kKgManyRowsW4 = 0.82;

// The best short-prompt plan of a call: its time in seconds (negative if there is none).
double plan_kg(int wk, int M, int K, int N, size_t part_cap, long long most, PfPlan* plan) {
  double best = -1.0;
  for (int k = 0; k < 2; ++k) {
    const KgTime& m = kKgTime[wk == WK_W4][k];
    const int bm = 32 << k;
    const long long tiles = (long long)((M + bm - 1) / bm) * ((N + 63) / 64);
    const double mb = (double)tiles * K * (2.0 * bm + 64.0 * (wk == WK_W4 ? 0.5 : 1.0)) * 1e-6;
    for (const int S : {1, 2, 3, 4, 6, 8}) {
      const long long wgs = tiles * S;
      const double part = (double)wgs * bm * 64 * sizeof(float);
      if (wgs > most) break;
      if (S > 1 && (part > (double)part_cap || tiles > (long long)(kCounterBytes / sizeof(unsigned)))) break;
      const int steps = (K / 32 + 4 * S - 1) / (4 * S);
      const long long full = wgs / (256LL * m.cap), rest = wgs - full * 256LL * m.cap;
      double s[3] = {m.s[0], m.s[1], m.s[2]};
      if (wk == WK_W4 && bm == 64 && M > kKgRows) s[1] = kKgManyRowsW4;
      double st = (double)full * s[m.cap - 1];
      if (rest > 0) st += s[(rest + 255) / 256 - 1];
      const double t = m.t0 + steps * st + m.mb * mb + (S > 1 ? m.x0 + m.xs * S + m.xmb * part * 1e-6 : 0.0);
      if (best < 0.0 || t * 1e-6 < best) best = t * 1e-6, *plan = PfPlan{true, 0, S, 0, bm};
    }
  }
  return best;
}

// Time model of the large tiles (prefill_kernel.h), microseconds: t0 + rounds of 256
// workgroups (one per CU) x 64-wide K tiles x s + the bytes the tiles read, mb per MB + the
// split-K exchange, xs per split and xmb per MB of partial tiles.  128x128 fits a CU twice: a
// round of 512 workgroups costs s2 a K tile, one of up to 256 s.  With two K groups a further
// round costs rr, nothing running beside its start.  The balanced schedule (256x256 only)
// runs sk K tiles and moves partials of about every tile: 2 + 0.075 a tile.
// Fitted to MI355X measurements of every shape and split (M = 256-2048, nine shapes from
// 1024x3072 to 12288x4096), 2-5 % rms; 128x384 carries 3 % more than its fit, since its close
// calls were lost (W8 2048x6144 at M = 2048 52.5 us against 51.0 on 256x256).  128x128 is for
// grids of one to two rounds: W8 2048x6144 at M = 1024 36.8 us against 41.5 with two K groups;
// 128x384 for those 256x256 leaves short of a round: W8 2048x6144 M = 1300 46.7 against 52;
// the balanced schedule at 4096x12288, M = 2048 184 against 205.
struct TiledTime {
  int shape;
  double t0, s, s2, mb, xs, xmb, rr;
};
constexpr TiledTime kTiledTime[2][4] = {  // W8, W4
    {{PF_128x128, 5.39, 0.798, 0.822, 0.0153, 0.900, 0.269, 0},
     {PF_256x256, 7.34, 1.213, 0, 0.0232, 3.00, 0.127, 0},
     {PF_128x128_K2, 5.80, 0.438, 0, 0.0105, 0.40, 0.30, 4.5},
     {PF_128x384, 6.03, 1.201, 0, 0.0294, -1, 0, 0}},
    {{PF_128x128, 6.07, 0.906, 0.943, 0.0095, 0.737, 0.249, 0},
     {PF_256x256, 7.15, 1.522, 0, 0.0168, 2.90, 0.133, 0},
     {PF_128x128_K2, 6.10, 0.590, 0, 0.0078, 0.40, 0.30, 4.0},
     {PF_128x384, 6.44, 1.445, 0, 0.0264, -1, 0, 0}}};

// The best large-tile plan of a call; *t its time in seconds.
PfPlan plan_tiled(int wk, int M, int K, int N, size_t part_cap, double* t) {
  const int nk = K / 64;
  PfPlan best{true, PF_128x128_K2, 1, 0, 0};
  *t = -1.0;
  for (const TiledTime& m : kTiledTime[wk == WK_W4]) {
    int bm, bn, waves;
    prefill_geometry(m.shape, &bm, &bn, &waves);
    const int per_cu = m.s2 > 0 ? 2 : 1;
    const long long tiles = (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
    const double base = m.t0 + m.mb * 1e-6 * (double)tiles * K * (2.0 * bm + bn * (wk == WK_W4 ? 0.5 : 1.0));
    const bool counters = tiles <= (long long)(kCounterBytes / sizeof(unsigned));
    auto take = [&](double us, int S, int sk) {
      if (*t < 0.0 || us * 1e-6 < *t) *t = us * 1e-6, best = PfPlan{true, m.shape, S, sk, 0};
    };
    for (int S = 1; S <= 16; S *= 2) {
      const double part = (double)tiles * S * waves * 128 * 64 * sizeof(float);
      if (nk % S != 0 || (S > 1 && (nk / S < 2 || m.xs < 0 || part > (double)part_cap || !counters))) break;
      if (S > 1 && tiles * (S / 2) >= 256LL * per_cu) break;  // split-K exists to fill the chip
      const long long wgs = tiles * S, rest = wgs % (256 * per_cu);
      const double rounds = (double)(wgs / (256 * per_cu)) * (per_cu == 2 ? m.s2 : m.s) +
                            (rest == 0 ? 0.0 : rest > 256 ? m.s2 : m.s);
      take(base + rounds * (nk / S) + (double)((wgs - 1) / (256 * per_cu)) * m.rr +
               (S > 1 ? m.xs * S + m.xmb * 1e-6 * (double)tiles * S * bm * bn * sizeof(float) : 0.0), S, 0);
    }
    // the balanced schedule: every CU the same run of (tile, K tile) units, across tiles
    if (m.shape == PF_256x256 && tiles % 256 != 0 && tiles > 128 && counters &&
        (double)tiles * 2 * waves * 128 * 64 * sizeof(float) <= (double)part_cap) {
      const int sk = (int)((tiles * nk + 255) / 256);
      if (prefill_balanced_ok(tiles, nk, sk)) take(base + 2.0 + 0.075 * (double)tiles + sk * m.s, 1, sk);
    }
  }
  return best;
}

// Whether a W4 call may use the large tiles: they round the group scales into the fp16
// weights, where the 16-row tiles and the short-prompt kernel multiply fp32 dots by them, so
// calls on the 16-row tiles' side of this line (their time against tiles of 128x128 and
// 256x256, microseconds) keep the fp32 form.
// The line is fixed: it decides the arithmetic of a call, not which tile is the fastest, so its
// constants stay as they are when plan_tiled's are fitted again.  It takes the workspace into
// account as the splits of the large tiles do: a smaller one can move a call to the fp32 side.
bool w4_large_tiles(int M, int K, int N, size_t part_cap) {
  const double row_wgs = (double)((M + 15) / 16) * ((N + 127) / 128);
  const double t_rows = 5.8 + std::max(1.0, row_wgs / 256) * 2.7e-3 * K;
  const int nk = K / 64;
  for (const int big : {0, 1}) {
    const int b = big ? 256 : 128, per_cu = big ? 1 : 2, waves = big ? 8 : 4;
    const long long tiles = (long long)((M + b - 1) / b) * ((N + b - 1) / b);
    for (int S = 1; S <= 16; S *= 2) {
      if (nk % S != 0 || nk / S < 2) break;
      if (S > 1 && ((double)tiles * S * waves * 128 * 64 * sizeof(float) > (double)part_cap ||
                    tiles > (long long)(kCounterBytes / sizeof(unsigned)) || tiles * (S / 2) >= 256LL * per_cu))
        break;
      const long long wgs = tiles * S;
      const int occ = (wgs > 256 && per_cu > 1) ? 2 : 1;
      const double t_tile = big ? 1.96 : (occ == 2 ? 1.35 : 0.48);
      const double t = 5.0 + (double)((wgs + 256LL * occ - 1) / (256LL * occ)) * (nk / S) * t_tile * 1.3 +
                       (S > 1 ? 1.45 * S + 0.012 * wgs + 0.1e-6 * (double)wgs * b * b * sizeof(float) : 0.0);
      if (t < t_rows) return true;
    }
  }
  return false;
}

PfPlan plan_prefill(int wk, int M, int K, int N, size_t part_cap, bool force_tiled) {
  // rows: 16-row tiles, 4 waves over the whole K per 128 columns, 7.1 us (W4 5.8) + max(1,
  // workgroups / 256) x 3.4 ns (W4 2.7) per K row
  const bool w4 = wk == WK_W4;
  const double row_wgs = (double)((M + 15) / 16) * ((N + 127) / 128);
  const double t_rows = (w4 ? 5.8e-6 : 7.1e-6) + std::max(1.0, row_wgs / 256) * (w4 ? 2.7e-9 : 3.4e-9) * K;
  double t_tiled = 0.0;
  const PfPlan tiled = plan_tiled(wk, M, K, N, part_cap, &t_tiled);
  if (force_tiled) return tiled;
  PfPlan best{false, PF_128x128_K2, 1, 0, 0};
  double best_t = t_rows;
  const bool large = !w4 || w4_large_tiles(M, K, N, part_cap);
  if (large && t_tiled < best_t) best = tiled, best_t = t_tiled;
  // the short-prompt kernel, where its model is 10 % ahead (the rows model is off by about
  // that much): 2048x2048 at M = 128 13.6 -> 8.1 us (W8), 6144x2048 21.5 -> 13.3 (W4)
  PfPlan kg;
  const double t_kg = plan_kg(wk, M, K, N, part_cap, large ? kKgWorkgroups : 1LL << 20, &kg);
  if (t_kg >= 0.0 && t_kg < (!w4 && M > kKgRows ? 0.83 : 0.9) * best_t) return kg;
  return best;
}

// Tile order of a plan with one tile per workgroup (or its K splits): each XCD runs one
// contiguous eighth of the order, and the order goes down gm row tiles before the next
// column tile, so an XCD's run covers about gm row tiles x (run / gm) column tiles.
// gm minimises what one run reads into its XCD's L2: rows x (BM x K fp16 activations)
// + columns x (the weights of BN columns).  QLIN_PREFILL_GM overrides it (0: the order
// in groups of 8 row tiles with workgroups in launch order).
int prefill_tile_group(int wk, int M, int K, int N, int shape) {
  const char* e = getenv("QLIN_PREFILL_GM");
  if (e && *e) return std::max(0, atoi(e));
  int bm, bn, waves;
  prefill_geometry(shape, &bm, &bn, &waves);
  const long long tm = (M + bm - 1) / bm, tn = (N + bn - 1) / bn;
  const long long run = std::max<long long>(1, (tm * tn + 7) / 8);
  const double arow = (double)bm * K * 2.0, wcol = (double)K * bn * (wk == WK_W4 ? 0.5 : 1.0);
  int best = 1;
  double best_c = 0.0;
  for (int gm = 1; gm <= 64; gm *= 2) {
    const long long h = std::min<long long>(gm, tm);
    const long long rows = std::min(h, run), cols = (run + h - 1) / h;
    const double c = (double)rows * arow + (double)cols * wcol;
    if (gm == 1 || c < best_c) best_c = c, best = gm;
    if (gm >= tm) break;
  }
  return best;
}

int a16_linear(const char* fn, int wk, const void* x, int x_dtype, int M, int K, int64_t ldx, const void* w,
               const void* scale, int s_dtype, const uint8_t* zero, int group, int N, void* out, int out_dtype,
               int64_t ldo, const void* residual, int64_t ldr, void* ws, size_t wsb, void* stream) {
  QL_TRY(check_common(fn, M, K, N));
  if (M == 0 || N == 0) return QLIN_OK;
  if (!x) return fail(QLIN_ERR_INVALID, "%s: null x", fn);
  if (x_dtype != QLIN_F16) return fail(QLIN_ERR_UNSUPPORTED, "%s: activation dtype %d (fp16 only)", fn, x_dtype);
  if (!dtype_scale_ok(s_dtype)) return fail(QLIN_ERR_UNSUPPORTED, "%s: scale dtype %d", fn, s_dtype);
  if (!dtype_out_ok(out_dtype)) return fail(QLIN_ERR_UNSUPPORTED, "%s: output dtype %d", fn, out_dtype);
  if (K % 32 != 0) return fail(QLIN_ERR_UNSUPPORTED, "%s: K=%d is not a multiple of 32", fn, K);
  if (ldx < K) return fail(QLIN_ERR_INVALID, "%s: x row stride %lld < K", fn, (long long)ldx);
  if (!aligned(x, 16) || ldx % 8 != 0)
    return fail(QLIN_ERR_UNSUPPORTED, "%s: x must be 16-byte aligned with a row stride multiple of 8", fn);
  if (wk == WK_W4) QL_TRY(check_group(fn, group, K));
  QL_TRY(check_weight(fn, w, scale, zero, N, wk));
  QL_TRY(check_out16(fn, out, ldo, N, "out"));
  if (residual) QL_TRY(check_out16(fn, residual, ldr, N, "residual"));
  // More than 16 rows: the LDS-tiled MFMA kernel (tile shape and split-K from a time
  // model) or row tiles of 16 through the skinny kernel, whichever the model prefers.
  // QLIN_PREFILL ("skinny" or "tiled"), QLIN_PREFILL_SHAPE and QLIN_PREFILL_SPLITS
  // override the choice for tuning.
  const char* pimpl = getenv("QLIN_PREFILL");
  const bool force_skinny = pimpl && strcmp(pimpl, "skinny") == 0;
  const bool force_tiled = pimpl && strcmp(pimpl, "tiled") == 0;
  // the DMA kernel addresses activations with 32-bit byte offsets
  const bool fits32 = ((long long)(M - 1) * ldx + K) * 2 < (1LL << 31);
  const size_t part_cap = (ws && wsb > kPartBase) ? wsb - kPartBase : 0;
  if (M > 16 && K % 64 == 0 && !force_skinny) {
    TlArgs t;
    t.x = (const _Float16*)x;
    t.ldx = ldx;
    t.w = (const uint8_t*)w;
    t.s = scale;
    t.z = zero;
    t.M = M;
    t.N = N;
    t.K = K;
    t.group = (wk == WK_W4) ? group : 32;
    t.sdt = s_dtype;
    t.out = out;
    t.ldo = ldo;
    t.odt = out_dtype;
    t.res = residual;
    t.ldr = ldr;
    t.splits = 1;
    t.part = nullptr;
    t.cnt = nullptr;
    t.sk = 0;
    t.gm = 0;
    if (fits32) {
      PfPlan p = plan_prefill(wk, M, K, N, part_cap, force_tiled);
      if (getenv("QLIN_PREFILL_VERBOSE"))
        fprintf(stderr, "qlin prefill plan M=%d K=%d N=%d: %s shape=%d splits=%d sk=%d\n", M, K, N,
                p.kg ? "short" : p.tiled ? "tiled" : "skinny", p.kg ? p.kg : p.shape, p.splits, p.sk);
      const char* e = getenv("QLIN_PREFILL_SHAPE");
      const char* e2 = getenv("QLIN_PREFILL_SPLITS");
      const char* e3 = getenv("QLIN_PREFILL_SK");
      if ((e && *e) || (e2 && *e2) || (e3 && *e3)) {
        p.tiled = true;
        p.kg = 0;
        if (e && *e) p.shape = atoi(e);
        p.splits = (e2 && *e2) ? atoi(e2) : 1;
        p.sk = (e3 && *e3) ? atoi(e3) : 0;
        int bm, bn, waves;
        prefill_geometry(p.shape, &bm, &bn, &waves);
        const size_t tiles = (size_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
        if (!prefill_shape_ok(p.shape))
          return fail(QLIN_ERR_UNSUPPORTED, "%s: QLIN_PREFILL_SHAPE=%d unknown", fn, p.shape);
        if (p.splits < 1 || (K / 64) % p.splits != 0 ||
            (p.splits > 1 && (tiles * p.splits * waves * 128 * 64 * sizeof(float) > part_cap ||
                              tiles > kCounterBytes / sizeof(unsigned))))
          return fail(QLIN_ERR_UNSUPPORTED, "%s: QLIN_PREFILL_SPLITS=%d unusable here", fn, p.splits);
        // (the 128x384 tile has no balanced schedule)
        if (p.sk != 0 && (p.sk < 0 || p.splits != 1 || p.shape == PF_128x384 || !prefill_balanced_ok((long long)tiles, K / 64, p.sk) ||
                          tiles * 2 * waves * 128 * 64 * sizeof(float) > part_cap ||
                          tiles > kCounterBytes / sizeof(unsigned)))
          return fail(QLIN_ERR_UNSUPPORTED, "%s: QLIN_PREFILL_SK=%d unusable here", fn, p.sk);
      }
      // QLIN_PREFILL_KG="rows,splits" forces the short-prompt kernel (tuning)
      const char* ek = getenv("QLIN_PREFILL_KG");
      int kbm = 0, ksp = 0;
      if (ek && sscanf(ek, "%d,%d", &kbm, &ksp) == 2) {
        const size_t tiles = kbm > 0 ? (size_t)((M + kbm - 1) / kbm) * ((N + 63) / 64) : 0;
        if ((kbm != 32 && kbm != 64) || ksp < 1 || ksp > 64 || tiles * ksp > (1u << 24) ||
            (ksp > 1 && (tiles * ksp * kbm * 64 * sizeof(float) > part_cap || tiles > kCounterBytes / sizeof(unsigned))))
          return fail(QLIN_ERR_UNSUPPORTED, "%s: QLIN_PREFILL_KG=%d,%d unusable here", fn, kbm, ksp);
        p = PfPlan{true, 0, ksp, 0, kbm};
      }
      if (p.kg) {
        t.splits = p.splits;
        if (p.splits > 1) {
          t.cnt = (unsigned*)ws;
          t.part = (float*)((char*)ws + kPartBase);
        }
        return hip_status(fn, launch_prefill_kg(t, wk, zero != nullptr, p.kg, (hipStream_t)stream));
      }
      if (p.tiled || force_tiled) {
        t.splits = p.splits;
        t.sk = p.sk;
        if (p.sk == 0) t.gm = prefill_tile_group(wk, M, K, N, p.shape);
        if (p.splits > 1 || p.sk > 0) {
          t.cnt = (unsigned*)ws;
          t.part = (float*)((char*)ws + kPartBase);
        }
        return hip_status(fn, launch_prefill(t, wk, zero != nullptr, p.shape, (hipStream_t)stream));
      }
    }
  }
  SkArgs a = base_args();
  a.x = x;
  a.ldx = ldx;
  a.M = M;
  a.K = K;
  a.seg[0] = make_seg(w, scale, zero, N, 0);
  a.nseg = 1;
  a.ncols = N;
  a.group = (wk == WK_W4) ? group : 32;
  a.sdt = s_dtype;
  a.out = out;
  a.ldo = ldo;
  a.odt = out_dtype;
  a.res = residual;
  a.ldr = ldr;
  Problem P{ACT_F16, wk, EPI_STORE, zero != nullptr, M, K, a.group, 1, N};
  return plan_and_launch(fn, P, a, ws, wsb, (hipStream_t)stream);
}

}  // namespace

namespace qlin {

int set_error(int code, const char* msg) { return fail(code, "%s", msg); }

int gemm_i8_scratch(const char* fn, const int8_t* a_q, const float* a_s, int M, int K, const int8_t* b,
                    const void* b_s, int bs_dtype, int N, void* out, int64_t ldo, const void* residual,
                    int64_t ldr, void* scratch, size_t scratch_bytes, void* stream) {
  g_err[0] = 0;
  return engine_gemm(fn, WK_W8, a_q, a_s, M, K, b, b_s, bs_dtype, nullptr, 64, N, out, ldo, residual, ldr,
                     scratch, scratch_bytes, stream, true);
}

size_t counter_bytes() { return kCounterBytes; }
size_t poll_bytes() { return kPollBytes; }

}  // namespace qlin

extern "C" {

int qlin_version(void) { return QLIN_ABI_VERSION; }

const char* qlin_last_error(void) { return g_err; }

size_t qlin_workspace_bytes(void) { return kWorkspaceBytes; }

int qlin_gemm_i8(const int8_t* a_q, const float* a_s, int M, int K, const int8_t* b, const void* b_s, int bs_dtype,
                 int N, void* out, int64_t ldo, const void* residual, int64_t ldr, void* workspace,
                 size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  return engine_gemm("qlin_gemm_i8", WK_W8, a_q, a_s, M, K, b, b_s, bs_dtype, nullptr, 64, N, out, ldo, residual,
                     ldr, workspace, workspace_bytes, stream);
}

int qlin_gemm_w4(const int8_t* a_q, const float* a_s, int M, int K, const uint8_t* b, const void* b_s,
                 int bs_dtype, const uint8_t* b_z, int group, int N, void* out, int64_t ldo, const void* residual,
                 int64_t ldr, void* workspace, size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  return engine_gemm("qlin_gemm_w4", WK_W4, a_q, a_s, M, K, b, b_s, bs_dtype, b_z, group, N, out, ldo, residual,
                     ldr, workspace, workspace_bytes, stream);
}

int qlin_proj3_i8(const int8_t* a_q, const float* a_s, int M, int K, const int8_t* w1, const void* s1, int n1,
                  const int8_t* w2, const void* s2, int n2, const int8_t* w3, const void* s3, int n3, int bs_dtype,
                  void* out, int64_t ldo, void* workspace, size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  return engine_proj3("qlin_proj3_i8", WK_W8, a_q, a_s, M, K, w1, s1, nullptr, n1, w2, s2, nullptr, n2, w3, s3,
                      nullptr, n3, bs_dtype, 64, out, ldo, workspace, workspace_bytes, stream);
}

int qlin_proj3_w4(const int8_t* a_q, const float* a_s, int M, int K, const uint8_t* w1, const void* s1,
                  const uint8_t* z1, int n1, const uint8_t* w2, const void* s2, const uint8_t* z2, int n2,
                  const uint8_t* w3, const void* s3, const uint8_t* z3, int n3, int bs_dtype, int group, void* out,
                  int64_t ldo, void* workspace, size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  return engine_proj3("qlin_proj3_w4", WK_W4, a_q, a_s, M, K, w1, s1, z1, n1, w2, s2, z2, n2, w3, s3, z3, n3,
                      bs_dtype, group, out, ldo, workspace, workspace_bytes, stream);
}

int qlin_mlp_gate_up_i8(const int8_t* a_q, const float* a_s, int M, int K, const int8_t* wg, const void* sg,
                        const int8_t* wu, const void* su, int bs_dtype, int N, void* out, void* workspace,
                        size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  return engine_gate_up("qlin_mlp_gate_up_i8", WK_W8, EPI_GATEUP, a_q, a_s, M, K, wg, sg, nullptr, wu, su, nullptr,
                        bs_dtype, 64, N, out, nullptr, nullptr, workspace, workspace_bytes, stream);
}

int qlin_mlp_gate_up_w4(const int8_t* a_q, const float* a_s, int M, int K, const uint8_t* wg, const void* sg,
                        const uint8_t* zg, const uint8_t* wu, const void* su, const uint8_t* zu, int bs_dtype,
                        int group, int N, void* out, void* workspace, size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  return engine_gate_up("qlin_mlp_gate_up_w4", WK_W4, EPI_GATEUP, a_q, a_s, M, K, wg, sg, zg, wu, su, zu, bs_dtype,
                        group, N, out, nullptr, nullptr, workspace, workspace_bytes, stream);
}

int qlin_mlp_gate_up_quant_i8(const int8_t* a_q, const float* a_s, int M, int K, const int8_t* wg, const void* sg,
                              const int8_t* wu, const void* su, int bs_dtype, int N, int8_t* out_q, float* out_s,
                              void* workspace, size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  return engine_gate_up("qlin_mlp_gate_up_quant_i8", WK_W8, EPI_GATEUP_Q, a_q, a_s, M, K, wg, sg, nullptr, wu, su,
                        nullptr, bs_dtype, 64, N, nullptr, out_q, out_s, workspace, workspace_bytes, stream);
}

int qlin_mlp_gate_up_quant_w4(const int8_t* a_q, const float* a_s, int M, int K, const uint8_t* wg, const void* sg,
                              const uint8_t* zg, const uint8_t* wu, const void* su, const uint8_t* zu,
                              int bs_dtype, int group, int N, int8_t* out_q, float* out_s, void* workspace,
                              size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  return engine_gate_up("qlin_mlp_gate_up_quant_w4", WK_W4, EPI_GATEUP_Q, a_q, a_s, M, K, wg, sg, zg, wu, su, zu,
                        bs_dtype, group, N, nullptr, out_q, out_s, workspace, workspace_bytes, stream);
}

int qlin_linear_w8(const void* x, int x_dtype, int M, int K, int64_t ldx, const int8_t* w, const void* scale,
                   int s_dtype, int N, void* out, int out_dtype, int64_t ldo, const void* residual, int64_t ldr,
                   void* workspace, size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  return a16_linear("qlin_linear_w8", WK_W8, x, x_dtype, M, K, ldx, w, scale, s_dtype, nullptr, 32, N, out,
                    out_dtype, ldo, residual, ldr, workspace, workspace_bytes, stream);
}

int qlin_linear_w4(const void* x, int x_dtype, int M, int K, int64_t ldx, const uint8_t* w, const void* scale,
                   int s_dtype, const uint8_t* zero, int group, int N, void* out, int out_dtype, int64_t ldo,
                   const void* residual, int64_t ldr, void* workspace, size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  return a16_linear("qlin_linear_w4", WK_W4, x, x_dtype, M, K, ldx, w, scale, s_dtype, zero, group, N, out,
                    out_dtype, ldo, residual, ldr, workspace, workspace_bytes, stream);
}

// ---------------------------------------------------------------------------
// Activation producers (kernels/norm.py) and the linears that make their own
// activations from them
// ---------------------------------------------------------------------------

static ProArgs pro_from(const qlin_producer* p) {
  ProArgs a{};
  a.kind = p->kind;
  a.x = p->x;
  a.ldx = p->ldx;
  a.xdt = p->x_dtype;
  a.g = p->g;
  a.ldg = p->ldg;
  a.w = p->w;
  a.wdt = p->w_dtype;
  a.hd = p->hd;
  a.one_plus = p->one_plus;
  a.eps = p->eps;
  a.q = p->q;
  a.s = p->s;
  return a;
}

static int produce(const char* fn, ProArgs p, int M, int K, void* stream) {
  if (M < 0 || K < 0) return fail(QLIN_ERR_INVALID, "%s: bad sizes M=%d K=%d", fn, M, K);
  if (M == 0 || K == 0) return QLIN_OK;
  if (!p.q || !p.s) return fail(QLIN_ERR_INVALID, "%s: null q or s", fn);
  size_t none = 0;
  QL_TRY(setup_pro(fn, p, M, K, nullptr, &none));
  return hip_status(fn, launch_producer(p, M, K, (hipStream_t)stream));
}

int qlin_rmsnorm_quant(const void* x, int64_t ldx, int x_dtype, const void* w, int w_dtype, int M, int K, float eps,
                       int one_plus, int8_t* q, float* s, void* stream) {
  g_err[0] = 0;
  ProArgs p{};
  p.kind = PRO_RMSNORM;
  p.x = x;
  p.ldx = ldx;
  p.xdt = x_dtype;
  p.w = w;
  p.wdt = w_dtype;
  p.one_plus = one_plus ? 1 : 0;
  p.eps = eps;
  p.q = q;
  p.s = s;
  return produce("qlin_rmsnorm_quant", p, M, K, stream);
}

int qlin_gate_mul_quant(const void* a, int64_t lda, const void* g, int64_t ldg, int dtype, int M, int N, int hd,
                        int8_t* q, float* s, void* stream) {
  g_err[0] = 0;
  ProArgs p{};
  p.kind = PRO_GATE_MUL;
  p.x = a;
  p.ldx = lda;
  p.xdt = dtype;
  p.g = g;
  p.ldg = ldg;
  p.hd = hd;
  p.q = q;
  p.s = s;
  return produce("qlin_gate_mul_quant", p, M, N, stream);
}

int qlin_norm_gated_quant(const void* v, const void* z, int64_t ldz, int dtype, const void* w, int w_dtype, int T,
                          int N, int hd, float eps, int8_t* q, float* s, void* stream) {
  g_err[0] = 0;
  ProArgs p{};
  p.kind = PRO_NORM_GATED;
  p.x = v;
  p.ldx = N;
  p.xdt = dtype;
  p.g = z;
  p.ldg = ldz;
  p.w = w;
  p.wdt = w_dtype;
  p.hd = hd;
  p.eps = eps;
  p.q = q;
  p.s = s;
  return produce("qlin_norm_gated_quant", p, T, N, stream);
}

int qlin_pro_exp_f32(const float* x, float* y, int n, void* stream) {
  g_err[0] = 0;
  if (n < 0) return fail(QLIN_ERR_INVALID, "qlin_pro_exp_f32: n=%d", n);
  if (n > 0 && (!x || !y)) return fail(QLIN_ERR_INVALID, "qlin_pro_exp_f32: null pointer");
  return hip_status("qlin_pro_exp_f32", launch_pro_exp(x, y, n, (hipStream_t)stream));
}

#define QL_PRO_ARG(fn)                                                      \
  if (!pro) return fail(QLIN_ERR_INVALID, "%s: null producer", fn);        \
  const ProArgs pa = pro_from(pro);

int qlin_pro_gemm_i8(const qlin_producer* pro, int M, int K, const int8_t* b, const void* b_s, int bs_dtype, int N,
                     void* out, int64_t ldo, const void* residual, int64_t ldr, void* workspace,
                     size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  QL_PRO_ARG("qlin_pro_gemm_i8")
  return engine_gemm("qlin_pro_gemm_i8", WK_W8, nullptr, nullptr, M, K, b, b_s, bs_dtype, nullptr, 64, N, out, ldo,
                     residual, ldr, workspace, workspace_bytes, stream, false, &pa);
}

int qlin_pro_gemm_w4(const qlin_producer* pro, int M, int K, const uint8_t* b, const void* b_s, int bs_dtype,
                     const uint8_t* b_z, int group, int N, void* out, int64_t ldo, const void* residual, int64_t ldr,
                     void* workspace, size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  QL_PRO_ARG("qlin_pro_gemm_w4")
  return engine_gemm("qlin_pro_gemm_w4", WK_W4, nullptr, nullptr, M, K, b, b_s, bs_dtype, b_z, group, N, out, ldo,
                     residual, ldr, workspace, workspace_bytes, stream, false, &pa);
}

int qlin_pro_proj3_i8(const qlin_producer* pro, int M, int K, const int8_t* w1, const void* s1, int n1,
                      const int8_t* w2, const void* s2, int n2, const int8_t* w3, const void* s3, int n3, int bs_dtype,
                      void* out, int64_t ldo, void* workspace, size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  QL_PRO_ARG("qlin_pro_proj3_i8")
  return engine_proj3("qlin_pro_proj3_i8", WK_W8, nullptr, nullptr, M, K, w1, s1, nullptr, n1, w2, s2, nullptr, n2,
                      w3, s3, nullptr, n3, bs_dtype, 64, out, ldo, workspace, workspace_bytes, stream, &pa);
}

int qlin_pro_proj3_w4(const qlin_producer* pro, int M, int K, const uint8_t* w1, const void* s1, const uint8_t* z1,
                      int n1, const uint8_t* w2, const void* s2, const uint8_t* z2, int n2, const uint8_t* w3,
                      const void* s3, const uint8_t* z3, int n3, int bs_dtype, int group, void* out, int64_t ldo,
                      void* workspace, size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  QL_PRO_ARG("qlin_pro_proj3_w4")
  return engine_proj3("qlin_pro_proj3_w4", WK_W4, nullptr, nullptr, M, K, w1, s1, z1, n1, w2, s2, z2, n2, w3, s3, z3,
                      n3, bs_dtype, group, out, ldo, workspace, workspace_bytes, stream, &pa);
}

int qlin_pro_mlp_gate_up_quant_i8(const qlin_producer* pro, int M, int K, const int8_t* wg, const void* sg,
                                  const int8_t* wu, const void* su, int bs_dtype, int N, int8_t* out_q, float* out_s,
                                  void* workspace, size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  QL_PRO_ARG("qlin_pro_mlp_gate_up_quant_i8")
  return engine_gate_up("qlin_pro_mlp_gate_up_quant_i8", WK_W8, EPI_GATEUP_Q, nullptr, nullptr, M, K, wg, sg, nullptr,
                        wu, su, nullptr, bs_dtype, 64, N, nullptr, out_q, out_s, workspace, workspace_bytes, stream,
                        &pa);
}

int qlin_pro_mlp_gate_up_quant_w4(const qlin_producer* pro, int M, int K, const uint8_t* wg, const void* sg,
                                  const uint8_t* zg, const uint8_t* wu, const void* su, const uint8_t* zu,
                                  int bs_dtype, int group, int N, int8_t* out_q, float* out_s, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  QL_PRO_ARG("qlin_pro_mlp_gate_up_quant_w4")
  return engine_gate_up("qlin_pro_mlp_gate_up_quant_w4", WK_W4, EPI_GATEUP_Q, nullptr, nullptr, M, K, wg, sg, zg, wu,
                        su, zu, bs_dtype, group, N, nullptr, out_q, out_s, workspace, workspace_bytes, stream, &pa);
}

int qlin_w4_unpack(const uint8_t* packed, int K, int N, uint8_t* nib, void* stream) {
  g_err[0] = 0;
  if (K < 0 || N < 0 || K % 2) return fail(QLIN_ERR_INVALID, "qlin_w4_unpack: bad sizes K=%d N=%d", K, N);
  if ((long long)K * N == 0) return QLIN_OK;
  if (!packed || !nib) return fail(QLIN_ERR_INVALID, "qlin_w4_unpack: null pointer");
  return hip_status("qlin_w4_unpack", launch_w4_unpack(packed, K, N, nib, (hipStream_t)stream));
}

int qlin_w4_dequant_f32(const uint8_t* packed, const void* scale, int s_dtype, const uint8_t* zero, int group, int K,
                        int N, float* out, void* stream) {
  g_err[0] = 0;
  if (K < 0 || N < 0 || K % 2) return fail(QLIN_ERR_INVALID, "qlin_w4_dequant_f32: bad sizes K=%d N=%d", K, N);
  if (group <= 0 || K % group) return fail(QLIN_ERR_INVALID, "qlin_w4_dequant_f32: bad group %d", group);
  if (!dtype_scale_ok(s_dtype)) return fail(QLIN_ERR_UNSUPPORTED, "qlin_w4_dequant_f32: scale dtype %d", s_dtype);
  if ((long long)K * N == 0) return QLIN_OK;
  if (!packed || !scale || !out) return fail(QLIN_ERR_INVALID, "qlin_w4_dequant_f32: null pointer");
  return hip_status("qlin_w4_dequant_f32",
                    launch_w4_dequant(packed, scale, s_dtype, zero, group, K, N, out, (hipStream_t)stream));
}

int qlin_w8_dequant_f32(const int8_t* w, const void* scale, int s_dtype, int K, int N, float* out, void* stream) {
  g_err[0] = 0;
  if (K < 0 || N < 0) return fail(QLIN_ERR_INVALID, "qlin_w8_dequant_f32: bad sizes K=%d N=%d", K, N);
  if (!dtype_scale_ok(s_dtype)) return fail(QLIN_ERR_UNSUPPORTED, "qlin_w8_dequant_f32: scale dtype %d", s_dtype);
  if ((long long)K * N == 0) return QLIN_OK;
  if (!w || !scale || !out) return fail(QLIN_ERR_INVALID, "qlin_w8_dequant_f32: null pointer");
  return hip_status("qlin_w8_dequant_f32", launch_w8_dequant(w, scale, s_dtype, K, N, out, (hipStream_t)stream));
}

int qlin_requant_w4_sym(const float* w, int K, int N, int group, uint8_t* packed, uint16_t* scale_bf16,
                        void* stream) {
  g_err[0] = 0;
  if (K < 0 || N < 0) return fail(QLIN_ERR_INVALID, "qlin_requant_w4_sym: bad sizes K=%d N=%d", K, N);
  if ((group != 32 && group != 64) || K % group != 0)
    return fail(QLIN_ERR_INVALID, "qlin_requant_w4_sym: group %d must be 32 or 64 and divide K=%d", group, K);
  if (K / group > 65535) return fail(QLIN_ERR_UNSUPPORTED, "qlin_requant_w4_sym: K=%d too large", K);
  if ((long long)K * N == 0) return QLIN_OK;
  if (!w || !packed || !scale_bf16) return fail(QLIN_ERR_INVALID, "qlin_requant_w4_sym: null pointer");
  return hip_status("qlin_requant_w4_sym",
                    launch_requant_w4(w, K, N, group, packed, scale_bf16, (hipStream_t)stream));
}

int qlin_requant_w8_row(const float* w, int K, int N, int8_t* q, float* scale, void* stream) {
  g_err[0] = 0;
  if (K < 0 || N < 0) return fail(QLIN_ERR_INVALID, "qlin_requant_w8_row: bad sizes K=%d N=%d", K, N);
  if ((K + 63) / 64 > 65535) return fail(QLIN_ERR_UNSUPPORTED, "qlin_requant_w8_row: K=%d too large", K);
  if ((long long)K * N == 0) return QLIN_OK;
  if (!w || !q || !scale) return fail(QLIN_ERR_INVALID, "qlin_requant_w8_row: null pointer");
  return hip_status("qlin_requant_w8_row", launch_requant_w8(w, K, N, q, scale, (hipStream_t)stream));
}

int qlin_w4_repack_gptq(const int32_t* qweight, int K, int N, uint8_t* packed, void* stream) {
  g_err[0] = 0;
  if (K < 0 || N < 0 || K % 8 != 0)
    return fail(QLIN_ERR_INVALID, "qlin_w4_repack_gptq: K=%d must be a multiple of 8, N=%d", K, N);
  if ((long long)K * N == 0) return QLIN_OK;
  if (!qweight || !packed) return fail(QLIN_ERR_INVALID, "qlin_w4_repack_gptq: null pointer");
  return hip_status("qlin_w4_repack_gptq", launch_repack_gptq(qweight, K, N, packed, (hipStream_t)stream));
}

int qlin_w4_repack_awq(const int32_t* qweight, int K, int N, uint8_t* packed, void* stream) {
  g_err[0] = 0;
  if (K < 0 || N < 0 || K % 2 != 0 || N % 8 != 0)
    return fail(QLIN_ERR_INVALID, "qlin_w4_repack_awq: K=%d must be even and N=%d a multiple of 8", K, N);
  if ((long long)K * N == 0) return QLIN_OK;
  if (!qweight || !packed) return fail(QLIN_ERR_INVALID, "qlin_w4_repack_awq: null pointer");
  if (!aligned(packed, 8)) return fail(QLIN_ERR_UNSUPPORTED, "qlin_w4_repack_awq: packed must be 8-byte aligned");
  return hip_status("qlin_w4_repack_awq", launch_repack_awq(qweight, K, N, packed, (hipStream_t)stream));
}

int qlin_w4_repack_ct(const int32_t* weight_packed, int N, int W, int K, uint8_t* packed, void* stream) {
  g_err[0] = 0;
  if (N < 0 || W < 0 || K < 0 || K % 2 != 0 || (long long)K > 8LL * W)
    return fail(QLIN_ERR_INVALID, "qlin_w4_repack_ct: need even K <= 8 W (N=%d W=%d K=%d)", N, W, K);
  if (N % 16 != 0) return fail(QLIN_ERR_UNSUPPORTED, "qlin_w4_repack_ct: N=%d is not a multiple of 16", N);
  if ((long long)N * K == 0) return QLIN_OK;
  if (!weight_packed || !packed) return fail(QLIN_ERR_INVALID, "qlin_w4_repack_ct: null pointer");
  if (!aligned(weight_packed, 4) || !aligned(packed, 16))
    return fail(QLIN_ERR_UNSUPPORTED, "qlin_w4_repack_ct: weight_packed 4-byte and packed 16-byte aligned");
  if ((K / 2 + 63) / 64 > 65535) return fail(QLIN_ERR_UNSUPPORTED, "qlin_w4_repack_ct: K=%d too large", K);
  return hip_status("qlin_w4_repack_ct", launch_repack_ct(weight_packed, N, W, K, packed, (hipStream_t)stream));
}

int qlin_w4_zeros_unpack(const int32_t* qzeros, int G, int N, int awq_order, int add, uint8_t* zeros,
                         void* stream) {
  g_err[0] = 0;
  if (G < 0 || N < 0 || N % 8 != 0)
    return fail(QLIN_ERR_INVALID, "qlin_w4_zeros_unpack: N=%d must be a multiple of 8 (G=%d)", N, G);
  if (add < 0 || add > 240) return fail(QLIN_ERR_INVALID, "qlin_w4_zeros_unpack: add=%d out of range", add);
  if ((long long)G * N == 0) return QLIN_OK;
  if (!qzeros || !zeros) return fail(QLIN_ERR_INVALID, "qlin_w4_zeros_unpack: null pointer");
  return hip_status("qlin_w4_zeros_unpack",
                    launch_zeros_unpack(qzeros, G, N, awq_order ? 1 : 0, add, zeros, (hipStream_t)stream));
}

}  // extern "C"
