// Engine-signature calls outside the fast kernels' layout rules, gfx950: any N and
// pointers aligned only to their element size (the fast kernels need N % 16 == 0 and
// 16-byte aligned rows).  The reference's kernels mask every edge (kernels/gemm.py:50-57,
// kernels/w4.py:75-104), so a caller may hand it a weight of 4000 columns or a view
// into a larger tensor; this kernel takes those calls.
//
// Work split: a workgroup of 8 waves owns 128 columns and 16 or 32 rows; wave w folds
// the w-th eighth of K's 64-wide blocks.  Arithmetic per output:
//   W8: acc = fma(float(dot_b), a_s[b], acc) over the wave's blocks b, dot_b exact in int32;
//   W4: acc = fma(float(dot), a_s * w_s, acc) over sub-blocks of min(group, 64), dot of
//       the codes with (nibble - z) exact in int32 (kernels/w4.py:75-104);
// the eight partial sums are added in wave order, then the fast kernels' epilogues:
// y = fma(acc, column scale, residual) (W4: scale 1) stored as bf16 / fp16; or
// h = silu(g) * u, stored as bf16 or requantized per 64 columns (kernels/gemm.py:195-211).
// The split depends on K alone, so a row's result does not depend on M: rows of a batch
// equal single-row calls and chunked prompts equal unchunked ones.
//
// A row starts at any byte address, so a lane reads its 8 columns of a row with one
// unaligned 8-byte load (gfx950 takes them) and byte permutes turn 16 rows into the MFMA's
// B operands, as in the decode units.  A lane whose 8 columns would pass the end of the row
// reads the row's last 8 and keeps only the columns that are its own.
//
// Bound: HBM at decode rows, the fold (two VALU instructions per output and block) at
// prefill rows.  M = 2, K = 2048, N = 50021 (102 MB): 30.1 us (3.4 TB/s); one column per lane with byte
// loads, one wave per row, took 224.6 us. M = 304, K = 3712, N = 3001: 28 us (240 TFLOP/s), 782 us before.
// The 32-row forms take all 256 registers and spill (16 for W8, 36 for W4); the 28 us are with them.
#include <algorithm>

#include "qlin_dev.h"
#include "qlin_internal.h"

namespace qlin {

namespace {

constexpr int EW = 8;      // waves of a workgroup, each an eighth of K
constexpr int ECOLS = 128; // columns of a tile

typedef u32x2 u32x2_u __attribute__((aligned(1)));
typedef u32x4 u32x4_u __attribute__((aligned(1)));

template <typename T>
__device__ __forceinline__ T ld_any(const void* p) {  // a load at any byte address
  return *(const __attribute__((address_space(1))) T*)p;
}

// 8 consecutive bytes of a row from `p`; NARROW (rows of fewer than 8 columns): the row's
// n bytes, the last one repeated.
template <bool NARROW>
__device__ __forceinline__ u32x2 ld_cols(const uint8_t* p, int n) {
  if constexpr (!NARROW) return ld_any<u32x2_u>(p);
  uint64_t v = 0;
#pragma unroll
  for (int c = 0; c < 8; ++c) v |= (uint64_t)p[min(c, n - 1)] << (8 * c);
  return bitcast<u32x2>(v);
}

__device__ __forceinline__ i32x4 dot64(u32x4 a, u32x4 b) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(bitcast<i32x4>(a), bitcast<i32x4>(b), i32x4{0, 0, 0, 0}, 0, 0, 0);
}

// One 64-wide block in registers: the weights of the lane's 8 columns (16 rows W8, 8 byte
// rows W4), its activation operands and the scales of the rows it folds.
template <int WK, int RT>
struct EBlock {
  u32x2 w[WK == WK_W8 ? 16 : 8];
  u32x4 a[RT];
  float as[RT][4];
};

// a weight set of this tile: `w` / `s` / `z` at the lane's first column, n the row length
struct ESet {
  const uint8_t* w;
  const void* s;
  const uint8_t* z;
  int n;
  int c;
};

template <int WK, int RT, bool NARROW>
__device__ __forceinline__ void load_block(const EdgeArgs& a, const ESet& S, const int8_t* x, const float* xs,
                                           int b, const int (&ar)[RT], const int (&sr)[RT][4], EBlock<WK, RT>& B) {
  const int g = ((int)threadIdx.x & 63) >> 4;
  constexpr int R = WK == WK_W8 ? 16 : 8;  // byte rows of a lane group
  // (a uniform row address and a 32-bit lane offset: no 64-bit address per load)
  const uint32_t off = (uint32_t)(R * g) * (uint32_t)S.n + (uint32_t)S.c;
#pragma unroll
  for (int i = 0; i < R; ++i)
    B.w[i] = ld_cols<NARROW>(S.w + ((long long)b * (4 * R) + i) * S.n + off, S.n);
  const int nb = a.K >> 6;
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    B.a[t] = ld_any<u32x4_u>(x + b * 64 + (uint32_t)(ar[t] * a.K + 16 * g));
#pragma unroll
    for (int r = 0; r < 4; ++r) B.as[t][r] = (xs + b)[(uint32_t)(sr[t][r] * nb)];
  }
}

// Folds one block into acc[t][c] (row tile t, the lane's column c).  ONE: a single
// activation row, so only accumulator row 0 is read.
template <int WK, int RT, bool NARROW>
__device__ __forceinline__ void fold_block(const EdgeArgs& a, const ESet& S, int b, const EBlock<WK, RT>& B, bool one,
                                           f32x4 (&acc)[RT][8]) {
  if constexpr (WK == WK_W8) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      uint32_t x[4][4];
#pragma unroll
      for (int h = 0; h < 4; ++h) tr4(B.w[4 * h][q], B.w[4 * h + 1][q], B.w[4 * h + 2][q], B.w[4 * h + 3][q], x[h]);
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        i32x4 p[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) p[u] = dot64(B.a[t], u32x4{x[0][u], x[1][u], x[2][u], x[3][u]});
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[t][4 * q + u][0] = fmaf((float)p[u][0], B.as[t][0], acc[t][4 * q + u][0]);
        if (!one) {
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int r = 1; r < 4; ++r)
              acc[t][4 * q + u][r] = fmaf((float)p[u][r], B.as[t][r], acc[t][4 * q + u][r]);
        }
        __builtin_amdgcn_sched_barrier(0);  // (keeps one quarter's dots live at a time)
      }
    }
  } else {
    // nibbles as int8 16 (n - 8), even K then odd K; the activation operand permuted alike
    const int g = ((int)threadIdx.x & 63) >> 4;
    const int sub = a.group < 64 ? 2 : 1;
    for (int h = 0; h < sub; ++h) {
      // groups of 32: lane groups 0, 1 hold the first half of the block's K, 2, 3 the second
      const uint32_t keep = (sub == 1 || (g >> 1) == h) ? 0xFFFFFFFFu : 0u;
      const long long gi = (long long)((b * 64 + 32 * h) / a.group) * S.n + S.c;
      float ws[8];
      uint32_t zb[2];
      if constexpr (NARROW) {
#pragma unroll
        for (int c = 0; c < 8; ++c) ws[c] = load_scale(S.s, a.sdt, gi + min(c, S.n - 1)) * 0.0625f;
      } else {
        const bool f32 = a.sdt == DT_F32;
        const uint8_t* sp = (const uint8_t*)S.s + gi * (f32 ? 4 : 2);
        const u32x4 s0 = ld_any<u32x4_u>(sp), s1 = ld_any<u32x4_u>(sp + (f32 ? 16 : 0));
        cvt_scale4(s0, a.sdt, ws);
        cvt_scale4(f32 ? s1 : u32x4{s0.z, s0.w, 0, 0}, a.sdt, ws + 4);
#pragma unroll
        for (int c = 0; c < 8; ++c) ws[c] *= 0.0625f;
      }
      u32x2 zr = u32x2{0x08080808u, 0x08080808u};
      if (S.z) zr = ld_cols<NARROW>(S.z + gi, S.n);
      zb[0] = zr.x, zb[1] = zr.y;
      u32x4 ap[RT];
      i32x4 sx[RT];
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        const u32x4 v = B.a[t] & u32x4{keep, keep, keep, keep};
        ap[t] = u32x4{perm(v.y, v.x, 0x06040200u), perm(v.w, v.z, 0x06040200u), perm(v.y, v.x, 0x07050301u),
                      perm(v.w, v.z, 0x07050301u)};
        sx[t] = dot64(ap[t], u32x4{0x01010101u, 0x01010101u, 0x01010101u, 0x01010101u});
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        uint32_t lo[8], hi[8], e0[4], e1[4], o0[4], o1[4];
#pragma unroll
        for (int i = 0; i < 8; ++i) w4_split_i8x16(B.w[i][q], lo[i], hi[i]);
        tr4(lo[0], lo[1], lo[2], lo[3], e0);
        tr4(lo[4], lo[5], lo[6], lo[7], e1);
        tr4(hi[0], hi[1], hi[2], hi[3], o0);
        tr4(hi[4], hi[5], hi[6], hi[7], o1);
        int zc[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) zc[u] = (8 - (int)((zb[q] >> (8 * u)) & 0xFFu)) * 16;
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          i32x4 p[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) p[u] = dot64(ap[t], u32x4{e0[u], e1[u], o0[u], o1[u]});
#pragma unroll
          for (int u = 0; u < 4; ++u)
            acc[t][4 * q + u][0] =
                fmaf((float)(p[u][0] + zc[u] * sx[t][0]), B.as[t][0] * ws[4 * q + u], acc[t][4 * q + u][0]);
          if (!one) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
              for (int r = 1; r < 4; ++r)
                acc[t][4 * q + u][r] =
                    fmaf((float)(p[u][r] + zc[u] * sx[t][r]), B.as[t][r] * ws[4 * q + u], acc[t][4 * q + u][r]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
}

// Grid: x = tiles of 128 columns (of each projection in turn), y = tiles of 16 RT rows.
template <int WK, int RT, bool NARROW>
__global__ __launch_bounds__(64 * EW, 2) void edge_kernel(const EdgeArgs a, int ntiles) {
  __shared__ f32x4 red4[EW * 16 * ECOLS / 4];  // [wave][row][column position]
  float* red = (float*)red4;
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4;
  // neighbouring tiles share the cache lines that their edges cut: keep them on one XCD
  // (workgroup b runs on XCD b mod 8), which takes a contiguous run of the tiles
  const int xcd = (int)blockIdx.x & 7, per8 = ntiles >> 3, more = ntiles & 7;
  int tile = xcd * per8 + min(xcd, more) + ((int)blockIdx.x >> 3);
  int si = 0;
  const bool gate_up = a.epi != EPI_STORE;
  if (!gate_up)
    while (si + 1 < a.nseg && tile >= (a.seg[si].n + ECOLS - 1) / ECOLS) tile -= (a.seg[si++].n + ECOLS - 1) / ECOLS;
  const int n = a.seg[si].n, c0 = tile * ECOLS;
  const int cl = NARROW ? 0 : min(c0 + 8 * j, n - 8);  // the lane's first column
  const int row0 = (int)blockIdx.y * 16 * RT, rows = min(a.M - row0, 16 * RT);
  int ar[RT], sr[RT][4];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    ar[t] = min(16 * t + j, rows - 1);
#pragma unroll
    for (int r = 0; r < 4; ++r) sr[t][r] = min(16 * t + 4 * g + r, rows - 1);
  }
  const int8_t* const x = a.x + (long long)row0 * a.K;
  const float* const xs = a.xs + (long long)row0 * (a.K >> 6);
  const int nb = a.K >> 6, per = (nb + EW - 1) / EW;
  const int b0 = wave * per, b1 = min(nb, b0 + per);
  const bool one = rows == 1;
  const int pos = tid & (ECOLS - 1);  // this thread's column position in the epilogue
  const int pl = NARROW ? 0 : min(c0 + (pos & ~7), n - 8);
  const int col = NARROW ? pos : pl + (pos & 7);
  // a position keeps its column if no earlier lane has it
  const bool keep = NARROW ? pos < n : (c0 + (pos & ~7) < n && col >= c0 + (pos & ~7));
  float first[RT][4];  // gate sums, while up is computed
  const int nsets = gate_up ? 2 : 1;
  for (int set = 0; set < nsets; ++set) {
    const Seg& G = a.seg[gate_up ? set : si];
    const ESet S{G.w, G.s, G.z, n, cl};
    f32x4 acc[RT][8];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int c = 0; c < 8; ++c) acc[t][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    // (one block in registers at a time: two measured no faster and cost 60 registers)
    for (int b = b0; b < b1; ++b) {
      EBlock<WK, RT> B;
      load_block<WK, RT, NARROW>(a, S, x, xs, b, ar, sr, B);
      __builtin_amdgcn_sched_barrier(0);
      fold_block<WK, RT, NARROW>(a, S, b, B, one, acc);
    }
    const float cs = WK == WK_W8 ? load_scale(G.s, a.sdt, min(col, n - 1)) : 1.0f;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      if (set + t) __syncthreads();  // the sums of the last 16 rows have been read
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * g + r;
        if (16 * t + row < rows) {
          float* d = red + (wave * 16 + row) * ECOLS + 8 * j;
          *(f32x4*)d = f32x4{acc[t][0][r], acc[t][1][r], acc[t][2][r], acc[t][3][r]};
          *(f32x4*)(d + 4) = f32x4{acc[t][4][r], acc[t][5][r], acc[t][6][r], acc[t][7][r]};
        }
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 4 * i + (tid >> 7);  // uniform over a wave
        if (16 * t + row >= rows) continue;
        const long long m = row0 + 16 * t + row;
        float v = red[row * ECOLS + pos];
#pragma unroll
        for (int w = 1; w < EW; ++w) v += red[(w * 16 + row) * ECOLS + pos];
        if (!gate_up) {
          float y = v * cs;
          if (a.res && keep) y = fmaf(v, cs, load_act16(a.res, a.odt, m * a.ldr + G.col0 + col));
          if (keep) ((uint16_t*)a.out)[m * a.ldo + G.col0 + col] = to_out16(y, a.odt);
        } else if (set == 0) {
          first[t][i] = v * cs;
        } else {
          float h = silu(first[t][i]) * (v * cs);
          if (a.epi == EPI_GATEUP) {
            if (keep) ((uint16_t*)a.out)[m * a.ldo + col] = f32_to_bf16(h);
          } else {
            // the bf16 round trip, then the group's amax over the wave (64 columns; N % 64 == 0)
            h = bf16_to_f32(f32_to_bf16(h));
            float am = keep ? fabsf(h) : 0.0f;
#pragma unroll
            for (int s = 1; s < 64; s <<= 1) am = fmaxf(am, __shfl_xor(am, s));
            const float sc = fmaxf(am / 127.0f, 1e-8f);
            if (keep) a.oq[m * n + col] = (int8_t)round_i8(h / sc);
            if (keep && lane == 0) a.os[m * (n / 64) + col / 64] = sc;
          }
        }
      }
    }
  }
}

template <int WK>
void launch_wk(const EdgeArgs& a, int ntiles, bool narrow, hipStream_t st) {
  const dim3 wg(64 * EW);
  const dim3 g16((unsigned)ntiles, (unsigned)((a.M + 15) / 16)), g32((unsigned)ntiles, (unsigned)((a.M + 31) / 32));
  if (narrow) hipLaunchKernelGGL((edge_kernel<WK, 1, true>), g16, wg, 0, st, a, ntiles);
  // 32 rows share a tile's weight operands once there are more than 16
  else if (a.M <= 16) hipLaunchKernelGGL((edge_kernel<WK, 1, false>), g16, wg, 0, st, a, ntiles);
  else hipLaunchKernelGGL((edge_kernel<WK, 2, false>), g32, wg, 0, st, a, ntiles);
}

}  // namespace

hipError_t launch_edge(const EdgeArgs& e, int wk, hipStream_t st) {
  if (e.M <= 0 || e.ncols <= 0) return hipSuccess;
  // projections of fewer than 8 columns are read byte by byte, in a launch of their own
  const bool gate_up = e.epi != EPI_STORE;
  for (int narrow = 0; narrow < 2; ++narrow) {
    EdgeArgs a = e;
    int ntiles = 0;
    if (gate_up) {
      ntiles = (e.seg[0].n < 8) == (narrow != 0) ? (e.seg[0].n + ECOLS - 1) / ECOLS : 0;
    } else {
      a.nseg = 0;
      for (int i = 0; i < e.nseg; ++i) {
        if (e.seg[i].n <= 0 || (e.seg[i].n < 8) != (narrow != 0)) continue;
        a.seg[a.nseg++] = e.seg[i];
        ntiles += (e.seg[i].n + ECOLS - 1) / ECOLS;
      }
    }
    if (ntiles == 0) continue;
    // (the grid's y dimension holds 65535 row tiles)
    const int step = 16 * 65535;
    for (int m0 = 0; m0 < e.M; m0 += step) {
      EdgeArgs b = a;
      b.M = std::min(step, e.M - m0);
      b.x += (long long)m0 * e.K;
      b.xs += (long long)m0 * (e.K / 64);
      if (b.out) b.out = (uint16_t*)b.out + (long long)m0 * e.ldo;
      if (b.res) b.res = (const uint16_t*)b.res + (long long)m0 * e.ldr;
      if (b.oq) b.oq += (long long)m0 * e.ncols;
      if (b.os) b.os += (long long)m0 * (e.ncols / 64);
      if (wk == WK_W8) launch_wk<WK_W8>(b, ntiles, narrow != 0, st);
      else launch_wk<WK_W4>(b, ntiles, narrow != 0, st);
      const hipError_t err = hipGetLastError();
      if (err != hipSuccess) return err;
    }
  }
  return hipSuccess;
}

}  // namespace qlin
