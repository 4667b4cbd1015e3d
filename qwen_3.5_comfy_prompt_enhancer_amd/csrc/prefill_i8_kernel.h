// Tiled int8-activation GEMM for the engine-signature calls with more than 16 rows
// (prefill chunks), gfx950: int8 or W4 weights; the store epilogue and the fused
// gate/up epilogues (silu(g) * u, optionally requantized per 64 columns).
//
// Replaces the prefill-sized launches of gemm_i8, gemm_w4, proj3(_w4) and
// mlp_gate_up(_quant)(_w4) (kernels/gemm.py:20-312; kernels/w4.py:64-323) with the
// reference's arithmetic: an exact int32 dot per 64-wide activation block, then
// `acc += float(dot) * a_s[m, block]` in fp32 (W4: per 64-wide weight sub-block,
// `acc += float(dot) * (a_s * b_s[group, n])`, w4.py:103-104), then the column scale
// (W8) and either the residual and a 16-bit store (gemm.py:43-57) or, for gate/up
// (two weight sets feeding one tile), h = silu(g) * u, stored as bf16 or rounded
// through bf16 and quantized per 64 columns with max(amax / 127, 1e-8) and round
// half away from zero (gemm.py:195-211).
//
//   * Workgroup tile: 128 x 128 of 8 waves (2 x 2 wave tiles of 64 x 64, times two K
//     groups), or 64, 96, 128 or 160 rows x 64 columns of 4 waves (2 wave tiles times two K
//     groups) for calls whose rows or columns would leave the large tile half empty or the
//     chip half idle: with 137 rows the 128-row tile computes 256.  The host's time model
//     (abi.hip, tile_time) chooses; the K order and so the bits are the same.  A stage of
//     the LDS ring holds two activation blocks (128 K); group kg computes block
//     2 * stage + kg; at the end the two groups' accumulators are added through LDS, each
//     group finishing half of the 16-row blocks (group 0 finishing all of them left four of
//     eight waves idle in the epilogue: a W8 2048-hidden layer's linears at M = 512 134.2 ->
//     131.6 us with the producers, a W4 4096-hidden one's at M = 137 220.9 -> 216.7).
//   * MFMA: v_mfma_i32_16x16x64_i8, one instruction per 64-wide block, started from
//     an inline zero, with the weights as its A operand and the activations as B: lane
//     (g, j) supplies K bytes 16g..16g+15 of weight column 4j + t and of activation row j,
//     and accumulates 16 adjacent columns of row j.  So it folds one activation scale per
//     16-row block (four with the operands the other way round: gemm_i8 8192x2048 at M = 512
//     without a split 72.3 us against 69.3, 2048x6144 25.6 against 24.5; W4 1 %, gate/up
//     equal).  Weight bytes are N-contiguous in
//     LDS (as in HBM, rows padded per lane group); each lane reads 4 adjacent columns
//     of its 16 K rows (one dword per row) and 4x4 byte transposes turn them into the
//     4 operands.  W4: the nibbles become int8 16 * (n - 8) (even K then odd K), the
//     activation operand is permuted to the same order, and the scale product carries the
//     1/16 (exact); explicit zeros add (8 - z) * sum(a) from one more MFMA against all-ones.
//   * Copies: global -> registers (three stages ahead; two for gate/up and for 160 rows,
//     whose accumulators leave no second set of registers) -> LDS (one stage ahead), one
//     barrier per stage.  Every address in the loop is a per-thread value made before it plus
//     the stage's scalar offset.
//   * Bound: the fold, two VALU instructions per output and block (three for W4), at about
//     two thirds of their issue rate.  Reading the next stage's operands into registers
//     while the current one is folded (three LDS stages) changed nothing (27.9 us at
//     2048x8192 W8, M = 512; small tiles 2-5 % slower).
//   * Split-K: `splits` workgroups per tile over equal ranges of 64-wide blocks; each
//     stores its fp32 partial tile (both weight sets for gate/up; device-coherent) and
//     counts its arrival, and the last to arrive sums the partials in split order and
//     runs the epilogue.
//   * The K order of every output element is fixed (blocks in order within each K
//     group, then group 0 + group 1, then splits in order), so rows do not depend on M
//     or on the chunking for a given split count.
#pragma once

#include "qlin_dev.h"
#include "qlin_internal.h"

namespace qlin {

namespace {

constexpr int GROUP_M = 8;  // tile order: 8 row tiles per group share weight column tiles in L2

// RB: 16-row blocks of a wave tile; WNW: 64-column wave tiles per workgroup row.  A
// workgroup's tile is 32 RB rows x 64 WNW columns (2 x WNW wave tiles of 16 RB x 64, times
// two K groups): <4, 2> is the 128 x 128 tile of 8 waves, <RB, 1> tiles of 4 waves.
template <int WK, int NS, int RB, int WNW>
struct Gi8 {
  static constexpr int BM = 32 * RB;
  static constexpr int BN = 64 * WNW;
  static constexpr int WAVES = 4 * WNW;
  static constexpr int THREADS = 64 * WAVES;
  static constexpr bool W4 = WK == WK_W4;
  static constexpr int A_BLK = BM * 64;                 // activation bytes of one block
  static constexpr int B_ROWS = W4 ? 32 : 64;           // weight rows of one block
  // Weight rows are N-contiguous (128 bytes), with 64 bytes of padding after every
  // group of RG rows, RG = the rows of one MFMA lane group (16 int8, 8 packed).  The
  // four lane groups of a ds_read_b32 then start 16 dwords apart modulo the 64 banks
  // and read without bank conflicts (unpadded they all hit the same 16 banks).
  static constexpr int RG = W4 ? 8 : 16;
  static constexpr int B_PAD = 64;
  static constexpr int B_BLK = B_ROWS * BN + (B_ROWS / RG) * B_PAD;  // one block of one set
  static __device__ __forceinline__ int b_row(int r) { return r * BN + (r / RG) * B_PAD; }
  static constexpr int B_OFF = 2 * A_BLK;               // weights: [set][2 blocks]
  static constexpr int AS_OFF = B_OFF + NS * 2 * B_BLK;  // activation scales: [2][BM] fp32
  static constexpr int BS_OFF = AS_OFF + 2 * BM * 4;    // W4 group scales / 16: [set][2][BN] fp32
  static constexpr int BZ_OFF = BS_OFF + (W4 ? NS * 2 * BN * 4 : 0);  // W4: 16 (8 - zero), [set][2][BN] int32
  static constexpr int STAGE = BZ_OFF + (W4 ? NS * 2 * BN * 4 : 0);
  static constexpr int RED = 2 * WNW * 16 * RB * 64 * 4;  // one set of group 1's accumulators at the end
  static constexpr int LDS = (2 * STAGE > RED) ? 2 * STAGE : RED;
};

__device__ __forceinline__ uint32_t rfl(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// activation row r's 16-byte chunk c within a block: rows of 64 bytes, chunks swizzled
// so the 8-lane phases of ds_read_b128 hit distinct banks
__device__ __forceinline__ int a_off(int r, int c) { return r * 64 + 16 * (c ^ ((r >> 2) & 3)); }

}  // namespace

// Waves per SIMD a variant's registers are budgeted for: two (256 registers), or three
// (168) for the smallest tile.
template <int NS, int RB, int WNW>
constexpr int kI8Occ = (WNW == 1 && NS * RB <= 2) ? 3 : 2;

template <int WK, bool HZ, int EPI, int RB, int WNW>
__global__ __launch_bounds__(256 * WNW)
__attribute__((amdgpu_waves_per_eu(kI8Occ<(EPI == EPI_STORE) ? 1 : 2, RB, WNW>)))
void prefill_i8_kernel(const SkArgs a) {
  constexpr int NS = (EPI == EPI_STORE) ? 1 : 2;  // weight sets feeding one tile
  using G = Gi8<WK, NS, RB, WNW>;
  constexpr int BM = G::BM, BN = G::BN, THREADS = G::THREADS;
  static_assert(WNW == 1 || RB == 4, "the 8-wave tile has 128 rows");
  constexpr int NA = RB / WNW;                          // 16-byte activation chunks per thread and stage
  constexpr int NAS = (2 * BM + THREADS - 1) / THREADS;  // activation scales per thread and stage
  constexpr bool W4 = G::W4;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

  const int tid = threadIdx.x;
  const int wave = (int)rfl((uint32_t)tid >> 6), lane = tid & 63;
  const int j = lane & 15, g = lane >> 4;
  const int kg = wave / (2 * WNW), wm = (wave / WNW) & 1, wn = wave % WNW;
  const int M = a.M, K = a.K;
  // split-K: `S` workgroups per output tile, each over nk consecutive 64-wide blocks
  // from kb0
  // Workgroups go to the 8 XCDs in turn; with a.gm set, XCD x's workgroups (b = x,
  // x + 8, ...) take one contiguous run of the tile order (a tile's splits included).
  const int S = a.splits;
  const int b = (int)blockIdx.x, W = (int)gridDim.x;
  const int v = a.gm > 0 ? (b & 7) * (W >> 3) + min(b & 7, W & 7) + (b >> 3) : b;
  const int tile = v / S, split = v % S;
  const int nk = K / 64 / S;
  const int kb0 = split * nk;

  // grouped tile order: runs of consecutive tiles cover gm row tiles x a few column
  // tiles, so the workgroups of one XCD share activation and weight tiles in its L2
  const int tiles_m = (M + BM - 1) / BM, tiles_n = a.ntiles;
  const int gm = a.gm > 0 ? a.gm : GROUP_M;
  const int per_group = gm * tiles_n;
  const int grp = tile / per_group;
  const int first_m = grp * gm;
  const int gsize = min(tiles_m - first_m, gm);
  const int tm = first_m + (tile % per_group) % gsize;
  const int tn = (tile % per_group) / gsize;
  int si = 0;
  if constexpr (EPI == EPI_STORE) {
    if (a.nseg > 1 && tn >= a.seg[1].tile0) si = 1;
    if (a.nseg > 2 && tn >= a.seg[2].tile0) si = 2;
  }
  const Seg sg = a.seg[si];
  const uint8_t* wset[NS];
  const void* sset[NS];
  const uint8_t* zset[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    wset[s] = a.seg[si + s].w;
    sset[s] = a.seg[si + s].s;
    zset[s] = a.seg[si + s].z;
  }
  const int n = sg.n;
  const int ncol0 = (tn - sg.tile0) * BN;  // tile's first column within its matrix
  const int m0 = tm * BM;

  // ---------------- copies: global -> registers -> LDS ----------------
  // Per stage and thread: NA 16-byte chunks of activations, two (W4: one) of each weight
  // set, NAS activation scales, one W4 group scale and zero.  Rows past M and blocks past the last read
  // clamped, in-bounds addresses and are never used.
  const int8_t* xq = (const int8_t*)a.x;
  const int NG = K / 64;
  struct Regs {
    u32x4 av[NA];
    u32x4 bv[NS][W4 ? 1 : 2];
    float as_[NAS];
    uint32_t bs;  // W4: raw dword of one group scale of set tid / 256
    uint32_t bz;  // W4 with zeros: the matching zero
  };
  // The block of every activation and weight load below is uniform over a wave (its K group
  // is a function of the wave), so each address is a per-thread offset fixed for the whole loop plus the
  // block's offset in a scalar register: buffer loads over the activations, weights and
  // activation scales (the host keeps each under 2^31 bytes), no per-stage address
  // arithmetic on the vector ALU.
  const __amdgpu_buffer_rsrc_t xr = part_rsrc(xq, (unsigned)((long long)M * K));
  const __amdgpu_buffer_rsrc_t sr = part_rsrc(a.xs, (unsigned)((long long)M * NG * 4));
  __amdgpu_buffer_rsrc_t wr[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) wr[s] = part_rsrc(wset[s], (unsigned)((long long)(W4 ? K / 2 : K) * n));
  // Activation chunk q of a stage: block q / (4 BM), row, 16-byte chunk.  Its block (uniform
  // over a wave: 4 BM is a multiple of 64), global offset and place in a stage's LDS are
  // computed once: in the loop, the block's v_readfirstlane kept the compiler from moving any
  // of it out (382 VALU instructions in two stages instead of 336: gemm_i8 8192x2048 at
  // M = 1024 without a split 75.0 us against 69.2, gate/up 2048x6144 86.3 against 80.0).
  constexpr bool XB = THREADS == 4 * BM;  // chunk i is block i's: one offset for both
  int xk2[NA];
  unsigned xoff[NA], xdst[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int q = tid + THREADS * i;
    xk2[i] = XB ? i : (int)rfl((uint32_t)(q / (4 * BM)));
    const int r = (XB ? tid : q - 4 * BM * xk2[i]) >> 2, c = tid & 3;
    xoff[i] = (unsigned)(min(m0 + r, M - 1) * K + 16 * c);
    xdst[i] = (unsigned)(xk2[i] * G::A_BLK + a_off(r, c));
  }
  constexpr int BCH = BN / 16;                    // 16-byte chunks of a weight row
  constexpr int BPB = (W4 ? 32 : 64) * BCH;       // and of a block
  const int wk2 = W4 ? (int)rfl((uint32_t)tid / BPB) : 0;
  const int wrow = (tid % BPB) / BCH, wch = tid % BCH;  // W8: block i's row and chunk alike
  const unsigned woff = (unsigned)(wrow * n + ncol0 + 16 * wch);
  const unsigned wdst = (unsigned)(wk2 * G::B_BLK + G::b_row(wrow) + 16 * wch);
  // activation scale e of a stage: block e / BM, row e % BM
  constexpr bool SU = BM % 64 == 0;  // its block is uniform over a wave
  int sk2[NAS];
  unsigned soff[NAS];
#pragma unroll
  for (int i = 0; i < NAS; ++i) {
    const int e = tid + THREADS * i;
    sk2[i] = SU ? (int)rfl((uint32_t)(e / BM)) : e / BM;
    soff[i] = (unsigned)(min(m0 + e % BM, M - 1) * NG * 4);
  }
  auto fetch = [&](Regs& rg, int st) {
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int blk = kb0 + min(2 * st + xk2[i], nk - 1);
      rg.av[i] = bitcast<u32x4>(__builtin_amdgcn_raw_buffer_load_b128(xr, xoff[i], blk * 64, 0));
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if constexpr (W4) {
        const int blk = kb0 + min(2 * st + wk2, nk - 1);
        rg.bv[s][0] = bitcast<u32x4>(__builtin_amdgcn_raw_buffer_load_b128(wr[s], woff, blk * 32 * n, 0));
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int blk = kb0 + min(2 * st + i, nk - 1);
          rg.bv[s][i] = bitcast<u32x4>(__builtin_amdgcn_raw_buffer_load_b128(wr[s], woff, blk * 64 * n, 0));
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NAS; ++i) {
      const int e = tid + THREADS * i;
      if (e < 2 * BM) {
        const int blk = kb0 + min(2 * st + sk2[i], nk - 1);
        rg.as_[i] = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(sr, soff[i] + (SU ? 0 : 4 * blk), SU ? 4 * blk : 0, 0));
      }
    }
    if constexpr (W4) {
      // group scales (and zeros) of both blocks: 2 BN per set, thread tid takes one of
      // set tid / (2 BN)
      const int s = tid / (2 * BN);
      if (s < NS) {
        const int t2 = tid % (2 * BN), k2 = t2 / BN, c = t2 % BN;
        const int blk = kb0 + min(2 * st + k2, nk - 1);
        const long long gi = (long long)(blk * 64 / a.group) * n + ncol0 + c;
        rg.bs = ld_scale1_raw(sset[s], a.sdt, gi);  // converted at the LDS store
        if constexpr (HZ) rg.bz = ld_global<uint8_t>(zset[s] + gi);
      }
    }
  };
  auto store = [&](const Regs& rg, int buf) {
    uint8_t* base = lds + buf * G::STAGE;
#pragma unroll
    for (int i = 0; i < NA; ++i) *(u32x4*)(base + xdst[i]) = rg.av[i];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      uint8_t* sb = base + G::B_OFF + s * 2 * G::B_BLK;
      if constexpr (W4) {
        *(u32x4*)(sb + wdst) = rg.bv[s][0];
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i) *(u32x4*)(sb + i * G::B_BLK + wdst) = rg.bv[s][i];
      }
    }
#pragma unroll
    for (int i = 0; i < NAS; ++i) {
      const int e = tid + THREADS * i;
      if (e < 2 * BM) ((float*)(base + G::AS_OFF))[e] = rg.as_[i];
    }
    if constexpr (W4) {
      if (tid / (2 * BN) < NS) {
        // gi of the fetch has the parity of tid (n and ncol0 are even)
        ((float*)(base + G::BS_OFF))[tid] = cvt_scale1(rg.bs, a.sdt, tid) * 0.0625f;
        if constexpr (HZ) ((int*)(base + G::BZ_OFF))[tid] = (8 - (int)rg.bz) * 16;
      }
    }
  };

  f32x4 acc[NS][RB][4];
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[s][rb][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // WA: the weights are the MFMA's A operand and the activations its B operand: lane (g, j)
  // holds, of instruction t, D rows 4g + r = weight columns 16g + 4r + t and D column j =
  // activation row j.  So a lane folds one activation row per block of 16 (one a_s value
  // instead of four) and ends with 16 adjacent columns of it.  With zeros the other way
  // round: lane (g, j) ends with columns 4j .. 4j + 3 of rows 4g + r, and holds 4 group
  // scales and 4 zeros instead of 16 of each, which gate/up's registers have no room for
  // (its loop reloaded spilled addresses, waiting for the copies in flight: 4096x12288 at
  // M = 512 on 128x128 276 us against 210; store calls within 3 % but for 160 rows, 6 % behind).
  constexpr bool WA = !HZ;
  auto mfma = [](i32x4 w, i32x4 x) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(WA ? w : x, WA ? x : w, i32x4{0, 0, 0, 0}, 0, 0, 0);
  };
  constexpr int LC = WA ? 16 : 4, LR = 16 / LC;  // columns and rows (per block of 16) of a lane
  const int cb = wn * 64 + 4 * j;                // first of the 4 columns whose operand the lane builds
  const int ccol = WA ? wn * 64 + 16 * g : cb;   // first of the columns the lane accumulates
  using ScaleA = std::conditional_t<WA, float, f32x4>;  // a lane's activation scales of a block of 16 rows

  // Operands of one 64-wide block: a weight set's raw from LDS, and the activations'.
  struct Wop {
    uint32_t d[W4 ? 8 : 16];
  };
  struct Aop {
    i32x4 av[RB];
    ScaleA as[RB];
    i32x4 sx[HZ ? RB : 1];  // W4 with zeros: sums of the rows' codes (every column alike)
  };
  // (one address per operand and compile-time steps from it: 16 rows on, a row's chunks are
  // swizzled alike)
  const unsigned asrc = (unsigned)(kg * G::A_BLK + a_off(wm * 16 * RB + j, g));
  const unsigned ssrc = (unsigned)(G::AS_OFF + (kg * BM + wm * 16 * RB + (WA ? j : 4 * g)) * 4);
  const unsigned wsrc = (unsigned)(G::B_OFF + kg * G::B_BLK + G::b_row(G::RG * g) + cb);
  const unsigned bsrc = (unsigned)((kg * BN + ccol) * 4);
  auto load_a = [&](const uint8_t* base, Aop& o) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      o.av[rb] = *(const i32x4*)(base + asrc + rb * 1024);
      o.as[rb] = *(const ScaleA*)(base + ssrc + rb * 64);
      if constexpr (W4) {
        // slots in the order of the nibble split: even K of the 16, then odd K
        const u32x4 x = bitcast<u32x4>(o.av[rb]);
        o.av[rb] = bitcast<i32x4>(u32x4{perm(x.y, x.x, 0x06040200u), perm(x.w, x.z, 0x06040200u),
                                        perm(x.y, x.x, 0x07050301u), perm(x.w, x.z, 0x07050301u)});
      }
      if constexpr (HZ)
        o.sx[rb] = mfma(bitcast<i32x4>(u32x4{0x01010101u, 0x01010101u, 0x01010101u, 0x01010101u}), o.av[rb]);
    }
  };
  auto load_w = [&](const uint8_t* base, int s, Wop& o) {
#pragma unroll
    for (int i = 0; i < G::RG; ++i) o.d[i] = *(const uint32_t*)(base + wsrc + s * 2 * G::B_BLK + i * BN);
  };
  // columns whose dots are computed before their folds (4 RB registers each), so that the
  // folds run back to back instead of each waiting on its MFMA
  constexpr int DOTS = NS == 1 ? (RB == 3 || RB == 4 ? 4 : RB == 2 ? 2 : 1) : (RB <= 2 ? 2 : 1);
  // folds one block of set s; W4 group scales and zeros come from the stage (`base`) here,
  // where they are used, and take no registers before
  auto fold = [&](int s, const uint8_t* base, const Aop& A, const Wop& B) {
    f32x4 bs[LC / 4];
    i32x4 zc[LC / 4];
    if constexpr (W4) {
#pragma unroll
      for (int r = 0; r < LC / 4; ++r) {
        bs[r] = *(const f32x4*)(base + G::BS_OFF + bsrc + (s * 2 * BN + 4 * r) * 4);
        if constexpr (HZ) zc[r] = *(const i32x4*)(base + G::BZ_OFF + bsrc + (s * 2 * BN + 4 * r) * 4);
      }
    }
    u32x4 bv[4];
    if constexpr (W4) {
      uint32_t lo[8], hi[8], e0[4], e1[4], o0[4], o1[4];
#pragma unroll
      for (int i = 0; i < 8; ++i) w4_split_i8x16(B.d[i], lo[i], hi[i]);
      tr4(lo[0], lo[1], lo[2], lo[3], e0);
      tr4(lo[4], lo[5], lo[6], lo[7], e1);
      tr4(hi[0], hi[1], hi[2], hi[3], o0);
      tr4(hi[4], hi[5], hi[6], hi[7], o1);
#pragma unroll
      for (int t = 0; t < 4; ++t) bv[t] = u32x4{e0[t], e1[t], o0[t], o1[t]};
    } else {
      uint32_t x0[4], x1[4], x2[4], x3[4];
      tr4(B.d[0], B.d[1], B.d[2], B.d[3], x0);
      tr4(B.d[4], B.d[5], B.d[6], B.d[7], x1);
      tr4(B.d[8], B.d[9], B.d[10], B.d[11], x2);
      tr4(B.d[12], B.d[13], B.d[14], B.d[15], x3);
#pragma unroll
      for (int t = 0; t < 4; ++t) bv[t] = u32x4{x0[t], x1[t], x2[t], x3[t]};
    }
#pragma unroll
    for (int t0 = 0; t0 < 4; t0 += DOTS) {
      i32x4 p[RB][DOTS];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int t = 0; t < DOTS; ++t)
          p[rb][t] = mfma(bitcast<i32x4>(bv[t0 + t]), A.av[rb]);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int t = 0; t < DOTS; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float c = acc[s][rb][t0 + t][r];
            float as;
            if constexpr (WA) as = A.as[rb];
            else as = A.as[rb][r];
            if constexpr (W4) {
              // The MFMA sums 16 * (nibble - 8) * a: the dot is p / 16, exactly.  Rather
              // than shifting every p, the fold takes float(p) (exact: |p| < 2^24) against
              // the scale product divided by 16 (exact): fma(float(p), fl(a_s * b_s) / 16,
              // acc) is fma(float(p / 16), fl(a_s * b_s), acc) bit for bit.
              int v = p[rb][t][r];
              if constexpr (HZ) v += zc[WA ? r : 0][t0 + t] * A.sx[rb][WA ? 0 : r];
              acc[s][rb][t0 + t][r] = fmaf((float)v, as * bs[WA ? r : 0][t0 + t], c);
            } else {
              acc[s][rb][t0 + t][r] = fmaf((float)p[rb][t][r], as, c);
            }
          }
    }
  };

  // ---------------- K loop: stage st holds blocks 2st and 2st+1 ----------------
  // Stage s is stored to LDS buffer s & 1 one iteration ahead (after the barrier that
  // ended the last read of that buffer) and computed in iteration s.  Its copy into
  // registers is issued three iterations ahead with one weight set (two register
  // sets, the loop written for even and odd st so their indices are static) and two
  // iterations ahead with two (one register set: the gate/up accumulators need the
  // registers).  The copy goes out right after the registers' LDS store, before the
  // barrier, so its issue overlaps the wait there (gate/up 47 us instead of 51 at
  // M = 512; issuing the store and copy before the MFMAs instead measured 49).
  // Every copy and LDS store is issued unconditionally: stages past the last one read
  // the last block again (fetch clamps the block index) and are stored to the buffer
  // no one reads any more.  A copy issued under a condition made the wait insertion
  // assume, at the join, that its registers were the most recent loads: it waited for
  // every copy in flight (vmcnt(0)) before each stage's LDS stores and again before
  // the next copy, so a stage waited a whole memory round trip.
  const int nst = (nk + 1) / 2;
  auto compute = [&](int st) {
    if (2 * st + kg >= nk) return;
    const uint8_t* base = lds + (st & 1) * G::STAGE;
    Aop A;
    load_a(base, A);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      Wop B;
      load_w(base, s, B);
      fold(s, base, A, B);
    }
  };
  if constexpr (NS == 1 && RB <= 4) {
    Regs rg0, rg1;
    fetch(rg0, 0);
    store(rg0, 0);
    fetch(rg1, 1);
    fetch(rg0, 2);
    __syncthreads();
    // next: the registers holding stage st+1, stored now and refilled with stage st+3
    auto iter = [&](int st, Regs& next) {
      compute(st);
      store(next, (st + 1) & 1);
      fetch(next, st + 3);
      __syncthreads();
    };
    int st = 0;
    for (; st + 1 < nst; st += 2) {
      iter(st, rg1);
      iter(st + 1, rg0);
    }
    if (st < nst) iter(st, rg1);
  } else {
    Regs rg;
    fetch(rg, 0);
    store(rg, 0);
    fetch(rg, 1);
    __syncthreads();
    for (int st = 0; st < nst; ++st) {
      compute(st);
      store(rg, (st + 1) & 1);
      fetch(rg, st + 2);
      __syncthreads();
    }
  }
  // W8 column scales of the epilogue: in flight during the sums below
  u32x4 csraw[NS][LC / 4];
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int r = 0; r < LC / 4; ++r)
      csraw[s][r] = W4 ? u32x4{0u, 0u, 0u, 0u} : ld_scale4_raw(sset[s], a.sdt, ncol0 + ccol + 4 * r);

  // ---------------- K groups: group 0 + group 1 (fixed order), one set at a time ----------------
  // Each group finishes half of the 16-row blocks: it takes the other's sums of them (the two
  // are added either way round to the same bits) and runs their epilogue, so no wave sits out
  // the epilogue's divisions and exponentials.
  constexpr int WT = 2 * WNW;  // wave tiles (wm, wn) of one K group
  constexpr int RH = (RB + 1) / 2;
  auto mine = [&](int rb) { return (rb < RH) == (kg == 0); };
  const int wt = wave % WT;
  float* red = (float*)lds + wt * (16 * RB * 64) + lane;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    if (s > 0) __syncthreads();  // the previous set has been read
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      if (mine(rb)) continue;  // uniform over a wave
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[((rb * 4 + t) * 4 + r) * 64] = acc[s][rb][t][r];
    }
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      if (!mine(rb)) continue;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[s][rb][t][r] += red[((rb * 4 + t) * 4 + r) * 64];
    }
  }
  if (S > 1) {
    // Split-K: the partial tile of each weight set (wave tile w: the float4 (rb, t) of
    // every lane at byte ((rb * 4 + t) * 64 + lane) * 16 of its slot, slots
    // [split][set][wave]) goes out through device-coherent stores; each workgroup's
    // stores complete before it counts its arrival, and the last to arrive sums the
    // partials in split order.
    __shared__ int s_last;
    constexpr unsigned kSlot = 16u * RB * 64u * 4u;
    const __amdgpu_buffer_rsrc_t rs =
        part_rsrc(a.part + (long long)tile * S * NS * WT * (16 * RB * 64), (unsigned)(S * NS * WT) * kSlot);
    const unsigned lane_off = (unsigned)lane * 16u;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const unsigned base = (unsigned)((split * NS + s) * WT + wt) * kSlot + lane_off;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        if (!mine(rb)) continue;
#pragma unroll
        for (int t = 0; t < 4; ++t) st_coherent(acc[s][rb][t], rs, base + (unsigned)(rb * 4 + t) * 1024u);
      }
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);  // every partial store of this wave has completed
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (tid == 0) {
      const unsigned prev = __hip_atomic_fetch_add(a.cnt + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int last = prev == (unsigned)(S - 1);
      if (last) __hip_atomic_store(a.cnt + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_last = last;
    }
    __syncthreads();
    if (!s_last) return;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    for (int sp = 0; sp < S; ++sp) {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const unsigned base = (unsigned)((sp * NS + s) * WT + wt) * kSlot + lane_off;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          if (!mine(rb)) continue;
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const f32x4 v = ld_coherent(rs, base + (unsigned)(rb * 4 + t) * 1024u);
            acc[s][rb][t] = (sp == 0) ? v : acc[s][rb][t] + v;
          }
        }
      }
    }
  }

  // ---------------- epilogue ----------------
  // Value (i, c) of a lane's block of 16 rows: its row i (of LR) and column c (of LC).
  const int col = ncol0 + ccol;  // its first column within the matrix
  auto val = [&](int s, int rb, int i, int c) { return WA ? acc[s][rb][c & 3][c >> 2] : acc[s][rb][c & 3][i]; };
  float cs[NS][LC];
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int r = 0; r < LC / 4; ++r) {
      if constexpr (W4) cs[s][4 * r] = cs[s][4 * r + 1] = cs[s][4 * r + 2] = cs[s][4 * r + 3] = 1.0f;
      else cvt_scale4(csraw[s][r], a.sdt, &cs[s][4 * r]);
    }
  const int r0 = m0 + wm * 16 * RB + (WA ? j : 4 * g);
  constexpr int VC = LC < 8 ? LC : 8;  // 16-bit values of a store
  using V16 = std::conditional_t<VC == 8, u32x4, u32x2>;
  if constexpr (EPI == EPI_STORE) {
    // column scale (W8), residual, 16-bit store.  The output type and the residual
    // are uniform: branch once, outside the per-value code.
    const int ocol = sg.col0 + col;
    auto store_all = [&](auto bf16, auto with_res) {
      constexpr bool BF = decltype(bf16)::value, RES = decltype(with_res)::value;
      auto cvt2 = [](float v0, float v1) -> uint32_t {
        if constexpr (BF) return (uint32_t)f32_to_bf16(v0) | ((uint32_t)f32_to_bf16(v1) << 16);
        else return bitcast<uint32_t>(__builtin_convertvector((float __attribute__((ext_vector_type(2)))){v0, v1}, f16x2));
      };
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int i = 0; i < LR; ++i) {
          const int row = r0 + rb * 16 + i;
          if (!mine(rb) || row >= M) continue;
          uint16_t* const o = (uint16_t*)a.out + (long long)row * a.ldo + ocol;
#pragma unroll
          for (int h = 0; h < LC / VC; ++h) {
            // column scale and residual in one rounding (fmaf), the product alone
            // without a residual: the skinny kernel's epilogue rounds the same way
            V16 rv = V16(0u), ov;
            if constexpr (RES) rv = *(const V16*)((const uint16_t*)a.res + (long long)row * a.ldr + ocol + VC * h);
            float y[VC];
#pragma unroll
            for (int c = 0; c < VC; ++c) {
              const float v = val(0, rb, i, VC * h + c), k = cs[0][VC * h + c];
              if constexpr (RES) {
                const uint16_t hh = (uint16_t)(rv[c >> 1] >> (16 * (c & 1)));
                y[c] = fmaf(v, k, BF ? bf16_to_f32(hh) : (float)bitcast<_Float16>(hh));
              } else {
                y[c] = v * k;
              }
            }
#pragma unroll
            for (int c = 0; c < VC / 2; ++c) ov[c] = cvt2(y[2 * c], y[2 * c + 1]);
            *(V16*)(o + VC * h) = ov;
          }
        }
    };
    using T = std::true_type;
    using F = std::false_type;
    if (a.odt == DT_BF16) {
      if (a.res) store_all(T{}, T{});
      else store_all(T{}, F{});
    } else {
      if (a.res) store_all(F{}, T{});
      else store_all(F{}, F{});
    }
  } else {
    // h = silu(g) * u; bf16 store, or bf16 round trip and per-64-column int8 quant.
    // A row's 64 columns of this wave tile are the four lanes g of its j (WA) or the
    // sixteen lanes j of its g: the amax reduces over those lanes.
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      if (!mine(rb)) continue;
#pragma unroll
      for (int i = 0; i < LR; ++i) {
        const int row = r0 + rb * 16 + i;
        float h[LC];
#pragma unroll
        for (int c = 0; c < LC; ++c) h[c] = silu(val(0, rb, i, c) * cs[0][c]) * (val(1, rb, i, c) * cs[1][c]);
        if constexpr (EPI == EPI_GATEUP) {
          if (row < M) {
            uint16_t* const d = (uint16_t*)a.out + (long long)row * a.ncols + col;
#pragma unroll
            for (int v = 0; v < LC / VC; ++v) {
              V16 o;
#pragma unroll
              for (int c = 0; c < VC / 2; ++c)
                o[c] = (uint32_t)f32_to_bf16(h[VC * v + 2 * c]) | ((uint32_t)f32_to_bf16(h[VC * v + 2 * c + 1]) << 16);
              *(V16*)(d + VC * v) = o;
            }
          }
        } else {
          float am = 0.0f;
#pragma unroll
          for (int c = 0; c < LC; ++c) {
            h[c] = bf16_to_f32(f32_to_bf16(h[c]));  // bf16 round trip (kernels/gemm.py:198-200)
            am = fmaxf(am, fabsf(h[c]));
          }
          if constexpr (WA) {
            float am0, am1;
            lane_pair<16>(am, am0, am1);
            lane_pair<32>(fmaxf(am0, am1), am0, am1);
            am = fmaxf(am0, am1);
          } else {
            am = fmaxf(am, lane_xor<1>(am));
            am = fmaxf(am, lane_xor<2>(am));
            am = fmaxf(am, lane_xor<4>(am));
            am = fmaxf(am, lane_xor<8>(am));
          }
          const float sc = fmaxf(am / 127.0f, 1e-8f);
          const float inv = 1.0f / sc;
          if (row < M) {
            uint32_t qw[LC / 4];
#pragma unroll
            for (int q = 0; q < LC / 4; ++q) {
              qw[q] = 0;
#pragma unroll
              for (int t = 0; t < 4; ++t) qw[q] |= ((uint32_t)(quant_i8(h[4 * q + t], sc, inv) & 0xFF)) << (8 * t);
            }
            int8_t* const d = a.oq + (long long)row * a.ncols + col;
            if constexpr (WA) *(u32x4*)d = u32x4{qw[0], qw[1], qw[2], qw[3]};
            else *(uint32_t*)d = qw[0];
            if (WA ? g == 0 : j == 0) a.os[(long long)row * (a.ncols / 64) + col / 64] = sc;
          }
        }
      }
    }
  }
}

template <int WK, bool HZ, int EPI, int RB, int WNW>
static hipError_t launch_i8_t(const SkArgs& a, int tiles, hipStream_t st) {
  using G = Gi8<WK, (EPI == EPI_STORE) ? 1 : 2, RB, WNW>;
  static bool attr_set = false;  // benign race: every caller sets the same value
  if (!attr_set) {
    const hipError_t e = hipFuncSetAttribute((const void*)prefill_i8_kernel<WK, HZ, EPI, RB, WNW>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  hipLaunchKernelGGL((prefill_i8_kernel<WK, HZ, EPI, RB, WNW>), dim3(tiles), dim3(G::THREADS), (size_t)G::LDS, st, a);
  return hipGetLastError();
}

template <int WK, bool HZ, int EPI>
static hipError_t launch_i8_e(const SkArgs& a, int tile, int tiles, hipStream_t st) {
  switch (tile) {
    case I8_128x128: return launch_i8_t<WK, HZ, EPI, 4, 2>(a, tiles, st);
    case I8_64x64: return launch_i8_t<WK, HZ, EPI, 2, 1>(a, tiles, st);
    case I8_96x64: return launch_i8_t<WK, HZ, EPI, 3, 1>(a, tiles, st);
    default: break;
  }
  if constexpr (EPI == EPI_STORE) {  // (two weight sets' accumulators would spill)
    if (tile == I8_128x64) return launch_i8_t<WK, HZ, EPI, 4, 1>(a, tiles, st);
    if (tile == I8_160x64) return launch_i8_t<WK, HZ, EPI, 5, 1>(a, tiles, st);
  }
  return hipErrorInvalidValue;
}

template <int WK, bool HZ>
hipError_t launch_i8_w(const SkArgs& a, int epi, int tile, int tiles, hipStream_t st) {
  switch (epi) {
    case EPI_STORE: return launch_i8_e<WK, HZ, EPI_STORE>(a, tile, tiles, st);
    case EPI_GATEUP: return launch_i8_e<WK, HZ, EPI_GATEUP>(a, tile, tiles, st);
    default: return launch_i8_e<WK, HZ, EPI_GATEUP_Q>(a, tile, tiles, st);
  }
}

// the weight kinds, one source file each
extern template hipError_t launch_i8_w<WK_W8, false>(const SkArgs&, int, int, int, hipStream_t);
extern template hipError_t launch_i8_w<WK_W4, false>(const SkArgs&, int, int, int, hipStream_t);
extern template hipError_t launch_i8_w<WK_W4, true>(const SkArgs&, int, int, int, hipStream_t);

}  // namespace qlin
