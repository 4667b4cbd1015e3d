// GEMM for fp16 activations with few rows (17 to a few hundred), gfx950: tiles of 32 or 64
// rows x 64 columns whose K is split over the four waves of a workgroup, and over
// workgroups where the tiles leave CUs idle.
//
// out[M,N] = x[M,K] . dequant(W)[K,N] (+ residual), W in the engine layouts (int8 [K,N] with
// per-column scales, or packed nibbles [K/2,N] with per-group scales and optional zeros).
// Between the decode plans (16-row tiles, each re-reading the weights) and the large prefill
// tiles (few workgroups, long serial K loops and a large split-K exchange), a short prompt
// is bound by latency: how long the longest chain of loads, MFMAs and partial sums is.
//
//   * Wave u of the 4 S waves of a tile (S workgroups) takes a contiguous run of the 32-wide
//     K steps.  A wave copies its own activations and weights (16-byte LDS DMA into a ring of
//     three steps of its own) and waits for its own copies, so the K loop has no barrier.
//   * LDS: activation rows of 64 bytes with 16-byte chunk c at c ^ ((r >> 2) & 3); the i-th
//     weight row of lane group g (of its 8 int8 or 4 packed rows) at slot 4 i + g, so a wave's
//     read of its i-th rows is 256 contiguous bytes: both free of bank conflicts.
//   * 16 RB x 64 outputs per wave, v_mfma_f32_16x16x32_f16 on exactly converted weights (int8,
//     or nibble - z).  W8 column scales multiply the fp32 result; W4 group scales multiply the
//     group's fp32 dot where the wave's run leaves the group.
//   * The four waves' sums are added through LDS in wave order, each wave finishing a quarter
//     of the tile; with S > 1 the quarters are stored (device-coherent) and the last workgroup
//     to arrive adds the splits in order, every wave a quarter, all its loads in flight.
//     No workgroup waits for another.
//
// The K order depends on K, S and nothing else, so rows do not depend on their tile.
//
// Measured (weights from HBM), against the faster of the 16-row and large tiles: W8 M = 128
// 2048x2048 8.1 us (13.6), 6144x2048 13.9 (22.2), 4096x4096 14.5 (19.1); M = 32 12288x4096
// 16.9 (27.7); W4-g128 M = 128 6144x2048 13.3 (21.5); M = 32 4096x4096 9.9 (15.7).
#include "prefill_kernel.h"

namespace qlin {

namespace {

template <int WK, int RB>
struct KgGeo {
  static constexpr int BM = 16 * RB;
  static constexpr int A_BYTES = BM * 64;                        // one 32-wide step of the rows
  static constexpr int B_BYTES = (WK == WK_W8) ? 32 * 64 : 16 * 64;
  static constexpr int SC_BYTES = (WK == WK_W8) ? 0 : 1024;      // W4 scales and zeros (one copy)
  static constexpr int STEP = A_BYTES + B_BYTES + SC_BYTES;
  static constexpr int DMA = RB + 2;                             // copies per step
  static constexpr int RED = 4 * RB * 4 * 1024;                  // the four waves' sums
  static constexpr int LDS = (12 * STEP > RED) ? 12 * STEP : RED;
};

template <int WK, bool HZ, int RB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void prefill_kg_kernel(const TlArgs a) {
  using G = KgGeo<WK, RB>;
  constexpr bool W4 = WK == WK_W4;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ int s_last;
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = (int)rfl((uint32_t)tid >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int M = a.M, N = a.N, S = a.splits;
  // XCD x's workgroups (b = x, x + 8, ...) take one contiguous run of the order: a tile's
  // splits, then the row tiles of a column tile (the same weights), then the next columns
  const int b = (int)blockIdx.x, W = (int)gridDim.x;
  const int v = (b & 7) * (W >> 3) + min(b & 7, W & 7) + (b >> 3);
  const int tile = v / S, split = v - tile * S;
  const int tiles_m = (M + G::BM - 1) / G::BM;
  const int tn = tile / tiles_m, tm = tile - tn * tiles_m;
  const int m0 = tm * G::BM, n0 = tn * 64;
  // this wave's run of 32-wide steps
  const int T = a.K >> 5, u = split * 4 + wave;
  const int s0 = (int)((long long)T * u / (4 * S)), s1 = (int)((long long)T * (u + 1) / (4 * S));

  uint32_t offA[RB];
#pragma unroll
  for (int q = 0; q < RB; ++q) {
    const int r = 16 * q + (lane >> 2), c = (lane & 3) ^ ((r >> 2) & 3);
    offA[q] = (uint32_t)(((long long)min(m0 + r, M - 1) * a.ldx + 8 * c) * 2);  // rows past M are never stored
  }
  int col = n0 + 16 * (lane & 3);
  col = col < N ? col : n0;  // chunks past N (N % 16 == 0) re-read a valid one
  uint32_t offB[W4 ? 1 : 2];
#pragma unroll
  for (int q = 0; q < (W4 ? 1 : 2); ++q) {
    const int slot = 16 * q + (lane >> 2);
    offB[q] = (uint32_t)(((W4 ? 4 : 8) * (slot & 3) + (slot >> 2)) * N + col);
  }
  // W4: lanes 0 .. 4 ssz - 1 copy the step's 64 scales, 16 .. 19 its zeros, 16 bytes each;
  // the others (and columns past N) re-read the tile's first
  const int ssz = a.sdt == DT_F32 ? 4 : 2;
  const bool zlane = HZ && (lane >> 2) == 4;
  uint32_t offS = 0;
  if constexpr (W4) {
    if (lane < 4 * ssz && n0 + 16 * lane / ssz < N) offS = 16u * (uint32_t)lane;
    if (zlane && n0 + 16 * (lane & 3) < N) offS = 16u * (uint32_t)(lane & 3);
  }
  const bool pow2 = (a.group & (a.group - 1)) == 0;
  const int gsh = __builtin_ctz((unsigned)a.group);
  auto group_of = [&](int s) { return pow2 ? (32 * s) >> gsh : 32 * s / a.group; };

  const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds + (uint32_t)(wave * 3 * G::STEP);
  auto issue = [&](int step, uint32_t at) {  // `at`: byte offset of the step's buffer in the ring
    const int s = min(step, T - 1);          // (steps past the run are read and never used)
    const uint32_t base = rfl(ring + at);
    const void* xa = rfl_ptr(a.x + 32LL * s);
#pragma unroll
    for (int q = 0; q < RB; ++q) dma_s(xa, offA[q], rfl(base + 1024u * q));
    const void* wb = rfl_ptr(a.w + (long long)s * (W4 ? 16 : 32) * N);
#pragma unroll
    for (int q = 0; q < (W4 ? 1 : 2); ++q) dma_s(wb, offB[q], rfl(base + (uint32_t)G::A_BYTES + 1024u * q));
    if constexpr (W4) {
      const long long row = (long long)group_of(s) * N + n0;
      const uint8_t* ps = (const uint8_t*)a.s + row * ssz;
      if constexpr (HZ) ps = zlane ? a.z + row : ps;
      dma_v(ps + offS, rfl(base + (uint32_t)(G::A_BYTES + G::B_BYTES)));
    }
  };

  f32x4 acc[RB][4];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[rb][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 p[W4 ? RB : 1][4];  // W4: the current group's dot
  if constexpr (W4) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int t = 0; t < 4; ++t) p[rb][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  auto step_mma = [&](uint32_t at, bool leave) {  // leave: the run's next step is in another group
    const uint8_t* sA = lds + wave * 3 * G::STEP + at;
    const uint8_t* sB = sA + G::A_BYTES;
    f16x8 av[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const int r = 16 * rb + j;
      av[rb] = *(const f16x8*)(sA + r * 64 + 16 * (g ^ ((r >> 2) & 3)));
    }
    uint32_t d[W4 ? 4 : 8];
#pragma unroll
    for (int i = 0; i < (W4 ? 4 : 8); ++i) d[i] = *(const uint32_t*)(sB + (4 * i + g) * 64 + 4 * j);
    if constexpr (!W4) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const u32x4 h = u32x4{w8_pair_f16(d[0], d[1], t), w8_pair_f16(d[2], d[3], t), w8_pair_f16(d[4], d[5], t),
                              w8_pair_f16(d[6], d[7], t)};
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) acc[rb][t] = mfma_f16(av[rb], bitcast<f16x8>(h), acc[rb][t]);
      }
    } else {
      const uint8_t* sS = sB + G::B_BYTES;
      uint32_t zv = 0x08080808u;
      if constexpr (HZ) zv = *(const uint32_t*)(sS + 256 + 4 * j);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const f16x2 bias = w4_bias((zv >> (8 * t)) & 0xFFu);
        const u32x4 h = u32x4{w4_pair_f16(d[0], t, bias), w4_pair_f16(d[1], t, bias), w4_pair_f16(d[2], t, bias),
                              w4_pair_f16(d[3], t, bias)};
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) p[rb][t] = mfma_f16(av[rb], bitcast<f16x8>(h), p[rb][t]);
      }
      if (leave) {  // uniform
        u32x4 raw;
        if (ssz == 4) {
          raw = *(const u32x4*)(sS + 16 * j);
        } else {
          const u32x2 r2 = *(const u32x2*)(sS + 8 * j);
          raw = u32x4{r2.x, r2.y, 0u, 0u};
        }
        float sc[4];
        cvt_scale4(raw, a.sdt, sc);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[rb][t][r] = fmaf(p[rb][t][r], sc[t], acc[rb][t][r]);
            p[rb][t] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
      }
    }
  };

  issue(s0, 0);
  issue(s0 + 1, G::STEP);
  uint32_t at = 0;
  for (int s = s0; s < s1; ++s) {
    __builtin_amdgcn_sched_barrier(0);
    // step s copied (s + 1 may be in flight), and the reads of step s - 1 have returned
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(G::DMA));
    const uint32_t next = at >= G::STEP ? at - G::STEP : at + 2 * G::STEP;
    issue(s + 2, next);
    __builtin_amdgcn_sched_barrier(0);
    step_mma(at, W4 && (s + 1 == s1 || group_of(s + 1) != group_of(s)));
    at = at == 2 * G::STEP ? 0 : at + G::STEP;
  }
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));  // no copy may land after the ring is reused

  // the four waves' sums, in wave order: wave w finishes the (rb, t) slots RB w .. RB w + RB - 1
  __syncthreads();
  f32x4* red = (f32x4*)lds;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int t = 0; t < 4; ++t) red[(wave * RB * 4 + rb * 4 + t) * 64 + lane] = acc[rb][t];
  __syncthreads();
  f32x4 y[RB];
#pragma unroll
  for (int k = 0; k < RB; ++k) {
    y[k] = red[(wave * RB + k) * 64 + lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) y[k] = y[k] + red[(w * RB * 4 + wave * RB + k) * 64 + lane];
  }
  if (S > 1) {
    constexpr unsigned kPart = RB * 4 * 1024;  // bytes of a workgroup's partial tile
    const __amdgpu_buffer_rsrc_t rs = part_rsrc(a.part + (long long)tile * S * (kPart / 4), (unsigned)S * kPart);
    const unsigned off = (unsigned)(wave * RB * 64 + lane) * 16u;
#pragma unroll
    for (int k = 0; k < RB; ++k) st_coherent(y[k], rs, (unsigned)split * kPart + off + 1024u * k);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);  // this wave's partial stores have completed
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (tid == 0) {
      const unsigned prev = __hip_atomic_fetch_add(a.cnt + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_last = prev == (unsigned)(S - 1);
      if (s_last) __hip_atomic_store(a.cnt + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!s_last) return;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    for (int sp = 0; sp < S; ++sp) {
#pragma unroll
      for (int k = 0; k < RB; ++k) {
        const f32x4 q = ld_coherent(rs, (unsigned)sp * kPart + off + 1024u * k);
        y[k] = sp == 0 ? q : y[k] + q;
      }
    }
  }

  // epilogue: RB = 4: rows 16 wave + 4g + r, columns 4j .. 4j + 3; RB = 2: rows 16 (wave / 2)
  // + 4g + r, columns 4j + 2 (wave % 2) and the next
  const int rb = (wave * RB) >> 2, t0 = (wave * RB) & 3;
  const int colb = n0 + 4 * j + t0;
  if (colb >= N) return;
  float cs[4] = {1.f, 1.f, 1.f, 1.f};
  if constexpr (!W4) {
    float c4[4];
    cvt_scale4(ld_scale4_raw(a.s, a.sdt, n0 + 4 * j), a.sdt, c4);
#pragma unroll
    for (int k = 0; k < RB; ++k) cs[k] = RB == 4 ? c4[k] : (t0 ? c4[2 + k] : c4[k]);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = m0 + 16 * rb + 4 * g + r;
    if (row >= M) break;
    uint32_t o[RB / 2], rw[RB / 2];
    if (a.res) {
      const uint16_t* rp = (const uint16_t*)a.res + (long long)row * a.ldr + colb;
      if constexpr (RB == 4) {
        const u32x2 q = *(const u32x2*)rp;
        rw[0] = q.x, rw[1] = q.y;
      } else {
        rw[0] = *(const uint32_t*)rp;
      }
    }
#pragma unroll
    for (int k = 0; k < RB; k += 2) {
      float e0, e1;
      if (a.res) {  // (one rounding, spelled out: both tile heights give the same bits)
        const uint16_t h0 = (uint16_t)rw[k / 2], h1 = (uint16_t)(rw[k / 2] >> 16);
        e0 = fmaf(y[k][r], cs[k], a.odt == DT_BF16 ? bf16_to_f32(h0) : (float)bitcast<_Float16>(h0));
        e1 = fmaf(y[k + 1][r], cs[k + 1], a.odt == DT_BF16 ? bf16_to_f32(h1) : (float)bitcast<_Float16>(h1));
      } else {
        e0 = y[k][r] * cs[k];
        e1 = y[k + 1][r] * cs[k + 1];
      }
      o[k / 2] = (uint32_t)to_out16(e0, a.odt) | ((uint32_t)to_out16(e1, a.odt) << 16);
    }
    uint16_t* op = (uint16_t*)a.out + (long long)row * a.ldo + colb;
    if constexpr (RB == 4) *(u32x2*)op = u32x2{o[0], o[1]};
    else *(uint32_t*)op = o[0];
  }
}

template <int WK, bool HZ, int RB>
hipError_t launch_kg(const TlArgs& a, hipStream_t st) {
  using G = KgGeo<WK, RB>;
  const long long tiles = (long long)((a.M + G::BM - 1) / G::BM) * ((a.N + 63) / 64);
  static bool attr_set = false;  // benign race: every caller sets the same value
  if (!attr_set) {
    const hipError_t e = hipFuncSetAttribute((const void*)prefill_kg_kernel<WK, HZ, RB>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  hipLaunchKernelGGL((prefill_kg_kernel<WK, HZ, RB>), dim3((unsigned)(tiles * a.splits)), dim3(256), (size_t)G::LDS, st, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_prefill_kg(const TlArgs& a, int wk, bool hz, int bm, hipStream_t st) {
  if (bm == 32) {
    if (wk == WK_W8) return launch_kg<WK_W8, false, 2>(a, st);
    return hz ? launch_kg<WK_W4, true, 2>(a, st) : launch_kg<WK_W4, false, 2>(a, st);
  }
  if (wk == WK_W8) return launch_kg<WK_W8, false, 4>(a, st);
  return hz ? launch_kg<WK_W4, true, 4>(a, st) : launch_kg<WK_W4, false, 4>(a, st);
}

}  // namespace qlin
