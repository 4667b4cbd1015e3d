// Layout kernels.  W4 unpack and W4 / W8 dequantization to fp32 expose the exact
// integer / fp32 values the GEMM kernels consume, so the unpack and dequant can be
// checked bit for bit (quant_formats.py:6-9, kernels/w4.py:51-61, 103-104).  The
// load-time producers of the packed layouts, symmetric W4 per (group, column) and
// W8 per column (quant_formats.py:253-275), requantize fp32 weights on the GPU with
// the same arithmetic: fp32 amax, clamp at 1e-8, one correctly rounded division for
// the scale and one per weight, round half to even.
#include "qlin_dev.h"
#include "qlin_internal.h"

namespace qlin {

// nib[k][n] = nibble k of column n: byte (k/2, n), low nibble for even k.
__global__ void w4_unpack_kernel(const uint8_t* __restrict__ p, int K, int N, uint8_t* __restrict__ out) {
  const long long total = (long long)(K / 2) * N;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const long long jrow = i / N, col = i - jrow * N;
    const uint8_t b = p[i];
    out[(2 * jrow) * N + col] = b & 0x0F;
    out[(2 * jrow + 1) * N + col] = b >> 4;
  }
}

// out[k][n] = (nibble - z) * scale[k/group][n] in fp32; z = 8 when zeros are absent.
__global__ void w4_dequant_kernel(const uint8_t* __restrict__ p, const void* s, int sdt,
                                  const uint8_t* __restrict__ z, int group, int K, int N,
                                  float* __restrict__ out) {
  const long long total = (long long)(K / 2) * N;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const long long jrow = i / N, col = i - jrow * N;
    const uint8_t b = p[i];
    const long long k0 = 2 * jrow;
    const long long g0 = (k0 / group) * N + col, g1 = ((k0 + 1) / group) * N + col;
    const int z0 = z ? (int)z[g0] : 8, z1 = z ? (int)z[g1] : 8;
    out[k0 * N + col] = (float)((int)(b & 0x0F) - z0) * load_scale(s, sdt, g0);
    out[(k0 + 1) * N + col] = (float)((int)(b >> 4) - z1) * load_scale(s, sdt, g1);
  }
}

// out[k][n] = w[k][n] * scale[n] in fp32.
__global__ void w8_dequant_kernel(const int8_t* __restrict__ w, const void* s, int sdt, int K, int N,
                                  float* __restrict__ out) {
  const long long total = (long long)K * N;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const long long col = i % N;
    out[i] = (float)w[i] * load_scale(s, sdt, col);
  }
}

// ---------------------------------------------------------------------------
// Requantization (quant_formats.py:253-275).  Byte and fp32 element work, bound
// by HBM: a thread keeps its weights in registers between the amax and the codes, so a
// weight is read once (columns too long for that are read again from the caches).
// ---------------------------------------------------------------------------

// rint(w / sc) with the correctly rounded quotient's value, from a product with
// inv = fl(1 / sc): the product is within 2^-22 of the quotient relative, 3e-5 for
// quotients up to 128, so only a product within 1e-4 of a rounding tie needs the division
// (a division is about twelve instructions; with one per weight these kernels were bound
// by them, not by HBM).  Infinities and NaN take either form to the same value.
__device__ __forceinline__ float rint_div(float w, float sc, float inv) {
  const float t = w * inv;
  float r = rintf(t);
  if (__builtin_expect(fabsf(t - r) > 0.4999f, 0)) r = rintf(w / sc);
  return r;
}

// W4, C columns per thread (N % C == 0), the group's GROUP rows held in registers (C *
// GROUP = 128 of them): every weight is read once, all of a thread's loads in flight
// together.  K = 4096, N = 12288, groups of 32 / 64: 42 / 41.5 us (5.4 TB/s), 72 / 79 us
// with a second read of the rows and a division per weight.
template <int GROUP, int C>
__global__ __launch_bounds__(256) void requant_w4_kernel_reg(const float* __restrict__ w, int N,
                                                             uint8_t* __restrict__ packed,
                                                             uint16_t* __restrict__ sbf) {
  typedef float vec __attribute__((ext_vector_type(C)));
  const int n = C * (blockIdx.x * blockDim.x + threadIdx.x);
  const int gi = blockIdx.y;
  if (n >= N) return;
  const float* col = w + (long long)gi * GROUP * N;
  vec v[GROUP];
#pragma unroll
  for (int r = 0; r < GROUP; ++r)
    v[r] = __builtin_nontemporal_load((const vec*)(col + (long long)r * N + (uint32_t)n));
  float sc[C], inv[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    float amax = 0.0f;
#pragma unroll
    for (int r = 0; r < GROUP; ++r) amax = fmaxf(amax, fabsf(v[r][c]));
    sc[c] = fmaxf(amax, 1e-8f) / 7.0f;
    inv[c] = 1.0f / sc[c];
  }
  auto code = [&](float x, int c) {
    return (uint32_t)(int)(fminf(fmaxf(rint_div(x, sc[c], inv[c]), -8.0f), 7.0f) + 8.0f);
  };
  uint8_t* prow = packed + (long long)gi * (GROUP / 2) * N;
#pragma unroll
  for (int r = 0; r < GROUP; r += 2) {
    uint32_t word = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) word |= (code(v[r][c], c) | (code(v[r + 1][c], c) << 4)) << (8 * c);
    uint8_t* d = prow + (long long)(r / 2) * N + (uint32_t)n;
    if constexpr (C == 4) *(uint32_t*)d = word;
    else *(uint16_t*)d = (uint16_t)word;
  }
  uint32_t sw[2] = {0u, 0u};
#pragma unroll
  for (int c = 0; c < C; ++c) sw[c >> 1] |= (uint32_t)f32_to_bf16(sc[c]) << (16 * (c & 1));
  uint16_t* sd = sbf + (long long)gi * N + (uint32_t)n;
  if constexpr (C == 4) *(u32x2*)sd = u32x2{sw[0], sw[1]};
  else *(uint32_t*)sd = sw[0];
}

// W4: thread = (group g, column n).  sc = max(amax, 1e-8) / 7 over the group's rows;
// code = clamp(rint(w / sc), -8, 7) + 8; even K in the low nibble (quant_formats.py:
// 223-229, 246-250); the scale is stored as bf16 (round to nearest even).
__global__ void requant_w4_kernel(const float* __restrict__ w, int K, int N, int group,
                                  uint8_t* __restrict__ packed, uint16_t* __restrict__ sbf) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  const int gi = blockIdx.y;
  if (n >= N) return;
  const float* col = w + (long long)gi * group * N + n;
  float amax = 0.0f;
  for (int r = 0; r < group; ++r) amax = fmaxf(amax, fabsf(col[(long long)r * N]));
  const float sc = fmaxf(amax, 1e-8f) / 7.0f;
  uint8_t* prow = packed + (long long)gi * (group / 2) * N + n;
  for (int r = 0; r < group; r += 2) {
    const float q0 = fminf(fmaxf(rintf(col[(long long)r * N] / sc), -8.0f), 7.0f) + 8.0f;
    const float q1 = fminf(fmaxf(rintf(col[(long long)(r + 1) * N] / sc), -8.0f), 7.0f) + 8.0f;
    prow[(long long)(r / 2) * N] = (uint8_t)((int)q0 | ((int)q1 << 4));
  }
  sbf[(long long)gi * N + n] = f32_to_bf16(sc);
}

// W8 in one launch (N % 4 == 0): a workgroup of 1024 threads owns a strip of 4 L columns.
// Thread (q = tid / L) holds 4 columns of rows q, q + 1024 / L, ... in registers (NIT of
// them; the rows past those are read again from the caches for the second half), the
// columns' amax meets in LDS, and the codes are written from the registers: 512 rows of the
// wide form <8, 16>, 1024 / 2048 / 4096 of <4, 4> / <8, 4> / <16, 4>, whose last 12 spill.
// Bound by HBM and the second read of the other rows (7/8 of 4096 in the wide form, about
// 1 MB a strip), and by a workgroup's read and write phases not overlapping (its registers
// hold one workgroup per CU).  K = 4096, N = 12288: 76 us, 4096 x 4096: 25 us, 2048 x 2048: 9.0 us,
// against 110 / 48.5 / 30 us in four launches (amax by atomics, codes with a division
// each, scale).
template <int NIT, int L>
__global__ __launch_bounds__(1024) void requant_w8_strip_kernel(const float* __restrict__ w, int K, int N, int strips,
                                                                int8_t* __restrict__ q, float* __restrict__ scale) {
  constexpr int RS = 1024 / L;  // rows per step
  __shared__ float part[16][4 * L];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // strips narrower than a cache line: neighbours on one XCD (workgroup b runs on XCD b mod 8)
  const int xcd = (int)blockIdx.x & 7, per8 = strips >> 3, more = strips & 7;
  const int strip = L < 8 ? xcd * per8 + min(xcd, more) + ((int)blockIdx.x >> 3) : (int)blockIdx.x;
  const int c4 = 4 * (tid & (L - 1)), n = 4 * L * strip + c4, r0 = tid / L;
  const bool valid = n < N;
  const uint32_t nn = valid ? (uint32_t)n : 0u;
  f32x4 v[NIT];
  f32x4 am = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NIT; ++i) {
    // (a row read twice leaves the amax as it is; a uniform address and a 32-bit offset)
    const int k0 = RS * i < K ? RS * i : 0;
    v[i] = *(const f32x4*)(w + (long long)k0 * N + ((uint32_t)min(r0, K - 1 - k0) * (uint32_t)N + nn));
  }
#pragma unroll 4
  for (int r = r0 + RS * NIT; r < K; r += RS) {
    const f32x4 x = *(const f32x4*)(w + (long long)r * N + nn);
#pragma unroll
    for (int c = 0; c < 4; ++c) am[c] = fmaxf(am[c], fabsf(x[c]));
  }
#pragma unroll
  for (int i = 0; i < NIT; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) am[c] = fmaxf(am[c], fabsf(v[i][c]));
#pragma unroll
  for (int s = L; s < 64; s <<= 1)
#pragma unroll
    for (int c = 0; c < 4; ++c) am[c] = fmaxf(am[c], __shfl_xor(am[c], s));
  if (lane < L) *(f32x4*)&part[wave][c4] = am;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const f32x4 x = *(const f32x4*)&part[i][c4];
#pragma unroll
    for (int c = 0; c < 4; ++c) am[c] = fmaxf(am[c], x[c]);
  }
  if (!valid) return;
  f32x4 sc, inv;
#pragma unroll
  for (int c = 0; c < 4; ++c) sc[c] = fmaxf(am[c], 1e-8f) / 127.0f, inv[c] = 1.0f / sc[c];
  if (tid < L) *(f32x4*)(scale + n) = sc;
  auto put = [&](int k0, const f32x4& x) {  // row k0 + r0
    uint32_t word = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      word |= ((uint32_t)(int)fminf(fmaxf(rint_div(x[c], sc[c], inv[c]), -127.0f), 127.0f) & 0xFFu) << (8 * c);
    *(uint32_t*)(q + (long long)k0 * N + ((uint32_t)r0 * (uint32_t)N + nn)) = word;
  };
#pragma unroll
  for (int i = 0; i < NIT; ++i)
    if (r0 + RS * i < K) put(RS * i, v[i]);
#pragma unroll 4
  for (int r = r0 + RS * NIT; r < K; r += RS) put(r - r0, *(const f32x4*)(w + (long long)r * N + nn));
}

// Any N, pass 1: the bits of max |w| over a block of rows of each column, merged with an
// unsigned atomic max (the order of non-negative floats is that of their bits) into
// `bits`, which starts at zero.
__global__ void w8_amax_kernel(const float* __restrict__ w, int K, int N, int rows, unsigned* __restrict__ bits) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const int r0 = blockIdx.y * rows, r1 = min(K, r0 + rows);
  float amax = 0.0f;
  for (int r = r0; r < r1; ++r) amax = fmaxf(amax, fabsf(w[(long long)r * N + n]));
  atomicMax(bits + n, bitcast<unsigned>(amax));
}

// the same, 4 columns per thread (N % 4 == 0)
__global__ void w8_amax_x4_kernel(const float* __restrict__ w, int K, int N, int rows, unsigned* __restrict__ bits) {
  const int n = 4 * (blockIdx.x * blockDim.x + threadIdx.x);
  if (n >= N) return;
  const int r0 = blockIdx.y * rows, r1 = min(K, r0 + rows);
  f32x4 amax = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int r = r0; r < r1; ++r) {
    const f32x4 v = *(const f32x4*)(w + (long long)r * N + n);
#pragma unroll
    for (int c = 0; c < 4; ++c) amax[c] = fmaxf(amax[c], fabsf(v[c]));
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) atomicMax(bits + n + c, bitcast<unsigned>(amax[c]));
}

__global__ void fill_u32_kernel(unsigned* __restrict__ p, int n, unsigned v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// W8, pass 2: code = clamp(rint(w / sc), -127, 127) with sc = max(amax, 1e-8) / 127.
__global__ void w8_quant_kernel(const float* __restrict__ w, int K, int N, const unsigned* __restrict__ bits,
                                int8_t* __restrict__ q) {
  const long long total = (long long)K * N;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const int n = (int)(i % N);
    const float sc = fmaxf(bitcast<float>(bits[n]), 1e-8f) / 127.0f;
    q[i] = (int8_t)(int)fminf(fmaxf(rintf(w[i] / sc), -127.0f), 127.0f);
  }
}

// the same, 4 consecutive elements per thread (N % 4 == 0, so they share a row)
__global__ void w8_quant_x4_kernel(const float* __restrict__ w, int K, int N, const unsigned* __restrict__ bits,
                                   int8_t* __restrict__ q) {
  const long long total4 = (long long)K * N / 4;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total4;
       i += (long long)gridDim.x * blockDim.x) {
    const int n = (int)((4 * i) % N);
    const f32x4 v = *(const f32x4*)(w + 4 * i);
    const u32x4 b = *(const u32x4*)(bits + n);
    uint32_t word = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float sc = fmaxf(bitcast<float>(b[c]), 1e-8f) / 127.0f;
      word |= ((uint32_t)(int)fminf(fmaxf(rintf(v[c] / sc), -127.0f), 127.0f) & 0xFFu) << (8 * c);
    }
    *(uint32_t*)(q + 4 * i) = word;
  }
}

// W8, pass 3: the amax bits become the fp32 scale, in place.
__global__ void w8_scale_kernel(int N, unsigned* __restrict__ bits) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n < N) bits[n] = bitcast<unsigned>(fmaxf(bitcast<float>(bits[n]), 1e-8f) / 127.0f);
}

// ---------------------------------------------------------------------------
// External int4 formats -> the engine layout (quant_formats.py:199-229, 355-466).
// GPTQ packs 8 K-nibbles of one column per int32 word (nibble j = bits 4j..4j+3 =
// row 8w + j), so the engine's pair bytes (even K low, odd K high) are the word's
// little-endian bytes: packed[4w + t][n] = byte t of qweight[w][n].  AWQ packs 8
// N-nibbles of one row per word in the order [0, 2, 4, 6, 1, 3, 5, 7]; column 8c + j
// sits at nibble kAwqRev[j] = [0, 4, 1, 5, 2, 6, 3, 7][j] of word c.
// ---------------------------------------------------------------------------

__constant__ int kAwqRev[8] = {0, 4, 1, 5, 2, 6, 3, 7};

// thread = (word row w, column n): one word in, its 4 bytes to 4 packed rows
__global__ void repack_gptq_kernel(const uint32_t* __restrict__ qw, int K, int N, uint8_t* __restrict__ packed) {
  const long long total = (long long)(K / 8) * N;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const long long w = i / N, n = i - w * N;
    const uint32_t v = qw[i];
#pragma unroll
    for (int t = 0; t < 4; ++t) packed[(4 * w + t) * N + n] = (uint8_t)(v >> (8 * t));
  }
}

// 4 columns per thread (N % 4 == 0): one 16-byte load, a 4x4 byte transpose, four
// 4-byte stores (row 4w + t gets byte t of the four words)
__global__ void repack_gptq_x4_kernel(const uint32_t* __restrict__ qw, int K, int N, uint8_t* __restrict__ packed) {
  const long long total4 = (long long)(K / 8) * N / 4;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total4;
       i += (long long)gridDim.x * blockDim.x) {
    const long long e = 4 * i, w = e / N, n = e - w * N;
    const u32x4 v = *(const u32x4*)(qw + e);
    uint32_t t4[4];
    tr4(v.x, v.y, v.z, v.w, t4);
#pragma unroll
    for (int t = 0; t < 4; ++t) *(uint32_t*)(packed + (4 * w + t) * N + n) = t4[t];
  }
}

// rows 2r and 2r+1 of word column c -> 8 pair bytes: byte b of `e` pairs the words'
// nibbles 2b (columns 0, 4, 1, 5 for b = 0, 1, 2, 3), byte b of `o` their nibbles 2b + 1
// (columns 2, 6, 3, 7).
__device__ __forceinline__ u32x2 awq_pairs(uint32_t lo, uint32_t hi) {
  const uint32_t e = (lo & 0x0F0F0F0Fu) | ((hi & 0x0F0F0F0Fu) << 4);
  const uint32_t o = ((lo >> 4) & 0x0F0F0F0Fu) | (hi & 0xF0F0F0F0u);
  return u32x2{perm(o, e, 0x06040200u), perm(o, e, 0x07050301u)};
}

// thread = (packed row, word); with W2, two words (an even word count, 16-byte stores).
// K = 4096, N = 12288: 8.7 us, 10.9 with a shift and a mask per nibble and 8-byte stores.
template <bool W2>
__global__ void repack_awq_kernel(const uint32_t* __restrict__ qw, int K, int N, uint8_t* __restrict__ packed) {
  const int W = N / 8, per = W2 ? W / 2 : W;
  const long long total = (long long)(K / 2) * per;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const long long r = i / per, c = i - r * per;
    if constexpr (W2) {
      const u32x2 lo = *(const u32x2*)(qw + (2 * r) * W + 2 * c), hi = *(const u32x2*)(qw + (2 * r + 1) * W + 2 * c);
      const u32x2 a = awq_pairs(lo.x, hi.x), b = awq_pairs(lo.y, hi.y);
      *(u32x4*)(packed + r * N + 16 * c) = u32x4{a.x, a.y, b.x, b.y};
    } else {
      *(u32x2*)(packed + r * N + 8 * c) = awq_pairs(qw[(2 * r) * W + c], qw[(2 * r + 1) * W + c]);
    }
  }
}

// compressed-tensors int4 (quant_formats.py:282-354): weight_packed int32 [N][W], 8
// straight-order K nibbles per word, one output feature per row.  Byte i of word w
// holds nibbles k = 8w + 2i (low) and 8w + 2i + 1 (high): exactly the engine's pair
// byte of packed row 4w + i, column n.  So the engine layout [K/2][N] is the byte
// transpose of the [N][4W] byte view, cut to K/2 rows.  A tile of 128 columns x 128
// packed rows goes through LDS: a thread loads 16 bytes of each of 4 source rows (V4: W %
// 4 == 0 and a 16-byte aligned source; word by word otherwise), transposes them 4 x 4 bytes
// at a time in registers and writes dwords of 4 columns; packed rows then leave as 128
// contiguous bytes.  K = 4096, N = 12288: 8.8 us, 16.5 through a 64 x 64 tile of single bytes.
template <bool V4>
__global__ __launch_bounds__(256) void repack_ct_kernel(const uint32_t* __restrict__ qw, int N, int W, int KB,
                                                        uint8_t* __restrict__ packed) {
  constexpr int T = 128, P = T / 4 + 1;  // row pitch in dwords
  __shared__ uint32_t t[T * P];          // [packed row j - j0][columns 4 nq .. 4 nq + 3]
  const int n0 = blockIdx.x * T, j0 = blockIdx.y * T;
  const int tid = threadIdx.x;
  {
    const int nq = tid >> 3, jc = 16 * (tid & 7);  // source rows n0 + 4 nq .. + 3, bytes j0 + jc .. + 15
    const int n = n0 + 4 * nq, wj = (j0 + jc) >> 2;
    u32x4 v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t* src = qw + (long long)min(n + r, N - 1) * W;
      if constexpr (V4) {
        v[r] = *(const u32x4*)(src + min(wj, W - 4));  // (words past the row are not stored)
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[r][q] = src[min(wj + q, W - 1)];
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t x[4];
      tr4(v[0][q], v[1][q], v[2][q], v[3][q], x);
#pragma unroll
      for (int b = 0; b < 4; ++b) t[(jc + 4 * q + b) * P + nq] = x[b];
    }
  }
  __syncthreads();
  const int c = 4 * (tid & 7), n = n0 + 4 * c;  // 16 columns
  if (n >= N) return;                           // N % 16 == 0: the 16 columns are all in range
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int jr = 32 * i + (tid >> 3), j = j0 + jr;
    if (j >= KB) break;
    const uint32_t* row = t + jr * P + c;
    *(u32x4*)(packed + (long long)j * N + n) = u32x4{row[0], row[1], row[2], row[3]};
  }
}

// z[g][8c + j] = nibble (awq ? kAwqRev[j] : j) of qzeros[g][c], plus `add`
__global__ void zeros_unpack_kernel(const uint32_t* __restrict__ qz, int G, int N, int awq, int add,
                                    uint8_t* __restrict__ z) {
  const long long total = (long long)G * N;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const long long g = i / N;
    const int n = (int)(i - g * N), c = n >> 3, j = n & 7;
    const int pos = awq ? kAwqRev[j] : j;
    z[i] = (uint8_t)(((qz[g * (N / 8) + c] >> (4 * pos)) & 0xFu) + (uint32_t)add);
  }
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

static dim3 grid_for(long long total) {
  long long blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  if (blocks < 1) blocks = 1;
  return dim3((unsigned)blocks);
}

hipError_t launch_w4_unpack(const uint8_t* p, int K, int N, uint8_t* out, hipStream_t st) {
  hipLaunchKernelGGL(w4_unpack_kernel, grid_for((long long)(K / 2) * N), dim3(256), 0, st, p, K, N, out);
  return hipGetLastError();
}

hipError_t launch_w4_dequant(const uint8_t* p, const void* s, int sdt, const uint8_t* z, int group, int K,
                             int N, float* out, hipStream_t st) {
  hipLaunchKernelGGL(w4_dequant_kernel, grid_for((long long)(K / 2) * N), dim3(256), 0, st, p, s, sdt, z,
                     group, K, N, out);
  return hipGetLastError();
}

hipError_t launch_w8_dequant(const int8_t* w, const void* s, int sdt, int K, int N, float* out,
                             hipStream_t st) {
  hipLaunchKernelGGL(w8_dequant_kernel, grid_for((long long)K * N), dim3(256), 0, st, w, s, sdt, K, N, out);
  return hipGetLastError();
}

hipError_t launch_requant_w4(const float* w, int K, int N, int group, uint8_t* packed, uint16_t* sbf,
                             hipStream_t st) {
  const dim3 wg(256);
  if (N % 4 == 0 && group == 32 && aligned16(w) && aligned16(packed) && aligned16(sbf))
    hipLaunchKernelGGL((requant_w4_kernel_reg<32, 4>), dim3((unsigned)((N / 4 + 255) / 256), (unsigned)(K / 32)), wg,
                       0, st, w, N, packed, sbf);
  else if (N % 2 == 0 && group == 64 && aligned16(w) && aligned16(packed) && aligned16(sbf))
    hipLaunchKernelGGL((requant_w4_kernel_reg<64, 2>), dim3((unsigned)((N / 2 + 255) / 256), (unsigned)(K / 64)), wg,
                       0, st, w, N, packed, sbf);
  else
    hipLaunchKernelGGL(requant_w4_kernel, dim3((unsigned)((N + 255) / 256), (unsigned)(K / group)), wg, 0, st, w, K, N,
                       group, packed, sbf);
  return hipGetLastError();
}

hipError_t launch_requant_w8(const float* w, int K, int N, int8_t* q, float* scale, hipStream_t st) {
  const bool x4 = N % 4 == 0 && aligned16(w) && aligned16(q) && aligned16(scale);
  // Longer columns take four launches that spread the rows over the chip: a strip walks all
  // of them on one CU, twice past its registers, from farther caches the longer it is, and a
  // second round of strips starts late.  us, strips / four launches: K = 16384: N = 64 45 / 34,
  // 1024 89 / 66, 4096 162 / 144; K = 12288: 1024 53 / 50, 4096 104 / 112, 6144 185 / 156;
  // K = 8192: 64 24 / 24, 4096 66 / 83, 8192 155 / 135; K = 6144: 6144 82 / 90.
  const int longest = N <= 256 ? 8192 : N <= 2048 ? 10240 : N < 6144 ? 12288 : 6144;
  if (x4 && K <= longest) {
    // 64 columns per strip where that leaves at least 128 strips, or where a strip's rows fit
    // the registers twice over; 16 columns otherwise (K = 4096: N = 6144 38 us against 46
    // with 64 columns, N = 8192 65 against 53, N = 16384 150 against 110; K = 1024, N = 6144
    // 19.4 against 13.0)
    const bool wide = N >= 8192 || (K <= 1024 && N >= 4096);
    const int strips = (N + (wide ? 63 : 15)) / (wide ? 64 : 16);
    const dim3 grid((unsigned)strips), wg(1024);
    if (wide) hipLaunchKernelGGL((requant_w8_strip_kernel<8, 16>), grid, wg, 0, st, w, K, N, strips, q, scale);
    else if (K <= 1024) hipLaunchKernelGGL((requant_w8_strip_kernel<4, 4>), grid, wg, 0, st, w, K, N, strips, q, scale);
    else if (K <= 2048) hipLaunchKernelGGL((requant_w8_strip_kernel<8, 4>), grid, wg, 0, st, w, K, N, strips, q, scale);
    else hipLaunchKernelGGL((requant_w8_strip_kernel<16, 4>), grid, wg, 0, st, w, K, N, strips, q, scale);
    return hipGetLastError();
  }
  unsigned* bits = (unsigned*)scale;  // amax bits first, the scale at the end
  const unsigned cb = (unsigned)((N + 255) / 256);
  constexpr int kRows = 64;  // rows per amax block: enough blocks to fill the chip
  hipLaunchKernelGGL(fill_u32_kernel, dim3(cb), dim3(256), 0, st, bits, N, 0u);
  const unsigned rb = (unsigned)((K + kRows - 1) / kRows);
  if (x4) {
    hipLaunchKernelGGL(w8_amax_x4_kernel, dim3((unsigned)((N / 4 + 255) / 256), rb), dim3(256), 0, st, w, K, N, kRows,
                       bits);
    hipLaunchKernelGGL(w8_quant_x4_kernel, grid_for((long long)K * N / 4), dim3(256), 0, st, w, K, N, bits, q);
  } else {
    hipLaunchKernelGGL(w8_amax_kernel, dim3(cb, rb), dim3(256), 0, st, w, K, N, kRows, bits);
    hipLaunchKernelGGL(w8_quant_kernel, grid_for((long long)K * N), dim3(256), 0, st, w, K, N, bits, q);
  }
  hipLaunchKernelGGL(w8_scale_kernel, dim3(cb), dim3(256), 0, st, N, bits);
  return hipGetLastError();
}

hipError_t launch_repack_gptq(const int32_t* qw, int K, int N, uint8_t* packed, hipStream_t st) {
  if (N % 4 == 0 && aligned16(qw) && aligned16(packed))
    hipLaunchKernelGGL(repack_gptq_x4_kernel, grid_for((long long)(K / 8) * N / 4), dim3(256), 0, st,
                       (const uint32_t*)qw, K, N, packed);
  else
    hipLaunchKernelGGL(repack_gptq_kernel, grid_for((long long)(K / 8) * N), dim3(256), 0, st, (const uint32_t*)qw,
                       K, N, packed);
  return hipGetLastError();
}

hipError_t launch_repack_awq(const int32_t* qw, int K, int N, uint8_t* packed, hipStream_t st) {
  const uint32_t* q = (const uint32_t*)qw;
  const long long words = (long long)(K / 2) * (N / 8);
  if (N % 16 == 0 && aligned16(qw) && aligned16(packed))
    hipLaunchKernelGGL(repack_awq_kernel<true>, grid_for(words / 2), dim3(256), 0, st, q, K, N, packed);
  else
    hipLaunchKernelGGL(repack_awq_kernel<false>, grid_for(words), dim3(256), 0, st, q, K, N, packed);
  return hipGetLastError();
}

hipError_t launch_repack_ct(const int32_t* qw, int N, int W, int K, uint8_t* packed, hipStream_t st) {
  const int KB = K / 2;
  const uint32_t* q = (const uint32_t*)qw;
  const dim3 grid((unsigned)((N + 127) / 128), (unsigned)((KB + 127) / 128)), wg(256);
  if (W % 4 == 0 && aligned16(qw)) hipLaunchKernelGGL(repack_ct_kernel<true>, grid, wg, 0, st, q, N, W, KB, packed);
  else hipLaunchKernelGGL(repack_ct_kernel<false>, grid, wg, 0, st, q, N, W, KB, packed);
  return hipGetLastError();
}

hipError_t launch_zeros_unpack(const int32_t* qz, int G, int N, int awq, int add, uint8_t* z, hipStream_t st) {
  hipLaunchKernelGGL(zeros_unpack_kernel, grid_for((long long)G * N), dim3(256), 0, st, (const uint32_t*)qz, G, N,
                     awq, add, z);
  return hipGetLastError();
}

}  // namespace qlin
