// Int8 activation path (src/kernel.rs:70-166, Q8Activation / dot_q8_0_i8 / matmul_q8_0_i8):
// activations quantized per 32-value block to i8 with an f32 scale, multiplied against Q8_0
// weights with i8 MFMAs. Results are bit-identical to the reference's scalar integer dot: the
// i32 block sums are exact whatever the order, and each output's blocks are folded by one lane,
// in block order, as s += ((f32)isum * dw) * dx with no fused multiply-add.
#include <hip/hip_runtime.h>

#include "deq.hpp"
#include "kernels.hpp"

namespace rehip {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// One thread per (row, 32-value block): Q8Activation::from_f32 (kernel.rs:88-105). d = max|x|/127
// (NaN never wins the max), inv = 1/d or 0, q = round-half-away(x * inv) clamped to [-127, 127],
// a NaN product gives 0. Division and rounding are the IEEE-exact device operations.
__global__ __launch_bounds__(256) void quantize_q8_act_kernel(const float* __restrict__ x, int rows, int n,
                                                              float* __restrict__ scales, int8_t* __restrict__ qs) {
  const int nb = n >> 5;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long long)rows * nb) return;
  const int row = (int)(i / nb), kb = (int)(i - (long long)row * nb);
  const float4* src = reinterpret_cast<const float4*>(x + (size_t)row * n + (size_t)kb * 32);
  float v[32];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float4 f = src[j];
    v[4 * j] = f.x;
    v[4 * j + 1] = f.y;
    v[4 * j + 2] = f.z;
    v[4 * j + 3] = f.w;
  }
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 32; ++j) amax = fmaxf(amax, fabsf(v[j]));
  const float d = amax / 127.0f;
  const float inv = d > 0.0f ? 1.0f / d : 0.0f;
  uint32_t packed[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    uint32_t w = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      float r = roundf(v[4 * j + b] * inv);
      r = r != r ? 0.0f : fminf(fmaxf(r, -127.0f), 127.0f);
      w |= ((uint32_t)(uint8_t)(int8_t)(int)r) << (8 * b);
    }
    packed[j] = w;
  }
  uint4* dst = reinterpret_cast<uint4*>(qs + (size_t)row * n + (size_t)kb * 32);
  dst[0] = make_uint4(packed[0], packed[1], packed[2], packed[3]);
  dst[1] = make_uint4(packed[4], packed[5], packed[6], packed[7]);
  scales[i] = d;
}

constexpr int kI8Chunk = 256;  // blocks of activation scales staged in LDS at a time (n <= 8192: one)
constexpr int kI8Ahead = 4;    // blocks whose operands are in flight ahead of the MFMA

// 1.5 * 2^23: an MFMA that starts from these bits leaves the bits of the float kI8Magic + isum
// (|isum| <= 32 * 128 * 127 < 2^22), so with bias = -kI8Magic * dw (exact: 13 significant bits) one
// fma gives round(isum * dw), the conversion and the first multiply of the fold in one operation.
constexpr float kI8Magic = 12582912.0f;
constexpr int kI8MagicBits = 0x4B400000;

// Y (rows x m) = Q8_0 W (m x n, tiled slabs) times quantized activations. Workgroup = 4 waves = two
// 64-row weight tiles x 32 activation rows; wave w owns 32 weight rows. Per block one
// v_mfma_i32_32x32x32_i8 (A = 32 activation rows x 32 i8, B = 32 i8 x 32 weight rows; lane l supplies
// row/column l%32 and bytes 16(l/32)..+15 of the block to both, so the i32 sums are the exact block dot
// products) and the f32 fold of the 16 results the lane holds: activation rows 8(i/4) + 4(l/32) + i%4
// of weight row l%32, three operations each (kI8Magic).
// The activations go through LDS in stages of kI8Ahead = 4 blocks, one whole 128-byte line of each
// row (a thread copies one 16-byte unit of a stage, loaded a stage ahead): read per block straight
// from the rows, an operand load touched 32 lines for 32 bytes of each, and the lines left the L1
// before their other three blocks were read. The activation scales of up to 256 blocks are staged
// block-major; weights load into registers kI8Ahead blocks ahead, at a scalar offset. No branch
// inside a stage (a branch between an MFMA and the reads of its result, or between a load and its
// use, makes the compiler wait for every outstanding load).
// The first stage's activations and scales are loaded together (one after the other, rows of 256 and 512 were
// 0.5-0.9 us slower than read straight from the rows). 4864 x 896, 961 rows: 32.4 -> 23.1 us, rows of 4864 154
// -> 107 us, rows of 256 4.9 -> 4.9 at 32 rows (the three-operation fold alone: 4864 x 896 34.8 -> 34.5 with the
// quantization).
// A scale that is not finite has no exact bias and leaves NaN: such rows are folded again at the end.
__global__ __launch_bounds__(256, 4) void q8_i8_gemm_kernel(const uint8_t* __restrict__ W, const float* __restrict__ xs,
                                                         const int8_t* __restrict__ xq, float* __restrict__ y, int m,
                                                         int n, int rows, int tiles) {
#pragma clang fp contract(off)
  extern __shared__ __align__(16) float dxs_flat[];     // min(nb, kI8Chunk) x 32
  float (*dxs)[32] = reinterpret_cast<float (*)[32]>(dxs_flat);
  __shared__ uint4 xb[2][32 * 8];                       // 16-byte unit u of row r at r * 8 + (u ^ (r / 2 % 8))
  constexpr uint32_t SLAB = 64 * 34;
  static_assert(kI8Ahead == 4, "a stage is one 128-byte line of a row");
  const int nb = n >> 5;
  const int r0 = blockIdx.y * 32;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = min(2 * (int)blockIdx.x + (wave >> 1), tiles - 1);   // past the last: computed, not stored
  const int h = lane >> 5, c = lane & 31;
  const int trow = (wave & 1) * 32 + c;                 // weight row inside the tile
  // the tile's slabs and the group's activation rows, each below 2 GiB (a matrix has at most 2^24 columns)
  const __amdgpu_buffer_rsrc_t wr = make_rsrc(W + (size_t)tile * nb * SLAB, (uint32_t)nb * SLAB);
  const __amdgpu_buffer_rsrc_t ar = make_rsrc(xq + (size_t)r0 * n, (uint32_t)min(32, rows - r0) * (uint32_t)n);
  const int wo = h * (64 * 16) + trow * 16, wdo = 2 * (64 * 16) + trow * 2;
  // this thread's unit of a stage (units past the row's end hold the next row's bytes, rows past the
  // last zeros: neither is used)
  const int xr = threadIdx.x >> 3, xu = threadIdx.x & 7;
  const int xo = xr * n + 16 * xu, xd = xr * 8 + (xu ^ ((xr >> 1) & 7));
  const int nst = (nb + kI8Ahead - 1) / kI8Ahead;
  auto load_x = [&](int st) __attribute__((always_inline)) {
    return bld16(ar, (uint32_t)(xo + 128 * min(st, nst - 1)));
  };
  v4i Bw[kI8Ahead];
  uint32_t D[kI8Ahead];
  auto load = [&](const int j, const int kb) __attribute__((always_inline)) {
    const int kn = min(kb, nb - 1);
    Bw[j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, wo, kn * (int)SLAB, 0));
    D[j] = __builtin_amdgcn_raw_buffer_load_b16(wr, wdo, kn * (int)SLAB, 0);
  };
  // scales of four of this thread's blocks of a row, every eighth from k0 of the chunk at kb0
  const int st = threadIdx.x & 31, sk = threadIdx.x >> 5;
  const float* srow = xs + (size_t)min(r0 + st, rows - 1) * nb;
  float sv[4];
  auto load_s = [&](const int kb0, const int kc, const int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) sv[u] = srow[kb0 + min(k0 + 8 * u, kc - 1)];
  };
  // the first stage's activations and scales go out together, ahead of the weights: one memory round trip
  uint4 xv = load_x(0);
  load_s(0, min(kI8Chunk, nb), sk);
#pragma unroll
  for (int j = 0; j < kI8Ahead; ++j) load(j, j);
  __builtin_amdgcn_sched_barrier(0);
  float s[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] = 0.0f;
  v16i magic;
#pragma unroll
  for (int i = 0; i < 16; ++i) magic[i] = kI8MagicBits;

  // one block: MFMA on slot j, refill slot j with block kb + kI8Ahead (clamped), fold
  auto step = [&](const int j, const int kb, const uint4* xrow, const float* dxrow) __attribute__((always_inline)) {
    const v4i a = *reinterpret_cast<const v4i*>(xrow + ((2 * j + h) ^ ((c >> 1) & 7)));
    const v16i acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, Bw[j], magic, 0, 0, 0);
    const float dw = f16_bits_to_f32(D[j]);
    const float bias = -kI8Magic * dw;
    __builtin_amdgcn_sched_barrier(0);    // slot j is free: the refill takes its registers
    load(j, kb + kI8Ahead);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float4 dx = *reinterpret_cast<const float4*>(dxrow + 8 * g + 4 * h);
      const float dxv[4] = {dx.x, dx.y, dx.z, dx.w};
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const int i = 4 * g + jj;
        const float t = __builtin_fmaf(__int_as_float(acc[i]), dw, bias) * dxv[jj];   // not contracted (see above)
        s[i] = s[i] + t;
      }
    }
    __builtin_amdgcn_sched_barrier(0);   // else every refill moves ahead of the stage's first wait
  };

  xb[0][xd] = xv;
  xv = load_x(1);
  int buf = 0;
  for (int kb0 = 0; kb0 < nb; kb0 += kI8Chunk) {
    const int kc = min(kI8Chunk, nb - kb0);
    if (kb0) __syncthreads();
    // scales of 32 activation rows x kc blocks -> dxs[block][row]
    for (int k0 = sk; k0 < kc; k0 += 8 * 4) {
      if (kb0 || k0 != sk) load_s(kb0, kc, k0);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (k0 + 8 * u < kc) dxs[k0 + 8 * u][st] = sv[u];
    }
    const int full = kc & ~(kI8Ahead - 1);
#pragma unroll 1
    for (int k = 0; k < full; k += kI8Ahead) {
      __syncthreads();                    // the stage is there; everyone has read the one before it
      xb[buf ^ 1][xd] = xv;
      xv = load_x((kb0 + k) / kI8Ahead + 2);
      __builtin_amdgcn_sched_barrier(0);
      const uint4* xrow = xb[buf] + c * 8;
#pragma unroll
      for (int j = 0; j < kI8Ahead; ++j) step(j, kb0 + k + j, xrow, dxs[k + j]);
      buf ^= 1;
    }
  }
  // blocks past the last whole stage (only in the last chunk: kI8Chunk is a multiple of 4)
  __syncthreads();
  const int tail = nb & ~(kI8Ahead - 1);
#pragma unroll
  for (int j = 0; j < kI8Ahead - 1; ++j)
    if (tail + j < nb) step(j, tail + j, xb[buf] + c * 8, dxs[(tail & (kI8Chunk - 1)) + j]);
  bool nan = false;                       // inf * dw - inf: every sum of such a row is NaN
#pragma unroll
  for (int i = 0; i < 16; ++i) nan |= s[i] != s[i];
  if (__any(nan)) {
    const int8_t* arow = xq + (size_t)min(r0 + c, rows - 1) * n + 16 * h;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll 1
    for (int kb = 0; kb < nb; ++kb) {
      load(0, kb);
      const v4i a = *reinterpret_cast<const v4i*>(arow + (size_t)kb * 32);
      const v16i acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, Bw[0], v16i{}, 0, 0, 0);
      const float dw = f16_bits_to_f32(D[0]);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float dx = xs[(size_t)min(r0 + 8 * (i >> 2) + 4 * h + (i & 3), rows - 1) * nb + kb];
        const float t = ((float)acc[i] * dw) * dx;
        s[i] = s[i] + t;
      }
    }
  }
  const int wrow = tile * 64 + trow;
  if (wrow >= m || 2 * (int)blockIdx.x + (wave >> 1) >= tiles) return;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = r0 + 8 * (i >> 2) + 4 * h + (i & 3);
    if (r < rows) y[(size_t)r * m + wrow] = s[i];
  }
}

constexpr int kSegWaves = 4;    // K segments (one per wave) of one output tile
constexpr int kSegBlocks = 4;   // blocks per wave per round

// Long rows over few output tiles: one 32 x 32 output tile per workgroup of kSegWaves waves. A
// round covers kSegWaves * kSegBlocks consecutive blocks; wave w takes kSegBlocks of them and
// computes their terms ((f32)isum * dw) * dx in parallel with the other waves (one i8 MFMA per
// block, as q8_i8_gemm_kernel), then the running sums (16 per lane) pass from wave to wave
// through LDS, each wave adding its terms in block order: the same fold, in the same order, as
// one lane walking all blocks, with only the adds serial. The next round's operands load during
// the folds (keeping two rounds in flight measured no faster: the compiler's wait counts then
// drain every outstanding load at the round's first MFMA).
__global__ __launch_bounds__(64 * kSegWaves) void q8_i8_gemm_seg_kernel(const uint8_t* __restrict__ W,
                                                                         const float* __restrict__ xs,
                                                                         const int8_t* __restrict__ xq,
                                                                         float* __restrict__ y, int m, int n,
                                                                         int rows) {
#pragma clang fp contract(off)
  constexpr int S = kSegWaves, KBs = kSegBlocks, RB = S * KBs;
  static_assert(kI8Chunk % RB == 0, "scale chunks hold whole rounds");
  extern __shared__ __align__(16) float dxs_flat[];   // min(nb, kI8Chunk) x 32 scales
  float (*dxs)[32] = reinterpret_cast<float (*)[32]>(dxs_flat);
  __shared__ float sbuf[16][64];          // running sums, [result register][lane]
  const int nb = n >> 5;
  const int grp = blockIdx.x;             // 32 weight rows: tile grp/2, rows 32 (grp%2) ..
  const int tile = grp >> 1;
  const int r0 = blockIdx.y * 32;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int h = lane >> 5, c = lane & 31;
  const int trow = (grp & 1) * 32 + c;
  const uint8_t* wb = W + (size_t)tile * nb * (64 * 34) + h * (64 * 16) + trow * 16;
  const uint8_t* wd = W + (size_t)tile * nb * (64 * 34) + 2 * (64 * 16) + trow * 2;
  const int8_t* arow = xq + (size_t)min(r0 + c, rows - 1) * n + 16 * h;
  const int rounds = (nb + RB - 1) / RB;
  v4i A[KBs], Bw[KBs];
  uint32_t D[KBs];
  auto load = [&](int rr, v4i (&a)[KBs], v4i (&b)[KBs], uint32_t (&d)[KBs]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < KBs; ++j) {
      const int kb = min(rr * RB + wave * KBs + j, nb - 1);
      a[j] = *reinterpret_cast<const v4i*>(arow + (size_t)kb * 32);
      b[j] = *reinterpret_cast<const v4i*>(wb + (size_t)kb * (64 * 34));
      d[j] = *reinterpret_cast<const uint16_t*>(wd + (size_t)kb * (64 * 34));
    }
  };
  load(0, A, Bw, D);
  float s[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] = 0.0f;
  auto round = [&](int rr, v4i (&a)[KBs], v4i (&b)[KBs], uint32_t (&d)[KBs]) __attribute__((always_inline)) {
    const int b0 = rr * RB;
    const int kc0 = b0 / kI8Chunk * kI8Chunk;     // first block of the staged scale chunk
    if (b0 == kc0) {
      // scales of 32 activation rows x the chunk's blocks -> dxs[block][row], 8 loads in flight
      const int kc = min(kI8Chunk, nb - kc0);
      __syncthreads();                    // the previous chunk's readers are done
      for (int e0 = threadIdx.x; e0 < kc * 32; e0 += 64 * S * 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int e = e0 + 64 * S * u;
          const int t = e / kc, k = e - t * kc;
          v[u] = e < kc * 32 ? xs[(size_t)min(r0 + t, rows - 1) * nb + kc0 + k] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int e = e0 + 64 * S * u;
          const int t = e / kc, k = e - t * kc;
          if (e < kc * 32) dxs[k][t] = v[u];
        }
      }
      __syncthreads();
    }
    float tm[KBs][16];
#pragma unroll
    for (int j = 0; j < KBs; ++j) {
      const v16i acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[j], b[j], v16i{}, 0, 0, 0);
      const float dw = f16_bits_to_f32(d[j]);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int kl = min(b0 + wave * KBs + j, nb - 1) - kc0;   // clamped blocks are not folded
        const float4 dx = *reinterpret_cast<const float4*>(&dxs[kl][8 * g + 4 * h]);
        const float dxv[4] = {dx.x, dx.y, dx.z, dx.w};
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) tm[j][4 * g + jj] = ((float)acc[4 * g + jj] * dw) * dxv[jj];
      }
    }
    if (rr + 1 < rounds) load(rr + 1, a, b, d);   // the next round's operands load during the folds
    // ordered fold: waves 0 .. S-1 in turn, each continuing the running sums of the one before
    for (int w = 0; w < S; ++w) {
      if (wave == w) {
        if (rr > 0 || w > 0) {
#pragma unroll
          for (int i = 0; i < 16; ++i) s[i] = sbuf[i][lane];
        }
#pragma unroll
        for (int j = 0; j < KBs; ++j) {
          if (b0 + w * KBs + j < nb) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = s[i] + tm[j][i];
          }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) sbuf[i][lane] = s[i];
      }
      __syncthreads();
    }
  };
  for (int rr = 0; rr < rounds; ++rr) round(rr, A, Bw, D);
  if (wave != 0) return;
  const int wr = tile * 64 + trow;
  if (wr >= m) return;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = r0 + 8 * (i >> 2) + 4 * h + (i & 3);
    if (r < rows) y[(size_t)r * m + wr] = sbuf[i][lane];
  }
}

constexpr int kI8GemvRows = 16;       // weight rows per workgroup
constexpr int kI8GemvMaxBlocks = 960; // 16 x (nb + 1) f32 terms in LDS, at most 61.5 KB (n <= 30720)

// One activation row (matvec_q8_0_i8, kernel.rs:145-154). Workgroup = 256 threads = 16 weight
// rows x 16 block lanes: thread (row, j) computes the terms ((f32)isum * dw) * dx of blocks
// j, j + 16, ... of its row (isum by v_dot4_i32_i8, exact) into LDS; then one lane per row adds
// its row's terms in block order.
__global__ __launch_bounds__(256) void q8_i8_gemv_kernel(const uint8_t* __restrict__ W, const float* __restrict__ xs,
                                                         const int8_t* __restrict__ xq, float* __restrict__ y, int m,
                                                         int n) {
#pragma clang fp contract(off)
  extern __shared__ float terms[];               // kI8GemvRows x (nb + 1)
  const int nb = n >> 5;
  const int stride = nb + 1;
  const int r = threadIdx.x & (kI8GemvRows - 1), j = threadIdx.x >> 4;
  const int row = blockIdx.x * kI8GemvRows + r;         // may pass m: padding rows are zero
  const int tile = row >> 6, trow = row & 63;
  const uint8_t* slab0 = W + (size_t)tile * nb * (64 * 34);
  for (int kb = j; kb < nb; kb += 16) {
    const uint8_t* slab = slab0 + (size_t)kb * (64 * 34);
    const uint4 w0 = *reinterpret_cast<const uint4*>(slab + trow * 16);
    const uint4 w1 = *reinterpret_cast<const uint4*>(slab + 64 * 16 + trow * 16);
    const float dw = f16_bits_to_f32(*reinterpret_cast<const uint16_t*>(slab + 2 * (64 * 16) + trow * 2));
    const uint4 a0 = *reinterpret_cast<const uint4*>(xq + (size_t)kb * 32);
    const uint4 a1 = *reinterpret_cast<const uint4*>(xq + (size_t)kb * 32 + 16);
    int isum = 0;
    isum = __builtin_amdgcn_sdot4((int)w0.x, (int)a0.x, isum, false);
    isum = __builtin_amdgcn_sdot4((int)w0.y, (int)a0.y, isum, false);
    isum = __builtin_amdgcn_sdot4((int)w0.z, (int)a0.z, isum, false);
    isum = __builtin_amdgcn_sdot4((int)w0.w, (int)a0.w, isum, false);
    isum = __builtin_amdgcn_sdot4((int)w1.x, (int)a1.x, isum, false);
    isum = __builtin_amdgcn_sdot4((int)w1.y, (int)a1.y, isum, false);
    isum = __builtin_amdgcn_sdot4((int)w1.z, (int)a1.z, isum, false);
    isum = __builtin_amdgcn_sdot4((int)w1.w, (int)a1.w, isum, false);
    terms[r * stride + kb] = ((float)isum * dw) * xs[kb];
  }
  __syncthreads();
  if (j != 0 || row >= m) return;
  float acc = 0.0f;
  for (int kb = 0; kb < nb; ++kb) acc = acc + terms[r * stride + kb];
  y[row] = acc;
}

}  // namespace

hipError_t launch_quantize_q8_act(const float* x, int rows, int n, float* scales, int8_t* qs, hipStream_t s) {
  const long long blocks = (long long)rows * (n >> 5);
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(quantize_q8_act_kernel, dim3((unsigned)((blocks + 255) / 256)), dim3(256), 0, s, x, rows, n,
                     scales, qs);
  return hipGetLastError();
}

hipError_t launch_q8_i8_gemm(const uint8_t* W, int tiles, const float* xs, const int8_t* xq, float* y, int m, int n,
                             int rows, hipStream_t s) {
  if (rows == 0) return hipSuccess;
  if (rows == 1 && (n >> 5) <= kI8GemvMaxBlocks) {
    const size_t lds = (size_t)kI8GemvRows * ((n >> 5) + 1) * sizeof(float);
    hipLaunchKernelGGL(q8_i8_gemv_kernel, dim3((unsigned)(tiles * (64 / kI8GemvRows))), dim3(256), lds, s, W, xs, xq,
                       y, m, n);
    return hipGetLastError();
  }
  const unsigned rgroups = (unsigned)((rows + 31) / 32);
  // long rows over few output tiles: split each tile's fold over the waves of a workgroup
  if ((n >> 5) >= 64 && (size_t)tiles * 2 * rgroups < 512) {
    const size_t lds = (size_t)min(n >> 5, kI8Chunk) * 32 * sizeof(float);
    hipLaunchKernelGGL(q8_i8_gemm_seg_kernel, dim3((unsigned)tiles * 2, rgroups), dim3(64 * kSegWaves), lds, s, W,
                       xs, xq, y, m, n, rows);
    return hipGetLastError();
  }
  const size_t lds = (size_t)min(n >> 5, kI8Chunk) * 32 * sizeof(float);
  hipLaunchKernelGGL(q8_i8_gemm_kernel, dim3((unsigned)(tiles + 1) / 2, rgroups), dim3(256), lds, s, W, xs, xq, y, m, n,
                     rows, tiles);
  return hipGetLastError();
}

}  // namespace rehip
