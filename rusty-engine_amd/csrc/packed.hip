// GEMM over packed bf16 operands: Y[N x m] = X[N x K] * W[m x K]^T for many activation rows.
//
// The tiled GEMM (gemm.hip) decodes a weight tile and converts the activation rows again in every
// workgroup that uses them; from a few hundred rows on, that VALU and LDS-write work and the f32
// activation reads bound it, not the matrix cores. Here one launch (pack_kernel) writes both
// operands once, as bf16 MFMA fragments, and the GEMM's inner loop is LDS DMA, fragment reads and
// MFMAs only.
//
// Packed layout: a fragment is 32 rows x 16 k, 1 KiB, in the operand order of
// v_mfma_f32_32x32x16_bf16: lane l's 16 bytes are row l % 32, k 8 (l / 32) .. + 7. Fragment
// (g, ks) of an operand (rows 32g.., k 16ks..) is at (g * KS + ks) * 1024, KS = ceil(K / 32) * 2.
// A fragment read is then 64 consecutive 16-byte units (no bank conflicts) and a stage is copied
// to LDS in contiguous 1 KiB pieces. K past the row is zero in both operands; rows past the
// matrix are not written (they feed outputs that are not stored).
//
// f32 mode: a second plane of each operand holds the bf16 rounding of what the first leaves, and every
// product is w_hi x_hi + w_hi x_lo + w_lo x_hi in f32 accumulators, each term within 2^-16 relative, as in
// the tiled GEMM. BF16 weights leave nothing: one plane and two products, w x_hi + w x_lo. NP: products
// per pair of operands (1 in bf16 mode, 3 or 2 in f32 mode).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>

#include "deq.hpp"
#include "kernels.hpp"
#include "qfrag.hpp"

namespace rehip {

namespace {

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4_t;

// s_waitcnt vmcnt(N) lgkmcnt(0): at most N copies of this wave still in flight, every fragment read
// done (the builtin, so the compiler's own wait counting sees it)
template <int N>
__device__ __forceinline__ void wait_copies() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
}

// 8 values -> one fragment unit (bf16, round to nearest even) and the unit of their remainders
template <bool SP>
__device__ __forceinline__ void store_unit(uint8_t* dst, size_t lo, const float (&v)[8]) {
  bf16x8_t h;
#pragma unroll
  for (int i = 0; i < 8; ++i) h[i] = (__bf16)v[i];
  *reinterpret_cast<bf16x8_t*>(dst) = h;
  if constexpr (SP) {
    bf16x8_t l;
#pragma unroll
    for (int i = 0; i < 8; ++i) l[i] = (__bf16)(v[i] - (float)h[i]);
    *reinterpret_cast<bf16x8_t*>(dst + lo) = l;
  }
}

// byte offset of the unit of (row, k), k a multiple of 8
__device__ __forceinline__ size_t unit_off(int row, int k, int KS) {
  return ((size_t)(row >> 5) * KS + (k >> 4)) * 1024 + ((k >> 3) & 1) * 512 + (row & 31) * 16;
}

// the 8 elements k.. of a row-major row (K % 8 == 0 and 16-byte aligned rows), widened to f32
template <uint32_t T>
__device__ __forceinline__ void load8(const void* p, size_t i, float (&v)[8]) {
  if constexpr (T == 0) {
    const float4* q = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(p) + i);
    const float4 a = q[0], b = q[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
    const uint4 u = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p) + i);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (T == 1) {
        v[2 * j] = f16_bits_to_f32(w[j] & 0xFFFFu);
        v[2 * j + 1] = f16_bits_to_f32(w[j] >> 16);
      } else {
        v[2 * j] = __uint_as_float(w[j] << 16);
        v[2 * j + 1] = __uint_as_float(w[j] & 0xFFFF0000u);
      }
    }
  }
}

// One wave packs 32 rows x 64 k of a row-major operand: lane l takes row l % 32 and, of each of
// the four k steps, half l / 32, so a row's 64 k are read as whole lines and each store
// instruction writes one whole fragment.
constexpr int kRowPackK = 64;
template <uint32_t T, bool SP>
__device__ __forceinline__ void pack_rows(const void* src, int rows, int K, int KS, int g, int kc, uint8_t* dst,
                                          size_t lo) {
  const int lane = threadIdx.x & 63;
  const int row = 32 * g + (lane & 31);
  const int k0 = kRowPackK * kc + 8 * (lane >> 5);
  if (row >= rows) return;
  float v[4][8];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int k = k0 + 16 * j;
    if (k < K) {
      load8<T>(src, (size_t)row * K + k, v[j]);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[j][i] = 0.0f;
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int k = k0 + 16 * j;
    if (k < 16 * KS) store_unit<SP>(dst + unit_off(row, k, KS), lo, v[j]);
  }
}

// One wave packs one 32-quant chunk of a slab's 64 rows (lane = row): the four units of the
// chunk's two 16-element runs. second: of W2 (which may be the same matrix as W).
template <int T, bool SP>
__device__ __forceinline__ void pack_chunk(const PackArgs& p, bool second, int tile, int c) {
  using B = Blk<T>;
  const void* W = second ? p.W2 : p.W;
  const int lane = threadIdx.x & 63;
  const int kb = c / B::NCH, cc = c - kb * B::NCH;
  const uint8_t* slab = (const uint8_t*)W + ((size_t)tile * p.KB + kb) * B::SLAB;
  int row = 64 * tile + lane - p.w_row0;
  if (p.W2) {
    if (row >= p.w_rows) return;          // (the other matrix's groups would follow)
    row = 2 * row - (row & 31) + (second ? 32 : 0);
  }
  Run a, b;
  B::chunk(slab, lane, cc, a, b);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const Run& r = h ? b : a;
    const int k = kb * B::QK + r.e;
    if (k >= p.K) continue;               // K % 32 == 0: a run is wholly inside or outside
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = run_value(r, i);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float w[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) w[i] = v[8 * u + i];
      store_unit<SP>(p.Wp + unit_off(row, k + 8 * u, p.KS), p.w_lo, w);
    }
  }
}

template <uint32_t T> inline constexpr bool kRowMajor = (T == 0 || T == 1 || T == 30);

// Both operands in one launch: workgroups below w_groups pack W (four chunks each, or four
// 32-row x 64-k pieces of a row-major one), the rest pack X.
template <uint32_t T, bool SP>
__global__ __launch_bounds__(256) void pack_kernel(PackArgs p) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kcs = (16 * p.KS + kRowPackK - 1) / kRowPackK;
  if ((int)blockIdx.x < p.w_groups) {
    const int job = (int)blockIdx.x * 4 + wave;
    if constexpr (kRowMajor<T>) {
      const int g = job / kcs;
      if (32 * g >= p.w_rows) return;
      constexpr size_t ES = T == 0 ? 4 : 2;
      pack_rows<T, SP && T != 30>((const uint8_t*)p.W + (size_t)p.w_row0 * p.K * ES, p.w_rows, p.K, p.KS, g,
                                  job - g * kcs, p.Wp, p.w_lo);
    } else {
      const int nch = p.KB * Blk<(int)T>::NCH;
      const int t = job / nch, nt = (p.w_rows + 63) / 64;
      const bool second = t >= nt;
      if (t >= (p.W2 ? 2 * nt : nt)) return;
      pack_chunk<(int)T, SP>(p, second, p.w_row0 / 64 + (second ? t - nt : t), job - t * nch);
    }
  } else {
    const int job = ((int)blockIdx.x - p.w_groups) * 4 + wave;
    const int g = job / kcs;
    if (32 * g >= p.x_rows) return;
    pack_rows<0, SP>(p.x, p.x_rows, p.K, p.KS, g, job - g * kcs, p.Xp, p.x_lo);
  }
}

// The GEMM. A workgroup of WM x WN waves computes BM weight rows x BN activation rows in stages of
// 32 k (two fragments deep), with NB stage buffers in LDS filled by DMA and the operands of two stages in
// registers. A wave's body for stage s, whose operands it has read: wait for its own copies of stage s + 1
// and for the workgroup (all waves have then read stage s), then multiply stage s, reading the operands of
// stage s + 1 among the first half of the MFMAs and refilling stage s's buffer with stage s + NB among
// the second. So one barrier per stage, copies that have NB - 1 stages to land, and no read that waits for
// a copy or MFMA that waits for its stage's reads.
// The activations are the A operand (rows of D): a lane then holds one weight row's column of D,
// and a store instruction writes two whole 128-byte runs of two output rows.
// SW: the SwiGLU epilogue. The weights are the A operand, so a lane holds one activation row and runs of
// four consecutive weight rows, and writes h as 8-byte halves of the next GEMM's fragment units.
template <int BM, int BN, int WM, int WN, int NB, int NP, bool SW>
__global__ __launch_bounds__(WM* WN * 64) void packed_gemm_kernel(PackedGemmArgs p) {
  constexpr int NWAVE = WM * WN, KK = 2;                        // k steps of 16 per stage
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  constexpr int PX = NP > 1 ? 2 : 1, PW = NP == 3 ? 2 : 1;      // planes
  constexpr int WQ = BM / 32 * KK * PW, XQ = BN / 32 * KK * PX;  // 1 KiB pieces per stage
  constexpr int NI = (WQ + XQ) / NWAVE;
  constexpr int SB = (WQ + XQ) * 1024;
  static_assert((WQ + XQ) % NWAVE == 0 && NB >= 2 && NB * SB <= (int)kMaxLdsBytes, "stage split");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[NB * SB];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;

  // XCD x (workgroup % 8) takes a contiguous run of tiles; tiles are ordered in bands of
  // kBand activation tiles, weight tiles outer, so the workgroups running together on one XCD
  // share both operands in its L2
  const int mt = (p.m + BM - 1) / BM, nt = (p.N + BN - 1) / BN;
  const int total = mt * nt * p.splits, per = (total + 7) / 8;
  int t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (t >= total || (int)(blockIdx.x >> 3) >= per) return;
  const int split = t / (mt * nt);
  t -= split * (mt * nt);
  constexpr int kBand = 4;
  const int band = t / (kBand * mt), bw = min(kBand, nt - band * kBand);
  t -= band * kBand * mt;
  const int mtile = t / bw, ntile = band * kBand + (t - mtile * bw);

  const int s0 = split * p.steps_per_split;
  const int ns = min(p.KS / KK - s0, p.steps_per_split);
  const __amdgpu_buffer_rsrc_t wr = make_rsrc(p.Wp, p.w_bytes);
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(p.Xp, p.x_bytes);
  // this wave's pieces of a stage: source offset of stage 0 (piece q: plane, 32-row group, k step)
  uint32_t src[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int q = wave * NI + j;
    const bool isw = q < WQ;
    const int r = isw ? q : q - WQ, n = isw ? BM / 32 * KK : BN / 32 * KK;
    const int plane = r / n, g = (r - plane * n) / KK, kk = r % KK;
    const int g0 = isw ? mtile * (BM / 32) : ntile * (BN / 32);
    src[j] = (uint32_t)plane * (isw ? p.w_lo : p.x_lo) + ((uint32_t)(g0 + g) * (uint32_t)p.KS + (uint32_t)(KK * s0 + kk)) * 1024u;
  }
  // copy j of this wave's share of stage s; a stage past the end reads past the resource: zeros, no
  // memory traffic
  auto dma = [&](int s, uint8_t* buf, int j) {
    const uint32_t vo = s < ns ? (uint32_t)lane * 16u : kQOob;
    const uint32_t so = (uint32_t)min(s, ns - 1) * (KK * 1024u);
    const int q = wave * NI + j;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(q < WQ ? wr : xr, (lds_void_t*)(buf + 1024 * q), 16, (int)vo,
                                             (int)(src[j] + so), 0, 0);
  };
  f32x16_t acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.0f;

  // a whole stage's operands
  struct Ops { bf16x8_t w[KK][PW][TM], x[KK][PX][TN]; };
  constexpr int NR1 = PW * TM + PX * TN, NR = KK * NR1;   // fragment reads per k step and stage
  constexpr int NM = KK * TM * TN * NP;                   // MFMAs per stage
  // per k step: the first planes' activations and weights, then the second planes'
  auto read = [&](const uint8_t* buf, Ops& o, int i) {
    const int kk = i / NR1, pl = i % NR1 / (TM + TN), f = i % NR1 % (TM + TN);
    if (f < TN)
      o.x[kk][pl][f] = *reinterpret_cast<const bf16x8_t*>(
          buf + (WQ + pl * (BN / 32 * KK) + KK * (wn * TN + f) + kk) * 1024 + lane * 16);
    else
      o.w[kk][pl][f - TN] = *reinterpret_cast<const bf16x8_t*>(
          buf + (pl * (BM / 32 * KK) + KK * (wm * TM + f - TN) + kk) * 1024 + lane * 16);
  };
  // MFMA i of a stage: per k step the w_hi x_hi products, then w_hi x_lo and w_lo x_hi
  auto mma = [&](const Ops& o, int i) {
    const int kk = i / (NM / KK), term = i / (TM * TN) % NP, m = i / TN % TM, n = i % TN;
    const bf16x8_t x = o.x[kk][term == 1][n], w = o.w[kk][term == 2][m];
    acc[n][m] = SW ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x, acc[n][m], 0, 0, 0)
                   : __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, w, acc[n][m], 0, 0, 0);
  };
  auto sync = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  int cur = 0;
  auto step = [&](int s, const Ops& now, Ops& then) {
    const int next = cur == (NB - 1) * SB ? 0 : cur + SB;
    wait_copies<(NB - 2) * NI>();              // stage s + 1 has landed (this wave's pieces)
    sync();                                // everyone's pieces; everyone has read stage s
    // reads among the first half of the MFMAs (the last has landed when the stage ends), copies
    // spread over the second: issued together they would queue in the address unit ahead of every
    // wave's MFMAs
    constexpr int RM = (2 * NR + NM - 1) / NM, H = NM / 2;
#pragma unroll
    for (int i = 0; i < NM; ++i) {
#pragma unroll
      for (int r = i * RM; r < (i + 1) * RM && r < NR; ++r) read(smem + next, then, r);
#pragma unroll
      for (int j = 0; j < NI; ++j)
        if (i == H + j * (NM - H) / NI) dma(s + NB, smem + cur, j);
      mma(now, i);
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = next;
  };
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) dma(i, smem + i * SB, j);
  wait_copies<(NB - 1) * NI>();
  sync();
  Ops e, o;                                // operands of even and odd stages
#pragma unroll
  for (int i = 0; i < NR; ++i) read(smem, e, i);
#pragma unroll 1
  for (int s = 0; s < ns; s += 2) {
    step(s, e, o);
    step(s + 1, o, e);                     // past the end: zeros
  }
  wait_copies<0>();                            // no copy into LDS outlives the workgroup

  if constexpr (SW) {
    static_assert(TM % 2 == 0, "whole gate / up pairs per wave");
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int x = BN * ntile + BN / WN * wn + 32 * j + (lane & 31);
      if (x >= p.N) continue;
#pragma unroll
      for (int i = 0; i < TM; i += 2) {
        const int k0 = (BM * mtile + BM / WM * wm + 32 * i) / 2;   // h columns k0 .. k0 + 31
        if (2 * k0 >= p.m) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          bf16x4_t hi, lo;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = silu_mul(acc[j][i][4 * q + e], acc[j][i + 1][4 * q + e]);
            hi[e] = (__bf16)v;
            lo[e] = (__bf16)(v - (float)hi[e]);
          }
          uint8_t* d = p.Hp + unit_off(x, k0 + 8 * q, p.KSh) + 8 * (lane >> 5);
          *reinterpret_cast<bf16x4_t*>(d) = hi;
          if constexpr (NP > 1) *reinterpret_cast<bf16x4_t*>(d + p.h_lo) = lo;
        }
      }
    }
    return;
  }
  if (p.add) {                             // (splits 1)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int w = BM * mtile + BM / WM * wm + 32 * i + (lane & 31);
        if (w >= p.m) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int x = BN * ntile + BN / WN * wn + 32 * j + 4 * (lane >> 5) + 8 * (r >> 2) + (r & 3);
          const size_t o = (size_t)x * p.ldy + w;
          if (x < p.N) p.Y[o] = p.add[o] + acc[j][i][r];
        }
      }
    return;
  }
  float* Y = p.splits > 1 ? p.partial + (size_t)split * p.split_stride : p.Y;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int x0 = BN * ntile + BN / WN * wn + 32 * j + 4 * (lane >> 5);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int w = BM * mtile + BM / WM * wm + 32 * i + (lane & 31);
      if (w >= p.m) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int x = x0 + 8 * (r >> 2) + (r & 3);
        if (x < p.N) {
          float* y = Y + (size_t)x * p.ldy + w;
          if (p.splits > 1) *y = acc[j][i][r];
          else __builtin_nontemporal_store(acc[j][i][r], y);
        }
      }
    }
  }
}

template <int BM, int BN, int WM, int WN, int NB, int NP, bool SW = false>
hipError_t launch_shape(const PackedGemmArgs& a, hipStream_t s, hipEvent_t done) {
  const int total = ((a.m + BM - 1) / BM) * ((a.N + BN - 1) / BN) * a.splits;
  const int grid = (total + 7) / 8 * 8;
  auto* k = packed_gemm_kernel<BM, BN, WM, WN, NB, NP, SW>;
  if (done) hipExtLaunchKernelGGL(k, dim3((unsigned)grid), dim3(WM * WN * 64), 0, s, nullptr, done, 0, a);
  else hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(WM * WN * 64), 0, s, a);
  return hipGetLastError();
}

template <uint32_t T>
hipError_t launch_pack_t(const PackArgs& a, unsigned grid, bool sp, hipStream_t s) {
  if (sp) hipLaunchKernelGGL((pack_kernel<T, true>), dim3(grid), dim3(256), 0, s, a);
  else hipLaunchKernelGGL((pack_kernel<T, false>), dim3(grid), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_pack(uint32_t type, PackArgs a, bool sp, hipStream_t s) {
  const long kcs = (16 * a.KS + kRowPackK - 1) / kRowPackK;
  long wjobs;
  if (type == 0 || type == 1 || type == 30) wjobs = (long)((a.w_rows + 31) / 32) * kcs;
  else wjobs = (long)((a.w_rows + 63) / 64) * a.KB * (type == T_Q4_K || type == T_Q5_K || type == T_Q6_K ? 8 : 1);
  if (a.W2) wjobs *= 2;
  const long xjobs = (long)((a.x_rows + 31) / 32) * kcs;
  a.w_groups = (int)((wjobs + 3) / 4);
  const unsigned grid = (unsigned)(a.w_groups + (xjobs + 3) / 4);
  if (grid == 0) return hipSuccess;
  switch (type) {
    case 0: return launch_pack_t<0>(a, grid, sp, s);
    case 1: return launch_pack_t<1>(a, grid, sp, s);
    case 30: return launch_pack_t<30>(a, grid, sp, s);
    case T_Q4_0: return launch_pack_t<T_Q4_0>(a, grid, sp, s);
    case T_Q5_0: return launch_pack_t<T_Q5_0>(a, grid, sp, s);
    case T_Q8_0: return launch_pack_t<T_Q8_0>(a, grid, sp, s);
    case T_Q4_K: return launch_pack_t<T_Q4_K>(a, grid, sp, s);
    case T_Q5_K: return launch_pack_t<T_Q5_K>(a, grid, sp, s);
    case T_Q6_K: return launch_pack_t<T_Q6_K>(a, grid, sp, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_packed_gemm(const PackedGemmArgs& a, PackedTile tile, int products, hipStream_t s, hipEvent_t done) {
  using T = PackedTile;
  if (a.Hp) {
    if (a.splits != 1) return hipErrorInvalidValue;
    if (products == 3) {
      if (tile == T::k256x128) return launch_shape<256, 128, 4, 2, 3, 3, true>(a, s, done);
      if (tile == T::k128x128) return launch_shape<128, 128, 2, 2, 4, 3, true>(a, s, done);
      if (tile == T::k128x64) return launch_shape<128, 64, 2, 2, 3, 3, true>(a, s, done);
    } else if (products == 1) {
      if (tile == T::k256x256) return launch_shape<256, 256, 2, 4, 4, 1, true>(a, s, done);
      if (tile == T::k128x128) return launch_shape<128, 128, 2, 2, 4, 1, true>(a, s, done);
    }
    return hipErrorInvalidValue;
  }
  if (products == 3) {
    if (tile == T::k256x128) return launch_shape<256, 128, 4, 2, 3, 3>(a, s, done);
    if (tile == T::k192x128) return launch_shape<192, 128, 2, 2, 4, 3>(a, s, done);
    if (tile == T::k128x128) return launch_shape<128, 128, 2, 2, 4, 3>(a, s, done);
    if (tile == T::k128x64) return launch_shape<128, 64, 2, 2, 3, 3>(a, s, done);
  } else if (products == 2) {
    if (tile == T::k256x128) return launch_shape<256, 128, 4, 2, 4, 2>(a, s, done);
    if (tile == T::k192x128) return launch_shape<192, 128, 2, 2, 4, 2>(a, s, done);
    if (tile == T::k128x128) return launch_shape<128, 128, 2, 2, 3, 2>(a, s, done);
    if (tile == T::k128x64) return launch_shape<128, 64, 2, 2, 4, 2>(a, s, done);
  } else if (products == 1) {
    if (tile == T::k256x256) return launch_shape<256, 256, 2, 4, 4, 1>(a, s, done);
    if (tile == T::k192x128) return launch_shape<192, 128, 2, 2, 4, 1>(a, s, done);
    if (tile == T::k128x128) return launch_shape<128, 128, 2, 2, 4, 1>(a, s, done);
  }
  return hipErrorInvalidValue;
}

PackedPlan plan_packed(int m, int rows, int K, int products, bool pairs, int splits) {
  // The fullest CU's tiles times the stages of one, at the measured time of a stage (32 k; us, on
  // 961 x 4864 x 896, 961 x 896 x 4864, 4096^3 and 2048 x 14336 x 4096), plus the bytes of the
  // outputs and, for K slices, of the partial tiles and their reduce at 4 TB/s and its launch.
  struct Shape { PackedTile t; int bm, bn; double us; };
  static const Shape bf[] = {{PackedTile::k256x256, 256, 256, 0.74}, {PackedTile::k192x128, 192, 128, 0.295},
                             {PackedTile::k128x128, 128, 128, 0.222}};
  static const Shape f32[] = {{PackedTile::k256x128, 256, 128, 0.95}, {PackedTile::k192x128, 192, 128, 0.80},
                              {PackedTile::k128x128, 128, 128, 0.55}, {PackedTile::k128x64, 128, 64, 0.36}};
  // two products: 0.62 .. 0.75 of three (0.85 for one workgroup of 128 x 128 per CU)
  static const Shape f32b[] = {{PackedTile::k256x128, 256, 128, 0.66}, {PackedTile::k192x128, 192, 128, 0.55},
                               {PackedTile::k128x128, 128, 128, 0.38}, {PackedTile::k128x64, 128, 64, 0.26}};
  const Shape* sh = products == 3 ? f32 : products == 2 ? f32b : bf;
  const int ns = products > 1 ? 4 : 3, steps = (K + 31) / 32;
  const double out_us = (double)m * rows * 4 / 4e6;
  const int first = splits ? splits : 1, last = splits ? splits : pairs ? 1 : 8;
  PackedPlan best;
  best.us = 1e30;
  for (int i = 0; i < ns; ++i) {
    if (pairs && sh[i].t == PackedTile::k192x128) continue;   // three 32-row groups per wave
    const long tiles = (long)((m + sh[i].bm - 1) / sh[i].bm) * ((rows + sh[i].bn - 1) / sh[i].bn);
    for (int sp_n = first; sp_n <= last; ++sp_n) {
      const int per = (steps + sp_n - 1) / sp_n;
      if (!splits && sp_n > 1 &&
          (per < 4 || (steps + per - 1) / per != sp_n || (double)sp_n * rows * m * 4 > (32 << 20))) continue;
      double us = (double)((tiles * sp_n + 255) / 256) * per * sh[i].us + out_us * sp_n;
      if (sp_n > 1) us += 2.0 + out_us * (sp_n + 1);
      if (us < best.us) best = {sh[i].t, sp_n, per, us};
    }
  }
  return best;
}

}  // namespace rehip
