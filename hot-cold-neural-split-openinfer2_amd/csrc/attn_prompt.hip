// Grouped-query attention for prompts on gfx950's matrix cores: the
// projections and the attention of GroupedQueryAttention.forward
// (engine.py:90-125) for calls with many token rows.
//
//   k_proj       C = X W^T, fp16 rows times fp8 e4m3fn weights (widened
//                exactly to fp16), fp32 sums; epilogue q / k / v (RoPE, q to a
//                buffer, k and v into the cache) or o_proj (out and x + out)
//
// Rounded to fp16: x_n, q, k, v before and after RoPE, the attention output
// and out; everything between them is fp32.
#include "attn_kernels.h"
#include "capi_util.h"
#include "decode_util.h"
#include "ffn_kernels.h"

namespace oi2 {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kHalfHead = kHeadDim / 2;

__device__ __forceinline__ uint32_t pack_f16x2(float a, float b) {
  return (uint32_t)float_to_half_bits(a) | ((uint32_t)float_to_half_bits(b) << 16);
}

__device__ __forceinline__ h8 fp8x8_h8(uint32_t d0, uint32_t d1) {
  const h4 lo = __builtin_shufflevector(fp8x2_to_f16x2(d0, false), fp8x2_to_f16x2(d0, true), 0, 1, 2, 3);
  const h4 hi = __builtin_shufflevector(fp8x2_to_f16x2(d1, false), fp8x2_to_f16x2(d1, true), 0, 1, 2, 3);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

__device__ __forceinline__ f32x16 mfma32(h8 a, h8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// 16 bytes per lane into LDS at dst + 16 lane; the uniform part of the
// address in the scalar offset.
__device__ __forceinline__ void dma16(rsrc_t r, uint8_t* dst, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)dst, 16, voff, soff, 0, 0);
}

// ── projections ──────────────────────────────────────────────────────────────
//
// Workgroup tile: 64 WM token rows x 128 weight rows (one head), four waves
// in 2 x 2, each 32 WM rows x the 32-row B tiles {32 wn ..} and {64 + 32 wn ..}.
// v_mfma_f32_32x32x16_f16, lane l = (l % 32, h = l / 32): A[l % 32][K 8 h ..],
// B[K 8 h ..][l % 32], element j of D at row 8 (j / 4) + 4 h + j % 4, column
// l % 32.  Only the pairing of A and B along K matters, so lane half h takes
// the h-th half of each K block.
//
// Both operands go to LDS by DMA (no registers, no LDS store instructions),
// three buffers, one barrier per K block.  A DMA puts lane l's 16 bytes at
// dst + 16 l, so rows cannot be padded; instead lane l fetches the chunk that
// belongs there under swz below.
//
// What bounds it: at 512 tokens (q / k / v: 25.8 GFLOP in 31.3 us, 823
// TFLOP/s; o_proj 17.2 GFLOP in 20.4 us) the matrix cores are busy about 40 %
// of the time; a block's waves wait for its DMAs (the weights and rows come
// from beyond L2) and a grid of 192 or 256 workgroups is one round on 256
// CUs.  The single-token GEMV this replaces from 9 rows on re-read the
// weights for every 8 rows: 64 launches of 17.2 + 8.2 us at 512 tokens.
// Position of 16-byte chunk c of a row of C chunks: 256 bytes of LDS (all 64
// banks) hold 16 / C rows, and 16 consecutive rows' chunk c fall on distinct
// banks.
template <int C>
__device__ __forceinline__ int swz(int row, int c) { return c ^ ((row / (16 / C)) & (C - 1)); }

// A fragments of step st (16 K) of a staged block.
template <int WM, int KB>
__device__ __forceinline__ void proj_read_a(const uint8_t* sA, int wm, int st, h8 (&av)[WM]) {
  const int l = lane_id(), r = l & 31, h = l >> 5;
#pragma unroll
  for (int ms = 0; ms < WM; ++ms) {
    const int row = 32 * WM * wm + 32 * ms + r;
    av[ms] = *reinterpret_cast<const h8*>(sA + row * (2 * KB) + 16 * swz<KB / 8>(row, KB / 16 * h + st));
  }
}

// The fp8 weights of steps 2 p and 2 p + 1.
template <int KB>
__device__ __forceinline__ void proj_read_b(const uint8_t* sB, int wn, int p, u32x4 (&bv)[2]) {
  const int l = lane_id(), r = l & 31, h = l >> 5;
#pragma unroll
  for (int nb = 0; nb < 2; ++nb) {
    const int row = 64 * nb + 32 * wn + r;
    bv[nb] = *reinterpret_cast<const u32x4*>(sB + row * KB + 16 * swz<KB / 16>(row, KB / 32 * h + p));
  }
}

template <int WM, int KB>
__global__ __launch_bounds__(256, KB == 64 ? 2 : 1) void k_proj(ProjArgs a, int mt, int n_heads) {
  constexpr int kBM = 64 * WM;
  constexpr int kPA = kBM * KB * 2;            // bytes of an A buffer
  constexpr int kPB = kHeadDim * KB;           // bytes of a B buffer (fp8)
  constexpr int kCA = KB / 8, kCB = KB / 16;   // 16-byte chunks per row
  constexpr int kDA = WM * KB / 32, kDB = KB / 32, kDma = kDA + kDB;   // DMAs per wave and block
  __shared__ __align__(1024) uint8_t sA0[kPA], sA1[kPA], sA2[kPA];
  __shared__ __align__(1024) uint8_t sB0[kPB], sB1[kPB], sB2[kPB];
  const int b = blockIdx.x, q = b >> 3;
  const int hb = (q / mt) * 8 + (b & 7);
  if (hb >= n_heads) return;                   // the whole workgroup
  const int m0 = (q % mt) * kBM;
  const int l = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = w >> 1, wn = w & 1;
  const uint8_t* W;
  int blk;
  if (hb < a.blocks0) {
    W = a.w0;
    blk = hb;
  } else if (hb < a.blocks0 + a.blocks1) {
    W = a.w1;
    blk = hb - a.blocks0;
  } else {
    W = a.w2;
    blk = hb - a.blocks0 - a.blocks1;
  }
  // DMA i of a wave fills the 1 KB at 1024 (w + 4 i) of the A (then the B)
  // buffer; token rows past the call read zero
  const rsrc_t rx = rsrc(a.x, (uint32_t)a.rows * kH * 2);
  const rsrc_t rw = rsrc(W + (size_t)blk * kHeadDim * kH, (uint32_t)kHeadDim * kH);
  uint32_t aoff[kDA], boff[kDB];
#pragma unroll
  for (int i = 0; i < kDA; ++i) {
    const int row = 64 / kCA * (w + 4 * i) + l / kCA;
    aoff[i] = (uint32_t)(m0 + row) * (kH * 2) + 16 * swz<kCA>(row, l % kCA);
  }
#pragma unroll
  for (int i = 0; i < kDB; ++i) {
    const int row = 64 / kCB * (w + 4 * i) + l / kCB;
    boff[i] = (uint32_t)row * kH + 16 * swz<kCB>(row, l % kCB);
  }
  // DMAs [i0, i1) of block kb
  auto issue = [&](int kb, int i0, int i1, uint8_t* sA, uint8_t* sB) {
#pragma unroll
    for (int i = 0; i < kDA; ++i)
      if (i >= i0 && i < i1) dma16(rx, sA + 1024 * (w + 4 * i), aoff[i], kb * KB * 2);
#pragma unroll
    for (int i = 0; i < kDB; ++i)
      if (i + kDA >= i0 && i + kDA < i1) dma16(rw, sB + 1024 * (w + 4 * i), boff[i], kb * KB);
  };
  f32x16 acc[WM][2];
#pragma unroll
  for (int ms = 0; ms < WM; ++ms) acc[ms][0] = acc[ms][1] = f32x16{};
  constexpr int kNB = kH / KB;
  // Block kb's DMAs have landed when at most the next block's kDma are
  // outstanding; the barrier then makes every wave's visible.
  auto landed = [&]() {
    static_assert(kDma == 12 || kDma == 8 || kDma == 6 || kDma == 4, "the wait counts below");
    if constexpr (kDma == 12) asm volatile("s_waitcnt vmcnt(12) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if constexpr (kDma == 8) asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if constexpr (kDma == 6) asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if constexpr (kDma == 4) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  // Software pipeline over the steps: a step's MFMAs run while the next
  // step's A fragments come from LDS, its weights (read a step earlier still)
  // are widened and the weights of the pair of steps after it are read.
  h8 av[2][WM], bf[2][2];
  u32x4 bv[2][2];
  auto widen = [&](const u32x4 (&v)[2], int half, h8 (&o)[2]) {
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) o[nb] = fp8x8_h8(v[nb][2 * half], v[nb][2 * half + 1]);
  };
  auto mma = [&](int cur) {
#pragma unroll
    for (int ms = 0; ms < WM; ++ms)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) acc[ms][nb] = mfma32(av[cur][ms], bf[cur][nb], acc[ms][nb]);
  };
  // Block kb from cA / cB; its step 0 is in av[0], bf[0] and the weights of
  // its steps 0, 1 in bv[0].  Once the last step's A fragments are read every
  // wave is done with the block: block kb + 1 is waited for, and block kb + 3
  // may go to this block's buffers.  Its DMAs are spread kPer a step over the
  // last step and the next block's (all at once they hold the wave's issue,
  // and with it the MFMAs, for the ~770 cycles the CU takes to accept them).
  constexpr int kSt = KB / 16;   // steps of a block
  constexpr int kPer = 3;        // DMAs per step
  static_assert(kPer * (kSt - 1) >= kDma, "a block's DMAs are issued before the next wait");
  auto block = [&](int kb, uint8_t* cA, uint8_t* cB, const uint8_t* nA, const uint8_t* nB, uint8_t* pA, uint8_t* pB) {
    const int kl = kb + 2 < kNB ? kb + 2 : kNB - 1;   // past the end: an unused block again
#pragma unroll
    for (int st = 0; st < kSt; ++st) {
      const int cur = st & 1, nx = cur ^ 1, pc = (st >> 1) & 1;
      if (st < kSt - 1)
        proj_read_a<WM, KB>(cA, wm, st + 1, av[nx]);
      else
        proj_read_a<WM, KB>(nA, wm, 0, av[nx]);
      if (cur == 0 && st < kSt - 2) proj_read_b<KB>(cB, wn, st / 2 + 1, bv[pc ^ 1]);
      if (st < kSt - 2)
        issue(kl, kPer * (st + 1), kPer * (st + 2), pA, pB);
      else if (st == kSt - 1)
        issue(kb + 3 < kNB ? kb + 3 : kNB - 1, 0, kPer, cA, cB);
      widen(cur == 0 ? bv[pc] : bv[pc ^ 1], cur ^ 1, bf[nx]);
      mma(cur);
      if (cur == 0 && st < kSt - 2)
        __builtin_amdgcn_sched_group_barrier(0x100, WM + 2, 0);
      else
        __builtin_amdgcn_sched_group_barrier(0x100, WM, 0);
#pragma unroll
      for (int i = 0; i < 2 * WM; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 8 / (2 * WM), 0);
        if (i < kPer) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (st == kSt - 2) {
        landed();
        proj_read_b<KB>(nB, wn, 0, bv[pc ^ 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  issue(0, 0, kDma, sA0, sB0);
  issue(1, 0, kDma, sA1, sB1);
  landed();
  issue(2, 0, kPer, sA2, sB2);
  proj_read_a<WM, KB>(sA0, wm, 0, av[0]);
  proj_read_b<KB>(sB0, wn, 0, bv[0]);
  widen(bv[0], 0, bf[0]);
  constexpr int kEven = kNB / 3 * 3;
#pragma unroll 1
  for (int kb = 0; kb < kEven; kb += 3) {
    block(kb, sA0, sB0, sA1, sB1, sA2, sB2);
    block(kb + 1, sA1, sB1, sA2, sB2, sA0, sB0);
    block(kb + 2, sA2, sB2, sA0, sB0, sA1, sB1);
  }
  block(kEven, sA0, sB0, sA1, sB1, sA2, sB2);
  if constexpr (kNB - kEven == 2) block(kEven + 1, sA1, sB1, sA2, sB2, sA0, sB0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    // no DMA outlives the loop
  __syncthreads();

  // Epilogue through LDS, so that a thread has 8 neighbouring outputs of a
  // row (and, half a head further, their RoPE partners) and loads and stores
  // 16 bytes at a time: element by element from the accumulators, with a
  // table load, a row split and two 2-byte stores each, it took 8 us of a
  // 24 us tile.  y rounded to fp16: dims 0 .. 63 in sA0, 64 .. 127 in sA1.
  uint16_t* y0 = reinterpret_cast<uint16_t*>(sA0);
  uint16_t* y1 = reinterpret_cast<uint16_t*>(sA1);
  {
    const int j = 32 * wn + (l & 31), h = l >> 5;
#pragma unroll
    for (int ms = 0; ms < WM; ++ms)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int o = (32 * WM * wm + 32 * ms + 8 * (e >> 2) + 4 * h + (e & 3)) * kHalfHead + j;
        y0[o] = float_to_half_bits(acc[ms][0][e]);
        y1[o] = float_to_half_bits(acc[ms][1][e]);
      }
  }
  __syncthreads();
  const bool rot = hb < a.blocks0 + a.blocks1;
#pragma unroll
  for (int it = 0; it < kBM * 8 / 256; ++it) {
    const int i = threadIdx.x + 256 * it, r = i >> 3, j = 8 * (i & 7), row = m0 + r;
    if (row >= a.rows) break;
    u32x4 v0 = *reinterpret_cast<const u32x4*>(y0 + r * kHalfHead + j);
    u32x4 v1 = *reinterpret_cast<const u32x4*>(y1 + r * kHalfHead + j);
    if (a.mode == 1) {
      const size_t o = (size_t)row * kH + hb * kHeadDim + j;
      *reinterpret_cast<u32x4_a2*>(a.out + o) = v0;
      *reinterpret_cast<u32x4_a2*>(a.out + o + kHalfHead) = v1;
      if (a.residual) {
        const u32x4 r0 = *reinterpret_cast<const u32x4*>(a.residual + o);
        const u32x4 r1 = *reinterpret_cast<const u32x4*>(a.residual + o + kHalfHead);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          v0[d] = pack_f16x2(half_lo(r0[d]) + half_lo(v0[d]), half_hi(r0[d]) + half_hi(v0[d]));
          v1[d] = pack_f16x2(half_lo(r1[d]) + half_lo(v1[d]), half_hi(r1[d]) + half_hi(v1[d]));
        }
        *reinterpret_cast<u32x4_a2*>(a.x_out + o) = v0;
        *reinterpret_cast<u32x4_a2*>(a.x_out + o + kHalfHead) = v1;
      }
      continue;
    }
    const int bt = row / a.seq, t = row - bt * a.seq;
    if (rot) {
      // engine.py:150-157: cat(x1 cos - x2 sin, x1 sin + x2 cos), the tables
      // cast to fp16; products and sum in fp32, rounded once to fp16
      const f32x4_a4* pc = reinterpret_cast<const f32x4_a4*>(a.cos + (size_t)t * kHalfHead + j);
      const f32x4_a4* ps = reinterpret_cast<const f32x4_a4*>(a.sin + (size_t)t * kHalfHead + j);
      const f32x4 c[2] = {pc[0], pc[1]}, s[2] = {ps[0], ps[1]};
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        float o0[2], o1[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const float x0 = k ? half_hi(v0[d]) : half_lo(v0[d]), x1 = k ? half_hi(v1[d]) : half_lo(v1[d]);
          const float cc = round_f16(c[d >> 1][2 * (d & 1) + k]), ss = round_f16(s[d >> 1][2 * (d & 1) + k]);
          o0[k] = x0 * cc - x1 * ss;
          o1[k] = x0 * ss + x1 * cc;
        }
        v0[d] = pack_f16x2(o0[0], o0[1]);
        v1[d] = pack_f16x2(o1[0], o1[1]);
      }
    }
    uint16_t* dst;
    if (hb < a.blocks0) {
      dst = a.q + (size_t)row * a.q_width + blk * kHeadDim + j;
    } else {
      uint16_t* cache = rot ? a.k_cache : a.v_cache;
      dst = cache + (((size_t)bt * a.n_kv + blk) * a.cap + (a.past + t)) * kHeadDim + j;
    }
    *reinterpret_cast<u32x4*>(dst) = v0;
    *reinterpret_cast<u32x4*>(dst + kHalfHead) = v1;
  }
}

}  // namespace

// The tile: the smallest whose tiles fit one workgroup per CU (64 rows, else
// 128 rows, on 128-wide K blocks: three deep buffers of one workgroup fill a
// CU's LDS); past that 128 rows on 64-wide K blocks, two workgroups a CU.
// Measured, q / k / v (48 heads) and o_proj (32 heads) in us:
//   rows   64-row        128-row       128-row, 64-wide K
//   100    18.3  15.8    26.9  23.6    28.1  25.2
//   300    20.6  17.8    28.9  25.2    30.4  27.2
//   512    37.4  20.4    31.3  26.8    32.8  28.1
//   768    55.5  37.4    58.7  31.5    49.6  31.8
//   1000   66.7  43.1    64.0  34.6    57.7  37.2
void launch_proj(const ProjArgs& a, int n_heads, hipStream_t st) {
  const int cus = device_cus();
  const int mt1 = (a.rows + 63) / 64, mt2 = (a.rows + 127) / 128, n8 = (n_heads + 7) / 8 * 8;
  if (mt1 * n_heads <= cus)
    hipLaunchKernelGGL((k_proj<1, 128>), dim3(n8 * mt1), dim3(256), 0, st, a, mt1, n_heads);
  else if (mt2 * n_heads <= cus)
    hipLaunchKernelGGL((k_proj<2, 128>), dim3(n8 * mt2), dim3(256), 0, st, a, mt2, n_heads);
  else
    hipLaunchKernelGGL((k_proj<2, 64>), dim3(n8 * mt2), dim3(256), 0, st, a, mt2, n_heads);
}

}  // namespace oi2
