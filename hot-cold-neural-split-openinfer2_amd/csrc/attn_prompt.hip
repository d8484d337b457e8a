// Grouped-query attention for prompts on gfx950's matrix cores: the
// projections and the attention of GroupedQueryAttention.forward
// (engine.py:90-125) for calls with several token rows.
//
//   k_proj       C = X W^T, fp16 rows times fp8 e4m3fn weights (widened
//                exactly to fp16), fp32 sums; epilogue q / k / v (RoPE, q to a
//                buffer, k and v into the cache) or o_proj (out and x + out)
//   k_proj_few   the same for 6 to 32 rows
//   k_flash      attention of 64 query rows of a head per workgroup over the
//                cache positions they see
//
// Rounded to fp16: x_n, q, k, v before and after RoPE (rope_f16), the attention
// output and out; everything between them is fp32.
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
  if (b == 0)
    for (int i = threadIdx.x; i < a.n_counters; i += 256) a.counters[i] = 0u;
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
    const int i = threadIdx.x + 256 * it, r = i >> 3, j = 8 * (i & 7), row = a.row0 + m0 + r;
    if (m0 + r >= a.rows) break;
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
      const f32x4_a4* pc = reinterpret_cast<const f32x4_a4*>(a.cos + (size_t)t * kHalfHead + j);
      const f32x4_a4* ps = reinterpret_cast<const f32x4_a4*>(a.sin + (size_t)t * kHalfHead + j);
      const f32x4 c[2] = {pc[0], pc[1]}, s[2] = {ps[0], ps[1]};
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const f16x2 x0 = as_f16x2(v0[d]), x1 = as_f16x2(v1[d]);
        f16x2 o0, o1;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int e = 2 * (d & 1) + k;
          const RopePair o = rope_f16(x0[k], x1[k], (_Float16)c[d >> 1][e], (_Float16)s[d >> 1][e]);
          o0[k] = o.a;
          o1[k] = o.b;
        }
        v0[d] = __builtin_bit_cast(uint32_t, o0);
        v1[d] = __builtin_bit_cast(uint32_t, o1);
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

// ── projections of a few rows ────────────────────────────────────────────────
//
// At most 16 NT rows: bound by the weight stream.  Workgroup: 16 weight rows
// of a head, the eight RoPE pairs (j, j + 64) from j0 on as columns 0-7 and
// 8-15 of one 16x16x32 MFMA, its eight waves 512 K each; the waves' sums meet
// in LDS.  Lane l = (t, q) = (l % 16, l / 16) takes 16 bytes (16 K, two steps)
// of weight row t and the same 16 K of token t straight from memory: nothing
// is shared between the waves, so nothing goes through LDS before the sums.
// 8 rows: q / k / v 11.0 us (the single-token GEMV 18.2), o_proj 7.5 (9.6);
// a layer at 12 rows 30 us (k_proj's 64-row tiles: 46), at 32 rows 48 (53),
// and at 48 rows, four token tiles, 67 (61).
constexpr int kFewThreads = 512, kFewWaves = 8;

template <int NT>
__global__ __launch_bounds__(kFewThreads, 4) void k_proj_few(ProjArgs a) {
  __shared__ f32x4 s_r[kFewWaves][kWave];
  const int l = lane_id(), t = l & 15, q = l >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hb = blockIdx.x >> 3, j0 = 8 * (blockIdx.x & 7);
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < a.n_counters; i += kFewThreads) a.counters[i] = 0u;
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
  const uint8_t* pw = W + (size_t)(blk * kHeadDim + j0 + (t & 7) + kHalfHead * (t >> 3)) * kH + 512 * w + 16 * q;
  const rsrc_t rx = rsrc(a.x, (uint32_t)a.rows * kH * 2);      // rows past the call read zero
  const uint32_t x0 = ((uint32_t)t * kH + 512 * w + 16 * q) * 2;
  f32x4 acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int kB = NT == 1 ? 8 : 4;                          // 64-wide K chunks loaded together
#pragma unroll 1
  for (int c0 = 0; c0 < 8; c0 += kB) {
    u32x4 wv[kB], xv[kB][NT][2];
#pragma unroll
    for (int c = 0; c < kB; ++c) {
      wv[c] = load16_nt(pw + 64 * (c0 + c));
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int s = 0; s < 2; ++s)
          xv[c][nt][s] = bld16(rx, x0 + nt * (16 * kH * 2) + 128 * (c0 + c) + 16 * s);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kB; ++c)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const h8 b = fp8x8_h8(wv[c][2 * s], wv[c][2 * s + 1]);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, xv[c][nt][s]), b, acc[nt], 0, 0, 0);
      }
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    if (nt > 0) __syncthreads();                               // the previous sums are read
    s_r[w][l] = acc[nt];
    __syncthreads();
    // thread i < 128: row i / 8, pair i % 8
    const int r = threadIdx.x >> 3, p = threadIdx.x & 7, row = a.row0 + 16 * nt + r, j = j0 + p;
    if (r >= 16 || 16 * nt + r >= a.rows) continue;
    float y0 = 0.0f, y1 = 0.0f;
#pragma unroll
    for (int k = 0; k < kFewWaves; ++k) {
      y0 += s_r[k][16 * (r >> 2) + p][r & 3];
      y1 += s_r[k][16 * (r >> 2) + 8 + p][r & 3];
    }
    y0 = round_f16(y0);
    y1 = round_f16(y1);
    if (a.mode == 1) {
      const size_t o = (size_t)row * kH + hb * kHeadDim + j;
      a.out[o] = float_to_half_bits(y0);
      a.out[o + kHalfHead] = float_to_half_bits(y1);
      if (a.residual) {
        a.x_out[o] = float_to_half_bits(half_bits_to_float(a.residual[o]) + y0);
        a.x_out[o + kHalfHead] = float_to_half_bits(half_bits_to_float(a.residual[o + kHalfHead]) + y1);
      }
      continue;
    }
    const int bt = row / a.seq, tt = row - bt * a.seq;
    float o0 = y0, o1 = y1;
    if (hb < a.blocks0 + a.blocks1) {
      const size_t e = (size_t)tt * kHalfHead + j;
      const RopePair o = rope_f16((_Float16)y0, (_Float16)y1, (_Float16)a.cos[e], (_Float16)a.sin[e]);
      o0 = (float)o.a;
      o1 = (float)o.b;
    }
    uint16_t* dst;
    if (hb < a.blocks0) {
      dst = a.q + (size_t)row * a.q_width + blk * kHeadDim + j;
    } else {
      uint16_t* cache = hb < a.blocks0 + a.blocks1 ? a.k_cache : a.v_cache;
      dst = cache + (((size_t)bt * a.n_kv + blk) * a.cap + (a.past + tt)) * kHeadDim + j;
    }
    dst[0] = float_to_half_bits(o0);
    dst[kHalfHead] = float_to_half_bits(o1);
  }
}

// ── attention ────────────────────────────────────────────────────────────────
//
// Workgroup: 64 query rows of one head over the positions they see, 32 NK a
// tile, 2 NK waves.  Wave (qs, kv) = (w & 1, w >> 1) takes query rows 32 qs ..
// and the kv-th 32 positions of every tile with its own running max, sum and
// output (flash-style); the NK position parts meet in LDS at the end.
//
// The scores are taken transposed, S^T = K Q^T (32x32x16 MFMAs), so that a
// lane holds 16 scores of ONE query (column l % 32): max, sum and rescaling
// are per lane, one exchange with lane l ^ 32 for the max.  Element j of lane
// half h is position 8 (j / 4) + 4 h + j % 4; out^T += V^T P^T takes the
// probabilities as they lie, K step s the elements 8 s .. 8 s + 7, with the
// positions of V^T stored in that order.
//
// Probabilities stay 32-bit: p 2^10 = hi + lo in two fp16 parts (hi truncated,
// lo the rest, at least 21 bits; the 2^10 keeps lo of small p out of the
// subnormals and cancels in the division by the sum), two MFMAs per fragment.
// What both truncate is below 2^-21 p or 2^-34 (the sum keeps it): at most
// n 2^-34 of the output over n positions, and the layer's error against float64
// is the fp32 kernels' (512 rows 7.8e-4 with either).
//
// What bounds it: the chain of one tile (scores, max, probabilities, output:
// 24 MFMAs and ~200 vector instructions a wave) and, causal, the longest row
// tile's chain of tiles.  512 rows 16 us (one workgroup per query row and
// head, the single-token kernel: 134), 1300 rows 39 us (split kernel: 1078).
// Reading a tile's eight K fragments ahead of its MFMAs changed nothing.
//
// K goes to LDS by DMA; V through registers, 4 positions x 8 dims a thread,
// transposed to rows of one dim.  Both two buffers, one barrier per tile.
constexpr int kFQ = 64;                        // query rows per workgroup
constexpr float kLog2e = 1.44269504088896341f;

// Byte offset of 16-byte chunk c (8 positions) of V^T's row d.  The transposed
// stores (rows 8 apart) and the fragment reads (16 consecutive rows) both
// spread over all banks.
template <int NK>
__device__ __forceinline__ int vt_off(int d, int c) {
  if (NK == 4) return d * 256 + 16 * (c ^ (((d >> 3) ^ d) & 15));
  return (d ^ ((d >> 3) & 1)) * 128 + 16 * (c ^ (((d >> 4) ^ (d >> 1)) & 7));
}

__device__ __forceinline__ bool f16_nonfinite(uint32_t h) { return (h & 0x7C00u) == 0x7C00u; }

template <int NK>
__global__ __launch_bounds__(128 * NK, 4 / NK) void k_flash(FlashArgs a, int n_qt) {
  constexpr int kFP = 32 * NK;                 // positions per tile
  constexpr int kW = 2 * NK;                   // waves
  __shared__ __align__(1024) uint8_t sK0[kFP * 256], sK1[kFP * 256];
  __shared__ __align__(1024) uint8_t sV0[kHeadDim * kFP * 2], sV1[kHeadDim * kFP * 2];
  __shared__ float s_m[kW][32], s_l[kW][32];
  __shared__ uint32_t s_bad[3][NK];            // tile kt % 3: its positions with a non-finite v
  __shared__ uint32_t s_redo;
  const int b = blockIdx.x;
  // the four heads of blocks 8 apart share an XCD: with up to 8 kv heads they
  // are of one kv head, whose K and V its L2 then holds
  const int hq = (b & 7) * (kH / kHeadDim / 8) + ((b >> 3) & 3), rest = b >> 5;
  const int bt = rest / n_qt, q0 = (n_qt - 1 - rest % n_qt) * kFQ;   // the longest rows first
  const int g = hq / (kH / kHeadDim / a.n_kv);
  const int t = threadIdx.x, l = lane_id(), r = l & 31, h = l >> 5;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6), qs = w & 1, kv = w >> 1;
  const int n_pos = a.past + a.seq;
  const int n_see = a.causal ? min(a.past + q0 + kFQ, n_pos) : n_pos;   // positions this workgroup reads
  const int n_kt = (n_see + kFP - 1) / kFP;

  const size_t head = ((size_t)bt * a.n_kv + g) * a.cap * kHeadDim;
  const rsrc_t rk = rsrc(a.k_cache + head, (uint32_t)n_pos * 256);
  const rsrc_t rv = rsrc(a.v_cache + head, (uint32_t)n_pos * 256);
  // K DMA i: rows 4 (w + kW i) + l / 16, chunk l % 16
  uint32_t koff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 4 * (w + kW * i) + (l >> 4);
    koff[i] = (uint32_t)row * 256 + 16 * swz<16>(row, l & 15);
  }
  // V: positions 4 (t / 16) .. + 3, dims 8 (t % 16) .. + 7
  const int pg = t >> 4, dc = t & 15;
  const uint32_t voff = (uint32_t)(4 * pg) * 256 + 16 * dc;
  const int og = (pg >> 2) * 4 + (pg & 1) * 2 + ((pg >> 1) & 1);   // its 4-position group in V^T's order
  u32x4 vr[4];
  auto load_k = [&](int kt, uint8_t* sK) {
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16(rk, sK + 1024 * (w + kW * i), koff[i] + (uint32_t)kt * (kFP * 256), 0);
  };
  auto load_v = [&](int kt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) vr[i] = bld16(rv, voff + (uint32_t)kt * (kFP * 256) + 256 * i);
  };
  // whether some row of the workgroup must not see some position of tile kt
  auto masked = [&](int kt) { return a.causal && (kt + 1) * kFP > a.past + q0 + 1; };
  // A non-finite v cannot go through the products: a masked position's
  // probability is 0, and so is the low part of one that fp16 holds exactly, and
  // 0 times it would be NaN where the row does not see it, or sees infinity.  It
  // always leaves a non-finite sum, so the tiles are run without looking for it;
  // a workgroup that ends with such a sum runs them once more with `careful`.
  bool careful = false;
  auto store_v = [&](int kt, uint8_t* sV) {
    if (careful) {
      // non-finite v go in as 0, and their positions are noted and added one by
      // one to the rows that see them
      uint32_t bad = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const uint32_t x = vr[i][d];
          const uint32_t lo = f16_nonfinite(x) ? 0xFFFFu : 0u, hi = f16_nonfinite(x >> 16) ? 0xFFFF0000u : 0u;
          vr[i][d] = x & ~(lo | hi);
          if (lo | hi) bad |= 1u << i;
        }
      if (bad) atomicOr(&s_bad[kt % 3][pg >> 3], bad << (4 * (pg & 7)));
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const uint32_t x0 = vr[0][d], x1 = vr[1][d], x2 = vr[2][d], x3 = vr[3][d];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const uint32_t sel = k ? 0x07060302u : 0x05040100u;
        const int row = 8 * dc + 2 * d + k;
        *reinterpret_cast<u32x2v*>(sV + vt_off<NK>(row, og >> 1) + 8 * (og & 1)) =
            u32x2v{__builtin_amdgcn_perm(x1, x0, sel), __builtin_amdgcn_perm(x3, x2, sel)};
      }
    }
  };

  // this lane's query row, all 128 dims: B operand, K step st dims 16 st + 8 h
  const int tq = q0 + 32 * qs + r;                        // row within the sequence
  const int tc = tq < a.seq ? tq : a.seq - 1;             // rows past it repeat the last one, not stored
  const uint16_t* pq = a.q + ((size_t)bt * a.seq + tc) * kH + hq * kHeadDim + 8 * h;
  h8 qf[8];
#pragma unroll
  for (int st = 0; st < 8; ++st) qf[st] = *reinterpret_cast<const h8*>(pq + 16 * st);
  const int lim = a.causal ? a.past + tc + 1 : n_pos;     // positions this row sees
  const float sc2 = a.scale * kLog2e;
  const float ninf = -__builtin_inff();

  f32x16 o[4];
  float m, lsum;                                          // of this lane's positions; m of both halves

  auto tile = [&](int kt, const uint8_t* cK, const uint8_t* cV, uint8_t* nK, uint8_t* nV) {
    // K's DMAs (the only loads in flight) and V's stores of this tile are done
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // of the tile before, which every wave is done with; the one after the
    // next's, a barrier before its first use
    if (careful && t < NK) s_bad[(kt + 2) % 3][t] = 0;
    const bool more = kt + 1 < n_kt;
    if (more) {
      load_k(kt + 1, nK);
      load_v(kt + 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    const int p0 = kt * kFP + 32 * kv;                    // this wave's first position
    const bool live = p0 < n_see;
    if (live) {
      f32x16 s = {}, s1 = {};                             // two chains: an MFMA's result takes a while
#pragma unroll
      for (int st = 0; st < 8; ++st) {
        const int row = 32 * kv + r;
        const h8 kf = *reinterpret_cast<const h8*>(cK + row * 256 + 16 * swz<16>(row, 2 * st + h));
        if (st & 1) s1 = mfma32(kf, qf[st], s1);
        else s = mfma32(kf, qf[st], s);
      }
      s += s1;
      if (masked(kt) || p0 + 32 > n_pos) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int p = p0 + 8 * (j >> 2) + 4 * h + (j & 3);
          s[j] = p < lim ? s[j] : ninf;
        }
      }
      float cm = s[0];
#pragma unroll
      for (int j = 1; j < 16; ++j) cm = fmaxf(cm, s[j]);
      cm = fmaxf(cm, __shfl_xor(cm, 32)) * sc2;
      // The sums are taken against m, which follows the row's max only once
      // that is 2^5 above it (p 2^10 stays within fp16's range): most tiles
      // then skip the 65 products of the rescaling.
      const bool up = cm > m + 5.0f;
      if (__any(up)) {
        const float mn = up ? cm : m;
        const float alpha = m == mn ? 1.0f : __builtin_amdgcn_exp2f(m - mn);   // exp2(-inf) = 0
        lsum *= alpha;
#pragma unroll
        for (int d = 0; d < 4; ++d) o[d] *= alpha;
        m = mn;
      }
      const float ref = (m == ninf ? 0.0f : m) - 10.0f;   // p comes out times 2^10
      float p[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        p[j] = __builtin_amdgcn_exp2f(fmaf(s[j], sc2, -ref));
        lsum += p[j];
      }
      h8 ph[2], pl[2];
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        u32x4 uh, ul;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float e0 = p[8 * s2 + 2 * k], e1 = p[8 * s2 + 2 * k + 1];
          const uint32_t hi = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(e0, e1));
          uh[k] = hi;
          ul[k] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(fmaf(half_lo(hi), -1.0f, e0), fmaf(half_hi(hi), -1.0f, e1)));
        }
        ph[s2] = __builtin_bit_cast(h8, uh);
        pl[s2] = __builtin_bit_cast(h8, ul);
      }
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const int row = 32 * d + r;
          const h8 vf = *reinterpret_cast<const h8*>(cV + vt_off<NK>(row, 4 * kv + 2 * s2 + h));
          o[d] = mfma32(vf, ph[s2], o[d]);
          o[d] = mfma32(vf, pl[s2], o[d]);
        }
      if (careful) {
        uint32_t bad = s_bad[kt % 3][kv];
        while (bad) {
          const int pos = __builtin_ctz(bad);             // of this wave's 32
          bad &= bad - 1;
          const int jj = 4 * (pos >> 3) + (pos & 3), hh = (pos >> 2) & 1;
          float pv = 0.0f;
#pragma unroll
          for (int j = 0; j < 16; ++j) pv = j == jj ? p[j] : pv;
          pv = __shfl(pv, r + 32 * hh);
          const uint16_t* v = a.v_cache + head + (size_t)(p0 + pos) * kHeadDim;
#pragma unroll
          for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int j = 0; j < 16; ++j) {
              const uint16_t x = v[32 * d + 8 * (j >> 2) + 4 * h + (j & 3)];
              if (p0 + pos < lim && f16_nonfinite(x)) o[d][j] = fmaf(pv, half_bits_to_float(x), o[d][j]);
            }
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more) store_v(kt + 1, nV);
  };
  if (t == 0) s_redo = 0u;                                // set after the first tile's barrier at the earliest
#pragma unroll 1
  for (;;) {
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] = f32x16{};
    m = ninf;
    lsum = 0.0f;
    load_k(0, sK0);
    load_v(0);
    if (careful) {
      if (t < 2 * NK) s_bad[t / NK][t % NK] = 0;
      __syncthreads();
    }
    store_v(0, sV0);
#pragma unroll 1
    for (int kt = 0; kt < n_kt; kt += 2) {
      tile(kt, sK0, sV0, sK1, sV1);
      if (kt + 1 < n_kt) tile(kt + 1, sK1, sV1, sK0, sV0);
    }
    if (!careful) {
      float z = 0.0f;                                     // NaN once a sum is not finite
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int j = 0; j < 16; ++j) z = fmaf(o[d][j], 0.0f, z);
      if (__any(z != z) && l == 0) s_redo = 1u;
    }
    __syncthreads();                                      // the tiles are no longer read
    if (careful || s_redo == 0u) break;
    careful = true;
  }
  lsum += __shfl_xor(lsum, 32);                           // of the wave's positions
  // wave (qs, kv) finishes dims kOut kv .. of its rows: every wave leaves its
  // sums of each wave's dims in that wave's buffer (a wave with no position
  // has m = -inf)
  constexpr int kD = 4 / NK, kOut = 32 * kD;   // 32-dim tiles, dims per finishing wave
  float* xch[4] = {reinterpret_cast<float*>(sK0), reinterpret_cast<float*>(sK1), reinterpret_cast<float*>(sV0),
                   reinterpret_cast<float*>(sV1)};        // by dim tile: [qs][source kv][16 values][64 lanes]
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int j = 0; j < 16; ++j) xch[d][((qs * NK + kv) * 16 + j) * 64 + l] = o[d][j];
  if (h == 0) {
    s_m[w][r] = m;
    s_l[w][r] = lsum;
  }
  __syncthreads();
  float M = ninf, L = 0.0f, e[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k) M = fmaxf(M, s_m[qs + 2 * k][r]);
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    const float mk = s_m[qs + 2 * k][r];
    e[k] = mk == ninf ? 0.0f : __builtin_amdgcn_exp2f(mk - M);
    L = fmaf(e[k], s_l[qs + 2 * k][r], L);
  }
  const float inv = 1.0f / L;
  if (tq < a.seq) {
    uint16_t* po = a.out + ((size_t)bt * a.seq + tq) * kH + hq * kHeadDim + kOut * kv;
#pragma unroll
    for (int dd = 0; dd < kD; ++dd) {
      const int d = kD * kv + dd;
      const float* mine = reinterpret_cast<const float*>(d < 2 ? (d ? sK1 : sK0) : (d == 2 ? sV0 : sV1));
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = 4 * q4 + i;
          v[i] = 0.0f;
#pragma unroll
          for (int k = 0; k < NK; ++k) v[i] = fmaf(e[k], mine[((qs * NK + k) * 16 + j) * 64 + l], v[i]);
          v[i] *= inv;
        }
        *reinterpret_cast<u32x2v*>(po + 32 * dd + 8 * q4 + 4 * h) =
            u32x2v{pack_f16x2(v[0], v[1]), pack_f16x2(v[2], v[3])};
      }
    }
  }
}

}  // namespace

// Up to 32 rows (16 with 96 heads, whose 768 workgroups of two token tiles take
// longer: a layer at 32 rows 105 against 92 us) k_proj_few.  From there the
// smallest tile whose tiles fit one workgroup per CU (64 rows, else 128 rows,
// on 128-wide K blocks: three deep buffers of one workgroup fill a CU's LDS);
// past that 128 rows on 64-wide K blocks, two workgroups a CU.
// Measured, q / k / v (48 heads) and o_proj (32 heads) in us:
//   rows   64-row        128-row       128-row, 64-wide K
//   100    18.3  15.8    26.9  23.6    28.1  25.2
//   300    20.6  17.8    28.9  25.2    30.4  27.2
//   512    37.4  20.4    31.3  26.8    32.8  28.1
//   768    55.5  37.4    58.7  31.5    49.6  31.8
//   1000   66.7  43.1    64.0  34.6    57.7  37.2
static_assert(kH == 4096, "kProjMaxRows");
void launch_proj(const ProjArgs& a, int n_heads, hipStream_t st) {
  if (a.rows <= 16 || (a.rows <= 32 && n_heads <= 64)) {
    if (a.rows <= 16) hipLaunchKernelGGL(k_proj_few<1>, dim3(8 * n_heads), dim3(kFewThreads), 0, st, a);
    else hipLaunchKernelGGL(k_proj_few<2>, dim3(8 * n_heads), dim3(kFewThreads), 0, st, a);
    return;
  }
  const int cus = device_cus();
  const int mt1 = (a.rows + 63) / 64, mt2 = (a.rows + 127) / 128, n8 = (n_heads + 7) / 8 * 8;
  if (mt1 * n_heads <= cus)
    hipLaunchKernelGGL((k_proj<1, 128>), dim3(n8 * mt1), dim3(256), 0, st, a, mt1, n_heads);
  else if (mt2 * n_heads <= cus)
    hipLaunchKernelGGL((k_proj<2, 128>), dim3(n8 * mt2), dim3(256), 0, st, a, mt2, n_heads);
  else
    hipLaunchKernelGGL((k_proj<2, 64>), dim3(n8 * mt2), dim3(256), 0, st, a, mt2, n_heads);
}

// Four position parts (eight waves, 128 positions a tile) while every
// workgroup has a CU to itself, else two (two workgroups a CU): 1300 rows, 672
// workgroups, 38.6 against 49.1 us; 9 rows over 4000 positions, 32 workgroups,
// the layer 90 against 110 us.
void launch_flash(const FlashArgs& a, hipStream_t st) {
  const int n_qt = (a.seq + kFQ - 1) / kFQ, wgs = kH / kHeadDim * n_qt * a.batch;
  if (wgs <= device_cus())
    hipLaunchKernelGGL(k_flash<4>, dim3(wgs), dim3(512), 0, st, a, n_qt);
  else
    hipLaunchKernelGGL(k_flash<2>, dim3(wgs), dim3(256), 0, st, a, n_qt);
}

}  // namespace oi2
