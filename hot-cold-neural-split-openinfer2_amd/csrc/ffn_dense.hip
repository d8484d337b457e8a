// sparse_ffn (engine.py:173-209) on dense weights, exactly as the reference
// engine calls it: the hot half as the fp16 tensors SparseFFNLayer widens its
// fp8 file to (gate/up (n_hot, H), down (H, n_hot)), the cold half as the fp32
// tensors ColdWeightStore.read_neurons returns (gate/up (n, H), down (H, n)),
// x (rows, H) fp16.  Either half may also come as fp16, bf16 or fp32.
//
//   h     = act(x G^T) * (act)(x U^T)   per half, fp32 (engine.py:163-170)
//   y     = h_hot D_hot^T + h_cold D_cold^T   fp32
//   out   = fp16(y)
//
// Two kernels for both halves together, bound by the weight stream:
//   k_dense_up   one workgroup per tile of neurons of a half: its eight waves split
//                the hidden dimension and meet in LDS, where the activation is
//                applied; h (fp32) goes to the workspace.
//   k_dense_down one workgroup per 16 outputs: the eight waves split the hot
//                neurons, then the cold ones, on the same sums and meet in LDS;
//                the only writer of its y and out.
// Up to 64 tokens a pass, in tiles of 16, each weight loaded once for all of
// them.  Products on the matrix cores: fp16 weights with the fp16 x as they
// are (16x16x32 f16, exact products), everything else in fp32 (16x16x4 f32):
// bf16 and fp32 weights, and the whole down product, whose h stays fp32.
// 13 tokens, 3584 fp16 hot and 538 fp32 cold neurons (115 MB of weights), the
// whole Python call with its cast of the fp32 y to x's type (a third launch):
// with one GEMV pass per four tokens, four launches each, 184 us, with these two
// (24 + 18) 43.
#include "capi_util.h"
#include "ffn_kernels.h"

namespace oi2 {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));

constexpr int kDThreads = 512;        // 8 waves
constexpr int kDWaves = 8;
constexpr int kDTile = 16;            // outputs and tokens per tile
constexpr int kDMaxTiles = 4;         // token tiles per pass

__device__ __forceinline__ u32x4 rload16(rsrc_t r, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
}

template <int DT>
constexpr uint32_t dsize() { return DT == OI2_DTYPE_F32 ? 4u : 2u; }

// 8 weights of dtype DT as floats.
template <int DT>
__device__ __forceinline__ void widen8(const u32x4 (&v)[dsize<DT>() / 2], float w[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if constexpr (DT == OI2_DTYPE_F32) {
      w[i] = as_f32(v[i >> 2][i & 3]);
    } else {
      const uint32_t d = v[0][i >> 1];
      const uint16_t b = (uint16_t)(i & 1 ? d >> 16 : d & 0xFFFFu);
      w[i] = DT == OI2_DTYPE_BF16 ? bf16_bits_to_float(b) : half_bits_to_float(b);
    }
  }
}

// Lane l = (t, q) = (l % 16, l / 16) of both MFMA forms: A[t][K of q],
// B[K of q][t], element e of D at row 4 q + e, column t.  Only the pairing of
// A and B along K matters, so group q takes 8 neighbouring K of each 32.
__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

struct DenseHalf {
  const void* gate;
  const void* up;
  const void* down;
  int n, dt, ldh;             // neurons, dtype, row stride of h (a multiple of 32)
  float* h;                   // (rows of the pass, ldh) fp32, zero past n
};

struct DenseArgs {
  const uint16_t* x;          // the pass's first token
  int rows;                   // tokens of the pass
  DenseHalf half[2];          // hot, cold
  int relu, both;
  float* y32;                 // may be null
  uint16_t* out;              // may be null
};

// Element (row, column) of the waves' sums of one 16 x 16 tile, added in wave
// order.
__device__ __forceinline__ float red_sum(const f32x4 (*s)[kWave], int row, int col) {
  float v = 0.0f;
#pragma unroll
  for (int w = 0; w < kDWaves; ++w) v += s[w][16 * (row >> 2) + col][row & 3];
  return v;
}

// Neurons of a gate/up tile.  16-bit weights: 16, gate and up rows in MFMAs of
// their own.  fp32 weights: 8, columns 0-7 of one MFMA their gate rows, 8-15
// their up rows; with 16 a tile took 24 us (its fp32 MFMAs and 512 KB of
// weights) and set the launch's end, and 16-bit tiles of 8 read the tokens
// twice as often (13 tokens 33 against 28 us for 3584 fp16 neurons, 64 tokens
// 78 against 62).
template <int DT>
constexpr int tile_neurons() { return DT == OI2_DTYPE_F32 ? 8 : 16; }
inline int tile_neurons_of(int dt) { return dt == OI2_DTYPE_F32 ? 8 : 16; }

// Tile `tile` of a half for NT token tiles.  Wave w takes K 512 w ..
// 512 w + 511.
template <int DT, int NT>
__device__ __forceinline__ void dense_up_tile(const DenseArgs& a, const DenseHalf& hf, int tile,
                                              f32x4 (*s_r)[kDWaves][kWave]) {
  constexpr int kN = tile_neurons<DT>(), kS = kN / 8;   // neurons, weight streams per lane
  const int l = lane_id(), t = l & 15, q = l >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // rows past n repeat the last one (their h is stored as zero)
  const size_t e0 = (size_t)min(tile * kN + t % kN, hf.n - 1) * kH + 512 * w + 8 * q;
  const uint8_t* pw[kS];
#pragma unroll
  for (int s = 0; s < kS; ++s)
    pw[s] = static_cast<const uint8_t*>((kS == 2 ? s == 0 : t < 8) ? hf.gate : hf.up) + e0 * dsize<DT>();
  const rsrc_t rx = rsrc(a.x, (uint32_t)a.rows * kH * 2);
  const uint32_t x0 = ((uint32_t)t * kH + 512 * w + 8 * q) * 2;
  f32x4 acc[kS][NT];
#pragma unroll
  for (int s = 0; s < kS; ++s)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[s][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int kB = 4;                        // 32-wide K chunks loaded together
  constexpr int kR = dsize<DT>() / 2;          // 16-byte pieces of 8 weights
#pragma unroll 1
  for (int c0 = 0; c0 < 16; c0 += kB) {
    u32x4 xv[kB][NT], wv[kB][kS][kR];
#pragma unroll
    for (int c = 0; c < kB; ++c) {
      const uint32_t k = 32 * (c0 + c);
#pragma unroll
      for (int s = 0; s < kS; ++s)
#pragma unroll
        for (int p = 0; p < kR; ++p) wv[c][s][p] = load16(pw[s] + k * dsize<DT>() + 16 * p);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) xv[c][nt] = rload16(rx, x0 + 2 * k + nt * (kDTile * kH * 2));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kB; ++c)
#pragma unroll
      for (int s = 0; s < kS; ++s)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          if constexpr (DT == OI2_DTYPE_F16) {
            acc[s][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                __builtin_bit_cast(h8, xv[c][nt]), __builtin_bit_cast(h8, wv[c][s][0]), acc[s][nt], 0, 0, 0);
          } else {
            float wf[8];
            widen8<DT>(wv[c][s], wf);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const uint32_t d = xv[c][nt][i >> 1];
              acc[s][nt] = mfma_f32(half_bits_to_float((uint16_t)(i & 1 ? d >> 16 : d & 0xFFFFu)), wf[i], acc[s][nt]);
            }
          }
        }
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    if (nt > 0) __syncthreads();               // the previous tile's sums are read
#pragma unroll
    for (int s = 0; s < kS; ++s) s_r[s][w][l] = acc[s][nt];
    __syncthreads();
    const int i = threadIdx.x, r = i / kN, n = i % kN, m = kDTile * nt + r;
    if (i < kN * kDTile && m < a.rows) {
      const float g = red_sum(s_r[0], r, n), u = kS == 2 ? red_sum(s_r[kS - 1], r, n) : red_sum(s_r[0], r, 8 + n);
      hf.h[(size_t)m * hf.ldh + tile * kN + n] = tile * kN + n < hf.n ? gated_act(g, u, a.relu, a.both) : 0.0f;
    }
  }
}

// Workgroups: the `first_tiles` tiles of the half with the wider weights
// first, then the other's.
template <int NT>
__global__ __launch_bounds__(kDThreads, NT == 4 ? 2 : 4) void k_dense_up(DenseArgs a, int first, int first_tiles) {
  __shared__ f32x4 s_r[2][kDWaves][kWave];
  int tile = blockIdx.x, hi = first;
  if (tile >= first_tiles) {
    tile -= first_tiles;
    hi = 1 - first;
  }
  const DenseHalf& hf = a.half[hi];
  if (hf.dt == OI2_DTYPE_F16) dense_up_tile<OI2_DTYPE_F16, NT>(a, hf, tile, s_r);
  else if (hf.dt == OI2_DTYPE_F32) dense_up_tile<OI2_DTYPE_F32, NT>(a, hf, tile, s_r);
  else dense_up_tile<OI2_DTYPE_BF16, NT>(a, hf, tile, s_r);
}

// acc += the pass's h times the down rows j0 + t over this wave's eighth of
// the half's 32-neuron chunks.  The rows' stride is n, any alignment.  A lane
// whose 8 neurons would pass the row's end takes the row's last 8 instead and
// drops those that are not its own: past the end lies the next row, or the
// end of the matrix, where a 16-byte load that is only partly in range reads
// all zero.
template <int DT, int NT>
__device__ __forceinline__ void dense_down_half(const DenseArgs& a, const DenseHalf& hf, int j0, f32x4 (&acc)[NT]) {
  const int l = lane_id(), t = l & 15, q = l >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_ch = hf.ldh / 32;
  const int c_lo = w * n_ch / kDWaves, c_hi = (w + 1) * n_ch / kDWaves;
  const rsrc_t rd = rsrc(hf.down, (uint32_t)((size_t)kH * hf.n * dsize<DT>()));
  const rsrc_t rh = rsrc(hf.h, (uint32_t)a.rows * hf.ldh * 4);
  const uint32_t d0 = (uint32_t)(j0 + t) * (uint32_t)hf.n;
  const uint32_t h0 = (uint32_t)t * hf.ldh * 4;
  if (hf.n < 8) {                              // element by element, in one wave
    if (w > 0) return;
    float dw[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t e = q == 0 && i < hf.n ? d0 + i : (kNoOff / dsize<DT>());
      if constexpr (DT == OI2_DTYPE_F32) {
        dw[i] = as_f32(__builtin_amdgcn_raw_buffer_load_b32(rd, 4 * e, 0, 0));
      } else {
        const uint16_t b = __builtin_amdgcn_raw_buffer_load_b16(rd, 2 * e, 0, 0);
        dw[i] = DT == OI2_DTYPE_BF16 ? bf16_bits_to_float(b) : half_bits_to_float(b);
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const uint32_t ho = q == 0 ? h0 + 4 * i + (uint32_t)nt * kDTile * hf.ldh * 4 : kNoOff;
        acc[nt] = mfma_f32(as_f32(bld4(rh, ho)), dw[i], acc[nt]);
      }
    }
    return;
  }
  constexpr int kB = NT == 1 ? 8 : NT == 2 ? 4 : 2;
  constexpr int kR = dsize<DT>() / 2;
#pragma unroll 1
  for (int c0 = c_lo; c0 < c_hi; c0 += kB) {
    u32x4 dv[kB][kR];
    u32x4 hv[kB][NT][2];
#pragma unroll
    for (int c = 0; c < kB; ++c) {
      const int k = 32 * (c0 + c) + 8 * q, kk = min(k, hf.n - 8);
      const bool in = c0 + c < c_hi && k < hf.n;
      const uint32_t od = in ? dsize<DT>() * (d0 + kk) : kNoOff;
#pragma unroll
      for (int p = 0; p < kR; ++p) dv[c][p] = rload16(rd, od + 16 * p);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const uint32_t ho = in ? h0 + 4 * kk + (uint32_t)nt * kDTile * hf.ldh * 4 : kNoOff;
        hv[c][nt][0] = rload16(rh, ho);
        hv[c][nt][1] = rload16(rh, ho + 16);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kB; ++c) {
      const int drop = 32 * (c0 + c) + 8 * q + 8 - hf.n;   // elements of the lane before
      float dw[8];
      widen8<DT>(dv[c], dw);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const bool own = i >= drop;
        const float d = own ? dw[i] : 0.0f;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const float h = as_f32(hv[c][nt][i >> 2][i & 3]);
          acc[nt] = mfma_f32(own ? h : 0.0f, d, acc[nt]);
        }
      }
    }
  }
}

template <int NT>
__global__ __launch_bounds__(kDThreads, 2) void k_dense_down(DenseArgs a) {
  __shared__ f32x4 s_y[kDWaves][kWave];
  const int l = lane_id(), w = threadIdx.x >> 6, j0 = blockIdx.x * kDTile;
  f32x4 acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const DenseHalf& hf = a.half[k];
    if (hf.n == 0) continue;
    if (hf.dt == OI2_DTYPE_F16) dense_down_half<OI2_DTYPE_F16, NT>(a, hf, j0, acc);
    else if (hf.dt == OI2_DTYPE_F32) dense_down_half<OI2_DTYPE_F32, NT>(a, hf, j0, acc);
    else dense_down_half<OI2_DTYPE_BF16, NT>(a, hf, j0, acc);
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    if (nt > 0) __syncthreads();
    s_y[w][l] = acc[nt];
    __syncthreads();
    const int i = threadIdx.x, r = i >> 4;
    if (i < 256) {
      const int m = kDTile * nt + r;
      if (m < a.rows) {
        const float y = red_sum(s_y, r, i & 15);
        const size_t o = (size_t)m * kH + j0 + (i & 15);
        if (a.y32) a.y32[o] = y;
        if (a.out) a.out[o] = float_to_half_bits(y);
      }
    }
  }
}

__global__ __launch_bounds__(256) void k_dense_zero(int rows, float* y32, uint16_t* out) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < (size_t)rows * kH) {
    if (y32) y32[i] = 0.0f;
    if (out) out[i] = 0;
  }
}

template <int NT>
void launch_pass(const DenseArgs& a, hipStream_t st) {
  auto size = [](int dt) { return dt == OI2_DTYPE_F32 ? 4 : 2; };
  const int first = a.half[1].n > 0 && size(a.half[1].dt) > size(a.half[0].dt) ? 1 : 0;
  auto tiles = [&](int k) { return a.half[k].ldh / tile_neurons_of(a.half[k].dt); };
  hipLaunchKernelGGL(k_dense_up<NT>, dim3(tiles(0) + tiles(1)), dim3(kDThreads), 0, st, a, first, tiles(first));
  hipLaunchKernelGGL(k_dense_down<NT>, dim3(kH / kDTile), dim3(kDThreads), 0, st, a);
}

int h_stride(int n) { return (n + 31) & ~31; }

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

bool dtype_ok(int dt) { return dt == OI2_DTYPE_F32 || dt == OI2_DTYPE_BF16 || dt == OI2_DTYPE_F16; }

}  // namespace
}  // namespace oi2

using namespace oi2;

extern "C" {

size_t oi2_sparse_ffn_dense_workspace_bytes(int32_t rows, int32_t n_hot, int32_t n_cold) {
  if (rows < 0 || n_hot < 0 || n_cold < 0) return 0;
  const size_t m = rows < kDTile * kDMaxTiles ? rows : kDTile * kDMaxTiles;   // tokens of a pass
  return 256 + align256(m * (size_t)h_stride(n_hot) * sizeof(float)) +
         align256(m * (size_t)h_stride(n_cold) * sizeof(float));
}

int oi2_sparse_ffn_dense(const uint16_t* x, int32_t rows, int32_t act, int32_t act_on_both,
                         int32_t n_hot, int32_t hot_dtype, const void* gate_hot, const void* up_hot,
                         const void* down_hot, int32_t n_cold, int32_t cold_dtype,
                         const void* gate_cold, const void* up_cold, const void* down_cold,
                         uint16_t* out, float* y32, void* workspace, size_t workspace_bytes,
                         void* stream) {
  clear_error();
  OI2_CHECK_ARG(rows >= 0 && n_hot >= 0 && n_cold >= 0, "negative size");
  OI2_CHECK_ARG(act == OI2_ACT_SILU || act == OI2_ACT_RELU, "act %d is not OI2_ACT_*", act);
  if (rows == 0) return OI2_OK;
  OI2_CHECK_ARG(x && (uintptr_t)x % 16 == 0, "x must be non-null and 16-byte aligned");
  OI2_CHECK_ARG(out || y32, "both outputs are null");
  OI2_CHECK_ARG(!out || (uintptr_t)out % 2 == 0, "out must be 2-byte aligned");
  // the buffer loads address each matrix with 32-bit byte offsets
  const size_t lim = (size_t)1 << 31;
  if (n_hot > 0) {
    OI2_CHECK_ARG(dtype_ok(hot_dtype), "hot_dtype %d is not OI2_DTYPE_F16, _F32 or _BF16", hot_dtype);
    OI2_CHECK_ARG(gate_hot && up_hot && down_hot, "hot weights are null");
    OI2_CHECK_ARG((uintptr_t)gate_hot % 16 == 0 && (uintptr_t)up_hot % 16 == 0,
                  "hot gate/up must be 16-byte aligned");
    OI2_CHECK_ARG((size_t)n_hot * kH * (hot_dtype == OI2_DTYPE_F32 ? 4 : 2) < lim,
                  "hot half too large (%d neurons)", n_hot);
  }
  if (n_cold > 0) {
    OI2_CHECK_ARG(dtype_ok(cold_dtype), "cold_dtype %d is not OI2_DTYPE_F16, _F32 or _BF16",
                  cold_dtype);
    OI2_CHECK_ARG(gate_cold && up_cold && down_cold, "cold weights are null");
    OI2_CHECK_ARG((uintptr_t)gate_cold % 16 == 0 && (uintptr_t)up_cold % 16 == 0,
                  "cold gate/up must be 16-byte aligned");
    OI2_CHECK_ARG((size_t)n_cold * kH * (cold_dtype == OI2_DTYPE_F32 ? 4 : 2) < lim,
                  "cold half too large (%d neurons)", n_cold);
  }
  const size_t need = oi2_sparse_ffn_dense_workspace_bytes(rows, n_hot, n_cold);
  OI2_CHECK_ARG(workspace && workspace_bytes >= need, "workspace of %zu bytes, %zu needed",
                workspace_bytes, need);
  hipStream_t st = (hipStream_t)stream;
  if (n_hot == 0 && n_cold == 0) {   // engine.py:207-208: zeros
    const size_t m = (size_t)rows * kH;
    hipLaunchKernelGGL(k_dense_zero, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, st, rows, y32, out);
    OI2_CHECK_LAUNCH();
    return OI2_OK;
  }
  uint8_t* ws = reinterpret_cast<uint8_t*>(workspace);
  const int pass = rows < kDTile * kDMaxTiles ? rows : kDTile * kDMaxTiles;
  DenseArgs a{};
  a.half[0] = {gate_hot, up_hot, down_hot, n_hot, hot_dtype, h_stride(n_hot), reinterpret_cast<float*>(ws)};
  a.half[1] = {gate_cold, up_cold, down_cold, n_cold, cold_dtype, h_stride(n_cold),
               reinterpret_cast<float*>(ws + align256((size_t)pass * h_stride(n_hot) * sizeof(float)))};
  a.relu = act == OI2_ACT_RELU;
  a.both = act_on_both ? 1 : 0;
  for (int r0 = 0; r0 < rows; r0 += pass) {
    a.x = x + (size_t)r0 * kH;
    a.rows = rows - r0 < pass ? rows - r0 : pass;
    a.y32 = y32 ? y32 + (size_t)r0 * kH : nullptr;
    a.out = out ? out + (size_t)r0 * kH : nullptr;
    if (a.rows <= kDTile) launch_pass<1>(a, st);
    else if (a.rows <= 2 * kDTile) launch_pass<2>(a, st);
    else launch_pass<4>(a, st);
    OI2_CHECK_LAUNCH();
  }
  return OI2_OK;
}

}  // extern "C"
