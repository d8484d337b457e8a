// Device split writer: the cold half of split_dense's per-layer loop
// (splitter.py:229-256) with quantize_int4 (splitter.py:81-108), producing the
// byte image of one section of cold_weights.bin in device memory.
//
// quantize_int4 per 128-element group g of a vector:
//   s = max(max|g|, 1e-8) / 7                        (fp32, correctly rounded)
//   q = clamp(round_half_even(g / s), -8, 7)         (fp32 divide, then rint)
//   nibbles: element 2k low, 2k + 1 high; scale stored as fp16 (RNE)
// Section: 16-byte header <HHIq (layer, expert, n_cold, 0), n_cold records
// of 6400 bytes, zero padding to a 4096-byte multiple.  Record: u16 nid, gate,
// up and down nibbles (2048 B each), gate/up/down scales (32 fp16 each), zero
// padding from byte 6338.
#include "capi_util.h"
#include "ffn_kernels.h"

namespace oi2 {

namespace {

constexpr int kPage = 4096;
constexpr int kHeader = 16;
constexpr int kRawRecord = kOffScales + 3 * kGroups * 2;   // 6338

struct QuantArgs {
  const float* src[3];        // gate, up, down
  int64_t row_stride[3];      // elements between consecutive source rows
  int64_t elem_stride[3];     // elements between consecutive vector elements
  const uint16_t* nids;
  const int32_t* rows;        // source row of record k
  int n;
  uint8_t* records;           // record k at records + 6400 k
};

typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// q = clamp(rint(x / s), -8, 7) as 4 bits, the quotient correctly rounded
// first.  inv = 1 / s gives x / s to within 3 ulp (1.5e-6 at |x / s| <= 7),
// which rounds to the same integer unless it lies that close to a tie; only
// then is the division made (a correctly rounded one is ~10 instructions).
// NaN and infinite operands behave in x inv as in x / s.
__device__ __forceinline__ uint32_t quant4(float x, float s, float inv) {
  float d = x * inv;
  float r = __builtin_rintf(d);
  if (__builtin_expect(fabsf(fabsf(d - r) - 0.5f) < 4e-6f, 0)) r = __builtin_rintf(__fdiv_rn(x, s));
  return (uint32_t)(int)fminf(fmaxf(r, -8.0f), 7.0f) & 0xFu;
}

__device__ __forceinline__ float group_scale(float amax) { return __fdiv_rn(fmaxf(amax, 1e-8f), 7.0f); }

// A vector whose elements are consecutive (gate and up rows): one workgroup
// per (record k, vector m).  Thread t takes elements
// 4 t .. 4 t + 3 of each 1024, so a wave's load is 1 KB in one piece and a
// group is half a wave.  (16 consecutive elements a thread made every load
// touch 64 pieces 64 bytes apart.)
__device__ __forceinline__ void quantize_row(const QuantArgs& a, int k, int m) {
  const int t = threadIdx.x;
  const float* v = a.src[m] + (int64_t)a.rows[k] * a.row_stride[m];
  f32x4 x[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) x[c] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_a4*>(v + 1024 * c + 4 * t));
  uint8_t* rec = a.records + (size_t)k * kRecBytes;
  uint16_t* out = reinterpret_cast<uint16_t*>(rec + kOffGate + m * (kH / 2)) + t;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    float amax = fmaxf(fmaxf(fabsf(x[c].x), fabsf(x[c].y)), fmaxf(fabsf(x[c].z), fabsf(x[c].w)));
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o, kWave));
    const float s = group_scale(amax), inv = __fdiv_rn(1.0f, s);
    out[256 * c] = (uint16_t)(quant4(x[c].x, s, inv) | (quant4(x[c].y, s, inv) << 4) | (quant4(x[c].z, s, inv) << 8) |
                              (quant4(x[c].w, s, inv) << 12));
    if ((t & 31) == 0)
      reinterpret_cast<uint16_t*>(rec + kOffScales + m * kGroups * 2)[8 * c + (t >> 5)] = float_to_half_bits(s);
  }
  if (m == 0) {
    if (t == 0) reinterpret_cast<uint16_t*>(rec)[0] = a.nids[k];
    if (t < (kRecBytes - kRawRecord) / 2) reinterpret_cast<uint16_t*>(rec + kRawRecord)[t] = 0;
  }
}

// Vectors whose elements are strided (the down matrix's columns): lanes are
// records, so that a load of one element reads neighbouring columns of one
// matrix row.  Workgroup: 64 records x kColGroups groups of 128 elements, wave
// w elements 32 w .. 32 w + 31 of each group; the next group's loads are in
// flight while one is quantised.  Neighbouring record tiles share the lines
// at their edges and run on one XCD.  (A workgroup per record and vector read
// 4 bytes of every line of the columns: a 10752-record section took 696 us.)
constexpr int kColGroups = 4;
__device__ __forceinline__ void quantize_cols(const QuantArgs& a, int tile, int m, int g0,
                                              float (&s_max)[2][4][kWave]) {
  const int l = lane_id(), w = threadIdx.x >> 6;
  const int k = tile * kWave + l, kc = k < a.n ? k : a.n - 1;
  const int64_t es = a.elem_stride[m];
  const float* v = a.src[m] + (int64_t)a.rows[kc] * a.row_stride[m] + (int64_t)(kGroup * g0 + 32 * w) * es;
  uint8_t* rec = a.records + (size_t)kc * kRecBytes;
  float x[2][32];
  auto load = [&](int g, float (&d)[32]) {
    const float* p = v + (int64_t)(kGroup * g) * es;
#pragma unroll
    for (int i = 0; i < 32; ++i) d[i] = p[i * es];
  };
  load(0, x[0]);
#pragma unroll
  for (int g = 0; g < kColGroups; ++g) {
    const int cur = g & 1;
    if (g + 1 < kColGroups) load(g + 1, x[cur ^ 1]);
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; ++i) amax = fmaxf(amax, fabsf(x[cur][i]));
    s_max[cur][w][l] = amax;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the next loads stay in flight
    amax = fmaxf(fmaxf(s_max[cur][0][l], s_max[cur][1][l]), fmaxf(s_max[cur][2][l], s_max[cur][3][l]));
    const float s = group_scale(amax), inv = __fdiv_rn(1.0f, s);
    u32x4 q = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 32; ++i) q[i >> 3] |= quant4(x[cur][i], s, inv) << (4 * (i & 7));
    if (k < a.n) {
      *reinterpret_cast<u32x4_a2*>(rec + kOffGate + m * (kH / 2) + (g0 + g) * (kGroup / 2) + 16 * w) = q;
      if (w == 0)
        reinterpret_cast<uint16_t*>(rec + kOffScales + m * kGroups * 2)[g0 + g] = float_to_half_bits(s);
    }
  }
  if (m == 0 && g0 == 0 && w == 0 && k < a.n) {
    reinterpret_cast<uint16_t*>(rec)[0] = a.nids[k];
    for (int i = 0; i < (kRecBytes - kRawRecord) / 2; ++i) reinterpret_cast<uint16_t*>(rec + kRawRecord)[i] = 0;
  }
}

// Header and trailing zero padding of a section with n records.
__device__ __forceinline__ void section_frame(uint8_t* section, int layer, int expert, int n, size_t body,
                                              size_t total) {
  const int t = threadIdx.x;
  if (t == 0) {
    uint32_t* h = reinterpret_cast<uint32_t*>(section);
    h[0] = (uint32_t)(layer & 0xFFFF) | ((uint32_t)(expert & 0xFFFF) << 16);
    h[1] = (uint32_t)n;
    h[2] = 0;
    h[3] = 0;
  }
  for (size_t i = body + t; i < total; i += kThreads) section[i] = 0;
}

// One launch (per kMaxRecords records): workgroup 0 frames the section, the next
// take the strided
// vectors (8 per tiles x kGroups / kColGroups each; the longest ones first),
// the rest one consecutive vector each.  Bound by memory: a 10752-record
// section reads 528 MB and writes 69 MB in 139 us, 4.3 TB/s (a large copy
// moves 4.8); in launches of their own 75 + 77 + 4 us, and 145 with the rows'
// loads not marked non-temporal.
struct SectionArgs {
  QuantArgs q;
  int rows_v[3], cols_v[3], n_rows, n_cols;   // vectors by kind
  int tiles, per;                             // 64-record tiles, and per XCD
  uint8_t* section;                           // null: framed by another launch
  int layer, expert, n;                       // n: the section's records (q.n the launch's)
  size_t body, total;
};
__global__ __launch_bounds__(kThreads) void k_quantize_section(SectionArgs a) {
  __shared__ float s_max[2][4][kWave];
  int b = blockIdx.x;
  if (b == 0) {
    if (a.section) section_frame(a.section, a.layer, a.expert, a.n, a.body, a.total);
    return;
  }
  b -= 1;
  constexpr int kParts = kGroups / kColGroups;
  const int x8 = 8 * a.per, cols = a.n_cols * kParts * x8;
  if (b < cols) {
    const int v = b / (kParts * x8), r = b - v * kParts * x8, part = r / x8, t = r - part * x8;
    // XCD t & 7 takes a run of tiles: neighbours share the lines at their edges
    const int tile = (t & 7) * a.per + (t >> 3);
    if (tile < a.tiles) quantize_cols(a.q, tile, a.cols_v[v], part * kColGroups, s_max);
    return;
  }
  b -= cols;
  quantize_row(a.q, b % a.q.n, a.rows_v[b / a.q.n]);
}

// A launch has at most 2^32 threads, which three workgroups a record would pass
// at 5.6 million records.
constexpr int kMaxRecords = 1 << 20;

size_t section_bytes(int64_t n) {
  const size_t body = kHeader + (size_t)n * kRecBytes;
  return (body + kPage - 1) / kPage * kPage;
}

}  // namespace

}  // namespace oi2

using namespace oi2;

extern "C" size_t oi2_section_bytes(int32_t n_cold) { return n_cold < 0 ? 0 : section_bytes(n_cold); }

extern "C" int oi2_quantize_section(int32_t layer, int32_t expert, int32_t n, const uint16_t* nids,
                                    const int32_t* rows, const float* gate, const float* up,
                                    const float* down, const int64_t* row_stride,
                                    const int64_t* elem_stride, uint8_t* section,
                                    size_t section_bytes_, void* stream) {
  OI2_CHECK_ARG(n >= 0, "n must be non-negative, got %d", n);
  OI2_CHECK_ARG(layer >= 0 && layer <= 0xFFFF && expert >= 0 && expert <= 0xFFFF,
                "layer and expert must fit the header's u16 fields");
  OI2_CHECK_ARG(section && (uintptr_t)section % 16 == 0, "section must be 16-byte aligned device memory");
  const size_t need = section_bytes(n);
  OI2_CHECK_ARG(section_bytes_ >= need, "section buffer of %zu bytes is smaller than the %zu required",
                section_bytes_, need);
  hipStream_t st = static_cast<hipStream_t>(stream);
  SectionArgs sa{};
  sa.section = section;
  sa.layer = layer;
  sa.expert = expert;
  sa.n = n;
  sa.body = (size_t)kHeader + (size_t)n * kRecBytes;
  sa.total = need;
  if (n > 0) {
    OI2_CHECK_ARG(nids && rows && gate && up && down && row_stride && elem_stride,
                  "nids, rows, gate, up, down and the strides are required");
    QuantArgs a{};
    a.src[0] = gate;
    a.src[1] = up;
    a.src[2] = down;
    for (int m = 0; m < 3; ++m) {
      OI2_CHECK_ARG(row_stride[m] >= 0 && elem_stride[m] >= 1, "strides must be non-negative (element: >= 1)");
      a.row_stride[m] = row_stride[m];
      a.elem_stride[m] = elem_stride[m];
    }
    for (int m = 0; m < 3; ++m) {
      if (elem_stride[m] == 1) sa.rows_v[sa.n_rows++] = m;
      else sa.cols_v[sa.n_cols++] = m;
    }
    sa.q = a;
  }
  int r0 = 0;
  do {                                         // once for an empty section, to frame it
    const int nr = n - r0 < kMaxRecords ? n - r0 : kMaxRecords;
    sa.q.n = nr;
    sa.q.nids = nids + r0;
    sa.q.rows = rows + r0;
    sa.q.records = section + kHeader + (size_t)r0 * kRecBytes;
    sa.tiles = (nr + kWave - 1) / kWave;
    sa.per = (sa.tiles + 7) / 8;
    const int grid = 1 + sa.n_cols * (kGroups / kColGroups) * 8 * sa.per + sa.n_rows * nr;
    hipLaunchKernelGGL(k_quantize_section, dim3(grid), dim3(kThreads), 0, st, sa);
    OI2_CHECK_LAUNCH();
    sa.section = nullptr;
    r0 += nr;
  } while (r0 < n);
  return OI2_OK;
}
