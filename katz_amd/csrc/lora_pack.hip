// The packed adapter buffers of ALL layers of a model in two launches: kh_lora_pack_bf16.
//
// Activating adapters (set_weights_and_activate_adapters, diffusers-hf/src/diffusers/utils/peft_utils.py:238-269) means, here,
// laying the active adapters of a layer out as A_cat [R,K], B_cat [N,R], col_scale [R] (katz_amd/lora.py), and for a layer behind
// a folded LayerNorm also A_cat * gamma with its two row terms.  For the 722 linears of SDXL that was some 9000 small torch
// operations (about 90 ms of host time); the bytes are 0.4 GB read and written, so a launch over all rows of all layers is bound by
// HBM and takes a fraction of a millisecond.  Two activations with the step behind each (768x768, ranks 64 + 32, then 16), with the
// one-call blocks: 181 -> 88 ms the first time a set is used, 59 where the same two sets take turns.
#include "kh_common.h"

namespace {

// rows of the device tables (64-bit words)
struct PackLayer {
  bf16_t* a;        // [R,K]
  bf16_t* a_norm;   // [R,K] = a * gamma, or null
  const bf16_t* gamma; const bf16_t* beta;
  float* ca1;       // [R] row sums of a_norm
  float* ca2;       // [R] a . beta
  bf16_t* b;        // [N,R]
  float* scale;     // [R]
  int64_t K, N, R, geglu;
  int64_t piece0, pieces;   // its slice of the piece table
};
struct PackPiece {
  const void* down;   // [rank,K]
  const void* up;     // [N,rank]
  int64_t rank, col, dtype;   // first packed column; 0 bf16, 1 fp16, 2 fp32
  int64_t mult;       // fp32 bits: the multiplier of its columns
};
static_assert(sizeof(PackLayer) == 14 * 8 && sizeof(PackPiece) == 6 * 8, "table rows");

__device__ __forceinline__ float element(const void* p, int dtype, size_t i) {
  if (dtype == 0) return (float)static_cast<const bf16_t*>(p)[i];
  if (dtype == 1) return (float)static_cast<const _Float16*>(p)[i];
  return static_cast<const float*>(p)[i];
}
// eight consecutive elements, rounded to bf16 (16-byte aligned rows only)
__device__ __forceinline__ u32x4 eight(const void* p, int dtype, size_t i) {
  if (dtype == 0) return *reinterpret_cast<const u32x4*>(static_cast<const bf16_t*>(p) + i);
  float f[8];
  if (dtype == 1) {
    typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
    const f16x8 v = *reinterpret_cast<const f16x8*>(static_cast<const _Float16*>(p) + i);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = (float)v[e];
  } else {
    const f32x4 a = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p) + i), b = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p) + i + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) { f[e] = a[e]; f[4 + e] = b[e]; }
  }
  return u32x4{pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]), pack_bf16x2(f[6], f[7])};
}

// the layer that owns row `row` of the concatenated rows: start[l] <= row < start[l + 1]
__device__ __forceinline__ int owner(const int32_t* start, int n, int row) {
  int lo = 0, hi = n;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (start[mid] <= row) lo = mid; else hi = mid;
  }
  return lo;
}

// A side: one wave per packed row of A_cat (K % 8 == 0)
__global__ __launch_bounds__(256) void lora_pack_a_kernel(const PackLayer* __restrict__ layers, const PackPiece* __restrict__ pieces,
                                                          const int32_t* __restrict__ start, int n, int rows) {
  const int row = (int)blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= rows) return;
  const int l = owner(start, n, row), r = row - start[l];
  const PackLayer L = layers[l];
  const void* src = nullptr;
  int dtype = 0;
  size_t base = 0;
  float mult = 0.f;
  for (int i = 0; i < (int)L.pieces; ++i) {
    const PackPiece p = pieces[L.piece0 + i];
    if (r >= (int)p.col && r < (int)(p.col + p.rank)) {
      src = p.down; dtype = (int)p.dtype; base = (size_t)(r - (int)p.col) * L.K; mult = __uint_as_float((uint32_t)p.mult);
    }
  }
  if (lane == 0) L.scale[r] = mult;
  double s1 = 0, s2 = 0;
  for (int k = lane * 8; k < (int)L.K; k += 512) {
    const u32x4 v = src != nullptr ? eight(src, dtype, base + k) : u32x4{0, 0, 0, 0};
    *reinterpret_cast<u32x4*>(L.a + (size_t)r * L.K + k) = v;
    if (L.a_norm != nullptr) {
      const u32x4 g = *reinterpret_cast<const u32x4*>(L.gamma + k), b = *reinterpret_cast<const u32x4*>(L.beta + k);
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[e] = pack_bf16x2(bf16_lo(v[e]) * bf16_lo(g[e]), bf16_hi(v[e]) * bf16_hi(g[e]));   // (a product of two bf16 is exact in fp32)
        s1 += (double)bf16_lo(o[e]) + (double)bf16_hi(o[e]);
        s2 += (double)(bf16_lo(v[e]) * bf16_lo(b[e])) + (double)(bf16_hi(v[e]) * bf16_hi(b[e]));
      }
      *reinterpret_cast<u32x4*>(L.a_norm + (size_t)r * L.K + k) = o;
    }
  }
  if (L.a_norm != nullptr) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) { s1 += __shfl_xor(s1, d, 64); s2 += __shfl_xor(s2, d, 64); }
    if (lane == 0) { L.ca1[r] = (float)s1; L.ca2[r] = (float)s2; }
  }
}

// B side: a thread per eight packed columns of one row of B_cat (R % 8 == 0); 256 threads cover 2048 / R rows.  Rows of a GEGLU
// projection come in blocks of 32 value rows and their 32 gate rows (katz_amd/lora.py interleave_geglu_rows).
__global__ __launch_bounds__(256) void lora_pack_b_kernel(const PackLayer* __restrict__ layers, const PackPiece* __restrict__ pieces,
                                                          const int32_t* __restrict__ start, int n) {
  const int l = owner(start, n, (int)blockIdx.x);
  const PackLayer L = layers[l];
  const int R = (int)L.R, per_row = R / 8, rows = 256 / per_row;
  const int t = threadIdx.x;
  const int row = ((int)blockIdx.x - start[l]) * rows + t / per_row, c0 = (t % per_row) * 8;
  if (t >= rows * per_row || row >= (int)L.N) return;
  int srow = row;
  if (L.geglu) srow = (row & 63) < 32 ? (row >> 6) * 32 + (row & 31) : (int)(L.N >> 1) + (row >> 6) * 32 + (row & 31);
  u32x4 v = {0, 0, 0, 0};
  for (int i = 0; i < (int)L.pieces; ++i) {
    const PackPiece p = pieces[L.piece0 + i];
    const int lo = (int)p.col, hi = (int)(p.col + p.rank), r = (int)p.rank;
    if (hi <= c0 || lo >= c0 + 8) continue;
    if (lo <= c0 && hi >= c0 + 8 && r % 8 == 0 && (c0 - lo) % 8 == 0) {
      v = eight(p.up, (int)p.dtype, (size_t)srow * r + (c0 - lo));
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int c = c0 + e;
        if (c >= lo && c < hi) {
          const uint32_t w = f32_to_bf16_bits(element(p.up, (int)p.dtype, (size_t)srow * r + (c - lo)));
          v[e >> 1] = (e & 1) ? (v[e >> 1] & 0xffffu) | (w << 16) : (v[e >> 1] & 0xffff0000u) | w;
        }
      }
    }
  }
  *reinterpret_cast<u32x4*>(L.b + (size_t)row * R + c0) = v;
}

// col_scale of many layers: table rows {address, first column, columns, fp32 bits}
__global__ __launch_bounds__(128) void lora_rescale_kernel(const int64_t* __restrict__ table) {
  const int64_t* r = table + (size_t)blockIdx.x * 4;
  float* dst = reinterpret_cast<float*>(r[0]) + r[1];
  for (int i = threadIdx.x; i < (int)r[2]; i += 128) dst[i] = __uint_as_float((uint32_t)r[3]);
}

}  // namespace

// See include/katz_hip.h.
KH_EXPORT int kh_lora_pack_bf16(const void* layers, const void* pieces, const int32_t* a_start, const int32_t* b_start, int64_t n_layers,
                                int64_t a_rows, int64_t b_blocks, void* stream) {
  if (!layers || !pieces || !a_start || !b_start || n_layers <= 0 || a_rows <= 0 || b_blocks <= 0) return KH_ERR_INVALID_ARG;
  if (a_rows > 0x7fffffff || b_blocks > 0x7fffffff || n_layers > (1 << 24)) return KH_ERR_TOO_LARGE;
  if (!kh_aligned16(layers) || !kh_aligned16(pieces)) return KH_ERR_ALIGNMENT;
  hipStream_t s = (hipStream_t)stream;
  kh_launch(KH_TAG_LORA_PACK, lora_pack_a_kernel, dim3((unsigned)((a_rows + 3) / 4)), dim3(256), 0, s, (const PackLayer*)layers,
            (const PackPiece*)pieces, a_start, (int)n_layers, (int)a_rows);
  if (const hipError_t e = hipGetLastError(); e != hipSuccess) return (int)e;
  kh_launch(KH_TAG_LORA_PACK, lora_pack_b_kernel, dim3((unsigned)b_blocks), dim3(256), 0, s, (const PackLayer*)layers, (const PackPiece*)pieces,
            b_start, (int)n_layers);
  KH_RETURN_LAST_ERROR();
}

KH_EXPORT int kh_lora_rescale(const int64_t* table, int64_t n, void* stream) {
  if (!table || n <= 0 || n > 0x7fffffff) return KH_ERR_INVALID_ARG;
  kh_launch(KH_TAG_LORA_PACK, lora_rescale_kernel, dim3((unsigned)n), dim3(128), 0, (hipStream_t)stream, table);
  KH_RETURN_LAST_ERROR();
}
