// K1, fp32: y = x W^T + b + ((x A_cat^T) * col_scale) B_cat^T (+ residual) on the fp32 matrix instruction (gfx950).
//
// The reference's LoRA linear (diffusers-hf/src/diffusers/models/lora.py:222-232, :451-457) in full precision: products and
// sums in fp32 (v_mfma_f32_32x32x2_f32), T = (x A_cat^T) * col_scale kept in fp32 between the two launches.
//
// Bound: the fp32 matrix rate (256 FLOP per clock and CU, 1/16 of bf16's), which the vector-ALU kernel in lora_gemm.hip (an
// FMA and two LDS reads per product) misses by a factor of 8.  Two launches: T first (32 x 32 tiles, the four waves of a
// workgroup split K), then the base GEMM with the rank columns as extra K steps -- computing T inside every column tile's
// workgroup would add R / 64 of the base FLOPs.  64 x 64 tiles, four waves of one 32 x 32 tile each: at 32 KB of LDS and 16
// accumulators per lane five workgroups share a CU, so tile counts that do not divide by 256 CUs spread evenly and the
// matrix pipe always has another wave to run; operand bytes are no issue at this rate (16 B per clock and CU).
// M 8192, N = K 640, rank 32: 84.5 us for both launches (87 TFLOP/s; a library fp32 GEMM reaches 133 here) against 465 us.
#include "kh_common.h"

namespace {

struct F32Params {
  const float *x, *w, *bias, *t, *b_cat, *res;
  float* y;
  int M, N, K, R;
};

constexpr int FB = 64;         // rows and columns of a tile
constexpr int FK = 32;         // K columns of a stage
constexpr int FLD = FK + 4;    // staged row: 144 bytes, so the 16 rows of a ds_read_b128 phase fall into distinct banks

// eight K columns of a 32-row operand panel: lane (l32, lh) holds columns 4 lh .. 4 lh + 3 of row l32, so element e of both
// operands feeds one matrix instruction (its two K columns are e and 4 + e)
__device__ __forceinline__ f32x16 mma8(const f32x4 a, const f32x4 b, f32x16 c) {
#pragma unroll
  for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], c, 0, 0, 0);
  return c;
}

// y = x W^T + t B_cat^T + bias + res.  K, R: multiples of 4.
__global__ __launch_bounds__(256, 4) void lora_gemm_f32_mfma_kernel(const F32Params p) {
  __shared__ __attribute__((aligned(16))) float sm[2][2 * FB * FLD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, lh = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;
  const int n_tiles = (p.N + FB - 1) / FB;
  const uint32_t tile = xcd_remap(blockIdx.x, gridDim.x);    // an XCD walks neighbouring tiles: its x rows stay in its L2
  const int m0 = (int)(tile / n_tiles) * FB, n0 = (int)(tile % n_tiles) * FB;
  const int K1 = (p.K + FK - 1) / FK, KT = K1 + (p.R + FK - 1) / FK;
  // this thread's four 16-byte pieces of a stage: rows r, r + 32 of x and of W, columns 4 c .. 4 c + 3
  const int r = tid >> 3, c = (tid & 7) * 4;
  int xr[2], wr[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    xr[q] = m0 + r + 32 * q < p.M ? m0 + r + 32 * q : p.M - 1;
    wr[q] = n0 + r + 32 * q < p.N ? n0 + r + 32 * q : p.N - 1;
  }
  f32x4 v[4];
  auto load = [&](int t) {
    const bool ext = t >= K1;
    const int k = (ext ? t - K1 : t) * FK + c, len = ext ? p.R : p.K;
    const float* xs = ext ? p.t : p.x;
    const float* ws = ext ? p.b_cat : p.w;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      v[q] = k < len ? *reinterpret_cast<const f32x4*>(xs + (size_t)xr[q] * len + k) : f32x4{0, 0, 0, 0};
      v[2 + q] = k < len ? *reinterpret_cast<const f32x4*>(ws + (size_t)wr[q] * len + k) : f32x4{0, 0, 0, 0};
    }
  };
  auto store = [&](float* s) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      *reinterpret_cast<f32x4*>(s + (r + 32 * q) * FLD + c) = v[q];
      *reinterpret_cast<f32x4*>(s + (FB + r + 32 * q) * FLD + c) = v[2 + q];
    }
  };
  f32x16 acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
  load(0);
  store(sm[0]);
  for (int t = 0; t < KT; ++t) {
    if (t + 1 < KT) load(t + 1);                 // in flight under the matrix instructions below
    __syncthreads();
    const float* s = sm[t & 1];
    const float* sx = s + (wm * 32 + l32) * FLD + 4 * lh;
    const float* sw = s + (FB + wn * 32 + l32) * FLD + 4 * lh;
#pragma unroll
    for (int g = 0; g < FK / 8; ++g)             // W first: a lane then holds one output row and runs of four columns
      acc = mma8(*reinterpret_cast<const f32x4*>(sw + 8 * g), *reinterpret_cast<const f32x4*>(sx + 8 * g), acc);
    if (t + 1 < KT) store(sm[(t + 1) & 1]);      // that buffer was last read before the barrier above
  }
  const int row = m0 + wm * 32 + l32;
  if (row >= p.M) return;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int col = n0 + wn * 32 + 8 * g + 4 * lh;
    f32x4 o = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    if (col + 4 <= p.N && p.N % 4 == 0) {
      if (p.bias != nullptr) o += *reinterpret_cast<const f32x4*>(p.bias + col);
      if (p.res != nullptr) o += *reinterpret_cast<const f32x4*>(p.res + (size_t)row * p.N + col);
      *reinterpret_cast<f32x4*>(p.y + (size_t)row * p.N + col) = o;
    } else {
      for (int e = 0; e < 4; ++e)
        if (col + e < p.N)
          p.y[(size_t)row * p.N + col + e] = o[e] + (p.bias ? p.bias[col + e] : 0.f) + (p.res ? p.res[(size_t)row * p.N + col + e] : 0.f);
    }
  }
}

// t = (x A_cat^T) * col_scale, 32 x 32 tiles; wave w takes the 8-column groups w, w + 4, ... of K straight from memory (x is
// read R / 32 times in all), the four partial tiles meet in LDS in a fixed order
__global__ __launch_bounds__(256) void lora_shrink_f32_kernel(const float* __restrict__ x, const float* __restrict__ a_cat,
                                                              const float* __restrict__ col_scale, float* __restrict__ t, int M, int K, int R) {
  __shared__ __attribute__((aligned(16))) f32x4 part[3][4][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, lh = lane >> 5;
  const int m0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const int xr = m0 + l32 < M ? m0 + l32 : M - 1, ar = r0 + l32 < R ? r0 + l32 : R - 1;
  const float* xs = x + (size_t)xr * K + 4 * lh;
  const float* as = a_cat + (size_t)ar * K + 4 * lh;
  f32x16 acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
  // a wave reads 32 consecutive columns at a time (whole 128-byte lines), two such blocks in flight
  const int nb = (K + 31) / 32;
  auto block = [&](int b, f32x4 (&va)[4], f32x4 (&vx)[4]) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int k = b * 32 + 8 * g;
      const bool in = k + 4 * lh < K;
      va[g] = in ? *reinterpret_cast<const f32x4*>(as + k) : f32x4{0, 0, 0, 0};
      vx[g] = in ? *reinterpret_cast<const f32x4*>(xs + k) : f32x4{0, 0, 0, 0};
    }
  };
  f32x4 va[2][4], vx[2][4];
  if (wave < nb) block(wave, va[0], vx[0]);
  for (int b = wave; b < nb; b += 8) {
    if (b + 4 < nb) block(b + 4, va[1], vx[1]);
#pragma unroll
    for (int g = 0; g < 4; ++g) acc = mma8(va[0][g], vx[0][g], acc);
    if (b + 4 < nb) {
      if (b + 8 < nb) block(b + 8, va[0], vx[0]);
#pragma unroll
      for (int g = 0; g < 4; ++g) acc = mma8(va[1][g], vx[1][g], acc);
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int g = 0; g < 4; ++g) part[wave - 1][g][lane] = f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  }
  __syncthreads();
  if (wave > 0 || m0 + l32 >= M) return;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    f32x4 o = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
#pragma unroll
    for (int s = 0; s < 3; ++s) o += part[s][g][lane];
    const int col = r0 + 8 * g + 4 * lh;
    if (col < R) *reinterpret_cast<f32x4*>(t + (size_t)(m0 + l32) * R + col) = o * *reinterpret_cast<const f32x4*>(col_scale + col);
  }
}

}  // namespace

// See include/katz_hip.h.
KH_EXPORT int kh_lora_linear_split_f32(const float* x, const float* w, const float* bias, const float* a_cat, const float* b_cat,
                                       const float* col_scale, float* t_scratch, const float* residual, float* y, int64_t M, int64_t N,
                                       int64_t K, int64_t R, void* stream) {
  if (!x || !w || !y || M <= 0 || N <= 0 || K <= 0 || R < 0) return KH_ERR_INVALID_ARG;
  if (R > 0 && (!a_cat || !b_cat || !col_scale || !t_scratch)) return KH_ERR_INVALID_ARG;
  if (K % 4 != 0 || R % 4 != 0) return KH_ERR_UNSUPPORTED;
  if (R > 128 || M > (1 << 24) || N > (1 << 24) || K > (1 << 24)) return KH_ERR_TOO_LARGE;
  if (!kh_aligned16(x) || !kh_aligned16(w) || !kh_aligned16(y) || (bias && !kh_aligned16(bias)) || (residual && !kh_aligned16(residual)) ||
      (R > 0 && (!kh_aligned16(a_cat) || !kh_aligned16(b_cat) || !kh_aligned16(col_scale) || !kh_aligned16(t_scratch))))
    return KH_ERR_ALIGNMENT;
  hipStream_t s = (hipStream_t)stream;
  const int64_t tiles = ((M + FB - 1) / FB) * ((N + FB - 1) / FB);
  if (tiles > 0x7fffffff) return KH_ERR_TOO_LARGE;
  if (R > 0) {
    kh_launch(KH_TAG_LORA_SHRINK, lora_shrink_f32_kernel, dim3((unsigned)((M + 31) / 32), (unsigned)((R + 31) / 32)), dim3(256), 0, s, x, a_cat,
              col_scale, t_scratch, (int)M, (int)K, (int)R);
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return (int)e;
  }
  const F32Params p = {x, w, bias, t_scratch, b_cat, residual, y, (int)M, (int)N, (int)K, (int)R};
  kh_launch(KH_TAG_LORA_GEMM_F32, lora_gemm_f32_mfma_kernel, dim3((unsigned)tiles), dim3(256), 0, s, p);
  KH_RETURN_LAST_ERROR();
}
