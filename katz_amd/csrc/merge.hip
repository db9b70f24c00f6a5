// Batched LoRA merge: W_l += scale_l * up_l . down_l for many layers in ONE launch (gfx950).
//
// Katz merges an adapter into the UNet weights before a request that uses it: for each of the 722 matched linears
// `unet_state_dict[key] += cur_up @ cur_down * scale` (patch_on_lora,
// diffusers-hf/src/diffusers/pipelines/controlnet/pipeline_controlnet_sd_xl_katz.py:1730-1747; diffusers' own
// _fuse_lora, diffusers-hf/src/diffusers/models/lora.py:403-433, is the same update in fp32).  That is 722 small
// matmuls, adds and a load_state_dict; here it is one kernel over a table of layers.  The update streams every
// weight once (read + write: HBM-bound), the rank-r product is a handful of MFMA steps per 128x128 tile:
//   * grid = all 128x128 tiles of all layers; a workgroup finds its layer in the tile prefix, a lane per entry;
//   * a lane's 16-byte pieces of W are requested before all else: their way from memory is the kernel's time, and the rest lies beside it
//     (requested between the stores, 8 bytes at a time, they were 32 round trips in a row);
//   * the up tile [128, r] and the down tile [r, 128] go to LDS, 64 ranks at a time, down with its rank axis turned inside;
//   * W' = bf16(float(W) + scale * acc): fp32 accumulate, one rounding (the reference rounds the product and the
//     scaled product to half first).
// 345 MB of weights (1280 wide, five blocks), float16 operands of rank 64: 325 -> 179 us (4.0 TB/s); rank 128 439 -> 234, rank 16 278 -> 159;
// 640 wide, six blocks, rank 32: 90 -> 51.  Workgroups of 512 threads with half the rows per wave: 205 us, four of 256 to a CU spill: 280.
// Adapter operands may be bf16 or fp16 storage (Katz keeps adapters as float16 arrays in shared memory,
// load_lora_shm_multi.py:49-61): fp16 operands use the f16 MFMA, so nothing is converted on the way.
#include "kh_common.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int MG_BM = 128, MG_BN = 128, MG_THREADS = 256;
constexpr int MG_RMAX = 128;                 // largest rank
constexpr int MG_RC = 64;                    // ranks in LDS at a time: with 128 two workgroups fit a CU in place of three (rank 128: 301 us instead of 234)

struct MergeRow {       // one layer; mirrors the six 64-bit words of the table in include/katz_hip.h
  uint64_t w, up, down; // device addresses: W [N,K] bf16, up [N,r], down [r,K]
  int64_t N, K, r;
};

__host__ __device__ constexpr int mg_lds_bytes(int rp) { return ((MG_BM + MG_BN) * (rp + 8) + MG_BN / 8 * 16) * 2; }

template <bool F16>
__device__ __forceinline__ f32x4 mfma32(const u32x4 a, const u32x4 b, f32x4 c) {
  if constexpr (F16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
}

// rc_max: the most ranks in LDS at a time (a multiple of 32; sizes the LDS rows); a layer's own rank may be smaller.
template <bool F16>
__global__ __launch_bounds__(MG_THREADS, 3) void lora_merge_kernel(const MergeRow* __restrict__ table,
                                                                const int* __restrict__ tile_start, int n_layers,
                                                                const float* __restrict__ layer_scale, float scale, int rc_max) {
  extern __shared__ __align__(16) uint16_t mg_smem[];
  const int ldu = rc_max + 8;                 // sU row stride: rows 16-byte aligned, an odd multiple of 16 bytes
  uint16_t* sU = mg_smem;                     // [128][ldu]   up tile, rank axis contiguous
  uint16_t* sD = mg_smem + MG_BM * ldu;       // [128][ldu]   down tile by columns of W, rank axis contiguous; 16 more behind eight columns (banks)
  auto at = [&](int col) { return col * ldu + (col >> 3) * 16; };
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 15, lg = lane >> 4;
  // layer of this tile: the last l with tile_start[l] <= blockIdx.x (uniform over the workgroup)
  // (a lane per entry: a bisection is a chain of loads)
  int lo = 0, count = n_layers;
  const int bid = (int)blockIdx.x;
  while (count > 1) {
    const int stride = (count + 63) / 64, at = lane * stride;
    const int before = __popcll(__ballot(at < count && tile_start[lo + (at < count ? at : 0)] <= bid)) - 1;
    lo += before * stride;
    count = count - before * stride < stride ? count - before * stride : stride;
  }
  const MergeRow L = table[lo];
  const int N = (int)L.N, K = (int)L.K;
  const int r = (int)L.r;
  const int tn = (K + MG_BN - 1) / MG_BN;
  const int t = bid - tile_start[lo];
  const int m0 = (t / tn) * MG_BM, n0 = (t % tn) * MG_BN;
  if (m0 >= N) return;                        // a tile count larger than the layer's (uniform; before any barrier)
  const float s = scale * (layer_scale != nullptr ? layer_scale[lo] : 1.f);
  const uint16_t* up = reinterpret_cast<const uint16_t*>(L.up);
  const uint16_t* down = reinterpret_cast<const uint16_t*>(L.down);
  bf16_t* W = reinterpret_cast<bf16_t*>(L.w);

  // A wave owns 32 rows of the tile, a lane of it rows lr and 16 + lr, columns 32 j + 8 lg .. + 7
  const int row0 = m0 + wave * 32 + lr, col0 = n0 + lg * 8;
  const bool vec = (K & 7) == 0 && (L.w & 15) == 0, half = (K & 3) == 0 && (L.w & 7) == 0;   // pieces of 16 bytes; of 8
  u32x4 old[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      old[i][j] = vec && row0 + i * 16 < N && col0 + j * 32 < K ? *reinterpret_cast<const u32x4*>(W + (size_t)(row0 + i * 16) * K + col0 + j * 32) : u32x4{0, 0, 0, 0};

  // Operands in 16-byte pieces where the layer allows it (r % 8 == 0, K % 8 == 0, aligned bases: every linear of the UNet), else
  // element by element
  const bool fast = (L.r & 7) == 0 && (K & 7) == 0 && ((L.up | L.down) & 15) == 0;
  // Products with the row of W in the lane: fragment row m of the two tiles of 32 columns is column 8 (m / 4) + 4 tile + m % 4, so that a lane's
  // results of both are the eight columns of its piece
  f32x4 acc[2][4][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j][0] = acc[i][j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint16_t *fu = sU + (wave * 32 + lr) * ldu + lg * 8, *fd = sD + at(8 * (lr >> 2) + (lr & 3)) + lg * 8;
  for (int r0 = 0; r0 < r; r0 += rc_max) {
    const int rc = ((r - r0 < rc_max ? r - r0 : rc_max) + 31) & ~31;   // in whole MFMA steps, the excess zero-filled
    if (r0 > 0) __syncthreads();
    if (fast) {
      const int upr = rc / 8;                                   // pieces per up row
      for (int i = tid; i < MG_BM * upr; i += MG_THREADS) {
        const int row = i / upr, k = (i % upr) * 8;
        u32x4 v = u32x4{0, 0, 0, 0};
        if (m0 + row < N && r0 + k < r) v = *reinterpret_cast<const u32x4*>(up + (size_t)(m0 + row) * L.r + r0 + k);
        *reinterpret_cast<u32x4*>(sU + row * ldu + k) = v;
      }
      for (int i = tid; i < rc / 4 * (MG_BN / 8); i += MG_THREADS) {   // four ranks of eight columns
        const int k = i / (MG_BN / 8) * 4, col = (i % (MG_BN / 8)) * 8;
        u32x4 v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[e] = r0 + k + e < r && n0 + col < K ? *reinterpret_cast<const u32x4*>(down + (size_t)(r0 + k + e) * K + n0 + col) : u32x4{0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          auto one = [&](int e) { return (v[e][c >> 1] >> ((c & 1) * 16)) & 0xffffu; };
          *reinterpret_cast<u32x2*>(sD + at(col + c) + k) = u32x2{one(0) | one(1) << 16, one(2) | one(3) << 16};
        }
      }
    } else {
      for (int i = tid; i < MG_BM * rc; i += MG_THREADS) {
        const int row = i / rc, k = i % rc;
        sU[row * ldu + k] = (m0 + row < N && r0 + k < r) ? up[(size_t)(m0 + row) * L.r + r0 + k] : (uint16_t)0;
      }
      for (int i = tid; i < rc / 4 * MG_BN; i += MG_THREADS) {  // four ranks of a column
        const int k = i / MG_BN * 4, col = i % MG_BN;
        uint32_t v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = r0 + k + e < r && n0 + col < K ? down[(size_t)(r0 + k + e) * K + n0 + col] : (uint16_t)0;
        *reinterpret_cast<u32x2*>(sD + at(col) + k) = u32x2{v[0] | v[1] << 16, v[2] | v[3] << 16};
      }
    }
    __syncthreads();
    for (int k0 = 0; k0 < rc; k0 += 32) {
      const u32x4 b0 = *reinterpret_cast<const u32x4*>(fu + k0), b1 = *reinterpret_cast<const u32x4*>(fu + 16 * ldu + k0);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const u32x4 a = *reinterpret_cast<const u32x4*>(fd + at(j * 32) + h * 4 * ldu + k0);
          acc[0][j][h] = mfma32<F16>(a, b0, acc[0][j][h]);
          acc[1][j][h] = mfma32<F16>(a, b1, acc[1][j][h]);
        }
    }
  }

  // W' = bf16(W + s * acc): fp32 sum, one rounding
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = row0 + i * 16;
    if (row >= N) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = col0 + j * 32;
      auto sum = [&](float w, int e) { return w + s * acc[i][j][e >> 2][e & 3]; };
      auto sums = [&](uint32_t w, int e) { return pack_bf16x2(sum(bf16_lo(w), 2 * e), sum(bf16_hi(w), 2 * e + 1)); };
      if (vec) {
        if (col >= K) continue;
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = sums(old[i][j][e], e);
        *reinterpret_cast<u32x4*>(W + (size_t)row * K + col) = o;   // (through the L2: 182 us instead of 179)
      } else if (half) {
#pragma unroll
        for (int e = 0; e < 4; e += 2)
          if (col + 2 * e < K) {
            u32x2* w = reinterpret_cast<u32x2*>(W + (size_t)row * K + col + 2 * e);
            const u32x2 v = *w;
            *w = u32x2{sums(v[0], e), sums(v[1], e + 1)};
          }
      } else {
        bf16_t* w = W + (size_t)row * K + col;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (col + e < K) w[e] = (bf16_t)sum((float)w[e], e);
      }
    }
  }
}

}  // namespace

// See include/katz_hip.h.
KH_EXPORT int kh_lora_merge_grouped_bf16(const uint64_t* table, const int32_t* tile_start, const float* layer_scale,
                                         int64_t n_layers, int64_t total_tiles, int64_t max_rank, float scale,
                                         int operands_fp16, void* stream) {
  if (!table || !tile_start || n_layers <= 0 || total_tiles <= 0 || max_rank <= 0) return KH_ERR_INVALID_ARG;
  if (total_tiles > 0x7fffffffL || n_layers > (1 << 24) || max_rank > MG_RMAX) return KH_ERR_TOO_LARGE;
  static_assert(sizeof(MergeRow) == 6 * sizeof(uint64_t), "table row layout");
  const MergeRow* rows = reinterpret_cast<const MergeRow*>(table);
  const int rc = max_rank < MG_RC ? ((int)max_rank + 31) & ~31 : MG_RC, lds = mg_lds_bytes(rc);
  hipError_t e = operands_fp16 ? kh_allow_lds<lora_merge_kernel<true>>(mg_lds_bytes(MG_RC))
                               : kh_allow_lds<lora_merge_kernel<false>>(mg_lds_bytes(MG_RC));
  if (e != hipSuccess) return (int)e;
  if (operands_fp16)
    kh_launch(KH_TAG_LORA_MERGE, lora_merge_kernel<true>, dim3((unsigned)total_tiles), dim3(MG_THREADS), (size_t)lds,
              (hipStream_t)stream, rows, (const int*)tile_start, (int)n_layers, layer_scale, scale, rc);
  else
    kh_launch(KH_TAG_LORA_MERGE, lora_merge_kernel<false>, dim3((unsigned)total_tiles), dim3(MG_THREADS), (size_t)lds,
              (hipStream_t)stream, rows, (const int*)tile_start, (int)n_layers, layer_scale, scale, rc);
  KH_RETURN_LAST_ERROR();
}
