// K2, one launch: segmented multi-adapter LoRA delta  y[rows, :] += scale_a * bf16(x[rows, :] . A_a^T) . B_a^T  per request
// segment (rows [seg_start[s], seg_start[s+1]) use adapter seg_adapter[s], negative: none) for gfx950.
//
// The per-request form of the reference's LoRA linear (diffusers-hf/src/diffusers/models/lora.py:222-232, :451-457)
// with y already holding the base projection; the reference has no batched heterogeneous-adapter path.  Same arithmetic
// as kh_sgmv_shrink_bf16 followed by kh_sgmv_expand_bf16 (t rounded to bf16 between the two products, the product
// rounded to bf16 before it is added to y), but t never leaves the workgroup: one launch instead of two and no round
// trip of t through memory.  Bound: HBM (x read once, y read and written once; the adapter matrices come from L2).
//
// A workgroup (8 waves) owns BM = 64 or 128 rows of one segment.
//   phase 1: T[BM, RA] = x_tile . A_a^T over K in 64-column stages (a ring of buffer-addressed LDS DMA); RA = 64 where the adapter's rank
//            allows, else 128.  T is rounded to bf16 and written to LDS in the stage layout, so that
//   phase 2: for every 128-column tile of y:  acc = T . B_a[tile]^T  (K = the adapter's padded rank, one or two stages of
//            B from L2, requested while the previous tile is being finished), times the adapter's scale, rounded, transposed through
//            LDS and added to the y pieces, which were requested five tiles ahead (128 rows: one).
// What bounds it at a request's sizes is not HBM's rate but the chain of latencies -- segment table, 20 stages, 5 .. 10 tiles -- in workgroups
// that are one to a CU.  Hence as many stages under way as 128 KB hold (seven of 16 KB instead of two of 32: with 128 rows and all 128 rank rows
// a stage took 0.45 us), the y pieces of the first five tiles (128 rows: of the first) requested while phase 1 runs, and 64-row blocks while they fit one
// round of the 256 CUs, so that fewer of them repeat phase 1 for other columns.
// 8 requests of 256 .. 1024 rows at 1280 -> 1280, ranks 8 .. 128: 24.9 -> 19.8 us.
// Rows / columns of A_a / B_a beyond the adapter's rank are zero by contract, so the padded rank only saves work.
// Batches with few row blocks deal the column tiles of y to several workgroups, each of which repeats
// phase 1 for its rows: x is then read from L2 more than once, which such small batches do not notice.
// Grouped form (kh_sgmv_fused_grouped_bf16): several layers that read the same x with the same segments (the to_k / to_v
// projections of every cross-attention read the one text context) in one launch, blockIdx.z = (layer, column range),
// per-layer A / B / y from a device table: 77-row requests give a single layer's launch a few microseconds of traffic,
// 120 layers fill the chip.
#include "kh_common.h"
#include <type_traits>

namespace {

typedef __attribute__((address_space(3))) void* lptr_t;
typedef __amdgpu_buffer_rsrc_t rsrc_t;

template <int VM, int LGKM>
__device__ __forceinline__ void wait_cnt() {  // gfx9 encoding: vmcnt = [15:14|3:0], expcnt = [6:4], lgkmcnt = [11:8]
  __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | ((LGKM & 15) << 8) | ((VM >> 4) << 14));
}

struct FusedParams {
  const bf16_t* x; const bf16_t* a_all; const bf16_t* b_all; bf16_t* y;
  const int* seg_start; const int* seg_adapter; const int* adapter_rank; const float* adapter_scale;
  int K, N, RP;
  int tiles_per_z;   // 128-column tiles of y per workgroup: blockIdx.z selects the range (T is recomputed per range)
  int z_per_layer;   // column ranges per layer (grid.z = layers x z_per_layer)
  const uint64_t* table;   // grouped form: rows {a_all, b_all, y} of device pointers, one per layer; null: the fields above
};

constexpr int RING = 128 * 1024;                  // phase 1's stages; phase 2: T, then two buffers of a B tile
constexpr int B_TILE = 2 * 128 * 128;             // 128 y columns x 128 rank columns, as two 64-column stages
constexpr int C_OFF = RING;                       // staging of 64 output rows x (128 + 8) columns
constexpr int LDC = 128 + 8;
constexpr int LDS_BYTES = C_OFF + 64 * LDC * 2;
static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");

template <int BM>
__global__ __launch_bounds__(512, 2) void sgmv_fused_kernel(const FusedParams p) {
#if __HIP_DEVICE_COMPILE__   // the host pass only needs the kernel's symbol (it cannot lower the buffer-resource type)
  constexpr int TI = BM / 64, T_BYTES = 2 * BM * 128;   // a wave's 32-row tiles; T as two 64-column stages of 128-byte rows
  // tiles whose y pieces are under way or here.  128 rows: those of the second tile would only be in the way of phase 1's short ring (8 x 4096 rows
  // at 640 33.1 -> 32.3 us without them, rank 64 29.9 -> 29.3, at 1280 55.9 -> 53.9)
  constexpr int YD = BM == 64 ? 5 : 1;
  static_assert(T_BYTES + 2 * B_TILE <= RING, "T and the B buffers lie in the ring");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int seg = blockIdx.y;
  const int r0 = p.seg_start[seg], r1 = p.seg_start[seg + 1], ad = p.seg_adapter[seg];
  const int m0 = blockIdx.x * BM;
  if (ad < 0 || m0 >= r1 - r0) return;            // uniform over the workgroup
  const int M = r1 - r0;                          // rows of this segment
  const int rank = p.adapter_rank[ad];            // multiple of 32, <= RP
  const float scale = p.adapter_scale[ad];
  const int K = p.K, N = p.N, RP = p.RP;
  const int layer = (int)blockIdx.z / p.z_per_layer, zz = (int)blockIdx.z % p.z_per_layer;
  const bf16_t* a_all = p.a_all; const bf16_t* b_all = p.b_all; bf16_t* y_all = p.y;
  if (p.table != nullptr) {
    const uint64_t* row = p.table + (size_t)layer * 3;
    a_all = reinterpret_cast<const bf16_t*>(row[0]); b_all = reinterpret_cast<const bf16_t*>(row[1]); y_all = reinterpret_cast<bf16_t*>(row[2]);
  }
  const bf16_t* x = p.x + (size_t)r0 * K;
  bf16_t* y = y_all + (size_t)r0 * N;
  const bf16_t* A = a_all + (size_t)ad * RP * K;
  const bf16_t* B = b_all + (size_t)ad * N * RP;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;        // 2 x 4 waves: a wave owns BM / 2 rows x 32 columns of a BM x 128 tile
  const int l32 = lane & 31, lh = lane >> 5;
  const int sw = (l32 >> 1) & 7;

  auto clamp32 = [](size_t bytes) { return (int)(uint32_t)(bytes < 0xFFFFFFFFull ? bytes : 0xFFFFFFFFull); };
  auto mk = [&](const bf16_t* base, size_t bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(base), 0, clamp32(bytes), 0x00020000); };

  // ---- phase 2's requests: B tile j; the y pieces of tile j (those of the first tiles go out while phase 1 runs) ----
  const int j0 = zz * p.tiles_per_z;
  const int n_tiles = (N / 128 - j0) < p.tiles_per_z ? (N / 128 - j0) : p.tiles_per_z;   // tiles j0 .. j0 + n_tiles - 1
  const int ks_total = rank / 16;                 // MFMA steps over the padded rank (2, 4, 6 or 8)
  const int nstage = (rank + 63) / 64;            // B stages per tile (1 or 2)
  // B tile j: rows n0 .. n0+127 of B (row stride RP), 64 rank columns per stage; 16 units of 8 rows x 128 bytes per stage, two per wave
  const rsrc_t rs_b = mk(B, (size_t)N * RP * 2);
  uint32_t vb[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int r = (wave * 2 + q) * 8 + (lane >> 3);
    vb[q] = (uint32_t)r * (uint32_t)RP * 2u + (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
  }
  constexpr int CPR = 16, ECH = 64 * CPR / 512;   // 16-byte pieces per staged row; per thread and 64-row pass: 2
  u32x4 yr[YD][TI][ECH];                          // this thread's y pieces
  // (the first stage of the first B tile goes out ahead of phase 1, into the staging tile)
  auto b_stage = [&](int j, int s) { return j == 0 && s == 0 ? smem + C_OFF : smem + T_BYTES + (j & 1) * B_TILE + s * (128 * 128); };
  auto tile_row = [&](int ps, int srow) { return m0 + (TI == 2 ? (srow >> 5) * 64 + ps * 32 + (srow & 31) : srow); };   // of a pass's staged row
  auto issue_b = [&](int j, int s) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_b, (lptr_t)(b_stage(j, s) + (wave * 2 + q) * 1024), 16, vb[q] + s * 128, (j0 + j) * 128 * RP * 2, 0, 0);
  };
  auto issue_y = [&](int j, u32x4 (&d)[TI][ECH]) {
#pragma unroll
    for (int ps = 0; ps < TI; ++ps)
#pragma unroll
      for (int q = 0; q < ECH; ++q) {
        const int c = tid + q * 512, srow = c / CPR, ch = c % CPR;
        int grow = tile_row(ps, srow);
        grow = grow < M ? grow : M - 1;
        d[ps][q] = *reinterpret_cast<const u32x4*>(y + (size_t)grow * N + (j0 + j) * 128 + ch * 8);
      }
  };

  // ---- phase 1: T = x_tile . A^T ----
  // DMA units of 8 rows x 128 bytes: TI of x and one or two of A per wave and stage; a lane's byte offset (row, swizzled piece)
  // never changes, the K tile is a scalar offset
  const rsrc_t rs_x = mk(x + (size_t)m0 * K, (size_t)(M - m0) * K * 2);
  const rsrc_t rs_a = mk(A, (size_t)RP * K * 2);
  uint32_t vx[TI], va[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int r = (wave + 8 * q) * 8 + (lane >> 3);
    const uint32_t pcb = (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
    if (q < TI) {
      int row = m0 + r; row = row < M ? row : M - 1;
      vx[q < TI ? q : 0] = (uint32_t)(row - m0) * (uint32_t)K * 2u + pcb;
    }
    va[q] = r < rank ? (uint32_t)r * (uint32_t)K * 2u + pcb : 0xFFFFFFFFu;   // (rows beyond the rank: zeros, not read from memory)
  }
  // fragments of a 64-column stage: rows (wm * BM / 2 + i * 32 + l32) of the first operand, (wn * 32 + l32) of the second
  struct Fr { bf16x8 a[4][TI]; bf16x8 b[4]; };
  auto read_frags = [&](const char* st_a, const char* st_b, Fr& f) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int po = ((2 * ks + lh) ^ sw) * 16;
#pragma unroll
      for (int i = 0; i < TI; ++i) f.a[ks][i] = *reinterpret_cast<const bf16x8*>(st_a + (wm * (BM / 2) + i * 32 + l32) * 128 + po);
      f.b[ks] = *reinterpret_cast<const bf16x8*>(st_b + (wn * 32 + l32) * 128 + po);
    }
  };
  f32x16 acc[TI];
  auto zero_acc = [&]() {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][v] = 0.f;
  };
  auto mma = [&](const Fr& f, int ks_n) {   // the first ks_n 16-column steps of the stage
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      if (ks < ks_n) {
#pragma unroll
        for (int i = 0; i < TI; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[ks][i], f.b[ks], acc[i], 0, 0, 0);
      }
  };
  const int KT = K / 64;
  zero_acc();
  Fr f;
  auto shrink = [&](auto au) {                    // au: A units per wave
    constexpr int AU = decltype(au)::value, STAGE = (BM + AU * 64) * 128, NST = RING / STAGE, PD = NST - 1, CNT = TI + AU;
    const bool mine = wn * 32 < AU * 64;          // (waves whose rank columns lie beyond RA only move operands)
    auto issue1 = [&](int t, int st) {
      const int so = t * 128;
#pragma unroll
      for (int q = 0; q < TI; ++q) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_x, (lptr_t)(smem + st + (wave + 8 * q) * 1024), 16, vx[q], so, 0, 0);
#pragma unroll
      for (int q = 0; q < AU; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_a, (lptr_t)(smem + st + BM * 128 + (wave + 8 * q) * 1024), 16, va[q], so, 0, 0);
    };
#pragma unroll
    for (int t = 0; t < PD; ++t)
      if (t < KT) issue1(t, t * STAGE);
    int st = 0, fill = PD * STAGE;                // stages of tile t and of tile t + PD
    auto step = [&](int t) {
      // this wave's loads of tile t are complete (y pieces among the younger ones only make it wait for more)
      if (t + PD <= KT) wait_cnt<CNT*(PD - 1), 0>(); else wait_cnt<0, 0>();
      __builtin_amdgcn_s_barrier();               // everyone's are, and everyone has read tile t-1
      if (t + PD < KT) issue1(t + PD, fill);      // into the stage of tile t-1
      if (mine) {
        read_frags(smem + st, smem + st + BM * 128, f);
        mma(f, 4);
      }
      st = st + STAGE == NST * STAGE ? 0 : st + STAGE;
      fill = fill + STAGE == NST * STAGE ? 0 : fill + STAGE;
    };
    // the y pieces of tile i after step i of every YD-th part of the stages
    int t = 0;
#pragma unroll
    for (int i = 0; i < YD; ++i) {
      if (i < n_tiles) issue_y(i, yr[i]);
      for (; t < (i + 1) * KT / YD; ++t) step(t);
    }
  };
  issue_b(0, 0);
  if (rank <= 64) shrink(std::integral_constant<int, 1>{}); else shrink(std::integral_constant<int, 2>{});
  __syncthreads();   // the ring is dead
  if (nstage > 1) issue_b(0, 1);

  // T, rounded to bf16, into the stage layout (row r, logical 16-byte piece c of stage s at physical piece c ^ ((r/2) % 8));
  // a lane holds column wn * 32 + l32 of rows 8 * (v / 4) + 4 * lh + (v % 4) of each of its two 32-row tiles
  {
    const int col = wn * 32 + l32, s = col >> 6, cc = col & 63, piece = cc >> 3, within = (cc & 7) * 2;
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int r = wm * (BM / 2) + i * 32 + 8 * (v >> 2) + 4 * lh + (v & 3);
        *reinterpret_cast<bf16_t*>(smem + s * (BM * 128) + r * 128 + ((piece ^ ((r >> 1) & 7)) * 16) + within) = (bf16_t)acc[i][v];
      }
  }

  // ---- phase 2: y tile += scale * T . B_tile^T for every 128-column tile ----
  const bool full = m0 + BM <= M;
  __syncthreads();   // T is written
  bf16_t* sC = reinterpret_cast<bf16_t*>(smem + C_OFF);
  auto tile = [&](int j, u32x4 (&yc)[TI][ECH]) {
    // B tile j (this wave's share) is here; what is younger -- a wave's memory operations complete in order --, the stores of the tile
    // before and the y pieces requested with them, may still be on its way
    if (j > 0 && full && j - 1 + YD < n_tiles) wait_cnt<2 * TI * ECH, 0>(); else if (j > 0 && full) wait_cnt<TI * ECH, 0>(); else wait_cnt<0, 0>();
    __builtin_amdgcn_s_barrier();
    if (j + 1 < n_tiles) {                        // flies under this tile's MFMAs and epilogue
      issue_b(j + 1, 0);
      if (nstage > 1) issue_b(j + 1, 1);
    }
    zero_acc();
    for (int s = 0; s < nstage; ++s) {
      read_frags(smem + s * (BM * 128), b_stage(j, s), f);
      const int left = ks_total - 4 * s;
      mma(f, left < 4 ? left : 4);
    }
    if (j == 0) __syncthreads();                  // its B lies in the staging tile
    // epilogue: passes of 64 rows (of 128: the waves' upper / lower 32-row tiles): scale, round, transpose through LDS, add y
#pragma unroll
    for (int i = 0; i < TI; ++i) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = wm * 32 + 8 * (v >> 2) + 4 * lh + (v & 3);
        sC[row * LDC + wn * 32 + l32] = (bf16_t)(acc[i][v] * scale);
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < ECH; ++q) {
        const int c = tid + q * 512, srow = c / CPR, ch = c % CPR;
        const int grow = tile_row(i, srow);
        if (grow < M) {
          u32x4 o = *reinterpret_cast<const u32x4*>(sC + srow * LDC + ch * 8);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = pack_bf16x2(bf16_lo(o[e]) + bf16_lo(yc[i][q][e]), bf16_hi(o[e]) + bf16_hi(yc[i][q][e]));
          *reinterpret_cast<u32x4*>(y + (size_t)grow * N + (j0 + j) * 128 + ch * 8) = o;
        }
      }
      __syncthreads();
    }
    if (j + YD < n_tiles) issue_y(j + YD, yc);
  };
  for (int j = 0; j < n_tiles; j += YD) {
#pragma unroll
    for (int i = 0; i < YD; ++i) {
      if (j + i >= n_tiles) break;
      tile(j + i, yr[i]);
    }
  }
#endif
}

}  // namespace

namespace {

int sgmv_fused_impl(const void* x, const void* a_all, const void* b_all, void* y, const uint64_t* table, int64_t n_layers,
                    const int32_t* seg_start, const int32_t* seg_adapter, const int32_t* adapter_rank, const float* adapter_scale,
                    int64_t n_segments, int64_t max_seg_rows, int64_t N, int64_t K, int64_t RP, void* stream) {
  if (!x || !seg_start || !seg_adapter || !adapter_rank || !adapter_scale) return KH_ERR_INVALID_ARG;
  if (table == nullptr && (!a_all || !b_all || !y)) return KH_ERR_INVALID_ARG;
  if (n_segments <= 0 || max_seg_rows <= 0 || N <= 0 || K <= 0 || RP <= 0 || n_layers <= 0) return KH_ERR_INVALID_ARG;
  if (RP > 128) return KH_ERR_TOO_LARGE;
  if (K % 64 != 0 || N % 128 != 0 || RP % 32 != 0) return KH_ERR_UNSUPPORTED;
  if (n_segments > 65535 || max_seg_rows > (1 << 24) || N > (1 << 24) || K > (1 << 24)) return KH_ERR_TOO_LARGE;
  if (!kh_aligned16(x) || (table == nullptr && (!kh_aligned16(a_all) || !kh_aligned16(b_all) || !kh_aligned16(y))) ||
      (table != nullptr && ((uintptr_t)table & 7) != 0))
    return KH_ERR_ALIGNMENT;
  FusedParams p;
  p.x = (const bf16_t*)x; p.a_all = (const bf16_t*)a_all; p.b_all = (const bf16_t*)b_all; p.y = (bf16_t*)y;
  p.seg_start = seg_start; p.seg_adapter = seg_adapter; p.adapter_rank = adapter_rank; p.adapter_scale = adapter_scale;
  p.K = (int)K; p.N = (int)N; p.RP = (int)RP; p.table = table;
  // Row blocks of 64 while they about fit one round of the CUs (not all segments have max_seg_rows rows), of 128 otherwise: two rounds of 64
  // rows cost more than one of 128 (8 x 4096 rows: 40 against 32 us; 4 x 3136: 19 against 24).  Few row blocks: the column tiles of y are dealt to
  // several workgroups, each of which recomputes its rows' T, while that brings their number nearer to the CUs' (7 x 744 rows: 27 us with
  // one range, 20 with three, 28 with four, more than the CUs).
  const int bm = (max_seg_rows + 63) / 64 * n_segments * n_layers > 320 ? 128 : 64;
  const int64_t row_blocks = (max_seg_rows + bm - 1) / bm;
  const int64_t row_wgs = row_blocks * n_segments * n_layers, n_tiles = N / 128;
  int64_t z = 300 / row_wgs;
  z = z < 1 ? 1 : z < n_tiles ? z : n_tiles;
  p.tiles_per_z = (int)((n_tiles + z - 1) / z);
  z = (n_tiles + p.tiles_per_z - 1) / p.tiles_per_z;
  p.z_per_layer = (int)z;
  if (z * n_layers > 65535) return KH_ERR_TOO_LARGE;
  auto go = [&](auto bmc) {
    constexpr int BM = decltype(bmc)::value;
    if (hipError_t e = kh_allow_lds<sgmv_fused_kernel<BM>>(LDS_BYTES); e != hipSuccess) return (int)e;
    kh_launch(KH_TAG_SGMV_FUSED, sgmv_fused_kernel<BM>, dim3((unsigned)row_blocks, (unsigned)n_segments, (unsigned)(z * n_layers)), dim3(512), LDS_BYTES,
              (hipStream_t)stream, p);
    KH_RETURN_LAST_ERROR();
  };
  return bm == 128 ? go(std::integral_constant<int, 128>{}) : go(std::integral_constant<int, 64>{});
}

}  // namespace

// See include/katz_hip.h.
KH_EXPORT int kh_sgmv_fused_bf16(const void* x, const void* a_all, const void* b_all, void* y, const int32_t* seg_start,
                                 const int32_t* seg_adapter, const int32_t* adapter_rank, const float* adapter_scale,
                                 int64_t n_segments, int64_t max_seg_rows, int64_t N, int64_t K, int64_t RP, void* stream) {
  return sgmv_fused_impl(x, a_all, b_all, y, nullptr, 1, seg_start, seg_adapter, adapter_rank, adapter_scale, n_segments, max_seg_rows,
                         N, K, RP, stream);
}

// See include/katz_hip.h.
KH_EXPORT int kh_sgmv_fused_grouped_bf16(const void* x, const uint64_t* table, int64_t n_layers, const int32_t* seg_start,
                                         const int32_t* seg_adapter, const int32_t* adapter_rank, const float* adapter_scale,
                                         int64_t n_segments, int64_t max_seg_rows, int64_t N, int64_t K, int64_t RP, void* stream) {
  if (!table) return KH_ERR_INVALID_ARG;
  return sgmv_fused_impl(x, nullptr, nullptr, nullptr, table, n_layers, seg_start, seg_adapter, adapter_rank, adapter_scale, n_segments,
                         max_seg_rows, N, K, RP, stream);
}
