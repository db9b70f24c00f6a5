// Parameters shared by the LoRA GEMM kernels (host fills, kernels read by value).
#pragma once
#include "kh_common.h"
#include <type_traits>

struct LoraGemmParams {
  const bf16_t* x;
  const bf16_t* w;
  const bf16_t* bias;      // may be null
  const bf16_t* a_cat;     // [R,K] (unused when R == 0)
  const bf16_t* b_cat;     // [N,R]
  const float* col_scale;  // [R]
  const bf16_t* t_ext;     // [M, ldt] precomputed, already scaled shrink result (null: compute it in the kernel)
  int ldt;
  int t_nsplit;            // > 0: W rows come in blocks of t_nsplit rows; block j uses T columns [j*R, (j+1)*R)
  // grouped launch: blockIdx.y selects a row {w, bias, b_cat, t_ext, y} of this device table (null: single layer)
  const uint64_t* grp;
  int dbg;  // always 0 unless the library is built with -DKH_TUNING (kernel experiments; not part of the C ABI)
  const bf16_t* res;       // [M,N] residual added in the epilogue, may be null
  bf16_t* y;
  int M, N, K, R;
  int m_tiles, n_tiles, n_chunk, n_chunks;  // n_chunk = N tiles walked by one workgroup
  // tile -> XCD map (xg_n > 0): the 8 XCDs form an xg_m x xg_n grid over the tile matrix, each owning a block of
  // xr_m x xr_n tiles (see launch_pcfg); 0: contiguous ranges of the (m block, n chunk) list per XCD
  int xg_n, xr_m, xr_n;
  // segmented launch (sg_mode != 0): blockIdx.y = segment s of a batch of requests; rows [sg_start[s], sg_start[s+1])
  // of x / y, weights of adapter sg_adapter[s] (negative: the segment is skipped) at w + adapter * sg_wstride.
  // sg_mode 1 (shrink): y = x . W_a^T.  sg_mode 2 (expand): y += sg_scale[a] * (x . W_a^T) over the first
  // sg_rank[a] K columns (x = the shrink result, row stride K).  M = the longest segment.
  const int32_t* sg_start; const int32_t* sg_adapter; const int32_t* sg_rank; const float* sg_scale;
  int sg_mode; long sg_wstride;
  int geglu;                                // 1: W rows are (value,gate) interleaved in 32-column groups, y is [M,N/2]
  // 3x3 convolution as an implicit GEMM (conv_cin > 0): x is an NHWC image [Nb, conv_h, conv_w, conv_cin], row m
  // of the GEMM is output pixel m of [Nb, conv_ho, conv_wo], K = 9 * conv_cin ordered (kh, kw, ci), padding 1
  int conv_cin, conv_h, conv_w, conv_ho, conv_wo, conv_stride;
  // shrink inside the GEMM launch (il_blocks > 0): the first il_blocks workgroups compute t_ext = the shrink of x
  // (a_cat, col_scale) in 64x64 tiles and count themselves into il_cnt[row block]; the GEMM workgroups wait for their
  // row block's count before they read t_ext.  il_cnt: ceil(M / 128) + 1 ints, zero when the launch starts (arrivals
  // per row block, then a time-out flag); the launch leaves the arrivals in them.
  int il_blocks = 0;
  int il_tile = 0, il_waves = 0;        // lora_gemm_fine.hip: rows and columns of a shrink tile, waves that share its sum
  int il_cols = 0;                      // column tiles of T per 64 rows beside 128 x 128 and 256 x 128 tiles (il_col_tiles)
  int* il_cnt = nullptr;
  // two-launch / in-launch forms: rank columns >= r_used of t_ext and b_cat are all zero (0: unknown, use R); the
  // 128x128 / 256x128 and 256x320 kernels then skip the MFMA steps that would only add zeros
  int r_used = 0;
  // LayerNorm folded into the GEMM (ln_part != nullptr): x is the input of a LayerNorm over its K columns whose affine
  // weight is already multiplied into w (and a_cat); the epilogue finishes the normalisation per output row,
  //   y[m,n] = rstd_m * (acc[m,n] - mean_m * ln_c1[n]) + ln_c2[n]   (ln_c1 = row sums of w, ln_c2 = bias + w . beta),
  // with mean / rstd from the row's 16 partial (sum, sum of squares) pairs in ln_part.  The shrink of such a layer
  // stores t = ((x . a^T) - mean * ln_ca1 + ln_ca2 / rstd) * col_scale, i.e. the adapter's share divided by rstd.
  const float* ln_part = nullptr;   // [16][M][2]
  const float* ln_c1 = nullptr;     // [N]
  const float* ln_c2 = nullptr;     // [N]
  const float* ln_ca1 = nullptr;    // [ldt] (shrink)
  const float* ln_ca2 = nullptr;    // [ldt]
  float ln_eps = 0.f;
  int ln_lds = 0;                   // byte offset of the workgroup's mean / rstd arrays in dynamic LDS (set by the launcher)
  // Row statistics of the output for a following folded LayerNorm (st_part != nullptr): column tile j writes the
  // (sum, sum of squares) of its columns of every row to st_part[j][row]; tile 0 also zeroes the slots past the last tile.
  float* st_part = nullptr;         // [16][M][2]
  // Weight prefetch (pf != nullptr): the launch also touches every 128-byte line of pf[0 .. 128 * pf_lines), the weights
  // of the NEXT launch of this family, so that they wait in the memory-side cache when that launch asks for them (a
  // step reads 2.5 GB of weights once each: every launch would otherwise meet its weights in HBM, where the XCDs that
  // share a weight block each fetch it again).  Set from kh_set_weight_prefetch by the entry points.
  // Cross-attention in the epilogue (xa_k != nullptr): the layer is an attention's to_q and an output tile holds queries of
  // one sample by whole 64-wide heads -- 32, 64 or 128 queries of one or two heads on the fine tiles (xattn_tile.h), 128 of two
  // on the 128x128 / 8-wave tiles (lora_gemm_pipe.hip); instead of storing them the workgroup runs
  // softmax(q k^T * scale) v for them against the xa_S <= 96 keys of those heads and stores that to xa_o (rows like y's,
  // head h at columns 64 h).  Rows m belong to batch sample m / xa_T (xa_T % 128 == 0); k / v: [B, S, heads * 64] views.
  const bf16_t* xa_k = nullptr; const bf16_t* xa_v = nullptr; bf16_t* xa_o = nullptr;
  int xa_S = 0, xa_T = 0;
  long xa_ldk = 0, xa_ldv = 0, xa_ldo = 0, xa_bsk = 0, xa_bsv = 0;
  float xa_scale_log2e = 0.f;
  // GroupNorm statistics of a convolution's result as a by-product of its epilogue (gn_part != nullptr; 3x3 convolutions on
  // the 160-column tiles): a tile holds whole groups of gn_cg channels of BM pixels of one image (gn_hw pixels each), and
  // its workgroup writes their (sum, sum of squares) over conv + gn_add[image][c] to gn_part[image][group][row tile of
  // the image][2] -- the layout kh_group_norm_bf16's second pass folds.
  float* gn_part = nullptr; const bf16_t* gn_add = nullptr;
  int gn_cg = 0, gn_hw = 0;
  const void* pf[3] = {nullptr, nullptr, nullptr};   // up to three ranges: weights, A_cat, B_cat of that launch
  uint32_t pf_lines[3] = {0, 0, 0};
};

// bit 24 of the `flags` of kh_lora_linear_split_bf16 / _norm_bf16 / _xattn_bf16: no launch whose workgroups wait for others of it (see include/katz_hip.h)
constexpr int KH_FLAG_NO_WAIT = 1 << 24;

// Weight prefetch of a launch with its own shrink: by the idle waves of the shrink workgroups when the first range is short
__host__ __device__ inline bool il_prefetch_by_idle_waves(const LoraGemmParams& p) { return p.pf_lines[0] <= ((8u << 20) >> 7); }

// The XCD grid of mt x nt tiles of bm x bn: the one whose per-XCD block of rm x rn tiles touches the fewest operand rows, padding counted as cost.
struct KhXcdGrid { int gn, rm, rn; };      // XCDs side by side in a row of tiles; the block
inline KhXcdGrid kh_xcd_grid(int mt, int nt, int bm, int bn) {
  KhXcdGrid g = {0, 0, 0};
  double best = 0;
  for (int gm = 1; gm <= 8; gm *= 2) {
    const int gn = 8 / gm, rm = (mt + gm - 1) / gm, rn = (nt + gn - 1) / gn;
    const double cost = ((double)rm * bm + (double)rn * bn) * (8.0 * rm * rn) / ((double)mt * nt);
    if (g.gn == 0 || cost < best) { best = cost; g = {gn, rm, rn}; }
  }
  return g;
}

// Do `cols` column tiles of T per 64 rows find a CU each beside the 128 x 128 GEMM tiles, on every XCD?  (2304 / 1280 / 1280: 72 pieces and 180 tiles
// are 252 in all but 9 + 25 on an XCD: a second round, 21.3 us in place of 19.4 with 36 pieces; K 2048 27.4 and 23.4)
inline bool il_fits_beside(const LoraGemmParams& p, int cols) {
  const KhXcdGrid g = kh_xcd_grid((p.M + 127) / 128, (p.N + 127) / 128, 128, 128);
  return ((p.M + 63) / 64 * cols + 7) / 8 + g.rm * g.rn <= 32;
}

// In-launch shrink on 64 x 32 tiles: a single layer with R = 64 columns of T, or with 128 of which at most the first 96 are
// in use (two adapters of ranks 64 + 32, say), short enough in K that its GEMM tiles would otherwise wait for T, and
// small enough in M that the two or three tiles per 64 rows fit beside the GEMM tiles (M 2048 / N 1280 / K 1280, rank 64: 19.2 us on one 64 x 64
// tile per 64 rows).  The GEMM tiles never multiply the columns the shrink leaves unwritten (r_used bounds their K loop).
// Decided on the host: the kernels get the number of column tiles (p.il_cols), more than one per 64 columns of T where they are narrow.
inline int il_col_tiles(const LoraGemmParams& p) {
  const int narrow = p.ldt != p.R ? 0 : p.R == 64 ? 2 : p.R == 128 && p.r_used > 0 && p.r_used <= 96 ? 3 : 0;
  return narrow > 0 && p.K <= 2560 && il_fits_beside(p, narrow) ? narrow : p.ldt / 64;
}
__device__ __forceinline__ bool il_narrow(const LoraGemmParams& p) { return p.il_cols * 64 > p.ldt; }

// The pending weight prefetch of this host thread (kh_set_weight_prefetch), handed to the next launch.
void kh_take_weight_prefetch(LoraGemmParams& p);

// bytes of dynamic LDS a launch with a folded LayerNorm adds: mean, 1/std of a tile's rows, c1, c2 of its columns, 2 * max(BM, 128) + 2 * BN floats at most
// (192 x 320 tiles use all of it)
constexpr int KH_LN_LDS = 4096;
constexpr int KH_LN_SLOTS = 16;     // partial pairs per row: at most 16 column tiles (N <= 2048 with 128-column tiles)

// Touch lines first, first + n_wg * NT, ... of the prefetch range: one dword per line and lane, loaded into 256 bytes of
// LDS that belong to this wave alone and that its own later DMA overwrites (a wave's loads land in order), so no
// register and no wait is spent on data nobody reads.  wg / n_wg: this workgroup's index among those that take part.
__device__ __forceinline__ void kh_prefetch_lines(const void* const (&pf)[3], const uint32_t (&lines)[3], char* wave_lds, int wg, int n_wg,
                                                  int tid, int nt) {
#if __HIP_DEVICE_COMPILE__
  if (pf[0] == nullptr) return;
  // four rounds over the first range (64 MB with 256 workgroups of 512 threads), one over the others (adapter matrices),
  // no loop; the per-lane offset carries the round, because only it is checked against the range: an offset beyond the
  // range reads nothing
  const uint32_t first = ((uint32_t)wg * (uint32_t)nt + (uint32_t)tid) << 7, step = ((uint32_t)n_wg * (uint32_t)nt) << 7;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(pf[k] != nullptr ? pf[k] : pf[0]), 0,
                                                                        pf[k] != nullptr ? (int)(lines[k] << 7) : 0, 0x00020000);
#pragma unroll
    for (uint32_t r = 0; r < (k == 0 ? 4u : 1u); ++r) {
      const uint32_t off = first + r * step;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)wave_lds, 4, off >= first ? off : 0xFFFFFFFFu, 0, 0, 0);
    }
  }
#endif
}

// Bring a block of W into this XCD's L2: the 128-byte lines of K columns 64 c0 .. 64 (c0 + nc) of rows row0 .. row0 + rows, thread i of n
// taking lines i, i + n, ... (loaded like the hint above: into LDS nobody reads).  The workgroups of an XCD that share the block take
// a share each.  Without it all of them meet the same cold lines at the same time, and a CU takes about 55 GB/s of lines that come from
// memory, 110 GB/s of lines its L2 has.
// NC: nc's largest value where that is known, so that a line's row and column come without a division.
template <int NC = 0>
__device__ __forceinline__ void kh_touch_rows(const bf16_t* w, int N, int K, int row0, int rows, int c0, int nc, char* wave_lds, int i, int n) {
#if __HIP_DEVICE_COMPILE__
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(w), 0, (int)((size_t)N * K * 2), 0x00020000);
  if (row0 + rows > N) rows = N - row0;
  if (64 * (c0 + nc) > K) nc = K / 64 - c0;
  const int per = NC > 0 ? NC : nc;
  for (int l = i; l < rows * per; l += n) {
    const int r = l / per, c = l - r * per;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)wave_lds, 4,
                                             c < nc ? (uint32_t)(row0 + r) * (uint32_t)K * 2u + (uint32_t)(c0 + c) * 128u : 0xFFFFFFFFu, 0, 0, 0);
  }
#endif
}
// ... from the start of a kernel, where the block is at most 3 MB of the XCD's 4 MB (and W below 2 GiB)
__device__ __forceinline__ bool kh_touch_pays(int N, int K, int rows) { return (size_t)rows * K * 2 <= (3u << 20) && (size_t)N * K * 2 < (1ull << 31); }

// The same from waves that have nothing else to do (the idle half of an in-launch shrink workgroup): as many rounds as
// the ranges need, up to 16 (the first range) / 4 (the others), in a loop.
__device__ __forceinline__ void kh_prefetch_lines_idle(const void* const (&pf)[3], const uint32_t (&lines)[3], char* wave_lds, int wg, int n_wg,
                                                       int tid, int nt) {
#if __HIP_DEVICE_COMPILE__
  if (pf[0] == nullptr) return;
  const uint32_t first = ((uint32_t)wg * (uint32_t)nt + (uint32_t)tid) << 7, step = ((uint32_t)n_wg * (uint32_t)nt) << 7;
  // (three calls: indexed in a loop the arrays went to scratch memory in some kernels)
  auto range = [&](const void* at, uint32_t n, uint32_t cap) {
    if (at == nullptr) return;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(at), 0, (int)(n << 7), 0x00020000);
    const uint32_t bytes = n << 7;                       // at most 2 GiB
    uint32_t rounds = (bytes + step - 1) / step;
    rounds = rounds < cap ? rounds : cap;
    for (uint32_t r = 0; r < rounds; ++r)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)wave_lds, 4, first + r * step, 0, 0, 0);
  };
  range(pf[0], lines[0], 16u);
  range(pf[1], lines[1], 4u);
  range(pf[2], lines[2], 4u);
#endif
}

// a column tile's pair for one output row, and (from tile 0) zeros in the slots no tile writes
__device__ __forceinline__ void kh_ln_store_stats(float* part, int row, int M, int tile, int n_tiles, float s, float q) {
  u32x2* dst = reinterpret_cast<u32x2*>(part) + row;
  dst[(size_t)tile * M] = u32x2{__float_as_uint(s), __float_as_uint(q)};
  if (tile == 0)
    for (int t = n_tiles; t < KH_LN_SLOTS; ++t) dst[(size_t)t * M] = u32x2{0u, 0u};
}

// sum over the 16 lanes of a DPP row (lanes 16k .. 16k+15), the result in every lane: four cross-lane adds in the VALU
__device__ __forceinline__ float kh_row16_sum(float v) {
  auto dpp = [](float x, auto ctrl) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  v += dpp(v, std::integral_constant<int, 0xb1>{});    // quad_perm [1,0,3,2]
  v += dpp(v, std::integral_constant<int, 0x4e>{});    // quad_perm [2,3,0,1]
  v += dpp(v, std::integral_constant<int, 0x141>{});   // row_half_mirror
  v += dpp(v, std::integral_constant<int, 0x140>{});   // row_mirror
  return v;
}

// mean and 1/std (or std, `want_sigma`) of ROWS consecutive rows from m0 into out_mean / out_2 (LDS), by all NT threads
// of the workgroup, in two steps so that the loads fly while the kernel sets up its operands.  A wave takes sixteen rows
// at a time: lane = (slot group g = lane / 16, row = lane % 16) loads the pairs of slots g, 4 + g, 8 + g, 12 + g (every
// load instruction reads four whole 128-byte lines of the slot-major buffer [slot][row][2]), adds them up, and the four
// groups meet by two cross-lane adds: a fixed order, deterministic.  M = rows of the buffer, D = the row's length.
// Same formula as the stand-alone LayerNorm kernel: biased variance, rstd = rsqrt(var + eps).
template <int ROWS, int NT>
struct KhLnTileStats {
  static constexpr int PASSES = (ROWS + (NT / 64) * 16 - 1) / ((NT / 64) * 16);
  static_assert(KH_LN_SLOTS == 16 && ROWS % 16 == 0 && NT % 64 == 0, "four slot groups of four, sixteen rows per wave and pass");
  u32x2 v[PASSES][4];

  __device__ __forceinline__ void load(const float* part, int m0, int M, int tid) {
    const int lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const u32x2* src = reinterpret_cast<const u32x2*>(part) + (size_t)g * M;
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps) {
      const int r = ((tid >> 6) + ps * (NT / 64)) * 16 + r16;          // beyond ROWS: a valid address, never stored
      const int row = m0 + r < M ? m0 + r : M - 1;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[ps][j] = src[(size_t)(4 * j) * M + row];
    }
  }
  __device__ __forceinline__ void finish(int D, float eps, int tid, float* out_mean, float* out_2, bool want_sigma) const {
    const int lane = tid & 63, r16 = lane & 15, g = lane >> 4;
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps) {
      const int r = ((tid >> 6) + ps * (NT / 64)) * 16 + r16;
      float s = 0.f, q = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) { s += __uint_as_float(v[ps][j][0]); q += __uint_as_float(v[ps][j][1]); }
      s += __shfl_xor(s, 16, 64); q += __shfl_xor(q, 16, 64);
      s += __shfl_xor(s, 32, 64); q += __shfl_xor(q, 32, 64);
      if (g == 0 && r < ROWS) {
        const float mean = s / (float)D;
        float var = q / (float)D - mean * mean;
        var = var > 0.f ? var : 0.f;
        out_mean[r] = mean;
        out_2[r] = want_sigma ? sqrtf(var + eps) : rsqrtf(var + eps);
      }
    }
  }
};

// one thread's share of a row's statistics: the (sum, sum of squares) of the eight bf16 values of a 16-byte piece
__device__ __forceinline__ void kh_piece_sums(const u32x4 o, float& s, float& q) {
  s = 0.f; q = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = bf16_lo(o[e]), b = bf16_hi(o[e]);
    s += a; q += a * a;
    s += b; q += b * b;
  }
}

// Software-pipelined kernel (lora_gemm_pipe.hip); needs K % 32 == 0.  tile_sel: 0 automatic, >= 16 forces a tile.
int lora_gemm_pipe_launch(const LoraGemmParams& p, int tile_sel, hipStream_t stream);
// 3x3 convolution (conv_* fields set, R == 0, K == 9 * conv_cin, conv_cin % 32 == 0).
int lora_gemm_pipe_launch_conv(const LoraGemmParams& p, hipStream_t stream);
// Segmented multi-adapter form (sg_* fields set; plain GEMM per segment, K % 32 == 0).
int lora_gemm_pipe_launch_sgmv(const LoraGemmParams& p, int n_segments, hipStream_t stream);
// Grouped form: grid.y = n_groups, per-group pointers from p.grp; rank columns (p.R > 0) as extra K tiles.
int lora_gemm_pipe_launch_grouped(const LoraGemmParams& p, int n_groups, hipStream_t stream);
// Shrink and GEMM in one launch for shapes whose 128x128 tiles leave CUs idle (p.a_cat / col_scale / b_cat set, p.t_ext =
// scratch for the shrink result, p.il_cnt = counters); KH_ERR_UNSUPPORTED when the shape does not qualify.
int lora_gemm_pipe_il_form(const LoraGemmParams& p);          // 0: not taken
int lora_gemm_pipe_launch_il(const LoraGemmParams& p, int form, hipStream_t stream);
// query projection + cross-attention in its epilogue (xa_k set)
bool lora_gemm_pipe_xattn_ok(const LoraGemmParams& p);
int lora_gemm_pipe_launch_xattn(const LoraGemmParams& p, bool il, hipStream_t stream);     // il: with its shrink (the call has an il form)
// (32 * row_groups) x 160 tiles whose 8 waves are row_groups x k-slices (lora_gemm_ksplit.hip), tile codes 40 and 41;
// plain or K-extended GEMM with bias / residual, K % 64 == 0.  row_groups 2 or 4.
int lora_gemm_ksplit_launch(const LoraGemmParams& p, int row_groups, hipStream_t stream);
// the convolution that also leaves GroupNorm statistics (gn_cg / gn_hw set): row groups of the 160-column tiles it would run
// on, 0 when the rules give it other tiles or the groups do not fit them
int lora_gemm_conv_gn_row_groups(const LoraGemmParams& p);
// Fine tiles (lora_gemm_fine.hip), with the sums in the order of the 128 x 128 (order 0), the 128 x 160 (order 2) or the 64 x 160 kernel
// (order 4); plain or K-extended GEMM and 3x3 convolutions (in order 0 on 128 x 128 and 128 / 160 / 192 x 160, without GroupNorm statistics).
// ok: what the kernel takes at all; form: -1 where order 0 is not suited (orders 2 and 4: the caller has seen to N % 160 and the number of tiles).
bool lora_gemm_fine_ok(const LoraGemmParams& p);
int lora_gemm_fine_form(const LoraGemmParams& p, int order);
int lora_gemm_rounds_form(const LoraGemmParams& p);          // of a convolution or a linear layer with many rows in order 0; -1: none
int lora_gemm_geglu_form(const LoraGemmParams& p);           // of a GEGLU projection; -2: the 256 x 320 tiles of lora_gemm_wide.hip, -1: neither
int lora_gemm_fine_launch(const LoraGemmParams& p, int form, hipStream_t stream);
// the fine tile that a call with T given runs on, -1 where another kernel is chosen
int lora_gemm_pipe_fine_form(const LoraGemmParams& p);
// Shrink and GEMM in one launch on fine tiles that leave CUs idle (p.a_cat / col_scale / b_cat set, p.t_ext = scratch for the shrink result,
// p.il_cnt = counters)
int lora_gemm_fine_il_form(LoraGemmParams p);                 // -1: not taken
int lora_gemm_fine_launch_il(LoraGemmParams p, int form, hipStream_t stream);
bool lora_gemm_fine_grouped_ok(const LoraGemmParams& p);     // many layers on the same few rows (p.grp)
int lora_gemm_fine_launch_grouped(const LoraGemmParams& p, int n_groups, hipStream_t stream);
// a query projection with its cross-attention: 1 or 2 launches, 0 where lora_gemm_pipe_launch_xattn takes it; two launches: the second, T given
int lora_gemm_fine_xattn_launches(const LoraGemmParams& p, bool may_wait);
int lora_gemm_fine_launch_xattn(const LoraGemmParams& p, bool may_wait, hipStream_t stream);
int lora_gemm_fine_launch_il128(LoraGemmParams p, hipStream_t stream);   // ... on 128 x 128 tiles, for lora_gemm_pipe_launch_il
// how many waves share a sum of the stand-alone shrink of this call (lora_shrink.hip)
int lora_shrink_waves(int64_t M, int64_t K, int64_t R, int group, int r_used);
// Shrink and GEMM in one launch on the 128 x 160 tiles, every workgroup computing a piece of T first (p.a_cat / col_scale /
// b_cat set, p.t_ext = scratch for the shrink result, p.il_cnt = counters, p.r_used <= 96 of R = 128).
bool lora_gemm_fine_coop_ok(const LoraGemmParams& p);
int lora_gemm_fine_launch_coop(const LoraGemmParams& p, hipStream_t stream);
int lora_gemm_fine_coop_timeouts(int* count, int clear);
// Wide-tile variant (lora_gemm_wide.hip): 256 x 320 tiles, 8 waves; plain or K-extended GEMM with bias / residual /
// GEGLU; M % 256 == 0, N % 320 == 0, K % 64 == 0.
bool lora_gemm_wide_ok(const LoraGemmParams& p);
int lora_gemm_wide_launch(LoraGemmParams p, hipStream_t stream);

// The shrink of a layer, optionally with a folded LayerNorm in front (ln_part != nullptr; lora_shrink.hip).
int lora_shrink_ln_launch(const void* x, const void* a_cat, const float* col_scale, void* t, int64_t M, int64_t K, int64_t R,
                          const float* ln_part, const float* ln_ca1, const float* ln_ca2, float ln_eps, hipStream_t stream, int group, int r_used);

extern "C" int kh_lora_shrink_bf16(const void* x, const void* a_cat, const float* col_scale, void* t, int64_t M, int64_t K,
                                   int64_t R, void* stream);

// Kernel experiments (timestamps, frozen operands, alternative tile maps) exist only in builds with -DKH_TUNING; the
// shipped library compiles them out and its entry points reject the flag bits that would select them.
#ifdef KH_TUNING
#define KH_DBG(p, bit) (((p).dbg & (bit)) != 0)
#else
#define KH_DBG(p, bit) false
#endif
