// LoRA shrink for layers that share an input: t[M,R] = bf16((x[M,K] . A_cat[R,K]^T) * col_scale[R]).
//
// The low-rank "down" projection of the reference's LoRA linear
// (diffusers-hf/src/diffusers/models/lora.py:224-225, down(hidden_states)) for all adapters of one or
// several layers that read the same x at once: to_q / to_k / to_v of a self-attention take the same
// normalised hidden states, so their A matrices are stacked into one A_cat and x is read once.
// The result stays L2-resident (M*R*2 bytes, ~1 MB) and is consumed by kh_lora_linear_pre_bf16, which
// then runs the base GEMM without the per-tile shrink recompute of the fused kernel.
//
// Bound: the vector L1 path (64 B/clk per CU).  2*M*K*R FLOPs are ~1 GFLOP, but M*R is so small that
// filling 256 CUs means 32x32 or 64x64 output tiles, and a tile of a x b outputs pulls (a+b)*K*2
// bytes through its CU's L1.  A workgroup owns TR*32 rows x TC*32 rank columns; its NW waves split K.
// Each wave streams its 64-column chunks (dealt round-robin) through a PRIVATE two-stage LDS ring
// with global_load_lds: 8 rows x 128 contiguous bytes per instruction, i.e. whole cache lines (with
// 64-byte rows every line is fetched by two different steps and has left the 32 KB L1 in between; a
// fragment load straight from global memory has every lane in a row of its own and runs at a quarter
// of the L1 rate).  A private ring needs no barrier: the wave waits for its own loads (vmcnt), reads
// the fragments, and refills the stage it has just read.  Partial sums of the NW waves meet in LDS
// in a fixed order (deterministic).
// Tried and dropped: splitting K across workgroups with a last-arriver reduction (the device-scope
// release is an L2 write-back on a multi-XCD part: 40 us); direct global -> register fragments (L1
// tag rate, 3-4x slower at K = 5120).
#include "lora_shrink_tile.h"

namespace {

// GROUP > 0: the rank columns come in groups of GROUP (one stacked layer each) of which only the first C::TC * 32 are in
// use; blockIdx.y counts groups, and the tile's workgroup zeroes the group's padding columns for its rows.
template <class C, int GROUP = 0>
__global__ __launch_bounds__(C::NW * 64) void lora_shrink_kernel(const ShrinkParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int STEP = GROUP > 0 ? GROUP : C::TC * 32;
  const int m0 = (int)blockIdx.x * C::TR * 32, r0 = (int)blockIdx.y * STEP;
  lora_shrink_tile<C, false, C::NW * 64>(p, m0, r0, smem);
  if constexpr (GROUP > C::TC * 32) {
    constexpr int PIECES = (GROUP - C::TC * 32) / 8;   // 16-byte pieces per row
    for (int i = threadIdx.x; i < C::TR * 32 * PIECES; i += C::NW * 64) {
      const int row = m0 + i / PIECES;
      if (row < p.M) *reinterpret_cast<u32x4*>(p.t + (size_t)row * p.R + r0 + C::TC * 32 + (i % PIECES) * 8) = u32x4{0, 0, 0, 0};
    }
  }
}

template <class C, int GROUP = 0>
int launch_shrink(const ShrinkParams& p, hipStream_t stream) {
  if (hipError_t e = kh_allow_lds<lora_shrink_kernel<C, GROUP>>(C::LDS); e != hipSuccess) return (int)e;
  constexpr int STEP = GROUP > 0 ? GROUP : C::TC * 32;
  dim3 grid((unsigned)((p.M + C::TR * 32 - 1) / (C::TR * 32)), (unsigned)((p.R + STEP - 1) / STEP));
  kh_launch(KH_TAG_LORA_SHRINK, lora_shrink_kernel<C, GROUP>, grid, dim3(C::NW * 64), C::LDS, stream, p);
  KH_RETURN_LAST_ERROR();
}

// Few rows: 16 x 16 tiles (lora_shrink16_tile)
template <int NW>
__global__ __launch_bounds__(NW * 64) void lora_shrink16_kernel(const ShrinkParams p, int group, int tiles) {   // tiles: in use per group
#if __HIP_DEVICE_COMPILE__
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, m0 = (int)blockIdx.x * 16, g = (int)blockIdx.y / tiles, tile = (int)blockIdx.y % tiles;
  lora_shrink16_tile<NW, false>(p, m0, g * group + tile * 16, smem);
  if (tile == tiles - 1) {                              // the group's padding columns of these rows
    const int pieces = group / 8 - tiles * 2;
    for (int i = tid; i < 16 * pieces; i += NW * 64) {
      const int row = m0 + i / pieces;
      if (row < p.M) *reinterpret_cast<u32x4*>(p.t + (size_t)row * p.R + g * group + tiles * 16 + (i % pieces) * 8) = u32x4{0, 0, 0, 0};
    }
  }
#endif
}

template <int NW>
int launch_shrink16(const ShrinkParams& p, int group, int tiles, hipStream_t stream) {
  constexpr int LDS = SHRINK16_LDS<NW>;
  if (hipError_t e = kh_allow_lds<lora_shrink16_kernel<NW>>(LDS); e != hipSuccess) return (int)e;
  dim3 grid((unsigned)((p.M + 15) / 16), (unsigned)(p.R / group * tiles));
  kh_launch(KH_TAG_LORA_SHRINK, lora_shrink16_kernel<NW>, grid, dim3(NW * 64), LDS, stream, p, group, tiles);
  KH_RETURN_LAST_ERROR();
}

// What a call's sizes choose: the tiles, and how many waves share a sum (chunk t of 64 columns is added up by wave t % waves, then wave after wave).
enum ShrinkTiles { GROUP_32x96, TILE_64x64, TILE_32x64, TILE_16x16, TILE_32x32 };
struct ShrinkPlan {
  ShrinkTiles tiles;
  int waves;
  int group, used;      // rank columns of a layer; 16-column tiles of them that are in use (TILE_16x16)
};

ShrinkPlan shrink_plan(int64_t M, int64_t K, int64_t R, int group, int r_used) {
  const int64_t kc = K / 64;
  const auto even = [&](int a, int b) { return kc % a == 0 || kc % b != 0 ? a : b; };   // prefer a count that deals the chunks out evenly
  const int grp = group > 0 ? group : (int)R, used = (group > 0 && r_used > 0 && r_used < group ? r_used : grp) / 16;
  // several stacked layers of rank 96 in 128 on many rows (q / k / v of the 64 x 64 level): one-wave workgroups, each a
  // 32-row x 96-column tile of one layer over the whole K, five to a CU.  With K this short a tile is a handful of chunks
  // and its time is load latency, not bytes: more independent workgroups per CU win (16.3 us against 20.8 with the 64 x 64
  // tiles below at M 8192, K 640, three layers; 64 x 96 tiles of four waves 21.4, 128 x 96 tiles of two waves 25.3, although
  // both read fewer bytes).  A single layer (R 128) stays with the 64 x 64 tiles: 8.4 us against 13.2.
  if (group == 128 && r_used > 64 && r_used <= 96 && R % 128 == 0 && R >= 256 && M >= 4096) return {GROUP_32x96, 1, grp, used};
  // the largest output tile that still gives most CUs a workgroup (a 64x64 tile reads half the bytes per output of a 32x64 one)
  if (R % 64 == 0 && ((M + 63) / 64) * (R / 64) >= 160) return {TILE_64x64, even(4, 5), grp, used};
  if (R % 64 == 0 && ((M + 31) / 32) * (R / 64) >= 256) return {TILE_32x64, even(4, 5), grp, used};
  // 16 x 16 tiles while they get a CU each (the wave counts are those of the 32 x 32 tiles: the order of the sum)
  return {R % grp == 0 && (M + 15) / 16 * (R / grp) * used <= 256 ? TILE_16x16 : TILE_32x32, even(8, 5), grp, used};
}

template <int TR, int TC>
int launch_shrink_waves(const ShrinkParams& p, int waves, hipStream_t stream) {
  switch (waves) {
    case 4: if constexpr (TC == 2) return launch_shrink<SCfg<4, TR, TC>>(p, stream); break;
    case 5: return launch_shrink<SCfg<5, TR, TC>>(p, stream);
    case 8: if constexpr (TC == 1) return launch_shrink<SCfg<8, TR, TC>>(p, stream); break;
  }
  return KH_ERR_UNSUPPORTED;
}

}  // namespace

KH_EXPORT int kh_lora_shrink_bf16(const void* x, const void* a_cat, const float* col_scale, void* t, int64_t M,
                                  int64_t K, int64_t R, void* stream) {
  return lora_shrink_ln_launch(x, a_cat, col_scale, t, M, K, R, nullptr, nullptr, nullptr, 0.f, (hipStream_t)stream, 0, 0);
}

// For launches that bring their shrink along with the sums of its own launch.
int lora_shrink_waves(int64_t M, int64_t K, int64_t R, int group, int r_used) { return shrink_plan(M, K, R, group, r_used).waves; }

// The shrink, optionally of a layer with a folded LayerNorm (ln_part != nullptr; see ShrinkParams).
// group / r_used (both 0: nothing known): the R columns are stacked layers of `group` packed rank columns each, of which
// the columns >= r_used are padding (A_cat rows of zeros) that need not be computed.
int lora_shrink_ln_launch(const void* x, const void* a_cat, const float* col_scale, void* t, int64_t M, int64_t K, int64_t R,
                          const float* ln_part, const float* ln_ca1, const float* ln_ca2, float ln_eps, hipStream_t s,
                          int group, int r_used) {
  if (!x || !a_cat || !col_scale || !t || M <= 0 || K <= 0 || R <= 0) return KH_ERR_INVALID_ARG;
  if (ln_part != nullptr && (!ln_ca1 || !ln_ca2)) return KH_ERR_INVALID_ARG;
  if (K % 64 != 0 || R % 32 != 0) return KH_ERR_UNSUPPORTED;
  if (R > 65535 * 32 || M > (1 << 24)) return KH_ERR_TOO_LARGE;
  if (!kh_aligned16(x) || !kh_aligned16(a_cat) || !kh_aligned16(t) || (ln_part && !kh_aligned16(ln_part))) return KH_ERR_ALIGNMENT;
  ShrinkParams p;
  p.x = (const bf16_t*)x; p.a_cat = (const bf16_t*)a_cat; p.col_scale = col_scale; p.t = (bf16_t*)t;
  p.M = (int)M; p.K = (int)K; p.R = (int)R;
  p.ln_part = ln_part; p.ln_ca1 = ln_ca1; p.ln_ca2 = ln_ca2; p.ln_eps = ln_eps;
  const ShrinkPlan plan = shrink_plan(M, K, R, group, r_used);
  switch (plan.tiles) {
    case GROUP_32x96: return launch_shrink<SCfg<1, 1, 3>, 128>(p, s);
    case TILE_64x64: return launch_shrink_waves<2, 2>(p, plan.waves, s);
    case TILE_32x64: return launch_shrink_waves<1, 2>(p, plan.waves, s);
    case TILE_16x16: return plan.waves == 8 ? launch_shrink16<8>(p, plan.group, plan.used, s) : launch_shrink16<5>(p, plan.group, plan.used, s);
    default: return launch_shrink_waves<1, 1>(p, plan.waves, s);
  }
}
