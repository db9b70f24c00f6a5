// K1, narrow-output variant: y = [x | T] . [W | B_cat]^T (+ bias, + residual) on bf16 MFMA (gfx950) with
// (32*WM) x 160 output tiles, for layers whose 128x128 tiles would leave much of the chip idle.
//
// Same arithmetic as the two-launch form of lora_gemm_pipe.hip (the reference's LoRA linear,
// diffusers-hf/src/diffusers/models/lora.py:224-225 after a separate shrink launch): T = the scaled
// shrink result, so the adapters' rank columns are extra K tiles of the base GEMM.
//
// Why another tile shape: N = 1280 = 2^8 * 5.  At M = 2048 the 128x128 tiling has 160 tiles for 256 CUs;
// 64x160 has exactly 256, 128x160 has 256 at M = 8192 / N = 640.  A factor 5 does not divide over 8
// waves in M or N, so the waves split K instead: a workgroup's 8 waves form WM row groups of 32 rows times
// WK = 8 / WM k-slices; a wave owns a 32 x 160 strip of accumulators (5 MFMA tiles) and multiplies only its
// own 16-column slices of every 64-column stage (1 x fragment + 5 W fragments per 5 MFMAs).  After the K
// loop the k-slices of a row group meet in LDS and are added in a fixed order (deterministic), then the
// epilogue is the usual one (bias in fp32, round, transpose through LDS, residual, 16-byte row stores).
//
// Operand movement as in lora_gemm_pipe.hip: global -> LDS by global_load_lds (8 rows x 128 bytes per
// instruction, XOR-swizzled pieces), a ring of 3 stages, loads two stages ahead, one barrier per stage,
// fragments double-buffered in registers.  (32*WM + 160) / 8 DMA units per stage do not divide by 8 waves:
// waves below N_HI issue one more than the others, and every wait picks its count by a wave-uniform branch.
#include "kh_common.h"
#include "lora_gemm.h"

namespace {

typedef const __attribute__((address_space(1))) void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;
typedef __amdgpu_buffer_rsrc_t rsrc_t;
template <int I> using IC = std::integral_constant<int, I>;

template <int VM, int LGKM>
__device__ __forceinline__ void wait_cnt() {  // gfx9 encoding: vmcnt = [15:14|3:0], expcnt = [6:4], lgkmcnt = [11:8]
  __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | ((LGKM & 15) << 8) | ((VM >> 4) << 14));
}

template <int WM_, int NST_ = 4>
struct KCfg {
  static constexpr int WM = WM_, WK = 8 / WM_;       // row groups x k-slices = 8 waves
  static constexpr int BM = 32 * WM, BN = 160, BK = 64, NST = NST_, TN = 5;   // NST ring stages: loads run NST - 1 K tiles ahead
  static constexpr int KSW = 4 / WK;                 // 16-column MFMA steps of a stage per wave
  static constexpr int UNITS = (BM + BN) / 8;        // DMA instructions per stage (8 rows x 128 B each)
  static constexpr int LPS_LO = UNITS / 8, N_HI = UNITS % 8, LPS_HI = LPS_LO + (N_HI ? 1 : 0);
  static constexpr int STAGE = (BM + BN) * 128;
  static constexpr int RING = NST * STAGE;
  static constexpr int PART = (WK - 1) * WM * 80 * 64 * 4;   // fp32 partial strips of the k-slices 1 .. WK-1
  static constexpr int LDC = BN + 8;
  static constexpr int SC = BM * LDC * 2;
  static constexpr int LDS = RING > PART + SC ? RING : PART + SC;
  static constexpr int OPC = BM * (BN / 8);          // 16-byte output pieces per tile
  static constexpr int OPT = (OPC + 511) / 512;      // per thread
  static_assert(WM == 2 || WM == 4, "row groups");
  static_assert(LDS <= 160 * 1024, "LDS budget");
};

template <class C>
__global__ __launch_bounds__(512, 2) void lora_gemm_ksplit_kernel(const LoraGemmParams p) {
#if __HIP_DEVICE_COMPILE__   // the host pass only needs the kernel's symbol (it cannot lower the buffer-resource type)
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int BM = C::BM, BN = C::BN, TN = C::TN, KSW = C::KSW, NST = C::NST, STAGE = C::STAGE;
  constexpr int LPS_LO = C::LPS_LO, LPS_HI = C::LPS_HI, N_HI = C::N_HI;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / C::WK, wk = wave % C::WK;
  const int l32 = lane & 31, lh = lane >> 5;

  // the next launch's weights
  kh_prefetch_lines(p.pf, p.pf_lines, smem + wave * 1024, blockIdx.x, gridDim.x, tid, 512);
  // tile of this workgroup: XCD b % 8 owns a block of xr_m x xr_n tiles (its W rows stay in its L2)
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int m_blk = (xcd / p.xg_n) * p.xr_m + local / p.xr_n;
  const int n_blk = (xcd % p.xg_n) * p.xr_n + local % p.xr_n;
  if (local / p.xr_n >= p.xr_m || m_blk >= p.m_tiles || n_blk >= p.n_tiles) return;  // padding of the grid
  const int m0 = m_blk * BM, n0 = n_blk * BN;
  const int M = p.M, N = p.N, K = p.K;
  const int KT1 = K / 64;
  const int KT = KT1 + (p.t_ext != nullptr ? p.R / 64 : 0);
  const bool has_hi = wave < N_HI;
  // folded LayerNorm: mean and 1/std of this tile's x rows, read in the epilogue (the barriers of the K loop lie between)
  // and the two per-column terms of this column tile; requested here, finished once the bias loads are under way
  float* sMu = reinterpret_cast<float*>(smem + p.ln_lds);
  float* sRs = sMu + 256;
  float* sc1 = sRs + 256;
  float* sc2 = sc1 + 256;
  KhLnTileStats<BM, 512> ln_stats;
  float ln_c1v = 0.f, ln_c2v = 0.f;
  if (p.ln_part != nullptr) {
    ln_stats.load(p.ln_part, m0, M, tid);
    if (tid < BN) {
      ln_c1v = n0 + tid < N ? p.ln_c1[n0 + tid] : 0.f;
      ln_c2v = n0 + tid < N ? p.ln_c2[n0 + tid] : 0.f;
    }
  }


  // DMA of this lane: unit u = wave + 8*q covers stage rows u*8 .. u*8+7 (x rows first, then W rows); LDS slot = lane:
  // row lane/8, physical piece lane%8, which holds logical piece (lane%8) ^ ((row/2)%8).  The loads are buffer loads:
  // a byte offset per lane that never changes (voff: row and piece) plus a scalar byte offset per K tile, so that the
  // loop carries no vector address arithmetic (with per-lane 64-bit pointers the adds and selects of every stage sat in
  // the same issue stream as the MFMAs and the loop ran at the sum of both).  Every buffer here is shorter than 2 GiB.
  uint32_t voff[LPS_HI], voff2[LPS_HI];
  constexpr int XQ = BM / 64;                          // units q < XQ are x rows for every wave, the others W rows
#pragma unroll
  for (int q = 0; q < LPS_HI; ++q) {
    int u = wave + 8 * q;
    u = u < C::UNITS ? u : C::UNITS - 1;               // never issued (has_hi), keep the offset valid
    const int r = u * 8 + (lane >> 3);
    const uint32_t pcb = (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
    if (r < BM) {
      int row = m0 + r; row = row < M ? row : M - 1;
      voff[q] = (uint32_t)row * (uint32_t)K * 2u + pcb;
      voff2[q] = ((uint32_t)row * (uint32_t)p.ldt + (uint32_t)(p.t_nsplit > 0 ? (n0 / p.t_nsplit) * p.R : 0)) * 2u + pcb;
    } else {
      int row = n0 + r - BM; row = row < N ? row : N - 1;
      voff[q] = (uint32_t)row * (uint32_t)K * 2u + pcb;
      voff2[q] = (uint32_t)row * (uint32_t)p.R * 2u + pcb;
    }
  }
  const rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.x), 0, (int)((size_t)M * K * 2), 0x00020000);
  const rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.w), 0, (int)((size_t)N * K * 2), 0x00020000);
  const rsrc_t rs_t = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.t_ext != nullptr ? p.t_ext : p.x), 0,
                                                         p.t_ext != nullptr ? (int)((size_t)M * p.ldt * 2) : 0, 0x00020000);
  const rsrc_t rs_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.t_ext != nullptr ? p.b_cat : p.w), 0,
                                                         p.t_ext != nullptr ? (int)((size_t)N * p.R * 2) : 0, 0x00020000);
  auto issue = [&](int t, auto stc) {                  // K tile t into ring stage stc
    char* stage = smem + decltype(stc)::value * STAGE;
    if (t < KT1) {
      const int so = t * 128;
#pragma unroll
      for (int q = 0; q < LPS_HI; ++q) {
        if (q < LPS_LO || has_hi) {
          __builtin_amdgcn_raw_ptr_buffer_load_lds(q < XQ ? rs_x : rs_w, (lptr_t)(stage + (wave + 8 * q) * 1024), 16, voff[q], so, 0, 0);
        }
      }
    } else {
      const int so = (t - KT1) * 128;
#pragma unroll
      for (int q = 0; q < LPS_HI; ++q)
        if (q < LPS_LO || has_hi)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(q < XQ ? rs_t : rs_b, (lptr_t)(stage + (wave + 8 * q) * 1024), 16, voff2[q], so, 0, 0);
    }
  };
  // wait until at most n of this wave's younger K tiles are outstanding (and its LDS reads are done)
  constexpr int PD = NST - 1;                            // prefetch distance in K tiles
  static_assert(NST == 3 || NST == 4, "groups of 6 or 4 written-out steps");
  auto wait_younger = [&](int n) {
    if (n >= PD - 1) { if (has_hi) wait_cnt<LPS_HI * (PD - 1), 0>(); else wait_cnt<LPS_LO * (PD - 1), 0>(); }
    else if (n == 1) { if (has_hi) wait_cnt<LPS_HI, 0>(); else wait_cnt<LPS_LO, 0>(); }
    else wait_cnt<0, 0>();
  };

  // fragment addresses: byte offsets into a stage that never change (the stage is a compile-time constant of every
  // unrolled step and lands in the instruction's offset field; stage 2 lies beyond that field's 64 KB and gets a
  // second set)
  struct Fr { bf16x8 a[KSW]; bf16x8 b[KSW][TN]; };
  const int sw = (l32 >> 1) & 7;
  int fa[KSW], fb[KSW], fa2[KSW], fb2[KSW];
#pragma unroll
  for (int k = 0; k < KSW; ++k) {
    const int po = ((2 * (wk * KSW + k) + lh) ^ sw) * 16;
    fa[k] = (wm * 32 + l32) * 128 + po;
    fb[k] = (BM + l32) * 128 + po;
    fa2[k] = fa[k] + 2 * STAGE;
    fb2[k] = fb[k] + 2 * STAGE;
  }
  auto read_frags = [&](auto stc, Fr& f) {
    constexpr int ST = decltype(stc)::value;
#pragma unroll
    for (int k = 0; k < KSW; ++k) {
      const char* pa = ST >= 2 ? smem + fa2[k] + (ST - 2) * STAGE : smem + fa[k] + ST * STAGE;
      const char* pb = ST >= 2 ? smem + fb2[k] + (ST - 2) * STAGE : smem + fb[k] + ST * STAGE;
      f.a[k] = *reinterpret_cast<const bf16x8*>(pa);
#pragma unroll
      for (int j = 0; j < TN; ++j) f.b[k][j] = *reinterpret_cast<const bf16x8*>(pb + j * 32 * 128);
    }
  };
  f32x16 acc[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;
  auto mma = [&](const Fr& f) {
#pragma unroll
    for (int k = 0; k < KSW; ++k)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[k], f.b[k][j], acc[j], 0, 0, 0);
  };

  // bias of this lane's columns, requested before the loop
  float bv[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = n0 + j * 32 + l32;
    bv[j] = (p.bias != nullptr && col < N) ? (float)p.bias[col] : 0.f;
  }
  if (p.ln_part != nullptr) {
    ln_stats.finish(K, p.ln_eps, tid, sMu, sRs, false);
    if (tid < BN) { sc1[tid] = ln_c1v; sc2[tid] = ln_c2v; }
  }
  wait_cnt<0, 15>();

  // K loop.  Step t: tile t is in registers (cur); tile t+1 becomes visible at the barrier, after which every wave has
  // read tile t out of its stage, so that stage takes tile t+1+PD.  lcm(NST, 2) steps (ring stages x two register
  // buffers) are written out, so the stage of every access is a constant; the steady group carries no conditions.
  Fr f0, f1;
  issue(0, IC<0>{});
  if (KT > 1) issue(1, IC<1>{});
  if (PD > 2 && KT > 2) issue(2, IC<2>{});
  wait_younger(KT - 1);
  __builtin_amdgcn_s_barrier();
  if (KT > PD) issue(PD, IC<PD>{});
  read_frags(IC<0>{}, f0);
  // st_next: stage of tile t+1; st_fill: stage that tile t+1+PD refills (= stage of tile t)
  auto step = [&](int t, const Fr& cur, Fr& nxt, auto st_next, auto st_fill, auto steady) {
    if constexpr (decltype(steady)::value) {
      wait_younger(PD - 1);
      __builtin_amdgcn_s_barrier();
      issue(t + 1 + PD, st_fill);
      read_frags(st_next, nxt);
    } else if (t + 1 < KT) {
      wait_younger(KT - 2 - t);
      __builtin_amdgcn_s_barrier();
      if (t + 1 + PD < KT) issue(t + 1 + PD, st_fill);
      read_frags(st_next, nxt);
    }
    mma(cur);
  };
  constexpr int U = (NST % 2 == 0) ? NST : 2 * NST;
  using T1 = std::true_type; using T0 = std::false_type;
  int t = 0;
  for (; t + U + PD < KT; t += U) {
    step(t, f0, f1, IC<1 % NST>{}, IC<0>{}, T1{});
    step(t + 1, f1, f0, IC<2 % NST>{}, IC<1 % NST>{}, T1{});
    step(t + 2, f0, f1, IC<3 % NST>{}, IC<2 % NST>{}, T1{});
    step(t + 3, f1, f0, IC<4 % NST>{}, IC<3 % NST>{}, T1{});
    if constexpr (U == 6) {
      step(t + 4, f0, f1, IC<5 % NST>{}, IC<4 % NST>{}, T1{});
      step(t + 5, f1, f0, IC<6 % NST>{}, IC<5 % NST>{}, T1{});
    }
  }
  for (; t < KT; t += U) {
    step(t, f0, f1, IC<1 % NST>{}, IC<0>{}, T0{});
    if (t + 1 < KT) step(t + 1, f1, f0, IC<2 % NST>{}, IC<1 % NST>{}, T0{});
    if (t + 2 < KT) step(t + 2, f0, f1, IC<3 % NST>{}, IC<2 % NST>{}, T0{});
    if (t + 3 < KT) step(t + 3, f1, f0, IC<4 % NST>{}, IC<3 % NST>{}, T0{});
    if constexpr (U == 6) {
      if (t + 4 < KT) step(t + 4, f0, f1, IC<5 % NST>{}, IC<4 % NST>{}, T0{});
      if (t + 5 < KT) step(t + 5, f1, f0, IC<6 % NST>{}, IC<5 % NST>{}, T0{});
    }
  }
  __syncthreads();   // the ring is dead: partial strips and the staging tile reuse it

  // residual pieces of this thread, requested before the reduction
  u32x4 rr[C::OPT];
  if (p.res != nullptr) {
#pragma unroll
    for (int q = 0; q < C::OPT; ++q) {
      const int c = tid + q * 512, srow = c / (BN / 8), ch = c % (BN / 8);
      const int grow = m0 + srow, gcol = n0 + ch * 8;
      rr[q] = (c < C::OPC && grow < M && gcol < N) ? *reinterpret_cast<const u32x4*>(p.res + (size_t)grow * N + gcol)
                                                  : u32x4{0, 0, 0, 0};
    }
  }
  // k-slices 1 .. WK-1 hand their strips to slice 0 of their row group: 20 x 16 bytes per lane, lane-contiguous
  // (writer lane = reader lane, so the layout is free)
  f32x4* part = reinterpret_cast<f32x4*>(smem);
  if (wk > 0) {
    f32x4* dst = part + ((size_t)((wk - 1) * C::WM + wm) * 20) * 64 + lane;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        dst[(j * 4 + g) * 64] = f32x4{acc[j][4 * g], acc[j][4 * g + 1], acc[j][4 * g + 2], acc[j][4 * g + 3]};
  }
  __syncthreads();
  bf16_t* sC = reinterpret_cast<bf16_t*>(smem + C::PART);
  if (wk == 0) {
#pragma unroll
    for (int s = 1; s < C::WK; ++s) {                  // fixed order: deterministic
      const f32x4* srcp = part + ((size_t)((s - 1) * C::WM + wm) * 20) * 64 + lane;
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 v = srcp[(j * 4 + g) * 64];
          acc[j][4 * g] += v[0]; acc[j][4 * g + 1] += v[1]; acc[j][4 * g + 2] += v[2]; acc[j][4 * g + 3] += v[3];
        }
    }
    if (p.ln_part != nullptr) {
      // y = rstd_row * (acc - mean_row * c1_col) + c2_col: four consecutive rows per accumulator group
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int trow = wm * 32 + 8 * g + 4 * lh;
        const f32x4 mu = *reinterpret_cast<const f32x4*>(sMu + trow), rs = *reinterpret_cast<const f32x4*>(sRs + trow);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const float c1 = sc1[j * 32 + l32], c2 = sc2[j * 32 + l32];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            sC[(trow + e) * C::LDC + j * 32 + l32] = (bf16_t)(rs[e] * (acc[j][4 * g + e] - mu[e] * c1) + c2);
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int col = j * 32 + l32;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int row = wm * 32 + 8 * (v >> 2) + 4 * lh + (v & 3);
          sC[row * C::LDC + col] = (bf16_t)(acc[j][v] + bv[j]);
        }
      }
    }
  }
  __syncthreads();
  const KhOut yout(p.y, (size_t)M * N * 2);
  if (p.st_part != nullptr) {
    // as below, and every row's (sum, sum of squares) over this tile's columns for a following folded LayerNorm: the 20
    // pieces of a row meet in LDS (the partial strips are dead) and are added in a fixed order
    float* sp = reinterpret_cast<float*>(smem);          // [BM][20][2]
    static_assert(BM * 20 * 8 <= C::PART, "row statistics fit the dead partial strips");
#pragma unroll
    for (int q = 0; q < C::OPT; ++q) {
      const int c = tid + q * 512, srow = c / (BN / 8), ch = c % (BN / 8);
      const int grow = m0 + srow, gcol = n0 + ch * 8;
      const bool ok = c < C::OPC && grow < M && gcol < N;
      u32x4 o = ok ? *reinterpret_cast<const u32x4*>(sC + srow * C::LDC + ch * 8) : u32x4{0, 0, 0, 0};
      if (p.res != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[e] = pack_bf16x2(bf16_lo(o[e]) + bf16_lo(rr[q][e]), bf16_hi(o[e]) + bf16_hi(rr[q][e]));
      }
      if (ok) yout.store16(((size_t)grow * N + gcol) * 2, o);
      float ps, pq;
      kh_piece_sums(o, ps, pq);
      if (c < C::OPC) *reinterpret_cast<u32x2*>(sp + 2 * c) = u32x2{__float_as_uint(ps), __float_as_uint(pq)};
    }
    __syncthreads();
    if (tid < BM && m0 + tid < M) {
      float s = 0.f, q2 = 0.f;
#pragma unroll
      for (int ch = 0; ch < BN / 8; ++ch) { s += sp[2 * (tid * (BN / 8) + ch)]; q2 += sp[2 * (tid * (BN / 8) + ch) + 1]; }
      kh_ln_store_stats(p.st_part, m0 + tid, M, n_blk, p.n_tiles, s, q2);
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < C::OPT; ++q) {
    const int c = tid + q * 512, srow = c / (BN / 8), ch = c % (BN / 8);
    const int grow = m0 + srow, gcol = n0 + ch * 8;
    if (c < C::OPC && grow < M && gcol < N) {
      u32x4 o = *reinterpret_cast<const u32x4*>(sC + srow * C::LDC + ch * 8);
      if (p.res != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[e] = pack_bf16x2(bf16_lo(o[e]) + bf16_lo(rr[q][e]), bf16_hi(o[e]) + bf16_hi(rr[q][e]));
      }
      yout.store16(((size_t)grow * N + gcol) * 2, o);
    }
  }
#endif
}

template <class C>
int launch_ksplit(LoraGemmParams p, hipStream_t stream) {
  p.m_tiles = (p.M + C::BM - 1) / C::BM;
  p.n_tiles = (p.N + C::BN - 1) / C::BN;
  static_assert(C::LDS + KH_LN_LDS <= 160 * 1024, "LDS budget with the row statistics");
  if (hipError_t e = kh_allow_lds<lora_gemm_ksplit_kernel<C>>(C::LDS + KH_LN_LDS); e != hipSuccess) return (int)e;
  if (p.st_part != nullptr && p.n_tiles > KH_LN_SLOTS) return KH_ERR_UNSUPPORTED;
  p.ln_lds = C::LDS;
  const size_t lds = (size_t)C::LDS + (p.ln_part != nullptr ? KH_LN_LDS : 0);
  // the XCD grid whose per-XCD block touches the fewest operand rows, padding counted as cost
  double best = 0;
  p.xg_n = 0;
  for (int gm = 1; gm <= 8; gm *= 2) {
    const int gn = 8 / gm;
    const int rm = (p.m_tiles + gm - 1) / gm, rn = (p.n_tiles + gn - 1) / gn;
    const double cost = ((double)rm * C::BM + (double)rn * C::BN) * (8.0 * rm * rn) / ((double)p.m_tiles * p.n_tiles);
    if (p.xg_n == 0 || cost < best) { best = cost; p.xg_n = gn; p.xr_m = rm; p.xr_n = rn; }
  }
  const unsigned grid = 8u * (unsigned)p.xr_m * (unsigned)p.xr_n;
  kh_launch(KH_TAG_LORA_GEMM, lora_gemm_ksplit_kernel<C>, dim3(grid), dim3(512), lds, stream, p);
  KH_RETURN_LAST_ERROR();
}

}  // namespace

// every operand is addressed as a buffer with 32-bit byte offsets: shorter than 2 GiB each
static bool ks_fits_buffers(const LoraGemmParams& p) {
  const size_t lim = (size_t)1 << 31;
  return (size_t)p.M * p.K * 2 < lim && (size_t)p.N * p.K * 2 < lim && (size_t)p.M * (p.ldt > 0 ? p.ldt : 1) * 2 < lim && (size_t)p.N * (p.R > 0 ? p.R : 1) * 2 < lim;
}

static bool lora_gemm_ksplit_ok(const LoraGemmParams& p) {
  const bool plain = p.R == 0 || p.t_ext != nullptr;
  return plain && ks_fits_buffers(p) && p.grp == nullptr && p.sg_mode == 0 && p.conv_cin == 0 && !p.geglu && p.K % 64 == 0 && p.K >= 64 &&
         (p.t_ext == nullptr || (p.R % 64 == 0 && p.ldt % 8 == 0)) && (p.t_nsplit == 0 || p.t_nsplit % 160 == 0) &&
         p.N % 8 == 0;
}

int lora_gemm_ksplit_launch(const LoraGemmParams& p, int row_groups, hipStream_t stream) {
  if (!lora_gemm_ksplit_ok(p)) return KH_ERR_UNSUPPORTED;
  return row_groups == 4 ? launch_ksplit<KCfg<4>>(p, stream) : launch_ksplit<KCfg<2>>(p, stream);
}
