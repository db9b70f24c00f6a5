// K1 / K1c, fine tiles: y = x W^T (+ T B_cat^T, + bias, + residual, LayerNorm folded in / row statistics out) and 3x3
// convolutions on BM x BN output tiles small enough that a few hundred rows still give every CU a workgroup.
//
// Same arithmetic as the two-launch form of lora_gemm_pipe.hip (the reference's LoRA linear,
// diffusers-hf/src/diffusers/models/lora.py:224-225, T made by a launch in front), bit for bit as one of the kernels for more
// rows: the order of every sum is that kernel's (below), which is what the tests compare with.
//
// What bounds these calls: not the matrix pipe and not HBM's rate but a CU's operand stream.  A CU takes about 55 GB/s of
// lines that come from memory and 110 GB/s of lines its L2 has, all CUs together 17 TB/s out of the L2s; a 128 x 128 tiling of M = 1000 /
// N = 1280 streams 32 KB a stage into each of 80 CUs and takes 16 us, whether M is 150 or 2000.  Hence
//   * small tiles: 64 x 80 gives 256 workgroups there, 18 KB a stage;
//   * four waves that only move operands beside four or eight that only compute: a wave that does both stands in the queue of the address
//     unit (16 clocks per 1 KB instruction) while its MFMAs wait (64 x 160 tiles: 1330 clocks a stage together, 860 apart).  Eight (GEGLU and
//     order 2) are two to a SIMD, so that one's LDS reads run under the other's MFMAs;
//   * a ring of as many stages as LDS holds (up to 16), and
//   * the XCD's block of W fetched into its L2 by all its workgroups before the K loop meets it.
//
// Orders (ORD): the 128 x 128 / 256 x 320 kernels add along K one 16-column step after the other (0), the 160-column kernels in four
// slices of 16 (4) or two of 32 (2) of every 64 columns that are added at the end.  v_mfma 16x16x32 gives the bits of two chained 16-column steps of
// 32x32x16, and 16x16x16 those of one, so 16-row tiles can follow either.  Row statistics are sums over 128 columns (order 0) or
// 160 (orders 2 and 4): layers that leave them run on tiles of that width.
//
// Operands reach LDS by buffer loads (8 rows x 128 bytes per instruction, XOR-swizzled pieces, rows past M read zeros).
#include "kh_common.h"
#include "lora_gemm.h"
#include "lora_shrink_tile.h"
#include "xattn_tile.h"

// Bounded waits of the cooperative shrink that have run out on this GPU; read (and cleared) by kh_lora_split_timeouts
// together with the count of the in-launch shrink of lora_gemm_pipe.hip.
static __device__ int kh_coop_timeout_count;

namespace {

typedef __attribute__((address_space(3))) void* lptr_t;
typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef short s16x4 __attribute__((ext_vector_type(4)));

template <int VM, int LGKM>
__device__ __forceinline__ void wait_cnt() {  // gfx9 encoding: vmcnt = [15:14|3:0], expcnt = [6:4], lgkmcnt = [11:8]
  __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | ((LGKM & 15) << 8) | ((VM >> 4) << 14));
}

// until at most n K tiles of LPS loads each are outstanding (n >= N: N tiles)
template <int LPS, int N>
__device__ __forceinline__ void wait_tiles(int n) {
  if constexpr (N <= 0) wait_cnt<0, 0>();
  else if (n >= N) wait_cnt<LPS * N, 0>();
  else wait_tiles<LPS, N - 1>(n);
}

// a bare barrier (a fence would drain the prefetches), kept in place among the memory accesses around it
__device__ __forceinline__ void ring_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

constexpr int cmax(int a, int b) { return a > b ? a : b; }
constexpr int cmin(int a, int b) { return a < b ? a : b; }

constexpr int GTAB_LO = 0x3800, GTAB_N = 2560;           // gates 2^-15 <= |gate| < 32, per sign

template <int BM_, int BN_, int ORD_, bool GLU_ = false>
struct FCfg {
  static constexpr int BM = BM_, BN = BN_, ORD = ORD_;
  static constexpr bool GLU = GLU_;                      // GEGLU epilogue
  static constexpr int CW = GLU || ORD == 2 ? 8 : 4, CT = CW * 64, NT = CT + 256;   // computing waves (and four that move operands), their threads, all threads
  static constexpr int TAB = GLU ? 2 * GTAB_N * 2 : 0;   // its table of bf16(gelu(gate)), see lora_gemm_wide.hip
  // computing waves: WM row groups x WN column groups x WK k-slices
  static constexpr int WK = ORD == 0 ? 1 : ORD, WN = GLU ? 4 : ORD == 2 ? 2 : ORD != 0 ? 1 : BM == 32 ? (BN >= 64 ? 4 : 2) : BN % 128 != 0 && BN != 160 ? 1 : 2,
                       WM = CW / (WK * WN);
  // 32-row MFMA tiles for the slices where the tile divides into them, 16-row tiles otherwise (16x16x16 has half the rate)
  static constexpr int MF = ORD == 4 && BN % 32 == 0 ? 32 : 16, G = MF == 32 ? 4 : 1;     // G: groups of four rows per lane and tile
  static constexpr int TM = BM / (MF * WM), TN = BN / (MF * WN);                           // a wave's MFMA tiles
  static constexpr int KS = ORD == 0 ? 2 : 1;                                            // its k-steps per stage
  // operand order of the matrix instructions: (W, x) leaves four columns of a row in a lane, so that the epilogue writes 8 bytes at a time
  // (128 x 320: 5.6 K clocks against 8.4 K), (x, W) four rows of a column.  One x fragment per W fragment is the exception: the K loop of 64 x 80
  // takes 8.8 K clocks with (x, W) and 9.9 K with (W, x), more than the epilogue saves.
  static constexpr bool XW = BM == 64 && BN == 80 && ORD == 0;
  static constexpr bool DB = TM * TN * G * 4 <= 96 && BM <= 128 && !GLU;      // two fragment buffers where the registers allow it
  static constexpr bool SA = CW == 8;                    // one buffer of x fragments: 168 registers a wave
  static constexpr int BK = 64, ROWB = BK * 2, PPR = BK / 8, UR = 64 / PPR;      // a stage row's bytes, 16-byte pieces; rows per DMA instruction
  static constexpr int ROWS = BM + BN, STAGE = ROWS * ROWB;
  static constexpr int UNITS = ROWS / UR, LPS_LO = UNITS / 4, N_HI = UNITS % 4, LPS_HI = LPS_LO + (N_HI ? 1 : 0);
  static constexpr int XQ = BM / UR / 4;                                         // DMA units q < XQ are x rows for every wave
  static constexpr int LDC = BN + 8;
  // partial sums of the k-slices (NH passes over the row tiles) / row statistics
  static constexpr int NH = WK > 1 && CW * TM * TN * G > 80 ? 2 : 1;
  static constexpr int PART = GLU ? 0 : WK > 1 ? CW * TM / NH * TN * G * 1024 : (BM * (BN / 8) * 8 + 1023) / 1024 * 1024;
  static constexpr int TAIL = PART + BM * LDC * 2;
  static constexpr int NST = cmin(16, (159 * 1024 - KH_LN_LDS - TAB) / STAGE), PD = NST - 1;  // as many stages as fit, but at most 16
  static constexpr int TAB_OFF = cmax(NST * STAGE, TAIL), TOUCH_OFF = TAB_OFF + TAB, LDS = TOUCH_OFF + CW * 256;   // (where prefetched dwords nobody reads land)
  static constexpr int OPC = BM * (BN / 8), OPT = (OPC + NT - 1) / NT;             // 16-byte output pieces: per tile, per thread
  static_assert(WM * WN * WK == CW && TM * MF * WM == BM && TN * MF * WN == BN && TM % NH == 0 && TM / NH * TN * G % WK == 0, "tile");
  static_assert(BM % 32 == 0 && XQ * UR * 4 == BM && ROWS % UR == 0, "whole DMA instructions");
  static_assert(NST >= 2 && LPS_HI * (PD - 1) < 63 && LDS + KH_LN_LDS <= 160 * 1024, "ring");
};

// CONV: x is an NHWC image and row m of the GEMM is output pixel m of a 3x3 convolution with padding 1 (K = 9 * Cin ordered
// (kh, kw, ci)): a stage is 64 channels of one tap, taps outside the image read zeros (an offset beyond the buffer).
// Rows come in segments of seg_rows (an image of a convolution that leaves statistics, everything otherwise) that start a tile of their own.
//
// COOP: the launch computes its own shrink, cooperatively.  These tiles fill every CU, so there is no idle CU for shrink
// workgroups beside the GEMM ones; instead EVERY workgroup first computes one piece of T -- 32 rows x 96 rank columns: the
// n_tiles = 4 x (ldt / 128) workgroups of a row block of 128 rows share that block's 4 row quarters x ldt / 128 column
// groups of T, workgroup n_blk takes quarter n_blk % 4 of group n_blk / 4 --, stores it write-through, zeroes the 32
// padding columns of its group, counts itself into the row block's counter and then runs its GEMM tile; before its first
// request for T (the last K tiles) it waits, bounded, for the row block's count and reads T past the L2.  A workgroup
// never waits before its own piece is out, so the launch makes progress in whatever order its workgroups become
// resident, as long as no OTHER launch whose workgroups wait for each other shares the device with it (the binding does
// not use this form on a second stream).
//
// IL: a launch whose tiles leave enough CUs idle brings the shrink along: its first il_blocks workgroups compute one 16 x 16 (or 32 x 32) tile
// of T each, store it write-through and count themselves into the counter of their 128 rows; the GEMM workgroups wait, bounded, for
// that count before their first request for T.  The shrink workgroups have the lowest ids and wait for nothing, so they are resident
// before anything waits for them.
//
// GRP: n_groups layers that read the same few rows in one launch (LoraGemmParams::grp, T given); a workgroup takes one tile of one layer.
enum { T_GIVEN = 0, T_COOP = 1, T_IL = 2, T_GRP = 3 };
using ILTileWide = SCfg<4, 2, 2>;               // the pieces beside 128 x 128 tiles: 64 x 64 ...
using ILTileNarrow = SCfg<4, 2, 1>;             // ... and 64 x 32 (il_narrow)
constexpr int il_lds(int waves) { return waves == 8 ? cmax(SHRINK16_LDS<8>, SCfg<8, 1, 1, 2>::LDS) : cmax(SHRINK16_LDS<5>, SCfg<5, 1, 1, 3>::LDS); }
//
// XA: the layer is an attention's to_q; a tile's rows are queries of one sample, its columns whole heads, and the epilogue runs the cross-attention on
// them (xattn_tile.h).
template <class C, bool CONV, int TMODE, bool XA = false>
__global__ __launch_bounds__(C::NT, TMODE == T_COOP ? 1 : C::CW == 8 ? 3 : 2) void lora_gemm_fine_kernel(const LoraGemmParams p0, const int seg_rows, const int seg_tiles) {
#if __HIP_DEVICE_COMPILE__   // the host pass only needs the kernel's symbol (it cannot lower the buffer-resource type)
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int BM = C::BM, BN = C::BN, TM = C::TM, TN = C::TN, KS = C::KS, NST = C::NST, PD = C::PD;
  constexpr int BK = C::BK, ROWB = C::ROWB, UR = C::UR, PPR = C::PPR, STAGE = C::STAGE, LPS_LO = C::LPS_LO, LPS_HI = C::LPS_HI, XQ = C::XQ;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool producer = wave >= C::CW;                 // the last four waves move operands, the others compute
  const int pw = C::CW == 4 || producer ? wave & 3 : wave & (C::CW - 1), wm = pw / (C::WK * C::WN), wn = pw / C::WK % C::WN, wk = pw % C::WK;
  const int lr = lane % C::MF, lg = lane / C::MF;      // row inside an MFMA tile, 16-byte (8-byte) piece of a k-step

  constexpr bool COOP = TMODE == T_COOP, GRP = TMODE == T_GRP;
  // GRP: the row tiles of a layer's columns follow each other on one XCD, so that W comes from memory once
  LoraGemmParams pg;
  int gm_blk = 0, gn_blk = 0;
  if constexpr (GRP) {
    const int local = (int)blockIdx.x >> 3, tile = local / p0.m_tiles * 8 + ((int)blockIdx.x & 7), layer = tile / p0.n_tiles;
    if (layer >= p0.il_blocks) return;                 // (il_blocks: the number of layers)
    gm_blk = local % p0.m_tiles;
    gn_blk = tile - layer * p0.n_tiles;
    const uint64_t* const g = p0.grp + (size_t)layer * 5;
    pg = p0;
    pg.w = reinterpret_cast<const bf16_t*>(g[0]);
    pg.bias = reinterpret_cast<const bf16_t*>(g[1]);
    pg.b_cat = reinterpret_cast<const bf16_t*>(g[2]);
    pg.t_ext = reinterpret_cast<const bf16_t*>(g[3]);
    pg.y = reinterpret_cast<bf16_t*>(g[4]);
  }
  const LoraGemmParams& p = GRP ? pg : p0;
  if constexpr (TMODE == T_IL) {
    if ((int)blockIdx.x < p.il_blocks) {
      constexpr bool BIG = BM == 128 && BN == 128;
      const int r = p.r_used > 0 ? p.r_used : p.R, size = BIG ? 64 : p.il_tile, gx = (p.M + size - 1) / size, ct = BIG ? p.il_cols : (r + size - 1) / size;
      const int bx = (int)blockIdx.x % gx, by = (int)blockIdx.x / gx;
      // padding to a multiple of 8 (the XCD map of the rest); idle waves
      if (by >= (BIG ? ct : ct * (p.ldt / p.R)) || (!BIG && wave >= p.il_waves)) return;
      if (BIG && wave >= 4) {
        // The piece is the work of waves 0 .. 3.  When most of its own loads are out, the others hint the next launch's weights (by the GEMM workgroups
        // in front of their own operands the 1024 x 1024 step took 2 % longer) and fetch what is left of the XCD's block of W into its L2: M 2048 /
        // N 1280 / K 1280, rank 96, weights from HBM / from the memory-side cache 17.7 / 16.8 us, 17.9 / 18.1 by the computing waves as in the other
        // forms, 20.1 / 16.4 by nobody.  (The piece's barriers wait until these waves have ended.)
        const int xcd = (int)blockIdx.x & 7, wgs = (gx * ct - xcd + 7) / 8, KT1 = p.K / BK;
        char* lds = smem + C::TOUCH_OFF + (wave - 4) * 256;
        auto touch = [&](int t) {
          const int rows = p.xr_n * BN, row0 = (xcd % p.xg_n) * rows, i = ((int)blockIdx.x >> 3) * 256 + tid - 256;
          // (the last, shorter block by its true width: 3952 / 640 / 640 20.1 us instead of 19.7 with the constant)
          if (t + 8 <= KT1) kh_touch_rows<8>(p.w, p.N, p.K, row0, rows, t, 8, lds, i, wgs * 256);
          else kh_touch_rows(p.w, p.N, p.K, row0, rows, t, 8, lds, i, wgs * 256);
        };
        __builtin_amdgcn_s_sleep(127);                       // 8128 clocks, about 10 stages of the K loop
        const bool hints = il_prefetch_by_idle_waves(p);
        if (hints) kh_prefetch_lines_idle(p.pf, p.pf_lines, lds, (int)blockIdx.x, gx * ct, tid - 256, 256);
        for (int t = p.pf[0] != nullptr ? 24 : 8; t < KT1; t += 8) {   // (a caller that hints has had these weights hinted, too)
          touch(t);
          if (t >= 24) __builtin_amdgcn_s_sleep(48);
        }
        __builtin_amdgcn_s_waitcnt(0);                        // (nothing lands in LDS that is no longer this workgroup's)
        return;
      }
      ShrinkParams sp;
      sp.x = p.x; sp.a_cat = p.a_cat; sp.col_scale = p.col_scale; sp.t = const_cast<bf16_t*>(p.t_ext);
      sp.M = p.M; sp.K = p.K; sp.R = p.ldt;
      sp.ln_part = p.ln_part; sp.ln_ca1 = p.ln_ca1; sp.ln_ca2 = p.ln_ca2; sp.ln_eps = p.ln_eps;
      const int r0 = by / ct * p.R + by % ct * size;
      static_assert(cmax(ILTileWide::LDS, ILTileNarrow::LDS) <= C::TOUCH_OFF || !BIG, "the shrink tiles' rings");
      static_assert(il_lds(5) <= C::LDS, "the shrink tiles' rings");
      if constexpr (BIG) {
        if (il_narrow(p)) lora_shrink_tile<ILTileNarrow, true, 256>(sp, bx * 64, by * 32, smem);
        else lora_shrink_tile<ILTileWide, true, 256>(sp, bx * 64, by * 64, smem);
      } else if (il_lds(8) <= C::LDS && p.il_waves == 8) {
        if (size == 16) lora_shrink16_tile<8, true>(sp, bx * 16, r0, smem);
        else lora_shrink_tile<SCfg<8, 1, 1, 2>, true, 512>(sp, bx * 32, r0, smem);
      } else {
        if (size == 16) lora_shrink16_tile<5, true>(sp, bx * 16, r0, smem);
        else lora_shrink_tile<SCfg<5, 1, 1, 3>, true, 320>(sp, bx * 32, r0, smem);
      }
      __builtin_amdgcn_s_waitcnt(0);                          // this thread's write-through stores have completed
      __syncthreads();
      if (tid == 0) __hip_atomic_fetch_add(p.il_cnt + bx * size / 128, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
  }
  const int bid = (int)blockIdx.x - (TMODE == T_IL ? p.il_blocks : 0), n_wg = (int)gridDim.x - (TMODE == T_IL ? p.il_blocks : 0);
  // tile of this workgroup: XCD b % 8 owns a block of xr_m x xr_n tiles (its W rows stay in its L2)
  const int xcd = bid & 7, local = bid >> 3;
  const int m_blk = GRP ? gm_blk : (xcd / p.xg_n) * p.xr_m + local / p.xr_n;
  const int n_blk = GRP ? gn_blk : (xcd % p.xg_n) * p.xr_n + local % p.xr_n;
  if (!GRP && (local / p.xr_n >= p.xr_m || m_blk >= p.m_tiles || n_blk >= p.n_tiles)) return;  // padding of the grid
  const int M = p.M, N = p.N, K = p.K;
  const int seg = m_blk / seg_tiles, m0 = seg * seg_rows + (m_blk % seg_tiles) * BM, n0 = n_blk * BN;
  const int seg_end = (seg + 1) * seg_rows, rows = (seg_end < M ? seg_end : M) - m0;   // rows of this tile that exist (may exceed BM)
  // T made by a launch in front: its rank columns are extra K tiles
  constexpr bool EXT = !CONV;
  const int KT1 = K / BK, r_ext = p.r_used > 0 ? p.r_used : p.R;
  const int KT = KT1 + (EXT && p.t_ext != nullptr ? (r_ext + BK - 1) / BK : 0);
  const bool has_hi = pw < C::N_HI;

  if constexpr (COOP) {
    static_assert(SCfg<4, 1, 3>::LDS <= C::TOUCH_OFF && BM == 128, "the shrink piece's rings fit the GEMM ring; four quarters per row block");
    // this workgroup's piece of T = bf16((x . A_cat^T) * col_scale) (with a folded LayerNorm in front: the form documented at
    // ShrinkParams), then the padding columns, then the arrival
    const int q4 = n_blk & 3, grp = n_blk >> 2;
    ShrinkParams sp;
    sp.x = p.x; sp.a_cat = p.a_cat; sp.col_scale = p.col_scale; sp.t = const_cast<bf16_t*>(p.t_ext);
    sp.M = M; sp.K = K; sp.R = p.ldt;
    sp.ln_part = p.ln_part; sp.ln_ca1 = p.ln_ca1; sp.ln_ca2 = p.ln_ca2; sp.ln_eps = p.ln_eps;
    // (a quarter that starts past the last row has nothing to compute: the tile's addressing assumes m0 < M)
    if (m0 + 32 * q4 < M) lora_shrink_tile<SCfg<4, 1, 3>, true, C::NT>(sp, m0 + 32 * q4, grp * 128, smem);
    if (tid < 128) {   // columns 96 .. 127 of the group: 32 rows x 4 pieces of 16 bytes
      const int row = m0 + 32 * q4 + (tid >> 2);
      if (row < M) {
        uint32_t* dst = reinterpret_cast<uint32_t*>(const_cast<bf16_t*>(p.t_ext) + (size_t)row * p.ldt + grp * 128 + 96 + (tid & 3) * 8);
#pragma unroll
        for (int e = 0; e < 4; ++e) __hip_atomic_store(dst + e, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __builtin_amdgcn_s_waitcnt(0);                          // this thread's write-through stores have completed
    __syncthreads();
    if (tid == 0) __hip_atomic_fetch_add(p.il_cnt + m_blk, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // of a stage row, the piece that a 16-byte piece is stored as: 16 rows at one piece fill the 64 banks
  auto swz = [](int row) { return (PPR == 8 ? row >> 1 : row) & (PPR - 1); };
  // DMA of this lane: unit u = pw + 4*q covers stage rows u*UR .. u*UR+UR-1 (x rows, W rows); LDS slot = lane: row
  // lane/PPR, physical piece lane%PPR, which holds logical piece (lane%PPR) ^ swz(row).  Formed by the waves that move operands only (large tiles kept
  // these offsets over the computing waves' loop, in scratch memory; 1 / 1280 / 1280 8.7 -> 8.45 us, 154 / 640 / 2048 9.6 -> 9.45), or by all ahead of the
  // branch where that is faster (988 / 1280 / 1280 12.7 us instead of 13.05).
  constexpr uint32_t OOB = 0x80000000u;                // every buffer here is shorter than 2 GiB
  uint32_t voff[LPS_HI], voff2[EXT ? LPS_HI : 1];
  int tapmask[CONV ? XQ : 1];                          // CONV: bit t = tap t of this lane's row is inside the image
  constexpr bool AHEAD = C::CW == 4 && BM * BN < 128 * 128 && !(BM == 32 && BN == 32);
  // (behind the branch the kernel's arguments would be a load of their own: here they come with the others)
  if constexpr (C::CW == 4 && !AHEAD && BM * BN <= 128 * 128) asm volatile("" ::"s"(p.x), "s"(p.w), "s"(p.t_ext), "s"(p.b_cat), "s"(p.ldt), "s"(p.t_nsplit));
  auto offsets = [&] {
#pragma unroll
    for (int q = 0; q < LPS_HI; ++q) {
      int u = pw + 4 * q;
      u = u < C::UNITS ? u : C::UNITS - 1;               // never issued (has_hi), keep the offset valid
      const int r = u * UR + lane / PPR;
      const uint32_t pcb = (uint32_t)(((lane % PPR) ^ swz(r)) * 16);
      if (CONV && q < XQ) {
        int row = m0 + r; row = row < M ? row : M - 1;
        const int wo = row % p.conv_wo, t2 = row / p.conv_wo, ho = t2 % p.conv_ho, nb = t2 / p.conv_ho;
        const int hi0 = ho * p.conv_stride - 1, wi0 = wo * p.conv_stride - 1;
        int mask = 0;
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
          const int hi = hi0 + tap / 3, wi = wi0 + tap % 3;
          mask |= (hi >= 0 && hi < p.conv_h && wi >= 0 && wi < p.conv_w) ? (1 << tap) : 0;
        }
        tapmask[q < XQ ? q : 0] = mask;
        // relative to one row and one pixel in front of the image (the buffer's base), so that it is never negative
        voff[q] = (uint32_t)(((nb * p.conv_h + hi0 + 1) * p.conv_w + wi0 + 1) * p.conv_cin) * 2u + pcb;
      } else if (q < XQ) {
        voff[q] = (uint32_t)(m0 + r) * (uint32_t)K * 2u + pcb;        // rows past M lie beyond the buffer: zeros
      } else {
        voff[q] = (uint32_t)(n0 + r - BM) * (uint32_t)K * 2u + pcb;
      }
      if (EXT && p.t_ext != nullptr)
        voff2[q] = q < XQ ? ((uint32_t)(m0 + r) * (uint32_t)p.ldt + (uint32_t)(p.t_nsplit > 0 ? (n0 / p.t_nsplit) * p.R : 0)) * 2u + pcb
                          : (uint32_t)(n0 + r - BM) * (uint32_t)p.R * 2u + pcb;
    }
  };
  if constexpr (AHEAD) offsets();
  // fragments: row lr of each block of MF rows; of a k-step the lane's 16-byte piece lg (16x16x16: its 8 bytes lg)
  constexpr bool HALF = C::ORD == 4 && C::MF == 16;
  using Frag = typename std::conditional<HALF, s16x4, bf16x8>::type;
  using Acc = typename std::conditional<C::MF == 32, f32x16, f32x4>::type;
  struct Fr { Frag a[KS][TM], b[KS][TN]; };
  int fa[KS], fb[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    const int po = HALF ? ((2 * wk + (lg >> 1)) ^ swz(lr)) * 16 + (lg & 1) * 8 : ((C::MF == 16 ? 4 * (C::ORD == 0 ? k : wk) + lg : 2 * wk + lg) ^ swz(lr)) * 16;
    fa[k] = (wm * (BM / C::WM) + lr) * ROWB + po;
    fb[k] = (BM + wn * (BN / C::WN) + lr) * ROWB + po;
  }
  auto read_frags = [&](int st, Fr& f) {
#pragma unroll
    for (int k = 0; k < KS; ++k) {
#pragma unroll
      for (int i = 0; i < TM; ++i) f.a[k][i] = *reinterpret_cast<const Frag*>(smem + st + fa[k] + i * C::MF * ROWB);
#pragma unroll
      for (int j = 0; j < TN; ++j) f.b[k][j] = *reinterpret_cast<const Frag*>(smem + st + fb[k] + j * C::MF * ROWB);
    }
  };
  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4 * C::G; ++e) acc[i][j][e] = 0.f;
  auto mfma = [&](const Frag& x, const Frag& w, Acc& c) {
    const Frag& u = C::XW ? x : w;
    const Frag& v = C::XW ? w : x;
    if constexpr (HALF) c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(u, v, c, 0, 0, 0);
    else if constexpr (C::MF == 32) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(u, v, c, 0, 0, 0);
    else c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(u, v, c, 0, 0, 0);
  };
  auto mma = [&](const Fr& f) {
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) mfma(f.a[k][i], f.b[k][j], acc[i][j]);
  };

  // K loop.  Step t: tile t is in the computing waves' registers (cur); tile t+1 becomes visible at the barrier, after which
  // every wave has read tile t out of its stage, so that stage takes tile t + NST.  Both kinds of waves pass KT barriers.
  // (the epilogue's per-row and per-column terms are the producers' to fetch: ten registers less in the computing waves)
  float* sMu = reinterpret_cast<float*>(smem + C::LDS);      // [LNR] mean, [LNR] 1/std, [BN] x 2
  constexpr int LNR = cmax(BM, 128);
  float* sRs = sMu + LNR;
  float* sc1 = sRs + LNR;
  float* sc2 = sc1 + BN;
  static_assert((2 * LNR + 2 * BN) * 4 <= KH_LN_LDS, "per-row and per-column terms");
  typedef XAttnFine<cmax(BN / 64, 1), 256, C::LDC> XAttn;
  XAttn kv;                                            // XA: the keys and values, in the producers
  if (producer) {
    if constexpr (!AHEAD) offsets();
    const size_t x_bytes = CONV ? (size_t)(M / (p.conv_ho * p.conv_wo)) * p.conv_h * p.conv_w * p.conv_cin * 2 : (size_t)M * K * 2;
    const size_t x_lead = CONV ? (size_t)(p.conv_w + 1) * p.conv_cin * 2 : 0;
    const rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(p.x) - x_lead), 0,
                                                           (int)(x_bytes + x_lead), 0x00020000);
    const rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.w), 0, (int)((size_t)N * K * 2), 0x00020000);
    const bool has_t = EXT && p.t_ext != nullptr;
    const rsrc_t rs_t = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(has_t ? p.t_ext : p.x), 0,
                                                           has_t ? (int)((size_t)M * p.ldt * 2) : 0, 0x00020000);
    const rsrc_t rs_bx = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(has_t ? p.b_cat : p.w), 0,
                                                            has_t ? (int)((size_t)N * p.R * 2) : 0, 0x00020000);
    // CONV: K tiles are requested in order, so the tap and the channel offset of the next request are running scalars
    int cv_tap = 0, cv_kw = 0, cv_c0 = 0, cv_shift = 0, cv_row = 0;
    uint32_t xvo[XQ];
#pragma unroll
    for (int q = 0; q < XQ; ++q) xvo[q] = (!CONV || (tapmask[CONV ? q : 0] & 1)) ? voff[q] : OOB;
    auto issue = [&](int t, int st) {                    // K tile t into the ring stage at byte offset st
      char* stage = smem + st;
      const int so = t * ROWB;
      if (EXT && t >= KT1) {                             // columns of T and B_cat; past the last rank column: zeros
        if ((COOP || TMODE == T_IL) && t == KT1) {
          // first request for T: wait (bounded) until every workgroup of these 128 rows has delivered its piece
          if (lane == 0) {
            int it = 0, want = p.n_tiles;
            if (TMODE == T_IL) {
              const int left = M - m0 / 128 * 128;
              if (BM == 128 && BN == 128) want = ((left < 128 ? left : 128) + 63) / 64 * p.il_cols;
              else want = ((left < 128 ? left : 128) + p.il_tile - 1) / p.il_tile * ((r_ext + p.il_tile - 1) / p.il_tile) * (p.ldt / p.R);
            }
            while (__hip_atomic_load(p.il_cnt + m0 / 128, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < want && ++it < (1 << 20))
              __builtin_amdgcn_s_sleep(8);
            if (it >= (1 << 20)) {
              __hip_atomic_store(p.il_cnt + (p.M + 127) / 128, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              __hip_atomic_fetch_add(&kh_coop_timeout_count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
          }
        }
        const int c = (t - KT1) * BK;
#pragma unroll
        for (int q = 0; q < LPS_HI; ++q) {
          if (q < LPS_LO || has_hi) {
            const int r = (pw + 4 * q) * UR + lane / PPR, col = c + ((lane % PPR) ^ swz(r)) * 8;
            const uint32_t vo = col < r_ext ? voff2[EXT ? q : 0] : OOB;
            // T was written inside this launch, maybe on another XCD: read past the (non-coherent) L2
            if ((COOP || TMODE == T_IL) && q < XQ) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_t, (lptr_t)(stage + (pw + 4 * q) * 1024), 16, vo, c * 2, 0, 17 /* sc0 sc1 */);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(q < XQ ? rs_t : rs_bx, (lptr_t)(stage + (pw + 4 * q) * 1024), 16, vo, c * 2, 0, 0);
          }
        }
        return;
      }
#pragma unroll
      for (int q = 0; q < LPS_HI; ++q) {
        if (q < LPS_LO || has_hi) {
          lptr_t dst = (lptr_t)(stage + (pw + 4 * q) * 1024);
          if (q < XQ) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_x, dst, 16, xvo[q], CONV ? (cv_shift + cv_c0) * 2 : so, 0, 0);
          else __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_w, dst, 16, voff[q], so, 0, 0);
        }
      }
      if (CONV) {
        cv_c0 += BK;
        if (cv_c0 == p.conv_cin) {
          cv_c0 = 0; ++cv_tap; ++cv_kw; cv_shift += p.conv_cin;
          if (cv_kw == 3) { cv_kw = 0; cv_row += p.conv_w * p.conv_cin; cv_shift = cv_row; }
#pragma unroll
          for (int q = 0; q < XQ; ++q) xvo[q] = ((tapmask[CONV ? q : 0] >> cv_tap) & 1) ? voff[q] : OOB;
        }
      }
    };
    // until at most n of this wave's younger K tiles are outstanding (and its LDS reads are done)
    auto wait_younger = [&](int n) {
      if (has_hi) wait_tiles<LPS_HI, PD - 1>(n); else wait_tiles<LPS_LO, PD - 1>(n);
    };

    // requested now, used after the K loop (older than every DMA load, so no wait falls in between)
    constexpr int CP = (BN + 255) / 256;
    const int ptid = tid - C::CT;
    KhLnTileStats<GRP ? cmin(BM, 128) : BM, 256> ln_stats;
    float c1v[CP], c2v[CP];
    uint16_t biasv[CP];
    if (p.ln_part != nullptr) ln_stats.load(p.ln_part, m0, M, ptid);
    if constexpr (XA) kv.load(p, m0, n0, ptid);
#pragma unroll
    for (int c = 0; c < CP; ++c) {
      const int col = n0 + (ptid + 256 * c < BN ? ptid + 256 * c : 0);
      c1v[c] = p.ln_part != nullptr ? p.ln_c1[col] : 0.f;
      c2v[c] = p.ln_part != nullptr ? p.ln_c2[col] : 0.f;
      biasv[c] = p.ln_part == nullptr && p.bias != nullptr ? reinterpret_cast<const uint16_t*>(p.bias)[col] : (uint16_t)0;
    }
    // K tiles go out in order as their stages come free; those of a T that is being made beside this tile once the loop is under
    // way (the wait for it holds up every step behind it; 300 / 640 / 640, rank 64, on 32 x 64 tiles: 10.4 us with it in front of the loop, 6.6 here)
    const int KTI = TMODE == T_IL ? KT1 : KT;
#pragma unroll
    for (int t = 0; t < PD; ++t)
      if (t < KTI) issue(t, t * STAGE);
    wait_younger(KTI - 1);
    ring_barrier();
    if (KTI > PD) issue(PD, PD * STAGE);
    int st = 0, t = 0;                                 // stage of tile t
    for (; t + NST < KTI; ++t) {
      wait_younger(PD - 1);
      ring_barrier();
      issue(t + NST, st);
      st = st + STAGE == NST * STAGE ? 0 : st + STAGE;
    }
    int next = KTI;                                    // first tile that is not out yet
    for (; t + 1 < KT; ++t) {
      if constexpr (TMODE == T_IL)
        for (; next < KT && next < t + NST && (t >= 4 || 2 * t >= KT1 - 1); ++next) issue(next, next % NST * STAGE);
      wait_younger(next - t - 2);
      ring_barrier();
    }
    if (p.ln_part != nullptr) ln_stats.finish(K, p.ln_eps, ptid, sMu, sRs, false);
#pragma unroll
    for (int c = 0; c < CP; ++c)
      if (const int col = ptid + 256 * c; col < BN) { sc1[col] = c1v[c]; sc2[col] = p.ln_part != nullptr ? c2v[c] : bf16_bits_to_f32(biasv[c]); }
  } else {
    // W's lines into the XCD's L2 ahead of the ring (kh_touch_rows): 24 stages now, then 8 every 8 stages (M 988, N 1280, K 1280: 10.4 ->
    // 9.9 us; K 5120 38.4 -> 30.5; x, which the launch in front has just written, is not worth it)
    // (lines by a constant division only for large tiles: 154 / 1280 / 2048 took 10.9 us with it instead of 10.7, 3952 / 640 / 640 20.1 instead of 19.9)
    auto touch = [&](int t, auto n) {
      if (!GRP && !(TMODE == T_IL && BM == 128 && BN == 128) && t < KT1)
        kh_touch_rows<(BM * BN > 128 * 128) ? decltype(n)::value : 0>(p.w, N, K, (xcd % p.xg_n) * p.xr_n * BN, p.xr_n * BN, t, n, smem + C::TOUCH_OFF + pw * 256, local * C::CT + tid, p.xr_m * p.xr_n * C::CT);
    };
    // (a GEGLU projection has so many columns that its first tile queued behind 24 stages: 988 / 10240 / 1280 from HBM 36.4 -> 34.7 us).
    // The next launch's weights come behind this launch's own first lines, from waves that wait for them anyway.
    constexpr int TOUCH = C::GLU ? 8 : 24;
    constexpr std::integral_constant<int, 8> EIGHT{};
    touch(0, std::integral_constant<int, TOUCH>{});
    if (!GRP && !(TMODE == T_IL && BM == 128 && BN == 128 && il_prefetch_by_idle_waves(p)))
      kh_prefetch_lines(p.pf, p.pf_lines, smem + C::TOUCH_OFF + pw * 256, bid, n_wg, tid, C::CT);
    uint16_t* gtab = reinterpret_cast<uint16_t*>(smem + C::TAB_OFF);
    if constexpr (C::GLU) {
#pragma unroll 4
      for (int i = tid; i < 2 * GTAB_N; i += C::CT) {
        const uint32_t bits = (uint32_t)(i >= GTAB_N ? 0x8000 + (i - GTAB_N) : i) + GTAB_LO;
        gtab[i] = (uint16_t)pack_bf16x2(kh_gelu_erf(bf16_lo(bits)), 0.f);
      }
    }
    ring_barrier();
    int st = 0;
    if constexpr (C::SA) {
      // Two waves per SIMD compute, so that one's reads run under the other's matrix instructions, and a wave has 168 registers: one set of x fragments,
      // each replaced behind the instruction of a k-step that used it last, and two fragments of W.  The barrier that shows the next stage lies behind the
      // reads of this stage's last fragments, three columns before its end.
      static_assert(TN >= 3 && C::MF == 16, "columns of a stage");
      constexpr int G = KS * TN, NB = G % 2 == 0 ? 2 : TN;   // columns of a stage; fragments of W in registers (a stage ends where it began)
      Frag a[TM], b[NB];
      auto read_a = [&](int st, int k, int i) { a[i] = *reinterpret_cast<const Frag*>(smem + st + fa[k] + i * C::MF * ROWB); };
      auto read_b = [&](int st, int g) { b[g % NB] = *reinterpret_cast<const Frag*>(smem + st + fb[g / TN] + g % TN * C::MF * ROWB); };
      auto stage = [&](auto last_tag) {
        constexpr bool LAST = decltype(last_tag)::value;
        int nxt = st;
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int k = g / TN, j = g % TN;
          if (!LAST && g == G - NB) {
            nxt = st + STAGE == NST * STAGE ? 0 : st + STAGE;
            wait_cnt<63, 0>();
            ring_barrier();
          }
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            mfma(a[i], b[g % NB], acc[i][j]);
            if (j == TN - 1 && (k + 1 < KS || !LAST)) {
              read_a(k + 1 < KS ? st : nxt, k + 1 < KS ? k + 1 : 0, i);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
          if (g + NB < G) read_b(st, g + NB);
          else if (!LAST) read_b(nxt, g + NB - G);
          __builtin_amdgcn_sched_barrier(0);
        }
        st = nxt;
      };
#pragma unroll
      for (int i = 0; i < TM; ++i) read_a(0, 0, i);
#pragma unroll
      for (int g = 0; g < NB; ++g) read_b(0, g);
      for (int t = 0; t + 1 < KT; ++t) {
        if ((t & 7) == 0) touch(t + TOUCH, EIGHT);
        stage(std::false_type{});
      }
      stage(std::true_type{});
    } else if constexpr (!C::DB) {
      // One set of W fragments, replaced one by one behind the matrix instructions that used them last, and two of x, a k-step each: the
      // reads of the next k-step run under the matrix instructions of this one.  (A whole stage read and then multiplied takes the sum of both
      // where the operands arrive in time: GEGLU on 64 x 320 tiles, 2048 / 5120 / 640, 25.2 -> 24.0 us.)  The barrier that shows the next stage lies before the last k-step, whose fragments have
      // been read by then, so that the stage can be filled again.
      Frag a[2][TM], b[TN];
      auto read_a = [&](int st, int k, int set) {
#pragma unroll
        for (int i = 0; i < TM; ++i) a[set][i] = *reinterpret_cast<const Frag*>(smem + st + fa[k] + i * C::MF * ROWB);
      };
      auto read_b = [&](int st, int k, int j) { b[j] = *reinterpret_cast<const Frag*>(smem + st + fb[k] + j * C::MF * ROWB); };
      auto mma1 = [&](int set, int j) {
#pragma unroll
        for (int i = 0; i < TM; ++i) mfma(a[set][i], b[j], acc[i][j]);
      };
      auto kstep = [&](int set, int st_next, int k_next) {   // x in a[set]; the next k-step's fragments: step k_next of stage st_next
        read_a(st_next, k_next, 1 - set);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          mma1(set, j);
          read_b(st_next, k_next, j);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      auto next_stage = [&]() {
        st = st + STAGE == NST * STAGE ? 0 : st + STAGE;
        wait_cnt<63, 0>();
        ring_barrier();
      };
      read_a(0, 0, 0);
#pragma unroll
      for (int j = 0; j < TN; ++j) read_b(0, 0, j);
      if constexpr (KS == 2) {
        for (int t = 0; t + 1 < KT; ++t) {
          if ((t & 7) == 0) touch(t + TOUCH, EIGHT);
          kstep(0, st, 1);
          next_stage();
          kstep(1, st, 0);
        }
        kstep(0, st, 1);
      } else {
        int t = 0;
        for (; t + 2 < KT; t += 2) {
          if ((t & 7) == 0) touch(t + TOUCH, EIGHT);
          next_stage();
          kstep(0, st, 0);
          next_stage();
          kstep(1, st, 0);
        }
        if (t + 1 < KT) {
          next_stage();
          kstep(0, st, 0);
#pragma unroll
          for (int i = 0; i < TM; ++i) a[0][i] = a[1][i];
        }
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) mma1(KS == 2 ? 1 : 0, j);
    } else {
    Fr f0, f1;
    read_frags(0, f0);
    auto step = [&](const Fr& cur, Fr& nxt) {
      st = st + STAGE == NST * STAGE ? 0 : st + STAGE;
      wait_cnt<63, 0>();
      ring_barrier();
      read_frags(st, nxt);
      mma(cur);
    };
    int t = 0;
    for (; t + 2 < KT; t += 2) {
      if ((t & 7) == 0) touch(t + TOUCH, EIGHT);
      step(f0, f1);
      step(f1, f0);
    }
    if (t + 1 < KT) { step(f0, f1); mma(f1); }
    else mma(f0);
    }
  }

  // residual pieces of this thread, requested before the reductions
  u32x4 rr[C::OPT];
  if (p.res != nullptr) {
#pragma unroll
    for (int q = 0; q < C::OPT; ++q) {
      const int c = tid + q * C::NT, srow = c / (BN / 8), ch = c % (BN / 8);
      rr[q] = (c < C::OPC && srow < rows) ? *reinterpret_cast<const u32x4*>(p.res + (size_t)(m0 + srow) * N + n0 + ch * 8) : u32x4{0, 0, 0, 0};
    }
  }
  __syncthreads();   // the ring is dead: partial sums and the staging tiles reuse it
  if constexpr (XA)
    if (producer) kv.store(smem + (C::TAIL + 15) / 16 * 16, tid - C::CT);

  // the k-slices meet in LDS: every wave leaves all its tiles and finishes every WK-th of them
  f32x4* part = reinterpret_cast<f32x4*>(smem);
  bf16_t* sC = reinterpret_cast<bf16_t*>(smem + C::PART);
  auto finish = [&](const f32x4 s, int i, int j, int g) {   // the four outputs of group g of tile (i, j) in this lane
    const int at = (C::MF == 32 ? 8 * g : 0) + 4 * lg;       // first of the four: columns of row lr (XW: rows of column lr) of the tile
    const int row = wm * (BM / C::WM) + i * C::MF + (C::XW ? at : lr), col = wn * (BN / C::WN) + j * C::MF + (C::XW ? lr : at);
    if constexpr (C::XW) {
      f32x4 mu = {0.f, 0.f, 0.f, 0.f}, rs = {1.f, 1.f, 1.f, 1.f};
      if (p.ln_part != nullptr) { mu = *reinterpret_cast<const f32x4*>(sMu + row); rs = *reinterpret_cast<const f32x4*>(sRs + row); }
      const float c1 = sc1[col], c2 = sc2[col];
#pragma unroll
      for (int e = 0; e < 4; ++e) sC[(row + e) * C::LDC + col] = (bf16_t)(rs[e] * (s[e] - mu[e] * c1) + c2);
    } else {
      float mu = 0.f, rs = 1.f;
      if (p.ln_part != nullptr) { mu = sMu[row]; rs = sRs[row]; }
      const f32x4 c1 = *reinterpret_cast<const f32x4*>(sc1 + col), c2 = *reinterpret_cast<const f32x4*>(sc2 + col);
      bf16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (bf16_t)(rs * (s[e] - mu * c1[e]) + c2[e]);
      *reinterpret_cast<bf16x4*>(sC + row * C::LDC + col) = o;
    }
  };
  auto group = [&](const Acc& v, int g) { return f32x4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]}; };
  if constexpr (C::WK == 1) {
    if (!producer) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) finish(group(acc[i][j], 0), i, j, 0);
    }
  } else {
    constexpr int UH = TM / C::NH * TN * C::G;           // groups of a pass
#pragma unroll
    for (int h = 0; h < C::NH; ++h) {
      if (h > 0) __syncthreads();
      if (!producer) {
#pragma unroll
        for (int i = 0; i < TM / C::NH; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int g = 0; g < C::G; ++g) part[(pw * UH + (i * TN + j) * C::G + g) * 64 + lane] = group(acc[h * (TM / C::NH) + i][j], g);
      }
      __syncthreads();
      if (!producer) {
#pragma unroll
        for (int u = 0; u < UH / C::WK; ++u) {
          const int at = u * C::WK + wk, ij = at / C::G;
          f32x4 s = part[((pw - wk) * UH + at) * 64 + lane];
#pragma unroll
          for (int k = 1; k < C::WK; ++k) {              // slice after slice
            const f32x4 o = part[((pw - wk + k) * UH + at) * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] += o[e];
          }
          finish(s, h * (TM / C::NH) + ij / TN, ij % TN, at % C::G);
        }
      }
    }
  }
  __syncthreads();
  if constexpr (XA) {
    static_assert(C::WK == 1 && !C::GLU && !CONV && BN % 64 == 0 && C::LDC % 8 == 0 && (C::TAIL + 15) / 16 * 16 + XAttn::LDS_BYTES <= C::LDS, "cross-attention");
    static_assert(BN / 64 * (BM / 32) <= 8, "a wave per 32 queries of a head");
    if (wave < BN / 64 * (BM / 32)) XAttn::unit(p, sC, smem + (C::TAIL + 15) / 16 * 16, wave / (BM / 32), wave % (BM / 32), m0, n0, lane);
    return;
  }
  if constexpr (C::GLU) {
    // staged columns come in groups of 64 = 32 value columns then their 32 gate columns
    constexpr int OPR = BN / 16, GCH = (BM * OPR + C::NT - 1) / C::NT;
    const int out_ld = N / 2;
    const KhOut gout(p.y, (size_t)M * out_ld * 2);
    const uint16_t* gtab = reinterpret_cast<const uint16_t*>(smem + C::TAB_OFF);
#pragma unroll
    for (int q = 0; q < GCH; ++q) {
      const int c = tid + q * C::NT, srow = c / OPR, oc = c % OPR, grp = oc >> 2, sub = oc & 3;
      if (c >= BM * OPR || srow >= rows) continue;
      const u32x4 hv = *reinterpret_cast<const u32x4*>(sC + srow * C::LDC + grp * 64 + sub * 8);
      const u32x4 gv = *reinterpret_cast<const u32x4*>(sC + srow * C::LDC + grp * 64 + 32 + sub * 8);
      u32x4 ar;                                            // gelu(gate) rounded to bf16 before the product
      bool outside = false;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t lo = gv[e] & 0xffffu, hi = gv[e] >> 16;
        const uint32_t olo = (lo & 0x7fffu) - GTAB_LO, ohi = (hi & 0x7fffu) - GTAB_LO;
        outside = outside || olo >= (uint32_t)GTAB_N || ohi >= (uint32_t)GTAB_N;
        const uint32_t ilo = (olo < (uint32_t)GTAB_N ? olo : 0u) + (lo >> 15) * GTAB_N;
        const uint32_t ihi = (ohi < (uint32_t)GTAB_N ? ohi : 0u) + (hi >> 15) * GTAB_N;
        ar[e] = (uint32_t)gtab[ilo] | ((uint32_t)gtab[ihi] << 16);
      }
      if (outside) {                                       // tiny, huge or non-finite gates: evaluate directly
#pragma unroll
        for (int e = 0; e < 4; ++e) ar[e] = pack_bf16x2(kh_gelu_erf(bf16_lo(gv[e])), kh_gelu_erf(bf16_hi(gv[e])));
      }
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = pack_bf16x2(bf16_lo(hv[e]) * bf16_lo(ar[e]), bf16_hi(hv[e]) * bf16_hi(ar[e]));
      gout.store16(((size_t)(m0 + srow) * out_ld + (n0 >> 1) + grp * 32 + sub * 8) * 2, o);
    }
    return;
  }
  const KhOut yout(p.y, (size_t)M * N * 2);
  float* sp = reinterpret_cast<float*>(smem);          // row statistics: [BM][BN / 8][2], the partial sums are dead
#pragma unroll
  for (int q = 0; q < C::OPT; ++q) {
    const int c = tid + q * C::NT, srow = c / (BN / 8), ch = c % (BN / 8);
    const bool ok = c < C::OPC && srow < rows;
    u32x4 o = ok ? *reinterpret_cast<const u32x4*>(sC + srow * C::LDC + ch * 8) : u32x4{0, 0, 0, 0};
    if (p.res != nullptr) {
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = pack_bf16x2(bf16_lo(o[e]) + bf16_lo(rr[q][e]), bf16_hi(o[e]) + bf16_hi(rr[q][e]));
    }
    if (ok) yout.store16(((size_t)(m0 + srow) * N + n0 + ch * 8) * 2, o);
    if (!CONV && p.st_part != nullptr) {
      float ps, pq;
      kh_piece_sums(o, ps, pq);
      if constexpr (BN == 128) {                         // the 16 pieces of a row sit in 16 neighbouring lanes
        ps = kh_row16_sum(ps);
        pq = kh_row16_sum(pq);
        if (ch == 0 && ok) kh_ln_store_stats(p.st_part, m0 + srow, M, n_blk, p.n_tiles, ps, pq);
      } else if (c < C::OPC) {
        *reinterpret_cast<u32x2*>(sp + 2 * c) = u32x2{__float_as_uint(ps), __float_as_uint(pq)};
      }
    }
    if (CONV && C::ORD != 0 && p.gn_part != nullptr && p.res != nullptr && ok) *reinterpret_cast<u32x4*>(sC + srow * C::LDC + ch * 8) = o;
  }
  if (!CONV && BN != 128 && p.st_part != nullptr) {
    __syncthreads();
    if (tid < BM && tid < rows) {
      float s = 0.f, q2 = 0.f;
#pragma unroll
      for (int ch = 0; ch < BN / 8; ++ch) { s += sp[2 * (tid * (BN / 8) + ch)]; q2 += sp[2 * (tid * (BN / 8) + ch) + 1]; }
      kh_ln_store_stats(p.st_part, m0 + tid, M, n_blk, p.n_tiles, s, q2);
    }
  }
  if constexpr (CONV && C::ORD != 0) if (p.gn_part != nullptr) {
    // GroupNorm statistics as a by-product (LoraGemmParams::gn_part): (sum, sum of squares) of the stored values plus the per-(image,
    // channel) term over this tile's pixels of one image and whole groups of channels; sums in fixed orders
    constexpr int PCS = BN / 8, RP = 25;                      // 16-byte pieces per row, row parts (those of the 64 x 160 kernel)
    float* colp = sp;                                         // [RP][BN][2]
    float* cols = colp + RP * BN * 2;                         // [BN][2]
    static_assert((RP * BN * 2 + BN * 2) * 4 <= C::PART, "column sums fit the dead partial sums");
    const int cg = p.gn_cg, ng = BN / cg, G = N / cg, nrow = rows < BM ? rows : BM;
    const float ad = (tid < BN && p.gn_add != nullptr) ? (float)p.gn_add[(size_t)seg * N + n0 + tid] : 0.f;
    __syncthreads();
    if (tid < RP * PCS) {
      const int ch = tid % PCS, prt = tid / PCS;
      float cs[8], cq[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) cs[e] = cq[e] = 0.f;
#pragma unroll
      for (int i = 0; i < (BM + RP - 1) / RP; ++i) {
        const int r = prt + i * RP;
        if (r < nrow) {
          const u32x4 v = *reinterpret_cast<const u32x4*>(sC + r * C::LDC + ch * 8);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float a = bf16_lo(v[e]), b2 = bf16_hi(v[e]);
            cs[2 * e] += a; cq[2 * e] = fmaf(a, a, cq[2 * e]);
            cs[2 * e + 1] += b2; cq[2 * e + 1] = fmaf(b2, b2, cq[2 * e + 1]);
          }
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) *reinterpret_cast<f32x2*>(colp + (prt * BN + ch * 8 + e) * 2) = f32x2{cs[e], cq[e]};
    }
    __syncthreads();
    if (tid < BN) {
      float s = 0.f, q = 0.f;
#pragma unroll
      for (int prt = 0; prt < RP; ++prt) { const f32x2 v = *reinterpret_cast<const f32x2*>(colp + (prt * BN + tid) * 2); s += v[0]; q += v[1]; }
      *reinterpret_cast<f32x2*>(cols + tid * 2) = f32x2{s + (float)nrow * ad, q + 2.f * ad * s + (float)nrow * ad * ad};
    }
    __syncthreads();
    if (tid < ng) {
      float s = 0.f, q = 0.f;
      for (int c = tid * cg; c < (tid + 1) * cg; ++c) { s += cols[2 * c]; q += cols[2 * c + 1]; }
      *reinterpret_cast<f32x2*>(p.gn_part + (((size_t)seg * G + n0 / cg + tid) * seg_tiles + m_blk % seg_tiles) * 2) = f32x2{s, q};
    }
  }
#endif
}

// the tiles of a call and their XCD grid
template <class C>
bool plan_tiles(LoraGemmParams& p, int seg_rows) {
  if (p.N % C::BN != 0 || (p.t_nsplit > 0 && p.t_nsplit % C::BN != 0)) return false;
  p.m_tiles = p.M / seg_rows * ((seg_rows + C::BM - 1) / C::BM);
  p.n_tiles = p.N / C::BN;
  const KhXcdGrid g = kh_xcd_grid(p.m_tiles, p.n_tiles, C::BM, C::BN);
  p.xg_n = g.gn; p.xr_m = g.rm; p.xr_n = g.rn;
  return p.st_part == nullptr || p.n_tiles <= KH_LN_SLOTS;
}

// ... and its shrink's: a CU each beside the GEMM's on every XCD; 16 x 16 where they fit (T is there sooner)
template <class C>
bool plan_il(LoraGemmParams& p) {
  if (!plan_tiles<C>(p, p.M) || il_lds(p.il_waves) > C::LDS) return false;
  const int r = p.r_used > 0 ? p.r_used : p.R;
  for (p.il_tile = 16; p.il_tile <= 32; p.il_tile *= 2) {
    const long pieces = (long)((p.M + p.il_tile - 1) / p.il_tile) * ((r + p.il_tile - 1) / p.il_tile) * (p.ldt / p.R);
    if ((pieces + 7) / 8 + (long)p.xr_m * p.xr_n > 32) continue;
    p.il_blocks = (int)((pieces + 7) / 8 * 8);
    return true;
  }
  return false;
}

template <class C, bool CONV, int TMODE = T_GIVEN, bool XA = false>
int launch_fine(LoraGemmParams p, hipStream_t stream) {
  const int seg_rows = CONV && p.gn_part != nullptr ? p.conv_ho * p.conv_wo : p.M;
  if (!plan_tiles<C>(p, seg_rows)) return KH_ERR_UNSUPPORTED;
  if constexpr (TMODE == T_IL && !(C::BM == 128 && C::BN == 128))
    if (!plan_il<C>(p)) return KH_ERR_UNSUPPORTED;
  if (hipError_t e = kh_allow_lds<lora_gemm_fine_kernel<C, CONV, TMODE, XA>>(C::LDS + KH_LN_LDS); e != hipSuccess) return (int)e;
  const unsigned grid = (unsigned)(TMODE == T_IL ? p.il_blocks : 0) + 8u * (unsigned)p.xr_m * (unsigned)p.xr_n;
  kh_launch(CONV ? KH_TAG_CONV : KH_TAG_LORA_GEMM, lora_gemm_fine_kernel<C, CONV, TMODE, XA>, dim3(grid), dim3(C::NT), (size_t)C::LDS + KH_LN_LDS, stream, p,
            seg_rows, (seg_rows + C::BM - 1) / C::BM);
  KH_RETURN_LAST_ERROR();
}

}  // namespace

// What the kernel takes, whatever the tile: whole 64-column stages, T given where there are rank columns, operands that one buffer
// descriptor spans.
bool lora_gemm_fine_ok(const LoraGemmParams& p) {
  const size_t lim = (size_t)1 << 31;
  if (p.grp != nullptr || p.sg_mode != 0 || p.xa_k != nullptr || p.K % 64 != 0 || (p.R > 0 && p.t_ext == nullptr)) return false;
  if (p.ldt % 8 != 0 || (size_t)p.N * p.K * 2 >= lim || (size_t)p.N * p.R * 2 >= lim || (size_t)p.M * (p.ldt > 0 ? p.ldt : 1) * 2 >= lim) return false;
  if (p.conv_cin == 0) return (size_t)p.M * p.K * 2 < lim;
  const size_t xb = ((size_t)(p.M / (p.conv_ho * p.conv_wo)) * p.conv_h + 1) * p.conv_w * p.conv_cin * 2 + 2 * (size_t)p.conv_cin;
  return p.conv_cin % 64 == 0 && xb < lim && p.R == 0;
}

// Forms: order 0 on 64 x 80 (0), 128 x 80 (1), 32 x 128 (2), 64 x 128 (3); order 4 on 32 x 160 (4), 64 x 160 (5), 64 x 80 (6);
// GEGLU on 64 x 320 (7), 128 x 320 (8), 160 x 320 (17), 192 x 320 (18); order 2 on 128 x 160 (9); order 0 on 32 x 32 (10), 32 x 64 (11), 64 x 64 (12);
// order 4 on 32 x 32 (13), 32 x 64 (14), 64 x 64 (15); order 0 on 128 x 128 (16), 128 x 160 (19), 160 x 160 (20), 192 x 160 (21).
//
// Order 2: eight waves of 64 x 80, two k-slices of four, and waves of their own for the operands, in place of eight 32 x 160 strips that did
// both.  us per launch, weights from HBM (strips, then four waves of 64 x 160): convolutions 640 -> 640 at 2 x 64 x 64 70.9 -> 63.0, 1920 -> 640 190 -> 167, 960 -> 320 at
// 2 x 128 x 128 198 -> 173; (four, then eight) 640 -> 640 at 2 x 64 x 64 62.0 -> 59.2, 320 -> 320 at 2 x 128 x 128 69.9 -> 66.1, 1280 -> 1280 at 2 x 64 x 64 239 -> 214, 1920 -> 640 159 both;
// linear layers with adapters 8192 / 640 / 640 20.1 -> 18.6, 8192 / 640 / 2560 44.3 -> 42.0.
//
// Few rows: the shrink of a call with adapters runs inside the launch, on CUs that its tiles leave idle (T_IL).  The shrink's sums are those of
// its own launch and the tiles' those of the order, so one launch and two give the same bits.
template <class F>
static int with_il_tile(int form, F f) {
  switch (form) {
    case 0: return f(FCfg<64, 80, 0>{});
    case 1: return f(FCfg<128, 80, 0>{});
    case 2: return f(FCfg<32, 128, 0>{});
    case 3: return f(FCfg<64, 128, 0>{});
    case 4: return f(FCfg<32, 160, 4>{});
    case 5: return f(FCfg<64, 160, 4>{});
    case 7: return f(FCfg<64, 320, 0, true>{});
    case 8: return f(FCfg<128, 320, 0, true>{});
    case 10: return f(FCfg<32, 32, 0>{});
    case 11: return f(FCfg<32, 64, 0>{});
    case 12: return f(FCfg<64, 64, 0>{});
    case 13: return f(FCfg<32, 32, 4>{});
    case 14: return f(FCfg<32, 64, 4>{});
    case 15: return f(FCfg<64, 64, 4>{});
    default: return KH_ERR_UNSUPPORTED;
  }
}

// the pieces of T (16 or 32 wide) that a launch of this form brings along; 0: it leaves no CUs for them
static int shrink_beside(LoraGemmParams& p, int form) {
  if (p.t_ext == nullptr || p.R <= 0 || p.ldt != (p.t_nsplit > 0 ? p.N / p.t_nsplit : 1) * p.R) return 0;
  p.il_waves = lora_shrink_waves(p.M, p.K, p.ldt, p.R, p.r_used);
  if (p.il_waves != 5 && p.il_waves != 8) return 0;
  return with_il_tile(form, [&](auto c) { return plan_il<decltype(c)>(p) ? KH_OK : KH_ERR_UNSUPPORTED; }) == KH_OK ? p.il_tile : 0;
}

// GEGLU projections: of 64 / 128 / 160 / 192 x 320 tiles and the 256 x 320 ones of lora_gemm_wide.hip (-2) those whose rounds of the CUs take least; -1: 128 x 128 tiles.
// A round costs about 100 rows more than its tiles have (its start, its epilogue; the 256-row tiles, whose waves move their own operands, 150).
// us per launch without adapters, weights from HBM, before (in several rounds 128 x 320 on four computing waves, or 128 x 128) -> now: N 10240 / K 1280, M 512 22.7 ->
// 22.1, 1024 34.5 -> 31.4, 1152 48 -> 34.6, 1280 55.5 -> 35.5, 1400 57.4 -> 40.3, 1536 47.8 -> 40.5, 1800 69.8 -> 56.0, 1976 71.4 -> 58.1, 2048 (256 rows) 55.8, 58.9 on 128;
// N 5120 / K 640, M 1100 17.8 -> 16.0, 2304 28.7 -> 21.5, 3072 30.1 -> 25.7, 3952 44.2 -> 35.4, 4096 (256 rows) 33.7, 4608 50.3 -> 40.5, 6000 64.6 -> 50.6, 7200 77.7 -> 62.8,
// 8192 (256 rows) 64.2, 69.6 on 192.
// The 192-row tile has eight registers more than its wave: four lane constants and a fragment of the last stage go through scratch, 36 bytes a lane, all of it
// ahead of the loop over K or behind it.
int lora_gemm_geglu_form(const LoraGemmParams& p) {
  if (!lora_gemm_fine_ok(p) || p.st_part != nullptr || p.res != nullptr || p.N % 320 != 0 || p.t_nsplit % 320 != 0) return -1;
  if ((long)((p.M + 63) / 64) * (p.N / 320) <= 128) return -1;           // (up to half a round of 64 x 320 the 128 x 128 tiles are as fast)
  const auto cost = [&](int bm, int more) {
    const KhXcdGrid g = kh_xcd_grid((p.M + bm - 1) / bm, p.N / 320, bm, 320);
    return ((long)g.rm * g.rn + 31) / 32 * (bm + more);
  };
  constexpr struct { int form, bm; } tiles[] = {{7, 64}, {8, 128}, {17, 160}, {18, 192}};
  int best = -1;
  long least = 0;
  for (const auto& t : tiles)
    if (const long c = cost(t.bm, 100); best < 0 || c < least) { least = c; best = t.form; }
  return lora_gemm_wide_ok(p) && cost(256, 150) < least ? -2 : best;
}

// Which of them, for a layer whose sums follow `order`; -1 where none fits and the larger tiles of the other families win.  A
// convolution that leaves GroupNorm statistics does so per 64 rows.
//
// Linear layers: a CU's time is the rows it streams, BM + BN of K columns each, so the tile with the fewest of them whose workgroups fit
// one round of the 256 CUs (a workgroup fills a CU, so a second round costs as much as the first).  Where the launch is to bring its shrink along,
// the first that leaves the CUs for 16 x 16 pieces of it; where the loop is long enough to hide the larger pieces, the first that leaves them for
// 32 x 32 ones if there is no other, or if its loop (us: 3 + 2.9e-5 a row and column of K) and those pieces (8 + 2.3e-3 K) are through before the larger
// tile's loop (16 / 32: 512 / 1280 / 5120, 96 40.3 / 24.6, 154 21.6 / 20.5, 700 / 640 / 2560, 64 22.4 / 14.1, 400 / 1280 / 2048, 96 16.2 / 12.5; against that 308 / 1280 /
// 2048, 64 12.0 / 13.3, 512 / 640 / 2560, 64 13.7 / 14.7, 308 / 1280 / 1280, 64 8.4 / 11.3); else two launches.  A T that is given leaves all CUs to the tiles (988 / 1280 / 1280, 64 11.3 us on tiles that leave some -> 10.0, K 5120 35.6 -> 30.7; 700 / 640 /
// 2560 22.4 -> 11.2): the order of the sums is the same.
// us per call, weights from HBM (M / N / K, rank: without the tiles of 32 and 64 columns -> now): 1 / 1280 / 1280, 16 12.1 -> 8.4;
// 77 / 1280 / 2048, 32 14.1 -> 9.2; 154 / 1280 / 2048, 96 13.4 -> 10.7; 64 / 1280 / 5120, 32 36.7 -> 17.4; 256 / 1280 / 5120, 32 32.1 -> 20.6;
// 512 / 1280 / 1280, 32 10.1 -> 9.3; 300 / 640 / 640, 64 7.3 -> 6.4; no adapters: 154 / 640 / 2048 12.1 -> 8.3, 655 / 1280 / 2048 12.2 -> 11.1.
int lora_gemm_fine_form(const LoraGemmParams& p, int order) {
  if (!lora_gemm_fine_ok(p)) return -1;
  const long hw = p.gn_part != nullptr ? (long)p.conv_ho * p.conv_wo : p.M, nb = p.M / hw;
  auto tiles_of = [&](int bm, int bn) { return nb * ((hw + bm - 1) / bm) * (p.N / bn); };
  auto fits = [&](int bm, int bn) { return p.N % bn == 0 && p.t_nsplit % bn == 0 && (p.st_part == nullptr || p.N / bn <= KH_LN_SLOTS) && tiles_of(bm, bn) <= 256; };
  auto pieces_of = [&](int size) { return (long)((p.M + size - 1) / size) * (((p.r_used > 0 ? p.r_used : p.R) + size - 1) / size) * (p.ldt / p.R); };
  if (p.geglu) {
    const int form = order == 0 ? lora_gemm_geglu_form(p) : -1;
    return form >= 0 ? form : -1;
  }
  if (order == 2) return 9;
  if (p.conv_cin > 0) return p.gn_part != nullptr ? (80 % p.gn_cg == 0 && fits(64, 80) ? 6 : 5) : fits(32, 160) ? 4 : 5;
  struct Tile { int form, bm, bn; };
  constexpr Tile tiles0[] = {{10, 32, 32}, {11, 32, 64}, {12, 64, 64}, {0, 64, 80}, {2, 32, 128}, {3, 64, 128}, {1, 128, 80}};
  constexpr Tile tiles4[] = {{13, 32, 32}, {14, 32, 64}, {15, 64, 64}, {4, 32, 160}, {5, 64, 160}};
  const bool stats = p.st_part != nullptr, brings = p.t_ext != nullptr && p.a_cat != nullptr && p.R > 0;   // (a T that is given needs no CUs)
  const Tile* const all = order == 0 ? tiles0 : tiles4;
  const Tile* const end = all + (order == 0 ? 7 : 5);
  const int width = order == 0 ? 128 : 160;
  auto first = [&](int piece, const Tile* stop) {       // piece: the shrink's pieces beside the tiles, 0: none needed
    for (const Tile* t = all; t != stop; ++t) {
      if (!fits(t->bm, t->bn) || (stats && t->bn != width)) continue;
      if (piece == 0) return t;
      if (tiles_of(t->bm, t->bn) + pieces_of(piece) > 256) continue;      // (a part of what shrink_beside asks, and much cheaper)
      if (LoraGemmParams q = p; shrink_beside(q, t->form) == piece) return t;
    }
    return stop;
  };
  if (brings) {
    const Tile* const a = first(16, end);
    const Tile* const b = p.K >= 1280 ? first(32, a) : a;      // (a smaller tile, if any)
    auto loop = [&](const Tile* t) { return 3 + 2.9e-5 * p.K * (t->bm + t->bn); };
    const double pieces = 8 + 2.3e-3 * p.K;
    if (b != a && (a == end || (loop(b) < loop(a) && pieces < loop(a)))) return b->form;
    if (a != end) return a->form;
  }
  const Tile* const t = first(0, end);
  return t != end ? t->form : -1;
}

// Many rows, sums in the order of the 128 x 128 kernel: of 128 x 128 (convolutions) and 128 / 160 / 192 x 160 tiles those whose rounds of the CUs stream the fewest rows
// (us go with rounds x (BM + BN): one round of 160 x 160 / 192 x 160 at 1536 / 3840 / 1280 21.1 / 21.3, of 256 x 128 24.3; 1800 rows: two of the first 34.0, one of the second
// 23.6 and of the third 24.9; convolutions 320 -> 320 at 2 x 104 x 152, two rounds of 128 / 160 / 192 61.5 / 62.7 / 70.7).  A round is what the fullest XCD gets.
static long rounds_cost(const LoraGemmParams& p, int bm, int bn) {
  const KhXcdGrid g = kh_xcd_grid((p.M + bm - 1) / bm, (p.N + bn - 1) / bn, bm, bn);
  return ((long)g.rm * g.rn + 31) / 32 * (bm + bn);
}

// -1: none divides the columns, or others win.
// Convolutions, before on 128 x 128 tiles whose waves both move operands and compute, two workgroups to a CU or one (us, weights from HBM): 320 -> 320 at 2 x 72 x 72 47.7 -> 27.6,
// 2 x 96 x 96 52.6 -> 34.2, 2 x 104 x 152 81.3 -> 60.2, 2 x 128 x 120 80.7 -> 60.6, 640 -> 320 at 2 x 96 x 96 95 -> 60.5, 2 x 88 x 120 108 -> 69.5, 640 -> 640 at 2 x 64 x 76 94 -> 65,
// 1280 -> 640 at 2 x 56 x 56 166 -> 99, 1280 -> 1280 at 4 x 24 x 24 100 -> 83, 2 x 36 x 36 90 -> 87.
// Where 128 x 128 is one round (that kernel, these tiles): few columns are as fast there or faster (320 -> 320 at 1 x 104 x 88 25.6, 27.6, at 2 x 68 x 68 26.2, 27.7,
// 960 -> 320 at 2 x 64 x 72 64.0, 65.7), many are faster here (640 -> 1280 at 2 x 36 x 32 53.7, 46.8); 640 may be either (640 -> 640 at 2 x 46 x 46 43.4, 43.5, at 2 x 48 x 48 45.1, 45.9,
// 1920 -> 640 at 2 x 56 x 56 137 both, 320 -> 640 at 2 x 52 x 52 27.5, 26.8, 960 -> 640 at 2 x 48 x 56 70.7, 66.0, 1280 -> 640 at 2 x 48 x 52 96.2, 84.1) and stays there.  So do
// short sums (128 -> 320 at 2 x 64 x 64 14.3, 16.4, 256 -> 320 at 2 x 70 x 70 22.5, 23.8) and few tiles (1280 -> 1280 at 8 x 8 88, 112).
// Linear layers without row statistics (which go by 128 columns), before on 256 x 128 or 128 x 128 tiles, T given: 1300 / 3840 / 1280 21.8 -> 19.0, 1536 25.5 -> 21.1, 1800
// 25.4 -> 23.6, 5120 / 1280 / 1280 22.7 -> 19.8, K 5120 71.7 -> 60.6, 4608 / 1920 / 640 25.8 -> 21.4, 6000 27.5 -> 24.2, 10000 / 640 / 640 14.5 -> 12.9.
int lora_gemm_rounds_form(const LoraGemmParams& p) {
  const bool conv = p.conv_cin > 0;
  if (!lora_gemm_fine_ok(p) || p.gn_part != nullptr || p.geglu) return -1;
  const long tiles = (long)((p.M + 127) / 128) * ((p.N + 127) / 128);
  // one round of 128 x 128 with a long sum (us, T given or none, before on tiles whose eight waves do both): 2304 / 1280 / 5120 53.5 -> 42.4, 2432 51.4 -> 41.8, K 2560 29.5 -> 23.2,
  // 4608 / 640 / 2560, R 128 47.3 -> 41.9 with its shrink, 700 / 3840 / 2560 26.9 -> 25.7; half a round is as fast there (1024 / 2048 / 4096 25.7, 26.3 here), and so are shorter sums
  if (!conv && tiles > 128 && tiles <= 256 && p.K >= 2560 && p.N % 128 == 0 && p.t_nsplit % 128 == 0 && (p.st_part == nullptr || p.N / 128 <= KH_LN_SLOTS) && rounds_cost(p, 128, 128) == 256) return 16;
  if (p.st_part != nullptr) return -1;
  if (conv ? tiles <= 128 || (rounds_cost(p, 128, 128) == 256 && (p.K < 2560 || p.N < 1024)) : tiles <= 256) return -1;
  int best = -1;
  long least = conv ? 0 : rounds_cost(p, 256, 128);
  constexpr struct { int form, bm, bn; } all[] = {{16, 128, 128}, {19, 128, 160}, {20, 160, 160}, {21, 192, 160}};
  for (const auto& t : all) {
    if (p.N % t.bn != 0 || (p.t_nsplit > 0 && p.t_nsplit % t.bn != 0) || (!conv && t.form == 16)) continue;
    if (const long c = rounds_cost(p, t.bm, t.bn); least == 0 || c < least) { least = c; best = t.form; }
  }
  return best;
}

int lora_gemm_fine_launch(const LoraGemmParams& p, int form, hipStream_t stream) {
  const bool conv = p.conv_cin > 0;
  // (a forced form comes here without the rule above)
  if (!lora_gemm_fine_ok(p) || (p.geglu ? (form != 7 && form != 8 && form != 17 && form != 18) || p.st_part != nullptr || p.res != nullptr : form == 7 || form == 8 || form == 17 || form == 18)) return KH_ERR_UNSUPPORTED;
  switch (form) {
    case 0: return conv ? KH_ERR_UNSUPPORTED : launch_fine<FCfg<64, 80, 0>, false>(p, stream);
    case 1: return conv ? KH_ERR_UNSUPPORTED : launch_fine<FCfg<128, 80, 0>, false>(p, stream);
    case 2: return conv ? KH_ERR_UNSUPPORTED : launch_fine<FCfg<32, 128, 0>, false>(p, stream);
    case 3: return conv ? KH_ERR_UNSUPPORTED : launch_fine<FCfg<64, 128, 0>, false>(p, stream);
    case 4: return conv ? launch_fine<FCfg<32, 160, 4>, true>(p, stream) : launch_fine<FCfg<32, 160, 4>, false>(p, stream);
    case 5: return conv ? launch_fine<FCfg<64, 160, 4>, true>(p, stream) : launch_fine<FCfg<64, 160, 4>, false>(p, stream);
    case 6: return conv ? launch_fine<FCfg<64, 80, 4>, true>(p, stream) : KH_ERR_UNSUPPORTED;
    case 7: return launch_fine<FCfg<64, 320, 0, true>, false>(p, stream);
    case 8: return launch_fine<FCfg<128, 320, 0, true>, false>(p, stream);
    case 17: return launch_fine<FCfg<160, 320, 0, true>, false>(p, stream);
    case 18: return launch_fine<FCfg<192, 320, 0, true>, false>(p, stream);
    case 16: return conv ? launch_fine<FCfg<128, 128, 0>, true>(p, stream) : launch_fine<FCfg<128, 128, 0>, false>(p, stream);
    case 19: return conv ? launch_fine<FCfg<128, 160, 0>, true>(p, stream) : launch_fine<FCfg<128, 160, 0>, false>(p, stream);
    case 20: return conv ? launch_fine<FCfg<160, 160, 0>, true>(p, stream) : launch_fine<FCfg<160, 160, 0>, false>(p, stream);
    case 21: return conv ? launch_fine<FCfg<192, 160, 0>, true>(p, stream) : launch_fine<FCfg<192, 160, 0>, false>(p, stream);
    case 9: return conv ? launch_fine<FCfg<128, 160, 2>, true>(p, stream) : launch_fine<FCfg<128, 160, 2>, false>(p, stream);
    case 10: return conv ? KH_ERR_UNSUPPORTED : launch_fine<FCfg<32, 32, 0>, false>(p, stream);
    case 11: return conv ? KH_ERR_UNSUPPORTED : launch_fine<FCfg<32, 64, 0>, false>(p, stream);
    case 12: return conv ? KH_ERR_UNSUPPORTED : launch_fine<FCfg<64, 64, 0>, false>(p, stream);
    case 13: return conv ? KH_ERR_UNSUPPORTED : launch_fine<FCfg<32, 32, 4>, false>(p, stream);
    case 14: return conv ? KH_ERR_UNSUPPORTED : launch_fine<FCfg<32, 64, 4>, false>(p, stream);
    case 15: return conv ? KH_ERR_UNSUPPORTED : launch_fine<FCfg<64, 64, 4>, false>(p, stream);
    default: return KH_ERR_UNSUPPORTED;
  }
}

// The cooperative form (see the kernel): the layers whose 128 x 160 tiles fill the chip -- exactly the shapes the rule in
// lora_gemm_pipe_launch gives these tiles --, T of one or several stacked layers with 128 packed rank columns each of which
// at most 96 are in use, four column tiles per 128 rank columns of T.
bool lora_gemm_fine_coop_ok(const LoraGemmParams& p) {
  if (!(p.t_ext != nullptr && p.a_cat != nullptr && p.col_scale != nullptr && p.il_cnt != nullptr)) return false;
  if (!lora_gemm_fine_ok(p) || p.conv_cin > 0 || p.geglu || p.t_nsplit % 160 != 0 || p.N % 160 != 0 || p.R != 128 || p.r_used <= 0 || p.r_used > 96 || p.ldt % 128 != 0) return false;
  const long tiles = (long)((p.M + 127) / 128) * ((p.N + 127) / 128), m128 = (p.M + 127) / 128, n160 = p.N / 160;
  if (!(tiles > 256 && tiles <= 384 && m128 * n160 <= 256)) return false;
  const bool t_ok = p.t_nsplit == 0 ? p.ldt == p.R : (p.N % p.t_nsplit == 0 && p.ldt == (p.N / p.t_nsplit) * p.R);
  return t_ok && n160 == 4 * (p.ldt / 128) && n160 <= KH_LN_SLOTS;
}

// this file's share of kh_lora_split_timeouts (synchronous)
int lora_gemm_fine_coop_timeouts(int* count, int clear) {
  int v = 0;
  hipError_t e = hipMemcpyFromSymbol(&v, HIP_SYMBOL(kh_coop_timeout_count), sizeof(int), 0, hipMemcpyDeviceToHost);
  if (e != hipSuccess) return (int)e;
  *count = v;
  if (clear && v != 0) {
    const int zero = 0;
    e = hipMemcpyToSymbol(HIP_SYMBOL(kh_coop_timeout_count), &zero, sizeof(int), 0, hipMemcpyHostToDevice);
    if (e != hipSuccess) return (int)e;
  }
  return KH_OK;
}

int lora_gemm_fine_launch_coop(const LoraGemmParams& p, hipStream_t stream) {
  if (!lora_gemm_fine_coop_ok(p)) return KH_ERR_UNSUPPORTED;
  return launch_fine<FCfg<128, 160, 2>, false, T_COOP>(p, stream);
}

// Shrink inside the launch (IL): the form of lora_gemm_fine_form, where its tiles leave the CUs.
// us per call, weights from HBM, two launches -> one: M 154 / N 1280 / K 2048, rank 96 14.9 -> 10.7; 512 / 1280 / 1280, rank 32 12.9 -> 9.3;
// 512 / 1280 / 5120 30.9 -> 24.0; 988 / 1280 / 1280, rank 16 15.8 -> 12.2 (64 x 80 tiles and two launches 13.7); GEGLU 640 / 10240 / 1280, rank 16 36.3 -> 33.4.
int lora_gemm_fine_il_form(LoraGemmParams p) {
  if (p.a_cat == nullptr || p.col_scale == nullptr || p.il_cnt == nullptr || p.conv_cin > 0) return -1;
  const int form = lora_gemm_pipe_fine_form(p);
  const int piece = shrink_beside(p, form);
  return piece == 16 || (piece == 32 && p.K >= 1280) ? form : -1;   // (the rule of the forms)
}

// Many layers on the same few rows (the context projections of every cross-attention).  Bound by their weights, which come from memory once each: a
// tile is 128 columns of a layer, and so many of its rows, up to 160, that no second workgroup asks for those weights.  us per launch, two-per-CU tiles of
// 128 x 128 -> these: 120 layers of 2048 -> 1280, 154 rows, rank columns 128 284 -> 188 (3.4 TB/s of weights), 77 rows, 64 199 -> 151, 308 rows, 64 440 -> 269,
// 20 rows, 64 175 -> 136; 20 layers of 2048 -> 640, 154 rows, 128 34.8 -> 19.3; 60 layers, 600 rows, 64 316 -> 239.
template <int BM>
static int launch_grouped(LoraGemmParams p, int n_groups, hipStream_t stream) {
  using C = FCfg<BM, 128, 0>;
  p.m_tiles = (p.M + BM - 1) / BM;
  p.n_tiles = p.N / 128;
  p.il_blocks = n_groups;
  const long tiles = (long)n_groups * p.n_tiles, grid = (tiles + 7) / 8 * 8 * p.m_tiles;
  if (grid > 0x7fffffffL) return KH_ERR_TOO_LARGE;
  if (hipError_t e = kh_allow_lds<lora_gemm_fine_kernel<C, false, T_GRP>>(C::LDS + KH_LN_LDS); e != hipSuccess) return (int)e;
  kh_launch(KH_TAG_LORA_GEMM, lora_gemm_fine_kernel<C, false, T_GRP>, dim3((unsigned)grid), dim3(512), (size_t)C::LDS + KH_LN_LDS, stream, p, p.M, p.m_tiles);
  KH_RETURN_LAST_ERROR();
}

bool lora_gemm_fine_grouped_ok(const LoraGemmParams& p) {
  const size_t lim = (size_t)1 << 31;
  return p.K % 64 == 0 && p.N % 128 == 0 && p.M <= 640 && (size_t)p.M * p.K * 2 < lim && (size_t)p.N * p.K * 2 < lim && (size_t)p.N * (p.R > 0 ? p.R : 1) * 2 < lim &&
         (size_t)p.M * p.ldt * 2 < lim;
}

int lora_gemm_fine_launch_grouped(const LoraGemmParams& p, int n_groups, hipStream_t stream) {
  const int tiles = (p.M + 159) / 160, rows = (p.M + tiles - 1) / tiles;
  return rows <= 32 ? launch_grouped<32>(p, n_groups, stream) : rows <= 64 ? launch_grouped<64>(p, n_groups, stream) : rows <= 96 ? launch_grouped<96>(p, n_groups, stream)
         : rows <= 128 ? launch_grouped<128>(p, n_groups, stream) : launch_grouped<160>(p, n_groups, stream);
}

// Shrink inside the launch, 128 x 128 tiles: form 1 of lora_gemm_pipe_il_form.  Against the kernel of lora_gemm_pipe.hip, whose eight
// waves both moved operands and computed 64 x 32 each, us per call with statistics, rank 96, weights from the memory-side cache / from HBM:
// 2048 / 1280 / 1280 17.2 -> 16.8 / 20.0 -> 17.7; 2048 / 1280 / 5120 41.5 -> 38.5 / 54.5 -> 43.3; rank 64 without statistics 18.0 -> 16.3 / -.
int lora_gemm_fine_launch_il128(LoraGemmParams p, hipStream_t stream) {
  using C = FCfg<128, 128, 0>;
  p.il_cols = il_col_tiles(p);
  p.il_blocks = ((p.M + 63) / 64 * p.il_cols + 7) / 8 * 8;
  return launch_fine<C, false, T_IL>(p, stream);
}

int lora_gemm_fine_launch_il(LoraGemmParams p, int form, hipStream_t stream) {
  p.il_waves = lora_shrink_waves(p.M, p.K, p.ldt, p.R, p.r_used);
  return with_il_tile(form, [&](auto c) { return launch_fine<decltype(c), false, T_IL>(p, stream); });
}

// A query projection with its cross-attention in the epilogue (the shapes of lora_gemm_pipe_xattn_ok: whole 128-row and 128-column tiles, samples of
// whole 128-row tiles).  Fewer than 1024 rows: the tile of the projection alone, with the shrink beside it where 16 x 16
// pieces find CUs; else 128 x 128.  Bound by the operand stream like the projection alone; the attention adds 1 to 2 us at the end.  Against 128 x 128
// tiles whose eight waves both move operands and compute (lora_gemm_pipe.hip) and, below 1024 rows, a shrink in a launch of its own, us per call, weights
// from HBM, 77 keys: 512 / 1280 / 1280, rank 32 of 64 24.7 -> 11.3, rank 64 25.6 -> 15.1, without adapters 20.6 -> 11.2; 256 / 640 / 640, 16 18.0 -> 9.2;
// 768 / 1280 / 1280, 48 25.4 -> 15.0; 896, 64 26.0 -> 19.2; 1024, 16 23.0 -> 21.3; 1536, 32 23.1 -> 19.8; 2048, rank 96 24.0 -> 19.2, without 21.4 -> 19.0.
// Same bits.  Pieces of T that do not fit beside the tiles on every XCD stay there (2304 / 1280 / 1280, 128 26.8).
namespace {
template <class F>
int with_xattn_tile(int form, F f) {
  switch (form) {
    case 2: return f(FCfg<32, 128, 0>{});
    case 3: return f(FCfg<64, 128, 0>{});
    case 11: return f(FCfg<32, 64, 0>{});
    case 12: return f(FCfg<64, 64, 0>{});
    default: return f(FCfg<128, 128, 0>{});
  }
}

// the projection alone, as the rule of the forms sees it
LoraGemmParams xattn_projection(const LoraGemmParams& p) {
  LoraGemmParams q = p;
  q.xa_k = nullptr;
  return q;
}

// form and whether it brings the shrink; form -1: lora_gemm_pipe.hip's tiles
struct XAttnForm { int form; bool il; };
XAttnForm xattn_form(const LoraGemmParams& p, bool may_wait) {
  LoraGemmParams q = xattn_projection(p);
  if (!lora_gemm_fine_ok(q)) return {-1, false};
  const bool brings = may_wait && q.R > 0 && q.a_cat != nullptr && q.il_cnt != nullptr;
  if (brings && lora_gemm_pipe_il_form(p) != 0) return il_fits_beside(q, il_col_tiles(q)) ? XAttnForm{16, true} : XAttnForm{-1, false};
  if (q.M >= 1024) return {16, false};
  // whole heads: the first of 64 and 128 columns in the order of their operand rows
  for (const int form : {11, 12, 2, 3}) {
    const int bm = form == 2 || form == 11 ? 32 : 64, bn = form == 2 || form == 3 ? 128 : 64;
    if ((long)(q.M / bm) * (q.N / bn) <= 256) return {form, brings && shrink_beside(q, form) == 16};
  }
  return {16, false};
}
}  // namespace

int lora_gemm_fine_xattn_launches(const LoraGemmParams& p, bool may_wait) {
  const XAttnForm f = xattn_form(p, may_wait);
  return f.form < 0 ? 0 : p.R == 0 || f.il ? 1 : 2;
}

int lora_gemm_fine_launch_xattn(const LoraGemmParams& pin, bool may_wait, hipStream_t stream) {
  const XAttnForm f = xattn_form(pin, may_wait);
  if (f.form < 0) return KH_ERR_UNSUPPORTED;
  LoraGemmParams p = pin;
  if (!f.il) return with_xattn_tile(f.form, [&](auto c) { return launch_fine<decltype(c), false, T_GIVEN, true>(p, stream); });
  if (f.form == 16) {
    p.il_cols = il_col_tiles(p);
    p.il_blocks = ((p.M + 63) / 64 * p.il_cols + 7) / 8 * 8;
  } else {
    p.il_waves = lora_shrink_waves(p.M, p.K, p.ldt, p.R, p.r_used);
  }
  return with_xattn_tile(f.form, [&](auto c) { return launch_fine<decltype(c), false, T_IL, true>(p, stream); });
}
