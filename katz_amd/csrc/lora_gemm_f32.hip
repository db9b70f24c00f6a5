// K1, fp32: y = x W^T + b + ((x A_cat^T) * col_scale) B_cat^T (+ residual) at fp32 precision (gfx950).
//
// The reference's LoRA linear (diffusers-hf/src/diffusers/models/lora.py:222-232, :451-457) in full precision.
//
// The fp32 matrix instruction gives 256 FLOP per clock and CU, bf16's sixteen times that.  So every operand is split into three bf16 numbers
// that add up to it exactly (24 bits = 8 + 8 + 8), and six of their nine products are summed in fp32 by the bf16 instruction, all but the three that
// are at most 2^-24 of their factors' product each (x: lower parts of 2^-7 and 2^-16, W: 2^-8 and 2^-17): 2.7 times the fp32 rate.  The sums of 32
// columns are formed apart and added to the running sum with rounding (the matrix instruction truncates), so the error is below that of the fp32
// instruction: against 64 bits 1.0e-7 instead of 4.5e-7 at K 640, 2.5e-7 instead of 13e-7 at K 5120 (2-norm, normal inputs).
// Three bf16 numbers hold operands from 2^-103 on; tiles that meet smaller ones, or whose sums are not finite, are formed by the fp32 instruction
// (M 8192, N = K 640: 110 us where every tile is).
//
// Two launches.  The first forms T = (x A_cat^T) * col_scale (fp32 instruction, kept in fp32) and splits W and B_cat once into planes that the
// GEMM moves as they are; x is split by the GEMM itself (its planes would be one and a half times x's bytes, out and in again), whose rank
// columns are extra K steps.  What bounds the GEMM then: the matrix pipe, 1920 clocks of a 128 x 160 tile's 32-column stage at the 1.7 - 2
// GHz it leaves, beside about 1750 clocks of LDS traffic; measured 1.5 us a stage and 11 us around them.
// M 8192, N = K 640, rank 32: 84.6 -> 50.3 us for both launches (fp32 instruction on 64 x 64 tiles before).
#include "kh_common.h"

namespace {

struct F32Params {
  const float *x, *w, *bias, *t, *b_cat, *res;
  const void* planes;      // [W | B_cat] split into three bf16 planes (lora_split_w_kernel)
  float* y;
  int M, N, K, R;
};

constexpr int SHR_NS = 2, SHR_LDS = 8 * SHR_NS * 8192;   // the shrink's rings: blocks of a wave, bytes
constexpr int FB = 64;         // rows and columns of a tile of the form without planes
constexpr int FK = 32;         // K columns of a stage
constexpr int FLD = FK + 4;    // its staged row: 144 bytes, so the 16 rows of a ds_read_b128 phase fall into distinct banks

// eight K columns of a 32-row operand panel: lane (l32, lh) holds columns 4 lh .. 4 lh + 3 of row l32, so element e of both
// operands feeds one matrix instruction (its two K columns are e and 4 + e)
__device__ __forceinline__ f32x16 mma8(const f32x4 a, const f32x4 b, f32x16 c) {
#pragma unroll
  for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], c, 0, 0, 0);
  return c;
}

// a barrier that waits for this wave's own LDS accesses, kept in place among them
__device__ __forceinline__ void stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);          // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int N>
__device__ __forceinline__ void vm_wait() {    // vmcnt = [15:14|3:0]
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// a = hi + mid + lo exactly, 8 bits of a's 24 each.  x: hi is the upper half of a (|mid| <= 2^-7 |a|, |lo| <= 2^-16 |a|).  Four at a time.
__device__ __forceinline__ void split4(const f32x4 v, u32x2& hi, u32x2& mid, u32x2& lo) {
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float a = v[2 * e], b = v[2 * e + 1];
    const uint32_t ah = __float_as_uint(a) & 0xffff0000u, bh = __float_as_uint(b) & 0xffff0000u;
    hi[e] = __builtin_amdgcn_perm(bh, ah, 0x07060302u);
    const float ar = a - __uint_as_float(ah), br = b - __uint_as_float(bh);
    uint32_t m = pack_bf16x2(ar, br);
    asm("" : "+v"(m));                         // (one conversion for both: the compiler would take the halves from two more)
    mid[e] = m;
    lo[e] = pack_bf16x2(ar - bf16_lo(m), br - bf16_hi(m));
  }
}
// W and B_cat, which are split once: hi is the number nearest to a (2^-8, 2^-17), so that no product left out exceeds 2^-24 of its factors'
__device__ __forceinline__ void split4_nearest(const f32x4 v, u32x2& hi, u32x2& mid, u32x2& lo) {
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float a = v[2 * e], b = v[2 * e + 1];
    hi[e] = pack_bf16x2(a, b);
    const float ar = a - bf16_lo(hi[e]), br = b - bf16_hi(hi[e]);
    mid[e] = pack_bf16x2(ar, br);
    lo[e] = pack_bf16x2(ar - bf16_lo(mid[e]), br - bf16_hi(mid[e]));
  }
}

// the smallest operand so far that is not zero: its bits shifted left by one, less one
__device__ __forceinline__ void track_least(const f32x4 v, uint32_t& least) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t t = (__float_as_uint(v[e]) << 1) - 1u;
    least = least < t ? least : t;
  }
}
// The three planes hold a number exactly where bf16 reaches down to its last bit, and as normal numbers from 2^-103 on.  Smaller ones would lose
// their lower planes (rows of 2^-118 came out 9e-6 off, of 2^-122 1.5e-4), so the tiles that meet them are formed by the fp32 instruction.
__device__ __forceinline__ bool too_small(uint32_t least) { return least < (24u << 24) - 1u; }

// W and B_cat as the GEMM's W operand: per stage of 32 K columns (those of W, then those of B_cat, zeros behind the last) and group of 16 rows
// three blocks of 1 KB, the planes hi, mid and lo, in the order in which the 64 lanes of a wave hold a matrix operand (lane 16 g + r: columns
// 8 g .. 8 g + 7 of row r), so that the GEMM moves whole blocks and reads them without an address computation or a bank conflict.
__device__ __forceinline__ void split_w_block(const F32Params& p, int block, int lane) {
  const int groups = (p.N + 15) / 16, t = block / groups, grp = block % groups, K1 = (p.K + FK - 1) / FK;
  const bool ext = t >= K1;
  const int row = grp * 16 + (lane & 15), k = (ext ? t - K1 : t) * FK + (lane >> 4) * 8, len = ext ? p.R : p.K;
  const float* src = (ext ? p.b_cat : p.w) + (size_t)row * len + k;
  const bool in = row < p.N;
  const f32x4 v0 = in && k < len ? *reinterpret_cast<const f32x4*>(src) : f32x4{0, 0, 0, 0};
  const f32x4 v1 = in && k + 4 < len ? *reinterpret_cast<const f32x4*>(src + 4) : f32x4{0, 0, 0, 0};
  u32x2 h[2], m[2], l[2];
  uint32_t least = 0xffffffffu;
  track_least(v0, least);
  track_least(v1, least);
  split4_nearest(v0, h[0], m[0], l[0]);
  split4_nearest(v1, h[1], m[1], l[1]);
  if (too_small(least)) h[0][0] = 0x7fc07fc0u;             // (NaN: no sum of this row of W will be finite)
  char* dst = const_cast<char*>(reinterpret_cast<const char*>(p.planes)) + (size_t)block * 3072 + lane * 16;
  *reinterpret_cast<u32x4*>(dst) = u32x4{h[0][0], h[0][1], h[1][0], h[1][1]};
  *reinterpret_cast<u32x4*>(dst + 1024) = u32x4{m[0][0], m[0][1], m[1][0], m[1][1]};
  *reinterpret_cast<u32x4*>(dst + 2048) = u32x4{l[0][0], l[0][1], l[1][0], l[1][1]};
}

// WM x WN waves of (16 TM) x 80 outputs
template <int WM_, int WN_, int TM_>
struct GCfg {
  static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = 5, NT = WM * WN * 64, BM = WM * TM * 16, BN = WN * 80;
  static constexpr int PLANE = BM * FK * 2, XST = 3 * PLANE, WST = BN / 16 * 3072, NSW = 3, WOFF = 2 * XST, FLAG = WOFF + NSW * WST, LDS = FLAG + 16;   // FLAG: x has an operand too small for its planes
  static constexpr int PI = BM * 8 / NT;                                  // pieces of four columns of x a thread has of a stage
  static constexpr int WB = BN / 16 * 3, DU = (WB + WM * WN - 1) / (WM * WN);   // blocks of W: of a stage, of a wave
  static constexpr int AHEAD = 3;                                         // stages of x on their way from memory
  static_assert(PI * NT == BM * 8 && PI <= TN && WB >= DU * WM * WN - WB && LDS <= 160 * 1024, "tile");
};

// y = x W^T + t B_cat^T + bias + res.  K, R: multiples of 4.
template <class C>
__global__ __launch_bounds__(C::NT, 2) void lora_gemm_f32_split_kernel(const F32Params p, const int n_tiles) {
#if __HIP_DEVICE_COMPILE__   // the host pass only needs the kernel's symbol (it cannot lower the buffer-resource type)
  typedef __amdgpu_buffer_rsrc_t rsrc_t;
  typedef __attribute__((address_space(3))) void* lptr_t;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int TM = C::TM, TN = C::TN, AHEAD = C::AHEAD;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const uint32_t tile = xcd_remap(blockIdx.x, gridDim.x);    // an XCD walks neighbouring tiles: its x rows stay in its L2
  const int m0 = (int)(tile / n_tiles) * C::BM, n0 = (int)(tile % n_tiles) * C::BN;
  const int K1 = (p.K + FK - 1) / FK, KT = K1 + (p.R + FK - 1) / FK;
  // x's row r of a stage, 16-byte piece c of a plane: pieces are exchanged so that 16 rows at one piece fill the banks
  auto at = [](int r, int c) { return r * (FK * 2) + ((c ^ (r >> 2)) & 3) * 16; };
  const int wm = wave / C::WN, wn = wave % C::WN;

  // This thread's pieces of x: eight neighbouring threads read the 128 bytes of a row.  Buffer loads, without a branch: the compiler then
  // knows how many younger loads to leave under way.  Columns past the end are offsets beyond the buffer (zeros).
  const int c4 = (tid & 7) * 4;
  const rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.x + (size_t)m0 * p.K), 0, 0x7fffffff, 0x00020000);
  const rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.R > 0 ? p.t + (size_t)m0 * p.R : p.x), 0, 0x7fffffff, 0x00020000);
  uint32_t least = 0xffffffffu;
  uint32_t offk[C::PI], offr[C::PI];
  int to[C::PI];
#pragma unroll
  for (int q = 0; q < C::PI; ++q) {
    const int r = (tid >> 3) + q * (C::NT / 8), row = r < p.M - m0 ? r : p.M - m0 - 1;      // (rows past the end are never stored)
    offk[q] = ((uint32_t)row * (uint32_t)p.K + (uint32_t)c4) * 4u;
    offr[q] = ((uint32_t)row * (uint32_t)p.R + (uint32_t)c4) * 4u;
    to[q] = at(r, c4 >> 3) + (c4 & 4) * 2;
  }
  auto load = [&](int t, f32x4 (&g)[C::PI]) {
    const bool ext = t >= K1;
    const int k = (ext ? t - K1 : t) * FK, len = ext ? p.R : p.K;
    const uint32_t past = (uint32_t)((len - 1 - k - c4) >> 31) << 31;        // beyond the buffer from column len on
#pragma unroll
    for (int q = 0; q < C::PI; ++q)
      g[q] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ext ? rt : rx, (ext ? offr[q] : offk[q]) | past, k * 4, 0));
  };
  auto store = [&](int t, int q, const f32x4 (&g)[C::PI]) {
    char* st = smem + (t & 1) * C::XST + to[q];
    u32x2 hi, mid, lo;
    split4(g[q], hi, mid, lo);
    *reinterpret_cast<u32x2*>(st) = hi;
    *reinterpret_cast<u32x2*>(st + C::PLANE) = mid;
    *reinterpret_cast<u32x2*>(st + 2 * C::PLANE) = lo;
  };
  // W's blocks by LDS DMA, three stages ahead (past the last stage the last one again; the last blocks twice where the waves' shares do not divide)
  const int groups = (p.N + 15) / 16, grp0 = n0 / 16;
  auto fetch = [&](int t, int st) {
    const int tt = t < KT ? t : KT - 1;
    const rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(p.planes)) + ((size_t)tt * groups + grp0) * 3072, 0,
                                                         (groups - grp0) * 3072, 0x00020000);      // (groups past the last: zeros)
#pragma unroll
    for (int u = 0; u < C::DU; ++u) {
      int blk = wave + u * (C::WM * C::WN);
      blk = blk < C::WB ? blk : blk - C::WM * C::WN;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lptr_t)(smem + C::WOFF + st + blk * 1024), 16, (uint32_t)(blk * 1024 + lane * 16), 0, 0, 0);
    }
  };

  // The six products that can weigh more than 2^-24, summed for the stage alone and then added: the matrix instruction cuts off
  // what it adds to, which on a running sum of one sign would build up.
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 x[3][TM], w[3][TN];
  int ax[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) ax[i] = at(wm * (TM * 16) + i * 16 + lr, lg);
  const int aw = C::WOFF + wn * 5 * 3072 + lane * 16;
  const char* xst = smem;                                    // x of the stage whose fragments are read next, W of it, W's place to fill
  int wst = 0, wfill = 0;
  auto read_x = [&](int s) {
#pragma unroll
    for (int i = 0; i < TM; ++i) x[s][i] = *reinterpret_cast<const bf16x8*>(xst + s * C::PLANE + ax[i]);
  };
  auto read_w = [&](int s) {
#pragma unroll
    for (int j = 0; j < TN; ++j) w[s][j] = *reinterpret_cast<const bf16x8*>(smem + wst + aw + (j * 3 + s) * 1024);
  };
  auto next_read = [&](int t) {                              // (from stage t on)
    xst = smem + (t & 1) * C::XST;
    wst = wst + C::WST == C::NSW * C::WST ? 0 : wst + C::WST;
  };
  auto next_fetch = [&](int t) {
    fetch(t, wfill);
    wfill = wfill + C::WST == C::NSW * C::WST ? 0 : wfill + C::WST;
  };
  // Stage t, whose fragments are in registers: its products -- product by product over all tiles, so that none waits for the one before it
  // --, behind a plane's last product the plane of stage t + 1 (which is visible), and between them stage t + 2's pieces of x are split and
  // stored.  W first: a lane then holds one output row and runs of four columns.
  auto stage = [&](int t, f32x4 (&g)[C::PI]) {
    next_read(t + 1);
    next_fetch(t + 3);
    __builtin_amdgcn_sched_barrier(0);
    constexpr int sx[6] = {1, 0, 0, 1, 2, 0}, sw[6] = {1, 2, 1, 0, 0, 0};    // (the heaviest last)
    f32x4 c[TM][TN];
#pragma unroll
    for (int q = 0; q < 6; ++q) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
          c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[sw[q]][j], x[sx[q]][i], q == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : c[i][j], 0, 0, 0);
      if (q == 1) read_w(2);
      if (q == 2) read_w(1);
      if (q == 3) read_x(1);
      if (q == 4) read_x(2);
      if (q == 5) { read_x(0); read_w(0); }
      if (q < C::PI) store(t + 2, q, g);
    }
    f32x4 was[C::PI];
#pragma unroll
    for (int q = 0; q < C::PI; ++q) was[q] = g[q];
    load(t + 2 + AHEAD, g);
#pragma unroll
    for (int q = 0; q < C::PI; ++q) track_least(was[q], least);       // (not in front of the loads: 64 rows, K 5120, N 1280 120 us, 125 .. 128 there)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[i][j] += c[i][j];
    // W of stage t + 2 has landed when only what was requested behind it is under way: x of the last stage, W and x of this one
    __builtin_amdgcn_sched_barrier(0);
    vm_wait<C::DU + 2 * C::PI>();
    stage_barrier();                                         // stage t + 1 has been read, stage t + 2 is there
  };
  f32x4 g[AHEAD][C::PI], g0[C::PI];                          // (loads past the last stage: zeros)
  int* const flag = reinterpret_cast<int*>(smem + C::FLAG);
  if (tid == 0) *flag = 0;
  load(0, g0);
  load(1, g[1]);
  load(2, g[2]);
  load(3, g[0]);
  __builtin_amdgcn_sched_barrier(0);
  next_fetch(0); next_fetch(1);
#pragma unroll
  for (int q = 0; q < C::PI; ++q) {
    store(0, q, g0);
    store(1, q, g[1]);
    track_least(g0[q], least);
    track_least(g[1][q], least);
  }
  __builtin_amdgcn_sched_barrier(0);
  load(4, g[1]);
  __builtin_amdgcn_sched_barrier(0);
  next_fetch(2);
  __builtin_amdgcn_sched_barrier(0);
  vm_wait<C::PI + C::DU>();                                  // W of the first two stages
  stage_barrier();
#pragma unroll
  for (int s = 0; s < 3; ++s) { read_x(s); read_w(s); }
  stage_barrier();
  static_assert(AHEAD == 3, "g[(t + 2) % 3]: stage t + 2");
  for (int t = 0; t < KT; t += AHEAD) {
#pragma unroll
    for (int d = 0; d < AHEAD; ++d) {
      if (t + d >= KT) break;
      stage(t + d, g[(d + 2) % AHEAD]);
    }
  }
  vm_wait<0>();                                              // (no load into LDS outlives the wave)
  if (too_small(least)) *flag = 1;
  stage_barrier();

  // A result that is not finite (an input that is not, an overflow, an operand too small for three bf16 numbers) says nothing about what full
  // products give: such waves form their tile again, with the fp32 instruction, straight from memory.
  bool bad = *flag != 0;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) bad = bad || !(fabsf(acc[i][j][e]) < __builtin_inff());
  if (__ballot(bad) != 0) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int part = 0; part < (p.R > 0 ? 2 : 1); ++part) {
      const float *xp = part ? p.t : p.x, *wp = part ? p.b_cat : p.w;
      const int len = part ? p.R : p.K;
      for (int k0 = 0; k0 < len; k0 += 16) {                 // lane lg holds columns k0 + 4 lg .. + 3 of both operands: element e of all lanes is a step
        const int k = k0 + 4 * lg;
        f32x4 xv[TM], wv[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int row = m0 + wm * (TM * 16) + i * 16 + lr;
          xv[i] = k < len ? *reinterpret_cast<const f32x4*>(xp + (size_t)(row < p.M ? row : p.M - 1) * len + k) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int row = n0 + wn * 80 + j * 16 + lr;
          wv[j] = k < len ? *reinterpret_cast<const f32x4*>(wp + (size_t)(row < p.N ? row : p.N - 1) * len + k) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[j][e], xv[i][e], c, 0, 0, 0);
            acc[i][j] += c;
          }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = m0 + wm * (TM * 16) + i * 16 + lr;
    if (row >= p.M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wn * 80 + j * 16 + 4 * lg;
      f32x4 o = acc[i][j];
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
#endif
}

template <class C>
int launch_split(const F32Params& p, hipStream_t s) {
  const long n_tiles = (p.N + C::BN - 1) / C::BN, tiles = (long)((p.M + C::BM - 1) / C::BM) * n_tiles;
  if (tiles > 0x7fffffff) return KH_ERR_TOO_LARGE;
  if (hipError_t e = kh_allow_lds<lora_gemm_f32_split_kernel<C>>(C::LDS); e != hipSuccess) return (int)e;
  kh_launch(KH_TAG_LORA_GEMM_F32, lora_gemm_f32_split_kernel<C>, dim3((unsigned)tiles), dim3(C::NT), (size_t)C::LDS, s, p, (int)n_tiles);
  KH_RETURN_LAST_ERROR();
}

// t = (x A_cat^T) * col_scale on 32 x 32 tiles; wave w takes the 32-column blocks w, w + 8, ... of K through a ring of its own in LDS (buffer
// loads of whole 128-byte lines; with every lane reading its own row the L1's tags bound it: 12 us at M 8192, K 640, rank 32), the
// eight partial tiles meet in a fixed order.  x is read R / 32 times in all.  That is the first `shrink` workgroups; the others split W and B_cat, a
// block per wave.
__global__ __launch_bounds__(512) void lora_prepare_f32_kernel(const F32Params p, const float* __restrict__ a_cat, const float* __restrict__ col_scale,
                                                               const int shrink, const int blocks) {
#if __HIP_DEVICE_COMPILE__   // the host pass only needs the kernel's symbol (it cannot lower the buffer-resource type)
  typedef __amdgpu_buffer_rsrc_t rsrc_t;
  typedef __attribute__((address_space(3))) void* lptr_t;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, lh = lane >> 5;
  if ((int)blockIdx.x >= shrink) {
    const int block = ((int)blockIdx.x - shrink) * 8 + wave;
    if (block < blocks) split_w_block(p, block, lane);
    return;
  }
  const int M = p.M, K = p.K, R = p.R, m_tiles = (M + 31) / 32;
  const int m0 = (int)blockIdx.x % m_tiles * 32, r0 = (int)blockIdx.x / m_tiles * 32;
  float* t = const_cast<float*>(p.t);
  const rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.x + (size_t)m0 * K), 0, 0x7fffffff, 0x00020000);
  const rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a_cat + (size_t)r0 * K), 0, 0x7fffffff, 0x00020000);
  // a block: 32 rows of x, 32 of A_cat, 128 bytes each, 8 rows to a load; piece c of row r sits at piece c ^ (r & 7)
  char* ring = smem + wave * (SHR_NS * 8192);
  const int c4 = ((lane & 7) ^ (lane >> 3)) * 4;
  uint32_t xo[4], ao[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int r = u * 8 + (lane >> 3);
    xo[u] = ((uint32_t)(m0 + r < M ? r : M - 1 - m0) * (uint32_t)K + (uint32_t)c4) * 4u;
    ao[u] = ((uint32_t)(r0 + r < R ? r : R - 1 - r0) * (uint32_t)K + (uint32_t)c4) * 4u;
  }
  const int nb = (K + 31) / 32, n = (nb - wave + 7) / 8;
  auto fetch = [&](int i) {                                  // this wave's block i (past the last: zeros)
    const int b = wave + 8 * i;
    char* st = ring + (i % SHR_NS) * 8192;
    const uint32_t past = (uint32_t)((K - 1 - b * 32 - c4) >> 31) << 31;     // columns past the end: offsets beyond the buffer, zeros
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lptr_t)(st + u * 1024), 16, xo[u] | past, b * 128, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lptr_t)(st + 4096 + u * 1024), 16, ao[u] | past, b * 128, 0, 0);
    }
  };
  f32x16 acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
#pragma unroll
  for (int i = 0; i < SHR_NS - 1; ++i) fetch(i);
  for (int i = 0; i < n; ++i) {
    fetch(i + SHR_NS - 1);                                   // its place was read in the step before
    vm_wait<8 * (SHR_NS - 1)>();
    const char* st = ring + (i % SHR_NS) * 8192 + l32 * 128;
    f32x4 va[4], vx[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int at = ((2 * g + lh) ^ (l32 & 7)) * 16;
      vx[g] = *reinterpret_cast<const f32x4*>(st + at);
      va[g] = *reinterpret_cast<const f32x4*>(st + 4096 + at);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);                      // lgkmcnt(0): read before the place is filled again
#pragma unroll
    for (int g = 0; g < 4; ++g) acc = mma8(va[g], vx[g], acc);
  }
  vm_wait<0>();
  __syncthreads();
  f32x4(*part)[4][64] = reinterpret_cast<f32x4(*)[4][64]>(smem);
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
    for (int s = 0; s < 7; ++s) o += part[s][g][lane];
    const int col = r0 + 8 * g + 4 * lh;
    if (col < R) *reinterpret_cast<f32x4*>(t + (size_t)(m0 + l32) * R + col) = o * *reinterpret_cast<const f32x4*>(col_scale + col);
  }
#endif
}

// The same without planes: both operands on the fp32 matrix instruction (64 x 64 tiles, four waves of one 32 x 32 tile), for few rows on many columns
// (kh_lora_linear_planes_f32_pays) and for calls whose planes take more than a GiB.  A stage's 32 columns are summed in two chains apart from the
// running sum, which the matrix instruction would cut off at every addition: K 640 / 1280 / 5120 4.5e-7 / 6.4e-7 / 13e-7 -> 1.2e-7 / 1.4e-7 / 2.4e-7
// against 64 bits (planes 1.0e-7 / 1.3e-7 / 2.4e-7), for 12 % of the launch (64 x 10240 x 1280 32.2 -> 36.3 us).
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
    f32x16 c[2];                                 // the stage's own sums
#pragma unroll
    for (int e = 0; e < 16; ++e) c[0][e] = c[1][e] = 0.f;
#pragma unroll
    for (int g = 0; g < FK / 8; ++g)             // W first: a lane then holds one output row and runs of four columns
      c[g % 2] = mma8(*reinterpret_cast<const f32x4*>(sw + 8 * g), *reinterpret_cast<const f32x4*>(sx + 8 * g), c[g % 2]);
    if (t + 1 < KT) store(sm[(t + 1) & 1]);      // that buffer was last read before the barrier above
    acc += c[0] + c[1];
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

}  // namespace

static int f32_args(const float* x, const float* w, const float* bias, const float* a_cat, const float* b_cat, const float* col_scale,
                    const float* t_scratch, const float* residual, const float* y, int64_t M, int64_t N, int64_t K, int64_t R) {
  if (!x || !w || !y || M <= 0 || N <= 0 || K <= 0 || R < 0) return KH_ERR_INVALID_ARG;
  if (R > 0 && (!a_cat || !b_cat || !col_scale || !t_scratch)) return KH_ERR_INVALID_ARG;
  if (K % 4 != 0 || R % 4 != 0) return KH_ERR_UNSUPPORTED;
  if (R > 128 || M > (1 << 24) || N > (1 << 24) || K > (1 << 24)) return KH_ERR_TOO_LARGE;
  if (!kh_aligned16(x) || !kh_aligned16(w) || !kh_aligned16(y) || (bias && !kh_aligned16(bias)) || (residual && !kh_aligned16(residual)) ||
      (R > 0 && (!kh_aligned16(a_cat) || !kh_aligned16(b_cat) || !kh_aligned16(col_scale) || !kh_aligned16(t_scratch))))
    return KH_ERR_ALIGNMENT;
  return KH_OK;
}

static int launch_prepare(const F32Params& p, const float* a_cat, const float* col_scale, int64_t blocks, hipStream_t s) {
  const int64_t shrink = p.R > 0 ? (int64_t)((p.M + 31) / 32) * ((p.R + 31) / 32) : 0, grid = shrink + (blocks + 7) / 8;
  if (grid > 0x7fffffff) return KH_ERR_TOO_LARGE;
  if (grid == 0) return KH_OK;
  if (hipError_t e = kh_allow_lds<lora_prepare_f32_kernel>(SHR_LDS); e != hipSuccess) return (int)e;
  kh_launch(KH_TAG_LORA_SHRINK, lora_prepare_f32_kernel, dim3((unsigned)grid), dim3(512), shrink > 0 ? (size_t)SHR_LDS : 0, s, p, a_cat, col_scale, (int)shrink, (int)blocks);
  KH_RETURN_LAST_ERROR();
}

// See include/katz_hip.h.
KH_EXPORT int kh_lora_linear_split_f32(const float* x, const float* w, const float* bias, const float* a_cat, const float* b_cat,
                                       const float* col_scale, float* t_scratch, const float* residual, float* y, int64_t M, int64_t N,
                                       int64_t K, int64_t R, void* stream) {
  if (const int rc = f32_args(x, w, bias, a_cat, b_cat, col_scale, t_scratch, residual, y, M, N, K, R); rc != KH_OK) return rc;
  const int64_t tiles = ((M + FB - 1) / FB) * ((N + FB - 1) / FB);
  if (tiles > 0x7fffffff) return KH_ERR_TOO_LARGE;
  const F32Params p = {x, w, bias, t_scratch, b_cat, residual, nullptr, y, (int)M, (int)N, (int)K, (int)R};
  if (const int rc = launch_prepare(p, a_cat, col_scale, 0, (hipStream_t)stream); rc != KH_OK) return rc;
  kh_launch(KH_TAG_LORA_GEMM_F32, lora_gemm_f32_mfma_kernel, dim3((unsigned)tiles), dim3(256), 0, (hipStream_t)stream, p);
  KH_RETURN_LAST_ERROR();
}

// See include/katz_hip.h: bytes of the planes, 0 where the form is not taken (rows of a tile are addressed with 32-bit offsets; a GiB of
// scratch at most).
KH_EXPORT int64_t kh_lora_linear_planes_f32_bytes(int64_t N, int64_t K, int64_t R) {
  if (N <= 0 || K <= 0 || R < 0 || N > (1 << 24) || K >= (1 << 22) || R > 128) return 0;
  const int64_t bytes = ((K + FK - 1) / FK + (R + FK - 1) / FK) * ((N + 15) / 16) * 3072;
  return bytes <= ((int64_t)1 << 30) ? bytes : 0;
}

// Planes cost W three times more (read, written, read again as 6 of 4 bytes), the fp32 instruction the matrix pipe.  Estimates of both launches in us,
// within 10 % of what was measured for 1 .. 1024 rows at 640 x 640 .. 12288 x 12288: some 6 us before and behind the loop, a pass over W at
// 5 TB/s, 4 us where x comes in several rows of tiles, and per stage of 32 columns the time of the tile that is taken (rounds of 256 CUs).  Planes
// give the smaller error and stay up to a tenth slower.  M / N / K, planes / fp32 instruction: 64 / 10240 / 1280 62.8 / 49.6; 192 / 5120 / 640 33.0 / 27.6;
// 128 / 8192 / 8192 344 / 266; 256 / 12288 / 12288 1010 / 755; 256 / 10240 / 1280 78 / 87; 64 / 1280 / 5120 136 / 167; 1024 / 640 / 640 26.6 / 26.3.
KH_EXPORT int kh_lora_linear_planes_f32_pays(int64_t M, int64_t N, int64_t K, int64_t R) {
  if (M <= 0 || N <= 0 || K <= 0 || R < 0 || M > (1 << 24) || N > (1 << 24) || K > (1 << 24) || R > 128) return 0;
  auto rounds = [&](int64_t bm, int64_t bn) { return (double)(((M + bm - 1) / bm * ((N + bn - 1) / bn) + 255) / 256); };
  const double stages = (double)((K + FK - 1) / FK + (R + FK - 1) / FK), small = rounds(64, 80), mid = 1.1 * rounds(128, 80), big = 1.65 * rounds(128, 160);
  const double tile = small == 1 ? 0.77 : small == 2 ? 1.16 : 0.25 + 0.5 * small, least = tile < mid ? tile : mid, instr = 0.2 + 0.59 * rounds(FB, FB);
  const double planes = 6 + 2e-6 * (double)N * (double)K + (M > 64 ? 4 : 0) + stages * (least < big ? least : big);
  return planes <= 1.1 * (5.5 + stages * (instr > 0.98 ? instr : 0.98)) ? 1 : 0;
}

KH_EXPORT int kh_lora_linear_planes_f32(const float* x, const float* w, const float* bias, const float* a_cat, const float* b_cat,
                                        const float* col_scale, float* t_scratch, void* planes, const float* residual, float* y, int64_t M,
                                        int64_t N, int64_t K, int64_t R, void* stream) {
  if (const int rc = f32_args(x, w, bias, a_cat, b_cat, col_scale, t_scratch, residual, y, M, N, K, R); rc != KH_OK) return rc;
  if (!planes) return KH_ERR_INVALID_ARG;
  if (!kh_aligned16(planes)) return KH_ERR_ALIGNMENT;
  const int64_t bytes = kh_lora_linear_planes_f32_bytes(N, K, R);
  if (bytes == 0) return KH_ERR_UNSUPPORTED;
  hipStream_t s = (hipStream_t)stream;
  const F32Params p = {x, w, bias, t_scratch, b_cat, residual, planes, y, (int)M, (int)N, (int)K, (int)R};
  if (const int rc = launch_prepare(p, a_cat, col_scale, bytes / 3072, s); rc != KH_OK) return rc;
  // the tile whose rounds of 256 CUs cost least (clocks of a 32-column stage; two workgroups of the small ones share a CU)
  auto cost = [&](int64_t bm, int64_t bn, double clk) { return (double)(((M + bm - 1) / bm * ((N + bn - 1) / bn) + 255) / 256) * clk; };
  const double big = cost(128, 160, 2000), mid = cost(128, 80, 1050), small = cost(64, 80, 600);
  if (big <= mid && big <= small) return launch_split<GCfg<4, 2, 2>>(p, s);
  return mid <= small ? launch_split<GCfg<8, 1, 1>>(p, s) : launch_split<GCfg<4, 1, 1>>(p, s);
}
