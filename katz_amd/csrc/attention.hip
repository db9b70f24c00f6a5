// K3: flash-style attention forward on bf16 MFMA for gfx950, head_dim 64, no mask, no dropout:
//   o = softmax(q k^T * scale) v
// replacing the F.scaled_dot_product_attention call of the reference's attention processor
// (diffusers-hf/src/diffusers/models/attention_processor.py:1269-1283).  q/k/v/o are addressed in
// the projection layout [B, tokens, heads*64] (head h = columns 64h..64h+63) through explicit
// row / batch strides, so the [B,h,T,64] transposes of the reference (:1269-1272, :1280) are never
// materialised.
//
// One workgroup = 4 (or 2) waves = 128 (64) queries of one (batch, head); each wave owns 32 queries.
// Per 64-key tile (K and V in LDS, three stages):
//   S^T = K . Q^T      (A = K fragment from LDS, B = Q fragment held in registers)
//   so every lane holds 32 scores of ONE query (query = lane%32): the row max / row sum are
//   in-lane reductions plus one exchange between the two 32-lane halves.
//   O^T += V^T . P^T   (A = V^T fragment from LDS, transposed by the read (ds_read_tr16_b64), B = P straight from the score registers:
//   the MFMA K index is a free permutation as long as both operands agree on it.)
//
// What bounds it: the vector ALU (exp, scale, maximum, conversion: about 1000 of the 1300 clocks a wave spends on a tile with three waves per SIMD) and,
// on most grids, the last round of workgroups (640 on 256 CUs: three on some, 2.5 on average).  K and V went through registers before, V transposed by
// eight 4-byte LDS writes and 16 vector instructions per thread and tile; by DMA into unpadded swizzled tiles, us per call (batch, tokens, heads):
// 2 x 4096 x 10 129 -> 120, 2 x 3952 x 10 125 -> 114, 2 x 1024 x 20 27.2 -> 24.8, 1 x 3952 x 10 86.7 -> 78.7, 1 x 988 x 20 18.7 -> 17.4, 2 x 256 x 20 6.9 -> 5.9,
// 988 queries on 77 keys 6.7 -> 5.8.  Same bits.  Transposing reads as inline assembly, without the compiler's wait for every DMA in front of them and
// with the DMA a whole step ahead, measured the same; 64 queries per workgroup everywhere 160 us at 2 x 4096 x 10, 25.5 at 2 x 1024 x 20.
#include "kh_common.h"
#include <type_traits>

namespace {

constexpr int HD = 64;        // head dim
constexpr int KV = 64;        // keys per tile
constexpr float NEG_BIG = -1.0e30f;
constexpr float RESCALE_LOG2 = 8.0f;   // the running maximum moves only for jumps above 2^8

struct AttnParams {
  const bf16_t* q; const bf16_t* k; const bf16_t* v; bf16_t* o;
  int B, H, T, S;
  long ldq, ldk, ldv, ldo;   // row strides (elements)
  long bsq, bsk, bsv, bso;   // batch strides (elements)
  float scale_log2e;
  int q_blocks;
};

typedef __attribute__((address_space(3))) void* lptr_t;
typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef __attribute__((address_space(3))) bf16x4* ltr_t;

constexpr int ROWB = HD * 2;                 // bytes of a K or V row in LDS, unpadded
constexpr int TILE = KV * ROWB;              // of a tile of either
constexpr int NST = 3;                       // stages of K and V

template <int VM>
__device__ __forceinline__ void wait_vm() {  // vmcnt = VM, the other counters unconstrained (gfx9 encoding)
  __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | (15 << 8) | ((VM >> 4) << 14));
}

// the larger of lanes l and l + 32, in both, without a trip through LDS
__device__ __forceinline__ float half_max(float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}

template <int NW>   // waves per workgroup: NW*32 queries
// Two waves per SIMD at least: that caps a wave at 256 registers, which makes the compiler keep MFMA results in
// VGPRs (the softmax reads them every tile; from AGPRs every score and every rescaled output costs extra moves).
__global__ __launch_bounds__(NW * 64, 2) void attention_kernel(const AttnParams p) {
#if __HIP_DEVICE_COMPILE__   // the host pass only needs the kernel's symbol (it cannot lower the buffer-resource type)
  constexpr int UPW = 8 / NW;                // 1 KB DMA instructions per wave and tile of K, and of V
  extern __shared__ __attribute__((aligned(16))) char smem[];   // [NST][K tile, V tile] (named arrays: the compiler waits for every DMA in front of a read)

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, lh = lane >> 5;
  const uint32_t total = (uint32_t)p.q_blocks * p.H * p.B;
  const uint32_t logical = xcd_remap(blockIdx.x, total);
  const int qb = logical % p.q_blocks;
  const int bh = logical / p.q_blocks;
  const int h = bh % p.H, b = bh / p.H;

  const bf16_t* qp = p.q + (size_t)b * p.bsq + (size_t)h * HD;
  const bf16_t* kp = p.k + (size_t)b * p.bsk + (size_t)h * HD;
  const bf16_t* vp = p.v + (size_t)b * p.bsv + (size_t)h * HD;
  bf16_t* op = p.o + (size_t)b * p.bso + (size_t)h * HD;

  // Q fragments: query = q0 + l32, d = ks*16 + lh*8 .. +7
  const int qrow = qb * (NW * 32) + wave * 32 + l32;
  const int qrow_c = qrow < p.T ? qrow : p.T - 1;
  bf16x8 qf[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    qf[ks] = *reinterpret_cast<const bf16x8*>(qp + (size_t)qrow_c * p.ldq + ks * 16 + lh * 8);

  f32x16 oacc[2];
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) oacc[dt][v] = 0.f;
  float m_run = NEG_BIG, l_run = 0.f;

  const int n_tiles = (p.S + KV - 1) / KV;

  // K and V tiles go straight to LDS, two tiles ahead: a DMA instruction is 8 keys of 128 bytes, lane l key l / 8, and the 16-byte piece it fetches
  // is swizzled by the key so that the reads below spread over the banks.  Keys past S lie beyond the buffer: zeros.
  auto swz_k = [](int key) { return (key >> 1) & 7; };
  auto swz_v = [](int key) { return (key & 2) << 1; };
  uint32_t koff[UPW], voff[UPW];
#pragma unroll
  for (int i = 0; i < UPW; ++i) {
    const int key = (wave * UPW + i) * 8 + (lane >> 3);
    koff[i] = (uint32_t)key * (uint32_t)p.ldk * 2u + (uint32_t)(((lane & 7) ^ swz_k(key)) * 16);
    voff[i] = (uint32_t)key * (uint32_t)p.ldv * 2u + (uint32_t)(((lane & 7) ^ swz_v(key)) * 16);
  }
  auto load_tile = [&](int t, int st) {      // tile t into the stage at byte st
    const int s0 = t * KV, last = (p.S - s0 < KV ? p.S - s0 : KV) - 1;
    const rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(kp + (size_t)s0 * p.ldk), 0, (int)(uint32_t)((last * p.ldk + HD) * 2), 0x00020000);
    const rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(vp + (size_t)s0 * p.ldv), 0, (int)(uint32_t)((last * p.ldv + HD) * 2), 0x00020000);
#pragma unroll
    for (int i = 0; i < UPW; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (lptr_t)(smem + st + (wave * UPW + i) * 1024), 16, koff[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < UPW; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (lptr_t)(smem + st + TILE + (wave * UPW + i) * 1024), 16, voff[i], 0, 0, 0);
  };
  // K fragment: key l32 of 32, pieces 2 ks + lh.  V^T fragment: ds_read_tr16_b64 gives lane i of 16 the i-th element of four rows of which the lanes
  // 4r .. 4r + 3 address the r-th (32 bytes): four keys of dimension i.
  int ka[4], va[2];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) ka[ks] = l32 * ROWB + ((2 * ks + lh) ^ swz_k(l32)) * 16;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt) {
    const int r = (lane & 15) >> 2, piece = dt * 4 + ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
    va[dt] = TILE + (4 * lh + r) * ROWB + (piece ^ swz_v(r)) * 16 + (lane & 1) * 8;
  }
  load_tile(0, 0);
  if (n_tiles > 1) load_tile(1, 2 * TILE);
  int stg = 0;                               // stage of the current tile

  // One 64-key tile.  MASK: the tile may reach beyond S (only the last one can).
  auto tile_step = [&](int t, auto mask_tag) {
    constexpr bool MASK = decltype(mask_tag)::value;
    if (t + 1 < n_tiles) wait_vm<2 * UPW>(); else wait_vm<0>();      // this wave's share of tile t is there
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();            // everybody's; and nobody reads tile t - 1 any more, whose stage tile t + 2 takes
    asm volatile("" ::: "memory");

    // S^T tiles: st[kt][v] : key = t*64 + kt*32 + 8*(v/4) + 4*lh + v%4, query = l32
    f32x16 st[2];
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(smem + stg + ka[ks] + kt * 32 * ROWB);
        st[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], ks == 0 ? zero : st[kt], 0, 0, 0);
      }
    }
    if constexpr (MASK) {
      const int s0 = t * KV;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int key = s0 + kt * 32 + 8 * (v >> 2) + 4 * lh + (v & 3);
          if (key >= p.S) st[kt][v] = NEG_BIG;
        }
    }
    float mx = NEG_BIG;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int v = 0; v < 16; ++v) mx = fmaxf(mx, st[kt][v]);
    mx = half_max(mx);
    // Lazy running maximum: the reference point of the exponentials only moves when the row maximum has grown by
    // more than 2^RESCALE_LOG2 in the exponent domain; until then p = exp2(s - m) may exceed 1 (by at most that
    // factor, harmless in fp32 / bf16) and numerator and denominator stay consistent.  Moving it rescales
    // the 32 output accumulators, which is then rare -- and skipped for the whole wave when no lane moves.
    const bool move = (mx - m_run) * p.scale_log2e > RESCALE_LOG2;
    if (__builtin_amdgcn_ballot_w64(move) != 0) {
      const float m_new = move ? mx : m_run;
      const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * p.scale_log2e);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) oacc[dt][v] *= alpha;
    }
    const float mb = m_run * p.scale_log2e;
    bf16x8 pf[2][2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int v = 0; v < 16; v += 2) {
        const float e0 = __builtin_amdgcn_exp2f(st[kt][v] * p.scale_log2e - mb);
        const float e1 = __builtin_amdgcn_exp2f(st[kt][v + 1] * p.scale_log2e - mb);
        pf[kt][v >> 3][v & 7] = (bf16_t)e0;
        pf[kt][v >> 3][(v & 7) + 1] = (bf16_t)e1;
      }
    // O^T += V^T . P^T : A fragment row d = dt*32 + l32, element e <-> key kt*32 + 8*(2s + e/4) + 4*lh + e%4.
    // Row sums ride along on the matrix pipe, which has cycles to spare here (the vector ALU does not):
    // ones^T . P^T puts sum_k P[k][q] of all 64 keys (both lane halves) into every row of column q, i.e. into every
    // register of the lanes of query q.  The denominator is then the sum of the same rounded P values the numerator
    // uses.  Its MFMAs sit between those of the two output tiles, so nothing waits on their dependency chain.
    const bf16_t one = (bf16_t)1.0f;
    const bf16x8 ones = {one, one, one, one, one, one, one, one};
    f32x16 rsum = zero;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int dt = 0; dt < 2; ++dt) {
          // (the swizzle repeats every four keys)
          const char* base = smem + stg + va[dt] + (kt * 32 + 16 * s) * ROWB;
          const bf16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((ltr_t)(base));
          const bf16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((ltr_t)(base + 8 * ROWB));
          bf16x8 vf;
#pragma unroll
          for (int e = 0; e < 4; ++e) { vf[e] = v0[e]; vf[4 + e] = v1[e]; }
          oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[kt][s], oacc[dt], 0, 0, 0);
        }
        rsum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, pf[kt][s], rsum, 0, 0, 0);
      }
    l_run += rsum[0];

    // (behind the reads of V: the compiler waits for every DMA that is out in front of a transposing read)
    if (t + 2 < n_tiles) load_tile(t + 2, stg >= 2 * TILE ? stg - 2 * TILE : stg + 4 * TILE);
    stg = stg == 2 * (NST - 1) * TILE ? 0 : stg + 2 * TILE;
  };
  const int full_tiles = p.S / KV;
  for (int t = 0; t < full_tiles; ++t) tile_step(t, std::false_type{});
  if (full_tiles < n_tiles) tile_step(full_tiles, std::true_type{});

  const float inv = 1.0f / l_run;   // the MFMA row sums already cover the keys of both lane halves
  // A lane holds runs of 4 dims (8 bytes); lanes l and l + 32 hold the two halves of every 16-byte piece of their query's
  // row.  Two pieces at a time, the pair trades halves (v_permlane32_swap: the upper half of the first register against the
  // lower half of the second), after which lane l owns the even piece and lane l + 32 the odd one: 16-byte stores.
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int gp = 0; gp < 2; ++gp) {
      const int ge = 2 * gp, go = 2 * gp + 1;
      const uint32_t e0 = pack_bf16x2(oacc[dt][4 * ge + 0] * inv, oacc[dt][4 * ge + 1] * inv);
      const uint32_t e1 = pack_bf16x2(oacc[dt][4 * ge + 2] * inv, oacc[dt][4 * ge + 3] * inv);
      const uint32_t o0 = pack_bf16x2(oacc[dt][4 * go + 0] * inv, oacc[dt][4 * go + 1] * inv);
      const uint32_t o1 = pack_bf16x2(oacc[dt][4 * go + 2] * inv, oacc[dt][4 * go + 3] * inv);
      const auto s0 = __builtin_amdgcn_permlane32_swap(e0, o0, false, false);
      const auto s1 = __builtin_amdgcn_permlane32_swap(e1, o1, false, false);
      const u32x4 piece = {s0[0], s1[0], s0[1], s1[1]};
      if (qrow < p.T) {
        const size_t off = (size_t)qrow * p.ldo + dt * 32 + 8 * (2 * gp + lh);
        *reinterpret_cast<u32x4*>(op + off) = piece;   // (plain: written through the L2, 32 bytes of a row at a time gained nothing)
      }
    }
#endif
}

}  // namespace

KH_EXPORT int kh_attention_bf16(const void* q, const void* k, const void* v, void* o, int64_t B, int64_t H, int64_t T,
                                int64_t S, int64_t head_dim, int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo,
                                int64_t bsq, int64_t bsk, int64_t bsv, int64_t bso, float scale, void* stream) {
  if (!q || !k || !v || !o || B <= 0 || H <= 0 || T <= 0 || S <= 0) return KH_ERR_INVALID_ARG;
  if (head_dim != HD) return KH_ERR_UNSUPPORTED;
  if ((ldq | ldk | ldv | ldo | bsq | bsk | bsv | bso) % 8 != 0) return KH_ERR_ALIGNMENT;
  if (ldq < H * HD || ldk < H * HD || ldv < H * HD || ldo < H * HD) return KH_ERR_INVALID_ARG;
  if (!kh_aligned16(q) || !kh_aligned16(k) || !kh_aligned16(v) || !kh_aligned16(o)) return KH_ERR_ALIGNMENT;
  AttnParams p;
  p.q = (const bf16_t*)q; p.k = (const bf16_t*)k; p.v = (const bf16_t*)v; p.o = (bf16_t*)o;
  p.B = (int)B; p.H = (int)H; p.T = (int)T; p.S = (int)S;
  p.ldq = ldq; p.ldk = ldk; p.ldv = ldv; p.ldo = ldo;
  p.bsq = bsq; p.bsk = bsk; p.bsv = bsv; p.bso = bso;
  p.scale_log2e = scale * 1.4426950408889634f;
  // 128 queries per workgroup; 64 for short key sequences on small grids (cross-attention), for a finer spread
  const bool small = ((T + 127) / 128) * H * B < 512 && S <= 256;
  const int qpw = small ? 64 : 128;
  p.q_blocks = (int)((T + qpw - 1) / qpw);
  const long grid = (long)p.q_blocks * H * B;
  if (grid > 0x7fffffffL) return KH_ERR_TOO_LARGE;
  if (small)
    kh_launch(KH_TAG_ATTENTION, attention_kernel<2>, dim3((unsigned)grid), dim3(128), 2 * NST * TILE, (hipStream_t)stream, p);
  else
    kh_launch(KH_TAG_ATTENTION, attention_kernel<4>, dim3((unsigned)grid), dim3(256), 2 * NST * TILE, (hipStream_t)stream, p);
  KH_RETURN_LAST_ERROR();
}
