// K3: flash-style attention forward on bf16 MFMA for gfx950, head_dim 64, no mask, no dropout:
//   o = softmax(q k^T * scale) v
// replacing the F.scaled_dot_product_attention call of the reference's attention processor
// (diffusers-hf/src/diffusers/models/attention_processor.py:1269-1283).  q/k/v/o are addressed in
// the projection layout [B, tokens, heads*64] (head h = columns 64h..64h+63) through explicit
// row / batch strides, so the [B,h,T,64] transposes of the reference (:1269-1272, :1280) are never
// materialised.
//
// One workgroup = 4 waves = 128 queries of one (batch, head), 32 each, or 64, 16 each (Wave below: the same bits).
// Per 64-key tile (K and V in LDS, three stages):
//   S^T = K . Q^T      (A = K fragment from LDS, B = Q fragment held in registers)
//   so every lane holds 32 scores of ONE query (query = lane%32): the row max / row sum are
//   in-lane reductions plus one exchange between the two 32-lane halves.
//   O^T += V^T . P^T   (A = V^T fragment from LDS, transposed by the read (ds_read_tr16_b64), B = P straight from the score registers:
//   the MFMA K index is a free permutation as long as both operands agree on it.)
//
// What bounds it: the vector ALU (exp, scale, maximum, conversion: about 1000 of the 1200 clocks a wave of 32 queries spends on a tile with three waves per
// SIMD) and, before the last round's workgroups were halved, that round (620 of 128 queries on 256 CUs: three on some, 2.4 on average).  A wave of 16
// reads as many bytes of K and V from LDS as one of 32, so only those workgroups are halved that would leave CUs idle.  us per launch in a graph, all of 128
// queries (64 on two waves for short keys on small grids) -> now, one run (batch, tokens, heads): 2 x 4096 x 10 113.3 -> 100.5, 2 x 3952 x 10 109.7 -> 95.8, 2 x 1024 x 20 23.5 -> 20.6,
// 1 x 3952 x 10 73.6 -> 60.3, 1 x 988 x 20 16.8 -> 15.7, 2 x 256 x 20 5.7 -> 4.9, 988 queries on 77 keys 5.5 -> 4.8, 2 x 3952 x 10 on 77 9.4 -> 8.7.
// K and V by DMA into unpadded swizzled tiles, V transposed by the read, took 114 us where registers and eight 4-byte
// LDS writes a thread took 125 (2 x 3952 x 10).  Transposing reads as inline assembly, without the compiler's wait for every DMA in front of
// them and with the DMA a whole step ahead, measured the same; 64 queries per workgroup everywhere 113 us at 2 x 3952 x 10.
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
  int n32;                   // workgroups of 128 queries (a multiple of 8, or all of them)
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

// ... of the four lanes that hold scores of query l % 16
__device__ __forceinline__ float quarter_max(float v) {
  const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return half_max(fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1])));
}

// Shapes of a wave with QW queries.  Either way a lane holds scores of one query, score i of 2 QW (i = register tile * registers + register), eight in a
// row are a k-step's P fragment, and every sum runs over the keys in the same order: v_mfma 16x16x32 gives the bits of two chained steps of 32x32x16 if
// keys and dimensions sit at the same places of those steps.  For QW 16 the rows of K that a tile multiplies are chosen accordingly.
template <int QW>
struct Wave {
  using Acc = typename std::conditional<QW == 32, f32x16, f32x4>::type;
  static constexpr int NA = QW == 32 ? 16 : 4;           // registers of a tile
  static constexpr int NK = KV / QW, ND = HD / QW;       // tiles of scores, of the output
  static constexpr int KS = QW == 32 ? 4 : 2;            // k-steps over the dimensions and over the keys of a tile of 64
  static __device__ __forceinline__ Acc mfma(const bf16x8& a, const bf16x8& b, const Acc& c) {
#if __HIP_DEVICE_COMPILE__
    if constexpr (QW == 32) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
#else
    return c;
#endif
  }
};

// Queries q0 .. q0 + 4 QW of a head, four waves.
template <int QW>
__device__ __forceinline__ void attention_unit(const AttnParams& p, const int q0, const int bh, char* smem) {
#if __HIP_DEVICE_COMPILE__   // the host pass only needs the kernel's symbol (it cannot lower the buffer-resource type)
  typedef Wave<QW> W;
  typedef typename W::Acc Acc;
  constexpr int UPW = 2;                     // 1 KB DMA instructions per wave and tile of K, and of V

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane % QW, lg = lane / QW;  // query of the wave, part of its scores
  const int h = bh % p.H, b = bh / p.H;

  const bf16_t* qp = p.q + (size_t)b * p.bsq + (size_t)h * HD;
  const bf16_t* kp = p.k + (size_t)b * p.bsk + (size_t)h * HD;
  const bf16_t* vp = p.v + (size_t)b * p.bsv + (size_t)h * HD;
  bf16_t* op = p.o + (size_t)b * p.bso + (size_t)h * HD;

  // Q fragments: query q0 + lq, d = ks * (HD / KS) + lg*8 .. +7
  const int qrow = q0 + wave * QW + lq;
  const int qrow_c = qrow < p.T ? qrow : p.T - 1;
  bf16x8 qf[W::KS];
#pragma unroll
  for (int ks = 0; ks < W::KS; ++ks)
    qf[ks] = *reinterpret_cast<const bf16x8*>(qp + (size_t)qrow_c * p.ldq + ks * (HD / W::KS) + lg * 8);

  Acc zero;
#pragma unroll
  for (int v = 0; v < W::NA; ++v) zero[v] = 0.f;
  Acc oacc[W::ND];
#pragma unroll
  for (int dt = 0; dt < W::ND; ++dt) oacc[dt] = zero;
  float m_run = NEG_BIG, l_run = 0.f;

  const int n_tiles = (p.S + KV - 1) / KV;

  // K and V tiles go straight to LDS, two tiles ahead: a DMA instruction is 8 keys of 128 bytes, lane l key l / 8, and the 16-byte piece it fetches
  // is swizzled by the key so that the reads below spread over the banks.  Keys past S lie beyond the buffer: zeros.
  auto swz_k = [](int key) { return QW == 32 ? (key >> 1) & 7 : ((key & 7) >> 1) | ((key >> 2) & 4); };
  auto swz_v = [](int key) { return QW == 32 ? (key & 2) << 1 : (key & 2) << 1 | (key & 4) >> 1; };
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
  // K fragments, pieces (8 / KS) ks + lg: QW 32 key lq of the tile's 32; QW 16 key 16 (lq / 8) + 8 a + lq % 8 of 32 keys for their tiles a = 0, 1.
  // V^T fragments: ds_read_tr16_b64 gives lane i of 16 the i-th element of four rows of which the lanes 4r .. 4r + 3 address the r-th (32 bytes): four
  // keys of dimension i.
  int ka[4], va[W::ND];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int key = QW == 32 ? lq : 16 * (lq >> 3) + 8 * (i >> 1) + (lq & 7), piece = QW == 32 ? 2 * i + lg : 4 * (i & 1) + lg;
    ka[i] = key * ROWB + (piece ^ swz_k(key)) * 16;
  }
#pragma unroll
  for (int dt = 0; dt < W::ND; ++dt) {
    const int r = (lane & 15) >> 2, half = (lane & 3) >> 1;
    const int key = QW == 32 ? 4 * lg + r : 16 * (lg >> 1) + 4 * (lg & 1) + r, piece = QW == 32 ? dt * 4 + ((lane >> 4) & 1) * 2 + half : dt * 2 + half;
    va[dt] = TILE + key * ROWB + (piece ^ swz_v(QW == 32 ? r : key)) * 16 + (lane & 1) * 8;
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

    // S^T tiles: st[kt][v], query lq, key t*64 + kt*32 + 8*(v/4) + 4*lg + v%4 (QW 32) or t*64 + (kt/2)*32 + 16*(lg/2) + 8*(kt%2) + 4*(lg%2) + v
    Acc st[W::NK];
#pragma unroll
    for (int kt = 0; kt < W::NK; ++kt) {
#pragma unroll
      for (int ks = 0; ks < W::KS; ++ks) {
        const int at = QW == 32 ? ka[ks] + kt * 32 * ROWB : ka[(kt & 1) * 2 + ks] + (kt >> 1) * 32 * ROWB;
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(smem + stg + at);
        st[kt] = W::mfma(kf, qf[ks], ks == 0 ? zero : st[kt]);
      }
    }
    if constexpr (MASK) {
      const int s0 = t * KV;
#pragma unroll
      for (int kt = 0; kt < W::NK; ++kt)
#pragma unroll
        for (int v = 0; v < W::NA; ++v) {
          const int key = s0 + (QW == 32 ? kt * 32 + 8 * (v >> 2) + 4 * lg + (v & 3) : (kt >> 1) * 32 + 16 * (lg >> 1) + 8 * (kt & 1) + 4 * (lg & 1) + v);
          if (key >= p.S) st[kt][v] = NEG_BIG;
        }
    }
    float mx = NEG_BIG;
#pragma unroll
    for (int kt = 0; kt < W::NK; ++kt)
#pragma unroll
      for (int v = 0; v < W::NA; ++v) mx = fmaxf(mx, st[kt][v]);
    mx = QW == 32 ? half_max(mx) : quarter_max(mx);
    // Lazy running maximum: the reference point of the exponentials only moves when the row maximum has grown by
    // more than 2^RESCALE_LOG2 in the exponent domain; until then p = exp2(s - m) may exceed 1 (by at most that
    // factor, harmless in fp32 / bf16) and numerator and denominator stay consistent.  Moving it rescales
    // the output accumulators, which is then rare -- and skipped for the whole wave when no lane moves.
    const bool move = (mx - m_run) * p.scale_log2e > RESCALE_LOG2;
    if (__builtin_amdgcn_ballot_w64(move) != 0) {
      const float m_new = move ? mx : m_run;
      const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * p.scale_log2e);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < W::ND; ++dt)
#pragma unroll
        for (int v = 0; v < W::NA; ++v) oacc[dt][v] *= alpha;
    }
    const float mb = m_run * p.scale_log2e;
    bf16x8 pf[W::KS];
#pragma unroll
    for (int i = 0; i < W::NK * W::NA; i += 2) {
      const float e0 = __builtin_amdgcn_exp2f(st[i / W::NA][i % W::NA] * p.scale_log2e - mb);
      const float e1 = __builtin_amdgcn_exp2f(st[i / W::NA][i % W::NA + 1] * p.scale_log2e - mb);
      pf[i >> 3][i & 7] = (bf16_t)e0;
      pf[i >> 3][(i & 7) + 1] = (bf16_t)e1;
    }
    // O^T += V^T . P^T : A fragment row d = dt*QW + lane % QW, its keys those of the P fragment's elements.
    // Row sums ride along on the matrix pipe, which has cycles to spare here (the vector ALU does not):
    // ones^T . P^T puts sum_k P[k][q] of all 64 keys (all lane parts) into every row of column q, i.e. into every
    // register of the lanes of query q.  The denominator is then the sum of the same rounded P values the numerator
    // uses.  Its MFMAs sit between those of the output tiles, so nothing waits on their dependency chain.
    const bf16_t one = (bf16_t)1.0f;
    const bf16x8 ones = {one, one, one, one, one, one, one, one};
    Acc rsum = zero;
#pragma unroll
    for (int s = 0; s < W::KS; ++s) {
#pragma unroll
      for (int dt = 0; dt < W::ND; ++dt) {
        // (the swizzles repeat every eight keys)
        const char* base = smem + stg + va[dt] + s * (KV / W::KS) * ROWB;
        const bf16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((ltr_t)(base));
        const bf16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((ltr_t)(base + 8 * ROWB));
        bf16x8 vf;
#pragma unroll
        for (int e = 0; e < 4; ++e) { vf[e] = v0[e]; vf[4 + e] = v1[e]; }
        oacc[dt] = W::mfma(vf, pf[s], oacc[dt]);
      }
      rsum = W::mfma(ones, pf[s], rsum);
    }
    l_run += rsum[0];

    // (behind the reads of V: the compiler waits for every DMA that is out in front of a transposing read)
    if (t + 2 < n_tiles) load_tile(t + 2, stg >= 2 * TILE ? stg - 2 * TILE : stg + 4 * TILE);
    stg = stg == 2 * (NST - 1) * TILE ? 0 : stg + 2 * TILE;
  };
  const int full_tiles = p.S / KV;
  for (int t = 0; t < full_tiles; ++t) tile_step(t, std::false_type{});
  if (full_tiles < n_tiles) tile_step(full_tiles, std::true_type{});

  const float inv = 1.0f / l_run;   // the MFMA row sums already cover the keys of all lane parts
  // A lane holds runs of 4 dims (8 bytes); the halves of every 16-byte piece of a query's row lie in two lanes, 32 (QW 32) or 16 apart.  Two pieces at a
  // time, the pair trades halves (v_permlane32_swap, v_permlane16_swap: the upper lanes of the first register against the lower lanes of the second), after
  // which one lane owns the first piece and the other one the second: 16-byte stores.
#pragma unroll
  for (int i = 0; i < (QW == 32 ? 4 : 2); ++i) {
    const int te = QW == 32 ? i >> 1 : 2 * i, to = QW == 32 ? te : te + 1, ge = QW == 32 ? 8 * (i & 1) : 0, go = QW == 32 ? ge + 4 : 0;   // tiles, first registers
    const uint32_t e0 = pack_bf16x2(oacc[te][ge + 0] * inv, oacc[te][ge + 1] * inv);
    const uint32_t e1 = pack_bf16x2(oacc[te][ge + 2] * inv, oacc[te][ge + 3] * inv);
    const uint32_t o0 = pack_bf16x2(oacc[to][go + 0] * inv, oacc[to][go + 1] * inv);
    const uint32_t o1 = pack_bf16x2(oacc[to][go + 2] * inv, oacc[to][go + 3] * inv);
    u32x4 piece;
    if constexpr (QW == 32) {
      const auto s0 = __builtin_amdgcn_permlane32_swap(e0, o0, false, false);
      const auto s1 = __builtin_amdgcn_permlane32_swap(e1, o1, false, false);
      piece = u32x4{s0[0], s1[0], s0[1], s1[1]};
    } else {
      const auto s0 = __builtin_amdgcn_permlane16_swap(e0, o0, false, false);
      const auto s1 = __builtin_amdgcn_permlane16_swap(e1, o1, false, false);
      piece = u32x4{s0[0], s1[0], s0[1], s1[1]};
    }
    if (qrow < p.T) {
      const int d = QW == 32 ? te * 32 + 8 * (2 * (i & 1) + lg) : (te + (lg & 1)) * 16 + 8 * (lg >> 1);
      *reinterpret_cast<u32x4*>(op + (size_t)qrow * p.ldo + d) = piece;   // (plain: written through the L2, 32 bytes of a row at a time gained nothing)
    }
  }
#endif
}

// The first n32 workgroups take 128 queries with four waves of 32, the others 64 with four of 16.
// Two waves per SIMD at least: that caps a wave at 256 registers, which makes the compiler keep MFMA results in
// VGPRs (the softmax reads them every tile; from AGPRs every score and every rescaled output costs extra moves).
__global__ __launch_bounds__(256, 2) void attention_kernel(const AttnParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];   // [NST][K tile, V tile] (named arrays: the compiler waits for every DMA in front of a read)
  const uint32_t n32 = (uint32_t)p.n32;
  if (blockIdx.x < n32) {
    const uint32_t u = xcd_remap(blockIdx.x, n32);
    attention_unit<32>(p, (int)(u % p.q_blocks) * 128, (int)(u / p.q_blocks), smem);
  } else {                                                       // (n32 is a multiple of 8, so the XCDs go on round-robin)
    const uint32_t v = xcd_remap(blockIdx.x - n32, gridDim.x - n32), u = n32 + v / 2;
    const int q0 = (int)(u % p.q_blocks) * 128 + (int)(v & 1) * 64;
    if (q0 < p.T) attention_unit<16>(p, q0, (int)(u / p.q_blocks), smem);
  }
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
  // 128 queries per workgroup, and 64 for those of the last round of the 256 CUs where that round is at most half full, so that no CU gets a whole
  // workgroup more than others get (the halves then find a CU each; in a fuller round they only cost more: 400 of 128 queries, 2560 x 10 x 2, 49.8 us whole,
  // 50.2 split; 720, 2304 x 10 x 4, 67.5 and 73.8); everything is 64 where there is no whole round (a CU with two waves per SIMD instead of one: 240
  // workgroups, 1444 x 20, 23.3 -> 22.5 us).
  const long units = (T + 127) / 128 * H * B, rest = units % 256;
  p.q_blocks = (int)((T + 127) / 128);
  const long n32 = units < 256 ? 0 : rest <= 128 ? units - rest : units, grid = n32 + 2 * (units - n32);
  if (grid > 0x7fffffffL) return KH_ERR_TOO_LARGE;
  p.n32 = (int)n32;
  kh_launch(KH_TAG_ATTENTION, attention_kernel, dim3((unsigned)grid), dim3(256), 2 * NST * TILE, (hipStream_t)stream, p);
  KH_RETURN_LAST_ERROR();
}
