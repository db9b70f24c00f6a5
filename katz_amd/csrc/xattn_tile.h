// Cross-attention of a staged query tile in the epilogue of lora_gemm_fine.hip (LoraGemmParams::xa_k): the tile is BM queries of BN / 64 heads, a
// wave takes 32 queries of one head against the at most 96 keys of its sample.  The arithmetic, and so the bits, are those of XAttnTile
// (lora_gemm_pipe.hip): one pass over all keys, one query per lane, the row sums as one more MFMA.
//
// Keys and values wait in the registers of the waves that move operands (requested before the ring, 24 registers a head, in waves that use
// few others) and go to LDS when the ring is dead; V is transposed by the read (ds_read_tr16_b64, as in attention.hip).
#pragma once
#include "kh_common.h"
#include "lora_gemm.h"

namespace {

template <int HEADS, int NT, int LDQ>   // heads of a tile; threads that load; elements of a staged query row
struct XAttnFine {
  static constexpr int XS = 96, ROWB = 128, ROUNDS = HEADS * XS * 8 / NT;
  static constexpr int K_BYTES = HEADS * XS * ROWB, LDS_BYTES = 2 * K_BYTES;
  static_assert(ROUNDS * NT == HEADS * XS * 8, "whole rounds of 16-byte pieces");
  u32x4 rk[ROUNDS], rv[ROUNDS];

  static __device__ __forceinline__ int swz_k(int key) { return (key >> 1) & 7; }
  static __device__ __forceinline__ int swz_v(int key) { return (key & 2) << 1; }

  // keys beyond S: zeros (their scores are masked, their weights zero)
  __device__ __forceinline__ void load(const LoraGemmParams& p, int m0, int n0, int tid) {
    const int b = m0 / p.xa_T;
    const bf16_t* const kp = p.xa_k + (size_t)b * p.xa_bsk + n0;
    const bf16_t* const vp = p.xa_v + (size_t)b * p.xa_bsv + n0;
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
      const int c = tid + i * NT, hh = c / (XS * 8), key = c % (XS * 8) >> 3, pc = c & 7;
      const bool in = key < p.xa_S;
      rk[i] = in ? *reinterpret_cast<const u32x4*>(kp + (size_t)key * p.xa_ldk + hh * 64 + pc * 8) : u32x4{0u, 0u, 0u, 0u};
      rv[i] = in ? *reinterpret_cast<const u32x4*>(vp + (size_t)key * p.xa_ldv + hh * 64 + pc * 8) : u32x4{0u, 0u, 0u, 0u};
    }
  }

  __device__ __forceinline__ void store(char* kv, int tid) const {
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
      const int c = tid + i * NT, row = c >> 3, key = row % XS, pc = c & 7;   // (head hh's rows follow those of hh - 1)
      *reinterpret_cast<u32x4*>(kv + row * ROWB + (pc ^ swz_k(key)) * 16) = rk[i];
      *reinterpret_cast<u32x4*>(kv + K_BYTES + row * ROWB + (pc ^ swz_v(key)) * 16) = rv[i];
    }
  }

  // queries 32 qg .. of head hh of the tile, by one wave; sQ: the staged tile, kv: what store left
  static __device__ __forceinline__ void unit(const LoraGemmParams& p, const bf16_t* sQ, const char* kv, int hh, int qg, int m0, int n0, int lane) {
#if __HIP_DEVICE_COMPILE__
    typedef __attribute__((address_space(3))) bf16x4* ltr_t;
    const int l32 = lane & 31, lh = lane >> 5, S = p.xa_S;
    bf16x8 qf[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) qf[ks] = *reinterpret_cast<const bf16x8*>(sQ + (qg * 32 + l32) * LDQ + hh * 64 + ks * 16 + lh * 8);
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // S^T tiles: st[kt][v]: key = kt*32 + 8*(v/4) + 4*lh + v%4, query = l32
    const char* const sK = kv + hh * XS * ROWB;
    f32x16 st[3];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int kt = 0; kt < 3; ++kt) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(sK + (kt * 32 + l32) * ROWB + ((2 * ks + lh) ^ swz_k(l32)) * 16);
        st[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], ks == 0 ? zero : st[kt], 0, 0, 0);
      }
    float mx = -1.0e30f;
#pragma unroll
    for (int kt = 0; kt < 3; ++kt)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int key = kt * 32 + 8 * (v >> 2) + 4 * lh + (v & 3);
        if (key >= S) st[kt][v] = -1.0e30f;
        mx = fmaxf(mx, st[kt][v]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mb = mx * p.xa_scale_log2e;
    bf16x8 pf[3][2];
#pragma unroll
    for (int kt = 0; kt < 3; ++kt)
#pragma unroll
      for (int v = 0; v < 16; v += 2) {
        pf[kt][v >> 3][v & 7] = (bf16_t)__builtin_amdgcn_exp2f(st[kt][v] * p.xa_scale_log2e - mb);
        pf[kt][v >> 3][(v & 7) + 1] = (bf16_t)__builtin_amdgcn_exp2f(st[kt][v + 1] * p.xa_scale_log2e - mb);
      }
    // O^T += V^T . P^T: A fragment row d = dt*32 + l32, element e <-> key kt*32 + 8*(2s + e/4) + 4*lh + e%4 (see attention.hip)
    const bf16_t one = (bf16_t)1.0f;
    const bf16x8 ones = {one, one, one, one, one, one, one, one};
    const char* const sV = kv + K_BYTES + hh * XS * ROWB;
    int va[2];
#pragma unroll
    for (int dt = 0; dt < 2; ++dt) {
      const int r = (lane & 15) >> 2, piece = dt * 4 + ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
      va[dt] = (4 * lh + r) * ROWB + (piece ^ swz_v(r)) * 16 + (lane & 1) * 8;
    }
    f32x16 oacc[2] = {zero, zero}, rsum = zero;
#pragma unroll
    for (int kt = 0; kt < 3; ++kt)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int dt = 0; dt < 2; ++dt) {
          const char* const base = sV + va[dt] + (kt * 32 + 16 * s) * ROWB;
          const bf16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((ltr_t)(base));
          const bf16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((ltr_t)(base + 8 * ROWB));
          bf16x8 vf;
#pragma unroll
          for (int e = 0; e < 4; ++e) { vf[e] = v0[e]; vf[4 + e] = v1[e]; }
          oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[kt][s], oacc[dt], 0, 0, 0);
        }
        rsum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, pf[kt][s], rsum, 0, 0, 0);
      }
    // lanes l and l + 32 trade halves, so that each stores whole 16-byte pieces (see attention.hip)
    const float inv = 1.0f / rsum[0];
    bf16_t* const op = p.xa_o + (size_t)(m0 + qg * 32 + l32) * p.xa_ldo + n0 + hh * 64;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int gp = 0; gp < 2; ++gp) {
        const int ge = 8 * gp, go = 8 * gp + 4;
        const uint32_t e0 = pack_bf16x2(oacc[dt][ge] * inv, oacc[dt][ge + 1] * inv), e1 = pack_bf16x2(oacc[dt][ge + 2] * inv, oacc[dt][ge + 3] * inv);
        const uint32_t o0 = pack_bf16x2(oacc[dt][go] * inv, oacc[dt][go + 1] * inv), o1 = pack_bf16x2(oacc[dt][go + 2] * inv, oacc[dt][go + 3] * inv);
        const auto s0 = __builtin_amdgcn_permlane32_swap(e0, o0, false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(e1, o1, false, false);
        *reinterpret_cast<u32x4*>(op + dt * 32 + 8 * (2 * gp + lh)) = u32x4{s0[0], s1[0], s0[1], s1[1]};
      }
#endif
  }
};

}  // namespace
