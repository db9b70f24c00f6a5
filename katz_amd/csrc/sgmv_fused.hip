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
//            B from L2, requested three tiles ahead), times the adapter's scale, rounded and added to the y pieces, which were
//            requested five tiles ahead (128 rows: one), in the registers that held the products: no staging, one barrier a tile.
// What bounds it at a request's sizes is not HBM's rate but the chain of latencies -- segment table, 20 stages, 5 .. 10 tiles -- in workgroups
// that are one to a CU.  Hence as many stages under way as 128 KB hold (eight of 16 KB; five of 24 with all 128 rank rows), a stage's fragments
// read while the stage before is multiplied, the y pieces of the first five tiles (128 rows: of the first) requested while phase 1 runs, the
// results written through the L2 (behind plain stores the launch ended with all of y still to be written: 1 us of 20), and 64-row blocks while
// they fit one round of the 256 CUs, so that fewer of them repeat phase 1 for other columns.
// 8 requests of 256 .. 1024 rows at 1280 -> 1280, ranks 8 .. 128: 20.1 -> 17.6 us, all of rank 32 19.5 -> 15.1; 2 x 1024 rows 13.5 -> 12.9 (launches in a graph).
// Rows / columns of A_a / B_a beyond the adapter's rank are zero by contract, so the padded rank only saves work.
// Batches with few row blocks deal the column tiles of y to several workgroups, each of which repeats phase 1 for its rows: x is then read from
// L2 more than once, which such small batches do not notice.  How many is decided by the segments' true lengths, which only the device knows
// (up to 64 segments): with the host's bound -- every segment as long as the longest -- five segments of 650 rows were 275 workgroups, a
// second round for 19 of them (27.2 -> 11.5 us), and 16 of 1280 .. 2852 rows at 640 a second round of nine (40.1 -> 33.0).
// Grouped form (kh_sgmv_fused_grouped_bf16): several layers that read the same x with the same segments (the to_k / to_v
// projections of every cross-attention read the one text context) in one launch,
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
  int n_segments;    // dealt form: at most 64 segments, workgroups dealt by their table; 0: blockIdx = (row block, segment, layer and column range)
  int n_layers, row_blocks;
  int tiles_per_z;   // 128-column tiles of y per workgroup: blockIdx.z selects the range (T is recomputed per range)
  int z_per_layer;   // column ranges per layer (grid.z = layers x z_per_layer)
  const uint64_t* table;   // grouped form: rows {a_all, b_all, y} of device pointers, one per layer; null: the fields above
};

constexpr int CUS = 256;
#if defined(KH_PLAIN_STORES)
constexpr int STORE_POLICY = 0;
#else
constexpr int STORE_POLICY = 16;                  // sc1: through the L2
#endif
constexpr int B_TILE = 2 * 128 * 128;             // 128 y columns x 128 rank columns, as two 64-column stages
constexpr int RING = 128 * 1024;                  // phase 1: stages of x, then those of A; phase 2: T, and all but the first of the buffers of B tiles
constexpr int D = 3;                              // B tiles requested ahead: D + 1 buffers, buffer k at RING - k B_TILE
constexpr int LDS_BYTES = RING + B_TILE;
static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");

template <int BM>
__global__ __launch_bounds__(512, 2) void sgmv_fused_kernel(const FusedParams p) {
#if __HIP_DEVICE_COMPILE__   // the host pass only needs the kernel's symbol (it cannot lower the buffer-resource type)
  constexpr int TI = BM / 32, T_BYTES = 2 * BM * 128;   // a wave's 16-row tiles; T as two 64-column stages of 128-byte rows
  constexpr int XU = BM / 64;                     // units of 8 rows of x per wave and stage
  // tiles whose y pieces are under way or here.  128 rows: those of the second tile would only be in the way of phase 1's short ring (8 x 4096 rows
  // at 640 33.1 -> 32.3 us without them, rank 64 29.9 -> 29.3, at 1280 55.9 -> 53.9)
  constexpr int YD = BM == 64 ? 5 : 1;
  static_assert(T_BYTES + D * B_TILE <= RING, "T and the B buffers lie in the ring");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int all_tiles = p.N / 128;

  // ---- which rows of which segment, which column tiles ----
  int m0, layer, r0, M, ad, rank, j0, n_tiles;
  float scale;
  if (p.n_segments > 0) {
    // A lane per segment: its row blocks, then their running sum.  Whole rounds of CUS blocks take all columns; what is left over is dealt by
    // column ranges to as many workgroups as there are CUs -- by the blocks that the segments really have, which the host does not know --, the
    // ranges of a block eight workgroups apart, on one XCD.
    int st = 0, end = 0, a = -1;
    if (lane < p.n_segments) { st = p.seg_start[lane]; end = p.seg_start[lane + 1]; a = p.seg_adapter[lane]; }
    const int rows = a >= 0 && end > st ? end - st : 0;
    int rk = 0;
    float sc = 0.f;
    if (rows > 0) { rk = p.adapter_rank[a]; sc = p.adapter_scale[a]; }
    int blocks = (rows + BM - 1) / BM;
    blocks = blocks < p.row_blocks ? blocks : p.row_blocks;
    // (blocks of adapters of more than 64 in the upper half of the word, where 64 segments' blocks fit half a word)
    const bool halves = p.row_blocks < 1024;
    uint32_t sum = (uint32_t)blocks | (halves && rk > 64 ? (uint32_t)blocks << 16 : 0u);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) { const uint32_t v = __shfl_up(sum, o, 64); if (lane >= o) sum += v; }
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)sum, 63);
    const int heavy = halves ? (int)(total >> 16) : 0, per_layer = (int)(halves ? total & 0xffff : total);
    const int nb = per_layer * p.n_layers;
    int upto = (int)(halves ? sum & 0xffff : sum);       // blocks up to this lane's segment
    wait_cnt<0, 0>();                             // (or the compiler waits for them, and all behind them, among phase 1's loads)
    const int u = (int)blockIdx.x, full = nb / CUS * CUS;
    int b = u, last = nb;
    j0 = 0; n_tiles = all_tiles;
    if (u >= full) {
      const int left = nb - full, left8 = (left + 7) & ~7;
      if (left == 0) return;
      int z = CUS / left8;
      z = z < all_tiles ? z : all_tiles;
      int v = u - full;
      // A range more for the blocks of adapters of more than 64 where that fits beside the others: a stage of theirs is 24 KB, of the others 12 or 16
      // (8 requests of mixed ranks 18.6 -> 17.6 us, 16 of 357 .. 961 rows 26.0 -> 22.9; the wait for the ranks before the sum
      // does not show: within 0.05 either way without it)
      const int h8 = (heavy + 7) & ~7, l8 = (nb - heavy + 7) & ~7;
      if (full == 0 && p.n_layers == 1 && heavy > 0 && heavy < nb && z < all_tiles && h8 * (z + 1) + l8 * z <= CUS) {
        const bool mine = v < h8 * (z + 1);
        upto = mine ? (int)(sum >> 16) : upto - (int)(sum >> 16);
        v = mine ? v : v - h8 * (z + 1);
        last = mine ? heavy : nb - heavy;
        z = mine ? z + 1 : z;
      }
      const int per = (all_tiles + z - 1) / z;
      z = (all_tiles + per - 1) / per;
      const int w = v % (8 * z);
      b = full + v / (8 * z) * 8 + w % 8;
      if (b >= last) return;                      // uniform over the workgroup
      j0 = w / 8 * per;
      n_tiles = all_tiles - j0 < per ? all_tiles - j0 : per;
    }
    layer = b / per_layer;
    const int bl = b % per_layer;
    const int seg = __builtin_ctzll(__ballot(upto > bl));
    m0 = (bl - (__builtin_amdgcn_readlane(upto, seg) - __builtin_amdgcn_readlane(blocks, seg))) * BM;
    r0 = __builtin_amdgcn_readlane(st, seg);
    M = __builtin_amdgcn_readlane(rows, seg);     // rows of this segment
    ad = __builtin_amdgcn_readlane(a, seg);
    rank = __builtin_amdgcn_readlane(rk, seg);    // multiple of 32, <= RP
    scale = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, sc), seg));
  } else {
    const int seg = blockIdx.y;
    r0 = p.seg_start[seg]; M = p.seg_start[seg + 1] - r0; ad = p.seg_adapter[seg];
    m0 = blockIdx.x * BM;
    if (ad < 0 || m0 >= M) return;                // uniform over the workgroup
    rank = p.adapter_rank[ad]; scale = p.adapter_scale[ad];
    layer = (int)blockIdx.z / p.z_per_layer;
    j0 = (int)blockIdx.z % p.z_per_layer * p.tiles_per_z;
    n_tiles = all_tiles - j0 < p.tiles_per_z ? all_tiles - j0 : p.tiles_per_z;
  }
  const int K = p.K, N = p.N, RP = p.RP;
  // (in scalar registers by name: a descriptor that the compiler takes for a wave's own costs a loop around each of its loads)
  auto uni = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  m0 = uni(m0); layer = uni(layer); r0 = uni(r0); M = uni(M); ad = uni(ad); rank = uni(rank); j0 = uni(j0); n_tiles = uni(n_tiles);
  const bf16_t* a_all = p.a_all; const bf16_t* b_all = p.b_all; bf16_t* y_all = p.y;
  if (p.table != nullptr) {
    const uint64_t* row = p.table + (size_t)layer * 3;
    auto entry = [&](int i) { const uint64_t v = row[i]; return (uint64_t)(uint32_t)uni((int)(v >> 32)) << 32 | (uint32_t)uni((int)v); };
    a_all = reinterpret_cast<const bf16_t*>(entry(0)); b_all = reinterpret_cast<const bf16_t*>(entry(1)); y_all = reinterpret_cast<bf16_t*>(entry(2));
  }
  const bf16_t* x = p.x + (size_t)r0 * K;
  bf16_t* y = y_all + (size_t)r0 * N;
  const bf16_t* A = a_all + (size_t)ad * RP * K;
  const bf16_t* B = b_all + (size_t)ad * N * RP;

  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;        // 2 x 4 waves: a wave owns BM / 2 rows x 32 columns of a BM x 128 tile
  const int lr = lane & 15, lg = lane >> 4;

  auto clamp32 = [](size_t bytes) { return (int)(uint32_t)(bytes < 0xFFFFFFFFull ? bytes : 0xFFFFFFFFull); };
  auto mk = [&](const bf16_t* base, size_t bytes) {
    const uint64_t a = (uint64_t)base;
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>((uint64_t)(uint32_t)uni((int)(a >> 32)) << 32 | (uint32_t)uni((int)a)), 0,
                                             uni(clamp32(bytes)), 0x00020000);
  };

  // Stages are 128-byte rows of eight 16-byte pieces.  x and T: piece c of row r at c ^ (r / 2 % 8), fragment rows in order.  A and B: fragment
  // row m of the two 16-row tiles of a wave's 32 rows is row 8 (m / 4) + 4 tile + m % 4, so that a lane's results of both tiles are eight
  // neighbouring columns of one row (one 16-byte piece of T or y); the swizzle that keeps those 16 rows on different banks is another one.
  auto swz = [](int r) { return ((r >> 1) & 1) | ((r >> 3) & 3) << 1; };

  // ---- requests.  Phase 1: DMA units of 8 rows x 128 bytes, XU of x and one or two of A per wave and stage; a lane's byte offset (row, swizzled
  // piece) never changes, the K tile is a scalar offset.  Rows beyond the segment or the rank: offsets beyond the buffer, zeros. ----
  const int KT = K / 64;
  const rsrc_t rs_x = mk(x + (size_t)m0 * K, (size_t)(M - m0) * K * 2);
  const rsrc_t rs_a = mk(A, (size_t)RP * K * 2);
  const rsrc_t rs_b = mk(B, (size_t)N * RP * 2);
  const rsrc_t rs_y = mk(y + (size_t)m0 * N, (size_t)(M - m0) * N * 2);
  uint32_t vx[XU], va[2], vb[2], vy[TI], gone[TI];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int r = (wave + 8 * q) * 8 + (lane >> 3), rb = (wave * 2 + q) * 8 + (lane >> 3);
    if (q < XU) vx[q < XU ? q : 0] = r < M - m0 ? (uint32_t)r * (uint32_t)K * 2u + (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16) : 0xFFFFFFFFu;
    va[q] = r < rank ? (uint32_t)r * (uint32_t)K * 2u + (uint32_t)(((lane & 7) ^ swz(r)) * 16) : 0xFFFFFFFFu;
    vb[q] = (uint32_t)rb * (uint32_t)RP * 2u + (uint32_t)(((lane & 7) ^ swz(rb)) * 16);
  }
  // phase 2: B tile j: rows n0 .. n0+127 of B (row stride RP), 64 rank columns per stage, 16 units per stage, two per wave; y pieces of tile j: rows
  // 16 i + lr of the wave's, columns 8 lg .. 8 lg + 7
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    const int r = wm * (BM / 2) + i * 16 + lr;
    gone[i] = (uint32_t)((M - m0 - 1 - r) >> 31);
    vy[i] = ((uint32_t)r * (uint32_t)N * 2u + (uint32_t)((j0 * 128 + wn * 32 + lg * 8) * 2)) | gone[i];
  }
  auto b_stage = [&](int j, int s) { return smem + RING - (j & D) * B_TILE + s * (128 * 128); };
  auto issue_b = [&](int j, int s) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_b, (lptr_t)(b_stage(j, s) + (wave * 2 + q) * 1024), 16, vb[q] + s * 128, (j0 + j) * 128 * RP * 2, 0, 0);
  };
  u32x4 yr[YD][TI];
  auto issue_y = [&](int j, u32x4 (&d)[TI]) {     // (past the last tile: no memory is read, but the request counts)
    const uint32_t past = (uint32_t)((n_tiles - 1 - j) >> 31);
#pragma unroll
    for (int i = 0; i < TI; ++i)
      d[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_y, vy[i] | past, j < n_tiles ? j * 256 : 0, 0));
  };

  auto body = [&](auto au) {                      // au: A units per wave, and 64-column stages of the rank
    constexpr int AU = decltype(au)::value, NST = RING / (BM * 128 + AU * 8192), CNT = XU + AU, AOFF = NST * BM * 128;
    // ---- phase 1: T = x_tile . A^T ----
    const bool mine = wn * 32 < rank;             // (waves whose rank columns lie beyond the rank only move operands)
    struct Fr { bf16x8 a[2][TI]; bf16x8 b[2][2]; };
    auto issue = [&](int t, int slot) {
#pragma unroll
      for (int q = 0; q < XU; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_x, (lptr_t)(smem + slot * (BM * 128) + (wave + 8 * q) * 1024), 16, vx[q], t * 128, 0, 0);
#pragma unroll
      for (int q = 0; q < AU; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_a, (lptr_t)(smem + AOFF + slot * (AU * 8192) + (wave + 8 * q) * 1024), 16, va[q], t * 128, 0, 0);
    };
    const int wrow = 8 * (lr >> 2) + (lr & 3);    // (+ 4: second tile; its swizzle is the same)
    auto read_frags = [&](int slot, Fr& f) {
      const char *sx = smem + slot * (BM * 128) + (wm * (BM / 2) + lr) * 128, *sa = smem + AOFF + slot * (AU * 8192) + (wn * 32 + wrow) * 128;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int i = 0; i < TI; ++i) f.a[ks][i] = *reinterpret_cast<const bf16x8*>(sx + i * 2048 + ((4 * ks + lg) ^ (lr >> 1)) * 16);
#pragma unroll
        for (int h = 0; h < 2; ++h) f.b[ks][h] = *reinterpret_cast<const bf16x8*>(sa + h * 512 + ((4 * ks + lg) ^ swz(wrow)) * 16);
      }
    };
    f32x4 acc[TI][2];
    auto zero_acc = [&]() {
#pragma unroll
      for (int i = 0; i < TI; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
#pragma unroll
    for (int s = 0; s < AU; ++s) issue_b(0, s);
#pragma unroll 1
    for (int t = 0; t < (KT < NST ? KT : NST); ++t) issue(t, t);
    zero_acc();
    auto mma = [&](const Fr& f) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int h = 0; h < 2; ++h) acc[i][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.b[ks][h], f.a[ks][i], acc[i][h], 0, 0, 0);
    };
    if constexpr (BM == 64) {
      // a stage's fragments are read while the stage before is multiplied
      Fr f0, f1;
      int slot = 0, t = 0;                        // stage t, whose fragments are in registers or under way to them, and its place
      auto step = [&](Fr& cur, Fr& next) {
        wait_cnt<CNT*(NST - 2), 0>();             // this wave's loads of stage t + 1 are complete, its fragments of stage t read
        __builtin_amdgcn_s_barrier();             // everyone's are
        __builtin_amdgcn_sched_barrier(0);
        issue(t + NST, slot);
        slot = slot + 1 == NST ? 0 : slot + 1;
        ++t;
        if (mine) {
          read_frags(slot, next);
          mma(cur);
        }
      };
      // (the loop in pairs of stages, the last NST stages by themselves, from f0 on: they request nothing)
      const int head = KT > NST ? KT - NST : 0;
      if (KT >= NST) wait_cnt<CNT*(NST - 1), 0>(); else wait_cnt<0, 0>();
      __builtin_amdgcn_s_barrier();
      if (KT >= NST ? head & 1 : (NST - KT) & 1) {
        if (mine) read_frags(0, f1);
        if (KT > NST) step(f1, f0);
      } else if (mine) {
        read_frags(0, f0);
      }
#pragma unroll 1
      while (t + 4 < head) {
        step(f0, f1);
        step(f1, f0);
      }
      // (here, so that the last stages are behind them: the waits count only those)
#pragma unroll
      for (int i = 0; i < YD; ++i) issue_y(i, yr[i]);
#pragma unroll 1
      while (t < head) {
        step(f0, f1);
        step(f1, f0);
      }
      auto last = [&](auto rc, Fr& cur, Fr& next) { // r stages follow
        constexpr int r = decltype(rc)::value;
        if (r >= KT) return;
        if constexpr (r > 0) {
          wait_cnt<CNT*(r - 1), 0>();
          __builtin_amdgcn_s_barrier();
          __builtin_amdgcn_sched_barrier(0);
          slot = slot + 1 == NST ? 0 : slot + 1;
        }
        if (mine) {
          if constexpr (r > 0) read_frags(slot, next);
          mma(cur);
        }
      };
      auto both = [&](auto rc) {
        constexpr int r = decltype(rc)::value;
        if constexpr (r < NST) {
          if constexpr ((NST - 1 - r) % 2 == 0) last(rc, f0, f1); else last(rc, f1, f0);
        }
      };
      both(std::integral_constant<int, 7>{}); both(std::integral_constant<int, 6>{}); both(std::integral_constant<int, 5>{});
      both(std::integral_constant<int, 4>{}); both(std::integral_constant<int, 3>{}); both(std::integral_constant<int, 2>{});
      both(std::integral_constant<int, 1>{}); both(std::integral_constant<int, 0>{});
      static_assert(NST >= 4 && NST <= 8, "the last stages");
    } else {
      // (128 rows: two stages of fragments beside all else do not fit the registers)
      Fr f;
      int slot = 0;
#pragma unroll
      for (int i = 0; i < YD; ++i) issue_y(i, yr[i]);
#pragma unroll 1
      for (int t = 0; t < KT; ++t) {
        if (t == 0 && NST <= KT) wait_cnt<CNT*(NST - 1), 0>();
        else if (t + NST <= KT + 1) wait_cnt<CNT*(NST - 2), 0>();
        else wait_cnt<0, 0>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (t > 0 && t + NST - 1 < KT) issue(t + NST - 1, slot == 0 ? NST - 1 : slot - 1);
        if (mine) {
          read_frags(slot, f);
          mma(f);
        }
        slot = slot + 1 == NST ? 0 : slot + 1;
      }
    }
    wait_cnt<0, 0>();                             // (the y pieces)
    __builtin_amdgcn_s_barrier();                 // the ring is dead
    __builtin_amdgcn_sched_barrier(0);

    // ---- phase 2: y tile += scale * T . B_tile^T for every 128-column tile ----
#pragma unroll
    for (int j = 1; j <= D; ++j)
#pragma unroll
      for (int s = 0; s < AU; ++s)
        if (j < n_tiles) issue_b(j, s);
    // T, rounded to bf16, into the stage layout
    if (mine) {
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const u32x4 o = {pack_bf16x2(acc[i][0][0], acc[i][0][1]), pack_bf16x2(acc[i][0][2], acc[i][0][3]),
                         pack_bf16x2(acc[i][1][0], acc[i][1][1]), pack_bf16x2(acc[i][1][2], acc[i][1][3])};
        const int c = wn * 4 + lg;
        *reinterpret_cast<u32x4*>(smem + (c >> 3) * (BM * 128) + (wm * (BM / 2) + i * 16 + lr) * 128 + (((c & 7) ^ (lr >> 1)) * 16)) = o;
      }
    }
    const int steps = (rank + 31) / 32;           // MFMA steps over the padded rank
    bf16x8 tf[2 * AU][TI];
    constexpr int CB = 2 * AU, ST = TI;           // requests of a B tile, stores of a tile
    auto tile = [&](int j, auto ic, u32x4 (&yc)[TI]) {
      // B tile j (this wave's share) is here; what is younger -- a wave's memory operations complete in order --, the next tiles of B and the
      // stores of the tiles before, may still be on its way
      constexpr int i0 = decltype(ic)::value;     // tile j is the first (0), one of those up to D, or a later one
      const int ahead = n_tiles - 1 - j;
      if constexpr (i0 == 0) wait_cnt<63, 0>();
      else if (ahead >= 2) wait_cnt<2 * CB + i0 * ST, 0>();
      else if (ahead == 1) wait_cnt<CB + i0 * ST, 0>();
      else wait_cnt<i0 * ST, 0>();
      __builtin_amdgcn_s_barrier();               // everyone's is, everyone has read tile j - 1 (tile 0: has written its part of T)
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (i0 == 0) {
#pragma unroll
        for (int ks = 0; ks < 2 * AU; ++ks)
          if (ks < steps) {
#pragma unroll
            for (int i = 0; i < TI; ++i)
              tf[ks][i] = *reinterpret_cast<const bf16x8*>(smem + (ks >> 1) * (BM * 128) + (wm * (BM / 2) + i * 16 + lr) * 128 + ((((ks & 1) * 4 + lg) ^ (lr >> 1)) * 16));
          }
      } else {
#pragma unroll
        for (int s = 0; s < AU; ++s)
          if (j + D < n_tiles) issue_b(j + D, s);
      }
      zero_acc();
#pragma unroll
      for (int ks = 0; ks < 2 * AU; ++ks)
        if (ks < steps) {
          const char* sb = b_stage(j, ks >> 1) + (wn * 32 + wrow) * 128 + ((((ks & 1) * 4 + lg) ^ swz(wrow)) * 16);
          const bf16x8 b0 = *reinterpret_cast<const bf16x8*>(sb), b1 = *reinterpret_cast<const bf16x8*>(sb + 512);
#pragma unroll
          for (int i = 0; i < TI; ++i) {
            acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0, tf[ks][i], acc[i][0], 0, 0, 0);
            acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b1, tf[ks][i], acc[i][1], 0, 0, 0);
          }
        }
      // scale, round, add to the y pieces
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t v = pack_bf16x2(acc[i][e >> 1][2 * (e & 1)] * scale, acc[i][e >> 1][2 * (e & 1) + 1] * scale);
          o[e] = pack_bf16x2(bf16_lo(v) + bf16_lo(yc[i][e]), bf16_hi(v) + bf16_hi(yc[i][e]));
        }
        // (no scalar offset: for such stores the compiler leaves out the wait state without which the next vector instruction overwrote the second
        // half of a row's piece now and then)
        __builtin_amdgcn_raw_buffer_store_b128(o, rs_y, (vy[i] + j * 256) | gone[i], 0, STORE_POLICY);
      }
      if (j + YD < n_tiles) issue_y(j + YD, yc);
    };
    // the first tiles by themselves: their y pieces are here
    auto early = [&](auto ic) {
      constexpr int i = decltype(ic)::value;
      if (i < n_tiles) tile(i, std::integral_constant<int, i < D ? i : D>{}, yr[i % YD]);
    };
    early(std::integral_constant<int, 0>{});
    if constexpr (YD > 1) {
      early(std::integral_constant<int, 1>{}); early(std::integral_constant<int, 2>{});
      early(std::integral_constant<int, 3>{}); early(std::integral_constant<int, 4>{});
      for (int j = YD; j < n_tiles; j += YD) {
#pragma unroll
        for (int i = 0; i < YD; ++i) {
          if (j + i >= n_tiles) break;
          tile(j + i, std::integral_constant<int, D>{}, yr[i]);
        }
      }
    } else {
#pragma unroll 1
      for (int j = 1; j < n_tiles; ++j) tile(j, std::integral_constant<int, 1>{}, yr[0]);
    }
    wait_cnt<0, 0>();                             // (or the compiler counts them as under way in the other body)
  };
  if (rank <= 64) body(std::integral_constant<int, 1>{}); else body(std::integral_constant<int, 2>{});
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
  // rows cost more than one of 128 (8 x 4096 rows: 40 against 32 us; 4 x 3136: 19 against 24).  (A 128-row tile of y has to lie within 32 bits.)
  // The rest is dealt on the device; more segments than a wave has lanes, or workgroups than a grid may have threads, by the host's bound.
  const int bm = (max_seg_rows + 63) / 64 * n_segments * n_layers > 320 && N <= (1 << 23) ? 128 : 64;
  const int64_t row_blocks = (max_seg_rows + bm - 1) / bm;
  const int64_t row_wgs = row_blocks * n_segments * n_layers, n_tiles = N / 128;
  if (n_layers > 65535) return KH_ERR_TOO_LARGE;
  p.n_layers = (int)n_layers; p.row_blocks = (int)row_blocks;
  dim3 grid;
  if (n_segments <= 64 && row_wgs <= (1 << 20)) {
    p.n_segments = (int)n_segments; p.tiles_per_z = 0; p.z_per_layer = 0;
    const int64_t most = (row_wgs + 7) / 8 * 8 * n_tiles;
    grid = dim3((unsigned)(row_wgs > CUS ? row_wgs + CUS : most < CUS ? most : CUS));
  } else {
    int64_t z = 300 / row_wgs;
    z = z < 1 ? 1 : z < n_tiles ? z : n_tiles;
    p.n_segments = 0;
    p.tiles_per_z = (int)((n_tiles + z - 1) / z);
    p.z_per_layer = (int)((n_tiles + p.tiles_per_z - 1) / p.tiles_per_z);
    grid = dim3((unsigned)row_blocks, (unsigned)n_segments, (unsigned)(p.z_per_layer * n_layers));
  }
  auto go = [&](auto bmc) {
    constexpr int BM = decltype(bmc)::value;
    if (hipError_t e = kh_allow_lds<sgmv_fused_kernel<BM>>(LDS_BYTES); e != hipSuccess) return (int)e;
    kh_launch(KH_TAG_SGMV_FUSED, sgmv_fused_kernel<BM>, grid, dim3(512), LDS_BYTES, (hipStream_t)stream, p);
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
