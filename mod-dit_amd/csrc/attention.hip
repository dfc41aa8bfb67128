// Dense and block-sparse flash-attention forward for gfx950 (CDNA4).
//
// One workgroup = 4 wave64s = 128 query rows (each wave owns 32 rows as two 16-row blocks);
// keys stream in tiles of 64 (the mask's key-block granularity). Per key tile each wave
// computes, on bf16/fp16 MFMA 16x16x32,
//   S^T (64 keys x 32 queries) = K . Q^T      4 key x 2 query blocks, D/32 steps
//   O^T (d x 32 queries)      += V^T . P^T    D/16 x 2 blocks, 2 steps
// Computing the transposed products puts one query per lane column and block, so the rescale
// of O is a per-lane multiply, and the S^T accumulators of key blocks 2t and 2t+1 are the
// B operand of P^T's step t (the V operand is read in the same key order), so P never
// leaves registers.
//
// What bounds it is the board's power limit: the clock falls until the power fits, so time
// follows the energy of the work, not its schedule. The 16x16x32 shape does the same
// products for less (2.19 against 1.86 PFLOP/s for 32x32x16 on random operands at the
// limit). Its price, two queries per lane and with them twice the row reductions, is kept
// off most tiles: a lane compares its own scores with the running max, and the row max is
// exchanged and moved only where one of them lies far above it (settle). Against the 32x32x16
// kernel with a max per tile, on structured inputs: dense 24 heads x 115,200, D = 128 155.9 ->
// 146.5 ms; block-sparse 40 x 69,120 21.3 -> 20.4 ms; 48 x 17,776, D = 64 1.55 -> 1.44 ms.
// Weighing a tile against the max as it is, and computing it again where that overflows, takes
// the lanes' max off too (147.1, 20.8 and 1.46 ms) but costs peaked rows up to 40 %.
//
// K and V tiles go straight from HBM into LDS (buffer_load ... lds, no register
// staging), both row-major with an XOR swizzle on 16-byte chunks that keeps the operand
// reads bank-conflict free; V^T fragments come out of the row-major V tile through
// ds_read_b64_tr_b16. Two stages per operand. The loop is software pipelined:
// iteration j computes S_{j+1}, then O += P_j V_j together with the softmax of S_{j+1}, while
// K_{j+2} and V_{j+1} stream in; one barrier per tile.
//
// The sparse variant walks a per-(head, query tile) list of key tiles, each entry
// carrying two row bits (query rows 0-63 / 64-127 of the tile); a wave whose bit is
// clear skips the math but still issues its share of the tile's DMA.
//
// Reference semantics: flash_attn_func (MoD/mod/triton_flash_sparsity.py:320-321) for
// the dense pass incl. its LSE; block_sparse_sage2_attn_cuda at 128q x 64k tiles
// (MoD/mod/attn_mask.py:296-317) for the sparse pass, computed here in bf16/fp16 with
// fp32 softmax instead of SageAttention's quantisation.
#include "common.h"
#include "lds_dma.h"

#include <cfloat>

namespace moddit {
namespace {

constexpr int kBM = 128;  // query rows per workgroup
constexpr int kBN = 64;   // keys per tile
constexpr int kThreads = 256;

template <int D>
struct AttnLds {
  static constexpr int kRowBytes = D * 2;                 // one token row, no padding
  static constexpr int kTileBytes = kBN * kRowBytes;      // one 64-key K or V tile
  static constexpr int kTotal = 4 * kTileBytes;           // K ring (2) + V ring (2)
  static constexpr int kChunks = D / 8;                   // 16-byte chunks per row
  static constexpr int kRowsPerWindow = 1024 / kRowBytes; // rows per 1 KB DMA window
  static constexpr int kWindows = kTileBytes / 1024;      // DMA windows per tile
};

struct AttnParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  float* lse;
  int64_t q_sb, q_sh, q_ss;
  int64_t k_sb, k_sh, k_ss;
  int64_t v_sb, v_sh, v_ss;
  int64_t o_sb, o_sh, o_ss;
  int heads;
  int q_len;
  int kv_len;
  int origin;    // token index of grid row/column 0 (-63..0); see moddit_block_sparse_fwd
  int n_qtiles;
  int n_ktiles;
  int xcd_run;    // workgroup -> tile order (xcd_remap)
  float scale_log2;  // softmax_scale * log2(e)
  const int32_t* counts;
  const int32_t* entries;
  int cap;
  uint32_t k_bytes;  // byte span of one head's K rows [0, kv_len)
  uint32_t v_bytes;
  // fused sparsity map (map != nullptr only for the kMap kernels)
  uint16_t* map;     // fp16 (B*H, map_nblk, map_nblk)
  int map_q_off;     // token of video row 0 (== key offset)
  int map_kt0;       // grid key tile holding video key 0
  int map_nblk;      // video blocks per side
  int map_block;     // 64 or 128
  int map_valid;     // video tokens that exist: min(map_nblk*map_block, seq_len - map_q_off)
  float map_scale;   // softmax scale applied to q before rounding
  float map_log_thr; // ln(threshold)
  // split key range (kSplit kernels): `n_split` workgroups per query tile
  int n_split;
  float* part_o;   // [tile][piece][128][D]: unnormalised O of the piece, relative to its max
  float* part_ml;  // [tile][piece][128][2]: running max (log2 units) and row sum
};

// 16-byte chunk swizzles (XOR on the chunk index) that make the MFMA operand reads
// bank-conflict free: K rows are read one row per lane (A operand of S^T), V rows
// through ds_read_b64_tr_b16 (eight keys x 16 dims per half-wave).
template <int D>
__device__ __forceinline__ int swz_k(int r) { return (r / (128 / D)) % (D / 8); }
template <int D>
__device__ __forceinline__ int swz_v(int key) { return 2 * ((key / (128 / D)) % (D / 16)); }

// The running maxima move only on tiles where some lane of the wave holds a score more than
// kRescaleSlack log2 units above its row's; there every row's max moves to the tile's if that
// is larger. Softmax is shift-invariant, so results do not depend on it but for the rounding of
// P, whose weights reach 2^kRescaleSlack at most: a row's largest is exact (1) where the max is
// its own. 6 keeps the error against 64 bits below what 8 units in a kernel with a max per
// row and tile gave, over five seeds of each: 28,800 tokens + text, D = 128, bf16 2.04-2.17e-3
// of the result (2.16-2.22e-3; 8 here: 2.12-2.24e-3); fp16 2.55-2.74e-4 (2.67-2.80e-4; 2.65-
// 2.82e-4). 4 would take another 4-5 % off, and costs rows whose deviation is 2 to 8 2-3 %.
constexpr float kRescaleSlack = 6.0f;

// Waves per SIMD that the registers are held to. D = 128 takes 212-228 (two waves). D = 64 fits
// four in 124-128 (left alone, up to 134; the aligned dense kernel keeps seven invariants of
// its last tile in scratch), the fused map three. Where a launch has four workgroups per CU,
// three waves leave a quarter of them to a second round: 8 heads x 16,384, exact rows, a
// tenth of the tiles: 132 against 104 us.
constexpr int attn_waves(int head_dim, bool map) { return head_dim == 128 ? 2 : (map ? 3 : 4); }

typedef short s16x4 __attribute__((ext_vector_type(4)));

// ds_read_b64_tr_b16: within each 16-lane group, lane i receives element i%4 of the
// 4-element rows addressed by lanes i/4, i/4+4, i/4+8, i/4+12.
__device__ __forceinline__ s16x4 lds_read_tr16(const unsigned char* a) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(a));
}

// Map flush granularity of the fused map pass (key tiles per flush; the LDS count ring
// holds two flushes so that a flush never races the next tiles' counts).
constexpr int kMapFlush = 64;
constexpr int kMapCountBytes = 4 * 2 * kMapFlush * 4;  // int per (wave, ring slot)

// kSplit: one workgroup takes the piece `blockIdx % n_split` of a query tile's key tiles (or
// list entries) and leaves its unnormalised fp32 O, max and sum for combine_kernel.
template <int D, typename E, bool kSparse, bool kRagged, bool kMap = false, bool kSplit = false>
__global__ __launch_bounds__(kThreads, attn_waves(D, kMap)) __attribute__((amdgpu_waves_per_eu(attn_waves(D, kMap), attn_waves(D, kMap)))) void attention_fwd_kernel(AttnParams p) {
  using L = AttnLds<D>;
  using V8 = typename E::vec8;
  constexpr int kKC = D / 32;  // MFMA k-steps over d for S^T
  constexpr int kDB = D / 16;  // 16-row blocks of O^T
  constexpr int kWinPerWave = L::kWindows / 4;

  extern __shared__ __align__(16) unsigned char smem[];
  unsigned char* const k_ring = smem;
  unsigned char* const v_ring = smem + 2 * L::kTileBytes;

  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int g = lane >> 4;
  const int c16 = lane & 15;

  const int tile = kSplit ? blockIdx.x / p.n_split : xcd_remap(blockIdx.x, gridDim.x, p.xcd_run);
  const int qt = tile % p.n_qtiles;
  const int bh = tile / p.n_qtiles;
  const int b = bh / p.heads;
  const int h = bh - b * p.heads;

  const uint16_t* qb = p.q + b * p.q_sb + h * p.q_sh;
  const uint16_t* kb = p.k + b * p.k_sb + h * p.k_sh;
  const uint16_t* vb = p.v + b * p.v_sb + h * p.v_sh;

  int n_iter;
  const int32_t* list = nullptr;
  if (kSparse) {
    const int64_t slot = static_cast<int64_t>(h) * p.n_qtiles + qt;
    n_iter = p.counts[slot];
    n_iter = n_iter < 0 ? 0 : (n_iter < p.cap ? n_iter : p.cap);
    list = p.entries + slot * p.cap;
  } else {
    n_iter = p.n_ktiles;
  }
  int it0 = 0;  // first key tile (dense) of this workgroup's piece
  if constexpr (kSplit) {
    const int piece = blockIdx.x - tile * p.n_split;
    const int first = static_cast<int>(static_cast<int64_t>(n_iter) * piece / p.n_split);
    n_iter = static_cast<int>(static_cast<int64_t>(n_iter) * (piece + 1) / p.n_split) - first;
    if (kSparse)
      list += first;
    else
      it0 = first;
  }
  // A wave whose 32 rows are all padding takes part in the staging only: 2 of the 52 waves of a
  // head of 1,577 tokens, two of the four of a 41-row tail.
  const int first_row = p.origin + qt * kBM + __builtin_amdgcn_readfirstlane(wave) * 32;
  const int wbit = first_row < p.q_len && first_row + 31 >= 0 ? 1 << (wave >> 1) : 0;

  // ---- Q fragments (B operand of S^T = K Q^T): lane holds query 16qq + c16, dims 32c + 8g.. ----
  // Grid rows outside [0, q_len) are padding: they load a clamped row and store nothing.
  const int q_row0 = p.origin + qt * kBM + wave * 32 + c16;  // and + 16
  V8 qf[2][kKC];
#pragma unroll
  for (int qq = 0; qq < 2; ++qq) {
    const int q_row = q_row0 + 16 * qq;
    const int r = q_row < 0 ? 0 : (q_row < p.q_len ? q_row : p.q_len - 1);
    const u32x4* src = reinterpret_cast<const u32x4*>(qb + r * p.q_ss);
#pragma unroll
    for (int c = 0; c < kKC; ++c) qf[qq][c] = as_vec8<V8>(src[4 * c + g]);
  }
  __builtin_amdgcn_s_waitcnt(0);

  // ---- direct global -> LDS staging (buffer_load ... lds, 16 B per lane) ----
  // DMA window w writes LDS bytes [w*1024, w*1024+1024) of a stage, lane l at l*16. The
  // per-lane source is chosen so that the window holds the swizzled rows.
  const u32x4 k_rsrc = raw_rsrc(kb, p.k_bytes);
  const u32x4 v_rsrc = raw_rsrc(vb, p.v_bytes);
  const uint32_t k_lds = lds_addr(k_ring);
  const uint32_t v_lds = lds_addr(v_ring);
  uint32_t k_src[kWinPerWave];
  uint32_t v_src[kWinPerWave];
#pragma unroll
  for (int i = 0; i < kWinPerWave; ++i) {
    const int w = wave * kWinPerWave + i;
    const int r = w * L::kRowsPerWindow + (lane * 16) / L::kRowBytes;  // LDS row
    const int pch = ((lane * 16) % L::kRowBytes) / 16;                  // physical chunk
    const int kq = pch ^ swz_k<D>(r);                                   // logical chunk
    const int vq = pch ^ swz_v<D>(r);
    k_src[i] = static_cast<uint32_t>((r * p.k_ss + kq * 8) * 2);
    v_src[i] = static_cast<uint32_t>((r * p.v_ss + vq * 8) * 2);
  }
  const uint32_t k_tile_bytes = static_cast<uint32_t>(kBN * p.k_ss * 2);
  const uint32_t v_tile_bytes = static_cast<uint32_t>(kBN * p.v_ss * 2);
  // Grid origin in bytes (two's complement). Keys before token 0 get offsets that wrap
  // to >= 2^31, beyond every range the buffer descriptors admit, so they load zeros.
  const uint32_t k_org = static_cast<uint32_t>(p.origin * static_cast<int>(p.k_ss) * 2);
  const uint32_t v_org = static_cast<uint32_t>(p.origin * static_cast<int>(p.v_ss) * 2);

  auto dma_k = [&](int kt, int stage) {
    const uint32_t to = static_cast<uint32_t>(kt) * k_tile_bytes;
#pragma unroll
    for (int i = 0; i < kWinPerWave; ++i) {
      const uint32_t dst = k_lds + stage * L::kTileBytes + (wave * kWinPerWave + i) * 1024;
      if constexpr (kRagged)
        lds_dma16(k_rsrc, dst, k_src[i] + to + k_org, 0);
      else
        lds_dma16(k_rsrc, dst, k_src[i], to);
    }
  };
  auto dma_v = [&](int kt, int stage) {
    const uint32_t to = static_cast<uint32_t>(kt) * v_tile_bytes;
#pragma unroll
    for (int i = 0; i < kWinPerWave; ++i) {
      const uint32_t dst = v_lds + stage * L::kTileBytes + (wave * kWinPerWave + i) * 1024;
      if constexpr (kRagged)
        lds_dma16(v_rsrc, dst, v_src[i] + to + v_org, 0);
      else
        lds_dma16(v_rsrc, dst, v_src[i], to);
    }
  };

  // ---- LDS operand addressing ----
  // K (A operand of S^T): lane reads row 16kb + c16, logical chunk 4c + g.
  uint32_t k_rd[kKC];
#pragma unroll
  for (int c = 0; c < kKC; ++c)
    k_rd[c] = static_cast<uint32_t>(c16 * L::kRowBytes + (((4 * c + g) ^ swz_k<D>(c16)) * 16));
  // V (A operand of O^T, via ds_read_b64_tr_b16): in 16-lane group g lane c16 addresses key
  // 4g + c16/4 (+ 32t + 16s) and dims 16db + 4(c16%4).., and receives dim 16db + c16 of keys
  // 32t + 16s + 4g .. +3. With s = 0 and 1 in the two halves of the operand, k index 8g + e
  // is key 32t + 4g + e (e < 4) or 32t + 12 + 4g + e: the keys of the lane's own scores in
  // key blocks 2t and 2t + 1, so P needs no shuffle.
  const int v_key0 = 4 * g + (c16 >> 2);
  uint32_t v_rd[kDB];
#pragma unroll
  for (int db = 0; db < kDB; ++db) {
    const int d = db * 16 + 4 * (c16 & 3);
    v_rd[db] = static_cast<uint32_t>(v_key0 * L::kRowBytes + (((d >> 3) ^ swz_v<D>(v_key0)) * 16) + (d & 7) * 2);
  }

  f32x4 oacc[kDB][2];
#pragma unroll
  for (int db = 0; db < kDB; ++db) oacc[db][0] = oacc[db][1] = f32x4{};
  float m_run[2] = {-FLT_MAX, -FLT_MAX};  // never -inf: no difference of maxima is NaN
  float l_run[2] = {0.f, 0.f};  // this lane's keys only

  auto decode = [&](int e_raw, int& kt, int& flags) {
    const int e = __builtin_amdgcn_readfirstlane(e_raw);
    kt = e >> 2;
    // An entry outside the grid's key tiles [0, n_ktiles) holds no key of the sequence
    // (a 128-token block mask on a sequence that ends in the first half of its last
    // block lists such a tile): it is executed by no wave; its DMA loads a tile in range.
    flags = (kt >= 0 && kt < p.n_ktiles) ? (e & 3) : 0;
    kt = kt < 0 ? 0 : (kt < p.n_ktiles ? kt : p.n_ktiles - 1);
  };
  auto entry = [&](int i) -> int { return kSparse ? list[i] : (((it0 + i) << 2) | 3); };

  // s[kb][qq][j]: key 16kb + 4g + j, query 16qq + c16
  auto qk = [&](const unsigned char* ks, f32x4 (&s)[4][2]) {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) s[kb][0] = s[kb][1] = f32x4{};
#pragma unroll
    for (int c = 0; c < kKC; ++c) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const V8 a = *reinterpret_cast<const V8*>(ks + k_rd[c] + 16 * kb * L::kRowBytes);
        s[kb][0] = E::mma16(a, qf[0][c], s[kb][0]);
        s[kb][1] = E::mma16(a, qf[1][c], s[kb][1]);
      }
    }
    // D = 128: K reads four fragments ahead of their products, one per two products. Left to
    // itself the compiler issues most reads right before their use, and each pair of them is
    // waited for: with it, 128 to 256 workgroups of 64 to 256 tiles took 2-6 % longer (4 heads x
    // 4,096 tokens, all tiles: 90 against 86 us), exact rows 3-4 %, and at the power limit 1-2 %
    // (dense 24 x 115,200: 147.9 against 146.5 ms). 6 to 12 ahead are no better. D = 64 spills.
    if constexpr (D == 128) {
      constexpr int kReads = 4 * kKC, kAhead = 4;
      __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);  // 0x100: LDS reads
#pragma unroll
      for (int i = 0; i < kReads - kAhead; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);     // 0x008: MFMAs
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 2 * kAhead, 0);
    }
  };
  // O += P V: of its 2 kDB steps in the order (t, db), [i0, i1)
  auto pv = [&](const unsigned char* vs, const V8 (&pb)[2][2], int i0 = 0, int i1 = D / 8) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int db = 0; db < kDB; ++db) {
        if (t * kDB + db < i0 || t * kDB + db >= i1) continue;
        const unsigned char* a = vs + v_rd[db] + t * 32 * L::kRowBytes;
        const s16x4 lo = lds_read_tr16(a);
        const s16x4 hi = lds_read_tr16(a + 16 * L::kRowBytes);
        const u32x4 w = {__builtin_bit_cast(u32x2, lo).x, __builtin_bit_cast(u32x2, lo).y,
                         __builtin_bit_cast(u32x2, hi).x, __builtin_bit_cast(u32x2, hi).y};
        oacc[db][0] = E::mma16(as_vec8<V8>(w), pb[0][t], oacc[db][0]);
        oacc[db][1] = E::mma16(as_vec8<V8>(w), pb[1][t], oacc[db][1]);
      }
    }
  };
  // Moves the running maxima, and sets alpha and rescale, only where a lane of the wave holds a
  // score more than kRescaleSlack above its row's max.
  auto settle = [&](const f32x4 (&s)[4][2], float (&alpha)[2], bool& rescale) {
    float mx[2];
#pragma unroll
    for (int qq = 0; qq < 2; ++qq) {
      mx[qq] = s[0][qq][0];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j) mx[qq] = fmaxf(mx[qq], s[kb][qq][j]);
    }
    const float over = fmaxf(__builtin_fmaf(mx[0], p.scale_log2, -m_run[0]),
                             __builtin_fmaf(mx[1], p.scale_log2, -m_run[1]));
    if (__builtin_expect(__ballot(over > kRescaleSlack) != 0ull, 0)) {
#pragma unroll
      for (int qq = 0; qq < 2; ++qq) {
        const float m_new = fmaxf(m_run[qq], max_over_groups(mx[qq]) * p.scale_log2);
        alpha[qq] = __builtin_amdgcn_exp2f(m_run[qq] - m_new);
        l_run[qq] *= alpha[qq];
        m_run[qq] = m_new;
      }
      rescale = true;
    }
  };
  // P = exp2(s - m) and its share of the row sums
  auto weigh = [&](const f32x4 (&s)[4][2], V8 (&pb)[2][2]) {
#pragma unroll
    for (int qq = 0; qq < 2; ++qq) {
      float rs = 0.f;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][qq][j], p.scale_log2, -m_run[qq]));
          rs += e;
          pb[qq][kb >> 1][(kb & 1) * 4 + j] = static_cast<typename E::elem>(e);
        }
      l_run[qq] += rs;
    }
  };
  // keys outside the sequence: a score of -inf
  auto mask = [&](f32x4 (&s)[4][2], int kt) {
    const int key0 = p.origin + kt * kBN;
    // comparing the constant 16kb + j against per-tile bounds keeps no per-element value live
    const int lo = -key0 - 4 * g;           // key >= 0       <=> 16kb + j >= lo
    const int hi = p.kv_len - key0 - 4 * g; // key < kv_len   <=> 16kb + j < hi
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool out = 16 * kb + j < lo || 16 * kb + j >= hi;
        s[kb][0][j] = out ? -INFINITY : s[kb][0][j];
        s[kb][1][j] = out ? -INFINITY : s[kb][1][j];
      }
  };
  auto crosses_edge = [&](int kt) -> bool {
    if constexpr (!kRagged) return false;
    const int key0 = p.origin + kt * kBN;
    return key0 < 0 || key0 + kBN > p.kv_len;
  };
  auto rescale_o = [&](const float (&alpha)[2]) {
#pragma unroll
    for (int db = 0; db < kDB; ++db) {
      oacc[db][0] *= alpha[0];
      oacc[db][1] *= alpha[1];
    }
  };

  // ---- prologue: K_0, V_0 -> stage 0, K_1 -> K stage 1; S_0 -> P_0 ----
  V8 pb[2][2];
  bool act_cur = false;
  int e_n1 = 0, e_n2 = 0;
  if (n_iter > 0) {
    const int e0 = entry(0);
    if (n_iter > 1) e_n1 = entry(1);
    if (n_iter > 2) e_n2 = entry(2);
    int kt0, f0;
    decode(e0, kt0, f0);
    dma_k(kt0, 0);
    dma_v(kt0, 0);
    if (n_iter > 1) {
      int kt1, f1;
      decode(e_n1, kt1, f1);
      dma_k(kt1, 1);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    act_cur = (f0 & wbit) != 0;
    if (act_cur) {
      f32x4 s[4][2];
      qk(k_ring, s);
      if (crosses_edge(kt0)) mask(s, kt0);
      float alpha[2];
      bool rescale;
      settle(s, alpha, rescale);
      weigh(s, pb);
    }
    __syncthreads();  // K stage 0 is refilled by the first iteration
  }

  // Iteration j: S_{j+1} = K_{j+1} Q^T, O += P_j V_j, P_{j+1} = softmax(S_{j+1}); K_{j+2}
  // and V_{j+1} stream into the stages freed by iteration j-1.
  bool pend = false;
  float pend_alpha[2] = {1.f, 1.f};
  for (int j = 0; j < n_iter; ++j) {
    const bool has1 = j + 1 < n_iter;
    const bool has2 = j + 2 < n_iter;
    int kt1 = 0, f1 = 0, kt2 = 0, f2 = 0;
    if (has1) decode(e_n1, kt1, f1);
    if (has2) decode(e_n2, kt2, f2);
    int e_n3 = 0;
    if (j + 3 < n_iter) e_n3 = entry(j + 3);
    if (has2) dma_k(kt2, j & 1);
    if (has1) dma_v(kt1, (j + 1) & 1);
    __builtin_amdgcn_sched_barrier(0);

    if (pend) {
      rescale_o(pend_alpha);
      pend = false;
    }
    const bool act_next = has1 && ((f1 & wbit) != 0);
    const unsigned char* vs = v_ring + (j & 1) * L::kTileBytes;
    const unsigned char* ks1 = k_ring + ((j + 1) & 1) * L::kTileBytes;
    if (act_cur && act_next) {
      f32x4 s[4][2];
      // The P.V steps lie where something else waits. D = 128: some under the max of the new
      // scores, the others under their weights (10 and 6 of 16; 12 and 4: 3 % slower on small
      // launches; 16 and 0: 4-7 % there and 3 % on large dense calls); left to itself the
      // scheduler spreads the S products over them, and the softmax waits. D = 64: half the
      // products and as much softmax, which starts sooner after P.V; four waves cover the rest.
      constexpr int kUnderMax = 10;
      if constexpr (D == 64) pv(vs, pb);
      qk(ks1, s);
      if (crosses_edge(kt1)) mask(s, kt1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (D == 128) pv(vs, pb, 0, kUnderMax);
      settle(s, pend_alpha, pend);
      if constexpr (D == 128) pv(vs, pb, kUnderMax);
      V8 pn[2][2];
      weigh(s, pn);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        pb[0][t] = pn[0][t];
        pb[1][t] = pn[1][t];
      }
    } else {
      if (act_cur) pv(vs, pb);
      if (act_next) {
        f32x4 s[4][2];
        qk(ks1, s);
        if (crosses_edge(kt1)) mask(s, kt1);
        settle(s, pend_alpha, pend);
        weigh(s, pb);
      }
    }
    act_cur = act_next;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    e_n1 = e_n2;
    e_n2 = e_n3;
  }
  if (pend) rescale_o(pend_alpha);

  // ---- epilogue ----
  float l_tot[2];
#pragma unroll
  for (int qq = 0; qq < 2; ++qq) l_tot[qq] = sum_over_groups(l_run[qq]);
  if constexpr (kSplit) {
#pragma unroll
    for (int qq = 0; qq < 2; ++qq) {
      const int64_t row = static_cast<int64_t>(blockIdx.x) * kBM + wave * 32 + 16 * qq + c16;
#pragma unroll
      for (int db = 0; db < kDB; ++db)
        *reinterpret_cast<f32x4*>(p.part_o + row * D + db * 16 + 4 * g) = oacc[db][qq];
      if (g == 0) {
        p.part_ml[2 * row] = m_run[qq];
        p.part_ml[2 * row + 1] = l_tot[qq];
      }
    }
    return;
  }
#pragma unroll
  for (int qq = 0; qq < 2; ++qq) {
    const int q_row = q_row0 + 16 * qq;
    if (q_row < 0 || q_row >= p.q_len) continue;
    const float inv = l_tot[qq] > 0.f ? 1.f / l_tot[qq] : 0.f;
    uint16_t* orow = p.o + b * p.o_sb + h * p.o_sh + q_row * p.o_ss;
#pragma unroll
    for (int db = 0; db < kDB; ++db) {
      u32x2 w;
      w.x = pack2(E::from_float(oacc[db][qq][0] * inv), E::from_float(oacc[db][qq][1] * inv));
      w.y = pack2(E::from_float(oacc[db][qq][2] * inv), E::from_float(oacc[db][qq][3] * inv));
      *reinterpret_cast<u32x2*>(orow + db * 16 + 4 * g) = w;
    }
    if (p.lse != nullptr && g == 0) {
      const int64_t li = static_cast<int64_t>(bh) * p.q_len + q_row;
      p.lse[li] = l_tot[qq] > 0.f ? (m_run[qq] + log2f(l_tot[qq])) * 0.69314718055994531f : -INFINITY;
    }
  }

  if constexpr (kMap) {
    // ---- fused sparsity map: with this tile's final LSE in registers, sweep the video
    // key tiles again with bf16(q*scale) and count the scores below lse + ln(threshold)
    // (MoD/mod/cuda_flash_sparsity_kernel.cu:82-163). The grid origin puts every video
    // block on this tile's 64/128-row boundaries, so the counts of waves (0,1) / (2,3)
    // (or all four, for 128-blocks) are whole map cells.
    const int vrow_tile = p.origin + qt * kBM - p.map_q_off;  // multiple of 128
    if (vrow_tile + kBM <= 0 || vrow_tile >= p.map_valid) return;  // uniform per workgroup
    float thr[2];
#pragma unroll
    for (int qq = 0; qq < 2; ++qq) {
      const int vrow = vrow_tile + wave * 32 + 16 * qq + c16;
      const bool row_ok = vrow >= 0 && vrow < p.map_valid;
      // the LSE exactly as stored above
      const float lse_row = l_tot[qq] > 0.f ? (m_run[qq] + log2f(l_tot[qq])) * 0.69314718055994531f : -INFINITY;
      thr[qq] = row_ok ? lse_row + p.map_log_thr : -INFINITY;
      // q scaled in fp32 and rounded to the storage type (reference :86-92)
      const int q_row = q_row0 + 16 * qq;
      const int r = q_row < 0 ? 0 : (q_row < p.q_len ? q_row : p.q_len - 1);
      const u32x4* src = reinterpret_cast<const u32x4*>(qb + r * p.q_ss);
#pragma unroll
      for (int c = 0; c < kKC; ++c) {
        const u32x4 raw = src[4 * c + g];
        uint16_t e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = E::from_float(E::to_float(u16_at(raw, j)) * p.map_scale);
        qf[qq][c] = as_vec8<V8>(u32x4{pack2(e[0], e[1]), pack2(e[2], e[3]), pack2(e[4], e[5]),
                                      pack2(e[6], e[7])});
      }
    }
    // K-only pass: all four 16 KB stages of the K and V rings form one K ring, filled
    // three tiles ahead; the count ring sits past them.
    int* cnt = reinterpret_cast<int*>(smem + 4 * L::kTileBytes);
    const int n_vt = p.map_nblk * p.map_block / kBN;
    uint16_t* out_bh = p.map + static_cast<int64_t>(bh) * p.map_nblk * p.map_nblk;
    const float inv_area = 1.0f / static_cast<float>(p.map_block * p.map_block);
#pragma unroll
    for (int t = 0; t < 3; ++t)
      if (t < n_vt) dma_k(p.map_kt0 + t, t);
    // Each wave issues kWinPerWave DMAs per K tile (4 at d=128, 2 at d=64), and vector
    // memory operations retire in issue order: tile 0 has landed once at most the two
    // later tiles' DMAs are outstanding.
    static_assert(3 * kWinPerWave < 16, "vmcnt immediate holds at most 15");
    if (n_vt >= 3)
      MODDIT_WAIT_VM_LGKM0(2 * kWinPerWave);
    else
      MODDIT_WAIT_VM_LGKM0(0);
    __syncthreads();
    for (int j = 0; j < n_vt; ++j) {
      // stage (j+3)%4 held tile j-1, read in the previous iteration (barrier since)
      if (j + 3 < n_vt) dma_k(p.map_kt0 + j + 3, (j + 3) & 3);
      __builtin_amdgcn_sched_barrier(0);
      f32x4 s[4][2];
      qk(k_ring + (j & 3) * L::kTileBytes, s);
      int total = 0;
      const bool last = j * kBN + kBN > p.map_valid;  // keys past the sequence end are not counted
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bool in = !last || j * kBN + 16 * kb + 4 * g + i < p.map_valid;
          total += __builtin_popcountll(__ballot(s[kb][0][i] < thr[0] && in));
          total += __builtin_popcountll(__ballot(s[kb][1][i] < thr[1] && in));
        }
      if (lane == 0) cnt[wave * 2 * kMapFlush + (j % (2 * kMapFlush))] = total;
      // tile j+1 must have landed; the DMAs of tiles j+2 and j+3 (and any map stores,
      // which are younger than tile j+1's DMA) may stay outstanding
      if (j + 3 < n_vt)
        MODDIT_WAIT_VM_LGKM0(2 * kWinPerWave);
      else if (j + 2 < n_vt)
        MODDIT_WAIT_VM_LGKM0(kWinPerWave);
      else
        MODDIT_WAIT_VM_LGKM0(0);
      __syncthreads();
      const int slot_hi = j % kMapFlush;
      if (slot_hi == kMapFlush - 1 || j + 1 == n_vt) {
        const int j0 = j - slot_hi;
        const int hb = ((j / kMapFlush) & 1) * kMapFlush;
        if (p.map_block == 64) {
          if (tid < 2 * kMapFlush) {
            const int qsub = tid / kMapFlush;
            const int sl = tid % kMapFlush;
            const int qblk = vrow_tile / 64 + qsub;
            if (sl <= slot_hi && qblk >= 0 && qblk < p.map_nblk) {
              const int c = cnt[(2 * qsub) * 2 * kMapFlush + hb + sl] +
                            cnt[(2 * qsub + 1) * 2 * kMapFlush + hb + sl];
              out_bh[static_cast<int64_t>(qblk) * p.map_nblk + j0 + sl] =
                  Fp16::from_float(static_cast<float>(c) * inv_area);
            }
          }
        } else {
          if (tid < kMapFlush / 2) {
            const int sl = tid;
            const int qblk = vrow_tile / 128;
            if (2 * sl + 1 <= slot_hi && qblk < p.map_nblk) {
              int c = 0;
#pragma unroll
              for (int w = 0; w < 4; ++w)
                c += cnt[w * 2 * kMapFlush + hb + 2 * sl] + cnt[w * 2 * kMapFlush + hb + 2 * sl + 1];
              out_bh[static_cast<int64_t>(qblk) * p.map_nblk + j0 / 2 + sl] =
                  Fp16::from_float(static_cast<float>(c) * inv_area);
            }
          }
        }
      }
    }
  }
}

// The pieces of a query tile -> its rows of O and LSE: with m the largest of the pieces'
// maxima, O = sum_i 2^(m_i - m) O_i / sum_i 2^(m_i - m) l_i, in fp32 and in piece order
// (deterministic). Bound by reading the partials back, mostly from L2 and the last-level
// cache. A workgroup takes kCombineRows rows of one tile, a thread four of its columns.
constexpr int kCombineRows = 16;

template <int D, typename E>
__global__ __launch_bounds__(kThreads) void combine_kernel(AttnParams p) {
  constexpr int kCols = D / 4;  // threads per row
  constexpr int kRowsPerPass = kThreads / kCols;
  const int tile = blockIdx.x / (kBM / kCombineRows);
  const int r_first = (blockIdx.x % (kBM / kCombineRows)) * kCombineRows;
  const int qt = tile % p.n_qtiles;
  const int bh = tile / p.n_qtiles;
  const int b = bh / p.heads;
  const int h = bh - b * p.heads;
  const int d = (threadIdx.x % kCols) * 4;
  for (int r = r_first + threadIdx.x / kCols; r < r_first + kCombineRows; r += kRowsPerPass) {
    const int q_row = p.origin + qt * kBM + r;
    if (q_row < 0 || q_row >= p.q_len) continue;
    const int64_t row0 = static_cast<int64_t>(tile) * p.n_split * kBM + r;
    float m = -FLT_MAX;  // the kernels' own start value
    for (int i = 0; i < p.n_split; ++i) m = fmaxf(m, p.part_ml[2 * (row0 + i * kBM)]);
    float l = 0.f;
    f32x4 o = f32x4{};
    for (int i = 0; i < p.n_split; ++i) {
      const int64_t row = row0 + i * kBM;
      const float w = __builtin_amdgcn_exp2f(p.part_ml[2 * row] - m);
      l += p.part_ml[2 * row + 1] * w;
      o += *reinterpret_cast<const f32x4*>(p.part_o + row * D + d) * w;
    }
    const float inv = l > 0.f ? 1.f / l : 0.f;
    u32x2 w2;
    w2.x = pack2(E::from_float(o[0] * inv), E::from_float(o[1] * inv));
    w2.y = pack2(E::from_float(o[2] * inv), E::from_float(o[3] * inv));
    *reinterpret_cast<u32x2*>(p.o + b * p.o_sb + h * p.o_sh + q_row * p.o_ss + d) = w2;
    if (p.lse != nullptr && d == 0)
      p.lse[static_cast<int64_t>(bh) * p.q_len + q_row] =
          l > 0.f ? (m + log2f(l)) * 0.69314718055994531f : -INFINITY;
  }
}

template <int D, typename E, bool kSparse, bool kRagged, bool kMap = false, bool kSplit = false>
int launch_attention_impl(const AttnParams& p, int batch, hipStream_t stream) {
  using L = AttnLds<D>;
  auto kernel = attention_fwd_kernel<D, E, kSparse, kRagged, kMap, kSplit>;
  constexpr int kLds = L::kTotal + (kMap ? kMapCountBytes : 0);
  static LaunchSetup once;
  if (set_dynamic_lds_once(once, reinterpret_cast<const void*>(kernel), kLds) != hipSuccess) {
    set_error("attention: cannot reserve %d bytes of LDS", kLds);
    return MODDIT_EHIP;
  }
  const int64_t tiles = static_cast<int64_t>(batch) * p.heads * p.n_qtiles;
  if (tiles == 0) return MODDIT_OK;
  const int64_t grid = kSplit ? tiles * p.n_split : tiles;
  if (grid > 0x7fffffff) {
    set_error("attention: too many tiles (%lld)", static_cast<long long>(tiles));
    return MODDIT_EINVAL;
  }
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kThreads), kLds, stream, p);
  MODDIT_CHECK_LAUNCH("attention");
  if constexpr (kSplit) {
    hipLaunchKernelGGL((combine_kernel<D, E>), dim3(static_cast<unsigned>(tiles * (kBM / kCombineRows))),
                       dim3(kThreads), 0, stream, p);
    MODDIT_CHECK_LAUNCH("attention (combine)");
  }
  return MODDIT_OK;
}

template <int D, typename E, bool kSparse>
int launch_attention(const AttnParams& p, int batch, hipStream_t stream) {
  // The fused map pass addresses video key tiles that may extend past the last key
  // (partial last block): always the range-checked path.
  if (p.map != nullptr) return launch_attention_impl<D, E, false, true, true>(p, batch, stream);
  // The split kernel exists in the range-checked form only (its masking is one scalar test
  // per key tile).
  if (p.n_split > 1) return launch_attention_impl<D, E, kSparse, true, false, true>(p, batch, stream);
  // Key counts that are a multiple of the tile (on an unshifted grid) need no clamping
  // or masking at all.
  if (p.kv_len % kBN == 0 && p.origin == 0)
    return launch_attention_impl<D, E, kSparse, false>(p, batch, stream);
  return launch_attention_impl<D, E, kSparse, true>(p, batch, stream);
}

// ---- how many pieces a query tile's key range is split into ----
// A launch of one workgroup per query tile leaves CUs idle when it has few tiles (a text
// tail, a short clip, few heads): its time is a whole key sweep however few they are. The
// sweep is then split over `n_split` workgroups per tile, at the price of writing and
// re-reading fp32 partial outputs and one more launch. The choice compares estimates of
// both, from the time a key tile takes with k workgroups on a CU (cu_tile_us: fitted to 166
// measured shapes of 1 to 512 query tiles by 16 to 512 key tiles, 1 to 32 pieces each). List
// lengths are known on the device only: a block-sparse list is taken to hold a quarter of its
// capacity. On those shapes the choice is never slower than no split, on average 3.5 % from
// the best of 1..32 pieces and at worst 25 % (sweeps of 16 key tiles, which are kept at two
// pieces): 256 text rows x 24 heads over 29,019 keys, D = 128 (48 tiles): 590 us unsplit,
// 135 in 10 pieces; over 115,419 keys 2,318 and 465 us; 4,096 tokens x 2 heads, D = 64 (64
// tiles): 66 and 29 us. Two tiles per CU no longer gain (432 tiles of 36 key tiles: 47 us
// unsplit, 59 us in two). A list that holds less than a twentieth of its capacity loses the
// second launch, 4 us (32 tiles of one entry, D = 64: 13.4 -> 17.5 us a call).
constexpr int kMaxSplit = 64;
// Key tiles per piece at the least: below 16 key tiles the second launch costs a dense call
// what the split saves. A list's estimate is rough: real lists
// hold a tenth to all of their capacity.
constexpr int kMinPieceDense = 8;
constexpr int kMinPieceSparse = 4;

double cu_tile_us(int head_dim, int64_t k) {
  constexpr double k128[4] = {1.33, 1.81, 3.14, 4.05}, k64[4] = {0.97, 1.17, 1.72, 2.19};
  if (head_dim == 128) return k <= 4 ? k128[k - 1] : k128[3] + 1.01 * (k - 4);
  return k <= 4 ? k64[k - 1] : k64[3] + 0.46 * (k - 4);
}

int split_for(int64_t tiles, int64_t key_tiles, int min_piece, int head_dim) {
  constexpr double kCus = 256, kFixedTiles = 2.5, kLaunchUs = 4.0, kPartialBytesPerUs = 4.0e6;
  int best = 1;
  double best_us = 0.0;
  for (int s = 1; s <= kMaxSplit; ++s) {
    if (s > 1 && key_tiles < static_cast<int64_t>(s) * min_piece) break;
    const int64_t per_cu = static_cast<int64_t>((tiles * s + kCus - 1) / kCus);
    double us = cu_tile_us(head_dim, per_cu) * (static_cast<double>(key_tiles) / s + kFixedTiles);
    if (s > 1) us += kLaunchUs + tiles * s * (kBM * (head_dim + 2) * 8.0) / kPartialBytesPerUs;
    if (s == 1 || us < 0.97 * best_us) {
      best = s;
      best_us = us;
    }
  }
  return best;
}

int64_t q_tiles_of(int q_len, int origin) { return (static_cast<int64_t>(q_len) - origin + kBM - 1) / kBM; }

int dense_split(int batch, int heads, int q_len, int kv_len, int head_dim) {
  return split_for(static_cast<int64_t>(batch) * heads * q_tiles_of(q_len, 0),
                   (static_cast<int64_t>(kv_len) + kBN - 1) / kBN, kMinPieceDense, head_dim);
}

int sparse_split(int batch, int heads, int q_len, int head_dim, int origin, int cap) {
  return split_for(static_cast<int64_t>(batch) * heads * q_tiles_of(q_len, origin), cap / 4,
                   kMinPieceSparse, head_dim);
}

int64_t split_workspace_bytes(int64_t tiles, int n_split, int head_dim) {
  return n_split > 1 ? tiles * n_split * kBM * (head_dim + 2) * static_cast<int64_t>(sizeof(float)) : 0;
}

struct SplitArgs {
  void* workspace;
  int64_t bytes;
};

struct MapArgs {
  void* out;
  int q_off;
  int video_blocks;
  int block;
  float log_thr;
};

int attention_entry(const void* q, const void* k, const void* v, void* o, float* lse, int batch,
                    int heads, int q_len, int kv_len, int head_dim, const int64_t* qs,
                    const int64_t* ks, const int64_t* vs, const int64_t* os, float scale,
                    int dtype, const int32_t* counts, const int32_t* entries, int n_qtiles,
                    int cap, int origin, moddit_stream_t stream, const MapArgs* map = nullptr,
                    const SplitArgs* split = nullptr) {
  clear_error();
  MODDIT_CHECK_ARG(q && k && v && o, "attention: null tensor pointer");
  MODDIT_CHECK_ARG(qs && ks && vs && os, "attention: null stride array");
  MODDIT_CHECK_ARG(scale > 0.f && std::isfinite(scale), "attention: softmax_scale must be positive");
  MODDIT_CHECK_ARG(batch >= 0 && heads >= 0 && q_len >= 0 && kv_len >= 0,
                   "attention: negative size");
  if (head_dim != 64 && head_dim != 128) {
    set_error("attention: head_dim must be 64 or 128, got %d", head_dim);
    return MODDIT_EUNSUPPORTED;
  }
  if (dtype != MODDIT_BF16 && dtype != MODDIT_FP16) {
    set_error("attention: dtype must be bf16 or fp16");
    return MODDIT_EUNSUPPORTED;
  }
  MODDIT_CHECK_ARG(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(o),
                   "attention: q/k/v/o must be 16-byte aligned");
  const int64_t* all[4] = {qs, ks, vs, os};
  for (int t = 0; t < 4; ++t)
    for (int j = 0; j < 3; ++j)
      MODDIT_CHECK_ARG(all[t][j] >= 0 && all[t][j] % 8 == 0,
                       "attention: strides must be non-negative multiples of 8 elements");
  // the fused map pass aligns the grid to 128-row tiles itself
  MODDIT_CHECK_ARG(origin > (map ? -kBM : -kBN) && origin <= 0,
                   "attention: grid_origin must be in (-64, 0], got %d", origin);
  const bool sparse = counts != nullptr;
  const int nq = (q_len - origin + kBM - 1) / kBM;
  if (sparse) {
    MODDIT_CHECK_ARG(entries != nullptr, "attention: tile entries missing");
    MODDIT_CHECK_ARG(n_qtiles == nq, "attention: n_qtiles=%d but q_len=%d (grid origin %d) needs %d",
                     n_qtiles, q_len, origin, nq);
    MODDIT_CHECK_ARG(cap > 0, "attention: cap must be positive");
  }
  if (q_len == 0 || batch == 0 || heads == 0) return MODDIT_OK;
  MODDIT_CHECK_ARG(kv_len > 0 || sparse, "attention: kv_len must be positive for dense attention");

  AttnParams p;
  p.q = static_cast<const uint16_t*>(q);
  p.k = static_cast<const uint16_t*>(k);
  p.v = static_cast<const uint16_t*>(v);
  p.o = static_cast<uint16_t*>(o);
  p.lse = lse;
  p.q_sb = qs[0]; p.q_sh = qs[1]; p.q_ss = qs[2];
  p.k_sb = ks[0]; p.k_sh = ks[1]; p.k_ss = ks[2];
  p.v_sb = vs[0]; p.v_sh = vs[1]; p.v_ss = vs[2];
  p.o_sb = os[0]; p.o_sh = os[1]; p.o_ss = os[2];
  p.heads = heads;
  p.q_len = q_len;
  p.kv_len = kv_len;
  p.origin = origin;
  p.n_qtiles = nq;
  p.n_ktiles = (kv_len - origin + kBN - 1) / kBN;
  p.xcd_run = xcd_run_for(static_cast<int64_t>(kv_len) * head_dim * 2 * 2);  // K and V
  p.scale_log2 = scale * 1.4426950408889634f;
  p.counts = counts;
  p.entries = entries;
  p.cap = cap;
  if (sparse && kv_len == 0) {
    set_error("attention: kv_len must be positive");
    return MODDIT_EINVAL;
  }
  // Per-head K/V spans are addressed with 32-bit buffer offsets; a whole 64-key tile past
  // the last row must also stay below 2^31.
  const int64_t k_span = (static_cast<int64_t>(kv_len) - 1) * ks[2] * 2 + head_dim * 2;
  const int64_t v_span = (static_cast<int64_t>(kv_len) - 1) * vs[2] * 2 + head_dim * 2;
  const int64_t max_off = (static_cast<int64_t>(p.n_ktiles) * kBN) * (ks[2] > vs[2] ? ks[2] : vs[2]) * 2;
  if (k_span > 0x7fffffffLL || v_span > 0x7fffffffLL || max_off > 0x7fffffffLL) {
    set_error("attention: one head's K/V span exceeds 2 GiB of 32-bit offsets");
    return MODDIT_EUNSUPPORTED;
  }
  p.k_bytes = static_cast<uint32_t>(k_span);
  p.v_bytes = static_cast<uint32_t>(v_span);
  p.map = nullptr;
  if (map != nullptr) {
    const int vt = map->video_blocks * map->block;
    p.map = static_cast<uint16_t*>(map->out);
    p.map_q_off = map->q_off;
    p.map_kt0 = (map->q_off - origin) / kBN;
    p.map_nblk = map->video_blocks;
    p.map_block = map->block;
    p.map_valid = vt < q_len - map->q_off ? vt : q_len - map->q_off;
    p.map_scale = scale;
    p.map_log_thr = map->log_thr;
    // largest byte offset a video key tile forms
    const int64_t map_off = (static_cast<int64_t>(map->q_off) - origin + vt) * ks[2] * 2;
    if (map_off > 0x7fffffffLL) {
      set_error("flash_fwd_map: one head's K span exceeds 2 GiB of 32-bit offsets");
      return MODDIT_EUNSUPPORTED;
    }
  }

  p.n_split = 1;
  if (split != nullptr && split->workspace != nullptr) {
    const int n_split = sparse ? sparse_split(batch, heads, q_len, head_dim, origin, cap)
                               : dense_split(batch, heads, q_len, kv_len, head_dim);
    const int64_t tiles = static_cast<int64_t>(batch) * heads * nq;
    const int64_t need = split_workspace_bytes(tiles, n_split, head_dim);
    MODDIT_CHECK_ARG(split->bytes >= need, "attention: workspace of %lld bytes, %lld needed",
                     static_cast<long long>(split->bytes), static_cast<long long>(need));
    MODDIT_CHECK_ARG(aligned16(split->workspace), "attention: workspace must be 16-byte aligned");
    if (n_split > 1) {
      p.n_split = n_split;
      p.part_o = static_cast<float*>(split->workspace);
      p.part_ml = p.part_o + tiles * n_split * kBM * head_dim;
    }
  }

  hipStream_t st = as_stream(stream);
  const bool bf = dtype == MODDIT_BF16;
  if (head_dim == 128) {
    if (bf) return sparse ? launch_attention<128, Bf16, true>(p, batch, st)
                          : launch_attention<128, Bf16, false>(p, batch, st);
    return sparse ? launch_attention<128, Fp16, true>(p, batch, st)
                  : launch_attention<128, Fp16, false>(p, batch, st);
  }
  if (bf) return sparse ? launch_attention<64, Bf16, true>(p, batch, st)
                        : launch_attention<64, Bf16, false>(p, batch, st);
  return sparse ? launch_attention<64, Fp16, true>(p, batch, st)
                : launch_attention<64, Fp16, false>(p, batch, st);
}

}  // namespace
}  // namespace moddit

extern "C" int moddit_flash_fwd(const void* q, const void* k, const void* v, void* o, float* lse,
                                int batch, int heads, int q_len, int kv_len, int head_dim,
                                const int64_t q_strides[3], const int64_t k_strides[3],
                                const int64_t v_strides[3], const int64_t o_strides[3],
                                float softmax_scale, int dtype, moddit_stream_t stream) {
  return moddit::attention_entry(q, k, v, o, lse, batch, heads, q_len, kv_len, head_dim,
                                 q_strides, k_strides, v_strides, o_strides, softmax_scale, dtype,
                                 nullptr, nullptr, 0, 0, 0, stream);
}

extern "C" int64_t moddit_flash_fwd_workspace_bytes(int batch, int heads, int q_len, int kv_len,
                                                    int head_dim) {
  using namespace moddit;
  if (batch <= 0 || heads <= 0 || q_len <= 0 || kv_len <= 0) return 0;
  return split_workspace_bytes(static_cast<int64_t>(batch) * heads * q_tiles_of(q_len, 0),
                               dense_split(batch, heads, q_len, kv_len, head_dim), head_dim);
}

extern "C" int moddit_flash_fwd_ws(const void* q, const void* k, const void* v, void* o, float* lse,
                                   int batch, int heads, int q_len, int kv_len, int head_dim,
                                   const int64_t q_strides[3], const int64_t k_strides[3],
                                   const int64_t v_strides[3], const int64_t o_strides[3],
                                   float softmax_scale, int dtype, void* workspace,
                                   int64_t workspace_bytes, moddit_stream_t stream) {
  const moddit::SplitArgs split{workspace, workspace_bytes};
  return moddit::attention_entry(q, k, v, o, lse, batch, heads, q_len, kv_len, head_dim,
                                 q_strides, k_strides, v_strides, o_strides, softmax_scale, dtype,
                                 nullptr, nullptr, 0, 0, 0, stream, nullptr, &split);
}

extern "C" int64_t moddit_block_sparse_fwd_workspace_bytes(int batch, int heads, int q_len,
                                                           int head_dim, int cap, int grid_origin) {
  using namespace moddit;
  if (batch <= 0 || heads <= 0 || q_len <= 0 || cap <= 0 || grid_origin > 0 || grid_origin <= -kBN)
    return 0;
  return split_workspace_bytes(static_cast<int64_t>(batch) * heads * q_tiles_of(q_len, grid_origin),
                               sparse_split(batch, heads, q_len, head_dim, grid_origin, cap), head_dim);
}

extern "C" int moddit_block_sparse_fwd_ws(const void* q, const void* k, const void* v, void* o,
                                          float* lse, int batch, int heads, int q_len, int kv_len,
                                          int head_dim, const int64_t q_strides[3],
                                          const int64_t k_strides[3], const int64_t v_strides[3],
                                          const int64_t o_strides[3], float softmax_scale,
                                          int dtype, const int32_t* counts, const int32_t* entries,
                                          int n_qtiles, int cap, int grid_origin, void* workspace,
                                          int64_t workspace_bytes, moddit_stream_t stream) {
  if (counts == nullptr) {
    moddit::set_error("block_sparse_fwd: counts must not be NULL");
    return MODDIT_EINVAL;
  }
  const moddit::SplitArgs split{workspace, workspace_bytes};
  return moddit::attention_entry(q, k, v, o, lse, batch, heads, q_len, kv_len, head_dim,
                                 q_strides, k_strides, v_strides, o_strides, softmax_scale, dtype,
                                 counts, entries, n_qtiles, cap, grid_origin, stream, nullptr, &split);
}

extern "C" int moddit_flash_fwd_map(const void* q, const void* k, const void* v, void* o,
                                    float* lse, void* map_out, int batch, int heads, int seq_len,
                                    int head_dim, const int64_t q_strides[3],
                                    const int64_t k_strides[3], const int64_t v_strides[3],
                                    const int64_t o_strides[3], float softmax_scale,
                                    float log_threshold, int video_offset, int video_blocks,
                                    int block_size, int dtype, moddit_stream_t stream) {
  using namespace moddit;
  clear_error();
  MODDIT_CHECK_ARG(map_out != nullptr, "flash_fwd_map: map_out must not be NULL");
  MODDIT_CHECK_ARG(block_size == 64 || block_size == 128,
                   "flash_fwd_map: block_size must be 64 or 128, got %d", block_size);
  MODDIT_CHECK_ARG(video_blocks > 0, "flash_fwd_map: video_blocks must be positive");
  MODDIT_CHECK_ARG(video_offset >= 0, "flash_fwd_map: video offset must be non-negative");
  // the last block may be partial, but must hold at least one token
  MODDIT_CHECK_ARG(static_cast<int64_t>(video_offset) + static_cast<int64_t>(video_blocks - 1) * block_size < seq_len,
                   "flash_fwd_map: video region exceeds sequence length");
  MODDIT_CHECK_ARG(!std::isnan(log_threshold), "flash_fwd_map: NaN threshold");
  // grid shifted so that video row 0 starts a 128-row tile
  const int origin = video_offset - ((video_offset + kBM - 1) / kBM) * kBM;
  MapArgs m{map_out, video_offset, video_blocks, block_size, log_threshold};
  return attention_entry(q, k, v, o, lse, batch, heads, seq_len, seq_len, head_dim, q_strides,
                         k_strides, v_strides, o_strides, softmax_scale, dtype, nullptr, nullptr,
                         0, 0, origin, stream, &m);
}

extern "C" int moddit_block_sparse_fwd(const void* q, const void* k, const void* v, void* o,
                                       float* lse, int batch, int heads, int q_len, int kv_len,
                                       int head_dim, const int64_t q_strides[3],
                                       const int64_t k_strides[3], const int64_t v_strides[3],
                                       const int64_t o_strides[3], float softmax_scale, int dtype,
                                       const int32_t* counts, const int32_t* entries,
                                       int n_qtiles, int cap, int grid_origin,
                                       moddit_stream_t stream) {
  if (counts == nullptr) {
    moddit::set_error("block_sparse_fwd: counts must not be NULL");
    return MODDIT_EINVAL;
  }
  return moddit::attention_entry(q, k, v, o, lse, batch, heads, q_len, kv_len, head_dim,
                                 q_strides, k_strides, v_strides, o_strides, softmax_scale, dtype,
                                 counts, entries, n_qtiles, cap, grid_origin, stream);
}
