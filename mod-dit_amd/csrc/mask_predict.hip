// Mask prediction for gfx950: M^T S line statistics, line prediction/selection,
// block-diagonal mode, block mask + attention tile lists, and the refresh merge (the
// ridge solve between M^T S and the selection is in fit.hip). All of it is HBM-bound
// integer/byte work; none of it is reshaped onto MFMA.
//
// Floating-point contraction is disabled in this file: the prediction
// cur + (cur - last) / T must round exactly like the reference's separate fp32 ops.
#pragma clang fp contract(off)

#include "common.h"

namespace moddit {
namespace {

// =====================================================================================
// M^T S (MoD/mod/cuda_lstsq_kernel.cu:17-162, 421-482; torch twin cuda_lstsq.py:91-139)
// =====================================================================================
//
// fp32 maps: three workgroup roles over one launch, all reading the map with 128-byte
// rows per wave:
//   diagonal bands  : 64 diagonals per workgroup, lane = diagonal, waves stride rows
//   column strips   : 64 columns per workgroup, lane = column, waves stride rows
//   frame blocks    : one workgroup per head sums the n/bpf diagonal bpf x bpf blocks
// Sums accumulate in fp64 and are rounded once (deterministic: fixed order).

constexpr int kMtsThreads = 256;

struct MtsParams {
  const float* map;
  int heads;
  int n;
  int bpf;
  int n_bands;   // ceil((2n-1)/64)
  int n_strips;  // ceil(n/64)
  float* out;    // (H, 3n)
};

__global__ __launch_bounds__(kMtsThreads) void mts_kernel(MtsParams p) {
  __shared__ double s_wide[kMtsThreads];

  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int n = p.n;
  const int nd = 2 * n - 1;
  const int F = 3 * n;

  int role_id = blockIdx.x;
  double acc = 0.0;

  if (role_id < p.heads * p.n_bands) {
    // ---- diagonal band ----
    const int h = role_id / p.n_bands;
    const int band = role_id % p.n_bands;
    const int dk = band * 64 + lane;  // diagonal index, offset = dk - (n-1)
    const int off = dk - (n - 1);
    const int off_lo = band * 64 - (n - 1);
    const int off_hi = band * 64 + 63 - (n - 1);
    const int r_lo = off_hi < 0 ? -off_hi : 0;
    const int r_hi = off_lo > 0 ? n - off_lo : n;
    const int64_t base = static_cast<int64_t>(h) * n * n;
    if (dk < nd) {
#pragma unroll 4
      for (int r = r_lo + wave; r < r_hi; r += 4) {
        const int c = r + off;
        if (c >= 0 && c < n) acc += static_cast<double>(p.map[base + static_cast<int64_t>(r) * n + c]);
      }
    }
    s_wide[tid] = acc;
    __syncthreads();
    if (wave == 0 && dk < nd) {
      for (int w = 1; w < 4; ++w) acc += s_wide[w * 64 + lane];
      p.out[static_cast<int64_t>(h) * F + dk] = static_cast<float>(acc);
    }
    return;
  }
  role_id -= p.heads * p.n_bands;

  if (role_id < p.heads * p.n_strips) {
    // ---- column strip ----
    const int h = role_id / p.n_strips;
    const int strip = role_id % p.n_strips;
    const int c = strip * 64 + lane;
    const int64_t base = static_cast<int64_t>(h) * n * n;
    if (c < n) {
#pragma unroll 4
      for (int r = wave; r < n; r += 4) acc += static_cast<double>(p.map[base + static_cast<int64_t>(r) * n + c]);
    }
    s_wide[tid] = acc;
    __syncthreads();
    if (wave == 0 && c < n) {
      for (int w = 1; w < 4; ++w) acc += s_wide[w * 64 + lane];
      p.out[static_cast<int64_t>(h) * F + nd + c] = static_cast<float>(acc);
    }
    return;
  }
  role_id -= p.heads * p.n_strips;

  // ---- frame-diagonal blocks ----
  const int h = role_id;
  const int bpf = p.bpf;
  const int nb = n / bpf;
  const int per = bpf * bpf;
  const int64_t total = static_cast<int64_t>(nb) * per;
  const int64_t base = static_cast<int64_t>(h) * n * n;
  for (int64_t idx = tid; idx < total; idx += kMtsThreads) {
    const int f = static_cast<int>(idx / per);
    const int rem = static_cast<int>(idx % per);
    const int i = rem / bpf;
    const int j = rem % bpf;
    acc += static_cast<double>(p.map[base + static_cast<int64_t>(f * bpf + i) * n + (f * bpf + j)]);
  }
  s_wide[tid] = acc;
  __syncthreads();
  for (int s = kMtsThreads / 2; s > 0; s >>= 1) {
    if (tid < s) s_wide[tid] += s_wide[tid + s];
    __syncthreads();
  }
  if (tid == 0) p.out[static_cast<int64_t>(h) * F + F - 1] = static_cast<float>(s_wide[0]);
}

// -------------------------------------------------------------------------------------
// Single pass over an fp16 map (the product path): mts_tile_kernel reads every cell once and
// leaves one record of partial sums per tile, mts_sum_kernel adds the records of each line.
//
// A tile is 512 columns x 4R rows; each of the workgroup's four waves owns R rows, a lane 8
// consecutive columns. Column sums stay in the lane. A diagonal moves one column to the
// right per row, so the lane's 8 diagonal sums do too: their registers are renamed (the row
// loop is unrolled by 8), the one that crosses to the next lane moves by a wave shift, and
// the one that leaves the last lane is stored to LDS. Nothing is reduced across lanes, and
// no atomic is used: with 23 LDS atomics per 8 x 16 cells and global atomics per tile, which
// this replaced, both launches took 60 us at n = 1800 x 24 (155.5 MB) and, where rows are not
// 16-byte aligned, 67 us at n = 275 x 48 (7 MB); 51 (3.0 TB/s) and 13.5 us now. It issues 41
// VALU instructions per row of 64 x 8 cells, half of them fp64, on four waves per SIMD (112
// VGPRs); a second register stage of loads gains nothing. Loads that would pass the map's end
// are moved back and shifted (edge_row); read cell by cell, as the last rows of a map and all
// of a small one were at first, 16 x 16 blocks x 24 heads took 23.7 us (15.2 with the atomics,
// 12.3 now).
//
// Exactness: every finite fp16 value is a multiple of 2^-24 below 2^16, so any sum of at
// most 8192 of them needs at most 53 significant bits and is exact in fp64 in any order; a
// tile's share of one line is at most 4R <= 256 cells. The records are then added as int64
// in units of 2^-24 and rounded once to fp32: every output is the correctly rounded sum,
// whatever the tile shape. Records that are not finite (inf/NaN inputs) are added in float
// instead, in a fixed order (inf/NaN semantics only).
constexpr int kMtsTileThreads = 256;
constexpr int kMtsWaves = kMtsTileThreads / 64;
constexpr int kMtsCols = 8;                    // columns per lane
constexpr int kMtsTileC = 64 * kMtsCols;       // 512
// Rows per wave: 64, or 16 for maps too small to fill the GPU with the taller tiles.
constexpr int kMtsRowsTall = 64;
constexpr int kMtsRowsShort = 16;
constexpr int64_t kMtsFillTiles = 512;         // two workgroups per CU
// A map's line sums over c cells stay below 2^63 units of 2^-24 while c <= 2^23 (an fp16
// value is below 2^40 units). Diagonal and column outputs sum n cells; the frame-block
// output sums (n / bpf) * bpf^2 = n * min(bpf, n) cells, which the entry point bounds.
constexpr int kMts1MaxN = 1 << 20;
constexpr int64_t kMts1MaxFrameCells = int64_t{1} << 23;

// Record of a tile: its diagonals' sums (index kl = (c - C0) - (r - R0) + rows - 1), its
// columns' sums, the frame-block sum in int64 units and its non-finite part.
__host__ __device__ constexpr int mts_tile_diags(int rows) { return kMtsTileC + kMtsWaves * rows - 1; }
__host__ __device__ constexpr int mts_record_doubles(int rows) { return mts_tile_diags(rows) + kMtsTileC + 2; }

inline int mts_rows_for(int heads, int n) {
  const int64_t ct = (n + kMtsTileC - 1) / kMtsTileC;
  const int tall = kMtsWaves * kMtsRowsTall;
  return heads * ct * ((n + tall - 1) / tall) >= kMtsFillTiles ? kMtsRowsTall : kMtsRowsShort;
}

struct Mts1Params {
  const uint16_t* map;
  int heads;
  int n;
  int bpf;
  int n_rt;        // row tiles per head
  int n_ct;        // column tiles per head
  double* records; // [head][row tile][column tile][mts_record_doubles(rows)]
  float* out;      // (H, 3n)
};

// x of the previous lane (0 in lane 0)
__device__ __forceinline__ double wave_shift_up(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(u), 0x138, 0xf, 0xf, true);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(u >> 32), 0x138, 0xf, 0xf, true);
  return __builtin_bit_cast(double, static_cast<uint64_t>(lo) | (static_cast<uint64_t>(hi) << 32));
}

__device__ __forceinline__ double read_lane(double x, int lane) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(u), lane);
  const uint32_t hi = __builtin_amdgcn_readlane(static_cast<int>(u >> 32), lane);
  return __builtin_bit_cast(double, static_cast<uint64_t>(lo) | (static_cast<uint64_t>(hi) << 32));
}

template <int kRows>
__global__ __launch_bounds__(kMtsTileThreads, 3) void mts_tile_kernel(Mts1Params p) {
  constexpr int kWaveDiag = kMtsTileC + kRows - 1;
  constexpr int kTileDiag = mts_tile_diags(kRows);
  __shared__ double s_diag[kMtsWaves][kWaveDiag];
  __shared__ double s_col[kMtsWaves][kMtsTileC];
  __shared__ long long s_frame[kMtsWaves];
  __shared__ double s_special[kMtsWaves];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  // wave-uniform, so that the row tests and addresses below are scalar
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = p.n;
  const int tiles = p.n_rt * p.n_ct;
  const int h = blockIdx.x / tiles;
  const int t = blockIdx.x - h * tiles;
  const int R0 = (t / p.n_ct) * (kMtsWaves * kRows);
  const int C0 = (t % p.n_ct) * kMtsTileC;
  const int rs = R0 + wave * kRows;        // this wave's first row
  const int c0 = C0 + lane * kMtsCols;     // this lane's first column
  const int64_t cells = static_cast<int64_t>(p.heads) * n * n;
  const int64_t head0 = static_cast<int64_t>(h) * n * n;
  const int frame_end = (n / p.bpf) * p.bpf;
  // columns past the row's end are loaded with the next row's cells and cleared
  u32x4 keep;
#pragma unroll
  for (int w = 0; w < 4; ++w)
    keep[w] = (c0 + 2 * w < n ? 0xffffu : 0u) | (c0 + 2 * w + 1 < n ? 0xffff0000u : 0u);

  double cacc[kMtsCols], dacc[kMtsCols];
#pragma unroll
  for (int j = 0; j < kMtsCols; ++j) cacc[j] = dacc[j] = 0.0;
  double fsum = 0.0;
  double leaving = 0.0;  // lane i: the diagonal that left the last lane after row i
  // the cells of one row, with the lane's diagonal of column j in register (j - rr) & 7
  auto add_row = [&](u32x4 w, int rr) {
#pragma unroll
    for (int j = 0; j < kMtsCols; ++j) {
      const double x = static_cast<double>(Fp16::to_float(u16_at(w, j)));
      cacc[j] += x;
      dacc[(j - rr) & 7] += x;
    }
  };
  // its frame-block cells, if the row's frame meets the tile's columns
  auto add_frame = [&](u32x4 w, int r) {
    const int f0 = r < frame_end ? r / p.bpf * p.bpf : n;
    if (f0 < C0 + kMtsTileC && f0 + p.bpf > C0) {
#pragma unroll
      for (int j = 0; j < kMtsCols; ++j)
        if (static_cast<unsigned>(c0 + j - f0) < static_cast<unsigned>(p.bpf))
          fsum += static_cast<double>(Fp16::to_float(u16_at(w, j)));
    }
  };
  // one row down, the diagonals are one column further: the sum at column 7 goes to the next
  // lane, the last lane's is complete
  auto step_down = [&](double& edge, int row) {
    const double out = read_lane(edge, 63);
    leaving = lane == row ? out : leaving;
    edge = wave_shift_up(edge);
  };
  // the lane's cells of a row near the map's end or past it (zeros): the 16 bytes that end with
  // the map instead of those past its end, shifted into place
  auto edge_row = [&](int r) -> u32x4 {
    u32x4 w = u32x4{};
    if (r >= n) return w;
    const int64_t at = head0 + static_cast<int64_t>(r) * n + (c0 < n ? c0 : 0);
    if (cells >= kMtsCols) {
      const int64_t from = at < cells - kMtsCols ? at : cells - kMtsCols;
      const int drop = static_cast<int>(at - from);  // 0..7 cells
      __builtin_memcpy(&w, p.map + from, 16);
#pragma unroll
      for (int b = 1; b < kMtsCols; b *= 2)  // right by 1, 2, 4 cells
        if (drop & b) {
          const uint64_t lo = w[0] | static_cast<uint64_t>(w[1]) << 32;
          const uint64_t hi = w[2] | static_cast<uint64_t>(w[3]) << 32;
          const uint64_t l = b == 4 ? hi : lo >> (16 * b) | hi << (64 - 16 * b);
          const uint64_t h2 = b == 4 ? 0 : hi >> (16 * b);
          w = u32x4{static_cast<uint32_t>(l), static_cast<uint32_t>(l >> 32),
                    static_cast<uint32_t>(h2), static_cast<uint32_t>(h2 >> 32)};
        }
    } else {  // fewer cells than a load holds
      for (int j = 0; j < kMtsCols; ++j)
        if (at + j < cells) w[j >> 1] |= static_cast<uint32_t>(p.map[at + j]) << (16 * (j & 1));
    }
    return w;
  };
#pragma unroll 1
  for (int r8 = 0; r8 < kRows; r8 += 8) {
    const int r = rs + r8;
    u32x4 raw[8];
    if (r + 8 <= n && head0 + static_cast<int64_t>(r + 7) * n + C0 + kMtsTileC <= cells) {
      // eight whole rows, 16 bytes per lane at any 2-byte address
      const uint16_t* src = p.map + head0 + static_cast<int64_t>(r) * n + (c0 < n ? c0 : C0);
#pragma unroll
      for (int rr = 0; rr < 8; ++rr) __builtin_memcpy(&raw[rr], src + static_cast<int64_t>(rr) * n, 16);
    } else {
#pragma unroll
      for (int rr = 0; rr < 8; ++rr) raw[rr] = edge_row(r + rr);
    }
#pragma unroll
    for (int rr = 0; rr < 8; ++rr) {
      raw[rr] &= keep;
      add_row(raw[rr], rr);
      step_down(dacc[(7 - rr) & 7], r8 + rr);
      __builtin_amdgcn_sched_barrier(0);  // or all 64 cells are converted first, and spill
    }
    // The frame cells apart from the sums above, which stay free of branches. The empty asm
    // keeps the compiler from moving the sums below these branches, and from carrying the
    // 64 converted cells across them: either spills.
#pragma unroll
    for (int j = 0; j < kMtsCols; ++j) asm volatile("" : "+v"(cacc[j]), "+v"(dacc[j]));
#pragma unroll
    for (int rr = 0; rr < 8; ++rr) {
      asm volatile("" : "+v"(raw[rr]));
      add_frame(raw[rr], r + rr);
    }
  }
  // after the last row's shift, register j of lane l holds the diagonal of column 8l + j - 1
#pragma unroll
  for (int j = 0; j < kMtsCols; ++j) {
    const int kl = lane * kMtsCols + j - 1;
    if (kl >= 0) s_diag[wave][kl] = dacc[j];
    s_col[wave][lane * kMtsCols + j] = cacc[j];
  }
  if (lane < kRows) s_diag[wave][kWaveDiag - 1 - lane] = leaving;
  // frame-block partial: each lane's sum (at most 512 cells) is exact in fp64 and converts
  // exactly to int64 units
  long long fq = 0;
  double special = 0.0;
  if (__builtin_isfinite(fsum))
    fq = static_cast<long long>(fsum * 0x1p24);
  else
    special = fsum;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    fq += __shfl_xor(fq, o);
    special += __shfl_xor(special, o);
  }
  if (lane == 0) {
    s_frame[wave] = fq;
    s_special[wave] = special;
  }
  __syncthreads();

  double* rec = p.records + static_cast<int64_t>(blockIdx.x) * mts_record_doubles(kRows);
  // wave w's index is kl minus the rows below it in the tile
  for (int kl = tid; kl < kTileDiag; kl += kMtsTileThreads) {
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < kMtsWaves; ++w) {
      const int i = kl - (kMtsWaves - 1 - w) * kRows;
      if (i >= 0 && i < kWaveDiag) sum += s_diag[w][i];
    }
    rec[kl] = sum;
  }
  for (int c = tid; c < kMtsTileC; c += kMtsTileThreads)
    rec[kTileDiag + c] = (s_col[0][c] + s_col[1][c]) + (s_col[2][c] + s_col[3][c]);
  if (tid == 0) {
    rec[kTileDiag + kMtsTileC] =
        __builtin_bit_cast(double, (s_frame[0] + s_frame[1]) + (s_frame[2] + s_frame[3]));
    rec[kTileDiag + kMtsTileC + 1] = (s_special[0] + s_special[1]) + (s_special[2] + s_special[3]);
  }
}

// Exact sum of finite fp64 partials (multiples of 2^-24); non-finite ones apart, in float.
struct MtsSum {
  long long q = 0;
  float special = 0.f;
  __device__ __forceinline__ void add(double x) {
    if (__builtin_isfinite(x))
      q += static_cast<long long>(x * 0x1p24);
    else
      special += static_cast<float>(x);
  }
  __device__ __forceinline__ float result() const {
    return (special != 0.f || special != special) ? special : static_cast<float>(q) * 0x1p-24f;
  }
};

// One thread per diagonal and column output, one wave per head's frame-block output.
template <int kRows>
__global__ __launch_bounds__(kMtsTileThreads) void mts_sum_kernel(Mts1Params p) {
  constexpr int kTileR = kMtsWaves * kRows;
  constexpr int kTileDiag = mts_tile_diags(kRows);
  constexpr int kRec = mts_record_doubles(kRows);
  const int n = p.n;
  const int nd = 2 * n - 1;
  const int64_t F = 3 * static_cast<int64_t>(n);
  const int groups = static_cast<int>((F - 1 + kMtsTileThreads - 1) / kMtsTileThreads) + 1;
  const int h = blockIdx.x / groups;
  const int g = blockIdx.x - h * groups;
  const double* rec = p.records + static_cast<int64_t>(h) * p.n_rt * p.n_ct * kRec;
  float* out = p.out + static_cast<int64_t>(h) * F;
  if (g == groups - 1) {  // frame blocks: lanes stride the tiles
    if (threadIdx.x >= 64) return;
    long long q = 0;
    double special = 0.0;
    for (int64_t t = threadIdx.x; t < static_cast<int64_t>(p.n_rt) * p.n_ct; t += 64) {
      q += __builtin_bit_cast(long long, rec[t * kRec + kTileDiag + kMtsTileC]);
      special += rec[t * kRec + kTileDiag + kMtsTileC + 1];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      q += __shfl_xor(q, o);
      special += __shfl_xor(special, o);
    }
    if (threadIdx.x == 0) {
      MtsSum sum;
      sum.q = q;
      sum.special = static_cast<float>(special);
      out[F - 1] = sum.result();
    }
    return;
  }
  const int64_t i = static_cast<int64_t>(g) * kMtsTileThreads + threadIdx.x;
  if (i >= F - 1) return;
  MtsSum sum;
  if (i < nd) {
    // diagonal offset c - r = off crosses row tile rt at columns [R0 + off, R0 + off + kTileR)
    const int off = static_cast<int>(i) - (n - 1);
    for (int rt = 0; rt < p.n_rt; ++rt) {
      const int first = rt * kTileR + off;
      const int last = first + kTileR - 1;
      if (last < 0 || first >= n) continue;
      const int ct0 = (first < 0 ? 0 : first) / kMtsTileC;
      const int ct1 = (last < n ? last : n - 1) / kMtsTileC;
      for (int ct = ct0; ct <= ct1; ++ct)
        sum.add(rec[(static_cast<int64_t>(rt) * p.n_ct + ct) * kRec + first - ct * kMtsTileC + kTileR - 1]);
    }
  } else {
    const int c = static_cast<int>(i) - nd;
    for (int rt = 0; rt < p.n_rt; ++rt)
      sum.add(rec[(static_cast<int64_t>(rt) * p.n_ct + c / kMtsTileC) * kRec + kTileDiag + c % kMtsTileC]);
  }
  out[i] = sum.result();
}

template <int kRows>
int launch_mts_fp16(Mts1Params& q, hipStream_t st) {
  q.n_rt = (q.n + kMtsWaves * kRows - 1) / (kMtsWaves * kRows);
  q.n_ct = (q.n + kMtsTileC - 1) / kMtsTileC;
  const int64_t grid = static_cast<int64_t>(q.heads) * q.n_rt * q.n_ct;
  const int64_t sums = static_cast<int64_t>(q.heads) *
                       ((3 * static_cast<int64_t>(q.n) - 1 + kMtsTileThreads - 1) / kMtsTileThreads + 1);
  MODDIT_CHECK_ARG(grid < 0x7fffffff && sums < 0x7fffffff, "mts: shape too large");
  hipLaunchKernelGGL((mts_tile_kernel<kRows>), dim3(static_cast<unsigned>(grid)),
                     dim3(kMtsTileThreads), 0, st, q);
  MODDIT_CHECK_LAUNCH("mts");
  hipLaunchKernelGGL((mts_sum_kernel<kRows>), dim3(static_cast<unsigned>(sums)),
                     dim3(kMtsTileThreads), 0, st, q);
  MODDIT_CHECK_LAUNCH("mts (sum)");
  return MODDIT_OK;
}

// =====================================================================================
// Line prediction + k-smallest selection (MoD/mod/attn_mask.py:351-370)
// =====================================================================================
//
// One workgroup per head. Keys are (ordered(pred) << 14 | index) — unique, so the k-th
// smallest key is found exactly by a 6-pass 8-bit radix select (48 bits), and the k
// selected indices are compacted in ascending index order.

constexpr int kSelThreads = 1024;
constexpr int kSelMaxItems = 16384;  // 3n-1 <= 16384
constexpr int kIdxBits = 14;

__device__ __forceinline__ uint32_t ordered_bits(float v) {
  uint32_t u = __float_as_uint(v);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0xffffffffu;  // NaN orders last
  if (u == 0x80000000u) u = 0;                              // -0 == +0
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ int block_exclusive_scan(int v, int* s_wave, int* total) {
  // 1024 threads = 16 wave64s.
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(incl, o);
    if (lane >= o) incl += t;
  }
  if (lane == 63) s_wave[wave] = incl;
  __syncthreads();
  if (wave == 0) {
    int w = lane < 16 ? s_wave[lane] : 0;
    int wincl = w;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      const int t = __shfl_up(wincl, o);
      if (lane >= o) wincl += t;
    }
    if (lane < 16) s_wave[lane] = wincl - w;  // exclusive per wave
    if (lane == 15) s_wave[16] = wincl;
  }
  __syncthreads();
  const int res = s_wave[wave] + incl - v;
  *total = s_wave[16];
  __syncthreads();
  return res;
}

__global__ __launch_bounds__(kSelThreads) void select_kernel(const float* __restrict__ x_cur,
                                                             const float* __restrict__ x_last,
                                                             int n, float inv_T_unused, int T,
                                                             int k, int32_t* __restrict__ sel) {
  extern __shared__ __align__(16) unsigned char sel_smem[];
  unsigned long long* keys = reinterpret_cast<unsigned long long*>(sel_smem);
  __shared__ int hist[256];
  __shared__ int s_wave[17];
  __shared__ unsigned long long s_prefix;
  __shared__ int s_kk;

  const int h = blockIdx.x;
  const int tid = threadIdx.x;
  const int F = 3 * n;
  const int items = 3 * n - 1;
  const int nd = 2 * n - 1;
  const float Tf = static_cast<float>(T);
  const float* xc = x_cur + static_cast<int64_t>(h) * F;
  const float* xl = x_last + static_cast<int64_t>(h) * F;

  for (int i = tid; i < items; i += kSelThreads) {
    float cur, last;
    if (i < n) {  // column line i: c = X[:, 2n-1+i] / 2
      cur = xc[nd + i] / 2.0f;
      last = xl[nd + i] / 2.0f;
    } else {  // diagonal line i-n: d = X[:, i-n]
      cur = xc[i - n];
      last = xl[i - n];
    }
    const float step = (cur - last) / Tf;
    const float pred = cur + step;
    keys[i] = (static_cast<unsigned long long>(ordered_bits(pred)) << kIdxBits) |
              static_cast<unsigned long long>(i);
  }
  if (tid == 0) {
    s_prefix = 0ull;
    s_kk = k;
  }
  __syncthreads();

  unsigned long long mask_hi = 0ull;
  for (int shift = 40; shift >= 0; shift -= 8) {
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    const unsigned long long prefix = s_prefix;
    for (int i = tid; i < items; i += kSelThreads) {
      const unsigned long long key = keys[i];
      if ((key & mask_hi) == prefix) atomicAdd(&hist[(key >> shift) & 255u], 1);
    }
    __syncthreads();
    if (tid < 64) {
      const int h0 = hist[4 * tid], h1 = hist[4 * tid + 1], h2 = hist[4 * tid + 2],
                h3 = hist[4 * tid + 3];
      const int local = h0 + h1 + h2 + h3;
      int incl = local;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(incl, o);
        if (tid >= o) incl += t;
      }
      const int excl = incl - local;
      const int kk = s_kk;
      if (excl < kk && kk <= incl) {
        int before = excl;
        int digit = 4 * tid;
        if (kk > before + h0) {
          before += h0;
          digit++;
          if (kk > before + h1) {
            before += h1;
            digit++;
            if (kk > before + h2) {
              before += h2;
              digit++;
            }
          }
        }
        s_prefix = prefix | (static_cast<unsigned long long>(digit) << shift);
        s_kk = kk - before;
      }
    }
    mask_hi |= 255ull << shift;
    __syncthreads();
  }
  const unsigned long long kth = s_prefix;

  // Ordered compaction of {key <= kth} by index.
  const int chunk = (items + kSelThreads - 1) / kSelThreads;
  const int i0 = tid * chunk;
  int cnt = 0;
  for (int i = i0; i < i0 + chunk && i < items; ++i) cnt += keys[i] <= kth ? 1 : 0;
  int total = 0;
  int pos = block_exclusive_scan(cnt, s_wave, &total);
  int32_t* out = sel + static_cast<int64_t>(h) * k;
  for (int i = i0; i < i0 + chunk && i < items; ++i) {
    if (keys[i] <= kth) {
      if (pos < k) out[pos] = i;
      ++pos;
    }
  }
}

__global__ void check_bd_kernel(const float* __restrict__ x, int heads, int F, float thr,
                                uint8_t* __restrict__ mode) {
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  if (h < heads && mode[h] == MODDIT_MODE_SPARSE) {
    if (x[static_cast<int64_t>(h) * F + F - 1] <= thr) mode[h] = MODDIT_MODE_BLOCK_DIAGONAL;
  }
}

// =====================================================================================
// Block mask + attention tile lists (MoD/mod/attn_mask.py:440-559, 296-311)
// =====================================================================================
//
// One wave per (head, 128-row query tile): a lane owns 8 consecutive mask columns per pass
// of 512, so a tile needs neither LDS nor a barrier to place its entries in ascending order
// (one scan of the lanes' counts per pass), and narrow masks keep as many waves busy as wide
// ones. Workgroups of 256 columns x 8 rows that stepped through eight tiles together, which
// this replaced, left 220 of 256 threads idle at 279 columns: 38 us there (48 heads), 24 us
// at 225 x 24 heads, and 44 us for the mask alone at 1,800 x 24 (78 MB), against 19.5, 9.5
// and 22 us (3.5 TB/s of mask bytes) now.

constexpr int kMaskThreads = 256;  // four waves
constexpr int kMaskWaves = kMaskThreads / 64;
constexpr int kMaskCols = 8;       // columns per lane and pass
constexpr int kMaskPass = 64 * kMaskCols;

// Appends the entries (key_tile << 2 | row bits) of one pass's active columns (bit c of
// m0 / m1: column j0 + c is active in the tile's first / second row) to the list, which
// holds `written` entries so far; returns the new length. Key tiles from kv_tiles on are
// dropped, entries past `cap` counted but not stored. All lanes of the wave take part.
__device__ __forceinline__ int emit_tiles(unsigned m0, unsigned m1, int j0, int lane, int per_col,
                                          bool both, int kv_tiles, int32_t* out, int cap,
                                          int written) {
  unsigned any = m0 | m1;
  // columns wholly below the key-tile limit, and one that it may cut in half
  const int left = kv_tiles - j0 * per_col;  // key tiles from this lane's first column on
  const int whole = left <= 0 ? 0 : (left / per_col < kMaskCols ? left / per_col : kMaskCols);
  const int part = whole < kMaskCols && left > 0 ? left - whole * per_col : 0;
  any &= (1u << (whole + (part > 0 ? 1 : 0))) - 1u;
  const int cut = part > 0 && ((any >> whole) & 1u) ? per_col - part : 0;
  const int cnt = __builtin_popcount(any) * per_col - cut;
  int incl = cnt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(incl, o);
    if (lane >= o) incl += v;
  }
  int pos = written + incl - cnt;
  while (any != 0u) {
    const int c = __builtin_ctz(any);
    any &= any - 1u;
    const int bits = both ? 3 : static_cast<int>(((m0 >> c) & 1u) | (((m1 >> c) & 1u) << 1));
    const int kt = (j0 + c) * per_col;
    if (pos < cap) out[pos] = (kt << 2) | bits;
    ++pos;
    if (per_col == 2 && kt + 1 < kv_tiles) {
      if (pos < cap) out[pos] = ((kt + 1) << 2) | bits;
      ++pos;
    }
  }
  return written + __builtin_amdgcn_readlane(incl, 63);
}

// bit c of the result = byte c (0 or 1) of v; no partial product carries into the top byte
__device__ __forceinline__ unsigned byte_bits(uint64_t v) {
  return static_cast<unsigned>((v * 0x0102040810204080ull) >> 56);
}

struct MaskParams {
  const int32_t* sel;      // (H, k)
  int k;
  const uint8_t* mode;     // (H)
  int n;                   // video blocks per side
  int bpf;
  int layout;
  int nb;                  // mask blocks per side
  int text_blocks;
  int block;               // 64 or 128
  int union_rows;
  uint8_t* mask_out;       // (H, nb, nb) or null
  int32_t* counts;         // (H, n_qtiles) or null
  int32_t* entries;        // (H, n_qtiles, cap) or null
  int n_qtiles;
  int cap;
};

// LDS of the line-based mask kernel: the selected columns and diagonals as bytes, each at an
// 8-byte aligned offset plus zero padding for the unaligned 8-byte windows.
__host__ __device__ inline int mask_diag_offset(int n) { return (n + 7) & ~7; }
__host__ __device__ inline int mask_lds_bytes(int n) {
  return mask_diag_offset(n) + ((2 * n - 1 + 7) & ~7) + 8;
}

// Tiles per workgroup: the selected-line byte maps are built in LDS once per workgroup
// and serve this many consecutive query tiles of the head.
constexpr int kMaskTilesPerWg = 8;

__global__ __launch_bounds__(kMaskThreads) void mask_tiles_kernel(MaskParams p) {
  extern __shared__ __align__(16) unsigned char mk_smem[];
  uint8_t* colsel = mk_smem;                          // n bytes
  uint8_t* diagsel = mk_smem + mask_diag_offset(p.n);  // 2n-1 bytes
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wg_per_head = (p.n_qtiles + kMaskTilesPerWg - 1) / kMaskTilesPerWg;
  const int h = blockIdx.x / wg_per_head;
  const int t_begin = (blockIdx.x % wg_per_head) * kMaskTilesPerWg;
  const int t_end = t_begin + kMaskTilesPerWg < p.n_qtiles ? t_begin + kMaskTilesPerWg : p.n_qtiles;
  const int n = p.n;
  const int nb = p.nb;
  const int mode = p.mode ? p.mode[h] : MODDIT_MODE_SPARSE;

  for (int i = tid; i < mask_lds_bytes(n) / 8; i += kMaskThreads)
    reinterpret_cast<uint64_t*>(mk_smem)[i] = 0;
  __syncthreads();
  const int32_t* s = p.sel + static_cast<int64_t>(h) * p.k;
  for (int i = tid; i < p.k; i += kMaskThreads) {
    const int idx = s[i];
    if (idx >= 0 && idx < n) colsel[idx] = 1;
    else if (idx >= n && idx < 3 * n - 1) diagsel[idx - n] = 1;
  }
  __syncthreads();

  // mask rows / columns [video0, video0 + n) are the video's; the others (the text of the
  // hunyuan / cogvideox layouts, all cells of the 'other' layout) are true throughout
  const int video0 = p.layout == MODDIT_LAYOUT_COGVIDEOX ? p.text_blocks
                     : p.layout == MODDIT_LAYOUT_OTHER   ? nb
                                                         : 0;
  const bool full = mode == MODDIT_MODE_FULL;
  const bool bd = mode == MODDIT_MODE_BLOCK_DIAGONAL;
  const int per_tile = p.block == 64 ? 2 : 1;
  const int per_col = p.block == 64 ? 1 : 2;
  const bool both = p.block == 128 || p.union_rows;
  constexpr uint64_t kOnes = 0x0101010101010101ull;

  // 8 consecutive bytes of an LDS byte map from index i >= 0
  auto window = [](const uint8_t* map, int i) -> uint64_t {
    const uint64_t* w = reinterpret_cast<const uint64_t*>(map) + (i >> 3);
    const int sh = (i & 7) * 8;
    const uint64_t lo = w[0];
    return sh ? (lo >> sh) | (w[1] << (64 - sh)) : lo;
  };
  // the mask bytes (0/1) of columns j0 .. j0+7 in video row iv (iv < 0: a text row)
  auto row_bytes = [&](int iv, int j0) -> uint64_t {
    if (j0 >= nb) return 0;
    const uint64_t valid = nb - j0 >= kMaskCols ? kOnes : kOnes >> (8 * (kMaskCols - (nb - j0)));
    if (full || iv < 0) return valid;
    const int jv0 = j0 - video0;
    uint64_t r;
    if (jv0 >= 0 && jv0 + kMaskCols <= n) {
      // selected columns, then the diagonals jv - iv + n - 1 in [0, 2n-2]
      r = window(colsel, jv0) | window(diagsel, jv0 - iv + n - 1);
      if (bd) {
        const int f0 = iv / p.bpf * p.bpf;  // columns of the row's frame: [f0, f0 + bpf)
        int a = f0 - jv0;
        int b = f0 + p.bpf - jv0;
        a = a < 0 ? 0 : a;
        b = b > kMaskCols ? kMaskCols : b;
        if (a < b) r |= (kOnes >> (8 * (kMaskCols - (b - a)))) << (8 * a);
      }
    } else {
      r = 0;
#pragma unroll
      for (int c = 0; c < kMaskCols; ++c) {
        const int jv = jv0 + c;
        const bool video = jv >= 0 && jv < n;
        if (!video || colsel[jv] || diagsel[jv - iv + n - 1] || (bd && jv / p.bpf == iv / p.bpf))
          r |= 1ull << (8 * c);
      }
    }
    return r & valid;
  };
  // one 8-byte store where the row holds all eight columns (rows start at any byte
  // address; global stores need no alignment), bytes at its end
  auto store_row = [&](int row, int j0, uint64_t bytes) {
    uint8_t* dst = p.mask_out + (static_cast<int64_t>(h) * nb + row) * nb + j0;
    if (j0 + kMaskCols <= nb) {
      __builtin_memcpy(dst, &bytes, 8);
    } else {
      for (int c = 0; c < kMaskCols && j0 + c < nb; ++c) dst[c] = (bytes >> (8 * c)) & 1;
    }
  };

  for (int t = t_begin + (tid >> 6); t < t_end; t += kMaskWaves) {
    const int r0 = t * per_tile;
    const bool has_r1 = per_tile == 2 && r0 + 1 < nb;
    const int v0 = r0 - video0;
    const int iv0 = v0 >= 0 && v0 < n ? v0 : -1;
    const int iv1 = v0 + 1 >= 0 && v0 + 1 < n ? v0 + 1 : -1;
    const int64_t slot = static_cast<int64_t>(h) * p.n_qtiles + t;
    int32_t* out = p.counts ? p.entries + slot * p.cap : nullptr;
    int written = 0;
    for (int jb = 0; jb < nb; jb += kMaskPass) {
      const int j0 = jb + lane * kMaskCols;
      const uint64_t b0 = row_bytes(iv0, j0);
      const uint64_t b1 = has_r1 ? row_bytes(iv1, j0) : 0;
      if (p.mask_out && j0 < nb) {
        store_row(r0, j0, b0);
        if (has_r1) store_row(r0 + 1, j0, b1);
      }
      if (out != nullptr)
        written = emit_tiles(byte_bits(b0), byte_bits(b1), j0, lane, per_col, both, nb * per_col,
                             out, p.cap, written);
    }
    if (out != nullptr && lane == 0) p.counts[slot] = written < p.cap ? written : p.cap;
  }
}

// Tile lists of a caller's bool mask (MoD/mod/attn_mask.py:296-311), with the mask bytes read
// 8 at a time at any byte address. Bound by reading the mask; with the byte loads and the
// workgroup scans that this replaced: 28 us at 64 blocks x 2 heads (8 workgroups), 36 us at
// 454 x 24, 37 us at 225 x 24; 4.2, 9.8 and 6.5 us now.
struct MaskTilesParams {
  const uint8_t* mask;  // (H, n_rows, nb), any nonzero byte is true
  int64_t head_stride;
  int64_t row_stride;
  int heads;
  int n_rows;
  int nb;
  int block;
  int union_rows;
  int kv_tiles;  // key tiles at or beyond are dropped
  int32_t* counts;
  int32_t* entries;
  int n_qtiles;
  int cap;
};

__global__ __launch_bounds__(kMaskThreads) void tiles_from_mask_kernel(MaskTilesParams p) {
  const int lane = threadIdx.x & 63;
  const int64_t slot = static_cast<int64_t>(blockIdx.x) * kMaskWaves + (threadIdx.x >> 6);
  if (slot >= static_cast<int64_t>(p.heads) * p.n_qtiles) return;
  const int h = static_cast<int>(slot / p.n_qtiles);
  const int t = static_cast<int>(slot - static_cast<int64_t>(h) * p.n_qtiles);
  const int per_tile = p.block == 64 ? 2 : 1;
  const int per_col = p.block == 64 ? 1 : 2;
  const int r0 = t * per_tile;
  const uint8_t* row0 = p.mask + h * p.head_stride + r0 * p.row_stride;
  const uint8_t* row1 = row0 + p.row_stride;
  const bool has_r1 = per_tile == 2 && r0 + 1 < p.n_rows;
  const bool both = p.block == 128 || p.union_rows;

  // bit c: byte c of the 8 mask bytes at `row + j` is nonzero (columns past nb: clear)
  auto load_bits = [&](const uint8_t* row, int j) -> unsigned {
    uint64_t v = 0;
    if (j + kMaskCols <= p.nb) {
      __builtin_memcpy(&v, row + j, 8);
    } else {
      for (int c = 0; j + c < p.nb; ++c) v |= static_cast<uint64_t>(row[j + c]) << (8 * c);
    }
    const uint64_t low7 = 0x7f7f7f7f7f7f7f7full;
    return byte_bits(((((v & low7) + low7) | v) >> 7) & 0x0101010101010101ull);
  };

  int written = 0;
  for (int jb = 0; jb < p.nb; jb += kMaskPass) {
    const int j0 = jb + lane * kMaskCols;
    const unsigned m0 = j0 < p.nb ? load_bits(row0, j0) : 0u;
    const unsigned m1 = has_r1 && j0 < p.nb ? load_bits(row1, j0) : 0u;
    written = emit_tiles(m0, m1, j0, lane, per_col, both, p.kv_tiles,
                         p.entries + slot * p.cap, p.cap, written);
  }
  if (lane == 0) p.counts[slot] = written < p.cap ? written : p.cap;
}

// =====================================================================================
// Refresh merge (MoD/mod/attn_mask.py:671-675)
// =====================================================================================
__global__ void refresh_merge_kernel(const uint16_t* __restrict__ prev,
                                     const uint16_t* __restrict__ cur,
                                     const uint8_t* __restrict__ mask, int64_t mhs, int64_t mrs,
                                     int heads, int n, uint16_t* out) {
  const int64_t total = static_cast<int64_t>(heads) * n * n;
  for (int64_t idx = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; idx < total;
       idx += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t h = idx / (static_cast<int64_t>(n) * n);
    const int64_t rem = idx - h * n * n;
    const int64_t i = rem / n;
    const int64_t j = rem - i * n;
    const bool m = mask[h * mhs + i * mrs + j] != 0;
    out[idx] = m ? cur[idx] : prev[idx];
  }
}

}  // namespace
}  // namespace moddit

using namespace moddit;

extern "C" int64_t moddit_mts_workspace_bytes(int heads, int n) {
  if (heads <= 0 || n <= 0) return 0;
  const int rows = mts_rows_for(heads, n);
  const int64_t n_rt = (n + kMtsWaves * rows - 1) / (kMtsWaves * rows);
  const int64_t n_ct = (n + kMtsTileC - 1) / kMtsTileC;
  return heads * n_rt * n_ct * mts_record_doubles(rows) * static_cast<int64_t>(sizeof(double));
}

extern "C" int moddit_mts(const void* map, int map_dtype, int heads, int n, int blocks_per_frame,
                          void* workspace, float* mts_out, moddit_stream_t stream) {
  clear_error();
  MODDIT_CHECK_ARG(map && mts_out, "mts: null pointer argument");
  MODDIT_CHECK_ARG(map_dtype == MODDIT_FP16 || map_dtype == MODDIT_FP32,
                   "mts: map dtype must be fp16 or fp32");
  MODDIT_CHECK_ARG(heads >= 0 && n > 0, "mts: invalid shape heads=%d n=%d", heads, n);
  MODDIT_CHECK_ARG(blocks_per_frame > 0, "mts: blocks_per_frame must be positive, got %d",
                   blocks_per_frame);
  if (heads == 0) return MODDIT_OK;
  hipStream_t st = as_stream(stream);
  if (map_dtype == MODDIT_FP16) {
    MODDIT_CHECK_ARG(workspace != nullptr, "mts: fp16 maps need a workspace of "
                     "moddit_mts_workspace_bytes(heads, n) bytes");
    MODDIT_CHECK_ARG(aligned16(workspace), "mts: workspace must be 16-byte aligned");
    MODDIT_CHECK_ARG(n <= kMts1MaxN, "mts: n=%d exceeds %d", n, kMts1MaxN);
    MODDIT_CHECK_ARG(static_cast<int64_t>(n) * (blocks_per_frame < n ? blocks_per_frame : n) <=
                         kMts1MaxFrameCells,
                     "mts: n * min(blocks_per_frame, n) = %lld frame-block cells exceed %lld "
                     "(the exact fp16 sum's int64 range)",
                     static_cast<long long>(n) * (blocks_per_frame < n ? blocks_per_frame : n),
                     static_cast<long long>(kMts1MaxFrameCells));
    Mts1Params q;
    q.map = static_cast<const uint16_t*>(map);
    q.heads = heads;
    q.n = n;
    q.bpf = blocks_per_frame;
    q.records = static_cast<double*>(workspace);
    q.out = mts_out;
    return mts_rows_for(heads, n) == kMtsRowsTall ? launch_mts_fp16<kMtsRowsTall>(q, st)
                                                  : launch_mts_fp16<kMtsRowsShort>(q, st);
  }
  MtsParams p;
  p.map = static_cast<const float*>(map);
  p.heads = heads;
  p.n = n;
  p.bpf = blocks_per_frame;
  p.n_bands = (2 * n - 1 + 63) / 64;
  p.n_strips = (n + 63) / 64;
  p.out = mts_out;
  const int64_t grid = static_cast<int64_t>(heads) * (p.n_bands + p.n_strips + 1);
  MODDIT_CHECK_ARG(grid < 0x7fffffff, "mts: shape too large");
  hipLaunchKernelGGL(mts_kernel, dim3(static_cast<unsigned>(grid)), dim3(kMtsThreads), 0, st, p);
  MODDIT_CHECK_LAUNCH("mts");
  return MODDIT_OK;
}

// Closed form of M^T M + lambda I (MoD/mod/cuda_lstsq.py:42-89). Column order of M:
// [2n-1 diagonals by offset -(n-1)..n-1][n columns][1 frame-block-diagonal].
extern "C" int moddit_mtm_host(int n, int blocks_per_frame, double regularization,
                               double* mtm_out) {
  clear_error();
  MODDIT_CHECK_ARG(mtm_out != nullptr, "mtm: null output");
  MODDIT_CHECK_ARG(n > 0 && blocks_per_frame > 0, "mtm: invalid n=%d bpf=%d", n, blocks_per_frame);
  const int nd = 2 * n - 1;
  const int64_t F = 3 * static_cast<int64_t>(n);
  for (int64_t i = 0; i < F * F; ++i) mtm_out[i] = 0.0;
  const int bpf = blocks_per_frame;
  const int nbk = n / bpf;
  for (int kd = 0; kd < nd; ++kd) {
    const int off = kd - (n - 1);
    const int aoff = off < 0 ? -off : off;
    mtm_out[kd * F + kd] = static_cast<double>(n - aoff);
    for (int c = 0; c < n; ++c) {
      // diagonal with col-row = off crosses column c iff row = c - off is in [0, n)
      const bool hit = off >= 0 ? (c >= off) : (c < n + off);
      if (hit) {
        mtm_out[kd * F + nd + c] = 1.0;
        mtm_out[(nd + c) * F + kd] = 1.0;
      }
    }
    const double db = aoff < bpf ? static_cast<double>(nbk) * (bpf - aoff) : 0.0;
    mtm_out[kd * F + (F - 1)] = db;
    mtm_out[(F - 1) * F + kd] = db;
  }
  for (int c = 0; c < n; ++c) {
    mtm_out[(nd + c) * F + nd + c] = static_cast<double>(n);
    const double vb = c < nbk * bpf ? static_cast<double>(bpf) : 0.0;
    mtm_out[(nd + c) * F + (F - 1)] = vb;
    mtm_out[(F - 1) * F + nd + c] = vb;
  }
  mtm_out[(F - 1) * F + (F - 1)] = static_cast<double>(nbk) * bpf * bpf;
  for (int64_t i = 0; i < F; ++i) mtm_out[i * F + i] += regularization;
  return MODDIT_OK;
}

extern "C" int moddit_select_lines(const float* x_cur, const float* x_last, int heads, int n,
                                   int predict_T, int top_k, int32_t* sel_out,
                                   moddit_stream_t stream) {
  clear_error();
  MODDIT_CHECK_ARG(x_cur && x_last && sel_out, "select_lines: null pointer argument");
  MODDIT_CHECK_ARG(n > 0 && heads >= 0, "select_lines: invalid shape");
  MODDIT_CHECK_ARG(predict_T != 0, "select_lines: predict_T must be nonzero");
  const int items = 3 * n - 1;
  MODDIT_CHECK_ARG(items <= kSelMaxItems, "select_lines: 3n-1=%d exceeds %d", items, kSelMaxItems);
  MODDIT_CHECK_ARG(top_k > 0, "select_lines: top_k must be positive, got %d", top_k);
  const int k = top_k < items ? top_k : items;
  if (heads == 0) return MODDIT_OK;
  const size_t lds = static_cast<size_t>(items) * sizeof(unsigned long long);
  static LaunchSetup once;
  if (set_dynamic_lds_once(once, reinterpret_cast<const void*>(select_kernel),
                           kSelMaxItems * 8) != hipSuccess) {
    set_error("select_lines: cannot reserve LDS");
    return MODDIT_EHIP;
  }
  hipLaunchKernelGGL(select_kernel, dim3(heads), dim3(kSelThreads), lds, as_stream(stream), x_cur,
                     x_last, n, 0.f, predict_T, k, sel_out);
  MODDIT_CHECK_LAUNCH("select_lines");
  return MODDIT_OK;
}

extern "C" int moddit_check_bd(const float* x, int heads, int features, float threshold,
                               uint8_t* mode, moddit_stream_t stream) {
  clear_error();
  MODDIT_CHECK_ARG(x && mode, "check_bd: null pointer argument");
  MODDIT_CHECK_ARG(heads >= 0 && features > 0, "check_bd: invalid shape");
  if (heads == 0) return MODDIT_OK;
  hipLaunchKernelGGL(check_bd_kernel, dim3((heads + 63) / 64), dim3(64), 0, as_stream(stream), x,
                     heads, features, threshold, mode);
  MODDIT_CHECK_LAUNCH("check_bd");
  return MODDIT_OK;
}

static int check_tile_outputs(int n_rows, int nb, int block_size, int n_qtiles, int cap) {
  const int64_t tokens = static_cast<int64_t>(n_rows) * block_size;
  const int64_t need_q = (tokens + 127) / 128;
  MODDIT_CHECK_ARG(n_qtiles == need_q, "mask tiles: n_qtiles=%d but %lld mask tokens need %lld",
                   n_qtiles, static_cast<long long>(tokens), static_cast<long long>(need_q));
  MODDIT_CHECK_ARG(cap >= nb * (block_size / 64), "mask tiles: cap=%d below %d key tiles", cap,
                   nb * (block_size / 64));
  return MODDIT_OK;
}

extern "C" int moddit_mask_from_lines(const int32_t* sel, int heads, int k, const uint8_t* mode,
                                      int n, int blocks_per_frame, int layout, int nb,
                                      int text_blocks, int block_size, int union_rows,
                                      uint8_t* mask_out, int32_t* counts, int32_t* entries,
                                      int n_qtiles, int cap, moddit_stream_t stream) {
  clear_error();
  MODDIT_CHECK_ARG(sel != nullptr || k == 0, "mask_from_lines: null selection");
  MODDIT_CHECK_ARG(heads >= 0 && n > 0 && nb > 0 && k >= 0, "mask_from_lines: invalid shape");
  MODDIT_CHECK_ARG(blocks_per_frame > 0, "mask_from_lines: blocks_per_frame must be positive");
  MODDIT_CHECK_ARG(block_size == 64 || block_size == 128, "mask_from_lines: block_size must be 64 or 128");
  MODDIT_CHECK_ARG(layout >= 0 && layout <= MODDIT_LAYOUT_OTHER, "mask_from_lines: bad layout");
  MODDIT_CHECK_ARG((counts == nullptr) == (entries == nullptr),
                   "mask_from_lines: counts and entries go together");
  if (layout == MODDIT_LAYOUT_WAN) MODDIT_CHECK_ARG(nb == n, "mask_from_lines: wan layout needs nb == n");
  if (layout == MODDIT_LAYOUT_HUNYUAN) MODDIT_CHECK_ARG(nb >= n, "mask_from_lines: hunyuan layout needs nb >= n");
  if (layout == MODDIT_LAYOUT_COGVIDEOX)
    MODDIT_CHECK_ARG(text_blocks >= 0 && nb - text_blocks == n,
                     "mask_from_lines: cogvideox layout needs nb - text_blocks == n");
  if (counts) {
    int rc = check_tile_outputs(nb, nb, block_size, n_qtiles, cap);
    if (rc) return rc;
  } else {
    n_qtiles = static_cast<int>((static_cast<int64_t>(nb) * block_size + 127) / 128);
  }
  if (heads == 0) return MODDIT_OK;
  MaskParams p{};
  p.sel = sel;
  p.k = k;
  p.mode = mode;
  p.n = n;
  p.bpf = blocks_per_frame;
  p.layout = layout;
  p.nb = nb;
  p.text_blocks = text_blocks;
  p.block = block_size;
  p.union_rows = union_rows;
  p.mask_out = mask_out;
  p.counts = counts;
  p.entries = entries;
  p.n_qtiles = n_qtiles;
  p.cap = cap;
  const size_t lds = static_cast<size_t>(mask_lds_bytes(n));
  MODDIT_CHECK_ARG(lds <= 65536, "mask_from_lines: n=%d too large", n);
  const int64_t grid = static_cast<int64_t>(heads) * ((n_qtiles + kMaskTilesPerWg - 1) / kMaskTilesPerWg);
  hipLaunchKernelGGL(mask_tiles_kernel, dim3(static_cast<unsigned>(grid)),
                     dim3(kMaskThreads), lds, as_stream(stream), p);
  MODDIT_CHECK_LAUNCH("mask_from_lines");
  return MODDIT_OK;
}

extern "C" int moddit_mask_to_tiles(const uint8_t* mask, int heads, int n_rows, int n_cols,
                                    int64_t mask_head_stride, int64_t mask_row_stride,
                                    int block_size, int union_rows, int kv_tiles,
                                    int32_t* counts, int32_t* entries, int n_qtiles, int cap,
                                    moddit_stream_t stream) {
  clear_error();
  MODDIT_CHECK_ARG(mask && counts && entries, "mask_to_tiles: null pointer argument");
  MODDIT_CHECK_ARG(heads >= 0 && n_rows > 0 && n_cols > 0, "mask_to_tiles: invalid shape");
  MODDIT_CHECK_ARG(mask_head_stride >= 0 && mask_row_stride >= n_cols,
                   "mask_to_tiles: invalid mask strides");
  MODDIT_CHECK_ARG(block_size == 64 || block_size == 128, "mask_to_tiles: block_size must be 64 or 128");
  int rc = check_tile_outputs(n_rows, n_cols, block_size, n_qtiles, cap);
  if (rc) return rc;
  if (heads == 0) return MODDIT_OK;
  MaskTilesParams p;
  p.mask = mask;
  p.head_stride = mask_head_stride;
  p.row_stride = mask_row_stride;
  p.heads = heads;
  p.n_rows = n_rows;
  p.nb = n_cols;
  p.block = block_size;
  p.union_rows = union_rows;
  p.kv_tiles = kv_tiles < 0 ? 0 : kv_tiles;
  p.counts = counts;
  p.entries = entries;
  p.n_qtiles = n_qtiles;
  p.cap = cap;
  const int64_t grid = (static_cast<int64_t>(heads) * n_qtiles + kMaskWaves - 1) / kMaskWaves;
  MODDIT_CHECK_ARG(grid <= 0x7fffffff, "mask_to_tiles: shape too large");
  hipLaunchKernelGGL(tiles_from_mask_kernel, dim3(static_cast<unsigned>(grid)),
                     dim3(kMaskThreads), 0, as_stream(stream), p);
  MODDIT_CHECK_LAUNCH("mask_to_tiles");
  return MODDIT_OK;
}

extern "C" int moddit_refresh_merge(const void* prev, const void* cur, const uint8_t* mask,
                                    int64_t mask_head_stride, int64_t mask_row_stride, int heads,
                                    int n, void* out, moddit_stream_t stream) {
  clear_error();
  MODDIT_CHECK_ARG(prev && cur && mask && out, "refresh_merge: null pointer argument");
  MODDIT_CHECK_ARG(heads >= 0 && n >= 0, "refresh_merge: invalid shape");
  const int64_t total = static_cast<int64_t>(heads) * n * n;
  if (total == 0) return MODDIT_OK;
  int64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(refresh_merge_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                     as_stream(stream), static_cast<const uint16_t*>(prev),
                     static_cast<const uint16_t*>(cur), mask, mask_head_stride, mask_row_stride,
                     heads, n, static_cast<uint16_t*>(out));
  MODDIT_CHECK_LAUNCH("refresh_merge");
  return MODDIT_OK;
}
