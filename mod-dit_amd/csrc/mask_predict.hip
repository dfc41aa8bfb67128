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
// Single pass over an fp16 map (the product path). One workgroup per (head, 512-row x
// 256-column tile) reads its cells once with 16-byte loads. Each thread owns 8 consecutive
// columns of one 64-row slab of the tile and keeps its column sums and, per 16-row
// sub-block, the sums of the 23 diagonals its 8 x 16 cells lie on in fp64 registers.
// Every finite fp16 value is a multiple of 2^-24 below 2^16, so any sum of at most 8192 of
// them needs at most 53 significant bits and is exact in fp64 in any order; a tile's
// share of one line is at most 512 cells. The eight slabs' column sums and the threads'
// overlapping diagonal sums are combined in LDS (still exact), and each workgroup adds
// its column, diagonal and frame-block partials into an int64 accumulator per output
// (units of 2^-24) with global integer atomics: exact and order-independent, so every
// output is the correctly rounded fp32 of the exact sum in any workgroup order
// (deterministic), and the map is read once (155.5 MB at the headline). A partial that is
// not finite (inf/NaN inputs) goes into a float side accumulator instead (inf/NaN
// semantics only, also order-independent). The tile shape minimises the global atomics
// per cell for its area (256 column + 767 diagonal partials per 131,072 cells): contended
// atomics, not the loads, were what bounded the 64-row-block version of this pass.
constexpr int kMts1Threads = 256;
constexpr int kMts1Cols = 8;         // columns per thread
constexpr int kMts1Sub = 16;         // rows per register sub-block
constexpr int kMts1Slab = 64;        // rows per thread
constexpr int kMts1ColThreads = 32;  // threads across a tile's columns
constexpr int kMts1Slabs = kMts1Threads / kMts1ColThreads;   // 8
constexpr int kMts1TileC = kMts1ColThreads * kMts1Cols;      // 256
constexpr int kMts1TileR = kMts1Slabs * kMts1Slab;           // 512
constexpr int kMts1Diag = kMts1Cols + kMts1Sub - 1;          // 23
constexpr int kMts1TileDiag = kMts1TileC + kMts1TileR - 1;   // 767
// Exactness of the int64 accumulators: an fp16 value is below 2^16, i.e. 2^40 units of
// 2^-24, so a sum over c cells stays below 2^63 while c <= 2^23. Diagonal and column
// outputs sum n cells; the frame-block output sums (n / bpf) * bpf^2 = n * min(bpf, n)
// cells, which the entry point bounds (kMts1MaxFrameCells).
constexpr int kMts1MaxN = 1 << 20;
constexpr int64_t kMts1MaxFrameCells = int64_t{1} << 23;

struct Mts1Params {
  const uint16_t* map;
  int heads;
  int n;
  int bpf;
  int n_rt;  // row tiles per head
  int n_ct;  // column tiles per head
  unsigned long long* acc;  // (H, 3n) int64 units of 2^-24 (two's complement)
  float* special;           // (H, 3n) sums of the non-finite partials
  float* out;               // (H, 3n)
};

// Adds an exact fp64 partial (a multiple of 2^-24, |x| < 2^25) to an output.
__device__ __forceinline__ void mts1_flush(const Mts1Params& p, int64_t idx, double x) {
  if (x == 0.0) return;
  if (__builtin_isfinite(x)) {
    atomicAdd(&p.acc[idx], static_cast<unsigned long long>(static_cast<long long>(x * 0x1p24)));
  } else {
    atomicAdd(&p.special[idx], static_cast<float>(x));
  }
}

__global__ void mts1_zero_kernel(Mts1Params p) {
  const int64_t total = static_cast<int64_t>(p.heads) * 3 * p.n;
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    p.acc[i] = 0ull;
    p.special[i] = 0.f;
  }
}

template <bool kVec>
__global__ __launch_bounds__(kMts1Threads) void mts1_kernel(Mts1Params p) {
  __shared__ double s_diag[kMts1TileDiag];
  __shared__ double s_col[kMts1Slabs][kMts1TileC];
  __shared__ long long s_frame[kMts1Threads / 64];
  const int tid = threadIdx.x;
  const int tc = tid % kMts1ColThreads;
  const int tr = tid / kMts1ColThreads;
  const int tiles = p.n_rt * p.n_ct;
  const int h = blockIdx.x / tiles;
  const int t = blockIdx.x - h * tiles;
  const int R0 = (t / p.n_ct) * kMts1TileR;
  const int C0 = (t % p.n_ct) * kMts1TileC;
  const int n = p.n;
  const int nd = 2 * n - 1;
  const int64_t F = 3 * static_cast<int64_t>(n);
  const int frame_end = (n / p.bpf) * p.bpf;
  for (int i = tid; i < kMts1TileDiag; i += kMts1Threads) s_diag[i] = 0.0;
  __syncthreads();

  const int c0 = C0 + tc * kMts1Cols;   // this thread's first column
  const int rs = R0 + tr * kMts1Slab;   // this thread's first row
  const uint16_t* base = p.map + static_cast<int64_t>(h) * n * n;
  const int64_t out0 = static_cast<int64_t>(h) * F;
  // frames of the first and last owned columns inside the frame blocks (-1: none)
  const int c_last = (c0 + kMts1Cols - 1 < frame_end ? c0 + kMts1Cols - 1 : frame_end - 1);
  const int cf_lo = c0 < frame_end ? c0 / p.bpf : -1;
  const int cf_hi = c0 < frame_end ? c_last / p.bpf : -1;
  double cacc[kMts1Cols];
#pragma unroll
  for (int j = 0; j < kMts1Cols; ++j) cacc[j] = 0.0;
  double fsum = 0.0;
  if (c0 < n) {
    for (int s0 = 0; s0 < kMts1Slab; s0 += kMts1Sub) {
      if (rs + s0 >= n) break;
      double dacc[kMts1Diag];
#pragma unroll
      for (int d = 0; d < kMts1Diag; ++d) dacc[d] = 0.0;
#pragma unroll
      for (int rr = 0; rr < kMts1Sub; ++rr) {
        const int r = rs + s0 + rr;
        if (r < n) {
          const uint16_t* row = base + static_cast<int64_t>(r) * n;
          uint16_t v[kMts1Cols];
          if constexpr (kVec) {
            const u32x4 w = *reinterpret_cast<const u32x4*>(row + c0);
#pragma unroll
            for (int j = 0; j < kMts1Cols; ++j) v[j] = u16_at(w, j);
          } else {
#pragma unroll
            for (int j = 0; j < kMts1Cols; ++j) v[j] = c0 + j < n ? row[c0 + j] : 0;
          }
          double x[kMts1Cols];
#pragma unroll
          for (int j = 0; j < kMts1Cols; ++j) {
            x[j] = static_cast<double>(Fp16::to_float(v[j]));
            cacc[j] += x[j];
            dacc[j - rr + kMts1Sub - 1] += x[j];
          }
          // frame-block cells: only rows whose frame meets the owned columns
          const int rframe = r < frame_end ? r / p.bpf : -2;
          if (rframe >= cf_lo && rframe <= cf_hi) {
#pragma unroll
            for (int j = 0; j < kMts1Cols; ++j)
              if (c0 + j < frame_end && (c0 + j) / p.bpf == rframe) fsum += x[j];
          }
        }
      }
      // local diagonal kl = (c - C0) - (r - R0) + 511 of accumulator d
#pragma unroll
      for (int d = 0; d < kMts1Diag; ++d) {
        const int kl = (c0 - C0) + d - (kMts1Sub - 1) - (rs - R0) - s0 + (kMts1TileR - 1);
        if (dacc[d] != 0.0) atomicAdd(&s_diag[kl], dacc[d]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < kMts1Cols; ++j) s_col[tr][tc * kMts1Cols + j] = cacc[j];
  // frame-block partial of the workgroup: each thread's sum (at most 512 cells) is exact in
  // fp64 and converts exactly to int64 units; the workgroup adds them as integers
  long long fq = 0;
  if (__builtin_isfinite(fsum))
    fq = static_cast<long long>(fsum * 0x1p24);
  else
    atomicAdd(&p.special[out0 + F - 1], static_cast<float>(fsum));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) fq += __shfl_xor(fq, o);
  if ((tid & 63) == 0) s_frame[tid >> 6] = fq;
  __syncthreads();
  if (tid == 0) {
    long long tot = 0;
    for (int w = 0; w < kMts1Threads / 64; ++w) tot += s_frame[w];
    if (tot != 0) atomicAdd(&p.acc[out0 + F - 1], static_cast<unsigned long long>(tot));
  }
  // column partials: the eight slabs' sums of one column (at most 512 cells, exact)
  for (int c = tid; c < kMts1TileC; c += kMts1Threads) {
    double sum = 0.0;
#pragma unroll
    for (int sl = 0; sl < kMts1Slabs; ++sl) sum += s_col[sl][c];
    if (C0 + c < n) mts1_flush(p, out0 + nd + C0 + c, sum);
  }
  // diagonal partials: global index k = (c - r) + n - 1 = kl - 511 + C0 - R0 + n - 1
  for (int kl = tid; kl < kMts1TileDiag; kl += kMts1Threads) {
    const int k = kl - (kMts1TileR - 1) + C0 - R0 + n - 1;
    if (k >= 0 && k < nd) mts1_flush(p, out0 + k, s_diag[kl]);
  }
}

__global__ void mts1_finalize_kernel(Mts1Params p) {
  const int64_t total = static_cast<int64_t>(p.heads) * 3 * p.n;
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const float sp = p.special[i];
    p.out[i] = (sp != 0.f || sp != sp)
                   ? sp
                   : static_cast<float>(static_cast<long long>(p.acc[i])) * 0x1p-24f;
  }
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
  return static_cast<int64_t>(heads) * 3 * n * (sizeof(unsigned long long) + sizeof(float));
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
    q.n_rt = (n + kMts1TileR - 1) / kMts1TileR;
    q.n_ct = (n + kMts1TileC - 1) / kMts1TileC;
    const int64_t total = static_cast<int64_t>(heads) * 3 * n;
    q.acc = static_cast<unsigned long long*>(workspace);
    q.special = reinterpret_cast<float*>(q.acc + total);
    q.out = mts_out;
    const int64_t grid = static_cast<int64_t>(heads) * q.n_rt * q.n_ct;
    MODDIT_CHECK_ARG(grid < 0x7fffffff, "mts: shape too large");
    int64_t fill = (total + 255) / 256;
    if (fill > 4096) fill = 4096;
    hipLaunchKernelGGL(mts1_zero_kernel, dim3(static_cast<unsigned>(fill)), dim3(256), 0, st, q);
    MODDIT_CHECK_LAUNCH("mts (zero)");
    const bool vec = n % 8 == 0 && aligned16(map);
    auto kernel = vec ? mts1_kernel<true> : mts1_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kMts1Threads), 0, st, q);
    MODDIT_CHECK_LAUNCH("mts");
    hipLaunchKernelGGL(mts1_finalize_kernel, dim3(static_cast<unsigned>(fill)), dim3(256), 0, st, q);
    MODDIT_CHECK_LAUNCH("mts (finalize)");
    return MODDIT_OK;
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
