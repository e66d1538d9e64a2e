// Stable LSD radix sort of particles by cell id.
//
// Binning (locate_particles, mesh.tcc:1097-1153) gives each particle a cell;
// the scatter kernels need the particles grouped by cell with ascending
// particle ids inside each cell. Sorting the pairs (cell, id) with a stable
// sort over the id-ordered input gives exactly that. Each pass is
//   hist:    per tile, a digit histogram (LDS atomics),
//   scan:    exclusive scan of the digit-major histogram table,
//   scatter: per tile, stable ranks from wave64 ballots (one-bit ballots
//            form each lane's digit-match mask), written at the scanned
//            offsets.
// The first pass reads the particles' cells themselves. A pass costs launches
// and tile latency rather than bytes at the sizes a step has, so digits are as
// wide as makes the passes few (up to 10 bits: 2 passes up to a million cells,
// where 8-bit digits took 3), and tiles shrink with the number of particles so
// that they still cover the device. One sort with 8-bit digits, 4096-key tiles
// and 5 launches a pass -> this: 8k particles 67 -> 26 us, 24k 64 -> 34, 262k
// (3 passes -> 2) 96 -> 42, 2.1M 133 -> 103, 5.2M 180 -> 140.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mpmx_kernels.h"

namespace mpmx {

static constexpr int kSortBlock = 256;
static constexpr int kWaves = kSortBlock / 64;
static constexpr int kMaxBits = 10;
static constexpr int kMaxBins = 1 << kMaxBits;
static constexpr int kScanTile = 1024;
// Up to this many table entries one workgroup scans the table in one launch.
static constexpr int kScanOne = 32768;
// Up to this many scan tiles, every tile sums the totals before it itself.
static constexpr int kScanDirect = 2048;

// Rounds of kSortBlock keys per tile: short tiles for few particles (a tile is
// a chain of dependent rounds, 1 us each), long ones where the table, a row of
// digits per tile, would cost more than the rounds.
static inline int rounds_for(int64_t n) {
  return n < (64 << 10) ? 1 : (n < (512 << 10) ? 4 : (n < (2 << 20) ? 8 : 16));
}
static inline int64_t tiles_for(int64_t n) {
  const int64_t t = (int64_t)kSortBlock * rounds_for(n);
  return (n + t - 1) / t;
}

// Passes and the bits of a pass's digit for keys up to max_key.
struct Digits {
  int passes, width;
};
static inline Digits digits_for(int max_key) {
  int bits = 1;
  while (bits < 31 && (1ll << bits) <= (long long)max_key) ++bits;
  const int passes = (bits + kMaxBits - 1) / kMaxBits;
  return {passes, (bits + passes - 1) / passes};
}

int64_t radix_sort_temp_ints(int64_t n, int max_key) {
  const int64_t table = std::max<int64_t>(tiles_for(n), 1) << digits_for(max_key).width;
  return 2 * n + table + (table + kScanTile - 1) / kScanTile + 64;
}

// keys: cell in [0, ncells) else max_key
template <bool FIRST>
__device__ __forceinline__ int load_key(const int* keys, int64_t i, int max_key) {
  const int c = keys[i];
  return !FIRST || (c >= 0 && c < max_key) ? c : max_key;
}

template <bool FIRST>
__global__ __launch_bounds__(kSortBlock) void k_rs_hist(const int* keys, int64_t n, int max_key,
                                                        int shift, int nbins, int rounds,
                                                        int* hist, int64_t nblocks) {
  __shared__ int bins[kMaxBins];
  for (int b = threadIdx.x; b < nbins; b += kSortBlock) bins[b] = 0;
  __syncthreads();
  const int64_t base = blockIdx.x * (int64_t)(kSortBlock * rounds);
  for (int r = 0; r < rounds; ++r) {
    const int64_t i = base + r * kSortBlock + threadIdx.x;
    if (i < n) atomicAdd(&bins[(load_key<FIRST>(keys, i, max_key) >> shift) & (nbins - 1)], 1);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < nbins; b += kSortBlock) hist[b * nblocks + blockIdx.x] = bins[b];
}

// Exclusive scan of `total` ints in place: each 1024-element tile is scanned
// by one block (4 consecutive elements per thread, wave prefix sums by
// shuffles), then the totals of the tiles before it are added.

__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int u = __shfl_up(v, off, 64);
    if (lane >= off) v += u;
  }
  return v;
}

// block-wide exclusive scan of one value per thread (WAVES * 64 threads);
// returns the exclusive prefix and writes the block total to *total
template <int WAVES>
__device__ __forceinline__ int block_excl_scan(int v, int* total) {
  __shared__ int wsum[WAVES];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int incl = wave_incl_scan(v);
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  int before = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    before += (w < wave) ? wsum[w] : 0;
    tot += wsum[w];
  }
  __syncthreads();
  *total = tot;
  return before + incl - v;
}

// The whole table (at most kScanOne entries) by one workgroup.
__global__ __launch_bounds__(1024) void k_rs_scan_one(int* a, int total) {
  constexpr int PER = kScanOne / 1024;
  const int per = (total + 1023) / 1024, b = threadIdx.x * per;
  int v[PER], s = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    v[j] = (j < per && b + j < total) ? a[b + j] : 0;
    s += v[j];
  }
  int tot;
  int run = block_excl_scan<16>(s, &tot);
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (j < per && b + j < total) a[b + j] = run;
    run += v[j];
  }
}

__global__ __launch_bounds__(256) void k_rs_scan_tiles(int* a, int64_t total, int* tile_sums) {
  const int64_t base = blockIdx.x * (int64_t)kScanTile + threadIdx.x * 4;
  int v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = (base + j < total) ? a[base + j] : 0;
  const int s = (v[0] + v[1]) + (v[2] + v[3]);
  int tot;
  int run = block_excl_scan<4>(s, &tot);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (base + j < total) a[base + j] = run;
    run += v[j];
  }
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = tot;
}

// exclusive scan of the tile sums (any count) by one block
__global__ __launch_bounds__(256) void k_rs_scan_sums(int* sums, int64_t n) {
  __shared__ int carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int64_t b = 0; b < n; b += 256) {
    const int64_t i = b + threadIdx.x;
    const int v = i < n ? sums[i] : 0;
    int tot;
    const int ex = block_excl_scan<4>(v, &tot);
    if (i < n) sums[i] = carry + ex;
    __syncthreads();
    if (threadIdx.x == 0) carry += tot;
    __syncthreads();
  }
}

// DIRECT: `sums` holds the tiles' totals, summed here up to the block's own;
// else their exclusive scan.
template <bool DIRECT>
__global__ __launch_bounds__(256) void k_rs_scan_add(int* a, int64_t total, const int* sums) {
  int add = 0;
  if constexpr (DIRECT) {
    int s = 0;
    for (int i = threadIdx.x; i < (int)blockIdx.x; i += 256) s += sums[i];
    (void)block_excl_scan<4>(s, &add);
  } else {
    add = sums[blockIdx.x];
  }
  const int64_t base = blockIdx.x * (int64_t)kScanTile;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t i = base + j * 256 + threadIdx.x;
    if (i < total) a[i] += add;
  }
}

template <bool FIRST>
__global__ __launch_bounds__(kSortBlock) void k_rs_scatter(const int* kin, const int* vin,
                                                           int* kout, int* vout, int64_t n,
                                                           int max_key, int shift, int bits,
                                                           int rounds, const int* hist,
                                                           int64_t nblocks) {
  __shared__ int base[kMaxBins];
  __shared__ unsigned short wcount[kWaves][kMaxBins];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int nbins = 1 << bits;
  for (int b = tid; b < nbins; b += kSortBlock) {
    base[b] = hist[b * nblocks + blockIdx.x];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) wcount[w][b] = 0;
  }
  __syncthreads();
  const unsigned long long lt = (1ull << lane) - 1ull;
  const int64_t tbase = blockIdx.x * (int64_t)(kSortBlock * rounds);
  for (int r = 0; r < rounds; ++r) {
    const int64_t i = tbase + r * kSortBlock + tid;
    const bool valid = i < n;
    int key = 0, val = 0, digit = 0;
    if (valid) {
      key = load_key<FIRST>(kin, i, max_key);
      val = FIRST ? (int)i : vin[i];
      digit = (key >> shift) & (nbins - 1);
    }
    unsigned long long mask = __ballot(valid);
    for (int b = 0; b < bits; ++b) {
      const int bit = (digit >> b) & 1;
      const unsigned long long bal = __ballot(bit);
      mask &= bit ? bal : ~bal;
    }
    const int rank = __popcll(mask & lt);
    if (valid && rank == 0) wcount[wave][digit] = (unsigned short)__popcll(mask);
    __syncthreads();
    if (valid) {
      int off = base[digit] + rank;
      for (int w = 0; w < wave; ++w) off += wcount[w][digit];
      kout[off] = key;
      vout[off] = val;
    }
    if (r + 1 == rounds) break;  // the same for every thread
    __syncthreads();
    for (int b = tid; b < nbins; b += kSortBlock) {
      int tot = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        tot += wcount[w][b];
        wcount[w][b] = 0;
      }
      base[b] += tot;
    }
    __syncthreads();
  }
}

void radix_sort_by_cell(const int* cell, int64_t n, int max_key, int* keys_out, int* vals_out,
                        int* tmp, hipStream_t st) {
  if (n <= 0) return;
  const int rounds = rounds_for(n);
  const int64_t nb = tiles_for(n);
  int* hist = tmp + 2 * n;
  const auto [passes, width] = digits_for(max_key);
  const int nbins = 1 << width;
  const int64_t total = nbins * nb;
  const int64_t ntiles = (total + kScanTile - 1) / kScanTile;
  int* tile_sums = hist + total;
  const int* sk = cell;
  const int* sv = nullptr;
  for (int pass = 0; pass < passes; ++pass) {
    // the passes alternate between the outputs and tmp and end in the outputs
    const bool out = (passes - 1 - pass) % 2 == 0;
    int* dk = out ? keys_out : tmp;
    int* dv = out ? vals_out : tmp + n;
    const int shift = width * pass;
    const dim3 g((unsigned)nb), b(kSortBlock);
    if (pass == 0)
      hipLaunchKernelGGL((k_rs_hist<true>), g, b, 0, st, sk, n, max_key, shift, nbins, rounds,
                         hist, nb);
    else
      hipLaunchKernelGGL((k_rs_hist<false>), g, b, 0, st, sk, n, max_key, shift, nbins, rounds,
                         hist, nb);
    if (total <= kScanOne) {
      hipLaunchKernelGGL(k_rs_scan_one, dim3(1), dim3(1024), 0, st, hist, (int)total);
    } else {
      hipLaunchKernelGGL(k_rs_scan_tiles, dim3((unsigned)ntiles), dim3(256), 0, st, hist, total,
                         tile_sums);
      if (ntiles <= kScanDirect) {
        hipLaunchKernelGGL((k_rs_scan_add<true>), dim3((unsigned)ntiles), dim3(256), 0, st, hist,
                           total, tile_sums);
      } else {
        hipLaunchKernelGGL(k_rs_scan_sums, dim3(1), dim3(256), 0, st, tile_sums, ntiles);
        hipLaunchKernelGGL((k_rs_scan_add<false>), dim3((unsigned)ntiles), dim3(256), 0, st, hist,
                           total, tile_sums);
      }
    }
    if (pass == 0)
      hipLaunchKernelGGL((k_rs_scatter<true>), g, b, 0, st, sk, sv, dk, dv, n, max_key, shift,
                         width, rounds, hist, nb);
    else
      hipLaunchKernelGGL((k_rs_scatter<false>), g, b, 0, st, sk, sv, dk, dv, n, max_key, shift,
                         width, rounds, hist, nb);
    sk = dk;
    sv = dv;
  }
}

}  // namespace mpmx
