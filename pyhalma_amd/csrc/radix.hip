// Stable LSD radix sort (8-bit digits).  Per pass: a per-block digit histogram, an
// exclusive scan of each digit's row of the digit-major [digit][block] table (a block per
// digit, which also writes the digit's total), then a stable scatter (each block adds the
// exclusive scan of the 256 digit totals, taken in LDS, to its row offsets) in which each
// wavefront ranks a contiguous part of the tile by digit on its own (ranks among equal
// digits of 64 keys from eight ballots, the wavefront's running counts in LDS), the
// wavefronts' counts are put together once, and the tile is sorted by digit in LDS and
// written digit run by digit run, consecutive threads to consecutive addresses.
//
// Bound by memory latency and the barriers of a tile.  A scatter pass of 8M pairs takes
// 45 us (2.8 TB/s), of 1.9M 16, of 24k 5.2; with 256 keys ranked per round by the whole
// workgroup, four barriers each, it took 56, 19 and 11.5.  Large inputs take tiles of 4096
// keys (longer runs per digit), small ones of 1024 (more blocks).
#include "radix.h"

#include <algorithm>

namespace halma {

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kSmall = 4, kLarge = 16;         // keys per thread of a tile
constexpr int64_t kLargeKeys = int64_t{1} << 20;  // inputs from this size take large tiles

inline int64_t tiles_of(int64_t n) {
    const int64_t tile = kThreads * (n >= kLargeKeys ? kLarge : kSmall);
    return n > 0 ? (n + tile - 1) / tile : 1;
}

template <int kRounds>
__global__ __launch_bounds__(kThreads) void k_radix_hist(const uint32_t* __restrict__ keys,
                                                         int64_t n, int shift, int64_t nb,
                                                         int32_t* __restrict__ hist) {
    __shared__ int h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = static_cast<int64_t>(blockIdx.x) * (kThreads * kRounds);
    uint32_t k[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const int64_t i = base + r * kThreads + threadIdx.x;
        k[r] = i < n ? keys[i] : 0;
    }
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
        if (base + r * kThreads + threadIdx.x < n) atomicAdd(&h[(k[r] >> shift) & 0xff], 1);
    __syncthreads();
    hist[static_cast<int64_t>(threadIdx.x) * nb + blockIdx.x] = h[threadIdx.x];
}

// exclusive scan of one int per thread over the block (256 threads)
__device__ int block_excl_scan(int v, int* sh /* kWaves */) {
    const int lane = __lane_id(), w = threadIdx.x / kWave;
    int x = v;
    for (int d = 1; d < kWave; d <<= 1) {
        const int y = __shfl_up(x, d, kWave);
        if (lane >= d) x += y;
    }
    if (lane == kWave - 1) sh[w] = x;
    __syncthreads();
    int before = 0;
    for (int k = 0; k < w; ++k) before += sh[k];
    __syncthreads();
    return before + x - v;
}

// Exclusive scan of one digit's row hist[d][0 .. nb) into offs (a block per digit, 1024
// entries per round, four consecutive per thread); the row's total goes to tot[d].
__global__ __launch_bounds__(kThreads) void k_radix_rows(const int32_t* __restrict__ hist,
                                                         int64_t nb, int32_t* __restrict__ offs,
                                                         int32_t* __restrict__ tot) {
    __shared__ int scan_sh[kWaves];
    __shared__ int last;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * nb;
    int run = 0;
    for (int64_t c = 0; c < nb; c += 4 * kThreads) {
        const int64_t j0 = c + 4 * threadIdx.x;
        int v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = j0 + u < nb ? hist[row + j0 + u] : 0;
        const int local = (v[0] + v[1]) + (v[2] + v[3]);
        const int excl = block_excl_scan(local, scan_sh);
        int o = run + excl;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (j0 + u < nb) offs[row + j0 + u] = o;
            o += v[u];
        }
        // the round's total: the last thread's exclusive prefix plus its own entries
        if (threadIdx.x == kThreads - 1) last = excl + local;
        __syncthreads();
        run += last;
        __syncthreads();
    }
    if (threadIdx.x == 0) tot[blockIdx.x] = run;
}

// Stable scatter of one tile: wavefront w ranks keys [w part, (w + 1) part) of the tile in
// order, 64 at a time.
template <int kRounds>
__global__ __launch_bounds__(kThreads) void k_radix_scatter(
    const uint32_t* __restrict__ keys, const int32_t* __restrict__ vals, int64_t n, int shift,
    int64_t nb, const int32_t* __restrict__ offs, const int32_t* __restrict__ tot,
    uint32_t* __restrict__ keys_out, int32_t* __restrict__ vals_out) {
    constexpr int kTile = kThreads * kRounds;
    __shared__ int wcnt[kWaves][256];  // counts of a wavefront, then its digits' first places
    __shared__ int loff[256];          // a digit's first place in the sorted tile
    __shared__ int scan_sh[kWaves];
    __shared__ int64_t run[256];
    __shared__ uint32_t sk[kTile];
    __shared__ int32_t sv[kTile];
    const int tid = threadIdx.x;
    const int lane = __lane_id();
    const int w = tid / kWave;
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kTile;
    const int64_t first = base + w * (kWave * kRounds) + lane;
    uint32_t kk[kRounds];
    int32_t vv[kRounds];
    int rk[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const int64_t i = first + r * kWave;
        kk[r] = i < n ? keys[i] : 0;
        vv[r] = i < n ? (vals ? vals[i] : static_cast<int32_t>(i)) : 0;
    }
    {  // start of the digit's run: the totals of the smaller digits plus this block's row offset
        const int row = offs[static_cast<int64_t>(tid) * nb + blockIdx.x];
        run[tid] = static_cast<int64_t>(block_excl_scan(tot[tid], scan_sh)) + row;
    }
#pragma unroll
    for (int k = 0; k < 256; k += kWave) wcnt[w][k + lane] = 0;
    const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const bool valid = first + r * kWave < n;
        const int digit = (kk[r] >> shift) & 0xff;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const bool bit = (digit >> b) & 1;
            const uint64_t m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        // the wavefront's counts: read by every lane of the digit, then raised by its last
        // (LDS accesses of one wavefront stay in order)
        const int before = valid ? wcnt[w][digit] : 0;
        const int rank = __popcll(peers & lt);
        __builtin_amdgcn_wave_barrier();
        if (valid && (peers >> lane) == 1ull) wcnt[w][digit] = before + rank + 1;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        rk[r] = valid ? before + rank : -1;
    }
    __syncthreads();
    int sum = 0;
    int part[kWaves];
#pragma unroll
    for (int k = 0; k < kWaves; ++k) {
        part[k] = sum;
        sum += wcnt[k][tid];
    }
    const int at = block_excl_scan(sum, scan_sh);
    loff[tid] = at;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) wcnt[k][tid] = at + part[k];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
        if (rk[r] >= 0) {
            const int pos = wcnt[w][(kk[r] >> shift) & 0xff] + rk[r];
            sk[pos] = kk[r];
            sv[pos] = vv[r];
        }
    __syncthreads();
    const int64_t left = n - base;
    const int tile_n = left < kTile ? static_cast<int>(left) : kTile;
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const int j = r * kThreads + tid;
        if (j < tile_n) {
            const uint32_t key = sk[j];
            const int d = (key >> shift) & 0xff;
            const int64_t dest = run[d] + (j - loff[d]);
            keys_out[dest] = key;
            vals_out[dest] = sv[j];
        }
    }
}

}  // namespace

// Enough for every sort of at most n pairs: a caller may size it for its largest, and the
// small tiles of just under kLargeKeys pairs need the longest tables up to 4M pairs.
size_t radix_workspace_bytes(int64_t n) {
    const int64_t nb = std::max(tiles_of(n), tiles_of(std::min(n, kLargeKeys - 1)));
    Carver c(nullptr);
    c.take<int32_t>(256 * nb);
    c.take<int32_t>(256 * nb);
    c.take<int32_t>(256);
    c.take<uint32_t>(n > 0 ? n : 1);
    c.take<int32_t>(n > 0 ? n : 1);
    return c.used;
}

int radix_sort_pairs(const uint32_t* keys_in, const int32_t* vals_in, uint32_t* keys_out,
                     int32_t* vals_out, int64_t n, int bits, void* ws, hipStream_t st) {
    if (n <= 0) return 0;
    if (n > INT32_MAX) return set_error(HALMA_E_LIMIT, "radix sort: too many keys");
    const int64_t nb = tiles_of(n);
    const bool large = n >= kLargeKeys;
    Carver c(ws);
    int32_t* hist = c.take<int32_t>(256 * nb);
    int32_t* offs = c.take<int32_t>(256 * nb);
    int32_t* tot = c.take<int32_t>(256);
    uint32_t* tk = c.take<uint32_t>(n);
    int32_t* tv = c.take<int32_t>(n);
    const int passes = bits <= 0 ? 1 : (bits + 7) / 8;
    // ping-pong so that the last pass lands in the output arrays
    const uint32_t* kin = keys_in;
    const int32_t* vin = vals_in;
    for (int p = 0; p < passes; ++p) {
        const bool to_out = ((passes - 1 - p) % 2) == 0;
        uint32_t* kout = to_out ? keys_out : tk;
        int32_t* vout = to_out ? vals_out : tv;
        auto hist_kernel = large ? k_radix_hist<kLarge> : k_radix_hist<kSmall>;
        hist_kernel<<<static_cast<unsigned>(nb), kThreads, 0, st>>>(kin, n, 8 * p, nb, hist);
        HALMA_LAUNCH_CHECK();
        k_radix_rows<<<256, kThreads, 0, st>>>(hist, nb, offs, tot);
        HALMA_LAUNCH_CHECK();
        auto scatter = large ? k_radix_scatter<kLarge> : k_radix_scatter<kSmall>;
        scatter<<<static_cast<unsigned>(nb), kThreads, 0, st>>>(kin, vin, n, 8 * p, nb, offs, tot,
                                                                kout, vout);
        HALMA_LAUNCH_CHECK();
        kin = kout;
        vin = vout;
    }
    return 0;
}

}  // namespace halma
