// Potential-minimum centre of every halo: the fixed-point iteration
//   c <- c + a(c) / w(c),   a = sum_j m_j (x_j - c) (r^2 + eps^2)^(-3/2),
//                           w = sum_j m_j (r^2 + eps^2)^(-3/2)
// (the gradient step of Phi = -G S that never increases Phi), until every halo's step is
// at most tol * eps, then S at the centres.
//
// An iteration is one pass over the particles of the haloes still moving: a wavefront per
// chunk of kChunk particles (coalesced 16-byte loads, eight in flight per lane, FP32
// sub-tiles of 8 terms with Kahan sums, a fixed FP64 butterfly), then a wavefront per halo
// that adds the chunk sums in a fixed order and moves the centre.  The centres stay on the
// device: the host queues iterations kBatch at a time, one batch ahead of the count of
// moving haloes it reads back, and the kernels of haloes that have arrived return at once.
// What bounds it: reading 16 bytes per particle and iteration.  60 Hernquist haloes of
// 5e4-5e5 particles (11.7M, 31 iterations until the last one arrives): 1.20 ms; a launch of
// the batched softened sums per iteration with the step as tensor operations took 12.0 ms,
// most of it the host's.
#include <math.h>

#include <algorithm>
#include <vector>

#include "halma_common.h"
#include "soft_pair.h"
#include "staging.h"

namespace halma {

namespace {

constexpr int kChunk = 2048;  // particles of a wavefront's item
constexpr int kBatch = 4;     // iterations queued between two read-backs

struct __attribute__((aligned(8))) CentreDesc {
    int64_t src_off;
    int32_t src_len, first;  // first chunk
};

__global__ void k_centre_pack(const float* __restrict__ m, const float* __restrict__ x,
                              const float* __restrict__ y, const float* __restrict__ z,
                              int64_t n, float4* __restrict__ out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) out[i] = make_float4(x[i], y[i], z[i], m[i]);
}

__global__ void k_centre_init(int n_halo, int* __restrict__ moving, int* __restrict__ iters,
                              double* __restrict__ steps, int* __restrict__ left) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n_halo) {
        moving[i] = 1;
        iters[i] = 0;
        steps[i] = INFINITY;
    }
    if (i < 2) left[i] = 0;
}

// The sums of one chunk at its halo's centre: a and w (kModeAcc, part[4 k ..]) or S
// (kModePot, part[k]).  Bound by the loads: S of 11.7M particles (188 MB) in 28.7 us, 6.5
// TB/s, where 4096 particles per wavefront taken from a shared queue (k_soft_few) take
// 52 us: twice the wavefronts, none of them waiting for a counter.
template <int MODE>
__global__ __launch_bounds__(256) void k_centre_part(const float4* __restrict__ src,
                                                     const CentreDesc* __restrict__ halos,
                                                     const int* __restrict__ chunk_halo,
                                                     int n_chunks, const double* __restrict__ c,
                                                     const int* __restrict__ moving, float e2,
                                                     double* __restrict__ part) {
    constexpr int NQ = n_planes(MODE);
    const int lane = __lane_id();
    const int k = __builtin_amdgcn_readfirstlane(
        static_cast<int>(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave));
    if (k >= n_chunks) return;
    const int h = chunk_halo[k];
    if (moving && !moving[h]) return;
    const CentreDesc d = halos[h];
    const TestPt t = split_test(c[3 * h], c[3 * h + 1], c[3 * h + 2]);
    const int j0 = (k - d.first) * kChunk;
    const int last = min(d.src_len, j0 + kChunk) - 1;
    const float4* sp = src + d.src_off;
    float as[NQ], ac[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) as[q] = ac[q] = 0.0f;
    for (int j = j0 + lane; j - lane <= last; j += kSub * kWave) {
        float4 p[kSub];
#pragma unroll
        for (int s = 0; s < kSub; ++s) p[s] = sp[min(j + s * kWave, last)];
        float ps[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) ps[q] = 0.0f;
#pragma unroll
        for (int s = 0; s < kSub; ++s) {
            if (j + s * kWave > last) p[s].w = 0.0f;  // beyond the chunk: no mass
            pair_term<MODE, false>(ps, p[s], t, e2);
        }
#pragma unroll
        for (int q = 0; q < NQ; ++q) kahan(as[q], ac[q], ps[q]);
    }
    // lanes a and a ^ m add the same two values: every lane ends with the same total
    double v[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) v[q] = static_cast<double>(as[q]) + static_cast<double>(ac[q]);
#pragma unroll
    for (int m = kWave / 2; m >= 1; m >>= 1)
#pragma unroll
        for (int q = 0; q < NQ; ++q) v[q] = v[q] + __shfl_xor(v[q], m, kWave);
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) part[static_cast<int64_t>(k) * NQ + q] = v[q];
    }
}

// a halo's sums over its chunks: lane-strided, then the butterfly
template <int NQ>
__device__ __forceinline__ void halo_sums(const CentreDesc& d, const double* __restrict__ part,
                                          int lane, double v[NQ]) {
    const int nch = (d.src_len + kChunk - 1) / kChunk;
#pragma unroll
    for (int q = 0; q < NQ; ++q) v[q] = 0.0;
    for (int k = lane; k < nch; k += kWave)
#pragma unroll
        for (int q = 0; q < NQ; ++q) v[q] += part[static_cast<int64_t>(d.first + k) * NQ + q];
#pragma unroll
    for (int m = kWave / 2; m >= 1; m >>= 1)
#pragma unroll
        for (int q = 0; q < NQ; ++q) v[q] = v[q] + __shfl_xor(v[q], m, kWave);
}

// One wavefront per halo: the step of a moving halo, and whether it moves on; left[turn]
// counts the haloes that do, and the other word, whose count was copied to the host before
// this launch, is cleared for the next iteration.
__global__ __launch_bounds__(256) void k_centre_step(const CentreDesc* __restrict__ halos,
                                                     int n_halo, const double* __restrict__ part,
                                                     double limit, double* __restrict__ c,
                                                     int* __restrict__ moving,
                                                     int* __restrict__ iters,
                                                     double* __restrict__ steps,
                                                     int* __restrict__ left, int turn) {
    const int lane = __lane_id();
    const int h = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
    if (blockIdx.x == 0 && threadIdx.x == 0) left[turn ^ 1] = 0;
    if (h >= n_halo || !moving[h]) return;
    double v[4];
    halo_sums<4>(halos[h], part, lane, v);
    if (lane != 0) return;
    double s2 = 0.0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const double step = v[3] > 0.0 ? v[q] / v[3] : 0.0;
        c[3 * h + q] += step;
        s2 += step * step;
    }
    const double len = sqrt(s2);
    steps[h] = len;
    iters[h] += 1;
    const bool on = len > limit;
    moving[h] = on;
    if (on) atomicAdd(left + turn, 1);
}

__global__ __launch_bounds__(256) void k_centre_pot(const CentreDesc* __restrict__ halos,
                                                    int n_halo, const double* __restrict__ part,
                                                    double* __restrict__ S) {
    const int lane = __lane_id();
    const int h = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
    if (h >= n_halo) return;
    double v[1];
    halo_sums<1>(halos[h], part, lane, v);
    if (lane == 0) S[h] = v[0];
}

struct CentreWs {
    float4* src4;
    CentreDesc* halos;
    int* chunk_halo;
    double* part;
    int* moving;
    int* left;  // haloes still moving after iteration i, at i % 2
    size_t bytes;
};

int64_t centre_chunks(int64_t H, const int64_t* off) {
    int64_t n = 0;
    for (int64_t h = 0; h < H; ++h) n += (off[h + 1] - off[h] + kChunk - 1) / kChunk;
    return n;
}

CentreWs carve_centre(void* base, int64_t H, int64_t n, int64_t n_chunks) {
    Carver c(base);
    CentreWs w;
    w.src4 = c.take<float4>(std::max<int64_t>(n, 1));
    w.halos = c.take<CentreDesc>(std::max<int64_t>(H, 1));
    w.chunk_halo = c.take<int>(std::max<int64_t>(n_chunks, 1));
    w.part = c.take<double>(4 * std::max<int64_t>(n_chunks, 1));
    w.moving = c.take<int>(std::max<int64_t>(H, 1));
    w.left = c.take<int>(2);
    w.bytes = c.used;
    return w;
}

int check_centre(int64_t H, const int64_t* off, int max_iter) {
    if (H < 0 || !off || H > INT32_MAX || max_iter < 0)
        return set_error(HALMA_E_ARG, "halma_refine_centres: bad halo count, offsets or max_iter");
    for (int64_t h = 0; h < H; ++h) {
        if (off[h + 1] < off[h]) return set_error(HALMA_E_ARG, "offsets must not decrease");
        if (off[h + 1] - off[h] > INT32_MAX - kChunk)
            return set_error(HALMA_E_ARG, "halo %lld: too many particles",
                             static_cast<long long>(h));
    }
    if (H > 0 && centre_chunks(H, off) > INT32_MAX)
        return set_error(HALMA_E_LIMIT, "too many work items");
    return 0;
}

}  // namespace

}  // namespace halma

using namespace halma;

extern "C" {

size_t halma_refine_centres_workspace_size(int64_t n_halo, const int64_t* offsets, int max_iter) {
    if (check_centre(n_halo, offsets, max_iter)) return 0;
    if (n_halo == 0) return carve_centre(nullptr, 0, 0, 0).bytes;
    return carve_centre(nullptr, n_halo, offsets[n_halo] - offsets[0],
                        centre_chunks(n_halo, offsets))
        .bytes;
}

int halma_refine_centres(int64_t n_halo, const int64_t* offsets, const float* m, const float* x,
                         const float* y, const float* z, double eps, double tol, int max_iter,
                         double* centres, double* S, int32_t* iters, double* steps, void* ws,
                         size_t ws_bytes, void* stream) {
    int rc = check_centre(n_halo, offsets, max_iter);
    if (rc) return rc;
    if (!(eps >= 0.0) || !isfinite(eps)) return set_error(HALMA_E_ARG, "eps must be >= 0");
    if (n_halo == 0) return 0;
    const int64_t n = offsets[n_halo] - offsets[0], s0 = offsets[0];
    if (!centres || !S || !iters || !steps || (n > 0 && (!m || !x || !y || !z)))
        return set_error(HALMA_E_ARG, "halma_refine_centres: null pointer");
    const int64_t n_chunks = centre_chunks(n_halo, offsets);
    const int H = static_cast<int>(n_halo), nc = static_cast<int>(n_chunks);
    CentreWs w = carve_centre(ws, n_halo, n, n_chunks);
    if (!ws || ws_bytes < w.bytes)
        return set_error(HALMA_E_WORKSPACE, "workspace %zu < required %zu", ws_bytes, w.bytes);
    hipStream_t st = static_cast<hipStream_t>(stream);
    std::vector<CentreDesc> halos(static_cast<size_t>(n_halo));
    std::vector<int32_t> chunk_halo(static_cast<size_t>(n_chunks));
    int32_t at = 0;
    for (int h = 0; h < H; ++h) {
        CentreDesc& d = halos[h];
        d.src_off = offsets[h] - s0;
        d.src_len = static_cast<int32_t>(offsets[h + 1] - offsets[h]);
        d.first = at;
        for (int j = 0; j < d.src_len; j += kChunk) chunk_halo[at++] = h;
    }
    rc = upload_async(w.halos, halos.data(), halos.size() * sizeof(CentreDesc), st);
    if (!rc) rc = upload_async(w.chunk_halo, chunk_halo.data(), chunk_halo.size() * sizeof(int32_t), st);
    if (rc) return rc;
    if (n > 0) {
        k_centre_pack<<<static_cast<unsigned>((n + 255) / 256), 256, 0, st>>>(
            m + s0, x + s0, y + s0, z + s0, n, w.src4);
        HALMA_LAUNCH_CHECK();
    }
    k_centre_init<<<static_cast<unsigned>((n_halo + 256) / 256), 256, 0, st>>>(H, w.moving, iters,
                                                                               steps, w.left);
    HALMA_LAUNCH_CHECK();
    const float e2 = static_cast<float>(eps * eps);
    const unsigned gc = static_cast<unsigned>((n_chunks + 3) / 4);
    const unsigned gh = static_cast<unsigned>((n_halo + 3) / 4);
    long long* words = pinned_words(2);
    if (!words) return set_error(HALMA_E_STATE, "pinned host buffer unavailable");
    volatile int* host = reinterpret_cast<volatile int*>(words);
    hipEvent_t done[2] = {nullptr, nullptr};
    bool pending[2] = {false, false};
    hipError_t e = hipEventCreateWithFlags(&done[0], hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&done[1], hipEventDisableTiming);
    int launched = 0;
    for (int b = 0; e == hipSuccess && launched < max_iter; ++b) {
        const int q = b & 1;
        for (int i = 0; i < kBatch && launched < max_iter && e == hipSuccess; ++i, ++launched) {
            if (nc > 0)
                k_centre_part<kModeAcc><<<gc, 256, 0, st>>>(w.src4, w.halos, w.chunk_halo, nc,
                                                            centres, w.moving, e2, w.part);
            k_centre_step<<<gh, 256, 0, st>>>(w.halos, H, w.part, tol * eps, centres, w.moving,
                                              iters, steps, w.left, launched & 1);
            e = hipGetLastError();
        }
        if (e == hipSuccess)
            e = hipMemcpyAsync(const_cast<int*>(host) + q, w.left + ((launched - 1) & 1),
                               sizeof(int), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipEventRecord(done[q], st);
        if (e != hipSuccess) break;
        pending[q] = true;
        if (b > 0) {  // the batch before this one
            e = hipEventSynchronize(done[q ^ 1]);
            pending[q ^ 1] = false;
            if (e == hipSuccess && host[q ^ 1] == 0) break;
        }
    }
    // the words are this thread's next call's, too: no copy is left in flight
    for (int q = 0; q < 2; ++q) {
        if (pending[q]) {
            const hipError_t e1 = hipEventSynchronize(done[q]);
            if (e == hipSuccess) e = e1;
        }
        if (done[q]) (void)hipEventDestroy(done[q]);
    }
    if (e != hipSuccess) return hip_fail(e, "centring iteration", __FILE__, __LINE__);
    if (nc > 0) {
        k_centre_part<kModePot><<<gc, 256, 0, st>>>(w.src4, w.halos, w.chunk_halo, nc, centres,
                                                    nullptr, e2, w.part);
        HALMA_LAUNCH_CHECK();
    }
    k_centre_pot<<<gh, 256, 0, st>>>(w.halos, H, w.part, S);
    HALMA_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
