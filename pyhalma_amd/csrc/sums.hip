// Per-halo sums over CSR ranges in double-double: the four masses of the ram-pressure energy
// test (halo_gas.py:466-489) and the mass-weighted sum of a per-member value (the potential
// energy of the centring).
//
// A halo is cut into chunks of kChunk members, a wavefront each (lanes in stride, a fixed
// butterfly), and a wavefront per halo adds the chunks' sums: two launches, every value read
// once.  Bound by the chain of double-double additions of a lane (32 of each sum): 24 gas
// haloes of 1e3-2e5 cells take 44 us (one weighted sum over 6 haloes of up to 2e5: 28 us);
// the masked masses as tensor expressions with a group reduction each (one workgroup for a
// halo, positions and extents summed along) took 1.2 ms, the weighted sum 240 us.
#include <algorithm>
#include <vector>

#include "halma_common.h"
#include "staging.h"

namespace halma {

namespace {

constexpr int kChunk = 2048;
constexpr int kThreads = 256;

struct __attribute__((aligned(8))) SumDesc {
    int64_t off;
    int32_t len, first;  // members, first chunk
};

struct SumArgs {
    const void* m;
    int m_t;
    const void* temp;
    int temp_t;
    const uint8_t* bound;
    const double* s;
};

__device__ __forceinline__ void wave_dd(double (&v)[2]) {
    for (int m = kWave / 2; m >= 1; m >>= 1) {
        const double h2 = __shfl_xor(v[0], m, kWave), l2 = __shfl_xor(v[1], m, kWave);
        // both lanes of a pair add the lower lane's sum and then the upper one's
        if (__lane_id() & m) {
            double h = h2, l = l2;
            dd_add_dd(h, l, v[0], v[1]);
            v[0] = h;
            v[1] = l;
        } else {
            dd_add_dd(v[0], v[1], h2, l2);
        }
    }
}

// NQ = 4: all, cold and bound, cold and not bound, hot and not bound masses (cold: T < 5e4,
// hot: not cold); NQ = 1: sum m s
template <int NQ>
__global__ __launch_bounds__(kThreads) void k_sums_part(const SumDesc* __restrict__ halos,
                                                        const int* __restrict__ chunk_halo,
                                                        int n_chunks, SumArgs a,
                                                        double* __restrict__ part) {
    const int lane = __lane_id();
    const int c = static_cast<int>((blockIdx.x * blockDim.x + threadIdx.x) / kWave);
    if (c >= n_chunks) return;
    const SumDesc d = halos[chunk_halo[c]];
    const int j0 = (c - d.first) * kChunk, j1 = min(d.len, j0 + kChunk);
    double acc[NQ][2];
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[q][0] = acc[q][1] = 0.0;
    for (int j = j0 + lane; j < j1; j += 4 * kWave) {
        double m[4], t[4];
        bool b[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = j + u * kWave;
            const int64_t i = d.off + (k < j1 ? k : j1 - 1);
            m[u] = ldf(a.m, a.m_t, i);
            t[u] = NQ == 4 ? ldf(a.temp, a.temp_t, i) : a.s[i];
            b[u] = NQ == 4 && a.bound[i] != 0;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (j + u * kWave >= j1) break;
            if constexpr (NQ == 4) {
                const bool cold = t[u] < 5 * 1e4;
                dd_add(acc[0][0], acc[0][1], m[u]);
                dd_add(acc[1][0], acc[1][1], cold && b[u] ? m[u] : 0.0);
                dd_add(acc[2][0], acc[2][1], cold && !b[u] ? m[u] : 0.0);
                dd_add(acc[3][0], acc[3][1], !cold && !b[u] ? m[u] : 0.0);
            } else {
                dd_add(acc[0][0], acc[0][1], m[u] * t[u]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        wave_dd(acc[q]);
        if (lane == 0) {
            part[(static_cast<int64_t>(c) * NQ + q) * 2] = acc[q][0];
            part[(static_cast<int64_t>(c) * NQ + q) * 2 + 1] = acc[q][1];
        }
    }
}

template <int NQ>
__global__ __launch_bounds__(kThreads) void k_sums_halo(const SumDesc* __restrict__ halos,
                                                        int n_halo,
                                                        const double* __restrict__ part,
                                                        double* __restrict__ out) {
    const int lane = __lane_id();
    const int h = static_cast<int>((blockIdx.x * blockDim.x + threadIdx.x) / kWave);
    if (h >= n_halo) return;
    const SumDesc d = halos[h];
    const int nch = (d.len + kChunk - 1) / kChunk;
    double v[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        double acc[2] = {0.0, 0.0};
        for (int c = lane; c < nch; c += kWave) {
            const double* p = part + (static_cast<int64_t>(d.first + c) * NQ + q) * 2;
            dd_add_dd(acc[0], acc[1], p[0], p[1]);
        }
        wave_dd(acc);
        v[q] = acc[0] + acc[1];
    }
    if (lane != 0) return;
    if constexpr (NQ == 4) v[1] = v[0] != 0.0 ? v[1] / v[0] : 0.0;  // cold bound fraction
#pragma unroll
    for (int q = 0; q < NQ; ++q) out[static_cast<int64_t>(h) * NQ + q] = v[q];
}

struct SumWs {
    SumDesc* halos;
    int* chunk_halo;
    double* part;
    size_t bytes;
};

int64_t sum_chunks(int64_t H, const int64_t* off) {
    int64_t n = 0;
    for (int64_t h = 0; h < H; ++h) n += (off[h + 1] - off[h] + kChunk - 1) / kChunk;
    return n;
}

SumWs carve_sums(void* base, int64_t H, int64_t n_chunks) {
    Carver c(base);
    SumWs w;
    w.halos = c.take<SumDesc>(std::max<int64_t>(H, 1));
    w.chunk_halo = c.take<int>(std::max<int64_t>(n_chunks, 1));
    w.part = c.take<double>(8 * std::max<int64_t>(n_chunks, 1));
    w.bytes = c.used;
    return w;
}

int check_sums(int64_t H, const int64_t* off) {
    if (H < 0 || !off || H > INT32_MAX)
        return set_error(HALMA_E_ARG, "halo sums: bad halo count or offsets");
    for (int64_t h = 0; h < H; ++h)
        if (off[h + 1] < off[h] || off[h + 1] - off[h] > INT32_MAX - kChunk)
            return set_error(HALMA_E_ARG, "halo sums: offsets must not decrease");
    if (H > 0 && sum_chunks(H, off) > INT32_MAX)
        return set_error(HALMA_E_LIMIT, "too many work items");
    return 0;
}

template <int NQ>
int run_sums(int64_t H, const int64_t* off, const SumArgs& a, double* out, void* ws,
             size_t ws_bytes, hipStream_t st) {
    const int64_t n_chunks = sum_chunks(H, off);
    SumWs w = carve_sums(ws, H, n_chunks);
    if (!ws || ws_bytes < w.bytes)
        return set_error(HALMA_E_WORKSPACE, "workspace %zu < required %zu", ws_bytes, w.bytes);
    std::vector<SumDesc> halos(static_cast<size_t>(H));
    std::vector<int32_t> map(static_cast<size_t>(n_chunks));
    int32_t at = 0;
    for (int64_t h = 0; h < H; ++h) {
        halos[h] = {off[h], static_cast<int32_t>(off[h + 1] - off[h]), at};
        for (int64_t j = off[h]; j < off[h + 1]; j += kChunk) map[at++] = static_cast<int32_t>(h);
    }
    int rc = upload_async(w.halos, halos.data(), halos.size() * sizeof(SumDesc), st);
    if (!rc) rc = upload_async(w.chunk_halo, map.data(), map.size() * sizeof(int32_t), st);
    if (rc) return rc;
    if (n_chunks > 0) {
        k_sums_part<NQ><<<static_cast<unsigned>((n_chunks + 3) / 4), kThreads, 0, st>>>(
            w.halos, w.chunk_halo, static_cast<int>(n_chunks), a, w.part);
        HALMA_LAUNCH_CHECK();
    }
    k_sums_halo<NQ><<<static_cast<unsigned>((H + 3) / 4), kThreads, 0, st>>>(
        w.halos, static_cast<int>(H), w.part, out);
    HALMA_LAUNCH_CHECK();
    return 0;
}

}  // namespace

}  // namespace halma

using namespace halma;

extern "C" {

size_t halma_halo_sums_workspace_size(int64_t n_halo, const int64_t* offsets) {
    if (check_sums(n_halo, offsets)) return 0;
    return carve_sums(nullptr, n_halo, n_halo > 0 ? sum_chunks(n_halo, offsets) : 0).bytes;
}

int halma_gas_masses(int64_t n_halo, const int64_t* offsets, const void* m, int m_dtype,
                     const void* temp, int temp_dtype, const uint8_t* bound, double* out,
                     void* ws, size_t ws_bytes, void* stream) {
    int rc = check_sums(n_halo, offsets);
    if (rc) return rc;
    if ((m_dtype != HALMA_F32 && m_dtype != HALMA_F64) ||
        (temp_dtype != HALMA_F32 && temp_dtype != HALMA_F64))
        return set_error(HALMA_E_ARG, "bad dtype");
    if (n_halo == 0) return 0;
    if (!out || (offsets[n_halo] > offsets[0] && (!m || !temp || !bound)))
        return set_error(HALMA_E_ARG, "halma_gas_masses: null pointer");
    const SumArgs a{m, m_dtype, temp, temp_dtype, bound, nullptr};
    return run_sums<4>(n_halo, offsets, a, out, ws, ws_bytes, static_cast<hipStream_t>(stream));
}

int halma_weighted_sums(int64_t n_halo, const int64_t* offsets, const void* m, int m_dtype,
                        const double* s, double* out, void* ws, size_t ws_bytes, void* stream) {
    int rc = check_sums(n_halo, offsets);
    if (rc) return rc;
    if (m_dtype != HALMA_F32 && m_dtype != HALMA_F64) return set_error(HALMA_E_ARG, "bad dtype");
    if (n_halo == 0) return 0;
    if (!out || (offsets[n_halo] > offsets[0] && (!m || !s)))
        return set_error(HALMA_E_ARG, "halma_weighted_sums: null pointer");
    const SumArgs a{m, m_dtype, nullptr, HALMA_F64, nullptr, s};
    return run_sums<1>(n_halo, offsets, a, out, ws, ws_bytes, static_cast<hipStream_t>(stream));
}

}  // extern "C"
