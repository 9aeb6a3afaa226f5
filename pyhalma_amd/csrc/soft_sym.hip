// Softened self sums of many haloes with the pair symmetry used: S_i and a_i of soft.hip
// over the halo's own members, each pair's differences, distance, rule and powers of 1/r
// evaluated once and its terms added to both members.
//
// A halo is cut into blocks of 64 T members; a work item is a pair of blocks (A, B),
// A <= B, taken by one wavefront.  The members of A are its tests, T per lane in registers;
// the members of B stream through as wave-uniform scalars, eight at a time:
//   - test side: FP32 sums of the eight terms, added in FP64 per test and quantity (two
//     instructions, where a Kahan sum takes four);
//   - source side: per source the T terms of a lane in FP32, then the fixed tree over the
//     lanes (reduce8), FP64 from the first level at T = 8, from the third at T = 2: eight
//     terms meet in FP32, as on the test side.  A holds every test of the item, so the total
//     is the item's and goes straight to its slot.
// A diagonal item (A == B) takes all its ordered pairs on the test side.  A member's sums
// of one item go to the slot of the other block (mod the band width), in FP64: slot B for
// the members of A, slot A for the members of B; k_soft_sym_merge adds a member's slots in
// slot order.  Haloes of more than kSsBand blocks run in tiles of kSsBand x kSsBand blocks,
// a launch and a merge per tile, so that a member needs kSsBand slots at most.
//
// T = 8 (blocks of 512) from kSsBig members on, T = 2 (blocks of 128) below: what the tree
// costs per pair falls with T, and a halo of kSsBig members has 528 items of T = 8, one for
// every second SIMD.  The choice depends on the halo's own size alone, so a member's result
// depends on its halo only.
//
// Bound by the FP32 vector ALUs: 23 issue slots per pair distance (3 differences, 3 for
// r^2, 3 for the rule, 2 for the reciprocal root, 2 for its cube, 2 + 8 for the sums of the
// two sides), 1 for the FP64 sums and 2.4 for the tree at T = 8 (1.6 with its first three
// levels in FP32, i.e. 64 terms instead of 8: six haloes of 2e4-2e5 members 18.2 instead of
// 19.0 ms a call, the spread of S 1.36 times the one-sided kernel's instead of 0.94), i.e. 13.2
// per ordered pair; the one-sided kernel of soft.hip takes 21.5.
#include <math.h>

#include <algorithm>
#include <vector>

#include "halma_common.h"
#include "potential.h"
#include "soft_pair.h"
#include "soft_sym.h"
#include "staging.h"
#include "sym.h"
#include "wave_reduce.h"

namespace halma {

namespace {

constexpr int kSsBand = 64;          // blocks per band
constexpr int kSsQueues = 8;         // queues of a launch's items, heads in lines of their own
constexpr int kSsHead = 16;
constexpr int kSsBig = 16384;        // members from which a halo is cut into blocks of 512
// Slot bytes of the haloes that share a launch, at 32 bytes a slot (room for S and a, whatever
// the call asks for): the workspace grows by 2 kB a member up to here and no further, and a
// halo that would need more is left to soft.hip (a quarter of the room makes 20 haloes of 1e5
// members 60 -> 68 ms in more launches, and one of 1e6 413 -> 516 in narrower bands).
constexpr size_t kSsSlots = size_t(4) << 30;
constexpr size_t kSsSlotBytes = 32;
constexpr int64_t kSsMax = static_cast<int64_t>(kSsSlots / (kSsSlotBytes * kSsBand));

// members rows[off, off + n); slot s, plane q of member i at
// part[q * n_part + part_off + s * n + i]
struct __attribute__((aligned(8))) SsDesc {
    int64_t off, part_off;
    int32_t n, nb, wb, bs;
};

// planes kept per member: S, or a (3), or both
__host__ __device__ constexpr int ss_planes(int mode) {
    return ((mode & kModePot) ? 1 : 0) + ((mode & kModeAcc) ? 3 : 0);
}

// Eight sources (cnt of them exist; kFull: all) against the lane's T tests.  kCols: the
// source side's terms pj too (a's with the sign of x_j - t_i, as the test side's).
template <int MODE, int T, bool kCols, bool kFull>
__device__ __forceinline__ void ss_group(const float4* __restrict__ q0, int cnt, float e2,
                                         const float* x, const float* y, const float* z,
                                         const float* m, double (*R)[4], float (*pj)[8]) {
    constexpr int A = (MODE & kModePot) ? 1 : 0;
    float4 src[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        src[s] = uniform_load(q0 + (kFull ? s : min(s, cnt - 1)));
        if (!kFull && s >= cnt) src[s].w = 0.0f;
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        float ps[4];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const float4 q = src[s];
            const float dx = q.x - x[t], dy = q.y - y[t], dz = q.z - z[t];
            const float mn = fminf(fminf(fabsf(dx), fabsf(dy)), fabsf(dz));
            const float d2 =
                __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, e2)));
            const float v = mn != 0.0f ? __builtin_amdgcn_rsqf(d2) : 0.0f;
            if (MODE & kModePot) {
                ps[0] = s == 0 ? q.w * v : __builtin_fmaf(q.w, v, ps[0]);
                if (kCols) pj[0][s] = t == 0 ? m[t] * v : __builtin_fmaf(m[t], v, pj[0][s]);
            }
            if (MODE & kModeAcc) {
                const float v3 = v * (v * v);
                const float f = q.w * v3;
                ps[A + 0] = s == 0 ? f * dx : __builtin_fmaf(f, dx, ps[A + 0]);
                ps[A + 1] = s == 0 ? f * dy : __builtin_fmaf(f, dy, ps[A + 1]);
                ps[A + 2] = s == 0 ? f * dz : __builtin_fmaf(f, dz, ps[A + 2]);
                if (kCols) {
                    const float g = m[t] * v3;
                    pj[A + 0][s] = t == 0 ? g * dx : __builtin_fmaf(g, dx, pj[A + 0][s]);
                    pj[A + 1][s] = t == 0 ? g * dy : __builtin_fmaf(g, dy, pj[A + 1][s]);
                    pj[A + 2][s] = t == 0 ? g * dz : __builtin_fmaf(g, dz, pj[A + 2][s]);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < ss_planes(MODE); ++q) R[t][q] += static_cast<double>(ps[q]);
        // a test's terms stay together: interleaved over the tests, their differences and
        // powers need more registers than two wavefronts per SIMD have
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Item k of a launch: its tile {halo, band P, band Q, first item} by bisection, and the
// block pair within it (B-major; a diagonal tile holds A <= B alone).
__device__ __forceinline__ void ss_item(const int4* __restrict__ tiles, int n_tiles,
                                        const SsDesc* __restrict__ halos, int k, SsDesc& d, int& A,
                                        int& B) {
    int lo = 0, hi = n_tiles - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (uniform_load(tiles + mid).w <= k) lo = mid;
        else hi = mid - 1;
    }
    const int4 t = uniform_load(tiles + lo);
    d = uniform_load(halos + t.x);
    const int r = k - t.w;
    const int a0 = t.y * d.wb, b0 = t.z * d.wb;
    if (t.y != t.z) {
        const int na = min(d.nb, a0 + d.wb) - a0;
        A = a0 + r % na;
        B = b0 + r / na;
    } else {  // r = b (b + 1) / 2 + a, a <= b
        int b = static_cast<int>((sqrtf(8.0f * static_cast<float>(r) + 1.0f) - 1.0f) * 0.5f);
        while (b * (b + 1) / 2 > r) --b;
        while ((b + 1) * (b + 2) / 2 <= r) ++b;
        A = a0 + (r - b * (b + 1) / 2);
        B = b0 + b;
    }
}

template <int MODE, int T>
__global__ __launch_bounds__(256, 2) void k_soft_sym(const float4* __restrict__ rows,
                                                  const SsDesc* __restrict__ halos,
                                                  const int4* __restrict__ tiles, int n_tiles,
                                                  int n_items, float e2, double* __restrict__ part,
                                                  int64_t n_part, int* __restrict__ head) {
    constexpr int NP = ss_planes(MODE);
    constexpr int A0 = (MODE & kModePot) ? 1 : 0;
    constexpr int kBlock = T * kWave;
    const int lane = __lane_id();
    const int n_waves = static_cast<int>(gridDim.x * (blockDim.x / kWave));
    // the items after the first ones from a queue, of blocks of 128 from kSsQueues of them in
    // turn: one queue's additions follow one another by 7 ns (300 haloes of 5000 members have
    // 246k: S 2.8 ms, 1.6 this way)
    const int nq = T == 8 ? 1 : min(kSsQueues, static_cast<int>(gridDim.x));
    const int queue = static_cast<int>(blockIdx.x) % nq;
    int k = __builtin_amdgcn_readfirstlane(
        static_cast<int>(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave));
    for (bool first = true;; first = false) {
        if (!first) {
            int t = 0;
            if (lane == 0) t = atomicAdd(head + kSsHead * queue, 1);
            k = n_waves + __builtin_amdgcn_readfirstlane(t) * nq + queue;
        }
        if (k >= n_items) break;
        SsDesc d;
        int A, B;
        ss_item(tiles, n_tiles, halos, k, d, A, B);
        const float4* sp = rows + d.off;
        float x[T], y[T], z[T], m[T];
        double R[T][4];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int i = A * kBlock + t * kWave + lane;
            const float4 p = sp[min(i, d.n - 1)];
            x[t] = p.x;
            y[t] = p.y;
            z[t] = p.z;
            m[t] = i < d.n ? p.w : 0.0f;  // padding lanes add nothing to sources
#pragma unroll
            for (int q = 0; q < 4; ++q) R[t][q] = 0.0;
        }
        const int j0 = B * kBlock;
        const int cnt = min(kBlock, d.n - j0);
        float pj[4][8];
        if (A == B) {
            int g = 0;
            for (; g + 8 <= cnt; g += 8)
                ss_group<MODE, T, false, true>(sp + j0 + g, 8, e2, x, y, z, m, R, pj);
            if (g < cnt)
                ss_group<MODE, T, false, false>(sp + j0 + g, cnt - g, e2, x, y, z, m, R, pj);
        } else {
            double* out = part + d.part_off + static_cast<int64_t>(A % d.wb) * d.n + j0;
            const int s = (lane >> 3) & 7;
            for (int g = 0; g < cnt; g += 8) {
                if (g + 8 <= cnt)
                    ss_group<MODE, T, true, true>(sp + j0 + g, 8, e2, x, y, z, m, R, pj);
                else
                    ss_group<MODE, T, true, false>(sp + j0 + g, cnt - g, e2, x, y, z, m, R, pj);
#pragma unroll
                for (int q = 0; q < NP; ++q) {
                    const double tot = reduce8<T == 8 ? 0 : 2>(pj[q], lane);
                    if ((lane & 7) == 0 && g + s < cnt)
                        out[q * n_part + g + s] = q < A0 ? tot : -tot;
                }
            }
        }
        double* out = part + d.part_off + static_cast<int64_t>(B % d.wb) * d.n;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int i = A * kBlock + t * kWave + lane;
            if (i < d.n)
#pragma unroll
                for (int q = 0; q < NP; ++q) out[q * n_part + i] = R[t][q];
        }
    }
}

// Segment {halo, first member, members, slots} of a tile, one plane per blockIdx.z: each
// member's slots 0 .. slots-1 added in order, eight in flight, and the sum added to (or,
// for a member's first tile, written to) its outputs.  Bound by reading the slots: six
// haloes of 2e4-2e5 members (3.1 GB) take 0.65 ms, 4.8 TB/s; with a quarter of the threads, each
// adding four members' planes in turn, 1.58 ms.
template <int MODE>
__global__ __launch_bounds__(256) void k_soft_sym_merge(const SsDesc* __restrict__ halos,
                                                        const int4* __restrict__ segs, int n_segs,
                                                        const double* __restrict__ part,
                                                        int64_t n_part, double* __restrict__ pot,
                                                        double* __restrict__ acc) {
    constexpr int A0 = (MODE & kModePot) ? 1 : 0;
    const int q = blockIdx.z;
    for (int sg = blockIdx.y; sg < n_segs; sg += gridDim.y) {
        const int4 g = segs[sg];
        const SsDesc d = halos[g.x];
        const int nloc = g.w & 0xffffff;
        const bool fresh = (g.w >> 24) != 0;
        for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < g.z;
             k += gridDim.x * blockDim.x) {
            const int64_t i = g.y + k;
            const int64_t o = d.off + i;
            const double* pp = part + q * n_part + d.part_off + i;
            double* to = q < A0 ? pot + o : acc + 3 * o + (q - A0);
            double sum = fresh ? 0.0 : *to;
            for (int c = 0; c < nloc; c += 8) {
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    v[u] = c + u < nloc ? pp[static_cast<int64_t>(c + u) * d.n] : 0.0;
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (c + u < nloc) sum += v[u];
            }
            *to = sum;
        }
    }
}

__global__ void k_soft_sym_clear(int* __restrict__ p, int64_t n) {
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x)
        p[i] = 0;
}

struct SsLaunch {
    bool big;
    int32_t tile0, n_tiles, n_items, seg0, n_segs;
};

struct SsPlan {
    std::vector<SsDesc> halos;
    std::vector<int4> tiles, segs;
    std::vector<SsLaunch> launches;
    int64_t n_part = 0;  // slots of the largest group of haloes
};

// a halo of n members from row `off` on
SsDesc ss_desc(int64_t n, int64_t off) {
    SsDesc d;
    d.off = off;
    d.part_off = 0;
    d.n = static_cast<int32_t>(std::min<int64_t>(n, INT32_MAX));  // larger: not taken
    d.bs = n >= kSsBig ? 512 : 128;
    d.nb = static_cast<int32_t>((n + d.bs - 1) / d.bs);
    d.wb = std::max(1, std::min(d.nb, kSsBand));
    return d;
}

int plan_ss(int64_t H, const int64_t* off, SsPlan& p) {
    p = SsPlan();
    p.halos.resize(static_cast<size_t>(H));
    std::vector<int64_t> key(static_cast<size_t>(H), 0);
    size_t taken = 0;
    for (int64_t h = 0; h < H; ++h) {
        const int64_t n = off[h + 1] - off[h];
        p.halos[h] = ss_desc(n, off[h] - off[0]);
        if (n == 0 || !soft_sym_takes(n)) continue;
        key[h] = n;
        ++taken;
    }
    std::vector<int32_t> order = order_desc(key);
    order.resize(taken);
    size_t at = 0;
    while (at < order.size()) {
        // a group: haloes of one block size whose slots (at most four planes) fit together
        const bool big = p.halos[order[at]].bs == 512;
        size_t end = at;
        int64_t slots = 0;
        while (end < order.size()) {
            SsDesc& d = p.halos[order[end]];
            const int64_t s = static_cast<int64_t>(d.wb) * d.n;
            if ((d.bs == 512) != big) break;
            if (end > at && static_cast<size_t>(slots + s) * kSsSlotBytes > kSsSlots) break;
            d.part_off = slots;
            slots += s;
            ++end;
        }
        p.n_part = std::max(p.n_part, slots);
        const SsDesc& d0 = p.halos[order[at]];
        const int64_t K0 = (d0.nb + d0.wb - 1) / d0.wb;
        int P = 0, Q = 0;
        for (int64_t t = 0; t < K0 * (K0 + 1) / 2; ++t) {  // t = Q (Q + 1) / 2 + P
            SsLaunch l{big, static_cast<int32_t>(p.tiles.size()), 0, 0,
                       static_cast<int32_t>(p.segs.size()), 0};
            int64_t items = 0;
            for (size_t q = at; q < end; ++q) {
                const int32_t h = order[q];
                const SsDesc& d = p.halos[h];
                if (Q * d.wb >= d.nb) break;  // the haloes shrink
                const int na = std::min(d.nb, (P + 1) * d.wb) - P * d.wb;
                const int nq = std::min(d.nb, (Q + 1) * d.wb) - Q * d.wb;
                p.tiles.push_back(make_int4(h, P, Q, static_cast<int>(items)));
                items += P == Q ? static_cast<int64_t>(nq) * (nq + 1) / 2
                                : static_cast<int64_t>(na) * nq;
                auto seg = [&](int band, int nloc, bool fresh) {
                    const int64_t m0 = static_cast<int64_t>(band) * d.wb * d.bs;
                    const int64_t m1 = std::min<int64_t>(d.n, m0 + static_cast<int64_t>(d.wb) * d.bs);
                    p.segs.push_back(make_int4(h, static_cast<int>(m0), static_cast<int>(m1 - m0),
                                               (fresh ? 1 << 24 : 0) | nloc));
                };
                // a band's first tile is (0, Q) for the members of Q; band 0's is (0, 0)
                if (P == Q) {
                    seg(P, nq, Q == 0);
                } else {
                    seg(P, nq, false);
                    seg(Q, na, P == 0);
                }
            }
            if (items > INT32_MAX) return set_error(HALMA_E_LIMIT, "too many work items");
            l.n_tiles = static_cast<int32_t>(p.tiles.size()) - l.tile0;
            l.n_items = static_cast<int32_t>(items);
            l.n_segs = static_cast<int32_t>(p.segs.size()) - l.seg0;
            p.launches.push_back(l);
            if (++P > Q) {
                ++Q;
                P = 0;
            }
        }
        at = end;
    }
    return 0;
}

struct SsWs {
    SsDesc* halos;
    int4* tiles;
    int4* segs;
    int* heads;
    double* part;
    size_t bytes;
};

SsWs carve_ss(void* base, size_t halos, size_t tiles, size_t segs, size_t launches,
              int64_t n_part) {
    Carver c(base);
    SsWs w;
    w.halos = c.take<SsDesc>(std::max<size_t>(halos, 1));
    w.tiles = c.take<int4>(std::max<size_t>(tiles, 1));
    w.segs = c.take<int4>(std::max<size_t>(segs, 1));
    w.heads = c.take<int>(kSsQueues * kSsHead * std::max<size_t>(launches, 1));
    w.part = c.take<double>(4 * static_cast<size_t>(std::max<int64_t>(n_part, 1)));
    w.bytes = c.used;
    return w;
}

template <int MODE>
int launch_ss(const SsPlan& p, const SsWs& w, const float4* rows, float e2, double* pot,
              double* acc, hipStream_t st) {
    const int cus = std::max(device_cu_count(), 1);
    k_soft_sym_clear<<<16, 256, 0, st>>>(
        w.heads, static_cast<int64_t>(kSsQueues * kSsHead) * static_cast<int64_t>(p.launches.size()));
    HALMA_LAUNCH_CHECK();
    for (size_t q = 0; q < p.launches.size(); ++q) {
        const SsLaunch& l = p.launches[q];
        const int blocks = (l.n_items + 3) / 4;
        if (l.big)
            k_soft_sym<MODE, 8><<<std::min(blocks, cus * 2), 256, 0, st>>>(
                rows, w.halos, w.tiles + l.tile0, l.n_tiles, l.n_items, e2, w.part, p.n_part,
                w.heads + kSsQueues * kSsHead * q);
        else
            k_soft_sym<MODE, 2><<<std::min(blocks, cus * 4), 256, 0, st>>>(
                rows, w.halos, w.tiles + l.tile0, l.n_tiles, l.n_items, e2, w.part, p.n_part,
                w.heads + kSsQueues * kSsHead * q);
        HALMA_LAUNCH_CHECK();
        const dim3 grid(merge_width(p.segs.data() + l.seg0, l.n_segs),
                        static_cast<unsigned>(std::min(l.n_segs, 65535)), ss_planes(MODE));
        k_soft_sym_merge<MODE><<<grid, 256, 0, st>>>(w.halos, w.segs + l.seg0, l.n_segs, w.part,
                                                     p.n_part, pot, acc);
        HALMA_LAUNCH_CHECK();
    }
    return 0;
}

}  // namespace

bool soft_sym_takes(int64_t n) { return n <= kSsMax; }

size_t soft_sym_bytes(int64_t H, const int64_t* off) {
    // at least what the plan needs, without its tables: a group of haloes fits kSsSlots, two
    // after one another would not, and a group's largest halo has no more bands than any
    size_t tiles = 0, segs = 0, bands[2] = {0, 0};
    int64_t slots[2] = {0, 0};
    for (int64_t h = 0; h < H; ++h) {
        const SsDesc d = ss_desc(off[h + 1] - off[h], 0);
        if (d.n == 0 || !soft_sym_takes(d.n)) continue;
        const size_t K = static_cast<size_t>((d.nb + d.wb - 1) / d.wb);
        tiles += K * (K + 1) / 2;
        segs += K * K;
        slots[d.bs == 512] += static_cast<int64_t>(d.wb) * d.n;
        bands[d.bs == 512] = std::max(bands[d.bs == 512], K);
    }
    const int64_t room = static_cast<int64_t>(kSsSlots / kSsSlotBytes);
    size_t launches = 0;
    for (int c = 0; c < 2; ++c)
        launches += (static_cast<size_t>(2 * slots[c] / room) + 1) * (bands[c] * (bands[c] + 1) / 2);
    return carve_ss(nullptr, static_cast<size_t>(H), tiles, segs, std::min(launches, tiles),
                    std::min(std::max(slots[0], slots[1]), room))
        .bytes;
}

int soft_sym_run(int64_t H, const int64_t* off, const float4* rows, float e2, double* pot,
                 double* acc, void* ws, size_t ws_bytes, hipStream_t st) {
    SsPlan p;
    int rc = plan_ss(H, off, p);
    if (rc) return rc;
    SsWs w = carve_ss(ws, p.halos.size(), p.tiles.size(), p.segs.size(), p.launches.size(), p.n_part);
    if (ws_bytes < w.bytes)
        return set_error(HALMA_E_WORKSPACE, "workspace %zu < required %zu", ws_bytes, w.bytes);
    rc = upload_async(w.halos, p.halos.data(), p.halos.size() * sizeof(SsDesc), st);
    if (!rc) rc = upload_async(w.tiles, p.tiles.data(), p.tiles.size() * sizeof(int4), st);
    if (!rc) rc = upload_async(w.segs, p.segs.data(), p.segs.size() * sizeof(int4), st);
    if (rc) return rc;
    if (p.launches.empty()) return 0;
    if (pot && acc) return launch_ss<kModeBoth>(p, w, rows, e2, pot, acc, st);
    if (pot) return launch_ss<kModePot>(p, w, rows, e2, pot, nullptr, st);
    return launch_ss<kModeAcc>(p, w, rows, e2, nullptr, acc, st);
}

}  // namespace halma
