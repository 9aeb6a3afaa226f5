// Self-potential of many haloes with the pair symmetry used: S_i = sum_{j != i} m_j / r_ij
// over the halo's own members (the sum of particle_subroutines.f90:466-514 with tests =
// sources, as the unbinding's full passes need), each pair distance computed once and
// its two terms, m_j / r to S_i and m_i / r to S_j, accumulated together.
//
// A halo of n members is cut into blocks of kBlock = 512 members.  A work item is a pair of
// blocks (A, B), A <= B.  The members of A are the tests, kTests = 8 per lane in registers
// (test strip t: members 64 t .. 64 t + 63 of A); the members of B stream through as
// wave-uniform sources, eight at a time, in segments of kSeg = 32:
//   - test side: per test an FP32 sum of the eight terms, added in FP64 over the segment,
//     the segments' sums in FP64 in order;
//   - source side: per source two FP32 chains over a lane's tests 0-3 and 4-7, their sum
//     through a fixed tree over the lanes (reduce8, its last three levels in FP64).  The lanes
//     hold every test of the item, so the total goes straight to the member's slot.
// In a diagonal item (A == B) a source of strip s meets the strips t < s on both sides and
// strip s on the test side alone (all its ordered pairs); the strips above it are another
// source's.  Every member then has partial sums in nb + 1 slots (nb = blocks of its halo),
// each written by exactly one item: slot s < I (its block) from the source side of item
// (s, I), slot I from the test side of item (I, I), slots s > I from the test side of item
// (I, s), and slot nb from the source side of item (I, I).  The slots are merged in FP64 in
// slot order.
//
// A launch of kWaveItems items or more gives each item to a wavefront, which takes its
// segments in turn; one with fewer (a lone halo, the later passes of an unbinding) to a
// workgroup of sixteen wavefronts, a segment each, whose test sums meet in LDS and are
// added in segment order.  The same operations in the same order: a halo's sums do not
// depend on the other haloes of the call.
//
// Bound by the FP32 vector ALUs.  Per pair distance 11.5 issue slots (3 differences, 3 for
// r^2, 1.5 for the coordinate rule, 2 for the reciprocal root, 2 sums), 0.25 for the FP64
// sums, 0.5 for the two chains and the tree.  The rule is a running minimum of the
// |differences| of a strip's eight pairs per lane, one compare and a branch; the branch's
// side evaluates the rule pair by pair (a tenth of the eights in the clumps' FP32
// coordinates).  Pair by pair for all of them costs 3 slots.  The clump step's launches (8.0e9
// distances in the first) 2.80 -> 2.46 ms, the gas step's 16.8 -> 14.6 ms against two tests
// per lane with Kahan sums, the pair-by-pair rule and a tree per 128 tests.
#include <math.h>

#include <algorithm>
#include <vector>

#include "halma_common.h"
#include "potential.h"
#include "staging.h"
#include "sym.h"
#include "tuning.h"
#include "wave_reduce.h"

namespace halma {

namespace {

constexpr int kTests = 8;                 // tests per lane
constexpr int kBlock = kTests * kWave;    // members of a block
constexpr int kSeg = 32;                  // sources of a segment
constexpr int kSegs = kBlock / kSeg;
static_assert(kBlock == 128 * kSymK, "blocks of the plans");

// Below this many items a launch gives each to a workgroup (k_pot_sym_fine): the clump step
// (33k items in the first pass) is the same from 1024 to 8192, the bridged pairs' later passes
// (1-8k items) take 8.2 ms at 1024, 8.0 at 2048, 7.6 at 4096, 7.9 at 8192
constexpr int kWaveItems = 4096;

struct SymTests {
    float x[kTests], y[kTests], z[kTests], m[kTests];
};

__device__ __forceinline__ void load_tests(const float4* __restrict__ sp, int i0, int n, int lane,
                                           SymTests& T) {
#pragma unroll
    for (int t = 0; t < kTests; ++t) {
        const int i = i0 + t * kWave + lane;
        const float4 p = sp[min(i, n - 1)];
        T.x[t] = p.x;
        T.y[t] = p.y;
        T.z[t] = p.z;
        T.m[t] = i < n ? p.w : 0.0f;  // padding lanes add nothing to sources
    }
}

// Eight sources (cnt of them exist; kFull: all of them): strips t < lim on both sides, strip
// lim on the test side.  R: the tests' FP64 sums of the segment.  Returns the source side's
// total of source (lane >> 3) & 7, valid in the lanes with lane % 8 == 0.
template <bool kFull>
__device__ __forceinline__ double sym_group(const float4* __restrict__ q0, int cnt, int lim,
                                           const SymTests& T, double R[kTests], int lane) {
    float4 q[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        q[s] = uniform_load(q0 + (kFull ? s : min(s, cnt - 1)));
        if (!kFull && s >= cnt) q[s].w = 0.0f;
    }
    float p[2][8];
#pragma unroll
    for (int s = 0; s < 8; ++s) p[0][s] = p[1][s] = 0.0f;
#pragma unroll
    for (int t = 0; t < kTests; ++t) {
        if (t <= lim) {
            float v[8];
            inv_r_group<8>(q, T.x[t], T.y[t], T.z[t], v);
            float ps = q[0].w * v[0];
#pragma unroll
            for (int s = 1; s < 8; ++s) ps = __builtin_fmaf(q[s].w, v[s], ps);
            R[t] += static_cast<double>(ps);
            if (t < lim) {
#pragma unroll
                for (int s = 0; s < 8; ++s)
                    p[t / 4][s] = __builtin_fmaf(T.m[t], v[s], p[t / 4][s]);
            }
        }
        // a strip's terms stay together (registers)
        __builtin_amdgcn_sched_barrier(0);
    }
    if (lim == 0) return 0.0;
#pragma unroll
    for (int s = 0; s < 8; ++s) p[0][s] += p[1][s];
    return reduce8<3>(p[0], lane);
}

// Sources j0 .. j0 + cnt - 1 (a segment) of item (A, B): the source side to its slot (out,
// by member), the test side to R.
__device__ __forceinline__ void sym_segment(const float4* __restrict__ sp, int j0, int cnt,
                                            int lim, const SymTests& T, double R[kTests],
                                            float2* __restrict__ out, int lane) {
    const int s = (lane >> 3) & 7;
    for (int g = 0; g < cnt; g += 8) {
        const double tot = g + 8 <= cnt ? sym_group<true>(sp + j0 + g, 8, lim, T, R, lane)
                                        : sym_group<false>(sp + j0 + g, cnt - g, lim, T, R, lane);
        if ((lane & 7) == 0 && g + s < cnt) out[j0 + g + s] = split_sum(tot);
    }
}

struct SymItem {
    const float4* sp;  // the halo's members
    float2* pp;        // its slots
    int64_t stride;    // slots are laid out for the planned size
    int n, A, B, tslot, sslot;
    bool ok;
};

__device__ __forceinline__ SymItem sym_item(const float4* __restrict__ src,
                                            const SymDesc* __restrict__ halos,
                                            const int* __restrict__ live_n,
                                            const int4* __restrict__ items, int k,
                                            float2* __restrict__ part) {
    const int4 it = uniform_load(items + k);
    const SymDesc d = uniform_load(halos + it.x);
    SymItem r;
    r.n = live_n ? __builtin_amdgcn_readfirstlane(uniform_load(live_n + it.x)) : d.n;
    const int nb = (r.n + kBlock - 1) / kBlock;
    r.A = it.y;
    r.B = it.z;
    r.ok = r.B < nb && r.A <= r.B;
    r.sp = src + d.off;
    r.pp = part + d.part_off;
    r.stride = d.n;
    // test side: slot B (mod the band width); source side: slot A, or the diagonal slot
    r.tslot = r.B % d.wb;
    r.sslot = r.A < r.B ? r.A % d.wb : min(d.wb, nb);
    return r;
}

__global__ __launch_bounds__(256, 4) void k_pot_sym(const float4* __restrict__ src,
                                                 const SymDesc* __restrict__ halos,
                                                 const int* __restrict__ live_n,
                                                 const int4* __restrict__ items, int n_items,
                                                 const int64_t* __restrict__ n_items_dev,
                                                 float2* __restrict__ part,
                                                 int* __restrict__ head) {
    const int lane = __lane_id();
    if (n_items_dev) {
        const int64_t nd = uniform_load(n_items_dev);
        n_items = static_cast<int>(nd < n_items ? nd : n_items);
    }
    if (n_items < kWaveItems) return;  // k_pot_sym_fine takes the launch
    const int n_waves = static_cast<int>(gridDim.x * (blockDim.x / kWave));
    int k = __builtin_amdgcn_readfirstlane(
        static_cast<int>(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave));
    for (bool first = true;; first = false) {
        if (!first) {
            int t = 0;
            if (lane == 0) t = atomicAdd(head, 1);
            k = n_waves + __builtin_amdgcn_readfirstlane(t);
        }
        if (k >= n_items) break;
        const SymItem it = sym_item(src, halos, live_n, items, k, part);
        if (!it.ok) continue;
        SymTests T;
        load_tests(it.sp, it.A * kBlock, it.n, lane, T);
        double S[kTests];
#pragma unroll
        for (int t = 0; t < kTests; ++t) S[t] = 0.0;
        float2* out = it.pp + static_cast<int64_t>(it.sslot) * it.stride;
        const int j1 = min(it.n, (it.B + 1) * kBlock);
        int sg = 0;
        for (int j0 = it.B * kBlock; j0 < j1; j0 += kSeg, ++sg) {
            double R[kTests];
#pragma unroll
            for (int t = 0; t < kTests; ++t) R[t] = 0.0;
            sym_segment(it.sp, j0, min(kSeg, j1 - j0),
                        it.A == it.B ? sg * kSeg / kWave : kTests, T, R, out, lane);
#pragma unroll
            for (int t = 0; t < kTests; ++t) S[t] += R[t];
        }
        out = it.pp + static_cast<int64_t>(it.tslot) * it.stride;
#pragma unroll
        for (int t = 0; t < kTests; ++t) {
            const int i = it.A * kBlock + t * kWave + lane;
            if (i < it.n) out[i] = split_sum(S[t]);
        }
    }
}

// One item per workgroup of sixteen wavefronts, a segment each.
__global__ __launch_bounds__(1024) void k_pot_sym_fine(const float4* __restrict__ src,
                                                       const SymDesc* __restrict__ halos,
                                                       const int* __restrict__ live_n,
                                                       const int4* __restrict__ items,
                                                       int n_items,
                                                       const int64_t* __restrict__ n_items_dev,
                                                       float2* __restrict__ part,
                                                       int* __restrict__ head) {
    static_assert(kSegs * kWave == 1024, "one wavefront per segment of an item");
    __shared__ double seg[kSegs][kBlock];  // 64 KiB
    __shared__ int next_item;
    if (n_items_dev) {
        const int64_t nd = uniform_load(n_items_dev);
        n_items = static_cast<int>(nd < n_items ? nd : n_items);
    }
    if (n_items >= kWaveItems) return;  // k_pot_sym takes the launch
    const int lane = __lane_id();
    const int sg = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
    int k = static_cast<int>(blockIdx.x);
    for (bool first = true;; first = false) {
        if (!first) {
            __syncthreads();  // the previous item's LDS has been read
            if (threadIdx.x == 0) next_item = atomicAdd(head, 1);
            __syncthreads();
            k = static_cast<int>(gridDim.x) + __builtin_amdgcn_readfirstlane(next_item);
        }
        if (k >= n_items) break;
        const SymItem it = sym_item(src, halos, live_n, items, k, part);
        if (!it.ok) continue;  // the same for the whole workgroup
        const int j0 = it.B * kBlock + sg * kSeg;
        const int cnt = min(kSeg, it.n - j0);
        if (cnt > 0) {
            SymTests T;
            load_tests(it.sp, it.A * kBlock, it.n, lane, T);
            double R[kTests];
#pragma unroll
            for (int t = 0; t < kTests; ++t) R[t] = 0.0;
            sym_segment(it.sp, j0, cnt, it.A == it.B ? sg * kSeg / kWave : kTests, T, R,
                        it.pp + static_cast<int64_t>(it.sslot) * it.stride, lane);
#pragma unroll
            for (int t = 0; t < kTests; ++t) seg[sg][t * kWave + lane] = R[t];
        }
        __syncthreads();
        const int n_segs = min(kSegs, (it.n - it.B * kBlock + kSeg - 1) / kSeg);
        const int e = threadIdx.x, i = it.A * kBlock + e;
        if (e < kBlock && i < it.n) {
            double S = 0.0;
            for (int g = 0; g < n_segs; ++g) S += seg[g][e];
            it.pp[static_cast<int64_t>(it.tslot) * it.stride + i] = split_sum(S);
        }
    }
}

// The slots of one tile launch added into each affected member's FP64 sum (out, cleared
// before the first launch): segment s = {halo, first member, count, role << 24 | local
// slots}; the member adds its local slots 0 .. nloc - 1 in order, then, on a diagonal
// tile, the diagonal slot.  With one band a member's slots 0..nb are added in order.  Bound
// by reading the slots: up to 128 workgroups to a segment (merge_width), since a launch of few
// large haloes has few segments (24 gas haloes of 1e3-2e5 cells: 62 -> 22.6 us a launch against 32
// for every segment); as many for each of 20000 haloes of 100 members, nearly all without a
// member, took 555 us, 32 took 330, the one that they need 20.
__global__ __launch_bounds__(256) void k_sym_merge_tile(const SymDesc* __restrict__ halos,
                                                        const int4* __restrict__ segs, int nseg,
                                                        const int64_t* __restrict__ member_base,
                                                        const float2* __restrict__ part,
                                                        double* __restrict__ out) {
    for (int s = blockIdx.y; s < nseg; s += gridDim.y) {
        const int4 sg = segs[s];
        const SymDesc d = halos[sg.x];
        const int nloc = sg.w & 0xffffff;
        const bool diag = (sg.w >> 24) == 2;
        for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < sg.z; k += gridDim.x * blockDim.x) {
            const int64_t i = sg.y + k;
            const float2* pp = part + d.part_off + i;
            const int64_t g = member_base[sg.x] + i;
            double acc = out[g];
            for (int c = 0; c < nloc; c += 8) {
                float2 q[8];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    q[u] = c + u < nloc ? pp[static_cast<int64_t>(c + u) * d.n]
                                        : make_float2(0.0f, 0.0f);
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (c + u < nloc) acc += static_cast<double>(q[u].x) + static_cast<double>(q[u].y);
            }
            if (diag) {
                const float2 q = pp[static_cast<int64_t>(min(d.wb, d.nb)) * d.n];
                acc += static_cast<double>(q.x) + static_cast<double>(q.y);
            }
            out[g] = acc;
        }
    }
}

__global__ void k_sym_zero(double* __restrict__ p, int64_t n) {
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x)
        p[i] = 0.0;
}

__global__ void k_sym_pack(const float* __restrict__ m, const float* __restrict__ x,
                           const float* __restrict__ y, const float* __restrict__ z, int64_t n,
                           float4* __restrict__ out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) out[i] = make_float4(x[i], y[i], z[i], m[i]);
}

// One block per tile (P, Q) of a halo: its items (A, B), B-major, A <= B, from the
// tile's first item index on.
__global__ __launch_bounds__(256) void k_sym_expand(const int4* __restrict__ tiles,
                                                    const SymDesc* __restrict__ halos,
                                                    int4* __restrict__ items) {
    const int4 t = tiles[blockIdx.x];
    const SymDesc d = halos[t.x];
    const int wb = d.wb, nb = d.nb;
    const int a0 = t.y * wb, a1 = min(nb, (t.y + 1) * wb);
    const int b0 = t.z * wb, b1 = min(nb, (t.z + 1) * wb);
    int64_t at = t.w;
    for (int B = b0; B < b1; ++B) {
        const int ae = t.y == t.z ? B + 1 : a1;  // diagonal tile: A <= B
        for (int A = a0 + static_cast<int>(threadIdx.x); A < ae; A += blockDim.x)
            items[at + (A - a0)] = make_int4(t.x, A, B, 0);
        at += ae - a0;
    }
}

__global__ void k_sym_clear(int* __restrict__ p) {
    if (threadIdx.x == 0) *p = 0;
}

struct SymWs {
    float4* src4;
    SymDesc* halos;
    int4* items;
    float2* part;
    int4* segs;
    int4* tiles;
    int64_t* base;
    int* head;
    size_t bytes;
};

// n_segs: the merge segments of a banded plan (at most two per halo and tile)
SymWs carve_sym(void* b, const SymPlan& p, int64_t H, int64_t n_segs) {
    Carver c(b);
    SymWs w;
    w.src4 = c.take<float4>(std::max<int64_t>(p.n_members, 1));
    w.halos = c.take<SymDesc>(std::max<int64_t>(H, 1));
    w.items = c.take<int4>(std::max<int64_t>(p.n_items, 1));
    w.part = c.take<float2>(std::max<int64_t>(p.n_part, 1));
    w.segs = c.take<int4>(std::max<int64_t>(n_segs, 1));
    w.tiles = c.take<int4>(std::max<size_t>(p.tiles.size(), 1));
    w.base = c.take<int64_t>(H + 1);
    w.head = c.take<int>(64);
    w.bytes = c.used;
    return w;
}

}  // namespace

int plan_sym(int64_t H, const int64_t* off, SymPlan& plan, bool with_items, int max_members,
             int band) {
    plan = SymPlan();
    plan.halos.resize(H);
    int64_t part = 0;
    std::vector<int64_t> work(H);
    for (int64_t h = 0; h < H; ++h) {
        const int64_t n = off[h + 1] - off[h];
        if (n < 0 || n > INT32_MAX) return set_error(HALMA_E_ARG, "halo %lld: bad offsets",
                                                      static_cast<long long>(h));
        SymDesc& d = plan.halos[h];
        d.off = off[h] - off[0];
        d.part_off = part;
        d.n = static_cast<int32_t>(n);
        d.nb = (max_members != 0 && d.n > max_members) ? 0 : sym_blocks(d.n);
        d.wb = (band > 0 && d.nb > band) ? band : d.nb + 1;
        d.pad = 0;
        part += static_cast<int64_t>(std::min(d.wb, d.nb) + 1) * n;
        work[h] = n;
    }
    plan.order = order_desc(work);
    int64_t n_items = 0;
    for (int64_t h = 0; h < H; ++h) {
        const int64_t nb = plan.halos[h].nb;
        n_items += nb * (nb + 1) / 2;
    }
    if (n_items > INT32_MAX) return set_error(HALMA_E_LIMIT, "too many work items");
    plan.n_items = n_items;
    if (with_items) {
        int64_t tiles = 1;
        for (int64_t h = 0; h < H; ++h) {
            const SymDesc& d = plan.halos[h];
            const int64_t K = d.nb > 0 ? (d.nb + d.wb - 1) / d.wb : 0;
            tiles = std::max<int64_t>(tiles, K * (K + 1) / 2);
        }
        plan.launch_off.push_back(0);
        plan.seg_off.push_back(0);
        int64_t at = 0;  // items listed so far
        for (int64_t t = 0; t < tiles; ++t) {
            for (int32_t h : plan.order) {
                const SymDesc& d = plan.halos[h];
                const int nb = d.nb, wb = d.wb;
                const int64_t K = nb > 0 ? (nb + wb - 1) / wb : 0;
                if (t >= K * (K + 1) / 2) continue;
                int Q = 0;
                while (static_cast<int64_t>(Q + 1) * (Q + 2) / 2 <= t) ++Q;
                const int P = static_cast<int>(t - static_cast<int64_t>(Q) * (Q + 1) / 2);
                const int b0 = Q * wb, b1 = std::min(nb, (Q + 1) * wb);
                const int a0 = P * wb, a1 = std::min(nb, (P + 1) * wb);
                plan.tiles.push_back(make_int4(h, P, Q, static_cast<int>(at)));
                at += P == Q ? static_cast<int64_t>(b1 - b0) * (b1 - b0 + 1) / 2
                             : static_cast<int64_t>(b1 - b0) * (a1 - a0);
                // the members of bands P and Q take this tile's slots into their sums
                auto seg = [&](int band, int role, int nloc) {
                    const int64_t m0 = static_cast<int64_t>(band) * wb * 4 * 128;
                    const int64_t m1 = std::min<int64_t>(d.n, m0 + static_cast<int64_t>(wb) * 512);
                    plan.segs.push_back(make_int4(h, static_cast<int>(m0),
                                                  static_cast<int>(m1 - m0), (role << 24) | nloc));
                };
                if (P == Q) {
                    seg(P, 2, b1 - b0);
                } else {
                    seg(P, 0, b1 - b0);
                    seg(Q, 1, a1 - a0);
                }
            }
            plan.launch_off.push_back(at);
            plan.seg_off.push_back(static_cast<int64_t>(plan.segs.size()));
        }
        if (at != n_items) return set_error(HALMA_E_STATE, "symmetric plan: item count");
    }
    plan.n_members = off[H] - off[0];
    plan.n_part = part;
    return 0;
}

unsigned merge_width(const int4* segs, int64_t n) {
    int64_t most = 1, blocks = 0;
    for (int64_t s = 0; s < n; ++s) {
        const int64_t b = (segs[s].z + 255) / 256;
        most = std::max(most, b);
        blocks += b;
    }
    if (n <= 0) return 1;
    const int64_t want = std::max((2 * blocks + n - 1) / n, (8192 + n - 1) / n);
    return static_cast<unsigned>(std::min<int64_t>({want, most, 128}));
}

int expand_sym_items(const int4* d_tiles, int64_t n_tiles, const SymDesc* d_halos, int4* items,
                     hipStream_t st) {
    if (n_tiles <= 0) return 0;
    if (n_tiles > INT32_MAX) return set_error(HALMA_E_LIMIT, "too many symmetric tiles");
    k_sym_expand<<<static_cast<unsigned>(n_tiles), 256, 0, st>>>(d_tiles, d_halos, items);
    HALMA_LAUNCH_CHECK();
    return 0;
}

int launch_pot_sym(const SymPlan& plan, const float4* src4, const SymDesc* d_halos,
                   const int* live_n, const int4* d_items, const int64_t* n_items_dev,
                   float2* part, int* head, hipStream_t st, bool reset_head) {
    if (reset_head) {
        k_sym_clear<<<1, 64, 0, st>>>(head);
        HALMA_LAUNCH_CHECK();
    }
    const int n_items = static_cast<int>(plan.n_items);
    if (n_items == 0) return 0;
    int cus = device_cu_count();
    if (cus <= 0) cus = 256;
    // both forms are queued when the item count is known only on the device and the plan
    // allows either (the one not chosen returns at once); the device count never exceeds
    // the planned n_items
    if (n_items >= kWaveItems) {
        const int grid = std::max(1, std::min(cus * 8, (n_items + 3) / 4));
        k_pot_sym<<<grid, 256, 0, st>>>(src4, d_halos, live_n, d_items, n_items, n_items_dev,
                                        part, head);
        HALMA_LAUNCH_CHECK();
    }
    if (n_items < kWaveItems || n_items_dev) {
        const int grid = std::max(1, std::min(cus, n_items));
        k_pot_sym_fine<<<grid, 1024, 0, st>>>(src4, d_halos, live_n, d_items, n_items,
                                              n_items_dev, part, head);
        HALMA_LAUNCH_CHECK();
    }
    return 0;
}

}  // namespace halma

using namespace halma;

extern "C" {

double halma_pot_sym_error_bound(void) { return pot_sym_error_bound(); }

size_t halma_pot_sum_self_workspace_size(int64_t n_halo, const int64_t* offsets) {
    if (n_halo < 0 || !offsets) return 0;
    for (int64_t h = 0; h < n_halo; ++h)
        if (offsets[h + 1] < offsets[h]) return 0;
    SymPlan plan;
    if (plan_sym(n_halo, offsets, plan, true, 0, kSymBand)) return 0;
    return carve_sym(nullptr, plan, n_halo, static_cast<int64_t>(plan.segs.size())).bytes;
}

int halma_pot_sum_self_batched(int64_t n_halo, const int64_t* offsets, const float* m,
                               const float* x, const float* y, const float* z, double* out,
                               void* ws, size_t ws_bytes, void* stream) {
    if (n_halo < 0 || !offsets) return set_error(HALMA_E_ARG, "bad halo count or offsets");
    if (n_halo == 0) return 0;
    for (int64_t h = 0; h < n_halo; ++h)
        if (offsets[h + 1] < offsets[h]) return set_error(HALMA_E_ARG, "offsets must not decrease");
    const int64_t n = offsets[n_halo] - offsets[0];
    if (n == 0) return 0;
    if (!m || !x || !y || !z || !out) return set_error(HALMA_E_ARG, "null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    // haloes of more than kSymBand blocks run tile by tile (slots O(n kSymBand) per member)
    SymPlan plan;
    int rc = plan_sym(n_halo, offsets, plan, true, 0, kSymBand);
    if (rc) return rc;
    SymWs w = carve_sym(ws, plan, n_halo, static_cast<int64_t>(plan.segs.size()));
    if (ws_bytes < w.bytes)
        return set_error(HALMA_E_WORKSPACE, "workspace %zu < required %zu", ws_bytes, w.bytes);
    const int64_t o0 = offsets[0];
    k_sym_pack<<<static_cast<unsigned>((n + 255) / 256), 256, 0, st>>>(m + o0, x + o0, y + o0,
                                                                       z + o0, n, w.src4);
    HALMA_LAUNCH_CHECK();
    std::vector<int64_t> base(n_halo + 1);
    for (int64_t h = 0; h <= n_halo; ++h) base[h] = offsets[h] - o0;
    rc = upload_async(w.halos, plan.halos.data(), plan.halos.size() * sizeof(SymDesc), st);
    if (!rc) rc = upload_async(w.base, base.data(), base.size() * sizeof(int64_t), st);
    if (!rc && !plan.tiles.empty())
        rc = upload_async(w.tiles, plan.tiles.data(), plan.tiles.size() * sizeof(int4), st);
    if (!rc && !plan.segs.empty())
        rc = upload_async(w.segs, plan.segs.data(), plan.segs.size() * sizeof(int4), st);
    if (!rc)
        rc = expand_sym_items(w.tiles, static_cast<int64_t>(plan.tiles.size()), w.halos,
                              w.items, st);
    if (rc) return rc;
    double* o = out + o0;
    k_sym_zero<<<256, 256, 0, st>>>(o, n);
    HALMA_LAUNCH_CHECK();
    int cus = device_cu_count();
    if (cus <= 0) cus = 256;
    const int64_t T = static_cast<int64_t>(plan.launch_off.size()) - 1;
    for (int64_t t = 0; t < T; ++t) {
        const int64_t i0 = plan.launch_off[t], ni = plan.launch_off[t + 1] - i0;
        const int64_t s0 = plan.seg_off[t], ns = plan.seg_off[t + 1] - s0;
        if (ni > 0) {
            k_sym_clear<<<1, 64, 0, st>>>(w.head);
            HALMA_LAUNCH_CHECK();
            if (ni >= kWaveItems) {
                const int grid = static_cast<int>(std::min<int64_t>(cus * 8, (ni + 3) / 4));
                k_pot_sym<<<grid, 256, 0, st>>>(w.src4, w.halos, nullptr, w.items + i0,
                                                static_cast<int>(ni), nullptr, w.part, w.head);
            } else {
                const int grid = static_cast<int>(std::min<int64_t>(cus, ni));
                k_pot_sym_fine<<<grid, 1024, 0, st>>>(w.src4, w.halos, nullptr, w.items + i0,
                                                      static_cast<int>(ni), nullptr, w.part,
                                                      w.head);
            }
            HALMA_LAUNCH_CHECK();
        }
        if (ns > 0) {
            const dim3 mg(merge_width(plan.segs.data() + s0, ns),
                          static_cast<unsigned>(std::min<int64_t>(ns, 65535)));
            k_sym_merge_tile<<<mg, 256, 0, st>>>(w.halos, w.segs + s0, static_cast<int>(ns),
                                                 w.base, w.part, o);
            HALMA_LAUNCH_CHECK();
        }
    }
    return 0;
}

}  // extern "C"
