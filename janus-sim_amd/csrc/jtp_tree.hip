// Radix tree (Karras LBVH) over the sorted Morton keys with integer-exact dual (m+, m-) monopoles and boxes, built
// bottom-up in LDS; walk groups and cell offset tables.
//
// Reference behaviour replaced:
//   build_bvh_tp + delta_tp / range_tp / split_tp / clz64_tp (src/nbody_gpu_twopass.rs:356-447):
//     same radix-tree topology and node numbers (same delta with the index tie-break), found from the leaves up
//     instead of by a range and split search per node; leaves are encoded here as ~sorted_index instead of n-1+index.
//   init_leaves_tp + reduce_tp (nbody_gpu_twopass.rs:450-561) build ONE species per tree in FP32
//     with atomics; here one tree holds both species and every node keeps separate (n+, sum x+) and
//     (n-, sum x-) as exact 64-bit integer sums of fixed-point coordinates, so the monopoles are
//     independent of summation order and bit-reproducible.  The dual-monopole node is the design of
//     src/nbody_gpu.rs:603-874 (init_leaves/reduce_com); no periodic unfolding is needed because a
//     radix-tree node is a Morton-prefix range and never straddles the periodic boundary.
#include "jtp_internal.h"
#include "jtp_device.h"

namespace jtp {

struct alignas(16) NodeSum {  // 64 bytes: the stage copy reads this layout
    uint64_t sp[3];
    uint64_t sm[3];
    uint32_t np, nm;
    uint32_t pad[2];
};
static_assert(sizeof(NodeSum) == 64, "NodeSum layout");

__device__ inline int clz64_dev(uint64_t x) { return x == 0 ? 64 : __clzll((long long)x); }

// Common prefix length of the (key, index) strings of neighbours i and i + 1, plus one; 0 outside [0, n).
__device__ inline uint32_t delta1(const uint64_t* __restrict__ k, int64_t n, int64_t i) {
    if (i < 0 || i + 1 >= n) return 0;
    const uint64_t a = k[i], b = k[i + 1];
    return 1u + (a == b ? 64u + (uint32_t)clz64_dev((uint64_t)(i ^ (i + 1))) : (uint32_t)clz64_dev(a ^ b));
}

// Quotient s / cnt for s < 2^63 and a quotient below 2^33, rc = 1 / cnt in double: the double estimate is within 1 of
// it and the remainder settles which (a 64-bit integer division is ~10x the instructions).
__device__ inline uint64_t quot_u64(uint64_t s, uint32_t cnt, double rc) {
    uint64_t q = (uint64_t)((double)s * rc);
    const int64_t r = (int64_t)(s - q * (uint64_t)cnt);
    if (r < 0) --q;
    else if (r >= (int64_t)cnt) ++q;
    return q;
}
// Rounded integer mean of a fixed-point coordinate sum.
__device__ inline uint32_t mean_fixed(uint64_t s, uint32_t cnt, double rc) {
    return (uint32_t)quot_u64(s + (uint64_t)(cnt >> 1), cnt, rc);
}
__device__ inline double mean_fixed_f64(uint64_t s, uint32_t cnt, double rc) {
    const uint64_t q = quot_u64(s, cnt, rc), r = s - q * (uint64_t)cnt;
    return (double)q + (double)r / (double)cnt;
}

// Walk records of one node, written as soon as its sums and box are final.
//   FP32: {com+ xyz (fixed), q+ (float bits)}, {com- xyz, q-}
//   FP64: {com+ xyz (fixed units, as double), q+}, {com- xyz, q-}
// q = sigma G |m| n; an empty species gets the box centre and q = 0.
template <int PREC>
__device__ inline void write_mono(int32_t p, const NodeSum& s, const uint32_t mn[3], const uint32_t mx[3],
                                  void* mono, double qp, double qm) {
    const double rp = s.np ? 1.0 / (double)s.np : 0.0, rm = s.nm ? 1.0 / (double)s.nm : 0.0;
    if (PREC == JTP_FP64) {
        const double c[3] = {(double)mn[0] + 0.5 * (double)(mx[0] - mn[0]),
                             (double)mn[1] + 0.5 * (double)(mx[1] - mn[1]),
                             (double)mn[2] + 0.5 * (double)(mx[2] - mn[2])};
        double4 a, b;
        if (s.np)
            a = make_double4(mean_fixed_f64(s.sp[0], s.np, rp), mean_fixed_f64(s.sp[1], s.np, rp),
                             mean_fixed_f64(s.sp[2], s.np, rp), qp * (double)s.np);
        else
            a = make_double4(c[0], c[1], c[2], 0.0);
        if (s.nm)
            b = make_double4(mean_fixed_f64(s.sm[0], s.nm, rm), mean_fixed_f64(s.sm[1], s.nm, rm),
                             mean_fixed_f64(s.sm[2], s.nm, rm), -qm * (double)s.nm);
        else
            b = make_double4(c[0], c[1], c[2], 0.0);
        ((double4*)mono)[2 * p] = a;
        ((double4*)mono)[2 * p + 1] = b;
    } else {
        const uint32_t c[3] = {mn[0] + (mx[0] - mn[0]) / 2, mn[1] + (mx[1] - mn[1]) / 2, mn[2] + (mx[2] - mn[2]) / 2};
        const float qpf = (float)qp, qmf = (float)qm;
        uint4 a, b;
        if (s.np)
            a = make_uint4(mean_fixed(s.sp[0], s.np, rp), mean_fixed(s.sp[1], s.np, rp), mean_fixed(s.sp[2], s.np, rp),
                           __float_as_uint(qpf * (float)s.np));
        else
            a = make_uint4(c[0], c[1], c[2], __float_as_uint(0.0f));
        if (s.nm)
            b = make_uint4(mean_fixed(s.sm[0], s.nm, rm), mean_fixed(s.sm[1], s.nm, rm), mean_fixed(s.sm[2], s.nm, rm),
                           __float_as_uint(-qmf * (float)s.nm));
        else
            b = make_uint4(c[0], c[1], c[2], __float_as_uint(0.0f));
        ((uint4*)mono)[2 * p] = a;
        ((uint4*)mono)[2 * p + 1] = b;
    }
}

// ------------------------------------------------------------------ bottom-up build
// A node of the radix tree is a run [f, l] of sorted leaves; with d(i) the common prefix of neighbours i and i + 1, it
// is the right child of its parent if d(f - 1) > d(l) and the left child otherwise, and the parent's split lies at that
// neighbour pair.  So a run that is complete needs two prefix lengths to know where it belongs, the two children of a
// parent meet at the parent's split, and the node's number is known with its side: f for a right child, l for a left
// one (0 for the root), as in Karras's construction.  (Agglomerative construction: Apetrei, Fast and Simple Agglomerative LBVH
// Construction, 2014.)
//
// One workgroup holds up to kBtM consecutive items (leaves or finished subtrees) in LDS.  Every thread starts from its
// item and climbs: it leaves its run at the parent's split; the second of the two to arrive merges and climbs on.
// Only the box travels; the species sums of a run are differences of prefix sums over the items, exact in 64 bits.
// When the climb has ended, one thread per finished node computes its records, all lanes busy, and writes them.  What
// stays unmerged (a run whose parent reaches beyond the items) is carried into the next round with the next leaves, and
// at the end goes to the workgroup's list in memory.  The next launch does the same with the lists of several
// workgroups as its items, down to one workgroup.
//
// The prefix lengths between the unmerged runs of a round have no inner local maximum (it would be a split whose two
// sides are there), so they fall and then rise: at most 2 x 80 of them (48 key bits and 32 index bits each way).
//
// Measured against the build it replaces (a range and split search per node, then three launches climbing through node
// records in device memory), the whole tree phase: 0.30 -> 0.08 ms at 2e4 particles, 0.35 -> 0.14 ms at 5.2e5, 4.4 -> 2.4
// ms at 2.2e7 beside the particle mesh.  The first launch is bound by VALU and LDS latency of the climb (~14 levels, few
// lanes left at the upper ones), not by HBM (96 bytes a leaf).
constexpr int kBtM = 384;      // items and threads of a workgroup: 48 KB of LDS, three workgroups per CU
constexpr int kBtLeft = 160;   // most unmerged runs of a round
constexpr int kBtLists = 28;   // lists per workgroup of a later launch: ~15 runs each
constexpr int kBtFinal = 64;   // most lists that the last launch's one workgroup takes
constexpr int kBtRounds = 8;   // most rounds of a workgroup of the first launch
constexpr int32_t kNoNode = (int32_t)0x80000000;

struct BtItem {  // one run: box, species sums, leaf range
    uint32_t mn[3], mx[3];
    uint64_t sp[3], sm[3];
    uint32_t np, nm;
    uint32_t first, last;
};
static_assert(sizeof(BtItem) == 88, "BtItem layout");

struct BtArgs {
    const uint64_t* keys;
    const uint4* parts;
    int64_t n;
    uint4* geo;
    int2* kids;
    void* mono;
    double qp, qm;
    const BtItem* in;       // kBtLeft per list
    const int32_t* in_cnt;  // items of each list
    int32_t nlists, lists_per_wg;
    int64_t span;           // first launch: leaves per workgroup
    BtItem* out;            // kBtLeft per workgroup
    int32_t* out_cnt;
    int32_t* cellnode;      // node of each start cell of the walk
    int32_t cell_prefix;    // 1 + prefix length (bits) of a start cell
    int32_t cell_shift;
    int32_t* counters;
};

// Inclusive prefix sum of a uint64 across the wavefront (the DPP pattern of wave_incl_scan_dpp).
// (bound_ctrl: lanes without a source read 0, so that no register has to be cleared for them)
template <int CTRL, int ROWS>
__device__ inline uint64_t dpp_add_u64(uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, ROWS, 0xf, ROWS == 0xf);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, ROWS, 0xf, ROWS == 0xf);
    return v + (((uint64_t)hi << 32) | lo);
}
__device__ inline uint64_t wave_incl_scan_u64(uint64_t v) {
    v = dpp_add_u64<0x111, 0xf>(v);
    v = dpp_add_u64<0x112, 0xf>(v);
    v = dpp_add_u64<0x114, 0xf>(v);
    v = dpp_add_u64<0x118, 0xf>(v);
    v = dpp_add_u64<0x142, 0xa>(v);
    return dpp_add_u64<0x143, 0xc>(v);
}

__device__ inline void lds_release() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local"); }
__device__ inline void lds_acquire() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local"); }

template <int PREC, bool LEAVES>
__global__ __launch_bounds__(kBtM, 4) void k_build(BtArgs a) {
    constexpr int W = kBtM / 64;
    constexpr uint32_t kLeafH = 0x8000u;  // handle of an item; a merged run's handle is its split
    __shared__ uint32_t ifirst[kBtM], ilast[kBtM];
    __shared__ uint8_t dl[kBtM + 2];           // dl[k]: prefix length + 1 before item k
    __shared__ uint64_t psum[6][kBtM + 1];     // exclusive prefix sums of sp, sm
    __shared__ uint32_t pcnt[2][kBtM + 1];
    __shared__ uint32_t state[kBtM + 2];       // handle + 1 of the run that waits at a split (last two: at the ends)
    __shared__ uint32_t ab[kBtM];              // items [a, b] of the run merged at a split, a | b << 16
    __shared__ uint32_t box[6][kBtM];          // its box
    __shared__ uint32_t ibox[6][kBtM];         // the items' boxes
    __shared__ uint16_t ord[kBtM];             // handle + 1 of the unmerged run that starts at an item
    __shared__ uint64_t wsum[W][6];
    __shared__ uint32_t wcnt[W][2];
    __shared__ int32_t woff[W + 1];
    __shared__ int32_t loff[LEAVES ? 1 : kBtFinal + 1];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;

    // the input: leaves [pos, end), or the items of the lists [l0, l1) numbered through
    int64_t pos, end;
    int l0 = 0, l1 = 0;
    if (LEAVES) {
        pos = (int64_t)blockIdx.x * a.span;
        end = pos + a.span < a.n ? pos + a.span : a.n;
    } else {
        l0 = (int)blockIdx.x * a.lists_per_wg;
        l1 = min(l0 + a.lists_per_wg, a.nlists);
        if (t == 0) {
            int s = 0;
            for (int i = l0; i < l1; ++i) {
                loff[i - l0] = s;
                s += min(a.in_cnt[i], kBtLeft);
            }
            loff[l1 - l0] = s;
        }
        __syncthreads();
        pos = 0;
        end = loff[l1 - l0];
    }

    BtItem it;  // the thread's item
    int nleft = 0;
    while (true) {
        const int64_t rem = end - pos;
        const int m = rem < kBtM - nleft ? nleft + (int)rem : kBtM;
        const bool have = t < m;
        const bool fresh = have && t >= nleft;
        if (fresh) {
            const int64_t i = pos + (t - nleft);
            if (LEAVES) {
                const uint4 r = a.parts[i];
                const uint32_t p[3] = {r.x, r.y, r.z};
                const bool plus = (int32_t)r.w > 0;
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    it.mn[x] = it.mx[x] = p[x];
                    it.sp[x] = plus ? p[x] : 0;
                    it.sm[x] = plus ? 0 : p[x];
                }
                it.np = plus ? 1u : 0u;
                it.nm = plus ? 0u : 1u;
                it.first = it.last = (uint32_t)i;
            } else {
                int lo = 0, hi = l1 - l0;  // the list that holds item i
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (loff[mid] <= (int)i) lo = mid; else hi = mid;
                }
                it = a.in[(int64_t)(l0 + lo) * kBtLeft + ((int)i - loff[lo])];
            }
        }
        pos += m - nleft;
        if (have) {
            ifirst[t] = it.first;
            ilast[t] = it.last;
            dl[t + 1] = (uint8_t)delta1(a.keys, a.n, (int64_t)it.last);
            if (t == 0) dl[0] = (uint8_t)delta1(a.keys, a.n, (int64_t)it.first - 1);
#pragma unroll
            for (int x = 0; x < 3; ++x) {
                ibox[x][t] = it.mn[x];
                ibox[3 + x][t] = it.mx[x];
            }
        }
        ab[t] = ~0u;
        ord[t] = 0;
        for (int k = t; k < kBtM + 2; k += kBtM) state[k] = 0;
        // prefix sums over the items
        uint64_t v[6];
        uint32_t c[2];
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            v[x] = wave_incl_scan_u64(have ? it.sp[x] : 0);
            v[3 + x] = wave_incl_scan_u64(have ? it.sm[x] : 0);
        }
        c[0] = (uint32_t)wave_incl_scan_dpp(have ? (int)it.np : 0);
        c[1] = (uint32_t)wave_incl_scan_dpp(have ? (int)it.nm : 0);
        if (lane == 63) {
#pragma unroll
            for (int x = 0; x < 6; ++x) wsum[w][x] = v[x];
            wcnt[w][0] = c[0];
            wcnt[w][1] = c[1];
        }
        __syncthreads();
        for (int i = 0; i < w; ++i) {
#pragma unroll
            for (int x = 0; x < 6; ++x) v[x] += wsum[i][x];
            c[0] += wcnt[i][0];
            c[1] += wcnt[i][1];
        }
#pragma unroll
        for (int x = 0; x < 6; ++x) psum[x][t + 1] = v[x];
        pcnt[0][t + 1] = c[0];
        pcnt[1][t + 1] = c[1];
        if (t < 6) psum[t][0] = 0;
        if (t < 2) pcnt[t][0] = 0;

        // the climb: at most m merges per thread
        if (have) {
            if (LEAVES && fresh && max((int)dl[t], (int)dl[t + 1]) < a.cell_prefix)
                a.cellnode[a.keys[it.first] >> a.cell_shift] = ~(int32_t)it.first;  // alone in its start cell
            int ra = t, rb = t;
            uint32_t h = kLeafH | (uint32_t)t;
            uint32_t b6[6] = {it.mn[0], it.mn[1], it.mn[2], it.mx[0], it.mx[1], it.mx[2]};
            while (true) {
                const int dL = dl[ra], dR = dl[rb + 1];
                if (dL == 0 && dR == 0) {  // the whole tree
                    a.counters[kCtrRoot] = 1;
                    break;
                }
                const bool right = dL > dR;
                if (right ? ra == 0 : rb == m - 1) {
                    state[right ? kBtM : kBtM + 1] = h + 1;
                    break;
                }
                const int g = right ? ra - 1 : rb;
                lds_release();
                const uint32_t old = atomicExch(&state[g], h + 1);
                if (old == 0) break;
                lds_acquire();
                const uint32_t oh = old - 1;
                if (oh & kLeafH) {
                    const int o = (int)(oh & ~kLeafH);
                    if (right) ra = o; else rb = o;
#pragma unroll
                    for (int x = 0; x < 3; ++x) {
                        b6[x] = min(b6[x], ibox[x][o]);
                        b6[3 + x] = max(b6[3 + x], ibox[3 + x][o]);
                    }
                } else {
                    const uint32_t oab = ab[oh];
                    if (right) ra = (int)(oab & 0xffffu); else rb = (int)(oab >> 16);
#pragma unroll
                    for (int x = 0; x < 3; ++x) {
                        b6[x] = min(b6[x], box[x][oh]);
                        b6[3 + x] = max(b6[3 + x], box[3 + x][oh]);
                    }
                }
                ab[g] = (uint32_t)ra | ((uint32_t)rb << 16);
#pragma unroll
                for (int x = 0; x < 6; ++x) box[x][g] = b6[x];
                h = (uint32_t)g;
            }
        }
        __syncthreads();

        // the finished nodes, one per split
        if (t < m && ab[t] != ~0u) {
            const int ra = (int)(ab[t] & 0xffffu), rb = (int)(ab[t] >> 16);
            const int32_t f = (int32_t)ifirst[ra], l = (int32_t)ilast[rb], g = (int32_t)ilast[t];
            const int dL = dl[ra], dR = dl[rb + 1];
            const int32_t id = dL == 0 && dR == 0 ? 0 : (dL > dR ? f : l);
            NodeSum s;
#pragma unroll
            for (int x = 0; x < 3; ++x) {
                s.sp[x] = psum[x][rb + 1] - psum[x][ra];
                s.sm[x] = psum[3 + x][rb + 1] - psum[3 + x][ra];
            }
            s.np = pcnt[0][rb + 1] - pcnt[0][ra];
            s.nm = pcnt[1][rb + 1] - pcnt[1][ra];
            const uint32_t mn[3] = {box[0][t], box[1][t], box[2][t]}, mx[3] = {box[3][t], box[4][t], box[5][t]};
            // box as (centre, first) and (extent, last): the walk's box test needs no further arithmetic, and
            // min = centre - extent / 2, max = min + extent recover the corners exactly
            uint32_t e[3], nc[3];
#pragma unroll
            for (int x = 0; x < 3; ++x) {
                e[x] = mx[x] - mn[x];
                nc[x] = mn[x] + e[x] / 2;
            }
            a.geo[2 * (int64_t)id] = make_uint4(nc[0], nc[1], nc[2], (uint32_t)f);
            a.geo[2 * (int64_t)id + 1] = make_uint4(e[0], e[1], e[2], (uint32_t)l);
            a.kids[id] = make_int2(f == g ? ~g : g, g + 1 == l ? ~l : g + 1);
            write_mono<PREC>(id, s, mn, mx, a.mono, a.qp, a.qm);
            if (dl[t + 1] >= a.cell_prefix && max(dL, dR) < a.cell_prefix) a.cellnode[a.keys[f] >> a.cell_shift] = id;
        }
        // the unmerged runs, in order
        for (int k = t; k < kBtM + 2; k += kBtM) {
            const uint32_t h1 = state[k];
            if (h1 == 0 || (k < kBtM && ab[k] != ~0u)) continue;
            const uint32_t h = h1 - 1;
            ord[h & kLeafH ? h & ~kLeafH : ab[h] & 0xffffu] = (uint16_t)h1;
        }
        __syncthreads();
        const uint32_t h1 = ord[t];
        const uint64_t bal = __ballot(h1 != 0);
        if (lane == 0) woff[w] = (int)__popcll(bal);
        if (h1) {
            const uint32_t h = h1 - 1;
            const bool leaf = (h & kLeafH) != 0;
            const int rb = leaf ? t : (int)(ab[h] >> 16);
            it.first = ifirst[t];
            it.last = ilast[rb];
#pragma unroll
            for (int x = 0; x < 3; ++x) {
                it.mn[x] = leaf ? ibox[x][t] : box[x][h];
                it.mx[x] = leaf ? ibox[3 + x][t] : box[3 + x][h];
                it.sp[x] = psum[x][rb + 1] - psum[x][t];
                it.sm[x] = psum[3 + x][rb + 1] - psum[3 + x][t];
            }
            it.np = pcnt[0][rb + 1] - pcnt[0][t];
            it.nm = pcnt[1][rb + 1] - pcnt[1][t];
        }
        __syncthreads();
        int rank = 0, total = 0;
        for (int i = 0; i < W; ++i) {
            if (i < w) rank += woff[i];
            total += woff[i];
        }
        rank += (int)__popcll(bal & lanemask_lt());
        if (total > kBtLeft) {  // no sorted keys give this: report it
            if (t == 0) a.counters[kCtrErr] = 5;
            total = kBtLeft;
        }
        if (pos >= end) {
            if (a.out_cnt) {
                if (h1 && rank < kBtLeft) a.out[(int64_t)blockIdx.x * kBtLeft + rank] = it;
                if (t == 0) a.out_cnt[blockIdx.x] = total;
            }
            return;
        }
        // to threads 0 .. total - 1, through the LDS of the sums and boxes (read above)
        BtItem* stage = (BtItem*)&psum[0][0];
        static_assert(sizeof(BtItem) * kBtLeft <= sizeof(psum), "staging fits");
        if (h1 && rank < kBtLeft) stage[rank] = it;
        __syncthreads();
        if (t < total) it = stage[t];
        nleft = total;
        __syncthreads();
    }
}

// Sums of every node (the stage export; the walk needs only the monopoles), a wavefront per node.  A node's leaves are added
// as whole chunks of kSumChunk, summed before, and what is left at its ends: the root's wavefront alone took 1 ms at 2e5
// particles reading leaf by leaf.
constexpr int kSumChunk = 512;

__device__ inline void add_sums(NodeSum& s, const NodeSum& o) {
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        s.sp[x] += o.sp[x];
        s.sm[x] += o.sm[x];
    }
    s.np += o.np;
    s.nm += o.nm;
}
// The lane's share of the leaves [f, l).
__device__ inline void add_leaves(NodeSum& s, const uint4* __restrict__ parts, int64_t f, int64_t l) {
    for (int64_t k = f + lane_id(); k < l; k += 64) {
        const uint4 r = parts[k];
        const bool plus = (int32_t)r.w > 0;
        const NodeSum o = {{plus ? r.x : 0u, plus ? r.y : 0u, plus ? r.z : 0u},
                           {plus ? 0u : r.x, plus ? 0u : r.y, plus ? 0u : r.z},
                           plus ? 1u : 0u,
                           plus ? 0u : 1u,
                           {0, 0}};
        add_sums(s, o);
    }
}
__device__ inline void write_sums(NodeSum s, NodeSum* __restrict__ out) {
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        s.sp[x] = wave_sum(s.sp[x]);
        s.sm[x] = wave_sum(s.sm[x]);
    }
    s.np = wave_sum(s.np);
    s.nm = wave_sum(s.nm);
    if (lane_id() == 0) *out = s;
}
__device__ inline int64_t wave_index() { return (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); }

__global__ __launch_bounds__(256) void k_chunk_sums(const uint4* __restrict__ parts, int64_t nchunk,
                                                    NodeSum* __restrict__ chunks) {
    const int64_t c = wave_index();
    if (c >= nchunk) return;
    NodeSum s{};
    add_leaves(s, parts, c * kSumChunk, (c + 1) * kSumChunk);
    write_sums(s, chunks + c);
}

__global__ __launch_bounds__(256) void k_node_sums(const uint4* __restrict__ parts, const uint4* __restrict__ geo,
                                                   int64_t nI, const NodeSum* __restrict__ chunks,
                                                   NodeSum* __restrict__ out) {
    const int64_t nw = (int64_t)gridDim.x * (blockDim.x >> 6);
    for (int64_t i = wave_index(); i < nI; i += nw) {
        const int64_t f = geo[2 * i].w, e = (int64_t)geo[2 * i + 1].w + 1;
        const int64_t c0 = (f + kSumChunk - 1) / kSumChunk, c1 = e / kSumChunk;
        NodeSum s{};
        if (e > nI + 1) {  // a node that a failed build left unwritten
        } else if (c1 <= c0) {
            add_leaves(s, parts, f, e);
        } else {
            add_leaves(s, parts, f, c0 * kSumChunk);
            for (int64_t c = c0 + lane_id(); c < c1; c += 64) add_sums(s, chunks[c]);
            add_leaves(s, parts, c1 * kSumChunk, e);
        }
        write_sums(s, out + i);
    }
}

hipError_t stage_node_sums(Ctx& c, int64_t n, hipStream_t s) {
    if (n < 2) return hipSuccess;
    const int64_t nb = (n - 1 + 3) / 4, nchunk = n / kSumChunk;
    NodeSum* chunks = (NodeSum*)c.keys1;  // free after the sort; 64 bytes to 512 of its 8
    static_assert(sizeof(NodeSum) <= kSumChunk * sizeof(uint64_t), "the chunks' sums fit");
    if (nchunk > 0) k_chunk_sums<<<dim3((unsigned)((nchunk + 3) / 4)), dim3(256), 0, s>>>(c.parts, nchunk, chunks);
    k_node_sums<<<dim3((unsigned)(nb < 65536 ? nb : 65536)), dim3(256), 0, s>>>(c.parts, c.node_geo, n - 1, chunks,
                                                                               (NodeSum*)c.node_sum);
    return hipGetLastError();
}

// ------------------------------------------------------------------ cell offsets
// out[c] = first sorted index whose cell (key >> shift) is >= c, for c in [0, ncells].
// Every entry is written exactly once, by the particle that starts the run.
__global__ void k_cell_start(const uint64_t* __restrict__ keys, int64_t n, int shift, int64_t ncells,
                             int32_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t c = (int64_t)(keys[i] >> shift);
    const int64_t cp = (i == 0) ? -1 : (int64_t)(keys[i - 1] >> shift);
    for (int64_t cc = cp + 1; cc <= c; ++cc) out[cc] = (int32_t)i;
    if (i == n - 1)
        for (int64_t cc = c + 1; cc <= ncells; ++cc) out[cc] = (int32_t)n;
}
__global__ void k_fill_i32(int32_t* __restrict__ out, int64_t m, int32_t v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) out[i] = v;
}

hipError_t launch_fill_i32(int32_t* out, int64_t m, int32_t v, hipStream_t s) {
    if (m > 0) k_fill_i32<<<dim3((unsigned)((m + kBlock - 1) / kBlock)), dim3(kBlock), 0, s>>>(out, m, v);
    return hipGetLastError();
}

hipError_t launch_cell_start(const uint64_t* keys, int64_t n, int shift, int64_t ncells, int32_t* out,
                             hipStream_t s) {
    if (n == 0) {
        k_fill_i32<<<dim3((unsigned)((ncells + 1 + kBlock - 1) / kBlock)), dim3(kBlock), 0, s>>>(out, ncells + 1, 0);
    } else {
        k_cell_start<<<dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, s>>>(keys, n, shift, ncells,
                                                                                       out);
    }
    return hipGetLastError();
}

// ------------------------------------------------------------------ walk groups
// Groups are runs of <= gs consecutive sorted particles inside one level-4 Morton cell
// (edge L/16).  cell4[c] = first sorted particle of cell c: the sort's gather has written it for the cells that hold
// any, the others (kNoCell) take the next cell's here; cell4[4096] = n.  goff[c] = index of the first group of cell c;
// counters[0] = number of groups.  One workgroup, the cells from the last to the first: two scans and no search of the
// keys (19.8 -> 4 us at 2e4 particles, all of it on the way to the build).
constexpr int kNCell4 = 1 << (3 * kGroupLevelBits);
constexpr int32_t kNoCell = 0x7fffffff;

__global__ __launch_bounds__(1024) void k_group_offsets(int32_t n, int gs, int32_t* __restrict__ cell4,
                                                        int32_t* __restrict__ goff, int32_t* __restrict__ counters) {
    __shared__ uint32_t next_s[16], sum_s[16];
    constexpr int per = kNCell4 / 1024;
    static_assert(per == 4, "one int4 a thread");
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    int4* q = (int4*)(cell4 + kNCell4 - per * (tid + 1));
    const int4 in = *q;
    const int32_t raw[per] = {in.w, in.z, in.y, in.x};
    // the running minimum of the starts, as a maximum with 0 for none
    uint32_t m[per];
#pragma unroll
    for (int j = 0; j < per; ++j) m[j] = max(j ? m[j - 1] : 0u, (uint32_t)(kNoCell - raw[j]));
    const uint32_t incl = wave_incl_max_dpp(m[per - 1]);
    if (lane == 63) next_s[w] = incl;
    const uint32_t up = (uint32_t)__shfl_up((int)incl, 1, 64);
    __syncthreads();
    uint32_t prev = max((uint32_t)(kNoCell - n), lane ? up : 0u);
    for (int i = 0; i < w; ++i) prev = max(prev, next_s[i]);
    int32_t start[per + 1];  // start[0]: of the cell after this thread's
    start[0] = kNoCell - (int32_t)prev;
    uint32_t v[per], s = 0;
#pragma unroll
    for (int j = 0; j < per; ++j) {
        start[j + 1] = kNoCell - (int32_t)max(prev, m[j]);
        v[j] = (uint32_t)((start[j] - start[j + 1] + gs - 1) / gs);
        s += v[j];
    }
    *q = make_int4(start[4], start[3], start[2], start[1]);
    const uint32_t sum = (uint32_t)wave_incl_scan_dpp((int)s);
    if (lane == 63) sum_s[w] = sum;
    __syncthreads();
    uint32_t after = sum - s, tot = 0;  // groups of the cells after this one
    for (int i = 0; i < 16; ++i) {
        if (i < w) after += sum_s[i];
        tot += sum_s[i];
    }
#pragma unroll
    for (int j = 0; j < per; ++j) {
        after += v[j];
        goff[kNCell4 - 1 - (per * tid + j)] = (int32_t)(tot - after);
    }
    if (tid == 0) {
        cell4[kNCell4] = n;
        goff[kNCell4] = (int32_t)tot;
        counters[kCtrNGroups] = (int32_t)tot;
    }
}

// The groups, and the list of those to walk first.  A run of Morton-consecutive particles that straddles the boundary of a
// large cell has a box that can reach across a dense region it has no part in; such a group opens everything there and
// takes up to 16 ms beside a mean of 0.22 (2.2e7 clustered particles), and whatever was pulled last set the end of the
// launch.  Their smallest enclosing Morton cell reaches far beyond them (the keys kEarlySpan / 2 group sizes before and after
// the run tell; in a level-4 cell with fewer particles than that none does), which also marks
// ~3 % of harmless groups; with all of those first, the long ones overlap the rest.  Walk before -> after: 1.76 ->
// 1.46 ms (1000003 clustered particles), 13.9 -> 12.7 (2.75e6, FP64), 39.0 -> 37.9 (2.2e7).
__global__ void k_groups(const uint64_t* __restrict__ keys, int64_t n, const int32_t* __restrict__ cell4,
                         const int32_t* __restrict__ goff, int gs, int64_t gmax, int2* __restrict__ groups,
                         int32_t* __restrict__ early, int32_t early_max, int32_t* __restrict__ counters) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= gmax || g >= goff[kNCell4]) return;
    int lo = 0, hi = kNCell4;  // find c with goff[c] <= g < goff[c+1]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (goff[mid] <= g) lo = mid; else hi = mid;
    }
    // skip empty cells that share the same offset
    int c = lo;
    const int64_t j = g - goff[c];
    const int32_t first = cell4[c] + (int32_t)(j * gs);
    int32_t cnt = min((int32_t)gs, cell4[c + 1] - first);
    if (cell4[c + 1] - cell4[c] > gs * (kEarlySpan / 2)) {  // a thinner level-4 cell: no cell within it is that full
        const int64_t last = (int64_t)first + cnt - 1, before = first - (int64_t)gs * (kEarlySpan / 2),
                      after = last + (int64_t)gs * (kEarlySpan / 2);
        const uint64_t kf = keys[first];
        const int prefix = clz64_dev(kf ^ keys[last]);
        if ((before >= 0 && clz64_dev(kf ^ keys[before]) >= prefix) ||
            (after < n && clz64_dev(kf ^ keys[after]) >= prefix)) {
            const int32_t k = atomicAdd(&counters[kCtrEarly], 1);
            if (k < early_max) {
                early[k] = (int32_t)g;
                cnt |= kEarlyMark;
            }
        }
    }
    groups[g] = make_int2(first, cnt);
}

// Clears what an evaluation counts, the cells' starts (cell4), and the start cells of the walk: cellnode[c] is the node whose leaves are exactly
// the particles of Morton cell c of level start_level (such a prefix range is one subtree; ~leaf for a single particle,
// kNoNode for none), written by the build; the walk seeds each group's traversal with the 27 cells around it.
__global__ void k_reset(int32_t* __restrict__ counters, int32_t* __restrict__ cellnode,
                        int32_t* __restrict__ cell4) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 4096) cellnode[i] = kNoNode;
    if (i < kNCell4) cell4[i] = kNoCell;
    if (i < kCtrTotal) counters[i] = 0;
}
hipError_t launch_reset(Ctx& c, hipStream_t s) {
    k_reset<<<dim3(16), dim3(256), 0, s>>>(c.dev_counters, c.cellnode, c.cell4);
    return hipGetLastError();
}

template <int PREC>
static hipError_t launch_build(Ctx& c, int64_t n, hipStream_t s) {
    BtArgs a{};
    a.keys = c.keys0;
    a.parts = c.parts;
    a.n = n;
    a.geo = c.node_geo;
    a.kids = c.node_kids;
    a.mono = c.node_mono;
    a.qp = c.p.g_constant * c.m_plus;
    a.qm = c.p.g_constant * c.m_minus;
    a.cellnode = c.cellnode;
    a.cell_prefix = 1 + 1 + 3 * c.start_level;  // + 1: the keys' top bit is 0
    a.cell_shift = 63 - 3 * c.start_level;
    a.counters = c.dev_counters;
    // rounds per workgroup: as many as leave 2048 workgroups (several per CU), at most kBtRounds
    int64_t rounds = n / ((int64_t)kBtM * 2048);
    rounds = rounds < 1 ? 1 : (rounds > kBtRounds ? kBtRounds : rounds);
    a.span = kBtM + (rounds - 1) * (kBtM - 16);
    int64_t lists = (n + a.span - 1) / a.span;
    BtItem* items = (BtItem*)c.node_sum;  // free here: the gather has read the records that were in it
    int32_t* cnt = c.bt_count;
    int64_t used = 0;  // lists placed so far: ~37 bytes a particle of the buffer's 64
    auto room = [&](int64_t k) {
        return (used + k) * kBtLeft * (int64_t)sizeof(BtItem) <= c.cap_n * (int64_t)sizeof(NodeSum) &&
               used + k <= bt_count_size(c.cap_n);
    };
    if (!room(lists)) return hipErrorInvalidValue;
    a.out = items;
    a.out_cnt = cnt;
    k_build<PREC, true><<<dim3((unsigned)lists), dim3(kBtM), 0, s>>>(a);
    while (lists > 1) {
        a.in = items;
        a.in_cnt = cnt;
        a.nlists = (int32_t)lists;
        items += lists * kBtLeft;
        cnt += lists;
        used += lists;
        const bool last = lists <= kBtFinal;
        a.lists_per_wg = last ? (int32_t)lists : kBtLists;
        lists = last ? 1 : (lists + kBtLists - 1) / kBtLists;
        if (!last && !room(lists)) return hipErrorInvalidValue;
        a.out = last ? nullptr : items;
        a.out_cnt = last ? nullptr : cnt;
        k_build<PREC, false><<<dim3((unsigned)lists), dim3(kBtM), 0, s>>>(a);
    }
    return hipGetLastError();
}

hipError_t build_tree(Ctx& c, int64_t n, hipStream_t s) {
    int32_t* goff = c.cell4 + (kNCell4 + 1);
    k_group_offsets<<<dim3(1), dim3(1024), 0, s>>>((int32_t)n, c.p.group_size, c.cell4, goff, c.dev_counters);
    if (c.n_groups_max > 0)
        k_groups<<<dim3((unsigned)((c.n_groups_max + kBlock - 1) / kBlock)), dim3(kBlock), 0, s>>>(
            c.keys0, n, c.cell4, goff, c.p.group_size, c.n_groups_max, c.groups, c.early, (int32_t)early_cap(c.cap_n),
            c.dev_counters);
    if (n >= 2) return c.p.precision == JTP_FP64 ? launch_build<JTP_FP64>(c, n, s) : launch_build<JTP_FP32>(c, n, s);
    return hipGetLastError();
}

}  // namespace jtp
