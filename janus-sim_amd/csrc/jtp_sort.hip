// Fixed-point conversion, Morton keys and stable LSD radix sorts for gfx950: the particles by their
// Morton keys (narrow keys, see below), and (64-bit key, int32 index) pairs for the initial conditions.
//
// Reference behaviour replaced: compute_morton_all + radix_histogram /
// radix_prefix_sum / radix_scatter + reorder_by_idx_* (src/nbody_gpu_twopass.rs:
// 1447-1658).  The reference sort is a stable LSD radix sort, so its output is
// the unique stable argsort of the keys; this one is too, with a parallel
// digit-major scan instead of the reference's serial per-bucket prefix loop and
// an LDS-staged tile reorder so that the scatter writes contiguous runs.
#include "jtp_internal.h"
#include "jtp_device.h"

namespace jtp {

// ------------------------------------------------------------------ fixed point
__device__ inline uint32_t to_fixed(double x, double L) {
    double t = x / L + 0.5;
    t -= floor(t);
    uint64_t w = (uint64_t)(t * 4294967296.0);
    if (w >= 4294967296ULL) w -= 4294967296ULL;
    return (uint32_t)w;
}

__global__ void k_fixed_from_f64(const double* __restrict__ pos, uint32_t* __restrict__ out, int64_t n3,
                                 double L) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n3) out[i] = to_fixed(pos[i], L);
}
__global__ void k_fixed_from_f32(const float* __restrict__ pos, uint32_t* __restrict__ out, int64_t n3,
                                 double L) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n3) out[i] = to_fixed((double)pos[i], L);
}

hipError_t launch_fixed_from_f64(const double* pos, uint32_t* out, int64_t n3, double L, hipStream_t s) {
    if (n3 > 0)
        k_fixed_from_f64<<<dim3((unsigned)((n3 + kBlock - 1) / kBlock)), dim3(kBlock), 0, s>>>(pos, out, n3, L);
    return hipGetLastError();
}
hipError_t launch_fixed_from_f32(const float* pos, uint32_t* out, int64_t n3, double L, hipStream_t s) {
    if (n3 > 0)
        k_fixed_from_f32<<<dim3((unsigned)((n3 + kBlock - 1) / kBlock)), dim3(kBlock), 0, s>>>(pos, out, n3, L);
    return hipGetLastError();
}

// ------------------------------------------------------------------ Morton keys
// Reference-compatible keys from f32 positions (compute_morton_all, nbody_gpu_twopass.rs:1458-1484):
// ix = (unsigned) fminf(fmaxf((x + box_half) * inv_cell, 0), 2^21 - 1), same interleave.
__global__ void k_morton_keys_f32(const float* __restrict__ pos, uint64_t* __restrict__ keys, int64_t n,
                                  float box_half, float inv_cell) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t c[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float g = __fmul_rn(__fadd_rn(pos[3 * i + a], box_half), inv_cell);
        c[a] = (uint32_t)fminf(fmaxf(g, 0.0f), 2097151.0f);
    }
    keys[i] = spread3_21(c[0]) | (spread3_21(c[1]) << 1) | (spread3_21(c[2]) << 2);
}

// compute_morton_f32 (nbody_gpu_twopass.rs:302-326): 10 bits per axis of (x + box_half) * 1024 / L in f32,
// the float-to-u32 conversion saturating (negative and NaN -> 0) and clamped to 1023, key = mc << 32 | i.
__device__ inline uint32_t cell10(float x) {
    return !(x > 0.0f) ? 0u : (x >= 1024.0f ? 1023u : (uint32_t)x);
}
__global__ void k_morton30_keys_f32(const float* __restrict__ pos, uint64_t* __restrict__ keys,
                                    int32_t* __restrict__ idx, int64_t n, float box_half) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float scale = __fdiv_rn(1024.0f, __fmul_rn(2.0f, box_half));
    const uint32_t cx = cell10(__fmul_rn(__fadd_rn(pos[3 * i], box_half), scale));
    const uint32_t cy = cell10(__fmul_rn(__fadd_rn(pos[3 * i + 1], box_half), scale));
    const uint32_t cz = cell10(__fmul_rn(__fadd_rn(pos[3 * i + 2], box_half), scale));
    // a 10-bit value sits in the low bits of the 21-bit spread, so spread3_21 gives the 30-bit interleave
    const uint64_t mc = spread3_21(cx) | (spread3_21(cy) << 1) | (spread3_21(cz) << 2);
    keys[i] = (mc << 32) | (uint64_t)(uint32_t)i;
    idx[i] = (int32_t)i;
}

hipError_t launch_morton30_keys_f32(const float* pos, uint64_t* keys, int32_t* idx, int64_t n, float box_half,
                                    hipStream_t s) {
    if (n > 0)
        k_morton30_keys_f32<<<dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, s>>>(pos, keys, idx, n,
                                                                                                box_half);
    return hipGetLastError();
}

hipError_t launch_morton_keys_f32(const float* pos, uint64_t* keys, int64_t n, float box_half, float inv_cell,
                                  hipStream_t s) {
    if (n > 0)
        k_morton_keys_f32<<<dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, s>>>(pos, keys, n,
                                                                                              box_half, inv_cell);
    return hipGetLastError();
}

// ------------------------------------------------------------------ radix sort
// (64-bit key, index) pairs.  Pass structure (8-bit digits, stable):
//   k_radix_hist    per-tile digit counts, stored digit-major: hist[d * nblk + b]
//   k_scan_chunks   exclusive scan of 2048-entry chunks of hist, chunk totals -> part[]
//   k_scan_part     exclusive scan of part[] (one workgroup)
//   k_radix_scatter stable in-tile ranks (wavefront bit-match + per-wave LDS counters),
//                   LDS reorder of the tile by digit, contiguous global writes.
// Digit-major exclusive prefix of the counts is exactly the global start of
// digit d's run for tile b.

constexpr int kScanChunk = 2048;

__global__ __launch_bounds__(256) void k_radix_hist(const uint64_t* __restrict__ keys, int64_t n, int shift,
                                                    uint32_t* __restrict__ hist, int nblk) {
    __shared__ uint32_t h[256];
    const int tid = threadIdx.x;
    h[tid] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kSortTile;
#pragma unroll
    for (int r = 0; r < kSortIPT; ++r) {
        int64_t idx = base + r * 256 + tid;
        if (idx < n) atomicAdd(&h[(uint32_t)(keys[idx] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[(int64_t)tid * nblk + blockIdx.x] = h[tid];
}

__global__ __launch_bounds__(256) void k_scan_chunks(uint32_t* __restrict__ data, int64_t m,
                                                     uint32_t* __restrict__ part) {
    __shared__ uint32_t lds[4];
    const int tid = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * kScanChunk + tid * 8;
    uint32_t v[8], s = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        v[i] = (base + i < m) ? data[base + i] : 0u;
        s += v[i];
    }
    uint32_t tot;
    uint32_t off = block256_excl_scan(s, lds, &tot);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if (base + i < m) data[base + i] = off;
        off += v[i];
    }
    if (tid == 0) part[blockIdx.x] = tot;
}

__global__ __launch_bounds__(256) void k_scan_part(uint32_t* __restrict__ part, int64_t np) {
    __shared__ uint32_t lds[4];
    __shared__ uint32_t carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int64_t b0 = 0; b0 < np; b0 += 256) {
        int64_t i = b0 + threadIdx.x;
        uint32_t v = (i < np) ? part[i] : 0u;
        uint32_t tot;
        uint32_t off = block256_excl_scan(v, lds, &tot);
        uint32_t c = carry;
        if (i < np) part[i] = c + off;
        __syncthreads();
        if (threadIdx.x == 0) carry = c + tot;
        __syncthreads();
    }
}

// Wavefront w of the block owns the contiguous slice [512 w, 512 w + 512) of the tile (lane l
// holds the keys at 512 w + 64 r + l, r = 0..7), so the ranks follow the input order with no
// block barrier between rounds: a round's rank is the wave's running count of the digit (its own
// LDS counters, read and then bumped by the digit's first lane, in program order within the wave)
// plus the number of earlier lanes holding the digit.  One block step then turns the per-wave
// counts into each wave's start within the tile's run of the digit.
__global__ __launch_bounds__(256) void k_radix_scatter(const uint64_t* __restrict__ kin,
                                                       const int32_t* __restrict__ vin,
                                                       uint64_t* __restrict__ kout, int32_t* __restrict__ vout,
                                                       int64_t n, int shift, const uint32_t* __restrict__ hist,
                                                       const uint32_t* __restrict__ part, int nblk) {
    static_assert(kSortTile == 4 * 64 * kSortIPT, "four wavefronts of kSortIPT keys per lane");
    __shared__ uint32_t wcnt[4][256];  // per-wave digit counts, then each wave's start in the tile
    __shared__ int64_t gbase[256];
    __shared__ uint32_t scan_lds[4];
    __shared__ uint64_t skeys[kSortTile];
    __shared__ int32_t svals[kSortTile];

    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const int b = blockIdx.x;
    const int64_t base = (int64_t)b * kSortTile;
    const int64_t wbase = base + (int64_t)w * 64 * kSortIPT + lane;
    const uint64_t lt = lanemask_lt();

    uint64_t key[kSortIPT];
    int32_t val[kSortIPT];
    uint32_t rk[kSortIPT];
#pragma unroll
    for (int r = 0; r < kSortIPT; ++r) {
        const int64_t idx = wbase + r * 64;
        if (idx < n) {
            key[r] = kin[idx];
            val[r] = vin[idx];
        } else {
            key[r] = 0;
            val[r] = 0;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) wcnt[i][tid] = 0;
    __syncthreads();

    uint32_t* mine = wcnt[w];
#pragma unroll
    for (int r = 0; r < kSortIPT; ++r) {
        const bool valid = wbase + r * 64 < n;
        const uint32_t d = (uint32_t)(key[r] >> shift) & 255u;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const bool bs = (d >> bit) & 1u;
            const uint64_t bb = __ballot(bs);
            peers &= bs ? bb : ~bb;
        }
        const uint32_t before = mine[d];
        rk[r] = before + (uint32_t)__popcll(peers & lt);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // every lane's read before the bump
        if (valid && (peers & lt) == 0) mine[d] = before + (uint32_t)__popcll(peers);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __syncthreads();
    // digit tid: the tile's run starts at toff; wave ww's keys of the digit follow those of waves < ww
    {
        const uint32_t c0 = wcnt[0][tid], c1 = wcnt[1][tid], c2 = wcnt[2][tid], c3 = wcnt[3][tid];
        const uint32_t toff = block256_excl_scan(c0 + c1 + c2 + c3, scan_lds, nullptr);
        wcnt[0][tid] = toff;
        wcnt[1][tid] = toff + c0;
        wcnt[2][tid] = toff + c0 + c1;
        wcnt[3][tid] = toff + c0 + c1 + c2;
        const int64_t hidx = (int64_t)tid * nblk + b;
        gbase[tid] = (int64_t)hist[hidx] + (int64_t)part[hidx / kScanChunk] - (int64_t)toff;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortIPT; ++r) {
        if (wbase + r * 64 < n) {
            const uint32_t d = (uint32_t)(key[r] >> shift) & 255u;
            const uint32_t l = mine[d] + rk[r];
            skeys[l] = key[r];
            svals[l] = val[r];
        }
    }
    __syncthreads();
    const int64_t cnt = (n - base) < kSortTile ? (n - base) : kSortTile;
    for (int l = tid; l < cnt; l += 256) {
        const uint64_t k = skeys[l];
        const uint32_t d = (uint32_t)(k >> shift) & 255u;
        const int64_t o = gbase[d] + l;
        kout[o] = k;
        vout[o] = svals[l];
    }
}

hipError_t radix_sort_pairs(Ctx& c, int64_t n, hipStream_t s) {
    if (n <= 1) return hipGetLastError();
    const int nblk = (int)((n + kSortTile - 1) / kSortTile);
    const int64_t m = (int64_t)nblk * 256;
    const int64_t nchunk = (m + kScanChunk - 1) / kScanChunk;
    uint64_t* ka = c.keys0;
    uint64_t* kb = c.keys1;
    int32_t* va = c.vals0;
    int32_t* vb = c.vals1;
    for (int shift = 0; shift < 64; shift += 8) {
        k_radix_hist<<<dim3(nblk), dim3(256), 0, s>>>(ka, n, shift, c.hist, nblk);
        k_scan_chunks<<<dim3((unsigned)nchunk), dim3(256), 0, s>>>(c.hist, m, c.hist_blk);
        k_scan_part<<<dim3(1), dim3(256), 0, s>>>(c.hist_blk, nchunk);
        k_radix_scatter<<<dim3(nblk), dim3(256), 0, s>>>(ka, va, kb, vb, n, shift, c.hist, c.hist_blk, nblk);
        uint64_t* tk = ka; ka = kb; kb = tk;
        int32_t* tv = va; va = vb; vb = tv;
    }
    // an even number of passes: the result is back in keys0/vals0
    return hipGetLastError();
}

// ------------------------------------------------------------------ device copy
// Streaming copy (16-byte words when both pointers and the size allow it).  Also the
// reference copy kernel for calibrating HBM byte counters.
__global__ void k_copy16(const uint4* __restrict__ src, uint4* __restrict__ dst, int64_t n16) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

hipError_t device_copy(void* dst, const void* src, size_t bytes, hipStream_t s) {
    if (bytes == 0) return hipSuccess;
    const bool aligned = (((uintptr_t)dst | (uintptr_t)src | bytes) & 15) == 0;
    if (!aligned) return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, s);
    const int64_t n16 = (int64_t)(bytes / 16);
    int64_t blocks = (n16 + kBlock - 1) / kBlock;
    if (blocks > 65536) blocks = 65536;
    k_copy16<<<dim3((unsigned)blocks), dim3(kBlock), 0, s>>>((const uint4*)src, (uint4*)dst, n16);
    return hipGetLastError();
}

// ------------------------------------------------------------------ particle sort
// Particles by the top 48 bits of their 63-bit Morton keys (kKeySortMask), stable, 8-bit digits d0 .. d5.  A
// digit that has been sorted by is not carried on: d0 and d1 travel in 2 and 1 bytes, d2 .. d5 in a 32-bit word,
// and the 64-bit keys are computed again from the records in the final gather.  (With 64-bit keys in every pass
// the passes moved 192 bytes a particle; these move 104.)
//
// Small sets (up to kSmallTiles tiles): the key kernel counts d0, every later pass counts its own digit, and the
// scatter workgroups add up the tiles' counts themselves: two launches a pass.
//
// Larger sets are first partitioned by d5 (a Morton octant prefix: 128 segments), with their 16-byte records;
// then d0 .. d4 are sorted by inside each segment, tiles and digit offsets per segment.  That takes no more
// passes, and the final gather reads records of one segment, a few MB that its XCD's L2 holds (each XCD gathers a
// contiguous part): from input order it fetched a whole 128-byte line for every 16-byte record.
//
// Measured (positions to gathered records), ms: 2e4 particles 0.17 -> 0.08, 5.2e5 0.20 -> 0.14, 1e6 0.22 -> 0.15, 4.2e6
// 0.43 -> 0.32, 2.2e7 1.96 -> 1.36.
constexpr int kSegs = 128;          // d5 has 7 bits: bit 63 of a key is 0
constexpr int kSmallTiles = 128;    // a scatter workgroup reads this many tiles' counts: ~3 us; above (2.6e5 particles)
                                    // segments are the faster path (5.2e5: 0.14 ms against 0.18 with 6144-key tiles)
constexpr int kSmallIpt = 8;        // keys per thread of small tiles (2048): 10 tiles at 2e4 particles
constexpr int kPartIpt = 8;         // the partition holds 16-byte records in LDS
constexpr int kPartTile = kBlock * kPartIpt;

__device__ inline uint64_t key48(uint32_t x, uint32_t y, uint32_t z) { return morton_fixed(x, y, z) >> kKeyLowBits; }

struct SortArgs {
    int64_t n;
    const uint32_t* hi_in;    // digits above those already sorted by
    const void* lo_in;        // d0 and d1 (uint16) or the one of them left (uint8)
    const uint32_t* val_in;
    uint32_t* hi_out;
    uint8_t* lo_out;
    uint32_t* val_out;
    uint32_t* hist;           // counts [tile][256], then (segments) those of the segment's tiles before
    const uint32_t* seg_tot;  // particles of each segment; nullptr: one segment
    uint32_t* dig_tot;        // segments: counts [segment][256]
    int32_t nblk;             // tiles (one segment)
    int32_t shift;            // of the digit in hi_in
};

// Tile `b` of the segments' tiles: its particles [base, base + cnt), its segment and that one's start; false beyond the last.
// 256 threads or more, all of them; seg >= 0 asks for a segment instead: base its start, cnt its tiles, b its first tile.
template <int TILE>
__device__ inline bool seg_find(const uint32_t* __restrict__ tot, int& seg, int& b, int64_t& base, int& cnt,
                                uint32_t& seg_start, uint32_t* lds /* 10 */) {
    const int t = threadIdx.x;
    if (t == 4) lds[4] = 0;
    const uint32_t c = t < kSegs ? tot[t] : 0;
    const uint32_t nt = (c + TILE - 1) / TILE;
    uint32_t ci = (uint32_t)wave_incl_scan_dpp((int)c), ti = (uint32_t)wave_incl_scan_dpp((int)nt);
    if (t == 63) {
        lds[0] = ci;
        lds[1] = ti;
    }
    __syncthreads();
    if (t >= 64 && t < kSegs) {
        ci += lds[0];
        ti += lds[1];
    }
    if (t < kSegs && (seg >= 0 ? t == seg : (uint32_t)b >= ti - nt && (uint32_t)b < ti)) {
        lds[4] = 1;
        lds[8] = (uint32_t)t;
        lds[9] = ci - c;
        if (seg >= 0) {
            lds[5] = ci - c;
            lds[6] = nt;
            lds[7] = ti - nt;
        } else {
            const uint32_t off = ((uint32_t)b - (ti - nt)) * TILE;
            lds[5] = ci - c + off;
            lds[6] = c - off < TILE ? c - off : TILE;
            lds[7] = (uint32_t)b;
        }
    }
    __syncthreads();
    base = lds[5];
    cnt = (int)lds[6];
    b = (int)lds[7];
    seg = (int)lds[8];
    seg_start = lds[9];
    return lds[4] != 0;
}

// Keys and packed records (x, y, z, species) in input order, and each tile's counts of d0.
template <int IPT>
__global__ __launch_bounds__(256) void k_sort_keys(const uint32_t* __restrict__ pos, const int8_t* __restrict__ species,
                                                   int64_t n, uint4* __restrict__ rec, uint16_t* __restrict__ lo,
                                                   uint32_t* __restrict__ hi, uint32_t* __restrict__ hist) {
    __shared__ uint32_t h[256];
    const int tid = threadIdx.x;
    h[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const int64_t i = (int64_t)blockIdx.x * (256 * IPT) + r * 256 + tid;
        if (i < n) {
            const uint32_t x = pos[3 * i], y = pos[3 * i + 1], z = pos[3 * i + 2];
            const uint64_t k = key48(x, y, z);
            rec[i] = make_uint4(x, y, z, (uint32_t)(int32_t)species[i]);
            lo[i] = (uint16_t)k;
            hi[i] = (uint32_t)(k >> 16);
            atomicAdd(&h[(uint32_t)k & 255u], 1u);
        }
    }
    __syncthreads();
    hist[(int64_t)blockIdx.x * 256 + tid] = h[tid];
}

// Each tile's counts of the pass's digit.
template <int IPT, int LO, bool SEG>
__global__ __launch_bounds__(256) void k_sort_hist(SortArgs a) {
    __shared__ uint32_t h[256];
    __shared__ uint32_t lds[10];
    const int tid = threadIdx.x;
    constexpr int TILE = 256 * IPT;
    int b = (int)blockIdx.x, cnt, seg = -1;
    uint32_t seg_start = 0;
    int64_t base = (int64_t)b * TILE;
    if (SEG) {
        if (!seg_find<TILE>(a.seg_tot, seg, b, base, cnt, seg_start, lds)) return;
    } else {
        cnt = a.n - base < TILE ? (int)(a.n - base) : TILE;
    }
    h[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const int l = r * 256 + tid;
        if (l < cnt) {
            const uint32_t d = LO == 8 ? (uint32_t)((const uint8_t*)a.lo_in)[base + l]
                                       : (a.hi_in[base + l] >> a.shift) & 255u;
            atomicAdd(&h[d], 1u);
        }
    }
    __syncthreads();
    a.hist[(int64_t)b * 256 + tid] = h[tid];
}

// Each tile's counts -> those of its segment's tiles before it, and the segment's counts.  A workgroup takes DIG digits of one
// segment, its 1024 / DIG groups of threads a run of the tiles each.  Several workgroups a segment, because a set may lie in
// one of them: with one each and four runs a digit, 4.1e6 particles of one octant cell took 1.50 ms to sort (1.22 with 32
// digits a workgroup, 1.34 with 128) and 2.2e7 took 2.75 (2.41; 2.48 with 64).  The workgroups cost 3 us a pass at 32 digits
// where the tiles are few, nothing at 128 (3e5 and 1e6 particles in a full box: 0.10 and 0.13 ms to sort; with 32 0.11 and 0.15).
constexpr int64_t kScanWide = (int64_t)2 << 20;  // 32 digits from this many particles (4.1e6 crowded: 1.88 ms a call before
                                                // the segments, 1.93 with 128 digits, 1.85 with 32)
template <int TILE, int DIG>
__global__ __launch_bounds__(1024) void k_sort_segscan(SortArgs a) {
    constexpr int RUNS = 1024 / DIG;
    __shared__ uint32_t part[RUNS][DIG];
    __shared__ uint32_t lds[10];
    const int g = threadIdx.x / DIG, dd = threadIdx.x % DIG, d = (int)blockIdx.y * DIG + dd;
    int seg = (int)blockIdx.x, first = 0, nt;
    uint32_t seg_start;
    int64_t start;
    if (!seg_find<TILE>(a.seg_tot, seg, first, start, nt, seg_start, lds)) return;
    if (nt == 0) return;
    const int q = (nt + RUNS - 1) / RUNS, t0 = g * q < nt ? g * q : nt, t1 = t0 + q < nt ? t0 + q : nt;
    uint32_t* h = a.hist + (int64_t)first * 256 + d;
    uint32_t s = 0;
#pragma unroll 8
    for (int t = t0; t < t1; ++t) s += h[(int64_t)t * 256];
    part[g][dd] = s;
    __syncthreads();
    uint32_t run = 0;
    for (int i = 0; i < g; ++i) run += part[i][dd];
    if (g == RUNS - 1) a.dig_tot[seg * 256 + d] = run + s;
#pragma unroll 8
    for (int t = t0; t < t1; ++t) {
        const uint32_t v = h[(int64_t)t * 256];
        h[(int64_t)t * 256] = run;
        run += v;
    }
}

// In-tile stable ranks: wavefront w owns the contiguous slice [64 IPT w, 64 IPT (w + 1)) of the tile (lane l holds the
// keys at 64 r + l of it), so the ranks follow the input order with no barrier between rounds: a round's rank is the
// wave's running count of the digit (its own LDS counters, read and then bumped by the digit's first lane, in program
// order within the wave) plus the number of earlier lanes holding the digit.  Then the per-wave counts become each
// wave's start within the tile's run of the digit; returns the tile's start of digit tid.
template <int IPT>
__device__ inline uint32_t tile_ranks(const uint32_t dig[IPT], int nmine, uint16_t (*wcnt)[256], uint32_t* scan_lds,
                                      uint16_t rk[IPT], int bits) {
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const uint64_t lt = lanemask_lt();
#pragma unroll
    for (int i = 0; i < 4; ++i) wcnt[i][tid] = 0;
    __syncthreads();
    uint16_t* mine = wcnt[w];
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const bool valid = r * 64 + lane < nmine;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            if (bit >= bits) break;
            const bool bs = (dig[r] >> bit) & 1u;
            const uint64_t bb = __ballot(bs);
            peers &= bs ? bb : ~bb;
        }
        const uint32_t before = mine[dig[r]];
        rk[r] = (uint16_t)(before + (uint32_t)__popcll(peers & lt));
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // every lane's read before the bump
        if (valid && (peers & lt) == 0) mine[dig[r]] = (uint16_t)(before + (uint32_t)__popcll(peers));
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __syncthreads();
    const uint32_t c0 = wcnt[0][tid], c1 = wcnt[1][tid], c2 = wcnt[2][tid], c3 = wcnt[3][tid];
    const uint32_t toff = block256_excl_scan(c0 + c1 + c2 + c3, scan_lds, nullptr);
    wcnt[0][tid] = (uint16_t)toff;
    wcnt[1][tid] = (uint16_t)(toff + c0);
    wcnt[2][tid] = (uint16_t)(toff + c0 + c1);
    wcnt[3][tid] = (uint16_t)(toff + c0 + c1 + c2);
    return toff;
}

// One pass: ranks in the tile, the tile reordered by digit in LDS, contiguous global writes.
template <int IPT, int LO, bool IDENT, bool KEYOUT, bool SEG>
__global__ __launch_bounds__(256) void k_sort_scatter(SortArgs a) {
    constexpr int TILE = 256 * IPT;
    using LoT = typename std::conditional<LO == 16, uint16_t, uint8_t>::type;
    __shared__ uint16_t wcnt[4][256];
    __shared__ uint32_t gbase[256];
    __shared__ uint32_t lds[10];
    __shared__ uint32_t shi[TILE];
    __shared__ uint32_t sval[TILE];
    __shared__ LoT slo[LO ? TILE : 1];
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    int b = (int)blockIdx.x, cnt, seg = -1;
    uint32_t seg_start = 0;
    int64_t base = (int64_t)b * TILE;
    if (SEG) {
        if (!seg_find<TILE>(a.seg_tot, seg, b, base, cnt, seg_start, lds)) return;
    } else {
        cnt = a.n - base < TILE ? (int)(a.n - base) : TILE;
    }
    const int w0 = w * 64 * IPT;
    const int nmine = cnt - w0 < 0 ? 0 : (cnt - w0 < 64 * IPT ? cnt - w0 : 64 * IPT);
    uint32_t hi[IPT], val[IPT], dig[IPT];
    LoT lo[IPT];
    uint16_t rk[IPT];
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const int l = r * 64 + lane;
        const int64_t i = base + w0 + l;
        const bool in = l < nmine;
        hi[r] = in ? a.hi_in[i] : 0;
        val[r] = IDENT ? (uint32_t)i : (in ? a.val_in[i] : 0);
        lo[r] = LO && in ? ((const LoT*)a.lo_in)[i] : (LoT)0;
        dig[r] = LO ? (uint32_t)lo[r] & 255u : (hi[r] >> a.shift) & 255u;
    }
    // where the tile's run of digit tid starts
    uint32_t before = 0, tot = 0;
    if (SEG) {
        before = seg_start + a.hist[(int64_t)b * 256 + tid];
        tot = a.dig_tot[seg * 256 + tid];
    } else {
#pragma unroll 16
        for (int t = 0; t < a.nblk; ++t) {
            const uint32_t v = a.hist[t * 256 + tid];
            before += t < b ? v : 0;
            tot += v;
        }
    }
    const uint32_t start = block256_excl_scan(tot, lds, nullptr) + before;
    const uint32_t toff = tile_ranks<IPT>(dig, nmine, wcnt, lds, rk, 8);
    gbase[tid] = start - toff;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        if (r * 64 + lane < nmine) {
            const uint32_t l = (uint32_t)wcnt[w][dig[r]] + rk[r];
            shi[l] = hi[r];
            sval[l] = val[r];
            if (LO) slo[l] = lo[r];
        }
    }
    __syncthreads();
#pragma unroll 4
    for (int l = tid; l < cnt; l += 256) {
        const uint32_t h = shi[l];
        const uint32_t x = LO ? (uint32_t)slo[l] : 0u;
        const uint32_t d = LO ? x & 255u : (h >> a.shift) & 255u;
        const uint32_t o = gbase[d] + (uint32_t)l;
        if (KEYOUT) a.hi_out[o] = h;
        if (LO == 16) a.lo_out[o] = (uint8_t)(x >> 8);
        a.val_out[o] = sval[l];
    }
}

// ---- partition by d5
__device__ inline uint32_t top_digit(uint32_t x, uint32_t y, uint32_t z) { return (uint32_t)(morton_fixed(x, y, z) >> 56); }

// Counts of d5, digit-major: hist[d * nblk + b].
__global__ __launch_bounds__(256) void k_part_hist(const uint32_t* __restrict__ pos, int64_t n,
                                                   uint32_t* __restrict__ hist, int nblk) {
    __shared__ uint32_t h[kSegs];
    const int tid = threadIdx.x;
    if (tid < kSegs) h[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPartIpt; ++r) {
        const int64_t i = (int64_t)blockIdx.x * kPartTile + r * 256 + tid;
        if (i < n) atomicAdd(&h[top_digit(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2])], 1u);
    }
    __syncthreads();
    if (tid < kSegs) hist[(int64_t)tid * nblk + blockIdx.x] = h[tid];
}

// One workgroup per digit: exclusive scan over the tiles; tot[d] = the digit's total.
__global__ __launch_bounds__(1024) void k_part_scan(uint32_t* __restrict__ hist, int nblk, uint32_t* __restrict__ tot) {
    __shared__ uint32_t lds[16];
    const int tid = threadIdx.x, w = tid >> 6;
    uint32_t* h = hist + (int64_t)blockIdx.x * nblk;
    uint32_t carry = 0;
    for (int t0 = 0; t0 < nblk; t0 += 4096) {  // four consecutive tiles per thread
        uint32_t v[4], s = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int t = t0 + 4 * tid + k;
            v[k] = t < nblk ? h[t] : 0;
            s += v[k];
        }
        const uint32_t incl = (uint32_t)wave_incl_scan_dpp((int)s);
        if ((tid & 63) == 63) lds[w] = incl;
        __syncthreads();
        uint32_t off = carry + incl - s;
        for (int i = 0; i < 16; ++i) {
            if (i < w) off += lds[i];
            carry += lds[i];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int t = t0 + 4 * tid + k;
            if (t < nblk) h[t] = off;
            off += v[k];
        }
    }
    if (tid == 0) tot[blockIdx.x] = carry;
}

// Records (x, y, z, input index << 1 | species +1) and the lower 40 key bits, in segment order.
__global__ __launch_bounds__(256) void k_part_scatter(const uint32_t* __restrict__ pos,
                                                      const int8_t* __restrict__ species, int64_t n,
                                                      const uint32_t* __restrict__ hist, int nblk,
                                                      const uint32_t* __restrict__ tot, uint4* __restrict__ rec,
                                                      uint8_t* __restrict__ lo, uint32_t* __restrict__ hi) {
    __shared__ uint16_t wcnt[4][256];
    __shared__ uint32_t gbase[256];
    __shared__ uint32_t lds[8];
    __shared__ uint4 srec[kPartTile];
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const int64_t base = (int64_t)blockIdx.x * kPartTile;
    const int cnt = n - base < kPartTile ? (int)(n - base) : kPartTile;
    const int w0 = w * 64 * kPartIpt;
    const int nmine = cnt - w0 < 0 ? 0 : (cnt - w0 < 64 * kPartIpt ? cnt - w0 : 64 * kPartIpt);
    uint4 q[kPartIpt];
    uint32_t dig[kPartIpt];
    uint16_t rk[kPartIpt];
#pragma unroll
    for (int r = 0; r < kPartIpt; ++r) {
        const int l = r * 64 + lane;
        const int64_t i = base + w0 + l;
        q[r] = make_uint4(0u, 0u, 0u, 0u);
        if (l < nmine)
            q[r] = make_uint4(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], ((uint32_t)i << 1) | (species[i] > 0 ? 1u : 0u));
        dig[r] = top_digit(q[r].x, q[r].y, q[r].z);
    }
    const uint32_t segtot = tid < kSegs ? tot[tid] : 0;
    uint32_t start = block256_excl_scan(segtot, lds, nullptr);
    if (tid < kSegs) start += hist[(int64_t)tid * nblk + blockIdx.x];
    const uint32_t toff = tile_ranks<kPartIpt>(dig, nmine, wcnt, lds, rk, 7);
    gbase[tid] = start - toff;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPartIpt; ++r)
        if (r * 64 + lane < nmine) srec[(uint32_t)wcnt[w][dig[r]] + rk[r]] = q[r];
    __syncthreads();
#pragma unroll 4
    for (int l = tid; l < cnt; l += 256) {
        const uint4 r = srec[l];
        const uint64_t k = key48(r.x, r.y, r.z);
        const uint32_t o = gbase[(uint32_t)(k >> 40)] + (uint32_t)l;
        rec[o] = r;
        lo[o] = (uint8_t)k;
        hi[o] = (uint32_t)(k >> 8);
    }
}

// ---- gather
// parts[i] = (x, y, z, species) of the i-th particle in key order (reorder_by_idx_*, nbody_gpu_twopass.rs:1490-1514, fused
// into one 16-byte record), its key and its input index.  With ts, also the start of every Morton-aligned tile of 8^3 PM
// cells (lt = log2 G - 3 tile bits per axis; the tile index is a prefix of the key), and with cells that of every level
// kGroupLevelBits cell that holds any (the walk's groups; a search of the keys for them took 20 us at 2e4 particles and
// 44 beside other boxes' work): the particle that begins a run of tiles writes the starts of the tiles up to its own, so
// every entry is written once, ts[ntile] = n.  Lanes read the previous particle's tile from their neighbour; lane 0
// gathers it again.  SEG: records in segment order with the input index beside the species, workgroups dealt so that each
// XCD gathers a contiguous part.
template <bool SEG>
__global__ __launch_bounds__(256) void k_gather_parts(const uint4* __restrict__ rec, const uint32_t* __restrict__ idx,
                                                      uint4* __restrict__ parts, uint64_t* __restrict__ keys,
                                                      int32_t* __restrict__ perm, int64_t n, int32_t* __restrict__ ts,
                                                      int lt, int32_t* __restrict__ cells) {
    int64_t blk = blockIdx.x;
    if (SEG) blk = (int64_t)(blockIdx.x % kXcds) * (gridDim.x / kXcds) + blockIdx.x / kXcds;
    const int64_t i = blk * blockDim.x + threadIdx.x;
    const bool in = i < n;
    const bool edge = (threadIdx.x & 63) == 0 && i > 0 && in && (ts || cells);
    uint4 r = make_uint4(0u, 0u, 0u, 0u), before = r;
    if (edge) before = rec[idx[i - 1]];
    if (in) {
        const uint32_t k = idx[i];
        r = rec[k];
        perm[i] = (int32_t)(SEG ? r.w >> 1 : k);
        if (SEG) r.w = r.w & 1u ? 1u : 0xffffffffu;
        parts[i] = r;
        keys[i] = morton_fixed(r.x, r.y, r.z) & kKeySortMask;
    }
    auto tile_of = [&](const uint4& q, int sh) {
        return (int32_t)(spread3_21(q.x >> sh) | (spread3_21(q.y >> sh) << 1) | (spread3_21(q.z >> sh) << 2));
    };
    if (cells) {
        const int32_t c = in ? tile_of(r, 32 - kGroupLevelBits) : -1;
        int32_t cp = __shfl_up(c, 1, 64);
        if ((threadIdx.x & 63) == 0) cp = edge ? tile_of(before, 32 - kGroupLevelBits) : -1;
        if (in && c != cp) cells[c] = (int32_t)i;
    }
    if (!ts) return;
    const int sh = 32 - lt;
    const int32_t ntile = 1 << (3 * lt);
    const int32_t tc = in ? tile_of(r, sh) : ntile;
    int32_t tp = __shfl_up(tc, 1, 64);
    if ((threadIdx.x & 63) == 0) tp = edge ? tile_of(before, sh) : -1;
    if (!in) return;
    for (int32_t t = tp + 1; t <= tc; ++t) ts[t] = (int32_t)i;
    if (i == n - 1)
        for (int32_t t = tc + 1; t <= ntile; ++t) ts[t] = (int32_t)n;
}

// ---- host side
template <int IPT, int LO, bool IDENT, bool KEYOUT, bool SEG>
static void sort_pass(const SortArgs& a, unsigned nblk, bool counted, hipStream_t s) {
    if (!counted) k_sort_hist<IPT, LO, SEG><<<dim3(nblk), dim3(256), 0, s>>>(a);
    if (SEG && a.n < kScanWide) k_sort_segscan<256 * IPT, 128><<<dim3(kSegs, 2), dim3(1024), 0, s>>>(a);
    else if (SEG) k_sort_segscan<256 * IPT, 32><<<dim3(kSegs, 8), dim3(1024), 0, s>>>(a);
    k_sort_scatter<IPT, LO, IDENT, KEYOUT, SEG><<<dim3(nblk), dim3(256), 0, s>>>(a);
}

// One segment; the result (input indices in key order) in vals1.
template <int IPT>
static void sort_small(Ctx& c, const uint32_t* pos, const int8_t* species, uint4* rec, int64_t n, hipStream_t s) {
    const unsigned nblk = (unsigned)((n + 256 * IPT - 1) / (256 * IPT));
    uint32_t *ha = (uint32_t*)c.keys1, *hb = ha + c.cap_n;
    uint16_t* lo16 = (uint16_t*)c.keys0;
    uint8_t* lo8 = (uint8_t*)c.keys0 + 2 * c.cap_n;
    uint32_t *v0 = (uint32_t*)c.vals0, *v1 = (uint32_t*)c.vals1;
    k_sort_keys<IPT><<<dim3(nblk), dim3(256), 0, s>>>(pos, species, n, rec, lo16, ha, c.hist);
    SortArgs a{};
    a.n = n;
    a.hist = c.hist;
    a.nblk = (int32_t)nblk;
    a.hi_in = ha; a.hi_out = hb; a.lo_in = lo16; a.lo_out = lo8; a.val_out = v0;
    sort_pass<IPT, 16, true, true, false>(a, nblk, true, s);
    a.hi_in = hb; a.hi_out = ha; a.lo_in = lo8; a.val_in = v0; a.val_out = v1;
    sort_pass<IPT, 8, false, true, false>(a, nblk, false, s);
    for (int p = 0; p < 3; ++p) {  // d2, d3, d4
        a.hi_in = p & 1 ? hb : ha; a.hi_out = p & 1 ? ha : hb;
        a.val_in = p & 1 ? v0 : v1; a.val_out = p & 1 ? v1 : v0;
        a.shift = 8 * p;
        sort_pass<IPT, 0, false, true, false>(a, nblk, false, s);
    }
    a.hi_in = hb; a.val_in = v0; a.val_out = v1; a.shift = 24;
    sort_pass<IPT, 0, false, false, false>(a, nblk, false, s);
}

// Partitioned by d5; the result (places in segment order) in vals1.
template <int IPT>
static void sort_segments(Ctx& c, const uint32_t* pos, const int8_t* species, uint4* rec, int64_t n, hipStream_t s) {
    const int npart = (int)((n + kPartTile - 1) / kPartTile);
    const unsigned nblk = (unsigned)(n / (256 * IPT) + kSegs);  // at most: every segment ends with a partial tile
    uint32_t *ha = (uint32_t*)c.keys1, *hb = ha + c.cap_n;
    uint8_t* lo8 = (uint8_t*)c.keys0;
    uint32_t *v0 = (uint32_t*)c.vals0, *v1 = (uint32_t*)c.vals1;
    uint32_t* tot = c.hist;  // kSegs totals, 256 of each segment, then the counts
    uint32_t* dig = c.hist + kSegs;
    uint32_t* hist = dig + kSegs * 256;
    k_part_hist<<<dim3(npart), dim3(256), 0, s>>>(pos, n, hist, npart);
    k_part_scan<<<dim3(kSegs), dim3(1024), 0, s>>>(hist, npart, tot);
    k_part_scatter<<<dim3(npart), dim3(256), 0, s>>>(pos, species, n, hist, npart, tot, rec, lo8, ha);
    SortArgs a{};
    a.n = n;
    a.hist = hist;
    a.seg_tot = tot;
    a.dig_tot = dig;
    a.hi_in = ha; a.hi_out = hb; a.lo_in = lo8; a.val_out = v1;
    sort_pass<IPT, 8, true, true, true>(a, nblk, false, s);
    for (int p = 0; p < 3; ++p) {  // d1, d2, d3
        a.hi_in = p & 1 ? ha : hb; a.hi_out = p & 1 ? hb : ha;
        a.val_in = p & 1 ? v0 : v1; a.val_out = p & 1 ? v1 : v0;
        a.shift = 8 * p;
        sort_pass<IPT, 0, false, true, true>(a, nblk, false, s);
    }
    a.hi_in = ha; a.val_in = v0; a.val_out = v1; a.shift = 24;
    sort_pass<IPT, 0, false, false, true>(a, nblk, false, s);
}

// Counts: the small path's kSmallTiles tiles, or the segments' tiles and totals (tiles of 2048 at least), or the
// partition's tiles.
int64_t sort_hist_size(int64_t cap) { return (cap / (256 * kSmallIpt) + 2 * kSegs + 1) * 256 + kSegs; }

hipError_t sort_particles(Ctx& c, const uint32_t* pos, const int8_t* species, int64_t n, int32_t* ts, int32_t* cells,
                          hipStream_t s) {
    if (n <= 0) {
        if (!ts) return hipGetLastError();
        return launch_fill_i32(ts, ((int64_t)1 << (3 * (c.logG - 3))) + 1, 0, s);
    }
    uint4* rec = (uint4*)c.node_sum;  // until the tree build, which follows the gather
    const uint32_t* idx = (const uint32_t*)c.vals1;
    const unsigned nb = (unsigned)((n + kBlock - 1) / kBlock);
    const int lt = c.logG - 3;
    if (n <= (int64_t)kSmallTiles * 256 * kSmallIpt) {
        sort_small<kSmallIpt>(c, pos, species, rec, n, s);
        k_gather_parts<false><<<dim3(nb), dim3(kBlock), 0, s>>>(rec, idx, c.parts, c.keys0, c.vals0, n, ts, lt, cells);
    } else {
        // tiles of 6144 once there are enough for the CUs: longer runs per digit
        if (n < (int64_t)4 << 20) sort_segments<kSmallIpt>(c, pos, species, rec, n, s);
        else sort_segments<kSortIPT>(c, pos, species, rec, n, s);
        const unsigned nbx = (nb + kXcds - 1) / kXcds * kXcds;
        k_gather_parts<true><<<dim3(nbx), dim3(kBlock), 0, s>>>(rec, idx, c.parts, c.keys0, c.vals0, n, ts, lt, cells);
    }
    return hipGetLastError();
}

}  // namespace jtp
