// k_bin.hip -- tile binning by direct placement (the render/train fast path).
//
// Replaces duplicate-with-keys + the pair sort (tile_binner_cpu.cpp:59-99,
// sorter_cpu.cpp:6-44; scatter.cl:73-154 + radix_sort_kv_cl.h) with the same
// result: per tile, the indices of the Gaussians whose tile rectangle covers
// it, in (depth bits, index) order, plus [start, end) ranges (empty tiles
// (0, 0)).
//
// Input is each view's Gaussians in depth order: a stable sort by the float
// bits of depth, so equal depths keep index order, with culled Gaussians last.
// Two levels, because a Gaussian covers tens of tiles but few bins of 4 x 4
// tiles (47 tiles, 6 bins on average at 1M Gaussians, 1080p):
//
//   level 1, bin lists: the depth order is cut into chunks (bin_layout).
//     coarse_count:  per (chunk, bin) the Gaussians whose rectangle meets the
//                    bin, by a difference array over the bin grid in LDS (four
//                    LDS atomics per Gaussian, whatever its size).
//     coarse_scan, coarse_starts: each bin's column of that table scanned over
//                    the chunks, then the bins' totals scanned: the place of
//                    every (bin, chunk) run in one array of records.
//     coarse_place:  every Gaussian writes a record (index, mask of the bin's
//                    tiles its rectangle covers) into each of its bins'
//                    runs.  The rank inside a run comes from one 64-bit lane
//                    mask per (wave, bin) in LDS: a lane sets its bit in its
//                    bins' masks and counts the bits below its own, so order is
//                    kept and no record is moved twice.
//   level 2, tile lists: a bin's records are cut into C2 groups of chunks.
//     tile_count:    per (tile, group) the records whose mask has the tile.
//     scan:          one exclusive scan of that tile-major table gives every
//                    (tile, group)'s first slot, the tiles' starts and the total.
//     tile_place:    a wave owns one row of tiles of a bin and a group; it
//                    reads 64 records at a time and, per tile, compacts the
//                    indices whose bit is set with one ballot: the slots of one
//                    step are consecutive, so a store is one run of up to 64
//                    indices and a tile's cursor is one scalar.
//   ranges: (start, end) of a tile are the scanned entries of its first group
//           and of the next tile's first group.
//
// What bounds it: the pairs' 4 bytes written once (189 MB at 1M Gaussians,
// 1080p), the records (8 bytes, 6 per Gaussian, scattered in short runs)
// written once and read twice, and the launches' latency at small sizes.
// One level (a wave per group of Gaussians and 8 x 8-tile bin, one visit per
// Gaussian and bin, 15 of 64 lanes live) took 377 us for those 47M pairs, and
// 275 us where a first raster round let it skip part of them; these kernels
// take 53 (coarse_place), 26 (tile_count) and 67 us (tile_place), 2.8 TB/s of
// pairs.  At 10k Gaussians and 256 x 256 pixels placement went from 165 to
// 5 us, at 1M and 4K from 1004 to 261 us, at 16 views of 1M (371M pairs) from
// 2740 to 869 us.
#include "gs_device.h"
#include "gs_internal.h"
#include "gs_wave.h"

namespace gsb {

// A bin is BT x BT tiles; a record is a Gaussian index and the mask of the
// bin's tiles it covers (bit BT * y + x).
template <int BT>
struct Bins;
template <>
struct Bins<4> {
    using Rec = uint2;  // (index, mask)
};
template <>
struct Bins<8> {
    using Rec = uint4;  // (index, unused, mask low, mask high)
};

struct Rect {
    int x0, y0, x1, y1;  // half open
    __device__ __forceinline__ explicit Rect(uint32_t R)
        : x0((int)(R & 0xFFu)), y0((int)((R >> 16) & 0xFFu)), x1((int)((R >> 8) & 0xFFu)), y1((int)(R >> 24)) {}
    __device__ __forceinline__ bool empty() const { return x0 >= x1 || y0 >= y1; }
};

// The bins a rectangle meets, [x0, x1) x [y0, y1) of the bin grid.
template <int BT>
__device__ __forceinline__ Rect bins_of(const Rect& t) {
    Rect b(0u);
    if (!t.empty()) {
        b.x0 = t.x0 / BT;
        b.y0 = t.y0 / BT;
        b.x1 = (t.x1 + BT - 1) / BT;
        b.y1 = (t.y1 + BT - 1) / BT;
    }
    return b;
}

// Bits [a, b) of a word, 0 <= a, b <= 32.
__device__ __forceinline__ uint32_t bits_range(int a, int b) {
    const uint32_t lo = a < 32 ? ~0u << a : 0u;
    return b < 32 ? lo & ~(~0u << b) : lo;
}

template <int BT>
__device__ __forceinline__ typename Bins<BT>::Rec make_record(uint32_t id, const Rect& t, int bx, int by) {
    const int xa = max(t.x0 - BT * bx, 0), xb = min(t.x1 - BT * bx, BT);
    const int ya = max(t.y0 - BT * by, 0), yb = min(t.y1 - BT * by, BT);
    const uint32_t row = bits_range(xa, xb);
    if constexpr (BT == 4) {
        return make_uint2(id, (row * 0x1111u) & bits_range(4 * ya, 4 * yb));
    } else {
        const uint32_t rows = row * 0x01010101u;
        return make_uint4(id, 0u, rows & bits_range(min(8 * ya, 32), min(8 * yb, 32)),
                          rows & bits_range(max(8 * ya - 32, 0), max(8 * yb - 32, 0)));
    }
}

// The mask bits of tile row y, in the low BT bits.
__device__ __forceinline__ uint32_t mask_row(const uint2& r, int y) { return r.y >> (4 * y); }
__device__ __forceinline__ uint32_t mask_row(const uint4& r, int y) { return (y < 4 ? r.z : r.w) >> (8 * (y & 3)); }

__device__ __forceinline__ int4 view_info(const BinArgs& a, int v) { return a.views ? a.views[v] : a.view0; }

// The Gaussian of depth rank r of view v and its packed tile rectangle
// (x0 | x1 << 8 | y0 << 16 | y1 << 24; 0 when culled).
__device__ __forceinline__ uint2 rect_record(const BinArgs& a, int v, const int4& vi, uint32_t r) {
    const size_t seg = (size_t)v * a.N;
    const uint32_t id = a.sidx ? a.sidx[(seg + r) * (size_t)a.sidx_stride] >> a.sidx_shift : r;
    if (a.rect_idx) return make_uint2(a.rect_idx[seg + id], id);  // packed beforehand, in index order
    const int rad = a.radii[seg + id];
    uint2 rec = make_uint2(0u, id);
    if (rad > 0) {
        const float2 m = a.means2D[seg + id];
        int mn[2], mx[2];
        gsd::get_rect(m.x, m.y, rad, vi.x, vi.y, mn, mx);
        rec.x = (uint32_t)mn[0] | ((uint32_t)mx[0] << 8) | ((uint32_t)mn[1] << 16) | ((uint32_t)mx[1] << 24);
    }
    return rec;
}

// Depth ranks [r0, r1) of chunk c: the first S chunks hold 256, the others CH.
__device__ __forceinline__ void chunk_ranks(const BinArgs& a, int c, uint32_t& r0, uint32_t& r1) {
    const int late = max(c - a.S, 0);
    r0 = 256u * (uint32_t)(c - late) + (uint32_t)a.CH * (uint32_t)late;
    r1 = min(r0 + (c < a.S ? 256u : (uint32_t)a.CH), (uint32_t)a.N);
}

// One block per (view, chunk): the depth-ordered rectangle records of the
// chunk and its count in every bin of the view.
//
// Here and in coarse_place the chunks go round the XCDs one by one, not in a run
// to each: the nearest chunks have the most records and the last ones, of culled
// Gaussians, none, so with runs one XCD had most of the work (4M Gaussians, 1.7M
// of them in view, 1080p: coarse_count 61 -> 41 us, coarse_place 133 -> 91; 1M,
// all in view: 12.6 -> 12.7 and 54.6 -> 50.9).  From eight views on a run is a
// whole view or more, and this kernel keeps the runs: the rectangles it gathers
// from are then in one L2 (16 views of 1M: 156 us against 235).
template <int BT>
__global__ __launch_bounds__(256) void coarse_count_kernel(BinArgs a) {
    __shared__ int dif[2 * GS_BIN_MAX_BINS];  // (columns + 1) x (rows + 1)
    const int q = a.V >= 8 ? gsd::xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x;
    const int v = q / a.C1, c = q - v * a.C1;
    const int4 vi = view_info(a, v);
    const int nbx = (vi.x + BT - 1) / BT, nby = (vi.y + BT - 1) / BT, W1 = nbx + 1;
    const int tid = threadIdx.x;
    for (int i = tid; i < W1 * (nby + 1); i += 256) dif[i] = 0;
    __syncthreads();
    uint32_t r0, r1;
    chunk_ranks(a, c, r0, r1);
    for (uint32_t r = r0 + (uint32_t)tid; r < r1; r += 256u) {
        const uint2 rec = rect_record(a, v, vi, r);
        a.rects[(size_t)v * a.N + r] = rec;
        const Rect t(rec.x);
        if (!t.empty()) {
            const Rect b = bins_of<BT>(t);
            atomicAdd(&dif[b.y0 * W1 + b.x0], 1);
            atomicAdd(&dif[b.y0 * W1 + b.x1], -1);
            atomicAdd(&dif[b.y1 * W1 + b.x0], -1);
            atomicAdd(&dif[b.y1 * W1 + b.x1], 1);
        }
    }
    __syncthreads();
    if (tid < nby) {
        int* row = dif + tid * W1;
        int s = 0;
#pragma unroll 4
        for (int x = 0; x < nbx; x++) {
            s += row[x];
            row[x] = s;
        }
    }
    __syncthreads();
    uint32_t* tab = a.table1 + (size_t)c * a.NB + (uint32_t)vi.z;
    if (tid < nbx) {
        int s = 0;
#pragma unroll 4
        for (int y = 0; y < nby; y++) {
            s += dif[y * W1 + tid];
            tab[y * nbx + tid] = (uint32_t)s;
        }
    }
}

// Each bin's column of the (chunk, bin) table turned into its exclusive scan
// over the chunks, and the bin's total: 16 bins (one 64-byte row segment) per
// block, the chunks split over 64 slices.
__global__ __launch_bounds__(1024) void coarse_scan_kernel(uint32_t* __restrict__ table, int C1, uint32_t NB,
                                                           uint32_t* __restrict__ tot) {
    __shared__ uint32_t s_w[64][16];
    const int l = threadIdx.x & 15, w = threadIdx.x >> 4;
    const uint32_t b = blockIdx.x * 16u + (uint32_t)l;
    const bool ok = b < NB;
    const int per = (C1 + 63) / 64;
    const int c0 = w * per, c1 = min(C1, c0 + per);
    uint32_t s = 0u;
#pragma unroll 8
    for (int c = c0; c < c1; c++) s += ok ? table[(size_t)c * NB + b] : 0u;
    s_w[w][l] = s;
    __syncthreads();
    uint32_t run = 0u, all = 0u;
#pragma unroll 8
    for (int k = 0; k < 64; k++) {
        const uint32_t x = s_w[k][l];
        run += k < w ? x : 0u;
        all += x;
    }
    if (w == 0 && ok) tot[b] = all;
    if (ok) {
#pragma unroll 8
        for (int c = c0; c < c1; c++) {
            const uint32_t x = table[(size_t)c * NB + b];
            table[(size_t)c * NB + b] = run;
            run += x;
        }
    }
}

// One block: the bins' first records (NB + 1 entries), the record count, and
// the flag (may be null) when the records outgrow their buffer.
__global__ __launch_bounds__(1024) void coarse_starts_kernel(const uint32_t* __restrict__ tot, uint32_t NB,
                                                             uint32_t cap, uint32_t* __restrict__ start,
                                                             unsigned long long* __restrict__ total,
                                                             uint32_t* __restrict__ overflow) {
    __shared__ unsigned long long s_w[16];
    unsigned long long carry = 0ull;
    for (uint32_t b0 = 0; b0 < NB; b0 += 1024u) {
        const uint32_t b = b0 + threadIdx.x;
        const unsigned long long x = b < NB ? tot[b] : 0u;
        unsigned long long sum;
        const unsigned long long ex = carry + gsw::block_exclusive_scan<unsigned long long>(x, s_w, &sum);
        if (b < NB) start[b] = (uint32_t)min(ex, (unsigned long long)0xFFFFFFFFu);
        carry += sum;
    }
    if (threadIdx.x == 0) {
        start[NB] = (uint32_t)min(carry, (unsigned long long)0xFFFFFFFFu);
        *total = carry;
        if (overflow && carry > cap) *overflow = 1u;
    }
}

// One block per (view, chunk): writes the chunk's records.  256 Gaussians per
// round, 64 per wave; MAXB: the largest bin count of a view.  A Gaussian of
// more than BIG bins is handled by its whole wave, one bin per lane, so a few
// that cover the view do not serialise on one lane each.
constexpr int BIG = 16;

template <int BT, int MAXB>
__global__ __launch_bounds__(256) void coarse_place_kernel(BinArgs a) {
    __shared__ uint64_t s_m[4][MAXB];     // per wave and bin: the lanes of this round whose Gaussian meets it
    __shared__ uint32_t s_base[4][MAXB];  // per wave and bin: the wave's first record of this round
    __shared__ uint32_t s_cur[MAXB];      // per bin: the next record
    using Rec = typename Bins<BT>::Rec;
    Rec* const coarse = reinterpret_cast<Rec*>(a.coarse);
    const int q = blockIdx.x;
    const int v = q / a.C1, c = q - v * a.C1;
    const int4 vi = view_info(a, v);
    const int nbx = (vi.x + BT - 1) / BT, nby = (vi.y + BT - 1) / BT, nb = nbx * nby;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const uint32_t* col = a.table1 + (size_t)c * a.NB + (uint32_t)vi.z;
    for (int b = tid; b < nb; b += 256) {
        s_cur[b] = a.start[(uint32_t)vi.z + b] + col[b];
#pragma unroll
        for (int k = 0; k < 4; k++) s_m[k][b] = 0ull;
    }
    uint32_t r0, r1;
    chunk_ranks(a, c, r0, r1);
    const uint2* rects = a.rects + (size_t)v * a.N;
    uint2 nxt = r0 + (uint32_t)tid < r1 ? rects[r0 + tid] : make_uint2(0u, 0u);
    __syncthreads();
    for (uint32_t base = r0; base < r1; base += 256u) {
        const uint2 rec = nxt;
        nxt = base + 256u + (uint32_t)tid < r1 ? rects[base + 256u + tid] : make_uint2(0u, 0u);
        const Rect t(rec.x);
        const Rect b = bins_of<BT>(t);
        const int bw = b.x1 - b.x0, cnt = bw * (b.y1 - b.y0);
        const uint64_t big = __ballot(cnt > BIG);
        const uint64_t bit = 1ull << lane;
        const int b0 = b.y0 * nbx + b.x0;
        if (cnt <= BIG) {
            int bin = b0, x = 0;
            for (int k = 0; k < cnt; k++) {
                atomicOr((unsigned long long*)&s_m[w][bin], (unsigned long long)bit);
                const bool wrap = ++x == bw;
                bin += wrap ? nbx - bw + 1 : 1;
                x = wrap ? 0 : x;
            }
        }
        for (uint64_t m = big; m != 0ull; m &= m - 1ull) {
            const int j = __builtin_ctzll(m);
            const Rect bj = bins_of<BT>(Rect((uint32_t)__builtin_amdgcn_readlane((int)rec.x, j)));
            const int wj = bj.x1 - bj.x0, nj = wj * (bj.y1 - bj.y0);
            for (int k = lane; k < nj; k += 64)
                atomicOr((unsigned long long*)&s_m[w][(bj.y0 + k / wj) * nbx + bj.x0 + k % wj], 1ull << j);
        }
        __syncthreads();
        for (int k = tid; k < nb; k += 256) {
            uint32_t at = s_cur[k];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                s_base[j][k] = at;
                at += (uint32_t)__popcll(s_m[j][k]);
            }
            s_cur[k] = at;
        }
        __syncthreads();
        // a record's slot: its wave's first one, then the lanes below whose Gaussian meets the bin
        if (cnt <= BIG) {
            int bin = b0, x = 0, y = 0;
#pragma unroll 2
            for (int k = 0; k < cnt; k++) {
                const uint32_t slot = s_base[w][bin] + (uint32_t)__popcll(s_m[w][bin] & (bit - 1ull));
                if (slot < a.coarse_cap) coarse[slot] = make_record<BT>(rec.y, t, b.x0 + x, b.y0 + y);
                const bool wrap = ++x == bw;
                bin += wrap ? nbx - bw + 1 : 1;
                x = wrap ? 0 : x;
                y += wrap ? 1 : 0;
            }
        }
        for (uint64_t m = big; m != 0ull; m &= m - 1ull) {
            const int j = __builtin_ctzll(m);
            const Rect tj((uint32_t)__builtin_amdgcn_readlane((int)rec.x, j));
            const uint32_t id = (uint32_t)__builtin_amdgcn_readlane((int)rec.y, j);
            const Rect bj = bins_of<BT>(tj);
            const int wj = bj.x1 - bj.x0, nj = wj * (bj.y1 - bj.y0);
            for (int k = lane; k < nj; k += 64) {
                const int x = bj.x0 + k % wj, y = bj.y0 + k / wj, bin = y * nbx + x;
                const uint32_t slot = s_base[w][bin] + (uint32_t)__popcll(s_m[w][bin] & ((1ull << j) - 1ull));
                if (slot < a.coarse_cap) coarse[slot] = make_record<BT>(id, tj, x, y);
            }
        }
        __syncthreads();
        if (base + 256u < r1) {
            for (int k = tid; k < nb; k += 256) {
#pragma unroll
                for (int j = 0; j < 4; j++) s_m[j][k] = 0ull;
            }
            __syncthreads();
        }
    }
}

// The bin, group and records of a level-2 block (uniform).
struct BinGroup {
    int v, g, bx, by;
    int4 vi;
    uint32_t s, e;  // records
};

template <int BT>
__device__ __forceinline__ BinGroup bin_group(const BinArgs& a) {
    const int q = gsd::xcd_remap(blockIdx.x, gridDim.x);
    BinGroup o;
    const uint32_t gb = (uint32_t)(q / a.C2);
    o.g = q - (int)gb * a.C2;
    o.v = 0;
    if (a.views)
        while (o.v + 1 < a.V && (uint32_t)a.views[o.v + 1].z <= gb) o.v++;
    o.vi = view_info(a, o.v);
    const int nbx = (o.vi.x + BT - 1) / BT;
    const int local = (int)(gb - (uint32_t)o.vi.z);
    o.bx = local % nbx;
    o.by = local / nbx;
    const int c0 = o.g * a.GC, c1 = c0 + a.GC;
    const uint32_t first = a.start[gb];
    o.s = first + a.table1[(size_t)c0 * a.NB + gb];
    o.e = c1 < a.C1 ? first + a.table1[(size_t)c1 * a.NB + gb] : a.start[gb + 1];
    o.s = min(o.s, a.coarse_cap);
    o.e = min(o.e, a.coarse_cap);
    return o;
}

// Global index of tile (x, y) of a block's bin, or -1 outside the view.
template <int BT>
__device__ __forceinline__ int bin_tile(const BinGroup& b, int x, int y) {
    const int tx = b.bx * BT + x, ty = b.by * BT + y;
    return tx < b.vi.x && ty < b.vi.y ? b.vi.w + ty * b.vi.x + tx : -1;
}

// One block per (bin, group): each wave counts every fourth run of 64 records
// for all tiles of the bin.
template <int BT>
__global__ __launch_bounds__(256) void tile_count_kernel(BinArgs a) {
    using Rec = typename Bins<BT>::Rec;
    __shared__ uint32_t s_n[4][BT * BT];
    const BinGroup b = bin_group<BT>(a);
    const Rec* coarse = reinterpret_cast<const Rec*>(a.coarse);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (blockIdx.x == 0 && threadIdx.x == 0) a.table2[a.table2_len - 1] = 0u;
    uint32_t n[BT * BT];
#pragma unroll
    for (int k = 0; k < BT * BT; k++) n[k] = 0u;
    for (uint32_t r = b.s + 64u * w; r < b.e; r += 256u) {
        Rec x{};
        if (r + (uint32_t)lane < b.e) x = coarse[r + lane];
#pragma unroll
        for (int k = 0; k < BT * BT; k++) n[k] += (uint32_t)__popcll(__ballot((mask_row(x, k / BT) >> (k % BT)) & 1u));
    }
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < BT * BT; k++) s_n[w][k] = n[k];
    }
    __syncthreads();
    if (threadIdx.x < BT * BT) {
        const int k = threadIdx.x;
        const int t = bin_tile<BT>(b, k % BT, k / BT);
        if (t >= 0) a.table2[(size_t)t * a.C2 + b.g] = s_n[0][k] + s_n[1][k] + s_n[2][k] + s_n[3][k];
    }
}

// One block per (bin, group), one row of BT tiles per wave.  PRE runs of 64
// records are loaded ahead of the one being compacted.  Slots past the
// capacity are dropped and raise the overflow flag.
template <int BT>
__global__ __launch_bounds__(64 * BT) void tile_place_kernel(BinArgs a) {
    using Rec = typename Bins<BT>::Rec;
    const BinGroup b = bin_group<BT>(a);
    if (b.s >= b.e) return;
    const Rec* coarse = reinterpret_cast<const Rec*>(a.coarse);
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t cur[BT];
#pragma unroll
    for (int k = 0; k < BT; k++) {
        const int t = bin_tile<BT>(b, k, w);
        cur[k] = t >= 0 ? a.scanned[(size_t)t * a.C2 + b.g] : 0u;
    }
    constexpr int PRE = 4;
    Rec nxt[PRE];
#pragma unroll
    for (int p = 0; p < PRE; p++) {
        const uint32_t r = b.s + 64u * p + (uint32_t)lane;
        nxt[p] = Rec{};
        if (r < b.e) nxt[p] = coarse[r];
    }
    for (uint32_t base = b.s; base < b.e; base += 64u * PRE) {
        Rec rec[PRE];
#pragma unroll
        for (int p = 0; p < PRE; p++) {
            rec[p] = nxt[p];
            const uint32_t r = base + 64u * (PRE + p) + (uint32_t)lane;
            nxt[p] = Rec{};
            if (r < b.e) nxt[p] = coarse[r];
        }
#pragma unroll
        for (int p = 0; p < PRE; p++) {
            const uint32_t m = mask_row(rec[p], w);
#pragma unroll
            for (int k = 0; k < BT; k++) {
                const bool in = (m >> k) & 1u;
                const uint64_t bal = __ballot(in);
                const uint32_t at = cur[k] + __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32),
                                                                       __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
                if (in && at < a.capacity) a.out[at] = rec[p].x;
                cur[k] += (uint32_t)__popcll(bal);
            }
        }
    }
    uint32_t most = 0u;
#pragma unroll
    for (int k = 0; k < BT; k++) most = max(most, cur[k]);
    if (lane == 0 && most > a.capacity) *a.overflow = 1u;
}

// One thread per global tile.
// Ranges are clamped to the pair capacity, so that after an overflow (pairs
// dropped, flag raised) the rasterizers still read inside the buffer.
__global__ __launch_bounds__(256) void bin_ranges_kernel(const uint32_t* __restrict__ scanned, int C2,
                                                         uint32_t total_tiles, uint32_t capacity,
                                                         uint32_t* __restrict__ ranges) {
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= total_tiles) return;
    uint32_t s = min(scanned[(size_t)g * C2], capacity);
    uint32_t e = min(scanned[(size_t)(g + 1) * C2], capacity);
    if (s == e) s = e = 0u;
    ranges[2 * (size_t)g] = s;
    ranges[2 * (size_t)g + 1] = e;
}

}  // namespace gsb

using namespace gsb;

// Views of up to 1024 bins of 4 x 4 tiles (2048 x 2048 pixels, say) use those,
// larger views bins of 8 x 8: the bin masks of a block then always fit a few
// workgroups per CU, and the larger rectangles of a larger view meet as many bins
// as before (at 4K, 1M Gaussians: 6.9 records per Gaussian instead of 18).
int bin_side(int max_gx, int max_gy) {
    const int b4 = ((max_gx + 3) / 4) * ((max_gy + 3) / 4);
    return b4 <= GS_BIN_MAX_BINS ? 4 : 8;
}

int bin_count_of_view(int side, int gx, int gy) { return ((gx + side - 1) / side) * ((gy + side - 1) / side); }

// Chunks: 256 .. 4096 Gaussians, the largest that still gives 512 chunks (two
// blocks per CU) so that small scenes spread over the chip and large ones keep
// the (chunk, bin) table small; 2048 at most while that table has 32 MB or less,
// and the first 128 chunks, of the nearest Gaussians, 256: from inside a scene
// those meet tens of bins each (43 on average in the first thousand, 4 over all)
// and one block of 4096 of them outlasted all others (4M Gaussians, 1.7M in view,
// 1080p: coarse_place 353 us; 154 with the near chunks cut, 91 with both).
// Groups: enough level-2 blocks to fill the
// chip several times (8192) and about one per 512 Gaussians beyond, so that
// the bins where a scene is densest do not leave one long block at the end; in
// views of few bins up to one per 128 Gaussians, since with 64 groups a bin the
// few blocks of a view of one bin walked 60 thousand records each (4M Gaussians,
// 64 x 64 pixels: tile_count 127 and tile_place 298 us, now 12 and 32;
// 1M at 160 x 120: 22 and 44, now 11 and 20).
void bin_layout(BinArgs& a) {
    const size_t vn = (size_t)a.V * (size_t)a.N;
    int rounds = 1;
    while (rounds < 16 && vn / (256u * 2u * (size_t)rounds) >= 512u) {
        if (rounds >= 8 && ((size_t)a.N / (256u * (size_t)rounds) + 1u) * a.NB * 4u <= (size_t)32 << 20) break;
        rounds *= 2;
    }
    a.CH = 256 * rounds;
    a.S = rounds > 1 ? std::min(128, a.N / 2048) : 0;
    a.C1 = a.S + (a.N - 256 * a.S + a.CH - 1) / a.CH;
    const size_t blocks = std::min(std::max<size_t>(8192u, vn / 512u), std::max<size_t>(vn / 128u, (size_t)64u * a.NB));
    const int want = (int)std::max<size_t>(blocks / a.NB, 1u);
    a.GC = (a.C1 + want - 1) / want;
    a.C2 = (a.C1 + a.GC - 1) / a.GC;
    a.table1_len = (size_t)a.C1 * a.NB;
    a.table2_len = (size_t)a.total_tiles * a.C2 + 1;
}

size_t bin_record_bytes(const BinArgs& a) { return a.side == 4 ? 8 : 16; }

size_t bin_workspace_bytes(const BinArgs& a) {
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    return al((size_t)a.V * a.N * 8) + al(a.table1_len * 4) + al((size_t)a.NB * 4) + al(((size_t)a.NB + 1) * 4) +
           2 * al(a.table2_len * 4) + al(((size_t)scan_partials_needed((uint32_t)a.table2_len) + 1) * 8);
}

void bin_carve(BinArgs& a, void* workspace) {
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    char* w = static_cast<char*>(workspace);
    a.rects = reinterpret_cast<uint2*>(w); w += al((size_t)a.V * a.N * 8);
    a.table1 = reinterpret_cast<uint32_t*>(w); w += al(a.table1_len * 4);
    a.tot = reinterpret_cast<uint32_t*>(w); w += al((size_t)a.NB * 4);
    a.start = reinterpret_cast<uint32_t*>(w); w += al(((size_t)a.NB + 1) * 4);
    a.table2 = reinterpret_cast<uint32_t*>(w); w += al(a.table2_len * 4);
    a.scanned = reinterpret_cast<uint32_t*>(w); w += al(a.table2_len * 4);
    a.partial = reinterpret_cast<unsigned long long*>(w);
}

template <int BT>
static hipError_t bin_lists(const BinArgs& a, hipStream_t s, unsigned long long* records, bool counted) {
    const unsigned chunks = (unsigned)(a.V * a.C1);
    if (!counted) {
        coarse_count_kernel<BT><<<chunks, 256, 0, s>>>(a);
        coarse_scan_kernel<<<(a.NB + 15) / 16, 1024, 0, s>>>(a.table1, a.C1, a.NB, a.tot);
        coarse_starts_kernel<<<1, 1024, 0, s>>>(a.tot, a.NB, a.coarse_cap, a.start, records,
                                                a.record_overflow);
    }
    if (a.max_bins <= 256)
        coarse_place_kernel<BT, 256><<<chunks, 256, 0, s>>>(a);
    else if (a.max_bins <= 512)
        coarse_place_kernel<BT, 512><<<chunks, 256, 0, s>>>(a);
    else if (a.max_bins <= GS_BIN_MAX_BINS)
        coarse_place_kernel<BT, GS_BIN_MAX_BINS><<<chunks, 256, 0, s>>>(a);
    else
        return hipErrorInvalidValue;
    tile_count_kernel<BT><<<a.NB * (unsigned)a.C2, 256, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_bin_lists(const BinArgs& a, hipStream_t s, unsigned long long* records, uint32_t* total32,
                            unsigned long long* total64, bool counted) {
    const hipError_t e = a.side == 4 ? bin_lists<4>(a, s, records, counted) : bin_lists<8>(a, s, records, counted);
    if (e != hipSuccess) return e;
    return launch_scan_u32_exclusive(a.table2, (uint32_t)a.table2_len, a.scanned, a.partial, s, total32, total64);
}

hipError_t launch_bin_place(const BinArgs& a, hipStream_t s) {
    if (a.side == 4)
        tile_place_kernel<4><<<a.NB * (unsigned)a.C2, 256, 0, s>>>(a);
    else
        tile_place_kernel<8><<<a.NB * (unsigned)a.C2, 512, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_bin_ranges(const BinArgs& a, uint32_t* ranges, hipStream_t s) {
    if (a.total_tiles == 0) return hipSuccess;
    bin_ranges_kernel<<<(a.total_tiles + 255) / 256, 256, 0, s>>>(a.scanned, a.C2, (uint32_t)a.total_tiles, a.capacity,
                                                                 ranges);
    return hipGetLastError();
}
