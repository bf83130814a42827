// k_raster.hip -- tile rasterization, forward and backward.
//
// One 256-thread workgroup (four wave64s) per 16x16 tile, one thread per
// pixel.  The tile's depth-sorted Gaussians are staged in LDS in batches of
// BATCH entries (position, conic+opacity, colour); every lane then reads the
// same LDS slot (a broadcast, no bank conflicts).  The forward stops a pixel
// when its transmittance would fall below 1e-4 and the workgroup when all its
// pixels stopped; it records T_final, the contributor count and the list index
// (+1) of the last contributor.
//
// The backward walks the same list back to front from the largest last
// contributor in the tile.  Each pixel recovers T_i = T/(1-alpha) exactly as
// the reference CPU backward (cpu/rasterizer_backward_cpu.cpp:69-134); the
// nine per-Gaussian gradient terms are summed across the wave with packed
// permlane-swap/DPP steps (no LDS traffic), across the four waves with LDS
// atomics, and land in HBM with one float atomic per (tile, Gaussian,
// component), issued by consecutive lanes per Gaussian.  What bounds the
// backward: VALU issue (71 instructions per visited entry and wave, 27 of them
// the sums), and below about two workgroups per CU the latency of that chain.
//
// Multi-view: the same tile bodies run over a global (view, tile) list, either
// one workgroup per global tile or a persistent grid that takes tiles from
// per-XCD atomic queues.  Workgroup-to-tile maps are XCD-aware throughout.
#include "gs_device.h"

namespace gsr {

using gsd::smin;

// Wave w of a tile (threads 64w .. 64w+63) covers one block of its pixels:
// in the forward the 8 x 8 quadrant (w & 1, w >> 1), in the backward the
// 16 x 4 strip of rows 4w .. 4w+3 (measured: each layout is the faster one
// for its kernel).  Per LDS batch, mask[w][c] bit b is set when entry 64c + b
// can pass the alpha cut somewhere in block w (see strip_hits); each wave
// visits only its set bits.
// One staged entry: 48 bytes, read with one base address and immediate
// offsets (mean, conic + opacity, colour).
struct Staged {
    float2 xy;
    float2 pad;
    float4 co;
    float4 rgb;
};

template <int BATCH>
struct FwdSmem {
    Staged e[BATCH];
    uint64_t mask[4][BATCH / 64];
};

// Block-hit bits of one staged entry: bit w set when the Gaussian can pass the
// 1/255 alpha cut at some pixel centre of block w of the tile whose top-left
// pixel is (x0, y0): QUAD, the 8 x 8 quadrant (w & 1, w >> 1); else the strip
// of rows y0 + 4w .. y0 + 4w + 3, columns x0 .. x0 + 15.
// alpha = o * exp(-Q/2) with Q = a u^2 + 2 b u v + c v^2 ((a, b, c) the conic,
// (u, v) the pixel minus the mean), so passing needs Q <= r2 = 2 ln(255 o).
// The least Q over a rectangle is 0 when the mean lies inside it, else the
// least of its minima along the four edges; along an edge Q is a quadratic
// in one variable whose minimum lies at its vertex clamped to the edge.
// Margins, so that a strip without the bit has no pixel that passes:
//  - the rasterizer's float Q has a relative rounding error below about
//    8 eps tr^2/det (its terms reach tr^2/det times Q), and so has the Q
//    computed here; the test is exact only where tr^2/det <= 1000 (together
//    at most 1e-3) and r2 is widened by 0.1 %, plus 1e-3 for the approximate
//    log used here;
//  - each rectangle is grown by half a pixel on every side.
// o < 1/255 never passes (no bits); a degenerate or too anisotropic conic
// gets every bit.  An entry with a non-finite mean or conic never passes in
// the rasterizer (its power is NaN) and gets no bits, so every visited entry
// is finite.
__device__ __forceinline__ float quad_form(float a, float b, float c, float u, float v) {
    return (a * u * u + c * v * v) + 2.0f * b * u * v;
}

template <bool QUAD>
__device__ __forceinline__ uint32_t strip_hits(float2 m, float4 co, float x0, float y0) {
    const float o = co.w;
    if (!(o >= 1.0f / 255.0f)) return 0u;
    const float a = co.x, b = co.y, c = co.z;
    if (!(__builtin_isfinite(m.x) && __builtin_isfinite(m.y) && __builtin_isfinite(a) && __builtin_isfinite(b) &&
          __builtin_isfinite(c) && __builtin_isfinite(o)))
        return 0u;
    const float det = a * c - b * b;
    const float tr = a + c;
    if (!(det > 0.0f) || !(tr * tr <= 1000.0f * det)) return 0xFu;
    // 2 ln(x) = 2 ln(2) log2(x)
    const float r2 = 1.38629436f * __builtin_amdgcn_logf(255.0f * o) * 1.001f + 1e-3f;
    constexpr float G = 0.5f;
    constexpr float BW = QUAD ? 7.0f : 15.0f, BH = QUAD ? 7.0f : 3.0f;  // block extent - 1
    // edge vertices: u* = -(b / a) v on the rows, v* = -(b / c) u on the columns
    const float ka = -b * __builtin_amdgcn_rcpf(a), kc = -b * __builtin_amdgcn_rcpf(c);
    uint32_t h = 0u;
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const float bx = x0 + (QUAD ? (float)(8 * (w & 1)) : 0.0f);
        const float by = y0 + (QUAD ? (float)(8 * (w >> 1)) : (float)(4 * w));
        const float u0 = bx - G - m.x, u1 = bx + (BW + G) - m.x;
        const float vl = kc * u0, vr = kc * u1;
        const float v0 = by - G - m.y, v1 = by + (BH + G) - m.y;
        float q = (u0 <= 0.0f && u1 >= 0.0f && v0 <= 0.0f && v1 >= 0.0f) ? 0.0f : 3.0e38f;
        q = fminf(q, quad_form(a, b, c, fminf(fmaxf(ka * v0, u0), u1), v0));
        q = fminf(q, quad_form(a, b, c, fminf(fmaxf(ka * v1, u0), u1), v1));
        q = fminf(q, quad_form(a, b, c, u0, fminf(fmaxf(vl, v0), v1)));
        q = fminf(q, quad_form(a, b, c, u1, fminf(fmaxf(vr, v0), v1)));
        h |= (q <= r2) ? (1u << w) : 0u;
    }
    return h;
}

// Staged conics are kept as (-a/2, -b, -c/2, o), so that the power
// -0.5 (a dx^2 + c dy^2) - b dx dy of rasterizer_cpu.cpp:159-161 becomes
// (a' dx^2 + c' dy^2) + b' dx dy.  Scaling by -1/2 and -1 is exact, so this is
// the same float value (away from subnormals) in one multiply fewer.
__device__ __forceinline__ float4 prescale(float4 co) { return make_float4(-0.5f * co.x, -co.y, -0.5f * co.z, co.w); }

__device__ __forceinline__ float power_of(const float4& co, float dx, float dy) {
    return (co.x * dx * dx + co.z * dy * dy) + co.y * dx * dy;
}

// Ballots the hit bits of 64 staged entries (one per lane of the calling wave,
// entries 64c .. 64c+63) into the four strips' masks.
template <int BATCH>
__device__ __forceinline__ void store_masks(uint64_t (&mask)[4][BATCH / 64], int c, uint32_t h, int lane) {
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const uint64_t b = __ballot((h >> w) & 1u);
        if (lane == 0) mask[w][c] = b;
    }
}

__device__ __forceinline__ uint64_t wave_uniform(uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// gradient sums per Gaussian: dop * (dx, dy, dx^2, dx dy, dy^2), rgb 3, opacity 1
constexpr int NG = 9;

template <int BATCH>
struct BwdSmem {
    Staged e[BATCH];
    uint64_t mask[4][BATCH / 64];
    uint32_t id[BATCH];
    float g[BATCH][NG];
    uint32_t maxlast;
};

struct PixOut {
    float* img;
    float* T_final;
    int* n_contrib;
    uint32_t* last_contrib;
};

// An entry at a pixel: the exponent and min(0.99, opacity e^power), with the
// 1/255 decision exact (gsd::alpha_fast / alpha_fix); ep = e^power.
struct Eval {
    float dx, dy, power, ep, alpha;
};

__device__ __forceinline__ Eval evaluate(const Staged& e, float fpx, float fpy) {
    Eval v;
    const float2 mm = e.xy;
    const float4 co = e.co;
    v.dx = mm.x - fpx;
    v.dy = mm.y - fpy;
    v.power = power_of(co, v.dx, v.dy);
    v.alpha = gsd::raster_alpha_wave(co.w, v.power, &v.ep);
    return v;
}

// Two entries whose chains (LDS reads, power, exponential) overlap.
__device__ __forceinline__ void evaluate2(const Staged& e0, const Staged& e1, float fpx, float fpy, Eval& a, Eval& b) {
    const float2 m0 = e0.xy, m1 = e1.xy;
    const float4 c0 = e0.co, c1 = e1.co;
    a.dx = m0.x - fpx;
    a.dy = m0.y - fpy;
    b.dx = m1.x - fpx;
    b.dy = m1.y - fpy;
    a.power = power_of(c0, a.dx, a.dy);
    b.power = power_of(c1, b.dx, b.dy);
    bool n0, n1;
    a.alpha = gsd::alpha_fast(c0.w, a.power, &a.ep, &n0);
    b.alpha = gsd::alpha_fast(c1.w, b.power, &b.ep, &n1);
    if (__ballot(n0 || n1) != 0ull) {
        gsd::alpha_fix(c0.w, a.power, n0, &a.alpha, &a.ep);
        gsd::alpha_fix(c1.w, b.power, n1, &b.alpha, &b.ep);
    }
}

template <int BATCH, bool PAIR>
__device__ __forceinline__ void fwd_tile(const RasterArgs& a, int tile, FwdSmem<BATCH>& sm, const PixOut& o) {
    const int tx = tile % a.gx, ty = tile / a.gx;
    const int t = threadIdx.x;
    // 8 x 8 quadrant (w & 1, w >> 1) per wave
    const int px = tx * gsd::TILE + 8 * ((t >> 6) & 1) + (t & 7), py = ty * gsd::TILE + 8 * (t >> 7) + ((t >> 3) & 7);
    const bool inside = px < a.W && py < a.H;
    const int pix = py * a.W + px;
    const uint32_t start = a.ranges[2 * tile], end = a.ranges[2 * tile + 1];
    const float fpx = (float)px, fpy = (float)py;
    const float tx0 = (float)(tx * gsd::TILE), ty0 = (float)(ty * gsd::TILE);
    const int lane = t & 63, w = t >> 6;
    float T = 1.0f, C0 = 0.0f, C1 = 0.0f, C2 = 0.0f;
    int cnt = 0;
    uint32_t last = 0;
    bool done = !inside;
    // One visited entry, predicated: every lane runs it and selects, so the
    // only branches are uniform (the CU's scalar unit, shared by its waves, is
    // not spent on exec-mask bookkeeping of per-pixel branches).
    auto blend = [&](const Eval& v, const float4& cl, uint32_t index, bool valid) {
        // rasterizer_cpu.cpp: skip if power > 0 or alpha < 1/255; stop
        // (without this entry) once T would fall below 1e-4
        const bool use = valid && !done && v.power <= 0.0f && v.alpha >= 1.0f / 255.0f;
        const float test_T = T * (1.0f - v.alpha);
        const bool take = use && test_T >= 0.0001f;  // T and alpha are finite here
        // used but no room left (one compare: the negated compare
        // would be a second, since the compiler keeps NaN semantics)
        done = done || (use != take);
        // colour += c alpha T, with the weight alpha T selected in or out;
        // the colour feeds no decision (T and alpha do), so its sums are
        // contracted to FMAs
        const float wt = take ? v.alpha * T : 0.0f;
        {
#pragma clang fp contract(fast)
            C0 += cl.x * wt;
            C1 += cl.y * wt;
            C2 += cl.z * wt;
        }
        T = take ? test_T : T;
        cnt += take ? 1 : 0;
        last = take ? index : last;
    };
    for (uint32_t base = start; base < end; base += BATCH) {
        if (__syncthreads_count(!done) == 0) break;
        for (int k = t; k < BATCH; k += 256) {
            uint32_t j = base + k;
            uint32_t h = 0u;
            if (j < end) {
                uint32_t id = a.values[(size_t)j * a.vstride];
                const float2 mm = a.means2D[id];
                const float4 cc = make_float4(a.conics[id * 3], a.conics[id * 3 + 1], a.conics[id * 3 + 2], a.opac[id]);
                sm.e[k].xy = mm;
                sm.e[k].co = prescale(cc);
                sm.e[k].rgb = make_float4(a.rgb[id * 3], a.rgb[id * 3 + 1], a.rgb[id * 3 + 2], 0.0f);
                h = strip_hits<true>(mm, cc, tx0, ty0);
            }
            store_masks<BATCH>(sm.mask, k >> 6, h, lane);
        }
        __syncthreads();
        const int nc = (int)(((end - base) < (uint32_t)BATCH ? (end - base) : (uint32_t)BATCH) + 63u) >> 6;
        for (int c = 0; c < nc; c++) {
            if (__ballot(!done) == 0ull) break;
            uint64_t m = wave_uniform(sm.mask[w][c]);
            while (m != 0ull) {
                if constexpr (!PAIR) {
                    const int k = (c << 6) + __builtin_ctzll(m);
                    m &= m - 1ull;
                    const Eval v = evaluate(sm.e[k], fpx, fpy);
                    blend(v, sm.e[k].rgb, base + (uint32_t)k + 1u, true);
                } else {
                    const int k0 = (c << 6) + __builtin_ctzll(m);
                    m &= m - 1ull;
                    const bool two = m != 0ull;
                    const int k1 = two ? (c << 6) + __builtin_ctzll(m) : k0;
                    m &= m - 1ull;  // 0 stays 0
                    const float4 cl0 = sm.e[k0].rgb, cl1 = sm.e[k1].rgb;
                    Eval v0, v1;
                    evaluate2(sm.e[k0], sm.e[k1], fpx, fpy, v0, v1);
                    blend(v0, cl0, base + (uint32_t)k0 + 1u, true);
                    blend(v1, cl1, base + (uint32_t)k1 + 1u, two);
                }
            }
        }
    }
    if (inside) {
        o.img[pix * 3 + 0] = C0 + T * a.bg0;
        o.img[pix * 3 + 1] = C1 + T * a.bg1;
        o.img[pix * 3 + 2] = C2 + T * a.bg2;
        if (o.T_final) o.T_final[pix] = T;
        if (o.n_contrib) o.n_contrib[pix] = cnt;
        if (o.last_contrib) o.last_contrib[pix] = last;
    }
}

// ---- packed wave reduction of the gradient terms ---------------------------
// Packed, two values share each exchange: v_permlane32_swap leaves value a
// summed over lane pairs {l, l+32} in lanes 0-31 and value b in lanes 32-63;
// v_permlane16_swap does the same between 16-lane rows.  swap16_sum of
// swap32_sum(a, b) and swap32_sum(c, d) holds a, c, b, d in rows 0 .. 3.
__device__ __forceinline__ float swap32_sum(float a, float b) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__device__ __forceinline__ float swap16_sum(float a, float b) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

// The nine sums of one visited entry over a wave's strip of 16 columns x 4
// rows (lane l at column l % 16, row l / 16).  dx depends on the column alone
// and dy on the row alone, so the six sums of dop times 1, dx, dy, dx^2, dx dy,
// dy^2 start as three values (dop, dop dy, dop dy^2) summed over the rows, and
// are multiplied by dx afterwards:
//   swap steps (rows): k0 = {dop, dop dy^2, dop dy, c0} and k1 = {c1, c1, c2,
//     c2} in rows 0 .. 3, each summed over the four rows, per column;
//   m1 = k0 dx and m2 = m1 dx carry the dx and dx^2 sums; row 1 and 3 of m1
//     hold nothing wanted, so k1 goes there;
//   DPP steps (columns): the values share a register as soon as their sums
//     repeat within a row: m1 takes the upper half of each row after the first
//     step, m2 the odd quarters after the second.
// 22 VALU instructions after the four products; nine separate terms took 28
// after eight products, and two selects to deliver (200k Gaussians at 720p:
// 343 -> 332 us, 10k at 256 x 256: 82 -> 77 us).
struct ReduceRole {
    bool odd_row, half, quarter;  // lane / 16 odd; lane & 8; lane & 4
    int term;                     // the sum this lane delivers (-1: none)
};

__device__ __forceinline__ ReduceRole reduce_role(int lane) {
    ReduceRole q;
    const int row = lane >> 4, p = lane & 15;
    q.odd_row = (row & 1) != 0;
    q.half = (lane & 8) != 0;
    q.quarter = (lane & 4) != 0;
    q.term = -1;
    if (p == 0) q.term = row == 0 ? 8 : (row == 1 ? 4 : (row == 2 ? 1 : 5));  // k0: 1, dy^2, dy, c0
    if (p == 8) q.term = row == 0 ? 0 : (row == 1 ? 6 : (row == 2 ? 3 : 7));  // m1: dx, c1, dx dy, c2
    if (p == 4 && row == 0) q.term = 2;                                       // m2: dx^2
    return q;
}

__device__ __forceinline__ float wave_reduce9(float dop, float dx, float dy, float c0, float c1, float c2,
                                              const ReduceRole& q) {
    const float py = dop * dy;
    const float h0 = swap32_sum(dop, py);
    const float h1 = swap32_sum(py * dy, c0);
    const float h2 = swap32_sum(c1, c2);
    float k0 = swap16_sum(h0, h1);
    const float k1 = swap16_sum(h2, h2);
    float m1 = k0 * dx;
    float m2 = m1 * dx;
    m1 = q.odd_row ? k1 : m1;
    constexpr int ROR8 = 0x128, HALF_MIRROR = 0x141, QUAD_XOR2 = 0x4E, QUAD_XOR1 = 0xB1;
    k0 += dpp_f<ROR8>(k0);
    m1 += dpp_f<ROR8>(m1);
    m2 += dpp_f<ROR8>(m2);
    k0 = q.half ? m1 : k0;
    k0 += dpp_f<HALF_MIRROR>(k0);
    m2 += dpp_f<HALF_MIRROR>(m2);
    k0 = q.quarter ? m2 : k0;
    k0 += dpp_f<QUAD_XOR2>(k0);
    k0 += dpp_f<QUAD_XOR1>(k0);
    return k0;
}

struct PixIn {
    const float* T_final;
    const uint32_t* last_contrib;
    const float* d_image;
};

template <int BATCH>
__device__ __forceinline__ void bwd_tile(const RasterArgs& a, int tile, BwdSmem<BATCH>& sm, const PixIn& in,
                                         const GradArgs& g) {
    const int tx = tile % a.gx, ty = tile / a.gx;
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int px = tx * gsd::TILE + (t & 15), py = ty * gsd::TILE + (t >> 4);
    const bool inside = px < a.W && py < a.H;
    const uint32_t start = a.ranges[2 * tile];
    const int pix = py * a.W + px;
    float T = 0.0f, dC0 = 0.0f, dC1 = 0.0f, dC2 = 0.0f;
    uint32_t last = 0;
    if (inside) {
        T = in.T_final[pix];
        last = in.last_contrib[pix];
        dC0 = in.d_image[pix * 3];
        dC1 = in.d_image[pix * 3 + 1];
        dC2 = in.d_image[pix * 3 + 2];
    }
    float acc0 = a.bg0, acc1 = a.bg1, acc2 = a.bg2;
    const float fpx = (float)px, fpy = (float)py;
    const float tx0 = (float)(tx * gsd::TILE), ty0 = (float)(ty * gsd::TILE);
    const int w = t >> 6;
    const ReduceRole role = reduce_role(lane);
    if (t == 0) sm.maxlast = 0;
    __syncthreads();
    if (last > 0) atomicMax(&sm.maxlast, last);
    // this wave's own largest last contributor: entries past it touch none of
    // its pixels, so the wave skips them
    uint32_t wlast = last;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t u = (uint32_t)__shfl_xor((int)wlast, o, 64);
        wlast = u > wlast ? u : wlast;
    }
    // every lane holds the maximum; readfirstlane lets the compiler keep it,
    // and the entry loop below, in scalar registers
    wlast = (uint32_t)__builtin_amdgcn_readfirstlane((int)wlast);
    __syncthreads();
    const uint32_t stop = sm.maxlast;

    // One visited entry, predicated as in the forward: its contribution is
    // selected in or out through the factors (visited entries are finite, so a
    // zero factor zeroes every term).
    struct Terms {
        float dop, aT;  // dL/d(opacity * G) times G; alpha T
        bool contrib;
    };
    auto gradient = [&](const Eval& v, const float4& cl, uint32_t j) -> Terms {
        Terms r;
        r.contrib = j < last && v.power <= 0.0f && v.alpha >= 1.0f / 255.0f;
        // T_i = T / (1 - alpha) as the reference recovers it
        // (rasterizer_backward_cpu.cpp:85), with the hardware reciprocal
        // (1 ulp): gradients need 1e-3, not bits.  alpha <= 0.99, so the
        // reference's guard 1 - alpha > 1e-6 always holds.
        const float Ti = T * __builtin_amdgcn_rcpf(1.0f - v.alpha);
        float dal;
        {
            // gradient-only arithmetic: contracted to FMAs (the
            // contributor decisions above stay uncontracted)
#pragma clang fp contract(fast)
            dal = Ti * ((cl.x - acc0) * dC0 + (cl.y - acc1) * dC1 + (cl.z - acc2) * dC2);
        }
        // dL/d(opacity * G) = dal * G; dL/dpower = opacity times that,
        // and the opacity is applied once per Gaussian when the sums
        // leave LDS (alpha >= 0.99 is the clamp: no gradient)
        r.dop = (r.contrib && v.alpha < 0.99f) ? dal * v.ep : 0.0f;
        r.aT = r.contrib ? v.alpha * Ti : 0.0f;
        // colour behind the next entry: alpha c + (1 - alpha) acc
        const float ac = r.contrib ? v.alpha : 0.0f;
        {
#pragma clang fp contract(fast)
            acc0 += ac * (cl.x - acc0);
            acc1 += ac * (cl.y - acc1);
            acc2 += ac * (cl.z - acc2);
        }
        T = r.contrib ? Ti : T;
        return r;
    };

    for (uint32_t hi = stop; hi > start;) {
        const uint32_t lo = (hi - start > (uint32_t)BATCH) ? hi - BATCH : start;
        const int n = (int)(hi - lo);
        __syncthreads();
        for (int k = t; k < BATCH; k += 256) {
            uint32_t h = 0u;
            if (k < n) {
                uint32_t id = a.values[(size_t)(lo + k) * a.vstride];
                sm.id[k] = id;
                const float2 mm = a.means2D[id];
                const float4 cc = make_float4(a.conics[id * 3], a.conics[id * 3 + 1], a.conics[id * 3 + 2], a.opac[id]);
                sm.e[k].xy = mm;
                sm.e[k].co = prescale(cc);
                sm.e[k].rgb = make_float4(a.rgb[id * 3], a.rgb[id * 3 + 1], a.rgb[id * 3 + 2], 0.0f);
                h = strip_hits<false>(mm, cc, tx0, ty0);
            }
            store_masks<BATCH>(sm.mask, k >> 6, h, lane);
#pragma unroll
            for (int c = 0; c < NG; c++) sm.g[k][c] = 0.0f;
        }
        __syncthreads();
        // this wave's entries, back to front from its last contributor
        const int kmax = wlast <= lo ? -1 : ((int)(wlast - lo) < n ? (int)(wlast - lo) : n) - 1;
        for (int ch = kmax >> 6; ch >= 0; ch--) {
            uint64_t bits = wave_uniform(sm.mask[w][ch]);
            if (ch == (kmax >> 6)) bits &= ~0ull >> (63 - (kmax & 63));
            while (bits != 0ull) {
                const int k = (ch << 6) + (63 - __builtin_clzll(bits));
                bits &= ~(1ull << (k & 63));
                const float4 cl = sm.e[k].rgb;
                const Eval v = evaluate(sm.e[k], fpx, fpy);
                const Terms r = gradient(v, cl, lo + (uint32_t)k);
                if (__ballot(r.contrib) != 0ull) {
                    const float sum = wave_reduce9(r.dop, v.dx, v.dy, r.aT * dC0, r.aT * dC1, r.aT * dC2, role);
                    if (role.term >= 0 && sum != 0.0f)
                        atomicAdd(&sm.g[0][0] + (__builtin_amdgcn_readfirstlane(k * NG) + role.term), sum);
                }
            }
        }
        __syncthreads();
        // One (Gaussian, term) per thread, nine consecutive lanes per Gaussian:
        // its atomics into one array are one request per line, four or five for
        // the nine terms.  With a thread per Gaussian and nine instructions of
        // 64 scattered lines each, the atomics held the kernel up by 105 us at
        // 1M Gaussians and 1080p (612 -> 474 us with this order), 332 -> 263 us
        // at 200k and 720p.
        // Sums of dop * (dx, dy, dx^2, dx dy, dy^2); times the opacity they are
        // those of dpow, and -> the reference's terms
        // (rasterizer_backward_cpu.cpp): d_mean = -(a Sx + b Sy, c Sy + b Sx),
        // d_conic = (-Sxx / 2, -Sxy, -Syy / 2); the staged conic is
        // (-a/2, -b, -c/2, o)
        for (int i = t; i < n * NG; i += 256) {
            const int k = i / NG, c = i - k * NG;
            const uint32_t id = sm.id[k];
            float v = (&sm.g[0][0])[i];
            float* dst;
            if (c < 5) {
                const float4 cs = sm.e[k].co;
                if (c < 2) {
                    const float ca = -2.0f * (c == 0 ? cs.x : cs.z), cb = -cs.y;
                    v = -(ca * (cs.w * v) + cb * (cs.w * sm.g[k][1 - c]));
                    dst = &g.d_means2D[id].x + c;
                } else {
                    v = (c == 3 ? -1.0f : -0.5f) * (cs.w * v);
                    dst = g.d_conics + (size_t)id * 3 + (c - 2);
                }
            } else {
                dst = c < 8 ? g.d_rgb + (size_t)id * 3 + (c - 5) : g.d_op + id;
            }
            if (v != 0.0f) unsafeAtomicAdd(dst, v);
        }
        hi = lo;
    }
}

template <int BATCH, bool PAIR>
__global__ __launch_bounds__(256) void raster_fwd_kernel(RasterArgs a, PixOut o) {
    __shared__ FwdSmem<BATCH> sm;
    fwd_tile<BATCH, PAIR>(a, gsd::xcd_remap(blockIdx.x, gridDim.x), sm, o);
}

template <int BATCH>
__global__ __launch_bounds__(256) void raster_bwd_kernel(RasterArgs a, PixIn in, GradArgs g) {
    __shared__ BwdSmem<BATCH> sm;
    bwd_tile<BATCH>(a, gsd::xcd_remap(blockIdx.x, gridDim.x), sm, in, g);
}

// ------------------------------------------------------------ multi-view ----
// View of a global tile (views are few; every thread of the group scans the
// same table, so the loop is uniform).
__device__ __forceinline__ int view_of(const MultiRaster& m, int gtile) {
    int v = 0;
    while (v + 1 < m.V && m.views[v + 1].w <= gtile) v++;
    return v;
}

__device__ __forceinline__ RasterArgs view_args(const MultiRaster& m, int v) {
    const int4 vi = m.views[v];  // (W, H, gx, first global tile)
    RasterArgs a;
    a.W = vi.x;
    a.H = vi.y;
    a.gx = vi.z;
    a.means2D = m.means2D + (size_t)v * m.N;
    a.conics = m.conics + (size_t)v * m.N * 3;
    a.opac = m.opac + (size_t)v * m.N;
    a.rgb = m.rgb + (size_t)v * m.N * 3;
    a.values = m.values;
    a.vstride = m.vstride;
    a.ranges = m.ranges + 2 * (size_t)vi.w;
    a.bg0 = m.bg0;
    a.bg1 = m.bg1;
    a.bg2 = m.bg2;
    return a;
}

// Next global tile: blockIdx.x (one group per tile, XCD-remapped), or from the
// persistent work queues.  The queues are 8 counters over 8 contiguous ranges of
// global tiles; a group starts on the queue of its own XCD (so neighbouring
// tiles share an L2) and moves to the next queue when one runs dry.  Every
// pass takes a fresh counter value, so each group leaves after at most
// total_tiles + 8 passes.
constexpr int NQ = 8;

struct QueueState {
    int q;     // queues tried so far
    int tile;  // broadcast slot
};

__device__ __forceinline__ bool next_tile(const MultiRaster& m, int& g, int& iter, QueueState* s) {
    if (m.counter == nullptr) {
        g = gsd::xcd_remap(blockIdx.x, gridDim.x);
        return iter++ == 0 && blockIdx.x < (unsigned)m.total_tiles;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (iter++ == 0) s->q = 0;
        const int k = m.total_tiles / NQ, r = m.total_tiles % NQ;
        int tile = -1;
        while (s->q < NQ) {
            const int qi = ((int)(blockIdx.x % NQ) + s->q) % NQ;
            const int len = k + (qi < r ? 1 : 0);
            const int i = (int)atomicAdd(&m.counter[qi], 1u);
            if (i < len) {
                tile = qi * k + (qi < r ? qi : r) + i;
                break;
            }
            s->q++;
        }
        s->tile = tile;
    }
    __syncthreads();
    g = s->tile;
    return g >= 0;
}

template <int BATCH>
__global__ __launch_bounds__(256) void raster_fwd_multi_kernel(MultiRaster m, MultiPix o) {
    __shared__ FwdSmem<BATCH> sm;
    __shared__ QueueState qs;
    int g, iter = 0;
    while (next_tile(m, g, iter, &qs)) {
        const int v = view_of(m, g);
        RasterArgs a = view_args(m, v);
        const size_t p0 = (size_t)m.pix_off[v];
        PixOut po{o.img + p0 * 3, o.T_final + p0, o.n_contrib + p0, o.last_contrib + p0};
        fwd_tile<BATCH, false>(a, g - m.views[v].w, sm, po);
    }
}

template <int BATCH>
__global__ __launch_bounds__(256) void raster_bwd_multi_kernel(MultiRaster m, MultiPix o, MultiGrads gr) {
    __shared__ BwdSmem<BATCH> sm;
    __shared__ QueueState qs;
    int g, iter = 0;
    while (next_tile(m, g, iter, &qs)) {
        const int v = view_of(m, g);
        RasterArgs a = view_args(m, v);
        const size_t p0 = (size_t)m.pix_off[v];
        PixIn pi{o.T_final + p0, o.last_contrib + p0, o.d_image + p0 * 3};
        const size_t n0 = (size_t)v * m.N;
        GradArgs ga{gr.d_means2D + n0, gr.d_conics + n0 * 3, gr.d_rgb + n0 * 3, gr.d_op + n0};
        bwd_tile<BATCH>(a, g - m.views[v].w, sm, pi, ga);
    }
}

}  // namespace gsr

using namespace gsr;

hipError_t launch_raster_fwd(const RasterArgs& a, int num_tiles, int batch, float* img, float* T_final, int* n_contrib,
                             uint32_t* last_contrib, hipStream_t s) {
    if (num_tiles <= 0) return hipSuccess;
    PixOut o{img, T_final, n_contrib, last_contrib};
    // Up to 1024 tiles (four waves per SIMD) a wave's own instruction chain sets
    // the pace, and two entries at a time overlap it: 43 -> 36 us at 256 tiles
    // (10k Gaussians), 70 -> 62 us at 520; from 3400 tiles on it is a draw.
    const bool pair = num_tiles <= 1024;
    switch (batch) {
#define FWD(B)                                                              \
    case B:                                                                 \
        if (pair) raster_fwd_kernel<B, true><<<num_tiles, 256, 0, s>>>(a, o); \
        else raster_fwd_kernel<B, false><<<num_tiles, 256, 0, s>>>(a, o);   \
        break
        FWD(64);
        FWD(128);
        FWD(256);
        FWD(512);
#undef FWD
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_raster_bwd(const RasterArgs& a, int num_tiles, int batch, const float* T_final,
                             const uint32_t* last_contrib, const float* d_image, const GradArgs& g, hipStream_t s) {
    if (num_tiles <= 0) return hipSuccess;
    PixIn in{T_final, last_contrib, d_image};
    switch (batch) {
        case 64: raster_bwd_kernel<64><<<num_tiles, 256, 0, s>>>(a, in, g); break;
        case 128: raster_bwd_kernel<128><<<num_tiles, 256, 0, s>>>(a, in, g); break;
        case 256: raster_bwd_kernel<256><<<num_tiles, 256, 0, s>>>(a, in, g); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// grid: one group per global tile, or `persistent_groups` groups pulling
// tiles from the 8 queue counters at m.counter (zero at launch).
hipError_t launch_raster_fwd_multi(const MultiRaster& m, const MultiPix& o, int batch, int persistent_groups,
                                   hipStream_t s) {
    if (m.total_tiles <= 0) return hipSuccess;
    int grid = m.counter ? persistent_groups : m.total_tiles;
    switch (batch) {
        case 64: raster_fwd_multi_kernel<64><<<grid, 256, 0, s>>>(m, o); break;
        case 128: raster_fwd_multi_kernel<128><<<grid, 256, 0, s>>>(m, o); break;
        case 256: raster_fwd_multi_kernel<256><<<grid, 256, 0, s>>>(m, o); break;
        case 512: raster_fwd_multi_kernel<512><<<grid, 256, 0, s>>>(m, o); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_raster_bwd_multi(const MultiRaster& m, const MultiPix& o, const MultiGrads& g, int batch,
                                   int persistent_groups, hipStream_t s) {
    if (m.total_tiles <= 0) return hipSuccess;
    int grid = m.counter ? persistent_groups : m.total_tiles;
    switch (batch) {
        case 64: raster_bwd_multi_kernel<64><<<grid, 256, 0, s>>>(m, o, g); break;
        case 128: raster_bwd_multi_kernel<128><<<grid, 256, 0, s>>>(m, o, g); break;
        case 256: raster_bwd_multi_kernel<256><<<grid, 256, 0, s>>>(m, o, g); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
