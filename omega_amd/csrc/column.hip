// column.hip -- projections of 3-D (ring-pair) sinograms by image columns.
//
// Every plane of a sinogram repeats the same transaxial LORs: an oblique LOR crosses the x and y boundaries of the
// image at the same parameters as its neighbours in the other planes, and between two of them it stays in one
// column of voxels (fixed x, y), moving along z. So a wave takes one transaxial bin and 64 planes, one per lane:
// the crossings of the bin (pixel, exit parameter) are traced once per handle and kept, and all lanes read them
// through scalar loads; a lane keeps only its z walk, and the lanes' voxels lie within one column, which is
// contiguous in a z-fastest image (Nz floats, a few cache lines) -- in the one-lane-per-LOR kernels every lane
// gathers from, or adds to, a line of its own.
//
// Forward projection: z-fastest copy of the image, sums in the walk's order with its float operations
// (bit-identical to the one-lane-per-LOR kernel). Backprojection: a workgroup owns a tile of columns and a share of
// the segments (bin, entries inside the tile) of the lists, accumulates in LDS in 64-bit fixed point (as the
// direct-plane kernels: float LDS atomics retire 15 times slower, and global float atomics at 21 G segments of 64
// bytes per second however few lanes a segment serves), and adds the tile to the image once, in runs of
// consecutive x.
//
// LORs whose set-up differs from their bin's (along an image axis in a direct plane, entering the image through an
// end face, dropped or displaced by rounding) are listed and take the one-lane-per-LOR walk.
#include "column.hpp"
#include "geom.hpp"
#include "siddon_device.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <type_traits>
#include <vector>

namespace omg {

constexpr uint32_t kCL = 64;        // planes per wave

struct ColStart { float tc, tx0, ty0; uint32_t xy; };   // where a bin's walk enters the image
struct ColSeg { uint32_t bin, k0, k1; };                // entries [k0, k1) of the lists lie in one tile
struct ColItem { uint32_t tile, s0, s1; };              // one workgroup's segments

struct ColPlan {
    int64_t first = 0, n = 0;
    bool ok = false;
    uint32_t bins = 0;
    const uint32_t* bin_of = nullptr;   // measurement-level subsets: the range's first plane in the index table
    uint32_t* off = nullptr;            // [bins + 1]; the allocation that holds the other lists too
    ColStart* start = nullptr;
    uint2* ent = nullptr;               // {x | y << 16, exit parameter}
    uint32_t tw = 0, th = 0, ntx = 0;   // tile width, height; tiles per row
    ColSeg* seg = nullptr;
    ColItem* item = nullptr;
    uint32_t items = 0, tpb = 0;
};

// A bin's records, one group of planes: the largest |value| as float bits, and the sum of the |values|.
struct ColPeak { uint32_t top; float sum; };

struct ColView {
    uint32_t bins, planes, tw, th, ntx;
    const uint32_t* off;
    const ColStart* start;
    const uint2* ent;
    const ColSeg* seg;
    const ColItem* item;
};

// ---- building ----------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t col_tile(uint32_t xy, uint32_t tw, uint32_t th, uint32_t ntx) {
    return (xy & 0xffffu) / tw + (xy >> 16) / th * ntx;
}

// The transaxial walk of bin j: visit(xy, exit parameter) for each pixel in order; false when the bin's LORs are
// irregular in every plane or miss the image.
template <typename Visit>
__device__ __forceinline__ bool col_walk(const SidArgs& a, uint32_t j, ColStart& st, Visit&& visit) {
    Ray r;
    fetch_ray_base(a, j, r);
    const float xdf = r.xd - r.xs, ydf = r.yd - r.ys;
    st = ColStart{__builtin_nanf(""), 0.f, 0.f, 0u};
    if (isinf(ydf) || isinf(xdf)) return false;
    int32_t ti = 0, tj = 0, ux = 0, uy = 0;
    float txu = 0.f, tyu = 0.f, tc = 0.f, tx0 = 1e8f, ty0 = 1e8f;
    // a LOR along one image axis crosses that axis only (siddon_setup's branches for oblique planes)
    auto along = [&](float b, float bmax, float d, float src, float dst, float diff, uint32_t N, int32_t& i, int32_t& u,
                     float& t0, float& tu) {
        t0 = (b - src) / diff;
        const float tb = (bmax - src) / diff, tmin = mn(t0, tb), tmax = mx(t0, tb);
        tc = tmin;
        if (tc >= tmax) return false;
        uint32_t vmin = 0, vmax = 0;
        if (src < dst) axis_inc(tc, tmin, tmax, tmax, vmin, vmax, t0, u, diff, b, d, src, N);
        else axis_dec(tc, tmin, tmax, tmax, vmin, vmax, t0, u, diff, b, d, src, N);
        i = src < dst ? 0 : (int32_t)N - 1;
        tu = d / fabsf(diff);
        return true;
    };
    if (fabsf(ydf) < 1e-8f) {
        tj = perp_start(a.by, r.yd, a.dy, a.Ny);
        if (fabsf(xdf) < 1e-8f || r.yd > a.bmaxy || r.yd < a.by ||
            !along(a.bx, a.bmaxx, a.dx, r.xs, r.xd, xdf, a.Nx, ti, ux, tx0, txu))
            return false;
    } else if (fabsf(xdf) < 1e-8f) {
        ti = perp_start(a.bx, r.xd, a.dx, a.Nx);
        if (r.xd > a.bmaxx || r.xd < a.bx ||
            !along(a.by, a.bmaxy, a.dy, r.ys, r.yd, ydf, a.Ny, tj, uy, ty0, tyu))
            return false;
    } else {
        uint32_t Np = 0;
        if (preloop2(a.bx, a.by, xdf, ydf, a.bmaxx, a.bmaxy, a.dx, a.dy, a.Nx, a.Ny, ti, tj, txu, tyu, Np, r.ys, r.xs,
                     r.yd, r.xd, tc, ux, uy, tx0, ty0))
            return false;
    }
    st = ColStart{tc, tx0, ty0, (uint32_t)ti | (uint32_t)tj << 16};
    while ((uint32_t)ti < a.Nx && (uint32_t)tj < a.Ny) {
        const bool y = ty0 < tx0;
        visit((uint32_t)ti | (uint32_t)tj << 16, y ? ty0 : tx0);
        if (y) { tj += uy; ty0 += tyu; }
        else { ti += ux; tx0 += txu; }
    }
    return true;
}

// Bin j's LOR misses the image, or enters it after 1e-3 of its way and leaves it before 1 - 1e-3: every crossing parameter
// of its walk then lies in [0, 1], and a length is a parameter step times the LOR's (as ring_table asks of all LORs of
// a direct-plane sinogram).
__device__ __forceinline__ bool col_ring(const SidArgs& a, uint32_t j) {
    Ray r;
    fetch_ray_base(a, j, r);
    double t0 = 0.0, t1 = 1.0;
    bool miss = false;
    auto clip = [&](double s, double e, double lo, double hi) {
        const double dd = e - s;
        if (dd == 0.0) {
            miss = miss || s < lo || s > hi;
            return;
        }
        const double ta = (lo - s) / dd, tb = (hi - s) / dd;
        t0 = fmax(t0, fmin(ta, tb));
        t1 = fmin(t1, fmax(ta, tb));
    };
    clip(r.xs, r.xd, a.bx, a.bmaxx);
    clip(r.ys, r.yd, a.by, a.bmaxy);
    return miss || t0 >= t1 || !(t0 < 1e-3 || t1 > 1.0 - 1e-3);
}

// One plan's arrays while it is built (blockIdx.y of the launches below).
struct ColTrace {
    int64_t first;               // index table: the range's first measurement
    uint32_t* cnt;               // [bins] entries
    uint32_t* tile_cnt;          // [tiles] segments
    int32_t* bad;                // not the same bins in every plane, or a LOR that starts or ends in the image
    uint32_t* group_cnt;         // [workgroups][tiles]
    uint32_t* tile_cur;          // [tiles] segments placed so far
    // filling pass; null: no plan
    const uint32_t* off;
    const uint32_t* tile_off;
    ColStart* start;
    uint2* ent;
    ColSeg* seg;
};
constexpr uint32_t kColBatch = 8;
struct ColTraces { ColTrace t[kColBatch]; };

// One lane per bin. Counting pass: entries, and segments per tile. Filling pass: the lists, and the
// segments in their tiles' ranges. The tiles' counters are shared by every bin, so a workgroup adds its own
// counts (LDS, up to kTileLds tiles) once; they stay in group_cnt for the filling pass.
constexpr uint32_t kTileLds = 2048;

__global__ __launch_bounds__(256) void k_col_trace(SidArgs a, uint32_t bins, uint32_t tw, uint32_t th, uint32_t ntx,
                                                   uint32_t tiles, bool fill, ColTraces all) {
    __shared__ uint32_t mine[kTileLds];
    const ColTrace& q = all.t[blockIdx.y];
    if (fill && !q.ent) return;
    if (a.index) a.plane_offset = q.first;
    uint32_t* tile_cnt = fill ? q.tile_cur : q.tile_cnt;
    const uint32_t j = blockIdx.x * 256 + threadIdx.x;
    const bool shared = tiles <= kTileLds;
    uint32_t* group = q.group_cnt + (size_t)blockIdx.x * tiles;
    for (uint32_t i = threadIdx.x; i < (shared ? tiles : 0u); i += 256) mine[i] = fill ? group[i] : 0u;
    __syncthreads();
    ColStart st;
    uint32_t n = 0, tile = 0xffffffffu;
    if (j < bins && !fill) {
        col_walk(a, j, st, [&](uint32_t xy, float) {
            const uint32_t t = col_tile(xy, tw, th, ntx);
            if (t != tile) atomicAdd(shared ? mine + t : tile_cnt + t, 1u);
            tile = t;
            n++;
        });
        q.cnt[j] = n;
        if (!col_ring(a, j)) *q.bad = 1;
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < (shared ? tiles : 0u); i += 256) {
        if (!fill) group[i] = mine[i];
        if (mine[i]) mine[i] = atomicAdd(tile_cnt + i, mine[i]);   // filling pass: this workgroup's first slot
    }
    if (!fill) return;
    __syncthreads();
    if (j >= bins) return;
    const uint32_t o = q.off[j];
    uint32_t k0 = o;
    n = o;
    tile = 0xffffffffu;
    auto close = [&]() {
        if (tile != 0xffffffffu)
            q.seg[q.tile_off[tile] + atomicAdd(shared ? mine + tile : tile_cnt + tile, 1u)] = ColSeg{j, k0, n};
    };
    col_walk(a, j, st, [&](uint32_t xy, float tn) {
        const uint32_t t = col_tile(xy, tw, th, ntx);
        if (t != tile) {
            close();
            tile = t;
            k0 = n;
        }
        q.ent[n++] = make_uint2(xy, __float_as_uint(tn));
    });
    close();
    q.start[j] = st;
}

// *bad = 1 unless measurement i of the range is bin index[i % bins] of plane i / bins.
__global__ __launch_bounds__(256) void k_col_check(const uint32_t* __restrict__ table, uint64_t n, uint32_t bins,
                                                   uint32_t per, ColTraces all) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint32_t* index = table + all.t[blockIdx.y].first;
    const uint32_t p = (uint32_t)(i / bins), c = index[i - (uint64_t)p * bins];
    if (c >= per || index[i] != c + p * per) *all.t[blockIdx.y].bad = 1;
}

__global__ void k_col_zero(uint32_t* p, uint32_t n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// ---- running -----------------------------------------------------------------------------------------
// dst[x + y Nx][z + lead] = src[x + y Nx + z Nx Ny], columns of `pitch` with zeros around the image's Nz; clears
// the launch's state. grid = (ceil(Nx / 32), Ny, ceil(pitch / 32)), block = (32, 8).
__global__ __launch_bounds__(256) void k_col_zfast(const float* __restrict__ src, float* __restrict__ dst, uint32_t Nx,
                                                   uint32_t Ny, uint32_t Nz, uint32_t pitch, uint32_t lead,
                                                   uint32_t* __restrict__ state) {
    __shared__ float t[32][33];
    const uint32_t x0 = blockIdx.x * 32, z0 = blockIdx.z * 32, y = blockIdx.y;
    if (blockIdx.x + blockIdx.y + blockIdx.z == 0 && threadIdx.y == 0 && threadIdx.x < 4) state[threadIdx.x] = 0u;
    for (uint32_t k = threadIdx.y; k < 32; k += 8) {
        const uint32_t x = x0 + threadIdx.x, z = z0 + k - lead;
        t[k][threadIdx.x] = x < Nx && z < Nz ? src[x + ((size_t)z * Ny + y) * Nx] : 0.f;
    }
    __syncthreads();
    for (uint32_t k = threadIdx.y; k < 32; k += 8) {
        const uint32_t x = x0 + k, z = z0 + threadIdx.x;
        if (x < Nx && z < pitch) dst[(x + (size_t)y * Nx) * pitch + z] = t[threadIdx.x][k];
    }
}

// The set-up of a LOR is its bin's: the bin's crossings are its own.
__device__ __forceinline__ bool col_regular(const Walk& w, const ColStart& st) {
    return !w.perp && w.tc == st.tc && w.tx0 == st.tx0 && w.ty0 == st.ty0 &&
           ((uint32_t)w.ti | (uint32_t)w.tj << 16) == st.xy;
}

// More than one z crossing per column is possible only if they lie closer together than a column's faces.
__device__ __forceinline__ bool col_steep(const Walk& w) {
    const float t = w.txu == 0.f ? w.tyu : w.tyu == 0.f ? w.txu : fminf(w.txu, w.tyu);
    return w.uz != 0 && w.tzu < 1.001f * t;
}

// A lane's z walk within the columns its wave passes. tk counts from `lead`; columns carry cells of no consequence in
// front of the image and behind it. `left` counts the steps that the LOR's walk may still take (0: it has ended). A
// lane that leaves the image stays in the end cell with tz0 = kColEnd; one that runs out of steps keeps tk and Lf = 0:
// their terms vanish without a test. `tc` is the same for every lane after each column (its exit), so it lives outside.
constexpr float kColEnd = 3e38f;
struct ColLane {
    float tz0, tzu, Lf;
    int32_t tk, uz, left;
};

__device__ __forceinline__ void col_end(ColLane& l) {
    l.left = 0;
    l.Lf = 0.f;
    l.tz0 = kColEnd;
}

// One column as the walk defines it: z crossings while they come first, then the exit. visit(parameter step, tk).
template <typename Visit>
__device__ __forceinline__ void col_step(ColLane& l, float tc, float tn, uint32_t Nz, uint32_t lead, Visit&& visit) {
    float t = tc;
    bool cross = l.left > 0 && l.tz0 < tn;
    while (__any(cross)) {
        if (cross) {
            visit(l.tz0 - t, l.tk);
            t = l.tz0;
            l.tz0 += l.tzu;
            l.tk += l.uz;
            l.left--;
            if ((uint32_t)l.tk - lead >= Nz || l.left == 0) col_end(l);
        }
        cross = l.left > 0 && l.tz0 < tn;
    }
    if (l.left > 0) {
        visit(tn - t, l.tk);
        if (--l.left == 0) col_end(l);
    }
}

// True when no lane can run out of steps in the next four columns (two per column, see `steep`).
__device__ __forceinline__ bool col_free(const ColLane& l) { return !__any(l.left > 0 && l.left <= 8); }

// Four entries of a list from k on by one scalar load (the lists never change); the allocation ends four later.
__device__ __forceinline__ void col_four(const uint2* ent, uint32_t k, uint2 (&e)[4]) {
    const auto* p = (const __attribute__((address_space(4))) uint32_t*)(uintptr_t)(ent + k);
#pragma unroll
    for (int j = 0; j < 4; j++) e[j] = make_uint2(p[2 * j], p[2 * j + 1]);
}

// One column of a lane that crosses at most one z plane in it: the pieces before and behind the crossing, piece(length,
// tk) and other(length, tk, crossed); an absent one has length 0. CHECK: the lane may run out of steps here.
template <bool CHECK, typename Piece, typename Other>
__device__ __forceinline__ void col_pair(ColLane& l, float tc, float tn, uint32_t Nz, uint32_t lead, Piece&& piece,
                                         Other&& other) {
    const bool cross = l.tz0 < tn;
    piece(fmaxf((cross ? l.tz0 : tn) - tc, 0.f) * l.Lf, l.tk);
    l.tk += cross ? l.uz : 0;
    if (CHECK) {
        l.left -= cross ? 1 : 0;
        l.Lf = cross && l.left <= 0 ? 0.f : l.Lf;
    }
    other(fmaxf(tn - l.tz0, 0.f) * l.Lf, l.tk, cross);
    l.tz0 = cross ? l.tz0 + l.tzu : l.tz0;
    l.tz0 = (uint32_t)l.tk - lead < Nz ? l.tz0 : kColEnd;
    if (CHECK && --l.left <= 0) {
        l.left = 0;
        l.Lf = 0.f;
        l.tz0 = kColEnd;
    }
}

// A wave's maximum and sum (of values >= 0), in lane 63: rows of 16 lanes first, then lane 15 of rows 0 and 2 into the
// rows behind, lane 31 into rows 2 and 3.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_or_0(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
template <typename Op>
__device__ __forceinline__ uint32_t wave_fold(uint32_t v, Op&& op) {
    v = op(v, dpp_or_0<0x111, 0xf>(v));
    v = op(v, dpp_or_0<0x112, 0xf>(v));
    v = op(v, dpp_or_0<0x114, 0xf>(v));
    v = op(v, dpp_or_0<0x118, 0xf>(v));
    v = op(v, dpp_or_0<0x142, 0xa>(v));
    return op(v, dpp_or_0<0x143, 0xc>(v));
}
__device__ __forceinline__ ColPeak wave_peak(float v) {
    v = fabsf(v);
    const uint32_t top = wave_fold(__float_as_uint(v), [](uint32_t a, uint32_t b) { return max(a, b); });
    const uint32_t sum = wave_fold(__float_as_uint(v), [](uint32_t a, uint32_t b) {
        return __float_as_uint(__uint_as_float(a) + __uint_as_float(b));
    });
    return ColPeak{top, __uint_as_float(sum)};   // NaN and Inf order above every number
}

// a * b, and 0 where a factor is 0 whatever the other one is
__device__ __forceinline__ float mul_or_zero(float a, float b) {
    float r;
    asm("v_mul_legacy_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

enum { COL_FP = 0, COL_OSEM = 1, COL_BP = 2 };

// One wave per bin and 64 planes, BPW bins one after the other. COL_FP: y = A img. COL_BP: the lanes' records for
// k_col_bp, {z walk, length, y * weight (weight alone when y is null)}, and with wrec the weights beside them.
// COL_OSEM: forward projection, ratio, records. peak, wpeak: each bin's of rec and wrec. state[1]: irregular LORs listed in
// `rest`. Measurements pass through LDS (a wave's lanes are a whole plane apart in
// them). A column of up to 64 NR - 1 slices is loaded into the wave's registers, lane z holding slice z, and every
// lane picks its slices by ds_bpermute; NR 0: lanes gather from memory. What bounds the forward projection: VALU,
// about 22 operations per column and 64 LORs besides 690 per LOR's set-up. 64 planes of 224 x 224 bins, 128 x 128 x 63:
// 217 us; 383 us with gathers (16 clocks of the texture address unit each, two per column) and 484 us by one lane per
// LOR.
template <int MODE, int BPW, int NR>
__global__ __launch_bounds__(256, MODE == COL_BP || NR > 1 ? 4 : MODE == COL_FP ? 6 : 5) void k_col_fp(
    ColView c, SidArgs a, uint32_t plane0, const float* __restrict__ Xz, const float* __restrict__ yin,
    float* __restrict__ yout, float4* __restrict__ rec, float* __restrict__ wrec, ColPeak* __restrict__ peak,
    ColPeak* __restrict__ wpeak, uint32_t* __restrict__ state, uint32_t* __restrict__ rest, float epps) {
    constexpr uint32_t NB = 4 * BPW;
    __shared__ float ys[kCL][NB + 1];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t bin0 = blockIdx.x * NB, pg = plane0 + blockIdx.y * kCL;
    if (MODE != COL_FP && yin) {
        for (uint32_t t = threadIdx.x; t < kCL * NB; t += 256) {
            const uint32_t b = t % NB, q = t / NB;
            ys[q][b] = bin0 + b < c.bins && pg + q < c.planes ? yin[(int64_t)(pg + q) * c.bins + bin0 + b] : 0.f;
        }
        __syncthreads();
    }
    const uint32_t p = pg + lane;
    const bool in = p < c.planes;
    constexpr uint32_t lead = NR ? 0u : 1u;
    const uint32_t zp = NR ? 64u * NR : a.Nz + 2;
    const __amdgpu_buffer_rsrc_t cols = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(Xz), 0, NR ? (int)(a.Nx * a.Ny * 256u * NR) : 0, 0x00027000);
    for (uint32_t i = 0; i < BPW; i++) {
        const uint32_t b = wave * BPW + i, bin = bin0 + b;
        if (bin >= c.bins) break;
        const int64_t lo = (int64_t)p * c.bins + bin;
        const ColStart st = c.start[bin];
        Walk w;
        float weight = 0.f, yhat = 0.f;
        const bool hit = in && siddon_setup<false>(a, lo, w, weight);
        const bool reg = hit && col_regular(w, st);
        {   // irregular LORs: a list for k_col_rest
            const uint64_t m = __ballot(hit && !reg);
            if (m) {
                uint32_t o = 0;
                if (lane == 0) o = atomicAdd(state + 1, (uint32_t)__popcll(m));
                o = __builtin_amdgcn_readfirstlane(o);
                if (hit && !reg) rest[o + __popcll(m & ((1ull << lane) - 1))] = (uint32_t)lo;
            }
        }
        if (MODE != COL_BP) {
            float ax = 0.f;
            if (__any(reg)) {
                ColLane l{w.tz0, w.tzu, w.L, w.tk + (int32_t)lead, w.uz, (int32_t)w.left};
                if (!reg) {
                    l.tk = 0;
                    l.uz = 0;
                    col_end(l);
                }
                const bool steep = __any(reg && col_steep(w));
                float tc = st.tc;
                const uint32_t e1 = __builtin_amdgcn_readfirstlane(c.off[bin + 1]);
                uint32_t k = __builtin_amdgcn_readfirstlane(c.off[bin]);
                while (k < e1) {
                    if (!steep) {
                        // straight line, four columns at a time, the next four loading meanwhile; behind the list's
                        // end its last column again, where no length is left
                        uint2 e[4], en[4];
                        float r0[4], r1[4], n0[4], n1[4];
                        auto load = [&](uint32_t kk, uint2 (&ee)[4], float* q0, float* q1) {
                            col_four(c.ent, kk, ee);
#pragma unroll
                            for (int j = 1; j < 4; j++) ee[j] = kk + j < e1 ? ee[j] : ee[j - 1];
#pragma unroll
                            for (int j = 0; j < 4 && NR; j++) {
                                const int32_t o =
                                    (int32_t)(((ee[j].x & 0xffffu) + (ee[j].x >> 16) * a.Nx) * (256u * NR));
                                auto slice = [&](uint32_t z) {
                                    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(cols, 4 * z, o, 0));
                                };
                                q0[j] = slice(lane);
                                if (NR > 1) q1[j] = slice(64 + lane);
                            }
                        };
                        auto batch = [&](auto check) {
                            float l1[4], l2[4], v1[4], v2[4];
                            const int32_t tk0 = l.tk;
#pragma unroll
                            for (int j = 0; j < 4; j++) {
                                const float tn = __uint_as_float(e[j].y);
                                const char* col = reinterpret_cast<const char*>(
                                    Xz + (size_t)((e[j].x & 0xffffu) + (e[j].x >> 16) * a.Nx) * zp);
                                auto voxel = [&](int32_t tk) {
                                    if (!NR) return *reinterpret_cast<const float*>(col + 4u * (uint32_t)tk);
                                    auto pick = [&](float q) {
                                        return __int_as_float(__builtin_amdgcn_ds_bpermute(4 * tk, __float_as_int(q)));
                                    };
                                    if (NR < 2) return pick(r0[j]);
                                    const float q0 = pick(r0[j]), q1 = pick(r1[j]);
                                    return (tk & 64) ? q1 : q0;
                                };
                                col_pair<decltype(check)::value>(
                                    l, tc, tn, a.Nz, lead,
                                    [&](float len, int32_t tk) { l1[j] = len; v1[j] = voxel(tk); },
                                    [&](float len, int32_t tk, bool) { l2[j] = len; v2[j] = voxel(tk); });
                                tc = tn;
                            }
                            // steps taken; a lane that has ended stays at 0
                            if (!decltype(check)::value) l.left = max(l.left - 4 - abs(l.tk - tk0), 0);
                            if ((uint32_t)l.tk - lead >= a.Nz) col_end(l);
#pragma unroll
                            for (int j = 0; j < 4; j++) {   // 0 times anything is 0 here: no term for an empty piece
                                ax += mul_or_zero(l1[j], v1[j]);
                                ax += mul_or_zero(l2[j], v2[j]);
                            }
                        };
                        load(k, e, r0, r1);
                        for (; k < e1; k += 4) {
                            load(k + 4 < e1 ? k + 4 : k, en, n0, n1);
                            __builtin_amdgcn_sched_barrier(0);
                            if (col_free(l)) batch(std::false_type());
                            else batch(std::true_type());
#pragma unroll
                            for (int j = 0; j < 4; j++) {
                                e[j] = en[j];
                                r0[j] = n0[j];
                                r1[j] = n1[j];
                            }
                        }
#pragma unroll
                        for (int j = 0; j < 4 && NR; j++) {   // a use on the way out keeps the loads ahead of the sums
                            asm volatile("" ::"v"(r0[j]));
                            if (NR > 1) asm volatile("" ::"v"(r1[j]));
                        }
                    } else {
                        const uint32_t ke = min(k + 4, e1);
                        for (; k < ke; k++) {
                            const uint2 e = c.ent[k];
                            const float tn = __uint_as_float(e.y);
                            const float* col = Xz + (size_t)((e.x & 0xffffu) + (e.x >> 16) * a.Nx) * zp;
                            col_step(l, tc, tn, a.Nz, lead, [&](float dt, int32_t tk) {
                                const float len = dt * l.Lf;
                                if (len > 0.f) ax += len * col[tk];
                            });
                            tc = tn;
                        }
                    }
                }
            }
            yhat = hit ? ax * weight : 0.f;
            if (MODE == COL_FP) {
                ys[lane][b] = yhat;
                continue;
            }
        }
        float v = 1.f;
        if (MODE == COL_OSEM) {
            v = 0.f;
            if (hit) {
                v = ys[lane][b] / ratio_den(a, lo, yhat, epps);
                if (isnan(v) || isinf(v)) v = epps;
            }
        } else if (yin) {
            v = ys[lane][b];
        }
        const float keep = reg ? v * weight : 0.f;
        // bit 15 of tk: more than one z crossing per column is possible
        const uint32_t steep = reg && col_steep(w) ? 0x8000u : 0u;
        rec[((size_t)blockIdx.y * c.bins + bin) * kCL + lane] =
            make_float4(w.tz0, w.L, keep, __uint_as_float((uint32_t)(w.tk + 1) | steep | w.left << 16));
        const ColPeak pk = wave_peak(keep);
        if (lane == 63) peak[(size_t)blockIdx.y * c.bins + bin] = pk;
        if (wrec) {
            const float kw = reg ? weight : 0.f;
            wrec[((size_t)blockIdx.y * c.bins + bin) * kCL + lane] = kw;
            const ColPeak pw = wave_peak(kw);
            if (lane == 63) wpeak[(size_t)blockIdx.y * c.bins + bin] = pw;
        }
    }
    if (MODE == COL_FP) {
        __syncthreads();
        for (uint32_t t = threadIdx.x; t < kCL * NB; t += 256) {
            const uint32_t b = t % NB, q = t / NB;
            if (bin0 + b < c.bins && pg + q < c.planes) yout[(int64_t)(pg + q) * c.bins + bin0 + b] = ys[q][b];
        }
    }
}

// The irregular LORs of a k_col_fp launch, one per lane, by the walk of the one-lane-per-LOR kernels: thread `i` of
// `step`.
struct ColRest {
    const uint32_t* list;
    const float* img;        // image (x fastest); null: backprojection of yin alone
    const float* yin;
    float* yout;             // forward projection
    float *rhs, *sens;
    float epps;
};

__device__ __forceinline__ void col_rest(const SidArgs& a, const ColRest& r, uint32_t n, uint32_t i, uint32_t step) {
    for (; i < n; i += step) {
        const int64_t lo = r.list[i];
        float v = !r.img && r.yin ? r.yin[lo] : 1.f, weight = 0.f;
        if (r.img) {
            float ax = 0.f;
            const bool hit = siddon_gather<false>(a, lo, r.img, ax, weight);
            const float yhat = hit ? ax * weight : 0.f;
            if (r.yout) {
                r.yout[lo] = yhat;
                continue;
            }
            v = r.yin[lo] / ratio_den(a, lo, yhat, r.epps);
            if (isnan(v) || isinf(v)) v = r.epps;
        }
        if (v == 0.f && !r.sens) continue;
        siddon_trace(a, lo, weight, [&](uint32_t ind, float len) {
            const float lw = len * weight;
            unsafeAtomicAdd(r.rhs + ind, v * lw);
            if (r.sens) unsafeAtomicAdd(r.sens + ind, lw);
        });
    }
}

__global__ __launch_bounds__(64) void k_col_rest(SidArgs a, const uint32_t* __restrict__ state, ColRest r) {
    col_rest(a, r, state[1], blockIdx.x * 64 + threadIdx.x, gridDim.x * 64);
}

// Backprojection. Blocks [0, rest_blocks) of x take the irregular LORs (first, as theirs are the longest chains);
// every other block one item: LDS accumulators [tile pixel][Nz + 2], int64 fixed point; the end cells are dropped.
// blockIdx.z 1: the weights into sens instead of the records' values into rhs. What bounds it: the LDS atomics (64
// lanes over one column's cells) and about 35 VALU operations per column and 64 LORs. 64 planes of 224 x 224 bins,
// 128 x 128 x 63: 285 us, with the records' launch 355 us; 5690 us by one lane per LOR (global float atomics).
__global__ __launch_bounds__(1024, 8) void k_col_bp(ColView c, SidArgs a, uint32_t plane0, uint32_t rest_blocks,
                                                    ColRest rest, const float4* __restrict__ rec,
                                                    const float* __restrict__ wrec, const ColPeak* __restrict__ peak,
                                                    const ColPeak* __restrict__ wpeak,
                                                    const uint32_t* __restrict__ state) {
    extern __shared__ unsigned long long acc64[];
    __shared__ uint32_t most[16], least[16];
    __shared__ float total[16];
    if (blockIdx.x < rest_blocks) {
        if (blockIdx.y + blockIdx.z == 0)
            col_rest(a, rest, state[1], blockIdx.x * blockDim.x + threadIdx.x, rest_blocks * blockDim.x);
        return;
    }
    const bool sens = blockIdx.z != 0;
    float* __restrict__ rhs = sens ? rest.sens : rest.rhs;
    const ColItem it = c.item[blockIdx.x - rest_blocks];
    const uint32_t x0 = it.tile % c.ntx * c.tw, y0 = it.tile / c.ntx * c.th;
    const uint32_t zp = a.Nz + 2, cells = c.tw * c.th * zp;
    auto bin_peak = [&](uint32_t q) {
        return q < it.s1 ? (sens ? wpeak : peak)[(size_t)blockIdx.y * c.bins + c.seg[q].bin] : ColPeak{0u, 0.f};
    };
    ColPeak pk = bin_peak(it.s0 + threadIdx.x);        // in flight while the cells are cleared
    for (uint32_t i = threadIdx.x; i < cells; i += blockDim.x) acc64[i] = 0ull;
    // The item's own scale: |term| <= peak * voxel diagonal, and a segment adds at most two terms to a voxel per lane.
    // One outlying LOR so costs bits where it passes only, and of its own size (the sum of the records bounds a voxel's,
    // not their number times the largest). Where not even the bins' largest terms keep 20 bits, the item adds floats.
    uint32_t top = 0, low = ~0u;
    float sum = 0.f;
    for (uint32_t q = it.s0 + threadIdx.x; q < it.s1; q += blockDim.x) {
        top = max(top, pk.top);
        low = min(low, pk.top ? pk.top : ~0u);
        sum += pk.sum;
        pk = bin_peak(q + blockDim.x);
    }
    top = wave_fold(top, [](uint32_t a, uint32_t b) { return max(a, b); });
    low = ~wave_fold(~low, [](uint32_t a, uint32_t b) { return max(a, b); });
    sum = __uint_as_float(wave_fold(__float_as_uint(sum), [](uint32_t a, uint32_t b) {
        return __float_as_uint(__uint_as_float(a) + __uint_as_float(b));
    }));
    if ((threadIdx.x & 63) == 63) {
        most[threadIdx.x >> 6] = top;
        least[threadIdx.x >> 6] = low;
        total[threadIdx.x >> 6] = sum;
    }
    __syncthreads();
    top = most[0];
    low = least[0];
    sum = total[0];
    for (uint32_t q = 1; q < blockDim.x >> 6; q++) {
        top = max(top, most[q]);
        low = min(low, least[q]);
        sum += total[q];
    }
    if (top == 0u) return;
    bool finite = top < 0x7f800000u;
    double up, down;
    {
        const float diag = sqrtf(a.dx * a.dx + a.dy * a.dy + a.dz * a.dz) * (1.f + 0x1p-10f);
        const float bt = finite ? __uint_as_float(top) * diag : 1.f;
        const float bs = 2.f * sum * diag * (1.f + 0x1p-10f);
        finite = finite && bs < __builtin_inff();
        fixed_scale(bt, finite ? fmaxf(bs, bt) : 1.f, up, down);
        finite = finite && (double)(__uint_as_float(low) * diag) * up >= 0x1p20;
    }
    const uint32_t lane = threadIdx.x & 63, p = plane0 + blockIdx.y * kCL + lane;
    ColLane l;
    float tzi = 0.f;
    l.tzu = 0.f;
    l.uz = 0;
    if (p < c.planes) {
        const float2 zz = *reinterpret_cast<const float2*>(a.z + (a.plane_col + p) * 2);
        l.tzu = a.dz / fabsf(zz.y - zz.x);
        tzi = fabsf(zz.y - zz.x) / a.dz;
        l.uz = zz.x < zz.y ? 1 : -1;
    }
    const int32_t uz = l.uz;
    const uint32_t waves = blockDim.x >> 6;
    uint32_t s = it.s0 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t group = (size_t)blockIdx.y * c.bins * kCL + lane;
    auto fetch = [&](uint32_t q) {
        const size_t o = group + (size_t)c.seg[q].bin * kCL;
        float4 r = rec[o];
        if (sens) r.z = wrec[o];
        return r;
    };
    float4 nx = s < it.s1 ? fetch(s) : make_float4(0.f, 0.f, 0.f, 0.f);
    for (; s < it.s1; s += waves) {
        const ColSeg sg = c.seg[s];
        const float4 r = nx;
        if (s + waves < it.s1) nx = fetch(s + waves);   // in flight during this segment
        const uint32_t o = c.off[sg.bin];
        const uint32_t bits = __float_as_uint(r.w);
        const float Lw = r.y * r.z;                       // length * record value; a term is a parameter step times it
        float tc = sg.k0 > o ? __uint_as_float(c.ent[sg.k0 - 1].y) : c.start[sg.bin].tc;
        l.tz0 = r.x;
        l.uz = uz;
        l.Lf = Lw;
        l.tk = (int32_t)(bits & 0x7fffu);
        l.left = (int32_t)(bits >> 16);
        if (r.z == 0.f) {
            l.tk = 0;
            l.uz = 0;
            col_end(l);
        }
        if (!__any(l.left > 0)) continue;
        const bool steep = __any(l.left > 0 && (bits & 0x8000u));
        if (l.tz0 < tc) {             // the z crossings before the tile
            const float n = fminf(floorf((tc - l.tz0) * tzi) + 1.f, (float)l.left);
            l.tz0 = __builtin_fmaf(n, l.tzu, l.tz0);
            l.tk += l.uz * (int32_t)n;
            l.left -= (int32_t)n;
            if ((uint32_t)(l.tk - 1) >= a.Nz) col_end(l);
        }
        l.left -= (int32_t)(sg.k0 - o);
        if (l.left <= 0) col_end(l);
        if (l.left > 0) {
            for (uint32_t k = sg.k0; k < sg.k1; k += 4) {
                if (finite && !steep) {
                    uint2 e[4];
                    col_four(c.ent, k, e);
                    auto batch = [&](auto check) {
                        const int32_t tk0 = l.tk;
#pragma unroll
                        for (uint32_t j = 0; j < 4; j++) {
                            if (j && k + j >= sg.k1) break;
                            const float tn = __uint_as_float(e[j].y);
                            unsigned long long* col =
                                acc64 + (((e[j].x >> 16) - y0) * c.tw + ((e[j].x & 0xffffu) - x0)) * zp;
                            col_pair<decltype(check)::value>(
                                l, tc, tn, a.Nz, 1u, [&](float len, int32_t tk) { lds_add_fixed(col + tk, len, up); },
                                [&](float len, int32_t tk, bool cross) {
                                    if (cross) lds_add_fixed(col + tk, len, up);
                                });
                            tc = tn;
                        }
                        if (!decltype(check)::value) l.left = max(l.left - 4 - abs(l.tk - tk0), 0);
                        if ((uint32_t)(l.tk - 1) >= a.Nz) col_end(l);
                    };
                    if (col_free(l)) batch(std::false_type());
                    else batch(std::true_type());
                } else {
                    for (uint32_t j = k; j < min(k + 4, sg.k1); j++) {
                        const uint2 e = c.ent[j];
                        const float tn = __uint_as_float(e.y);
                        const uint32_t ex = e.x & 0xffffu, ey = e.x >> 16;
                        unsigned long long* col = acc64 + ((ey - y0) * c.tw + (ex - x0)) * zp;
                        col_step(l, tc, tn, a.Nz, 1u, [&](float dt, int32_t tk) {
                            if (!(dt > 0.f)) return;
                            if (finite) lds_add_fixed(col + tk, dt * l.Lf, up);
                            else unsafeAtomicAdd(rhs + ex + (size_t)(ey + (size_t)(tk - 1) * a.Ny) * a.Nx, dt * l.Lf);
                        });
                        tc = tn;
                    }
                }
            }
        }
    }
    __syncthreads();
    if (!finite) return;
    // x fastest, so a wave's adds fall on runs of tw consecutive voxels
    for (uint32_t i = threadIdx.x; i < c.tw * c.th * a.Nz; i += blockDim.x) {
        const uint32_t lx = i % c.tw, q = i / c.tw, ly = q % c.th, z = q / c.th;
        const unsigned long long v = acc64[(ly * c.tw + lx) * zp + z + 1];
        if (v != 0ull) unsafeAtomicAdd(rhs + x0 + lx + (size_t)(y0 + ly + (size_t)z * a.Ny) * a.Nx, fixed_value(v, down));
    }
}

// ---- host ----------------------------------------------------------------------------------------------
struct ColBuffer {
    std::mutex mu;                  // held while a call's launches are issued
    hipStream_t s = nullptr;        // of the calls that used it last; their end is `done`
    hipEvent_t done = nullptr;      // (the null stream's buffer has none)
    float* p = nullptr;
    size_t floats = 0;
};

struct ColCache {
    std::vector<ColPlan*> e;
    std::mutex buffers_mu;
    std::vector<std::unique_ptr<ColBuffer>> buffers;
    size_t others = 0;              // of them for streams that are not the null stream
};

static void col_free(ColPlan* p) {
    hipFree(p->off);
    p->off = nullptr; p->start = nullptr; p->ent = nullptr; p->seg = nullptr; p->item = nullptr;
}

template <typename T>
static bool col_alloc(T** p, uint64_t n) {
    return hipMalloc(reinterpret_cast<void**>(p), (size_t)std::max<uint64_t>(n, 1) * sizeof(T)) == hipSuccess;
}

constexpr size_t kColLds = 76 * 1024;   // two workgroups of 16 waves per CU (one of 152 KB: 376 us, four of 38 KB: 310 us)
constexpr size_t kColPlans = 64;        // subsets of an index table that keep their lists
constexpr uint32_t kColRest = 32;       // workgroups of k_col_bp for the irregular LORs

// Columns per tile whose int64 accumulators fit LDS: 16 x 16 (64-byte runs of x) down to 1 x 1; 0: none.
static bool col_tile_size(uint32_t Nz, uint32_t* tw, uint32_t* th) {
    const size_t m = kColLds / (8 * ((size_t)Nz + 2));
    uint32_t w = 16, h = 16;
    while ((size_t)w * h > m && (w > 1 || h > 1)) {
        if (h >= w) h /= 2;
        else w /= 2;
    }
    *tw = w;
    *th = h;
    return (size_t)w * h <= m;
}

static size_t col_lds(uint32_t tw, uint32_t th, uint32_t Nz) { return (size_t)tw * th * (Nz + 2) * 8; }

// Lanes per workgroup of k_col_bp: a tile's LDS decides how many share a CU, 32 waves on it either way.
static uint32_t col_tpb(uint32_t tw, uint32_t th, uint32_t Nz) {
    const size_t lds = col_lds(tw, th, Nz);
    return lds > 38 * 1024 ? 1024 : lds > 19 * 1024 ? 512 : 256;
}

// The host's part of a plan from its counts (entries per bin, segments per tile): the layout, the items and the
// allocation, with the tables to upload. False when there is nothing to keep or it does not fit.
static bool col_layout_lists(const omg_geom* g, ColPlan* p, const uint32_t* hc, const uint32_t* ht, uint32_t tiles,
                             std::vector<uint32_t>& tables, size_t* at_toff) {
    std::vector<uint32_t> off((size_t)p->bins + 1), toff(tiles);
    uint64_t total = 0, segs = 0;
    for (uint32_t j = 0; j < p->bins; j++) {
        off[j] = (uint32_t)total;
        total += hc[j];
        if (total >= 0xFFFFFFF0ull) return false;
    }
    off[p->bins] = (uint32_t)total;
    for (uint32_t t = 0; t < tiles; t++) {
        toff[t] = (uint32_t)segs;
        segs += ht[t];
    }
    if (total * 8 + segs * 12 > (2ull << 30)) return false;
    // equal shares of the segments: one per wave at least (an item clears and adds its whole tile)
    std::vector<ColItem> items;
    p->tpb = col_tpb(p->tw, p->th, g->d.Nz);
    while (p->tpb > 256 && segs < 8 * 4096) p->tpb /= 2;    // few segments: more, smaller workgroups
    const uint64_t slots = 256 * (2048 / p->tpb);
    // four rounds of workgroups even out (294 us with two, 345 us with one)
    uint64_t share = std::max<uint64_t>(p->tpb / 64, (segs + 4 * slots - 1) / (4 * slots));
    for (uint64_t parts = ~0ull; share < segs && parts > 4 * slots - kColRest; share += (share + 63) / 64) {
        parts = 0;
        for (uint32_t t = 0; t < tiles; t++) parts += (ht[t] + share - 1) / share;
    }
    for (uint32_t t = 0; t < tiles; t++) {
        const uint32_t parts = (uint32_t)((ht[t] + share - 1) / share);
        for (uint32_t q = 0; q < parts; q++) {
            const uint32_t s0 = (uint32_t)((uint64_t)ht[t] * q / parts), s1 = (uint32_t)((uint64_t)ht[t] * (q + 1) / parts);
            items.push_back(ColItem{t, toff[t] + s0, toff[t] + s1});
        }
    }
    p->items = (uint32_t)items.size();
    if (p->items == 0) return false;
    // one allocation, the tables that the host made in front, uploaded by one copy
    auto round = [](size_t n) { return (n + 3) & ~(size_t)3; };
    *at_toff = round(off.size());
    const size_t at_item = *at_toff + round(tiles), at_start = at_item + round(3 * items.size());
    const size_t at_ent = at_start + 4 * (size_t)p->bins, at_seg = at_ent + 2 * (total + 4);
    tables.assign(at_start, 0u);
    std::copy(off.begin(), off.end(), tables.begin());
    std::copy(toff.begin(), toff.end(), tables.begin() + (ptrdiff_t)*at_toff);
    static_assert(sizeof(ColItem) == 12 && sizeof(ColSeg) == 12 && sizeof(ColStart) == 16, "table layout");
    std::memcpy(tables.data() + at_item, items.data(), items.size() * sizeof(ColItem));
    if (!col_alloc(&p->off, at_seg + 3 * segs)) return false;
    p->item = reinterpret_cast<ColItem*>(p->off + at_item);
    p->start = reinterpret_cast<ColStart*>(p->off + at_start);
    p->ent = reinterpret_cast<uint2*>(p->off + at_ent);
    p->seg = reinterpret_cast<ColSeg*>(p->off + at_seg);
    return true;
}

// Builds the plans in ps (the same number of measurements each, first and n set) together, kColBatch to a launch: between
// the launches and two waits, which are most of what one of them takes, they run beside each other. Sets their `ok`; one
// that is not ok holds nothing.
static void col_build(const omg_geom* g, const std::vector<ColPlan*>& ps, hipStream_t s) {
    const omg_geom_desc& d = g->d;
    const uint32_t per = d.size_x * d.size_y;
    uint32_t bins = per, tw = 0, th = 0;
    // with an index table a range has to be the same bins of every plane
    if (g->index_dev) bins = d.n_proj && ps[0]->n % d.n_proj == 0 ? (uint32_t)(ps[0]->n / d.n_proj) : 0u;
    if (bins == 0 || bins > per || !col_tile_size(d.Nz, &tw, &th)) return;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(k_col_bp), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)kColLds) != hipSuccess) {
        (void)hipGetLastError();
        return;
    }
    const uint32_t ntx = (d.Nx + tw - 1) / tw, tiles = ntx * ((d.Ny + th - 1) / th);
    const unsigned groups = grid_for(bins, 256);
    // [plans][bins], [plans][tiles + 1: bad] are read back together; [plans][tiles], for the filling pass, like the latter
    // cleared; [plans][workgroups][tiles]
    const uint64_t K = ps.size(), marks = tiles + 1ull, back = tiles <= kTileLds ? (uint64_t)groups * tiles : 0;
    const uint64_t at_marks = K * bins, at_cur = at_marks + K * marks, at_group = at_cur + K * tiles;
    const uint64_t words = at_group + K * back;
    uint32_t* temp = nullptr;
    std::vector<uint32_t> host(at_cur);
    std::vector<std::vector<uint32_t>> tables(ps.size());
    std::vector<ColTraces> traces((ps.size() + kColBatch - 1) / kColBatch, ColTraces{});
    if (words >= (1ull << 31) || !col_alloc(&temp, words)) {
        (void)hipGetLastError();
        return;
    }
    struct Temp {        // freed on every way out, after the copies from and to this function's tables
        uint32_t* p;
        hipStream_t s;
        ~Temp() { (void)hipStreamSynchronize(s); hipFree(p); }
    } const guard{temp, s};
    for (size_t k = 0; k < ps.size(); k++) {
        ColTrace& t = traces[k / kColBatch].t[k % kColBatch];
        t.first = ps[k]->first;
        t.cnt = temp + k * bins;
        t.tile_cnt = temp + at_marks + k * marks;
        t.bad = reinterpret_cast<int32_t*>(t.tile_cnt + tiles);
        t.tile_cur = temp + at_cur + k * tiles;
        t.group_cnt = temp + at_group + k * back;
        ps[k]->bins = bins;
        ps[k]->tw = tw;
        ps[k]->th = th;
        ps[k]->ntx = ntx;
        if (g->index_dev) ps[k]->bin_of = g->index_dev + ps[k]->first;
    }
    const SidArgs a = make_sid_args(g, 0, bins);
    auto trace = [&](bool fill) {
        for (size_t b = 0; b < traces.size(); b++) {
            const unsigned count = (unsigned)std::min<size_t>(kColBatch, ps.size() - b * kColBatch);
            if (!fill && g->index_dev)
                hipLaunchKernelGGL(k_col_check, dim3(grid_for(ps[0]->n, 256), count), dim3(256), 0, s, g->index_dev,
                                   (uint64_t)ps[0]->n, bins, per, traces[b]);
            hipLaunchKernelGGL(k_col_trace, dim3(groups, count), dim3(256), 0, s, a, bins, tw, th, ntx, tiles, fill,
                               traces[b]);
        }
        return hipGetLastError() == hipSuccess;
    };
    hipLaunchKernelGGL(k_col_zero, dim3(grid_for((int64_t)(at_group - at_marks), 256)), dim3(256), 0, s, temp + at_marks,
                       (uint32_t)(at_group - at_marks));
    if (!trace(false) || hipMemcpyAsync(host.data(), temp, host.size() * 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess) {
        (void)hipGetLastError();
        return;
    }
    bool any = false;
    for (size_t k = 0; k < ps.size(); k++) {
        ColPlan* p = ps[k];
        const uint32_t *hc = host.data() + k * bins, *ht = host.data() + at_marks + k * marks;
        size_t at_toff = 0;
        p->ok = ht[tiles] == 0 && col_layout_lists(g, p, hc, ht, tiles, tables[k], &at_toff) &&
                hipMemcpyAsync(p->off, tables[k].data(), tables[k].size() * 4, hipMemcpyHostToDevice, s) == hipSuccess;
        if (!p->ok) continue;
        ColTrace& t = traces[k / kColBatch].t[k % kColBatch];
        t.off = p->off;
        t.tile_off = p->off + at_toff;
        t.start = p->start;
        t.ent = p->ent;
        t.seg = p->seg;
        any = true;
    }
    const bool ok = !any || (trace(true) && hipStreamSynchronize(s) == hipSuccess);
    for (ColPlan* p : ps) {
        p->ok = p->ok && ok;
        if (!p->ok) col_free(p);
    }
    (void)hipGetLastError();
}

const ColPlan* col_plan(const omg_geom* gc, int64_t first, int64_t n, hipStream_t s, uint32_t min_planes) {
    omg_geom* g = const_cast<omg_geom*>(gc);
    const omg_geom_desc& d = g->d;
    // few planes leave lanes idle (min_planes); the records hold z in 15 bits and the steps left in 16
    if (d.mode != OMG_MODE_PET_SINO || d.projector_type != OMG_PROJ_SIDDON || d.tof_bins > 1 || g->force_generic ||
        d.reserved[3] != 0 || d.reserved[4] < 0 || d.n_proj < min_planes ||
        (uint64_t)d.Nx + d.Ny + d.Nz + 3 > 65535 || d.Nz > 32000 || n > 0xffffffffll ||
        (uint64_t)std::max(d.rays_xy, 1u) * std::max(d.rays_z, 1u) != 1)
        return nullptr;
    const uint64_t per = (uint64_t)d.size_x * d.size_y;
    if (!g->index_dev && ((uint64_t)n < min_planes * per || (uint64_t)n % per)) return nullptr;
    const std::lock_guard<std::mutex> lock(g->lists_mu);
    if (g->columns)
        for (ColPlan* p : g->columns->e)
            if (!g->index_dev || (p->first == first && p->n == n)) return p->ok ? p : nullptr;
    if (fixed_region_active() || (g->columns && g->columns->e.size() >= kColPlans) || is_capturing(s)) return nullptr;
    // Where an index table divides into ranges of this size, the caller goes through all of them: they are built together
    // (four plans of 576 bins take 220 us, one after the other 520 us), up to 8 at the first range, for which a caller of a
    // single range pays little, more at the second.
    std::vector<int64_t> firsts{first};
    const int64_t ranges = g->index_dev && n > 0 && first % n == 0 && d.meas_index_len % n == 0 ? d.meas_index_len / n : 0;
    const ColPlan* one = g->columns && g->columns->e.size() == 1 ? g->columns->e[0] : nullptr;
    if (one ? one->n == n && one->first % n == 0 && ranges <= (int64_t)kColPlans : !g->columns && ranges <= 8)
        for (int64_t f = 0; f < ranges * n; f += n)
            if (f != first && !(one && f == one->first)) firsts.push_back(f);
    std::vector<std::unique_ptr<ColPlan>> built;
    try {
        const RelaxedCapture relaxed;
        if (!g->columns) g->columns = new ColCache();
        g->columns->e.reserve(kColPlans);
        std::vector<ColPlan*> ps;
        for (const int64_t f : firsts) {
            built.emplace_back(new ColPlan());
            built.back()->first = f;
            built.back()->n = n;
            ps.push_back(built.back().get());
        }
        col_build(g, ps, s);
    } catch (const std::bad_alloc&) {       // no host memory for the tables: trace
        for (auto& p : built) col_free(p.get());
        return nullptr;
    }
    const ColPlan* p = built[0].get();
    for (auto& q : built) g->columns->e.push_back(q.release());
    return p->ok ? p : nullptr;
}

void col_release(omg_geom* g) {
    if (!g->columns) return;
    for (ColPlan* p : g->columns->e) {
        col_free(p);
        delete p;
    }
    for (auto& b : g->columns->buffers) {
        hipFree(b->p);
        if (b->done) hipEventDestroy(b->done);
    }
    delete g->columns;
    g->columns = nullptr;
}

// Work memory: [z-fastest image: Nx Ny pitch][records: 4 floats x bins x 64 x plane groups per pass][weights, with
// sens][the bins' peaks, of the weights too with sens][irregular LORs][state: 4].
constexpr uint64_t kColRecords = 8ull << 20;      // records per pass (128 MB): plane groups beyond take more passes

// Bins per wave: one where the wave walks (a lane's chain of columns is long, so the last waves would leave the chip
// idle: 218 us for the forward projection against 299 us with four), four for the records alone (longer runs of y:
// 73 against 84 us with two).
template <int MODE>
static void col_launch_fp(const ColView& c, const SidArgs& a, uint32_t g0, uint32_t groups, uint32_t nr, const float* Xz,
                          const float* yin, float* yout, float4* rec, float* wrec, ColPeak* peak,
                          ColPeak* wpeak, uint32_t* state, uint32_t* rest, float epps, hipStream_t s) {
    auto launch = [&](auto kern, uint32_t nb) {
        hipLaunchKernelGGL(kern, dim3((c.bins + nb - 1) / nb, groups), dim3(256), 0, s, c, a, g0 * kCL, Xz, yin, yout, rec,
                           wrec, peak, wpeak, state, rest, epps);
    };
    if (MODE == COL_BP) launch(k_col_fp<MODE, MODE == COL_BP ? 4 : 1, 1>, 16);
    else if (nr == 1) launch(k_col_fp<MODE, 1, 1>, 4);
    else if (nr == 2) launch(k_col_fp<MODE, 1, 2>, 4);
    else launch(k_col_fp<MODE, 1, 0>, 4);
}

struct ColLayout {
    uint32_t nr, pitch, all, pass;
    uint64_t per;
    size_t nimg, nrec, nw, npeak, need;
};

static ColLayout col_layout(const omg_geom* g, const ColPlan* pl, int64_t n, bool img, bool rec, bool sens) {
    const omg_geom_desc& d = g->d;
    ColLayout w;
    const bool small = (uint64_t)d.Nx * d.Ny * (d.Nz <= 63 ? 256 : 512) <= 0xffffffffull;   // a buffer's offsets
    w.nr = !small ? 0 : d.Nz <= 63 ? 1 : d.Nz <= 127 ? 2 : 0;
    w.pitch = w.nr ? 64 * w.nr : d.Nz + 2;
    w.all = (uint32_t)((n / pl->bins + kCL - 1) / kCL);
    w.per = (uint64_t)pl->bins * kCL;
    w.pass = (uint32_t)std::min<uint64_t>(w.all, std::max<uint64_t>(1, kColRecords / w.per));
    w.nimg = img ? ((size_t)d.Nx * d.Ny * w.pitch + 3) & ~(size_t)3 : 0;
    w.nrec = rec ? 4 * w.per * w.pass : 0;
    w.nw = sens ? w.per * w.pass : 0;
    w.npeak = rec ? 2 * (size_t)pl->bins * w.pass : 0;   // of one kind
    w.need = w.nimg + w.nrec + w.nw + (sens ? 2 : 1) * w.npeak + w.per * w.pass + 4;
    return w;
}

size_t col_work_floats(const omg_geom* g, const ColPlan* pl, int64_t n, bool img, bool rec, bool sens) {
    return col_layout(g, pl, n, img, rec, sens).need;
}

// A buffer for stream s, locked: the one that s used last, a new one, or one whose last call has ended. Null: none.
static ColBuffer* col_buffer(ColCache* c, hipStream_t s) {
    for (;;) {
        ColBuffer* own = nullptr;
        {
            const std::lock_guard<std::mutex> lock(c->buffers_mu);
            for (auto& b : c->buffers)
                if (b->s == s) own = b.get();
            if (!own && (c->others < kColStreams || !s)) {
                std::unique_ptr<ColBuffer> b(new ColBuffer());
                c->buffers.reserve(kColStreams + 1);
                if (s && hipEventCreateWithFlags(&b->done, hipEventDisableTiming) != hipSuccess) {
                    (void)hipGetLastError();
                    return nullptr;
                }
                b->mu.lock();
                b->s = s;
                c->others += s ? 1 : 0;
                c->buffers.push_back(std::move(b));
                return c->buffers.back().get();
            }
            for (size_t i = 0; !own && i < c->buffers.size(); i++) {
                ColBuffer* b = c->buffers[i].get();
                if (!b->s || !b->mu.try_lock()) continue;
                if (hipEventQuery(b->done) == hipSuccess) {
                    b->s = s;
                    return b;
                }
                (void)hipGetLastError();    // not ready
                b->mu.unlock();
            }
        }
        if (!own) return nullptr;
        own->mu.lock();             // another thread's call on s: the two come one after the other in any case
        if (own->s == s) return own;
        own->mu.unlock();           // given to another stream meanwhile
    }
}

ColWork::ColWork(const omg_geom* g, size_t floats, hipStream_t s, bool beside) : s_(s) {
    if (fixed_region_active() ? !scratch_fits(g, floats, s) : is_capturing(s)) return;
    if (fixed_region_active() || !beside) {
        if (scratch_reserve(const_cast<omg_geom*>(g), floats, s) == OMG_OK) p_ = scratch_ptr(g);
        else (void)hipGetLastError();
        return;
    }
    const RelaxedCapture relaxed;
    try {
        buf_ = col_buffer(g->columns, s);
    } catch (const std::bad_alloc&) {
    }
    if (!buf_) return;
    // The event also orders calls of a stream that has this handle's name only by now (hipStreamPerThread in another
    // thread, a destroyed stream's successor); on the stream itself it is nothing to wait for.
    bool ok = !buf_->done || hipStreamWaitEvent(s, buf_->done, 0) == hipSuccess;
    if (ok && buf_->floats < floats) {
        ok = (buf_->done ? hipEventSynchronize(buf_->done) : hipStreamSynchronize(s)) == hipSuccess;
        hipFree(buf_->p);
        buf_->p = nullptr;
        buf_->floats = 0;
        ok = ok && hipMalloc(reinterpret_cast<void**>(&buf_->p), floats * sizeof(float)) == hipSuccess;
        if (ok) buf_->floats = floats;
    }
    if (ok) p_ = buf_->p;
    else (void)hipGetLastError();
}

ColWork::~ColWork() {
    if (!buf_) return;
    if (p_ && buf_->done && hipEventRecord(buf_->done, s_) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipStreamSynchronize(s_);
    }
    buf_->mu.unlock();
}

// The plane groups of a call, pass after pass. yout: forward projection of img. Otherwise rhs (and sens) += the
// backprojection of the ratios (img given) or of yin (null: ones).
static int col_run(const omg_geom* g, const ColPlan* pl, int64_t first, int64_t n, const float* img, const float* yin,
                   float* yout, const float* add, float* rhs, float* sens, float epps, float* work, hipStream_t s,
                   bool timed) {
    const omg_geom_desc& d = g->d;
    const ColView c{pl->bins, (uint32_t)(n / pl->bins), pl->tw, pl->th, pl->ntx,
                    pl->off, pl->start, pl->ent, pl->seg, pl->item};
    SidArgs a = make_sid_args(g, first, n);
    a.plane_col = g->index_dev ? 0 : first;   // the z table's first plane (an index table's range holds every plane)
    a.add = add;
    const ColLayout w = col_layout(g, pl, n, img != nullptr, rhs != nullptr, sens != nullptr);
    const uint32_t nr = w.nr, pitch = w.pitch, all = w.all, pass = w.pass;
    g->column_calls.fetch_add(1, std::memory_order_relaxed);
    float* Xz = work;
    float4* rec = reinterpret_cast<float4*>(Xz + w.nimg);
    float* wrec = sens ? Xz + w.nimg + w.nrec : nullptr;
    ColPeak* peak = reinterpret_cast<ColPeak*>(Xz + w.nimg + w.nrec + w.nw);
    ColPeak* wpeak = sens ? peak + w.npeak / 2 : nullptr;
    uint32_t* rest = reinterpret_cast<uint32_t*>(peak + (sens ? 2 : 1) * (w.npeak / 2));
    uint32_t* state = rest + w.per * pass;
    const size_t lds = col_lds(c.tw, c.th, d.Nz);
    hipEvent_t stop = nullptr;
    if (timed) timing_begin(s, &stop);
    if (img)
        hipLaunchKernelGGL(k_col_zfast, dim3((d.Nx + 31) / 32, d.Ny, (pitch + 31) / 32), dim3(32, 8), 0, s, img, Xz, d.Nx,
                           d.Ny, d.Nz, pitch, nr ? 0u : 1u, state);
    OMG_CHECK_LAUNCH();
    for (uint32_t g0 = 0; g0 < all; g0 += pass) {
        const uint32_t groups = std::min(pass, all - g0);
        if (!img || g0) {
            hipLaunchKernelGGL(k_col_zero, dim3(1), dim3(256), 0, s, state, 4u);
            OMG_CHECK_LAUNCH();
        }
        if (yout) col_launch_fp<COL_FP>(c, a, g0, groups, nr, Xz, yin, yout, rec, wrec, peak, wpeak, state, rest, epps, s);
        else if (img) col_launch_fp<COL_OSEM>(c, a, g0, groups, nr, Xz, yin, yout, rec, wrec, peak, wpeak, state, rest, epps, s);
        else col_launch_fp<COL_BP>(c, a, g0, groups, nr, Xz, yin, yout, rec, wrec, peak, wpeak, state, rest, epps, s);
        OMG_CHECK_LAUNCH();
        const ColRest r{rest, img, yin, yout, rhs, sens, epps};
        if (yout) {
            hipLaunchKernelGGL(k_col_rest, dim3(1024), dim3(64), 0, s, a, state, r);
        } else {
            hipLaunchKernelGGL(k_col_bp, dim3(kColRest + pl->items, groups, sens ? 2 : 1), dim3(pl->tpb), lds, s,
                               c, a, g0 * kCL, kColRest, r, rec, wrec, peak, wpeak, state);
        }
        OMG_CHECK_LAUNCH();
    }
    if (timed) timing_end(s, stop);
    return OMG_OK;
}

int col_forward(const omg_geom* g, const ColPlan* pl, int64_t first, int64_t n, const float* img, float* y, float* work,
                hipStream_t s) {
    return col_run(g, pl, first, n, img, nullptr, y, nullptr, nullptr, nullptr, 0.f, work, s, true);
}

int col_backward(const omg_geom* g, const ColPlan* pl, int64_t first, int64_t n, const float* y, float* rhs, float* sens,
                 float* work, hipStream_t s) {
    return col_run(g, pl, first, n, nullptr, y, nullptr, nullptr, rhs, sens, 0.f, work, s, true);
}

int col_osem(const omg_geom* g, const ColPlan* pl, int64_t first, int64_t n, const float* img, const float* meas,
             const float* add, float* rhs, float* sens, float epps, float* work, hipStream_t s, bool timed) {
    return col_run(g, pl, first, n, img, meas, nullptr, add, rhs, sens, epps, work, s, timed);
}

}  // namespace omg
