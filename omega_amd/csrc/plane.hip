// plane.hip -- OSEM subset iterations of direct-plane sinograms from one 2-D system's lists.
//
// In a direct-plane sinogram (zs == zd on every plane) the walk of a LOR, its voxels and their lengths or
// weights, depends on the transaxial table only: every plane repeats the same 2-D system. The lists of that
// system are traced once per geometry handle by the projectors' own walks and kept (as the tube lists of
// projector 3 are), and a subset iteration becomes two sparse products with the subset's planes side by side:
//   k_plane_gather   the planes' slices, plane fastest: Xt[pixel][plane]
//   k_plane_fp       one lane per (LOR, plane): yhat, ratio, R[LOR][plane] = ratio * LOR weight
//   k_plane_bp       one lane per (pixel, plane): sum over the pixel's LORs in double, and the EM / OSL update
// The lanes of a wave that share a LOR (pixel) read the same list entry and one 32-byte run of Xt (R), so the
// walk's arithmetic (about 30 operations per voxel) and the scattered accumulation with its partial slices
// are gone; what is left is the list stream (8 bytes per entry and 8 planes) and L2 gathers. There are no
// atomics and the lists have a fixed order, so an iteration is deterministic. The forward sum keeps the
// walk's order and its float operations (a product and an add per voxel), the backprojection adds exact
// products in double and rounds once.
//
// Measured on a 128 x 128 x 63 image, 128 x 160 bins, 8 planes per subset, one subset step (with the sensitivity
// image / without; the kernels before it in brackets): Siddon 55 / 52 us (141 / 92: slices and accumulators in
// LDS), with 17 TOF bins 362 us (5968: one lane per LOR, every plane's bin weights evaluated twice), orthogonal
// 73 / 71 us (964 / 655: tube lists of every plane), interpolation 89 / 72 us (589 / 384). Odd 109 x 97 image,
// 8 planes of 142 x 91 bins, with prior: 50 us (478: global atomics). The lists take 50 MB (TOF: 340 MB). A
// handle's first call builds them, 0.8 ms with its allocations (interpolation 0.7, orthogonal 1.6, TOF 2.9 ms): two
// iterations of 8 subsets on a fresh handle take 1.7 ms against 2.0 ms tracing (orthogonal 2.8 against 25, interpolation
// 2.1 against 7.9, TOF 5.9 against 48 ms); one alone takes 0.1 ms more with Siddon.
#include "plane.hpp"
#include "geom.hpp"
#include "siddon_device.hpp"

#include <algorithm>
#include <cmath>
#include <memory>
#include <new>

namespace omg {

constexpr int kPB = 256;

struct PlanePlan {
    bool ok = false;
    bool interp = false;
    // Rows, pixels of a slice, pixel lists. Pixels nyx and up lie in the slices after the plane's own: the far-face
    // samples of the interpolation projector, and with Ny > Nx the Siddon rows along x, which step by Ny.
    uint32_t bins = 0, nyx = 0, npix = 0;
    uint32_t xrows = 0;                      // pixels that the forward projection reads (interpolation: nyx)
    uint64_t nent = 0;                       // entries of `ent`, padding included
    uint2* ent = nullptr;                    // row lists {pixel, length}; the padding points at pixel xrows
    uint32_t* off = nullptr;
    uint32_t* len = nullptr;                 // [row groups] padded entries per row
    uint4* samp = nullptr;                   // interpolation projector: forward samples
    uint32_t* soff = nullptr;
    uint32_t* slen = nullptr;
    uint2* cent = nullptr;                   // pixel lists {row, length}; the padding points at row `bins`
    uint32_t* cpos = nullptr;                // TOF: position in `ent` of every pixel-list entry
    uint32_t* coff = nullptr;
    uint32_t* clen = nullptr;
    float* w = nullptr;                      // [n_proj][bins] LOR weights
    float* share = nullptr;                  // TOF: [nent][pitch] bin shares
    uint32_t pitch = 0;
    int32_t* slice = nullptr;                // [n_proj]
    char* block = nullptr;                   // the allocation that holds all of these
    std::vector<int32_t> slice_host;
};

// ---- building ----------------------------------------------------------------------------------------
__global__ __launch_bounds__(kPB) void k_plane_set2(uint2* __restrict__ p, uint64_t n, uint32_t a) {
    const uint64_t i = (uint64_t)blockIdx.x * kPB + threadIdx.x;
    if (i < n) p[i] = make_uint2(a, 0u);
}
__global__ __launch_bounds__(kPB) void k_plane_set4(uint4* __restrict__ p, uint64_t n, uint32_t a) {
    const uint64_t i = (uint64_t)blockIdx.x * kPB + threadIdx.x;
    if (i < n) p[i] = make_uint4(a, 0u, 0u, 0u);
}
__global__ __launch_bounds__(kPB) void k_plane_set1(uint32_t* __restrict__ p, uint64_t n, uint32_t a) {
    const uint64_t i = (uint64_t)blockIdx.x * kPB + threadIdx.x;
    if (i < n) p[i] = a;
}

// Row lists -> unordered pixel lists: key = position in ent, value = {row, length}.
__global__ __launch_bounds__(kPB) void k_plane_transpose(uint32_t bins, const uint2* __restrict__ ent,
                                                         const float* __restrict__ lsum,
                                                         const uint32_t* __restrict__ off,
                                                         const uint32_t* __restrict__ cnt,
                                                         const uint32_t* __restrict__ coff,
                                                         uint32_t* __restrict__ cursor, uint32_t* __restrict__ key,
                                                         uint2* __restrict__ val) {
    const uint32_t row = blockIdx.x * (kPB / 64) + (threadIdx.x >> 6);
    if (row >= bins) return;
    for (uint32_t k = threadIdx.x & 63; k < cnt[row]; k += 64) {
        const uint32_t pos = off[row / kLI] + k * kLI + row % kLI;
        const uint2 e = ent[pos];
        const uint32_t c = atomicAdd(cursor + e.x, 1u);
        const size_t o = (size_t)coff[e.x / kLI] + (size_t)c * kLI + e.x % kLI;
        key[o] = pos;
        val[o] = make_uint2(row, lsum ? __float_as_uint(lsum[pos]) : e.y);
    }
}

// Orders each pixel's list by key (rank sort, one wave per pixel): the lists do not depend on the order in
// which k_plane_transpose's atomics retired. A lane holds one key and counts the smaller ones, 64 others at a time from
// the wave's registers (128 x 128 pixels, 128 x 160 LORs: 99 us; 328 us with every key read from memory).
__global__ __launch_bounds__(kPB) void k_plane_sort(uint32_t npix, const uint32_t* __restrict__ coff,
                                                    const uint32_t* __restrict__ count,
                                                    const uint32_t* __restrict__ key, const uint2* __restrict__ val,
                                                    uint2* __restrict__ cent, uint32_t* __restrict__ cpos) {
    const uint32_t pix = blockIdx.x * (kPB / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (pix >= npix) return;
    const uint32_t lane = threadIdx.x & 63;
    const size_t o = (size_t)coff[pix / kLI] + pix % kLI;
    const uint32_t n = count[pix];
    for (uint32_t i0 = 0; i0 < n; i0 += 64) {
        const uint32_t i = i0 + lane, ki = i < n ? key[o + (size_t)i * kLI] : 0u;
        uint32_t r = 0;
        for (uint32_t j0 = 0; j0 < n; j0 += 64) {
            // behind the list: larger than every key (a position below 2^32 - 16)
            const uint32_t kj = j0 + lane < n ? key[o + (size_t)(j0 + lane) * kLI] : ~0u;
#pragma unroll
            for (int t = 0; t < 64; t++) r += (uint32_t)__builtin_amdgcn_readlane((int)kj, t) < ki ? 1u : 0u;
        }
        if (i < n) {
            cent[o + (size_t)r * kLI] = val[o + (size_t)i * kLI];
            if (cpos) cpos[o + (size_t)r * kLI] = ki;
        }
    }
}

// ---- running -----------------------------------------------------------------------------------------
// (Every argument of k_plane_bp within 256 bytes, and what k_plane_fp waits for first together: a further line of them
// costs 0.1 us.)
struct PlaneRun {
    uint32_t bins, xrows, nyx, npix;
    uint32_t planes;                         // of this call
    uint32_t nx, nz;                         // image row length, slices
    uint32_t nent;
    const uint32_t *off, *len, *soff, *slen, *coff, *clen;
    const uint2 *ent, *cent;
    const uint4* samp;
    const uint32_t* cpos;
    const float* w;                          // of the call's first plane
    const int32_t* slice;                    // of the call's first plane
    const float* share;
    // interpolation projector: the planes' z table and the grid's z axis (others: null)
    const float* z;
    float bz, sz;
};

// Xt[chunk][pixel][PL]: the planes' slices side by side (and what follows them, up to xrows), and a zero row behind
// them for the padding entries. GATHER_BEHIND: xrows reach past the slice, to the image's end at most.
// GATHER_INTERP: the blend of the two slices that the plane's samples lie between.
enum { GATHER_SLICE = 0, GATHER_INTERP = 1, GATHER_BEHIND = 2 };
template <int PL, int MODE>
__global__ __launch_bounds__(kPB) void k_plane_gather(PlaneRun a, const float* __restrict__ x, float* __restrict__ Xt) {
    const uint32_t pix = blockIdx.x * kPB + threadIdx.x;
    if (pix > a.xrows) return;
    float v[PL];
#pragma unroll
    for (int p = 0; p < PL; p++) {
        const uint32_t plane = blockIdx.y * PL + p;
        v[p] = 0.f;
        if (plane < a.planes && pix < a.xrows) {
            const int32_t tk = a.slice[plane];
            if (MODE == GATHER_INTERP) {
                if (tk >= 0) {
                    const float u = ((0.f + a.z[2 * plane]) - a.bz) * a.sz * (float)a.nz - 0.5f;
                    const float f = floorf(u), c = u - f;
                    const uint32_t z0 = (uint32_t)fminf(fmaxf(f, 0.f), (float)(a.nz - 1));
                    const uint32_t z1 = (uint32_t)fminf(fmaxf(f + 1.f, 0.f), (float)(a.nz - 1));
                    v[p] = (1.f - c) * x[(size_t)z0 * a.nyx + pix] + c * x[(size_t)z1 * a.nyx + pix];
                }
            } else if (tk >= 0) {
                const size_t n = (size_t)tk * a.nyx + pix;
                if (MODE != GATHER_BEHIND || n < (size_t)a.nz * a.nyx) v[p] = x[n];
            }
        }
    }
    float* o = Xt + ((size_t)blockIdx.y * (a.xrows + 1) + pix) * PL;
#pragma unroll
    for (int p = 0; p < PL; p++) o[p] = v[p];
}

// Forward projection, ratio and R = ratio * weight (W = weight with SENS), one lane per (LOR, plane); row
// `bins` of R and W is zero (the pixel lists' padding).
template <int PL, bool INTERP, bool SENS>
__global__ __launch_bounds__(kPB) void k_plane_fp(PlaneRun a, const float* __restrict__ Xt,
                                                  const float* __restrict__ meas, const float* __restrict__ add,
                                                  float* __restrict__ R, float* __restrict__ W, float epps) {
    const uint32_t t = blockIdx.x * kPB + threadIdx.x;
    const uint32_t row = t / PL, p = t % PL, plane = blockIdx.y * PL + p;
    if (row > a.bins) return;
    const size_t o = ((size_t)blockIdx.y * (a.bins + 1) + row) * PL + p;
    if (row == a.bins || plane >= a.planes) {
        R[o] = 0.f;
        if (SENS) W[o] = 0.f;
        return;
    }
    const float* X = Xt + (size_t)blockIdx.y * (a.xrows + 1) * PL + p;
    const uint32_t g = row / kLI;
    float ax = 0.f;
    if (INTERP) {
        const uint4* e = a.samp + a.soff[g] + row % kLI;
        const uint32_t n = a.slen[g];
        for (uint32_t k = 0; k < n; k += 4) {
            uint4 q[4];
            float v[4][4];
#pragma unroll
            for (int j = 0; j < 4; j++) q[j] = e[(k + j) * kLI];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t i = q[j].x & 0x3fffffffu, fx = (q[j].x >> 30) & 1u, fy = (q[j].x >> 31) ? a.nx : 0u;
                v[j][0] = X[(size_t)i * PL];
                v[j][1] = X[(size_t)(i + fx) * PL];
                v[j][2] = X[(size_t)(i + fy) * PL];
                v[j][3] = X[(size_t)(i + fy + fx) * PL];
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float fa = __uint_as_float(q[j].y), fb = __uint_as_float(q[j].z);
                const float c0 = (1.f - fa) * v[j][0] + fa * v[j][1];
                const float c1 = (1.f - fa) * v[j][2] + fa * v[j][3];
                ax += __uint_as_float(q[j].w) * ((1.f - fb) * c0 + fb * c1);
            }
        }
    } else {
        const uint2* e = a.ent + a.off[g] + row % kLI;
        const uint32_t n = a.len[g];
        uint2 q[kLUnroll];
        float v[kLUnroll];
#pragma unroll
        for (uint32_t j = 0; j < kLUnroll; j++) q[j] = n ? e[j * kLI] : uint2{0u, 0u};
        for (uint32_t k = 0; k < n; k += kLUnroll) {
            uint2 qn[kLUnroll];
            const uint32_t kn = k + kLUnroll < n ? k + kLUnroll : k;   // the next entries load behind the voxels
#pragma unroll
            for (uint32_t j = 0; j < kLUnroll; j++) v[j] = X[(size_t)q[j].x * PL];
#pragma unroll
            for (uint32_t j = 0; j < kLUnroll; j++) qn[j] = e[(kn + j) * kLI];
#pragma unroll
            for (uint32_t j = 0; j < kLUnroll; j++) ax += __uint_as_float(q[j].y) * v[j];
#pragma unroll
            for (uint32_t j = 0; j < kLUnroll; j++) q[j] = qn[j];
        }
    }
    const bool in = a.slice[plane] >= 0;
    const size_t m = (size_t)plane * a.bins + row;
    const float w = in ? a.w[m] : 0.f;
    float d = ax * w + epps;
    if (add) d += add[m];
    float r = meas[m] / d;
    if (isnan(r) || isinf(r)) r = epps;
    R[o] = in ? r * w : 0.f;
    if (SENS) W[o] = w;
}

// Time of flight: per LOR the bins' forward sums (one lane per (LOR, plane), NQ * 4 bins in registers), the
// ratios, and per list entry T[entry][plane] = length * sum_b share_b ratio_b weight for the pixel lists.
template <int PL, int NQ, bool SENS>
__global__ __launch_bounds__(kPB) void k_plane_tof(PlaneRun a, uint32_t chunk, uint32_t nb, const float* __restrict__ Xt,
                                                   const float* __restrict__ meas, const float* __restrict__ add,
                                                   float* __restrict__ T, float* __restrict__ W, float epps) {
    const uint32_t t = blockIdx.x * kPB + threadIdx.x;
    const uint32_t row = t / PL, p = t % PL, plane = chunk * PL + p;
    if (row > a.bins) return;
    if (row == a.bins) {                     // the pixel lists' padding
        T[(size_t)a.nent * PL + p] = 0.f;
        if (SENS) W[(size_t)row * PL + p] = 0.f;
        return;
    }
    const bool in = plane < a.planes && a.slice[plane] >= 0;
    const float* X = Xt + (size_t)chunk * (a.xrows + 1) * PL + p;
    const uint32_t g = row / kLI, base = a.off[g] + row % kLI, n = a.len[g];
    const float4* sh = reinterpret_cast<const float4*>(a.share) + (size_t)base * NQ;
    float acc[4 * NQ];
#pragma unroll
    for (int b = 0; b < 4 * NQ; b++) acc[b] = 0.f;
    for (uint32_t k = 0; k < n; k += 2) {
        float v[2];
        float4 s[2][NQ];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint2 q = a.ent[base + (k + j) * kLI];
            v[j] = __uint_as_float(q.y) * X[(size_t)q.x * PL];
#pragma unroll
            for (int c = 0; c < NQ; c++) s[j][c] = sh[(size_t)(k + j) * kLI * NQ + c];
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
#pragma unroll
            for (int c = 0; c < NQ; c++) {
                acc[4 * c] += v[j] * s[j][c].x;
                acc[4 * c + 1] += v[j] * s[j][c].y;
                acc[4 * c + 2] += v[j] * s[j][c].z;
                acc[4 * c + 3] += v[j] * s[j][c].w;
            }
        }
    }
    const size_t nlor = (size_t)a.planes * a.bins, m = (size_t)plane * a.bins + row;
    const float w = in ? a.w[m] : 0.f;
    const float ad = in && add ? add[m] : 0.f;
#pragma unroll
    for (int b = 0; b < 4 * NQ; b++) {
        float r = 0.f;
        if (in && (uint32_t)b < nb) {
            float d = acc[b] * w + epps;
            if (add) d += ad;
            r = meas[m + (size_t)b * nlor] / d;
            if (isnan(r) || isinf(r)) r = epps;
        }
        acc[b] = r * w;
    }
    if (SENS) W[(size_t)row * PL + p] = w;
    for (uint32_t k = 0; k < n; k += 2) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            float s = 0.f;
#pragma unroll
            for (int c = 0; c < NQ; c++) {
                const float4 q = sh[(size_t)(k + j) * kLI * NQ + c];
                s += q.x * acc[4 * c];
                s += q.y * acc[4 * c + 1];
                s += q.z * acc[4 * c + 2];
                s += q.w * acc[4 * c + 3];
            }
            const uint32_t pos = base + (k + j) * kLI;
            T[(size_t)pos * PL + p] = __uint_as_float(a.ent[pos].y) * s;
        }
    }
}

// Sums of one pixel list: rhs of length * R (or of T, TOF), sens of length * W. The entries of the next batch load
// while the values of this one arrive (they are the chain's two links): 28 -> 23 us without sens, TOF 98 -> 53 us.
template <int PL, bool TOF, bool SENS>
__device__ __forceinline__ void plane_sums(const PlaneRun& a, uint32_t pix, const float* __restrict__ R,
                                           const float* __restrict__ W, double& rhs, double& sens) {
    const uint32_t g = pix / kLI, n = a.clen[g];
    const size_t o = (size_t)a.coff[g] + pix % kLI;
    const uint2* e = a.cent + o;
    const uint32_t* ep = TOF ? a.cpos + o : nullptr;
    uint2 q[kLUnroll];
    uint32_t at[kLUnroll];
    auto fetch = [&](uint32_t k, uint2 (&qq)[kLUnroll], uint32_t (&aa)[kLUnroll]) {
#pragma unroll
        for (uint32_t j = 0; j < kLUnroll; j++) {
            if (!TOF || SENS) qq[j] = e[(k + j) * kLI];
            if (TOF) aa[j] = ep[(k + j) * kLI];
        }
    };
    if (n) fetch(0, q, at);
    for (uint32_t k = 0; k < n; k += kLUnroll) {
        uint2 qn[kLUnroll];
        uint32_t an[kLUnroll];
        float v[kLUnroll], u[kLUnroll];
#pragma unroll
        for (uint32_t j = 0; j < kLUnroll; j++) {
            v[j] = R[(size_t)(TOF ? at[j] : q[j].x) * PL];
            if (SENS) u[j] = W[(size_t)q[j].x * PL];
        }
        fetch(k + kLUnroll < n ? k + kLUnroll : k, qn, an);   // the next entries load behind the values
#pragma unroll
        for (uint32_t j = 0; j < kLUnroll; j++) {
            if (TOF) rhs += (double)v[j];
            else rhs = __builtin_fma((double)__uint_as_float(q[j].y), (double)v[j], rhs);
            if (SENS) sens = __builtin_fma((double)__uint_as_float(q[j].y), (double)u[j], sens);
        }
#pragma unroll
        for (uint32_t j = 0; j < kLUnroll; j++) {
            if (!TOF || SENS) q[j] = qn[j];
            if (TOF) at[j] = an[j];
        }
    }
}

__device__ __forceinline__ float plane_update(float xo, float S, float rhs, const float* dU, size_t n, float epps,
                                              int pos) {
    float v = dU ? xo / (S + dU[n]) * rhs : xo / S * (rhs + epps);
    if (pos && v < epps) v = epps;
    return v;
}

// Plane of the call whose slice is z, or -1 (a scan of the call's planes).
__device__ __forceinline__ int32_t plane_at(const PlaneRun& a, int32_t z) {
    for (uint32_t q = 0; q < a.planes; q++)
        if (a.slice[q] == z) return (int32_t)q;
    return -1;
}

// The lists of pixel `pix` of slice z from the planes in the slices before it (pixels nyx and up).
template <int PL, bool SENS>
__device__ __forceinline__ void plane_carried(const PlaneRun& a, uint32_t pix, int32_t z, const float* __restrict__ R,
                                              const float* __restrict__ W, double& rhs, double& sens) {
    const size_t rows = (size_t)(a.bins + 1) * PL;
    for (uint32_t q = pix + a.nyx; q < a.npix && z > 0; q += a.nyx) {
        const int32_t p = plane_at(a, --z);
        if (p >= 0) plane_sums<PL, false, SENS>(a, q, R + (p / PL) * rows + p % PL, W + (p / PL) * rows + p % PL, rhs, sens);
    }
}

// Backprojection and update. The first `bpb` blocks hold the voxels of the call's planes [chunk0, chunk0 +
// chunks) of PL planes, one lane per (pixel, plane); with OTHERS the blocks behind them update the image's
// other slices (rhs = 0), 4 * 256 voxels of one slice each. CARRY: pixel lists nyx and up exist, whose voxels lie in
// the slices after their plane's own.
template <int PL, bool TOF, bool SENS, bool CARRY>
__global__ __launch_bounds__(kPB) void k_plane_bp(PlaneRun a, uint32_t bpb, uint32_t per_chunk, uint32_t chunk0,
                                                  const float* __restrict__ R, const float* __restrict__ W,
                                                  float* __restrict__ x, float* __restrict__ S,
                                                  const float* __restrict__ dU, float epps, int pos) {
    if (blockIdx.x < bpb) {
        const uint32_t ch = blockIdx.x / per_chunk;
        const uint32_t t = (blockIdx.x - ch * per_chunk) * kPB + threadIdx.x;
        const uint32_t pix = t / PL, p = t % PL, plane = (chunk0 + ch) * PL + p;
        if (pix >= a.nyx || plane >= a.planes) return;
        const int32_t tk = a.slice[plane];
        if (tk < 0) return;
        double rhs = 0.0, sens = 0.0;
        const size_t rows = (size_t)(a.bins + 1) * PL;
        plane_sums<PL, TOF, SENS>(a, pix, R + (TOF ? 0 : ch * rows) + p, W + (TOF ? 0 : ch * rows) + p, rhs, sens);
        if (CARRY) {
            if (a.z && tk == 0 && pix == 0) { rhs = 0.0; sens = 0.0; }   // the interpolation reference skips voxel 0
            plane_carried<PL, SENS>(a, pix, tk, R, W, rhs, sens);
        }
        const size_t n = (size_t)tk * a.nyx + pix;
        float s;
        if (SENS) {
            s = (float)sens;
            if (s < epps) s = epps;
            S[n] = s;
        } else {
            s = S[n];
        }
        x[n] = plane_update(x[n], s, (float)rhs, dU, n, epps, pos);
        return;
    }
    const uint32_t b = blockIdx.x - bpb, per = (a.nyx + 4 * kPB - 1) / (4 * kPB);
    const int32_t z = (int32_t)(b / per);
    if (plane_at(a, z) >= 0) return;
    for (uint32_t j = 0; j < 4; j++) {
        const uint32_t pix = (b % per) * 4 * kPB + j * kPB + threadIdx.x;
        if (pix >= a.nyx) return;
        double rhs = 0.0, sens = 0.0;
        if (CARRY) plane_carried<PL, SENS>(a, pix, z, R, W, rhs, sens);
        const size_t n = (size_t)z * a.nyx + pix;
        float s;
        if (SENS) {
            s = (float)sens;
            if (s < epps) s = epps;
            S[n] = s;
        } else {
            s = S[n];
        }
        x[n] = plane_update(x[n], s, (float)rhs, dU, n, epps, pos);
    }
}

// ---- plan: host ----------------------------------------------------------------------------------------
static void plan_free(PlanePlan* p) {
    hipFree(p->block);
    const std::vector<int32_t> keep = p->slice_host;
    *p = PlanePlan();
    p->slice_host = keep;
}

template <typename T>
static bool dev_alloc(T** p, uint64_t n) {
    return hipMalloc(reinterpret_cast<void**>(p), (size_t)std::max<uint64_t>(n, 1) * sizeof(T)) == hipSuccess;
}

// Offsets of padded, interleaved lists with the given entry counts; false when they pass 2^32 entries.
static bool list_layout(const std::vector<uint32_t>& cnt, std::vector<uint32_t>& off, std::vector<uint32_t>& len,
                        uint64_t* total) {
    const size_t groups = (cnt.size() + kLI - 1) / kLI;
    off.assign(groups, 0);
    len.assign(groups, 0);
    uint64_t t = 0;
    for (size_t g = 0; g < groups; g++) {
        uint32_t m = 0;
        for (size_t r = g * kLI; r < std::min(cnt.size(), (g + 1) * kLI); r++) m = std::max(m, cnt[r]);
        m = (m + kLUnroll - 1) / kLUnroll * kLUnroll;
        off[g] = (uint32_t)t;
        len[g] = m;
        t += (uint64_t)m * kLI;
        if (t >= 0xFFFFFFF0ull) return false;
    }
    *total = t;
    return true;
}

// Work memory of an iteration in floats: gathered slices; ratios (TOF: per entry, a chunk of planes at a time); weights.
struct PlaneWork { size_t xt, r, w; };
static PlaneWork plane_work(const PlanePlan* p, uint32_t chunks, uint32_t pl, bool tof) {
    const size_t rr = (size_t)(tof ? 1 : chunks) * (p->bins + 1) * pl;
    return PlaneWork{(size_t)chunks * (p->xrows + 1) * pl, tof ? (size_t)(p->nent + 1) * pl : rr, rr};
}

// Device memory that the lists may take, with the work memory of an iteration on every plane (omg_geom_desc.reserved[4],
// as the tube lists).
static uint64_t plan_budget(const omg_geom* g) {
    const int32_t r = g->d.reserved[4];
    if (r < 0) return 0;
    return (uint64_t)(r == 0 ? 16384 : r) << 20;
}

static bool plan_applies(const omg_geom* g) {
    const omg_geom_desc& d = g->d;
    if (d.mode != OMG_MODE_PET_SINO || g->force_generic || g->index_dev || plan_budget(g) == 0) return false;
    if ((uint64_t)std::max(d.rays_xy, 1u) * std::max(d.rays_z, 1u) != 1) return false;
    const bool tof = d.tof_bins > 1;
    if (d.projector_type == OMG_PROJ_SIDDON) {
        if (tof && d.tof_bins > 32) return false;      // the bins of a LOR are held in registers
    } else if (d.projector_type == OMG_PROJ_ORTH) {
        uint32_t plane = 0;
        if (!orth_plane_ok(g, &plane)) return false;
    } else if (d.projector_type == OMG_PROJ_INTERP) {
        if (tof) return false;
    } else {
        return false;
    }
    if ((uint64_t)d.Nx * d.Ny + d.Nx + 1 >= (1u << 30)) return false;
    for (uint32_t p = 0; p < d.n_proj; p++)
        if (!(g->z_host[2 * (size_t)p] == g->z_host[2 * (size_t)p + 1])) return false;
    return true;
}

// Lists per pixel longer than this keep the tracing kernels (the rank sort is quadratic in them).
constexpr uint32_t kMaxPixelList = 16384;

// Fills p; false (with everything freed) when the lists do not apply, do not fit or memory is short.
static bool plan_build(const omg_geom* g, PlanePlan* p, hipStream_t s) {
    const omg_geom_desc& d = g->d;
    const bool interp = d.projector_type == OMG_PROJ_INTERP, tof = d.tof_bins > 1;
    const bool orth = d.projector_type == OMG_PROJ_ORTH;
    const uint32_t bins = d.size_x * d.size_y;
    p->interp = interp;
    p->bins = bins;
    p->nyx = d.Nx * d.Ny;
    p->npix = p->nyx + (interp ? d.Nx + 1 : 0);
    // a row along x starts at its y times Ny (siddon_setup): with Ny > Nx it can end past the slice. The TOF kernels
    // hold one chunk of planes at a time and take no such rows, nor are lists many times the slice kept for them.
    if (!interp && !orth && !tof && d.Ny > d.Nx && d.Ny <= 16 * d.Nx && d.Ny < 32768)
        p->npix = std::max(p->nyx, (d.Ny - 1) * d.Ny + d.Nx);
    if (interp) interp_plane_slices(g, p->slice_host);
    else siddon_plane_slices(g, p->slice_host);
    // The lowest slice: voxels that a walk leaves out behind the image's end are out for every other plane too, so the
    // lists hold (or refuse, plane_put) all that any plane visits. The orthogonal projector, whose images are square and
    // whose tubes stay in their slice, has its own choice.
    uint32_t plane = d.n_proj;
    for (uint32_t q = 0; q < d.n_proj; q++)
        if (p->slice_host[q] >= 0 && (plane == d.n_proj || p->slice_host[q] < p->slice_host[plane])) plane = q;
    if (orth && !orth_plane_ok(g, &plane)) return false;
    if (plane == d.n_proj || bins == 0) return false;
    const uint64_t budget = plan_budget(g);

    PlaneFill f = {};
    f.npix = p->npix;
    f.slice_base = (uint32_t)p->slice_host[plane] * p->nyx;
    // counts, cleared and read back together: [pixels][bad][rows][samples of the rows]
    const uint64_t npix0 = p->npix, ncount = npix0 + 1 + (interp ? 2 : 1) * (uint64_t)bins;
    uint32_t *counts = nullptr, *key = nullptr;
    uint2* val = nullptr;
    float* lsum = nullptr;
    bool ok = dev_alloc(&counts, ncount);
    uint32_t *pixcnt = counts, *cnt = counts + npix0 + 1, *scnt = cnt + bins;
    auto trace = [&](const PlaneFill& q) {
        return (interp ? interp_plane_trace(g, plane, q, s) : orth ? orth_plane_trace(g, plane, q, s)
                : tof ? tof_plane_trace(g, plane, q, s) : siddon_plane_trace(g, plane, q, s)) == OMG_OK;
    };
    auto fill1 = [&](uint32_t* q, uint64_t n, uint32_t v) {
        hipLaunchKernelGGL(k_plane_set1, dim3(grid_for((int64_t)n, kPB)), dim3(kPB), 0, s, q, n, v);
    };
    std::vector<uint32_t> host(ncount), hc, hp, hs, off, len, soff, slen, coff, clen, tables;
    uint64_t nc = 0, ns = 0;
    if (ok) {
        fill1(pixcnt, npix0 + 1, 0u);
        f.cnt = cnt; f.pixcnt = pixcnt; f.scnt = scnt; f.bad = reinterpret_cast<int32_t*>(pixcnt + npix0);
        ok = trace(f) && hipMemcpyAsync(host.data(), counts, ncount * 4, hipMemcpyDeviceToHost, s) == hipSuccess &&
             hipStreamSynchronize(s) == hipSuccess && !host[npix0];
    }
    const auto rows = host.begin() + (ptrdiff_t)npix0 + 1;
    hp.assign(host.begin(), host.begin() + (ptrdiff_t)npix0);
    hc.assign(rows, rows + bins);
    if (interp) hs.assign(rows + bins, host.end());
    if (!interp) {       // only as far as the lists go
        while (p->npix > p->nyx && hp[p->npix - 1] == 0) p->npix--;
        hp.resize(p->npix);
    }
    p->xrows = interp ? p->nyx : p->npix;
    ok = ok && *std::max_element(hp.begin(), hp.end()) <= kMaxPixelList && list_layout(hc, off, len, &p->nent) &&
         list_layout(hp, coff, clen, &nc) && (!interp || list_layout(hs, soff, slen, &ns));
    p->pitch = tof ? (d.tof_bins + 3) / 4 * 4 : 0;
    if (p->pitch == 4) p->pitch = 8;
    if (p->pitch == 12) p->pitch = 16;
    if (p->pitch == 28) p->pitch = 32;
    if (ok) {
        const PlaneWork w = plane_work(p, (d.n_proj + 7) / 8, 8, tof);
        ok = p->nent * (8 + 4 + 4ull * p->pitch) + nc * (8 + 12 + 4) + ns * 16 + 4ull * bins * d.n_proj +
                 4ull * (w.xt + w.r + w.w) <= budget;
    }
    char* temp = nullptr;
    if (ok) {                // one allocation for the lists, one for what only their building needs
        for (const auto* t : {&off, &len, &soff, &slen, &coff, &clen}) tables.insert(tables.end(), t->begin(), t->end());
        tables.insert(tables.end(), p->slice_host.begin(), p->slice_host.end());
        size_t keep = 0, work = 0;
        auto take = [](size_t& at, uint64_t bytes) {
            const size_t unit = bytes >= (1u << 20) ? 2u << 20 : 256u, o = (at + unit - 1) & ~(unit - 1);
            at = o + (size_t)bytes;
            return o;
        };
        const size_t at_ent = take(interp ? work : keep, p->nent * 8);
        const size_t at_tables = take(keep, tables.size() * 4), at_cent = take(keep, nc * 8);
        const size_t at_w = take(keep, 4ull * bins * d.n_proj), at_samp = take(keep, ns * 16);
        const size_t at_share = take(keep, tof ? 4 * p->nent * p->pitch : 0), at_cpos = take(keep, tof ? 4 * nc : 0);
        // the interpolation projector's row lists serve the transposition only
        const size_t at_key = take(work, nc * 4), at_val = take(work, nc * 8), at_lsum = take(work, tof ? 4 * p->nent : 0);
        ok = dev_alloc(&p->block, keep) && dev_alloc(&temp, work) &&
             hipMemcpyAsync(p->block + at_tables, tables.data(), tables.size() * 4, hipMemcpyHostToDevice, s) == hipSuccess;
        uint32_t* t = reinterpret_cast<uint32_t*>(p->block + at_tables);
        p->off = t; p->len = t += off.size(); p->soff = t += len.size(); p->slen = t += soff.size();
        p->coff = t += slen.size(); p->clen = t += coff.size();
        p->slice = reinterpret_cast<int32_t*>(t += clen.size());
        p->cent = reinterpret_cast<uint2*>(p->block + at_cent);
        p->w = reinterpret_cast<float*>(p->block + at_w);
        if (interp) p->samp = reinterpret_cast<uint4*>(p->block + at_samp);
        if (tof) p->share = reinterpret_cast<float*>(p->block + at_share);
        if (tof) p->cpos = reinterpret_cast<uint32_t*>(p->block + at_cpos);
        if (tof) lsum = reinterpret_cast<float*>(temp + at_lsum);
        p->ent = reinterpret_cast<uint2*>((interp ? temp : p->block) + at_ent);
        key = reinterpret_cast<uint32_t*>(temp + at_key);
        val = reinterpret_cast<uint2*>(temp + at_val);
    }
    if (ok) {
        hipLaunchKernelGGL(k_plane_set2, dim3(grid_for((int64_t)p->nent, kPB)), dim3(kPB), 0, s, p->ent, p->nent, p->xrows);
        hipLaunchKernelGGL(k_plane_set2, dim3(grid_for((int64_t)nc, kPB)), dim3(kPB), 0, s, p->cent, nc, bins);
        if (tof) fill1(p->cpos, nc, (uint32_t)p->nent);
        if (interp)
            hipLaunchKernelGGL(k_plane_set4, dim3(grid_for((int64_t)ns, kPB)), dim3(kPB), 0, s, p->samp, ns, p->nyx);
        f.off = p->off; f.ent = p->ent; f.soff = p->soff; f.samp = p->samp;
        ok = trace(f);
        if (ok && tof) {
            // shares of the padding entries are read (times a zero voxel): they must be numbers
            fill1(reinterpret_cast<uint32_t*>(p->share), p->nent * p->pitch, 0u);
            ok = tof_plane_shares(g, plane, f, p->pitch, p->share, lsum, s) == OMG_OK;
        }
        ok = ok && (interp ? interp_plane_weights(g, p->w, s) : orth ? orth_plane_weights(g, p->w, s)
                           : siddon_plane_weights(g, p->w, s)) == OMG_OK;
    }
    if (ok) {
        // the second pass over the row counts (the same walk) left cnt as it was
        fill1(pixcnt, p->npix, 0u);
        hipLaunchKernelGGL(k_plane_transpose, dim3((bins + kPB / 64 - 1) / (kPB / 64)), dim3(kPB), 0, s, bins, p->ent,
                           lsum, p->off, cnt, p->coff, pixcnt, key, val);
        hipLaunchKernelGGL(k_plane_sort, dim3((p->npix + kPB / 64 - 1) / (kPB / 64)), dim3(kPB), 0, s, p->npix, p->coff,
                           pixcnt, key, val, p->cent, p->cpos);
        ok = hipGetLastError() == hipSuccess && hipStreamSynchronize(s) == hipSuccess;
    }
    if (!ok) (void)hipStreamSynchronize(s);      // copies from this function's tables
    hipFree(counts); hipFree(temp);
    if (interp) p->ent = nullptr;
    if (!ok) {
        (void)hipGetLastError();
        plan_free(p);
    }
    return ok;
}

const PlanePlan* plane_plan(const omg_geom* gc, hipStream_t s) {
    omg_geom* g = const_cast<omg_geom*>(gc);
    const std::lock_guard<std::mutex> lock(g->lists_mu);
    if (g->plane) return g->plane->ok ? g->plane : nullptr;
    std::unique_ptr<PlanePlan> p;
    try {
        if (!plan_applies(g) || fixed_region_active() || is_capturing(s)) return nullptr;
        const RelaxedCapture relaxed;
        p.reset(new PlanePlan());
        p->ok = plan_build(g, p.get(), s);
        g->plane = p.release();
    } catch (const std::bad_alloc&) {       // no host memory for the tables: trace
        if (p) plan_free(p.get());
        return nullptr;
    }
    return g->plane->ok ? g->plane : nullptr;
}

void plane_release(omg_geom* g) {
    if (!g->plane) return;
    plan_free(g->plane);
    delete g->plane;
    g->plane = nullptr;
}

// ---- subset iteration ------------------------------------------------------------------------------------
template <int PL>
static int run_planes(omg_geom* g, const PlanePlan* pl, const PlaneRun& a, const SidArgs& sa, float* x,
                      const float* meas, const float* add, float* S, bool sens, float epps, const float* dU, int pos,
                      hipStream_t s, bool* done) {
    const uint32_t chunks = (a.planes + PL - 1) / PL;
    const bool tof = pl->share != nullptr;
    const PlaneWork w = plane_work(pl, chunks, PL, tof);
    const size_t need = w.xt + w.r + (sens ? w.w : 0);
    *done = false;
    if (!scratch_fits(g, need, s)) return OMG_OK;
    if (scratch_reserve(g, need, s) != OMG_OK) {   // device memory short: the tracing kernels need less
        (void)hipGetLastError();
        return OMG_OK;
    }
    int rc = OMG_OK;
    *done = true;
    g->plane_calls.fetch_add(1, std::memory_order_relaxed);
    float* Xt = scratch_ptr(g);
    float* R = Xt + w.xt;
    float* W = R + w.r;
    hipEvent_t stop;
    timing_begin(s, &stop);
    const dim3 gg(grid_for((int64_t)a.xrows + 1, kPB), chunks);
    hipLaunchKernelGGL((pl->interp ? k_plane_gather<PL, GATHER_INTERP> : a.xrows > a.nyx ? k_plane_gather<PL, GATHER_BEHIND>
                        : k_plane_gather<PL, GATHER_SLICE>), gg, dim3(kPB), 0, s, a, x, Xt);
    OMG_CHECK_LAUNCH();
    const uint32_t per_chunk = grid_for((int64_t)a.nyx * PL, kPB);
    const uint32_t others = (a.nyx + 4 * kPB - 1) / (4 * kPB) * a.nz;
    const unsigned fpb = grid_for((int64_t)(a.bins + 1) * PL, kPB);
    if (tof) {
        for (uint32_t c = 0; c < chunks; c++) {
            auto launch = [&](auto kern) {
                hipLaunchKernelGGL(kern, dim3(fpb), dim3(kPB), 0, s, a, c, sa.tof_bins, Xt, meas, add, R, W, epps);
            };
            switch (pl->pitch / 4) {
                case 2: sens ? launch(k_plane_tof<PL, 2, true>) : launch(k_plane_tof<PL, 2, false>); break;
                case 4: sens ? launch(k_plane_tof<PL, 4, true>) : launch(k_plane_tof<PL, 4, false>); break;
                case 5: sens ? launch(k_plane_tof<PL, 5, true>) : launch(k_plane_tof<PL, 5, false>); break;
                case 6: sens ? launch(k_plane_tof<PL, 6, true>) : launch(k_plane_tof<PL, 6, false>); break;
                default: sens ? launch(k_plane_tof<PL, 8, true>) : launch(k_plane_tof<PL, 8, false>); break;
            }
            OMG_CHECK_LAUNCH();
            const unsigned blocks = per_chunk + (c == 0 ? others : 0);
            if (sens)
                hipLaunchKernelGGL((k_plane_bp<PL, true, true, false>), dim3(blocks), dim3(kPB), 0, s, a, per_chunk,
                                   per_chunk, c, R, W, x, S, dU, epps, pos);
            else
                hipLaunchKernelGGL((k_plane_bp<PL, true, false, false>), dim3(blocks), dim3(kPB), 0, s, a, per_chunk,
                                   per_chunk, c, R, W, x, S, dU, epps, pos);
            OMG_CHECK_LAUNCH();
        }
        timing_end(s, stop);
        return OMG_OK;
    }
    const dim3 fg(fpb, chunks), bg(per_chunk * chunks + others);
    const bool carry = a.npix > a.nyx;
    auto step = [&](auto fp, auto bp) {
        hipLaunchKernelGGL(fp, fg, dim3(kPB), 0, s, a, Xt, meas, add, R, W, epps);
        OMG_CHECK_LAUNCH();
        hipLaunchKernelGGL(bp, bg, dim3(kPB), 0, s, a, per_chunk * chunks, per_chunk, 0u, R, W, x, S, dU, epps, pos);
        OMG_CHECK_LAUNCH();
        return (int)OMG_OK;
    };
    if (pl->interp && sens) rc = step(k_plane_fp<PL, true, true>, k_plane_bp<PL, false, true, true>);
    else if (pl->interp) rc = step(k_plane_fp<PL, true, false>, k_plane_bp<PL, false, false, true>);
    else if (sens) rc = step(k_plane_fp<PL, false, true>, carry ? k_plane_bp<PL, false, true, true> : k_plane_bp<PL, false, true, false>);
    else rc = step(k_plane_fp<PL, false, false>, carry ? k_plane_bp<PL, false, false, true> : k_plane_bp<PL, false, false, false>);
    if (rc) return rc;
    timing_end(s, stop);
    return OMG_OK;
}

int plane_subset_iteration(omg_geom* g, const PlanePlan* pl, int64_t first, int64_t n, float* x, const float* meas,
                           const float* add, float* S, int32_t compute_sens, float epps, const float* dU,
                           int32_t positivity, hipStream_t s, bool* done) {
    const uint32_t planes = (uint32_t)(n / pl->bins);
    const SidArgs sa = make_sid_args(g, first, n);
    PlaneRun a;
    a.bins = pl->bins; a.nyx = pl->nyx; a.npix = pl->npix; a.xrows = pl->xrows; a.planes = planes;
    a.nx = g->d.Nx;
    a.nz = g->d.Nz;
    a.off = pl->off; a.len = pl->len; a.soff = pl->soff; a.slen = pl->slen; a.coff = pl->coff; a.clen = pl->clen;
    a.ent = pl->ent; a.cent = pl->cent; a.samp = pl->samp; a.cpos = pl->cpos;
    a.w = pl->w + (size_t)first * pl->bins;
    a.slice = pl->slice + first;
    a.nent = (uint32_t)pl->nent;      // below 2^32 (list_layout)
    a.share = pl->share;
    a.z = pl->interp ? g->z_dev + 2 * first : nullptr;
    a.bz = g->d.bz;
    a.sz = (float)(1.0 / ((double)g->d.dz * g->d.Nz));
    *done = false;
    // two planes of one slice would update its voxels twice
    std::vector<char> seen(g->d.Nz, 0);
    for (uint32_t p = 0; p < planes; p++) {
        const int32_t tk = pl->slice_host[(size_t)first + p];
        if (tk < 0) continue;
        if (seen[tk]) return OMG_OK;
        seen[tk] = 1;
    }
    // planes side by side per lane group: eight fill a 32-byte run; fewer where the call has fewer
    if (planes > 4) return run_planes<8>(g, pl, a, sa, x, meas, add, S, compute_sens != 0, epps, dU, positivity, s, done);
    if (planes > 2) return run_planes<4>(g, pl, a, sa, x, meas, add, S, compute_sens != 0, epps, dU, positivity, s, done);
    if (planes > 1) return run_planes<2>(g, pl, a, sa, x, meas, add, S, compute_sens != 0, epps, dU, positivity, s, done);
    return run_planes<1>(g, pl, a, sa, x, meas, add, S, compute_sens != 0, epps, dU, positivity, s, done);
}

}  // namespace omg
