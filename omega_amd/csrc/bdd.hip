// bdd.hip -- branchless distance-driven projector (projector type 5), CT flat-panel data.
//
// Semantics of projectorType5Forward / projectorType5Backward (source/opencl/projectorType5.cl:64-337,
// :381-756): the forward projection averages the volume over each detector pixel's footprint on every
// slab (x- or y-slabs, whichever the source direction is closer to) with four taps of the slab's
// summed-area table; the backprojection is voxel-driven and takes four taps of each projection's
// summed-area table over the voxel's footprint. Summed-area tables are built here on the device
// (prefix along z / columns first, then along the fast axis), and every tap is an exact FP32 bilinear
// interpolation in normalised coordinates with clamp-to-edge, where the reference uses texture
// filtering; the slab or projection coordinate selects its table exactly.
//
// gfx950 mapping: FP is one lane per (detector row, group of 8 detector columns, projection) -- the reference's
// grouping, which lets consecutive columns reuse two of the four taps -- over slab tables that a workgroup first
// interpolates along its rows' edges into LDS. BP is one lane per (x, y) column and a run of z; all lanes walk the
// projections in the same order, so the projection's table (e.g. 513 x 385 floats) stays resident in L2. The
// per-projection back-projection geometry is precomputed once per geometry handle (computeGeom5,
// source/Python/omegatomo/projector/init.py:6-37) and read through scalar loads.
#include "geom.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace omg {

struct BddArgs {
    uint32_t Nx, Ny, Nz, nRows, nCols, nProj;   // nProj: projections in this call
    float dx, dy, dz, bx, by, bz, pitchX, pitchY;
    float scaleX, scaleY, scaleZ;                // 1 / (d * (N + 1)), computeProjectorScalingValues
    const float* xyz;                            // 6 floats per projection (subset-offset)
    const float* uv;                             // 2 floats per projection (subset-offset)
    const float* geom5;                          // 16 floats per projection (subset-offset)
};

// ---- taps -------------------------------------------------------------------------------------------
// A tap is a bilinear interpolation of a W x H table at u W - 0.5, v H - 0.5 with clamp to edge. The tables
// carry one replicated column and row on every side (pitch W + 2), so that a clamped coordinate is a cell index
// in [0, W] whose two columns are neighbours: no second index, and one 8-byte load per row.
struct Cell {
    int32_t i;       // the cell's first column / row, -1 .. n - 1 (the table pointers skip the padding)
    float a, na;     // fraction and 1 - fraction
};

__device__ __forceinline__ Cell cell(float u, float n, float top) {   // top = n - 1
    const float c = u * n - 0.5f;
    const float f = floorf(c);
    Cell r;
    r.a = c - f;
    r.na = 1.f - r.a;
    r.i = (int32_t)__builtin_amdgcn_fmed3f(f, -1.f, top);
    return r;
}

struct __attribute__((packed, aligned(4))) F2 { float x, y; };

// Byte offset of a cell's first row: both factors fit 24 bits (one full-rate multiply).
__device__ __forceinline__ int32_t row_off(const Cell& y, uint32_t pitch) { return __mul24(y.i, (int)pitch); }

// The tap at column cell x (byte offset off of its first entry in the row) of the two rows at T0 and T1.
__device__ __forceinline__ float tap(const char* __restrict__ T0, const char* __restrict__ T1, int32_t off,
                                     const Cell& x, const Cell& y) {
    const F2 p = *reinterpret_cast<const F2*>(T0 + off), q = *reinterpret_cast<const F2*>(T1 + off);
    const float r0 = x.na * p.x + x.a * p.y;
    const float r1 = x.na * q.x + x.a * q.y;
    return y.na * r0 + y.a * r1;
}

// Correctly rounded square root and quotient x / d for a divisor whose correctly rounded reciprocal r is known,
// from the hardware's estimate and fused steps (Markstein, "Computation of elementary functions on the IBM RISC
// System/6000 processor", 1990), for arguments whose results neither overflow nor are denormal.
__device__ __forceinline__ float sqrt_rn(float x) {
    const float y = __builtin_amdgcn_rsqf(x);
    float g = x * y, h = 0.5f * y;
    const float r = __builtin_fmaf(-h, g, 0.5f);
    g = __builtin_fmaf(g, r, g);
    h = __builtin_fmaf(h, r, h);
    return __builtin_fmaf(__builtin_fmaf(-g, g, x), h, g);
}
__device__ __forceinline__ float div_rn(float x, float d, float r) {
    const float q = x * r;
    return __builtin_fmaf(__builtin_fmaf(-q, d, x), r, q);
}

__device__ __forceinline__ float len3(float x, float y, float z) { return sqrtf(x * x + y * y + z * z); }

// ---- summed-area tables ----------------------------------------------------------------------------
// Volume: IY, Ny slabs of (Nx+1) x (Nz+1), and IX, Nx slabs of (Ny+1) x (Nz+1), z fastest; first row and column
// zero; padded as above, the z pitch rounded up to four entries (zpitch). The sums run along z first, then along
// the slab's other axis, each one after the other in float.
__host__ __device__ __forceinline__ uint32_t zpitch(uint32_t Nz) { return (Nz + 3 + 3) & ~3u; }

// z sums, x fastest -> z fastest: a wave holds 64 columns of one image row and turns 32 z at a time through LDS
// (one lane per column storing both x-fastest tables put the x slabs' stores on a line each: 272 us at 256^3 and
// 2 x 146 us for the second sums, against 104 and 2 x 52 us). Lands in IY's cells, not yet summed along x.
__global__ __launch_bounds__(256) void k_sat_z(BddArgs a, const float* __restrict__ vol, float* __restrict__ IY) {
    __shared__ float tile[4][32][65];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t x = blockIdx.x * 64 + lane, y = blockIdx.y * 4 + wave;
    const uint32_t zp = zpitch(a.Nz);
    const bool in = x < a.Nx && y < a.Ny;
    float acc = 0.f;
    for (uint32_t z0 = 0; z0 < a.Nz; z0 += 32) {
#pragma unroll
        for (uint32_t k = 0; k < 32; k++) {
            acc += in && z0 + k < a.Nz ? vol[x + (size_t)y * a.Nx + (size_t)(z0 + k) * a.Nx * a.Ny] : 0.f;
            tile[wave][k][lane] = acc;
        }
        __syncthreads();
        const uint32_t z = z0 + (lane & 31);
        for (uint32_t r = lane >> 5; r < 64; r += 2)
            if (y < a.Ny && blockIdx.x * 64 + r < a.Nx && z < a.Nz)
                IY[((size_t)y * (a.Nx + 3) + blockIdx.x * 64 + r + 2) * zp + z + 2] = tile[wave][lane & 31][r];
        __syncthreads();
    }
}

// Sums of slab blockIdx.y along its other axis (n columns): in(c) = src + c * stride, the table's column c + 2 at
// dst. One lane per z; the zero columns, the replicated ones and the z padding too. dst may be src.
__global__ __launch_bounds__(64) void k_sat_slab(const float* src, float* dst, uint32_t n, uint32_t Nz, size_t slab_in,
                                                 size_t stride, size_t slab_out) {
    const uint32_t e = blockIdx.x * 64 + threadIdx.x, zp = zpitch(Nz);
    if (e > Nz + 1) return;
    float* out = dst + blockIdx.y * slab_out + e;
    out[0] = 0.f;
    out[zp] = 0.f;
    const uint32_t pads = e == Nz + 1 ? zp - 1 - e : 0;    // the last z again in the entries behind it
    for (uint32_t j = 0; j < 2; j++)
        for (uint32_t q = 1; q <= pads; q++) out[(size_t)j * zp + q] = 0.f;
    const float* in = src + blockIdx.y * slab_in + e;
    float acc = 0.f;
    for (uint32_t c0 = 0; c0 < n; c0 += 8) {
        float v[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) v[j] = e >= 2 && c0 + j < n ? in[(c0 + j) * stride] : 0.f;
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) {
            if (c0 + j < n) {
                acc += v[j];
                for (uint32_t q = 0; q <= pads; q++) out[(size_t)(c0 + j + 2) * zp + q] = acc;
            }
        }
    }
    for (uint32_t q = 0; q <= pads; q++) out[(size_t)(n + 2) * zp + q] = acc;
}

// Sinogram tables: sums along the columns per detector row first; nProj tables of (nCols+1) x (nRows+1).
__global__ __launch_bounds__(256) void k_sat_sino_cols(BddArgs a, const float* __restrict__ y, float* __restrict__ S) {
    const uint32_t r = blockIdx.x * 256 + threadIdx.x, k = blockIdx.y;
    if (r >= a.nRows) return;
    const size_t P = a.nRows + 3, H = a.nCols + 3;
    float* T = S + (size_t)k * P * H + r + 2;
    const float* in = y + r + (size_t)k * a.nRows * a.nCols;
    float acc = 0.f;
    for (uint32_t c0 = 0; c0 < a.nCols; c0 += 8) {
        float v[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) v[j] = c0 + j < a.nCols ? in[(size_t)(c0 + j) * a.nRows] : 0.f;
#pragma unroll
        for (uint32_t j = 0; j < 8; j++) {
            acc += v[j];
            if (c0 + j < a.nCols) T[(size_t)(c0 + j + 2) * P] = acc;
        }
    }
}

// Sums along the fast axis of 64 rows of a W x H table (padded pitch W + 2), 64 columns at a time through LDS,
// and the table's zero first row and column and its padding. grid = (ceil((H + 2) / 64), tables). (One lane per
// row straight from memory took 236 us for 45 views of 512 x 384, against 72 us.)
__global__ __launch_bounds__(256) void k_sat_rows(float* __restrict__ tables, uint32_t W, uint32_t H) {
    __shared__ float t[64][65];
    const uint32_t P = W + 2;
    float* T = tables + (size_t)blockIdx.y * P * (H + 2);
    const uint32_t row0 = blockIdx.x * 64;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float acc = 0.f;
    // padded rows 2 .. H hold sums (rows 1 .. H-1 of the table); rows 0 and 1 are zero
    for (uint32_t c0 = 0; c0 < W - 1; c0 += 64) {
        for (uint32_t r = wave; r < 64; r += 4) {
            const uint32_t row = row0 + r;
            if (row >= 2 && row <= H && c0 + lane < W - 1) t[r][lane] = T[(size_t)row * P + 2 + c0 + lane];
        }
        __syncthreads();
        if (threadIdx.x < 64) {
            const uint32_t n = min(64u, W - 1 - c0);
            for (uint32_t i = 0; i < n; i++) {
                acc += t[threadIdx.x][i];
                t[threadIdx.x][i] = acc;
            }
        }
        __syncthreads();
        for (uint32_t r = wave; r < 64; r += 4) {
            const uint32_t row = row0 + r;
            if (row >= 2 && row <= H && c0 + lane < W - 1) {
                const float v = t[r][lane];
                T[(size_t)row * P + 2 + c0 + lane] = v;
                if (c0 + lane == W - 2) T[(size_t)row * P + W + 1] = v;            // the last column again
                if (row == H) {                                                   // the last row again
                    T[(size_t)(H + 1) * P + 2 + c0 + lane] = v;
                    if (c0 + lane == W - 2) T[(size_t)(H + 1) * P + W + 1] = v;
                }
            } else if (row < 2 && c0 + lane < W - 1) {
                T[(size_t)row * P + 2 + c0 + lane] = 0.f;
                if (c0 + lane == W - 2) T[(size_t)row * P + W + 1] = 0.f;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 128) {
        const uint32_t row = row0 + (threadIdx.x >> 1);
        if (row < H + 2) T[(size_t)row * P + (threadIdx.x & 1)] = 0.f;             // first column and its pad
    }
}

// ---- forward projection ----------------------------------------------------------------------------
constexpr int kCols = 8;
constexpr uint32_t kXcds = 8;

// A workgroup holds `rb` detector rows of one view with all their column groups, one lane per (row, group). Per
// slab the row's two edges fix two column cells of the slab's table, so the table is first interpolated along them
// for every z, h[row][z] = {left edge, right edge}, into LDS (one item of four z per lane: four 16-byte loads),
// and a tap is then one LDS read of two neighbouring z and three operations per edge. The next slab's h is written
// while this one's is read (two buffers, one barrier per slab). The operations of a tap and their order are the
// reference's. Each XCD gets a contiguous range of blocks, so that the blocks that sweep one view's slabs together
// share an L2. What bounds it: VALU, about 38 operations per pixel and slab. 256^3, 45 views of 512 x 384:
// 6.85 -> 2.2 ms (one lane per (row, group) with four full bilinear taps from memory; with shared cells and 8-byte
// loads, still from memory, 4.5 ms: 4.5 loads per pixel and slab at 16 clocks each). LDS false: h is formed at
// every tap from memory, for volumes with more slices than LDS holds two rows of (about 10000).
template <bool LDS>
__global__ __launch_bounds__(256) void k_bdd_fp(BddArgs a, uint32_t per_xcd, uint32_t per_view, uint32_t rb,
                                                const float* __restrict__ IY, const float* __restrict__ IX,
                                                float* __restrict__ out) {
    extern __shared__ float4 lds4[];
    const uint32_t groups = (a.nCols + kCols - 1) / kCols, gl = min(groups, 256u), gc = (groups + 255) / 256;
    const uint32_t block = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    const uint32_t k = block / per_view;                        // one view per block: its table is uniform
    if (k >= a.nProj) return;
    const uint32_t b = block - k * per_view;
    const uint32_t row0 = b / gc * rb, rr = threadIdx.x / gl;
    const uint32_t g = b % gc * gl + threadIdx.x % gl;
    const uint32_t r = row0 + rr, c0 = g * kCols;
    const bool live = rr < rb && r < a.nRows && g < groups;
    const float* P = a.xyz + (size_t)k * 6;
    const float sx = P[0], sy = P[1], sz = P[2];
    const float ux = a.uv[(size_t)k * 2], uy = a.uv[(size_t)k * 2 + 1];
    const bool ydir = fabsf(sx) <= fabsf(sy);
    // slab axis: y-slabs sample IY in (x, z); x-slabs sample IX in (y, z). Edge slopes of detector row q:
    auto slopes = [&](uint32_t q, float& L0, float& L1) {
        const float i1 = (float)q - (float)a.nRows / 2.f + .5f;
        const float x = P[3] + i1 * ux, y = P[4] + i1 * uy;
        const float dRx = x - ux * 0.5f, dRy = y - uy * 0.5f;
        const float dLx = x + ux * 0.5f, dLy = y + uy * 0.5f;
        L0 = ydir ? (dLx - sx) / (dLy - sy) : (dLy - sy) / (dLx - sx);
        L1 = ydir ? (dRx - sx) / (dRy - sy) : (dRy - sy) / (dRx - sx);
    };
    const float apuT = ydir ? (a.bx - sx - a.dx / 2.f) : (a.by - sy - a.dy / 2.f);
    const float apuV = ydir ? a.by - sy : a.bx - sx;
    const float apuZ = (a.bz - sz - a.dz / 2.f);
    const float dslab = ydir ? a.dy : a.dx;
    const float scaleT = ydir ? a.scaleX : a.scaleY;
    const float Wf = (float)(ydir ? a.Nx + 1 : a.Ny + 1), Hf = (float)(a.Nz + 1);
    const float Wt = Wf - 1.f, Ht = Hf - 1.f;
    const uint32_t nslab = ydir ? a.Ny : a.Nx, zp = zpitch(a.Nz), quads = zp / 4;
    const size_t slab = (size_t)((ydir ? a.Nx : a.Ny) + 3) * zp;
    const float* T = (ydir ? IY : IX) + zp;                     // the table's own first column
    float2* h0 = reinterpret_cast<float2*>(lds4);               // [2][rb][zp]
    float* rowL = reinterpret_cast<float*>(h0 + 2 * (size_t)rb * zp);   // [rb][2]
    if (LDS && threadIdx.x < rb) slopes(row0 + threadIdx.x, rowL[2 * threadIdx.x], rowL[2 * threadIdx.x + 1]);
    __syncthreads();
    auto build = [&](float v, float4* h) {                      // h of the slab at T
        for (uint32_t it = threadIdx.x; it < rb * quads; it += 256) {
            const uint32_t q = it / quads, zq = it - q * quads;
            const float a0 = v * rowL[2 * q] - apuT, a1 = v * rowL[2 * q + 1] - apuT;
            const Cell cl = cell(fminf(a0, a1) * scaleT, Wf, Wt), cr = cell(fmaxf(a0, a1) * scaleT, Wf, Wt);
            const float4* pl = reinterpret_cast<const float4*>(T + (ptrdiff_t)cl.i * (ptrdiff_t)zp) + zq;
            const float4* pr = reinterpret_cast<const float4*>(T + (ptrdiff_t)cr.i * (ptrdiff_t)zp) + zq;
            const float4 l0 = pl[0], l1 = pl[quads], r0 = pr[0], r1 = pr[quads];
            h[2 * it] = make_float4(cl.na * l0.x + cl.a * l1.x, cr.na * r0.x + cr.a * r1.x,
                                    cl.na * l0.y + cl.a * l1.y, cr.na * r0.y + cr.a * r1.y);
            h[2 * it + 1] = make_float4(cl.na * l0.z + cl.a * l1.z, cr.na * r0.z + cr.a * r1.z,
                                        cl.na * l0.w + cl.a * l1.w, cr.na * r0.w + cr.a * r1.w);
        }
    };
    const float i1 = (float)r - (float)a.nRows / 2.f + .5f, i2 = (float)c0 - (float)a.nCols / 2.f + .5f;
    const float dxp = P[3] + i1 * ux, dyp = P[4] + i1 * uy, dzp = P[5] + i2 * a.pitchY;
    const float dUz = dzp + a.pitchY * 0.5f, dDz = dzp - a.pitchY * 0.5f;
    const float ex = dxp - sx, ey = dyp - sy, ez = dzp - sz;
    const float inv = 1.f / len3(ex, ey, ez);
    float kerroin = a.dx * a.dy * a.dz;
    kerroin /= ydir ? fabsf(ey * inv) : fabsf(ex * inv);
    const float Z0 = ydir ? (dUz - sz) / (dyp - sy) : (dUz - sz) / (dxp - sx);
    const float Z1 = ydir ? (dDz - sz) / (dyp - sy) : (dDz - sz) / (dxp - sx);
    float L0, L1;
    slopes(r, L0, L1);
    const int maxZZ = min(kCols, (int)a.nCols - (int)c0);
    float temp[kCols];
#pragma unroll
    for (int q = 0; q < kCols; q++) temp[q] = 0.f;
    float half = dslab / 2.f;
    if (LDS) {
        build(half + apuV, lds4);
        __syncthreads();
    }
    for (uint32_t jj = 0; jj < nslab; jj++) {
        const float v = half + apuV;
        half += dslab;
        if (LDS) T += slab;
        if (LDS && jj + 1 < nslab) build(half + apuV, lds4 + ((jj + 1) & 1) * (size_t)rb * quads * 2);
        if (live) {
            const float a0 = v * L0 - apuT, a1 = v * L1 - apuT;
            const float b0 = v * Z0 - apuZ, b1 = v * Z1 - apuZ;
            const float tl = fminf(a0, a1), tr = fmaxf(a0, a1);
            float zu = fminf(b0, b1), zd = fmaxf(b0, b1);
            const float invArea = 1.f / fabsf((tl - tr) * (zu - zd));
            zu *= a.scaleZ; zd *= a.scaleZ;
            const float2* h = h0 + ((size_t)(jj & 1) * rb + rr) * zp + 1;
            const Cell cl = cell(tl * scaleT, Wf, Wt), cr = cell(tr * scaleT, Wf, Wt);   // LDS false
            const float* hl = T + (ptrdiff_t)cl.i * (ptrdiff_t)zp + 1;
            const float* hr = T + (ptrdiff_t)cr.i * (ptrdiff_t)zp + 1;
            auto taps = [&](float z, float& l, float& rt) {
                const Cell c = cell(z, Hf, Ht);
                float2 p, q;
                if (LDS) {
                    p = h[c.i];
                    q = h[c.i + 1];
                } else {
                    p = make_float2(cl.na * hl[c.i] + cl.a * hl[c.i + (int)zp], cr.na * hr[c.i] + cr.a * hr[c.i + (int)zp]);
                    q = make_float2(cl.na * hl[c.i + 1] + cl.a * hl[c.i + 1 + (int)zp],
                                    cr.na * hr[c.i + 1] + cr.a * hr[c.i + 1 + (int)zp]);
                }
                l = c.na * p.x + c.a * q.x;
                rt = c.na * p.y + c.a * q.y;
            };
            float A, B, C, D;
            taps(zu, D, A);
            taps(zd, B, C);
            temp[0] += (C + D - A - B) * invArea;
            const float step = fabsf(zu - zd);
#pragma unroll
            for (int q = 1; q < kCols; q++) {
                D = B; A = C;
                zd += step;
                taps(zd, B, C);
                temp[q] += (C + D - A - B) * invArea;
            }
        }
        if (LDS) __syncthreads();
        else T += slab;
    }
    if (!live) return;
#pragma unroll
    for (int q = 0; q < kCols; q++)
        if (q < maxZZ) out[r + (size_t)(c0 + q) * a.nRows + (size_t)k * a.nRows * a.nCols] = temp[q] * kerroin;
}

// ---- backprojection (voxel-driven) -------------------------------------------------------------------
// One lane per (x, y) column and NZ voxels along z. Where a voxel's faces fall across the panel's rows does not
// depend on z: the geometry's panels stand along z (geom5: o[8] = o[9] = o[10] = 0), and the faces' scales
// tLU, tRD depend on z only through lu2 * o[14], the rounding residue of a zero, which is lost in the sum for all
// z of a lane unless the first and the last differ. So the row cells (Ax, Dx) and all divisions are formed once per
// (column, view); the panel columns that the lane's voxels fall on are interpolated along both cells once,
// win[column][lane] = {at Ax, at Dx} in LDS, and a voxel reads its two column cells there. Waves whose window
// passes kWin columns, or whose faces' scales differ along z, take every tap from memory. Operations and order are
// the reference's. What bounds it: VALU, about 90 operations per voxel and view. 256^3, 45 views of 512 x 384:
// 4.55 -> 1.8 ms (every voxel by itself, four full taps of 16 loads; with shared cells but taps from memory 2.8).
constexpr int kWin = 16;

template <int NZ, bool SENS>
__global__ __launch_bounds__(256, 4) void k_bdd_bp(BddArgs a, const float* __restrict__ S, float* __restrict__ vol,
                                                   float* __restrict__ sens) {
    __shared__ float2 win[kWin][256];
    const uint32_t Nxy = a.Nx * a.Ny;
    const uint32_t rem = blockIdx.x * 256 + threadIdx.x, kz0 = blockIdx.y * NZ;
    if (rem >= Nxy) return;
    const uint32_t j = rem / a.Nx, i = rem - j * a.Nx;
    const float vx = (float)i * a.dx + a.dx / 2.f + a.bx;
    const float vy = (float)j * a.dy + a.dy / 2.f + a.by;
    const float kokoX = (float)(a.nRows + 1) * a.pitchX, kokoY = (float)(a.nCols + 1) * a.pitchY;
    const float invKx = 1.f / kokoX, invKy = 1.f / kokoY;
    const float Wf = (float)(a.nRows + 1), Hf = (float)(a.nCols + 1);
    const float Wt = Wf - 1.f, Ht = Hf - 1.f;
    const uint32_t pitch = 4u * (a.nRows + 3);
    const char* T0 = reinterpret_cast<const char*>(S) + pitch + 4;
    float temp[NZ], ws[NZ];
#pragma unroll
    for (int z = 0; z < NZ; z++) { temp[z] = 0.f; ws[z] = 0.f; }
    for (uint32_t kk = 0; kk < a.nProj; kk++) {
        const float* o = a.geom5 + (size_t)kk * 16;
        const float s0 = o[0], s1 = o[1], s2 = o[2];
        const bool sxDim = fabsf(s0) <= fabsf(s1);
        float lu0, lu1, rd0, rd1;
        if (sxDim) {
            const bool pos = s1 > 0.f;
            lu0 = pos ? vx - a.dx / 2.f : vx + a.dx / 2.f;
            rd0 = pos ? vx + a.dx / 2.f : vx - a.dx / 2.f;
            lu1 = vy; rd1 = vy;
        } else {
            const bool pos = s0 > 0.f;
            lu1 = pos ? vy + a.dy / 2.f : vy - a.dy / 2.f;
            rd1 = pos ? vy - a.dy / 2.f : vy + a.dy / 2.f;
            lu0 = vx; rd0 = vx;
        }
        lu0 -= s0; lu1 -= s1;
        rd0 -= s0; rd1 -= s1;
        const float nl = -lu0 * o[12] + -lu1 * o[13], nr = -rd0 * o[12] + -rd1 * o[13];
        auto vzc = [&](uint32_t kz) { return (float)kz * a.dz + a.dz / 2.f + a.bz; };
        auto lz = [&](uint32_t kz) { return vzc(kz) - a.dz / 2.f - s2; };
        auto rz = [&](uint32_t kz) { return vzc(kz) + a.dz / 2.f - s2; };
        float dl = nl + -lz(kz0) * o[14], dr = nr + -rz(kz0) * o[14];
        const bool same = dl == nl + -lz(kz0 + NZ - 1) * o[14] && dr == nr + -rz(kz0 + NZ - 1) * o[14];
        const float vdx = vx - s0, vdy = vy - s1;
        const float q2 = vdx * vdx + vdy * vdy;
        const float dk = sxDim ? a.dy : a.dx, vk = sxDim ? fabsf(vdy) : fabsf(vdx), rk = 1.f / vk;
        float tLU, tRD;
        Cell ca, cd;
        auto columns = [&]() {
            tLU = o[15] / dl;
            tRD = o[15] / dr;
            const float pl0 = lu0 * tLU + s0 - o[3], pl1 = lu1 * tLU + s1 - o[4];
            const float pr0 = rd0 * tRD + s0 - o[3], pr1 = rd1 * tRD + s1 - o[4];
            float Ax = pl0 * o[6] + pl1 * o[7] + a.pitchX / 2.f, Dx = pr0 * o[6] + pr1 * o[7] + a.pitchX / 2.f;
            if (Dx > Ax) { const float t = Ax; Ax = Dx; Dx = t; }
            ca = cell(Ax * invKx, Wf, Wt);
            cd = cell(Dx * invKx, Wf, Wt);
        };
        auto edges = [&](uint32_t kz, Cell& ya, Cell& yd) {
            const float pl2 = lz(kz) * tLU + s2 - o[5], pr2 = rz(kz) * tRD + s2 - o[5];
            float Ay = pl2 * o[11] + a.pitchY / 2.f, Dy = pr2 * o[11] + a.pitchY / 2.f;
            if (Dy > Ay) { const float t = Ay; Ay = Dy; Dy = t; }
            ya = cell(Ay * invKy, Hf, Ht);
            yd = cell(Dy * invKy, Hf, Ht);
        };
        auto add = [&](int z, float apu) {
            const float vdz = vzc(kz0 + z) - s2;
            const float kerroin = div_rn(dk * sqrt_rn(q2 + vdz * vdz), vk, rk);
            temp[z] += apu != 0.f ? apu * kerroin : 0.f;
            if (SENS) ws[z] += apu != 0.f ? kerroin : 0.f;
        };
        columns();
        // panel columns of the lane's voxels: the cells are monotone in z
        Cell y0, y1, y2, y3;
        edges(kz0, y0, y1);
        edges(kz0 + NZ - 1, y2, y3);
        const int lo = min(min(y0.i, y1.i), min(y2.i, y3.i));
        const int n = max(max(y0.i, y1.i), max(y2.i, y3.i)) + 2 - lo;
        if (__all(same && n <= kWin)) {
            const char* Ta = T0 + 4 * ca.i;
            const char* Td = T0 + 4 * cd.i;
#pragma unroll
            for (int r = 0; r < kWin; r += 4) {
                if (!__any(r < n)) break;
                F2 p[4], q[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int off = __mul24(min(lo + r + e, (int)a.nCols + 1), (int)pitch);
                    p[e] = *reinterpret_cast<const F2*>(Ta + off);
                    q[e] = *reinterpret_cast<const F2*>(Td + off);
                }
#pragma unroll
                for (int e = 0; e < 4; e++)
                    win[r + e][threadIdx.x] = make_float2(ca.na * p[e].x + ca.a * p[e].y, cd.na * q[e].x + cd.a * q[e].y);
            }
#pragma unroll
            for (int z = 0; z < NZ; z++) {
                Cell ya, yd;
                edges(kz0 + z, ya, yd);
                const float2 a0 = win[ya.i - lo][threadIdx.x], a1 = win[ya.i - lo + 1][threadIdx.x];
                const float2 d0 = win[yd.i - lo][threadIdx.x], d1 = win[yd.i - lo + 1][threadIdx.x];
                const float A = ya.na * a0.x + ya.a * a1.x, C = ya.na * a0.y + ya.a * a1.y;
                const float B = yd.na * d0.x + yd.a * d1.x, D = yd.na * d0.y + yd.a * d1.y;
                add(z, A + D - C - B);
            }
        } else {
            const char* T1 = T0 + pitch;
#pragma unroll
            for (int z = 0; z < NZ; z++) {
                __builtin_amdgcn_sched_barrier(0);
                dl = nl + -lz(kz0 + z) * o[14];
                dr = nr + -rz(kz0 + z) * o[14];
                columns();
                Cell ya, yd;
                edges(kz0 + z, ya, yd);
                const int32_t ra = row_off(ya, pitch), rd = row_off(yd, pitch), oa = 4 * ca.i, od = 4 * cd.i;
                const float A = tap(T0, T1, ra + oa, ca, ya), B = tap(T0, T1, rd + oa, ca, yd);
                const float C = tap(T0, T1, ra + od, cd, ya), D = tap(T0, T1, rd + od, cd, yd);
                add(z, A + D - C - B);
            }
        }
        T0 += (size_t)pitch * (a.nCols + 3);
    }
#pragma unroll
    for (int z = 0; z < NZ; z++) {
        if (kz0 + z < a.Nz) {
            const size_t n = rem + (size_t)(kz0 + z) * Nxy;
            vol[n] += temp[z];
            if (SENS) sens[n] += ws[z];
        }
    }
}

static BddArgs make_bdd_args(const omg_geom* g, int64_t first, uint32_t nproj) {
    BddArgs a;
    a.Nx = g->d.Nx; a.Ny = g->d.Ny; a.Nz = g->d.Nz;
    a.nRows = g->d.size_x; a.nCols = g->d.size_y; a.nProj = nproj;
    a.dx = g->d.dx; a.dy = g->d.dy; a.dz = g->d.dz;
    a.bx = g->d.bx; a.by = g->d.by; a.bz = g->d.bz;
    a.pitchX = g->d.dPitchX; a.pitchY = g->d.dPitchY;
    a.scaleX = 1.f / (g->d.dx * (float)(g->d.Nx + 1));
    a.scaleY = 1.f / (g->d.dy * (float)(g->d.Ny + 1));
    a.scaleZ = 1.f / (g->d.dz * (float)(g->d.Nz + 1));
    a.xyz = g->x_dev + first * 6;
    a.uv = g->z_dev + first * 2;
    a.geom5 = g->bdd_geom5 + first * 16;
    return a;
}

}  // namespace omg

using namespace omg;

// Host: per-projection back-projection geometry, computeGeom5 (init.py:6-37) in float arithmetic.
int bdd_prepare(omg_geom* g) {
    OMG_REQUIRE(!g->d.ct_pitch, "projector_type 5 supports the uV (2 floats per projection) panel description");
    OMG_REQUIRE(g->d.dPitchX > 0.f && g->d.dPitchY > 0.f, "projector_type 5 needs dPitchX and dPitchY");
    const uint32_t P = g->d.n_proj;
    std::vector<float> x(P * 6), uv(P * 2), out((size_t)P * 16);
    OMG_CHECK_HIP(hipMemcpy(x.data(), g->x_dev, x.size() * sizeof(float), hipMemcpyDeviceToHost));
    OMG_CHECK_HIP(hipMemcpy(uv.data(), g->z_dev, uv.size() * sizeof(float), hipMemcpyDeviceToHost));
    const float indX = (float)g->d.size_x / 2.f, indY = (float)g->d.size_y / 2.f;
    const float c0[3] = {g->d.bx + 0.5f * g->d.Nx * g->d.dx, g->d.by + 0.5f * g->d.Ny * g->d.dy,
                         g->d.bz + 0.5f * g->d.Nz * g->d.dz};
    for (uint32_t k = 0; k < P; k++) {
        const float* p = &x[(size_t)k * 6];
        const float sd = std::hypot(p[3] - p[0], p[4] - p[1]), sc = std::hypot(c0[0] - p[0], c0[1] - p[1]);
        if (sc > 0.f) g->bdd_mag = std::max(g->bdd_mag, sd / sc);
        const float s[3] = {p[0], p[1], p[2]}, d[3] = {p[3], p[4], p[5]};
        const float ax[3] = {uv[2 * k] * indX, uv[2 * k + 1] * indX, 0.f};
        const float ay[3] = {0.f, 0.f, indY * g->d.dPitchY};
        float d3[3], d2[3], e[3];
        for (int c = 0; c < 3; c++) { d3[c] = d[c] - ax[c] - ay[c]; d2[c] = ax[c] - ay[c]; }
        for (int c = 0; c < 3; c++) e[c] = d3[c] - d[c];
        const float lx = std::sqrt(ax[0] * ax[0] + ax[1] * ax[1] + ax[2] * ax[2]);
        const float ly = std::sqrt(ay[0] * ay[0] + ay[1] * ay[1] + ay[2] * ay[2]);
        const float cp[3] = {d2[1] * e[2] - d2[2] * e[1], d2[2] * e[0] - d2[0] * e[2], d2[0] * e[1] - d2[1] * e[0]};
        float* o = &out[(size_t)k * 16];
        for (int c = 0; c < 3; c++) {
            o[c] = s[c]; o[3 + c] = d3[c]; o[6 + c] = ax[c] / lx; o[9 + c] = ay[c] / ly; o[12 + c] = cp[c];
        }
        o[15] = cp[0] * (s[0] - d[0]) + cp[1] * (s[1] - d[1]) + cp[2] * (s[2] - d[2]);
    }
    OMG_CHECK_HIP(hipMalloc(reinterpret_cast<void**>(&g->bdd_geom5), out.size() * sizeof(float)));
    OMG_CHECK_HIP(hipMemcpy(g->bdd_geom5, out.data(), out.size() * sizeof(float), hipMemcpyHostToDevice));
    return OMG_OK;
}

void bdd_release(omg_geom* g) {
    hipFree(g->bdd_geom5);
    g->bdd_geom5 = nullptr;
}

int bdd_forward(const omg_geom* g, int64_t first, int64_t n, const float* img, float* y, hipStream_t s) {
    const int64_t per = (int64_t)g->d.size_x * g->d.size_y;
    const uint32_t nproj = (uint32_t)(n / per);
    BddArgs a = make_bdd_args(g, first, nproj);
    const uint32_t zp = zpitch(a.Nz), groups = (a.nCols + kCols - 1) / kCols;
    const size_t slab_y = (size_t)(a.Nx + 3) * zp, slab_x = (size_t)(a.Ny + 3) * zp;
    const size_t sy = slab_y * a.Ny, sx = slab_x * a.Nx;
    // detector rows per workgroup: as many as its lanes and 40 KB of LDS take (four workgroups a CU), one at least
    const size_t row_lds = 2 * sizeof(float2) * (size_t)zp + 2 * sizeof(float);
    uint32_t rb = groups < 256 ? 256 / groups : 1;
    while (rb > 1 && rb * row_lds > 40 * 1024) rb--;
    const bool in_lds = rb * row_lds <= 160 * 1024;
    int rc = scratch_reserve(const_cast<omg_geom*>(g), sy + sx, s);
    if (rc) return rc;
    float* IY = scratch_ptr(g);
    float* IX = scratch_ptr(g) + sy;
    hipLaunchKernelGGL(k_sat_z, dim3((a.Nx + 63) / 64, (a.Ny + 3) / 4), dim3(256), 0, s, a, img, IY);
    OMG_CHECK_LAUNCH();
    const unsigned zb = (a.Nz + 2 + 63) / 64;
    // x slabs first: they read the z sums that the y slabs then sum in place
    hipLaunchKernelGGL(k_sat_slab, dim3(zb, a.Nx), dim3(64), 0, s, IY + 2 * zp, IX, a.Ny, a.Nz, (size_t)zp, slab_y,
                       slab_x);
    OMG_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_sat_slab, dim3(zb, a.Ny), dim3(64), 0, s, IY + 2 * zp, IY, a.Nx, a.Nz, slab_y, (size_t)zp,
                       slab_y);
    OMG_CHECK_LAUNCH();
    const size_t lds = in_lds ? rb * row_lds : 0;
    if (lds > 64 * 1024)   // every time: a device's attribute, and any thread's call
        OMG_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_bdd_fp<true>),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const uint32_t per_view = (a.nRows + rb - 1) / rb * ((groups + 255) / 256);
    const uint32_t per_xcd = (uint32_t)(((uint64_t)per_view * nproj + kXcds - 1) / kXcds);
    hipLaunchKernelGGL(in_lds ? k_bdd_fp<true> : k_bdd_fp<false>, dim3(per_xcd * kXcds), dim3(256), lds, s, a, per_xcd,
                       per_view, rb, IY, IX, y);
    OMG_CHECK_LAUNCH();
    return OMG_OK;
}

int bdd_backward(const omg_geom* g, int64_t first, int64_t n, const float* yin, float* rhs, float* sens, hipStream_t s) {
    const int64_t per = (int64_t)g->d.size_x * g->d.size_y;
    const uint32_t nproj = (uint32_t)(n / per);
    BddArgs a = make_bdd_args(g, first, nproj);
    int rc = scratch_reserve(const_cast<omg_geom*>(g), (size_t)(a.nRows + 3) * (a.nCols + 3) * nproj, s);
    if (rc) return rc;
    float* S = scratch_ptr(g);
    hipLaunchKernelGGL(k_sat_sino_cols, dim3(grid_for(a.nRows, 256), nproj), dim3(256), 0, s, a, yin, S);
    OMG_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_sat_rows, dim3((a.nCols + 3 + 63) / 64, nproj), dim3(256), 0, s, S, a.nRows + 1, a.nCols + 1);
    OMG_CHECK_LAUNCH();
    const uint32_t Nxy = a.Nx * a.Ny;
    auto launch = [&](auto kern, uint32_t nz) {
        hipLaunchKernelGGL(kern, dim3(grid_for(Nxy, 256), (a.Nz + nz - 1) / nz), dim3(256), 0, s, a, S, rhs, sens);
    };
    // eight voxels per lane while their columns fit the window (a voxel spans about step of them) and that leaves
    // the chip (1024 SIMDs) several waves each; else two
    const float step = g->bdd_mag * a.dz / a.pitchY * 1.2f;
    if (8.f * step + 3.f <= (float)kWin && (uint64_t)Nxy * a.Nz >= (uint64_t)8 * 64 * 4096) {
        if (sens) launch(k_bdd_bp<8, true>, 8);
        else launch(k_bdd_bp<8, false>, 8);
    } else if (4.f * step + 3.f <= (float)kWin && (uint64_t)Nxy * a.Nz >= (uint64_t)4 * 64 * 4096) {
        if (sens) launch(k_bdd_bp<4, true>, 4);
        else launch(k_bdd_bp<4, false>, 4);
    } else {
        if (sens) launch(k_bdd_bp<2, true>, 2);
        else launch(k_bdd_bp<2, false>, 2);
    }
    OMG_CHECK_LAUNCH();
    return OMG_OK;
}
