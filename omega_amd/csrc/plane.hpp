// plane.hpp -- the lists of a direct-plane sinogram's one 2-D system, shared by its planes (plane.hip).
#pragma once
#include "common.hpp"

#include <vector>

struct omg_geom;

namespace omg {

// Lists are interleaved by kLI rows and padded to a multiple of kLUnroll entries: entry k of row r sits at
// off[r / kLI] + k * kLI + r % kLI, so the rows that a wave holds read one contiguous run per k.
constexpr uint32_t kLI = 8;
constexpr uint32_t kLUnroll = 8;

// Where the tracing kernels put a row's entries. Counting pass: ent null, cnt[row] and the pixels' counts.
// Filling pass: ent (and for the interpolation projector samp) and the LOR weights of every plane.
struct PlaneFill {
    uint32_t npix;               // pixel lists: Nx * Ny, and those of the slices behind (PlanePlan)
    uint32_t slice_base;         // linear index of the traced plane's slice
    uint32_t* cnt;               // [rows] entries
    uint32_t* pixcnt;            // [npix] entries
    uint32_t* scnt;              // [rows] forward samples (interpolation projector)
    int32_t* bad;                // set when a voxel lies outside the lists
    const uint32_t* off;         // [row groups]
    uint2* ent;                  // {pixel, float bits}
    const uint32_t* soff;
    uint4* samp;                 // {pixel | x step << 30 | y step << 31, x fraction, y fraction, length}
};

// A visited voxel of row `row`: counted, or stored as entry k.
__device__ __forceinline__ void plane_put(const PlaneFill& f, uint32_t row, uint32_t& k, uint32_t ind, float w) {
    const uint32_t pix = ind - f.slice_base;
    if (pix >= f.npix) {
        *f.bad = 1;
        return;
    }
    if (f.ent) f.ent[(size_t)f.off[row / kLI] + k * kLI + row % kLI] = make_uint2(pix, __float_as_uint(w));
    else atomicAdd(f.pixcnt + pix, 1u);
    k++;
}

struct PlanePlan;

// The lists of g, built on the first call that may allocate and wait (not under stream capture, not in a
// no-allocation call); null when they do not apply or do not fit.
const PlanePlan* plane_plan(const omg_geom* g, hipStream_t s);
void plane_release(omg_geom* g);

// One OSEM / OSL-OSEM subset iteration from the lists: planes [first, first + n / bins) of distinct slices.
// *done false: nothing was launched (work memory short in a no-allocation call or under stream capture).
int plane_subset_iteration(omg_geom* g, const PlanePlan* pl, int64_t first, int64_t n, float* x, const float* meas,
                           const float* add, float* S, int32_t compute_sens, float epps, const float* dU,
                           int32_t positivity, hipStream_t s, bool* done);

// Tracing launches, one per projector (siddon.hip, orth.hip, interp.hip): the rows of plane `plane` into f,
// and the LOR weights of all planes ([n_proj][bins]).
int siddon_plane_trace(const omg_geom* g, uint32_t plane, const PlaneFill& f, hipStream_t s);
int siddon_plane_weights(const omg_geom* g, float* w, hipStream_t s);
int tof_plane_trace(const omg_geom* g, uint32_t plane, const PlaneFill& f, hipStream_t s);
int tof_plane_shares(const omg_geom* g, uint32_t plane, const PlaneFill& f, uint32_t pitch, float* share, float* lsum,
                     hipStream_t s);
int orth_plane_trace(const omg_geom* g, uint32_t plane, const PlaneFill& f, hipStream_t s);
int orth_plane_weights(const omg_geom* g, float* w, hipStream_t s);
int interp_plane_trace(const omg_geom* g, uint32_t plane, const PlaneFill& f, hipStream_t s);
int interp_plane_weights(const omg_geom* g, float* w, hipStream_t s);
// Image slices of the planes as the projector's own arithmetic places them (-1: the plane misses the image).
void siddon_plane_slices(const omg_geom* g, std::vector<int32_t>& out);
void interp_plane_slices(const omg_geom* g, std::vector<int32_t>& out);
// True when every tube of a projector-2 direct-plane sinogram stays in its slice and the planes lie at the same offset
// from their slice centres but for rounding; *plane: the one to trace.
bool orth_plane_ok(const omg_geom* g, uint32_t* plane);

}  // namespace omg
