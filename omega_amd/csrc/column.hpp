// column.hpp -- 3-D sinogram projections by image columns (column.hip).
#pragma once
#include "common.hpp"

struct omg_geom;

namespace omg {

struct ColPlan;

// The transaxial lists that serve measurements [first, first + n) of g, built on the first call that may allocate
// and wait; null when they do not apply or do not fit, or with fewer than min_planes planes. A wave's 64 lanes are
// planes, so its time hardly falls with their number: with 64 the forward projection gains 2.3 times (half of that
// with kColPlanes), the backprojection 16 times (kColPlanesBack; 1380 -> 209 us
// with 30 planes of 208 x 128 bins, 123 x 123 x 27 voxels).
constexpr uint32_t kColPlanes = 32, kColPlanesBack = 12;
const ColPlan* col_plan(const omg_geom* g, int64_t first, int64_t n, hipStream_t s, uint32_t min_planes = kColPlanes);
void col_release(omg_geom* g);

// y = A img.
int col_forward(const omg_geom* g, const ColPlan* pl, int64_t first, int64_t n, const float* img, float* y,
                hipStream_t s, bool* done);
// rhs += A^T y (y null: A^T 1); with sens also sens += A^T 1.
int col_backward(const omg_geom* g, const ColPlan* pl, int64_t first, int64_t n, const float* y, float* rhs, float* sens,
                 hipStream_t s, bool* done);
// rhs += A^T (meas / (A img + epps (+ add))), NaN and Inf ratios -> epps; with sens also sens += A^T 1. work: null, or
// col_osem_work floats (calls without sens) that the caller keeps, 16-byte aligned.
size_t col_osem_work(const omg_geom* g, const ColPlan* pl, int64_t n);
int col_osem(const omg_geom* g, const ColPlan* pl, int64_t first, int64_t n, const float* img, const float* meas,
             const float* add, float* rhs, float* sens, float epps, float* work, hipStream_t s, bool* done);

}  // namespace omg
