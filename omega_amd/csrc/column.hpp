// column.hpp -- 3-D sinogram projections by image columns (column.hip).
#pragma once
#include "common.hpp"

struct omg_geom;

namespace omg {

struct ColPlan;

// The transaxial lists that serve measurements [first, first + n) of g, built on the first call that may allocate
// and wait; null when they do not apply or do not fit, or with fewer than min_planes planes. A wave's 64 lanes are
// planes, so its time hardly falls with their number. One lane per LOR / by columns, us, 208 x 128 bins on 123 x 123 x 27
// voxels and 224 x 224 bins on 128 x 128 x 63:
//   planes   forward            backward            fused step
//   8        70/174   102/318   590/263  1174/493   615/392  1157/751
//   16       105/177  183/322   1132/268 2109/499   1104/397 2117/757
//   31       170/179  317/322   2050/274 4022/506   2000/404 3934/766
//   64       310/184  607/331   3962/287 7977/520   3962/414 7864/779
// So forward projections go by columns from kColPlanes on, backprojections from kColPlanesBack. The fused and frames steps
// keep the forward projection's line, by these figures a late one (theirs lies at 8).
constexpr uint32_t kColPlanes = 32, kColPlanesBack = 12;
const ColPlan* col_plan(const omg_geom* g, int64_t first, int64_t n, hipStream_t s, uint32_t min_planes = kColPlanes);
void col_release(omg_geom* g);

// Floats of work memory of a call on n measurements: forward projection (img), backprojection (rec), both, with sens.
size_t col_work_floats(const omg_geom* g, const ColPlan* pl, int64_t n, bool img, bool rec, bool sens);

// Work memory of one call (or of one after the other on one stream), held until the object ends; null (trace instead)
// where there is none to be had. The no-allocation region while one is held. Else, with `beside`, for the projections
// that may run beside each other on several streams and threads of one handle (forward projections and sensitivity
// images, whose tracing kernels touch the caller's arrays only): a buffer of the stream, kept for its next call, up to
// kColStreams of them, then that of a stream which has finished. The others share the handle's scratch, as their
// tracing kernels do. Null while s is being captured: neither lives as long as a caller's graph.
// The null stream's buffer is its own for good. Others end a call by an event, 3 us on the GPU: a stream may be gone,
// or its name be another's, when the buffer is wanted next.
constexpr size_t kColStreams = 4;
struct ColBuffer;
class ColWork {
public:
    ColWork(const omg_geom* g, size_t floats, hipStream_t s, bool beside);
    ~ColWork();
    ColWork(const ColWork&) = delete;
    ColWork& operator=(const ColWork&) = delete;
    float* get() const { return p_; }

private:
    ColBuffer* buf_ = nullptr;
    float* p_ = nullptr;
    hipStream_t s_;
};

// `work`: col_work_floats of 16-byte aligned memory. timed: record the launches (omg_timing_enable).
// y = A img.
int col_forward(const omg_geom* g, const ColPlan* pl, int64_t first, int64_t n, const float* img, float* y, float* work,
                hipStream_t s);
// rhs += A^T y (y null: A^T 1); with sens also sens += A^T 1.
int col_backward(const omg_geom* g, const ColPlan* pl, int64_t first, int64_t n, const float* y, float* rhs, float* sens,
                 float* work, hipStream_t s);
// rhs += A^T (meas / (A img + epps (+ add))), NaN and Inf ratios -> epps; with sens also sens += A^T 1.
int col_osem(const omg_geom* g, const ColPlan* pl, int64_t first, int64_t n, const float* img, const float* meas,
             const float* add, float* rhs, float* sens, float epps, float* work, hipStream_t s, bool timed = true);

}  // namespace omg
