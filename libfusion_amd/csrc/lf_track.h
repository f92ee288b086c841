// Device-resident Gauss-Newton tracking state shared by reduce.hip (kernels)
// and system.cpp (the host classes that sequence them).
#pragma once

#include <hip/hip_runtime.h>

#include "libfusion_amd.h"

// The Gauss-Newton state of a frame after one of its steps.
struct LfGnState {
    double est[12];        // current estimate T (reference camera -> current camera), 3x4 row-major
    float icp_error, rgb_error, stddev;
    float last_icp_error;  // icp error before the last step (last_icp_error of compute_transform(ctx))
    int icp_count, rgb_count;
    int active;            // 0 once the current level broke out of its loop
    int invalid;           // an error became NaN this frame
    int iterations;        // Gauss-Newton steps taken this frame
    int pad;
};

// A frame's pose for a reader that waits for nothing: record n is the state's record[n & 1],
// and a copy of one caught between its stores does not match its check.
struct LfPoseRecord {
    double pose[12];
    unsigned long long number;  // in the order of the frames (0: empty)
    unsigned long long check;
};
__host__ __device__ inline unsigned long long lf_pose_check(const LfPoseRecord &r) {
    unsigned long long h = 0;  // an empty record's
    for (int k = 0; k < 12; ++k) {
        h = (h ^ __builtin_bit_cast(unsigned long long, r.pose[k])) * 0x9E3779B97F4A7C15ull;
        h ^= h >> 29;
    }
    h = (h ^ r.number) * 0x9E3779B97F4A7C15ull;
    return h ^ h >> 32;
}

// One tracker's state in device memory.  Poses are 3x4 row-major doubles.
struct LfTrackState {
    LfGnState gn;        // after the last step that was taken
    LfGnState slot[2];   // after step k - 1, in slot k & 1: read by step k's launch while it writes the other
    double prev[12];     // Revertable<SE3d>::prev (revertable.h:7-45)
    double init[12];     // initial estimate (identity in DenseOdometry)
    int success;         // result of the last finished frame
    int pad;
    // odometry chain (DenseOdometry::trackFrame, rgbd_odometry.cpp:18-48)
    double pose[12];     // T_world_camera of the current frame
    float pose24[24];    // float T_world_camera and T_camera_world for the mapping kernels
    LfPoseRecord record[2];  // pose after the last frame and the one before it (of a batch's systems)
    // the last Gauss-Newton step's FP64 sums: A = w H_icp + H_rgb and b in
    // create_jtjjtr<6,7> order (0-26), ICP r^2 / count (27 / 28), RGB r^2 /
    // count (29 / 30)
    double sums[32];
};

// Per-level inputs of one tracking iteration.
struct LfTrackLevel {
    const float *curr_vmap, *curr_nmap, *last_vmap, *last_nmap;
    const float *curr_I, *last_I, *dIdx, *dIdy;
    int cols, rows;
    lf_intrinsics K;
    int half_maps;  // the maps hold FP16 (nmap 4 x FP16, intensity and gradients FP16; vmaps stay float4)
};

// Scratch floats needed by the stand-alone reductions and by a tracker's steps
// (partial rows of the workgroups).
size_t lf_reduce_partials(void);
size_t lf_track_scratch_floats(void);

// Schedule position of one Gauss-Newton step within a tracked frame.
struct LfStepFlags {
    int step;                 // index within the frame; 0 starts the estimate at init (replaces lf_track_begin)
    int end;                  // the launch after the last step: its solve and lf_track_finish
    int first_of_level;       // first iteration of a pyramid level (resets the error history)
    // the step before
    int prev_first_of_level;
    int prev_grid;            // its workgroups
    int context_mode;         // compute_transform(ctx) (icp_tracker.cpp:210-314): NaN errors are not
                              // flagged and the finish always succeeds with update = estimate^-1
    unsigned long long record;  // number of the frame's pose record (0: none is written)
    double init[12];          // initial estimate, 3x4 row-major (step 0)
};

// One Gauss-Newton iteration of DenseTracking::compute_transform
// (icp_tracker.cpp:50-140) in one launch, entirely on the device: the previous
// step's sums, FP64 solve, SE3 update and divergence checks, then this step's
// fused ICP + RGB reduction.  A frame is its steps in order and one launch with end set.
// scratch: lf_track_scratch_floats().  *grid: the workgroups used.
int lf_track_step(const LfTrackLevel &lv, float *scratch, LfTrackState *st, const LfStepFlags &f, float icp_weight,
                  hipStream_t stream, int *grid);
// Start a frame's estimate at T (3x4 doubles, host): est = prev = init = T.
// Only needed when a frame schedules no step.
int lf_track_begin(LfTrackState *st, const double *T12, hipStream_t stream);
// End of a tracked frame: success test, update = est^-1 (or identity), chain the
// odometry pose and refresh pose24.  Only needed when a frame schedules no step.
int lf_track_finish(LfTrackState *st, unsigned long long record, hipStream_t stream);
// Set the odometry pose directly (first frame / restart): T given as 3x4 doubles (host).
int lf_track_set_pose(LfTrackState *st, const double *T12, unsigned long long record, hipStream_t stream);
// The state into pinned host memory (there once the stream has come this far).
int lf_track_read(const LfTrackState *st, LfTrackState *host, hipStream_t stream);

// Batched tracking: one step of several systems in one launch.  A job is
// the launch arguments of one system's step (lf_track_job_bytes each);
// lf_track_job_make fills one and reports its grid, lf_track_job_skip marks a
// system with nothing at this index.  lf_track_batch_step runs step jobs[0..n)
// (device memory) with a grid of gmax workgroups per system (the largest job
// grid).  A job made with share n takes 1/n of the resident workgroups (at
// least one), so n systems together fill the grid once; each lane then sums
// several pixels, and the system's sums equal lf_track_step's up to FP64
// summation order (exactly, for share 1).
// The jobs of one batch share one map format (half_maps as in their LfTrackLevel).
size_t lf_track_job_bytes(void);
// share: systems sharing the launch (the job's grid is 1/share of a lone
// system's); wgs > 0 sets the grid instead.
int lf_track_job_make(const LfTrackLevel &lv, float *scratch, LfTrackState *st, const LfStepFlags &f,
                      float icp_weight, int share, int wgs, void *job, int *grid);
void lf_track_job_skip(void *job);
int lf_track_batch_step(const void *jobs, int n, int gmax, int half_maps, hipStream_t stream);
// The end jobs of n systems (made with end set), whatever their numbers of steps.
int lf_track_batch_end(const void *jobs, int n, hipStream_t stream);
