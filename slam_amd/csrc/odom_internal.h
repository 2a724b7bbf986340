// odom_internal.h -- launchers of the HIP kernels (odom_kernels.hip), called by
// the host class (odom_host.cpp).  All launchers are asynchronous on `s`.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "odom_device.h"
#include "slam_odom.h"
#include "slam_splat.h"
#include "slam_surfel.h"

namespace slam {

// The statistics of the state last read back to the host (by odom_track,
// odom_get_pose or odom_get_stats), without a device round trip; for a caller
// that has just made one of those calls.  ODOM_ERR_ARG before any readback.
int odom_stats_last_read(odom_handle c, odom_stats* s);

// surfel_clean without its wait for the surfel count, for a caller that goes
// on enqueuing: until a surfel_* call that needs the count waits for it, the
// model has at most *upper surfels (those before and the new points), their
// number in device memory at *dev_count (which may exceed *upper where the
// buffer is full).
int surfel_clean_enqueue(surfel_handle c, const float pose[16], int time, float conf_threshold, int time_delta);
// The current model, its surfels (an upper bound) and, while a count is
// outstanding, the device's count (else null).
void surfel_model_enqueued(surfel_handle c, const float** dev_ptr, int* upper, const int** dev_count);
// splat_combined_predict of a device model of min(n, *dev_count) surfels.
int splat_predict_counted(splat_handle c, const float pose[16], const float* model, int n, const int* dev_count,
                          float depth_cutoff, float conf_threshold, int time, int max_time, int time_delta);

// The streams that the handles' work goes to.
hipStream_t surfel_stream(surfel_handle c);
hipStream_t splat_stream(splat_handle c);

// Launch shape of a step kernel at one level (replaces GPUConfig.h's
// threads/blocks table; chosen by the autotuner).
struct StepShape {
    int threads;    // 64, 128, 256 or 512
    int ppt;        // pixels per thread: 1, 2, 4, 8 or 16
};

// Kernel names and the shapes they support, for the autotuner.
int step_shape_supported(StepShape sh);

// ---- preprocessing (a1-a13) ----
void launch_bilateral(const uint16_t* src, int src_pitch, uint16_t* dst, int w, int h, float maxD,
                      hipStream_t s);
// depth pyramid -> vertex+normal maps of all levels in one launch
struct VNLevels {
    uint16_t* depth[kLevels];       // written by launch_depth_pyramid_maps (level 0 unless it is src)
    const uint16_t* src;            // level 0
    int src_pitch;                  // in elements
    float* vmap[kLevels];
    float* nmap[kLevels];
    int w[kLevels], h[kLevels];
    float fx_inv[kLevels], fy_inv[kLevels], cx[kLevels], cy[kLevels];
    float cutoff;
};
// initICP's depth levels from a.src and the three levels' vertex and normal
// maps, in one launch.
void launch_depth_pyramid_maps(const VNLevels& a, hipStream_t s);
// RGBA32F vertex/normal maps -> planar pyramids (copyMaps + resize, optional
// rigid transform), plus the vertex z plane kept for verticesToDepth.
struct ModelLevels {
    const float4* v4;
    const float4* n4;
    int v_pitch, n_pitch;           // in float4 elements
    float* vmap[kLevels];
    float* nmap[kLevels];
    int w[kLevels], h[kLevels];
    float* vz;                      // w0*h0 z values (may be null)
    int transform;
    float R[9], t[3];
    const float* pose_dev;          // if set: [R|t] (3x4 row-major) read on the device
};
void launch_model_maps(const ModelLevels& a, hipStream_t s);
// The three levels of up to two pyramids in one launch: a depth pyramid (a8,
// a9) from the vertex z plane `vz` (verticesToDepth, cutoff; float levels), or
// with vz null an intensity pyramid (a10, a11) from colour (rgb, pitch, ch;
// uint8 levels).
struct PyrSrc {
    const float* vz;
    float cutoff;
    const uint8_t* rgb;
    int pitch, ch;
    void* dst[kLevels];
};
struct PyrJob {
    PyrSrc p[2];
    int count;
    int w0, h0;
    TrackState* fresh;              // if set: a sequence starts (no motion yet, no SO3 failure)
};
void launch_pyramid(const PyrJob& j, hipStream_t s);
// derivatives (a12) + static photometric source mask, all levels of all pairs
struct PrepLevels {
    const uint8_t* img[kLevels];
    const float* depth[kLevels];
    short2* dxy[kLevels];
    float* zsrc[kLevels];
    int w[kLevels], h[kLevels];
    float minScale[kLevels];
};
void launch_rgb_prep(const PrepLevels& a, hipStream_t s);
// The same for every pair, G pixels of a row a thread; max_groups: the most
// groups of G that any pair has, per level.
void launch_rgb_prep_pairs(const PairDesc* pairs, int npairs, int G, const int max_groups[kLevels], hipStream_t s);
// G of a launch over so many level-0 pixels (1 or 4).
int rgb_prep_group_size(long long pixels);
// The pose (3x4 row-major) that the next call starts from.
void launch_set_pose(TrackState* st, const float pose[12], hipStream_t s);

// ---- tracking (a14-a21) ----
struct StepLaunch {
    const PairDesc* pairs;          // device array
    int npairs;
    const int* blk_pair;            // device table, per level (null when npairs == 1)
    int total_blocks;               // blocks of this level over all pairs
    long long pixels = 0;           // of this level over all pairs
    StepShape shape;
};
// SO3 pre-alignment; max_px_l2: largest level-2 pixel count over the pairs
// The SO3 loop; with begin, its last launch also does launch_track_begin's work.
// spin_limit < 0: one launch per iteration; else the one-launch loop (when
// the pairs fit), whose barrier waits give up after spin_limit polls.  With
// prep (one pair), launch_rgb_prep's work is done too: by extra blocks of the
// one-launch loop, or by a launch of its own before the per-iteration form.
void launch_so3(const PairDesc* pairs, int npairs, const TrackParams* begin, int spin_limit, hipStream_t s,
                const PrepLevels* prep = nullptr);
void launch_track_begin(const PairDesc* pairs, int npairs, const TrackParams& P, hipStream_t s);
// warm start: seed from the network prediction (6 floats per pair, device),
// optionally kept only when the level-2 ICP association is not worse than plain
void launch_seed_select(const PairDesc* pairs, int npairs, const float* pred, float t_scale, float r_scale,
                        int select, const TrackParams& P, hipStream_t s);
// network input (cnn_kernels.hip) from 160x120 level-2 buffers
void cnn_launch_prepare(const float* depth_a, const uint8_t* image_a, const uint16_t* depth_b, const uint8_t* image_b,
                        int n, size_t frame_stride, void* x, hipStream_t s);
// Gauss-Newton iteration k (global index over the call) at (level, iter).
// mode 0: tracking (the prologue finishes iteration k-1, which ran at
// prev_level); mode 1: parity pass with the constants of state slot 0,
// partials into parity 0 (totals by launch_reduce_dbg).
void launch_step_a(const StepLaunch& L, int level, int iter, int k, int prev_level, const TrackParams& P, int mode,
                   uint8_t* dbg_mask, hipStream_t s);
void launch_step_b(const StepLaunch& L, int level, int iter, int k, const TrackParams& P, int mode, hipStream_t s);
// Finish iteration k-1 and store the state of iteration k, one workgroup of
// `threads` (256 or 512: those of the pass A that follows) per pair
// (followed by launch_step_a with mode 1).
void launch_solve(const PairDesc* pairs, int npairs, int level, int iter, int k, int prev_level, const TrackParams& P,
                  int threads, hipStream_t s);
// Policy calls: the start of every entry (hyp entries per handle; the
// prediction or the constant-velocity extrapolation), and the judge of two
// refinements per handle (slot >= 0: after the coarse levels, from state
// slot `slot`; slot < 0: after the call).
void launch_seed_policy(const PairDesc* pairs, int nentries, int hyp, const float* pred, float t_scale, float r_scale,
                        hipStream_t s);
void launch_judge(const PairDesc* pairs, int nhandles, const TrackParams& P, int slot, int level, hipStream_t s);
// finishes the last iteration (K-1, at last_level), revert, result
void launch_track_end(const PairDesc* pairs, int npairs, const TrackParams& P, int K, int last_level, hipStream_t s);
// FP64 totals of a parity pass: which 0 = pass A (ICP sums, count, sigma), 1 = pass B
void launch_reduce_dbg(const PairDesc* pairs, int which, int level, hipStream_t s);
void launch_so3_step_dbg(const PairDesc* pairs, const float* consts27, double* out11, uint8_t* mask,
                         hipStream_t s);

// Constant tables of the kernels (the bilateral's spatial factors), per device.
void init_device_tables();

// Host copy of the device exp (same operation sequence): tables and tests.
float bexpf_host(float x);

}  // namespace slam
