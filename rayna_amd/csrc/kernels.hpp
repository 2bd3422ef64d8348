// Interface between the host renderer and the wavefront kernels of kernels.hip.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layout.hpp"

namespace rayna {

// Path state of one chunk of samples, structure-of-arrays in HBM.  A chunk holds samples [s0, s0 + n_spp) of
// every pixel; slot i is sample s0 + i % n_spp of pixel i / n_spp, so a pixel's samples are neighbours (a wave
// traces 64 samples of one pixel, or all the samples of a few neighbouring pixels).
struct PathBuffers {
    float *ox, *oy, *oz;     // ray origin
    float *dx, *dy, *dz;     // ray direction (unit)
    float *tr, *tg, *tb;     // path throughput
    float *lr, *lg, *lb;     // radiance gathered so far; the sample's value once the path ends
    float *hit_t;            // closest-hit distance
    uint32_t *hit_ref;       // kind << 28 | index, 0 on a miss
    uint32_t *hit_aux;       // HIT_AUX_* bits; the object-space distance of a transformed object's hit
    uint32_t *hit_sub;       // an instance's hit: the reference of its primitive inside the instanced mesh BVH
    int32_t *hit_rank;       // optional (parity queries): rank of the closest primitive
    float *sdf_nx, *sdf_ny, *sdf_nz;  // scenes with unbounded objects: the shading normal of an SDF hit
};

struct FrameParams {
    GViewport vp;
    uint32_t width, height;
    uint32_t spp;            // samples per pixel of the frame
    uint32_t sdim;           // isqrt(spp): the stratified grid is sdim x sdim
    uint32_t key0, key1;     // Philox key
    uint32_t ray_depth;
    uint32_t n_pixels;
    uint32_t s0;             // first sample of the chunk
    uint32_t n_spp;          // samples per pixel in the chunk
    uint32_t n_slots;        // slots in the chunk: n_pixels * n_spp
    int32_t mode;            // RAYNA_MODE_*
    uint32_t *checks = nullptr;  // validation on: RAYNA_CHECKS violation counters (RAYNA_CHECK_*), else null
    uint32_t rays_stored = 0;    // k_generate stored this chunk's camera rays (else the first kernels compute them)
};

// One request of a batch, as seen by one chunk of paths: its slots are [slot_base, slot_base + n_slots), sample
// s0 + l % n_spp of pixel l / n_spp for local slot l (pixel-major, like a single frame).
struct RequestParams {
    GViewport vp;
    uint32_t width, height, spp, sdim;
    uint32_t key0, key1, ray_depth, n_pixels;
    uint32_t s0, n_spp, slot_base, n_slots;
    int32_t root, first_sdf, n_sdfs, skybox;  // the request's scene within the merged scene set
    int32_t sky_image;                        // RAYNA_SKY_HDRI: its image
    uint32_t sum_offset;                      // its 3 * n_pixels floats in the batch's sum and output buffers
    int32_t layout;                           // output layout (RAYNA_LAYOUT_*)
    uint32_t first_piece;                     // 1 if the chunk holds the request's first samples
};

// The requests of a batch chunk.  reqs == nullptr: a single frame described by FrameParams and SceneView.
struct BatchView {
    const RequestParams *reqs;
    uint32_t n_reqs;
    uint32_t *slot_req;  // request (index into reqs) of every slot, written by generate
};

// Inputs and outputs of the adjoint replay (path replay backpropagation) of a frame.
struct AdjointParams {
    const float *d_image;    // dloss/d(frame mean), 3 floats per pixel in row-major pixel order
    double inv_spp;          // 1 / samples per pixel: the share of each sample
    double *grad;            // copies x n_materials x 3 gradient accumulators
    uint32_t n_materials;
    uint32_t copies;         // gradient copies (a block adds into copy blockIdx % copies)
};

// Traversal tuning of the extend kernel: a wave takes new rays once `refill_lanes` of its lanes are idle,
// claiming `wave_batch` queue positions per atomic.
// packet_depths: the bounces (depth < packet_depths) traced as wave packets (k_extend_packet) where a chunk's
// samples of a pixel are neighbouring slots.
struct ExtendTuning {
    uint32_t refill_lanes = 32;
    uint32_t wave_batch = 128;
    uint32_t packet_depths = 1;
};

// Shade grid: blocks of 256 threads per compute unit (grid-stride over the queue).
constexpr int SHADE_BLOCKS_PER_CU = 16;

// The camera ray of every slot (the throughput and radiance fields are left as they are: the first shade takes
// them as 1 and 0, and the adjoint replay reads the primal radiance still held there).  With bv.reqs,
// fp.n_slots is the chunk's slot count and the requests come from bv.
void launch_generate(const FrameParams &fp, const PathBuffers &pb, const BatchView &bv, hipStream_t s);
// Claim counters of one k_extend or k_march launch: its work is cut into CLAIM_PARTS contiguous parts, each with its
// own counter, one 128-byte line apart, and on a line after them a word per part that is set once its last claim is
// taken (CLAIM_WORDS words in all, zeroed before the launch).
#ifndef RAYNA_CLAIM_PARTS
#define RAYNA_CLAIM_PARTS 4
#endif
constexpr uint32_t CLAIM_PARTS = RAYNA_CLAIM_PARTS;
constexpr uint32_t CLAIM_WORDS = (CLAIM_PARTS + 1) * 32;

// Deepest ray_depth that options may ask for.
constexpr uint32_t MAX_RAY_DEPTH = 1000;

// k_trace's counters of closest-hit queries, one 128-byte line apart (SEGMENT_WORDS words of 32 bits in all).  A wave
// adds to the counter of its block, so each holds what a whole chunk may come to: 2^32 paths to the depth limit.
using SegmentCounter = unsigned long long;
constexpr uint32_t SEGMENT_PARTS = 64;
constexpr uint32_t SEGMENT_STRIDE = 128 / sizeof(SegmentCounter);
constexpr uint32_t SEGMENT_WORDS = SEGMENT_PARTS * 32;
static_assert((SegmentCounter)-1 >> 32 >= MAX_RAY_DEPTH + 1, "a query counter may overflow");

// queue == nullptr: identity queue of fp.n_slots entries; else queue[0 .. *count)
// overflow: traversal stack entries beyond the LDS part, extend_block() * grid * (stack_need - extend_lds_stack());
// work: CLAIM_WORDS zeroed words, the counters the launch's waves take rays from
void launch_extend(const SceneView &sv, const FrameParams &fp, const PathBuffers &pb, const int32_t *queue,
                   const uint32_t *count, uint32_t depth, int grid, int2 *overflow, uint32_t *work,
                   const ExtendTuning &tune, const BatchView &bv, hipStream_t s);
// How many of a chunk's depths, from the camera rays on, get a launch of extend (and march) and one of shade each; the
// paths that are left go to their ends in one launch (launch_trace).  All depths (2^32 - 1) for the non-PBR modes and
// validation.
//
// Without unbounded objects: the camera rays where they are traced as packets, and for a large chunk over a tree that
// is not small the first bounce too: its rays start from one point per wave, which k_extend's seven waves per SIMD use
// better than k_trace's mix of depths.  (1080p, 64 samples, first bounce apart against not: 45.6 and 48.6 ms with
// 1.3 M triangles, 34.6 and 36.5 with 1290 (235 nodes), 28.2 and 28.3 with 480 spheres (40 nodes), 27.3 and 25.9 in the
// Cornell box; at 640x360x64, 8.04 and 7.99 ms with 1.3 M triangles.)  With media or instances k_trace has four waves
// per SIMD against k_extend's six, and the size of the tree does not matter: 521 spheres with a medium 1080p at 16, 33
// and 64 samples 12.0 and 12.6, 23.8 and 25.1, 45.8 and 48.4 ms, transformed objects 5.44 and 5.69, 10.5 and 11.4, 19.8
// and 21.7.  Without packets the camera rays are a launch of their own then as well, which pays later: RTTNW 1080p at 16,
// 33 and 64 samples, depth limit 10, 10.53 and 10.30, 19.8 and 20.4, 36.8 and 38.5 ms, depth limit 2, 6.44 and 6.40, 12.5
// and 12.8, 23.6 and 24.4.
//
// With unbounded objects: k_march's waves are full and each at one SDF, k_trace_sdf's do not wait for a depth's
// longest march.  So the largest chunks launch the camera rays and the first bounce, where most of the work is; small
// ones the camera rays, most of which march past everything; the smallest, where every launch is a wait, and those in
// between none.  The lines were drawn on the first of these scenes; device ms with 0, 1, 2 and all depths launched:
//                          64x36x2                 161x91x9                640x360x4               640x360x8
//   bulb, blobs, medium    3.19 3.50 3.87 6.11     4.52 4.55 5.03 8.79     7.24 6.33 7.06 11.2     9.64 7.40 7.88 12.8
//   the bulb alone         2.61 3.51 3.64 5.79     3.08 3.92 4.60 8.37     4.34 4.84 5.27 9.88     5.51 5.47 6.04 11.4
//   the blobs alone        0.65 0.98 1.16 1.44     1.13 1.80 2.25 3.63     1.60 2.22 2.87 4.83     2.28 2.62 3.42 5.74
//   60 bounded, a sphere   0.52 0.54 0.60 0.75     0.91 0.93 0.82 1.00     1.77 1.71 1.39 1.49     1.87 2.15 1.76 1.84
//                          640x360x24              640x360x64              1280x720x64             1280x720x128
//   bulb, blobs, medium    12.0 11.9 10.7 16.5     17.5 18.2 18.5 23.7     44.1 42.4 40.5 49.9     81.2 72.2 67.4 76.9
//   the bulb alone         7.19 7.42 8.12 14.6     9.79 12.0 12.6 19.3     22.0 23.5 24.4 34.3     36.9 37.9 40.6 52.8
//   the blobs alone        2.69 4.03 4.54 7.89     4.49 5.58 6.23 10.4     12.9 13.2 13.5 19.1     24.5 23.6 23.0 29.3
//   60 bounded, a sphere   2.44 2.78 2.65 2.53     3.83 4.59 4.89 4.87     12.2 13.5 13.0 13.9     24.0 25.5 24.0 25.6
// So between 2^14 and 2^21 paths a scene of one SDF would do better with no launch apart, and one of mostly bounded
// objects with two; the rule's choice is within 5% of a launch per depth or faster on all of them but the last at
// 320x180x8 and 640x360x4 and x8 (1.38 against 1.29, 1.71 against 1.49, 2.15 against 1.84).
//
// Of scenes that are all but nothing else than marches (at most MARCHED_NODES tree nodes), those of several unbounded
// objects leave a k_trace_sdf wave's lanes at different ones, so they launch the first bounce from fewer paths on
// (with 0 and 2 depths launched: two sets of blobs 640x360x16 7.0 and 5.9 ms, x64 13.2 and 11.0, 1280x720x32 20.7 and
// 16.5; six spheres 640x360x16 2.32 and 2.17, 1280x720x32 8.1 and 7.6; the bulb and the blobs 640x360x64 17.5 and 18.5,
// 1280x720x32 26.7 and 25.9: BULB_BOUNCE_SLOTS with a Mandelbulb, SDF_WHOLE_SLOTS without) and, where paths end after two
// or three vertices, every depth (with none and all launched, depth limits 0, 1 and 2: two sets of blobs 640x360x16 3.8
// and 1.9, 5.0 and 3.1, 5.6 and 4.0 ms; the bulb and the blobs 640x360x64 6.1 and 4.5, 7.9 and 7.5, 9.2 and 9.3,
// 1280x720x40 10.8 and 8.3, 15.6 and 12.5, 17.9 and 15.7).  Camera rays alone: one set of blobs 1280x720x40 6.1 and 5.7,
// the bulb 5.1 and 5.8.
//
// A batch's chunk of that size that mixes scenes with and without unbounded objects launches four depths: in one wave of
// k_trace_sdf a mesh's traversal stalls the marches and the other way round, where k_extend and k_march take each kind
// in full waves.  (64 requests of three scenes, two of them without SDFs, in chunks of up to 2^29 paths, three in flight,
// with 2, 3, 4 and all depths launched: shortest first 1972, 1844, 1760 and 1701 ms, in the order given 2115, 1956, 1871
// and 1799; 24 smaller requests in one chunk 74.1, 71.8, 71.0 and 76.9.)
constexpr uint32_t SDF_CAMERA_SLOTS = 1u << 14, SDF_WHOLE_SLOTS = 1u << 21, SDF_BOUNCE_SLOTS = 1u << 26;
constexpr uint32_t MIXED_DEPTHS = 4, BULB_BOUNCE_SLOTS = 3u << 23;
constexpr int32_t MARCHED_NODES = 4;
constexpr uint32_t FIRST_BOUNCE_SLOTS = 1u << 24;
constexpr uint32_t LANES_BOUNCE_SLOTS = 1u << 26;
constexpr int32_t FIRST_BOUNCE_NODES = 128;
uint32_t launched_depths(const SceneView &sv, const FrameParams &fp, const ExtendTuning &tune, const BatchView &bv);
// first_depth 0: every slot's path from its camera ray; first_depth > 0: the paths launch_shade kept at the depth before.
// The radiance field holds each path's radiance at the end.  overflow and work as for launch_extend; segments:
// SEGMENT_WORDS zeroed words, the closest-hit queries (launch_count_segments).
void launch_trace(const SceneView &sv, const FrameParams &fp, const PathBuffers &pb, const int32_t *queue,
                  const uint32_t *count, uint32_t first_depth, int grid, int2 *overflow, uint32_t *work,
                  SegmentCounter *segments, const ExtendTuning &tune, const AdjointParams *adjoint, const BatchView &bv,
                  hipStream_t s);
void launch_shade(const SceneView &sv, const FrameParams &fp, const PathBuffers &pb, const int32_t *queue_in,
                  const uint32_t *count_in, int32_t *queue_out, uint32_t *count_out, uint32_t depth, int grid,
                  const AdjointParams *adjoint, const BatchView &bv, hipStream_t s);
// The unbounded SDF objects of each queued path (n_sdf per path; in a batch, each request's own), marched
// after launch_extend with its hit as the cut, then merged into the hit record; the paths whose closest hit
// becomes an SDF get their shading normal in pb.sdf_n*.  mt: two planes of mt_stride >= count * n_sdf floats
// (outcome, march iteration).  work: CLAIM_WORDS zeroed words.  sdf_queue: room for every queued path; sdf_count: one
// zeroed counter.  No-op for n_sdf == 0.
void launch_march(const SceneView &sv, const FrameParams &fp, const PathBuffers &pb, const int32_t *queue,
                  const uint32_t *count, uint32_t n_sdf, float *mt, uint64_t mt_stride, uint32_t *work, int grid,
                  int merge_grid, const ExtendTuning &tune, const BatchView &bv, int32_t *sdf_queue,
                  uint32_t *sdf_count, hipStream_t s);
// Pixels per block of the resolve kernels for n samples per pixel in the chunk: a block stages its pixels'
// samples (three channels, rows of n | 1 floats) in LDS so that its loads are coalesced; from 1040 samples per
// pixel on, a block sums 256 pixels straight from HBM.  A small stage keeps many blocks per CU: the 1080p,
// 64-sample resolve took 0.459 ms with 4160 floats per channel, 0.324 with 2080, 0.279 with 1040.
constexpr uint32_t RESOLVE_STAGE = 1040;  // floats per channel
constexpr uint32_t resolve_pixels_per_block(uint32_t n) {
    return (n | 1u) > RESOLVE_STAGE ? 256u : (RESOLVE_STAGE / (n | 1u) > 256u ? 256u : RESOLVE_STAGE / (n | 1u));
}
// Batch chunks: per request, the running per-pixel sum of the chunk's samples (in sample order) and, at the
// request's last chunk, its sample mean in its layout at out + sum_offset.  blocks: the most resolve blocks of
// one request of the chunk (its pixels / resolve_pixels_per_block(its n_spp), rounded up).
void launch_resolve_batch(const BatchView &bv, uint32_t blocks, const PathBuffers &pb, float *sum, hipStream_t s);
void launch_finalize_batch(const BatchView &bv, const uint32_t *final_reqs, uint32_t n_final, uint32_t max_pixels,
                           const float *sum, float *out, hipStream_t s);
void launch_sum_grad(const double *grad, uint32_t n, uint32_t copies, double *out, hipStream_t s);
// The non-PBR render modes: the mode colour of each slot's camera ray (after launch_extend at depth 0) into
// its radiance field.
void launch_shade_mode(const SceneView &sv, const FrameParams &fp, const PathBuffers &pb, int grid, hipStream_t s);
// The UI's 8-bit conversion of a row-major float image (width * height * 3) to RGBA.
void launch_to_srgb8(const float *img, uint32_t n_pixels, uint8_t *rgba, hipStream_t s);
// A chunk's closest-hit queries, added to *segments (first: set): first_count, the lengths of queues 1 to n - 1 and the
// SEGMENT_PARTS counters of launch_trace.
struct SegmentCount {
    const uint32_t *queue_count;
    uint32_t n, first_count;
    const SegmentCounter *parts;
    unsigned long long *segments;
    uint32_t first;
};
// Where a frame's means go: the accumulation buffer (three planes; fresh: it holds nothing yet), and the image, the
// accumulated sum over `frames`.
struct FrameOutput {
    float *acc, *image;
    double frames;
    int32_t layout;  // RAYNA_LAYOUT_*
    uint32_t fresh;
};
// The chunk's samples added to the frame's per-pixel sums, and the chunk's queries counted.  out: the chunk is the
// frame's last, and its sums go to the output instead (launch_finalize is then not needed; it checks the pixels under
// validation, which this does not).
void launch_resolve(const FrameParams &fp, const PathBuffers &pb, float *sum, uint32_t chunk_samples, int first,
                    const SegmentCount &sc, const FrameOutput *out, hipStream_t s);
void launch_finalize(const FrameParams &fp, const float *sum, const FrameOutput &out, hipStream_t s);
void launch_fill_u32(uint32_t *p, uint32_t value, uint32_t n, hipStream_t s);
// Whether launch_extend traces this depth as wave packets (k_extend_packet).  At depth 0 of a single request the
// packets compute the camera rays themselves, so only the march and the non-PBR modes need k_generate's rays.
bool extend_packets(const SceneView &sv, const FrameParams &fp, const ExtendTuning &tune, const BatchView &bv,
                    uint32_t depth);
// The VALU issue-rate calibration kernel over `blocks` blocks of 256 lanes (out: one float per lane); returns
// the wave64 VALU instructions its chains issue (loop and set-up instructions not counted).
uint64_t launch_valu_peak(float *out, uint32_t blocks, uint32_t iters, hipStream_t s);
void launch_sqrt_check(uint32_t first, uint32_t count, unsigned long long *mismatches, uint32_t blocks, hipStream_t s);
void launch_count_segments(const SegmentCount &sc, hipStream_t s);

// The static workspace of rayna_adjoint_static (a file-scope device array of adjoint_scratch_doubles()
// doubles): its address on `device`, which must be the current device (taken on the first call per device).
hipError_t adjoint_scratch(int device, double **ptr);
size_t adjoint_scratch_doubles();

int extend_lds_stack();
int extend_blocks_per_cu();  // resident extend blocks per CU (the persistent grid is this times the CU count)
int extend_block();
int march_blocks_per_cu();
int march_block();

}  // namespace rayna
