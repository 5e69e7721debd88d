// Kernel-side types and launch declarations shared by kernels.hip and the
// host runtime (runtime.hip).
#pragma once

#include "xt_device.h"
#include "xt_guide.h"

namespace xt {

#ifndef XT_TRACE_BLOCK
#define XT_TRACE_BLOCK 256
#endif
#ifndef XT_TRACE_LDS_DEPTH
#define XT_TRACE_LDS_DEPTH 16
#endif
#ifndef XT_SHADE_BLOCK
#define XT_SHADE_BLOCK 512
#endif
constexpr int SHADE_BLOCK = XT_SHADE_BLOCK;          // threads per block of the shade kernel
// Guided and normal-mapped shading, long for every vertex, takes blocks of half
// the size, whose waves wait less for each other at the appends (512 -> 256:
// guided room 7700 -> 7461 us, normal-mapped plane 6768 -> 6634).  The plain
// forms would pay more for twice the atomics on the queue lengths, which are
// served one after another (Cornell box 1235 -> 1293 us, room 10853 -> 10600).
__host__ __device__ constexpr int shade_block(bool guide, bool nmap) { return guide || nmap ? SHADE_BLOCK / 2 : SHADE_BLOCK; }
constexpr int TRACE_BLOCK = XT_TRACE_BLOCK;          // lanes per block of the traversal kernels
constexpr int TRACE_LDS_DEPTH = XT_TRACE_LDS_DEPTH;  // LDS stack entries per lane
// queue length (an upper bound the host knows) from which the traversal
// kernels hand out rays in chunks from a cursor (DYN, xt_traverse.h)
#ifndef XT_TRAV_DYN_MIN
#define XT_TRAV_DYN_MIN (8u << 20)
#endif
constexpr uint32_t TRAV_DYN_MIN = XT_TRAV_DYN_MIN;

// Where the current batch lies in the render: pixel range, paths, first
// sample.  Host-driven renders pass it in WaveParams; graph replays read it
// from device memory (WaveParams::cursor), advanced by k_advance_cursor.
struct BatchCursor {
    uint32_t first_pixel, num_pixels;
    uint32_t num_paths;
    uint32_t sample0;      // global index of the batch's first sample
    uint32_t s_rel;        // the same, counted from the render's first sample
};

// Per-batch constants of the wavefront pipeline.
struct WaveParams {
    uint32_t width, height;
    uint32_t first_pixel, num_pixels;   // pixel range of the batch
    uint32_t num_paths;                 // num_pixels * samples in the batch
    uint32_t sample0;                   // global sample index of the batch's first sample
    uint32_t seed, stream;
    uint32_t integrator, flags;
    int32_t max_depth, rr_start;
    float rr_prob, eps, shadow_margin;
    float tan_x, tan_y;
    float cam[16];
    const BatchCursor* cursor;          // non-null: the batch fields above are read from here
};

__device__ __forceinline__ BatchCursor batch_of(const WaveParams& wp) {
    if (wp.cursor) return *wp.cursor;
    return BatchCursor{wp.first_pixel, wp.num_pixels, wp.num_paths, wp.sample0, 0u};
}

// Batch schedule of one render: S samples of pix_chunk pixels per batch.
struct BatchPlan {
    uint32_t npix, pix_chunk, S, spp, spp_offset;
};

// Extension-ray queue, SoA of float4 (64 B per entry):
//   o = (origin, pdf of the BSDF sample that made the ray; -1 = delta)
//   d = (direction, path id)
//   w = (path weight, vertex index v | flags << 24)   v = vertex the ray will hit (1 = camera hit)
//   e = (material_eval of the sample, env-light pdf of the direction)
//   rec = training-record index of the vertex that sampled the ray (INVALID: none);
//         only touched while training records are kept
struct PathQueue {
    float4* o;
    float4* d;
    float4* w;
    float4* e;
    uint32_t* rec;
};
// Queue lengths, four words: 2 k is the length of path queue k, 2 k + 1 that of
// the shadow queue filled beside it.  A pair is one 64-bit counter to the shade
// kernel, which appends to both with one atomic.
__host__ __device__ __forceinline__ uint32_t* path_count(uint32_t* counts, int k) { return counts + 2 * k; }
__host__ __device__ __forceinline__ uint32_t* shadow_count(uint32_t* counts, int k) { return counts + 2 * k + 1; }
__host__ __device__ __forceinline__ unsigned long long* pair_count(uint32_t* counts, int k) {
    return (unsigned long long*)(counts + 2 * k);
}
constexpr uint32_t QF_PENDING = 1u;   // the previous vertex's NEE result waits in pending[id]

// Shadow-ray queue (48 B per entry):
//   o = (origin, tmax), d = (direction, path id), c = (contribution, mode: 1 = store to pending)
struct ShadowQueue {
    float4* o;
    float4* d;
    float4* c;
};

// Per-vertex training record written while rendering (96 B, six float4):
//   a = (p.xyz, n.x)  b = (n.yz, wo.xy)  c = (wo.z, dir.xyz)
//   d = (pdf, W.xyz)  e = (E.xyz, path id | 1 << 31 if the vertex was guided)
//   f = (pre.xyz, 0)
// p, n, wo: the query; dir and pdf: the sampled direction and its strategy
// pdf; W: path throughput before the vertex; E: the vertex's sample weight
// f cos / pdf; pre: the path radiance collected up to and including the
// vertex's own light sample (written when the next vertex is shaded).
// After the path ends, C = (L_path - pre) / W is the vertex's estimate of
// f cos L_i / pdf along dir, and L_i = C / E.
struct TrainRec {
    float4 a, b, c, d, e, f;
};
constexpr uint32_t TREC_GUIDED = 1u << 31;

// Decoded mixture per path-queue entry, SoA per lobe j:
// lobes_mk[j * stride + i] = (mu, kappa) as four halves, lobes2[j * stride +
// i] = (alpha, alpha * vmf_norm(kappa)) in fp32 with kappa the stored half
// value; 128 bytes per entry.  Readers renormalise mu, so sampling and pdf
// see the same distribution.
constexpr int G_LOBE_FIELDS = 4 * G_LOBES;
__host__ __device__ __forceinline__ uint32_t pack_half2(float a, float b) {
    const _Float16 ha = (_Float16)a, hb = (_Float16)b;
    return (uint32_t)__builtin_bit_cast(uint16_t, ha) | ((uint32_t)__builtin_bit_cast(uint16_t, hb) << 16);
}
__host__ __device__ __forceinline__ float half_lo(uint32_t v) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(v & 0xFFFFu)); }
__host__ __device__ __forceinline__ float half_hi(uint32_t v) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(v >> 16)); }
// (normalised mu, kappa) of one stored lobe
__host__ __device__ __forceinline__ float4 unpack_lobe(uint2 v) {
    const f3 mu = normalize(mk(half_lo(v.x), half_hi(v.x), half_lo(v.y)));
    return make_float4(mu.x, mu.y, mu.z, half_hi(v.y));
}

struct GuideRender {
    const uint2* lobes_mk; // null: guiding off
    const float2* lobes2;
    uint32_t stride;
    float prob;            // probability of sampling the guide (one-sample MIS with the BSDF)
    TrainRec* recs;        // null: no training records
    uint32_t rec_base;     // record index of this bounce's first queue entry
    uint32_t rec_cap;
    uint32_t max_vertex;   // guide surface vertices 1..max_vertex only (0: all)
};

// ---- unified batches: many renders (items) share one wavefront
//
// The items' paths are numbered one after another (item k owns
// [path_base, path_base + paths), sample-major inside the item as a single
// render numbers them); the batch walks that path space in windows of up to
// `window` paths, each window one pass of the count-driven bounce loop.  A
// queue entry's path id is window-relative; item_of[id] names its item, whose
// record gives the render's parameters, scene and film.

struct MultiItem {
    WaveParams wp;          // the render's parameters (the batch fields are unused)
    const float4* nodes;    // its scene's BVH nodes and leaf-ordered triangles
    const float4* tris;
    uint32_t scene;         // index into MultiBatch::scenes
    uint32_t npix;          // width * height
    uint32_t spp_offset;
    uint32_t film_f64;
    void* film;             // device film (+= radiance sums, as xt_render)
    uint64_t path_base;     // first path of the item in the batch
    uint64_t paths;         // npix * spp
};

// The current window and the items it overlaps (written by k_window_plan).
struct MultiCursor {
    uint64_t g0;            // first path of the window
    uint32_t n;             // paths in the window (0: past the end)
    uint32_t first_item;    // first item overlapping the window
    uint32_t num_overlap;   // items overlapping the window
    uint32_t pad;
};

struct MultiBatch {
    const MultiItem* items;
    const DevScene* scenes;
    uint32_t num_items;
    uint32_t window;
    uint64_t total_paths;
    MultiCursor* cursor;
    uint32_t* item_of;      // per path of the window
    uint32_t* units;        // window plan: accumulation units before each overlapping item (num_overlap + 1)
};

template <bool ANY, int LDS_DEPTH, bool COUNT, bool MULTI = false, bool DYN = false>
__global__ void k_trace(DevScene sc, const float4* ray_o, const float4* ray_d, int ray_stride,
                        const uint32_t* count_ptr, uint32_t count_fixed, float4* hits, uint8_t* occluded,
                        int hit_prim_ids, int tmax_from_ray, uint32_t* ovf, uint32_t* dyn,
                        unsigned long long* visit_totals,
                        uint32_t* clear_a, uint32_t* clear_b, const uint32_t* item_of = nullptr,
                        const MultiItem* items = nullptr);
template <bool DYN>
__global__ void k_shadow_multi(ShadowQueue sq, const uint32_t* count, float4* radiance, float4* pending, uint32_t* ovf,
                               uint32_t* dyn, const uint32_t* item_of, const MultiItem* items);
template <bool MULTI, bool DYN>
__global__ void k_trace_shadow(DevScene sc, const float4* ray_o, const float4* ray_d, float4* hits, ShadowQueue sq,
                               uint32_t* counts, int cur, float4* radiance, float4* pending, uint32_t* ovf, uint32_t* dyn,
                               uint32_t* counts_out, const uint32_t* item_of = nullptr, const MultiItem* items = nullptr);
__global__ void k_window_init(MultiBatch mb);
__global__ void k_window_plan(MultiBatch mb);
__global__ void k_window_advance(MultiBatch mb);
__global__ void k_count_from_window(uint32_t* count, const MultiCursor* c);
__global__ void k_generate_multi(MultiBatch mb, PathQueue q, float4* radiance);
template <bool NMAP>
__global__ void k_shade_multi(MultiBatch mb, PathQueue qin, const uint32_t* count_in, const float4* hits,
                              PathQueue qout, unsigned long long* counts_out, ShadowQueue sq,
                              float4* radiance, float4* pending);
template <bool NMAP>
__global__ void k_shade_multi_open(MultiBatch mb, PathQueue qin, const uint32_t* count_in, const float4* hits,
                                   PathQueue qout, unsigned long long* counts_out, ShadowQueue sq, float4* radiance,
                                   float4* pending);
__global__ void k_accumulate_multi(MultiBatch mb, const float4* radiance);

// Arguments of k_walk.  MULTI uses mb, the others wp and scene; QUEUE (paths
// taken up in mid-flight) uses q, count and pending, the others number the
// paths of the batch or window themselves.
struct WalkArgs {
    WaveParams wp;
    const DevScene* scene;
    MultiBatch mb;
    PathQueue q;
    const uint32_t* count;
    const float4* pending;
    float4* radiance;
    uint32_t lanes;                 // rays a wave keeps in flight (1..64)
    uint32_t* ovf;                  // traversal spill columns
    uint32_t* dyn;                  // chunk cursor and block counter, zero between launches
    uint32_t max_vertex = 0xFFFFFFFFu;   // a path that goes on past it is left there and sets *overrun
    uint32_t* overrun;              // null: the depth cap ends every path
    unsigned long long* rays;       // null, or running totals of extension and shadow rays
    unsigned long long* rays_out;   // where the launch leaves them, and *overrun (mapped host memory)
};
// waves per SIMD of k_walk (at 3 instead of 4, with no spill instead of 28
// registers', it measured the same; the normal-mapping form needs 256 VGPRs)
constexpr int WALK_WAVES = 4, WALK_WAVES_NMAP = 2;
// Most paths of a batch that are walked instead of queued.  A walked path costs
// the longest of its wave's rays at every vertex, a queued one its share of two
// launches per round; where a batch has few paths the launches, their gaps and
// the slowest ray of each cost more.  Walked paths are best as many as there are
// lanes for, 262,144 (131,072 with normal maps, whose lanes then take two each):
// beyond, waves begin again with full-length paths.  Walked / queued us, at 229 k,
// 262 k, 328 k paths: 100 k triangle room (depth 16) 2240 / 2425, 2260 / 2410, 3180 /
// 2840; Cornell box (depth 8) 530 / 587, 537 / 594, 794 / 692; material zoo 861 / 863,
// 875 / 865, 1180 / 982; 0.5 M triangle canyon under a sky 1450 / 1494, 1529 / 1529,
// 1930 / 1702; with normal-mapped materials room 3257 / 3273, 3330 / 3340, 4350 /
// 3440, Cornell box 766 / 803, 774 / 811, 990 / 886.
// In an open scene (scene_open) most paths leave early, and later ones fill
// their lanes.  Walked / queued at 328 k, 461 k, 655 k: 0.5 M triangle field 562 /
// 922, 776 / 993, 970 / 1118, with depth 20 442 / 777, 550 / 821, 660 / 916; object in
// a lat-long sky 444 / 598, 454 / 617, 533 / 676; normal-mapped plane 785 / 993 at
// 328 k, 1060 / 1150 at 459 k, 1176 / 1248 at 524 k, 1468 / 1354 at 590 k.
// Without a depth cap the last paths go on for many rounds: at 328 k, 459 k,
// 590 k, 655 k Cornell box 1332 / 1350, 1545 / 1573, 1734 / 1752, 1821 / 1884; zoo
// 2168 / 2235, 2405 / 2544, 2651 / 2810, 2788 / 2916; room 4960 / 5277, 5970 / 6002,
// 6670 / 6650, 7015 / 6975 (8800 / 8106 at 922 k); with normal-mapped materials Cornell
// box 1556 / 1582, 1917 / 1744, room 6270 / 6010, 7605 / 6910.
constexpr uint32_t WALK_MAX = 4u << 16;
constexpr uint32_t WALK_MAX_OPEN = 10u << 16, WALK_MAX_OPEN_NMAP = 8u << 16;
constexpr uint32_t WALK_MAX_UNCAPPED = 10u << 16, WALK_MAX_UNCAPPED_NMAP = 5u << 16;
// Paths of a queue that are walked to their ends instead of queued on: the
// last rounds of a large batch (material zoo at 460 k paths, us: 1782 from
// 32 Ki, 1646 from 128 Ki, 1577 from 256 Ki, 1519 from 384 Ki; 100 k triangle
// room at 460 k: 3326, 3328, 3272, 3671).
constexpr uint32_t WALK_TAIL = 1u << 18;
// Waves that few paths are spread over, by leaving lanes empty: a wave's step
// takes as long as the slowest of its rays, so 6 k paths ran in 735 us at 64
// paths a wave and in 545 / 427 / 413 / 406 us over 512 / 1024 / 2048 / 4096
// waves (before paths had two lanes).
constexpr uint32_t WALK_SPREAD = 2048;
// Paths up to which a wave holds at most 32, each with a second lane for its
// shadow ray: as many as 4 waves per SIMD hold.  100 k triangle room, us, one
// lane a path against two: 14 k paths 1111 / 757, 57 k 1763 / 1053, 115 k 2000 /
// 1364; at 230 k, where two lanes a path need twice the waves, 2220 / 2347.
constexpr uint32_t WALK_PAIRS = 1u << 17;
template <bool QUEUE, bool NMAP, bool MULTI>
__global__ void k_walk(WalkArgs a);

__global__ void k_generate(WaveParams wp, PathQueue q, float4* radiance);
template <bool DYN>
__global__ void k_trace_camera(DevScene sc, WaveParams wp, float4* hits, uint32_t* ovf, uint32_t* dyn,
                               unsigned long long* clear);
template <bool GUIDE, bool NMAP, bool SORT, bool FIRST>
__global__ void k_shade(WaveParams wp, const DevScene* scene, PathQueue qin, const uint32_t* count_in, const float4* hits,
                        PathQueue qout, unsigned long long* counts_out, ShadowQueue sq,
                        float4* radiance, float4* pending, GuideRender gr);
template <bool NMAP>
__global__ void k_shade_open(WaveParams wp, const DevScene* scene, PathQueue qin, const uint32_t* count_in,
                             const float4* hits, PathQueue qout, unsigned long long* counts_out, ShadowQueue sq,
                             float4* radiance, float4* pending, GuideRender gr);
template <bool COUNT, bool DYN = false>
__global__ void k_shadow(DevScene sc, ShadowQueue sq, const uint32_t* count, float4* radiance, float4* pending,
                         uint32_t* ovf, uint32_t* dyn, unsigned long long* visit_totals, const uint32_t* counts4,
                         uint32_t* counts_out);
__global__ void k_accumulate(WaveParams wp, const float4* radiance, void* film, int film_f64, const uint32_t* overrun);
__global__ void k_zero_u32(uint32_t* p, uint32_t n);
constexpr int VALU_PROBE_CHAINS = 16;   // FMA chains per lane of k_valu_probe
__global__ void k_valu_probe(uint32_t iters, float* out);
__global__ void k_cursor_init(BatchCursor* c, BatchPlan plan, uint32_t* dyn);
__global__ void k_advance_cursor(BatchCursor* c, BatchPlan plan);
__global__ void k_count_from_cursor(uint32_t* count, const BatchCursor* c);

}  // namespace xt
