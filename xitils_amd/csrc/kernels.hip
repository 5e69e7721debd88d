// gfx950 kernels: ray queries and the wavefront path tracer.
//
// Wavefront pipeline per batch of paths (one path = one pixel sample):
//   extend (camera rays) -> shade -> [extend + shadow -> shade]* -> accumulate
// (guided and counting renders begin with generate; a batch of few paths, or
// a large one's last, is one launch: k_walk)
// extend  : closest hit for every queued ray         (Scene::intersect, Scene.h:30)
// shade   : one StandardPathTracer / NaivePathTracer loop step
//           (PathTracer.h:147-246 / 65-101): emission at the new vertex,
//           roulette, BSDF sample -> next queue, light sample -> shadow queue
// shadow  : any hit for every shadow ray             (Scene::intersectAny, Scene.h:34)
// Queues are compacted with one atomic per block for both (wave
// ballots + an LDS prefix); per-wave atomics on the two queue counters were
// the shade kernel's bottleneck.
// Radiance is kept per path id and summed in the reference's order (BSDF-hit
// emission of vertex v+1 before the light sample of vertex v), so the image
// does not depend on queue order.
#include "kernels.h"
#include "xt_traverse.h"
#include "xt_nmap.h"

namespace xt {

// Block-aggregated appends to two queues at once (extension and shadow): one
// 64-bit atomic per block on the pair of their lengths (low and high word).
// Every block's atomics go to the same two words and are served one after
// another.  Against an atomic per queue, shade launches of queues that stay in
// the caches: 40.4 -> 34.7 us (Cornell box, 1 M paths), 172 -> 165 (100 k
// triangle room, 3.7 M); of 100 M paths, bound by memory: no change.
// Every thread of the block must call it (the callers' loops are
// block-uniform).  Returns this thread's slots (valid when its predicate is
// set).
template <int BLOCK>
__device__ __forceinline__ uint2 block_append2(unsigned long long* counters, bool pa, bool pb,
                                               uint32_t* sh /* 2 * (BLOCK / 64) + 2 words of LDS */) {
    constexpr int NW = BLOCK / 64;
    const uint64_t ma = __ballot(pa), mb = __ballot(pb);
    const uint32_t wave = threadIdx.x / 64, lane = __lane_id();
    const uint64_t below = (1ull << lane) - 1ull;
    if (lane == 0) {
        sh[wave] = (uint32_t)__popcll(ma);
        sh[NW + wave] = (uint32_t)__popcll(mb);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t ta = 0, tb = 0;
        for (int w = 0; w < NW; ++w) {
            uint32_t ca = sh[w], cb = sh[NW + w];
            sh[w] = ta;
            sh[NW + w] = tb;
            ta += ca;
            tb += cb;
        }
        const unsigned long long both = (unsigned long long)ta | ((unsigned long long)tb << 32);
        const unsigned long long at = both ? atomicAdd(counters, both) : 0ull;
        sh[2 * NW] = (uint32_t)at;
        sh[2 * NW + 1] = (uint32_t)(at >> 32);
    }
    __syncthreads();
    uint2 r = make_uint2(sh[2 * NW] + sh[wave] + (uint32_t)__popcll(ma & below),
                         sh[2 * NW + 1] + sh[NW + wave] + (uint32_t)__popcll(mb & below));
    __syncthreads();   // sh is reused by the next iteration
    return r;
}

// VALU issue probe: VALU_PROBE_CHAINS independent fp32 FMA chains per lane
// (one VALU instruction per step, enough independent work to cover the FMA
// latency at 8 waves per SIMD) and no memory traffic; `out` is written only
// if the sums take a value they never take, which keeps the chains live.
__global__ __launch_bounds__(256) void k_valu_probe(uint32_t iters, float* out) {
    float a[VALU_PROBE_CHAINS];
#pragma unroll
    for (int k = 0; k < VALU_PROBE_CHAINS; ++k) a[k] = 1.0f + 1e-6f * (float)(threadIdx.x + 64 * k);
    for (uint32_t i = 0; i < iters; ++i) {
#pragma unroll
        for (int k = 0; k < VALU_PROBE_CHAINS; ++k) a[k] = __builtin_fmaf(a[k], 0.9999999f, 1e-7f);
    }
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < VALU_PROBE_CHAINS; ++k) sum += a[k];
    if (sum == -1.0f) out[blockIdx.x] = sum;
}

__global__ void k_zero_u32(uint32_t* p, uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// ---------------------------------------------------------------- ray queries

// Adds a wave's visit counts to the 64-bit totals (counting build only).
__device__ __forceinline__ void flush_counts(unsigned long long* totals, const VisitCount& vc) {
    unsigned long long a = vc.nodes, b = vc.tris;
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off);
        b += __shfl_xor(b, off);
    }
    if (__lane_id() == 0) {
        atomicAdd(&totals[0], a);
        atomicAdd(&totals[1], b);
    }
}

// The loop of the traversal kernels: the rays of `ch` (and, DYN, of the cursor
// `dyn`) by persistent waves with in-place lane refill.  load(i) sets up ray i
// in r and t, finish(i, occluded) takes its result out of t.
template <bool ANY, int LDS_DEPTH, bool COUNT, bool DYN, class SV, class Load, class Finish>
__device__ __forceinline__ void trace_queue(RayChunks ch, uint32_t* dyn, const SV& sv, const RayPre& r, Trav& t,
                                            const float4* top, uint32_t* my_lds, uint32_t* my_ovf, size_t nthreads,
                                            VisitCount& vc, Load load, Finish finish) {
    const uint64_t below = (1ull << __lane_id()) - 1ull;
    uint32_t rid = INVALID;   // the lane's ray; INVALID: none
    while (true) {
        const uint64_t busy = wave_ballot(rid != INVALID);
        const uint32_t nidle = 64u - wave_count(busy);
        if (nidle >= (uint32_t)REFILL_IDLE) {
            if (DYN && ch.next >= ch.end && !ch.exhausted) chunks_refill(ch, dyn);
            if (ch.next < ch.end) {
                const uint32_t my = ch.next + (uint32_t)__popcll(~busy & below);
                if (rid == INVALID && my < ch.end) {
                    rid = my;
                    load(rid);
                }
                ch.next = min(ch.next + nidle, ch.end);
            } else if (busy == 0) {
                break;
            }
        }
        const bool active = rid != INVALID;
        bool occ = false;
        const bool done = trav_step<ANY, LDS_DEPTH, COUNT, DYN>(active, sv, r, t, top, my_lds, TRACE_BLOCK, my_ovf, nthreads, vc, &occ);
        if (active && done) {
            finish(rid, occ);
            rid = INVALID;
        }
    }
}

// A closest-hit ray's entry of the hit queue.
__device__ __forceinline__ float4 hit_record(const Trav& t, uint32_t id) {
    return t.best_slot != INVALID ? make_float4(t.best_t, __uint_as_float(id), t.b0, t.b1)
                                  : make_float4(INFINITY, __uint_as_float(INVALID), 0.0f, 0.0f);
}

// What a shadow ray adds: unoccluded contributions go straight to the path
// radiance, or to pending[] when the path continues (see k_shade).
__device__ __forceinline__ void shadow_record(const ShadowQueue& sq, uint32_t i, bool occ, float4* radiance, float4* pending) {
    const float4 c4 = sq.c[i];
    const uint32_t id = __float_as_uint(sq.d[i].w);
    const f3 c = occ ? splat(0.0f) : xyz(c4);
    if (c4.w != 0.0f) {
        pending[id] = f4(c, 0.0f);
    } else if (!occ) {
        radiance[id] = f4(xyz(radiance[id]) + c, 0.0f);
    }
}

// Ray queries over a ray array (stride in float4 between rays): closest hit
// (ANY = false) -> hits[i] = (t, slot or prim id, b0, b1); any hit ->
// occluded[i].  Persistent waves with in-place lane refill (xt_traverse.h).
// MULTI: the rays of a unified batch's queue, each traced in its own item's
// scene (item_of[path id] -> the item's nodes and triangles, per lane).
// Bounded to 8 waves per SIMD, which every form but the chunked multi-scene
// one (7, where 8 spills two registers) reaches without spilling.
//
// Bound by VALU issue, and for any hit by L1 accesses too: a node visit is some
// 180 VALU instructions and 4 loads, and the kernel issued 0.76-0.84 G
// wave-instructions per ms where independent FMAs reach 0.81-0.88.  Lane state
// kept as masks and counts in scalar registers (the ray id tells an idle lane),
// the outward push one fma a plane, child counts from the sort's masks and
// stack reads that stay LDS reads: 1080p field 62.8 -> 61.3 ms a frame, 100 k
// triangle room 12.85 -> 12.46, 16 rooms batch 4.07 -> 3.84, bounce-ray query
// 437 -> 427 us.  (Grid steps held as whole floats in the nodes' spare words:
// 1% faster frames, but the bounce-ray query 450 us.)
template <bool ANY, int LDS_DEPTH, bool COUNT, bool MULTI, bool DYN>
__global__ __launch_bounds__(TRACE_BLOCK, DYN && MULTI ? 7 : 8) void k_trace(DevScene sc, const float4* __restrict__ ray_o,
                                                        const float4* __restrict__ ray_d, int ray_stride,
                                                        const uint32_t* __restrict__ count_ptr, uint32_t count_fixed,
                                                        float4* __restrict__ hits, uint8_t* __restrict__ occluded,
                                                        int hit_prim_ids, int tmax_from_ray, uint32_t* __restrict__ ovf,
                                                        uint32_t* __restrict__ dyn,
                                                        unsigned long long* __restrict__ visit_totals,
                                                        uint32_t* __restrict__ clear_a, uint32_t* __restrict__ clear_b,
                                                        const uint32_t* __restrict__ item_of,
                                                        const MultiItem* __restrict__ items) {
    __shared__ uint32_t lds[LDS_DEPTH * TRACE_BLOCK];
    // the next round's queue counters (their last readers ran before this
    // kernel in stream order), so the bounce loop needs no clearing launches
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (clear_a) *clear_a = 0u;
        if (clear_b) *clear_b = 0u;
    }
    __shared__ float4 top[TOP_F4];
    stage_top_nodes(top, sc);
    const uint32_t n = count_ptr ? *count_ptr : count_fixed;
    const size_t nthreads = (size_t)gridDim.x * blockDim.x;
    const size_t gtid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t* my_lds = lds + threadIdx.x;
    uint32_t* my_ovf = ovf ? ovf + gtid : nullptr;
    const uint32_t nwaves = (uint32_t)(nthreads / 64), wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(gtid / 64));
    RayChunks ch = chunks_first<DYN>(wave, nwaves, n);
    VisitCount vc;
    RayPre r;
    Trav t;
    TravView view{sc.nodes, sc.tris, MULTI ? 0u : sc.top_nodes};
    auto load = [&](uint32_t i) {
        const float4 o4 = ray_o[(size_t)i * ray_stride], d4 = ray_d[(size_t)i * ray_stride];
        if constexpr (MULTI) {
            const MultiItem& it = items[item_of[__float_as_uint(d4.w)]];
            view.nodes = it.nodes;
            view.tris = it.tris;
        }
        r = ray_setup(xyz(o4), xyz(d4));
        trav_init(t, tmax_from_ray ? o4.w : INFINITY);   // extension rays: tMax = Infinity (PathTracer.h:167)
    };
    auto finish = [&](uint32_t i, bool occ) {
        if (ANY) occluded[i] = occ ? 1 : 0;
        else hits[i] = hit_record(t, hit_prim_ids && t.best_slot != INVALID ? prim_of_slot(view, t.best_slot) : t.best_slot);
    };
    if constexpr (MULTI) trace_queue<ANY, LDS_DEPTH, COUNT, DYN>(ch, dyn, view, r, t, top, my_lds, my_ovf, nthreads, vc, load, finish);
    else trace_queue<ANY, LDS_DEPTH, COUNT, DYN>(ch, dyn, sc, r, t, top, my_lds, my_ovf, nthreads, vc, load, finish);
    if constexpr (DYN) chunks_release(dyn);
    if (COUNT) flush_counts(visit_totals, vc);
}

#define XT_INST_TRACE(ANY, COUNT, MULTI, DYN)                                                                      \
    template __global__ void k_trace<ANY, TRACE_LDS_DEPTH, COUNT, MULTI, DYN>(                                     \
        DevScene, const float4*, const float4*, int, const uint32_t*, uint32_t, float4*, uint8_t*, int, int,       \
        uint32_t*, uint32_t*, unsigned long long*, uint32_t*, uint32_t*, const uint32_t*, const MultiItem*);
XT_INST_TRACE(false, false, false, false)
XT_INST_TRACE(true, false, false, false)
XT_INST_TRACE(false, true, false, false)
XT_INST_TRACE(true, true, false, false)
XT_INST_TRACE(false, false, true, false)
XT_INST_TRACE(false, false, true, true)
XT_INST_TRACE(false, false, false, true)
XT_INST_TRACE(true, false, false, true)
XT_INST_TRACE(false, true, false, true)
XT_INST_TRACE(true, true, false, true)
#undef XT_INST_TRACE

// ---------------------------------------------------------------- wavefront PT

// Camera ray of a pixel's sample (PinholeCamera::generateRay, Camera.h:45-55)
// at the jittered film position of RenderTargetTile::GenerateFilmPosition
// (RenderTarget.h:68-80).
__device__ __forceinline__ void camera_ray(const WaveParams& wp, uint32_t pixel, uint32_t sample, f3* o, f3* d) {
    const uint32_t x = pixel % wp.width, y = pixel / wp.width;
    Rng rng{make_uint2(wp.seed, wp.stream), pixel, sample};
    uint4 b0 = rng.block(0, 0);
    float ux = Rng::to_unit(b0.x), uy = Rng::to_unit(b0.y);
    float fx = (float)x, fy = (float)y;
    fx /= (float)wp.width;
    fy /= (float)wp.height;
    fy = 1.0f - fy;
    fx += (ux - 0.5f) / (float)wp.width;
    fy += (uy - 0.5f) / (float)wp.height;
    f3 dc = normalize(mk(wp.tan_x * (fx - 0.5f) * 2, wp.tan_y * (fy - 0.5f) * 2, 1));
    *o = xf_point(wp.cam, mk(0, 0, 0));
    *d = xf_vector(wp.cam, dc);
}

// Camera rays of a batch's paths.
__global__ __launch_bounds__(256) void k_generate(WaveParams wp, PathQueue q, float4* __restrict__ radiance) {
    const BatchCursor bc = batch_of(wp);
    const uint32_t P = bc.num_paths;
    for (uint32_t id = blockIdx.x * blockDim.x + threadIdx.x; id < P; id += gridDim.x * blockDim.x) {
        uint32_t s_local = id / bc.num_pixels;
        uint32_t pixel = bc.first_pixel + (id - s_local * bc.num_pixels);
        f3 o, d;
        camera_ray(wp, pixel, bc.sample0 + s_local, &o, &d);
        // e (the sampling record) and the radiance slot of a camera ray are
        // implied by its vertex index 1: the shade step reads neither
        q.o[id] = make_float4(o.x, o.y, o.z, 0.0f);
        q.d[id] = make_float4(d.x, d.y, d.z, __uint_as_float(id));
        q.w[id] = make_float4(1.0f, 1.0f, 1.0f, __uint_as_float(1u));
        if (q.rec) q.rec[id] = INVALID;
    }
}

// Material-sorted shading (XT_FLAG_SORT_MATERIALS): the block's queue
// entries [base, base + blockDim.x) are partitioned by shading key (miss,
// then 1 + material type of the hit) before they are shaded, stably, so each
// wave of the block mostly shades one kind of BSDF instead of every kind the
// queue mixes.  Returns this thread's entry offset within the block; every
// thread of the block must call it (the callers' loops are block-uniform).
constexpr int SHADE_KEYS = 1 + XT_MAT_COUNT_ + 1;   // miss, material types, entries past the queue end
template <int BLOCK>
__device__ __forceinline__ uint32_t block_sort_by_material(const DevScene& sc, const float4* __restrict__ hits,
                                                           uint32_t base, uint32_t n,
                                                           uint32_t* sh /* (BLOCK / 64 + 1) * SHADE_KEYS + BLOCK */) {
    constexpr int NW = BLOCK / 64;
    const uint32_t i = base + threadIdx.x;
    uint32_t key = SHADE_KEYS - 1;
    if (i < n) {
        const uint32_t slot = __float_as_uint(hits[i].y);
        key = 0;
        if (slot != INVALID) {
            const uint32_t m = __float_as_uint(in_global(sc.tris)[(size_t)slot * TRI_F4 + 1].w);
            key = 1 + min(in_global((const uint32_t*)sc.mats)[(size_t)m * (sizeof(xt_material) / 4)], (uint32_t)XT_MAT_COUNT_);
        }
    }
    const uint32_t wave = threadIdx.x / 64, lane = __lane_id();
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t rank = 0;
#pragma unroll
    for (int k = 0; k < SHADE_KEYS; ++k) {
        const uint64_t m = __ballot(key == (uint32_t)k);
        if (key == (uint32_t)k) rank = (uint32_t)__popcll(m & below);
        if (lane == 0) sh[wave * SHADE_KEYS + k] = (uint32_t)__popcll(m);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        // key-major, then wave order: every wave's share of a key after the
        // earlier waves' share of it, and after every entry of a smaller key
        uint32_t total = 0;
        for (int k = 0; k < SHADE_KEYS; ++k)
            for (int w = 0; w < NW; ++w) {
                const uint32_t c = sh[w * SHADE_KEYS + k];
                sh[w * SHADE_KEYS + k] = total;
                total += c;
            }
    }
    __syncthreads();
    uint32_t* order = sh + (NW + 1) * SHADE_KEYS;
    order[sh[wave * SHADE_KEYS + key] + rank] = threadIdx.x;
    __syncthreads();
    const uint32_t mine = order[threadIdx.x];
    __syncthreads();   // sh is reused by the next iteration
    return mine;
}

// The result of shading one queue entry: the extension ray and the light
// sample it pushes, if any.
struct ShadeOut {
    bool push_ext = false, push_sh = false, guided = false;
    f3 ext_o{0.0f, 0.0f, 0.0f}, ext_d{0.0f, 0.0f, 0.0f}, ext_w{0.0f, 0.0f, 0.0f}, ext_e{0.0f, 0.0f, 0.0f};
    float ext_pdf = 0.0f, ext_pe = 0.0f;
    uint32_t ext_v = 0;
    Surf s;
    f3 sh_o{0.0f, 0.0f, 0.0f}, sh_d{0.0f, 0.0f, 0.0f}, sh_c{0.0f, 0.0f, 0.0f};
    float sh_tmax = 0.0f;
    uint32_t id = 0;
};

// Path id -> (pixel, sample) of a single render's batch (as k_generate).
struct CursorMap {
    const WaveParams& wp;
    __device__ __forceinline__ uint2 operator()(uint32_t id) const {
        const BatchCursor bc = batch_of(wp);
        const uint32_t s_local = id / bc.num_pixels;
        return make_uint2(bc.first_pixel + (id - s_local * bc.num_pixels), bc.sample0 + s_local);
    }
};

// The batch's camera rays, made where they are traced and again where their
// hits are shaded (k_shade's FIRST form), so the first round has no ray queue:
// writing and reading one cost 144 bytes a path and a launch, making the rays
// twice some 300 VALU instructions (1080p field, 132 M paths: 58.06 -> 57.32 ms a
// frame, of which k_generate 1.44, while the camera rays' trace went from 12.9
// to 13.6; Cornell box 1239 -> 1232 us).
template <bool DYN>
__global__ __launch_bounds__(TRACE_BLOCK, 8) void k_trace_camera(DevScene sc, WaveParams wp, float4* __restrict__ hits,
                                                                 uint32_t* __restrict__ ovf, uint32_t* __restrict__ dyn,
                                                                 unsigned long long* __restrict__ clear) {
    __shared__ uint32_t lds[TRACE_LDS_DEPTH * TRACE_BLOCK];
    if (blockIdx.x == 0 && threadIdx.x == 0) *clear = 0ull;   // the next round's queues
    __shared__ float4 top[TOP_F4];
    stage_top_nodes(top, sc);
    const size_t nthreads = (size_t)gridDim.x * blockDim.x;
    const size_t gtid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t nwaves = (uint32_t)(nthreads / 64), wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(gtid / 64));
    const RayChunks ch = chunks_first<DYN>(wave, nwaves, batch_of(wp).num_paths);
    const CursorMap pmap{wp};
    VisitCount vc;
    RayPre r;
    Trav t;
    trace_queue<false, TRACE_LDS_DEPTH, false, DYN>(
        ch, dyn, sc, r, t, top, lds + threadIdx.x, ovf ? ovf + gtid : nullptr, nthreads, vc,
        [&](uint32_t i) {
            f3 o, d;
            const uint2 ps = pmap(i);
            camera_ray(wp, ps.x, ps.y, &o, &d);
            r = ray_setup(o, d);
            trav_init(t, INFINITY);   // tMax = Infinity (PathTracer.h:167)
        },
        [&](uint32_t i, bool) { hits[i] = hit_record(t, t.best_slot); });
    if constexpr (DYN) chunks_release(dyn);
}
template __global__ void k_trace_camera<false>(DevScene, WaveParams, float4*, uint32_t*, uint32_t*, unsigned long long*);
template __global__ void k_trace_camera<true>(DevScene, WaveParams, float4*, uint32_t*, uint32_t*, unsigned long long*);

// One StandardPathTracer / NaivePathTracer loop step (PathTracer.h:147-246 /
// 65-101) for queue entry i: emission at the new vertex, roulette, BSDF
// sample -> extension ray, light sample -> shadow ray.
// Per-render constants of the shade step.
struct ShadeConst {
    bool standard, can_sample, uniform_bary;
    EnvNee envn;
    float p_area;
    uint2 key;
};
__device__ __forceinline__ ShadeConst shade_const(const WaveParams& wp, const DevScene& sc) {
    ShadeConst c;
    c.standard = wp.integrator == XT_INTEGRATOR_STANDARD;
    c.can_sample = sc.num_lights > 0;
    c.envn = env_nee_setup(sc.env, c.standard && (wp.flags & XT_FLAG_ENV_NEE) != 0, c.can_sample);
    c.p_area = c.can_sample ? 1.0f - c.envn.p_select : 0.0f;
    c.uniform_bary = (wp.flags & XT_FLAG_UNIFORM_BARY) != 0;
    c.key = make_uint2(wp.seed, wp.stream);
    return c;
}

// A path's arrival at a vertex: the ray that reached it (direction, BSDF
// sample) and the path's state.
struct VertexIn {
    f3 d, weight, meval;
    float pdf_prev, pe_prev;
    uint32_t v, qflags, id;
    float4 h;          // hit record of the ray
    f3 rad, pend;      // radiance so far; light sample of the previous vertex (QF_PENDING)
};

// One loop step of the path at `in`; i: its guide lobes' entry.  put_rad(rad)
// takes the path's radiance up to here.
// WHICH: all kinds of ray, or only such as are known to miss or to hit.
enum class Rays { ALL, MISS, HIT };
template <bool GUIDE, bool NMAP, Rays WHICH = Rays::ALL, class PathMap, class PutRad>
__device__ __forceinline__ void shade_vertex(const WaveParams& wp, const DevScene& sc, const ShadeConst& sc0,
                                             const VertexIn& in, const GuideRender& gr, uint32_t i, const PathMap& pmap,
                                             PutRad put_rad, ShadeOut& out) {
    const bool standard = sc0.standard;
    const bool can_sample = sc0.can_sample;
    const EnvNee envn = sc0.envn;
    const float p_area = sc0.p_area;
    const bool uniform_bary = sc0.uniform_bary;
    const uint2 key = sc0.key;
    bool& push_ext = out.push_ext;
    bool& push_sh = out.push_sh;
    bool& guided = out.guided;
    f3& ext_o = out.ext_o;
    f3& ext_d = out.ext_d;
    f3& ext_w = out.ext_w;
    f3& ext_e = out.ext_e;
    float& ext_pdf = out.ext_pdf;
    float& ext_pe = out.ext_pe;
    uint32_t& ext_v = out.ext_v;
    Surf& s = out.s;
    f3& sh_o = out.sh_o;
    f3& sh_d = out.sh_d;
    f3& sh_c = out.sh_c;
    float& sh_tmax = out.sh_tmax;
    const uint32_t id = out.id = in.id;
        const uint32_t v = in.v, qflags = in.qflags;
        const float4 h = in.h;
        const float pdf_prev = in.pdf_prev, pe_prev = in.pe_prev;
        const f3 d = in.d, meval = in.meval, pend = in.pend;
        f3 weight = in.weight, rad = in.rad;
        const uint32_t slot = __float_as_uint(h.y);
        const bool hit = WHICH == Rays::ALL ? slot != INVALID : WHICH == Rays::HIT;
        xt_material mat;
        bool emissive = false;
        if (hit) {
            s = make_surf<NMAP>(sc, slot, d, h.z, h.w);
            mat = in_global(sc.mats)[s.mat];
            emissive = mat.type == XT_MAT_EMISSION;
        }
        // ---- radiance arriving along the ray that reached this vertex
        if (v == 1 && standard) {
            if (!hit) {
                if (sc.env.has_sky) rad += weight * env_radiance(sc.env, d);          // PathTracer.h:133-136
            } else if (emissive) {
                rad += weight * emitted(mat, -d, s.n);                                // PathTracer.h:143-145
            }
        } else if (standard) {
            if (!hit) {
                if (sc.env.has_sky) {                                                  // PathTracer.h:192-195
                    f3 Le = env_radiance(sc.env, d);
                    if (envn.on && pdf_prev >= 0.0f) {
                        // power heuristic; a direction the sky sampler cannot produce
                        // (pe = 0) or an unbounded BSDF pdf keeps the full weight
                        const float mis = (pe_prev > 0.0f && pdf_prev < INFINITY)
                                              ? (pdf_prev * pdf_prev) / (pdf_prev * pdf_prev + pe_prev * pe_prev)
                                              : 1.0f;
                        rad += weight * mis * meval * Le;
                    } else {
                        rad += weight * meval * Le;
                    }
                }
            } else if (emissive) {                                                     // PathTracer.h:171-189
                float mis;
                if (pdf_prev >= 0.0f && can_sample) {
                    float pl = in_global(sc.light_pdf)[slot] * p_area;
                    float cosL = fabsf(dot(d, s.sn));
                    float distSq = h.x * h.x;
                    pl *= distSq / cosL;
                    mis = (pdf_prev * pdf_prev) / (pdf_prev * pdf_prev + pl * pl);
                } else {
                    mis = 1.0f;
                }
                if (mis > 0.0f) rad += weight * mis * meval * emitted(mat, -d, s.n);
            }
        } else {                                                                       // PathTracer.h:75-98
            if (!hit) {
                if (sc.env.has_sky) rad += clamp_pos(weight * env_radiance(sc.env, d));
            } else if (emissive) {
                rad += weight * emitted(mat, -d, s.n);
            }
        }
        if (qflags & QF_PENDING) rad += pend;  // light sample of the previous vertex
        put_rad(rad);

        bool live = hit && !emissive;
        Rng rng{key, 0u, 0u};
        if (live) {
            const uint2 ps = pmap(id);   // path id -> (pixel, sample)
            rng.pixel = ps.x;
            rng.sample = ps.y;
        }
        if (live && standard) {
            if (v > 1) {                                       // PathTracer.h:239-245
                weight = weight * meval;
                if (is_zero(weight)) live = false;
            }
            if (live && wp.max_depth > 0 && (int)v > wp.max_depth) live = false;
            uint4 blk0 = make_uint4(0, 0, 0, 0);
            if (live) blk0 = rng.block(v, 0);
            if (live && (int)(v + 1) > wp.rr_start) {          // PathTracer.h:149-155
                if (Rng::to_unit(blk0.x) >= wp.rr_prob) live = false;
                else weight = div(weight, wp.rr_prob);
            }
            if (live) {
                const Frame fs = make_frame(s.sn);   // BasisVectors(shading.n), shared by both samplers
                f3 wi = splat(0.0f);
                float pdfB = 0.0f;
                f3 me;
                // Guided vertex: one-sample MIS of the learned mixture (probability
                // gr.prob) and the BSDF sampler; the strategy pdf is the mixture
                // pdf wherever the BSDF pdf is positive, and zero elsewhere.
                guided = GUIDE && gr.lobes_mk != nullptr && !mat_is_delta(mat.type) &&
                         (gr.max_vertex == 0 || v <= gr.max_vertex);
                const WalkKey wk{key, rng.pixel, rng.sample, v};
                auto l4 = [&](int j) { return unpack_lobe(gr.lobes_mk[(size_t)j * gr.stride + i]); };
                auto l2 = [&](int j) { return gr.lobes2[(size_t)j * gr.stride + i]; };
                // (a NaN BSDF pdf -- GGX D at a grazing half vector -- stays NaN, so
                // the light-sample MIS below drops that sample as the plain path does)
                auto strategy_pdf = [&](f3 dir, float pb) {
                    if (pb != pb) return pb;
                    return pb > 0.0f ? gr.prob * guide_pdf_lobes(l4, l2, dir) + (1.0f - gr.prob) * pb : 0.0f;
                };
                if (guided) {
                    const uint4 blk3 = rng.block(v, 3);
                    // The random walk's sampling density is not its getPDF (an
                    // approximation, Main.cpp:245), so a walk-sampled direction is
                    // weighted with its throughput, the unbiased estimate of f / p:
                    // me = throughput * p^ / (c q + (1 - c) p^), the one-sample MIS
                    // whose weights (computed with p^) still sum to one.
                    const bool walk = NMAP && mat.type == XT_MAT_MICROFACET_NMAP;
                    float pb;
                    f3 fc;
                    if (Rng::to_unit(blk3.x) < gr.prob) {
                        wi = guide_sample_lobes(l4, l2, Rng::to_unit(blk3.y), Rng::to_unit(blk3.z),
                                                Rng::to_unit(blk3.w));
                        fc = mat_eval<NMAP>(mat, s, wi, &pb, wk, D_WALK_EVAL2);
                    } else if (walk) {
                        fc = mat_sample<NMAP>(mat, s, fs, blk0, wk, &wi, &pb) * pb;
                    } else {
                        mat_sample<NMAP>(mat, s, fs, blk0, wk, &wi, &pdfB);
                        fc = mat_eval<NMAP>(mat, s, wi, &pb, wk, D_WALK_EVAL2);
                    }
                    pdfB = strategy_pdf(wi, pb);
                    if (!(pdfB > 0.0f)) pdfB = 0.0f;
                    me = pdfB > 0.0f ? div(fc, pdfB) : splat(0.0f);
                    if (!finite3(me)) me = splat(0.0f);
                } else {
                    me = mat_sample<NMAP>(mat, s, fs, blk0, wk, &wi, &pdfB);
                }
                if (!is_zero(me)) {                            // PathTracer.h:165-167
                    push_ext = true;
                    ext_d = wi;
                    ext_o = s.p + wp.eps * wi;
                    ext_w = weight;
                    ext_e = me;
                    ext_pdf = pdfB;
                    ext_v = v + 1;
                    ext_pe = (envn.on && pdfB >= 0.0f) ? envn.p_select * env_nee_pdf(sc.env, envn, normalize(wi), s.sn)
                                                       : 0.0f;
                }
                // ---- light sample (PathTracer.h:202-233)
                uint4 blk1 = rng.block(v, 1);
                bool sample_env = false;
                if (envn.on) sample_env = !can_sample || Rng::to_unit(blk1.x) < envn.p_select;
                if (sample_env) {
                    if (pdfB >= 0.0f) {
                        f3 ld = env_nee_sample(sc.env, envn, fs, Rng::to_unit(blk1.w), Rng::to_unit(blk1.y),
                                               Rng::to_unit(blk1.z));
                        float pe = envn.p_select * env_nee_pdf(sc.env, envn, ld, s.sn);
                        float pb;
                        f3 fc = mat_eval<NMAP>(mat, s, ld, &pb, wk, D_WALK_EVAL);
                        if (guided) pb = strategy_pdf(ld, pb);
                        const float mis = (pe * pe) / (pb * pb + pe * pe);
                        if (pe > 0.0f && !is_zero(fc) && mis > 0.0f) {   // NaN mis: dropped
                            f3 c = div(weight * mis * fc * env_radiance(sc.env, ld), pe);
                            push_sh = true;
                            sh_d = ld;
                            sh_o = s.p + wp.eps * ld;
                            sh_tmax = INFINITY;
                            sh_c = c;
                        }
                    }
                } else if (can_sample) {
                    uint2 lo = in_global(sc.light_objs)[blk1.y % sc.num_lights];
                    uint32_t lslot = in_global(sc.light_slots)[lo.x + blk1.z % lo.y];
                    uint4 blk2 = rng.block(v, 2);
                    float t0, t1;
                    if (uniform_bary) {
                        float su = sqrtf(Rng::to_unit(blk2.x));
                        t0 = 1.0f - su;
                        t1 = Rng::to_unit(blk2.y) * su;
                    } else {                                   // TriangleIndexed.h:184-192
                        float a = Rng::to_unit(blk2.x), b = Rng::to_unit(blk2.y), c = Rng::to_unit(blk2.z);
                        float sum = a + b + c;
                        if (sum == 0.0f) {
                            a = b = c = 1.0f;
                            sum = 3.0f;
                        }
                        float inv = 1.0f / sum;
                        t0 = a * inv;
                        t1 = b * inv;
                    }
                    const auto lt = in_global(sc.tris) + (size_t)lslot * TRI_F4;
                    float4 l0 = lt[0], l1 = lt[1], l2 = lt[2];
                    f3 q0 = xyz(l0), q1 = xyz(l1), q2 = xyz(l2);
                    f3 lp = lerp3(q0, q1, q2, t0, t1);
                    f3 ln = normalize(cross(q1 - q0, q2 - q0));
                    f3 lsn = ln;
                    if (__float_as_uint(l2.w) & TRI_FLAG_NORMALS) {
                        const auto nr = in_global(sc.normals) + (size_t)lslot * TRI_F4;
                        lsn = normalize(lerp3(xyz(nr[0]), xyz(nr[1]), xyz(nr[2]), t0, t1));
                    }
                    ln = normalize(ln);
                    lsn = normalize(lsn);
                    float pdfL = in_global(sc.light_pdf)[lslot] * p_area;
                    float dist = length(lp - s.p);
                    f3 sd = div(lp - s.p, dist);
                    if (dot(sd, ln) < 0) {
                        float distSq = dist * dist;
                        float mis;
                        float pb;
                        f3 fc = mat_eval<NMAP>(mat, s, sd, &pb, wk, D_WALK_EVAL);
                        if (guided) pb = strategy_pdf(sd, pb);
                        if (pdfB >= 0.0f) {
                            float cosL = fabsf(dot(-sd, lsn));
                            pb *= cosL / distSq;
                            mis = (pdfL * pdfL) / (pb * pb + pdfL * pdfL);
                        } else {
                            mis = 0.0f;
                        }
                        if (mis > 0.0f) {
                            float G = fabsf(dot(-sd, lsn)) / distSq;
                            const xt_material lm = in_global(sc.mats)[__float_as_uint(l1.w)];
                            f3 c = div(weight * mis * fc * emitted(lm, -sd, ln) * G, pdfL);
                            push_sh = true;
                            sh_d = sd;
                            sh_o = s.p + wp.eps * sd;
                            sh_tmax = dist - wp.shadow_margin;
                            sh_c = c;
                        }
                    }
                }
            }
        } else if (live) {  // NaivePathTracer (PathTracer.h:86-100), then the roulette of the next loop head
            uint4 blk0 = rng.block(v, 0);
            f3 wi = splat(0.0f);
            float pdfB = 0.0f;
            const WalkKey wk{key, rng.pixel, rng.sample, v};
            weight = weight * mat_sample<NMAP>(mat, s, make_frame(s.sn), blk0, wk, &wi, &pdfB);
            if (is_zero(weight)) live = false;
            if (live && wp.max_depth > 0 && (int)v > wp.max_depth) live = false;
            if (live && (int)(v + 1) > wp.rr_start) {
                uint4 nb = rng.block(v + 1, 0);
                if (Rng::to_unit(nb.x) >= wp.rr_prob) live = false;
                else weight = div(weight, wp.rr_prob);
            }
            if (live) {
                push_ext = true;
                ext_d = wi;
                ext_o = s.p + wp.eps * wi;
                ext_w = weight;
                ext_e = splat(1.0f);
                ext_pdf = pdfB;
                ext_v = v + 1;
            }
        }
}

// shade_vertex of queue entry i.
// FIRST: the camera ray of path i, as k_trace_camera traced it.
template <bool GUIDE, bool NMAP, bool FIRST, Rays WHICH = Rays::ALL, class PathMap>
__device__ __forceinline__ void shade_entry(const WaveParams& wp, const DevScene& sc, const ShadeConst& sc0,
                                            const PathQueue& qin, const float4* __restrict__ hits,
                                            float4* __restrict__ radiance, float4* __restrict__ pending,
                                            const GuideRender& gr, uint32_t i, const PathMap& pmap, ShadeOut& out) {
    VertexIn in;
    in.h = hits[i];
    if constexpr (FIRST) {
        f3 o;
        const uint2 ps = pmap(i);
        camera_ray(wp, ps.x, ps.y, &o, &in.d);
        in.id = i;
        in.v = 1u;
        in.qflags = 0u;
        in.pdf_prev = in.pe_prev = 0.0f;
        in.weight = in.meval = splat(1.0f);
        in.rad = in.pend = splat(0.0f);
    } else {
        const float4 o4 = qin.o[i], d4 = qin.d[i], w4 = qin.w[i];
        in.id = __float_as_uint(d4.w);
        const uint32_t vf = __float_as_uint(w4.w);
        in.v = vf & 0xFFFFFFu;
        in.qflags = vf >> 24;
        // a camera ray (vertex 1) has no sampling record and no radiance yet:
        // the generate step writes neither
        const float4 e4 = in.v > 1 ? qin.e[i] : make_float4(1.0f, 1.0f, 1.0f, 0.0f);
        in.pdf_prev = o4.w;
        in.pe_prev = e4.w;
        in.d = xyz(d4);
        in.meval = xyz(e4);
        in.weight = xyz(w4);
        in.rad = in.v > 1 ? xyz(radiance[in.id]) : splat(0.0f);
        in.pend = (in.qflags & QF_PENDING) ? xyz(pending[in.id]) : splat(0.0f);
        if (GUIDE && gr.recs) {
            // the vertex that sampled this ray: radiance up to and including its light sample
            const uint32_t rin = qin.rec[i];
            if (rin != INVALID) gr.recs[rin].f = f4(in.rad + in.pend, 0.0f);
        }
    }
    const uint32_t id = in.id;
    shade_vertex<GUIDE, NMAP, WHICH>(wp, sc, sc0, in, gr, i, pmap, [&](f3 rad) { radiance[id] = f4(rad, 0.0f); }, out);
}

// Compacted appends of a block's shaded entries (every thread of the block
// calls it): the extension ray with its training record, the shadow ray.
template <bool GUIDE, int BLOCK>
__device__ __forceinline__ void shade_emit(ShadeOut& o, const PathQueue& qout,
                                           unsigned long long* __restrict__ counts_out, const ShadowQueue& sq,
                                           const GuideRender& gr, uint32_t* append_lds) {
    // guided light samples: a non-finite contribution is dropped, never summed
    if (GUIDE && o.push_sh && !finite3(o.sh_c)) o.push_sh = false;
    const uint2 slots = block_append2<BLOCK>(counts_out, o.push_ext, o.push_sh, append_lds);
    const uint32_t ei = slots.x, si = slots.y;
    if (o.push_ext) {
        uint32_t fl = o.push_sh ? QF_PENDING : 0u;
        qout.o[ei] = f4(o.ext_o, o.ext_pdf);
        qout.d[ei] = f4(o.ext_d, __uint_as_float(o.id));
        qout.w[ei] = f4(o.ext_w, __uint_as_float(o.ext_v | (fl << 24)));
        qout.e[ei] = f4(o.ext_e, o.ext_pe);
        if (GUIDE && gr.recs) {
            const uint32_t ri = gr.rec_base + ei;
            const bool keep = ri < gr.rec_cap && ri >= gr.rec_base;
            qout.rec[ei] = keep ? ri : INVALID;
            if (keep) {
                TrainRec& rr = gr.recs[ri];
                const Surf& s = o.s;
                rr.a = make_float4(s.p.x, s.p.y, s.p.z, s.sn.x);
                rr.b = make_float4(s.sn.y, s.sn.z, s.wo.x, s.wo.y);
                rr.c = make_float4(s.wo.z, o.ext_d.x, o.ext_d.y, o.ext_d.z);
                rr.d = make_float4(o.ext_pdf, o.ext_w.x, o.ext_w.y, o.ext_w.z);
                rr.e = f4(o.ext_e, __uint_as_float(o.id | (o.guided ? TREC_GUIDED : 0u)));
            }
        }
    }
    if (o.push_sh) {
        sq.o[si] = f4(o.sh_o, o.sh_tmax);
        sq.d[si] = f4(o.sh_d, __uint_as_float(o.id));
        sq.c[si] = f4(o.sh_c, o.push_ext ? 1.0f : 0.0f);
    }
}

// The forms without normal mapping (but the guided sorted one, at 144 VGPRs)
// are bounded to 4 waves per SIMD, which they reach without spilling.
// FIRST: the first round of an unguided render, whose queue is the batch's
// paths themselves.
template <bool GUIDE, bool NMAP, bool SORT, bool FIRST>
__global__ __launch_bounds__(shade_block(GUIDE, NMAP), NMAP || (GUIDE && SORT) ? 1 : 4) void k_shade(WaveParams wp, const DevScene* __restrict__ scene, PathQueue qin,
                                               const uint32_t* __restrict__ count_in, const float4* __restrict__ hits,
                                               PathQueue qout, unsigned long long* __restrict__ counts_out,
                                               ShadowQueue sq, float4* __restrict__ radiance,
                                               float4* __restrict__ pending, GuideRender gr) {
    // the scene record is read through a pointer: by value its fields
    // occupy scalar registers for the whole kernel and spill (111 SGPR
    // spills, 556 lane reads, 112 VGPRs; through the pointer 32, 80, 103)
    const DevScene& sc = *scene;
    const uint32_t n = FIRST ? batch_of(wp).num_paths : *count_in;
    const uint32_t stride = gridDim.x * blockDim.x;
    constexpr int BLOCK = shade_block(GUIDE, NMAP);
    __shared__ uint32_t append_lds[2 * (BLOCK / 64) + 2];
    __shared__ uint32_t sort_lds[SORT ? (BLOCK / 64 + 1) * SHADE_KEYS + BLOCK : 1];
    const CursorMap pmap{wp};
    const ShadeConst c0 = shade_const(wp, sc);
    // whole-block iterations so the appends below always see every thread
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += stride) {
        const uint32_t i = base + (SORT ? block_sort_by_material<BLOCK>(sc, hits, base, n, sort_lds) : threadIdx.x);
        ShadeOut o;
        if (i < n) shade_entry<GUIDE, NMAP, FIRST>(wp, sc, c0, qin, hits, radiance, pending, gr, i, pmap, o);
        shade_emit<GUIDE, BLOCK>(o, qout, counts_out, sq, gr, append_lds);
    }
}

// A block's share of a queue in which many rays have left for the sky: misses
// are shaded as they come, hits are collected and shaded by the whole block at
// a time, so the long code of a hit does not run for the few lanes of a wave
// that hit (11 of 64 in the second round of the 1080p field, 9 in the
// normal-mapped plane's).  1080p field, 132 M paths, 57.5 -> 55.3 ms a frame, its
// second round 6.1 -> 4.3 ms, now some 3.3 TB/s; plane at 6.2 M paths 8.0 -> 6.8.
// A first round, whose camera rays miss together, is faster in queue order
// (plane 6.72 against 6.87 ms).  Where nearly every ray hits it costs nothing
// that shows: 100 k triangle room at 655 k paths 3.70 ms under a sky and without.
// list: 2 * BLOCK entries, wave_hits: one count per wave.
template <int BLOCK, class Miss, class Hit>
__device__ __forceinline__ void shade_open(uint32_t n, const float4* __restrict__ hits, const PathQueue& qout,
                                           unsigned long long* __restrict__ counts_out, const ShadowQueue& sq,
                                           uint32_t* append_lds, uint32_t* list, uint32_t* wave_hits, Miss miss, Hit hit) {
    const GuideRender gr{};
    const uint32_t stride = gridDim.x * blockDim.x, wave = threadIdx.x / 64;
    uint32_t waiting = 0;   // entries of list: below BLOCK between iterations
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += stride) {
        const uint32_t i = base + threadIdx.x;
        const bool hits_i = i < n && __float_as_uint(hits[i].y) != INVALID;
        if (i < n && !hits_i) miss(i);
        const uint64_t mask = wave_ballot(hits_i);
        if (__lane_id() == 0) wave_hits[wave] = (uint32_t)__popcll(mask);
        __syncthreads();
        uint32_t at = waiting;
        for (uint32_t w = 0; w < BLOCK / 64; ++w) {
            const uint32_t c = wave_hits[w];
            if (w < wave) at += c;
            waiting += c;
        }
        if (hits_i) list[at + (uint32_t)__popcll(mask & ((1ull << __lane_id()) - 1ull))] = i;
        __syncthreads();
        const bool last = n - base <= stride;
        while (waiting >= (uint32_t)BLOCK || (last && waiting)) {
            const uint32_t take = min(waiting, (uint32_t)BLOCK);
            waiting -= take;
            ShadeOut o;
            if (threadIdx.x < take) hit(list[waiting + threadIdx.x], o);
            shade_emit<false, BLOCK>(o, qout, counts_out, sq, gr, append_lds);   // ends with every list entry read
        }
    }
}

template <bool NMAP>
__global__ __launch_bounds__(shade_block(false, NMAP), NMAP ? 1 : 4) void k_shade_open(WaveParams wp, const DevScene* __restrict__ scene,
                                                                       PathQueue qin, const uint32_t* __restrict__ count_in,
                                                                       const float4* __restrict__ hits, PathQueue qout,
                                                                       unsigned long long* __restrict__ counts_out,
                                                                       ShadowQueue sq, float4* __restrict__ radiance,
                                                                       float4* __restrict__ pending, GuideRender gr) {
    constexpr int BLOCK = shade_block(false, NMAP);
    __shared__ uint32_t append_lds[2 * (BLOCK / 64) + 2], list[2 * BLOCK], wave_hits[BLOCK / 64];
    const DevScene& sc = *scene;
    const CursorMap pmap{wp};
    const ShadeConst c0 = shade_const(wp, sc);
    shade_open<BLOCK>(
        *count_in, hits, qout, counts_out, sq, append_lds, list, wave_hits,
        [&](uint32_t i) {
            ShadeOut o;
            shade_entry<false, NMAP, false, Rays::MISS>(wp, sc, c0, qin, hits, radiance, pending, gr, i, pmap, o);
        },
        [&](uint32_t i, ShadeOut& o) {
            shade_entry<false, NMAP, false, Rays::HIT>(wp, sc, c0, qin, hits, radiance, pending, gr, i, pmap, o);
        });
}
#define XT_INST_SHADE_OPEN(N)                                                                                         \
    template __global__ void k_shade_open<N>(WaveParams, const DevScene*, PathQueue, const uint32_t*, const float4*,   \
                                             PathQueue, unsigned long long*, ShadowQueue, float4*, float4*, GuideRender);
XT_INST_SHADE_OPEN(false)
XT_INST_SHADE_OPEN(true)
#undef XT_INST_SHADE_OPEN

#define XT_INST_SHADE(G, N, S, F)                                                                                \
    template __global__ void k_shade<G, N, S, F>(WaveParams, const DevScene*, PathQueue, const uint32_t*, const float4*,     \
                                                 PathQueue, unsigned long long*, ShadowQueue, float4*, float4*,       \
                                                 GuideRender);
XT_INST_SHADE(false, false, false, false)
XT_INST_SHADE(true, false, false, false)
XT_INST_SHADE(false, true, false, false)
XT_INST_SHADE(true, true, false, false)
XT_INST_SHADE(false, false, true, false)
XT_INST_SHADE(true, false, true, false)
XT_INST_SHADE(false, true, true, false)
XT_INST_SHADE(true, true, true, false)
XT_INST_SHADE(false, false, false, true)
XT_INST_SHADE(false, true, false, true)
XT_INST_SHADE(false, false, true, true)
XT_INST_SHADE(false, true, true, true)
#undef XT_INST_SHADE

// Any-hit for queued shadow rays; unoccluded contributions go straight to the
// path radiance, or to pending[] when the path continues (see k_shade).
// Bounded to 8 waves per SIMD, which every form reaches without spilling.
template <bool COUNT, bool DYN>
__global__ __launch_bounds__(TRACE_BLOCK, 8) void k_shadow(DevScene sc, ShadowQueue sq, const uint32_t* __restrict__ count,
                                                        float4* __restrict__ radiance, float4* __restrict__ pending,
                                                        uint32_t* __restrict__ ovf, uint32_t* __restrict__ dyn,
                                                        unsigned long long* __restrict__ visit_totals,
                                                        const uint32_t* __restrict__ counts4,
                                                        uint32_t* __restrict__ counts_out) {
    __shared__ uint32_t lds[TRACE_LDS_DEPTH * TRACE_BLOCK];
    // the round's final queue counts (shade, which appends them, ran before
    // this kernel) to the host's pinned ring, in place of a copy launch
    if (counts_out && blockIdx.x == 0 && threadIdx.x < 4) counts_out[threadIdx.x] = counts4[threadIdx.x];
    __shared__ float4 top[TOP_F4];
    stage_top_nodes(top, sc);
    const uint32_t n = *count;
    const size_t nthreads = (size_t)gridDim.x * blockDim.x;
    const size_t gtid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t* my_lds = lds + threadIdx.x;
    uint32_t* my_ovf = ovf ? ovf + gtid : nullptr;
    const uint32_t nwaves = (uint32_t)(nthreads / 64), wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(gtid / 64));
    RayChunks ch = chunks_first<DYN>(wave, nwaves, n);
    VisitCount vc;
    RayPre r;
    Trav t;
    trace_queue<true, TRACE_LDS_DEPTH, COUNT, DYN>(
        ch, dyn, sc, r, t, top, my_lds, my_ovf, nthreads, vc,
        [&](uint32_t i) {
            const float4 o4 = sq.o[i];
            r = ray_setup(xyz(o4), xyz(sq.d[i]));
            trav_init(t, o4.w);
        },
        [&](uint32_t i, bool occ) { shadow_record(sq, i, occ, radiance, pending); });
    if constexpr (DYN) chunks_release(dyn);
    if (COUNT) flush_counts(visit_totals, vc);
}
#define XT_INST_SHADOW(COUNT, DYN)                                                                               \
    template __global__ void k_shadow<COUNT, DYN>(DevScene, ShadowQueue, const uint32_t*, float4*, float4*, uint32_t*, \
                                                  uint32_t*, unsigned long long*, const uint32_t*, uint32_t*);
XT_INST_SHADOW(false, false)
XT_INST_SHADOW(true, false)
XT_INST_SHADOW(false, true)
XT_INST_SHADOW(true, true)
#undef XT_INST_SHADOW

// film[pixel] += radiance of each of the batch's samples, in sample order
// (overrun: null, or set when paths of the batch were left unfinished, and the
// film then stays as it is).
__global__ __launch_bounds__(256) void k_accumulate(WaveParams wp, const float4* __restrict__ radiance, void* film,
                                                    int film_f64, const uint32_t* __restrict__ overrun) {
    if (overrun && *overrun) return;
    const BatchCursor bc = batch_of(wp);
    const uint32_t np = bc.num_pixels, S = bc.num_paths / bc.num_pixels;
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < np; p += gridDim.x * blockDim.x) {
        size_t o = 3 * (size_t)(bc.first_pixel + p);
        if (film_f64) {
            double* f = (double*)film;
            double r = f[o], g = f[o + 1], b = f[o + 2];
            for (uint32_t s = 0; s < S; ++s) {
                float4 L = radiance[(size_t)s * np + p];
                r += (double)L.x;
                g += (double)L.y;
                b += (double)L.z;
            }
            f[o] = r;
            f[o + 1] = g;
            f[o + 2] = b;
        } else {
            float* f = (float*)film;
            float r = f[o], g = f[o + 1], b = f[o + 2];
            for (uint32_t s = 0; s < S; ++s) {
                float4 L = radiance[(size_t)s * np + p];
                r += L.x;
                g += L.y;
                b += L.z;
            }
            f[o] = r;
            f[o + 1] = g;
            f[o + 2] = b;
        }
    }
}

// ---------------------------------------------------------------- device-side batch schedule

__device__ __forceinline__ BatchCursor cursor_at(const BatchPlan& pl, uint32_t px0, uint32_t s0, uint32_t base) {
    BatchCursor c;
    c.first_pixel = px0;
    c.num_pixels = min(pl.pix_chunk, pl.npix - px0);
    c.s_rel = s0;
    c.sample0 = base + s0;
    c.num_paths = c.num_pixels * min(pl.S, pl.spp - s0);
    return c;
}

// First batch of a render whose first sample is plan.spp_offset; clears a
// chunk cursor that nothing else has (dyn, or null).
__global__ void k_cursor_init(BatchCursor* c, BatchPlan plan, uint32_t* dyn) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    *c = cursor_at(plan, 0, 0, plan.spp_offset);
    if (dyn) dyn[0] = dyn[1] = 0u;
}

// Next batch: the next pixel chunk, or the first chunk of the next S samples.
// Past the last batch the cursor holds zero paths.
__global__ void k_advance_cursor(BatchCursor* c, BatchPlan plan) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    BatchCursor cur = *c;
    const uint32_t base = cur.sample0 - cur.s_rel;   // the render's first sample (plan.spp_offset is not used here)
    uint32_t px0 = cur.first_pixel + plan.pix_chunk;
    uint32_t s0 = cur.s_rel;
    if (px0 >= plan.npix) {
        px0 = 0;
        s0 += plan.S;
    }
    if (s0 >= plan.spp) {
        cur.num_paths = 0;
        *c = cur;
        return;
    }
    *c = cursor_at(plan, px0, s0, base);
}

__global__ void k_count_from_cursor(uint32_t* count, const BatchCursor* c) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *count = c->num_paths;
}

}  // namespace xt

// ---------------------------------------------------------------- unified batches

namespace xt {

// Window [0, window) of the batch.
__global__ void k_window_init(MultiBatch mb) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    MultiCursor c{};
    c.g0 = 0;
    c.n = (uint32_t)min((uint64_t)mb.window, mb.total_paths);
    *mb.cursor = c;
}

// The next window (n = 0 past the end).
__global__ void k_window_advance(MultiBatch mb) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    MultiCursor c = *mb.cursor;
    c.g0 += mb.window;
    c.n = c.g0 < mb.total_paths ? (uint32_t)min((uint64_t)mb.window, mb.total_paths - c.g0) : 0u;
    *mb.cursor = c;
}

// The items the window overlaps and their accumulation units: item
// first_item + j accumulates min(npix, its paths in the window) pixels,
// numbered from units[j].
__global__ void k_window_plan(MultiBatch mb) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    MultiCursor c = *mb.cursor;
    const uint64_t lo = c.g0, hi = c.g0 + c.n;
    uint32_t k = 0;
    while (k < mb.num_items && mb.items[k].path_base + mb.items[k].paths <= lo) ++k;
    c.first_item = k;
    uint32_t j = 0, u = 0;
    for (; c.n > 0 && k < mb.num_items && mb.items[k].path_base < hi; ++k, ++j) {
        const MultiItem& it = mb.items[k];
        const uint64_t a = max(it.path_base, lo), b = min(it.path_base + it.paths, hi);
        mb.units[j] = u;
        u += (uint32_t)min((uint64_t)it.npix, b - a);
    }
    mb.units[j] = u;
    c.num_overlap = j;
    *mb.cursor = c;
}

__global__ void k_count_from_window(uint32_t* count, const MultiCursor* c) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *count = c->n;
}

// The window's overlapping item holding window path id (largest j with
// path_base <= g0 + id).
__device__ __forceinline__ uint32_t window_item(const MultiBatch& mb, const MultiCursor& c, uint32_t id) {
    const uint64_t g = c.g0 + id;
    uint32_t lo = c.first_item, hi = c.first_item + c.num_overlap - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (mb.items[mid].path_base <= g) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Camera rays of the window's paths (k_generate per item).
__global__ __launch_bounds__(256) void k_generate_multi(MultiBatch mb, PathQueue q, float4* __restrict__ radiance) {
    const MultiCursor c = *mb.cursor;
    for (uint32_t id = blockIdx.x * blockDim.x + threadIdx.x; id < c.n; id += gridDim.x * blockDim.x) {
        const uint32_t k = window_item(mb, c, id);
        const MultiItem& it = mb.items[k];
        const uint64_t local = c.g0 + id - it.path_base;
        const uint32_t s_local = (uint32_t)(local / it.npix);
        const uint32_t pixel = (uint32_t)(local - (uint64_t)s_local * it.npix);
        const WaveParams& wp = it.wp;
        f3 o, d;
        camera_ray(wp, pixel, it.spp_offset + s_local, &o, &d);
        q.o[id] = make_float4(o.x, o.y, o.z, 0.0f);   // e and radiance: implied by vertex 1, as above
        q.d[id] = make_float4(d.x, d.y, d.z, __uint_as_float(id));
        q.w[id] = make_float4(1.0f, 1.0f, 1.0f, __uint_as_float(1u));
        mb.item_of[id] = k;
    }
}

// Path id -> (pixel, sample) of a unified batch's path.
struct ItemMap {
    const MultiItem& it;
    uint64_t g0;
    __device__ __forceinline__ uint2 operator()(uint32_t id) const {
        const uint64_t local = g0 + id - it.path_base;
        const uint32_t s_local = (uint32_t)(local / it.npix);
        return make_uint2((uint32_t)(local - (uint64_t)s_local * it.npix), it.spp_offset + s_local);
    }
};

// The shade step of a unified batch: each entry with its item's parameters
// and scene (unguided).
template <bool NMAP>
__global__ __launch_bounds__(shade_block(false, NMAP), NMAP ? 1 : 4) void k_shade_multi(MultiBatch mb, PathQueue qin,
                                                             const uint32_t* __restrict__ count_in,
                                                             const float4* __restrict__ hits, PathQueue qout,
                                                             unsigned long long* __restrict__ counts_out, ShadowQueue sq,
                                                             float4* __restrict__ radiance, float4* __restrict__ pending) {
    const uint32_t n = *count_in;
    const uint64_t g0 = mb.cursor->g0;
    const uint32_t stride = gridDim.x * blockDim.x;
    constexpr int BLOCK = shade_block(false, NMAP);
    __shared__ uint32_t append_lds[2 * (BLOCK / 64) + 2];
    const GuideRender gr{};
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += stride) {
        const uint32_t i = base + threadIdx.x;
        ShadeOut o;
        if (i < n) {
            const MultiItem& it = mb.items[mb.item_of[__float_as_uint(qin.d[i].w)]];
            const DevScene& sc = mb.scenes[it.scene];
            shade_entry<false, NMAP, false>(it.wp, sc, shade_const(it.wp, sc), qin, hits, radiance, pending, gr, i,
                                     ItemMap{it, g0}, o);
        }
        shade_emit<false, BLOCK>(o, qout, counts_out, sq, gr, append_lds);
    }
}
template <bool NMAP>
__global__ __launch_bounds__(shade_block(false, NMAP), NMAP ? 1 : 4) void k_shade_multi_open(MultiBatch mb, PathQueue qin,
                                                             const uint32_t* __restrict__ count_in,
                                                             const float4* __restrict__ hits, PathQueue qout,
                                                             unsigned long long* __restrict__ counts_out, ShadowQueue sq,
                                                             float4* __restrict__ radiance, float4* __restrict__ pending) {
    constexpr int BLOCK = shade_block(false, NMAP);
    __shared__ uint32_t append_lds[2 * (BLOCK / 64) + 2], list[2 * BLOCK], wave_hits[BLOCK / 64];
    const uint64_t g0 = mb.cursor->g0;
    const GuideRender gr{};
    shade_open<BLOCK>(
        *count_in, hits, qout, counts_out, sq, append_lds, list, wave_hits,
        [&](uint32_t i) {
            const MultiItem& it = mb.items[mb.item_of[__float_as_uint(qin.d[i].w)]];
            const DevScene& sc = mb.scenes[it.scene];
            ShadeOut o;
            shade_entry<false, NMAP, false, Rays::MISS>(it.wp, sc, shade_const(it.wp, sc), qin, hits, radiance, pending, gr, i,
                                                        ItemMap{it, g0}, o);
        },
        [&](uint32_t i, ShadeOut& o) {
            const MultiItem& it = mb.items[mb.item_of[__float_as_uint(qin.d[i].w)]];
            const DevScene& sc = mb.scenes[it.scene];
            shade_entry<false, NMAP, false, Rays::HIT>(it.wp, sc, shade_const(it.wp, sc), qin, hits, radiance, pending, gr, i,
                                                       ItemMap{it, g0}, o);
        });
}
template __global__ void k_shade_multi_open<false>(MultiBatch, PathQueue, const uint32_t*, const float4*, PathQueue,
                                                   unsigned long long*, ShadowQueue, float4*, float4*);
template __global__ void k_shade_multi_open<true>(MultiBatch, PathQueue, const uint32_t*, const float4*, PathQueue,
                                                  unsigned long long*, ShadowQueue, float4*, float4*);
template __global__ void k_shade_multi<false>(MultiBatch, PathQueue, const uint32_t*, const float4*, PathQueue,
                                              unsigned long long*, ShadowQueue, float4*, float4*);
template __global__ void k_shade_multi<true>(MultiBatch, PathQueue, const uint32_t*, const float4*, PathQueue,
                                             unsigned long long*, ShadowQueue, float4*, float4*);

// Any-hit for a unified batch's shadow queue, each ray in its item's scene.
// 8 waves per SIMD, without spilling.
template <bool DYN>
__global__ __launch_bounds__(TRACE_BLOCK, 8) void k_shadow_multi(ShadowQueue sq, const uint32_t* __restrict__ count,
                                                              float4* __restrict__ radiance, float4* __restrict__ pending,
                                                              uint32_t* __restrict__ ovf, uint32_t* __restrict__ dyn,
                                                              const uint32_t* __restrict__ item_of,
                                                              const MultiItem* __restrict__ items) {
    __shared__ uint32_t lds[TRACE_LDS_DEPTH * TRACE_BLOCK];
    const uint32_t n = *count;
    const size_t nthreads = (size_t)gridDim.x * blockDim.x;
    const size_t gtid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t* my_lds = lds + threadIdx.x;
    uint32_t* my_ovf = ovf ? ovf + gtid : nullptr;
    const uint32_t nwaves = (uint32_t)(nthreads / 64), wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(gtid / 64));
    RayChunks ch = chunks_first<DYN>(wave, nwaves, n);
    VisitCount vc;
    RayPre r;
    Trav t;
    TravView view{nullptr, nullptr, 0u};
    trace_queue<true, TRACE_LDS_DEPTH, false, DYN>(
        ch, dyn, view, r, t, nullptr, my_lds, my_ovf, nthreads, vc,
        [&](uint32_t i) {
            const float4 o4 = sq.o[i], d4 = sq.d[i];
            const MultiItem& it = items[item_of[__float_as_uint(d4.w)]];
            view.nodes = it.nodes;
            view.tris = it.tris;
            r = ray_setup(xyz(o4), xyz(d4));
            trav_init(t, o4.w);
        },
        [&](uint32_t i, bool occ) { shadow_record(sq, i, occ, radiance, pending); });
    if constexpr (DYN) chunks_release(dyn);
}
template __global__ void k_shadow_multi<false>(ShadowQueue, const uint32_t*, float4*, float4*, uint32_t*, uint32_t*,
                                               const uint32_t*, const MultiItem*);
template __global__ void k_shadow_multi<true>(ShadowQueue, const uint32_t*, float4*, float4*, uint32_t*, uint32_t*,
                                              const uint32_t*, const MultiItem*);

// A round's extension rays and the shadow rays of the round before, which do
// not depend on each other, in one launch: a launch lasts as long as its slowest
// rays, so below some millions of paths two launches end with two stretches of
// a nearly idle chip, and below half a million one queue does not fill it at
// all.  16 rooms at 128 x 128 in one batch 3.80 -> 2.80 ms, Cornell box at 1 M
// paths 1511 -> 1247 us, 100 k triangle room at 3.7 M 12.33 -> 10.88 ms (guided
// 9.17 -> 7.68), normal-mapped plane 8.30 -> 7.96, 1080p field at 132 M 58.9 ->
// 58.3.  A path's contributions are added in the same order: its shadow ray
// still ends before its next vertex is shaded.
// DYN: a wave takes chunks of extension rays while there are any, then of
// shadow rays.  Otherwise the two queues are one row of rays with an even
// share per wave, and only the wave at the seam traces both kinds.
template <bool MULTI, bool DYN>
__global__ __launch_bounds__(TRACE_BLOCK, DYN && MULTI ? 7 : 8) void k_trace_shadow(
    DevScene sc, const float4* __restrict__ ray_o, const float4* __restrict__ ray_d, float4* __restrict__ hits, ShadowQueue sq,
    uint32_t* __restrict__ counts, int cur, float4* __restrict__ radiance, float4* __restrict__ pending,
    uint32_t* __restrict__ ovf, uint32_t* __restrict__ dyn, uint32_t* __restrict__ counts_out,
    const uint32_t* __restrict__ item_of, const MultiItem* __restrict__ items) {
    __shared__ uint32_t lds[TRACE_LDS_DEPTH * TRACE_BLOCK];
    const uint32_t np = *path_count(counts, cur), ns = *shadow_count(counts, cur);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        // the lengths to the host's pinned ring, and the next round's queues
        // (last read by the previous round) emptied
        if (counts_out) {
            *path_count(counts_out, cur) = np;
            *shadow_count(counts_out, cur) = ns;
        }
        *pair_count(counts, 1 - cur) = 0ull;
    }
    __shared__ float4 top[MULTI ? 1 : TOP_F4];
    if constexpr (!MULTI) stage_top_nodes(top, sc);
    const size_t nthreads = (size_t)gridDim.x * blockDim.x;
    const size_t gtid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t* my_lds = lds + threadIdx.x;
    uint32_t* my_ovf = ovf ? ovf + gtid : nullptr;
    const uint32_t nwaves = (uint32_t)(nthreads / 64), wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(gtid / 64));
    RayChunks ext, sha;
    if constexpr (DYN) {
        ext = chunks_first<true>(wave, nwaves, np);
        sha = chunks_queued(nwaves, ns);
    } else {
        chunks_joint(wave, nwaves, np, ns, &ext, &sha);
    }
    VisitCount vc;
    auto scene_of = [&](uint32_t id, TravView& view) {
        if constexpr (MULTI) {
            const MultiItem& it = items[item_of[id]];
            view.nodes = it.nodes;
            view.tris = it.tris;
        }
    };
    auto trace = [&](const auto& sv, TravView& view) {
        RayPre r;
        Trav t;
        trace_queue<false, TRACE_LDS_DEPTH, false, DYN>(
            ext, dyn, sv, r, t, MULTI ? nullptr : top, my_lds, my_ovf, nthreads, vc,
            [&](uint32_t i) {
                const float4 d4 = ray_d[i];
                scene_of(__float_as_uint(d4.w), view);
                r = ray_setup(xyz(ray_o[i]), xyz(d4));
                trav_init(t, INFINITY);   // tMax = Infinity (PathTracer.h:167)
            },
            [&](uint32_t i, bool) { hits[i] = hit_record(t, t.best_slot); });
    };
    auto trace_shadow = [&](const auto& sv, TravView& view) {
        RayPre r;
        Trav t;
        trace_queue<true, TRACE_LDS_DEPTH, false, DYN>(
            sha, dyn + 2, sv, r, t, MULTI ? nullptr : top, my_lds, my_ovf, nthreads, vc,
            [&](uint32_t i) {
                const float4 o4 = sq.o[i], d4 = sq.d[i];
                scene_of(__float_as_uint(d4.w), view);
                r = ray_setup(xyz(o4), xyz(d4));
                trav_init(t, o4.w);
            },
            [&](uint32_t i, bool occ) { shadow_record(sq, i, occ, radiance, pending); });
    };
    TravView view{nullptr, nullptr, 0u}, shadow_view{nullptr, nullptr, 0u};
    if constexpr (MULTI) {
        trace(view, view);
        trace_shadow(shadow_view, shadow_view);
    } else {
        trace(sc, view);
        trace_shadow(sc, shadow_view);
    }
    if constexpr (DYN) {
        chunks_release(dyn);
        chunks_release(dyn + 2);
    }
}
#define XT_INST_TRACE_SHADOW(MULTI, DYN)                                                                              \
    template __global__ void k_trace_shadow<MULTI, DYN>(DevScene, const float4*, const float4*, float4*, ShadowQueue,  \
                                                        uint32_t*, int, float4*, float4*, uint32_t*, uint32_t*,        \
                                                        uint32_t*, const uint32_t*, const MultiItem*);
XT_INST_TRACE_SHADOW(false, false)
XT_INST_TRACE_SHADOW(false, true)
XT_INST_TRACE_SHADOW(true, false)
XT_INST_TRACE_SHADOW(true, true)
#undef XT_INST_TRACE_SHADOW

// film[pixel] += the window's samples of that pixel, in sample order, for
// every item the window overlaps (one thread per item pixel).
__global__ __launch_bounds__(256) void k_accumulate_multi(MultiBatch mb, const float4* __restrict__ radiance) {
    const MultiCursor c = *mb.cursor;
    if (c.n == 0) return;
    const uint32_t total = mb.units[c.num_overlap];
    for (uint32_t u = blockIdx.x * blockDim.x + threadIdx.x; u < total; u += gridDim.x * blockDim.x) {
        uint32_t lo = 0, hi = c.num_overlap - 1;
        while (lo < hi) {
            const uint32_t mid = (lo + hi + 1) >> 1;
            if (mb.units[mid] <= u) lo = mid;
            else hi = mid - 1;
        }
        const MultiItem& it = mb.items[c.first_item + lo];
        const uint64_t a = max(it.path_base, c.g0), b = min(it.path_base + it.paths, c.g0 + c.n);
        const uint64_t first = a - it.path_base + (u - mb.units[lo]);   // local index of this pixel's first sample
        const uint64_t last = b - it.path_base;
        const uint32_t pixel = (uint32_t)(first % it.npix);
        const size_t o = 3 * (size_t)pixel;
        if (it.film_f64) {
            double* f = (double*)it.film;
            double rr = f[o], gg = f[o + 1], bb = f[o + 2];
            for (uint64_t l = first; l < last; l += it.npix) {
                const float4 L = radiance[it.path_base + l - c.g0];
                rr += (double)L.x;
                gg += (double)L.y;
                bb += (double)L.z;
            }
            f[o] = rr;
            f[o + 1] = gg;
            f[o + 2] = bb;
        } else {
            float* f = (float*)it.film;
            float rr = f[o], gg = f[o + 1], bb = f[o + 2];
            for (uint64_t l = first; l < last; l += it.npix) {
                const float4 L = radiance[it.path_base + l - c.g0];
                rr += L.x;
                gg += L.y;
                bb += L.z;
            }
            f[o] = rr;
            f[o + 1] = gg;
            f[o + 2] = bb;
        }
    }
}

// ---------------------------------------------------------------- whole paths in one launch

// Paths followed from their camera ray (or from where the queue left them) to
// their end in one launch: a lane keeps its path's state in registers and
// loops over shadow ray, extension ray and shade step; lanes whose path has
// ended take the next path of the wave's chunk.  The same functions in the
// same order per path as the queued kernels, so the same radiance.
//
// Between vertices the wave traces every path's two rays to their ends, then
// shades together.  A full wave's lane traces them one after the other (going
// on to its extension ray as soon as WALK_SWITCH lanes, or all that are left,
// have their shadow ray done).  With at most 32 paths -- few in all, or the
// last of a wave, moved together -- lane l + 32 traces the shadow ray while
// lane l traces the extension ray: such a wave's time is the chain of its
// slowest path, some 17 us of traversal and 14 of shading a vertex (1 k
// triangles), where one ray after the other took 40 us.  96 x 64: 373 -> 293 us;
// 800 x 800, paths ended by roulette alone: 2.83 -> 2.55 ms.
#ifndef XT_WALK_SWITCH
#define XT_WALK_SWITCH 8
#endif
template <bool QUEUE, bool NMAP, bool MULTI>
__global__ __launch_bounds__(TRACE_BLOCK, NMAP ? WALK_WAVES_NMAP : WALK_WAVES) void k_walk(WalkArgs a) {
    __shared__ uint32_t lds[TRACE_LDS_DEPTH * TRACE_BLOCK];
    __shared__ float4 top[TOP_F4];
    __shared__ uint32_t counted[2];
    const WaveParams& wp0 = a.wp;
    const MultiBatch& mb = a.mb;
    if (threadIdx.x < 2) counted[threadIdx.x] = 0u;
    if constexpr (!MULTI) stage_top_nodes(top, *a.scene);
    __syncthreads();
    uint32_t n = QUEUE ? *a.count : MULTI ? mb.cursor->n : batch_of(wp0).num_paths;
    if (a.overrun && *a.overrun) n = 0u;   // the render has failed
    const size_t nthreads = (size_t)gridDim.x * blockDim.x;
    const size_t gtid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t* my_lds = lds + threadIdx.x;
    uint32_t* my_ovf = a.ovf ? a.ovf + gtid : nullptr;
    const uint32_t nwaves = (uint32_t)(nthreads / 64), wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(gtid / 64));
    const uint32_t lanes = a.lanes, lane = __lane_id();
    const uint64_t below = (1ull << lane) - 1ull;
    RayChunks ch = chunks_first<true>(wave, nwaves, n, lanes);
    const GuideRender gr{};
    const CursorMap cmap{wp0};
    ShadeConst c0;
    if constexpr (!MULTI) c0 = shade_const(wp0, *a.scene);
    // the lane's path: its next extension ray, the sample that made it, the
    // radiance so far and the light sample its shadow ray decides on
    bool alive = false, has_ext = false, has_sh = false;
    uint32_t id = 0, v = 0, item = 0, n_ext = 0, n_sh = 0;
    f3 eo = splat(0.0f), ed = eo, weight = eo, meval = eo, rad = eo, c = eo, so = eo, sd = eo;
    float pdf = 0.0f, pe = 0.0f, stmax = 0.0f;
    enum { IDLE, SHADOW, EXTEND, SWITCH };   // SWITCH: shadow ray done, extension ray next
    bool pair = lanes <= 32;   // two lanes per path
    RayPre r;
    Trav t;
    TravView view{nullptr, nullptr, 0u};
    while (true) {
        uint64_t busy = wave_ballot(alive);
        const uint32_t nidle = lanes - wave_count(busy);
        const bool refill = busy == 0 || nidle * 4 >= lanes;
        if (refill && ch.next >= ch.end && !ch.exhausted) chunks_refill(ch, a.dyn);
        if (refill && ch.next < ch.end) {
            const uint32_t my = ch.next + (uint32_t)__popcll(~busy & below);
            if (!alive && lane < lanes && my < ch.end) {
                if constexpr (QUEUE) {
                    const float4 o4 = a.q.o[my], d4 = a.q.d[my], w4 = a.q.w[my];
                    id = __float_as_uint(d4.w);
                    const uint32_t vf = __float_as_uint(w4.w);
                    v = vf & 0xFFFFFFu;
                    const bool has_pend = ((vf >> 24) & QF_PENDING) != 0;
                    const float4 e4 = v > 1 ? a.q.e[my] : make_float4(1.0f, 1.0f, 1.0f, 0.0f);
                    pdf = o4.w;
                    pe = e4.w;
                    meval = xyz(e4);
                    weight = xyz(w4);
                    rad = v > 1 ? xyz(a.radiance[id]) : splat(0.0f);
                    c = has_pend ? xyz(a.pending[id]) : splat(0.0f);
                    eo = xyz(o4);
                    ed = xyz(d4);
                } else {
                    id = my;
                    if constexpr (MULTI) {
                        const MultiCursor mc = *mb.cursor;
                        item = window_item(mb, mc, id);
                        const MultiItem& it = mb.items[item];
                        const uint2 ps = ItemMap{it, mc.g0}(id);
                        camera_ray(it.wp, ps.x, ps.y, &eo, &ed);
                    } else {
                        const uint2 ps = cmap(id);
                        camera_ray(wp0, ps.x, ps.y, &eo, &ed);
                    }
                    v = 1;
                    pdf = pe = 0.0f;
                    weight = meval = splat(1.0f);
                    rad = c = splat(0.0f);
                }
                if constexpr (MULTI) {
                    view.nodes = mb.items[item].nodes;
                    view.tris = mb.items[item].tris;
                }
                alive = has_ext = true;
                has_sh = false;
            }
            ch.next = min(ch.next + nidle, ch.end);
            busy = wave_ballot(alive);
        }
        if (busy == 0) break;
        if (!pair && ch.exhausted && ch.next >= ch.end && wave_count(busy) <= 32) {
            // the wave's last paths, moved to its first lanes
            pair = true;
            uint32_t* const from = lds + (threadIdx.x & ~63u);   // the stacks are empty here
            if (alive) from[__popcll(busy & below)] = lane;
            const bool keep = lane < wave_count(busy);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const int src = keep ? (int)from[lane] : (int)lane;
            auto move3 = [&](f3 x) { return mk(__shfl(x.x, src), __shfl(x.y, src), __shfl(x.z, src)); };
            eo = move3(eo);
            ed = move3(ed);
            weight = move3(weight);
            meval = move3(meval);
            rad = move3(rad);
            c = move3(c);
            so = move3(so);
            sd = move3(sd);
            pdf = __shfl(pdf, src);
            pe = __shfl(pe, src);
            stmax = __shfl(stmax, src);
            id = __shfl(id, src);
            v = __shfl(v, src);
            if constexpr (MULTI) {
                item = __shfl(item, src);
                view.nodes = mb.items[item].nodes;
                view.tris = mb.items[item].tris;
            }
            const uint32_t flags = __shfl((uint32_t)has_ext | (uint32_t)has_sh << 1, src);
            alive = keep;
            has_ext = keep && (flags & 1u);
            has_sh = keep && (flags & 2u);
        }
        // the rays of this vertex: a path's light sample c is added now (a path
        // that ends) or at its next vertex, unless the shadow ray is blocked
        int mode = !alive ? IDLE : has_sh && !pair ? SHADOW : has_ext ? EXTEND : IDLE;
        bool occluded = false;
        n_sh += alive && has_sh ? 1u : 0u;
        f3 ro = mode == SHADOW ? so : eo, rd = mode == SHADOW ? sd : ed;
        float rt = mode == SHADOW ? stmax : INFINITY;   // extension rays: tMax = Infinity (PathTracer.h:167)
        if (pair) {
            const int owner = (int)(lane & 31u);
            const bool theirs = __shfl((int)(alive && has_sh), owner) != 0;
            const f3 o2 = mk(__shfl(so.x, owner), __shfl(so.y, owner), __shfl(so.z, owner));
            const f3 d2 = mk(__shfl(sd.x, owner), __shfl(sd.y, owner), __shfl(sd.z, owner));
            const float t2 = __shfl(stmax, owner);
            if (lane >= 32 && theirs) {
                mode = SHADOW;
                ro = o2;
                rd = d2;
                rt = t2;
            }
            if constexpr (MULTI) {
                const uint32_t it2 = __shfl(item, owner);
                if (lane >= 32 && theirs) {
                    view.nodes = mb.items[it2].nodes;
                    view.tris = mb.items[it2].tris;
                }
            }
        }
        n_ext += mode == EXTEND ? 1u : 0u;
        if (mode != IDLE) {
            r = ray_setup(ro, rd);
            trav_init(t, rt);
        }
        while (true) {
            const uint64_t tracing = __ballot(mode == SHADOW || mode == EXTEND);
            const uint64_t waiting = __ballot(mode == SWITCH);
            if ((tracing | waiting) == 0) break;
            if (tracing == 0 || __popcll(waiting) >= XT_WALK_SWITCH) {
                if (mode == SWITCH) {
                    r = ray_setup(eo, ed);
                    trav_init(t, INFINITY);
                    mode = EXTEND;
                    ++n_ext;
                }
            }
            const bool active = mode == SHADOW || mode == EXTEND;
            bool occ = false, done;
            if constexpr (MULTI)
                done = trav_step_mixed<TRACE_LDS_DEPTH>(active, mode == SHADOW, view, r, t, top, my_lds, TRACE_BLOCK, my_ovf,
                                                        nthreads, &occ);
            else
                done = trav_step_mixed<TRACE_LDS_DEPTH>(active, mode == SHADOW, *a.scene, r, t, top, my_lds, TRACE_BLOCK,
                                                        my_ovf, nthreads, &occ);
            if (active && done) {
                if (mode == SHADOW) occluded = occ;
                mode = mode == SHADOW && has_ext && alive ? SWITCH : IDLE;
            }
        }
        if (pair) occluded = (wave_ballot(occluded) >> (lane & 31u) >> 32) & 1ull;
        if (alive && has_sh) {
            if (occluded) c = splat(0.0f);
            if (!has_ext) {
                if (!occluded) rad += c;
                a.radiance[id] = f4(rad, 0.0f);
                alive = false;
            }
        }
        if (alive) {
            VertexIn in;
            in.d = ed;
            in.weight = weight;
            in.meval = meval;
            in.pdf_prev = pdf;
            in.pe_prev = pe;
            in.v = v;
            in.qflags = QF_PENDING;   // c is zero without a light sample
            in.id = id;
            in.h = t.best_slot != INVALID
                       ? make_float4(t.best_t, __uint_as_float(t.best_slot), t.b0, t.b1)
                       : make_float4(INFINITY, __uint_as_float(INVALID), 0.0f, 0.0f);
            in.rad = rad;
            in.pend = c;
            ShadeOut o;
            auto put = [&](f3 x) { rad = x; };
            if constexpr (MULTI) {
                const MultiItem& it = mb.items[item];
                const DevScene& sc = mb.scenes[it.scene];
                shade_vertex<false, NMAP>(it.wp, sc, shade_const(it.wp, sc), in, gr, 0, ItemMap{it, mb.cursor->g0}, put, o);
            } else {
                shade_vertex<false, NMAP>(wp0, *a.scene, c0, in, gr, 0, cmap, put, o);
            }
            has_ext = o.push_ext;
            has_sh = o.push_sh;
            eo = o.ext_o;
            ed = o.ext_d;
            weight = o.ext_w;
            meval = o.ext_e;
            pdf = o.ext_pdf;
            pe = o.ext_pe;
            v = o.ext_v;
            c = o.sh_c;
            so = o.sh_o;
            sd = o.sh_d;
            stmax = o.sh_tmax;
            if (has_ext && v > a.max_vertex) {
                // the render fails, and no wave takes another chunk
                atomicOr(a.overrun, 1u);
                atomicMax(&a.dyn[0], ch.n);
                has_ext = has_sh = false;
            }
            if (!has_ext && !has_sh) {
                a.radiance[id] = f4(rad, 0.0f);
                alive = false;
            }
        }
    }
    if (a.rays) {
        for (int off = 32; off > 0; off >>= 1) {
            n_ext += __shfl_xor(n_ext, off);
            n_sh += __shfl_xor(n_sh, off);
        }
        if (lane == 0) {
            atomicAdd(&counted[0], n_ext);
            atomicAdd(&counted[1], n_sh);
        }
    }
    // as chunks_release; the last block to leave also hands out the ray totals
    __syncthreads();
    if (threadIdx.x == 0) {
        if (a.rays) {
            atomicAdd(&a.rays[0], (unsigned long long)counted[0]);
            atomicAdd(&a.rays[1], (unsigned long long)counted[1]);
        }
        __threadfence();
        if (atomicAdd(&a.dyn[1], 1u) == gridDim.x - 1) {
            atomicExch(&a.dyn[0], 0u);
            atomicExch(&a.dyn[1], 0u);
            if (a.rays) {
                a.rays_out[0] = atomicAdd(&a.rays[0], 0ull);
                a.rays_out[1] = atomicAdd(&a.rays[1], 0ull);
                a.rays_out[2] = a.overrun ? atomicOr(a.overrun, 0u) : 0u;
            }
        }
    }
}
template __global__ void k_walk<false, false, false>(WalkArgs);
template __global__ void k_walk<true, false, false>(WalkArgs);
template __global__ void k_walk<false, true, false>(WalkArgs);
template __global__ void k_walk<true, true, false>(WalkArgs);
template __global__ void k_walk<false, false, true>(WalkArgs);
template __global__ void k_walk<false, true, true>(WalkArgs);

}  // namespace xt
