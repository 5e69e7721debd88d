// VonMisesFisherDistribution<N> (VonMisesFisherDistribution.h:9-217) on the
// device: mixture pdf, the reference's sampler, and the EM fit
// approximateBySEM, batched over many independent distributions.  Mixtures
// travel in the reference's encoding (encode/decode, :37-58): 5 floats per
// lobe (mu.xyz, kappa, alpha), the last lobe's alpha omitted and recovered as
// 1 minus the running sum.
//
// The fit runs one wave64 per sample set when there are enough sets to fill
// the chip, else a block of several waves per set (fit_waves).  Either way
// lane l of a wave sums samples l, l + 64, ... of the set in that order and a
// butterfly of commutative adds reduces the lanes, so both forms give the
// same bits: EM stops on a signed difference, whose step count a different
// summation order would change.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "runtime.h"
#include "xt_guide.h"

using namespace xt;

namespace {

constexpr int VMF_MAX_LOBES = 16;
constexpr float VMF_PI = 3.14159265358979323846f;

__device__ __forceinline__ void vmf_decode_lobe(const float* enc, int N, int k, float acc, f3* mu, float* kappa,
                                                float* alpha) {
    *mu = mk(enc[5 * k], enc[5 * k + 1], enc[5 * k + 2]);
    *kappa = enc[5 * k + 3];
    *alpha = (k < N - 1) ? enc[5 * k + 4] : 1.0f - acc;
}

// eval (:60-66): sum_k alpha_k vMF_k(w), alphas decoded as in :47-58.
__global__ void k_vmf_eval(int N, const float* __restrict__ enc, uint32_t num_dists, const uint32_t* __restrict__ dist,
                           const float* __restrict__ dirs, uint32_t n, float* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t d = dist ? dist[i] : 0u;
    if (d >= num_dists) {
        out[i] = NAN;
        return;
    }
    const float* e = enc + (size_t)d * (5 * N - 1);
    const f3 w = mk(dirs[3 * (size_t)i], dirs[3 * (size_t)i + 1], dirs[3 * (size_t)i + 2]);
    float acc = 0.0f, v = 0.0f;
    for (int k = 0; k < N; ++k) {
        VmfLobe lb;
        vmf_decode_lobe(e, N, k, acc, &lb.mu, &lb.kappa, &lb.alpha);
        acc += lb.alpha;
        v += lb.alpha * vmf_lobe_pdf(lb, w);
    }
    out[i] = v;
}

// sample (:162-201) with uniforms (lobe choice, disk radius, disk angle, W).
__global__ void k_vmf_sample(int N, const float* __restrict__ enc, uint32_t num_dists, const uint32_t* __restrict__ dist,
                             const float* __restrict__ uni, uint32_t n, float* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t d = dist ? dist[i] : 0u;
    float* o = out + 3 * (size_t)i;
    if (d >= num_dists) {
        o[0] = o[1] = o[2] = NAN;
        return;
    }
    const float* e = enc + (size_t)d * (5 * N - 1);
    const float* u = uni + 4 * (size_t)i;
    // Sampler::randiAlongNormalizedWeights (Sampler.h:52-61): u <= running sum
    float acc = 0.0f, accum = 0.0f;
    f3 mu = mk(0, 0, 0);
    float kappa = 0.0f, alpha = 0.0f;
    int sel = N - 1;
    for (int k = 0; k < N; ++k) {
        vmf_decode_lobe(e, N, k, acc, &mu, &kappa, &alpha);
        acc += alpha;
        if (k == N - 1) break;
        accum += alpha;
        if (u[0] <= accum) {
            sel = k;
            break;
        }
    }
    (void)sel;
    if (mu.x == 0.0f && mu.y == 0.0f && mu.z == 0.0f) {
        o[0] = o[1] = o[2] = 0.0f;
        return;
    }
    const float r = sqrtf(u[1]);
    const float theta = 2.0f * VMF_PI * u[2] - VMF_PI;
    const float vx = r * cosf(theta), vy = r * sinf(theta);
    float W = 1.0f;
    if (kappa > 0.0f) W = 1.0f + powf(kappa, -1.0f) * logf(u[3] + (1.0f - u[3]) * expf(-2.0f * kappa));
    const float s = safe_sqrt(1.0f - powf(W, 2.0f));
    const Frame fr = make_frame(normalize(mu));
    const f3 g = normalize(to_world(fr, W, s * vx, s * vy));
    o[0] = g.x;
    o[1] = g.y;
    o[2] = g.z;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
    return v;
}

// approximateBySEM (:68-160) for sample sets samples[off[f] .. off[f+1]).
template <int N>
__global__ __launch_bounds__(256) void k_vmf_fit(const float* __restrict__ smp, const uint32_t* __restrict__ off,
                                                 uint32_t nfits, const float* __restrict__ init_u,
                                                 float* __restrict__ enc, int32_t* __restrict__ steps_out) {
    constexpr float KappaLimit = 1000.0f;
    constexpr int StepMax = 100000;
    constexpr float DiffThreshold = 1e-6f;
    const uint32_t nw = (gridDim.x * blockDim.x) >> 6;
    const int l = __lane_id();
    for (uint32_t f = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; f < nfits; f += nw) {
        const uint32_t b = off[f], e = off[f + 1];
        const uint32_t n = e > b ? e - b : 0u;
        f3 mu[N];
        float ka[N], al[N];
        int steps = 0;
        _Pragma("unroll") for (int j = 0; j < N; ++j) {          // default distribution (:24-35)
            mu[j] = mk(1, 0, 0);
            ka[j] = 0.0f;
            al[j] = j == 0 ? 1.0f : 0.0f;
        }
        if (n == 1) {                          // :79-86
            const f3 x = mk(smp[3 * (size_t)b], smp[3 * (size_t)b + 1], smp[3 * (size_t)b + 2]);
            _Pragma("unroll") for (int j = 0; j < N; ++j) {
                mu[j] = x;
                ka[j] = KappaLimit;
            }
        } else if (n > 1) {
            const float* iu = init_u + (size_t)2 * N * f;
            _Pragma("unroll") for (int j = 0; j < N; ++j) {      // :89-98
                const float theta = asinf(iu[2 * j]);
                const float phi = 2.0f * VMF_PI * iu[2 * j + 1] - VMF_PI;
                mu[j] = mk(cosf(theta) * cosf(phi), cosf(theta) * sinf(phi), sinf(theta));
                ka[j] = 0.5f;
                al[j] = 1.0f / N;
            }
            f3 lmu[N];
            float lka[N];
            int step = 0;
            for (step = 0; step < StepMax; ++step) {
                float sa[N];
                f3 sr[N];
                _Pragma("unroll") for (int j = 0; j < N; ++j) {
                    sa[j] = 0.0f;
                    sr[j] = mk(0, 0, 0);
                }
                for (uint32_t i = b + l; i < e; i += 64) {   // E-step (:109-120), responsibilities without alpha
                    const f3 x = mk(smp[3 * (size_t)i], smp[3 * (size_t)i + 1], smp[3 * (size_t)i + 2]);
                    float v[N];
                    float gsum = 0.0f;
                    _Pragma("unroll") for (int j = 0; j < N; ++j) {
                        VmfLobe lb{mu[j], ka[j], 0.0f};
                        v[j] = vmf_lobe_pdf(lb, x);
                        gsum += v[j];
                    }
                    _Pragma("unroll") for (int j = 0; j < N; ++j) {
                        const float z = gsum > 0.0f ? v[j] / gsum : 0.0f;
                        sa[j] += z;
                        sr[j] += z * x;
                    }
                }
                _Pragma("unroll") for (int j = 0; j < N; ++j) {          // M-step (:123-139)
                    const float a = wave_sum(sa[j]);
                    f3 r = mk(wave_sum(sr[j].x), wave_sum(sr[j].y), wave_sum(sr[j].z));
                    r = div(r, a);
                    al[j] = a / (float)n;
                    const float rl = length(r);
                    float k = (3 * rl - powf(rl, 3.0f)) / (1.0f - dot(r, r));
                    mu[j] = normalize(r);
                    if (k > KappaLimit) k = KappaLimit;
                    if (k < 0.0f) k = 0.0f;
                    ka[j] = k;
                }
                if (step > 0) {                        // :141-148
                    float diff = 0.0f;
                    _Pragma("unroll") for (int j = 0; j < N; ++j) {
                        const f3 dm = mu[j] - lmu[j];
                        diff += dot(dm, dm);
                        diff += (ka[j] - lka[j]) * 0.1f;
                    }
                    if (diff < DiffThreshold) break;
                }
                _Pragma("unroll") for (int j = 0; j < N; ++j) {
                    lmu[j] = mu[j];
                    lka[j] = ka[j];
                }
            }
            steps = step < StepMax ? step + 1 : StepMax;
        }
        if (l == 0) {                                  // encode (:37-45)
            float* o = enc + (size_t)(5 * N - 1) * f;
            _Pragma("unroll") for (int j = 0; j < N; ++j) {
                o[5 * j] = mu[j].x;
                o[5 * j + 1] = mu[j].y;
                o[5 * j + 2] = mu[j].z;
                o[5 * j + 3] = ka[j];
                if (j < N - 1) o[5 * j + 4] = al[j];
            }
            if (steps_out) steps_out[f] = steps;
        }
    }
}

// k_vmf_fit with a block of W waves per sample set.  One wave per set leaves
// the chip idle with few sets, and its E-step is a serial chain of
// ceil(n / 64) rounds of N pdfs and divisions: 96 sets of 3000 samples, 6
// lobes, took 11.5 ms a call (bound by the set of most steps, 36 us a step).
// Here wave w evaluates the responsibilities of rounds
// w, w + W, ... and leaves them in LDS beside the samples; then each of the
// 4 N sums (z, z x, z y, z z of a lobe) is one wave's, which adds the rounds
// in order and reduces its lanes: every rounding is k_vmf_fit's.  The M-step
// takes one lane per lobe of wave 0.  The same call takes 2.8 ms, 7.5 us a step:
// some 3 us of it the M-step's own chain and the barriers, the rest issue.
//
// The block has its CU to itself (152 KB of LDS): the samples of sets of up to
// 3072 stay in LDS for all steps, and the responsibilities of as many rounds
// as fit are one batch between two barriers.
template <int N, int W>
struct FitShared {
    static constexpr int SAMPLE_ROUNDS = 48;   // rounds of 64 samples kept in LDS
    // rounds of responsibilities per batch: whole turns of the W waves, at most SAMPLE_ROUNDS
    static constexpr int TURNS = (152 * 1024 - SAMPLE_ROUNDS * 768) / (N * 256 * W);
    static constexpr int ROUNDS = W * (TURNS * W > SAMPLE_ROUNDS ? SAMPLE_ROUNDS / W : TURNS);
    static_assert(TURNS >= 1 && SAMPLE_ROUNDS % W == 0, "a batch holds a round of every wave");
    float z[ROUNDS][N][64];
    float x[SAMPLE_ROUNDS][3][64];
    float sum[4 * N];
    float mu[N][3], kappa[N], norm[N];
    int stop;
};

// wave_sum with cross-lane moves in place of LDS shuffles: the same tree (from
// distance 8 on the lanes repeat, so a rotation of a row is the exchange).
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float wave_sum_dpp(float v) {
    v += __shfl_xor(v, 32);
    v += __shfl_xor(v, 16);
    v += dpp_move<0x128>(v);   // row_ror:8
    v += dpp_move<0x124>(v);   // row_ror:4
    v += dpp_move<0x122>(v);   // row_ror:2
    v += dpp_move<0x121>(v);   // row_ror:1
    return v;
}

template <int N, int W>
__global__ __launch_bounds__(64 * W) void k_vmf_fit_block(const float* __restrict__ smp, const uint32_t* __restrict__ off,
                                                          uint32_t nfits, const float* __restrict__ init_u,
                                                          float* __restrict__ enc, int32_t* __restrict__ steps_out) {
    constexpr float KappaLimit = 1000.0f;
    constexpr int StepMax = 100000;
    constexpr float DiffThreshold = 1e-6f;
    __shared__ FitShared<N, W> sh;
    const int l = __lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (uint32_t f = blockIdx.x; f < nfits; f += gridDim.x) {
        const uint32_t b = off[f], e = off[f + 1];
        const uint32_t n = e > b ? e - b : 0u;
        const uint32_t rounds = (n + 63) / 64;
        const bool resident = rounds <= (uint32_t)FitShared<N, W>::SAMPLE_ROUNDS;
        auto load_round = [&](uint32_t r, uint32_t to) {   // samples of round r, zeros past the end
            const uint32_t i = r * 64 + l;
            f3 x = mk(0, 0, 0);
            if (i < n) {
                const size_t o = 3 * ((size_t)b + i);
                x = mk(smp[o], smp[o + 1], smp[o + 2]);
            }
            sh.x[to][0][l] = x.x;
            sh.x[to][1][l] = x.y;
            sh.x[to][2][l] = x.z;
        };
        int steps = 0;
        f3 mu = mk(1, 0, 0), lmu = mu;   // lane j of wave 0: lobe j
        float ka = 0.0f, al = l == 0 ? 1.0f : 0.0f, lka = 0.0f;
        if (n == 1) {                          // :79-86
            mu = mk(smp[3 * (size_t)b], smp[3 * (size_t)b + 1], smp[3 * (size_t)b + 2]);
            ka = KappaLimit;
        } else if (n > 1) {
            if (w == 0 && l < N) {             // :89-98
                const float* iu = init_u + (size_t)2 * N * f;
                const float theta = asinf(iu[2 * l]);
                const float phi = 2.0f * VMF_PI * iu[2 * l + 1] - VMF_PI;
                mu = mk(cosf(theta) * cosf(phi), cosf(theta) * sinf(phi), sinf(theta));
                ka = 0.5f;
                al = 1.0f / N;
            }
            if (resident)
                for (uint32_t r = w; r < rounds; r += W) load_round(r, r);
            int step = 0;
            for (step = 0; step < StepMax; ++step) {
                if (w == 0 && l < N) {
                    sh.mu[l][0] = mu.x;
                    sh.mu[l][1] = mu.y;
                    sh.mu[l][2] = mu.z;
                    sh.kappa[l] = ka;
                    sh.norm[l] = ka == 0.0f ? 1.0f / (4.0f * VMF_PI) : vmf_norm(ka);   // vmf_lobe_pdf
                }
                __syncthreads();
                constexpr int CHAINS = (4 * N + W - 1) / W;
                float acc[CHAINS];
                _Pragma("unroll") for (int c = 0; c < CHAINS; ++c) acc[c] = 0.0f;
                for (uint32_t r0 = 0; r0 < rounds; r0 += FitShared<N, W>::ROUNDS) {
                    const uint32_t nr = min(rounds - r0, (uint32_t)FitShared<N, W>::ROUNDS);
                    for (uint32_t r = w; r < nr; r += W) {   // E-step (:109-120), responsibilities without alpha
                        const uint32_t rx = resident ? r0 + r : r;
                        if (!resident) load_round(r0 + r, r);
                        const bool in = (r0 + r) * 64 + l < n;
                        const f3 x = mk(sh.x[rx][0][l], sh.x[rx][1][l], sh.x[rx][2][l]);
                        float v[N];
                        float gsum = 0.0f;
                        _Pragma("unroll") for (int j = 0; j < N; ++j) {
                            const float k = sh.kappa[j];
                            const f3 m = mk(sh.mu[j][0], sh.mu[j][1], sh.mu[j][2]);
                            v[j] = k == 0.0f ? sh.norm[j] : sh.norm[j] * expf(k * (dot(x, m) - 1.0f));
                            gsum += v[j];
                        }
                        _Pragma("unroll") for (int j = 0; j < N; ++j)
                            sh.z[r][j][l] = gsum > 0.0f && in ? v[j] / gsum : 0.0f;
                    }
                    __syncthreads();
                    _Pragma("unroll") for (int c = 0; c < CHAINS; ++c) {
                        const int k = w + c * W, j = k >> 2, q = k & 3;
                        if (k >= 4 * N) break;
                        float a = acc[c];
                        const float* z = &sh.z[0][j][l];
                        if (q == 0) {
#pragma unroll 8
                            for (uint32_t r = 0; r < nr; ++r) a += z[r * N * 64];
                        } else {
                            const float* x = &sh.x[resident ? r0 : 0][q - 1][l];
#pragma unroll 8
                            for (uint32_t r = 0; r < nr; ++r) a += z[r * N * 64] * x[r * 192];
                        }
                        acc[c] = a;
                    }
                    if (r0 + nr < rounds) __syncthreads();   // the next batch overwrites z and x
                }
                _Pragma("unroll") for (int c = 0; c < CHAINS; ++c) {
                    const int k = w + c * W;
                    if (k >= 4 * N) break;
                    const float a = wave_sum_dpp(acc[c]);
                    if (l == 0) sh.sum[k] = a;
                }
                __syncthreads();
                if (w == 0) {
                    float d0 = 0.0f, d1 = 0.0f;
                    if (l < N) {                       // M-step (:123-139)
                        const float a = sh.sum[4 * l];
                        f3 r = mk(sh.sum[4 * l + 1], sh.sum[4 * l + 2], sh.sum[4 * l + 3]);
                        r = div(r, a);
                        al = a / (float)n;
                        const float rl = length(r);
                        float k = (3 * rl - powf(rl, 3.0f)) / (1.0f - dot(r, r));
                        mu = normalize(r);
                        if (k > KappaLimit) k = KappaLimit;
                        if (k < 0.0f) k = 0.0f;
                        ka = k;
                        const f3 dm = mu - lmu;
                        d0 = dot(dm, dm);
                        d1 = (ka - lka) * 0.1f;
                    }
                    float diff = 0.0f;                 // :141-148
                    _Pragma("unroll") for (int j = 0; j < N; ++j) {
                        diff += __shfl(d0, j);
                        diff += __shfl(d1, j);
                    }
                    lmu = mu;
                    lka = ka;
                    if (l == 0) sh.stop = step > 0 && diff < DiffThreshold;
                }
                __syncthreads();
                if (sh.stop) break;
            }
            steps = step < StepMax ? step + 1 : StepMax;
        }
        if (w == 0 && l < N) {                         // encode (:37-45)
            float* o = enc + (size_t)(5 * N - 1) * f + 5 * l;
            o[0] = mu.x;
            o[1] = mu.y;
            o[2] = mu.z;
            o[3] = ka;
            if (l < N - 1) o[4] = al;
            if (l == 0 && steps_out) steps_out[f] = steps;
        }
        __syncthreads();   // sh.stop is read before the next set writes it
    }
}

// Whether a call takes a block per set.  A block needs sets with work for its
// waves, and fewer sets than a wave each would fill the chip with.  6 lobes,
// a wave against a block per set: 1024 sets of 256 samples 4.6 / 2.1 ms, 400
// of 256 3.3 / 1.4 ms, 1024 of 3000 19.2 / 6.1 ms, 1 of 3000 1.7 / 0.46 ms;
// 1 lobe, 96 of 3000 (2 steps) 0.26 / 0.25 ms.  The line lies on the safe side of
// where the forms cross, not there: with 6 and 12 lobes the block is still the
// faster one at 2048 sets of 256 (8.5 / 5.8, 43 / 14 ms) and of 64 (5.1 / 3.2, 5.2 /
// 4.5), the wave at 8192 sets of 64 (8.3 / 9.8, 13.4 / 14.7); with one lobe they
// differ by 10% from 64 sets on, the wave ahead.
constexpr int FIT_BLOCK_WAVES = 16;
bool fit_in_blocks(uint32_t nfits, uint32_t num_samples) {
    return nfits <= 1024 && num_samples / nfits >= 256;
}

template <int N>
void launch_fit(bool blocks, hipStream_t st, const float* smp, const uint32_t* off, uint32_t nfits, const float* iu,
                float* enc, int32_t* steps) {
    if (blocks) {
        hipLaunchKernelGGL((k_vmf_fit_block<N, FIT_BLOCK_WAVES>), dim3(nfits), dim3(64 * FIT_BLOCK_WAVES), 0, st, smp, off,
                           nfits, iu, enc, steps);
        return;
    }
    const uint32_t grid = std::max(1u, std::min((nfits + 3) / 4, 4096u));
    hipLaunchKernelGGL(k_vmf_fit<N>, dim3(grid), dim3(256), 0, st, smp, off, nfits, iu, enc, steps);
}

using FitLauncher = void (*)(bool, hipStream_t, const float*, const uint32_t*, uint32_t, const float*, float*,
                             int32_t*);
const FitLauncher kFit[VMF_MAX_LOBES + 1] = {nullptr,         launch_fit<1>,  launch_fit<2>,  launch_fit<3>,
                                             launch_fit<4>,   launch_fit<5>,  launch_fit<6>,  launch_fit<7>,
                                             launch_fit<8>,   launch_fit<9>,  launch_fit<10>, launch_fit<11>,
                                             launch_fit<12>,  launch_fit<13>, launch_fit<14>, launch_fit<15>,
                                             launch_fit<16>};

// Device copies of host arrays (or the caller's device pointers).
struct Staged {
    xt_device* dev;
    hipStream_t st;
    std::vector<void*> owned;
    Staged(xt_device* d, hipStream_t stream) : dev(d), st(stream) {}
    ~Staged() {
        if (!owned.empty()) hipStreamSynchronize(st);   // also after an error halfway
        for (void* p : owned) dev->stage.give(p);
    }
    template <class T>
    hipError_t in(const T* src, size_t count, bool on_device, const T** dst) {
        if (on_device || count == 0 || !src) {
            *dst = src;
            return hipSuccess;
        }
        T* d = nullptr;
        hipError_t e = dev->stage.take(count * sizeof(T), (void**)&d);
        if (e != hipSuccess) return e;
        owned.push_back(d);
        *dst = d;
        return hipMemcpyAsync(d, src, count * sizeof(T), hipMemcpyHostToDevice, st);
    }
    template <class T>
    hipError_t out(T* user, size_t count, bool on_device, T** dst) {
        if (on_device || count == 0) {
            *dst = user;
            return hipSuccess;
        }
        T* d = nullptr;
        hipError_t e = dev->stage.take(count * sizeof(T), (void**)&d);
        if (e != hipSuccess) return e;
        owned.push_back(d);
        *dst = d;
        return hipSuccess;
    }
};

xt_status vmf_check(xt_device* dev, uint32_t num_lobes) {
    if (!dev) return xt_fail(XT_ERR_INVALID_ARGUMENT, "device is NULL");
    if (num_lobes < 1 || num_lobes > (uint32_t)VMF_MAX_LOBES)
        return xt_fail(XT_ERR_INVALID_ARGUMENT, "num_lobes must be in [1, 16]");
    XT_HIP(hipSetDevice(dev->ordinal));
    return XT_OK;
}

}  // namespace

extern "C" {

xt_status xt_vmf_eval(xt_device* dev, uint32_t num_lobes, const float* encoded, uint32_t num_dists,
                      const uint32_t* dist_of_dir, const float* dirs, uint32_t n, float* pdf, int on_device) {
    xt_status s = vmf_check(dev, num_lobes);
    if (s != XT_OK) return s;
    if (n == 0) return XT_OK;
    if (!encoded || !dirs || !pdf || num_dists == 0) return xt_fail(XT_ERR_INVALID_ARGUMENT, "NULL or empty argument");
    const hipStream_t st = hipStreamPerThread;
    Staged sg(dev, st);
    const float *d_enc, *d_dirs;
    const uint32_t* d_dist;
    float* d_out;
    const size_t E = 5 * num_lobes - 1;
    XT_HIP(sg.in(encoded, E * num_dists, on_device, &d_enc));
    XT_HIP(sg.in(dist_of_dir, dist_of_dir ? (size_t)n : 0, on_device, &d_dist));
    XT_HIP(sg.in(dirs, 3 * (size_t)n, on_device, &d_dirs));
    XT_HIP(sg.out(pdf, n, on_device, &d_out));
    hipLaunchKernelGGL(k_vmf_eval, dim3((n + 255) / 256), dim3(256), 0, st, (int)num_lobes, d_enc, num_dists, d_dist,
                       d_dirs, n, d_out);
    XT_HIP(hipGetLastError());
    if (!on_device) XT_HIP(hipMemcpyAsync(pdf, d_out, n * sizeof(float), hipMemcpyDeviceToHost, st));
    XT_HIP(hipStreamSynchronize(st));
    return XT_OK;
}

xt_status xt_vmf_sample(xt_device* dev, uint32_t num_lobes, const float* encoded, uint32_t num_dists,
                        const uint32_t* dist_of_sample, const float* uniforms, uint32_t n, float* dirs, int on_device) {
    xt_status s = vmf_check(dev, num_lobes);
    if (s != XT_OK) return s;
    if (n == 0) return XT_OK;
    if (!encoded || !uniforms || !dirs || num_dists == 0) return xt_fail(XT_ERR_INVALID_ARGUMENT, "NULL or empty argument");
    const hipStream_t st = hipStreamPerThread;
    Staged sg(dev, st);
    const float *d_enc, *d_u;
    const uint32_t* d_dist;
    float* d_out;
    const size_t E = 5 * num_lobes - 1;
    XT_HIP(sg.in(encoded, E * num_dists, on_device, &d_enc));
    XT_HIP(sg.in(dist_of_sample, dist_of_sample ? (size_t)n : 0, on_device, &d_dist));
    XT_HIP(sg.in(uniforms, 4 * (size_t)n, on_device, &d_u));
    XT_HIP(sg.out(dirs, 3 * (size_t)n, on_device, &d_out));
    hipLaunchKernelGGL(k_vmf_sample, dim3((n + 255) / 256), dim3(256), 0, st, (int)num_lobes, d_enc, num_dists, d_dist,
                       d_u, n, d_out);
    XT_HIP(hipGetLastError());
    if (!on_device) XT_HIP(hipMemcpyAsync(dirs, d_out, 3 * (size_t)n * sizeof(float), hipMemcpyDeviceToHost, st));
    XT_HIP(hipStreamSynchronize(st));
    return XT_OK;
}

xt_status xt_vmf_fit(xt_device* dev, uint32_t num_lobes, const float* samples, uint32_t num_samples,
                     const uint32_t* offsets, uint32_t num_fits, const float* init_uniforms, float* encoded,
                     int32_t* steps, int on_device) {
    xt_status s = vmf_check(dev, num_lobes);
    if (s != XT_OK) return s;
    if (num_fits == 0) return XT_OK;
    if (!offsets || !init_uniforms || !encoded || (num_samples && !samples))
        return xt_fail(XT_ERR_INVALID_ARGUMENT, "NULL argument");
    const hipStream_t st = hipStreamPerThread;
    // the kernel reads samples[offsets[f] .. offsets[f+1]): validate the ranges
    std::vector<uint32_t> hoff(num_fits + 1);
    if (on_device) XT_HIP(hipMemcpy(hoff.data(), offsets, hoff.size() * 4, hipMemcpyDeviceToHost));
    else std::copy(offsets, offsets + num_fits + 1, hoff.begin());
    for (uint32_t f = 0; f < num_fits; ++f)
        if (hoff[f + 1] < hoff[f]) return xt_fail(XT_ERR_INVALID_ARGUMENT, "offsets must be non-decreasing");
    if (hoff[num_fits] > num_samples) return xt_fail(XT_ERR_INVALID_ARGUMENT, "offsets exceed num_samples");
    Staged sg(dev, st);
    const float *d_smp, *d_iu;
    const uint32_t* d_off;
    float* d_enc;
    int32_t* d_steps = nullptr;
    const size_t E = 5 * num_lobes - 1;
    XT_HIP(sg.in(samples, 3 * (size_t)num_samples, on_device, &d_smp));
    XT_HIP(sg.in(offsets, (size_t)num_fits + 1, on_device, &d_off));
    XT_HIP(sg.in(init_uniforms, (size_t)2 * num_lobes * num_fits, on_device, &d_iu));
    XT_HIP(sg.out(encoded, E * num_fits, on_device, &d_enc));
    if (steps) XT_HIP(sg.out(steps, num_fits, on_device, &d_steps));
    kFit[num_lobes](fit_in_blocks(num_fits, hoff[num_fits] - hoff[0]), st, d_smp, d_off, num_fits, d_iu, d_enc, d_steps);
    XT_HIP(hipGetLastError());
    if (!on_device) {
        XT_HIP(hipMemcpyAsync(encoded, d_enc, E * num_fits * sizeof(float), hipMemcpyDeviceToHost, st));
        if (steps) XT_HIP(hipMemcpyAsync(steps, d_steps, num_fits * sizeof(int32_t), hipMemcpyDeviceToHost, st));
    }
    XT_HIP(hipStreamSynchronize(st));
    return XT_OK;
}

}  // extern "C"
