// train.hip -- one training step of the avatar network on the device.
//
// Restates Testbed::train_nerf_step (instant-ngp/src/testbed_nerf.cu:
// 3176-3400) for the INSTA path, as this sequence of kernels on one stream:
//   rays      generate_training_samples_nerf (1105-1285): per ray a training
//             image ((i + rays_total) * n_images / n_rays, 1082-1103) and a
//             PCG32 stream advanced by 8 draws per ray (1143): pixel xy, a
//             draw the reference spends on motion blur, the start jitter;
//             march through the image frame's occupancy grid from
//             max(t_box, 0) + dt * jitter, at most max_steps samples; a ray
//             whose sample range would cross the cap is dropped (1239-1242)
//   deform    posed -> canonical with the frame of each ray (core.cu:442-526)
//   infer     the context's inference network (MFMA) on every marched sample
//   loss      compute_loss_kernel_train_nerf (1305-1643): product
//             transmittance T *= 1 - alpha until T < 1e-4, random background
//             (the same PCG32 stream: draws 2-4 of the ray), Huber(0.1) / 5
//             per channel, dL/d(rgb logit) = w * dL/drgb * s(1 - s),
//             dL/d(density logit) = sigma * dt * dL/drgb . (T rgb - suffix),
//             scaled by loss_scale / n_rays; the composited samples are
//             compacted into a batch of at most target_samples (1543-1560)
//   forward   on the compacted batch: hash grid (FP32, the plain encode)
//             and the MLPs on FP32 MFMA, keeping every activation the
//             backward needs, feature-major [feature][sample]
//   backward  both MLPs on FP32 MFMA over the compacted batch (ReLU masks
//             from the stored activations) into dL/dencoding, stored for
//             every level and then scattered into the hash tables: levels
//             that fit in LDS by a workgroup per level, feature and chunk
//             (FP64 LDS atomics; packed FP16 ones with FP16 gradients), larger
//             ones partitioned by table slice and accumulated slice by slice in
//             LDS the same way, or, where a table exceeds kPartMaxEntries, by
//             global atomics (FP64; packed FP16), one level per XCD at a time
//   wgrad     weight gradients dW = sum_n delta_n x_n^T as per-chunk partial
//             products on FP32 MFMA (samples as the K dimension, operands
//             staged through LDS), then a fixed-order sum over chunks:
//             deterministic MLP gradients
//   adam      Kingma & Ba with bias correction over all parameters, after
//             removing the loss scale
// Extra dims (16 per frame) enter the density MLP as 16 more inputs, 1.0 or
// the ray's frame values by the selector the deformation writes; their
// columns of W0 get gradients like the encoding's, the values themselves
// none (latent-code optimisation is off in the reference configuration).
// Training images hold sRGB colour with straight alpha, as the reference's
// 8-bit images do.  Declared simplifications against the reference: no
// density/colour regularisers, no error map, rays never masked out.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>
#include <type_traits>

#include "context.hpp"
#include "encoding.hpp"
#include "march.hpp"

namespace insta {

enum : uint32_t {
    kTRays = 0,      // rays kept (ray list length)
    kTSamples = 1,   // samples reserved
    kTLimit = 2,     // first sample of the ray that crossed the cap
    kTValid = 3,     // samples marched into the buffers
    kTUsed = 4,      // samples composited before termination
    kTLoss = 5,      // float bits: sum of per-ray loss / n_rays
    kTCompactRes = 6,  // compacted samples reserved
    kTCompactN = 7,    // compacted samples kept (<= compact capacity)
    kTRound0 = 8,      // samples evaluated in each window (kRounds counters)
    kTQueue = 12,      // queries left for the deformation's second pass
    kTCounters = 13
};

// Evaluation windows over each ray's marched samples: samples [kWin[w],
// kWin[w + 1]) of the rays still alive are deformed and evaluated in round
// w, then each ray's transmittance advances over them (the loss kernel's
// arithmetic); a ray whose transmittance fell below 1e-4, or whose samples
// ran out, takes no further round.  The loss reads exactly the samples the
// rounds evaluated, so the step computes what one pass over every marched
// sample would.  Once trained, most rays stop within a sample or two of the
// surface, so the first window holds one sample (a first window of 4 or 8
// measured 10-90 % slower rounds).
constexpr uint32_t kRounds = 4;
constexpr uint32_t kWin[kRounds + 1] = {0u, 1u, 4u, 16u, 0xffffffffu};

constexpr int kW = 64;
constexpr int kDOut = 16;
constexpr int kCin = 32;             // density outputs + 16 SH
constexpr uint32_t kMlpThreads = 256;  // backward: one weight copy in LDS per block
// Samples per weight-gradient partial: a batch in 64 chunks of whole LDS
// slices (32 samples), between 128 and 1,024 samples each.  A chunk's slices
// follow one another, so a small batch in chunks of 1,024 sat on a few CUs
// (1,000 samples: 48 us, in chunks of 128 9 us).
constexpr uint32_t kChunk = 1024, kChunkMin = 128, kChunksFew = 64;
__host__ __device__ inline uint32_t wgrad_chunk(uint32_t n) {
    const uint32_t c = (n + 32u * kChunksFew - 1u) / (32u * kChunksFew) * 32u;
    return c < kChunkMin ? kChunkMin : (c > kChunk ? kChunk : c);
}
// chunks of any batch of up to cap samples, at most
inline uint32_t wgrad_chunks(uint32_t cap) {
    return std::max((cap + kChunk - 1) / kChunk, std::min(kChunksFew, (cap + kChunkMin - 1) / kChunkMin));
}
constexpr uint32_t kRaySeedStride = 8;
// One wave per workgroup of the per-ray kernels: a step has thousands of rays
// where the chip has 1,024 SIMDs, and each lane walks its ray's samples one
// after another, so a wave wants a CU (its L1, its memory port) to itself.
// 8,192 rays, waves of four a workgroup / one: loss 180 / 108 us, the four
// rounds' kernels 135 / 48 us, rays 124 / 111 us.
constexpr uint32_t kRayThreads = 64;
constexpr uint32_t kRayWaves = kRayThreads / 64;
// backward: wave-level run sums on levels where one marching step covers at
// most this fraction of a cell (runs of about two or more samples per entry)
constexpr float kRunMaxStepCells = 0.5f;

// activation rows (feature-major, row stride = sample capacity)
template <int E>
struct Act {
    static constexpr int ENC = 0, H1 = E, DENS = E + kW, SH = E + kW + kDOut, H2 = E + kW + kCin,
                         H3 = H2 + kW, N = H3 + kW;
};
// delta rows
struct Dact {
    static constexpr int DRGB = 0, DH3 = 4, DH2 = DH3 + kW, DDENS = DH2 + kW, DH1 = DDENS + kDOut, N = DH1 + kW;
};
// parameter offsets (density MLP, colour MLP), row-major [out][in]
template <int E>
struct Off {
    static constexpr uint32_t W0 = 0, W1 = W0 + kW * E, W2 = W1 + kDOut * kW, W3 = W2 + kW * kCin, W4 = W3 + kW * kW,
                              N = W4 + 3 * kW;
};

// XCDs of the device: workgroups of one XCD share its L2
constexpr uint32_t kXcds = 8;

struct TrainState {
    uint32_t n_images = 0, width = 0, height = 0;
    bool far = false;              // an image's camera is far_camera
    float4* images = nullptr;
    TrainImage* meta = nullptr;
    // supervision of the training set (nullptr: none): mask id and
    // camera-axis depth per pixel, [n][h][w]
    uint8_t* seg = nullptr;
    float* depth = nullptr;
    std::vector<int32_t> frames;
    // workspace
    uint32_t ray_cap = 0, sample_cap = 0, compact_cap = 0;
    float4* ray_d = nullptr;
    float4* ray_o = nullptr;       // origin, w = length of the unnormalised direction
    int32_t* ray_frame = nullptr;
    uint32_t *ray_img = nullptr, *ray_pix = nullptr, *ray_src = nullptr, *ray_base = nullptr, *ray_cnt = nullptr;
    float4 *s_cpos = nullptr, *s_cdir = nullptr, *s_out = nullptr, *s_dout = nullptr;
    // evaluation rounds: per ray transmittance, alive flag and the first slot
    // of its samples in the round buffers (r_*: one window's samples, packed)
    float* ray_T = nullptr;
    uint32_t *ray_alive = nullptr, *ray_gbase = nullptr;
    float4 *r_pos = nullptr, *r_cpos = nullptr, *r_cdir = nullptr, *r_out = nullptr;
    int32_t* s_hit = nullptr;
    uint32_t* c_idx = nullptr;     // compacted batch: sample index
    float4* c_dout = nullptr;      // compacted batch: dL/d(rgb logits, density logit)
    float *act = nullptr, *dact = nullptr, *part = nullptr;
    float* t_buf = nullptr;        // march t values, step-major [max_steps][rays of the step]: the rounds and the loss read them
    // optimizer
    float *grad = nullptr, *adam_m = nullptr, *adam_v = nullptr;
    // hash-table gradients added to by global atomics (a table above
    // kPartMaxEntries only): FP64, or under FP16 accumulation kHalfCopies
    // partial tables; summed into grad afterwards
    double2* grad_d = nullptr;
    __half2* grad_h = nullptr;      // (the same memory)
    // partitioned scatter: its levels (0: none, or tables too large for it), the
    // records of one pass and their directory
    uint32_t part_levels = 0;
    void* recs = nullptr;
    uint32_t* rec_dir = nullptr;
    float* denc = nullptr;         // dL/dencoding of the batch [32][batch cap], for the scatters
    // LDS-scattered levels (a prefix of the levels, entries [0, lds_end)):
    // one partial table per chunk of the batch, [kScatterMaxChunks][2 lds_end]
    float* grad_p = nullptr;
    uint32_t lds_levels = 0, lds_end = 0;
    uint32_t* counters = nullptr;
    uint32_t* h_counters = nullptr;
    uint64_t rays_total = 0;
    uint32_t rays_per_batch = 1u << 12;
    // two counters, as the reference keeps them: the training step
    // (Testbed::m_training_step, which times the density-grid updates and
    // resumes at the saved value + 1 on snapshot load, testbed.cu:3011) and
    // Adam's own step (bias correction; restarts with fresh moments)
    uint32_t training_step = 0;
    uint32_t adam_step = 0;
    // Ema optimizer: running average of the weights and its debiased copy
    float *ema = nullptr, *ema_infer = nullptr;
    uint32_t ema_step = 0;
    bool have_grad = false;
    // network plugin: per-sample extra dims of the last forward ([cap][X]) and
    // its batch size (0: no stored forward; a training step overwrites it)
    float* net_extra = nullptr;
    uint32_t net_extra_cap = 0;
    uint32_t net_n = 0;
};

namespace {

__global__ void train_clear_kernel(uint32_t* counters, uint32_t limit) {
    const uint32_t i = threadIdx.x;
    if (i < kTCounters) counters[i] = i == kTLimit ? limit : 0u;
}

__global__ void fill_zero_kernel(uint32_t* p, uint64_t n) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = 0u;
}

__global__ void train_count_kernel(uint32_t* counters) {
    if (threadIdx.x == 0) counters[kTValid] = min(counters[kTSamples], counters[kTLimit]);
}

__global__ void train_compact_count_kernel(uint32_t* counters, uint32_t cap) {
    if (threadIdx.x == 0) counters[kTCompactN] = min(counters[kTCompactRes], cap);
}

struct RayArgs {
    RenderArgs box;               // render box, G, dt, max_steps (grid set per ray)
    const TrainImage* meta;
    const uint8_t* grids_lin;     // [slot][G^3/8]
    size_t grid_bytes;
    uint32_t n_images, width, height, max_samples;
    int32_t fixed_slot;           // >= -1: every ray marches this slot's grid
};

INSTA_DEV bool train_ray(const RayArgs& a, uint32_t i, uint32_t n_rays, uint64_t rays_total, Pcg32 rng,
                         uint32_t& img, uint32_t& pix, V3& o, V3& d, float& dn, float& t0, RenderArgs& ra) {
    img = (uint32_t)((((uint64_t)i + rays_total) * a.n_images / n_rays) % a.n_images);
    rng.advance((uint64_t)i * kRaySeedStride);
    const float x = rng.next_float();
    const float y = rng.next_float();
    (void)rng.next_float();  // motion-blur time in the reference
    const float jitter = rng.next_float();
    const uint32_t px = min((uint32_t)(x * (float)a.width), a.width - 1u);
    const uint32_t py = min((uint32_t)(y * (float)a.height), a.height - 1u);
    pix = px + py * a.width;
    const TrainImage& c = a.meta[img];
    const V3 d0 = v3((x - c.cx) * (float)a.width / c.fx, (y - c.cy) * (float)a.height / c.fy, 1.0f);
    d = v3(c.M[0] * d0.x + c.M[1] * d0.y + c.M[2] * d0.z, c.M[4] * d0.x + c.M[5] * d0.y + c.M[6] * d0.z,
           c.M[8] * d0.x + c.M[9] * d0.y + c.M[10] * d0.z);
    dn = norm(d);
    d = v3(d.x / dn, d.y / dn, d.z / dn);
    o = v3(c.M[3], c.M[7], c.M[11]);
    ra = a.box;
    ra.grid = a.grids_lin + (size_t)((a.fixed_slot >= -1 ? a.fixed_slot : c.frame) + 1) * a.grid_bytes;
    const float tb = box_ray_tmin(ra, o, d);
    if (tb == 3.40282347e38f) return false;
    t0 = fmaxf(tb, 0.0f) + a.box.dt * jitter;
    return true;
}

template <bool kFar>
__global__ __launch_bounds__(kRayThreads) void train_rays_kernel(RayArgs a, uint32_t n_rays, uint64_t rays_total,
                                                         Pcg32 rng, float4* __restrict__ ray_d,
                                                         float4* __restrict__ ray_o,
                                                         int32_t* __restrict__ ray_frame,
                                                         uint32_t* __restrict__ ray_img,
                                                         uint32_t* __restrict__ ray_pix,
                                                         uint32_t* __restrict__ ray_src,
                                                         uint32_t* __restrict__ ray_base,
                                                         uint32_t* __restrict__ ray_cnt,
                                                         float* __restrict__ t_buf,
                                                         float* __restrict__ ray_T,
                                                         uint32_t* __restrict__ ray_alive,
                                                         uint32_t* __restrict__ counters) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t img = 0, pix = 0, count = 0;
    V3 o = v3(0, 0, 0), d = v3(0, 0, 1), idir = v3(0, 0, 1);
    float t0 = 0.0f, dn = 1.0f;
    RenderArgs ra = a.box;
    if (i < n_rays && train_ray(a, i, n_rays, rays_total, rng, img, pix, o, d, dn, t0, ra)) {
        idir = v3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
        // sample t values to step-major scratch (t_buf[j * n_rays + i])
        bool exited;
        count = walk_samples<kFar>(ra, o, d, idir, t0, a.box.max_steps, exited,
                                   [&](uint32_t j, float tj) { t_buf[(size_t)j * n_rays + i] = tj; });
    }
    const uint32_t base = block_reserve<kRayWaves>(&counters[kTSamples], count);
    const bool fits = base + count <= a.max_samples;
    if (count > 0 && !fits && base < a.max_samples) atomicMin(&counters[kTLimit], base);
    const bool keep = count > 0 && fits;
    const uint32_t r = block_append<kRayWaves>(&counters[kTRays], keep);
    if (!keep) return;
    ray_d[r] = make_float4(d.x, d.y, d.z, 0.0f);
    ray_o[r] = make_float4(o.x, o.y, o.z, dn);
    ray_frame[r] = a.meta[img].frame;
    ray_img[r] = img;
    ray_pix[r] = pix;
    ray_src[r] = i;
    ray_base[r] = base;
    ray_cnt[r] = count;
    ray_T[r] = 1.0f;
    ray_alive[r] = 1u;
}

template <int NIN, int NOUT>
INSTA_DEV void store_rows(float* __restrict__ act, uint32_t ld, int row0, uint32_t i, const float* v) {
#pragma unroll
    for (int k = 0; k < NOUT; ++k) act[(size_t)(row0 + k) * ld + i] = v[k];
}

// Forward with stored activations over the compacted batch, on
// v_mfma_f32_16x16x4f32 (the layout of the FP32 inference kernel): phase A,
// one thread per sample, encodes (FP32, the scalar encode's arithmetic) into
// LDS and stores the encoding, extra-dims and SH rows; phase B runs each
// wave's 64 samples, 16 columns at a time, through the density MLP and the
// colour MLP's hidden layers with the weights as A operands, storing every
// layer's rows from the accumulators (lane l holds rows 4(l/16)..+3 of
// column l%16, contiguous along the batch).  The training step needs no
// output layer (dL/doutput comes from the loss kernel); the network plugin's
// forward asks for it through `out` (rgb logits and the density logit per
// batch entry).  Extra dims come from the frame table by the selector, or
// per sample from x_extra [n][X] when given.
typedef float tf_f4 __attribute__((ext_vector_type(4)));
constexpr uint32_t kFwdTile = 256;

// Column blocks of 16 samples a wave of the forward and backward kernels
// takes: four, or one where the batch is small, so that a workgroup has 64
// samples instead of 256, a quarter of the levels a wave to encode, and a
// quarter of the latency.
// 1,000 samples: backward 58 -> 16 us, forward 40 -> 13 us; at 100,000 (head)
// four columns: forward 145 us, one column 148 us, backward 84 / 82 us; above
// that one column costs the forward more (126 against 121 us at 8,192 rays).
constexpr uint32_t kSmallBatch = 65536;
INSTA_DEV uint32_t tile_columns(uint32_t n) { return n <= kSmallBatch ? 1u : 4u; }
// workgroups that cover any batch of up to cap samples
uint32_t mlp_blocks(uint32_t cap) {
    return std::max((cap + kFwdTile - 1) / kFwdTile, (std::min(cap, kSmallBatch) + kFwdTile / 4 - 1) / (kFwdTile / 4));
}

template <int L, int X>
__global__ __launch_bounds__(256) void train_forward_kernel(const float* __restrict__ params,
                                                          const float* __restrict__ table, GridParams gp,
                                                          const float* __restrict__ frame_extra, uint32_t n_frames,
                                                          const uint32_t* __restrict__ n_dev,
                                                          const uint32_t* __restrict__ c_idx,
                                                          const float4* __restrict__ cpos,
                                                          const float4* __restrict__ cdir,
                                                          const float* __restrict__ x_extra,
                                                          float* __restrict__ act, uint32_t ld,
                                                          float4* __restrict__ out) {
    constexpr int E = 2 * L, DIN = E + X, KB0 = DIN / 4, S = DIN + 1;
    static_assert(DIN % 4 == 0, "K blocks of 4");
    using A = Act<DIN>;
    using O = Off<DIN>;
    __shared__ float s_x[kFwdTile * S];
    const uint32_t n = *n_dev;
    const uint32_t cols = tile_columns(n), samples = 64u * cols;
    const uint32_t base = blockIdx.x * samples;
    if (base >= n) return;  // whole block past the batch
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t m = lane & 15u, g = lane >> 4;
    {
        const uint32_t i = base + tid % samples;
        const int part = __builtin_amdgcn_readfirstlane((int)(tid / samples)), per = (int)(L / 4u * cols);
        float* row = s_x + tid % samples * S;
        if (i < n) {
            const uint32_t smp = c_idx[i];
            const float4 p4 = cpos[smp], d4 = cdir[smp];
            const V3 x = v3(p4.x, p4.y, p4.z);
            // two levels' gathers in flight; rolled, so that a level's
            // corners do not all live at once (one wave per SIMD)
#pragma unroll 2
            for (int l = part * per; l < (part + 1) * per; ++l) {
                float f[2];
                encode_level<2>(table, gp, (uint32_t)l, x, f);
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    row[2 * l + k] = f[k];
                    act[(size_t)(A::ENC + 2 * l + k) * ld + i] = f[k];
                }
            }
            if (part == 0) {
                if constexpr (X > 0) {
                    const uint32_t sel = __float_as_uint(d4.w);
                    const float* fx = x_extra ? x_extra + (size_t)smp * X
                                              : (sel != kExtraOnes && sel <= n_frames ? frame_extra + (size_t)(sel - 1u) * X
                                                                                      : nullptr);
#pragma unroll
                    for (int e = 0; e < X; ++e) {
                        const float v = fx ? fx[e] : 1.0f;
                        row[E + e] = v;
                        act[(size_t)(A::ENC + E + e) * ld + i] = v;
                    }
                }
                float sh[16];
                sh16(d4.x * 2.0f - 1.0f, d4.y * 2.0f - 1.0f, d4.z * 2.0f - 1.0f, sh);
                store_rows<16, 16>(act, ld, A::SH, i, sh);
            }
        } else if (part == 0) {
#pragma unroll
            for (int k = 0; k < DIN; ++k) row[k] = 0.0f;
        }
    }
    __syncthreads();
    const float* W0 = params + O::W0;
    const float* W1 = params + O::W1;
    const float* W2 = params + O::W2;
    const float* W3 = params + O::W3;
    for (uint32_t nb = 0; nb < cols; ++nb) {
        const uint32_t s = (wave * cols + nb) * 16 + m;  // column (sample) of this lane
        const uint32_t i = base + s;
        const bool live = i < n;
        const float* xr = s_x + s * S;
        // SH of the column's sample; lane group g feeds K rows 4g..4g+3
        float shg[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (live) {
            const float4 d4 = cdir[c_idx[i]];
            float sh[16];
            sh16(d4.x * 2.0f - 1.0f, d4.y * 2.0f - 1.0f, d4.z * 2.0f - 1.0f, sh);
#pragma unroll
            for (int b = 0; b < 4; ++b) shg[b] = g == 0 ? sh[b] : (g == 1 ? sh[4 + b] : (g == 2 ? sh[8 + b] : sh[12 + b]));
        }
        // density layer 0: H1 = relu(W0 x)
        tf_f4 h[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            tf_f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int kb = 0; kb < KB0; ++kb)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(W0[(16 * t + m) * DIN + 4 * kb + g], xr[4 * kb + g], acc, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                h[t][q] = fmaxf(acc[q], 0.0f);
                if (live) act[(size_t)(A::H1 + 16 * t + 4 * g + q) * ld + i] = h[t][q];
            }
        }
        // density output: 16 rows, K = H1 in the order 16t + 4g + b
        tf_f4 dn = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int b = 0; b < 4; ++b)
                dn = __builtin_amdgcn_mfma_f32_16x16x4f32(W1[m * kW + 16 * t + 4 * g + b], h[t][b], dn, 0, 0, 0);
        if (live)
#pragma unroll
            for (int q = 0; q < 4; ++q) act[(size_t)(A::DENS + 4 * g + q) * ld + i] = dn[q];
        // colour layer 0: K = density outputs (4g + b) then SH (16 + 4g + b)
        tf_f4 r[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            tf_f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int b = 0; b < 4; ++b)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(W2[(16 * t + m) * kCin + 4 * g + b], dn[b], acc, 0, 0, 0);
#pragma unroll
            for (int b = 0; b < 4; ++b)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(W2[(16 * t + m) * kCin + 16 + 4 * g + b], shg[b], acc, 0, 0,
                                                           0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                r[t][q] = fmaxf(acc[q], 0.0f);
                if (live) act[(size_t)(A::H2 + 16 * t + 4 * g + q) * ld + i] = r[t][q];
            }
        }
        // colour layer 1
        tf_f4 h3[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            tf_f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(W3[(16 * t + m) * kW + 16 * s2 + 4 * g + b], r[s2][b],
                                                               acc, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                h3[t][q] = fmaxf(acc[q], 0.0f);
                if (live) act[(size_t)(A::H3 + 16 * t + 4 * g + q) * ld + i] = h3[t][q];
            }
        }
        if (out) {
            // colour output (3 rows of W4, padded to 16): lane group 0 holds
            // rows 0..3 of its column; the density logit is density output 0
            const float* W4 = params + O::W4;
            tf_f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(m < 3 ? W4[m * kW + 16 * s2 + 4 * g + b] : 0.0f,
                                                               h3[s2][b], acc, 0, 0, 0);
            if (live && g == 0) out[i] = make_float4(acc[0], acc[1], acc[2], dn[0]);
        }
    }
}

struct LossArgs {
    const float4* images;
    const uint8_t* seg;   // mask ids (nullptr: no masks)
    const float* depth;   // camera-axis depth, 0 = none (nullptr: no depth images)
    uint32_t width, height;
    float dt, density_bias, loss_scale_per_ray, inv_rays;
    float seg_weight, depth_weight;
};

INSTA_DEV float sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }

// one sample's transmittance step, exactly as the loss kernel composites
INSTA_DEV float transmit(float T, float density_logit, float density_bias, float dt) {
    const float sigma = expf(density_logit + density_bias);
    const float alpha = 1.0f - expf(-sigma * dt);
    return T * (1.0f - alpha);
}

// f(j, load(j)) for j = 0..n-1 in order until it returns false.  A lane's walk
// over its ray is a chain of memory latencies if each sample is loaded when it
// is wanted: four are loaded while the four before them are worked on.
// 8,192 rays: loss 193 us without, 180 us (108 us with one wave a workgroup);
// gathers of the four rounds 64 -> 41 us (32 us).
template <class V, class Load, class F>
INSTA_DEV void walk_ray(uint32_t n, Load load, F f) {
    if (n == 0) return;
    V next[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) next[k] = load(min(k, n - 1u));
    for (uint32_t j = 0; j < n; j += 4) {
        V cur[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            cur[k] = next[k];
            next[k] = load(min(j + 4u + k, n - 1u));
        }
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            if (j + k < n && !f(j + k, cur[k])) return;
    }
}

// Round `w` gather: the window's samples of every alive ray, packed into the
// round buffers (each ray's samples contiguous from ray_gbase).
__global__ __launch_bounds__(kRayThreads) void train_gather_kernel(uint32_t lo, uint32_t hi,
                                                           const uint32_t* __restrict__ ray_base,
                                                           const uint32_t* __restrict__ ray_cnt,
                                                           const uint32_t* __restrict__ ray_alive,
                                                           uint32_t* __restrict__ ray_gbase,
                                                           const float4* __restrict__ ray_o,
                                                           const float4* __restrict__ ray_d,
                                                           const uint32_t* __restrict__ ray_src,
                                                           const float* __restrict__ t_buf, uint32_t t_stride,
                                                           float4* __restrict__ r_pos,
                                                           uint32_t* __restrict__ counters, uint32_t round_slot) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r == 0) counters[kTQueue] = 0u;  // this round's
    uint32_t n = 0;
    if (r < counters[kTRays] && ray_alive[r]) {
        const uint32_t cnt = ray_cnt[r];
        n = cnt > lo ? min(cnt, hi) - lo : 0u;
    }
    const uint32_t g = block_reserve<kRayWaves>(&counters[round_slot], n);
    if (n == 0) return;
    ray_gbase[r] = g;
    // posed positions from the march's t values (the march's own arithmetic)
    const float4 o4 = ray_o[r], d4 = ray_d[r];
    const V3 o = v3(o4.x, o4.y, o4.z), d = v3(d4.x, d4.y, d4.z);
    const float* __restrict__ tr = t_buf + ray_src[r];
    walk_ray<float>(
        n, [&](uint32_t k) { return tr[(size_t)(lo + k) * t_stride]; },
        [&](uint32_t k, float t) {
            const V3 pos = o + d * t;
            r_pos[g + k] = make_float4(pos.x, pos.y, pos.z, __uint_as_float(r));
            return true;
        });
}

// Round `w` scatter and transmittance: each alive ray's evaluated samples go
// back to their marched slots, and its transmittance advances over them; the
// ray stays alive only while it is >= 1e-4 with samples left past the window.
__global__ __launch_bounds__(kRayThreads) void train_round_kernel(uint32_t lo, uint32_t hi, float density_bias, float dt,
                                                          const uint32_t* __restrict__ ray_base,
                                                          const uint32_t* __restrict__ ray_cnt,
                                                          uint32_t* __restrict__ ray_alive,
                                                          const uint32_t* __restrict__ ray_gbase,
                                                          float* __restrict__ ray_T,
                                                          const float4* __restrict__ r_cpos,
                                                          const float4* __restrict__ r_cdir,
                                                          const float4* __restrict__ r_out,
                                                          float4* __restrict__ s_cpos, float4* __restrict__ s_cdir,
                                                          float4* __restrict__ s_out,
                                                          const uint32_t* __restrict__ counters) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= counters[kTRays] || !ray_alive[r]) return;
    const uint32_t cnt = ray_cnt[r];
    const uint32_t n = cnt > lo ? min(cnt, hi) - lo : 0u;
    const uint32_t base = ray_base[r] + lo, g = ray_gbase[r];
    float T = ray_T[r];
    bool alive = n > 0;
    struct Sample {
        float4 out, cpos, cdir;
    };
    walk_ray<Sample>(
        n, [&](uint32_t k) { return Sample{r_out[g + k], r_cpos[g + k], r_cdir[g + k]}; },
        [&](uint32_t k, const Sample& q) {
            s_cpos[base + k] = q.cpos;
            s_cdir[base + k] = q.cdir;
            s_out[base + k] = q.out;
            if (alive) {
                T = transmit(T, q.out.w, density_bias, dt);
                if (T < 1e-4f) alive = false;
            }
            return true;
        });
    ray_T[r] = T;
    ray_alive[r] = alive && cnt > hi ? 1u : 0u;
}
// sRGB transfer functions with the reference's constants (common_device.cuh:31-61)
INSTA_DEV float srgb_to_linear(float c) { return c <= 0.04045f ? c / 12.92f : powf((c + 0.055f) / 1.055f, 2.4f); }
INSTA_DEV float linear_to_srgb(float c) { return c < 0.0031308f ? 12.92f * c : 1.055f * powf(c, 0.41666f) - 0.055f; }

__global__ __launch_bounds__(kRayThreads) void train_loss_kernel(LossArgs a, Pcg32 rng0,
                                                         const uint32_t* __restrict__ ray_src,
                                                         const uint32_t* __restrict__ ray_img,
                                                         const uint32_t* __restrict__ ray_pix,
                                                         const uint32_t* __restrict__ ray_base,
                                                         const uint32_t* __restrict__ ray_cnt,
                                                         const float4* __restrict__ ray_o,
                                                         const float4* __restrict__ ray_d,
                                                         const float* __restrict__ t_buf, uint32_t t_stride,
                                                         const float4* __restrict__ s_out,
                                                         uint32_t* __restrict__ c_idx, float4* __restrict__ c_dout,
                                                         uint32_t compact_cap, uint32_t* __restrict__ counters) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = r < counters[kTRays];
    float ray_loss = 0.0f;
    uint32_t used = 0, base = 0;
    float acc[3] = {0.0f, 0.0f, 0.0f}, grad[3] = {0.0f, 0.0f, 0.0f};
    // depth supervision: the composited depth and dL/dD (0: none for this ray)
    float depth_ray = 0.0f, dgrad = 0.0f;
    V3 org = v3(0.0f, 0.0f, 0.0f), dir = v3(0.0f, 0.0f, 1.0f);
    const float* __restrict__ tr = t_buf;  // this ray's march t values, stride t_stride
    struct RaySample {
        float4 out;
        float t;
    };
    const auto load_sample = [&](uint32_t j, bool with_t) {
        return RaySample{s_out[base + j], with_t ? tr[(size_t)j * t_stride] : 0.0f};
    };
    if (valid) {
        base = ray_base[r];
        tr = t_buf + ray_src[r];
        const uint32_t cnt = ray_cnt[r];
        Pcg32 rng = rng0;
        rng.advance((uint64_t)ray_src[r] * kRaySeedStride);
        (void)rng.next_float();
        (void)rng.next_float();
        // linear colour space with sRGB training (testbed_nerf.cu:1419-1443):
        // the random background goes to linear, is blended behind the
        // premultiplied linear texel (read_rgba of an 8-bit sRGB image,
        // common_device.cuh:658-671), then target and background return to sRGB
        const size_t texel = (size_t)ray_img[r] * a.width * a.height + ray_pix[r];
        const float4 tex = a.images[texel];
        const float texc[3] = {tex.x, tex.y, tex.z};
        float bg[3], target[3];
        for (int c = 0; c < 3; ++c) {
            const float bg_lin = srgb_to_linear(rng.next_float());
            bg[c] = linear_to_srgb(bg_lin);
            target[c] = linear_to_srgb(srgb_to_linear(texc[c]) * tex.w + (1.0f - tex.w) * bg_lin);
        }
        // segmentation and depth supervision (testbed_nerf.cu:1476-1497): mask
        // ids 120/130/140 weight the colour gradient; ids <= 90 or > 250 and
        // near-transparent texels get no depth term; the target is the depth
        // texel times the unnormalised direction's length (0 texel: none)
        float seg_w = 1.0f, lam = a.depth_weight;
        if (a.seg) {
            const uint32_t id = a.seg[texel];
            if (id == 120u || id == 130u || id == 140u) seg_w = a.seg_weight;
            if (id <= 90u || id > 250u) lam = 0.0f;
            if (tex.w < 0.001f) lam = 0.0f;
        }
        const float4 ro = ray_o[r], rd = ray_d[r];
        org = v3(ro.x, ro.y, ro.z);
        dir = v3(rd.x, rd.y, rd.z);
        const float target_depth = ro.w * ((lam > 0.0f && a.depth) ? a.depth[texel] : -1.0f);
        const bool supervise_depth = target_depth > 0.0f;
        float T = 1.0f;
        walk_ray<RaySample>(
            cnt, [&](uint32_t j) { return load_sample(j, supervise_depth); },
            [&](uint32_t, const RaySample& q) {
                if (T < 1e-4f) return false;
                const float sigma = expf(q.out.w + a.density_bias);
                const float alpha = 1.0f - expf(-sigma * a.dt);
                const float w = alpha * T;
                acc[0] = acc[0] + w * sigmoid(q.out.x);
                acc[1] = acc[1] + w * sigmoid(q.out.y);
                acc[2] = acc[2] + w * sigmoid(q.out.z);
                if (supervise_depth) {
                    const V3 p = org + dir * q.t;
                    depth_ray = depth_ray + w * norm(p - org);
                }
                T = T * (1.0f - alpha);  // = transmit(T, o.w, ...), which the rounds use
                ++used;
                return true;
            });
        // L1 depth loss (depth_loss_type's default, testbed_nerf.cu:133-139)
        if (supervise_depth) dgrad = copysignf(1.0f, depth_ray - target_depth) * lam;
        if (used == cnt) {
            for (int c = 0; c < 3; ++c) acc[c] = acc[c] + T * bg[c];
        }
        // Huber(0.1) / 5 per channel (testbed_nerf.cu:141-157, 1299)
        for (int c = 0; c < 3; ++c) {
            const float diff = acc[c] - target[c];
            const float ad = fabsf(diff);
            const float l = ad > 0.1f ? ad - 0.05f : (0.5f / 0.1f) * diff * diff;
            grad[c] = (ad > 0.1f ? (diff > 0.0f ? 1.0f : -1.0f) : diff / 0.1f) / 5.0f * seg_w;
            ray_loss += l / 5.0f;
        }
        ray_loss = ray_loss / 3.0f * a.inv_rays;
    }
    // compaction of the composited samples into the training batch
    const uint32_t cb = block_reserve<kRayWaves>(&counters[kTCompactRes], used);
    const uint32_t n_c = cb < compact_cap ? min(used, compact_cap - cb) : 0u;
    if (valid) {
        const float ls = a.loss_scale_per_ray;
        float T = 1.0f;
        float acc2[3] = {0.0f, 0.0f, 0.0f}, depth2 = 0.0f;
        const auto backprop = [&](uint32_t j, const RaySample& q) {
            const float4 o = q.out;
            const float sg[3] = {sigmoid(o.x), sigmoid(o.y), sigmoid(o.z)};
            const float sigma = expf(o.w + a.density_bias);
            const float alpha = 1.0f - expf(-sigma * a.dt);
            const float w = alpha * T;
            for (int c = 0; c < 3; ++c) acc2[c] = acc2[c] + w * sg[c];
            T = T * (1.0f - alpha);
            float dsig = 0.0f;
            float drgb[3];
            for (int c = 0; c < 3; ++c) {
                drgb[c] = ls * (w * grad[c] * (sg[c] * (1.0f - sg[c])));
                dsig = dsig + grad[c] * (T * sg[c] - (acc[c] - acc2[c]));
            }
            if (dgrad != 0.0f) {
                // dD/dsigma_j / dt = T_{j+1} depth_j - (depth suffix after j)
                const V3 p = org + dir * q.t;
                const float dj = norm(p - org);
                depth2 = depth2 + w * dj;
                dsig = dsig + dgrad * (T * dj - (depth_ray - depth2));
            }
            c_idx[cb + j] = base + j;
            c_dout[cb + j] = make_float4(drgb[0], drgb[1], drgb[2], ls * (sigma * (a.dt * dsig)));
            return true;
        };
        walk_ray<RaySample>(n_c, [&](uint32_t j) { return load_sample(j, dgrad != 0.0f); }, backprop);
    }
    // statistics, one atomic each per workgroup
    __shared__ uint32_t s_used;
    __shared__ float s_loss;
    if (threadIdx.x == 0) {
        s_used = 0u;
        s_loss = 0.0f;
    }
    __syncthreads();
    uint32_t u = used;
    float lsum = ray_loss;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        u += __shfl_xor(u, off);
        lsum += __shfl_xor(lsum, off);
    }
    if ((threadIdx.x & 63u) == 0) {
        atomicAdd(&s_used, u);
        atomicAdd(&s_loss, lsum);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (s_used) atomicAdd(&counters[kTUsed], s_used);
        if (s_loss != 0.0f) atomicAdd(reinterpret_cast<float*>(&counters[kTLoss]), s_loss);
    }
}

// Gradients of the LDS-scattered entries into grad_tab: the sum of the
// scatter's chunk partials ([chunk][feature][lds_end]) in chunk order.
__global__ void grad_partials_reduce_kernel(const float* __restrict__ grad_p, uint32_t lds_end, uint32_t chunks,
                                            float* __restrict__ grad_tab) {
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= lds_end) return;
    float a = 0.0f, b = 0.0f;
    for (uint32_t c = 0; c < chunks; ++c) {
        a = a + grad_p[(size_t)(2u * c) * lds_end + e];
        b = b + grad_p[(size_t)(2u * c + 1u) * lds_end + e];
    }
    *reinterpret_cast<float2*>(grad_tab + 2 * (size_t)e) = make_float2(a, b);
}

// Sum of v over the run of equal keys that starts at this lane, in the run's
// first lane (other lanes' sums are partial).  Runs are maximal stretches of
// consecutive lanes with one key; every lane of the wave is active.
INSTA_DEV float2 run_sum(uint32_t key, float2 v, bool& head) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t prev = __shfl_up(key, 1u);
    head = lane == 0u || prev != key;
    const uint64_t heads = __ballot(head);
    if (heads == ~0ull) return v;  // no two neighbours share a key
    const uint64_t later = lane == 63u ? 0ull : heads & (~0ull << (lane + 1u));
    const uint32_t end = later ? (uint32_t)__builtin_ctzll(later) - 1u : 63u;
#pragma unroll
    for (uint32_t off = 1; off < 64u; off <<= 1) {
        const float ox = __shfl_down(v.x, off), oy = __shfl_down(v.y, off);
        if (lane + off <= end) {
            v.x = v.x + ox;
            v.y = v.y + oy;
        }
    }
    return v;
}

// Hash-grid scatter of the leading levels whose tables fit in LDS (at most
// kLdsEntries entries each): a workgroup adds its chunk's corner gradients
// into an LDS copy of the level's table, then stores the whole table as its
// chunk's partial (plain coalesced stores, no global atomics);
// grad_partials_reduce_kernel sums the partials in chunk order.
// FP32 gradients (scatter_lds64_kernel): one workgroup per (chunk, level,
// feature) with FP64 LDS atomics.  An FP32 LDS atomic retires 200 G lanes/s
// over the chip, an FP64 one 1,760 G (random entries or 64 hot ones alike), so
// the table holds doubles, one feature of them; recomputing the corners for
// the other feature costs less than the adds did, and neither conflicts nor
// runs of equal entries need care.  The sums are exact but for one rounding.
// 237,000 samples on the eight levels of the small shapes: 77 us, with FP32 atomics and run sums 167; 100,003
// random samples, two levels: 30 us against 194.
// H16 (scatter_lds_kernel): one workgroup per (chunk, level), packed FP16
// atomics, one per corner; on levels in run_mask a wave first sums runs of
// consecutive samples with one corner.
constexpr uint32_t kLdsEntries = 16384;
constexpr uint32_t kScatterThreads = 1024;
constexpr uint32_t kScatterChunk = 8192;    // samples per workgroup
constexpr uint32_t kScatterMaxChunks = 64;  // partial tables

// The leading levels whose tables fit in LDS, as a mask, and the first entry
// after them.
uint32_t lds_scatter_levels(const GridParams& gp, int n_levels, uint32_t* end) {
    uint32_t mask = 0, e = 0;
    for (int l = 0; l < n_levels && gp.size[l] <= kLdsEntries; ++l) {
        mask |= 1u << l;
        e = gp.offset[l] + gp.size[l];
    }
    *end = e;
    return mask;
}

// partial tables: [chunk][feature][lds_end]
__global__ __launch_bounds__(kScatterThreads) void scatter_lds64_kernel(GridParams gp,
                                                                        const uint32_t* __restrict__ n_dev,
                                                                        const uint32_t* __restrict__ c_idx,
                                                                        const float4* __restrict__ cpos,
                                                                        const float* __restrict__ denc_g, uint32_t ld,
                                                                        float* __restrict__ grad_p, uint32_t lds_end) {
    __shared__ double tab[kLdsEntries];  // 128 KB: one workgroup per CU
    const uint32_t l = blockIdx.y, f = blockIdx.z;
    const uint32_t n = *n_dev;
    const uint32_t chunk = (n + gridDim.x - 1) / gridDim.x;
    // an empty chunk still stores its (zero) partial
    const uint32_t s0 = min(n, blockIdx.x * chunk), s1 = min(n, s0 + chunk);
    const uint32_t size = gp.size[l];
    for (uint32_t j = threadIdx.x; j < size; j += kScatterThreads) tab[j] = 0.0;
    __syncthreads();
    const float* __restrict__ de = denc_g + (size_t)(2u * l + f) * ld;
    // the next sample is loaded before this one's corners are added
    uint32_t i = s0 + threadIdx.x;
    float4 pn = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float en = 0.0f;
    if (i < s1) {
        pn = cpos[c_idx[i]];
        en = de[i];
    }
    while (i < s1) {
        const V3 x = xyz(pn);
        const float e = en;
        i += kScatterThreads;
        if (i < s1) {
            pn = cpos[c_idx[i]];
            en = de[i];
        }
        uint32_t corner[8];
        float weight[8];
        cell_corners(gp, l, x, corner, weight);
#pragma unroll
        for (uint32_t c = 0; c < 8; ++c) {
            const float w = weight[c];
            unsafeAtomicAdd(&tab[corner[c]], (double)(w * e));
        }
    }
    __syncthreads();
    float* __restrict__ dst = grad_p + ((size_t)blockIdx.x * 2u + f) * lds_end + gp.offset[l];
    for (uint32_t j = threadIdx.x; j < size; j += kScatterThreads) dst[j] = (float)tab[j];
}

__global__ __launch_bounds__(kScatterThreads) void scatter_lds_kernel(GridParams gp, const uint32_t* __restrict__ n_dev,
                                                                      const uint32_t* __restrict__ c_idx,
                                                                      const float4* __restrict__ cpos,
                                                                      const float* __restrict__ denc_g, uint32_t ld,
                                                                      uint32_t run_mask, float* __restrict__ grad_p,
                                                                      uint32_t lds_end) {
    __shared__ __half2 tab[kLdsEntries];  // 64 KB: two workgroups per CU
    const uint32_t l = blockIdx.y;  // grid.y: the LDS-scattered levels
    const uint32_t n = *n_dev;
    const uint32_t chunk = (n + gridDim.x - 1) / gridDim.x;
    // an empty chunk still stores its (zero) partial
    const uint32_t s0 = min(n, blockIdx.x * chunk), s1 = min(n, s0 + chunk);
    const uint32_t size = gp.size[l], off = gp.offset[l];
    for (uint32_t j = threadIdx.x; j < size; j += kScatterThreads) tab[j] = __floats2half2_rn(0.0f, 0.0f);
    __syncthreads();
    const bool runs = (run_mask >> l) & 1u;
    // every thread runs every round (run_sum needs whole waves); the next
    // round's sample is loaded before this round's corners are added
    const uint32_t rounds = (s1 - s0 + kScatterThreads - 1) / kScatterThreads;
    auto load = [&](uint32_t q, float4& p4, float& e0, float& e1) {
        const uint32_t i = s0 + q * kScatterThreads + threadIdx.x;
        if (i < s1) {
            p4 = cpos[c_idx[i]];
            e0 = denc_g[(size_t)(2 * l) * ld + i];
            e1 = denc_g[(size_t)(2 * l + 1) * ld + i];
        } else {
            p4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            e0 = e1 = 0.0f;
        }
    };
    float4 pn;
    float en0 = 0.0f, en1 = 0.0f;
    if (rounds) load(0, pn, en0, en1);
    for (uint32_t q = 0; q < rounds; ++q) {
        const bool valid = s0 + q * kScatterThreads + threadIdx.x < s1;
        const V3 x = xyz(pn);
        const float e0 = en0, e1 = en1;
        if (q + 1 < rounds) load(q + 1, pn, en0, en1);
        uint32_t corner[8];
        float weight[8];
        cell_corners(gp, l, x, corner, weight);
#pragma unroll
        for (uint32_t c = 0; c < 8; ++c) {
            const float w = weight[c];
            const uint32_t idx = corner[c];
            float2 v = make_float2(w * e0, w * e1);
            bool lead = valid;
            if (runs) {
                bool head;
                v = run_sum(valid ? idx : ~0u, v, head);
                lead = valid && head;
            }
            if (lead) unsafeAtomicAdd(&tab[idx], __floats2half2_rn(v.x, v.y));
        }
    }
    __syncthreads();
    float* __restrict__ dst = grad_p + (size_t)blockIdx.x * 2u * lds_end + off;
    for (uint32_t j = threadIdx.x; j < size; j += kScatterThreads) {
        const float2 v = __half22float2(tab[j]);
        dst[j] = v.x;
        dst[lds_end + j] = v.y;
    }
}

// Hash-grid scatter of the levels whose tables exceed LDS, one level's
// samples after the other on one XCD.  Workgroups are dispatched round-robin
// over the eight XCDs (block b on XCD b % 8), each with a 4 MB L2, so block b
// takes the levels b % 8, b % 8 + 8, ... of the list, a level's samples before
// the next level's: a table of 2^19 entries (4 MB) is added to from one L2
// while it is resident, instead of every table's lines moving between eight
// L2s and HBM.  On the levels of run_mask the corner gradients of consecutive
// samples that land on one entry (coarse levels along one ray) are summed
// across the wave first and added by one lane.
// FP32: FP64 atomics, so that the sums are exact but for one rounding however
// many samples share an entry; neighbouring lanes first pair up, so that an
// entry's two adds are neighbours in one memory request.
// H16: one packed FP16 atomic per corner, into one of kHalfCopies partial
// tables (by block of kLevelThreads samples; a level's first copy before its
// second), which keep the rounding of many small adds in check and are summed
// in a fixed order afterwards.
// Bound by the L2's atomics, about one request per clock and XCD: a plugin pass
// of 100,000 samples near the skin at T = 2^20 takes 1,305 us; with one FP32
// copy of the tables per XCD 2,220, with FP32 atomics straight into the
// gradients 1,118, but sums of 8,192 crowded samples were off by 1.2e-6 of
// themselves (now below 2^-22).
constexpr uint32_t kLevelThreads = 256;
constexpr uint32_t kHalfCopies = 8;
// Where no table exceeds kPartMaxEntries (the partition's directory) the levels
// are partitioned instead, kPartPass samples at a time (352 MB of records at
// full size), batches of any size: a plugin pass at full size takes 157 / 172 /
// 191 us for 300 / 4,000 / 8,192 samples; with FP32 atomics for these batches
// 152 / 183 / 232 us, and sums off by up to 9e-7 of themselves.
constexpr uint32_t kPartMaxEntries = 1u << 19;
constexpr uint32_t kPartPass = 1u << 18;
constexpr uint32_t kPartSlices = 64;  // one wave scans a chunk's slice counts
template <bool H16>
__global__ __launch_bounds__(kLevelThreads) void scatter_levels_kernel(GridParams gp, uint32_t level_mask,
                                                                       uint32_t run_mask, uint32_t blocks,
                                                                       const uint32_t* __restrict__ n_dev,
                                                                       const uint32_t* __restrict__ c_idx,
                                                                       const float4* __restrict__ cpos,
                                                                       const float* __restrict__ denc_g, uint32_t ld,
                                                                       double* __restrict__ grad_d,
                                                                       __half2* __restrict__ grad_h,
                                                                       uint64_t entries) {
    // blocks: sample blocks per level, a multiple of kHalfCopies
    const uint32_t k = blockIdx.x / kXcds, li = (k / blocks) * kXcds + blockIdx.x % kXcds;
    uint32_t b = k % blocks, copy = 0;
    if constexpr (H16) {
        const uint32_t per_copy = blocks / kHalfCopies;
        copy = b / per_copy;
        b = (b % per_copy) * kHalfCopies + copy;
    }
    const uint32_t n = *n_dev, s0 = b * kLevelThreads;
    if (li >= (uint32_t)__popc(level_mask) || (s0 + (threadIdx.x & ~63u)) >= n) return;  // whole waves
    uint32_t rest = level_mask;
    for (uint32_t j = 0; j < li; ++j) rest &= rest - 1u;  // drop the li lowest levels of the list
    const uint32_t l = (uint32_t)__builtin_ctz(rest);
    const uint32_t off = gp.offset[l];
    const bool runs = (run_mask >> l) & 1u;
    const bool valid = s0 + threadIdx.x < n, odd = threadIdx.x & 1u;
    const uint32_t i = valid ? s0 + threadIdx.x : n - 1u;  // tail lanes repeat the last sample and add nothing
    const float4 p4 = cpos[c_idx[i]];
    const float e0 = valid ? denc_g[(size_t)(2u * l) * ld + i] : 0.0f;
    const float e1 = valid ? denc_g[(size_t)(2u * l + 1u) * ld + i] : 0.0f;
    const V3 x = xyz(p4);
    uint32_t corner[8];
    float weight[8];
    cell_corners(gp, l, x, corner, weight);
#pragma unroll
    for (uint32_t c = 0; c < 8; ++c) {
        const float w = weight[c];
        uint32_t idx = off + corner[c];
        float2 v = make_float2(w * e0, w * e1);
        bool lead = valid;
        if (runs) {
            bool head;
            v = run_sum(valid ? idx : ~0u, v, head);
            lead = valid && head;
        }
        if constexpr (H16) {
            if (lead) unsafeAtomicAdd(grad_h + copy * entries + idx, __floats2half2_rn(v.x, v.y));
        } else {
            if (!lead) idx = ~0u;
            // quad_perm 0,0,2,2 and 1,1,3,3: the even, then the odd lane's
            // sample of each pair, its features on the pair's two lanes
            const uint32_t ie = dpp<0xA0>(idx), io = dpp<0xF5>(idx);
            const float ye = __uint_as_float(dpp<0xA0>(__float_as_uint(v.y)));
            const float xo = __uint_as_float(dpp<0xF5>(__float_as_uint(v.x)));
            const float ve = odd ? ye : v.x, vo = odd ? v.y : xo;
            if (ie != ~0u) unsafeAtomicAdd(grad_d + 2u * (size_t)ie + (odd ? 1u : 0u), (double)ve);
            if (io != ~0u) unsafeAtomicAdd(grad_d + 2u * (size_t)io + (odd ? 1u : 0u), (double)vo);
        }
    }
}

// The same levels in two kernels without global atomics (an XCD's L2 retires
// about one request of them per clock, 5.6 ms per 10^6 samples at full size).
// partition_kernel writes each chunk's corner
// gradients as records (entry, value), sorted by slice of the level's table;
// accumulate_kernel, one workgroup per (slice, level), adds its slice's records
// of every chunk into an LDS copy of the slice and stores it: every entry of
// the level is written once, so the gradients need no clearing either.
// FP32: 12-byte records, slices of up to 8,192 entries, FP64 LDS atomics (as
// scatter_lds64_kernel).  H16: 8-byte records of FP16 pairs (runs summed first,
// as in scatter_levels_kernel), the same slices; chunk c is of copy
// c % kHalfCopies, and the slice's copies are accumulated one after the other
// and summed in order.  Bound by the records' trip through memory (8 corners
// x 12 bytes, written and read) and, FP16, its LDS atomics: 100,003 random
// samples at full size take 50 + 82 us (scatter_levels_kernel: 698), the
// 225,000 samples of a training step under FP16 83 + 140 us (718).  With
// slices of 8,192 entries on every level the small dense ones, a few crowded
// slices, set the second kernel's time (310 and 250 us).
template <bool H16>
struct Part {
    static constexpr uint32_t kChunkSamples = H16 ? kLevelThreads : 1024u;
    static constexpr uint32_t kLanes = H16 ? 32u : 64u;  // lanes reading one chunk's records
    struct Rec32 {
        uint32_t idx;
        float x, y;
    };
    struct Rec16 {
        uint32_t idx;
        __half2 v;
    };
    using Rec = std::conditional_t<H16, Rec16, Rec32>;
    static constexpr uint32_t kMaxChunks = kPartPass / kChunkSamples;
    // per chunk: record slots, directory words (first record of each slice, end)
    static constexpr uint32_t kRecs = 8u * kChunkSamples;
    static constexpr uint32_t kDir = kPartSlices + 1u;
};
// A level has at most kPartSlices slices of 2^shift entries, and above 32 of
// them: a small dense level's records, which all fall near the skin, still
// spread over many workgroups.
INSTA_DEV uint32_t slice_shift(uint32_t size) {
    const uint32_t m = (size - 1u) / kPartSlices;
    return m ? 32u - (uint32_t)__builtin_clz(m) : 0u;
}

template <bool H16>
__global__ __launch_bounds__(Part<H16>::kChunkSamples) void partition_kernel(
    GridParams gp, uint32_t first_level, uint32_t run_mask, uint32_t pass0, const uint32_t* __restrict__ n_dev,
    const uint32_t* __restrict__ c_idx, const float4* __restrict__ cpos, const float* __restrict__ denc_g, uint32_t ld,
    typename Part<H16>::Rec* __restrict__ recs, uint32_t* __restrict__ dir) {
    using P = Part<H16>;
    __shared__ uint32_t s_cnt[kPartSlices], s_base[kPartSlices];
    const uint32_t n = *n_dev, s0 = pass0 + blockIdx.x * P::kChunkSamples;
    if (s0 >= n) return;
    const uint32_t l = first_level + blockIdx.y, t = threadIdx.x;
    const uint32_t shift = slice_shift(gp.size[l]);
    for (uint32_t j = t; j < kPartSlices; j += P::kChunkSamples) s_cnt[j] = 0u;
    __syncthreads();
    const bool valid = s0 + t < n;
    const uint32_t i = valid ? s0 + t : n - 1u;  // tail lanes repeat the last sample and emit nothing
    const float4 p4 = cpos[c_idx[i]];
    const float e0 = denc_g[(size_t)(2u * l) * ld + i], e1 = denc_g[(size_t)(2u * l + 1u) * ld + i];
    const V3 x = xyz(p4);
    uint32_t corner[8];
    float weight[8];
    cell_corners(gp, l, x, corner, weight);
    uint32_t idx[8], rank[8];
    float2 v[8];
#pragma unroll
    for (uint32_t c = 0; c < 8; ++c) {
        const float w = weight[c];
        idx[c] = corner[c];
        v[c] = make_float2(w * e0, w * e1);
        bool lead = valid;
        if constexpr (H16) {
            if ((run_mask >> l) & 1u) {
                bool head;
                v[c] = run_sum(valid ? idx[c] : ~0u, v[c], head);
                lead = valid && head;
            }
        }
        if (lead)
            rank[c] = atomicAdd(&s_cnt[idx[c] >> shift], 1u);
        else
            idx[c] = ~0u;
    }
    __syncthreads();
    // first record of each slice (one wave; at most 64 slices)
    const size_t chunk = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
    if (t < 64u) {
        const uint32_t cnt = t < kPartSlices ? s_cnt[t] : 0u;
        uint32_t incl = cnt;
#pragma unroll
        for (uint32_t o = 1; o < 64u; o <<= 1) {
            const uint32_t up = __shfl_up(incl, o);
            if (t >= o) incl += up;
        }
        if (t < kPartSlices) {
            s_base[t] = incl - cnt;
            dir[chunk * P::kDir + t] = incl - cnt;
            if (t == kPartSlices - 1u) dir[chunk * P::kDir + t + 1u] = incl;
        }
    }
    __syncthreads();
    typename P::Rec* __restrict__ out = recs + chunk * P::kRecs;
#pragma unroll
    for (uint32_t c = 0; c < 8; ++c) {
        if (idx[c] == ~0u) continue;
        const uint32_t slot = s_base[idx[c] >> shift] + rank[c];
        const uint32_t e = idx[c] & ((1u << shift) - 1u);
        if constexpr (H16)
            out[slot] = {e, __floats2half2_rn(v[c].x, v[c].y)};
        else
            out[slot] = {e, v[c].x, v[c].y};
    }
}

constexpr uint32_t kAccThreads = 1024;
template <bool H16>
__global__ __launch_bounds__(kAccThreads) void accumulate_kernel(GridParams gp, uint32_t first_level, uint32_t pass0,
                                                                 uint32_t chunks, const uint32_t* __restrict__ n_dev,
                                                                 const typename Part<H16>::Rec* __restrict__ recs,
                                                                 const uint32_t* __restrict__ dir,
                                                                 float* __restrict__ grad_tab) {
    using P = Part<H16>;
    constexpr uint32_t kSlice = kPartMaxEntries / kPartSlices;
    constexpr uint32_t kCopies = H16 ? kHalfCopies : 1u;
    constexpr uint32_t kPer = kSlice / kAccThreads;  // entries per thread
    struct D2 {
        double x, y;
    };
    using Entry = std::conditional_t<H16, __half2, D2>;
    __shared__ Entry tab[kSlice];  // 32 KB of FP16 pairs, 128 KB of FP64 pairs
    __shared__ uint2 s_dir[P::kMaxChunks];  // this slice's records of each chunk
    const uint32_t l = first_level + blockIdx.y, t = threadIdx.x;
    const uint32_t lane = t % P::kLanes, reader = t / P::kLanes;
    const uint32_t size = gp.size[l], shift = slice_shift(size), e0 = blockIdx.x << shift;
    if (e0 >= size) return;
    const uint32_t here = min(1u << shift, size - e0);
    const uint32_t n = *n_dev;
    if (pass0 && n <= pass0) return;  // nothing to add to the first pass's sums
    const uint32_t used = n > pass0 ? min((n - pass0 + P::kChunkSamples - 1u) / P::kChunkSamples, chunks) : 0u;
    for (uint32_t ch = t; ch < used; ch += kAccThreads) {
        const uint32_t* d = dir + ((size_t)blockIdx.y * chunks + ch) * P::kDir + blockIdx.x;
        s_dir[ch] = make_uint2(d[0], d[1]);
    }
    float2* __restrict__ out = reinterpret_cast<float2*>(grad_tab) + gp.offset[l] + e0;
    float2 acc[kPer];
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) {
        const uint32_t e = t + kAccThreads * q;
        acc[q] = pass0 && e < here ? out[e] : make_float2(0.0f, 0.0f);
    }
    for (uint32_t copy = 0; copy < kCopies; ++copy) {
        for (uint32_t e = t; e < here; e += kAccThreads) {
            if constexpr (H16)
                tab[e] = __floats2half2_rn(0.0f, 0.0f);
            else
                tab[e] = {0.0, 0.0};
        }
        __syncthreads();
        for (uint32_t ch = copy + reader * kCopies; ch < used; ch += kCopies * (kAccThreads / P::kLanes)) {
            const uint2 seg = s_dir[ch];
            const typename P::Rec* __restrict__ rec = recs + ((size_t)blockIdx.y * chunks + ch) * P::kRecs;
            auto add = [&](const typename P::Rec& x) {
                if constexpr (H16) {
                    unsafeAtomicAdd(&tab[x.idx], x.v);
                } else {
                    unsafeAtomicAdd(&tab[x.idx].x, (double)x.x);
                    unsafeAtomicAdd(&tab[x.idx].y, (double)x.y);
                }
            };
            uint32_t r = seg.x + lane;
            for (; r + 3u * P::kLanes < seg.y; r += 4u * P::kLanes) {  // four loads in flight
                const typename P::Rec a = rec[r], b = rec[r + P::kLanes], c = rec[r + 2u * P::kLanes],
                                      d = rec[r + 3u * P::kLanes];
                add(a);
                add(b);
                add(c);
                add(d);
            }
            for (; r < seg.y; r += P::kLanes) add(rec[r]);
        }
        __syncthreads();
#pragma unroll
        for (uint32_t q = 0; q < kPer; ++q) {
            const uint32_t e = t + kAccThreads * q;
            if (e >= here) break;
            const Entry v = tab[e];
            if constexpr (H16) {
                acc[q].x = acc[q].x + __low2float(v);
                acc[q].y = acc[q].y + __high2float(v);
            } else {
                acc[q].x = (float)((double)acc[q].x + v.x);
                acc[q].y = (float)((double)acc[q].y + v.y);
            }
        }
    }
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) {
        const uint32_t e = t + kAccThreads * q;
        if (e < here) out[e] = acc[q];
    }
}

// Gradients of the entries [first, entries) into grad_tab: the FP64 sums,
// rounded.
__global__ void grad_doubles_store_kernel(const double2* __restrict__ grad_d, uint64_t first, uint64_t entries,
                                          float* __restrict__ grad_tab) {
    for (uint64_t e = first + blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; e < entries;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const double2 v = grad_d[e];
        *reinterpret_cast<float2*>(grad_tab + 2 * e) = make_float2((float)v.x, (float)v.y);
    }
}

// The same of the FP16 copies, summed in copy order.
__global__ void grad_copies_reduce_kernel(const __half2* __restrict__ grad_h, uint64_t first, uint64_t entries,
                                          float* __restrict__ grad_tab) {
    for (uint64_t e = first + blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; e < entries;
         e += (uint64_t)gridDim.x * blockDim.x) {
        float a = 0.0f, b = 0.0f;
#pragma unroll
        for (uint32_t x = 0; x < kHalfCopies; ++x) {
            const __half2 h = grad_h[x * entries + e];
            a = a + __low2float(h);
            b = b + __high2float(h);
        }
        grad_tab[2 * e] = a;
        grad_tab[2 * e + 1] = b;
    }
}

// Backward of both MLPs over a block of 256 compacted samples (64 of a small
// batch), on FP32 MFMA in the forward kernel's layout (16 samples per step of a
// wave): the deltas through the transposed weights (held in LDS), the ReLU
// masks from the stored activations, each delta's rows stored for the weight
// gradients, and dL/dencoding through LDS to memory for the hash-grid
// scatters.  Bound by the latency of its chain of layers at 2 waves a SIMD, not
// by bandwidth (1.7 KB a sample): the masks of all layers are loaded at once
// (8,192 rays 228 -> 197 us, 1,000 samples 58 -> 48 us, 16 us in small tiles).
template <int L, int X>
__global__ __launch_bounds__(kMlpThreads) void train_backward_kernel(const float* __restrict__ params,
                                                                       const uint32_t* __restrict__ n_dev,
                                                                       const float* __restrict__ act,
                                                                       const float4* __restrict__ dout,
                                                                       float* __restrict__ dact, uint32_t ld,
                                                                       float* __restrict__ denc_g) {
    constexpr int E = 2 * L, DIN = E + X;  // encoding, density input (+ extra dims)
    using A = Act<DIN>;
    using O = Off<DIN>;
    typedef float bf4 __attribute__((ext_vector_type(4)));
    __shared__ __attribute__((aligned(16))) float w[O::N];  // both MLPs' weights
    __shared__ float s_denc[E][kMlpThreads];   // dL/dencoding of the block's samples
    const uint32_t n = *n_dev;
    const uint32_t cols = tile_columns(n), samples = 64u * cols;
    const uint32_t base = blockIdx.x * samples;
    if (base >= n) return;  // whole block past the batch
    static_assert(O::N % 4 == 0, "whole float4s of weights");
#pragma unroll 8
    for (uint32_t e = 4u * threadIdx.x; e < O::N; e += 4u * kMlpThreads)
        *reinterpret_cast<float4*>(w + e) = *reinterpret_cast<const float4*>(params + e);
    __syncthreads();
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t m = lane & 15u, g = lane >> 4;
    for (uint32_t nb = 0; nb < cols; ++nb) {
        // Opaque copies of 0 and ld: the weight reads (LDS) and the row
        // addresses of act/dact are formed inside this loop.  Loop-invariant,
        // they were otherwise hoisted out of it into ~360 registers (1 wave
        // per SIMD); recomputed per block of 16 samples, 248 (2 waves).
        uint32_t z = 0, ldz = ld;
        asm volatile("" : "+s"(z), "+s"(ldz));
        const float* W0 = w + O::W0 + z;
        const float* W1 = w + O::W1 + z;
        const float* W2 = w + O::W2 + z;
        const float* W3 = w + O::W3 + z;
        const float* W4 = w + O::W4 + z;
        const uint32_t s = (wave * cols + nb) * 16 + m;  // column (sample) of this lane
        const uint32_t i = base + s;
        const bool live = i < n;
        // the masks of all layers at once: loaded layer by layer, each layer
        // waited for its own
        bool on1[16], on2[16], on3[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const uint32_t row = 16 * (k / 4) + 4 * g + k % 4;
            on3[k] = live && act[(size_t)(A::H3 + row) * ldz + i] > 0.0f;
            on2[k] = live && act[(size_t)(A::H2 + row) * ldz + i] > 0.0f;
            on1[k] = live && act[(size_t)(A::H1 + row) * ldz + i] > 0.0f;
        }
        const float4 d4 = live ? dout[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        // colour output layer: dH3 = relu'(H3) (W4^T dRGB), K = 3 rgb rows (+ one zero)
        const float b_rgb = g == 0 ? d4.x : (g == 1 ? d4.y : (g == 2 ? d4.z : 0.0f));
        bf4 dh3[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            bf4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(g < 3 ? W4[g * kW + 16 * t + m] : 0.0f, b_rgb, acc, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t row = 16 * t + 4 * g + q;
                dh3[t][q] = on3[4 * t + q] ? acc[q] : 0.0f;
                if (live) dact[(size_t)(Dact::DH3 + row) * ldz + i] = dh3[t][q];
            }
        }
        // colour hidden layer: dH2 = relu'(H2) (W3^T dH3)
        bf4 dh2[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            bf4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(W3[(16 * s2 + 4 * g + b) * kW + 16 * t + m], dh3[s2][b],
                                                               acc, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t row = 16 * t + 4 * g + q;
                dh2[t][q] = on2[4 * t + q] ? acc[q] : 0.0f;
                if (live) dact[(size_t)(Dact::DH2 + row) * ldz + i] = dh2[t][q];
            }
        }
        // colour input restricted to the density outputs: dD = (W2^T dH2)[0..15], + dL/d(density logit) on row 0
        bf4 dd = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int b = 0; b < 4; ++b)
                dd = __builtin_amdgcn_mfma_f32_16x16x4f32(W2[(16 * t + 4 * g + b) * kCin + m], dh2[t][b], dd, 0, 0, 0);
        if (g == 0) dd[0] = dd[0] + d4.w;  // density logit = density-MLP output 0
        if (live)
#pragma unroll
            for (int q = 0; q < 4; ++q) dact[(size_t)(Dact::DDENS + 4 * g + q) * ldz + i] = dd[q];
        // density hidden layer: dH1 = relu'(H1) (W1^T dD)
        bf4 dh1[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            bf4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int b = 0; b < 4; ++b)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(W1[(4 * g + b) * kW + 16 * t + m], dd[b], acc, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t row = 16 * t + 4 * g + q;
                dh1[t][q] = on1[4 * t + q] ? acc[q] : 0.0f;
                if (live) dact[(size_t)(Dact::DH1 + row) * ldz + i] = dh1[t][q];
            }
        }
        // dL/dencoding = (W0^T dH1)[0..E), the extra dims' rows not needed
#pragma unroll
        for (int te = 0; te < E / 16; ++te) {
            bf4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(W0[(16 * s2 + 4 * g + b) * DIN + 16 * te + m],
                                                               dh1[s2][b], acc, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) s_denc[16 * te + 4 * g + q][s] = acc[q];
        }
    }
    __syncthreads();
    const uint32_t i = base + tid % samples, part = tid / samples;
    if ((i & ~63u) >= n) return;  // whole wave past the batch (no barrier follows)
    const bool valid = i < n;
    if (valid && part == 0) {
        const float4 d4 = dout[i];
        dact[(size_t)(Dact::DRGB + 0) * ld + i] = d4.x;
        dact[(size_t)(Dact::DRGB + 1) * ld + i] = d4.y;
        dact[(size_t)(Dact::DRGB + 2) * ld + i] = d4.z;
    }
    // dL/dencoding for the scatter kernels
    if (valid)
#pragma unroll 4
        for (uint32_t e = part; e < E; e += 4u / cols) denc_g[(size_t)e * ld + i] = s_denc[e][tid % samples];
}


struct WProduct {
    uint32_t d_row, x_row, O, I, out;
};
struct WArgs {
    WProduct p[5];
};

// partial[c][out + o*I + i] = sum over samples n of chunk c of
// dact[d_row + o][n] * act[x_row + i][n], on v_mfma_f32_16x16x4f32: the
// samples are the K dimension; kS-sample slices of both operands are staged
// through LDS (each thread loads 4 consecutive samples of kPass rows of
// each operand as float4, coalesced along the samples), wave w owns input
// tile i = 16w..16w+15 and the four output tiles o = 0..63 of it, one MFMA
// per tile and 4 samples (A = 16 outputs x 4 samples, B = 4 samples x 16
// inputs).
typedef float wg_f4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void wgrad_kernel(WArgs wa, const uint32_t* __restrict__ n_dev,
                                                    const float* __restrict__ act, const float* __restrict__ dact,
                                                    uint32_t ld, float* __restrict__ part, uint32_t n_mlp) {
    constexpr uint32_t kS = 32;            // samples per LDS slice
    constexpr uint32_t kP = kS + 4;        // LDS row pitch: fragment reads (16 rows x 4 samples) spread over the banks
    constexpr uint32_t kRowsPass = 1024u / kS;  // rows one pass of 256 threads covers (kS / 4 threads per row)
    constexpr uint32_t kPass = 64u / kRowsPass;
    __shared__ float Ds[64 * kP];
    __shared__ float Xs[64 * kP];
    const WProduct pr = wa.p[blockIdx.y];
    const uint32_t n = *n_dev;
    const uint32_t chunk = wgrad_chunk(n), s0 = blockIdx.x * chunk;
    if (s0 >= n) return;
    const uint32_t s1 = min(s0 + chunk, n);
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const uint32_t m = lane & 15u, g = lane >> 4;   // fragment row / k of this lane
    const uint32_t n_ot = (pr.O + 15u) / 16u;       // output tiles in use
    const bool active = 16u * wave < pr.I;          // this wave's input tile exists
    const bool vec = (ld & 3u) == 0u;               // rows 16-byte aligned
    const uint32_t c4 = (t % (kS / 4u)) * 4u;       // this thread's first sample in a slice
    const uint32_t r0 = t / (kS / 4u);              // its rows r0 + kRowsPass p
    wg_f4 acc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] = wg_f4{0.0f, 0.0f, 0.0f, 0.0f};
    const float* dp[kPass];
    const float* xp[kPass];
#pragma unroll
    for (uint32_t q = 0; q < kPass; ++q) {
        const uint32_t row = r0 + kRowsPass * q;
        dp[q] = row < pr.O ? dact + (size_t)(pr.d_row + row) * ld : nullptr;
        xp[q] = row < pr.I ? act + (size_t)(pr.x_row + row) * ld : nullptr;
    }
    auto ld4 = [&](const float* p, uint32_t smp) -> float4 {
        if (!p) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (vec && smp + 4u <= s1) return *reinterpret_cast<const float4*>(p + smp);
        return make_float4(smp < s1 ? p[smp] : 0.0f, smp + 1u < s1 ? p[smp + 1u] : 0.0f,
                           smp + 2u < s1 ? p[smp + 2u] : 0.0f, smp + 3u < s1 ? p[smp + 3u] : 0.0f);
    };
    // next slice in registers while the current one is multiplied
    float4 dn[kPass], xn[kPass];
    auto fetch = [&](uint32_t s) {
#pragma unroll
        for (uint32_t q = 0; q < kPass; ++q) {
            dn[q] = ld4(dp[q], s + c4);
            xn[q] = ld4(xp[q], s + c4);
        }
    };
    fetch(s0);
    for (uint32_t s = s0; s < s1; s += kS) {
#pragma unroll
        for (uint32_t q = 0; q < kPass; ++q) {
            const uint32_t row = r0 + kRowsPass * q;
            *reinterpret_cast<float4*>(&Ds[row * kP + c4]) = dn[q];
            *reinterpret_cast<float4*>(&Xs[row * kP + c4]) = xn[q];
        }
        __syncthreads();
        if (s + kS < s1) fetch(s + kS);
        // one output tile (O <= 16) or all four (rows past O are zero):
        // straight-line MFMAs, the accumulators stay in place
        auto mma = [&](auto tiles) {
#pragma unroll
            for (uint32_t k0 = 0; k0 < kS; k0 += 4u) {
                const float b = Xs[(16u * wave + m) * kP + k0 + g];
#pragma unroll
                for (uint32_t ot = 0; ot < decltype(tiles)::value; ++ot)
                    acc[ot] = __builtin_amdgcn_mfma_f32_16x16x4f32(Ds[(16u * ot + m) * kP + k0 + g], b, acc[ot],
                                                                    0, 0, 0);
            }
        };
        if (active) {
            if (n_ot <= 1u)
                mma(std::integral_constant<uint32_t, 1>{});
            else
                mma(std::integral_constant<uint32_t, 4>{});
        }
        __syncthreads();
    }
    if (!active) return;
    // lane holds C[o = 16 ot + 4 g + j][i = 16 wave + m]
    const uint32_t ii = 16u * wave + m;
#pragma unroll
    for (uint32_t ot = 0; ot < 4u; ++ot)
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) {
            const uint32_t o = 16u * ot + 4u * g + j;
            if (o < pr.O && ii < pr.I) part[(size_t)blockIdx.x * n_mlp + pr.out + o * pr.I + ii] = acc[ot][j];
        }
}

__global__ void wgrad_reduce_kernel(const float* __restrict__ part, const uint32_t* __restrict__ n_dev,
                                    uint32_t n_mlp, float* __restrict__ grad) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_mlp) return;
    const uint32_t n = *n_dev, chunk = wgrad_chunk(n), nc = (n + chunk - 1) / chunk;
    // eight interleaved running sums (chunk c into sum c mod 8), added in a
    // fixed order: deterministic, with eight independent loads in flight
    float s[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t c = 0;
    for (; c + 8 <= nc; c += 8)
#pragma unroll
        for (uint32_t r = 0; r < 8; ++r) s[r] += part[(size_t)(c + r) * n_mlp + p];
#pragma unroll
    for (uint32_t r = 0; r < 8; ++r)
        if (c + r < nc) s[r] += part[(size_t)(c + r) * n_mlp + p];
    grad[p] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}

// Unscale, optionally step Adam.  grad[] receives dL/dparam (unscaled).
__global__ void adam_kernel(float* __restrict__ params, float* __restrict__ grad, float* __restrict__ m,
                            float* __restrict__ v, uint64_t n_params, float inv_scale, float lr, float b1, float b2,
                            float eps, float bc1, float bc2, float l2_reg, uint32_t apply) {
    for (uint64_t p = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; p < n_params;
         p += (uint64_t)gridDim.x * blockDim.x) {
        float g = grad[p] * inv_scale;
        grad[p] = g;
        if (apply) {
            g = g + l2_reg * params[p];
            const float mm = b1 * m[p] + (1.0f - b1) * g;
            const float vv = b2 * v[p] + (1.0f - b2) * (g * g);
            m[p] = mm;
            v[p] = vv;
            params[p] = params[p] - lr * (mm / bc1) / (sqrtf(vv / bc2) + eps);
        }
    }
}

// Ema around the optimizer: a = decay * a + (1 - decay) * w (a starts at 0
// with the first update), and the debiased average a * debias, debias =
// 1 / (1 - decay^t), for inference
__global__ void ema_kernel(const float* __restrict__ w, float* __restrict__ a, float* __restrict__ infer,
                           uint64_t n, float decay, float debias, uint32_t first) {
    for (uint64_t p = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; p < n; p += (uint64_t)gridDim.x * blockDim.x) {
        const float prev = first ? 0.0f : a[p];
        const float v = decay * prev + (1.0f - decay) * w[p];
        a[p] = v;
        infer[p] = v * debias;
    }
}

template <class T>
bool train_alloc(T*& p, size_t bytes) {
    return hipMalloc(reinterpret_cast<void**>(&p), bytes) == hipSuccess;
}

void free_workspace_train(TrainState* ts) {
    dev_free(ts->ray_d); dev_free(ts->ray_o); dev_free(ts->ray_frame); dev_free(ts->ray_img); dev_free(ts->ray_pix);
    dev_free(ts->ray_src); dev_free(ts->ray_base); dev_free(ts->ray_cnt);
    dev_free(ts->s_cpos); dev_free(ts->s_cdir); dev_free(ts->s_out); dev_free(ts->s_hit);
    dev_free(ts->c_idx); dev_free(ts->c_dout); dev_free(ts->act); dev_free(ts->dact); dev_free(ts->part);
    dev_free(ts->t_buf);
    dev_free(ts->denc); dev_free(ts->recs); dev_free(ts->rec_dir);
    ts->part_levels = 0;
    dev_free(ts->ray_T); dev_free(ts->ray_alive); dev_free(ts->ray_gbase);
    dev_free(ts->r_pos); dev_free(ts->r_cpos); dev_free(ts->r_cdir); dev_free(ts->r_out);
    ts->ray_cap = ts->sample_cap = ts->compact_cap = 0;
}

uint32_t largest_table(const insta_ctx* ctx) {
    const GridParams gp = grid_params(ctx);
    return *std::max_element(gp.size, gp.size + ctx->cfg.n_levels);
}

// rays, marched samples and the compacted batch grow independently to the
// largest request seen
// grow the training workspace to hold n_rays rays, n_samples marched samples
// and a compacted batch of n_compact (insta_reserve only)
insta_status grow_train_workspace(insta_ctx* ctx, TrainState* ts, uint32_t n_rays, uint32_t n_samples,
                                  uint32_t n_compact) {
    if (n_rays <= ts->ray_cap && n_samples <= ts->sample_cap && n_compact <= ts->compact_cap) return INSTA_OK;
    const uint32_t rc = std::max(n_rays, ts->ray_cap), sc = std::max(n_samples, ts->sample_cap);
    const uint32_t cc = std::max(n_compact, ts->compact_cap);
    free_workspace_train(ts);
    const int DIN = (int)(ctx->cfg.n_levels * 2 + ctx->cfg.n_extra_dims);
    const size_t act_rows = (size_t)DIN + 224, n_mlp = ctx->layout.n_mlp_params;
    bool ok = true;
    ok = ok && train_alloc(ts->ray_d, rc * sizeof(float4)) && train_alloc(ts->ray_o, rc * sizeof(float4)) &&
         train_alloc(ts->ray_frame, rc * sizeof(int32_t));
    ok = ok && train_alloc(ts->ray_img, rc * 4) && train_alloc(ts->ray_pix, rc * 4) && train_alloc(ts->ray_src, rc * 4);
    ok = ok && train_alloc(ts->ray_base, rc * 4) && train_alloc(ts->ray_cnt, rc * 4);
    ok = ok && train_alloc(ts->s_cpos, sc * sizeof(float4));
    ok = ok && train_alloc(ts->s_cdir, sc * sizeof(float4)) && train_alloc(ts->s_out, sc * sizeof(float4));
    ok = ok && train_alloc(ts->s_hit, sc * sizeof(int32_t));
    ok = ok && train_alloc(ts->ray_T, rc * sizeof(float)) && train_alloc(ts->ray_alive, rc * 4) &&
         train_alloc(ts->ray_gbase, rc * 4);
    ok = ok && train_alloc(ts->r_pos, sc * sizeof(float4)) && train_alloc(ts->r_cpos, sc * sizeof(float4));
    ok = ok && train_alloc(ts->r_cdir, sc * sizeof(float4)) && train_alloc(ts->r_out, sc * sizeof(float4));
    ok = ok && train_alloc(ts->c_idx, cc * sizeof(uint32_t)) && train_alloc(ts->c_dout, cc * sizeof(float4));
    ok = ok && train_alloc(ts->act, act_rows * cc * sizeof(float));
    ok = ok && train_alloc(ts->dact, (size_t)Dact::N * cc * sizeof(float));
    ok = ok && train_alloc(ts->part, (size_t)wgrad_chunks(cc) * n_mlp * sizeof(float));
    ok = ok && train_alloc(ts->t_buf, (size_t)rc * ctx->cfg.max_steps * sizeof(float));
    ok = ok && train_alloc(ts->denc, (size_t)2 * INSTA_MAX_LEVELS * cc * sizeof(float));
    const uint32_t big = ctx->cfg.n_levels - (uint32_t)__builtin_popcount(ts->lds_levels);
    if (big && largest_table(ctx) <= kPartMaxEntries) {
        const size_t pass = std::min(cc, kPartPass);
        const size_t c32 = (pass + Part<false>::kChunkSamples - 1) / Part<false>::kChunkSamples;
        const size_t c16 = (pass + Part<true>::kChunkSamples - 1) / Part<true>::kChunkSamples;
        const size_t rec_bytes = std::max(c32 * Part<false>::kRecs * sizeof(Part<false>::Rec),
                                          c16 * Part<true>::kRecs * sizeof(Part<true>::Rec));
        const size_t dirs = std::max(c32 * Part<false>::kDir, c16 * Part<true>::kDir);
        ok = ok && train_alloc(ts->recs, big * rec_bytes) && train_alloc(ts->rec_dir, big * dirs * sizeof(uint32_t));
        if (ok) ts->part_levels = big;
    }
    if (!ok) {
        free_workspace_train(ts);
        set_error("training workspace allocation failed");
        return INSTA_ERR_OOM;
    }
    ts->ray_cap = rc;
    ts->sample_cap = sc;
    ts->compact_cap = cc;
    return INSTA_OK;
}

// a step or plugin call must fit the reserved workspace: nothing is allocated per call
insta_status check_train_workspace(const TrainState* ts, uint32_t n_rays, uint32_t n_samples, uint32_t n_compact,
                                   const char* who) {
    if (n_rays <= ts->ray_cap && n_samples <= ts->sample_cap && n_compact <= ts->compact_cap) return INSTA_OK;
    set_error(std::string(who) + ": needs " + std::to_string(n_rays) + " rays, " + std::to_string(n_samples) +
              " samples, a batch of " + std::to_string(n_compact) + "; reserved " + std::to_string(ts->ray_cap) +
              " / " + std::to_string(ts->sample_cap) + " / " + std::to_string(ts->compact_cap) +
              ": reserve them with insta_reserve (train_rays, train_samples, train_batch)");
    return INSTA_ERR_STATE;
}

template <int L, int X>
insta_status launch_train_forward(insta_ctx* ctx, TrainState* ts, hipStream_t stream) {
    const uint32_t cap = ts->compact_cap;
    const uint32_t* n_dev = ts->counters + kTCompactN;
    const float* table = ctx->d_params + ctx->layout.n_mlp_params;
    const GridParams gp = grid_params(ctx);
    const dim3 sgrid(mlp_blocks(cap));
    hipLaunchKernelGGL((train_forward_kernel<L, X>), sgrid, dim3(kFwdTile), 0, stream, ctx->d_params, table, gp,
                       ctx->d_frame_extra, ctx->cfg.max_frames, n_dev, ts->c_idx, ts->s_cpos, ts->s_cdir,
                       static_cast<const float*>(nullptr), ts->act, cap, static_cast<float4*>(nullptr));
    INSTA_HIP(hipGetLastError());
    return INSTA_OK;
}

template <bool H16>
void launch_partition(TrainState* ts, const GridParams& gp, uint32_t run_mask, uint32_t pass0, float* grad_tab,
                      hipStream_t stream) {
    using P = Part<H16>;
    const uint32_t cap = ts->compact_cap, first = (uint32_t)__builtin_popcount(ts->lds_levels);
    const uint32_t chunks = (std::min(cap - pass0, kPartPass) + P::kChunkSamples - 1) / P::kChunkSamples;
    typename P::Rec* recs = reinterpret_cast<typename P::Rec*>(ts->recs);
    const uint32_t* n_dev = ts->counters + kTCompactN;
    hipLaunchKernelGGL(partition_kernel<H16>, dim3(chunks, ts->part_levels), dim3(P::kChunkSamples), 0, stream, gp,
                       first, run_mask, pass0, n_dev, ts->c_idx, ts->s_cpos, ts->denc, cap, recs, ts->rec_dir);
    hipLaunchKernelGGL(accumulate_kernel<H16>, dim3(kPartSlices, ts->part_levels), dim3(kAccThreads), 0, stream, gp,
                       first, pass0, chunks, n_dev, recs, ts->rec_dir, grad_tab);
}

template <int L, int X>
insta_status launch_train_backward(insta_ctx* ctx, TrainState* ts, const insta_train_config& tc, hipStream_t stream) {
    constexpr int DIN = 2 * L + X;
    using A = Act<DIN>;
    using O = Off<DIN>;
    const uint32_t cap = ts->compact_cap;
    const uint32_t* n_dev = ts->counters + kTCompactN;
    const GridParams gp = grid_params(ctx);
    const uint32_t n_mlp = (uint32_t)ctx->layout.n_mlp_params;
    const dim3 sgrid(mlp_blocks(cap));
    float* grad_tab = ts->grad + n_mlp;
    // levels whose tables fit in LDS are scattered by scatter_lds64_kernel
    // (FP16: scatter_lds_kernel), the others partitioned or, with tables too
    // large for that, by scatter_levels_kernel
    const uint32_t lds_mask = ts->lds_levels, lds_end = ts->lds_end;
    const uint32_t big_mask = ((1u << L) - 1u) & ~lds_mask;
    // levels whose cells span at least 1 / kRunMaxStepCells marching steps
    uint32_t run_mask = 0;
    for (int l = 0; l < L; ++l)
        if (ctx->cfg.dt * gp.scale[l] <= kRunMaxStepCells) run_mask |= 1u << l;
    hipLaunchKernelGGL((train_backward_kernel<L, X>), sgrid, dim3(kMlpThreads), 0, stream, ctx->d_params, n_dev, ts->act,
                       ts->c_dout, ts->dact, cap, ts->denc);
    INSTA_HIP(hipGetLastError());
    const uint32_t chunks =
        std::min<uint32_t>(std::max<uint32_t>((cap + kScatterChunk - 1) / kScatterChunk, 1u), kScatterMaxChunks);
    if (lds_mask) {
        const dim3 grid(chunks, __builtin_popcount(lds_mask));
        if (tc.grid_grad_fp16)
            hipLaunchKernelGGL(scatter_lds_kernel, grid, dim3(kScatterThreads), 0, stream, gp, n_dev, ts->c_idx,
                               ts->s_cpos, ts->denc, cap, run_mask, ts->grad_p, lds_end);
        else
            hipLaunchKernelGGL(scatter_lds64_kernel, dim3(grid.x, grid.y, 2), dim3(kScatterThreads), 0, stream, gp,
                               n_dev, ts->c_idx, ts->s_cpos, ts->denc, cap, ts->grad_p, lds_end);
        hipLaunchKernelGGL(grad_partials_reduce_kernel, dim3((lds_end + 255) / 256), dim3(256), 0, stream, ts->grad_p,
                           lds_end, chunks, grad_tab);
        INSTA_HIP(hipGetLastError());
    }
    if (big_mask && ts->part_levels) {
        for (uint32_t pass0 = 0; pass0 < cap; pass0 += kPartPass) {
            if (tc.grid_grad_fp16)
                launch_partition<true>(ts, gp, run_mask, pass0, grad_tab, stream);
            else
                launch_partition<false>(ts, gp, run_mask, pass0, grad_tab, stream);
        }
        INSTA_HIP(hipGetLastError());
    } else if (big_mask) {
        const uint64_t entries = ctx->layout.n_grid_params / 2;
        const uint32_t blocks =
            ((cap + kLevelThreads - 1) / kLevelThreads + kHalfCopies - 1) / kHalfCopies * kHalfCopies;
        const uint32_t slots = (__builtin_popcount(big_mask) + kXcds - 1) / kXcds;
        const dim3 grid(kXcds * slots * blocks);
        if (tc.grid_grad_fp16) {
            // clear this backward's copies (fill kernels: capturable)
            hipLaunchKernelGGL(fill_zero_kernel, dim3(2048), dim3(256), 0, stream,
                               reinterpret_cast<uint32_t*>(ts->grad_h), kHalfCopies * entries);
            hipLaunchKernelGGL(scatter_levels_kernel<true>, grid, dim3(kLevelThreads), 0, stream, gp, big_mask,
                               run_mask, blocks, n_dev, ts->c_idx, ts->s_cpos, ts->denc, cap,
                               reinterpret_cast<double*>(ts->grad_d), ts->grad_h, entries);
            hipLaunchKernelGGL(grad_copies_reduce_kernel, dim3(2048), dim3(256), 0, stream, ts->grad_h,
                               (uint64_t)lds_end, entries, grad_tab);
        } else {
            hipLaunchKernelGGL(fill_zero_kernel, dim3(2048), dim3(256), 0, stream,
                               reinterpret_cast<uint32_t*>(ts->grad_d + lds_end), 4 * (entries - lds_end));
            hipLaunchKernelGGL(scatter_levels_kernel<false>, grid, dim3(kLevelThreads), 0, stream, gp, big_mask,
                               run_mask, blocks, n_dev, ts->c_idx, ts->s_cpos, ts->denc, cap,
                               reinterpret_cast<double*>(ts->grad_d), ts->grad_h, entries);
            hipLaunchKernelGGL(grad_doubles_store_kernel, dim3(2048), dim3(256), 0, stream, ts->grad_d,
                               (uint64_t)lds_end, entries, grad_tab);
        }
        INSTA_HIP(hipGetLastError());
    }
    WArgs wa;
    wa.p[0] = WProduct{Dact::DH1, A::ENC, kW, DIN, O::W0};
    wa.p[1] = WProduct{Dact::DDENS, A::H1, kDOut, kW, O::W1};
    wa.p[2] = WProduct{Dact::DH2, A::DENS, kW, kCin, O::W2};
    wa.p[3] = WProduct{Dact::DH3, A::H2, kW, kW, O::W3};
    wa.p[4] = WProduct{Dact::DRGB, A::H3, 3, kW, O::W4};
    const uint32_t n_chunks = wgrad_chunks(cap);
    hipLaunchKernelGGL(wgrad_kernel, dim3(n_chunks, 5), dim3(256), 0, stream, wa, n_dev, ts->act, ts->dact, cap,
                       ts->part, n_mlp);
    INSTA_HIP(hipGetLastError());
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3((n_mlp + 255) / 256), dim3(256), 0, stream, ts->part, n_dev, n_mlp,
                       ts->grad);
    INSTA_HIP(hipGetLastError());
    return INSTA_OK;
}

// ---- NerfNetwork plugin (nerf_network.h:238-383): forward with stored
// activations and backward on caller-given samples, through the training
// step's kernels; the batch is the caller's samples in order (c_idx = i).
__global__ void net_prepare_kernel(const float* __restrict__ coords, uint32_t n, uint32_t stride, uint32_t X,
                                   float4* __restrict__ cpos, float4* __restrict__ cdir, uint32_t* __restrict__ c_idx,
                                   float* __restrict__ x_extra, uint32_t* __restrict__ counters) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) counters[kTCompactN] = n;
    if (i >= n) return;
    const float* c = coords + (size_t)i * stride;
    cpos[i] = make_float4(c[0], c[1], c[2], 0.0f);
    cdir[i] = make_float4(c[8], c[9], c[10], __uint_as_float(kExtraOnes));
    c_idx[i] = i;
    // the density input's extra dims are the coordinate's last X floats
    // (forward_impl's extract_expressions, nerf_network.h:253-262)
    for (uint32_t e = 0; e < X; ++e) x_extra[(size_t)i * X + e] = c[stride - X + e];
}

// param_gradients_mode Overwrite / Accumulate
__global__ void net_grad_out_kernel(const float* __restrict__ g, float* __restrict__ out, uint64_t n,
                                    uint32_t accumulate) {
    for (uint64_t p = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; p < n; p += (uint64_t)gridDim.x * blockDim.x)
        out[p] = accumulate ? out[p] + g[p] : g[p];
}

// Input gradients of the backward (dL_dinput rows 0..2 and the direction rows
// 8..10; the reference backpropagates through the position and direction
// encodings only, nerf_network.h:318-380): dL/dencoding as the backward stored
// it and dL/dSH = W2[:, 16:32]^T dH2 from the stored deltas; the position through
// the derivative of each level's trilinear weights (scale_l per axis) times
// the corner features, the direction (input in [0,1], d = 2 x - 1) through
// the derivatives of the 16 SH polynomials.
INSTA_DEV void sh16_grad(float x, float y, float z, const float* g, float out[3]) {
    const float C1 = 0.48860251190291987f, C2 = 1.0925484305920792f, C3 = 0.94617469575755997f;
    const float C4 = 0.54627421529603959f, C5 = 0.59004358992664352f, C6 = 2.8906114426405538f;
    const float C7 = 0.45704579946446572f, C8 = 0.3731763325901154f, C9 = 1.4453057213202769f;
    float dx = 0.0f, dy = 0.0f, dz = 0.0f;
    dy += g[1] * -C1;
    dz += g[2] * C1;
    dx += g[3] * -C1;
    dx += g[4] * (C2 * y); dy += g[4] * (C2 * x);
    dy += g[5] * (-C2 * z); dz += g[5] * (-C2 * y);
    dz += g[6] * (2.0f * C3 * z);
    dx += g[7] * (-C2 * z); dz += g[7] * (-C2 * x);
    dx += g[8] * (2.0f * C4 * x); dy += g[8] * (-2.0f * C4 * y);
    dx += g[9] * (-6.0f * C5 * x * y); dy += g[9] * (C5 * (3.0f * y * y - 3.0f * x * x));
    dx += g[10] * (C6 * y * z); dy += g[10] * (C6 * x * z); dz += g[10] * (C6 * x * y);
    dy += g[11] * (C7 * (1.0f - 5.0f * z * z)); dz += g[11] * (-10.0f * C7 * y * z);
    dz += g[12] * (C8 * (15.0f * z * z - 3.0f));
    dx += g[13] * (C7 * (1.0f - 5.0f * z * z)); dz += g[13] * (-10.0f * C7 * x * z);
    dx += g[14] * (2.0f * C9 * x * z); dy += g[14] * (-2.0f * C9 * y * z); dz += g[14] * (C9 * (x * x - y * y));
    dx += g[15] * (C5 * (3.0f * y * y - 3.0f * x * x)); dy += g[15] * (6.0f * C5 * x * y);
    out[0] = dx;
    out[1] = dy;
    out[2] = dz;
}

template <int L, int X>
__global__ __launch_bounds__(128) void net_input_grad_kernel(const float* __restrict__ params,
                                                             const float* __restrict__ table, GridParams gp,
                                                             uint32_t n, const float4* __restrict__ cpos,
                                                             const float4* __restrict__ cdir,
                                                             const float* __restrict__ dact,
                                                             const float* __restrict__ denc_g, uint32_t ld,
                                                             float* __restrict__ dL_dinput, uint32_t stride) {
    constexpr int E = 2 * L, DIN = E + X;
    using O = Off<DIN>;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float dsh[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) dsh[j] = 0.0f;
#pragma unroll 16
    for (int k = 0; k < kW; ++k) {
        const float d2 = dact[(size_t)(Dact::DH2 + k) * ld + i];
#pragma unroll
        for (int j = 0; j < 16; ++j) dsh[j] += params[O::W2 + k * kCin + 16 + j] * d2;
    }
    const float4 p4 = cpos[i];
    float gx[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll 2
    for (int l = 0; l < L; ++l) {
        const float sc = gp.scale[l];
        const float de0 = denc_g[(size_t)(2 * l) * ld + i], de1 = denc_g[(size_t)(2 * l + 1) * ld + i];
        float frac[3], weight[8];
        float2 v[8];
        cell_fetch(gp, (uint32_t)l, xyz(p4), reinterpret_cast<const char*>(table + 2 * (size_t)gp.offset[l]), v, frac,
                   weight);
#pragma unroll
        for (uint32_t c = 0; c < 8; ++c) {
            float wk[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) wk[k] = ((c >> k) & 1u) ? frac[k] : 1.0f - frac[k];
            const float s = de0 * v[c].x + de1 * v[c].y;
            gx[0] += s * (((c & 1u) ? sc : -sc) * wk[1] * wk[2]);
            gx[1] += s * (((c & 2u) ? sc : -sc) * wk[0] * wk[2]);
            gx[2] += s * (((c & 4u) ? sc : -sc) * wk[0] * wk[1]);
        }
    }
    const float4 d4 = cdir[i];
    float gd[3];
    sh16_grad(d4.x * 2.0f - 1.0f, d4.y * 2.0f - 1.0f, d4.z * 2.0f - 1.0f, dsh, gd);
    float* o = dL_dinput + (size_t)i * stride;
    o[0] = gx[0];
    o[1] = gx[1];
    o[2] = gx[2];
    o[8] = 2.0f * gd[0];
    o[9] = 2.0f * gd[1];
    o[10] = 2.0f * gd[2];
}

template <int L, int X>
insta_status launch_net_forward(insta_ctx* ctx, TrainState* ts, float4* out, hipStream_t stream) {
    const uint32_t cap = ts->compact_cap;
    const float* table = ctx->d_params + ctx->layout.n_mlp_params;
    hipLaunchKernelGGL((train_forward_kernel<L, X>), dim3(mlp_blocks(cap)), dim3(kFwdTile), 0, stream,
                       ctx->d_params, table, grid_params(ctx), ctx->d_frame_extra, ctx->cfg.max_frames,
                       ts->counters + kTCompactN, ts->c_idx, ts->s_cpos, ts->s_cdir,
                       X ? static_cast<const float*>(ts->net_extra) : nullptr, ts->act, cap, out);
    INSTA_HIP(hipGetLastError());
    return INSTA_OK;
}

template <int L, int X>
insta_status launch_net_input_grad(insta_ctx* ctx, TrainState* ts, uint32_t n, float* dL_dinput, uint32_t stride,
                                   hipStream_t stream) {
    const float* table = ctx->d_params + ctx->layout.n_mlp_params;
    hipLaunchKernelGGL((net_input_grad_kernel<L, X>), dim3((n + 127) / 128), dim3(128), 0, stream, ctx->d_params,
                       table, grid_params(ctx), n, ts->s_cpos, ts->s_cdir, ts->dact, ts->denc, ts->compact_cap, dL_dinput,
                       stride);
    INSTA_HIP(hipGetLastError());
    return INSTA_OK;
}

}  // namespace

bool train_supported(const insta_config& c) {
    return c.n_neurons == 64 && c.density_out == 16 && c.sh_degree == 4 && (c.n_extra_dims == 0 || c.n_extra_dims == 16) &&
           c.density_hidden_layers == 1 && c.rgb_hidden_layers == 2 && c.n_features_per_level == 2 &&
           (c.n_levels == 8 || c.n_levels == 16);
}

void free_train(insta_ctx* ctx) {
    TrainState* ts = ctx->train;
    if (!ts) return;
    free_workspace_train(ts);
    dev_free(ts->images); dev_free(ts->meta); dev_free(ts->seg); dev_free(ts->depth);
    dev_free(ts->grad); dev_free(ts->grad_d); dev_free(ts->grad_p);
    dev_free(ts->adam_m); dev_free(ts->adam_v); dev_free(ts->counters); dev_free(ts->net_extra);
    if (ctx->net_src == ts->ema_infer) ctx->net_src = nullptr;
    dev_free(ts->ema); dev_free(ts->ema_infer);
    if (ts->h_counters) (void)hipHostFree(ts->h_counters);
    delete ts;
    ctx->train = nullptr;
}

// gradients, optimizer moments and counters: created once per context
static insta_status ensure_train_state(insta_ctx* ctx, hipStream_t stream) {
    if (!ctx->train) {
        TrainState* ts = new (std::nothrow) TrainState();
        if (!ts) {
            set_error("host allocation failed");
            return INSTA_ERR_OOM;
        }
        ctx->train = ts;
        const uint64_t np = ctx->layout.n_params;
        ts->lds_levels = lds_scatter_levels(grid_params(ctx), (int)ctx->cfg.n_levels, &ts->lds_end);
        bool ok = train_alloc(ts->grad, np * sizeof(float)) && train_alloc(ts->adam_m, np * sizeof(float)) &&
                  train_alloc(ts->adam_v, np * sizeof(float)) && train_alloc(ts->ema, np * sizeof(float)) &&
                  train_alloc(ts->ema_infer, np * sizeof(float)) &&
                  (largest_table(ctx) <= kPartMaxEntries ||
                   train_alloc(ts->grad_d, kHalfCopies * (ctx->layout.n_grid_params / 2) * sizeof(__half2))) &&
                  (ts->lds_end == 0 ||
                   train_alloc(ts->grad_p, (size_t)kScatterMaxChunks * 2 * ts->lds_end * sizeof(float))) &&
                  train_alloc(ts->counters, kTCounters * sizeof(uint32_t)) &&
                  hipHostMalloc((void**)&ts->h_counters, kTCounters * sizeof(uint32_t), hipHostMallocDefault) ==
                      hipSuccess;
        if (!ok) {
            free_train(ctx);
            set_error("training state allocation failed");
            return INSTA_ERR_OOM;
        }
        ts->grad_h = reinterpret_cast<__half2*>(ts->grad_d);
        INSTA_HIP(hipMemsetAsync(ts->adam_m, 0, np * sizeof(float), stream));
        INSTA_HIP(hipMemsetAsync(ts->adam_v, 0, np * sizeof(float), stream));
    }
    return INSTA_OK;
}

insta_status set_training_set(insta_ctx* ctx, uint32_t n_images, uint32_t width, uint32_t height, const float* rgba,
                              const insta_camera* cams, const int32_t* frames, hipStream_t stream) {
    insta_status st = ensure_train_state(ctx, stream);
    if (st != INSTA_OK) return st;
    TrainState* ts = ctx->train;
    dev_free(ts->images);
    dev_free(ts->meta);
    dev_free(ts->seg);    // a new set starts without supervision
    dev_free(ts->depth);
    const size_t px = (size_t)n_images * width * height;
    if (!train_alloc(ts->images, px * sizeof(float4)) || !train_alloc(ts->meta, n_images * sizeof(TrainImage))) {
        set_error("training image allocation failed");
        return INSTA_ERR_OOM;
    }
    std::vector<TrainImage> meta(n_images);
    bool far = false;
    for (uint32_t i = 0; i < n_images; ++i) {
        TrainImage& m = meta[i];
        for (int k = 0; k < 12; ++k) m.M[k] = cams[i].matrix[k];
        m.fx = cams[i].focal_px[0];
        m.fy = cams[i].focal_px[1];
        m.cx = cams[i].screen_center[0];
        m.cy = cams[i].screen_center[1];
        m.frame = frames[i];
        m.pad[0] = m.pad[1] = m.pad[2] = 0;
        const float origin[3] = {m.M[3], m.M[7], m.M[11]};
        far |= far_camera(origin, ctx->cfg.dt);
    }
    INSTA_HIP(hipMemcpyAsync(ts->images, rgba, px * sizeof(float4), hipMemcpyDeviceToDevice, stream));
    INSTA_HIP(hipMemcpyAsync(ts->meta, meta.data(), n_images * sizeof(TrainImage), hipMemcpyHostToDevice, stream));
    INSTA_HIP(hipStreamSynchronize(stream));  // `meta` is pageable host memory
    ts->frames.assign(frames, frames + n_images);
    ts->n_images = n_images;
    ts->far = far;
    ts->width = width;
    ts->height = height;
    ts->rays_total = 0;
    return INSTA_OK;
}

insta_status set_training_supervision(insta_ctx* ctx, const uint8_t* seg, const float* depth, hipStream_t stream) {
    TrainState* ts = ctx->train;
    const size_t px = (size_t)ts->n_images * ts->width * ts->height;
    dev_free(ts->seg);
    dev_free(ts->depth);
    if ((seg && !train_alloc(ts->seg, px)) || (depth && !train_alloc(ts->depth, px * sizeof(float)))) {
        dev_free(ts->seg);
        dev_free(ts->depth);
        set_error("training supervision allocation failed");
        return INSTA_ERR_OOM;
    }
    if (seg) INSTA_HIP(hipMemcpyAsync(ts->seg, seg, px, hipMemcpyDeviceToDevice, stream));
    if (depth) INSTA_HIP(hipMemcpyAsync(ts->depth, depth, px * sizeof(float), hipMemcpyDeviceToDevice, stream));
    return INSTA_OK;
}

insta_status train_step(insta_ctx* ctx, const insta_train_config& tc, insta_train_stats* stats, hipStream_t stream) {
    TrainState* ts = ctx->train;
    ts->net_n = 0;  // the step reuses the network plugin's activation buffers
    const uint32_t n_rays = tc.n_rays ? tc.n_rays : ts->rays_per_batch;
    insta_status st = check_train_workspace(ts, n_rays, tc.max_samples, tc.target_samples, "train_step");
    if (st != INSTA_OK) return st;
    // the step evaluates its samples with the training weights (under an Ema
    // optimizer the inference network holds the average between steps)
    const float* inference_src = net_params(ctx);
    if (inference_src != ctx->d_params) {
        ctx->net_src = nullptr;
        st = prepare_network(ctx, stream);
        if (st != INSTA_OK) return st;
    }
    const uint64_t np = ctx->layout.n_params;
    // the marched-sample cap is the step's (a larger reservation changes nothing)
    const uint32_t cap = tc.max_samples;
    hipLaunchKernelGGL(train_clear_kernel, dim3(1), dim3(64), 0, stream, ts->counters, cap);
    INSTA_HIP(hipGetLastError());

    Pcg32 rng = Pcg32::seeded(tc.seed);
    rng.advance(ts->rays_total * kRaySeedStride);
    RayArgs ra{};
    ra.box.G = ctx->cfg.grid_size;
    ra.box.dt = ctx->cfg.dt;
    ra.box.max_steps = ctx->cfg.max_steps;
    for (int k = 0; k < 3; ++k) {
        ra.box.lo[k] = ctx->render_lo[k];
        ra.box.hi[k] = ctx->render_hi[k];
    }
    ra.meta = ts->meta;
    ra.grids_lin = ctx->d_grids_lin;
    ra.grid_bytes = (size_t)ctx->cfg.grid_size * ctx->cfg.grid_size * ctx->cfg.grid_size / 8;
    ra.n_images = ts->n_images;
    ra.width = ts->width;
    ra.height = ts->height;
    ra.max_samples = cap;
    ra.fixed_slot = tc.occupancy_slot;
    hipLaunchKernelGGL(ts->far ? train_rays_kernel<true> : train_rays_kernel<false>,
                       dim3((n_rays + kRayThreads - 1) / kRayThreads), dim3(kRayThreads), 0, stream, ra, n_rays, ts->rays_total, rng, ts->ray_d, ts->ray_o, ts->ray_frame, ts->ray_img, ts->ray_pix, ts->ray_src, ts->ray_base,
                       ts->ray_cnt, ts->t_buf, ts->ray_T, ts->ray_alive, ts->counters);
    INSTA_HIP(hipGetLastError());
    hipLaunchKernelGGL(train_count_kernel, dim3(1), dim3(64), 0, stream, ts->counters);
    // deform and evaluate the marched samples window by window, only while
    // their rays are still alive
    const dim3 rgrid((n_rays + kRayThreads - 1) / kRayThreads);
    for (uint32_t w = 0; w < kRounds; ++w) {
        const uint32_t lo = kWin[w], hi = kWin[w + 1];
        hipLaunchKernelGGL(train_gather_kernel, rgrid, dim3(kRayThreads), 0, stream, lo, hi, ts->ray_base, ts->ray_cnt,
                           ts->ray_alive, ts->ray_gbase, ts->ray_o, ts->ray_d, ts->ray_src, ts->t_buf, n_rays,
                           ts->r_pos, ts->counters, kTRound0 + w);
        INSTA_HIP(hipGetLastError());
        const uint32_t* n_round = ts->counters + kTRound0 + w;
        // the deformation kernels stride over the round's samples: a grid for
        // at most the window's samples and 2^20 threads, not for the sample
        // capacity (empty workgroups of a 2^24-thread grid cost ~15 us a launch)
        const uint32_t round_grid =
            (uint32_t)std::min<uint64_t>(std::min<uint64_t>(cap, (uint64_t)n_rays * (hi - lo)), 1u << 20);
        st = launch_deform_samples(ctx, -1, ts->ray_frame, n_round, round_grid, ts->r_pos, ts->ray_d, ts->s_hit,
                                   ts->r_cpos, ts->r_cdir, ctx->d_misses, ts->r_out, ts->counters + kTQueue, stream);
        if (st != INSTA_OK) return st;
        st = launch_network_samples(ctx, n_round, cap, ts->r_cpos, ts->r_cdir, ts->r_out, stream);
        if (st != INSTA_OK) return st;
        hipLaunchKernelGGL(train_round_kernel, rgrid, dim3(kRayThreads), 0, stream, lo, hi, ctx->cfg.density_logit_bias,
                           ctx->cfg.dt, ts->ray_base, ts->ray_cnt, ts->ray_alive, ts->ray_gbase, ts->ray_T,
                           ts->r_cpos, ts->r_cdir, ts->r_out, ts->s_cpos, ts->s_cdir, ts->s_out, ts->counters);
        INSTA_HIP(hipGetLastError());
    }
    LossArgs la;
    la.images = ts->images;
    la.seg = ts->seg;
    la.depth = ts->depth;
    la.seg_weight = tc.seg_weight;
    la.depth_weight = tc.depth_weight;
    la.width = ts->width;
    la.height = ts->height;
    la.dt = ctx->cfg.dt;
    la.density_bias = ctx->cfg.density_logit_bias;
    la.loss_scale_per_ray = tc.loss_scale / (float)n_rays;
    la.inv_rays = 1.0f / (float)n_rays;
    hipLaunchKernelGGL(train_loss_kernel, rgrid, dim3(kRayThreads), 0, stream, la, rng, ts->ray_src,
                       ts->ray_img, ts->ray_pix, ts->ray_base, ts->ray_cnt, ts->ray_o, ts->ray_d, ts->t_buf,
                       n_rays, ts->s_out,
                       ts->c_idx, ts->c_dout,
                       ts->compact_cap, ts->counters);
    INSTA_HIP(hipGetLastError());
    hipLaunchKernelGGL(train_compact_count_kernel, dim3(1), dim3(64), 0, stream, ts->counters, ts->compact_cap);
    const bool x16 = ctx->cfg.n_extra_dims != 0;
    st = ctx->cfg.n_levels == 8 ? (x16 ? launch_train_forward<8, 16>(ctx, ts, stream) : launch_train_forward<8, 0>(ctx, ts, stream))
                                : (x16 ? launch_train_forward<16, 16>(ctx, ts, stream) : launch_train_forward<16, 0>(ctx, ts, stream));
    if (st != INSTA_OK) return st;
    st = ctx->cfg.n_levels == 8
             ? (x16 ? launch_train_backward<8, 16>(ctx, ts, tc, stream) : launch_train_backward<8, 0>(ctx, ts, tc, stream))
             : (x16 ? launch_train_backward<16, 16>(ctx, ts, tc, stream) : launch_train_backward<16, 0>(ctx, ts, tc, stream));
    if (st != INSTA_OK) return st;
    const uint32_t t = ts->adam_step + (tc.apply_update ? 1u : 0u);
    const float bc1 = tc.apply_update ? 1.0f - (float)std::pow((double)tc.beta1, (double)t) : 1.0f;
    const float bc2 = tc.apply_update ? 1.0f - (float)std::pow((double)tc.beta2, (double)t) : 1.0f;
    hipLaunchKernelGGL(adam_kernel, dim3(2048), dim3(256), 0, stream, ctx->d_params, ts->grad, ts->adam_m, ts->adam_v,
                       np, 1.0f / tc.loss_scale, tc.learning_rate, tc.beta1, tc.beta2, tc.epsilon, bc1, bc2,
                       tc.l2_reg, tc.apply_update);
    INSTA_HIP(hipGetLastError());
    if (tc.apply_update) {
        if (tc.ema_decay > 0.0f) {
            // the weight average renders use; training keeps its own weights
            ts->ema_step += 1;
            const float debias = (float)(1.0 / (1.0 - std::pow((double)tc.ema_decay, (double)ts->ema_step)));
            hipLaunchKernelGGL(ema_kernel, dim3(2048), dim3(256), 0, stream, ctx->d_params, ts->ema, ts->ema_infer,
                               np, tc.ema_decay, debias, ts->ema_step == 1 ? 1u : 0u);
            INSTA_HIP(hipGetLastError());
            ctx->net_src = ts->ema_infer;
        } else {
            ts->ema_step = 0;
            ctx->net_src = nullptr;
        }
        st = prepare_network(ctx, stream);
        if (st != INSTA_OK) return st;
    } else if (inference_src != net_params(ctx)) {
        ctx->net_src = inference_src == ctx->d_params ? nullptr : inference_src;  // back to what renders used
        st = prepare_network(ctx, stream);
        if (st != INSTA_OK) return st;
    }
    INSTA_HIP(hipMemcpyAsync(ts->h_counters, ts->counters, kTCounters * sizeof(uint32_t), hipMemcpyDeviceToHost,
                             stream));
    INSTA_HIP(hipStreamSynchronize(stream));
    const uint32_t* hc = ts->h_counters;
    if (stats) {
        stats->n_rays = n_rays;
        stats->n_rays_used = hc[kTRays];
        stats->n_samples = hc[kTValid];
        stats->n_samples_used = hc[kTUsed];
        stats->n_samples_evaluated = 0;
        for (uint32_t w = 0; w < kRounds; ++w) stats->n_samples_evaluated += hc[kTRound0 + w];
        float loss;
        std::memcpy(&loss, &hc[kTLoss], 4);
        stats->loss = loss;
    }
    ts->rays_total += n_rays;
    ts->have_grad = true;
    if (tc.apply_update) {
        ts->adam_step = t;
        ts->training_step += 1;
    }
    if (stats) {
        stats->step = ts->training_step;
        stats->adam_step = ts->adam_step;
    }
    // adaptive ray count (testbed_nerf.cu:3402-3410): rays * target /
    // compacted batch, rounded up to a multiple of 128, at most 2^18 rays
    const uint32_t measured = std::max(std::min(hc[kTUsed], ts->compact_cap), 1u);
    double next = (double)n_rays * tc.target_samples / measured;
    next = std::min(std::max(next, 128.0), (double)(1u << 18));
    ts->rays_per_batch = ((uint32_t)next + 127u) & ~127u;
    return INSTA_OK;
}

void reset_inference_average(insta_ctx* ctx) {
    if (ctx->train) ctx->train->ema_step = 0;
    ctx->net_src = nullptr;
}

bool train_has_gradients(const insta_ctx* ctx) { return ctx->train && ctx->train->have_grad; }
bool train_has_set(const insta_ctx* ctx) { return ctx->train && ctx->train->n_images > 0; }
const std::vector<int32_t>& train_frames(const insta_ctx* ctx) { return ctx->train->frames; }
TrainSetView train_set_view(const insta_ctx* ctx) {
    const TrainState* ts = ctx->train;
    if (!ts) return TrainSetView{};
    return TrainSetView{ts->meta, ts->n_images, ts->width, ts->height};
}
uint32_t train_step_count(const insta_ctx* ctx) { return ctx->train ? ctx->train->training_step : 0u; }

insta_status get_gradients(insta_ctx* ctx, float* out, hipStream_t stream) {
    INSTA_HIP(hipMemcpyAsync(out, ctx->train->grad, ctx->layout.n_params * sizeof(float), hipMemcpyDeviceToDevice,
                             stream));
    return INSTA_OK;
}

insta_status train_export(insta_ctx* ctx, bool with_optimizer, TrainSnapshot& out, hipStream_t stream) {
    out = TrainSnapshot{};
    TrainState* ts = ctx->train;
    if (!ts) return INSTA_OK;
    out.present = true;
    out.step = ts->training_step;
    out.adam_step = ts->adam_step;
    out.rays_per_batch = ts->rays_per_batch;
    out.rays_total = ts->rays_total;
    if (ts->n_images && ts->meta) {
        std::vector<TrainImage> meta(ts->n_images);
        INSTA_HIP(hipMemcpyAsync(meta.data(), ts->meta, meta.size() * sizeof(TrainImage), hipMemcpyDeviceToHost,
                                 stream));
        INSTA_HIP(hipStreamSynchronize(stream));
        out.n_images = ts->n_images;
        out.width = ts->width;
        out.height = ts->height;
        out.cams.resize((size_t)ts->n_images * 16);
        for (uint32_t i = 0; i < ts->n_images; ++i) {
            float* c = out.cams.data() + (size_t)i * 16;
            std::memcpy(c, meta[i].M, 12 * sizeof(float));
            c[12] = meta[i].fx;
            c[13] = meta[i].fy;
            c[14] = meta[i].cx;
            c[15] = meta[i].cy;
        }
    }
    if (with_optimizer) {
        const uint64_t np = ctx->layout.n_params;
        out.m.resize(np);
        out.v.resize(np);
        INSTA_HIP(hipMemcpyAsync(out.m.data(), ts->adam_m, np * sizeof(float), hipMemcpyDeviceToHost, stream));
        INSTA_HIP(hipMemcpyAsync(out.v.data(), ts->adam_v, np * sizeof(float), hipMemcpyDeviceToHost, stream));
        INSTA_HIP(hipStreamSynchronize(stream));
    }
    return INSTA_OK;
}

insta_status train_import(insta_ctx* ctx, const TrainSnapshot& in, hipStream_t stream) {
    insta_status st = ensure_train_state(ctx, stream);
    if (st != INSTA_OK) return st;
    TrainState* ts = ctx->train;
    const uint64_t np = ctx->layout.n_params;
    // Testbed::load_snapshot resumes at training_step + 1 (testbed.cu:3011)
    ts->training_step = in.step + 1;
    ts->rays_per_batch = in.rays_per_batch;
    ts->rays_total = in.rays_total;
    if (in.m.size() == np && in.v.size() == np) {
        INSTA_HIP(hipMemcpyAsync(ts->adam_m, in.m.data(), np * sizeof(float), hipMemcpyHostToDevice, stream));
        INSTA_HIP(hipMemcpyAsync(ts->adam_v, in.v.data(), np * sizeof(float), hipMemcpyHostToDevice, stream));
        INSTA_HIP(hipStreamSynchronize(stream));  // pageable sources
        ts->adam_step = in.adam_step;
    } else {
        INSTA_HIP(hipMemsetAsync(ts->adam_m, 0, np * sizeof(float), stream));
        INSTA_HIP(hipMemsetAsync(ts->adam_v, 0, np * sizeof(float), stream));
        ts->adam_step = 0;  // fresh moments restart the bias correction
    }
    return INSTA_OK;
}

insta_status reset_optimizer(insta_ctx* ctx, hipStream_t stream) {
    TrainState* ts = ctx->train;
    const uint64_t np = ctx->layout.n_params;
    // stream-ordered fill kernels: no device-wide stall, capturable
    hipLaunchKernelGGL(fill_zero_kernel, dim3(1024), dim3(256), 0, stream, reinterpret_cast<uint32_t*>(ts->adam_m), np);
    hipLaunchKernelGGL(fill_zero_kernel, dim3(1024), dim3(256), 0, stream, reinterpret_cast<uint32_t*>(ts->adam_v), np);
    INSTA_HIP(hipGetLastError());
    ts->adam_step = 0;
    return INSTA_OK;
}

// ---- NerfNetwork plugin entry points --------------------------------------
namespace {
insta_status ensure_net_workspace(insta_ctx* ctx, uint32_t n, hipStream_t) {
    if (!ctx->train) {
        set_error("network plugin: no workspace: reserve one with insta_reserve (train_samples, train_batch)");
        return INSTA_ERR_STATE;
    }
    TrainState* ts = ctx->train;
    insta_status st = check_train_workspace(ts, 0, n, n, "network plugin");
    if (st != INSTA_OK) return st;
    if (ctx->cfg.n_extra_dims && ts->net_extra_cap < n) {
        set_error("network plugin: extra-dims workspace smaller than the batch: reserve with insta_reserve");
        return INSTA_ERR_STATE;
    }
    return INSTA_OK;
}
}  // namespace

insta_status reserve_training(insta_ctx* ctx, uint32_t rays, uint32_t samples, uint32_t batch, hipStream_t stream) {
    insta_status st = ensure_train_state(ctx, stream);
    if (st != INSTA_OK) return st;
    TrainState* ts = ctx->train;
    st = grow_train_workspace(ctx, ts, rays, samples, batch);
    if (st != INSTA_OK) return st;
    const uint32_t X = ctx->cfg.n_extra_dims;
    if (X && ts->net_extra_cap < ts->compact_cap) {
        dev_free(ts->net_extra);
        ts->net_extra_cap = 0;
        if (hipMalloc(reinterpret_cast<void**>(&ts->net_extra), (size_t)ts->compact_cap * X * sizeof(float)) !=
            hipSuccess) {
            set_error("network plugin workspace allocation failed");
            return INSTA_ERR_OOM;
        }
        ts->net_extra_cap = ts->compact_cap;
    }
    return INSTA_OK;
}

insta_status network_forward(insta_ctx* ctx, const float* coords, uint32_t n, uint32_t stride, float* out,
                             hipStream_t stream) {
    insta_status st = ensure_net_workspace(ctx, n, stream);
    if (st != INSTA_OK) return st;
    TrainState* ts = ctx->train;
    const uint32_t X = ctx->cfg.n_extra_dims;
    hipLaunchKernelGGL(net_prepare_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, coords, n, stride, X, ts->s_cpos,
                       ts->s_cdir, ts->c_idx, ts->net_extra, ts->counters);
    INSTA_HIP(hipGetLastError());
    float4* o = reinterpret_cast<float4*>(out);
    const bool x16 = X != 0;
    st = ctx->cfg.n_levels == 8 ? (x16 ? launch_net_forward<8, 16>(ctx, ts, o, stream) : launch_net_forward<8, 0>(ctx, ts, o, stream))
                                : (x16 ? launch_net_forward<16, 16>(ctx, ts, o, stream) : launch_net_forward<16, 0>(ctx, ts, o, stream));
    if (st != INSTA_OK) return st;
    ts->net_n = n;
    return INSTA_OK;
}

uint32_t network_forward_batch(const insta_ctx* ctx) { return ctx->train ? ctx->train->net_n : 0u; }

insta_status network_backward(insta_ctx* ctx, uint32_t n, uint32_t stride, const float* dL_dout, float* grad_out,
                              bool accumulate, float* dL_dinput, hipStream_t stream) {
    TrainState* ts = ctx->train;
    const uint64_t np = ctx->layout.n_params;
    INSTA_HIP(hipMemcpyAsync(ts->c_dout, dL_dout, (size_t)n * sizeof(float4), hipMemcpyDeviceToDevice, stream));
    insta_train_config tc{};
    tc.grid_grad_fp16 = 0;
    const bool x16 = ctx->cfg.n_extra_dims != 0;
    insta_status st =
        ctx->cfg.n_levels == 8
            ? (x16 ? launch_train_backward<8, 16>(ctx, ts, tc, stream) : launch_train_backward<8, 0>(ctx, ts, tc, stream))
            : (x16 ? launch_train_backward<16, 16>(ctx, ts, tc, stream) : launch_train_backward<16, 0>(ctx, ts, tc, stream));
    if (st != INSTA_OK) return st;
    hipLaunchKernelGGL(net_grad_out_kernel, dim3(1024), dim3(256), 0, stream, ts->grad, grad_out, np,
                       accumulate ? 1u : 0u);
    INSTA_HIP(hipGetLastError());
    if (dL_dinput) {
        st = ctx->cfg.n_levels == 8
                 ? (x16 ? launch_net_input_grad<8, 16>(ctx, ts, n, dL_dinput, stride, stream)
                        : launch_net_input_grad<8, 0>(ctx, ts, n, dL_dinput, stride, stream))
                 : (x16 ? launch_net_input_grad<16, 16>(ctx, ts, n, dL_dinput, stride, stream)
                        : launch_net_input_grad<16, 0>(ctx, ts, n, dL_dinput, stride, stream));
        if (st != INSTA_OK) return st;
    }
    return INSTA_OK;
}

}  // namespace insta
