// density.hip -- density-grid update of training: the occupancy grid as an
// EMA of the network's optical thickness (Testbed::update_density_grid_nerf,
// instant-ngp/src/testbed_nerf.cu:2774-2861, one cascade, one step):
//   samples   generate_grid_samples_nerf_nonuniform (487-516): n_uniform
//             cells at any density and n_nonuniform cells above 0.01 (up to
//             10 probes of a multiplicative-hash cell sequence), a random
//             position inside each cell; both sets read the same PCG32 state,
//             which then advances by 2^32 (pcg32's default jump)
//   order     counting sort of the samples by (posed frame, Morton cell): the
//             cells come from a multiplicative sequence and the frames from a
//             random stream, so in drawing order a wave's 64 nearest-triangle
//             walks would share nothing
//   warp      each position to canonical space through its random posed frame
//             (warp_random_samples, src/core.cu:528-579)
//   splat     density MLP at the canonical position (extra dims all 1.0, as
//             extract_expressions_random writes, nerf_network.h:107-127),
//             optical thickness
//             exp(logit + bias) * dt, atomicMax on the float bits into the
//             cell (splat_grid_samples_nerf_max_nearest_neighbor, 518-534)
//   ema       grid = max(grid * decay, new) unless negative
//             (ema_grid_samples_nerf, 554-577)
//   bitfield  cell occupied when grid > min(0.01, mean of max(grid, 0))
//             (update_density_grid_mean_and_bitfield + grid_to_bitfield,
//             2863-2878, 585-609), written into an occupancy slot
// The mean is a two-stage fixed-order reduction, so the bitfield is a
// deterministic function of the grid.
#include <algorithm>

#include "context.hpp"
#include "encoding.hpp"

namespace insta {

struct DensityGridState {
    float* grid = nullptr;      // [G^3] Morton order
    float* tmp = nullptr;       // [G^3] this update's splats
    float4* rec = nullptr;      // [cap] drawn samples: position, posed frame (bits)
    uint32_t* idx = nullptr;    // [cap] their cells
    float4* srec = nullptr;     // [cap] the samples by (frame, cell)
    uint32_t* sidx = nullptr;   // [cap]
    uint32_t* bins = nullptr;   // [kMaxBins] samples per bin, then each bin's next slot
    uint32_t* bin_sums = nullptr;  // [kMaxBins / kScanBins]
    float* partial = nullptr;   // [G^3 / kReduce] block sums
    float* mean = nullptr;      // [1]
    float* h_mean = nullptr;    // pinned mirror
    uint32_t cap = 0;
    uint32_t step = 0;
    uint32_t marked_n = 0;      // training images at the last untrained-cell marking
    Pcg32 rng{0, 0};
};

namespace {

constexpr uint32_t kThreads = 256;
constexpr uint32_t kReduce = 1024;    // cells per first-stage block
// Sort bins: at most 2^20 (and about one per sample), the frames times equal
// runs of the Morton order.  At 2^20 samples of three frames a bin is a box
// of 2 x 2 x 2 cells of the 128^3 grid.
constexpr uint32_t kMaxBins = 1u << 20;
constexpr uint32_t kScanBins = 1024;  // bins per workgroup of the scan
constexpr float kMinOpticalThickness = 0.01f;  // NERF_MIN_OPTICAL_THICKNESS (testbed_nerf.cu:63)

__global__ void dg_fill_kernel(float* p, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

// mark_untrained_density_grid (testbed_nerf.cu:391-431): -1 for a cell that
// no training camera sees (centre widened by the half-diagonal against each
// camera's centred frustum), 0 for a seen cell that was untrained (or always
// with `clear`); one thread per cell, Morton order, one cascade
__global__ void dg_mark_kernel(float* __restrict__ grid, uint32_t G, const TrainImage* __restrict__ meta,
                               uint32_t n_images, float half_x, float half_y, uint32_t clear) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= G * G * G) return;
    const float x = (float)compact3(i), y = (float)compact3(i >> 1), z = (float)compact3(i >> 2);
    const float px = ((x + 0.5f) / (float)G - 0.5f) * 1.0f + 0.5f;
    const float py = ((y + 0.5f) / (float)G - 0.5f) * 1.0f + 0.5f;
    const float pz = ((z + 0.5f) / (float)G - 0.5f) * 1.0f + 0.5f;
    const float radius = 0.5f * 1.73205080757f * 1.0f / (float)G;
    bool seen = false;
    for (uint32_t j = 0; j < n_images && !seen; ++j) {
        const TrainImage& c = meta[j];
        const float lx = px - c.M[3], ly = py - c.M[7], lz = pz - c.M[11];
        const float cx = lx * c.M[0] + ly * c.M[4] + lz * c.M[8];
        const float cy = lx * c.M[1] + ly * c.M[5] + lz * c.M[9];
        const float cz = lx * c.M[2] + ly * c.M[6] + lz * c.M[10];
        seen = cz > 0.0f && fabsf(cx) - radius < cz / c.fx * half_x && fabsf(cy) - radius < cz / c.fy * half_y;
    }
    const float g = grid[i];
    if (clear || (g < 0.0f) != !seen) grid[i] = seen ? 0.0f : -1.0f;
}

// The sample's posed frame is the warp's draw (warp_random_samples): the
// stream `frames` advanced by (first + i) * n_meshes gives
// floor(u * n_meshes), so the last frame is never chosen.
__global__ void dg_samples_kernel(uint32_t n, uint32_t step, float thresh, uint32_t G, const float* __restrict__ grid,
                                  Pcg32 rng, Pcg32 frames, uint32_t first, uint32_t n_meshes, uint32_t bin_shift,
                                  uint32_t frame_bins, float4* __restrict__ rec, uint32_t* __restrict__ idx_out,
                                  uint32_t* __restrict__ bins) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t cells = G * G * G;
    rng.advance((uint64_t)i * 4u);
    (void)rng.next_float();  // cascade choice; one cascade here
    uint32_t idx = 0;
    for (uint32_t j = 0; j < 10; ++j) {
        idx = ((i + step * n) * 56924617u + j * 19349663u + 96925573u) % cells;
        if (grid[idx] > thresh) break;
    }
    const uint32_t x = compact3(idx), y = compact3(idx >> 1), z = compact3(idx >> 2);
    const float rx = rng.next_float(), ry = rng.next_float(), rz = rng.next_float();
    const float g = (float)G;
    frames.advance((uint64_t)(first + i) * n_meshes);
    const uint32_t frame = (uint32_t)(frames.next_float() * (float)n_meshes);
    rec[first + i] = make_float4((((float)x + rx) / g - 0.5f) * 1.0f + 0.5f, (((float)y + ry) / g - 0.5f) * 1.0f + 0.5f,
                                 (((float)z + rz) / g - 0.5f) * 1.0f + 0.5f, __uint_as_float(frame));
    idx_out[first + i] = idx;
    atomicAdd(bins + frame * frame_bins + (idx >> bin_shift), 1u);
}

// sum over the workgroup's kScanBins threads' values, in every thread
__device__ inline uint32_t block_sum(uint32_t v, uint32_t* s) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63u) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    uint32_t t = 0;
    for (uint32_t w = 0; w < kScanBins / 64; ++w) t += s[w];
    __syncthreads();
    return t;
}

__global__ __launch_bounds__(kScanBins) void dg_bin_sums_kernel(const uint32_t* __restrict__ bins, uint32_t n_bins,
                                                                uint32_t* __restrict__ sums) {
    __shared__ uint32_t s[kScanBins / 64];
    const uint32_t i = blockIdx.x * kScanBins + threadIdx.x;
    const uint32_t t = block_sum(i < n_bins ? bins[i] : 0u, s);
    if (threadIdx.x == 0) sums[blockIdx.x] = t;
}

// bins[i] <- samples in the bins before i (at most kScanBins workgroups)
__global__ __launch_bounds__(kScanBins) void dg_bin_scan_kernel(uint32_t* __restrict__ bins, uint32_t n_bins,
                                                                const uint32_t* __restrict__ sums) {
    __shared__ uint32_t s[kScanBins / 64];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const uint32_t i = blockIdx.x * kScanBins + t;
    uint32_t run = block_sum(t < blockIdx.x ? sums[t] : 0u, s);
    const uint32_t v = i < n_bins ? bins[i] : 0u;
    uint32_t incl = v;
#pragma unroll
    for (uint32_t o = 1; o < 64u; o <<= 1) {
        const uint32_t up = __shfl_up(incl, o);
        if (lane >= o) incl += up;
    }
    if (lane == 63u) s[wave] = incl;
    __syncthreads();
    for (uint32_t w = 0; w < wave; ++w) run += s[w];
    if (i < n_bins) bins[i] = run + incl - v;
}

// the drawn samples into their bins (their order inside a bin varies; every
// use of a sample is its own)
__global__ void dg_order_kernel(uint32_t n, uint32_t bin_shift, uint32_t frame_bins, const float4* __restrict__ rec,
                                const uint32_t* __restrict__ idx, uint32_t* __restrict__ bins,
                                float4* __restrict__ srec, uint32_t* __restrict__ sidx) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 r = rec[i];
    const uint32_t c = idx[i];
    const uint32_t slot = atomicAdd(bins + __float_as_uint(r.w) * frame_bins + (c >> bin_shift), 1u);
    srec[slot] = r;
    sidx[slot] = c;
}

// Density logit (output 0 of the density MLP) at canonical positions, optical
// thickness max-splatted into the sample's cell.  The hidden layer is a
// contraction over the batch, so it runs on v_mfma_f32_16x16x4f32: phase A,
// one thread per sample, encodes into LDS; phase B, a wave's 64 samples in
// four blocks of 16 columns, weights as A operands held in registers (lane l:
// row l % 16, k l / 16) and the extra dims' columns (all 1.0) as the starting
// accumulator; the one output row needed is a dot product on the vector ALUs
// (16 terms per lane, then the four lane groups), not a padded MFMA tile.
// Bound by the table gathers of phase A: 1,048,576 samples at L = 16, T =
// 2^19 take 547 us; with one thread per sample running the MLP as FMA
// chains on scalar weights, and the samples in drawing order, 894 us.
typedef float dg_f4 __attribute__((ext_vector_type(4)));
constexpr uint32_t kSplatTile = 256;
template <int L, int X>
__global__ __launch_bounds__(kSplatTile) void dg_splat_kernel(const float* __restrict__ params,
                                                              const float* __restrict__ table, GridParams gp,
                                                              const float4* __restrict__ pos,
                                                              const uint32_t* __restrict__ idx, uint32_t n, float dt,
                                                              float bias, float* __restrict__ tmp) {
    constexpr int E = 2 * L, DIN = E + X, KB = E / 4, S = E + 1;
    constexpr int W = 64;
    __shared__ float s_x[kSplatTile * S];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t m = lane & 15u, g = lane >> 4;
    const uint32_t base = blockIdx.x * kSplatTile;
    {
        const uint32_t i = min(base + tid, n - 1u);  // lanes past the end repeat the last sample
        const V3 x = xyz(pos[i]);
        float* row = s_x + tid * S;
#pragma unroll 2
        for (int l = 0; l < L; ++l) {
            float f[2];
            encode_level<2>(table, gp, (uint32_t)l, x, f);
            row[2 * l] = f[0];
            row[2 * l + 1] = f[1];
        }
    }
    float a[4][KB];
    dg_f4 first[4], w1[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) a[t][kb] = params[(16 * t + m) * DIN + 4 * kb + g];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t r = 16 * t + 4 * g + q;
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < X; ++e) sum = sum + params[r * DIN + E + e];
            first[t][q] = sum;
            w1[t][q] = params[W * DIN + r];
        }
    }
    __syncthreads();
    for (uint32_t nb = 0; nb < 4; ++nb) {
        const uint32_t s = wave * 64 + nb * 16 + m;  // sample (column) of this lane
        const float* xr = s_x + s * S;
        float logit = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            dg_f4 h = first[t];
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
                h = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][kb], xr[4 * kb + g], h, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) logit = __builtin_fmaf(w1[t][q], fmaxf(h[q], 0.0f), logit);
        }
        logit += __shfl_xor(logit, 16);
        logit += __shfl_xor(logit, 32);
        if (g == 0 && base + s < n) {
            const float thickness = expf(logit + bias) * dt;
            atomicMax(reinterpret_cast<uint32_t*>(tmp) + idx[base + s], __float_as_uint(thickness));
        }
    }
}

// NerfNetwork::density (nerf_network.h:385-414): the density MLP's 16
// outputs at canonical positions, extra dims 1.0 (extract_expressions_random
// writes 1.0, nerf_network.h:107-127); out [n][16], output 0 the density logit
template <int L, int X>
__global__ __launch_bounds__(128) void density_outputs_kernel(const float* __restrict__ params,
                                                              const float* __restrict__ table, GridParams gp,
                                                              const float* __restrict__ pos, uint32_t n,
                                                              float* __restrict__ out) {
    constexpr int E = 2 * L + X;
    constexpr int W = 64;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const V3 x = v3(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]);
    float enc[E];
#pragma unroll
    for (int l = 0; l < L; ++l) encode_level<2>(table, gp, (uint32_t)l, x, enc + 2 * l);
#pragma unroll
    for (int e = 2 * L; e < E; ++e) enc[e] = 1.0f;
    float h[W];
    dense<E, W, true>(params, enc, h);
    float o[16];
    dense<W, 16, false>(params + W * E, h, o);
#pragma unroll
    for (int k = 0; k < 16; ++k) out[(size_t)i * 16 + k] = o[k];
}

__global__ void dg_ema_kernel(float* __restrict__ grid, const float* __restrict__ tmp, float decay, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float prev = grid[i];
    grid[i] = prev < 0.0f ? prev : fmaxf(prev * decay, tmp[i]);
}

// stage 1: block b sums max(grid, 0) / n over cells [b*kReduce, (b+1)*kReduce)
__global__ __launch_bounds__(kThreads) void dg_reduce_kernel(const float* __restrict__ grid, uint32_t n,
                                                              float* __restrict__ partial) {
    __shared__ float s[kThreads];
    const uint32_t b = blockIdx.x, t = threadIdx.x;
    const float inv = 1.0f / (float)n;
    float acc = 0.0f;
    for (uint32_t k = 0; k < kReduce / kThreads; ++k) {
        const uint32_t i = b * kReduce + k * kThreads + t;
        if (i < n) acc += fmaxf(grid[i], 0.0f) * inv;
    }
    s[t] = acc;
    __syncthreads();
    for (uint32_t o = kThreads / 2; o > 0; o >>= 1) {
        if (t < o) s[t] += s[t + o];
        __syncthreads();
    }
    if (t == 0) partial[b] = s[0];
}

// stage 2: one block sums the partials in a fixed order
__global__ __launch_bounds__(kThreads) void dg_mean_kernel(const float* __restrict__ partial, uint32_t nb,
                                                            float* __restrict__ mean) {
    __shared__ float s[kThreads];
    const uint32_t t = threadIdx.x;
    float acc = 0.0f;
    for (uint32_t i = t; i < nb; i += kThreads) acc += partial[i];
    s[t] = acc;
    __syncthreads();
    for (uint32_t o = kThreads / 2; o > 0; o >>= 1) {
        if (t < o) s[t] += s[t + o];
        __syncthreads();
    }
    if (t == 0) mean[0] = s[0];
}

__global__ void dg_bitfield_kernel(const float* __restrict__ grid, const float* __restrict__ mean,
                                   uint8_t* __restrict__ bits, uint32_t n_bytes) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_bytes) return;
    const float thresh = fminf(kMinOpticalThickness, mean[0]);
    uint32_t v = 0;
    for (uint32_t j = 0; j < 8; ++j) v |= grid[8 * i + j] > thresh ? (1u << j) : 0u;
    bits[i] = (uint8_t)v;
}

bool dg_alloc(void* p, size_t bytes) { return hipMalloc(reinterpret_cast<void**>(p), bytes) == hipSuccess; }

}  // namespace

void free_density_grid(insta_ctx* ctx) {
    DensityGridState* d = ctx->density;
    if (!d) return;
    dev_free(d->grid); dev_free(d->tmp); dev_free(d->partial); dev_free(d->mean);
    dev_free(d->rec); dev_free(d->idx); dev_free(d->srec); dev_free(d->sidx); dev_free(d->bins); dev_free(d->bin_sums);
    if (d->h_mean) (void)hipHostFree(d->h_mean);
    delete d;
    ctx->density = nullptr;
}

insta_status update_density_grid(insta_ctx* ctx, uint32_t slot, uint32_t n_frames, const insta_density_grid_config& c,
                                 float* grid_out, float* mean_out, hipStream_t stream) {
    const uint32_t G = ctx->cfg.grid_size, cells = G * G * G;
    const uint32_t n = c.n_uniform + c.n_nonuniform;
    if (!ctx->density) {
        DensityGridState* d = new (std::nothrow) DensityGridState();
        if (!d) {
            set_error("host allocation failed");
            return INSTA_ERR_OOM;
        }
        ctx->density = d;
        const uint32_t nb = (cells + kReduce - 1) / kReduce;
        if (!dg_alloc(&d->grid, cells * 4) || !dg_alloc(&d->tmp, cells * 4) || !dg_alloc(&d->partial, nb * 4) ||
            !dg_alloc(&d->mean, 4) ||
            hipHostMalloc(reinterpret_cast<void**>(&d->h_mean), 4, hipHostMallocDefault) != hipSuccess) {
            free_density_grid(ctx);
            set_error("density grid allocation failed");
            return INSTA_ERR_OOM;
        }
    }
    DensityGridState* d = ctx->density;
    if (n > d->cap) {
        dev_free(d->rec);
        dev_free(d->idx);
        dev_free(d->srec);
        dev_free(d->sidx);
        d->cap = 0;
        if ((!d->bins && !dg_alloc(&d->bins, kMaxBins * 4)) ||
            (!d->bin_sums && !dg_alloc(&d->bin_sums, kMaxBins / kScanBins * 4)) ||
            !dg_alloc(&d->rec, (size_t)n * 16) || !dg_alloc(&d->idx, (size_t)n * 4) ||
            !dg_alloc(&d->srec, (size_t)n * 16) || !dg_alloc(&d->sidx, (size_t)n * 4)) {
            set_error("density grid sample allocation failed");
            return INSTA_ERR_OOM;
        }
        d->cap = n;
    }
    const dim3 cgrid((cells + kThreads - 1) / kThreads), block(kThreads);
    if (d->step == 0) {
        d->rng = Pcg32::seeded(c.seed);
        hipLaunchKernelGGL(dg_fill_kernel, cgrid, block, 0, stream, d->grid, cells);
    }
    // cells no training camera sees, on the first update and whenever the
    // number of training images changed (the reference keys this to
    // training step 0, where its first update runs, testbed_nerf.cu:2795-2806)
    const TrainSetView tv = train_set_view(ctx);
    if (tv.n_images > 0 && (d->step == 0 || tv.n_images != d->marked_n)) {
        hipLaunchKernelGGL(dg_mark_kernel, cgrid, block, 0, stream, d->grid, G, tv.meta, tv.n_images,
                           (float)tv.width * 0.5f, (float)tv.height * 0.5f, d->step == 0 ? 1u : 0u);
        d->marked_n = tv.n_images;
    }
    hipLaunchKernelGGL(dg_fill_kernel, cgrid, block, 0, stream, d->tmp, cells);
    // frames for the warp: a second stream, advanced per update
    Pcg32 wr = Pcg32::seeded(c.seed ^ 0x9e3779b9u);
    wr.advance((uint64_t)d->step << 32);
    // bins: frames 0 .. n_frames - 2 (one at least) times runs of 2^bin_shift
    // Morton cells, at most kMaxBins and about one per sample
    const uint32_t n_meshes = n_frames - 1, bin_frames = std::max(n_meshes, 1u);
    uint32_t max_bins = kScanBins;
    while (max_bins < n && max_bins < kMaxBins) max_bins <<= 1;
    uint32_t bin_shift = 0;
    while (((uint64_t)bin_frames * (cells >> bin_shift)) > max_bins && (cells >> bin_shift) > 1) ++bin_shift;
    const uint32_t frame_bins = cells >> bin_shift, n_bins = bin_frames * frame_bins;
    const uint32_t scan_blocks = (n_bins + kScanBins - 1) / kScanBins;
    hipLaunchKernelGGL(dg_fill_kernel, dim3((n_bins + kThreads - 1) / kThreads), block, 0, stream,
                       reinterpret_cast<float*>(d->bins), n_bins);
    if (c.n_uniform)
        hipLaunchKernelGGL(dg_samples_kernel, dim3((c.n_uniform + kThreads - 1) / kThreads), block, 0, stream,
                           c.n_uniform, d->step, -0.01f, G, d->grid, d->rng, wr, 0u, n_meshes, bin_shift, frame_bins,
                           d->rec, d->idx, d->bins);
    if (c.n_nonuniform)
        hipLaunchKernelGGL(dg_samples_kernel, dim3((c.n_nonuniform + kThreads - 1) / kThreads), block, 0, stream,
                           c.n_nonuniform, d->step, kMinOpticalThickness, G, d->grid, d->rng, wr, c.n_uniform,
                           n_meshes, bin_shift, frame_bins, d->rec, d->idx, d->bins);
    hipLaunchKernelGGL(dg_bin_sums_kernel, dim3(scan_blocks), dim3(kScanBins), 0, stream, d->bins, n_bins, d->bin_sums);
    hipLaunchKernelGGL(dg_bin_scan_kernel, dim3(scan_blocks), dim3(kScanBins), 0, stream, d->bins, n_bins, d->bin_sums);
    hipLaunchKernelGGL(dg_order_kernel, dim3((n + kThreads - 1) / kThreads), block, 0, stream, n, bin_shift, frame_bins,
                       d->rec, d->idx, d->bins, d->srec, d->sidx);
    INSTA_HIP(hipGetLastError());
    d->rng.advance(1ull << 32);
    // the drawn records and the first bin's counter are done with: the warp's
    // queue and its length
    hipLaunchKernelGGL(dg_fill_kernel, dim3(1), block, 0, stream, reinterpret_cast<float*>(d->bins), 1u);
    insta_status st = launch_deform_records(ctx, d->srec, n, reinterpret_cast<uint2*>(d->rec), d->bins, stream);
    if (st != INSTA_OK) return st;
    const float* table = ctx->d_params + ctx->layout.n_mlp_params;
    const GridParams gp = grid_params(ctx);
    const dim3 sgrid((n + kSplatTile - 1) / kSplatTile);
#define INSTA_SPLAT(L_, X_)                                                                                     \
    hipLaunchKernelGGL((dg_splat_kernel<L_, X_>), sgrid, dim3(kSplatTile), 0, stream, ctx->d_params, table, gp, d->srec,   \
                       d->sidx, n, ctx->cfg.dt, ctx->cfg.density_logit_bias, d->tmp)
    const bool x16 = ctx->cfg.n_extra_dims != 0;
    if (ctx->cfg.n_levels == 8) {
        if (x16) INSTA_SPLAT(8, 16);
        else INSTA_SPLAT(8, 0);
    } else {
        if (x16) INSTA_SPLAT(16, 16);
        else INSTA_SPLAT(16, 0);
    }
#undef INSTA_SPLAT
    INSTA_HIP(hipGetLastError());
    hipLaunchKernelGGL(dg_ema_kernel, cgrid, block, 0, stream, d->grid, d->tmp, c.decay, cells);
    const uint32_t nb = (cells + kReduce - 1) / kReduce;
    hipLaunchKernelGGL(dg_reduce_kernel, dim3(nb), block, 0, stream, d->grid, cells, d->partial);
    hipLaunchKernelGGL(dg_mean_kernel, dim3(1), block, 0, stream, d->partial, nb, d->mean);
    hipLaunchKernelGGL(dg_bitfield_kernel, dim3((cells / 8 + kThreads - 1) / kThreads), block, 0, stream, d->grid,
                       d->mean, ctx->grid(slot), cells / 8);
    INSTA_HIP(hipGetLastError());
    st = launch_grid_linear(ctx, slot, stream);
    if (st != INSTA_OK) return st;
    if (grid_out) INSTA_HIP(hipMemcpyAsync(grid_out, d->grid, cells * 4, hipMemcpyDeviceToDevice, stream));
    if (mean_out) {
        INSTA_HIP(hipMemcpyAsync(d->h_mean, d->mean, 4, hipMemcpyDeviceToHost, stream));
        INSTA_HIP(hipStreamSynchronize(stream));
        *mean_out = *d->h_mean;
    }
    ctx->grid_built[slot] = 1;
    ++d->step;
    return INSTA_OK;
}

insta_status launch_density_outputs(insta_ctx* ctx, const float* pos, uint32_t n, float* out, hipStream_t stream) {
    if (n == 0) return INSTA_OK;
    const GridParams gp = grid_params(ctx);
    const float* table = ctx->d_params + ctx->layout.n_mlp_params;
    const dim3 grid((n + 127) / 128), block(128);
    const bool x16 = ctx->cfg.n_extra_dims == 16;
    if (ctx->cfg.n_levels == 8)
        hipLaunchKernelGGL((x16 ? density_outputs_kernel<8, 16> : density_outputs_kernel<8, 0>), grid, block, 0, stream,
                           ctx->d_params, table, gp, pos, n, out);
    else
        hipLaunchKernelGGL((x16 ? density_outputs_kernel<16, 16> : density_outputs_kernel<16, 0>), grid, block, 0,
                           stream, ctx->d_params, table, gp, pos, n, out);
    INSTA_HIP(hipGetLastError());
    return INSTA_OK;
}

insta_status density_export(insta_ctx* ctx, DensitySnapshot& out, hipStream_t stream) {
    out = DensitySnapshot{};
    DensityGridState* d = ctx->density;
    if (!d || d->step == 0) return INSTA_OK;  // never populated
    const uint32_t G = ctx->cfg.grid_size, cells = G * G * G;
    out.grid.resize(cells);
    // the grid was last written on the caller's stream: copy there (pageable
    // destination), without stalling other streams of the device
    INSTA_HIP(hipMemcpyAsync(out.grid.data(), d->grid, (size_t)cells * 4, hipMemcpyDeviceToHost, stream));
    INSTA_HIP(hipStreamSynchronize(stream));
    out.step = d->step;
    out.rng_state = d->rng.state;
    out.rng_inc = d->rng.inc;
    return INSTA_OK;
}

insta_status density_import(insta_ctx* ctx, const DensitySnapshot& in, uint32_t slot, hipStream_t stream) {
    const uint32_t G = ctx->cfg.grid_size, cells = G * G * G;
    if (in.grid.empty()) {
        if (ctx->density) ctx->density->step = 0;
        return INSTA_OK;
    }
    if (in.grid.size() != cells) {
        set_error("density grid: size does not match the context's grid");
        return INSTA_ERR_INVALID;
    }
    if (!ctx->density) {
        DensityGridState* d = new (std::nothrow) DensityGridState();
        if (!d) {
            set_error("host allocation failed");
            return INSTA_ERR_OOM;
        }
        ctx->density = d;
        const uint32_t nb = (cells + kReduce - 1) / kReduce;
        if (!dg_alloc(&d->grid, cells * 4) || !dg_alloc(&d->tmp, cells * 4) || !dg_alloc(&d->partial, nb * 4) ||
            !dg_alloc(&d->mean, 4) ||
            hipHostMalloc(reinterpret_cast<void**>(&d->h_mean), 4, hipHostMallocDefault) != hipSuccess) {
            free_density_grid(ctx);
            set_error("density grid allocation failed");
            return INSTA_ERR_OOM;
        }
    }
    DensityGridState* d = ctx->density;
    INSTA_HIP(hipMemcpyAsync(d->grid, in.grid.data(), (size_t)cells * 4, hipMemcpyHostToDevice, stream));
    d->step = in.step ? in.step : 1;
    d->rng.state = in.rng_state;
    d->rng.inc = in.rng_inc;
    // mean and bitfield as after an update (update_density_grid_mean_and_bitfield)
    const dim3 block(kThreads);
    const uint32_t nb = (cells + kReduce - 1) / kReduce;
    hipLaunchKernelGGL(dg_reduce_kernel, dim3(nb), block, 0, stream, d->grid, cells, d->partial);
    hipLaunchKernelGGL(dg_mean_kernel, dim3(1), block, 0, stream, d->partial, nb, d->mean);
    hipLaunchKernelGGL(dg_bitfield_kernel, dim3((cells / 8 + kThreads - 1) / kThreads), block, 0, stream, d->grid,
                       d->mean, ctx->grid(slot), cells / 8);
    INSTA_HIP(hipGetLastError());
    insta_status st = launch_grid_linear(ctx, slot, stream);
    if (st != INSTA_OK) return st;
    INSTA_HIP(hipStreamSynchronize(stream));  // pageable source
    ctx->grid_built[slot] = 1;
    return INSTA_OK;
}

insta_status reset_density_grid(insta_ctx* ctx) {
    if (ctx->density) ctx->density->step = 0;
    return INSTA_OK;
}

}  // namespace insta
