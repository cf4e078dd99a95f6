// march.hpp -- ray/box, occupancy-grid stepping, Sobol jitter and
// wave-aggregated list helpers shared by the render and training marches
// (instant-ngp/src/testbed_nerf.cu:186-208, 313-337, 634-686;
// random_val.cuh:159-288).
#pragma once

#include <cmath>

#include "context.hpp"

namespace insta {

struct RenderArgs {
    float M[12];
    float cx, cy, fx, fy;
    float off_x, off_y;
    uint32_t width, height, spp, G, max_steps;
    float dt, min_transmittance, density_bias;
    float lo[3], hi[3];
    const uint8_t* grid;
};

// ---- Sobol / Owen scrambling (random_val.cuh:159-288) ---------------------
INSTA_DEV uint32_t lk_permutation(uint32_t x, uint32_t seed) {
    x += seed;
    x ^= x * 0x6c50b47cu;
    x ^= x * 0xb82f1e52u;
    x ^= x * 0xc7afe638u;
    x ^= x * 0x8d22f6e6u;
    return x;
}
INSTA_DEV uint32_t owen_scramble(uint32_t x, uint32_t seed) {
    return __builtin_bitreverse32(lk_permutation(__builtin_bitreverse32(x), seed));
}
INSTA_DEV uint32_t hash_combine(uint32_t seed, uint32_t v) { return seed ^ (v + (seed << 6) + (seed >> 2)); }
// dimension 0 of the Sobol sequence is the bit-reversed index
INSTA_DEV float ld_random_val0(uint32_t index, uint32_t seed) {
    const float S = (float)(1.0 / 4294967296.0);
    index = owen_scramble(index, seed);
    return (float)owen_scramble(__builtin_bitreverse32(index), hash_combine(seed, 0u)) * S;
}

// ---- march helpers (testbed_nerf.cu:186-208, 313-337) --------------------
INSTA_DEV bool box_contains(const RenderArgs& a, V3 p) {
    return p.x >= a.lo[0] && p.x <= a.hi[0] && p.y >= a.lo[1] && p.y <= a.hi[1] && p.z >= a.lo[2] && p.z <= a.hi[2];
}

// density_grid_occupied_at for one cascade (testbed_nerf.cu:313-337), read
// from the linear-order copy of the Morton bitfield (same bits).
INSTA_DEV bool occupied(const uint8_t* __restrict__ grid, uint32_t G, V3 pos) {
    const float g = (float)G;
    const float px = ((pos.x - 0.5f) * 1.0f + 0.5f) * g;
    const float py = ((pos.y - 0.5f) * 1.0f + 0.5f) * g;
    const float pz = ((pos.z - 0.5f) * 1.0f + 0.5f) * g;
    int ix = (int)px, iy = (int)py, iz = (int)pz;
    const int hi = (int)G - 1;
    ix = ix < 0 ? 0 : (ix > hi ? hi : ix);
    iy = iy < 0 ? 0 : (iy > hi ? hi : iy);
    iz = iz < 0 ? 0 : (iz > hi ? hi : iz);
    const uint32_t idx = (uint32_t)ix + G * ((uint32_t)iy + G * (uint32_t)iz);
    return (grid[idx >> 3] >> (idx & 7u)) & 1u;
}

// where a ray at t leaves the voxel of pos
INSTA_DEV float next_voxel(float t, V3 pos, V3 dir, V3 idir, uint32_t res) {
    const float r = (float)res;
    const V3 p = v3(r * pos.x, r * pos.y, r * pos.z);
    const float tx = (floorf(p.x + 0.5f + 0.5f * signf(dir.x)) - p.x) * idir.x;
    const float ty = (floorf(p.y + 0.5f + 0.5f * signf(dir.y)) - p.y) * idir.y;
    const float tz = (floorf(p.z + 0.5f + 0.5f * signf(dir.z)) - p.z) * idir.z;
    const float tn = fminf(fminf(tx, ty), tz);
    return t + fmaxf(tn / r, 0.0f);
}

INSTA_DEV float advance_to_next_voxel(float t, float dt, V3 pos, V3 dir, V3 idir, uint32_t res) {
    const float t_target = next_voxel(t, pos, dir, idir, res);
    do {
        t += dt;
    } while (t < t_target);
    return t;
}

// The walk along a ray (one step per sample, one jump per empty voxel) waits
// for an occupancy bit before each step, and neither step needs it: the next
// position if this one is occupied (t + dt) and if it is empty (the next
// voxel) depend on t alone.  So kSpec positions ahead are formed as if the
// ray stayed in occupied cells (or in empty ones, whichever it was in last),
// their bits are loaded together, and the walk takes them in order up to the
// first that is different: the t values visited are those of the walk one bit
// at a time.  Bound by that chain of loads in small frames (64 x 64 of the
// small sphere, 85 samples a ray: 124 -> 108 us with the rays' t values
// reloaded four at a time too; eight ahead: 7 % slower) and by the vector ALUs
// in large ones.
constexpr int kSpec = 4;
struct Ahead {
    float t[kSpec + 1];
    bool in[kSpec], occ[kSpec];
    INSTA_DEV Ahead(const RenderArgs& a, V3 o, V3 d, V3 idir, float t0, bool through_occupied) {
        t[0] = t0;
#pragma unroll
        for (int q = 0; q < kSpec; ++q) {
            const V3 pos = o + d * t[q];
            in[q] = box_contains(a, pos);
            occ[q] = occupied(a.grid, a.G, pos);
            // (a position outside the box ends the walk: nothing is formed past it)
            t[q + 1] = through_occupied ? t[q] + a.dt
                                        : (in[q] ? advance_to_next_voxel(t[q], a.dt, pos, d, idir, a.G) : t[q]);
        }
    }
};

// Far cameras, some 10^5 away: a step may be below the last bit of t somewhere
// in the box, where advance_to_next_voxel would never end (and the walks form
// it ahead also for a ray all of whose cells are occupied).  The host tells
// (far_camera) and launches kernels of their own, so that the others' stay as
// they are (64 x 64 frame of the small sphere 370 us; with the test in every
// step, or once per ray, 385 us).
inline bool far_camera(const float origin[3], float dt) {
    // no ray's t in the box is larger: the box lies within [0, 1]^3, voxels end within one of it
    const float end = std::fabs(origin[0]) + std::fabs(origin[1]) + std::fabs(origin[2]) + 8.0f;
    return !(end + 0.5f * dt > end);
}

// The walk of a far ray, a position at a time (walk_samples; with no samples
// wanted, `most` 0, skip_empty).  One that stands still in an empty cell ends
// there, exited.
template <class Sample>
INSTA_DEV uint32_t walk_far(const RenderArgs& a, V3 o, V3 d, V3 idir, float& t, uint32_t most, bool& exited,
                            Sample&& sample) {
    uint32_t count = 0;
    exited = false;
    do {
        const V3 pos = o + d * t;
        const bool occ = occupied(a.grid, a.G, pos);
        exited = !box_contains(a, pos);
        if (exited || (occ && most == 0)) break;
        const float target = occ ? t : next_voxel(t, pos, d, idir, a.G);
        if (occ) sample(count++, t);
        do {
            const float next = t + a.dt;
            exited = !occ && !(next > t);
            t = next;
        } while (!exited && t < target);
    } while (!exited && (most == 0 || count < most));
    return count;
}

// Walk from t to the next occupied position inside the box.  Returns false
// if the ray leaves the box first.
template <bool kFar>
INSTA_DEV bool skip_empty(const RenderArgs& a, V3 o, V3 d, V3 idir, float& t) {
    if constexpr (kFar) {
        bool exited;
        walk_far(a, o, d, idir, t, 0u, exited, [](uint32_t, float) {});
        return !exited;
    }
    while (true) {
        const Ahead w(a, o, d, idir, t, false);
#pragma unroll
        for (int q = 0; q < kSpec; ++q) {
            t = w.t[q];
            if (!w.in[q]) return false;
            if (w.occ[q]) return true;
        }
        t = w.t[kSpec];
    }
}

// Up to `most` samples from t: sample(j, t) for each, in order; t ends at the
// next unvisited position.  exited: the ray left the box.
template <bool kFar, class Sample>
INSTA_DEV uint32_t walk_samples(const RenderArgs& a, V3 o, V3 d, V3 idir, float& t, uint32_t most, bool& exited,
                                Sample&& sample) {
    exited = false;
    if constexpr (kFar) return most ? walk_far(a, o, d, idir, t, most, exited, sample) : 0u;
    uint32_t count = 0;
    bool through = true;  // the last position seen was occupied
    while (count < most && !exited) {
        const Ahead w(a, o, d, idir, t, through);
        bool go = true;
        float at = t;
        t = w.t[kSpec];
#pragma unroll
        for (int q = 0; q < kSpec; ++q) {
            if (!go) continue;
            if (count >= most || !w.in[q]) {
                exited = count < most;
                t = w.t[q];
                go = false;
            } else {
                if (w.occ[q]) sample(count++, w.t[q]);
                if (w.occ[q] != through) {  // the positions ahead were formed the other way
                    at = w.t[q];
                    go = false;
                    t = -1.0f;
                }
            }
        }
        if (t == -1.0f) {
            through = !through;
            t = through ? at + a.dt : advance_to_next_voxel(at, a.dt, o + d * at, d, idir, a.G);
        }
    }
    return count;
}

INSTA_DEV float box_ray_tmin(const RenderArgs& a, V3 o, V3 d) {
    float tmin = (a.lo[0] - o.x) / d.x, tmax = (a.hi[0] - o.x) / d.x;
    if (tmin > tmax) { float s = tmin; tmin = tmax; tmax = s; }
    float tymin = (a.lo[1] - o.y) / d.y, tymax = (a.hi[1] - o.y) / d.y;
    if (tymin > tymax) { float s = tymin; tymin = tymax; tymax = s; }
    if (tmin > tymax || tymin > tmax) return 3.40282347e38f;
    if (tymin > tmin) tmin = tymin;
    if (tymax < tmax) tmax = tymax;
    float tzmin = (a.lo[2] - o.z) / d.z, tzmax = (a.hi[2] - o.z) / d.z;
    if (tzmin > tzmax) { float s = tzmin; tzmin = tzmax; tzmax = s; }
    if (tmin > tzmax || tzmin > tmax) return 3.40282347e38f;
    if (tzmin > tmin) tmin = tzmin;
    return tmin;
}

// Reservations: one atomic per workgroup of `kWaves` full waves, every thread
// calling.  Atomics on one counter retire one at a time over the whole chip,
// about 6.4 ns each (with one per wave, the 16,384 waves of a 1024 x 1024
// frame spent 105 us of their ray set-up on it), so a workgroup sums its
// waves' counts in LDS first.

// exclusive prefix of v over the workgroup, plus one atomic reservation
template <uint32_t kWaves>
INSTA_DEV uint32_t block_reserve(uint32_t* counter, uint32_t v) {
    __shared__ uint32_t s_wave[kWaves], s_base;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t incl = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t up = __shfl_up(incl, o);
        if (lane >= (uint32_t)o) incl += up;
    }
    if (lane == 63u) s_wave[wave] = incl;
    __syncthreads();
    uint32_t before = 0, total = 0;
#pragma unroll
    for (uint32_t w = 0; w < kWaves; ++w) {
        if (w < wave) before += s_wave[w];
        total += s_wave[w];
    }
    if (threadIdx.x == 0) s_base = total ? atomicAdd(counter, total) : 0u;
    __syncthreads();
    const uint32_t slot = s_base + before + incl - v;
    __syncthreads();  // a later reservation reuses the LDS words
    return slot;
}

// this thread's slot in a list (only meaningful if `want`)
template <uint32_t kWaves>
INSTA_DEV uint32_t block_append(uint32_t* counter, bool want) {
    return block_reserve<kWaves>(counter, want ? 1u : 0u);
}

INSTA_DEV uint32_t wave_max(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor(v, o));
    return v;
}

// Step-major order within a wave's sample range: sample j of lane l sits at
// wave_base + (samples of steps < j over the wave's lanes) + (lanes below l
// with more than j samples).  Lanes are adjacent rays, so neighbouring
// samples are the same step of neighbouring pixels.  Every lane of the wave
// calls this with the same j sequence (j < the wave's largest count).
struct StepMajor {
    uint32_t running = 0;
    INSTA_DEV uint32_t next(uint32_t j, uint32_t count, bool& mine) {
        const uint64_t act = __ballot(j < count);
        const uint32_t lane = threadIdx.x & 63u;
        const uint64_t below = act & ((1ull << lane) - 1ull);
        const uint32_t slot = running + (uint32_t)__popcll(below);
        running += (uint32_t)__popcll(act);
        mine = j < count;
        return slot;
    }
};

}  // namespace insta
