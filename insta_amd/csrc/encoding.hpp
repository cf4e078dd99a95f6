// encoding.hpp -- hash-grid encoding, spherical-harmonics direction
// encoding and the bias-free dense layer, shared by the inference and
// training kernels.
//
// Hash grid convention (the reference delegates it to tiny-cuda-nn, absent
// from its tree; Instant-NGP, Mueller et al. 2022): level l uses scale s_l =
// b^l * N_min - 1 and resolution ceil(s_l) + 1; position x maps to
// x * s_l + 0.5, whose floor/fraction give the cell and trilinear weights;
// dense levels index x + y r + z r^2, hashed levels
// (x * 1 ^ y * 2654435761 ^ z * 805459861) mod T.
#pragma once

#include "context.hpp"

namespace insta {

// table entry of corner cg on a level: dense levels index x + y r + z r^2
// (wrapped into the level's table), hashed levels use the spatial hash
INSTA_DEV uint32_t grid_index(const uint32_t cg[3], bool dense, uint32_t res, uint32_t size) {
    if (dense) {
        uint32_t idx = cg[0] + cg[1] * res + cg[2] * (res * res);
        if (idx >= size) idx %= size;
        return idx;
    }
    return (cg[0] ^ (cg[1] * 2654435761u) ^ (cg[2] * 805459861u)) & (size - 1u);
}

// Position x's cell on level l: its lower corner g, the offset in it and the
// trilinear weights, corner c's bit d the upper one on axis d.
INSTA_DEV void cell_weights(float sc, V3 x, uint32_t g[3], float frac[3], float w[8]) {
    const float px = x.x * sc + 0.5f, py = x.y * sc + 0.5f, pz = x.z * sc + 0.5f;
    const float fx = floorf(px), fy = floorf(py), fz = floorf(pz);
    frac[0] = px - fx, frac[1] = py - fy, frac[2] = pz - fz;
    g[0] = (uint32_t)(int32_t)fx, g[1] = (uint32_t)(int32_t)fy, g[2] = (uint32_t)(int32_t)fz;
    const float u0 = 1.0f - frac[0], u1 = 1.0f - frac[1], u2 = 1.0f - frac[2];
    const float xy[4] = {u0 * u1, frac[0] * u1, u0 * frac[1], frac[0] * frac[1]};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        w[c] = xy[c] * u2;
        w[c + 4] = xy[c] * frac[2];
    }
}

// Entries of a cell's corners on a dense level, wrapped as grid_index: only
// positions outside [0, 1]^3 need it, so the callers test the whole cell once
// (tested corner by corner, every corner's load sat behind a branch of its own
// and the eight loads went out one after another).
INSTA_DEV void dense_corners(const uint32_t g[3], uint32_t res, uint32_t size, uint32_t idx[8]) {
    const uint32_t res2 = res * res, first = g[0] + g[1] * res + g[2] * res2;
#pragma unroll
    for (uint32_t c = 0; c < 8; ++c) {
        idx[c] = first + (c & 1u) + ((c & 2u) ? res : 0u) + ((c & 4u) ? res2 : 0u);
        if (idx[c] >= size) idx[c] %= size;
    }
}

constexpr uint32_t kPrimeY = 2654435761u, kPrimeZ = 805459861u;

// The eight corners of position x's cell on level l: table entries (as
// grid_index) and weights, for the gradient scatters.
INSTA_DEV void cell_corners(const GridParams& gp, uint32_t l, V3 x, uint32_t idx[8], float w[8]) {
    uint32_t g[3];
    float frac[3];
    cell_weights(gp.scale[l], x, g, frac, w);
    const uint32_t res = gp.res[l], size = gp.size[l];
    if ((gp.dense_mask >> l) & 1u) {
        const uint32_t res2 = res * res;
        const uint32_t first = g[0] + g[1] * res + g[2] * res2;
#pragma unroll
        for (uint32_t c = 0; c < 8; ++c)
            idx[c] = first + (c & 1u) + ((c & 2u) ? res : 0u) + ((c & 4u) ? res2 : 0u);
        // inside the grid the last corner's entry is the largest
        if (!(g[0] < res && g[1] < res && g[2] < res && idx[7] < size)) dense_corners(g, res, size, idx);
    } else {
        const uint32_t hy = g[1] * kPrimeY, hz = g[2] * kPrimeZ;
        const uint32_t yz[4] = {hy ^ hz, (hy + kPrimeY) ^ hz, hy ^ (hz + kPrimeZ), (hy + kPrimeY) ^ (hz + kPrimeZ)};
#pragma unroll
        for (uint32_t c = 0; c < 8; ++c) idx[c] = ((g[0] + (c & 1u)) ^ yz[c >> 1]) & (size - 1u);
    }
}

// Values of the corners' entries (E: an entry of two features, base: the
// level's table), the offsets in the cell and the weights.  Coherent positions
// (renders) are bound by the instructions of this function, scattered ones by
// cache lookups, one per lane and load.  So the corners of an x pair come with
// one load: neighbours on dense levels; on hashed ones the two hashes of an
// even x differ in bit 0 only.  Of an odd x, the lower corner comes with its
// pair all the same and the upper one by itself (kPairs: no lane waits for the
// others' way), or lanes with an odd x load all corners by themselves
// (kEvenPairs: two ways, but no bytes for nothing), or all lanes do (kSingle).
// Offsets are computed in bytes (the hash's factors times the entry's size),
// dense rows lie at four scalar bases, and which half of its aligned pair a
// corner is follows from the cell's parity, the factors being odd.
// 16-level head, us, corners one after another / kSingle / kPairs / kEvenPairs:
//   FP32 render at 512 x 512              1,355 / 1,294 / 1,255 / 1,330
//   1,048,576 positions near the skin, FP32 617 / 623 / 560 / 504, BF16 458 / 387 / 383 / 331
//   anywhere,                          FP32 817 / 892 / 853 / 830, BF16 628 / 587 / 616 / 525
//   on a lattice,                      FP32 679 / 703 / 706 / 695, BF16 505 / 500 / 589 / 527
// so renders, training and the density grid take kPairs, inference calls, whose
// positions may come in any order, kEvenPairs.
enum Corners { kPairs, kEvenPairs, kSingle };
template <class E, Corners kMode = kPairs>
INSTA_DEV void cell_fetch(const GridParams& gp, uint32_t l, V3 x, const char* __restrict__ base, E v[8], float frac[3],
                          float w[8]) {
    struct Two {  // aligned as one entry: half of the pairs start at an odd one
        E a, b;
    };
    constexpr uint32_t S = sizeof(E);
    uint32_t g[3];
    cell_weights(gp.scale[l], x, g, frac, w);
    const uint32_t size = gp.size[l];
    if ((gp.dense_mask >> l) & 1u) {
        // a dense level has at most 2^26 entries, so a slab of it less than
        // 2^18: the byte strides fit the 24-bit multiplier
        const uint32_t res = gp.res[l], row = res * S, slab = res * res * S;
        const uint32_t at = g[0] * S + __umul24(g[1], row) + __umul24(g[2], slab);
        // inside the grid the last corner's entry is the largest
        if (__builtin_expect(g[0] < res && g[1] < res && g[2] < res && at + row + slab + S < size * S, 1)) {
            const char* rows[4] = {base, base + row, base + slab, base + slab + row};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const Two t = *reinterpret_cast<const Two*>(rows[j] + at);
                v[2 * j] = t.a;
                v[2 * j + 1] = t.b;
            }
        } else {
            uint32_t idx[8];
            dense_corners(g, res, size, idx);
#pragma unroll
            for (int c = 0; c < 8; ++c) v[c] = *reinterpret_cast<const E*>(base + idx[c] * S);
        }
    } else {
        const uint32_t mask = (size - 1u) * S;
        const uint32_t hy = g[1] * (kPrimeY * S), hz = g[2] * (kPrimeZ * S);
        const uint32_t hy1 = hy + kPrimeY * S, hz1 = hz + kPrimeZ * S;
        const uint32_t yz[4] = {hy ^ hz, hy1 ^ hz, hy ^ hz1, hy1 ^ hz1};
        const uint32_t x0 = g[0] * S, x1 = x0 + S;
        const bool apart = g[0] & 1u;
        if (kMode == kSingle || (kMode == kEvenPairs && apart)) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[2 * j] = *reinterpret_cast<const E*>(base + ((x0 ^ yz[j]) & mask));
                v[2 * j + 1] = *reinterpret_cast<const E*>(base + ((x1 ^ yz[j]) & mask));
            }
            return;
        }
        Two t[4];  // level tables hold an even number of entries
#pragma unroll
        for (int j = 0; j < 4; ++j) t[j] = *reinterpret_cast<const Two*>(base + ((x0 ^ yz[j]) & (mask & ~S)));
        E up[4];
        if (kMode == kPairs && apart) {
#pragma unroll
            for (int j = 0; j < 4; ++j) up[j] = *reinterpret_cast<const E*>(base + ((x1 ^ yz[j]) & mask));
        }
        const bool upper = (g[0] ^ g[1] ^ g[2]) & 1u;  // rows 0 and 3; rows 1 and 2 the other half
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool odd = (j == 0 || j == 3) ? upper : !upper;
            v[2 * j] = odd ? t[j].b : t[j].a;
            const E other = odd ? t[j].a : t[j].b;
            v[2 * j + 1] = kMode == kPairs && apart ? up[j] : other;
        }
    }
}

// Features of position x on level l; kMode as in cell_fetch (F = 2).
template <int F, Corners kMode = kPairs>
INSTA_DEV void encode_level(const float* __restrict__ table, const GridParams& gp, uint32_t l, V3 x, float acc[F]) {
    float w[8];
    const char* base = reinterpret_cast<const char*>(table + (size_t)gp.offset[l] * F);
#pragma unroll
    for (int f = 0; f < F; ++f) acc[f] = 0.0f;
    if constexpr (F == 2) {
        float2 v[8];
        float frac[3];
        cell_fetch<float2, kMode>(gp, l, x, base, v, frac, w);
#pragma unroll
        for (uint32_t c = 0; c < 8; ++c) {
            acc[0] = acc[0] + w[c] * v[c].x;
            acc[1] = acc[1] + w[c] * v[c].y;
        }
        return;
    }
    uint32_t idx[8];
    cell_corners(gp, l, x, idx, w);
    if constexpr (F == 4) {
#pragma unroll
        for (uint32_t c = 0; c < 8; ++c) {
            const float4 v = *reinterpret_cast<const float4*>(base + (size_t)idx[c] * 16u);
            acc[0] = acc[0] + w[c] * v.x;
            acc[1] = acc[1] + w[c] * v.y;
            acc[2] = acc[2] + w[c] * v.z;
            acc[3] = acc[3] + w[c] * v.w;
        }
    } else if constexpr (F != 2) {
#pragma unroll
        for (uint32_t c = 0; c < 8; ++c) {
            const float* e = reinterpret_cast<const float*>(base + (size_t)idx[c] * (4u * F));
#pragma unroll
            for (int f = 0; f < F; ++f) acc[f] = acc[f] + w[c] * e[f];
        }
    }
}

// real SH bands 0..3 of a direction in [-1,1]^3 (see the oracle for the
// normalisation constants' closed forms)
INSTA_DEV void sh16(float x, float y, float z, float* o) {
    const float xy = x * y, xz = x * z, yz = y * z, x2 = x * x, y2 = y * y, z2 = z * z;
    o[0] = 0.28209479177387814f;
    o[1] = -0.48860251190291987f * y;
    o[2] = 0.48860251190291987f * z;
    o[3] = -0.48860251190291987f * x;
    o[4] = 1.0925484305920792f * xy;
    o[5] = -1.0925484305920792f * yz;
    o[6] = 0.94617469575755997f * z2 - 0.31539156525251999f;
    o[7] = -1.0925484305920792f * xz;
    o[8] = 0.54627421529603959f * x2 - 0.54627421529603959f * y2;
    o[9] = 0.59004358992664352f * y * (-3.0f * x2 + y2);
    o[10] = 2.8906114426405538f * xy * z;
    o[11] = 0.45704579946446572f * y * (1.0f - 5.0f * z2);
    o[12] = 0.3731763325901154f * z * (5.0f * z2 - 3.0f);
    o[13] = 0.45704579946446572f * x * (1.0f - 5.0f * z2);
    o[14] = 1.4453057213202769f * z * (x2 - y2);
    o[15] = 0.59004358992664352f * x * (-x2 + 3.0f * y2);
}

// bias-free dense layer, row-major W[out][in]; weights are wave-uniform and
// reach the FMAs as scalar operands
template <int NIN, int NOUT, bool RELU>
INSTA_DEV void dense(const float* __restrict__ W, const float* x, float* y) {
#pragma unroll
    for (int o = 0; o < NOUT; ++o) {
        float acc = 0.0f;
#pragma unroll
        for (int i = 0; i < NIN; ++i) acc = __builtin_fmaf(W[o * NIN + i], x[i], acc);
        y[o] = RELU ? (acc > 0.0f ? acc : 0.0f) : acc;
    }
}

}  // namespace insta
