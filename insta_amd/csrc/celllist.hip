// celllist.hip -- per-cell candidate lists for the nearest-triangle query of
// the sample deformation (`warp`, src/core.cu:442-526, which calls
// closest_triangle, bvh.cuh:48-96, once per sample).
//
// The reference answers every query by a BVH traversal.  Here the marched
// samples of a frame all lie in occupied cells of the frame's occupancy grid,
// so the build below gives each occupied cell (split into S^3 sub-cells) the
// short list of triangles that can be nearest to a point inside it; a query
// in such a sub-cell scans that list instead of walking the tree.  The
// invariant that makes the answer identical to the BVH's (and to brute
// force) is stated with the layout in common.hpp.
//
// Build, per slot, all on the device and capturable into a graph (no host
// reads, no memsets, grids sized by the caps):
//   1. words: snapshot of the linear occupancy bits, popcount per 64 cells
//   2. scan:  exclusive prefix of the popcounts (one workgroup)
//   3. cells: linear index of each occupied cell, in rank order
//   4. lists: (S = 4) one workgroup per occupied cell gathers the triangles that can
//             matter to any of its sub-cells, then takes each one's seed
//             (nearest triangle at the centre), bound U^2 (from the 8
//             corners), count and entries from those; it claims its entries
//             with one atomic (layout order varies, contents do not)
//   5. count, fill: (other splits, and cells with too many candidates for LDS)
//             one lane per sub-cell: nearest triangle at the centre
//             (BVH), the bound U^2 from the 8 corners, a bounded BVH range walk
//             counting the triangles whose box is within U; the same walk
//             writes the entries, seed first
//   6. sort:  one wave per list orders the entries after the seed by box
//             distance (rank by counting)
//   7. finish: lists valid unless the occupied cells exceeded the cap
#include "context.hpp"

namespace insta {
namespace {

constexpr uint32_t kClThreads = 256;
constexpr uint32_t kScanThreads = 1024;
constexpr uint32_t kClMaxBlocks = 8192;
// a list holds its seed and at most 64 * kSortPerLane more entries (the sort
// kernel's reach); longer ones leave their sub-cell to the BVH
constexpr uint32_t kSortPerLane = 8;
constexpr uint32_t kMaxList = 1u + 64u * kSortPerLane;

__global__ void cl_begin_kernel(uint32_t* __restrict__ state) {
    if (threadIdx.x < kClState) state[threadIdx.x] = 0u;
}

__global__ void cl_invalidate_kernel(uint32_t* __restrict__ state, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) state[kClState * i + 2] = 0u;
}

__global__ void cl_words_kernel(const uint64_t* __restrict__ lin, uint32_t n_words, uint64_t* __restrict__ bits,
                                uint32_t* __restrict__ rank) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_words) return;
    const uint64_t w = lin[i];
    bits[i] = w;
    rank[i] = (uint32_t)__popcll(w);
}

// rank[i] <- popcounts before word i; state[0] = occupied cells,
// state[3] = 1 when they exceed the cap.  One workgroup, bound by latency: it
// reads uint4s side by side, the next tile's while it scans this one (128^3
// cells, 32,768 words: 9.5 us, with a run of 32 words a thread 58).
__global__ __launch_bounds__(kScanThreads) void cl_scan_kernel(uint32_t* __restrict__ rank, uint32_t n_words,
                                                               uint32_t cap, uint32_t* __restrict__ state) {
    __shared__ uint32_t part[kScanThreads / 64];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    // whole uint4s: the grid's edge is a multiple of 8, its words of 8 too
    uint4* __restrict__ r4 = reinterpret_cast<uint4*>(rank);
    const uint32_t n4 = n_words / 4u;
    const auto load = [&](uint32_t i) { return i < n4 ? r4[i] : make_uint4(0u, 0u, 0u, 0u); };
    uint32_t carry = 0;
    uint4 next = load(t);
    for (uint32_t base = 0; base < n4; base += kScanThreads) {
        const uint4 v = next;
        next = load(base + kScanThreads + t);
        const uint32_t s = v.x + v.y + v.z + v.w;
        uint32_t incl = s;
#pragma unroll
        for (uint32_t o = 1; o < 64u; o <<= 1) {
            const uint32_t up = __shfl_up(incl, o);
            if (lane >= o) incl += up;
        }
        if (lane == 63u) part[wave] = incl;
        __syncthreads();
        uint32_t before = 0, total = 0;
#pragma unroll
        for (uint32_t w = 0; w < kScanThreads / 64; ++w) {
            if (w < wave) before += part[w];
            total += part[w];
        }
        const uint32_t x = carry + before + incl - s;
        if (base + t < n4) r4[base + t] = make_uint4(x, x + v.x, x + v.x + v.y, x + v.x + v.y + v.z);
        carry += total;
        __syncthreads();  // the next tile reuses part
    }
    if (t == 0) {
        state[0] = carry;
        state[3] = carry > cap ? 1u : 0u;
    }
}

__global__ void cl_cells_kernel(const uint64_t* __restrict__ bits, const uint32_t* __restrict__ rank, uint32_t n_words,
                                uint32_t cap, uint32_t* __restrict__ cells) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_words) return;
    uint64_t w = bits[i];
    uint32_t r = rank[i];
    while (w) {
        const uint32_t j = (uint32_t)__ffsll((unsigned long long)w) - 1u;
        if (r < cap) cells[r] = i * 64u + j;
        ++r;
        w &= w - 1ull;
    }
}

struct ClArgs {
    MeshView m;
    const uint32_t* cells;
    uint32_t* left;       // [cap] ranks of the cells cl_cell_kernel's first launch left to its second
                          // (state[5] of them)
    uint32_t* walk;       // [cap] by rank: 1 where it left the cell to the per-lane kernels
    uint32_t all;         // the per-lane kernels take every cell
    uint2* head;
    uint32_t* ent;
    uint32_t* state;
    uint32_t G, S, cap, ent_cap;
};

// First of n list entries.  Lists too long to keep claim theirs too, so that
// the total tells what capacity would hold all; over a large, densely occupied
// grid it passes 2^32 (256^3 sub-cells around a 16,000-triangle mesh: above 6e9), and
// a 32-bit count would hand out the first entries again.
INSTA_DEV uint64_t claim_entries(uint32_t* state, uint32_t n) {
    return atomicAdd(reinterpret_cast<unsigned long long*>(state + kClClaim), (unsigned long long)n);
}

// sub-cell `sub` of occupied cell `cell`, grown by kCellEps
INSTA_DEV void sub_box(const ClArgs& a, uint32_t cell, uint32_t sub, float4& lo, float4& hi) {
    const uint32_t cx = cell % a.G, cy = (cell / a.G) % a.G, cz = cell / (a.G * a.G);
    const uint32_t sx = sub % a.S, sy = (sub / a.S) % a.S, sz = sub / (a.S * a.S);
    const float inv = 1.0f / (float)(a.G * a.S);
    lo = make_float4((float)(cx * a.S + sx) * inv - kCellEps, (float)(cy * a.S + sy) * inv - kCellEps,
                     (float)(cz * a.S + sz) * inv - kCellEps, 0.0f);
    hi = make_float4((float)(cx * a.S + sx + 1u) * inv + kCellEps, (float)(cy * a.S + sy + 1u) * inv + kCellEps,
                     (float)(cz * a.S + sz + 1u) * inv + kCellEps, 0.0f);
}

INSTA_DEV void tri_verts(const MeshView& m, uint32_t t, V3& a, V3& b, V3& c) {
    const float4 r0 = m.btris[3 * t], r1 = m.btris[3 * t + 1], r2 = m.btris[3 * t + 2];
    a = v3(r0.x, r0.y, r0.z);
    b = v3(r0.w, r1.x, r1.y);
    c = v3(r1.z, r1.w, r2.x);
}

// squared distance between two boxes
INSTA_DEV float box_box_sq(float4 alo, float4 ahi, float4 blo, float4 bhi) {
    const float dx = fmaxf(fmaxf(alo.x - bhi.x, blo.x - ahi.x), 0.0f);
    const float dy = fmaxf(fmaxf(alo.y - bhi.y, blo.y - ahi.y), 0.0f);
    const float dz = fmaxf(fmaxf(alo.z - bhi.z, blo.z - ahi.z), 0.0f);
    return dx * dx + dy * dy + dz * dz;
}

// U^2: the largest squared distance from a corner of the box to triangle t,
// with a relative margin over the rounding of the distances and boxes
INSTA_DEV float seed_bound(const MeshView& m, uint32_t t, float4 lo, float4 hi) {
    V3 a, b, c;
    tri_verts(m, t, a, b, c);
    float mx = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const V3 q = v3(k & 1 ? hi.x : lo.x, k & 2 ? hi.y : lo.y, k & 4 ? hi.z : lo.z);
        mx = fmaxf(mx, tri_distance_sq(a, b, c, q));
    }
    return mx * (1.0f + 0x1p-10f) + 0x1p-40f;
}

// Every triangle (BVH order) whose box lies within squared distance U2 of the
// box [lo, hi], in tree order: emit(t, d2).  Depth-first over the implicit
// 4-ary heap; at most 3 pending siblings per inner level.
template <class Emit>
INSTA_DEV void bvh_range(const MeshView& m, float4 lo, float4 hi, float U2, uint32_t* stack, uint32_t stride,
                         Emit&& emit) {
    const uint32_t shift = 2u * m.k;
    int sp = 0;
    uint32_t node = 0;
    for (;;) {
        if (node < m.leaf_base) {
            const uint32_t first = 4u * node + 1u;
            uint32_t next = kNoNode;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint32_t ch = first + c;
                if (box_box_sq(lo, hi, m.nodes[2 * ch], m.nodes[2 * ch + 1]) <= U2) {
                    if (next != kNoNode) stack[(sp++) * stride] = next;
                    next = ch;
                }
            }
            if (next != kNoNode) {
                node = next;
                continue;
            }
        } else {
            const uint32_t j = node - m.leaf_base;
            const uint32_t b = (uint32_t)(((uint64_t)j * m.nf) >> shift);
            const uint32_t e = (uint32_t)(((uint64_t)(j + 1) * m.nf) >> shift);
            for (uint32_t t = b; t < e; ++t) {
                V3 va, vb, vc;
                tri_verts(m, t, va, vb, vc);
                const float4 tlo = make_float4(fminf(fminf(va.x, vb.x), vc.x), fminf(fminf(va.y, vb.y), vc.y),
                                               fminf(fminf(va.z, vb.z), vc.z), 0.0f);
                const float4 thi = make_float4(fmaxf(fmaxf(va.x, vb.x), vc.x), fmaxf(fmaxf(va.y, vb.y), vc.y),
                                               fmaxf(fmaxf(va.z, vb.z), vc.z), 0.0f);
                const float d2 = box_box_sq(lo, hi, tlo, thi);
                if (d2 <= U2) emit(t, d2);
            }
        }
        if (sp == 0) break;
        node = stack[(--sp) * stride];
    }
}

// One workgroup per occupied cell.  The sub-cells' lists come from one
// candidate set: with D the largest distance from a corner of the cell to the
// triangle nearest its centre and r half a sub-cell's diagonal, a sub-cell's
// own bound U is at most D + r (its seed is no farther from its centre than
// that triangle, and its corners are within r of its centre), so every entry
// of its list lies within D + r of the cell.  The workgroup walks the tree
// level by level (the frontier's children side by side) and gathers the
// triangles' boxes in LDS; then thread = (sub-cell, share of the candidates),
// the shares' seeds, corner distances and counts combined through LDS: the
// same seed, bound, box distances and entries as a walk of the sub-cell's own,
// whose chain of node loads and divergence (a sub-cell beside the mesh's pole
// visits hundreds of triangles) set the per-lane kernels' time.  Bound by the
// seeds' exact distances over the candidates: a 9,976-triangle head's 8,622
// cells (17 M entries) take 382 + 86 us (second launch); one lane per sub-cell,
// counting and filling walks, 1,029 + 444 us.
// A second launch (kSecond) takes the cells with more than kCellCand candidates
// with larger workgroups and lists, up to kCellCand2 of them; cells with more go
// to the per-lane kernels.
constexpr uint32_t kCellThreads = 256, kCellCand = 1024;
constexpr uint32_t kCellThreads2 = 1024, kCellCand2 = 3072;

// slot of this thread's item in an LDS list of kCellCand (>= kCellCand: full);
// whole waves call
INSTA_DEV uint32_t lds_append(uint32_t* n, bool live) {
    const uint64_t mask = __ballot(live);
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t base = 0;
    if (lane == 0 && mask) base = atomicAdd(n, (uint32_t)__popcll(mask));
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    return base + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
}

template <bool kSecond>
__global__ __launch_bounds__(kSecond ? kCellThreads2 : kCellThreads) void cl_cell_kernel(ClArgs a) {
    constexpr uint32_t kThreads = kSecond ? kCellThreads2 : kCellThreads, kWaves = kThreads / 64u;
    constexpr uint32_t kCand = kSecond ? kCellCand2 : kCellCand;  // candidates, and tree nodes of a level
    __shared__ uint16_t s_node[2][kCand], s_tri[kCand];
    __shared__ float s_lo[kCand][3], s_hi[kCand][3];
    __shared__ uint32_t s_n[2], s_cand;
    __shared__ uint64_t s_base;
    __shared__ uint32_t s_u[kThreads], s_v[kThreads], s_w[kThreads];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t S3 = a.S * a.S * a.S, shares = kThreads / S3;
    const uint32_t sub = tid % S3, share = tid / S3;
    const uint32_t n_cells = kSecond ? a.state[5] : min(a.state[0], a.cap);
    const uint32_t shift = 2u * a.m.k, n_leaves = 1u << shift;
    auto box = [&](uint32_t q, float4& lo, float4& hi) {
        lo = make_float4(s_lo[q][0], s_lo[q][1], s_lo[q][2], 0.0f);
        hi = make_float4(s_hi[q][0], s_hi[q][1], s_hi[q][2], 0.0f);
    };
    for (uint32_t ci = blockIdx.x; ci < n_cells; ci += gridDim.x) {
        const uint32_t rank = kSecond ? a.left[ci] : ci, cell = a.cells[rank];
        float4 lo, hi, blo, bhi, tmp;  // this thread's sub-cell; the whole cell
        sub_box(a, cell, sub, lo, hi);
        sub_box(a, cell, 0u, blo, tmp);
        sub_box(a, cell, S3 - 1u, tmp, bhi);
        const V3 mid = v3((blo.x + bhi.x) * 0.5f, (blo.y + bhi.y) * 0.5f, (blo.z + bhi.z) * 0.5f);
        // a triangle near the cell's centre: the nearest of the leaf nearest
        // by box (any triangle bounds the candidates; a near one tightly)
        uint64_t nearest = ~0ull;
        for (uint32_t j = tid; j < n_leaves; j += kThreads) {
            const uint32_t node = a.m.leaf_base + j;
            const float d = box_distance_sq(a.m.nodes[2 * node], a.m.nodes[2 * node + 1], mid);
            const uint64_t key = (uint64_t)__float_as_uint(d) << 32 | j;
            nearest = key < nearest ? key : nearest;
        }
        const uint32_t dmin = wave_min_bits((uint32_t)(nearest >> 32));
        const uint32_t jmin = wave_min_bits((uint32_t)(nearest >> 32) == dmin ? (uint32_t)nearest : 0xffffffffu);
        if (lane == 0) {
            s_u[wave] = dmin;
            s_v[wave] = jmin;
        }
        if (tid < 2u) s_n[tid] = tid == 0 ? 1u : 0u;
        if (tid == 0) {
            s_cand = 0u;
            s_node[0][0] = 0;
        }
        __syncthreads();
        uint32_t wl = 0;
        for (uint32_t w = 1; w < kWaves; ++w)
            if (s_u[w] < s_u[wl]) wl = w;
        const uint32_t leaf0 = s_v[wl];
        float best_d = 3.40282347e38f;
        uint32_t first = 0;
        V3 va, vb, vc;
        {
            const uint32_t t0 = (uint32_t)(((uint64_t)leaf0 * a.m.nf) >> shift);
            const uint32_t t1 = (uint32_t)(((uint64_t)(leaf0 + 1) * a.m.nf) >> shift);
            uint32_t d = 0xffffffffu;
            for (uint32_t t = t0 + lane; t < t1; t += 64u) {  // (each wave alike)
                tri_verts(a.m, t, va, vb, vc);
                const uint32_t x = __float_as_uint(tri_distance_sq(va, vb, vc, mid));
                if (x < d) {
                    d = x;
                    first = t;
                }
            }
            const uint32_t dm = wave_min_bits(d);
            first = wave_min_bits(d == dm ? first : 0xffffffffu);
            if (first == 0xffffffffu || dm > 0x7f7fffffu) first = t0;
        }
        tri_verts(a.m, first, va, vb, vc);
        const V3 corner = v3(lane & 1 ? bhi.x : blo.x, lane & 2 ? bhi.y : blo.y, lane & 4 ? bhi.z : blo.z);
        best_d = __uint_as_float(~wave_min_bits(~__float_as_uint(tri_distance_sq(va, vb, vc, corner))));
        const float D = sqrtf(best_d), r = 0.5f * sqrtf(sqnorm(xyz(hi) - xyz(lo)));
        const float C2 = (D + r) * (D + r) * (1.0f + 0x1p-8f) + 0x1p-30f;
        // the tree, a level at a time
        uint32_t cur = 0;
        bool overflow = !(C2 < 3.0e38f);
        for (uint32_t depth = 0; depth < a.m.k && !overflow; ++depth) {
            const uint32_t n_cur = s_n[cur];
            for (uint32_t b = 0; b < 4u * n_cur; b += kThreads) {
                const uint32_t j = b + tid;
                const bool in = j < 4u * n_cur;
                const uint32_t ch = in ? 4u * s_node[cur][j / 4u] + 1u + (j & 3u) : 1u;
                const bool live = in && box_box_sq(blo, bhi, a.m.nodes[2 * ch], a.m.nodes[2 * ch + 1]) <= C2;
                const uint32_t slot = lds_append(&s_n[cur ^ 1u], live);
                if (live && slot < kCand) s_node[cur ^ 1u][slot] = (uint16_t)ch;
            }
            __syncthreads();
            cur ^= 1u;
            overflow = s_n[cur] > kCand;
            if (tid == 0) s_n[cur ^ 1u] = 0u;
            __syncthreads();
        }
        // the surviving leaves' triangles, 16 threads a leaf
        if (!overflow) {
            const uint32_t n_cur = s_n[cur];
            for (uint32_t b = 0; b < n_cur; b += kThreads / 16u) {
                const uint32_t li = b + tid / 16u;
                const uint32_t j = li < n_cur ? s_node[cur][li] - a.m.leaf_base : 0u;
                const uint32_t t0 = (uint32_t)(((uint64_t)j * a.m.nf) >> shift);
                const uint32_t t1 = li < n_cur ? (uint32_t)(((uint64_t)(j + 1) * a.m.nf) >> shift) : t0;
                for (uint32_t t = t0 + tid % 16u; __ballot(t < t1) != 0ull; t += 16u) {
                    bool live = t < t1;
                    float4 tlo, thi;
                    if (live) {
                        tri_verts(a.m, t, va, vb, vc);
                        tlo = make_float4(fminf(fminf(va.x, vb.x), vc.x), fminf(fminf(va.y, vb.y), vc.y),
                                          fminf(fminf(va.z, vb.z), vc.z), 0.0f);
                        thi = make_float4(fmaxf(fmaxf(va.x, vb.x), vc.x), fmaxf(fmaxf(va.y, vb.y), vc.y),
                                          fmaxf(fmaxf(va.z, vb.z), vc.z), 0.0f);
                        live = box_box_sq(blo, bhi, tlo, thi) <= C2;
                    }
                    const uint32_t slot = lds_append(&s_cand, live);
                    if (live && slot < kCand) {
                        s_tri[slot] = (uint16_t)t;
                        s_lo[slot][0] = tlo.x; s_lo[slot][1] = tlo.y; s_lo[slot][2] = tlo.z;
                        s_hi[slot][0] = thi.x; s_hi[slot][1] = thi.y; s_hi[slot][2] = thi.z;
                    }
                }
            }
            __syncthreads();
            overflow = s_cand > kCand || s_cand == 0u;
        }
        if (overflow) {  // left to the second launch, or (too many for it as well) to the per-lane kernels
            if (tid == 0) {
                const bool walk = kSecond || s_cand > kCellCand2;  // (s_cand: all of them where the tree's levels fit)
                a.walk[rank] = walk ? 1u : 0u;
                if (!walk) a.left[atomicAdd(&a.state[5], 1u)] = rank;
            }
            __syncthreads();
            continue;
        }
        if (tid == 0) a.walk[rank] = 0u;
        const uint32_t n_cand = s_cand;
        // the seed: nearest to the sub-cell's centre (the order and prune margin of bvh_closest)
        const V3 ctr = v3((lo.x + hi.x) * 0.5f, (lo.y + hi.y) * 0.5f, (lo.z + hi.z) * 0.5f);
        uint32_t best = 0x7f7fffffu, best_key = 0xffffffffu;  // distance bits; original id << 16 | triangle
        float bound = prune_bound(3.40282347e38f);
        for (uint32_t q = share; q < n_cand; q += shares) {
            uint32_t key = 0;
            float4 tlo, thi;
            box(q, tlo, thi);
            if (box_distance_sq(tlo, thi, ctr) > bound) continue;
            const uint32_t d = triangle_candidate<false>(a.m, s_tri[q], ctr, bound, key);
            if (d < best || (d == best && key < best_key)) {
                best = d;
                best_key = key;
                bound = prune_bound(__uint_as_float(d));
            }
        }
        s_u[tid] = best;
        s_v[tid] = best_key;
        __syncthreads();
        for (uint32_t q = 0; q < shares; ++q) {
            const uint32_t d = s_u[q * S3 + sub], key = s_v[q * S3 + sub];
            if (d < best || (d == best && key < best_key)) {
                best = d;
                best_key = key;
            }
        }
        const uint32_t seed = best_key & 0xffffu;
        const bool found = best_key != 0xffffffffu;
        // U^2 as seed_bound: the corners dealt over the shares
        float mx = 0.0f;
        if (found) tri_verts(a.m, seed, va, vb, vc);
        for (uint32_t k = share; k < 8u && found; k += shares)
            mx = fmaxf(mx, tri_distance_sq(va, vb, vc, v3(k & 1 ? hi.x : lo.x, k & 2 ? hi.y : lo.y, k & 4 ? hi.z : lo.z)));
        s_w[tid] = __float_as_uint(mx);
        __syncthreads();
        for (uint32_t q = 0; q < min(shares, 8u); ++q) mx = fmaxf(mx, __uint_as_float(s_w[q * S3 + sub]));
        const float U2 = mx * (1.0f + 0x1p-10f) + 0x1p-40f;
        uint32_t mine = 0;  // candidates of this share within the bound, the seed apart
        for (uint32_t q = share; q < n_cand && found; q += shares) {
            float4 tlo, thi;
            box(q, tlo, thi);
            if (box_box_sq(lo, hi, tlo, thi) <= U2) mine += s_tri[q] != seed ? 1u : 0u;
        }
        __syncthreads();  // (s_u, s_v, s_w are free)
        s_u[tid] = mine;
        __syncthreads();
        uint32_t count = found ? 1u : 0u, before = 1;
        for (uint32_t q = 0; q < shares; ++q) {
            const uint32_t c = s_u[q * S3 + sub];
            count += c;
            if (q < share) before += c;
        }
        // the sub-cells' entries: one claim for the workgroup, then each one's offset
        if (share == 0) s_v[sub] = count;
        __syncthreads();
        if (wave == 0) {
            const uint32_t c = lane < S3 ? s_v[lane] : 0u;
            uint32_t incl = c;
#pragma unroll
            for (uint32_t o = 1; o < 64u; o <<= 1) {
                const uint32_t up = __shfl_up(incl, o);
                if (lane >= o) incl += up;
            }
            if (lane == 63u) s_base = claim_entries(a.state, incl);
            if (lane < S3) s_w[lane] = incl - c;
        }
        __syncthreads();
        const uint64_t off = s_base + s_w[sub];
        uint2 hd = make_uint2(0u, kNoList);
        if (found && count <= kMaxList && off + count <= a.ent_cap)
            hd = make_uint2((uint32_t)off, count | (seed << 16));
        if (share == 0) {
            a.head[(size_t)rank * S3 + sub] = hd;
            if (hd.y == kNoList) atomicAdd(&a.state[4], 1u);
        }
        if (hd.y != kNoList) {
            uint32_t* e = a.ent + off;
            if (share == 0) e[0] = seed;  // box distance 0: scanned first
            uint32_t k = before;
            for (uint32_t q = share; q < n_cand; q += shares) {
                float4 tlo, thi;
                box(q, tlo, thi);
                const float d2 = box_box_sq(lo, hi, tlo, thi);
                const uint32_t t = s_tri[q];
                if (d2 <= U2 && t != seed) e[k++] = (__float_as_uint(d2) & 0xffff0000u) | t;
            }
        }
        __syncthreads();  // the next cell reuses the LDS lists
    }
}

// Whether the per-lane kernels walk the cell of this rank.  They visit the cells
// in rank order and pass over the others: neighbouring waves then walk
// neighbouring cells, whose nodes and triangles the CU's cache still holds (in
// the order the cells were left in, a 32^3 grid of 1,109 cells took 7,700 us
// to build, 7,080 in rank order; all cells one lane per sub-cell, 6,600: the
// cells left here, of over 3,072 candidates, set the time either way).
INSTA_DEV bool walked(const ClArgs& a, uint32_t rank) { return a.all || a.walk[rank]; }

__global__ __launch_bounds__(kClThreads) void cl_count_kernel(ClArgs a) {
    extern __shared__ uint32_t stack[];  // [stack_depth(k)][kClThreads]
    const uint32_t S3 = a.S * a.S * a.S;
    const uint32_t n_sub = min(a.state[0], a.cap) * S3;
    for (uint32_t i = blockIdx.x * kClThreads + threadIdx.x; i < n_sub; i += gridDim.x * kClThreads) {
        const uint32_t rank = i / S3;
        if (!walked(a, rank)) continue;
        float4 lo, hi;
        sub_box(a, a.cells[rank], i % S3, lo, hi);
        const V3 ctr = v3((lo.x + hi.x) * 0.5f, (lo.y + hi.y) * 0.5f, (lo.z + hi.z) * 0.5f);
        const Hit h = bvh_closest(a.m, ctr, stack + threadIdx.x, kClThreads);
        uint2 hd = make_uint2(0u, kNoList);
        if (h.idx >= 0) {
            const float U2 = seed_bound(a.m, (uint32_t)h.idx, lo, hi);
            const uint32_t seed = (uint32_t)h.idx;
            uint32_t count = 1;  // the seed, then every other triangle of the walk
            bvh_range(a.m, lo, hi, U2, stack + threadIdx.x, kClThreads,
                      [&](uint32_t t, float) { count += t != seed ? 1u : 0u; });
            const uint64_t off = claim_entries(a.state, count);
            if (count <= kMaxList && off + count <= a.ent_cap)
                hd = make_uint2((uint32_t)off, count | ((uint32_t)h.idx << 16));
        }
        if (hd.y == kNoList) atomicAdd(&a.state[4], 1u);
        a.head[i] = hd;
    }
}

__global__ __launch_bounds__(kClThreads) void cl_fill_kernel(ClArgs a) {
    extern __shared__ uint32_t stack[];  // [stack_depth(k)][kClThreads]
    const uint32_t S3 = a.S * a.S * a.S;
    const uint32_t n_sub = min(a.state[0], a.cap) * S3;
    for (uint32_t i = blockIdx.x * kClThreads + threadIdx.x; i < n_sub; i += gridDim.x * kClThreads) {
        const uint32_t rank = i / S3;
        if (!walked(a, rank)) continue;
        const uint2 hd = a.head[i];
        if (hd.y == kNoList) continue;
        const uint32_t count = hd.y & 0xffffu, seed = hd.y >> 16;
        float4 lo, hi;
        sub_box(a, a.cells[rank], i % S3, lo, hi);
        const float U2 = seed_bound(a.m, seed, lo, hi);
        uint32_t* e = a.ent + hd.x;
        e[0] = seed;  // box distance 0: scanned first
        uint32_t k = 1;
        bvh_range(a.m, lo, hi, U2, stack + threadIdx.x, kClThreads, [&](uint32_t t, float d2) {
            if (t != seed && k < count) e[k++] = (__float_as_uint(d2) & 0xffff0000u) | t;
        });
    }
}

// Sort each list's entries after the seed by key (truncated box distance,
// then triangle): one wave per sub-cell ranks the keys by counting the smaller
// ones (keys are distinct), then writes them to their ranks.  The keys are
// read from memory once, into registers (key q of lane l is entry l + 64 q);
// the counting pass broadcasts them from there lane by lane (readlane), so it
// issues no memory reads.  Every store follows all of the wave's loads, so no
// entry is overwritten before it is read.  Most lists have at most 64 keys
// (31 on average on the 9,976-triangle head): they take one key per lane and
// straight-line steps of eight; the next list's head is loaded meanwhile.
// 544,000 lists of the head: 248 us, with the eight-key loop for all 824.
__global__ __launch_bounds__(kClThreads) void cl_sort_kernel(ClArgs a) {
    const uint32_t S3 = a.S * a.S * a.S;
    const uint32_t n_sub = min(a.state[0], a.cap) * S3;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t n_waves = gridDim.x * (kClThreads / 64u);
    uint32_t i = blockIdx.x * (kClThreads / 64u) + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64u));
    uint2 next = i < n_sub ? a.head[i] : make_uint2(0u, kNoList);
    for (; i < n_sub; i += n_waves) {
        const uint2 hd = next;
        if (i + n_waves < n_sub) next = a.head[i + n_waves];
        if (hd.y == kNoList) continue;
        const uint32_t n = (hd.y & 0xffffu) - 1u;
        uint32_t* e = a.ent + hd.x + 1u;
        if (n <= 64u) {
            const uint32_t key = lane < n ? e[lane] : 0xffffffffu;
            uint32_t rank = 0;
            for (uint32_t l0 = 0; l0 < n; l0 += 8u) {  // lanes past n hold no smaller key
#pragma unroll
                for (uint32_t l = 0; l < 8u; ++l)
                    rank += (uint32_t)__builtin_amdgcn_readlane((int)key, (int)(l0 + l)) < key ? 1u : 0u;
            }
            if (lane < n) e[rank] = key;
            continue;
        }
        uint32_t key[kSortPerLane], rank[kSortPerLane];
#pragma unroll
        for (uint32_t q = 0; q < kSortPerLane; ++q) {
            const uint32_t x = lane + 64u * q;
            key[q] = x < n ? e[x] : 0xffffffffu;
            rank[q] = 0u;
        }
        const uint32_t nq = (n + 63u) / 64u;  // key slots in use (wave-uniform)
#pragma unroll
        for (uint32_t qs = 0; qs < kSortPerLane; ++qs) {
            if (qs >= nq) break;
            const uint32_t cnt = min(64u, n - 64u * qs);
            for (uint32_t l = 0; l < cnt; ++l) {
                const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)key[qs], (int)l);
#pragma unroll
                for (uint32_t q = 0; q < kSortPerLane; ++q)
                    if (q < nq) rank[q] += v < key[q] ? 1u : 0u;
            }
        }
#pragma unroll
        for (uint32_t q = 0; q < kSortPerLane; ++q)
            if (lane + 64u * q < n) e[rank[q]] = key[q];
    }
}

__global__ void cl_finish_kernel(uint32_t* __restrict__ state) {
    if (threadIdx.x != 0) return;
    state[1] = state[kClClaim + 1] ? 0xffffffffu : state[kClClaim];
    state[2] = state[3] == 0u ? 1u : 0u;
}

ClArgs cl_args(insta_ctx* ctx, uint32_t slot) {
    ClArgs a;
    const size_t G = ctx->cfg.grid_size, S = ctx->cfg.cell_split;
    a.m = ctx->mesh(slot);
    a.cells = ctx->d_cl_cells + slot * (size_t)ctx->cfg.cell_list_cells;
    a.head = ctx->d_cl_head + slot * (size_t)ctx->cfg.cell_list_cells * S * S * S;
    a.ent = ctx->d_cl_ent + slot * (size_t)ctx->cfg.cell_list_entries;
    a.state = ctx->d_cl_state + kClState * (size_t)slot;
    a.left = ctx->d_cl_left + 2 * slot * (size_t)ctx->cfg.cell_list_cells;
    a.walk = a.left + ctx->cfg.cell_list_cells;
    // a workgroup per cell pays for 64 sub-cells, not for 8 or 1: the small
    // sphere at S = 2 takes 230 + 150 us one lane per sub-cell, 920 us so
    a.all = S == 4 ? 0u : 1u;
    a.G = (uint32_t)G;
    a.S = (uint32_t)S;
    a.cap = ctx->cfg.cell_list_cells;
    a.ent_cap = ctx->cfg.cell_list_entries;
    return a;
}

}  // namespace

insta_status alloc_cell_lists(insta_ctx* ctx) {
    if (ctx->cfg.cell_split == 0) return INSTA_OK;
    const size_t n = ctx->n_slots, G = ctx->cfg.grid_size, S = ctx->cfg.cell_split;
    const size_t words = G * G * G / 64;
    const size_t cells = ctx->cfg.cell_list_cells, ents = ctx->cfg.cell_list_entries;
    bool ok = true;
    auto alloc = [&](void** p, size_t bytes) {
        if (ok && hipMalloc(p, bytes) != hipSuccess) ok = false;
    };
    alloc((void**)&ctx->d_cl_bits, n * words * sizeof(uint64_t));
    alloc((void**)&ctx->d_cl_rank, n * words * sizeof(uint32_t));
    alloc((void**)&ctx->d_cl_cells, n * cells * sizeof(uint32_t));
    alloc((void**)&ctx->d_cl_left, 2 * n * cells * sizeof(uint32_t));
    alloc((void**)&ctx->d_cl_head, n * cells * S * S * S * sizeof(uint2));
    alloc((void**)&ctx->d_cl_ent, n * ents * sizeof(uint32_t));
    alloc((void**)&ctx->d_cl_state, n * kClState * sizeof(uint32_t));
    if (!ok) {
        free_cell_lists(ctx);
        set_error("device allocation of the candidate lists failed (lower cell_list_cells / cell_list_entries)");
        return INSTA_ERR_OOM;
    }
    // every slot starts without lists
    if (hipMemset(ctx->d_cl_state, 0, n * kClState * sizeof(uint32_t)) != hipSuccess) {
        free_cell_lists(ctx);
        set_error("candidate list state initialisation failed");
        return INSTA_ERR_HIP;
    }
    return INSTA_OK;
}

void free_cell_lists(insta_ctx* ctx) {
    dev_free(ctx->d_cl_bits);
    dev_free(ctx->d_cl_rank);
    dev_free(ctx->d_cl_cells);
    dev_free(ctx->d_cl_left);
    dev_free(ctx->d_cl_head);
    dev_free(ctx->d_cl_ent);
    dev_free(ctx->d_cl_state);
}

insta_status launch_cell_lists_invalidate(insta_ctx* ctx, uint32_t first, uint32_t n, hipStream_t stream) {
    if (!ctx->d_cl_state || n == 0) return INSTA_OK;
    hipLaunchKernelGGL(cl_invalidate_kernel, dim3((n + 255) / 256), dim3(256), 0, stream,
                       ctx->d_cl_state + kClState * first, n);
    INSTA_HIP(hipGetLastError());
    return INSTA_OK;
}

insta_status launch_cell_lists(insta_ctx* ctx, uint32_t slot, hipStream_t stream) {
    if (!ctx->d_cl_state) return INSTA_OK;
    const ClArgs a = cl_args(ctx, slot);
    const size_t G = ctx->cfg.grid_size;
    const uint32_t n_words = (uint32_t)(G * G * G / 64);
    uint64_t* bits = ctx->d_cl_bits + slot * (size_t)n_words;
    uint32_t* rank = ctx->d_cl_rank + slot * (size_t)n_words;
    const uint64_t* lin = reinterpret_cast<const uint64_t*>(ctx->grid_lin(slot));
    hipLaunchKernelGGL(cl_begin_kernel, dim3(1), dim3(64), 0, stream, a.state);
    hipLaunchKernelGGL(cl_words_kernel, dim3((n_words + 255) / 256), dim3(256), 0, stream, lin, n_words, bits, rank);
    hipLaunchKernelGGL(cl_scan_kernel, dim3(1), dim3(kScanThreads), 0, stream, rank, n_words, a.cap, a.state);
    hipLaunchKernelGGL(cl_cells_kernel, dim3((n_words + 255) / 256), dim3(256), 0, stream, bits, rank, n_words, a.cap,
                       ctx->d_cl_cells + slot * (size_t)ctx->cfg.cell_list_cells);
    const size_t shmem = (size_t)stack_depth(ctx->bvh_k) * kClThreads * sizeof(uint32_t);
    const uint64_t max_sub = (uint64_t)a.cap * a.S * a.S * a.S;
    // (after the per-cell kernels most lanes pass over their cell)
    const uint32_t blocks =
        (uint32_t)std::min<uint64_t>((max_sub + kClThreads - 1) / kClThreads, a.all ? kClMaxBlocks : 1024u);
    if (!a.all) {
        hipLaunchKernelGGL(cl_cell_kernel<false>, dim3(std::min(a.cap, kClMaxBlocks)), dim3(kCellThreads), 0, stream, a);
        hipLaunchKernelGGL(cl_cell_kernel<true>, dim3(std::min(a.cap, 512u)), dim3(kCellThreads2), 0, stream, a);
    }
    hipLaunchKernelGGL(cl_count_kernel, dim3(blocks), dim3(kClThreads), shmem, stream, a);
    hipLaunchKernelGGL(cl_fill_kernel, dim3(blocks), dim3(kClThreads), shmem, stream, a);
    hipLaunchKernelGGL(cl_sort_kernel, dim3(kClMaxBlocks), dim3(kClThreads), 0, stream, a);
    hipLaunchKernelGGL(cl_finish_kernel, dim3(1), dim3(64), 0, stream, a.state);
    INSTA_HIP(hipGetLastError());
    return INSTA_OK;
}

insta_status launch_mesh_occupancy(insta_ctx* ctx, uint32_t slot, float threshold, hipStream_t stream) {
    insta_status st = launch_occupancy(ctx, slot, threshold, stream);
    if (st != INSTA_OK) return st;
    st = launch_grid_linear(ctx, slot, stream);
    if (st != INSTA_OK) return st;
    return launch_cell_lists(ctx, slot, stream);
}

}  // namespace insta
