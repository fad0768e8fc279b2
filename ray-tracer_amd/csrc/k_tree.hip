// k_tree.hip -- triangle tree: construction and per-ray traversal (gfx950).
//
// Results are those of the reference's traversal and intersection
// (projects/CUDA-Engine/source/RayTracer.cu:1152-1614, 1711-1774): a ray's
// hit is the closest (or any) triangle that the ray-triangle test accepts and
// that is a candidate of the ray's chain of hierarchy nodes -- its object's
// sphere passes the top node, and its own sphere every node down to the leaf.
// The tests of one (ray, triangle) pair commute, so the tree finds the
// triangles that the ray test accepts and the node tests run only on those
// that would improve the ray's result, instead of on every pair.
//
// The tree is a four-wide bounding-box tree: a binary tree merged bottom up
// over the triangles in Morton order, from which each wide node takes the
// children of the largest surface.  It is rebuilt on the device at scene load
// and after object updates (262,604 triangles: 0.35 ms, bound by the
// latency of its 26 launches and of the merging rounds).
#include <algorithm>
#include <cmath>
#include <utility>

#include "rsh_kernels.hpp"

namespace rsh {

namespace {

constexpr uint32_t TREE_LEAF = 4;              // triangles per leaf
constexpr uint32_t TREE_EMPTY = 0xFFFFFFFFu;
constexpr uint32_t TREE_IS_LEAF = 0x80000000u; // child word: leaf flag, (count - 1) << 29, first record
constexpr uint32_t CODE_BITS = 9;              // Morton code bits per axis (three sorting passes)

inline uint32_t grid_for(uint64_t n, uint32_t block) {
    const uint64_t g = (n + block - 1) / block;
    return g ? (uint32_t)g : 1u;
}

// Order-preserving map of floats to unsigned words (atomicMin / atomicMax).
__device__ __forceinline__ uint32_t ordered(float f) {
    const uint32_t b = __float_as_uint(f);
    return (b >> 31) ? ~b : b | 0x80000000u;
}
__device__ __forceinline__ float unordered(uint32_t u) {
    return __uint_as_float((u >> 31) ? u & 0x7FFFFFFFu : ~u);
}

__device__ __forceinline__ float wave_min_f(float x) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) x = fminf(x, __shfl_xor(x, d, 64));
    return x;
}
__device__ __forceinline__ float wave_max_f(float x) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) x = fmaxf(x, __shfl_xor(x, d, 64));
    return x;
}

__device__ __forceinline__ float half_surface(float4 lo, float4 hi) {
    const float x = hi.x - lo.x, y = hi.y - lo.y, z = hi.z - lo.z;
    return x * y + y * z + z * x;
}

// bounds: ordered words of the scene box (lo xyz, hi xyz) and the largest
// triangle-sphere radius.
__global__ void k_tree_clear(uint32_t* bounds) {
    if (threadIdx.x < 3) bounds[threadIdx.x] = ordered(INFINITY);
    else if (threadIdx.x < 6) bounds[threadIdx.x] = ordered(-INFINITY);
    else if (threadIdx.x == 6) bounds[6] = ordered(0.0f);
}

// Box of triangle t: every ray that both the line test against its bounding
// sphere (ray_may_hit_sphere) and ray_triangle accept meets it once it is
// widened by the ray's margin (k_tree_trace).  ray_triangle's FP32 acceptance
// holds the line to the triangle except where the ray is nearly parallel to
// its plane: there u, v and t may be off along the plane by any amount, but
// the line still runs within ~5e-7 |tvec| / sin(e1, e2) of the plane where it
// passes the triangle's sphere.  The box therefore covers the triangle and the
// disc that its plane cuts from the sphere; a triangle with sin(e1, e2) < 0.02
// (no reliable plane) the whole sphere.  A non-finite triangle is never hit
// (every term of the test becomes NaN) and gets an empty box.
// The bounds' atomics all go to one line, at about 12 ns each: a block of 1024
// adds its own, and there are 64 (262,604 triangles: 330 us with seven atomics
// a wave, 12 so).
constexpr uint32_t PRIM_BLOCKS = 64;
__global__ void __launch_bounds__(1024) k_tree_prims(const float4* tri_sphere, const float4* tri_mt, uint32_t T,
                                                    float4* box, uint32_t* bounds, float* area) {
    __shared__ uint32_t s_bounds[7];
    __shared__ float s_area[16];
    if (threadIdx.x < 7) s_bounds[threadIdx.x] = threadIdx.x < 3 ? ordered(INFINITY) : threadIdx.x < 6 ? ordered(-INFINITY) : ordered(0.0f);
    __syncthreads();
    v3 all_lo = mk(INFINITY, INFINITY, INFINITY), all_hi = mk(-INFINITY, -INFINITY, -INFINITY);
    float all_r = 0.0f, sum = 0.0f;
    for (uint32_t t = blockIdx.x * 1024 + threadIdx.x; t < T; t += gridDim.x * 1024) {
        v3 lo = mk(INFINITY, INFINITY, INFINITY), hi = mk(-INFINITY, -INFINITY, -INFINITY);
        const v3 a = xyz(tri_mt[3 * (size_t)t]), e1 = xyz(tri_mt[3 * (size_t)t + 1]), e2 = xyz(tri_mt[3 * (size_t)t + 2]);
        const float4 s = tri_sphere[t];
        const v3 n = cross(e1, e2);
        const float nn = dot(n, n), ll = dot(e1, e1) * dot(e2, e2);
        const bool plane = nn > 4e-4f * ll && nn > 1e-30f;
        const float inv = plane ? 1.0f / nn : 0.0f;
        // half-extent of the disc on an axis: r sqrt(1 - n_axis^2 / |n|^2), widened for its rounding
        const float hx = s.w * fminf(1.0f, sqrtf(fmaxf(0.0f, 1.0f - n.x * n.x * inv)) + 2e-3f);
        const float hy = s.w * fminf(1.0f, sqrtf(fmaxf(0.0f, 1.0f - n.y * n.y * inv)) + 2e-3f);
        const float hz = s.w * fminf(1.0f, sqrtf(fmaxf(0.0f, 1.0f - n.z * n.z * inv)) + 2e-3f);
        const v3 b = a + e1, c = a + e2;
        const v3 l = mk(fminf(fminf(a.x, fminf(b.x, c.x)), s.x - hx), fminf(fminf(a.y, fminf(b.y, c.y)), s.y - hy),
                        fminf(fminf(a.z, fminf(b.z, c.z)), s.z - hz));
        const v3 h = mk(fmaxf(fmaxf(a.x, fmaxf(b.x, c.x)), s.x + hx), fmaxf(fmaxf(a.y, fmaxf(b.y, c.y)), s.y + hy),
                        fmaxf(fmaxf(a.z, fmaxf(b.z, c.z)), s.z + hz));
        const float all = ((a.x + a.y) + a.z) + ((e1.x + e1.y) + e1.z) + ((e2.x + e2.y) + e2.z) + ((s.x + s.y) + s.z) + s.w;
        if (isfinite(all)) {
            lo = l; hi = h;
            all_lo = mk(fminf(all_lo.x, l.x), fminf(all_lo.y, l.y), fminf(all_lo.z, l.z));
            all_hi = mk(fmaxf(all_hi.x, h.x), fmaxf(all_hi.y, h.y), fmaxf(all_hi.z, h.z));
            all_r = fmaxf(all_r, s.w);
            sum += half_surface(f4(l, 0.0f), f4(h, 0.0f));
        }
        box[2 * (size_t)t] = f4(lo, 0.0f);
        box[2 * (size_t)t + 1] = f4(hi, 0.0f);
    }
    const float m[7] = {wave_min_f(all_lo.x), wave_min_f(all_lo.y), wave_min_f(all_lo.z),
                        wave_max_f(all_hi.x), wave_max_f(all_hi.y), wave_max_f(all_hi.z), wave_max_f(all_r)};
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d, 64);
    if ((threadIdx.x & 63u) == 0) {
        s_area[threadIdx.x >> 6] = sum;
#pragma unroll
        for (int i = 0; i < 3; i++) atomicMin(&s_bounds[i], ordered(m[i]));
#pragma unroll
        for (int i = 3; i < 7; i++) atomicMax(&s_bounds[i], ordered(m[i]));
    }
    __syncthreads();
    if (threadIdx.x < 3) atomicMin(&bounds[threadIdx.x], s_bounds[threadIdx.x]);
    else if (threadIdx.x < 7) atomicMax(&bounds[threadIdx.x], s_bounds[threadIdx.x]);
    else if (threadIdx.x == 7) {
        float all = 0.0f;
        for (uint32_t i = 0; i < 16; i++) all += s_area[i];
        area[blockIdx.x] = all;
    }
}

__device__ __forceinline__ uint32_t spread10(uint32_t x) {
    x = (x | (x << 16)) & 0x030000FFu;
    x = (x | (x << 8)) & 0x0300F00Fu;
    x = (x | (x << 4)) & 0x030C30C3u;
    return (x | (x << 2)) & 0x09249249u;
}

// Morton code of the box centre over the scene box.
__global__ void __launch_bounds__(256) k_tree_codes(const float4* box, uint32_t T, const uint32_t* bounds,
                                                    uint32_t* codes, uint32_t* ids) {
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t >= T) return;
    const v3 c = (xyz(box[2 * (size_t)t]) + xyz(box[2 * (size_t)t + 1])) * 0.5f;
    const v3 lo = mk(unordered(bounds[0]), unordered(bounds[1]), unordered(bounds[2]));
    const v3 hi = mk(unordered(bounds[3]), unordered(bounds[4]), unordered(bounds[5]));
    const v3 ex = hi - lo;
    auto q = [](float x, float l, float e) { return min(f2u(((x - l) / e) * (float)(1u << CODE_BITS)), (1u << CODE_BITS) - 1u); };   // NaN -> 0
    codes[t] = (spread10(q(c.z, lo.z, ex.z)) << 2) | (spread10(q(c.y, lo.y, ex.y)) << 1) | spread10(q(c.x, lo.x, ex.x));
    ids[t] = t;
}

// The binary tree, bottom up: clusters in Morton order, of which in each round
// every two that are one another's best partner -- the union of the smallest
// surface within MERGE_RADIUS places -- become one (parallel locally ordered
// clustering, Meister and Bittner 2018).  Against the radix tree over the same
// codes a ray takes 16 to 32 % fewer node steps and as many or fewer leaf steps
// (camera and diffuse rays; shadow rays' change little), and radius 8 or 16 is no
// better than 4: office camera pass 0.58 -> 0.48 ms, soft-shadow frame 3.14 ->
// 2.97, 1M diffuse rays 0.741 -> 0.678, 16-view batch 7.86 -> 7.64.
// A workgroup merges MERGE_CHUNK neighbouring clusters in LDS down to a
// sixteenth, the next launch what 16 workgroups have left, until one is left:
// three launches for 262,604 triangles with 10, 10 and 24 rounds, where a
// launch a round would take 42 and a compaction each (the tree's quality is
// the same: a partner is rarely across the chunk's edge).  A round is bound by
// its three barriers.
constexpr uint32_t MERGE_CHUNK = 2048;
constexpr uint32_t MERGE_KEEP = MERGE_CHUNK / 16;
constexpr uint32_t MERGE_RADIUS = 4;
// Rounds of best partners (28 at most seen); then neighbours merge in pairs,
// which bounds the rounds and the tree's depth: MERGE_ROUNDS + 11 a launch.
constexpr uint32_t MERGE_ROUNDS = 40;

// Marks a node that is no leaf: of more than TREE_LEAF triangles, or of fewer
// whose halves have less surface than the whole: a leaf's step costs about four
// of a node's (leaves wherever four triangles fit: 16-view batch 7.80 ms, so
// 7.64; office frame 1.862, 1.847; 1M diffuse rays 0.668, 0.678).
constexpr uint32_t TREE_SPLIT = 0x80000000u;

struct MergeArgs {
    uint32_t T;
    const uint32_t* ids;         // triangles in Morton order
    const float4* box;           // triangle boxes
    const uint32_t* in;          // later launches: MERGE_KEEP slots for each workgroup of the one before,
    const uint32_t* in_count;    // and how many of them are used
    uint32_t in_groups;
    uint32_t* out;
    uint32_t* out_count;
    uint32_t base;               // nodes of this launch: MERGE_CHUNK for each workgroup from here on
    float4* node;                // node i < T: i-th triangle in Morton order; (lo, left child), (hi, right child)
    uint32_t* size;              // triangles below a node >= T, and TREE_SPLIT
    const float* area;           // half surfaces of the triangles' boxes, summed by each of area_blocks blocks
    uint32_t area_blocks;
    TreeMeasure* measure;        // written by the last launch
    bool last;
};

template <bool FIRST>
__global__ void __launch_bounds__(1024) k_tree_merge(MergeArgs A) {
    __shared__ float s_box[6][MERGE_CHUNK];
    __shared__ uint32_t s_id[MERGE_CHUNK], s_size[MERGE_CHUNK];
    __shared__ uint16_t s_best[MERGE_CHUNK];
    __shared__ uint32_t s_sum[32];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    uint32_t n = 0;
    auto load = [&](uint32_t at, uint32_t id, uint32_t size, float4 lo, float4 hi) {
        s_box[0][at] = lo.x; s_box[1][at] = lo.y; s_box[2][at] = lo.z;
        s_box[3][at] = hi.x; s_box[4][at] = hi.y; s_box[5][at] = hi.z;
        s_id[at] = id; s_size[at] = size;
    };
    auto surface = [&](uint32_t i) {
        return half_surface(make_float4(s_box[0][i], s_box[1][i], s_box[2][i], 0.0f),
                            make_float4(s_box[3][i], s_box[4][i], s_box[5][i], 0.0f));
    };
    if (FIRST) {
        const uint32_t p0 = blockIdx.x * MERGE_CHUNK;
        n = min(MERGE_CHUNK, A.T - p0);
        for (uint32_t i = tid; i < n; i += 1024) {
            const size_t t = A.ids[p0 + i];
            const float4 lo = A.box[2 * t], hi = A.box[2 * t + 1];
            A.node[2 * (size_t)(p0 + i)] = lo;
            A.node[2 * (size_t)(p0 + i) + 1] = hi;
            load(i, p0 + i, 1u, lo, hi);
        }
    } else {
        const uint32_t g0 = blockIdx.x * 16;
        for (uint32_t slot = tid; slot < MERGE_CHUNK; slot += 1024) {
            const uint32_t g = slot / MERGE_KEEP, k = slot % MERGE_KEEP;
            uint32_t before = 0, mine = 0, all = 0;
            for (uint32_t i = 0; i < 16; i++) {
                const uint32_t c = g0 + i < A.in_groups ? A.in_count[g0 + i] : 0u;
                before += i < g ? c : 0u;
                mine = i == g ? c : mine;
                all += c;
            }
            n = all;
            if (k < mine) {
                const uint32_t id = A.in[(size_t)(g0 + g) * MERGE_KEEP + k];
                load(before + k, id, id < A.T ? 1u : A.size[id] & ~TREE_SPLIT, A.node[2 * (size_t)id], A.node[2 * (size_t)id + 1]);
            }
        }
    }
    __syncthreads();
    const uint32_t target = A.last ? 1u : max(1u, n / 16);
    uint32_t next = A.base + blockIdx.x * MERGE_CHUNK;
    for (uint32_t round = 0; n > target; round++) {
        for (uint32_t i = tid; i < n; i += 1024) {
            // Of equal surfaces the neighbour i ^ 1 comes first, then the lower
            // place: an order of the pairs, so the first pair of all chooses one
            // another and every round merges.  (Infinite and NaN surfaces are
            // never chosen; where none is finite, neighbours pair up.)
            const uint32_t next_to = (i ^ 1u) < n ? i ^ 1u : i - 1u;
            uint32_t best = next_to;
            if (round < MERGE_ROUNDS) {
                const float lx = s_box[0][i], ly = s_box[1][i], lz = s_box[2][i];
                const float hx = s_box[3][i], hy = s_box[4][i], hz = s_box[5][i];
                auto area = [&](uint32_t j) {
                    return half_surface(
                        make_float4(fminf(lx, s_box[0][j]), fminf(ly, s_box[1][j]), fminf(lz, s_box[2][j]), 0.0f),
                        make_float4(fmaxf(hx, s_box[3][j]), fmaxf(hy, s_box[4][j]), fmaxf(hz, s_box[5][j]), 0.0f));
                };
                float least = area(next_to);
                if (!(least < INFINITY)) least = INFINITY;
                const uint32_t j1 = min(n - 1, i + MERGE_RADIUS);
                for (uint32_t j = i > MERGE_RADIUS ? i - MERGE_RADIUS : 0u; j <= j1; j++) {
                    const float c = area(j);
                    if (j != i && c < least) { least = c; best = j; }
                }
            } else {
                best = (i ^ 1u) < n ? i ^ 1u : i;
            }
            s_best[i] = (uint16_t)best;
        }
        __syncthreads();
        float4 lo[2], hi[2];
        uint32_t id[2], size[2], kid[2];
        bool split[2];
        unsigned long long kept[2], merged[2];
#pragma unroll
        for (uint32_t e = 0; e < 2; e++) {
            const uint32_t i = tid + e * 1024;
            bool keep = false, merge = false;
            if (i < n) {
                const uint32_t m = s_best[i];
                const bool pair = m != i && s_best[m] == i;
                keep = !pair || i < m;
                merge = pair && i < m;
                if (keep) {
                    const uint32_t o = merge ? m : i;
                    lo[e] = make_float4(fminf(s_box[0][i], s_box[0][o]), fminf(s_box[1][i], s_box[1][o]), fminf(s_box[2][i], s_box[2][o]), 0.0f);
                    hi[e] = make_float4(fmaxf(s_box[3][i], s_box[3][o]), fmaxf(s_box[4][i], s_box[4][o]), fmaxf(s_box[5][i], s_box[5][o]), 0.0f);
                    id[e] = s_id[i];
                    kid[e] = s_id[o];
                    size[e] = s_size[i] + (merge ? s_size[o] : 0u);
                    split[e] = size[e] > TREE_LEAF || surface(i) + surface(o) < half_surface(lo[e], hi[e]);
                }
            }
            kept[e] = __ballot(keep);
            merged[e] = __ballot(merge);
            if (lane == 0) s_sum[e * 16 + wave] = (uint32_t)__popcll(kept[e]) | (uint32_t)__popcll(merged[e]) << 16;
        }
        __syncthreads();       // sums written, and every read of the clusters done
        uint32_t incl = lane < 32 ? s_sum[lane] : 0u;
#pragma unroll
        for (uint32_t d = 1; d < 32; d <<= 1) {
            const uint32_t up = (uint32_t)__shfl_up((int)incl, d, 64);
            incl += lane >= d ? up : 0u;
        }
        const uint32_t total = (uint32_t)__shfl((int)incl, 31, 64);
        const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
        for (uint32_t e = 0; e < 2; e++) {
            const uint32_t slot = e * 16 + wave;
            const uint32_t upto = (uint32_t)__shfl((int)incl, (int)slot, 64);
            if (kept[e] >> lane & 1ull) {
                const uint32_t k0 = (upto & 0xFFFFu) - (uint32_t)__popcll(kept[e]);
                const uint32_t m0 = (upto >> 16) - (uint32_t)__popcll(merged[e]);
                uint32_t me = id[e];
                if (merged[e] >> lane & 1ull) {
                    me = next + m0 + (uint32_t)__popcll(merged[e] & below);
                    A.node[2 * (size_t)me] = make_float4(lo[e].x, lo[e].y, lo[e].z, __uint_as_float(id[e]));
                    A.node[2 * (size_t)me + 1] = make_float4(hi[e].x, hi[e].y, hi[e].z, __uint_as_float(kid[e]));
                    A.size[me] = size[e] | (split[e] ? TREE_SPLIT : 0u);
                }
                load(k0 + (uint32_t)__popcll(kept[e] & below), me, size[e], lo[e], hi[e]);
            }
        }
        n = total & 0xFFFFu;
        next += total >> 16;
        __syncthreads();
    }
    for (uint32_t i = tid; i < n; i += 1024) A.out[(size_t)blockIdx.x * MERGE_KEEP + i] = s_id[i];
    if (tid == 0) A.out_count[blockIdx.x] = n;
    if (A.last && tid < 64) {
        float sum = tid < A.area_blocks ? A.area[tid] : 0.0f;
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d, 64);
        if (tid == 0) {
            const float root = surface(0);
            *A.measure = TreeMeasure{sum / root, root};
        }
    }
}

// Wide node w, built from a binary node: the child of the largest surface is
// replaced by its two children until there are four or only leaves are left.  Its inner children become the next level's
// wide nodes at `next` on, as counted in *count.  Triangles take the order of
// the children; k_tree_records fills the leaves when all nodes are there (a
// level is a chain of loads that other XCDs have written: 21 us a level with
// the leaves in it, 14 without).
struct EmitArgs {
    uint32_t T;
    const float4* node;
    const uint32_t* size;
    const uint32_t* root;
    uint2* queue;           // (binary node, its first place in tree order) of every wide node, in breadth-first order
    uint32_t* count;        // wide nodes per level, then their number
    TreeNode* nodes;        // (hi of a child: .w its binary node)
};
constexpr uint32_t TREE_LEVELS = 320;      // deeper than six merging launches can make it

__device__ void emit_node(const EmitArgs& A, uint32_t w, uint32_t next, uint32_t* count) {
    uint32_t id[4], size[4];
    float4 lo[4], hi[4];
    float area[4];          // of a child that can be split, else -1
    uint32_t n = 0;
    auto put = [&](uint32_t k, uint32_t c) {
        const float4* b = A.node + 2 * (size_t)c;
        id[k] = c; lo[k] = b[0]; hi[k] = b[1];
        size[k] = c < A.T ? 1u : A.size[c];
        area[k] = size[k] & TREE_SPLIT ? fmaxf(half_surface(lo[k], hi[k]), 0.0f) : -1.0f;     // NaN -> 0
    };
    const uint2 of = A.queue[w];
    put(0, __float_as_uint(A.node[2 * (size_t)of.x].w));
    put(1, __float_as_uint(A.node[2 * (size_t)of.x + 1].w));
    n = 2;
    for (; n < 4; n++) {
        uint32_t k = 0;
#pragma unroll
        for (uint32_t i = 1; i < 4; i++)
            if (i < n && area[i] > area[k]) k = i;
        if (area[k] < 0.0f) break;
        const uint32_t left = __float_as_uint(lo[k].w), right = __float_as_uint(hi[k].w);
        put(k, left); put(n, right);
    }
    uint32_t inner = 0;
    for (uint32_t k = 0; k < n; k++) inner += size[k] >> 31;
    uint32_t at = inner ? next + atomicAdd(count, inner) : 0u;
    uint32_t first = of.y;
    TreeNode out;
    for (uint32_t k = 0; k < 4; k++) {
        uint32_t word = TREE_EMPTY, from = 0u;
        float4 l = make_float4(INFINITY, INFINITY, INFINITY, 0.0f), h = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
        if (k < n) {
            l = lo[k]; h = hi[k]; from = id[k];
            if (size[k] & TREE_SPLIT) {
                A.queue[at] = make_uint2(id[k], first);
                word = at++;
            } else {
                word = TREE_IS_LEAF | ((size[k] - 1u) << 29) | first;
            }
            first += size[k] & ~TREE_SPLIT;
        }
        out.child[k][0] = make_float4(l.x, l.y, l.z, __uint_as_float(word));
        out.child[k][1] = make_float4(h.x, h.y, h.z, __uint_as_float(from));
    }
    A.nodes[w] = out;
}

// The root, and the level counts cleared.  Up to TREE_LEAF triangles: one leaf.
__global__ void k_tree_root(EmitArgs A) {
    for (uint32_t i = threadIdx.x; i <= TREE_LEVELS; i += blockDim.x)
        A.count[i] = (i == 0 && A.T > TREE_LEAF) || (i == TREE_LEVELS && A.T <= TREE_LEAF) ? 1u : 0u;
    if (threadIdx.x != 0) return;
    const uint32_t root = A.root[0];
    A.queue[0] = make_uint2(root, 0u);
    if (A.T > TREE_LEAF) return;
    TreeNode out;
    for (uint32_t k = 0; k < 4; k++) {
        const uint32_t word = k == 0 ? TREE_IS_LEAF | ((A.T - 1u) << 29) : TREE_EMPTY;
        const v3 l = k == 0 ? xyz(A.node[2 * (size_t)root]) : mk(INFINITY, INFINITY, INFINITY);
        const v3 h = k == 0 ? xyz(A.node[2 * (size_t)root + 1]) : mk(-INFINITY, -INFINITY, -INFINITY);
        out.child[k][0] = f4(l, __uint_as_float(word));
        out.child[k][1] = f4(h, __uint_as_float(root));
    }
    A.nodes[0] = out;
}

// One level of wide nodes.
__global__ void __launch_bounds__(256) k_tree_level(EmitArgs A, uint32_t level) {
    uint32_t start = 0;
    for (uint32_t k = 0; k < level; k++) start += A.count[k];
    const uint32_t n = A.count[level];
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
        emit_node(A, start + i, start + n, A.count + level + 1);
}

// The levels from `level` on in one workgroup, until none is left or `last` is
// done.
__global__ void __launch_bounds__(1024) k_tree_tail(EmitArgs A, uint32_t level, uint32_t last) {
    __shared__ uint32_t s_n;
    uint32_t start = 0;
    for (uint32_t k = 0; k < level; k++) start += A.count[k];
    for (; level <= last; level++) {
        __syncthreads();
        if (threadIdx.x == 0) s_n = __hip_atomic_load(A.count + level, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const uint32_t n = s_n;
        if (n == 0u) break;
        for (uint32_t i = threadIdx.x; i < n; i += 1024u) emit_node(A, start + i, start + n, A.count + level + 1);
        __threadfence_block();
        start += n;
    }
    if (threadIdx.x == 0 && last == TREE_LEVELS - 2u) A.count[TREE_LEVELS] = start;
}

// Triangle records in tree order, 64 B each: (sphere), (v0, triangle id),
// (e1, object), (e2, -); a thread for each child of a wide node, which fills a
// leaf's.  ids: triangles in Morton order; objects: (first triangle, ...) of
// each of the K objects, which tile [0, T) in order.
__global__ void __launch_bounds__(256) k_tree_records(EmitArgs A, const uint32_t* ids, const float4* tri_sphere,
                                                      const float4* tri_mt, const uint4* objects, uint32_t K,
                                                      float4* rec) {
    const uint32_t j = blockIdx.x * 256 + threadIdx.x, w = j >> 2;
    if (w >= A.count[TREE_LEVELS]) return;
    const float4* child = A.nodes[w].child[j & 3u];
    const uint32_t word = __float_as_uint(child[0].w);
    if (!(word & TREE_IS_LEAF) || word == TREE_EMPTY) return;
    const uint32_t n = ((word >> 29) & 3u) + 1u, first = word & 0x1FFFFFFFu;
    // the n binary leaves below the child
    uint32_t l[TREE_LEAF] = {__float_as_uint(child[1].w), 0u, 0u, 0u};
    for (uint32_t m = 1; m < n; m++) {
        bool done = false;
#pragma unroll
        for (uint32_t k = 0; k < TREE_LEAF; k++) {
            if (done || k >= m || l[k] < A.T) continue;
            const float4* b = A.node + 2 * (size_t)l[k];
            const uint32_t right = __float_as_uint(b[1].w);
            l[k] = __float_as_uint(b[0].w);
#pragma unroll
            for (uint32_t i = 1; i < TREE_LEAF; i++)
                if (i == m) l[i] = right;
            done = true;
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < TREE_LEAF; k++) {
        if (k >= n) break;
        const uint32_t t = ids[l[k]];
        uint32_t a = 0, b = K;      // objects[a].x <= t < objects[b].x (b = K: end)
        while (b - a > 1) {
            const uint32_t m = (a + b) >> 1;
            if (objects[m].x <= t) a = m; else b = m;
        }
        float4* r = rec + 4 * (size_t)(first + k);
        r[0] = tri_sphere[t];
        r[1] = f4(xyz(tri_mt[3 * (size_t)t]), __uint_as_float(t));
        r[2] = f4(xyz(tri_mt[3 * (size_t)t + 1]), __uint_as_float(a));
        r[3] = f4(xyz(tri_mt[3 * (size_t)t + 2]), 0.0f);
    }
}

// ------------------------------------------------------------- traversal --
// Four lanes per sorted ray (a quad): lane q tests child q of a node or
// triangle q of a leaf; 16 rays, one wave, per workgroup.  Nearest child first;
// the others wait on the ray's stack in LDS.
// Large passes are bound by VALU issue (1080p atrium camera pass: 295M
// instructions, 0.48 ms of issue in 0.52 ms) and the loads behind it, small
// ones by the latency of the longest ray's steps (14k rays: 0.12 ms).  Waves
// hide that latency: 8 a SIMD (64 VGPRs, 11 of the closest-hit kernel's spilled;
// 3.0 / 4.5 KB of LDS) against 7 with 6 KB: 1080p atrium frame 2.97 -> 2.92 ms,
// 16-view batch 8.65 -> 8.08, 1M diffuse rays 0.863 -> 0.806, soft shadows 3.45 ->
// 3.15; 6 waves 2 to 4 % slower than 7, 5 waves 6 to 10 %.  One thread per ray needs half the
// instructions but waits twice as long per step: its seven or eight loads of a
// node touch 64 lines each, and a leaf's triangles follow one another (same
// camera pass 0.62-0.76 ms, the 14k rays 0.28 ms).  Against the work-item kernel
// (k_traverse64) with its culling and work list, traversal alone: the frame's
// 8 passes 4.77 -> 1.84 ms, a query of 1M diffuse rays 9.18 -> 0.52 ms, one of
// 100k shadow rays 0.54 -> 0.12 ms.
constexpr uint32_t STACK = 48, SMALL_STACK = 6;       // the latter: used of it in the tests of a full stack

template <int CTRL>
__device__ __forceinline__ uint32_t quad_u(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, true);
}
constexpr int QUAD_XOR1 = 0xB1, QUAD_XOR2 = 0x4E;                     // quad_perm [1,0,3,2], [2,3,0,1]
constexpr int QUAD_ROT1 = 0x39, QUAD_ROT2 = 0x4E, QUAD_ROT3 = 0x93;   // [1,2,3,0], [2,3,0,1], [3,0,1,2]
template <int CTRL>
__device__ __forceinline__ unsigned long long quad_u64(unsigned long long x) {
    return ((unsigned long long)quad_u<CTRL>((uint32_t)(x >> 32)) << 32) | quad_u<CTRL>((uint32_t)x);
}

// The candidate test of the reference for (ray at sorted position pos,
// triangle): the batch-boundary range of its object, the object's sphere
// against the top node (RAH: neither), and the triangle's sphere against every
// node of the ray's chain.
__device__ __forceinline__ bool is_candidate(const TreeParams& P, const uint32_t* off, uint32_t pos, uint32_t tri,
                                             uint32_t obj, float4 sph) {
    uint32_t span = P.rays_per_top;
    bool ok = true;
    for (uint32_t k = P.depth; ok && k-- > 0; span /= P.branch) {
        const size_t g = off[k] + pos / span;
        const float4 S = P.nodes[2 * g], C = P.nodes[2 * g + 1];
        const float2 a = P.aux[g];
        if (k + 1 == P.depth && P.algorithm != 1) {
            const uint4 r = P.obj_range[obj];
            ok = !(tri >= r.z && tri < r.w) && sphere_node(S, C, P.obj_sphere[obj], a.x, a.y);
        }
        ok = ok && sphere_node(S, C, sph, a.x, a.y);
    }
    return ok;
}

// A ray's factors of the slab arithmetic.
struct Slabs {
    float ix, iy, iz;              // 1 / direction
    float lx, ly, lz, hx, hy, hz;  // box planes lo - e and hi + e: t = plane * i + l (or h)
    float slack;
    bool plain;
};
__device__ __forceinline__ Slabs make_slabs(const TreeParams& P, v3 o, v3 d, float dd) {
    Slabs s;
    // Per-ray margin of the boxes: at least the line test's, 1e-4 (|c - o|_1 +
    // r) + 1e-6, for every triangle of the scene box, and the slab arithmetic's
    // own rounding.  That works on coordinates, not on differences as the tests
    // above do: o +- e, its product with 1 / d and the box planes are each off by
    // up to 2^-24 of |o| + far1, a margin per axis of 3 2^-24 |o| (taken as 4e-7)
    // beside what the first term holds.  Without it a scene of 10 units lost 0.008 %
    // of its hits 50,000 units from the origin, 0.3 % at 100,000.
    const v3 slo = mk(unordered(P.bounds[0]), unordered(P.bounds[1]), unordered(P.bounds[2]));
    const v3 shi = mk(unordered(P.bounds[3]), unordered(P.bounds[4]), unordered(P.bounds[5]));
    const float far1 = fmaxf(fabsf(slo.x - o.x), fabsf(shi.x - o.x)) + fmaxf(fabsf(slo.y - o.y), fabsf(shi.y - o.y)) +
                       fmaxf(fabsf(slo.z - o.z), fabsf(shi.z - o.z));
    const float e = 1.1e-4f * (far1 + unordered(P.bounds[6])) + 1e-5f;
    const v3 ao = mk(fabsf(o.x), fabsf(o.y), fabsf(o.z));
    const v3 m = mk(__builtin_fmaf(4e-7f, ao.x, e), __builtin_fmaf(4e-7f, ao.y, e), __builtin_fmaf(4e-7f, ao.z, e));
    // Rays whose magnitudes leave the range of the slab arithmetic visit every
    // box (all factors 0: no box is rejected).
    s.plain = dd >= 1e-24f && dd <= 1e24f && far1 + fmaxf(ao.x, fmaxf(ao.y, ao.z)) <= 1e15f;
    auto inverse = [&](float x) {
        return s.plain ? hw_rcp(fabsf(x) < 1e-18f ? (x < 0.0f ? -1e-18f : 1e-18f) : x) : 0.0f;
    };
    s.ix = inverse(d.x); s.iy = inverse(d.y); s.iz = inverse(d.z);
    s.lx = s.plain ? -(o.x + m.x) * s.ix : 0.0f; s.ly = s.plain ? -(o.y + m.y) * s.iy : 0.0f;
    s.lz = s.plain ? -(o.z + m.z) * s.iz : 0.0f;
    s.hx = s.plain ? -(o.x - m.x) * s.ix : 0.0f; s.hy = s.plain ? -(o.y - m.y) * s.iy : 0.0f;
    s.hz = s.plain ? -(o.z - m.z) * s.iz : 0.0f;
    s.slack = 0.01f * hw_rcp(hw_sqrt(dd));
    return s;
}
// Entry distance of a child's box, and whether the ray meets it before lim.
__device__ __forceinline__ bool meets(const Slabs& s, float4 lo, float4 hi, float lim, float& tn) {
    const float x0 = __builtin_fmaf(lo.x, s.ix, s.lx), x1 = __builtin_fmaf(hi.x, s.ix, s.hx);
    const float y0 = __builtin_fmaf(lo.y, s.iy, s.ly), y1 = __builtin_fmaf(hi.y, s.iy, s.hy);
    const float z0 = __builtin_fmaf(lo.z, s.iz, s.lz), z1 = __builtin_fmaf(hi.z, s.iz, s.hz);
    tn = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), 0.0f));
    const float tf = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fminf(fmaxf(z0, z1), lim));
    return !(tn > tf) && __float_as_uint(lo.w) != TREE_EMPTY;
}

template <int KIND>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(8, 8))) k_tree_trace(const TreeParams P) {
    __shared__ uint32_t s_stack[STACK][16];
    __shared__ uint16_t s_near[KIND == 0 ? STACK : 1][16];     // entry distance, upper half (rounded down)
    const uint32_t lane = threadIdx.x, q = lane & 3u, ray = lane >> 2;
    const uint32_t* off = P.ps ? P.ps->offset : P.level_offset;
    // Workgroups go to the 8 XCDs in turn; 64 neighbours (1024 sorted rays) stay
    // on one, whose L2 then holds their part of the tree (atrium frame 2.91 ->
    // 2.86 ms; an eighth of the pass on each XCD: 2.95, and 12 % slower on the
    // batch, whose parts differ in length).
    const uint32_t b = blockIdx.x;
    const uint32_t blk = b < (gridDim.x & ~511u) ? (b & ~511u) | ((b & 7u) << 6) | ((b >> 3) & 63u) : b;
    const uint32_t pos = blk * 16 + ray;
    if (pos >= (P.ps ? P.ps->N : P.N)) return;
    const float4 r0 = P.rec0[pos], r1 = P.rec1[pos];
    const uint32_t slot = __float_as_uint(r0.w);
    const v3 d = xyz(r1), o = xyz(r0) + d * EPS;
    const float dd = dot(d, d);
    const float tmax = r1.w;
    const unsigned long long miss = P.hit_mode == 0 ? MISS64 : (unsigned long long)MISS32;
    const float none = __int_as_float(0x7FC00000);
    const Slabs S = make_slabs(P, o, d, dd);
    unsigned long long best = miss;
    bool occluded = false, verify = false;
    // hi: the range test's bound (NaN: none), lim: the boxes'
    float hi = KIND == 1 ? tmax : none;
    float lim = KIND == 1 && S.plain ? tmax * 1.002f + S.slack : INFINITY;
    uint32_t sp = 0, best_rec = TREE_EMPTY;
    uint32_t scan = TREE_EMPTY;                // next record of a scan over all triangles
    // A NaN direction is never hit (every comparison of ray_triangle's results
    // fails).
    uint32_t cur = dd == dd ? 0u : TREE_EMPTY;
    // The next entry that may still hold a nearer hit.
    auto pop = [&]() -> uint32_t {
        while (sp > 0) {
            sp--;
            const uint32_t c = s_stack[sp][ray];
            if (KIND == 1 || !(__uint_as_float((uint32_t)s_near[sp][ray] << 16) > lim)) return c;
        }
        return TREE_EMPTY;
    };
    for (;;) {
        while (!(cur & TREE_IS_LEAF)) {
            const float4* nb = P.tree[cur].child[q];
            const float4 a = nb[0], b = nb[1];
            const uint32_t ch = __float_as_uint(a.w);
            float tn;
            const bool in = meets(S, a, b, lim, tn);
            const uint32_t key = in ? (__float_as_uint(tn) & ~3u) | q : 0xFFFFFFFCu | q;
            uint32_t n = (uint32_t)__popc((uint32_t)(__ballot(in) >> (lane & 60u)) & 15u);
            // rank of the lane's child among the hit ones, nearest first
            const uint32_t rank = (quad_u<QUAD_ROT1>(key) < key ? 1u : 0u) + (quad_u<QUAD_ROT2>(key) < key ? 1u : 0u) +
                                  (quad_u<QUAD_ROT3>(key) < key ? 1u : 0u);
            const bool full = sp + n > P.stack;    // no ray of a scene of ordinary depth
            if (in && !full) {
                const uint32_t at = sp + n - 1u - rank;
                s_stack[at][ray] = ch;
                if (KIND == 0) s_near[at][ray] = (uint16_t)(__float_as_uint(tn) >> 16);
            }
            sp = full ? 0u : sp + n;
            n = full ? 0u : n;
            scan = full ? 0u : scan;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");     // pushed by one lane, popped by four
            if (n != 0u) cur = s_stack[--sp][ray];
            else cur = pop();
        }
        if (cur == TREE_EMPTY) {
            if (scan < P.T) {
                // the stack was full: the ray takes every triangle in turn
                if (scan == 0u) {
                    verify = true;
                    best = miss;
                    if (KIND == 0) hi = none;
                }
                cur = TREE_IS_LEAF | (min(P.T - scan, TREE_LEAF) - 1u) << 29 | scan;
                scan += TREE_LEAF;
            } else {
                if (KIND == 1 || verify || best_rec == TREE_EMPTY) break;
                // The closest accepted triangle is the answer if it is a
                // candidate (nearly always); otherwise the ray starts over and
                // tests every triangle that would improve its result.
                const float4* rec = P.records + 4 * (size_t)best_rec;
                if (is_candidate(P, off, pos, __float_as_uint(rec[1].w), __float_as_uint(rec[2].w), rec[0])) break;
                verify = true;
                best = miss;
                hi = none;
                lim = INFINITY;
                cur = 0u;
                continue;
            }
        }
        const uint32_t first = cur & 0x1FFFFFFFu, n = ((cur >> 29) & 3u) + 1u;
        const uint32_t j = first + (q < n ? q : 0u);
        const float4* rec = P.records + 4 * (size_t)j;
        // The triangle first: both tests have to accept, about three in four
        // spheres do, and the sphere's answer would cost a trip to memory ahead
        // of the triangle's own (1080p atrium frame 2.58 -> 2.54 ms, 100k shadow
        // rays 212 -> 197 us, against sphere first).
        if (q < n) {
            const float4 A = rec[1], B = rec[2], C = rec[3];
            const float th = ray_triangle(o, d, xyz(A), xyz(B), xyz(C));
            const uint32_t tri = __float_as_uint(A.w);
            unsigned long long rc = miss;
            if (KIND == 1) {
                if (th > EPS && th < tmax) rc = 0ull;
            } else if (th > EPS) {
                rc = pack_hit(th, tri, P.hit_mode);
            }
            if (rc < best) {
                const float4 sph = rec[0];
                const bool may = P.line_only ? ray_may_hit_sphere(o, d, dd, sph)
                                             : ray_may_hit_sphere_range(o, d, dd, sph, EPS, hi);
                if (may && ((KIND == 0 && !verify) || is_candidate(P, off, pos, tri, __float_as_uint(B.w), sph))) {
                    best = rc;
                    best_rec = j;
                }
            }
        }
        if (KIND == 1) {
            uint32_t any = best == 0ull ? 1u : 0u;
            any |= quad_u<QUAD_XOR1>(any);
            any |= quad_u<QUAD_XOR2>(any);
            if (any) { occluded = true; break; }
        } else {
            // the quad agrees on its closest record
            unsigned long long m = quad_u64<QUAD_XOR1>(best);
            uint32_t mr = quad_u<QUAD_XOR1>(best_rec);
            if (m < best) { best = m; best_rec = mr; }
            m = quad_u64<QUAD_XOR2>(best);
            mr = quad_u<QUAD_XOR2>(best_rec);
            if (m < best) { best = m; best_rec = mr; }
            if (P.hit_mode == 0) {
                hi = __uint_as_float((uint32_t)(best >> 32));
                if (S.plain) lim = hi != hi ? INFINITY : hi * 1.002f + S.slack;
            }
        }
        cur = pop();
    }
    if (q != 0u) return;
    if (KIND == 1) {
        if (occluded) P.shadow[slot] = MISS32;
    } else {
        P.closest[slot] = best;
    }
}

// The same for small passes, a wave per ray: each step takes up to 16 entries
// off the ray's stack, one to a quad, so a ray that meets hundreds of boxes is a
// chain of tens of steps instead of hundreds.  It visits boxes that a nearer hit
// would have spared, on SIMDs that a small pass leaves idle.
constexpr uint32_t WAVE_STACK = 512, SMALL_WAVE_STACK = 16;

// Up to how many rays a wave each is the faster.  How long a quad's chain of
// steps is decides, and that goes with the triangle boxes a line through the
// scene meets (TreeMeasure::boxes).  Whole queries, quad and wave in us:
//   boxes  scene                  33000 rays    65536        131072
//     6    plain room, diffuse     131   144   144   180    156   243
//    13    atrium, diffuse         227   169   199   220    226   338
//    25    office, primary         211   170   226   243    247   400
//    25    office, diffuse         193   166   227   229    256   365
//    29    soup of 10k, diffuse    448   220   490   300    568   489
//   115    2k large triangles      878   257   911   395   1080   648
//   170    100k, sparse            305   199   346   276    423   441
//   259    soup of 100k, primary   672   257   730   506   1203   697
//   259    soup of 100k, diffuse   982   313  1119   488   1363   845
// The limit is 32768 up to 12 boxes, where the plain room's lie together, and
// grows with them to four times that, where the first of the long ones meet.
// With 32768 for all, 33,000 rays of the long scenes were slower than by testing
// every candidate (soup, primary 579; 10k, diffuse 364; large triangles 428).
// A frame's rays walk together, and a quad's chains are the shorter for it:
// camera and mirror rays meet at half as many (office frame of 512x512, 44,000
// mirror rays: 483 us with a quad a ray, 510 with a wave), camera rays at 49152 at
// most (quad and wave: office 297 and 326, soup 523 and 509, 100k overlapping 498
// and 489; 76800: soup 568 and 673), and shadow rays, which end at the first
// occluder, not above 32768 in any scene (soup, 512x512, 90,000: 853 and 963).
// A device-sized pass, as captured frames have, is taken by its capacity: the
// workgroups past its rays end at once (replayed 64x64 frame with two bounces
// and shadows, soup: 1275 us with a quad a ray, 438 so).
inline uint32_t wave_rays(const TreeParams& p) {
    const uint32_t rays = (uint32_t)(32768.0f * std::fmin(8.0f, std::fmax(1.0f, p.boxes / 12.0f)));     // a query's, before its cap
    if (!p.frame) return std::min(rays, 131072u);
    if (p.kind == 1) return 32768u;
    return p.line_only ? std::min(rays / 2, 49152u) : std::min(std::max(rays / 2, 32768u), 131072u);
}

template <int KIND>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(8, 8))) k_tree_trace_wave(const TreeParams P) {
    __shared__ uint32_t s_stack[WAVE_STACK];
    __shared__ uint16_t s_near[KIND == 0 ? WAVE_STACK : 1];    // entry distance, upper half (rounded down)
    const uint32_t lane = threadIdx.x, q = lane & 3u, quad = lane >> 2, pos = blockIdx.x;
    if (pos >= (P.ps ? P.ps->N : P.N)) return;
    const uint32_t* off = P.ps ? P.ps->offset : P.level_offset;
    const float4 r0 = P.rec0[pos], r1 = P.rec1[pos];
    const v3 d = xyz(r1), o = xyz(r0) + d * EPS;
    const float dd = dot(d, d);
    const float tmax = r1.w;
    const unsigned long long miss = P.hit_mode == 0 ? MISS64 : (unsigned long long)MISS32;
    const float none = __int_as_float(0x7FC00000);
    const Slabs S = make_slabs(P, o, d, dd);
    unsigned long long best = miss;
    uint32_t best_rec = TREE_EMPTY;
    bool occluded = false, verify = false;
    float hi = KIND == 1 ? tmax : none;
    float lim = KIND == 1 && S.plain ? tmax * 1.002f + S.slack : INFINITY;
    uint32_t scan = TREE_EMPTY;                // next record of a scan over all triangles
    uint32_t sp = dd == dd ? 1u : 0u;          // a NaN direction is never hit
    if (lane == 0) {
        s_stack[0] = 0u;
        if (KIND == 0) s_near[0] = 0;
    }
    for (;;) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");     // pushed by one lane, taken by others
        uint32_t j = TREE_EMPTY;               // the lane's triangle
        if (sp != 0u) {
            const uint32_t m = min(min(sp, 16u), (P.stack - sp) / 3u);
            if (m == 0u) {                     // full: the ray takes every triangle in turn
                sp = 0u;
                scan = 0u;
                verify = true;
                best = miss;
                if (KIND == 0) hi = none;
                continue;
            }
            sp -= m;
            uint32_t cur = TREE_EMPTY;
            if (quad < m) {
                const uint32_t at = sp + m - 1u - quad;
                const uint32_t c = s_stack[at];
                if (KIND == 1 || !(__uint_as_float((uint32_t)s_near[at] << 16) > lim)) cur = c;
            }
            bool in = false;
            uint32_t ch = 0u, rank = 0u;
            float tn = 0.0f;
            if (!(cur & TREE_IS_LEAF)) {       // whole quads
                const float4* nb = P.tree[cur].child[q];
                const float4 a = nb[0], b = nb[1];
                ch = __float_as_uint(a.w);
                in = meets(S, a, b, lim, tn);
                const uint32_t key = in ? (__float_as_uint(tn) & ~3u) | q : 0xFFFFFFFCu | q;
                rank = (quad_u<QUAD_ROT1>(key) < key ? 1u : 0u) + (quad_u<QUAD_ROT2>(key) < key ? 1u : 0u) +
                       (quad_u<QUAD_ROT3>(key) < key ? 1u : 0u);
            } else if (cur != TREE_EMPTY) {
                const uint32_t n = ((cur >> 29) & 3u) + 1u;
                if (q < n) j = (cur & 0x1FFFFFFFu) + q;
            }
            // the nearest of the topmost entry on top
            const unsigned long long mask = __ballot(in), from = mask >> (lane & 60u);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // all entries taken
            if (in) {
                const uint32_t at = sp + (uint32_t)__popcll(from >> 4) + (uint32_t)__popc((uint32_t)from & 15u) - 1u - rank;
                s_stack[at] = ch;
                if (KIND == 0) s_near[at] = (uint16_t)(__float_as_uint(tn) >> 16);
            }
            sp += (uint32_t)__popcll(mask);
        } else if (scan < P.T) {
            if (scan + lane < P.T) j = scan + lane;
            scan += 64u;
        } else {
            if (KIND == 1 || verify || best_rec == TREE_EMPTY) break;
            // as in k_tree_trace
            const float4* rec = P.records + 4 * (size_t)best_rec;
            if (is_candidate(P, off, pos, __float_as_uint(rec[1].w), __float_as_uint(rec[2].w), rec[0])) break;
            verify = true;
            best = miss;
            hi = none;
            lim = INFINITY;
            if (lane == 0) { s_stack[0] = 0u; s_near[0] = 0; }
            sp = 1u;
            continue;
        }
        unsigned long long mine = best;
        uint32_t mine_rec = best_rec;
        if (j != TREE_EMPTY) {
            const float4* rec = P.records + 4 * (size_t)j;
            const float4 A = rec[1], B = rec[2], C = rec[3];
            const float th = ray_triangle(o, d, xyz(A), xyz(B), xyz(C));
            const uint32_t tri = __float_as_uint(A.w);
            unsigned long long rc = miss;
            if (KIND == 1) {
                if (th > EPS && th < tmax) rc = 0ull;
            } else if (th > EPS) {
                rc = pack_hit(th, tri, P.hit_mode);
            }
            if (rc < best) {
                const float4 sph = rec[0];
                const bool may = P.line_only ? ray_may_hit_sphere(o, d, dd, sph)
                                             : ray_may_hit_sphere_range(o, d, dd, sph, EPS, hi);
                if (may && ((KIND == 0 && !verify) || is_candidate(P, off, pos, tri, __float_as_uint(B.w), sph))) {
                    mine = rc;
                    mine_rec = j;
                }
            }
        }
        if (__ballot(mine < best) == 0ull) continue;
        if (KIND == 1) { occluded = true; break; }
#pragma unroll
        for (int x = 32; x > 0; x >>= 1) {
            const unsigned long long om = __shfl_xor(mine, x, 64);
            const uint32_t orec = (uint32_t)__shfl_xor((int)mine_rec, x, 64);
            if (om < mine) { mine = om; mine_rec = orec; }
        }
        best = mine;
        best_rec = mine_rec;
        if (P.hit_mode == 0) {
            hi = __uint_as_float((uint32_t)(best >> 32));
            if (S.plain) lim = hi != hi ? INFINITY : hi * 1.002f + S.slack;
        }
    }
    if (lane != 0u) return;
    const uint32_t slot = __float_as_uint(r0.w);
    if (KIND == 1) {
        if (occluded) P.shadow[slot] = MISS32;
    } else {
        P.closest[slot] = best;
    }
}

}  // namespace

// One allocation for what the traversal reads, one for the construction.  The I
// wide nodes with an inner child have four children each and the B others two
// triangles or more, every leaf child one: T >= 4 I - (I + B - 1) + 2 B and B <=
// 3 I + 1, so I + B <= 2 T / 3 (one for a scene of a single leaf).
inline uint32_t wide_nodes(uint32_t T) { return (uint32_t)(2 * (uint64_t)T / 3) + 1u; }

hipError_t TreeBuild::reserve(uint32_t T) {
    struct Slab {
        char* p;
        size_t off = 0;
        void take(DevBuf& b, size_t bytes) {
            if (p) { b.p = p + off; b.bytes = bytes; }
            off += (bytes + 255) & ~(size_t)255;
        }
    };
    // binary nodes: T leaves, T for the first merging launch, then MERGE_CHUNK a workgroup
    const uint32_t groups = (T + MERGE_CHUNK - 1) / MERGE_CHUNK;
    size_t binary = 2 * (size_t)T;
    for (uint32_t g = groups; g > 1;) { g = (g + 15) / 16; binary += (size_t)g * MERGE_CHUNK; }
    const size_t wide = wide_nodes(T);
    hipError_t e = hipSuccess;
    for (int pass = 0; pass < 2 && e == hipSuccess; pass++) {      // sizes, then addresses
        Slab a{pass ? keep.as<char>() : nullptr}, b{pass ? work.as<char>() : nullptr};
        a.take(nodes, wide * sizeof(TreeNode)); a.take(records, (size_t)T * 64); a.take(bounds, 64);
        b.take(box, (size_t)T * 32); b.take(node, binary * 32); b.take(size, binary * 4);
        b.take(left, ((size_t)groups * 2 + 2) * MERGE_KEEP * 4); b.take(left_count, ((size_t)groups * 2 + 2) * 4);
        b.take(scodes, (size_t)T * 4); b.take(sids, (size_t)T * 4); b.take(queue, wide * 8);
        b.take(count, (TREE_LEVELS + 1) * 4); b.take(codes, (size_t)T * 4); b.take(ids, (size_t)T * 4);
        b.take(sc.ping_k, (size_t)T * 4); b.take(sc.ping_v, (size_t)T * 4); b.take(sc.hist, sort_hist_bytes(T));
        b.take(sc.digit_totals, 512 * 4);
        if (pass) break;
        e = keep.reserve(a.off);
        if (e == hipSuccess) e = work.reserve(b.off);
    }
    return e;
}

void TreeBuild::release() {
    keep.release();
    work.release();
}

hipError_t TreeBuild::build(const float4* tri_sphere, const float4* tri_mt, const uint4* objects, uint32_t K, uint32_t T,
                            TreeMeasure* measure, hipStream_t s) {
    if (T == 0 || T > TREE_MAX_TRIANGLES || K == 0) return hipErrorInvalidValue;
    float4* bx = box.as<float4>();
    uint32_t* bd = bounds.as<uint32_t>();
    k_tree_clear<<<1, 64, 0, s>>>(bd);
    const uint32_t prim_blocks = min(grid_for(T, 1024), PRIM_BLOCKS);
    float* sums = queue.as<float>();        // (256 B at least; the queue is filled after the merge has read them)
    k_tree_prims<<<prim_blocks, 1024, 0, s>>>(tri_sphere, tri_mt, T, bx, bd, sums);
    k_tree_codes<<<grid_for(T, 256), 256, 0, s>>>(bx, T, bd, codes.as<uint32_t>(), ids.as<uint32_t>());
    const hipError_t e = run_radix_sort(codes.as<uint32_t>(), ids.as<uint32_t>(), T, 3 * CODE_BITS,
                                        scodes.as<uint32_t>(), sids.as<uint32_t>(), sc, s);
    if (e != hipSuccess) return e;
    MergeArgs M{};
    M.T = T; M.ids = sids.as<uint32_t>(); M.box = bx; M.base = T;
    M.node = node.as<float4>(); M.size = size.as<uint32_t>();
    M.out = left.as<uint32_t>(); M.out_count = left_count.as<uint32_t>();
    M.area = sums; M.area_blocks = prim_blocks; M.measure = measure;
    uint32_t groups = (T + MERGE_CHUNK - 1) / MERGE_CHUNK;
    M.last = groups == 1;
    k_tree_merge<true><<<groups, 1024, 0, s>>>(M);
    M.base += T;
    while (!M.last) {
        // each launch's clusters follow those of the one before
        M.in = M.out; M.in_count = M.out_count; M.in_groups = groups;
        M.out += (size_t)groups * MERGE_KEEP; M.out_count += groups;
        groups = (groups + 15) / 16;
        M.last = groups == 1;
        k_tree_merge<false><<<groups, 1024, 0, s>>>(M);
        M.base += groups * MERGE_CHUNK;
    }
    EmitArgs A{T, M.node, M.size, M.out, queue.as<uint2>(), count.as<uint32_t>(), nodes.as<TreeNode>()};
    k_tree_root<<<1, 64, 0, s>>>(A);
    if (T > TREE_LEAF) {
        // a level has at most 4^level nodes: the first and the last levels in one
        // workgroup, the wide ones between with a launch each
        uint32_t level = 0;
        if (T > 16384) {
            k_tree_tail<<<1, 1024, 0, s>>>(A, 0u, 4u);
            for (level = 5; level < 12; level++) k_tree_level<<<grid_for(T / 8, 256), 256, 0, s>>>(A, level);
        }
        k_tree_tail<<<1, 1024, 0, s>>>(A, level, TREE_LEVELS - 2u);
    }
    k_tree_records<<<grid_for(4 * (uint64_t)wide_nodes(T), 256), 256, 0, s>>>(A, M.ids, tri_sphere, tri_mt, objects, K,
                                                                              records.as<float4>());
    return hipGetLastError();
}

void launch_tree_trace(const TreeParams& p, hipStream_t s) {
    if (!p.N) return;
    const bool wave = p.walk == WALK_WAVE || (p.walk != WALK_QUAD && p.N <= wave_rays(p));
    TreeParams q = p;
    if (wave) {
        q.stack = p.small_stack ? SMALL_WAVE_STACK : WAVE_STACK;
        if (p.kind == 1) k_tree_trace_wave<1><<<p.N, 64, 0, s>>>(q);
        else k_tree_trace_wave<0><<<p.N, 64, 0, s>>>(q);
        return;
    }
    q.stack = p.small_stack ? SMALL_STACK : STACK;
    if (p.kind == 1) k_tree_trace<1><<<grid_for(p.N, 16), 64, 0, s>>>(q);
    else k_tree_trace<0><<<grid_for(p.N, 16), 64, 0, s>>>(q);
}

}  // namespace rsh
