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
// The tree is a four-wide bounding-box tree over the triangles in Morton
// order: Karras' radix tree, from which each wide node takes the children of
// the largest surface.  It is rebuilt on the device at scene load and after
// object updates (262,604 triangles: about 0.25 ms, bound by the latency of
// its 30 launches).
#include <utility>

#include "rsh_kernels.hpp"

namespace rsh {

namespace {

constexpr uint32_t TREE_LEAF = 4;              // triangles per leaf
constexpr uint32_t TREE_EMPTY = 0xFFFFFFFFu;
constexpr uint32_t TREE_IS_LEAF = 0x80000000u; // child word: leaf flag, (count - 1) << 29, first record
constexpr uint32_t CODE_BITS = 9;              // Morton code bits per axis (three sorting passes)
constexpr uint32_t BLOCK_SHIFT = 3;            // range boxes: 8 children per block level

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
__global__ void __launch_bounds__(256) k_tree_prims(const float4* tri_sphere, const float4* tri_mt, uint32_t T,
                                                    float4* box, uint32_t* bounds) {
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    v3 lo = mk(INFINITY, INFINITY, INFINITY), hi = mk(-INFINITY, -INFINITY, -INFINITY);
    float r = 0.0f;
    if (t < T) {
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
        if (isfinite(all)) { lo = l; hi = h; r = s.w; }
        box[2 * (size_t)t] = f4(lo, 0.0f);
        box[2 * (size_t)t + 1] = f4(hi, 0.0f);
    }
    const float m[7] = {wave_min_f(lo.x), wave_min_f(lo.y), wave_min_f(lo.z),
                        wave_max_f(hi.x), wave_max_f(hi.y), wave_max_f(hi.z), wave_max_f(r)};
    if ((threadIdx.x & 63u) == 0) {
#pragma unroll
        for (int i = 0; i < 3; i++) atomicMin(&bounds[i], ordered(m[i]));
#pragma unroll
        for (int i = 3; i < 7; i++) atomicMax(&bounds[i], ordered(m[i]));
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

// Triangle records in tree order, 64 B each: (sphere), (v0, triangle id),
// (e1, object), (e2, -), and their boxes (block level 0).
// objects: (first triangle, ...) of each of the K objects, which tile [0, T) in order.
__global__ void __launch_bounds__(256) k_tree_records(const uint32_t* ids, const float4* tri_sphere,
                                                      const float4* tri_mt, const uint4* objects, uint32_t K,
                                                      const float4* box, uint32_t T, float4* rec, float4* blk) {
    const uint32_t j = blockIdx.x * 256 + threadIdx.x;
    if (j >= T) return;
    const uint32_t t = ids[j];
    uint32_t a = 0, b = K;      // objects[a].x <= t < objects[b].x (b = K: end)
    while (b - a > 1) {
        const uint32_t m = (a + b) >> 1;
        if (objects[m].x <= t) a = m; else b = m;
    }
    rec[4 * (size_t)j] = tri_sphere[t];
    rec[4 * (size_t)j + 1] = f4(xyz(tri_mt[3 * (size_t)t]), __uint_as_float(t));
    rec[4 * (size_t)j + 2] = f4(xyz(tri_mt[3 * (size_t)t + 1]), __uint_as_float(a));
    rec[4 * (size_t)j + 3] = f4(xyz(tri_mt[3 * (size_t)t + 2]), 0.0f);
    blk[2 * (size_t)j] = box[2 * (size_t)t];
    blk[2 * (size_t)j + 1] = box[2 * (size_t)t + 1];
}

__device__ __forceinline__ void grow(v3& lo, v3& hi, const float4* b) {
    const float4 l = b[0], h = b[1];
    lo = mk(fminf(lo.x, l.x), fminf(lo.y, l.y), fminf(lo.z, l.z));
    hi = mk(fmaxf(hi.x, h.x), fmaxf(hi.y, h.y), fmaxf(hi.z, h.z));
}

// Boxes of aligned runs of 8 entries of the level below.
__global__ void __launch_bounds__(256) k_tree_blocks(const float4* in, uint32_t n, float4* out, uint32_t m) {
    const uint32_t j = blockIdx.x * 256 + threadIdx.x;
    if (j >= m) return;
    v3 lo = mk(INFINITY, INFINITY, INFINITY), hi = mk(-INFINITY, -INFINITY, -INFINITY);
    for (uint32_t i = j << BLOCK_SHIFT; i < ((j + 1) << BLOCK_SHIFT) && i < n; i++) grow(lo, hi, in + 2 * (size_t)i);
    out[2 * (size_t)j] = f4(lo, 0.0f);
    out[2 * (size_t)j + 1] = f4(hi, 0.0f);
}

struct BlockLevels {
    uint32_t off[12];      // first entry of each level
    uint32_t levels;
};

// Box of the records [a, b]: whole blocks of the highest level that fits,
// single entries at the ragged ends.
__device__ void range_box(const float4* blk, const BlockLevels& L, uint32_t a, uint32_t b, v3& lo, v3& hi) {
    lo = mk(INFINITY, INFINITY, INFINITY); hi = mk(-INFINITY, -INFINITY, -INFINITY);
    uint32_t e = b + 1;      // [a, e) in units of the current level
    for (uint32_t k = 0;; k++) {
        const float4* p = blk + 2 * (size_t)L.off[k];
        constexpr uint32_t W = 1u << BLOCK_SHIFT;
        if (k + 1 == L.levels || e - a <= W) {
            for (uint32_t i = a; i < e; i++) grow(lo, hi, p + 2 * (size_t)i);
            return;
        }
        while (a & (W - 1u)) { grow(lo, hi, p + 2 * (size_t)a); a++; }
        while (e & (W - 1u)) { e--; grow(lo, hi, p + 2 * (size_t)e); }
        a >>= BLOCK_SHIFT; e >>= BLOCK_SHIFT;
        if (a >= e) return;
    }
}

// Radix tree over the sorted codes (Karras 2012): internal node i covers the
// records [range.x, range.y]; child words: internal index, or TREE_IS_LEAF |
// record.  Equal codes are told apart by their positions.
__global__ void __launch_bounds__(256) k_tree_link(const uint32_t* codes, uint32_t T, uint2* range, uint2* child) {
    const int i = (int)(blockIdx.x * 256 + threadIdx.x);
    const int n = (int)T;
    if (i >= n - 1) return;
    auto delta = [&](int a, int b) -> int {
        if (b < 0 || b >= n) return -1;
        const uint32_t x = codes[a] ^ codes[b];
        return x ? __clz((int)x) : 32 + __clz(a ^ b);
    };
    const int d = delta(i, i + 1) > delta(i, i - 1) ? 1 : -1;
    const int dmin = delta(i, i - d);
    int lmax = 2;
    while (delta(i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dn = delta(i, j);
    int s = 0;
    for (int t = (l + 1) >> 1;; t = (t + 1) >> 1) {
        if (delta(i, i + (s + t) * d) > dn) s += t;
        if (t == 1) break;
    }
    const int g = i + s * d + (d < 0 ? d : 0);
    const int a = i < j ? i : j, b = i < j ? j : i;
    range[i] = make_uint2((uint32_t)a, (uint32_t)b);
    child[i] = make_uint2(a == g ? TREE_IS_LEAF | (uint32_t)g : (uint32_t)g,
                          b == g + 1 ? TREE_IS_LEAF | (uint32_t)(g + 1) : (uint32_t)(g + 1));
}

// Boxes of the radix tree's internal nodes.
__global__ void __launch_bounds__(256) k_tree_boxes(uint32_t T, const uint2* range, const float4* blk, BlockLevels L,
                                                    float4* ibox) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i + 1u >= T) return;
    const uint2 r = range[i];
    v3 lo, hi;
    range_box(blk, L, r.x, r.y, lo, hi);
    ibox[2 * (size_t)i] = f4(lo, 0.0f);
    ibox[2 * (size_t)i + 1] = f4(hi, 0.0f);
}

// Wide node w, built from radix node `root`: the child of the largest surface
// is replaced by its two children until there are four or only leaves are
// left.  Its inner children become the next level's wide nodes at `next` on,
// as counted in *count.
struct EmitArgs {
    uint32_t T;
    const uint2* range;
    const uint2* child;
    const float4* ibox;
    const float4* blk;
    uint32_t* queue;        // radix node of every wide node, in breadth-first order
    uint32_t* count;        // wide nodes per level
    TreeNode* nodes;
};
constexpr uint32_t TREE_LEVELS = 64;

__device__ void emit_node(const EmitArgs& A, uint32_t w, uint32_t next, uint32_t* count) {
    uint32_t cw[4] = {TREE_EMPTY, TREE_EMPTY, TREE_EMPTY, TREE_EMPTY};
    float4 lo[4], hi[4];
    float area[4];          // of a child that can be split, else -1
    uint32_t n = 0;
    auto put = [&](uint32_t k, uint32_t c) {
        const bool one = c & TREE_IS_LEAF;
        const uint32_t id = c & ~TREE_IS_LEAF;
        const uint2 r = one ? make_uint2(id, id) : A.range[id];
        const float4* b = (one ? A.blk : A.ibox) + 2 * (size_t)id;
        lo[k] = b[0]; hi[k] = b[1];
        const bool leaf = r.y - r.x + 1u <= TREE_LEAF;
        cw[k] = leaf ? TREE_IS_LEAF | ((r.y - r.x) << 29) | r.x : c;
        const float dx = hi[k].x - lo[k].x, dy = hi[k].y - lo[k].y, dz = hi[k].z - lo[k].z;
        area[k] = leaf ? -1.0f : fmaxf(dx * dy + dy * dz + dz * dx, 0.0f);     // NaN -> 0
    };
    const uint2 c0 = A.child[A.queue[w]];
    put(0, c0.x); put(1, c0.y);
    n = 2;
    for (; n < 4; n++) {
        uint32_t k = 0;
#pragma unroll
        for (uint32_t i = 1; i < 4; i++)
            if (i < n && area[i] > area[k]) k = i;
        if (area[k] < 0.0f) break;
        const uint2 c = A.child[cw[k]];
        put(k, c.x); put(n, c.y);
    }
    uint32_t inner = 0;
    for (uint32_t k = 0; k < n; k++) inner += (cw[k] & TREE_IS_LEAF) ? 0u : 1u;
    uint32_t at = inner ? next + atomicAdd(count, inner) : 0u;
    TreeNode out;
    for (uint32_t k = 0; k < 4; k++) {
        uint32_t word = TREE_EMPTY;
        float4 l = make_float4(INFINITY, INFINITY, INFINITY, 0.0f), h = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
        if (k < n) {
            word = cw[k]; l = lo[k]; h = hi[k];
            if (!(word & TREE_IS_LEAF)) { A.queue[at] = word; word = at++; }
        }
        out.child[k][0] = make_float4(l.x, l.y, l.z, __uint_as_float(word));
        out.child[k][1] = make_float4(h.x, h.y, h.z, 0.0f);
    }
    A.nodes[w] = out;
}

// The root, and the level counts cleared.  Up to TREE_LEAF triangles: one leaf.
__global__ void k_tree_root(EmitArgs A) {
    if (threadIdx.x < TREE_LEVELS) A.count[threadIdx.x] = threadIdx.x == 0 && A.T > TREE_LEAF ? 1u : 0u;
    if (threadIdx.x != 0) return;
    A.queue[0] = 0u;
    if (A.T > TREE_LEAF) return;
    v3 lo = mk(INFINITY, INFINITY, INFINITY), hi = mk(-INFINITY, -INFINITY, -INFINITY);
    for (uint32_t i = 0; i < A.T; i++) grow(lo, hi, A.blk + 2 * (size_t)i);
    TreeNode out;
    for (uint32_t k = 0; k < 4; k++) {
        const uint32_t word = k == 0 ? TREE_IS_LEAF | ((A.T - 1u) << 29) : TREE_EMPTY;
        const v3 l = k == 0 ? lo : mk(INFINITY, INFINITY, INFINITY), h = k == 0 ? hi : mk(-INFINITY, -INFINITY, -INFINITY);
        out.child[k][0] = f4(l, __uint_as_float(word));
        out.child[k][1] = f4(h, 0.0f);
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
        if (n == 0u) return;
        for (uint32_t i = threadIdx.x; i < n; i += 1024u) emit_node(A, start + i, start + n, A.count + level + 1);
        __threadfence_block();
        start += n;
    }
}

// ------------------------------------------------------------- traversal --
// Four lanes per sorted ray (a quad): lane q tests child q of a node or
// triangle q of a leaf; 16 rays, one wave, per workgroup.  Nearest child first;
// the others wait on the ray's stack in LDS.
// Large passes are bound by VALU issue (1080p atrium camera pass: 308M
// instructions, 0.50 ms of issue in 0.60 ms) and the loads behind it, small
// ones by the latency of the longest ray's steps (14k rays: 0.12 ms).  Waves
// hide that latency: 8 a SIMD (64 VGPRs, 9 of the closest-hit kernel's spilled;
// 3.0 / 4.5 KB of LDS) against 7 with 6 KB: 1080p atrium frame 2.97 -> 2.92 ms,
// 16-view batch 8.65 -> 8.08, 1M diffuse rays 0.863 -> 0.806, soft shadows 3.45 ->
// 3.15; 6 waves 2 to 4 % slower than 7, 5 waves 6 to 10 %.  One thread per ray needs half the
// instructions but waits twice as long per step: its seven or eight loads of a
// node touch 64 lines each, and a leaf's triangles follow one another (same
// camera pass 0.62-0.76 ms, the 14k rays 0.28 ms).  Against the work-item kernel
// (k_traverse64) with its culling and work list, traversal alone: the frame's
// 8 passes 4.77 -> 2.06 ms, a query of 1M diffuse rays 9.18 -> 0.63 ms, one of
// 100k shadow rays 0.54 -> 0.13 ms.
constexpr uint32_t STACK = 48;

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
    // r) + 1e-6, for every triangle of the scene box, which also covers the
    // rounding of the slab arithmetic.
    const v3 slo = mk(unordered(P.bounds[0]), unordered(P.bounds[1]), unordered(P.bounds[2]));
    const v3 shi = mk(unordered(P.bounds[3]), unordered(P.bounds[4]), unordered(P.bounds[5]));
    const float far1 = fmaxf(fabsf(slo.x - o.x), fabsf(shi.x - o.x)) + fmaxf(fabsf(slo.y - o.y), fabsf(shi.y - o.y)) +
                       fmaxf(fabsf(slo.z - o.z), fabsf(shi.z - o.z));
    const float e = 1.1e-4f * (far1 + unordered(P.bounds[6])) + 1e-5f;
    // Rays whose magnitudes leave the range of the slab arithmetic visit every
    // box (all factors 0: no box is rejected).
    s.plain = dd >= 1e-24f && dd <= 1e24f && far1 <= 1e15f;
    auto inverse = [&](float x) {
        return s.plain ? hw_rcp(fabsf(x) < 1e-18f ? (x < 0.0f ? -1e-18f : 1e-18f) : x) : 0.0f;
    };
    s.ix = inverse(d.x); s.iy = inverse(d.y); s.iz = inverse(d.z);
    s.lx = s.plain ? -(o.x + e) * s.ix : 0.0f; s.ly = s.plain ? -(o.y + e) * s.iy : 0.0f;
    s.lz = s.plain ? -(o.z + e) * s.iz : 0.0f;
    s.hx = s.plain ? -(o.x - e) * s.ix : 0.0f; s.hy = s.plain ? -(o.y - e) * s.iy : 0.0f;
    s.hz = s.plain ? -(o.z - e) * s.iz : 0.0f;
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
            if (KIND == 1 || !(__uint_as_float((uint32_t)s_near[sp][ray] << 16) > lim)) return s_stack[sp][ray];
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
            uint32_t n = in ? 1u : 0u;
            n += quad_u<QUAD_XOR1>(n);
            n += quad_u<QUAD_XOR2>(n);
            // rank of the lane's child among the hit ones, nearest first
            const uint32_t rank = (quad_u<QUAD_ROT1>(key) < key ? 1u : 0u) + (quad_u<QUAD_ROT2>(key) < key ? 1u : 0u) +
                                  (quad_u<QUAD_ROT3>(key) < key ? 1u : 0u);
            const bool full = sp + n > STACK;  // no ray of a scene of ordinary depth
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
        const float4 sph = rec[0];
        const bool may = q < n && (P.line_only ? ray_may_hit_sphere(o, d, dd, sph)
                                               : ray_may_hit_sphere_range(o, d, dd, sph, EPS, hi));
        if (may) {
            const float4 A = rec[1], B = rec[2], C = rec[3];
            const float th = ray_triangle(o, d, xyz(A), xyz(B), xyz(C));
            const uint32_t tri = __float_as_uint(A.w);
            unsigned long long rc = miss;
            if (KIND == 1) {
                if (th > EPS && th < tmax) rc = 0ull;
            } else if (th > EPS) {
                rc = pack_hit(th, tri, P.hit_mode);
            }
            if (rc < best && ((KIND == 0 && !verify) || is_candidate(P, off, pos, tri, __float_as_uint(B.w), sph))) {
                best = rc;
                best_rec = j;
            }
        }
        // the quad agrees on its closest record
        unsigned long long m = quad_u64<QUAD_XOR1>(best);
        uint32_t mr = quad_u<QUAD_XOR1>(best_rec);
        if (m < best) { best = m; best_rec = mr; }
        m = quad_u64<QUAD_XOR2>(best);
        mr = quad_u<QUAD_XOR2>(best_rec);
        if (m < best) { best = m; best_rec = mr; }
        if (KIND == 1) {
            if (best == 0ull) { occluded = true; break; }
        } else if (P.hit_mode == 0) {
            hi = __uint_as_float((uint32_t)(best >> 32));
            if (S.plain) lim = hi != hi ? INFINITY : hi * 1.002f + S.slack;
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

}  // namespace

// One allocation for what the traversal reads, one for the construction.  A
// wide node with an inner child has four children, of which every leaf holds a
// triangle, and a bottom one covers five or more triangles, so there are at
// most (T - 1) / 3 of them (and one for a scene of a single leaf).
hipError_t TreeBuild::reserve(uint32_t T) {
    struct Slab {
        char* p;
        size_t off = 0;
        void take(DevBuf& b, size_t bytes) {
            if (p) { b.p = p + off; b.bytes = bytes; }
            off += (bytes + 255) & ~(size_t)255;
        }
    };
    uint64_t blocks = 0;
    for (uint64_t n = T;; n = (n + 7) / 8) { blocks += n; if (n <= 1) break; }
    const size_t wide = (size_t)T / 3 + 1;
    hipError_t e = hipSuccess;
    for (int pass = 0; pass < 2 && e == hipSuccess; pass++) {      // sizes, then addresses
        Slab a{pass ? keep.as<char>() : nullptr}, b{pass ? work.as<char>() : nullptr};
        a.take(nodes, wide * sizeof(TreeNode)); a.take(records, (size_t)T * 64); a.take(bounds, 64);
        b.take(box, (size_t)T * 32); b.take(blk, (size_t)blocks * 32); b.take(scodes, (size_t)T * 4);
        b.take(sids, (size_t)T * 4); b.take(queue, wide * 4); b.take(count, TREE_LEVELS * 4);
        b.take(codes, (size_t)T * 4); b.take(ids, (size_t)T * 4); b.take(sc.ping_k, (size_t)T * 4);
        b.take(sc.ping_v, (size_t)T * 4); b.take(sc.hist, sort_hist_bytes(T));
        b.take(sc.digit_totals, 512 * 4); b.take(range, (size_t)T * 8); b.take(child, (size_t)T * 8);
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
                            hipStream_t s) {
    if (T == 0 || T > (1u << 29) || K == 0) return hipErrorInvalidValue;
    float4* bx = box.as<float4>();       // the triangles' boxes, then the radix nodes'
    float4* bk = blk.as<float4>();
    uint32_t* bd = bounds.as<uint32_t>();
    k_tree_clear<<<1, 64, 0, s>>>(bd);
    k_tree_prims<<<grid_for(T, 256), 256, 0, s>>>(tri_sphere, tri_mt, T, bx, bd);
    k_tree_codes<<<grid_for(T, 256), 256, 0, s>>>(bx, T, bd, codes.as<uint32_t>(), ids.as<uint32_t>());
    const hipError_t e = run_radix_sort(codes.as<uint32_t>(), ids.as<uint32_t>(), T, 3 * CODE_BITS,
                                        scodes.as<uint32_t>(), sids.as<uint32_t>(), sc, s);
    if (e != hipSuccess) return e;
    k_tree_records<<<grid_for(T, 256), 256, 0, s>>>(sids.as<uint32_t>(), tri_sphere, tri_mt, objects, K, bx, T,
                                                    records.as<float4>(), bk);
    BlockLevels L{};
    uint32_t n = T, off = 0;
    L.levels = 1;
    while (n > 8 && L.levels < 12) {
        const uint32_t m = (n + 7) / 8;
        L.off[L.levels] = off + n;
        k_tree_blocks<<<grid_for(m, 256), 256, 0, s>>>(bk + 2 * (size_t)off, n, bk + 2 * (size_t)(off + n), m);
        off += n;
        n = m;
        L.levels++;
    }
    EmitArgs A{T, range.as<uint2>(), child.as<uint2>(), bx, bk, queue.as<uint32_t>(), count.as<uint32_t>(),
               nodes.as<TreeNode>()};
    k_tree_root<<<1, 64, 0, s>>>(A);
    if (T > TREE_LEAF) {
        k_tree_link<<<grid_for(T, 256), 256, 0, s>>>(scodes.as<uint32_t>(), T, range.as<uint2>(), child.as<uint2>());
        k_tree_boxes<<<grid_for(T, 256), 256, 0, s>>>(T, range.as<uint2>(), bk, L, bx);
        // a level has at most 4^level nodes: the first and the last levels in one
        // workgroup, the wide ones between with a launch each
        uint32_t level = 0;
        if (T > 16384) {
            k_tree_tail<<<1, 1024, 0, s>>>(A, 0u, 4u);
            for (level = 5; level < 11; level++) k_tree_level<<<grid_for(T / 8, 256), 256, 0, s>>>(A, level);
        }
        k_tree_tail<<<1, 1024, 0, s>>>(A, level, TREE_LEVELS - 2u);
    }
    return hipGetLastError();
}

void launch_tree_trace(const TreeParams& p, hipStream_t s) {
    if (!p.N) return;
    if (p.kind == 1) k_tree_trace<1><<<grid_for(p.N, 16), 64, 0, s>>>(p);
    else k_tree_trace<0><<<grid_for(p.N, 16), 64, 0, s>>>(p);
}

}  // namespace rsh
