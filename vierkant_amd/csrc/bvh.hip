// bvh.hip - mesh -> BVH build (LBVH) and closest/any-hit traversal for gfx950.
//
// The reference hands triangles to the Vulkan driver (RayBuilder::create_mesh_structures,
// src/RayBuilder.cpp:98-303, vkCmdBuildAccelerationStructuresKHR :274) and traces with TraceRay
// (shaders/slang/raypipeline.slang:182); both are opaque. This file is the MI355X replacement.
//
// Build (all on the GPU, one stream):
//   k_bounds    bounds of the triangles' AABB centers, index check
//   k_morton    30-bit Morton code of the AABB center in the centroid bounds
//   radix sort  (code, triangle) pairs, project-written (radix_sort.hip)
//   k_karras    binary radix tree over the sorted codes (Karras 2012), ties broken by position; or, with
//               VKRT_BUILDER_PLOC, agglomerative clustering over the sorted leaves (k_ploc_*)
//   k_leaves    triangles in leaf order, straight from the mesh: exact AABBs and 64-B records (v0, e1, e2,
//               original index)
//   k_box_*     unions of leaf boxes (segment prefix/suffix unions and a sparse table of segment unions)
//   k_layout    BVH2 nodes holding both children's boxes (64 B), each the union over its leaf run; subtrees of
//               <= max_leaf_size triangles collapsed into leaves over the contiguous sorted range
//
// Traversal: one ray per lane, front-to-back descent with a per-lane stack. Box tests are padded so
// that a box is never culled when it holds a triangle the reference test accepts (see slab_interval),
// and equal-t hits resolve to the lowest original triangle index, so results are identical to the
// brute-force loop over intersect(Triangle, Ray).
#include <algorithm>
#include <cfloat>
#include <chrono>
#include <cmath>
#include <cstring>
#include <initializer_list>
#include <memory>
#include <utility>
#include <vector>

#include "context.hpp"
#include "kernels.hpp"
#include "bvh_types.hpp"
#include "radix_sort.hpp"
#include "vierkant/rt_math.hpp"

using namespace vierkant::rt;

namespace vkrt
{

__device__ __forceinline__ vec3 ld3(const float *p) { return vec3{p[0], p[1], p[2]}; }

__device__ __forceinline__ bool finite3(const vec3 &v)
{
    return __builtin_isfinite(v.x) && __builtin_isfinite(v.y) && __builtin_isfinite(v.z);
}

// ---------------------------------------------------------------------------------------------
// build kernels
// ---------------------------------------------------------------------------------------------
//! an indexed mesh as the build reads it: vertex i's position at pos + i * stride
struct mesh_view
{
    const uint8_t *pos;
    const uint32_t *idx;
    uint32_t stride, n_tri, n_vert;
};

//! triangle j's vertices; an index past the vertices reads vertex 0 (and `ok` turns false: the build then fails)
__device__ __forceinline__ void load_triangle(const mesh_view &m, uint32_t j, vec3 &v0, vec3 &v1, vec3 &v2, bool &ok)
{
    uint32_t i0 = m.idx[3 * (size_t)j], i1 = m.idx[3 * (size_t)j + 1], i2 = m.idx[3 * (size_t)j + 2];
    ok = i0 < m.n_vert && i1 < m.n_vert && i2 < m.n_vert;
    if(!ok) i0 = i1 = i2 = 0;
    v0 = ld3(reinterpret_cast<const float *>(m.pos + (size_t)i0 * m.stride));
    v1 = ld3(reinterpret_cast<const float *>(m.pos + (size_t)i1 * m.stride));
    v2 = ld3(reinterpret_cast<const float *>(m.pos + (size_t)i2 * m.stride));
}

//! a triangle's exact box, lo xyz then hi xyz. A triangle with a non-finite vertex never yields a finite t (the
//! reference test then produces NaN), so it gets an empty box and is never visited (returns false)
__device__ __forceinline__ bool triangle_box(const vec3 &v0, const vec3 &v1, const vec3 &v2, float b[6])
{
    const bool finite = finite3(v0) && finite3(v1) && finite3(v2);
    b[0] = finite ? fminf(fminf(v0.x, v1.x), v2.x) : FLT_MAX;
    b[1] = finite ? fminf(fminf(v0.y, v1.y), v2.y) : FLT_MAX;
    b[2] = finite ? fminf(fminf(v0.z, v1.z), v2.z) : FLT_MAX;
    b[3] = finite ? fmaxf(fmaxf(v0.x, v1.x), v2.x) : -FLT_MAX;
    b[4] = finite ? fmaxf(fmaxf(v0.y, v1.y), v2.y) : -FLT_MAX;
    b[5] = finite ? fmaxf(fmaxf(v0.z, v1.z), v2.z) : -FLT_MAX;
    return finite;
}

//! the bounds of the triangles' box centers, as one partial result per workgroup (k_morton combines them). No
//! atomics: 1.8M triangles' wave minima meeting on six words of one line took 1.92 ms of the 13.4 ms build (an
//! update of a line that every XCD writes costs 11 ns, one after the other). Two workgroups per CU keep the
//! partials few enough for every k_morton workgroup to read them all.
constexpr uint32_t BOUNDS_BLOCK = 512, BOUNDS_PARTIALS = 512;
__global__ void __launch_bounds__(BOUNDS_BLOCK) k_bounds(mesh_view m, float *__restrict__ partial,
                                                         uint32_t *__restrict__ err)
{
    __shared__ float part[6][BOUNDS_BLOCK / 64];
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    bool all_ok = true;
    for(uint32_t j = blockIdx.x * BOUNDS_BLOCK + threadIdx.x; j < m.n_tri; j += gridDim.x * BOUNDS_BLOCK)
    {
        vec3 v0, v1, v2;
        bool ok;
        float b[6];
        load_triangle(m, j, v0, v1, v2, ok);
        all_ok = all_ok && ok;
        if(!triangle_box(v0, v1, v2, b)) continue;
        for(int k = 0; k < 3; ++k)
        {
            const float c = 0.5f * b[k] + 0.5f * b[3 + k];
            lo[k] = fminf(lo[k], c);
            hi[k] = fmaxf(hi[k], c);
        }
    }
    if(!all_ok) atomicOr(err, 1u);
    for(int k = 0; k < 3; ++k)
    {
        for(int off = 32; off > 0; off >>= 1)
        {
            lo[k] = fminf(lo[k], __shfl_xor(lo[k], off));
            hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], off));
        }
        if((threadIdx.x & 63u) == 0)
        {
            part[k][threadIdx.x >> 6] = lo[k];
            part[3 + k][threadIdx.x >> 6] = hi[k];
        }
    }
    __syncthreads();
    if(threadIdx.x < 6)
    {
        float x = part[threadIdx.x][0];
        for(uint32_t w = 1; w < BOUNDS_BLOCK / 64; ++w)
            x = threadIdx.x < 3 ? fminf(x, part[threadIdx.x][w]) : fmaxf(x, part[threadIdx.x][w]);
        partial[6 * blockIdx.x + threadIdx.x] = x;
    }
}

__device__ __forceinline__ uint32_t spread10(uint32_t x)
{
    x &= 0x3ffu;
    x = (x | (x << 16)) & 0x030000ffu;
    x = (x | (x << 8)) & 0x0300f00fu;
    x = (x | (x << 4)) & 0x030c30c3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
}

//! 30-bit Morton code of each triangle's box center in the bounds that the n_partial partial results give. The
//! boxes are computed again from the mesh, which costs less than writing and reading them back would.
__global__ void __launch_bounds__(256) k_morton(mesh_view m, const float *__restrict__ partial, uint32_t n_partial,
                                                uint32_t *__restrict__ keys, uint32_t *__restrict__ vals)
{
    __shared__ float part[6][4];
    float cb[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for(uint32_t p = threadIdx.x; p < n_partial; p += 256)
        for(int a = 0; a < 6; ++a) cb[a] = a < 3 ? fminf(cb[a], partial[6 * p + a]) : fmaxf(cb[a], partial[6 * p + a]);
    for(int a = 0; a < 6; ++a)
    {
        for(int off = 32; off > 0; off >>= 1)
        {
            const float o = __shfl_xor(cb[a], off);
            cb[a] = a < 3 ? fminf(cb[a], o) : fmaxf(cb[a], o);
        }
        if((threadIdx.x & 63u) == 0) part[a][threadIdx.x >> 6] = cb[a];
    }
    __syncthreads();
    const uint32_t j = blockIdx.x * 256 + threadIdx.x;
    if(j >= m.n_tri) return;
    vec3 v0, v1, v2;
    bool ok;
    float b[6];
    load_triangle(m, j, v0, v1, v2, ok);
    uint32_t code = 0;
    if(triangle_box(v0, v1, v2, b))
    {
        uint32_t q[3];
        for(int a = 0; a < 3; ++a)
        {
            const float lo = fminf(fminf(part[a][0], part[a][1]), fminf(part[a][2], part[a][3]));
            const float hi = fmaxf(fmaxf(part[3 + a][0], part[3 + a][1]), fmaxf(part[3 + a][2], part[3 + a][3]));
            float c = 0.5f * b[a] + 0.5f * b[3 + a];
            float ext = hi - lo;
            float f = ext > 0.f ? (c - lo) / ext : 0.5f;
            f = fminf(fmaxf(f, 0.f), 1.f);
            q[a] = min(1023u, static_cast<uint32_t>(f * 1024.f));
        }
        code = (spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2]);
    }
    keys[j] = code;
    vals[j] = j;
}

__device__ __forceinline__ int delta(const uint32_t *__restrict__ keys, int n, int i, int j)
{
    if(j < 0 || j >= n) return -1;
    uint32_t a = keys[i], b = keys[j];
    if(a == b) return 32 + __clz(static_cast<uint32_t>(i ^ j));
    return __clz(a ^ b);
}

//! Karras 2012 binary radix tree. child refs: >= 0 internal node, < 0 leaf at sorted position ~ref.
__global__ void k_karras(const uint32_t *__restrict__ keys, int n, int2 *__restrict__ child, uint2 *__restrict__ range)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n - 1) return;
    const int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = delta(keys, n, i, i - d);
    int lmax = 2;
    while(delta(keys, n, i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for(int t = lmax / 2; t >= 1; t /= 2)
        if(delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = delta(keys, n, i, j);
    int s = 0;
    for(int div = 2;; div *= 2)
    {
        int t = (l + div - 1) / div;
        if(delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
        if(t <= 1) break;
    }
    const int gamma = i + s * d + min(d, 0);
    const int first = min(i, j), last = max(i, j);
    int left = (first == gamma) ? ~gamma : gamma;
    int right = (last == gamma + 1) ? ~(gamma + 1) : gamma + 1;
    child[i] = make_int2(left, right);
    range[i] = make_uint2(first, last);
}

//! (box arrays are 8-byte aligned: three 8-byte accesses per box)
__device__ __forceinline__ void load_box(const float *p, float b[6])
{
    const float2 *q = reinterpret_cast<const float2 *>(p);
    for(int a = 0; a < 3; ++a)
    {
        const float2 v = q[a];
        b[2 * a] = v.x, b[2 * a + 1] = v.y;
    }
}

__device__ __forceinline__ void store_box(float *p, const float b[6])
{
    float2 *q = reinterpret_cast<float2 *>(p);
    for(int a = 0; a < 3; ++a) q[a] = make_float2(b[2 * a], b[2 * a + 1]);
}

//! the triangles in leaf order, straight from the mesh: their leaf records (material and flags cleared) and, with
//! BOXES, their boxes
template<bool BOXES>
__global__ void __launch_bounds__(256) k_leaves(mesh_view m, const uint32_t *__restrict__ order,
                                                float *__restrict__ tbox, float4 *__restrict__ tris)
{
    const uint32_t j = blockIdx.x * 256 + threadIdx.x;
    if(j >= m.n_tri) return;
    const uint32_t src = min(order[j], m.n_tri - 1u);// (a malformed tree, rejected for its depth, leaves gaps)
    vec3 v0, v1, v2;
    bool ok;
    load_triangle(m, src, v0, v1, v2, ok);
    if constexpr(BOXES)
    {
        float b[6];
        triangle_box(v0, v1, v2, b);
        store_box(tbox + 6 * (size_t)j, b);
    }
    const vec3 e1 = v1 - v0, e2 = v2 - v0;
    float4 *t = tris + (TRI_BYTES / 16) * (size_t)j;
    t[0] = make_float4(v0.x, v0.y, v0.z, e1.x);
    t[1] = make_float4(e1.y, e1.z, e2.x, e2.y);
    t[2] = make_float4(e2.z, __uint_as_float(src), 0.f, 0.f);
    t[3] = make_float4(0.f, 0.f, 0.f, 0.f);
}

//! Node boxes without a bottom-up hand-off. Every internal node covers a contiguous run [first, last] of the
//! leaf order (`range`), so its box is the union of those leaves' boxes. The leaves are cut into segments of
//! BOX_SEG: k_box_scan writes, per leaf, the union from its segment's start (pre) and to its segment's end
//! (suf), and each segment's union (level 0 of a sparse table, levels 1.. by k_box_sparse: level k holds the
//! union of 2^k segments from each start). A run that crosses segments is suf[first], pre[last] and at most two
//! overlapping table entries; a run inside one segment is pre or suf when it touches the segment's start or
//! end, else a loop over its (at most BOX_SEG - 2) leaves. Every pass reads what earlier kernels wrote, so no
//! box crosses between workgroups, or XCDs, inside a kernel. A min or max is exact whatever the grouping, so
//! the boxes are the ones the pairwise union up the tree gives; only leaves' boxes are combined (the padding
//! past the last leaf is never read into a union).
constexpr uint32_t BOX_SEG = 64;

__device__ __forceinline__ void box_union(float a[6], const float b[6])
{
    for(int k = 0; k < 3; ++k) a[k] = fminf(a[k], b[k]);
    for(int k = 3; k < 6; ++k) a[k] = fmaxf(a[k], b[k]);
}

//! one segment of BOX_SEG leaves per workgroup (one wave): inclusive prefix and suffix unions in LDS
__global__ void __launch_bounds__(BOX_SEG) k_box_scan(uint32_t n, const float *__restrict__ tbox,
                                                      float *__restrict__ pre, float *__restrict__ suf,
                                                      float *__restrict__ seg)
{
    __shared__ float sp[6][BOX_SEG], ss[6][BOX_SEG];
    const uint32_t t = threadIdx.x, j = blockIdx.x * BOX_SEG + t;
    const uint32_t cnt = min(BOX_SEG, n - blockIdx.x * BOX_SEG);// leaves in this segment
    float a[6], b[6];
    if(t < cnt) load_box(tbox + 6 * (size_t)j, a);
    else
        for(int k = 0; k < 6; ++k) a[k] = 0.f;// past the last leaf: never combined into a leaf's union
    for(int k = 0; k < 6; ++k) b[k] = a[k];
    for(uint32_t off = 1; off < BOX_SEG; off <<= 1)
    {
        for(int k = 0; k < 6; ++k)
        {
            sp[k][t] = a[k];
            ss[k][t] = b[k];
        }
        __syncthreads();
        if(t >= off)
        {
            float o[6];
            for(int k = 0; k < 6; ++k) o[k] = sp[k][t - off];
            box_union(a, o);
        }
        if(t + off < cnt)
        {
            float o[6];
            for(int k = 0; k < 6; ++k) o[k] = ss[k][t + off];
            box_union(b, o);
        }
        __syncthreads();
    }
    if(t < cnt)
    {
        store_box(pre + 6 * (size_t)j, a);
        store_box(suf + 6 * (size_t)j, b);
    }
    if(t == 0)
        store_box(seg + 6 * (size_t)blockIdx.x, b);// leaf 0's suffix: the segment
}

//! sparse-table levels k .. k + 2 from level k - 1: entry i of level k + d is the union of 2^(d + 1) entries of level
//! k - 1, 2^(k - 1) apart, while the last of them is inside (i + 2^(k + d) <= nseg). Three levels a launch: the
//! table of 1.8M leaves has 15, and a launch each took 3 us of which the work was a fraction.
constexpr uint32_t SPARSE_LEVELS = 3;
__global__ void __launch_bounds__(256) k_box_sparse(uint32_t nseg, uint32_t k, uint32_t levels, float *__restrict__ table)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    const uint32_t step = 1u << (k - 1);
    if((size_t)i + 2 * step > nseg) return;
    const float *from = table + 6 * ((size_t)(k - 1) * nseg + i);
    float a[6], b[6];
    load_box(from, a);
    uint32_t taken = 1;
    for(uint32_t d = 0; d < SPARSE_LEVELS && k + d < levels; ++d)
    {
        const uint32_t want = 2u << d;
        if((size_t)i + (size_t)want * step > nseg) return;
        for(; taken < want; ++taken)
        {
            load_box(from + 6 * (size_t)taken * step, b);
            box_union(a, b);
        }
        store_box(table + 6 * ((size_t)(k + d) * nseg + i), a);
    }
}

//! the leaves' boxes and their unions, as k_layout reads them
struct leaf_unions
{
    const float *tbox, *pre, *suf, *table;
    uint32_t n, nseg;
};

//! the union of leaf boxes first .. last
__device__ __forceinline__ void run_box(const leaf_unions &l, uint32_t first, uint32_t last, float o[6])
{
    const uint32_t sf = first / BOX_SEG, sl = last / BOX_SEG;
    float x[6];
    if(sf == sl)
    {
        const bool at_end = last % BOX_SEG == BOX_SEG - 1 || last == l.n - 1;
        if(first % BOX_SEG == 0) load_box(l.pre + 6 * (size_t)last, o);
        else if(at_end) load_box(l.suf + 6 * (size_t)first, o);
        else
        {
            load_box(l.tbox + 6 * (size_t)first, o);
            for(uint32_t j = first + 1; j <= last; ++j)
            {
                load_box(l.tbox + 6 * (size_t)j, x);
                box_union(o, x);
            }
        }
    }
    else
    {
        load_box(l.suf + 6 * (size_t)first, o);
        load_box(l.pre + 6 * (size_t)last, x);
        box_union(o, x);
        if(sl > sf + 1)
        {
            const uint32_t lo = sf + 1, count = sl - 1 - lo + 1;
            const uint32_t k = 31u - __builtin_clz(count);
            load_box(l.table + 6 * ((size_t)k * l.nseg + lo), x);
            box_union(o, x);
            load_box(l.table + 6 * ((size_t)k * l.nseg + (sl - 1) - (1u << k) + 1), x);
            box_union(o, x);
        }
    }
}

//! the sparse table's depth for nseg segments: levels 0 .. floor(log2(nseg))
static uint32_t box_levels(uint32_t nseg)
{
    uint32_t l = 1;
    while((2ull << (l - 1)) <= nseg) ++l;
    return l;
}

__device__ __forceinline__ float pad_lo(float x) { return x - fabsf(x) * BOX_PAD; }
__device__ __forceinline__ float pad_hi(float x) { return x + fabsf(x) * BOX_PAD; }

//! BVH2 node i from its children's leaf runs: child k's box is the union over its run (each node is one node's
//! child, so no node's box is computed twice, and none is stored on its own)
__global__ void __launch_bounds__(256) k_layout(leaf_unions l, const int2 *__restrict__ child,
                                                const uint2 *__restrict__ range, uint32_t max_leaf,
                                                vkrt_bvh_node *__restrict__ nodes)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if(i + 1 >= l.n) return;
    const int2 c = child[i];
    float bx[2][6];
    int ref[2];
    const int cr[2] = {c.x, c.y};
    for(int k = 0; k < 2; ++k)
    {
        uint32_t first, last;
        if(cr[k] < 0)
        {
            first = last = ~cr[k];
            load_box(l.tbox + 6 * (size_t)first, bx[k]);
        }
        else
        {
            const uint2 cr_range = range[cr[k]];
            first = cr_range.x, last = cr_range.y;
            run_box(l, first, last, bx[k]);
        }
        const uint32_t count = last - first + 1;
        ref[k] = (cr[k] < 0 || count <= max_leaf) ? ~static_cast<int>((first << 3) | (count - 1)) : cr[k];
        for(int a = 0; a < 3; ++a) bx[k][a] = pad_lo(bx[k][a]);
        for(int a = 3; a < 6; ++a) bx[k][a] = pad_hi(bx[k][a]);
    }
    vkrt_bvh_node nd;
    nd.a = make_float4(bx[0][0], bx[0][3], bx[0][1], bx[0][4]);
    nd.b = make_float4(bx[1][0], bx[1][3], bx[1][1], bx[1][4]);
    nd.c = make_float4(bx[0][2], bx[0][5], bx[1][2], bx[1][5]);
    nd.d = make_int4(ref[0], ref[1], 0, 0);
    nodes[i] = nd;
}

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------
//! what a build's kernels count and its host side reads: one block in device memory, cleared at the start of a
//! build and copied to the context's pinned host memory by k_report (a kernel's store and the synchronization
//! take 10 us; a copy into pageable memory took 25 us besides). Counters that many workgroups update lie on
//! lines of their own.
struct ploc_round
{
    uint32_t nc, base, buf;// clusters, nodes made so far, which of the two lists holds the clusters
};
constexpr uint32_t MAX_LEVELS = STACK_SIZE + 2;// of the 4-wide collapse: each goes at least one binary level down
struct bvh_state
{
    uint32_t err;// an index past the vertices
    uint32_t pad0[31];
    double sah;  // sum of the children's SAH terms (divided by the root's area on the host)
    uint32_t pad1[30];
    uint32_t leaves;
    uint32_t pad2[31];
    uint32_t depth;// of the binary tree, its root counting 1
    uint32_t pad3[31];
    uint32_t stack;// worst-case traversal stack of the 4-wide tree
    uint32_t pad4[31];
    uint32_t level[MAX_LEVELS + 2];// 4-wide nodes per level
    uint32_t top_levels;           // levels that the collapse's first launch took
    ploc_round ploc[2];            // the clusters before an even and an odd round
    uint32_t ploc_left, ploc_nodes;// clusters left and nodes made after the last tail
    vkrt_bvh_node root;  // of the binary tree, where one is given
    vkrt_bvh4_node root4;// of the 4-wide tree
};

__global__ void __launch_bounds__(256) k_state_clear(bvh_state *__restrict__ st)
{
    uint32_t *w = reinterpret_cast<uint32_t *>(st);
    for(uint32_t i = threadIdx.x; i < sizeof(bvh_state) / 4; i += 256) w[i] = 0u;
}

__global__ void __launch_bounds__(256) k_report(const bvh_state *__restrict__ st, const vkrt_bvh_node *__restrict__ nodes,
                                                const vkrt_bvh4_node *__restrict__ nodes4, bvh_state *__restrict__ host)
{
    const uint32_t *src = reinterpret_cast<const uint32_t *>(st);
    uint32_t *dst = reinterpret_cast<uint32_t *>(host);
    for(uint32_t i = threadIdx.x; i < offsetof(bvh_state, root) / 4; i += 256) dst[i] = src[i];
    if(nodes && threadIdx.x < sizeof(vkrt_bvh_node) / 4)
        dst[offsetof(bvh_state, root) / 4 + threadIdx.x] = reinterpret_cast<const uint32_t *>(nodes)[threadIdx.x];
    if(nodes4 && threadIdx.x < sizeof(vkrt_bvh4_node) / 4)
        dst[offsetof(bvh_state, root4) / 4 + threadIdx.x] = reinterpret_cast<const uint32_t *>(nodes4)[threadIdx.x];
}

//! the state as the host reads it, once everything queued before has run; the root nodes of what is given too
static const bvh_state &read_state(vkrt_ctx *ctx, const vkrt_bvh_node *nodes, const vkrt_bvh4_node *nodes4)
{
    bvh_state *host = ctx->pinned_as<bvh_state>();
    k_report<<<1, 256, 0, ctx->stream>>>(ctx->state.as<bvh_state>(), nodes, nodes4, host);
    VKRT_HIP(hipGetLastError());
    VKRT_HIP(hipStreamSynchronize(ctx->stream));
    return *host;
}

//! a single leaf's bounds (at most 8 triangles): the union of its triangles' boxes (tbox, in leaf order), padded
//! like every node box
static void single_leaf_info(vkrt_bvh *bvh, const float *tbox, hipStream_t s)
{
    vkrt_bvh_info &info = bvh->info;
    info.depth = 1;
    info.sah_cost = 0.f;
    info.n_leaves = bvh->empty ? 0 : 1;
    if(bvh->empty) return;
    const uint32_t v = static_cast<uint32_t>(~bvh->root_ref), first = v >> 3, count = (v & 7u) + 1;
    std::vector<float> box(6 * (size_t)count);
    VKRT_HIP(hipMemcpyAsync(box.data(), tbox + 6 * (size_t)first, box.size() * 4, hipMemcpyDeviceToHost, s));
    VKRT_HIP(hipStreamSynchronize(s));
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for(uint32_t k = 0; k < count; ++k)
        for(int a = 0; a < 3; ++a)
        {
            lo[a] = std::min(lo[a], box[6 * (size_t)k + a]);
            hi[a] = std::max(hi[a], box[6 * (size_t)k + 3 + a]);
        }
    for(int a = 0; a < 3; ++a)
    {
        info.bounds[a] = lo[a] - std::fabs(lo[a]) * BOX_PAD;
        info.bounds[3 + a] = hi[a] + std::fabs(hi[a]) * BOX_PAD;
    }
}

//! the binary tree a build works on
struct binary_tree
{
    vkrt_bvh_node *nodes;
    int2 *child;
    uint2 *range;// the run of leaves below each node
};

static void build_topology_ploc(vkrt_ctx *ctx, vkrt_bvh *bvh, const mesh_view &mesh, const binary_tree &bin,
                                const uint32_t *sorted);

static void build_topology(vkrt_ctx *ctx, vkrt_bvh *bvh, const mesh_view &mesh, const binary_tree &bin)
{
    hipStream_t s = ctx->stream;
    const uint32_t n = bvh->n_tri;
    // scratch: centroid bounds, sort keys, sort temp
    device_buffer &tmp = ctx->scratch[2];
    const size_t key_bytes = (size_t)n * sizeof(uint32_t), partial_bytes = BOUNDS_PARTIALS * 6 * sizeof(float);
    tmp.reserve(partial_bytes + 2 * key_bytes + radix_sort_temp_bytes(n));
    float *partial = tmp.as<float>();
    uint32_t *keys = reinterpret_cast<uint32_t *>(tmp.as<uint8_t>() + partial_bytes);
    void *sort_tmp = tmp.as<uint8_t>() + partial_bytes + 2 * key_bytes;
    // PLOC puts the sorted triangles into an order of its own
    const bool ploc = bvh->builder == VKRT_BUILDER_PLOC && n >= 2;
    uint32_t *order = ploc ? keys + n : bvh->order.as<uint32_t>();

    bvh_state *st = ctx->state.as<bvh_state>();
    k_state_clear<<<1, 256, 0, s>>>(st);
    const uint32_t n_partial = std::min(BOUNDS_PARTIALS, div_up(n, BOUNDS_BLOCK));
    k_bounds<<<n_partial, BOUNDS_BLOCK, 0, s>>>(mesh, partial, &st->err);
    k_morton<<<div_up(n, 256), 256, 0, s>>>(mesh, partial, n_partial, keys, order);
    radix_sort_pairs(s, keys, order, n, 30, sort_tmp);
    if(n >= 2)
    {
        const uint32_t ni = n - 1;
        if(ploc) build_topology_ploc(ctx, bvh, mesh, bin, order);
        else
            k_karras<<<div_up(ni, 256), 256, 0, s>>>(keys, (int)n, bin.child, bin.range);
    }
    VKRT_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------
// PLOC (Meister & Bittner 2018): agglomerative clustering over the Morton-sorted leaves. Each round every
// cluster finds, within PLOC_RADIUS positions of the sorted list, the cluster whose merged box has the
// smallest surface area; mutual nearest neighbours merge into a new node at the lower position, and the list
// is compacted. Pairs are ordered by (area, lower position, higher position), so the globally smallest pair
// is always mutual and every round merges. Nodes are numbered down from n - 2 in merge order, so the root is
// node 0 and parents precede children; leaves are finally put in depth-first order so that every subtree
// covers a contiguous range, which the leaf collapse of k_layout and the refit rely on.
//
// A 1.8M-triangle build takes 64 rounds, 30 of them over fewer than 1,024 clusters, so what a round costs besides
// its work decides: two launches a round, with no count read by the host, and the last rounds in one workgroup
// that keeps its clusters in LDS (nine launches and a host round trip a round took 5.0 ms; now 1.1 ms).
// ---------------------------------------------------------------------------------------------
constexpr int PLOC_RADIUS = 16;    // default search radius
constexpr int PLOC_MAX_RADIUS = 32;
constexpr int PLOC_BLOCK = 256;
constexpr int PLOC_SPAN = 4 * PLOC_BLOCK;// positions whose neighbour a workgroup finds: its tile and a radius each side
constexpr uint32_t PLOC_TAIL = 1024;     // clusters that one workgroup finishes
constexpr uint32_t PLOC_MAX_CLIMB = 4096;// bound of the upward walks; deeper trees are rejected after the collapse

//! the positions of a tile whose neighbours' neighbours are inside the workgroup's span
__host__ __device__ constexpr uint32_t ploc_tile(int radius) { return PLOC_SPAN - 2 * radius; }

//! what a cluster does in a round: merge with the cluster `code` positions on, or one of these
constexpr int8_t PLOC_GONE = 0, PLOC_STAYS = -128;

//! the two cluster lists: box corners, with the cluster's node (a leaf: ~position) in lo.w and its leaf count in
//! hi.w, as bits
struct ploc_lists
{
    float4 *lo[2], *hi[2];
};

//! the tree under construction: node k's children, leaf count and parent
struct ploc_tree
{
    int2 *child;
    uint32_t *cnt;
    int32_t *parent;
    uint32_t ni;
};

__device__ __forceinline__ float merged_half_area(const float2 a[3], const float2 b[3])
{
    const float dx = fmaxf(a[0].y, b[0].y) - fminf(a[0].x, b[0].x);
    const float dy = fmaxf(a[1].y, b[1].y) - fminf(a[1].x, b[1].x);
    const float dz = fmaxf(a[2].y, b[2].y) - fminf(a[2].x, b[2].x);
    return dx * dy + dy * dz + dz * dx;
}

__global__ void __launch_bounds__(256) k_ploc_init(mesh_view m, const uint32_t *__restrict__ order, float4 *__restrict__ lo,
                                                   float4 *__restrict__ hi, bvh_state *__restrict__ st)
{
    const uint32_t j = blockIdx.x * 256 + threadIdx.x;
    if(j == 0) st->ploc[0] = ploc_round{m.n_tri, 0u, 0u};
    if(j >= m.n_tri) return;
    vec3 v0, v1, v2;
    bool ok;
    float b[6];
    load_triangle(m, order[j], v0, v1, v2, ok);
    triangle_box(v0, v1, v2, b);
    lo[j] = make_float4(b[0], b[1], b[2], __int_as_float(~static_cast<int32_t>(j)));
    hi[j] = make_float4(b[3], b[4], b[5], __uint_as_float(1u));
}

//! node `id` over clusters a and b (their node and leaf count); returns its leaf count
__device__ __forceinline__ uint32_t ploc_node(const ploc_tree &t, int32_t id, int32_t a, int32_t b, uint32_t na, uint32_t nb)
{
    t.child[id] = make_int2(a, b);
    t.cnt[id] = na + nb;
    if(a >= 0) t.parent[a] = id;
    if(b >= 0) t.parent[b] = id;
    return na + nb;
}

//! the nearest neighbour of every cluster within the window (ties go to the smallest position, which is the
//! smallest pair in (area, lower, higher) order), and what each cluster does: code, and per tile the clusters kept
//! and merged. A thread takes four neighbouring positions, so a box read from LDS serves four of them (one position
//! a thread read 64 16-B words each, 180 us for 1.8M clusters); boxes lie by position mod 4, so that a wave's
//! reads are consecutive. RADIUS 0: the radius is the argument.
template<int RADIUS>
__global__ void __launch_bounds__(PLOC_BLOCK) k_ploc_nn(const bvh_state *__restrict__ st, uint32_t parity, int radius_arg,
                                                        ploc_lists l, int8_t *__restrict__ code,
                                                        uint32_t *__restrict__ counts)
{
    constexpr int QUARTER = (PLOC_SPAN + 2 * PLOC_MAX_RADIUS) / 4;
    __shared__ float2 box[3][4 * QUARTER];
    __shared__ int16_t nn[PLOC_SPAN];
    __shared__ uint32_t wave_count[PLOC_BLOCK / 64];
    const int radius = RADIUS ? RADIUS : radius_arg;
    const ploc_round round = st->ploc[parity];
    const int nc = static_cast<int>(round.nc), tile = static_cast<int>(ploc_tile(radius));
    const int start = static_cast<int>(blockIdx.x) * tile;
    if(round.nc <= PLOC_TAIL || start >= nc) return;
    const float4 *__restrict__ lo = l.lo[round.buf], *__restrict__ hi = l.hi[round.buf];
    const int span0 = start - radius;// the position of nn[0]
    for(int s = threadIdx.x; s < PLOC_SPAN + 2 * radius; s += PLOC_BLOCK)
    {
        const int j = span0 - radius + s;
        if(j < 0 || j >= nc) continue;
        const float4 a = lo[j], b = hi[j];
        const int slot = (s & 3) * QUARTER + (s >> 2);
        box[0][slot] = make_float2(a.x, b.x);
        box[1][slot] = make_float2(a.y, b.y);
        box[2][slot] = make_float2(a.z, b.z);
    }
    __syncthreads();
    const int t = static_cast<int>(threadIdx.x);
    auto load = [&](int c, float2 v[3]) {
        const int slot = (c & 3) * QUARTER + t + (c >> 2);
        v[0] = box[0][slot], v[1] = box[1][slot], v[2] = box[2][slot];
    };
    float2 own[4][3];
    for(int k = 0; k < 4; ++k) load(k + radius, own[k]);
    float best[4] = {0.f, 0.f, 0.f, 0.f};
    int best_c[4] = {-1, -1, -1, -1};
    const int j0 = span0 - radius + 4 * t;
    auto step = [&](int c) {
        const int j = j0 + c;
        const bool there = j >= 0 && j < nc;
        float2 v[3];
        load(c, v);
#pragma unroll
        for(int k = 0; k < 4; ++k)
        {
            const int o = c - radius - k;
            if(o < -radius || o > radius || o == 0) continue;
            const float d = merged_half_area(own[k], v);
            if(there && (best_c[k] < 0 || d < best[k]))
            {
                best[k] = d;
                best_c[k] = c;
            }
        }
    };
    if constexpr(RADIUS != 0)
    {
#pragma unroll
        for(int c = 0; c < 2 * RADIUS + 4; ++c) step(c);
    }
    else
        for(int c = 0; c < 2 * radius + 4; ++c) step(c);
    for(int k = 0; k < 4; ++k) nn[4 * t + k] = static_cast<int16_t>(4 * t + best_c[k] - radius);
    __syncthreads();
    uint32_t kept = 0, merged = 0;
    for(int m = 0; m < 4; ++m)
    {
        const int i = t + m * PLOC_BLOCK;
        const bool mine = i >= radius && i < PLOC_SPAN - radius && span0 + i < nc;
        int8_t what = PLOC_GONE;
        if(mine)
        {
            const int j = nn[i];
            const bool mutual = nn[j] == i;
            what = !mutual ? PLOC_STAYS : (i < j ? static_cast<int8_t>(j - i) : PLOC_GONE);
            code[span0 + i] = what;
        }
        kept += __popcll(__ballot(mine && what != PLOC_GONE));
        merged += __popcll(__ballot(mine && what > 0));
    }
    if((threadIdx.x & 63u) == 0) wave_count[threadIdx.x >> 6] = kept | (merged << 16);
    __syncthreads();
    if(threadIdx.x == 0)
        counts[blockIdx.x] = (wave_count[0] + wave_count[1]) + (wave_count[2] + wave_count[3]);
}

//! the round's merges and the compacted list. A tile's place is the sum of the tiles before it, which every
//! workgroup adds up for itself (at most 1,900 of them at 1.8M clusters, from L2): no scan launches and no waiting.
__global__ void __launch_bounds__(PLOC_BLOCK) k_ploc_merge(bvh_state *__restrict__ st, uint32_t parity, int radius,
                                                           ploc_lists l, const int8_t *__restrict__ code,
                                                           const uint32_t *__restrict__ counts, ploc_tree tree)
{
    __shared__ uint32_t wave_kept[PLOC_BLOCK / 64], wave_merged[PLOC_BLOCK / 64], wave_sum[PLOC_BLOCK / 64];
    const ploc_round round = st->ploc[parity];
    const uint32_t tile = ploc_tile(radius), start = blockIdx.x * tile;
    if(round.nc <= PLOC_TAIL)
    {
        if(blockIdx.x == 0 && threadIdx.x == 0) st->ploc[parity ^ 1u] = round;// left to the tail
        return;
    }
    if(start >= round.nc) return;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t kept = 0, merged = 0;// of the tiles before
    for(uint32_t b = threadIdx.x; b < blockIdx.x; b += PLOC_BLOCK)
    {
        const uint32_t c = counts[b];
        kept += c & 0xffffu;
        merged += c >> 16;
    }
    for(int off = 32; off > 0; off >>= 1)
    {
        kept += __shfl_xor(kept, off);
        merged += __shfl_xor(merged, off);
    }
    int8_t what[4];
    uint32_t mine = 0;// kept | merged << 16 of this thread's four positions
    for(uint32_t k = 0; k < 4; ++k)
    {
        const uint32_t p = 4 * threadIdx.x + k;
        what[k] = p < tile && start + p < round.nc ? code[start + p] : PLOC_GONE;
        mine += (what[k] != PLOC_GONE ? 1u : 0u) + (what[k] > 0 ? 0x10000u : 0u);
    }
    uint32_t scan = mine;
    for(int off = 1; off < 64; off <<= 1)
    {
        const uint32_t y = __shfl_up(scan, off);
        if(lane >= (uint32_t)off) scan += y;
    }
    if(lane == 63) wave_sum[wave] = scan;
    if(lane == 0)
    {
        wave_kept[wave] = kept;
        wave_merged[wave] = merged;
    }
    __syncthreads();
    kept = (wave_kept[0] + wave_kept[1]) + (wave_kept[2] + wave_kept[3]);
    merged = (wave_merged[0] + wave_merged[1]) + (wave_merged[2] + wave_merged[3]);
    uint32_t before = scan - mine, total = 0;
    for(uint32_t w = 0; w < PLOC_BLOCK / 64; ++w)
    {
        before += w < wave ? wave_sum[w] : 0u;
        total += wave_sum[w];
    }
    if(start + tile >= round.nc && threadIdx.x == 0)
        st->ploc[parity ^ 1u] = ploc_round{kept + (total & 0xffffu), round.base + merged + (total >> 16), round.buf ^ 1u};
    const float4 *__restrict__ lo = l.lo[round.buf], *__restrict__ hi = l.hi[round.buf];
    float4 *__restrict__ out_lo = l.lo[round.buf ^ 1u], *__restrict__ out_hi = l.hi[round.buf ^ 1u];
    uint32_t pos = kept + (before & 0xffffu), made = round.base + merged + (before >> 16);
    for(uint32_t k = 0; k < 4; ++k)
    {
        if(what[k] == PLOC_GONE) continue;
        const uint32_t i = start + 4 * threadIdx.x + k;
        float4 a = lo[i], b = hi[i];
        if(what[k] > 0)
        {
            const float4 c = lo[i + what[k]], d = hi[i + what[k]];
            const int32_t id = static_cast<int32_t>(tree.ni - 1u - made);
            ++made;
            const uint32_t n = ploc_node(tree, id, __float_as_int(a.w), __float_as_int(c.w), __float_as_uint(b.w),
                                         __float_as_uint(d.w));
            a = make_float4(fminf(a.x, c.x), fminf(a.y, c.y), fminf(a.z, c.z), __int_as_float(id));
            b = make_float4(fmaxf(b.x, d.x), fmaxf(b.y, d.y), fmaxf(b.z, d.z), __uint_as_float(n));
        }
        out_lo[pos] = a;
        out_hi[pos] = b;
        ++pos;
    }
}

//! every remaining round of at most PLOC_TAIL clusters in one workgroup, one cluster a thread (three barriers a
//! round, 1.5 us, against the two launches of the kernels above)
__global__ void __launch_bounds__(PLOC_TAIL) k_ploc_tail(bvh_state *__restrict__ st, uint32_t parity, int radius,
                                                         ploc_lists l, ploc_tree tree)
{
    __shared__ float2 box[3][PLOC_TAIL];
    __shared__ int32_t node[PLOC_TAIL];
    __shared__ uint32_t leaves[PLOC_TAIL];
    __shared__ int16_t nn[PLOC_TAIL];
    __shared__ uint32_t wave_sum[PLOC_TAIL / 64];
    const ploc_round round = st->ploc[parity];
    const int i = static_cast<int>(threadIdx.x);
    if(round.nc > PLOC_TAIL)
    {
        if(i == 0) st->ploc_left = round.nc;
        return;
    }
    int nc = static_cast<int>(round.nc);
    uint32_t base = round.base;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    float2 me[3];
    int32_t id = 0;
    uint32_t n = 0;
    if(i < nc)
    {
        const float4 a = l.lo[round.buf][i], b = l.hi[round.buf][i];
        me[0] = make_float2(a.x, b.x), me[1] = make_float2(a.y, b.y), me[2] = make_float2(a.z, b.z);
        id = __float_as_int(a.w);
        n = __float_as_uint(b.w);
        for(int k = 0; k < 3; ++k) box[k][i] = me[k];
        node[i] = id;
        leaves[i] = n;
    }
    __syncthreads();
    while(nc > 1)
    {
        const bool active = i < nc;
        int best_j = -1;
        if(active)
        {
            float best = 0.f;
            const int first = max(0, i - radius), last = min(nc - 1, i + radius);
            for(int j = first; j <= last; ++j)
            {
                if(j == i) continue;
                const float2 v[3] = {box[0][j], box[1][j], box[2][j]};
                const float d = merged_half_area(me, v);
                if(best_j < 0 || d < best)
                {
                    best = d;
                    best_j = j;
                }
            }
            nn[i] = static_cast<int16_t>(best_j);
        }
        __syncthreads();
        const bool mutual = active && nn[best_j] == i;
        const bool merges = mutual && i < best_j, keep = active && !(mutual && i > best_j);
        float2 other[3];
        int32_t other_id = 0;
        uint32_t other_n = 0;
        if(merges)
        {
            for(int k = 0; k < 3; ++k) other[k] = box[k][best_j];
            other_id = node[best_j];
            other_n = leaves[best_j];
        }
        const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
        const uint64_t km = __ballot(keep), mm = __ballot(merges);
        if(lane == 0) wave_sum[wave] = __popcll(km) | (static_cast<uint32_t>(__popcll(mm)) << 16);
        __syncthreads();
        uint32_t before = 0, total = 0;
        for(uint32_t w = 0; w < PLOC_TAIL / 64; ++w)
        {
            before += w < wave ? wave_sum[w] : 0u;
            total += wave_sum[w];
        }
        if(merges)
        {
            const int32_t made = static_cast<int32_t>(tree.ni - 1u - (base + (before >> 16) + __popcll(mm & below)));
            n = ploc_node(tree, made, id, other_id, n, other_n);
            id = made;
            for(int k = 0; k < 3; ++k)
                me[k] = make_float2(fminf(me[k].x, other[k].x), fmaxf(me[k].y, other[k].y));
        }
        if((total >> 16) == 0u)
        {
            // every round merges the smallest pair at least, unless areas are NaN (an infinite extent times zero):
            // the build then fails
            if(i == 0) st->ploc_left = 0u;
            return;
        }
        const int to = static_cast<int>((before & 0xffffu) + __popcll(km & below));
        if(keep)
        {
            for(int k = 0; k < 3; ++k) box[k][to] = me[k];
            node[to] = id;
            leaves[to] = n;
        }
        nc = static_cast<int>(total & 0xffffu);
        base += total >> 16;
        __syncthreads();
        if(i < nc)
        {
            for(int k = 0; k < 3; ++k) me[k] = box[k][i];
            id = node[i];
            n = leaves[i];
        }
    }
    if(i == 0)
    {
        st->ploc_left = 1u;
        st->ploc_nodes = base;
    }
}

__device__ __forceinline__ uint32_t leaf_count(const uint32_t *__restrict__ cnt, int32_t ref)
{
    return ref < 0 ? 1u : cnt[ref];
}

//! the depth-first position of the first leaf of nodes a .. b - 1: the leaf counts of all left siblings on the way
//! up to a node before a, whose position an earlier launch found (parents precede children). Launched over
//! ranges that grow eightfold, so a climb is a few steps (up to the root from everywhere took 199 us)
__global__ void __launch_bounds__(256) k_ploc_first(uint32_t a, uint32_t b, ploc_tree tree, uint32_t *__restrict__ first)
{
    const uint32_t k = a + blockIdx.x * 256 + threadIdx.x;
    if(k >= b) return;
    uint32_t off = 0;
    int32_t cur = static_cast<int32_t>(k);
    for(uint32_t step = 0; cur > 0 && step < PLOC_MAX_CLIMB; ++step)
    {
        const int32_t up = tree.parent[cur];
        const int2 c = tree.child[up];
        if(c.y == cur) off += leaf_count(tree.cnt, c.x);
        cur = up;
        if(cur > 0 && static_cast<uint32_t>(cur) < a)
        {
            off += first[cur];
            break;
        }
    }
    first[k] = off;
}

//! the leaves in depth-first order: each node's range, its leaf children's positions and their triangles
__global__ void __launch_bounds__(256) k_ploc_emit(ploc_tree tree, const uint32_t *__restrict__ first,
                                                   const uint32_t *__restrict__ order_in, uint32_t *__restrict__ order_out,
                                                   uint2 *__restrict__ range)
{
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if(k >= tree.ni) return;
    const uint32_t f = first[k];
    range[k] = make_uint2(f, f + tree.cnt[k] - 1u);
    int2 c = tree.child[k];
    const uint32_t right = f + leaf_count(tree.cnt, c.x);
    if(c.x < 0)
    {
        order_out[f] = order_in[~c.x];
        c.x = ~static_cast<int32_t>(f);
    }
    if(c.y < 0)
    {
        order_out[right] = order_in[~c.y];
        c.y = ~static_cast<int32_t>(right);
    }
    tree.child[k] = c;
}

static void build_topology_ploc(vkrt_ctx *ctx, vkrt_bvh *bvh, const mesh_view &mesh, const binary_tree &bin,
                                const uint32_t *sorted)
{
    hipStream_t s = ctx->stream;
    const int radius = bvh->ploc_radius ? static_cast<int>(bvh->ploc_radius) : PLOC_RADIUS;
    const uint32_t n = bvh->n_tri, ni = n - 1, tiles = div_up(n, ploc_tile(radius));
    // working set: two cluster lists, what each cluster does, counts per tile, the tree's counts, parents and
    // first leaves
    device_buffer &w = ctx->scratch[3];
    const size_t bytes = (size_t)n * 65 + (size_t)tiles * 4 + (size_t)ni * 12 + 512;
    w.reserve(bytes);
    uint8_t *q = w.as<uint8_t>();
    auto take = [&q](size_t b) {
        uint8_t *r = q;
        q += (b + 15) & ~size_t(15);
        return r;
    };
    ploc_lists l;
    for(int k = 0; k < 2; ++k)
    {
        l.lo[k] = reinterpret_cast<float4 *>(take((size_t)n * 16));
        l.hi[k] = reinterpret_cast<float4 *>(take((size_t)n * 16));
    }
    int8_t *code = reinterpret_cast<int8_t *>(take(n));
    uint32_t *counts = reinterpret_cast<uint32_t *>(take((size_t)tiles * 4));
    ploc_tree tree{bin.child, reinterpret_cast<uint32_t *>(take((size_t)ni * 4)),
                   reinterpret_cast<int32_t *>(take((size_t)ni * 4)), ni};
    uint32_t *first = reinterpret_cast<uint32_t *>(take((size_t)ni * 4));
    VKRT_REQUIRE(q <= w.as<uint8_t>() + bytes, "PLOC working set overrun");

    bvh_state *st = ctx->state.as<bvh_state>();
    k_ploc_init<<<div_up(n, 256), 256, 0, s>>>(mesh, sorted, l.lo[0], l.hi[0], st);
    // rounds are launched without asking how many clusters are left: as many as a list that shrinks by a fifth each
    // time needs (a round with too few clusters passes them on, 4 us), the tail, and eight more at a time while
    // the tail finds too many
    uint32_t round = 0, nc = n, todo = 0;
    for(double k = n; k > PLOC_TAIL; k *= 0.82) ++todo;
    while(true)
    {
        const uint32_t grid = div_up(nc, ploc_tile(radius));// (the list never grows)
        for(uint32_t stop = round + todo; round < stop; ++round)
        {
            if(radius == PLOC_RADIUS)
                k_ploc_nn<PLOC_RADIUS><<<grid, PLOC_BLOCK, 0, s>>>(st, round & 1u, radius, l, code, counts);
            else
                k_ploc_nn<0><<<grid, PLOC_BLOCK, 0, s>>>(st, round & 1u, radius, l, code, counts);
            k_ploc_merge<<<grid, PLOC_BLOCK, 0, s>>>(st, round & 1u, radius, l, code, counts, tree);
        }
        k_ploc_tail<<<1, PLOC_TAIL, 0, s>>>(st, round & 1u, radius, l, tree);
        const bvh_state &got = read_state(ctx, nullptr, nullptr);
        VKRT_REQUIRE(got.ploc_left >= 1 && got.ploc_left < nc, "PLOC made no progress");
        nc = got.ploc_left;
        if(nc == 1)
        {
            VKRT_REQUIRE(got.ploc_nodes == ni, "PLOC did not build n - 1 nodes");
            break;
        }
        todo = 8;
    }
    for(uint32_t a = 0, b = 1024; a < ni; a = b, b *= 8)
    {
        const uint32_t stop = std::min(b, ni);
        k_ploc_first<<<div_up(stop - a, 256), 256, 0, s>>>(a, stop, tree, first);
    }
    k_ploc_emit<<<div_up(ni, 256), 256, 0, s>>>(tree, first, sorted, bvh->order.as<uint32_t>(), bin.range);
    VKRT_HIP(hipGetLastError());
}

//! parts of one allocation, one after the other, each at a multiple of 256 B
static void place(device_buffer &mem, std::initializer_list<std::pair<vkrt_bvh::part *, size_t>> parts)
{
    size_t total = 0;
    for(const auto &[p, bytes]: parts) total += (bytes + 255) & ~size_t(255);
    mem.reserve(total);
    uint8_t *at = mem.as<uint8_t>();
    for(const auto &[p, bytes]: parts)
    {
        p->ptr = at;
        p->bytes = bytes;
        at += (bytes + 255) & ~size_t(255);
    }
}

//! the BVH's memory, with room for node_cap 4-wide nodes
static void allocate(vkrt_bvh *bvh, uint32_t node_cap)
{
    const size_t n = bvh->n_tri;
    // (a step at the last leaf reads one record past it)
    place(bvh->memory, {{&bvh->nodes4, (size_t)node_cap * sizeof(vkrt_bvh4_node)}, {&bvh->tris, (n + 1) * TRI_BYTES},
                        {&bvh->indices, n * 3 * sizeof(uint32_t)}, {&bvh->order, n * sizeof(uint32_t)},
                        {&bvh->wide_range, node_cap * sizeof(uint2)}});
    bvh->node_cap = node_cap;
    bvh->joint = static_cast<size_t>(bvh->tris.as<uint8_t>() - bvh->nodes4.as<uint8_t>()) + bvh->tris.bytes <= 0xffffffffull;
}

//! how many 4-wide nodes a build makes room for before it knows: measured over heightfields, spheres, the room and
//! triangle soups, both builders, a triangle takes 0.42 to 0.53 of a node at one triangle a leaf, 0.25 to 0.31 at two,
//! 0.15 to 0.20 at four and 0.07 to 0.11 at eight. A tree that needs more (a regular grid at one triangle a leaf:
//! 0.67) is collapsed again into a larger allocation. Knowing the place beforehand saves the build a copy of the
//! nodes and a second pass over the mesh, and the allocation overlaps the kernels queued before it.
static uint32_t node_guess(const vkrt_bvh *bvh)
{
    const double per_tri = 0.07 + 0.5 / bvh->max_leaf;
    return static_cast<uint32_t>(std::min<double>(bvh->n_tri, bvh->n_tri * per_tri + 8));
}

//! leaf records and boxes from the mesh, and the boxes' unions (in scratch): the start of a refit and, after the
//! topology, of a build
static leaf_unions leaf_pass(vkrt_ctx *ctx, vkrt_bvh *bvh, const mesh_view &mesh)
{
    hipStream_t s = ctx->stream;
    const uint32_t n = bvh->n_tri;
    // (the sort's scratch is done with; a single leaf's box is read back from here)
    ctx->scratch[2].reserve((size_t)n * 6 * sizeof(float));
    float *tbox = ctx->scratch[2].as<float>();
    k_leaves<true><<<div_up(n, 256), 256, 0, s>>>(mesh, bvh->order.as<uint32_t>(), tbox, bvh->tris.as<float4>());
    if(n < 2) return leaf_unions{tbox, nullptr, nullptr, nullptr, n, 0u};
    // per-leaf prefix and suffix unions, then the segments' sparse table
    const uint32_t nseg = div_up(n, BOX_SEG), levels = box_levels(nseg);
    device_buffer &w = ctx->scratch[3];
    w.reserve(((size_t)2 * n + (size_t)levels * nseg) * 6 * sizeof(float));
    float *pre = w.as<float>(), *suf = pre + 6 * (size_t)n, *table = suf + 6 * (size_t)n;
    k_box_scan<<<nseg, BOX_SEG, 0, s>>>(n, tbox, pre, suf, table);
    for(uint32_t k = 1; k < levels; k += SPARSE_LEVELS)
        k_box_sparse<<<div_up(nseg, 256), 256, 0, s>>>(nseg, k, levels, table);
    VKRT_HIP(hipGetLastError());
    return leaf_unions{tbox, pre, suf, table, n, nseg};
}

// ---------------------------------------------------------------------------------------------
// 4-wide collapse: top-down, one BVH4 node per work item. A work item starts from a BVH2 node's two
// children and repeatedly opens the internal child with the largest surface area until it has four
// children or only leaves; each internal child becomes a new work item. The boxes are the BVH2's (already
// padded), so traversal stays conservative. Every item also carries the traversal stack depth on entry
// (the sum of pushes, children - 1, over its ancestors); the maximum decides whether the collapse fits the
// fixed stack.
// ---------------------------------------------------------------------------------------------
struct collapse_child
{
    int32_t ref;
    float lo[3], hi[3];
};

__device__ __forceinline__ collapse_child child_of(const vkrt_bvh_node &nd, int k)
{
    collapse_child c;
    const float4 xy = k == 0 ? nd.a : nd.b;
    c.ref = k == 0 ? nd.d.x : nd.d.y;
    c.lo[0] = xy.x;
    c.hi[0] = xy.y;
    c.lo[1] = xy.z;
    c.hi[1] = xy.w;
    c.lo[2] = k == 0 ? nd.c.x : nd.c.z;
    c.hi[2] = k == 0 ? nd.c.y : nd.c.w;
    return c;
}

__device__ __forceinline__ float half_area(const collapse_child &c)
{
    const float dx = c.hi[0] - c.lo[0], dy = c.hi[1] - c.lo[1], dz = c.hi[2] - c.lo[2];
    return dx * dy + dy * dz + dz * dx;
}

__device__ __forceinline__ double child_area(const collapse_child &c)
{
    const double dx = fmax(0.0, (double)c.hi[0] - c.lo[0]), dy = fmax(0.0, (double)c.hi[1] - c.lo[1]),
                 dz = fmax(0.0, (double)c.hi[2] - c.lo[2]);
    return 2.0 * (dx * dy + dy * dz + dz * dx);
}

//! one level of the collapse. The work item of 4-wide node i is queue[i] = (BVH2 node, stack depth on entry, the
//! BVH2 node's depth): nodes are numbered level by level, so the queue's index is the node's. The level's
//! nodes and its children's are st->level[0 .. level + 1]; a workgroup takes its children's slots with one
//! atomic per 256 items (a child each took 63 us per level at 1.8M triangles on three words that every XCD
//! writes), which also lays a node's children side by side. The grid may be larger or smaller than the level.
//! A level opens every BVH2 node once, so the tree's depth, leaves and SAH terms are summed on the way (a pass of
//! its own, climbing the parents for the depth, took 608 us). Nodes deeper than the stack end the descent: the
//! build then fails. Nodes at or past n4_cap are counted and queued but not written (with n4_cap 0 a build wants the
//! sums only); n4_range[i] is the run of leaves below node i.
//! TOP: one workgroup takes the levels from the root on while they fit it (five in a full tree; a launch each took
//! 8 us); `level` otherwise counts from the first level it left.
constexpr uint32_t COLLAPSE_BLOCK = 256, COLLAPSE_GRID = 1024;
template<bool TOP>
__global__ void __launch_bounds__(COLLAPSE_BLOCK) k_collapse(const vkrt_bvh_node *__restrict__ n2,
                                                             const uint2 *__restrict__ range, int4 *__restrict__ queue,
                                                             uint32_t level, uint32_t n4_cap,
                                                             vkrt_bvh4_node *__restrict__ n4,
                                                             uint2 *__restrict__ n4_range, bvh_state *__restrict__ st)
{
    __shared__ uint32_t wave_sum[COLLAPSE_BLOCK / 64], slot_base;
    __shared__ double wave_sah[COLLAPSE_BLOCK / 64];
    __shared__ uint32_t wave_leaves[COLLAPSE_BLOCK / 64], wave_depth[COLLAPSE_BLOCK / 64],
            wave_stack[COLLAPSE_BLOCK / 64];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    double sah = 0.0;
    uint32_t leaves = 0, depth = 0, stack = 0;
    uint32_t first = 0, count = 1;// the level's first node and its nodes
    if constexpr(TOP)
    {
        level = 0;
        if(threadIdx.x == 0)
        {
            queue[0] = make_int4(0, 0, 1, 0);
            st->level[0] = 1u;
        }
        __syncthreads();
    }
    else
    {
        // (each lane reads a level's count: a loop over them waited for one after the other)
        level += st->top_levels;
        if(level >= MAX_LEVELS) return;
        uint32_t sum = lane < level ? st->level[lane] : 0u;
        if(lane + 64u < level) sum += st->level[lane + 64u];
        for(int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
        first = sum;
        count = st->level[level];
    }
    while(true)
    {
        const uint32_t next = first + count;
        for(uint32_t base = blockIdx.x * COLLAPSE_BLOCK; base < count; base += gridDim.x * COLLAPSE_BLOCK)
        {
            const bool active = base + threadIdx.x < count;
            const uint32_t me = first + base + threadIdx.x;
            collapse_child ch[4];
            uint32_t ch_depth[4] = {0, 0, 0, 0};// depth of the BVH2 node each child came from
            int cnt = 0;
            uint32_t inner = 0, depth_here = 0;
            int32_t node_here = 0;
            if(active)
            {
                const int4 item = queue[me];
                node_here = item.x;
                auto open = [&](int slot_a, int slot_b, int32_t node, uint32_t d) {
                    const vkrt_bvh_node nd = n2[node];
                    ch[slot_a] = child_of(nd, 0);
                    ch[slot_b] = child_of(nd, 1);
                    ch_depth[slot_a] = ch_depth[slot_b] = d;
                    depth = max(depth, d);
                    for(const int k: {slot_a, slot_b})
                    {
                        const double a = child_area(ch[k]);
                        if(ch[k].ref >= 0) sah += a;
                        else
                        {
                            sah += ((static_cast<uint32_t>(~ch[k].ref) & 7u) + 1) * a;
                            ++leaves;
                            depth = max(depth, d + 1);
                        }
                    }
                };
                open(0, 1, item.x, static_cast<uint32_t>(item.z));
                cnt = 2;
    #pragma unroll
                for(int step = 0; step < 2; ++step)
                {
                    int best = -1;
                    float best_a = -1.0f;
    #pragma unroll
                    for(int j = 0; j < 3; ++j)
                    {
                        if(j >= cnt || ch[j].ref < 0) continue;
                        const float a = half_area(ch[j]);
                        if(a > best_a)
                        {
                            best_a = a;
                            best = j;
                        }
                    }
                    if(best < 0) break;
                    // (constant slots: an array indexed by `best` would live in scratch memory)
                    if(best == 0) open(0, 2 + step, ch[0].ref, ch_depth[0] + 1);
                    else if(best == 1) open(1, 2 + step, ch[1].ref, ch_depth[1] + 1);
                    else open(2, 3, ch[2].ref, ch_depth[2] + 1);
                    ++cnt;
                }
                depth_here = static_cast<uint32_t>(item.y) + (cnt - 1);
                stack = max(stack, depth_here);
    #pragma unroll
                for(int j = 0; j < 4; ++j)
                    inner += j < cnt && ch[j].ref >= 0 && ch_depth[j] <= (uint32_t)STACK_SIZE ? 1u : 0u;
            }
            // the children's slots: an exclusive scan over the workgroup and one atomic
            uint32_t sum = inner;
            for(int off = 1; off < 64; off <<= 1)
            {
                const uint32_t y = __shfl_up(sum, off);
                if(lane >= (uint32_t)off) sum += y;
            }
            if(lane == 63) wave_sum[wave] = sum;
            __syncthreads();
            uint32_t before = 0, total = 0;
            for(uint32_t w = 0; w < COLLAPSE_BLOCK / 64; ++w)
            {
                before += w < wave ? wave_sum[w] : 0u;
                total += wave_sum[w];
            }
            if(threadIdx.x == 0) slot_base = next + (total ? atomicAdd(&st->level[level + 1], total) : 0u);
            __syncthreads();
            uint32_t slot = slot_base + before + sum - inner;
            if(active)
            {
                vkrt_bvh4_node out;
                float lo[3][4], hi[3][4];
                int32_t refs[4];
    #pragma unroll
                for(int j = 0; j < 4; ++j)
                {
                    for(int a = 0; a < 3; ++a)
                    {
                        lo[a][j] = j < cnt ? ch[j].lo[a] : 0.0f;
                        hi[a][j] = j < cnt ? ch[j].hi[a] : 0.0f;
                    }
                    refs[j] = EMPTY_CHILD;
                    if(j >= cnt) continue;
                    if(ch[j].ref < 0) refs[j] = ch[j].ref;
                    else if(ch_depth[j] <= (uint32_t)STACK_SIZE)
                    {
                        refs[j] = static_cast<int32_t>(slot);
                        queue[slot++] = make_int4(ch[j].ref, static_cast<int32_t>(depth_here),
                                                  static_cast<int32_t>(ch_depth[j] + 1), 0);
                    }
                }
                out.lox = make_float4(lo[0][0], lo[0][1], lo[0][2], lo[0][3]);
                out.hix = make_float4(hi[0][0], hi[0][1], hi[0][2], hi[0][3]);
                out.loy = make_float4(lo[1][0], lo[1][1], lo[1][2], lo[1][3]);
                out.hiy = make_float4(hi[1][0], hi[1][1], hi[1][2], hi[1][3]);
                out.loz = make_float4(lo[2][0], lo[2][1], lo[2][2], lo[2][3]);
                out.hiz = make_float4(hi[2][0], hi[2][1], hi[2][2], hi[2][3]);
                out.child = make_int4(refs[0], refs[1], refs[2], refs[3]);
                out.pad = make_int4(0, 0, 0, 0);
                if(me < n4_cap)
                {
                    n4[me] = out;
                    n4_range[me] = range[node_here];
                }
            }
        }
        if constexpr(!TOP) break;
        // the next level, when there is one and it fits (its nodes' queue entries are this workgroup's own stores)
        __syncthreads();
        ++level;
        first = next;
        count = __hip_atomic_load(&st->level[level], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if(count == 0 || count > COLLAPSE_BLOCK) break;
    }
    if(TOP && threadIdx.x == 0) st->top_levels = level;
    if(!TOP && blockIdx.x * COLLAPSE_BLOCK >= count) return;// (the whole workgroup: it had no item)
    for(int off = 32; off > 0; off >>= 1)
    {
        sah += __shfl_xor(sah, off);
        leaves += __shfl_xor(leaves, off);
        depth = max(depth, (uint32_t)__shfl_xor(depth, off));
        stack = max(stack, (uint32_t)__shfl_xor(stack, off));
    }
    if(lane == 0)
    {
        wave_sah[wave] = sah;
        wave_leaves[wave] = leaves;
        wave_depth[wave] = depth;
        wave_stack[wave] = stack;
    }
    __syncthreads();
    if(threadIdx.x == 0)
    {
        for(uint32_t w = 1; w < COLLAPSE_BLOCK / 64; ++w)
        {
            sah += wave_sah[w];
            leaves += wave_leaves[w];
            depth = max(depth, wave_depth[w]);
            stack = max(stack, wave_stack[w]);
        }
        atomicAdd(&st->sah, sah);
        if(leaves) atomicAdd(&st->leaves, leaves);
        atomicMax(&st->depth, depth);
        atomicMax(&st->stack, stack);
    }
}

//! refit of the 4-wide layout, a thread per child slot: a child's box is the union over its run of leaves, as when
//! the tree was built, so the collapse's shape, its worst-case stack depth and the choice of the 4-wide walk stay
//! what the build recorded
__global__ void __launch_bounds__(256) k_wide_refit(leaf_unions l, uint32_t n4_count, const uint2 *__restrict__ n4_range,
                                                    vkrt_bvh4_node *__restrict__ n4)
{
    const uint32_t i = (blockIdx.x * 256 + threadIdx.x) >> 2, j = threadIdx.x & 3u;
    if(i >= n4_count) return;
    const int32_t ref = reinterpret_cast<const int32_t *>(&n4[i].child)[j];
    if(ref == EMPTY_CHILD) return;
    uint2 r;
    if(ref >= 0) r = n4_range[ref];
    else
    {
        uint32_t count;
        const uint32_t v = static_cast<uint32_t>(~ref);
        r.x = v >> 3;
        count = (v & 7u) + 1u;
        r.y = r.x + count - 1u;
    }
    float b[6];
    run_box(l, r.x, r.y, b);
    float *f = reinterpret_cast<float *>(&n4[i]) + j;// lox hix loy hiy loz hiz, four floats each
    for(int a = 0; a < 3; ++a)
    {
        f[8 * a] = pad_lo(b[a]);
        f[8 * a + 4] = pad_hi(b[3 + a]);
    }
}

//! the root's box from its two child boxes: rb as (lo, hi) pairs per axis, bounds as lo xyz then hi xyz
static void root_bounds(const vkrt_bvh_node &root, float rb[6], float bounds[6])
{
    const float r[6] = {std::min(root.a.x, root.b.x), std::max(root.a.y, root.b.y), std::min(root.a.z, root.b.z),
                        std::max(root.a.w, root.b.w), std::min(root.c.x, root.c.z), std::max(root.c.y, root.c.w)};
    for(int a = 0; a < 6; ++a) rb[a] = r[a];
    for(int a = 0; a < 3; ++a)
    {
        bounds[a] = r[2 * a];
        bounds[3 + a] = r[2 * a + 1];
    }
}

//! a root's box from its used children
static void root_bounds(const vkrt_bvh4_node &root, float bounds[6])
{
    const float *planes[6] = {&root.lox.x, &root.loy.x, &root.loz.x, &root.hix.x, &root.hiy.x, &root.hiz.x};
    const int32_t child[4] = {root.child.x, root.child.y, root.child.z, root.child.w};
    bool first = true;
    for(int j = 0; j < 4; ++j)
    {
        if(child[j] == EMPTY_CHILD) continue;
        for(int a = 0; a < 6; ++a)
            bounds[a] = first ? planes[a][j] : (a < 3 ? std::min(bounds[a], planes[a][j]) : std::max(bounds[a], planes[a][j]));
        first = false;
    }
}

//! the BVH2 collapsed into the BVH4 used for traversal and the tree's statistics; false when the nodes did not fit
//! (n_nodes4 then says how many there are)
static bool collapse(vkrt_ctx *ctx, vkrt_bvh *bvh, const binary_tree &bin)
{
    hipStream_t s = ctx->stream;
    // (a 4-wide node takes in at least one node of the binary tree)
    const uint32_t most_nodes = bvh->n_nodes, cap = bvh->allow_wide ? bvh->node_cap : 0u;
    ctx->scratch[2].reserve((size_t)most_nodes * sizeof(int4));
    int4 *queue = ctx->scratch[2].as<int4>();
    bvh_state *st = ctx->state.as<bvh_state>();
    vkrt_bvh4_node *n4 = bvh->nodes4.as<vkrt_bvh4_node>();
    uint2 *n4_range = bvh->wide_range.as<uint2>();
    k_collapse<true><<<1, COLLAPSE_BLOCK, 0, s>>>(bin.nodes, bin.range, queue, 0u, cap, n4, n4_range, st);
    // the other levels are launched without asking how many there are: as many as balanced trees of this size have and
    // some more (a level that is not there costs its launch, 2 us), then in turns until the last one is empty
    uint32_t level = 0, todo = 2;
    for(size_t k = 1; k < most_nodes; k *= 4) ++todo;
    const bvh_state *got = nullptr;
    while(true)
    {
        for(uint32_t stop = level + todo; level < stop; ++level)
        {
            // (the first of them has a parent level of at most COLLAPSE_BLOCK nodes)
            const uint64_t most =
                    std::min<uint64_t>(most_nodes, level < 12 ? 4ull * COLLAPSE_BLOCK << (2 * level) : most_nodes);
            k_collapse<false><<<std::min(COLLAPSE_GRID, div_up(most, COLLAPSE_BLOCK)), COLLAPSE_BLOCK, 0, s>>>(
                    bin.nodes, bin.range, queue, level, cap, n4, n4_range, st);
        }
        got = &read_state(ctx, bin.nodes, nullptr);
        if(got->err) throw error(VKRT_E_INVALID_ARG, "triangle index out of range of the vertex count");
        if(got->depth > (uint32_t)STACK_SIZE) throw error(VKRT_E_INTERNAL, "BVH deeper than the traversal stack");
        if(got->top_levels + level >= MAX_LEVELS || got->level[got->top_levels + level] == 0) break;
        todo = 4;
    }
    uint64_t total = 0;
    for(uint32_t l = 0; l < MAX_LEVELS; ++l) total += got->level[l];
    VKRT_REQUIRE(total <= most_nodes, "BVH4 collapse overflow");
    vkrt_bvh_info &info = bvh->info;
    float rb[6];
    root_bounds(got->root, rb, info.bounds);
    const double dx = std::max(0.0, (double)rb[1] - rb[0]), dy = std::max(0.0, (double)rb[3] - rb[2]),
                 dz = std::max(0.0, (double)rb[5] - rb[4]);
    const double root_area = std::max(1e-30, 2.0 * (dx * dy + dy * dz + dz * dx));
    info.depth = std::max(1u, got->depth);
    info.sah_cost = static_cast<float>(1.0 + got->sah / root_area);// 1: the root's own visit
    info.n_leaves = got->leaves;
    if(!bvh->allow_wide) return true;
    bvh->n_nodes4 = static_cast<uint32_t>(total);
    bvh->stack4 = got->stack;
    bvh->root4 = 0;
    return total <= cap;
}

//! the end of a build: the leaves, the binary tree, and its collapse (kept off when its worst-case stack depth exceeds
//! STACK_SIZE)
static void build_tree(vkrt_ctx *ctx, vkrt_bvh *bvh, const mesh_view &mesh, const binary_tree &bin)
{
    hipStream_t s = ctx->stream;
    const uint32_t n = bvh->n_tri;
    const leaf_unions leaves = leaf_pass(ctx, bvh, mesh);
    bvh->n_nodes = n - 1u;
    bvh->root_ref = n <= bvh->max_leaf ? ~static_cast<int>(n - 1u) : 0;
    if(n >= 2)
        k_layout<<<div_up(n - 1u, 256), 256, 0, s>>>(leaves, bin.child, bin.range, bvh->max_leaf, bin.nodes);
    VKRT_HIP(hipGetLastError());
    if(bvh->root_ref < 0)
    {
        if(read_state(ctx, nullptr, nullptr).err)
            throw error(VKRT_E_INVALID_ARG, "triangle index out of range of the vertex count");
        bvh->root4 = bvh->root_ref;// a single leaf
        bvh->wide = bvh->allow_wide;
        single_leaf_info(bvh, ctx->scratch[2].as<float>(), s);
        return;
    }
    if(!collapse(ctx, bvh, bin))
    {
        // more nodes than there was room for: the same again in a larger allocation
        device_buffer old = std::move(bvh->memory);
        const vkrt_bvh::part indices = bvh->indices, order = bvh->order;
        allocate(bvh, bvh->n_nodes4);
        VKRT_HIP(hipMemcpyAsync(bvh->indices.ptr, indices.ptr, indices.bytes, hipMemcpyDeviceToDevice, s));
        VKRT_HIP(hipMemcpyAsync(bvh->order.ptr, order.ptr, order.bytes, hipMemcpyDeviceToDevice, s));
        mesh_view moved = mesh;
        moved.idx = bvh->indices.as<uint32_t>();
        k_leaves<false><<<div_up(n, 256), 256, 0, s>>>(moved, bvh->order.as<uint32_t>(), nullptr, bvh->tris.as<float4>());
        k_state_clear<<<1, 256, 0, s>>>(ctx->state.as<bvh_state>());
        VKRT_REQUIRE(collapse(ctx, bvh, bin), "BVH4 collapse overflow");
    }
    // the 4-wide walk addresses nodes with 32-bit byte offsets (node4_intervals)
    bvh->wide = bvh->allow_wide && bvh->stack4 <= (uint32_t)STACK_SIZE &&
                (uint64_t)bvh->n_nodes4 * sizeof(vkrt_bvh4_node) <= 0xffffffffull;
    if(bvh->wide) return;
    // the binary tree stays where traversal uses it
    const size_t ni = n - 1u;
    place(bvh->binary, {{&bvh->nodes, ni * sizeof(vkrt_bvh_node)}, {&bvh->child, ni * sizeof(int2)},
                        {&bvh->range, ni * sizeof(uint2)}});
    VKRT_HIP(hipMemcpyAsync(bvh->nodes.ptr, bin.nodes, bvh->nodes.bytes, hipMemcpyDeviceToDevice, s));
    VKRT_HIP(hipMemcpyAsync(bvh->child.ptr, bin.child, bvh->child.bytes, hipMemcpyDeviceToDevice, s));
    VKRT_HIP(hipMemcpyAsync(bvh->range.ptr, bin.range, bvh->range.bytes, hipMemcpyDeviceToDevice, s));
}

//! the rest of the info block after a build or a refit
static void refresh_info(vkrt_bvh *bvh)
{
    bvh->info.n_tri = bvh->n_tri;
    bvh->info.n_nodes = bvh->n_nodes;
    bvh->info.device_bytes = bvh->memory.bytes + bvh->binary.bytes;
    bvh->info.n_wide_nodes = bvh->wide ? bvh->n_nodes4 : 0;
    bvh->info.wide_stack = bvh->stack4;
}

}// namespace vkrt

using namespace vkrt;

extern "C" {

int vkrt_bvh_build(vkrt_ctx *ctx, const float *positions, uint32_t n_vert, uint32_t stride_bytes,
                   const uint32_t *indices, uint32_t n_tri, const vkrt_bvh_params *params, int flags, vkrt_bvh **out)
{
    return guarded(ctx, [&] {
        VKRT_REQUIRE(out, "null output handle");
        *out = nullptr;
        VKRT_REQUIRE(stride_bytes >= 12 && stride_bytes % 4 == 0, "stride must be >= 12 and a multiple of 4");
        VKRT_REQUIRE(n_tri == 0 || (positions && indices && n_vert), "null mesh arrays");
        VKRT_REQUIRE(n_tri < (1u << 28), "at most 2^28 - 1 triangles per BVH");
        uint32_t leaf = params && params->max_leaf_size ? params->max_leaf_size : 2;
        VKRT_REQUIRE(leaf >= 1 && leaf <= (uint32_t)MAX_LEAF, "max_leaf_size must be in 1..8");
        VKRT_REQUIRE(!params || params->builder == VKRT_BUILDER_LBVH || params->builder == VKRT_BUILDER_PLOC,
                     "builder must be VKRT_BUILDER_LBVH or VKRT_BUILDER_PLOC");
        VKRT_REQUIRE(!params || params->width == 0 || params->width == 2 || params->width == 4,
                     "width must be 0 (auto), 2 or 4");
        auto t_start = std::chrono::steady_clock::now();
        auto bvh = std::make_unique<vkrt_bvh>();
        bvh->device = ctx->device;
        bvh->n_tri = n_tri;
        bvh->n_vert = n_vert;
        bvh->max_leaf = leaf;
        bvh->empty = n_tri == 0;
        bvh->allow_wide = !params || params->width != 2;
        bvh->builder = params ? params->builder : VKRT_BUILDER_LBVH;
        VKRT_REQUIRE(!params || params->ploc_radius <= (uint32_t)PLOC_MAX_RADIUS, "ploc_radius must be in 0..32");
        bvh->ploc_radius = params ? params->ploc_radius : 0u;
        if(n_tri)
        {
            ctx->state.reserve(sizeof(bvh_state));
            const size_t pos_bytes = (size_t)(n_vert - 1) * stride_bytes + 12;
            const uint8_t *dpos =
                    input(ctx, 0, reinterpret_cast<const uint8_t *>(positions), pos_bytes, flags);
            const uint32_t *didx = input(ctx, 1, indices, (size_t)n_tri * 3, flags);
            // the binary tree is scratch: most builds keep only its collapse
            const size_t ni = n_tri - 1u, node_bytes = (ni * sizeof(vkrt_bvh_node) + 255) & ~size_t(255),
                         child_bytes = (ni * sizeof(int2) + 255) & ~size_t(255);
            ctx->scratch[4].reserve(node_bytes + child_bytes + ni * sizeof(uint2));
            uint8_t *tree = ctx->scratch[4].as<uint8_t>();
            const binary_tree bin{reinterpret_cast<vkrt_bvh_node *>(tree), reinterpret_cast<int2 *>(tree + node_bytes),
                                  reinterpret_cast<uint2 *>(tree + node_bytes + child_bytes)};
            allocate(bvh.get(), bvh->allow_wide ? node_guess(bvh.get()) : 0u);
            VKRT_HIP(hipMemcpyAsync(bvh->indices.ptr, didx, (size_t)n_tri * 3 * sizeof(uint32_t),
                                    hipMemcpyDeviceToDevice, ctx->stream));
            const mesh_view mesh{dpos, bvh->indices.as<uint32_t>(), stride_bytes, n_tri, n_vert};
            build_topology(ctx, bvh.get(), mesh, bin);
            build_tree(ctx, bvh.get(), mesh, bin);
            VKRT_HIP(hipStreamSynchronize(ctx->stream));
        }
        else single_leaf_info(bvh.get(), nullptr, ctx->stream);
        bvh->info.build_ms = std::chrono::duration<float, std::milli>(std::chrono::steady_clock::now() - t_start).count();
        refresh_info(bvh.get());
        *out = bvh.release();
    });
}

int vkrt_bvh_refit(vkrt_ctx *ctx, vkrt_bvh *bvh, const float *positions, uint32_t stride_bytes, int flags)
{
    return guarded(ctx, [&] {
        VKRT_REQUIRE(bvh, "null bvh");
        VKRT_REQUIRE(stride_bytes >= 12 && stride_bytes % 4 == 0, "stride must be >= 12 and a multiple of 4");
        if(bvh->empty) return;
        VKRT_REQUIRE(positions, "null positions");
        ctx->state.reserve(sizeof(bvh_state));
        hipStream_t s = ctx->stream;
        const size_t pos_bytes = (size_t)(bvh->n_vert - 1) * stride_bytes + 12;
        const uint8_t *dpos = input(ctx, 0, reinterpret_cast<const uint8_t *>(positions), pos_bytes, flags);
        const leaf_unions leaves = leaf_pass(
                ctx, bvh, mesh_view{dpos, bvh->indices.as<uint32_t>(), stride_bytes, bvh->n_tri, bvh->n_vert});
        if(bvh->root_ref < 0) single_leaf_info(bvh, ctx->scratch[2].as<float>(), s);
        else
        {
            // the topology stays, and with it depth, leaves and SAH cost: only the boxes and bounds change
            vkrt_bvh4_node *n4 = bvh->wide ? bvh->nodes4.as<vkrt_bvh4_node>() : nullptr;
            vkrt_bvh_node *n2 = bvh->nodes.as<vkrt_bvh_node>();
            if(n4)
                k_wide_refit<<<div_up((uint64_t)bvh->n_nodes4 * 4, 256), 256, 0, s>>>(leaves, bvh->n_nodes4,
                                                                                     bvh->wide_range.as<uint2>(), n4);
            if(n2)
                k_layout<<<div_up(bvh->n_nodes, 256), 256, 0, s>>>(leaves, bvh->child.as<int2>(), bvh->range.as<uint2>(),
                                                                   bvh->max_leaf, n2);
            const bvh_state &got = read_state(ctx, n2, n4);
            float rb[6];
            if(n4) root_bounds(got.root4, bvh->info.bounds);
            else root_bounds(got.root, rb, bvh->info.bounds);
        }
        refresh_info(bvh);
    });
}

int vkrt_bvh_validate(vkrt_ctx *ctx, const vkrt_bvh *bvh, const float *positions, uint32_t stride_bytes, int flags,
                      vkrt_bvh_check *out)
{
    return guarded(ctx, [&] {
        VKRT_REQUIRE(bvh && out, "null bvh or output");
        VKRT_REQUIRE(stride_bytes >= 12 && stride_bytes % 4 == 0, "stride must be >= 12 and a multiple of 4");
        VKRT_REQUIRE(bvh->empty || positions, "null positions");
        *out = vkrt_bvh_check{};
        out->wide = bvh->wide ? 1u : 0u;
        if(bvh->empty)
        {
            out->ok = 1;
            out->stack_ok = 1;
            return;
        }
        hipStream_t s = ctx->stream;
        const uint32_t n = bvh->n_tri;
        auto fetch = [&](const void *src, size_t bytes, bool device, std::vector<uint8_t> &dst) {
            dst.resize(bytes);
            if(!bytes) return;
            VKRT_HIP(hipMemcpyAsync(dst.data(), src, bytes, device ? hipMemcpyDeviceToHost : hipMemcpyHostToHost, s));
        };
        std::vector<uint8_t> h_nodes, h_nodes4, h_tris, h_idx, h_pos;
        if(bvh->wide) fetch(bvh->nodes4.ptr, (size_t)bvh->n_nodes4 * sizeof(vkrt_bvh4_node), true, h_nodes4);
        else if(bvh->root_ref >= 0) fetch(bvh->nodes.ptr, (size_t)bvh->n_nodes * sizeof(vkrt_bvh_node), true, h_nodes);
        fetch(bvh->tris.ptr, (size_t)n * TRI_BYTES, true, h_tris);
        fetch(bvh->indices.ptr, (size_t)n * 3 * sizeof(uint32_t), true, h_idx);
        fetch(positions, (size_t)(bvh->n_vert - 1) * stride_bytes + 12, (flags & VKRT_DEVICE_PTRS) != 0, h_pos);
        VKRT_HIP(hipStreamSynchronize(s));
        const auto *nodes = reinterpret_cast<const vkrt_bvh_node *>(h_nodes.data());
        const auto *nodes4 = reinterpret_cast<const vkrt_bvh4_node *>(h_nodes4.data());
        const auto *tris = reinterpret_cast<const float4 *>(h_tris.data());
        const auto *idx = reinterpret_cast<const uint32_t *>(h_idx.data());
        std::vector<uint32_t> seen(n, 0);
        auto vertex = [&](uint32_t v, int a) {
            float x;
            std::memcpy(&x, h_pos.data() + (size_t)v * stride_bytes + 4 * a, 4);
            return x;
        };
        auto violation = [&](uint32_t kind, uint32_t node, uint32_t slot, uint32_t tri, const float *box,
                             const float *outer, int n_outer) {
            if(out->box_violations++ != 0) return;
            out->bad_kind = kind;
            out->bad_node = node;
            out->bad_slot = slot;
            out->bad_tri = tri;
            std::memcpy(out->bad_box, box, sizeof out->bad_box);
            for(int a = 0; a < n_outer; ++a) out->bad_outer[a] = outer[a];
        };
        // a leaf's triangles: counted, and their vertices inside the box the parent stores for the leaf
        auto leaf = [&](int32_t ref, const float *box, uint32_t node, uint32_t slot) {
            const uint32_t v = static_cast<uint32_t>(~ref), first = v >> 3, count = (v & 7u) + 1;
            if((uint64_t)first + count > n)
            {
                ++out->bad_refs;
                return;
            }
            for(uint32_t k = first; k < first + count; ++k)
            {
                ++out->tris_reached;
                uint32_t orig;
                std::memcpy(&orig, &tris[(TRI_BYTES / 16) * (size_t)k + 2].y, 4);
                if(orig >= n)
                {
                    ++out->bad_refs;
                    continue;
                }
                ++seen[orig];
                if(!box) continue;
                bool finite = true, inside = true;
                float outside[3] = {0.f, 0.f, 0.f};
                for(int c = 0; c < 3; ++c)
                {
                    const uint32_t vi = idx[3 * (size_t)orig + c];
                    if(vi >= bvh->n_vert)
                    {
                        finite = false;
                        break;
                    }
                    bool in = true;
                    for(int a = 0; a < 3; ++a)
                    {
                        const float x = vertex(vi, a);
                        finite = finite && std::isfinite(x);
                        in = in && x >= box[a] && x <= box[3 + a];
                    }
                    if(!in && inside)
                        for(int a = 0; a < 3; ++a) outside[a] = vertex(vi, a);
                    inside = inside && in;
                }
                // non-finite triangles get empty boxes
                if(finite && !inside) violation(2, node, slot, orig, box, outside, 3);
            }
        };
        auto inside = [](const float *in, const float *outer) {
            for(int a = 0; a < 3; ++a)
                if(!(in[a] >= outer[a] && in[3 + a] <= outer[3 + a])) return false;
            return true;
        };
        uint32_t recorded = 0;
        if(bvh->root_ref < 0)
        {
            leaf(bvh->root_ref, nullptr, 0, 0);// a single leaf: no box is stored for it
            out->stack_bound = 0;
        }
        else if(bvh->wide)
        {
            recorded = bvh->stack4;
            struct item
            {
                int32_t node;
                uint32_t depth;
                float box[6];
                bool has_box;
            };
            std::vector<item> todo{{0, 0u, {}, false}};
            while(!todo.empty())
            {
                const item it = todo.back();
                todo.pop_back();
                if(it.node < 0 || (uint32_t)it.node >= bvh->n_nodes4)
                {
                    ++out->bad_refs;
                    continue;
                }
                const vkrt_bvh4_node &nd = nodes4[it.node];
                const int32_t ch[4] = {nd.child.x, nd.child.y, nd.child.z, nd.child.w};
                const float *lx = &nd.lox.x, *hx = &nd.hix.x, *ly = &nd.loy.x, *hy = &nd.hiy.x, *lz = &nd.loz.x,
                            *hz = &nd.hiz.x;
                uint32_t used = 0;
                for(int j = 0; j < 4; ++j) used += ch[j] != EMPTY_CHILD ? 1u : 0u;
                const uint32_t depth_here = it.depth + (used ? used - 1 : 0);
                out->stack_bound = std::max(out->stack_bound, depth_here);
                for(int j = 0; j < 4; ++j)
                {
                    if(ch[j] == EMPTY_CHILD) continue;
                    const float b[6] = {lx[j], ly[j], lz[j], hx[j], hy[j], hz[j]};
                    if(it.has_box && !inside(b, it.box)) violation(1, it.node, j, 0, b, it.box, 6);
                    if(ch[j] < 0) leaf(ch[j], b, it.node, j);
                    else
                    {
                        item c{ch[j], depth_here, {}, true};
                        std::memcpy(c.box, b, sizeof b);
                        todo.push_back(c);
                    }
                }
            }
        }
        else
        {
            // binary tree: the stack holds at most one entry per ancestor of the deepest node
            recorded = bvh->info.depth;
            struct item
            {
                int32_t node;
                uint32_t depth;
                float box[6];
                bool has_box;
            };
            std::vector<item> todo{{0, 1u, {}, false}};
            while(!todo.empty())
            {
                const item it = todo.back();
                todo.pop_back();
                if(it.node < 0 || (uint32_t)it.node >= bvh->n_nodes)
                {
                    ++out->bad_refs;
                    continue;
                }
                const vkrt_bvh_node &nd = nodes[it.node];
                out->stack_bound = std::max(out->stack_bound, it.depth + 1);
                const float b[2][6] = {{nd.a.x, nd.a.z, nd.c.x, nd.a.y, nd.a.w, nd.c.y},
                                       {nd.b.x, nd.b.z, nd.c.z, nd.b.y, nd.b.w, nd.c.w}};
                const int32_t ch[2] = {nd.d.x, nd.d.y};
                for(int j = 0; j < 2; ++j)
                {
                    if(it.has_box && !inside(b[j], it.box)) violation(1, it.node, j, 0, b[j], it.box, 6);
                    if(ch[j] < 0) leaf(ch[j], b[j], it.node, j);
                    else
                    {
                        item c{ch[j], it.depth + 1, {}, true};
                        std::memcpy(c.box, b[j], sizeof b[j]);
                        todo.push_back(c);
                    }
                }
            }
        }
        for(uint32_t k = 0; k < n; ++k) out->tris_not_once += seen[k] != 1 ? 1u : 0u;
        out->stack_ok = (bvh->root_ref < 0 || out->stack_bound == recorded) && out->stack_bound <= (uint32_t)STACK_SIZE;
        out->ok = out->tris_not_once == 0 && out->box_violations == 0 && out->bad_refs == 0 && out->stack_ok &&
                  out->tris_reached == n;
    });
}

int vkrt_bvh_get_info(const vkrt_bvh *bvh, vkrt_bvh_info *out)
{
    if(!bvh || !out) return VKRT_E_INVALID_ARG;
    *out = bvh->info;
    return VKRT_OK;
}

void vkrt_bvh_destroy(vkrt_bvh *bvh)
{
    if(!bvh) return;
    (void)hipSetDevice(bvh->device);
    delete bvh;
}

}// extern "C"
