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
//   k_leaves    triangles in leaf order, straight from the mesh: exact AABBs and 48-B records (v0, e1, e2,
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
#include <memory>
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
    if(!(finite3(v0) && finite3(v1) && finite3(v2)))
    {
        b[0] = b[1] = b[2] = FLT_MAX;
        b[3] = b[4] = b[5] = -FLT_MAX;
        return false;
    }
    b[0] = fminf(fminf(v0.x, v1.x), v2.x), b[1] = fminf(fminf(v0.y, v1.y), v2.y), b[2] = fminf(fminf(v0.z, v1.z), v2.z);
    b[3] = fmaxf(fmaxf(v0.x, v1.x), v2.x), b[4] = fmaxf(fmaxf(v0.y, v1.y), v2.y), b[5] = fmaxf(fmaxf(v0.z, v1.z), v2.z);
    return true;
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

//! the triangles in leaf order, straight from the mesh: their boxes, and with RECORDS the 48-B leaf records
//! (v0, e1, e2, original index; the last two words are cleared)
template<bool RECORDS>
__global__ void __launch_bounds__(256) k_leaves(mesh_view m, const uint32_t *__restrict__ order,
                                                float *__restrict__ tbox, float4 *__restrict__ tris)
{
    const uint32_t j = blockIdx.x * 256 + threadIdx.x;
    if(j >= m.n_tri) return;
    const uint32_t src = order[j];
    vec3 v0, v1, v2;
    bool ok;
    float b[6];
    load_triangle(m, src, v0, v1, v2, ok);
    triangle_box(v0, v1, v2, b);
    store_box(tbox + 6 * (size_t)j, b);
    if constexpr(RECORDS)
    {
        const vec3 e1 = v1 - v0, e2 = v2 - v0;
        tris[3 * (size_t)j + 0] = make_float4(v0.x, v0.y, v0.z, e1.x);
        tris[3 * (size_t)j + 1] = make_float4(e1.y, e1.z, e2.x, e2.y);
        tris[3 * (size_t)j + 2] = make_float4(e2.z, __uint_as_float(src), 0.f, 0.f);
    }
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

//! sparse-table level k from level k - 1: entry i = union of entries i and i + 2^(k-1), for i + 2^k <= nseg
__global__ void k_box_sparse(uint32_t nseg, uint32_t k, float *__restrict__ table)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t half = 1u << (k - 1);
    if((size_t)i + 2 * half > nseg) return;
    const float *lo = table + 6 * ((size_t)(k - 1) * nseg + i);
    const float *hi = table + 6 * ((size_t)(k - 1) * nseg + i + half);
    float a[6], b[6];
    load_box(lo, a);
    load_box(hi, b);
    box_union(a, b);
    store_box(table + 6 * ((size_t)k * nseg + i), a);
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
    vkrt_bvh_node root;
};

__global__ void __launch_bounds__(256) k_state_clear(bvh_state *__restrict__ st)
{
    uint32_t *w = reinterpret_cast<uint32_t *>(st);
    for(uint32_t i = threadIdx.x; i < sizeof(bvh_state) / 4; i += 256) w[i] = 0u;
}

__global__ void __launch_bounds__(256) k_report(const bvh_state *__restrict__ st, const vkrt_bvh_node *__restrict__ nodes,
                                                bvh_state *__restrict__ host)
{
    const uint32_t *src = reinterpret_cast<const uint32_t *>(st);
    uint32_t *dst = reinterpret_cast<uint32_t *>(host);
    for(uint32_t i = threadIdx.x; i < offsetof(bvh_state, root) / 4; i += 256) dst[i] = src[i];
    if(nodes && threadIdx.x < sizeof(vkrt_bvh_node) / 4)
        dst[offsetof(bvh_state, root) / 4 + threadIdx.x] = reinterpret_cast<const uint32_t *>(nodes)[threadIdx.x];
}

//! the state as the host reads it, once everything queued before has run; with nodes, the root node too
static const bvh_state &read_state(vkrt_ctx *ctx, const vkrt_bvh_node *nodes)
{
    bvh_state *host = ctx->pinned_as<bvh_state>();
    k_report<<<1, 256, 0, ctx->stream>>>(ctx->state.as<bvh_state>(), nodes, host);
    VKRT_HIP(hipGetLastError());
    VKRT_HIP(hipStreamSynchronize(ctx->stream));
    return *host;
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

//! a single leaf's bounds (at most 8 triangles): the union of its triangles' boxes (tbox, in leaf order), padded
//! like every node box
static void single_leaf_info(vkrt_bvh *bvh, hipStream_t s)
{
    vkrt_bvh_info &info = bvh->info;
    info.depth = 1;
    info.sah_cost = 0.f;
    info.n_leaves = bvh->empty ? 0 : 1;
    if(bvh->empty) return;
    const uint32_t v = static_cast<uint32_t>(~bvh->root_ref), first = v >> 3, count = (v & 7u) + 1;
    std::vector<float> box(6 * (size_t)count);
    VKRT_HIP(hipMemcpyAsync(box.data(), bvh->tbox.as<float>() + 6 * (size_t)first, box.size() * 4,
                            hipMemcpyDeviceToHost, s));
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

static void build_topology_ploc(vkrt_ctx *ctx, vkrt_bvh *bvh);

static void build_topology(vkrt_ctx *ctx, vkrt_bvh *bvh, const mesh_view &mesh)
{
    hipStream_t s = ctx->stream;
    const uint32_t n = bvh->n_tri;
    bvh->tbox.reserve((size_t)n * 6 * sizeof(float));
    // scratch: centroid bounds, sort keys, sort temp
    device_buffer &tmp = ctx->scratch[2];
    const size_t key_bytes = (size_t)n * sizeof(uint32_t), partial_bytes = BOUNDS_PARTIALS * 6 * sizeof(float);
    tmp.reserve(partial_bytes + key_bytes + radix_sort_temp_bytes(n));
    float *partial = tmp.as<float>();
    uint32_t *keys = reinterpret_cast<uint32_t *>(tmp.as<uint8_t>() + partial_bytes);
    void *sort_tmp = tmp.as<uint8_t>() + partial_bytes + key_bytes;
    bvh->order.reserve(key_bytes);
    uint32_t *order = bvh->order.as<uint32_t>();

    bvh_state *st = ctx->state.as<bvh_state>();
    k_state_clear<<<1, 256, 0, s>>>(st);
    const uint32_t n_partial = std::min(BOUNDS_PARTIALS, div_up(n, BOUNDS_BLOCK));
    k_bounds<<<n_partial, BOUNDS_BLOCK, 0, s>>>(mesh, partial, &st->err);
    k_morton<<<div_up(n, 256), 256, 0, s>>>(mesh, partial, n_partial, keys, order);
    radix_sort_pairs(s, keys, order, n, 30, sort_tmp);
    if(n >= 2)
    {
        const uint32_t ni = n - 1;
        bvh->child.reserve(ni * sizeof(int2));
        bvh->range.reserve(ni * sizeof(uint2));
        if(bvh->builder == VKRT_BUILDER_PLOC)
        {
            k_leaves<false><<<div_up(n, 256), 256, 0, s>>>(mesh, order, bvh->tbox.as<float>(), nullptr);
            build_topology_ploc(ctx, bvh);
        }
        else
            k_karras<<<div_up(ni, 256), 256, 0, s>>>(keys, (int)n, bvh->child.as<int2>(), bvh->range.as<uint2>());
    }
    VKRT_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------
// PLOC (Meister & Bittner 2018): agglomerative clustering over the Morton-sorted leaves. Each round every
// cluster finds, within PLOC_RADIUS positions of the sorted list, the cluster whose merged box has the
// smallest surface area; mutual nearest neighbours merge into a new node at the lower position, and the list
// is compacted. Pairs are ordered by (area, lower position, higher position), so the globally smallest pair
// is always mutual and every round merges. Internal nodes are numbered in merge order, then renumbered so the
// root is node 0 and parents precede children; leaves are finally put in depth-first order so that every
// subtree covers a contiguous range, which the leaf collapse of k_layout and the refit rely on.
// ---------------------------------------------------------------------------------------------
constexpr int PLOC_RADIUS = 16;    // default search radius
constexpr int PLOC_MAX_RADIUS = 32;
constexpr int PLOC_BLOCK = 256;
constexpr uint32_t PLOC_MAX_DEPTH = 4096;// bound of the upward walks; deeper trees are rejected after layout

__device__ __forceinline__ float merged_half_area(const float4 &alo, const float4 &ahi, const float4 &blo,
                                                  const float4 &bhi)
{
    const float dx = fmaxf(ahi.x, bhi.x) - fminf(alo.x, blo.x);
    const float dy = fmaxf(ahi.y, bhi.y) - fminf(alo.y, blo.y);
    const float dz = fmaxf(ahi.z, bhi.z) - fminf(alo.z, blo.z);
    return dx * dy + dy * dz + dz * dx;
}

__global__ void k_ploc_init(const float *__restrict__ tbox, uint32_t n, int32_t *__restrict__ cl_id,
                            float4 *__restrict__ lo, float4 *__restrict__ hi, int32_t *__restrict__ parent_int,
                            uint32_t ni)
{
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if(j < ni) parent_int[j] = -1;
    if(j >= n) return;
    const float *b = tbox + 6 * (size_t)j;
    cl_id[j] = ~static_cast<int32_t>(j);
    lo[j] = make_float4(b[0], b[1], b[2], 0.f);
    hi[j] = make_float4(b[3], b[4], b[5], 0.f);
}

//! nearest neighbour of every cluster within the window; ties go to the smallest position, which is the
//! smallest pair in (area, lower, higher) order
__global__ void __launch_bounds__(PLOC_BLOCK) k_ploc_nn(const float4 *__restrict__ lo, const float4 *__restrict__ hi,
                                                        uint32_t nc, int radius, int32_t *__restrict__ nn)
{
    __shared__ float4 slo[PLOC_BLOCK + 2 * PLOC_MAX_RADIUS], shi[PLOC_BLOCK + 2 * PLOC_MAX_RADIUS];
    const int base = static_cast<int>(blockIdx.x * PLOC_BLOCK) - radius;
    for(int k = threadIdx.x; k < PLOC_BLOCK + 2 * radius; k += PLOC_BLOCK)
    {
        const int g = base + k;
        if(g >= 0 && g < static_cast<int>(nc))
        {
            slo[k] = lo[g];
            shi[k] = hi[g];
        }
    }
    __syncthreads();
    const int i = static_cast<int>(blockIdx.x * PLOC_BLOCK + threadIdx.x);
    if(i >= static_cast<int>(nc)) return;
    const int li = threadIdx.x + radius;
    float best = 0.f;
    int bj = -1;
    for(int o = -radius; o <= radius; ++o)
    {
        const int j = i + o;
        if(o == 0 || j < 0 || j >= static_cast<int>(nc)) continue;
        const float d = merged_half_area(slo[li], shi[li], slo[li + o], shi[li + o]);
        if(bj < 0 || d < best)
        {
            best = d;
            bj = j;
        }
    }
    nn[i] = bj;
}

__global__ void k_ploc_flags(const int32_t *__restrict__ nn, uint32_t nc, uint32_t *__restrict__ merge,
                             uint32_t *__restrict__ keep)
{
    const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if(i >= static_cast<int>(nc)) return;
    const int j = nn[i];
    const bool mutual = nn[j] == i;
    merge[i] = (mutual && i < j) ? 1u : 0u;
    keep[i] = (mutual && i > j) ? 0u : 1u;
}

__device__ __forceinline__ uint32_t leaf_count(const uint32_t *__restrict__ cnt, int32_t ref)
{
    return ref < 0 ? 1u : cnt[ref];
}

__global__ void k_ploc_merge(const int32_t *__restrict__ nn, uint32_t nc, const uint32_t *__restrict__ merge,
                             const uint32_t *__restrict__ moff, const uint32_t *__restrict__ keep,
                             const uint32_t *__restrict__ koff, uint32_t base, const int32_t *__restrict__ cl_id,
                             const float4 *__restrict__ lo, const float4 *__restrict__ hi,
                             int32_t *__restrict__ out_id, float4 *__restrict__ out_lo, float4 *__restrict__ out_hi,
                             int2 *__restrict__ child, uint32_t *__restrict__ cnt, int32_t *__restrict__ parent_int,
                             int32_t *__restrict__ parent_leaf)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= nc || !keep[i]) return;
    const uint32_t pos = koff[i];
    if(!merge[i])
    {
        out_id[pos] = cl_id[i];
        out_lo[pos] = lo[i];
        out_hi[pos] = hi[i];
        return;
    }
    const uint32_t j = static_cast<uint32_t>(nn[i]);
    const int32_t id = static_cast<int32_t>(base + moff[i]);
    const int32_t a = cl_id[i], b = cl_id[j];
    child[id] = make_int2(a, b);
    cnt[id] = leaf_count(cnt, a) + leaf_count(cnt, b);
    if(a < 0) parent_leaf[~a] = id;
    else parent_int[a] = id;
    if(b < 0) parent_leaf[~b] = id;
    else parent_int[b] = id;
    const float4 la = lo[i], lb = lo[j], ha = hi[i], hb = hi[j];
    out_id[pos] = id;
    out_lo[pos] = make_float4(fminf(la.x, lb.x), fminf(la.y, lb.y), fminf(la.z, lb.z), 0.f);
    out_hi[pos] = make_float4(fmaxf(ha.x, hb.x), fmaxf(ha.y, hb.y), fmaxf(ha.z, hb.z), 0.f);
}

//! internal node k becomes ni - 1 - k: the last merge (the root) is node 0 and parents precede children
__global__ void k_ploc_renumber(uint32_t ni, uint32_t n, const int2 *__restrict__ child, const uint32_t *__restrict__ cnt,
                                const int32_t *__restrict__ parent_int, const int32_t *__restrict__ parent_leaf,
                                int2 *__restrict__ child2, uint32_t *__restrict__ cnt2, int32_t *__restrict__ parent_int2,
                                int32_t *__restrict__ parent_leaf2)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    auto map = [ni](int32_t r) { return r < 0 ? r : static_cast<int32_t>(ni - 1u) - r; };
    if(k < ni)
    {
        const uint32_t nk = ni - 1u - k;
        const int2 c = child[k];
        child2[nk] = make_int2(map(c.x), map(c.y));
        cnt2[nk] = cnt[k];
        parent_int2[nk] = parent_int[k] < 0 ? -1 : map(parent_int[k]);
    }
    if(k < n) parent_leaf2[k] = map(parent_leaf[k]);
}

//! depth-first position of every leaf and the first position of every internal node's range: the leaf
//! counts of all left siblings on the way up
__global__ void k_ploc_dfs(uint32_t ni, uint32_t n, const int2 *__restrict__ child, const uint32_t *__restrict__ cnt,
                           const int32_t *__restrict__ parent_int, const int32_t *__restrict__ parent_leaf,
                           uint32_t *__restrict__ leaf_pos, uint2 *__restrict__ range)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if(k < n)
    {
        uint32_t off = 0;
        int32_t cur = ~static_cast<int32_t>(k), node = parent_leaf[k];
        for(uint32_t step = 0; node >= 0 && step < PLOC_MAX_DEPTH; ++step)
        {
            const int2 c = child[node];
            if(c.y == cur) off += leaf_count(cnt, c.x);
            cur = node;
            node = parent_int[node];
        }
        leaf_pos[k] = off;
    }
    if(k < ni)
    {
        uint32_t off = 0;
        int32_t cur = static_cast<int32_t>(k), node = parent_int[k];
        for(uint32_t step = 0; node >= 0 && step < PLOC_MAX_DEPTH; ++step)
        {
            const int2 c = child[node];
            if(c.y == cur) off += leaf_count(cnt, c.x);
            cur = node;
            node = parent_int[node];
        }
        range[k] = make_uint2(off, off + cnt[k] - 1u);
    }
}

//! leaves to depth-first order: the triangle order and leaf child refs
__global__ void k_ploc_permute(uint32_t ni, uint32_t n, const uint32_t *__restrict__ leaf_pos,
                               const uint32_t *__restrict__ order_in, uint32_t *__restrict__ order_out,
                               const int2 *__restrict__ child_in, int2 *__restrict__ child_out)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if(k < n)
    {
        const uint32_t d = leaf_pos[k];
        if(d >= n) return;// only a malformed tree gets here; its depth is rejected
        order_out[d] = order_in[k];
    }
    if(k < ni)
    {
        const int2 c = child_in[k];
        auto map = [leaf_pos](int32_t r) { return r < 0 ? ~static_cast<int32_t>(leaf_pos[~r]) : r; };
        child_out[k] = make_int2(map(c.x), map(c.y));
    }
}

__global__ void __launch_bounds__(1024) k_scan_local(const uint32_t *__restrict__ in, uint32_t n,
                                                     uint32_t *__restrict__ out, uint32_t *__restrict__ block_sums)
{
    __shared__ uint32_t wsum[16];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t i = blockIdx.x * 1024 + threadIdx.x;
    const uint32_t x = i < n ? in[i] : 0u;
    uint32_t sc = x;
    for(int off = 1; off < 64; off <<= 1)
    {
        const uint32_t y = __shfl_up(sc, off);
        if(lane >= (uint32_t)off) sc += y;
    }
    if(lane == 63) wsum[wave] = sc;
    __syncthreads();
    if(threadIdx.x < 16)
    {
        const uint32_t w = wsum[threadIdx.x];
        uint32_t acc = w;
        for(int off = 1; off < 16; off <<= 1)
        {
            const uint32_t y = __shfl_up(acc, off, 16);
            if(threadIdx.x >= (uint32_t)off) acc += y;
        }
        wsum[threadIdx.x] = acc - w;
        if(threadIdx.x == 15) block_sums[blockIdx.x] = acc;
    }
    __syncthreads();
    if(i < n) out[i] = wsum[wave] + sc - x;
}

//! exclusive scan of the per-block sums in one workgroup, 1024 at a time with a running carry
__global__ void __launch_bounds__(1024) k_scan_blocks(uint32_t *__restrict__ data, uint32_t n)
{
    __shared__ uint32_t wsum[16];
    __shared__ uint32_t carry;
    if(threadIdx.x == 0) carry = 0;
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for(uint32_t base = 0; base < n; base += 1024)
    {
        const uint32_t i = base + threadIdx.x;
        const uint32_t x = i < n ? data[i] : 0u;
        uint32_t sc = x;
        for(int off = 1; off < 64; off <<= 1)
        {
            const uint32_t y = __shfl_up(sc, off);
            if(lane >= (uint32_t)off) sc += y;
        }
        if(lane == 63) wsum[wave] = sc;
        __syncthreads();
        if(threadIdx.x < 16)
        {
            const uint32_t w = wsum[threadIdx.x];
            uint32_t acc = w;
            for(int off = 1; off < 16; off <<= 1)
            {
                const uint32_t y = __shfl_up(acc, off, 16);
                if(threadIdx.x >= (uint32_t)off) acc += y;
            }
            wsum[threadIdx.x] = acc - w;
        }
        __syncthreads();
        const uint32_t c = carry;
        if(i < n) data[i] = c + wsum[wave] + sc - x;
        __syncthreads();
        if(threadIdx.x == 1023) carry = c + wsum[wave] + sc;
        __syncthreads();
    }
}

__global__ void __launch_bounds__(1024) k_scan_add(const uint32_t *__restrict__ in, uint32_t n,
                                                   uint32_t *__restrict__ out, const uint32_t *__restrict__ block_off,
                                                   uint32_t *__restrict__ total)
{
    const uint32_t i = blockIdx.x * 1024 + threadIdx.x;
    if(i >= n) return;
    const uint32_t v = out[i] + block_off[blockIdx.x];
    out[i] = v;
    if(i == n - 1) *total = v + in[i];
}

//! exclusive prefix sum of n values; *total receives the sum. block_sums holds div_up(n, 1024) entries
static void exclusive_scan(hipStream_t s, const uint32_t *in, uint32_t *out, uint32_t n, uint32_t *block_sums,
                           uint32_t *total)
{
    const uint32_t nb = div_up(n, 1024);
    k_scan_local<<<nb, 1024, 0, s>>>(in, n, out, block_sums);
    k_scan_blocks<<<1, 1024, 0, s>>>(block_sums, nb);
    k_scan_add<<<nb, 1024, 0, s>>>(in, n, out, block_sums, total);
}

static void build_topology_ploc(vkrt_ctx *ctx, vkrt_bvh *bvh)
{
    hipStream_t s = ctx->stream;
    const uint32_t radius = bvh->ploc_radius ? bvh->ploc_radius : PLOC_RADIUS;
    const uint32_t n = bvh->n_tri, ni = n - 1;
    // working set: two cluster lists (ids, lo, hi), neighbours, flags and offsets, leaf counts, scan sums
    device_buffer &w = ctx->scratch[3];
    const size_t nb = div_up(n, 1024);
    const size_t bytes = (size_t)n * (2 * 4 + 4 * 16 + 4 + 4 * 4 + 4 + 4) + (size_t)ni * 8 + nb * 4 + 512;
    w.reserve(bytes);
    uint8_t *q = w.as<uint8_t>();
    auto take = [&q](size_t b) {
        uint8_t *r = q;
        q += (b + 15) & ~size_t(15);
        return r;
    };
    int32_t *id[2] = {reinterpret_cast<int32_t *>(take((size_t)n * 4)), reinterpret_cast<int32_t *>(take((size_t)n * 4))};
    float4 *lo[2] = {reinterpret_cast<float4 *>(take((size_t)n * 16)), reinterpret_cast<float4 *>(take((size_t)n * 16))};
    float4 *hi[2] = {reinterpret_cast<float4 *>(take((size_t)n * 16)), reinterpret_cast<float4 *>(take((size_t)n * 16))};
    int32_t *nn = reinterpret_cast<int32_t *>(take((size_t)n * 4));
    uint32_t *merge = reinterpret_cast<uint32_t *>(take((size_t)n * 4));
    uint32_t *moff = reinterpret_cast<uint32_t *>(take((size_t)n * 4));
    uint32_t *keep = reinterpret_cast<uint32_t *>(take((size_t)n * 4));
    uint32_t *koff = reinterpret_cast<uint32_t *>(take((size_t)n * 4));
    uint32_t *leaf_pos = reinterpret_cast<uint32_t *>(take((size_t)n * 4));
    uint32_t *cnt = reinterpret_cast<uint32_t *>(take((size_t)ni * 4));
    uint32_t *sums = reinterpret_cast<uint32_t *>(take(nb * 4));
    uint32_t *totals = reinterpret_cast<uint32_t *>(take(16));
    int32_t *parent_int = reinterpret_cast<int32_t *>(take((size_t)ni * 4));
    int32_t *parent_leaf = reinterpret_cast<int32_t *>(take((size_t)n * 4));
    VKRT_REQUIRE(q <= w.as<uint8_t>() + bytes, "PLOC working set overrun");

    int2 *child = bvh->child.as<int2>();
    k_ploc_init<<<div_up(n, 256), 256, 0, s>>>(bvh->tbox.as<float>(), n, id[0], lo[0], hi[0], parent_int, ni);
    uint32_t nc = n, base = 0;
    int cur = 0;
    uint32_t rounds = 0;
    while(nc > 1)
    {
        VKRT_REQUIRE(++rounds <= n, "PLOC made no progress");
        k_ploc_nn<<<div_up(nc, PLOC_BLOCK), PLOC_BLOCK, 0, s>>>(lo[cur], hi[cur], nc, static_cast<int>(radius), nn);
        k_ploc_flags<<<div_up(nc, 256), 256, 0, s>>>(nn, nc, merge, keep);
        exclusive_scan(s, merge, moff, nc, sums, totals);
        exclusive_scan(s, keep, koff, nc, sums, totals + 1);
        k_ploc_merge<<<div_up(nc, 256), 256, 0, s>>>(nn, nc, merge, moff, keep, koff, base, id[cur], lo[cur], hi[cur],
                                                     id[cur ^ 1], lo[cur ^ 1], hi[cur ^ 1], child, cnt, parent_int,
                                                     parent_leaf);
        uint32_t t[2];
        VKRT_HIP(hipMemcpyAsync(t, totals, 8, hipMemcpyDeviceToHost, s));
        VKRT_HIP(hipStreamSynchronize(s));
        VKRT_REQUIRE(t[0] >= 1 && t[1] == nc - t[0], "PLOC round inconsistent");
        base += t[0];
        nc = t[1];
        cur ^= 1;
    }
    VKRT_REQUIRE(base == ni, "PLOC did not build n - 1 nodes");
    // the cluster lists and flag arrays are free now: renumbered tree (root first), then depth-first leaf
    // positions and ranges, then the permuted copies
    int2 *child2 = reinterpret_cast<int2 *>(lo[0]);
    uint32_t *cnt2 = merge;
    int32_t *pint2 = reinterpret_cast<int32_t *>(moff);
    int32_t *pleaf2 = reinterpret_cast<int32_t *>(keep);
    k_ploc_renumber<<<div_up(n, 256), 256, 0, s>>>(ni, n, child, cnt, parent_int, parent_leaf, child2, cnt2, pint2,
                                                   pleaf2);
    k_ploc_dfs<<<div_up(n, 256), 256, 0, s>>>(ni, n, child2, cnt2, pint2, pleaf2, leaf_pos, bvh->range.as<uint2>());
    uint32_t *order_in = koff;
    VKRT_HIP(hipMemcpyAsync(order_in, bvh->order.ptr, (size_t)n * 4, hipMemcpyDeviceToDevice, s));
    k_ploc_permute<<<div_up(n, 256), 256, 0, s>>>(ni, n, leaf_pos, order_in, bvh->order.as<uint32_t>(), child2, child);
    VKRT_HIP(hipGetLastError());
}

//! the leaf records, the BVH2's nodes and the root, from the mesh and a topology: the last part of a build and the
//! whole of a refit, which keeps the topology
static void build_bounds(vkrt_ctx *ctx, vkrt_bvh *bvh, const mesh_view &mesh)
{
    hipStream_t s = ctx->stream;
    const uint32_t n = bvh->n_tri;
    bvh->tris.reserve((size_t)n * 3 * sizeof(float4));
    k_leaves<true><<<div_up(n, 256), 256, 0, s>>>(mesh, bvh->order.as<uint32_t>(), bvh->tbox.as<float>(),
                                                  bvh->tris.as<float4>());
    if(n >= 2)
    {
        const uint32_t ni = n - 1;
        // scratch: per-leaf prefix and suffix unions, then the segments' sparse table
        const uint32_t nseg = div_up(n, BOX_SEG), levels = box_levels(nseg);
        device_buffer &w = ctx->scratch[3];
        w.reserve(((size_t)2 * n + (size_t)levels * nseg) * 6 * sizeof(float));
        float *pre = w.as<float>(), *suf = pre + 6 * (size_t)n, *table = suf + 6 * (size_t)n;
        k_box_scan<<<nseg, BOX_SEG, 0, s>>>(n, bvh->tbox.as<float>(), pre, suf, table);
        for(uint32_t k = 1; k < levels; ++k)
            k_box_sparse<<<div_up(nseg, 256), 256, 0, s>>>(nseg, k, table);
        bvh->n_nodes = ni;
        bvh->nodes.reserve((size_t)ni * sizeof(vkrt_bvh_node));
        const leaf_unions l{bvh->tbox.as<float>(), pre, suf, table, n, nseg};
        k_layout<<<div_up(ni, 256), 256, 0, s>>>(l, bvh->child.as<int2>(), bvh->range.as<uint2>(), bvh->max_leaf,
                                                 bvh->nodes.as<vkrt_bvh_node>());
        bvh->root_ref = (n <= bvh->max_leaf) ? ~static_cast<int>(n - 1) : 0;
    }
    else
    {
        bvh->n_nodes = 0;
        bvh->root_ref = ~0;// a leaf holding the single triangle
    }
    VKRT_HIP(hipGetLastError());
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
    int32_t src;// (BVH2 parent node << 1) | side: where the box is stored, re-read by a refit
    float lo[3], hi[3];
};

__device__ __forceinline__ collapse_child child_of(const vkrt_bvh_node &nd, int32_t node, int k)
{
    collapse_child c;
    const float4 xy = k == 0 ? nd.a : nd.b;
    c.ref = k == 0 ? nd.d.x : nd.d.y;
    c.src = (node << 1) | k;
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
//! build then fails. n4 null: the sums only.
constexpr uint32_t COLLAPSE_BLOCK = 256, COLLAPSE_GRID = 1024;
__global__ void __launch_bounds__(COLLAPSE_BLOCK) k_collapse(const vkrt_bvh_node *__restrict__ n2,
                                                             int4 *__restrict__ queue, uint32_t level,
                                                             vkrt_bvh4_node *__restrict__ n4,
                                                             bvh_state *__restrict__ st)
{
    __shared__ uint32_t wave_sum[COLLAPSE_BLOCK / 64], slot_base;
    __shared__ double wave_sah[COLLAPSE_BLOCK / 64];
    __shared__ uint32_t wave_leaves[COLLAPSE_BLOCK / 64], wave_depth[COLLAPSE_BLOCK / 64],
            wave_stack[COLLAPSE_BLOCK / 64];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t first = 0;// the level's first node
    for(uint32_t l = 0; l < level; ++l) first += st->level[l];
    const uint32_t count = st->level[level], next = first + count;
    double sah = 0.0;
    uint32_t leaves = 0, depth = 0, stack = 0;
    for(uint32_t base = blockIdx.x * COLLAPSE_BLOCK; base < count; base += gridDim.x * COLLAPSE_BLOCK)
    {
        const bool active = base + threadIdx.x < count;
        const uint32_t me = first + base + threadIdx.x;
        collapse_child ch[4];
        uint32_t ch_depth[4] = {0, 0, 0, 0};// depth of the BVH2 node each child came from
        int cnt = 0;
        uint32_t inner = 0, depth_here = 0;
        if(active)
        {
            const int4 item = queue[me];
            auto open = [&](int slot_a, int slot_b, int32_t node, uint32_t d) {
                const vkrt_bvh_node nd = n2[node];
                ch[slot_a] = child_of(nd, node, 0);
                ch[slot_b] = child_of(nd, node, 1);
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
            int32_t refs[4], srcs[4];
#pragma unroll
            for(int j = 0; j < 4; ++j)
            {
                srcs[j] = j < cnt ? ch[j].src : -1;
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
            out.src = make_int4(srcs[0], srcs[1], srcs[2], srcs[3]);
            if(n4) n4[me] = out;
        }
    }
    if(blockIdx.x * COLLAPSE_BLOCK >= count) return;// (the whole workgroup: it had no item)
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

__global__ void k_collapse_root(int4 *__restrict__ queue, bvh_state *__restrict__ st)
{
    queue[0] = make_int4(0, 0, 1, 0);
    st->level[0] = 1u;
}

//! refit of the 4-wide layout: every used child slot re-reads its box from the BVH2 node it was collapsed
//! from (the BVH2 keeps its topology and node numbering on refit), so the collapse's shape, its worst-case
//! stack depth and the choice of the 4-wide walk stay what the build recorded
__global__ void k_wide_refit(const vkrt_bvh_node *__restrict__ n2, uint32_t n4_count, vkrt_bvh4_node *__restrict__ n4)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n4_count) return;
    vkrt_bvh4_node nd = n4[i];
    float *lox = &nd.lox.x, *hix = &nd.hix.x, *loy = &nd.loy.x, *hiy = &nd.hiy.x, *loz = &nd.loz.x, *hiz = &nd.hiz.x;
    const int32_t src[4] = {nd.src.x, nd.src.y, nd.src.z, nd.src.w};
    for(int j = 0; j < 4; ++j)
    {
        if(src[j] < 0) continue;
        const vkrt_bvh_node p = n2[src[j] >> 1];
        const collapse_child c = child_of(p, src[j] >> 1, src[j] & 1);
        lox[j] = c.lo[0];
        hix[j] = c.hi[0];
        loy[j] = c.lo[1];
        hiy[j] = c.hi[1];
        loz[j] = c.lo[2];
        hiz[j] = c.hi[2];
    }
    n4[i] = nd;
}

//! refreshes the boxes of an existing 4-wide layout after the BVH2 was refitted (no change of shape)
static void refit_wide(vkrt_ctx *ctx, vkrt_bvh *bvh)
{
    if(bvh->empty || !bvh->wide || bvh->root4 < 0 || bvh->n_nodes4 == 0) return;
    k_wide_refit<<<div_up(bvh->n_nodes4, 256), 256, 0, ctx->stream>>>(bvh->nodes.as<vkrt_bvh_node>(), bvh->n_nodes4,
                                                                       bvh->nodes4.as<vkrt_bvh4_node>());
    VKRT_HIP(hipGetLastError());
}

//! the end of a build: the BVH2 collapsed into the BVH4 used for traversal (kept off when its worst-case stack
//! depth exceeds STACK_SIZE), the tree's statistics, and what the kernels before found wrong
static void build_wide(vkrt_ctx *ctx, vkrt_bvh *bvh)
{
    hipStream_t s = ctx->stream;
    bvh->wide = false;
    bvh->n_nodes4 = 0;
    bvh->stack4 = 0;
    auto check_indices = [](const bvh_state &st) {
        if(st.err) throw error(VKRT_E_INVALID_ARG, "triangle index out of range of the vertex count");
    };
    if(bvh->root_ref < 0)
    {
        check_indices(read_state(ctx, nullptr));
        bvh->root4 = bvh->root_ref;// a single leaf
        bvh->wide = bvh->allow_wide;
        single_leaf_info(bvh, s);
        return;
    }
    // (a 4-wide node takes in at least one node of the binary tree)
    const size_t cap = bvh->n_nodes;
    ctx->scratch[2].reserve(cap * sizeof(int4));
    int4 *queue = ctx->scratch[2].as<int4>();
    vkrt_bvh4_node *n4 = nullptr;
    if(bvh->allow_wide)
    {
        ctx->scratch[3].reserve(cap * sizeof(vkrt_bvh4_node));
        n4 = ctx->scratch[3].as<vkrt_bvh4_node>();
    }
    const vkrt_bvh_node *n2 = bvh->nodes.as<vkrt_bvh_node>();
    bvh_state *st = ctx->state.as<bvh_state>();
    k_collapse_root<<<1, 1, 0, s>>>(queue, st);
    // the levels are launched without asking how many there are: as many as balanced trees of this size have and
    // some more (a level that is not there costs its launch, 2 us), then in turns until the last one is empty
    uint32_t level = 0, todo = 6;
    for(size_t k = 1; k < cap; k *= 4) ++todo;
    const bvh_state *got = nullptr;
    while(true)
    {
        for(uint32_t stop = std::min(level + todo, MAX_LEVELS); level < stop; ++level)
        {
            const uint64_t most = std::min<uint64_t>(cap, level < 16 ? 1ull << (2 * level) : cap);
            k_collapse<<<std::min(COLLAPSE_GRID, div_up(most, COLLAPSE_BLOCK)), COLLAPSE_BLOCK, 0, s>>>(n2, queue, level,
                                                                                                         n4, st);
        }
        got = &read_state(ctx, n2);
        check_indices(*got);
        if(got->depth > (uint32_t)STACK_SIZE) throw error(VKRT_E_INTERNAL, "BVH deeper than the traversal stack");
        if(got->level[level] == 0) break;
        VKRT_REQUIRE(level < MAX_LEVELS, "BVH4 collapse did not end");
        todo = 4;
    }
    uint64_t total = 0;
    for(uint32_t l = 0; l < level; ++l) total += got->level[l];
    VKRT_REQUIRE(total <= cap, "BVH4 collapse overflow");
    vkrt_bvh_info &info = bvh->info;
    float rb[6];
    root_bounds(got->root, rb, info.bounds);
    const double dx = std::max(0.0, (double)rb[1] - rb[0]), dy = std::max(0.0, (double)rb[3] - rb[2]),
                 dz = std::max(0.0, (double)rb[5] - rb[4]);
    const double root_area = std::max(1e-30, 2.0 * (dx * dy + dy * dz + dz * dx));
    info.depth = std::max(1u, got->depth);
    info.sah_cost = static_cast<float>(1.0 + got->sah / root_area);// 1: the root's own visit
    info.n_leaves = got->leaves;
    if(!bvh->allow_wide) return;
    bvh->n_nodes4 = static_cast<uint32_t>(total);
    bvh->stack4 = got->stack;
    bvh->root4 = 0;
    // the nodes move from the scratch, sized for the most there could be, into an array of their number
    const size_t bytes = (size_t)bvh->n_nodes4 * sizeof(vkrt_bvh4_node);
    bvh->nodes4.reserve(bytes);
    VKRT_HIP(hipMemcpyAsync(bvh->nodes4.ptr, n4, bytes, hipMemcpyDeviceToDevice, s));
    // the 4-wide walk addresses nodes with 32-bit byte offsets (node4_intervals)
    bvh->wide = bvh->stack4 <= (uint32_t)STACK_SIZE && (uint64_t)bytes <= 0xffffffffull;
}

//! the rest of the info block after a build or a refit
static void refresh_info(vkrt_bvh *bvh)
{
    bvh->info.n_tri = bvh->n_tri;
    bvh->info.n_nodes = bvh->n_nodes;
    bvh->info.device_bytes = bvh->nodes.bytes + bvh->tris.bytes + bvh->nodes4.bytes;
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
            bvh->indices.reserve((size_t)n_tri * 3 * sizeof(uint32_t));
            const uint32_t *didx = input(ctx, 1, indices, (size_t)n_tri * 3, flags);
            VKRT_HIP(hipMemcpyAsync(bvh->indices.ptr, didx, (size_t)n_tri * 3 * sizeof(uint32_t),
                                    hipMemcpyDeviceToDevice, ctx->stream));
            const mesh_view mesh{dpos, bvh->indices.as<uint32_t>(), stride_bytes, n_tri, n_vert};
            build_topology(ctx, bvh.get(), mesh);
            build_bounds(ctx, bvh.get(), mesh);
            build_wide(ctx, bvh.get());
            VKRT_HIP(hipStreamSynchronize(ctx->stream));
        }
        else single_leaf_info(bvh.get(), ctx->stream);
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
        build_bounds(ctx, bvh, mesh_view{dpos, bvh->indices.as<uint32_t>(), stride_bytes, bvh->n_tri, bvh->n_vert});
        refit_wide(ctx, bvh);
        if(bvh->root_ref < 0) single_leaf_info(bvh, s);
        else
        {
            // the topology stays, and with it depth, leaves and SAH cost: only the bounds change
            float rb[6];
            root_bounds(read_state(ctx, bvh->nodes.as<vkrt_bvh_node>()).root, rb, bvh->info.bounds);
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
        fetch(bvh->nodes.ptr, (size_t)bvh->n_nodes * sizeof(vkrt_bvh_node), true, h_nodes);
        if(bvh->wide) fetch(bvh->nodes4.ptr, (size_t)bvh->n_nodes4 * sizeof(vkrt_bvh4_node), true, h_nodes4);
        fetch(bvh->tris.ptr, (size_t)n * 3 * sizeof(float4), true, h_tris);
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
                std::memcpy(&orig, &tris[3 * (size_t)k + 2].y, 4);
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
