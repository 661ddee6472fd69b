// bvh_types.hpp - BVH layout shared by the build, the traversal kernels and the C ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "context.hpp"

//! BVH2 node holding both children's boxes (64 B, four 16-B loads)
struct vkrt_bvh_node
{
    float4 a;// child 0: lo.x hi.x lo.y hi.y
    float4 b;// child 1: lo.x hi.x lo.y hi.y
    float4 c;// lo.z hi.z of child 0, lo.z hi.z of child 1
    int4 d;  // child refs: >= 0 internal node, < 0 leaf ~((first << 3) | (count - 1))
};

//! 4-wide node collapsed from the BVH2 (128 B): children's boxes by plane, so one node visit is seven
//! 16-B loads and four slab tests; an unused slot has child ref EMPTY_CHILD (its box is never read)
struct vkrt_bvh4_node
{
    float4 lox, hix, loy, hiy, loz, hiz;
    int4 child;// >= 0 BVH4 node, < 0 leaf (the BVH2 leaf encoding), EMPTY_CHILD unused
    int4 pad;
};

namespace vkrt
{
//! the walk that a BVH's layout takes: the binary tree, or the 4-wide collapse with nodes and records within reach of
//! one base (joint) or each from its own
enum walk_layout : uint32_t
{
    WALK_BINARY = 0,
    WALK_JOINT = 1,
    WALK_APART = 2
};
}// namespace vkrt

struct vkrt_bvh
{
    //! a part of the BVH's one allocation
    struct part
    {
        void *ptr = nullptr;
        size_t bytes = 0;
        template<class T>
        T *as() const
        {
            return static_cast<T *>(ptr);
        }
    };
    int device = 0;
    uint32_t n_tri = 0, n_vert = 0, n_nodes = 0, max_leaf = 4;
    uint32_t builder = 0;// VKRT_BUILDER_*
    uint32_t ploc_radius = 0;// 0: default
    int32_t root_ref = 0;
    bool empty = true;
    // One allocation holds the 4-wide collapse, used by traversal when its worst-case stack fits (wide == true), the
    // leaf records behind it, so that a walk reaches both with 32-bit offsets from one base (joint == true unless
    // they pass 4 GiB, from some 41M triangles at two a leaf), and what a refit needs: the mesh's indices, the
    // leaves' order and the run of leaves below each 4-wide node. (Freeing a large allocation takes 250 to 500 us:
    // eight of them took 1.7 of the 4.1 ms that building and destroying a 1.8M-triangle BVH took.)
    vkrt::device_buffer memory;
    part nodes4, tris, indices, order, wide_range;
    uint32_t node_cap = 0;// 4-wide nodes there is room for
    // the binary tree with its children and runs, kept only where traversal walks it: no 4-wide collapse
    vkrt::device_buffer binary;
    part nodes, child, range;
    bool joint = true;
    int32_t root4 = 0;
    uint32_t n_nodes4 = 0, stack4 = 0;
    bool wide = false, allow_wide = true;
    vkrt_bvh_info info{};

    vkrt::walk_layout walk() const { return !wide ? vkrt::WALK_BINARY : joint ? vkrt::WALK_JOINT : vkrt::WALK_APART; }
};

namespace vkrt
{

constexpr int32_t MAX_LEAF = 8;
constexpr int STACK_SIZE = 64;      // traversal stack entries per ray; the build rejects deeper trees
constexpr float BOX_PAD = 0x1p-16f; // relative growth of every stored box coordinate
constexpr float T_PAD = 0x1p-16f;   // relative growth of every slab interval
constexpr uint32_t TRI_TWO_SIDED = 1u;// flag bit in a leaf triangle record: never culled as a back face
constexpr uint32_t TRI_ALPHA_MASK = 2u;// flag bit: the record's material is alpha-masked (any-hit test)
//! a leaf record: v0, e1, e2 (nine floats), original triangle index, material, flags, and a gap of 16 B. At 64 B two
//! records lie like the seven 16-B words of a 4-wide node (see fetch7), and none crosses a 64-B line
constexpr uint32_t TRI_BYTES = 64;
constexpr int32_t EMPTY_CHILD = 0x7fffffff;// unused BVH4 child slot (no node index reaches it)

}// namespace vkrt
