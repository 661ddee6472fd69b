// intersect.hip - batched versions of vierkant's intersect(...) overloads and the brute-force
// closest/any-hit loop, for gfx950.
//
// Pairwise kernels evaluate the reference arithmetic (vierkant/rt_math.hpp) one element per lane.
// The brute-force kernel tiles (rays x triangle chunks): the matrix cores sort out the pairs that can hit, those
// take the reference's test, and a lane merges its best hit into a per-ray 64-bit key (ordered t << 32 | prim)
// with one atomic min, so ties on t resolve to the lowest triangle index no matter which chunk finishes first.
#include <cfloat>
#include <mutex>

#include "context.hpp"
#include "kernels.hpp"
#include "vierkant/rt_math.hpp"

using namespace vierkant::rt;

namespace vkrt
{

__device__ __forceinline__ vec3 ld3(const float *p) { return vec3{p[0], p[1], p[2]}; }

__device__ __forceinline__ void load_ray(const float4 *__restrict__ rays, uint32_t i, vec3 &o, float &tmin, vec3 &d,
                                         float &tmax)
{
    float4 a = rays[2 * i], b = rays[2 * i + 1];
    o = vec3{a.x, a.y, a.z};
    tmin = a.w;
    d = vec3{b.x, b.y, b.z};
    tmax = b.w;
}

// ---------------------------------------------------------------------------------------------
// pairwise tests
// ---------------------------------------------------------------------------------------------
__global__ void k_pair_tri(const float *__restrict__ tris, const float4 *__restrict__ rays, uint32_t n,
                           vkrt_tri_result *__restrict__ out)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n) return;
    vec3 o, d;
    float tmin, tmax;
    load_ray(rays, i, o, tmin, d, tmax);
    const float *t9 = tris + 9 * (size_t)i;
    vec3 v0 = ld3(t9), v1 = ld3(t9 + 3), v2 = ld3(t9 + 6);
    float t = 0.f, u = 0.f, v = 0.f;
    bool hit = mt_reference(o, d, v0, v1 - v0, v2 - v0, t, u, v);
    out[i] = hit ? vkrt_tri_result{INTERSECT, t, u, v} : vkrt_tri_result{REJECT, 0.f, 0.f, 0.f};
}

__global__ void k_pair_aabb(const float *__restrict__ boxes, const float4 *__restrict__ rays, uint32_t n,
                            vkrt_result *__restrict__ out)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n) return;
    vec3 o, d;
    float tmin, tmax;
    load_ray(rays, i, o, tmin, d, tmax);
    const float *b = boxes + 6 * (size_t)i;
    float dist = 0.f;
    uint32_t type = aabb_reference(ld3(b), ld3(b + 3), o, d, dist);
    out[i] = vkrt_result{type, type ? dist : 0.f};
}

__global__ void k_pair_obb(const float *__restrict__ obbs, const float4 *__restrict__ rays, uint32_t n,
                           vkrt_result *__restrict__ out)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n) return;
    vec3 o, d;
    float tmin, tmax;
    load_ray(rays, i, o, tmin, d, tmax);
    const float *b = obbs + 15 * (size_t)i;
    const vec3 axis[3] = {ld3(b + 3), ld3(b + 6), ld3(b + 9)};
    float dist = 0.f;
    uint32_t type = obb_reference(ld3(b), axis, ld3(b + 12), o, d, dist);
    out[i] = vkrt_result{type, type ? dist : 0.f};
}

__global__ void k_pair_sphere(const float *__restrict__ spheres, const float4 *__restrict__ rays, uint32_t n,
                              vkrt_result *__restrict__ out)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n) return;
    vec3 o, d;
    float tmin, tmax;
    load_ray(rays, i, o, tmin, d, tmax);
    const float *s = spheres + 4 * (size_t)i;
    float dist = 0.f;
    uint32_t type = sphere_reference(ld3(s), s[3], o, d, dist);
    out[i] = vkrt_result{type, type ? dist : 0.f};
}

__global__ void k_pair_plane(const float *__restrict__ planes, const float4 *__restrict__ rays, uint32_t n,
                             vkrt_result *__restrict__ out)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n) return;
    vec3 o, d;
    float tmin, tmax;
    load_ray(rays, i, o, tmin, d, tmax);
    const float *p = planes + 4 * (size_t)i;
    const float c[4] = {p[0], p[1], p[2], p[3]};
    float dist = 0.f;
    uint32_t type = plane_reference(c, o, d, dist);
    out[i] = vkrt_result{type, type ? dist : 0.f};
}

__global__ void k_pair_tri_box(const float *__restrict__ tris, const float *__restrict__ boxes, uint32_t n,
                               uint32_t *__restrict__ out)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n) return;
    float t[9], b[6];
    for(int k = 0; k < 9; ++k) t[k] = tris[9 * (size_t)i + k];
    for(int k = 0; k < 6; ++k) b[k] = boxes[6 * (size_t)i + k];
    out[i] = tri_box_overlap(t, b, b + 3);
}

__global__ void k_pair_tri_tri(const float *__restrict__ ta, const float *__restrict__ tb, uint32_t n,
                               uint32_t *__restrict__ out)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n) return;
    float a[9], b[9];
    for(int k = 0; k < 9; ++k) a[k] = ta[9 * (size_t)i + k], b[k] = tb[9 * (size_t)i + k];
    out[i] = tri_tri_overlap(a, b);
}

// ---------------------------------------------------------------------------------------------
// shared helpers
// ---------------------------------------------------------------------------------------------
__global__ void k_fill_u64(uint64_t *__restrict__ p, uint32_t n, uint64_t value)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i < n) p[i] = value;
}

__global__ void k_fill_u8(uint8_t *__restrict__ p, uint32_t n, uint8_t value)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i < n) p[i] = value;
}

// ---------------------------------------------------------------------------------------------
// brute force
// ---------------------------------------------------------------------------------------------
// A hit needs a = tvec.(d x e2), b = d.(tvec x e1) and c = det - a - b all of det's sign, and each of the three
// is a product of a vector of the triangle and one of the ray, (edge, vertex x edge) . (o x d, d) in six
// components about any origin: a contraction, so the matrix cores find the few pairs that can hit and only
// those take the reference's test, whose decision and bits stand. With -ffp-contract=off that test is some 45
// VALU instructions a pair; the filter leaves 3.5 of them (min3, max3, max, half a max3) beside six
// 32x32x16 bf16 MFMAs per 32 x 32 pairs.
//
// The factors go in as two bf16 parts each, hi + mid, off by 2^-16 of the factor; a lane's half holds the
// triangle's hi or mid parts and the two MFMAs of a product take the ray's hi and its mid parts. With
// P = |d| E (|f| + V) (E the longest edge and V the farthest vertex of 32 triangles, f the point of the ray's line
// nearest to the origin, all about a vertex of the chunk; o x d = f x d, so rays from far away lose no more than near
// ones) the parts are off by at most 2^-15 P, the 24 terms' sum by less than 2^-19 P, and f itself and the reference's
// own a, b and det by less than 2^-18 |d| E (|o| + V): a pair whose three values are not all above
// -|d| E (2^-14 (|f| + V) + 2^-18 |o|) - 2^-70, nor all below its negative, is no hit of the reference's. 2^-70 covers
// what is lost below the normal range while every factor stays below 2^40; a ray or a tile beyond that takes every pair.
// A triangle with a NaN or an infinity is never hit (det is not finite, so t comes out NaN or 0 x infinity): it takes the
// place of another one of its tile in the filter and fails the reference's test where that one is asked for.
//
// 65,536 rays x 20,480 triangles: 1,210 us with the reference's test for every pair, 242 so (origins a thousand radii
// away 375, without f 1,630; the scene at 1e13, where nothing has a bound, 1,196, and 1,590 where a record is read for
// each ray of a lane; a NaN in every 256th triangle or every 32nd ray 270, and 1,540 where it takes its chunk's or its
// wave's bound with it), the matrix cores busy for 48 % of them and 69 VALU instructions a wave per 32 x 32 pairs,
// 48 of them the filter's. Two products of 32 x 32 in flight per wave, at two or three waves a SIMD, are no faster:
// 248 - 255.
constexpr float BRUTE_LIMIT = 0x1p40f;
constexpr int BRUTE_STAGE = 256;// triangles in LDS at a time, one a thread
constexpr int BRUTE_TILES = BRUTE_STAGE / 32;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

//! six values as two bf16 parts each, two zeros behind
__device__ __forceinline__ void split_bf16(const vec3 &p, const vec3 &q, bf16x8 &hi, bf16x8 &mid)
{
    const float x[8] = {p.x, p.y, p.z, q.x, q.y, q.z, 0.f, 0.f};
#pragma unroll
    for(int k = 0; k < 8; ++k)
    {
        hi[k] = static_cast<__bf16>(x[k]);
        mid[k] = static_cast<__bf16>(x[k] - static_cast<float>(hi[k]));
    }
}

//! no smaller than |v|, also where the squares underflow
__device__ __forceinline__ float norm_above(const vec3 &v) { return sqrtf(dot(v, v)) + 0x1p-60f; }

__device__ __forceinline__ bool finite3(const vec3 &v)
{
    return __builtin_isfinite(v.x) && __builtin_isfinite(v.y) && __builtin_isfinite(v.z);
}

__device__ __forceinline__ uint32_t half_wave_max(uint32_t x)
{
#pragma unroll
    for(int off = 16; off > 0; off >>= 1) x = max(x, static_cast<uint32_t>(__shfl_xor(static_cast<int>(x), off)));
    return x;
}

//! the smallest of three values, and of their negatives: neither reaches zero unless all lie on one side of it
__device__ __forceinline__ float above(float a, float b, float c) { return fminf(fminf(a, b), c); }
__device__ __forceinline__ float below(float a, float b, float c) { return fminf(fminf(-a, -b), -c); }

//! the middle one of three values; of those that are numbers where one or two are NaN
__device__ __forceinline__ float middle(float a, float b, float c) { return fmaxf(fminf(a, b), fminf(fmaxf(a, b), c)); }

//! a wave takes 32 * GROUPS rays over its workgroup's triangles; lanes l and l + 32 hold one ray, and 16
//! triangles each of every 32
template<bool ANY, int GROUPS>
__global__ void __launch_bounds__(256, GROUPS > 2 ? 3 : 4) k_brute(const float4 *__restrict__ rays, uint32_t n_ray,
                                                  const float *__restrict__ tris, uint32_t n_tri, uint32_t chunk,
                                                  uint64_t *__restrict__ keys, uint8_t *__restrict__ occluded)
{
    __shared__ bf16x8 parts[BRUTE_TILES][3][64];
    __shared__ float4 records[BRUTE_STAGE][3];// v0, e1, e2 for the reference's test
    __shared__ float2 extent[BRUTE_TILES];    // E, V

    const uint32_t lane = threadIdx.x & 63u, half = lane >> 5;
    const uint32_t t0 = blockIdx.y * chunk, count = min(n_tri - t0, chunk);
    // the origin for the chunk, a vertex that one stray or non-finite triangle does not carry off
    const vec3 c0 = ld3(tris + 9 * (size_t)t0), c1 = ld3(tris + 9 * (size_t)(t0 + count / 2u)),
               c2 = ld3(tris + 9 * (size_t)(t0 + count - 1u));
    auto origin = [](float a, float b, float c) {
        const float m = middle(a, b, c);
        // (a scalar: the same in every lane, which the compiler does not see)
        return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(fabsf(m) < BRUTE_LIMIT ? m : 0.f)));
    };
    const vec3 centre{origin(c0.x, c1.x, c2.x), origin(c0.y, c1.y, c2.y), origin(c0.z, c1.z, c2.z)};

    bf16x8 ray_hi[GROUPS], ray_mid[GROUPS];
    float ray_d[GROUPS], ray_o[GROUPS], best[GROUPS];
    uint32_t best_i[GROUPS];
    bool unbounded = true;// each group has a ray that takes every pair
    const uint32_t first_ray = (blockIdx.x * 4u + (threadIdx.x >> 6)) * (32u * GROUPS) + (lane & 31u);
#pragma unroll
    for(int g = 0; g < GROUPS; ++g)
    {
        const uint32_t r = first_ray + 32u * g;
        vec3 o{0.f, 0.f, 0.f}, d{0.f, 0.f, 1.f};
        float tmin = 0.f, tmax = -1.f;
        if(r < n_ray) load_ray(rays, r, o, tmin, d, tmax);
        o = o - centre;
        const float dd = dot(d, d);
        const vec3 foot = dd > 0x1p-100f ? o - d * (dot(o, d) / dd) : o;
        split_bf16(cross(foot, d), d, ray_hi[g], ray_mid[g]);
        ray_o[g] = norm_above(foot) + 0x1p-4f * norm_above(o);
        ray_d[g] = norm_above(d);
        bool none = !(tmin < tmax);// no t lies inside
        if(!(ray_o[g] < BRUTE_LIMIT && ray_d[g] < BRUTE_LIMIT && ray_o[g] * ray_d[g] < BRUTE_LIMIT))
        {
            ray_d[g] = __int_as_float(0x7fc00000);
            // a NaN or an infinite origin makes every t a NaN or infinite, an infinite direction makes it NaN or +-0
            none |= !finite3(o) || d.x != d.x || d.y != d.y || d.z != d.z || (tmin >= 0.f && !finite3(d));
        }
        if(none) ray_d[g] = -__int_as_float(0x7f800000);// no pair is taken
        best[g] = tmax;
        best_i[g] = VKRT_INVALID_PRIM;
        unbounded = unbounded && __any(ray_d[g] != ray_d[g]);
    }

    auto test = [&](int g, const vec3 &o, const vec3 &d, float tmin, const float4 &q0, const float4 &q1,
                    const float4 &q2, uint32_t prim) {
        float t, u, v;
        if(!mt_fast_window(o, d, vec3{q0.x, q0.y, q0.z}, vec3{q0.w, q1.x, q1.y}, vec3{q1.z, q1.w, q2.x}, tmin, best[g],
                           t, u, v))
            return;
        // (ANY: the ray takes no pair any more)
        if(ANY) ray_d[g] = -__int_as_float(0x7f800000);
        else best[g] = t;
        best_i[g] = prim;
    };
    for(uint32_t done = 0; done < count; done += BRUTE_STAGE)
    {
        const uint32_t base = t0 + done, n = min(count - done, static_cast<uint32_t>(BRUTE_STAGE));
        if(done) __syncthreads();
        {
            vec3 v0 = centre, e1{0.f, 0.f, 0.f}, e2{0.f, 0.f, 0.f};
            if(threadIdx.x < n)
            {
                const float *t = tris + 9 * (size_t)(base + threadIdx.x);
                v0 = ld3(t);
                e1 = ld3(t + 3) - v0;
                e2 = ld3(t + 6) - v0;
            }
            records[threadIdx.x][0] = make_float4(v0.x, v0.y, v0.z, e1.x);
            records[threadIdx.x][1] = make_float4(e1.y, e1.z, e2.x, e2.y);
            records[threadIdx.x][2] = make_float4(e2.z, 0.f, 0.f, 0.f);
            v0 = v0 - centre;
            float e, v;// E and V of this triangle, E NaN where it has no bound
            auto measure = [&] {
                const float l1 = norm_above(e1);
                e = fmaxf(fmaxf(l1, norm_above(e2)), norm_above(e1 - e2));
                v = norm_above(v0) + l1;
                const bool bounded = e < BRUTE_LIMIT && v < BRUTE_LIMIT && e * v < BRUTE_LIMIT;
                if(!bounded) e = __int_as_float(0x7fc00000);
                return bounded;
            };
            if(__any(!measure()))
            {
                // (stand-ins for triangles that are never hit; a tile of nothing else lies below every bound)
                const bool whole = threadIdx.x < n && finite3(v0) && finite3(e1) && finite3(e2);
                const uint64_t wave_whole = __ballot(whole);
                const uint32_t tile_whole = static_cast<uint32_t>(half ? wave_whole >> 32 : wave_whole);
                const int from = static_cast<int>(32u * half) + max(__ffs(static_cast<int>(tile_whole)) - 1, 0);
                float *part[9] = {&v0.x, &v0.y, &v0.z, &e1.x, &e1.y, &e1.z, &e2.x, &e2.y, &e2.z};
#pragma unroll
                for(int k = 0; k < 9; ++k)
                {
                    const float x = __shfl(*part[k], from);
                    if(!whole) *part[k] = tile_whole ? x : 0.f;
                }
                measure();
                if(!tile_whole) e = -__int_as_float(0x7f800000);
            }
            const vec3 e3 = e1 - e2;
            const uint32_t tile = threadIdx.x >> 5, row = threadIdx.x & 31u;
            bf16x8 hi, mid;
            split_bf16(e2, cross(v0, e2), hi, mid);
            parts[tile][0][row] = hi;
            parts[tile][0][32 + row] = mid;
            split_bf16(vec3{0.f, 0.f, 0.f} - e1, cross(e1, v0), hi, mid);
            parts[tile][1][row] = hi;
            parts[tile][1][32 + row] = mid;
            split_bf16(e3, cross(v0 + e1, e3), hi, mid);
            parts[tile][2][row] = hi;
            parts[tile][2][32 + row] = mid;
            // compared as integers a NaN is above every number, and -infinity above that
            e = __uint_as_float(half_wave_max(__float_as_uint(e)));
            v = __uint_as_float(half_wave_max(__float_as_uint(v) & 0x7fffffffu));
            if(row == 0) extent[tile] = make_float2(e, v);
        }
        __syncthreads();

        const uint32_t n_tile = (n + 31u) / 32u;
        float bound = extent[0].x;
#pragma unroll
        for(int tile = 1; tile < BRUTE_TILES; ++tile) bound = fminf(bound, extent[tile].x);
        if(unbounded || bound != bound)
        {
            // no bound in the whole stage: every pair, a record read once for the lane's rays
            vec3 o[GROUPS], d[GROUPS];
            float tmin[GROUPS];
#pragma unroll
            for(int g = 0; g < GROUPS; ++g)
            {
                float tmax;
                o[g] = d[g] = vec3{0.f, 0.f, 0.f};
                tmin[g] = __int_as_float(0x7f800000);
                if(!(ray_d[g] == -__int_as_float(0x7f800000)))
                    load_ray(rays, first_ray + 32u * g, o[g], tmin[g], d[g], tmax);
            }
#pragma unroll 1
            for(uint32_t row = half; row < n; row += 2u)
            {
                const float4 q0 = records[row][0], q1 = records[row][1], q2 = records[row][2];
#pragma unroll
                for(int g = 0; g < GROUPS; ++g) test(g, o[g], d[g], tmin[g], q0, q1, q2, base + row);
            }
            continue;
        }
        for(uint32_t tile = 0; tile < n_tile; ++tile)
        {
            bf16x8 part[3];
#pragma unroll
            for(int k = 0; k < 3; ++k) part[k] = parts[tile][k][lane];
            const float2 ev = extent[tile];
            const uint32_t row0 = 32u * tile + 4u * half;
#pragma unroll
            for(int g = 0; g < GROUPS; ++g)
            {
                f32x16 m[3];
#pragma unroll
                for(int k = 0; k < 3; ++k)
                {
                    const f32x16 zero = {};
                    m[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(part[k], ray_hi[g], zero, 0, 0, 0);
                    m[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(part[k], ray_mid[g], m[k], 0, 0, 0);
                }
                const float margin = ray_d[g] * ev.x * (ray_o[g] + ev.y) * 0x1p-14f + 0x1p-70f;
                float nearest = -__int_as_float(0x7f800000);
#pragma unroll
                for(int i = 0; i < 16; ++i)
                    nearest = fmaxf(fmaxf(nearest, above(m[0][i], m[1][i], m[2][i])),
                                    below(m[0][i], m[1][i], m[2][i]));
                if(nearest < -margin) continue;

                // a NaN margin gets here for rays that take no pair too, and for those past the end
                if(ray_d[g] == -__int_as_float(0x7f800000)) continue;
                vec3 o, d;
                float tmin, tmax;
                load_ray(rays, first_ray + 32u * g, o, tmin, d, tmax);
                auto test_row = [&](uint32_t row) {
                    test(g, o, d, tmin, records[row][0], records[row][1], records[row][2], base + row);
                };
                if(__any(!(margin < __int_as_float(0x7f800000))))
                {
                    // no bound for some ray: every pair, a step's records asked for ahead of its tests
#pragma unroll 4
                    for(uint32_t i = 0; i < 16; ++i)
                        if(row0 + 8u * (i >> 2) + (i & 3u) < n) test_row(row0 + 8u * (i >> 2) + (i & 3u));
                    continue;
                }
                uint32_t mask = 0;
#pragma unroll
                for(int i = 0; i < 16; ++i)
                    mask |= fmaxf(above(m[0][i], m[1][i], m[2][i]), below(m[0][i], m[1][i], m[2][i])) < -margin
                                ? 0u
                                : 1u << i;
                while(mask)
                {
                    const uint32_t i = __ffs(static_cast<int>(mask)) - 1, row = row0 + 8u * (i >> 2) + (i & 3u);
                    mask &= mask - 1u;
                    if(row >= n) break;
                    test_row(row);
                    if(ANY && ray_d[g] == -__int_as_float(0x7f800000)) break;
                }
            }
            if(ANY)
            {
                bool open = false;
#pragma unroll
                for(int g = 0; g < GROUPS; ++g) open |= !(ray_d[g] == -__int_as_float(0x7f800000));
                if(!__any(open)) break;
            }
        }
    }
#pragma unroll
    for(int g = 0; g < GROUPS; ++g)
    {
        if(best_i[g] == VKRT_INVALID_PRIM) continue;
        if(ANY) occluded[first_ray + 32u * g] = 1;
        else atomicMin((unsigned long long *)&keys[first_ray + 32u * g], hit_key(best[g], best_i[g]));
    }
}

__global__ void k_brute_finalize(const float4 *__restrict__ rays, uint32_t n_ray, const float *__restrict__ tris,
                                 const uint64_t *__restrict__ keys, vkrt_hit *__restrict__ hits)
{
    uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if(r >= n_ray) return;
    uint64_t key = keys[r];
    vkrt_hit h{__int_as_float(0x7f800000), 0.f, 0.f, VKRT_INVALID_PRIM};
    if(key != ~0ull)
    {
        uint32_t prim = static_cast<uint32_t>(key & 0xffffffffu);
        vec3 o, d;
        float tmin, tmax;
        load_ray(rays, r, o, tmin, d, tmax);
        const float *p = tris + 9 * (size_t)prim;
        const vec3 v0 = ld3(p);
        float t = 0.f, u = 0.f, v = 0.f;
        mt_reference(o, d, v0, ld3(p + 3) - v0, ld3(p + 6) - v0, t, u, v);
        h = vkrt_hit{t, u, v, prim};
    }
    hits[r] = h;
}

// ---------------------------------------------------------------------------------------------
// compute_aabb: per axis the first point attaining the min (max), as the sequential glm::min/max
// fold of src/intersection.cpp:100-104 keeps the earlier of equal values; NaN never wins a compare.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ uint64_t wave_min_u64(uint64_t x)
{
    for(int off = 32; off > 0; off >>= 1)
    {
        uint64_t y = __shfl_xor(x, off);
        x = y < x ? y : x;
    }
    return x;
}

__device__ __forceinline__ uint64_t wave_max_u64(uint64_t x)
{
    for(int off = 32; off > 0; off >>= 1)
    {
        uint64_t y = __shfl_xor(x, off);
        x = y > x ? y : x;
    }
    return x;
}

__global__ void __launch_bounds__(256) k_aabb_reduce(const float *__restrict__ pts, uint32_t n,
                                                     uint64_t *__restrict__ keys)
{
    uint64_t mn[3] = {~0ull, ~0ull, ~0ull}, mx[3] = {0, 0, 0};
    for(uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    {
        for(int a = 0; a < 3; ++a)
        {
            float c = pts[3 * (size_t)i + a];
            if(c != c) continue;
            uint64_t ord = ordered_bits(c + 0.0f);
            uint64_t kmin = (ord << 32) | i, kmax = (ord << 32) | (0xffffffffu - i);
            mn[a] = kmin < mn[a] ? kmin : mn[a];
            mx[a] = kmax > mx[a] ? kmax : mx[a];
        }
    }
    for(int a = 0; a < 3; ++a)
    {
        uint64_t lo = wave_min_u64(mn[a]), hi = wave_max_u64(mx[a]);
        if((threadIdx.x & 63) == 0)
        {
            if(lo != ~0ull) atomicMin((unsigned long long *)&keys[a], lo);
            if(hi != 0) atomicMax((unsigned long long *)&keys[3 + a], hi);
        }
    }
}

__global__ void k_aabb_finalize(const float *__restrict__ pts, const uint64_t *__restrict__ keys,
                                float *__restrict__ out6)
{
    int a = threadIdx.x;
    if(a >= 6) return;
    const float init = a < 3 ? FLT_MAX : -FLT_MAX;
    uint64_t k = keys[a];
    float r = init;
    if(a < 3 && k != ~0ull)
    {
        float v = pts[3 * (size_t)(k & 0xffffffffu) + a];
        r = v < init ? v : init;
    }
    else if(a >= 3 && k != 0)
    {
        float v = pts[3 * (size_t)(0xffffffffu - (k & 0xffffffffu)) + (a - 3)];
        r = init < v ? v : init;
    }
    out6[a] = r;
}

//! compute_bounding_sphere (src/intersection.cpp:25-92): the extremum indices come from k_aabb_reduce's
//! keys (first occurrence of the strict minimum / maximum, NaN never wins), then one workgroup seeds the
//! sphere from the axis with the largest squared extent and grows it in index order. Per chunk of 1024
//! points the block finds the first point outside the current sphere, that lane applies the reference's
//! update, and the scan resumes after it: the exact sequential result, in parallel within each chunk.
constexpr int SPHERE_BLOCK = 1024;

__global__ void __launch_bounds__(SPHERE_BLOCK) k_sphere_grow(const float *__restrict__ pts, uint32_t n,
                                                             const uint64_t *__restrict__ keys,
                                                             float *__restrict__ out4)
{
    __shared__ float sph[4];
    __shared__ uint32_t first;
    const uint32_t tid = threadIdx.x;
    if(tid == 0)
    {
        uint32_t pmin[3], pmax[3];
        for(int a = 0; a < 3; ++a)
        {
            const float v0 = pts[a];
            const bool nan0 = v0 != v0;// a NaN first coordinate is never replaced
            pmin[a] = (nan0 || keys[a] == ~0ull) ? 0u : static_cast<uint32_t>(keys[a] & 0xffffffffu);
            pmax[a] = (nan0 || keys[3 + a] == 0ull) ? 0u : 0xffffffffu - static_cast<uint32_t>(keys[3 + a] & 0xffffffffu);
        }
        float best = 0.f;
        int axis = 0;
        for(int a = 0; a < 3; ++a)
        {
            const float *p1 = pts + 3 * (size_t)pmin[a], *p2 = pts + 3 * (size_t)pmax[a];
            const float dx = p2[0] - p1[0], dy = p2[1] - p1[1], dz = p2[2] - p1[2];
            const float d2 = (dx * dx + dy * dy) + dz * dz;
            if(d2 > best)
            {
                best = d2;
                axis = a;
            }
        }
        const float *p1 = pts + 3 * (size_t)pmin[axis], *p2 = pts + 3 * (size_t)pmax[axis];
        sph[0] = (p1[0] + p2[0]) / 2.f;
        sph[1] = (p1[1] + p2[1]) / 2.f;
        sph[2] = (p1[2] + p2[2]) / 2.f;
        sph[3] = sqrtf(best) / 2.f;
    }
    __syncthreads();
    for(uint32_t base = 0; base < n; base += SPHERE_BLOCK)
    {
        const uint32_t i = base + tid;
        float px = 0.f, py = 0.f, pz = 0.f;
        if(i < n)
        {
            px = pts[3 * (size_t)i];
            py = pts[3 * (size_t)i + 1];
            pz = pts[3 * (size_t)i + 2];
        }
        uint32_t start = 0;
        while(true)
        {
            const float cx = sph[0], cy = sph[1], cz = sph[2], r = sph[3];
            const float vx = px - cx, vy = py - cy, vz = pz - cz;
            const float d2 = (vx * vx + vy * vy) + vz * vz;
            const bool outside = i < n && tid >= start && d2 > r * r;
            if(tid == 0) first = 0xffffffffu;
            __syncthreads();
            if(outside) atomicMin(&first, tid);
            __syncthreads();
            const uint32_t f = first;
            if(f == 0xffffffffu) break;
            if(tid == f)
            {
                const float d = sqrtf(d2);
                const float k = 0.5f + (r / d) / 2;
                sph[0] = px * (1.f - k) + cx * k;
                sph[1] = py * (1.f - k) + cy * k;
                sph[2] = pz * (1.f - k) + cz * k;
                sph[3] = (r + d) / 2;
            }
            __syncthreads();
            start = f + 1;
        }
        __syncthreads();
    }
    if(tid == 0)
    {
        out4[0] = sph[0];
        out4[1] = sph[1];
        out4[2] = sph[2];
        out4[3] = sph[3];
    }
}

// ---------------------------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------------------------
void launch_fill_u64(hipStream_t s, uint64_t *p, uint32_t n, uint64_t value)
{
    if(!n) return;
    k_fill_u64<<<div_up(n, 256), 256, 0, s>>>(p, n, value);
}

void launch_fill_u8(hipStream_t s, uint8_t *p, uint32_t n, uint8_t value)
{
    if(!n) return;
    k_fill_u8<<<div_up(n, 256), 256, 0, s>>>(p, n, value);
}

//! launches k_brute over (workgroups of rays) x (chunks of triangles)
template<bool ANY>
static void brute(vkrt_ctx *ctx, const float *tris, uint32_t n_tri, const float4 *rays, uint32_t n_ray,
                  uint64_t *keys, uint8_t *occ)
{
    const uint32_t stages = div_up(n_tri, BRUTE_STAGE);
    // 128 rays a wave spread a triangle's loads and its preparation over more products once each SIMD gets 16 such
    // waves; with fewer, waves of 32 rays fill the card better. 65,536 rays x 80 / 1,280 triangles (512 / 2,560
    // waves of 128): 21 / 34 us with 128 rays, 14 / 32 with 32; 16,384 x 20,480 (10,240): 82 and 78; 32,768 x
    // 20,480 (20,480): 130 and 148
    const bool few = static_cast<uint64_t>(div_up(n_ray, 128)) * stages < 16384;
    const uint32_t blocks = div_up(n_ray, few ? 128 : 512);
    // chunks of whole stages, as many as fill the card some five times over (2,048, 4,096 and 16,384 workgroups:
    // 245, 242 and 255 us) and no more than a grid can have
    const uint32_t chunks = min(stages, min(div_up(4096, blocks), 65535u));
    const uint32_t chunk = min(static_cast<uint64_t>(div_up(stages, chunks)) * BRUTE_STAGE, static_cast<uint64_t>(n_tri));
    const dim3 grid(blocks, div_up(n_tri, chunk));
    if(few) k_brute<ANY, 1><<<grid, 256, 0, ctx->stream>>>(rays, n_ray, tris, n_tri, chunk, keys, occ);
    else k_brute<ANY, 4><<<grid, 256, 0, ctx->stream>>>(rays, n_ray, tris, n_tri, chunk, keys, occ);
}

void brute_closest(vkrt_ctx *ctx, const float *tris, uint32_t n_tri, const float4 *rays, uint32_t n_ray,
                   uint64_t *keys, vkrt_hit *hits)
{
    launch_fill_u64(ctx->stream, keys, n_ray, ~0ull);
    if(n_tri) brute<false>(ctx, tris, n_tri, rays, n_ray, keys, nullptr);
    k_brute_finalize<<<div_up(n_ray, 256), 256, 0, ctx->stream>>>(rays, n_ray, tris, keys, hits);
}

void brute_any(vkrt_ctx *ctx, const float *tris, uint32_t n_tri, const float4 *rays, uint32_t n_ray, uint8_t *occ)
{
    launch_fill_u8(ctx->stream, occ, n_ray, 0);
    if(n_tri) brute<true>(ctx, tris, n_tri, rays, n_ray, nullptr, occ);
}

// ---------------------------------------------------------------------------------------------
// allocation-free brute force: its scratch (the 64-bit hit keys) is
// a file-scope device array, so a call allocates nothing. Each GPU holds its own copy of the array;
// the host reaches it only through the address hipGetSymbolAddress returns on that device (the
// array's name on the host is a stand-in, not a device address).
// ---------------------------------------------------------------------------------------------
constexpr size_t NOALLOC_BYTES = (size_t)VKRT_NOALLOC_MAX_RAY * sizeof(uint64_t);

static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

constexpr int NOALLOC_MAX_DEVICES = 64;
static std::mutex g_scratch_mutex;
static void *g_scratch_ptr[NOALLOC_MAX_DEVICES];

//! resolves `scratch` on the context's device (current when this runs, from vkrt_create), once per device
void noalloc_scratch_init(vkrt_ctx *ctx)
{
    if(ctx->device < 0 || ctx->device >= NOALLOC_MAX_DEVICES) return;// the entry point then reports it
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if(!g_scratch_ptr[ctx->device])
    {
        void *p = nullptr;
        VKRT_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        VKRT_REQUIRE(p, "hipGetSymbolAddress returned no address for the allocation-free scratch");
        g_scratch_ptr[ctx->device] = p;
    }
    ctx->noalloc_scratch = g_scratch_ptr[ctx->device];
}

}// namespace vkrt

// =============================================================================================
// C ABI
// =============================================================================================
using namespace vkrt;

template<class Out, class K>
static int pairwise(vkrt_ctx *ctx, const float *prims, size_t floats_per, const vkrt_ray *rays, uint32_t n, Out *out,
                    int flags, K kernel)
{
    return guarded(ctx, [&] {
        VKRT_REQUIRE(n == 0 || (prims && rays && out), "null array argument");
        if(n == 0) return;
        const float *dp = input(ctx, 0, prims, n * floats_per, flags);
        const vkrt_ray *dr = input(ctx, 1, rays, n, flags);
        Out *dout = output(ctx, 2, out, n, flags);
        kernel<<<div_up(n, 256), 256, 0, ctx->stream>>>(dp, reinterpret_cast<const float4 *>(dr), n, dout);
        VKRT_HIP(hipGetLastError());
        finish_output(ctx, 2, out, n, flags);
        finish_call(ctx, flags);
    });
}

extern "C" {

int vkrt_intersect_triangles(vkrt_ctx *ctx, const float *tris, const vkrt_ray *rays, uint32_t n,
                             vkrt_tri_result *out, int flags)
{
    return pairwise(ctx, tris, 9, rays, n, out, flags, k_pair_tri);
}

int vkrt_intersect_aabbs(vkrt_ctx *ctx, const float *boxes, const vkrt_ray *rays, uint32_t n, vkrt_result *out,
                         int flags)
{
    return pairwise(ctx, boxes, 6, rays, n, out, flags, k_pair_aabb);
}

int vkrt_intersect_obbs(vkrt_ctx *ctx, const float *obbs, const vkrt_ray *rays, uint32_t n, vkrt_result *out,
                        int flags)
{
    return pairwise(ctx, obbs, 15, rays, n, out, flags, k_pair_obb);
}

int vkrt_intersect_spheres(vkrt_ctx *ctx, const float *spheres, const vkrt_ray *rays, uint32_t n,
                           vkrt_result *out, int flags)
{
    return pairwise(ctx, spheres, 4, rays, n, out, flags, k_pair_sphere);
}

int vkrt_intersect_planes(vkrt_ctx *ctx, const float *planes, const vkrt_ray *rays, uint32_t n, vkrt_result *out,
                          int flags)
{
    return pairwise(ctx, planes, 4, rays, n, out, flags, k_pair_plane);
}

int vkrt_tri_box_overlap(vkrt_ctx *ctx, const float *tris, const float *boxes, uint32_t n, uint32_t *out, int flags)
{
    return guarded(ctx, [&] {
        VKRT_REQUIRE(n == 0 || (tris && boxes && out), "null array argument");
        if(n == 0) return;
        const float *dt = input(ctx, 0, tris, (size_t)n * 9, flags);
        const float *db = input(ctx, 1, boxes, (size_t)n * 6, flags);
        uint32_t *dout = output(ctx, 2, out, n, flags);
        k_pair_tri_box<<<div_up(n, 256), 256, 0, ctx->stream>>>(dt, db, n, dout);
        VKRT_HIP(hipGetLastError());
        finish_output(ctx, 2, out, n, flags);
        finish_call(ctx, flags);
    });
}

int vkrt_tri_tri_overlap(vkrt_ctx *ctx, const float *tris_a, const float *tris_b, uint32_t n, uint32_t *out,
                         int flags)
{
    return guarded(ctx, [&] {
        VKRT_REQUIRE(n == 0 || (tris_a && tris_b && out), "null array argument");
        if(n == 0) return;
        const float *da = input(ctx, 0, tris_a, (size_t)n * 9, flags);
        const float *db = input(ctx, 1, tris_b, (size_t)n * 9, flags);
        uint32_t *dout = output(ctx, 2, out, n, flags);
        k_pair_tri_tri<<<div_up(n, 256), 256, 0, ctx->stream>>>(da, db, n, dout);
        VKRT_HIP(hipGetLastError());
        finish_output(ctx, 2, out, n, flags);
        finish_call(ctx, flags);
    });
}

int vkrt_compute_aabb(vkrt_ctx *ctx, const float *points, uint32_t n, float *out6, int flags)
{
    return guarded(ctx, [&] {
        VKRT_REQUIRE(out6 && (n == 0 || points), "null array argument");
        const float *dp = input(ctx, 0, points, (size_t)n * 3, flags);
        float *dout = output(ctx, 2, out6, 6, flags);
        ctx->scratch[0].reserve(6 * sizeof(uint64_t));
        uint64_t *keys = ctx->scratch[0].as<uint64_t>();
        launch_fill_u64(ctx->stream, keys, 3, ~0ull);
        launch_fill_u64(ctx->stream, keys + 3, 3, 0ull);
        if(n)
        {
            uint32_t blocks = div_up(n, 256);
            if(blocks > 4 * (uint32_t)ctx->cu_count) blocks = 4 * ctx->cu_count;
            k_aabb_reduce<<<blocks, 256, 0, ctx->stream>>>(dp, n, keys);
        }
        k_aabb_finalize<<<1, 64, 0, ctx->stream>>>(dp, keys, dout);
        VKRT_HIP(hipGetLastError());
        finish_output(ctx, 2, out6, 6, flags);
        finish_call(ctx, flags);
    });
}

int vkrt_compute_bounding_sphere(vkrt_ctx *ctx, const float *points, uint32_t n, float *out4, int flags)
{
    return guarded(ctx, [&] {
        VKRT_REQUIRE(out4 && (n == 0 || points), "null array argument");
        float *dout = output(ctx, 2, out4, 4, flags);
        if(n == 0)
        {
            // the reference reads vertices[0] of an empty array; here the sphere is all zeros
            const float zero[4] = {0.f, 0.f, 0.f, 0.f};
            VKRT_HIP(hipMemcpyAsync(dout, zero, sizeof zero, hipMemcpyHostToDevice, ctx->stream));
            VKRT_HIP(hipStreamSynchronize(ctx->stream));
        }
        else
        {
            const float *dp = input(ctx, 0, points, (size_t)n * 3, flags);
            ctx->scratch[0].reserve(6 * sizeof(uint64_t));
            uint64_t *keys = ctx->scratch[0].as<uint64_t>();
            launch_fill_u64(ctx->stream, keys, 3, ~0ull);
            launch_fill_u64(ctx->stream, keys + 3, 3, 0ull);
            uint32_t blocks = div_up(n, 256);
            if(blocks > 4 * (uint32_t)ctx->cu_count) blocks = 4 * ctx->cu_count;
            k_aabb_reduce<<<blocks, 256, 0, ctx->stream>>>(dp, n, keys);
            k_sphere_grow<<<1, SPHERE_BLOCK, 0, ctx->stream>>>(dp, n, keys, dout);
            VKRT_HIP(hipGetLastError());
        }
        finish_output(ctx, 2, out4, 4, flags);
        finish_call(ctx, flags);
    });
}

int vkrt_intersect_brute_closest(vkrt_ctx *ctx, const float *tris, uint32_t n_tri, const vkrt_ray *rays,
                                 uint32_t n_ray, vkrt_hit *out, int flags)
{
    return guarded(ctx, [&] {
        VKRT_REQUIRE((n_tri == 0 || tris) && (n_ray == 0 || (rays && out)), "null array argument");
        if(n_ray == 0) return;
        const float *dt = input(ctx, 0, tris, (size_t)n_tri * 9, flags);
        const vkrt_ray *dr = input(ctx, 1, rays, n_ray, flags);
        vkrt_hit *dh = output(ctx, 2, out, n_ray, flags);
        ctx->scratch[1].reserve((size_t)n_ray * sizeof(uint64_t));
        brute_closest(ctx, dt, n_tri, reinterpret_cast<const float4 *>(dr), n_ray, ctx->scratch[1].as<uint64_t>(),
                      dh);
        VKRT_HIP(hipGetLastError());
        finish_output(ctx, 2, out, n_ray, flags);
        finish_call(ctx, flags);
    });
}

int vkrt_intersect_brute_closest_noalloc(vkrt_ctx *ctx, const float *tris, uint32_t n_tri, const vkrt_ray *rays,
                                         uint32_t n_ray, vkrt_hit *out, int flags)
{
    return guarded(ctx, [&] {
        VKRT_REQUIRE(flags & VKRT_DEVICE_PTRS,
                     "vkrt_intersect_brute_closest_noalloc takes device pointers only (VKRT_DEVICE_PTRS)");
        VKRT_REQUIRE((n_tri == 0 || tris) && (n_ray == 0 || (rays && out)), "null array argument");
        VKRT_REQUIRE(n_tri <= VKRT_NOALLOC_MAX_TRI,
                     "vkrt_intersect_brute_closest_noalloc: n_tri exceeds VKRT_NOALLOC_MAX_TRI (262144)");
        VKRT_REQUIRE(n_ray <= VKRT_NOALLOC_MAX_RAY,
                     "vkrt_intersect_brute_closest_noalloc: n_ray exceeds VKRT_NOALLOC_MAX_RAY (786432)");
        VKRT_REQUIRE(ctx->noalloc_scratch, "no allocation-free scratch on this device");
        if(n_ray == 0) return;
        uint64_t *keys = static_cast<uint64_t *>(ctx->noalloc_scratch);
        // every key brute_closest reads is written first in the same call, by a fill kernel, so nothing left by
        // an earlier call is read
        brute_closest(ctx, tris, n_tri, reinterpret_cast<const float4 *>(rays), n_ray, keys, out);
        VKRT_HIP(hipGetLastError());
        finish_call(ctx, flags);
    });
}

int vkrt_intersect_brute_any(vkrt_ctx *ctx, const float *tris, uint32_t n_tri, const vkrt_ray *rays,
                             uint32_t n_ray, uint8_t *occluded, int flags)
{
    return guarded(ctx, [&] {
        VKRT_REQUIRE((n_tri == 0 || tris) && (n_ray == 0 || (rays && occluded)), "null array argument");
        if(n_ray == 0) return;
        const float *dt = input(ctx, 0, tris, (size_t)n_tri * 9, flags);
        const vkrt_ray *dr = input(ctx, 1, rays, n_ray, flags);
        uint8_t *docc = output(ctx, 2, occluded, n_ray, flags);
        brute_any(ctx, dt, n_tri, reinterpret_cast<const float4 *>(dr), n_ray, docc);
        VKRT_HIP(hipGetLastError());
        finish_output(ctx, 2, occluded, n_ray, flags);
        finish_call(ctx, flags);
    });
}

}// extern "C"
