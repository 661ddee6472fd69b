// radix_sort.hip - stable LSD radix sort of (uint32 key, uint32 value) pairs, 8-bit digits.
//
// One pass per digit, three kernels per pass:
//   k_rs_hist    per-tile 256-bin histogram in LDS, stored digit-major (hist[d * tiles + tile])
//   k_rs_scan    exclusive scan of each digit's row, one workgroup per digit, and the digit's total
//   k_rs_scatter stable scatter: within a round of 256 items a wave64 finds the lanes holding the same
//                digit with 8 ballots (match-any), ranks by popcount below its lane, and waves are
//                ordered through per-wave digit counts in LDS; the digits' bases are the scan of the 256 totals,
//                which every workgroup makes for itself
// Tiles are 256 threads x ROUNDS rounds; item k of thread t is tile_base + 256 k + t, so loads are coalesced
// and the in-tile order (round, thread) is the input order, which keeps the sort stable.
#include "context.hpp"
#include "radix_sort.hpp"

namespace vkrt
{

constexpr uint32_t RS_THREADS = 256, RS_BINS = 256;
// rounds per tile: what a round costs is its five barriers, one after the other, so a sort too small to give each
// CU a tile of eight rounds takes tiles of two (20k keys: 11.1 us a scatter at eight rounds, 5.0 at two)
constexpr uint32_t RS_ROUNDS = 8, RS_ROUNDS_SMALL = 2, RS_SMALL = 256 * RS_ROUNDS * RS_THREADS;

static uint32_t rs_tiles(uint32_t n) { return div_up(n, RS_THREADS * (n < RS_SMALL ? RS_ROUNDS_SMALL : RS_ROUNDS)); }

template<uint32_t ROUNDS>
__global__ void __launch_bounds__(RS_THREADS) k_rs_hist(const uint32_t *__restrict__ keys, uint32_t n, uint32_t shift,
                                                        uint32_t tiles, uint32_t *__restrict__ hist)
{
    __shared__ uint32_t h[RS_BINS];
    h[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * (ROUNDS * RS_THREADS);
    for(uint32_t k = 0; k < ROUNDS; ++k)
    {
        uint32_t i = base + k * RS_THREADS + threadIdx.x;
        if(i < n) atomicAdd(&h[(keys[i] >> shift) & 0xffu], 1u);
    }
    __syncthreads();
    hist[threadIdx.x * tiles + blockIdx.x] = h[threadIdx.x];
}

//! exclusive scan of x over the workgroup of 256 (wsum: 4 words of LDS); `total` is the whole sum
__device__ __forceinline__ uint32_t block_scan(uint32_t x, uint32_t *wsum, uint32_t &total)
{
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t s = x;
    for(int off = 1; off < 64; off <<= 1)
    {
        const uint32_t y = __shfl_up(s, off);
        if(lane >= (uint32_t)off) s += y;
    }
    if(lane == 63) wsum[wave] = s;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
    for(uint32_t w = 0; w < RS_THREADS / 64; ++w)
    {
        before += w < wave ? wsum[w] : 0u;
        total += wsum[w];
    }
    return before + s - x;
}

//! digit blockIdx.x's row of tile counts, scanned in place, and its total. Rows lie one after the other, so the 256
//! of them fill the chip (one workgroup over the whole table took 210 us a pass at 1.8M keys, 839 us of a build;
//! the rows take 4.8 us a pass)
__global__ void __launch_bounds__(RS_THREADS) k_rs_scan(uint32_t *__restrict__ hist, uint32_t tiles,
                                                        uint32_t *__restrict__ totals)
{
    __shared__ uint32_t wsum[2][RS_THREADS / 64];
    uint32_t *row = hist + (size_t)blockIdx.x * tiles;
    uint32_t carry = 0, turn = 0;
    for(uint32_t base = 0; base < tiles; base += RS_THREADS, turn ^= 1u)
    {
        const uint32_t i = base + threadIdx.x;
        uint32_t total;
        // (the sums alternate between two sets, so one barrier a turn is enough)
        const uint32_t before = block_scan(i < tiles ? row[i] : 0u, wsum[turn], total);
        if(i < tiles) row[i] = carry + before;
        carry += total;
    }
    if(threadIdx.x == 0) totals[blockIdx.x] = carry;
}

template<uint32_t ROUNDS>
__global__ void __launch_bounds__(RS_THREADS) k_rs_scatter(const uint32_t *__restrict__ keys_in,
                                                           const uint32_t *__restrict__ vals_in, uint32_t n,
                                                           uint32_t shift, uint32_t tiles,
                                                           const uint32_t *__restrict__ offsets,
                                                           const uint32_t *__restrict__ totals,
                                                           uint32_t *__restrict__ keys_out,
                                                           uint32_t *__restrict__ vals_out)
{
    __shared__ uint32_t gbase[RS_BINS];
    __shared__ uint32_t wcount[RS_THREADS / 64][RS_BINS];
    __shared__ uint32_t wsum[RS_THREADS / 64];
    const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
    uint32_t all;
    const uint32_t digit_base = block_scan(totals[t], wsum, all);
    gbase[t] = digit_base + offsets[t * tiles + blockIdx.x];
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const uint32_t base = blockIdx.x * (ROUNDS * RS_THREADS);
    for(uint32_t k = 0; k < ROUNDS; ++k)
    {
        for(uint32_t w = 0; w < RS_THREADS / 64; ++w) wcount[w][t] = 0;
        __syncthreads();
        const uint32_t i = base + k * RS_THREADS + t;
        const bool valid = i < n;
        uint32_t key = 0, val = 0, d = 0;
        if(valid)
        {
            key = keys_in[i];
            val = vals_in[i];
            d = (key >> shift) & 0xffu;
        }
        uint64_t peers = __ballot(valid);
        for(int b = 0; b < 8; ++b)
        {
            const bool bit = (d >> b) & 1u;
            const uint64_t ones = __ballot(valid && bit);
            peers &= bit ? ones : ~ones;
        }
        const uint32_t rank = __popcll(peers & lt_mask);
        if(valid && rank == 0) wcount[wave][d] = __popcll(peers);
        __syncthreads();
        if(valid)
        {
            uint32_t off = gbase[d] + rank;
            for(uint32_t w = 0; w < wave; ++w) off += wcount[w][d];
            keys_out[off] = key;
            vals_out[off] = val;
        }
        __syncthreads();
        uint32_t add = 0;
        for(uint32_t w = 0; w < RS_THREADS / 64; ++w) add += wcount[w][t];
        gbase[t] += add;
        __syncthreads();
    }
}

size_t radix_sort_temp_bytes(uint32_t n)
{
    return ((size_t)rs_tiles(n) + 1) * RS_BINS * sizeof(uint32_t) + 2 * (size_t)n * sizeof(uint32_t) + 256;
}

void radix_sort_pairs(hipStream_t s, uint32_t *keys, uint32_t *vals, uint32_t n, uint32_t key_bits, void *temp)
{
    if(n <= 1) return;
    const uint32_t tiles = rs_tiles(n);
    uint32_t *totals = static_cast<uint32_t *>(temp), *hist = totals + RS_BINS;
    uint32_t *k_alt = hist + (size_t)tiles * RS_BINS;
    uint32_t *v_alt = k_alt + n;
    uint32_t *kin = keys, *vin = vals, *kout = k_alt, *vout = v_alt;
    const uint32_t passes = div_up(key_bits, 8);
    for(uint32_t p = 0; p < passes; ++p)
    {
        const uint32_t shift = 8 * p;
        if(n < RS_SMALL) k_rs_hist<RS_ROUNDS_SMALL><<<tiles, RS_THREADS, 0, s>>>(kin, n, shift, tiles, hist);
        else k_rs_hist<RS_ROUNDS><<<tiles, RS_THREADS, 0, s>>>(kin, n, shift, tiles, hist);
        k_rs_scan<<<RS_BINS, RS_THREADS, 0, s>>>(hist, tiles, totals);
        if(n < RS_SMALL)
            k_rs_scatter<RS_ROUNDS_SMALL><<<tiles, RS_THREADS, 0, s>>>(kin, vin, n, shift, tiles, hist, totals, kout, vout);
        else k_rs_scatter<RS_ROUNDS><<<tiles, RS_THREADS, 0, s>>>(kin, vin, n, shift, tiles, hist, totals, kout, vout);
        std::swap(kin, kout);
        std::swap(vin, vout);
    }
    if(kin != keys)
    {
        VKRT_HIP(hipMemcpyAsync(keys, kin, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, s));
        VKRT_HIP(hipMemcpyAsync(vals, vin, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, s));
    }
}

}// namespace vkrt
