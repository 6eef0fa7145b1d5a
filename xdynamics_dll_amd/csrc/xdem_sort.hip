// xdem_sort.hip -- stable LSD radix sort of (cell hash, index) pairs and the cell table, for gfx950.
//
// 8-bit digits over tiles of 4,096 pairs, blocks of 1,024 threads. Up to kSmall pairs one block does
// everything in LDS (after a kernel that clears the cell table). Beyond, two kernels a digit:
//   k_hist      per-tile digit counts (LDS atomics) -> hist[tile][digit]; the first digit's launch
//               has further blocks that clear the cell table meanwhile
//   k_scatter   adds up the counts of the earlier tiles and of all tiles itself (no scan kernel
//               between: a block reads the whole table, 1 KB a tile, coalesced and from L2), ranks
//               its pairs among equal digits, reorders the tile in LDS by digit and writes runs of
//               equal digits. That reading grows with the square of the tiles: beyond kTableTiles
//               of them two kernels between, k_chunk_sums and k_chunk_bases, leave a block one row
//               and its own chunk's earlier tiles to read.
// and k_bounds, the first and one-past-last position of every occupied cell. A wave ranks its own 64
// pairs at a time with wave64 ballots against counters of its own, so the block synchronises only
// once for all of them; ranks respect input order, which makes the sort stable.
//
// Bound by latency up to about a million pairs: the kernels of a call take 84 -> 48 us for 120,000
// pairs and 21 key bits and 131 -> 64 us for 1,048,575 (three kernels a digit, one of them a scan by
// one work-group, and separate copies and fills).
#include "xdem_sort.hpp"

namespace xdem {
namespace {

constexpr uint32_t kThreads = 1024;
constexpr uint32_t kWaves = kThreads / 64;
constexpr uint32_t kItems = 4;
constexpr uint32_t kTile = kThreads * kItems;
constexpr uint32_t kSmall = kThreads * 8;   // pairs that one block sorts, 2, 4 or 8 a thread
constexpr uint32_t kChunk = 32;      // tiles whose counts are added up together beyond kTableTiles
// The most tiles whose whole table every block reads: the reorder launcher takes 67 us either way
// for 1,000,000 pairs, 109 against 84 for 2,000,000, 240 against 123 for 4,000,000 and 8,540 against
// 1,004 for 32,000,000 (the kernels of one scan by one work-group 143, 204, 358 and 2,750); 49
// against 56 for 100,000.
constexpr uint32_t kTableTiles = 256;
constexpr uint32_t kNone = 0xffffffffu;

// Both cell tables from entry b * kThreads on, by nb blocks.
__device__ __forceinline__ void clear_cells(uint32_t* cstart, uint32_t* cend, uint32_t ncell, uint32_t b, uint32_t nb)
{
    for (size_t i = (size_t)b * kThreads + threadIdx.x; i < ncell; i += (size_t)nb * kThreads) {
        cstart[i] = kNone;
        cend[i] = 0u;
    }
}

__global__ __launch_bounds__(kThreads) void k_clear(uint32_t* cstart, uint32_t* cend, uint32_t ncell)
{
    clear_cells(cstart, cend, ncell, blockIdx.x, gridDim.x);
}

__global__ __launch_bounds__(kThreads) void k_hist(const uint32_t* __restrict__ keys, uint32_t n, uint32_t shift,
                                                   uint32_t* __restrict__ hist, uint32_t ntiles, uint32_t* cstart,
                                                   uint32_t* cend, uint32_t ncell)
{
    if (blockIdx.x >= ntiles) {
        clear_cells(cstart, cend, ncell, blockIdx.x - ntiles, gridDim.x - ntiles);
        return;
    }
    __shared__ uint32_t cnt[256];
    if (threadIdx.x < 256u) cnt[threadIdx.x] = 0u;
    __syncthreads();
    const uint32_t base = blockIdx.x * kTile + threadIdx.x;
#pragma unroll
    for (uint32_t s = 0; s < kItems; s++) {
        const uint32_t idx = base + s * kThreads;
        if (idx < n) atomicAdd(&cnt[(keys[idx] >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 256u) hist[blockIdx.x * 256u + threadIdx.x] = cnt[threadIdx.x];
}

// Exclusive scan of one value per thread over threads 0..255 (4 waves); every thread of the block
// calls it, threads past 255 get nothing of use.
__device__ __forceinline__ uint32_t scan256(uint32_t v, uint32_t* wsum)
{
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (uint32_t off = 1; off < 64u; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63u && w < 4u) wsum[w] = x;
    __syncthreads();
    uint32_t pre = 0;
    for (uint32_t q = 0; q < 4u && q < w; q++) pre += wsum[q];
    __syncthreads();
    return pre + x - v;
}

// The tile's ranking. Item s of a thread is pair wave * 64 ITEMS + s * 64 + lane of the tile; items
// past the tile's end come last and count as digit 255, after every pair. place[s]: the item's
// position in the tile sorted by digit; start[d]: the first position of digit d.
template <uint32_t ITEMS>
__device__ __forceinline__ void rank_tile(const uint32_t (&digit)[ITEMS], uint32_t (&place)[ITEMS], uint32_t (*cnt)[256],
                                          uint32_t* start, uint32_t* wsum)
{
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint64_t lt = lane == 0u ? 0ull : (~0ull >> (64u - lane));
    for (uint32_t q = lane; q < 256u; q += 64u) cnt[w][q] = 0u;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (uint32_t s = 0; s < ITEMS; s++) {
        const uint32_t d = digit[s];
        uint64_t peers = ~0ull;   // lanes of this wave holding the same digit
#pragma unroll
        for (uint32_t b = 0; b < 8u; b++) {
            const bool bit = (d >> b) & 1u;
            const uint64_t m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        const uint32_t before = (uint32_t)__popcll(peers & lt);
        const uint32_t c = cnt[w][d];
        place[s] = c + before;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (before == 0u) cnt[w][d] = c + (uint32_t)__popcll(peers);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    uint32_t total = 0;
    if (tid < 256u) {
#pragma unroll
        for (uint32_t q = 0; q < kWaves; q++) {
            const uint32_t c = cnt[q][tid];
            cnt[q][tid] = total;
            total += c;
        }
    }
    const uint32_t first = scan256(total, wsum);
    if (tid < 256u) start[tid] = first;
    __syncthreads();
#pragma unroll
    for (uint32_t s = 0; s < ITEMS; s++) place[s] += start[digit[s]] + cnt[w][digit[s]];
}

// The counts of kChunk tiles added up, a chunk a block: a quarter of the block adds up a quarter of
// the chunk's tiles.
__device__ __forceinline__ uint32_t chunk_part(const uint32_t* __restrict__ hist, uint32_t chunk, uint32_t end)
{
    const uint32_t d = threadIdx.x & 255u, t0 = chunk * kChunk + (threadIdx.x >> 8) * (kChunk / 4u);
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t u = 0; u < kChunk / 4u; u++) sum += t0 + u < end ? hist[(t0 + u) * 256u + d] : 0u;
    return sum;
}

__global__ __launch_bounds__(kThreads) void k_chunk_sums(const uint32_t* __restrict__ hist, uint32_t ntiles,
                                                         uint32_t* __restrict__ sums)
{
    __shared__ uint32_t s_part[kThreads];
    const uint32_t tid = threadIdx.x;
    s_part[tid] = chunk_part(hist, blockIdx.x, ntiles);
    __syncthreads();
    if (tid < 256u)
        sums[blockIdx.x * 256u + tid] = s_part[tid] + s_part[256u + tid] + s_part[512u + tid] + s_part[768u + tid];
}

// The chunks' sums to the first position of each digit of each chunk, in place, by one block: a
// quarter of it takes a quarter of the chunks.
__global__ __launch_bounds__(kThreads) void k_chunk_bases(uint32_t* __restrict__ sums, uint32_t nchunk)
{
    __shared__ uint32_t s_part[kThreads], s_wsum[4], s_first[256];
    const uint32_t tid = threadIdx.x, d = tid & 255u, g = tid >> 8, per = (nchunk + 3u) / 4u;
    const uint32_t lo = min(nchunk, g * per), hi = min(nchunk, lo + per);
    uint32_t part = 0;
    for (uint32_t t = lo; t < hi; t += 8u) {
#pragma unroll
        for (uint32_t u = 0; u < 8u; u++) part += t + u < hi ? sums[(t + u) * 256u + d] : 0u;
    }
    s_part[tid] = part;
    __syncthreads();
    const uint32_t all = s_part[d] + s_part[256u + d] + s_part[512u + d] + s_part[768u + d];
    const uint32_t first = scan256(all, s_wsum);
    if (tid < 256u) s_first[tid] = first;
    __syncthreads();
    uint32_t run = s_first[d];
    for (uint32_t q = 0; q < g; q++) run += s_part[q * 256u + d];
    for (uint32_t t = lo; t < hi; t += 8u) {
        uint32_t c[8];
#pragma unroll
        for (uint32_t u = 0; u < 8u; u++) c[u] = t + u < hi ? sums[(t + u) * 256u + d] : 0u;
#pragma unroll
        for (uint32_t u = 0; u < 8u; u++) {
            if (t + u < hi) sums[(t + u) * 256u + d] = run;
            run += c[u];
        }
    }
}

// BASES: the counts of whole chunks come added up (k_chunk_bases). As a branch of one kernel the
// other reading's sorts took 1 to 2 percent longer.
template <bool BASES>
__global__ __launch_bounds__(kThreads) void k_scatter(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                      uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
                                                      uint32_t* __restrict__ vout2, uint32_t n, uint32_t shift,
                                                      const uint32_t* __restrict__ hist, uint32_t ntiles,
                                                      const uint32_t* __restrict__ bases)
{
    __shared__ uint32_t s_keys[kTile], s_vals[kTile];
    __shared__ uint32_t s_cnt[kWaves][256];
    __shared__ uint32_t s_start[256], s_gbase[256], s_wsum[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint32_t base = blockIdx.x * kTile;
    uint32_t key[kItems], val[kItems], digit[kItems], place[kItems];
#pragma unroll
    for (uint32_t s = 0; s < kItems; s++) {
        const uint32_t idx = base + (w * kItems + s) * 64u + lane;
        key[s] = idx < n ? kin[idx] : 0u;
        val[s] = idx < n ? vin[idx] : 0u;
        digit[s] = idx < n ? (key[s] >> shift) & 255u : 255u;
    }
    // digit d of this tile goes after all smaller digits and after digit d of the earlier tiles:
    // a quarter of the block adds up a quarter of the tiles' counts
    if (BASES) {
        const uint32_t chunk = blockIdx.x / kChunk;
        s_keys[tid] = chunk_part(hist, chunk, blockIdx.x);
        __syncthreads();
        if (tid < 256u)
            s_gbase[tid] = bases[chunk * 256u + tid] + s_keys[tid] + s_keys[256u + tid] + s_keys[512u + tid] + s_keys[768u + tid];
    } else {
        const uint32_t d = tid & 255u, g = tid >> 8, per = (ntiles + 3u) / 4u;
        const uint32_t lo = min(ntiles, g * per), hi = min(ntiles, lo + per);
        uint32_t pre = 0, all = 0, t = lo;
        for (; t + 8u <= hi; t += 8u) {
            uint32_t c[8];
#pragma unroll
            for (uint32_t u = 0; u < 8u; u++) c[u] = hist[(t + u) * 256u + d];
#pragma unroll
            for (uint32_t u = 0; u < 8u; u++) {
                all += c[u];
                pre += t + u < blockIdx.x ? c[u] : 0u;
            }
        }
        for (; t < hi; t++) {
            const uint32_t c = hist[t * 256u + d];
            all += c;
            pre += t < blockIdx.x ? c : 0u;
        }
        s_keys[tid] = pre;
        s_vals[tid] = all;
        __syncthreads();
        pre = all = 0;
        if (tid < 256u)
#pragma unroll
            for (uint32_t q = 0; q < 4u; q++) {
                pre += s_keys[q * 256u + tid];
                all += s_vals[q * 256u + tid];
            }
        const uint32_t first = scan256(all, s_wsum);
        if (tid < 256u) s_gbase[tid] = first + pre;
    }
    rank_tile<kItems>(digit, place, s_cnt, s_start, s_wsum);
#pragma unroll
    for (uint32_t s = 0; s < kItems; s++) {
        s_keys[place[s]] = key[s];
        s_vals[place[s]] = val[s];
    }
    __syncthreads();
    const uint32_t valid = min(n - base, kTile);
#pragma unroll
    for (uint32_t s = 0; s < kItems; s++) {
        const uint32_t p = s * kThreads + tid;
        if (p < valid) {
            const uint32_t k = s_keys[p], v = s_vals[p], d = (k >> shift) & 255u;
            const uint32_t o = s_gbase[d] + (p - s_start[d]);
            kout[o] = k;
            vout[o] = v;
            if (vout2) vout2[o] = v;
        }
    }
}

// Cell bounds (impl:317-360) of n sorted hashes; with kcopy, also the copies of a single digit's sort
// (whose source is the caller's arrays).
__global__ __launch_bounds__(256) void k_bounds(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals,
                                                uint32_t* kcopy, uint32_t* vcopy, uint32_t* sorted_index,
                                                uint32_t* cstart, uint32_t* cend, uint32_t n)
{
    const uint32_t id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= n) return;
    const uint32_t h = keys[id], prev = id ? keys[id - 1u] : 0u;
    if (kcopy) {
        const uint32_t v = vals[id];
        kcopy[id] = h;
        vcopy[id] = v;
        sorted_index[id] = v;
    }
    if (id == 0u || h != prev) {
        cstart[h] = id;
        if (id) cend[prev] = id;
    }
    if (id == n - 1u) cend[h] = id + 1u;
}

// All digits of up to kThreads * ITEMS pairs, the copies and the cell bounds, by one block.
template <uint32_t ITEMS>
__global__ __launch_bounds__(kThreads) void k_sort_small(uint32_t* hash, uint32_t* index, uint32_t* sorted_index,
                                                         uint32_t* cstart, uint32_t* cend, uint32_t n, uint32_t npass)
{
    __shared__ uint32_t s_keys[kThreads * ITEMS], s_vals[kThreads * ITEMS];
    __shared__ uint32_t s_cnt[kWaves][256];
    __shared__ uint32_t s_start[256], s_wsum[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    uint32_t key[ITEMS], val[ITEMS], digit[ITEMS], place[ITEMS];
#pragma unroll
    for (uint32_t s = 0; s < ITEMS; s++) {
        const uint32_t idx = (w * ITEMS + s) * 64u + lane;
        key[s] = idx < n ? hash[idx] : 0u;
        val[s] = idx < n ? index[idx] : 0u;
    }
    for (uint32_t p = 0; p < npass; p++) {
#pragma unroll
        for (uint32_t s = 0; s < ITEMS; s++) {
            const uint32_t idx = (w * ITEMS + s) * 64u + lane;
            if (p) {
                key[s] = s_keys[idx];
                val[s] = s_vals[idx];
            }
            digit[s] = idx < n ? (key[s] >> (8u * p)) & 255u : 255u;
        }
        __syncthreads();
        rank_tile<ITEMS>(digit, place, s_cnt, s_start, s_wsum);
#pragma unroll
        for (uint32_t s = 0; s < ITEMS; s++) {
            s_keys[place[s]] = key[s];
            s_vals[place[s]] = val[s];
        }
        __syncthreads();
    }
    for (uint32_t p = tid; p < n; p += kThreads) {
        const uint32_t h = s_keys[p], v = s_vals[p];
        hash[p] = h;
        index[p] = v;
        sorted_index[p] = v;
        const uint32_t prev = p ? s_keys[p - 1u] : 0u;
        if (p == 0u || h != prev) {
            cstart[h] = p;
            if (p) cend[prev] = p;
        }
        if (p == n - 1u) cend[h] = p + 1u;
    }
}

}  // namespace

size_t cell_sort_scratch_bytes(uint32_t n)
{
    const size_t ntiles = (n + kTile - 1) / kTile;
    return sizeof(uint32_t) * 256 * (ntiles ? ntiles : 1);
}

hipError_t cell_sort(uint32_t* hash, uint32_t* index, uint32_t* sorted_index, uint32_t* cstart, uint32_t* cend, uint32_t n,
                     uint32_t ncell, uint32_t* const buf[4], void* scratch, hipStream_t stream)
{
    uint32_t bits = 1;
    while (bits < 32u && (1ull << bits) < (unsigned long long)ncell) bits++;
    const uint32_t npass = (bits + 7u) / 8u;
    const uint32_t clear_blocks = std::min(512u, (ncell - 1u) / kThreads + 1u);   // ncell > 0
    if (n <= kSmall) {
        hipLaunchKernelGGL(k_clear, dim3(clear_blocks), dim3(kThreads), 0, stream, cstart, cend, ncell);
        if (n > 4u * kThreads)
            hipLaunchKernelGGL(k_sort_small<8>, dim3(1), dim3(kThreads), 0, stream, hash, index, sorted_index, cstart, cend, n, npass);
        else if (n > 2u * kThreads)
            hipLaunchKernelGGL(k_sort_small<4>, dim3(1), dim3(kThreads), 0, stream, hash, index, sorted_index, cstart, cend, n, npass);
        else if (n)
            hipLaunchKernelGGL(k_sort_small<2>, dim3(1), dim3(kThreads), 0, stream, hash, index, sorted_index, cstart, cend, n, npass);
        return hipGetLastError();
    }
    const uint32_t ntiles = (n + kTile - 1u) / kTile;
    uint32_t* hist = static_cast<uint32_t*>(scratch);
    const uint32_t *ksrc = hash, *vsrc = index;
    for (uint32_t p = 0; p < npass; p++) {
        // the last digit goes to the caller's arrays, unless they are its source
        const bool out = p + 1u == npass && npass > 1u;
        uint32_t* kdst = out ? hash : buf[2u * (p & 1u)];
        uint32_t* vdst = out ? index : buf[2u * (p & 1u) + 1u];
        const uint32_t extra = p == 0u ? clear_blocks : 0u;
        hipLaunchKernelGGL(k_hist, dim3(ntiles + extra), dim3(kThreads), 0, stream, ksrc, n, 8u * p, hist, ntiles, cstart,
                           cend, ncell);
        uint32_t* vcopy = out ? sorted_index : nullptr;
        if (ntiles <= kTableTiles) {
            hipLaunchKernelGGL(k_scatter<false>, dim3(ntiles), dim3(kThreads), 0, stream, ksrc, vsrc, kdst, vdst, vcopy, n,
                               8u * p, hist, ntiles, (const uint32_t*)nullptr);
        } else {
            // a row of 256 for each chunk, in an array that this digit neither reads nor writes
            uint32_t* bases = out ? buf[2u * (p & 1u)] : (p ? sorted_index : buf[2]);
            const uint32_t nchunk = (ntiles + kChunk - 1u) / kChunk;
            hipLaunchKernelGGL(k_chunk_sums, dim3(nchunk), dim3(kThreads), 0, stream, hist, ntiles, bases);
            hipLaunchKernelGGL(k_chunk_bases, dim3(1), dim3(kThreads), 0, stream, bases, nchunk);
            hipLaunchKernelGGL(k_scatter<true>, dim3(ntiles), dim3(kThreads), 0, stream, ksrc, vsrc, kdst, vdst, vcopy, n,
                               8u * p, hist, ntiles, (const uint32_t*)bases);
        }
        ksrc = kdst;
        vsrc = vdst;
    }
    const bool copy = npass == 1u;
    hipLaunchKernelGGL(k_bounds, dim3((n + 255u) / 256u), dim3(256), 0, stream, ksrc, vsrc, copy ? hash : nullptr,
                       copy ? index : nullptr, sorted_index, cstart, cend, n);
    return hipGetLastError();
}

}  // namespace xdem
