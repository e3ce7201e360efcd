// k_readback.hip — a world's state as transfer objects, built on the device.
//
// ALIEN packs its transfer objects on the device as well (source/EngineGpuKernels/DataAccessKernels.cu),
// with an atomic cursor.  Here the records come out in ascending id order (ties by index), so the
// cells' ids are sorted once per set (a cell keeps its id and slot for the set's life) and the
// particles' ids on every read-back, by a stable radix sort of 8-bit digits that skips the digits in
// which no two keys differ.  The pack kernels gather a record per thread, stage 256 of them in LDS
// and store them to pinned host memory as one contiguous run.
//
// Bound: the link to the host.  Stores of 8 bytes per lane to pinned memory reached 55 GB/s on an
// MI355X, a DMA copy of the same bytes 57 GB/s; a kernel needs no device staging buffer and no
// second launch, which is what counts for small worlds (65 KB: 15 us, launch and wait included).
// get_data with this against one pageable copy per array and a conversion on the host: 1,200 cells
// 490 -> 63 us, 80,021 cells 6.6 -> 0.57 ms, 1,000,000 cells with 136,000 particles 186 -> 4.0 ms,
// 4,000,000 cells 775 -> 13.7 ms (544 MB: 40 GB/s).
#include "../../include/alien_hip.h"
#include "kernels_common.hpp"
#include "readback.hpp"

namespace alien {

constexpr int kPackThreads = 256;
constexpr int kCellWords = int(sizeof(alien_cell_to) / 4);
constexpr int kPartWords = int(sizeof(alien_particle_to) / 4);
static_assert(kCellWords == 34 && offsetof(alien_cell_to, pos) == 80 && offsetof(alien_cell_to, color) == 104 &&
                  offsetof(alien_cell_to, age) == 108 && offsetof(alien_cell_to, livingState) == 112 &&
                  offsetof(alien_cell_to, creatureId) == 116 && offsetof(alien_cell_to, activationTime) == 128,
              "the pack kernel writes the record word by word");
static_assert(kPartWords == 8 && offsetof(alien_particle_to, energy) == 8 && offsetof(alien_particle_to, color) == 28,
              "the pack kernel writes the record word by word");

// ---- stable radix sort -----------------------------------------------------------------------------
// One pass per digit: per-tile digit counts, an exclusive scan of each digit's row of tile counts, and
// the scatter, which ranks a tile's keys in order (256 at a time: a wave finds the lanes with its
// digit by eight ballots).
constexpr int kSortThreads = 256;
constexpr int kSortRounds = kSortTile / kSortThreads;

__global__ void __launch_bounds__(kSortThreads) k_sort_count(const unsigned long long* keys, int n, int shift,
                                                             uint32_t* counts, int tiles) {
    __shared__ uint32_t h[256];
    const int tid = int(threadIdx.x);
    h[tid] = 0u;
    __syncthreads();
    const int first = int(blockIdx.x) * kSortTile;
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const int k = first + r * kSortThreads + tid;
        if (k < n) atomicAdd(&h[uint32_t(keys[k] >> shift) & 255u], 1u);
    }
    __syncthreads();
    counts[size_t(tid) * tiles + blockIdx.x] = h[tid];
}

// row d of the counts: exclusive scan over the tiles, total behind the rows
__global__ void __launch_bounds__(kSortThreads) k_sort_rows(uint32_t* counts, int tiles) {
    uint32_t* row = counts + size_t(blockIdx.x) * tiles;
    uint32_t sum = 0u;
    for (int t0 = 0; t0 < tiles; t0 += kSortThreads) {
        const int t = t0 + int(threadIdx.x);
        const uint32_t v = t < tiles ? row[t] : 0u;
        uint32_t total;
        const uint32_t off = block_exclusive_scan(v, total);
        if (t < tiles) row[t] = sum + off;
        sum += total;
    }
    if (threadIdx.x == 0) counts[size_t(256) * tiles + blockIdx.x] = sum;
}

__global__ void __launch_bounds__(kSortThreads) k_sort_scatter(const unsigned long long* keys, const int* vals, int n,
                                                               int shift, const uint32_t* counts, int tiles,
                                                               unsigned long long* keysOut, int* valsOut) {
    constexpr int kWaves = kSortThreads / 64;
    __shared__ uint32_t base[256];
    __shared__ uint32_t cnt[kWaves][256];
    const int tid = int(threadIdx.x), lane = tid & 63, wave = tid >> 6;
    uint32_t total;
    const uint32_t before = block_exclusive_scan(counts[size_t(256) * tiles + tid], total);
    base[tid] = before + counts[size_t(tid) * tiles + blockIdx.x];
#pragma unroll
    for (int v = 0; v < kWaves; ++v) cnt[v][tid] = 0u;
    __syncthreads();
    const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const int first = int(blockIdx.x) * kSortTile;
    for (int r = 0; r < kSortRounds; ++r) {
        if (first + r * kSortThreads >= n) break;  // (the same for the whole workgroup)
        const int k = first + r * kSortThreads + tid;
        const bool on = k < n;
        const unsigned long long key = on ? keys[k] : 0ull;
        const uint32_t d = uint32_t(key >> shift) & 255u;
        unsigned long long same = __ballot(on);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const unsigned long long set = __ballot((d >> b) & 1u);
            same &= (d >> b) & 1u ? set : ~set;
        }
        const int rank = __builtin_popcountll(same & below);
        if (on && rank == 0) cnt[wave][d] = uint32_t(__builtin_popcountll(same));
        __syncthreads();
        if (on) {
            uint32_t at = base[d] + uint32_t(rank);
            for (int v = 0; v < wave; ++v) at += cnt[v][d];
            keysOut[at] = key;
            valsOut[at] = vals[k];
        }
        __syncthreads();
        uint32_t sum = 0u;
#pragma unroll
        for (int v = 0; v < kWaves; ++v) {
            sum += cnt[v][tid];
            cnt[v][tid] = 0u;
        }
        base[tid] += sum;
        __syncthreads();
    }
}

// OR of the keys' differences from a reference key: the digits worth a pass
__device__ __forceinline__ void merge_differing(unsigned long long x, unsigned long long* differing) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x |= __shfl_xor(x, o, 64);
    if ((threadIdx.x & 63) == 0 && x) atomicOr(differing, x);
}

// ---- cells -----------------------------------------------------------------------------------------
// keys of the world's cells: by slot, or (slotOf given) by index
__global__ void __launch_bounds__(kPackThreads) k_cell_keys(const unsigned long long* cid, const int* slotOf, int n,
                                                            unsigned long long* keys, int* vals,
                                                            unsigned long long* differing) {
    const int k = int(blockIdx.x) * kPackThreads + int(threadIdx.x);
    unsigned long long x = 0ull;
    if (k < n) {
        const unsigned long long key = cid[slotOf ? slotOf[k] : k];
        keys[k] = key;
        vals[k] = k;
        x = key ^ cid[0];
    }
    merge_differing(x, differing);
}

// rank of every slot (or index) in the sorted order; flags equal neighbours
__global__ void __launch_bounds__(kPackThreads) k_cell_ranks(const unsigned long long* keys, const int* vals, int n,
                                                             int* rankOf, unsigned long long* equal) {
    const int r = int(blockIdx.x) * kPackThreads + int(threadIdx.x);
    if (r >= n) return;
    rankOf[vals[r]] = r;
    if (equal && r > 0 && keys[r] == keys[r - 1]) atomicOr(equal, 1ull);
}

// this read-back's order from the slots' ranks: index at every rank and rank of every index
__global__ void __launch_bounds__(kPackThreads) k_cell_order(const int* slotOf, const int* rankOfSlot, int n, int* order,
                                                             int* rankOf) {
    const int i = int(blockIdx.x) * kPackThreads + int(threadIdx.x);
    if (i >= n) return;
    const int r = rankOfSlot[slotOf[i]];
    order[r] = i;
    rankOf[i] = r;
}

// records first .. first + count - 1 of the order
__global__ void __launch_bounds__(kPackThreads) k_pack_cells(PackCells a, int first, int count, uint2* out) {
    __shared__ __align__(16) uint32_t rec[kPackThreads * kCellWords];
    const int k0 = int(blockIdx.x) * kPackThreads;
    const int cnt = min(kPackThreads, count - k0);
    const int tid = int(threadIdx.x);
    if (tid < cnt) {
        const int i = a.order[first + k0 + tid];
        const int sl = a.slot[i];
        const uint32_t f = a.flags[i];
        const int nc = flags_num_conn(f);
        const bool bar = flags_barrier(f);
        uint32_t* r = rec + tid * kCellWords;
        const unsigned long long id = a.cid[sl];
        r[0] = uint32_t(id);
        r[1] = uint32_t(id >> 32);
        uint32_t t[kMaxBonds], d[kMaxBonds], g[kMaxBonds];
#pragma unroll
        for (int b = 0; b < kMaxBonds; ++b) {
            t[b] = b < nc ? uint32_t(a.btgt[size_t(b) * a.plane + i]) : 0u;
            d[b] = b < nc ? __float_as_uint(a.brest[size_t(b) * a.plane + i]) : 0u;
            g[b] = b < nc ? __float_as_uint(a.bang[size_t(b) * a.plane + i]) : 0u;
        }
#pragma unroll
        for (int b = 0; b < kMaxBonds; ++b) {
            r[2 + 3 * b] = b < nc ? uint32_t(a.rankOf[t[b]]) : 0u;
            r[3 + 3 * b] = d[b];
            r[4 + 3 * b] = g[b];
        }
        const float2 p = a.pos[i], v = a.vel[i];
        r[20] = __float_as_uint(p.x);
        r[21] = __float_as_uint(p.y);
        r[22] = __float_as_uint(v.x);
        r[23] = __float_as_uint(v.y);
        r[24] = __float_as_uint(a.energy[sl]);
        r[25] = __float_as_uint(a.stiff[sl]);
        r[26] = uint32_t(flags_color(f)) | uint32_t(flags_max_conn(f)) << 8 | uint32_t(nc) << 16 | (bar ? 1u << 24 : 0u);
        // a non-barrier cell ages by one per step; a barrier cell is Ready after any step
        r[27] = a.ageBase[sl] + (bar ? 0u : a.steps);
        const uint32_t living = a.living && !(bar && a.stepped) ? uint32_t(a.living[sl]) : 0u;
        CellExtra x{};
        if (a.extra) x = a.extra[sl];
        r[28] = living | uint32_t(x.cellFunction) << 8 | uint32_t(x.ancestorMutationId) << 16 | uint32_t(x.selected) << 24;
        r[29] = a.creature[sl];
        r[30] = x.mutationId;
        r[31] = x.genomeComplexity;
        r[32] = a.activation ? a.activation[sl] : 0u;
        r[33] = 0u;
    }
    __syncthreads();
    const uint2* src = reinterpret_cast<const uint2*>(rec);
    uint2* dst = out + size_t(k0) * (kCellWords / 2);
    for (int q = tid; q < cnt * (kCellWords / 2); q += kPackThreads) dst[q] = src[q];
}

// ---- particles -------------------------------------------------------------------------------------
// Entries of a world's particles: 0 .. np-1 its live range (particles killed in the last step are still
// in it, marked), then with splitting the np records of halves that wait for the next map.
__device__ __forceinline__ bool entry_lives(const PackParticles& a, int e) {
    if (e < a.np) return (a.pflags[e] & kParticleDead) == 0;
    return e < a.entries && (a.halves[e - a.np].color & kStagedPending) != 0u;
}

__global__ void __launch_bounds__(kPackThreads) k_part_count(PackParticles a, uint32_t* tileCount) {
    const int first = int(blockIdx.x) * kPartTile;
    uint32_t n = 0;
#pragma unroll
    for (int r = 0; r < kPartTile / kPackThreads; ++r) n += entry_lives(a, first + r * kPackThreads + int(threadIdx.x)) ? 1u : 0u;
    uint32_t total;
    block_exclusive_scan(n, total);
    if (threadIdx.x == 0) tileCount[blockIdx.x] = total;
}

// exclusive scan of the tile counts by one workgroup; result[0] the total, result[1] cleared for the
// keys' differences
__global__ void __launch_bounds__(1024) k_part_offsets(uint32_t* tileCount, int tiles, unsigned long long* result) {
    uint32_t sum = 0u;
    for (int t0 = 0; t0 < tiles; t0 += 1024) {
        const int t = t0 + int(threadIdx.x);
        const uint32_t v = t < tiles ? tileCount[t] : 0u;
        uint32_t total;
        const uint32_t off = block_exclusive_scan(v, total);
        if (t < tiles) tileCount[t] = sum + off;
        sum += total;
    }
    if (threadIdx.x == 0) {
        result[0] = sum;
        result[1] = 0ull;
    }
}

// ids and entries of the living particles, in entry order
__global__ void __launch_bounds__(kPackThreads) k_part_keys(PackParticles a, const uint32_t* tileOffset,
                                                            unsigned long long* keys, int* vals,
                                                            unsigned long long* result) {
    uint32_t at = tileOffset[blockIdx.x];
    unsigned long long diff = 0ull;
    const unsigned long long ref = a.pid[0];
    for (int r = 0; r < kPartTile / kPackThreads; ++r) {
        const int e = int(blockIdx.x) * kPartTile + r * kPackThreads + int(threadIdx.x);
        const bool on = entry_lives(a, e);
        uint32_t total;
        const uint32_t off = block_exclusive_scan(on ? 1u : 0u, total);
        if (on) {
            const unsigned long long key = e < a.np ? a.pid[e] : a.halves[e - a.np].id;
            keys[at + off] = key;
            vals[at + off] = e;
            diff |= key ^ ref;
        }
        at += total;
    }
    merge_differing(diff, &result[1]);
}

__global__ void __launch_bounds__(kPackThreads) k_pack_particles(PackParticles a, const int* order, int first, int count,
                                                                 uint2* out) {
    __shared__ __align__(16) uint32_t rec[kPackThreads * kPartWords];
    const int k0 = int(blockIdx.x) * kPackThreads;
    const int cnt = min(kPackThreads, count - k0);
    const int tid = int(threadIdx.x);
    if (tid < cnt) {
        const int e = order[first + k0 + tid];
        uint32_t* r = rec + tid * kPartWords;
        unsigned long long id;
        float en;
        float2 p, v;
        uint32_t color;
        if (e < a.np) {
            id = a.pid[e];
            en = a.pen[e];
            p = a.ppos[e];
            v = a.pvel[e];
            color = a.pflags[e] & kParticleColorMask;
            const int ps = a.pslot[e];
            if (a.selected && ps >= 0) color |= uint32_t(a.selected[ps]) << 8;
        } else {
            const StagedParticle h = a.halves[e - a.np];
            id = h.id;
            en = h.energy;
            p = h.pos;
            v = h.vel;
            color = h.color & kParticleColorMask;
        }
        r[0] = uint32_t(id);
        r[1] = uint32_t(id >> 32);
        r[2] = __float_as_uint(en);
        r[3] = __float_as_uint(p.x);
        r[4] = __float_as_uint(p.y);
        r[5] = __float_as_uint(v.x);
        r[6] = __float_as_uint(v.y);
        r[7] = color;
    }
    __syncthreads();
    const uint2* src = reinterpret_cast<const uint2*>(rec);
    uint2* dst = out + size_t(k0) * (kPartWords / 2);
    for (int q = tid; q < cnt * (kPartWords / 2); q += kPackThreads) dst[q] = src[q];
}

// ---- launches --------------------------------------------------------------------------------------
static unsigned blocks_of(int n, int per) { return unsigned((n + per - 1) / per); }

int launch_radix_sort(const SortBuffers& b, int n, unsigned long long differing, hipStream_t s) {
    int at = 0;
    const int tiles = int(blocks_of(n, kSortTile));
    for (int shift = 0; shift < 64 && n > 1; shift += 8) {
        if (((differing >> shift) & 255ull) == 0ull) continue;
        hipLaunchKernelGGL(k_sort_count, dim3(tiles), dim3(kSortThreads), 0, s, b.keys[at], n, shift, b.counts, tiles);
        hipLaunchKernelGGL(k_sort_rows, dim3(256), dim3(kSortThreads), 0, s, b.counts, tiles);
        hipLaunchKernelGGL(k_sort_scatter, dim3(tiles), dim3(kSortThreads), 0, s, b.keys[at], b.vals[at], n, shift, b.counts,
                           tiles, b.keys[at ^ 1], b.vals[at ^ 1]);
        at ^= 1;
    }
    return at;
}

void launch_cell_keys(const unsigned long long* cid, const int* slotOf, int n, const SortBuffers& b,
                      unsigned long long* differing, hipStream_t s) {
    hipLaunchKernelGGL(k_cell_keys, dim3(blocks_of(n, kPackThreads)), dim3(kPackThreads), 0, s, cid, slotOf, n, b.keys[0],
                       b.vals[0], differing);
}

void launch_cell_ranks(const unsigned long long* keys, const int* vals, int n, int* rankOf, unsigned long long* equal,
                       hipStream_t s) {
    hipLaunchKernelGGL(k_cell_ranks, dim3(blocks_of(n, kPackThreads)), dim3(kPackThreads), 0, s, keys, vals, n, rankOf, equal);
}

void launch_cell_order(const int* slotOf, const int* rankOfSlot, int n, int* order, int* rankOf, hipStream_t s) {
    hipLaunchKernelGGL(k_cell_order, dim3(blocks_of(n, kPackThreads)), dim3(kPackThreads), 0, s, slotOf, rankOfSlot, n, order,
                       rankOf);
}

void launch_pack_cells(const PackCells& a, int first, int count, void* out, hipStream_t s) {
    hipLaunchKernelGGL(k_pack_cells, dim3(blocks_of(count, kPackThreads)), dim3(kPackThreads), 0, s, a, first, count,
                       static_cast<uint2*>(out));
}

void launch_part_keys(const PackParticles& a, uint32_t* tileCount, const SortBuffers* b, unsigned long long* result,
                      hipStream_t s) {
    const int tiles = int(blocks_of(a.entries, kPartTile));
    hipLaunchKernelGGL(k_part_count, dim3(tiles), dim3(kPackThreads), 0, s, a, tileCount);
    hipLaunchKernelGGL(k_part_offsets, dim3(1), dim3(1024), 0, s, tileCount, tiles, result);
    if (b) hipLaunchKernelGGL(k_part_keys, dim3(tiles), dim3(kPackThreads), 0, s, a, tileCount, b->keys[0], b->vals[0], result);
}

void launch_pack_particles(const PackParticles& a, const int* order, int first, int count, void* out, hipStream_t s) {
    hipLaunchKernelGGL(k_pack_particles, dim3(blocks_of(count, kPackThreads)), dim3(kPackThreads), 0, s, a, order, first, count,
                       static_cast<uint2*>(out));
}

}  // namespace alien
