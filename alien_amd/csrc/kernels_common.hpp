// kernels_common.hpp — device helpers shared by the kernel files.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "device_math.hpp"
#include "engine_types.hpp"

namespace alien {

__device__ __forceinline__ void slot_of(f2 p, int W, int H, int& sx, int& sy) {
    sx = wrap_int(floor_int(p.x), W);
    sy = wrap_int(floor_int(p.y), H);
}
// floor(a / b) for 0 <= a < 2^24, 0 < b < 2^24: the product with the approximate reciprocal is
// within a few units of the quotient, the corrections make it exact
__device__ __forceinline__ int div_small(int a, int b) {
    int q = int(float(a) * __builtin_amdgcn_rcpf(float(b)));
    while ((q + 1) * b <= a) ++q;
    while (q > 0 && q * b > a) --q;
    return q;
}
// floor(s / binSize) for a slot coordinate (a shift for power-of-two bins)
__device__ __forceinline__ int bin_coord(const DevWorld& w, int s) {
    return w.binShift >= 0 ? s >> w.binShift : div_small(s, w.binSize);
}
__device__ __forceinline__ int cell_bin_local(const DevWorld& w, int sx, int sy) {
    int bx = min(bin_coord(w, sx), w.nbx - 1), by = min(bin_coord(w, sy), w.nby - 1);
    return by * w.nbx + bx;
}
__device__ __forceinline__ int part_bin_local(const DevWorld& w, int sx, int sy) {
    int bx = min(sx / kParticleBin, w.pnbx - 1), by = min(sy / kParticleBin, w.pnby - 1);
    return by * w.pnbx + bx;
}
__device__ __forceinline__ int wrap_small(int x, int n) { return x < 0 ? x + n : (x >= n ? x - n : x); }

// global new-cell index range of local cell bin b
__device__ __forceinline__ void cell_bin_range(const Ctx& c, const DevWorld& w, int b, int& s, int& e) {
    uint32_t base = c.start[w.binOff];
    s = w.cellOff + int(c.start[w.binOff + b] - base);
    e = w.cellOff + int(c.start[w.binOff + b + 1] - base);
}
// (clamped to the world's particle capacity: a map beyond it is reported by the particle scatter)
__device__ __forceinline__ void part_bin_range(const Ctx& c, const DevWorld& w, int b, int& s, int& e) {
    uint32_t base = c.start[w.pbinOff];
    s = w.partOff + min(int(c.start[w.pbinOff + b] - base), w.partCap);
    e = w.partOff + min(int(c.start[w.pbinOff + b + 1] - base), w.partCap);
}

// bin coordinates of a position (on the torus up to rounding; anything else takes the general wrap),
// and its global bin index
__device__ __forceinline__ void cell_bin_xy(const DevWorld& w, f2 p, int& bx, int& by) {
    int sx = static_cast<int>(__builtin_floorf(p.x)), sy = static_cast<int>(__builtin_floorf(p.y));
    if (uint32_t(sx) >= uint32_t(w.W) || uint32_t(sy) >= uint32_t(w.H)) slot_of(p, w.W, w.H, sx, sy);
    bx = min(bin_coord(w, sx), w.nbx - 1);
    by = min(bin_coord(w, sy), w.nby - 1);
}
__device__ __forceinline__ int cell_bin_of(const DevWorld& w, f2 p) {
    int bx, by;
    cell_bin_xy(w, p, bx, by);
    return w.binOff + by * w.nbx + bx;
}

// enters cell k in the far list of global bin gb; the bin's parts are listed once it has more than a lane merges
// in (k_sort.hip)
__device__ __forceinline__ void list_far(const FarCells& f, int groupShift, int* next, int gb, int k) {
    next[k] = atomicExch(&f.head[gb], k);
    const int n = atomicAdd(&f.count[gb], 1);
    f.group[gb >> groupShift] = 1;
    if (n == kFarWalk || (n > kFarWalk && n % 64 == 0)) f.list[atomicAdd(f.total, 1)] = make_int2(gb, n / 64);
}

// moves the active lanes' cells between groups in the sums of groups: one atomic per group that gains or
// loses any
__device__ __forceinline__ void add_per_key(int* sums, int key, int unit) {
    const int lane = int(threadIdx.x) & 63;
    for (unsigned long long m = __ballot(true); m != 0ull;) {
        const int lead = __builtin_ctzll(m), k = __builtin_amdgcn_readlane(key, lead);
        const unsigned long long same = __ballot(key == k);
        if (lane == lead) atomicAdd(&sums[k], unit * __builtin_popcountll(same));
        m &= ~same;
    }
}
__device__ __forceinline__ void shift_groups(int* sums, int* supers, int from, int to) {
    add_per_key(sums, from, -1);
    add_per_key(sums, to, 1);
    const int sf = from / kSuperGroups, st = to / kSuperGroups;
    if (sf != st) {
        add_per_key(supers, sf, -1);
        add_per_key(supers, st, 1);
    }
}

// flat bins that a cell with near move code `move` crossed
__device__ __forceinline__ int move_bins(const DevWorld& w, uint32_t move) {
    const int m = int(move) - 1, y = m >= 6 ? 1 : (m >= 3 ? 0 : -1);
    return m - 3 * y - 4 + y * w.nbx;
}

// base[i] through a 32-bit byte offset, which a 64-bit address of a signed index costs four operations
// more than (a set's cells times 8 bytes, and a world's bins times 4, stay below 2^32)
template <class T> __device__ __forceinline__ T* at32(T* base, uint32_t i) {
    using Byte = typename std::conditional<std::is_const<T>::value, const char, char>::type;
    return reinterpret_cast<T*>(reinterpret_cast<Byte*>(base) + uint32_t(i * uint32_t(sizeof(T))));
}
template <class T> __device__ __forceinline__ T ld32(const T* base, uint32_t i) { return *at32(base, i); }
template <class T> __device__ __forceinline__ void st32(T* base, uint32_t i, T v) { *at32(base, i) = v; }
static_assert(uint64_t(kMaxSetCells) * 8 < (uint64_t(1) << 32), "32-bit byte offsets");

// Next-step bin of the cell at end-of-step index k: end-of-step position pNew; bOld, its bin in this
// step's map (the bin of its start-of-step position, counted from the world's first).  The next map
// looks for a bin's cells in the bins one and one row of bins around (counted along the rows, so a step
// across the end of a row is near, one across the torus' edge is not).
__device__ __forceinline__ void bin_next(const Ctx& c, const DevWorld& w, int k, f2 pNew, int bOld) {
    int bx, by;
    cell_bin_xy(w, pNew, bx, by);
    const int b = by * w.nbx + bx;
    const int d = b - bOld;
    uint32_t move = 0u;
    if (d != 0) {
        const int y = d > 1 ? 1 : (d < -1 ? -1 : 0), x = d - y * w.nbx;
        move = uint32_t(3 * (y + 1) + x + 2);
        if (x < -1 || x > 1) {
            move = kFarCode;
            list_far(c.farNext, c.groupShift, c.farLink, w.binOff + b, k);
        }
        const int from = (w.binOff + bOld) >> c.groupShift, to = (w.binOff + b) >> c.groupShift;
        if (from != to) shift_groups(c.groupSumNext, c.superSumNext, from, to);
    }
    st32(c.binOf, uint32_t(k), int(uint32_t(b) | move << kMoveShift));
}

__device__ __forceinline__ void pbin_for_next_step(const Ctx& c, const DevWorld& w, int k, f2 p, uint32_t* hist) {
    int sx, sy;
    slot_of(p, w.W, w.H, sx, sy);
    int gb = w.pbinOff + part_bin_local(w, sx, sy);
    c.pbinOf[k] = gb;
    atomicAdd(&hist[gb], 1u);
}

// Inclusive sum over the 64 lanes of a wave (all lanes active), with DPP row shifts and row
// broadcasts instead of LDS permutes: sums of up to four lanes, of eight, of the 16-lane row, then
// row 0's total into row 1 and row 2's into row 3, then lane 31's prefix into rows 2 and 3.
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t x) {
    uint32_t v = x;
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x111, 0xf, 0xf, true));   // row_shr:1
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x112, 0xf, 0xf, true));   // row_shr:2
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x113, 0xf, 0xf, true));   // row_shr:3
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x114, 0xf, 0xe, false));  // row_shr:4, lanes 4-15
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x118, 0xf, 0xc, false));  // row_shr:8, lanes 8-15
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x142, 0xa, 0xf, false));  // row_bcast:15, rows 1, 3
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x143, 0xc, 0xf, false));  // row_bcast:31, rows 2, 3
    return v;
}

// the value of lane 63 (a wave total after an inclusive scan), read as a scalar
__device__ __forceinline__ int wave_last(int v) { return __builtin_amdgcn_readlane(v, 63); }

// exclusive scan across the block (blockDim multiple of 64, at most 1024); block total in `total`
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t& total) {
    __shared__ uint32_t waveSums[17];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int numWaves = blockDim.x >> 6;
    uint32_t inc = wave_inclusive_scan(v);
    if (lane == 63) waveSums[wave] = inc;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t s = 0;
        for (int k = 0; k < numWaves; ++k) {
            uint32_t t = waveSums[k];
            waveSums[k] = s;
            s += t;
        }
        waveSums[16] = s;
    }
    __syncthreads();
    uint32_t res = inc - v + waveSums[wave];
    total = waveSums[16];
    __syncthreads();
    return res;
}

// Several kernels run the cells' and the particles' work of a phase in one launch, each part on its
// own workgroups: a workgroup's place among those of its part
struct Span {
    int block, blocks;
};

// grid-stride iteration over the blocks of live particles (the table the particle bin sort writes
// for the live ranges it publishes)
template <class F> __device__ __forceinline__ void for_live_particles(const Ctx& c, Span at, F&& f) {
    const int n = *c.numPartBlocks;
    for (int e = at.block; e < n; e += at.blocks) {
        const int2 blk = c.partBlocks[e];
        const int live = c.ctr[blk.x].numParticles;
        const DevWorld& w = c.worlds[blk.x];
        const int k = blk.y + int(threadIdx.x);
        if (k < w.partOff + live) f(blk.x, w, k);
    }
}

}  // namespace alien
