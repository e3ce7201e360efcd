// k_sort.hip — spatial hash: counting sort of cells and energy particles by bin.
//
// Replaces ALIEN's CellMap / ParticleMap (source/EngineGpuKernels/Map.cuh:71-280), which insert
// pointers into a dense world-size grid with atomicCAS chains (cell map) or last-writer-wins
// stores (particle map).  Here every bin of every world is one offset.  The cells' map holds them by
// bin and inside a bin by previous index (R1), so the map order is the logical order of the step.  The
// kernels that produce the end-of-step positions record each cell's next bin and the direction it went
// (binOf); the next map finds a bin's cells where they can be: almost all are still in the bin, and a
// cell that moved comes from one of the eight bins around.  So a wave that builds the map of consecutive
// bins reads what was recorded for the cells of three stretches of the last map — its own bins, the row
// above, the row below — and needs no lists.  Where the bins start follows from where they started in the
// last map and from the cells that changed groups of 256 bins since (groupSum: their numbers, added up by
// the kernels that record the bins, one atomic per wave and group).  The map takes one launch.
// (Recording every mover in a list of its new bin and counting it out of the old one cost three
// device-scope atomics each, which the memory side executes: 40 of 143 us of the fluid pass with 4M
// cells; clearing those lists and a scan over all bins with tiles that wait for the tiles before them,
// 34 us more.  Steps then and now: 256k cells 26.5 and 22.1 us, 4M 168 and 139 us, 0.84M in bodies
// with bonds 314 and 300 us.  A launch of its own that counts the groups took 18 us at 4M.)
// Only cells that moved further, or across the torus' edge, or that are in no map yet are entered in a
// list per bin ("far").  Particles: counted with atomics, scattered, then sorted inside their bins.
#include "kernels.hpp"
#include "particle_steps.hpp"

namespace alien {

__global__ void k_fill_u32(uint32_t* p, uint32_t v, size_t n) {
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    size_t stride = size_t(gridDim.x) * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

// bins of the current state, used after data is set and after introspection: the current state
// is in no map order yet (every bin of the last map is empty), so every cell is a far one of the
// coming step
__global__ void k_cell_bin(Ctx c) {
    int2 blk = c.cellBlocks[blockIdx.x];
    const DevWorld w = c.worlds[blk.x];
    int i = blk.y + int(threadIdx.x);
    if (i >= w.cellOff + w.numCells) return;
    int bx, by;
    cell_bin_xy(w, to_f2(c.A.pos[i]), bx, by);
    const int gb = w.binOff + by * w.nbx + bx;
    c.binOf[i] = int(uint32_t(gb - w.binOff) | kFarMove);
    list_far(c.far, c.groupShift, c.farLink, gb, i);
}

// (the groups gain their far cells; a wave for 256 bins)
__global__ void k_seed_sums(Ctx c) {
    const int g0 = (int(blockIdx.x) * int(blockDim.x) + int(threadIdx.x)) / 64 * kGroupBins, lane = int(threadIdx.x) & 63;
    if (g0 >= c.numCellBins) return;
    const int4 n = reinterpret_cast<const int4*>(c.far.count + g0)[lane];
    const int lanes = (1 << c.groupShift) / 4;
    int sum = n.x + n.y + n.z + n.w;
    for (int o = 1; o < lanes; o *= 2) sum += __shfl_xor(sum, o, 64);
    if (lane % lanes != 0) return;
    const int g = (g0 + 4 * lane) >> c.groupShift;
    c.groupSum[g] = sum;
    if (sum) atomicAdd(&c.superSum[g / kSuperGroups], sum);
}

__global__ void k_part_bin(Ctx c) {
    for_live_particles(c, {int(blockIdx.x), int(gridDim.x)}, [&](int, const DevWorld& w, int i) {
        if (c.A.pflags[i] & kParticleDead)
            c.pbinOf[i] = -1;
        else
            pbin_for_next_step(c, w, i, to_f2(c.A.ppos[i]), c.count);
        // a half split off particle i at the end of the last step
        if (c.splitStage > 0) {
            const StagedParticle& r = c.splitStaged[i];
            if (r.color & kStagedPending)
                pbin_for_next_step(c, w, c.splitStage + i, to_f2(r.pos), c.count);
            else
                c.pbinOf[c.splitStage + i] = -1;
        }
    });
}

// The bins whose cells can be in bins [b0, b0 + nb) of a world without having moved far: three stretches
// of bins, above, around and below, disjoint and in order (in narrow worlds they join).
struct Reach {
    int lo[3], hi[3];
};
__device__ __forceinline__ Reach reach_of(const DevWorld& w, int b0, int nb) {
    const int n = w.nbx * w.nby;
    Reach r;
    r.lo[0] = max(b0 - w.nbx - 1, 0);
    r.hi[0] = max(min(b0 + nb - w.nbx + 1, b0 - 1), r.lo[0]);
    r.lo[1] = max(b0 - 1, 0);
    r.hi[1] = min(b0 + nb + 1, n);
    r.hi[2] = min(b0 + nb + w.nbx + 1, n);
    r.lo[2] = min(max(b0 + w.nbx - 1, b0 + nb + 1), r.hi[2]);
    return r;
}
// the same as places in the last map, counted from the world's first cell
struct Places {
    int s[3], e[3];
};
__device__ __forceinline__ Places places_of(const Reach& r, const uint32_t* prev) {
    const int base = int(prev[0]);
    Places p;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        p.s[k] = int(prev[r.lo[k]]) - base;
        p.e[k] = int(prev[r.hi[k]]) - base;
    }
    return p;
}

__device__ __forceinline__ int world_of(const Ctx& c, int gb) { return c.numWorlds == 1 ? 0 : c.groupWorld[gb / kGroupBins]; }
__device__ __forceinline__ uint32_t move_of(int x) { return uint32_t(x) >> kMoveShift; }
// the recorded bin, counted from bin b0
__device__ __forceinline__ uint32_t bin_from(int x, int b0) { return (uint32_t(x) & kBinMask) - uint32_t(b0); }

// what cells [i0, end) of a world recorded, 64 per round, with all the loads in flight.  The first rounds
// load without a look at the end (the array goes on beyond it, kBinOfPad).
template <int kRounds>
__device__ __forceinline__ void load_rounds(const int* binOf, int i0, int end, int lane, int (&x)[kRounds]) {
    static_assert(64 * kRounds <= kBinOfPad, "loads beyond the end");
    const int* at = binOf + i0;
#pragma unroll
    for (int q = 0; q < kRounds; ++q)
        if (q < kRounds - 1 || i0 + 64 * q < end) x[q] = at[lane + 64 * q];
}

// ---------------------------------------------------------------------------------------------
// Offsets of the particle bins in one pass: a workgroup takes the next tile of bins (tickets in the order
// the workgroups start), sums its bins up and publishes the sum, then finds the sum of all bins before
// it by looking back over what the tiles before it published (decoupled look-back: a tile publishes its
// own sum before it looks back, and every tile before it holds an earlier ticket and has started, so each
// wait ends).  `count` stays: the particle scatter counts its bins down to zero, which leaves them
// cleared for the step after next (the two histograms alternate).
// ---------------------------------------------------------------------------------------------
constexpr int kScanItems = 8;  // consecutive particle bins per thread
constexpr int kMapThreads = 256;
constexpr int kPartScanTile = kMapThreads * kScanItems;
// tile status word: flag (bits 62-63: 1 the tile's sum, 2 the sum up to and including the tile),
// launch epoch (bits 32-61), value (bits 0-31)
constexpr unsigned long long kTileSum = 1ull << 62, kTileInclusive = 2ull << 62;
constexpr uint32_t kEpochMask = 0x3fffffffu;
constexpr int kLookBackSpins = 1 << 22;  // far beyond any wait for a running tile

// Workgroup b runs on XCD b % 8: of `blocks` (a multiple of 8) each XCD gets one contiguous run, so the
// rows that neighbouring waves share stay in its L2
__device__ __forceinline__ int xcd_run(int b, int blocks) { return (b % kXcdCount) * (blocks / kXcdCount) + b / kXcdCount; }

__device__ __forceinline__ bool tile_status_ready(unsigned long long w, uint32_t epoch) {
    return (w >> 62) != 0ull && uint32_t((w >> 32) & kEpochMask) == epoch;
}

__device__ __forceinline__ void part_scan(const Ctx& c, int tiles) {
    __shared__ int sTile;
    __shared__ uint32_t sEpoch, sPrefix;
    const int tid = int(threadIdx.x), lane = tid & 63;
    // All atomics here are relaxed (agent scope): a status word carries its whole message (flag,
    // epoch, value), and the epoch and ticket a launch reads were written by the launches before
    // it.  Ordered ones would write back or invalidate the XCD's L2 at every store and load.
    if (tid == 0) {
        const uint32_t e = __hip_atomic_load(c.mapEpoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // the epoch has been read when the ticket is taken; the last ticket's holder advances it
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        sEpoch = e & kEpochMask;
        sTile = int(__hip_atomic_fetch_add(c.mapTicket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    }
    __syncthreads();
    const int tile = sTile;
    const uint32_t epoch = sEpoch;
    const unsigned long long ep = (unsigned long long)epoch << 32;
    const uint32_t n = uint32_t(c.numBins);
    const uint32_t base = uint32_t(c.numCellBins) + uint32_t(tile) * uint32_t(kPartScanTile) + uint32_t(tid * kScanItems);
    uint32_t v[kScanItems];
    if (base + 8 <= n) {
        const uint4 a = *reinterpret_cast<const uint4*>(c.count + base);
        const uint4 b = *reinterpret_cast<const uint4*>(c.count + base + 4);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) v[k] = base + k < n ? c.count[base + k] : 0u;
    }
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) s += v[k];
    uint32_t total;
    const uint32_t off = block_exclusive_scan(s, total);
    if (tid == 0)
        __hip_atomic_store(&c.mapStatus[tile], (tile == 0 ? kTileInclusive : kTileSum) | ep | total, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    if (tid < 64) {
        // the first wave looks back, 64 tiles at a time, until a tile with its inclusive sum
        uint32_t prefix = 0;
        if (tile > 0) {
            for (int j = tile - 1;; j -= 64) {
                const int idx = j - lane;
                unsigned long long w = kTileInclusive | ep;  // before the first tile: sum 0
                if (idx >= 0) {
                    // (bounded: a tile that never published would be a bug; the step then reports
                    // an error instead of hanging)
                    for (int spin = 0;; ++spin) {
                        w = __hip_atomic_load(&c.mapStatus[idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if (tile_status_ready(w, epoch)) break;
                        if (spin >= kLookBackSpins) {
                            atomicOr(&c.sc->errors, 2);
                            w = kTileInclusive | ep;
                            break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                    }
                }
                const unsigned long long incl = __ballot((w >> 62) == 2ull);
                const int stop = incl ? __builtin_ctzll(incl) : 64;
                uint32_t val = lane <= stop ? uint32_t(w) : 0u;
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) val += __shfl_xor(val, o, 64);
                prefix += val;
                if (incl) break;
            }
            if (lane == 0)
                __hip_atomic_store(&c.mapStatus[tile], kTileInclusive | ep | (prefix + total), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        if (lane == 0) sPrefix = prefix;
    }
    __syncthreads();
    // (a particle bin's offset counts from its world's first; the first bin's is also the end of the
    // last cell bin)
    uint32_t o = uint32_t(c.cellCount) + sPrefix + off;
    uint32_t st8[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        st8[k] = o;
        o += v[k];
    }
    if (base + 8 <= n) {
        *reinterpret_cast<uint4*>(c.start + base) = make_uint4(st8[0], st8[1], st8[2], st8[3]);
        *reinterpret_cast<uint4*>(c.start + base + 4) = make_uint4(st8[4], st8[5], st8[6], st8[7]);
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
            if (base + k < n) c.start[base + k] = st8[k];
    }
    if (base < n && n <= base + kScanItems) c.start[n] = o;
    // the last ticket: every ticket is gone; reset the ticket and advance the epoch for the next
    // launch
    if (tile == tiles - 1 && tid == 0) {
        __hip_atomic_store(c.mapTicket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_fetch_add(c.mapEpoch, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---------------------------------------------------------------------------------------------
// The cells' map.  One wave per group puts every cell of its bins at its rank by A index, i.e. by its place
// in the last map (R1).  It goes over the bins' reach in that order, 64 cells at a time, with the first
// rounds' loads of all three stretches in flight together: the wave is a chain of latencies (table,
// offsets, cells, stores; 9 us at 1024 waves, 33 us at 16384, where the VALU's share is 15).  Each XCD
// takes one run of groups (the rows that neighbouring waves share: 7 of 40 us).
//  - The bins' own cells that left are counted per bin; the near movers into the bins are counted and, met
//    in order, listed in LDS.  That gives the bins' sizes, and with the groups before it their offsets.
//  - The bins' own cells that stayed hold their old order: a stayer's rank is its place in the bin's
//    old stretch, minus the cells that left the bin before it, plus the movers into it from lower places.
//  - A listed mover from a lower place comes behind the listed ones of its bin before it, one from a
//    higher place behind the stayers as well.  If there are more than the list holds, another run over
//    the reach places them, the lanes of one bin in turns (256k cells of 1 to 2 units a step: the map 61 us
//    with one bin of a round after the other, 26 with turns).
//  - Far cells: the near cells of a bin with few of them take its first places, and at the end the bin's lane
//    merges its far cells in (256k cells that move 5 units a step: a step of 158 us with a wave for each far
//    cell, 58 so; 1M of them 500 and 111).  Bins with more far cells than a lane takes (kFarWalk) get a wave
//    per 64 of them: it counts the cells of the group before them over the group's reach, and their ranks
//    along the list; the near cells of such a bin add the list's smaller indices.
// ---------------------------------------------------------------------------------------------
constexpr int kMapWaves = kMapThreads / 64;
constexpr int kScatterList = 192;  // movers into a group's bins listed (typically 5 to 25), a multiple of 8
constexpr int kScatterRounds = 5;  // rounds of a stretch loaded at once (258 bins at up to 1.24 cells per bin)
constexpr int kFarBlocks = 256;    // workgroups for the bins with many far cells, at most
static_assert(kGroupBins == 4 * 64, "four bins per lane");

template <int kBins> struct ScatterShared {
    int prev[kBins + 4];  // places in the last map, counted from the world's first cell
    union {
        int start[kBins + 4];  // the same in the new map
        uint32_t out[kBins];   // before it is known: cells that left the bin
    };
    uint32_t before[kBins], after[kBins];  // near movers into the bin from lower and higher places
    union {
        int2 list[kScatterList];   // (A index in the world, bin)
        struct {                   // the other run
            uint32_t met[kBins];   // movers placed so far
            uint16_t turn[kBins];  // lane whose turn it is
        } run;
    };
};

// cells that the world's groups before global group g gained since the last map
__device__ __forceinline__ int gained_before(const Ctx& c, const DevWorld& w, int g, int lane) {
    const int first = w.binOff >> c.groupShift;
    const int s0 = (first + kSuperGroups - 1) / kSuperGroups, s1 = g / kSuperGroups;
    int n = 0;
    if (s0 < s1) {
        for (int k = first + lane; k < s0 * kSuperGroups; k += 64) n += c.groupSum[k];
        for (int k = s0 + lane; k < s1; k += 64) n += c.superSum[k];
        for (int k = s1 * kSuperGroups + lane; k < g; k += 64) n += c.groupSum[k];
    } else {
        for (int k = first + lane; k < g; k += 64) n += c.groupSum[k];
    }
    return wave_last(int(wave_inclusive_scan(uint32_t(n))));
}

// the next step's sums, and the far lists of the group's bins where there are any, start empty (their last
// readers ran a step ago)
template <int kBins> __device__ __forceinline__ void clear_next(const Ctx& c, int g, int lane) {
    if (lane == 0) {
        c.groupSumNext[g] = 0;
        if (g % kSuperGroups == 0) c.superSumNext[g / kSuperGroups] = 0;
    }
    if (c.farNext.group[g] == 0) return;
    if (lane < kBins / 4) {
        reinterpret_cast<int4*>(c.farNext.count + g * kBins)[lane] = make_int4(0, 0, 0, 0);
        reinterpret_cast<int4*>(c.farNext.head + g * kBins)[lane] = make_int4(kNone, kNone, kNone, kNone);
    }
    if (lane == 0) c.farNext.group[g] = 0;
}

// far cells of global bin gb with A index below i
__device__ __forceinline__ int rank_far(const Ctx& c, int gb, int i) {
    int n = 0;
    for (int j = c.far.head[gb]; j != kNone; j = c.farLink[j]) n += j < i ? 1 : 0;
    return n;
}

// (the passes read the cells' state through `sorted`: a copy of it in map order costs more than it saves)
__device__ __forceinline__ void place_cell(const Ctx& c, const DevWorld& w, int i, int dest) {
    st32(c.sorted, uint32_t(w.cellOff + dest), w.cellOff + i);
}

// The far cells of bins with more than kFarWalk: one wave per entry, 64 of a bin's list
template <int kBins> __device__ __forceinline__ void far_scatter(const Ctx& c, int wave, int waves, int lane) {
    const int total = *c.far.total;
    for (int q = wave; q < total; q += waves) {
        const int2 entry = c.far.list[q];
        const int gb = entry.x, first = 64 * entry.y;
        const DevWorld& w = c.worlds[world_of(c, gb)];
        if (!w.active) continue;
        // this lane's cell, and its rank among the list's
        int own = kNone, rank = 0;
        for (int j = c.far.head[gb], n = 0; j != kNone && n < first + 64; j = c.farLink[j], ++n) own = n - first == lane ? j : own;
        for (int j = c.far.head[gb]; j != kNone; j = c.farLink[j]) rank += j < own ? 1 : 0;
        const int g = gb / kBins, b0 = g * kBins - w.binOff;
        const uint32_t t = uint32_t(gb - w.binOff - b0);
        const int i = own - w.cellOff;
        const uint32_t* prev = c.startPrev + w.binOff;
        const Places p = places_of(reach_of(w, b0, min(kBins, w.nbx * w.nby - b0)), prev);
        const int* binOf = c.binOf + w.cellOff;
        const int4 fc = lane < kBins / 4 ? reinterpret_cast<const int4*>(c.far.count + g * kBins)[lane] : make_int4(0, 0, 0, 0);
        const int base = int(prev[b0] - prev[0]) + gained_before(c, w, g, lane);
        const uint32_t b = uint32_t(4 * lane);
        // cells of the group's bins before this one, and the bin's near cells before the lane's
        uint32_t n = (b < t ? uint32_t(fc.x) : 0u) + (b + 1u < t ? uint32_t(fc.y) : 0u) + (b + 2u < t ? uint32_t(fc.z) : 0u) +
                     (b + 3u < t ? uint32_t(fc.w) : 0u);
        for (int k = 0; k < 3; ++k)
            for (int j0 = p.s[k]; j0 < p.e[k]; j0 += 256) {
                int x[4];
                load_rounds(binOf, j0, p.e[k], lane, x);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const bool in = j0 + 64 * r + lane < p.e[k] && move_of(x[r]) != kFarCode;
                    const uint32_t u = in ? bin_from(x[r], b0) : ~0u;
                    n += u < t ? 1u : 0u;
                    for (unsigned long long m = __ballot(u == t); m != 0ull; m &= m - 1ull)
                        rank += j0 + 64 * r + __builtin_ctzll(m) < i ? 1 : 0;
                }
            }
        const int at = base + wave_last(int(wave_inclusive_scan(n))) + rank;
        if (own != kNone) place_cell(c, w, i, at);
    }
}

// Merges the k far cells of a bin (at most kMax) into its places `seg`, whose first m hold its other cells in
// order
template <int kMax> __device__ __forceinline__ void merge_far(int* seg, const int* link, int head, int k, int m) {
    int f[kMax], to[kMax];
#pragma unroll
    for (int s = 0; s < kMax; ++s) {
        f[s] = s < k ? head : 0x7fffffff;
        if (s + 1 < k) head = link[head];
    }
#pragma unroll
    for (int s = 0; s < kMax; ++s) {
        to[s] = 0;
#pragma unroll
        for (int j = 0; j < kMax; ++j) to[s] += f[j] < f[s] ? 1 : 0;
    }
    // the others from the last one on, up behind the far cells before them; those before all stay
    for (; m > 0; --m) {
        const int e = seg[m - 1];
        int n = 0;
#pragma unroll
        for (int s = 0; s < kMax; ++s) n += f[s] < e ? 1 : 0;
        if (n == 0) break;
#pragma unroll
        for (int s = 0; s < kMax; ++s) to[s] += f[s] > e ? 1 : 0;
        seg[m - 1 + n] = e;
    }
#pragma unroll
    for (int s = 0; s < kMax; ++s)
        if (s < k) seg[m + to[s]] = f[s];
}

template <int kBins>
__device__ __forceinline__ void cell_scatter(const Ctx& c, ScatterShared<kBins>& S, int g, int lane) {
    const bool binLane = lane < kBins / 4;  // (four bins each)
    const int g0 = g * kBins;
    if (g0 >= c.numCellBins) return;
    const DevWorld& w = c.worlds[world_of(c, g0)];
    const int b0 = g0 - w.binOff, bins = w.nbx * w.nby;
    const uint32_t* prev = c.startPrev + w.binOff;
    const int prevBase = int(prev[0]);
    const uint4 pv = binLane ? *reinterpret_cast<const uint4*>(prev + b0 + 4 * lane) : make_uint4(0u, 0u, 0u, 0u);
    const uint32_t pvEnd = prev[b0 + kBins];
    uint4* startOut = reinterpret_cast<uint4*>(c.start + g0) + lane;
    const bool last = g0 + kBins == c.numCellBins;  // its end is stored too
    clear_next<kBins>(c, g, lane);
    if (!w.active || b0 >= bins) {
        // a world left out keeps its map; padding ends with the world
        const uint32_t d = uint32_t(w.cellOff - prevBase), end = uint32_t(w.cellOff + w.numCells);
        if (binLane) *startOut = w.active ? make_uint4(end, end, end, end) : make_uint4(pv.x + d, pv.y + d, pv.z + d, pv.w + d);
        if (last && lane == 0) c.start[c.numCellBins] = end;
        return;
    }
    const int nb = min(kBins, bins - b0);
    const int p0 = int(prev[b0]) - prevBase, p1 = int(prev[b0 + nb]) - prevBase;  // the bins' own cells
    const Places p = places_of(reach_of(w, b0, nb), prev);
    const bool farCells = c.far.group[g] != 0;
    bool manyFar = false;  // some bin has more than its lane merges in
    const int* binOf = c.binOf + w.cellOff;
    const int base = p0 + gained_before(c, w, g, lane);
    int x[3][kScatterRounds];
#pragma unroll
    for (int k = 0; k < 3; ++k) load_rounds(binOf, p.s[k], p.e[k], lane, x[k]);
    if (binLane) {
        reinterpret_cast<int4*>(S.prev)[lane] =
            make_int4(int(pv.x) - prevBase, int(pv.y) - prevBase, int(pv.z) - prevBase, int(pv.w) - prevBase);
        reinterpret_cast<uint4*>(S.out)[lane] = make_uint4(0u, 0u, 0u, 0u);
        reinterpret_cast<uint4*>(S.before)[lane] = make_uint4(0u, 0u, 0u, 0u);
        reinterpret_cast<uint4*>(S.after)[lane] = make_uint4(0u, 0u, 0u, 0u);
    }
    if (lane == 0) S.prev[kBins] = int(pvEnd) - prevBase;
    __syncwarp();
    int listed = 0;  // movers into the bins so far (listed up to the list's size)
    // cells i0 + lane of the stretch around the bins (k == 1), above or below: what they recorded
    auto meet = [&](int k, int y, int i0) {
        if (i0 >= p.e[k]) return;
        const int i = i0 + lane;
        const uint32_t move = move_of(y), t = bin_from(y, b0);
        const bool into = i < p.e[k] && move != 0u && move != kFarCode && t < uint32_t(nb);
        if (k == 1 && move != 0u && i >= p0 && i < p1) {
            int old;
            if (move != kFarCode) {
                old = int(t) - move_bins(w, move);
            } else {  // the last bin that starts at or before the cell
                old = 0;
#pragma unroll
                for (int s = kBins / 2; s > 0; s >>= 1)
                    if (S.prev[old + s] <= i) old += s;
            }
            atomicAdd(&S.out[old], 1u);
        }
        const unsigned long long m = __ballot(into);
        if (m == 0ull) return;
        if (into) {
            atomicAdd(k == 0 || (k == 1 && i < S.prev[t]) ? &S.before[t] : &S.after[t], 1u);
            const int q = int(__builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), uint32_t(listed))));
            if (q < kScatterList) S.list[q] = make_int2(i, int(t));
        }
        listed += __builtin_popcountll(m);
    };
#pragma unroll
    for (int k = 0; k < 3; ++k) {
#pragma unroll
        for (int q = 0; q < kScatterRounds; ++q) meet(k, x[k][q], p.s[k] + 64 * q);
        for (int i0 = p.s[k] + 64 * kScatterRounds; i0 < p.e[k]; i0 += 256) {
            int y[4];
            load_rounds(binOf, i0, p.e[k], lane, y);
#pragma unroll
            for (int q = 0; q < 4; ++q) meet(k, y[q], i0 + 64 * q);
        }
    }
    __syncwarp();
    // sizes and offsets
    {
        uint32_t v[4] = {0u, 0u, 0u, 0u};
        if (binLane) {
            const uint4 o = reinterpret_cast<const uint4*>(S.out)[lane];
            const uint4 f = reinterpret_cast<const uint4*>(S.before)[lane], a = reinterpret_cast<const uint4*>(S.after)[lane];
            const int next = S.prev[4 * lane + 4];
            v[0] = pv.y - pv.x - o.x + f.x + a.x, v[1] = pv.z - pv.y - o.y + f.y + a.y;
            v[2] = pv.w - pv.z - o.z + f.z + a.z, v[3] = uint32_t(next + prevBase) - pv.w - o.w + f.w + a.w;
        }
        if (farCells) {
            const int4 fc = binLane ? *reinterpret_cast<const int4*>(c.far.count + g0 + 4 * lane) : make_int4(0, 0, 0, 0);
            manyFar = __any(max(max(fc.x, fc.y), max(fc.z, fc.w)) > kFarWalk);
            v[0] += uint32_t(fc.x), v[1] += uint32_t(fc.y), v[2] += uint32_t(fc.z), v[3] += uint32_t(fc.w);
        }
        const uint32_t sum = v[0] + v[1] + v[2] + v[3];
        const int s0 = base + int(wave_inclusive_scan(sum) - sum);
        const int4 s = make_int4(s0, s0 + int(v[0]), s0 + int(v[0] + v[1]), s0 + int(v[0] + v[1] + v[2]));
        const uint32_t off = uint32_t(w.cellOff);
        if (binLane) {
            reinterpret_cast<int4*>(S.start)[lane] = s;
            *startOut = make_uint4(off + uint32_t(s.x), off + uint32_t(s.y), off + uint32_t(s.z), off + uint32_t(s.w));
        }
        if (lane == 63) {
            S.start[kBins] = s0 + int(sum);
            if (last) c.start[c.numCellBins] = off + uint32_t(w.numCells);
        }
    }
    __syncwarp();
    // far cells before cell i in bin t, where they are not merged in at the end
    auto far_before = [&](int t, int i) {
        return manyFar && c.far.count[g0 + t] > kFarWalk ? rank_far(c, g0 + t, w.cellOff + i) : 0;
    };
    const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    unsigned long long leftPrev = 0ull;  // the round before: own cells that left their bin
    int longStart = -1, longGone = 0;    // the bin that reaches into this round: its cells that left before it
    auto stay = [&](int y, int i0) {
        const int i = i0 + lane;
        const bool own = i >= p0 && i < p1;
        const uint32_t move = move_of(y), t = bin_from(y, b0);
        const unsigned long long left = __ballot(own && move != 0u);
        const bool stays = own && move == 0u;
        const int sb = stays ? S.prev[t] : i0;
        const unsigned long long old = __ballot(sb < i0);
        if (old) {  // (all of one bin)
            const int from = __builtin_amdgcn_readlane(sb, __builtin_ctzll(old));
            if (from != longStart) {
                longStart = from;
                longGone = __builtin_popcountll(from > i0 - 64 ? leftPrev >> (from - (i0 - 64)) : leftPrev);
                for (int j0 = from; j0 < i0 - 64; j0 += 64) {
                    const int j = j0 + lane;
                    longGone += __builtin_popcountll(__ballot(j < i0 - 64 && move_of(binOf[min(j, i0)]) != 0u));
                }
            }
        }
        if (stays) {
            const int gone = sb < i0 ? longGone + __builtin_popcountll(left & below)
                                     : __builtin_popcountll(left & below & ~((1ull << (sb - i0)) - 1ull));
            place_cell(c, w, i, S.start[t] + i - sb - gone + int(S.before[t]) + far_before(int(t), i));
        }
        longGone += __builtin_popcountll(left);
        leftPrev = left;
    };
#pragma unroll
    for (int q = 0; q < kScatterRounds; ++q)
        if (p.s[1] + 64 * q < p1) stay(x[1][q], p.s[1] + 64 * q);
    for (int i0 = p.s[1] + 64 * kScatterRounds; i0 < p1; i0 += 256) {
        int y[4];
        load_rounds(binOf, i0, p1, lane, y);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (i0 + 64 * q < p1) stay(y[q], i0 + 64 * q);
    }
    // a mover's place, n: movers into its bin before it
    auto place_mover = [&](int i, int t, int n) {
        int at = S.start[t] + n;
        if (i >= S.prev[t]) {  // behind the stayers
            at += S.start[t + 1] - S.start[t] - int(S.before[t] + S.after[t]);
            if (farCells) at -= c.far.count[g0 + t];
        }
        place_cell(c, w, i, at + far_before(t, i));
    };
    if (listed <= kScatterList) {
        for (int q0 = 0; q0 < listed; q0 += 64) {
            const int q = q0 + lane;
            const bool on = q < listed;
            const int2 m = S.list[on ? q : 0];
            int n = 0;
            // (few bins get more than one)
            if (__ballot(on && S.before[m.y] + S.after[m.y] > 1u)) {
                const int end = min(listed, q0 + 64);
                for (int j = 0; j < end; j += 8) {
                    int4 v[4];  // (two of the list each; the reads in flight together)
#pragma unroll
                    for (int u = 0; u < 4; ++u) v[u] = reinterpret_cast<const int4*>(S.list)[j / 2 + u];
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        n += (v[u].y == m.y && j + 2 * u < q ? 1 : 0) + (v[u].w == m.y && j + 2 * u + 1 < q ? 1 : 0);
                }
            }
            if (on) place_mover(m.x, m.y, n);
        }
    } else {
        if (binLane) {
            reinterpret_cast<uint4*>(S.run.met)[lane] = make_uint4(0u, 0u, 0u, 0u);
            reinterpret_cast<uint2*>(S.run.turn)[lane] = make_uint2(~0u, ~0u);
        }
        __syncwarp();
        for (int k = 0; k < 3; ++k)
            for (int i0 = p.s[k]; i0 < p.e[k]; i0 += 64) {
                const int i = i0 + lane;
                const int y = binOf[min(i, p.e[k] - 1)];
                const uint32_t move = move_of(y), t = bin_from(y, b0);
                const bool into = i < p.e[k] && move != 0u && move != kFarCode && t < uint32_t(nb);
                // Lanes of one bin take turns, whoever comes first: a lane's movers before it are those met in
                // the rounds before, and the turns of lower lanes
                bool waits = into;
                int n = into ? int(S.run.met[t]) : 0;
                for (uint32_t turn = 0; __any(waits); turn += 64u) {
                    if (waits) S.run.turn[t] = uint16_t(turn + uint32_t(lane));
                    __syncwarp();
                    const uint32_t who = into ? S.run.turn[t] : ~0u;
                    if ((who ^ turn) < uint32_t(lane)) ++n;
                    waits = waits && who != turn + uint32_t(lane);
                    __syncwarp();
                }
                if (into) {
                    atomicAdd(&S.run.met[t], 1u);
                    place_mover(i, int(t), n);
                }
                __syncwarp();
            }
    }
    if (farCells && binLane) {
        __threadfence_block();  // (the near cells' places)
        const int4 fc = *reinterpret_cast<const int4*>(c.far.count + g0 + 4 * lane);
        const int4 head = *reinterpret_cast<const int4*>(c.far.head + g0 + 4 * lane);
        for (int k = 0; k < 4; ++k) {
            const int t = 4 * lane + k, n = k < 2 ? (k == 0 ? fc.x : fc.y) : (k == 2 ? fc.z : fc.w);
            const int h = k < 2 ? (k == 0 ? head.x : head.y) : (k == 2 ? head.z : head.w);
            if (n == 0 || n > kFarWalk) continue;
            int* seg = c.sorted + w.cellOff + S.start[t];
            const int m = S.start[t + 1] - S.start[t] - n;
            if (__any(n > 4))
                merge_far<kFarWalk>(seg, c.farLink, h, n, m);
            else
                merge_far<4>(seg, c.farLink, h, n, m);
        }
    }
}

__device__ __forceinline__ void particles_to_bins(const Ctx& c, int b, int partBlocks) {
    if (b < partBlocks) return part_scatter(c, {b, partBlocks});
    // the particles that cells emitted this step
    const int2 blk = c.cellBlocks[b - partBlocks];
    const DevWorld& w = c.worlds[blk.x];
    const int i = blk.y + int(threadIdx.x);
    if (i < w.cellOff + w.numCells) part_scatter_staged(c, w, i);
}
__global__ void k_part_scatter(Ctx c, int partBlocks) { particles_to_bins(c, int(blockIdx.x), partBlocks); }
__global__ void __launch_bounds__(kMapThreads) k_part_scan(Ctx c, int tiles) { part_scan(c, tiles); }

// The map of a step, on workgroups of one launch: the cells, the far cells, and of the particles the offsets of
// their bins (scanTiles) or, where those were found before, their places (partBlocks live ones,
// stagedBlocks the cells' emitted ones).  It opens the
// step: clears the per-step list counters and advances the worlds' timesteps if asked (a step without
// bond work has no later reader of them).
template <int kBins>
__global__ void __launch_bounds__(kMapThreads)
k_map(Ctx c, int scanTiles, int partBlocks, int stagedBlocks, int groupBlocks, int farBlocks, StepCounters* open, int advance) {
    __shared__ __align__(16) ScatterShared<kBins> S[kMapWaves];
    int b = int(blockIdx.x);
    const int tid = int(threadIdx.x), lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = int(blockDim.x) >> 6;
    if (b == 0) {
        if (tid == 0) *c.farNext.total = 0;
        if (open && tid == 0) {
            open->candidates = 0;
            open->liveParticles = 0;
        }
        if (advance)
            for (int wi = tid; wi < c.numWorlds; wi += int(blockDim.x)) c.ctr[wi].timestep += 1ull;
    }
    if (b < scanTiles) return part_scan(c, scanTiles);
    b -= scanTiles;
    if (b < groupBlocks) return cell_scatter<kBins>(c, S[wave], xcd_run(b, groupBlocks) * waves + wave, lane);
    b -= groupBlocks;
    if (b < partBlocks + stagedBlocks) return particles_to_bins(c, b, partBlocks);
    b -= partBlocks + stagedBlocks;
    if (b < farBlocks) far_scatter<kBins>(c, b * waves + wave, farBlocks * waves, lane);
}

void launch_fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t s) {
    if (n == 0) return;
    size_t g = (n + 255) / 256;
    if (g > 4096) g = 4096;
    hipLaunchKernelGGL(k_fill_u32, dim3(unsigned(g)), dim3(256), 0, s, p, v, n);
}

void launch_seed_bins(const Ctx& c, const LaunchShape& sh, hipStream_t s) {
    // no last map (every bin of it empty), every cell a far one of the coming step
    launch_fill_u32(const_cast<uint32_t*>(c.startPrev), 0u, size_t(c.numBins) + 1, s);
    launch_fill_u32(reinterpret_cast<uint32_t*>(c.far.head), uint32_t(kNone), size_t(c.numCellBins), s);
    launch_fill_u32(reinterpret_cast<uint32_t*>(c.far.count), 0u, size_t(c.numCellBins), s);
    launch_fill_u32(reinterpret_cast<uint32_t*>(c.far.group), 0u, size_t(c.numCellBins >> c.groupShift), s);
    launch_fill_u32(reinterpret_cast<uint32_t*>(c.far.total), 0u, 1, s);
    launch_fill_u32(reinterpret_cast<uint32_t*>(c.superSum), 0u, size_t((c.numCellBins >> c.groupShift) / kSuperGroups + 1), s);
    if (sh.cellBlocks) hipLaunchKernelGGL(k_cell_bin, dim3(sh.cellBlocks), dim3(sh.cellThreads), 0, s, c);
    if (c.numCellBins) hipLaunchKernelGGL(k_seed_sums, dim3(c.numCellBins / kGroupBins / 4 + 1), dim3(256), 0, s, c);
    if (sh.partBlocks) hipLaunchKernelGGL(k_part_bin, dim3(sh.partGrid), dim3(sh.partThreads), 0, s, c);
}

int map_scan_tiles(int partBins) { return (partBins + kPartScanTile - 1) / kPartScanTile; }

// The maps of a step; with `open` it also opens the step, with `advanceTimestep` the worlds' timesteps.
// The particles' takes two launches, one for their bins' offsets and one for their places.  `chain`: the
// offsets come with the cells' map, and launch_part_scatter is to follow at the head of the particles'
// chain, beside the next cell pass; otherwise the offsets come first and the places with the cells' map.
void launch_map(const Ctx& c, const LaunchShape& sh, hipStream_t s, bool chain, StepCounters* open, bool advanceTimestep) {
    const bool particles = sh.hasParticles && sh.partBlocks;
    const int tiles = particles ? map_scan_tiles(c.numBins - c.numCellBins) : 0;
    const int threads = sh.cellThreads, waves = threads / 64;
    const int blocks = c.cellCount > 0 ? ((c.numCellBins >> c.groupShift) + waves - 1) / waves : 0;
    const int groups = (blocks + kXcdCount - 1) / kXcdCount * kXcdCount;
    const int far = std::min(64 * sh.cellBlocks, kFarBlocks);
    const bool with = chain && threads == kMapThreads;  // (the scan's tiles are of kMapThreads)
    if (!with && tiles) hipLaunchKernelGGL(k_part_scan, dim3(tiles), dim3(kMapThreads), 0, s, c, tiles);
    const int scan = with ? tiles : 0, parts = particles && !chain ? sh.partGrid : 0;
    const int staged = particles && !chain && c.partStage > 0 ? sh.cellBlocks : 0;
    const auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(std::max(scan + groups + parts + staged + far, 1)), dim3(threads), 0, s, c, scan, parts,
                           staged, groups, far, open, advanceTimestep ? 1 : 0);
    };
    c.groupShift == 8 ? run(k_map<256>) : (c.groupShift == 6 ? run(k_map<64>) : run(k_map<16>));
}

void launch_part_scatter(const Ctx& c, const LaunchShape& sh, hipStream_t s) {
    if (!sh.hasParticles || !sh.partBlocks) return;
    const int staged = c.partStage > 0 ? sh.cellBlocks : 0;
    hipLaunchKernelGGL(k_part_scatter, dim3(sh.partGrid + staged), dim3(sh.cellThreads), 0, s, c, sh.partGrid);
}

}  // namespace alien
