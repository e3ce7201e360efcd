// k_neighbor.hip — the neighbour passes: fluid (SPH pressure and viscosity, overlap push, barriers, fusion
// candidates) and collision (repulsion, momentum exchange, overlap push, fusion candidates), with the
// end-of-step state of the cells that have no bonds (CellProcessor::calcFluidForces_reconnectCells_
// correctOverlap and calcCollisions_reconnectCells_correctOverlap, source/EngineGpuKernels/
// CellProcessor.cuh:122-365).
//
// The map is in logical order (cells by bin, inside a bin by previous index), so the three stencil
// bins of a cell in one bin row are one contiguous range of the map, and one wave takes 64
// consecutive map positions:
//  1. Every lane finds its three ranges, without the bins and bin rows that lie beyond its reach (the
//     squared distance to the bin's edge, in the same rounded operations as the test itself, so no
//     neighbour is lost): 5 candidates a cell instead of 9.6 at one cell per bin.
//  2. The union of the lanes' ranges, one stretch of the map per stencil row, is staged in LDS.
//  3. The lanes' lists are laid end to end and tested 64 candidates at a time, whoever they belong
//     to: a wave spends its total over 64, not its longest list.  A bit per list start tells a lane
//     its list's owner; the hits of a round, in lane order, go straight to the wave's list of pairs,
//     which is thereby ordered by owner and inside by visiting order.
//  4. The pairs are evaluated one per lane, and every owner adds its pairs' terms in visiting order
//     (the float sums of a sequential stencil walk, bit for bit).
// The pass is bound by VALU issue, so the pair terms use the short exact reciprocals and roots
// (mid_rcp, mid_sqrt; one range check per pair), indices become 32-bit byte offsets (a 64-bit
// address costs four operations), 1 / density is stored instead of the density, and sets without bond
// work run a variant without flags, bonds, barriers and fusion.
// Steps of a fluid world before (lists cut and pairs compacted per 64-candidate round, edge cells alone
// in their lanes) and now, with the map as it was: 256k cells 35 -> 26.5 us, 4M 172 -> 168 us.
// Records for all pairs of a wave in bodies (the tests ran up to five times before): 134k cells 158 -> 152
// us, with the edge waves and fewer cells per wave (kFluidShiftMin) 10751 cells 108 -> 91.5 us.
//
// Cells of the first and last bin column have a stencil that wraps around the torus: their ranges
// come in two pieces.  They are left to waves of their own, eight for a group of rows' pairs of edge bins (one row
// in small sets; the cells of a body there, one after the other, took 16 of 32 us of a small world), that take a
// cell at a time with 64 of its candidates side by side; walked alone by a lane of the pass, they were its last
// waves to end.  (With eight waves for every row, a tall world spent its time on empty ones, and more than 16 cells
// or 64 candidates were walked by a lane each: 256k cells of 64 x 8192 units, reach 2.5, a step of 340 us, 151 so;
// bodies there 117 and 96; 64k fluid cells with reach 8, 281 and 152.)
// A wave whose stretches do not fit the stage (uneven density: bodies next to empty space, drops) tests the lists of
// its first lanes; the other lanes go over their ranges by themselves, and so do all of a wave with long lists
// (dense worlds, wide reach: above 72 candidates a cell).  A list of any length fits otherwise: the tests go on
// until the pair records are full, and again after their pairs.  (When cells with more than 64 candidates and the
// lanes beyond the stage walked all nine bins, a candidate at a time: bodies 210k cells in fluid 146 -> 117 us a
// step, in collision 147 -> 124, drops of 2.7 cells a unit square 115 -> 54, a million cells at 2 a unit square, reach
// 1.3, 376 -> 147, at 1 and reach 4, 375 -> 286.)
// Collision worlds run the same pass.  In a body most neighbours are bonded, and a bonded pair adds nothing
// but a rare push, so the pairs found are first sifted (8 to 2 a cell).  The pass before walked strips of
// bin columns row by row, with the rows' halo staged again by every chunk, all nine bins tested and a list
// as long as the longest lane's: 3300 VALU operations for 64 cells of a body; now 0.84M cells in bodies 110
// -> 84 us (a step, with no copy of the cells' state in the map any more, 300 -> 260), 18k cells 25 -> 12.5
// us (85 -> 68), eight worlds of 1024^2 in one set: a step 210 -> 175 us.
#include "kernels.hpp"
#include "neighbor_device.hpp"
#include "particle_steps.hpp"

namespace alien {

// The pass's variants: fluid worlds of sets without bond work, and with; collision worlds.
enum class Pass { kFree, kBonds, kCollide };
template <Pass kPass> constexpr bool kBonded = kPass != Pass::kFree;  // (collision worlds have bonds in general)
constexpr int kFluidWaves = 4;   // waves per workgroup at most
// staged candidates of the three stencil rows: three rows of 66 bins at one cell per bin; with bonds,
// bodies of four cells a bin next to empty space
constexpr int kFreeStage = 288, kBondStage = 344;
// pair records at a time: a fluid's cells have about one each at one cell per bin; with bonds, bodies with
// ten neighbours a cell
constexpr int kFreePairs = 128, kBondPairs = 512;
// Lists longer than this in the mean are not laid out: their pairs come to one owner after the other, whose sums are
// a serial chain, and the lanes go over their ranges by themselves (walk_ranges).  Steps of fluid cells with 48 | 64 |
// 80 as the limit: 1 a unit square and reach 2.4, 223, 160 and 153 us; 0.25 and 8, 152, 152 and 153 (280 with lists);
// drops of 2.7 in sparse surroundings and reach 4, 186, 184 and 197.
constexpr int kLongLists = 72;
static_assert(64 * kLongLists + 64 <= 8192, "a bit for each candidate of a wave's lists, and of a lane without one");

// LDS of one wave: 6 KB (8 KB with bonds), six (five) waves per SIMD (the owners' velocities, densities
// and flags come from their registers, by cross-lane permutes).  With bonds, while the tests ran again for pairs
// without a record: room for 448 staged cells and 896 pairs at four waves was 1 % slower in bodies, for 288
// and 384 5 to 10 %.
template <int kStage, int kPairs> struct FluidShared {
    // staged candidates: their positions, and behind them their A indices (the last round of tests reads
    // up to 63 positions past the last list, and counts nothing there)
    float2 cpos[kStage + kStage / 2];
    __device__ int& caidx(int x) { return reinterpret_cast<int*>(cpos + kStage)[x]; }
    float2 pos[64];  // the wave's own cells; no position for a lane that does not test
    uint16_t first[64];  // each owner's first pair
    uint16_t own[64];    // pairs up to the owner's own place in its list
    uint16_t pair[kPairs];  // pair records: staged neighbour, owner << 9
    union {
        struct {
            // per list: its row boundaries (flat, two 16-bit halves) and what to add to a flat index
            // for the candidate's place, row by row
            int4 rec[64];
            uint32_t start[256];  // bit f: a list starts at flat index f
        } t;
        struct {
            float4 a[64];  // density term, overlap push, barrier (A index + 1)
            float4 b[64];  // pressure and viscosity terms
        } r;
    } u;
};
template <bool kBonds>
using FluidWave = FluidShared<kBonds ? kBondStage : kFreeStage, kBonds ? kBondPairs : kFreePairs>;
static_assert(sizeof(FluidWave<true>) <= 8000 && sizeof(FluidWave<false>) <= 6826, "20 and 24 waves per CU");
static_assert(kBondStage <= 512 && kFreeStage >= 126, "9-bit staged entries; room to read past the last list");

__device__ __forceinline__ int lanes_below(unsigned long long mask, int add) {
    return int(__builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), uint32_t(add))));
}

// the cell at map position m
__device__ __forceinline__ Nb map_nb(const Ctx& c, int m) {
    Nb o;
    o.aidx = c.sorted[m];
    o.pos = to_f2(ld32(c.A.pos, o.aidx));
    o.vel = to_f2(ld32(c.A.vel, o.aidx));
    o.dens = ld32(c.A.dens, o.aidx);
    o.flags = ld32(c.A.flags, o.aidx);
    o.lidx = m;
    return o;
}

// the terms of a pair of fluid cells (pair_term<true>, CellProcessor.cuh:144-231): a = density term,
// overlap push; b = pressure, viscosity
struct FluidTerms {
    float rho;
    f2 D, Fp, Fv;
};
template <bool kForce>
__device__ __forceinline__ FluidTerms fluid_terms(const DevParams& P, f2 pd, f2 vd, float si, float oi, bool force) {
    const float d2 = lensq(pd);
    float d = mid_sqrt(d2);
    float invD = mid_rcp(d);
    if (!mid_range(d2)) {
        d = __builtin_sqrtf(d2);
        invD = 1.0f / d;
    }
    const float q = d * P.invH;
    const float r = 2.0f - q;
    const float wNear = kTwoThirds - q * q + 0.5f * q * q * q, wFar = mid_div<6>(r * r * r);
    const float gNear = -2.0f * q + 1.5f * q * q, gFar = -0.5f * r * r;
    const bool near = q < 1.0f, far = q < 2.0f;
    FluidTerms t;
    t.rho = (near ? wNear : (far ? wFar : 0.0f)) * kKernelNorm * P.invH2;
    const float kd = (near ? gNear : (far ? gFar : 0.0f)) * kKernelNorm * P.invH3;
    t.D = {0.0f, 0.0f};
    if (d < P.minDistance) {
        const f2 p = mul(pd, P.minDistance);
        t.D = f2{mid_div<5>(p.x), mid_div<5>(p.y)};
        if (!mid_range(p.x) || !mid_range(p.y)) t.D = dvd(p, 5.0f);
    }
    t.Fp = t.Fv = f2{0.0f, 0.0f};
    const bool on = d > kNearZero && (!kForce || force);
    const f2 fp = mul(mul(mul(pd, -invD), si + oi), kd);
    // (d * d + 0.25 lies in the middle range: d is a neighbour's distance, at most 64)
    const f2 fv = mul(mul(mul(mul(vd, oi), d), kd), mid_rcp(d * d + 0.25f));
    if (on) {
        t.Fp = fp;
        t.Fv = fv;
    }
    return t;
}

// end of the pass for a cell of a set without bond work (cell_finish without bonds and barriers)
__device__ __forceinline__ void finish_free(const Ctx& c, const DevWorld& w, const DevParams& P, int k, f2 pos, f2 vel,
                                            uint32_t flags, int slot, float rho, f2 D, f2 Fp, f2 Fv, int bOld) {
    const f2 F = add(f2{0.0f, 0.0f}, add(mul(Fp, P.pressure), mul(Fv, P.viscosity)));
    const f2 pc = add(pos, D);
    f2 v = add(vel, F);
    if (lensq(v) > P.maxVelSq) v = mul(unit(v), P.maxVelocity);
    const f2 zero = {0.0f, 0.0f};
    const float dt = P.dt;
    const f2 p2 = torus_pos(add(pc, add(mul(v, dt), mul(mul(mul(zero, dt), dt), 0.5f))), w.W, w.H);
    v = add(v, mul(mul(add(zero, zero), 0.5f), dt));
    v = mul(v, 1.0f - P.friction);
    float inv = mid_rcp(rho);
    if (!mid_range(rho)) inv = 1.0f / rho;
    st32(c.B.flags, k, flags);
    st32(c.B.slot, k, slot);
    st32(c.B.dens, k, inv);
    st32(c.B.pos, k, to_float2(p2));
    st32(c.B.vel, k, to_float2(v));
    bin_next(c, w, k, p2, bOld);
}

// a cell whose stencil is walked by one lane, entry by entry
template <bool kFluid> __device__ __forceinline__ void walk_alone(const Ctx& c, int wi, int m) {
    const DevWorld& w = c.worlds[wi];
    const DevParams& P = c.params[wi];
    const uint32_t* start = c.start + w.binOff;
    const int off = w.cellOff - int(start[0]);
    const Nb s = map_nb(c, m);
    int bx, by;
    cell_bin_xy(w, s.pos, bx, by);
    atomicAdd(&c.sc->directCells, 1ull);
    cell_direct<kFluid>(c, w, P, wi, s, [&](auto&& visit) {
        for (int k = 0; k < 9; ++k) {
            const int b = wrap_small(by + k / 3 - 1, w.nby) * w.nbx + wrap_small(bx + k % 3 - 1, w.nbx);
            const int e = off + int(start[b + 1]);
            for (int j = off + int(start[b]); j < e; ++j) visit(map_nb(c, j));
        }
    });
}

// A cell of the pass whose lane goes over its ranges by itself: the map positions lo[k] on, ns[k] of each stencil
// row, with the loads of four candidates in flight.  Adds up in visiting order, as the pairs of a wave's lists do.
template <Pass kPass>
__device__ __forceinline__ void walk_ranges(const Ctx& c, const DevWorld& w, const DevParams& P, int wi, int m, int aidx, f2 pos,
                                            f2 vel, float inv, uint32_t flags, const int bt[kMaxBonds], const int lo[3],
                                            const int ns[3], bool seam, Acc& acc) {
    constexpr bool kFluid = kPass != Pass::kCollide, kBonds = kBonded<kPass>;
    constexpr int kAhead = 4;
    const float Wf = float(w.W), Hf = float(w.H);
    Nb s;
    s.pos = pos, s.vel = vel, s.dens = inv, s.flags = flags, s.aidx = aidx, s.lidx = m;
    int3 at = make_int3(lo[0], lo[1], lo[2]), n = make_int3(ns[0], ns[1], ns[2]);
#pragma unroll 1
    for (int k = 0; k < 3; ++k) {
        int x = at.x;
        const int end = x + n.x;
        at.x = at.y, at.y = at.z, n.x = n.y, n.y = n.z;
        for (; x < end; x += kAhead) {
            Nb o[kAhead];
#pragma unroll
            for (int q = 0; q < kAhead; ++q) o[q].aidx = ld32(c.sorted, uint32_t(min(x + q, end - 1)));
#pragma unroll
            for (int q = 0; q < kAhead; ++q) {
                const uint32_t a = uint32_t(o[q].aidx);
                o[q].pos = to_f2(ld32(c.A.pos, a));
                o[q].vel = to_f2(ld32(c.A.vel, a));
                if (kFluid) o[q].dens = ld32(c.A.dens, a);
                if (kBonds) o[q].flags = ld32(c.A.flags, a);
            }
#pragma unroll
            for (int q = 0; q < kAhead; ++q) {
                o[q].lidx = x + q;
                const f2 pd = stencil_delta(pos, o[q].pos, Wf, Hf, kFluid && seam);
                if (!(lensq(pd) <= P.reachSq) || x + q >= end) continue;
                if constexpr (kPass == Pass::kFree) {
                    // (the cell itself, at distance 0, adds its own density term and zeros)
                    const FluidTerms t = fluid_terms<false>(P, pd, sub(vel, o[q].vel), inv, o[q].dens, true);
                    acc.rho = acc.rho + t.rho;
                    acc.D = add(acc.D, t.D);
                    acc.Fp = add(acc.Fp, t.Fp);
                    acc.Fv = add(acc.Fv, t.Fv);
                } else {
                    if (!kFluid && x + q == m) continue;
                    float t[kPairTerms];
                    const uint32_t f = pair_term<kFluid>(c, w, P, wi, s, o[q], is_bonded(bt, o[q].aidx - w.cellOff), t, kFluid && seam,
                                                         [&] { return make_int2(m, o[q].lidx); });
                    acc_add<kFluid>(acc, f, t);
                }
            }
        }
    }
}

// The cells of the first and last bin column, in units: the last bin of row u - 1 and the first bin of row u, which
// follow each other in the map.  A group of units (edgeUnits) is shared by kEdgeWaves waves, this one number `part`, a
// cell at a time in turn, with 64 of its candidates side by side.
template <Pass kPass> __device__ __forceinline__ void edge_cells(const Ctx& c, int wi, int group, int part) {
    constexpr bool kFluid = kPass != Pass::kCollide;
    const DevWorld& w = c.worlds[wi];
    const DevParams& P = c.params[wi];
    const int lane = int(threadIdx.x) & 63;
    const uint32_t* start = c.start + w.binOff;
    const int off = w.cellOff - int(start[0]);
    const int units = kFluid ? c.edgeUnits : c.collideEdgeUnits, u = group * units + lane;
    int unitAt = 0, unitN = 0;
    if (lane < units && u <= w.nby) {
        unitAt = off + int(start[max(u * w.nbx - 1, 0)]);
        unitN = off + int(start[u < w.nby ? u * w.nbx + 1 : u * w.nbx]) - unitAt;
    }
    const int unitEnd = int(wave_inclusive_scan(uint32_t(unitN))), cells = wave_last(unitEnd);
    const float Wf = float(w.W), Hf = float(w.H), reachSq = P.reachSq;
    const float w0 = sph_w(0.0f) * P.invH2;
    for (int t = part; t < cells; t += kEdgeWaves) {
        const int k = __builtin_popcountll(__ballot(unitEnd <= t));
        const int m = t + __builtin_amdgcn_readlane(unitAt - (unitEnd - unitN), k);
        const Nb s = map_nb(c, m);  // (the same on every lane)
        int bx, by;
        cell_bin_xy(w, s.pos, bx, by);
        // lane k < 9: the stencil bin k in visiting order
        int lo = 0, n = 0;
        if (lane < 9) {
            const int b = wrap_small(by + lane / 3 - 1, w.nby) * w.nbx + wrap_small(bx + lane % 3 - 1, w.nbx);
            lo = off + int(start[b]);
            n = off + int(start[b + 1]) - lo;
        }
        const int inc = int(wave_inclusive_scan(uint32_t(n)));
        const int total = wave_last(inc);
        const bool keepSelf = kFluid && flags_barrier(s.flags);
        const int slot = c.A.slot[s.aidx];
        int bt[kMaxBonds];
        if constexpr (kPass != Pass::kFree) load_bonds(c, s, bt);
        Acc a;
        acc_init(a, s);
        auto from = [](float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
        for (int f0 = 0; f0 < total; f0 += 64) {
            // candidate f0 + lane of the list
            int at = 0;
#pragma unroll
            for (int q = 0; q < 9; ++q) {
                const int begin = __builtin_amdgcn_readlane(inc - n, q);
                at = f0 + lane >= begin ? __builtin_amdgcn_readlane(lo, q) + f0 + lane - begin : at;
            }
            const bool in = f0 + lane < total;
            Nb o = s;
            if (in) o = map_nb(c, at);
            const float d2 = lensq(kFluid ? torus_delta(s.pos, o.pos, Wf, Hf) : sub(o.pos, s.pos));
            const bool hit = in && d2 <= reachSq && (o.aidx != s.aidx || keepSelf);
            unsigned long long hits = __ballot(hit);
            // the own density term, at its place in the order (after the round's hits before it, or after all)
            const unsigned long long self = __ballot(in && o.aidx == s.aidx);
            bool pending = kFluid && !keepSelf && self != 0ull;
            const int selfAt = pending ? __builtin_ctzll(self) : 64;
            auto add_own = [&](int l) {
                if (pending && l > selfAt) {
                    a.rho = a.rho + w0;
                    pending = false;
                }
            };
            if constexpr (kPass == Pass::kFree) {
                const FluidTerms t = fluid_terms<false>(P, torus_delta(s.pos, o.pos, Wf, Hf), sub(s.vel, o.vel), s.dens, o.dens, true);
                for (; hits; hits &= hits - 1ull) {
                    const int l = __builtin_ctzll(hits);
                    add_own(l);
                    a.rho = a.rho + from(t.rho, l);
                    a.D = add(a.D, f2{from(t.D.x, l), from(t.D.y, l)});
                    a.Fp = add(a.Fp, f2{from(t.Fp.x, l), from(t.Fp.y, l)});
                    a.Fv = add(a.Fv, f2{from(t.Fv.x, l), from(t.Fv.y, l)});
                }
            } else {
                float t[kPairTerms];
#pragma unroll
                for (int v = 0; v < kPairTerms; ++v) t[v] = 0.0f;
                uint32_t f = 0u;
                if (hit)
                    f = pair_term<kFluid>(c, w, P, wi, s, o, is_bonded(bt, o.aidx - w.cellOff), t, true,
                                          [&] { return make_int2(s.lidx, o.lidx); });
                for (; hits; hits &= hits - 1ull) {
                    const int l = __builtin_ctzll(hits);
                    add_own(l);
                    float tt[kPairTerms];
#pragma unroll
                    for (int v = 0; v < kPairTerms; ++v) tt[v] = from(t[v], l);
                    acc_add<kFluid>(a, uint32_t(__builtin_amdgcn_readlane(int(f), l)), tt);
                }
            }
            add_own(65);
        }
        if (lane != 0) continue;
        if constexpr (kPass == Pass::kFree)
            finish_free(c, w, P, m, s.pos, s.vel, s.flags, slot, a.rho, a.D, a.Fp, a.Fv, by * w.nbx + bx);
        else
            cell_finish<kFluid>(c, w, P, wi, s, slot, bt, a, by * w.nbx + bx);
    }
}

// Wave v of the world: 64 (fewer in small sets, fluidShift) consecutive map positions of the first bin row, of the last one, or of those
// between (each of the three parts has its own last wave, so that no wave has lanes whose stencil rows
// are at different ends of the map).  Returns the map position that this lane is left to walk alone, or -1.
template <Pass kPass>
__device__ __forceinline__ int fluid_wave(const Ctx& c, FluidWave<kBonded<kPass>>& S, int wi, int v) {
    constexpr bool kBonds = kBonded<kPass>, kCollide = kPass == Pass::kCollide;
    constexpr int kStage = kBonds ? kBondStage : kFreeStage, kPairs = kBonds ? kBondPairs : kFreePairs;
    const int lane = int(threadIdx.x) & 63;
    // the world and its parameters are read once, before any store: read through references,
    // every use after a global store would load them again
    const DevWorld w = c.worlds[wi];
    const DevParams P = c.params[wi];
    const uint32_t* start = c.start + w.binOff;
    const int off = w.cellOff - int(start[0]);
    int m0, mEnd;
    bool seam = false;
    {
        const int r1 = int(start[w.nbx] - start[0]), r2 = int(start[(w.nby - 1) * w.nbx] - start[0]);
        const int sh = kCollide ? c.collideShift : c.fluidShift, more = (1 << sh) - 1;
        const int v1 = (r1 + more) >> sh, v2 = v1 + ((r2 - r1 + more) >> sh);
        const int at = v < v1 ? v << sh : (v < v2 ? r1 + ((v - v1) << sh) : r2 + ((v - v2) << sh));
        m0 = w.cellOff + at;
        mEnd = w.cellOff + min(at + more + 1, v < v1 ? r1 : (v < v2 ? r2 : w.numCells));
        // (in grids of at least eight bins each way, two stencil neighbours lie less than three bin edges
        // apart, less than half the world: away from the seam rows the plain difference equals the torus
        // difference bit for bit)
        // (collision pairs are tested by their plain difference, R13: no neighbours across the seam)
        if (!kCollide) seam = v < v1 || v >= v2 || w.nbx < 8 || w.nby < 8;
    }
    if ((P.motion == 0) == kCollide || m0 >= mEnd) return -1;  // (a wave past its world)
    const int m = m0 + lane;
    const bool active = m < mEnd;
    const float Wf = float(w.W), Hf = float(w.H);
    const float w0 = kCollide ? 0.0f : sph_w(0.0f) * P.invH2;  // a cell's own density term

    int aidx = 0, slot = 0;
    f2 pos = {0.0f, 0.0f}, vel = {0.0f, 0.0f};
    float inv = 0.0f;
    uint32_t flags = 0u;
    if (active) {
        aidx = ld32(c.sorted, m);
        pos = to_f2(ld32(c.A.pos, aidx));
        vel = to_f2(ld32(c.A.vel, aidx));
        if (!kCollide) inv = ld32(c.A.dens, aidx);
        flags = ld32(c.A.flags, aidx);
        slot = ld32(c.A.slot, aidx);
    }
    // the own bonds, early: the pairs ask the owners for them
    int bt[kMaxBonds];
#pragma unroll
    for (int b = 0; b < kMaxBonds; ++b)
        bt[b] = kBonds && active && b < flags_num_conn(flags) ? c.A.btgt[b * c.cellCap + aidx] : -1;
    int bx, by;
    cell_bin_xy(w, pos, bx, by);
    // (rounding may put a position on the far edge itself, which is bin 0, or it may be no number)
    const bool plain = pos.x < Wf && pos.y < Hf;
    const bool edge = bx == 0 || bx == w.nbx - 1;
    const bool mine = active && !edge;  // (edge cells belong to the edge waves)
    bool alone = mine && !plain;
    // the ranges; a bin (or bin row) next to the cell's is left out when its near edge is out of reach
    int lo[3] = {0, 0, 0}, ns[3] = {0, 0, 0};
    if (mine && !alone) {
        const float X0 = float(bx * w.binSize);
        const float l = pos.x - X0, r = pos.x - (X0 + float(w.binSize));
        const int b0 = l * l <= P.reachSq ? bx - 1 : bx, b1 = r * r <= P.reachSq ? bx + 2 : bx + 1;
        const int rows[3] = {by == 0 ? w.nby - 1 : by - 1, by, by == w.nby - 1 ? 0 : by + 1};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint32_t rb = uint32_t(rows[k] * w.nbx);
            lo[k] = off + int(ld32(start, rb + uint32_t(b0)));
            ns[k] = off + int(ld32(start, rb + uint32_t(b1))) - lo[k];
        }
    }
    // up and down rows out of reach
    if (mine && !alone) {
        const float Y0 = float(by * w.binSize);
        const float up = pos.y - Y0, down = pos.y - (by == w.nby - 1 ? Hf : Y0 + float(w.binSize));
        if (up * up > P.reachSq) ns[0] = 0;
        if (down * down > P.reachSq) ns[2] = 0;
    }
    Acc acc;
    {
        Nb self;
        self.pos = pos;
        acc_init(acc, self);
    }
    // The staged stretch of each stencil row, [u0, u0 + un): from the left bin of the first testing lane to
    // the right bin of the last one (both grow with the lane: a wave is in the torus' first bin row, in its
    // last one, or in neither).  Lists that are long in the mean are not laid out.  If the rows do not fit the
    // stage, the first lanes take what fits.  The other lanes go over their ranges each for itself, as all do
    // where fewer than 16 would fit.
    unsigned long long group = __ballot(mine && !alone);
    if (wave_last(int(wave_inclusive_scan(uint32_t(ns[0] + ns[1] + ns[2])))) > kLongLists * __builtin_popcountll(group)) group = 0ull;
    {
        const int first = group ? __builtin_ctzll(group) : 0;
        const int bxF = __builtin_amdgcn_readlane(bx, first), byF = __builtin_amdgcn_readlane(by, first);
        int u0[3], un[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            u0[k] = group ? off + int(start[wrap_small(byF + k - 1, w.nby) * w.nbx + bxF - 1]) : 0;
            un[k] = 0;
        }
        for (int keep = 64; group;) {
            const int last = 63 - __builtin_clzll(group);
            const int bxL = __builtin_amdgcn_readlane(bx, last), byL = __builtin_amdgcn_readlane(by, last);
#pragma unroll
            for (int k = 0; k < 3; ++k)
                un[k] = off + int(start[wrap_small(byL + k - 1, w.nby) * w.nbx + bxL + 2]) - u0[k];
            if (__builtin_expect(un[0] + un[1] + un[2] <= kStage, 1)) break;
            keep >>= 1;
            group &= keep >= 16 ? ((1ull << keep) - 1ull) << first : 0ull;
            if (!group) un[0] = un[1] = un[2] = 0;
        }
        const int un01 = un[0] + un[1], unAll = un01 + un[2];
        const bool tests = __builtin_amdgcn_inverse_ballot_w64(group);
        {
            const int g0 = u0[0], g1 = u0[1] - un[0], g2 = u0[2] - un01;
            constexpr int kLoads = (kStage + 63) / 64;
            int a[kLoads];
            float2 v[kLoads];
#pragma unroll
            for (int q = 0; q < kLoads; ++q) {
                const int x = lane + 64 * q;
                a[q] = x < unAll ? ld32(c.sorted, uint32_t(x + (x < un[0] ? g0 : (x < un01 ? g1 : g2)))) : 0;
            }
#pragma unroll
            for (int q = 0; q < kLoads; ++q)
                if (64 * q < unAll) v[q] = ld32(c.A.pos, uint32_t(a[q]));
#pragma unroll
            for (int q = 0; q < kLoads; ++q)
                if (lane + 64 * q < unAll) {
                    S.cpos[lane + 64 * q] = v[q];
                    S.caidx(lane + 64 * q) = a[q];
                }
        }
        S.pos[lane] = tests ? to_float2(pos) : make_float2(__builtin_nanf(""), 0.0f);
        // A lane without a list gets one entry that no test accepts, so that list k belongs to lane k.
        const int nt = tests ? ns[0] + ns[1] + ns[2] : 1;
        const int inc = int(wave_inclusive_scan(uint32_t(nt)));
        const int flat = inc - nt, flatAll = group ? wave_last(inc) : 0;
        const int selfBase = m0 - u0[1] + un[0];  // the own entry of lane 0
        // the lists' tests and pairs, as many rounds of tests at a time as there is room for their pairs
        for (int from = 0, to = 0; from < flatAll; from = to) {
            {
                int4 rec = make_int4(flat | flat << 16, -flat, -flat, -flat);
                if (tests) {
                    const int b1 = flat + ns[0], b2 = b1 + ns[1];
                    rec.x = b1 | b2 << 16 | (kPass == Pass::kBonds && flags_barrier(flags) ? int(0x80000000u) : 0);
                    rec.y = lo[0] - u0[0] - flat;
                    rec.z = lo[1] - u0[1] + un[0] - b1;
                    rec.w = lo[2] - u0[2] + un01 - b2;
                }
                S.u.t.start[lane] = 0u;
                S.u.t.start[lane + 64] = 0u;
                if (flatAll > 4096 - 64) {
                    S.u.t.start[lane + 128] = 0u;
                    S.u.t.start[lane + 192] = 0u;
                }
                S.u.t.rec[lane] = rec;
                if (!kCollide) S.own[lane] = 0xffff;
                __syncwarp();
                atomicOr(&S.u.t.start[flat >> 5], 1u << (flat & 31));
                __syncwarp();
            }
            int numPairs = 0;
            auto test = [&](auto seamTag) {
                constexpr bool kSeam = decltype(seamTag)::value;
                int owners = __builtin_popcountll(__ballot(flat < from)) - 1;  // lists that started before this round, minus one
                int f0 = from;
                for (; f0 < flatAll; f0 += 64) {
                    const uint32_t s0 = __builtin_amdgcn_readfirstlane(S.u.t.start[f0 >> 5]);
                    const uint32_t s1 = __builtin_amdgcn_readfirstlane(S.u.t.start[(f0 >> 5) + 1]);
                    const unsigned long long starts = (static_cast<unsigned long long>(s1) << 32) | s0;
                    const int owner = lanes_below(starts >> 1, owners + int(s0 & 1u));
                    owners += __builtin_popcountll(starts);
                    const int f = f0 + lane;
                    const bool in = f < flatAll;
                    const int4 rec = S.u.t.rec[owner];
                    const f2 ps = to_f2(S.pos[owner]);
                    const int b1 = rec.x & 0xffff, b2 = kBonds ? (rec.x >> 16) & 0x7fff : rec.x >> 16;
                    const int x = f + (f < b1 ? rec.y : (f < b2 ? rec.z : rec.w));
                    const f2 pn = to_f2(S.cpos[x]);
                    const float d2 = lensq(kSeam ? torus_delta(ps, pn, Wf, Hf) : sub(ps, pn));
                    // a barrier cell meets itself as a barrier neighbour; any other cell adds its own
                    // density term at its place in the visiting order, without a pair
                    const bool self = in && x == owner + selfBase;
                    const bool hit = in && d2 <= P.reachSq && (!self || (kPass == Pass::kBonds && rec.x < 0));
                    const unsigned long long hits = __ballot(hit);
                    const int rank = lanes_below(hits, numPairs);
                    if (numPairs + __builtin_popcountll(hits) > kPairs) break;
                    if (__builtin_amdgcn_inverse_ballot_w64(starts)) S.first[owner] = uint16_t(rank);
                    if (!kCollide && self) S.own[owner] = uint16_t(rank);
                    if (hit) S.pair[rank] = uint16_t(x | owner << 9);
                    numPairs += __builtin_popcountll(hits);
                }
                to = min(f0, flatAll);
            };
            if (seam)
                test(std::true_type{});
            else
                test(std::false_type{});
            __syncwarp();
            // (a list may have started before these tests, or start after them)
            int pairs0 = flat < from ? 0 : (flat < to ? S.first[lane] : numPairs);
            int pairs1 = inc < from ? 0 : (inc < to ? S.first[lane + 1] : numPairs);
            const int ownAt = kCollide || (kBonds && flags_barrier(flags)) ? -1 : S.own[lane];
            int rend = numPairs;
            if constexpr (kCollide) {
                // Most neighbours in a body are bonded, and a bonded pair adds only its overlap push (closer
                // than minDistance, not for a barrier cell): the other records go, bit 15 marks what stays of
                // the bonded ones.  (In place: a round's records land at or before their own places.)
                int kept = 0;
                const int from0 = pairs0, from1 = pairs1;
                pairs0 = pairs1 = 0;
                for (int p0 = 0; p0 < rend; p0 += 64) {
                    const int p = p0 + lane;
                    const int r = p < rend ? S.pair[p] : 0;
                    const int x = r & 0x1ff, ol = r >> 9;
                    const uint32_t sf = uint32_t(__shfl(int(flags), ol, 64));
                    bool bonded = false;
                    if (__any(p < rend && flags_num_conn(sf) > 0)) {
                        const int oa = S.caidx(x) - w.cellOff;
#pragma unroll
                        for (int b = 0; b < kMaxBonds; ++b) {
                            const int partner = __shfl(bt[b], ol, 64);  // (every lane takes part)
                            bonded = bonded || partner == oa;
                        }
                    }
                    const bool push = !flags_barrier(sf) && lensq(sub(to_f2(S.pos[ol]), to_f2(S.cpos[x]))) <= P.overlapBelowSq;
                    const bool stays = p < rend && (!bonded || push);
                    const unsigned long long m = __ballot(stays);
                    if (stays) S.pair[lanes_below(m, kept)] = uint16_t(r | (bonded ? 0x8000 : 0));
                    // the owners' first and last records move along
                    if (from0 > p0 && from0 <= p0 + 64) pairs0 = kept + __builtin_popcountll(m & (~0ull >> (p0 + 64 - from0)));
                    if (from1 > p0 && from1 <= p0 + 64) pairs1 = kept + __builtin_popcountll(m & (~0ull >> (p0 + 64 - from1)));
                    kept += __builtin_popcountll(m);
                }
                rend = kept;
                __syncwarp();
            }
            for (int p0 = 0; p0 < rend; p0 += 64) {
                // pair terms, one pair per lane
                float4 ra = make_float4(0.0f, 0.0f, 0.0f, 0.0f), rb = ra;
                const int p = p0 + lane;
                int x = 0, ol = 0, bonded = 0;  // (bonded: of a collision pair)
                if (p < rend) {
                    const int r = S.pair[p];
                    x = r & 0x1ff;
                    ol = (r >> 9) & 63;
                    bonded = r >> 15;
                }
                // the owner's state, from its registers
                const f2 sv = {__shfl(vel.x, ol, 64), __shfl(vel.y, ol, 64)};
                const float si = kCollide ? 0.0f : __shfl(inv, ol, 64);
                const f2 sp = to_f2(S.pos[ol]);
                const uint32_t sf = kBonds ? uint32_t(__shfl(int(flags), ol, 64)) : 0u;
                const int sa = kBonds ? __shfl(aidx, ol, 64) : 0;
                int sb[kMaxBonds];
                if constexpr (kPass == Pass::kBonds) {
                    // (no permutes for a round without a bonded owner)
                    if (__any(flags_num_conn(sf) > 0)) {
    #pragma unroll
                        for (int b = 0; b < kMaxBonds; ++b) sb[b] = __shfl(bt[b], ol, 64);
                    } else {
    #pragma unroll
                        for (int b = 0; b < kMaxBonds; ++b) sb[b] = -1;
                    }
                }
                if (p < rend) {
                    const int oa = S.caidx(x);
                    const f2 op = to_f2(S.cpos[x]);
                    const f2 ov = to_f2(ld32(c.A.vel, uint32_t(oa)));
                    const float oi = kCollide ? 0.0f : ld32(c.A.dens, uint32_t(oa));
                    const f2 pd = stencil_delta(sp, op, Wf, Hf, seam);
                    const f2 vd = sub(sv, ov);
                    if constexpr (kCollide) {
                        Nb s, o;
                        s.pos = sp, s.vel = sv, s.flags = sf, s.aidx = sa;
                        o.pos = op, o.vel = ov, o.flags = ld32(c.A.flags, uint32_t(oa)), o.aidx = oa;
                        float t[kPairTerms] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
                        const uint32_t f = pair_term<false>(c, w, P, wi, s, o, bonded != 0, t, false, [&] {
                            return make_int2(m0 + ol, x + (x < un[0] ? u0[0] : (x < un01 ? u0[1] - un[0] : u0[2] - un01)));
                        });
                        ra = make_float4(t[0], t[1], t[2], t[3]);
                        rb = make_float4(t[4], t[5], __int_as_float(int(f)), 0.0f);
                    } else if constexpr (!kBonds) {
                        const FluidTerms t = fluid_terms<false>(P, pd, vd, si, oi, true);
                        ra = make_float4(t.rho, t.D.x, t.D.y, 0.0f);
                        rb = make_float4(t.Fp.x, t.Fp.y, t.Fv.x, t.Fv.y);
                    } else {
                        const uint32_t of = ld32(c.A.flags, uint32_t(oa));
                        if (flags_barrier(of)) {
                            ra.x = len2(pd);
                            ra.w = __int_as_float(oa + 1);
                        } else {
                            const bool bonded = is_bonded(sb, oa - w.cellOff);
                            const int nc = flags_num_conn(sf);
                            const bool bari = flags_barrier(sf);
                            const FluidTerms t = fluid_terms<true>(P, pd, vd, si, oi, !bonded);
                            ra = make_float4(t.rho, bari ? 0.0f : t.D.x, bari ? 0.0f : t.D.y, 0.0f);
                            rb = make_float4(t.Fp.x, t.Fp.y, t.Fv.x, t.Fv.y);
                            if (!bonded && !bari && nc < flags_max_conn(sf) && flags_num_conn(of) < flags_max_conn(of) &&
                                lensq(vd) > P.fusionBelowSq) {
                                const int sl = m0 + ol, olx = x + (x < un[0] ? u0[0] : (x < un01 ? u0[1] - un[0] : u0[2] - un01));
                                if (sl < olx) {
                                    const float ei = c.energy[w.cellOff + c.A.slot[sa]];
                                    const float ej = c.energy[w.cellOff + c.A.slot[oa]];
                                    if (ei <= P.maxBindingEnergy && ej <= P.maxBindingEnergy) push_candidate(c, sl, olx, wi);
                                }
                            }
                        }
                    }
                }
                __syncwarp();  // (the test's records, and the round before, are done with)
                S.u.r.a[lane] = ra;
                S.u.r.b[lane] = rb;
                __syncwarp();
                // every owner adds its pairs of this round in visiting order; terms a pair does not have
                // are zero, which leaves a sum that started at +0 unchanged bit for bit
                const int j1 = min(pairs1, min(p0 + 64, rend));
                for (int j = max(pairs0, p0); j < j1; ++j) {
                    const float4 ta = S.u.r.a[j - p0], tb = S.u.r.b[j - p0];
                    if constexpr (kCollide) {
                        acc_add_collision(acc, uint32_t(__float_as_int(tb.z)), f2{ta.x, ta.y}, f2{ta.z, ta.w}, f2{tb.x, tb.y});
                        continue;
                    }
                    acc.rho = j == ownAt ? acc.rho + w0 : acc.rho;
                    if constexpr (kBonds) {
                        // of the barrier neighbours only the first ten count, and of those the first
                        // nearest one (CellProcessor.cuh:234-246)
                        const bool bar = __float_as_int(ta.w) != 0;
                        const bool nearest = bar && acc.numBarrier < 10 && (acc.cb < 0 || ta.x < acc.cbDist);
                        acc.cb = nearest ? __float_as_int(ta.w) - 1 : acc.cb;
                        acc.cbDist = nearest ? ta.x : acc.cbDist;
                        acc.numBarrier += bar ? 1 : 0;
                        acc.rho = bar ? acc.rho : acc.rho + ta.x;
                    } else {
                        acc.rho = acc.rho + ta.x;
                    }
                    acc.D = add(acc.D, f2{ta.y, ta.z});
                    acc.Fp = add(acc.Fp, f2{tb.x, tb.y});
                    acc.Fv = add(acc.Fv, f2{tb.z, tb.w});
                }
            }
            if (!kCollide && tests && ownAt == pairs1) acc.rho = acc.rho + w0;  // the own term after all pairs
            __syncwarp();
        }
    }
    const bool walks = mine && !alone && !__builtin_amdgcn_inverse_ballot_w64(group);
    if (__builtin_expect(__any(walks), 0)) {
        const unsigned long long all = __ballot(walks);
        // (counted here: after a store the compiler would read the map's offsets through the vector path)
        if (lane == 0) {
            atomicAdd(&c.sc->fallbackChunks, 1ull);
            atomicAdd(&c.sc->directCells, (unsigned long long)(__builtin_popcountll(all)));
        }
        if (walks) walk_ranges<kPass>(c, w, P, wi, m, aidx, pos, vel, inv, flags, bt, lo, ns, seam, acc);
    }
    if (!mine) return -1;
    if (alone) return m;
    const int bOld = by * w.nbx + bx;
    if constexpr (kBonds) {
        Nb self;
        self.pos = pos;
        self.vel = vel;
        self.dens = inv;
        self.flags = flags;
        self.aidx = aidx;
        self.lidx = m;
        cell_finish<!kCollide>(c, w, P, wi, self, slot, bt, acc, bOld);
    } else {
        finish_free(c, w, P, m, pos, vel, flags, slot, acc.rho, acc.D, acc.Fp, acc.Fv, bOld);
    }
    return -1;
}

// With bonds also a stage of the particles' chain, on the launch's first workgroups (sets with bond work):
// their bin sort, or with the late chain their scatter
template <Pass kPass>
__global__ void __launch_bounds__(64 * kFluidWaves) __attribute__((amdgpu_waves_per_eu(kBonded<kPass> ? 5 : 6)))
k_neighbor(Ctx c, int partBlocks, int late, int edgeBlocks, int tableBlocks) {
    constexpr bool kBonds = kBonded<kPass>, kFluid = kPass != Pass::kCollide;
    __shared__ FluidWave<kBonds> SS[kFluidWaves];
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    int block = int(blockIdx.x);
    if constexpr (kBonds) {
        if (block < partBlocks)
            return late ? part_scatter(c, {block, partBlocks}) : part_binsort(c, {block, partBlocks});
        block -= partBlocks;
    }
    if (block < edgeBlocks) {
        const int2 blk = (kFluid ? c.edgeBlocks : c.collideEdgeBlocks)[block];
        const int wi = blk.x;
        edge_cells<kPass>(c, wi, (blk.y + wave) / kEdgeWaves, (blk.y + wave) % kEdgeWaves);
        return;
    }
    block -= edgeBlocks;
    // XCD-aware: workgroup b runs on XCD b % 8, which sweeps one contiguous band of the map, so the
    // stencil rows its waves share stay in its L2
    const int per = (tableBlocks + kXcdCount - 1) / kXcdCount;
    const int e = (block % kXcdCount) * per + block / kXcdCount;
    if (e >= tableBlocks) return;
    const int2 blk = (kFluid ? c.fluidBlocks : c.collideBlocks)[e];
    const int m = fluid_wave<kPass>(c, SS[wave], blk.x, blk.y + wave);
    // (rare: its parameters are read again, so that the waves above do not carry them)
    if (m >= 0) walk_alone<kFluid>(c, blk.x, m);
}

// The particles' stage goes with the first launch.  A set with collision worlds but no bond work at all still
// runs the one collision variant.
void launch_neighbor(const Ctx& c, const LaunchShape& sh, hipStream_t s, bool withParticles) {
    int parts = withParticles && sh.hasParticles && sh.partBlocks ? (sh.lateParticles ? sh.partGrid : sh.pbinBlocks) : 0;
    const int late = sh.lateParticles ? 1 : 0;
    const auto grid = [&](int edges, int table) {
        return dim3(parts + edges + (table + kXcdCount - 1) / kXcdCount * kXcdCount);
    };
    const dim3 threads(sh.cellThreads);
    if (sh.collideBlocks) {
        hipLaunchKernelGGL(k_neighbor<Pass::kCollide>, grid(sh.collideEdgeBlocks, sh.collideBlocks), threads, 0, s, c, parts, late,
                           sh.collideEdgeBlocks, sh.collideBlocks);
        parts = 0;
    }
    if (sh.hasBondWork && (sh.fluidBlocks || parts))
        hipLaunchKernelGGL(k_neighbor<Pass::kBonds>, grid(sh.edgeBlocks, sh.fluidBlocks), threads, 0, s, c, parts, late,
                           sh.edgeBlocks, sh.fluidBlocks);
    else if (sh.fluidBlocks)
        hipLaunchKernelGGL(k_neighbor<Pass::kFree>, grid(sh.edgeBlocks, sh.fluidBlocks), threads, 0, s, c, 0, 0, sh.edgeBlocks,
                           sh.fluidBlocks);
}

}  // namespace alien
