// k_neighbor.hip — the collision neighbour pass, and the launch of both passes.
//
// One wave owns a strip of bin columns and walks it row by row (see "Row streaming" below).  Per
// row it (1) tests the 3x3 bin stencil of every cell with the neighbour predicate on squared
// lengths and records the neighbours as a bit mask in visiting order, (2) evaluates all neighbour
// pairs of the row one pair per lane, and (3) lets every cell add its pairs' terms in visiting
// order, which gives the float sums of a sequential stencil walk bit for bit.  A cell with more
// than 64 stencil candidates, or a strip whose rows do not fit LDS, walks its stencil
// sequentially instead (same order, same results).  A workgroup of a fluid world exits at once.
#include <type_traits>

#include "kernels.hpp"
#include "neighbor_device.hpp"
#include "particle_steps.hpp"

namespace alien {

// ---------------------------------------------------------------------------------------------
// Row streaming.  A workgroup (one wave) owns a strip of up to kStripMax bin columns and a chunk of
// staged rows, and walks them top to bottom with staged rows Y-1, Y, Y+1 in LDS.  A staged row is
// kSub consecutive bin rows (1, or 2 for sparse worlds, so that one pass has enough cells for the
// 64 lanes); each bin row covers the strip plus one halo column on each side, its entries stored
// bin by bin in rank order (R1), so the three stencil bins of a cell in one bin row are one
// contiguous range.  While row Y is computed, the entries of row Y+2 and the bin counters of row
// Y+3 are on their way into registers; row Y+2 is committed once row Y-1 is no longer needed.  The
// three staged rows share one ring pool of entries (positions counted up without wrapping, stored
// modulo kPool): a row takes the pool space right after the previous one, so any three
// consecutive rows of up to kPool entries together fit, however they are distributed.
// ---------------------------------------------------------------------------------------------
constexpr int kRowBins = kStripMax + 2;            // halo columns of one bin row
constexpr int kSubMax = 2;                         // bin rows per staged row, at most
constexpr int kPool = kRowPool;
constexpr int kPoolMask = kPool - 1;
constexpr int kPairCap = 128;  // pair records per evaluation window
constexpr int kPosMirror = 64;
static_assert((kPool & kPoolMask) == 0 && kPool <= 256, "pair records keep an 8-bit pool position");
static_assert(kRowCap <= 2 * kRowThreads, "a row in flight holds at most two entries per lane");
static_assert(kSubMax * kRowBins <= 3 * kRowThreads && kSubMax * kRowBins < 256,
              "bin slots: three per lane, 8-bit ids");

// LDS of one wave, for staged rows of up to kMaxSub bin rows
template <int kMaxSub>
struct RowShared {
    static constexpr int kStageBins = kMaxSub * kRowBins;  // bin slots of one staged row (row major)
    // per ring row: pool position of the first entry of every bin slot, then the end; per ring
    // row and bin row, map positions of the first entries of the left halo bin, the first interior
    // bin and the right halo bin (the interior bins of a bin row are contiguous in the map)
    int rs[3][kStageBins + 1];
    int rm[3][kMaxSub][3];
    // entries of the staged rows, by pool position modulo kPool; positions 0..kPosMirror-1 are
    // repeated after the end so that a stencil range of up to 64 entries reads without wrapping
    float2 pos[kPool + kPosMirror];
    float2 vel[kPool];
    uint16_t flags[kPool];  // the bits the pass reads of an entry's flags (flags16)
    int aidx[kPool];
    uint8_t sbin[kPool];  // bin slot: bin row * HX + halo column
    // the row in flight
    int nrs[kStageBins + 1];
    int nrm[kMaxSub][3];
    uint8_t nebin[kRowCap];  // entry of the row -> bin slot
    union {
        struct {
            // while a row is computed, the pair records of the current window: the cell's pool
            // position, and the neighbour as bonded << 15 | ring row << 8 | pool position
            uint8_t pself[kPairCap];
            uint16_t pnb[kPairCap];
        } pr;
    } u;
};

// registers of a row in flight: bin counters of the bin slots lane, lane + 64, lane + 128, then
// the entries lane and lane + 64 in map order
template <int kSub>
struct RowFlight {
    static constexpr int kSlots = kSub == 2 ? 3 : 2;  // bin slots per lane
    uint32_t s0[kSlots], s1[kSlots];
    int aidx[2];
    float2 pos[2], vel[2];
    uint32_t flags[2];
    int total;
};

struct StripGeom {
    int x0, IX, HX;  // first interior bin column, interior columns, halo columns (IX + 2)
    int nbx, nby, binOff, cellOff;
    uint32_t base;   // start[] value of the world's first bin
    bool seam;       // the staged rows or columns wrap around the torus
};

// map segment of halo column hx: 0 the left halo bin, 1 the interior, 2 the right halo bin; and
// the segment's first halo column
__device__ __forceinline__ int seg_of(int hx, int HX) { return hx == 0 ? 0 : (hx == HX - 1 ? 2 : 1); }
__device__ __forceinline__ int seg_first(int seg, int HX) { return seg == 0 ? 0 : (seg == 2 ? HX - 1 : 1); }

// bin row (0 or 1) of bin slot j
template <int kSub>
__device__ __forceinline__ int slot_row(int j, int HX) { return kSub == 2 && j >= HX ? 1 : 0; }

// An entry's flags in LDS: bond counts (bits 0..7) and the barrier bit (moved to bit 8), the only
// bits the pass reads of a neighbour; a cell's own full flags are read again before its writes.
__device__ __forceinline__ uint16_t flags16(uint32_t f) { return uint16_t((f & 0xFFu) | ((f & kBarrierBit) >> 8)); }
__device__ __forceinline__ uint32_t flags32(uint16_t p) { return (uint32_t(p) & 0xFFu) | ((uint32_t(p) & 0x100u) << 8); }

// logical index of the staged entry at pool position pp (already reduced modulo kPool) of ring row r
template <int kSub, class RS>
__device__ __forceinline__ int row_lidx(const RS& S, const StripGeom& g, int r, int pp) {
    const int j = S.sbin[pp];
    const int t = slot_row<kSub>(j, g.HX);
    const int seg = seg_of(j - t * g.HX, g.HX);
    return S.rm[r][t][seg] + ((pp - S.rs[r][t * g.HX + seg_first(seg, g.HX)]) & kPoolMask);
}

// the staged entry at pool position pp of ring row r; without its logical index if !kLidx
template <int kSub, class RS, bool kLidx = true>
__device__ __forceinline__ Nb row_nb(const RS& S, const StripGeom& g, int r, int pp) {
    Nb o;
    o.pos = to_f2(S.pos[pp]);
    o.vel = to_f2(S.vel[pp]);
    o.dens = 0.0f;
    o.flags = flags32(S.flags[pp]);
    o.aidx = S.aidx[pp];
    o.lidx = kLidx ? row_lidx<kSub>(S, g, r, pp) : -1;
    return o;
}

template <bool kFluid>
__device__ __forceinline__ Nb global_nb(const Ctx& c, int a, int l) {
    Nb o;
    o.pos = to_f2(c.A.pos[a]);
    o.vel = to_f2(c.A.vel[a]);
    o.dens = kFluid ? c.A.dens[a] : 0.0f;
    o.flags = c.A.flags[a];
    o.aidx = a;
    o.lidx = l;
    return o;
}

// bin of halo column hx in bin row yy (both wrapped around the torus)
__device__ __forceinline__ int strip_bin(const StripGeom& g, int yy, int hx) {
    return g.binOff + wrap_small(yy, g.nby) * g.nbx + wrap_small(g.x0 - 1 + hx, g.nbx);
}

// A: bin counters of staged row Y
template <int kSub>
__device__ __forceinline__ void row_issue_counts(const Ctx& c, const StripGeom& g, int Y, RowFlight<kSub>& F) {
    const int lane = threadIdx.x;
#pragma unroll
    for (int q = 0; q < RowFlight<kSub>::kSlots; ++q) {
        const int j = lane + q * kRowThreads;
        F.s0[q] = F.s1[q] = 0u;
        if (j < kSub * g.HX) {
            const int t = slot_row<kSub>(j, g.HX);
            const int gb = strip_bin(g, kSub * Y + t, j - t * g.HX);
            F.s0[q] = c.start[gb];
            F.s1[q] = c.start[gb + 1];
        }
    }
}

// B: slots of the row's bins, then the entry loads (map-order copy, contiguous per bin)
template <int kSub, class RS>
__device__ __forceinline__ void row_issue_entries(const Ctx& c, const StripGeom& g, RS& S, RowFlight<kSub>& F) {
    constexpr int kSlots = RowFlight<kSub>::kSlots;
    const int lane = threadIdx.x;
    const int SB = kSub * g.HX;
    int n[kSlots], inc[kSlots];
#pragma unroll
    for (int q = 0; q < kSlots; ++q) {
        n[q] = lane + q * kRowThreads < SB ? int(F.s1[q] - F.s0[q]) : 0;
        inc[q] = int(wave_inclusive_scan(uint32_t(n[q])));
    }
    const int tot0 = wave_last(inc[0]), tot1 = wave_last(inc[1]);
    F.total = tot0 + tot1 + (kSlots > 2 ? wave_last(inc[kSlots - 1]) : 0);
#pragma unroll
    for (int q = 0; q < kSlots; ++q) {
        const int j = lane + q * kRowThreads;
        if (j >= SB) continue;
        const int off = inc[q] - n[q] + (q >= 1 ? tot0 : 0) + (q >= 2 ? tot1 : 0);
        const int t = slot_row<kSub>(j, g.HX);
        const int hx = j - t * g.HX;
        S.nrs[j] = off;
        if (hx <= 1 || hx == g.HX - 1) S.nrm[t][seg_of(hx, g.HX)] = g.cellOff + int(F.s0[q] - g.base);
        for (int e = 0; e < n[q]; ++e) S.nebin[off + e] = uint8_t(j);
    }
    if (lane == 0) S.nrs[SB] = F.total;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int e = lane + q * kRowThreads;
        if (e < F.total) {
            const int j = S.nebin[e];
            const int t = slot_row<kSub>(j, g.HX);
            const int seg = seg_of(j - t * g.HX, g.HX);
            const int m = S.nrm[t][seg] + (e - S.nrs[t * g.HX + seg_first(seg, g.HX)]);
            F.aidx[q] = c.sorted[m];
            F.pos[q] = c.mpos[m];
            F.vel[q] = c.mvel[m];
            F.flags[q] = c.mflags[m];
        }
    }
}

// C: the row into ring row r at pool position head.  The row was read from the map copy bin by
// bin, and the map holds every bin's cells by previous index (R1): an entry's place in the row is
// its rank in its bin.
template <int kSub, class RS>
__device__ __forceinline__ void row_commit(const StripGeom& g, RS& S, const RowFlight<kSub>& F, int r, int head) {
    const int lane = threadIdx.x;
    const int SB = kSub * g.HX;
    for (int i = lane; i <= SB; i += kRowThreads) S.rs[r][i] = head + S.nrs[i];
    if (lane < 3 * kSub) S.rm[r][lane / 3][lane % 3] = S.nrm[lane / 3][lane % 3];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int e = lane + q * kRowThreads;
        if (e < F.total) {
            const int j = S.nebin[e];
            const int a = F.aidx[q];
            const int pp = (head + e) & kPoolMask;
            S.pos[pp] = F.pos[q];
            if (pp < kPosMirror) S.pos[kPool + pp] = F.pos[q];
            S.vel[pp] = F.vel[q];
            S.flags[pp] = flags16(F.flags[q]);
            S.aidx[pp] = a;
            S.sbin[pp] = uint8_t(j);
        }
    }
    __syncthreads();
}

// element r (0..2) of a three-element register array, without indexing it at run time (which
// would place the array in scratch memory)
__device__ __forceinline__ int pick3(const int (&a)[3], int r) { return r == 0 ? a[0] : (r == 1 ? a[1] : a[2]); }

// The cells of staged row Y (ring row rc; rows Y-1 and Y+1 in rm_ and rp).
template <bool kFluid, int kSub, class RS>
__device__ __forceinline__ void row_compute(const Ctx& c, const DevWorld& w, const DevParams& P, int wi,
                                            const StripGeom& g, RS& S, int rm_, int rc, int rp) {
    const int lane = threadIdx.x;
    const float Wf = float(w.W), Hf = float(w.H);
    // the cells: the interior bins of each bin row of the staged row
    const int cs0 = S.rs[rc][1];
    const int n0 = S.rs[rc][g.IX + 1] - cs0;
    const int cs1 = kSub == 2 ? S.rs[rc][g.HX + 1] : 0;
    const int ncell = n0 + (kSub == 2 ? S.rs[rc][g.HX + g.IX + 1] - cs1 : 0);
    const float w0 = kFluid ? sph_w(0.0f) * P.invH2 : 0.0f;  // a fluid cell's own density term
    for (int q0 = 0; q0 < ncell; q0 += kRowThreads) {
        // candidates of this lane's cell: three contiguous pool ranges, one per stencil bin row
        const int q = q0 + lane;
        const bool active = q < ncell;
        Nb self;
        int bt[kMaxBonds];
        int a0s[3] = {0, 0, 0}, ns[3] = {0, 0, 0}, ringOf[3] = {rm_, rc, rp};
        unsigned long long mask = 0ull, bmask = 0ull;
        bool direct = false;
        int selfIdx = -1;  // fluid: number of the cell's pairs that come before its own density term
        const int t = kSub == 2 && q >= n0 ? 1 : 0;    // the cell's bin row in the staged row
        const int su = t == 0 ? cs0 + q : cs1 + (q - n0);  // pool position, not wrapped
        const int sp = su & kPoolMask;
        int slot = 0;
        if (active) {
            self = row_nb<kSub>(S, g, rc, sp);
            slot = c.A.slot[self.aidx];  // needed only at the end: loaded early
            load_bonds(c, self, bt);
            const int hx = S.sbin[sp] - t * g.HX;
            // stencil bin rows (ring row, bin row): above, own, below
            int subOf[3] = {0, 0, 0};
            if (kSub == 2) {
                ringOf[0] = t == 0 ? rm_ : rc;
                subOf[0] = t == 0 ? 1 : 0;
                ringOf[1] = rc;
                subOf[1] = t;
                ringOf[2] = t == 0 ? rc : rp;
                subOf[2] = t == 0 ? 1 : 0;
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const int b0 = subOf[k] * g.HX + hx;
                a0s[k] = S.rs[ringOf[k]][b0 - 1];
                ns[k] = S.rs[ringOf[k]][b0 + 2] - a0s[k];
            }
            if (ns[0] + ns[1] + ns[2] > 64) {
                direct = true;
            } else {
                const bool hasBonds = flags_num_conn(self.flags) > 0;
                // fluid: the cell's own density term needs no pair evaluation; only its place in
                // the visiting order is kept (a barrier cell meets itself as a barrier instead);
                // collision: the cell is not its own neighbour
                const bool keepSelf = kFluid && flags_barrier(self.flags);
                const int selfFlat = ns[0] + (su - a0s[1]);  // the cell's own visiting index
                // predicated tests, one mask bit per candidate in visiting order (one copy of the
                // loop for chunks on the torus seam, one for the rest)
                auto test = [&](auto seamTag) {
                    constexpr bool kSeam = decltype(seamTag)::value;
                    auto dsq = [&](f2 o) {
                        return kFluid ? lensq(kSeam ? torus_delta(self.pos, o, Wf, Hf) : sub(self.pos, o))
                                      : lensq(sub(o, self.pos));  // R13
                    };
                    int cidx = 0;
#pragma unroll
                    for (int r = 0; r < 3; ++r) {
                        const int pb = a0s[r] & kPoolMask, n = ns[r];
                        unsigned long long rowMask = 0ull;
                        for (int u = 0; u < n; u += 2) {
                            // two candidates per iteration; the second is read even past the
                            // range end (within the mirrored pool) and trimmed below
                            const f2 p0 = to_f2(S.pos[pb + u]);
                            const f2 p1 = to_f2(S.pos[pb + u + 1]);
                            rowMask |= dsq(p0) <= P.reachSq ? (1ull << u) : 0ull;
                            rowMask |= dsq(p1) <= P.reachSq ? (2ull << u) : 0ull;
                        }
                        rowMask &= n >= 64 ? ~0ull : (1ull << n) - 1ull;
                        mask |= rowMask << cidx;
                        cidx += n;
                    }
                };
                if (g.seam)
                    test(std::true_type{});
                else
                    test(std::false_type{});
                if (!keepSelf) mask &= ~(1ull << selfFlat);
                if (kFluid && !keepSelf) selfIdx = __builtin_popcountll(mask & ((1ull << selfFlat) - 1ull));
                if (hasBonds) {
                    // which of the neighbours are bonded
                    const bool bari = flags_barrier(self.flags);
                    unsigned long long m = mask;
                    while (m) {
                        const int ci = __builtin_ctzll(m);
                        m &= m - 1ull;
                        const int r = ci < ns[0] ? 0 : (ci < ns[0] + ns[1] ? 1 : 2);
                        const int rest = ci - (r == 0 ? 0 : (r == 1 ? ns[0] : ns[0] + ns[1]));
                        const int np = (pick3(a0s, r) + rest) & kPoolMask;
                        if (!is_bonded(bt, S.aidx[np] - w.cellOff)) continue;
                        if constexpr (!kFluid) {
                            // a bonded collision pair adds only its overlap push (closer than
                            // minDistance, not for a barrier cell): otherwise it adds nothing and
                            // leaves the list (the distance as the pair term takes it)
                            const f2 o = to_f2(S.pos[np]);
                            const float d2 = lensq(g.seam ? torus_delta(self.pos, o, Wf, Hf) : sub(self.pos, o));
                            if (bari || d2 > P.overlapBelowSq) {
                                mask &= ~(1ull << ci);
                                continue;
                            }
                        }
                        bmask |= 1ull << ci;
                    }
                }
            }
        }
        const int count = __builtin_popcountll(mask);
        const int inc = int(wave_inclusive_scan(uint32_t(count)));
        const int numPairs = wave_last(inc);
        const int pbase = inc - count;

        Acc a;
        if (active) acc_init(a, self);
        for (int W0 = 0; W0 < numPairs; W0 += kPairCap) {
            const int wend = min(numPairs, W0 + kPairCap);
            // owners write the records of their pairs inside this window
            if (count > 0 && pbase < wend && pbase + count > W0) {
                unsigned long long m = mask;
                for (int p = pbase; m; ++p) {
                    const int ci = __builtin_ctzll(m);
                    m &= m - 1ull;
                    if (p < W0 || p >= wend) continue;
                    int r = 0, rest = ci;
                    if (rest >= ns[0]) {
                        rest -= ns[0];
                        r = 1;
                        if (rest >= ns[1]) {
                            rest -= ns[1];
                            r = 2;
                        }
                    }
                    const int np = (pick3(a0s, r) + rest) & kPoolMask;
                    const uint32_t bonded = uint32_t((bmask >> ci) & 1ull);
                    S.u.pr.pself[p - W0] = uint8_t(sp);
                    S.u.pr.pnb[p - W0] = uint16_t((bonded << 15) | (uint32_t(pick3(ringOf, r)) << 8) | uint32_t(np));
                }
            }
            __syncthreads();
            for (int off = W0; off < wend; off += kRowThreads) {
                // pair terms, one pair per lane
                const int p = off + lane;
                float tm[kPairTerms];
#pragma unroll
                for (int v = 0; v < kPairTerms; ++v) tm[v] = 0.0f;
                uint32_t f = 0u;
                if (p < wend) {
                    const uint32_t rec = S.u.pr.pnb[p - W0];
                    const int ps = S.u.pr.pself[p - W0], ro = int((rec >> 8) & 3u), po = int(rec & 0xFFu);
                    const Nb s = row_nb<kSub, RS, false>(S, g, rc, ps);
                    const Nb o = row_nb<kSub, RS, false>(S, g, ro, po);
                    f = pair_term<kFluid>(c, w, P, wi, s, o, (rec >> 15) != 0u, tm, g.seam, [&] {
                        return make_int2(row_lidx<kSub>(S, g, rc, ps), row_lidx<kSub>(S, g, ro, po));
                    });
                }
                // the owner adds its pairs of this round in visiting order, reading each from the
                // lane that evaluated it (every lane takes part in every exchange)
                const int lo = max(pbase, off), hi = min(pbase + count, min(off + kRowThreads, wend));
                const int n = count > 0 ? max(0, hi - lo) : 0;
                for (int j = 0; __any(j < n); ++j) {
                    const int src = (lo + j - off) & (kRowThreads - 1);
                    float tt[kPairTerms];
#pragma unroll
                    for (int v = 0; v < kPairTerms; ++v) tt[v] = __shfl(tm[v], src, kRowThreads);
                    const uint32_t ff = uint32_t(__shfl(int(f), src, kRowThreads));
                    const bool on = j < n;
                    if constexpr (kFluid) a.rho = on && lo + j - pbase == selfIdx ? a.rho + w0 : a.rho;
                    acc_add_sel<kFluid>(a, on, ff, tt);
                }
            }
            __syncthreads();
        }
        if (active && selfIdx == count) a.rho = a.rho + w0;  // the own term after all pairs
        if (active) {
            // the cell's full flags, from the start-of-step arrays (the map copy holds a bin's
            // entries in arrival order, not at their logical indices)
            self.flags = c.A.flags[self.aidx];
            if (direct) {
                atomicAdd(&c.sc->directCells, 1ull);
                cell_direct<kFluid>(c, w, P, wi, self, [&](auto&& visit) {
#pragma unroll
                    for (int r = 0; r < 3; ++r)
                        for (int u = a0s[r]; u < a0s[r] + ns[r]; ++u)
                            visit(row_nb<kSub>(S, g, ringOf[r], u & kPoolMask));
                });
            } else {
                // the bond targets are loaded again rather than kept in registers through the pair
                // work (few cells have bonds in a fluid world; the loads hit the cache)
                int bt2[kMaxBonds];
                load_bonds(c, self, bt2);
                cell_finish<kFluid>(c, w, P, wi, self, slot, bt2, a);
            }
        }
    }
}

// A chunk with a row too dense for LDS: every cell walks its stencil in global memory, entries of
// a bin by increasing previous index (selection over the bin), same order and results.
template <bool kFluid>
__device__ __forceinline__ void rows_direct(const Ctx& c, const DevWorld& w, const DevParams& P, int wi, const StripGeom& g, int y0,
                            int IY) {
    const uint32_t base = g.base;
    auto binRange = [&](int gb, int& s0, int& n) {
        s0 = g.cellOff + int(c.start[gb] - base);
        n = int(c.start[gb + 1] - c.start[gb]);
    };
    for (int y = y0; y < y0 + IY; ++y) {
        const int rowFirst = g.binOff + y * g.nbx + g.x0;
        const int m0 = g.cellOff + int(c.start[rowFirst] - base);
        const int m1 = g.cellOff + int(c.start[rowFirst + g.IX] - base);
        for (int m = m0 + int(threadIdx.x); m < m1; m += kRowThreads) {
            // the bin of map position m: the last bin of the row segment starting at or before m
            int lo = 0, hi = g.IX;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (g.cellOff + int(c.start[rowFirst + mid] - base) <= m)
                    lo = mid;
                else
                    hi = mid;
            }
            const int hx = lo + 1;
            // (the map holds every bin's cells by previous index: a cell's logical index is its map
            // position)
            const int i = c.sorted[m];
            const Nb self = global_nb<kFluid>(c, i, m);
            cell_direct<kFluid>(c, w, P, wi, self, [&](auto&& visit) {
                for (int dy = -1; dy <= 1; ++dy)
                    for (int dx = -1; dx <= 1; ++dx) {
                        int s0, n;
                        binRange(strip_bin(g, y + dy, hx + dx), s0, n);
                        for (int t = 0; t < n; ++t) visit(global_nb<kFluid>(c, c.sorted[s0 + t], s0 + t));
                    }
            });
        }
    }
}

// Whether staged rows y0-1 .. y0+IY (kSub bin rows each) each fit a row in flight and every three
// consecutive ones the pool (the same answer on every lane).
template <int kSub>
__device__ __forceinline__ bool stage_fits(const Ctx& c, const StripGeom& g, int y0, int IY) {
    const int lane = threadIdx.x;
    int total = 0;
    if (lane < IY + 2) {
        const int Y = y0 - 1 + lane;
#pragma unroll
        for (int t = 0; t < kSub; ++t) {
            const int yy = kSub * Y + t;
            const int rowFirst = g.binOff + wrap_small(yy, g.nby) * g.nbx + g.x0;
            total += int(c.start[rowFirst + g.IX] - c.start[rowFirst]);
            const int gl = strip_bin(g, yy, 0), gr = strip_bin(g, yy, g.IX + 1);
            total += int(c.start[gl + 1] - c.start[gl]) + int(c.start[gr + 1] - c.start[gr]);
        }
    }
    const int three = total + __shfl_down(total, 1, kRowThreads) + __shfl_down(total, 2, kRowThreads);
    return !__any(total > kRowCap || (lane < IY && three > kPool));
}

// One chunk of IY staged rows from staged row y0 (kSub bin rows each); false (and nothing done)
// when its staged rows do not fit the LDS.
template <bool kFluid, int kSub, class RS>
__device__ __forceinline__ bool chunk_rows(const Ctx& c, const DevWorld& w, const DevParams& P, int wi,
                                           StripGeom& g, RS& S, int y0, int IY) {
    const int nbyS = g.nby / kSub;
    // Away from the seam no staged bin wraps, and two stencil neighbours lie less than three bin
    // edges apart (the last column and row absorb less than one edge of remainder) while half the
    // world is at least four: the torus difference is the plain difference there, bit for bit.
    g.seam = g.x0 == 0 || g.x0 + g.IX >= g.nbx || y0 == 0 || y0 + IY >= nbyS || g.nbx < 8 || g.nby < 8;
    if (!stage_fits<kSub>(c, g, y0, IY)) return false;

    RowFlight<kSub> F, G;
    int head = 0;  // pool position of the next committed row
    // rows y0-1, y0, y0+1 into ring rows 0, 1, 2
    for (int r = 0; r < 3; ++r) {
        row_issue_counts<kSub>(c, g, y0 - 1 + r, F);
        row_issue_entries<kSub>(c, g, S, F);
        row_commit<kSub>(g, S, F, r, head);
        head += F.total;
    }
    if (IY >= 2) row_issue_counts<kSub>(c, g, y0 + 2, F);
    for (int y = y0; y < y0 + IY; ++y) {
        const int rc = (y - y0 + 1) % 3;
        const int rm_ = (rc + 2) % 3, rp = (rc + 1) % 3;
        const bool next = y + 2 <= y0 + IY;  // row y+2 is the lower halo of row y+1
        if (next) {
            row_issue_entries<kSub>(c, g, S, F);
            if (y + 3 <= y0 + IY) row_issue_counts<kSub>(c, g, y + 3, G);
        }
        row_compute<kFluid, kSub>(c, w, P, wi, g, S, rm_, rc, rp);
        if (next) {
            row_commit<kSub>(g, S, F, rm_, head);  // row y+2 replaces row y-1
            head += F.total;
#pragma unroll
            for (int q = 0; q < RowFlight<kSub>::kSlots; ++q) {
                F.s0[q] = G.s0[q];
                F.s1[q] = G.s1[q];
            }
        }
    }
    return true;
}

// A collision world staged two bin rows at a time (sparse rows) runs a chunk whose two-row stages
// do not fit as single bin rows over the same bins.
// (four waves per SIMD, 128 VGPRs without scratch: at 133 VGPRs and three waves the eight-world batch ran
// 13 % slower)
template <bool kFluid>
__global__ void __launch_bounds__(kRowThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
k_neighbor_rows(Ctx c, int sortBlocks) {
    __shared__ RowShared<kFluid ? 1 : kSubMax> S;
    // (the particles' bin sort, on workgroups of its own, in sets with bond work)
    if (int(blockIdx.x) < sortBlocks) {
        part_binsort(c, {int(blockIdx.x), sortBlocks});
        return;
    }
    const int2 tb = c.tileBlocks[int(blockIdx.x) - sortBlocks];
    if (tb.x < 0) return;
    const int wi = tb.x;
    // the world and its parameters are read once, before any store: read through references,
    // every use after a global store would load them again
    const DevWorld w = c.worlds[wi];
    const DevParams P = c.params[wi];
    if ((P.motion == 0) != kFluid) return;
    const int strip = tb.y % w.ntx, chunk = tb.y / w.ntx;
    StripGeom g;
    g.x0 = strip * w.tileX;
    g.IX = min(w.tileX, w.nbx - g.x0);
    g.HX = g.IX + 2;
    g.nbx = w.nbx;
    g.nby = w.nby;
    g.binOff = w.binOff;
    g.cellOff = w.cellOff;
    g.base = c.start[w.binOff];
    g.seam = true;
    const int y0 = chunk * w.tileY;  // in staged rows of w.rowsPerStage bin rows
    const int IY = min(w.tileY, w.nby / w.rowsPerStage - y0);
    const int by0 = w.rowsPerStage * y0, bIY = w.rowsPerStage * IY;  // the chunk in bin rows
    bool done = false;
    // (fluid worlds are always staged one bin row at a time: the two-row variant would cost the
    // fluid kernel a third of its resident waves in registers)
    if constexpr (!kFluid)
        if (w.rowsPerStage == 2) done = chunk_rows<kFluid, 2>(c, w, P, wi, g, S, y0, IY);
    if (!done) done = chunk_rows<kFluid, 1>(c, w, P, wi, g, S, by0, bIY);
    if (!done) {
        // too crowded for the LDS staging: every cell walks its stencil in global memory, and the
        // owner-counted part of the region's bins is empty
        if (threadIdx.x == 0) atomicAdd(&c.sc->fallbackChunks, 1ull);
        rows_direct<kFluid>(c, w, P, wi, g, by0, bIY);
    }
}

int neighbor_blocks_per_cu() {
    int n = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_neighbor_rows<false>, kRowThreads, 0);
    return e == hipSuccess ? std::max(1, n) : 1;
}

void launch_fluid(const Ctx& c, const LaunchShape& sh, hipStream_t s, int sortBlocks);

void launch_neighbor(const Ctx& c, const LaunchShape& sh, hipStream_t s, bool withPartSort) {
    // (the bin sort goes with the first launch)
    int sort = withPartSort && sh.hasParticles && sh.partBlocks ? sh.pbinBlocks : 0;
    const bool collision = sh.hasCollision && sh.tileBlocks;
    if (sh.fluidBlocks || (sort && !collision)) {
        launch_fluid(c, sh, s, sort);
        sort = 0;
    }
    if (collision) {
        sort *= sh.binThreads / kRowThreads;
        hipLaunchKernelGGL(k_neighbor_rows<false>, dim3(sort + sh.tileBlocks), dim3(kRowThreads), 0, s, c, sort);
    }
}

}  // namespace alien
