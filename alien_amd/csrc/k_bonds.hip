// k_bonds.hip — bonded cells and structural operations.
//
// Connection forces (CellProcessor::calcConnectionForces, source/EngineGpuKernels/CellProcessor.cuh:
// 408-491) run twice per step around the Verlet position update (:525-544) and before the velocity
// update (:546-559), over the staged cells (cells with bonds, and barrier cells).  Angle forces that
// the reference adds to the neighbours with float atomics are written by the owner into per-bond
// slots and gathered by the receiver in its own bond order (R7).  Structural operations follow
// CellConnectionProcessor (source/EngineGpuKernels/CellConnectionProcessor.cuh): fusion pairs
// claim their cells and bond neighbours and apply only when every claim holds (R5); bond deletion
// works from per-cell flags (R6).
//
// The phase is a chain of launches, each of which needs all cells of the one before it.  Short ones
// cost their latency, not their work (18,000 cells: 2 to 12 us each), so what is independent shares a
// launch: the living states, and on workgroups of their own the stages of the particles' chain
// (particle_steps.hpp).  A step of 18,000 bonded cells with 700 particles took 126 us in 22 launches and
// takes 90 us in 11; 10,700 cells at ALIEN's default parameters 176 us in 27 and 124 us in 12; 840,000
// bonded cells without particles 336 us and 331 us.
#include "kernels.hpp"
#include "particle_steps.hpp"

namespace alien {

// The kernels below run one thread per cell of the worlds that can have bonded or barrier cells
// (bond block table) and act on the staged cells: those the neighbour pass found bonded or barrier
// (stage), which is the set CellProcessor's bonded-cell passes cover.  Cells bonded by this step's
// fusion are not among them.
__device__ __forceinline__ bool staged_cell(const Ctx& c, int block, int& x, int& wi, uint8_t& stage) {
    const int2 blk = c.bondBlocks[block];
    wi = blk.x;
    x = blk.y + int(threadIdx.x);
    const DevWorld& w = c.worlds[wi];
    stage = 0;
    if (x >= w.cellOff + w.numCells) return false;
    stage = c.stage[x];
    return stage != 0;
}

// Angle forces act every third step; on the others no partner has written any.
__device__ __forceinline__ bool angle_step(const Ctx& c, int wi) { return (c.ctr[wi].timestep % 3ull) == 0ull; }

// a partner's bond targets (-1: none) and flags, from the record the first pass leaves on an angle step
__device__ __forceinline__ uint32_t partner_list(const Ctx& c, int o, int (&t)[kMaxBonds]) {
    const int4 a = c.lists[2 * o], b = c.lists[2 * o + 1];
    t[0] = a.x, t[1] = a.y, t[2] = a.z, t[3] = a.w, t[4] = b.x, t[5] = b.y;
    return uint32_t(b.z);
}

// Connection forces of a staged cell: own force plus per-bond angle forces for the partners; pass 1
// also runs checkConnections (CellProcessor.cuh:493-523) on the moved positions.  The partners' data of
// all the cell's bonds is loaded up front, so the loads are in flight together (lanes skip the slots
// beyond their cell's bonds: 7 % faster than loading all six).
// Pass 0 finds the bond targets in start-of-step indices, as the neighbour pass left them, and
// renumbers them to the end-of-step order: it takes its own list from B (which it rewrites) and its
// partners' lists from A, so that no thread reads a list another rewrites.
// What a pass needs of a partner lies in one 16-byte record (bonded, moved): a gather costs the L1 a line
// per lane whatever its width.  Records, and no markers read or written on the steps without angle forces:
// 0.84M cells in bodies, a step 260 -> 248 us; with the bond lists of an angle step in records too (its
// partners' planes: seven gathers for each bond and pass), 242 us, eight worlds 172 -> 162 us.
// In the second pass the cells stand at pos + shift; the bond vector is taken as the start-of-pass
// difference plus the difference of the shifts, which keeps the FP32 result close to the exact one
// (rounding pos + shift first would cost up to ulp(world size)).
template <int kPass> __device__ __forceinline__ void conn_own(const Ctx& c, int block) {
    const int cap = c.cellCap;
    int x, wi;
    uint8_t stage;
    if (!staged_cell(c, block, x, wi, stage)) return;
    const DevWorld& w = c.worlds[wi];
    const DevParams& P = c.params[wi];
    const uint32_t fx = c.B.flags[x];
    const int nc = flags_num_conn(fx);
    // the partners' indices, in A (pass 0) or B (pass 1)
    int tl[kMaxBonds];
    float4 part[kMaxBonds];  // (what the bonds' partners have in the pass's record)
#pragma unroll
    for (int b = 0; b < kMaxBonds; ++b) tl[b] = b < nc ? w.cellOff + c.B.btgt[b * cap + x] : x;
#pragma unroll
    for (int b = 0; b < kMaxBonds; ++b) {
        part[b] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (b < nc) part[b] = (kPass == 0 ? c.bonded : c.moved)[tl[b]];
    }
    if constexpr (kPass == 0) {
#pragma unroll
        for (int b = 0; b < kMaxBonds; ++b)
            if (b < nc) c.B.btgt[b * cap + x] = __float_as_int(part[b].w) - w.cellOff;
    }
    const bool considerAngles = angle_step(c, wi);
    if (kPass == 0 && considerAngles && nc > 0) {
        int own[kMaxBonds];
#pragma unroll
        for (int b = 0; b < kMaxBonds; ++b) own[b] = b < nc ? __float_as_int(part[b].w) - w.cellOff : -1;
        c.lists[2 * x] = make_int4(own[0], own[1], own[2], own[3]);
        c.lists[2 * x + 1] = make_int4(own[4], own[5], int(fx), 0);
    }
    if (nc == 0 || flags_barrier(fx)) {
        if (considerAngles) c.valid[x] = 0u;
        if (kPass == 1) c.stretched[x] = 0;  // checkConnections skips barrier cells
        return;
    }
    const float Wf = float(w.W), Hf = float(w.H);
    f2 px, shx = {0.0f, 0.0f};
    if constexpr (kPass == 0) {
        px = to_f2(c.B.pos[x]);
    } else {
        const float4 own = c.moved[x];
        px = f2{own.x, own.y};
        shx = f2{own.z, own.w};
    }
    const float sx = c.bstiff[x];
    const float kx2 = sx * sx;
    f2 disp[kMaxBonds];
    float kc2[kMaxBonds], rest[kMaxBonds];
#pragma unroll
    for (int b = 0; b < kMaxBonds; ++b) {
        kc2[b] = 0.0f;
        rest[b] = 0.0f;
        disp[b] = f2{0.0f, 0.0f};
        if (b < nc) {
            const float so = kPass == 0 ? part[b].z : c.bstiff[tl[b]];
            kc2[b] = so * so;
            rest[b] = c.B.brest[b * cap + x];
            disp[b] = torus_delta(f2{part[b].x, part[b].y}, px, Wf, Hf);
            if constexpr (kPass == 1) disp[b] = add(disp[b], sub(f2{part[b].z, part[b].w}, shx));
        }
    }
    // the bond before the first is the last one
    f2 prevDisp = disp[0];
    int lastTarget = tl[0];
#pragma unroll
    for (int b = 1; b < kMaxBonds; ++b)
        if (b == nc - 1) {
            prevDisp = disp[b];
            lastTarget = tl[b];
        }
    f2 force = {0.0f, 0.0f};
    uint32_t v = 0u;
    bool tooLong = false;
    const float maxBind = P.maxBindingDistance[flags_color(fx) % kColors];
#pragma unroll
    for (int b = 0; b < kMaxBonds; ++b) {
        if (b >= nc) break;
        const int o = tl[b];
        const f2 d = disp[b];
        const float ad = len2(d);
        if (kPass == 1 && ad > maxBind) tooLong = true;  // checkConnections on new positions
        const float dev = ad - rest[b];
        force = add(force, dvd(mul(mul(unit(d), dev), kx2 + kc2[b]), 6.0f));
        bool skipped = false;  // a bond whose actual angle is negative keeps the previous vector
        if (considerAngles && (nc > 2 || (nc == 2 && b == 0))) {
            const int lc = b == 0 ? lastTarget : tl[b > 0 ? b - 1 : 0];
            uint32_t fo;
            int lt[kMaxBonds];
            if constexpr (kPass == 0) {
                fo = c.A.flags[o];
                const int no = flags_num_conn(fo);
                // (the partner's list: its loads in flight together)
#pragma unroll
                for (int j = 0; j < kMaxBonds; ++j) lt[j] = j < no ? c.A.btgt[j * cap + o] : -1;
            } else {
                fo = partner_list(c, o, lt);
            }
            bool tri = false;
#pragma unroll
            for (int j = 0; j < kMaxBonds; ++j) tri = tri || lt[j] == lc - w.cellOff;
            if (!tri) {
                const float angle = angle_of(d);
                const float prevAngle = angle_of(prevDisp);
                const float act = sub_angle(angle, prevAngle);
                if (act < 0.0f) {
                    skipped = true;
                } else {
                    const float ref = c.B.bang[b * cap + x];
                    const float strength = fabsf(ref - act) / 2000.0f * kx2;
                    f2 f1 = mul(dvd(unit(d), fmaxf(len2(d), P.minDistance)), strength);
                    rot_cw(f1);
                    f2 fb = mul(dvd(unit(prevDisp), fmaxf(len2(prevDisp), P.minDistance)), strength);
                    rot_ccw(fb);
                    if (ref < act) {
                        f1 = mul(f1, -1.0f);
                        fb = mul(fb, -1.0f);
                    }
                    if (!flags_barrier(fo)) {
                        c.out1[b * cap + x] = to_float2(f1);
                        v |= 1u << b;
                    }
                    if (!flags_barrier((kPass == 0 ? c.A : c.B).flags[lc])) {
                        c.out2[b * cap + x] = to_float2(fb);
                        v |= 1u << (6 + b);
                    }
                    force = sub(force, add(f1, fb));
                }
            }
        }
        if (!skipped) prevDisp = d;
    }
    c.own[x] = to_float2(force);
    if (considerAngles) c.valid[x] = v;
    if (tooLong) c.stage[x] = uint8_t(stage | kDropBonds);
    if (kPass == 1) c.stretched[x] = tooLong ? 1 : 0;
}

// (at most 80 VGPRs, six waves per SIMD: the partner loads are latency-bound)
template <bool kLate> __global__ void __attribute__((amdgpu_waves_per_eu(6))) k_conn_first(Ctx c, int partBlocks) {
    const int b = int(blockIdx.x);
    if (b < partBlocks)
        kLate ? part_binsort(c, {b, partBlocks}) : part_move(c, {b, partBlocks});
    else
        conn_own<0>(c, b - partBlocks);
}

template <bool kLate> __global__ void __attribute__((amdgpu_waves_per_eu(6))) k_conn_second(Ctx c, int partBlocks) {
    const int b = int(blockIdx.x);
    if (b < partBlocks)
        kLate ? part_target(c, {b, partBlocks}) : part_apply(c, {b, partBlocks});
    else
        conn_own<1>(c, b - partBlocks);
}

// own force plus the angle forces the partners wrote for this cell, in its bond order (R7); the
// partners' markers are loaded up front
__device__ __forceinline__ f2 gather_conn(const Ctx& c, const DevWorld& w, int wi, int x, int nc) {
    const int cap = c.cellCap;
    f2 acc = {0.0f, 0.0f};
    acc = add(acc, to_f2(c.own[x]));
    if (!angle_step(c, wi)) return acc;
    const int xl = x - w.cellOff;
    int pt[kMaxBonds];
    uint32_t vps[kMaxBonds];
#pragma unroll
    for (int q = 0; q < kMaxBonds; ++q) pt[q] = q < nc ? w.cellOff + c.B.btgt[q * cap + x] : x;
#pragma unroll
    for (int q = 0; q < kMaxBonds; ++q) vps[q] = q < nc ? c.valid[pt[q]] : 0u;
#pragma unroll
    for (int q = 0; q < kMaxBonds; ++q) {
        const uint32_t vp = vps[q];
        if (vp == 0u) continue;  // the partner wrote no angle force this pass
        const int p = pt[q];
        int lt[kMaxBonds];
        const int np = flags_num_conn(partner_list(c, p, lt));
        int b = -1;
#pragma unroll
        for (int kk = kMaxBonds - 1; kk >= 0; --kk) b = lt[kk] == xl ? kk : b;
        if (b < 0) continue;
        if (vp & (1u << b)) acc = add(acc, to_f2(c.out1[b * cap + p]));
        const int b2 = (b + 1) % np;
        if (vp & (1u << (6 + b2))) acc = add(acc, to_f2(c.out2[b2 * cap + p]));
    }
    return acc;
}

// Verlet position step (CellProcessor.cuh:525-544): the displacement is stored and applied after
// the second force pass
__device__ __forceinline__ void conn_pos(const Ctx& c, int block) {
    int x, wi;
    uint8_t stage;
    if (!staged_cell(c, block, x, wi, stage)) return;
    const DevWorld& w = c.worlds[wi];
    const DevParams& P = c.params[wi];
    const uint32_t fx = c.B.flags[x];
    const float dt = P.dt;
    const f2 v = to_f2(c.B.vel[x]), p = to_f2(c.B.pos[x]);
    if (flags_barrier(fx)) {
        const f2 sh = mul(v, dt);
        c.moved[x] = make_float4(p.x, p.y, sh.x, sh.y);
        return;
    }
    const f2 s1 = gather_conn(c, w, wi, x, flags_num_conn(fx));
    const f2 sh = add(mul(v, dt), mul(mul(mul(s1, dt), dt), 0.5f));  // x/2 == x*0.5 exactly
    c.moved[x] = make_float4(p.x, p.y, sh.x, sh.y);
    c.s2[x] = to_float2(s1);
}

template <bool kLate> __global__ void k_conn_pos(Ctx c, int partBlocks) {
    const int b = int(blockIdx.x);
    if (b < partBlocks)
        kLate ? part_move(c, {b, partBlocks}) : part_target(c, {b, partBlocks});
    else
        conn_pos(c, b - partBlocks);
}

// Verlet velocity step and friction (CellProcessor.cuh:546-559, 707-723); the moved position is
// written here, and its bin recorded for the next step's map
__device__ __forceinline__ void conn_vel(const Ctx& c, int block) {
    int x, wi;
    uint8_t stage;
    if (!staged_cell(c, block, x, wi, stage)) return;
    const DevWorld& w = c.worlds[wi];
    const DevParams& P = c.params[wi];
    const float dt = P.dt, friction = P.friction;
    // on an inner-friction step the velocity is left before friction for the next launch
    const bool inner = P.innerFriction > 0.0f && (c.ctr[wi].timestep % 3ull) == 0ull;
    // every load before the first store, so that they are in flight together
    const uint32_t fx = c.B.flags[x];
    const float4 at = c.moved[x];
    const f2 p = {at.x, at.y}, sh = {at.z, at.w}, v0 = to_f2(c.B.vel[x]), s2 = to_f2(c.s2[x]);
    // (the map gives the cell's start-of-step index at its end-of-step index)
    const f2 pOld = to_f2(c.A.pos[c.sorted[x]]);
    f2 s1 = {0.0f, 0.0f};
    if (!flags_barrier(fx)) s1 = gather_conn(c, w, wi, x, flags_num_conn(fx));
    const f2 p2 = torus_pos(add(p, sh), w.W, w.H);
    c.B.pos[x] = to_float2(p2);
    bin_next(c, w, x, p2, cell_bin_of(w, pOld) - w.binOff);
    if (flags_barrier(fx)) return;
    const f2 acc = mul(add(s1, s2), 0.5f);
    f2 v = add(v0, mul(acc, dt));
    if (inner) {
        c.s2[x] = to_float2(v);  // the start-of-pass velocity of the inner friction
    } else {
        v = mul(v, 1.0f - friction);
    }
    c.B.vel[x] = to_float2(v);
}

// applyInnerFriction (CellProcessor.cuh:678-705) every third step, then applyFriction (:707-723).
// Jacobi (rule R11): each bond is relaxed twice for the cell, once for its own visit and once for
// the partner's visit of the bond, toward the partner's start-of-pass velocity, in bond order;
// barrier partners are skipped.
__device__ __forceinline__ void inner_friction(const Ctx& c, const DevWorld& w, const DevParams& P, int x, int nc,
                                               const int t[kMaxBonds]) {
    const float f = P.innerFriction;
    f2 vp[kMaxBonds];
    bool use[kMaxBonds];
#pragma unroll
    for (int b = 0; b < kMaxBonds; ++b) {
        use[b] = false;
        vp[b] = f2{0.0f, 0.0f};
        if (b < nc) {
            use[b] = !flags_barrier(c.B.flags[t[b]]);
            if (use[b]) vp[b] = to_f2(c.s2[t[b]]);
        }
    }
    f2 v = to_f2(c.s2[x]);
    for (int visit = 0; visit < 2; ++visit)
#pragma unroll
        for (int b = 0; b < kMaxBonds; ++b)
            if (b < nc && use[b]) {
                const f2 avg = mul(add(v, vp[b]), 0.5f);
                v = add(mul(v, 1.0f - f), mul(avg, f));
            }
    v = mul(v, 1.0f - P.friction);
    c.B.vel[x] = to_float2(v);
}

// CellProcessor.cuh:786-790: a cell with more energy than cellMaxBindingEnergy loses its bonds
__device__ __forceinline__ bool above_max_energy(const Ctx& c, const DevWorld& w, const DevParams& P, int x) {
    return !flags_barrier(c.B.flags[x]) && c.energy[w.cellOff + c.B.slot[x]] > P.maxBindingEnergy;
}

// Inner friction, and the marks of the structural operations: whether the cell or a bond partner loses
// its bonds (R6), from the kDropBonds bits of the passes before and, with a finite maximum, from the
// energies as absorption left them.  A cell sets its own bits here while its partners read its byte:
// they take kDropBonds from the passes before or test the same energy, and get the same answer either way.
__device__ __forceinline__ void friction_and_marks(const Ctx& c, int block) {
    const int cap = c.cellCap;
    int x, wi;
    uint8_t stage;
    if (!staged_cell(c, block, x, wi, stage)) return;
    const DevWorld& w = c.worlds[wi];
    const DevParams& P = c.params[wi];
    const uint32_t fx = c.B.flags[x];
    const int nc = flags_num_conn(fx);
    int t[kMaxBonds];
#pragma unroll
    for (int b = 0; b < kMaxBonds; ++b) t[b] = b < nc ? w.cellOff + c.B.btgt[b * cap + x] : x;
    uint32_t m = 0u;
#pragma unroll
    for (int b = 0; b < kMaxBonds; ++b)
        if (b < nc) m |= c.stage[t[b]];
    bool own = (stage & kDropBonds) != 0;
    bool any = own || (m & kDropBonds) != 0u;
    if (P.maxBindingEnergy < __builtin_huge_valf()) {
        if (above_max_energy(c, w, P, x)) own = any = true;
#pragma unroll
        for (int b = 0; b < kMaxBonds; ++b)
            if (b < nc && above_max_energy(c, w, P, t[b])) any = true;
    }
    if (any) c.stage[x] = uint8_t(kStagedCell | (own ? kDropBonds : 0) | kMarkedCell);
    if (!(P.innerFriction > 0.0f) || (c.ctr[wi].timestep % 3ull) != 0ull || flags_barrier(fx)) return;
    inner_friction(c, w, P, x, nc, t);
}

// ---------------------------------------------------------------------------------------------
// living states of the worlds that track them (rule R17, cellDeathConsequences None), one thread
// per end-of-step cell.  The three phases alternate between the two state buffers (living at the
// start of the step -> livingNext -> living -> livingNext, the next step's start).
// ---------------------------------------------------------------------------------------------
constexpr uint8_t kReady = 0, kUnderConstruction = 1, kActivating = 2, kDetaching = 3, kReviving = 4, kDying = 5;

__device__ __forceinline__ bool living_cell(const Ctx& c, int block, int& x, int& wi) {
    const int2 blk = c.livingBlocks[block];
    wi = blk.x;
    x = blk.y + int(threadIdx.x);
    const DevWorld& w = c.worlds[wi];
    return x < w.cellOff + w.numCells;
}

// checkConnections' Detaching marks on the partners of cells with an overstretched bond
// (CellProcessor.cuh:515-520), then aging (:561-594)
__device__ __forceinline__ void living_mark_age(const Ctx& c, int block) {
    const int cap = c.cellCap;
    int x, wi;
    if (!living_cell(c, block, x, wi)) return;
    const DevWorld& w = c.worlds[wi];
    const uint32_t fx = c.B.flags[x];
    const int sl = w.cellOff + c.B.slot[x];
    uint8_t st = c.living[sl];
    if (w.bondWork) {  // (stretched marks exist for the staged cells of worlds with bond work)
        const int nc = flags_num_conn(fx);
        for (int b = 0; b < nc; ++b)
            if (c.stretched[w.cellOff + c.B.btgt[b * cap + x]]) st = kDetaching;
    }
    if (!flags_barrier(fx)) {
        const uint32_t act = c.activation[sl];
        if (st == kReady && act > 0u) c.activation[sl] = act - 1u;
    }
    c.livingNext[sl] = st;
}

// the state transitions (CellProcessor.cuh:596-676) from the states after the marks
__device__ __forceinline__ void living_transition(const Ctx& c, int block) {
    const int cap = c.cellCap;
    int x, wi;
    if (!living_cell(c, block, x, wi)) return;
    const DevWorld& w = c.worlds[wi];
    const uint32_t fx = c.B.flags[x];
    const int sl = w.cellOff + c.B.slot[x];
    const uint8_t st = c.livingNext[sl];
    uint8_t next = st;
    if (flags_barrier(fx)) {
        next = kReady;
    } else if (st == kActivating || st == kReviving || st == kDetaching) {
        next = kReady;  // Detaching -> Ready under cellDeathConsequences None
    } else if (st == kUnderConstruction) {
        const uint32_t cr = c.creature[sl];
        const int nc = flags_num_conn(fx);
        for (int b = 0; b < nc; ++b) {
            const int ps = w.cellOff + c.B.slot[w.cellOff + c.B.btgt[b * cap + x]];
            if (c.creature[ps] == cr && c.livingNext[ps] == kActivating) next = kActivating;
        }
    }
    c.living[sl] = next;
}

// decay (CellProcessor.cuh:775-858): energy below cellMinEnergy -> Dying; the partners of a cell
// that becomes Dying -> Detaching unless they are or become Dying (cellDeathProbability 0)
__device__ __forceinline__ bool below_min_energy(const Ctx& c, const DevWorld& w, const DevParams& P, uint32_t f, int sl) {
    return !flags_barrier(f) && c.energy[sl] < P.minEnergy[flags_color(f)];
}

__device__ __forceinline__ void living_decay(const Ctx& c, int block) {
    const int cap = c.cellCap;
    int x, wi;
    if (!living_cell(c, block, x, wi)) return;
    const DevWorld& w = c.worlds[wi];
    const DevParams& P = c.params[wi];
    const uint32_t fx = c.B.flags[x];
    const int sl = w.cellOff + c.B.slot[x];
    const uint8_t st = c.living[sl];
    uint8_t next = st;
    if (below_min_energy(c, w, P, fx, sl)) {
        next = kDying;
    } else if (st != kDying) {
        const int nc = flags_num_conn(fx);
        for (int b = 0; b < nc; ++b) {
            const int p = w.cellOff + c.B.btgt[b * cap + x];
            const int ps = w.cellOff + c.B.slot[p];
            if (below_min_energy(c, w, P, c.B.flags[p], ps) && c.living[ps] != kDying) next = kDetaching;
        }
    }
    c.livingNext[sl] = next;
}

// A set without bond work has no bonded or barrier cell: aging with the activation count
// (CellProcessor.cuh:561-594), the transitions (:596-676; UnderConstruction stays without an
// Activating partner) and the decay to Dying (:775-858; no partner to mark Detaching) of the three
// kernels above need no partner, and one pass per cell gives their end-of-step state.
__global__ void k_living_unbonded(Ctx c) {
    int x, wi;
    if (!living_cell(c, int(blockIdx.x), x, wi)) return;
    const DevWorld& w = c.worlds[wi];
    const DevParams& P = c.params[wi];
    const uint32_t fx = c.B.flags[x];
    const int sl = w.cellOff + c.B.slot[x];
    uint8_t st = c.living[sl];
    if (!flags_barrier(fx)) {
        const uint32_t act = c.activation[sl];
        if (st == kReady && act > 0u) c.activation[sl] = act - 1u;
    }
    if (flags_barrier(fx) || st == kActivating || st == kReviving || st == kDetaching) st = kReady;
    if (below_min_energy(c, w, P, fx, sl)) st = kDying;
    c.livingNext[sl] = st;
}

// the velocity step, the marks and ages of the living states (from this step's overstretched bonds),
// and the absorptions
template <bool kLate> __global__ void k_conn_vel(Ctx c, int partBlocks, int bondBlocks) {
    int b = int(blockIdx.x);
    if (b < partBlocks) return kLate ? part_apply(c, {b, partBlocks}) : part_absorb(c, {b, partBlocks});
    b -= partBlocks;
    if (b < bondBlocks) return conn_vel(c, b);
    living_mark_age(c, b - bondBlocks);
}

__global__ void k_marks(Ctx c, int absorbBlocks, int bondBlocks) {
    int b = int(blockIdx.x);
    if (b < absorbBlocks) return part_absorb(c, {b, absorbBlocks});
    b -= absorbBlocks;
    if (b < bondBlocks)
        friction_and_marks(c, b);
    else
        living_transition(c, b - bondBlocks);
}

// ---------------------------------------------------------------------------------------------
// structural operations (CellConnectionProcessor.cuh), R5/R6
// ---------------------------------------------------------------------------------------------
template <class F> __device__ __forceinline__ void for_claim_set(const Ctx& c, const DevWorld& w, int a, int b, F&& f) {
    const int cap = c.cellCap;
    f(a);
    int na = flags_num_conn(c.B.flags[a]);
    for (int k = 0; k < na; ++k) f(w.cellOff + c.B.btgt[k * cap + a]);
    f(b);
    int nb = flags_num_conn(c.B.flags[b]);
    for (int k = 0; k < nb; ++k) f(w.cellOff + c.B.btgt[k * cap + b]);
}

__device__ __forceinline__ unsigned long long claim_key(const DevWorld& w, int a, int b) {
    return (static_cast<unsigned long long>(uint32_t(a - w.cellOff)) << 32) | uint32_t(b - w.cellOff);
}

// A cell that loses its bonds this step, or has a partner that does, fuses with none.  Unbonded cells
// have no marks: of the reasons to lose bonds, too much energy applies to them as well.
__device__ __forceinline__ bool fusion_barred(const Ctx& c, const DevWorld& w, const DevParams& P, int x) {
    const uint8_t stage = c.stage[x];
    if (stage != 0) return (stage & kMarkedCell) != 0;
    return P.maxBindingEnergy < __builtin_huge_valf() && above_max_energy(c, w, P, x);
}

__device__ __forceinline__ void fuse_claim(const Ctx& c, Span at) {
    const int n = min(c.sc->candidates, c.candCap);
    for (int q = at.block * blockDim.x + threadIdx.x; q < n; q += at.blocks * blockDim.x) {
        int4 cd = c.cand[q];
        const DevWorld& w = c.worlds[cd.z];
        if (fusion_barred(c, w, c.params[cd.z], cd.x) || fusion_barred(c, w, c.params[cd.z], cd.y)) {
            c.cand[q].w = 0;
            continue;
        }
        unsigned long long key = claim_key(w, cd.x, cd.y);
        for_claim_set(c, w, cd.x, cd.y, [&](int x) { atomicMin(&c.claim[x], key); });
    }
}

// the fusion claims, and the living states' decay (which reads the bond lists before fusions change them)
__global__ void k_fuse_claim(Ctx c, int candBlocks) {
    const int b = int(blockIdx.x);
    if (b < candBlocks)
        fuse_claim(c, {b, candBlocks});
    else
        living_decay(c, b - candBlocks);
}

// tryAddConnectionOneWay (CellConnectionProcessor.cuh:274-427) without angle alignment
__device__ bool would_overlap(const Ctx& c, const DevWorld& w, int c1, f2 otherPos) {
    const int cap = c.cellCap;
    const int n = flags_num_conn(c.B.flags[c1]);
    if (n < 2) return false;
    const f2 p1 = to_f2(c.B.pos[c1]);
    for (int i = 0; i < n; ++i) {
        const int cc = w.cellOff + c.B.btgt[i * cap + c1];
        const int nc = w.cellOff + c.B.btgt[((i + 1) % n) * cap + c1];
        const int ncl = nc - w.cellOff;
        const int ncc = flags_num_conn(c.B.flags[cc]);
        bool both = false;
        for (int j = 0; j < ncc; ++j)
            if (c.B.btgt[j * cap + cc] == ncl) {
                both = true;
                break;
            }
        if (!both) continue;
        if (segments_cross(p1, otherPos, to_f2(c.B.pos[cc]), to_f2(c.B.pos[nc]))) return true;
    }
    return false;
}

__device__ bool add_one_way(const Ctx& c, const DevWorld& w, int c1, int c2, f2 posDelta) {
    const int cap = c.cellCap;
    const float Wf = float(w.W), Hf = float(w.H);
    uint32_t f = c.B.flags[c1];
    const int n = flags_num_conn(f);
    if (n == kMaxBonds) return false;
    if (would_overlap(c, w, c1, to_f2(c.B.pos[c2]))) return false;
    const float newAngle = angle_of(posDelta);
    const float dist = len2(posDelta);
    const int c2l = c2 - w.cellOff;
    const f2 p1 = to_f2(c.B.pos[c1]);
    if (n == 0) {
        c.B.btgt[c1] = c2l;
        c.B.brest[c1] = dist;
        c.B.bang[c1] = 360.0f;
        c.B.flags[c1] = flags_with_num_conn(f, 1);
        return true;
    }
    if (n == 1) {
        const f2 cd = torus_delta(to_f2(c.B.pos[w.cellOff + c.B.btgt[c1]]), p1, Wf, Hf);
        const float prevAngle = angle_of(cd);
        float angleDiff = newAngle - prevAngle;
        if (angleDiff < 0.0f) angleDiff += 360.0f;
        if (fabsf(angleDiff) < kNearZero || fabsf(angleDiff - 360.0f) < kNearZero ||
            fabsf(angleDiff + 360.0f) < kNearZero)
            return false;
        c.B.bang[cap + c1] = angleDiff;
        c.B.bang[c1] = 360.0f - angleDiff;
        c.B.btgt[cap + c1] = c2l;
        c.B.brest[cap + c1] = dist;
        c.B.flags[c1] = flags_with_num_conn(f, 2);
        return true;
    }
    int index = 0;
    float prevAngle = 0.0f, nextAngle = 0.0f;
    bool found = false;
    for (; index < n; ++index) {
        const int prevIndex = (index + n - 1) % n;
        prevAngle = angle_of(torus_delta(to_f2(c.B.pos[w.cellOff + c.B.btgt[prevIndex * cap + c1]]), p1, Wf, Hf));
        nextAngle = angle_of(torus_delta(to_f2(c.B.pos[w.cellOff + c.B.btgt[index * cap + c1]]), p1, Wf, Hf));
        if (angle_between(prevAngle, nextAngle, newAngle) || prevIndex == index) {
            found = true;
            break;
        }
    }
    if (!found) return false;
    const float refAngle = c.B.bang[index * cap + c1];
    const float angleDiff1 = sub_angle(newAngle, prevAngle);
    const float angleDiff2 = sub_angle(nextAngle, prevAngle);
    const float frac = angleDiff2 != 0.0f ? angleDiff1 / angleDiff2 : 0.5f;
    float afp = refAngle * frac;
    afp = fminf(afp, refAngle);
    if (afp < kNearZero) return false;
    if (index == 0) index = n;
    for (int j = n; j > index; --j) {
        c.B.btgt[j * cap + c1] = c.B.btgt[(j - 1) * cap + c1];
        c.B.brest[j * cap + c1] = c.B.brest[(j - 1) * cap + c1];
        c.B.bang[j * cap + c1] = c.B.bang[(j - 1) * cap + c1];
    }
    c.B.btgt[index * cap + c1] = c2l;
    c.B.brest[index * cap + c1] = dist;
    c.B.bang[index * cap + c1] = afp;
    c.B.bang[((index + 1) % (n + 1)) * cap + c1] = refAngle - afp;
    c.B.flags[c1] = flags_with_num_conn(f, n + 1);
    return true;
}

__global__ void k_fuse_apply(Ctx c) {
    const int n = min(c.sc->candidates, c.candCap);
    const int cap = c.cellCap;
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) {
        int4 cd = c.cand[q];
        if (!cd.w) continue;
        const DevWorld& w = c.worlds[cd.z];
        const int a = cd.x, b = cd.y;
        unsigned long long key = claim_key(w, a, b);
        bool ok = true;
        for_claim_set(c, w, a, b, [&](int x) { ok = ok && (c.claim[x] == key); });
        if (!ok) continue;
        // lockAndtryAddConnections (CellConnectionProcessor.cuh:249-272)
        const uint32_t fa = c.B.flags[a], fb = c.B.flags[b];
        const int na = flags_num_conn(fa), nb = flags_num_conn(fb);
        bool already = false;
        for (int k = 0; k < na; ++k) already = already || (c.B.btgt[k * cap + a] == b - w.cellOff);
        if (already) continue;
        if (!(na < flags_max_conn(fa) && nb < flags_max_conn(fb))) continue;
        // tryAddConnections (:211-240)
        const f2 posDelta = torus_delta(to_f2(c.B.pos[b]), to_f2(c.B.pos[a]), float(w.W), float(w.H));
        int st[kMaxBonds];
        float sr[kMaxBonds], sa[kMaxBonds];
        for (int k = 0; k < kMaxBonds; ++k) {
            st[k] = c.B.btgt[k * cap + a];
            sr[k] = c.B.brest[k * cap + a];
            sa[k] = c.B.bang[k * cap + a];
        }
        if (!add_one_way(c, w, a, b, posDelta)) continue;
        if (!add_one_way(c, w, b, a, mul(posDelta, -1.0f))) {
            c.B.flags[a] = fa;
            for (int k = 0; k < kMaxBonds; ++k) {
                c.B.btgt[k * cap + a] = st[k];
                c.B.brest[k * cap + a] = sr[k];
                c.B.bang[k * cap + a] = sa[k];
            }
        }
    }
}

__device__ __forceinline__ void fuse_reset(const Ctx& c, Span at) {
    const int n = min(c.sc->candidates, c.candCap);
    for (int q = at.block * blockDim.x + threadIdx.x; q < n; q += at.blocks * blockDim.x) {
        int4 cd = c.cand[q];
        if (!cd.w) continue;
        const DevWorld& w = c.worlds[cd.z];
        for_claim_set(c, w, cd.x, cd.y, [&](int x) { c.claim[x] = ~0ull; });
    }
}

// deleteConnectionOneWay (CellConnectionProcessor.cuh:429-448)
__device__ void delete_one_way(const Ctx& c, int c1, int targetLocal) {
    const int cap = c.cellCap;
    uint32_t f = c.B.flags[c1];
    const int n = flags_num_conn(f);
    for (int i = 0; i < n; ++i) {
        if (c.B.btgt[i * cap + c1] == targetLocal) {
            const float angleToAdd = c.B.bang[i * cap + c1];
            for (int j = i; j < n - 1; ++j) {
                c.B.btgt[j * cap + c1] = c.B.btgt[(j + 1) * cap + c1];
                c.B.brest[j * cap + c1] = c.B.brest[(j + 1) * cap + c1];
                c.B.bang[j * cap + c1] = c.B.bang[(j + 1) * cap + c1];
            }
            if (i < n - 1)
                c.B.bang[i * cap + c1] += angleToAdd;
            else
                c.B.bang[c1] += angleToAdd;
            c.B.flags[c1] = flags_with_num_conn(f, n - 1);
            return;
        }
    }
}

__device__ __forceinline__ void delete_bonds(const Ctx& c, int block) {
    const int cap = c.cellCap;
    int x, wi;
    uint8_t stage;
    if (!staged_cell(c, block, x, wi, stage) || !(stage & kMarkedCell)) return;
    const DevWorld& w = c.worlds[wi];
    const int nc = flags_num_conn(c.B.flags[x]);
    int snap[kMaxBonds];
    for (int b = 0; b < nc; ++b) snap[b] = c.B.btgt[b * cap + x];
    for (int b = 0; b < nc; ++b)
        if ((stage | c.stage[w.cellOff + snap[b]]) & kDropBonds) delete_one_way(c, x, snap[b]);
}

// Last launch of the step: frees the claims of this step's candidates, drops the bonds of the marked
// cells (a pair with a marked cell claimed nothing, so the two touch different cells) and advances
// every world's timestep (SimulationCudaFacade.cu:140-143).
__global__ void k_fuse_end(Ctx c, int candBlocks) {
    const int b = int(blockIdx.x);
    if (b == 0)
        for (int wi = threadIdx.x; wi < c.numWorlds; wi += blockDim.x) c.ctr[wi].timestep += 1ull;
    if (b < candBlocks)
        fuse_reset(c, {b, candBlocks});
    else
        delete_bonds(c, b - candBlocks);
}

// The phase after the neighbour pass in sets with bond work (SimulationKernelsLauncher.cu:38-91), with
// the particles' chain from the movement on: their bin sort ran with the neighbour pass.  Energies
// change in the absorptions only; before them the neighbour pass read them for fusion candidates, after
// them the marks and the decay do.
// The particles' chain goes along: movement in the first launch to absorption in the fourth, or all of it a
// launch later (lateParticles), which lets the scan of their bins share the launch of the cells' map (a
// launch of its own was 4.5 us of a step's 64.5 with 18k cells in bodies; now 59.4).
void launch_bonds(const Ctx& c, const LaunchShape& sh, hipStream_t s, Recorder* rec) {
    const int parts = sh.hasParticles && sh.partBlocks ? sh.partGrid : 0;
    const int sort = parts ? sh.pbinBlocks : 0;
    const int bonds = sh.bondBlocks, living = sh.livingBlocks, cand = sh.candGrid;
    const dim3 t(sh.cellThreads);
#define L(name, kernel, grid, ...)                                         \
    do {                                                                   \
        if (rec) rec->mark(name);                                          \
        hipLaunchKernelGGL(kernel, dim3(grid), t, 0, s, __VA_ARGS__);      \
    } while (0)
    if (sh.lateParticles) {
        L("conn_first", k_conn_first<true>, sort + bonds, c, sort);
        L("conn_pos", k_conn_pos<true>, parts + bonds, c, parts);
        L("conn_second", k_conn_second<true>, parts + bonds, c, parts);
        L("conn_vel", k_conn_vel<true>, parts + bonds + living, c, parts, bonds);
    } else {
        L("conn_first", k_conn_first<false>, parts + bonds, c, parts);
        L("conn_pos", k_conn_pos<false>, parts + bonds, c, parts);
        L("conn_second", k_conn_second<false>, parts + bonds, c, parts);
        L("conn_vel", k_conn_vel<false>, parts + bonds + living, c, parts, bonds);
    }
    const int absorb = sh.lateParticles ? parts : 0;
    L("marks", k_marks, absorb + bonds + living, c, absorb, bonds);
    L("fuse_claim", k_fuse_claim, cand + living, c, cand);
    L("fuse_apply", k_fuse_apply, cand, c);
    L("fuse_end", k_fuse_end, cand + bonds, c, cand);
#undef L
}

// a set without bond work has no staged cell, and the scan at the start of the step advanced the
// timesteps
void launch_living_unbonded(const Ctx& c, const LaunchShape& sh, hipStream_t s, Recorder* rec) {
    if (!sh.livingBlocks) return;
    if (rec) rec->mark("living_unbonded");
    hipLaunchKernelGGL(k_living_unbonded, dim3(sh.livingBlocks), dim3(sh.cellThreads), 0, s, c);
}

}  // namespace alien
