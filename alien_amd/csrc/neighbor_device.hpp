// neighbor_device.hpp — what the fluid and the collision neighbour pass share: the neighbour predicate,
// the terms of a pair, the sums of a cell and its end-of-pass state.
//
// ALIEN: calcCollisions_reconnectCells_correctOverlap / calcFluidForces_reconnectCells_correctOverlap
// (source/EngineGpuKernels/CellProcessor.cuh:122-365), then checkForces/applyForces (:367-406); for
// cells without bonds also the Verlet updates and friction of the same step (:525-559, :707-723),
// which reduce to local operations when the connection forces are zero.
//
// Divisions by per-world constants (1/h, 1/h^2, 1/h^3), by a cell's density, by |d| and by the
// collision and viscosity denominators are products with the correctly rounded reciprocal (R16
// of the oracle), and the length comparisons |v| > c are tests of |v|^2 against the exact
// threshold of the correctly rounded square root.
#pragma once

#include "kernels_common.hpp"

namespace alien {

struct Nb {
    f2 pos, vel;
    float dens;  // 1 / density (fluid)
    uint32_t flags;
    int aidx;  // index in the start-of-step arrays (A)
    int lidx;  // index in the end-of-step arrays (B), the logical index of this step
};

__device__ __forceinline__ void push_candidate(const Ctx& c, int a, int b, int w) {
    int q = atomicAdd(&c.sc->candidates, 1);
    if (q < c.candCap)
        c.cand[q] = make_int4(a, b, w, 1);
    else
        atomicOr(&c.sc->errors, 1);
}

// what a neighbour pair contributes
constexpr uint32_t kPairBarrier = 1u;  // fluid: a barrier neighbour (A index, distance)
constexpr uint32_t kPairSelf = 2u;     // fluid: the cell itself (density term only)
constexpr uint32_t kPairOverlap = 4u;  // overlap correction
constexpr uint32_t kPairForce = 8u;    // force terms
constexpr int kPairTerms = 7;

// neighbour predicate (fluid: CellProcessor.cuh:137-143; collision: Map.cuh:189 with
// CellProcessor.cuh:290-296): |d| <= R tested as |d|^2 <= reachSq, which is exactly equivalent.
// Cells are never detached here (detached cells come from cell functions), so the detached rule
// never applies.
template <bool kFluid>
__device__ __forceinline__ bool is_neighbor(const Nb& s, const Nb& o, float Wf, float Hf, float reachSq) {
    if constexpr (kFluid)
        return lensq(torus_delta(s.pos, o.pos, Wf, Hf)) <= reachSq;
    else
        return o.aidx != s.aidx && lensq(sub(o.pos, s.pos)) <= reachSq;
}

// The contribution of neighbour o to cell s, for a pair that passed is_neighbor.  The logical
// indices of the two cells are needed only for a fusion candidate: lidxOf() returns them as
// (s, o) when asked.
template <bool kFluid, class LidxOf>
__device__ __forceinline__ uint32_t pair_term(const Ctx& c, const DevWorld& w, const DevParams& P, int wi, const Nb& s,
                                              const Nb& o, bool bonded, float* t, bool seam, LidxOf&& lidxOf) {
    const float Wf = float(w.W), Hf = float(w.H);
    const float cmd = P.minDistance;
    const bool bari = flags_barrier(s.flags);
    const f2 pd = stencil_delta(s.pos, o.pos, Wf, Hf, seam);
    const float d = len2(pd);
    uint32_t f = 0u;
    if constexpr (kFluid) {
        // CellProcessor.cuh:144-231
        if (flags_barrier(o.flags)) {
            t[0] = __int_as_float(o.aidx);
            t[1] = d;
            return kPairBarrier;
        }
        t[0] = sph_w(d * P.invH) * P.invH2;
        if (o.aidx == s.aidx) return kPairSelf;
        if (!bari && d < cmd) {
            const f2 D = dvd(mul(pd, cmd), 5.0f);
            t[1] = D.x;
            t[2] = D.y;
            f |= kPairOverlap;
        }
        if (bonded) return f;
        const f2 vd = sub(s.vel, o.vel);
        const float factor = s.dens + o.dens;  // 1/density_i + 1/density_j
        if (fabsf(d) > kNearZero) {
            const float kd = sph_dw(d * P.invH) * P.invH3;
            const f2 Fp = mul(mul(mul(pd, 1.0f / (-d)), factor), kd);
            const f2 Fv = mul(mul(mul(mul(vd, o.dens), d), kd), 1.0f / (d * d + 0.25f));
            t[3] = Fp.x;
            t[4] = Fp.y;
            t[5] = Fv.x;
            t[6] = Fv.y;
            f |= kPairForce;
        }
        if (flags_num_conn(s.flags) < flags_max_conn(s.flags) && flags_num_conn(o.flags) < flags_max_conn(o.flags) &&
            !bari && lensq(vd) > P.fusionBelowSq) {
            const int2 L = lidxOf();
            if (L.x < L.y) {
                const float ei = c.energy[w.cellOff + c.A.slot[s.aidx]];
                const float ej = c.energy[w.cellOff + c.A.slot[o.aidx]];
                if (ei <= P.maxBindingEnergy && ej <= P.maxBindingEnergy) push_candidate(c, L.x, L.y, wi);
            }
        }
    } else {
        // CellProcessor.cuh:297-361.  f(j,i) mirrors f(i,j): unit(-d) = -unit(d) and
        // (-dv).(-d) = dv.d exactly, so only the barrier factor and the branch differ.
        if (!bari && d < cmd) {
            const f2 D = dvd(mul(pd, cmd), 5.0f);
            t[0] = D.x;
            t[1] = D.y;
            f |= kPairOverlap;
        }
        if (bonded) return f;
        const f2 vd = sub(s.vel, o.vel);
        const float dvp = dot2(vd, pd);
        const bool appr = dot2(pd, vd) < 0.0f;
        const bool barj = flags_barrier(o.flags);
        const bool fastI = appr && lensq(s.vel) > P.fastSq;
        const bool fastJ = appr && lensq(o.vel) > P.fastSq;
        f2 fastT = {0.0f, 0.0f}, repT = {0.0f, 0.0f};
        if (fastI || fastJ) fastT = mul(mul(pd, dvp), 1.0f / (-2.0f * (d * d + 0.25f)));
        if (!(fastI && fastJ)) repT = mul(mul(unit(pd), P.collisionDistance - d), P.repulsion);
        const f2 fij = mul(fastI ? fastT : repT, bari ? 2.0f : 1.0f);
        // -f(j,i); unit() of a (near) zero vector is (1,0) in both directions, so there the
        // repulsion is not mirrored
        const f2 fjRep = mul(repT, barj ? 2.0f : 1.0f);
        const f2 nfji = fastJ ? mul(fastT, barj ? 2.0f : 1.0f) : (d > kNearZero ? fjRep : neg(fjRep));
        t[2] = fij.x;
        t[3] = fij.y;
        t[4] = nfji.x;
        t[5] = nfji.y;
        f |= kPairForce;
        if (flags_num_conn(s.flags) < flags_max_conn(s.flags) && flags_num_conn(o.flags) < flags_max_conn(o.flags) &&
            appr && !bari && !barj && lensq(vd) > P.fusionBelowSq) {
            const int2 L = lidxOf();
            if (L.x < L.y) {
                const float ei = c.energy[w.cellOff + c.A.slot[s.aidx]];
                const float ej = c.energy[w.cellOff + c.A.slot[o.aidx]];
                if (ei <= P.maxBindingEnergy && ej <= P.maxBindingEnergy) push_candidate(c, L.x, L.y, wi);
            }
        }
    }
    return f;
}

// per-cell sums of the pass, added in visiting order.  Of the barrier neighbours only the first
// ten count, and of those the first nearest one (CellProcessor.cuh:234-246); it is tracked as the
// barriers arrive.
struct Acc {
    f2 F, pc, D, Fp, Fv;
    float rho;
    int numBarrier;
    int cb;  // nearest barrier (A index), -1 if none
    float cbDist;
};

__device__ __forceinline__ void acc_init(Acc& a, const Nb& s) {
    a.F = {0.0f, 0.0f};
    a.pc = s.pos;
    a.D = {0.0f, 0.0f};
    a.Fp = {0.0f, 0.0f};
    a.Fv = {0.0f, 0.0f};
    a.rho = 0.0f;
    a.numBarrier = 0;
    a.cb = -1;
    a.cbDist = 0.0f;
}

template <bool kFluid>
__device__ __forceinline__ void acc_add(Acc& a, uint32_t f, const float* t) {
    if constexpr (kFluid) {
        if (f & kPairBarrier) {
            if (a.numBarrier < 10 && (a.cb < 0 || t[1] < a.cbDist)) {
                a.cb = __float_as_int(t[0]);
                a.cbDist = t[1];
            }
            ++a.numBarrier;
            return;
        }
        a.rho = a.rho + t[0];
        if (f & kPairSelf) return;
        if (f & kPairOverlap) a.D = add(a.D, f2{t[1], t[2]});
        if (f & kPairForce) {
            a.Fp = add(a.Fp, f2{t[3], t[4]});
            a.Fv = add(a.Fv, f2{t[5], t[6]});
        }
    } else {
        if (f & kPairOverlap) a.pc = add(a.pc, f2{t[0], t[1]});
        if (f & kPairForce) {
            a.F = add(a.F, f2{t[2], t[3]});
            a.F = add(a.F, f2{t[4], t[5]});
        }
    }
}

// acc_add of a collision pair without branches, for terms zeroed before pair_term wrote them.  Adding a
// zero term leaves a sum that started at +0 unchanged bit for bit (such a sum is never -0), so the flags
// select only for the position sum, which starts at the cell's position.
__device__ __forceinline__ void acc_add_collision(Acc& a, uint32_t f, f2 push, f2 f1, f2 f2nd) {
    const f2 pc = add(a.pc, push);
    if (f & kPairOverlap) a.pc = pc;
    a.F = add(add(a.F, f1), f2nd);
}

__device__ __forceinline__ void load_bonds(const Ctx& c, const Nb& s, int bt[kMaxBonds]) {
    const int nci = flags_num_conn(s.flags);
#pragma unroll
    for (int b = 0; b < kMaxBonds; ++b) bt[b] = b < nci ? c.A.btgt[b * c.cellCap + s.aidx] : -1;
}

__device__ __forceinline__ bool is_bonded(const int bt[kMaxBonds], int jLocal) {
    bool bonded = false;
#pragma unroll
    for (int b = 0; b < kMaxBonds; ++b) bonded = bonded || (bt[b] == jLocal);
    return bonded;
}

// Barrier reflection, applyForces, and the end-of-step writes of one cell.  A bonded or barrier
// cell is marked staged for the bond kernels of the step.
template <bool kFluid>
__device__ __forceinline__ void cell_finish(const Ctx& c, const DevWorld& w, const DevParams& P, int wi, const Nb& s,
                                            int slot, const int bt[kMaxBonds], Acc& a, int bOld = -1) {
    const int cap = c.cellCap;
    const float Wf = float(w.W), Hf = float(w.H);
    const int i = s.aidx, k = s.lidx;
    const f2 pi = s.pos, vi = s.vel;
    const uint32_t fi = s.flags;
    const int nci = flags_num_conn(fi);
    const bool bari = flags_barrier(fi);
    f2 F = a.F, pc = a.pc;
    if constexpr (kFluid) {
        if (a.cb >= 0) {  // barrier reflection, CellProcessor.cuh:234-274
            const int cb = a.cb;
            const float cbDist = a.cbDist;
            const f2 pb = to_f2(c.A.pos[cb]);
            const f2 vb = to_f2(c.A.vel[cb]);
            const int nb = flags_num_conn(c.A.flags[cb]);
            f2 rr = {0.0f, 0.0f};
            if (nb <= 1) {
                rr = torus_delta(pi, pb, Wf, Hf);
            } else {
                const float angleToCell = angle_of(torus_delta(pi, pb, Wf, Hf));
                for (int q = 0; q < nb; ++q) {
                    const f2 o1 = to_f2(c.A.pos[w.cellOff + c.A.btgt[q * cap + cb]]);
                    const f2 o2 = to_f2(c.A.pos[w.cellOff + c.A.btgt[((q + 1) % nb) * cap + cb]]);
                    const float a1 = angle_of(torus_delta(o1, pb, Wf, Hf));
                    const float a2 = angle_of(torus_delta(o2, pb, Wf, Hf));
                    if (angle_between(a1, a2, angleToCell)) {
                        rr = sub(o2, o1);
                        rot_ccw(rr);
                        break;
                    }
                }
            }
            const f2 vr = sub(vi, vb);
            const float dd = dot2(vr, rr);
            if (dd < 0.0f) {
                const float trs = fmaxf(0.05f, lensq(rr));
                const float td = fmaxf(0.05f, cbDist);
                F = add(F, dvd(sub(add(sub(vr, dvd(mul(mul(rr, 2.0f), dd), trs)), vb), vi), td));
            }
        }
        F = add(F, add(mul(a.Fp, P.pressure), mul(a.Fv, P.viscosity)));
        pc = add(pi, a.D);
    }

    // the cell in the end-of-step order; bond targets stay in start-of-step indices until the
    // first connection pass renumbers them
    c.B.flags[k] = fi;
    c.B.slot[k] = slot;
    if constexpr (kFluid) c.B.dens[k] = 1.0f / a.rho;
    float stiff = 0.0f;
    if constexpr (kFluid) {
        // (unrolled: a loop to nci would index bt at run time and place it in scratch memory)
#pragma unroll
        for (int b = 0; b < kMaxBonds; ++b)
            if (b < nci) {
                c.B.btgt[b * cap + k] = bt[b];
                c.B.brest[b * cap + k] = c.A.brest[b * cap + i];
                c.B.bang[b * cap + k] = c.A.bang[b * cap + i];
            }
        if (nci > 0) stiff = c.stiff[w.cellOff + slot];
    } else {
        // (collision worlds are mostly bonded cells: their bond data is loaded before any of it
        // is stored, so that the loads are in flight together)
        float brest[kMaxBonds], bang[kMaxBonds];
#pragma unroll
        for (int b = 0; b < kMaxBonds; ++b) {
            brest[b] = b < nci ? c.A.brest[b * cap + i] : 0.0f;
            bang[b] = b < nci ? c.A.bang[b * cap + i] : 0.0f;
        }
        stiff = nci > 0 ? c.stiff[w.cellOff + slot] : 0.0f;
#pragma unroll
        for (int b = 0; b < kMaxBonds; ++b)
            if (b < nci) {
                c.B.btgt[b * cap + k] = bt[b];
                c.B.brest[b * cap + k] = brest[b];
                c.B.bang[b * cap + k] = bang[b];
            }
    }
    if (nci > 0) {
        c.bstiff[k] = stiff;
        c.bonded[i] = make_float4(pc.x, pc.y, stiff, __int_as_float(k));
    }
    // checkForces (CellProcessor.cuh:367-386): a bonded cell whose force is above cellMaxForce loses
    // all its bonds with probability cellMaxForceDecayProb (deleting the bonds of an unbonded cell
    // would change nothing)
    // (the per-colour threshold is read from memory: indexing the register copy of the
    // parameters by a run-time colour would place the whole copy in scratch memory)
    uint8_t stage = bari || nci != 0 ? kStagedCell : 0;
    if (P.decayProb > 0.0f && nci > 0 && !bari && lensq(F) > c.params[wi].maxForceSq[flags_color(fi)]) {
        const unsigned long long id = c.cid[w.cellOff + slot];
        if (uniform_draw(w.seed, c.ctr[wi].timestep, id, kStreamForceDecay) < P.decayProb) stage |= kDropBonds;
    }
    f2 v = vi;
    if (!bari) {  // applyForces
        v = add(v, F);
        if (lensq(v) > P.maxVelSq) v = mul(unit(v), P.maxVelocity);
    }
    if (!bari && nci == 0) {
        // no bonds: both connection-force passes yield zero, so the Verlet position and velocity
        // updates and friction of this step are applied here with the same operations
        const f2 zero = {0.0f, 0.0f};
        const float dt = P.dt;
        const f2 p2 = torus_pos(add(pc, add(mul(v, dt), mul(mul(mul(zero, dt), dt), 0.5f))), w.W, w.H);
        const f2 acc = mul(add(zero, zero), 0.5f);
        v = add(v, mul(acc, dt));
        v = mul(v, 1.0f - P.friction);
        c.B.pos[k] = to_float2(p2);
        c.B.vel[k] = to_float2(v);
        bin_next(c, w, k, p2, bOld >= 0 ? bOld : cell_bin_of(w, pi) - w.binOff);
    } else {
        c.B.pos[k] = to_float2(pc);
        c.B.vel[k] = to_float2(v);
    }
    if (w.bondWork) c.stage[k] = stage;
}

// One cell, neighbours visited one after another (forEachNb calls visit(o) in stencil order).
template <bool kFluid, class ForEach>
__device__ __forceinline__ void cell_direct(const Ctx& c, const DevWorld& w, const DevParams& P, int wi, const Nb& s,
                                            ForEach&& forEachNb) {
    const float Wf = float(w.W), Hf = float(w.H);
    int bt[kMaxBonds];
    load_bonds(c, s, bt);
    Acc a;
    acc_init(a, s);
    forEachNb([&](const Nb& o) {
        if (!is_neighbor<kFluid>(s, o, Wf, Hf, P.reachSq)) return;
        float t[kPairTerms];
        const uint32_t f = pair_term<kFluid>(c, w, P, wi, s, o, is_bonded(bt, o.aidx - w.cellOff), t, true,
                                             [&] { return make_int2(s.lidx, o.lidx); });
        acc_add<kFluid>(a, f, t);
    });
    cell_finish<kFluid>(c, w, P, wi, s, c.A.slot[s.aidx], bt, a);
}

}  // namespace alien
