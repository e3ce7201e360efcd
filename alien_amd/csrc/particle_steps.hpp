// particle_steps.hpp — the per-step work on energy particles: their map, movement, particle-particle
// fusion, absorption into cells and reflection at barrier cells (ALIEN RadiationProcessor::movement/
// collision, source/EngineGpuKernels/RadiationProcessor.cuh:61-170).  Each is the body of a kernel of
// its own beside the fluid pass (k_particles.hip), and a part of the launches of the bond phase
// (k_sort.hip, k_neighbor.hip, k_bonds.hip).
//
// The reference resolves concurrent fusions and absorptions with tryLock and skips on contention.
// Here the outcome is fixed (R8): a particle targets the winner of its 1x1 slot in the particle map
// (lowest index, pre-move position); it fuses only into a target that is not fusing itself, and a
// sink accepts the lowest-index fusing particle; a cell accepts the lowest-index absorbing
// particle.  Claims are atomicMin on indices, which is order independent.
#pragma once

#include "kernels_common.hpp"

namespace alien {

// particle i (A index or staging slot) of bin gb to its place in the map (the order inside the bin
// is fixed by the bin sort)
__device__ __forceinline__ void scatter_particle(const Ctx& c, const DevWorld& w, int gb, int i) {
    const int rel = int(c.start[gb] - c.start[w.pbinOff]) + int(atomicSub(&c.count[gb], 1u)) - 1;
    if (rel < w.partCap)
        c.psorted[w.partOff + rel] = i;
    else
        atomicOr(&c.sc->errors, 4);  // (the host keeps room for a step's emissions: not reached)
}

__device__ __forceinline__ void part_scatter(const Ctx& c, Span at) {
    for_live_particles(c, at, [&](int, const DevWorld& w, int i) {
        const int gb = c.pbinOf[i];
        if (gb >= 0) scatter_particle(c, w, gb, i);
        // the particle split off particle i at the end of the last step (cleared once read)
        if (c.splitStage > 0) {
            const int st = c.splitStage + i;
            const int g2 = c.pbinOf[st];
            if (g2 >= 0) {
                c.pbinOf[st] = -1;
                scatter_particle(c, w, g2, st);
            }
        }
    });
}

// the particle cell i emitted this step, from its staging slot (cleared once read)
__device__ __forceinline__ void part_scatter_staged(const Ctx& c, const DevWorld& w, int i) {
    const int st = c.partStage + i;
    const int gb = c.pbinOf[st];
    if (gb < 0) return;
    c.pbinOf[st] = -1;
    scatter_particle(c, w, gb, st);
}

// Sort the entries [s, e) of a particle bin ascending.  Up to 16 in registers, every entry to its rank
// among the bin's (their indices are distinct); no register array is indexed at run time, which would
// place it in scratch memory.
template <int kMax> __device__ __forceinline__ void sort_ranked(int* arr, int s, int n) {
    int v[kMax];
#pragma unroll
    for (int k = 0; k < kMax; ++k) v[k] = k < n ? arr[s + k] : 0x7fffffff;
#pragma unroll
    for (int k = 0; k < kMax; ++k) {
        int rank = 0;
#pragma unroll
        for (int j = 0; j < kMax; ++j) rank += v[j] < v[k] ? 1 : 0;
        if (k < n) arr[s + rank] = v[k];
    }
}
__device__ __forceinline__ void sort_part_bin(int* arr, int s, int e) {
    const int n = e - s;
    if (n <= 1) return;
    if (n <= 4) {
        sort_ranked<4>(arr, s, n);
    } else if (n <= 8) {
        sort_ranked<8>(arr, s, n);
    } else if (n <= 16) {
        sort_ranked<16>(arr, s, n);
    } else {
        for (int k = s + 1; k < e; ++k) {
            const int x = arr[k];
            int j = k - 1;
            while (j >= s && arr[j] > x) {
                arr[j + 1] = arr[j];
                --j;
            }
            arr[j + 1] = x;
        }
    }
}

// Particle map in logical order (the particles cell radiation emitted this step, from their staging
// slots, sort behind every live particle's index); also publishes the new number of live
// particles per world and the table of live particle blocks.  One thread per bin of the bin block
// table, in workgroups of any size that divides its blocks'.
__device__ __forceinline__ void part_binsort(const Ctx& c, Span at) {
    if (at.block == 0) {
        for (int wi = threadIdx.x; wi < c.numWorlds; wi += blockDim.x) {
            const DevWorld& w = c.worlds[wi];
            const int live = min(int(c.start[w.pbinOff + w.pnbx * w.pnby] - c.start[w.pbinOff]), w.partCap);
            c.ctr[wi].numParticles = live;
            if (live > 0) atomicAdd(&c.sc->liveParticles, live);
        }
        __syncthreads();
        // the table of live particle blocks, world by world
        const int ppb = c.partBlockParticles;
        int base = 0;
        for (int wi = 0; wi < c.numWorlds; ++wi) {
            const DevWorld& w = c.worlds[wi];
            if (!w.active) continue;
            const int nb = (c.ctr[wi].numParticles + ppb - 1) / ppb;
            for (int j = int(threadIdx.x); j < nb; j += int(blockDim.x)) c.partBlocks[base + j] = make_int2(wi, w.partOff + j * ppb);
            base += nb;
        }
        if (threadIdx.x == 0) *c.numPartBlocks = base;
    }
    const int parts = c.blockThreads / int(blockDim.x);  // workgroups per table entry
    const int2 blk = c.pbinBlocks[at.block / parts];
    const DevWorld w = c.worlds[blk.x];
    const int gb = blk.y + (at.block % parts) * int(blockDim.x) + int(threadIdx.x);
    if (gb >= w.pbinOff + w.pnbx * w.pnby) return;
    int s, e;
    part_bin_range(c, w, gb - w.pbinOff, s, e);
    sort_part_bin(c.psorted, s, e);
}

// A particle's slot inside its bin, four bits each way (the last bins reach up to 15 units)
__device__ __forceinline__ uint32_t slot_code(const DevWorld& w, int sx, int sy) {
    const int bx = min(sx / kParticleBin, w.pnbx - 1), by = min(sy / kParticleBin, w.pnby - 1);
    return uint32_t(sx - bx * kParticleBin) | uint32_t(sy - by * kParticleBin) << 4;
}

// The movement of the particles in map order (RadiationProcessor.cuh:61-70: position += velocity *
// dt on the torus) into the end-of-step arrays, one thread per particle of the new live ranges; a
// particle emitted this step comes from its staging record.
__device__ __forceinline__ void part_move(const Ctx& c, Span at) {
    // (the start-of-step and end-of-step arrays are distinct)
    const float2* __restrict__ appos = c.A.ppos;
    const float2* __restrict__ apvel = c.A.pvel;
    const float* __restrict__ apen = c.A.pen;
    const int* __restrict__ aplast = c.A.plast;
    const int* __restrict__ apslot = c.A.pslot;
    const uint8_t* __restrict__ apflags = c.A.pflags;
    const unsigned long long* __restrict__ apid = c.A.pid;
    float2* __restrict__ bppos = c.B.ppos;
    float2* __restrict__ bpvel = c.B.pvel;
    float* __restrict__ bpen = c.B.pen;
    int* __restrict__ bplast = c.B.plast;
    int* __restrict__ bpslot = c.B.pslot;
    uint8_t* __restrict__ bpflags = c.B.pflags;
    unsigned long long* __restrict__ bpid = c.B.pid;
    for_live_particles(c, at, [&](int wi, const DevWorld& w, int k) {
        const float dt = c.params[wi].dt;
        const int src = c.psorted[k];
        const auto code = [&](f2 p) {  // the pre-move slot
            int sx, sy;
            slot_of(p, w.W, w.H, sx, sy);
            c.pcode[k] = uint8_t(slot_code(w, sx, sy));
        };
        const bool rad = c.partStage > 0 && src >= c.partStage;
        if (rad || (c.splitStage > 0 && src >= c.splitStage)) {
            const StagedParticle r = rad ? c.staged[src - c.partStage] : c.splitStaged[src - c.splitStage];
            if (!rad) c.splitStaged[src - c.splitStage].color = r.color & ~kStagedPending;  // (in the arrays now)
            const f2 v = to_f2(r.vel);
            code(to_f2(r.pos));
            bppos[k] = to_float2(torus_pos(add(to_f2(r.pos), mul(v, dt)), w.W, w.H));
            bpvel[k] = r.vel;
            bpen[k] = r.energy;
            bplast[k] = kNone;
            bpslot[k] = kNone;
            bpflags[k] = uint8_t(r.color & kParticleColorMask);
            bpid[k] = r.id;
            return;
        }
        const f2 v = to_f2(apvel[src]), p = to_f2(appos[src]);
        code(p);
        bppos[k] = to_float2(torus_pos(add(p, mul(v, dt)), w.W, w.H));
        bpvel[k] = to_float2(v);
        bpen[k] = apen[src];
        bplast[k] = aplast[src];
        bpslot[k] = apslot[src];
        bpflags[k] = apflags[src];
        bpid[k] = apid[src];
    });
}

// The particle map winner of the slot of position p (R2): the first particle of the bin whose
// pre-move slot matches; particle k fuses into it when it is another particle closer than sqrt(0.5)
// after the move.  Returns the target or -1.  (The movement leaves the slots in map order, a byte each:
// the search through map and positions was a chain of two loads for every entry; steps of 134k cells
// with default parameters 148.4 -> 137.3 us, of 1M radiating ones 142.3 -> 134.2.)
__device__ __forceinline__ int particle_target(const Ctx& c, const DevWorld& w, int k, f2 p) {
    int sx, sy;
    slot_of(p, w.W, w.H, sx, sy);
    const uint32_t code = slot_code(w, sx, sy);
    int s, e;
    part_bin_range(c, w, part_bin_local(w, sx, sy), s, e);
    int t = -1;
    for (int m = s; m < e && t < 0; m += 8) {
        uint32_t x[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) x[q] = m + q < e ? uint32_t(c.pcode[m + q]) : 0x100u;
#pragma unroll
        for (int q = 7; q >= 0; --q) t = x[q] == code ? m + q : t;
    }
    return t >= 0 && t != k && lensq(sub(p, to_f2(c.B.ppos[t]))) < 0.5f ? t : -1;
}

// Targets and fusion claims in one pass: a particle claims its target when the target does not
// fuse itself, which it finds by computing the target's own target (the same function of the same
// moved positions; fusing particles are rare).
__device__ __forceinline__ void part_target(const Ctx& c, Span at) {
    for_live_particles(c, at, [&](int, const DevWorld& w, int k) {
        const f2 p = to_f2(c.B.ppos[k]);
        const int want = particle_target(c, w, k, p);
        c.want[k] = want;
        if (want >= 0 && particle_target(c, w, want, to_f2(c.B.ppos[want])) < 0) atomicMin(&c.fclaim[want], k);
        // cell hit this step: lowest-index cell of the slot at map-build time (cellMap.getFirst),
        // the first of the bin's cells in map order (a bin holds its cells by previous index)
        int cell = -1;
        if (want < 0) {
            const f2 q = add(p, to_f2(c.B.pvel[k]));
            int qx, qy;
            slot_of(q, w.W, w.H, qx, qy);
            int cs, ce;
            cell_bin_range(c, w, cell_bin_local(w, qx, qy), cs, ce);
            // (four cells' loads in flight)
            for (int m = cs; m < ce && cell < 0; m += 4) {
                f2 a[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) a[j] = to_f2(c.A.pos[c.sorted[min(m + j, ce - 1)]]);
#pragma unroll
                for (int j = 3; j >= 0; --j) {
                    int ax, ay;
                    slot_of(a[j], w.W, w.H, ax, ay);
                    if (m + j < ce && ax == qx && ay == qy) cell = m + j;
                }
            }
        }
        c.absorbCell[k] = cell;
    });
}

__device__ __forceinline__ void part_apply(const Ctx& c, Span at) {
    for_live_particles(c, at, [&](int wi, const DevWorld& w, int k) {
        const DevParams& P = c.params[wi];
        const int q = c.fclaim[k];
        if (q != kClaimFree) {
            // sink: merge the lowest-index particle fusing into it (RadiationProcessor.cuh:86-93)
            c.fclaim[k] = kClaimFree;
            const float eq = c.B.pen[q], ek = c.B.pen[k];
            if (eq > kNearZero && ek > kNearZero) {
                const float f1 = eq / (eq + ek);
                const f2 vq = to_f2(c.B.pvel[q]), vk = to_f2(c.B.pvel[k]);
                c.B.pvel[k] = to_float2(add(mul(vq, f1), mul(vk, 1.0f - f1)));
                c.B.pen[k] = ek + eq;
                c.B.plast[k] = kNone;
                c.B.pen[q] = 0.0f;
                c.B.pflags[q] = uint8_t(c.B.pflags[q] | kParticleDead);
            }
            c.absorbCell[k] = -1;
            return;
        }
        if (c.want[k] >= 0) return;
        const int cm = c.absorbCell[k];
        if (cm < 0) return;
        // the cell as the neighbour pass found it (through the map: a barrier cell does not move
        // or change speed in that pass, and no cell changes its flags or slot there)
        const int ca = c.sorted[cm];
        const uint32_t fc = c.A.flags[ca];
        if (flags_barrier(fc)) {  // reflection (:99-106)
            const f2 vb = to_f2(c.A.vel[ca]);
            const f2 vr = sub(to_f2(c.B.pvel[k]), vb);
            const f2 rr = torus_delta(to_f2(c.B.ppos[k]), to_f2(c.A.pos[ca]), float(w.W), float(w.H));
            const float d = dot2(vr, rr);
            if (d < 0.0f) {
                const float trs = fmaxf(0.1f, lensq(rr));
                c.B.pvel[k] = to_float2(add(sub(vr, dvd(mul(mul(rr, 2.0f), d), trs)), vb));
            }
            c.absorbCell[k] = -1;
            return;
        }
        if (c.B.plast[k] == c.A.slot[ca] || P.absorption[flags_color(fc) % kColors] < kNearZero) {
            c.absorbCell[k] = -1;
            return;
        }
        atomicMin(&c.cclaim[cm], k);
    });
}

// RadiationProcessor::splitting (RadiationProcessor.cuh:172-204), after absorption: with
// probability 0.01 (R9 draw keyed by the particle id) a particle above particleSplitEnergy of its
// colour halves its energy and splits in two, 1/5 of a random unit vector u either side of its
// position, their velocities its own -/+ u radiationVelocityPerturbation / (E/2 + 1).  The new half
// goes to the split staging slot of the particle's index and into the next step's histogram, so
// that the next map sorts it behind the particles that lived, in index order (R18); its id is
// kCreatedParticleId | kSplitParticleId | timestep << 32 | local index.
__device__ __forceinline__ void split_particle(const Ctx& c, const DevWorld& w, int wi, int k) {
    const DevParams& P = c.params[wi];
    const unsigned long long id = c.B.pid[k];
    const unsigned long long ts = c.ctr[wi].timestep - (c.timestepAdvanced ? 1ull : 0ull);
    if (!(uniform_draw(w.seed, ts, id, kStreamSplit) < 0.01f)) return;
    const int col = c.B.pflags[k] & kParticleColorMask;
    float e = c.B.pen[k];
    if (!(e > P.splitEnergy[col % kColors])) return;
    e = e * 0.5f;
    f2 u = to_f2(unit_vector_of_angle(uniform_draw(w.seed, ts, id, kStreamSplitAngle) * 360.0f));
    const f2 p = to_f2(c.B.ppos[k]);
    const f2 d = {u.x / 5.0f, u.y / 5.0f};
    const f2 other = torus_pos(add(p, d), w.W, w.H);
    const f2 self = torus_pos(sub(p, d), w.W, w.H);
    u = mul(u, P.radVelPert / (e + 1.0f));
    const f2 v = to_f2(c.B.pvel[k]);
    c.B.pen[k] = e;
    c.B.ppos[k] = to_float2(self);
    c.B.pvel[k] = to_float2(sub(v, u));
    StagedParticle r;
    r.pos = to_float2(other);
    r.vel = to_float2(add(v, u));
    r.energy = e;
    r.color = uint32_t(col) | kStagedPending;
    r.id = kCreatedParticleId | kSplitParticleId | ((ts & 0x3fffffffull) << 32) | (unsigned long long)uint32_t(k - w.partOff);
    c.splitStaged[k] = r;
    pbin_for_next_step(c, w, c.splitStage + k, other, c.countNext);
}

// absorption (:108-165); also bins the surviving particles for the next step
__device__ __forceinline__ void part_absorb(const Ctx& c, Span at) {
    for_live_particles(c, at, [&](int wi, const DevWorld& w, int k) {
        const int cm = c.absorbCell[k];
        if (cm >= 0 && c.cclaim[cm] == k) {
            c.cclaim[cm] = kClaimFree;
            const DevParams& P = c.params[wi];
            const int ca = c.sorted[cm];
            const uint32_t fc = c.A.flags[ca];
            const float ra = P.absorption[flags_color(fc) % kColors];
            float e = c.B.pen[k];
            float transfer = e * ra;
            if (e < 0.01f) transfer = e;
            const int cslot = c.A.slot[ca];
            float* ce = &c.energy[w.cellOff + cslot];
            *ce = *ce + transfer;
            e = e - transfer;
            c.B.pen[k] = e;
            if (e < kNearZero)
                c.B.pflags[k] = uint8_t(c.B.pflags[k] | kParticleDead);
            else
                c.B.plast[k] = cslot;
        }
        if (c.B.pflags[k] & kParticleDead) {
            c.pbinOf[k] = -1;
            return;
        }
        if (c.splitStage > 0 && c.params[wi].splits) split_particle(c, w, wi, k);
        pbin_for_next_step(c, w, k, to_f2(c.B.ppos[k]), c.countNext);
    });
}

}  // namespace alien
