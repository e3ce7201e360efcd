// engine_types.hpp — device-visible layout of a world set.
//
// A world set is any number of independent worlds stored back to back in one segmented SoA.  A
// plain simulation is a world set of one world; the batch and the server use the same kernels.
// Every index stored in a world's arrays (bond targets, cell slots, last absorbed cell, particle
// slots) is local to that world, so a world's ranges can be copied between sets unchanged.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace alien {

constexpr int kMaxBonds = 6;
constexpr int kColors = 7;
constexpr int kParticleBin = 8;  // edge of the energy-particle bins, in world units
constexpr int kNone = -1;
constexpr int kClaimFree = 0x7fffffff;
// binOf: the cell's next bin, counted from its world's first (below 2^28: bins are at least two units wide
// and worlds span at most 2^30 square units), and in the bits above it how the cell came there: 0 it stayed,
// 1 to 9 from the bin around in that direction, kFarCode from further
constexpr int kMoveShift = 28;
constexpr uint32_t kBinMask = (1u << kMoveShift) - 1u, kFarCode = 15u, kFarMove = kFarCode << kMoveShift;
// Bins per wave of the cells' map (a group): 256, in sets with more than kDenseBins cells per bin 64, with twice that
// 16 (Ctx::groupShift).  With many cells to a bin there are few bins, and a wave goes over the cells of its own and
// of the rows next to them: 262k cells at nine to a bin, 114 waves for the whole map, 173 us of a step of 329 with
// 256, 251 with 64, 224 with 16; at four to a bin 76, 58 and 55; at 16 to a bin 286, 250 and 236.  At one to a bin
// the groups' sums cost more: 4M cells 151 us with 256, 190 with 64; 0.84M in bodies 224 and 235.
// A world's bins are padded to a multiple of kGroupBins.
constexpr int kGroupBins = 256, kDenseBins = 3;
constexpr int kBinOfPad = 576;     // entries of binOf that may be read (and not used) past the last cell
constexpr int kSuperGroups = 256;  // groups per sum of groups
// Cells per wave of the fluid pass, as a power of two: 64, and in sets with fewer than a wave per SIMD (1024)
// half as many, down to 16, as long as they give a SIMD one wave at most.  The pass is one wave's latency
// there (10751 cells in bodies: a step of 106 us with 64, 97 with 32, 92 with 16); with more cells the
// wave's fixed work counts (134k cells in bodies: 159, 157 and 162 us; 256k free ones: 22, 26 and 32 us).
constexpr int kFluidShiftMin = 4;
// waves of the neighbour passes for a group of units of two edge bins (k_neighbor.hip); units per group: as few as
// keep a set's edge waves at kEdgeWavesMost, two and a half for a SIMD, or less.  A step, us: 150k fluid cells of
// 707 x 1010 units 24.4 with 4096 as the limit, 21.7 with 2048; cells in bodies of 926 x 1115 units 145.2 with 2048,
// 141.9 with 2560, 141.4 with 4096, of 1024 x 1024 units 133.2, 133.2 and 136.5; 17k fluid cells of 214 x 296 units
// 16.1 with 1024, 16.9 with 512, 20.2 with 256.
constexpr int kEdgeWaves = 8, kEdgeUnitsMost = 8, kEdgeWavesMost = 2560;
constexpr int kXcdCount = 8;  // XCDs of an MI355X: workgroup b of a launch runs on XCD b % 8
// Size limits of one world set.  Cell indices, bin offsets and the bond planes ([kMaxBonds][cap],
// addressed as b * cap + x) are 32-bit ints in the kernels, so a set holds at most
// (2^31 - 1) / kMaxBonds cells; particle indices and the uint32 bin scan over cells plus particles
// stay in range with at most 2^30 particles.  At ~530 B per cell the cell limit is ~190 GB
// of the 288 GB of HBM.
constexpr int64_t kMaxSetCells = (int64_t(0x7fffffff)) / kMaxBonds;  // 357,913,941
constexpr int64_t kMaxSetParticles = int64_t(1) << 30;

// cell flags word
constexpr uint32_t kNumConnMask = 0xFu;        // bits 0..3
constexpr uint32_t kMaxConnShift = 4;          // bits 4..7
constexpr uint32_t kColorShift = 8;            // bits 8..15
constexpr uint32_t kBarrierBit = 1u << 16;
constexpr uint32_t kDetachedBit = 1u << 17;
// stage byte of a cell (Ctx::stage)
constexpr uint8_t kStagedCell = 1, kDropBonds = 2, kMarkedCell = 4;
// particle flags byte
constexpr uint8_t kParticleColorMask = 0x7F;
constexpr uint8_t kParticleDead = 0x80;
// ids of the particles cell radiation creates: this bit, the timestep (bits 32-61) and the local
// index of the emitting cell (bits 0-31)
constexpr unsigned long long kCreatedParticleId = 1ull << 63;
// with this bit too: the particle came from a split (timestep in bits 32-61, index of the particle
// that split in bits 0-31)
constexpr unsigned long long kSplitParticleId = 1ull << 62;

__host__ __device__ inline int flags_num_conn(uint32_t f) { return int(f & kNumConnMask); }
__host__ __device__ inline int flags_max_conn(uint32_t f) { return int((f >> kMaxConnShift) & 0xFu); }
__host__ __device__ inline int flags_color(uint32_t f) { return int((f >> kColorShift) & 0xFFu); }
__host__ __device__ inline bool flags_barrier(uint32_t f) { return (f & kBarrierBit) != 0; }
__host__ __device__ inline int flags_detached(uint32_t f) { return (f & kDetachedBit) ? 1 : 0; }
__host__ __device__ inline uint32_t flags_with_num_conn(uint32_t f, int n) {
    return (f & ~kNumConnMask) | (uint32_t(n) & kNumConnMask);
}

// per-world simulation parameters (physics subset of SimulationParameters)
struct DevParams {
    float dt;
    int motion;  // 0 fluid, 1 collision
    float smoothing, viscosity, pressure;
    float collisionDistance, repulsion;
    float friction, maxVelocity, minDistance, fusionVelocity, maxBindingEnergy;
    float maxBindingDistance[kColors];
    float absorption[kColors];
    // neighbour predicate without the square root: sqrt(s) <= R  <=>  s <= reachSq, where R is the
    // interaction radius (2 h for fluid, cellMaxCollisionDistance for collision) and reachSq the
    // largest float whose correctly rounded square root does not exceed R
    float reachSq;
    // the same for the other length comparisons of the pass: |v| > maxVelocity <=> |v|^2 > maxVelSq,
    // |v| > 0.5 <=> |v|^2 > fastSq, |dv| < fusionVelocity <=> |dv|^2 <= fusionBelowSq,
    // |d| < minDistance <=> |d|^2 <= overlapBelowSq
    float maxVelSq, fastSq, fusionBelowSq, overlapBelowSq;
    float invH, invH2, invH3;  // 1/h, 1/h^2, 1/h^3 (fluid)
    float innerFriction;       // applied every third step to bonded cells (0: off)
    float decayProb;           // cellMaxForceDecayProb (0: off)
    float maxForceSq[kColors];  // |F| > cellMaxForce  <=>  |F|^2 > maxForceSq (as reachSq)
    float minEnergy[kColors];   // cellMinEnergy
    // cell radiation (CellProcessor.cuh:725-773); radiates: radiationProb > 0 and some colour has
    // a positive high-radiation factor or age strength
    int radiates;
    int splits;                  // some colour has a finite particleSplitEnergy
    float splitEnergy[kColors];  // particleSplitEnergy (RadiationProcessor::splitting)
    float radProb, radVelMul, radVelPert;
    int radMinAge[kColors];
    float highRadFactor[kColors], highRadMinEnergy[kColors], radAgeStrength[kColors];
};

// per-world geometry and placement in the set
struct DevWorld {
    int W, H;
    int binSize, nbx, nby;  // cell bins (row-major)
    int binShift;           // log2(binSize) when binSize is a power of two, else -1
    int pnbx, pnby;         // particle bins of kParticleBin units
    int cellOff, numCells;  // hot and cold cell arrays
    int binOff;             // first cell bin in the combined bin arrays
    int pbinOff;            // first particle bin in the combined bin arrays
    int partOff, partCap;   // particle arrays
    int bondWork;           // 1 if a bonded or barrier cell exists or can appear by fusion
    int livingWork;         // 1 if living states are tracked on the device (see WorldSet::build)
    unsigned long long seed;  // key of the world's random draws
    // timestep at which the cells' base ages (ageBase) were taken: a non-barrier cell ages by one
    // every step, so its age at the start of step t is ageBase + (t - ageTs)
    unsigned long long ageTs;
    int active;  // 0: left out of every launch (frozen)
};

// per-world device counters
struct DevCounters {
    unsigned long long timestep;
    int numParticles;  // live particles at [partOff, partOff + numParticles)
    int pad;
};

// global counters of one step (reset at the start of every step)
struct StepCounters {
    int candidates;  // fusion candidate pairs
    int errors;      // bit 0: candidate list overflow; bit 1: map-build look-back gave up;
                     // bit 2: a world's particles exceeded its particle capacity
    int liveParticles;  // energy particles alive after this step's particle sort, all worlds
    // neighbour-pass paths since the data was set (not reset per step): waves with too many candidates to
    // stage or to list at once, and the cells that went over their candidates alone
    unsigned long long fallbackChunks;
    unsigned long long directCells;
};

// hot per-cell / per-particle state; two of these exist and alternate every step
struct HotBuffers {
    float2* pos;
    float2* vel;
    float* dens;  // 1 / density of a fluid cell (set to 1 when a world changes its parameters, motion included)
    uint32_t* flags;
    int* slot;    // local cold slot of the cell (stable identity)
    int* btgt;    // [kMaxBonds][cellCap] local logical index of the bond partner
    float* brest; // [kMaxBonds][cellCap]
    float* bang;  // [kMaxBonds][cellCap]
    float2* ppos;
    float2* pvel;
    float* pen;
    int* plast;   // local cold slot of the last absorbing cell, kNone if none
    int* pslot;   // local particle slot (host-side selection state), kNone for created particles
    uint8_t* pflags;
    unsigned long long* pid;  // particle id
};

// a particle emitted by cell radiation, in its staging slot (one record: one cache line touched to
// write it and one to read it)
struct __align__(16) StagedParticle {
    float2 pos;  // pre-move position
    float2 vel;
    float energy;
    uint32_t color;  // | kStagedPending for a split half not yet in the particle arrays
    unsigned long long id;
};
// a split half waits in its record from the end of one step to the movement of the next (and is
// part of the world's state in between: get_data, statistics and rebuilt sets include it)
constexpr uint32_t kStagedPending = 0x100u;

// pass-through fields of a cell that no kernel of the step reads (genomeComplexity as its bits)
struct CellExtra {
    uint32_t mutationId, genomeComplexity;
    uint8_t cellFunction, ancestorMutationId, selected, pad;
};

// Cells that the map cannot find near their new bin (k_sort.hip): a list per bin, and of the bins with
// more than kFarWalk of them a list of their parts of 64.
constexpr int kFarWalk = 16;
struct FarCells {
    int* head;   // [numCellBins] one of the bin's, kNone without any; Ctx::farLink goes on
    int* count;  // [numCellBins]
    int* group;  // [groups] whether the group's bins have any
    int* total;  // entries in the list
    int2* list;  // (global bin, part); one array for both steps: read before it is written
};

// Every launch of a forked graph copies the context (launch.hip): a step of a small radiating world, 70 us in nine
// launches, took 2.5 us more with 128 bytes more in it, so its numbers lie together without gaps.
struct Ctx {
    int numWorlds;
    int cellCap;  // total cells (= sum of numCells)
    int partCap;  // total particle slots
    int numBins;  // cell bins + particle bins of all worlds
    int numCellBins;  // cell bins of all worlds, each world's padded to a multiple of kGroupBins
    int cellCount;    // cells of all worlds
    int groupShift;   // 1 << groupShift bins per group of the map: 8, 6 or 4
    int candCap;
    int timestepAdvanced;  // 1 if the step's map scan advanced the worlds' timesteps
    // Particles emitted by cell radiation during a step are written at partStage + (cell index),
    // behind the worlds' particle ranges (partStage = 0: no staging area), and enter the step's
    // particle map like the live particles.
    int partStage;
    // Particles split off at the end of a step: staging slot splitStage + k for the particle at k
    // (0: no split staging area), record splitStaged[k]; they enter the next step's map behind the
    // particles that lived and before that step's radiation
    int splitStage;
    int blockThreads;        // cells, bins or living cells per entry of cellBlocks .. livingBlocks
    int partBlockParticles;  // particles per entry of partBlocks
    int fluidShift, collideShift;     // waves of the fluid / collision pass take 1 << shift cells
    int edgeUnits, collideEdgeUnits;  // edge units that kEdgeWaves waves share
    const DevWorld* worlds;
    const DevParams* params;
    DevCounters* ctr;
    StepCounters* sc;
    HotBuffers A;  // state at the start of the step (read)
    HotBuffers B;  // state at the end of the step (written)
    float* energy;  // cold [cellCap], indexed by cellOff + slot
    float* stiff;   // cold [cellCap]
    unsigned long long* cid;  // cold [cellCap]: cell id (key of the cell's random draws)
    uint32_t* ageBase;        // cold [cellCap]: cell age at the world's ageTs
    StagedParticle* staged;  // [cellCap]: the particle of staging slot partStage + i at staged[i]
    StagedParticle* splitStaged;
    // living states of the worlds with livingWork, cold by slot: `living` holds the state at the
    // start of the step, `livingNext` the other buffer (the step's phases alternate between the
    // two and leave the end-of-step state in `livingNext`, the next step's `living`)
    uint8_t* living;
    uint8_t* livingNext;
    uint32_t* activation;     // cold [cellCap]: activationTime (worlds with livingWork)
    uint32_t* creature;       // cold [cellCap]: creatureId (worlds with livingWork)
    uint8_t* stretched;       // [cellCap] end-of-step staged cell had a bond beyond cellMaxBindingDistance
    int* binOf;     // [cellCap] next bin of A-cell i, and how it came there (kBinMask, kMoveShift)
    int* pbinOf;    // [partCap] global bin of A-particle i, -1 if dead
    // Particles per bin: counted with atomics by the kernels that produce the end-of-step particle
    // positions (and by seeding), brought back to zero by the particle scatter.
    uint32_t* count;      // [numBins] start-of-step state
    uint32_t* countNext;  // [numBins] end-of-step state (next step's `count`)
    const int* groupWorld;  // [numCellBins / kGroupBins] the bins' world
    // Cells that the groups of cell bins, and kSuperGroups of those, gained (or lost) since the
    // last map; ...Next: for the next step (built during this step)
    int* groupSum;
    int* groupSumNext;
    int* superSum;
    int* superSumNext;
    uint32_t* start;      // [numBins + 1] offsets of this step's map (relative to the world's first bin's)
    const uint32_t* startPrev;  // [numBins + 1] the last step's map
    // far cells of this step's map, and of the next (entered during this step)
    FarCells far, farNext;
    int* farLink;  // [cellCap] the bin's next far cell (kNone ends a list)
    // one-pass scan of the particle bins: per tile of bins a status word (flag, launch epoch, sum), the launch epoch
    // and the tile ticket
    unsigned long long* mapStatus;
    uint32_t* mapEpoch;
    uint32_t* mapTicket;
    int* sorted;   // [cellCap] map order (bin, then previous index) -> A index
    float4* bonded;  // [cellCap] by A index, of bonded cells: position after the neighbour pass, stiffness, new index
    int* psorted;  // [partCap]
    uint8_t* pcode;  // [partCap] by map position: the particle's slot inside its bin before the movement
    // [cellCap] kStagedCell: the end-of-step cell is staged (bonded or barrier at the neighbour pass);
    // kDropBonds: it loses all its bonds at the end of the step; kMarkedCell: it or a bond partner
    // does.  The neighbour pass writes the byte of every cell of the bond-work worlds.
    uint8_t* stage;
    float2* own;    // [cellCap]
    int4* lists;    // [2 * cellCap] on angle steps, of bonded cells: their bond targets (-1: none), flags, unused
    float4* moved;  // [cellCap] position after the neighbour pass, and displacement of the first Verlet step
    float* bstiff;  // [cellCap] stiffness of a bonded cell in end-of-step order (written by the neighbour pass)
    float2* s2;     // [cellCap] connection force of the first pass
    float2* out1;  // [kMaxBonds][cellCap]
    float2* out2;
    uint32_t* valid;  // [cellCap]
    unsigned long long* claim;  // [cellCap]
    int4* cand;                 // [candCap] (a, b, world, live)
    int* want;        // [partCap]
    int* fclaim;      // [partCap]
    int* absorbCell;  // [partCap]
    int* cclaim;      // [cellCap]
    const int2* cellBlocks;  // per block: (world, first global cell index)
    const int2* bondBlocks;  // the same over the worlds with bond work
    const int2* pbinBlocks;  // per block: (world, first global bin index) over particle bins
    // per block of partBlockParticles live particles: (world, first global particle index), over
    // the active worlds' live ranges; written by the host when the tables are built and by the
    // particle bin sort for the ranges it publishes (*numPartBlocks entries)
    int2* partBlocks;
    int* numPartBlocks;
    const int2* fluidBlocks;  // per workgroup of the fluid pass: (world, its first wave)
    const int2 *collideBlocks, *collideEdgeBlocks;  // the same of the collision pass
    const int2* edgeBlocks;  // per workgroup: (world, its first edge wave), see k_neighbor.hip
    const int2* livingBlocks;  // per block: (world, first global cell index) over livingWork worlds
};

}  // namespace alien
