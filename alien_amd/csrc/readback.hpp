// readback.hpp — device-side packing of transfer objects (k_readback.hip) and its host plumbing
// (readback.cpp).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <functional>

#include "engine_types.hpp"

namespace alien {

constexpr int kSortTile = 4096;  // keys per workgroup of the radix sort
constexpr int kPartTile = 2048;  // particle entries per workgroup of the live-particle compaction

// ping-pong keys and values, and the digit counts: 256 rows of one count per tile, then 256 totals
struct SortBuffers {
    unsigned long long* keys[2];
    int* vals[2];
    uint32_t* counts;
    static size_t bytes(size_t n) { return 24 * n + 1024 * ((n + kSortTile - 1) / kSortTile + 1); }
    // carved out of `bytes(n)` bytes at p (8-byte aligned)
    static SortBuffers at(void* p, size_t n) {
        SortBuffers b;
        b.keys[0] = static_cast<unsigned long long*>(p);
        b.keys[1] = b.keys[0] + n;
        b.vals[0] = reinterpret_cast<int*>(b.keys[1] + n);
        b.vals[1] = b.vals[0] + n;
        b.counts = reinterpret_cast<uint32_t*>(b.vals[1] + n);
        return b;
    }
};

// one world's cells: arrays from its first cell (hot ones by index, cold ones by slot)
struct PackCells {
    const int *order, *rankOf, *slot;
    const uint32_t* flags;
    const float2 *pos, *vel;
    const int* btgt;
    const float *brest, *bang;
    size_t plane;  // distance of the bond planes
    const unsigned long long* cid;
    const float *energy, *stiff;
    const uint32_t *ageBase, *creature;
    uint32_t steps;        // steps since the ages were taken
    bool stepped;          // any
    const uint8_t* living;  // null: every cell Ready without an activation count
    const uint32_t* activation;
    const CellExtra* extra;  // null: all zero
};

// one world's particles: arrays from its first particle slot
struct PackParticles {
    int np, entries;
    const float2 *ppos, *pvel;
    const float* pen;
    const int* pslot;
    const uint8_t* pflags;
    const unsigned long long* pid;
    const StagedParticle* halves;  // null without splitting
    const uint8_t* selected;       // by particle slot; null: all zero
};

// keys[0], vals[0] sorted by key, stable, over the bits set in `differing`; returns the index of the
// buffers that hold the result
int launch_radix_sort(const SortBuffers& b, int n, unsigned long long differing, hipStream_t s);
// *differing (cleared by the caller) collects the bits in which the keys differ
void launch_cell_keys(const unsigned long long* cid, const int* slotOf, int n, const SortBuffers& b,
                      unsigned long long* differing, hipStream_t s);
void launch_cell_ranks(const unsigned long long* keys, const int* vals, int n, int* rankOf, unsigned long long* equal,
                       hipStream_t s);
void launch_cell_order(const int* slotOf, const int* rankOfSlot, int n, int* order, int* rankOf, hipStream_t s);
void launch_pack_cells(const PackCells& a, int first, int count, void* out, hipStream_t s);
// result[0] the living particles, and with `b` their ids and entries in b, result[1] the bits in which
// the ids differ
void launch_part_keys(const PackParticles& a, uint32_t* tileCount, const SortBuffers* b, unsigned long long* result,
                      hipStream_t s);
void launch_pack_particles(const PackParticles& a, const int* order, int first, int count, void* out, hipStream_t s);

// A pinned transfer buffer of kBytes, from a pool that keeps at most kKept of them for the next caller
// (any thread).
class PinnedBuffer {
public:
    static constexpr size_t kBytes = size_t(2) << 20;
    static constexpr size_t kKept = 8;
    PinnedBuffer();
    ~PinnedBuffer();
    PinnedBuffer(const PinnedBuffer&) = delete;
    PinnedBuffer& operator=(const PinnedBuffer&) = delete;
    void* data() const { return p_; }

private:
    void* p_ = nullptr;
};

// Copies n records of `size` bytes to `out` through pinned buffers: pack(first, count, to) launches
// on `s` the kernel that writes records first .. first + count - 1 to pinned memory.
void read_records(size_t n, size_t size, void* out, hipStream_t s,
                  const std::function<void(size_t, size_t, void*)>& pack);

// f(begin, end) over consecutive pieces of [0, n), on up to eight threads; the exception of the first piece
// that throws one goes on to the caller
void for_ranges(size_t n, const std::function<void(size_t, size_t)>& f);

}  // namespace alien
