// How launches divide their work: plain arithmetic shared by the kernels,
// the launch code and the CPU tests (which compile this header with the host
// compiler), so it includes nothing of HIP.
#pragma once

#include <stdint.h>

namespace spg {

// Waves that walk n rays (before the cap by occupancy): one per 64 rays, and
// below 256 * 64 rays up to 256 waves with fewer rays each, one wave per CU
// (a wave's time is that of its longest chain of steps, and lanes that wait
// for other kinds of steps lengthen it).  96 or 128 rays per wave: the
// 256x256 frame's walk takes 228 and 240 us instead of 200; 48 rays and at
// least 512 waves: 214; 80 rays: 230.
__host__ __device__ inline uint32_t walk_waves(uint32_t n)
{
    const uint32_t full = n / 64u + (n % 64u != 0u ? 1u : 0u);
    const uint32_t few = n < 256u ? n : 256u;
    return full > few ? full : few ? few : 1u;
}

// The chunks of a list of n rays for `waves` waves: chunk j holds rays
// [begin(j), end(j)).  An even share of the list, at most maxChunk rays.  No
// sum here passes n, so none wraps for any 32-bit n.
struct WorkChunks
{
    uint32_t n, chunk, chunks;
    __host__ __device__ inline WorkChunks(uint32_t rays, uint32_t waves, uint32_t maxChunk)
        : n(rays)
    {
        const uint32_t last = n ? n - 1u : 0u, share = last / waves + 1u;
        chunk = share < maxChunk ? share : maxChunk;
        chunks = n ? last / chunk + 1u : 0u;
    }
    __host__ __device__ inline uint32_t begin(uint32_t j) const { return j * chunk; }
    __host__ __device__ inline uint32_t end(uint32_t j) const
    {
        const uint32_t lo = j * chunk, left = n - lo;
        return lo + (chunk < left ? chunk : left);
    }
};

// A wave refills its idle lanes once kRefill of them wait (or all do): each
// refill stalls the wave on the new rays' loads and setup, so refilling one
// lane per iteration adds a memory round trip to nearly every step, while
// waiting for all 64 leaves the wave running its longest ray alone.  Scene
// walk: 40 instead of 32 costs 2-3% (box 1820 against 1771 us, room 4532
// against 4386); mesh walk: 48 instead of 32 costs 2% (527 against 516 us).
constexpr uint32_t kSceneRefill = 32, kMeshRefill = 32;
// The top kShort entries of each lane's stack live in LDS (kShort * 256
// bytes per wave), deeper ones spill to global memory: 40 for the scene walk
// costs the room 4% (4539 us against 4359), 80 for the mesh walk gains
// nothing over 32.
constexpr int kSceneShortStack = 16, kMeshShortStack = 32;
// The spill area's first entry: what no walk keeps in LDS (2.1 MB per entry on
// 256 CUs).
constexpr int kMinShortStack =
    kSceneShortStack < kMeshShortStack ? kSceneShortStack : kMeshShortStack;

// Refill thresholds of the scene walk that a batch's tuner times against the
// default (24 grid scenes at 2^22 paths in flight: 5.06 ms per sample with
// 32, 4.92 with 40, 5.05 with 48; eight grid scenes of 64 to 512 pixels a
// side at 2^20: 1.13, 1.14, 1.16).
constexpr uint32_t kRefillSweep[] = {40, 48};
// A candidate of the tuner replaces the best so far only where its time is
// shorter by more than 2%: timings of one shape differ by 1-4% from run to
// run.
inline bool tuned_better(float ms, float best) { return ms < 0.98f * best; }

// Where record i of a list of `words` words each begins (i * words passes 2^32
// from 715,827,883 rays of 6 words on).
__host__ __device__ inline uint64_t record_at(uint32_t i, uint32_t words)
{
    return (uint64_t)i * words;
}

// A grid-stride loop's next index, n at its end: `i + step` would wrap where n
// is within a step of 2^32, and the thread would start over for ever.
__host__ __device__ inline uint32_t stride_next(uint32_t i, uint32_t step, uint32_t n)
{
    return n - i > step ? i + step : n;
}

// Blocks of `block` threads for n items, at most `most`.
__host__ __device__ inline uint32_t stride_blocks(uint32_t n, uint32_t block, uint32_t most)
{
    const uint32_t need = n / block + (n % block != 0u ? 1u : 0u);
    return need < most ? need : most;
}

}  // namespace spg
