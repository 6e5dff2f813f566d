// How a traversal launch deals its rays to its waves (host and device; no HIP
// header, so the rule can be checked on its own).
#pragma once
#include <stdint.h>

namespace kp {

// Rays of a chunk taken from the work counter, and of one near a queue's end.
constexpr uint32_t kChunk = 256;
constexpr uint32_t kTailChunk = 64;

// Occlusion launches of at most this many rays per block split their rays
// (k_occluded5<true>).
constexpr uint32_t kSplitRays = 512;

// Thin launches: up to kThinMost rays per SIMD are spread over one wave a SIMD
// (up to kThinOne) or two, the idle lanes taking parts of them.
template <bool kAny>
constexpr uint32_t kThinOne = kAny ? 32u : 8u;
template <bool kAny>
constexpr uint32_t kThinMost = kAny ? 64u : 128u;

// Whether the first chunks of n rays over `waves` waves hold every ray, so
// that the work counter is not used.
constexpr bool first_chunks_hold_all(uint64_t n, uint32_t waves) { return n <= (uint64_t)waves * kChunk; }

// Rays of a wave's first chunk: wave w of a launch (or of a part of one with a
// queue of its own) starts with rays [w F, (w + 1) F) of the queue's n.
//
// Up to kChunk rays per wave: every ray in a first chunk; more: the first
// chunks hold about half the rays (256 .. 4096 per wave) and the counter's
// chunks balance the rest.  First chunks are multiples of 64 rays (as many
// waves as that takes), except that a small launch whose rays can be split
// (thin_most > 0) uses one or two waves per SIMD with fewer rays each: the
// idle lanes then take parts of the rays from the start.  A grid's blocks are
// placed one a CU before a CU gets a second, so its first `simds` waves have a
// SIMD each, however many waves a SIMD the grid holds in all (five, four where
// the kernel needs more registers, fewer where a batch is tuned so); a grid of
// fewer waves has one SIMD per wave.  1,000 closest-hit rays take 15.2 us with
// at least four rays a wave and 13.7 so, 2,000 occlusion rays 36 us with 64 a
// wave and 27 so (20.5 with the hand-out of single children).  One wave per
// SIMD or two: 16,384 closest-hit rays 37.6 us (14.5 each where three
// launches are in flight) and 33.4 (14.2), 65,536 74.7 (28.3) and 61.1
// (26.5), 100,000 84 (64 a wave, 33.6) and 77 (33.0); occlusion 16,384
// 26.1 (10.6) and 24.7 (11.9), 65,536 43.4 (17.5) and 37.2 (17.0),
// 100,000 48 (64 a wave, 20.3) and 45.4 (20.8).  All five a SIMD take
// 65,536 closest-hit rays 54 us, but 36 with three launches in flight.
// Multiples of 64 leave some waves without rays, which costs the launch
// and helps others in flight (800,000 rays 278 and 184 us; evenly dealt
// 248 and 191).  The first launch of a pass (even), whose camera rays
// take about the same time each, deals them evenly: a batch of eight
// scenes 931 -> 893 us; later bounces gain nothing by it.
constexpr uint32_t first_chunk(uint32_t n, uint32_t waves, uint32_t simds, uint32_t thin_one, uint32_t thin_most,
                               bool even) {
    const uint32_t one = waves < simds ? waves : simds;
    if (n <= one * thin_most) {
        const uint32_t two = waves < 2u * one ? waves : 2u * one;
        const uint32_t used = n <= one * thin_one ? one : two;
        return (n + used - 1u) / used;
    }
    if (first_chunks_hold_all(n, waves)) {
        const uint32_t f = (n + waves - 1u) / waves;
        return even ? (f < 64u ? 64u : f) : (f + 63u) & ~63u;
    }
    const uint32_t f = (n / (2u * waves)) & ~63u;
    return f < kChunk ? kChunk : (f > 4096u ? 4096u : f);
}

}  // namespace kp
