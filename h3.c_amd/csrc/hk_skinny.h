/* Offsets of the skinny GEMM's buffer loads (hk_gemm.hip), apart from the
 * kernel so that a CPU test can walk every load of a launch.
 *
 * A load reads at its lane offset plus its scalar offset, and the hardware
 * lets it through when the lane offset is below the buffer's bytes less the
 * scalar offset.  That difference must not be negative: as an unsigned number
 * it would let any lane offset through.  So the scalar offset never passes
 * the last k step, whatever step the pipeline asks for, and what makes a load
 * beyond the end return zeros is its lane offset alone. */
#ifndef HK_SKINNY_H
#define HK_SKINNY_H

#include <stdint.h>

/* k steps (of 64 bf16, 128 bytes a row) loaded ahead of the MFMAs, for W;
 * the ring they go round in */
enum { HK_SKINNY_RING = 4 };

/* The scalar offset of k step `step` of `k_steps`. */
constexpr uint32_t hk_skinny_k_bytes(uint32_t step, uint32_t k_steps) {
    return (step < k_steps ? step : k_steps - 1u) * 128u;
}

/* The lane offset of a load: `offset`, or past any operand (whose bytes end
 * 2 K + 4096 below 2^32) for a step past the end of its piece. */
constexpr uint32_t hk_skinny_lane(uint32_t offset, uint32_t step,
                                  uint32_t piece_steps) {
    return step < piece_steps ? offset : 0xfffff000u;
}

#endif
