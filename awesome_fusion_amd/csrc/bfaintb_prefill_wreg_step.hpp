// Where in a K-step of bfaintb_prefill_wreg_kernel everything beside the matrix instructions stands: plain constants, which the kernel is written by and
// which a host program can replay.
#pragma once
#include <stdint.h>

namespace bfaintb {

// A step is 8 MT slots of one matrix instruction.  In a slot, in this order: the barrier, a fragment of A, a quad's codes and scale, a request for memory.
// The stages of LDS go round by threes; Now is the one this step multiplies from, Next and After the two behind it.  The step
//   reads     fragments of A: Now's, from the ninth on, and behind the barrier Next's first eight;
//             quads (a column block's codes and group scale): Next's from the third on, and behind the barrier After's first two;
//   requests  A of step kt + 2, into After; codes (rows) and group scales of step kt + 3, into Now; packed codes of step kt + 2, into registers.
// So what one step reads ahead of its barrier, A of Now and codes of Next, is where the requests behind that barrier go: they have to be there, every
// wave's of them, when the barrier opens.
template <int BITS, bool GROUPED, bool PACKED, int MT>
struct WregStep {
    static constexpr uint32_t kUnits = 2u * MT, kSlots = 8u * MT, kBarrierSlot = kSlots - 24u;

    // Requests: codes and group scales in their order, the copies of A spread among them; packed codes, which the next step waits for at its
    // start, ahead of them (us, among the copies / ahead: 577 x 13824 x 5120 4-bit g128 95.7 / 86.2, 8-bit 89.5 / 80.6; 300 x 28672 x 4096 79.9 / 72.0).
    static constexpr uint32_t kACopies = MT / 2u, kCodeCopies = PACKED ? 0u : BITS / 2u;
    static constexpr uint32_t kCodes = (GROUPED ? 1u : 0u) + (PACKED ? 4u : kCodeCopies), kRequests = kCodes + kACopies;
    static constexpr uint32_t copies_before(uint32_t r) { return !PACKED ? r * kACopies / kRequests : r < kCodes ? 0u : r - kCodes; }
    static constexpr uint32_t request_slot(uint32_t r) { return 2u + r * (kSlots - 2u) / kRequests; }
    static constexpr uint32_t requests_before(uint32_t slot)
    {
        uint32_t r = 0;
        while (r < kRequests && request_slot(r) < slot) ++r;
        return r;
    }
    static constexpr uint32_t behind_codes()  // requests of a step behind its last one for codes or scales
    {
        uint32_t r = 0;
        while (r - copies_before(r) < kCodes) ++r;
        return kRequests - r;
    }

    // LDS reads: of unit un's fragment (un < 8: the next step's), of a quad (quad < 2: the step's after).  A quad is read a quarter of a step before
    // it is prepared; the last one six slots before the barrier, which waits for it: with 8 blocks a quarter of a step would be too late.
    static constexpr uint32_t kLastQuadSlot = kBarrierSlot - 6u;
    static constexpr uint32_t frag_slot(uint32_t un) { return un >= 8u ? 4u * (un - 8u) : kBarrierSlot + 3u * un; }
    static constexpr uint32_t quad_slot(uint32_t quad)
    {
        if (quad >= 2u) return (quad - 2u) * MT < kLastQuadSlot ? (quad - 2u) * MT : kLastQuadSlot;
        return (quad + 6u) * MT > kBarrierSlot ? (quad + 6u) * MT : kBarrierSlot + 1u;
    }
    static constexpr uint32_t quad_reads(uint32_t quad)
    {
        return (PACKED || (BITS == 4 && (quad & 1u) != 0u) ? 0u : 1u) + (GROUPED ? 1u : 0u);
    }
    static constexpr uint32_t reads_at(uint32_t slot)
    {
        uint32_t n = 0;
        for (uint32_t un = 0; un < kUnits; ++un) n += frag_slot(un) == slot ? 1u : 0u;
        for (uint32_t quad = 0; quad < 8u; ++quad) n += quad_slot(quad) == slot ? quad_reads(quad) : 0u;
        return n;
    }
    // LDS reads that may be in flight: behind the last fragment of group g and before the group begins
    static constexpr uint32_t in_flight(uint32_t g)
    {
        uint32_t n = 0;
        const uint32_t last = frag_slot(4u * g + 3u);
        for (uint32_t slot = last + 1u; slot < 16u * g + (g < 2u ? kSlots : 0u); ++slot) n += reads_at(slot % kSlots);
        return n;
    }
};

}  // namespace bfaintb
