// Replays the K-steps of bfaintb_prefill_wreg_kernel, every form, as its waves may run against one another: between two barriers any wave may be
// anywhere.  Checked of every barrier: what is read of LDS behind it has landed (every wave has waited for its part); what is copied to LDS behind it
// goes to no place that is read behind it, or whose reads from before may still be on their way; and of every group of matrix instructions, that
// it waits for its fragments.
#include "../../awesome_fusion_amd/csrc/bfaintb_prefill_wreg_step.hpp"

#include <cstdio>
#include <deque>
#include <vector>

using bfaintb::WregStep;

struct Item {
    char kind;      // 'a': a tile of A, 'c': codes or scales, 'p': packed codes, to registers
    uint32_t step;  // whose it is
    uint32_t unit;  // fragments: which
    uint32_t stage() const { return step % 3u; }
};

static int g_faults = 0, g_form_faults = 0;
#define CHECK(ok, ...) do { if (!(ok) && ++g_faults && ++g_form_faults <= 2) { printf(__VA_ARGS__); printf("\n"); } } while (0)

static void drain(std::deque<Item>& q, uint32_t left) { while (q.size() > left) q.pop_front(); }  // (either kind completes in order)

template <int BITS, bool GROUPED, bool PACKED, int MT>
static void replay()
{
    using S = WregStep<BITS, GROUPED, PACKED, MT>;
    char form[64];
    g_form_faults = 0;
    snprintf(form, sizeof(form), "%d bits, %s, %s, %d blocks", BITS, GROUPED ? "groups" : "columns", PACKED ? "packed" : "rows", MT);
    std::deque<Item> vm, lds;
    std::vector<Item> read, copied;  // since the last barrier (reads: and those that were in flight there)
    std::vector<Item> late;          // copies in flight at the last barrier
    auto barrier = [&](uint32_t at) {
        for (const Item& r : read)
            for (const Item& c : copied)
                CHECK(r.kind != c.kind || r.stage() != c.stage(), "%s: behind the barrier of step %d, '%c' of step %u is copied to where step %u's is read", form, (int)at - 1, c.kind, c.step, r.step);
        for (const Item& r : read)
            for (const Item& c : late)
                CHECK(r.kind != c.kind || r.step != c.step, "%s: behind the barrier of step %d, '%c' of step %u is read and may not have landed", form, (int)at - 1, r.kind, r.step);
        read.assign(lds.begin(), lds.end());
        late.assign(vm.begin(), vm.end());
        copied.clear();
    };
    auto read_lds = [&](char kind, uint32_t step, uint32_t unit) { lds.push_back({kind, step, unit}), read.push_back({kind, step, unit}); };
    // the prologue: A of step 1 on its way, what is before it landed; the fragments and quads that a step finds read
    for (uint32_t i = 0; i < S::kACopies; ++i) vm.push_back({'a', 1, 0});
    for (uint32_t un = 0; un < 8; ++un) read_lds('a', 0, un);
    for (uint32_t i = 0; i < S::quad_reads(0) + S::quad_reads(1); ++i) read_lds('c', 1, 0);
    for (uint32_t kt = 0; kt < 13; ++kt) {
        if (PACKED) drain(vm, S::behind_codes());
        for (const Item& v : vm) CHECK(v.kind != 'p' || v.step != kt + 1, "%s: step %u begins without the packed codes it converts", form, kt);
        uint32_t quads = 0, frags = 0, requests = 0;
        for (uint32_t slot = 0; slot < S::kSlots; ++slot) {
            if (slot % 16u == 0u) {
                drain(lds, S::in_flight(slot / 16u));
                for (const Item& r : lds) CHECK(r.kind != 'a' || r.step != kt || r.unit / 4u != slot / 16u, "%s: step %u, slot %u multiplies a fragment that is on its way", form, kt, slot);
            }
            if (slot == S::kBarrierSlot) {
                drain(vm, S::requests_before(slot));
                drain(lds, 0);
                barrier(kt + 1);
            }
            for (uint32_t un = 0; un < S::kUnits; ++un)
                if (S::frag_slot(un) == slot) read_lds('a', un < 8 ? kt + 1 : kt, un), ++frags;
            for (uint32_t quad = 0; quad < 8; ++quad) {
                if (S::quad_slot(quad) != slot) continue;
                for (uint32_t i = 0; i < S::quad_reads(quad); ++i) read_lds('c', quad < 2 ? kt + 2 : kt + 1, 0);
                ++quads;
            }
            const uint32_t r = S::requests_before(slot);
            CHECK(S::requests_before(slot + 1) - r <= 1, "%s: two requests in a slot", form);
            if (S::requests_before(slot + 1) == r) continue;
            const bool of_a = S::copies_before(r + 1) != S::copies_before(r), scales = GROUPED && r == S::copies_before(r);
            const Item it = of_a ? Item{'a', kt + 2, 0} : PACKED && !scales ? Item{'p', kt + 2, 0} : Item{'c', kt + 3, 0};
            vm.push_back(it), ++requests;
            if (it.kind != 'p') copied.push_back(it);
        }
        CHECK(quads == 8 && frags == S::kUnits && requests == S::kRequests, "%s: %u quads, %u fragments, %u requests a step", form, quads, frags, requests);
    }
}

template <int MT>
static void replay_height()
{
    replay<8, false, false, MT>(), replay<8, true, false, MT>(), replay<4, false, false, MT>(), replay<4, true, false, MT>();
    replay<8, false, true, MT>(), replay<8, true, true, MT>(), replay<4, false, true, MT>(), replay<4, true, true, MT>();
}

int main()
{
    replay_height<8>(), replay_height<10>(), replay_height<12>(), replay_height<14>(), replay_height<16>();
    if (g_faults == 0) printf("all steps in order\n");
    return g_faults != 0;
}
