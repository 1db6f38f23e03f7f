// Rows of the tiles' pair-state table as the contact phase finds them, on the
// host: a row holds its live entries, then a claimed slot whose tag is not
// written yet, behind it what earlier rows left. Prints each lookup that is
// wrong; the exit status is their number.
#include <cstdio>
#include <vector>

#include "../../libgran_amd/csrc/pair_row.h"

using namespace hg;

static int wrong = 0;

static void expect(const char *what, const std::vector<uint32_t> &tags, uint32_t count, uint32_t j, uint32_t slot) {
    const uint32_t got = row_slot(count, j, [&](uint32_t s) { return tags[s]; });
    if (got == slot) return;
    std::printf("%s: partner %u of %u entries in slot %u, not %u\n", what, j, count, got, slot);
    wrong++;
}

int main() {
    for (uint32_t bond : {0u, kBondBit}) {
        // [5, 9] lost 5: [9 | 9]. Another thread claims slot 1 for a new partner
        // and has not written its tag.
        const std::vector<uint32_t> left{9u | bond, 9u | bond};
        expect("before the claim", left, 1, 9, 0);
        expect("claimed slot holds the old tag", left, 2, 9, 0);
        // [2, 5, 7, 9] lost 2 and 5: [7, 9 | 7, 9], two slots claimed, the
        // second one written first
        const std::vector<uint32_t> two{7u | bond, 9u | bond, 7u, 3u};
        expect("two claimed", two, 4, 7, 0);
        expect("two claimed", two, 4, 9, 1);
        expect("two claimed", two, 4, 3, 3);
    }
    const std::vector<uint32_t> row{1, kNoEntry, 4u | kBondBit, 6};
    expect("an ended entry between", row, 4, 4, 2);
    expect("not in the row", row, 4, 5, kNoRowSlot);
    expect("beyond the row", row, 3, 6, kNoRowSlot);
    expect("an empty row", row, 0, 1, kNoRowSlot);
    // a slot comes back from the queue as it went in, however long the row
    for (uint32_t place : {0u, 1u, kTilePlaces - 1u})
        for (uint32_t slot : {0u, 1u, 4094u, 4095u, 4096u, 70000u, kNoRowSlot - 1u, kNoRowSlot}) {
            const uint32_t word = queue_word(place, slot);
            if (queue_place(word) == place && queue_slot(word) == slot) continue;
            std::printf("place %u, slot %u came back as %u, %u\n", place, slot, queue_place(word), queue_slot(word));
            wrong++;
        }
    if (kNoRowSlot <= 4095u) wrong++;
    return wrong;
}
