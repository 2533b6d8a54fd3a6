// patch_deal.h over all patches of up to 32 channel blocks and 1300 positions: every unit is dealt once, and a patch that four rounds of 256
// threads hold takes no more.  Prints "ok" when all do.
#include <cmath>
#include <cstdio>
#include <vector>

#include "../z-ant_amd/csrc/patch_deal.h"

int main() {
    for (int blocks = 1; blocks <= 32; ++blocks)
        for (int positions = 9; positions <= 1300; positions += blocks > 8 ? 7 : 1) {
            const bool flat = patch_flat(blocks, positions);
            const int rounds = patch_rounds(blocks, positions, flat), per_block = (positions + 255) / 256, fewest = (blocks * positions + 255) / 256;
            if (fewest <= PATCH_ROUNDS_AHEAD ? rounds > PATCH_ROUNDS_AHEAD : rounds > blocks * per_block) {
                std::printf("%d blocks of %d: %d rounds\n", blocks, positions, rounds);
                return 1;
            }
            std::vector<int> dealt(size_t(blocks) * positions, 0);
            for (int ulp = -2; ulp <= 2; ++ulp) {  // (a reciprocal instruction may be off by one)
                float inv = 1.0f / float(positions);
                for (int i = 0; i < std::abs(ulp); ++i) inv = std::nextafter(inv, ulp < 0 ? 0.0f : 2.0f);
                for (int r = 0; r < rounds; ++r)
                    for (int tid = 0; tid < 256; ++tid) {
                        int block = r / per_block, p = (r % per_block) * 256 + tid;
                        if (flat) p = patch_unit_flat(r, tid, positions, inv, &block);
                        if (p < 0 || block < 0) { std::printf("%d blocks of %d: round %d thread %d\n", blocks, positions, r, tid); return 1; }
                        if (block < blocks && p < positions) ++dealt[size_t(block) * positions + p];
                    }
            }
            for (int n : dealt)
                if (n != 5) { std::printf("%d blocks of %d: a unit %d times\n", blocks, positions, n); return 1; }
        }
    std::puts("ok");
    return 0;
}
