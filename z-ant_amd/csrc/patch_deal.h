// How the units of a block's input patch -- `positions` of each of `blocks` blocks of 16 channels -- are dealt to the 256 threads that copy
// it; usable from host code (no HIP headers needed) and, under hipcc, from kernels.
#pragma once

#if defined(__HIPCC__)
#define ZANT_DEAL_FN __host__ __device__ __forceinline__
#else
#define ZANT_DEAL_FN inline
#endif

// Rounds of units that a thread holds while another stage runs: more are not fetched ahead.
constexpr int PATCH_ROUNDS_AHEAD = 4;

// A round is 256 positions of one channel block, whose index is then the same for all threads; or, `flat`, 256 units of all blocks in a
// row, which takes a division a unit but leaves no threads idle.
ZANT_DEAL_FN int patch_rounds(int blocks, int positions, bool flat) {
    return flat ? (blocks * positions + 255) >> 8 : blocks * ((positions + 255) >> 8);
}
// Flat where rounds by block are too many to be fetched ahead and those in a row fewer: 72 -> 432 -> 72 on 512 maps of 28x28 1040 -> 1004
// us, 72 -> 72 -> 112 on 32 of 9x9 with stride 2 12.5 -> 11.7.  Kernels of their own: the code for both costs narrow blocks 0.3 us a launch
// and MobileNetV2-0.35 2 %.
ZANT_DEAL_FN bool patch_flat(int blocks, int positions) {
    const int by_block = patch_rounds(blocks, positions, false);
    return by_block > PATCH_ROUNDS_AHEAD && patch_rounds(blocks, positions, true) < by_block;
}

// p / d for 0 <= p < 2^20 with inv = 1.0f / d to within a few units in the last place: (p + 1/2) / d is at least 1 / 2d away from a whole
// number, further than reciprocal and fma err.
ZANT_DEAL_FN int quick_div(int p, float inv) { return int(__builtin_fmaf(float(p), inv, 0.5f * inv)); }

// Thread `tid`'s position and block in a round of a flat deal; a block past the last one: none.
ZANT_DEAL_FN int patch_unit_flat(int round, int tid, int positions, float inv_positions, int *block) {
    const int u = round * 256 + tid;
    *block = quick_div(u, inv_positions);
    return u - *block * positions;
}
