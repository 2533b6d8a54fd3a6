// Matrix-core f32 convolution on split operands (conv_split_f32.hip): what the dispatch in conv_f32.hip needs of it.
#pragma once
#include "common.h"

// max without the NaN-quieting pass the compiler puts in front of fmaxf (an MFMA result is never a signalling NaN); a NaN
// operand yields the other one, like fmaxf
__device__ __forceinline__ float vmax(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float vmax3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// A convolution seen as one flat sequence of output slots (output positions, or 2x2 pooling windows with a fused pool) over
// "strips": a strip is a run of whole output columns of one image (the whole image unless it is too wide for LDS).  The
// input rows of a strip with their padding follow one another strip after strip, so the rows a run of slots needs are one
// run of padded rows, wherever it starts and however many images it touches.
struct FlatGeom {
    int PW, PHI;            // patch columns; padded input rows of one strip
    int P1s;                // patch positions allocated (a multiple of 4)
    int rs, cs;             // padded input rows / columns from one slot to the next
    int SR, SC;             // slots of a strip: rows, columns
    int slot_cols;          // slot columns of a whole image (strips x SC may exceed it)
    int n_strips;           // strips per image
    int n_slots;            // slots in all
    int S;                  // slots per tile
    int n_chunks, n_kblocks, n_tiles;
    int x_c4;               // the input is stored [N][C/4][H][W][4]
    FastDiv d_im, d_sc, d_pw, d_phi, d_strips, d_kw;
};

struct SplitPlan {
    int MT, WM, WN;         // 32-slot tiles of a wave (x 32 channels); waves over slots and over channels
    int pair;               // steps of 8 channels, two taps per matrix instruction
    int nsub;               // groups of 16 channels per step
    FlatGeom f;
    size_t lds_bytes;
    size_t wp_bytes;        // packed weights
};

// Whether the kernel takes this convolution (with the fused 2x2/2 max pool or without), and the tiling it would run with.  `slot`
// keeps the tiling for the next call with the same geometry.
bool zant_conv_split_plan(const ConvGeom &g, bool pool, int num_cus, SplitPlan *plan, zant_pack_slot *slot = nullptr);
// What a layer counts against ZANT_HIP_STATIC_SCRATCH_BYTES.  The limit is stated in f32 weights; the static array itself has
// room for their three terms and padding.
size_t zant_conv_split_fixed_bytes(const ConvGeom &g);
// Packs the weights (unless `slot` holds them) and launches.
int zant_conv_split_run(zant_ctx *ctx, const float *x, const float *w, const float *bias, float *y, const ConvGeom &g,
                        const SplitPlan &plan, int relu, bool pool, zant_pack_slot *slot, int x_c4);

// Convolutions of short sums (conv_short_f32.hip): whether the kernel can take this one, whether it is then the better one of the two
// (packed_once: the split kernel's weights are packed once for many calls), and its launch (no scratch).
bool zant_conv_short_ok(const ConvGeom &g);
bool zant_conv_short_better(const ConvGeom &g, bool packed_once);
int zant_conv_short_run(zant_ctx *ctx, const float *x, const float *w, const float *bias, float *y, const ConvGeom &g, int relu);
