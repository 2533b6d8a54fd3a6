// What the inverted residual block kernels share: a block's kernel arguments and their preparation (qblock_i8.hip).
#pragma once
#include "quant_common.h"
#include "quant_layout.h"

struct QBlockArgs {
    int N, H, W, OH, OW, stride;
    int CBin, Cin32, Ce32, CBe, CBo;   // input channel blocks (16) / chunks (32); expanded chunks / blocks; output blocks
    int Co;                            // output channels (the rest of the last block is padding)
    int NB, TH, PH, PW, P, Ppad, Q;    // tile: images, output rows, patch rows / columns / positions, output positions
    int n_row_tiles, n_tiles;
    int o_xl, o_e, o_w1, o_w2, o_wdw, o_tab, o_act, o_ptab, o_qtab;  // LDS byte offsets
    int packed_units;                  // 16-byte units of weights and tables: the LDS bytes from o_w1 to the end of the position tables
    int split;                         // stage D deals (position tile, channel chunk) units to the waves (few position tiles)
    int zp1, zp2;                      // zero points of the three convolutions' own outputs
    float zp3f;
    QAct act1, act2;
    int has_act1, has_act2;
    uint32_t pad_e4;                   // the depthwise input zero point ^ 0x80 in every byte
    int half_last;                     // the last chunk of expanded channels holds at most 16 real ones
    int has_res, fast_div;             // fast_div: the scales allow the unscaled division sequence
    float ry_rcp;                      // refined reciprocal of ry_scale
    float ra_scale, rb_scale, ry_scale;  // residual add: a = projection output, b = block input, y = sum
    int ra_zp, rb_zp, ry_zp;
};

// The activation part of a block's tables: QB_ACT_HEAD bytes of QBlockActHead, then the two activation tables, each at an address of
// its convolution's zero point's parity (quant_common.h).
constexpr int QB_ACT_HEAD = 32, QB_ACT_TABLE = 272, QB_ACT_BYTES = QB_ACT_HEAD + 2 * QB_ACT_TABLE;
struct QBlockActHead {
    int lo1, hi1, lo2, hi2;  // the entries between which each table changes
    int unused[4];
};
// The position tables.  Of a patch position (Ppad entries): x the patch row, bit 31 set for a halo column or past the patch; y the byte
// offset of its first unit from that of the tile's first image, patch row 0, column 0.  Of an output position (Q rounded up to 32): x
// the byte offset of its top-left tap in the patch, y that of its first output unit from the tile's first one.
typedef int2 QBlockPos;
static_assert(sizeof(QBlockActHead) == QB_ACT_HEAD && QB_ACT_BYTES % 16 == 0 && QB_ACT_TABLE >= 257, "layout of the tables");

#ifdef __HIPCC__
__device__ __forceinline__ RequantLut qb_lut(const char *act, int table, int lo, int hi, int zp) {
    const int base = int(lds_address(act)) + QB_ACT_HEAD + table * QB_ACT_TABLE + (zp & 1);
    RequantLut t;
    t.t0 = zq_as_float(unsigned(base + zp));
    t.lo = zq_as_float(unsigned(base + lo));
    t.hi = zq_as_float(unsigned(base + hi));
    return t;
}
#endif

// What a launch needs of one block: its kernel arguments, LDS bytes, instantiation and packed weights.
struct QBlockPrep {
    QBlockArgs a;
    size_t lds_bytes;
    int CO32, MQv;
    const uint4 *packed;  // weights, requantisation, activation and position tables
};

// Plans a block's tile, (re)packs its weights and tables into `slot` (or the context workspace) and fills the kernel
// arguments.  force_nb > 0: tiles of exactly that many whole images, or 1.  plan_only: no packing, no pointers needed.
int zant_qblock_prepare(zant_ctx *ctx, const int64_t xdim[4], const zant_qconv_desc *expand, const zant_qconv_desc *dw, int64_t dw_stride,
                        const zant_qconv_desc *project, int residual, float add_scale, int add_zp, const int64_t ydim[4], bool plan_only,
                        zant_pack_slot *slot, int force_nb, QBlockPrep *out);

// zant_qblock_chain on one image a workgroup, activations in LDS from block to block (qblock_image_i8.hip); 1 when the blocks do not
// fit that or there are too many images.
int zant_qblock_image_chain(zant_ctx *ctx, int n, const zant_qblock_call *calls, bool query_only);
