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
    uint32_t pad_e4;                   // the depthwise input zero point ^ 0x80 in every byte
    int half_last;                     // the last chunk of expanded channels holds at most 16 real ones
    int has_res, fast_div;             // fast_div: the scales allow the unscaled division sequence
    float ry_rcp;                      // refined reciprocal of ry_scale
    float ra_scale, rb_scale, ry_scale;  // residual add: a = projection output, b = block input, y = sum
    int ra_zp, rb_zp, ry_zp;
    QAct act1, act2;                   // what only the tables are made from comes last: the kernels load their arguments in wide pieces
    int has_act1, has_act2;
};

// The activation part of a block's tables: QB_ACT_HEAD bytes of QBlockActHead, then the two activation tables, each at an address of
// its convolution's zero point's parity (quant_common.h).
constexpr int QB_ACT_HEAD = 4, QB_ACT_TABLE = 258, QB_ACT_BYTES = (QB_ACT_HEAD + 2 * QB_ACT_TABLE + 15) / 16 * 16;
struct QBlockActHead {
    uint8_t lo1, hi1, lo2, hi2;  // the entries between which each table changes
};
static_assert(sizeof(QBlockActHead) == QB_ACT_HEAD && QB_ACT_TABLE % 2 == 0 && QB_ACT_TABLE >= 257, "layout of the tables");
// The position tables, 16 bits an entry: what is more in LDS is a smaller tile, a workgroup less on a CU or a block that does not fit (with
// 8 bytes an entry 96 -> 576 -> 96 channels did not, 64 -> 192 -> 64 on 1024 maps of 20x20 took 171 us instead of 141).  Of a patch
// position (Ppad entries): its row among those of the tile's images, QB_POS_PAD set for a halo column, past the patch and, in tiles of
// whole images, for the rows above and below an image.  Of an output position (Q rounded up to 32): its top-left tap's patch position.
typedef uint16_t QBlockPos;
constexpr int QB_POS_PAD = 0x8000;

#ifdef __HIPCC__
// `head`: the four bytes of QBlockActHead, in a scalar register
__device__ __forceinline__ unsigned qb_act_head(const char *act) { return __builtin_amdgcn_readfirstlane(*reinterpret_cast<const unsigned *>(act)); }
__device__ __forceinline__ RequantLut qb_lut(const char *act, unsigned head, int table, int zp) {
    const int base = int(lds_address(act)) + QB_ACT_HEAD + table * QB_ACT_TABLE + (zp & 1);
    const int lo = (head >> (16 * table)) & 255, hi = (head >> (16 * table + 8)) & 255;
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

// LDS bytes that a block takes of a chain on one image a workgroup: input patch of `positions`, `weights` and tables, expanded patch,
// projection sums of `outputs`.
static inline size_t zant_qblock_image_bytes(int Cin32, int Ce32, int co32, int64_t positions, int64_t outputs, int64_t weights) {
    const size_t Ppad = size_t(positions + 31) & ~size_t(31), Qpad = size_t(outputs + 31) & ~size_t(31);
    return size_t(Cin32 + Ce32) * 2 * Ppad * 16 + size_t(weights) + QB_ACT_BYTES + (Ppad + Qpad) * sizeof(QBlockPos) + Qpad / 32 * co32 * 4096;
}

// zant_qblock_chain on one image a workgroup, activations in LDS from block to block (qblock_image_i8.hip); 1 when the blocks do not
// fit that or there are too many images.
int zant_qblock_image_chain(zant_ctx *ctx, int n, const zant_qblock_call *calls, bool query_only);
