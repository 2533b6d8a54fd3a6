// Which blocks and chains of inverted residual blocks are taken (host code only): what LDS has room for, but no block of half-empty matrix
// tiles that the three layers by themselves outrun.  Prints "ok" when all are as expected.
#include <cstdio>
#include <cstring>

#include "quant_layout.h"

struct Block { int cin, ce, co, stride; bool residual; };

int main() {
    zant_ctx ctx;
    ctx.num_cus = 256;
    struct { int64_t images, h; int n; Block b[3]; bool refused; } cases[] = {
        // one block of weights that leave room for a row or two: up to a tile a CU
        {1, 3, 1, {{96, 576, 96, 1, true}}}, {8, 8, 1, {{96, 576, 96, 1, true}}}, {32, 6, 1, {{96, 576, 96, 1, true}}},
        {512, 8, 1, {{96, 576, 96, 1, true}}, true}, {512, 3, 1, {{96, 576, 96, 1, true}}, true}, {1024, 7, 1, {{112, 448, 112, 1, true}}, true},
        // one image a workgroup
        {100, 16, 2, {{48, 192, 72, 2, false}, {72, 288, 72, 1, true}}},
        {256, 16, 3, {{64, 192, 96, 2, false}, {96, 288, 96, 1, true}, {96, 288, 96, 1, true}}},
        {256, 12, 3, {{56, 224, 56, 1, true}, {56, 224, 56, 1, true}, {56, 224, 56, 1, true}}},
        {256, 8, 2, {{64, 128, 128, 1, false}, {128, 256, 128, 1, true}}},
        {100, 20, 3, {{40, 120, 64, 2, false}, {64, 192, 64, 1, true}, {64, 192, 64, 1, true}}},
    };
    for (const auto &k : cases) {
        zant_qconv_desc d[3][3];
        zant_qblock_call calls[3];
        int64_t dim[4][4];
        std::memset(d, 0, sizeof(d));
        dim[0][0] = k.images; dim[0][1] = k.b[0].cin; dim[0][2] = dim[0][3] = k.h;
        for (int b = 0; b < k.n; ++b) {
            const Block &s = k.b[b];
            const int io[3][2] = {{s.cin, s.ce}, {s.ce, s.ce}, {s.ce, s.co}};
            for (int i = 0; i < 3; ++i) {
                d[b][i].C = io[i][0]; d[b][i].K = io[i][1]; d[b][i].n_wscale = 1;
                d[b][i].x_scale = d[b][i].y_scale = d[b][i].act_scale = 1.0f;
            }
            dim[b + 1][0] = k.images; dim[b + 1][1] = s.co;
            dim[b + 1][2] = dim[b + 1][3] = (dim[b][2] - 1) / s.stride + 1;
            calls[b] = {nullptr, dim[b], &d[b][0], &d[b][1], s.stride, &d[b][2], s.residual, 1.0f, 0, nullptr, dim[b + 1], nullptr};
        }
        const Block &s = k.b[0];
        const int rc = k.n > 1 ? zant_qblock_chain(&ctx, ZantChain::images, k.n, calls, true)
                               : zant_qblock_blocked(&ctx, nullptr, dim[0], &d[0][0], &d[0][1], s.stride, &d[0][2], s.residual, 1.0f, 0, nullptr,
                                                     dim[1], true, nullptr);
        if (rc != (k.refused ? 1 : ZANT_OK)) {
            std::printf("%ld images of %ldx%ld, %d -> %d -> %d: %d\n", long(k.images), long(k.h), long(k.h), s.cin, s.ce, s.co, rc);
            return 1;
        }
    }
    std::puts("ok");
    return 0;
}
