// f32 convolution of short sums (few input channels, or 1x1 filters over few) on the f32 matrix cores.
//
//   D[k, p] = sum_{c,kh,kw} W[k, c, kh, kw] * X[n(p), c, ih(p,kh), iw(p,kw)]      (reference op_convolution.zig:42-331)
//
// With few terms a sum the output dominates: a 32 x 32 block is 4 KB of stores, some 1500 cycles of a SIMD's share of the HBM
// bandwidth, and v_mfma_f32_32x32x2_f32 adds two terms to it in 64.  So there is nothing to stage, split or pack: a wave gathers
// its 32 positions' terms straight from the vector cache, two consecutive terms c*T + t for each position (lanes 0-31 the
// first, lanes 32-63 the second), and multiplies them with the weights of up to 96 output channels, which the workgroup has
// copied to LDS as they are.  Padding is a range-checked load that returns zero.  One launch, no scratch, f32 arithmetic throughout.
// Kernel times against the kernels that ran these layers before (one thread an output, or one a position, or the split kernel and its
// packing): 387x3x57x92 to 109 5x5 filters 7270 -> 500 us, 64x2x56x56 to 64 3x3 filters 131 -> 18, 64x16x56x56 to 64 1x1 filters
// 223 -> 16, 64x1x56x56 to 128 3x3 filters 32 -> 21, 64x64x56x56 to 64 1x1 filters 52 -> 32.  What bounds it: stores, whose 128-byte runs
// reach 3 to 5 TB/s, and from some 64 terms on the matrix pipes.  Plain stores, not streaming ones: what the next operator reads stays in
// the last-level cache (a 2x2 pool behind 3055x1x28x28 to 32 filters 85 us less), and consecutive tiles, whose runs share cache lines,
// go to one XCD (186624 positions, 128 filters 34 -> 28 us on cold buffers).  One case is no faster, and 2 to 8 us slower of 90: 3055x1x28x28 to
// 32 3x3 filters, where both kernels wait for 265 MB of stores.
#include <algorithm>

#include "conv_split_f32.h"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

struct ShortGeom {
    int terms, steps;            // terms of a sum; pairs of them
    int n_pos, n_tiles;          // output positions of the batch; tiles of 32
    FastDiv d_terms, d_taps, d_kw, d_plane, d_ow;
};

constexpr int kGroup = 8;        // pairs of terms a lane loads at a time

constexpr size_t short_lds_bytes(int kb, int steps) {
    return size_t(2 * steps) * (kb * 32 + 1) * 4 + size_t(kb) * 32 * 4 + size_t((steps + kGroup - 1) / kGroup * kGroup * 2) * 8;
}

// Workgroups of four waves, KB blocks of 32 output channels; a wave walks tiles of 32 positions.
// LDS: [term][KB * 32 channels, one word of padding] weights (the padding keeps the transposing copy off one bank), bias, and per
// term where it lies relative to a position's first: byte offset, filter row and column.
template <int KB, bool HALVES>
__global__ void __launch_bounds__(256, KB > 2 ? 2 : 4)
conv_f32_short_kernel(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias, float *__restrict__ y,
                      ConvGeom g, ShortGeom s, int relu) {
    constexpr int COLS = KB * 32, PITCH = COLS + 1;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    uint2 *tab = reinterpret_cast<uint2 *>(lds);
    const int tab_n = (s.steps + kGroup - 1) / kGroup * kGroup * 2;
    float *bias_l = reinterpret_cast<float *>(tab + tab_n);
    float *wl = bias_l + COLS;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, lh = lane >> 5;
    const int k0 = blockIdx.y * COLS, kn = min(g.K - k0, COLS);
    const int plane = g.H * g.W, oplane = g.OH * g.OW;

    for (int e = tid; e < tab_n; e += 256) {
        const int c = int(fastdiv(unsigned(e), s.d_taps)), t = e - c * g.KH * g.KW;
        const int kh = int(fastdiv(unsigned(t), s.d_kw)), kw = t - kh * g.KW;
        uint2 v;
        v.x = unsigned(c * plane + kh * g.dh * g.W + kw * g.dw) * 4u;
        v.y = unsigned(kh * g.dh) << 16 | unsigned(kw * g.dw);
        if (e >= s.terms) v = uint2{0u, 0x7fff0000u};  // a row below every image (H + pad < 2^15): loads as zero
        tab[e] = v;
    }
    for (int i = tid; i < COLS; i += 256) bias_l[i] = bias != nullptr && i < kn ? bias[k0 + i] : 0.0f;
    const float *wk = w + int64_t(k0) * s.terms;
    for (int i = tid; i < COLS * s.terms; i += 256) {
        const int col = int(fastdiv(unsigned(i), s.d_terms));
        wl[(i - col * s.terms) * PITCH + col] = col < kn ? wk[i] : 0.0f;
    }
    if (s.terms & 1)
        for (int i = tid; i < COLS; i += 256) wl[s.terms * PITCH + i] = 0.0f;
    __syncthreads();

    const float *wa = wl + lh * PITCH + l32;
    const uint2 *tp = tab + lh;
    const int64_t img = int64_t(g.C) * plane;
    const int chunks = (s.n_tiles + 3) >> 2;
    auto tile_of = [&](int i) {  // neighbouring tiles on one XCD
        const int xcd = i & 7, q = chunks >> 3, rem = chunks & 7;
        return (xcd * q + min(xcd, rem) + (i >> 3)) * 4 + wave;
    };
    // where a lane's position lies: its filter's first row and column, their byte in the input and the output's byte, both from the
    // tile's first image
    int n0, pos_ok, ih0, iw0, at0;
    unsigned out0;
    auto enter = [&](int tile) {
        n0 = int(fastdiv(unsigned(tile * 32), s.d_plane));
        const int p = tile * 32 + l32, pc = min(p, s.n_pos - 1);
        pos_ok = p < s.n_pos;
        const int n = int(fastdiv(unsigned(pc), s.d_plane)), pos = pc - n * oplane;
        const int oh = int(fastdiv(unsigned(pos), s.d_ow)), ow = pos - oh * g.OW;
        ih0 = oh * g.sh - g.pt;
        iw0 = ow * g.sw - g.pl;
        at0 = ((n - n0) * int(img) + ih0 * g.W + iw0) * 4;  // (negative above an image: only padding is there)
        out0 = unsigned(((n - n0) * g.K + lh * 4) * oplane + pos) * 4u;  // < 2^31: checked on the host
    };
    auto gather = [&](int s0, float (&b)[kGroup]) {
        const int64_t left = (g.N - n0) * img * 4;
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(x + n0 * img), 0, int(min(left, int64_t(0x7ffffffc))), 0x00027000);
        uint2 e[kGroup];
#pragma unroll
        for (int j = 0; j < kGroup; ++j) e[j] = tp[2 * (s0 + j)];
#pragma unroll
        for (int j = 0; j < kGroup; ++j) {
            const bool ok = unsigned(ih0 + int(e[j].y >> 16)) < unsigned(g.H) && unsigned(iw0 + int(e[j].y & 0xffffu)) < unsigned(g.W);
            const int off = ok ? at0 + int(e[j].x) : int(0x80000000u);  // past every range
            b[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, 0, 0));
        }
    };
    int i = blockIdx.x;
    if (i >= chunks || tile_of(i) >= s.n_tiles) return;  // (tiles are missing in the last chunk only, which is the last of its workgroup)
    float b0[kGroup], b1[kGroup];
    enter(tile_of(i));
    gather(0, b0);
    while (true) {
        f32x16 acc[KB];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[kb][v] = 0.0f;
        // A group's 16 terms (8 with HALVES) are summed from zero and then added to the total; an instruction rounds once a term,
        // so that is what keeps the sum closer to 64 bits than three split terms' (2-norm 7.1e-8 against 7.2e-8 at 32 terms, 8.8e-8
        // against 1.15e-7 at 64, 9.6e-8 against 1.66e-7 at 128) and than one running f32 sum's (9.0e-8 against 1.55e-7 at 75).
        constexpr int CHUNK = HALVES ? kGroup / 2 : kGroup;
        auto multiply = [&](int s0, const float (&b)[kGroup]) {
#pragma unroll
            for (int j0 = 0; j0 < kGroup; j0 += CHUNK) {
                if (s0 + j0 >= s.steps) break;
                f32x16 part[KB];
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int v = 0; v < 16; ++v) part[kb][v] = 0.0f;
                auto step = [&](int j) {
#pragma unroll
                    for (int kb = 0; kb < KB; ++kb)
                        part[kb] = __builtin_amdgcn_mfma_f32_32x32x2f32(wa[2 * (s0 + j) * PITCH + kb * 32], b[j], part[kb], 0, 0, 0);
                };
                if (s0 + j0 + CHUNK <= s.steps) {
#pragma unroll
                    for (int j = 0; j < CHUNK; ++j) step(j0 + j);
                } else {
#pragma unroll
                    for (int j = 0; j < CHUNK - 1; ++j)
                        if (s0 + j0 + j < s.steps) step(j0 + j);
                }
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[kb][v] += part[kb][v];
            }
        };
        for (int s0 = 0; s0 < s.steps; s0 += 2 * kGroup) {
            if (s0 + kGroup < s.steps) gather(s0 + kGroup, b1);
            multiply(s0, b0);
            if (s0 + kGroup < s.steps) {
                if (s0 + 2 * kGroup < s.steps) gather(s0 + 2 * kGroup, b0);
                multiply(s0 + kGroup, b1);
            }
        }
        char *yb = reinterpret_cast<char *>(y + (int64_t(n0) * g.K + k0) * oplane);
        const unsigned oplane4 = unsigned(oplane) * 4u;
        unsigned off = out0;
        const bool stores = pos_ok;
        // the next tile's first terms are requested ahead of this one's stores: a wave's loads are answered behind older stores
        i += gridDim.x;
        const bool more = i < chunks && tile_of(i) < s.n_tiles;
        if (more) {
            enter(tile_of(i));
            gather(0, b0);
        }
        int row0 = lh * 4;
        asm volatile("" : "+v"(row0));  // opaque, so that the biases are not kept in registers over the tiles
        const float floor = relu ? 0.0f : __builtin_nanf("");  // (the max with a NaN is the other operand, a NaN among them)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            if (kb * 32 >= kn) break;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = row0 + kb * 32 + (v >> 2) * 8 + (v & 3);
                if (stores && (kb * 32 + 32 <= kn || row < kn)) *reinterpret_cast<float *>(yb + off) = vmax(acc[kb][v] + bias_l[row], floor);
                off += (v & 3) == 3 ? 5u * oplane4 : oplane4;
            }
        }
        if (!more) break;
    }
}

template <int KB, bool HALVES>
int launch(zant_ctx *ctx, const float *x, const float *w, const float *bias, float *y, const ConvGeom &g, const ShortGeom &s, int groups,
           int relu) {
    const size_t lds = short_lds_bytes(KB, s.steps);
    const int resident = ctx->num_cus * int(std::max<size_t>(1, std::min<size_t>(KB == 1 ? 7 : 6 - KB, 160 * 1024 / lds)));
    // (eight at least, so that the chunk with tiles missing is some wave's last: see the kernel's tile order)
    const int wgs = std::min((s.n_tiles + 3) / 4, std::max(8, (resident + groups - 1) / groups));
    KernelTimer kt(ctx);
    ZANT_KERNEL_NAME(ctx, "conv_f32_short_kernel<%d,%s>", KB, HALVES ? "true" : "false");
    hipLaunchKernelGGL((conv_f32_short_kernel<KB, HALVES>), dim3(unsigned(wgs), unsigned(groups)), dim3(256), lds, ctx->stream, x, w, bias, y, g, s, relu);
    ZANT_LAUNCH_CHECK(ctx);
    return ZANT_OK;
}

}  // namespace

bool zant_conv_short_ok(const ConvGeom &g) {
    const int64_t terms = int64_t(g.C) * g.KH * g.KW, oplane = int64_t(g.OH) * g.OW, img = int64_t(g.C) * g.H * g.W;
    if (terms > 448 || oplane * g.N + 64 >= (int64_t(1) << 31)) return false;
    if (short_lds_bytes(1, int(terms + 1) / 2) > 64 * 1024) return false;
    const int64_t span = std::min<int64_t>(g.N, 31 / oplane + 2);  // images a tile can touch
    if (span * img * 4 >= 0x70000000 || span * g.K * oplane * 4 >= 0x70000000) return false;
    // filter rows and columns are 16-bit fields of a table, and a term past the last has to lie below every image
    return int64_t(g.H) + g.pt < 32767 && int64_t(g.KH - 1) * g.dh < 32767 && int64_t(g.KW - 1) * g.dw < 65536;
}

// Where it is the better kernel for a layer the split one takes too.  1x1 filters: up to 128 channels (64x64x56x56 to 16 / 64
// filters 43 -> 17 / 52 -> 32 us with the packing the split kernel needs, 128 channels to 64 filters 67 -> 52; to 128 filters
// 64 channels 57 -> 53 and 128 channels 80 -> 88).  Other filters: only where the packing launch weighs, short sums to few channels
// (64x5x56x56 to 32 3x3 filters 16.6 -> 15.6 us, to 64 of them 22.9 -> 25.7) and layers of few positions (1512 positions, 90 terms
// 11.3 -> 8.2 us; 10296, 117 terms 9.5 -> 9.9).  Layers of a few hundred positions, where one launch less saves the same 4 us, are
// left to the split kernel: its behaviour at the edges of the f32 range is pinned on them.
bool zant_conv_short_better(const ConvGeom &g, bool packed_once) {
    const int64_t terms = int64_t(g.C) * g.KH * g.KW, positions = int64_t(g.N) * g.OH * g.OW;
    if (positions < 320) return false;
    if (g.KH * g.KW == 1) return terms <= (g.K > 64 ? 95 : 128);
    if (packed_once) return false;
    return (terms <= 45 && g.K <= 32) || (terms <= 90 && positions <= 8192);
}

int zant_conv_short_run(zant_ctx *ctx, const float *x, const float *w, const float *bias, float *y, const ConvGeom &g, int relu) {
    ShortGeom s;
    s.terms = g.C * g.KH * g.KW;
    s.steps = (s.terms + 1) / 2;
    s.n_pos = g.N * g.OH * g.OW;
    s.n_tiles = (s.n_pos + 31) / 32;
    s.d_terms = make_fastdiv(unsigned(s.terms));
    s.d_taps = make_fastdiv(unsigned(g.KH * g.KW));
    s.d_kw = make_fastdiv(unsigned(g.KW));
    s.d_plane = make_fastdiv(unsigned(g.OH * g.OW));
    s.d_ow = make_fastdiv(unsigned(g.OW));
    // Two or three blocks of channels a workgroup: one block alone gathers the input too often (34 filters over 47 channels, 1.2
    // million positions: 112 against 128 us), four leave two waves a SIMD (128 filters, 9 terms: 49 us against 21).  Fewer while
    // LDS lacks room or the tiles alone leave SIMDs without a wave.
    const int blocks = (g.K + 31) / 32;
    int kb = blocks % 3 == 0 ? 3 : std::min(blocks, 2);
    while (kb > 1 && (short_lds_bytes(kb, s.steps) > 64 * 1024 || int64_t(s.n_tiles) * ((blocks + kb - 1) / kb) < int64_t(ctx->num_cus) * 4)) --kb;
    const int groups = (blocks + kb - 1) / kb;
    if (s.terms > 16 && s.terms <= 36) {  // where sums of 16 terms would be less exact than what the split kernel gives
        if (kb == 1) return launch<1, true>(ctx, x, w, bias, y, g, s, groups, relu);
        if (kb == 2) return launch<2, true>(ctx, x, w, bias, y, g, s, groups, relu);
        return launch<3, true>(ctx, x, w, bias, y, g, s, groups, relu);
    }
    if (kb == 1) return launch<1, false>(ctx, x, w, bias, y, g, s, groups, relu);
    if (kb == 2) return launch<2, false>(ctx, x, w, bias, y, g, s, groups, relu);
    return launch<3, false>(ctx, x, w, bias, y, g, s, groups, relu);
}
