// f32 convolution (conv_lean / OnnxConvLean, reference op_convolution.zig:42-331): entry points, dispatch, and the kernels
// of layers with few input channels.
//
// The reference materialises a zero-padded copy, an im2col matrix, a transposed weight matrix and a matmul result.  Here a
// convolution is one implicit-GEMM kernel (conv_split_f32.hip); layers of short sums are bound by writing their output and run on
// conv_short_f32.hip, with a fused pool on the kernels here.  A direct kernel (one thread per output element) covers what is left.
#include <algorithm>
#include <mutex>

#include "common.h"
#include "conv_split_f32.h"
#include "conv_tile.h"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// One thread per output element; any stride / dilation / pads / kernel size.
__global__ void __launch_bounds__(256) conv_f32_direct_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                             const float *__restrict__ bias, float *__restrict__ y,
                                                             ConvGeom g, int relu) {
    const int64_t total = int64_t(g.N) * g.K * g.OH * g.OW;
    const int64_t step = int64_t(gridDim.x) * blockDim.x;
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += step) {
        const int ow = int(i % g.OW);
        const int oh = int((i / g.OW) % g.OH);
        const int k = int((i / (int64_t(g.OW) * g.OH)) % g.K);
        const int n = int(i / (int64_t(g.OW) * g.OH * g.K));
        float acc = 0.0f;
        for (int c = 0; c < g.C; ++c) {
            const float *xp = x + (int64_t(n) * g.C + c) * g.H * g.W;
            const float *wq = w + (int64_t(k) * g.C + c) * g.KH * g.KW;
            for (int kh = 0; kh < g.KH; ++kh) {
                const int ih = oh * g.sh - g.pt + kh * g.dh;
                if (ih < 0 || ih >= g.H) continue;
                for (int kw = 0; kw < g.KW; ++kw) {
                    const int iw = ow * g.sw - g.pl + kw * g.dw;
                    if (iw < 0 || iw >= g.W) continue;
                    acc = __builtin_fmaf(xp[ih * g.W + iw], wq[kh * g.KW + kw], acc);
                }
            }
        }
        float r = acc + (bias ? bias[k] : 0.0f);
        if (relu) r = r > 0.0f ? r : 0.0f;
        y[i] = r;
    }
}

// Few-input-channel convolution fused with ReLU and a 2x2 / stride-2 max pool (stride-1, undilated
// convolution).  One thread owns one POOLED position: it keeps the (KH+1) x (KW+1) input patch of each
// channel in registers, forms the four convolution outputs of the pooling window for every output
// channel, and writes only their (ReLU'd) maximum: the full-resolution activation never reaches HBM.
template <int C, int KH, int KW>
__global__ void __launch_bounds__(256)
conv_f32_smallc_pool_kernel(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
                            float *__restrict__ y, ConvGeom g, int POH, int POW, int relu) {
    constexpr int PH = KH + 1, PW = KW + 1, CKK = C * KH * KW;
    const int64_t pplane = int64_t(POH) * POW;
    const int64_t total = int64_t(g.N) * pplane;
    const int64_t step = int64_t(gridDim.x) * blockDim.x;
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += step) {
        const int n = int(i / pplane);
        const int pos = int(i - int64_t(n) * pplane);
        const int ph = pos / POW, pw = pos - ph * POW;
        const int ih0 = 2 * ph - g.pt, iw0 = 2 * pw - g.pl;
        float patch[C][PH][PW];
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int r = 0; r < PH; ++r)
#pragma unroll
                for (int q = 0; q < PW; ++q) {
                    const int ih = ih0 + r, iw = iw0 + q;
                    const bool ok = ih >= 0 && ih < g.H && iw >= 0 && iw < g.W;
                    patch[c][r][q] = ok ? x[((int64_t(n) * C + c) * g.H + ih) * g.W + iw] : 0.0f;
                }
        float *yp = y + int64_t(n) * g.K * pplane + pos;
        // The weights of a channel are wave-uniform (scalar loads).  Those of channel k + 1 are requested before the
        // arithmetic of channel k, so the scalar-load latency hides behind 4 * CKK FMAs instead of stalling every channel.
        float wcur[CKK], wnext[CKK];
        const float *bp = bias ? bias : w;  // always loadable: the value is dropped below when there is no bias
        float bcur = bias ? bp[0] : 0.0f, bnext = 0.0f;
#pragma unroll
        for (int e = 0; e < CKK; ++e) wcur[e] = w[e];
        for (int k = 0; k < g.K; ++k) {
            const int kn = k + 1 < g.K ? k + 1 : k;
            const float *wk = w + int64_t(kn) * CKK;
#pragma unroll
            for (int e = 0; e < CKK; ++e) wnext[e] = wk[e];
            const float bl = bp[kn];
            __builtin_amdgcn_sched_barrier(0);  // keep the requests ahead of the arithmetic
            bnext = bias ? bl : 0.0f;
            float a00 = 0.f, a01 = 0.f, a10 = 0.f, a11 = 0.f;
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int kh = 0; kh < KH; ++kh)
#pragma unroll
                    for (int kw = 0; kw < KW; ++kw) {
                        const float wv = wcur[(c * KH + kh) * KW + kw];
                        a00 = __builtin_fmaf(patch[c][kh][kw], wv, a00);
                        a01 = __builtin_fmaf(patch[c][kh][kw + 1], wv, a01);
                        a10 = __builtin_fmaf(patch[c][kh + 1][kw], wv, a10);
                        a11 = __builtin_fmaf(patch[c][kh + 1][kw + 1], wv, a11);
                    }
            // adding the same bias is monotone and so is its rounding: max(a_i + b) == max(a_i) + b exactly
            float r = fmaxf(fmaxf(a00, a01), fmaxf(a10, a11)) + bcur;
            if (relu) r = r > 0.0f ? r : 0.0f;  // max and ReLU commute (both monotone)
            yp[int64_t(k) * pplane] = r;
#pragma unroll
            for (int e = 0; e < CKK; ++e) wcur[e] = wnext[e];
            bcur = bnext;
        }
    }
}

// Single-channel 3x3 first layer + ReLU + MaxPool 2x2/2 on the matrix cores (stride 1, no padding).
//   D[k, p] = sum_t W[k, t] * X[window(p) + tap t]: output channels are the MFMA rows (32 per workgroup), pooled
// positions the columns, and the nine taps the reduction axis, two per v_mfma_f32_32x32x2_f32: (0,0)|(0,1), (1,0)|(1,1),
// (2,0)|(2,1), (0,2)|(1,2), (2,2)|none.  The pairing makes the address of a lane's tap a per-lane base plus an offset
// that is the same for both halves of the wave; the tenth, absent tap reads a word holding 1.0 against the channel's bias
// as its weight, so the matrix cores add the bias too.
// A workgroup copies `imgs` whole images to LDS and walks their pooled positions 32 at a time per wave; the four members
// of a pooling window are four accumulator tiles of the same lane, so the pool is a register-wise max (then ReLU, which
// commutes with it).  20 MFMAs produce 32 positions x 32 channels.  Vector instructions of a SIMD's other waves do not
// hide behind its matrix instructions here (a tile's wall time measured as the sum of both), so everything around the
// MFMAs is kept to a minimum: two instructions per output value and a store without address arithmetic.
template <bool RELU, bool FULLK>
__global__ void __launch_bounds__(256, 4) conv_f32_c1k3_pool_mfma_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                                     const float *__restrict__ bias, float *__restrict__ y,
                                                                     int N, int H, int W, int K, int POH, int POW, int imgs,
                                                                     FastDiv dpp, FastDiv dpw, int y_c4) {
    extern __shared__ __attribute__((aligned(16))) float img_lds[];  // [imgs][H][W], four words (1, 0, 0, 0), weights, bias
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform by construction; says so to the compiler (LDS
                                                                // copy destinations then stay in scalar registers)
    const int l32 = lane & 31, lh = lane >> 5;
    const int HW = H * W, PP = POH * POW;
    const int n0 = blockIdx.x * imgs, imgs_here = min(imgs, N - n0);
    const int kb = blockIdx.y * 32;
    const int cnt = imgs_here * HW;
    const float *src = x + int64_t(n0) * HW;
    if ((HW & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0) {
        for (int i = tid; i < (cnt >> 2); i += 256)
            reinterpret_cast<f32x4 *>(img_lds)[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(src) + i);
    } else {
        for (int i = tid; i < cnt; i += 256) img_lds[i] = src[i];
    }
    // [0]: the word the absent tenth tap of the upper half-wave reads -- 1.0, against the channel's bias as its weight, so
    // the last MFMA adds the bias; [1..3]: zero
    const int one_idx = imgs * HW;
    if (tid < 4) img_lds[one_idx + tid] = tid == 0 ? 1.0f : 0.0f;
    // Weights and bias of the workgroup's 32 channels go through LDS: one coalesced read per workgroup, where per-lane
    // reads would be 21 scattered loads per wave, queued in front of the other workgroups' image loads on the CU.
    float *wl = img_lds + one_idx + 4;  // [32][9] weights, then [32] bias
    for (int i = tid; i < 32 * 9 + 32; i += 256) {
        float v = 0.0f;
        if (i < 32 * 9) {
            if (kb + i / 9 < K) v = w[int64_t(kb) * 9 + i];
        } else if (bias != nullptr && kb + i - 32 * 9 < K) {
            v = bias[kb + i - 32 * 9];
        }
        wl[i] = v;
    }
    __syncthreads();

    // this lane's A operands: channel kb + l32, tap pair member lh; the tenth "tap" is the bias
    float wa[5];
    {
        const float *wr = wl + l32 * 9;
        wa[0] = wr[0 + lh];
        wa[1] = wr[3 + lh];
        wa[2] = wr[6 + lh];
        wa[3] = wr[lh ? 5 : 2];
        wa[4] = lh ? wl[32 * 9 + l32] : wr[8];
    }

    const int total = imgs_here * PP;
    // store bases of this lane group's 16 output channels: workgroup-uniform, pinned to scalar registers
    unsigned long long ybase[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const unsigned long long a = reinterpret_cast<unsigned long long>(y + (int64_t(n0) * K + kb + (v >> 2) * 8 + (v & 3)) * PP);
        // (the builtin returns int: without the casts the low word would be sign-extended over the high one)
        const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(unsigned(a))));
        const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(unsigned(a >> 32))));
        ybase[v] = (static_cast<unsigned long long>(hi) << 32) | static_cast<unsigned long long>(lo);
    }
    // quad-blocked output ([N][K/4][PP][4]): this lane's four groups of four consecutive channels are four 16-byte units,
    // 2 * PP units apart; their bases (group offset included) likewise sit in scalar registers
    unsigned long long ybase4[4];
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
        const unsigned long long a = reinterpret_cast<unsigned long long>(y + (int64_t(n0) * K + kb + gq * 8) * PP);
        const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(unsigned(a))));
        const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(unsigned(a >> 32))));
        ybase4[gq] = (static_cast<unsigned long long>(hi) << 32) | static_cast<unsigned long long>(lo);
    }
    for (int p0 = wave * 32; p0 < total; p0 += 4 * 32) {
        // Waves with more steps left go first.  Left alone the SIMD serves its oldest waves first: the youngest workgroup on
        // a CU then runs most of its steps after the others are gone, one wave per SIMD, which keeps the matrix pipe half
        // busy; with the laggards in front the four waves of a SIMD finish together.
        {
            const int left = (total - p0 + 127) >> 7;
            if (left >= 5) __builtin_amdgcn_s_setprio(3);
            else if (left >= 3) __builtin_amdgcn_s_setprio(2);
            else if (left == 2) __builtin_amdgcn_s_setprio(1);
            else __builtin_amdgcn_s_setprio(0);
        }
        const int p = p0 + l32;
        const bool valid = p < total;
        const unsigned pc_ = valid ? unsigned(p) : 0u;
        const unsigned img = fastdiv(pc_, dpp), pp = pc_ - img * unsigned(PP);
        const unsigned pr = fastdiv(pp, dpw), pcol = pp - pr * unsigned(POW);
        const int wb = int(img) * HW + int(2 * pr) * W + int(2 * pcol);  // window origin in LDS
        const int a012 = wb + lh, a3 = wb + 2 + lh * W;
        f32x16 acc[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[j][v] = 0.0f;
        float b[5][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int to = (j >> 1) * W + (j & 1);  // window member (dy, dx)
            b[0][j] = img_lds[a012 + to];
            b[1][j] = img_lds[a012 + to + W];
            b[2][j] = img_lds[a012 + to + 2 * W];
            b[3][j] = img_lds[a3 + to];
            b[4][j] = img_lds[lh ? one_idx : wb + to + 2 * W + 2];
        }
        // tap pairs outermost: consecutive MFMAs go to different accumulators
#pragma unroll
        for (int t = 0; t < 5; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(wa[t], b[t][j], acc[j], 0, 0, 0);
        if (valid) {
            // One 32-bit byte offset per lane and a uniform base per output channel, kept in scalar registers (the host
            // checks that N * K * PP * 4 fits in 32 bits): the stores need no address arithmetic in the vector unit, which
            // this kernel's matrix instructions leave little room for.  The bias came in through the tenth tap; adding the
            // same bias to the four window members is monotone, so the maximum below is pool(conv + bias) exactly.
            const unsigned byte_off = ((unsigned(img) * unsigned(K) + unsigned(lh * 4)) * unsigned(PP) + pp) * 4u;
            // The first three window members first, for all 16 values: the fourth accumulator tile is the one the last
            // MFMA is still writing, and these 16 instructions are the distance its readers must keep from it.
            float m3[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) m3[v] = vmax3(acc[0][v], acc[1][v], acc[2][v]);
            __builtin_amdgcn_sched_barrier(0);
            if (y_c4) {
                // quad (kb + gq*8 + lh*4) / 4 of image n0 + img: unit ((img * K/4 + lh) * PP + pp) past the group's base
                const unsigned off16 = ((unsigned(img) * unsigned(K >> 2) + unsigned(lh)) * unsigned(PP) + pp) * 16u;
#pragma unroll
                for (int gq = 0; gq < 4; ++gq) {
                    if (FULLK || kb + gq * 8 + lh * 4 < K) {  // K is a multiple of 4 here: a quad is whole or absent
                        f32x4 o4;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            o4[e] = RELU ? vmax3(m3[gq * 4 + e], acc[3][gq * 4 + e], 0.0f) : vmax(m3[gq * 4 + e], acc[3][gq * 4 + e]);
                        // (a store of more than 8 bytes reads its data over the next cycles: the two wait states keep the
                        // next vector write to these registers -- which the compiler cannot tell apart through the
                        // statement -- behind it)
                        asm volatile("global_store_dwordx4 %0, %1, %2\n\ts_nop 1" : : "v"(off16), "v"(o4), "s"(ybase4[gq]) : "memory");
                    }
                }
            } else {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int dk = (v >> 2) * 8 + (v & 3);
                if (FULLK || kb + lh * 4 + dk < K) {
                    const float o = RELU ? vmax3(m3[v], acc[3][v], 0.0f) : vmax(m3[v], acc[3][v]);
                    asm volatile("global_store_dword %0, %1, %2" : : "v"(byte_off), "v"(o), "s"(ybase[v]) : "memory");
                }
            }
            }
        }
    }
}

}  // namespace

int zant_conv_resolve(const int64_t xdim[4], const int64_t wdim[4], const int64_t *stride, int n_stride,
                      const int64_t *pads, int n_pads, const int64_t *dil, int n_dil, int64_t group,
                      const char *auto_pad, int64_t s[2], int64_t d[2], int64_t p[4]) {
    if (group >= 0 && group != 1) return ZANT_InvalidDimensions;  // op_convolution.zig:60-65
    if (!stride || n_stride < 1) return ZANT_WrongStride;
    s[0] = stride[0];                                              // :68
    s[1] = n_stride > 1 ? stride[1] : stride[0];                   // :69
    d[0] = (dil && n_dil > 0) ? dil[0] : 1;                        // :70
    d[1] = dil ? (n_dil > 1 ? dil[1] : (n_dil > 0 ? dil[0] : 1)) : 1;  // :71
    if (s[0] <= 0 || s[1] <= 0 || d[0] <= 0 || d[1] <= 0) return ZANT_WrongStride;
    const int64_t dkh = (wdim[2] - 1) * d[0] + 1, dkw = (wdim[3] - 1) * d[1] + 1;  // :74-75
    p[0] = p[1] = p[2] = p[3] = 0;  // h_begin, w_begin, h_end, w_end
    if (auto_pad) {
        const bool upper = !strcmp(auto_pad, "SAME_UPPER"), lower = !strcmp(auto_pad, "SAME_LOWER");
        if (upper || lower) {
            const int64_t oh = ceil_div64(xdim[2], s[0]), ow = ceil_div64(xdim[3], s[1]);  // :92-93
            int64_t th = (oh - 1) * s[0] + dkh - xdim[2], tw = (ow - 1) * s[1] + dkw - xdim[3];  // :96-97
            if (th < 0) th = 0;
            if (tw < 0) tw = 0;
            if (upper) { p[0] = th / 2; p[2] = th - p[0]; p[1] = tw / 2; p[3] = tw - p[1]; }  // :101-104
            else { p[2] = th / 2; p[0] = th - p[2]; p[3] = tw / 2; p[1] = tw - p[3]; }         // :106-109
        } else if (!strcmp(auto_pad, "NOTSET")) {
            if (!pads) return ZANT_InvalidPadding;  // :120-125
            if (n_pads >= 4) { p[0] = pads[0]; p[1] = pads[1]; p[2] = pads[2]; p[3] = pads[3]; }  // :114-119
        }
        // "VALID" and unknown strings: no padding (:88-89, :126-128)
    }
    // auto_pad == null: pads are ignored (:86)
    return ZANT_OK;
}

extern "C" int zant_hip_conv2d_out_shape(const int64_t xdim[4], const int64_t wdim[4], const int64_t *stride,
                                         int n_stride, const int64_t *pads, int n_pads, const int64_t *dil, int n_dil,
                                         int64_t group, const char *auto_pad, int64_t ydim[4]) {
    // OnnxConv, op_convolution.zig:647-732
    if (!xdim || !wdim || !ydim) return ZANT_NullPointer;
    if (group >= 0 && group != 1) return ZANT_InvalidDimensions;
    if (!stride || n_stride < 1) return ZANT_WrongStride;
    const int64_t sh = stride[0], sw = n_stride > 1 ? stride[1] : stride[0];
    const int64_t dh = (dil && n_dil > 0) ? dil[0] : 1;
    const int64_t dw = dil ? (n_dil > 1 ? dil[1] : (n_dil > 0 ? dil[0] : 1)) : 1;
    if (sh <= 0 || sw <= 0) return ZANT_WrongStride;
    const int64_t dkh = (wdim[2] - 1) * dh + 1, dkw = (wdim[3] - 1) * dw + 1;
    const int64_t H = xdim[2], W = xdim[3];
    int64_t oh, ow;
    if (auto_pad) {
        if (!strcmp(auto_pad, "VALID")) {
            oh = (H - dkh) / sh + 1; ow = (W - dkw) / sw + 1;
        } else if (!strcmp(auto_pad, "SAME_UPPER") || !strcmp(auto_pad, "SAME_LOWER")) {
            oh = ceil_div64(H, sh); ow = ceil_div64(W, sw);
        } else if (!strcmp(auto_pad, "NOTSET")) {
            if (pads) {
                if (n_pads < 4) return ZANT_InvalidPadding;  // :713-715
                oh = (H + pads[0] + pads[2] - dkh) / sh + 1;
                ow = (W + pads[1] + pads[3] - dkw) / sw + 1;
            } else {
                oh = (H - dkh) / sh + 1; ow = (W - dkw) / sw + 1;  // :717-718
            }
        } else {
            return ZANT_InvalidPadding;  // :720-722
        }
    } else {
        const int64_t th = (pads && n_pads >= 4) ? pads[0] + pads[2] : 0;  // :725-728
        const int64_t tw = (pads && n_pads >= 4) ? pads[1] + pads[3] : 0;
        oh = (H + th - dkh) / sh + 1; ow = (W + tw - dkw) / sw + 1;
    }
    ydim[0] = xdim[0]; ydim[1] = wdim[0]; ydim[2] = oh; ydim[3] = ow;
    return ZANT_OK;
}

extern "C" int zant_hip_conv2d_f32(zant_ctx *ctx, const float *x, const int64_t xdim[4], const float *w,
                                   const int64_t wdim[4], const float *bias, float *y, const int64_t ydim[4],
                                   const int64_t *stride, int n_stride, const int64_t *pads, int n_pads,
                                   const int64_t *dil, int n_dil, int64_t group, const char *auto_pad, int fuse_act) {
    return zant_conv2d_f32_slot(ctx, x, xdim, w, wdim, bias, y, ydim, stride, n_stride, pads, n_pads, dil, n_dil, group, auto_pad,
                                fuse_act, nullptr);
}

// ---- zant_hip_conv2d_f32_static: the same convolution for callers that cannot allocate ---------------------------
//
// The matrix-core kernel's scratch (the packed weights) lives in a static device array instead of the context workspace;
// three bf16 terms a weight and the kernel's own padding take at most four times the limit that is stated in f32 weights.
// `scratch` below is only the host-side handle of that array: every device holds its own copy at its own address, which
// hipGetSymbolAddress returns and which is what kernels, copies and fills must be given.  The array is shared by every call
// on a device and keeps the previous call's contents; each call re-packs the weights before its convolution kernel, in stream
// order, so calls on ONE stream are safe back to back, while calls that overlap on one device (two contexts, two streams) race.
static __device__ __align__(256) unsigned char scratch[4 * ZANT_HIP_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices];        // device address of `scratch` per device, nullptr until resolved
hipError_t g_scratch_err[kMaxDevices];   // what hipGetSymbolAddress returned on that device
bool g_scratch_tried[kMaxDevices];
}  // namespace

void zant_conv_static_scratch_init(int device) {
    if (device < 0 || device >= kMaxDevices) return;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_tried[device]) return;
    g_scratch_tried[device] = true;
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));  // `device` is current (see the caller)
    g_scratch_err[device] = e;
    g_scratch_ptr[device] = e == hipSuccess ? ptr : nullptr;
}

extern "C" int zant_hip_conv2d_f32_static(zant_ctx *ctx, const float *x, const int64_t xdim[4], const float *w,
                                          const int64_t wdim[4], const float *bias, float *y, const int64_t ydim[4],
                                          const int64_t *stride, int n_stride, const int64_t *pads, int n_pads,
                                          const int64_t *dil, int n_dil, int64_t group, const char *auto_pad,
                                          int fuse_act) {
    if (!ctx) return ZANT_NullPointer;
    if (ctx->device < 0 || ctx->device >= kMaxDevices) return ZANT_InvalidInput;
    void *ptr;
    hipError_t e;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        ptr = g_scratch_ptr[ctx->device];
        e = g_scratch_err[ctx->device];
    }
    if (!ptr) return zant_fail_hip(ctx, e == hipSuccess ? hipErrorNotInitialized : e, "hipGetSymbolAddress(scratch)");
    zant_pack_slot slot;
    slot.dev = ptr;
    slot.bytes = 4 * ZANT_HIP_STATIC_SCRATCH_BYTES;
    slot.fixed = true;
    return zant_conv2d_f32_slot(ctx, x, xdim, w, wdim, bias, y, ydim, stride, n_stride, pads, n_pads, dil, n_dil, group,
                                auto_pad, fuse_act, &slot);
}

namespace {
// Layers that zant_hip_conv2d_f32_static takes whatever the size of their weights, on the direct kernel: fewer than 64 output
// positions, or no tile of whole output rows (32 to 256 positions x 32 or 64 channels, 8 input channels a step, two staging
// buffers in half of LDS) of which they fill half.  Callers rely on that line; it does not follow what the matrix-core kernel
// can tile, which is more.
bool needs_no_scratch(const ConvGeom &g) {
    if (int64_t(g.N) * g.OH * g.OW < 64 || int64_t(g.N) * g.C * g.H * g.W >= (int64_t(1) << 40)) return true;
    const size_t cap = 80 * 1024 - (size_t((g.K + 63) / 64) * 64 * sizeof(float) + 8);
    auto tile = [&](int WM, int WN, TilePlan *p) {
        return zant_plan_conv_tiles(g, WM, WN, 8, 8, sizeof(float), cap, p, false, 0, 32, 0, 2, 4, 256, 4096);
    };
    TilePlan narrow, wide;
    const bool ok_n = tile(4, 1, &narrow), ok_w = g.K > 32 && tile(2, 2, &wide);
    if (ok_w && !(ok_n && narrow.eff > wide.eff + 0.25)) return wide.eff < 0.5;
    return !ok_n || narrow.eff < 0.5;
}
}  // namespace

int zant_conv2d_f32_slot(zant_ctx *ctx, const float *x, const int64_t xdim[4], const float *w, const int64_t wdim[4],
                         const float *bias, float *y, const int64_t ydim[4], const int64_t *stride, int n_stride,
                         const int64_t *pads, int n_pads, const int64_t *dil, int n_dil, int64_t group, const char *auto_pad,
                         int fuse_act, zant_pack_slot *slot, int x_c4) {
    if (!ctx || !xdim || !wdim || !ydim) return ZANT_NullPointer;
    zant_log("OnnxConvLean1");
    int64_t s[2], d[2], p[4];
    int rc = zant_conv_resolve(xdim, wdim, stride, n_stride, pads, n_pads, dil, n_dil, group, auto_pad, s, d, p);
    if (rc) { zant_log(rc == ZANT_InvalidPadding ? "OnnxConvLeanError2" : "OnnxConvLeanError1"); return rc; }
    for (int i = 0; i < 4; ++i)
        if (xdim[i] <= 0 || wdim[i] <= 0 || xdim[i] > INT32_MAX || wdim[i] > INT32_MAX) return ZANT_InvalidDimensions;
    const int64_t PH = xdim[2] + p[0] + p[2], PW = xdim[3] + p[1] + p[3];
    const int64_t dkh = (wdim[2] - 1) * d[0] + 1, dkw = (wdim[3] - 1) * d[1] + 1;
    if (PH < dkh || PW < dkw) return ZANT_InvalidDimensions;               // op_convolution.zig:250, :394
    if (xdim[1] != wdim[1]) return ZANT_InputTensorsWrongShape;            // im2col cols != kernel rows (op_mat_mul.zig:34)
    const int64_t OH = (PH - dkh) / s[0] + 1, OW = (PW - dkw) / s[1] + 1;  // :247-248
    if (ydim[0] != xdim[0] || ydim[1] != wdim[0] || ydim[2] != OH || ydim[3] != OW) return ZANT_InvalidDimensions;  // :212-217
    if (OH > INT32_MAX || OW > INT32_MAX || PH > INT32_MAX || PW > INT32_MAX) return ZANT_InvalidDimensions;
    if (!x || !w || !y) return ZANT_NullPointer;
    if (fuse_act != ZANT_ACT_NONE && fuse_act != ZANT_ACT_RELU) return ZANT_InvalidInput;

    ConvGeom g;
    g.N = int(xdim[0]); g.C = int(xdim[1]); g.H = int(xdim[2]); g.W = int(xdim[3]);
    g.K = int(wdim[0]); g.CG = int(wdim[1]); g.KH = int(wdim[2]); g.KW = int(wdim[3]);
    g.OH = int(OH); g.OW = int(OW);
    g.sh = int(s[0]); g.sw = int(s[1]); g.dh = int(d[0]); g.dw = int(d[1]);
    g.pt = int(p[0]); g.pl = int(p[1]); g.groups = 1;
    const int relu = fuse_act == ZANT_ACT_RELU;
    zant_log("OnnxConvLean2");

    SplitPlan plan;
    const bool no_room = slot && slot->fixed && zant_conv_split_fixed_bytes(g) > ZANT_HIP_STATIC_SCRATCH_BYTES;
    const bool short_ok = !x_c4 && zant_conv_short_ok(g);
    const bool split_first = x_c4 || no_room || !short_ok || !zant_conv_short_better(g, slot && !slot->fixed);
    if (split_first && zant_conv_split_plan(g, false, ctx->num_cus, &plan, slot) && !(no_room && needs_no_scratch(g))) {
        rc = zant_conv_split_run(ctx, x, w, bias, y, g, plan, relu, false, slot, x_c4);
        if (rc == ZANT_OK) zant_log("OnnxConvLean4");
        return rc;
    }
    if (x_c4) return ZANT_InvalidInput;  // only the matrix-core kernel reads the quad-blocked layout (see zant_conv2d_f32_c4_caps)
    const int64_t total = int64_t(g.N) * g.K * g.OH * g.OW;
    // (sums of one or two terms for few outputs: a thread an output is done before the other kernel has its weights in LDS,
    // 7514 positions, 36 filters 4.5 against 4.8 us, 24192 positions, 19 filters 5.2 against 4.6)
    if (short_ok && (int64_t(g.C) * g.KH * g.KW > 2 || total > 400 * 1000)) {
        rc = zant_conv_short_run(ctx, x, w, bias, y, g, relu);
        if (rc == ZANT_OK) zant_log("OnnxConvLean4");
        return rc;
    }
    int64_t blocks = ceil_div64(total, 256);
    if (blocks > int64_t(ctx->num_cus) * 32) blocks = int64_t(ctx->num_cus) * 32;
    KernelTimer kt(ctx);
    ZANT_KERNEL_NAME(ctx, "conv_f32_direct_kernel");
    hipLaunchKernelGGL(conv_f32_direct_kernel, dim3(unsigned(blocks)), dim3(256), 0, ctx->stream, x, w, bias, y, g, relu);
    ZANT_LAUNCH_CHECK(ctx);
    zant_log("OnnxConvLean4");
    return ZANT_OK;
}

// Conv (+ReLU) + MaxPool 2x2/2 in one kernel (few-channel first layers: direct kernel; many-channel layers: the
// implicit-GEMM kernel with a register-wise pool in its epilogue); returns 1 when the shape is
// not one this kernel takes (the caller then runs the two operators separately).
int zant_conv2d_f32_fused_pool(zant_ctx *ctx, const float *x, const int64_t xdim[4], const float *w, const int64_t wdim[4],
                               const float *bias, float *y, const int64_t ydim[4], const int64_t *stride, int n_stride,
                               const int64_t *pads, int n_pads, const int64_t *dil, int n_dil, int64_t group,
                               const char *auto_pad, int relu, bool query_only, zant_pack_slot *slot, int x_c4, int y_c4) {
    int64_t s[2], d[2], p[4];
    if (zant_conv_resolve(xdim, wdim, stride, n_stride, pads, n_pads, dil, n_dil, group, auto_pad, s, d, p)) return 1;
    if (s[0] != 1 || s[1] != 1 || d[0] != 1 || d[1] != 1 || xdim[1] != wdim[1]) return 1;
    const int C = int(wdim[1]), KH = int(wdim[2]), KW = int(wdim[3]);
    const bool k133 = C == 1 && KH == 3 && KW == 3, k155 = C == 1 && KH == 5 && KW == 5, k333 = C == 3 && KH == 3 && KW == 3;
    const int64_t OH = xdim[2] + p[0] + p[2] - KH + 1, OW = xdim[3] + p[1] + p[3] - KW + 1;
    if (OH < 2 || OW < 2) return 1;
    if (ydim[0] != xdim[0] || ydim[1] != wdim[0] || ydim[2] != OH / 2 || ydim[3] != OW / 2) return 1;
    for (int i = 0; i < 4; ++i)
        if (xdim[i] <= 0 || wdim[i] <= 0 || xdim[i] > INT32_MAX || wdim[i] > INT32_MAX) return 1;
    ConvGeom g;
    g.N = int(xdim[0]); g.C = C; g.H = int(xdim[2]); g.W = int(xdim[3]);
    g.K = int(wdim[0]); g.CG = C; g.KH = KH; g.KW = KW; g.OH = int(OH); g.OW = int(OW);
    g.sh = g.sw = g.dh = g.dw = 1; g.pt = int(p[0]); g.pl = int(p[1]); g.groups = 1;
    if (!k133 && !k155 && !k333) {
        // many-channel layers: the implicit-GEMM kernel with the pool folded into its epilogue
        SplitPlan plan;
        if (!zant_conv_split_plan(g, true, ctx ? ctx->num_cus : 256, &plan, slot)) return 1;
        if (query_only) return ZANT_OK;
        if (y_c4) return ZANT_InvalidInput;  // (zant_conv2d_f32_c4_caps says which kernel writes that layout)
        return zant_conv_split_run(ctx, x, w, bias, y, g, plan, relu, true, slot, x_c4);
    }
    if (query_only) return ZANT_OK;
    if (x_c4) return ZANT_InvalidInput;
    const int POH = int(OH / 2), POW = int(OW / 2);
    if (k133 && g.pt == 0 && g.pl == 0 && OH == xdim[2] - 2 && OW == xdim[3] - 2 && int64_t(g.H) * g.W * 4 <= 40 * 1024 &&
        int64_t(POH) * POW < (1 << 20) && int64_t(g.N) * g.K * POH * POW < (int64_t(1) << 30)) {
        // the matrix-core first layer: four whole images per workgroup (fewer if they do not fit in 40 KB of LDS); with
        // its 104 registers four workgroups share a CU, which measured better than eight images and two workgroups
        const int imgs = int(std::min<int64_t>(4, (40 * 1024) / (int64_t(g.H) * g.W * 4)));
        const dim3 grid(unsigned(ceil_div64(g.N, imgs)), unsigned(ceil_div64(g.K, 32)));
        KernelTimer kt(ctx);
        const size_t lds = size_t(imgs) * g.H * g.W * 4 + 16 + (32 * 9 + 32) * 4;
        const FastDiv dpp = make_fastdiv(unsigned(POH * POW)), dpw = make_fastdiv(unsigned(POW));
        const bool fullk = g.K % 32 == 0;
        ZANT_KERNEL_NAME(ctx, "conv_f32_c1k3_pool_mfma_kernel<%s,%s>", relu ? "true" : "false", fullk ? "true" : "false");
#define ZANT_C1K3(R, F)                                                                                                      \
    hipLaunchKernelGGL((conv_f32_c1k3_pool_mfma_kernel<R, F>), grid, dim3(256), lds, ctx->stream, x, w, bias, y, g.N, g.H, g.W, g.K, \
                       POH, POW, imgs, dpp, dpw, (y_c4 && g.K % 4 == 0) ? 1 : 0)
        if (y_c4 && g.K % 4 != 0) return ZANT_InvalidInput;
        if (relu) { if (fullk) ZANT_C1K3(true, true); else ZANT_C1K3(true, false); }
        else { if (fullk) ZANT_C1K3(false, true); else ZANT_C1K3(false, false); }
#undef ZANT_C1K3
        ZANT_LAUNCH_CHECK(ctx);
        return ZANT_OK;
    }
    if (y_c4) return ZANT_InvalidInput;
    const int64_t positions = int64_t(g.N) * POH * POW;
    const unsigned pb = unsigned(std::min<int64_t>(ceil_div64(positions, 256), int64_t(ctx->num_cus) * 16));
    KernelTimer kt(ctx);
    ZANT_KERNEL_NAME(ctx, "conv_f32_smallc_pool_kernel<%s>", k133 ? "1,3,3" : k155 ? "1,5,5" : "3,3,3");
    if (k133) hipLaunchKernelGGL((conv_f32_smallc_pool_kernel<1, 3, 3>), dim3(pb), dim3(256), 0, ctx->stream, x, w, bias, y, g, POH, POW, relu);
    else if (k155) hipLaunchKernelGGL((conv_f32_smallc_pool_kernel<1, 5, 5>), dim3(pb), dim3(256), 0, ctx->stream, x, w, bias, y, g, POH, POW, relu);
    else hipLaunchKernelGGL((conv_f32_smallc_pool_kernel<3, 3, 3>), dim3(pb), dim3(256), 0, ctx->stream, x, w, bias, y, g, POH, POW, relu);
    ZANT_LAUNCH_CHECK(ctx);
    return ZANT_OK;
}

// Which kernel will run a convolution node decides which of its tensors may be quad-blocked: the implicit-GEMM kernel
// reads that layout (with the fused pool or without), the single-channel 3x3 first-layer kernel with the fused pool
// writes it.  The conditions repeat those of zant_conv2d_f32_slot / zant_conv2d_f32_fused_pool above.
void zant_conv2d_f32_c4_caps(const int64_t xdim[4], const int64_t wdim[4], const int64_t ydim[4], const int64_t *stride,
                             int n_stride, const int64_t *pads, int n_pads, const int64_t *dil, int n_dil, int64_t group,
                             const char *auto_pad, bool fuse_pool, int *in_ok, int *out_ok) {
    *in_ok = *out_ok = 0;
    int64_t s[2], d[2], p[4];
    if (zant_conv_resolve(xdim, wdim, stride, n_stride, pads, n_pads, dil, n_dil, group, auto_pad, s, d, p)) return;
    for (int i = 0; i < 4; ++i)
        if (xdim[i] <= 0 || wdim[i] <= 0 || xdim[i] > INT32_MAX || wdim[i] > INT32_MAX) return;
    if (xdim[1] != wdim[1]) return;
    const int64_t PH = xdim[2] + p[0] + p[2], PW = xdim[3] + p[1] + p[3];
    const int64_t dkh = (wdim[2] - 1) * d[0] + 1, dkw = (wdim[3] - 1) * d[1] + 1;
    if (PH < dkh || PW < dkw) return;
    const int64_t OH = (PH - dkh) / s[0] + 1, OW = (PW - dkw) / s[1] + 1;
    if (OH > INT32_MAX || OW > INT32_MAX) return;
    ConvGeom g;
    g.N = int(xdim[0]); g.C = int(xdim[1]); g.H = int(xdim[2]); g.W = int(xdim[3]);
    g.K = int(wdim[0]); g.CG = int(wdim[1]); g.KH = int(wdim[2]); g.KW = int(wdim[3]);
    g.OH = int(OH); g.OW = int(OW);
    g.sh = int(s[0]); g.sw = int(s[1]); g.dh = int(d[0]); g.dw = int(d[1]);
    g.pt = int(p[0]); g.pl = int(p[1]); g.groups = 1;
    SplitPlan plan;
    if (!fuse_pool) {
        *in_ok = (g.C % 4 == 0) && zant_conv_split_plan(g, false, 256, &plan);
        return;
    }
    if (s[0] != 1 || s[1] != 1 || d[0] != 1 || d[1] != 1) return;
    const bool k133 = g.C == 1 && g.KH == 3 && g.KW == 3, k155 = g.C == 1 && g.KH == 5 && g.KW == 5,
               k333 = g.C == 3 && g.KH == 3 && g.KW == 3;
    if (!k133 && !k155 && !k333) {
        *in_ok = (g.C % 4 == 0) && zant_conv_split_plan(g, true, 256, &plan);
        return;
    }
    const int POH = int(OH / 2), POW = int(OW / 2);
    *out_ok = k133 && g.K % 4 == 0 && g.pt == 0 && g.pl == 0 && OH == xdim[2] - 2 && OW == xdim[3] - 2 &&
              int64_t(g.H) * g.W * 4 <= 40 * 1024 && int64_t(POH) * POW < (1 << 20) &&
              int64_t(g.N) * g.K * POH * POW < (int64_t(1) << 30) && ydim[2] == POH && ydim[3] == POW;
}

namespace {
__global__ void __launch_bounds__(256) from_c4_f32_kernel(const f32x4 *__restrict__ x, float *__restrict__ y, int64_t units,
                                                          int64_t HW) {
    const int64_t step = int64_t(gridDim.x) * blockDim.x;
    for (int64_t u = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; u < units; u += step) {
        const int64_t q = u / HW, pos = u - q * HW;  // q = n * C/4 + quad: NCHW plane 4q + e
        const f32x4 v = x[u];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[(q * 4 + e) * HW + pos] = v[e];
    }
}
}  // namespace

int zant_from_c4_f32(zant_ctx *ctx, const float *x, int64_t N, int64_t C, int64_t HW, float *y) {
    if (!ctx || !x || !y) return ZANT_NullPointer;
    if (C % 4 != 0) return ZANT_InvalidInput;
    const int64_t units = N * (C / 4) * HW;
    if (units == 0) return ZANT_OK;
    const unsigned blocks = unsigned(std::min<int64_t>(ceil_div64(units, 256), int64_t(ctx->num_cus) * 16));
    hipLaunchKernelGGL(from_c4_f32_kernel, dim3(blocks), dim3(256), 0, ctx->stream, reinterpret_cast<const f32x4 *>(x), y, units, HW);
    ZANT_LAUNCH_CHECK(ctx);
    return ZANT_OK;
}
