// Consecutive inverted residual blocks of MobileNetV2 on the int8 matrix cores, one image a workgroup from the first block to the
// last: for batches that leave the chip's CUs an image or two each.
//
// Bound by latency: a late block is a few dozen matrix instructions, and what it takes is a chain of dependent steps -- weights from
// memory, operand reads, products, table look-ups, barriers.  So nothing of a block waits that need not: its weights and tables
// come into LDS while the block before it computes, its input is written there by the block before it (and kept for the
// residual add), its arguments are in the scalar cache from the start, and sixteen waves share every stage.  A stage's units --
// (32 positions x 32 expanded channels) in the expansion, (32 output positions x 32 expanded channels) in the depthwise and
// projection stage, (32 positions x 8 output channels) in the last -- are dealt to the waves one by one, and the projection's
// sums meet in LDS by integer additions, whose order does not matter.  The arithmetic is qblock_kernel's: the same bytes.
// MobileNetV2-0.35's last 14 blocks, one image: 139 us as two tile chains and a block, 97 with eight waves, 82 with sixteen, 71 with the
// tables packed beside the weights (they were the longest unit) and the arguments prefetched, 69 with lookups by address.  Of a block's 5 us the expansion
// takes 1.3, depthwise and projection 2, the last stage 1.2, mostly vector instructions of three or four waves a SIMD.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "qblock_i8.h"

namespace {

typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i32x4 lds_i32x4;

constexpr int kThreads = 1024, kWaves = 16;
constexpr int kAhead = 4;       // 16-byte units of the next block's weights a thread holds while the expansion runs
constexpr int kMaxBlocks = 15;  // what the kernel argument segment (4 KB) has room for
constexpr size_t kLdsMax = 160 * 1024;

// One block; the LDS offsets in `a` are those of the chain's plan.
struct ImageLink {
    const uint4 *packed;
    uint8_t *y;
    QBlockArgs a;
    int co32;      // blocks of 32 output channels
    int o_r;       // projection sums: [32-position tile][32-channel block][accumulator register][lane]
    int late;      // LDS has no room for this block's weights while the block before it runs: they are loaded after it
};
struct ImageChain {
    const uint4 *x;
    int n;
    ImageLink link[kMaxBlocks];
};
static_assert(sizeof(ImageChain) <= 4096, "kernel arguments");

__device__ __forceinline__ i32x4 as_i32x4(const uint4 &v) {
    i32x4 r;
    r[0] = int(v.x); r[1] = int(v.y); r[2] = int(v.z); r[3] = int(v.w);
    return r;
}

// What this wave wrote to LDS is there and its reads are done; global loads and stores stay in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// units [from, all) of a block's packed weights and tables: memory -> LDS
__device__ __forceinline__ void copy_weights(const ImageLink &l, char *lds, int tid, int from) {
    i32x4 *dst = reinterpret_cast<i32x4 *>(lds + l.a.o_w1);
    const int units = l.a.packed_units;
    for (int i0 = from; i0 < units; i0 += kAhead * kThreads) {
        i32x4 v[kAhead];
#pragma unroll
        for (int r = 0; r < kAhead; ++r) v[r] = *reinterpret_cast<const i32x4 *>(l.packed + min(i0 + r * kThreads + tid, units - 1));
#pragma unroll
        for (int r = 0; r < kAhead; ++r)
            if (i0 + r * kThreads + tid < units) dst[i0 + r * kThreads + tid] = v[r];
    }
}

__device__ __forceinline__ void image_block(const ImageLink &l, const ImageLink &next, bool has_next, int img, char *lds) {
    const QBlockArgs &a = l.a;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, lh = lane >> 5;
    const int co32 = l.co32;
    const uint4 *XL = reinterpret_cast<const uint4 *>(lds + a.o_xl);   // [Cin32*2][Ppad] units of 16 channels
    const uint4 *W1 = reinterpret_cast<const uint4 *>(lds + a.o_w1);   // [Cin32][Ce32][2][32]
    const uint4 *W2 = reinterpret_cast<const uint4 *>(lds + a.o_w2);   // [Ce32][co32][2][32]
    const uint32_t *WDW = reinterpret_cast<const uint32_t *>(lds + a.o_wdw);  // [Ce/4][9][4] dwords
    const int Ce = a.Ce32 * 32;
    const float *m1 = reinterpret_cast<const float *>(lds + a.o_tab);
    const int *c1 = reinterpret_cast<const int *>(m1 + Ce);
    const float *m2 = reinterpret_cast<const float *>(c1 + Ce);
    const int *c2 = reinterpret_cast<const int *>(m2 + Ce);
    const float *m3 = reinterpret_cast<const float *>(c2 + Ce);
    const int *c3 = reinterpret_cast<const int *>(m3 + co32 * 32);
    const QBlockPos *ptab = reinterpret_cast<const QBlockPos *>(lds + a.o_ptab), *qtab = reinterpret_cast<const QBlockPos *>(lds + a.o_qtab);
    int *R = reinterpret_cast<int *>(lds + l.o_r);
    const unsigned head = qb_act_head(lds + a.o_act);
    const RequantLut lut1 = qb_lut(lds + a.o_act, head, 0, a.zp1), lut2 = qb_lut(lds + a.o_act, head, 1, a.zp2);
    const unsigned xl_a = lds_address(lds + a.o_xl), e_a = lds_address(lds + a.o_e);  // expanded patch: [Ce32*2][Ppad] units
    const int n_ptiles = a.Ppad >> 5, nq_tiles = (a.Q + 31) >> 5;

    // ---- the next block's weights set out; the projection sums start from zero ----
    const bool ahead = has_next && !next.late;
    i32x4 w[kAhead];
    if (ahead) {
#pragma unroll
        for (int r = 0; r < kAhead; ++r) w[r] = *reinterpret_cast<const i32x4 *>(next.packed + min(r * kThreads + tid, next.a.packed_units - 1));
    }
    for (int i = tid; i < nq_tiles * co32 * 256; i += kThreads) reinterpret_cast<uint4 *>(R)[i] = uint4{0u, 0u, 0u, 0u};

    // ---- expansion ----
    const int b_units = a.Ce32 * n_ptiles;
    const float inv_np = 1.0f / float(n_ptiles);
    for (int u = wave; u < b_units; u += kWaves) {
        const int kb = small_div(u, n_ptiles, inv_np), ptile = u - kb * n_ptiles, kch = kb * 32 + lh * 4;
        i32x4 xb;
        qb_read128(xb, xl_a + unsigned(lh * a.Ppad + ptile * 32 + l32) * 16u, 0);
        const i32x4 wa0 = as_i32x4(W1[kb * 64 + lh * 32 + l32]);
        const bool padp = ptab[ptile * 32 + l32] & QB_POS_PAD;  // the depthwise convolution's padding: its zero point instead of an expansion
        i32x16 acc[1];
        float mv[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            acc[0][v] = c1[kch + (v >> 2) * 8 + (v & 3)];
            mv[v] = m1[kch + (v >> 2) * 8 + (v & 3)];
        }
        qb_ready(xb, 0);
        acc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wa0, xb, acc[0], 0, 0, 0);
        for (int chunk = 1; chunk < a.Cin32; ++chunk)
            acc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(as_i32x4(W1[(chunk * a.Ce32 + kb) * 64 + lh * 32 + l32]),
                                                           as_i32x4(XL[(2 * chunk + lh) * a.Ppad + ptile * 32 + l32]), acc[0], 0, 0, 0);
        const bool half = a.half_last && kb == a.Ce32 - 1;  // at most 16 real channels: the upper half is padding
        uint32_t d[1][4];
        if (half) qb_requant_lookup_n<2, 1>(acc, mv, lut1, d);
        else qb_requant_lookup_n<4, 1>(acc, mv, lut1, d);
        const auto s0 = __builtin_amdgcn_permlane32_swap(d[0][0], d[0][2], false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(d[0][1], d[0][3], false, false);
        i32x4 out;
        out[0] = padp ? int(a.pad_e4) : int(s0[0]); out[1] = padp ? int(a.pad_e4) : int(s0[1]);
        out[2] = padp ? int(a.pad_e4) : int(s1[0]); out[3] = padp ? int(a.pad_e4) : int(s1[1]);
        if (!half || !lh)
            *reinterpret_cast<lds_i32x4 *>(e_a + unsigned((2 * kb + lh) * a.Ppad + ptile * 32 + l32) * 16u) = out;
    }
    // the next block's weights to LDS
    if (ahead) {
        i32x4 *dst = reinterpret_cast<i32x4 *>(lds + next.a.o_w1);
#pragma unroll
        for (int r = 0; r < kAhead; ++r)
            if (r * kThreads + tid < next.a.packed_units) dst[r * kThreads + tid] = w[r];
        copy_weights(next, lds, tid, kAhead * kThreads);
    }
    lds_barrier();

    // ---- depthwise 3x3 + projection ----
    {
        const bool diag_mine = (l32 >> 4) == lh;  // the diagonal element of row l32 lies in this lane's half of the columns
        const int diag_q = (l32 >> 2) & 3;
        const uint32_t dm0 = diag_mine && diag_q == 0 ? 0xffffffffu : 0u, dm1 = diag_mine && diag_q == 1 ? 0xffffffffu : 0u,
                       dm2 = diag_mine && diag_q == 2 ? 0xffffffffu : 0u, dm3 = diag_mine && diag_q == 3 ? 0xffffffffu : 0u;
        const int d_units = nq_tiles * a.Ce32;
        const float inv_ce = 1.0f / float(a.Ce32);
        const unsigned row_b = unsigned(a.PW) * 16u;
        for (int u = wave; u < d_units; u += kWaves) {
            const int j = small_div(u, a.Ce32, inv_ce), ch = u - j * a.Ce32, kch = ch * 32 + lh * 4;
            const bool half = a.half_last && ch == a.Ce32 - 1;
            const unsigned r0 = e_a + unsigned((2 * ch + lh) * a.Ppad) * 16u + unsigned(qtab[j * 32 + l32]) * 16u,  // top-left tap
                           r1 = r0 + row_b, r2 = r1 + row_b;
            const uint32_t *wk = WDW + ((ch * 32 + l32) >> 2) * 36 + (l32 & 3);
            uint32_t wd[9];
#pragma unroll
            for (int t = 0; t < 9; ++t) wd[t] = wk[t * 4];
            i32x16 acc2;
            float mv[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                acc2[v] = c2[kch + (v >> 2) * 8 + (v & 3)];
                mv[v] = m2[kch + (v >> 2) * 8 + (v & 3)];
            }
            i32x4 tap[9];
            qb_read128(tap[0], r0, 0); qb_read128(tap[1], r0, 16); qb_read128(tap[2], r0, 32);
            qb_read128(tap[3], r1, 0); qb_read128(tap[4], r1, 16); qb_read128(tap[5], r1, 32);
            qb_read128(tap[6], r2, 0); qb_read128(tap[7], r2, 16); qb_read128(tap[8], r2, 32);
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                i32x4 wa;
                wa[0] = int(wd[t] & dm0); wa[1] = int(wd[t] & dm1); wa[2] = int(wd[t] & dm2); wa[3] = int(wd[t] & dm3);
                qb_ready(tap[t], 8 - t);
                acc2 = __builtin_amdgcn_mfma_i32_32x32x32_i8(wa, tap[t], acc2, 0, 0, 0);
            }
            uint32_t d[4];
            if (half) qb_requant_lookup<2>(acc2, mv, lut2, d);
            else qb_requant_lookup<4>(acc2, mv, lut2, d);
            const auto s0 = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
            i32x4 db;
            db[0] = int(s0[0]); db[1] = int(s0[1]); db[2] = int(s1[0]); db[3] = int(s1[1]);
            for (int kb3 = 0; kb3 < co32; ++kb3) {
                i32x16 acc3;
#pragma unroll
                for (int v = 0; v < 16; ++v) acc3[v] = 0;
                acc3 = __builtin_amdgcn_mfma_i32_32x32x32_i8(as_i32x4(W2[(ch * co32 + kb3) * 64 + lh * 32 + l32]), db, acc3, 0, 0, 0);
                int *sum = R + (j * co32 + kb3) * 1024 + lane;
#pragma unroll
                for (int v = 0; v < 16; ++v) atomicAdd(sum + v * 64, acc3[v]);
            }
        }
    }
    lds_barrier();

    // ---- requantisation (and the residual add): to the next block's patch and to memory ----
    {
        const float inv_ow = 1.0f / float(a.OW);
        const int units = nq_tiles * co32 * 4;
        const float inv_co = 1.0f / float(co32);
        for (int u = wave; u < units; u += kWaves) {
            const int gq = u & 3, j = small_div(u >> 2, co32, inv_co), kb3 = (u >> 2) - j * co32, cbq = kb3 * 2 + (gq >> 1);
            if (cbq >= a.CBo) continue;
            const int q = j * 32 + l32;
            if (q >= a.Q) continue;
            const int qr = small_div(q, a.OW, inv_ow), qc = q - qr * a.OW;
            const unsigned byte = unsigned(gq & 1) * 8u + unsigned(lh) * 4u;
            uint32_t o = 0;
            // eight output channels past the last real one are padding of the blocked layout: zeros
            const bool real = kb3 * 32 + gq * 8 < a.Co;
            if (real) {
                uint32_t xr = 0;
                if (a.has_res)  // (stride 1: the output position's own place in the patch)
                    xr = *reinterpret_cast<const uint32_t *>(lds + a.o_xl + (unsigned(cbq * a.Ppad + (qr + 1) * a.PW + qc + 1) * 16u + byte));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int k = kb3 * 32 + gq * 8 + lh * 4 + e;
                    const int sum = R[((j * co32 + kb3) * 16 + gq * 4 + e) * 64 + lane] + c3[k];
                    const float r = __builtin_rintf(float(sum) * m3[k]) + a.zp3f;
                    if (a.has_res) {
                        const float va = __builtin_amdgcn_fmed3f(r, 0.0f, 255.0f);
                        const float fa = (va - float(a.ra_zp)) * a.ra_scale;
                        const float fb = (float(((xr ^ 0x80808080u) >> (8 * e)) & 0xffu) - float(a.rb_zp)) * a.rb_scale;
                        const float qv = div_by(fa + fb, a.ry_scale, a.ry_rcp, a.fast_div);
                        o = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_rintf(qv) + float(a.ry_zp), e, o);
                    } else {
                        o = __builtin_amdgcn_cvt_pk_u8_f32(r, e, o);
                    }
                }
                o ^= 0x80808080u;
            }
            if (has_next)
                *reinterpret_cast<uint32_t *>(lds + next.a.o_xl + (unsigned(cbq * next.a.Ppad + (qr + 1) * next.a.PW + qc + 1) * 16u + byte)) = o;
            const unsigned at = ((unsigned(img) * unsigned(a.CBo) + unsigned(cbq)) * unsigned(a.OH) + unsigned(qr)) * unsigned(a.OW) + unsigned(qc);
            *reinterpret_cast<uint32_t *>(l.y + (at * 16u + byte)) = o;  // (< 2^31: checked on the host)
        }
    }
    lds_barrier();
}

__global__ void __launch_bounds__(kThreads, 4) qblock_image_chain_kernel(ImageChain c) {
    extern __shared__ __attribute__((aligned(256))) char lds[];
    const int tid = threadIdx.x, img = blockIdx.x;
    {
        // every block's arguments into the scalar cache now: each line would cost a stage a trip to memory (1.7 us of setup a block)
        unsigned touched = 0;
        for (int b = 0; b < c.n; ++b) {
            const unsigned *line = reinterpret_cast<const unsigned *>(&c.link[b]);
#pragma unroll
            for (int i = 0; i < int(sizeof(ImageLink) / 4); i += 15) touched += line[i];
        }
        asm volatile("" ::"s"(touched));
    }
    {
        // the first block: weights, tables and its input patch (positions outside the image are left as they are: the expansion
        // replaces what they yield)
        const ImageLink &l = c.link[0];
        const QBlockArgs &a = l.a;
        const float inv_p = 1.0f / float(a.P), inv_pw = 1.0f / float(a.PW);
        i32x4 *XL = reinterpret_cast<i32x4 *>(lds + a.o_xl);
        const int a_units = a.CBin * a.P;
        for (int u0 = tid; u0 < a_units; u0 += 4 * kThreads) {
            i32x4 v[4];
            int dst[4];
            bool ok[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int u = min(u0 + r * kThreads, a_units - 1);
                const int cb = small_div(u, a.P, inv_p), p = u - cb * a.P, ph = small_div(p, a.PW, inv_pw), pw = p - ph * a.PW;
                const int ih = ph - 1, iw = pw - 1;
                dst[r] = cb * a.Ppad + p;
                ok[r] = u0 + r * kThreads < a_units && ih >= 0 && ih < a.H && iw >= 0 && iw < a.W;
                const uint4 *src = ok[r] ? c.x + ((int64_t(img) * a.CBin + cb) * a.H + ih) * int64_t(a.W) + iw : c.x;
                v[r] = *reinterpret_cast<const i32x4 *>(src);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (ok[r]) XL[dst[r]] = v[r];
        }
        copy_weights(l, lds, tid, 0);
    }
    lds_barrier();
    for (int b = 0; b < c.n; ++b) {
        const ImageLink &l = c.link[b];
        const bool has_next = b + 1 < c.n;
        const ImageLink &next = c.link[has_next ? b + 1 : b];
        image_block(l, next, has_next, img, lds);
        if (has_next && next.late) {
            copy_weights(next, lds, tid, 0);
            lds_barrier();
        }
    }
}

size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

// LDS of a chain.  What a block keeps while it runs -- input patch, weights and tables -- is filled while the block before it runs, so
// neighbours lie at opposite ends, with the running block's expanded patch and projection sums between them.  Where that does
// not fit, the next block's weights and tables (the inner part of its end) come late.  Returns the bytes, 0: no room.
size_t plan_lds(ImageChain &c) {
    struct Need { size_t xl, w, e, r; };
    auto need_of = [](const ImageLink &l) {
        const QBlockArgs &a = l.a;
        Need n;
        n.xl = align256(size_t(a.Cin32) * 2 * a.Ppad * 16);
        n.w = size_t(a.packed_units) * 16;
        n.e = align256(size_t(a.Ce32) * 2 * a.Ppad * 16);
        n.r = size_t((a.Q + 31) / 32) * l.co32 * 4096;
        return n;
    };
    size_t total = 0;
    for (int b = 0; b < c.n; ++b) {
        const Need n = need_of(c.link[b]);
        size_t bytes = n.xl + n.w + n.e + n.r;
        if (b + 1 < c.n) {
            const Need m = need_of(c.link[b + 1]);
            c.link[b + 1].late = bytes + m.xl + m.w > kLdsMax;
            bytes += m.xl + (c.link[b + 1].late ? 0 : m.w);
        }
        if (bytes > kLdsMax) return 0;
        total = std::max(total, bytes);
    }
    c.link[0].late = 0;
    for (int b = 0; b < c.n; ++b) {
        ImageLink &l = c.link[b];
        QBlockArgs &a = l.a;
        const Need n = need_of(l);
        const bool low = b % 2 == 0;
        const size_t xl = low ? 0 : total - n.xl, w = low ? n.xl : xl - n.w, e = low ? w + n.w : w - n.e, r = low ? e + n.e : e - n.r;
        const int move = int(w) - a.o_w1;  // (what lies behind the weights keeps its distance from them)
        a.o_xl = int(xl); a.o_e = int(e); l.o_r = int(r);
        a.o_w1 += move; a.o_w2 += move; a.o_wdw += move; a.o_tab += move; a.o_act += move; a.o_ptab += move; a.o_qtab += move;
    }
    return total;
}

}  // namespace

// Up to one image a CU always: 53 chains of four blocks on maps of 3x3 to 14x14, 8 to 56 channels, at 256 images 1.24 to 1.94 times as fast.
// With a second round of images where blocks are wide and their maps small, so that few images fill a tile's matrix instructions and the
// weights weigh: at 512 images 144 expanded channels and more on maps of up to 9x9 1.01 to 1.48 times as fast, 192 on 10x10 69.6 us against
// 63.8 as tiles, 64 on 6x6 35.1 against 30.3; 96 on 5x5 and 6x6, where two images leave a tile's waves uneven work, 38.2 against 42.4, on
// 7x7 39.1 against 37.3.  MobileNetV2-0.35's last 14 blocks, which are three launches as tiles: 256 images 78 us (149), 512 148 (163).
bool zant_qblock_images_better(zant_ctx *ctx, int n, const zant_qblock_call *calls) {
    if (calls[0].xdim[0] <= ctx->num_cus) return true;
    for (int b = 0; b < n; ++b) {
        const int64_t map = calls[b].xdim[2] * calls[b].xdim[3], expanded = calls[b].expand->K;
        if (map > 81 || expanded < (map >= 25 && map <= 36 ? 96 : 144)) return false;
    }
    return true;
}

int zant_qblock_image_chain(zant_ctx *ctx, int n, const zant_qblock_call *calls, bool query_only) {
    // Up to two images a CU; past that tiles of several images were the faster (MobileNetV2-0.35's last 14 blocks at 700 217 us against 192).
    if (n < 2 || n > kMaxBlocks || !calls[0].xdim || calls[0].xdim[0] > 2 * int64_t(ctx->num_cus)) return 1;
    ImageChain c;
    std::memset(&c, 0, sizeof(c));
    c.n = n;
    c.x = reinterpret_cast<const uint4 *>(calls[0].x);
    for (int b = 0; b < n; ++b) {
        const zant_qblock_call &k = calls[b];
        if (!query_only && (!k.x || !k.y)) return ZANT_NullPointer;
        if (!query_only && b > 0 && k.x != calls[b - 1].y) return 1;
        QBlockPrep prep;
        const int rc = zant_qblock_prepare(ctx, k.xdim, k.expand, k.dw, k.dw_stride, k.project, k.residual, k.add_scale, k.add_zp, k.ydim,
                                           query_only, k.slot, 1, &prep);
        if (rc) return rc;
        if (prep.a.n_row_tiles != 1 || prep.a.NB != 1 || k.xdim[0] != calls[0].xdim[0]) return 1;
        ImageLink &l = c.link[b];
        l.packed = prep.packed;
        l.y = k.y;
        l.a = prep.a;
        l.co32 = prep.CO32;
    }
    const size_t lds = plan_lds(c);
    if (!lds) return 1;
    if (query_only) return ZANT_OK;
    if (!zant_raise_lds_limit(ctx, reinterpret_cast<const void *>(&qblock_image_chain_kernel), int(kLdsMax))) return ZANT_HipError;
    KernelTimer kt(ctx);
    ZANT_KERNEL_NAME(ctx, "qblock_image_chain_kernel x %d", n);
    hipLaunchKernelGGL(qblock_image_chain_kernel, dim3(unsigned(calls[0].xdim[0])), dim3(kThreads), lds, ctx->stream, c);
    ZANT_LAUNCH_CHECK(ctx);
    return ZANT_OK;
}
