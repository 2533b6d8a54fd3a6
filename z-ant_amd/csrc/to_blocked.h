// NCHW u8 -> [N][CB][H][W][16] signed (value - 128), as a piece of a kernel: alone (to_blocked_kernel) or beside the packing of
// weights, whose launch it then shares.
// Against the kernel that took planes of odd lengths byte by byte, and the two launches: 256x120x45x45 to 64 3x3 filters, kernels,
// 136 -> 102 us, 43x15x47x3 17.4 -> 9.4 (the layout 9 -> 3, its launch 3); whole calls on small tensors 21 - 27 -> 17 - 24 us.  Planes of
// whole dwords take what they took (256x96x48x48 17 us); their calls lose the launch.
#pragma once
#include "quant_layout.h"

struct BlockedJob {
    const uint8_t *x;
    uint4 *xb;
    unsigned quads;          // quads of positions, counted through the whole tensor: ceil(HW / 4) for every (image, channel block)
    unsigned CB, HW, HW4;    // HW4 = ceil(HW / 4)
    int C;
    FastDiv d_hw4, d_cb;
    unsigned blocks() const { return (quads + 63) / 64; }
};
// False for tensors too large for 32-bit counting (zant_to_blocked takes those too).
bool zant_blocked_job(const uint8_t *x, int64_t N, int64_t C, int64_t HW, void *xb, BlockedJob *j);

// A workgroup of 256 turns 64 quads of positions x 16 channels; channels beyond C are 0 (their weights are 0 too).
// Wavefront g loads the dwords of channels 4g .. 4g+3, a quad per lane (256 contiguous bytes per load; planes start and end
// anywhere: a plane's last quad is read from four bytes before its end and shifted), transposes its 4 x 4 bytes with byte
// permutes (dword b: position b, channels 4g .. 4g+3) and writes the four dwords to LDS row g; then thread u gathers unit u's four
// dwords (one per row, consecutive lanes on consecutive banks) and stores its 16 bytes: a workgroup's stores are one run of 4 KB.
// (One tile per workgroup: with two, all eight loads of a thread in flight together, the kernel was slower.)
__device__ __forceinline__ void blocked_tile(const BlockedJob &j, unsigned block) {
    __shared__ __attribute__((aligned(16))) uint32_t stage[4][256];
    typedef uint32_t u32_any __attribute__((aligned(1)));
    const unsigned g = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const unsigned qi = block * 64u + lane;
    uint32_t r[4] = {0u, 0u, 0u, 0u};  // r[c] = 4 consecutive positions of channel c0 + c
    if (qi < j.quads) {
        const unsigned row = fastdiv(qi, j.d_hw4), q = qi - row * j.HW4;  // row = image * CB + channel block
        const unsigned n = fastdiv(row, j.d_cb), cb = row - n * j.CB;
        const int c0 = int(cb) * 16 + int(g) * 4;
        const uint8_t *img = j.x + int64_t(n) * j.C * j.HW;
        uint32_t v[4];
        if (j.HW >= 4) {
            // The four loads leave together: a channel past C reads channel C - 1 instead of branching around its load
            // (with a branch per load the compiler waited for each one before the next), and is zeroed afterwards.
            const unsigned at = min(4 * q, j.HW - 4), shift = 8 * (4 * q - at);
#pragma unroll
            for (int c = 0; c < 4; ++c)
                v[c] = __builtin_nontemporal_load(reinterpret_cast<const u32_any *>(img + int64_t(min(c0 + c, j.C - 1)) * j.HW + at));
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] >>= shift;
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint8_t *p = img + int64_t(min(c0 + c, j.C - 1)) * j.HW;
                v[c] = uint32_t(p[0]) | uint32_t(p[min(1u, j.HW - 1)]) << 8 | uint32_t(p[j.HW - 1]) << 16;
            }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) r[c] = c0 + c < j.C ? v[c] ^ 0x80808080u : 0u;
    }
    const uint32_t lo01 = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u);  // r0.0 r1.0 r0.1 r1.1
    const uint32_t hi01 = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);  // r0.2 r1.2 r0.3 r1.3
    const uint32_t lo23 = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u);
    const uint32_t hi23 = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
    uint4 o;  // dword b: position b, channels c0 .. c0+3
    o.x = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
    o.y = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
    o.z = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
    o.w = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
    *reinterpret_cast<uint4 *>(&stage[g][lane * 4]) = o;
    __syncthreads();
    const unsigned u = threadIdx.x, qu = block * 64u + (u >> 2);
    if (qu < j.quads) {
        const unsigned row = fastdiv(qu, j.d_hw4), pos = (qu - row * j.HW4) * 4u + (u & 3u);
        if (pos < j.HW) j.xb[int64_t(row) * j.HW + pos] = make_uint4(stage[0][u], stage[1][u], stage[2][u], stage[3][u]);
    }
}
