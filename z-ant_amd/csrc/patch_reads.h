// LDS bank conflicts of the operand reads of a tile plan (conv_tile.h), as a function of the patch row pitch.  Plain C++, so that a
// test can compare it with the definition on the host.
#pragma once
#include <cstdint>

// A lane reads the 16-byte unit of its position slot; the LDS serves 16 such units per cycle when they lie in 16 different
// groups of four banks (unit index mod 16), and takes one more cycle for every further distinct unit of a group.  Consecutive
// lanes take consecutive positions of the (pooled) output, so the units a pass of 16 lanes touches are spaced by the stride, by
// two columns with a fused pool, by a patch row at a row change and by a patch image at an image change: on small maps a pitch of
// 8 or 16 units puts whole columns of the tile into the same banks.
//
// What a pass touches is a few runs of columns, a patch row each.  The runs do not depend on the pitch, so they are found once, as masks
// of the banks they take (a run that meets a bank again is cut there); a pitch rotates each mask by its row, and the passes' cycles
// are the largest counts of the masks' bits.  A plan's search for its pitch takes 1 to 4 us of the host this way, 5 to 21 lane by lane.
class PatchReads {
public:
    // WM * MT position tiles of 32 slots; NB images x TH rows x OW columns of positions (windows of 2x2 of them, TH / 2 x POW, with
    // `pool`, four position tiles being the members of 32 windows), PH patch rows an image, strides sh, sw.
    PatchReads(int WM, int MT, int NB, int TH, int PH, int OW, int sh, int sw, bool pool, int POW) {
        const int cols = pool ? POW : OW, rows = pool ? TH / 2 : TH, step = (pool ? 2 : 1) * sw, members = pool ? 4 : 1;
        int period = 16;  // columns of a run before its banks come round again
        for (int s = step; period > 1 && !(s & 1); s >>= 1) period >>= 1;
        const int tiles = WM * (pool ? MT / 4 : MT);
        for (int m = 0; m < members; ++m) {
            const int dr = pool ? (m >> 1) * sh : 0, dc = pool ? (m & 1) * sw : 0;
            int img = 0, r = 0, c = 0;
            for (int pass = 0; pass < tiles * 2; ++pass) {
                if (passes_ >= kPasses) return;
                bool origin = false, absent = false;  // is unit 0 read by a position; does a lane without one read it
                for (int left = 16; left > 0;) {
                    if (img >= NB || r >= rows) { absent = true; break; }  // (so are all lanes behind)
                    const int taken = left < cols - c ? left : cols - c;
                    int len = taken;
                    left -= taken;
                    const int row = img * PH + (pool ? 2 : 1) * r * sh + dr;
                    origin |= row == 0 && c * step + dc == 0;
                    for (int at = c * step + dc; len > 0; len -= period, at += period * step) {
                        const int n = len < period ? len : period;
                        unsigned mask = 0;
                        if (step == 1) mask = (1u << n) - 1u;
                        else for (int i = 0; i < n; ++i) mask |= 1u << ((i * step) & 15);
                        add(row, rotate(mask, at));
                    }
                    c += taken;
                    if (c == cols) { c = 0; if (++r == rows) { r = 0; ++img; } }
                }
                if (absent && !origin) add(0, 1u);
                end_[passes_++] = n_;
            }
        }
    }
    // The average number of cycles per 16-lane pass (1 = conflict-free) for patch rows of `pw` units.
    double cycles(int pw) const {
        long total = 0;
        for (int p = 0, k = 0; p < passes_; ++p) {
            unsigned b0 = 0, b1 = 0, b2 = 0, b3 = 0, b4 = 0;  // bit b of these five: the count of bank b, in binary
            for (; k < end_[p]; ++k) {
                unsigned m = rotate(mask_[k], row_[k] * pw), t = b0 & m;
                b0 ^= m; m = t; t = b1 & m;
                b1 ^= m; m = t; t = b2 & m;
                b2 ^= m; m = t; t = b3 & m;
                b3 ^= m; b4 |= t;
            }
            unsigned most = 0xffffu;
            int worst = 0;
            const unsigned bits[5] = {b0, b1, b2, b3, b4};
            for (int i = 4; i >= 0; --i)
                if (most & bits[i]) { most &= bits[i]; worst |= 1 << i; }
            total += worst > 1 ? worst : 1;
        }
        return double(total) / double(passes_);
    }

private:
    static constexpr int kPasses = 64, kRuns = kPasses * 17;
    static unsigned rotate(unsigned mask, int by) {
        by &= 15;
        return (mask << by | mask >> (16 - by)) & 0xffffu;
    }
    void add(int row, unsigned mask) { row_[n_] = row; mask_[n_] = uint16_t(mask); ++n_; }
    int n_ = 0, passes_ = 0;
    int row_[kRuns], end_[kPasses];
    uint16_t mask_[kRuns];
};
