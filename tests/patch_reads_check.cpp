// PatchReads (patch_reads.h) against the definition, lane by lane, over random tile shapes: prints "ok" when all agree.
#include <cstdio>
#include <cstdlib>

#include "../z-ant_amd/csrc/patch_reads.h"

struct Tile { int WM, MT, NB, TH, PH, OW, sh, sw, POW; };

// cycles of a 16-lane pass, averaged: the most distinct units that share a group of four banks
static double by_lane(const Tile &t, bool pool, int pw) {
    const int per_img = t.TH * t.OW, per_img_p = pool ? (t.TH / 2) * t.POW : 1;
    long total = 0, passes = 0;
    for (int wm = 0; wm < t.WM; ++wm)
        for (int i = 0; i < t.MT; ++i)
            for (int half = 0; half < 2; ++half) {
                int unit[16], n_unit = 0, load[16] = {0}, worst = 1;
                for (int l = half * 16; l < half * 16 + 16; ++l) {
                    int img, r, c;
                    if (pool) {
                        const int p = (wm * (t.MT / 4) + i / 4) * 32 + l, rem = p % per_img_p;
                        img = p / per_img_p;
                        r = 2 * (rem / t.POW) + ((i & 3) >> 1);
                        c = 2 * (rem % t.POW) + (i & 1);
                    } else {
                        const int q = (wm * t.MT + i) * 32 + l, rem = q % per_img;
                        img = q / per_img;
                        r = rem / t.OW;
                        c = rem % t.OW;
                    }
                    const int u = img < t.NB && r < t.TH ? (img * t.PH + r * t.sh) * pw + c * t.sw : 0;
                    bool seen = false;
                    for (int k = 0; k < n_unit; ++k) seen |= unit[k] == u;
                    if (!seen) { unit[n_unit++] = u; ++load[u & 15]; }
                }
                for (int b = 0; b < 16; ++b) worst = load[b] > worst ? load[b] : worst;
                total += worst;
                ++passes;
            }
    return double(total) / double(passes);
}

int main() {
    srand(1);
    for (int n = 0; n < 20000; ++n) {
        const bool pool = rand() % 3 == 0;
        Tile t;
        t.WM = rand() % 2 ? 4 : 2;
        t.MT = pool ? 4 : 1 + rand() % 6;
        t.OW = (pool ? 2 : 1) + rand() % (rand() % 2 ? 40 : 200);
        t.sh = pool ? 1 : 1 + rand() % 4;
        t.sw = pool ? 1 : 1 + rand() % 17;
        t.NB = 1 + rand() % (rand() % 2 ? 3 : 40);
        t.TH = pool ? 2 * (1 + rand() % 8) : 1 + rand() % 16;
        t.POW = pool ? t.OW / 2 : 0;
        t.PH = (t.TH - 1) * t.sh + 1 + rand() % 5;
        const PatchReads reads(t.WM, t.MT, t.NB, t.TH, t.PH, t.OW, t.sh, t.sw, pool, t.POW);
        const int pw0 = (t.OW - 1) * t.sw + 1 + rand() % 4;
        for (int pw = pw0; pw < pw0 + 4; ++pw)
            if (by_lane(t, pool, pw) != reads.cycles(pw)) {
                printf("differs: WM %d MT %d NB %d TH %d PH %d OW %d strides %d %d pool %d pitch %d\n", t.WM, t.MT, t.NB, t.TH, t.PH, t.OW,
                       t.sh, t.sw, int(pool), pw);
                return 1;
            }
    }
    printf("ok\n");
    return 0;
}
