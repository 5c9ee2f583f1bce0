// walk_sight against the masks key by key, on the host: a walk position is reported whole for a wave's 32 queries exactly
// where every one of them sees every key of its tile. Prints the number of waves compared; 1 on the first difference.
#include <stdio.h>
#include <stdlib.h>

#include "fv_internal.h"

static long waves = 0;
static int check(const fv::FlashParams& p, int bm) {
    const int nkt = (p.sk + 63) / 64;
    for (int q0 = 0; q0 < p.sq; q0 += bm) {
        const int qlen = p.sq - q0 < bm ? p.sq - q0 : bm;
        const fv::TileWalk w = fv::mask_tile_walk(p, q0, qlen, nkt);
        for (int first = q0; first + 32 <= q0 + qlen; first += 32, waves++) {
            const fv::WalkSight s = fv::walk_sight(p, w, first);
            // (the last tile of a walk is asked key by key, its keys may end)
            for (int e = 0; e + 1 < w.ne; e++) {
                const int t = e < w.n0 ? e : e < w.n0 + w.n1 ? w.a1 + (e - w.n0) : w.a2 + (e - w.n0 - w.n1);
                bool whole = true;
                for (int q = first; q < first + 32 && whole; q++) {
                    const fv::LaneMask m = fv::lane_mask(p, q);
                    for (int x = 64 * t; x < 64 * t + 64 && whole; x++) whole = x < m.a_hi || x >= m.c_lo || (x >= m.w_lo && x < m.w_hi);
                }
                // (a pair of positions may be called cut where both are whole, in different ranges; never the other way round)
                if (s.all(e, e) != whole || (s.all(e, e + 1) && !whole) || (e > 0 && s.all(e - 1, e) && !whole)) {
                    printf("mode %d ft %d win %d sink %d vs %d frames %d chunk %d radius %d sq %d sk %d: queries %d, position %d, tile %d: %d\n",
                           p.mask_mode, p.ft, p.win, p.sink, p.vs, p.frames, p.chunk, p.radius, p.sq, p.sk, first, e, t, (int)whole);
                    return 1;
                }
            }
        }
    }
    return 0;
}

int main() {
    const int fts[] = {1, 7, 32, 50, 64, 100, 129, 390};
    for (int bm : {128, 256})
        for (int ft : fts) {
            fv::FlashParams p{};
            p.ft = ft;
            p.mask_mode = 1;
            for (p.win = 0; p.win < 5; p.win++)
                for (p.sink = 0; p.sink < 4; p.sink++)
                    for (int s : {300, 5 * ft + 333}) {
                        p.sq = p.sk = s;
                        if (check(p, bm)) return 1;
                        p.sk = 2 * s + 17;
                        if (check(p, bm)) return 1;
                    }
            p.mask_mode = 2;
            p.win = p.sink = 0;
            for (p.vs = 0; p.vs < 200; p.vs += 67)
                for (p.frames = 3; p.frames < 14; p.frames += 5)
                    for (p.chunk = 0; p.chunk < 4; p.chunk++)
                        for (p.radius = 0; p.radius <= p.frames; p.radius += 1 + p.radius) {
                            p.ve = p.vs + p.frames * ft;
                            p.sq = p.sk = p.ve + 37;
                            if (check(p, bm)) return 1;
                        }
        }
    printf("%ld\n", waves);
    return 0;
}
