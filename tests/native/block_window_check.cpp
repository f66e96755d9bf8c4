// Host-only check of the MFMA decode's block-table window (part_range, wave_range,
// window_covers and window_lane in attention_body.h), built and run by
// tests/test_block_window.py: every entry a wave uses belongs to a block that
// holds keys of its row, whether its window was requested before the row's length
// was known or by the wave itself, and lies inside the window.
#include <cstdio>

#include "../../pagedattentionmetal_amd/csrc/kernels/attention_body.h"

using namespace pam;

// the lanes the kernel reads for tile t of a row of nlb blocks (load_tile)
static bool tile_ok(int t, int bs, int bsh, int window_blk, int nlb, bool early) {
    for (int row = 0; row < 16; row += bs >= 16 ? 16 : 1) {
        const int j = t * 16 + row;
        const int lane = bs >= 16 ? (j >> bsh) - window_blk : window_lane(j, bsh, window_blk, nlb);
        if (lane < 0 || lane > 63) return false;
        int blk = window_blk + lane;
        if (!early && blk >= nlb) blk = nlb - 1;  // refresh_window loads no entry past the row
        if (blk >= nlb) return false;
    }
    return true;
}

int main() {
    long used = 0;
    for (int bs : {8, 16, 32, 128})
        for (int L = 1; L <= 1200; L += L < 420 ? 1 : 13)
            for (int tpp : {1, 2, 3, 5, 8, 16, 17, 32, 64, 128}) {
                const int bsh = __builtin_ctz((unsigned)bs), nlb = (L + bs - 1) / bs;
                const RowCtx c{nullptr, 0, L, 0};
                const int parts = part_range(c, 0, tpp * 16).nparts;
                for (int part = 0; part < parts; part++) {
                    const PartRange wg = part_range(c, part, tpp * 16);
                    const int early_blk = (int)((long)part * tpp * 16 / bs);
                    if (early_blk >= nlb) return printf("window starts past the row: L %d block %d part %d\n", L, bs, part), 1;
                    for (int w = 0; w < kMfmaWaves; w++) {
                        const PartRange pr = wave_range(wg, w, kMfmaWaves);
                        for (int t = pr.t_begin; t < pr.t_end; t++) {
                            const bool early = window_covers(early_blk, pr.t_end, bsh);
                            // a wave's own window may be refreshed at any tile up to 16 before
                            const int own = ((t - t % 16 < pr.t_begin ? pr.t_begin : t - t % 16) * 16) >> bsh;
                            if (!tile_ok(t, bs, bsh, early ? early_blk : own, nlb, early)) {
                                printf("L %d block %d partition %d x %d tiles, wave %d, tile %d\n", L, bs, part, tpp, w, t);
                                return 1;
                            }
                            used++;
                        }
                    }
                }
            }
    printf("ok %ld tiles\n", used);
    return 0;
}
