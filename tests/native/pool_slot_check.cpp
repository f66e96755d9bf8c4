// Host-only check that the row-block kernels address a pool's token slots in 64 bits
// (pool_slot and KeySlots in rows_body.h): block tables of pools
// with more than 2^31 slots.  Built and run by tests/test_pool_slots.py (no kernel
// launches).
#include <cstdio>
#include <type_traits>

#include "../../pagedattentionmetal_amd/csrc/kernels/rows_body.h"

using namespace pam;

int main() {
    for (int bs : {1, 8, 16, 24, 256})
        for (int64_t first : {(int64_t)5, ((int64_t)1 << 31) - 2, ((int64_t)1 << 31) + 3, (int64_t)0xFFFFFFF0, (int64_t)3 << 33}) {
            const int64_t b0 = first / bs;
            if (b0 + 4 > 0x7FFFFFFF) continue;  // block ids are 32 bits
            const int32_t bt[4] = {(int32_t)b0, (int32_t)b0 + 3, (int32_t)b0 + 1, (int32_t)b0 + 2};
            BackwardParams p{};
            p.block_table = bt;
            p.block_size = bs;
            p.window_start = bs / 2;
            p.seq_len = 4 * bs;
            const KeySlots keys(p);
            for (int j = -1; j <= 4 * bs; j++) {
                const bool inside = j >= p.window_start && j < p.seq_len;
                const __int128 want = inside ? (__int128)bt[j / bs] * bs + j % bs : -1;
                if ((__int128)keys.at(j) != want) return printf("KeySlots: block size %d, block %d, key %d\n", bs, bt[0], j), 1;
                if (inside && (__int128)pool_slot(bt[j / bs], bs, j % bs) != want)
                    return printf("pool_slot: block size %d, block %d, key %d\n", bs, bt[0], j), 1;
            }
        }
    typedef RowTiles<float, float, 2, 2> Tiles;
    // the loads take the slot as it is
    static_assert(std::is_same<decltype(&Tiles::issue_k), void (Tiles::*)(const AttnParams &, int64_t, int)>::value, "K");
    static_assert(std::is_same<decltype(&Tiles::issue_v), void (Tiles::*)(const AttnParams &, int64_t, int)>::value, "V");
    printf("ok\n");
    return 0;
}
