/* Host-side check of the launch that merges key splits (flash-attn-rtx5060_amd/csrc/fa_sched.h): its grid covers every row
 * and stays below 2^32 threads for as many rows as a launch with one thread per four elements does. */
#include <stdio.h>
#include "fa_sched.h"

int main(void)
{
    int fails = 0, shared = 0;
    for (int D = 64; D <= 128; D += 64)
        for (int n = 2; n <= 64; n += n < 12 ? 1 : 13)
            for (int bit = 0; bit <= 28; ++bit)
                for (int off = -1; off <= 1; ++off) {
                    const long long rows = (1LL << bit) + off;
                    const long long plain = (rows + fa_combine_rows(D, 1) - 1) / fa_combine_rows(D, 1) * 256;
                    if (rows < 1 || plain >= 1LL << 32) continue;
                    const int groups = fa_combine_groups(rows, D, n), per = fa_combine_rows(D, groups);
                    const long long blocks = (rows + per - 1) / per;
                    const int ok = (groups == 1 || (groups == 8 && n > 8)) && per >= 1 && blocks * per >= rows && blocks * 256 < 1LL << 32;
                    if (!ok && fails++ < 10) printf("D %d splits %d rows %lld: %d groups, %lld blocks\n", D, n, rows, groups, blocks);
                    shared += groups == 8;
                    if (n > 8 && rows <= 1 << 20 && groups != 8 && fails++ < 10) printf("D %d splits %d rows %lld: not shared\n", D, n, rows);
                }
    return fails != 0 || shared == 0;
}
