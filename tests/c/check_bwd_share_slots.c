/* Host-side check that no launch of the key-owning backward kernel uses more shares than the caller's buffer of parts
 * was sized for (flash-attn-rtx5060_amd/csrc/fa_bwd_layout.h), whatever number of compute units the device reports,
 * and that a whole MI355X cuts what the size was made for. */
#include <stdio.h>
#include "fa_bwd_layout.h"

int main(void)
{
    static const int lens[] = {128, 512, 1000, 2048, 5001}, units[] = {8, 32, 64, 128, 256, 304}, masks[][3] = {{0, -1, -1}, {1, -1, -1}, {1, 300, -1}};
    static const int chunks[] = {1, 8, 24, 264, 1000}, rests[] = {0, 1, 2, 7, 8};
    int fails = 0, cut = 0, refused = 0;
    for (int D = 64; D <= 128; D += 64)
    for (unsigned l = 0; l < sizeof(lens) / sizeof(*lens); ++l)
        for (unsigned m = 0; m < sizeof(masks) / sizeof(*masks); ++m)
            for (int G = 1; G <= 8; G += 7)
                for (unsigned c = 0; c < sizeof(chunks) / sizeof(*chunks); ++c)
                    for (unsigned r = 0; r < sizeof(rests) / sizeof(*rests); ++r) {
                        const int S = lens[l], chunk = chunks[c], rest = rests[r];
                        int L, R, per_head = 0;
                        if (rest >= chunk) continue;
                        fa_mask_bounds(2 * S, masks[m][0], masks[m][1], masks[m][2], &L, &R);
                        for (int kb = 0; kb < (S + 255) / 256; ++kb) per_head += G * fa_bwd_walk_tiles(S, S, R, L, kb);
                        const int slots = fa_bwd_share_slots(D, chunk, rest, G, S, R, L, per_head);
                        for (unsigned u = 0; u < sizeof(units) / sizeof(*units); ++u)
                            for (int last = 0; last < 2; ++last) {
                                const int heads = last ? rest : chunk;
                                if (heads == 0) continue;
                                const int want = fa_bwd_shares(D, heads, G, S, R, L, per_head, units[u]);
                                const int got = fa_bwd_launch_shares(D, heads, G, S, R, L, per_head, units[u], slots);
                                if (got > slots || (got != 0 && got != want) || (units[u] == 256 && got != want)) {
                                    if (fails++ < 10) printf("D %d S %d G %d chunk %d rest %d units %d: %d shares of %d, %d slots\n", D, S, G, chunk, rest, units[u], got, want, slots);
                                }
                                cut += got != 0;
                                refused += want > slots;
                            }
                    }
    if (cut == 0 || refused == 0) { printf("nothing cut (%d) or nothing refused (%d)\n", cut, refused); return 1; }
    return fails != 0;
}
