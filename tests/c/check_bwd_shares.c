/* Host-side check of how the backward pass cuts the key blocks' walks into equal shares
 * (flash-attn-rtx5060_amd/csrc/fa_bwd_layout.h).  Follows what the key-owning kernel and the adding kernel do:
 *  1. every pair of every walk is done exactly once, in the order of the walk, shares differ by at most one pair;
 *  2. a part of a walk goes to a slot of its own; the adding kernel's rule names every cut walk exactly once and
 *     adds exactly the parts that were written for it, in the order of the walk;
 *  3. the workgroups' shares are a permutation. */
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "fa_bwd_layout.h"

static int fails = 0;
#define CHECK(cond, ...) do { if (!(cond)) { if (fails++ < 20) { printf(__VA_ARGS__); printf("\n"); } } } while (0)

static void check(int heads, int G, int S, int causal, int wl, int wr, int shares)
{
    int L, R;
    fa_mask_bounds(2 * S, causal, wl, wr, &L, &R);
    const int nkb = (S + 255) / 256;
    int per_head = 0;
    for (int kb = 0; kb < nkb; ++kb) per_head += G * fa_bwd_walk_tiles(S, S, R, L, kb);
    const int total = heads * per_head;
    if (total < shares) return;                                      /* (every share has at least one pair) */
    int *next = calloc((size_t)heads * nkb, sizeof(int));            /* pairs of the walk done so far */
    int *slot_walk = malloc(sizeof(int) * (size_t)shares * FA_BWD_PARTS_PER_SHARE);
    int *done = calloc((size_t)heads * nkb, sizeof(int)), *whole = calloc((size_t)heads * nkb, sizeof(int));
    char *seen = calloc((size_t)shares, 1);
    memset(slot_walk, 0xff, sizeof(int) * (size_t)shares * FA_BWD_PARTS_PER_SHARE);
    for (int b = 0; b < shares; ++b) {
        const int s = fa_bwd_share_of(b, shares);
        CHECK(s >= 0 && s < shares && !seen[s], "share %d of block %d", s, b);
        if (s >= 0 && s < shares) seen[s] = 1;
    }
    for (int s = 0; s < shares; ++s) {
        int at = fa_bwd_share_begin(s, shares, total);
        const int begin = at, end = fa_bwd_share_begin(s + 1, shares, total);
        CHECK(end - begin >= total / shares && end - begin <= total / shares + 1, "share %d has %d of %d", s, end - begin, total);
        while (at < end) {
            int h, kb, wb, len;
            fa_bwd_walk_at(at, per_head, G, S, S, R, L, &h, &kb, &wb, &len);
            CHECK(h >= 0 && h < heads && kb >= 0 && kb < nkb && at >= wb && at < wb + len, "walk of %d", at);
            const int from = at - wb, n = end - at < len - from ? end - at : len - from, w = h * nkb + kb;
            CHECK(next[w] == from, "walk %d: pair %d after %d", w, from, next[w]);
            next[w] = from + n;
            at += n;
            if (n == len) { whole[w]++; continue; }
            const int slot = fa_bwd_part_slot(s, from);
            /* (what the kernel derives at the end of the walk from the position alone) */
            int h2, kb2, wb2, len2;
            fa_bwd_walk_at(at - 1, per_head, G, S, S, R, L, &h2, &kb2, &wb2, &len2);
            CHECK((begin > wb2 || at < wb2 + len2) && fa_bwd_part_slot(s, begin > wb2 ? 1 : 0) == slot && h2 == h && kb2 == kb, "slot of share %d", s);
            CHECK(slot_walk[slot] == -1, "slot %d written twice", slot);
            slot_walk[slot] = w;
        }
    }
    for (int s = 1; s < shares; ++s) {                                /* the adding kernel */
        const int cut = fa_bwd_share_begin(s, shares, total);
        int h, kb, wb, len;
        fa_bwd_walk_at(cut, per_head, G, S, S, R, L, &h, &kb, &wb, &len);
        if (cut == wb || fa_bwd_share_begin(s - 1, shares, total) > wb) continue;
        int last = s;
        while (fa_bwd_share_begin(last + 1, shares, total) < wb + len) ++last;
        const int w = h * nkb + kb;
        done[w]++;
        CHECK(slot_walk[fa_bwd_part_slot(s - 1, 0)] == w, "first part of walk %d", w);
        slot_walk[fa_bwd_part_slot(s - 1, 0)] = -2;
        for (int p = s; p <= last; ++p) {
            CHECK(slot_walk[fa_bwd_part_slot(p, 1)] == w, "part %d of walk %d", p, w);
            slot_walk[fa_bwd_part_slot(p, 1)] = -2;
        }
    }
    for (int w = 0; w < heads * nkb; ++w) CHECK(whole[w] + done[w] == 1, "walk %d: whole %d, added %d", w, whole[w], done[w]);
    for (int i = 0; i < shares * FA_BWD_PARTS_PER_SHARE; ++i) CHECK(slot_walk[i] < 0, "slot %d was never added", i);
    free(next); free(slot_walk); free(done); free(whole); free(seen);
}

int main(void)
{
    static const int lens[] = {1, 63, 64, 255, 256, 257, 511, 1000, 2048, 4096, 5001}, masks[][3] = {{0, -1, -1}, {1, -1, -1}, {1, 0, -1}, {1, 300, -1}, {0, 64, 700}, {0, -1, 0}};
    for (unsigned l = 0; l < sizeof(lens) / sizeof(*lens); ++l)
        for (unsigned m = 0; m < sizeof(masks) / sizeof(*masks); ++m)
            for (int heads = 1; heads <= 16; heads += 5)
                for (int G = 1; G <= 8; G += 7)
                    for (int shares = 8; shares <= 256; shares = shares * 2 + 8)
                        check(heads, G, lens[l], masks[m][0], masks[m][1], masks[m][2], shares);
    if (fails) printf("%d failures\n", fails);
    return fails != 0;
}
