// Where a walked 64-row tile of the backward kernels sits in LDS, as plain integer arithmetic shared by the
// device code and a host-side check (compiled as C by the tests): which 16-byte chunk of the source a direct
// global->LDS load instruction puts where, and which LDS byte each lane addresses in the two read patterns.
#ifndef FA_BWD_LAYOUT_H
#define FA_BWD_LAYOUT_H

#include "fa_sched.h"

#if defined(__HIPCC__)
#define FA_LAYOUT_HD __host__ __device__ __forceinline__
#else
#define FA_LAYOUT_HD static inline
#endif

// One 16-byte-chunk swizzle that serves both read patterns, so that the tile sits in LDS once.  A row holds
// cpr = D/8 chunks (16 at D = 128, 8 at D = 64); logical chunk c of row r is stored at chunk position c ^ swz(r).
// ds_read_b128 by 16 lanes on 16 consecutive rows and one logical chunk needs 16 different positions inside
// 256 bytes (a bijection of the row's low bits); ds_read_b64_tr_b16 by 32 lanes on 4 consecutive rows x 4
// consecutive chunks needs the 4 rows in 4 different 64-byte groups (the two high bits follow the row's low
// bits).  Invariant under row += 16, not under row += 8.
FA_LAYOUT_HD int fa_u_swz(int cpr, int row)
{
    return cpr == 16 ? (((row & 3) << 2) | ((row >> 2) & 3)) : ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));
}

// Direct load: slot P (0 .. 64*cpr-1; lane l of the n-th wave instruction of a tile has P = 64 n + l) lands at LDS
// byte 16 P of the tile.  Returns the byte offset in the source tile it has to be fetched from.
FA_LAYOUT_HD int fa_bwd_load_source(int D, int P, int row_bytes)
{
    const int cpr = D / 8, row = P / cpr, pos = P % cpr;
    return row * row_bytes + ((pos ^ fa_u_swz(cpr, row)) << 4);
}

// ds_read_b128, A operand with rows = tile rows: lane (l32 = lane % 32, half = lane / 32) reads 16 bytes =
// head-dim values 16 s + 8 half .. + 7 of row l32 (+ 32 per row block, added as an immediate).
FA_LAYOUT_HD int fa_bwd_row_read(int D, int lane, int s)
{
    const int cpr = D / 8, half = lane >> 5, l32 = lane & 31;
    return l32 * D * 2 + (((2 * s + half) ^ fa_u_swz(cpr, l32)) << 4);
}

// ds_read_b64_tr_b16, A operand with rows = head dim (32-value block db), k = tile rows: the lane addresses the 8
// bytes = head-dim values 32 db + 16 (l32 / 16) + 4 (l16 % 4) .. + 3 of tile row 4 half + l16 / 4 + 8 hi (+ 16 per
// 16-row slice, added as an immediate); the instruction transposes among the 16 lanes that share l32 / 16 and half.
FA_LAYOUT_HD int fa_bwd_tr_read(int D, int lane, int db, int hi)
{
    const int cpr = D / 8, half = lane >> 5, l32 = lane & 31, l16 = lane & 15;
    const int row = 4 * half + (l16 >> 2) + 8 * hi, dq = l32 >> 4, c4 = l16 & 3;
    const int c = 4 * db + 2 * dq + (c4 >> 1);
    return row * D * 2 + ((c ^ fa_u_swz(cpr, row)) << 4) + ((c4 & 1) << 3);
}

// Where the 2 KiB dS block (32-query block qb, 32-key block kb) of a head lies in the five-product form's workspace,
// in blocks from the head's start.  Blocks are grouped in squares of 8 x 8 (256 queries x 256 keys, 128 KiB): the
// key-owning kernel (a workgroup = 8 or 4 key blocks, walking query tiles) and the query-owning kernel (a workgroup = 8 or 4
// query blocks, walking key tiles) then each work through one contiguous 128 KiB square for four tiles in a row
// (with whole block rows the query-owning kernel's eight waves read 512 KiB apart: 0.87 ms against 0.82 on B2 H32
// S8192 D128); inside a square the key block runs fastest, so the two blocks a query-owning wave needs per key tile
// are neighbours.
FA_LAYOUT_HD long long fa_ds_squares_per_side(int S) { return ((S + 31) / 32 + 7) / 8; }
FA_LAYOUT_HD long long fa_ds_blocks_per_head(int S) { return fa_ds_squares_per_side(S) * fa_ds_squares_per_side(S) * 64; }
FA_LAYOUT_HD long long fa_ds_block_index(int S, int qb, int kb)
{
    return (((long long)(qb >> 3) * fa_ds_squares_per_side(S) + (kb >> 3)) << 6) + ((qb & 7) << 3) + (kb & 7);
}

// ---- Equal shares of the key-owning kernel's work.  The walk of a key block (256 keys of a K/V head) visits the 64-query
// tiles that see one of its keys, for each of the G query heads that share the K/V head: G * tiles pairs, in that order
// (head by head, from the last tile down).  Under a causal mask block 0 walks all tiles and the last block four of
// them; a problem with few key blocks leaves CUs idle.  The walks of all blocks, block by block and head by head, are
// therefore laid end to end and cut into shares that differ by at most one pair (no more shares than pairs).
FA_LAYOUT_HD int fa_bwd_tiles_of_keys(int S, int Sk, int Lq, int Rq, int first, int keys)
{
    int lo, hi;
    fa_tile_range(S, 64, Lq, Rq, first, Sk - first < keys ? Sk - first : keys, &lo, &hi);
    return hi - lo + 1;
}
FA_LAYOUT_HD int fa_bwd_walk_tiles(int S, int Sk, int Lq, int Rq, int kblock) { return fa_bwd_tiles_of_keys(S, Sk, Lq, Rq, kblock * 256, 256); }
// Share of workgroup `block`: with workgroups dealt round robin over the eight XCDs, each XCD gets consecutive shares
// (a head or two of the list: what runs there at a time reads the same tiles).  `shares` is a multiple of eight.
FA_LAYOUT_HD int fa_bwd_share_of(int block, int shares) { return (block & 7) * (shares >> 3) + (block >> 3); }
FA_LAYOUT_HD int fa_bwd_share_begin(int share, int shares, int total) { return (int)((long long)share * total / shares); }
// The walk that pair `at` (of the whole list) belongs to: K/V head (counted from the launch's first) and key block, its
// first pair and its length.  per_head: pairs of one head's walks.
FA_LAYOUT_HD void fa_bwd_walk_at(int at, int per_head, int G, int S, int Sk, int Lq, int Rq, int *head, int *kblock, int *begin, int *len)
{
    const int h = (int)((unsigned)at / (unsigned)per_head);
    int from = h * per_head, kb = 0, n = G * fa_bwd_walk_tiles(S, Sk, Lq, Rq, 0);
    while (at >= from + n) {
        from += n;
        n = G * fa_bwd_walk_tiles(S, Sk, Lq, Rq, ++kb);
    }
    *head = h; *kblock = kb; *begin = from; *len = n;
}
// Where a share leaves the fp32 sums of a walk it does only a part of: the end of a walk that an earlier share began
// (from > 0, always the share's first walk) in the first of its two slots, a walk it begins and does not finish (its
// last) in the second.
#define FA_BWD_PARTS_PER_SHARE 2
FA_LAYOUT_HD int fa_bwd_part_slot(int share, int from) { return FA_BWD_PARTS_PER_SHARE * share + (from > 0 ? 0 : 1); }

// Whether the key-owning kernel with shares is built: not at head dimension 128 with dropout, which is out of registers
// (the 80-260 bytes of scratch memory that the shares cost it are touched in the tile loop).
#if defined(__cplusplus)
constexpr
#endif
FA_LAYOUT_HD int fa_bwd_can_share(int D, int dropout) { return !(D == 128 && dropout); }
// Whether the key-owning kernel's items differ in length: masked, and not a window of at most half the length.
FA_LAYOUT_HD int fa_bwd_uneven(int S, int Sk, int L, int R) { return (L < S + Sk || R < S + Sk) && 2LL * L > (long long)S; }
// How many equal shares the walks of a launch over `heads` K/V heads are cut into, or 0 to leave every walk to one
// workgroup: cut when the longest of a few workgroups (walking the items as a snake, or nearly in rounds when the
// hardware hands them out) has more than 4/3 of a share and 3 to 9 pairs, what writing and adding the parts costs, to do.
// (Why 4/3: the chip is at its power cap, and compute units that idle leave their power to the others.)  Backward pass,
// fp16, longest : share in pairs, cut against whole: causal D128 B1 H32/8 S4096 256 : 68 493 against 938 us, B1 H8 S2048
// 32 : 4.5 102 against 157, B1 H16 S1024 16 : 2.5 77 against 93, B2 H8 S512 8 : 2 51 against 59, without a mask B1 H40 S2048
// 64 : 40 330 against 370; and not cut: B1 H32 S2048 32 : 18 195 against 184, B6 H8 S2048 36 : 27 266 against 233, without a
// mask B2 H16 S512 D64 8 : 2 47 against 44.
// Head dimension 64: an uncut launch has items of 128 keys, two workgroups to a compute unit, so the longest is counted in
// pairs of 128 keys.  In units of a share's pair of 256, a workgroup that has its compute unit to itself takes 4/5 for one and
// two side by side 11/20 each; a cut costs 15 (256 shares; less with fewer).  Backward pass, fp16, longest : share, cut against
// whole, us: causal B1 H8 S2048 32 : 4.5 57 / 62, B1 H32/8 S2048 128 : 18 100 / 191, B1 H12 S3000 47 : 14 96 / 105, no mask B1 H4
// S8192 128 : 64 265 / 277; and not cut: causal B1 H16 S1024 16 : 2.5 43 / 37.5, B4 H8 S1024 16 : 5 49 / 40, B2 H8 S512 8 : 2 30 /
// 24, B5 H8 S4096 130 : 85 399 / 368, window 4000 B2 H8 S16000 260 : 229 994 / 877, no mask B1 H16 S2048 32 : 16 81 / 74.
FA_LAYOUT_HD long long fa_bwd_item_load(long long at, long long g, long long items, int snake, int heads, int n_kblocks, int keys, int G, int S, int Lq, int Rq)
{
    long long sum = 0;
    for (long long pass = 0; pass * g < items; ++pass) {
        const long long item = pass * g + (snake && (pass & 1) ? g - 1 - at : at);
        if (item >= items) continue;
        int head, kblock;
        fa_item_decode(item, heads, n_kblocks, 0, &head, &kblock);
        sum += (long long)G * fa_bwd_tiles_of_keys(S, S, Lq, Rq, kblock * keys, keys);
    }
    return sum;
}
FA_LAYOUT_HD int fa_bwd_shares(int D, int heads, int G, int S, int Lq, int Rq, int walk_head, int compute_units)
{
    const int keys = D == 64 ? 128 : 256, n_kblocks = (S + keys - 1) / keys;
    const long long total = (long long)heads * walk_head, items = (long long)heads * n_kblocks, slots = (long long)compute_units * (256 / keys);
    if (walk_head <= 0 || total > 0x3fffffffLL) return 0;
    long long shares = total / 2 / 8 * 8;          // at least two pairs each
    if (shares > compute_units) shares = compute_units / 8 * 8;
    if (shares < 8) return 0;
    const int snake = fa_bwd_uneven(S, S, Rq, Lq) && items < 16 * slots;
    const long long g = items < slots ? items : slots;
    long long worst = 0, worst_two = 0;            // of one workgroup, of the two of a compute unit
    for (int probe = 0; probe < 8; ++probe) {
        const long long at = probe == 7 ? (items - 1) % g : probe * (g - 1) / 6;
        const long long one = fa_bwd_item_load(at, g, items, snake, heads, n_kblocks, keys, G, S, Lq, Rq);
        if (one > worst) worst = one;
        if (D == 64 && at + compute_units < g) {
            const long long two = one + fa_bwd_item_load(at + compute_units, g, items, snake, heads, n_kblocks, keys, G, S, Lq, Rq);
            if (two > worst_two) worst_two = two;
        }
    }
    if (D == 64) {
        const long long sixtieths = 48 * worst > 33 * worst_two ? 48 * worst : 33 * worst_two;
        return sixtieths > 80 * total / shares + 900 * shares / 256 ? (int)shares : 0;
    }
    return 3 * worst > 4 * (total / shares) + 9 + 18 * shares / 256 ? (int)shares : 0;
}
// The buffer of the parts is sized on the host without a device, for FA_BWD_SHARE_UNITS compute units (a whole MI355X):
// the shares of the larger of the launches over a whole chunk of K/V heads and over the `rest` that is left (0: none).
#define FA_BWD_SHARE_UNITS 256
FA_LAYOUT_HD int fa_bwd_share_slots(int D, int chunk, int rest, int G, int S, int Lq, int Rq, int walk_head)
{
    const int whole = fa_bwd_shares(D, chunk, G, S, Lq, Rq, walk_head, FA_BWD_SHARE_UNITS);
    const int last = rest > 0 ? fa_bwd_shares(D, rest, G, S, Lq, Rq, walk_head, FA_BWD_SHARE_UNITS) : 0;
    return whole > last ? whole : last;
}
// The shares of one launch: by the compute units of the device it runs on, which may cut what FA_BWD_SHARE_UNITS would
// leave whole (a partition with 32 units: S 512, causal, chunks of 264 heads and a rest of 2, 32 shares where the buffer
// holds 8), and none when the buffer has fewer slots than that.
FA_LAYOUT_HD int fa_bwd_launch_shares(int D, int heads, int G, int S, int Lq, int Rq, int walk_head, int compute_units, int slots)
{
    const int shares = fa_bwd_shares(D, heads, G, S, Lq, Rq, walk_head, compute_units);
    return shares <= slots ? shares : 0;
}

#endif
