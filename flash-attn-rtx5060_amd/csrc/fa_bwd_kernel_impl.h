// FlashAttention backward for gfx950 (MI355X): dQ, dK, dV from Q, K, V, O, dO and the logsumexp the forward
// pass writes.  The reference has no backward pass (its L output is accepted and never written, reference
// src/flash_forward.h:602,628-644); this is the consumer of the logsumexp this library emits.
//
//   P  = exp(scale * Q K^T - LSE)            (recomputed; masked pairs are 0)
//   dV = P^T dO
//   dP = dO V^T,   delta_i = sum_t dO_it O_it
//   dS = P o (dP - delta)
//   dQ = scale * dS K,   dK = scale * dS^T Q
//
// Two kernels: fa_bwd_dq (a workgroup owns 256 queries and walks the key tiles; it also writes delta and the
// rescaled logsumexp for the second kernel) and fa_bwd_dkdv (a workgroup owns 256 or 128 keys of one K/V head and walks
// the query tiles of the query heads that share it); no atomics, every output element has one writer, results
// are the same bits from run to run.
// Template flags: LAYOUT 0 = contiguous [B,H,S,D] with S a multiple of 128 and as many keys; 1 (strided) = the
// same lengths with row, head and batch strides from the arguments and grouped K/V heads; 2 (general) = that
// plus any lengths (query i at key position i + Sk - S, ragged last tiles).  Each keeps its instruction stream
// free of what it does not need.  ALIBI subtracts slope[h] * |position - key| from the scaled score.  DROPOUT
// replays the forward pass's keep decisions from (seed, head, query position, key).  (Either one is instantiated
// for all three layouts, both together for the general one only.)
// Layouts 0 and 1 also have a five-product form (fa_bwd_prepare, fa_bwd_dkdv<WRITE_DS>, fa_bwd_dq_from_ds below).
// Both walkers use the building blocks of the forward kernel: 32x32x16 MFMA with the thing a wave owns on the
// lane (query in fa_bwd_dq, key in fa_bwd_dkdv), so that the owner's operands are B operands loaded once into
// registers, the walked tiles are A operands streamed through LDS by direct global->LDS loads, and an
// accumulator tile is already laid out as the B operand of the next product.
// A walked tile that is needed both row-wise (ds_read_b128) and transposed (ds_read_b64_tr_b16) sits in LDS
// once, under a swizzle that is bank-conflict-free for both.
#ifndef FA_BWD_KERNEL_IMPL_H
#define FA_BWD_KERNEL_IMPL_H
#include "fa_fwd_kernel_impl.h"
#include "fa_bwd_args.h"
#include "fa_bwd_layout.h"

namespace {

constexpr int kBwdWaves = 8;            // 8 waves x 32 owned rows = 256 rows per workgroup, two waves per SIMD
constexpr int kBwdStages = 3;           // LDS ring: with three stages one barrier per tile is enough
constexpr float kLog2e = 1.44269504088896340736f;
// K^T fragments that the key-owning kernel keeps in LDS (see there); the dropout words take the place of one
constexpr int fa_bwd_parked(int D, bool dropout) { return D == 128 ? (dropout ? 6 : 7) : 0; }
constexpr int kDsBlockBytes = 2048;     // one 32-query x 32-key block of dS in the storage type

// Takes the word by value on purpose: __builtin_bit_cast applied directly to an element of a vector
// (`__builtin_bit_cast(float, v[e])`) reads element 0 whatever e is with this compiler.
__device__ __forceinline__ float as_f32(uint32_t w) { return __builtin_bit_cast(float, w); }

// per-lane LDS addresses of the two read patterns in the stage being read; everything else about a fragment
// (which of the stage's tiles, which 32-row block, which 16-row slice) is an immediate offset of the read
template <int D> struct TileReader {
    static constexpr int CPR = D / 8, ROWB = D * 2, KS = D / 16, DB = D / 32;
    uint32_t row_addr[KS];      // ds_read_b128: A operand rows = tile rows, k = 16 head-dim values of slice s
    uint32_t tr_addr[DB][2];    // ds_read_b64_tr_b16: A operand rows = head dim (block db), k = 16 tile rows (two reads of 8)
    __device__ __forceinline__ void init(int lane, uint32_t stage_base)
    {
#pragma unroll
        for (int s = 0; s < KS; ++s) row_addr[s] = stage_base + (uint32_t)fa_bwd_row_read(D, lane, s);
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int hi = 0; hi < 2; ++hi) tr_addr[db][hi] = stage_base + (uint32_t)fa_bwd_tr_read(D, lane, db, hi);
    }
    // move to another stage of the ring (delta in bytes, wave-uniform)
    __device__ __forceinline__ void advance(int delta)
    {
#pragma unroll
        for (int s = 0; s < KS; ++s) row_addr[s] += delta;
#pragma unroll
        for (int db = 0; db < DB; ++db) { tr_addr[db][0] += delta; tr_addr[db][1] += delta; }
    }
    // row-wise fragment: head-dim slice s, 32-row block b of the tile at byte `tile` of the stage
    __device__ __forceinline__ u32x4 rows(int tile, int s, int b) const { return lds_read_b128(row_addr[s] + (uint32_t)(tile + b * 32 * ROWB)); }
    // transposed fragment: 16-row slice t2, head-dim block db of the tile at byte `tile` of the stage
    __device__ __forceinline__ u32x4 transposed(int tile, int t2, int db) const
    {
        const u32x2 lo = lds_read_tr(tr_addr[db][0] + (uint32_t)(tile + (16 * t2) * ROWB));
        const u32x2 hi = lds_read_tr(tr_addr[db][1] + (uint32_t)(tile + (16 * t2) * ROWB));
        return u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
};

// one 64-row tile global -> LDS: wave w of NW issues instructions w, w + NW, ...
template <int D, int NW = kBwdWaves> struct TileLoader {
    static constexpr int CPR = D / 8, ROWB = D * 2, TILEB = 64 * ROWB, IPW = TILEB / 1024 / NW;
    uint32_t g[IPW];
    int wave, lane;
    // row_bytes: distance between consecutive rows of the source in bytes
    __device__ __forceinline__ void init(int wave_, int lane_, int row_bytes)
    {
        wave = wave_; lane = lane_;
#pragma unroll
        for (int i = 0; i < IPW; ++i) {
            g[i] = (uint32_t)fa_bwd_load_source(D, (i * NW + wave) * 64 + lane, row_bytes);
        }
    }
    __device__ __forceinline__ void load(const uint16_t *tile_src, uint32_t lds_tile) const
    {
#pragma unroll
        for (int i = 0; i < IPW; ++i)
            dma_16(reinterpret_cast<const char *>(tile_src), g[i], lds_tile + (i * NW + wave) * 1024);
    }
    // a tile whose last rows lie past the end of the tensor: they are filled with copies of row `valid - 1`
    __device__ __forceinline__ void load_ragged(const uint16_t *tile_src, uint32_t lds_tile, int valid, int row_bytes) const
    {
        // (the empty asm keeps the address arithmetic of this rare path inside its branch: hoisted out of the
        // tile loop it would occupy registers for the whole kernel)
        int ln = lane;
        asm volatile("" : "+v"(ln));
#pragma unroll
        for (int i = 0; i < IPW; ++i) {
            const int P = (i * NW + wave) * 64 + ln, row = P / CPR, pos = P % CPR;
            const int src_row = row < valid ? row : valid - 1;
            dma_16(reinterpret_cast<const char *>(tile_src), (uint32_t)(src_row * row_bytes + ((pos ^ fa_u_swz(CPR, row)) << 4)),
                   lds_tile + (i * NW + wave) * 1024);
        }
    }
};

// 256 bytes (64 floats) global -> LDS in one wave instruction: lane l copies the float at src[index] to LDS
// byte lds + 4*l
__device__ __forceinline__ void dma_4(const float *src, int index, uint32_t lds)
{
    const uint64_t b = (uint64_t)src;
    const uint32_t b_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
    const uint32_t b_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    const uint64_t ub = ((uint64_t)b_hi << 32) | (uint64_t)b_lo;
    const uint32_t voff = (uint32_t)index * 4u;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(ub) : "memory", "m0");
}

// s_waitcnt vmcnt(n) for a wave-uniform run-time n (the instruction takes an immediate)
__device__ __forceinline__ void wait_vm_upto(int n)
{
    switch (n) {
#define FA_WAIT_CASE(k) case k: wait_vm<k>(); break;
    FA_WAIT_CASE(0) FA_WAIT_CASE(1) FA_WAIT_CASE(2) FA_WAIT_CASE(3) FA_WAIT_CASE(4) FA_WAIT_CASE(5) FA_WAIT_CASE(6) FA_WAIT_CASE(7)
    FA_WAIT_CASE(8) FA_WAIT_CASE(9) FA_WAIT_CASE(10) FA_WAIT_CASE(11) FA_WAIT_CASE(12) FA_WAIT_CASE(13) FA_WAIT_CASE(14) FA_WAIT_CASE(15)
    FA_WAIT_CASE(16)
#undef FA_WAIT_CASE
    default: wait_vm<0>(); break;
    }
}

// dma_16 with the streaming hint: data that is read exactly once should not displace what others re-read from L2
__device__ __forceinline__ void dma_16_stream(const char *base, uint32_t voff, uint32_t lds)
{
    const uint64_t b = (uint64_t)base;
    const uint32_t b_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
    const uint32_t b_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    const uint64_t ub = ((uint64_t)b_hi << 32) | (uint64_t)b_lo;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                 :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(ub) : "memory", "m0");
}

// the lane index, read from the hardware and tied to the place of the call: what follows from it is formed there instead of
// once at the top and kept in registers
__device__ __forceinline__ int lane_here()
{
    int ln = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(ln));
    return ln;
}

__device__ __forceinline__ f32x16 zero16()
{
    f32x16 z;
#pragma unroll
    for (int r = 0; r < 16; ++r) z[r] = 0.0f;
    return z;
}

// The kernel's arguments, read again from the kernel-argument segment: what is taken from the by-value argument
// is loaded once in front of the item loop and then kept in scalar registers through every tile loop; a use behind
// this call loads it where it is needed (scalar loads from a segment that stays in the scalar cache).
__device__ __forceinline__ const FaBwdArgs &args_reloaded()
{
    typedef const __attribute__((address_space(4))) FaBwdArgs *KernargPtr;
    KernargPtr ka = (KernargPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ka));
    return *(const FaBwdArgs *)ka;
}

__device__ __forceinline__ const uint16_t *head_ptr(const uint16_t *p, const FaBwdTensor &t, int b, int h)
{
    return p + (long long)b * t.bs + (long long)h * t.hs;
}
__device__ __forceinline__ uint16_t *head_ptr(uint16_t *p, const FaBwdTensor &t, int b, int h)
{
    return p + (long long)b * t.bs + (long long)h * t.hs;
}

// ---------------------------------------------------------------------------------------------------------
// dQ: a workgroup owns 256 queries (lane = query), walks the key tiles of its visible range.
// LDS stage: K (read row-wise for S^T = K Q^T and transposed for dQ^T += K^T dS^T), V (row-wise, dP^T = V dO^T).
// ---------------------------------------------------------------------------------------------------------
template <bool BF16, int D, bool MASKED, int LAYOUT, bool ALIBI, bool DROPOUT>
__global__ void __launch_bounds__(kBwdWaves * 64, 2) fa_bwd_dq(const FaBwdArgs a)
{
    constexpr bool STRIDES = LAYOUT >= 1, GENERAL = LAYOUT == 2, ONE_ITEM = STRIDES && D == 128 && !(DROPOUT && MASKED && !GENERAL);
    static_assert(LAYOUT >= 0 && LAYOUT <= 2, "0 the reference's layout, 1 strided, 2 general");
    static_assert(!GENERAL || MASKED, "the general instantiations always carry the mask code (ragged tiles need it)");

    typedef Num<BF16> N;
    typedef TileReader<D> Reader;
    typedef TileLoader<D> Loader;
    constexpr int KS = Reader::KS, DB = Reader::DB, TILEB = Loader::TILEB, STAGEB = 2 * TILEB, IPW = Loader::IPW;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int S = a.S, Sk = GENERAL ? a.Sk : a.S, off = GENERAL ? a.Sk - a.S : 0;
    const int n_qblocks = (S + 255) / 256;
    // one head per XCD at a time, long blocks first: the workgroups that share a head's K and V share an L2
    // Work items: one workgroup per item, or (grid smaller than the list) a resident grid that walks the
    // longest-first list as a snake, pass 0 forwards, pass 1 backwards, ..., which pairs long items with short ones.
    const long long n_items = (long long)a.B * a.H * n_qblocks;
    for (int pass = 0; !ONE_ITEM || pass < 1; ++pass) {       // (128-wide strided and general instantiations: exactly one item, no loop)
    const long long item = (long long)pass * gridDim.x + ((pass & 1) ? gridDim.x - 1 - blockIdx.x : blockIdx.x);
    if (item >= n_items) break;
    if (pass > 0) __syncthreads();          // (the LDS stages: other waves may still be reading the last tile)
    // (the lane index is taken from the hardware once per work item and tied to this place: what is derived from
    // it would otherwise be computed in front of the item loop and kept in registers through every tile loop)
    int lane = ONE_ITEM ? (int)threadIdx.x & 63 : (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    if (!ONE_ITEM) asm volatile("" : "+v"(lane));
    const int half = lane >> 5, l32 = lane & 31;
    int bh, qblock;
    fa_item_decode(item, a.B * a.H, n_qblocks, MASKED ? 1 : 0, &bh, &qblock);
    const int b = bh / a.H, h = bh - b * a.H, hk = STRIDES ? h / (a.H / a.Hk) : h;
    const int q_rs = STRIDES ? a.q.rs : D, k_rs = STRIDES ? a.k.rs : D, v_rs = STRIDES ? a.v.rs : D;
    const int o_rs = STRIDES ? a.o.rs : D, g_rs = STRIDES ? a.dO_.rs : D, dq_rs = STRIDES ? a.dq.rs : D;
    const uint16_t *Qh, *Kh, *Vh, *Oh, *dOh;
    uint16_t *dQh;
    if (STRIDES) {
        Qh = head_ptr(a.Q, a.q, b, h); Kh = head_ptr(a.K, a.k, b, hk); Vh = head_ptr(a.V, a.v, b, hk);
        Oh = head_ptr(a.O, a.o, b, h); dOh = head_ptr(a.dO, a.dO_, b, h); dQh = head_ptr(a.dQ, a.dq, b, h);
    } else {
        const size_t head_off = (size_t)bh * S * D;
        Qh = a.Q + head_off; Kh = a.K + head_off; Vh = a.V + head_off; Oh = a.O + head_off; dOh = a.dO + head_off;
        dQh = a.dQ + head_off;
    }
    const int q0 = qblock * 256, qw = q0 + wave * 32;
    const bool active = qw < S;                    // the last block may own fewer than 256 rows
    const int my_q = active ? (GENERAL && qw + l32 >= S ? S - 1 : qw + l32) : (GENERAL ? 0 : l32);   // row to load
    const bool row_ok = active && qw + l32 < S;
    const int my_pos = qw + l32 + off;             // key position of this lane's query (masks, ALiBi)

    u32x4 qf[KS], gf[KS];           // Q^T and dO^T as B operands: lane = (query, head-dim slice 8*half..+7 of each 16)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        qf[s] = *reinterpret_cast<const u32x4 *>(Qh + (size_t)my_q * q_rs + 16 * s + 8 * half);
        gf[s] = *reinterpret_cast<const u32x4 *>(dOh + (size_t)my_q * g_rs + 16 * s + 8 * half);
    }
    // logsumexp in exp2 units; a row that saw no key has -inf there and takes +inf here, which makes every P 0
    const float lse_raw = a.lse[(size_t)bh * S + my_q];
    float lse_l2 = (GENERAL && lse_raw == -INFINITY) ? INFINITY : lse_raw * kLog2e;
    // delta_i = sum_t dO_it O_it: this lane holds half of row i of dO already; the other half is on lane ^ 32.
    // Both are written out for fa_bwd_dkdv, which runs after this kernel.
    float delta = 0.0f;
    {
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const u32x4 o = *reinterpret_cast<const u32x4 *>(Oh + (size_t)my_q * o_rs + 16 * s + 8 * half);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const uint32_t ow = o[w], gw = gf[s][w];
                delta += storage_to_f32<BF16>((uint16_t)(ow & 0xffffu)) * storage_to_f32<BF16>((uint16_t)(gw & 0xffffu));
                delta += storage_to_f32<BF16>((uint16_t)(ow >> 16)) * storage_to_f32<BF16>((uint16_t)(gw >> 16));
            }
        }
        delta += swap_halves(delta);
        if (row_ok && half == 0) {
            a.delta[(size_t)bh * S + my_q] = -delta / a.drop_scale;
            a.lse2[(size_t)bh * S + my_q] = (GENERAL && lse_raw == -INFINITY) ? -INFINITY : (a.drop_log - lse_raw) / a.key_scale;
        }
    }
    const float c = a.scale * kLog2e;
    float slope_l2 = 0.0f;
    if (ALIBI) slope_l2 = a.alibi[h] * kLog2e;

    int t0, t1, my_lo = 1, my_hi = 0;
    fa_tile_range(Sk, 64, a.L, a.R, q0 + off, S - q0 < 256 ? S - q0 : 256, &t0, &t1);
    if (active) fa_tile_range(Sk, 64, a.L, a.R, qw + off, GENERAL && S - qw < 32 ? S - qw : 32, &my_lo, &my_hi);

    Reader rd; rd.init(lane, lds0);
    Loader ldk, ldv;
    ldk.init(wave, lane, k_rs * 2);
    if (STRIDES) ldv.init(wave, lane, v_rs * 2);
    auto issue = [&](int tile, int stage) __attribute__((always_inline)) {
        const uint32_t base = lds0 + stage * STAGEB;
        if (GENERAL && (tile + 1) * 64 > Sk) {
            ldk.load_ragged(Kh + (size_t)tile * 64 * k_rs, base, Sk - tile * 64, k_rs * 2);
            ldv.load_ragged(Vh + (size_t)tile * 64 * v_rs, base + TILEB, Sk - tile * 64, v_rs * 2);
        } else {
            ldk.load(Kh + (size_t)tile * 64 * k_rs, base);
            (STRIDES ? ldv : ldk).load(Vh + (size_t)tile * 64 * v_rs, base + TILEB);
        }
    };

    f32x16 dq[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) dq[db] = zero16();

    // 32 keys (block kb of the tile in the stage being read) against this wave's 32 queries
    auto half_tile = [&](bool edge, int t, int kb) __attribute__((always_inline)) {
        constexpr int k_tile = 0, v_tile = TILEB;
        f32x16 sx = zero16(), dp = zero16();
#pragma unroll
        for (int s = 0; s < KS; ++s) sx = N::mfma(rd.rows(k_tile, s, kb), qf[s], sx);      // S^T = K Q^T
#pragma unroll
        for (int s = 0; s < KS; ++s) dp = N::mfma(rd.rows(v_tile, s, kb), gf[s], dp);      // dP^T = V dO^T
        const int first = t * 64 + 32 * kb + 4 * half;                      // key of accumulator row 0 on this lane
        if (MASKED && edge) {            // wave-uniform; a masked score becomes -inf and its P exactly 0
            int hi = my_pos + a.R, lo = my_pos - a.L - first;                // visible: lo <= 8*(r/4) + r%4 <= hi
            if (GENERAL && hi > Sk - 1) hi = Sk - 1;
            hi -= first;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (8 * (r >> 2) + (r & 3) > hi || 8 * (r >> 2) + (r & 3) < lo) sx[r] = -INFINITY;
        }
        // dropout: the forward kept key j of this query iff byte r of this block is >= the threshold, and scaled
        // the kept probabilities; the same factor reaches dP, while the softmax Jacobian sees the undropped P
        DropWords dw;
        if (DROPOUT) dw = dropout_words(a.seed_lo, a.seed_hi, (uint32_t)bh, (uint32_t)my_pos, (uint32_t)(2 * (2 * t + kb) + half));
        uint32_t ds[8];                                  // dS^T in B-operand order
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float v[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int r = 2 * i + e;
                float x = __builtin_fmaf(sx[r], c, -lse_l2);
                if (ALIBI) x = __builtin_fmaf(-slope_l2, __builtin_fabsf((float)(first + 8 * (r >> 2) + (r & 3) - my_pos)), x);
                const float p = __builtin_amdgcn_exp2f(x);
                float dpr = dp[r];
                if (DROPOUT) dpr = dropout_keep_byte(dw, r, a.drop_threshold) ? dpr * a.drop_scale : 0.0f;
                v[e] = p * (dpr - delta);
            }
            ds[i] = N::pack2(v[0], v[1]);
        }
#pragma unroll
        for (int n = 0; n < 2 * DB; ++n) {                // dQ^T += K^T dS^T
            const int h2 = n / DB, db = n % DB;
            const u32x4 bfrag = {ds[4 * h2], ds[4 * h2 + 1], ds[4 * h2 + 2], ds[4 * h2 + 3]};
            dq[db] = N::mfma(rd.transposed(k_tile, 2 * kb + h2, db), bfrag, dq[db]);
        }
    };

    if (t0 <= t1) {
        // Tiles are fetched two ahead: tile t+2 is issued at the end of iteration t, into the stage tile t-1 was
        // read from (free for everyone since this iteration's barrier).  A wait for "everything in flight" in the
        // middle of an iteration -- the compiler's own, around a register it spilled -- then only meets loads
        // that were issued a whole iteration earlier.
        issue(t0, 0);
        if (t0 + 1 <= t1) issue(t0 + 1, 1);
        wait_vm<0>();
        // the owner's operands have landed too: say so, or the compiler waits for them inside the loop, where
        // its wait would also cover the asynchronous tile loads
#pragma unroll
        for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[s]), "+v"(gf[s]));
        asm volatile("" : "+v"(lse_l2), "+v"(delta), "+v"(slope_l2));
        int stage = 0;
        for (int t = t0; t <= t1; ++t) {
            const int next = stage == kBwdStages - 1 ? 0 : stage + 1;
            if (t + 1 <= t1) wait_vm<2 * IPW>();                // tile t has landed, tile t+1 may still be in flight
            else wait_vm<0>();
            phase_barrier();                                    // tile t is in LDS for everyone; tile t-1's stage is free
            if (my_lo <= t && t <= my_hi) {
                const bool edge = MASKED && (fa_tile_class(64, a.L, a.R, qw + off, 32, t) == 1 || (GENERAL && (t + 1) * 64 > Sk));
                half_tile(edge, t, 0);
                half_tile(edge, t, 1);
            }
            if (t + 2 <= t1) issue(t + 2, next == kBwdStages - 1 ? 0 : next + 1);
            rd.advance(next == 0 ? -(kBwdStages - 1) * STAGEB : STAGEB);
            stage = next;
        }
    }
    if (row_ok) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                u32x2 w;
                w[0] = N::pack2(dq[db][4 * g] * a.scale, dq[db][4 * g + 1] * a.scale);
                w[1] = N::pack2(dq[db][4 * g + 2] * a.scale, dq[db][4 * g + 3] * a.scale);
                *reinterpret_cast<u32x2 *>(dQh + (size_t)my_q * dq_rs + 32 * db + 8 * g + 4 * half) = w;
            }
    }
    }   // next work item
}

// ---------------------------------------------------------------------------------------------------------
// dK, dV: a workgroup owns 32 NW keys of one K/V head (256, or 128 in the five-product form's uncut launches at head dimension
// 64; lane = key), walks the query tiles that see them, for each
// of the query heads that share the K/V head.
// LDS stage: Q (row-wise for S = Q K^T, transposed for dK^T += Q^T dS), dO (row-wise for dP = dO V^T, transposed
// for dV^T += dO^T P), the 64 words each that the accumulators of S and dP start from (FaBwdArgs).
// ---------------------------------------------------------------------------------------------------------
// WRITE_DS (the five-product form): every 32-query x 32-key block of dS that a wave forms is also written to
// a.ds_blocks, in the wave's operand order, for fa_bwd_dq_from_ds.
// SHARES (with WRITE_DS): the walks cut into equal shares, see fa_bwd_layout.h.
// ONE_ITEM: no loop around the work item (see launch_bwd).
template <bool BF16, int D, bool MASKED, int LAYOUT, bool ALIBI, bool DROPOUT, bool WRITE_DS = false, bool SHARES = false, int NW = kBwdWaves,
          bool ONE_ITEM = LAYOUT >= 1 && D == 128 && !WRITE_DS>
__global__ void __launch_bounds__(NW * 64, 2) fa_bwd_dkdv(const FaBwdArgs a)
{
    constexpr bool STRIDES = LAYOUT >= 1, GENERAL = LAYOUT == 2;
    static_assert(!SHARES || (WRITE_DS && !ONE_ITEM), "a share is several walks, one pass of the item loop each");
    static_assert(!WRITE_DS || LAYOUT <= 1 || (!ALIBI && !DROPOUT), "general lengths: dS blocks without ALiBi and dropout only");
    typedef Num<BF16> N;
    typedef TileReader<D> Reader;
    typedef TileLoader<D, NW> Loader;
    constexpr int BK = 32 * NW;                   // keys per workgroup
    constexpr int KS = Reader::KS, DB = Reader::DB, TILEB = Loader::TILEB, STAGEB = 2 * TILEB + 512, IPW = Loader::IPW;
    // LDS reads run this many matrix instructions ahead (at head dimension 128 what the registers hold: three with less of K
    // in LDS, or with fewer address registers and an instruction more per read, measured 1-4 % slower on every shape tried).
    // Masked walks with ALiBi, and masked shares in the reference's layout, hold one: with two they reload spilled values in
    // every tile or walk, behind a wait for all loads and stores in flight.  Backward pass, causal, two ahead / one, us: ALiBi
    // B2 H16 S4096 424 / 396, B4 H16 S2048 250 / 232, B1 H8 S2048 stored [B,S,H,D] (shares) 92.6 / 86.2, B1 H32/4 S2048 149.7 /
    // 144.9 (B2 H32/8 S4096 840 / 853 the other way); without ALiBi, shares, B1 H8 S2048 87.0 / 86.0, B1 H16 S1024 66.4 / 64.2.
    constexpr bool TIGHT = WRITE_DS && MASKED && (ALIBI || (LAYOUT == 0 && SHARES));
    constexpr int PD = D == 64 ? 4 : DROPOUT || TIGHT ? 1 : 2;
    constexpr int NSTG = kBwdStages;                                  // LDS stages; pairs are requested NSTG - 1 ahead
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int S = a.S, Sk = GENERAL ? a.Sk : a.S, off = GENERAL ? a.Sk - a.S : 0;
    const int G = STRIDES ? a.H / a.Hk : 1;
    const int n_kblocks = (Sk + BK - 1) / BK;
    // one K/V head per XCD at a time; key block 0 is seen by the most queries and goes first
    // (work items as in fa_bwd_dq; the list here is ascending in the key block, which is longest first under a
    // causal mask: key block 0 is seen by every query)
    const long long n_items = (long long)a.heads * n_kblocks;
    // Equal shares: the walks of all key blocks one behind the other, cut into as many shares as there are
    // workgroups (fa_bwd_layout.h); a share covers the end of one walk, whole walks, and the beginning of another.
    // (What this needs besides the position `share_at` is read and formed again at each place that uses it: scalar
    // registers held through the tile loop are spilled into vector registers, which the 128-wide kernels do not have.)
    int share_at = 0;
    if (SHARES) share_at = fa_bwd_share_begin(fa_bwd_share_of((int)blockIdx.x, (int)gridDim.x), (int)gridDim.x, a.walk_total);
    for (int pass = 0; !ONE_ITEM || pass < 1; ++pass) {       // (128-wide strided and general instantiations: exactly one item, no loop)
    const long long item = (long long)pass * gridDim.x + ((pass & 1) ? gridDim.x - 1 - blockIdx.x : blockIdx.x);
    if (!SHARES && item >= n_items) break;
    if (pass > 0) __syncthreads();
    int lane = ONE_ITEM ? (int)threadIdx.x & 63 : (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    if (!ONE_ITEM) asm volatile("" : "+v"(lane));
    const int half = lane >> 5, l32 = lane & 31;
    int bhk, kblock;
    int walk_from = 0, walk_pairs = 0;             // shares: the (query head, query tile) pairs of the walk this pass does
    if (SHARES) {
        const FaBwdArgs &f = args_reloaded();
        const int end = fa_bwd_share_begin(fa_bwd_share_of((int)blockIdx.x, (int)gridDim.x) + 1, (int)gridDim.x, f.walk_total);
        if (share_at >= end) break;
        int walk_begin, walk_len;
        fa_bwd_walk_at(share_at, f.walk_head, G, S, Sk, f.R + off, f.L - off, &bhk, &kblock, &walk_begin, &walk_len);
        walk_from = share_at - walk_begin;
        walk_pairs = end - share_at < walk_len - walk_from ? end - share_at : walk_len - walk_from;
        share_at += walk_pairs;
    } else {
        fa_item_decode(item, a.heads, n_kblocks, 0, &bhk, &kblock);
    }
    bhk += a.head0;
    const int b = bhk / a.Hk, hk = bhk - b * a.Hk;
    const int q_rs = STRIDES ? a.q.rs : D, g_rs = STRIDES ? a.dO_.rs : D, k_rs = STRIDES ? a.k.rs : D, v_rs = STRIDES ? a.v.rs : D;
    const uint16_t *Kh, *Vh;
    if (STRIDES) {
        Kh = head_ptr(a.K, a.k, b, hk); Vh = head_ptr(a.V, a.v, b, hk);
    } else {
        const size_t head_off = (size_t)bhk * S * D;
        Kh = a.K + head_off; Vh = a.V + head_off;
    }
    const int k0 = kblock * BK, kw = k0 + wave * 32;
    const bool active = kw < Sk;
    const int my_k = kw + l32;                     // this lane's key (masks, ALiBi)
    const int my_kc = active ? (GENERAL && my_k >= Sk ? Sk - 1 : my_k) : (GENERAL ? 0 : l32);     // row to load

    u32x4 kf[KS], vf[KS];           // K^T and V^T as B operands: lane = (key, head-dim slice)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        kf[s] = *reinterpret_cast<const u32x4 *>(Kh + (size_t)my_kc * k_rs + 16 * s + 8 * half);
        vf[s] = *reinterpret_cast<const u32x4 *>(Vh + (size_t)my_kc * v_rs + 16 * s + 8 * half);
    }
    const float c = a.key_scale * kLog2e;

    // the query tiles that see these keys: the query at index i (position i + off) sees key j iff
    // j - R - off <= i <= j + L - off: the forward bounds with the two sides exchanged and shifted
    const int Lq = a.R + off, Rq = a.L - off;
    int t0, t1, my_lo = 1, my_hi = 0;
    fa_tile_range(S, 64, Lq, Rq, k0, Sk - k0 < BK ? Sk - k0 : BK, &t0, &t1);
    if (active) fa_tile_range(S, 64, Lq, Rq, kw, GENERAL && Sk - kw < 32 ? Sk - kw : 32, &my_lo, &my_hi);

    Reader rd; rd.init(lane, lds0);
    uint32_t stat_addr = lds0 + 2 * TILEB + 16 * half;       // this lane's logsumexp / delta words in the stage being read
    const uint32_t drop_lds = lds0 + NSTG * STAGEB + wave * 1024;       // dropout: 1 KB per wave behind the ring
    Loader ldq, ldg;
    if (!STRIDES || GENERAL) ldq.init(wave, lane, q_rs * 2);      // (general: only its ragged tiles go through these two)
    if (GENERAL) ldg.init(wave, lane, g_rs * 2);
    // strided layouts: where the walked query head starts (Q, dO, its rescaled logsumexps and deltas), formed when the
    // walk moves to the next head of the group and carried in eight scalar registers; the strides themselves are
    // read again at every fetch
    const uint16_t *walk_q = nullptr, *walk_g = nullptr;
    const float *walk_lse = nullptr, *walk_delta = nullptr;
    auto walk_head = [&](int g) __attribute__((always_inline)) {
        const FaBwdArgs &f = args_reloaded();
        const int h = hk * G + g;
        walk_q = head_ptr(f.Q, f.q, b, h); walk_g = head_ptr(f.dO, f.dO_, b, h);
        walk_lse = f.lse2 + ((size_t)b * f.H + h) * S; walk_delta = f.delta + ((size_t)b * f.H + h) * S;
    };
    // g: query head inside the group of this K/V head
    auto issue = [&](int g, int tile, int stage) __attribute__((always_inline)) {
        const uint32_t base = lds0 + stage * STAGEB;
        const int h = hk * G + g;
        const uint16_t *Qh, *dOh;
        const float *lse_h, *delta_h;
        if (STRIDES) {
            Qh = walk_q; dOh = walk_g; lse_h = walk_lse; delta_h = walk_delta;
        } else {
            Qh = a.Q + (size_t)bhk * S * D; dOh = a.dO + (size_t)bhk * S * D;
            lse_h = a.lse2 + ((size_t)b * a.H + h) * S; delta_h = a.delta + ((size_t)b * a.H + h) * S;
        }
        if (GENERAL && (tile + 1) * 64 > S) {
            const int valid = S - tile * 64;
            ldq.load_ragged(Qh + (size_t)tile * 64 * q_rs, base, valid, q_rs * 2);
            ldg.load_ragged(dOh + (size_t)tile * 64 * g_rs, base + TILEB, valid, g_rs * 2);
            int ln = lane;
            asm volatile("" : "+v"(ln));
            if (wave == 0) dma_4(lse_h + tile * 64, ln < valid ? ln : valid - 1, base + 2 * TILEB);
            if (wave == 1) dma_4(delta_h + tile * 64, ln < valid ? ln : valid - 1, base + 2 * TILEB + 256);
        } else if (STRIDES) {
            // (the lanes' source offsets are formed here, from the hardware's lane index and freshly loaded strides:
            // kept in registers from the top of the item they are spilled, and every reload in the tile loop waits
            // for all loads in flight)
            const FaBwdArgs &f = args_reloaded();
            int ln = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
            asm volatile("" : "+v"(ln));
            Loader lq, lg;
            lq.init(wave, ln, f.q.rs * 2);
            lg.init(wave, ln, f.dO_.rs * 2);
            lq.load(Qh + (size_t)tile * 64 * f.q.rs, base);
            lg.load(dOh + (size_t)tile * 64 * f.dO_.rs, base + TILEB);
            if (wave == 0) dma_4(lse_h + tile * 64, ln, base + 2 * TILEB);
            if (wave == 1) dma_4(delta_h + tile * 64, ln, base + 2 * TILEB + 256);
        } else {
            ldq.load(Qh + (size_t)tile * 64 * q_rs, base);
            ldq.load(dOh + (size_t)tile * 64 * g_rs, base + TILEB);
            if (wave == 0) dma_4(lse_h + tile * 64, lane, base + 2 * TILEB);
            if (wave == 1) dma_4(delta_h + tile * 64, lane, base + 2 * TILEB + 256);
        }
    };
    f32x16 dk[DB], dv[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) { dk[db] = zero16(); dv[db] = zero16(); }
    // Head dimension 128: the kernel needs every register it can have (two waves per SIMD: 256), and a value the compiler
    // spills to scratch memory inside the tile loop comes back behind a wait for ALL loads and stores in flight.  The last
    // PARKED of the K^T fragments, which every half tile uses once, are kept in LDS instead (a plane of 16 bytes per lane
    // each, written once per work item) and read like any A operand: K's, because dP, dS and P are not alive yet where they
    // are used.  (One K and one V fragment, as before the reads ran ahead: spills of 80-360 bytes inside the loop.  What is
    // left of spills: see PD.)
    constexpr int PARKED = fa_bwd_parked(D, DROPOUT);
    constexpr uint32_t kParkPlane = 16u * NW * 64u;
    const uint32_t park_lds = lds0 + NSTG * STAGEB + (DROPOUT ? NW * 1024 : 0);       // (behind the dropout words)
    const uint32_t park_addr = park_lds + 16u * ((uint32_t)wave * 64u + (uint32_t)lane);
    auto parked = [&](int plane) __attribute__((always_inline)) {
        return *(volatile __attribute__((address_space(3))) u32x4 *)(uintptr_t)(park_addr + kParkPlane * (uint32_t)plane);
    };

    // Dropout decisions of the 32 x 32 block (query block qb of tile t, this wave's keys).  A Philox block covers sixteen
    // keys of ONE query, and a lane here owns a key: lane (l32, half) draws for query 32 qb + l32 the sixteen bytes of the
    // keys 8 g + 4 half + e (word g, byte e); the 4 x 4 bytes of four neighbouring lanes are transposed in registers, so that
    // a word holds four queries of ONE key, and the words change lanes through 1 KB of LDS that belong to the wave.
    // (Bound by the vector ALU: ten Philox rounds, then a comparison and a select per element for P and for dP.  With the bytes
    // compared in front of the exchange and sixteen bits put together on both sides of it, p = 0.1: B16 H16 S512 D64 no mask
    // 121 us, now 112; B16 H32 S1534 D128 causal 2036 / 1644; B4 H32 S1024 D128 no mask 404 / 273; all of the backward pass.)
    // (Head dimension 64: what the draws of a head have in common is kept in four registers; the 128-wide kernels have none left.
    // With it against all twenty products per draw: B16 H16 S512 D64 no mask, forward and backward, 138.5 against 140.1 us, B4 H16 S2048
    // 244.4 / 247.1, B8 H16 S1000 161.2 / 163.9.)
    DropAhead ahead = {0, 0, 0, 0, 0};
    uint32_t ahead_of = 0xffffffffu;
    auto draw = [&](uint32_t bhq, int t, int qb) __attribute__((always_inline)) {
        const int ln = lane_here(), key = ln & 31, quarter = ln >> 5;
        // (the seed's registers are tied to this place too: the ten rounds' keys would otherwise be kept in twenty registers)
        uint32_t seed_lo = a.seed_lo, seed_hi = a.seed_hi;
        asm volatile("" : "+s"(seed_lo), "+s"(seed_hi));
        const uint32_t query = (uint32_t)(t * 64 + 32 * qb + key + off);
        const DropWords dw = D == 64 ? dropout_words(ahead, seed_lo, seed_hi, query) : dropout_words(seed_lo, seed_hi, bhq, query, (uint32_t)(2 * (kw >> 5) + quarter));
        const uint32_t sel1 = (ln & 1) ? 0x03070105u : 0x06020400u, sel2 = (ln & 2) ? 0x03020706u : 0x05040100u;
        u32x4 w;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            uint32_t x = dw.w[g];
            x = __builtin_amdgcn_perm((uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xf, 0xf, true), x, sel1);
            w[g] = __builtin_amdgcn_perm((uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xf, 0xf, true), x, sel2);
        }
        *(__attribute__((address_space(3))) u32x4 *)(uintptr_t)(drop_lds + 16u * (uint32_t)ln) = w;
        __builtin_amdgcn_sched_barrier(0);
    };

    // A tile: its 64 queries, 32 (block qb) at a time, against this wave's 32 keys.  Per block four products: S = Q K^T, dP =
    // dO V^T, dV^T += dO^T P, dK^T += Q^T dS, NF matrix instructions that each read one fragment of the tile from LDS.
    // The fragments are read PD instructions ahead, across the blocks of the tile, and what the vector ALU does (P from S, dS
    // from P and dP) is dealt in pairs of elements over the instructions behind the one that its inputs come from.
    // (What bounds it: the dependent chain of a block on two waves per SIMD, then the power cap -- on zeros instead of unit
    // normal values the 64-wide kernel takes 232 us instead of 353.  Left to the compiler every read was waited for at once.
    // B2 H16 S4096 without a mask, D64 fp16 397 us before, 353 now; whole backward passes: B2 H32/8 S4096 D128 bf16 882 / 819,
    // B2 H32 S8192 D128 3270 / 3010, B4 H16 S1000 D128 96 / 90, B8 H16 S1000 D64 100 / 93.)
    auto whole_tile = [&](bool edge, float slope_l2, uint32_t bhq, int t) __attribute__((always_inline)) {
        constexpr int q_tile = 0, g_tile = TILEB, NH = 2 * KS + 4 * DB, NF = 2 * NH;
        u32x4 fr[NF], fb[NF];
        auto fetch = [&](int n) __attribute__((always_inline)) {
            const int qb = n / NH, i = n % NH;
            if (i < KS) {
                fr[n] = rd.rows(q_tile, i, qb);
                if (i >= KS - PARKED) fb[n] = parked(i - (KS - PARKED));
            } else if (i < 2 * KS) {
                fr[n] = rd.rows(g_tile, i - KS, qb);
            } else {
                const int m = (i - 2 * KS) % (2 * DB);
                fr[n] = rd.transposed(i < 2 * KS + 2 * DB ? g_tile : q_tile, 2 * qb + m / DB, m % DB);
            }
        };
        f32x16 sx, dp;
        // the accumulators of block qb start from what the row's exponent and row sum subtract: -lse / scale, -delta.  With
        // dropout from (ln(1 / (1 - p)) - lse) / scale and -delta (1 - p): P then carries the factor 1 / (1 - p) that both dV
        // and dS need before they are rounded to the storage type (a factor at the end would leave fp16's subnormal range
        // 1 / (1 - p) times larger: dK and dQ at p = 0.9, dO of 1e-3, nine times as far off)
        auto start = [&](f32x16 &acc, int qb, uint32_t at) __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const u32x4 w = lds_read_b128(stat_addr + at + (uint32_t)(32 * qb + 8 * g) * 4u);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[4 * g + e] = as_f32(w[e]);
            }
        };
        start(sx, 0, 0);
#pragma unroll
        for (int n = 0; n < PD; ++n) fetch(n);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
            if (DROPOUT) draw(bhq, t, qb);
            const int n0 = qb * NH;
#pragma unroll
            for (int s = 0; s < KS; ++s) {                                   // S = Q K^T: rows = queries, column (lane) = key
                const int n = n0 + s;
                if (n + PD < NF) fetch(n + PD);
                sx = N::mfma(fr[n], s >= KS - PARKED ? fb[n] : kf[s], sx);
                if (s == KS - 2) { if (DROPOUT) dp = zero16(); else start(dp, qb, 256u); }
                __builtin_amdgcn_sched_barrier(0);
            }
            const int first = t * 64 + 32 * qb + 4 * half;                      // query of accumulator row 0 on this lane
            if (MASKED && edge) {            // wave-uniform; a masked score becomes -inf and its P exactly 0
                int hi = my_k + Rq, lo = my_k - Lq - first;                      // visible: lo <= 8*(r/4) + r%4 <= hi
                if (GENERAL && hi > S - 1) hi = S - 1;
                hi -= first;
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (8 * (r >> 2) + (r & 3) > hi || 8 * (r >> 2) + (r & 3) < lo) sx[r] = -INFINITY;
            }
            // accumulator row r is query 32*qb + 8*(r/4) + 4*half + r%4 of the tile
            uint32_t kept[4];                // dropout: byte e of word g belongs to row 4 g + e
            if (DROPOUT) {
                const int ln = lane_here(), key = ln & 31;
                const uint32_t src = drop_lds + (uint32_t)(((key >> 2) & 1) * 512 + (ln >> 5) * 64 + (key & 3) * 16 + (key >> 3) * 4);
#pragma unroll
                for (int g = 0; g < 4; ++g) kept[g] = *(const __attribute__((address_space(3))) uint32_t *)(src + 128u * g);
            }
            auto keeps = [&](int r) __attribute__((always_inline)) { return ((kept[r >> 2] >> (8 * (r & 3))) & 255u) >= a.drop_threshold; };
            uint32_t pp[8], ds[8];
            // rows 2 i and 2 i + 1: P, kept in fp32 in sx for dS, and what multiplied V
            auto p_pair = [&](int i) __attribute__((always_inline)) {
                float pd[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int r = 2 * i + e;
                    float x = sx[r] * c;
                    if (ALIBI) x = __builtin_fmaf(-slope_l2, __builtin_fabsf((float)(first + 8 * (r >> 2) + (r & 3) + off - my_k)), x);
                    sx[r] = __builtin_amdgcn_exp2f(x);
                    pd[e] = !DROPOUT || keeps(r) ? sx[r] : 0.0f;
                }
                pp[i] = N::pack2(pd[0], pd[1]);
                asm volatile("" : "+v"(pp[i]));
            };
            f32x4 del;
            auto ds_pair = [&](int i) __attribute__((always_inline)) {
                float v[2];
                if (DROPOUT && i % 2 == 0) {
                    const u32x4 w = lds_read_b128(stat_addr + 256u + (uint32_t)(32 * qb + 4 * i) * 4u);
#pragma unroll
                    for (int e = 0; e < 4; ++e) del[e] = as_f32(w[e]);
                }
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int r = 2 * i + e;
                    float dpr = dp[r];
                    if (DROPOUT) dpr = (keeps(r) ? dpr : 0.0f) + del[r & 3];       // (in units of 1 / (1 - p), the factor that P has)
                    v[e] = sx[r] * dpr;
                }
                ds[i] = N::pack2(v[0], v[1]);     // dS, same operand order
                asm volatile("" : "+v"(ds[i]));
            };
            // dP (KS instructions) with P pairs from its second on; dV (2 DB) with the P pairs that are left and, from its
            // second on, dS pairs; dK with the rest.  A pair is ready in front of the instruction that reads it: the 16-query
            // slice h2 of P or dS needs the pairs 4 h2 .. 4 h2 + 3.
            constexpr int P_IN_DP = 6;
            int np = 0, nd = 0;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int n = n0 + KS + s;
                if (n + PD < NF) fetch(n + PD);
                dp = N::mfma(fr[n], vf[s], dp);
                const int upto = s * P_IN_DP / (KS - 1);
#pragma unroll
                for (int i = np; i < upto; ++i) p_pair(i);
                np = upto;
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int m = 0; m < 2 * DB; ++m) {                // dV^T += dO^T P
                const int n = n0 + 2 * KS + m, h2 = m / DB;
                if (n + PD < NF) fetch(n + PD);
                const u32x4 bfrag = {pp[4 * h2], pp[4 * h2 + 1], pp[4 * h2 + 2], pp[4 * h2 + 3]};
                dv[m % DB] = N::mfma(fr[n], bfrag, dv[m % DB]);
                if (m == 0)
#pragma unroll
                    for (int i = np; i < 8; ++i) p_pair(i);
                const int upto = m * 6 / (2 * DB - 1);
#pragma unroll
                for (int i = nd; i < upto; ++i) ds_pair(i);
                nd = upto;
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int m = 0; m < 2 * DB; ++m) {                // dK^T += Q^T dS
                const int n = n0 + 2 * KS + 2 * DB + m, h2 = m / DB;
                if (n + PD < NF) fetch(n + PD);
                const u32x4 bfrag = {ds[4 * h2], ds[4 * h2 + 1], ds[4 * h2 + 2], ds[4 * h2 + 3]};
                dk[m % DB] = N::mfma(fr[n], bfrag, dk[m % DB]);
                if (m == 0)
#pragma unroll
                    for (int i = nd; i < 8; ++i) ds_pair(i);
                if (m == 1 && qb == 0) start(sx, 1, 0);       // (P has been used)
                __builtin_amdgcn_sched_barrier(0);
            }
            if (WRITE_DS) {
                // Block (32-query block 2t + qb, this wave's 32-key block) of dS, 2 KiB, as the registers hold it: this
                // lane's key against the queries 8g + 4*half + 0..3, g = 0..3.  Two store instructions of 1 KiB each,
                // lane l writing bytes 16 l .. 16 l + 15 of its KiB: queries of g = 0, 1 in the first, g = 2, 3 in the second.
                // (bhq: the QUERY head, batch * H + head; the blocks of the query heads that share this K/V head are apart)
                const long long block = (long long)(bhq - (uint32_t)(a.head0 * G)) * fa_ds_blocks_per_head(S) + fa_ds_block_index(S, 2 * t + qb, kw >> 5);
                // (Inline assembly: the block's address stays in two scalar registers and the lane's offset in one
                // vector register that lives for these two instructions only -- as a 64-bit vector address it cost
                // the registers that made the compiler spill inside the tile loop, and every reload from scratch
                // memory there waits for all tile loads in flight.  Streaming stores: the blocks are read once, by
                // another kernel, and should not displace the walked tiles from L2.  The wait states cover the rule
                // that a store of more than 8 bytes must not be followed at once by a write of its data registers.)
                const uint64_t dst = (uint64_t)(reinterpret_cast<char *>(a.ds_blocks) + block * kDsBlockBytes);
                const uint64_t ub = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(dst >> 32)) << 32) |
                                    (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)dst);
                const uint32_t voff = 16u * __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
                u32x4 w0 = {ds[0], ds[1], ds[2], ds[3]}, w1 = {ds[4], ds[5], ds[6], ds[7]};
                // (general lengths: a lane whose key lies past the end has worked on a copy of the last key; what the
                // query-owning kernel multiplies with the padding rows of its last key tile must be zero)
                if (GENERAL && my_k >= Sk) { w0 = u32x4{0, 0, 0, 0}; w1 = u32x4{0, 0, 0, 0}; }
                asm volatile("global_store_dwordx4 %0, %1, %3 nt\n\tglobal_store_dwordx4 %0, %2, %3 offset:1024 nt\n\ts_nop 1"
                             :: "v"(voff), "v"(w0), "v"(w1), "s"(ub) : "memory");
            }
        }
    };

    if (t0 <= t1) {
        // from the last query tile down to the diagonal: every workgroup of a head then starts on the same tile
        // and the ones that run together keep reading the same tiles out of L2; then the next head of the group
        // (head, tile) pairs are fetched two ahead, as in fa_bwd_dq
        // (shares: from pair `walk_from` of the walk, `walk_pairs` of them)
        const int per_head = t1 - t0 + 1;
        const int first_g = SHARES ? walk_from / per_head : 0, first_t = SHARES ? t1 - (walk_from - first_g * per_head) : t1;
        int pairs_left = SHARES ? walk_pairs : G * per_head;    // (WRITE_DS) pairs still to come
        int ig = first_g, it = first_t;                         // the next pair to fetch
        auto issue_next = [&](int stage) __attribute__((always_inline)) {
            issue(ig, it, stage);
            if (--it < t0) {
                it = t1; ++ig;
                if (STRIDES && ig < G) walk_head(ig);
            }
        };
        if (STRIDES) walk_head(first_g);
        issue_next(0);
        if (SHARES ? pairs_left > 1 : ig < G) issue_next(1);
        // (read while K and V are on their way, not behind the wait for them)
        uint32_t tiny_scale = __builtin_bit_cast(uint32_t, a.key_scale) ^ __builtin_bit_cast(uint32_t, a.scale);
        asm volatile("" : "+s"(tiny_scale));
        wait_vm<0>();
#pragma unroll
        for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(kf[s]), "+v"(vf[s]));
        if (__builtin_expect(tiny_scale != 0, 0)) {         // (see FaBwdArgs)
#pragma unroll
            for (int s = 0; s < KS; ++s)
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint32_t two = kf[s][w];
                    kf[s][w] = N::pack2(storage_to_f32<BF16>((uint16_t)(two & 0xffffu)) * kTinyScaleKeys, storage_to_f32<BF16>((uint16_t)(two >> 16)) * kTinyScaleKeys);
                }
        }
        // from here on the parked fragments live in LDS, and their registers are free
        // (one plane of 16 bytes per thread for every parked fragment: consecutive lanes, consecutive 16 bytes)
#pragma unroll
        for (int i = 0; i < PARKED; ++i) *(__attribute__((address_space(3))) u32x4 *)(uintptr_t)(park_addr + kParkPlane * i) = kf[KS - PARKED + i];
        int stage = 0;
        // WRITE_DS: the dS stores this wave made in the last two iterations, and the pairs still to come.  The next
        // pair is then requested in front of an iteration's work instead of behind it.
        int st1 = 0, st2 = 0;
        constexpr bool TOP = WRITE_DS;
        for (int g = first_g, t_from = first_t; SHARES ? pairs_left > 0 : g < G; ++g, t_from = t1) {
            float slope_l2 = 0.0f;
            if (ALIBI) slope_l2 = a.alibi[hk * G + g] * kLog2e;
            for (int t = t_from; t >= t0 && (!SHARES || pairs_left > 0); --t) {
                const int next = stage == NSTG - 1 ? 0 : stage + 1, prev = stage == 0 ? NSTG - 1 : stage - 1;
                const bool more = t - 1 >= t0 || g + 1 < G;
                --pairs_left;
                if (WRITE_DS) {
                    // This pair has landed when at most what was issued behind it is outstanding (memory operations
                    // complete in the order they were issued): the loads of the pairs requested since, and the dS
                    // stores made since.  Requests at the top of an iteration put a pair's loads in front of that
                    // iteration's stores, so a store that takes long to be acknowledged holds up no load needed now.
                    const int loads = wave < 2 ? 2 * IPW + 1 : 2 * IPW;     // waves 0 and 1 also fetch lse / delta
                    wait_vm_upto((pairs_left > 0 ? loads : 0) + st1 + st2);
                } else if (more) {                              // this pair has landed, the next may still be in flight
                    if (wave < 2) wait_vm<2 * IPW + 1>(); else wait_vm<2 * IPW>();     // waves 0 and 1 also fetch lse / delta
                } else wait_vm<0>();
                phase_barrier();
                if (TOP && (SHARES ? pairs_left > 1 : ig < G)) issue_next(prev);
                st2 = st1;
                st1 = (WRITE_DS && my_lo <= t && t <= my_hi) ? 4 : 0;
                if (my_lo <= t && t <= my_hi) {
                    const bool edge = MASKED && (fa_tile_class(64, Lq, Rq, kw, 32, t) == 1 || (GENERAL && (t + 1) * 64 > S));
                    const uint32_t bhq = (uint32_t)(b * a.H + hk * G + g);        // the head the forward keyed its dropout on
                    if (DROPOUT && D == 64 && bhq != ahead_of) {
                        ahead = dropout_ahead(a.seed_lo, a.seed_hi, bhq, (uint32_t)(2 * (kw >> 5) + half));
                        ahead_of = bhq;
                    }
                    whole_tile(edge, slope_l2, bhq, t);
                }
                if (!TOP && ig < G) issue_next(prev);
                rd.advance(next == 0 ? -(NSTG - 1) * STAGEB : STAGEB);
                stat_addr += next == 0 ? -(NSTG - 1) * STAGEB : STAGEB;
                stage = next;
            }
        }
    }
    // (the lane's row and column offset are derived again here, from the hardware's lane index and tied to this
    // place: taken from the values computed at the top, the compiler forms the store addresses there and keeps
    // them in registers, or in scratch memory, through the whole loop)
    int lane_e = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane_e));
    const int key_e = kw + (lane_e & 31), half_e = lane_e >> 5;
    int part_slot = -1;
    if (SHARES) {
        const FaBwdArgs &f = args_reloaded();
        const int share = fa_bwd_share_of((int)blockIdx.x, (int)gridDim.x), begin = fa_bwd_share_begin(share, (int)gridDim.x, f.walk_total);
        int head, kb, walk_begin, walk_len;
        fa_bwd_walk_at(share_at - 1, f.walk_head, G, S, Sk, f.R + off, f.L - off, &head, &kb, &walk_begin, &walk_len);
        if (begin > walk_begin || share_at < walk_begin + walk_len) part_slot = fa_bwd_part_slot(share, begin > walk_begin ? 1 : 0);
    }
    if (SHARES && part_slot >= 0) {
        // part of a walk: the fp32 sums as the registers hold them, 1 KiB per store instruction, for fa_bwd_add_parts
        if (active) {
            float *part = args_reloaded().partials + (size_t)part_slot * (2 * 256 * D) + wave * (32 * D) + 4 * lane_e;
#pragma unroll
            for (int i = 0; i < 4 * DB; ++i) {
                *reinterpret_cast<f32x4 *>(part + 256 * i) = f32x4{dk[i / 4][4 * (i % 4)], dk[i / 4][4 * (i % 4) + 1], dk[i / 4][4 * (i % 4) + 2], dk[i / 4][4 * (i % 4) + 3]};
                *reinterpret_cast<f32x4 *>(part + 256 * D + 256 * i) = f32x4{dv[i / 4][4 * (i % 4)], dv[i / 4][4 * (i % 4) + 1], dv[i / 4][4 * (i % 4) + 2], dv[i / 4][4 * (i % 4) + 3]};
            }
        }
    } else if (active && key_e < Sk) {
        uint16_t *dKh, *dVh;
        int dk_rs = D, dv_rs = D;
        if (STRIDES) {
            const FaBwdArgs &f = args_reloaded();
            dKh = head_ptr(f.dK, f.dk, b, hk); dVh = head_ptr(f.dV, f.dv, b, hk);
            dk_rs = f.dk.rs; dv_rs = f.dv.rs;
        } else {
            dKh = a.dK + (size_t)bhk * S * D; dVh = a.dV + (size_t)bhk * S * D;
        }
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                u32x2 wk, wv;
                wk[0] = N::pack2(dk[db][4 * g] * a.scale, dk[db][4 * g + 1] * a.scale);
                wk[1] = N::pack2(dk[db][4 * g + 2] * a.scale, dk[db][4 * g + 3] * a.scale);
                wv[0] = N::pack2(dv[db][4 * g], dv[db][4 * g + 1]);
                wv[1] = N::pack2(dv[db][4 * g + 2], dv[db][4 * g + 3]);
                *reinterpret_cast<u32x2 *>(dKh + (size_t)key_e * dk_rs + 32 * db + 8 * g + 4 * half_e) = wk;
                *reinterpret_cast<u32x2 *>(dVh + (size_t)key_e * dv_rs + 32 * db + 8 * g + 4 * half_e) = wv;
            }
    }
    }   // next work item
}

// ---------------------------------------------------------------------------------------------------------
// The five-product form (regular lengths in the reference's or a strided layout, no ALiBi).  fa_bwd_dq above and fa_bwd_dkdv each recompute S and dP: seven
// products for five.  Here fa_bwd_dkdv, which has every dS block in registers as the operand of dK += dS^T Q,
// also writes it out (WRITE_DS), and dQ = scale * dS K is one product over those blocks: every output element
// still has exactly one writer and the same inputs give the same bits.  The price is S*S_kv storage-type elements
// per head written once and read once, so this kernel is bound by HBM bandwidth, not by the matrix cores.
//
// fa_bwd_prepare: delta_i = sum_t dO_it O_it and the logsumexp, in the units that FaBwdArgs states, which fa_bwd_dkdv fetches per
// query tile (fa_bwd_dq writes them in the seven-product form).
// Bound by HBM: O and dO read once.  A workgroup takes kPrepareRows rows per thread of one head: the head is found once, by
// scalar arithmetic (one row per thread found it with two 64-bit divisions each), and a thread has the loads of all its rows
// in flight together.  B2 H32 S4096 D128 stored [B,S,H,D], 136 MB: 26.6 us before, 23.9 (5.7 TB/s) now; the whole backward
// pass there 862 / 857 us, B16 H16 S1024 D64 196.7 / 194.6, B4 H16 S2048 D64 152.3 / 149.5, B1 H32 S2048 D128 148.5 / 147.0.
// ---------------------------------------------------------------------------------------------------------
constexpr int kPrepareRows = 4;               // rows per thread
constexpr long long kPrepareGrid = 1 << 16;   // workgroups of a launch at most (far below the 2^32 threads a launch may hold); they walk what is beyond
constexpr int fa_bwd_prepare_rows(int D) { return kPrepareRows * (256 / (D / 8)); }       // rows per workgroup
template <bool BF16, int D, bool STRIDED>
__global__ void __launch_bounds__(256) fa_bwd_prepare(const FaBwdArgs a)
{
    constexpr int TPR = D / 8, STEP = 256 / TPR;  // threads per row, 16 bytes each; rows that the workgroup reads at a time
    const int S = a.S, pieces = (S + fa_bwd_prepare_rows(D) - 1) / fa_bwd_prepare_rows(D);
    // heads stored inside rows ([B,S,H,D]): neighbouring workgroups take neighbouring heads, as they lie in memory
    const bool heads_inside = STRIDED && a.o.hs < a.o.rs;
    const unsigned blocks = (unsigned)a.B * (unsigned)a.H * (unsigned)pieces;
    for (unsigned block = blockIdx.x; block < blocks; block += gridDim.x) {
    int b, h, piece;
    if (heads_inside) {
        b = (int)(block / (unsigned)(a.H * pieces));
        const int in_b = (int)(block - (unsigned)b * (unsigned)(a.H * pieces));
        piece = in_b / a.H;
        h = in_b - piece * a.H;
    } else {
        const int bh = (int)(block / (unsigned)pieces);
        piece = (int)(block - (unsigned)bh * (unsigned)pieces);
        b = bh / a.H;
        h = bh - b * a.H;
    }
    const long long row0 = ((long long)b * a.H + h) * S;
    const uint16_t *o_head = STRIDED ? head_ptr(a.O, a.o, b, h) : a.O + row0 * D, *g_head = STRIDED ? head_ptr(a.dO, a.dO_, b, h) : a.dO + row0 * D;
    const long long o_rs = STRIDED ? a.o.rs : D, g_rs = STRIDED ? a.dO_.rs : D;
    const int slot = (int)threadIdx.x % TPR, first = piece * fa_bwd_prepare_rows(D) + (int)threadIdx.x / TPR;
    u32x4 o[kPrepareRows], g[kPrepareRows];
#pragma unroll
    for (int n = 0; n < kPrepareRows; ++n) {
        const int i = first + n * STEP < S ? first + n * STEP : S - 1;
        o[n] = *reinterpret_cast<const u32x4 *>(o_head + i * o_rs + slot * 8);
        g[n] = *reinterpret_cast<const u32x4 *>(g_head + i * g_rs + slot * 8);
    }
    // the row's thread number n writes the row of step n
    const int mine = first + slot * STEP;
    const bool writes = slot < kPrepareRows && mine < S;
    const float l = writes ? a.lse[row0 + mine] : 0.0f;
    float delta = 0.0f;
#pragma unroll
    for (int n = 0; n < kPrepareRows; ++n) {
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const uint32_t ow = o[n][w], gw = g[n][w];
            sum += storage_to_f32<BF16>((uint16_t)(ow & 0xffffu)) * storage_to_f32<BF16>((uint16_t)(gw & 0xffffu));
            sum += storage_to_f32<BF16>((uint16_t)(ow >> 16)) * storage_to_f32<BF16>((uint16_t)(gw >> 16));
        }
#pragma unroll
        for (int m = 1; m < TPR; m <<= 1) sum += __shfl_xor(sum, m);
        if (slot == n) delta = sum;
    }
    if (writes) {
        a.delta[row0 + mine] = -delta / a.drop_scale;
        a.lse2[row0 + mine] = l == -INFINITY ? -INFINITY : (a.drop_log - l) / a.key_scale;
    }
    }
}

// The same for sequences of at most a quarter of such a workgroup's rows, whose heads would leave most of its threads without a
// row: rows of all heads one behind the other, one per group of threads.  us, a piece of one head per workgroup / this: D64
// B512 H16 S16 12.2 / 7.6, B2048 H16 S1 35.9 / 4.8, D128 B1024 H16 S8 21.9 / 13.5; B256 H32 S33 28.2 / 30.5, and at D64 B128 H16
// S64 the backward pass 50.8 / 51.3.
template <bool BF16, int D, bool STRIDED>
__global__ void __launch_bounds__(256) fa_bwd_prepare_short(const FaBwdArgs a)
{
    constexpr int TPR = D / 8;                    // threads per row, 16 bytes each
    const long long n_rows = (long long)a.B * a.H * a.S;
    const int c = (int)threadIdx.x % TPR * 8;
    for (long long first = (long long)blockIdx.x * (256 / TPR); first < n_rows; first += (long long)gridDim.x * (256 / TPR)) {
    const long long row = first + (int)threadIdx.x / TPR, r = row < n_rows ? row : n_rows - 1;
    const uint16_t *o_row = a.O + r * D, *g_row = a.dO + r * D;
    if (STRIDED) {                                // row r of the [B,H,S] order, wherever the tensors keep it
        const long long bh = r / a.S;
        const int i = (int)(r - bh * a.S), b = (int)(bh / a.H), h = (int)(bh - (long long)b * a.H);
        o_row = head_ptr(a.O, a.o, b, h) + (long long)i * a.o.rs;
        g_row = head_ptr(a.dO, a.dO_, b, h) + (long long)i * a.dO_.rs;
    }
    const u32x4 o = *reinterpret_cast<const u32x4 *>(o_row + c), g = *reinterpret_cast<const u32x4 *>(g_row + c);
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const uint32_t ow = o[w], gw = g[w];
        sum += storage_to_f32<BF16>((uint16_t)(ow & 0xffffu)) * storage_to_f32<BF16>((uint16_t)(gw & 0xffffu));
        sum += storage_to_f32<BF16>((uint16_t)(ow >> 16)) * storage_to_f32<BF16>((uint16_t)(gw >> 16));
    }
#pragma unroll
    for (int m = 1; m < TPR; m <<= 1) sum += __shfl_xor(sum, m);
    if (row < n_rows && c == 0) {
        const float l = a.lse[row];
        a.delta[row] = -sum / a.drop_scale;
        a.lse2[row] = l == -INFINITY ? -INFINITY : (a.drop_log - l) / a.key_scale;
    }
    }
}

// The parts of the walks that fa_bwd_dkdv cut between its workgroups' shares: dK and dV of such a key block are the sums
// of its parts, added in the order of the walk (the same bits every run).  Workgroup (share c, wave w, dK or dV): the 32
// keys of wave w in the block that the boundary in front of share c cuts, if it cuts one and is the first to do so.
// Bound by HBM: 256 KB per part at head dimension 128, read once; a thread has all its slots of a part in flight at once
// (one slot after the other, the 57 parts of B1 H8/1 S2048's first block took 0.7 ms).
template <bool BF16, int D, bool STRIDED>
__global__ void __launch_bounds__(256) fa_bwd_add_parts(const FaBwdArgs a, int n_shares)
{
    constexpr int SLOTS = 8 * D / 256;            // 16-byte slots per thread: 32 keys x D floats over 256 threads
    const int share = (int)blockIdx.x / (2 * kBwdWaves) + 1, wave = (int)blockIdx.x / 2 % kBwdWaves, which = (int)blockIdx.x % 2;
    const int S = a.S, G = STRIDED ? a.H / a.Hk : 1;
    const int cut = fa_bwd_share_begin(share, n_shares, a.walk_total);
    int bhk, kblock, begin, len;
    fa_bwd_walk_at(cut, a.walk_head, G, S, S, a.R, a.L, &bhk, &kblock, &begin, &len);
    if (cut == begin || fa_bwd_share_begin(share - 1, n_shares, a.walk_total) > begin) return;
    int last = share;                             // the share that holds the walk's end
    while (fa_bwd_share_begin(last + 1, n_shares, a.walk_total) < begin + len) ++last;
    constexpr size_t PART = 2 * 256 * D;
    const float *src = a.partials + (size_t)which * (256 * D) + wave * (32 * D) + 4 * (int)threadIdx.x;
    f32x4 sum[SLOTS];
#pragma unroll
    for (int n = 0; n < SLOTS; ++n) sum[n] = *reinterpret_cast<const f32x4 *>(src + fa_bwd_part_slot(share - 1, 0) * PART + 1024 * n);
#pragma unroll 4
    for (int s = share; s <= last; ++s)
#pragma unroll
        for (int n = 0; n < SLOTS; ++n) sum[n] += *reinterpret_cast<const f32x4 *>(src + fa_bwd_part_slot(s, 1) * PART + 1024 * n);
    bhk += a.head0;
    const int b = bhk / a.Hk, hk = bhk - b * a.Hk;
    uint16_t *out = which == 0 ? (STRIDED ? head_ptr(a.dK, a.dk, b, hk) : a.dK + (size_t)bhk * S * D)
                               : (STRIDED ? head_ptr(a.dV, a.dv, b, hk) : a.dV + (size_t)bhk * S * D);
    const int rs = STRIDED ? (which == 0 ? a.dk.rs : a.dv.rs) : D, lane = (int)threadIdx.x % 64, key = kblock * 256 + wave * 32 + (lane & 31);
    const float scale = which == 0 ? a.scale : 1.0f;
    if (key >= S) return;
#pragma unroll
    for (int n = 0; n < SLOTS; ++n) {
        const int i = n * 4 + (int)threadIdx.x / 64, col = 32 * (i / 4) + 8 * (i % 4) + 4 * (lane >> 5);
        u32x2 w;
        w[0] = Num<BF16>::pack2(sum[n][0] * scale, sum[n][1] * scale);
        w[1] = Num<BF16>::pack2(sum[n][2] * scale, sum[n][3] * scale);
        *reinterpret_cast<u32x2 *>(out + (size_t)key * rs + col) = w;
    }
}

// dQ^T += K^T dS^T over the dS blocks fa_bwd_dkdv<WRITE_DS> wrote.  A workgroup owns 32 NW queries (NW waves x one
// 32-query block, lane = query) and walks the key tiles of its visible range.  LDS stage: the K tile (read
// transposed, as in fa_bwd_dq) and, per wave, the two 2 KiB dS blocks of its query block against the tile's keys,
// fetched by that wave alone.  A block comes in as it lies in memory except that the 64-byte groups of four keys
// are XOR-permuted among the four 512-byte planes, so that the transposing read of a half-wave -- four keys, all
// 32 queries, i.e. one group in each plane -- touches every LDS bank once.
template <bool BF16, int D, bool MASKED, int LAYOUT, int NW, int NST>
__global__ void __launch_bounds__(NW * 64, 2) fa_bwd_dq_from_ds(const FaBwdArgs a)
{
    constexpr bool STRIDED = LAYOUT >= 1, GENERAL = LAYOUT == 2;      // (general: any length S = S_kv)
    typedef Num<BF16> N;
    typedef TileReader<D> Reader;
    typedef TileLoader<D, NW> Loader;
    constexpr int DB = Reader::DB, TILEB = Loader::TILEB, IPW = Loader::IPW;
    constexpr int WAVE_DS = 2 * kDsBlockBytes;                 // a wave's two blocks of a key tile
    constexpr int STAGEB = TILEB + NW * WAVE_DS, ROWS = 32 * NW;
    constexpr int AHEAD = NST - 1;                             // tiles are requested this many ahead
    static_assert((AHEAD - 1) * (IPW + 4) <= 16, "more requests in flight than wait_vm_upto counts");
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int S = a.S;
    const int n_qblocks = (S + ROWS - 1) / ROWS;
    const int group = STRIDED ? a.H / a.Hk : 1, heads_q = a.heads * group, head0_q = a.head0 * group;
    const long long n_items = (long long)heads_q * n_qblocks;
    for (int pass = 0;; ++pass) {
    const long long item = (long long)pass * gridDim.x + ((pass & 1) ? gridDim.x - 1 - blockIdx.x : blockIdx.x);
    if (item >= n_items) break;
    if (pass > 0) __syncthreads();          // (the LDS stages: other waves may still be reading the last tile)
    int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane));
    const int half = lane >> 5, l32 = lane & 31, l16 = lane & 15;
    int bh, qblock;
    fa_item_decode(item, heads_q, n_qblocks, MASKED ? 1 : 0, &bh, &qblock);
    bh += head0_q;
    const uint16_t *Kh = a.K + (size_t)bh * S * D;
    uint16_t *dQh = a.dQ + (size_t)bh * S * D;
    int k_rs = D, dq_rs = D;
    if (STRIDED) {                                 // (bh counts query heads; the K/V head of query head h is h / (H / Hk))
        const int b = bh / a.H, h = bh - b * a.H;
        Kh = head_ptr(a.K, a.k, b, h / group);
        dQh = head_ptr(a.dQ, a.dq, b, h);
        k_rs = a.k.rs; dq_rs = a.dq.rs;
    }
    const int q0 = qblock * ROWS, qw = q0 + wave * 32;
    const bool active = qw < S;                    // the last block may own fewer rows
    int t0, t1, my_lo = 1, my_hi = 0;
    fa_tile_range(S, 64, a.L, a.R, q0, S - q0 < ROWS ? S - q0 : ROWS, &t0, &t1);
    if (active) fa_tile_range(S, 64, a.L, a.R, qw, GENERAL && S - qw < 32 ? S - qw : 32, &my_lo, &my_hi);
    // this head's dS blocks; this wave reads those of query block qw / 32
    const char *ds_head = reinterpret_cast<const char *>(a.ds_blocks) + (long long)(bh - head0_q) * fa_ds_blocks_per_head(S) * kDsBlockBytes;
    const int my_qb = active ? qw >> 5 : 0;

    Reader rd; rd.init(lane, lds0);
    Loader ldk; ldk.init(wave, lane, k_rs * 2);
    // Source of the 16 bytes lane l brings in with instruction w (0, 1) of a block: LDS slot 64 w + l of the block
    // = plane p = 2 w + l / 32, position l % 32; that position holds key ((l % 32 / 4) ^ p) * 4 + l % 4, which lies
    // in memory at 1 KiB * w + 512 * (l / 32) + 16 * key.
    uint32_t ds_src[2];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const int p = 2 * w + half, key = ((((l32 >> 2) ^ p) & 7) << 2) | (l32 & 3);
        ds_src[w] = (uint32_t)(1024 * w + 512 * half + 16 * key);
    }
    // Transposing read of a B operand (lane = query l32, keys 16 t2 + 4 half + {0..3} and + 8 of a block): the lane
    // addresses the 8 bytes that hold queries 16 (l32 / 16) + 4 (l16 % 4) .. + 3 of key 16 t2 + 8 hi + 4 half + l16 / 4.
    // Those four queries are quad 4 (l32 / 16) + l16 % 4 = 2 g + h of the block, written by fa_bwd_dkdv's lane
    // (key, half h) as its g-th pair of words: plane p = 2 (g / 2) + h, 16-byte slot of the key, byte 8 (g % 2).
    uint32_t ds_rd[2];
    {
        const int quad = 4 * (l32 >> 4) + (l16 & 3), g = quad >> 1, hq = quad & 1;
        const int p = 2 * (g >> 1) + hq;
#pragma unroll
        for (int hi = 0; hi < 2; ++hi)
            ds_rd[hi] = lds0 + TILEB + wave * WAVE_DS +
                        (uint32_t)(512 * p + ((((2 * hi + half) ^ p) & 3) << 6) + 16 * (l16 >> 2) + 8 * (g & 1));
    }
    auto issue = [&](int tile, int stage) __attribute__((always_inline)) {
        const uint32_t base = lds0 + stage * STAGEB;
        if (GENERAL && (tile + 1) * 64 > S) ldk.load_ragged(Kh + (size_t)tile * 64 * k_rs, base, S - tile * 64, k_rs * 2);
        else ldk.load(Kh + (size_t)tile * 64 * k_rs, base);
        if (my_lo <= tile && tile <= my_hi) {
            const char *src = ds_head + fa_ds_block_index(S, my_qb, 2 * tile) * kDsBlockBytes;      // (and its neighbour 2 tile + 1)
            const uint32_t dst = base + TILEB + wave * WAVE_DS;
#pragma unroll
            for (int n = 0; n < 4; ++n)         // block 2 tile (n = 0, 1), block 2 tile + 1 (n = 2, 3)
                dma_16_stream(src, (uint32_t)((n >> 1) * kDsBlockBytes) + ds_src[n & 1], dst + n * 1024);
        }
    };
    // the blocks fa_bwd_dkdv wrote: its wave with the 32 keys from `key0` on visits the query tiles of this range
    auto block_written = [&](int key0) __attribute__((always_inline)) {
        if (GENERAL && key0 >= S) return false;          // (a wave of the key-owning kernel without any key)
        int lo, hi;
        fa_tile_range(S, 64, a.R, a.L, key0, GENERAL && S - key0 < 32 ? S - key0 : 32, &lo, &hi);
        return lo <= (qw >> 6) && (qw >> 6) <= hi;
    };

    f32x16 dq[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) dq[db] = zero16();

    if (t0 <= t1) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (t0 + u <= t1) issue(t0 + u, u);
        int stage = 0;
        for (int t = t0; t <= t1; ++t) {
            const int next = stage == NST - 1 ? 0 : stage + 1;
            // tile t has landed when at most the requests of the tiles behind it are outstanding
            int later = 0;
#pragma unroll
            for (int u = 1; u < AHEAD; ++u)
                if (t + u <= t1) later += my_lo <= t + u && t + u <= my_hi ? IPW + 4 : IPW;
            wait_vm_upto(later);
            phase_barrier();
            if (my_lo <= t && t <= my_hi) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    if ((MASKED || GENERAL) && !block_written(64 * t + 32 * kb)) continue;       // wave-uniform
#pragma unroll
                    for (int t2 = 0; t2 < 2; ++t2) {
                        const u32x2 lo = lds_read_tr(ds_rd[0] + (uint32_t)(kb * kDsBlockBytes + 256 * t2));
                        const u32x2 hi = lds_read_tr(ds_rd[1] + (uint32_t)(kb * kDsBlockBytes + 256 * t2));
                        const u32x4 bfrag = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
                        for (int db = 0; db < DB; ++db) dq[db] = N::mfma(rd.transposed(0, 2 * kb + t2, db), bfrag, dq[db]);
                    }
                }
            }
            if (t + AHEAD <= t1) issue(t + AHEAD, stage == 0 ? NST - 1 : stage - 1);       // (the stage tile t - 1 was read from)
            const int delta = next == 0 ? -(NST - 1) * STAGEB : STAGEB;
            rd.advance(delta);
            ds_rd[0] += delta; ds_rd[1] += delta;
            stage = next;
        }
    }
    if (active && (!GENERAL || qw + l32 < S)) {
        const int my_q = qw + l32;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                u32x2 w;
                w[0] = N::pack2(dq[db][4 * g] * a.scale, dq[db][4 * g + 1] * a.scale);
                w[1] = N::pack2(dq[db][4 * g + 2] * a.scale, dq[db][4 * g + 3] * a.scale);
                *reinterpret_cast<u32x2 *>(dQh + (size_t)my_q * dq_rs + 32 * db + 8 * g + 4 * half) = w;
            }
    }
    }   // next work item
}

template <bool BF16, int D, bool MASKED, int LAYOUT, bool ALIBI, bool DROPOUT>
hipError_t launch_bwd(const FaBwdArgs &a_in, int compute_units, hipStream_t stream, bool configure_only = false)
{
    constexpr int TILEB = 64 * D * 2;
    FaBwdArgs a = a_in;
    const int all_heads = a.B * a.Hk, group = a.Hk > 0 ? a.H / a.Hk : 1;
    a.head0 = 0;
    a.heads = all_heads;
    const int smem_dq = kBwdStages * 2 * TILEB;
    auto smem_kv = [](int waves) { return kBwdStages * (2 * TILEB + 512) + (DROPOUT ? waves * 1024 : 0) + fa_bwd_parked(D, DROPOUT) * 16 * waves * 64; };
    const int smem_dkdv = smem_kv(kBwdWaves);
    // The key-owning kernel of the five-product form, head dimension 64: four waves, 128 keys, two workgroups per CU, whose
    // waves wait at barriers of their own.  Backward pass, four waves against eight: causal B8 H16 S1000 94 against 97 us, B4
    // H16 S2048 150 / 153, window 700 B1 H32 S8192 249 / 254, no mask B16 H16 S512 96 / 100, without a mask and ALiBi B23 H32
    // S256 90 / 95; B6 H32/8 S4096 1698 / 1670 and B32 H8 S300 45 / 42 the other way.
    constexpr int NWK = D == 64 ? 4 : kBwdWaves, KEYS_K = 32 * NWK, GROUPS_K = kBwdWaves / NWK;
    const int smem_dkdv_ds = smem_kv(NWK);
    constexpr bool EITHER = LAYOUT == 1 && D == 128 && DROPOUT && MASKED;        // the key-owning kernel is built with the item loop and without
    auto kq = fa_bwd_dq<BF16, D, MASKED, LAYOUT, ALIBI, DROPOUT>;
    auto kkv = fa_bwd_dkdv<BF16, D, MASKED, LAYOUT, ALIBI, DROPOUT>;
    // the five-product form: regular lengths (the reference's layout or a strided one) with dropout or ALiBi, any
    // length S = S_kv without them
    constexpr bool FIVE = LAYOUT <= 1 || (!ALIBI && !DROPOUT);
    constexpr int FL = FIVE ? LAYOUT : 0;
    constexpr bool CAN_SHARE = FIVE && fa_bwd_can_share(D, DROPOUT);
    // the query-owning kernel from dS blocks: 8 waves (256 queries) and three LDS stages, or 4 waves and four stages, or, at
    // head dimension 64, 4 waves and three stages, two workgroups per CU
    auto smem_dq_ds = [](int waves, int stages) { return stages * (TILEB + waves * 2 * kDsBlockBytes); };
    // the LDS opt-in is per (instantiation, device) and is made once, not on every launch
    static std::atomic<unsigned long long> configured{0ull};
    const unsigned long long dev_bit = 1ull << fa_launch_device();
    if (!(configured.load(std::memory_order_relaxed) & dev_bit)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kq), hipFuncAttributeMaxDynamicSharedMemorySize, smem_dq);
        if (e != hipSuccess) return e;
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(kkv), hipFuncAttributeMaxDynamicSharedMemorySize, smem_dkdv);
        if (e != hipSuccess) return e;
        if constexpr (EITHER) {
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(fa_bwd_dkdv<BF16, D, MASKED, LAYOUT, ALIBI, DROPOUT, false, false, kBwdWaves, false>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, smem_dkdv);
            if (e != hipSuccess) return e;
        }
        if constexpr (FIVE) {
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(fa_bwd_dkdv<BF16, D, MASKED, FL, ALIBI, DROPOUT, true, false, NWK>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, smem_dkdv_ds);
            if (e != hipSuccess) return e;
            if constexpr (CAN_SHARE) {
                e = hipFuncSetAttribute(reinterpret_cast<const void *>(fa_bwd_dkdv<BF16, D, MASKED, FL, ALIBI, DROPOUT, true, true>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, smem_dkdv);
                if (e != hipSuccess) return e;
            }
            if constexpr (D == 128 || MASKED) {
                e = hipFuncSetAttribute(reinterpret_cast<const void *>(fa_bwd_dq_from_ds<BF16, D, MASKED, FL, 8, 3>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, smem_dq_ds(8, 3));
                if (e != hipSuccess) return e;
            }
            if constexpr (D == 64) {
                e = hipFuncSetAttribute(reinterpret_cast<const void *>(fa_bwd_dq_from_ds<BF16, D, MASKED, FL, 4, 3>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, smem_dq_ds(4, 3));
                if (e != hipSuccess) return e;
            }
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(fa_bwd_dq_from_ds<BF16, D, MASKED, FL, 4, 4>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, smem_dq_ds(4, 4));
            if (e != hipSuccess) return e;
        }
        configured.fetch_or(dev_bit, std::memory_order_relaxed);
    }
    if (configure_only) return hipSuccess;     // (fa_init: the opt-in alone, so that no launch inside a stream capture makes it)
    // Masked problems with between one and sixteen items per compute unit: a resident grid (one workgroup per CU,
    // 8 waves at two per SIMD) walks the list as a snake, which pairs every long item with a short one; otherwise
    // one workgroup per item, handed out by the hardware as CUs free up.  Causal fp16, snake against dispatch:
    // B1 H32 S4096 D128 477 against 639 us, B1 H64 S2048 D128 273 against 370, B4 H16 S2048 D64 160 against 221,
    // B8 H32 S1024 D64 194 against 237, c3's shape 3.59 against 3.64 ms; without a mask (items all alike) the
    // hardware's order is 1-7 % ahead.
    // (a window of at most half the length leaves the items alike too: c4's shape 1.14 ms in the hardware's order,
    // 1.16 as a snake)
    const unsigned resident = (unsigned)compute_units;
    // (the general instantiations always carry the mask code: without a bound on either side, L = R = S + S_kv, their
    // items are alike as well)
    // (The 128-wide strided and general instantiations are launched one workgroup per item only: with the item loop
    // around them they spill ten times as much, and a reload inside the tile loop waits for every tile load in
    // flight: c3's shape stored [B,S,H,D] 4.1 ms against 3.8.  The 64-wide ones have the registers for the loop, and the
    // strided ones with dropout, which serve the reference's layout too, spill outside the tile loop only: with the loop where
    // the grid is a snake, without it elsewhere.  Seven products, p = 0.1, one item per workgroup / snake, us: causal B4 H16
    // S2048 D128 424 / 310, B1 H32 S4096 740 / 562, B8 H32 S512 151 / 134; with the loop where it is not needed B1 H16 S1024
    // 115 / 120, window 1000 B1 H32 S8192 646 / 671.)
    // (The kernels of the five-product form have the loop in every layout: the key-owning one keeps K^T fragments in LDS and
    // spills at most 24 bytes with it, 84 with dropout, which are touched per item or walked head and not per tile.)
    const bool uneven_items = MASKED && fa_bwd_uneven(a.S, a.Sk, a.L, a.R);
    const bool uneven = (LAYOUT == 0 || D == 64 || EITHER) && uneven_items;
    auto grid_if = [&](bool snake, long long items, unsigned groups_per_cu = 1u) {
        const unsigned g = (unsigned)items, all = groups_per_cu * resident;
        return (snake && g > all && g < 16u * all) ? all : g;
    };
    auto grid_for = [&](long long items) { return grid_if(uneven, items); };
    if constexpr (FIVE) {
        if (a.ds_blocks != nullptr) {
            // delta and the rescaled logsumexp, for all heads at once; then, for as many heads at a time as the
            // workspace holds dS blocks for: dK, dV and the dS blocks; dQ from the blocks
            constexpr int rows = fa_bwd_prepare_rows(D), short_rows = 256 / (D / 8);       // rows of a workgroup
            const bool short_heads = 4 * a.S <= rows;
            const long long prepare_blocks = short_heads ? ((long long)a.B * a.H * a.S + short_rows - 1) / short_rows : (long long)a.B * a.H * ((a.S + rows - 1) / rows);
            const dim3 prepare_grid((unsigned)(prepare_blocks < kPrepareGrid ? prepare_blocks : kPrepareGrid));
            if (short_heads) hipLaunchKernelGGL((fa_bwd_prepare_short<BF16, D, FL >= 1>), prepare_grid, dim3(256), 0, stream, a);
            else hipLaunchKernelGGL((fa_bwd_prepare<BF16, D, FL >= 1>), prepare_grid, dim3(256), 0, stream, a);
            const int chunk = a.ds_heads > 0 && a.ds_heads < all_heads ? a.ds_heads : all_heads;
            for (int h0 = 0; h0 < all_heads; h0 += chunk) {
                a.head0 = h0;
                a.heads = all_heads - h0 < chunk ? all_heads - h0 : chunk;
                const unsigned launch_k = grid_if(uneven_items, (long long)a.heads * ((a.Sk + KEYS_K - 1) / KEYS_K), GROUPS_K);
                unsigned n_shares = 0;
                if constexpr (CAN_SHARE) {
                    if (a.partials != nullptr) n_shares = (unsigned)fa_bwd_launch_shares(D, a.heads, group, a.S, a.R, a.L, a.walk_head, (int)resident, a.share_slots);
                    if (n_shares != 0) {
                        a.walk_total = a.heads * a.walk_head;
                        hipLaunchKernelGGL((fa_bwd_dkdv<BF16, D, MASKED, FL, ALIBI, DROPOUT, true, true>), dim3(n_shares), dim3(kBwdWaves * 64), smem_dkdv, stream, a);
                        hipLaunchKernelGGL((fa_bwd_add_parts<BF16, D, FL >= 1>), dim3((n_shares - 1) * 2 * kBwdWaves), dim3(256), 0, stream, a, (int)n_shares);
                    }
                }
                if (n_shares == 0)
                    hipLaunchKernelGGL((fa_bwd_dkdv<BF16, D, MASKED, FL, ALIBI, DROPOUT, true, false, NWK>), dim3(launch_k), dim3(NWK * 64), smem_dkdv_ds, stream, a);
                // Fewer than two 256-query items per CU: 128-query ones, twice as many, and a deeper ring, since a CU that
                // walks one item waits for the latency of its tiles.  Backward pass, causal, 128 against 256 queries: B2 H16
                // S2048 D128 (256 items) 162 against 177 us, B1 H8 S2048 D128 88 against 97, B1 H4 S4096 D64 86 against 98, B1 H16
                // S1024 D64 45 against 50; with 512 items level (B8 H16 S1000 D64 108 both), with 1024 K is read twice as often
                // for nothing (B2 H32/8 S4096 D128 910 against 887).
                const long long heads_q = (long long)a.heads * group, items_q = heads_q * ((a.S + 255) / 256);
                if (items_q < 2LL * compute_units) {
                    const unsigned launch_q = grid_if(uneven_items, heads_q * ((a.S + 127) / 128));
                    hipLaunchKernelGGL((fa_bwd_dq_from_ds<BF16, D, MASKED, FL, 4, 4>), dim3(launch_q), dim3(4 * 64), smem_dq_ds(4, 4), stream, a);
                } else if (D == 64 && !uneven_items) {
                    // 64-wide and items alike: 128-query ones, two workgroups per CU that wait at barriers and for their first
                    // tiles at different times.  Backward pass, 128 against 256 queries: no mask B16 H16 S512 96.5 / 101.4 us,
                    // with dropout 113.8 / 117.7, B2 H16 S8192 2064 / 2080, window 700 B2 H32 S8192 501 / 508.  Causal items,
                    // which K read twice as often and shorter pairs of the snake cost more: B4 H16 S2048 151.5 / 149.5,
                    // B16 H16 S1024 196.0 / 194.6, B6 H32/8 S4096 1741 / 1730; B8 H32 S1024 189.0 / 193.4 the other way.
                    if constexpr (D == 64)
                        hipLaunchKernelGGL((fa_bwd_dq_from_ds<BF16, D, MASKED, FL, 4, 3>), dim3((unsigned)(heads_q * ((a.S + 127) / 128))), dim3(4 * 64),
                                           smem_dq_ds(4, 3), stream, a);
                } else if constexpr (D == 128 || MASKED) {
                    const unsigned launch_q = grid_if(uneven_items, items_q);
                    hipLaunchKernelGGL((fa_bwd_dq_from_ds<BF16, D, MASKED, FL, 8, 3>), dim3(launch_q), dim3(8 * 64), smem_dq_ds(8, 3), stream, a);
                }
            }
            return hipGetLastError();
        }
    }
    const unsigned launch_q = grid_for((long long)a.B * a.H * ((a.S + 255) / 256));
    const unsigned launch_k = grid_for((long long)a.B * a.Hk * ((a.Sk + 255) / 256));
    hipLaunchKernelGGL(kq, dim3(launch_q), dim3(kBwdWaves * 64), smem_dq, stream, a);
    if constexpr (EITHER) {
        if ((long long)launch_k < (long long)a.B * a.Hk * ((a.Sk + 255) / 256)) {
            hipLaunchKernelGGL((fa_bwd_dkdv<BF16, D, MASKED, LAYOUT, ALIBI, DROPOUT, false, false, kBwdWaves, false>), dim3(launch_k), dim3(kBwdWaves * 64), smem_dkdv, stream, a);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL(kkv, dim3(launch_k), dim3(kBwdWaves * 64), smem_dkdv, stream, a);
    return hipGetLastError();
}

}  // namespace

#endif
