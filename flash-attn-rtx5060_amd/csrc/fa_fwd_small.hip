// Problems too small to fill the chip with 128-row blocks: 32 query rows per workgroup, whose waves share the keys.
//
// A block of the tile kernels (fa_fwd_kernel_impl.h) walks its key tiles one behind the other, two iterations more than it has
// tiles; where few blocks leave most compute units idle, that chain of latencies is the time of the call.  Here all NW waves of
// a workgroup hold the same 32 queries, take the key tiles in turn, each on its own -- a wave brings its tiles into LDS of its
// own and waits for nobody -- and meet once, at the end, to merge what they have.  Four times as many workgroups, an NW-th of
// the walk.  K and V are read once per 32 rows instead of once per 128, which is why larger problems keep the tile kernels.
//
//  * A tile is 8 KB of K and 8 KB of V: 64 keys at head dimension 64, 32 at 128.  One stage each: the next K tile is requested as
//    soon as the last fragment of the current one has been read, the next V tile behind PV, so each has the other half of an
//    iteration to arrive in.
//  * Layouts, products and operands are the tile kernels': S^T = K Q^T with v_mfma_f32_32x32x16, P from the accumulators straight
//    into O^T = V^T P^T, V^T by ds_read_b64_tr_b16.
//  * The merge goes through the waves' own LDS: reference points and row sums, then the rescaled accumulators, summed in the
//    order of the waves.
//
// Bound by latency: at B1 H4 S256 D64, 32 workgroups of one tile per wave, 4.5 us from launch to launch, of which an empty launch
// takes 2 (tile kernels 6.8: 1.7 us of set-up, six iterations of 0.8 of one wave per SIMD, 0.7 for the epilogue).  GPU time, tile
// kernels / this: causal B1 H4 S256 D64 8.4 / 4.9 us, B1 H16 S512 D64 11.4 / 6.3, D128 14.6 / 9.3, B1 H8 S1024 D128 22.1 / 13.2, B1 H4
// S8192 D64 87.5 / 61.1, window 200 B1 H16 S1024 D64 12.2 / 10.1, slopes B1 H16 S1024 D64 20.3 / 12.1.
#include "fa_fwd_kernel_impl.h"

namespace {

template <bool BF16, int D, bool ALIBI, int NW>
__global__ void __launch_bounds__(NW * 64, 2) fa_fwd_small(const FaKernelArgs a)
{
    constexpr int KT = 64 * 64 / D;               // keys per tile
    constexpr int CPR = D / 8, ROWB = D * 2, TILEB = KT * ROWB, INSTR = TILEB / 1024;
    constexpr int KS = D / 16, DB = D / 32, KB = KT / 32;
    constexpr int WAVEB = 2 * TILEB;              // a wave's LDS
    static_assert(TILEB == 8192 && 32 * D * 4 <= WAVEB, "a wave's part of O takes the place of its tiles");
    typedef Num<BF16> N;
    typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
    typedef __attribute__((address_space(3))) f32x2 lds_f32x2;

    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, l32 = lane & 31, l16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (blockIdx.y != 0) {
        first_rows_item<BF16, D, ALIBI, true, false, false, NW>(a, blockIdx.x, wave, lds0);
        return;
    }
    if ((long long)blockIdx.x >= a.n_items) return;       // (the grid is as wide as its wider row)
    const uint32_t lds_k = lds0 + wave * WAVEB, lds_v = lds_k + TILEB, lds_stat = lds0 + NW * WAVEB;

    int list_bh, qblock, hi, hk;
    fa_item_decode(blockIdx.x, a.BH, a.n_qblocks, a.descending, &list_bh, &qblock);
    const int bi = fa_strided_heads(list_bh, a.H, a.Hk, &hi, &hk), bh = bi * a.H + hi;
    const uint16_t *Qh = a.Q + (size_t)bi * a.q_bs + (size_t)hi * a.q_hs;
    const char *Kh = reinterpret_cast<const char *>(a.K + (size_t)bi * a.k_bs + (size_t)hk * a.k_hs);
    const char *Vh = reinterpret_cast<const char *>(a.V + (size_t)bi * a.v_bs + (size_t)hk * a.v_hs);
    const int S = a.S, Sk = a.Sk, pos_off = Sk - S, q0 = qblock * 32;
    const int my_q = q0 + l32 < S ? q0 + l32 : S - 1;     // (a row past the end works on a copy of the last one and stores nothing)
    const int q_pos = my_q + pos_off, rows = S - q0 < 32 ? S - q0 : 32;
    int t0, t1;
    fa_tile_range(Sk, KT, a.L, a.R, q0 + pos_off, rows, &t0, &t1);

    // direct global -> LDS loads of a whole tile; rows past the last key are fetched from it and masked
    auto request = [&](const char *head, int rs, int tile, uint32_t lds, bool is_k) __attribute__((always_inline)) {
        const uint32_t rb = (uint32_t)rs * 2u;
        const char *src = head + (size_t)tile * KT * rb;
        const int last = Sk - 1 - tile * KT;
#pragma unroll
        for (int n = 0; n < INSTR; ++n) {
            const int P = n * 64 + lane, row = P / CPR, pos = P % CPR;
            dma_16(src, (uint32_t)(row < last ? row : last) * rb + (uint32_t)((pos ^ (is_k ? k_swz<CPR>(row) : v_swz<CPR>(row))) << 4), lds + n * 1024);
        }
    };
    int tile = t0 + wave;
    if (tile <= t1) request(Kh, a.k_rs, tile, lds_k, true);

    u32x4 qf[KS];                                 // Q^T: lane = (query l32, head-dim slice 8 * half .. + 7 of each 16)
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const u32x4 *>(Qh + (size_t)my_q * a.q_rs + 16 * s + 8 * half);
    if (tile <= t1) request(Vh, a.v_rs, tile, lds_v, false);

    const float cs = a.scale_log2e;
    const float slope = ALIBI ? a.alibi[bh % a.H] : 0.0f, neg_slope_raw = ALIBI ? -slope / a.scale : 0.0f;
    uint32_t koff[KS], voff[DB];
#pragma unroll
    for (int s = 0; s < KS; ++s) koff[s] = lds_k + (uint32_t)(l32 * ROWB + (((2 * s + half) ^ k_swz<CPR>(l32)) << 4));
    {
        const int row0 = 4 * half + (l16 >> 2), dq = l32 >> 4, c4 = l16 & 3;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            const int c = 4 * db + 2 * dq + (c4 >> 1);
            voff[db] = lds_v + (uint32_t)(row0 * ROWB + ((c ^ v_swz<CPR>(row0)) << 4) + ((c4 & 1) << 3));
        }
    }
    f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] = 0.0f;
    float m_run = kNoReference, l_run = 0.0f;
    // (Q is waited for here, once: inside the loop the compiler's wait would also be one for the tiles)
    wait_vm<INSTR>();
#pragma unroll
    for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[s]));

    for (; tile <= t1; tile += NW) {
        wait_vm<INSTR>();                         // K(tile) has landed; V(tile), requested behind it, may be in flight
        f32x16 sx[KB];
        const int first = tile * KT + 4 * half;   // key of accumulator row 0 on this lane
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                sx[kb][r] = ALIBI ? __builtin_fabsf((float)(q_pos - first - 32 * kb - 8 * (r >> 2) - (r & 3))) * neg_slope_raw : 0.0f;
        u32x4 fr[KS * KB];
#pragma unroll
        for (int n = 0; n < KS * KB; ++n) fr[n] = lds_read_b128(koff[n / KB] + (uint32_t)((n % KB) * 32 * ROWB));
#pragma unroll
        for (int n = 0; n < KS * KB; ++n) sx[n % KB] = N::mfma(fr[n], qf[n / KB], sx[n % KB]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // (every fragment is in registers)
        const bool more = tile + NW <= t1;
        if (more) request(Kh, a.k_rs, tile + NW, lds_k, true);

        // some row of the block does not see all keys of the tile (wave-uniform)
        if ((tile + 1) * KT > Sk || fa_tile_class(KT, a.L, a.R, q0 + pos_off, rows, tile) != 2) {
            const int j_hi = (q_pos + a.R < Sk - 1 ? q_pos + a.R : Sk - 1) - first, j_lo = q_pos - a.L - first;
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int j = 32 * kb + 8 * (r >> 2) + (r & 3);
                    if (j > j_hi || j < j_lo) sx[kb][r] = -INFINITY;
                }
        }
        float mx = max_plain(sx[0][0], sx[KB - 1][15]);
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = KB == 2 ? fmaxf(fmaxf(mx, sx[0][r]), sx[KB - 1][r]) : fmaxf(mx, sx[0][r]);
        mx = max_of_halves(mx);
        const bool grow = __builtin_fmaf(mx, cs, -m_run * cs) > kRescaleLog2;
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
            const float m_new = grow ? mx : m_run, alpha = __builtin_amdgcn_exp2f((m_run - m_new) * cs);
            l_run *= alpha;
            m_run = m_new;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
        }
        const float nmc = -m_run * cs;
        uint32_t pk[8 * KB];
        float l_b = 0.0f;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float e0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sx[kb][2 * i], cs, nmc));
                const float e1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sx[kb][2 * i + 1], cs, nmc));
                l_run += e0; l_b += e1;
                pk[8 * kb + i] = N::pack2(e0, e1);
            }
        l_run += l_b;

        if (more) wait_vm<INSTR>(); else wait_vm<0>();      // V(tile); K(tile + NW) may be in flight
#pragma unroll
        for (int t2 = 0; t2 < 2 * KB; ++t2) {
            const u32x4 p = {pk[4 * t2], pk[4 * t2 + 1], pk[4 * t2 + 2], pk[4 * t2 + 3]};
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const u32x2 lo = lds_read_tr(voff[db] + (uint32_t)((16 * t2) * ROWB)), hi2 = lds_read_tr(voff[db] + (uint32_t)((16 * t2 + 8) * ROWB));
                o[db] = N::mfma(u32x4{lo[0], lo[1], hi2[0], hi2[1]}, p, o[db]);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (more) request(Vh, a.v_rs, tile + NW, lds_v, false);
    }

    // ---- the merge
    const int lane_e = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), row_e = lane_e & 31, half_e = lane_e >> 5;
    l_run += swap_halves(l_run);
    if (half_e == 0) *(lds_f32x2 *)(uintptr_t)(lds_stat + (uint32_t)((wave * 32 + row_e) * 8)) = f32x2{m_run, l_run};
    __syncthreads();
    float m_all = kNoReference;
#pragma unroll
    for (int w = 0; w < NW; ++w) m_all = fmaxf(m_all, (*(const lds_f32x2 *)(uintptr_t)(lds_stat + (uint32_t)((w * 32 + row_e) * 8)))[0]);
    const float f = __builtin_amdgcn_exp2f((m_run - m_all) * cs);
    // [row][16-byte column c at c ^ (row & 7)]: the lanes of a store are 32 rows of one column
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int c = 8 * db + 2 * g + half_e;
            *(lds_f32x4 *)(uintptr_t)(lds_k + (uint32_t)(row_e * (D * 4) + ((c ^ (row_e & 7)) << 4))) =
                f32x4{o[db][4 * g] * f, o[db][4 * g + 1] * f, o[db][4 * g + 2] * f, o[db][4 * g + 3] * f};
        }
    __syncthreads();
    // rows of a causal head that first_rows_item writes
    const int f_rows = a.first_parts > 0 ? 32 - pos_off : 0;
    for (int at = tid; at < 32 * CPR; at += NW * 64) {
        const int row = at / CPR, c = at % CPR, q = q0 + row;
        if (q >= S || q < f_rows) continue;
        float m = kNoReference, l = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) m = fmaxf(m, (*(const lds_f32x2 *)(uintptr_t)(lds_stat + (uint32_t)((w * 32 + row) * 8)))[0]);
        f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f}, y = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const f32x2 st = *(const lds_f32x2 *)(uintptr_t)(lds_stat + (uint32_t)((w * 32 + row) * 8));
            l += st[1] * __builtin_amdgcn_exp2f((st[0] - m) * cs);
            const uint32_t base = lds0 + (uint32_t)(w * WAVEB + row * (D * 4));
            x += *(const lds_f32x4 *)(uintptr_t)(base + (uint32_t)(((2 * c) ^ (row & 7)) << 4));
            y += *(const lds_f32x4 *)(uintptr_t)(base + (uint32_t)(((2 * c + 1) ^ (row & 7)) << 4));
        }
        // (a row that sees no key; not where l is NaN, that row is NaN.  With the regular kernels' lengths every row sees one: a sum of
        // zero is one of scores that are all -inf, and 0 / 0 says so)
        const bool empty = l == 0.0f && !(Sk == S && S % 128 == 0);
        const float inv = empty ? 0.0f : 1.0f / l;
        const u32x4 w4 = {N::pack2(x[0] * inv, x[1] * inv), N::pack2(x[2] * inv, x[3] * inv), N::pack2(y[0] * inv, y[1] * inv), N::pack2(y[2] * inv, y[3] * inv)};
        *reinterpret_cast<u32x4 *>(a.O + (size_t)bi * a.o_bs + (size_t)hi * a.o_hs + (size_t)q * a.o_rs + 8 * c) = w4;
        if (a.lse != nullptr && c == 0) a.lse[(size_t)bh * S + q] = empty ? -INFINITY : m * a.scale + __builtin_logf(l);
    }
}

template <bool BF16, int D, bool ALIBI, int NW>
hipError_t launch_small(const FaKernelArgs &a, hipStream_t stream, bool configure_only)
{
    constexpr size_t smem = NW * 16384 + NW * 32 * 8;
    auto kern = fa_fwd_small<BF16, D, ALIBI, NW>;
    static std::atomic<unsigned long long> configured{0ull};
    const unsigned long long dev_bit = 1ull << fa_launch_device();
    if (!(configured.load(std::memory_order_relaxed) & dev_bit)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        if (e != hipSuccess) return e;
        configured.fetch_or(dev_bit, std::memory_order_relaxed);
    }
    if (configure_only) return hipSuccess;
    const unsigned items = (unsigned)a.n_items, first = (unsigned)(a.BH * a.first_parts);
    hipLaunchKernelGGL(kern, dim3(items > first ? items : first, first > 0 ? 2 : 1), dim3(NW * 64), smem, stream, a);
    return hipGetLastError();
}

}  // namespace

// a.n_items workgroups (heads times 32-row blocks) of `waves` (4 or 8) waves
hipError_t fa_launch_forward_small(const FaKernelArgs &a, int bf16, int D, int waves, hipStream_t stream, bool configure_only)
{
    const int alibi = a.alibi != nullptr;
#define FA_SMALL(BF, DD, AL, WV) \
    if (bf16 == BF && D == DD && alibi == AL && waves == WV) return launch_small<BF != 0, DD, AL != 0, WV>(a, stream, configure_only);
#define FA_SMALLS(BF, DD) FA_SMALL(BF, DD, 0, 4) FA_SMALL(BF, DD, 1, 4) FA_SMALL(BF, DD, 0, 8) FA_SMALL(BF, DD, 1, 8)
    FA_SMALLS(0, 64) FA_SMALLS(0, 128) FA_SMALLS(1, 64) FA_SMALLS(1, 128)
#undef FA_SMALLS
#undef FA_SMALL
    return hipErrorInvalidValue;
}

hipError_t fa_configure_forward_small()
{
    FaKernelArgs a = {};
    static const float slope_stand_in = 0.0f;      // (only tested against null)
    for (int combo = 0; combo < 16; ++combo) {
        a.alibi = (combo & 1) ? &slope_stand_in : nullptr;
        const hipError_t e = fa_launch_forward_small(a, (combo >> 1) & 1, (combo & 4) ? 128 : 64, (combo & 8) ? 8 : 4, nullptr, true);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
