// Few queries behind long keys (decoding): a kernel of its own, and the merge of key splits.
//
// At most 32 query rows read a K/V head -- the G query heads that share it, times S new positions -- so the path is
// bound by HBM: every byte of K and V is read once and feeds one or two 16-column matrix instructions.  What the
// tile kernels (fa_fwd_kernel_impl.h) do for reuse is in the way here: their waves share 64-key tiles through a
// workgroup barrier, so that the loads in flight drain at every tile.  Here nothing is shared.  A wave walks pieces
// of its own (32 keys at head dimension 128, 64 at 64: 8 KB of K, 8 KB of V), the waves of a workgroup taking
// consecutive pieces, and requests the next piece as soon as the registers of the current one are free; they meet
// once, at the end, to merge their partial results through LDS.
//
//  * S^T = K Q^T with v_mfma_f32_16x16x32: K rows go from HBM straight into the A operand (lane = key, 16 bytes of
//    the head dimension: the four instructions of a row read its 256 bytes), Q^T is the B operand, read from LDS.  The
//    accumulator has the query on the lane and four keys of every 16 in it, so the softmax reductions are in-register
//    plus two half swaps.
//  * O^T += V^T P^T: the P accumulators of two 16-key blocks are, packed, the B operand of 32 keys.  V arrives in
//    whole rows, goes through 8 KB of LDS that belong to the wave alone (no barrier), and comes back transposed
//    (ds_read_b64_tr_b16); 32-byte columns are XOR-swizzled by the row, so neither side has bank conflicts.
//  * K and V are read with the non-temporal hint when there is more of them than stays in the memory-side cache: a
//    read-only loop over 2 GB runs at 7.1 TB/s with it and at 6.2 without (512 MB: 7.0 against 6.1).  Here, with the
//    hint against without: B4 H32 S_kv 32768 (2.1 GB) 329 against 369 us, B16 H32/8 S_kv 8192 (537 MB) 87 against 98,
//    B1 H64/8 S_kv 32768 (134 MB) 33.5 against 35.5; but B8 H32/8 S_kv 2048 (67 MB, called again and again) 18.5 against 17.2.
//  * Four waves per workgroup, four workgroups per CU (up to 16 rows: 128 registers): both launches of B4 H32 S_kv 32768
//    324 us, with eight waves 329, with sixteen 334 (before the splits followed the load of the busiest CU, see
//    fa_fwd_auto_splits; since then 308, of which this kernel 306 = 7.0 TB/s).
//
// Measured, both launches of a call, against the tile kernels, each with the splits that "auto" takes for it: B4 H32 S_kv
// 32768 308 us against 370, B16 H32/8 S_kv 8192 82.6 against 96.5, B1 H32/8 S_kv 1003 10.4 against 16.5 (with the call's host
// time, two microseconds of the difference).
#include "fa_fwd_kernel_impl.h"

namespace {

constexpr int kDecodeWaves = 4;

template <bool BF16> __device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c)
{
    if (BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
// maximum and sum over the four lanes l, l ^ 16, l ^ 32, l ^ 48, in all four
__device__ __forceinline__ float max_of_quarters(float x)
{
    float a = x, b = x, m;
    asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_max_f32 %2, %0, %1" : "+v"(a), "+v"(b), "=v"(m));
    return max_of_halves(m);
}
__device__ __forceinline__ float sum_of_quarters(float x)
{
    float a = x, b = x, m;
    asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_add_f32 %2, %0, %1" : "+v"(a), "+v"(b), "=v"(m));
    a = m; b = m;
    asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_add_f32 %2, %0, %1" : "+v"(a), "+v"(b), "=v"(m));
    return m;
}

// the lane index, read from the hardware and tied to the place of the call
__device__ __forceinline__ int lane_again()
{
    int ln = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(ln));
    return ln;
}

// ---- what merges the parts of a row's key splits (fa_combine_splits, and the decoding kernel's own merge)
// A part of weight zero is left out, not multiplied: what it holds may be infinite.
// (the choice in front of the product, so that sums of products stay fused, with one rounding each)
__device__ __forceinline__ f32x4 merge_weighted(f32x4 part, float w)
{
    const f32x4 none = {0.0f, 0.0f, 0.0f, 0.0f};
    return (w > 0.0f ? part : none) * w;
}
struct MergeSum {
    // running reference point and sum of weights (logsumexps are scaled scores, of any size: kNoReference is one for raw
    // scores; from the lowest finite number the differences below are never NaN)
    float m = -__FLT_MAX__, l = 0.0f;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
};
typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void part_store(float *p, f32x4 v)
{
    const u64x2 w = __builtin_bit_cast(u64x2, v);
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(p), w[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(p) + 1, w[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The parts of a row's four elements, eight at a time, of group `group` of `groups` that take eight in turn.  AGENT: parts that
// other workgroups of this launch have stored at the device's scope.
template <bool AGENT>
__device__ __forceinline__ void merge_parts(MergeSum &sum, const float *lse_row, const float *o_row, size_t lse_step, size_t o_step, int n, int group, int groups)
{
    constexpr int BATCH = 8;
    for (int s0 = BATCH * group; s0 < n; s0 += BATCH * groups) {
        float lse[BATCH];
        f32x4 o[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            const int s = s0 + u < n ? s0 + u : n - 1;
            if (AGENT) {
                lse[u] = __hip_atomic_load(&lse_row[(size_t)s * lse_step], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=v"(o[u]) : "v"(o_row + (size_t)s * o_step) : "memory");
            } else {
                lse[u] = lse_row[(size_t)s * lse_step];
                o[u] = *reinterpret_cast<const f32x4 *>(o_row + (size_t)s * o_step);
            }
        }
        if (AGENT)
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]), "+v"(o[4]), "+v"(o[5]), "+v"(o[6]), "+v"(o[7]) :: "memory");
        float mx = sum.m;
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            if (s0 + u >= n) lse[u] = -INFINITY;
            mx = fmaxf(mx, lse[u]);
        }
        const float alpha = __expf(sum.m - mx);
        sum.acc = merge_weighted(sum.acc, alpha);
        sum.l *= alpha;
        sum.m = mx;
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            const float w = __expf(lse[u] - mx);
            sum.acc += merge_weighted(o[u], w);
            sum.l += w;
        }
    }
}
// A group's sum added to those of the groups in front of it; w: its weight against the largest reference point of all groups
__device__ __forceinline__ void merge_group(f32x4 &acc, float &l, f32x4 group_acc, float group_l, float w)
{
    acc += merge_weighted(group_acc, w);
    l += group_l * w;
}

// NB: 16-row blocks of queries (R <= 16 * NB rows); NW: waves per workgroup; NT: K and V with the streaming hint
template <bool BF16, int D, int NB, int NW, bool ALIBI, bool NT>
__global__ void __launch_bounds__(NW * 64, NB == 1 ? 4 : 2) fa_fwd_decode(const FaKernelArgs a)
{
    constexpr int KP = 32 * (128 / D);            // keys per piece
    constexpr int ROWB = D * 2, CPR = D / 8, RPI = 64 / CPR;
    constexpr int KSL = D / 32;                   // 32-wide slices of the head dimension (QK^T)
    constexpr int JB = KP / 16;                   // 16-key blocks of a piece
    constexpr int DB = D / 16;                    // 16-wide blocks of the head dimension (PV)
    constexpr int VI = KP / RPI;                  // 1 KB instructions per piece of V (and of K: JB * KSL)
    constexpr int PIECEB = KP * ROWB;             // 8 KB
    typedef Num<BF16> N;
    typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
    typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
    typedef __attribute__((address_space(3))) float lds_f32;

    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
    const uint32_t lds_q = lds0 + NW * PIECEB;                        // Q^T fragments, [row block][slice][lane]
    const uint32_t lds_stat = lds_q + NB * KSL * 1024;                // [wave][row]: reference point, row sum
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // consecutive workgroups read consecutive key ranges of one K/V head
    const int n_splits = a.n_splits;
    // (heads interleaved within the rows, [B,S,H,D]: workgroups are dealt round robin over the XCDs, and neighbouring heads
    // lie in the same pages, so each XCD gets a run of the list instead of every eighth item -- otherwise every XCD's
    // address translation walks all pages: B60 H64 S_kv 3000 D64 520 against 608 us, B4 H16 S_kv 27270 D64 87 against 98;
    // for whole heads in a piece the plain order is level or better, B16 H32/8 S_kv 8192 82 against 85)
    unsigned block = blockIdx.x;
    if (a.k_hs < a.k_rs) {
        const unsigned per = gridDim.x >> 3, rest = gridDim.x & 7, xcd = blockIdx.x & 7;
        block = xcd * per + (xcd < rest ? xcd : rest) + (blockIdx.x >> 3);
    }
    const unsigned item = block / (unsigned)n_splits;
    const int split = (int)(block - item * (unsigned)n_splits);
    const int b = (int)(item / (unsigned)a.Hk), hk = (int)(item - (unsigned)b * (unsigned)a.Hk);
    const int S = a.S, Sk = a.Sk, pos_off = Sk - S, G = a.pack, R = G * S;
    const int h0 = hk * G, bh = b * a.H + h0;
    const uint16_t *Qh = a.Q + (size_t)b * a.q_bs + (size_t)h0 * a.q_hs;
    const char *Kh = reinterpret_cast<const char *>(a.K + (size_t)b * a.k_bs + (size_t)hk * a.k_hs);
    const char *Vh = reinterpret_cast<const char *>(a.V + (size_t)b * a.v_bs + (size_t)hk * a.v_hs);

    // the keys that some row sees, in pieces, and this workgroup's share of them
    const int key_lo = pos_off - a.L > 0 ? pos_off - a.L : 0;
    const int all_lo = key_lo / KP, n_pieces = (Sk - 1) / KP - all_lo + 1;
    const int per_split = (n_pieces + n_splits - 1) / n_splits;
    const int p_begin = all_lo + split * per_split;
    const int p_end = split * per_split + per_split < n_pieces ? p_begin + per_split : all_lo + n_pieces;

    const uint32_t k_rb = (uint32_t)a.k_rs * 2u, v_rb = (uint32_t)a.v_rs * 2u;      // row strides in bytes
    u32x4 kr[JB * KSL], vr[VI];
    auto request = [&](int piece) __attribute__((always_inline)) {
        // (what follows from the lane index is formed anew at every piece: held through the loop it is spilled)
        const int ln = lane_again();
        const uint32_t k_row0 = (uint32_t)(ln & 15) * k_rb, v_row0 = (uint32_t)(ln / CPR) * v_rb;
        const int first = piece * KP;
        const char *kp = Kh + (size_t)first * k_rb, *vp = Vh + (size_t)first * v_rb;
        // (rows past the end are read from the last row and masked)
        const uint32_t last = (uint32_t)(Sk - 1 - first), k_last = last * k_rb, v_last = last * v_rb;
#pragma unroll
        for (int j = 0; j < JB; ++j) {
            uint32_t off = k_row0 + (uint32_t)(16 * j) * k_rb;
            off = (last < (uint32_t)(KP - 1) && off > k_last ? k_last : off) + 16u * (uint32_t)(ln >> 4);
#pragma unroll
            for (int s = 0; s < KSL; ++s) {
                const u32x4 *src = reinterpret_cast<const u32x4 *>(kp + off + 64 * s);
                kr[j * KSL + s] = NT ? __builtin_nontemporal_load(src) : *src;
            }
        }
#pragma unroll
        for (int i = 0; i < VI; ++i) {
            uint32_t off = v_row0 + (uint32_t)(RPI * i) * v_rb;
            off = (last < (uint32_t)(KP - 1) && off > v_last ? v_last : off) + 16u * (uint32_t)(ln % CPR);
            const u32x4 *src = reinterpret_cast<const u32x4 *>(vp + off);
            vr[i] = NT ? __builtin_nontemporal_load(src) : *src;
        }
    };
    int piece = p_begin + wave;
    if (piece < p_end) request(piece);

    // Q^T: lane (row l16, quarter g) of slice s holds head-dim values 32 s + 8 g .. + 7; missing rows are zero
    for (int i = tid; i < NB * 16 * CPR; i += NW * 64) {
        const int row = i / CPR, c = i % CPR;
        u32x4 w = {0, 0, 0, 0};
        if (row < R) {
            const int rh = row / S;
            w = *reinterpret_cast<const u32x4 *>(Qh + (size_t)rh * a.q_hs + (size_t)(row - rh * S) * a.q_rs + 8 * c);
        }
        *(lds_u32x4 *)(uintptr_t)(lds_q + (uint32_t)(((row >> 4) * KSL + (c >> 2)) * 1024 + ((c & 3) * 16 + (row & 15)) * 16)) = w;
    }
    int pos[NB];                                  // key position of this lane's query
    float slope_raw[NB];                          // ALiBi: -slope / scale, in raw score units per key of distance
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int row = 16 * nb + l16 < R ? 16 * nb + l16 : R - 1, rh = row / S;
        pos[nb] = row - rh * S + pos_off;
        slope_raw[nb] = ALIBI ? -a.alibi[h0 + rh] / a.scale : 0.0f;
    }
    const float cs = a.scale_log2e, thresh = kRescaleLog2 / cs;
    float m_run[NB], l_run[NB];
    f32x4 o[NB][DB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        m_run[nb] = kNoReference;
        l_run[nb] = 0.0f;
#pragma unroll
        for (int db = 0; db < DB; ++db) o[nb][db] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // the wave's 8 KB of LDS: row r of the piece at r * ROWB, its 32-byte column c at c ^ v_col(r)
    const uint32_t lds_v = lds0 + wave * PIECEB;
    auto v_col = [](int row) __attribute__((always_inline)) { return D == 128 ? row & 7 : (row >> 1) & 3; };
    // (the i-th instruction of a piece brings row RPI * i + lane / CPR: v_col of it differs from that of i = 0 by a
    // constant, D = 128: bit 2 for odd i)
    const uint32_t v_wr = lds_v + (uint32_t)((lane / CPR) * ROWB + ((((lane % CPR) >> 1) ^ v_col(lane / CPR)) << 5) + ((lane & 1) << 4));
    const int tr_row = 4 * g + (l16 >> 2);
    const uint32_t v_rd = lds_v + (uint32_t)(tr_row * ROWB + (v_col(tr_row) << 5) + ((l16 & 3) << 3));
    __syncthreads();

    for (; piece < p_end; piece += NW) {
#pragma unroll
        for (int i = 0; i < VI; ++i)
            *(lds_u32x4 *)(uintptr_t)((v_wr ^ (D == 128 && (i & 1) ? 128u : 0u)) + (uint32_t)(RPI * i * ROWB)) = vr[i];
        __builtin_amdgcn_sched_barrier(0);       // (V's registers are free before Q's are needed)
        f32x4 s[NB][JB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
            for (int j = 0; j < JB; ++j) s[nb][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < KSL; ++i) {
                const u32x4 qf = *(const lds_u32x4 *)(uintptr_t)(lds_q + (uint32_t)((nb * KSL + i) * 1024 + lane * 16));
#pragma unroll
                for (int j = 0; j < JB; ++j) s[nb][j] = mfma16<BF16>(kr[j * KSL + i], qf, s[nb][j]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (piece + NW < p_end) request(piece + NW);      // (the registers of this piece are free)
        __builtin_amdgcn_sched_barrier(0);

        const int first = piece * KP;
        // some row does not see all keys of the piece (wave-uniform)
        const bool edge = first < pos_off + S - 1 - a.L || first + KP - 1 > pos_off + a.R || first + KP > Sk;
        u32x4 p[NB][JB / 2];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (ALIBI) {
                const float base = (float)(pos[nb] - first - 4 * g);
#pragma unroll
                for (int j = 0; j < JB; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[nb][j][r] = __builtin_fmaf(__builtin_fabsf(base - (float)(16 * j + r)), slope_raw[nb], s[nb][j][r]);
            }
            if (edge) {
                const int hi = (pos[nb] + a.R < Sk - 1 ? pos[nb] + a.R : Sk - 1) - first - 4 * g, lo = pos[nb] - a.L - first - 4 * g;
#pragma unroll
                for (int j = 0; j < JB; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (16 * j + r > hi || 16 * j + r < lo) s[nb][j][r] = -INFINITY;
            }
            float mx = s[nb][0][0];
#pragma unroll
            for (int j = 0; j < JB; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[nb][j][r]);
            mx = max_of_quarters(mx);
            const bool grow = mx > m_run[nb] + thresh;
            if (__builtin_amdgcn_ballot_w64(grow) != 0) {
                const float m_new = grow ? mx : m_run[nb], alpha = __builtin_amdgcn_exp2f((m_run[nb] - m_new) * cs);
                l_run[nb] *= alpha;
                m_run[nb] = m_new;
#pragma unroll
                for (int db = 0; db < DB; ++db) o[nb][db] *= alpha;
            }
            const float nmc = -m_run[nb] * cs;
#pragma unroll
            for (int j = 0; j < JB; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    s[nb][j][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[nb][j][r], cs, nmc));
                    l_run[nb] += s[nb][j][r];
                }
#pragma unroll
            for (int t = 0; t < JB / 2; ++t)
                p[nb][t] = u32x4{N::pack2(s[nb][2 * t][0], s[nb][2 * t][1]), N::pack2(s[nb][2 * t][2], s[nb][2 * t][3]),
                                 N::pack2(s[nb][2 * t + 1][0], s[nb][2 * t + 1][1]), N::pack2(s[nb][2 * t + 1][2], s[nb][2 * t + 1][3])};
        }
        // (this wave's LDS operations complete in order: its V rows are in before these reads)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int t = 0; t < JB / 2; ++t)
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const uint32_t at = v_rd ^ (uint32_t)(db << 5);
                const u32x2 lo = lds_read_tr(at + (uint32_t)((32 * t) * ROWB)), hi = lds_read_tr(at + (uint32_t)((32 * t + 16) * ROWB));
                const u32x4 vf = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) o[nb][db] = mfma16<BF16>(vf, p[nb][t], o[nb][db]);
            }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }

    // ---- merge of the waves: reference points and row sums first, then the rescaled accumulators, 16 rows at a time,
    // summed over the waves in their order
    const int lane_e = lane_again(), l16_e = lane_e & 15, g_e = lane_e >> 4, tid_e = wave * 64 + lane_e;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        l_run[nb] = sum_of_quarters(l_run[nb]);
        if (g_e == 0) {
            *(lds_f32 *)(uintptr_t)(lds_stat + (uint32_t)((wave * 16 * NB + 16 * nb + l16_e) * 8)) = m_run[nb];
            *(lds_f32 *)(uintptr_t)(lds_stat + (uint32_t)((wave * 16 * NB + 16 * nb + l16_e) * 8 + 4)) = l_run[nb];
        }
    }
    __syncthreads();                              // (also: every wave has read its last V piece)
    const size_t part = n_splits > 1 ? ((size_t)split * a.BH + bh) * S : 0;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        if (16 * nb >= R) break;
        const int rows = R - 16 * nb < 16 ? R - 16 * nb : 16;
        if (nb > 0) __syncthreads();
        // (32-byte column pairs aside, 16-byte column c of row q sits at c ^ q: consecutive rows on different banks)
        if (l16_e < rows) {
            float m_all = kNoReference;
#pragma unroll
            for (int w = 0; w < NW; ++w)
                m_all = fmaxf(m_all, *(const lds_f32 *)(uintptr_t)(lds_stat + (uint32_t)((w * 16 * NB + 16 * nb + l16_e) * 8)));
            const float f = __builtin_amdgcn_exp2f((m_run[nb] - m_all) * cs);
#pragma unroll
            for (int db = 0; db < DB; ++db)
                *(lds_f32x4 *)(uintptr_t)(lds0 + (uint32_t)(wave * (16 * D * 4) + l16_e * (D * 4) + (((4 * db + g_e) ^ l16_e) << 4))) = o[nb][db] * f;
        }
        __syncthreads();
        for (int i = tid_e; i < rows * (D / 4); i += NW * 64) {
            const int q = i / (D / 4), c = i % (D / 4), row = 16 * nb + q;
            float m_all = kNoReference, mw[NW], l_all = 0.0f;
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                mw[w] = *(const lds_f32 *)(uintptr_t)(lds_stat + (uint32_t)((w * 16 * NB + row) * 8));
                m_all = fmaxf(m_all, mw[w]);
            }
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                l_all += *(const lds_f32 *)(uintptr_t)(lds_stat + (uint32_t)((w * 16 * NB + row) * 8 + 4)) * __builtin_amdgcn_exp2f((mw[w] - m_all) * cs);
                acc += *(const lds_f32x4 *)(uintptr_t)(lds0 + (uint32_t)(w * (16 * D * 4) + q * (D * 4) + ((c ^ q) << 4)));
            }
            const bool empty = l_all == 0.0f;     // no key of this row in this share (a NaN is one's: as -inf, the merge would drop it)
            acc *= empty ? 0.0f : 1.0f / l_all;
            const float lse = empty ? -INFINITY : m_all * a.scale + __builtin_logf(l_all);
            if (n_splits > 1) {
                if (a.merge != nullptr) {         // (for a workgroup that may run on another XCD, see below)
                    part_store(a.o_part + (part + row) * D + 4 * c, acc);
                    if (c == 0) __hip_atomic_store(&a.lse_part[part + row], lse, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                } else {
                    *reinterpret_cast<f32x4 *>(a.o_part + (part + row) * D + 4 * c) = acc;
                    if (c == 0) a.lse_part[part + row] = lse;
                }
            } else {
                const int rh = row / S;
                u32x2 w2;
                w2[0] = N::pack2(acc[0], acc[1]);
                w2[1] = N::pack2(acc[2], acc[3]);
                *reinterpret_cast<u32x2 *>(a.O + (size_t)b * a.o_bs + (size_t)(h0 + rh) * a.o_hs + (size_t)(row - rh * S) * a.o_rs + 4 * c) = w2;
                if (a.lse != nullptr && c == 0) a.lse[(size_t)bh * S + row] = lse;
            }
        }
    }
    if (n_splits == 1 || a.merge == nullptr) return;

    // ---- the head's splits merged by the workgroup that finishes the last of them, in the order of the splits.  Parts are
    // stored and loaded at the device's scope, past the L2 of the XCD, so a store that has been acknowledged is seen from
    // every XCD, and no cache has to be written back: a workgroup waits for its stores, counts itself, and who counts last
    // finds all parts.
    // (Bound by latency: three trips to memory, against a launch, its gap and two trips.  GPU time of a call by two launches /
    // this: B1 H32/8 S_kv 1003 bf16 8.1 / 7.9 us, B2 H32 S_kv 1155 11.9 / 11.3, B4 H32/8 S_kv 1616 9.2 / 8.6, B1 H8/1 S_kv 2000 8.4 /
    // 8.6; with the host's part the first takes 9.9 / 7.4.)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    volatile __attribute__((address_space(3))) unsigned *arrived = (volatile __attribute__((address_space(3))) unsigned *)(uintptr_t)lds_stat;
    if (tid_e == 0) *arrived = atomicAdd(&a.merge[item * kFaMergeStride], 1u);
    __syncthreads();
    if (*arrived != (unsigned)n_splits - 1u) return;
    if (tid_e == 0) __hip_atomic_store(&a.merge[item * kFaMergeStride], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // fa_combine_splits' groups of splits, its batches and its order of sums, so that a call's bits do not depend on which of the two
    // merges it; here a group is whichever threads get to it (of its eight groups, those behind the last split add nothing).
    // (At most 256 output places of four elements; from 9 splits on at most 32 KB of parts, so 2048 / splits of them and 455 sums.)
    constexpr int TPR = D / 4, ALL = NW * 64;
    const size_t n_rows = (size_t)a.BH * S;
    const int pairs = R * TPR, all_groups = fa_combine_groups((long long)n_rows, D, n_splits);
    const int groups = all_groups == 1 ? 1 : n_splits < 8 * all_groups ? (n_splits + 7) / 8 : all_groups, sums = pairs * groups;
    auto write = [&](int pair, f32x4 acc, float m, float l) __attribute__((always_inline)) {
        const int row = pair / TPR, t = pair - row * TPR, rh = row / S;
        const bool empty = l == 0.0f;
        acc *= empty ? 0.0f : 1.0f / l;
        u32x2 w2;
        w2[0] = N::pack2(acc[0], acc[1]);
        w2[1] = N::pack2(acc[2], acc[3]);
        *reinterpret_cast<u32x2 *>(a.O + (size_t)b * a.o_bs + (size_t)(h0 + rh) * a.o_hs + (size_t)(row - rh * S) * a.o_rs + 4 * t) = w2;
        if (a.lse != nullptr && t == 0) a.lse[(size_t)bh * S + row] = empty ? -INFINITY : m + __logf(l);
    };
    const uint32_t lds_scalars = lds0 + (uint32_t)sums * 16u;
    for (int at = tid_e; at < sums; at += ALL) {
        const int group = groups > 1 ? at / pairs : 0, pair = at - group * pairs, row = pair / TPR, t = pair - row * TPR;
        const size_t grow = (size_t)bh * S + row;
        MergeSum sum;
        merge_parts<true>(sum, a.lse_part + grow, a.o_part + grow * D + 4 * t, n_rows, n_rows * D, n_splits, group, all_groups);
        if (groups == 1) {
            write(pair, sum.acc, sum.m, sum.l);
        } else {
            *(lds_f32x4 *)(uintptr_t)(lds0 + (uint32_t)at * 16u) = sum.acc;
            *(lds_f32 *)(uintptr_t)(lds_scalars + (uint32_t)at * 8u) = sum.m;
            *(lds_f32 *)(uintptr_t)(lds_scalars + (uint32_t)at * 8u + 4u) = sum.l;
        }
    }
    if (groups == 1) return;
    __syncthreads();
    for (int pair = tid_e; pair < pairs; pair += ALL) {
        float m = -__FLT_MAX__, l = 0.0f;
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int g = 0; g < groups; ++g) m = fmaxf(m, *(const lds_f32 *)(uintptr_t)(lds_scalars + (uint32_t)(g * pairs + pair) * 8u));
        for (int g = 0; g < groups; ++g) {
            const uint32_t scalars = lds_scalars + (uint32_t)(g * pairs + pair) * 8u;
            merge_group(acc, l, *(const lds_f32x4 *)(uintptr_t)(lds0 + (uint32_t)(g * pairs + pair) * 16u), *(const lds_f32 *)(uintptr_t)(scalars + 4u),
                        __expf(*(const lds_f32 *)(uintptr_t)scalars - m));
        }
        write(pair, acc, m, l);
    }
}

// Merges the partial results of a launch with key splits: for every query row,
//   LSE = log sum_s exp(LSE_s),  O = sum_s exp(LSE_s - LSE) * O_s
// (a split that saw no key of the row has LSE_s = -inf and weight 0).  A thread has four output elements of a row and
// takes eight splits at a time, logsumexps and partial rows requested together: one trip to memory for up to eight
// splits.  With more of them GROUPS threads share the four elements, taking eight splits in turn, and their sums meet
// in LDS.  A part of weight 0 is left out, not multiplied: what it holds may be infinite (a split's own keys decide),
// and the places of the last batch behind the last split hold that split's part once more.
template <bool BF16, int D, int GROUPS>
__global__ void __launch_bounds__(256) fa_combine_splits(const FaKernelArgs a)
{
    constexpr int TPR = D / 4;                    // threads per (row, group)
    constexpr int ROWS = 256 / (TPR * GROUPS);    // rows per workgroup
    const int t = threadIdx.x % TPR, group = threadIdx.x / TPR % GROUPS, r = threadIdx.x / (TPR * GROUPS);
    const long long n_rows = (long long)a.BH * a.S;
    long long row = (long long)blockIdx.x * ROWS + r;
    const bool live = row < n_rows;
    if (!live) row = n_rows - 1;
    MergeSum sum;
    merge_parts<false>(sum, a.lse_part + row, a.o_part + row * D + 4 * t, (size_t)n_rows, (size_t)n_rows * D, a.n_splits, group, GROUPS);
    float m = sum.m, l = sum.l;
    f32x4 acc = sum.acc;
    if (GROUPS > 1) {
        __shared__ float sm[GROUPS * ROWS], sl[GROUPS * ROWS];
        __shared__ f32x4 so[256];
        so[threadIdx.x] = acc;
        if (t == 0) { sm[r * GROUPS + group] = m; sl[r * GROUPS + group] = l; }
        __syncthreads();
        if (group != 0) return;
#pragma unroll
        for (int i = 0; i < GROUPS; ++i) m = fmaxf(m, sm[r * GROUPS + i]);
        l = 0.0f;
        acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < GROUPS; ++i) {
            merge_group(acc, l, so[(r * GROUPS + i) * TPR + t], sl[r * GROUPS + i], __expf(sm[r * GROUPS + i] - m));
        }
    }
    if (!live) return;
    const bool empty = l == 0.0f;                 // (not where l is NaN, from a logsumexp of +inf: that row is NaN)
    acc *= empty ? 0.0f : 1.0f / l;
    const int bh = (int)(row / a.S), q = (int)(row - (long long)bh * a.S);
    const int bi = bh / a.H, hi = bh - bi * a.H;
    uint16_t *dst = a.O + (size_t)bi * a.o_bs + (size_t)hi * a.o_hs + (size_t)q * a.o_rs + 4 * t;
    u32x2 w2;
    w2[0] = Num<BF16>::pack2(acc[0], acc[1]);
    w2[1] = Num<BF16>::pack2(acc[2], acc[3]);
    *reinterpret_cast<u32x2 *>(dst) = w2;
    if (a.lse != nullptr && t == 0) a.lse[row] = empty ? -INFINITY : m + __logf(l);
}

template <bool BF16, int D, int NB, int NW, bool ALIBI, bool NT>
hipError_t launch_decode(const FaKernelArgs &a, hipStream_t stream, bool configure_only)
{
    constexpr size_t smem = NW * 8192 + NB * (D / 32) * 1024 + NW * 16 * NB * 8;
    auto kern = fa_fwd_decode<BF16, D, NB, NW, ALIBI, NT>;
    static std::atomic<unsigned long long> configured{0ull};
    const unsigned long long dev_bit = 1ull << fa_launch_device();
    if (!(configured.load(std::memory_order_relaxed) & dev_bit)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        if (e != hipSuccess) return e;
        configured.fetch_or(dev_bit, std::memory_order_relaxed);
    }
    if (configure_only) return hipSuccess;
    hipLaunchKernelGGL(kern, dim3((unsigned)a.n_items), dim3(NW * 64), smem, stream, a);
    return hipGetLastError();
}

}  // namespace

// a.n_items workgroups (K/V heads times splits), four waves each; rows: query rows per K/V head, at most 32;
// streaming: read K and V with the non-temporal hint
hipError_t fa_launch_forward_decode(const FaKernelArgs &a, int bf16, int D, int rows, int streaming, hipStream_t stream, bool configure_only)
{
    const int alibi = a.alibi != nullptr, blocks = rows > 16 ? 2 : 1;
#define FA_DEC(BF, DD, NBV, AL, NT) \
    if (bf16 == BF && D == DD && blocks == NBV && alibi == AL && streaming == NT) \
        return launch_decode<BF != 0, DD, NBV, kDecodeWaves, AL != 0, NT != 0>(a, stream, configure_only);
#define FA_DEC_A(BF, DD, NBV) FA_DEC(BF, DD, NBV, 0, 0) FA_DEC(BF, DD, NBV, 0, 1) FA_DEC(BF, DD, NBV, 1, 0) FA_DEC(BF, DD, NBV, 1, 1)
#define FA_DECS(BF, DD) FA_DEC_A(BF, DD, 1) FA_DEC_A(BF, DD, 2)
    FA_DECS(0, 64) FA_DECS(0, 128) FA_DECS(1, 64) FA_DECS(1, 128)
#undef FA_DECS
#undef FA_DEC_A
#undef FA_DEC
    return hipErrorInvalidValue;
}

hipError_t fa_configure_forward_decode()
{
    FaKernelArgs a = {};
    static const float slope_stand_in = 0.0f;      // (only tested against null)
    for (int bf16 = 0; bf16 < 2; ++bf16)
        for (int D = 64; D <= 128; D += 64)
            for (int rows = 16; rows <= 32; rows += 16)
                for (int combo = 0; combo < 4; ++combo) {
                    a.alibi = (combo & 1) ? &slope_stand_in : nullptr;
                    const hipError_t e = fa_launch_forward_decode(a, bf16, D, rows, combo >> 1, nullptr, true);
                    if (e != hipSuccess) return e;
                }
    return hipSuccess;
}

hipError_t fa_launch_combine_splits(const FaKernelArgs &a, int bf16, int D, hipStream_t stream)
{
    const long long n_rows = (long long)a.BH * a.S;
    const int groups = fa_combine_groups(n_rows, D, a.n_splits);
    const int rows_per_block = fa_combine_rows(D, groups);
    const unsigned grid = (unsigned)((n_rows + rows_per_block - 1) / rows_per_block);
#define FA_COMBINE(BF, DD, GR) \
    if (bf16 == BF && D == DD && groups == GR) hipLaunchKernelGGL((fa_combine_splits<BF != 0, DD, GR>), dim3(grid), dim3(256), 0, stream, a);
    FA_COMBINE(0, 64, 1) FA_COMBINE(0, 64, 8) FA_COMBINE(0, 128, 1) FA_COMBINE(0, 128, 8)
    FA_COMBINE(1, 64, 1) FA_COMBINE(1, 64, 8) FA_COMBINE(1, 128, 1) FA_COMBINE(1, 128, 8)
#undef FA_COMBINE
    return hipGetLastError();
}
