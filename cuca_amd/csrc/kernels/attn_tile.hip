// attn_tile.hip -- paged attention of many query rows of one sequence over f16
// pools (a prefill chunk, verification rows), on the matrix cores: what
// attn_rows.hip describes (its ranges, statuses and generic kernel), for
// head_dim 64, 128 and 256 and groups of 1, 2, 4 and 8.
//
// A workgroup is four waves, a wave 32 query rows of one head: up to four
// heads of a KV head, then more rows; the last rows' workgroups, which see
// the most keys in causal calls, start first.  A tile is 64 positions (four
// paged blocks, from a multiple of 64 on, so that a row's sums depend on its
// own range alone): its K and V rows are copied straight into LDS, a block a
// wave, while the tile before computes, K one tile further ahead than V.
//
//  * S^T = K Q^T as v_mfma_f32_32x32x16_f16: a lane holds 32 keys' scores of
//    one row, so the softmax is the lane's own but for one exchange between
//    the wave's halves, and the weights are already the operand of O^T = V^T
//    P^T once the value product counts its keys in the scores' order.  V^T is
//    read from V's rows by the transposing LDS read.  Rows of 256 bytes would
//    all start on one bank: 16-byte pieces are stored exchanged by row (K: by
//    key mod 16, V: pairs of pieces by key mod 4), in the source addresses of
//    the copies; no bank conflicts (SQ_LDS_BANK_CONFLICT 0).
//  * A weight enters the value product as two f16 parts, hi = f16(p) and lo =
//    f16(p - hi), 22 bits of it.  Weights are held times 2^12, at most 2^15 (the
//    running maximum is raised only by steps above 2^3, so most tiles skip the
//    accumulators' rescale), so lo keeps its bits for weights down to 2^-15 of
//    the largest, and 2^-37 of it below (times 2^7 after steps of 2^8: down to
//    2^-10).
//  * A tile's value product is summed from zero, lo and hi in one chain, and
//    then added: the accumulators round once every 64 keys.  (The chain run in
//    the accumulators themselves rounds eight times; values that cancel then lost
//    1.4 times what one rounding every 16 keys loses, and 3 times what this does.)
//  * The next tile's score products issue between this one's exponentials and
//    conversions, two matrix instructions and eight scores' arithmetic a step; a
//    wave's last tile has none, and weighs only the 16 keys its ranges reach.
//
// What bounds it (causal 4096 rows, 32 heads over 8 of 128): the matrix cores are
// busy 44 % of the launch (SQ_VALU_MFMA_BUSY_CYCLES); each wave, two a SIMD,
// alternates between them and the vector unit (a value product has no arithmetic
// to hide behind), and waits for copies and the tile's barrier 23 % and for issue
// 33 % of its time (SQ_WAIT_ANY, SQ_WAIT_INST_ANY / SQ_WAVE_CYCLES).  MI355X, us,
// before (16-key blocks, 16x16x16 products, a row tile of 16) -> after: causal
// 4096 rows of 32 heads over 8 of 128: 505 -> 221 (218 with the chain in the
// accumulators); with a window of 256 71 -> 48; 2048 rows of 16 heads over 8 of
// 256: 197 -> 107; 8 rows after 4096 keys, 32 heads over 4: 279 -> 109 (one
// workgroup a head group: latency); 8 rows alone, 32 heads over 8: 5.7 -> 6.7 (a
// tile's 64 keys are copied for 8).
#include "common.h"

#pragma clang fp contract(off)

typedef _Float16 at_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 at_h4 __attribute__((ext_vector_type(4)));
typedef short at_s4 __attribute__((ext_vector_type(4)));
typedef _Float16 at_h2 __attribute__((ext_vector_type(2)));
typedef float at_f16v __attribute__((ext_vector_type(16)));
typedef float at_f2 __attribute__((ext_vector_type(2)));

// e less half H of p, exact where p is e rounded: one instruction (the
// compiler makes a conversion and a subtraction of it)
template <int H> __device__ static inline float at_less(float e, at_h2 p) {
    float o;
    if (H == 0) asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(o) : "v"(p), "v"(e));
    else asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(o) : "v"(p), "v"(e));
    return o;
}

template <int D, int HW, int KT>
__device__ static inline void attn_tile_body(const AttnRowsArgs &a) {
    constexpr int RT = 4 / HW;          // row tiles of 32 a workgroup
    constexpr int RB = 2 * D;           // bytes of a key's (or value's) row
    constexpr int CPR = D / 8;          // 16-byte pieces of it
    constexpr int RPC = 64 / CPR;       // rows a copy (1 KB, a wave)
    constexpr int NC = KT / 4 / RPC;    // copies a wave makes of K, and of V
    constexpr int NB = KT / 16;         // paged blocks a tile
    constexpr int NK = KT / 32, NJ = D / 16, ND = D / 32;
    __shared__ __align__(16) unsigned char kv[2][2][KT * RB]; // [tile % 2][K, V]
    __shared__ int span[2][RT];
    if (blockDim.x != 256) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int G = a.n_head / a.n_kv, hgs = G / HW;
    const int kvh = blockIdx.x % a.n_kv, t_id = blockIdx.x / a.n_kv;
    const int tile = (int)gridDim.x / (a.n_kv * hgs) - 1 - t_id / hgs;
    const int hd = (t_id % hgs) * HW + wave % HW, head = kvh * G + hd;
    const int rt = wave / HW;
    const int c = lane & 31, h = lane >> 5;
    const int row = (tile * RT + rt) * 32 + c;
    const bool in_call = row < a.rows;
    int lo = 0, hi = 0;
    if (in_call) {
        lo = a.ranges[2 * (int64_t)row];
        hi = a.ranges[2 * (int64_t)row + 1];
    }
    const bool valid = in_call && lo >= 0 && hi > lo && (int64_t)hi <= (int64_t)a.max_blocks * 16;
    const bool reports = kvh == 0 && hd == 0 && h == 0;
    if (in_call && !valid && reports) record_bad(a.status + CUCA_STATUS_KV_RANGE, (uint32_t)row, 0xffffffffu);
    // the wave's positions: the union [wlo, whi) of its rows' ranges, and the
    // part [ilo, ihi) inside all of them
    int wlo = valid ? lo : 0x7fffffff, whi = valid ? hi : 0;
    int ilo = valid ? lo : 0, ihi = valid ? hi : 0x7fffffff;
#pragma unroll
    for (int off = 1; off < 32; off <<= 1) {
        wlo = min(wlo, (int)xor_partner_bits((uint32_t)wlo, off));
        whi = max(whi, (int)xor_partner_bits((uint32_t)whi, off));
        ilo = max(ilo, (int)xor_partner_bits((uint32_t)ilo, off));
        ihi = min(ihi, (int)xor_partner_bits((uint32_t)ihi, off));
    }
    wlo = __builtin_amdgcn_readfirstlane(wlo);
    whi = __builtin_amdgcn_readfirstlane(whi);
    ilo = __builtin_amdgcn_readfirstlane(ilo);
    ihi = __builtin_amdgcn_readfirstlane(ihi);
    if (lane == 0 && wave % HW == 0) {
        span[0][rt] = wlo;
        span[1][rt] = whi;
    }
    __syncthreads();
    int tlo = span[0][0], thi = span[1][0];
#pragma unroll
    for (int i = 1; i < RT; i++) {
        tlo = min(tlo, span[0][i]);
        thi = max(thi, span[1][i]);
    }
    tlo = __builtin_amdgcn_readfirstlane(tlo);
    thi = __builtin_amdgcn_readfirstlane(thi);
    // the query operand: lane (c, h) holds row c's dims 16 j + 8 h .. + 7.  A
    // negative scale moves into its sign, so that a larger product is a larger score.
    // (At least the smallest normal number, so that a masked score of -inf
    // stays -inf.)
    float scale2 = __builtin_fabsf(a.scale * 1.4426950408889634f);
    if (scale2 < 1.17549435e-38f) scale2 = 1.17549435e-38f;
    at_h8 q[NJ];
    {
        const _Float16 *qr =
            reinterpret_cast<const _Float16 *>(a.q) + (int64_t)(in_call ? row : 0) * a.q_ld + (int64_t)head * D + 8 * h;
        const uint32_t flip = a.scale < 0.0f ? 0x80008000u : 0u;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const uint2 p = *reinterpret_cast<const uint2 *>(qr + 16 * j), r = *reinterpret_cast<const uint2 *>(qr + 16 * j + 4);
            q[j] = __builtin_bit_cast(at_h8, u32x4{p.x ^ flip, p.y ^ flip, r.x ^ flip, r.y ^ flip});
        }
    }
    at_f16v acc[ND];
#pragma unroll
    for (int d = 0; d < ND; d++) acc[d] = at_f16v{};
    float m = -3.40282347e38f, l = 0.0f; // (lowest: a score of -inf less m is -inf)
    bool bad = false;
    if (thi > 0) { // uniform over the workgroup
        const int b0 = tlo >> 4, b1 = (thi - 1) >> 4, t0 = tlo / KT, t1 = (thi - 1) / KT;
        const uint8_t *pk = static_cast<const uint8_t *>(a.pool_k), *pv = static_cast<const uint8_t *>(a.pool_v);
        uint32_t tabv = 0;
        bool tabbad = false;
        int tw = 0; // the window's first tile
        auto load_tab = [&](int t) { // the 64 entries from tile t's first block on
            tw = t;
            tabv = a.table[min(max(t * NB + lane, b0), b1)];
            tabbad = __ballot((int64_t)tabv >= a.n_blocks) != 0;
        };
        // a wave's copies: keys w KT / 4 ... of the tile, RPC a copy
        uint32_t offk[NC], offv[NC];
#pragma unroll
        for (int i = 0; i < NC; i++) {
            const int key = (wave * (KT / 4) + RPC * i + lane / CPR) & 15, slot = lane % CPR;
            const int kx = D == 64 ? key >> 1 : key, vx = (D == 64 ? (key >> 1) & 1 : key & 3) << 2;
            offk[i] = key * RB + ((slot ^ kx) << 4);
            offv[i] = key * RB + ((slot ^ vx) << 4);
        }
        const int wblk = wave * (KT / 4) / 16; // the wave's block of a tile
        auto copy = [&](auto IV, int t) { // tile t of K (0) or V (1) into its buffer
            constexpr int V = IV.value;
            uint32_t blk = (uint32_t)__builtin_amdgcn_readlane((int)tabv, (t - tw) * NB + wblk);
            if ((int64_t)blk >= a.n_blocks) blk = 0;
            const uint64_t at = ((uint64_t)blk * a.n_kv + kvh) * 16 * RB;
            const uint64_t src = (uint64_t)(V ? pv : pk) + at;
            const uint32_t(&off)[NC] = V ? offv : offk;
#pragma unroll
            for (int i = 0; i < NC; i++) {
                const uint32_t dst = (uint32_t)(uintptr_t)&kv[t & 1][V][(wave * (KT / 4) + RPC * i) * RB];
                lds_copy16(off[i], src, dst);
            }
        };
        // operand addresses within a buffer
        const int kx = (D == 64 ? (c >> 1) & 7 : c & 15);
        uint32_t ka[NJ], va[ND];
#pragma unroll
        for (int j = 0; j < NJ; j++) ka[j] = c * RB + (((2 * j + h) ^ kx) << 4);
        {
            const int i = lane & 15, r4 = i >> 2, vx = (D == 64 ? (r4 >> 1) & 1 : r4) << 2;
#pragma unroll
            for (int d = 0; d < ND; d++) {
                // (rows 16 t + 8 g + 4 h + r4: bit 1 of a row's number at D 64 is bit 1 of r4)
                const int chunk = 4 * d + 2 * ((lane >> 4) & 1) + ((i & 3) >> 1);
                va[d] = (4 * h + r4) * RB + ((chunk ^ vx) << 4) + 8 * (i & 1);
            }
        }
        at_f16v st[NK]; // scores: lane (c, h) holds row c, position KT t + 32 k + 8 (i / 4) + 4 h + i % 4 in st[k][i]
        auto score = [&](int t, at_f16v (&o)[NK]) {
            const unsigned char *kb = kv[t & 1][0];
#pragma unroll
            for (int k = 0; k < NK; k++) o[k] = at_f16v{};
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int k = 0; k < NK; k++)
                    o[k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                        *reinterpret_cast<const at_h8 *>(kb + ka[j] + 32 * k * RB), q[j], o[k], 0, 0, 0);
        };
        std::integral_constant<int, 0> K0;
        std::integral_constant<int, 1> V1;
        load_tab(t0);
        copy(K0, t0);
        copy(V1, t0);
        if (t0 < t1) copy(K0, t0 + 1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        score(t0, st);
        __syncthreads();
        for (int t = t0; t <= t1; t++) {
            // the tile's bad blocks
            if (tabbad) { // uniform
#pragma unroll 1
                for (int s = 0; s < NB; s++) {
                    const int b = t * NB + s;
                    const uint32_t blk = (uint32_t)__builtin_amdgcn_readlane((int)tabv, (t - tw) * NB + s);
                    if ((int64_t)blk >= a.n_blocks && valid && lo < 16 * b + 16 && hi > 16 * b) {
                        bad = true;
                        if (reports)
                            record_bad(a.status + CUCA_STATUS_KV_RANGE, (uint32_t)row, (uint32_t)max(16 * b, lo));
                    }
                }
            }
            // (a window of the table ends two tiles before its last entry's)
            if ((t + 3 - tw) * NB > 64) load_tab(t + 1);
            if (t < t1) copy(V1, t + 1);
            if (t + 1 < t1) copy(K0, t + 2);
            if (KT * t < whi && KT * (t + 2) > wlo) { // uniform over the wave
                if (KT * t < ilo || KT * (t + 1) > ihi) {
                    // position 32 k + 8 (i / 4) + i % 4 - off is in the row's range where that is < len
                    const uint32_t off = (valid ? lo : 0) - KT * t - 4 * h, len = valid ? hi - lo : 0x7fffffff;
#pragma unroll
                    for (int k = 0; k < NK; k++)
#pragma unroll
                        for (int i = 0; i < 16; i++)
                            st[k][i] = (uint32_t)(32 * k + 8 * (i >> 2) + (i & 3)) - off < len ? st[k][i] : -__builtin_huge_valf();
                }
                float bm = -__builtin_huge_valf();
#pragma unroll
                for (int k = 0; k < NK; k++)
#pragma unroll
                    for (int i = 0; i < 16; i++) bm = fmaxf(bm, st[k][i]);
                bm = fmaxf(bm, xor_partner(bm, 32)) * scale2;
                const bool up = bm > m + 3.0f;
                if (__ballot(up)) {
                    const float corr = up ? __builtin_amdgcn_exp2f(m - bm) : 1.0f;
                    l *= corr;
#pragma unroll
                    for (int d = 0; d < ND; d++) acc[d] *= corr;
                    m = up ? bm : m;
                }
                const float m12 = 12.0f - m;
                uint32_t ph[NK][8], pl[NK][8];
                at_f16v sn[NK];
                float s0 = 0.0f, s1 = 0.0f;
                auto weigh = [&](int n) { // score pair n's weights
                    const int k = n >> 3, i = 2 * (n & 7);
                    const float e0 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[k][i], scale2, m12));
                    const float e1 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[k][i + 1], scale2, m12));
                    s0 += e0;
                    s1 += e1;
                    const at_h2 p = __builtin_convertvector(at_f2{e0, e1}, at_h2);
                    ph[k][i >> 1] = __builtin_bit_cast(uint32_t, p);
                    pl[k][i >> 1] = __builtin_bit_cast(
                        uint32_t, __builtin_convertvector(at_f2{at_less<0>(e0, p), at_less<1>(e1, p)}, at_h2));
                };
                if (KT * (t + 1) < whi) { // uniform over the wave
                    // the next tile's scores on the matrix cores, this one's weights beside them
                    const unsigned char *kb = kv[(t + 1) & 1][0];
                    at_h8 kf[2][NK];
#pragma unroll
                    for (int k = 0; k < NK; k++) {
                        kf[0][k] = *reinterpret_cast<const at_h8 *>(kb + ka[0] + 32 * k * RB);
                    }
                    constexpr int PAIRS = NK * 8 / NJ < 1 ? 1 : NK * 8 / NJ; // score pairs a step
#pragma unroll
                    for (int j = 0; j < NJ; j++) {
#pragma unroll
                        for (int k = 0; k < NK && j + 1 < NJ; k++)
                            kf[(j + 1) & 1][k] = *reinterpret_cast<const at_h8 *>(kb + ka[j + 1] + 32 * k * RB);
#pragma unroll
                        for (int k = 0; k < NK; k++)
                            sn[k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[j & 1][k], q[j], j ? sn[k] : at_f16v{}, 0, 0, 0);
#pragma unroll
                        for (int n = j * PAIRS; n < (j + 1) * PAIRS && n < 8 * NK; n++) weigh(n);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else { // the wave's last tile: no next one; 16 keys past its ranges have weights of zero
#pragma unroll
                    for (int s = 0; s < KT / 16; s++) {
                        if (s && KT * t + 16 * s >= whi) {
#pragma unroll
                            for (int n = 4 * s; n < 4 * s + 4; n++) ph[n >> 3][n & 7] = pl[n >> 3][n & 7] = 0;
                            continue;
                        }
#pragma unroll
                        for (int n = 4 * s; n < 4 * s + 4; n++) {
                            weigh(n);
                            if (n & 1) __builtin_amdgcn_sched_barrier(0); // (spills otherwise)
                        }
                    }
#pragma unroll
                    for (int k = 0; k < NK; k++) sn[k] = st[k];
                }
                l += s0 + s1;
                const unsigned char *vb = kv[t & 1][1];
                typedef __attribute__((address_space(3))) at_s4 *lds4;
                auto value = [&](int d, int s) { // columns 32 d .. of keys 16 s .. 16 s + 15
                    const at_s4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(vb + va[d] + 16 * s * RB));
                    const at_s4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(vb + va[d] + (16 * s + 8) * RB));
                    return __builtin_bit_cast(at_h8, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
                };
                // a slice of 32 columns at a time from zero, added to its accumulators
                // beside the next slice's products
                constexpr int NS = KT / 16;
                at_f16v sum[2];
                at_h8 v[2];
                v[0] = value(0, 0);
#pragma unroll
                for (int d = 0; d < ND; d++)
#pragma unroll
                    for (int s = 0; s < NS; s++) {
                        const int n = d * NS + s;
                        if (n + 1 < ND * NS) v[(n + 1) & 1] = value((n + 1) / NS, (n + 1) % NS);
                        const uint32_t *hp = &ph[s >> 1][4 * (s & 1)], *lp = &pl[s >> 1][4 * (s & 1)];
                        const at_h8 bh = __builtin_bit_cast(at_h8, u32x4{hp[0], hp[1], hp[2], hp[3]});
                        const at_h8 bl = __builtin_bit_cast(at_h8, u32x4{lp[0], lp[1], lp[2], lp[3]});
                        sum[d & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[n & 1], bl, s ? sum[d & 1] : at_f16v{}, 0, 0, 0);
                        sum[d & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[n & 1], bh, sum[d & 1], 0, 0, 0);
                        if (d && s) { // (not behind the first: the slice's sums are not there yet)
#pragma unroll
                            for (int i = 16 * (s - 1) / (NS - 1); i < 16 * s / (NS - 1); i++)
                                acc[d - 1][i] += sum[(d - 1) & 1][i];
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                acc[ND - 1] += sum[(ND - 1) & 1];
#pragma unroll
                for (int k = 0; k < NK; k++) st[k] = sn[k];
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
    }
    l += __shfl_xor(l, 32);
    const bool zero = !valid || bad;
    _Float16 *orow =
        reinterpret_cast<_Float16 *>(a.out) + (int64_t)(in_call ? row : 0) * a.out_ld + (int64_t)head * D + 4 * h;
    bool fin = true;
    const float rl = 1.0f / l;
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            // the quotient: the reciprocal's product and its remainder
            const float o = acc[d][i] * rl;
            acc[d][i] = zero ? 0.0f : __builtin_fmaf(__builtin_fmaf(-o, l, acc[d][i]), rl, o);
            fin = fin && __builtin_fabsf(acc[d][i]) < __builtin_huge_valf();
        }
    // both halves of a row agree (the exchange outside the &&: behind it only
    // lanes whose own is true would ask, and the compiler takes the answer as known)
    const int fin_other = __shfl_xor((int)fin, 32);
    fin = fin && fin_other;
    // A weight of zero times an infinite or NaN value outside the row's range
    // is a NaN that the row must not see: such a row (its weights are finite)
    // is done again position by position.
    const bool again = in_call && !fin && __builtin_fabsf(l) < __builtin_huge_valf();
    if (in_call && !again) {
#pragma unroll
        for (int d = 0; d < ND; d++)
#pragma unroll
            for (int i = 0; i < 16; i += 4) {
                at_h4 o;
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = (_Float16)pin_f32(acc[d][i + e]);
                *reinterpret_cast<at_h4 *>(orow + 32 * d + 2 * i) = o;
            }
    }
    uint32_t todo = (uint32_t)__ballot(again);
    while (todo) { // uniform
        const int r = __builtin_ctz(todo);
        todo &= todo - 1;
        attn_rows_one<_Float16>(a, (tile * RT + rt) * 32 + r, head, lane);
    }
}

#define CUCA_ATTN_TILE(D, HW, KT, OCC)                                                                        \
    extern "C" __global__ __launch_bounds__(256, OCC) void cuca_attn_tile_f16_d##D##_h##HW(AttnRowsArgs a) {   \
        attn_tile_body<D, HW, KT>(a);                                                                         \
    }
CUCA_ATTN_TILE(64, 1, 64, 2)
CUCA_ATTN_TILE(64, 2, 64, 2)
CUCA_ATTN_TILE(64, 4, 64, 2)
CUCA_ATTN_TILE(128, 1, 64, 2)
CUCA_ATTN_TILE(128, 2, 64, 2)
CUCA_ATTN_TILE(128, 4, 64, 2)
CUCA_ATTN_TILE(256, 1, 64, 1)
CUCA_ATTN_TILE(256, 2, 64, 1)
CUCA_ATTN_TILE(256, 4, 64, 1)
