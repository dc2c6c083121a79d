// qms.hip -- the quantized matmul of several activation rows (decode batches
// of two and more, verification rows): the CPU engine's quantized matmul
// (QmmWeight, qmm.rs) bit for bit, as qmm.hip computes it, for tiles of two
// to four rows whose expanded form fits the LDS.
//
// The arithmetic is qmm.hip's: sixteen lane chains per weight row and
// activation row, lane l adding block by block, in row order, (float)P * (dw
// * dx) with the product and the sum rounded separately, P the exact integer
// pair sum; the fixed hsum tree at the end.  That is a dot, a multiply and an
// add a (block, lane, weight row, activation row), which bounds the kernel;
// everything else is shared or done once:
//
//  * A workgroup (4 to 16 waves) quantises the tile's activation rows once, whole,
//    into LDS (Acts::new, qmm.rs:1217-1343), for 32 to 64 weight rows; the
//    chunked kernel quantised a tile again for every 16.
//  * A wave is 16 chains x 4 lane groups, each lane RW weight rows (gate and
//    up for the GLU) by MJ activation rows: the weight pair is extracted once
//    for MJ dots, and the activation pairs (one 16-byte LDS read is four
//    blocks) serve RW.
//  * Weight pairs are exact f16 integers (the nibble or byte under an f16
//    exponent where it stands, the bias subtracted), so the LDS holds the
//    activation pairs alone, 2 bytes a value: four rows of 14336 values fit.
//  * dw * dx: lane l computes the products of block l of a group, and the
//    chain of block b reads them from lane b by a DPP row broadcast folded
//    into the multiply (as qmd.hip).
//  * Weight groups stream through a ring of D register slots.
//  * A matrix of few rows (down, o): the tile's rows are cut over JS waves of
//    the workgroup, since its chains are all the parallelism there is.
//
// What bounds it: the vector unit's issue rate (the chain arithmetic and the
// pair extraction), at four rows of the head 4.0 (Q4_0: 2.4) TB/s of weights;
// where a matrix has few rows, the chains' own latency.  Measured on MI355X
// against the chunked kernel at 3 / 4 / 8 rows of Q4_0, us: gate and up 14336
// x 4096 50.7 -> 29.2, 51.3 -> 34.4, 85.3 -> 61.1; down 4096 x 14336 36 ->
// 29.1, 36 -> 29.2, 50 -> 40.3; 4096 x 4096 12.3 -> 10.5 at four; the 128256 x
// 4096 head 215 -> 103, 217 -> 125, 424 -> 225 (Q8_0 234 -> 141 at four).
#include "common.h"

template <int FMT> __device__ static inline uint32_t qms_pair(const u32x4 &v, int i) {
    if (FMT == 0) { // dword i / 4: nibbles 4 (i % 4) and 16 + 4 (i % 4)
        const uint32_t d = v[i >> 2] >> ((i & 2) ? 8 : 0);
        const uint32_t p = (i & 1) ? and_or_b32(d, 0x00f000f0u, 0x54005400u) : and_or_b32(d, 0x000f000fu, 0x64006400u);
        const _Float16 bias = (_Float16)((i & 1) ? 72.0f : 1032.0f);
        return __builtin_bit_cast(uint32_t, __builtin_bit_cast(qmm_h2, p) - qmm_h2{bias, bias});
    }
    const uint32_t p = __builtin_amdgcn_perm(0x64646464u, v[i >> 1], (i & 1) ? 0x04030401u : 0x04020400u);
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(qmm_h2, p) - qmm_h2{(_Float16)1152.0f, (_Float16)1152.0f});
}

// The dots of one weight pair with MJ activation pairs, exact in f32, an
// instruction each: the builtin compiles to the accumulating form (v_dot2c)
// behind a move of zero, twice that.  The hardware wants three wait states
// between a dot and another instruction that reads or writes its result; the
// compiler does not know these for dots, so the block ends with them.
template <int MJ> __device__ static inline void qms_dots(uint32_t w, const uint32_t (&x)[MJ], float (&o)[MJ]) {
    if constexpr (MJ == 2)
        asm("v_dot2_f32_f16 %0, %2, %3, 0\n\tv_dot2_f32_f16 %1, %2, %4, 0\n\ts_nop 2"
            : "=&v"(o[0]), "=&v"(o[1])
            : "v"(w), "v"(x[0]), "v"(x[1]));
    else if constexpr (MJ == 3)
        asm("v_dot2_f32_f16 %0, %3, %4, 0\n\tv_dot2_f32_f16 %1, %3, %5, 0\n\tv_dot2_f32_f16 %2, %3, %6, 0\n\ts_nop 2"
            : "=&v"(o[0]), "=&v"(o[1]), "=&v"(o[2])
            : "v"(w), "v"(x[0]), "v"(x[1]), "v"(x[2]));
    else
        asm("v_dot2_f32_f16 %0, %4, %5, 0\n\tv_dot2_f32_f16 %1, %4, %6, 0\n\tv_dot2_f32_f16 %2, %4, %7, 0\n\t"
            "v_dot2_f32_f16 %3, %4, %8, 0\n\ts_nop 2"
            : "=&v"(o[0]), "=&v"(o[1]), "=&v"(o[2]), "=&v"(o[3])
            : "v"(w), "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]));
}
template <int MJ>
__device__ static inline void qms_dots2(uint32_t w, uint32_t u, const uint32_t (&x)[MJ], float (&o)[MJ], float (&p)[MJ]) {
    if constexpr (MJ == 1)
        asm("v_dot2_f32_f16 %0, %2, %4, 0\n\tv_dot2_f32_f16 %1, %3, %4, 0\n\ts_nop 2"
            : "=&v"(o[0]), "=&v"(p[0])
            : "v"(w), "v"(u), "v"(x[0]));
    else if constexpr (MJ == 2)
        asm("v_dot2_f32_f16 %0, %4, %6, 0\n\tv_dot2_f32_f16 %1, %4, %7, 0\n\t"
            "v_dot2_f32_f16 %2, %5, %6, 0\n\tv_dot2_f32_f16 %3, %5, %7, 0\n\ts_nop 2"
            : "=&v"(o[0]), "=&v"(o[1]), "=&v"(p[0]), "=&v"(p[1])
            : "v"(w), "v"(u), "v"(x[0]), "v"(x[1]));
    else if constexpr (MJ == 3)
        asm("v_dot2_f32_f16 %0, %6, %8, 0\n\tv_dot2_f32_f16 %1, %6, %9, 0\n\tv_dot2_f32_f16 %2, %6, %10, 0\n\t"
            "v_dot2_f32_f16 %3, %7, %8, 0\n\tv_dot2_f32_f16 %4, %7, %9, 0\n\tv_dot2_f32_f16 %5, %7, %10, 0\n\ts_nop 2"
            : "=&v"(o[0]), "=&v"(o[1]), "=&v"(o[2]), "=&v"(p[0]), "=&v"(p[1]), "=&v"(p[2])
            : "v"(w), "v"(u), "v"(x[0]), "v"(x[1]), "v"(x[2]));
    else
        asm("v_dot2_f32_f16 %0, %8, %10, 0\n\tv_dot2_f32_f16 %1, %8, %11, 0\n\t"
            "v_dot2_f32_f16 %2, %8, %12, 0\n\tv_dot2_f32_f16 %3, %8, %13, 0\n\t"
            "v_dot2_f32_f16 %4, %9, %10, 0\n\tv_dot2_f32_f16 %5, %9, %11, 0\n\t"
            "v_dot2_f32_f16 %6, %9, %12, 0\n\tv_dot2_f32_f16 %7, %9, %13, 0\n\ts_nop 2"
            : "=&v"(o[0]), "=&v"(o[1]), "=&v"(o[2]), "=&v"(o[3]), "=&v"(p[0]), "=&v"(p[1]), "=&v"(p[2]), "=&v"(p[3])
            : "v"(w), "v"(u), "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]));
}

// LDS of a tile: per activation row the pairs (a 272-byte row of 16 lanes x
// 16 bytes for every four blocks: the 16 bytes of padding keep the
// quantisation's writes of four such rows off the same banks) and, padded by
// a group, the block scales.
#define QMS_ROW4 17
#define QMS_LDS_BYTES(J, NBP) ((J) * ((NBP) / 4 * QMS_ROW4 * 16 + ((NBP) + 16) * 4) + 4 * QMS_ROW4 * 16)

template <int FMT, int RW> struct QmsSlot {
    u32x4 w[RW];
    uint32_t s[RW];
};

// MODE 0: plain (the LM head's cap when asked) or GLU; 3: the Q|K|V
// projection with RoPE and the paged K/V store.  MJ activation rows a wave, D
// ring slots.
template <typename T, int FMT, bool GLU, int MODE, int RW, int MJ, int D>
__device__ static inline void qms_body(const QmmArgs &a) {
    using F = QFmt<FMT>;
    constexpr int G = F::G;
    static_assert(!GLU || RW == 2, "the GLU's two rows are gate and up");
    extern __shared__ __attribute__((aligned(16))) unsigned char qms_lds[];
    const int js = a.js, tj = a.tile_rows; // waves a tile's rows are cut over; rows a tile
    const int ng = a.ng, nbp = ng * G, nq4 = nbp >> 2;
    u32x4 *xe = reinterpret_cast<u32x4 *>(qms_lds); // [row][nbp / 4][17]
    float *xsc = reinterpret_cast<float *>(xe + (MJ * js) * nq4 * QMS_ROW4 + 4 * QMS_ROW4); // [row][nbp + 16]
    const int tid = threadIdx.x, lt = tid & (CUCA_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / CUCA_WAVE);
    const int r = lt >> 4, l = lt & 15;
    // XCD-aware: the tiles of a weight block on one XCD (id % 8), in a row
    const int kq = (int)blockIdx.x >> 3, wb = kq / a.ntile * 8 + ((int)blockIdx.x & 7), tile = kq % a.ntile;
    if (wb >= a.nrb) return; // the whole workgroup
    const int j0 = tile * tj, nj = min(tj, a.m - j0);
    const int jw = (wave % js) * MJ; // the wave's first row of the tile

    // 1. The loads of the first four items a thread (item: 8 values, four
    // threads a block, the tile's rows end to end), then the ring's first
    // groups behind them, so that the quantisation runs under their latency.
    const int nt = (int)blockDim.x, waves = nt / CUCA_WAVE;
    const int task = wb * (waves / js) + wave / js;
    const int per = 4 * nbp, total = per * MJ * js, sub = tid & 3;
    float xv[4][8];
    auto fetch = [&](int i0) {
#pragma unroll
        for (int it = 0; it < 4; it++) {
            const int idx = i0 + it * nt + tid, j = idx / per, b = (idx - j * per) >> 2;
            if (j < nj && b < a.nb) {
                qmm_load8<T>(reinterpret_cast<const T *>(a.x) + (int64_t)(j0 + j) * a.ldx + (int64_t)b * 32 + sub * 8,
                             xv[it]);
            } else { // past the row, or a row past the tile's
#pragma unroll
                for (int e = 0; e < 8; e++) xv[it][e] = 0.0f;
            }
        }
    };
    fetch(0);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t nrec = (uint32_t)((int64_t)a.rows * a.row_bytes);
    const __amdgpu_buffer_rsrc_t rw =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(a.w), 0, (int)nrec, QMD_RSRC_W3);
    const __amdgpu_buffer_rsrc_t ru =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(GLU ? a.w_up : a.w), 0, (int)nrec, QMD_RSRC_W3);
    int row[RW]; // the lane's output columns (GLU: one)
    uint32_t vchunk[RW], vscale[RW];
#pragma unroll
    for (int i = 0; i < RW; i++) {
        row[i] = GLU ? task * 4 + r : task * 4 * RW + 4 * i + r;
        // a row past the matrix streams the last row; its result is not stored
        const uint32_t rb = (uint32_t)min(row[i], a.rows - 1) * (uint32_t)a.row_bytes;
        vchunk[i] = rb + F::SCB + 16 * l;
        vscale[i] = rb + 4 * ((l % G) >> 1);
    }
    typedef QmsSlot<FMT, RW> Slot;
    Slot ring[D];
    auto load = [&](Slot &s, int g) {
        const int so = (g < ng ? g : ng - 1) * F::GB; // wave-uniform: the scalar offset
#pragma unroll
        for (int i = 0; i < RW; i++) {
            s.w[i] = __builtin_amdgcn_raw_buffer_load_b128(GLU && i ? ru : rw, vchunk[i], so, 0);
            s.s[i] = __builtin_amdgcn_raw_buffer_load_b32(GLU && i ? ru : rw, vscale[i], so, 0);
        }
    };
    qmd_for<0, D>([&](auto I) {
        load(ring[I.value], I.value);
        __builtin_amdgcn_sched_barrier(0);
    });

    // 2. Quantise (as qmd.hip): the pairs of lanes base + q of block b, and
    // the block scales.
    for (int i0 = 0; i0 < total; i0 += 4 * nt) {
        if (i0) fetch(i0);
#pragma unroll
        for (int it = 0; it < 4; it++) {
            const int idx = i0 + it * nt + tid;
            if (i0 + it * nt >= total) break; // uniform: the tile is done
            const int j = idx / per, b = (idx - j * per) >> 2;
            float amax = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(xv[it][e]));
            amax = fmaxf(amax, xor_partner(amax, 1));
            amax = fmaxf(amax, xor_partner(amax, 2));
            const float d = amax / 127.0f;
            const float id = d != 0.0f ? 1.0f / d : 0.0f;
            uint32_t own[4], other[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                own[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(qmm_quant(xv[it][2 * i] * id),
                                                                                 qmm_quant(xv[it][2 * i + 1] * id)));
                other[i] = xor_partner_bits(own[i], 2);
            }
            if (idx < total) {
                // threads 0/1 own elements 0-7 / 8-15, threads 2/3 16-23 /
                // 24-31; sub < 2 writes lanes 8s..8s+3, sub >= 2 lanes
                // 8s+4..8s+7 (s = sub & 1)
                const bool low = sub < 2;
                const int base = 8 * (sub & 1) + (low ? 0 : 4);
                uint32_t *dst = reinterpret_cast<uint32_t *>(xe + (j * nq4 + (b >> 2)) * QMS_ROW4 + base) + (b & 3);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t lo = low ? own[q >> 1] : other[2 + (q >> 1)];
                    const uint32_t hi = low ? other[q >> 1] : own[2 + (q >> 1)];
                    dst[4 * q] = __builtin_amdgcn_perm(hi, lo, (q & 1) ? 0x07060302u : 0x05040100u);
                }
                if (sub == 0) xsc[j * (nbp + 16) + b] = j < nj && b < a.nb ? (float)(_Float16)d : 0.0f;
            }
        }
    }
    if (tid < 16 * MJ * js) // the group past each row, read and not used
        xsc[(tid >> 4) * (nbp + 16) + nbp + (tid & 15)] = 0.0f;
    __syncthreads();

    // 3. The stream.  The LDS operands of the next four blocks, and the next
    // group's dx, are read one step ahead (past the last group: the padding).
    const int sh = 16 * (l & 1);
    const u32x4 *xl = xe + jw * nq4 * QMS_ROW4 + l;
    const float *xsl = xsc + jw * (nbp + 16) + (l % G);
    constexpr int NS = G / 4; // steps of four blocks a group
    float acc[RW][MJ];
#pragma unroll
    for (int i = 0; i < RW; i++)
#pragma unroll
        for (int j = 0; j < MJ; j++) acc[i][j] = 0.0f;
    u32x4 cx[MJ];
    float cdx[MJ];
#pragma unroll
    for (int j = 0; j < MJ; j++) {
        cx[j] = xl[j * nq4 * QMS_ROW4];
        cdx[j] = xsl[j * (nbp + 16)];
    }
    auto consume = [&](const Slot &s, int g) {
        float sc[RW][MJ];
#pragma unroll
        for (int i = 0; i < RW; i++) {
            const float dw = qmv_h2f(s.s[i] >> sh);
#pragma unroll
            for (int j = 0; j < MJ; j++) sc[i][j] = dw * cdx[j];
        }
#pragma unroll
        for (int j = 0; j < MJ; j++) cdx[j] = xsl[j * (nbp + 16) + (g + 1) * G];
        qmd_for<0, NS>([&](auto S4) {
            const u32x4 *xn = xl + (g * NS + S4.value + 1) * QMS_ROW4;
            u32x4 nx[MJ];
#pragma unroll
            for (int j = 0; j < MJ; j++) nx[j] = xn[j * nq4 * QMS_ROW4];
            qmd_for<0, 4>([&](auto Q) {
                constexpr int b = 4 * S4.value + Q.value;
                float p[RW][MJ];
                uint32_t xp[MJ];
#pragma unroll
                for (int j = 0; j < MJ; j++) xp[j] = cx[j][Q.value];
                if constexpr (RW == 2)
                    qms_dots2<MJ>(qms_pair<FMT>(s.w[0], b), qms_pair<FMT>(s.w[1], b), xp, p[0], p[1]);
                else
                    qms_dots<MJ>(qms_pair<FMT>(s.w[0], b), xp, p[0]);
                // the dots, then the products, then the sums: the chains'
                // instructions in between hide each other's latency
#pragma unroll
                for (int i = 0; i < RW; i++)
#pragma unroll
                    for (int j = 0; j < MJ; j++) p[i][j] = p[i][j] * qmd_bcast<b>(sc[i][j]);
#pragma unroll
                for (int i = 0; i < RW; i++)
#pragma unroll
                    for (int j = 0; j < MJ; j++) acc[i][j] = acc[i][j] + p[i][j];
            });
            // pin these four blocks' arithmetic here (the chains are read
            // only at the end, so the compiler would sink it)
#pragma unroll
            for (int i = 0; i < RW; i++)
#pragma unroll
                for (int j = 0; j < MJ; j++) asm volatile("" : "+v"(acc[i][j]));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < MJ; j++) cx[j] = nx[j];
        });
    };
    const int nr = (ng + D - 1) / D;
    for (int R = 0; R + 1 < nr; R++) {
        qmd_for<0, D>([&](auto I) {
            consume(ring[I.value], R * D + I.value);
            load(ring[I.value], (R + 1) * D + I.value);
        });
    }
    const int rem = ng - (nr - 1) * D; // 1..D groups in the last round
    qmd_for<0, D>([&](auto I) {
        if (I.value < rem) consume(ring[I.value], (nr - 1) * D + I.value);
    });

#pragma unroll
    for (int j = 0; j < MJ; j++) {
        const int jt = jw + j; // row of the tile
#pragma unroll
        for (int i = 0; i < (GLU ? 1 : RW); i++) {
            float o = qmm_hsum(acc[i][j]);
            if constexpr (GLU) {
                float g = o, u = qmm_hsum(acc[RW - 1][j]);
                if (a.clamp > 0.0f) { // Glu::apply's clamp (cpu.rs:364-368)
                    g = fminf(g, a.clamp);
                    u = fminf(fmaxf(u, -a.clamp), a.clamp);
                }
                o = (a.gelu ? act_gelu_tanh(g) : act_silu(g)) * u;
            } else if (MODE == 0 && a.cap_flags) { // cap_logits (cpu.rs:2603-2617)
                if (a.cap_flags & 1) o = o * a.mul1 + 0.0f;
                if (a.cap_flags & 2) o = o * a.mul2 + 0.0f;
                if (a.cap_flags & 4) o = tanhf(o * a.softcap_inv + 0.0f) * a.softcap + 0.0f;
            }
            if constexpr (MODE == 3) {
                qmm_rope_kv_store<T>(a, min(j0 + jt, a.m - 1), jt < nj, (int64_t)(j0 + jt) * a.out_ld, row[i], l, o);
            } else {
                if (l == 0 && row[i] < a.rows && jt < nj)
                    reinterpret_cast<T *>(a.out)[(int64_t)(j0 + jt) * a.out_ld + row[i]] = to_stored<T>(o);
            }
        }
    }
}

// Up to 128 registers (four waves a SIMD; the four-row Q8_0 kernels use all of
// them, nothing is spilled): 8 waves a workgroup, or (one weight row a lane) up to
// 16.  D ring slots: a Q8_0 group is half a Q4_0 group's values, so four slots
// cover the time of two.
#define CUCA_QMS(NAME, ...)                                                                \
    extern "C" __global__ __launch_bounds__(8 * CUCA_WAVE, 4) void NAME(QmmArgs a) {        \
        qms_body<__VA_ARGS__>(a);                                                          \
    }
#define CUCA_QMS_SLIM(NAME, ...)                                                           \
    extern "C" __global__ __launch_bounds__(16 * CUCA_WAVE, 4) void NAME(QmmArgs a) {       \
        qms_body<__VA_ARGS__>(a);                                                          \
    }
// w1: one weight row a lane; w2: two; j2, j3, j4: activation rows a wave.
#define CUCA_QMS_SET(TN, T, FN, FMT, D)                                                    \
    CUCA_QMS_SLIM(cuca_qms_##TN##_##FN##_w1_j2, T, FMT, false, 0, 1, 2, 2 * D)                  \
    CUCA_QMS(cuca_qms_##TN##_##FN##_w2_j2, T, FMT, false, 0, 2, 2, D)                      \
    CUCA_QMS(cuca_qms_##TN##_##FN##_w2_j3, T, FMT, false, 0, 2, 3, D)                      \
    CUCA_QMS(cuca_qms_##TN##_##FN##_w2_j4, T, FMT, false, 0, 2, 4, D)                      \
    CUCA_QMS(cuca_qms_glu_##TN##_##FN##_j2, T, FMT, true, 0, 2, 2, D)                      \
    CUCA_QMS(cuca_qms_glu_##TN##_##FN##_j3, T, FMT, true, 0, 2, 3, D)                      \
    CUCA_QMS(cuca_qms_glu_##TN##_##FN##_j4, T, FMT, true, 0, 2, 4, D)                      \
    CUCA_QMS_SLIM(cuca_qms_rope_kv_##TN##_##FN##_j2, T, FMT, false, 3, 1, 2, 2 * D)
CUCA_QMS_SET(f32, float, q4_0, 0, 2)
CUCA_QMS_SET(f32, float, q8_0, 1, 4)
CUCA_QMS_SET(f16, _Float16, q4_0, 0, 2)
CUCA_QMS_SET(f16, _Float16, q8_0, 1, 4)
