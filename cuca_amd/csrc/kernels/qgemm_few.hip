// qgemm_few.hip -- the matrix-core quantized matmul (cuca_hip_qgemm's
// arithmetic class: weights f16(d * q), activations f16(x), f32 sums) for
// the batches of decode: up to 128 activation rows, where the weights'
// stream from HBM is the bound.
//
// A workgroup is 8 waves, each over one 16-row tile of the weight (the GLU
// form: waves 0-3 gate tiles, 4-7 the up tiles of the same columns), and
// NT * 16 tokens.  The weights go straight to registers, a packing group
// (512 or 256 values of a row) at a time, the next group's loads in flight
// while this one is computed.  The activations, which all 8 waves need, are
// read from the caller's rows (f32 or f16), rounded to f16 and staged in LDS
// a group at a time, double-buffered, one barrier a group.  (Read by each
// wave for itself they were the bound: at 32 rows every compute unit then
// pulled the whole batch through its L1 for 16 weight rows, 19.7 us for a
// 4096 x 4096 weight.)
//
// k order.  A k-step of v_mfma_f32_16x16x32_f16 is one 32-value block b: a
// lane (r, u) holds weight row r's values 4u..4u+3 and 16+4u..16+4u+3 of the
// block.  In the packed layout these are the dwords of chunks 4u..4u+3 (64
// contiguous bytes a lane a group, four 16-byte loads), and of an activation
// row two contiguous pieces of 4 values.  The chunks hold (l, l + 16) pairs;
// the 16-bit halves of two chunks' dwords are exchanged (v_perm) so that a
// weight operand's 8 values come in element order.
//
// Measured on MI355X, Q4_0, Llama-3-8B shapes, f32 rows, whole call, 32 / 64
// / 128 rows against the tiled kernel that served them before: gate+up with
// SwiGLU 24 / 37 us (47 / 69; at 128 rows qgemm.hip's tiles of 64 tokens take it),
// down 19 / 28 / 37 (27 / 32 / 46), q/o 13 / 20 / 24 (16 / 23 / 34), Q|K|V 15 / 22 /
// 29 (21 / 31 / 45).  What bounds it: one workgroup fits a compute unit (204
// registers at 32 tokens), two waves a SIMD that meet at a barrier a packing
// group, so loads, dequantisation (about 14 vector instructions a block and row
// tile) and products take turns; then, for the small weights, the second launch
// of the sums.  Two groups of weights or activations in flight instead of one: no
// faster.
//
// Few weight tiles (grid y > 1): k is cut into ranges of whole groups and
// each range's sums go to its own rows of the workspace, which
// cuca_qgemm_reduce_* adds in order.
#include "common.h"

typedef _Float16 qf_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 qf_h4 __attribute__((ext_vector_type(4)));
typedef _Float16 qf_h8 __attribute__((ext_vector_type(8)));
typedef float qf_acc __attribute__((ext_vector_type(4)));
typedef uint32_t qf_u2 __attribute__((ext_vector_type(2)));

template <int FMT> struct QfFmt;
template <> struct QfFmt<0> { static constexpr int G = 16, GB = 288, SCB = 32, BPD = 4; }; // Q4_0: 4 blocks a dword
template <> struct QfFmt<1> { static constexpr int G = 8, GB = 272, SCB = 16, BPD = 2; };  // Q8_0: 2

// A lane's part of a packing group of one weight row: chunks 4u..4u+3 and
// the group's scales.
template <int FMT> struct QfW {
    u32x4 c[4];
    u32x4 s[QfFmt<FMT>::G / 8];
};

template <int FMT> __device__ static inline void qf_load(const uint8_t *grp, int u, QfW<FMT> &o) {
    using F = QfFmt<FMT>;
#pragma unroll
    for (int i = 0; i < 4; i++) o.c[i] = *reinterpret_cast<const u32x4 *>(grp + F::SCB + 64 * u + 16 * i);
#pragma unroll
    for (int i = 0; i < F::G / 8; i++) o.s[i] = *reinterpret_cast<const u32x4 *>(grp + 16 * i);
}

// The weight operands of the BPD blocks of the exchanged dwords d (element
// pairs (0,1), (2,3), (16,17), (18,19) past 4u), scales sc: f16(d * q), one
// rounding.  A nibble is placed under an f16 exponent where it stands: bits
// 0-3 under 1024 (0x6400), bits 4-7 under 64 (0x5400: its unit is bit 4), the
// upper two after one shift by 8; then the bias is subtracted (exactly).
template <int FMT>
__device__ static inline void qf_operands(const uint32_t (&d)[4], const _Float16 (&sc)[QfFmt<FMT>::BPD],
                                          qf_h8 (&o)[QfFmt<FMT>::BPD]) {
#pragma unroll
    for (int i = 0; i < QfFmt<FMT>::BPD; i++) {
#pragma unroll
        for (int p = 0; p < 4; p++) {
            uint32_t v;
            float bias;
            if (FMT == 0) {
                const uint32_t w = i < 2 ? d[p] : d[p] >> 8;
                v = i & 1 ? and_or_b32(w, 0x00f000f0u, 0x54005400u) : and_or_b32(w, 0x000f000fu, 0x64006400u);
                bias = i & 1 ? 72.0f : 1032.0f;
            } else {
                v = __builtin_amdgcn_perm(0x64646464u, d[p], i == 0 ? 0x04020400u : 0x04030401u);
                bias = 1152.0f;
            }
            const qf_h2 w2 = (__builtin_bit_cast(qf_h2, v) - qf_h2{(_Float16)bias, (_Float16)bias}) * qf_h2{sc[i], sc[i]};
            o[i][2 * p] = w2.x;
            o[i][2 * p + 1] = w2.y;
        }
    }
}

// Eight activations as f16.
__device__ static inline qf_h4 qf_half(f32x4 v) {
    return qf_h4{(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
}
__device__ static inline qf_h4 qf_half(qf_h4 v) { return v; }
template <typename X> struct QfPiece;
template <> struct QfPiece<float> { typedef f32x4 T; };
template <> struct QfPiece<_Float16> { typedef qf_h4 T; };

// X: the activations read (f32, f16); T: the output.  NT: tiles of 16 tokens.
template <typename X, typename T, int FMT, int NT, bool GLU>
__device__ static inline void qgemm_few_body(const QGemmFewArgs &a) {
    using F = QfFmt<FMT>;
    typedef typename QfPiece<X>::T Piece; // 4 activations
    constexpr int KS = F::G * 32;               // values of k a stage: a group
    constexpr int XST = KS + 4;              // a token's row in LDS: 8 bytes past a multiple of 128
    constexpr int PR = KS / 4;                  // pieces of 4 values a token's row
    constexpr int PPT = NT * 16 * (KS / 4) / 512; // pieces a thread stages
    __shared__ __attribute__((aligned(16))) _Float16 xs[2][NT * 16 * XST];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, u = lane >> 4;
    // workgroup id = 8 (n_ct (wt / 8) + token tile) + wt % 8: the token tiles
    // of a weight tile run on one XCD and read its weights from HBM once.  Fewer
    // than eight weight tiles would leave XCDs idle: there they go round in turn.
    const int id = blockIdx.x, chunk = id >> 3;
    const bool turn = a.n_tile < 8;
    const int wt = turn ? id % a.n_tile : chunk / a.n_ct * 8 + (id & 7), ct = turn ? id / a.n_tile : chunk % a.n_ct;
    if (wt >= a.n_tile || ct >= a.n_ct) return; // the whole workgroup
    const int t0 = ct * (NT * 16);
    const int c0 = GLU ? wt * 64 + (wave & 3) * 16 : wt * 128 + wave * 16; // the wave's first output column
    const int row = min(c0 + r, a.rows - 1);
    const uint8_t *wr = (GLU && wave >= 4 ? a.w_up : a.w) + (int64_t)row * a.row_bytes;
    const int g0 = (int)blockIdx.y * a.gs, g1 = min(a.ng, g0 + a.gs); // this split's groups
    if (g0 >= g1) return;
    // a thread's pieces of a stage: piece p = tid + 512 i, token p / PR, values 4 (p % PR)
    const X *xr[PPT];
#pragma unroll
    for (int i = 0; i < PPT; i++) {
        const int p = tid + 512 * i, tok = t0 + p / PR;
        xr[i] = reinterpret_cast<const X *>(a.x) + (int64_t)min(tok, a.m - 1) * a.ldx + 4 * (p % PR);
    }
    // the pieces of a group; past the row's end (its last group) they are
    // staged as zeros, as the packed weights are there
    struct Pieces {
        Piece v[PPT];
    };
    auto fetch = [&](int g, Pieces &px) {
        const int k = min(g, g1 - 1) * KS;
#pragma unroll
        for (int i = 0; i < PPT; i++) {
            const int p4 = 4 * ((tid + 512 * i) % PR);
            px.v[i] = *reinterpret_cast<const Piece *>(xr[i] + (k + p4 < a.k ? k : -p4));
        }
    };
    auto stage = [&](int g, const Pieces &px, _Float16 *dst) {
#pragma unroll
        for (int i = 0; i < PPT; i++) {
            const int p = tid + 512 * i, p4 = 4 * (p % PR);
            qf_h4 v = qf_half(px.v[i]);
            if (min(g, g1 - 1) * KS + p4 >= a.k) v = qf_h4{};
            *reinterpret_cast<qf_h4 *>(dst + p / PR * XST + p4) = v;
        }
    };
    qf_acc acc[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) acc[j] = qf_acc{0.0f, 0.0f, 0.0f, 0.0f};
    // One group from register slot w and LDS buffer xc, while group g + 2's
    // weights replace it and group g + 1's activations are staged.  The slots
    // are named, not rotated: moving a slot's registers waits for its loads.
    const uint8_t *wlast = wr + (int64_t)(g1 - 1) * F::GB;
    auto grp_at = [&](int g) { return g < g1 ? wr + (int64_t)g * F::GB : wlast; };
    auto group = [&](int g, QfW<FMT> &w, Pieces &px, const _Float16 *xc, _Float16 *xn) {
        const _Float16 *xb = xc + r * XST + 4 * u;
        constexpr int XB = F::BPD < 4 || NT == 4 ? 4 : 8; // blocks whose operands are held
        qf_h8 xv[XB][NT];
        auto read = [&](int b) {
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const _Float16 *xp = xb + 16 * j * XST + 32 * b;
                xv[b % XB][j] = __builtin_shufflevector(
                    *reinterpret_cast<const qf_h4 *>(xp), *reinterpret_cast<const qf_h4 *>(xp + 16), 0, 1, 2, 3, 4, 5, 6, 7);
            }
        };
        // (unconditional, the last group again past the end: behind a branch
        // the compiler cannot count the loads in flight and waits for all)
        stage(g + 1, px, xn);
        fetch(g + 2, px);
#pragma unroll
        for (int b = 0; b < XB; b++) read(b);
#pragma unroll
        for (int t = 0; t < 4; t++) { // dword of the chunks
            uint32_t d[4];
            d[0] = __builtin_amdgcn_perm(w.c[1][t], w.c[0][t], 0x05040100u);
            d[1] = __builtin_amdgcn_perm(w.c[3][t], w.c[2][t], 0x05040100u);
            d[2] = __builtin_amdgcn_perm(w.c[1][t], w.c[0][t], 0x07060302u);
            d[3] = __builtin_amdgcn_perm(w.c[3][t], w.c[2][t], 0x07060302u);
            _Float16 sc[F::BPD];
#pragma unroll
            for (int i = 0; i < F::BPD; i++) {
                const int b = t * F::BPD + i; // block of the group
                const uint32_t s2 = w.s[b >> 3][(b & 7) >> 1];
                sc[i] = __builtin_bit_cast(_Float16, (uint16_t)((b & 1) ? s2 >> 16 : s2 & 0xffffu));
            }
            qf_h8 wv[F::BPD];
            qf_operands<FMT>(d, sc, wv);
#pragma unroll
            for (int i = 0; i < F::BPD; i++) {
                const int b = t * F::BPD + i;
#pragma unroll
                for (int j = 0; j < NT; j++)
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[i], xv[b % XB][j], acc[j], 0, 0, 0);
                if (b + XB < F::G) read(b + XB);
            }
            __builtin_amdgcn_sched_barrier(0); // operands are read no further ahead
        }
        qf_load<FMT>(grp_at(g + 2), u, w);
        __syncthreads();
    };
    QfW<FMT> w0, w1;
    Pieces px;
    fetch(g0, px);
    qf_load<FMT>(grp_at(g0), u, w0);
    stage(g0, px, xs[0]);
    fetch(g0 + 1, px);
    qf_load<FMT>(grp_at(g0 + 1), u, w1);
    __syncthreads();
    int g = g0;
    for (; g + 1 < g1; g += 2) {
        group(g, w0, px, xs[0], xs[1]);
        group(g + 1, w1, px, xs[1], xs[0]);
    }
    if (g < g1) group(g, w0, px, xs[0], xs[1]);
    // accumulator e of lane (r, u): weight row 4u + e, token r of the tile
    if (gridDim.y > 1) { // partial rows: [split][gate, up][m][rows] f32
        float *part = a.part + ((int64_t)(int)blockIdx.y * (GLU ? 2 : 1) + (GLU ? wave >> 2 : 0)) * a.m * a.rows;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const int tok = t0 + 16 * j + r, c = c0 + 4 * u;
            if (tok >= a.m) continue;
            float *o = part + (int64_t)tok * a.rows + c;
            if (a.rows % 4 == 0 && c < a.rows) {
                *reinterpret_cast<f32x4 *>(o) = acc[j];
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (c + e < a.rows) o[e] = acc[j][e];
            }
        }
        return;
    }
    T *out = reinterpret_cast<T *>(a.out);
    if (GLU) { // the up sums through LDS to the wave of their gate columns
        float *us = reinterpret_cast<float *>(&xs[0][0]);
        if (wave >= 4) {
#pragma unroll
            for (int j = 0; j < NT; j++) *reinterpret_cast<f32x4 *>(us + (((wave - 4) * NT + j) * 64 + lane) * 4) = acc[j];
        }
        __syncthreads();
        if (wave >= 4) return;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const f32x4 up = *reinterpret_cast<const f32x4 *>(us + ((wave * NT + j) * 64 + lane) * 4);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float gv = acc[j][e], uv = up[e];
                if (a.clamp > 0.0f) { // Glu::apply's clamp (cpu.rs:364-368)
                    gv = fminf(gv, a.clamp);
                    uv = fminf(fmaxf(uv, -a.clamp), a.clamp);
                }
                acc[j][e] = (a.gelu ? act_gelu_tanh(gv) : act_silu(gv)) * uv;
            }
        }
    }
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int tok = t0 + 16 * j + r;
        if (tok >= a.m) continue;
        T *o = out + (int64_t)tok * a.out_ld + c0 + 4 * u;
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (c0 + 4 * u + e < a.rows) o[e] = to_stored<T>(acc[j][e]);
    }
}

#define CUCA_QGEMM_FEW(NAME, X, T, FMT, NT, GLU)                                            \
    extern "C" __global__ __launch_bounds__(512, 2) void NAME(QGemmFewArgs a) {             \
        qgemm_few_body<X, T, FMT, NT, GLU>(a);                                              \
    }
#define CUCA_QGEMM_FEW_NT(XN, X, TN, T, NT)                                                 \
    CUCA_QGEMM_FEW(cuca_qgemm_few_##XN##_##TN##_q4_0_n##NT, X, T, 0, NT, false)             \
    CUCA_QGEMM_FEW(cuca_qgemm_few_##XN##_##TN##_q8_0_n##NT, X, T, 1, NT, false)             \
    CUCA_QGEMM_FEW(cuca_qgemm_few_glu_##XN##_##TN##_q4_0_n##NT, X, T, 0, NT, true)          \
    CUCA_QGEMM_FEW(cuca_qgemm_few_glu_##XN##_##TN##_q8_0_n##NT, X, T, 1, NT, true)
CUCA_QGEMM_FEW_NT(f32, float, f32, float, 1)
CUCA_QGEMM_FEW_NT(f32, float, f32, float, 2)
CUCA_QGEMM_FEW_NT(f16, _Float16, f32, float, 1)
CUCA_QGEMM_FEW_NT(f16, _Float16, f32, float, 2)
CUCA_QGEMM_FEW_NT(f16, _Float16, f32, float, 4)
CUCA_QGEMM_FEW_NT(f16, _Float16, f16, _Float16, 1)
CUCA_QGEMM_FEW_NT(f16, _Float16, f16, _Float16, 2)
CUCA_QGEMM_FEW_NT(f16, _Float16, f16, _Float16, 4)

// Rows rounded to f16 (RNE) [m][k], eight values a thread (k is a multiple of
// 32); vec: the rows start 16-byte aligned.
template <typename X> __device__ static inline void qgemm_rows_body(const QGemmFewArgs &a) {
    const int64_t t = (int64_t)blockIdx.x * CUCA_BLOCK + threadIdx.x;
    const int64_t per = a.k / 8;
    if (t >= (int64_t)a.m * per) return;
    const int64_t r = t / per, c = (t - r * per) * 8;
    const X *src = reinterpret_cast<const X *>(a.x) + r * a.ldx + c;
    qf_h8 h;
    if (a.vec) {
        if (sizeof(X) == 4) {
            const f32x4 v0 = reinterpret_cast<const f32x4 *>(src)[0], v1 = reinterpret_cast<const f32x4 *>(src)[1];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                h[i] = (_Float16)v0[i];
                h[4 + i] = (_Float16)v1[i];
            }
        } else {
            h = *reinterpret_cast<const qf_h8 *>(src);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) h[i] = (_Float16)(float)src[i];
    }
    *reinterpret_cast<qf_h8 *>(reinterpret_cast<_Float16 *>(a.out) + r * a.k + c) = h;
}
extern "C" __global__ __launch_bounds__(CUCA_BLOCK) void cuca_qgemm_rows_f32(QGemmFewArgs a) { qgemm_rows_body<float>(a); }
extern "C" __global__ __launch_bounds__(CUCA_BLOCK) void cuca_qgemm_rows_f16(QGemmFewArgs a) {
    qgemm_rows_body<_Float16>(a);
}
