// qgemm.hip -- the quantized matmul for many activation rows (prefill, large
// batches) on gfx950's matrix cores: out[t][n] = x[t] . w[n] with the Q4_0 /
// Q8_0 weights dequantised to f16 and the activations rounded to f16, f32
// accumulation (v_mfma_f32_16x16x32_f16).  Up to 128 rows: qgemm_few.hip.
//
// This is the reference GPU engine's arithmetic class for its dense paths
// (dense_gemv_kernel / dense_dequant_kernel, moe_kernel.rs:1414-1600: float
// products of dequantised weights and unquantised activations), not the CPU
// engine's bits (cuca_hip_qmm keeps those).  Each weight is f16(d * q) and
// each activation f16(x), one rounding each; the error is bounded by
// (2^-10 + k 2^-24) sum_i |w_i x_i| and the parity tests hold it to that.
//
// Tiling.  A workgroup of 4 waves computes 256 weight rows (the GLU form: 128
// gate rows and the 128 up rows of the same columns) x NT * 16 tokens; a wave
// takes 64 rows (32 gate + 32 up) x every token of the tile, 4 x NT tiles of
// 16 x 16.  Each weight is dequantised once a workgroup, in the registers of
// the wave that multiplies it, and each activation operand that a wave reads
// from LDS feeds four products: 32 rows a wave (two products a read) had the
// LDS busy with the reads all the time.  Two workgroups fit a compute unit,
// two waves a SIMD, so that one wave's dequantisation (about 14 vector
// instructions an operand of 8 products) runs under the other's products.
// Down of the routed experts, whose grids are smaller, also takes 128 weight rows
// a workgroup, 32 a wave (RI = 2; runtime.cpp, moe_qgemm_common).
//
// k order.  The weights are read in the packed layout of qmm.hip.  A dot
// product may sum its terms in any order, so the k index of the operands is
// the packed layout's own.  k runs in chunks of 128 values, 4 k-steps of 32.
// A lane (r, u) of a wave loads 16 bytes of row r: lane chunk c0 + u of the
// group (c0 = the first of the k-chunk's lane chunks), whose dword t holds
// the pairs of the blocks BPD t ..; the four lanes u of a row then exchange
// dwords (a 4 x 4 transpose, two permlane swaps of two registers each) so
// that lane u holds dword u of the chunks c0 .. c0 + 3.  So a lane needs the
// scales of the blocks BPD u .. only, and one 16-byte load is four k-steps.
// Slot j of lane u in k-step s is then true position
//   Q4_0 (512-value groups, a k-chunk = quarter q):
//        512 g + 128 u + 16 j + 4 q + s
//   Q8_0 (256-value groups, a k-chunk = half q, two loads a chunk):
//        256 g + 64 u + 16 (j % 4) + 8 q + 2 s + j / 4
// and the activations are rewritten in that order once a call
// (qgemm_prep_body), then copied into LDS directly, a k-chunk ahead.
//
// Measured on MI355X, Q4_0, Llama-3-8B shapes at 4096 f16 rows, whole call:
// gate+up with SwiGLU 853-881 us (1.09-1.13 PFLOP/s, 0.44 of the dense peak;
// 1260 for the kernel before this one, 128 x 128 tiles of 32 x 32 x 16
// products), down 468-483 (794), q/o 142-149 (219).  Q8_0: 990-1000, 543-550
// and 165-167.  What bounds it: the products (two waves a SIMD take turns);
// Q8_0's loads carry twice the bytes.  Not faster: a second register set for the
// next chunk's weights spilled.  Tiles of 64 tokens (half the products a
// dequantised weight) where tiles of 128 leave compute units idle and k is too
// short to split, and past 64 rows where qgemm_few.hip's tiles take turns
// (runtime.cpp, qgemm_common); where k splits they are slower (down at 777 rows
// 136 -> 150 us).
#include "common.h"
#include <type_traits>

typedef _Float16 qg_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 qg_h8 __attribute__((ext_vector_type(8)));
typedef float qg_acc __attribute__((ext_vector_type(4)));
typedef uint32_t qg_u2 __attribute__((ext_vector_type(2)));

#define QG_KC 128         // values per k-chunk: 4 k-steps of 32

template <int FMT> struct QgFmt;
template <> struct QgFmt<0> { static constexpr int GB = 288, SCB = 32, KCG = 4, UNITS = 1; }; // Q4_0
template <> struct QgFmt<1> { static constexpr int GB = 272, SCB = 16, KCG = 2, UNITS = 2; }; // Q8_0

// A lane's weights of a k-chunk of one 16-row tile (Q4_0 one 16-byte load,
// Q8_0 two), and its scales there (Q4_0: blocks 4u..4u+3; Q8_0: 2u, 2u+1, in
// .x).
template <int FMT> struct QgW {
    u32x4 c[QgFmt<FMT>::UNITS];
    qg_u2 s;
};
// tile: a tile's first row, in scalar registers, with the bytes that its rows
// have (rows past the matrix read as zeros: the buffer's bounds check); off:
// the lane's row of it plus 16 u.  One vector register addresses all four
// tiles, where global loads took a pair for each.
struct QgTile {
    const uint8_t *p;
    uint32_t bytes;
};
__device__ static inline __amdgpu_buffer_rsrc_t qg_rsrc(const QgTile &t, int64_t at) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(t.p + at), 0, (int)t.bytes, 0x00020000);
}
template <int FMT> __device__ static inline u32x4 qg_load(const QgTile &t, int kc, int unit, uint32_t off) {
    using F = QgFmt<FMT>;
    const int part = (kc % F::KCG) * F::UNITS + unit; // four 64-byte pieces a group in both formats
    return __builtin_amdgcn_raw_buffer_load_b128(qg_rsrc(t, (int64_t)(kc / F::KCG) * F::GB + F::SCB + 64 * part), (int)off,
                                                 0, 0);
}
template <int FMT> __device__ static inline qg_u2 qg_load_scales(const QgTile &t, int kc, uint32_t off, int u) {
    using F = QgFmt<FMT>;
    const __amdgpu_buffer_rsrc_t grp = qg_rsrc(t, (int64_t)(kc / F::KCG) * F::GB);
    if (FMT == 0) return __builtin_amdgcn_raw_buffer_load_b64(grp, (int)(off - 8u * (uint32_t)u), 0, 0);
    return qg_u2{__builtin_amdgcn_raw_buffer_load_b32(grp, (int)(off - 12u * (uint32_t)u), 0, 0), 0u};
}

// Lane u's register t <-> lane t's register u (u the lane's row of 16).
__device__ static inline void qg_transpose(u32x4 &v) {
    const auto p02 = __builtin_amdgcn_permlane32_swap(v.x, v.z, false, false);
    const auto p13 = __builtin_amdgcn_permlane32_swap(v.y, v.w, false, false);
    const auto a = __builtin_amdgcn_permlane16_swap(p02[0], p13[0], false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(p02[1], p13[1], false, false);
    v = u32x4{a[0], a[1], b[0], b[1]};
}

__device__ static inline _Float16 qg_scale(qg_u2 s, int i) {
    const uint32_t w = i < 2 ? s.x : s.y;
    return __builtin_bit_cast(_Float16, (uint16_t)((i & 1) ? (w >> 16) : (w & 0xffffu)));
}

// The weight operand of k-step s (compile-time s), from its transposed
// dwords.  Q4_0: a nibble is placed under an f16 exponent where it stands
// (bits 0-3 under 1024, bits 4-7 under 64, the upper two after one shift),
// the bias subtracted (exactly), the block scale multiplied: f16(d * q), one
// rounding.
template <int FMT> __device__ static inline qg_h8 qg_dequant(const QgW<FMT> &w, int s) {
    qg_h8 o;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t v;
        float bias;
        _Float16 d;
        if (FMT == 0) {
            const uint32_t x = i < 2 ? w.c[0][s] : w.c[0][s] >> 8;
            v = i & 1 ? and_or_b32(x, 0x00f000f0u, 0x54005400u) : and_or_b32(x, 0x000f000fu, 0x64006400u);
            bias = i & 1 ? 72.0f : 1032.0f;
            d = qg_scale(w.s, i);
        } else { // the biased bytes under 0x64
            v = __builtin_amdgcn_perm(0x64646464u, w.c[(s >> 1) % QgFmt<FMT>::UNITS][2 * (s & 1) + (i >> 1)],
                                      i & 1 ? 0x04030401u : 0x04020400u);
            bias = 1152.0f;
            d = qg_scale(w.s, i & 1);
        }
        const qg_h2 p = (__builtin_bit_cast(qg_h2, v) - qg_h2{(_Float16)bias, (_Float16)bias}) * qg_h2{d, d};
        o[2 * i] = p.x;
        o[2 * i + 1] = p.y;
    }
    return o;
}

// True position of slot 0 of unit v = 4 s + u (k-step s, lane u) of k-chunk
// kc, and of slot j.
template <int FMT> __device__ static inline int qg_slot(int kc, int v, int j) {
    const int s = v >> 2, u = v & 3;
    if (FMT == 0) return 512 * (kc >> 2) + 128 * u + 16 * j + 4 * (kc & 3) + s;
    return 256 * (kc >> 1) + 64 * u + 16 * (j & 3) + 8 * (kc & 1) + 2 * s + (j >> 2);
}

__device__ static inline void qgemm_load8f(const float *p, float (&v)[8]) {
    const f32x4 a = reinterpret_cast<const f32x4 *>(p)[0];
    const f32x4 b = reinterpret_cast<const f32x4 *>(p)[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// The activations rewritten once per call, before the matmul: f16, in the
// slot order of the format (xp [n_ct * TM][kp], kp = 128 per k-chunk; zero
// past k and in the rows past m, up to the whole tile).  One thread per unit
// (token, k-chunk, v = 4 k-step + lane u) of 8 values.
template <typename T, int FMT> __device__ static inline void qgemm_prep_body(const QGemmArgs &a) {
    const int64_t u = (int64_t)blockIdx.x * CUCA_BLOCK + threadIdx.x;
    const int64_t per_row = (int64_t)a.nkc * 16;
    if (u >= (int64_t)a.mp * per_row) return;
    const int tok = (int)(u / per_row), rem = (int)(u - (int64_t)tok * per_row);
    const int kc = rem >> 4, v = rem & 15;
    const T *row = reinterpret_cast<const T *>(a.x) + (int64_t)(tok < a.m ? tok : 0) * a.ldx;
    qg_h8 o;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int k = qg_slot<FMT>(kc, v, j);
        o[j] = tok < a.m && k < a.k ? (_Float16)(float)row[k] : (_Float16)0.0f;
    }
    *reinterpret_cast<qg_h8 *>(a.xp + (int64_t)tok * a.kp + (int64_t)kc * QG_KC + 8 * v) = o; // xp: f16 bits
}

// SPLIT: workgroup (tile, split) takes k-chunks [split * kcs, ...) and
// writes its f32 sums to the partial rows of the workspace (qgemm_reduce
// adds the splits in order and applies the epilogue); otherwise the
// epilogue is applied here.
template <typename T, int FMT, int NT, bool GLU, int ACT, bool SPLIT, int MOE = 0, int RI = 4>
__device__ static inline void qgemm_body(const QGemmArgs &a) {
    using F = QgFmt<FMT>;
    constexpr int TM = NT * 16;
    static_assert(!GLU || RI == 4, "gate, gate, up, up");
    constexpr int COLS = 64 * RI / (GLU ? 2 : 1); // output columns of a workgroup
    // two buffers of a k-chunk's activations: rows of 256 bytes, 16-byte unit
    // v of row R at unit v ^ (R & 7), so that the reads of 8 rows at one unit
    // fall in different banks (rows r and r + 8 of a fragment share theirs: a read
    // takes 8 cycles, and the LDS pipe is active a quarter of the launch)
    __shared__ __attribute__((aligned(16))) _Float16 xs[2 * TM * QG_KC];
    const int split = SPLIT ? (int)blockIdx.y : 0;
    // XCD x (workgroups x, x + 8, ...) takes row tiles x, x + 8, ... in
    // groups of 8; a group's workgroups take its row tiles in turn, token
    // tile by token tile, so that the workgroups resident on the XCD at once
    // share their weight and activation tiles in its L2.  Fewer than eight
    // row tiles would leave XCDs idle: there the tiles go round in turn (256 x
    // 2048 at 777 rows 27.7 -> 23.5 us).
    const int id = blockIdx.x, xcd = id & 7, kq = id >> 3;
    int ct, rt;
    if (a.n_rt < 8) {
        ct = id / a.n_rt;
        rt = id - ct * a.n_rt;
    } else {
        const int n_rx = (a.n_rt - xcd + 7) >> 3; // row tiles of this XCD
        const int g = kq / (8 * a.n_ct), w = kq - g * 8 * a.n_ct;
        const int gsz = min(8, n_rx - 8 * g);
        if (gsz <= 0) return;
        ct = w / gsz;
        rt = (8 * g + (w - ct * gsz)) * 8 + xcd;
    }
    if (ct >= a.n_ct) return;
    // routed experts: the tile's expert and pairs (uniform); tiles past the
    // last are empty
    int ex = 0, p0 = 0, np = 0;
    if (MOE) {
        ex = a.tile_e[ct];
        if (ex < 0) return;
        p0 = a.tile_p0[ct];
        np = a.tile_n[ct];
    }
    const int kc0 = split * a.kcs;
    const int kc1 = min(a.nkc, kc0 + a.kcs);
    if (kc0 >= kc1) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, u = lane >> 4;
    const int tok0 = ct * TM;
    const int n0 = rt * COLS + wave * (COLS / 4); // the wave's first output column
    // the wave's 16-row tiles (GLU: gate, gate, up, up of the same columns)
    QgTile tile[RI];
#pragma unroll
    for (int i = 0; i < RI; i++) {
        const int r0 = n0 + 16 * (GLU ? i & 1 : i); // uniform
        const int left = max(0, min(16, a.rows - r0));
        const uint64_t p = (uint64_t)(uintptr_t)(GLU && i >= 2 ? a.w_up : a.w) + (uint64_t)((int64_t)r0 * a.row_bytes) +
                           (MOE ? (uint64_t)((int64_t)ex * a.estride) : 0);
        const uint64_t ps = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(p >> 32)) << 32) |
                            (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)p);
        tile[i].p = reinterpret_cast<const uint8_t *>((uintptr_t)ps);
        const uint64_t bytes = (uint64_t)left * (uint64_t)a.row_bytes; // (16 rows of k = 2^28 pass 32 bits; 15 do not)
        tile[i].bytes = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(bytes < 0xffffffffull ? bytes : 0xffffffffull));
    }
    const uint32_t woff = (uint32_t)r * (uint32_t)a.row_bytes + 16u * (uint32_t)u;
    // The copies: wave w fills LDS rows w TM / 4 .., four rows of 256 bytes an
    // instruction (lane L: row L / 16 of them, unit L % 16, from source unit
    // (L % 16) ^ (row & 7)).  The waits are written out below.
    uint32_t off[2];
#pragma unroll
    for (int i = 0; i < 2; i++)
        off[i] = 2u * ((uint32_t)(lane >> 4) * (uint32_t)a.kp + 8u * (uint32_t)((lane & 15) ^ ((4 * i + (lane >> 4)) & 7)));
    const uint64_t xv = (uint64_t)(uintptr_t)a.xp + 2 * (uint64_t)((int64_t)(tok0 + wave * (TM / 4)) * a.kp);
    const uint64_t xb = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(xv >> 32)) << 32) |
                        (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)xv);
    const uint64_t x4 = 8 * (uint64_t)a.kp; // bytes of four rows
    auto copy = [&](int kc, int buf) {
#pragma unroll
        for (int i = 0; i < TM / 16; i++) {
            const uint64_t src = xb + i * x4 + (uint64_t)kc * (2 * QG_KC);
            const uint32_t dst = (uint32_t)(uintptr_t)&xs[(buf * TM + wave * (TM / 4) + 4 * i) * QG_KC];
            lds_copy16(off[i & 1], src, dst);
        }
    };
    qg_acc acc[RI][NT];
#pragma unroll
    for (int i = 0; i < RI; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = qg_acc{};
    // weights: a tile's next chunk is requested into its own registers, right
    // after the last operand made from them (a second register set, a chunk
    // ahead, spilled)
    QgW<FMT> wv[RI];
    auto load = [&](int kc, int i, int unit) {
        const int c = kc < kc1 ? kc : kc1 - 1; // (the last again past the end, unused)
        wv[i].c[unit] = qg_load<FMT>(tile[i], c, unit, woff);
        if (unit == F::UNITS - 1) wv[i].s = qg_load_scales<FMT>(tile[i], c, woff, u);
    };
    // unit (4 s + u) ^ (r & 7) of row 16 j + r: the k-step's part is s ^ (r >>
    // 2 & 1), so two addresses and constant offsets serve every read
    const _Float16 *xe = xs + r * QG_KC + 8 * (u ^ (r & 3)) + 32 * ((r >> 2) & 1), *xo = xe + (r & 4 ? -32 : 32);
    qg_h8 b[NT];
    auto read = [&](int buf, int s, int j) {
        b[j] = *reinterpret_cast<const qg_h8 *>((s & 1 ? xo : xe) + (buf * TM + 16 * j) * QG_KC + 64 * (s >> 1));
    };
    constexpr int STEPS = 4 / F::UNITS; // k-steps a load
#pragma unroll
    for (int i = 0; i < RI; i++)
#pragma unroll
        for (int q = 0; q < F::UNITS; q++) load(kc0, i, q);
    copy(kc0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // (the buffer is a run-time value: unrolled by two with constant buffers,
    // the Q4_0 kernels spilled)
    for (int kc = kc0, buf = 0; kc < kc1; kc++, buf ^= 1) {
        if (kc + 1 < kc1) copy(kc + 1, buf ^ 1);
#pragma unroll
        for (int j = 0; j < NT; j++) read(buf, 0, j);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (s % STEPS == 0) {
#pragma unroll
                for (int i = 0; i < RI; i++) qg_transpose(wv[i].c[s / STEPS]);
            }
#pragma unroll
            for (int i = 0; i < RI; i++) {
                const qg_h8 av = qg_dequant<FMT>(wv[i], s);
                if (s % STEPS == STEPS - 1) {
                    __builtin_amdgcn_sched_barrier(0);
                    load(kc + 1, i, s / STEPS);
                }
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, b[j], acc[i][j], 0, 0, 0);
                    if (i == RI - 1 && s < 3) read(buf, s + 1, j); // the next k-step's operand
                }
                // an operand is dequantised no further ahead (the kernels spill otherwise)
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // The next chunk's copies have landed, and every wave is done with
        // this buffer.  Of a wave's loads only the weight loads above come
        // after its copies (a load does not pass an asm with a memory
        // clobber), so that many may stay in flight.
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((F::UNITS + 1) * RI) : "memory");
        __syncthreads();
    }
    // accumulator e of lane (r, u) in tile (i, j): weight row 16 i + 4 u + e
    // of the wave's, token 16 j + r.  The empty asm keeps a tile where it is
    // until its turn (copied out all at once, the tiles would set the
    // kernel's register count).
    constexpr int NI = GLU && !SPLIT ? 2 : RI;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int local = 16 * j + r;
        const int tok = tok0 + local;
        const bool live = MOE ? local < np : tok < a.m;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            asm volatile("" : "+v"(acc[i][j]));
            if constexpr (GLU && !SPLIT) asm volatile("" : "+v"(acc[i + 2][j]));
            if (!live) continue;
            const int c = n0 + 16 * (GLU ? i & 1 : i) + 4 * u;
            if (SPLIT) { // partial rows: [split][gate, up][m][rows] f32
                const int64_t mat = GLU ? (int64_t)split * 2 + (i >> 1) : split;
                float *o = a.part + (mat * a.m + tok) * a.rows + c;
                if ((a.rows & 3) == 0 && c < a.rows) {
                    *reinterpret_cast<f32x4 *>(o) = acc[i][j];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (c + e < a.rows) o[e] = acc[i][j][e];
                }
                continue;
            }
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] = acc[i][j][e];
                if constexpr (GLU) {
                    float gg = v[e], uu = acc[(i + 2) & 3][j][e];
                    if (a.clamp > 0.0f) { // Glu::apply's clamp (cpu.rs:364-368)
                        gg = fminf(gg, a.clamp);
                        uu = fminf(fmaxf(uu, -a.clamp), a.clamp);
                    }
                    v[e] = (ACT == 0 ? act_silu(gg) : act_gelu_tanh(gg)) * uu;
                }
            }
            // MoE: pair p0 + local; down, the f32 product times the pair's
            // routing weight into the scratch row
            const int64_t row = MOE ? p0 + local : tok;
            if (MOE == 2) {
                const float pw = a.pair_weight[row];
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] *= pw;
            }
            typedef typename std::conditional<MOE == 2, float, T>::type O;
            O *o = reinterpret_cast<O *>(a.out) + row * a.out_ld + c;
            if (a.vec && c + 3 < a.rows) {
                if (sizeof(O) == 4) {
                    *reinterpret_cast<f32x4 *>(o) = f32x4{v[0], v[1], v[2], v[3]};
                } else {
                    typedef _Float16 qg_h4 __attribute__((ext_vector_type(4)));
                    *reinterpret_cast<qg_h4 *>(o) = qg_h4{to_stored<_Float16>(v[0]), to_stored<_Float16>(v[1]),
                                                         to_stored<_Float16>(v[2]), to_stored<_Float16>(v[3])};
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (c + e < a.rows) o[e] = to_stored<O>(v[e]);
            }
        }
    }
}

// The splits' partial rows added in split order, then the epilogue: one
// thread per output.
template <typename T, bool GLU, int ACT> __device__ static inline void qgemm_reduce_body(const QGemmArgs &a) {
    const int64_t e = (int64_t)blockIdx.x * CUCA_BLOCK + threadIdx.x;
    if (e >= (int64_t)a.m * a.rows) return;
    const int tok = (int)(e / a.rows), n = (int)(e - (int64_t)tok * a.rows);
    float g = 0.0f, u = 0.0f;
    for (int sp = 0; sp < a.splits; sp++) {
        g = g + a.part[((int64_t)sp * (GLU ? 2 : 1) * a.m + tok) * a.rows + n];
        if (GLU) u = u + a.part[((int64_t)(sp * 2 + 1) * a.m + tok) * a.rows + n];
    }
    float o = g;
    if (GLU) {
        if (a.clamp > 0.0f) { // Glu::apply's clamp (cpu.rs:364-368)
            g = fminf(g, a.clamp);
            u = fminf(fmaxf(u, -a.clamp), a.clamp);
        }
        o = (ACT == 0 ? act_silu(g) : act_gelu_tanh(g)) * u;
    }
    reinterpret_cast<T *>(a.out)[(int64_t)tok * a.out_ld + n] = to_stored<T>(o);
}

// Routed experts: the token tiles of the grouped GEMM.  One workgroup:
// thread 0 walks the experts (offsets clamped into [0, max_pairs] and made
// non-decreasing, so no pair index leaves the pair arrays), giving expert e
// ceil(n_e / tm) tiles from tile ts[e] on; then every tile c < n_ct gets
// its expert (a binary search over ts), first pair and pair count, or -1
// past the last tile.
#define QG_MOE_MAX_EXPERTS 4096
__device__ static inline void qgemm_moe_plan_body(const QGemmArgs &a) {
    __shared__ int ts[QG_MOE_MAX_EXPERTS + 1], lo[QG_MOE_MAX_EXPERTS + 1];
    const int E = a.n_experts, tm = a.tm;
    if (threadIdx.x == 0) {
        int prev = 0, t = 0;
        for (int e = 0; e < E; e++) {
            int l = a.offsets[e], hh = a.offsets[e + 1];
            l = min(max(l, prev), a.max_pairs);
            hh = min(max(hh, l), a.max_pairs);
            ts[e] = t;
            lo[e] = l;
            t += (hh - l + tm - 1) / tm;
            prev = hh;
        }
        ts[E] = t;
        lo[E] = prev;
    }
    __syncthreads();
    for (int c = threadIdx.x; c < a.n_ct; c += blockDim.x) {
        if (c >= ts[E]) {
            a.tile_e[c] = -1;
            a.tile_p0[c] = 0;
            a.tile_n[c] = 0;
            continue;
        }
        int l = 0, hh = E - 1; // the last e with ts[e] <= c (experts without pairs share ts)
        while (l < hh) {
            const int mid = (l + hh + 1) >> 1;
            if (ts[mid] <= c) l = mid;
            else hh = mid - 1;
        }
        const int p0 = lo[l] + (c - ts[l]) * tm;
        const int end = lo[l + 1]; // the clamped end of expert l's pairs
        a.tile_e[c] = l;
        a.tile_p0[c] = p0;
        a.tile_n[c] = min(tm, end - p0);
    }
}

// The activation rows of the routed pairs, rewritten as qgemm_prep_body does
// into the tile layout: padded row ct * tm + i holds pair tile_p0[ct] + i of
// the tile (zero past tile_n[ct]); up reads row pair_token[p] of x (a token
// outside [0, m) gives a zero row, reported), down row p.  Tiles past the
// last are not written (the GEMM skips them).
template <typename T, int FMT> __device__ static inline void qgemm_moe_prep_body(const QGemmArgs &a) {
    const int64_t u = (int64_t)blockIdx.x * CUCA_BLOCK + threadIdx.x;
    const int64_t per_row = (int64_t)a.nkc * 16;
    if (u >= (int64_t)a.mp * per_row) return;
    const int prow = (int)(u / per_row), rem = (int)(u - (int64_t)prow * per_row);
    const int ct = prow / a.tm, i = prow - ct * a.tm;
    if (a.tile_e[ct] < 0) return;
    const int kc = rem >> 4, v = rem & 15;
    bool valid = i < a.tile_n[ct];
    int64_t src = 0;
    if (valid) {
        const int p = a.tile_p0[ct] + i;
        if (a.moe_up) {
            const int tok = a.pair_token[p];
            if (tok < 0 || tok >= a.m) {
                valid = false;
                if (rem == 0) record_bad(a.status + CUCA_STATUS_MOE_PAIR, (uint32_t)p, (uint32_t)tok);
            } else {
                src = tok;
            }
        } else {
            src = p;
        }
    }
    const T *row = reinterpret_cast<const T *>(a.x) + src * a.ldx;
    qg_h8 o;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int k = qg_slot<FMT>(kc, v, j);
        o[j] = valid && k < a.k ? (_Float16)(float)row[k] : (_Float16)0.0f;
    }
    *reinterpret_cast<qg_h8 *>(a.xp + (int64_t)prow * a.kp + (int64_t)kc * QG_KC + 8 * v) = o;
}

#define CUCA_QGEMM(NAME, BODY, ...)                                                        \
    extern "C" __global__ __launch_bounds__(256) void NAME(QGemmArgs a) { BODY<__VA_ARGS__>(a); }
// two workgroups a compute unit: at most 256 registers
#define CUCA_QGEMM_TILE(NAME, ...)                                                         \
    extern "C" __global__ __launch_bounds__(256, 2) void NAME(QGemmArgs a) { qgemm_body<__VA_ARGS__>(a); }
#define CUCA_QGEMM_SET(TN, T, FN, FMT)                                                     \
    CUCA_QGEMM(cuca_qgemm_prep_##TN##_##FN, qgemm_prep_body, T, FMT)                        \
    CUCA_QGEMM_TILE(cuca_qgemm_##TN##_##FN, T, FMT, 8, false, 0, false)                    \
    CUCA_QGEMM_TILE(cuca_qgemm_glu_##TN##_##FN##_silu, T, FMT, 8, true, 0, false)          \
    CUCA_QGEMM_TILE(cuca_qgemm_glu_##TN##_##FN##_gelu, T, FMT, 8, true, 1, false)
CUCA_QGEMM_SET(f32, float, q4_0, 0)
CUCA_QGEMM_SET(f32, float, q8_0, 1)
CUCA_QGEMM_SET(f16, _Float16, q4_0, 0)
CUCA_QGEMM_SET(f16, _Float16, q8_0, 1)
CUCA_QGEMM_TILE(cuca_qgemm_q4_0_split, float, 0, 8, false, 0, true)
CUCA_QGEMM_TILE(cuca_qgemm_q8_0_split, float, 1, 8, false, 0, true)
CUCA_QGEMM_TILE(cuca_qgemm_glu_q4_0_split, float, 0, 8, true, 0, true)
CUCA_QGEMM_TILE(cuca_qgemm_glu_q8_0_split, float, 1, 8, true, 0, true)
// tiles of 64 tokens
#define CUCA_QGEMM_T64(TN, T, FN, FMT)                                                     \
    CUCA_QGEMM_TILE(cuca_qgemm_##TN##_##FN##_t64, T, FMT, 4, false, 0, false)              \
    CUCA_QGEMM_TILE(cuca_qgemm_glu_##TN##_##FN##_silu_t64, T, FMT, 4, true, 0, false)      \
    CUCA_QGEMM_TILE(cuca_qgemm_glu_##TN##_##FN##_gelu_t64, T, FMT, 4, true, 1, false)
CUCA_QGEMM_T64(f32, float, q4_0, 0)
CUCA_QGEMM_T64(f32, float, q8_0, 1)
CUCA_QGEMM_T64(f16, _Float16, q4_0, 0)
CUCA_QGEMM_T64(f16, _Float16, q8_0, 1)
CUCA_QGEMM_TILE(cuca_qgemm_q4_0_split_t64, float, 0, 4, false, 0, true)
CUCA_QGEMM_TILE(cuca_qgemm_glu_q4_0_split_t64, float, 0, 4, true, 0, true)
extern "C" __global__ __launch_bounds__(256) void cuca_qgemm_moe_plan(QGemmArgs a) { qgemm_moe_plan_body(a); }
#define CUCA_QGEMM_MOE_UP(TN, T, FN, FMT, TM)                                              \
    CUCA_QGEMM_TILE(cuca_qgemm_moe_up_##TN##_##FN##_silu_t##TM, T, FMT, TM / 16, true, 0, false, 1) \
    CUCA_QGEMM_TILE(cuca_qgemm_moe_up_##TN##_##FN##_gelu_t##TM, T, FMT, TM / 16, true, 1, false, 1)
#define CUCA_QGEMM_MOE_DOWN(TN, T, FN, FMT, TM)                                            \
    CUCA_QGEMM_TILE(cuca_qgemm_moe_down_##TN##_##FN##_r128_t##TM, T, FMT, TM / 16, false, 0, false, 2, 2)
#define CUCA_QGEMM_MOE_SET(TN, T, FN, FMT)                                                 \
    CUCA_QGEMM(cuca_qgemm_moe_prep_##TN##_##FN, qgemm_moe_prep_body, T, FMT)               \
    CUCA_QGEMM_MOE_UP(TN, T, FN, FMT, 32)                                                  \
    CUCA_QGEMM_MOE_UP(TN, T, FN, FMT, 64)                                                  \
    CUCA_QGEMM_MOE_UP(TN, T, FN, FMT, 128)                                                 \
    CUCA_QGEMM_MOE_DOWN(TN, T, FN, FMT, 32)                                                \
    CUCA_QGEMM_MOE_DOWN(TN, T, FN, FMT, 64)                                                \
    CUCA_QGEMM_MOE_DOWN(TN, T, FN, FMT, 128)                                               \
    CUCA_QGEMM_TILE(cuca_qgemm_moe_down_##TN##_##FN##_t128, T, FMT, 8, false, 0, false, 2)
CUCA_QGEMM_MOE_SET(f32, float, q4_0, 0)
CUCA_QGEMM_MOE_SET(f32, float, q8_0, 1)
CUCA_QGEMM_MOE_SET(f16, _Float16, q4_0, 0)
CUCA_QGEMM_MOE_SET(f16, _Float16, q8_0, 1)
#define CUCA_QGEMM_RED(TN, T)                                                              \
    CUCA_QGEMM(cuca_qgemm_reduce_##TN, qgemm_reduce_body, T, false, 0)                     \
    CUCA_QGEMM(cuca_qgemm_reduce_glu_##TN##_silu, qgemm_reduce_body, T, true, 0)           \
    CUCA_QGEMM(cuca_qgemm_reduce_glu_##TN##_gelu, qgemm_reduce_body, T, true, 1)
CUCA_QGEMM_RED(f32, float)
CUCA_QGEMM_RED(f16, _Float16)

// ---------------------------------------------------------------------
// The dense f16 path for many rows: the weight dequantised once into a
// resident f16 copy (the reference GPU engine's dense_dequant_kernel,
// moe_kernel.rs:1560-1600, with f16 output), then a plain f16 GEMM (the
// library's, f32 accumulation) and, for the GLU, the epilogue below.
// ---------------------------------------------------------------------

// One thread per (weight row, group, lane chunk l): the 2 G values l and
// l + 16 of the group's G blocks, w16[row][32 b + e] = f16(d_b * q), one
// rounding (the product of an f16 scale and a small integer is exact in
// f32) -- the values qgemm's operands carry.  Blocks past k (a partial last
// group) are not written.
template <int FMT> __device__ static inline void qdequant_body(const QDequantArgs &a) {
    constexpr int G = FMT == 0 ? 16 : 8, GB = FMT == 0 ? 288 : 272, SCB = 2 * G;
    const int64_t t = (int64_t)blockIdx.x * CUCA_BLOCK + threadIdx.x;
    if (t >= (int64_t)a.n * a.ng * 16) return;
    const int l = (int)(t & 15);
    const int64_t rg = t >> 4;
    const int g = (int)(rg % a.ng);
    const int64_t row = rg / a.ng;
    const uint8_t *grp = a.w + row * a.row_bytes + (int64_t)g * GB;
    const u32x4 chunk = *reinterpret_cast<const u32x4 *>(grp + SCB + 16 * l);
    const uint16_t *sc = reinterpret_cast<const uint16_t *>(grp);
    _Float16 *dst = reinterpret_cast<_Float16 *>(a.out) + row * a.out_ld;
#pragma unroll
    for (int b = 0; b < G; b++) {
        const int blk = g * G + b;
        if (blk >= a.nb) break;
        const float d = (float)__builtin_bit_cast(_Float16, sc[b]);
        int q0, q1; // elements l and l + 16
        if (FMT == 0) {
            const uint32_t w = chunk[b >> 2];
            q0 = (int)((w >> (4 * (b & 3))) & 15u) - 8;
            q1 = (int)((w >> (16 + 4 * (b & 3))) & 15u) - 8;
        } else {
            const uint32_t w = chunk[b >> 1];
            q0 = (int)((w >> (8 * (b & 1))) & 255u) - 128;
            q1 = (int)((w >> (16 + 8 * (b & 1))) & 255u) - 128;
        }
        dst[32 * blk + l] = (_Float16)(d * (float)q0);
        dst[32 * blk + l + 16] = (_Float16)(d * (float)q1);
    }
}
extern "C" __global__ __launch_bounds__(CUCA_BLOCK) void cuca_qdequant_q4_0(QDequantArgs a) { qdequant_body<0>(a); }
extern "C" __global__ __launch_bounds__(CUCA_BLOCK) void cuca_qdequant_q8_0(QDequantArgs a) { qdequant_body<1>(a); }

// Activations rounded to f16 (RNE), the GEMM's operand: x [m][ldx] f32 ->
// xh [m][k]; eight values per thread (k % 8 == 0).
extern "C" __global__ __launch_bounds__(CUCA_BLOCK) void cuca_cvt_f16_f32(QDequantArgs a) {
    const int64_t t = (int64_t)blockIdx.x * CUCA_BLOCK + threadIdx.x;
    const int64_t per = a.k / 8;
    if (t >= (int64_t)a.m * per) return;
    const int64_t r = t / per, c = (t - r * per) * 8;
    const float *src = reinterpret_cast<const float *>(a.x) + r * a.ldx + c;
    float v[8];
    qgemm_load8f(src, v);
    f16x8 h;
#pragma unroll
    for (int i = 0; i < 8; i++) h[i] = (_Float16)v[i];
    *reinterpret_cast<f16x8 *>(reinterpret_cast<_Float16 *>(a.out) + r * a.out_ld + c) = h;
}
