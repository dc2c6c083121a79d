// qms_moe.hip -- the routed experts (MoE) at decode, from two tokens on: the
// CPU engine's bits (qmm.hip; the expert sum of cpu.rs:400-417), with the
// arithmetic of qms.hip.
//
// Workgroup (tile, split) takes one tile of the expert order (moe_tile_lookup:
// up to four pairs of one expert) and a contiguous range of the expert's row
// tasks (gate and up: four rows of each; down: eight rows).  It quantises the
// tile's activation rows once, whole, into LDS (QMS layout), and its four waves
// stream their tasks' weight groups through a ring of D register slots, the
// first slots' loads under the quantisation.  A weight pair is extracted once for
// all the tile's pairs; a tile of fewer than four pairs runs a body of its own
// (MJ), so that no chain is computed for a pair that is not there.  A task's
// sums go to LDS and a chunk of QMS_MOE_NT tasks is written after its stream,
// so that the ring's waits count its own loads only.  Where the splits are a
// multiple of eight, a split of all an expert's tiles meets in one XCD's L2.
//
// What bounds it: the vector unit's issue rate (Q4_0 and Q8_0 take the same
// time), as qms.hip.  Measured on MI355X, 128 experts of 768 over 2048, top 8,
// Zipf routing, f32 Q4_0, up + down, 2 / 4 / 8 / 16 / 32 / 64 tokens: 16 / 24 / 37
// / 65 / 106 / 176 us, against the kernel before it (tiles of one to four pairs
// by the mean, every tile's chains computed for all of them, dw * dx and the
// pairs' bias through LDS) 25 / 27 / 47 / 69 / 139 / 342.
#include "common.h"

#define QMS_MOE_WAVES 4
#define QMS_MOE_NT 16

// LDS: the tile (QMS_LDS_BYTES) and, per wave, the sums of a chunk's tasks.
#define QMS_MOE_LDS_BYTES(J, NBP) (QMS_LDS_BYTES(J, NBP) + QMS_MOE_WAVES * QMS_MOE_NT * (J) * 8 * 4)

// UP: gate and up with the activation; otherwise down, times the pair's
// weight.  MJ = p1 - p0 pairs of expert e, from p0 on.
template <typename T, int FMT, bool UP, int MJ, int D>
__device__ static inline void qms_moe_tile(const QmvArgs &a, unsigned char *lds, int e, int p0, int split) {
    using F = QFmt<FMT>;
    constexpr int G = F::G, NS = G / 4, RPT = UP ? 4 : 8; // steps a group, (output) rows a task
    const int ng = a.ng, nbp = a.nbp, nq4 = nbp >> 2;
    u32x4 *xe = reinterpret_cast<u32x4 *>(lds);                              // [row][nbp / 4][17]
    float *xsc = reinterpret_cast<float *>(xe + MJ * nq4 * QMS_ROW4);        // [row][nbp]
    const int tid = threadIdx.x, lt = tid & (CUCA_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / CUCA_WAVE);
    float *res = xsc + MJ * nbp + wave * (QMS_MOE_NT * MJ * 8);              // [task][MJ][2][4]
    const int r = lt >> 4, l = lt & 15;
    constexpr int NTH = QMS_MOE_WAVES * CUCA_WAVE;

    int64_t xr[MJ]; // the pairs' activation rows, or -1 (a bad token: zeros, no output)
#pragma unroll
    for (int j = 0; j < MJ; j++) {
        xr[j] = (int64_t)(p0 + j) * a.ldx;
        if (UP) {
            const int t = a.pair_token[p0 + j];
            const bool ok = t >= 0 && t < a.n_tokens;
            if (!ok && tid == 0) record_bad(a.status + CUCA_STATUS_MOE_PAIR, (uint32_t)(p0 + j), (uint32_t)t);
            xr[j] = ok ? (int64_t)t * a.ldx : -1;
        }
    }
    // items of 8 values, four threads a block, the tile's rows end to end
    const int per = 4 * nbp, total = per * MJ, sub = tid & 3;
    float xv[4][8];
    auto fetch = [&](int i0) {
#pragma unroll
        for (int it = 0; it < 4; it++) {
            const int idx = i0 + it * NTH + tid, j = idx / per, b = (idx - j * per) >> 2;
            int64_t row = xr[0];
#pragma unroll
            for (int i = 1; i < MJ; i++) row = j == i ? xr[i] : row;
            if (j < MJ && b < a.nb && row >= 0) {
                qmm_load8<T>(reinterpret_cast<const T *>(a.x) + row + (int64_t)b * 32 + sub * 8, xv[it]);
            } else {
#pragma unroll
                for (int q = 0; q < 8; q++) xv[it][q] = 0.0f;
            }
        }
    };
    fetch(0);
    __builtin_amdgcn_sched_barrier(0);

    const uint32_t nrec = (uint32_t)((int64_t)a.rows * a.row_bytes);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(a.w + (int64_t)e * a.w_estride), 0, (int)nrec, QMD_RSRC_W3);
    const __amdgpu_buffer_rsrc_t ru = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>((UP ? a.w_up : a.w) + (int64_t)e * a.w_estride), 0, (int)nrec, QMD_RSRC_W3);
    const int first = split * a.tps + wave, tend = min(a.ntask, (split + 1) * a.tps);
    const int nt = first < tend ? (tend - first + QMS_MOE_WAVES - 1) / QMS_MOE_WAVES : 0;

    typedef QmsSlot<FMT, 2> Slot;
    Slot ring[D];
    uint32_t vchunk[2], vscale[2]; // the load cursor: task lti, its group lg
    int lti = 0, lg = 0;
    auto seek = [&](int ti) { // past the wave's last task: that task's rows again, not used
        const int task = first + min(ti, max(nt - 1, 0)) * QMS_MOE_WAVES;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int row = UP ? task * 4 + r : task * 8 + 4 * i + r;
            const uint32_t rb = (uint32_t)min(row, a.rows - 1) * (uint32_t)a.row_bytes;
            vchunk[i] = rb + F::SCB + 16 * l;
            vscale[i] = rb + 4 * ((l % G) >> 1);
        }
    };
    auto load = [&](Slot &s) {
        const int so = lg * F::GB; // wave-uniform: the scalar offset
#pragma unroll
        for (int i = 0; i < 2; i++) {
            s.w[i] = __builtin_amdgcn_raw_buffer_load_b128(UP && i ? ru : rw, vchunk[i], so, 0);
            s.s[i] = __builtin_amdgcn_raw_buffer_load_b32(UP && i ? ru : rw, vscale[i], so, 0);
        }
        if (++lg == ng) {
            lg = 0;
            seek(++lti);
        }
    };
    auto prime = [&](int c0) {
        lti = c0;
        lg = 0;
        seek(lti);
        qmd_for<0, D>([&](auto I) {
            load(ring[I.value]);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    prime(0);

    // quantise (as qms.hip)
    for (int i0 = 0; i0 < total; i0 += 4 * NTH) {
        if (i0) fetch(i0);
#pragma unroll
        for (int it = 0; it < 4; it++) {
            const int idx = i0 + it * NTH + tid;
            if (i0 + it * NTH >= total) break; // uniform: the tile is done
            const int j = idx / per, b = (idx - j * per) >> 2;
            float amax = 0.0f;
#pragma unroll
            for (int q = 0; q < 8; q++) amax = fmaxf(amax, fabsf(xv[it][q]));
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
                const bool low = sub < 2;
                const int base = 8 * (sub & 1) + (low ? 0 : 4);
                uint32_t *dst = reinterpret_cast<uint32_t *>(xe + (j * nq4 + (b >> 2)) * QMS_ROW4 + base) + (b & 3);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t lo = low ? own[q >> 1] : other[2 + (q >> 1)];
                    const uint32_t hi = low ? other[q >> 1] : own[2 + (q >> 1)];
                    dst[4 * q] = __builtin_amdgcn_perm(hi, lo, (q & 1) ? 0x07060302u : 0x05040100u);
                }
                if (sub == 0) xsc[j * nbp + b] = b < a.nb ? (float)(_Float16)d : 0.0f;
            }
        }
    }
    __syncthreads();
    if (nt == 0) return;

    const int sh = 16 * (l & 1);
    const u32x4 *xl = xe + l;
    const float *xsl = xsc + (l % G);
    for (int c0 = 0; c0 < nt; c0 += QMS_MOE_NT) {
        if (c0) prime(c0);
        const int cn = min(QMS_MOE_NT, nt - c0), groups = cn * ng;
        int cti = 0, cg = 0; // consumed: task of the chunk, group
        float acc[2][MJ], cdx[MJ];
        u32x4 cx[MJ];
#pragma unroll
        for (int j = 0; j < MJ; j++) {
            acc[0][j] = acc[1][j] = 0.0f;
            cx[j] = xl[j * nq4 * QMS_ROW4];
            cdx[j] = xsl[j * nbp];
        }
        auto consume = [&](const Slot &s) {
            float sc[2][MJ];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const float dw = qmv_h2f(s.s[i] >> sh);
#pragma unroll
                for (int j = 0; j < MJ; j++) sc[i][j] = dw * cdx[j];
            }
            const int gn = cg + 1 == ng ? 0 : cg + 1; // the next group's operands, read a step ahead
#pragma unroll
            for (int j = 0; j < MJ; j++) cdx[j] = xsl[j * nbp + gn * G];
            qmd_for<0, NS>([&](auto S4) {
                const u32x4 *xn = xl + (S4.value + 1 < NS ? cg * NS + S4.value + 1 : gn * NS) * QMS_ROW4;
                u32x4 nx[MJ];
#pragma unroll
                for (int j = 0; j < MJ; j++) nx[j] = xn[j * nq4 * QMS_ROW4];
                qmd_for<0, 4>([&](auto Q) {
                    constexpr int b = 4 * S4.value + Q.value;
                    float p[2][MJ];
                    uint32_t xp[MJ];
#pragma unroll
                    for (int j = 0; j < MJ; j++) xp[j] = cx[j][Q.value];
                    qms_dots2<MJ>(qms_pair<FMT>(s.w[0], b), qms_pair<FMT>(s.w[1], b), xp, p[0], p[1]);
#pragma unroll
                    for (int i = 0; i < 2; i++)
#pragma unroll
                        for (int j = 0; j < MJ; j++) p[i][j] = p[i][j] * qmd_bcast<b>(sc[i][j]);
#pragma unroll
                    for (int i = 0; i < 2; i++)
#pragma unroll
                        for (int j = 0; j < MJ; j++) acc[i][j] = acc[i][j] + p[i][j];
                });
                // pin these four blocks' arithmetic here (as qms.hip)
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < MJ; j++) asm volatile("" : "+v"(acc[i][j]));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < MJ; j++) cx[j] = nx[j];
            });
            cg = gn;
            if (gn == 0) { // the task's last group: its sums to LDS
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < MJ; j++) {
                        const float o = qmm_hsum(acc[i][j]);
                        if (l == 0) res[((cti * MJ + j) * 2 + i) * 4 + r] = o;
                        acc[i][j] = 0.0f;
                    }
                cti++;
            }
        };
        const int nr = (groups + D - 1) / D;
        for (int R = 0; R + 1 < nr; R++) {
            qmd_for<0, D>([&](auto I) {
                consume(ring[I.value]);
                load(ring[I.value]);
            });
        }
        const int rem = groups - (nr - 1) * D; // 1..D groups in the last round
        qmd_for<0, D>([&](auto I) {
            if (I.value < rem) consume(ring[I.value]);
        });
        __builtin_amdgcn_wave_barrier();
        // the chunk's outputs: a lane takes (task, pair, row of the task)
        for (int i = lt; i < cn * MJ * RPT; i += CUCA_WAVE) {
            const int ti = i / (MJ * RPT), j = (i / RPT) % MJ, rr = i % RPT;
            const int row = (first + (c0 + ti) * QMS_MOE_WAVES) * RPT + rr;
            int64_t xj = xr[0];
#pragma unroll
            for (int q = 1; q < MJ; q++) xj = j == q ? xr[q] : xj;
            if (row >= a.rows || xj < 0) continue;
            float o = res[(ti * MJ + j) * 8 + rr];
            if constexpr (UP) {
                float u = res[(ti * MJ + j) * 8 + 4 + rr];
                if (a.clamp > 0.0f) { // Glu::apply's clamp (cpu.rs:364-368)
                    o = fminf(o, a.clamp);
                    u = fminf(fmaxf(u, -a.clamp), a.clamp);
                }
                o = (a.gelu ? act_gelu_tanh(o) : act_silu(o)) * u;
                reinterpret_cast<T *>(a.out)[(int64_t)(p0 + j) * a.out_ld + row] = to_stored<T>(o);
            } else { // CpuExpert::add_picks: y * weight (cpu.rs:400-417)
                reinterpret_cast<float *>(a.out)[(int64_t)(p0 + j) * a.out_ld + row] = o * a.pair_weight[p0 + j];
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

template <typename T, int FMT, bool UP, int D> __device__ static inline void qms_moe_body(const QmvArgs &a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char qms_moe_lds[];
    const int tile = blockIdx.x / a.splits, split = blockIdx.x - tile * a.splits;
    if (split * a.tps >= a.ntask) return; // no rows left for it (the whole workgroup)
    int e, p0, p1;
    // tiles of a.m pairs
    const bool any = a.m == 4   ? moe_tile_lookup<4>(a.offsets, a.n_experts, a.max_pairs, tile, &e, &p0, &p1)
                     : a.m == 2 ? moe_tile_lookup<2>(a.offsets, a.n_experts, a.max_pairs, tile, &e, &p0, &p1)
                                : moe_tile_lookup<1>(a.offsets, a.n_experts, a.max_pairs, tile, &e, &p0, &p1);
    if (!any) return; // the whole workgroup
    e = __builtin_amdgcn_readfirstlane(e);
    p0 = __builtin_amdgcn_readfirstlane(p0);
    const int np = __builtin_amdgcn_readfirstlane(p1) - p0;
    if (np == 4) qms_moe_tile<T, FMT, UP, 4, D>(a, qms_moe_lds, e, p0, split);
    else if (np == 3) qms_moe_tile<T, FMT, UP, 3, D>(a, qms_moe_lds, e, p0, split);
    else if (np == 2) qms_moe_tile<T, FMT, UP, 2, D>(a, qms_moe_lds, e, p0, split);
    else if (np == 1) qms_moe_tile<T, FMT, UP, 1, D>(a, qms_moe_lds, e, p0, split);
}

#define CUCA_QMS_MOE(NAME, ...)                                                                  \
    extern "C" __global__ __launch_bounds__(QMS_MOE_WAVES * CUCA_WAVE, 4) void NAME(QmvArgs a) { \
        qms_moe_body<__VA_ARGS__>(a);                                                            \
    }
#define CUCA_QMS_MOE_SET(TN, T, FN, FMT, D)                        \
    CUCA_QMS_MOE(cuca_qms_moe_up_##TN##_##FN, T, FMT, true, D)     \
    CUCA_QMS_MOE(cuca_qms_moe_down_##TN##_##FN, T, FMT, false, D)
// (D slots: as qms.hip, but three for Q8_0, down spills with four)
CUCA_QMS_MOE_SET(f32, float, q4_0, 0, 2)
CUCA_QMS_MOE_SET(f32, float, q8_0, 1, 3)
CUCA_QMS_MOE_SET(f16, _Float16, q4_0, 0, 2)
CUCA_QMS_MOE_SET(f16, _Float16, q8_0, 1, 3)
