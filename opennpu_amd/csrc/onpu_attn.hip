// Decode attention for one token (grouped-query), the step the reference runs on the host beside
// its int4 matmuls: onpu_attn_step / onpu_attn_step_bf16 (onpu_cpu.cpp:173-229): for query head h
// (kv head g = h / (Hq / Hkv)), s_j = scale * q_h . K[g][j] + mask[j], softmax over j (with an
// optional per-head sink logit that takes probability mass but has no value), out_h = sum_j p_j
// V[g][j]. fp32 arithmetic; the KV cache is fp32 or bf16 (widened exactly).
//
// Split over the sequence; HBM-bound at long context (K and V are read once). k_attn_mfma serves a bf16
// cache, k_attn_part an fp32 one:
// workgroup (c, g, z) takes rows [c C, c C + C) of kv head g for HG of the query heads that share
// it (group z), so each K and V row is read once for HG heads. A row is read by LPR = D / 8
// consecutive lanes, 16 bytes each (one wave instruction covers 64 / LPR consecutive rows), with
// AU rows per lane group in flight. Phase 1 scores the chunk's rows into LDS (a lane's 8 products
// per head, summed across its LPR lanes by DPP); the chunk's max and exp-sum per head follow from
// LDS while the first V loads fly; phase 2 accumulates p_j V[j] in registers (8 values of d per lane
// and head), sums the row slots of a wave by shuffles and the waves in LDS, and writes the chunk's
// (max, sum, o[HG][D]). k_attn_combine: per query head, the chunks' partials rescaled to the
// global max (and the sink) and divided by the total mass.
#include <algorithm>
#include <type_traits>

#include "onpu_launch.h"

namespace {

constexpr int AT = 512;                      // threads per workgroup (8 waves)
constexpr int AW = AT / 64;
constexpr int AU = 4;                        // rows per lane group in flight
constexpr int AP_MAX = 16384;                // floats of P per workgroup (64 KiB)
constexpr int TARGET_WG = 512;
constexpr int ATT_MAX_CH = 4096;             // chunks per kv head at most: 8M rows or more, past any cache

struct AttnArgs {
    const float * q;
    const void * K, * V;
    const float * mask, * sinks;
    float * ws, * out;
    int64_t S, hs, rs;
    float scale;
    int Hq, D, Hkv, rep, ngrp, C, nch;
};

__device__ __forceinline__ void load8(const float * p, float (&v)[8]) {
    const float4 a = *(const float4 *) p, b = *(const float4 *) (p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// sum over aligned groups of L lanes (L = 8, 16, 32), every lane of a group left with the sum: DPP
// within a row of 16 (xor 1 and 2 by quad permutes, then the half-row and row mirrors, which pair
// lanes of equal partial sums), one cross-row shuffle for 32
template <int CTRL> __device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int L> __device__ __forceinline__ float group_sum(float x) {
    x += dpp_f<0xB1>(x);                     // quad_perm [1, 0, 3, 2]
    x += dpp_f<0x4E>(x);                     // quad_perm [2, 3, 0, 1]
    x += dpp_f<0x141>(x);                    // row_half_mirror: lane i <-> 7 - i
    if (L >= 16) x += dpp_f<0x140>(x);       // row_mirror: lane i <-> 15 - i
    if (L >= 32) x += __shfl_xor(x, 16);
    return x;
}

__device__ __forceinline__ float wave_max(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wave_sum(float v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// LDS: P [HG][C], red [AW][HG][D], wmax / wsum [AW][HG], qs [HG][D]
template <int LPR, int HG>
__global__ __launch_bounds__(AT) void k_attn_part(AttnArgs a) {
    constexpr int RPW = 64 / LPR, RIT = AW * RPW * AU;          // row slots per wave; rows per pass
    extern __shared__ __align__(16) float lds[];
    const int D = a.D, C = a.C, c = blockIdx.x, g = blockIdx.y, z = blockIdx.z, t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6, li = lane % LPR, slot = lane / LPR;
    float * P = lds, * red = P + HG * C, * wmax = red + AW * HG * D, * wsum = wmax + AW * HG, * qs = wsum + AW * HG;
    const bool dl = 8 * li < D;                                  // this lane's 8 values of d exist
    const int64_t j0 = (int64_t) c * C;
    const int rows = (int) (a.S - j0 < C ? a.S - j0 : C);
    // lanes past D read column 0 (their values meet zero q and are never stored)
    const float * Kg = (const float *) a.K + (int64_t) g * a.hs + j0 * a.rs + 8 * (dl ? li : 0);
    const float * Vg = (const float *) a.V + (int64_t) g * a.hs + j0 * a.rs + 8 * (dl ? li : 0);
    // q of the group's heads: coalesced 16-byte loads (0 past rep), stored to LDS after the first
    // pass's K loads are issued; the barrier then waits for LDS only (a __syncthreads would also
    // wait for the K loads)
    const int nq = HG * D / 4, hq0 = z * HG, hqn = a.rep - hq0 < HG ? a.rep - hq0 : HG;
    // (loads unconditional, from clamped addresses, and masked where used: a load under a branch is
    // waited for where the branch rejoins, which would serialize the loads)
    const bool qok = t < nq && t * 4 < hqn * D;
    const float4 qv = *(const float4 *) (a.q + (int64_t) (g * a.rep + hq0) * D + (qok ? 4 * t : 0));
    // Row of (pass r0, step u, wave, slot): consecutive slots and waves take consecutive rows, so one
    // wave instruction reads RPW consecutive rows.
    float kv[AU][8];
    auto issue = [&](const float * base, int r0) {
#pragma unroll
        for (int u = 0; u < AU; u++) {
            // rows past the chunk re-read its last row: their scores are not stored, their V rows
            // not accumulated
            const int row = r0 + (u * AW + wave) * RPW + slot;
            load8(base + (int64_t) (row < rows ? row : rows - 1) * a.rs, kv[u]);
        }
    };
    issue(Kg, 0);
    if (t < nq) *(float4 *) (qs + 4 * t) = qok ? qv : make_float4(0.f, 0.f, 0.f, 0.f);
    __builtin_amdgcn_s_waitcnt(0xc07f);                                 // lgkmcnt(0): the LDS stores
    __builtin_amdgcn_s_barrier();
    float qr[HG][8];
#pragma unroll
    for (int h = 0; h < HG; h++) {
        const float4 a0 = dl ? *(const float4 *) (qs + h * D + 8 * li) : make_float4(0.f, 0.f, 0.f, 0.f);
        const float4 a1 = dl ? *(const float4 *) (qs + h * D + 8 * li + 4) : make_float4(0.f, 0.f, 0.f, 0.f);
        qr[h][0] = a0.x; qr[h][1] = a0.y; qr[h][2] = a0.z; qr[h][3] = a0.w;
        qr[h][4] = a1.x; qr[h][5] = a1.y; qr[h][6] = a1.z; qr[h][7] = a1.w;
    }

    // phase 1: scores into P
    for (int r0 = 0; r0 < rows; r0 += RIT) {
        if (r0 > 0) issue(Kg, r0);
#pragma unroll
        for (int u = 0; u < AU; u++) {
            const int row = r0 + (u * AW + wave) * RPW + slot;
            float sc[HG];
#pragma unroll
            for (int h = 0; h < HG; h++) {
                float x = 0.f;
#pragma unroll
                for (int e = 0; e < 8; e++) x += qr[h][e] * kv[u][e];
                sc[h] = group_sum<LPR>(x);                                   // the row's lanes
            }
            if (li == 0 && row < rows) {
                const float mk = a.mask ? a.mask[j0 + row] : 0.f;
#pragma unroll
                for (int h = 0; h < HG; h++) P[h * C + row] = sc[h] * a.scale + mk;
            }
        }
    }
    issue(Vg, 0);                           // phase 2's first V loads fly during the softmax
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();
    // chunk max and exp-sum per head (a chunk whose rows are all -inf gets
    // p = e^(-inf - 0) = 0; a NaN score, which the maximum skips, p = NaN)
#pragma unroll
    for (int h = 0; h < HG; h++) {
        float mx = -__builtin_inff();
        for (int r = t; r < rows; r += AT) mx = fmaxf(mx, P[h * C + r]);
        mx = wave_max(mx);
        if (lane == 0) wmax[wave * HG + h] = mx;
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int h = 0; h < HG; h++) {
        float mx = wmax[h];
#pragma unroll
        for (int w = 1; w < AW; w++) mx = fmaxf(mx, wmax[w * HG + h]);
        const float base = mx == -__builtin_inff() ? 0.f : mx;
        float l = 0.f;
        for (int r = t; r < rows; r += AT) {
            const float p = expf(P[h * C + r] - base);
            P[h * C + r] = p;
            l += p;
        }
        l = wave_sum(l);
        if (lane == 0) wsum[wave * HG + h] = l;
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();

    // phase 2: o[h][d] = sum_j P[h][j] V[j][d]
    float acc[HG][8];
#pragma unroll
    for (int h = 0; h < HG; h++)
#pragma unroll
        for (int e = 0; e < 8; e++) acc[h][e] = 0.f;
    for (int r0 = 0; r0 < rows; r0 += RIT) {
        if (r0 > 0) issue(Vg, r0);
#pragma unroll
        for (int u = 0; u < AU; u++) {
            const int row = r0 + (u * AW + wave) * RPW + slot;
            if (row < rows) {
#pragma unroll
                for (int h = 0; h < HG; h++) {
                    const float p = P[h * C + row];
#pragma unroll
                    for (int e = 0; e < 8; e++) acc[h][e] += p * kv[u][e];
                }
            }
        }
    }
    // sum the wave's row slots (lanes LPR apart), then the waves
#pragma unroll
    for (int h = 0; h < HG; h++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float x = acc[h][e];
#pragma unroll
            for (int o = LPR; o < 64; o <<= 1) x += __shfl_xor(x, o);
            acc[h][e] = x;
        }
    if (slot == 0 && dl) {
#pragma unroll
        for (int h = 0; h < HG; h++)
#pragma unroll
            for (int e = 0; e < 8; e++) red[(wave * HG + h) * D + 8 * li + e] = acc[h][e];
    }
    __syncthreads();
    float * wp = a.ws + (((int64_t) g * a.ngrp + z) * a.nch + c) * (HG * (2 + D));
    for (int i = t; i < HG * D; i += AT) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < AW; w++) sum += red[w * HG * D + i];
        wp[2 * HG + i] = sum;
    }
    if (t < HG) {
        float mx = wmax[t], l = 0.f;
#pragma unroll
        for (int w = 1; w < AW; w++) mx = fmaxf(mx, wmax[w * HG + t]);
#pragma unroll
        for (int w = 0; w < AW; w++) l += wsum[w * HG + t];
        wp[t] = mx;
        wp[HG + t] = l;
    }
}

// ---- bf16 KV: scores on the matrix cores, no workgroup barrier before the end
// A wave takes 16 KT rows at a time. Bound by VALU work and latency at short context, by HBM at long.
// (The kernel above, which bf16 took too, spent its time in four barriers, P in LDS per workgroup and a
// DPP sum per row and head. Both launches, us per call, Hq / Hkv / D at S rows: 32 / 8 / 128 at 8192
// 17.8 -> 12.0, at 65536 53.6 -> 52.0 (5.2 TB/s); 32 / 4 / 128 at 16384 36.8 -> 14.8; 64 / 8 / 64 at 65536
// 61.7 -> 30.9; 16 / 2 / 256 at 16384 44.6 -> 22.2; 40 / 8 / 128 at 65536 93.6 -> 53.1. Error against 64 bits at
// those layouts 1.6-2.2e-7 -> 1.6-1.85e-7.) A row of an
// MFMA's A operand is one of three bf16 parts of one of 4 heads' q (row 4 h + part): q cut at its bits,
// 8 + 8 + 8, so the parts sum to q exactly and the products with bf16 K are exact; the steps' sums
// add as a tree, and the three fp32 sums of a (head, row) end in one lane (16 h + row of the 16), which adds them: no cross-lane sum and
// one exp per score. p goes through the wave's own LDS to the V layout (8 values of d per lane, LPR
// lanes per row) and o accumulates in fp32 by v_mfma_f32_4x4x1 (on the VALU for one or two heads), with
// a running maximum per wave. K of the
// next pass is loaded after this one's scores, V after this one's products, into the same registers.
// At the end the row slots of a wave are summed by half-swaps that leave each lane fewer heads, the
// waves meet in LDS, and a chunk's (max, sum, o) goes to the workspace (or, with one chunk, to out).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int MT = 256, MW = MT / 64;

// a workgroup barrier that orders LDS accesses only: global loads stay in flight across it
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <bool MAX> __device__ __forceinline__ float row16(float x) {        // over a row of 16 lanes
    if (MAX) {
        x = fmaxf(x, dpp_f<0xB1>(x));
        x = fmaxf(x, dpp_f<0x4E>(x));
        x = fmaxf(x, dpp_f<0x141>(x));
        return fmaxf(x, dpp_f<0x140>(x));
    }
    return group_sum<16>(x);
}

// lanes 32 (16) apart: a's sum in the lower, b's in the upper half (of each 32)
template <int HALF> __device__ __forceinline__ float swap_sum(float a, float b) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 r = HALF == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false)
                            : __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r.x) + __uint_as_float(r.y);
}

// LDS: P [MW][16 KT][HG], ml [MW][HG][2], red [MW][HG][D] (first the A fragments, 1 KiB each)
template <int NS, int HG, int KT>
__global__ __launch_bounds__(MT, 2) void k_attn_mfma(AttnArgs a) {
    constexpr int LPR = 4 * NS, RPW = 64 / LPR, NSET = (HG + 3) / 4;
    extern __shared__ __align__(16) float lds[];
    const int D = a.D, c = blockIdx.x, g = blockIdx.y, z = blockIdx.z;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int key = lane & 15, quad = lane >> 4, li = lane % LPR, slot = lane / LPR;
    float * P = lds + w * 16 * KT * HG, * ml = lds + MW * 16 * KT * HG, * red = ml + 2 * MW * HG;
    const int64_t j0 = (int64_t) c * a.C;
    const int rows = (int) (a.S - j0 < a.C ? a.S - j0 : a.C);
    const uint16_t * Kg = (const uint16_t *) a.K + (int64_t) g * a.hs + j0 * a.rs;
    const uint16_t * Vg = (const uint16_t *) a.V + (int64_t) g * a.hs + j0 * a.rs + (8 * li < D ? 8 * li : 0);
    const int hq0 = z * HG, hqn = a.rep - hq0 < HG ? a.rep - hq0 : HG;      // q heads of this group
    uint4 kr[KT][NS], vr[KT][NS];
    float mk[KT];
    // mask values through a buffer that is empty without a mask (no branch: a load under one is
    // waited for, with everything before it, where the paths meet); K and V rows past the chunk
    // re-read its last row
    const __amdgpu_buffer_rsrc_t mr =
        __builtin_amdgcn_make_buffer_rsrc((void *) (a.mask ? a.mask + j0 : a.q), (short) 0, a.mask ? rows * 4 : 0, 0x00020000);
    auto load_k = [&](int r0) {
#pragma unroll
        for (int t = 0; t < KT; t++)
            mk[t] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(mr, (uint32_t) (4 * (r0 + 16 * t + key)), 0, 0));
#pragma unroll
        for (int t = 0; t < KT; t++) {
            const int row = r0 + 16 * t + key;
            const uint16_t * p = Kg + (int64_t) (row < rows ? row : rows - 1) * a.rs;
#pragma unroll
            for (int s = 0; s < NS; s++) {                                   // past D: column 0, zeroed below
                const int d = 32 * s + 8 * quad;
                kr[t][s] = *(const uint4 *) (p + (d < D ? d : 0));
            }
        }
    };
    auto load_v = [&](int r0) {
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int s = 0; s < NS; s++) {
                const int row = r0 + 16 * t + RPW * s + slot;
                vr[t][s] = *(const uint4 *) (Vg + (int64_t) (row < rows ? row : rows - 1) * a.rs);
            }
    };
    // A fragments of the scores: lane (row = lane & 15: head row / 4, part row % 4; k = 8 quad + e).
    // Wave w cuts fragments w, w + 4, ... for all; q is loaded before K and V, so that cutting it
    // overlaps their latency (the barrier waits for LDS only).
    constexpr int NF = (NSET * NS + MW - 1) / MW;
    const int part = key & 3;
    float4 q4[NF][2];
    bool qok[NF];
#pragma unroll
    for (int i = 0; i < NF; i++) {
        const int f = w + MW * i, h = 4 * (f / NS) + (key >> 2), d = 32 * (f % NS) + 8 * quad;
        qok[i] = h < hqn && d < D && part < 3;
        const float4 * qp = (const float4 *) (a.q + (int64_t) (g * a.rep + hq0) * D + (qok[i] ? h * D + d : 0));
        q4[i][0] = qp[0];
        q4[i][1] = qp[1];
    }
    __builtin_amdgcn_sched_barrier(0);                           // q's loads stay ahead
    int r0 = w * 16 * KT;
    load_k(r0);
    load_v(r0);
    const uint32_t cut0 = part >= 1 ? 0xffff0000u : 0u, cut1 = part == 2 ? 0xffff0000u : 0u;
#pragma unroll
    for (int i = 0; i < NF; i++) {
        const float x[8] = {q4[i][0].x, q4[i][0].y, q4[i][0].z, q4[i][0].w, q4[i][1].x, q4[i][1].y, q4[i][1].z, q4[i][1].w};
        uint32_t u[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {                            // x, x - its top part, less that one's
            const float y = x[e] - __uint_as_float(__float_as_uint(x[e]) & cut0);
            u[e] = qok[i] ? __float_as_uint(y - __uint_as_float(__float_as_uint(y) & cut1)) : 0u;
        }
        if (w + MW * i < NSET * NS)
            *((uint4 *) red + (w + MW * i) * 64 + lane) =
                make_uint4(__builtin_amdgcn_perm(u[1], u[0], 0x07060302u), __builtin_amdgcn_perm(u[3], u[2], 0x07060302u),
                           __builtin_amdgcn_perm(u[5], u[4], 0x07060302u), __builtin_amdgcn_perm(u[7], u[6], 0x07060302u));
    }
    lds_barrier();
    bf16x8 qa[NSET][NS];
#pragma unroll
    for (int f = 0; f < NSET * NS; f++) qa[f / NS][f % NS] = __builtin_bit_cast(bf16x8, *((const uint4 *) red + f * 64 + lane));
    f32x4 av[NSET][8] = {};                                      // o: element h % 4 of av[h / 4][e]
    float m[NSET], l[NSET];
#pragma unroll
    for (int h4 = 0; h4 < NSET; h4++) { m[h4] = -__builtin_inff(); l[h4] = 0.f; }

    auto pass = [&](auto more) {
        const int rn = r0 + MW * 16 * KT;
        float sc[KT][NSET];
#pragma unroll
        for (int t = 0; t < KT; t++) {
            f32x4 d[NSET][NS];                                               // a sum per step, added as a tree
#pragma unroll
            for (int s = 0; s < NS; s++) {
                uint4 kv = kr[t][s];
                if (D < 32 * NS && 32 * s + 8 * quad >= D) kv = make_uint4(0, 0, 0, 0);
#pragma unroll
                for (int h4 = 0; h4 < NSET; h4++)
                    d[h4][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[h4][s], __builtin_bit_cast(bf16x8, kv), (f32x4){0, 0, 0, 0}, 0, 0, 0);
            }
#pragma unroll
            for (int h4 = 0; h4 < NSET; h4++)
#pragma unroll
                for (int o = 1; o < NS; o *= 2)
#pragma unroll
                    for (int s = 0; s < NS; s += 2 * o) d[h4][s] += d[h4][s + o];
            const int row = r0 + 16 * t + key;
#pragma unroll
            for (int h4 = 0; h4 < NSET; h4++) {
                // (the lower parts' sums are NaN where an infinite K meets their zeros)
                const f32x4 y = d[h4][0];
                const float x = y[0] + (__builtin_isfinite(y[0]) ? y[1] + y[2] : 0.f);
                sc[t][h4] = row < rows ? x * a.scale + mk[t] : -__builtin_inff();
            }
        }
        if (more) load_k(rn);
        float al[NSET];
        bool up = false;
#pragma unroll
        for (int h4 = 0; h4 < NSET; h4++) {
            float mx = sc[0][h4];
#pragma unroll
            for (int t = 1; t < KT; t++) mx = fmaxf(mx, sc[t][h4]);
            mx = fmaxf(m[h4], row16<true>(mx));
            al[h4] = m[h4] == mx ? 1.f : expf(m[h4] - mx);                   // 0 from a first finite maximum
            up = up || m[h4] != mx;
            m[h4] = mx;
            l[h4] *= al[h4];
#pragma unroll
            for (int t = 0; t < KT; t++) {
                // 0 also while the maximum is -inf; NaN, which the maximum skips, stays NaN
                const float p = sc[t][h4] == -__builtin_inff() ? 0.f : expf(sc[t][h4] - mx);
                l[h4] += p;
                if (4 * h4 + quad < HG) P[(16 * t + key) * HG + 4 * h4 + quad] = p;
            }
        }
        // o of this pass alone, added to the scaled o of those before it: shorter sums, less rounding (not
        // at 8 heads of D > 128, which have no registers left for both)
        constexpr bool OWN = NS * HG < 64;
        float f[HG];
        const bool rescale = r0 >= MW * 16 * KT && __any(up);                // (the first pass finds o = 0)
        if (rescale) {
#pragma unroll
            for (int h = 0; h < HG; h++) {
                f[h] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(al[h / 4]), 16 * (h % 4)));
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (!OWN) av[h / 4][e][h % 4] *= f[h];
            }
        }
        f32x4 pv[NSET][8];
#pragma unroll
        for (int h4 = 0; h4 < NSET; h4++)
#pragma unroll
            for (int e = 0; e < 8; e++) pv[h4][e] = OWN ? (f32x4){0, 0, 0, 0} : av[h4][e];
        if (r0 + 16 * KT > rows) {                                           // rows past the chunk: p = 0, V = 0
#pragma unroll
            for (int t = 0; t < KT; t++)
#pragma unroll
                for (int s = 0; s < NS; s++)
                    if (r0 + 16 * t + RPW * s + slot >= rows) vr[t][s] = make_uint4(0, 0, 0, 0);
        }
        __builtin_amdgcn_wave_barrier();                                     // the wave's LDS is in order
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int s = 0; s < NS; s++) {
                // lane (16 slot + 4 b + c): p of head c (and 4 + c) and V of its own 8 columns; block b of
                // v_mfma_f32_4x4x1 multiplies the 4 heads by its lanes' columns, fp32, into the lane
                const float * pp = P + (16 * t + RPW * s + slot) * HG + (HG >= 4 ? lane & 3 : 0);
                const uint32_t u[4] = {vr[t][s].x, vr[t][s].y, vr[t][s].z, vr[t][s].w};
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float v = __uint_as_float(e & 1 ? u[e / 2] & 0xffff0000u : u[e / 2] << 16);
#pragma unroll
                    for (int h = 0; h < HG; h += HG >= 4 ? 4 : 1) {
                        if (HG >= 4) pv[h / 4][e] = __builtin_amdgcn_mfma_f32_4x4x1f32(pp[h], v, pv[h / 4][e], 0, 0, 0);
                        else pv[0][e][h] += pp[h] * v;
                    }
                }
            }
#pragma unroll
        for (int h = 0; h < HG; h++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float o = av[h / 4][e][h % 4], n = pv[h / 4][e][h % 4];
                av[h / 4][e][h % 4] = !OWN ? n : (rescale ? __builtin_fmaf(o, f[h], n) : o + n);
            }
        __builtin_amdgcn_wave_barrier();
        if (more) load_v(rn);
        r0 = rn;
    };
    while (r0 + MW * 16 * KT < rows) pass(std::true_type{});
    if (r0 < rows) pass(std::false_type{});
#pragma unroll
    for (int h4 = 0; h4 < NSET; h4++) {
        l[h4] = row16<false>(l[h4]);
        if (key == 0 && 4 * h4 + quad < HG) {
            ml[(w * HG + 4 * h4 + quad) * 2] = m[h4];
            ml[(w * HG + 4 * h4 + quad) * 2 + 1] = l[h4];
        }
    }
    float acc[HG][8];
#pragma unroll
    for (int h = 0; h < HG; h++)
#pragma unroll
        for (int e = 0; e < 8; e++) acc[h][e] = av[h / 4][e][h % 4];
    // sum the row slots; each halving leaves a lane the heads of its half while there are two or more
    int hb = 0;                                                              // first head of this lane
    constexpr int H1 = RPW >= 2 && HG >= 2 ? HG / 2 : HG, H2 = RPW >= 4 && H1 >= 2 ? H1 / 2 : H1;
    if (RPW >= 2) {
#pragma unroll
        for (int h = 0; h < H1; h++)
#pragma unroll
            for (int e = 0; e < 8; e++) acc[h][e] = swap_sum<32>(acc[h][e], acc[HG >= 2 ? h + H1 : h][e]);
        if (HG >= 2) hb += (lane >> 5) * H1;
    }
    if (RPW >= 4) {
#pragma unroll
        for (int h = 0; h < H2; h++)
#pragma unroll
            for (int e = 0; e < 8; e++) acc[h][e] = swap_sum<16>(acc[h][e], acc[H1 >= 2 ? h + H2 : h][e]);
        if (H1 >= 2) hb += ((lane >> 4) & 1) * H2;
    }
    if (RPW >= 8) {
#pragma unroll
        for (int h = 0; h < H2; h++)
#pragma unroll
            for (int e = 0; e < 8; e++) acc[h][e] += dpp_f<0x128>(acc[h][e]);   // row_ror:8
    }
    lds_barrier();                                               // every wave has its fragments: red is free
    if (8 * li < D) {
#pragma unroll
        for (int h = 0; h < H2; h++) {
            float4 * o = (float4 *) (red + (w * HG + hb + h) * D + 8 * li);
            o[0] = make_float4(acc[h][0], acc[h][1], acc[h][2], acc[h][3]);
            o[1] = make_float4(acc[h][4], acc[h][5], acc[h][6], acc[h][7]);
        }
    }
    lds_barrier();
    float * wp = a.ws + (((int64_t) g * a.ngrp + z) * a.nch + c) * (HG * (2 + D));
    constexpr int DP = 32 * NS;                                  // D rounded up: a power of two
    const int d = threadIdx.x % DP;
    for (int h = threadIdx.x / DP; h < HG && d < D; h += MT / DP) {
        float M = ml[2 * h], sum = 0.f, L = 0.f;
#pragma unroll
        for (int k = 1; k < MW; k++) M = fmaxf(M, ml[(k * HG + h) * 2]);
        const float sink = a.sinks && a.nch == 1 && h < hqn ? a.sinks[g * a.rep + hq0 + h] : -__builtin_inff();
        M = fmaxf(M, sink);
#pragma unroll
        for (int k = 0; k < MW; k++) {
            const float mk = ml[(k * HG + h) * 2], f = mk == -__builtin_inff() ? 0.f : expf(mk - M);
            sum += f * red[(k * HG + h) * D + d];
            L += f * ml[(k * HG + h) * 2 + 1];
        }
        if (a.nch == 1) {
            if (a.sinks) L += expf(sink - M);
            if (h < hqn) a.out[(int64_t) (g * a.rep + hq0 + h) * D + d] = sum / L;
            continue;
        }
        wp[2 * HG + h * D + d] = sum;
        if (d == 0) {
            wp[h] = M;
            wp[HG + h] = L;
        }
    }
}

// grid (Hq, ceil(D / 64)), 8 waves: out[h][d] = sum_c e^(m_c - M) o_c[d] / (sum_c e^(m_c - M) l_c +
// e^(sink - M)). A lane per column; every wave finds M and the denominator by itself, a chunk per
// lane, and sums chunks w, w + 8, ..., 8 o loads at a time; the first 8 go out before M is known, so
// that one memory latency covers up to 64 chunks. The waves meet in LDS once. Latency-bound (32 heads,
// 64 chunks: 4.4 us with a workgroup per head in four dependent passes, 2.7-3.8 now).
constexpr int CW = 8, CB = 8;
template <int HG>
__global__ __launch_bounds__(64 * CW) void k_attn_combine(AttnArgs a) {
    __shared__ float sred[CW][64];
    const int h = blockIdx.x, g = h / a.rep, hr = h - g * a.rep, z = hr / HG, hh = hr - z * HG;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), d = 64 * blockIdx.y + lane;
    const int64_t st = HG * (2 + a.D);
    const float * wp = a.ws + ((int64_t) g * a.ngrp + z) * a.nch * st;
    const float * wo = wp + 2 * HG + hh * a.D + (d < a.D ? d : 0);
    float ov[CB];
    auto load_o = [&](int b) {                                   // (past the chunks: the last, unused)
#pragma unroll
        for (int k = 0; k < CB; k++) {
            const int c = b + w + CW * k < a.nch ? b + w + CW * k : a.nch - 1;
            ov[k] = wo[c * st];
        }
    };
    load_o(0);
    const int c0 = lane < a.nch ? lane : a.nch - 1;
    const float m0 = wp[c0 * st + hh], l0 = wp[c0 * st + HG + hh], sink = a.sinks ? a.sinks[h] : -__builtin_inff();
    float M = fmaxf(m0, sink);
    for (int c = lane + 64; c < a.nch; c += 64) M = fmaxf(M, wp[c * st + hh]);
    M = wave_max(M);
    float den = 0.f, acc = 0.f;
    for (int b = 0; b < a.nch; b += 64) {
        const int c = b + lane;
        const float mc = c >= a.nch ? -__builtin_inff() : (b == 0 ? m0 : wp[c * st + hh]);
        // (a chunk without a finite score has sum 0 and weight 0)
        const float f = mc == -__builtin_inff() ? 0.f : expf(mc - M);
        if (c < a.nch) den += f * (b == 0 ? l0 : wp[c * st + HG + hh]);
#pragma unroll
        for (int k = 0; k < CB; k++)
            if (b + w + CW * k < a.nch)
                acc += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), w + CW * k)) * ov[k];
        if (b + 64 < a.nch) load_o(b + 64);
    }
    sred[w][lane] = acc;
    den = wave_sum(den) + (a.sinks ? expf(sink - M) : 0.f);
    __syncthreads();
    if (w == 0 && d < a.D) {
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < CW; i++) sum += sred[i][lane];
        a.out[(int64_t) h * a.D + d] = sum / den;
    }
}

int next_pow2(int v) {
    int p = 1;
    while (p < v) p *= 2;
    return p;
}

struct AttnPlan { int LPR, HG, ngrp, C, nch; };

// chunk rows: enough chunks for ~TARGET_WG workgroups, at least 64 rows each, P within AP_MAX
AttnPlan attn_plan(int Hq, int D, int Hkv, int64_t S) {
    AttnPlan p;
    const int rep = Hq / Hkv;
    p.LPR = next_pow2(D / 8) < 8 ? 8 : next_pow2(D / 8);
    p.HG = next_pow2(rep) > 8 ? 8 : next_pow2(rep);
    p.ngrp = (rep + p.HG - 1) / p.HG;
    int64_t nch = (TARGET_WG + (int64_t) Hkv * p.ngrp - 1) / ((int64_t) Hkv * p.ngrp);
    const int64_t nmax = (S + 63) / 64;
    if (nch > nmax) nch = nmax;
    if (nch < 1) nch = 1;
    int64_t C = ((S + nch - 1) / nch + 63) / 64 * 64;
    if (C > AP_MAX / p.HG) C = AP_MAX / p.HG;
    p.C = (int) C;
    p.nch = (int) ((S + C - 1) / C);
    return p;                                 // nch <= ATT_MAX_CH is checked by the launcher
}

size_t attn_lds(const AttnPlan & p, int D) {
    return sizeof(float) * ((size_t) p.HG * p.C + (size_t) AW * p.HG * D + 2 * AW * p.HG + (size_t) p.HG * D);
}

template <bool BF, int NS, int HG>
hipError_t run_attn(const AttnArgs & a, const AttnPlan & p, hipStream_t s) {
    const dim3 grid((unsigned) a.nch, (unsigned) a.Hkv, (unsigned) a.ngrp);
    if (BF) {
        constexpr int KT = NS >= 8 || HG >= 8 ? 1 : 2;
        const size_t lds = sizeof(float) * ((size_t) MW * 16 * KT * HG + 2 * MW * HG) +
                           std::max<size_t>(sizeof(float) * MW * HG * a.D, 1024 * (size_t) NS * ((HG + 3) / 4));
        k_attn_mfma<NS, HG, KT><<<grid, MT, lds, s>>>(a);
    } else {
        k_attn_part<4 * NS, HG><<<grid, AT, attn_lds(p, a.D), s>>>(a);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || (BF && a.nch == 1)) return e;
    k_attn_combine<HG><<<dim3((unsigned) a.Hq, (unsigned) (a.D + 63) / 64), 64 * CW, 0, s>>>(a);
    return hipGetLastError();
}

template <bool BF, int NS>
hipError_t run_attn_hg(const AttnArgs & a, const AttnPlan & p, hipStream_t s) {
    switch (p.HG) {
    case 1: return run_attn<BF, NS, 1>(a, p, s);
    case 2: return run_attn<BF, NS, 2>(a, p, s);
    case 4: return run_attn<BF, NS, 4>(a, p, s);
    case 8: return run_attn<BF, NS, 8>(a, p, s);
    default: return hipErrorInvalidValue;
    }
}

template <bool BF>
hipError_t run_attn_lpr(const AttnArgs & a, const AttnPlan & p, hipStream_t s) {
    switch (p.LPR) {
    case 8: return run_attn_hg<BF, 2>(a, p, s);
    case 16: return run_attn_hg<BF, 4>(a, p, s);
    case 32: return run_attn_hg<BF, 8>(a, p, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

int64_t attn_ws_bytes(int Hq, int D, int Hkv, int64_t S) {
    if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || D <= 0 || S <= 0) return 0;
    const AttnPlan p = attn_plan(Hq, D, Hkv, S);
    return (int64_t) Hkv * p.ngrp * p.nch * p.HG * (2 + D) * (int64_t) sizeof(float);
}

hipError_t launch_attn_step(const float * q, int Hq, int D, const void * K, const void * V, int kv_bf16, int Hkv,
                            int64_t S, int64_t hs, int64_t rs, const float * mask, const float * sinks, float scale,
                            float * out, void * ws, int64_t ws_bytes, hipStream_t s) {
    if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || S <= 0 || D <= 0 || D > 256 || D % 8) return hipErrorInvalidValue;
    if (Hq / Hkv > 16) return hipErrorInvalidValue;
    const int64_t al = kv_bf16 ? 8 : 4;             // 16-byte row starts for the vector loads
    if (rs % al || hs % al || ((uintptr_t) K | (uintptr_t) V | (uintptr_t) q) % 16) return hipErrorInvalidValue;
    if (ws_bytes < attn_ws_bytes(Hq, D, Hkv, S)) return hipErrorInvalidValue;
    AttnPlan p = attn_plan(Hq, D, Hkv, S);
    // One workgroup per head group, without the second launch, up to four of its passes (two at D > 128):
    // a call issued from Python pays for the launch, and at four passes about breaks even. us per call, two
    // launches -> one, issued from Python / replayed from a graph of 16 calls:
    //   32 / 8 heads, D = 128: 128 rows 9.7 / 7.8 -> 7.2 / 5.3, 384 9.4 / 7.9 -> 8.4 / 8.4, 512 9.7-10.9 / 7.8 ->
    //     9.9 / 9.9
    //   40 / 8 (8 heads per group): 128 rows 9.9 / 8.6 -> 7.5 / 7.5, 192 10.0 / 8.6 -> 8.9 / 8.9, 256 10.0-10.8 / 8.7
    //     -> 10.2 / 10.3
    //   64 / 8, D = 64: 256 rows 9.8 / 7.4 -> 8.1 / 8.1; 32 / 8, D = 64: 512 rows 10.0 / 6.8 -> 7.3 / 6.7
    //   8 / 8 and 16 / 8, D = 128: 384 rows 9.6 / 6.7 -> 7.2 / 6.1 and 9.9 / 7.0 -> 7.3 / 6.8, 512 9.5 / 6.7 -> 7.2 /
    //     7.2 and 9.9 / 7.1 -> 8.0 / 8.0
    //   D = 256, 16 / 2, 16 / 4 and 8 / 8: 128 rows 11.4 / 11.4, 10.0 / 8.9 and 10.1 / 6.9 -> 11.3 / 11.4, 8.1 / 8.2
    //     and 7.4 / 5.4; 300 rows in one workgroup 16.9 against 13.5
    const int64_t one = D > 128 ? 128 : (p.HG >= 8 ? 256 : 512);
    if (kv_bf16 && S <= one) {
        p.C = (int) S;
        p.nch = 1;
    }
    AttnArgs a;
    a.q = q; a.K = K; a.V = V; a.mask = mask; a.sinks = sinks; a.ws = (float *) ws; a.out = out;
    a.S = S; a.hs = hs; a.rs = rs; a.scale = scale;
    a.Hq = Hq; a.D = D; a.Hkv = Hkv; a.rep = Hq / Hkv; a.ngrp = p.ngrp; a.C = p.C; a.nch = p.nch;
    if (Hkv > 65535 || p.ngrp > 65535 || p.nch > ATT_MAX_CH) return hipErrorInvalidValue;
    return kv_bf16 ? run_attn_lpr<true>(a, p, s) : run_attn_lpr<false>(a, p, s);
}

// ------------------------------------------------------------------ Gated DeltaNet decode step
// One decode token of a Gated DeltaNet layer: the reference's host onpu_gdn_step (onpu_cpu.cpp:107-
// 171). k_gdn_conv: one thread per channel c of qkv: causal conv over the last Kc inputs (the same
// order of products as the reference), SiLU into co, and the conv state shifts by one. k_gdn_head:
// one workgroup per value head h: q, k of its key head L2-normalised (q also / sqrt Dk), beta =
// sigmoid(Wb x), decay = exp(-exp(A_log) softplus(Wa x + dt_bias)); the head's state S [Dk][Dv]
// goes to LDS scaled by decay while thread (d-column j, row group g) sums kv_j = sum_i S_ij k_i;
// delta = beta (v - kv); S += k delta^T and o = S^T q in a second pass over LDS, S written back;
// out = norm_w * o / sqrt(mean(o^2) + eps) * silu(z). Sums are block reductions (another order than
// the reference's sequential loops).
namespace {

__device__ __forceinline__ float gdn_silu(float v) { return v / (1.f + expf(-v)); }

__global__ __launch_bounds__(256) void k_gdn_conv(const float * __restrict__ qkv, const float * __restrict__ conv_w,
                                                  int Kc, float * __restrict__ conv_state, int L, int C,
                                                  float * __restrict__ co) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    float * st = conv_state + (int64_t) c * L;
    const float * w = conv_w + (int64_t) c * Kc;
    float s = w[Kc - 1] * qkv[c];
    for (int j = 0; j < Kc - 1; j++) s += w[j] * st[L - (Kc - 1) + j];
    co[c] = gdn_silu(s);
    for (int j = 0; j + 1 < L; j++) st[j] = st[j + 1];
    st[L - 1] = qkv[c];
}

// block sum over 256 threads (every thread gets the sum); red: 8 floats of LDS
__device__ __forceinline__ float gdn_block_sum(float v, float * red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

struct GdnArgs {
    const float * x, * z, * Wb, * Wa, * A_log, * dt_bias, * norm_w, * co;
    float * S, * out;
    float eps;
    int H, Hk, Hv, Dk, Dv;
};

// LDS: Sl [Dk][Dv], vec [4][max(Dk, Dv)] (q, k, delta / o), part [256 / Dv][Dv], red [8]
__global__ __launch_bounds__(256) void k_gdn_head(GdnArgs a) {
    extern __shared__ __align__(16) float lds[];
    const int h = blockIdx.x, t = threadIdx.x, Dk = a.Dk, Dv = a.Dv, rep = a.Hv / a.Hk, kh = h / rep;
    const int key_dim = a.Hk * Dk, mx = Dk > Dv ? Dk : Dv, G = 256 / Dv, j = t % Dv, g = t / Dv;
    float * Sl = lds, * qv = Sl + Dk * Dv, * kvec = qv + mx, * dv = kvec + mx, * ov = dv + mx;
    float * part = ov + mx, * red = part + G * Dv;
    float qq = 0.f, kk = 0.f;
    for (int i = t; i < Dk; i += 256) {
        const float qi = a.co[kh * Dk + i], ki = a.co[key_dim + kh * Dk + i];
        qv[i] = qi;
        kvec[i] = ki;
        qq += qi * qi;
        kk += ki * ki;
    }
    float pb = 0.f, pa = 0.f;
    for (int i = t; i < a.H; i += 256) {
        pb += a.Wb[(int64_t) h * a.H + i] * a.x[i];
        pa += a.Wa[(int64_t) h * a.H + i] * a.x[i];
    }
    qq = gdn_block_sum(qq, red);
    kk = gdn_block_sum(kk, red);
    const float b = gdn_block_sum(pb, red), av = gdn_block_sum(pa, red);
    const float qn = 1.f / sqrtf(qq + 1e-6f) / sqrtf((float) Dk), kn = 1.f / sqrtf(kk + 1e-6f);
    const float beta = 1.f / (1.f + expf(-b));
    const float ad = av + a.dt_bias[h];
    const float sp = ad > 20.f ? ad : log1pf(expf(ad));
    const float decay = expf(-expf(a.A_log[h]) * sp);
    // pass 1: S <- decay S into LDS, kv_j = sum_i S_ij k_i (row groups g, g + G, ...)
    float * Sh = a.S + (int64_t) h * Dk * Dv;
    float kv = 0.f;
    if (g < G)
        for (int i = g; i < Dk; i += G) {
            const float r = Sh[(int64_t) i * Dv + j] * decay;
            Sl[i * Dv + j] = r;
            kv += r * (kvec[i] * kn);
        }
    if (g < G) part[g * Dv + j] = kv;
    __syncthreads();
    if (t < Dv) {
        float s = 0.f;
        for (int r = 0; r < G; r++) s += part[r * Dv + t];
        dv[t] = (a.co[2 * key_dim + (int64_t) h * Dv + t] - s) * beta;
    }
    __syncthreads();
    // pass 2: S += k delta^T, o_j = sum_i S_ij q_i; S back to HBM
    float o = 0.f;
    if (g < G)
        for (int i = g; i < Dk; i += G) {
            const float r = Sl[i * Dv + j] + (kvec[i] * kn) * dv[j];
            Sh[(int64_t) i * Dv + j] = r;
            o += r * (qv[i] * qn);
        }
    if (g < G) part[g * Dv + j] = o;
    __syncthreads();
    float oj = 0.f;
    if (t < Dv) {
        for (int r = 0; r < G; r++) oj += part[r * Dv + t];
        ov[t] = oj;
    }
    const float ms = gdn_block_sum(t < Dv ? oj * oj : 0.f, red) / Dv;
    const float rn = 1.f / sqrtf(ms + a.eps);
    if (t < Dv) a.out[(int64_t) h * Dv + t] = a.norm_w[t] * (oj * rn) * gdn_silu(a.z[(int64_t) h * Dv + t]);
}

}  // namespace

int64_t gdn_ws_bytes(int Hk, int Hv, int Dk, int Dv) {
    return (int64_t) (2 * Hk * Dk + Hv * Dv) * (int64_t) sizeof(float);
}

hipError_t launch_gdn_step(const float * x, int H, const float * qkv, const float * z, const float * Wb,
                           const float * Wa, const float * conv_w, int Kc, float * conv_state, int L,
                           const float * A_log, const float * dt_bias, const float * norm_w, float eps, float * S,
                           int Hk, int Hv, int Dk, int Dv, float * out, void * ws, int64_t ws_bytes, hipStream_t s) {
    if (H <= 0 || Hk <= 0 || Hv <= 0 || Hv % Hk || Dk <= 0 || Dv <= 0 || 256 % Dv || Dv < 4 || Kc < 1 ||
        L < Kc - 1 || L < 1 || (int64_t) Dk * Dv > 32768)
        return hipErrorInvalidValue;
    if (ws_bytes < gdn_ws_bytes(Hk, Hv, Dk, Dv)) return hipErrorInvalidValue;
    const int C = 2 * Hk * Dk + Hv * Dv;
    float * co = (float *) ws;
    k_gdn_conv<<<(C + 255) / 256, 256, 0, s>>>(qkv, conv_w, Kc, conv_state, L, C, co);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    GdnArgs a;
    a.x = x; a.z = z; a.Wb = Wb; a.Wa = Wa; a.A_log = A_log; a.dt_bias = dt_bias; a.norm_w = norm_w; a.co = co;
    a.S = S; a.out = out; a.eps = eps; a.H = H; a.Hk = Hk; a.Hv = Hv; a.Dk = Dk; a.Dv = Dv;
    const int mx = Dk > Dv ? Dk : Dv;
    const size_t lds = sizeof(float) * ((size_t) Dk * Dv + 4 * (size_t) mx + (size_t) (256 / Dv) * Dv + 8);
    k_gdn_head<<<Hv, 256, lds, s>>>(a);
    return hipGetLastError();
}
