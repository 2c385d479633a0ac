// GPU weight codecs of libonpu_hip: quantize weights already in HBM (fp32 or bf16) into a format's
// tiled HBM layout (onpu_common.h), or transcode GGUF Q4_K super-blocks into q4nx tiles. The bytes are
// those of the quantizers in onpu_codec.h (the source behind the host's onpu_pack / onpu_pack_q4k).
//
// One lane per group, each kernel writing the tiles itself: a wave covers the 16 rows x 4 groups of one
// block (lane 4 r + j: row r, group j, so that dword q of all lanes is 256 contiguous bytes), or, for
// g128s, 64 rows of one block column. (Through a staging buffer and k_repack, allocated and freed per
// call, the same matrix paid 34 us of repacking and ~130 us of allocation on top.)
#include "onpu_codec.h"
#include "onpu_launch.h"

namespace {

constexpr int CODEC_THREADS = 256, CODEC_WAVES = CODEC_THREADS / 64;

// G weights at element off; W is aligned to its elements only
template <int G, bool BF>
__device__ __forceinline__ void load_group(const void * W, int64_t off, float (&x)[G]) {
    if (BF) {
        uint32_t d[G / 2];
        __builtin_memcpy(d, (const uint16_t *) W + off, sizeof(d));
#pragma unroll
        for (int i = 0; i < G / 2; i++) {
            x[2 * i] = __builtin_bit_cast(float, d[i] << 16);
            x[2 * i + 1] = __builtin_bit_cast(float, d[i] & 0xffff0000u);
        }
    } else {
        __builtin_memcpy(x, (const float *) W + off, sizeof(x));
    }
}

// ------------------------------------------------------------------ search quantizers
// The searches of onpu_codec.h without their divisions. VALU-bound: an IEEE division is ~10 of the ~19
// ops a pass takes per weight; without it a q4s candidate takes 12.5 ops per weight from bf16 (16 from
// fp32) instead of 36. (Counters, 24576 x 4096 q4s from bf16: 14.2 VALU instructions per weight and candidate
// with all that is around the two passes, one per 2.7 cycles of a SIMD; waves wait for memory in 5 % of
// their cycles and for their turn to issue in 64 %; q4nx 3 and 62 %.) Whole call, 12288 x 4096, from bf16 / fp32: q4s 882 / 870 -> 224 / 309 us, g128s
// 889 / 905 -> 247 / 338, q4nx 897 / 899 -> 361 / 396; Q4_0, which has no search, 200 / 222 -> 40 / 58
// (no staging); q4s 24576 x 4096 from bf16 1728 -> 439. Every value that reaches a code, a scale or a
// comparison is the same fp32 number as there:
//   - v x, l x (4-bit integer times bf16), v v, l sc, v d (d, sc are bf16 values) are exact products, so
//     one fma rounds as the multiply and the add do;
//   - a quotient only reaches rint(RN(x / d)). With r ~ 1 / d within 2^-23.9 of it relative,
//     e = fma(-d, r, 1) exact and rl = e r, fma(x, r, x rl) is RN of (x / d)(1 + t), |t| < 2^-46
//     ("div2"). That is RN(x / d) wherever x / d is further than 2^-46 of itself from every midpoint of
//     neighbouring floats:
//       d a bf16 value: an 8-bit d times a 25-bit midpoint differs from a 24-bit x, if at all, by
//         more than 2^-33 of x;
//       x a bf16 value, d = D 2^s with 2^23 <= D < 2^24: only midpoints next to a half-integer h,
//         |h| < 9, matter. x - d h is a multiple J of 2^(s-1) and d ulp / 2 is D / 2^m of those units,
//         m = 20..25, so both must agree to 2^-17: D within 74 of a multiple of 2^20, not on it (on
//         it, D / 2^m is a multiple of 1/32, and J = D / 2^m would give x more than 8 bits).
//         d0_risky() finds those (one d in 2^12);
//     and for those, and for fp32 x, one more step fma(fma(-d, y, x), r, y) with r = RN(1 / d) is the
//     correctly rounded quotient (Markstein 1990: y faithful, the remainder exact);
//   - in the error pass of a bf16 x, x r alone (off by 2^-19 at most) picks another integer than
//     RN(x / d) only on an exact tie, as other bf16 quotients are 2^-9 from a half-integer at least; on
//     a tie either choice leaves |v d - x| = |d| / 2, the same squared error.
// Groups whose magnitudes could overflow or go subnormal on the way, or with a NaN, take the original.
struct Rcp { float r, rl; };

template <bool EXACT>
__device__ __forceinline__ Rcp rcp_of(float d) {
    Rcp c;
    if (EXACT) c.r = 1.0f / d;
    else {
        const float a = __builtin_amdgcn_rcpf(d);
        c.r = __builtin_fmaf(__builtin_fmaf(-d, a, 1.0f), a, a);
    }
    c.rl = __builtin_fmaf(-d, c.r, 1.0f) * c.r;
    return c;
}
__device__ __forceinline__ float div2(float x, Rcp c) { return __builtin_fmaf(x, c.r, x * c.rl); }
__device__ __forceinline__ float div4(float x, float d, Rcp c) {
    const float y = div2(x, c);
    return __builtin_fmaf(__builtin_fmaf(-d, y, x), c.r, y);
}
__device__ __forceinline__ bool d0_risky(float d) {
    const uint32_t t = (__builtin_bit_cast(uint32_t, d) + 128u) & 0xfffffu;
    return t < 256u && t != 128u;
}

// eight codes as a tile dword (element e at nibble nib_pos(e))
__device__ __forceinline__ uint32_t tile_dword(const uint8_t * q) {
    uint32_t d = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) d |= (uint32_t) q[e] << (4 * nib_pos(e));
    return d;
}
template <int G>
__device__ __forceinline__ void tile_dwords(const uint8_t (&q)[G], uint32_t (&dw)[G / 8]) {
#pragma unroll
    for (int i = 0; i < G / 8; i++) dw[i] = tile_dword(q + 8 * i);
}
// the same from codes held as floats v, bias to add: byte b of the dword is
// (v[e] + bias) + 16 (v[e + 2] + bias), e = 0, 4, 1, 5
__device__ __forceinline__ uint32_t tile_dword(const float (&v)[8], float bias) {
    uint32_t d = 0;
#pragma unroll
    for (int b = 0; b < 4; b++) {
        const int e = 4 * (b & 1) + (b >> 1);
        d = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(v[e + 2], 16.0f, v[e] + 17.0f * bias), b, d);
    }
    return d;
}

// candidate values x_max / d of quant_sym, and their reciprocals
struct SymTab { float dv[16], rdv[16]; };
constexpr SymTab sym_tab() {
    SymTab t{};
    for (int c = 0; c < 16; c++) {
        t.dv[c] = c < 8 ? -9.0f + 2.5f * c / 7 : 6.5f + 1.5f * (c - 8) / 7;
        t.rdv[c] = 1.0f / t.dv[c];
    }
    return t;
}
__constant__ const SymTab SYM_TAB = sym_tab();

// sums of one candidate's first pass: v = clamp(rint(x / d0)), sum v v and sum v x
template <int G, bool BF, bool FULL>
__device__ __forceinline__ void sym_sums(const float (&x)[G], float d0, Rcp c, float & sqq, float & sqx) {
#pragma clang fp contract(off)
    sqq = 0;
    sqx = 0;
#pragma unroll
    for (int i = 0; i < G; i++) {
        const float y = FULL ? div4(x[i], d0, c) : div2(x[i], c);
        const float v = __builtin_amdgcn_fmed3f(__builtin_rintf(y), -8.0f, 7.0f);
        sqq = __builtin_fmaf(v, v, sqq);
        sqx = BF ? __builtin_fmaf(v, x[i], sqx) : sqx + v * x[i];
    }
}

// quant_sym of onpu_codec.h, the same codes and scale
template <int G, bool BF>
__device__ __forceinline__ void quant_sym_gpu(const float (&x)[G], uint32_t (&dw)[G / 8], uint16_t & d_bf) {
#pragma clang fp contract(off)
    float mx = 0;
#pragma unroll
    for (int i = 0; i < G; i++) mx = __builtin_fabsf(x[i]) > __builtin_fabsf(mx) ? x[i] : mx;
    const float amx = __builtin_fabsf(mx);
    const bool zero = mx == 0;
    bool ok = zero || (amx >= 0x1p-60f && amx <= 0x1p60f);
#pragma unroll
    for (int i = 0; i < G; i++) ok = ok && __builtin_fabsf(x[i]) <= amx;       // false for a NaN
    if (!__all(ok)) {
        uint8_t q[G];
        quant_sym<G>(x, q, d_bf);
        tile_dwords<G>(q, dw);
        return;
    }
    if (zero) mx = 1.0f;
    float best_e = __builtin_inff(), best_d = 1.0f;
#pragma nounroll
    for (int c = 0; c < 16; c++) {
        const float dv = SYM_TAB.dv[c], rdv = SYM_TAB.rdv[c];
        float d0 = mx * rdv;                                                   // RN(mx / dv): two steps
        d0 = __builtin_fmaf(__builtin_fmaf(-dv, d0, mx), rdv, d0);
        d0 = __builtin_fmaf(__builtin_fmaf(-dv, d0, mx), rdv, d0);
        const Rcp r0 = rcp_of<!BF>(d0);
        float sqq, sqx;
        if (!BF) sym_sums<G, BF, true>(x, d0, r0, sqq, sqx);
        else if (__any(d0_risky(d0))) sym_sums<G, BF, true>(x, d0, rcp_of<true>(d0), sqq, sqx);
        else sym_sums<G, BF, false>(x, d0, r0, sqq, sqx);
        const float d = bf16_round(sqq > 0 ? sqx / sqq : d0);
        float e = 0;
        const Rcp r1 = rcp_of<false>(d);
#pragma unroll
        for (int i = 0; i < G; i++) {
            const float y = BF ? x[i] * r1.r : div2(x[i], r1);
            const float v = __builtin_amdgcn_fmed3f(__builtin_rintf(y), -8.0f, 7.0f);
            const float r = __builtin_fmaf(v, d, -x[i]);
            e += r * r;
        }
        if (d != 0 && e < best_e) { best_e = e; best_d = d; }
    }
    if (zero) best_d = 1.0f;
    const Rcp rb = rcp_of<false>(best_d);
#pragma unroll
    for (int i = 0; i < G / 8; i++) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = __builtin_amdgcn_fmed3f(__builtin_rintf(div2(x[8 * i + e], rb)), -8.0f, 7.0f);
        dw[i] = tile_dword(v, 8.0f);
    }
    d_bf = f32_to_bf16(best_d);
}

// quant_asym32 of onpu_codec.h, the same codes, scale and min
template <bool BF>
__device__ __forceinline__ void quant_asym_gpu(const float (&x)[32], uint32_t (&dw)[4], uint16_t & s_bf, uint16_t & m_bf) {
#pragma clang fp contract(off)
    float lo = x[0], hi = x[0], sx = 0;
#pragma unroll
    for (int i = 0; i < 32; i++) {
        lo = x[i] < lo ? x[i] : lo;
        hi = hi < x[i] ? x[i] : hi;
        sx += x[i];
    }
    const float range = hi - lo;
    bool ok = !(range > 0) || (range >= 0x1p-40f && lo >= -0x1p20f && hi <= 0x1p20f);
#pragma unroll
    for (int i = 0; i < 32; i++) ok = ok && x[i] >= lo && x[i] <= hi;          // false for a NaN
    if (!__all(ok)) {
        uint8_t q[32];
        quant_asym32(x, q, s_bf, m_bf);
        tile_dwords<32>(q, dw);
        return;
    }
    const bool flat = !(range > 0);
    const float rg = flat ? 1.0f : range;
    float best_e = __builtin_inff(), best_s = rg / 15, best_m = lo;
    float t[32];
#pragma unroll
    for (int i = 0; i < 32; i++) t[i] = x[i] - lo;
#pragma nounroll
    for (int st = 0; st <= 20; st++) {
        const float isc = (-1.0f + 0.1f * st + 15.0f) / rg;
        float sl = 0, sll = 0, slx = 0;
#pragma unroll
        for (int i = 0; i < 32; i++) {
            const float l = __builtin_amdgcn_fmed3f(__builtin_rintf(isc * t[i]), 0.0f, 15.0f);
            sl += l;
            sll = __builtin_fmaf(l, l, sll);
            slx = BF ? __builtin_fmaf(l, x[i], slx) : slx + l * x[i];
        }
        const float D = 32 * sll - sl * sl;
        float sc = rg / 15, mn = lo;
        if (D > 0) {
            sc = (32 * slx - sl * sx) / D;
            mn = (sll * sx - sl * slx) / D;
        }
        sc = bf16_round(sc);
        mn = bf16_round(mn);
        const bool use = sc > 0;
        const Rcp c = rcp_of<false>(use ? sc : 1.0f);
        float e = 0;
#pragma unroll
        for (int i = 0; i < 32; i++) {
            const float l = __builtin_amdgcn_fmed3f(__builtin_rintf(div2(x[i] - mn, c)), 0.0f, 15.0f);
            const float d = __builtin_fmaf(l, sc, mn) - x[i];
            e += d * d;
        }
        if (use && e < best_e) { best_e = e; best_s = sc; best_m = mn; }
    }
    best_s = bf16_round(best_s);
    best_m = bf16_round(best_m);
    if (flat) { best_s = 1.0f; best_m = lo; }
    const Rcp c = rcp_of<false>(best_s);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++)
            v[e] = __builtin_amdgcn_fmed3f(__builtin_rintf(div2(x[8 * i + e] - best_m, c)), 0.0f, 15.0f);
        dw[i] = flat ? 0u : tile_dword(v, 0.0f);
    }
    s_bf = f32_to_bf16(best_s);
    m_bf = f32_to_bf16(best_m);
}

// a lane's group of 32 (row r, group j of a block) and its parameter(s) into the block
template <int FMT>
__device__ __forceinline__ void store_group32(uint8_t * blk, int lane, const uint32_t (&dw)[4], uint16_t s, uint16_t m) {
#pragma unroll
    for (int k = 0; k < 4; k++) *(uint32_t *) (blk + 256 * k + 4 * lane) = dw[k];
    if (FMT == ONPU_Q4NX) *(uint32_t *) (blk + 1024 + 4 * lane) = s | ((uint32_t) m << 16);
    else *(uint16_t *) (blk + 1024 + 2 * lane) = s;
}

// grid (waves / CODEC_WAVES, experts): W [e][N][ldw] (elements), out [e] tiles of ostride bytes. Rows
// and groups past the matrix are quantized as zeros, which gives the padding codes, with parameters 0.
template <int FMT, bool BF>
__global__ __launch_bounds__(CODEC_THREADS, FMT == ONPU_G128S ? 2 : 1) void k_quantize(const void * __restrict__ W, int64_t ldw, int64_t N,
                                                            int64_t K, int64_t NT, int64_t KB,
                                                            uint8_t * __restrict__ out, int64_t ostride) {
    constexpr int G = FMT == ONPU_G128S ? 128 : 32;
    const int lane = threadIdx.x & 63;
    const int64_t w = (int64_t) blockIdx.x * CODEC_WAVES + (threadIdx.x >> 6), e = blockIdx.y;
    // g128s: 4 row tiles per wave, a lane per row; else one tile, a lane per (row, group)
    const int64_t tq = w / KB, b = w - tq * KB, t = G == 128 ? 4 * tq + (lane >> 4) : tq;
    if (tq >= (G == 128 ? (NT + 3) / 4 : NT)) return;
    const int64_t n = G == 128 ? 64 * tq + lane : 16 * t + (lane >> 2), k = G == 128 ? 128 * b : 128 * b + 32 * (lane & 3);
    const bool in = n < N && k < K;
    float x[G];
    if (in) load_group<G, BF>(W, (e * N + n) * ldw + k, x);
    else {
#pragma unroll
        for (int i = 0; i < G; i++) x[i] = 0;
    }
    uint32_t dw[G / 8];
    uint16_t s = 0, m = 0;
    auto & x32 = *reinterpret_cast<float (*)[32]>(x);
    auto & dw4 = *reinterpret_cast<uint32_t (*)[4]>(dw);
    if (FMT == ONPU_Q4_0) {
        uint8_t q[32];
        quant_q4_0(x32, q, s);
        // through the 16-bit words of a GGUF block: for a subnormal scale (1 / d infinite) the codes pass
        // 15, and these words are what they have always been stored as
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint16_t w = (uint16_t) ((q[2 * j] | (q[16 + 2 * j] << 4)) | ((q[2 * j + 1] | (q[17 + 2 * j] << 4)) << 8));
            q[2 * j] = w & 15;
            q[16 + 2 * j] = (w >> 4) & 15;
            q[2 * j + 1] = (w >> 8) & 15;
            q[17 + 2 * j] = w >> 12;
        }
        tile_dwords<32>(q, dw4);
    } else if (FMT == ONPU_Q4NX) quant_asym_gpu<BF>(x32, dw4, s, m);
    else quant_sym_gpu<G, BF>(x, dw, s);
    if (!in) s = m = 0;
    uint8_t * blk = out + e * ostride + (t * KB + b) * fmt_blk(FMT);
    if (G == 32) store_group32<FMT>(blk, lane, dw4, s, m);
    else if (t < NT) {
        const int r = lane & 15;
#pragma unroll
        for (int c = 0; c < 4; c++)                                            // column octet c of each 32
            *(uint4 *) (blk + 256 * c + 16 * r) = make_uint4(dw[c], dw[(4 + c) % (G / 8)], dw[(8 + c) % (G / 8)], dw[(12 + c) % (G / 8)]);
        *(uint16_t *) (blk + 1024 + 2 * r) = s;
    }
}

// grid (waves / CODEC_WAVES, experts): Q4_K rows of K / 256 super-blocks, ld bytes apart, experts
// bstride bytes apart -> q4nx tiles. A wave covers one block: 16 rows x half a super-block. The
// sub-block's 32 code bytes and the 16 header bytes come in two and one 16-byte loads (byte by byte
// and through staging, a 12288 x 4096 matrix took 142 us per call; so 61). VALU-bound: nine pairs of
// scale and min per sub-block, four ops per weight each.
__global__ __launch_bounds__(CODEC_THREADS) void k_q4k(const uint8_t * __restrict__ blocks, int64_t ld,
                                                       int64_t bstride, int64_t N, int64_t NT, int64_t KB,
                                                       uint8_t * __restrict__ out, int64_t ostride) {
    const int lane = threadIdx.x & 63;
    const int64_t w = (int64_t) blockIdx.x * CODEC_WAVES + (threadIdx.x >> 6), e = blockIdx.y, t = w / KB, b = w - t * KB;
    if (t >= NT) return;
    const int64_t n = 16 * t + (lane >> 2);
    uint32_t dw[4] = {0, 0, 0, 0};
    uint16_t s = 0, m = 0;
    if (n < N) {
        const uint8_t * p = blocks + e * bstride + n * ld + (b >> 1) * Q4K_BLOCK;
        const int sub = (int) (4 * (b & 1)) + (lane & 3);
        uint32_t h[4], c[8];
        __builtin_memcpy(h, p, sizeof(h));
        __builtin_memcpy(c, p + 16 + (sub >> 1) * 32, sizeof(c));
        uint8_t q[32];
        q4k_sub(h, c, sub, q, s, m);
        tile_dwords<32>(q, dw);
    }
    store_group32<ONPU_Q4NX>(out + e * ostride + (t * KB + b) * fmt_blk(ONPU_Q4NX), lane, dw, s, m);
}

bool codec_grid(int64_t waves, int64_t ne, dim3 & grid) {
    const int64_t gx = (waves + CODEC_WAVES - 1) / CODEC_WAVES;
    if (ne > 65535 || gx >= ((int64_t) 1 << 31)) return false;
    grid = dim3((unsigned) gx, (unsigned) ne);
    return true;
}

template <bool BF>
hipError_t quantize(int fmt, const void * W, int64_t ldw, const Tiled & g, dim3 grid, uint8_t * out, int64_t ostride,
                    hipStream_t s) {
    switch (fmt) {
    case ONPU_Q4NX: k_quantize<ONPU_Q4NX, BF><<<grid, CODEC_THREADS, 0, s>>>(W, ldw, g.N, g.K, g.NT, g.KB, out, ostride); break;
    case ONPU_Q4S: k_quantize<ONPU_Q4S, BF><<<grid, CODEC_THREADS, 0, s>>>(W, ldw, g.N, g.K, g.NT, g.KB, out, ostride); break;
    case ONPU_G128S: k_quantize<ONPU_G128S, BF><<<grid, CODEC_THREADS, 0, s>>>(W, ldw, g.N, g.K, g.NT, g.KB, out, ostride); break;
    case ONPU_Q4_0: k_quantize<ONPU_Q4_0, BF><<<grid, CODEC_THREADS, 0, s>>>(W, ldw, g.N, g.K, g.NT, g.KB, out, ostride); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_quantize(int fmt, const void * W, int64_t ldw, int wbf16, int64_t N, int64_t K, int64_t ne,
                           uint8_t * out, int64_t ostride, hipStream_t s) {
    if (ne <= 0) return hipSuccess;
    const Tiled g = tiled_geom(fmt, N, K);
    dim3 grid;
    if (!codec_grid((fmt == ONPU_G128S ? (g.NT + 3) / 4 : g.NT) * g.KB, ne, grid)) return hipErrorInvalidValue;
    return wbf16 ? quantize<true>(fmt, W, ldw, g, grid, out, ostride, s)
                 : quantize<false>(fmt, W, ldw, g, grid, out, ostride, s);
}

hipError_t launch_q4k(const uint8_t * blocks, int64_t ld, int64_t bstride, int64_t N, int64_t K, int64_t ne,
                      uint8_t * out, int64_t ostride, hipStream_t s) {
    if (ne <= 0) return hipSuccess;
    const Tiled g = tiled_geom(ONPU_Q4NX, N, K);
    dim3 grid;
    if (!codec_grid(g.NT * g.KB, ne, grid)) return hipErrorInvalidValue;
    k_q4k<<<grid, CODEC_THREADS, 0, s>>>(blocks, ld, bstride, N, g.NT, g.KB, out, ostride);
    return hipGetLastError();
}
