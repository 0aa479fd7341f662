// skinny.hip -- batched GEMV / skinny GEMM on the fp16 matrix cores for
// 2 <= M <= 32 token rows and Q4_K / Q5_K / Q6_K weights of any K (the batched
// shape of phi4.rs:1257-1268: Y[m][n] = sum_k X[m][k] * W[n][k], X and Y f32
// row-major).
//
// Exact weights.  For super-block b of row n,
//     sum_k x_k w_k = d * sum_s sum_{k in s} sc_s (q_k - c) x_k
//                     + sum_s (c d sc_s - dmin mn_s) X_s
// (phi4.rs:481-542, w = d*sc*q - dmin*mn), X_s the sum of x over sub-block s and c
// the middle of the quants (8 or 16).  sc_s (q_k - c) is an integer of at most
// 1008, exact in fp16: the MFMA B operand carries it, the 8 sub-blocks of a block
// accumulate in the MFMA's f32 accumulator, and d, dmin are applied once per block.
// The sums' terms are small MFMAs (16x16x16) of the X_s against sc_s and mn_s.
// With c = 0 the f32 sums are those of products of one sign, about twice as large
// as what they come to, and 4 times as far from it where x has a mean (M > 16, of
// f16 activations, has c = 0: sc_s q_k <= 1953 < 2^11).
// Error to 64 bits, M <= 16, K = 8192, weights of mean zero (with c = 0; the VALU
// kernel's, f32 throughout): even rows Q4_K 1.1e-7 (2.5e-7; 1.9e-7), Q5_K 1.2e-7
// (2.6e-7; 2.0e-7), Q6_K 1.2e-7 (VALU 2.0e-7); log-normal rows 1.3e-7 to 1.6e-7
// (2.6e-7 to 3.0e-7; 1.8e-7 to 2.3e-7); rows with a mean 1.2e-7 to 1.7e-7
// (1.8e-6; 4.1e-7 to 4.3e-7).
//
// Activations.  A wave's K slice (one super-block) of token m is scaled by
// 2^-E (E from the slice maximum, so the values lie below 2^14) and split
// x = hi + lo, hi = fp16(x), lo = fp16(x - hi), off by at most 2^-23 of x or 2^-39
// of the slice maximum.  M <= 16: A rows 2m+h (h = 0 hi, 1 lo), 8 tokens per 16-row
// A tile (the GEMV bar, 1e-4).  16 < M <= 32: A rows are 16 tokens of hi only
// (error 2^-12, the MFMA bar 2e-3).  The X_s are scaled by 2^-(E+5)
// (|X_s| <= 32 max) and split the same way; d and dmin take the 2^E back.
//
// MFMA layouts (lane l): 16x16x32 f16 -- A row l%16 / B column l%16 at
// k = 8(l/16) .. +7; 16x16x16 f16 -- the same at k = 4(l/16) .. +3; D rows
// 4(l/16)+r of column l%16 in register r.
//
// Encoding pass.  The A operands depend only on X, so a small kernel
// (skinny_encode_kernel) builds them once per call into the workspace, in the
// lane order of the MFMA:
//   av   [TOK][B][8][64] f16x8  lane's 8 values of sub-block s
//   amin [TOK][B][64]    f16x4  lane's 4 sub-block sums (A operand of their terms)
//   pe   [TOK][B][16]    f32    2^E of the A tile's token r (8 or 16 of them)
// (B = K/256 columns, TOK A tiles), 8,768 bytes per (tile, column).  Every
// workgroup of the main kernel then loads its operands with 16-byte loads
// instead of reading all of X in f32 and converting it again: at 8 rows QKV
// 5120x3072 takes 9.5 us against 10.1 with the operands built in every wave,
// gate+up 16384x3072 13.8 against 14.5.  Short rows are the other way round (see
// go_skinny).
//
// Work split: a workgroup of W waves takes the 16-row tiles b, b + G, ... (G =
// gridDim.x), T of them at a time; wave w owns the super-block columns w,
// w + W, ... of every row.  It walks its columns: the column's A operands in
// registers (the next column's requested meanwhile), then the T tiles' 16
// blocks of that column, staged in the wave's private LDS ring by LDS DMA (the
// next units in flight).  The row sums of the T tiles stay in registers over
// all columns; one barrier per T tiles, then the waves' partials are added in
// wave order.
//
// Q6_K.  p = sc_s (q - 32) reaches 127 * 32 = 4064, 13 bits with sign: one
// fp16 holds it up to 2048, above that to the next even number.  B hi =
// fp16(p) and B lo = p - B hi (exact, one packed fma) are two MFMAs on the same
// A operand, so the weight stays exact at the hi/lo activations; with hi
// activations alone (M > 16) B hi is taken alone, its 2^-12 is that bar's.
// A 210-byte block starts 2 bytes past a dword when its index is odd: rows are
// loaded from the dword below (14 units of 16 bytes a row) and moved down 2
// bytes in registers (v_alignbyte).
//
// Bound: HBM at every M in principle (20.6 MB of Q6_K in 2.9 us); in fact a CU's
// intake (at K = 8192 and 8 rows 262 KB of A operands next to its 80 KB of
// weights) and the decode (counted at 8 rows: 200 VALU instructions a unit of 16
// columns x 256 for Q4_K, 240 for Q5_K; three waves a SIMD).
// Measured per call, graphs over 300 MB of weight copies, in us, against the
// VALU kernel (four rows a pass over the weights) and, at 27 rows, the row
// conversion + prefill GEMM + split reduction that took these shapes before:
//   3072x8192 Q6_K  8 rows 16.3 (69), 16 rows 19.5 (134), 27 rows 19.6 (29.7)
//   3072x8192 Q4_K  8 rows 14.2 (39), 16 rows 17.2 (71),  27 rows 18.0 (25.8)
// and against the form with one column a wave and a barrier per tile:
//   16384x3072 Q4_K 8 rows 13.8 (15.6), 27 rows 16.2 (18.3)
//   5120x3072 Q5_K  8 rows 9.5 (11.0),  27 rows 11.2 (12.4)
#include "device_common.h"
#include "internal.h"

#include <type_traits>

namespace rrr {

typedef _Float16 f16x8s __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4s __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2s __attribute__((ext_vector_type(2)));

// Lane offset past every weight byte (w_bytes + RRR_READ_SLACK must stay below
// it): such loads return zeros and move no data.
constexpr uint32_t SK_OOB = 0x80000000u;

__device__ __forceinline__ f16x2s sk_bits(uint32_t v) { return __builtin_bit_cast(f16x2s, v); }
__device__ __forceinline__ uint32_t sk_u32(f16x2s v) { return __builtin_bit_cast(uint32_t, v); }

// Four quant values times the scale as exact fp16: v_perm places the bytes of v under
// the exponent of 1024 (f16 0x64vv = 1024 + v).  Plain, the bytes are q and
// fma(1024 + q, sc, -1024 sc) = sc q < 2^11; less their middle c, they are 64 q / c
// and fma(1024 + 64 q / c, sc c / 64, -(1024 + 64) sc c / 64) = sc (q - c), where
// 17 sc has 11 bits and |sc (q - c)| <= 1008.
__device__ __forceinline__ void sk_scale4(uint32_t v, f16x2s sc2, f16x2s nb2, uint32_t &o01, uint32_t &o23)
{
    o01 = sk_u32(__builtin_elementwise_fma(sk_bits(__builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)), sc2, nb2));
    o23 = sk_u32(__builtin_elementwise_fma(sk_bits(__builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)), sc2, nb2));
}

// Q4_K (phi4.rs:481-510): element 32s + e of a block is nibble (s & 1) of
// qs[32 (s/2) + e].  Lane k-group kg takes e = 8kg .. 8kg+7 of every s.
struct SkQ4K {
    static constexpr uint32_t BS = 144, LROW = 144;   // bytes of a block, and of its row in LDS
    static constexpr bool MINS = true;                // a min term (d*sc*q - dmin*mn)
    static constexpr uint32_t MID = 8;                // the middle of the quants
    struct Raw { u32x4 hdr; u32x2 qs[4]; };
    __device__ static void load(Raw &r, const uint8_t *L, uint32_t o, uint32_t kg, uint32_t)
    {
        r.hdr = *(const u32x4 *)(L + o);
#pragma unroll
        for (int p = 0; p < 4; p++) r.qs[p] = *(const u32x2 *)(L + o + 16 + 32 * p + 8 * kg);
    }
    // quant values of sub-block s at the lane's 8 positions, one per byte (C: times 8)
    template <bool C>
    __device__ static void quants(const Raw &r, int s, uint32_t &v0, uint32_t &v1)
    {
        const u32x2 q = r.qs[s >> 1];
        if constexpr (C) {
            v0 = (s & 1 ? q.x >> 1 : q.x << 3) & 0x78787878u;
            v1 = (s & 1 ? q.y >> 1 : q.y << 3) & 0x78787878u;
        } else {
            v0 = (q.x >> (4 * (s & 1))) & 0x0F0F0F0Fu;
            v1 = (q.y >> (4 * (s & 1))) & 0x0F0F0F0Fu;
        }
    }
};

// Q5_K (phi4.rs:512-542): Q4_K's nibbles plus bit s of qh[e] as bit 4.
struct SkQ5K {
    static constexpr uint32_t BS = 176, LROW = 176;
    static constexpr bool MINS = true;
    static constexpr uint32_t MID = 16;
    struct Raw { u32x4 hdr; u32x2 qh; u32x2 qs[4]; };
    __device__ static void load(Raw &r, const uint8_t *L, uint32_t o, uint32_t kg, uint32_t)
    {
        r.hdr = *(const u32x4 *)(L + o);
        r.qh = *(const u32x2 *)(L + o + 16 + 8 * kg);
#pragma unroll
        for (int p = 0; p < 4; p++) r.qs[p] = *(const u32x2 *)(L + o + 48 + 32 * p + 8 * kg);
    }
    template <bool C>   // C: times 4
    __device__ static void quants(const Raw &r, int s, uint32_t &v0, uint32_t &v1)
    {
        const u32x2 q = r.qs[s >> 1];
        if constexpr (C) {
            v0 = ((s & 1 ? q.x >> 2 : q.x << 2) & 0x3C3C3C3Cu) | ((s < 7 ? r.qh.x << (6 - s) : r.qh.x >> 1) & 0x40404040u);
            v1 = ((s & 1 ? q.y >> 2 : q.y << 2) & 0x3C3C3C3Cu) | ((s < 7 ? r.qh.y << (6 - s) : r.qh.y >> 1) & 0x40404040u);
        } else {
            v0 = ((q.x >> (4 * (s & 1))) & 0x0F0F0F0Fu) | (((r.qh.x >> s) & 0x01010101u) << 4);
            v1 = ((q.y >> (4 * (s & 1))) & 0x0F0F0F0Fu) | (((r.qh.y >> s) & 0x01010101u) << 4);
        }
    }
};

// Q6_K (phi4.rs:444-479): element 32s + e of a block is nibble (s % 4) / 2 of
// ql[64 (s/4) + 32 (s & 1) + e] and bits 2 (s % 4) .. +1 of qh[32 (s/4) + e],
// minus 32, times sc[2s + e/16].  The block starts `odd` (0 or 2) bytes into
// its LDS row.
struct SkQ6K {
    static constexpr uint32_t BS = 210, LROW = 224;
    static constexpr bool MINS = false;
    struct Raw { u32x2 ql[4], qh[2]; uint32_t sc[4]; uint32_t d; };
    // 8 bytes at p + odd, p 8-byte aligned
    __device__ static u32x2 at(const uint8_t *p, uint32_t odd)
    {
        const u32x2 v = *(const u32x2 *)p;
        const uint32_t n = *(const uint32_t *)(p + 8);
        return u32x2{__builtin_amdgcn_alignbyte(v.y, v.x, odd), __builtin_amdgcn_alignbyte(n, v.y, odd)};
    }
    __device__ static void load(Raw &r, const uint8_t *L, uint32_t o, uint32_t kg, uint32_t odd)
    {
        const uint8_t *p = L + o;
#pragma unroll
        for (int i = 0; i < 4; i++) r.ql[i] = at(p + 32 * i + 8 * kg, odd);
#pragma unroll
        for (int i = 0; i < 2; i++) r.qh[i] = at(p + 128 + 32 * i + 8 * kg, odd);
        const u32x4 c = *(const u32x4 *)(p + 192);
        const uint32_t e = *(const uint32_t *)(p + 208);
        r.sc[0] = __builtin_amdgcn_alignbyte(c.y, c.x, odd);
        r.sc[1] = __builtin_amdgcn_alignbyte(c.z, c.y, odd);
        r.sc[2] = __builtin_amdgcn_alignbyte(c.w, c.z, odd);
        r.sc[3] = __builtin_amdgcn_alignbyte(e, c.w, odd);
        r.d = e >> (8 * odd);
    }
    template <bool>
    __device__ static void quants(const Raw &r, int s, uint32_t &v0, uint32_t &v1)
    {
        const int g = s >> 2, q = s & 3;
        const u32x2 l = r.ql[2 * g + (q & 1)], h = r.qh[g];
        v0 = ((l.x >> (4 * (q >> 1))) & 0x0F0F0F0Fu) | (((h.x >> (2 * q)) & 0x03030303u) << 4);
        v1 = ((l.y >> (4 * (q >> 1))) & 0x0F0F0F0Fu) | (((h.y >> (2 * q)) & 0x03030303u) << 4);
    }
};

// Four quant values (bytes < 64 of v) minus 32, times the scale, as fp16 hi + lo.
__device__ __forceinline__ void sk_scale4_q6(uint32_t v, f16x2s sc2, uint32_t (&hi)[2], uint32_t (&lo)[2])
{
    const f16x2s off = {(_Float16)1056.0f, (_Float16)1056.0f};
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const f16x2s q = sk_bits(__builtin_amdgcn_perm(0x64646464u, v, i ? 0x04030402u : 0x04010400u)) - off;
        const f16x2s h = q * sc2;
        hi[i] = sk_u32(h);
        lo[i] = sk_u32(__builtin_elementwise_fma(q, sc2, -h));
    }
}

// Staging geometry of one wave's 16 block pieces, loaded straight into LDS
// (16-byte LDS DMA: lane l of a load writes base + 16 l).  Load slot s covers
// rows s*RPS .. s*RPS+RPS-1 (lane l: unit l % UPB of row l / UPB) and has a
// 1 KB LDS slot of its own, so lanes past the slot's rows (which read nothing
// and write zeros) stay inside it.  A tile buffer is S slots.
template <class Q>
struct SkGeom {
    static constexpr uint32_t UPB = Q::LROW / 16;
    static constexpr uint32_t RPS = 64 / UPB;
    static constexpr int S = (16 + RPS - 1) / RPS;
    static constexpr uint32_t BUF = 1024 * S;
    // LDS offset of row r inside a tile buffer
    __device__ static uint32_t row_off(uint32_t r) { return (r / RPS) * 1024 + (r % RPS) * Q::LROW; }
};

// Workspace layout of the encoded activations (see the top of this file).
constexpr uint32_t SK_AV_UNIT = 8 * 64 * 16, SK_AMIN_UNIT = 64 * 8, SK_PE_UNIT = 16 * 4;
__host__ __device__ constexpr uint64_t sk_ws_bytes(uint32_t tok, uint32_t B)
{
    return (uint64_t)tok * B * (SK_AV_UNIT + SK_AMIN_UNIT + SK_PE_UNIT);
}
struct SkWs {
    uint32_t amin, pe, bytes;   // byte offsets of the parts (av at 0), and the end
    __host__ __device__ SkWs(uint32_t tok, uint32_t B)
        : amin(tok * B * SK_AV_UNIT), pe(amin + tok * B * SK_AMIN_UNIT), bytes(pe + tok * B * SK_PE_UNIT)
    {
    }
};

// max |.| and sum of 8 values
__device__ __forceinline__ float sk_max8(const float4 &u, const float4 &v)
{
    return fmaxf(fmaxf(fmaxf(fabsf(u.x), fabsf(u.y)), fmaxf(fabsf(u.z), fabsf(u.w))),
                 fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
}
__device__ __forceinline__ float sk_sum8(const float4 &u, const float4 &v)
{
    return ((u.x + u.y) + (u.z + u.w)) + ((v.x + v.y) + (v.z + v.w));
}
// E of a slice whose largest |x| is mx: mx / 2^E in [2^13, 2^14)
__device__ __forceinline__ int sk_exponent(float mx)
{
    int ex = 14;
    if (mx > 0.0f && __builtin_isfinite(mx)) (void)frexpf(mx, &ex);
    return ex - 14;
}
// v / 2^e in f16: its hi or lo half (ldexp: times 2^-e would overflow for a
// slice below 2^-113), 0 for a row past M
__device__ __forceinline__ _Float16 sk_half(float v, int e, bool lo, bool live)
{
    const float y = ldexpf(v, -e);
    const _Float16 hi = (_Float16)y;
    return live ? (lo ? (_Float16)(y - (float)hi) : hi) : (_Float16)0.0f;
}
__device__ __forceinline__ f16x8s sk_values(const float4 &u, const float4 &v, int e, bool lo, bool live)
{
    const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
    f16x8s h;
#pragma unroll
    for (int i = 0; i < 8; i++) h[i] = sk_half(f[i], e, lo, live);
    return h;
}

// The encoding pass: one workgroup of four waves per (super-block column, A
// tile), grid (B, TOK).  Lane (row r16, group kg) of wave q takes token tok's
// values 32 s + 8 kg + i (i < 8) of sub-blocks s = 2q, 2q + 1.  Bound by latency
// (a load, a maximum over the slice, a store): one wave for all eight sub-blocks
// was a chain of ~600 instructions (with this split QKV 5120x3072 at 16 rows
// went from 12.1 to 11.2 us a call).  HILO: 8 tokens (hi, lo rows) per A tile,
// else 16 tokens (hi rows).
template <bool HILO>
__global__ __launch_bounds__(256) void skinny_encode_kernel(const float *__restrict__ x, uint32_t M, uint32_t K,
                                                            uint8_t *ws, uint32_t tok_tiles)
{
    __shared__ float wmax[4][16], gsum[8][16];
    const uint32_t B = K / 256, c = blockIdx.x, tt = blockIdx.y, lane = threadIdx.x & 63, q = threadIdx.x >> 6;
    const uint32_t r16 = lane & 15, kg = lane >> 4;
    const SkWs o(tok_tiles, B);
    const uint32_t tok = HILO ? tt * 8 + (r16 >> 1) : tt * 16 + r16;
    const bool lo = HILO && (r16 & 1);
    const bool live = tok < M;
    const float4 *xp = (const float4 *)(x + (uint64_t)min(tok, M - 1) * K + c * 256 + 64 * q + 8 * kg);
    const float4 xv[4] = {xp[0], xp[1], xp[8], xp[9]};
    float mx = 0.0f, gs[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const float4 u = xv[2 * s], v = xv[2 * s + 1];
        mx = fmaxf(mx, sk_max8(u, v));
        gs[s] = sk_sum8(u, v);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
#pragma unroll
    for (int s = 0; s < 2; s++) {
        gs[s] = gs[s] + __shfl_xor(gs[s], 16, 64);
        gs[s] = gs[s] + __shfl_xor(gs[s], 32, 64);
    }
    if (kg == 0) {
        wmax[q][r16] = mx;
        gsum[2 * q][r16] = gs[0];
        gsum[2 * q + 1][r16] = gs[1];
    }
    __syncthreads();
    const int e = sk_exponent(fmaxf(fmaxf(wmax[0][r16], wmax[1][r16]), fmaxf(wmax[2][r16], wmax[3][r16])));
    u32x4 *ap = (u32x4 *)ws + (uint64_t)(tt * B + c) * 8 * 64 + lane;
#pragma unroll
    for (int s = 0; s < 2; s++)
        ap[(2 * q + s) * 64] = __builtin_bit_cast(u32x4, sk_values(xv[2 * s], xv[2 * s + 1], e, lo, live));
    if (q != 0) return;
    f16x4s am;
#pragma unroll
    for (int i = 0; i < 4; i++) am[i] = sk_half(gsum[(4 * kg + i) & 7][r16], e + 5, lo, live && kg < 2);
    ((u32x2 *)(ws + o.amin))[(uint64_t)(tt * B + c) * 64 + lane] = __builtin_bit_cast(u32x2, am);
    // lanes 0..15 hold A rows 0..15: rows 2t, 2t + 1 (HILO) or row t are token t
    if (lane < 16 && (!HILO || !(lane & 1)))
        ((float *)(ws + o.pe))[(tt * B + c) * 16 + (HILO ? lane >> 1 : lane)] = ldexpf(1.0f, e);
}

// The A operands of one super-block column: TOK A tiles, pe the 2^E of the
// lane's D-layout tokens (D row 4 kg + j holds A row 4 kg + j: HILO token
// 2 kg + j / 2, else token 4 kg + j).
template <int TOK, int DPT>
struct SkA {
    f16x8s av[TOK][8];
    f16x4s amin[TOK];
    float pe[TOK][DPT];
};

// The same operands of one column and one A tile of 8 tokens built by the wave that
// uses them, from its lane's values of the column (16 float4, two a sub-block):
// the bits of skinny_encode_kernel.
__device__ __forceinline__ void sk_build(SkA<1, 2> &x, const float4 (&xv)[16], uint32_t lane, uint32_t M)
{
    const uint32_t r16 = lane & 15, kg = lane >> 4;
    const bool lo = r16 & 1, live = (r16 >> 1) < M;
    float mx = 0.0f, gs[8];
#pragma unroll
    for (int s = 0; s < 8; s++) {
        mx = fmaxf(mx, sk_max8(xv[2 * s], xv[2 * s + 1]));
        gs[s] = lanes4_sum(sk_sum8(xv[2 * s], xv[2 * s + 1]));
    }
    const int e = sk_exponent(lanes4_max(mx));
#pragma unroll
    for (int s = 0; s < 8; s++) x.av[0][s] = sk_values(xv[2 * s], xv[2 * s + 1], e, lo, live);
#pragma unroll
    for (int i = 0; i < 4; i++) x.amin[0][i] = sk_half(kg == 0 ? gs[i] : gs[4 + i], e + 5, lo, live && kg < 2);
#pragma unroll
    for (int j = 0; j < 2; j++) x.pe[0][j] = ldexpf(1.0f, __shfl(e, 4 * kg + 2 * j, 64));
}

// Tile buffers a wave of a WMAX-wave workgroup gets out of the 160 KB of LDS.
template <class Q, int WMAX>
constexpr int sk_ring()
{
    constexpr int n = 160 * 1024 / (WMAX * (int)SkGeom<Q>::BUF);
    return n > 4 ? 4 : n;
}

// TOK A tiles (TPT tokens each); DPT = tokens of a tile per lane in the D
// layout; T tiles at a time.  At most WMAX waves, NB = sk_ring tile buffers
// per wave: units u + 1 .. u + NB - 1 stream in while unit u is multiplied
// (unit = column, tile).  DB: more than one column a wave, the next column's A
// operands requested one column ahead.  ENC: one column a wave, its A operands
// built here instead of by the encoding pass.
template <class Q, bool HILO, int TOK, int T, int WMAX, bool DB, bool ENC>
__global__ __launch_bounds__(64 * WMAX) void skinny_kernel(GemvArgs a, uint32_t ntiles)
{
    using G = SkGeom<Q>;
    constexpr int TPT = HILO ? 8 : 16, DPT = HILO ? 2 : 4, MP = TOK * TPT, NB = sk_ring<Q, WMAX>();
    constexpr int NA = DB ? TOK * (9 + (Q::MINS ? 1 : 0)) : 0;   // loads of one column's A operands
    constexpr int AHEAD = DB || NB - 1 < T ? NB - 1 : T;         // units issued before the first
    static_assert(!ENC || (HILO && TOK == 1 && !DB), "operands built in the wave: one column, one A tile");
    static_assert(NB >= 2 && NB * G::BUF >= (uint32_t)T * MP * 64, "ring: two units, and the wave's row sums");
    extern __shared__ float smem[];
    const uint32_t K = a.K, M = a.M, N = a.N, B = K / 256, W = blockDim.x / 64;
    const uint32_t t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t r16 = lane & 15, kg = lane >> 4;
    const uint32_t GR = gridDim.x, tile0 = blockIdx.x;
    const uint32_t Cw = (B - wave + W - 1) / W;          // this wave's columns wave, wave + W, ... (W <= B)
    uint8_t *L = (uint8_t *)smem + wave * NB * G::BUF;   // this wave's tile buffers, then its row sums

    const uint32_t row_bytes = B * Q::BS;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.W, a.w_bytes + RRR_READ_SLACK);

    // weight units: lane-fixed offsets, a uniform offset per load slot; rows
    // past 16 in the last slot read nothing
    const uint32_t rsel = min(lane / G::UPB, G::RPS - 1), vl = lane - (lane / G::UPB) * G::UPB;
    const bool lane_ok = lane < G::RPS * G::UPB;
    const bool last_ok = lane_ok && (G::S - 1) * G::RPS + rsel < 16;
    const uint32_t tile_bytes = 16 * row_bytes;
    // tile `tile` of the wave's column ci into buffer `buf` (S loads; past the
    // last tile or column: zeros).  Q6_K: an odd block from the dword below (a
    // tile's and a slot's first rows have even block numbers, as S * RPS = 16
    // and RPS = 4 rows)
    auto dma = [&](uint32_t ci, uint32_t tile, uint32_t buf) {
        const uint32_t c = wave + ci * W;
        const uint32_t odd = Q::MINS ? 0u : 2 * ((rsel * B + c) & 1);
        const uint32_t v = rsel * row_bytes + c * Q::BS - odd + 16 * vl;
        const bool live = ci < Cw && tile < ntiles;
        const uint32_t tb = live ? tile * tile_bytes : 0u;
        uint8_t *dst = L + buf * G::BUF;
#pragma unroll
        for (int s = 0; s < G::S; s++)
            lds_dma16<RRR_CPOL_NT>(rs, dst + 1024 * s, live && (s == G::S - 1 ? last_ok : lane_ok) ? v : SK_OOB,
                                   tb + s * G::RPS * row_bytes);
    };

    // A operands of the wave's column ci from the encoding pass (NA loads;
    // past the last column: no request)
    using A = SkA<TOK, DPT>;
    const SkWs o(TOK, B);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(a.ws, o.bytes);
    auto load_a = [&](A &x, uint32_t ci) {
        const uint32_t out = ci < Cw ? 0u : RRR_OOB, c = wave + ci * W;
#pragma unroll
        for (int tt = 0; tt < TOK; tt++) {
            const uint32_t u = tt * B + (ci < Cw ? c : 0u);
#pragma unroll
            for (int s = 0; s < 8; s++)
                x.av[tt][s] = __builtin_bit_cast(f16x8s, bload16_so(ra, (lane * 16 + s * 1024) | out, u * SK_AV_UNIT));
            if constexpr (Q::MINS)
                x.amin[tt] = __builtin_bit_cast(
                    f16x4s, __builtin_amdgcn_raw_buffer_load_b64(ra, (lane * 8) | out, o.amin + u * SK_AMIN_UNIT, 0));
            const uint32_t po = o.pe + u * SK_PE_UNIT;
            if constexpr (HILO) {
                const u32x2 p = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(ra, (8 * kg) | out, po, 0));
                x.pe[tt][0] = u2f(p.x);
                x.pe[tt][1] = u2f(p.y);
            } else {
                const u32x4 p = bload16_so(ra, (16 * kg) | out, po);
                x.pe[tt][0] = u2f(p.x);
                x.pe[tt][1] = u2f(p.y);
                x.pe[tt][DPT - 2] = u2f(p.z);
                x.pe[tt][DPT - 1] = u2f(p.w);
            }
        }
    };

    const uint32_t roff = G::row_off(r16);
    float tot[T][TOK][DPT];   // row sums of the T tiles over the wave's columns
    uint32_t buf = 0, tb0 = tile0;   // ring place of the next unit; the first of the T tiles

    // one unit: tile ti of the T (static), the column's A operands in x
    auto unit = [&](const A &x, uint32_t ci, auto tic) {
        constexpr int ti = decltype(tic)::value;
        // the unit NB - 1 ahead into the buffer the last unit left, once its
        // LDS reads are done (a DMA that is out of range writes its zeros at once)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        // (one column a wave: none past its T tiles)
        const uint32_t ahead = buf == 0 ? NB - 1 : buf - 1;
        if constexpr (DB || ti + NB - 1 < T) dma(ci + (ti + NB - 1) / T, tb0 + ((ti + NB - 1) % T) * GR, ahead);
        // this unit landed: issued before the next column's A operands if it
        // is one of the column's first NB - 1, after them otherwise
        constexpr int later = DB || ti + NB - 1 < T ? NB - 1 : T - 1 - ti;   // units issued after it
        constexpr int n = later * G::S + (ti <= NB - 2 ? NA : 0);
        wait_vm<(n < 63 ? n : 63)>();
        typename Q::Raw raw;
        const uint32_t odd = Q::MINS ? 0u : 2 * ((r16 * B + wave + ci * W) & 1);
        Q::load(raw, L + buf * G::BUF, roff, kg, odd);
        buf = buf + 1 == NB ? 0 : buf + 1;
        f32x4 acc[TOK];
#pragma unroll
        for (int tt = 0; tt < TOK; tt++) acc[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
        const f16x2s k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
        if constexpr (Q::MINS) {
            const float d = h2f(raw.hdr.x), dmin = h2f(raw.hdr.x >> 16);
            uint32_t scb[2], mnb[2];
            scale_min_bytes_k4(raw.hdr.y, raw.hdr.z, raw.hdr.w, scb, mnb);
            // B operands of the sub-block sums: sc and mn of sub-blocks 4 kg .. 4 kg + 3
            // (k-groups 2, 3 padding, whose A is 0)
            auto bytes4 = [&](uint32_t v) {
                const f16x2s a = sk_bits(__builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)) - k1024;
                const f16x2s b = sk_bits(__builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)) - k1024;
                return f16x4s{a[0], a[1], b[0], b[1]};
            };
            const f16x4s bsc = bytes4(kg == 0 ? scb[0] : scb[1]), bmin = bytes4(kg == 0 ? mnb[0] : mnb[1]);
#pragma unroll
            for (int s = 0; s < 8; s++) {
                // {sc_s, sc_s}, for centred quants times MID / 64, exactly: byte s under the
                // exponent of 1024 (16 MID), less that
                constexpr uint32_t base = HILO ? 16 * Q::MID : 1024, ex = base == 128 ? 0x58585858u : base == 256 ? 0x5C5C5C5Cu : 0x64646464u;
                const f16x2s sc2 = sk_bits(__builtin_amdgcn_perm(ex, scb[s >> 2], 0x04000400u + 0x00010001u * (s & 3))) -
                                   f16x2s{(_Float16)base, (_Float16)base};
                constexpr float off = HILO ? -1088.0f : -1024.0f;
                const f16x2s nb2 = sc2 * f16x2s{(_Float16)off, (_Float16)off};
                uint32_t v0, v1, b[4];
                Q::template quants<HILO>(raw, s, v0, v1);
                sk_scale4(v0, sc2, nb2, b[0], b[1]);
                sk_scale4(v1, sc2, nb2, b[2], b[3]);
                const f16x8s bv = __builtin_bit_cast(f16x8s, u32x4{b[0], b[1], b[2], b[3]});
#pragma unroll
                for (int tt = 0; tt < TOK; tt++) acc[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.av[tt][s], bv, acc[tt], 0, 0, 0);
                // one sub-block's B operand live at a time
                if constexpr (TOK > 1) __builtin_amdgcn_sched_barrier(0);
            }
            // the row partials
            const float ds = (32.0f * Q::MID) * d, dm = 32.0f * dmin;
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int tt = 0; tt < TOK; tt++) {
                const f32x4 sm = __builtin_amdgcn_mfma_f32_16x16x16f16(x.amin[tt], bmin, zero, 0, 0, 0);
                if constexpr (HILO) {
                    // the two terms of the X_s nearly cancel where these are large: the
                    // difference of the hi parts is taken exactly (the product's rounding
                    // comes back), then the lo parts join
                    const f32x4 ss = __builtin_amdgcn_mfma_f32_16x16x16f16(x.amin[tt], bsc, zero, 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < DPT; j++) {
                        const int h = 2 * j;
                        const float p = dm * sm[h];
                        float v = fmaf(ds, ss[h], -p) - fmaf(dm, sm[h], -p);
                        v = fmaf(-dm, sm[h + 1], fmaf(ds, ss[h + 1], v));
                        v = fmaf(d, acc[tt][h], fmaf(d, acc[tt][h + 1], v));
                        tot[ti][tt][j] = fmaf(x.pe[tt][j], v, tot[ti][tt][j]);
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < DPT; j++)
                        tot[ti][tt][j] = fmaf(x.pe[tt][j], fmaf(d, acc[tt][j], -dm * sm[j]), tot[ti][tt][j]);
                }
            }
        } else {
            const float d = h2f(raw.d);
            const uint32_t sel = 0x04000400u + 0x00010001u * (kg >> 1);   // byte kg / 16 of a scale pair
#pragma unroll
            for (int s = 0; s < 8; s++) {
                // {sc, sc} exactly: byte sc + 128 under the exponent of 1024, minus 1152
                const f16x2s sc2 = sk_bits(__builtin_amdgcn_perm(0x64646464u, raw.sc[s >> 1] ^ 0x80808080u, sel + 0x00020002u * (s & 1))) -
                                   f16x2s{(_Float16)1152.0f, (_Float16)1152.0f};
                uint32_t v0, v1, h0[2], h1[2], l0[2], l1[2];
                Q::template quants<HILO>(raw, s, v0, v1);
                sk_scale4_q6(v0, sc2, h0, l0);
                sk_scale4_q6(v1, sc2, h1, l1);
                const f16x8s bh = __builtin_bit_cast(f16x8s, u32x4{h0[0], h0[1], h1[0], h1[1]});
                const f16x8s bl = __builtin_bit_cast(f16x8s, u32x4{l0[0], l0[1], l1[0], l1[1]});
#pragma unroll
                for (int tt = 0; tt < TOK; tt++) {
                    acc[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.av[tt][s], bh, acc[tt], 0, 0, 0);
                    if constexpr (HILO) acc[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.av[tt][s], bl, acc[tt], 0, 0, 0);
                }
                if constexpr (TOK > 1) __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int tt = 0; tt < TOK; tt++)
#pragma unroll
                for (int j = 0; j < DPT; j++) {
                    const float sv = HILO ? acc[tt][2 * j] + acc[tt][2 * j + 1] : acc[tt][j];
                    tot[ti][tt][j] = fmaf(x.pe[tt][j], d * sv, tot[ti][tt][j]);
                }
        }
    };
    auto column = [&](const A &x, A &next, uint32_t ci) {
        if constexpr (DB) {
            load_a(next, ci + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        unit(x, ci, std::integral_constant<int, 0>{});
        if constexpr (T > 1) unit(x, ci, std::integral_constant<int, 1>{});
        if constexpr (T > 2) {
            unit(x, ci, std::integral_constant<int, 2>{});
            unit(x, ci, std::integral_constant<int, 3>{});
        }
    };

    // the first units of the T tiles
    auto start = [&] {
#pragma unroll
        for (int u = 0; u < AHEAD; u++) dma(u / T, tb0 + (u % T) * GR, u);
    };
    A x0, x1;
    if constexpr (ENC) {
        const float4 *xp = (const float4 *)(a.x + (uint64_t)min(r16 >> 1, M - 1) * K + wave * 256 + 8 * kg);
        float4 xv[16];
#pragma unroll
        for (int s = 0; s < 8; s++) {
            xv[2 * s] = xp[8 * s];
            xv[2 * s + 1] = xp[8 * s + 1];
        }
        __builtin_amdgcn_sched_barrier(0);
        start();
        sk_build(x0, xv, lane, M);
    }
    for (; tb0 < ntiles; tb0 += T * GR) {
        // the first columns' A operands, then the first units: loads return in
        // order, so unit 0 waits for the A operands and its own weights only
        if constexpr (!ENC) {
            load_a(x0, 0);
            __builtin_amdgcn_sched_barrier(0);
            start();
        } else if (tb0 != tile0) {
            start();
        }
#pragma unroll
        for (int ti = 0; ti < T; ti++)
#pragma unroll
            for (int tt = 0; tt < TOK; tt++)
#pragma unroll
                for (int j = 0; j < DPT; j++) tot[ti][tt][j] = 0.0f;
        buf = 0;
        if constexpr (DB) {
            for (uint32_t ci = 0; ci < Cw; ci += 2) {
                column(x0, x1, ci);
                if (ci + 1 < Cw) column(x1, x0, ci + 1);
            }
        } else {
            column(x0, x1, 0);
        }
        // the wave's row sums over its ring (every DMA into it has landed, its
        // reads are done)
        wait_vm<0>();
        float *pp = (float *)L + r16;
#pragma unroll
        for (int ti = 0; ti < T; ti++)
#pragma unroll
            for (int tt = 0; tt < TOK; tt++)
#pragma unroll
                for (int j = 0; j < DPT; j++)
                    pp[(ti * MP + tt * TPT + (HILO ? 2 * kg + j : 4 * kg + j)) * 16] = tot[ti][tt][j];
        __syncthreads();
        // the W waves' partials in wave order, in 64 bits (a 12-long f32 chain was a
        // tenth of the error; no time)
        for (uint32_t i = t; i < T * MP * 16; i += 64 * W) {
            const uint32_t ti = i / (MP * 16), m = (i >> 4) % MP, c = i & 15, row = (tb0 + ti * GR) * 16 + c;
            if (m < M && row < N) {
                float v = ordered_sum<WMAX, double>(smem + i, W, NB * G::BUF / 4);
                float *yp = a.y + (uint64_t)m * N + row;
                if (a.residual) v = *yp + v;
                *yp = v;
            }
        }
        // the ring takes the next tiles' weights; nothing to wait for (the
        // stores, too) after the last
        if (tb0 + T * GR < ntiles) __syncthreads();
    }
}

template <class Q, bool HILO, int TOK, int T, int WMAX, bool DB, bool ENC>
static hipError_t go_skinny_t(const GemvArgs &a, uint32_t waves, uint32_t ntiles, uint32_t grid, hipStream_t s)
{
    const size_t lds = (size_t)waves * sk_ring<Q, WMAX>() * SkGeom<Q>::BUF;
    hipLaunchKernelGGL((skinny_kernel<Q, HILO, TOK, T, WMAX, DB, ENC>), dim3(grid), dim3(64 * waves), lds, s, a, ntiles);
    return hipGetLastError();
}

// One workgroup per CU at most, the tiles spread evenly over them, T of them
// at a time (one per workgroup: 1, two: 2, more: 4, or 2 where two columns'
// operands of two A tiles, or of one beside the sums' terms, leave no registers
// for it: 20000x5120 at 8 rows 39 us with 4, which spill, 32 with 2).  C columns a wave, the
// fewest that need no more than WMAX waves.
template <class Q, bool HILO, int TOK, int WMAX, bool DB, bool ENC = false>
static hipError_t go_skinny_w(const GemvArgs &a, hipStream_t s)
{
    const uint32_t B = a.K / 256, ntiles = (a.N + 15) / 16;
    const uint32_t C = (B + WMAX - 1) / WMAX, waves = (B + C - 1) / C;
    const uint32_t cus = device_cu_count(), per = (ntiles + cus - 1) / cus, grid = (ntiles + per - 1) / per;
    if constexpr (!ENC)
        hipLaunchKernelGGL(skinny_encode_kernel<HILO>, dim3(B, TOK), dim3(256), 0, s, a.x, a.M, a.K, (uint8_t *)a.ws, (uint32_t)TOK);
    if (per == 1) return go_skinny_t<Q, HILO, TOK, 1, WMAX, DB, ENC>(a, waves, ntiles, grid, s);
    constexpr bool few = DB && (TOK == 2 || Q::MINS);
    if (per == 2 || few) return go_skinny_t<Q, HILO, TOK, 2, WMAX, DB, ENC>(a, waves, ntiles, grid, s);
    return go_skinny_t<Q, HILO, TOK, few ? 2 : 4, WMAX, DB, ENC>(a, waves, ntiles, grid, s);
}

bool skinny_supported(const GemvArgs &a)
{
    if (a.type != T_Q4_K && a.type != T_Q5_K && a.type != T_Q6_K) return false;
    if (a.M < 1 || a.M > 32 || a.K % 256 || a.K == 0) return false;   // 1: the last of a longer run of rows
    if (a.K > (1u << 16)) return false;   // 32-bit workspace offsets, with room
    if (!a.ws || a.ws_bytes < sk_ws_bytes(2, a.K / 256)) return false;
    return a.w_bytes + RRR_READ_SLACK < SK_OOB;
}

// Waves a workgroup: one a column to 12 columns, and to 16 with one A tile (16384 x
// 4096 at 8 rows Q4_K 15.8 us against 20.6 with two columns a wave, Q6_K 20.1
// against 21.8; 4096 x 4096 8.7 against 9.7); beyond, up to 12 (168 registers a
// lane; 16 waves would leave 128, and two columns' operands of one A tile spill),
// 8 where two columns' operands of two A tiles are held.
// To 8 columns and 8 rows the waves build their own operands: the pass costs a
// launch, the building in every wave a chain of ~600 instructions that waits on
// x (5 rows, 1024 to 5632 weight rows, K = 1024 4.2 to 4.9 us against 5.5 to 6.4 with the
// pass, 2048 5.8 to 7.0 against 6.3 to 7.5, 2560 7.3 to 8.9 against 6.9 to 8.5).
template <class Q, bool HILO, int TOK>
static hipError_t go_skinny(const GemvArgs &a, hipStream_t s)
{
    if constexpr (TOK == 1) {
        if (a.K <= 8 * 256) return go_skinny_w<Q, HILO, TOK, 8, false, true>(a, s);
        if (a.K > 12 * 256 && a.K <= 16 * 256) return go_skinny_w<Q, HILO, TOK, 16, false>(a, s);
    }
    if (a.K <= 12 * 256) return go_skinny_w<Q, HILO, TOK, 12, false>(a, s);
    return go_skinny_w<Q, HILO, TOK, TOK == 1 ? 12 : 8, true>(a, s);
}

template <class Q>
static hipError_t go_skinny_m(const GemvArgs &a, hipStream_t s)
{
    if (a.M <= 8) return go_skinny<Q, true, 1>(a, s);
    if (a.M <= 16) return go_skinny<Q, true, 2>(a, s);
    return go_skinny<Q, false, 2>(a, s);
}

hipError_t launch_skinny(const GemvArgs &a, hipStream_t s)
{
    if (!skinny_supported(a)) return hipErrorNotSupported;
    switch (a.type) {
    case T_Q4_K: return go_skinny_m<SkQ4K>(a, s);
    case T_Q5_K: return go_skinny_m<SkQ5K>(a, s);
    default: return go_skinny_m<SkQ6K>(a, s);
    }
}

}  // namespace rrr
