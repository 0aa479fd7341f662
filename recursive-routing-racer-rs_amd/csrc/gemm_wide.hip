// gemm_wide.hip -- the prefill GEMM for long prompts: Y[M][N] = X[M][K] . W[N][K]^T
// (or Y +=) with X in f16 and W first expanded to f16, once per launch of the
// GEMM (once per chunk of rows where a call's rows go through the workspace).
//
// gemm_dq_kernel (gemm.hip) dequantizes a weight tile again for every 256 rows
// of X, with half of its waves, and its 256 x 128 tiles leave the last round of
// the CUs part empty at many shapes.  Here expand_kernel writes W as f16 (the
// same values, one rounding each) into a workspace and gemm_wide_kernel is a
// plain f16 GEMM whose eight waves all multiply, with a choice of tile widths;
// without split K its outputs are gemm_dq_kernel's bit for bit.  Which of the
// two a call takes follows from the two estimates gemm_wide_cost and gemm_plan
// (about 3 % to 10 % off the times measured at 128 to 2,048 rows of nine
// shapes; a near tie goes to gemm_dq_kernel).  Measured, us, expansion
// included (gemm_dq_kernel in brackets): 2,048 rows 16384x3072 198 (216),
// 5120x3072 71 (100), 3072x8192 Q6_K 112 (130); 1,152 rows 145 (189), 53 (66),
// 88 (112); 1,024 rows 112 (109), 50 (50), 78 (78).
//
// Bound: the matrix cores at the clock the power limit leaves (2,048 x 16384 x
// 3072 without its LDS and global traffic still takes 80 % of the time), then
// LDS (192 KB read and 64 KB written per step of a 256 x 256 tile).  The
// expansion runs at 6 TB/s (21 us for 16384x3072).
//
// Expanded layout: blocks of 16 rows x 64 k (2 KB), block (n / 16, k / 64) at
// ((n / 16) * (K / 64) + k / 64) * 2048; inside, row r's 16-byte chunk c (8
// values) sits at slot 8 r + (c ^ ((r / 2) % 8)).  A wave's 16-byte LDS DMA copies
// half a block as it is; the 16 lanes the LDS serves at once (16 rows of one
// chunk) then hit 64 distinct banks.  X's rows take the same form, each lane
// fetching its slot's 16 bytes (a wave load covers 8 rows' 128-byte lines).
#include "device_common.h"
#include "internal.h"

#include <initializer_list>

namespace rrr {

typedef _Float16 f16x8w __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2w __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f16x2w gw_bits(uint32_t v) { return __builtin_bit_cast(f16x2w, v); }
__device__ __forceinline__ uint32_t gw_u32(f16x2w v) { return __builtin_bit_cast(uint32_t, v); }

// ---------------------------------------------------------------------------
// Weights to f16: a wave takes 16 rows of one super-block column (4 blocks of
// the layout, 8 KB back to back); lane l fills slot l of the blocks' upper
// halves (row l / 8) and of their lower halves (row 8 + l / 8), whose chunks are
// c0 and c0 ^ 4: the same 8 quant bytes' place, one nibble and the other.  Same
// arithmetic as gemm_dq_kernel's staging: f16(d * sc), f16(-dmin * mn), one fma
// rounding.
template <uint32_t TYPE>
__global__ __launch_bounds__(256) void expand_kernel(const uint8_t *__restrict__ W, uint32_t K, uint32_t units,
                                                     u32x4 *__restrict__ out)
{
    constexpr uint32_t BS = TYPE == T_Q4_K ? 144 : TYPE == T_Q5_K ? 176 : 210;
    const uint32_t lane = threadIdx.x & 63, u = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (u >= units) return;
    const uint32_t B = K / 256, nb = u / B, b = u - nb * B;   // 16-row group, super-block
    const uint32_t c0 = (lane & 7) ^ (lane >> 4), e = 8 * (c0 & 3);
    u32x4 *o = out + ((uint64_t)nb * B + b) * 512 + lane;
    auto ld2 = [](const uint8_t *q) {
        u32x2 v;
        __builtin_memcpy(&v, q, 8);
        return v;
    };
    auto pair = [](uint32_t v, int i) {   // bytes 2i, 2i + 1 of v under the exponent of 1024
        return gw_bits(__builtin_amdgcn_perm(0x64646464u, v, i ? 0x04030402u : 0x04010400u));
    };
    u32x4 hdr[2];
    u32x2 q[2][4], qh[2][2];
    uint32_t d6[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const uint8_t *p = W + ((uint64_t)(16 * nb + 8 * h + (lane >> 3)) * B + b) * BS;
        if constexpr (TYPE == T_Q6_K) {
            uint16_t d16;
            __builtin_memcpy(&hdr[h], p + 192, 16);
            __builtin_memcpy(&d16, p + 208, 2);
            d6[h] = d16;
#pragma unroll
            for (int i = 0; i < 4; i++) q[h][i] = ld2(p + 32 * i + e);
#pragma unroll
            for (int i = 0; i < 2; i++) qh[h][i] = ld2(p + 128 + 32 * i + e);
        } else {
            __builtin_memcpy(&hdr[h], p, 16);
#pragma unroll
            for (int i = 0; i < 4; i++) q[h][i] = ld2(p + (TYPE == T_Q4_K ? 16 : 48) + 32 * i + e);
            if constexpr (TYPE == T_Q5_K) qh[h][0] = ld2(p + 16 + e);
        }
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const uint32_t nib = (c0 >> 2) ^ h;   // chunk c0 ^ 4 h: 32-element sub-block 2 k + nib of block k
        if constexpr (TYPE == T_Q6_K) {
            const float d = h2f(d6[h]);
            const f16x2w K2 = {(_Float16)1056.0f, (_Float16)1056.0f};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                // elements 64 k + 32 nib + e ..: half g = k / 2, quarter 2 (k % 2) + nib of it
                const int g = k >> 1;
                const u32x2 l = {nib ? q[h][2 * g + 1].x : q[h][2 * g].x, nib ? q[h][2 * g + 1].y : q[h][2 * g].y};
                const uint32_t sb = (hdr[h][k] >> (16 * nib + 4 * ((e >> 4) << 1))) & 0xFFu;   // scale 4 k + 2 nib + e / 16
                const _Float16 A = (_Float16)__fmul_rn(d, (float)(int8_t)sb);
                const f16x2w A2 = {A, A};
                u32x4 r;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const uint32_t v = ((l[i] >> (4 * (k & 1))) & 0x0F0F0F0Fu) |
                                       (((qh[h][g][i] >> (4 * (k & 1) + 2 * nib)) & 0x03030303u) << 4);
                    r[2 * i] = gw_u32(A2 * (pair(v, 0) - K2));
                    r[2 * i + 1] = gw_u32(A2 * (pair(v, 1) - K2));
                }
                o[128 * k + 64 * h] = r;
            }
        } else {
            const float d = h2f(hdr[h].x), dmin = h2f(hdr[h].x >> 16);
            const f16x2w K2 = {(_Float16)1024.0f, (_Float16)1024.0f};
            uint32_t scb[2], mnb[2];
            scale_min_bytes_k4(hdr[h].y, hdr[h].z, hdr[h].w, scb, mnb);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t sh = 16 * (k & 1) + 8 * nib;   // sub-block 2 k + nib
                const _Float16 A = (_Float16)__fmul_rn(d, (float)((scb[k >> 1] >> sh) & 0xFFu));
                const _Float16 Bn = (_Float16)(-__fmul_rn(dmin, (float)((mnb[k >> 1] >> sh) & 0xFFu)));
                const f16x2w A2 = {A, A}, B2 = {Bn, Bn};
                u32x4 r;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    uint32_t v = (q[h][k][i] >> (4 * nib)) & 0x0F0F0F0Fu;
                    if constexpr (TYPE == T_Q5_K) v |= ((qh[h][0][i] >> (2 * k + nib)) & 0x01010101u) << 4;
                    r[2 * i] = gw_u32(__builtin_elementwise_fma(A2, pair(v, 0) - K2, B2));
                    r[2 * i + 1] = gw_u32(__builtin_elementwise_fma(A2, pair(v, 1) - K2, B2));
                }
                o[128 * k + 64 * h] = r;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Workgroup of 512 threads, tile 256 x BN, WM x 8 / WM waves, each UI x UJ 32x32
// tiles of v_mfma_f32_32x32x16_f16.  K steps of 64; NB stages of LDS (the step's
// 256 X rows and BN W rows) form a ring filled by LDS DMA.
//
// A step is four slices of 16 k: the fragments of the next slice are read into
// the second register set between the MFMAs of this one, one read and one DMA
// after each (issued in a row ahead of them: 1,024 x 16384 x 3072 took 107
// instead of 93 us).  Four waves of 128 x 128 read a quarter less LDS but run
// one to a SIMD: 125 us.  Before the last
// slice's MFMAs a wave waits for its own DMA of the next step and for its reads
// of this stage, and passes the step's one barrier: past it the next stage is
// whole, and this one takes the DMA of step s + NB.
template <int BN, int WM, int WN>
struct GwGeom {
    static constexpr int NW = WM * WN;                               // waves
    static constexpr int UI = 8 / WM, UJ = BN / 32 / WN;             // 32x32 tiles a wave
    static constexpr uint32_t STAGE = (256 + BN) * 128;              // bytes of a step in LDS
    static constexpr int NB = 160 * 1024 / (int)STAGE > 4 ? 4 : 160 * 1024 / (int)STAGE;
    static constexpr int UNITS = (256 + BN) / 8;                     // 1 KB DMA loads of a stage
    static constexpr int DPW = (UNITS + NW - 1) / NW, DMIN = UNITS / NW;   // a wave's loads: at most, at least
};

template <int BN, int WM, int WN, bool ACC>
__global__ __launch_bounds__(64 * WM * WN) void gemm_wide_kernel(const uint16_t *X, const uint8_t *Wx, float *Y, uint32_t K,
                                                        uint32_t N, uint32_t M, uint32_t cols, uint32_t tiles_m,
                                                        uint32_t tiles_n, const float *rscale, uint32_t mrows)
{
    using G = GwGeom<BN, WM, WN>;
    constexpr int NB = G::NB, UI = G::UI, UJ = G::UJ, NW = G::NW;
    static_assert(UJ * 32 * WN == BN && NB >= 2, "tile shape");
    extern __shared__ uint8_t gw_lds[];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wm = wave / WN, wn = wave % WN;

    // tile: workgroup id % 8 picks the XCD, whose tiles are consecutive in an
    // order of bands of four row tiles, so its L2 serves 4 x 8 tiles at a time
    const uint32_t T = tiles_m * tiles_n, xcd = blockIdx.x & 7, tq = T >> 3, tr = T & 7;
    const uint32_t o = xcd * tq + min(xcd, tr) + (blockIdx.x >> 3);
    const uint32_t band = o / (4 * tiles_n), in = o - band * 4 * tiles_n, bm = min(4u, tiles_m - 4 * band);
    const uint32_t mt = 4 * band + in % bm, nt = in / bm;
    const uint32_t m0 = mt * 256, n0 = nt * BN;

    const uint32_t steps = K / 64;
    const __amdgpu_buffer_rsrc_t xrs = make_rsrc(X, (uint64_t)M * K * 2);
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(Wx, (uint64_t)cols * K * 2);
    // load u of a stage: 8 rows of X (u < 32) or of W; this wave's are wave + NW i
    uint32_t voff[G::DPW];
#pragma unroll
    for (int i = 0; i < G::DPW; i++) {
        const uint32_t u = wave + NW * i, r = 8 * (u & 1) + (lane >> 3), ch = (lane & 7) ^ ((r >> 1) & 7);
        voff[i] = NW * i < 32 ? ((m0 + 8 * u + (lane >> 3)) * K + 8 * ch) * 2
                             : ((n0 + 8 * u - 256) / 16 * steps) * 2048 + 1024 * (u & 1) + 16 * lane;
    }
    // load i of this wave for step s into its stage (past the last step: out of
    // range, zeros)
    auto dma1 = [&](uint32_t s, uint32_t stage, int i) {
        const bool live = s < steps;
        uint8_t *dst = gw_lds + stage * G::STAGE;
        const uint32_t u = wave + NW * i;
        if (NW * i + NW - 1 >= G::UNITS && u >= G::UNITS) return;   // wave-uniform: no load of the stage
        if (NW * i < 32)
            lds_dma16<0>(xrs, dst + 1024 * u, live ? voff[i] : RRR_OOB, live ? s * 128 : 0u);
        else
            lds_dma16<0>(wrs, dst + 1024 * u, live ? voff[i] : RRR_OOB, live ? s * 2048 : 0u);
    };
    // fragments: lane l takes row l % 32, k 8 (l / 32) .. + 7 of the slice
    const uint32_t fr = lane & 31, fsw = (fr >> 1) & 7;
    struct Frag {
        f16x8w a[UI], b[UJ];
    };
    // part n of a slice's fragments: a0 b0 a1 b1 ... in the order of their first use
    auto frag_part = [&](Frag &f, uint32_t stage, int kq, int n) {
        const uint8_t *p = gw_lds + stage * G::STAGE + fr * 128 + 16 * (((lane >> 5) + 2 * kq) ^ fsw);
        const bool is_a = n < 2 * UI && n % 2 == 0;
        const int k = is_a ? n / 2 : n - (n / 2 + 1 < UI ? n / 2 + 1 : UI);
        if (is_a)
            f.a[k] = *(const f16x8w *)(p + (wm * UI + k) * 4096);
        else
            f.b[k] = *(const f16x8w *)(p + 32768 + (wn * UJ + k) * 4096);
    };
    f32x16 acc[UI][UJ];
#pragma unroll
    for (int i = 0; i < UI; i++)
#pragma unroll
        for (int j = 0; j < UJ; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    // The MFMAs of slice f with, one after each, the reads of the next slice (kq of
    // `stage`) and the loads d0 .. d1 - 1 of step s: issued in a row ahead of the
    // MFMAs they would leave the matrix core idle meanwhile.
    auto slice = [&](const Frag &f, Frag &next, uint32_t stage, int kq, uint32_t s, uint32_t dst, int d0, int d1) {
        int n = 0, d = d0;
#pragma unroll
        for (int j = 0; j < UJ; j++)
#pragma unroll
            for (int i = 0; i < UI; i++) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[i], f.b[j], acc[i][j], 0, 0, 0);
                const bool last = i + 1 == UI && j + 1 == UJ;
                do {
                    if (n < UI + UJ) frag_part(next, stage, kq, n++);
                } while (last && n < UI + UJ);
                do {
                    if (d < d1) dma1(s, dst, d++);
                } while (last && d < d1);
                __builtin_amdgcn_sched_barrier(0);
            }
    };

    constexpr int DH = (G::DPW + 1) / 2;   // a stage's loads go out in two halves
#pragma unroll
    for (int s = 0; s < NB; s++)
#pragma unroll
        for (int i = 0; i < (s + 1 < NB ? G::DPW : DH); i++) dma1(s, s, i);
    wait_vm<(NB - 2) * G::DMIN + (DH < G::DMIN ? DH : G::DMIN)>();
    barrier_lds();
    Frag f0, f1;
#pragma unroll
    for (int n = 0; n < UI + UJ; n++) frag_part(f0, 0, 0, n);
    uint32_t st = 0, pv = NB - 1;
    for (uint32_t s = 0; s < steps; s++) {
        const uint32_t nx = st + 1 == NB ? 0 : st + 1;
        slice(f0, f1, st, 1, s + NB - 1, pv, DH, G::DPW);
        slice(f1, f0, st, 2, 0, 0, 0, 0);
        slice(f0, f1, st, 3, 0, 0, 0, 0);
        wait_vm<(NB - 2) * G::DMIN>();
        barrier_lds();
        slice(f1, f0, nx, 0, s + NB, st, 0, DH);   // past the last step: stale, unused
        pv = st;
        st = nx;
    }
    wait_vm<0>();

    // lane l: output column l % 32 of a tile, rows 8 (r / 4) + 4 (l / 32) + r % 4;
    // per row tile its row scales (powers of two, exact) and (ACC) Y's values are
    // requested at once; rows past mrows and columns past cols are padding,
    // never stored (cols % 32 == 0)
    const __amdgpu_buffer_rsrc_t rsr = make_rsrc(rscale, rscale ? (uint64_t)mrows * 4 : 0u);
    const uint32_t nl = cols - n0;   // columns left from this tile on
#pragma unroll
    for (int i = 0; i < UI; i++) {
        const uint32_t mb = m0 + 32 * (wm * UI + i) + 4 * (lane >> 5);
        float *yb = Y + n0 + wn * UJ * 32 + fr;
        float sc[16], old[UJ][16];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const uint32_t mc = min(mb + 8 * (r >> 2) + (r & 3), mrows - 1);
            sc[r] = u2f(bload4(rsr, 4 * mc));
            if constexpr (ACC) {
#pragma unroll
                for (int j = 0; j < UJ; j++)
                    old[j][r] = Y[(uint64_t)mc * N + min(n0 + (wn * UJ + j) * 32, cols - 32) + fr];
            }
        }
#pragma unroll
        for (int j = 0; j < UJ; j++) {
            if ((wn * UJ + j) * 32 >= nl) continue;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const uint32_t m = mb + 8 * (r >> 2) + (r & 3);
                if (m >= mrows) continue;
                const float v = rscale ? acc[i][j][r] * sc[r] : acc[i][j][r];
                if constexpr (ACC)
                    yb[(uint64_t)m * N + 32 * j] = old[j][r] + v;
                else
                    __builtin_nontemporal_store(v, yb + (uint64_t)m * N + 32 * j);
            }
        }
    }
}

// The GEMM's time in us: rounds of up to 256 tiles over the CUs, each its steps
// of 64 k and its f32 stores.  A step of a full round takes `step`; emptier
// rounds run at a higher clock (a quarter of the tiles: about two thirds of it).
static float gw_cost(uint32_t K, uint32_t N, uint32_t M, uint32_t BN)
{
    const float step = BN == 256 ? 1.68f : BN == 192 ? 1.25f : BN == 160 ? 1.05f : BN == 128 ? 0.9f : BN == 96 ? 0.74f : 0.55f;
    const uint32_t tiles = (M + 255) / 256 * ((N + BN - 1) / BN);
    return gemm_rounds(tiles, K / 64 * step * 0.55f, K / 64 * step * 0.45f, BN * 0.045f);
}
// Columns per expansion into `bytes` of workspace: all, or the smallest equal
// parts (a multiple of 256) that fit.
static uint32_t gw_cols(uint32_t K, uint32_t N, size_t bytes)
{
    for (uint32_t parts = 1; parts <= N / 64; parts++) {
        const uint32_t c = parts == 1 ? N : ((N + parts - 1) / parts + 255) / 256 * 256;
        if ((uint64_t)c * K * 2 <= bytes) return c;
    }
    return 0;
}
static uint32_t gw_best(uint32_t K, uint32_t N, uint32_t M)
{
    uint32_t best = 256;
    for (uint32_t bn : {192u, 160u, 128u, 96u, 64u})
        if (gw_cost(K, N, M, bn) < gw_cost(K, N, M, best)) best = bn;
    return best;
}

uint32_t gemm_wide_tile(uint32_t K, uint32_t N, uint32_t M, size_t wx_bytes)
{
    const uint32_t c = gw_cols(K, N, wx_bytes);
    return c ? gw_best(K, c < N ? c : N, M) : 0;
}

float gemm_wide_cost(uint32_t K, uint32_t N, uint32_t M, size_t wx_bytes)
{
    const uint32_t c = gw_cols(K, N, wx_bytes);
    if (!c) return 1e30f;
    // the expansion: 2.56 bytes of traffic a weight at 6 TB/s; two launches
    float t = 0.0f;
    for (uint32_t n = 0; n < N; n += c) {
        const uint32_t cn = N - n < c ? N - n : c;
        t += (float)cn * K * 4.3e-7f + 9.0f + gw_cost(K, cn, M, gw_best(K, cn, M));
    }
    return t;
}

template <int BN, int WM, int WN>
static hipError_t go_wide(const uint16_t *X, const uint8_t *wx, float *Y, uint32_t K, uint32_t N, uint32_t M,
                          uint32_t cols, const float *rscale, uint32_t mrows, bool acc, hipStream_t s)
{
    using G = GwGeom<BN, WM, WN>;
    constexpr size_t lds = (size_t)G::NB * G::STAGE;
    const uint32_t tm = (mrows + 255) / 256, tn = (cols + BN - 1) / BN;
    if (acc)
        hipLaunchKernelGGL((gemm_wide_kernel<BN, WM, WN, true>), dim3(tm * tn), dim3(64 * G::NW), lds, s, X, wx, Y, K, N,
                           M, cols, tm, tn, rscale, mrows);
    else
        hipLaunchKernelGGL((gemm_wide_kernel<BN, WM, WN, false>), dim3(tm * tn), dim3(64 * G::NW), lds, s, X, wx, Y, K, N,
                           M, cols, tm, tn, rscale, mrows);
    return hipGetLastError();
}

hipError_t launch_gemm_wide(const uint16_t *X, const float *rscale, const uint8_t *W, uint32_t type, float *Y,
                            uint32_t K, uint32_t N, uint32_t M, uint32_t mrows, bool acc, void *wx, size_t wx_bytes,
                            hipStream_t s)
{
    const uint32_t c = gw_cols(K, N, wx_bytes);
    if (!c || N % 64 || K % 256 || mrows == 0 || mrows > M) return hipErrorNotSupported;
    for (uint32_t n = 0; n < N; n += c) {
        const uint32_t cn = N - n < c ? N - n : c, units = cn / 16 * (K / 256);
        const uint8_t *w = W + (uint64_t)n * (K / 256) * block_bytes(type);
        const dim3 grid((units + 3) / 4);
        switch (type) {
        case T_Q4_K: hipLaunchKernelGGL(expand_kernel<T_Q4_K>, grid, dim3(256), 0, s, w, K, units, (u32x4 *)wx); break;
        case T_Q5_K: hipLaunchKernelGGL(expand_kernel<T_Q5_K>, grid, dim3(256), 0, s, w, K, units, (u32x4 *)wx); break;
        case T_Q6_K: hipLaunchKernelGGL(expand_kernel<T_Q6_K>, grid, dim3(256), 0, s, w, K, units, (u32x4 *)wx); break;
        default: return hipErrorNotSupported;
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const uint8_t *x = (const uint8_t *)wx;
        switch (gw_best(K, cn, mrows)) {
        case 256: e = go_wide<256, 4, 2>(X, x, Y + n, K, N, M, cn, rscale, mrows, acc, s); break;
        case 192: e = go_wide<192, 4, 2>(X, x, Y + n, K, N, M, cn, rscale, mrows, acc, s); break;
        case 160: e = go_wide<160, 8, 1>(X, x, Y + n, K, N, M, cn, rscale, mrows, acc, s); break;
        case 128: e = go_wide<128, 4, 2>(X, x, Y + n, K, N, M, cn, rscale, mrows, acc, s); break;
        case 96: e = go_wide<96, 8, 1>(X, x, Y + n, K, N, M, cn, rscale, mrows, acc, s); break;
        default: e = go_wide<64, 4, 2>(X, x, Y + n, K, N, M, cn, rscale, mrows, acc, s); break;
        }
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace rrr
