// attn_flash.hip -- causal prefill attention on the matrix cores, the K/V blocks
// shared by a workgroup's waves (the per-token attention dispatches of
// phi4.rs:1304-1312 for all prompt tokens in one launch).
//
// The query rows of a KV head are flattened, row R = token * heads_per_kv +
// head, so any group size fills the tiles.  Workgroup (g, b) of eight waves
// takes 32 RG of them, RG = 8 / KQ: wave (rg, kq) holds 32 rows and works on
// keys 32 kq .. + 31 of every tile of TK = 32 KQ cache rows; the KQ partial
// results of a row group merge at the end through LDS.  The tiles (K and V,
// f16 as cached) come by LDS DMA, the next one while this one is multiplied,
// one barrier a tile.  The workgroups with the most keys are launched first.
//
// Per tile and wave, v_mfma_f32_32x32x16_f16 throughout (lane l: A row / B
// column l % 32 at k 8 (l / 32) .. + 7; D column l % 32, rows 8 (r / 4) + 4 (l /
// 32) + r % 4 in register r):
//   S^T = K . Q^T   keys x rows; Q^T in f16 hi + lo, held in registers
//   online softmax of the lane's row: 16 of its 32 scores in this lane, the
//                   others in lane l ^ 32; the reference max moves lazily
//   O^T += V^T . P^T dims x rows; P in f16 hi + lo.  A lane's scores are the 8 k
//                   slots of each P^T operand when V^T takes the same keys in
//                   the same order: keys 16 m + 4 (l / 32) + {0..3, 8..11}, two
//                   transposing LDS reads (ds_read_b64_tr_b16: 16 lanes address
//                   4 keys x 16 dims, lane i gets dim i of the 4 keys).
// A wave stops at the tile with its last row's last key and then only loads for
// the others.  Hidden keys in the tiles before enter the product with P = 0, and
// 0 times a V that is not finite would be NaN: such V are taken out of the
// operand, and the rows that do see them get their NaN at the end.
// The hi + lo scalings are those of the short form in attn.hip: Q by a power of
// two per row that puts its largest component in [2^13, 2^14), P (<= 8) by 2^12.
//
// Bound: a wave's chain through a tile (LDS reads, 16 MFMAs, the softmax, 16
// MFMAs: 1.65 us, of which 0.9 us MFMA for the SIMD's two waves).  In prompts,
// 2,000 rows of 8 x 3 heads 76 us (156 with a wave to 16 tokens and keys read by
// every wave), 1,000 rows 33 (57), 512 rows behind 256 22 (31); eight in a row
// from one graph 62, 30 and 20.  Measured and not kept: the next tile's scores
// between the exponentials (registers spill: 81 us), the upper waves' outputs one
// step late (75 to 85 us).
// Precision, to 64 bits, against the per-head form on the same rows: scores of
// standard deviation 1.5 2.4e-7 to 2.9e-7 (3.2e-7 to 3.9e-7), 6 4.7e-7 to
// 5.2e-7 (6.7e-7 to 7.2e-7); near 0, where the f32 sums are all of it, 1.0e-7 to
// 1.4e-7 on tiles of 128 keys (1.1e-7 to 1.5e-7) and 1.25e-7 to 1.35e-7 on tiles
// of 64, whose waves add up twice the keys (1.2e-7).
#include "device_common.h"
#include "internal.h"

namespace rrr {

typedef _Float16 f16x8a __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4a __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2a __attribute__((ext_vector_type(2)));
typedef short i16x4a __attribute__((ext_vector_type(4)));

template <int KQ>
struct AfGeom {
    static constexpr int RG = 8 / KQ;
    static constexpr uint32_t TK = 32 * KQ, TILE = TK * 256;          // keys of a tile, its bytes of K (or V)
    static constexpr uint32_t MERGE = (8 - RG) * 64 * (64 + 2) * 4;   // the other waves' O, max, sum
    static constexpr uint32_t NS = KQ == 2 ? 3 : 2;                   // places of a K and V tile in LDS
    static constexpr uint32_t LDS = 2 * NS * TILE > MERGE ? 2 * NS * TILE : MERGE;
    static constexpr uint32_t BYTES = LDS + (ATT_HD + 1) * 4;         // and the first rows with a V that is not finite
};

__device__ __forceinline__ f16x4a lds_tr4(const uint8_t *p)
{
    i16x4a v = {0, 0, 0, 0};
#if defined(__HIP_DEVICE_COMPILE__)
    v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4a *)p);
#endif
    return __builtin_bit_cast(f16x4a, v);
}

// v of lanes l % 32 + 32 (second) next to lanes l % 32 (first), as lane_pair<32>
__device__ __forceinline__ float other_half_max(float v)
{
    float a, b;
    lane_pair<32>(v, a, b);
    return fmaxf(a, b);
}
__device__ __forceinline__ float other_half_sum(float v)
{
    float a, b;
    lane_pair<32>(v, a, b);
    return a + b;
}

template <int KQ, bool F16OUT>
__global__ __launch_bounds__(512) void attn_flash_kernel(const float *__restrict__ qkv, uint32_t row_stride,
                                                         const uint16_t *kc, const uint16_t *vc, void *__restrict__ out,
                                                         uint32_t rows, uint32_t pos0, uint32_t n_kv, uint32_t hpk,
                                                         uint32_t blocks, float qscale)
{
    using G = AfGeom<KQ>;
    constexpr int RG = G::RG;
    constexpr uint32_t TK = G::TK;
    extern __shared__ uint8_t af_lds[];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t rg = wave % RG, kq = wave / RG, hb = lane >> 5;
    const uint32_t g = blockIdx.x % n_kv, b = blocks - 1 - blockIdx.x / n_kv;   // longest first
    const uint32_t total = rows * hpk, R0 = 32 * (RG * b + rg);
    const uint32_t R = R0 + (lane & 31), Rc = min(R, total - 1), tok = Rc / hpk, head = g * hpk + (Rc - tok * hpk);
    const uint32_t tpos = pos0 + tok;                                           // the row sees keys 0 .. tpos
    const uint32_t wlo = pos0 + min(R0, total - 1) / hpk;                       // the wave's first row's last key
    const uint32_t last = pos0 + min(32 * RG * (b + 1) - 1, total - 1) / hpk;   // the workgroup's last key
    const uint32_t tiles = last / TK + 1, kv_stride = n_kv * ATT_HD;
    const uint32_t whi = pos0 + min(R0 + 31, total - 1) / hpk;                  // the wave's last key
    const uint32_t mine = whi >= 32 * kq ? (whi - 32 * kq) / TK + 1 : 0u;       // the wave's tiles with a key of its rows

    // K and V tiles: load i of a wave covers cache rows 4 (wave + 8 i) .. + 3 of
    // the tile, lane l row l / 16 and the 16-byte chunk whose place is l % 16:
    // K's chunk c of row r at c ^ (r % 16), so 16 rows' reads of one chunk hit
    // 64 banks; V's at c ^ (4 (r % 4) + (r / 4) % 4), so that the transposing
    // reads' 8 rows x 64 bytes do
    const uint64_t cache_bytes = (uint64_t)(last + 1) * kv_stride * 2;
    const __amdgpu_buffer_rsrc_t krs = make_rsrc(kc, cache_bytes), vrs = make_rsrc(vc, cache_bytes);
    auto load_part = [&](uint32_t t, uint32_t place, int i) {   // K (i < KQ) and V loads of tile t
        const int j = i % KQ;
        const uint32_t r = 4 * (wave + 8 * j) + (lane >> 4), row = min(t * TK + r, last), s = lane & 15;   // past it: a repeat
        const uint32_t base = (row * kv_stride + g * ATT_HD) * 2;
        uint8_t *dst = af_lds + place * 2 * G::TILE + 1024 * (wave + 8 * j);
        if (i < KQ)
            lds_dma16<0>(krs, dst, base + 16 * (s ^ (r & 15)), 0);
        else
            lds_dma16<0>(vrs, dst + G::TILE, base + 16 * (s ^ (4 * (r & 3) + ((r >> 2) & 3))), 0);
    };
#pragma unroll
    for (int p = 0; p + 1 < (int)G::NS; p++)
#pragma unroll
        for (int i = 0; i < 2 * KQ; i++) load_part(p, p, i);

    // Q^T operands of the lane's row: dims 16 kk + 8 hb .. + 7
    f16x8a qh[8], ql[8];
    float qs;   // undoes the row's power of two on the scores
    {
        const float *q = qkv + (size_t)tok * row_stride + (size_t)head * ATT_HD + 8 * hb;
        float x[8][8], mx = 0.0f;
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
            const float4 u = *(const float4 *)(q + 16 * kk), v = *(const float4 *)(q + 16 * kk + 4);
            const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 8; i++) {
                x[kk][i] = f[i] * qscale;
                mx = fmaxf(mx, fabsf(x[kk][i]));
            }
        }
        mx = other_half_max(mx);
        int e = 0;
        if (mx > 0.0f && __builtin_isfinite(mx)) (void)frexpf(mx, &e);
        e = max(e, -100);   // 2^(e - 14) stays a normal f32: a masked score times it is -inf
        qs = ldexpf(1.0f, e - 14);
#pragma unroll
        for (int kk = 0; kk < 8; kk++)
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float v = ldexpf(x[kk][i], 14 - e);
                const _Float16 hi = (_Float16)v;
                qh[kk][i] = hi;
                ql[kk][i] = (_Float16)(v - (float)hi);
            }
    }

    f32x16 o[4];
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[dt][r] = 0.0f;
    float m = -__builtin_inff(), ls = 0.0f;   // reference max; this lane's share of the sum, times 2^12

    // LDS addresses: K fragment kk (16 dims) at kaddr ^ 32 kk, V^T fragment (dims
    // 32 dt .., keys 16 k2 + 8 x ..) at (vaddr ^ (64 dt ^ 32 x)) + 256 (16 k2 + 8 x):
    // the swizzled chunk differs from the lane's by constant bits, so one
    // register each does (sixteen would spill)
    const uint32_t krow = 32 * kq + (lane & 31), ti = lane & 15;
    const uint32_t kaddr = krow * 256 + 16 * (hb ^ (krow & 15));
    const uint32_t vaddr = G::TILE + (32 * kq + 4 * hb + (ti >> 2)) * 256 +
                           16 * ((2 * ((lane >> 4) & 1) + ((ti & 3) >> 1)) ^ (4 * (ti >> 2)) ^ hb) + 8 * (ti & 1);
    auto kfrag = [&](uint32_t ka, int kk) { return *(const f16x8a *)(af_lds + (ka ^ (32u * kk))); };
    auto vfrag = [&](uint32_t va, int k2, int dt) {
        f16x4a v[2];
#pragma unroll
        for (int x = 0; x < 2; x++)
            v[x] = lds_tr4(af_lds + (va ^ (64u * dt ^ 32u * x)) + 256 * (16 * k2 + 8 * x));
        return __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7);
    };
    // per dim the first cache row whose V was taken out, then whether any was
    uint32_t *bad = (uint32_t *)(af_lds + G::LDS);
    if (threadIdx.x < ATT_HD + 1) bad[threadIdx.x] = threadIdx.x < ATT_HD ? ~0u : 0u;
    uint32_t st = 0;   // place of tile t
    for (uint32_t t = 0; t < mine; t++) {
        // tile t landed in every wave, and every wave is done with tile t - 1
        wait_vm<(G::NS - 2) * 2 * KQ>();
        barrier_lds();
        const uint32_t c0 = t * TK + 32 * kq, sp = st == 0 ? G::NS - 1 : st - 1;   // sp: place of t - 1 and t + NS - 1
        uint32_t ka = kaddr + st * 2 * G::TILE, va = vaddr + st * 2 * G::TILE;
        asm volatile("" : "+v"(ka), "+v"(va));   // the fragments' addresses are made where they are used
        f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = 0.0f;
        f16x8a kf[8], av[2][4];
#pragma unroll
        for (int kk = 0; kk < 8; kk++) kf[kk] = kfrag(ka, kk);
        __builtin_amdgcn_sched_barrier(0);
        // all V^T reads here, between the MFMAs: ahead of the next DMA, for
        // which the compiler would make a transposing read wait.  The lo products
        // first, in the same sums: they round at their own size, and there is no
        // second sum to add
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[kk], ql[kk], s, 0, 0, 0);
            av[kk >> 2][kk & 3] = vfrag(va, kk >> 2, kk & 3);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int kk = 0; kk < 8; kk++) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[kk], qh[kk], s, 0, 0, 0);
        float bm = -__builtin_inff();
        bool poison = false;   // a V that is not finite, in a tile with hidden keys
        if (c0 + 31 > wlo) {   // the tile holds keys past some of the wave's rows
            f16x8a z = {};
#pragma unroll
            for (int i = 0; i < 8; i++) z = __builtin_elementwise_fma(av[i >> 2][i & 3], f16x8a{}, z);
            const u32x4 zb = __builtin_bit_cast(u32x4, z);
            poison = __builtin_amdgcn_ballot_w64((zb.x | zb.y | zb.z | zb.w) != 0u) != 0;
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (c0 + 8 * (r >> 2) + 4 * hb + (r & 3) > tpos) s[r] = -__builtin_inff();
        }
#pragma unroll
        for (int r = 0; r < 16; r++) bm = fmaxf(bm, s[r]);
        bm = other_half_max(bm) * qs;
        // the reference max moves only when the tile's passes it by more than
        // 3 (P <= 8, P * 2^12 inside f16); rescaling is then a branch that the
        // wave takes for any of its rows.  -inf: no key of the row yet
        const bool upd = bm > m + 3.0f;
        const float mn = upd ? bm : m;
        const float cf = upd && m != -__builtin_inff() ? __builtin_amdgcn_exp2f(m - mn) : 1.0f;
        if (__builtin_amdgcn_ballot_w64(cf != 1.0f)) {
            ls *= cf;
#pragma unroll
            for (int dt = 0; dt < 4; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[dt][r] *= cf;
        }
        m = mn;
        const float off = mn == -__builtin_inff() ? 0.0f : -mn;
        f16x8a pb[2], pl[2];
        float lt = 0.0f;
        // a tile's loads between the exponentials (in a row they hold the wave
        // up); past the last tile they repeat its rows, into a place no one reads
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
            if (r / 2 < 2 * KQ) load_part(t + G::NS - 1, sp, r / 2);
            // 2^12 by a product: in the exponent it would cost its argument, near 0
            // for the weights that count, up to four bits
            const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], qs, off)) * 4096.0f;
            const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r + 1], qs, off)) * 4096.0f;
            lt += p0 + p1;
            // both halves to nearest: what they lose has no sign (cut off, every
            // output came 7e-8 of its size short)
            const f16x2a hi = {(_Float16)p0, (_Float16)p1};
            const f16x2a lo = {(_Float16)(p0 - (float)hi[0]), (_Float16)(p1 - (float)hi[1])};
            pb[r >> 3][r & 7] = hi[0];
            pb[r >> 3][(r & 7) + 1] = hi[1];
            pl[r >> 3][r & 7] = lo[0];
            pl[r >> 3][(r & 7) + 1] = lo[1];
            __builtin_amdgcn_sched_barrier(0);
        }
        ls += lt;
        if (__builtin_expect(poison, 0)) {
#pragma unroll
            for (int k2 = 0; k2 < 2; k2++)
#pragma unroll
                for (int dt = 0; dt < 4; dt++) {
#pragma unroll
                    for (int i = 0; i < 8; i++)
                        if (!__builtin_isfinite((float)av[k2][dt][i])) {
                            atomicMin(bad + 32 * dt + (lane & 31), c0 + 16 * k2 + 8 * (i >> 2) + 4 * hb + (i & 3));
                            bad[ATT_HD] = 1;
                            av[k2][dt][i] = (_Float16)0.0f;
                        }
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
#pragma unroll
        for (int k2 = 0; k2 < 2; k2++) {
#pragma unroll
            for (int dt = 0; dt < 4; dt++) o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[k2][dt], pb[k2], o[dt], 0, 0, 0);
#pragma unroll
            for (int dt = 0; dt < 4; dt++) o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[k2][dt], pl[k2], o[dt], 0, 0, 0);
        }
        st = st + 1 == G::NS ? 0 : st + 1;
    }
    for (uint32_t t = mine; t < tiles; t++) {   // the other waves' tiles
        wait_vm<(G::NS - 2) * 2 * KQ>();
        barrier_lds();
        const uint32_t sp = st == 0 ? G::NS - 1 : st - 1;
#pragma unroll
        for (int i = 0; i < 2 * KQ; i++) load_part(t + G::NS - 1, sp, i);
        st = st + 1 == G::NS ? 0 : st + 1;
    }
    wait_vm<0>();   // the repeated tile's loads, before the LDS is used again
    ls = other_half_sum(ls);

    // the row group's other waves hand their rows to wave kq = 0, which merges
    // them in order; a wave that saw no key of a row holds max -inf, sum 0
    __syncthreads();
    float *mg = (float *)af_lds;
    if (kq > 0) {
        float *p = mg + (size_t)((kq - 1) * RG + rg) * 66 * 64 + lane;
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) p[(16 * dt + r) * 64] = o[dt][r];
        p[64 * 64] = m;
        p[65 * 64] = ls;
    }
    __syncthreads();
    if (kq > 0) return;
#pragma unroll
    for (int k = 1; k < KQ; k++) {
        const float *p = mg + (size_t)((k - 1) * RG + rg) * 66 * 64 + lane;
        const float mk = p[64 * 64], M = fmaxf(m, mk);
        const float a = m == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(m - M);
        const float c = mk == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(mk - M);
        ls = __builtin_fmaf(p[65 * 64], c, ls * a);
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[dt][r] = __builtin_fmaf(p[(16 * dt + r) * 64], c, o[dt][r] * a);
        m = M;
    }
    // registers 4 q .. 4 q + 3 are dims 8 q + 4 hb ..; lanes l and l ^ 32 swap
    // so that one holds 8 dims of quad q, the other of quad q + 1
    const uint32_t any_bad = bad[ATT_HD];
    const float inv = 1.0f / ls;
    const size_t oi = ((size_t)tok * n_kv * hpk + head) * ATT_HD;
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
#pragma unroll
        for (int q = 0; q < 4; q += 2) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(o[dt][4 * q + i] * inv),
                                                                __float_as_uint(o[dt][4 * q + 4 + i] * inv), false, false);
                v[i] = u2f(w[0]);
                v[4 + i] = u2f(w[1]);
            }
            if (R >= total) continue;
            const uint32_t dim = 32 * dt + 8 * (q + hb);
            if (__builtin_expect(any_bad != 0, 0)) {
#pragma unroll
                for (int i = 0; i < 8; i++)
                    if (bad[dim + i] <= tpos) v[i] = __builtin_nanf("");
            }
            const size_t d = oi + dim;
            if constexpr (F16OUT) {
                f16x8a h;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    asm volatile("" : "+v"(v[i]));   // the f32 result, then its rounding (no mixed-precision fold)
                    h[i] = (_Float16)v[i];
                }
                *(f16x8a *)((_Float16 *)out + d) = h;
            } else {
                *(float4 *)((float *)out + d) = make_float4(v[0], v[1], v[2], v[3]);
                *(float4 *)((float *)out + d + 4) = make_float4(v[4], v[5], v[6], v[7]);
            }
        }
}

template <int KQ>
static hipError_t go_flash(const float *qkv, uint32_t row_stride, uint32_t rows, const uint16_t *kc, const uint16_t *vc,
                           void *out, bool out_f16, uint32_t pos0, uint32_t n_kv, uint32_t hpk, float qscale, hipStream_t s)
{
    using G = AfGeom<KQ>;
    const uint32_t blocks = (rows * hpk + 32 * G::RG - 1) / (32 * G::RG);
    if (out_f16)
        hipLaunchKernelGGL((attn_flash_kernel<KQ, true>), dim3(blocks * n_kv), dim3(512), G::BYTES, s, qkv, row_stride, kc,
                           vc, out, rows, pos0, n_kv, hpk, blocks, qscale);
    else
        hipLaunchKernelGGL((attn_flash_kernel<KQ, false>), dim3(blocks * n_kv), dim3(512), G::BYTES, s, qkv, row_stride, kc,
                           vc, out, rows, pos0, n_kv, hpk, blocks, qscale);
    return hipGetLastError();
}

hipError_t launch_attn_flash(const float *qkv, uint32_t row_stride, uint32_t rows, const uint16_t *kc,
                             const uint16_t *vc, void *out, bool out_f16, uint32_t pos0, uint32_t n_kv, uint32_t hpk,
                             float qscale, uint32_t kq, hipStream_t s)
{
    switch (kq) {
    case 2: return go_flash<2>(qkv, row_stride, rows, kc, vc, out, out_f16, pos0, n_kv, hpk, qscale, s);
    case 4: return go_flash<4>(qkv, row_stride, rows, kc, vc, out, out_f16, pos0, n_kv, hpk, qscale, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace rrr
