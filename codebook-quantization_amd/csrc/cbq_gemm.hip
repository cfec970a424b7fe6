// Batched-token GEMM over a compressed matrix on the bf16 matrix cores
// (gfx950): decode to MFMA fragments once, then multiply fragments.
//
// out[t, m] = sum_k x[t, k] * W[m, k] for the batched calls of ck_linear_f32 /
// ck_linear_bf16 (rocm/compressed_kernel.h:52-73) that bring a workspace.
// Two launches per slab of rows (three when K is split):
//   1. frag_prep_kernel: x and a slab of W are written in fragment order,
//      1 KiB per 16 rows x 32 columns (lane l's 16 bytes: row l % 16, columns
//      8 (l / 16) .. +7), bf16.  fp32 x becomes three bf16 parts whose sum is
//      x exactly (cbq_split3's split), bf16 x one.  A codebook that holds
//      bf16 numbers only (every lossless one) gives W one part; other fp32
//      codebooks give it three (fp32 x, exact) or two (bf16 x, hi + lo).
//   2. frag_gemm_kernel: a plain bf16 GEMM over the fragments, fp32
//      accumulation: the sum runs over (W part, column group, x part); fp32
//      x gives fp32 outputs, bf16 x bf16.
//   3. frag_reduce_kernel adds the split-K partials in split order.
// Products of fp32 x with bf16 weights are exact (24-bit significands as
// 8 + 8 + 8 bits); with other weights the sum of the six largest of the nine
// part products, short of the whole by less than 2^-22.  From K = 256 on the
// folded sums more than make up for that; rel-L2 against 64 bits, this /
// exact products in the fp32 kernel's one chain: K = 32 1.3e-7 / 1.0e-7, 128
// 2.0e-7 / 2.0e-7, 256 2.0e-7 / 2.8e-7, 1024 2.1e-7 / 2.9e-7, 12288 2.3e-7 /
// 5.0e-7 (of one sign throughout: 1.2e-7 / 0.8e-7, 1.6e-7 / 1.6e-7, 1.2e-7 /
// 2.3e-7, 0.8e-7 / 1.2e-7, 0.8e-7 / 1.2e-7, with a mean of -5e-8).  Below,
// such a codebook is multiplied in fp32.  x's lower parts go down to 2^-133:
// of |x| under 2^-110 an absolute 2^-133 may be lost.
//
// Why decode first: a fused kernel gathers every weight again for each 512
// tokens, and on this chip the decode's VALU and LDS work adds to the MFMA
// time instead of running under it.  The transient fragments are bounded (a
// slab of kSlabBytes, or of 256 rows where those are more), mostly stay in the
// 256 MiB last-level cache (12288 x 4096 in one part: 96 MiB), and make both
// GEMM operands plain 1 KiB global -> LDS copies.
#include "cbq_device.h"

#include <algorithm>

// Estimated time of the fused bf16 kernel with its workspace (cbq_prefill.hip).
float cbq_prefill_us(int T, int M, int K);

namespace {

constexpr int kGBlock = 512;                   // GEMM: 8 waves, two per SIMD
constexpr int kGWaves = kGBlock / CBQ_WAVE;
constexpr int kPBlock = 256;                   // prep: 4 waves
constexpr int kPrepBlocks = 5;                 // prep blocks per CU (13 bits: 30 KiB of LDS each;
                                               // at 14, 47 KiB, three of them run at once)
constexpr int kPrepGroups = 8;                 // column groups (of 32) per W prep tile
constexpr size_t kFrag = 1024;                 // bytes of one fragment
constexpr size_t kSlabBytes = (size_t)384 << 20;
// fp32 x: the accumulators are added to totals and cleared every 4, 8 or 16
// column groups (fold_groups).  An MFMA rounds its accumulator; one chain of
// 3 K / 32 roundings at the magnitude of the whole sum left rel-L2 6.2e-7 at
// K = 4096 and 1.2e-6 at 12288 against 64 bits (the fp32 matrix cores: 4.1e-7
// and 7.0e-7 at 512 tokens).  With a fold of f groups of n the variance goes
// as 3 f / 2 (the chains) + n / (2 f) (the totals), least at f = sqrt(n / 3):
// 1.8e-7 at K = 2048, 2.5e-7 at 12288, for one addition per accumulator and
// 3 f MFMAs (T = 512, 4096 x 12288: 130 -> 142 us at f = 16).
int fold_groups(int n) { return n < 96 ? 4 : n < 400 ? 8 : 16; }
constexpr int kSixMinK = 256;                  // K of fp32 x times three-part weights
constexpr int kHeader = 256;                   // workspace header: the W part count

typedef unsigned short g_u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack2(uint32_t lo, uint32_t hi)
{
    g_u16x2 p;
    p.x = (unsigned short)lo;
    p.y = (unsigned short)hi;
    return __builtin_bit_cast(uint32_t, p);
}

// ---- prep ---------------------------------------------------------------------

// fp32 -> the three bf16 parts of cbq_split3 (truncations, so no part of a
// finite value overflows), packed two columns to a dword.  A non-finite x
// keeps its value in the first part (a NaN stays a NaN) and zeros in the
// others.
__device__ __forceinline__ void split3_finite(const float (&v)[8], cbq_u32x4 &h, cbq_u32x4 &m,
                                              cbq_u32x4 &l)
{
    cbq_split3(v, h, m, l);
    bool odd = false;
#pragma unroll
    for (int e = 0; e < 8; e++)
        odd |= (__float_as_uint(v[e]) & 0x7f800000u) == 0x7f800000u;
    if (odd) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const uint32_t u = __float_as_uint(v[e]);
            if ((u & 0x7f800000u) != 0x7f800000u) continue;
            const uint32_t hb = (u >> 16) | ((u & 0x7fffffu) ? 0x40u : 0u);
            const uint32_t keep = (e & 1) ? 0x0000ffffu : 0xffff0000u;
            h[e >> 1] = (h[e >> 1] & keep) | (hb << ((e & 1) * 16));
            m[e >> 1] &= keep;
            l[e >> 1] &= keep;
        }
    }
}

// x [T][K] -> fragments [T / 16][G][NP], one wave per (token block, group):
// lane l reads row l % 16, columns 8 (l / 16) .. +7 of the group (16 rows x
// 64 or 128 contiguous bytes) and writes its 16 bytes of each part; rows >= T
// are zero.
template <int NP>
__device__ __forceinline__ void prep_x(const void *__restrict__ x, uint8_t *__restrict__ xf, int T,
                                       int K, int64_t unit, int64_t units, int64_t stride)
{
    const int G = K >> 5, lane = threadIdx.x & (CBQ_WAVE - 1);
#pragma unroll 1
    for (; unit < units; unit += stride) {
        const int tb = (int)(unit / G), g = (int)(unit - (int64_t)tb * G);
        const int t = tb * 16 + (lane & 15);
        const size_t at = (size_t)t * K + (size_t)g * 32 + (lane >> 4) * 8;
        uint8_t *dst = xf + (size_t)unit * NP * kFrag + lane * 16;
        if constexpr (NP == 1) {
            cbq_u32x4 v = {0u, 0u, 0u, 0u};
            if (t < T) v = *(const cbq_u32x4 *)((const uint16_t *)x + at);
            *(cbq_u32x4 *)dst = v;
        } else {
            float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (t < T) {
                const cbq_f32x4 a = *(const cbq_f32x4 *)((const float *)x + at);
                const cbq_f32x4 b = *(const cbq_f32x4 *)((const float *)x + at + 4);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[e] = a[e];
                    v[4 + e] = b[e];
                }
            }
            cbq_u32x4 h, m, l;
            split3_finite(v, h, m, l);
            *(cbq_u32x4 *)dst = h;
            *(cbq_u32x4 *)(dst + kFrag) = m;
            *(cbq_u32x4 *)(dst + 2 * kFrag) = l;
        }
    }
}

// Part p of codebook value v as bf16 bits.  NW = 3: the exact truncation
// split (non-finite values whole in part 0); a zero lower part of a nonzero
// value is the smallest normal number of its sign instead, so that an
// infinite x times it keeps its sign rather than turning into a NaN (2^-126
// is below one part in 2^24 of every product that is not itself subnormal).
// NW = 2: hi and lo rounded to nearest, as the fused bf16 kernel has them.
template <int NW> __device__ __forceinline__ uint32_t cb_part(float v, int p)
{
    const uint32_t u = __float_as_uint(v);
    if constexpr (NW == 2) {
        const uint32_t hi = f32_to_bf16(v);
        return p == 0 ? hi : f32_to_bf16(v - __uint_as_float(hi << 16));
    } else {
        if ((u & 0x7f800000u) == 0x7f800000u)
            return p == 0 ? (u >> 16) | ((u & 0x7fffffu) ? 0x40u : 0u) : 0u;
        if (p == 0) return u >> 16;
        const float r = v - __uint_as_float(u & 0xffff0000u);
        const uint32_t ur = __float_as_uint(r);
        uint32_t b = ur >> 16;
        if (p == 2) b = __float_as_uint(r - __uint_as_float(ur & 0xffff0000u)) >> 16;
        if ((b & 0x7fffu) == 0 && (u & 0x7fffffffu)) b = (u >> 31 << 15) | 0x0080u;
        return b;
    }
}

// Row m of a 32-row superblock sits in fragment (m >> 2) & 1 at fragment row
// 4 (m >> 3) + (m & 3): the MFMA's D rows 4 q .. 4 q + 3 of the two
// fragments are then the 8 consecutive features 8 q .. 8 q + 7, so a lane
// stores 16 (bf16) or 32 (fp32) contiguous bytes.
__device__ __forceinline__ int frag_of(int m) { return (m >> 2) & 1; }
__device__ __forceinline__ int frag_row(int m) { return ((m >> 3) << 2) + (m & 3); }

// Fixed-width indices of rows [row0, row0 + M) -> fragments [M / 16][nw][G],
// nw the parts there is room for (1 or NW); a codebook that needs more leaves
// flag 0.
// A tile is 32 rows x 8 groups: the rows' words arrive in 16-byte pieces
// (two rows per wave load), go to LDS with an odd row stride, and thread
// (row, group) unpacks its 32 indices, gathers bf16 values from the LDS
// table (padded to 2^BITS, which is the index clamp) and writes four 16-byte
// pieces, 256 contiguous bytes per fragment and store.  The next tile's words
// are in registers while one is decoded.
template <int BITS, int NW>
__device__ __forceinline__ void prep_w(const uint32_t *__restrict__ words,
                                       const float *__restrict__ cb, int C,
                                       uint8_t *__restrict__ wf, int nw,
                                       int *__restrict__ flag, int row0, int M, int G, int blk,
                                       int nblk, uint16_t *s_tab, uint32_t *s_raw, int *s_flag)
{
    constexpr int NE = (1 << BITS) / kPBlock, NB = NE < 8 ? NE : 8;   // table entries per thread
    static_assert(NE % NB == 0, "whole batches");
    constexpr int RS = kPrepGroups * BITS + 1;             // LDS words per row
    constexpr int kPieces = kPrepGroups * BITS / 4;        // 16-byte pieces per row (<= 32)
    static_assert(kPieces <= 32, "two rows per wave load");
    constexpr int kLoads = 32 / (2 * (kPBlock / CBQ_WAVE));
    const int tid = threadIdx.x, lane = tid & (CBQ_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / CBQ_WAVE);
    if (tid == 0) *s_flag = 0;
    __syncthreads();
    int parts = 1;
    const int nb32 = (M + 31) >> 5, ng = (G + kPrepGroups - 1) / kPrepGroups;
    const int tiles = nb32 * ng;
    const int64_t RW = (int64_t)G * BITS;
#pragma unroll 1
    for (int p = 0; p < parts; p++) {
        // the table of this part; the first pass also finds out how many
        // parts the codebook needs
        int what = 0;
#pragma unroll 1
        for (int e0 = 0; e0 < NE; e0 += NB) {
            float v[NB];
#pragma unroll
            for (int e = 0; e < NB; e++) v[e] = cb[min((e0 + e) * kPBlock + tid, C - 1)];
#pragma unroll
            for (int e = 0; e < NB; e++) {
                const uint32_t u = __float_as_uint(v[e]);
                if (NW == 3 && (u & 0x7f800000u) == 0x7f800000u) what |= 2;
                if (NW == 3 ? (u & 0xffffu) != 0
                            : (cb_part<2>(v[e], 1) & 0x7fffu) != 0) what |= 1;
                s_tab[(e0 + e) * kPBlock + tid] = (uint16_t)cb_part<NW>(v[e], p);
            }
        }
        if (p == 0 && what) atomicOr(s_flag, what);
        __syncthreads();
        if (p == 0) {
            const int f = *s_flag;
            parts = (f & 2) ? 0 : f ? NW : 1;
            if (parts > nw || (NW == 3 && parts > 1 && G < kSixMinK / 32)) parts = 0;
            if (blk == 0 && tid == 0) *flag = parts;
            if (parts == 0) return;                        // the GEMM reads the indices
        }
        // this wave's rows 8 wave + 2 i + (lane >> 5), piece lane & 31
        const int c = lane & 31;
        auto load = [&](int tile, cbq_u32x4 (&r)[kLoads]) {
            const int b = tile / ng, g0 = (tile - b * ng) * kPrepGroups;
#pragma unroll
            for (int i = 0; i < kLoads; i++) {
                const int m = min(b * 32 + wave * 8 + 2 * i + (lane >> 5), M - 1);
                const uint32_t *src = words + (int64_t)(row0 + m) * RW;
                const int64_t w = (int64_t)g0 * BITS + 4 * c;
                if (c < kPieces) {
                    if (w + 4 <= RW) {
                        __builtin_memcpy(&r[i], src + w, 16);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; e++) r[i][e] = src[min(w + e, RW - 1)];
                    }
                }
            }
        };
        cbq_u32x4 r[kLoads];
        int tile = blk;
        if (tile < tiles) load(tile, r);
        for (; tile < tiles; tile += nblk) {
            lds_barrier();                                 // the last tile's words are read
            if (c < kPieces) {
#pragma unroll
                for (int i = 0; i < kLoads; i++) {
                    uint32_t *d = s_raw + (wave * 8 + 2 * i + (lane >> 5)) * RS + 4 * c;
#pragma unroll
                    for (int e = 0; e < 4; e++) d[e] = r[i][e];
                }
            }
            if (tile + nblk < tiles) load(tile + nblk, r);
            lds_barrier();
            const int b = tile / ng, g0 = (tile - b * ng) * kPrepGroups;
            const int row = tid & 31, g = g0 + (tid >> 5);
            uint32_t w[BITS];
#pragma unroll
            for (int i = 0; i < BITS; i++) w[i] = s_raw[row * RS + (tid >> 5) * BITS + i];
            if (g < G) {
                constexpr uint32_t mask2 = ((1u << BITS) - 1u) << 1;
                uint8_t *dst = wf + ((size_t)(b * 2 + frag_of(row)) * nw * G + (size_t)p * G + g) *
                                        kFrag + frag_row(row) * 16;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    uint32_t v[8];
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const int o = (q * 8 + j) * BITS, k = o >> 5, sh = o & 31;
                        uint32_t f2;                       // the index doubled: a byte offset
                        if (sh == 0) f2 = (w[k] << 1) & mask2;
                        else if (sh + BITS <= 32) f2 = (w[k] >> (sh - 1)) & mask2;
                        else f2 = __builtin_amdgcn_alignbit(w[k + 1], w[k], (uint32_t)(sh - 1)) & mask2;
                        v[j] = *(const uint16_t *)((const char *)s_tab + f2);
                    }
                    *(cbq_u32x4 *)(dst + q * 256) =
                        cbq_u32x4{pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]),
                                  pack2(v[6], v[7])};
                }
            }
        }
        __syncthreads();                                   // the table is rewritten next
    }
}

// Blocks [0, nxb) write x's fragments (the first slab's launch only), the
// rest W's.
template <int BITS, int NP>
__global__ __launch_bounds__(kPBlock, 4) void frag_prep_kernel(
    const void *__restrict__ x, uint8_t *__restrict__ xf, int T, int K, int nxb,
    const uint32_t *__restrict__ words, const float *__restrict__ cb, int C,
    uint8_t *__restrict__ wf, int nw, int *__restrict__ flag, int row0, int M)
{
    constexpr int NW = NP == 3 ? 3 : 2;
    __shared__ __attribute__((aligned(64))) uint16_t s_tab[1 << BITS];
    __shared__ uint32_t s_raw[32 * (kPrepGroups * BITS + 1)];
    __shared__ int s_flag;
    if ((int)blockIdx.x < nxb) {
        const int64_t units = (int64_t)((T + 15) >> 4) * (K >> 5);
        prep_x<NP>(x, xf, T, K,
                   (int64_t)blockIdx.x * (kPBlock / CBQ_WAVE) + threadIdx.x / CBQ_WAVE, units,
                   (int64_t)nxb * (kPBlock / CBQ_WAVE));
        return;
    }
    prep_w<BITS, NW>(words, cb, C, wf, nw, flag, row0, M, K >> 5, blockIdx.x - nxb,
                     gridDim.x - nxb, s_tab, s_raw, &s_flag);
}

// ---- GEMM ---------------------------------------------------------------------

// One wave's share of a block tile: TB token fragments x MB feature fragments
// (MB even); WT x WM waves; NST LDS stages of one column group.
template <int NP_, int TB_, int MB_, int WT_, int WM_, int NST_> struct GemmCfg {
    static constexpr int NP = NP_, TB = TB_, MB = MB_, WT = WT_, WM = WM_, NST = NST_;
    static constexpr int NW = NP == 3 ? 3 : 2;
    static constexpr int NA = WT * TB, NB = WM * MB;         // fragments of a tile
    static constexpr int TT = NA * 16, TM = NB * 16;
    static_assert(WT * WM == kGWaves && MB % 2 == 0, "8 waves, feature pairs");
};

// The K loop's stages for WP parts of W: one column group, all its parts.
template <class C, int WP> struct GemmStage {
    static constexpr int NST = WP == 1 ? C::NST : 2;
    // stages between a buffer's last read and its reuse: 1 leaves reads in
    // flight over the barrier, at the price of a stage of LDS
    static constexpr int LAG = NST >= 4 ? 1 : 0;
    // LDS reads of the running stage that may be in flight at its barrier:
    // those of its only product, or with several x parts of its last one.
    // LDS answers in order, so the stage before it has been read.
    static constexpr int READS = LAG == 0 ? 0 : C::NP > 1 ? C::TB : C::TB + C::MB;
    static constexpr int PIECES = C::NA * C::NP + C::NB * WP;
    static constexpr int PL = (PIECES + kGWaves - 1) / kGWaves;   // copies per wave and stage
    static constexpr int BYTES = PIECES * (int)kFrag;
    static constexpr int LDS = NST * BYTES;
    // products (W part, x part) of a stage.  Three parts of both: the six
    // largest of the nine; the others are below 2^-22 of the whole.
    static constexpr int NS = C::NP == 1 ? WP : WP == 1 ? 3 : 6;
    static constexpr int wpart(int i) { return NS == 6 ? (i < 3 ? 0 : i < 5 ? 1 : 2) : C::NP == 1 ? i : 0; }
    static constexpr int xpart(int i) { return NS == 6 ? (i < 3 ? i : i < 5 ? i - 3 : 0) : C::NP == 1 ? 0 : i; }
    static_assert(LDS <= 160 * 1024, "LDS");
};

struct GemmArgs {
    const uint8_t *xf;      // [T / 16][G][NP] fragments
    const uint8_t *wf;      // [M / 16][nw][G] fragments of the slab
    const int *flag;        // W parts in use; 0: the slab does not hold W
    void *out;              // out + slab offset, row stride ldo
    float *part;            // split-K partials [S][tiles] in fragment order
    // for flag 0: the caller's x, the slab's first index words, the codebook
    const void *x;
    const uint32_t *words;
    const float *cb;
    int C, bits;
    int T, M, ldo, G, nT, nM, S;
    int nw;                 // W parts the slab has room for
    int fold;               // column groups per chain (even)
};

// One fragment (1 KiB, lane l's 16 bytes at + 16 l) from global memory to LDS
// offset dst (wave-uniform).  Written as asm so that the compiler does not
// order LDS reads behind it: the K loop's own waits do.  M0 holds the LDS
// address; one wait state is needed between its write and the load, and five
// between a VALU write of the address's scalar registers (v_readfirstlane)
// and the load: the compiler does not count them inside inline assembly.
__device__ __forceinline__ void lds_copy_frag(uint32_t dst, const uint8_t *src, uint32_t lane16)
{
    const uint64_t p = (uint64_t)src;              // wave-uniform, in scalar registers
    const uint64_t q = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)p) |
                       (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(p >> 32)) << 32;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2"
                 :: "s"(__builtin_amdgcn_readfirstlane(dst)), "v"(lane16), "s"(q) : "m0");
}

// The wave's copies but the newest N have landed in LDS, and its LDS reads but
// the newest R are done; then the block's barrier: every wave's.
template <int N, int R> __device__ __forceinline__ void stage_barrier()
{
    static_assert(N >= 0 && N < 64 && R >= 0 && R < 16, "counter widths");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(%1)\n\ts_barrier" :: "n"(N), "n"(R) : "memory");
}

__device__ __forceinline__ uint32_t bf16_pair(float a, float b)
{
    return pack2(f32_to_bf16(a), f32_to_bf16(b));
}

// 8 consecutive features of token t
template <bool BF16OUT>
__device__ __forceinline__ void store8(void *out, int64_t ldo, int t, int m, int M,
                                       const float (&v)[8])
{
    if constexpr (BF16OUT) {
        uint16_t *o = (uint16_t *)out + (int64_t)t * ldo + m;
        uint16_t h[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const __bf16 b = (__bf16)v[e];               // v_cvt_pk_bf16_f32, nearest even
            __builtin_memcpy(&h[e], &b, 2);
        }
        if (m + 8 <= M && ((uintptr_t)o & 15) == 0) {
            *(cbq_u32x4 *)o = cbq_u32x4{pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]),
                                        pack2(h[6], h[7])};
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (m + e < M) o[e] = h[e];
        }
    } else {
        float *o = (float *)out + (int64_t)t * ldo + m;
        if (m + 8 <= M && ((uintptr_t)o & 15) == 0) {
            *(cbq_f32x4 *)o = cbq_f32x4{v[0], v[1], v[2], v[3]};
            *(cbq_f32x4 *)(o + 4) = cbq_f32x4{v[4], v[5], v[6], v[7]};
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (m + e < M) o[e] = v[e];
        }
    }
}

// Tile number -> (token tile, feature tile): bands of at most 8 token tiles,
// feature tiles outermost within a band, so the blocks that run together on
// one XCD read few distinct fragments of both operands.
__device__ __forceinline__ void tile_at(int tile, int nT, int nM, int &tt, int &tm)
{
    const int band = tile / (8 * nM), in = tile - band * 8 * nM;
    const int bt = min(8, nT - band * 8);
    tm = in / bt;
    tt = band * 8 + in - tm * bt;
}

// One wave's products without the fragments, on the fp32 matrix cores from the
// index stream: acc as the K loop leaves it.  For codebooks that the bf16
// parts cannot stand for (flag 0: an infinite value times a zero part of x
// would be a NaN), that need more parts than their caller reserved, or that
// are short of kSixMinK columns.  Column group g's step e takes columns 8 q + e of lane
// quarter q, for x and W alike.  Loads go out as the compiler places them and
// every wave decodes its own rows: a path for callers that do not say what
// their codebook holds, not for speed.
template <class Cfg>
__device__ __forceinline__ void fp32_fragments(const GemmArgs &a, uint8_t *lds, int t0, int m0,
                                               int wt, int wm, int g0, int n,
                                               cbq_f32x4 (&acc)[Cfg::TB][Cfg::MB], int lds_bytes)
{
    const int lane = threadIdx.x & (CBQ_WAVE - 1), q = lane >> 4, fr = lane & 15;
    const int bits = a.bits, C = min(a.C, 1 << bits);
    const uint32_t mask = (1u << bits) - 1u;
    constexpr int kSteps = Cfg::NP == 3 ? 4 : 1;     // in flight; the K loop sets the registers
    const float *tab = a.cb;
    if (C * 4 <= lds_bytes) {
        float *const s = (float *)lds;
        for (int i = threadIdx.x; i < C; i += kGBlock) s[i] = a.cb[i];
        lds_barrier();
        tab = s;
    }
    const uint32_t *row[Cfg::MB];
#pragma unroll
    for (int j = 0; j < Cfg::MB; j++) {
        const int f = (m0 >> 4) + wm * Cfg::MB + j;            // fragment -> feature
        const int m = (f >> 1) * 32 + (fr >> 2) * 8 + (f & 1) * 4 + (fr & 3);
        row[j] = a.words + (int64_t)min(m, a.M - 1) * a.G * bits;
    }
#pragma unroll 1
    for (int g = g0; g < g0 + n; g++) {
#pragma unroll kSteps
        for (int e = 0; e < 8; e++) {
            float xv[Cfg::TB], w[Cfg::MB];
            const int o = (q * 8 + e) * bits, k = o >> 5, k1 = min(k + 1, bits - 1);
#pragma unroll
            for (int j = 0; j < Cfg::MB; j++) {
                const uint32_t *const p = row[j] + (int64_t)g * bits;
                const uint32_t ix = __builtin_amdgcn_alignbit(p[k1], p[k], o & 31) & mask;
                w[j] = tab[min((int)ix, C - 1)];
            }
#pragma unroll
            for (int i = 0; i < Cfg::TB; i++) {
                const int t = min(t0 + (wt * Cfg::TB + i) * 16 + fr, a.T - 1);
                const size_t at = ((size_t)t * a.G + g) * 32 + q * 8 + e;
                xv[i] = Cfg::NP == 3 ? ((const float *)a.x)[at]
                                     : bf16_to_f32(((const uint16_t *)a.x)[at]);
            }
#pragma unroll
            for (int i = 0; i < Cfg::TB; i++)
#pragma unroll
                for (int j = 0; j < Cfg::MB; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], xv[i], acc[i][j], 0, 0, 0);
        }
    }
}

template <class Cfg, bool SPLIT>
__global__ __launch_bounds__(kGBlock, 2) void frag_gemm_kernel(GemmArgs a)
{
    constexpr int NP = Cfg::NP, TB = Cfg::TB, MB = Cfg::MB;
    constexpr int kLds1 = GemmStage<Cfg, 1>::LDS, kLdsN = GemmStage<Cfg, Cfg::NW>::LDS;
    constexpr bool FOLD = NP == 3, BF16OUT = NP == 1;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLds1 > kLdsN ? kLds1 : kLdsN];
    const int lane = threadIdx.x & (CBQ_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / CBQ_WAVE);
    const int wt = wave / Cfg::WM, wm = wave % Cfg::WM;

    // blocks go to the XCDs in turn: give each XCD a run of tiles
    const int nb = gridDim.x, xcd = blockIdx.x & 7;
    const int lin = xcd * (nb >> 3) + min(xcd, nb & 7) + (blockIdx.x >> 3);
    const int tiles = a.nT * a.nM;
    const int z = SPLIT ? lin / tiles : 0, tile = lin - z * tiles;
    int tt, tm;
    tile_at(tile, a.nT, a.nM, tt, tm);
    const int t0 = tt * Cfg::TT, m0 = tm * Cfg::TM;
    float *const part = SPLIT ? a.part + ((size_t)z * tiles + tile) * (Cfg::TT * Cfg::TM) : nullptr;

    const int nW = __builtin_amdgcn_readfirstlane(*a.flag);
    // this block's column groups [g0, g1)
    const int per = SPLIT ? (a.G + a.S - 1) / a.S : a.G;
    const int g0 = min(z * per, a.G), n = min(g0 + per, a.G) - g0;

    cbq_f32x4 acc[TB][MB], tot[FOLD ? TB : 1][FOLD ? MB : 1];
#pragma unroll
    for (int i = 0; i < TB; i++)
#pragma unroll
        for (int j = 0; j < MB; j++) {
            acc[i][j] = cbq_f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (FOLD) tot[i][j] = cbq_f32x4{0.f, 0.f, 0.f, 0.f};
        }

    // the K loop over WP parts of W
    auto all = [&](auto WPc) {
        using St = GemmStage<Cfg, decltype(WPc)::value>;
        constexpr int WP = decltype(WPc)::value, NST = St::NST, PL = St::PL, NS = St::NS;
        constexpr int LAG = St::LAG;
        constexpr int STAGE = St::BYTES;
        // This wave's pieces of a stage: piece p goes to LDS offset p KiB,
        // the W fragments first (part by part), then x's.
        const int nTB = (a.T + 15) >> 4, nMB = ((a.M + 31) >> 5) * 2;
        const uint8_t *base[PL];
        uint32_t dst[PL], step[PL];
#pragma unroll
        for (int i = 0; i < PL; i++) {
            int p = wave + i * kGWaves;
            if (p >= St::PIECES) p -= St::PIECES;            // a repeat: same bytes, same place
            dst[i] = (uint32_t)p * (uint32_t)kFrag;
            const int q = p - Cfg::NB * WP;
            step[i] = (uint32_t)kFrag * (q >= 0 ? NP : 1);
            base[i] =
                q >= 0 ? a.xf + ((size_t)min((t0 >> 4) + q % Cfg::NA, nTB - 1) * a.G * NP + q / Cfg::NA) * kFrag
                       : a.wf + ((size_t)min((m0 >> 4) + p % Cfg::NB, nMB - 1) * a.nw + p / Cfg::NB) *
                                    a.G * kFrag;
        }
        const uint32_t lane16 = lane * 16;
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
        // copy i of the next column group into LDS offset buf; past the end
        // the last one is copied again, so every wave keeps as many in flight
        int gi = g0;
        auto copy = [&](uint32_t buf, int i) {
            lds_copy_frag(lds0 + buf + dst[i], base[i] + (uint32_t)gi * step[i], lane16);
        };
        auto advance = [&]() { gi += gi + 1 < g0 + n ? 1 : 0; };
        const uint8_t *const rda = lds + (Cfg::NB * WP + wt * TB) * (int)kFrag + lane16;
        const uint8_t *const rdb = lds + wm * MB * (int)kFrag + lane16;
        cbq_u32x4 fa[2][TB], fb[2][MB];
        auto read_a = [&](uint32_t buf, int p, int i, cbq_u32x4 (&f)[TB]) {
            f[i] = *(const cbq_u32x4 *)(rda + buf + (i + p * Cfg::NA) * (int)kFrag);
        };
        auto read_b = [&](uint32_t buf, int p, int j, cbq_u32x4 (&f)[MB]) {
            f[j] = *(const cbq_u32x4 *)(rdb + buf + (j + p * Cfg::NB) * (int)kFrag);
        };
        uint32_t cur = 0;                                   // LDS offset of the running stage
        uint32_t old = (NST - 1) * STAGE;                   // and of the one before it
        // One stage whose first fragments are in fa[P0] / fb[Q0]: the next
        // product's fragments are read while the current one runs.  Before
        // the last product's MFMAs every wave has waited for its reads of the
        // stage (LAG 0) or of the one before it (LAG 1), so the barrier frees
        // that LDS for the next copies and publishes the next stage.
        // With three x parts the copies into it are spread over that
        // product's MFMAs: a wave that issues them all at once waits in the
        // memory pipeline's queue before its MFMAs (T = 1024, 8192 x 4096:
        // 184 -> 165 us; over the next stage's products too: 168). With one
        // part the stage is a third as long and the earlier copies matter
        // more (T = 333, 4096 x 4096: 51 us against 53 spread).
        auto stage = [&](auto P0, auto Q0) {
            constexpr int p0 = decltype(P0)::value, q0 = decltype(Q0)::value;
#pragma unroll
            for (int i = 0; i < NS; i++) {
                const int k = (p0 + i) & 1, q = (q0 + St::wpart(i)) & 1;
                const bool last = i == NS - 1;
                const bool next_a = last || NP > 1;
                const bool next_b = last || St::wpart(i + 1) != St::wpart(i);
                const int na = next_a ? TB : 0, nb = next_b ? MB : 0;
                const int np = last ? 0 : St::xpart(i + 1), nw = last ? 0 : St::wpart(i + 1);
                cbq_u32x4 (&an)[TB] = fa[NP > 1 ? k ^ 1 : p0 ^ 1];
                cbq_u32x4 (&bn)[MB] = fb[q ^ 1];
                const uint32_t free_buf = LAG ? old : cur;
                if (last) {
                    stage_barrier<(NST - 2 - LAG) * PL, St::READS>();
                    old = cur;
                    cur = cur + STAGE == NST * STAGE ? 0u : cur + STAGE;
                }
                auto read = [&](int r) {
                    if (r < nb) read_b(cur, nw, r, bn);
                    else read_a(cur, np, r - nb, an);
                };
                constexpr int NM = TB * MB;
                if constexpr (NP == 1) {
                    if (last)
#pragma unroll
                        for (int c = 0; c < PL; c++) copy(free_buf, c);
#pragma unroll
                    for (int r = 0; r < nb + na; r++) read(r);
                }
#pragma unroll
                for (int m = 0; m < NM; m++) {
                    if constexpr (NP > 1) {
                        // reads over the first half of the MFMAs, copies over all
#pragma unroll
                        for (int r = m * 2 * (na + nb) / NM;
                             r < (m + 1) * 2 * (na + nb) / NM && r < na + nb; r++)
                            read(r);
                        if (last)
#pragma unroll
                            for (int c = m * PL / NM; c < (m + 1) * PL / NM; c++)
                                copy(free_buf, c);
                    }
                    const int x = m / MB, w = m % MB;
                    acc[x][w] = cbq_mfma_bf16(fb[q][w], fa[NP > 1 ? k : p0][x], acc[x][w]);
                    if constexpr (NP > 1) __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (NP == 1) {
#pragma unroll
                    for (int r = 0; r < na + nb; r++) {
                        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
                    }
                    __builtin_amdgcn_sched_group_barrier(0x008, NM, 0);
                }
                if (last) advance();
            }
        };
        // fragment registers in use at the start of every second stage
        constexpr int P1 = NP > 1 ? NS & 1 : 1, Q1 = WP & 1;
        const std::integral_constant<int, 0> I0{};
        for (int b = 0; b < NST - LAG; b++) {
#pragma unroll
            for (int i = 0; i < PL; i++) copy(b * STAGE, i);
            advance();
        }
        stage_barrier<(NST - 1 - LAG) * PL, 0>();
#pragma unroll
        for (int i = 0; i < TB; i++) read_a(0, 0, i, fa[0]);
#pragma unroll
        for (int j = 0; j < MB; j++) read_b(0, 0, j, fb[0]);
        for (int s = 0; s < n;) {
            const int e = FOLD ? min(n, s + a.fold) : n;
            for (; s + 2 <= e; s += 2) {
                stage(I0, I0);
                stage(std::integral_constant<int, P1>{}, std::integral_constant<int, Q1>{});
            }
            if (s < e) {                                    // an odd last stage
                stage(I0, I0);
                s++;
            }
            if constexpr (FOLD) {
#pragma unroll
                for (int i = 0; i < TB; i++)
#pragma unroll
                    for (int j = 0; j < MB; j++) {
#pragma unroll
                        for (int r = 0; r < 4; r++) tot[i][j][r] += acc[i][j][r];
                        acc[i][j] = cbq_f32x4{0.f, 0.f, 0.f, 0.f};
                    }
            }
        }
        // no copy into LDS may outlive the block
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    if (n > 0 && nW == 1) all(std::integral_constant<int, 1>{});
    else if (n > 0 && nW > 1) all(std::integral_constant<int, Cfg::NW>{});
    if (nW == 0)
        fp32_fragments<Cfg>(a, lds, t0, m0, wt, wm, g0, n, acc, (int)sizeof(lds));
    else if constexpr (FOLD)
#pragma unroll
        for (int i = 0; i < TB; i++)
#pragma unroll
            for (int j = 0; j < MB; j++) acc[i][j] = tot[i][j];

    // acc[i][2 j + f][r]: token 16 (wt TB + i) + lane % 16 of the tile,
    // feature 32 (wm MB / 2 + j) + 8 (lane / 16) + 4 f + r
#pragma unroll
    for (int i = 0; i < TB; i++) {
        const int t = t0 + (wt * TB + i) * 16 + (lane & 15);
#pragma unroll
        for (int j = 0; j < MB / 2; j++) {
            if constexpr (SPLIT) {
                float *o = part + (((wave * TB + i) * (MB / 2) + j) * 2 * 64 + lane) * 4;
                *(cbq_f32x4 *)o = acc[i][2 * j];
                *(cbq_f32x4 *)(o + 256) = acc[i][2 * j + 1];
            } else {
                const int m = m0 + (wm * (MB / 2) + j) * 32 + (lane >> 4) * 8;
                const float v[8] = {acc[i][2 * j][0],     acc[i][2 * j][1],
                                    acc[i][2 * j][2],     acc[i][2 * j][3],
                                    acc[i][2 * j + 1][0], acc[i][2 * j + 1][1],
                                    acc[i][2 * j + 1][2], acc[i][2 * j + 1][3]};
                if (t < a.T && m < a.M) store8<BF16OUT>(a.out, a.ldo, t, m, a.M, v);
            }
        }
    }
}

// The sum of a tile's S partials, in split order; thread = (wave, i, j, lane)
// of frag_gemm_kernel's layout, 8 outputs each.
template <bool BF16OUT>
__global__ __launch_bounds__(256) void frag_reduce_kernel(GemmArgs a, int TB, int MB2, int WM,
                                                          int TT, int TM)
{
    const int tiles = a.nT * a.nM, per = TT * TM / 8;
    const int64_t total = (int64_t)tiles * per;
    for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < total;
         u += (int64_t)gridDim.x * 256) {
        const int tile = (int)(u / per), e = (int)(u - (int64_t)tile * per);
        const int lane = e & 63;
        int q = e >> 6;
        const int j = q % MB2;
        q /= MB2;
        const int i = q % TB, wave = q / TB;
        int tt, tm;
        tile_at(tile, a.nT, a.nM, tt, tm);
        const int t = tt * TT + ((wave / WM) * TB + i) * 16 + (lane & 15);
        const int m = tm * TM + ((wave % WM) * MB2 + j) * 32 + (lane >> 4) * 8;
        if (t >= a.T || m >= a.M) continue;
        const float *p = a.part + (size_t)tile * (TT * TM) + (size_t)(e >> 6) * 512 + lane * 4;
        const size_t zs = (size_t)tiles * (TT * TM);
        cbq_f32x4 lo = *(const cbq_f32x4 *)p, hi = *(const cbq_f32x4 *)(p + 256);
        for (int z = 1; z < a.S; z++) {
            const cbq_f32x4 x = *(const cbq_f32x4 *)(p + z * zs);
            const cbq_f32x4 y = *(const cbq_f32x4 *)(p + z * zs + 256);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                lo[r] += x[r];
                hi[r] += y[r];
            }
        }
        const float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        store8<BF16OUT>(a.out, a.ldo, t, m, a.M, v);
    }
}

// ---- plan and launch ------------------------------------------------------------

// Block tiles (tokens x features), largest first: x parts, TB, MB, WT, WM, stages
using Gemm1a = GemmCfg<1, 8, 4, 2, 4, 4>;      // 256 x 256
using Gemm1b = GemmCfg<1, 4, 4, 4, 2, 5>;      // 256 x 128
using Gemm1c = GemmCfg<1, 4, 2, 2, 4, 4>;      // 128 x 128
using Gemm1d = GemmCfg<1, 2, 2, 2, 4, 4>;      // 64 x 128
using Gemm1e = GemmCfg<1, 4, 6, 4, 2, 5>;      // 256 x 192
using Gemm3a = GemmCfg<3, 4, 4, 4, 2, 2>;      // 256 x 128
using Gemm3b = GemmCfg<3, 4, 4, 2, 4, 4>;      // 128 x 256
using Gemm3c = GemmCfg<3, 4, 2, 2, 4, 4>;      // 128 x 128
using Gemm3d = GemmCfg<3, 2, 4, 2, 4, 4>;      // 64 x 256
using Gemm3e = GemmCfg<3, 2, 2, 2, 4, 4>;      // 64 x 128

struct GemmShape {
    int TT, TM, TB, MB2, WM;
    float step;             // us per column group with every CU busy (one block per CU)
};
template <class C> constexpr GemmShape shape_of(float step)
{
    return {C::TT, C::TM, C::TB, C::MB / 2, C::WM, step};
}
constexpr int kShapes = 5;
// step: a launch of whole rounds at K = 4096 (T = 2048 x M = 8192 for one x
// part, T = 1024 x M = 8192 for three), time / rounds / 128
const GemmShape kShape1[kShapes] = {shape_of<Gemm1a>(0.86f), shape_of<Gemm1b>(0.49f),
                                    shape_of<Gemm1c>(0.26f), shape_of<Gemm1d>(0.19f),
                                    shape_of<Gemm1e>(0.66f)};
const GemmShape kShape3[kShapes] = {shape_of<Gemm3a>(1.36f), shape_of<Gemm3b>(1.25f),
                                    shape_of<Gemm3c>(0.72f), shape_of<Gemm3d>(0.67f),
                                    shape_of<Gemm3e>(0.40f)};

struct GemmPlan {
    int shape, S;
    int rows;               // rows per slab (a multiple of 256, or all M)
    float us;               // estimated time of the GEMM over all slabs
    float chain;            // of that, the column groups' steps
};

template <class C>
int launch_cfg(const GemmArgs &a, hipStream_t st)
{
    const dim3 grid((unsigned)(a.nT * a.nM * a.S));
    if (a.S > 1)
        hipLaunchKernelGGL((frag_gemm_kernel<C, true>), grid, dim3(kGBlock), 0, st, a);
    else
        hipLaunchKernelGGL((frag_gemm_kernel<C, false>), grid, dim3(kGBlock), 0, st, a);
    return cbq_launch_status("frag_gemm_kernel");
}

int launch_gemm(int NP, int shape, GemmArgs a, hipStream_t st)
{
    const GemmShape &s = NP == 3 ? kShape3[shape] : kShape1[shape];
    a.nT = (a.T + s.TT - 1) / s.TT;
    a.nM = (a.M + s.TM - 1) / s.TM;
    int rc = CK_ERR_ARG;
#define CBQ_G(N, I, CFG)                                                                       \
    if (NP == N && shape == I) rc = launch_cfg<CFG>(a, st);
    CBQ_G(1, 0, Gemm1a) CBQ_G(1, 1, Gemm1b) CBQ_G(1, 2, Gemm1c) CBQ_G(1, 3, Gemm1d) CBQ_G(1, 4, Gemm1e)
    CBQ_G(3, 0, Gemm3a) CBQ_G(3, 1, Gemm3b) CBQ_G(3, 2, Gemm3c) CBQ_G(3, 3, Gemm3d) CBQ_G(3, 4, Gemm3e)
#undef CBQ_G
    if (rc || a.S == 1) return rc;
    const int64_t total = (int64_t)a.nT * a.nM * s.TT * s.TM / 8;
    const int blocks = (int)std::min<int64_t>((total + 255) / 256, 8 * cbq_num_cus());
    if (NP == 1)
        hipLaunchKernelGGL(frag_reduce_kernel<true>, dim3(blocks), dim3(256), 0, st, a, s.TB, s.MB2,
                           s.WM, s.TT, s.TM);
    else
        hipLaunchKernelGGL(frag_reduce_kernel<false>, dim3(blocks), dim3(256), 0, st, a, s.TB,
                           s.MB2, s.WM, s.TT, s.TM);
    return cbq_launch_status("frag_reduce_kernel");
}

template <int BITS>
int launch_prep(int NP, const void *x, uint8_t *xf, int T, int K, bool with_x,
                const uint32_t *words, const float *cb, int C, uint8_t *wf, int nw, int *flag,
                int row0, int M, hipStream_t st)
{
    const int cus = cbq_num_cus();
    const int64_t units = (int64_t)((T + 15) >> 4) * (K >> 5);
    const int nxb = with_x ? (int)std::min<int64_t>((units + 3) / 4, kPrepBlocks * cus) : 0;
    const int64_t tiles = (int64_t)((M + 31) >> 5) * ((K / 32 + kPrepGroups - 1) / kPrepGroups);
    const int nwb = (int)std::min<int64_t>(tiles, kPrepBlocks * cus);
    if (NP == 3)
        hipLaunchKernelGGL((frag_prep_kernel<BITS, 3>), dim3(nxb + nwb), dim3(kPBlock), 0, st, x, xf,
                           T, K, nxb, words, cb, C, wf, nw, flag, row0, M);
    else
        hipLaunchKernelGGL((frag_prep_kernel<BITS, 1>), dim3(nxb + nwb), dim3(kPBlock), 0, st, x, xf,
                           T, K, nxb, words, cb, C, wf, nw, flag, row0, M);
    return cbq_launch_status("frag_prep_kernel");
}

size_t round256(size_t n) { return (n + 255) & ~(size_t)255; }
size_t x_bytes(int T, int K, int NP) { return (size_t)((T + 15) >> 4) * (K >> 5) * NP * kFrag; }
size_t w_bytes(int rows, int K, int nw)
{
    return (size_t)((rows + 31) >> 5) * 2 * (K >> 5) * nw * kFrag;
}
// W parts a fixed-width slab has room for: one where the codebook is said to
// hold bf16 numbers only (every lossless one), or a non-finite value (no
// fragments are written then).
int w_parts(int NP, int cb_kind)
{
    if (cb_kind == CBQ_CB_BF16 || (NP == 3 && cb_kind == CBQ_CB_NON_FINITE)) return 1;
    return NP == 3 ? 3 : 2;
}
size_t part_bytes(const GemmPlan &p, int T, int NP)
{
    if (p.S <= 1) return 0;
    const GemmShape &s = NP == 3 ? kShape3[p.shape] : kShape1[p.shape];
    return (size_t)((T + s.TT - 1) / s.TT) * ((p.rows + s.TM - 1) / s.TM) * s.TT * s.TM * p.S *
           sizeof(float);
}

// The tile and K split of least estimated time: rounds of the CUs x (column
// groups of a block x the shape's step + 5 us of prologue and epilogue), plus
// the partials' write and read at about 5 TB/s and 3 us for the extra launch.
// A split holds at least 8 column groups (a shorter chain is all prologue).
GemmPlan gemm_plan(int T, int M, int K, int NP, int nw)
{
    GemmPlan p;
    const size_t row = (size_t)(K >> 5) * nw * kFrag / 16;
    const int fit = (int)std::max<size_t>(256, kSlabBytes / row / 256 * 256);
    const int slabs = (M + fit - 1) / fit;
    p.rows = slabs == 1 ? M : ((M + slabs - 1) / slabs + 255) / 256 * 256;
    p.shape = 0;
    p.S = 1;
    const int G = K >> 5, cus = cbq_num_cus();
    const GemmShape *shapes = NP == 3 ? kShape3 : kShape1;
    float best = 0.f;
    for (int i = 0; i < kShapes; i++) {
        const GemmShape &s = shapes[i];
        const int64_t tiles = (int64_t)((T + s.TT - 1) / s.TT) * ((p.rows + s.TM - 1) / s.TM);
        for (int S = 1; S <= 16 && (S == 1 || G / S >= 8); S++) {
            if (S > 1 && tiles * S > 2 * cus) break;
            const float rounds = (float)((tiles * S + cus - 1) / cus);
            const float chain = rounds * (float)((G + S - 1) / S) * s.step;
            float t = chain + rounds * 5.f;
            if (S > 1) t += 3.f + (float)(tiles * S) * (float)(s.TT * s.TM) * 8.f * 2e-7f;
            if (best == 0.f || t < best) {
                best = t;
                p.shape = i;
                p.S = S;
                p.us = t * slabs;
                p.chain = chain * slabs;
            }
        }
    }
    return p;
}

// Workspace: header (W part count), x fragments, a slab of W fragments, the
// split-K partials.
GemmArgs gemm_args(const GemmPlan &p, int NP, int nw, const void *x, int T, int M, int K,
                   uint8_t *ws)
{
    GemmArgs a;
    uint8_t *const wf = ws + kHeader + round256(x_bytes(T, K, NP));
    a.xf = ws + kHeader;
    a.wf = wf;
    a.flag = (const int *)ws;
    a.out = nullptr;
    a.part = (float *)(wf + round256(w_bytes(p.rows, K, nw)));
    a.x = x;
    a.words = nullptr;
    a.cb = nullptr;
    a.C = a.bits = 0;
    a.T = T;
    a.M = 0;
    a.ldo = M;
    a.G = K >> 5;
    a.S = p.S;
    a.nT = a.nM = 0;
    a.nw = nw;
    a.fold = fold_groups((a.G + p.S - 1) / p.S);
    return a;
}

size_t gemm_ws_bytes(const GemmPlan &p, int NP, int nw, int T, int K)
{
    return kHeader + round256(x_bytes(T, K, NP)) + round256(w_bytes(p.rows, K, nw)) +
           part_bytes(p, T, NP);
}

// out [T][M] = x @ W^T over the slabs of W; BITS-wide indices.
template <int BITS>
int frag_linear(int NP, int nw, const void *x, const uint32_t *words, const float *cb, void *out,
                int T, int M, int K, int C, uint8_t *ws, hipStream_t st)
{
    const GemmPlan p = gemm_plan(T, M, K, NP, nw);
    GemmArgs a = gemm_args(p, NP, nw, x, T, M, K, ws);
    a.cb = cb;
    a.C = C;
    a.bits = BITS;
    for (int r0 = 0; r0 < M; r0 += p.rows) {
        a.M = std::min(p.rows, M - r0);
        a.words = words + (int64_t)r0 * (K >> 5) * BITS;
        a.out = (uint8_t *)out + (size_t)r0 * (NP == 3 ? 4 : 2);
        int rc = launch_prep<BITS>(NP, x, (uint8_t *)a.xf, T, K, r0 == 0, words, cb, C,
                                   (uint8_t *)a.wf, nw, (int *)ws, r0, a.M, st);
        if (!rc) rc = launch_gemm(NP, p.shape, a, st);
        if (rc) return rc;
    }
    return CK_SUCCESS;
}

// x alone (the split format's matrices are decoded by cbq_split.hip)
template <int NP>
__global__ __launch_bounds__(kPBlock) void frag_x_kernel(const void *__restrict__ x,
                                                         uint8_t *__restrict__ xf, int T, int K)
{
    prep_x<NP>(x, xf, T, K, (int64_t)blockIdx.x * (kPBlock / CBQ_WAVE) + threadIdx.x / CBQ_WAVE,
               (int64_t)((T + 15) >> 4) * (K >> 5), (int64_t)gridDim.x * (kPBlock / CBQ_WAVE));
}

// Below 33 tokens of fp32 (64 of bf16; 65 where K % 128 == 0) the few-token kernels of cbq_tiny.hip
// read the weights in place: T = 32 fp32, 12288 x 4096: 52 us against 66 here;
// T = 48: 77 against 68.
bool frag_shape(int T, int M, int K, bool f32)
{
    return T >= (f32 ? 33 : 64) && M > 0 && K > 0 && K % 32 == 0;
}

}  // namespace

// Workspace bytes of the fragment GEMM for fp32 (f32) or bf16 x; 0: the shape
// does not take it.  bf16 x has the fused kernel of cbq_prefill.hip beside
// it, which reads the index stream alone: decoding first pays unless the
// matrix is large against the tokens and K long (T = 512: 4096 x 12288 111
// against 97 us fused, 12288 x 4096 100 / 100, 4096 x 4096 51 / 62; T = 2048,
// 12288 x 4096: 221 / 263), so the smaller estimate is taken: 13-bit indices
// read and fragments written at 4.8 TB/s, two launches, the GEMM's plan.
// Codebooks of other values have two parts of W (T = 512, 4096 x 4096: 82
// against 62 us fused); of unknown kind, 8-bit ones are taken to.
// bits 0: any width the GEMM takes.
size_t cbq_frag_ws_bytes(int T, int M, int K, int bits, bool f32, int cb_kind)
{
    if (!frag_shape(T, M, K, f32) || !(bits == 0 || bits == 8 || (bits >= 10 && bits <= 14)))
        return 0;
    const int NP = f32 ? 3 : 1;
    const int nw = w_parts(NP, cb_kind);
    const GemmPlan p = gemm_plan(T, M, K, NP, nw);
    if (!f32) {
        const bool two = cb_kind == CBQ_CB_UNKNOWN ? bits == 8 : nw == 2;
        const float prep = (float)M * (float)K * (two ? 5.f : 3.6f) / 4.8e6f;
        const float fused = cbq_prefill_us(T, M, K);
        if (fused > 0.f && prep + 6.f + p.us * (two ? 1.9f : 1.f) > fused) return 0;
    }
    return gemm_ws_bytes(p, NP, nw, T, K);
}

// Estimated microseconds of the batched linear over a codebook of other than
// bf16 numbers and fp32 x, all launches: three table passes, three parts of
// every weight written (and, past the last-level cache, read from HBM), half
// as long again a step as with one part.  Fitted to 356 calls (M x K from
// 512 x 2048 to 12288 x 4096 and 5000 x 12288, 33 to 768 tokens, 8 to 13 bits):
// within 15%.
float cbq_frag_six_us(int T, int M, int K, int bits)
{
    const float mw = (float)M * (float)K * 1e-6f;
    const GemmPlan p = gemm_plan(T, M, K, 3, 3);
    return 6.7f + 1.46e-3f * (float)(1 << bits) + mw * (1.5f + 0.058f * (float)(bits - 8)) +
           2.3f * std::max(0.f, mw - 30.f) + 1.55f * p.chain + 0.95f * (p.us - p.chain);
}

// The batched linear over fixed-width indices with a workspace of at least
// cbq_frag_ws_bytes (16-byte aligned); -1: not handled here.
int cbq_frag_linear(const void *x, bool f32, const uint8_t *packed, const float *cb, void *out,
                    int T, int M, int K, int C, int bits, int cb_kind, void *ws,
                    size_t ws_bytes, hipStream_t st)
{
    const size_t need = cbq_frag_ws_bytes(T, M, K, bits, f32, cb_kind);
    if (!need || !ws || ws_bytes < need || (((uintptr_t)ws | (uintptr_t)x) & 15) != 0 ||
        ((uintptr_t)packed & 3) != 0)
        return -1;
#define CBQ_FL(B)                                                                              \
    case B:                                                                                    \
        return frag_linear<B>(f32 ? 3 : 1, w_parts(f32 ? 3 : 1, cb_kind), x,                   \
                              (const uint32_t *)packed, cb, out, T, M, K, C, (uint8_t *)ws, st);
    switch (bits) {
        CBQ_FL(8) CBQ_FL(10) CBQ_FL(11) CBQ_FL(12) CBQ_FL(13) CBQ_FL(14)
    default: return -1;
    }
#undef CBQ_FL
}

// x [T][K] as fragments: fp32 as three parts, bf16 as one.
int cbq_frag_x(const void *x, bool f32, void *xf, int T, int K, hipStream_t st)
{
    const int64_t units = (int64_t)((T + 15) >> 4) * (K >> 5);
    const int blocks = (int)std::min<int64_t>((units + 3) / 4, kPrepBlocks * cbq_num_cus());
    if (f32)
        hipLaunchKernelGGL(frag_x_kernel<3>, dim3(blocks), dim3(kPBlock), 0, st, x, (uint8_t *)xf, T,
                           K);
    else
        hipLaunchKernelGGL(frag_x_kernel<1>, dim3(blocks), dim3(kPBlock), 0, st, x, (uint8_t *)xf, T,
                           K);
    return cbq_launch_status("frag_x_kernel");
}

// ---- split-format matrices -------------------------------------------------------

// cbq_split.hip: rows [row0, row0 + M) of the matrix as fragments
// [M / 16][1][G] at wf, and the part count 1 at flag.
int cbq_split_frags(const cbq_split_matrix *m, int row0, int M, int K, uint8_t *wf, int *flag,
                    hipStream_t st);

static bool split_gemm_shape(int T, int M, int K)
{
    return T >= 1 && M > 0 && K > 0 && K % 1024 == 0 && (int64_t)M * K % 4096 == 0;
}

extern "C" size_t cbq_split_linear_gemm_ws_bytes(int T, int M, int K, int x_bf16)
{
    if (!split_gemm_shape(T, M, K)) return 0;
    const int NP = x_bf16 ? 1 : 3;
    return gemm_ws_bytes(gemm_plan(T, M, K, NP, 1), NP, 1, T, K);
}

extern "C" int cbq_split_linear_gemm(const void *x, int x_bf16, int T, const cbq_split_matrix *m,
                                     void *out, int M, int K, void *ws, size_t ws_bytes,
                                     hipStream_t stream)
{
    if (!x || !m || !out || !ws || !split_gemm_shape(T, M, K) || !m->cwords || !m->row_off ||
        !m->raw || !m->lut || m->n_chunks != (int64_t)M * K / 4096)
        return CK_ERR_ARG;
    if ((((uintptr_t)x | (uintptr_t)ws | (uintptr_t)m->cwords | (uintptr_t)m->raw |
          (uintptr_t)m->lut) & 15) != 0)
        return CK_ERR_ARG;
    if (ws_bytes < cbq_split_linear_gemm_ws_bytes(T, M, K, x_bf16)) return CK_ERR_ARG;
    const int NP = x_bf16 ? 1 : 3;
    const GemmPlan p = gemm_plan(T, M, K, NP, 1);
    GemmArgs a = gemm_args(p, NP, 1, x, T, M, K, (uint8_t *)ws);
    int rc = cbq_frag_x(x, !x_bf16, (void *)a.xf, T, K, stream);
    for (int r0 = 0; r0 < M && !rc; r0 += p.rows) {
        a.M = std::min(p.rows, M - r0);
        a.out = (uint8_t *)out + (size_t)r0 * (NP == 3 ? 4 : 2);
        rc = cbq_split_frags(m, r0, a.M, K, (uint8_t *)a.wf, (int *)ws, stream);
        if (!rc) rc = launch_gemm(NP, p.shape, a, stream);
    }
    return rc;
}
