// Quantised Dense for 3 to 16 activation rows in one launch on the matrix cores (Q4_K, Q8_0, Q4_0, IQ4_NL, Q6_K; K % 256 == 0).
//
// At these batch sizes the weights' bytes bound the work, but the vector ALUs contract at most four rows per reading of W
// (gemv_ks_body.hpp), and the split-K kernels (mmq.hip) need three dependent launches and 32-row tiles.  Here the activations
// live in registers as MFMA operands: a wavefront owns a 512-value slice of K for good (so K = 4096 is the eight wavefronts of
// one workgroup), and 16-row tiles of W stream past it through a wavefront-private ring of two LDS slots filled by DMA.  No
// wavefront waits for another before the sums of up to sixteen tiles meet in LDS, where the workgroup adds the slices and
// applies normalisation, bias, activation, gate and residual.
//
// Activations: x * 2^e (a power of two per row and slice) as the sum of two fp16 numbers, hi = fp16(x), lo = fp16(x - hi), both
// truncated: 20 significant bits, more than the 16-bit fixed point of the GEMV.  With up to 8 rows hi and lo share one 16-column operand
// (columns 4 g + {0, 1}: hi of rows 2 g, 2 g + 1; + {2, 3}: their lo, so that a lane holds both halves of its sums); up to 16
// rows are two such sets against the same converted weights.
//
// Weights become exact fp16 integers (code - offset; Q4_K: times the 6-bit sub-block scale); d, dmin and Q6_K's group scales
// multiply the finished sums of their block in fp32.  v_mfma_f32_16x16x32_f16 with A = activations and B = weights: lane
// (i = lane % 16, kg = lane / 16) holds weight row i and 8 of the 32 values, and its four results belong to weight row i.
//
// What bounds it: a prologue of 5 us (launch, a trip to memory for the activations, some 700 vector instructions per wavefront of
// conversion), during which the 20 MB of the chip's rings fill, then the weights' way from memory, about 5 TB/s.  Q4_K at 8 rows: 4096 x 4096
// 12.3 -> 9.6 us, 4096 -> 14336 18.6 -> 13.9, the gated pair of those 27.2 -> 19.5; Q6_K at 4 rows on a 128256 x 4096 head 166 -> 92 us.
// (Reading the activations 32 bytes per lane, reducing row by row and rounding hi to nearest cost 2 us more per launch.)
//
// More than eight slices are shared out over gridDim.y workgroups; their sums go to memory and the split-K reduction of
// mmq.hip finishes them.
#include "blocks.hpp"
#include "common.hpp"
#include "lds_dma.hpp"

#include <algorithm>
#include <type_traits>

namespace gq {

namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

constexpr int kSlice = 512;        // values of K per wavefront
constexpr int kMaxWaves = 8;
constexpr int kStageBytes = 8192;  // activations of half a slice on their way into operand order; afterwards the sums of finished tiles
constexpr int kMaxProblems = 4;

__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
__device__ __forceinline__ uint32_t as_u(h2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ uint32_t dup_h(float v) { h2 r; r.x = (_Float16)v; r.y = r.x; return as_u(r); }
__device__ __forceinline__ h2 hconst(float v) { return as_h2(dup_h(v)); }

// What a tile needs per format: kUnit values of K are one DMA unit, a row's share of it kChunks 16-byte chunks (an odd count:
// the 16 rows of a tile then start in 16 different groups of four LDS banks), of which kLive are read from memory.
template <int T> struct MV;
template <> struct MV<kQ4_K> { static constexpr int kUnit = 512, kChunks = 19, kLive = 18, kBytes = 144; };
template <> struct MV<kQ4_0> { static constexpr int kUnit = 512, kChunks = 19, kLive = 18, kBytes = 144; };
template <> struct MV<kIQ4_NL> { static constexpr int kUnit = 512, kChunks = 19, kLive = 18, kBytes = 144; };
template <> struct MV<kQ8_0> { static constexpr int kUnit = 256, kChunks = 17, kLive = 17, kBytes = 272; };
// (a super-block is 210 bytes: the odd ones of a row start two bytes off a dword boundary and are read from two bytes before)
template <> struct MV<kQ6_K> { static constexpr int kUnit = 256, kChunks = 15, kLive = 14, kBytes = 210; };

template <int T> struct MVG {
    static constexpr int kLoads = (16 * MV<T>::kChunks + 63) / 64;  // DMA instructions per unit
    static constexpr int kSlot = kLoads * 1024;
    static constexpr int kUnits = kSlice / MV<T>::kUnit;           // units per tile
    static constexpr int kRow = MV<T>::kChunks * 16;
    static_assert(kLoads == 4 || kLoads == 5, "the load sequences below are written for four or five instructions");
};

// LDS per wavefront: two slots, the staging area, [8][16] sub-block sums (Q4_K), 8 inverse scales; per workgroup 8 x 16 sums of squares
template <int T, int SETS> struct MVLds {
    static constexpr int kSums = T == kQ4_K ? 8 * 16 * 4 : 0;
    static constexpr int kWave = 2 * MVG<T>::kSlot + kStageBytes + kSums + 64;
    static constexpr int bytes(int waves) { return waves * kWave + kMaxWaves * 16 * 4; }
    static_assert(kMaxWaves * kWave + kMaxWaves * 64 <= 160 * 1024, "LDS");
};

struct MmvArgs {
    const uint8_t *W[kMaxProblems];
    const float *bias[kMaxProblems];
    float *y[kMaxProblems];
    int N[kMaxProblems], act[kMaxProblems], tile0[kMaxProblems], n0[kMaxProblems];
    int count, ntiles, M, K, nslices, ntot;
    const void *X[kMaxProblems];  // apart: every matrix has its own activations and wgs[j] workgroups from wg0[j] on
    int wg0[kMaxProblems], wgs[kMaxProblems], apart;
    const uint8_t *W2;       // gated pair: the second matrix, its bias
    const float *bias2;
    const float *residual;
    const float *gain;       // RMS normalisation (norm != 0); may be null
    float gain_offset, eps, inv_k;
    int norm;
    float *partial, *partial2, *xss;  // gridDim.y > 1: sums [gridDim.y][M][ntot] (per matrix of a pair), sums of squares [gridDim.y][M]
};

// The first loads of a wavefront in one piece: the activations (R rows; a lane's eight values of a row are two groups of four, 256 apart: whole lines per instruction) and the gain, then both
// slots' weight DMAs, then a wait for the activations only (the weights, issued behind them, stay in flight).  Written as one
// block because the compiler does not count the DMAs: its own wait for the activations would be a wait for everything.
#define MV_OA(i) [a##i] "=&v"(ra[i])
#define MV_OB(i) [b##i] "=&v"(rb[i])
#define MV_SO(i) [s##i] "s"(soff[i])
#define MV_XA(i) "buffer_load_dwordx4 %[a" #i "], %[xo], %[xr], %[s" #i "] offen\n\t"
#define MV_XB(i) "buffer_load_dwordx4 %[b" #i "], %[xo], %[xr], %[s" #i "] offen offset:1024\n\t"
#define MV_HA(i) "buffer_load_dwordx2 %[a" #i "], %[xo], %[xr], %[s" #i "] offen\n\t"
#define MV_HB(i) "buffer_load_dwordx2 %[b" #i "], %[xo], %[xr], %[s" #i "] offen offset:512\n\t"
#define MV_GAIN "buffer_load_dwordx4 %[ga], %[go], %[gr], 0 offen\n\tbuffer_load_dwordx4 %[gb], %[go], %[gr], 0 offen offset:1024\n\t"
#define MV_D(slot, j) "s_nop 0\n\tbuffer_load_dwordx4 %[v" #j "], %[r" #slot "], 0 offen lds\n\ts_add_u32 m0, m0, 0x400\n\t"
#define MV_DMA4(slot) "s_mov_b32 m0, %[l" #slot "]\n\t" MV_D(slot, 0) MV_D(slot, 1) MV_D(slot, 2) MV_D(slot, 3)
#define MV_DMA5(slot) MV_DMA4(slot) MV_D(slot, 4)
#define MV_IN [xo] "v"(xo), [go] "v"(go), [xr] "s"(xr), [gr] "s"(gr), [r0] "s"(r0), [r1] "s"(r1), [l0] "s"(l0), [l1] "s"(l1), [v0] "v"(voff[0]), \
        [v1] "v"(voff[1]), [v2] "v"(voff[2]), [v3] "v"(voff[3]), [v4] "v"(voff[4])
#define MV_4(F) F(0), F(1), F(2), F(3)
#define MV_T4(F) F(0) F(1) F(2) F(3)
#define MV_8(F) F(0), F(1), F(2), F(3), F(4), F(5), F(6), F(7)
#define MV_T8(F) F(0) F(1) F(2) F(3) F(4) F(5) F(6) F(7)
#define MV_G [ga] "=&v"(ga), [gb] "=&v"(gb)

template <int L, bool BF, int R, typename XV>
__device__ __forceinline__ void first_loads(XV (&ra)[R], XV (&rb)[R], u4 &ga, u4 &gb, uint32_t xo, uint32_t go, i32x4 xr, i32x4 gr, const uint32_t (&soff)[R],
                                            i32x4 r0, i32x4 r1, uint32_t l0, uint32_t l1, const uint32_t (&voff)[5]) {
#define MV_CASE(dma, wait, T, O)                                                                                                                \
    if constexpr (BF) asm volatile(T(MV_HA) T(MV_HB) MV_GAIN dma(0) dma(1) wait : O(MV_OA), O(MV_OB), MV_G : MV_IN, O(MV_SO) : "memory", "scc");                          \
    else asm volatile(T(MV_XA) T(MV_XB) MV_GAIN dma(0) dma(1) wait : O(MV_OA), O(MV_OB), MV_G : MV_IN, O(MV_SO) : "memory", "scc");
    if constexpr (R == 4 && L == 4) { MV_CASE(MV_DMA4, "s_waitcnt vmcnt(8)", MV_T4, MV_4) }
    else if constexpr (R == 4) { MV_CASE(MV_DMA5, "s_waitcnt vmcnt(10)", MV_T4, MV_4) }
    else if constexpr (L == 4) { MV_CASE(MV_DMA4, "s_waitcnt vmcnt(8)", MV_T8, MV_8) }
    else { MV_CASE(MV_DMA5, "s_waitcnt vmcnt(10)", MV_T8, MV_8) }
}

// |a|, |b|, |c|: the largest (written out: the compiler first canonicalises every operand of its own maximum)
__device__ __forceinline__ float max3_abs(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// v minus the low / high fp16 number of a dword (exact: one mixed-precision multiply-add)
__device__ __forceinline__ float minus_low(float v, uint32_t h) {
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(v));
    return r;
}
__device__ __forceinline__ float minus_high(float v, uint32_t h) {
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(v));
    return r;
}
__device__ __forceinline__ float as_f(uint32_t u) { return __builtin_bit_cast(float, u); }

// Eight products per lane of a step, for every set of eight activation rows.
template <int SETS>
__device__ __forceinline__ void step8(const uint32_t (&x)[SETS][64], int at, const uint32_t (&w)[4], f4 (&c)[SETS]) {
    const u4 wv = {w[0], w[1], w[2], w[3]};
#pragma unroll
    for (int s = 0; s < SETS; s++) {
        const u4 xv = {x[s][at], x[s][at + 1], x[s][at + 2], x[s][at + 3]};
        c[s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, xv), __builtin_bit_cast(h8, wv), c[s], 0, 0, 0);
    }
}
template <int SETS> __device__ __forceinline__ void clear(f4 (&c)[SETS]) {
#pragma unroll
    for (int s = 0; s < SETS; s++) c[s] = f4{0.f, 0.f, 0.f, 0.f};
}
template <int SETS> __device__ __forceinline__ void add_scaled(float d, const f4 (&p)[SETS], f4 (&acc)[SETS]) {
#pragma unroll
    for (int s = 0; s < SETS; s++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[s][r] = fmaf(d, p[s][r], acc[s][r]);
}

// ---- a unit's codes: read from the slot into registers, then contracted ------------------------------------------------
// row: this lane's weight row in the slot; half: only the first 256 values of the slice exist.
template <int T> struct Codes;

// 0x64006400 (1024, 1024) from a register: with two literals the compiler splits (u & mask) | magic into two instructions
__device__ __forceinline__ uint32_t magic_reg() {
    uint32_t m;
    asm("v_mov_b32 %0, 0x64006400" : "=v"(m));
    return m;
}

template <> struct Codes<kQ4_K> {
    u4 hd[2], c[2][2];
    __device__ __forceinline__ void read(const uint8_t *row, int kg, int) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            hd[q] = *reinterpret_cast<const u4 *>(row + 144 * q);
            c[q][0] = *reinterpret_cast<const u4 *>(row + 144 * q + 16 + 32 * kg);
            c[q][1] = *reinterpret_cast<const u4 *>(row + 144 * q + 32 + 32 * kg);
        }
    }
    // lane kg owns the 64-value group kg of every super-block: sub-blocks 2 kg (low nibbles) and 2 kg + 1 (high)
    template <int SETS>
    __device__ __forceinline__ void contract(const uint32_t (&x)[SETS][64], const uint32_t (&xsum)[SETS][4], int kg, int, bool half, f4 (&acc)[SETS]) const {
        const uint32_t magic = magic_reg();
        const uint32_t sel0 = (kg & 1) ? 0x04020402u : 0x04000400u, sel1 = sel0 + 0x00010001u;
        const bool hi = kg >= 2;
        const uint32_t m6 = hi ? 0x0F0F0F0Fu : 0x3F3F3F3Fu, m2 = hi ? 0x30303030u : 0u, sh = hi ? 4u : 0u;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            if (q == 1 && half) continue;
            const uint32_t a = hd[q].y, b = hd[q].z, e = hd[q].w;
            // 6-bit scales and minima of sub-blocks 0 .. 3 (kg < 2) or 4 .. 7 as bytes, without a branch
            const uint32_t sc = ((hi ? e : a) & m6) | ((a >> 2) & m2), mn = (((hi ? e : b) >> sh) & m6) | ((b >> 2) & m2);
            const h2 off = hconst(-1024.f);
            const h2 s0 = as_h2(__builtin_amdgcn_perm(0x64646464u, sc, sel0)) + off, s1 = as_h2(__builtin_amdgcn_perm(0x64646464u, sc, sel1)) + off;
            const h2 m0 = as_h2(__builtin_amdgcn_perm(0x64646464u, mn, sel0)) + off, m1 = as_h2(__builtin_amdgcn_perm(0x64646464u, mn, sel1)) + off;
            const h2 s1h = s1 * hconst(0.0625f);                                  // high nibbles arrive as 1024 + 16 n
            const h2 k0 = s0 * hconst(-1024.f), k1 = s1 * hconst(-64.f);
            f4 p[SETS], p2[SETS];
            clear<SETS>(p);
            clear<SETS>(p2);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                uint32_t wl[4], wh[4];
#pragma unroll
                for (int w = 0; w < 2; w++) {
                    const uint32_t u = c[q][s >> 1][2 * (s & 1) + w], v = u >> 8;
                    wl[2 * w] = as_u(__builtin_elementwise_fma(as_h2((u & 0x000F000Fu) | magic), s0, k0));
                    wl[2 * w + 1] = as_u(__builtin_elementwise_fma(as_h2((v & 0x000F000Fu) | magic), s0, k0));
                    wh[2 * w] = as_u(__builtin_elementwise_fma(as_h2((u & 0x00F000F0u) | magic), s1h, k1));
                    wh[2 * w + 1] = as_u(__builtin_elementwise_fma(as_h2((v & 0x00F000F0u) | magic), s1h, k1));
                }
                step8<SETS>(x, 32 * q + 4 * s, wl, p);
                step8<SETS>(x, 32 * q + 16 + 4 * s, wh, p);
            }
            // the minima against the sub-block sums (two fp16 halves each)
            const u2 mv = {as_u(m0), as_u(m1)};
#pragma unroll
            for (int t = 0; t < SETS; t++) {
                const u2 xv = {xsum[t][2 * q], xsum[t][2 * q + 1]};
                p2[t] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h4, xv), __builtin_bit_cast(h4, mv), p2[t], 0, 0, 0);
            }
            add_scaled<SETS>(half_bits_to_float(hd[q].x & 0xFFFFu), p, acc);
            add_scaled<SETS>(-half_bits_to_float(hd[q].x >> 16), p2, acc);
        }
    }
};

// four signed bytes as fp16 numbers
__device__ __forceinline__ void bytes_to_h(uint32_t u, uint32_t &lo, uint32_t &hi) {
    u ^= 0x80808080u;
    lo = as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + hconst(-1152.f));
    hi = as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + hconst(-1152.f));
}

// 8 bytes at byte offset `at` of a 4-byte-aligned row; at % 4 is 0 or 2 (PAR 0 / 1)
template <int PAR>
__device__ __forceinline__ void window8(const uint8_t *p, uint32_t &a, uint32_t &b) {
    const uint32_t *w = reinterpret_cast<const uint32_t *>(p - 2 * PAR);
    if constexpr (PAR == 0) { a = w[0]; b = w[1]; }
    else { const uint32_t x = w[0], y = w[1], z = w[2]; a = __builtin_amdgcn_alignbyte(y, x, 2); b = __builtin_amdgcn_alignbyte(z, y, 2); }
}

template <> struct Codes<kQ8_0> {
    uint32_t v[8][2], d[8];
    __device__ __forceinline__ void read(const uint8_t *row, int kg, int) {
#pragma unroll
        for (int b = 0; b < 8; b++) {
            if (b & 1) window8<0>(row + 34 * b + 2 + 8 * kg, v[b][0], v[b][1]);
            else window8<1>(row + 34 * b + 2 + 8 * kg, v[b][0], v[b][1]);
            d[b] = *reinterpret_cast<const uint16_t *>(row + 34 * b);
        }
    }
    template <int SETS>
    __device__ __forceinline__ void contract(const uint32_t (&x)[SETS][64], const uint32_t (&)[SETS][4], int, int h, bool, f4 (&acc)[SETS]) const {
#pragma unroll
        for (int b = 0; b < 8; b++) {
            uint32_t w[4];
            bytes_to_h(v[b][0], w[0], w[1]);
            bytes_to_h(v[b][1], w[2], w[3]);
            f4 p[SETS];
            clear<SETS>(p);
            step8<SETS>(x, 32 * h + 4 * b, w, p);
            add_scaled<SETS>(half_bits_to_float(d[b]), p, acc);
        }
    }
};

// lanes kg = 0, 1 take the low nibbles of code bytes 8 kg .. (values 8 kg ..), kg = 2, 3 the high ones (values 16 + 8 (kg - 2) ..)
struct Codes18 {
    uint32_t v[16][2], d[16];
    __device__ __forceinline__ void read(const uint8_t *row, int kg, int) {
#pragma unroll
        for (int b = 0; b < 16; b++) {
            if (b & 1) window8<0>(row + 18 * b + 2 + 8 * (kg & 1), v[b][0], v[b][1]);
            else window8<1>(row + 18 * b + 2 + 8 * (kg & 1), v[b][0], v[b][1]);
            d[b] = *reinterpret_cast<const uint16_t *>(row + 18 * b);
        }
    }
};
template <> struct Codes<kQ4_0> : Codes18 {
    template <int SETS>
    __device__ __forceinline__ void contract(const uint32_t (&x)[SETS][64], const uint32_t (&)[SETS][4], int kg, int, bool half, f4 (&acc)[SETS]) const {
        const uint32_t sh = kg >= 2 ? 4 : 0, magic = magic_reg();
        const h2 off = hconst(-1032.f);
#pragma unroll
        for (int b = 0; b < 16; b++) {
            if (b >= 8 && half) continue;
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t u = v[b][i] >> sh;
                w[2 * i] = as_u(as_h2((u & 0x000F000Fu) | magic) + off);
                w[2 * i + 1] = as_u(as_h2(((u >> 8) & 0x000F000Fu) | magic) + off);
            }
            f4 p[SETS];
            clear<SETS>(p);
            step8<SETS>(x, 4 * b, w, p);
            add_scaled<SETS>(half_bits_to_float(d[b]), p, acc);
        }
    }
};
template <> struct Codes<kIQ4_NL> : Codes18 {
    template <int SETS>
    __device__ __forceinline__ void contract(const uint32_t (&x)[SETS][64], const uint32_t (&)[SETS][4], int kg, int, bool half, f4 (&acc)[SETS]) const {
        const uint32_t sh = kg >= 2 ? 4 : 0;
        // the code book (int8: -127 -104 -83 -65 | -49 -35 -22 -10 | 1 13 25 38 | 53 69 89 113) with its sign bits flipped, four per dword
        const uint32_t t0 = 0xBFAD9881u ^ 0x80808080u, t1 = 0xF6EADDCFu ^ 0x80808080u, t2 = 0x26190D01u ^ 0x80808080u, t3 = 0x71594535u ^ 0x80808080u;
#pragma unroll
        for (int b = 0; b < 16; b++) {
            if (b >= 8 && half) continue;
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t idx = v[b][i] >> sh, low3 = idx & 0x07070707u;
                const uint32_t lo = __builtin_amdgcn_perm(t1, t0, low3), hi = __builtin_amdgcn_perm(t3, t2, low3);
                const uint32_t u = __builtin_amdgcn_perm(hi, lo, 0x03020100u | ((idx & 0x08080808u) >> 1));
                w[2 * i] = as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + hconst(-1152.f));
                w[2 * i + 1] = as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + hconst(-1152.f));
            }
            f4 p[SETS];
            clear<SETS>(p);
            step8<SETS>(x, 4 * b, w, p);
            add_scaled<SETS>(half_bits_to_float(d[b]), p, acc);
        }
    }
};

// One 16-value scale group is one v_mfma_f32_16x16x16_f16 (lane kg: its values 4 kg ..): the product of a scale and a code has 13
// bits, too many to fold the scale into an fp16 operand.
template <> struct Codes<kQ6_K> {
    uint32_t ql[2][2][2], qh[2][2], sc[4], d;  // [half][16-value column pair][quadrants 0 / 1]
    template <int PAR> static __device__ __forceinline__ uint32_t dword(const uint8_t *p) {
        const uint32_t *w = reinterpret_cast<const uint32_t *>(p);
        if constexpr (PAR == 0) return w[0];
        else return __builtin_amdgcn_alignbyte(w[1], w[0], 2);
    }
    template <int PAR> __device__ __forceinline__ void read_par(const uint8_t *row, int kg) {  // (PAR: the super-block starts two bytes into the row)
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int l = 0; l < 2; l++) {
#pragma unroll
                for (int q = 0; q < 2; q++) ql[h][l][q] = dword<PAR>(row + 64 * h + 32 * q + 16 * l + 4 * kg);
                qh[h][l] = dword<PAR>(row + 128 + 32 * h + 16 * l + 4 * kg);
            }
#pragma unroll
        for (int i = 0; i < 4; i++) sc[i] = dword<PAR>(row + 192 + 4 * i);
        d = *reinterpret_cast<const uint16_t *>(row + 208 + 2 * PAR);
    }
    __device__ __forceinline__ void read(const uint8_t *row, int kg, int h) {
        if (h == 0) read_par<0>(row, kg);
        else read_par<1>(row, kg);
    }
    template <int SETS>
    __device__ __forceinline__ void contract(const uint32_t (&x)[SETS][64], const uint32_t (&)[SETS][4], int, int hb, bool, f4 (&acc)[SETS]) const {
        const float df = half_bits_to_float(d);
        const h2 off = hconst(-1056.f);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int l = 0; l < 2; l++) {
                    const uint32_t a = (ql[h][l][q & 1] >> (q >= 2 ? 4 : 0)) & 0x0F0F0F0Fu;
                    const uint32_t b = (q == 3 ? qh[h][l] >> 2 : q == 2 ? qh[h][l] : q == 1 ? qh[h][l] << 2 : qh[h][l] << 4) & 0x30303030u;
                    const uint32_t u = a | b;
                    const u2 wv = {as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + off),
                                   as_u(as_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + off)};
                    const int j = 8 * h + 2 * q + l;
                    f4 p[SETS];
                    clear<SETS>(p);
#pragma unroll
                    for (int s = 0; s < SETS; s++) {
                        const u2 xv = {x[s][32 * hb + 2 * j], x[s][32 * hb + 2 * j + 1]};
                        p[s] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h4, xv), __builtin_bit_cast(h4, wv), p[s], 0, 0, 0);
                    }
                    const uint32_t sw = sc[j >> 2];
                    add_scaled<SETS>(df * ((j & 3) == 0 ? sbyte0(sw) : (j & 3) == 1 ? sbyte1(sw) : (j & 3) == 2 ? sbyte2(sw) : sbyte3(sw)), p, acc);
                    if ((j & 3) == 3) {  // (four groups in flight: left to itself the compiler keeps the results of all sixteen, and spills)
#pragma unroll
                        for (int s = 0; s < SETS; s++) asm volatile("" : "+v"(acc[s]));
                    }
                }
    }
};

// R values per lane (R = 4 or 8) reduced over the wavefront together: swaps of halves and of rows of 16 lanes fold two arrays
// into one per step, so that eight reductions take 18 instructions instead of 80.  The total of array m ends up in lane_of_row(m)
// and the other lanes of its class (row_of_lane).
template <int R> __device__ __forceinline__ constexpr int lane_of_row(int m) { return (m & 1) * 32 + ((m >> 1) & 1) * 16 + (R == 8 ? m >> 2 : 0); }
template <int R> __device__ __forceinline__ int row_of_lane(int lane) { return (lane >> 5) + 2 * ((lane >> 4) & 1) + (R == 8 ? 4 * (lane & 1) : 0); }
template <int R> __device__ __forceinline__ bool row_writer(int lane) { return (lane & 15) < (R == 8 ? 2 : 1); }
template <int R, class Op>
__device__ __forceinline__ float rows_reduce(const float (&a)[R], int lane, Op op) {
    float b[R / 2], c[R / 4];
#pragma unroll
    for (int i = 0; i < R / 2; i++) {
        const auto s = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a[2 * i]), __builtin_bit_cast(uint32_t, a[2 * i + 1]), false, false);
        b[i] = op(__builtin_bit_cast(float, (uint32_t)s[0]), __builtin_bit_cast(float, (uint32_t)s[1]));
    }
#pragma unroll
    for (int i = 0; i < R / 4; i++) {
        const auto s = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, b[2 * i]), __builtin_bit_cast(uint32_t, b[2 * i + 1]), false, false);
        c[i] = op(__builtin_bit_cast(float, (uint32_t)s[0]), __builtin_bit_cast(float, (uint32_t)s[1]));
    }
    auto dpp = [](float v, auto ctrl) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xF, 0xF, true));
    };
    float d = c[0];
    if constexpr (R == 8) {
        const float keep = (lane & 1) ? c[1] : c[0], send = (lane & 1) ? c[0] : c[1];
        d = op(keep, dpp(send, std::integral_constant<int, 0xB1>()));   // the neighbour's share of this lane's array
    } else {
        d = op(d, dpp(d, std::integral_constant<int, 0xB1>()));
    }
    d = op(d, dpp(d, std::integral_constant<int, 0x4E>()));
    d = op(d, dpp(d, std::integral_constant<int, 0x128>()));            // rotations by 8 and 4 within 16 lanes
    return op(d, dpp(d, std::integral_constant<int, 0x124>()));
}

__device__ __forceinline__ void wave_fence() {  // LDS operations of one wavefront execute in order: only the compiler has to keep them so
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// SETS sets of R activation rows (R = 4: half the columns of a set stay empty, and half the conversion undone)
template <int T, bool BF, int SETS, int R>
__global__ __launch_bounds__(512) void mmv_kernel(const void *__restrict__ Xall, const MmvArgs A) {
    typedef MV<T> F;
    typedef MVG<T> G;
    typedef MVLds<T, SETS> L;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15, kg = lane >> 4;
    const int waves = (int)(blockDim.x >> 6);
    const int slice0 = (int)blockIdx.y * waves, live = min(waves, A.nslices - slice0), slice = slice0 + wave;
    // this workgroup's tiles: bx, bx + gx, .. below end
    int gx = (int)gridDim.x, bx = (int)blockIdx.x, end = A.ntiles;
    const void *X = Xall;
    if (A.apart) {
        int wg0 = 0, first = 0;
        X = A.X[0];
        gx = A.wgs[0];
        end = A.tile0[1];
#pragma unroll
        for (int j = 1; j < kMaxProblems; j++) {
            const bool in = j < A.count && (int)blockIdx.x >= A.wg0[j];
            X = in ? A.X[j] : X;
            gx = in ? A.wgs[j] : gx;
            wg0 = in ? A.wg0[j] : wg0;
            first = in ? A.tile0[j] : first;
            end = in ? (j + 1 < kMaxProblems && j + 1 < A.count ? A.tile0[(j + 1) % kMaxProblems] : A.ntiles) : end;
        }
        bx = first + bx - wg0;
    }
    const int dual = A.W2 ? 1 : 0;
    const int nmt = ((end - bx + gx - 1) / gx) << dual;  // matrix tiles of this workgroup (a gated pair's alternate)
    const int64_t row_bytes = (int64_t)(A.K / 256) * F::kBytes;

    uint8_t *const mine = lds + wave * L::kWave;
    uint8_t *const area = mine + 2 * G::kSlot;
    float *const ssq = reinterpret_cast<float *>(lds + waves * L::kWave);
    const uint32_t slot0 = __builtin_amdgcn_readfirstlane((uint32_t)reinterpret_cast<uintptr_t>(mine));

    // unit u of this wavefront: part u % kUnits of matrix tile u / kUnits; past the end an empty buffer (the loads then move nothing)
    const int nunits = nmt * G::kUnits;
    auto unit_rsrc = [&](int u) __attribute__((always_inline)) -> i32x4 {
        const int mt = min(u, nunits - 1) / G::kUnits, h = u % G::kUnits;
        const int tile = bx + (mt >> dual) * gx;
        const uint8_t *W = A.W[0];
        int N = A.N[0], tile0 = 0;
#pragma unroll
        for (int j = 1; j < kMaxProblems; j++) {  // (selects among arguments in registers: an indexed argument is two trips to the scalar cache)
            const bool in = j < A.count && tile >= A.tile0[j];
            W = in ? A.W[j] : W;
            N = in ? A.N[j] : N;
            tile0 = in ? A.tile0[j] : tile0;
        }
        if (dual && (mt & 1)) W = A.W2;
        const int64_t row0 = (int64_t)(tile - tile0) * 16;
        // (an odd Q6_K super-block is read from the dword its first two bytes share with the one before)
        const int64_t at = row0 * row_bytes + (int64_t)slice * (2 * F::kBytes) + (G::kUnits == 2 ? h * (F::kBytes - (T == kQ6_K ? 2 : 0)) : 0);
        return make_rsrc(W + at, u < nunits ? (uint64_t)((int64_t)N * row_bytes - at) : 0);
    };
    uint32_t voff[5];
#pragma unroll
    for (int l = 0; l < 5; l++) {
        const int c = min(lane + 64 * l, 16 * F::kChunks - 1);
        voff[l] = (uint32_t)(c / F::kChunks) * (uint32_t)row_bytes + (uint32_t)min(c % F::kChunks, F::kLive - 1) * 16u;
    }
    auto fetch = [&](int u) __attribute__((always_inline)) {
        const i32x4 r = unit_rsrc(u);
#pragma unroll
        for (int l = 0; l < G::kLoads; l++) dma16(slot0 + (uint32_t)((u & 1) * G::kSlot + l * 1024), r, voff[l], 0);
    };

    const bool half = slice == A.nslices - 1 && (A.K % kSlice) != 0;  // the last slice holds 256 values only
    uint32_t x[SETS][64], xsum[SETS][4];
    float inv[SETS][2];
    if (wave < live) {
        constexpr int XB = BF ? 2 : 4;
        typedef std::conditional_t<BF, u2, u4> XV;
        const uint32_t k = (uint32_t)slice * kSlice + (uint32_t)lane * 4u;  // (a slice's second half that lies past the row: other rows' values or zeros, cleared below)
        XV ra[R], rb[R];
        u4 ga, gb;
        uint32_t soff[R];
#pragma unroll
        for (int m = 0; m < R; m++) soff[m] = __builtin_amdgcn_readfirstlane((uint32_t)min(m, A.M - 1) * (uint32_t)(A.K * XB));  // rows past the last re-read it
        first_loads<G::kLoads, BF, R>(ra, rb, ga, gb, k * XB, k * 4u, make_rsrc(X, (uint64_t)A.M * (uint64_t)A.K * XB),
                                      make_rsrc(A.gain, A.gain ? (uint64_t)A.K * 4 : 0), soff, unit_rsrc(0), unit_rsrc(1), slot0,
                                      slot0 + (uint32_t)G::kSlot, voff);
        float gl[8];
#pragma unroll
        for (int e = 0; e < 8; e++) gl[e] = A.gain ? as_f(e < 4 ? ga[e & 3] : gb[e & 3]) + A.gain_offset : 1.f;
        uint32_t *const sums = reinterpret_cast<uint32_t *>(area + kStageBytes);
        float *const invs = reinterpret_cast<float *>(area + kStageBytes + L::kSums);
#pragma unroll
        for (int s = 0; s < SETS; s++) {
            if (s > 0) {
#pragma unroll
                for (int m = 0; m < R; m++) {
                    const uint8_t *xp = static_cast<const uint8_t *>(X) + ((int64_t)min(R * s + m, A.M - 1) * A.K + k) * XB;
                    ra[m] = *reinterpret_cast<const XV *>(xp);
                    rb[m] = *reinterpret_cast<const XV *>(xp + (half ? 0 : 256 * XB));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            float v[R][8];
#pragma unroll
            for (int m = 0; m < R; m++)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    if constexpr (BF) {
                        const uint32_t w = e < 4 ? ra[m][(e & 3) >> 1] : rb[m][(e & 3) >> 1];
                        v[m][e] = as_f((e & 1) ? w & 0xFFFF0000u : w << 16);
                    } else {
                        v[m][e] = as_f(e < 4 ? ra[m][e & 3] : rb[m][e & 3]);
                    }
                }
            if (half) {  // (rows past the last need no clearing: nothing reads their columns)
#pragma unroll
                for (int m = 0; m < R; m++)
#pragma unroll
                    for (int e = 4; e < 8; e++) v[m][e] = 0.f;
            }
            const int mine_row = row_of_lane<R>(lane);
            if (A.norm) {
                float t[R];
#pragma unroll
                for (int m = 0; m < R; m++) {
                    t[m] = v[m][0] * v[m][0];
#pragma unroll
                    for (int e = 1; e < 8; e++) t[m] = fmaf(v[m][e], v[m][e], t[m]);
                }
                const float ss = rows_reduce<R>(t, lane, [](float a, float b) { return a + b; });
                if (row_writer<R>(lane)) ssq[wave * 16 + R * s + mine_row] = ss;
#pragma unroll
                for (int m = 0; m < R; m++)
#pragma unroll
                    for (int e = 0; e < 8; e++) v[m][e] *= gl[e];
            }
            // scale: every row's largest magnitude over the wavefront at once, then each row's factor from the lane that holds it
            float am[R];
#pragma unroll
            for (int m = 0; m < R; m++) {
                am[m] = max3_abs(v[m][0], v[m][1], v[m][2]);
                am[m] = max3_abs(v[m][3], v[m][4], am[m]);
                am[m] = max3_abs(v[m][5], v[m][6], am[m]);
                am[m] = max3_abs(v[m][7], v[m][7], am[m]);
            }
            float my_sc, my_iv;
            const float top = rows_reduce<R>(am, lane, [](float a, float b) { return max3_abs(a, b, b); });
            pow2_scale(top, my_sc, my_iv);
            if (row_writer<R>(lane)) invs[mine_row] = my_iv;
            uint32_t hi[R][4], lo[R][4];
#pragma unroll
            for (int m = 0; m < R; m++) {
                const float sc = as_f((uint32_t)__builtin_amdgcn_readlane(__builtin_bit_cast(int, my_sc), lane_of_row<R>(m)));
#pragma unroll
                for (int e = 0; e < 8; e++) v[m][e] *= sc;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    // operand order of four values: nibble masks peel values 0, 2 | 1, 3 off a dword pair, the others are read 0, 1 | 2, 3
                    constexpr bool NIB = T == kQ4_K || T == kQ4_0;
                    const int e0 = NIB ? (e >> 1) * 4 + (e & 1) : 2 * e, e1 = NIB ? e0 + 2 : e0 + 1;
                    // (truncated: what hi drops lo takes up, one mixed-precision multiply-add per value)
                    const h2 hp = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(v[m][e0], v[m][e1]));
                    const h2 lp = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(minus_low(v[m][e0], as_u(hp)), minus_high(v[m][e1], as_u(hp))));
                    hi[m][e] = as_u(hp);
                    lo[m][e] = as_u(lp);
                }
                if constexpr (T == kQ4_K) {  // sums of the 32-value sub-blocks (eight lanes each), as two fp16 halves
                    float s0 = (v[m][0] + v[m][1]) + (v[m][2] + v[m][3]), s1 = (v[m][4] + v[m][5]) + (v[m][6] + v[m][7]);
#define MV_DPP_ADD(ctrl)                                                                                                                   \
    s0 += as_f((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__builtin_bit_cast(uint32_t, s0), ctrl, 0xF, 0xF, true));                     \
    s1 += as_f((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__builtin_bit_cast(uint32_t, s1), ctrl, 0xF, 0xF, true));
                    MV_DPP_ADD(0xB1) MV_DPP_ADD(0x4E) MV_DPP_ADD(0x141)
#undef MV_DPP_ADD
                    const float sum = (lane & 1) ? s1 : s0;  // (even lanes write the sub-blocks of the first half, odd ones of the second)
                    h2 sp;
                    sp.x = (_Float16)sum;
                    sp.y = (_Float16)(sum - (float)sp.x);
                    if ((lane & 7) < 2) sums[m * 16 + 8 * (lane & 1) + (lane >> 3)] = as_u(sp);
                }
            }
            // An infinite activation leaves lo = inf - inf: it becomes 0, and hi alone carries the infinity through the products as the
            // reference's own sums do (NaN stays in hi; rows without an infinity never come here).
            if (__builtin_amdgcn_ballot_w64(top == __builtin_inff()) != 0) {
#pragma unroll
                for (int m = 0; m < R; m++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint32_t l = lo[m][e];
                        lo[m][e] = ((l & 0x7C00u) == 0x7C00u ? 0u : l & 0xFFFFu) | ((l & 0x7C000000u) == 0x7C000000u ? 0u : l & 0xFFFF0000u);
                    }
            }
            wave_fence();
            inv[s][0] = invs[2 * kg];
            inv[s][1] = invs[2 * kg + 1];
            if constexpr (T == kQ4_K) {
                const bool low = (i16 & 2) != 0;  // (the columns of the lo halves carry no sums: both halves of a sum sit in the hi column)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t t = sums[(2 * (i16 >> 2) + (i16 & 1)) * 16 + 8 * (q >> 1) + 2 * kg + (q & 1)];
                    xsum[s][q] = low ? 0u : t;
                }
            }
            // Operand order through the staging area, half a slice (32 octets x 16 columns) at a time: column c of octet o
            // sits at o * 16 + (c ^ (o & 15)) - the xor spreads the octets' stores over the banks, reads of one octet are whole lines.
#pragma unroll
            for (int q = 0; q < 2; q++) {
                // (o * 16 + (c ^ (o & 15)) in bytes is o * 272 with c * 16 xored in, and the octet a step reads, o(kg, j), is kg's part
                // plus j's without a carry: one xor per address)
                uint8_t *const st = area;
                const int to = (lane >> 1) * 256 + ((lane >> 1) & 15) * 16 + (lane & 1) * 8;  // half an octet: lane / 2's, lane % 2
#pragma unroll
                for (int m = 0; m < R; m++) {
                    const int c = 4 * (m >> 1) + (m & 1);
                    *reinterpret_cast<u2 *>(st + (to ^ (c * 16))) = u2{hi[m][2 * q], hi[m][2 * q + 1]};
                    *reinterpret_cast<u2 *>(st + (to ^ ((c + 2) * 16))) = u2{lo[m][2 * q], lo[m][2 * q + 1]};
                }
                wave_fence();
                if constexpr (T == kQ6_K) {
                    const int b = kg >> 1, at = b * 256 + (i16 ^ b) * 16 + (kg & 1) * 8;  // octet 2 j + b, half kg & 1
#pragma unroll
                    for (int j = 0; j < 16; j++) {
                        const u2 t = *reinterpret_cast<const u2 *>(st + (at ^ ((2 * j & 15) * 16)) + 512 * j);
                        x[s][32 * q + 2 * j] = t.x;
                        x[s][32 * q + 2 * j + 1] = t.y;
                    }
                } else {
                    constexpr bool K4 = T == kQ4_K;  // octet 8 kg + j, or 4 j + kg
                    const int at = K4 ? kg * 2048 + (i16 ^ (8 * (kg & 1))) * 16 : kg * 256 + (i16 ^ kg) * 16;
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const u4 t = *reinterpret_cast<const u4 *>(st + (at ^ ((K4 ? j : 4 * (j & 3)) * 16)) + (K4 ? 256 : 1024) * j);
#pragma unroll
                        for (int e = 0; e < 4; e++) x[s][32 * q + 4 * j + e] = t[e];
                    }
                }
                wave_fence();
            }
        }
    }

    constexpr int RR = R * SETS;
    constexpr int CAP = 16 / SETS;  // matrix tiles whose sums the staging area holds
    for (int base = 0; base < nmt; base += CAP) {
        const int n = min(CAP, nmt - base);
        if (wave < live) {
            for (int t = 0; t < n; t++) {
                f4 acc[SETS];
                clear<SETS>(acc);
#pragma unroll
                for (int h = 0; h < G::kUnits; h++) {
                    const int u = (base + t) * G::kUnits + h;
                    Codes<T> c;
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(G::kLoads) : "memory");  // unit u has landed; u + 1 may be on its way
                    c.read(mine + (u & 1) * G::kSlot + i16 * G::kRow, kg, h);
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot has been read before it is filled again
                    fetch(u + 2);
                    if (G::kUnits == 1 || h == 0 || !half) c.template contract<SETS>(x, xsum, kg, h, half, acc);
                }
#pragma unroll
                for (int s = 0; s < SETS; s++)
                    reinterpret_cast<float2 *>(area)[(t * SETS + s) * 64 + lane] =
                        make_float2((acc[s][0] + acc[s][2]) * inv[s][0], (acc[s][1] + acc[s][3]) * inv[s][1]);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (not a wait for the DMAs in flight)
        // thread -> (tile t, activation row m, weight row r)
        for (int e = tid; e < (n >> dual) * 16 * RR; e += (int)blockDim.x) {
            const int r = e & 15, m = (e >> 4) & (RR - 1), t = e / (16 * RR);
            if (m >= A.M) continue;
            const int tile = bx + ((base >> dual) + t) * gx;
            int p = 0;
#pragma unroll
            for (int j = 1; j < kMaxProblems; j++)
                if (j < A.count && tile >= A.tile0[j]) p = j;
            const int row = (tile - A.tile0[p]) * 16 + r;
            if (row >= A.N[p]) continue;
            const int64_t to = (int64_t)m * A.N[p] + row;
            const bool last = gridDim.y == 1;
            const float res = last && A.residual ? A.residual[to] : 0.f;  // (a residual may be y itself: one thread reads and writes an element)
            const float bias = last && A.bias[p] ? A.bias[p][row] : 0.f, bias2 = last && dual && A.bias2 ? A.bias2[row] : 0.f;
            const int at = (((t << dual) * SETS + m / R) * 64 + ((m % R) >> 1) * 16 + r) * 2 + (m & 1);
            float pv[kMaxWaves], pg[kMaxWaves], ps[kMaxWaves];
#pragma unroll
            for (int w = 0; w < kMaxWaves; w++) {  // (every slice's sums are requested before the first is added)
                const int ww = min(w, live - 1);
                const float *q = reinterpret_cast<const float *>(lds + ww * L::kWave + 2 * G::kSlot);
                pv[w] = q[at];
                pg[w] = dual ? q[at + SETS * 128] : 0.f;
                ps[w] = A.norm ? ssq[ww * 16 + m] : 0.f;
            }
            float v = 0.f, g = 0.f, ss = 0.f;
#pragma unroll
            for (int w = 0; w < kMaxWaves; w++)
                if (w < live) { v += pv[w]; g += pg[w]; ss += ps[w]; }
            if (!last) {
                const int64_t pto = ((int64_t)blockIdx.y * A.M + m) * A.ntot + A.n0[p] + row;
                A.partial[pto] = v;
                if (dual) A.partial2[pto] = g;
                if (A.norm && tile == 0 && r == 0) A.xss[(int)blockIdx.y * A.M + m] = ss;
                continue;
            }
            const float rn = A.norm ? 1.f / sqrtf(ss * A.inv_k + A.eps) : 1.f;
            v = apply_act(A.act[p], fmaf(v, rn, bias));
            if (dual) v *= fmaf(g, rn, bias2);
            if (A.residual) v += res;
            A.y[p][to] = v;
        }
        if (base + CAP < nmt) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the empty requests behind the last unit
}

struct Plan { int nslices, waves, groups; };
Plan plan_of(int64_t K) {
    Plan p;
    p.nslices = (int)((K + kSlice - 1) / kSlice);
    p.groups = (p.nslices + kMaxWaves - 1) / kMaxWaves;
    p.waves = (p.nslices + p.groups - 1) / p.groups;
    p.groups = (p.nslices + p.waves - 1) / p.waves;
    return p;
}

template <int T, bool BF, int SETS, int R>
int launch_mmv_rows(const void *x, const MmvArgs &a, const Plan &p, hipStream_t s) {
    typedef MVLds<T, SETS> L;
    static const bool lds_ok = [] {
        return hipFuncSetAttribute(reinterpret_cast<const void *>(mmv_kernel<T, BF, SETS, R>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   L::bytes(kMaxWaves)) == hipSuccess;
    }();
    if (!lds_ok) return fail(GQ_ERR_HIP, "mmv: cannot reserve %d bytes of LDS", L::bytes(kMaxWaves));
    // Eight wavefronts per CU, two per SIMD, as registers and LDS hold them: one workgroup of five to eight, two of three or four, four of
    // two, eight of one; the slices' groups share them, the tiles are dealt out round-robin.  (With one workgroup per CU, short rows left
    // three quarters of the chip's loads unissued from nine rows on: Q4_0 1024 -> 32768 at 12 rows 32.2 us for 18.8, Q8_0
    // 256 -> 32768 46.8 for 15.3 at 16.)  Two sets of rows convert for half a microsecond longer where a SIMD has both wavefronts
    // converting: a second workgroup of three or four wavefronts pays from three tiles per CU on (Q8_0 2048 -> 8192 at 12 rows, two tiles:
    // 13.1 us with it, 12.4 without; -> 16384, four tiles: 17.4 and 18.2).
    const int cus = device_cu_count();
    int per_cu = kMaxWaves / p.waves;
    if (SETS == 2 && per_cu == 2 && a.ntiles < 3 * cus) per_cu = 1;
    int gx = std::max(1, std::min(a.ntiles, cus * per_cu / p.groups));
    MmvArgs b = a;
    if (a.apart) {  // every matrix its share of the workgroups, in proportion to its tiles
        const int total = gx;
        gx = 0;
        for (int j = 0; j < a.count; j++) {
            const int tiles = (j + 1 < a.count ? a.tile0[j + 1] : a.ntiles) - a.tile0[j];
            b.wg0[j] = gx;
            b.wgs[j] = std::max(1, (int)((int64_t)total * tiles / a.ntiles));
            gx += b.wgs[j];
        }
    }
    return launch(mmv_kernel<T, BF, SETS, R>, dim3((unsigned)gx, (unsigned)p.groups), dim3((unsigned)p.waves * 64), (size_t)L::bytes(p.waves), s, x, b);
}

template <int T>
int launch_mmv_t(const void *x, bool bf, const MmvArgs &a, const Plan &p, hipStream_t s) {
    if (a.M <= 4) return bf ? launch_mmv_rows<T, true, 1, 4>(x, a, p, s) : launch_mmv_rows<T, false, 1, 4>(x, a, p, s);
    if (a.M <= 8) return bf ? launch_mmv_rows<T, true, 1, 8>(x, a, p, s) : launch_mmv_rows<T, false, 1, 8>(x, a, p, s);
    return bf ? launch_mmv_rows<T, true, 2, 8>(x, a, p, s) : launch_mmv_rows<T, false, 2, 8>(x, a, p, s);
}

}  // namespace

bool mmv_one_launch(int64_t K) { return plan_of(K).groups == 1; }

bool mmv_supported(int type, int64_t M, int64_t K, int64_t N, const void *x, const void *gain) {
    if (type != kQ4_K && type != kQ8_0 && type != kQ4_0 && type != kIQ4_NL && type != kQ6_K) return false;
    if (M < 3 || M > 16 || N < 1 || N > (int64_t)INT32_MAX / 64 || K < 256 || K > (1 << 20)) return false;
    if (K % (type == kQ6_K ? 512 : 256) != 0) return false;  // (Q6_K: rows of whole dwords)
    return ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(gain)) & 15) == 0;
}

// The same activations against `count` matrices (one with W2, bias2: a gated pair; a residual goes with one matrix only).  K of
// more than eight slices needs workspace and, for the reduction, N % 4 == 0 (the dispatch sends other N here in one launch only).  xs: activations of
// their own for every matrix (two or more of up to eight slices, no extras).
int launch_mmv(int type, const void *x, bool x_is_bf16, int64_t M, int64_t K, int count, const MmqSetItem *items, const MmqExtra *ex, hipStream_t s,
               const void *const *xs) {
    if (count < 1 || count > kMaxProblems) return fail(GQ_ERR_NOT_IMPLEMENTED, "mmv: a set of %d matrices is not implemented", count);
    const Plan p = plan_of(K);
    if (xs && (count < 2 || ex || p.groups > 1)) return fail(GQ_ERR_NOT_IMPLEMENTED, "mmv: activations per matrix in this form are not implemented");
    MmvArgs a = {};
    a.apart = xs ? 1 : 0;
    for (int i = 0; xs && i < count; i++) a.X[i] = xs[i];
    int64_t tiles = 0, ntot = 0;
    for (int i = 0; i < count; i++) {
        a.W[i] = items[i].W; a.bias[i] = items[i].bias; a.y[i] = items[i].y; a.N[i] = (int)items[i].N; a.act[i] = items[i].act;
        a.tile0[i] = (int)tiles; a.n0[i] = (int)ntot;
        tiles += (items[i].N + 15) / 16;
        ntot += items[i].N;  // (two launches: the sums' rows are whole float4)
        if (p.groups > 1 && items[i].N % 4 != 0) return fail(GQ_ERR_NOT_IMPLEMENTED, "mmv: N off 4 in two launches is not implemented");
    }
    if (tiles > INT32_MAX / 64 || ntot > INT32_MAX) return fail(GQ_ERR_NOT_IMPLEMENTED, "mmv: too many weight rows");
    a.count = count; a.ntiles = (int)tiles; a.M = (int)M; a.K = (int)K; a.nslices = p.nslices; a.ntot = (int)ntot;
    if (ex) {
        a.W2 = ex->W2; a.bias2 = ex->bias2; a.residual = ex->residual;
        if (ex->norm) { a.norm = 1; a.gain = ex->norm->gain; a.gain_offset = ex->norm->gain_offset; a.eps = ex->norm->eps; a.inv_k = 1.0f / (float)K; }
    }
    if (p.groups > 1) {
        const size_t xss_bytes = ((size_t)p.groups * M * sizeof(float) + 255) & ~(size_t)255, part = (size_t)p.groups * M * ntot;
        void *ws = nullptr;
        if (int rc = stream_workspace(s, xss_bytes + part * sizeof(float) * (a.W2 ? 2 : 1), &ws)) return rc;
        a.xss = static_cast<float *>(ws);
        a.partial = reinterpret_cast<float *>(static_cast<uint8_t *>(ws) + xss_bytes);
        a.partial2 = a.W2 ? a.partial + part : nullptr;
    }
    int rc;
    switch (type) {
    case kQ4_K: rc = launch_mmv_t<kQ4_K>(x, x_is_bf16, a, p, s); break;
    case kQ8_0: rc = launch_mmv_t<kQ8_0>(x, x_is_bf16, a, p, s); break;
    case kQ4_0: rc = launch_mmv_t<kQ4_0>(x, x_is_bf16, a, p, s); break;
    case kIQ4_NL: rc = launch_mmv_t<kIQ4_NL>(x, x_is_bf16, a, p, s); break;
    case kQ6_K: rc = launch_mmv_t<kQ6_K>(x, x_is_bf16, a, p, s); break;
    default: rc = fail(GQ_ERR_NOT_IMPLEMENTED, "mmv: ggml type %d is not implemented", type);
    }
    if (rc || p.groups == 1) return rc;
    return launch_split_k_finish(a.partial, a.partial2, a.xss, p.groups, M, K, count, items, ex, s);
}

}  // namespace gq
