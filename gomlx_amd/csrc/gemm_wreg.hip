// Quantised Dense for large batches in one GEMM: the weights go from their GGML blocks into MFMA operands in registers, so that no
// 16-bit image of them is written and read back (gemm_dma.hip's way, whose image pass is a third of a decoder layer at 512 rows).
//
// Tile: 256 weight rows x 32 TM activation rows per workgroup, four wavefronts of 64 weight rows x all the activation rows: a weight is
// converted by exactly one wavefront of the workgroup, and an activation fragment read from LDS feeds two matrix instructions.  One
// wavefront per SIMD: its 512 registers hold 64 x 256 sums beside two sets of fragments, and the conversion of the next 16 values of K
// (at most 4 vector-ALU instructions per matrix instruction) is placed between the matrix instructions of the present ones.
//
// Activations: 16-bit rows [M, K], 64 values of K per step by DMA through a ring of LDS stages (rows of 128 bytes, chunks swizzled as in
// gemm_dma.hip).  Weights: a wavefront copies the raw bytes of 256 values of its 64 rows (consecutive 16-byte chunks) by DMA into a
// piece of LDS of its own and takes them into registers when it starts on them; the copy of the next 256 values then has three steps
// to land.  Operand values: the exact fp32 weight, rounded once - the values of the two-pass route.
//
// What bounds it: a step of 64 values of K takes a 256-row tile 2700 cycles for 2048 of matrix instructions (conversion 390, DMAs 350, the
// rest waits around the step's barrier) at the 2.0 - 2.1 GHz that the power limit leaves the whole chip; 2.5 us pass before the first bytes
// arrive and 4 to 6 in the epilogue.  4096 -> 2 x 14336 in Q4_K at 512 rows: 119 us (1.0 PFLOP/s, activations' conversion included) where the
// image and the GEMM over it took 165.
#include "blocks.hpp"
#include "common.hpp"
#include "lds_dma.hpp"

#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <utility>

namespace gq {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int ROWB = 128;   // bytes of an activation row in a stage: 64 values
constexpr int kUnit = 256;  // values of K per raw weight copy

template <bool BF16> struct Op;
template <> struct Op<true> {
    typedef bf16x8 vec8;
    static __device__ __forceinline__ uint32_t pack(float a, float b) {
        typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
        bf2 v;
        v.x = (__bf16)a;
        v.y = (__bf16)b;
        return __builtin_bit_cast(uint32_t, v);
    }
    static __device__ __forceinline__ f32x16 mfma(vec8 a, vec8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};
template <> struct Op<false> {
    typedef f16x8 vec8;
    static __device__ __forceinline__ uint32_t pack(float a, float b) {
        h2 v;
        v.x = (_Float16)a;
        v.y = (_Float16)b;
        return __builtin_bit_cast(uint32_t, v);
    }
    static __device__ __forceinline__ f32x16 mfma(vec8 a, vec8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};
__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }

// Eight weights whose codes arrive as fp16 pairs (v0, v2), (v1, v3), (v4, v6), (v5, v7) - NATURAL: (v0, v1) ... - as operands
// code * s + c: one fp32 multiply-add per weight, rounded once (v_fma_mix).
template <bool BF16, bool NATURAL>
__device__ __forceinline__ void finish8(const h2 (&p)[4], float s, float c, uint32_t (&w)[4]) {
    auto v = [&](_Float16 h) __attribute__((always_inline)) { return fmaf((float)h, s, c); };
    if constexpr (NATURAL) {
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = Op<BF16>::pack(v(p[i].x), v(p[i].y));
    } else {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            w[2 * i] = Op<BF16>::pack(v(p[2 * i].x), v(p[2 * i + 1].x));
            w[2 * i + 1] = Op<BF16>::pack(v(p[2 * i].y), v(p[2 * i + 1].y));
        }
    }
}

// The raw bytes of one unit (256 values) of a 32-row tile as lane (row, half h of every 16 values) needs them.
//   kChunks: 16-byte chunks of a row;  load: out of the parked copy of the tile;
//   scale<G, HI>: multiplier and addend of the 32 values 64 G + 32 HI ..;  frag<BF16, G, KK>: operands 64 G + 16 KK + 8 h ..
template <int T> struct RawUnit;

template <> struct RawUnit<kQ4_K> {
    static constexpr int kChunks = 9;
    u32x4 hd;
    u32x2 c[4][2];
    __device__ __forceinline__ void load(const uint8_t *park, int row, int h) {
        const uint8_t *p = park + row * 144;
        hd = *reinterpret_cast<const u32x4 *>(p);
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int q = 0; q < 2; q++) c[g][q] = *reinterpret_cast<const u32x2 *>(p + 16 + 32 * g + 16 * q + 8 * h);
    }
    template <int G, int HI> __device__ __forceinline__ void scale(float &s, float &m) const {
        uint32_t sc, mn;
        q4k_scale_min(hd.y, hd.z, hd.w, 2 * G + HI, sc, mn);
        // (codes arrive as fp16 subnormals n 2^-24, those of the high nibbles as n 2^-20)
        s = half_bits_to_float(hd.x & 0xFFFFu) * ((float)sc * (HI ? 0x1p20f : 0x1p24f));
        m = -(half_bits_to_float(hd.x >> 16) * (float)mn);
    }
    template <bool BF16, int G, int KK> __device__ __forceinline__ void frag(float s, float m, uint32_t (&w)[4]) const {
        constexpr uint32_t mask = KK >= 2 ? 0x00F000F0u : 0x000F000Fu;
        const uint32_t a = c[G][KK & 1].x, b = c[G][KK & 1].y;
        const h2 p[4] = {as_h2(a & mask), as_h2((a >> 8) & mask), as_h2(b & mask), as_h2((b >> 8) & mask)};
        finish8<BF16, false>(p, s, m, w);
    }
};

// 18-byte blocks: fp16 d, 16 code bytes (values 0 .. 15 in the low nibbles, 16 .. 31 in the high ones)
template <int T> struct RawNibble {
    static constexpr int kChunks = 9;
    u32x2 c[8];
    uint32_t d[4];
    __device__ __forceinline__ void load(const uint8_t *park, int row, int h) {
        const uint32_t *p = reinterpret_cast<const uint32_t *>(park + row * 144);
#pragma unroll
        for (int g = 0; g < 4; g++) {  // a pair of blocks is nine dwords: the first's codes lie half a dword off
            const uint32_t *q = p + 9 * g;
            const uint32_t w0 = q[2 * h], w1 = q[2 * h + 1], w2 = q[2 * h + 2];
            c[2 * g] = u32x2{__builtin_amdgcn_alignbit(w1, w0, 16), __builtin_amdgcn_alignbit(w2, w1, 16)};
            c[2 * g + 1] = u32x2{q[5 + 2 * h], q[6 + 2 * h]};
            d[g] = __builtin_amdgcn_perm(q[4], q[0], 0x07060100u);  // (d of the first block, d of the second)
        }
    }
    template <int G, int HI> __device__ __forceinline__ void scale(float &s, float &m) const {
        s = half_bits_to_float(HI ? d[G] >> 16 : d[G] & 0xFFFFu);
        m = 0.f;
    }
    template <bool BF16, int G, int KK> __device__ __forceinline__ void frag(float s, float m, uint32_t (&w)[4]) const {
        const uint32_t u[2] = {c[2 * G + (KK >> 1)].x, c[2 * G + (KK >> 1)].y};
        h2 p[4];
        if constexpr (T == kQ4_0) {  // n - 8, exact, before the scale meets it: an infinite d gives the reference's infinities
            constexpr uint32_t mask = KK & 1 ? 0x00F000F0u : 0x000F000Fu;
            uint32_t magic = KK & 1 ? 0x54005400u : 0x64006400u;  // fp16 64 + n and 1024 + n
            asm("" : "+v"(magic));
            const h2 off = as_h2(KK & 1 ? 0xD480D480u : 0xE408E408u);  // -72, -1032
#pragma unroll
            for (int i = 0; i < 2; i++) {
                p[2 * i] = as_h2((u[i] & mask) | magic) + off;
                p[2 * i + 1] = as_h2(((u[i] >> 8) & mask) | magic) + off;
            }
            finish8<BF16, false>(p, s, m, w);
        } else {  // four code-book entries (+ 128, unsigned) at a time by byte permutes: see iq4nl_value
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t n = KK & 1 ? u[i] >> 4 : u[i];
                const uint32_t low3 = n & 0x07070707u;
                const uint32_t lo = __builtin_amdgcn_perm(0x766A5D4Fu, 0x3F2D1801u, low3), hi = __builtin_amdgcn_perm(0xF1D9C5B5u, 0xA6998D81u, low3);
                const uint32_t e = __builtin_amdgcn_perm(hi, lo, 0x03020100u | ((n & 0x08080808u) >> 1));
                const h2 off = as_h2(0xE480E480u);  // -1152
                p[2 * i] = as_h2(__builtin_amdgcn_perm(0x64646464u, e, 0x04010400u)) + off;
                p[2 * i + 1] = as_h2(__builtin_amdgcn_perm(0x64646464u, e, 0x04030402u)) + off;
            }
            finish8<BF16, true>(p, s, m, w);
        }
    }
};
template <> struct RawUnit<kQ4_0> : RawNibble<kQ4_0> {};
template <> struct RawUnit<kIQ4_NL> : RawNibble<kIQ4_NL> {};

template <> struct RawUnit<kQ8_0> {  // 34-byte blocks: fp16 d, 32 signed bytes
    static constexpr int kChunks = 17;
    u32x2 c[8][2];
    uint32_t d[4];
    __device__ __forceinline__ void load(const uint8_t *park, int row, int h) {
        const uint32_t *p = reinterpret_cast<const uint32_t *>(park + row * 272);
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const uint32_t *r = p + 17 * g;
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const uint32_t w0 = r[4 * q + 2 * h], w1 = r[4 * q + 2 * h + 1], w2 = r[4 * q + 2 * h + 2];
                c[2 * g][q] = u32x2{__builtin_amdgcn_alignbit(w1, w0, 16), __builtin_amdgcn_alignbit(w2, w1, 16)};
                c[2 * g + 1][q] = u32x2{r[9 + 4 * q + 2 * h], r[10 + 4 * q + 2 * h]};
            }
            d[g] = __builtin_amdgcn_perm(r[8], r[0], 0x07060100u);
        }
    }
    template <int G, int HI> __device__ __forceinline__ void scale(float &s, float &m) const {
        s = half_bits_to_float(HI ? d[G] >> 16 : d[G] & 0xFFFFu);
        m = 0.f;
    }
    template <bool BF16, int G, int KK> __device__ __forceinline__ void frag(float s, float m, uint32_t (&w)[4]) const {
        const uint32_t u[2] = {c[2 * G + (KK >> 1)][KK & 1].x, c[2 * G + (KK >> 1)][KK & 1].y};
        h2 p[4];
        const h2 off = as_h2(0xE480E480u);  // -1152: fp16 1024 + (q + 128) back to q, exact
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t e = u[i] ^ 0x80808080u;
            p[2 * i] = as_h2(__builtin_amdgcn_perm(0x64646464u, e, 0x04010400u)) + off;
            p[2 * i + 1] = as_h2(__builtin_amdgcn_perm(0x64646464u, e, 0x04030402u)) + off;
        }
        finish8<BF16, true>(p, s, m, w);
    }
};

template <int T, int TM> struct WregTile {
    static constexpr int kChunks = RawUnit<T>::kChunks;
    static constexpr int kParkTile = 32 * kChunks * 16;               // raw bytes of a 32-row tile
    static constexpr int kTileDmas = (32 * kChunks + 63) / 64;        // (the last one carries 32 chunks)
    static constexpr int kRawDmas = 2 * kTileDmas;
    static constexpr int kStage = 32 * TM * ROWB;
    static constexpr int kPark = 8 * kParkTile;                       // four wavefronts, two tiles each
    static constexpr int NS = 3 * kStage + kPark <= 160 * 1024 ? 3 : 2;
    static constexpr int kLds = NS * kStage + kPark;
    static_assert(kLds <= 160 * 1024, "stages + parked weights exceed LDS");
};

// One matrix, up to four that share the activations (matrix p owns workgroups wg0[p] .. of grid.x and columns n0[p] .. of the sums), or a
// gated pair (W[0], W[1]; 128 outputs per workgroup).  gridDim.z slices of units_per_slice units of K: with more than one the sums go to
// partial[z][M][ntot].
struct WregArgs {
    const uint16_t *X;
    const uint8_t *W[4];
    const float *bias[4];
    float *Y[4];
    int N[4], wg0[4], n0[4];
    int count, ntot, M, K, act, units_per_slice;
    int64_t row_bytes;
    const float *residual, *rowscale;
    float *partial;
};

template <int T, bool BF16, int TM, bool GATED>
__global__ __launch_bounds__(256, 1) void gemm_wreg_kernel(WregArgs a) {
    typedef WregTile<T, TM> G;
    typedef typename Op<BF16>::vec8 vec8;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 31, h = lane >> 5;
    int prob = 0;
    if constexpr (!GATED) {
#pragma unroll
        for (int j = 1; j < 4; j++)
            if (j < a.count && (int)blockIdx.x >= a.wg0[j]) prob = j;
    }
    const int N = a.N[prob], M = a.M, K = a.K;
    const int bm = blockIdx.y * (32 * TM);
    const int row0 = ((int)blockIdx.x - a.wg0[prob]) * (GATED ? 128 : 256) + wave * (GATED ? 32 : 64);  // first weight row of this wavefront
    const int units = K / kUnit, u0 = (int)blockIdx.z * a.units_per_slice, nu = min(a.units_per_slice, units - u0), nsteps = 4 * nu;

    // ---- DMA roles
    const i32x4 xrsrc = make_rsrc(a.X + (int64_t)bm * K, (uint64_t)(M - bm) * (uint64_t)K * 2);  // (rows past M read as zero)
    i32x4 wrsrc[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int r = GATED ? row0 : row0 + 32 * j;
        const uint8_t *W = GATED ? a.W[j] : a.W[prob];
        wrsrc[j] = make_rsrc(W + (int64_t)min(r, N) * a.row_bytes, (uint64_t)max(N - r, 0) * (uint64_t)a.row_bytes);  // (and rows past N)
    }
    // activations: wavefront w copies rows 8 (TM w + j) + lane / 8 of the tile, j = 0 .. TM - 1
    uint32_t xvoff[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int row = 8 * (TM * wave + j) + (lane >> 3);
        xvoff[j] = (uint32_t)row * (uint32_t)(K * 2) + (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 16u;
    }
    uint32_t wvoff[G::kTileDmas];
#pragma unroll
    for (int l = 0; l < G::kTileDmas; l++) {
        const int c = min(lane + 64 * l, 32 * G::kChunks - 1);
        wvoff[l] = (uint32_t)(c / G::kChunks) * (uint32_t)a.row_bytes + (uint32_t)((c % G::kChunks) * 16);
    }
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(lds);
    const uint32_t xdst = lds0 + (uint32_t)(TM * wave) * 1024u;
    uint8_t *const park = lds + G::NS * G::kStage + wave * (2 * G::kParkTile);
    const uint32_t wdst = lds0 + (uint32_t)(G::NS * G::kStage + wave * (2 * G::kParkTile));
    // (steps and units past the end re-read the last one: the data is never used)
    auto issue_x = [&](int step, uint32_t stage_off, int j) __attribute__((always_inline)) {
        const uint32_t soff = (uint32_t)(4 * u0 + min(step, nsteps - 1)) * (uint32_t)ROWB + (uint32_t)(j >> 1) * (uint32_t)(32 * K);
        dma16(xdst + stage_off + (uint32_t)j * 1024u, xrsrc, xvoff[j & 1], soff);
    };
    auto issue_w = [&](int unit, int j) __attribute__((always_inline)) {
        const uint32_t soff = (uint32_t)(u0 + min(unit, nu - 1)) * (uint32_t)(G::kChunks * 16);
#pragma unroll
            for (int l = 0; l < G::kTileDmas; l++)
                if (64 * l + 64 <= 32 * G::kChunks || lane < 32 * G::kChunks - 64 * l)
                    dma16(wdst + (uint32_t)(j * G::kParkTile + l * 1024), wrsrc[j], wvoff[l], soff);
    };
    // ---- activation fragments: row 32 t + lane % 32, chunk 2 kk + lane / 32, swizzled
    uint32_t aoff[4];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) aoff[kk] = (uint32_t)col * ROWB + (uint32_t)((2 * kk + h) ^ ((col >> 1) & 7)) * 16u;

    f32x16 acc[2][TM];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int t = 0; t < TM; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[j][t][r] = 0.f;

    vec8 xf[2][TM];
    uint32_t wf[2][2][4];  // [set][tile]
    RawUnit<T> raw[2];
    float sc[2], mn[2];
    auto frags = [&](uint32_t stage_off, int kk, int set) __attribute__((always_inline)) {
        const uint8_t *base = lds + stage_off + aoff[kk];
#pragma unroll
        for (int t = 0; t < TM; t++) xf[set][t] = *reinterpret_cast<const vec8 *>(base + t * 32 * ROWB);
    };
    auto convert = [&](int j, auto gc, auto kc) __attribute__((always_inline)) {
        constexpr int g = decltype(gc)::value, kk = decltype(kc)::value;
        if constexpr ((kk & 1) == 0) raw[j].template scale<g, (kk >> 1)>(sc[j], mn[j]);
        raw[j].template frag<BF16, g, kk>(sc[j], mn[j], wf[kk & 1][j]);
    };
    auto mfmas = [&](int set, int half) __attribute__((always_inline)) {
#pragma unroll
        for (int t = half * (TM / 2); t < (half + 1) * (TM / 2); t++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                acc[j][t] = Op<BF16>::mfma(xf[set][t], __builtin_bit_cast(vec8, u32x4{wf[set][j][0], wf[set][j][1], wf[set][j][2], wf[set][j][3]}), acc[j][t]);
    };
    // a vector-ALU share and, READS, an LDS read behind every matrix instruction of half a group
    auto interleave = [](auto reads) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (decltype(reads)::value) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, TM == 8 ? 3 : TM == 6 ? 4 : 6, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load_raw = [&]() __attribute__((always_inline)) {
        raw[0].load(park, col, h);
        raw[1].load(park + G::kParkTile, col, h);
    };

#define GQ_PUBLISH(left) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(left) : "memory")
    // Requests, in order: x(0) raw(0) x(1) | step s: x(s + NS - 1), and behind it, in the second and third step of a unit, the raw bytes
    // of the next unit's first and second tile.  A step ends when x(s + 1) has landed - the last step of a unit: the raw bytes too -;
    // what was requested after it may stay in flight.
#pragma unroll
    for (int j = 0; j < TM; j++) issue_x(0, 0, j);
    issue_w(0, 0);
    issue_w(0, 1);
    if constexpr (G::NS == 3) {
#pragma unroll
        for (int j = 0; j < TM; j++) issue_x(1, G::kStage, j);
    }
    GQ_PUBLISH((G::NS - 2) * TM);
    load_raw();
    frags(0, 0, 0);
    typedef std::integral_constant<int, 0> Zero;
    convert(0, Zero(), Zero());
    convert(1, Zero(), Zero());
    __builtin_amdgcn_sched_barrier(0);

    uint32_t stage = 0, fill = (G::NS - 1) * G::kStage;  // byte offsets: the stage that is read, the one that is filled
    auto next_stage = [](uint32_t s) __attribute__((always_inline)) { return s == (G::NS - 1) * G::kStage ? 0u : s + G::kStage; };
    for (int u = 0; u < nu; u++) {
        auto step = [&](auto gc) __attribute__((always_inline)) {
            constexpr int g = decltype(gc)::value;
            auto group = [&](auto kc) __attribute__((always_inline)) {
                constexpr int kk = decltype(kc)::value;
                // this step's DMAs go out one by one between half groups: several in a row hold the wavefront up for 50 cycles each
                auto slot = [&](int sl) __attribute__((always_inline)) {
#pragma unroll
                    for (int j = 0; j < TM; j++)
                        if (j * 6 / TM == sl) issue_x(4 * u + g + G::NS - 1, fill, j);
                };
                if constexpr (kk < 3) {
                    slot(2 * kk);
                    frags(stage, kk + 1, (kk + 1) & 1);
                    mfmas(kk & 1, 0);
                    convert(0, gc, std::integral_constant<int, kk + 1>());
                    interleave(std::true_type());
                    slot(2 * kk + 1);
                    if constexpr (kk == 2 && (g == 1 || g == 2)) issue_w(u + 1, g - 1);
                    mfmas(kk & 1, 1);
                    convert(1, gc, std::integral_constant<int, kk + 1>());
                    interleave(std::false_type());
                } else {
                    if constexpr (G::NS == 3) {
                        if constexpr (g == 0 || g == 3) GQ_PUBLISH(TM);
                        else if constexpr (g == 1) GQ_PUBLISH(TM + G::kTileDmas);
                        else GQ_PUBLISH(TM + 2 * G::kTileDmas);
                    } else {
                        if constexpr (g == 0 || g == 3) GQ_PUBLISH(0);
                        else GQ_PUBLISH(G::kTileDmas);
                    }
                    stage = next_stage(stage);
                    fill = next_stage(fill);
                    if constexpr (g == 3) load_raw();
                    frags(stage, 0, 0);
                    mfmas(1, 0);
                    if constexpr (g != 3) convert(0, std::integral_constant<int, (g + 1) & 3>(), Zero());
                    interleave(std::true_type());
                    mfmas(1, 1);
                    if constexpr (g == 3) convert(0, Zero(), Zero());
                    convert(1, std::integral_constant<int, (g + 1) & 3>(), Zero());
                    interleave(std::false_type());
                }
            };
            group(std::integral_constant<int, 0>());
            group(std::integral_constant<int, 1>());
            group(std::integral_constant<int, 2>());
            group(std::integral_constant<int, 3>());
        };
        step(std::integral_constant<int, 0>());
        step(std::integral_constant<int, 1>());
        step(std::integral_constant<int, 2>());
        step(std::integral_constant<int, 3>());
    }
    GQ_PUBLISH(0);  // the re-read DMAs of the last steps; all of LDS is free now

    // ---- epilogue: acc[j][t][r] is row m = 32 t + 8 (r / 4) + 4 h + r % 4, column n = lane % 32 of tile j
    // Half the sums at a time go through a piece of LDS of the wavefront's own and are finished and stored in loops that are not unrolled.
    // Stores count as outstanding memory operations, in order with loads: a load between two stores would wait for the first one's way to
    // memory (a row scale loaded per store made this 27 us of a 256 x 256 tile's 105), so row scales come from LDS and a residual is requested in
    // front of the stores before its own.  Sums (16 t + r) of a tile lie 64 floats apart, a lane's own beside its neighbours': eight rows of
    // 32 columns are 256 consecutive floats, row 4 (l / 8 % 2) + l / 16 and columns 4 (l % 8) .. + 3 in lane l's four.
    constexpr int TH = TM / 2;
    float *const xch = reinterpret_cast<float *>(lds + wave * (2 * TH * 4096));
    float *const srow = reinterpret_cast<float *>(lds + 4 * (2 * TH * 4096));
    static_assert(4 * (2 * TH * 4096) + 128 * TM <= G::kLds, "the epilogue's LDS");
    const bool sliced = !GATED && gridDim.z > 1;
    const int ld = sliced ? a.ntot : N;
    float *const Y = sliced ? a.partial + (int64_t)blockIdx.z * M * a.ntot + a.n0[prob] : a.Y[prob];
    const float *const R = sliced ? nullptr : a.residual;
    const float *const B0 = sliced ? nullptr : a.bias[prob], *const B1 = GATED ? a.bias[1] : nullptr;
    const int act = sliced ? kActNone : a.act;
    if (threadIdx.x < 32 * TM) {
        const int m = bm + (int)threadIdx.x;
        srow[threadIdx.x] = !sliced && a.rowscale && m < M ? a.rowscale[m] : 1.f;
    }
    // the biases of a lane's four columns of either tile (gated: of either matrix)
    float4 bias[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const float *const B = GATED && j ? B1 : B0;
        const int n = row0 + (GATED ? 0 : 32 * j) + 4 * (lane & 7);
        auto at = [&](int c) __attribute__((always_inline)) { return B && n + c < N ? B[n + c] : 0.f; };
        bias[j] = make_float4(at(0), at(1), at(2), at(3));
    }
    __syncthreads();
    auto finish = [&](float v0, float v1, float s, float b, float b1, auto activate) __attribute__((always_inline)) {
        if constexpr (GATED) return activate(fmaf(v0, s, b)) * fmaf(v1, s, b1);
        else return activate(fmaf(v0, s, b));
    };
    const int lr = 4 * ((lane >> 3) & 1) + (lane >> 4);  // a lane's row of eight
    // pass p, tile j, four columns a lane.  Rows and pointers need not be whole float4: these instructions ask for whole dwords (an element at a time, behind
    // a branch for its row and a switch for the activation, took 33 us of a 256 x 256 tile and 80 with a residual).
    auto store_vec = [&](int p, int j, auto activate) __attribute__((always_inline)) {
        const int n = row0 + 32 * j + 4 * (lane & 7);
        const float *const src = xch + j * (TH * 1024) + 4 * lane;
        const float4 b0 = j ? bias[1] : bias[0], b1 = bias[1];
        if (n + 4 > N) return;
        // (buffer stores and loads: what lies past the last row is dropped resp. zero, so that no branch stands between one row's LDS reads and the next's)
        const uint64_t tail = (uint64_t)(M - bm) * (uint64_t)ld * 4;
        const uint32_t bytes = tail > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)tail;
        const auto yr = __builtin_amdgcn_make_buffer_rsrc(Y + (int64_t)bm * ld, 0, bytes, 0x00020000);
        uint32_t at = ((uint32_t)(32 * TH * p + lr) * (uint32_t)ld + (uint32_t)n) * 4u;
        const uint32_t step = (uint32_t)ld * 32u;
        auto value = [&](int q) __attribute__((always_inline)) {
            float4 v = *reinterpret_cast<const float4 *>(src + 256 * q), w = v;
            if constexpr (GATED) w = *reinterpret_cast<const float4 *>(src + TH * 1024 + 256 * q);
            const float s = srow[32 * TH * p + 8 * q + lr];
            return make_float4(finish(v.x, w.x, s, b0.x, b1.x, activate), finish(v.y, w.y, s, b0.y, b1.y, activate), finish(v.z, w.z, s, b0.z, b1.z, activate),
                               finish(v.w, w.w, s, b0.w, b1.w, activate));
        };
        if (!R) {
#pragma unroll 4
            for (int q = 0; q < 4 * TH; q++, at += step)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, value(q)), yr, at, 0, 0);
            return;
        }
        // (y may be the residual itself: one thread reads and writes an element, and reads no other thread's)
        const auto rr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(R) + (int64_t)bm * ld, 0, bytes, 0x00020000);
        constexpr int D = TH == 3 ? 6 : 8;  // rows of the residual on their way
        float4 r[D];
#pragma unroll
        for (int i = 0; i < D; i++) r[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rr, at + i * step, 0, 0));
#pragma unroll 1
        for (int q = 0; q < 4 * TH; q += D, at += D * step) {
            float4 next[D];
#pragma unroll
            for (int i = 0; i < D; i++)  // (past this pass's last row: loaded and not used, inside the matrix or zero)
                next[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rr, at + (D + i) * step, 0, 0));
#pragma unroll
            for (int i = 0; i < D; i++) {
                float4 v = value(q + i);
                v.x += r[i].x; v.y += r[i].y; v.z += r[i].z; v.w += r[i].w;
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), yr, at + i * step, 0, 0);
                r[i] = next[i];
            }
        }
    };
    // the one to three columns in front of N that are no whole four: finished where they lie, one row after the other, then stored element by element
    auto store_tail = [&](int p, int j) __attribute__((always_inline)) {
        const int n = row0 + 32 * j + 4 * (lane & 7);
        float *const src = xch + j * (TH * 1024) + 4 * lane;
        const float4 b0 = j ? bias[1] : bias[0], b1 = bias[1];
        if (n >= N || n + 4 <= N) return;
#pragma unroll 1
        for (int q = 0; q < 4 * TH; q++) {
            const float s = srow[32 * TH * p + 8 * q + lr];
#pragma unroll 1
            for (int c = 0; c < 3; c++) {
                const float bc = c == 0 ? b0.x : c == 1 ? b0.y : b0.z, b1c = c == 0 ? b1.x : c == 1 ? b1.y : b1.z;
                src[256 * q + c] = finish(src[256 * q + c], GATED ? src[TH * 1024 + 256 * q + c] : 0.f, s, bc, b1c, [act](float v) { return apply_act(act, v); });
            }
        }
        const int64_t at = (int64_t)(bm + 32 * TH * p + lr) * ld + n;
        constexpr int D = TH == 3 ? 6 : 8;
#pragma unroll 1
        for (int q = 0; q < 4 * TH; q += D) {
            float r[D][3];
#pragma unroll
            for (int i = 0; i < D; i++)
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    r[i][c] = src[256 * (q + i) + c];
                    if (R && n + c < N && bm + 32 * TH * p + lr + 8 * (q + i) < M) r[i][c] += R[at + (int64_t)(8 * (q + i)) * ld + c];
                }
#pragma unroll
            for (int i = 0; i < D; i++)
#pragma unroll
                for (int c = 0; c < 3; c++)
                    if (n + c < N && bm + 32 * TH * p + lr + 8 * (q + i) < M) Y[at + (int64_t)(8 * (q + i)) * ld + c] = r[i][c];
        }
    };
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const int mp = bm + 32 * TH * p;
        if (mp >= M) break;
        asm volatile("" ::: "memory");
#pragma unroll
        for (int t = 0; t < TH; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                xch[(16 * t + r) * 64 + lane] = acc[0][p * TH + t][r];
                xch[(16 * (TH + t) + r) * 64 + lane] = acc[1][p * TH + t][r];
            }
        asm volatile("" ::: "memory");
#pragma unroll 1
        for (int j = 0; j < (GATED ? 1 : 2); j++) {
            if (act == kActNone) store_vec(p, j, [](float v) { return v; });
            else if (act == kActSilu) store_vec(p, j, [](float v) { return v / (1.0f + __expf(-v)); });
            else store_vec(p, j, [act](float v) { return apply_act(act, v); });
            if (N & 3) store_tail(p, j);
        }
    }
#undef GQ_PUBLISH
}

template <int T, bool BF16, int TM, bool GATED>
int launch_tile(const WregArgs &a, dim3 grid, hipStream_t s) {
    typedef WregTile<T, TM> G;
    static const bool lds_ok = [] {
        return hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_wreg_kernel<T, BF16, TM, GATED>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   G::kLds) == hipSuccess;
    }();
    if (!lds_ok) return fail(GQ_ERR_HIP, "gemm: cannot reserve %d bytes of LDS", G::kLds);
    return launch(gemm_wreg_kernel<T, BF16, TM, GATED>, grid, dim3(256), (size_t)G::kLds, s, a);
}
template <int T>
int launch_type(const WregArgs &a, bool bf16, int tm, bool gated, dim3 grid, hipStream_t s) {
    auto tiled = [&](auto rows) {
        constexpr int TM = decltype(rows)::value;
        if (gated) return launch_tile<T, false, TM, true>(a, grid, s);
        return bf16 ? launch_tile<T, true, TM, false>(a, grid, s) : launch_tile<T, false, TM, false>(a, grid, s);
    };
    return tm == 8 ? tiled(std::integral_constant<int, 8>()) : tm == 6 ? tiled(std::integral_constant<int, 6>()) : tiled(std::integral_constant<int, 4>());
}

}  // namespace

// cols: columns of an output, or of all sums side by side (the epilogue addresses a tile's rows by 32-bit byte offsets)
bool gemm_wreg_supported(int type, int64_t M, int64_t K, int64_t cols) {
    if (type != kQ4_K && type != kQ8_0 && type != kQ4_0 && type != kIQ4_NL) return false;
    return K % kUnit == 0 && K <= (1 << 22) && cols <= (1 << 21) && M <= INT32_MAX && (M + 127) / 128 <= 65535;
}

// x16: 16-bit activations [M, K] (bf16, or fp16 with one scale per row); slices > 1: the sums of each slice to partial[slice][M][columns of
// all matrices], else the finished outputs.
int launch_gemm_wreg(int type, bool bf16, const uint16_t *x16, int64_t M, int64_t K, int count, const MmqSetItem *items, const uint8_t *W2,
                     const float *bias2, int act, const float *residual, const float *rowscale, float *partial, int tm, int slices, hipStream_t s) {
    WregArgs a = {};
    const int wg_rows = W2 ? 128 : 256;
    int64_t wgs = 0, ntot = 0;
    for (int i = 0; i < count; i++) {
        a.W[i] = items[i].W; a.bias[i] = items[i].bias; a.Y[i] = items[i].y;
        a.N[i] = (int)items[i].N; a.wg0[i] = (int)wgs; a.n0[i] = (int)ntot;
        wgs += (items[i].N + wg_rows - 1) / wg_rows;
        ntot += items[i].N;
    }
    if (W2) { a.W[1] = W2; a.bias[1] = bias2; }
    const int units = (int)(K / kUnit), per = (units + slices - 1) / slices;
    if (slices < 1 || (slices - 1) * per >= units || (W2 && (slices != 1 || count != 1 || bf16 || !rowscale)) || (slices > 1 && !partial))
        return fail(GQ_ERR_INVALID, "gemm: %d slices of K = %lld", slices, (long long)K);
    a.count = count; a.ntot = (int)ntot; a.M = (int)M; a.K = (int)K; a.act = act; a.units_per_slice = per;
    a.X = x16; a.row_bytes = (int64_t)gq_row_bytes(type, K);
    a.residual = residual; a.rowscale = rowscale; a.partial = partial;
    const dim3 grid((unsigned)wgs, (unsigned)((M + 32 * tm - 1) / (32 * tm)), (unsigned)slices);
    switch (type) {
    case kQ4_K: return launch_type<kQ4_K>(a, bf16, tm, W2 != nullptr, grid, s);
    case kQ8_0: return launch_type<kQ8_0>(a, bf16, tm, W2 != nullptr, grid, s);
    case kQ4_0: return launch_type<kQ4_0>(a, bf16, tm, W2 != nullptr, grid, s);
    case kIQ4_NL: return launch_type<kIQ4_NL>(a, bf16, tm, W2 != nullptr, grid, s);
    default: return fail(GQ_ERR_NOT_IMPLEMENTED, "qdense: ggml type %d is not implemented", type);
    }
}

}  // namespace gq
