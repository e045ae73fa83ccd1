// ggml.Dequantize (ml/ggml/dequant.go:39-54) and ggml.EmbeddingLookupDecomposed
// (ml/ggml/gather.go:21-49) as gfx950 kernels.  Both are bit-exact with the reference
// arithmetic and bound by the fp32 writes (4 bytes out per 0.56-1.06 bytes in).
#include "blocks.hpp"
#include "common.hpp"

#include <algorithm>
#include <climits>

namespace gq {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
struct __attribute__((packed, aligned(2))) u32_a2 { uint32_t v; };
__device__ __forceinline__ uint32_t load_u32_a2(const uint8_t *p) { return reinterpret_cast<const u32_a2 *>(p)->v; }

// The bytes that four consecutive values (quad `q`: values 4 q .. 4 q + 3 of a run of blocks at `row`) come from, and their
// exact value: the arithmetic of dequant16<T>, four values at a time.
template <int T> struct Quad;

template <> struct Quad<kQ8_0> {
    uint32_t d, c;
    __device__ __forceinline__ void load(const uint8_t *row, int64_t q) {
        const uint8_t *b = row + (q >> 3) * 34;
        d = load_u16(b);
        c = load_u32_a2(b + 2 + 4 * (int)(q & 7));
    }
    __device__ __forceinline__ f32x4 value(int64_t) const {
        const float s = half_bits_to_float(d);
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = (float)(int32_t)(int8_t)(c >> (8 * j)) * s;  // ml/ggml/dequant.go:74
        return v;
    }
};

template <int T> struct QuadNibble {  // Q4_0, IQ4_NL: values 0..15 in the low nibbles, 16..31 in the high ones
    uint32_t d, c;
    __device__ __forceinline__ void load(const uint8_t *row, int64_t q) {
        const uint8_t *b = row + (q >> 3) * 18;
        d = load_u16(b);
        c = load_u32_a2(b + 2 + 4 * (int)(q & 3));
    }
    __device__ __forceinline__ f32x4 value(int64_t q) const {
        const float s = half_bits_to_float(d);
        const uint32_t n = c >> (4 * (int)((q >> 2) & 1));
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t nib = (n >> (8 * j)) & 0x0Fu;
            if constexpr (T == kQ4_0) v[j] = ((float)nib - 8.0f) * s;  // ml/ggml/dequant.go:108-112
            else v[j] = iq4nl_value(nib) * s;                         // ml/ggml/dequant.go:130-133
        }
        return v;
    }
};
template <> struct Quad<kQ4_0> : QuadNibble<kQ4_0> {};
template <> struct Quad<kIQ4_NL> : QuadNibble<kIQ4_NL> {};

template <> struct Quad<kQ4_K> {
    uint4 hd;
    uint32_t c;
    __device__ __forceinline__ void load(const uint8_t *row, int64_t q) {
        const uint8_t *sb = row + (q >> 6) * 144;
        hd = *reinterpret_cast<const uint4 *>(sb);
        c = *reinterpret_cast<const uint32_t *>(sb + 16 + 32 * (int)((q >> 4) & 3) + 4 * (int)(q & 7));
    }
    __device__ __forceinline__ f32x4 value(int64_t q) const {
        uint32_t sc, mn;
        q4k_scale_min(hd.y, hd.z, hd.w, (int)((q >> 3) & 7), sc, mn);
        const float ds = half_bits_to_float(hd.x & 0xFFFFu) * (float)sc;
        const float dm = half_bits_to_float(hd.x >> 16) * (float)mn;
        const uint32_t n = c >> (4 * (int)((q >> 3) & 1));
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = ds * (float)((n >> (8 * j)) & 0x0Fu) - dm;
        return v;
    }
};

template <> struct Quad<kQ6_K> {  // (block layout: see dequant16<kQ6_K>)
    uint32_t d, ql, qh;
    int sc;
    __device__ __forceinline__ void load(const uint8_t *row, int64_t q) {
        const uint8_t *sb = row + (q >> 6) * 210;
        const int l = (int)(q & 63), h = l >> 5, qd = (l >> 3) & 3;
        ql = load_u32_a2(sb + 64 * h + 32 * (qd & 1) + 4 * (l & 7));
        qh = load_u32_a2(sb + 128 + 32 * h + 4 * (l & 7));
        sc = (int)(int8_t)sb[192 + (l >> 2)];
        d = load_u16(sb + 208);
    }
    __device__ __forceinline__ f32x4 value(int64_t q) const {
        const int qd = (int)((q >> 3) & 3), nsh = (qd >> 1) * 4, hsh = 2 * qd;
        const float ds = half_bits_to_float(d) * (float)sc;
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t lo = (ql >> (8 * j + nsh)) & 0x0Fu, hi = (qh >> (8 * j + hsh)) & 0x03u;
            v[j] = ds * (float)((int)(lo | (hi << 4)) - 32);
        }
        return v;
    }
};

// A workgroup writes U x 1024 consecutive values of one output row, a lane four of them per store: a wavefront's store
// covers 1 KB without gaps and its loads one super-block (or eight blocks).  All loads of a lane's U quads are issued before
// the first value is formed.  Bound by the writes: 14336 x 4096 values of Q4_K take 51.6 us (5.2 TB/s), with NT 39.7 us
// (6.7 TB/s), where 16 values per lane in four stores 64 bytes apart took 85 us (3.1 TB/s).
// For gq_dequantize the whole matrix is one row (blocks follow each other without gaps and so do the values); a gather takes
// one row per index.
template <int T, int U, bool NT>
__global__ __launch_bounds__(256) void dequant_rows_kernel(const uint8_t *__restrict__ W, float *__restrict__ out, int64_t rows,
                                                           int64_t quads_per_row, uint32_t rows_per_wg, uint32_t chunks, int64_t row_bytes, const int32_t *__restrict__ indices,
                                                           int64_t vocab, int32_t *__restrict__ err_flag, uint32_t first_wg) {
    int64_t r = 0, src = 0;
    const uint32_t wg = first_wg + blockIdx.x;
    uint32_t chunk = wg, lane = threadIdx.x;
    bool bad = false;
    if (indices) {  // gather: row r of the output is row indices[r] of the table
        const uint32_t group = wg / chunks;
        chunk = wg - group * chunks;
        r = group;
        if (rows_per_wg > 1) {  // (rows of fewer than 256 quads: several of them to a workgroup; U is 1 then)
            const uint32_t sub = lane / (uint32_t)quads_per_row;
            r = (int64_t)group * rows_per_wg + sub;
            lane -= sub * (uint32_t)quads_per_row;
            if (sub >= rows_per_wg || r >= rows) return;
        }
        src = indices[r];
        bad = src < 0 || src >= vocab;
        if (bad) {
            src = 0;
            if (chunk == 0 && lane == 0 && err_flag != nullptr) *err_flag = 1;
        }
    }
    const uint8_t *row = W + src * row_bytes;
    f32x4 *o = reinterpret_cast<f32x4 *>(out) + r * quads_per_row;
    const int64_t q0 = (int64_t)chunk * (256 * U) + lane;
    Quad<T> b[U];
#pragma unroll
    for (int u = 0; u < U; u++) b[u].load(row, min(q0 + 256 * u, quads_per_row - 1));
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int64_t q = q0 + 256 * u;
        if (q >= quads_per_row) continue;
        f32x4 v = b[u].value(q);
        if (bad) v = f32x4{__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf("")};
        if constexpr (NT) __builtin_nontemporal_store(v, o + q);
        else o[q] = v;
    }
}

// Outputs from this size on are written around the caches (NT).  They would push themselves out again before the next
// operation reads them: dequantisation and an addition over its result 133.6 against 138.3 us at 235 MB; at 67 MB, which the
// 256 MB of Infinity Cache keep, 39.6 against 37.8.
constexpr int64_t kStreamBytes = (int64_t)128 << 20;

template <int T>
int launch_rows(const uint8_t *W, float *out, int64_t N, int64_t K, const int32_t *indices, int64_t vocab, int32_t *err_flag, hipStream_t s) {
    const int64_t row_bytes = (K / Geom<T>::vpb) * Geom<T>::bpb;
    const int64_t rows = indices ? N : 1, quads = (indices ? K : N * K) / 4;
    // (four quads per lane once that still leaves every CU two workgroups; below that more workgroups answer sooner)
    const bool wide = quads >= 1024 && rows * ((quads + 1023) / 1024) >= 2 * (int64_t)device_cu_count();
    const int64_t chunks = wide ? (quads + 1023) / 1024 : (quads + 255) / 256, per_wg = quads >= 256 || !indices ? 1 : 256 / quads;
    const int64_t groups = (rows + per_wg - 1) / per_wg;
    if (chunks > INT_MAX / groups) return fail(GQ_ERR_NOT_IMPLEMENTED, "dequantize: %lld x %lld values in one call", (long long)N, (long long)K);
    // (a launch takes fewer than 2^32 threads: a gather of more than 2^24 rows of 1024 values, 64 GB of them, needs several)
    constexpr int64_t kMaxWgs = ((int64_t)1 << 24) - 1;
    auto go = [&](auto kernel) {
        for (int64_t first = 0; first < groups * chunks; first += kMaxWgs)
            if (int rc = launch(kernel, dim3((unsigned)std::min(groups * chunks - first, kMaxWgs)), dim3(256), 0, s, W, out, rows, quads, (uint32_t)per_wg,
                                (uint32_t)chunks, row_bytes, indices, vocab, err_flag, (uint32_t)first))
                return rc;
        return (int)GQ_OK;
    };
    if (!wide) return go(dequant_rows_kernel<T, 1, false>);
    return rows * quads * 16 >= kStreamBytes ? go(dequant_rows_kernel<T, 4, true>) : go(dequant_rows_kernel<T, 4, false>);
}

int dispatch_rows(int type, const uint8_t *W, float *out, int64_t N, int64_t K, const int32_t *indices, int64_t vocab, int32_t *err_flag,
                  hipStream_t s) {
    switch (type) {
    case kQ8_0: return launch_rows<kQ8_0>(W, out, N, K, indices, vocab, err_flag, s);
    case kQ4_0: return launch_rows<kQ4_0>(W, out, N, K, indices, vocab, err_flag, s);
    case kIQ4_NL: return launch_rows<kIQ4_NL>(W, out, N, K, indices, vocab, err_flag, s);
    case kQ4_K: return launch_rows<kQ4_K>(W, out, N, K, indices, vocab, err_flag, s);
    case kQ6_K: return launch_rows<kQ6_K>(W, out, N, K, indices, vocab, err_flag, s);
    default: return fail(GQ_ERR_NOT_IMPLEMENTED, "dequantize: ggml type %d is not implemented", type);
    }
}

}  // namespace

int launch_dequantize(int type, const uint8_t *W, int64_t N, int64_t K, float *out, hipStream_t s) {
    return dispatch_rows(type, W, out, N, K, nullptr, 0, nullptr, s);
}

int launch_embedding_lookup(int type, const uint8_t *table, int64_t vocab, int64_t K, const int32_t *idx,
                            int64_t count, float *out, int32_t *err_flag, hipStream_t s) {
    return dispatch_rows(type, table, out, count, K, idx, vocab, err_flag, s);
}

}  // namespace gq
