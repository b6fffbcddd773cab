// igemm.hip - products of many activation columns for every weight format on
// gfx950: y[m][n] = dot(row n, column m) on int8 MFMA with exact integers.
//
// Contract: the GGML MUL_MAT semantics of crates/tensor/src/cpu_extra.rs:756-873
// (every column quantized on its own, every output dot_packed of a row and a
// column) and MUL_MAT_ID of cpu_index.rs:169-236, with the dots of
// crates/quant/src/matvec.rs:115-160 (Q8_0) and matvec_extra.rs:174-294 (K
// formats).
//
// Integers.  Per (column, row, block of 256) the K formats need
//   I = sum_j sc_g(j) * q_j * x_j   and, with mins, Mn = sum_g mn_g * bsum_g
// I runs on v_mfma_i32_32x32x32_i8 with int8 planes of sc * q as the weight
// operand, made in registers from the packed weights:
//   Q2_K  sc * q <= 45                      one plane
//   Q3_K  -(sc * q) in -128..124            one plane
//   Q4_K  sc = 8 sh + sl: sh * q, sl * q    two planes, I = 8 A + B
//   Q5_K, Q6_K  p = sc * q: p + 128 split into its high byte and its low byte
//         less 128                          two planes, I = 256 A + B
// so I is the reference's exact i32 whatever the values are (|I| < 2^31: at
// most 4096 * 128 * 256).  Mn runs on v_mfma_f32_32x32x16_f16 (bsum <= 2032 and
// mn <= 63 are exact, the sum stays below 2^24).  Q8_0 takes one MFMA per
// block of 32.
//
// F32 order.  A lane owns (column, row) pairs and adds one term per block in
// block order.  For Q8_0 and Q2_K that is the reference's own sequence, and
// every operation is the reference's, so their results are the reference's bit
// for bit; the others add da * (d * I - dmin * Mn), from 0 in block order, or
// in KS interleaved partial sums where the K split is taken.
#include <type_traits>

#include "rlq_device.hpp"
#include "rlq_internal.hpp"
#include "rlq_layout.hpp"
#include "rlq_q8k.hpp"

namespace rlq {

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------
// Activation image, written once per call.  Columns are grouped in tiles of
// 32, K in chunks of 256 (the last one of a Q8_0 row may be partial, the rest
// zero).  Per (tile, chunk), tile by tile:
//   q     [k-step 8][k half 2][column 32][16 int8]    8 KB
//   d     K formats: [column 32] f32; Q8_0: [k-step 8][column 32] f32    1 KB
//   bsum  (Q2_K, Q4_K, Q5_K) [group half 2][column 32][8 f16]    1 KB
// k-step s, half h, byte t hold block position 32 s + 16 h + t, in the slot
// order of rlq_layout.hpp for Q4_K and Q5_K (one k-step = one sub-block).
// After the tiles, one flag word per (tile, chunk): nonzero marks a data error
// in one of its columns.
// ---------------------------------------------------------------------------
constexpr uint32_t kIgTok = 32;
constexpr uint32_t kIgD = 8192, kIgBsum = 9216;

__host__ __device__ constexpr bool ig_mins(uint32_t t) { return t == kQ2_K || t == kQ4_K || t == kQ5_K; }
__host__ __device__ constexpr bool ig_slots(uint32_t t) { return t == kQ4_K || t == kQ5_K; }
__host__ __device__ constexpr uint32_t ig_pieces(uint32_t t) { return ig_mins(t) ? 10u : 9u; }  // 1 KB each

static uint64_t ig_chunks(uint64_t cols) { return (cols + 255) / 256; }

size_t igemm_image_bytes(uint32_t t, uint64_t tiles, uint64_t cols) {
    return tiles * ig_chunks(cols) * (ig_pieces(t) * 1024ull + 4);
}

struct IgImage {
    uint8_t* img;
    uint32_t* flags;
    uint32_t nchunk;
};
static IgImage ig_carve(void* base, uint32_t t, uint64_t tiles, uint64_t cols) {
    const uint64_t n = tiles * ig_chunks(cols);
    return IgImage{(uint8_t*)base, (uint32_t*)((uint8_t*)base + n * ig_pieces(t) * 1024), (uint32_t)ig_chunks(cols)};
}

// Which matrix and column an image column stands for.  Products of one or more
// matrices whose columns are contiguous: `groups` of cpg columns, tpg tiles
// each; group k uses matrix k / wn2 / r3 * wn2 + k % wn2 (MUL_MAT broadcast).
// Or dealt by igemm_route_kernel (tile_mat non-null): the matrix of each tile,
// kIgZero for products without one (their rows are 0) and columns no product
// uses, kIgNone for unused tiles; per image column its source and its output
// row (-1: none).
constexpr uint32_t kIgNone = ~0u, kIgZero = ~0u - 1;
struct IgMap {
    uint32_t cpg, tpg, wn2, r3;
    const uint32_t* tile_mat;
    const int32_t *src, *row;
};

// Columns of one (tile, chunk): 16 lanes per column, lane r16 holding positions
// 16 r16 .. +15, from f32 rows (x) or from rows of packed Q8_K / Q8_0 blocks
// (taken as given).
template <uint32_t T, bool PACKED>
__global__ __launch_bounds__(512) void igemm_act_kernel(const void* __restrict__ xsrc, IgMap map, uint32_t K,
                                                        uint32_t nchunk, uint8_t* __restrict__ img,
                                                        uint32_t* __restrict__ flags, unsigned long long* err_word,
                                                        const uint32_t* gate) {
    if (gate && *gate) return;
    const uint32_t c = blockIdx.x % nchunk, tile = blockIdx.x / nchunk;
    const uint32_t r16 = threadIdx.x & 15, tok = threadIdx.x >> 4;
    int64_t m = -1;
    if (map.tile_mat) {
        if (map.tile_mat[tile] == kIgNone) {
            if (threadIdx.x == 0) flags[blockIdx.x] = 0;
            return;
        }
        m = map.src[tile * kIgTok + tok];
    } else {
        const uint32_t g = tile / map.tpg, j = tile % map.tpg * kIgTok + tok;
        if (j < map.cpg) m = (int64_t)g * map.cpg + j;
    }
    const uint32_t e0 = c * 256 + r16 * 16;
    const bool live = m >= 0 && e0 < K;
    uint8_t* out = img + (uint64_t)blockIdx.x * (ig_pieces(T) * 1024);
    uint32_t q[4] = {0, 0, 0, 0};
    float d = 0.0f;
    int32_t bsum = 0;
    int bad = 0;
    if constexpr (PACKED) {
        if (live) {
            if constexpr (T == kQ8_0) {
                const uint16_t* b = (const uint16_t*)((const uint8_t*)xsrc + ((uint64_t)m * (K / 32) + e0 / 32) * 34);
                d = half_bits_to_float_exact(b[0]);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    q[k] = (uint32_t)b[1 + 8 * (r16 & 1) + 2 * k] | (uint32_t)b[2 + 8 * (r16 & 1) + 2 * k] << 16;
            } else {
                const uint32_t* b = (const uint32_t*)((const uint8_t*)xsrc + ((uint64_t)m * (K / 256) + c) * 292);
                d = __uint_as_float(b[0]);
#pragma unroll
                for (int k = 0; k < 4; ++k) q[k] = b[1 + 4 * r16 + k];
            }
        }
    } else {
        float v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] = 0.0f;
        if (live) {
            const float4* src = (const float4*)((const float*)xsrc + (uint64_t)m * K + e0);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float4 f = src[k];
                v[4 * k] = f.x, v[4 * k + 1] = f.y, v[4 * k + 2] = f.z, v[4 * k + 3] = f.w;
            }
        }
        if constexpr (T == kQ8_0) {
            uint32_t index;
            const int kind = q8_0_pair16(v, r16 & 1, q, d, index);
            if (kind >= 0) {
                bad = 1;
                if (!(r16 & 1))
                    report_error(err_word, kind == kKindNonFinite
                                               ? error_key((uint64_t)m, kKindNonFinite, (e0 / 32) * 32ull + index)
                                               : error_key((uint64_t)m, kKindScale, e0 / 32));
            }
        } else {
            const Q8KRow o = q8k_row16(v, r16);
#pragma unroll
            for (int k = 0; k < 4; ++k) q[k] = o.q[k];
            d = o.d, bsum = o.bsum;
            if (o.kind >= 0) {
                bad = 1;
                if (r16 == 0)
                    report_error(err_word, o.kind == kKindNonFinite
                                               ? error_key((uint64_t)m, kKindNonFinite, c * 256ull + o.index)
                                               : error_key((uint64_t)m, kKindScale, c));
            }
        }
    }
    const uint4 w = ig_slots(T) ? q45_slots(q, r16 & 1) : make_uint4(q[0], q[1], q[2], q[3]);
    *(uint4*)(out + (r16 >> 1) * 1024 + (r16 & 1) * 512 + tok * 16) = w;
    if constexpr (T == kQ8_0) {
        if (!(r16 & 1)) *(float*)(out + kIgD + (r16 >> 1) * 128 + tok * 4) = d;
    } else {
        if (r16 == 0) *(float*)(out + kIgD + tok * 4) = d;
    }
    if constexpr (ig_mins(T))
        *(_Float16*)(out + kIgBsum + (r16 >> 3) * 512 + tok * 16 + (r16 & 7) * 2) = (_Float16)bsum;
    if (!PACKED) bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) flags[blockIdx.x] = (uint32_t)bad;
}

// ---------------------------------------------------------------------------
// Weight operands
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint4 ig_ld16(const uint8_t* p) { return *(const uint4*)p; }
__device__ __forceinline__ uint32_t ig_word(const uint4& v, int i) {
    return i == 0 ? v.x : (i == 1 ? v.y : (i == 2 ? v.z : v.w));
}
__device__ __forceinline__ uint32_t pk_mul(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t pk_mad(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(
        uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b) + __builtin_bit_cast(u16x2, c)));
}
// Byte B of w in both 16-bit halves, zero- or sign-extended.
template <int B>
__device__ __forceinline__ uint32_t ubyte2(uint32_t w) {
    return __builtin_amdgcn_perm(0u, w, 0x0c000c00u | (uint32_t)B | (uint32_t)B << 16);
}
__device__ __forceinline__ uint32_t pair16(int32_t v) { return (uint32_t)(uint16_t)v | (uint32_t)v << 16; }

// p + 128 of four values (even and odd bytes as 16-bit pairs) -> the two planes
// of p: the high byte, and the low byte with its top bit flipped (p + 128 =
// 256 hi + (lo + 128)).
__device__ __forceinline__ void split_planes(uint32_t e, uint32_t o, int32_t& hi, int32_t& lo) {
    hi = (int32_t)__builtin_amdgcn_perm(o, e, 0x07030501u);
    lo = (int32_t)(__builtin_amdgcn_perm(o, e, 0x06020400u) ^ 0x80808080u);
}

// A 4-bit field of eight mins or scales (bytes of two words) as f16: 0x64kk is
// 1024 + kk.
__device__ __forceinline__ f16x2 ig_byte_half2(uint32_t w, uint32_t sel) {
    return __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, w, sel)) -
           (f16x2){(_Float16)1024.0f, (_Float16)1024.0f};
}

// One format: Raw holds a lane's loaded bytes of one (16-row tile, chunk) pair;
// Pre what a chunk's k-steps share; ops<S> the weight operand of k-step S.
// Lane (ln, kh) of a wave works on row ln % 16 = n of layout tile ln / 16 and k
// half kh.
template <uint32_t T>
struct Ig;

template <>
struct Ig<kQ2_K> {
    static constexpr uint32_t kChunk = kQ2KChunk;
    static constexpr int kPlanes = 1, kShift = 0;
    struct Raw {
        uint4 q[2], sc;
        uint32_t dd;
    };
    struct Pre {
        uint32_t c[4];
    };
    __device__ static void load(Raw& r, const uint8_t* p, uint32_t n, uint32_t kh) {
#pragma unroll
        for (uint32_t g = 0; g < 2; ++g) r.q[g] = ig_ld16(p + (16 * (2 * g + kh) + n) * 16);
        r.sc = ig_ld16(p + 1024 + n * 16);
        r.dd = *(const uint32_t*)(p + 1280 + n * 4);
    }
    __device__ static Pre pre(const Raw& r, uint32_t kh) {
        Pre o;
#pragma unroll
        for (int k = 0; k < 4; ++k) o.c[k] = (ig_word(r.sc, k) >> (8 * kh)) & 0x000f000fu;
        return o;
    }
    // scale index 8 (S / 4) + 2 (S % 4) + kh: word S / 2, half S % 2 of the shifted words
    template <int S>
    __device__ static void ops(const Raw& r, const Pre& c, i32x4& a, i32x4&) {
        const uint32_t w = c.c[S / 2];
        const uint32_t sc = __builtin_amdgcn_perm(0u, w, (S & 1) ? 0x03020302u : 0x01000100u);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            a[i] = (int32_t)pk_mul((ig_word(r.q[S / 4], i) >> (2 * (S % 4))) & 0x03030303u, sc);
    }
    __device__ static f16x8 mins(const Raw& r, uint32_t kh) {
        const uint32_t w0 = ((kh ? r.sc.z : r.sc.x) >> 4) & 0x0f0f0f0fu, w1 = ((kh ? r.sc.w : r.sc.y) >> 4) & 0x0f0f0f0fu;
        f16x8 m;
        const f16x2 a = ig_byte_half2(w0, 0x04010400u), b = ig_byte_half2(w0, 0x04030402u);
        const f16x2 c = ig_byte_half2(w1, 0x04010400u), d = ig_byte_half2(w1, 0x04030402u);
        m[0] = a[0], m[1] = a[1], m[2] = b[0], m[3] = b[1], m[4] = c[0], m[5] = c[1], m[6] = d[0], m[7] = d[1];
        return m;
    }
    __device__ static float d(const Raw& r) { return half_to_float(r.dd); }
    __device__ static float dmin(const Raw& r) { return half_to_float(r.dd >> 16); }
};

template <>
struct Ig<kQ3_K> {
    static constexpr uint32_t kChunk = kQ3KChunk;
    static constexpr int kPlanes = 1, kShift = 0;
    struct Raw {
        uint4 q[2], hm;
        uint32_t s0, s1, s2, d;
    };
    struct Pre {
        uint32_t c[4];
    };
    __device__ static void load(Raw& r, const uint8_t* p, uint32_t n, uint32_t kh) {
#pragma unroll
        for (uint32_t g = 0; g < 2; ++g) r.q[g] = ig_ld16(p + (16 * (2 * g + kh) + n) * 16);
        r.hm = ig_ld16(p + 1024 + n * 32 + 16 * kh);
        const uint32_t* s = (const uint32_t*)(p + 1536 + n * 12);
        r.s0 = s[0], r.s1 = s[1], r.s2 = s[2];
        r.d = *(const uint16_t*)(p + 1728 + n * 2);
    }
    __device__ static Pre pre(const Raw& r, uint32_t kh) {
        // 6-bit scales (matvec_extra.rs:200-210), 0..63 for -32..31
        Pre o;
        o.c[0] = (r.s0 & 0x0f0f0f0fu) | ((r.s2 << 4) & 0x30303030u);
        o.c[1] = (r.s1 & 0x0f0f0f0fu) | ((r.s2 << 2) & 0x30303030u);
        o.c[2] = ((r.s0 >> 4) & 0x0f0f0f0fu) | (r.s2 & 0x30303030u);
        o.c[3] = ((r.s1 >> 4) & 0x0f0f0f0fu) | ((r.s2 >> 2) & 0x30303030u);
#pragma unroll
        for (int k = 0; k < 4; ++k) o.c[k] = (o.c[k] >> (8 * kh)) & 0x003f003fu;
        return o;
    }
    // -(sc * (u - 4)) mod 256 with u = 0..7: u * (32 - s) + 4 (s - 32)
    template <int S>
    __device__ static void ops(const Raw& r, const Pre& c, i32x4& a, i32x4&) {
        const uint32_t s = __builtin_amdgcn_perm(0u, c.c[S / 2], (S & 1) ? 0x03020302u : 0x01000100u);
        const uint32_t neg = __builtin_bit_cast(uint32_t, (u16x2)((u16x2){32, 32} - __builtin_bit_cast(u16x2, s)));
        const uint32_t add = __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, neg) * (u16x2){0xfffc, 0xfffc}));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t low = (ig_word(r.q[S / 4], i) >> (2 * (S % 4))) & 0x03030303u;
            const uint32_t h = ig_word(r.hm, i);
            const uint32_t u = low | ((S < 2 ? h << (2 - S) : h >> (S - 2)) & 0x04040404u);
            const uint32_t e = pk_mad(u & 0x00ff00ffu, neg, add), o = pk_mad((u >> 8) & 0x00ff00ffu, neg, add);
            a[i] = (int32_t)__builtin_amdgcn_perm(o, e, 0x06020400u);
        }
    }
    __device__ static float d(const Raw& r) { return -half_to_float(r.d); }
};

// Q4_K / Q5_K header words: 6-bit scales and mins (get_scale_min_k4,
// crates/quant/src/decode.rs:216-235), four per word.
struct IgHead {
    uint32_t scA, scB, mnA, mnB;
};
__device__ __forceinline__ IgHead ig_head(const uint4& h) {
    IgHead q;
    q.scA = h.y & 0x3f3f3f3fu;
    q.scB = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u);
    q.mnA = h.z & 0x3f3f3f3fu;
    q.mnB = ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u);
    return q;
}
// mins of sub-blocks 4 kh .. 4 kh + 3, each against two 16-value sums
__device__ __forceinline__ f16x8 ig_head_mins(const uint4& h, uint32_t kh) {
    const IgHead q = ig_head(h);
    const uint32_t w = kh ? q.mnB : q.mnA;
    f16x8 m;
    const f16x2 a = ig_byte_half2(w, 0x04010400u), b = ig_byte_half2(w, 0x04030402u);
    m[0] = m[1] = a[0], m[2] = m[3] = a[1], m[4] = m[5] = b[0], m[6] = m[7] = b[1];
    return m;
}

template <>
struct Ig<kQ4_K> {
    static constexpr uint32_t kChunk = kQ4KChunk;
    static constexpr int kPlanes = 2, kShift = 3;
    struct Raw {
        uint4 q[4], h;
    };
    struct Pre {
        uint32_t hi[2], lo[2];
    };
    __device__ static void load(Raw& r, const uint8_t* p, uint32_t n, uint32_t kh) {
#pragma unroll
        for (uint32_t g = 0; g < 4; ++g) r.q[g] = ig_ld16(p + (g / 2) * 1024 + (16 * (2 * (g % 2) + kh) + n) * 16);
        r.h = ig_ld16(p + 2048 + n * 16);
    }
    __device__ static Pre pre(const Raw& r, uint32_t) {
        const IgHead q = ig_head(r.h);
        return Pre{{(q.scA >> 3) & 0x07070707u, (q.scB >> 3) & 0x07070707u}, {q.scA & 0x07070707u, q.scB & 0x07070707u}};
    }
    template <int S>
    __device__ static void ops(const Raw& r, const Pre& c, i32x4& a, i32x4& b) {
        const uint32_t sh = ubyte2<S % 4>(c.hi[S / 4]), sl = ubyte2<S % 4>(c.lo[S / 4]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t w = ig_word(r.q[S / 2], i), q = ((S & 1) ? w >> 4 : w) & 0x0f0f0f0fu;
            a[i] = (int32_t)pk_mul(q, sh);  // byte products <= 105: no carries between bytes
            b[i] = (int32_t)pk_mul(q, sl);
        }
    }
    __device__ static f16x8 mins(const Raw& r, uint32_t kh) { return ig_head_mins(r.h, kh); }
    __device__ static float d(const Raw& r) { return half_to_float(r.h.x); }
    __device__ static float dmin(const Raw& r) { return half_to_float(r.h.x >> 16); }
};

template <>
struct Ig<kQ5_K> {
    static constexpr uint32_t kChunk = kQ5KChunk;
    static constexpr int kPlanes = 2, kShift = 8;
    struct Raw {
        uint4 q[4], qh, h;
    };
    struct Pre {
        uint32_t sc[2];
    };
    __device__ static void load(Raw& r, const uint8_t* p, uint32_t n, uint32_t kh) {
#pragma unroll
        for (uint32_t g = 0; g < 4; ++g) r.q[g] = ig_ld16(p + (g / 2) * 1024 + (16 * (2 * (g % 2) + kh) + n) * 16);
        r.qh = ig_ld16(p + 2048 + n * 32 + 16 * kh);
        r.h = ig_ld16(p + 2560 + n * 16);
    }
    __device__ static Pre pre(const Raw& r, uint32_t) {
        const IgHead q = ig_head(r.h);
        return Pre{{q.scA, q.scB}};
    }
    template <int S>
    __device__ static void ops(const Raw& r, const Pre& c, i32x4& a, i32x4& b) {
        const uint32_t sc = ubyte2<S % 4>(c.sc[S / 4]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t w = ig_word(r.q[S / 2], i), h = ig_word(r.qh, i);
            const uint32_t u = (((S & 1) ? w >> 4 : w) & 0x0f0f0f0fu) | ((S < 4 ? h << (4 - S) : h >> (S - 4)) & 0x10101010u);
            const uint32_t e = pk_mad(u & 0x00ff00ffu, sc, 0x00800080u), o = pk_mad((u >> 8) & 0x00ff00ffu, sc, 0x00800080u);
            int32_t hi, lo;
            split_planes(e, o, hi, lo);
            a[i] = hi, b[i] = lo;
        }
    }
    __device__ static f16x8 mins(const Raw& r, uint32_t kh) { return ig_head_mins(r.h, kh); }
    __device__ static float d(const Raw& r) { return half_to_float(r.h.x); }
    __device__ static float dmin(const Raw& r) { return half_to_float(r.h.x >> 16); }
};

template <>
struct Ig<kQ6_K> {
    static constexpr uint32_t kChunk = kQ6KChunk;
    static constexpr int kPlanes = 2, kShift = 8;
    struct Raw {
        uint4 ql[4], qh[2], sc;
        uint32_t d;
    };
    struct Pre {
        uint32_t c[4];
    };
    __device__ static void load(Raw& r, const uint8_t* p, uint32_t n, uint32_t kh) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) r.ql[k] = ig_ld16(p + kh * 1024 + (16 * k + n) * 16);
#pragma unroll
        for (uint32_t g = 0; g < 2; ++g) r.qh[g] = ig_ld16(p + 2048 + n * 64 + 32 * g + 16 * kh);
        r.sc = ig_ld16(p + 3072 + n * 16);
        r.d = *(const uint16_t*)(p + 3328 + n * 2);
    }
    __device__ static Pre pre(const Raw& r, uint32_t kh) {
        Pre o;
#pragma unroll
        for (int k = 0; k < 4; ++k) o.c[k] = ig_word(r.sc, k) >> (8 * kh);
        return o;
    }
    // k-step S = 4 (half of the block) + side; scale index 2 S + kh
    template <int S>
    __device__ static void ops(const Raw& r, const Pre& c, i32x4& a, i32x4& b) {
        constexpr int kSide = S % 4, kG = S / 4;
        const int32_t s = __builtin_amdgcn_sbfe((int32_t)c.c[S / 2], 16 * (S % 2), 8);
        const uint32_t sc = pair16(s), add = pair16(128 - 32 * s);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t w = ig_word(r.ql[2 * kG + (kSide & 1)], i), h = ig_word(r.qh[kG], i);
            const uint32_t u = ((kSide < 2 ? w : w >> 4) & 0x0f0f0f0fu) |
                               ((kSide < 2 ? h << (4 - 2 * kSide) : h >> (2 * kSide - 4)) & 0x30303030u);
            const uint32_t e = pk_mad(u & 0x00ff00ffu, sc, add), o = pk_mad((u >> 8) & 0x00ff00ffu, sc, add);
            int32_t hi, lo;
            split_planes(e, o, hi, lo);
            a[i] = hi, b[i] = lo;
        }
    }
    __device__ static float d(const Raw& r) { return half_to_float(r.d); }
};

// Q8_0: a chunk of four layout pairs (eight blocks of 32)
struct IgQ8Raw {
    uint4 q[8];
    uint32_t d[4];
};

// ---------------------------------------------------------------------------
// The product
// ---------------------------------------------------------------------------
struct IgArgs {
    const uint8_t* w;
    uint32_t rows, ntiles16, nchunk, npairs;  // npairs: Q8_0 block pairs per row
    const uint8_t* img;
    const uint32_t* flags;
    uint32_t nflags;
    uint32_t NT, MT;  // workgroup tiles along rows and columns
    float* y;
    uint64_t ldy;
    const uint32_t* gate;  // nonzero: the call was refused (igemm_route_kernel)
    IgMap map;
    uint64_t mat_bytes;  // between the stack's matrices
};

__device__ __forceinline__ i32x16 ig_mfma(i32x4 a, i32x4 b, i32x16 c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// global -> LDS, 16 bytes per lane: lane l's 16 bytes at sbase + voff go to LDS
// address lds + 16 l (inline asm: the compiler would wait for every such load
// before any LDS read; ig_barrier orders them)
__device__ __forceinline__ void ig_g2l(const void* sbase, uint32_t voff, uint32_t lds) {
    asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "{m0}"(lds));
}
__device__ __forceinline__ void ig_barrier() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <uint32_t T, int TT, int KS>
constexpr uint32_t ig_lds() {
    return 2u * KS * TT * ig_pieces(T) * 1024u;
}

// A workgroup of four waves: RW = 4 / KS waves side by side along the rows (32
// each) times KS along K; every wave takes TT column tiles of 32.  Wave group
// kg takes chunks kg, kg + KS, ...; its activations are one LDS stage per
// step, filled one step ahead, its weights go straight to registers, also one
// step ahead.
//
// Bound: many columns, the VALU (unpacking the weights, about 11 operations
// per four Q5_K / Q6_K values and wave, and three to five per output and block)
// beside the MFMAs: Q6_K 4096x14336, 1000 columns, 193 us = 610 TOP/s (8.24 ms
// in passes of 8 columns); Q3_K 14336x4096, 512 columns, 87 us.  Few columns:
// the memory latency of each wave's steps, about 1.4 us.
template <uint32_t T, int TT, int KS>
__global__ __launch_bounds__(256, TT == 1 ? 3 : 2) void igemm_kernel(IgArgs g) {
    constexpr int RW = 4 / KS;
    constexpr uint32_t kPieces = ig_pieces(T), kTile = kPieces * 1024, kStage = KS * TT * kTile;
    if (g.gate && *g.gate) return;
    extern __shared__ __align__(16) uint8_t smem[];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t kg = wave / RW, rw = wave % RW, ln = lane & 31, kh = lane >> 5, n = ln & 15;
    // workgroups i, i + 8, ... share an XCD and its L2: each XCD gets a
    // contiguous run of row tiles with all their column tiles
    const uint32_t G = g.NT * g.MT, per = G / 8, rest = G % 8, xcd = blockIdx.x % 8;
    const uint32_t id = xcd * per + (xcd < rest ? xcd : rest) + blockIdx.x / 8;
    const uint32_t nt = id / g.MT, mt = id % g.MT;
    const uint8_t* w = g.w;
    uint32_t mat = 0;
    if (g.map.tile_mat) {
        mat = g.map.tile_mat[mt * TT];
        if (mat == kIgNone) return;
    } else {
        const uint32_t k = mt * TT / g.map.tpg;
        if (mt * TT % g.map.tpg * kIgTok >= g.map.cpg) return;  // a tile of padding
        mat = k / g.map.wn2 / g.map.r3 * g.map.wn2 + k % g.map.wn2;
    }
    if (mat != kIgZero) w += (uint64_t)mat * g.mat_bytes;
    const uint32_t nchunk = g.nchunk, steps = (nchunk + KS - 1) / KS;
    uint32_t t16 = (nt * RW + rw) * 2 + (ln >> 4);
    t16 = t16 < g.ntiles16 ? t16 : g.ntiles16 - 1;  // (rows past the end are never stored)
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
    const uint8_t* act = g.img + (uint64_t)mt * TT * nchunk * kTile;

    auto chunk_of = [&](uint32_t it) {
        const uint32_t c = it * KS + kg;
        return c < nchunk ? c : nchunk - 1;
    };
    // this group's stage of step it: RW waves copy TT * kPieces pieces
    auto issue = [&](uint32_t it) {
        const uint32_t c = chunk_of(it);
        const uint32_t to = lds0 + (it & 1) * kStage + kg * (TT * kTile);
#pragma unroll
        for (uint32_t p = 0; p < (TT * kPieces + RW - 1) / RW; ++p) {
            const uint32_t i = p * RW + rw;
            if ((TT * kPieces) % RW == 0 || i < TT * kPieces)
                ig_g2l(act + ((uint64_t)(i / kPieces) * nchunk + c) * kTile + (i % kPieces) * 1024, lane * 16, to + i * 1024);
        }
    };

    using F = std::conditional_t<T == kQ8_0, IgQ8Raw, typename std::conditional_t<T == kQ8_0, Ig<kQ6_K>, Ig<T>>::Raw>;
    F cur, nxt;
    auto load = [&](F& r, uint32_t it) {
        const uint32_t c = chunk_of(it);
        if constexpr (T == kQ8_0) {
            const uint8_t* base = w + (uint64_t)t16 * g.npairs * kQ80Chunk;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t P = 4 * c + j < g.npairs ? 4 * c + j : g.npairs - 1;
                const uint8_t* p = base + (uint64_t)P * kQ80Chunk;
                r.q[2 * j] = ig_ld16(p + (16 * kh + n) * 16);
                r.q[2 * j + 1] = ig_ld16(p + (16 * (2 + kh) + n) * 16);
                r.d[j] = *(const uint32_t*)(p + 1024 + n * 4);
            }
        } else {
            Ig<T>::load(r, w + ((uint64_t)t16 * nchunk + c) * Ig<T>::kChunk, n, kh);
        }
    };

    issue(0);
    load(cur, 0);
    // a data error in any column: this call writes nothing
    int bad = 0;
    for (uint32_t i = threadIdx.x; i < g.nflags; i += 256) bad |= (int)g.flags[i];
    if (__syncthreads_or(bad)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stage must land before its LDS is released
        return;
    }

    float y[TT][16];
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) y[t][i] = 0.0f;

    for (uint32_t it = 0; it < (mat == kIgZero ? 0 : steps); ++it) {
        ig_barrier();  // stage `it` has landed for every wave; the other one is free
        if (it + 1 < steps) {
            issue(it + 1);
            load(nxt, it + 1);
        }
        const uint32_t c = it * KS + kg;
        if (KS == 1 || c < nchunk) {
            const uint8_t* st = smem + (it & 1) * kStage + kg * (TT * kTile);
            const uint8_t* ab = st + kh * 512 + ln * 16;
            if constexpr (T == kQ8_0) {
#pragma unroll
                for (int s = 0; s < 8; ++s) {
                    if (4 * c + s / 2 >= g.npairs) break;
                    const i32x4 b = __builtin_bit_cast(i32x4, cur.q[s]);
                    const float dw = half_to_float((s & 1) ? cur.d[s / 2] >> 16 : cur.d[s / 2]);
#pragma unroll
                    for (int t = 0; t < TT; ++t) {
                        const i32x4 a = *(const i32x4*)(ab + t * kTile + s * 1024);
                        const i32x16 I = ig_mfma(a, b, (i32x16){});
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const float4 da = *(const float4*)(st + t * kTile + kIgD + s * 128 + (8 * q + 4 * kh) * 4);
                            const float dv[4] = {da.x, da.y, da.z, da.w};
#pragma unroll
                            for (int k = 0; k < 4; ++k) {
                                const float term = (float)I[4 * q + k] * (dw * dv[k]);  // matvec.rs:124-128
                                y[t][4 * q + k] = y[t][4 * q + k] + term;
                            }
                        }
                    }
                }
            } else {
                using W = Ig<T>;
                const typename W::Pre pre = W::pre(cur, kh);
                i32x16 A[TT], B[TT];
#pragma unroll
                for (int t = 0; t < TT; ++t) A[t] = (i32x16){}, B[t] = (i32x16){};
                auto kstep = [&](auto s_) {
                    constexpr int S = decltype(s_)::value;
                    i32x4 wa, wb;
                    W::template ops<S>(cur, pre, wa, wb);
#pragma unroll
                    for (int t = 0; t < TT; ++t) {
                        const i32x4 a = *(const i32x4*)(ab + t * kTile + S * 1024);
                        A[t] = ig_mfma(a, wa, A[t]);
                        if (W::kPlanes == 2) B[t] = ig_mfma(a, wb, B[t]);
                    }
                };
                kstep(std::integral_constant<int, 0>{});
                kstep(std::integral_constant<int, 1>{});
                kstep(std::integral_constant<int, 2>{});
                kstep(std::integral_constant<int, 3>{});
                kstep(std::integral_constant<int, 4>{});
                kstep(std::integral_constant<int, 5>{});
                kstep(std::integral_constant<int, 6>{});
                kstep(std::integral_constant<int, 7>{});
                const float d = W::d(cur);
                float dmin = 0.0f;
                f16x8 mins = {};
                if constexpr (ig_mins(T)) dmin = W::dmin(cur), mins = W::mins(cur, kh);
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    f32x16 mn = {};
                    if constexpr (ig_mins(T)) {
                        const f16x8 bs = *(const f16x8*)(st + t * kTile + kIgBsum + kh * 512 + ln * 16);
                        mn = __builtin_amdgcn_mfma_f32_32x32x16_f16(bs, mins, (f32x16){}, 0, 0, 0);
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float4 da = *(const float4*)(st + t * kTile + kIgD + (8 * q + 4 * kh) * 4);
                        const float dv[4] = {da.x, da.y, da.z, da.w};
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const int i = 4 * q + k;
                            const int32_t I = W::kPlanes == 2 ? (int32_t)(((uint32_t)A[t][i] << W::kShift) + (uint32_t)B[t][i])
                                                              : A[t][i];
                            if constexpr (T == kQ2_K) {  // matvec_extra.rs:193-195
                                const float term = (dv[k] * d) * (float)I - (dv[k] * dmin) * mn[i];
                                y[t][i] = y[t][i] + term;
                            } else {
                                float term = d * (float)I;
                                if constexpr (ig_mins(T)) term = __builtin_fmaf(-dmin, mn[i], term);
                                y[t][i] = __builtin_fmaf(dv[k], term, y[t][i]);
                            }
                        }
                    }
                }
            }
        }
        cur = nxt;
    }

    if (mat == kIgZero) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // its first stage must land before LDS is reused
    if constexpr (KS > 1) {  // the groups' partial sums, added in group order
        __syncthreads();
        float* red = (float*)smem;
        if (kg) {
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) red[(((kg - 1) * RW + rw) * TT + t) * 1024 + i * 64 + lane] = y[t][i];
        }
        __syncthreads();
        if (kg) return;
#pragma unroll
        for (int k = 0; k < KS - 1; ++k)
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) y[t][i] += red[((k * RW + rw) * TT + t) * 1024 + i * 64 + lane];
    }
    const uint32_t row = (nt * RW + rw) * 32 + ln;
    if (row >= g.rows) return;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const uint32_t tile = mt * TT + t;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t tok = 8 * (i / 4) + 4 * kh + (i % 4);
            if (g.map.tile_mat) {
                const int32_t r = g.map.row[tile * kIgTok + tok];
                if (r >= 0) g.y[(uint64_t)r * g.ldy + row] = y[t][i];
            } else {
                const uint32_t k = tile / g.map.tpg, j = tile % g.map.tpg * kIgTok + tok;
                if (j < g.map.cpg) g.y[((uint64_t)k * g.map.cpg + j) * g.ldy + row] = y[t][i];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Launch
// ---------------------------------------------------------------------------
template <uint32_t T, int TT, int KS>
static hipError_t ig_launch_one(IgArgs g, uint32_t tiles, hipStream_t s) {
    constexpr int RW = 4 / KS;
    g.NT = (g.rows + 32 * RW - 1) / (32 * RW);
    g.MT = tiles / TT;
    const uint64_t grid = (uint64_t)g.NT * g.MT;
    if (grid == 0 || grid > 0x7fffffffull) return hipErrorInvalidValue;
    static LdsLimit lim;
    constexpr uint32_t lds = ig_lds<T, TT, KS>();
    const hipError_t e = lim.raise((const void*)igemm_kernel<T, TT, KS>, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((igemm_kernel<T, TT, KS>), dim3((unsigned)grid), dim3(256), lds, s, g);
    return hipGetLastError();
}

// Shape of the workgroups, by the number of (32 rows x 32 columns) tiles.
// Up to 512 of them leave most SIMDs idle: four waves split K (1024x4096, 77
// columns, Q4_K / Q5_K / Q6_K: 13.4 / 16.2 / 14.2 us against 26 / 36 / 29
// without); up to 1100, two do (14336x4096, 64 columns: 21.9 / 31.5 / 29.9
// against 28.7 / 39 / 31.8).  Beyond, a wave takes two column tiles, so that
// the weights it unpacks serve both (14336x4096, 512 columns, Q3_K / Q5_K /
// Q6_K: 87 / 116 / 109 us against 124 / 147 / 153), with K still split in two
// up to 3000 tiles (4096x4096, 512 columns: Q3_K 36.1 against 41.5, Q6_K 38.8
// against 42.1).  Q4_K unpacks in fewest steps and keeps one column tile up to
// 4000 tiles (37 us against 45); Q8_0 and Q2_K cannot split K, and Q8_0, whose
// work is the f32 terms, keeps one column tile throughout (124 us against 137).
// pairs: two neighbouring column tiles may share a wave.
template <uint32_t T>
static hipError_t ig_launch(const IgArgs& g, uint32_t tiles, bool pairs, hipStream_t s) {
    const uint64_t live = g.map.tile_mat ? tiles : (uint64_t)tiles / g.map.tpg * ((g.map.cpg + kIgTok - 1) / kIgTok);
    const uint64_t n = (uint64_t)((g.rows + 31) / 32) * live;
    if constexpr (T == kQ8_0) {
        return ig_launch_one<T, 1, 1>(g, tiles, s);
    } else {
        if constexpr (T != kQ2_K) {
            if (n <= 512) return ig_launch_one<T, 1, 4>(g, tiles, s);
            if (n <= 1100) return ig_launch_one<T, 1, 2>(g, tiles, s);
            if (T != kQ4_K && n <= 3000 && pairs) return ig_launch_one<T, 2, T == kQ4_K ? 1 : 2>(g, tiles, s);
        }
        if (!pairs || n <= (T == kQ2_K || T == kQ4_K ? 4000 : 0)) return ig_launch_one<T, 1, 1>(g, tiles, s);
        return ig_launch_one<T, 2, 1>(g, tiles, s);
    }
}

template <uint32_t T>
static hipError_t ig_act(const void* x, bool packed, const IgMap& map, uint32_t K, uint32_t tiles, const IgImage& im,
                         unsigned long long* err, const uint32_t* gate, hipStream_t s) {
    const dim3 grid(tiles * im.nchunk);
    if (!packed)
        hipLaunchKernelGGL((igemm_act_kernel<T, false>), grid, dim3(512), 0, s, x, map, K, im.nchunk, im.img, im.flags, err,
                           gate);
    else if constexpr (!ig_mins(T))
        hipLaunchKernelGGL((igemm_act_kernel<T, true>), grid, dim3(512), 0, s, x, map, K, im.nchunk, im.img, im.flags, err,
                           gate);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

// The image of the columns, then the product.
static hipError_t ig_run(uint32_t t, const uint8_t* w, uint64_t rows, uint64_t cols, uint64_t mat_bytes, const void* x,
                         bool packed, const IgMap& map, uint32_t tiles, bool pairs, const IgImage& im, float* y, uint64_t ldy,
                         const uint32_t* gate, unsigned long long* err, hipStream_t s) {
    if (rows == 0 || cols == 0 || cols % (t == kQ8_0 ? 32 : 256) || tiles == 0 || rows > 0x7fffffffull ||
        cols > (1u << 30) || tiles > (1u << 20) || (uint64_t)tiles * im.nchunk > 0x7fffffffull)
        return hipErrorInvalidValue;
    IgArgs g{};
    g.w = w;
    g.rows = (uint32_t)rows;
    g.ntiles16 = (uint32_t)layout_tiles(rows);
    g.nchunk = im.nchunk;
    g.npairs = t == kQ8_0 ? (uint32_t)layout_chunks_per_tile(t, cols) : 0;
    g.img = im.img;
    g.flags = im.flags;
    g.nflags = tiles * im.nchunk;
    g.y = y;
    g.ldy = ldy;
    g.gate = gate;
    g.map = map;
    g.mat_bytes = mat_bytes;
    hipError_t e;
#define RLQ_IG(TYPE)                                                                        \
    case TYPE:                                                                              \
        e = ig_act<TYPE>(x, packed, map, (uint32_t)cols, tiles, im, err, gate, s);          \
        return e != hipSuccess ? e : ig_launch<TYPE>(g, tiles, pairs, s);
    switch (t) {
        RLQ_IG(kQ8_0)
        RLQ_IG(kQ2_K)
        RLQ_IG(kQ3_K)
        RLQ_IG(kQ4_K)
        RLQ_IG(kQ5_K)
        RLQ_IG(kQ6_K)
        default: return hipErrorInvalidValue;
    }
#undef RLQ_IG
}

// Column tiles of one group: from three on an even number, so that pairs of them
// can share a wave.
static uint64_t ig_group_tiles(uint64_t cpg) {
    const uint64_t t = (cpg + kIgTok - 1) / kIgTok;
    return t > 2 ? (t + 1) & ~1ull : t;
}

size_t igemm_bytes(uint32_t t, uint64_t groups, uint64_t cpg, uint64_t cols) {
    return igemm_image_bytes(t, groups * ig_group_tiles(cpg), cols);
}

hipError_t launch_igemm(uint32_t t, const uint8_t* w, uint64_t rows, uint64_t cols, const void* x, bool packed,
                        const IgStack& st, float* y, uint64_t ldy, void* scratch, unsigned long long* err_word,
                        hipStream_t s) {
    const uint64_t tpg = ig_group_tiles(st.cpg), tiles = tpg * st.groups;
    if (st.cpg == 0 || st.groups == 0 || tiles > (1u << 20)) return hipErrorInvalidValue;
    IgMap map{};
    map.cpg = (uint32_t)st.cpg, map.tpg = (uint32_t)tpg, map.wn2 = (uint32_t)st.wn2, map.r3 = (uint32_t)st.r3;
    return ig_run(t, w, rows, cols, st.mat_bytes, x, packed, map, (uint32_t)tiles, tpg % 2 == 0,
                  ig_carve(scratch, t, tiles, cols), y, ldy, nullptr, err_word, s);
}

// ---------------------------------------------------------------------------
// MUL_MAT_ID
// ---------------------------------------------------------------------------

// Checks the ids (the first one outside [-1, mats) refuses the call) and deals
// the products to image columns, matrix after matrix, each from a whole group
// of `unit` tiles on (one workgroup); then the products without a matrix (id
// -1) and the columns that no product uses, which are quantized for their
// errors only.  Where inside its run a product lands depends on the order of
// the LDS atomics; its result does not.  One workgroup: the counts stay in LDS,
// and a launch of its own costs less than a grid-wide sum.
__global__ __launch_bounds__(1024) void igemm_route_kernel(IgRoute r, uint32_t tiles, uint32_t unit,
                                                           uint32_t* __restrict__ tile_mat, int32_t* __restrict__ src,
                                                           int32_t* __restrict__ row, uint32_t* __restrict__ gate,
                                                           unsigned long long* err_word) {
    __shared__ uint32_t count[kIgMaxMats + 1], first[kIgMaxMats + 2], used[kIgMaxColumns / 32];
    __shared__ unsigned long long bad;
    const uint32_t tid = threadIdx.x, group = unit * kIgTok;
    if (tid == 0) bad = ~0ull;
    for (uint32_t i = tid; i <= r.mats; i += 1024) count[i] = 0;
    for (uint32_t i = tid; i < (r.columns + 31) / 32; i += 1024) used[i] = 0;
    for (uint32_t i = tid; i < tiles * kIgTok; i += 1024) src[i] = row[i] = -1;
    __syncthreads();
    auto column_of = [&](uint32_t i) { return i / r.slots * r.ncols + i % r.slots % r.ncols; };
    for (uint32_t i = tid; i < r.products; i += 1024) {
        const int32_t id = r.ids[i];
        if (id < -1 || id >= (int32_t)r.mats) {
            atomicMin(&bad, (unsigned long long)i);
        } else {
            atomicAdd(&count[id < 0 ? r.mats : (uint32_t)id], 1u);
            if (id >= 0) atomicOr(&used[column_of(i) / 32], 1u << (column_of(i) % 32));
        }
    }
    __syncthreads();
    if (tid == 0) {
        *gate = bad != ~0ull;
        if (bad != ~0ull) report_error(err_word, bounds_key(bad));
    }
    if (bad != ~0ull) return;
    auto is_used = [&](uint32_t c) { return (used[c / 32] >> (c % 32)) & 1u; };
    for (uint32_t c = tid; c < r.columns; c += 1024)
        if (!is_used(c)) atomicAdd(&count[r.mats], 1u);
    __syncthreads();
    if (tid == 0) {
        uint32_t t = 0;
        for (uint32_t m = 0; m <= r.mats; ++m) {
            first[m] = t;
            t += (count[m] + group - 1) / group * unit;
        }
        first[r.mats + 1] = t;
    }
    __syncthreads();
    for (uint32_t t = tid; t < tiles; t += 1024) {
        uint32_t m = 0;
        while (m <= r.mats && first[m + 1] <= t) ++m;
        tile_mat[t] = m > r.mats ? kIgNone : (m == r.mats ? kIgZero : m);
    }
    __syncthreads();
    for (uint32_t i = tid; i <= r.mats; i += 1024) count[i] = 0;
    __syncthreads();
    for (uint32_t i = tid; i < r.products; i += 1024) {
        const int32_t id = r.ids[i];
        const uint32_t m = id < 0 ? r.mats : (uint32_t)id;
        const uint32_t at = first[m] * kIgTok + atomicAdd(&count[m], 1u);
        row[at] = (int32_t)i;
        if (id >= 0) src[at] = (int32_t)column_of(i);
    }
    for (uint32_t c = tid; c < r.columns; c += 1024)
        if (!is_used(c)) src[first[r.mats] * kIgTok + atomicAdd(&count[r.mats], 1u)] = (int32_t)c;
}

// From 128 products a matrix on, two column tiles of one matrix share a wave.
static uint32_t ig_unit(const IgRoute& r) { return r.products / r.mats >= 128 ? 2 : 1; }
// Upper bound of the tiles: every run in use may leave its last group short.
static uint64_t ig_route_tiles(const IgRoute& r) {
    const uint64_t u = ig_unit(r), n = (uint64_t)r.products + r.columns;
    return (n / (u * kIgTok) + (r.products < r.mats ? r.products : r.mats) + 1) * u;
}

size_t igemm_ids_bytes(uint32_t t, uint64_t cols, const IgRoute& r) {
    const uint64_t tiles = ig_route_tiles(r);
    return igemm_image_bytes(t, tiles, cols) + 4 + tiles * (4 + kIgTok * 8);
}

hipError_t launch_igemm_ids(uint32_t t, const uint8_t* w, uint64_t rows, uint64_t cols, uint64_t mat_bytes, const void* x,
                            bool packed, const IgRoute& r, float* y, uint64_t ldy, void* scratch,
                            unsigned long long* err_word, hipStream_t s) {
    const uint64_t tiles = ig_route_tiles(r);
    if (r.products == 0 || r.mats == 0 || r.mats > kIgMaxMats || r.columns > kIgMaxColumns || tiles > (1u << 20))
        return hipErrorInvalidValue;
    const IgImage im = ig_carve(scratch, t, tiles, cols);
    uint32_t* gate = im.flags + tiles * im.nchunk;
    uint32_t* tile_mat = gate + 1;
    int32_t *src = (int32_t*)(tile_mat + tiles), *row = src + tiles * kIgTok;
    const uint32_t unit = ig_unit(r);
    hipLaunchKernelGGL(igemm_route_kernel, dim3(1), dim3(1024), 0, s, r, (uint32_t)tiles, unit, tile_mat, src, row, gate,
                       err_word);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    IgMap map{};
    map.tile_mat = tile_mat, map.src = src, map.row = row;
    return ig_run(t, w, rows, cols, mat_bytes, x, packed, map, (uint32_t)tiles, unit == 2, im, y, ldy, gate, err_word, s);
}

}  // namespace rlq
