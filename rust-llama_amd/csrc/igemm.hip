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
    return tiles * ig_chunks(cols) * (ig_pieces(t) * 1024ull + 4) + 4;  // (the image's flags, and one for all)
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
// each; group k uses matrix k / wn2 / r3 * wn2 + k % wn2 (MUL_MAT broadcast; one:
// a single group, which needs no divisions).
// Or dealt by igemm_route_kernel (tile_mat non-null): the matrix of each tile
// (low half; high half: its live columns, which come first), kIgZero for
// products without one (their rows are 0) and columns no product uses, kIgNone
// for unused tiles; per image column its source and its output
// row (-1: none).
constexpr uint32_t kIgNone = ~0u, kIgZero = ~0u - 1;
struct IgMap {
    uint32_t cpg, tpg, wn2, r3, one;
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
        const uint32_t g = map.one ? 0 : tile / map.tpg, j = (tile - g * map.tpg) * kIgTok + tok;
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

// One flag for all of many: every workgroup of the product reads them, so past
// kIgFlags of them (131072 columns of 512 values) a launch that folds them costs
// less (Q2_K 1024x1024, 100000 columns 553 -> 364 us; Q6_K 4096x4096, 32768 columns
// 2142 -> 2037).
constexpr uint64_t kIgFlags = 8192;
__global__ __launch_bounds__(1024) void igemm_flags_kernel(const uint32_t* __restrict__ flags, uint64_t n,
                                                           uint32_t* __restrict__ all) {
    int bad = 0;
    for (uint64_t i = threadIdx.x; i < n; i += 1024) bad |= (int)flags[i];
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) *all = (uint32_t)bad;
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

// One format: Raw holds a lane's loaded bytes of one (16-row tile, chunk) pair:
// head loads the scales, refill<S> the pieces that no k-step after S uses (kLoads
// of them in 16 bytes each, not next to each other); Pre is
// what a chunk's k-steps share; ops<S> makes the weight operand of k-step S.
// Lane (ln, kh) of a wave works on row ln % 16 = n of layout tile ln / 16 and k
// half kh.
template <uint32_t T>
struct Ig;

template <>
struct Ig<kQ2_K> {
    static constexpr uint32_t kChunk = kQ2KChunk;
    static constexpr int kLoads = 3;
    static constexpr int kPlanes = 1, kShift = 0;
    struct Raw {
        uint4 q[2], sc;
        uint32_t dd;
    };
    struct Pre {
        uint32_t c[4];
    };
    __device__ static void head(Raw& r, const uint8_t* p, uint32_t n) {
        r.sc = ig_ld16(p + 1024 + n * 16);
        r.dd = *(const uint32_t*)(p + 1280 + n * 4);
    }
    template <int S>
    __device__ static void refill(Raw& r, const uint8_t* p, uint32_t n, uint32_t kh) {
        if (S % 4 == 3) r.q[S / 4] = ig_ld16(p + (16 * (2 * (S / 4) + kh) + n) * 16);
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
    static constexpr int kLoads = 3;
    static constexpr int kPlanes = 1, kShift = 0;
    struct Raw {
        uint4 q[2], hm;
        uint32_t s0, s1, s2, d;
    };
    struct Pre {
        uint32_t c[4];
    };
    template <int S>
    __device__ static void refill(Raw& r, const uint8_t* p, uint32_t n, uint32_t kh) {
        if (S % 4 == 3) r.q[S / 4] = ig_ld16(p + (16 * (2 * (S / 4) + kh) + n) * 16);
        if (S == 7) r.hm = ig_ld16(p + 1024 + n * 32 + 16 * kh);
    }
    __device__ static void head(Raw& r, const uint8_t* p, uint32_t n) {
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
    static constexpr int kLoads = 5;
    static constexpr int kPlanes = 2, kShift = 3;
    struct Raw {
        uint4 q[4], h;
    };
    struct Pre {
        uint32_t hi[2], lo[2];
    };
    __device__ static void head(Raw& r, const uint8_t* p, uint32_t n) { r.h = ig_ld16(p + 2048 + n * 16); }
    template <int S>
    __device__ static void refill(Raw& r, const uint8_t* p, uint32_t n, uint32_t kh) {
        if (S & 1) r.q[S / 2] = ig_ld16(p + (S / 4) * 1024 + (16 * (2 * (S / 2 % 2) + kh) + n) * 16);
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
    static constexpr int kLoads = 6;
    static constexpr int kPlanes = 2, kShift = 8;
    struct Raw {
        uint4 q[4], qh, h;
    };
    struct Pre {
        uint32_t sc[2];
    };
    __device__ static void head(Raw& r, const uint8_t* p, uint32_t n) { r.h = ig_ld16(p + 2560 + n * 16); }
    template <int S>
    __device__ static void refill(Raw& r, const uint8_t* p, uint32_t n, uint32_t kh) {
        if (S & 1) r.q[S / 2] = ig_ld16(p + (S / 4) * 1024 + (16 * (2 * (S / 2 % 2) + kh) + n) * 16);
        if (S == 7) r.qh = ig_ld16(p + 2048 + n * 32 + 16 * kh);
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
    static constexpr int kLoads = 7;
    static constexpr int kPlanes = 2, kShift = 8;
    struct Raw {
        uint4 ql[4], qh[2], sc;
        uint32_t d;
    };
    struct Pre {
        uint32_t c[4];
    };
    __device__ static void head(Raw& r, const uint8_t* p, uint32_t n) {
        r.sc = ig_ld16(p + 3072 + n * 16);
        r.d = *(const uint16_t*)(p + 3328 + n * 2);
    }
    template <int S>
    __device__ static void refill(Raw& r, const uint8_t* p, uint32_t n, uint32_t kh) {
        if (S % 4 >= 2) r.ql[2 * (S / 4) + S % 2] = ig_ld16(p + kh * 1024 + (16 * (2 * (S / 4) + S % 2) + n) * 16);
        if (S % 4 == 3) r.qh[S / 4] = ig_ld16(p + 2048 + n * 64 + 32 * (S / 4) + 16 * kh);
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

template <int S>
using IgStep = std::integral_constant<int, S>;
// f(IgStep<0>), ..., f(IgStep<7>)
template <typename F>
__device__ __forceinline__ void ig_steps(F&& f) {
    f(IgStep<0>{}), f(IgStep<1>{}), f(IgStep<2>{}), f(IgStep<3>{});
    f(IgStep<4>{}), f(IgStep<5>{}), f(IgStep<6>{}), f(IgStep<7>{});
}
template <uint32_t T>
__device__ __forceinline__ void ig_load(typename Ig<T>::Raw& r, const uint8_t* p, uint32_t n, uint32_t kh) {
    ig_steps([&](auto s) { Ig<T>::template refill<decltype(s)::value>(r, p, n, kh); });
    Ig<T>::head(r, p, n);
}

// Q8_0: a chunk of four layout pairs (eight blocks of 32)
template <uint32_t T>
struct IgRaw {
    using Raw = typename Ig<T>::Raw;
};
template <>
struct IgRaw<kQ8_0> {
    struct Raw {
        uint4 q[8];
        uint32_t d[4];
    };
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
    uint32_t* refused;   // set to whether a data error suppressed every output, or null
};
// A data error in any column (`bad`: one that this thread saw): the call writes
// nothing.
__device__ __forceinline__ bool ig_refused(const IgArgs& g, int bad) {
    bad = __syncthreads_or(bad);
    if (g.refused && blockIdx.x == 0 && threadIdx.x == 0) *g.refused = (uint32_t)(bad != 0);
    return bad != 0;
}

__device__ __forceinline__ i32x16 ig_mfma(i32x4 a, i32x4 b, i32x16 c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// global -> LDS, 16 bytes per lane: lane l's 16 bytes at sbase + voff go to LDS
// address lds + 16 l (inline asm: the compiler would wait for every such load
// before any LDS read; ig_barrier orders them)
__device__ __forceinline__ void ig_g2l(const void* sbase, uint32_t voff, uint32_t lds) {
    asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "{m0}"(lds));
}
// Barrier after which a stage has landed for every wave: at most N of a wave's
// loads, all younger than the stage's, are still in flight.
template <int N>
__device__ __forceinline__ void ig_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// LDS writes of every wave are visible after it; loads to registers stay in flight.
__device__ __forceinline__ void ig_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <uint32_t T, int TT, int KS>
constexpr uint32_t ig_lds() {
    return 2u * KS * TT * ig_pieces(T) * 1024u;
}

// One block's term before the activation scale, from its integers.
template <uint32_t T>
__device__ __forceinline__ float ig_term(int32_t A, int32_t B, float mn, float d, float dmin) {
    const int32_t I = Ig<T>::kPlanes == 2 ? (int32_t)(((uint32_t)A << Ig<T>::kShift) + (uint32_t)B) : A;
    const float t = d * (float)I;
    return ig_mins(T) ? __builtin_fmaf(-dmin, mn, t) : t;
}
// Q2_K's whole term, in the reference's operations (matvec_extra.rs:193-195).
__device__ __forceinline__ float ig_q2_term(int32_t I, float mn, float da, float d, float dmin) {
    return (da * d) * (float)I - (da * dmin) * mn;
}

// The matrix of column tile `tile` (kIgNone: nothing to do), and how many of its
// columns are live.
__device__ __forceinline__ uint32_t ig_matrix(const IgMap& map, uint32_t tile, uint32_t& live) {
    if (map.tile_mat) {
        const uint32_t v = map.tile_mat[tile];
        live = kIgTok;
        if (v >= kIgZero) return v;
        live = v >> 16;
        return v & 0xffffu;
    }
    const uint32_t k = map.one ? 0 : tile / map.tpg, j = (tile - k * map.tpg) * kIgTok;
    if (j >= map.cpg) return kIgNone;  // a tile of padding
    live = map.cpg - j < kIgTok ? map.cpg - j : kIgTok;
    if (map.one) return 0;
    return k / map.wn2 / map.r3 * map.wn2 + k % map.wn2;
}
// Stores value i of a lane's sixteen (column 8 (i / 4) + 4 kh + i % 4 of the tile) of
// weight row `row`: the live columns of a group follow each other.
struct IgStore {
    float* y;             // column 0 of the tile, or output row 0
    uint32_t live;
    const int32_t* rows;  // the output row of each column (-1: none), or null
};
__device__ __forceinline__ IgStore ig_store(const IgArgs& g, uint32_t tile, uint32_t row) {
    const IgMap& map = g.map;
    if (map.tile_mat) return IgStore{g.y + row, 0, map.row + tile * kIgTok};
    const uint32_t k = map.one ? 0 : tile / map.tpg, j = (tile - k * map.tpg) * kIgTok;
    return IgStore{g.y + ((uint64_t)k * map.cpg + j) * g.ldy + row, map.cpg > j ? map.cpg - j : 0, nullptr};
}
__device__ __forceinline__ void ig_put(const IgStore& o, uint64_t ldy, uint32_t i, uint32_t kh, float v) {
    const uint32_t tok = 8 * (i / 4) + 4 * kh + (i % 4);
    if (o.rows) {
        const int32_t r = o.rows[tok];
        if (r >= 0) o.y[(uint64_t)r * ldy] = v;
    } else if (tok < o.live) {
        o.y[tok * ldy] = v;
    }
}

// A workgroup of four waves: RW = 4 / KS waves side by side along the rows (32
// each) times KS along K; every wave takes TT column tiles of 32.  Wave group
// kg takes chunks kg, kg + KS, ...; its activations are one LDS stage per
// step, filled one step ahead, its weights go straight to the registers that
// the k-steps free, so that three waves fit a SIMD (the barrier before a stage
// leaves those younger loads in flight).  With a second set of weight registers
// and two waves: Q4_K 4096x14336, 1000 columns 193 us against 176, Q5_K
// 14336x4096, 512 columns 122 against 111, Q2_K 80 against 77, Q6_K the same.
//
// Bound: many columns, the VALU (unpacking the weights, about 11 operations
// per four Q5_K / Q6_K values and wave, and three to five per output and block):
// Q6_K 4096x14336, 1000 columns, 201 us = 584 TOP/s (8.24 ms in passes of 8
// columns) with the VALU issuing during 68 % of the cycles, the MFMAs busy during
// 29 %, both during 17 %.
// (Four column tiles a wave, one wave per SIMD, unpack half as often but hide
// nothing: 220 us against 222, Q5_K 220 against 210.)  A step takes at
// least the memory latency, about 1.4 us: few tiles have a kernel of their own.
template <uint32_t T, int TT, int KS>
__global__ __launch_bounds__(256, 3) void igemm_kernel(IgArgs g) {
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
    uint32_t live;  // (every column is multiplied)
    const uint32_t mat = ig_matrix(g.map, mt * TT, live);
    if (mat == kIgNone) return;
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

    using F = typename IgRaw<T>::Raw;
    F cur, nxt;  // nxt: Q8_0 only
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
            ig_load<T>(r, w + ((uint64_t)t16 * nchunk + c) * Ig<T>::kChunk, n, kh);
        }
    };

    issue(0);
    load(cur, 0);
    int bad = 0;
    for (uint32_t i = threadIdx.x; i < g.nflags; i += 256) bad |= (int)g.flags[i];
    if (ig_refused(g, bad)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stage must land before its LDS is released
        return;
    }

    float y[TT][16];
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) y[t][i] = 0.0f;

    const uint32_t run = mat == kIgZero ? 0 : steps;
    if constexpr (T == kQ8_0) {
        for (uint32_t it = 0; it < run; ++it) {
            ig_barrier<0>();  // stage `it` has landed for every wave; the other one is free
            if (it + 1 < steps) {
                issue(it + 1);
                load(nxt, it + 1);
            }
            const uint8_t* st = smem + (it & 1) * kStage;
            const uint8_t* ab = st + kh * 512 + ln * 16;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                if (4 * it + s / 2 >= g.npairs) break;
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
            cur = nxt;
        }
    } else {
        using W = Ig<T>;
        // one step; more: the next step's stage is issued first, its weights
        // follow the last use of the registers they take
        auto step = [&](auto more_, uint32_t it) {
            constexpr bool more = decltype(more_)::value;
            const uint8_t* wn = w + ((uint64_t)t16 * nchunk + chunk_of(it + 1)) * W::kChunk;
            if (more) {
                issue(it + 1);
                asm volatile("" ::: "memory");  // no load of the next weights before the stage's
            }
            const uint8_t* st = smem + (it & 1) * kStage + kg * (TT * kTile);
            const uint8_t* ab = st + kh * 512 + ln * 16;
            const typename W::Pre pre = W::pre(cur, kh);
            const float d = W::d(cur);
            float dmin = 0.0f;
            f16x8 mins = {};
            if constexpr (ig_mins(T)) dmin = W::dmin(cur), mins = W::mins(cur, kh);
            if (more) W::head(cur, wn, n);
            i32x16 A[TT], B[TT];
#pragma unroll
            for (int t = 0; t < TT; ++t) A[t] = (i32x16){}, B[t] = (i32x16){};
            ig_steps([&](auto s_) {
                constexpr int S = decltype(s_)::value;
                i32x4 wa, wb;
                W::template ops<S>(cur, pre, wa, wb);
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    const i32x4 a = *(const i32x4*)(ab + t * kTile + S * 1024);
                    A[t] = ig_mfma(a, wa, A[t]);
                    if (W::kPlanes == 2) B[t] = ig_mfma(a, wb, B[t]);
                }
                if (more) W::template refill<S>(cur, wn, n, kh);
            });
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
                        if constexpr (T == kQ2_K)
                            y[t][i] = y[t][i] + ig_q2_term(A[t][i], mn[i], dv[k], d, dmin);
                        else
                            y[t][i] = __builtin_fmaf(dv[k], ig_term<T>(A[t][i], B[t][i], mn[i], d, dmin), y[t][i]);
                    }
                }
            }
        };
        for (uint32_t it = 0; it + 1 < run; ++it) {
            if (it == 0) ig_barrier<0>();
            else ig_barrier<W::kLoads>();
            step(std::true_type{}, it);
        }
        if (run) {
            ig_barrier<0>();
            if (KS == 1 || (run - 1) * KS + kg < nchunk) step(std::false_type{}, run - 1);
        }
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
        const IgStore o = ig_store(g, mt * TT + t, row);
#pragma unroll
        for (int i = 0; i < 16; ++i) ig_put(o, g.ldy, i, kh, y[t][i]);
    }
}

// Few tiles: one (32 rows x 32 columns) tile per workgroup, its chunks dealt to
// KS waves.  Nothing is staged: a wave reads its weights and activations
// straight into the registers that the k-steps free, one chunk ahead (the
// activations half a chunk), so the
// waves run apart and only meet to add up.  Q2_K parks each chunk's terms in
// LDS and every wave adds its share of the tile in block order.
//
// Bound: memory latency (a wave has two to four chunks), then the activations'
// way from L2 (8 KB a chunk and tile; lanes of dead columns read column 0).
// 14336x4096, 16 columns: Q4_K 13.9 us with the image's kernel (24.3 with staged
// activations and K split in two, 23.8 in decode passes), Q2_K 12.8 (25.4, 32.3);
// 4096x14336: Q2_K 15.5 (68, 123), whose staged kernel cannot split K.
template <uint32_t T, int KS>
__global__ __launch_bounds__(64 * KS) __attribute__((amdgpu_waves_per_eu(KS == 4 ? 3 : 4))) void igemm_few_kernel(IgArgs g) {
    constexpr uint32_t kTile = ig_pieces(T) * 1024;
    constexpr int kOwn = 16 / KS;  // accumulators of the tile that a wave adds up
    using W = Ig<T>;
    if (g.gate && *g.gate) return;
    __shared__ float part[(T == kQ2_K ? 2 : 1) * KS][16][64];
    __shared__ __align__(16) float das[KS][32];
    const uint32_t lane = threadIdx.x & 63, kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t ln = lane & 31, kh = lane >> 5, n = ln & 15, nchunk = g.nchunk;
    const uint32_t G = g.NT * g.MT, per = G / 8, rest = G % 8, xcd = blockIdx.x % 8;
    const uint32_t id = xcd * per + (xcd < rest ? xcd : rest) + blockIdx.x / 8;
    const uint32_t nt = id / g.MT, mt = id % g.MT;
    uint32_t live;
    const uint32_t mat = ig_matrix(g.map, mt, live);
    if (mat == kIgNone) return;
    const bool zero = mat == kIgZero;
    uint32_t t16 = nt * 2 + (ln >> 4);
    t16 = t16 < g.ntiles16 ? t16 : g.ntiles16 - 1;
    const uint8_t* wt = g.w + (zero ? 0 : (uint64_t)mat * g.mat_bytes) + (uint64_t)t16 * nchunk * W::kChunk;
    const uint32_t col = ln < live ? ln : 0;
    const uint8_t* at = g.img + (uint64_t)mt * nchunk * kTile;

    typename W::Raw r;
    i32x4 act[4];
    float da = 0.0f;
    f16x8 bs = {};
    auto load_act = [&](int s, uint32_t c) {
        act[s % 4] = *(const i32x4*)(at + (uint64_t)c * kTile + s * 1024 + kh * 512 + col * 16);
    };
    auto load_scales = [&](uint32_t c) {
        da = *(const float*)(at + (uint64_t)c * kTile + kIgD + col * 4);
        if (ig_mins(T)) bs = *(const f16x8*)(at + (uint64_t)c * kTile + kIgBsum + kh * 512 + col * 16);
    };
    const uint32_t c0 = kg < nchunk ? kg : nchunk - 1;
#pragma unroll
    for (int s = 0; s < 4; ++s) load_act(s, c0);
    load_scales(c0);
    ig_load<T>(r, wt + (uint64_t)c0 * W::kChunk, n, kh);
    int bad = 0;
    for (uint32_t i = threadIdx.x; i < g.nflags; i += 64 * KS) bad |= (int)g.flags[i];
    if (ig_refused(g, bad)) return;

    float y[16], own[kOwn];
#pragma unroll
    for (int i = 0; i < 16; ++i) y[i] = 0.0f;
#pragma unroll
    for (int i = 0; i < kOwn; ++i) own[i] = 0.0f;
    // one chunk; more: the loads of chunk c + KS follow the last use of what
    // they replace.  Q2_K: y is the chunk's term, otherwise the running sum.
    auto chunk = [&](auto more_, uint32_t c) {
        constexpr bool more = decltype(more_)::value;
        const uint8_t* wn = wt + (uint64_t)(c + KS) * W::kChunk;
        const typename W::Pre pre = W::pre(r, kh);
        const float d = W::d(r);
        float dmin = 0.0f;
        f16x8 mins = {};
        if constexpr (ig_mins(T)) dmin = W::dmin(r), mins = W::mins(r, kh);
        if (kh == 0) das[kg][ln] = da;
        if (more) W::head(r, wn, n);
        i32x16 A = {}, B = {};
        ig_steps([&](auto s_) {
            constexpr int S = decltype(s_)::value;
            i32x4 wa, wb;
            W::template ops<S>(r, pre, wa, wb);
            A = ig_mfma(act[S % 4], wa, A);
            if (W::kPlanes == 2) B = ig_mfma(act[S % 4], wb, B);
            if (more) W::template refill<S>(r, wn, n, kh);
            if (S < 4) load_act(S + 4, c);
            else if (more) load_act(S - 4, c + KS);
        });
        f32x16 mn = {};
        if constexpr (ig_mins(T)) mn = __builtin_amdgcn_mfma_f32_32x32x16_f16(bs, mins, (f32x16){}, 0, 0, 0);
        if (more) load_scales(c + KS);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 dq = *(const float4*)&das[kg][8 * q + 4 * kh];
            const float dv[4] = {dq.x, dq.y, dq.z, dq.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = 4 * q + k;
                if constexpr (T == kQ2_K) y[i] = ig_q2_term(A[i], mn[i], dv[k], d, dmin);
                else y[i] = __builtin_fmaf(dv[k], ig_term<T>(A[i], B[i], mn[i], d, dmin), y[i]);
            }
        }
    };
    if constexpr (T == kQ2_K) {
        for (uint32_t it = 0; it * KS < nchunk && !zero; ++it) {
            const uint32_t c = it * KS + kg;
            float(*p)[16][64] = part + (it & 1) * KS;
            if (c < nchunk) {
                if (c + KS < nchunk) chunk(std::true_type{}, c);
                else chunk(std::false_type{}, c);
#pragma unroll
                for (int i = 0; i < 16; ++i) p[kg][i][lane] = y[i];
            }
            ig_lds_barrier();  // (two buffers: the next step's terms go to the other one)
            const uint32_t m = nchunk - it * KS < KS ? nchunk - it * KS : KS;
            for (uint32_t j = 0; j < m; ++j)
#pragma unroll
                for (int i = 0; i < kOwn; ++i) own[i] = own[i] + p[j][kg * kOwn + i][lane];
        }
    } else {
        if (!zero && kg < nchunk) {
            uint32_t c = kg;
            for (; c + KS < nchunk; c += KS) chunk(std::true_type{}, c);
            chunk(std::false_type{}, c);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) part[kg][i][lane] = y[i];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < KS; ++j)
#pragma unroll
            for (int i = 0; i < kOwn; ++i) own[i] += part[j][kg * kOwn + i][lane];
    }
    const uint32_t row = nt * 32 + ln;
    if (row >= g.rows) return;
    const IgStore o = ig_store(g, mt, row);
#pragma unroll
    for (int k = 0; k < kOwn; ++k) ig_put(o, g.ldy, kg * kOwn + k, kh, own[k]);
}

// Few tiles of Q8_0: eight waves take one pair of blocks each per step, three
// steps ahead (19 registers a step), park both blocks' terms in LDS, and every
// wave adds two of the tile's sixteen accumulators over the step's sixteen
// blocks in order.  One buffer and two barriers a step, so that two workgroups
// fit a CU's LDS.  Bound: a step's LDS traffic (128 KB a workgroup) and f32 terms,
// 1.2 to 1.4 us.  4096x4096, 16 columns: 16.8 us (46 staged, 27 in decode passes);
// 4096x14336: 39 (138, 187).
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void igemm_few_q8_kernel(IgArgs g) {
    constexpr int KS = 8, D = 3;
    constexpr uint32_t kTile = ig_pieces(kQ8_0) * 1024;
    if (g.gate && *g.gate) return;
    __shared__ __align__(16) float2 part[2 * KS][8][64];  // [block][accumulator pair][lane]
    __shared__ __align__(16) float das[KS][2][32];
    const uint32_t lane = threadIdx.x & 63, kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t ln = lane & 31, kh = lane >> 5, n = ln & 15, npairs = g.npairs;
    const uint32_t G = g.NT * g.MT, per = G / 8, rest = G % 8, xcd = blockIdx.x % 8;
    const uint32_t id = xcd * per + (xcd < rest ? xcd : rest) + blockIdx.x / 8;
    const uint32_t nt = id / g.MT, mt = id % g.MT;
    uint32_t live;
    const uint32_t mat = ig_matrix(g.map, mt, live);
    if (mat == kIgNone) return;
    const bool zero = mat == kIgZero;
    uint32_t t16 = nt * 2 + (ln >> 4);
    t16 = t16 < g.ntiles16 ? t16 : g.ntiles16 - 1;
    const uint8_t* wt = g.w + (zero ? 0 : (uint64_t)mat * g.mat_bytes) + (uint64_t)t16 * npairs * kQ80Chunk;
    const uint32_t col = ln < live ? ln : 0, steps = zero ? 0 : (npairs + KS - 1) / KS;
    const uint8_t* at = g.img + (uint64_t)mt * g.nchunk * kTile;

    struct Step {
        i32x4 w[2], a[2];
        uint32_t dw;
        float da[2];
    } buf[D];
    auto load = [&](Step& q, uint32_t it) {
        const uint32_t want = it * KS + kg, P = want < npairs ? want : npairs - 1;
        const uint8_t* p = wt + (uint64_t)P * kQ80Chunk;
        const uint8_t* x = at + (uint64_t)(P / 4) * kTile;
#pragma unroll
        for (uint32_t b = 0; b < 2; ++b) {
            const uint32_t s = 2 * (P % 4) + b;
            q.w[b] = *(const i32x4*)(p + (16 * (2 * b + kh) + n) * 16);
            q.a[b] = *(const i32x4*)(x + s * 1024 + kh * 512 + col * 16);
            q.da[b] = *(const float*)(x + kIgD + s * 128 + col * 4);
        }
        q.dw = *(const uint32_t*)(p + 1024 + n * 4);
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load(buf[d], d);
    int bad = 0;
    for (uint32_t i = threadIdx.x; i < g.nflags; i += 64 * KS) bad |= (int)g.flags[i];
    if (ig_refused(g, bad)) return;

    float own[2] = {0.0f, 0.0f};
    auto step = [&](Step& q, uint32_t it) {
        if (it * KS + kg < npairs) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                if (kh == 0) das[kg][b][ln] = q.da[b];
                const float dw = half_to_float(b ? q.dw >> 16 : q.dw);
                const i32x16 I = ig_mfma(q.a[b], q.w[b], (i32x16){});
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float4 dq = *(const float4*)&das[kg][b][8 * k + 4 * kh];  // matvec.rs:124-128
                    part[2 * kg + b][2 * k][lane] = make_float2((float)I[4 * k] * (dw * dq.x), (float)I[4 * k + 1] * (dw * dq.y));
                    part[2 * kg + b][2 * k + 1][lane] =
                        make_float2((float)I[4 * k + 2] * (dw * dq.z), (float)I[4 * k + 3] * (dw * dq.w));
                }
            }
        }
        load(q, it + D);
        ig_lds_barrier();
        const uint32_t left = npairs - it * KS, m = 2 * (left < KS ? left : KS);
        if (m == 2 * KS) {
#pragma unroll
            for (int j = 0; j < 2 * KS; ++j) {
                const float2 t = part[j][kg][lane];
                own[0] = own[0] + t.x, own[1] = own[1] + t.y;
            }
        } else {
            for (uint32_t j = 0; j < m; ++j) {
                const float2 t = part[j][kg][lane];
                own[0] = own[0] + t.x, own[1] = own[1] + t.y;
            }
        }
        ig_lds_barrier();
    };
    for (uint32_t it = 0; it < steps; it += D) {
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (it + d < steps) step(buf[d], it + d);
    }
    const uint32_t row = nt * 32 + ln;
    if (row >= g.rows) return;
    const IgStore o = ig_store(g, mt, row);
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) ig_put(o, g.ldy, kg * 2 + k, kh, own[k]);
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
    if (grid == 0 || grid * 256 > 0xffffffffull) return hipErrorInvalidValue;
    static LdsLimit lim;
    constexpr uint32_t lds = ig_lds<T, TT, KS>();
    const hipError_t e = lim.raise((const void*)igemm_kernel<T, TT, KS>, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((igemm_kernel<T, TT, KS>), dim3((unsigned)grid), dim3(256), lds, s, g);
    return hipGetLastError();
}

template <uint32_t T, int KS>
static hipError_t ig_launch_few(IgArgs g, uint32_t tiles, hipStream_t s) {
    g.NT = (g.rows + 31) / 32;
    g.MT = tiles;
    const uint64_t grid = (uint64_t)g.NT * g.MT;
    if (grid == 0 || grid * 64 * KS > 0xffffffffull) return hipErrorInvalidValue;
    if constexpr (T == kQ8_0) hipLaunchKernelGGL(igemm_few_q8_kernel, dim3((unsigned)grid), dim3(512), 0, s, g);
    else hipLaunchKernelGGL((igemm_few_kernel<T, KS>), dim3((unsigned)grid), dim3(64 * KS), 0, s, g);
    return hipGetLastError();
}

// The kernel, by the number n of (32 rows x 32 columns) tiles; us of both sides
// at 4096 columns unless said otherwise.  pairs: two neighbouring column tiles
// may share a wave.
//  - One tile per workgroup while that still gives few workgroups.  16 waves to
//    160 tiles (4096x14336, 16 columns: Q4_K 16.3 against 18.7 with 8, Q2_K 15.5
//    against 18.0), 8 to 512 (14336 rows, 16 columns: Q4_K 13.9 against 15.6 with
//    4), then 4 until the kernel below, whose waves share activations, is
//    faster: 1700 tiles of Q3_K and Q6_K (4096 rows, 384 columns = 1536: 35.2
//    against 36.3 and 38.1 against 40.1; 512 columns = 2048: 43.6 against 38.1 and
//    47.2 against 42.0), 2048 of Q2_K (32.5 against 34.7; 14336 rows, 192 columns
//    = 2688: 38.0 against 38.6), 2700 of Q5_K (59.3 against 80; 256 columns = 3584:
//    76.8 against 67.4), 3500 of Q4_K (43.0 against 45.8; 53.0 against 56.1), 2000
//    of it with fewer chunks than waves (256 values a row: 2048 tiles 13.2 against
//    11.2, 28672 rows, 96 columns = 2688: 17.7 against 12.5; 768 values: 19.0 against
//    16.6), and 4000 where column tiles cannot be paired.  Q8_0 to 1024 (4096 rows, 256
//    columns: 40 against 48; 384 = 1536: 56 against 50; 14336 values a row, 256: 108
//    against 137), and to 1800 tiles of MUL_MAT_ID, whose count includes unused ones
//    (8 experts of 4096x14336, 10 products: 1152, 110 against 163; of 4096x4096, 79
//    tokens: 1664, 45 against 53; 128 of 512x2048, 206 tokens: 2256, 64 against 58).
//  - Beyond, two column tiles a wave, so that the weights it unpacks serve both
//    (14336 rows, 512 columns, Q3_K / Q5_K / Q6_K: 87 / 116 / 109 against 124 / 147 /
//    153), with K split in two to 3000 tiles (4096 rows, 512 columns: Q3_K 36.1
//    against 41.5, Q6_K 38.8 against 42.1).  Q2_K, whose unpacking is short, from
//    4000 tiles on; Q8_0, whose work is the f32 terms, never (124 against 137).
template <uint32_t T>
static hipError_t ig_launch(const IgArgs& g, uint32_t tiles, bool pairs, hipStream_t s) {
    const uint64_t live = g.map.tile_mat ? tiles : (uint64_t)tiles / g.map.tpg * ((g.map.cpg + kIgTok - 1) / kIgTok);
    const uint64_t n = (uint64_t)((g.rows + 31) / 32) * live;
    if constexpr (T == kQ8_0) {
        return n <= (g.map.tile_mat ? 1800 : 1024) ? ig_launch_few<T, 8>(g, tiles, s) : ig_launch_one<T, 1, 1>(g, tiles, s);
    } else {
        constexpr uint64_t kFew = T == kQ2_K ? 2048 : (T == kQ4_K ? 3500 : (T == kQ5_K ? 2700 : 1700));
        if (n <= 160 && g.nchunk >= 16) return ig_launch_few<T, 16>(g, tiles, s);
        if (n <= 512) return ig_launch_few<T, 8>(g, tiles, s);
        const uint64_t few = !pairs ? 4000 : (T == kQ4_K && g.nchunk < 4 ? 2000 : kFew);
        if (n <= few) return ig_launch_few<T, 4>(g, tiles, s);
        if (!pairs || (T == kQ2_K && n <= 4000)) return ig_launch_one<T, 1, 1>(g, tiles, s);
        if constexpr (T == kQ3_K || T == kQ6_K)
            if (n <= 3000) return ig_launch_one<T, 2, 2>(g, tiles, s);
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

// Whether the launches stay below 2^32 threads (HIP runs a part of a larger grid
// and reports nothing): 512 for each record of the image, 256 for each tile of
// 128 rows x 32 columns (or of 64 x 64) of the product.  igemm_few_kernel's
// grids are bounded by the tiles that it is chosen for.
static bool ig_takes(uint64_t rows, uint64_t cols, uint64_t tiles) {
    return rows <= 0x7fffffffull && cols <= (1u << 30) && tiles <= (1u << 20) &&
           tiles * ig_chunks(cols) * 512 <= 0xffffffffull && (rows + 127) / 128 * tiles * 256 <= 0xffffffffull;
}

// The image of the columns, then the product.
static hipError_t ig_run(uint32_t t, const uint8_t* w, uint64_t rows, uint64_t cols, uint64_t mat_bytes, const void* x,
                         bool packed, const IgMap& map, uint32_t tiles, bool pairs, const IgImage& im, float* y, uint64_t ldy,
                         const uint32_t* gate, unsigned long long* err, hipStream_t s, uint32_t* refused = nullptr) {
    if (rows == 0 || cols == 0 || cols % (t == kQ8_0 ? 32 : 256) || tiles == 0 || !ig_takes(rows, cols, tiles))
        return hipErrorInvalidValue;
    IgArgs g{};
    g.w = w;
    g.rows = (uint32_t)rows;
    g.ntiles16 = (uint32_t)layout_tiles(rows);
    g.nchunk = im.nchunk;
    g.npairs = t == kQ8_0 ? (uint32_t)layout_chunks_per_tile(t, cols) : 0;
    g.img = im.img;
    g.flags = im.flags;
    const uint64_t nflags = (uint64_t)tiles * im.nchunk;
    const bool fold = nflags > kIgFlags && !gate;
    g.nflags = fold ? 1 : (uint32_t)nflags;
    if (fold) g.flags = im.flags + nflags;
    g.y = y;
    g.ldy = ldy;
    g.gate = gate;
    g.map = map;
    g.mat_bytes = mat_bytes;
    g.refused = refused;
    hipError_t e;
#define RLQ_IG(TYPE)                                                                        \
    case TYPE:                                                                              \
        e = ig_act<TYPE>(x, packed, map, (uint32_t)cols, tiles, im, err, gate, s);          \
        if (e == hipSuccess && fold) {                                                      \
            hipLaunchKernelGGL(igemm_flags_kernel, dim3(1), dim3(1024), 0, s, im.flags, nflags, im.flags + nflags); \
            e = hipGetLastError();                                                          \
        }                                                                                   \
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

bool igemm_takes(uint64_t rows, uint64_t groups, uint64_t cpg, uint64_t cols) {
    return ig_takes(rows, cols, groups * ig_group_tiles(cpg));
}

size_t igemm_bytes(uint32_t t, uint64_t groups, uint64_t cpg, uint64_t cols) {
    return igemm_image_bytes(t, groups * ig_group_tiles(cpg), cols);
}

hipError_t launch_igemm(uint32_t t, const uint8_t* w, uint64_t rows, uint64_t cols, const void* x, bool packed,
                        const IgStack& st, float* y, uint64_t ldy, void* scratch, unsigned long long* err_word,
                        hipStream_t s, uint32_t* refused) {
    const uint64_t tpg = ig_group_tiles(st.cpg), tiles = tpg * st.groups;
    if (st.cpg == 0 || st.groups == 0 || !ig_takes(rows, cols, tiles)) return hipErrorInvalidValue;
    IgMap map{};
    map.cpg = (uint32_t)st.cpg, map.tpg = (uint32_t)tpg, map.wn2 = (uint32_t)st.wn2, map.r3 = (uint32_t)st.r3;
    map.one = st.groups == 1;
    return ig_run(t, w, rows, cols, st.mat_bytes, x, packed, map, (uint32_t)tiles, tpg % 2 == 0,
                  ig_carve(scratch, t, tiles, cols), y, ldy, nullptr, err_word, s, refused);
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
        uint32_t v = kIgNone;
        if (m == r.mats) {
            v = kIgZero;
        } else if (m < r.mats) {  // (a group's second tile may be empty: one column, of zeros)
            const uint32_t at = (t - first[m]) * kIgTok, left = count[m] > at ? count[m] - at : 1;
            v = m | (left < kIgTok ? left : kIgTok) << 16;
        }
        tile_mat[t] = v;
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

bool igemm_ids_takes(uint64_t rows, uint64_t cols, const IgRoute& r) {
    return r.products > 0 && r.mats > 0 && r.mats <= kIgMaxMats && r.columns <= kIgMaxColumns &&
           ig_takes(rows, cols, ig_route_tiles(r));
}

size_t igemm_ids_bytes(uint32_t t, uint64_t cols, const IgRoute& r) {
    const uint64_t tiles = ig_route_tiles(r);
    return igemm_image_bytes(t, tiles, cols) + 4 + tiles * (4 + kIgTok * 8);
}

hipError_t launch_igemm_ids(uint32_t t, const uint8_t* w, uint64_t rows, uint64_t cols, uint64_t mat_bytes, const void* x,
                            bool packed, const IgRoute& r, float* y, uint64_t ldy, void* scratch,
                            unsigned long long* err_word, hipStream_t s) {
    if (!igemm_ids_takes(rows, cols, r)) return hipErrorInvalidValue;
    const uint64_t tiles = ig_route_tiles(r);
    const IgImage im = ig_carve(scratch, t, tiles, cols);
    uint32_t* gate = im.flags + tiles * im.nchunk + 1;
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
