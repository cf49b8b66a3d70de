// lp_gemm_fact.hip - tiled bf16-MFMA product of fp32 activation rows with F32 /
// F16 / BF16 / Q2_K / Q3_K / Q5_K weights (prompt rows), at fp32 precision.
//
// These types multiply fp32 activations (dot_row_f32 .. dot_row_q5_k,
// src/matmul.cpp:63-314). The matrix unit's fp32 products run at a sixteenth of
// its bf16 rate, so an fp32 value is split into the three bf16 pieces it is the
// exact sum of, x = x1 + x2 + x3, and multiplied piece by piece with fp32
// accumulation:
//   BF16        w is one piece:             3 products
//   Q2_K, Q3_K  scale times code (<= 45, <= 128) is a bf16 value; d once per 256
//   Q5_K        the 5-bit code is one; d * scale once per 32 (on the VALU)
//   F16         w = w1 + w2 (8 + 3 bits):   5 products (x3 w2 is below 2^-24)
//   F32         w = w1 + w2 + w3:           6 products (the rest below 2^-24)
// The min terms of Q2_K / Q5_K (-dmin * m * sum x) take the sums of x per 16 / 32
// elements, split the same way, in one small product per 32 elements. Every 64
// elements the fp32 accumulators are added to 64-bit sums, so the result is nearer
// to the exact product than the fp32 dots of the GEMV kernels are.
//
// Work split: that of the int8 product (lp_gemm_i8t.hip). A stage is 64 elements:
// the activation tile is split and the weight tile decoded once per workgroup into
// LDS in operand order ([32 rows][16 k][half][row][8 bf16]); the next stage is in
// registers meanwhile.
//
// What bounds it (BF16, N 4096 K 4096 M 512, 87 us, 590 TFLOP/s of bf16 products, the
// GEMVs 1175 us, one pass over the weights per 4 rows; matrix unit busy 21 %): loads are
// hidden behind the products; splitting x and writing its planes (58 us alone) and the
// products (72 - 80 us alone) follow each other in every wave. Large: M 2048 N 14336
// 15890 -> 884 us, Q5_K N 4096 K 14336 M 2048 95144 -> 1230. Normwise errors against
// 64-bit sums 5e-8 .. 1e-7, the GEMVs' 0.7e-7 .. 3e-7.
#include <hip/hip_runtime.h>

#include "lp_dequant_one.h"
#include "lp_internal.h"

namespace lp {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));
typedef short s4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));

constexpr int kH = 528;                  // 32 rows x 16 B, padded: the 8 pieces of a row written together hit distinct banks
constexpr int kTile = 8 * kH;            // 32 rows x 64 elements of one plane

struct FactArgs {
    const uint8_t* w;
    const float* x;
    float* y;
    int M, N, K;
    size_t rb;
    int ntm, ntn;
};

template <uint32_t T>
struct Traits {
    static constexpr int kPlanes = T == T_F32 ? 3 : T == T_F16 ? 2 : 1;    // bf16 pieces of a weight
    static constexpr bool kQuant = T == T_Q2_K || T == T_Q3_K || T == T_Q5_K;
    static constexpr bool kMin = T == T_Q2_K || T == T_Q5_K;
    // staging tasks per row: 4 values of F32, 8 of F16 / BF16, 8 code bytes (16 values) of the others
    static constexpr int kTasks = T == T_F32 ? 16 : kQuant ? 4 : 8;
    // floats per row and stage: Q5_K d * scale x 2, m x 2, dmin; Q3_K d; Q2_K d, dmin, m x 4
    static constexpr int kScales = T == T_Q5_K ? 5 : T == T_Q2_K ? 6 : T == T_Q3_K ? 1 : 0;
};

__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {      // rounded to nearest even
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, b2));
}
__device__ __forceinline__ float lo_f32(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float hi_f32(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }
__device__ __forceinline__ float hi16(float v) { return __uint_as_float(__float_as_uint(v) & 0xffff0000u); }

// What a thread has met of the values whose pieces do not hold all their bits: the x
// tasks (a bit each) with a quadruple below 2^-100 that is not all zeros; F32 only: the
// largest finite magnitude from 2^20 up, and the x and w tasks with such values.
struct Ends {
    uint32_t tiny = 0, xbig = 0, wbig = 0;
    float big = 0.0f;
};

// v[4] as PL planes of 4 bf16 whose sum is v: each piece is the rest rounded to
// nearest. Values whose first piece would round to infinity, and infinities
// (their own first piece), are cut off instead. One comparison finds these and the
// quadruples that Ends counts (all zeros among them).
template <int PL, bool BIG, bool X>
__device__ __forceinline__ void split4(const float (&v)[4], u32x2 (&o)[PL], Ends& e, uint32_t bit) {
    float r[4];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        o[0][i] = pk_bf16(v[2 * i], v[2 * i + 1]);
        r[2 * i] = v[2 * i] - lo_f32(o[0][i]);
        r[2 * i + 1] = v[2 * i + 1] - hi_f32(o[0][i]);
        if constexpr (PL > 1) o[1][i] = pk_bf16(r[2 * i], r[2 * i + 1]);
        if constexpr (PL > 2)
            o[2][i] = pk_bf16(r[2 * i] - lo_f32(o[1][i]), r[2 * i + 1] - hi_f32(o[1][i]));
    }
    if constexpr (PL == 1) return;
    const float a = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
    constexpr float top = BIG ? 0x1p20f : 0x1.fe8p127f;
    constexpr uint32_t lo = X ? (127u - 100u) << 23 : 0u;
    if (__builtin_expect(__float_as_uint(a) - lo < __builtin_bit_cast(uint32_t, top) - lo, 1)) return;
    if (BIG && a >= top) {
#pragma unroll
        for (int i = 0; i < 4; i++) e.big = fmaxf(e.big, fabsf(v[i]) < __builtin_inff() ? fabsf(v[i]) : 0.0f);
        (X ? e.xbig : e.wbig) |= bit;
    }
    if (X && a > 0.0f && a < 0x1p-100f) e.tiny |= bit;
    if (a >= 0x1.fe8p127f) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            uint32_t q[2][3];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const float x = v[2 * i + k], x1 = hi16(x), r1 = fabsf(x) == __builtin_inff() ? 0.0f : x - x1;
                const float x2 = hi16(r1);
                q[k][0] = __float_as_uint(x1) >> 16;
                q[k][1] = __float_as_uint(x2) >> 16;
                q[k][2] = __float_as_uint(r1 - x2) >> 16;
            }
#pragma unroll
            for (int p = 0; p < PL; p++) o[p][i] = q[0][p] | (q[1][p] << 16);
        }
    }
}

template <uint32_t T>
struct WReg {
    u32x4 a;             // F32: 4 values; F16, BF16: 8
    u32x2 q, h;          // code bytes, high-bit bytes
    u32x4 hd;            // Q5_K header
    uint32_t s0, s1, d;  // scale bytes, d (and dmin)
};

// Task t of the 64-element stage s of the row at base + off. F32, F16, BF16: past
// the row's end its last bytes again.
template <uint32_t T>
__device__ __forceinline__ void w_load(WReg<T>& r, const uint8_t* base, uint32_t off, uint32_t rb, int s, int t) {
    if constexpr (T == T_F32 || T == T_F16 || T == T_BF16) {
        uint32_t o = (uint32_t)s * (T == T_F32 ? 256u : 128u) + 16u * t;
        o = off + (o < rb - 16 ? o : rb - 16);
        if constexpr (T == T_F32) r.a = *reinterpret_cast<const u32x4_a4*>(base + o);
        else r.a = *reinterpret_cast<const u32x4_a2*>(base + o);
    } else if constexpr (T == T_Q5_K) {
        const uint8_t* sb = base + (size_t)(s >> 2) * 176;
        r.hd = *reinterpret_cast<const u32x4_a4*>(sb + off);
        r.h = *reinterpret_cast<const u32x2_a2*>(sb + 16 + (off + 8u * t));
        r.q = *reinterpret_cast<const u32x2_a2*>(sb + 48 + 32 * (s & 3) + (off + 8u * t));
    } else if constexpr (T == T_Q3_K) {
        const uint8_t* sb = base + (size_t)(s >> 2) * 110;
        r.h = *reinterpret_cast<const u32x2_a2*>(sb + (off + 8u * t));
        r.q = *reinterpret_cast<const u32x2_a2*>(sb + 32 + 32 * ((s & 3) >> 1) + (off + 8u * t));
        // scale bytes of groups j = 4 (s & 3) + 2 u + (t >> 1), u = 0, 1: low nibbles
        // at 96 + (j & 7), high bits at 104 + (j & 3)
        const uint32_t j = 4 * (s & 3) + (t >> 1);
        r.s0 = sb[off + 96 + (j & 7)] | (uint32_t)sb[off + 96 + ((j + 2) & 7)] << 8;
        r.s1 = sb[off + 104 + (j & 3)] | (uint32_t)sb[off + 104 + ((j + 2) & 3)] << 8;
        r.d = load_u16(sb + 108 + off);
    } else {
        const uint8_t* sb = base + (size_t)(s >> 2) * 84;
        r.q = *reinterpret_cast<const u32x2_a2*>(sb + 16 + 32 * ((s & 3) >> 1) + (off + 8u * t));
        r.s0 = *reinterpret_cast<const uint32_t*>(sb + 4 * (s & 3) + off);      // the stage's 4 groups
        r.d = *reinterpret_cast<const uint32_t*>(sb + 80 + off);
    }
}

// LDS of one K group's stage: x planes, w planes, floats per weight row (kScales
// x BN), and for the types with mins the sums of x: 16 bytes per token and lane half.
template <uint32_t T, int BM, int BN>
struct Lay {
    static constexpr int x = 0;
    static constexpr int w = x + 3 * (BM / 32) * kTile;
    static constexpr int sc = w + Traits<T>::kPlanes * (BN / 32) * kTile;
    static constexpr int xs = (sc + 4 * Traits<T>::kScales * BN + 15) & ~15;
    static constexpr int bytes = xs + (Traits<T>::kMin ? 32 * BM : 0);
};

template <uint32_t T, int BM, int BN>
__device__ __forceinline__ void w_store(const WReg<T>& r, uint8_t* st, int n, int s, int t, bool on, Ends& ends, uint32_t bit) {
    typedef Lay<T, BM, BN> L;
    constexpr int PL = Traits<T>::kPlanes;
    uint8_t* wt = st + L::w + (n >> 5) * kTile + (n & 31) * 16;
    float* sc = reinterpret_cast<float*>(st + L::sc) + n;
    if constexpr (T == T_BF16) {
        *reinterpret_cast<u32x4*>(wt + t * kH) = on ? r.a : u32x4{0, 0, 0, 0};
    } else if constexpr (T == T_F32 || T == T_F16) {
#pragma unroll
        for (int h = 0; h < (T == T_F32 ? 1 : 2); h++) {
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if constexpr (T == T_F32) v[i] = __uint_as_float(r.a[i]);
                else v[i] = fp16_bits_to_f32(r.a[2 * h + (i >> 1)] >> (16 * (i & 1)));
                v[i] = on ? v[i] : 0.0f;
            }
            u32x2 o[PL];
            split4<PL, T == T_F32, false>(v, o, ends, bit);
            uint8_t* p = T == T_F32 ? wt + (t >> 1) * kH + 8 * (t & 1) : wt + t * kH + 8 * h;
#pragma unroll
            for (int k = 0; k < PL; k++) *reinterpret_cast<u32x2*>(p + k * (BN / 32) * kTile) = o[k];
        }
    } else {
        // values 8t .. 8t + 7 of the stage's two 32-element groups 2j, 2j + 1
        const int j = s & 3;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            float f = 1.0f;
            if constexpr (T == T_Q3_K) {
                const uint32_t k = 4 * j + 2 * u + (t >> 1);
                const uint32_t lo = (r.s0 >> (8 * u)) & 0xffu, hb = (r.s1 >> (8 * u)) & 0xffu;
                f = (float)((int)(((k < 8 ? lo : lo >> 4) & 15u) | (((hb >> (2 * (k >> 2))) & 3u) << 4)) - 32);
            } else if constexpr (T == T_Q2_K) {
                f = (float)((r.s0 >> (8 * (2 * u + (t >> 1)))) & 15u);
            }
            u32x4 o;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                uint32_t c;
                if constexpr (T == T_Q5_K)
                    c = ((r.q[i] >> (4 * u)) & 0x0f0f0f0fu) | (((r.h[i] >> (2 * j + u)) & 0x01010101u) << 4);
                else
                    c = (r.q[i] >> (4 * (j & 1) + 2 * u)) & 0x03030303u;
                if constexpr (T == T_Q3_K) c |= ((r.h[i] >> (2 * j + u)) & 0x01010101u) << 2;      // code + 4
                float v[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    v[k] = (float)((c >> (8 * k)) & 0xffu);
                    if constexpr (T == T_Q3_K) v[k] = (v[k] - 4.0f) * f;
                    if constexpr (T == T_Q2_K) v[k] *= f;
                }
                o[2 * i] = pk_bf16(v[0], v[1]);
                o[2 * i + 1] = pk_bf16(v[2], v[3]);
            }
            *reinterpret_cast<u32x4*>(wt + (4 * u + t) * kH) = o;
        }
        if constexpr (T == T_Q5_K) {
            if (t < 2) {
                uint32_t s6, m6;
                scale_min_k4(2 * j + t, r.hd.y, r.hd.z, r.hd.w, s6, m6);
                sc[t * BN] = fp16_bits_to_f32(r.hd.x) * (float)s6;
                sc[(2 + t) * BN] = (float)m6;
            } else if (t == 2) {
                sc[4 * BN] = fp16_bits_to_f32(r.hd.x >> 16);
            }
        } else if constexpr (T == T_Q2_K) {
            sc[(2 + t) * BN] = (float)((r.s0 >> (8 * t + 4)) & 15u);
            if (t < 2) sc[t * BN] = fp16_bits_to_f32(r.d >> (16 * t));
        } else {
            if (t == 0) sc[0] = fp16_bits_to_f32(r.d);
        }
    }
}

// Outputs that the pieces do not give are made again in fp32:
//  - infinite and NaN ones: the pieces of an infinity are (inf, 0, 0) and its product
//    with a zero piece of a finite value is NaN, so are partial sums past the fp32
//    range with opposite signs;
//  - those that bits below the pieces' last one could show in: bf16 ends at 2^-133
//    (the matrix unit keeps such denormals, and its fp32 results'), so the pieces of
//    an x are off by up to 2^-134 where it is below 2^-110, and the sum by up to
//    K 2^-134 times the largest weight: 2^16 in F16, below 2^28 in the quantized types
//    and 2^20 in F32 and BF16, or what was met in an F32 column beyond that. (F32 weights
//    have the same pieces beside the largest x of the row.) Outputs below K 2^-110 times
//    that size are suspect; ordinary sums do not come there by cancellation, their 64-bit
//    sums end in a whole zero or far above;
//  - the rows of x with four neighbours all below 2^-100, not all zero: BF16 weights are not
//    looked at on their way to LDS and may be of any size.
// What is left: a sum of values below 2^-134 among larger ones may come out 0, and of BF16
// weights beyond 2^20 those beside an x below 2^-110 whose three neighbours are larger count
// with its first bits.
//
// A wave makes an output or four at a time, its lanes side by side along K. Measured (us,
// plain / one infinite row / all x near 1e-30; with a lane per output before): BF16
// N 14336 K 4096 M 200 147 / 388 / 2590 (1080 / 30450), N 4096 M 12 21 / 65 / 175 (414 /
// 768), Q5_K M 200 197 / 598 / 3940 (3290 / 226800), N 4096 M 12 30 / 151 / 361 (1540 / 5470).
// The GEMVs: 33 and 1560, 70 and 2650.
template <uint32_t T>
__device__ __forceinline__ void decode8(const uint8_t* w, int k, float (&v)[8], float& mn) {
    mn = 0.0f;
    if constexpr (T == T_F32) {
        const u32x4 a = *reinterpret_cast<const u32x4_a4*>(w + 4l * k), b = *reinterpret_cast<const u32x4_a4*>(w + 4l * k + 16);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = __uint_as_float(a[i]), v[4 + i] = __uint_as_float(b[i]);
    } else if constexpr (T == T_F16 || T == T_BF16) {
        const u32x4 a = *reinterpret_cast<const u32x4_a2*>(w + 2l * k);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[2 * i] = T == T_F16 ? fp16_bits_to_f32(a[i]) : lo_f32(a[i]);
            v[2 * i + 1] = T == T_F16 ? fp16_bits_to_f32(a[i] >> 16) : hi_f32(a[i]);
        }
    } else {
        // 8 values of one 16-element group: their low bits' and high bits' bytes
        const int e = k & 255, j = e >> 4, g = e >> 5;
        u32x2 q, h = {0, 0};
        float d;
        int sh, hs = 0;
        if constexpr (T == T_Q2_K) {
            const uint8_t* b = w + (k >> 8) * 84l;
            d = fp16_bits_to_f32(rd16(b + 80)) * (float)(b[j] & 15);
            mn = fp16_bits_to_f32(rd16(b + 82)) * (float)(b[j] >> 4);
            q = *reinterpret_cast<const u32x2_a2*>(b + 16 + 32 * (g >> 2) + (e & 31));
            sh = 2 * (g & 3);
        } else if constexpr (T == T_Q3_K) {
            const uint8_t* b = w + (k >> 8) * 110l;
            d = fp16_bits_to_f32(rd16(b + 108)) * (float)(q3k_scale(b + 96, j) - 32);
            q = *reinterpret_cast<const u32x2_a2*>(b + 32 + 32 * (g >> 2) + (e & 31));
            h = *reinterpret_cast<const u32x2_a2*>(b + (e & 31));
            sh = 2 * (g & 3);
            hs = g;
        } else {
            const uint8_t* b = w + (k >> 8) * 176l;
            int sc, mi;
            scale_min(g, b + 4, sc, mi);
            d = fp16_bits_to_f32(rd16(b)) * (float)sc;
            mn = fp16_bits_to_f32(rd16(b + 2)) * (float)mi;
            q = *reinterpret_cast<const u32x2_a2*>(b + 48 + 32 * (g >> 1) + (e & 31));
            h = *reinterpret_cast<const u32x2_a2*>(b + 16 + (e & 31));
            sh = 4 * (g & 1);
            hs = g;
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t lo = (q[i >> 2] >> (8 * (i & 3) + sh)) & (T == T_Q5_K ? 15u : 3u), hi = (h[i >> 2] >> (8 * (i & 3) + hs)) & 1u;
            v[i] = d * (T == T_Q3_K ? (float)((int)(lo + 4 * hi) - 4) : (float)(T == T_Q5_K ? lo + 16 * hi : lo));
        }
    }
}
// R rows of x from m0 on (those past M: the last one) times column n, the sums of type S in
// every lane; the mins' sums apart, as the reference keeps them
template <uint32_t T, int R, typename S>
__device__ __forceinline__ void wave_dot(const FactArgs& g, int m0, int n, int lane, float (&out)[R]) {
    const uint8_t* w = g.w + (size_t)n * g.rb;
    S s[R] = {}, sm[R] = {};
#pragma unroll R == 1 ? 4 : 2
    for (int k = 8 * lane; k < g.K; k += 512) {
        float v[8], mn;
        decode8<T>(w, k, v, mn);
#pragma unroll
        for (int i = 0; i < R; i++) {
            const float* x = g.x + (size_t)(m0 + i < g.M ? m0 + i : g.M - 1) * g.K + k;
            const float4 a = *reinterpret_cast<const float4*>(x), b = *reinterpret_cast<const float4*>(x + 4);
            const float u[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int l = 0; l < 8; l++) {
                s[i] = __builtin_elementwise_fma((S)u[l], (S)v[l], s[i]);
                if constexpr (Traits<T>::kMin) sm[i] = __builtin_elementwise_fma((S)u[l], (S)mn, sm[i]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < R; i++) out[i] = (float)(Traits<T>::kMin ? wave_sum(s[i]) - wave_sum(sm[i]) : wave_sum(s[i]));
}
__device__ __forceinline__ bool suspect(float v, float below) {
    const float a = fabsf(v);
    return !(a == 0.0f || (a >= below && a < __builtin_inff()));
}

// LDS of the stages, and after them of the K groups' sums
template <uint32_t T, int MT, int NT, int WM, int WN, int WK>
constexpr int lds_bytes() {
    constexpr int red = WK > 1 ? WK * WM * WN * MT * NT * 8192 : 0;
    constexpr int bufs = WK * (WM * WN == 1 ? 1 : 2) * Lay<T, 32 * MT * WM, 32 * NT * WN>::bytes;
    return bufs > red ? bufs : red;
}

// MT x NT tiles of 32 x 32 per wave.
template <uint32_t T, int MT, int NT, int WM, int WN, int WK>
__global__ void __launch_bounds__(64 * WM * WN * WK, 2)
gemm_fact(FactArgs g) {
    constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN, GT = 64 * WM * WN;
    typedef Lay<T, BM, BN> L;
    typedef Traits<T> R;
    constexpr int XPT = BM * 16 / GT, WPT = (BN * R::kTasks + GT - 1) / GT, PL = R::kPlanes;
    static_assert(BM * 16 % GT == 0, "whole tasks");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x % GT, kg = WK > 1 ? (int)(threadIdx.x / GT) : 0;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    // a group of one wave needs no barrier and one buffer: its LDS operations are in order
    constexpr int NBUF = GT == 64 ? 1 : 2;
    uint8_t* const lds = smem + kg * NBUF * L::bytes;
    uint32_t* const again = reinterpret_cast<uint32_t*>(smem + lds_bytes<T, MT, NT, WM, WN, WK>());
    if (threadIdx.x == 0) *again = 0;      // whether the tile has outputs to make again
    Ends ends;

    // tile order: as in the int8 product (one near-square block of tiles per XCD)
    const int ntiles = g.ntm * g.ntn, bid = blockIdx.x;
    const int q8 = ntiles >> 3, r8 = ntiles & 7, xcd = bid & 7;
    const int tile = xcd * q8 + (xcd < r8 ? xcd : r8) + (bid >> 3);
    constexpr int kGroup = 512 / BM;
    const int grp = tile / (kGroup * g.ntn), in = tile - grp * kGroup * g.ntn;
    const int gm = g.ntm - grp * kGroup < kGroup ? g.ntm - grp * kGroup : kGroup;
    const int m0 = (grp * kGroup + in % gm) * BM, n0 = in / gm * BN;
    const int nst = (g.K + 63) >> 6, iters = (nst + WK - 1) / WK;

    float4 rx[XPT];
    WReg<T> rw[WPT];
    uint32_t xrow[XPT], woff[WPT];
    const uint32_t quad = tid & 15;                 // 4-element piece of this thread's x tasks
#pragma unroll
    for (int i = 0; i < XPT; i++) {
        const int row = (tid + i * GT) >> 4, m = m0 + row < g.M ? row : g.M - 1 - m0;
        xrow[i] = (uint32_t)m * (uint32_t)g.K;
    }
#pragma unroll
    for (int i = 0; i < WPT; i++) {
        const int p = tid + i * GT, row = BN * R::kTasks % GT == 0 || p < BN * R::kTasks ? p / R::kTasks : 0;
        const int n = n0 + row < g.N ? row : g.N - 1 - n0;
        woff[i] = (uint32_t)n * (uint32_t)g.rb;
    }
    const float* const xbase = g.x + (size_t)m0 * g.K;
    const uint8_t* const wbase = g.w + (size_t)n0 * g.rb;
    // No load depends on a branch: pieces past K re-read the row's last elements (a
    // stage past K the last stage's) and store() writes zeros for them.
    auto load = [&](int s) {
        s = s < nst ? s : nst - 1;
        const uint32_t e = 64u * s + 4u * quad, ec = e < (uint32_t)g.K ? e : (uint32_t)g.K - 4u;
#pragma unroll
        for (int i = 0; i < XPT; i++) rx[i] = *reinterpret_cast<const float4*>(xbase + (xrow[i] + ec));
#pragma unroll
        for (int i = 0; i < WPT; i++)
            w_load<T>(rw[i], wbase, woff[i], (uint32_t)g.rb, s, (tid + i * GT) % R::kTasks);
    };
    auto store = [&](int s, uint8_t* st) {
        const bool on = 64 * s + 4 * (int)quad < g.K;
#pragma unroll
        for (int i = 0; i < XPT; i++) {
            const int row = (tid + i * GT) >> 4;
            const float v[4] = {on ? rx[i].x : 0.0f, on ? rx[i].y : 0.0f, on ? rx[i].z : 0.0f, on ? rx[i].w : 0.0f};
            u32x2 o[3];
            split4<3, T == T_F32, true>(v, o, ends, 1u << i);
            uint8_t* p = st + L::x + (row >> 5) * kTile + (quad >> 1) * kH + (row & 31) * 16 + 8 * (quad & 1);
#pragma unroll
            for (int k = 0; k < 3; k++) *reinterpret_cast<u32x2*>(p + k * (BM / 32) * kTile) = o[k];
            if constexpr (R::kMin) {
                // sums of 16 (Q2_K) or 32 elements over 4 or 8 lanes, as three bf16
                // pieces in K slots 0..2 and 4..6 of a lane half
                float u = (v[0] + v[1]) + (v[2] + v[3]);
                u = dpp_step<0xb1, 0xf>(u);
                u = dpp_step<0x4e, 0xf>(u);
                if constexpr (T == T_Q5_K) u = dpp_step<0x141, 0xf>(u);        // row_half_mirror
                const float u1 = hi16(u), r = u - u1, u2 = hi16(r), u3 = r - u2;
                const u32x2 rec = {__builtin_amdgcn_perm(__float_as_uint(u2), __float_as_uint(u1), 0x07060302u),
                                   __float_as_uint(u3) >> 16};
                u32x2* xs = reinterpret_cast<u32x2*>(st + L::xs) + 2 * ((quad >> 3) * BM + row);
                if constexpr (T == T_Q2_K) {
                    if ((quad & 3) == 0) xs[(quad >> 2) & 1] = rec;
                } else {
                    if ((quad & 3) == 0) xs[(quad >> 2) & 1] = quad & 4 ? u32x2{0, 0} : rec;
                }
            }
        }
        const int sw = s < nst ? s : nst - 1;
#pragma unroll
        for (int i = 0; i < WPT; i++) {
            const int p = tid + i * GT, t = p % R::kTasks;
            if (BN * R::kTasks % GT == 0 || p < BN * R::kTasks)
                w_store<T, BM, BN>(rw[i], st, p / R::kTasks, sw, t, 64 * s + (R::kQuant ? 0 : 64 / R::kTasks * t) < g.K, ends, 1u << i);
        }
    };

    double sum[MT][NT][16];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < NT; r++)
#pragma unroll
            for (int i = 0; i < 16; i++) sum[t][r][i] = 0.0;

    const int col = lane & 31, half = lane >> 5;
    auto compute = [&](const uint8_t* st) {
        const uint8_t* xt = st + L::x + wm * MT * kTile + half * kH + col * 16;
        const uint8_t* wt = st + L::w + wn * NT * kTile + half * kH + col * 16;
        const float* sc = reinterpret_cast<const float*>(st + L::sc) + wn * NT * 32 + col;
        f16v P[MT][NT];
        float chain[T == T_Q5_K ? MT : 1][T == T_Q5_K ? NT : 1][16];
        // Per unit (the stage; a 32-element block of Q5_K) the smaller products come
        // first, so that only those of the first pieces are rounded at the sum's size.
        constexpr int KU = T == T_Q5_K ? 2 : 4;
        b8v B[KU][PL][NT];
        auto frag_b = [&](int u, int k, int p) {
#pragma unroll
            for (int r = 0; r < NT; r++)
                B[k][p][r] = *reinterpret_cast<const b8v*>(wt + (p * (BN / 32) + r) * kTile + 2 * (u * KU + k) * kH);
        };
#pragma unroll
        for (int u = 0; u < 4 / KU; u++) {
#pragma unroll
            for (int k = 0; k < 2 * KU; k++) {
                const int kk = k % KU;
                b8v A[3][MT];
                // with several planes of w the first is read again for its second use
                if (k < KU) {
#pragma unroll
                    for (int p = 0; p < PL; p++) frag_b(u, kk, p);
                } else if (PL > 1) {
                    frag_b(u, kk, 0);
                }
#pragma unroll
                for (int p = k < KU && PL == 1 ? 1 : 0; p < (k < KU ? 3 : 1); p++)
#pragma unroll
                    for (int t = 0; t < MT; t++)
                        A[p][t] = *reinterpret_cast<const b8v*>(xt + (p * (BM / 32) + t) * kTile + 2 * (u * KU + kk) * kH);
#pragma unroll
                for (int r = 0; r < NT; r++)
#pragma unroll
                    for (int t = 0; t < MT; t++) {
                        f16v c = k == 0 ? f16v{} : P[t][r];
                        // pieces i of x and o - i of w, o = 2, 1, then 0
                        if (k < KU) {
#pragma unroll
                            for (int o = 2; o >= 1; o--)
#pragma unroll
                                for (int i = 2; i >= 0; i--)
                                    if (o - i >= 0 && o - i < PL)
                                        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[i][t], B[kk][o - i][r], c, 0, 0, 0);
                        } else {
                            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[0][t], B[kk][0][r], c, 0, 0, 0);
                        }
                        P[t][r] = c;
                    }
            }
            if constexpr (T == T_Q5_K) {
#pragma unroll
                for (int r = 0; r < NT; r++) {
                    const float ds = sc[u * BN + 32 * r];
#pragma unroll
                    for (int t = 0; t < MT; t++)
#pragma unroll
                        for (int i = 0; i < 16; i++)
                            chain[t][r][i] = u == 0 ? P[t][r][i] * ds : fmaf(P[t][r][i], ds, chain[t][r][i]);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < NT; r++) {
            double d = 1.0, dm = 0.0;
            b8v mb;
            if constexpr (T == T_Q2_K || T == T_Q3_K) d = (double)sc[32 * r];
            if constexpr (R::kMin) {
                dm = -(double)sc[(T == T_Q5_K ? 4 : 1) * BN + 32 * r];
                const float ma = T == T_Q5_K ? sc[(2 + half) * BN + 32 * r] : sc[(2 + 2 * half) * BN + 32 * r];
                const float mc = T == T_Q5_K ? 0.0f : sc[(3 + 2 * half) * BN + 32 * r];
                const uint32_t a1 = __float_as_uint(ma) >> 16, c1 = __float_as_uint(mc) >> 16;
                const u32x4 o = {a1 | (a1 << 16), a1, c1 | (c1 << 16), c1};
                mb = __builtin_bit_cast(b8v, o);
            }
#pragma unroll
            for (int t = 0; t < MT; t++) {
                f16v am;
                if constexpr (R::kMin) {
                    const b8v xs = reinterpret_cast<const b8v*>(st + L::xs)[half * BM + (wm * MT + t) * 32 + col];
                    am = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xs, mb, f16v{}, 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    float v;
                    if constexpr (T == T_Q5_K) v = chain[t][r][i];
                    else v = P[t][r][i];
                    if constexpr (T == T_Q2_K || T == T_Q3_K) sum[t][r][i] = fma((double)v, d, sum[t][r][i]);
                    else sum[t][r][i] += (double)v;
                    if constexpr (R::kMin) sum[t][r][i] = fma((double)am[i], dm, sum[t][r][i]);
                }
            }
        }
    };

    // Group kg takes the stages kg, kg + WK, ..; while one computes from one LDS
    // buffer, the next is loaded into registers and then written to the other.
    load(kg);
    store(kg, lds);
    __syncthreads();
    for (int it = 0; it < iters; it++) {
        const int next = (it + 1) * WK + kg;
        if (WK > 1 && it == iters - 1) {        // few stages per group: no wait for a load nobody needs (19.6 -> 18.8 us)
            compute(lds + (NBUF == 2 ? (it & 1) * L::bytes : 0));
            break;
        }
        load(next);
        compute(lds + (NBUF == 2 ? (it & 1) * L::bytes : 0));
        if constexpr (NBUF == 1) __builtin_amdgcn_wave_barrier();
        store(next, lds + (NBUF == 2 ? ((it + 1) & 1) * L::bytes : 0));
        if constexpr (NBUF == 1) __builtin_amdgcn_wave_barrier();
        else __syncthreads();
    }

    // register j = (t * NT + r) * 16 + i of a lane: its token and weight row (the lane's
    // number is read again, so that the part below keeps no register through the loop)
    const int ln = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    auto mrow = [&](int j) { return m0 + (wm * MT + (j >> 4) / NT) * 32 + 8 * ((j & 15) >> 2) + 4 * (ln >> 5) + (j & 3); };
    auto nrow = [&](int j) { return n0 + (wn * NT + (j >> 4) % NT) * 32 + (ln & 31); };
    constexpr float kSize = T == T_F16 ? 0x1p16f : R::kQuant ? 0x1p28f : 0x1p20f;
    const float below = (float)g.K * (0x1p-110f * kSize);
    bool bad = false;
    auto put = [&](int j, float v) {
        const int m = mrow(j), n = nrow(j);
        if (m < g.M && n < g.N) g.y[(size_t)m * g.N + n] = v;
        bad |= suspect(v, below);
    };
    if constexpr (WK > 1) {
        __syncthreads();      // every wave is done with its buffer
        // All groups leave their sums in LDS; group kg adds those of registers kg,
        // kg + WK, .. in the groups' order (against one group adding the others' one
        // after the other: BF16 N 4096 K 4096 M 12 21.4 -> 19.6 us).
        double* red = reinterpret_cast<double*>(smem) + wave * MT * NT * 16 * 64 + ln;
        constexpr int kGrp = WM * WN * MT * NT * 16 * 64;
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < NT; r++)
#pragma unroll
                for (int i = 0; i < 16; i++) red[kg * kGrp + ((t * NT + r) * 16 + i) * 64] = sum[t][r][i];
        __syncthreads();
        for (int j = kg; j < MT * NT * 16; j += WK) {
            double u = red[j * 64];
#pragma unroll
            for (int q = 1; q < WK; q++) u += red[q * kGrp + j * 64];
            put(j, (float)u);
        }
    } else {
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < NT; r++)
#pragma unroll
                for (int i = 0; i < 16; i++) put((t * NT + r) * 16 + i, (float)sum[t][r][i]);
    }
    if (bad || ends.tiny || ends.big > 0.0f) *again = 1;
    __syncthreads();
    if (__builtin_expect(*again == 0, 1)) return;

    // of the tile's x and weight rows: the largest magnitude from 2^20 up, all bits set for tiny x rows
    uint32_t* const ex = reinterpret_cast<uint32_t*>(smem);
    const int tg = (int)(threadIdx.x % GT);
    for (int i = threadIdx.x; i < BM + BN; i += GT * WK) ex[i] = 0;
    __syncthreads();
    for (int i = 0; i < XPT; i++) {
        const uint32_t v = (ends.tiny >> i) & 1u ? ~0u : (ends.xbig >> i) & 1u ? __float_as_uint(ends.big) : 0u;
        if (v) atomicMax(ex + ((tg + i * GT) >> 4), v);
    }
    for (int i = 0; i < WPT; i++)
        if ((ends.wbig >> i) & 1u) atomicMax(ex + BM + (tg + i * GT) / R::kTasks, __float_as_uint(ends.big));
    __syncthreads();
    // units of four registers, i.e. of four rows in a column
    for (int u = kg; u < MT * NT * 4; u += WK) {
        const int m = mrow(4 * u), n = nrow(4 * u);
        float* const y = g.y + (size_t)m * g.N + n;
        uint32_t todo = 0, nans = 0, inf = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (m + i >= g.M || n >= g.N) continue;
            const float v = y[(size_t)i * g.N];
            const uint32_t xe = ex[m + i - m0], we = ex[BM + n - n0];
            const float size = fmaxf(kSize, __uint_as_float(xe > we ? xe : we));
            if (xe == ~0u || suspect(v, (float)g.K * 0x1p-110f * size)) todo |= 1u << i;
            if (v != v) nans |= 1u << i;
            if (!(fabsf(v) < __builtin_inff())) inf |= 1u << i;
        }
        // a NaN in x makes its row NaN: nothing to be made again
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint64_t b = __ballot((nans >> (i & 3)) & 1u) & (i < 4 ? 0xffffffffull : ~0xffffffffull);
            if (!b) continue;
            const float* x = g.x + (size_t)(__builtin_amdgcn_readlane(m, i < 4 ? 0 : 32) + (i & 3)) * g.K;
            bool nan = false;
            for (int k = 4 * ln; k < g.K && !__any(nan); k += 256) {
                const float4 a = *reinterpret_cast<const float4*>(x + k);
                nan = a.x != a.x || a.y != a.y || a.z != a.z || a.w != a.w;
            }
            if (__any(nan) && (ln >> 5) == (i >> 2)) todo &= ~(1u << (i & 3));
        }
        // non-finite ones singly in 64 bits (a lane's share may leave the fp32 range where
        // the sum does not), small ones of the four rows at once
        for (uint64_t left = __ballot(todo != 0); left; left &= left - 1) {
            const int l = __ffsll((unsigned long long)left) - 1;
            const int ml = __builtin_amdgcn_readlane(m, l), nl = __builtin_amdgcn_readlane(n, l);
            const uint32_t td = __builtin_amdgcn_readlane(todo, l), large = __builtin_amdgcn_readlane(inf, l) & td;
            for (int i = 0; i < 4; i++) {
                if (!((large >> i) & 1u)) continue;
                float v[1];
                wave_dot<T, 1, double>(g, ml + i, nl, ln, v);
                if (ln == l) y[(size_t)i * g.N] = v[0];
            }
            if (td == large) continue;
            float v[4];
            wave_dot<T, 4, float>(g, ml, nl, ln, v);
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (ln == l && (((td ^ large) >> i) & 1u)) y[(size_t)i * g.N] = v[i];
        }
    }
}

template <uint32_t T, int MT, int NT, int WM, int WN, int WK>
hipError_t launch_cfg(FactArgs g, hipStream_t st) {
    constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN;
    constexpr int lds = lds_bytes<T, MT, NT, WM, WN, WK>() + 16;            // and a flag
    static_assert(lds <= 160 * 1024, "LDS");
    g.ntm = (g.M + BM - 1) / BM;
    g.ntn = (g.N + BN - 1) / BN;
    hipLaunchKernelGGL((gemm_fact<T, MT, NT, WM, WN, WK>), dim3((unsigned)(g.ntm * g.ntn)), dim3(64 * WM * WN * WK), lds,
                       st, g);
    return hipGetLastError();
}

}  // namespace

namespace {
// The tile forms (as the int8 product's; 64 x 128 where the planes of the weights
// leave no LDS for 128 x 128). Measured, us, N 4096 K 4096:
//   BF16  M 64   (256 tiles of 32 x 32)   32x32x8 24.8, 32x32x4 30, 64x64x2 49
//         M 128  (512)                    32x32x4 41, 32x32x8 47, 64x64x2 51
//         M 256  (256 tiles of 64 x 64)   64x64x2 54, 64x64 76, 32x32x4 77
//         M 512  (512)                    64x64 95 (87 in a stream of calls), 64x64x2 107, 128x128 123
//         M 2048 (512 tiles of 128 x 128) 128x128 253, 64x64 343
//   F32   M 128  32x32x6 85, 64x64 119      M 256  64x64 119, 64x128 165
//         M 512  64x128 169, 64x64 225
// Several planes leave LDS for six K groups of 32 x 32 and for 64 x 128 at most.
enum Form { F32X32X8, F32X32X6, F32X32X4, F64X64X2, F64X64, F64X128, F128X128 };

template <uint32_t T>
Form pick_form(int M, int N) {
    const long cus = device_cu_count();
    auto tiles = [&](int b) { return (long)((M + b - 1) / b) * ((N + b - 1) / b); };
    constexpr bool one = Traits<T>::kPlanes == 1;
    if (!one) return tiles(32) <= 2 * cus || M <= 32 ? F32X32X6 : tiles(64) <= cus ? F64X64 : F64X128;
    if (tiles(32) <= cus) return F32X32X8;
    if (tiles(32) <= 2 * cus || M <= 32) return F32X32X4;
    if (tiles(64) <= cus) return F64X64X2;
    const long r64 = (tiles(64) + 2 * cus - 1) / (2 * cus), r128 = (tiles(128) + cus - 1) / cus;
    return 1.4 * r128 < r64 ? F128X128 : F64X64;
}

template <uint32_t T>
hipError_t launch_t(const FactArgs& g, hipStream_t st) {
    const Form f = pick_form<T>(g.M, g.N);
    if constexpr (Traits<T>::kPlanes == 1) {
        switch (f) {
            case F32X32X8: return launch_cfg<T, 1, 1, 1, 1, 8>(g, st);
            case F32X32X4: return launch_cfg<T, 1, 1, 1, 1, 4>(g, st);
            case F64X64X2: return launch_cfg<T, 1, 1, 2, 2, 2>(g, st);
            case F64X64: return launch_cfg<T, 1, 1, 2, 2, 1>(g, st);
            case F128X128: return launch_cfg<T, 1, 2, 4, 2, 1>(g, st);
            default: break;
        }
    } else {
        switch (f) {
            case F32X32X6: return launch_cfg<T, 1, 1, 1, 1, 6>(g, st);
            case F64X64: return launch_cfg<T, 1, 1, 2, 2, 1>(g, st);
            case F64X128: return launch_cfg<T, 1, 2, 2, 2, 1>(g, st);
            default: break;
        }
    }
    return hipErrorInvalidValue;
}
}  // namespace

// Where this product beats the GEMVs, which read the weights once per 4 rows: up to
// 32 rows its time depends on K alone and on the rounds of tiles, theirs on M N K, so the
// line is a number of outputs (for F16, F32, Q2_K and Q5_K one per round of tiles), twice as
// many at K <= 2048, where its launch and last reduction weigh more. Measured (us, GEMV
// against this):
//   BF16 K 4096: N 4096 M 5 18.7 / 19, M 6 21.0 / 19.5, M 12 31.5 / 18.8, M 33 82.5 / 20.0; N 1024
//     M 12 9.2 / 19, M 33 23.4 / 18.3. Whole passes of 4 rows cost the GEMV less: N 2048 M 12 15.5 /
//     18.5, M 13 19.4 / 18.6, M 16 19.6 / 18.7; N 3072 M 8 15.7 / 18.7, M 9 19.9 / 18.8; not at K 8192,
//     N 3072 M 8 36.0 / 32.9.
//   Q5_K K 4096: N 4096 M 6 30.4 / 27.7, M 12 66 / 28; K 3072: N 3072 M 8 20.6 / 22.0, M 9 25.2 / 22.3,
//     two rounds N 10240 M 6 38.3 / 39.6, M 7 41.1 / 39.5; K 2048 N 10240 M 8 22.6 / 27.9, M 9 29.1 /
//     28.0, N 14336 M 6 26.2 / 28.3, M 7 28.7 / 28.1; K 1024 N 10240 M 5 17.7 / 16.0.
//   Q2_K K 4096: N 4096 M 6 22.3 / 26, M 8 28.9 / 26.9, two rounds N 10240 M 6 40.3 / 48.9, M 7 51.8 /
//     48.8; K 2048 N 10240 M 8 22.9 / 26.7, M 9 29.0 / 26.7, N 14336 M 6 25.6 / 26.7, M 7 28.3 / 26.6.
//   Q3_K K 4096 N 4096 M 6 29.1 / 26.9.
//   F16, F32 (more products) K 4096: N 4096 M 8 24.4, 28.7 / 32, 37, M 12 37.4, 40.5 / 32.1, 36.5; F16
//     N 3072 M 16 29.5 / 31.5, K 8192 73.7 / 61.2; N 14336 (two rounds of tiles) F16 M 6 65.8 / 62.8, F32 M 6 86 / 73,
//     N 8200 F16 M 8 52.5 / 61.
//   K 1024, N 4096: BF16 M 8 7.9 / 7.2, M 12 10.5 / 7.2; F16 M 12 11.2 / 11.5, M 33 27 / 11.5.
// Large: N 14336 K 4096 M 200 BF16 1690 -> 140, Q5_K 2660 -> 186, Q3_K 2018 -> 150, Q2_K
// 1556 -> 168, F16 1547 -> 280, F32 2057 -> 329.
bool fact_gemm_preferred(uint32_t type, int M, int K, int N) {
    const long cus = device_cu_count(), rounds = ((long)((M + 31) / 32) * ((N + 31) / 32) + cus - 1) / cus;
    // a tile's weight rows (128) and x rows (128) are addressed with 32-bit offsets
    if (128 * fact_row_bytes(type, K) > (1ull << 32) || K > 1 << 25) return false;
    const long many = 12000 + 37000 * rounds;
    long line = 24000;
    switch (type) {
        case T_F32: line = many; break;
        case T_F16: line = N < 4096 && K > 2048 && K < 6144 && many < 50000 ? 50000 : many; break;
        case T_BF16: if (K > 2048 && K <= 6144 && M % 4 == 0) line = 30000; break;
        case T_Q2_K: line = K > 2048 ? 32000 * rounds : 32000; break;
        case T_Q5_K: if (K > 2048 && K < 4096) line = rounds > 1 ? 31000 * rounds : 25000; break;
    }
    if (K <= 2048) line *= 2;
    if ((type == T_Q2_K || type == T_Q5_K) && K > 1024 && K <= 2048 && rounds > 1) line = 45000 * rounds;
    return M >= (type == T_F16 ? 6 : 5) && (long)M * N >= line;
}

const char* fact_gemm_form(uint32_t type, int M, int N) {
    const Form f = type == T_F32 ? pick_form<T_F32>(M, N) : type == T_F16 ? pick_form<T_F16>(M, N) : pick_form<T_BF16>(M, N);
    switch (f) {
        case F32X32X8: return "fact_gemm 32x32x8";
        case F32X32X6: return "fact_gemm 32x32x6";
        case F32X32X4: return "fact_gemm 32x32x4";
        case F64X64X2: return "fact_gemm 64x64x2";
        case F64X64: return "fact_gemm 64x64";
        case F64X128: return "fact_gemm 64x128";
        default: return "fact_gemm 128x128";
    }
}

hipError_t launch_gemm_fact(uint32_t type, const uint8_t* w, const float* x, float* y, int M, int K, int N,
                            hipStream_t st) {
    if (M <= 0 || N <= 0) return hipSuccess;
    const FactArgs g{w, x, y, M, N, K, fact_row_bytes(type, K), 0, 0};
    switch (type) {
        case T_F32: return launch_t<T_F32>(g, st);
        case T_F16: return launch_t<T_F16>(g, st);
        case T_BF16: return launch_t<T_BF16>(g, st);
        case T_Q2_K: return launch_t<T_Q2_K>(g, st);
        case T_Q3_K: return launch_t<T_Q3_K>(g, st);
        case T_Q5_K: return launch_t<T_Q5_K>(g, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace lp
