// lp_gemm_i8t.hip - tiled int8-MFMA product of quantized activation rows with
// Q8_0 / Q4_0 / Q5_0 / Q4_K / Q6_K weights (prompt rows).
//
// y[m][n] = sum over 32-element blocks b of  xd[m][b] * wd[n][b] * P[m][n][b],
// P the exact int32 block sum (v_mfma_i32_32x32x32_i8, one block per
// instruction). The reference sums the same block terms in fp32
// (src/matmul_simd.cpp:143-342).
//
// Work split. A workgroup owns BM tokens x BN weight rows; its waves are
// WM x WN over the tile and WK over K (each of the WK groups stages and sums
// its own pairs of 128-element stages; the groups' sums are added through LDS
// at the end). A stage is 128 elements = 4 blocks: the activation codes are
// copied and the weights decoded to int8 once per workgroup into LDS in MFMA
// operand order ([32 rows][block][half][row][16 B], padded so that 8 pieces of a
// row or 4 blocks of 2 rows written together fall into distinct banks). The next
// stage's bytes are in registers while this one computes; two LDS buffers and one
// barrier per stage, or, where a group is one wave, one buffer and none.
//
// Scales. Multiplying xd * wd for every output and block on the VALU would cost
// a third operation beside the conversion and the fma, and its operands many LDS
// reads. The tile of products xd (x) wd comes from one bf16 MFMA instead: an fp32
// value is exactly the sum of three bf16 pieces, so K slots hold the products of
// the pieces and the matrix unit's fp32 sum is the product to its own rounding.
// The int32 block sums are turned into floats by the matrix unit too (magic
// below): what remains per output and block is a subtraction and an fma, the two
// VALU forms that run at twice the rate of the three-operand ones (2.4 - 2.9
// against 4.3 cycles per wave measured).
//
// What bounds it (Q8_0, N 14336 K 4096 M 2048: 505 us a call with the quantizer, 480
// TOPS; the chunked kernels it replaces 4170 us, which streamed the weights 64 times): with the
// products removed the loads and LDS writes alone take 350 of 128 x 128 tiles'
// time, with the loads removed the products 290; of the loads the 34-byte weight
// blocks are two thirds (64 rows touch 64 cache lines per load), so weights are
// read by pairs of blocks in 4-byte aligned pieces (567 -> 506 us on 64 x 64
// tiles). Errors against 64-bit sums are smaller than the replaced kernels'
// (7.5e-8 normwise against 0.96e-7 at K 4096, 1.8e-7 at K 18944).
#include <hip/hip_runtime.h>

#include "lp_chunks.h"
#include "lp_internal.h"

namespace lp {
namespace {

typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i16v __attribute__((ext_vector_type(16)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));
typedef short s4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// 16 bytes at any even address (global memory takes unaligned vector loads)
typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u32_a2 __attribute__((aligned(2)));

constexpr int kHalfStride = 528;                 // 32 rows x 16 B, padded
constexpr int kBlkStride = 2 * kHalfStride;      // two halves
constexpr int kTileBytes = 4 * kBlkStride;       // 32 rows x 128 elements

__device__ __forceinline__ u32x4 ld16(const uint8_t* p) { return *reinterpret_cast<const u32x4_a2*>(p); }

// bytes c (0..127) minus k (per byte, no borrow across bytes)
__device__ __forceinline__ uint32_t sub_bytes(uint32_t c, uint32_t k4) {
    return ((c | 0x80808080u) - k4) ^ 0x80808080u;
}

template <bool V>
struct Flag {
    static constexpr bool value = V;
};

struct I8tArgs {
    const uint8_t* w;
    ActView A;
    float* y;
    int M, N, K;
    size_t rb;
    int ntm, ntn;
    // grouped MoE rows: the route table (lp_route.h), its pairs' offset, bytes of one
    // expert's weights
    const uint8_t* route;
    int mg, multi, topk;
    long ebytes;
};

// Per-type staging of one 128-element stage of BN weight rows by GT threads.
// kMin: the type has a min term (-dmin * sum m * xs).
template <uint32_t T>
struct Traits {
    static constexpr bool kMin = T == T_Q4_K;
    static constexpr bool kSub16 = T == T_Q6_K;          // 16-element int8 scales
    static constexpr int kPieces = T == T_Q4_K ? 3 : 2;  // bf16 pieces of the block scale
    // staging tasks per row: a pair of blocks (Q8_0, Q4_0: their rows are 4-byte
    // aligned, as a pair is), a block (Q5_0), 16 bytes of codes (Q4_K, Q6_K)
    static constexpr int kTasks = T == T_Q4_K || T == T_Q5_0 ? 4 : 2;
};

template <uint32_t T>
struct WReg {
    u32x4 a, b, c, e;    // code bytes
    u32x4 h;             // header (Q4_K) or scales
    uint32_t d;
};
// 16 bytes at a 4-byte aligned address
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ u32x4 ld16_a4(const uint8_t* p) { return *reinterpret_cast<const u32x4_a4*>(p); }

// The thread's byte offset in the rows of a tile (local row n, task) and the
// load of stage s from it; base: the tile's first row. Offsets and the stage's
// uniform byte position keep the loads in the scalar-base + 32-bit-offset form.
template <uint32_t T>
__device__ __forceinline__ uint32_t w_off(int n, int task, uint32_t rb) {
    constexpr uint32_t per = T == T_Q8_0 ? 68 : T == T_Q4_0 ? 36 : T == T_Q5_0 ? 22 : 16;
    return (uint32_t)n * rb + (uint32_t)task * per;
}
template <uint32_t T>
__device__ __forceinline__ void w_load(WReg<T>& r, const uint8_t* base, uint32_t off, uint32_t last, int s, int task) {
    if constexpr (T == T_Q8_0 || T == T_Q4_0 || T == T_Q5_0) {
        // past K: the row's last blocks again
        const uint32_t o = off + (uint32_t)s * (T == T_Q8_0 ? 136u : T == T_Q4_0 ? 72u : 88u);
        const uint8_t* p = base + (o < last ? o : last);
        if constexpr (T == T_Q5_0) {
            r.d = load_u16(p);
            r.h.x = *reinterpret_cast<const u32_a2*>(p + 2);
            r.a = ld16(p + 6);
        } else {
            r.a = ld16_a4(p);
            r.b = ld16_a4(p + 16);
            if constexpr (T == T_Q8_0) {
                r.c = ld16_a4(p + 32);
                r.e = ld16_a4(p + 48);
            }
            r.d = *reinterpret_cast<const uint32_t*>(p + (T == T_Q8_0 ? 64 : 32));
        }
    } else if constexpr (T == T_Q4_K) {
        // task = 2 j + c: bytes 16c..16c+15 of the 64-element group j of this half
        const uint8_t* sb = base + (size_t)(s >> 1) * 144;
        r.h = *reinterpret_cast<const u32x4*>(sb + (off - 16u * task));
        r.a = *reinterpret_cast<const u32x4*>(sb + 16 + 64 * (s & 1) + off);
    } else {
        // Q6_K, task c: elements 16c..16c+15 of the half's four blocks
        const uint8_t* sb = base + (size_t)(s >> 1) * 210;
        const int h = s & 1;
        r.a = ld16(sb + 64 * h + off);
        r.b = ld16(sb + 64 * h + 32 + off);
        r.c = ld16(sb + 128 + 32 * h + off);
        const uint32_t o = off - 16u * task;
        const u32x2_a2 sc = *reinterpret_cast<const u32x2_a2*>(sb + 192 + 8 * h + o);
        r.h.x = sc.x;
        r.h.y = sc.y;
        r.d = load_u16(sb + 208 + o);
    }
}

// bits 31..16 of b above bits 31..16 of a: two bf16 in one dword (a first)
__device__ __forceinline__ uint32_t pk_hi(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float hi16(float v) { return __uint_as_float(__float_as_uint(v) & 0xffff0000u); }

// The operands of a scale product x (x) w on v_mfma_f32_32x32x8_bf16 (4 K slots
// for lanes < 32, 4 for the others), from the exact bf16 pieces x = x1 + x2 + x3
// and w = w1 + w2 (an fp16 value) or w1 + w2 + w3 (an fp16 value times a 6-bit
// one). bf16 ends at 2^-133, fp32 at 2^-149: x2 and x3 are held times 2^13 (x is at
// most 2^121.01, a 127th of an fp32 value) beside w times 2^-13, w', so that every x
// from 2^-123 up has its 24 bits (unscaled pieces of x 2^-126 kept 8) and a subnormal
// one those from 2^-146 up. Two pieces:
//                      x1 x1 x2 x2 . w1 w2 w1' w2' | 0 0 x3 x3 . w1 w2 w1' w2'
//          three:     x1 x1 x1 x2 . w1 w2 w3 w1' | x2 x2 x3 x3 . w2' w3' w1' w2'
// (all products but x3 w3, below 2^-32 of the whole). LDS holds them ready made,
// 8 bytes per lane.
constexpr float kUp = 0x1p13f;
constexpr uint32_t kDown = (13u << 7) * 0x00010001u;
constexpr float kMinUp = 0x1p6f;                          // of the Q4_K mins' product, its
constexpr uint32_t kMinDown = 6u << 23;                   // upper halves only
// Two bf16 divided by powers of two: their exponents less than they are by the halves
// of k, zeros left (the saturated difference; no piece here is below 2^-64).
__device__ __forceinline__ uint32_t down(uint32_t v, uint32_t k) {
    typedef unsigned short h2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(h2, v), __builtin_bit_cast(h2, k)));
}
template <int PIECES>
__device__ __forceinline__ void put_x(u32x2* lo, u32x2* hi, float x) {
    const float x1 = hi16(x), r = (x - x1) * kUp, x2 = hi16(r), x3 = r - x2;
    if constexpr (PIECES == 3) {
        *lo = u32x2{pk_hi(x1, x1), pk_hi(x1, x2)};
        *hi = u32x2{pk_hi(x2, x2), pk_hi(x3, x3)};
    } else {
        *lo = u32x2{pk_hi(x1, x1), pk_hi(x2, x2)};
        *hi = u32x2{0u, pk_hi(x3, x3)};
    }
}
template <int PIECES>
__device__ __forceinline__ void put_w(u32x2* lo, u32x2* hi, float w) {
    const float w1 = hi16(w), r = w - w1;
    if constexpr (PIECES == 3) {
        const float w2 = hi16(r), w3 = r - w2;
        const uint32_t p = pk_hi(w1, w2), q = down(p, kDown);
        *lo = u32x2{p, __builtin_amdgcn_perm(q, __float_as_uint(w3), 0x05040302u)};
        *hi = u32x2{down(pk_hi(w2, w3), kDown), q};
    } else {
        const uint32_t p = pk_hi(w1, r);
        *lo = u32x2{p, down(p, kDown)};
    }
}

// LDS of one K group's stage: codes of BM tokens and BN rows, then 8-byte
// records: xd [4 blocks][2 lane halves][BM], wd [4][1 half, Q4_K 2][BN] (Q6_K:
// [BN], d); Q6_K: ex [4][BN], a block's two scales as floats; Q4_K: floats ex
// [4][BN] mins, xs [4][BM], dm [BN].
template <uint32_t T, int BM, int BN>
struct Lay {
    static constexpr int a = 0;
    static constexpr int w = a + BM / 32 * kTileBytes;
    static constexpr int xd = w + BN / 32 * kTileBytes;
    static constexpr int wd = xd + 64 * BM;
    static constexpr int ex = wd + (T == T_Q6_K ? 8 : T == T_Q4_K ? 64 : 32) * BN;
    static constexpr int xs = ex + (T == T_Q6_K ? 32 * BN : T == T_Q4_K ? 16 * BN : 0);
    static constexpr int dm = xs + (T == T_Q4_K ? 16 * BM : 0);
    static constexpr int bytes = (dm + (T == T_Q4_K ? 4 * BN : 0) + 15) & ~15;
};

template <uint32_t T, int BM, int BN>
__device__ __forceinline__ void w_store(const WReg<T>& r, uint8_t* st, int n, int b0, int task) {
    typedef Lay<T, BM, BN> L;
    uint8_t* wt = st + L::w + (n >> 5) * kTileBytes + (n & 31) * 16;
    u32x2* wd = reinterpret_cast<u32x2*>(st + L::wd);
    if constexpr (T == T_Q8_0) {
        // dwords 0..16 of two 34-byte blocks: the codes of the first are 2 bytes off
        const uint32_t w[17] = {r.a[0], r.a[1], r.a[2], r.a[3], r.b[0], r.b[1], r.b[2], r.b[3], r.c[0],
                                r.c[1], r.c[2], r.c[3], r.e[0], r.e[1], r.e[2], r.e[3], r.d};
        uint8_t* const q = wt + 2 * task * kBlkStride;
        u32x4 v[4];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            v[i >> 2][i & 3] = alignb(w[i + 1], w[i], 2);
            v[2 + (i >> 2)][i & 3] = w[9 + i];
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            *reinterpret_cast<u32x4*>(q + u * kBlkStride) = v[2 * u];
            *reinterpret_cast<u32x4*>(q + u * kBlkStride + kHalfStride) = v[2 * u + 1];
            put_w<2>(wd + (2 * task + u) * BN + n, nullptr, fp16_bits_to_f32(u ? w[8] >> 16 : w[0]));
        }
    } else if constexpr (T == T_Q4_0) {
        const uint32_t w[9] = {r.a[0], r.a[1], r.a[2], r.a[3], r.b[0], r.b[1], r.b[2], r.b[3], r.d};
        uint8_t* const q = wt + 2 * task * kBlkStride;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            u32x4 lo, hi;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t c = u ? w[5 + i] : alignb(w[i + 1], w[i], 2);
                lo[i] = sub_bytes(c & 0x0f0f0f0fu, 0x08080808u);
                hi[i] = sub_bytes((c >> 4) & 0x0f0f0f0fu, 0x08080808u);
            }
            *reinterpret_cast<u32x4*>(q + u * kBlkStride) = lo;
            *reinterpret_cast<u32x4*>(q + u * kBlkStride + kHalfStride) = hi;
            put_w<2>(wd + (2 * task + u) * BN + n, nullptr, fp16_bits_to_f32(u ? w[4] >> 16 : w[0]));
        }
    } else if constexpr (T == T_Q5_0) {
        u32x4 lo, hi;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // four bits of qh spread to bit 4 of the four bytes
            const uint32_t l5 = (((r.h.x >> (4 * i)) & 15u) * 0x00204081u & 0x01010101u) << 4;
            const uint32_t h5 = (((r.h.x >> (16 + 4 * i)) & 15u) * 0x00204081u & 0x01010101u) << 4;
            lo[i] = sub_bytes((r.a[i] & 0x0f0f0f0fu) | l5, 0x10101010u);
            hi[i] = sub_bytes(((r.a[i] >> 4) & 0x0f0f0f0fu) | h5, 0x10101010u);
        }
        *reinterpret_cast<u32x4*>(wt + task * kBlkStride) = lo;
        *reinterpret_cast<u32x4*>(wt + task * kBlkStride + kHalfStride) = hi;
        put_w<2>(wd + task * BN + n, nullptr, fp16_bits_to_f32(r.d));
    } else if constexpr (T == T_Q4_K) {
        const int j = task >> 1, c = task & 1;
        u32x4 lo, hi;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = r.a[i] & 0x0f0f0f0fu;
            hi[i] = (r.a[i] >> 4) & 0x0f0f0f0fu;
        }
        *reinterpret_cast<u32x4*>(wt + (2 * j) * kBlkStride + c * kHalfStride) = lo;
        *reinterpret_cast<u32x4*>(wt + (2 * j + 1) * kBlkStride + c * kHalfStride) = hi;
        // this task's block: 2j + c
        const int b = (b0 & 4) + 2 * j + c;
        uint32_t sc, mn;
        scale_min_k4(b, r.h.y, r.h.z, r.h.w, sc, mn);
        put_w<3>(wd + 2 * task * BN + n, wd + (2 * task + 1) * BN + n, fp16_bits_to_f32(r.h.x) * (float)sc);
        reinterpret_cast<float*>(st + L::ex)[task * BN + n] = (float)mn;
        if (task == 0) reinterpret_cast<float*>(st + L::dm)[n] = fp16_bits_to_f32(r.h.x >> 16);
    } else {
        const int c = task;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            u32x4 q;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t l = g & 1 ? r.b[i] : r.a[i];
                const uint32_t nib = (g & 2 ? l >> 4 : l) & 0x0f0f0f0fu;
                const uint32_t hb = 2 * g <= 4 ? (r.c[i] << (4 - 2 * g)) : (r.c[i] >> 2);
                q[i] = sub_bytes(nib | (hb & 0x30303030u), 0x20202020u);
            }
            *reinterpret_cast<u32x4*>(wt + g * kBlkStride + c * kHalfStride) = q;
        }
        // blocks 2c and 2c + 1: their two int8 scales
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const uint32_t s = c ? r.h.y : r.h.x;
            const int s0 = (int)(s << (24 - 16 * u)) >> 24, s1 = (int)(s << (16 - 16 * u)) >> 24;
            reinterpret_cast<float2*>(st + L::ex)[(2 * c + u) * BN + n] = make_float2((float)s0, (float)s1);
        }
        if (c == 0) put_w<2>(wd + n, nullptr, fp16_bits_to_f32(r.d));
    }
}

// One output by the whole wave in fp32, as the few-row kernels form it. An infinite
// block scale has no pieces (inf - inf), so its product above is NaN where the plain
// one is an infinity: non-finite outputs are made again here, except in rows whose
// own scales are not finite (a NaN or infinite activation), which are NaN either way.
// Measured (us a call, Q8_0 N 4096 K 4096 M 512, plain 45 - 50): one infinite scale in the
// matrix 89, a NaN activation row 48; N 14336 M 2048 504, 516 with one infinite scale.
template <uint32_t T>
__device__ __forceinline__ float wave_dot(const ActView& A, int arow, const uint8_t* wrow, int K, int lane) {
    float s = 0.0f;
    if constexpr (T == T_Q5_0) {
        const int8_t* q = A.qs + (size_t)arow * K;
        for (int b = lane; b < K >> 5; b += 64) {
            const uint8_t* blk = wrow + b * 22;
            const uint32_t qh = load_u16(blk + 2) | load_u16(blk + 4) << 16;
            int P = 0;
            for (int e = 0; e < 32; e++) {
                const int nib = e < 16 ? blk[6 + e] & 15 : blk[6 + e - 16] >> 4;
                P += ((nib | (int)((qh >> e) & 1u) << 4) - 16) * q[32 * b + e];
            }
            s = fmaf(fp16_bits_to_f32(load_u16(blk)) * A.d[(size_t)arow * (K >> 5) + b], (float)P, s);
        }
    } else {
        for (int c = lane; c < K >> 6; c += 64) {
            typename Chunk<T>::Act a;
            typename Chunk<T>::Wt w;
            int is[Chunk<T>::NSUB];
            load_act<T>(A, K, arow, c, a);
            Chunk<T>::load_w(wrow, c, w);
            Chunk<T>::isums(w, a, is);
            s += Chunk<T>::partial(w, a, is, c);
        }
    }
    return wave_sum(s);
}
__device__ __forceinline__ bool finite(float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; }

// MT x NT tiles of 32 x 32 per wave. MOE: a token tile is a routed group (expert,
// first pair, n <= BM pairs); its rows are gathered and scattered by pair.
template <uint32_t T, int MT, int NT, int WM, int WN, int WK, bool MOE>
__global__ void __launch_bounds__(64 * WM * WN * WK, 2)
gemm_i8t(I8tArgs g) {
    constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN, GT = 64 * WM * WN;
    typedef Lay<T, BM, BN> L;
    typedef Traits<T> R;
    constexpr int APT = BM * 8 / GT, XPT = (BM * 4 + GT - 1) / GT, WPT = (BN * R::kTasks + GT - 1) / GT;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x % GT, kg = WK > 1 ? (int)(threadIdx.x / GT) : 0;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    // a group of one wave needs no barrier and one buffer: its LDS operations are in order
    constexpr int NBUF = GT == 64 ? 1 : 2;
    uint8_t* const lds = smem + kg * NBUF * L::bytes;

    // Each XCD takes a contiguous run of tiles (blocks are dealt to the 8 XCDs in
    // turn), ordered in groups of kGroup token tiles that walk the weight tiles
    // together: the tiles in flight on an XCD then form a near-square block, whose
    // operands its L2 serves
    const int bid = blockIdx.x;
    if constexpr (MOE) {
        g.ntm = *reinterpret_cast<const int*>(g.route);
        if (bid >= g.ntm * g.ntn) return;
    }
    const int ntiles = g.ntm * g.ntn;
    const int q8 = ntiles >> 3, r8 = ntiles & 7, xcd = bid & 7;
    const int tile = xcd * q8 + (xcd < r8 ? xcd : r8) + (bid >> 3);
    constexpr int kGroup = MOE ? 1 : 512 / BM;
    const int grp = tile / (kGroup * g.ntn), in = tile - grp * kGroup * g.ntn;
    const int gm = g.ntm - grp * kGroup < kGroup ? g.ntm - grp * kGroup : kGroup;
    int m0 = (grp * kGroup + in % gm) * BM;
    const int n0 = in / gm * BN;
    const int* pairs = nullptr;
    if constexpr (MOE) {
        const int4 gd = reinterpret_cast<const int4*>(g.route + 16)[grp];
        pairs = reinterpret_cast<const int*>(g.route + 16 + (size_t)g.mg * 16) + gd.y;
        g.w += gd.x * g.ebytes;
        g.M = gd.z;
        m0 = 0;
    }
    auto arow = [&](int m) {                     // the activation row of a token
        if constexpr (!MOE) return m;
        const int p = pairs[m];
        return g.multi ? p : p / g.topk;
    };
    auto yrow = [&](int m) { return (size_t)(MOE ? pairs[m] : m) * g.N; };
    const int nb = g.K >> 5;
    const int nst = (nb + 3) >> 2, iters = (nst + 2 * WK - 1) / (2 * WK);

    u32x4 ra[APT];
    float rx[XPT], rs[R::kMin ? XPT : 1];
    WReg<T> rw[WPT];
    uint32_t aoff[APT], xoff[XPT], woff[WPT], wlast[WPT];
#pragma unroll
    for (int i = 0; i < APT; i++) {
        const int p = tid + i * GT, m = m0 + (p >> 3) < g.M ? p >> 3 : g.M - 1 - m0;
        aoff[i] = (uint32_t)arow(m) * (uint32_t)g.K + 16u * (p & 7);
    }
#pragma unroll
    for (int i = 0; i < XPT; i++) {
        const int p = tid + i * GT, row = BM * 4 % GT == 0 || p < BM * 4 ? p >> 2 : 0;
        const int m = m0 + row < g.M ? row : g.M - 1 - m0;
        xoff[i] = (uint32_t)arow(m) * (uint32_t)nb + (p & 3);
    }
#pragma unroll
    for (int i = 0; i < WPT; i++) {
        const int p = tid + i * GT, row = BN * R::kTasks % GT == 0 || p < BN * R::kTasks ? p / R::kTasks : 0;
        const int n = n0 + row < g.N ? row : g.N - 1 - n0;
        woff[i] = w_off<T>(n, p % R::kTasks, (uint32_t)g.rb);
        wlast[i] = (uint32_t)n * (uint32_t)g.rb + (T == T_Q5_0 ? (uint32_t)(nb - 1) * 22u : (uint32_t)(nb - 2) * (T == T_Q8_0 ? 34u : 18u));
    }
    const int8_t* const abase = g.A.qs + (size_t)m0 * g.K;
    const float* const xbase = g.A.d + (size_t)m0 * nb;
    const float* const sbase = R::kMin ? g.A.sum + (size_t)m0 * nb : nullptr;
    const uint8_t* const wbase = g.w + (size_t)n0 * g.rb;
    // No load depends on a branch (a value merged from two paths would be waited
    // for where they meet). A stage past K re-reads the last one. Where K ends
    // inside a stage, codes and scales past it come from the workspace's next
    // bytes and from the row's last block; store() zeroes their activation scales.
    auto load = [&](int s) {
        s = s < nst ? s : nst - 1;
#pragma unroll
        for (int i = 0; i < APT; i++) ra[i] = *reinterpret_cast<const u32x4*>(abase + (size_t)s * 128 + aoff[i]);
#pragma unroll
        for (int i = 0; i < XPT; i++) {
            rx[i] = xbase[(size_t)s * 4 + xoff[i]];
            if constexpr (R::kMin) rs[i] = sbase[(size_t)s * 4 + xoff[i]];
        }
#pragma unroll
        for (int i = 0; i < WPT; i++) w_load<T>(rw[i], wbase, woff[i], wlast[i], s, (tid + i * GT) % R::kTasks);
    };
    auto store = [&](int s, uint8_t* st) {
        const int b0 = 4 * s;
#pragma unroll
        for (int i = 0; i < APT; i++) {
            const int p = tid + i * GT, row = p >> 3, pc = p & 7;
            *reinterpret_cast<u32x4*>(st + L::a + (row >> 5) * kTileBytes + (pc >> 1) * kBlkStride +
                                      (pc & 1) * kHalfStride + (row & 31) * 16) = ra[i];
        }
#pragma unroll
        for (int i = 0; i < XPT; i++) {
            const int p = tid + i * GT;
            if (BM * 4 % GT == 0 || p < BM * 4) {
                u32x2* xd = reinterpret_cast<u32x2*>(st + L::xd) + 2 * (p & 3) * BM + (p >> 2);
                put_x<R::kPieces>(xd, xd + BM, b0 + (p & 3) < nb ? rx[i] : 0.0f);
                if constexpr (R::kMin) reinterpret_cast<float*>(st + L::xs)[(p & 3) * BM + (p >> 2)] = b0 + (p & 3) < nb ? rs[i] : 0.0f;
            }
        }
#pragma unroll
        for (int i = 0; i < WPT; i++) {
            const int p = tid + i * GT;
            if (BN * R::kTasks % GT == 0 || p < BN * R::kTasks)
                w_store<T, BM, BN>(rw[i], st, p / R::kTasks, b0, p % R::kTasks);
        }
    };

    // Every two stages (256 elements) the fp32 chain of block terms is added to
    // the output's sum in 64 bits and starts again: a single fp32 chain over K/32
    // blocks rounds 2-3 times worse than the K-sliced sums of the small-M kernels,
    // and with 64-bit sums of the same 256-element chains the forms below, which
    // split K over 1 to 8 groups of waves, agree to the last fp32 bit (up to the
    // 64-bit sums' own rounding), so a row does not depend on the rows beside it.
    float acc[MT][NT][16];
    double sum[MT][NT][16];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < NT; r++)
#pragma unroll
            for (int i = 0; i < 16; i++) sum[t][r][i] = 0.0;
    auto flush = [&] {
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < NT; r++)
#pragma unroll
                for (int i = 0; i < 16; i++) sum[t][r][i] += (double)acc[t][r][i];
    };

    const int col = lane & 31, half = lane >> 5;
    const bool upper = half != 0;
    // int32 block sums come out of the matrix unit on top of the bits of 1.5 * 2^23,
    // i.e. as floats 12582912 + P (|P| < 2^22): one subtraction instead of a
    // conversion, which takes twice as long
    constexpr float kMagic = 12582912.0f;
    i16v magic;
#pragma unroll
    for (int i = 0; i < 16; i++) magic[i] = __float_as_int(kMagic);
    asm volatile("" : "+v"(magic));
    auto compute = [&](auto first, const uint8_t* st) {
        constexpr bool FIRST = decltype(first)::value;
        constexpr int KS = R::kSub16 ? 2 : 1;          // products per block
        const uint8_t* at = st + L::a + wm * MT * kTileBytes + col * 16 + half * (R::kSub16 ? 8 : kHalfStride);
        const uint8_t* wt = st + L::w + wn * NT * kTileBytes + col * 16 + half * (R::kSub16 ? 8 : kHalfStride);
        const s4v* xd = reinterpret_cast<const s4v*>(st + L::xd) + half * BM + wm * MT * 32 + col;
        const s4v* wd = reinterpret_cast<const s4v*>(st + L::wd) + (R::kPieces == 3 ? half * BN : 0) + wn * NT * 32 + col;
        const float2* ex = reinterpret_cast<const float2*>(st + L::ex) + wn * NT * 32 + col;
        // Operands of block b + 1 are requested while block b computes.
        i4v A[2][MT], B[2][NT];
        long A2[2][MT][2], B2[2][NT][2];
        s4v xv[2][MT], wv[2][NT];
        float2 ev[2][NT];
        auto frags = [&](int b, int k) {
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const uint8_t* p = at + t * kTileBytes + b * kBlkStride;
                if constexpr (R::kSub16) {
                    A2[k][t][0] = *reinterpret_cast<const long*>(p);
                    A2[k][t][1] = *reinterpret_cast<const long*>(p + kHalfStride);
                } else {
                    A[k][t] = *reinterpret_cast<const i4v*>(p);
                }
                xv[k][t] = xd[2 * b * BM + 32 * t];
            }
#pragma unroll
            for (int r = 0; r < NT; r++) {
                const uint8_t* p = wt + r * kTileBytes + b * kBlkStride;
                if constexpr (R::kSub16) {
                    B2[k][r][0] = *reinterpret_cast<const long*>(p);
                    B2[k][r][1] = *reinterpret_cast<const long*>(p + kHalfStride);
                    wv[k][r] = wd[32 * r];
                    ev[k][r] = ex[b * BN + 32 * r];
                } else {
                    B[k][r] = *reinterpret_cast<const i4v*>(p);
                    wv[k][r] = wd[(R::kPieces == 3 ? 2 : 1) * b * BN + 32 * r];
                }
            }
        };
        constexpr int NTILE = MT * NT;
        f16v S, P[KS];
        auto issue = [&](int i) {
            const int k = (i / NTILE) & 1, t = i % NTILE % MT, r = i % NTILE / MT;
            S = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(xv[k][t], wv[k][r], f16v{}, 0, 0, 0);
            if constexpr (R::kSub16) {
#pragma unroll
                for (int c = 0; c < 2; c++)
                    P[c] = __builtin_bit_cast(f16v, __builtin_amdgcn_mfma_i32_32x32x16_i8(A2[k][t][c], B2[k][r][c],
                                                                                               magic, 0, 0, 0));
            } else {
                P[0] = __builtin_bit_cast(f16v, __builtin_amdgcn_mfma_i32_32x32x32_i8(A[k][t], B[k][r], magic, 0, 0, 0));
            }
        };
        frags(0, 0);
        issue(0);
#pragma unroll
        for (int i = 0; i < 4 * NTILE; i++) {
            const int b = i / NTILE, k = b & 1, t = i % NTILE % MT, r = i % NTILE / MT;
            if (i % NTILE == 0 && b < 3) frags(b + 1, k ^ 1);
#pragma unroll
            for (int q = 0; q < 16; q++) {
                float v = P[0][q] - kMagic;
                if constexpr (R::kSub16) {
                    v *= ev[k][r].x;
                    v = fmaf(P[1][q] - kMagic, ev[k][r].y, v);     // exact: below 2^24
                }
                if (FIRST && b == 0) acc[t][r][q] = v * S[q];
                else acc[t][r][q] = fmaf(v, S[q], acc[t][r][q]);
            }
            // the sums are made here: the compiler would sink them to their use at
            // the end of the stage and keep every block's products until then
#pragma unroll
            for (int q = 0; q < 16; q++) asm volatile("" : "+v"(acc[t][r][q]));
            if (i + 1 < 4 * NTILE) issue(i + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (R::kMin) {
            // sum over the stage's four blocks of m * xs: K slots of lane half h
            // are blocks 2h, 2h + 1, three pieces of xs each, the second and third
            // times 2^6 beside m' = m times 2^-6 (as x2 and x3 of put_x; xs goes up to 2^128)
            const float* xs = reinterpret_cast<const float*>(st + L::xs) + wm * MT * 32 + col;
            const float* mn = reinterpret_cast<const float*>(st + L::ex) + wn * NT * 32 + col;
            const float* dm = reinterpret_cast<const float*>(st + L::dm) + wn * NT * 32 + col;
            b8v xa[MT];
#pragma unroll
            for (int t = 0; t < MT; t++) {
                u32x4 o;
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const float x = xs[(2 * half + u) * BM + 32 * t];
                    const float x1 = hi16(x), q = (x - x1) * kMinUp, x2 = hi16(q);
                    o[2 * u] = pk_hi(x1, x2);
                    o[2 * u + 1] = pk_hi(q - x2, 0.0f);
                }
                xa[t] = __builtin_bit_cast(b8v, o);
            }
#pragma unroll
            for (int r = 0; r < NT; r++) {
                u32x4 o;
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const float m = mn[(2 * half + u) * BN + 32 * r];
                    o[2 * u] = down(pk_hi(m, m), kMinDown);
                    o[2 * u + 1] = o[2 * u] >> 16;
                }
                const b8v mb = __builtin_bit_cast(b8v, o);
                const float nd = -dm[32 * r];
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    const f16v S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[t], mb, f16v{}, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[t][r][i] = fmaf(nd, S[i], acc[t][r][i]);
                }
            }
        }
    };

    // While stage s computes from one LDS buffer, stage s + 1 is loaded into
    // registers and then written to the other.
    // a wave whose token tile is past the group's pairs only stages
    const bool busy = !MOE || WM == 1 || wm * MT * 32 < g.M;
    // Group kg takes the pairs kg, kg + WK, .. of stages.
    load(2 * kg);
    store(2 * kg, lds);
    __syncthreads();
    auto stage = [&](auto first, int next) {
        constexpr bool FIRST = decltype(first)::value;
        load(next);
        if (busy) compute(first, lds + (FIRST || NBUF == 1 ? 0 : L::bytes));
        if constexpr (NBUF == 1) __builtin_amdgcn_wave_barrier();
        store(next, lds + (FIRST && NBUF == 2 ? L::bytes : 0));
        if constexpr (NBUF == 1) __builtin_amdgcn_wave_barrier();
        else __syncthreads();
    };
    for (int it = 0; it < iters; it++) {
        const int s = 2 * (it * WK + kg);
        stage(Flag<true>{}, s + 1);
        // few stages per group: the last one does not wait for a load nobody needs
        // (the same call 11.6 -> 11.0 us)
        if (WK > 1 && it == iters - 1) {
            if (busy) compute(Flag<false>{}, lds + (NBUF == 1 ? 0 : L::bytes));
            flush();
            break;
        }
        stage(Flag<false>{}, s + 2 * WK);
        if (busy) flush();
    }
    bool bad = false;
    // register j = (t * NT + r) * 16 + i of a lane: its token and weight row (the lane's
    // number is read again, so that the part below keeps no register through the loop:
    // two more than 168 cost a wave per SIMD)
    const int ln = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    auto mrow = [&](int j) { return m0 + (wm * MT + (j >> 4) / NT) * 32 + 8 * ((j & 15) >> 2) + 4 * (ln >> 5) + (j & 3); };
    auto nrow = [&](int j) { return n0 + (wn * NT + (j >> 4) % NT) * 32 + (ln & 31); };
    auto put = [&](int j, float v) {
        const int m = mrow(j), n = nrow(j);
        if (m < g.M && n < g.N) g.y[yrow(m) + n] = v;
    };
    if constexpr (WK > 1) {
        __syncthreads();      // every wave is done with its buffer
        // All groups leave their sums in LDS; group kg adds those of registers kg,
        // kg + WK, .. in the groups' order (against one group adding the others' one
        // after the other: Q8_0 N 4096 K 4096 M 16 13.1 -> 11.6 us with the quantizer).
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
            bad |= !finite((float)u);
            put(j, (float)u);
        }
    } else {
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < NT; r++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    bad |= !finite((float)sum[t][r][i]);
                    put((t * NT + r) * 16 + i, (float)sum[t][r][i]);
                }
    }
    // (without the hint the MoE prompt's kernel is laid out worse: 424 -> 459 us a layer)
    if (__builtin_expect(!__any(bad), 1)) return;
    for (int j = kg; j < MT * NT * 16; j += WK) {
        const int m = mrow(j), n = nrow(j);
        const bool in = m < g.M && n < g.N;
        float* const y = g.y + (in ? yrow(m) + n : 0);
        uint64_t left = __ballot(in && !finite(*y));
        if (!left) continue;
        // each half's 32 lanes look through the scales of its row
        bool nan = false;
        if (m < g.M)
            for (int b = ln & 31; b < nb; b += 32) nan |= !finite(g.A.d[(size_t)arow(m) * nb + b]);
        const uint64_t nans = __ballot(nan);
        if ((uint32_t)nans) left &= ~0xffffffffull;
        if (nans >> 32) left &= 0xffffffffull;
        for (; left; left &= left - 1) {
            const int l = __ffsll((unsigned long long)left) - 1;
            const int row = __builtin_amdgcn_readlane(n, l);
            const float v = wave_dot<T>(g.A, arow(__builtin_amdgcn_readlane(m, l)), g.w + (size_t)row * g.rb, g.K, ln);
            if (ln == l) *y = v;
        }
    }
}

template <uint32_t T, int MT, int NT, int WM, int WN, int WK, bool MOE = false>
hipError_t launch_cfg(I8tArgs g, hipStream_t st) {
    constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN;
    constexpr int red = WK > 1 ? WK * WM * WN * MT * NT * 8192 : 0;
    constexpr int bufs = WK * (WM * WN == 1 ? 1 : 2) * Lay<T, BM, BN>::bytes;
    constexpr int lds = bufs > red ? bufs : red;
    static_assert(lds <= 160 * 1024, "LDS");
    if (!MOE) g.ntm = (g.M + BM - 1) / BM;
    g.ntn = (g.N + BN - 1) / BN;
    hipLaunchKernelGGL((gemm_i8t<T, MT, NT, WM, WN, WK, MOE>), dim3((unsigned)(g.ntm * g.ntn)), dim3(64 * WM * WN * WK), lds,
                       st, g);
    return hipGetLastError();
}

}  // namespace

namespace {
// The tile forms, most parallel first. Measured (us per product, CUs 256, K 4096
// unless said; t32 / t64 / t128 are the tile counts):
//   Q8_0 N 4096 M 64     (t32 256)   32x32x8 12.6  64x64x2 24.6  64x64 30.9  128x128 65
//   Q8_0 N 4096 M 128    (t32 512)   32x32x4 17.2  32x32x8 21.9  64x64x2 25.0
//   Q8_0 N 4096 M 256    (t64 256)   64x64x2 27.1  32x32x4 31.0  64x64 33.3
//   Q8_0 N 4096 M 512    (t64 512)   64x64 46.2  64x64x2 52.7  128x128 69
//   Q8_0 N 4096 M 1024   (t128 256)  128x128 76.9  64x64 83.9
//   Q6_K N 14336 M 2048  (t128 1792) 128x128 740  64x64 830
// Short rows have fewer stage pairs than eight groups: with four the call loses the
// idle ones and half the last sum (kernel time with the quantizer, M 12, N 2048: K 256
// 8.3 -> 7.1, K 1024 8.6 -> 7.3, Q6_K 10.3 -> 8.4; K 1536 8.6 against 9.0), and where one
// pair is all of K and there are more tiles than CUs, four waves side by side read x once
// (Q6_K N 14336 K 256 10.2 -> 8.8, N 32768 16.3 -> 9.1, Q4_0 12.6 -> 7.5; at K 512 only
// from four tiles per CU, Q6_K N 32768 16.0 -> 11.9, N 14336 slower).
enum Form { F32X128, F32X32X8, F32X32X4, F64X64X2, F64X64, F128X128 };

Form pick_form(uint32_t type, int M, int K, int N) {
    const long cus = device_cu_count();
    auto tiles = [&](int b) { return (long)((M + b - 1) / b) * ((N + b - 1) / b); };
    // one 32 x 32 tile per CU: eight waves share its K; two per CU (or at most
    // 32 rows, where larger tiles are half padding): four waves
    if (tiles(32) <= cus) return K <= 1024 ? F32X32X4 : F32X32X8;
    if (M <= 32 && (K <= 256 || (K <= 512 && tiles(32) >= 4 * cus))) return F32X128;
    if (tiles(32) <= 2 * cus || M <= 32) return F32X32X4;
    if (tiles(64) <= cus) return F64X64X2;
    // two 64 x 64 workgroups per CU against one of 128 x 128, which does four
    // tiles' work in 1.55 - 1.9 times a round's time. The K-quants' 64 x 64
    // workgroups run in whole rounds of two per CU; the smaller Q8_0 / Q4_0 /
    // Q5_0 ones even out over the rounds.
    const bool kq = type == T_Q4_K || type == T_Q6_K;
    const long t64 = tiles(64), r128 = (tiles(128) + cus - 1) / cus;
    const double r64 = kq ? (double)((t64 + 2 * cus - 1) / (2 * cus)) : (double)t64 / (2 * cus);
    return r128 * (kq ? 1.6 : 1.9) < r64 ? F128X128 : F64X64;
}

template <uint32_t T>
hipError_t launch_t(const I8tArgs& g, Form f, hipStream_t st) {
    switch (f) {
        // (Q4_K comes here with more than 32 rows)
        case F32X128: if constexpr (T != T_Q4_K) return launch_cfg<T, 1, 1, 1, 4, 1>(g, st); return hipErrorInvalidValue;
        case F32X32X8: return launch_cfg<T, 1, 1, 1, 1, 8>(g, st);
        case F32X32X4: return launch_cfg<T, 1, 1, 1, 1, 4>(g, st);
        case F64X64X2: return launch_cfg<T, 1, 1, 2, 2, 2>(g, st);
        case F64X64: return launch_cfg<T, 1, 1, 2, 2, 1>(g, st);
        default: return launch_cfg<T, 2, 1, 2, 4, 1>(g, st);
    }
}
}  // namespace

// Where this kernel is the fastest one (weights aligned as the entry points check).
// Up to 32 rows its time depends on K alone (8 to 12 us with the quantizer), a GEMV's
// on N too: up to 8 rows the line is a number of outputs. Measured (us, GEMV against
// this): Q8_0 K 4096: N 1024 M 8 9.9 / 11.3, N 2048 M 5 9.9 / 11.2, N 4096 M 5 13.6 /
// 10.9, M 8 19.2 / 10.8; K 1024 N 4096 M 5 7.9 / 8.7, M 8 9.9 / 8.2; Q4_0 N 2048 M 5
// 9.4 / 11.0, N 4096 M 5 11.6 / 10.3; Q5_0 N 2048 M 8 11.1 / 13.6, N 4096 M 8 13.5 /
// 12.4. Beyond 8 rows their GEMVs run twice (N 14336 K 4096 M 16: Q4_0 65.8 -> 15.4,
// Q5_0 69 -> 18.9; Q8_0's 16-row kernel 54.9 -> 17.0; N 1024 K 1024 8.5 -> 8.3).
// Q6_K from 9 rows where 32-row tiles fill the CUs (N 14336 M 9 37.0 -> 20.6), else
// from 13 (K 4096, N 512 .. 4096: M 13 13.8 -> 13.2, M 17 18.8 -> 13.3, N 4096 M 512
// 382 -> 65; N 3584 K 18944 M 512 1327 -> 270). Short rows (K 1024: M 13 8.6 / 8.7,
// M 16 8.8 / 8.4; K 1536 M 16 9.3 / 10.5) stay there up to 15 rows, and 16 below K = 1024:
// from there on, 16 rows give the bits of the first 16 of a longer prompt.
// Q4_K where the 16-row chunks of the small-M kernel end (beyond 32 rows, 64 for
// up to 4096 weight rows) while one round of 128 x 128 tiles covers the product,
// and for K > 4096 not where that round would be half empty (N 14336 M 64 42 -> 27,
// M 256 82 -> 74.5, M 512 108 against 143 here; N 4096 M 512 59 -> 48, M 1024 94
// -> 77; N 4096 K 14336 M 256 102 -> 87, M 512 146 against 154 here, M 1024 266
// -> 250): beyond, the split-precision kernels' cheaper epilogue wins. It also wins at
// long K where this product's tiles are mostly padding: up to 64 rows on more than a 64 x 64
// tile per CU (K 4096: N 18944 M 33 39 / 48, M 64 46 / 48, N 28672 M 33 43 / 48, M 56 48 / 49, N 32768
// M 40 50 / 49; K 3072: N 24576 M 40 35 / 38, N 28672 M 48 39 / 39, N 32768 M 33 40 / 39; K 2048:
// N 18944 M 33 25 / 26, M 64 32 / 27), and 129..192 rows where the wide-token kernel fills the
// CUs (K 4096: N 14336 M 129 63 / 72, M 176 69 / 72, M 192 72 / 73, N 16384 M 144 70 / 72, M 160 74 / 72,
// N 12288, not that kernel, 81 / 72; K 5120 N 14336 M 129 78 / 88; K 3072 N 14336 M 129 53 / 56, M 160
// 57 / 56; K 2048 43 / 39).
// Q4_0 rows beyond 12000 on few weight rows: the GEMVs' two passes do not grow with K there
// (N 512 K 14336 M 9 18.5 / 22.3, M 12 21.7 / 22.5, M 13 22.8 / 22.5; K 18944 M 12 22.0 / 29.2; N 768
// K 14336 M 11 20.8 / 22.5, K 18944 M 9 30.7 / 29.1; N 1024 K 14336 M 9 22.3 / 22.5, M 10 25.1 / 22.5).
bool i8t_preferred(uint32_t type, int M, int K, int N) {
    const long cus = device_cu_count();
    switch (type) {
        case T_Q4_0:
            if (M <= 16 && N <= (K <= 16384 ? 768 : 512) && K > 650 * (10 + M)) return false;
            [[fallthrough]];
        case T_Q8_0: case T_Q5_0:
            return M > 8 || (M >= 5 && (long)M * N >= (type == T_Q5_0 || K < 2048 ? 32768 : 20000));
        case T_Q6_K: return M > 16 || (M >= (K < 2048 ? 16 : 13) && K >= 1024) || (M >= 9 && (N + 31) / 32 > cus);
        case T_Q4_K: {
            if (M <= 32 || (M <= 64 && N <= 4096)) return false;
            const long t64 = (long)((M + 63) / 64) * ((N + 63) / 64), t128 = (long)((M + 127) / 128) * ((N + 127) / 128);
            const long mn = (long)M * N;
            if (K >= 3072 && M <= 64 && t64 > cus && mn <= (K >= 4096 ? 1500000 : 1200000)) return false;
            if (K >= 3072 && M > 128 && M <= 192 && wt_auto_cfg(M, K, N) == 0 && mn <= (K >= 4096 ? 2600000 : 2100000))
                return false;
            return t128 <= cus && (K <= 4096 || t64 <= cus || 4 * t128 > 3 * cus);
        }
    }
    return false;
}

const char* i8t_form(uint32_t type, int M, int K, int N) {
    switch (pick_form(type, M, K, N)) {
        case F32X128: return "i8t 32x128";
        case F32X32X8: return "i8t 32x32x8";
        case F32X32X4: return "i8t 32x32x4";
        case F64X64X2: return "i8t 64x64x2";
        case F64X64: return "i8t 64x64";
        default: return "i8t 128x128";
    }
}

hipError_t launch_gemm_i8t(uint32_t type, const uint8_t* w, const ActView& A, float* y, int M, int K, int N,
                           hipStream_t st) {
    if (M <= 0 || N <= 0) return hipSuccess;
    I8tArgs g{w, A, y, M, N, K, row_bytes(type, K)};
    const Form f = pick_form(type, M, K, N);
    switch (type) {
        case T_Q8_0: return launch_t<T_Q8_0>(g, f, st);
        case T_Q4_0: return launch_t<T_Q4_0>(g, f, st);
        case T_Q5_0: return launch_t<T_Q5_0>(g, f, st);
        case T_Q4_K: return launch_t<T_Q4_K>(g, f, st);
        case T_Q6_K: return launch_t<T_Q6_K>(g, f, st);
    }
    return hipErrorInvalidValue;
}

// Grouped MoE: groups of up to 32 / 64 / 128 pairs, one token tile each, on 32 x 128,
// 64 x 64 and 128 x 128 tiles. A larger group decodes the expert's weights less often
// and leaves more of its last tile empty. Measured (us, 128 experts, K 2048, N 1536, by
// pairs per expert; groups of 32 / 64 / 128): Q4_K 19: 95 / 133 / 195, 25: 113 / 146 /
// 209, 40: 172 / 155 / 208, 62: 221 / 213 / 235, 94: 306 / 297 / 260, 187: 543 / 496 /
// 458; Q8_0 10: 122 / 124, 25: 152 / 142, 62: 235 / 202 / 236, 131: 392 / 336 / 378;
// Q6_K 25: 148 / 201, 40: 223 / 219, 62: 287 / 304 / 331, 94: 390 / 419 / 351.
// Against the kernels for few pairs per expert (us, quantizer and route included): Q4_K
// groups of 8 at 6 pairs per expert 75 against 92 here, groups of 16 (replaced) at 10 122
// against 92, at 62 492 against 217; Q8_0 groups of 4 at 2 108 against 113, at 3 142
// against 117, at 62 2198 against 207; Q6_K at 3 182 against 111. K 14336, N 4096, 8
// experts, Q4_K at 10 161 against 131.
int moe_i8t_group(uint32_t type, int rows, int K, int P, int E) {
    const bool small = type == T_Q8_0 || type == T_Q4_0;
    if (!(small || type == T_Q4_K || type == T_Q6_K)) return 0;
    if (type == T_Q4_K ? P <= 8 * (long)E : P < 3 * (long)E) return 0;
    if ((long)rows * K > 0xffffffffL) return 0;             // 32-bit activation offsets
    if (P < (small ? 16 : 32) * (long)E) return 32;
    return small || P <= 80 * (long)E ? 64 : 128;
}

namespace {
template <uint32_t T>
hipError_t launch_moe_t(const I8tArgs& g, int gsize, hipStream_t st) {
    switch (gsize) {
        case 32: return launch_cfg<T, 1, 1, 1, 4, 1, true>(g, st);
        case 64: return launch_cfg<T, 1, 1, 2, 2, 1, true>(g, st);
    }
    // (Q8_0 and Q4_0 stay at 64: moe_i8t_group)
    if constexpr (T == T_Q4_K || T == T_Q6_K)
        if (gsize == 128) return launch_cfg<T, 2, 1, 2, 4, 1, true>(g, st);
    return hipErrorInvalidValue;
}
}  // namespace

hipError_t launch_moe_i8t(uint32_t type, const uint8_t* w, const ActView& A, const void* route, int max_groups,
                          int gsize, int P, int E, int multi, int topk, float* y, int K, int N, hipStream_t st) {
    I8tArgs g{w, A, y, 0, N, K, row_bytes(type, K)};
    g.ntm = P / gsize + (P < E ? P : E);                    // sum over experts of ceil(c / gsize) at most
    g.route = static_cast<const uint8_t*>(route);
    g.mg = max_groups;
    g.multi = multi;
    g.topk = topk;
    g.ebytes = (long)g.rb * N;
    switch (type) {
        case T_Q8_0: return launch_moe_t<T_Q8_0>(g, gsize, st);
        case T_Q4_0: return launch_moe_t<T_Q4_0>(g, gsize, st);
        case T_Q4_K: return launch_moe_t<T_Q4_K>(g, gsize, st);
        case T_Q6_K: return launch_moe_t<T_Q6_K>(g, gsize, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace lp
