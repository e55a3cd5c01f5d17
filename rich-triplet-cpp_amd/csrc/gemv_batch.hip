// gemv_batch.hip -- batched GEMV, M = 2..8 activation rows (speculative
// verify): Y[m][n] = sum_k X[m][k] * W[n][k] on MFMA, every weight byte read
// once for all M rows (decode_gemma3.msl:416-518, MAX_BATCH 8).  Weights:
// Q4_K blocks, GGUF Q4_0 blocks, Q4Mat storage, or BF16.
//
// One MFMA step covers 32 values of K for a 16-row weight tile and up to four
// activation rows t of a group q (Q = ceil(M / 4) groups, one MFMA each):
//  * B is the weight tile: lane l = (n = l%16, g = l/16) supplies 8 weights
//    of row n; the same 8 positions of the activations stand in A, so each
//    format picks the positions its bytes hold (Fmt::kX*).
//  * A row i = 4t + lambda (lambda < Fmt::kLimbs) is limb lambda of activation
//    row 4q + t.  Rows i with no limb or past M hold whatever lies in LDS: a
//    row of A reaches only its own row of the result, and theirs are unused.
//  * The output lane (n, g) holds C[4g + r][n], r = 0..3: the limb dots of
//    activation row 4q + g for weight row n, combined in the lane.
//
// Exact activation limbs, so that the MFMA products are exact:
//  * BF16 weights (v_mfma_f32_16x16x32_bf16): three bf16 limbs with
//    h + m + l == x exactly.  Products of bf16 values are exact in f32, so
//    only the f32 accumulation rounds, as in an f32 dot product.
//  * 4-bit weights (v_mfma_i32_16x16x32_i8): the step is one 32-value block
//    with one scale, and x is a fixed-point integer of int8 limbs times a
//    power of two per block.  Each limb dot is an exact int32.
//    - Q4_K: the three limbs of the M = 1 kernel (q4k_mfma.hpp), within 2.5e-7
//      of the block's absmax.  Nibbles 0..15, so R = C0 * 65536 + C1 * 256 +
//      C2 stays below 32 * 15 * 2^22 < 2^31 and is converted once; the
//      minimum's term, -(dmin * mv_j) * sum(x) with x as the limbs hold it, is
//      a contraction over the super-block's eight sub-blocks and runs on
//      v_mfma_f32_16x16x4_f32 (quant_q4k.cpp:482-523).
//    - Q4_0, Q4Mat: four limbs (fixed4()), within 2^-30 of the block's absmax:
//      an f32 sum of the block's products rounds by more, also where a value
//      stands beside one a thousand times as large.  Signed values (nibble - 8,
//      or the two's-complement nibble) as int8 multiples of 16, so no offset
//      term is left.  The fourth limb's row of A costs no MFMA.
//
// Work split: a workgroup of 8 waves stages all M rows as limbs in LDS, KS
// waves share a 16-row tile's K (slots ks, ks + KS, ...) and their sums meet
// in LDS; 8 / KS tiles run side by side, and the workgroup walks tile groups
// blockIdx.x, + gridDim.x, ...  Where K is too long for LDS it is staged in
// chunks, or, where that is quicker, the chunks run in workgroups of their
// own and the last to arrive adds the partial sums (plan()).  Each wave keeps
// kDepth slots of weights in flight in registers, over chunk and group ends.
//
// Bound: short outputs by the chain launch -> x -> limbs -> MFMA -> store.
// The limbs cost about 90 VALU per 8 values in every workgroup (1024 x 3072,
// M = 8: 1.6 us of 7.5, reading x 1.1); long outputs by the epilogue's VALU,
// about 100 per slot at M <= 4 and 140 at M <= 8.  Keeping K inside the
// workgroup saves the merge through memory that every K longer than one slice
// used to pay (1.7 us).  Measured, before -> now, us per launch in a graph:
//   Q4_K  3072 x 3072   M = 4: 7.9 -> 6.0    M = 8: 9.7 -> 8.4
//   Q4_K  8192 x 3072   M = 4: 8.5 -> 7.3    M = 8: 10.4 -> 10.1
//   Q4_K  3072 x 8192   M = 4: 11.5 -> 10.5  M = 8: 14.5 -> 13.1
//   Q4_K  12288 x 12288 M = 4: 27.9 -> 28.8  M = 8: 32.1 -> 32.4
//   Q4_K  256 x 65536   M = 4: 23.0 -> 13.9  M = 8: 28.7 -> 20.2
//   BF16  3072 x 3072   M = 4: 10.0 -> 7.2   M = 8: 11.1 -> 8.7
//   BF16  12288 x 12288 M = 4: 52.2 -> 53.0  M = 8: 58.0 -> 58.3
//   Q4_0  4096 x 4096   M = 4: 18.7 -> 6.2   M = 8: 29.1 -> 9.2 (VALU before)
//   Q4_0  4096 x 11008  M = 4: 246 -> 10.5   M = 8: 616 -> 14.8
//   Q4Mat 4096 x 4096   M = 4: 15.6 -> 6.4   M = 8: 52.0 -> 9.6 (VALU before)
// (With three limbs Q4_0 and Q4Mat took 5% less at M = 8 and the same at M = 4,
// and were up to 4 times as far from float64 as the VALU kernels.)
#include "q4k_mfma.hpp"
#include "rt_common.hpp"
#include "rt_launch.hpp"

namespace rt_hip {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8;  // (16 for long outputs at M > 4, below)
constexpr int kDepth = 2;  // weight slots in flight per wave
constexpr uint32_t kNoRead = 0x7ffffff0u;

// ---- formats -------------------------------------------------------------
// A slot is the unit a wave loads: kSteps 32-value steps of one 16-row tile.
// load(): row n's bytes of slot `sl`, lane (n, g); rows past the resource's
// range and pieces past K read zeros.

struct BBf16 {
    static constexpr bool kInt = false, kMin = false;
    static constexpr int kLimbs = 3;
    static constexpr int kSteps = 4;  // 128 values
    static constexpr int kX0 = 8, kX1 = 4;  // lane group g: values 8g.. and 8g + 4..
    static constexpr bool kTail = true;     // K need not be whole slots
    struct Slot { u32x4 v[4]; };
    struct Tile {
        const uint8_t* base;
        int64_t left;
        uint32_t roff;
    };
    __device__ static Tile tile(const uint8_t* w, int64_t, int row0, int n_rows, int K, int lane) {
        const int64_t rb = 2 * static_cast<int64_t>(K);
        return Tile{w + row0 * rb, static_cast<int64_t>(n_rows - row0) * rb,
                    static_cast<uint32_t>((lane & 15) * rb)};
    }
    __device__ static void load(const Tile& t, bool live, int sl, int K, int lane, Slot& s) {
        const int64_t o = static_cast<int64_t>(sl) * 256;
        const BufRsrc rs = make_rsrc(t.base + o, live ? t.left - o : 0);
        const int g = lane >> 4;
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            const bool in = sl * 128 + 32 * st + 8 * g < K;
            s.v[st] = ld16(rs, in ? t.roff + static_cast<uint32_t>(64 * st + 16 * g) : 0xfffffff0u);
        }
    }
};

// 4-bit formats: a decoded slot is eight blocks' B operands and scales.
struct Dec4 {
    long b[8];
    float ds[8];
    float mn[2];  // Q4_K: -(dmin * mv) of sub-blocks g and 4 + g
};

__device__ __forceinline__ long pair64(uint32_t lo, uint32_t hi) {
    return static_cast<long>((static_cast<uint64_t>(hi) << 32) | lo);
}

struct BQ4k {
    static constexpr bool kInt = true, kMin = true;
    static constexpr int kLimbs = 3;
    static constexpr int kSteps = 8;  // one super-block
    static constexpr int kX0 = 8, kX1 = 4;
    static constexpr bool kTail = false;
    static constexpr bool kInterleave = false;
    struct Slot {
        u32x4 h;      // d | dmin << 16, scales[12]
        u32x2 p[4];   // qs[32c + 8g, +8), c = 0..3
    };
    struct Tile {
        const uint8_t* base;
        int64_t left;
        uint32_t roff;
    };
    __device__ static Tile tile(const uint8_t* w, int64_t, int row0, int n_rows, int K, int lane) {
        const int64_t rb = static_cast<int64_t>(K >> 8) * kQ4kBlockBytes;
        return Tile{w + row0 * rb, static_cast<int64_t>(n_rows - row0) * rb,
                    static_cast<uint32_t>((lane & 15) * rb)};
    }
    __device__ static void load(const Tile& t, bool live, int sl, int, int lane, Slot& s) {
        const int64_t o = static_cast<int64_t>(sl) * kQ4kBlockBytes;
        const BufRsrc rs = make_rsrc(t.base + o, live ? t.left - o : 0);
        const uint32_t g8 = static_cast<uint32_t>(lane >> 4) * 8u;
        s.h = ld16(rs, t.roff);
#pragma unroll
        for (int c = 0; c < 4; ++c)
            s.p[c] = __builtin_bit_cast(
                u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, static_cast<int>(t.roff + 16u + 32u * c + g8), 0, 0));
    }
    // Sub-block j's values k = 32j + t sit in byte 32*(j/2) + t of qs, low
    // nibble for even j and high for odd (quant_q4k.cpp:280-317); the 6-bit
    // scales four at a time (Q4KMat::scale_min, quant_q4k.cpp:58-69).
    __device__ static void decode(const Slot& s, int lane, Dec4& o) {
        const uint32_t h1 = s.h[1], h2 = s.h[2], h3 = s.h[3];
        const uint32_t sl = h1 & 0x3f3f3f3fu, sh = (h3 & 0x0f0f0f0fu) | ((h1 >> 2) & 0x30303030u);
        const uint32_t ml = h2 & 0x3f3f3f3fu, mh = ((h3 >> 4) & 0x0f0f0f0fu) | ((h2 >> 2) & 0x30303030u);
        const float d = f16_bits_to_f32(s.h[0] & 0xffffu), nd = -f16_bits_to_f32(s.h[0] >> 16);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            o.ds[j] = d * ubyte_f32(sl, j);
            o.ds[4 + j] = d * ubyte_f32(sh, j);
        }
        const uint32_t g8 = static_cast<uint32_t>(lane >> 4) * 8u;
        o.mn[0] = nd * static_cast<float>(__builtin_amdgcn_ubfe(ml, g8, 8));
        o.mn[1] = nd * static_cast<float>(__builtin_amdgcn_ubfe(mh, g8, 8));
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            o.b[2 * c] = pair64(s.p[c][0] & 0x0f0f0f0fu, s.p[c][1] & 0x0f0f0f0fu);
            o.b[2 * c + 1] = pair64((s.p[c][0] >> 4) & 0x0f0f0f0fu, (s.p[c][1] >> 4) & 0x0f0f0f0fu);
        }
    }
};

// 4 x 4 transpose over (lane group, register): out[j] of lane group g is
// in[g] of lane group j.  Four gfx950 permlane swaps.
__device__ __forceinline__ void transpose4(uint32_t (&a)[4]) {
    auto s0 = __builtin_amdgcn_permlane32_swap(a[0], a[2], false, false);
    auto s1 = __builtin_amdgcn_permlane32_swap(a[1], a[3], false, false);
    auto t0 = __builtin_amdgcn_permlane16_swap(s0[0], s1[0], false, false);
    auto t1 = __builtin_amdgcn_permlane16_swap(s0[1], s1[1], false, false);
    a[0] = t0[0];
    a[1] = t0[1];
    a[2] = t1[0];
    a[3] = t1[1];
}
// out[j] = lane group j's value, in every lane.
__device__ __forceinline__ void gather4(uint32_t v, uint32_t (&o)[4]) {
    auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    auto e = __builtin_amdgcn_permlane32_swap(r[0], r[0], false, false);
    auto d = __builtin_amdgcn_permlane32_swap(r[1], r[1], false, false);
    o[0] = e[0];
    o[1] = d[0];
    o[2] = e[1];
    o[3] = d[1];
}
// The scale of a block for four limbs and the exponent that takes its values
// to integers below 2^30: v * 2^e = A0 * 2^24 + A1 * 2^16 + A2 * 2^8 + A3, each
// multiplied by a weight * 16, so a limb dot's unit is k = 2^-(e + 4).  Blocks
// below 2^-115 share the scale whose k is f32's smallest value: values keep
// bits down to 2^-145.  An Inf/NaN makes k non-finite, and with it the output.
__device__ __forceinline__ void block_scale4(float amax, float& k, int& e) {
    const uint32_t bits = __float_as_uint(amax), eb = max((bits >> 23) & 0xffu, 11u);
    const float s = __uint_as_float((eb - 5u) << 23);
    k = eb == 0xffu ? amax : s * 0x1p-28f;
    e = 156 - static_cast<int>(eb);
}
// The four limb words (planes A0 .. A3; value i in byte i) of four values.  The
// bytes of R + 0x808080 are the digits of R in base 256 with the low three
// biased by 128; flipping their bit 7 makes them int8.
__device__ __forceinline__ void fixed4(const f32x4 v, int e, uint32_t (&w)[4]) {
    uint32_t b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        b[i] = static_cast<uint32_t>(static_cast<int>(__builtin_rintf(__builtin_ldexpf(v[i], e)))) + 0x808080u;
    // perm(hi, lo, sel): byte j of the result is byte sel_j of {hi:lo}
    const uint32_t l01 = __builtin_amdgcn_perm(b[1], b[0], 0x05010400u), l23 = __builtin_amdgcn_perm(b[3], b[2], 0x05010400u);
    const uint32_t h01 = __builtin_amdgcn_perm(b[1], b[0], 0x07030602u), h23 = __builtin_amdgcn_perm(b[3], b[2], 0x07030602u);
    w[3] = __builtin_amdgcn_perm(l23, l01, 0x05040100u) ^ 0x80808080u;
    w[2] = __builtin_amdgcn_perm(l23, l01, 0x07060302u) ^ 0x80808080u;
    w[1] = __builtin_amdgcn_perm(h23, h01, 0x05040100u) ^ 0x80808080u;
    w[0] = __builtin_amdgcn_perm(h23, h01, 0x07060302u);
}
// Signed nibbles of v (two's complement) as int8 multiples of 16.
__device__ __forceinline__ long signed16(uint32_t v) { return pair64((v << 4) & 0xf0f0f0f0u, v & 0xf0f0f0f0u); }

// GGUF Q4_0: 18-byte blocks (d f16, qs[16]; value j < 16 the low nibble of
// qs[j] minus 8, value 16 + j the high one; gguf.cpp:495-529).  A row's slot
// is 144 contiguous bytes: lane group g loads bytes [36g, 36g + 36), blocks
// 2g and 2g + 1 whole, and the transpose hands every lane dword g of each
// block: values 4g .. 4g + 3 and 16 + 4g .. 16 + 4g + 3.
struct BQ40 {
    static constexpr bool kInt = true, kMin = false;
    static constexpr int kLimbs = 4;
    static constexpr int kSteps = 8;
    static constexpr int kX0 = 4, kX1 = 16;  // values 4g.. and 4g + 16..
    static constexpr bool kTail = false;
    static constexpr bool kInterleave = false;
    struct Slot {
        u32x4 a, b;
        uint32_t c;
    };
    struct Tile {
        const uint8_t* base;
        int64_t left;
        uint32_t roff;
    };
    __device__ static Tile tile(const uint8_t* w, int64_t, int row0, int n_rows, int K, int lane) {
        const int64_t rb = static_cast<int64_t>(K >> 5) * kQ40BlockBytes;
        return Tile{w + row0 * rb, static_cast<int64_t>(n_rows - row0) * rb,
                    static_cast<uint32_t>((lane & 15) * rb + 36 * (lane >> 4))};
    }
    __device__ static void load(const Tile& t, bool live, int sl, int, int, Slot& s) {
        const int64_t o = static_cast<int64_t>(sl) * 144;
        const BufRsrc rs = make_rsrc(t.base + o, live ? t.left - o : 0);
        s.a = ld16(rs, t.roff);  // dword-aligned 16-byte loads
        s.b = ld16(rs, t.roff + 16);
        s.c = __builtin_amdgcn_raw_buffer_load_b32(rs, static_cast<int>(t.roff + 32), 0, 0);
    }
    __device__ static void decode(const Slot& s, int, Dec4& o) {
        uint32_t x[4], y[4], dd[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = __builtin_amdgcn_alignbyte(j < 3 ? s.a[j + 1] : s.b[0], s.a[j], 2);
        y[0] = s.b[1];
        y[1] = s.b[2];
        y[2] = s.b[3];
        y[3] = s.c;
        // both d's: the low half of dword 0, the high half of dword 4
        gather4((s.a[0] & 0xffffu) | (s.b[0] & 0xffff0000u), dd);
        transpose4(x);
        transpose4(y);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            o.ds[2 * j] = f16_bits_to_f32(dd[j] & 0xffffu);
            o.ds[2 * j + 1] = f16_bits_to_f32(dd[j] >> 16);
            o.b[2 * j] = signed16(x[j] ^ 0x88888888u);
            o.b[2 * j + 1] = signed16(y[j] ^ 0x88888888u);
        }
    }
};

// Q4Mat (rt_hip.h): packed nibbles, element 2i the low nibble of byte i, and
// f32 scales.  Lane group g loads groups 2g and 2g + 1 of the slot (32 bytes
// and two scales); after the transpose dword g of a group holds values 8g ..
// 8g + 7, the even ones in its low nibbles.
struct BQ4m {
    static constexpr bool kInt = true, kMin = false;
    static constexpr int kLimbs = 4;
    static constexpr int kSteps = 8;
    static constexpr int kX0 = 8, kX1 = 4;
    static constexpr bool kTail = true;
    static constexpr bool kInterleave = true;
    struct Slot {
        u32x4 a, b;
        uint32_t s0, s1;
    };
    struct Tile {
        const uint8_t* base;
        const uint8_t* sc;
        int64_t left, sleft;
        uint32_t roff, soff;
    };
    __device__ static Tile tile(const uint8_t* w, int64_t sc_off, int row0, int n_rows, int K, int lane) {
        const int64_t rb = K >> 1, sb = static_cast<int64_t>(K >> 5) * 4;
        return Tile{w + row0 * rb, w + sc_off + row0 * sb, static_cast<int64_t>(n_rows - row0) * rb,
                    static_cast<int64_t>(n_rows - row0) * sb,
                    static_cast<uint32_t>((lane & 15) * rb + 32 * (lane >> 4)),
                    static_cast<uint32_t>((lane & 15) * sb + 8 * (lane >> 4))};
    }
    __device__ static void load(const Tile& t, bool live, int sl, int K, int lane, Slot& s) {
        const int64_t o = static_cast<int64_t>(sl) * 128, os = static_cast<int64_t>(sl) * 32;
        const BufRsrc rs = make_rsrc(t.base + o, live ? t.left - o : 0);
        const BufRsrc rc = make_rsrc(t.sc + os, live ? t.sleft - os : 0);
        const int grp = sl * 8 + 2 * (lane >> 4), ng = K >> 5;
        const bool i0 = grp < ng, i1 = grp + 1 < ng;
        s.a = ld16(rs, i0 ? t.roff : kNoRead);
        s.b = ld16(rs, i1 ? t.roff + 16 : kNoRead);
        s.s0 = __builtin_amdgcn_raw_buffer_load_b32(rc, static_cast<int>(i0 ? t.soff : kNoRead), 0, 0);
        s.s1 = __builtin_amdgcn_raw_buffer_load_b32(rc, static_cast<int>(i1 ? t.soff + 4 : kNoRead), 0, 0);
    }
    __device__ static void decode(const Slot& s, int, Dec4& o) {
        uint32_t x[4] = {s.a[0], s.a[1], s.a[2], s.a[3]}, y[4] = {s.b[0], s.b[1], s.b[2], s.b[3]}, d0[4], d1[4];
        gather4(s.s0, d0);
        gather4(s.s1, d1);
        transpose4(x);
        transpose4(y);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            o.ds[2 * j] = __uint_as_float(d0[j]);
            o.ds[2 * j + 1] = __uint_as_float(d1[j]);
            o.b[2 * j] = signed16(x[j]);
            o.b[2 * j + 1] = signed16(y[j]);
        }
    }
};

// LDS of one staged slot for Q row groups:
//   4-bit: limbs [4 step pairs][4Q rows][4 g][kLimbs][2 steps][8 bytes], then
//          the units of the limb dots [4Q rows][8 steps] and (Q4_K) sums of x,
//          the same shape;
//   BF16:  limbs [4 steps][4Q rows][4 g][kLimbs][16 bytes].
// Step (pair) records are 16 bytes longer than their limbs, which spreads the
// lanes of a staging write, one step after another, over the banks.
template <class F>
__host__ __device__ constexpr int row_bytes() {  // of one step (pair)
    return 64 * F::kLimbs;
}
template <class F>
__host__ __device__ constexpr int step_bytes(int q) {
    return q * 4 * row_bytes<F>() + 16;
}
template <class F>
__host__ __device__ constexpr int limb_bytes(int q) {
    return 4 * step_bytes<F>(q);
}
template <class F>
__host__ __device__ constexpr int cst_bytes(int q) {
    return F::kInt ? q * 4 * 8 * 4 : 0;
}
template <class F>
__host__ __device__ constexpr int slot_lds(int q) {
    return limb_bytes<F>(q) + cst_bytes<F>(q) * (F::kMin ? 2 : 1);
}
constexpr int red_bytes(int waves, int q) { return waves * q * kWave * 4; }

// Sum and max over the aligned quad of lanes (every lane gets the same bits).
__device__ __forceinline__ uint32_t quad_sum(uint32_t v) {
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0xb1, 0xf, 0xf, false));
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x4e, 0xf, 0xf, false));
    return v;
}
__device__ __forceinline__ uint32_t quad_max(uint32_t v) {
    v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0xb1, 0xf, 0xf, false)));
    v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x4e, 0xf, 0xf, false)));
    return v;
}

// One launch's shape: tile groups of waves / KS tiles (KS = 1 << ks_log); K
// in `nslots` slots, staged `cslots` at a time.
// With slices > 1 (grid y) a workgroup takes one chunk alone and the chunks'
// partial sums meet in memory.
struct BatchShape {
    int n, k, m, ks_log, groups, nslots, cslots, nchunks, per;  // per: slots per wave and chunk, whole rings
    int slices, waves;
    int64_t sc_off;  // Q4Mat: byte offset of the scales
};

// Partials are stored and reloaded with agent-scope (device-coherent)
// accesses: they bypass the per-XCD L2, so the workgroup that reduces them
// sees every other XCD's stores once those have completed.
__device__ __forceinline__ void st_dev(float* p, float v) {
    __hip_atomic_store((__attribute__((address_space(1))) float*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_dev(const float* p) {
    return __hip_atomic_load((const __attribute__((address_space(1))) float*)p, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}

// Several weights on the same x in one launch: the tiles of the `count` jobs
// one after another (each N a multiple of 16, so a tile has one job); first[j]
// is job j's first tile.  Unused entries repeat the last job.
constexpr int kMaxJobs = 3;
struct BatchJobs {
    const uint8_t* w[kMaxJobs];
    float* y[kMaxJobs];
    int n[kMaxJobs], first[kMaxJobs];
};

// XP: units of 8 activations a thread holds while staging one chunk.  Up to 4
// the kernel fits 128 registers, so two workgroups may share a CU.
// FORM kMulti: W, n and Y of each tile come from `jobs`; n is the sum.  kBias:
// bias[n] is added as a row is stored (a form of its own: a test of the pointer
// in the others cost Q4_K batches of 8 rows 1.4%).
enum Form { kOne = 0, kMulti = 1, kBias = 2 };
template <class F, int Q, int XP, int NW, int FORM>
__global__ __launch_bounds__(NW * kWave) void k_gemv_batch(const uint8_t* __restrict__ W, const float* __restrict__ X,
                                                         int k, int m, int n, int ks_log, int cslots, int nslots,
                                                         int groups, int per, float* __restrict__ Y, int nchunks,
                                                         int64_t sc_off, float* __restrict__ P,
                                                         uint32_t* __restrict__ counters,
                                                         const float* __restrict__ bias, const BatchJobs jobs) {
    // (the arguments before Y are preloaded into SGPRs at wave launch)
    constexpr bool MULTI = FORM == kMulti;
    const BatchShape S{n, k, m, ks_log, groups, nslots, cslots, nchunks, per, static_cast<int>(gridDim.y), NW, sc_off};
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr int kLimb = limb_bytes<F>(Q), kCst = cst_bytes<F>(Q), kThreads = NW * kWave;
    constexpr int kRow = row_bytes<F>(), kStep = step_bytes<F>(Q), kG = 16 * F::kLimbs;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int KS = 1 << S.ks_log, ks = wave & (KS - 1), tw = wave >> S.ks_log, TW = NW >> S.ks_log;
    const int g = lane >> 4;
    uint8_t* const cst = lds + S.cslots * kLimb;    // scales, then sums
    uint8_t* const sums = cst + S.cslots * kCst;
    float* const red = reinterpret_cast<float*>(lds + S.cslots * slot_lds<F>(Q));

    // x of a chunk into registers: unit u = tid + kThreads * i of the chunk's
    // row-major sequence is 8 values of row m's step r / 4, lane group r % 4.
    // Rows past M fall outside the buffer's range and read zeros.
    f32x4 xa[XP], xb[XP];
    const BufRsrc xr = make_rsrc(X, static_cast<int64_t>(S.m) * S.k * 4);
    auto chunk_slots = [&](int c) { return min(S.cslots, S.nslots - c * S.cslots); };
    struct Units {  // (m, r) of this thread's units, one after another
        uint32_t upr, dm, dr, m, r;
        __device__ void next() {
            m += dm;
            r += dr;
            const uint32_t over = r >= upr ? 1u : 0u;
            m += over;
            r -= over ? upr : 0u;
        }
    };
    auto units_of = [&](int c) {
        Units u;
        u.upr = static_cast<uint32_t>(chunk_slots(c) * F::kSteps * 4);
        // upr is at least 16 and below 2^14: a reciprocal rounded up by 2^-17 of
        // itself gives exact quotients of values up to 1024
        const float inv = __builtin_amdgcn_rcpf(static_cast<float>(u.upr)) * 1.0000076f;
        u.dm = static_cast<uint32_t>(static_cast<float>(kThreads) * inv);
        u.dr = kThreads - u.dm * u.upr;
        u.m = static_cast<uint32_t>(static_cast<float>(tid) * inv);
        u.r = static_cast<uint32_t>(tid) - u.m * u.upr;
        return u;
    };
    auto load_x = [&](int c) {
        Units u = units_of(c);
        const uint32_t k0 = static_cast<uint32_t>(c * S.cslots * F::kSteps * 32);
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            const uint32_t e = k0 + (F::kX0 == 8 ? 8 * u.r : 32 * (u.r >> 2) + 4 * (u.r & 3));
            uint32_t off = u.m * static_cast<uint32_t>(4 * S.k) + 4 * e;
            if constexpr (F::kTail) off = e < static_cast<uint32_t>(S.k) ? off : kNoRead;
            xa[i] = __builtin_bit_cast(f32x4, ld16(xr, off));
            xb[i] = __builtin_bit_cast(f32x4, ld16(xr, off + 4 * F::kX1));
            u.next();
        }
    };
    // Limbs (and, for the 4-bit formats, the per-row block constants) into LDS.
    auto stage = [&](int c) {
        Units u = units_of(c);
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            const bool in = u.m < static_cast<uint32_t>(S.m);
            f32x4 a = xa[i], b = xb[i];
            if constexpr (F::kInt) {
                if constexpr (F::kInterleave) {
                    a = f32x4{xa[i][0], xa[i][2], xb[i][0], xb[i][2]};
                    b = f32x4{xa[i][1], xa[i][3], xb[i][1], xb[i][3]};
                }
                // Block (step, m) is the quad of units g = 0..3.  A NaN stays in the
                // maximum, and is the largest of the bit patterns.
                auto max2 = [](float p, float q) { return __builtin_elementwise_maximum(p, q); };
                float amax = max2(max2(max2(fabsf(a[0]), fabsf(a[1])), max2(fabsf(a[2]), fabsf(a[3]))),
                                  max2(max2(fabsf(b[0]), fabsf(b[1])), max2(fabsf(b[2]), fabsf(b[3]))));
                amax = __uint_as_float(quad_max(__float_as_uint(amax)));
                uint32_t wa[4], wb[4];
                float unit, sum = 0.0f;
                if constexpr (F::kLimbs == 4) {
                    int ex;
                    block_scale4(amax, unit, ex);
                    fixed4(a, ex, wa);
                    fixed4(b, ex, wb);
                } else {
                    float sc, inv;
                    q4k_mfma::sub_block_scale(amax, sc, inv);
                    unit = sc * (1.0f / 65536.0f);
                    uint32_t bits = 0;
                    q4k_mfma::limb_words(a, inv, wa[0], wa[1], wa[2], bits);
                    q4k_mfma::limb_words(b, inv, wb[0], wb[1], wb[2], bits);
                    // the sum of the 32 R, |R| <= 2^22, exactly: what the limbs
                    // leave out of x then meets w = P - min, half as large as P
                    sum = static_cast<float>(static_cast<int>(quad_sum(bits) - (0x4b400000u << 5))) * unit;
                }
                if (in) {
                    uint8_t* const dst = lds + (u.r >> 3) * kStep + u.m * kRow + (u.r & 3) * kG + ((u.r & 4) << 1);
#pragma unroll
                    for (int l = 0; l < F::kLimbs; ++l) *reinterpret_cast<u32x2*>(dst + 16 * l) = u32x2{wa[l], wb[l]};
                    if ((u.r & 3) == 0) {
                        const uint32_t o = (u.r >> 5) * kCst + u.m * 32 + (u.r & 28);
                        *reinterpret_cast<float*>(cst + o) = unit;
                        if constexpr (F::kMin) *reinterpret_cast<float*>(sums + o) = sum;
                    }
                }
            } else {
                u32x2 ha, ma, la, hb, mb, lb;
                bf16_limbs4(a, ha, ma, la);
                bf16_limbs4(b, hb, mb, lb);
                if (in) {
                    u32x4* d4 = reinterpret_cast<u32x4*>(lds + (u.r >> 2) * kStep + u.m * kRow + (u.r & 3) * kG);
                    d4[0] = u32x4{ha[0], ha[1], hb[0], hb[1]};
                    d4[1] = u32x4{ma[0], ma[1], mb[0], mb[1]};
                    d4[2] = u32x4{la[0], la[1], lb[0], lb[1]};
                }
            }
            u.next();
        }
    };

    int group = blockIdx.x, chunk = blockIdx.y;
    auto job_of = [&](int t) { return t >= jobs.first[2] ? 2 : (t >= jobs.first[1] ? 1 : 0); };
    auto tile_of = [&](int grp) {
        const int t = grp * TW + tw;
        if constexpr (MULTI) {
            const int j = job_of(t);
            const uint8_t* const w = j == 2 ? jobs.w[2] : (j == 1 ? jobs.w[1] : jobs.w[0]);
            const int n = j == 2 ? jobs.n[2] : (j == 1 ? jobs.n[1] : jobs.n[0]);
            const int first = j == 2 ? jobs.first[2] : (j == 1 ? jobs.first[1] : 0);
            return F::tile(w, S.sc_off, 16 * (t - first), n, S.k, lane);
        } else {
            return F::tile(W, S.sc_off, 16 * t, S.n, S.k, lane);
        }
    };
    typename F::Tile cur = tile_of(group);
    typename F::Slot ring[kDepth];
    // Slot i of this wave in chunk c (none past the chunk's end: an empty
    // range reads zeros and no memory).
    auto issue = [&](const typename F::Tile& t, int grp, int c, int i, typename F::Slot& dst) {
        const int sl = ks + (i << S.ks_log);
        const bool live = grp < S.groups && sl < chunk_slots(c);
        F::load(t, live, c * S.cslots + (live ? sl : 0), S.k, lane, dst);
    };

    load_x(chunk);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < kDepth; ++j) {
        issue(cur, group, chunk, j, ring[j]);
        __builtin_amdgcn_sched_barrier(0);
    }
    stage(chunk);
    lds_barrier();

    // This lane's A rows: (t, lambda) = ((l % 16) / 4, l % 4) of each group q.
    const int ai = lane & 15;
    const uint32_t a_base = static_cast<uint32_t>((ai >> 2) * kRow + g * kG + min(ai & 3, F::kLimbs - 1) * 16);
    // Sums as an f32 A operand: row i = 4t + q of it is activation row 4q + t.
    const uint32_t s_base = static_cast<uint32_t>((min(ai & 3, Q - 1) * 4 + (ai >> 2)) * 32 + 4 * g);

    // C: the even and the odd BF16 steps' dots of a chunk.  acc: the sum over
    // chunks, or over 4-bit slots.  Short chains round less than one long one.
    f32x4 C[2][Q];
    float acc[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        C[0][q] = C[1][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        acc[q] = 0.0f;
    }
    auto consume = [&](const typename F::Slot& slot, int sl) {
        const uint8_t* const lb = lds + sl * kLimb + a_base;
        if constexpr (!F::kInt) {
#pragma unroll
            for (int st = 0; st < 4; ++st)
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const bf16x8 A = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(lb + st * kStep + q * 4 * kRow));
                    C[st & 1][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, __builtin_bit_cast(bf16x8, slot.v[st]),
                                                                           C[st & 1][q], 0, 0, 0);
                }
        } else {
            Dec4 w;
            F::decode(slot, lane, w);
            // The minimum's term of this super-block, where its sum starts:
            // kept apart to the end, the two halves of each sum would grow
            // several times larger than the sum and round accordingly.
            f32x4 mins = {0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (F::kMin) {
                const uint8_t* const sb = sums + sl * kCst + s_base;
                mins = __builtin_amdgcn_mfma_f32_16x16x4f32(*reinterpret_cast<const float*>(sb), w.mn[0], mins, 0, 0, 0);
                mins = __builtin_amdgcn_mfma_f32_16x16x4f32(*reinterpret_cast<const float*>(sb + 16), w.mn[1], mins, 0,
                                                            0, 0);
            }
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const f32x4* kp = reinterpret_cast<const f32x4*>(cst + sl * kCst + (q * 4 + g) * 32);
                const f32x4 k0 = kp[0], k1 = kp[1];
                float sum = F::kMin ? mins[q] : 0.0f;
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const u32x4 a2 = *reinterpret_cast<const u32x4*>(lb + p * kStep + q * 4 * kRow);
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int j = 2 * p + e;
                        const i32x4 z = {0, 0, 0, 0};
                        const i32x4 c =
                            __builtin_amdgcn_mfma_i32_16x16x32_i8(pair64(a2[2 * e], a2[2 * e + 1]), w.b[j], z, 0, 0, 0);
                        const float kj = j < 4 ? k0[j & 3] : k1[j & 3];
                        if constexpr (F::kMin) {
                            // |R * nibble| sums below 2^31 (see above); the shifts wrap, the total does not
                            const uint32_t tot = (((static_cast<uint32_t>(c[0]) << 8) + static_cast<uint32_t>(c[1]))
                                                  << 8) + static_cast<uint32_t>(c[2]);
                            sum = __builtin_fmaf(w.ds[j], static_cast<float>(static_cast<int>(tot)) * kj, sum);
                        } else {
                            // (multiples of 16 below 2^28: both halves convert exactly)
                            const int hi = c[0] * 256 + c[1], lo = c[2] * 256 + c[3];
                            const float dot = __builtin_fmaf(static_cast<float>(hi), 65536.0f, static_cast<float>(lo));
                            sum = __builtin_fmaf(w.ds[j], dot * kj, sum);
                        }
                    }
                }
                acc[q] += sum;
            }
        }
    };

    for (;;) {
        // The next unit of work: this group's next chunk, or the next group.
        const bool last_chunk = S.slices > 1 || chunk + 1 == S.nchunks;
        const int ngroup = last_chunk ? group + static_cast<int>(gridDim.x) : group, nchunk = last_chunk ? 0 : chunk + 1;
        const typename F::Tile next = tile_of(min(ngroup, S.groups - 1));
        // (no products in a wave whose tile lies past the last row)
        const int cs = 16 * (group * TW + tw) < S.n ? chunk_slots(chunk) : 0;
        for (int i = 0; i < S.per; i += kDepth) {
#pragma unroll
            for (int j = 0; j < kDepth; ++j) {
                const int sl = ks + ((i + j) << S.ks_log);
                if (sl < cs) consume(ring[j], sl);
                __builtin_amdgcn_sched_barrier(0);
                const int ii = i + j + kDepth;
                if (ii < S.per)
                    issue(cur, group, chunk, ii, ring[j]);
                else if (ngroup < S.groups)
                    issue(next, ngroup, nchunk, ii - S.per, ring[j]);
            }
        }
        if constexpr (!F::kInt) {
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const f32x4 c = C[0][q] + C[1][q];
                acc[q] += (c[0] + c[1]) + c[2];
                C[0][q] = C[1][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
        if (last_chunk) {
            // Row n of the tile, activation row 4q + g.
            const int row = 16 * (group * TW + tw) + (lane & 15);
            float v[Q], add = 0.0f;
            if constexpr (FORM == kBias) add = bias[min(row, S.n - 1)];
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                v[q] = acc[q];
                acc[q] = 0.0f;
            }
            if (S.ks_log) {
                // The KS waves' sums in wave order.
#pragma unroll
                for (int q = 0; q < Q; ++q) red[(wave * Q + q) * kWave + lane] = v[q];
                lds_barrier();
                if (ks == 0) {
#pragma unroll
                    for (int q = 0; q < Q; ++q)
                        for (int j = 1; j < KS; ++j) v[q] += red[((wave + j) * Q + q) * kWave + lane];
                }
                if (ngroup < S.groups) lds_barrier();  // before the next group's sums
            }
            const int64_t total = static_cast<int64_t>(S.m) * S.n;
            const bool mine = ks == 0 && row < S.n;
            if (S.slices > 1) {
                // Every wave's partials have completed, then one arrival per
                // workgroup; the last to arrive adds them in slice order (the
                // result does not depend on which) and resets the counter.
                // The ordering rests on the accesses themselves: the partials
                // are agent-scope stores (written through past the XCD's L2)
                // whose completion every wave has waited for (vmcnt(0))
                // before the barrier and the arrival, and the merging
                // workgroup reads them with agent-scope loads, issued once
                // the arrival's result is known.  A release/acquire on the
                // arrival would write back and invalidate the XCD's whole L2
                // in every workgroup: measured 15.8 against 10.2 us for Q4_K
                // 8192 x 3072 at M = 8.
                if (mine)
#pragma unroll
                    for (int q = 0; q < Q; ++q)
                        if (4 * q + g < S.m)
                            st_dev(P + blockIdx.y * total + static_cast<int64_t>(4 * q + g) * S.n + row, v[q]);
                wait_vmcnt<0>();
                lds_barrier();
                uint32_t* const flag = reinterpret_cast<uint32_t*>(lds);  // the limbs are dead
                if (tid == 0)
                    *flag = __hip_atomic_fetch_add(counters + group, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                lds_barrier();
                if (*flag != static_cast<uint32_t>(S.slices - 1)) return;
                if (mine)
#pragma unroll
                    for (int q = 0; q < Q; ++q)
                        if (4 * q + g < S.m) {
                            const float* const src = P + static_cast<int64_t>(4 * q + g) * S.n + row;
                            v[q] = ld_dev(src);
                            for (int j = 1; j < S.slices; ++j) v[q] += ld_dev(src + j * total);
                        }
                if (tid == 0) __hip_atomic_store(counters + group, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (mine) {
                if constexpr (FORM == kBias)
#pragma unroll
                    for (int q = 0; q < Q; ++q) v[q] += add;
                float* y = Y;
                int yn = S.n, yrow = row;
                if constexpr (MULTI) {
                    const int j = job_of(group * TW + tw);
                    y = j == 2 ? jobs.y[2] : (j == 1 ? jobs.y[1] : jobs.y[0]);
                    yn = j == 2 ? jobs.n[2] : (j == 1 ? jobs.n[1] : jobs.n[0]);
                    yrow -= 16 * (j == 2 ? jobs.first[2] : (j == 1 ? jobs.first[1] : 0));
                }
#pragma unroll
                for (int q = 0; q < Q; ++q)
                    if (4 * q + g < S.m) y[static_cast<int64_t>(4 * q + g) * yn + yrow] = v[q];
            }
        }
        if (ngroup >= S.groups) break;
        group = ngroup;
        chunk = nchunk;
        cur = next;
        if (S.nchunks > 1) {
            load_x(chunk);
            lds_barrier();  // every wave is done with the limbs in LDS
            stage(chunk);
            lds_barrier();
        }
    }
}

// Two workgroups of `cs`-slot chunks fit one CU: LDS, and registers (XP <= 4).
template <class F>
bool two_fit(int64_t cs, int m, int q) {
    return 2 * (cs * slot_lds<F>(q) + red_bytes(kWaves, q)) <= static_cast<int64_t>(lds_cap()) &&
           cs * F::kSteps * 4 * m <= 4 * kWaves * kWave;
}

// The launch shape: the least estimated time over the splits of K between the
// waves of a workgroup (KS) and, with `sliced`, between workgroups.  Costs in
// units of 0.1 us above the launch: one workgroup alone on its CU, and (".2")
// two that share it, as the grid of a shape makes them (`turns`: how many
// workgroups, or pairs of them, a CU runs one after another).
//   stage  per 1024 activations staged: every slice, and in an unsliced launch
//          every chunk of every turn (once when one chunk holds all of K)
//   slot   per weight slot of each wave
//   again  per staging that waits for the products before it
//   red    per turn, the waves' sums where KS > 1
//   merge, slice, sums   a merge through memory, per slice, and per 10^6 partial sums
//   turn, turn1          per turn after the first, sliced and not
//   narrow per slot and halving of KS: fewer waves of a tile read longer runs
//          of a row each
// Fitted to times of every split at 46 sizes from 16 x 256 to 262144 x 1024 and
// 16 x 131072 at M = 2, 4, 5 and 8, in each format: the shape taken is within
// 1.1% of the best of a size on average, and within 13% but for BF16 128256 x
// 2048 (26%: 114 us with KS = 1, 90 with 8).
struct Cost {
    double stage, stage2, slot, slot2, again, red, merge, slice, sums, turn, turn1, narrow;
};
template <class F, int Q>
constexpr Cost cost_of() {
    if constexpr (!F::kInt)
        return Q == 1 ? Cost{1.7, 2.0, 10.0, 19.0, 1.4, 0.34, 18.0, 3.7, 38.0, 11.0, 12.0, 0.05}
                      : Cost{1.4, 1.8, 11.0, 21.0, 2.2, 5.0, 10.0, 4.9, 30.0, 15.0, 4.3, 0.099};
    else if constexpr (F::kMin)
        return Q == 1 ? Cost{1.4, 2.1, 9.6, 18.0, 16.0, 3.0, 9.4, 4.2, 28.0, 12.0, 0.18, 0.063}
                      : Cost{1.7, 2.3, 9.8, 18.0, 0.23, 2.6, 11.0, 5.7, 15.0, 10.0, 6.1, 0.05};
    else
        return Q == 1 ? Cost{1.5, 2.1, 7.6, 14.0, 11.0, 2.0, 8.2, 4.1, 29.0, 18.0, 5.0, 0.13}
                      : Cost{1.2, 2.3, 9.8, 15.0, 2.5, 1.6, 9.2, 5.5, 14.0, 12.0, 6.6, 0.051};
}

// Workgroups of `cs`-slot chunks that share a CU in an unsliced launch: two
// where they fit; BF16 streams as fast from one (65536 x 2560, M = 4: 62.6 us
// against 66.1).
template <class F>
int64_t unsliced_per_cu(int64_t cs, int m, int q) {
    return F::kInt && two_fit<F>(cs, m, q) ? 2 : 1;
}

template <class F, int Q>
bool plan(int64_t n, int64_t k, int m, bool sliced, BatchShape* out) {
    const int64_t cus = device_info().cus;
    const int64_t tiles = (n + 15) / 16, nslots = (k + F::kSteps * 32 - 1) / (F::kSteps * 32);
    const int64_t lds = static_cast<int64_t>(lds_cap());
    // Chunks: what LDS holds, and 8 units of x per thread.
    const int64_t fit = (lds - red_bytes(kWaves, Q)) / slot_lds<F>(Q);
    const int64_t by_x = 8 * kWaves * kWave / (static_cast<int64_t>(F::kSteps) * 4 * m);
    const int64_t cmax = fit < by_x ? fit : by_x;
    if (cmax < 1) return false;
    const int64_t cmin = (nslots + cmax - 1) / cmax;
    // Long outputs at M > 4 whose limbs leave room for one workgroup per CU:
    // 16 waves, each with tiles of its own (8 waves leave the matrix cores
    // waiting: Q4_K 128256 x 3072, M = 8: 75.0 us with 8, 63 with 16).
    if (F::kInt && Q == 2 && cmin == 1 && tiles >= 16 * cus &&
        nslots * slot_lds<F>(Q) + red_bytes(16, Q) <= lds &&
        2 * (nslots * slot_lds<F>(Q) + red_bytes(kWaves, Q)) > lds) {
        const int64_t p = (nslots + kDepth - 1) / kDepth * kDepth;
        *out = BatchShape{static_cast<int>(n), static_cast<int>(k), m, 0, static_cast<int>((tiles + 15) / 16),
                          static_cast<int>(nslots), static_cast<int>(nslots), 1, static_cast<int>(p), 1, 16, 0};
        return true;
    }
    constexpr Cost C = cost_of<F, Q>();
    double cost = -1.0;
    const int fs = tune_param("BATCH_SLICES", 0), fk = tune_param("BATCH_KS", -1);
    static const int kSlices[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 16, 20, 24, 32, 48, 64, 96, 128};
    for (const int64_t slices : kSlices) {
        if (slices > 1 && (!sliced || slices < cmin || slices > nslots)) continue;
        if (fs && slices != fs) continue;
        const int64_t nchunks = slices > 1 ? slices : cmin;
        const int64_t cs = (nslots + nchunks - 1) / nchunks;
        if (cs * (nchunks - 1) >= nslots) continue;  // an empty last chunk
        const double stage = static_cast<double>(cs * F::kSteps * 32 * m) / 1024.0;
        const int64_t per_cu = slices > 1 ? (two_fit<F>(cs, m, Q) ? 2 : 1) : unsliced_per_cu<F>(cs, m, Q);
        for (int lg = 0; lg <= 3; ++lg) {
            if (fk >= 0 && lg != fk) continue;
            const int64_t groups = (tiles + (kWaves >> lg) - 1) / (kWaves >> lg);
            if (slices > 1 && groups > static_cast<int64_t>(kArrivalCounters)) continue;
            const int64_t per = (cs + (1 << lg) - 1) >> lg, all = groups * slices;
            const bool shared = per_cu == 2 && all > cus;
            const double turns = static_cast<double>((all + cus - 1) / cus) * (shared ? 0.5 : 1.0);
            const double n_stage = slices == 1 && nchunks == 1 ? 1.0 : turns * static_cast<double>(slices > 1 ? 1 : nchunks);
            const double n_slot = turns * static_cast<double>(per * (slices > 1 ? 1 : nchunks));
            double t = n_stage * stage * (shared ? C.stage2 : C.stage) + n_slot * (shared ? C.slot2 : C.slot);
            t += C.narrow * static_cast<double>(3 - lg) * n_slot + (lg ? C.red * turns : 0.0);
            if (slices > 1)
                t += C.merge + C.slice * static_cast<double>(slices) + C.sums * static_cast<double>(slices * m * n) * 1e-6 +
                     C.turn * (turns - 1.0);
            else
                t += C.turn1 * (turns - 1.0) + (nchunks > 1 ? C.again * (n_stage - 1.0) : 0.0);
            if (cost >= 0.0 && t >= cost) continue;
            cost = t;
            *out = BatchShape{static_cast<int>(n),      static_cast<int>(k),  m, lg, static_cast<int>(groups),
                              static_cast<int>(nslots), static_cast<int>(cs), static_cast<int>(nchunks),
                              static_cast<int>((per + kDepth - 1) / kDepth * kDepth), static_cast<int>(slices), kWaves, 0};
        }
    }
    return cost >= 0.0;
}

// jobs: null for one weight w, else n is the sum of theirs (w and y unused).
template <class F, int Q, int FORM>
hipError_t run(const void* w, const float* x, float* y, int64_t n, int64_t k, int m, int64_t sc_off, hipStream_t s,
               const float* bias, const BatchJobs* jobs = nullptr) {
    BatchShape S;
    if (!plan<F, Q>(n, k, m, true, &S)) return hipErrorInvalidValue;
    float* part = nullptr;
    uint32_t* counters = nullptr;
    if (S.slices > 1) {
        // Without scratch (it may not grow under a stream capture) K stays
        // inside the workgroups.
        hipError_t e;
        counters = arrival_counters(s, &e);
        if (counters)
            part = static_cast<float*>(workspace(static_cast<size_t>(S.slices) * m * n * sizeof(float), s, &e));
        if (!part && !plan<F, Q>(n, k, m, false, &S)) return hipErrorInvalidValue;
    }
    S.sc_off = sc_off;
    const size_t lds = static_cast<size_t>(S.cslots) * slot_lds<F>(Q) + red_bytes(S.waves, Q);
    const int64_t slots = (S.waves == kWaves ? unsliced_per_cu<F>(S.cslots, m, Q) : 1) *
                          static_cast<int64_t>(device_info().cus);
    const dim3 grid(static_cast<unsigned>(S.slices > 1 || S.groups < slots ? S.groups : slots),
                    static_cast<unsigned>(S.slices));
    const int threads = S.waves * kWave;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(static_cast<unsigned>(threads)), lds, s, static_cast<const uint8_t*>(w), x, S.k, S.m, S.n,
                           S.ks_log, S.cslots, S.nslots, S.groups, S.per, y, S.nchunks, S.sc_off, part, counters, bias,
                           FORM == kMulti ? *jobs : BatchJobs{});
        return hipGetLastError();
    };
    const int xp = static_cast<int>((static_cast<int64_t>(S.cslots) * F::kSteps * 4 * m + threads - 1) / threads);
    if constexpr (F::kInt && Q == 2) {
        if (S.waves == 16) return go(k_gemv_batch<F, Q, 4, 16, FORM>);
    }
    if (xp <= 1) return go(k_gemv_batch<F, Q, 1, kWaves, FORM>);
    if (xp <= 2) return go(k_gemv_batch<F, Q, 2, kWaves, FORM>);
    if (xp <= 4) return go(k_gemv_batch<F, Q, 4, kWaves, FORM>);
    return go(k_gemv_batch<F, Q, 8, kWaves, FORM>);
}

template <class F>
hipError_t dispatch(const void* w, const float* x, float* y, int64_t n, int64_t k, int m, int64_t sc_off,
                    hipStream_t s, const float* bias) {
    if (bias)
        return m <= 4 ? run<F, 1, kBias>(w, x, y, n, k, m, sc_off, s, bias)
                      : run<F, 2, kBias>(w, x, y, n, k, m, sc_off, s, bias);
    return m <= 4 ? run<F, 1, kOne>(w, x, y, n, k, m, sc_off, s, nullptr)
                  : run<F, 2, kOne>(w, x, y, n, k, m, sc_off, s, nullptr);
}

template <class F>
size_t workspace_of(int64_t n, int64_t k, int m) {
    BatchShape S;
    const bool ok = m <= 4 ? plan<F, 1>(n, k, m, true, &S) : plan<F, 2>(n, k, m, true, &S);
    return ok && S.slices > 1 ? static_cast<size_t>(S.slices) * m * n * sizeof(float) : 0;
}

}  // namespace

size_t gemv_batch_workspace_bytes(int fmt, int64_t n, int64_t k, int m) {
    if (m < 2 || m > 8) return 0;
    switch (fmt) {
        case RT_HIP_Q4K: return workspace_of<BQ4k>(n, k, m);
        case RT_HIP_BF16: return workspace_of<BBf16>(n, k, m);
        case RT_HIP_Q4_0: return workspace_of<BQ40>(n, k, m);
        case RT_HIP_Q4MAT: return workspace_of<BQ4m>(n, k, m);
    }
    return 0;
}

hipError_t launch_gemv_batch(int fmt, const void* w, const float* x, float* y, int64_t n, int64_t k, int m,
                             hipStream_t s, const float* bias) {
    if (m < 2 || m > 8) return hipErrorInvalidValue;
    switch (fmt) {
        case RT_HIP_Q4K: return dispatch<BQ4k>(w, x, y, n, k, m, 0, s, bias);
        case RT_HIP_BF16: return dispatch<BBf16>(w, x, y, n, k, m, 0, s, bias);
        case RT_HIP_Q4_0: return dispatch<BQ40>(w, x, y, n, k, m, 0, s, bias);
        case RT_HIP_Q4MAT:
            return dispatch<BQ4m>(w, x, y, n, k, m, static_cast<int64_t>(q4mat_scales_offset(n, k)), s, bias);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_gemv_batch_q4k_multi(int count, const void* const* w, const float* x, float* const* y,
                                       const int64_t* n, int64_t k, int m, hipStream_t s) {
    if (count < 1 || count > kMaxJobs || m < 2 || m > 8) return hipErrorInvalidValue;
    BatchJobs jobs;
    int64_t total = 0;
    for (int j = 0; j < kMaxJobs; ++j) {
        const int i = j < count ? j : count - 1;
        if (n[i] % 16 != 0) return hipErrorInvalidValue;
        jobs.w[j] = static_cast<const uint8_t*>(w[i]);
        jobs.y[j] = y[i];
        jobs.n[j] = static_cast<int>(n[i]);
        jobs.first[j] = j < count ? static_cast<int>(total / 16) : jobs.first[i];
        if (j < count) total += n[i];
    }
    if (total > 0x7fffffff) return hipErrorInvalidValue;
    return m <= 4 ? run<BQ4k, 1, kMulti>(nullptr, x, nullptr, total, k, m, 0, s, nullptr, &jobs)
                  : run<BQ4k, 2, kMulti>(nullptr, x, nullptr, total, k, m, 0, s, nullptr, &jobs);
}

}  // namespace rt_hip
