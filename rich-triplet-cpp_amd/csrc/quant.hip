// quant.hip -- Q4_K dequantization (to f32 or bf16) and quantization.
//
// Dequant: one lane per 8 (bf16) or 4 (f32) consecutive outputs, so every
// store instruction writes 1 KB of contiguous output; bit-exact with
// Q4KMat::dequantize_row_into (quant_q4k.cpp:280-317) because both products
// are exact and only the subtraction rounds.  The bf16 variant rounds that
// f32 value to nearest-even, as flux_dequant_q4k's bfloat() conversion does
// (shaders/flux.msl:78-79).
//
// Quantize: one wave per four 256-value super-blocks, lane l holding values
// 4l..4l+3 of each (sub-block l/8).  Every arithmetic step gives the bits of
// the reference's (quant_q4k.cpp:71-158): min/max are exact whatever the
// reduction order, the scalars of a sub-block and block take IEEE divisions
// and reciprocals (hipcc's default correctly-rounded f32 divide), no
// contraction (the library builds with -ffp-contract=off), the division of
// each value is a correctly rounded one from the sub-block's reciprocal, and
// the f16 header conversion is the reference's truncating one restated on
// bits.
#include "q4k_mfma.hpp"
#include "rt_common.hpp"
#include "rt_launch.hpp"

namespace rt_hip {
namespace {

// One lane per kPer consecutive outputs of a super-block: 8 for bf16 (32
// lanes per block), 4 for f32 (64 lanes); either way a wave's store covers
// 1 KB of contiguous output.  Sub-block sb's 32 values are the low (even
// sb) or high nibbles of qs chunk sb/2, so a lane reads kPer qs bytes and
// the 16-byte header.  w = (d*sv)*q - dmin*mv: the product is exact in f32,
// so the fma rounds only the subtraction, as the reference does.  bf16 is
// v_cvt_pk_bf16_f32, round-to-nearest-even with NaN quieting: identical to
// the reference's f32 -> bf16 (bf16.hpp:50-60) on every f32, NaNs included
// (checked on the device against the bit rule).
template <bool BF16>
__device__ __forceinline__ void dequant_unit(const uint8_t* __restrict__ W, void* __restrict__ out, int64_t u) {
    constexpr int kPer = BF16 ? 8 : 4;
    constexpr int kLanesPerSub = 32 / kPer;
    constexpr int kLanesPerBlk = 8 * kLanesPerSub;
    const int64_t blk = u / kLanesPerBlk;
    const int l = static_cast<int>(u % kLanesPerBlk);
    const int sb = l / kLanesPerSub, part = l % kLanesPerSub;
    const uint8_t* bp = W + blk * kQ4kBlockBytes;
    const u32x4 hd = ld16(bp);
    const uint8_t* qp = bp + 16 + (sb >> 1) * 32 + part * kPer;
    uint32_t q[2];
    if constexpr (BF16) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(qp);
        q[0] = v[0];
        q[1] = v[1];
    } else {
        q[0] = *reinterpret_cast<const uint32_t*>(qp);
        q[1] = 0;
    }
    uint32_t sv, mv;
    decode_scale_min(make_scale_sel(sb), hd[1], hd[2], hd[3], sv, mv);
    const float sc = f16_bits_to_f32(hd[0] & 0xffffu) * static_cast<float>(sv);
    const float mn = f16_bits_to_f32(hd[0] >> 16) * static_cast<float>(mv);
    const uint32_t sh = static_cast<uint32_t>(sb & 1) * 4u;
    float w[kPer];
#pragma unroll
    for (int e = 0; e < kPer; ++e)
        w[e] = __builtin_fmaf(sc, static_cast<float>((q[e >> 2] >> (8 * (e & 3) + sh)) & 15u), -mn);
    const int64_t o = blk * kQ4kBlockElems + sb * 32 + part * kPer;
    if constexpr (BF16) {
        *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(out) + o) =
            u32x4{bf16_pair(w[0], w[1]), bf16_pair(w[2], w[3]), bf16_pair(w[4], w[5]), bf16_pair(w[6], w[7])};
    } else {
        *reinterpret_cast<f32x4*>(static_cast<float*>(out) + o) = f32x4{w[0], w[1], w[2], w[3]};
    }
}

// Grid-stride over units, kUnroll per lane per round so that several loads
// are in flight per wave; one lane per unit made 52 K short waves for a
// 8192 x 3072 weight, and wave launch, not HBM, set the time.
constexpr int kUnroll = 4;

template <bool BF16>
__global__ __launch_bounds__(256) void k_dequant_q4k(const uint8_t* __restrict__ W, void* __restrict__ out,
                                                     int64_t units) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
    for (int64_t u0 = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; u0 < units; u0 += stride * kUnroll) {
#pragma unroll
        for (int j = 0; j < kUnroll; ++j) {
            const int64_t u = u0 + j * stride;
            if (u < units) dequant_unit<BF16>(W, out, u);
        }
    }
}

// A GEMM's two input conversions in one launch: units [0, wunits)
// dequantize W to bf16, the next aunits convert 8 f32 activations each to
// bf16 (the same rounding).
__global__ __launch_bounds__(256) void k_dequant_q4k_cvt(const uint8_t* __restrict__ W, uint16_t* __restrict__ wout,
                                                         int64_t wunits, const float* __restrict__ A,
                                                         uint16_t* __restrict__ aout, int64_t aunits) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 256, total = wunits + aunits;
    for (int64_t u0 = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; u0 < total; u0 += stride * kUnroll) {
#pragma unroll
        for (int j = 0; j < kUnroll; ++j) {
            const int64_t u = u0 + j * stride;
            if (u < wunits) {
                dequant_unit<true>(W, wout, u);
            } else if (u < total) {
                const int64_t i = u - wunits;
                const f32x4 a = reinterpret_cast<const f32x4*>(A)[2 * i];
                const f32x4 b = reinterpret_cast<const f32x4*>(A)[2 * i + 1];
                reinterpret_cast<u32x4*>(aout)[i] = u32x4{bf16_pair(a[0], a[1]), bf16_pair(a[2], a[3]),
                                                          bf16_pair(b[0], b[1]), bf16_pair(b[2], b[3])};
            }
        }
    }
}

// --- quantizer -------------------------------------------------------------

// Rust-style saturating f32 -> u8 (quant_q4k.cpp:27-35).
__device__ __forceinline__ uint32_t sat_u8(float v) {
    if (!(v > 0.0f)) return 0;
    if (v >= 255.0f) return 255;
    return static_cast<uint32_t>(v);
}

// Truncating f32 -> f16 bits (bf16.hpp:101-126).
__device__ __forceinline__ uint32_t f32_to_f16_trunc(float v) {
    const uint32_t bits = __float_as_uint(v);
    const uint32_t sign = (bits >> 16) & 0x8000u;
    const int32_t exp = static_cast<int32_t>((bits >> 23) & 0xffu);
    const uint32_t mant = bits & 0x7fffffu;
    if (exp == 0xff) return sign | 0x7c00u | (mant >> 13);
    const int32_t e16 = exp - 127 + 15;
    if (e16 >= 0x1f) return sign | 0x7c00u;
    if (e16 <= 0) {
        if (e16 < -10) return sign;
        const uint32_t m = mant | 0x800000u;
        return sign | (m >> (static_cast<uint32_t>(1 - e16) + 13u));
    }
    return sign | (static_cast<uint32_t>(e16) << 10) | (mant >> 13);
}

// std::min / std::max argument order of the reference (first wins on ties).
__device__ __forceinline__ float ref_max(float a, float b) { return a < b ? b : a; }

// The value of another lane: DPP control c (0xb1: lane ^ 1, 0x4e: lane ^ 2,
// 0x141: mirrored within 8 lanes, 0x128: lane ^ 8), lane ^ 16, lane ^ 32.
template <int C>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t x) {
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), C, 0xf, 0xf, true));
}
template <int C>
__device__ __forceinline__ float dpp_f32(float x) {
    return __uint_as_float(dpp_u32<C>(__float_as_uint(x)));
}
__device__ __forceinline__ uint32_t lane_xor16(uint32_t x, int lane) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return (lane & 16) ? r[0] : r[1];
}
__device__ __forceinline__ uint32_t lane_xor32(uint32_t x, int lane) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return (lane & 32) ? r[0] : r[1];
}
// The largest / the OR over the 8 lanes l + 8 j.
__device__ __forceinline__ float max_of_8(float x, int lane) {
    x = fmaxf(x, dpp_f32<0x128>(x));
    x = fmaxf(x, __uint_as_float(lane_xor16(__float_as_uint(x), lane)));
    return fmaxf(x, __uint_as_float(lane_xor32(__float_as_uint(x), lane)));
}
__device__ __forceinline__ uint32_t or_of_8(uint32_t x, int lane) {
    x |= dpp_u32<0x128>(x);
    x |= lane_xor16(x, lane);
    return x | lane_xor32(x, lane);
}
// x of the lane that has this lane's sub-block (8 lanes) of block B.
template <int B>
__device__ __forceinline__ float from_owner(float x) {
    return __uint_as_float(static_cast<uint32_t>(
        __builtin_amdgcn_ds_swizzle(static_cast<int>(__float_as_uint(x)), 0x18 | ((2 * B) << 5))));
}

// The nibble of v: min(15, sat_u8((v + mn) / sc + 0.5)) with r = 1 / sc and
// lim = 15 sc (exact: 21 bits), or sc = r = lim = 0 for a sub-block whose
// nibbles are all 0.  Above lim the nibble is 15 either way; NaN and negative
// sums become 0 in the clamp.  Two remainder steps make q the correctly
// rounded quotient (P. Markstein, Computation of elementary functions on the
// IBM RISC System/6000, 1990): the first leaves q within one ulp, the second,
// on an exact remainder and a correctly rounded r, rounds as a division does.
// Quotients too small for that are far below the 0.5 that would matter.
__device__ __forceinline__ uint32_t nibble(float v, float mn, float sc, float r, float lim) {
    const float x = __builtin_amdgcn_fmed3f(v + mn, 0.0f, lim);
    float q = x * r;
    q = __builtin_fmaf(__builtin_fmaf(-sc, q, x), r, q);
    q = __builtin_fmaf(__builtin_fmaf(-sc, q, x), r, q);
    return static_cast<uint32_t>(q + 0.5f);
}

// Bound: the bytes (reading the f32 weight), once the VALU work per value is
// small: with one block per wave every lane computed its sub-block's and
// block's scalars (9 divisions, 8 lanes for one sub-block, 64 for one block)
// and 4 values' nibbles, about 300 instructions per 256 values, and the VALU
// bound the kernel.  With four blocks per wave the min / max reduction ends
// with one sub-block in each pair of lanes (reduce-scatter over the blocks),
// so the scalars are computed once for all four.  8192 x 3072: 57.3 -> 22.5 us
// (2.0 -> 5.1 TB/s); 8192 x 12288: 214 -> 99 us.
__global__ __launch_bounds__(256) void k_quantize_q4k(const float* __restrict__ w, uint8_t* __restrict__ out,
                                                      int64_t blocks) {
    const int64_t blk0 = (static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6)) * 4;
    if (blk0 >= blocks) return;
    const int lane = threadIdx.x & 63;
    f32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)  // (past the end: the last block again, not stored)
        v[i] = *reinterpret_cast<const f32x4*>(w + min(blk0 + i, blocks - 1) * 256 + 4 * lane);

    // Step 1: sub-block (8 lanes) min / max, seeded with +-inf as the
    // reference's loop is, so a NaN input is skipped exactly as there.
    float lo[4], hi[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        lo[i] = __builtin_inff();
        hi[i] = -__builtin_inff();
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            lo[i] = fminf(lo[i], v[i][e]);
            hi[i] = fmaxf(hi[i], v[i][e]);
        }
    }
    // lanes with bit 2 (then bit 1) set go on with the later half of the blocks
    const bool b2 = (lane & 4) != 0, b1 = (lane & 2) != 0;
    float lo2[2], hi2[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        lo2[i] = fminf(b2 ? lo[i + 2] : lo[i], dpp_f32<0x141>(b2 ? lo[i] : lo[i + 2]));
        hi2[i] = fmaxf(b2 ? hi[i + 2] : hi[i], dpp_f32<0x141>(b2 ? hi[i] : hi[i + 2]));
    }
    float smin = fminf(b1 ? lo2[1] : lo2[0], dpp_f32<0x4e>(b1 ? lo2[0] : lo2[1]));
    float smax = fmaxf(b1 ? hi2[1] : hi2[0], dpp_f32<0x4e>(b1 ? hi2[0] : hi2[1]));
    smin = fminf(smin, dpp_f32<0xb1>(smin));
    smax = fmaxf(smax, dpp_f32<0xb1>(smax));
    // from here on this lane has sub-block lane / 8 of block (lane & 6) / 2
    float sub_min = 0.0f, range = smax;
    if (!(smin >= 0.0f)) {
        sub_min = smin;
        range = smax > smin ? smax - smin : 0.0f;
    }
    const float sub_scale = range > 0.0f ? range / 15.0f : 0.0f;
    // Step 2: block maxima over the 8 sub-blocks.
    const float max_scale = max_of_8(ref_max(0.0f, sub_scale), lane);
    const float max_min = max_of_8(ref_max(0.0f, -sub_min), lane);
    const float d = max_scale > 0.0f ? max_scale / 63.0f : 0.0f;
    const float dmin = max_min > 0.0f ? max_min / 63.0f : 0.0f;
    // Step 3: 6-bit scale and min of this lane's sub-block.
    uint32_t sv = 0, mv = 0;
    if (d > 0.0f) {
        const float inv = 1.0f / d;
        sv = min(63u, sat_u8(sub_scale * inv + 0.5f));
    }
    if (dmin > 0.0f) {
        const float inv = 1.0f / dmin;
        mv = min(63u, sat_u8(-sub_min * inv + 0.5f));
    }
    // Step 4: f16 header (truncating).
    const uint32_t d16 = f32_to_f16_trunc(d), m16 = f32_to_f16_trunc(dmin);
    const float dv = f16_bits_to_f32(d16), mvv = f16_bits_to_f32(m16);
    // Step 6: nibbles with the f16-rounded scales (all 0 for a scale of 0,
    // infinite or NaN).
    const float sc0 = dv * static_cast<float>(sv), mn0 = mvv * static_cast<float>(mv);
    const bool some = sc0 > 0.0f && sc0 < __builtin_inff();
    const float sc1 = some ? sc0 : 0.0f, r1 = some ? 1.0f / sc0 : 0.0f;
    uint32_t qn[4];
    auto block_nibbles = [&](const f32x4& x, float sc, float mn, float r) {
        const float lim = 15.0f * sc;
        uint32_t q = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) q |= nibble(x[e], mn, sc, r, lim) << (8 * e);
        return q;
    };
    qn[0] = block_nibbles(v[0], from_owner<0>(sc1), from_owner<0>(mn0), from_owner<0>(r1));
    qn[1] = block_nibbles(v[1], from_owner<1>(sc1), from_owner<1>(mn0), from_owner<1>(r1));
    qn[2] = block_nibbles(v[2], from_owner<2>(sc1), from_owner<2>(mn0), from_owner<2>(r1));
    qn[3] = block_nibbles(v[3], from_owner<3>(sc1), from_owner<3>(mn0), from_owner<3>(r1));
    // Value 4*lane+e sits in chunk c = lane/16; lanes with (lane%16) < 8 hold
    // low nibbles, lane+8 the matching high nibbles.  Of each pair of blocks
    // the former lanes store the first, the latter the second.
    const bool b3 = (lane & 8) != 0;
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
        const uint32_t own = b3 ? qn[i + 1] : qn[i], got = dpp_u32<0x128>(b3 ? qn[i] : qn[i + 1]);
        const uint32_t word = b3 ? got | (own << 4) : own | (got << 4);
        const int64_t blk = blk0 + i + (b3 ? 1 : 0);
        if (blk < blocks)
            *reinterpret_cast<uint32_t*>(out + blk * kQ4kBlockBytes + 16 + 32 * (lane >> 4) + 4 * (lane & 7)) = word;
    }
    // Step 5: pack the 12 scale bytes (pack_scales, quant_q4k.cpp:43-55), each
    // sub-block j's share in its place.
    const int j = lane >> 3, sh = 8 * (j & 3);
    const bool up = j >= 4;
    const uint32_t s0 = or_of_8((up ? (sv & 0x30u) << 2 : sv) << sh, lane);
    const uint32_t s1 = or_of_8((up ? (mv & 0x30u) << 2 : mv) << sh, lane);
    const uint32_t s2 = or_of_8(up ? ((sv & 0x0fu) | ((mv & 0x0fu) << 4)) << sh : 0u, lane);
    const int64_t blk = blk0 + (lane >> 1);
    if (lane < 8 && (lane & 1) == 0 && blk < blocks)
        *reinterpret_cast<u32x4*>(out + blk * kQ4kBlockBytes) = u32x4{d16 | (m16 << 16), s0, s1, s2};
}

// Reference row-major Q4_K blocks -> tiled layout (q4k_mfma.hpp): one thread
// per (tile, super-block, lane) writes that lane's header dword and its two
// 16-byte halves of qs; rows past N are written as zeros.  With hd > 0 the
// rows of each head of hd rows are interleaved on the way: tiled row 2j of a
// head takes source row j, row 2j + 1 takes source row j + hd / 2 (the
// half-split RoPE pairs become adjacent rows).
__global__ __launch_bounds__(256) void k_q4k_tile(const uint8_t* __restrict__ src,
                                                  uint8_t* __restrict__ dst, int64_t n, int nb,
                                                  int64_t threads, int hd) {
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (gid >= threads) return;
    const int l = static_cast<int>(gid & 63);
    const int64_t tb = gid >> 6;  // tile * nb + b
    const int b = static_cast<int>(tb % nb);
    const int64_t t = tb / nb;
    const int g = l >> 4;
    const int64_t row = t * 16 + (l & 15);
    uint8_t* out = dst + tb * q4k_mfma::kTiledBlockBytes;
    uint32_t hdr = 0;
    u32x4 qa = {0u, 0u, 0u, 0u}, qb = {0u, 0u, 0u, 0u};
    if (row < n) {
        int64_t srow = row;
        if (hd > 0) {
            const int64_t r = row % hd;
            srow = row - r + (r >> 1) + ((r & 1) ? hd / 2 : 0);
        }
        const uint8_t* blk = src + (srow * nb + b) * kQ4kBlockBytes;
        const u32x4 h = ld16(blk);
        uint32_t sv0, mv0, sv1, mv1;
        decode_scale_min(make_scale_sel(2 * g), h[1], h[2], h[3], sv0, mv0);
        decode_scale_min(make_scale_sel(2 * g + 1), h[1], h[2], h[3], sv1, mv1);
        const uint32_t dbyte = (h[0] >> (8 * g)) & 0xffu;
        hdr = sv0 | (sv1 << 6) | (mv0 << 12) | (mv1 << 18) | (dbyte << 24);
        qa = ld16(blk + 16 + 32 * g);
        qb = ld16(blk + 32 + 32 * g);
    }
    reinterpret_cast<uint32_t*>(out)[l] = hdr;
    reinterpret_cast<u32x4*>(out + q4k_mfma::kTiledQa)[l] = qa;
    reinterpret_cast<u32x4*>(out + q4k_mfma::kTiledQb)[l] = qb;
}

}  // namespace

// Grid for `units` lanes of work: one round of kUnroll units per lane, at
// most 8 workgroups per CU.
static dim3 unit_grid(int64_t units) {
    const int64_t want = (units + 256 * kUnroll - 1) / (256 * kUnroll), cap = 8 * device_info().cus;
    return dim3(static_cast<unsigned>(want < cap ? (want < 1 ? 1 : want) : cap));
}

hipError_t launch_dequant_q4k(const void* w, void* out, bool bf16, int64_t n, int64_t k,
                              hipStream_t s) {
    const int64_t units = n * k / (bf16 ? 8 : 4);
    if (bf16)
        hipLaunchKernelGGL(k_dequant_q4k<true>, unit_grid(units), dim3(256), 0, s, static_cast<const uint8_t*>(w),
                           out, units);
    else
        hipLaunchKernelGGL(k_dequant_q4k<false>, unit_grid(units), dim3(256), 0, s, static_cast<const uint8_t*>(w),
                           out, units);
    return hipGetLastError();
}

hipError_t launch_dequant_q4k_cvt(const void* w, uint16_t* wout, int64_t n, int64_t k, const float* a,
                                  uint16_t* aout, int64_t a_elems, hipStream_t s) {
    const int64_t wunits = n * k / 8, aunits = a_elems / 8;
    hipLaunchKernelGGL(k_dequant_q4k_cvt, unit_grid(wunits + aunits), dim3(256), 0, s,
                       static_cast<const uint8_t*>(w), wout, wunits, a, aout, aunits);
    return hipGetLastError();
}

hipError_t launch_quantize_q4k(const float* w, void* blocks, int64_t n, int64_t k,
                               hipStream_t s) {
    const int64_t nblk = n * (k / 256);
    const unsigned grid = static_cast<unsigned>((nblk + 15) / 16);
    hipLaunchKernelGGL(k_quantize_q4k, dim3(grid), dim3(256), 0, s, w, static_cast<uint8_t*>(blocks), nblk);
    return hipGetLastError();
}

hipError_t launch_q4k_tile(const void* blocks, void* tiled, int64_t n, int64_t k, hipStream_t s, int head_dim) {
    const int nb = static_cast<int>(k / 256);
    const int64_t threads = (n + 15) / 16 * nb * 64;
    const int64_t grid = (threads + 255) / 256;
    hipLaunchKernelGGL(k_q4k_tile, dim3(static_cast<unsigned>(grid)), dim3(256), 0, s,
                       static_cast<const uint8_t*>(blocks), static_cast<uint8_t*>(tiled), n, nb,
                       threads, head_dim);
    return hipGetLastError();
}

}  // namespace rt_hip
