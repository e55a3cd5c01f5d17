// flux_attention.hip -- FLUX's multi-head attention with no mask (every token
// attends to every token), streamed over key tiles with an online softmax:
// the reference's flux_attention (src/shaders/flux.msl:145-331) and the CPU
// attention it replaces (src/flux.cpp:282-323).
//
// q, k, v, out: [T][n_heads * D] f32 rows; D = head_dim, a multiple of 8 up
// to 128 (the reference's limits, metal_flux.mm:443-452).
// out[i][h] = sum_j softmax_j(scale * q_i . k_j) v_j for head h.
//
// A workgroup owns a block of 32 queries per wave (8 waves, 4 where the blocks
// would leave CUs idle) of one head and streams K and V once for all of them
// in tiles of 32 keys through LDS rings.
//
// f32 products on the bf16 matrix cores.  Every f32 factor is split into three
// bf16 limbs with h + m + l == x exactly (24 bits of significand; K and Q where
// the last bit is 2^-133 or more, V and P always, see kUp), and a product is the
// six limb products hh, hm, mh, mm, hl, lh on v_mfma_f32_32x32x16_bf16: products
// of bf16 values are exact in f32 and the three left out (ml, lm, ll) are
// together below 2^-24 of the product, at most the rounding of one f32
// multiplication.  The matrix cores do a bf16 product at
// 16 times the f32 rate, so six cost 3/8 of one f32 product.  Q's limbs live
// in registers (split once per block), K's and V's are split as each tile is
// staged, P's in the registers its scores were computed in:
//  * S^T = K Q^T per 32-key x 32-query tile: lane (h = l/32, n = l%32) supplies
//    K[key n] and Q[query n], dims 16a + 8h .. + 7 of step a; the result
//    leaves lane (h, n) holding query n's scores against keys 8i + 4h + r
//    (register 4i + r).  hh and the five corrections have accumulators of
//    their own, added at the end.
//  * Online softmax per query: the running maximum; each half of a query's
//    keys keeps its own denominator (added at the end); the accumulator is
//    rescaled by exp(m_old - m_new) where a maximum of the wave moved
//    (flux.msl:232-271).  Exponentials are powers of two: log2(e) and the scale
//    are in Q's limbs.
//  * O^T += V^T P^T: lane (h, n) supplies P[query n] of the eight keys it
//    holds in registers 8s .. 8s + 7 and V[those keys][dim 32c + n], which V's
//    LDS rows (one per dim, keys in that order) hold as 16 bytes; the result
//    leaves lane (h, n) holding O[query n][dims 32c + 8i + 4h + r].
// From a tile that holds a value of 2^64 or more in K, of 2^48 in V, an infinity
// or a NaN, or throughout a block with a query of 2^55 or more, the block takes f32
// MFMA steps on the staged f32 tiles: products that overflow and infinities
// then behave as in f32 arithmetic (a limb's product could overflow to the
// other sign).  A loop of its own: the limb loop has no registers to spare.
// It costs what f32 steps do: t = 4352, 24 x 128 with an infinity in one head
// 2790 us, in the middle tile of all 2090 (with f32 MFMA throughout 2070; with
// the operands read from memory step by step 10650 and 7020).
//
// The head is padded to DP in {32, 64, 128} dims with zeros (they add
// nothing to a score and are never stored).  Keys past T are masked to -inf
// (weight 0), their tile rows zero-filled by the loads' range check; query
// rows past T are computed and not stored.
//
// Bound: the matrix cores.  A 32-key tile of a CU's 256 queries is 96 MFMAs a
// wave, 6144 cycles a SIMD; between them come the softmax and the limb splits,
// about 440 VALU instructions a wave and tile.  Measured at t = 4352, 24 heads
// of 128: 2070 us with f32 MFMA (71% of that unit's peak, where 1480 us is the
// least), 1175-1290 us with limbs: MFMA busy 57% at the 1.76 GHz the power
// limit leaves (2.2 GHz when half idle), which also sets the spread.  Without
// the limb staging it would be 1075.
// t = 1280: 230 -> 160 us; t = 2622, 18 x 88: 750 -> 330; t = 477, 13 x 128:
// 87 -> 61; t = 466, 9 x 64: 39 -> 33; t = 100, 12 x 64: 13.5 -> 12.8 (t = 33,
// 4 x 32: 5.9 -> 6.5).  The error against float64 at t = 4352 fell from 1.6e-6
// to 8.5e-7.
//  * Of the two waves of a SIMD one is in its products (priority 1) while the
//    other does its softmax and staging, a barrier between phases: 1250 us;
//    free-running waves 1410.
//  * Tiles go through LDS copies of the raw f32 (no registers), are split once
//    and read by all 8 waves: blocks of 128 queries halve the reuse of the
//    splits and are taken only where 256 leave CUs idle.
#include <cmath>

#include "rt_common.hpp"
#include "rt_launch.hpp"

namespace rt_hip {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kBK = 32;  // keys per tile
constexpr uint32_t kNoRead = 0x7ffffff0u;  // past every tile's range: reads zeros

// V and the weights P enter the limbs times 2^16: bf16 has f32's exponents but 7
// bits, so the third limb of a value below 2^-109 would fall below bf16's
// smallest value, 2^-133.  With the factor every bit of an f32 value (2^-149 and
// up) is in reach.  (The matrix unit keeps bf16 values below 2^-126.)
constexpr float kUp = 0x1p16f, kDown = 0x1p-32f;

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// LDS: a ring of two tiles of K limbs [3][32 keys][DP] bf16, then one of three
// tiles of V limbs [3][DP dims][32 keys], then each wave's share of a tile's
// K and V as they are in memory, then the first tile without limbs.
template <int DP>
constexpr int limb_plane() {
    return 64 * DP;
}
// K units (key, 8 dims) and V units (4 keys, 1 dim) a thread stages: 4 DP and
// 8 DP of them in all.
constexpr int k_units(int dp, int nt) { return (4 * dp + nt - 1) / nt; }
constexpr int v_units(int dp, int nt) { return (8 * dp + nt - 1) / nt; }
template <int DP, int NW>
constexpr int raw_wave_bytes() {  // per wave: 2 x 16 bytes a lane and K unit, 4 x 4 a lane and V unit
    return 64 * (32 * k_units(DP, NW * 64) + 16 * v_units(DP, NW * 64));
}
template <int DP, int NW>
constexpr int raw_bytes() {
    return NW * raw_wave_bytes<DP, NW>();
}
template <int DP, int NW>
constexpr size_t flux_lds_bytes() {
    return static_cast<size_t>(15) * limb_plane<DP>() + raw_bytes<DP, NW>() + 16;
}
// 16-byte granule gr (8 dims) of a key's row: rows are exchanged granule-wise
// so that the 16 lanes an LDS read serves together hit distinct banks.
template <int DP>
__device__ __forceinline__ int k_off(int key, int gr) {
    constexpr int kMask = DP / 8 - 1, kShift = DP == 128 ? 0 : (DP == 64 ? 1 : 2);
    return key * (2 * DP) + ((gr ^ ((key >> kShift) & kMask & 15)) << 4);
}
// 16-byte unit u = 2s + h of a dim's row: keys 16s + 4h + {0..3, 8..11}.
__device__ __forceinline__ int v_off(int dim, int u) { return dim * 64 + ((u ^ ((dim >> 2) & 3)) << 4); }

// Three bf16 limbs of a pair, packed: h + m + l == x for finite x that bf16
// can hold (each residual is exact in f32).
__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = bf16_pair(a, b);
    const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
    m = bf16_pair(ra, rb);
    l = bf16_pair(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xffff0000u));
}
__device__ __forceinline__ void split8(const float (&v)[8], u32x4& h, u32x4& m, u32x4& l) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t hh, mm, ll;
        split2(v[2 * i], v[2 * i + 1], hh, mm, ll);
        h[i] = hh;
        m[i] = mm;
        l[i] = ll;
    }
}
// Adds the squares of a pair's high limbs to acc: NaN or infinite once one of
// them is NaN or 2^64 or more in magnitude.  A sum that stays finite bounds
// every value of K and, times 2^16, of V; with |q| < 2^55 a score (128 products
// below 2^119) and each of its limb products stays finite too, and so does a
// sum of T < 2^31 products of V and P (2^64 2^16 each).
constexpr float kQLimit = 0x1p55f;
__device__ __forceinline__ float limb_check(uint32_t h, float acc) {
    const bf16x2 v = __builtin_bit_cast(bf16x2, h);
    return __builtin_amdgcn_fdot2_f32_bf16(v, v, acc, false);
}
__device__ __forceinline__ bool not_finite(float x) { return (__float_as_uint(x) & 0x7fffffffu) >= 0x7f800000u; }

__device__ __forceinline__ f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                   0);
}

// Partial states of a split query block: O [BQ][DP], then m [BQ], l [BQ].
constexpr int piece_floats(int bq, int dp) { return bq * dp + 2 * bq; }

// Stored and reloaded with agent-scope (device-coherent) accesses: they
// bypass the per-XCD L2, so the workgroup that merges sees the other
// workgroup's stores once those have completed.
__device__ __forceinline__ void st_dev(float* p, float v) {
    __hip_atomic_store((__attribute__((address_space(1))) float*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_dev(const float* p) {
    return __hip_atomic_load((const __attribute__((address_space(1))) float*)p, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}

// This wave's LDS reads and writes, or its copies into LDS, are done (and no
// access moves across).
__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void copies_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The value of lane l ^ 32.
__device__ __forceinline__ float other_half(float x, int h) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(h ? r[0] : r[1]);
}

// Work: item i = (head i / nqb, query block i % nqb) over key tiles
// [0, ntile).  Without `part` workgroup (head, block) = (blockIdx.x,
// blockIdx.y) does one whole item.  With it (more items than workgroup
// slots) the flat sequence of (item, tile) units is cut into gridDim.x equal
// ranges of `per` >= ntile units, one per workgroup, so every workgroup does
// the same work and no partial round is left at the end.  An item cut by
// the boundary between workgroups w and w + 1 has two pieces: each stores
// its state (o, m, l) in part[w][piece] and counts its arrival in cnt[w];
// the second to arrive merges the two states and stores the output.
template <int DP, int NW>
__global__ __launch_bounds__(NW* kWave, NW == 4 && DP <= 64 ? 2 : 1) void k_flux_attn(const float* __restrict__ Q, const float* __restrict__ K,
                                                          const float* __restrict__ V, float* __restrict__ O, int T,
                                                          int n_heads, int D, float scale2, float* __restrict__ part,
                                                          uint32_t* __restrict__ cnt, int per) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ uint32_t arrival;
    constexpr int NT = NW * kWave, BQ = 32 * NW;
    constexpr int KS = DP / 16, NC = DP / 32;      // MFMA steps over the dims, 32-dim output blocks
    constexpr int kPlane = limb_plane<DP>();
    constexpr int KU = k_units(DP, NT), VU = v_units(DP, NT);
    uint8_t* const ldsV = lds + 6 * kPlane;
    int* const first_bad = reinterpret_cast<int*>(lds + 15 * kPlane + raw_bytes<DP, NW>());
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    uint8_t* const raw = lds + 15 * kPlane + wave * raw_wave_bytes<DP, NW>();
    const int64_t stride = static_cast<int64_t>(n_heads) * D;
    const int ntile = (T + kBK - 1) / kBK, nqb = (T + BQ - 1) / BQ;
    // Two phases alternate: products (priority 1) and softmax + staging.  With
    // 8 waves, w and w + 4 share a SIMD and the second group of four runs one
    // phase behind the first, so that one wave of a SIMD has the matrix cores
    // while the other has the VALU.
    constexpr bool kTwo = NW == 8;
    const bool second = kTwo && wave >= 4;

    // the units of this workgroup
    int64_t u, u_end;
    if (part) {
        u = static_cast<int64_t>(blockIdx.x) * per;
        u_end = min(u + per, static_cast<int64_t>(n_heads) * nqb * ntile);
    } else {
        const int64_t item = static_cast<int64_t>(blockIdx.x) * nqb + blockIdx.y;
        u = item * ntile;
        u_end = u + ntile;
    }
    while (u < u_end) {
        const int64_t item = u / ntile;
        const int t0 = static_cast<int>(u % ntile);
        const int t1 = static_cast<int>(min(static_cast<int64_t>(ntile), t0 + (u_end - u)));
        u += t1 - t0;
        const int head = static_cast<int>(item / nqb), q0 = static_cast<int>(item % nqb) * BQ;
        const float* kb = K + static_cast<int64_t>(head) * D;
        const float* vb = V + static_cast<int64_t>(head) * D;

        // A tile's K and V, copied into the wave's own LDS (no registers) in a
        // product phase; the limbs enter the rings in the phase after it.
        const int vdim = tid % DP, vquad = tid / DP;
        const uint32_t s4 = static_cast<uint32_t>(stride * 4);
        auto load_tile = [&](int i0) {
            const int base = (t0 + i0) * kBK, rows = min(kBK, T - base);
            const uint32_t bytes = static_cast<uint32_t>(((rows - 1) * stride + D) * 4);
            const BufRsrc rk = make_rsrc_n(kb + base * stride, bytes);
            const BufRsrc rv = make_rsrc_n(vb + base * stride, bytes);
#pragma unroll
            for (int i = 0; i < KU; ++i) {
                const int id = tid + NT * i, key = id / (DP / 8), dim = 8 * (id % (DP / 8));
                const uint32_t off = dim < D && key < kBK ? static_cast<uint32_t>(key) * s4 + 4 * dim : kNoRead;
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(
                        rk, (__attribute__((address_space(3))) void*)(raw + (2 * i + j) * 1024), 16,
                        static_cast<int>(off + 16u * j), 0, 0, 0);
            }
            // (kNoRead plus up to 31 rows stays past the range and below 2^32)
            const uint32_t off = vdim < D && vquad < 8 ? static_cast<uint32_t>(4 * vquad) * s4 + 4 * vdim : kNoRead;
#pragma unroll
            for (int i = 0; i < VU; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(
                        rv, (__attribute__((address_space(3))) void*)(raw + KU * 2048 + (4 * i + j) * 256), 4,
                        static_cast<int>(off + static_cast<uint32_t>(4 * i * (NT / DP) + j) * s4), 0, 0, 0);
        };
        auto stage_tile = [&](int i0) {
            uint8_t* const sk = lds + (i0 & 1) * 3 * kPlane;
            uint8_t* const sv = ldsV + (i0 % 3) * 3 * kPlane;
            float bad = 0.0f;
#pragma unroll
            for (int i = 0; i < KU; ++i) {
                const int id = tid + NT * i, key = id / (DP / 8), gr = id % (DP / 8);
                if (KU * NT > 4 * DP && id >= 4 * DP) break;
                const f32x4 x0 = *reinterpret_cast<const f32x4*>(raw + 2 * i * 1024 + lane * 16);
                const f32x4 x1 = *reinterpret_cast<const f32x4*>(raw + (2 * i + 1) * 1024 + lane * 16);
                const float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
                u32x4 a, b, c;
                split8(x, a, b, c);
                uint8_t* const d = sk + k_off<DP>(key, gr);
                *reinterpret_cast<u32x4*>(d) = a;
                *reinterpret_cast<u32x4*>(d + kPlane) = b;
                *reinterpret_cast<u32x4*>(d + 2 * kPlane) = c;
#pragma unroll
                for (int e = 0; e < 4; ++e) bad = limb_check(a[e], bad);
            }
#pragma unroll
            for (int i = 0; i < VU; ++i) {
                const int dim = vdim, quad = vquad + i * (NT / DP);
                if (VU * NT > 8 * DP && quad >= 8) break;
                // keys 4 quad .. + 3 = 16s + 8a + 4h' ..: unit 2s + h', half a
                const int s = quad >> 2, a8 = (quad >> 1) & 1, hh = quad & 1;
                u32x2 a, b, c;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    uint32_t x, y, z;
                    const uint8_t* const src = raw + KU * 2048 + (4 * i + 2 * e) * 256 + lane * 4;
                    split2(*reinterpret_cast<const float*>(src) * kUp, *reinterpret_cast<const float*>(src + 256) * kUp, x, y,
                           z);
                    a[e] = x;
                    b[e] = y;
                    c[e] = z;
                }
                uint8_t* const d = sv + v_off(dim, 2 * s + hh) + 8 * a8;
                *reinterpret_cast<u32x2*>(d) = a;
                *reinterpret_cast<u32x2*>(d + kPlane) = b;
                *reinterpret_cast<u32x2*>(d + 2 * kPlane) = c;
#pragma unroll
                for (int e = 0; e < 2; ++e) bad = limb_check(a[e], bad);
            }
            if (not_finite(bad)) atomicMin(first_bad, i0);
        };

        lds_wait();  // (of the item before: the copies overwrite it)
        load_tile(0);
        // this lane's query row (n of the wave's 32): dims 16a + 8h .. + 7
        const int qrow = q0 + wave * 32 + n;
        const float* qb = Q + static_cast<int64_t>(head) * D;
        u32x4 qh[KS], qm[KS], ql[KS];
        bool qbad = false;
        f32x4 qx[KS][2];  // all loads in flight at once; rows past T read row T - 1 (not stored)
#pragma unroll
        for (int a = 0; a < KS; ++a) {
            const int dim = min(16 * a + 8 * h, D - 8);
            const f32x4* p = reinterpret_cast<const f32x4*>(qb + min(qrow, T - 1) * stride + dim);
            qx[a][0] = p[0];
            qx[a][1] = p[1];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int a = 0; a < KS; ++a) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                x[e] = 16 * a + 8 * h < D ? qx[a][e >> 2][e & 3] : 0.0f;
                qbad |= !(fabsf(x[e]) < kQLimit);
                x[e] *= scale2;  // (the scores then come out scaled)
            }
            split8(x, qh[a], qm[a], ql[a]);
            __builtin_amdgcn_sched_barrier(0);
        }
        f32x16 o[NC];  // o[c][4i + r]: O[query n][dim 32c + 8i + 4h + r]
#pragma unroll
        for (int c = 0; c < NC; ++c) o[c] = f32x16{};
        float m_run = -__builtin_inff(), l_run = 0.0f;  // of query n; l of this half's keys

        // Scores of query n, times scale log2(e), masked and turned into weights;
        // the running state (m in powers of two) and the accumulator moved to
        // the new maximum.
        auto softmax = [&](f32x16& s, int base) {
            float mx = -__builtin_inff();
            if (base + kBK > T) {
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (base + 8 * (e >> 2) + 4 * h + (e & 3) >= T) s[e] = -__builtin_inff();
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[e]);
            mx = fmaxf(mx, other_half(mx, h));
            const float m_new = fmaxf(m_run, mx);  // finite for finite scores: key `base` is valid
            const float alpha = exp2_fast(m_run - m_new);  // 0 on the first tile
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                s[e] = exp2_fast(s[e] - m_new);  // -inf -> 0
                sum += s[e];
            }
            l_run = l_run * alpha + sum;
            m_run = m_new;
            if (__builtin_amdgcn_ballot_w64(!(alpha == 1.0f)) != 0) {
#pragma unroll
                for (int c = 0; c < NC; ++c) o[c] *= alpha;
            }
        };

        constexpr int kMask = (DP / 8 - 1) & 15, kShift = DP == 128 ? 0 : (DP == 64 ? 1 : 2);
        const int kbase = n * (2 * DP) + ((h ^ ((n >> kShift) & 1)) << 4);
        f32x16 s;
        u32x4 ph[2], pm[2], pl[2];  // limbs of P: keys of registers 8t .. 8t + 7
        f32x16 sc;
        // The fragments of one step: limbs of 16 dims of K, or of 16 keys of V
        // for a 32-dim block.  Steps run one behind the next step's reads (the
        // products of a step cover their latency; the scheduling barriers keep
        // the reads ahead).
        u32x4 fr[2][3];
        auto read3 = [&](u32x4 (&f)[3], const uint8_t* p) {
#pragma unroll
            for (int l = 0; l < 3; ++l) f[l] = *reinterpret_cast<const u32x4*>(p + l * kPlane);
        };
        // k_off(n, 2a + h) in two parts, recomputed each tile (opaque to the
        // compiler, which would keep all KS of them in registers)
        int kx = 0;
        auto k_frag = [&](int i0, int a) -> const uint8_t* {
            return lds + (i0 & 1) * 3 * kPlane + kbase + ((2 * a) << 4 ^ kx);
        };
        auto v_frag = [&](const uint8_t* st, int j) -> const uint8_t* {  // j = t * NC + c
            return st + v_off(32 * (j % NC) + n, 2 * (j / NC) + h);
        };
        // S^T of tile i0; fr[buf] holds step 0.
        auto scores = [&](int i0, int buf) {
            sc = f32x16{};
            s = f32x16{};
#pragma unroll
            for (int a = 0; a < KS; ++a) {
                u32x4(&f)[3] = fr[(a + buf) & 1];
                if (a + 1 < KS) read3(fr[(a + 1 + buf) & 1], k_frag(i0, a + 1));
                __builtin_amdgcn_sched_barrier(0);
                s = mma(f[0], qh[a], s);
                sc = mma(f[0], qm[a], sc);
                sc = mma(f[1], qh[a], sc);
                sc = mma(f[1], qm[a], sc);
                sc = mma(f[0], ql[a], sc);
                sc = mma(f[2], qh[a], sc);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        int nt = t1 - t0;  // tiles the limb loop takes
        // O^T += V^T P^T of tile i0, then the scores of tile i0 + 1.
        auto products = [&](int i0) {
            kx = ((n >> kShift) & kMask & ~1) << 4;
            asm volatile("" : "+v"(kx));
            const uint8_t* const st = ldsV + (i0 % 3) * 3 * kPlane;
            read3(fr[0], v_frag(st, 0));
#pragma unroll
            for (int j = 0; j < 2 * NC; ++j) {
                u32x4(&f)[3] = fr[j & 1];
                read3(fr[(j + 1) & 1], j + 1 < 2 * NC ? v_frag(st, j + 1) : k_frag(i0 + 1, 0));
                __builtin_amdgcn_sched_barrier(0);
                const int t = j / NC, c = j % NC;
                o[c] = mma(f[2], ph[t], o[c]);
                o[c] = mma(f[0], pl[t], o[c]);
                o[c] = mma(f[1], pm[t], o[c]);
                o[c] = mma(f[1], ph[t], o[c]);
                o[c] = mma(f[0], pm[t], o[c]);
                o[c] = mma(f[0], ph[t], o[c]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (kTwo || i0 + 1 < nt) scores(i0 + 1, 0);
        };

        __syncthreads();  // every wave is done with the previous item's LDS
        if (tid == 0) *first_bad = nt;
        __syncthreads();
        copies_wait();
        stage_tile(0);
        // The second group, a phase behind, stages its share of a tile one
        // phase ahead of the first group's.
        const int ahead = second ? 2 : 1;
        if (second && nt > 1) {
            lds_wait();  // the copies overwrite what stage_tile(0) read
            load_tile(1);
            copies_wait();
            stage_tile(1);
        }
        if (qbad) atomicMin(first_bad, 0);
        __syncthreads();
        // Product phase i: O += P V of tile i - 1, then the scores of tile i.
        // Softmax phase i: the weights of tile i, and this thread's share of
        // tile i + ahead into LDS.  Tile i + 1 is whole before the first
        // group's product phase i + 1 (the second group wrote its share two
        // phases before, the first group one).  A tile's K was last read in
        // the second group's phase i, two phases before the slot is written
        // again; its V one product phase later, hence three slots.
        if (second) lds_barrier();
        nt = min(nt, __builtin_amdgcn_readfirstlane(*first_bad));
        if (t0 + ahead < t1) load_tile(ahead);
        kx = ((n >> kShift) & kMask & ~1) << 4;
        read3(fr[0], k_frag(0, 0));
        scores(0, 0);
        for (int i = 0; i < nt; ++i) {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(0);
            if (kTwo) lds_barrier();
            __builtin_amdgcn_sched_barrier(0);
            s += sc;
            softmax(s, (t0 + i) * kBK);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                float p[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) p[e] = s[8 * t + e] * kUp;
                split8(p, ph[t], pm[t], pl[t]);
            }
            // (opaque: the compiler would compute them in the next phase)
#pragma unroll
            for (int t = 0; t < 2; ++t) asm volatile("" : "+v"(ph[t]), "+v"(pm[t]), "+v"(pl[t]));
            copies_wait();
            if (t0 + i + ahead < t1) stage_tile(i + ahead);
            __builtin_amdgcn_sched_barrier(0);
            lds_barrier();
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
            nt = min(nt, __builtin_amdgcn_readfirstlane(*first_bad));
            if (t0 + i + 1 + ahead < t1) load_tile(i + 1 + ahead);
            products(i);  // (past the last tile: scores of whatever the slot holds, unused)
        }
        __builtin_amdgcn_s_setprio(0);
        if (kTwo && !second) lds_barrier();
        // The rest of a block that met a value without limbs, in f32.  The raw
        // copies of a tile, every wave's share, hold it whole: K units of 4 dims
        // at 16 bytes a lane, V units of one dim at 4.  Half h takes dims 8a + 4h
        // .. + 3 of a step.
        float unit = kDown;  // of o
        if (nt < t1 - t0) {
            unit = 1.0f;
#pragma unroll
            for (int c = 0; c < NC; ++c) o[c] *= kDown;
            const uint8_t* const shares = lds + 15 * kPlane;
            constexpr int kShare = raw_wave_bytes<DP, NW>(), kRows = NT / DP;
            const float* const qp = qb + min(qrow, T - 1) * stride;  // (rows past T are not stored)
            copies_wait();
            for (int tile = t0 + nt; tile < t1; ++tile) {
                load_tile(tile - t0);
                copies_wait();
                __syncthreads();
                s = f32x16{};
#pragma unroll 4
                for (int a = 0; a < DP / 8; ++a) {
                    const int id = n * (DP / 8) + a, tt = id % NT, dim = 8 * a + 4 * h;
                    const f32x4 ka = *reinterpret_cast<const f32x4*>(shares + (tt >> 6) * kShare +
                                                                     (2 * (id / NT) + h) * 1024 + (tt & 63) * 16);
                    const f32x4 qa = *reinterpret_cast<const f32x4*>(qp + min(dim, D - 4));
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        s = __builtin_amdgcn_mfma_f32_32x32x2f32(ka[e], dim < D ? qa[e] : 0.0f, s, 0, 0, 0);
                }
                s *= scale2;
                softmax(s, tile * kBK);
#pragma unroll
                for (int e = 0; e < 16; ++e) {  // key 8 (e / 4) + 4h + e % 4
                    const int quad = 2 * (e >> 2) + h;
#pragma unroll
                    for (int c = 0; c < NC; ++c) {
                        const int tt = (quad % kRows) * DP + 32 * c + n;
                        const float va = *reinterpret_cast<const float*>(
                            shares + (tt >> 6) * kShare + KU * 2048 + (4 * (quad / kRows) + (e & 3)) * 256 + (tt & 63) * 4);
                        o[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(va, s[e], o[c], 0, 0, 0);
                    }
                }
                __syncthreads();  // every wave has read this tile's shares
            }
        }
        l_run += other_half(l_run, h);

        if (t0 > 0 || t1 < ntile) {
            // One of two pieces of the item: its state, then the arrival.
            const int piece = t0 == 0 ? 0 : 1;
            const int bnd = static_cast<int>(blockIdx.x) - piece;  // the boundary that cut the item
            constexpr int kPiece = piece_floats(BQ, DP);
            float* mine = part + (static_cast<int64_t>(bnd) * 2 + piece) * kPiece;
            const int qi = wave * 32 + n;
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int e = 0; e < 16; ++e) st_dev(mine + qi * DP + 32 * c + 8 * (e >> 2) + 4 * h + (e & 3), o[c][e]);
            if (h == 0) {
                st_dev(mine + BQ * DP + qi, m_run);
                st_dev(mine + BQ * DP + BQ + qi, unit == 1.0f ? -l_run : l_run);  // l > 0: its sign is o's unit
            }
            wait_vmcnt<0>();
            __syncthreads();
            // Relaxed: the state went out in agent-scope stores that every wave
            // has waited for before the barrier, and the merging piece reads it
            // with agent-scope loads once the arrival's result is known.  (A
            // release wrote the XCD's whole L2 back: 700 tokens, 100 heads of 64
            // 134 us, 121 without.)
            if (tid == 0) arrival = __hip_atomic_fetch_add(cnt + bnd, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            if (arrival == 0) continue;  // the other piece merges
            // Merge: m = max, each side scaled by exp(m_side - m).  Two terms,
            // so the result does not depend on which piece merges.
            const float* other = part + (static_cast<int64_t>(bnd) * 2 + (1 - piece)) * kPiece;
            const float mo = ld_dev(other + BQ * DP + qi), lu = ld_dev(other + BQ * DP + BQ + qi), lo = fabsf(lu);
            const float unit_o = __builtin_signbit(lu) ? 1.0f : kDown;
            const float m = fmaxf(m_run, mo);
            float am = exp2_fast(m_run - m), ao = exp2_fast(mo - m);
            l_run = l_run * am + lo * ao;
            if (unit != unit_o) {
                am *= unit;
                ao *= unit_o;
                unit = 1.0f;
            }
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    o[c][e] = o[c][e] * am + ld_dev(other + qi * DP + 32 * c + 8 * (e >> 2) + 4 * h + (e & 3)) * ao;
            if (tid == 0) __hip_atomic_store(cnt + bnd, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // out[query n][dims 32c + 8i + 4h ..]: divide by the denominator
        if (qrow < T) {
            float* dst = O + qrow * stride + static_cast<int64_t>(head) * D;
            const float inv = unit / l_run;
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int dim = 32 * c + 8 * i + 4 * h;
                    if (dim < D)
                        *reinterpret_cast<f32x4*>(dst + dim) =
                            f32x4{o[c][4 * i], o[c][4 * i + 1], o[c][4 * i + 2], o[c][4 * i + 3]} * inv;
                }
        }
    }
}

// Workgroup slots of the 8-wave form: one per CU (152 KB of LDS at 128 dims,
// 256 registers a wave).
int flux_slots() { return static_cast<int>(device_info().cus); }

int padded_dims(int head_dim) { return head_dim <= 32 ? 32 : (head_dim <= 64 ? 64 : 128); }

template <int DP, int NW>
hipError_t run(const float* q, const float* k, const float* v, float* out, int64_t t, int n_heads, int d, float* part, uint32_t* cnt, hipStream_t s) {
    constexpr int BQ = 32 * NW;
    const int64_t nqb = (t + BQ - 1) / BQ, ntile = (t + kBK - 1) / kBK, items = n_heads * nqb;
    const size_t lds = flux_lds_bytes<DP, NW>();
    // log2(e) / sqrt(d): the scale of flux.cpp:290 and metal_flux.mm:264
    const float scale2 = static_cast<float>(1.4426950408889634 / std::sqrt(static_cast<double>(d)));
    if (!part) {
        const dim3 grid(static_cast<unsigned>(n_heads), static_cast<unsigned>(nqb));
        hipLaunchKernelGGL((k_flux_attn<DP, NW>), grid, dim3(NW * kWave), lds, s, q, k, v, out,
                           static_cast<int>(t), n_heads, d, scale2, nullptr, nullptr, 0);
    } else {
        const int slots = flux_slots();
        const int64_t per = (items * ntile + slots - 1) / slots;  // >= ntile: more items than slots
        hipLaunchKernelGGL((k_flux_attn<DP, NW>), dim3(static_cast<unsigned>(slots)), dim3(NW * kWave),
                           lds, s, q, k, v, out, static_cast<int>(t), n_heads, d, scale2, part, cnt,
                           static_cast<int>(per));
    }
    return hipGetLastError();
}

// 4-wave workgroups where their blocks of 128 queries are at most one per CU
// (twice the workgroups, each with about 0.6 of the time), where one such
// block holds all queries, or where 256-query blocks would be cut although
// the 128-query ones are at most two per CU: such calls take no workspace, and
// up to 64 dims two of them share a CU (t = 384, 150 x 64: 63 us one at a
// time, 44 in pairs).
bool half_blocks(int64_t t, int n_heads) {
    const int64_t items = n_heads * ((t + 127) / 128), slots = flux_slots();
    return t <= 128 || items <= slots || (items <= 2 * slots && n_heads * ((t + 255) / 256) > slots);
}

template <int DP>
hipError_t run_dp(const float* q, const float* k, const float* v, float* out, int64_t t, int n_heads, int d, float* part, uint32_t* cnt, hipStream_t s) {
    if (half_blocks(t, n_heads))
        return run<DP, 4>(q, k, v, out, t, n_heads, d, nullptr, nullptr, s);
    return run<DP, 8>(q, k, v, out, t, n_heads, d, part, cnt, s);
}

}  // namespace

size_t flux_attention_workspace(int64_t t, int n_heads, int head_dim) {
    const int64_t items = n_heads * ((t + 255) / 256);
    const int slots = flux_slots();
    if (items <= slots || half_blocks(t, n_heads)) return 0;
    return static_cast<size_t>(slots) * 2 * piece_floats(256, padded_dims(head_dim)) * sizeof(float);
}

hipError_t launch_flux_attention(const float* q, const float* k, const float* v, float* out, int64_t t, int n_heads,
                                 int head_dim, float* part, uint32_t* counters, hipStream_t s) {
    if (part && (!counters || static_cast<size_t>(flux_slots()) > kArrivalCounters)) return hipErrorInvalidValue;
    switch (padded_dims(head_dim)) {
        case 32: return run_dp<32>(q, k, v, out, t, n_heads, head_dim, part, counters, s);
        case 64: return run_dp<64>(q, k, v, out, t, n_heads, head_dim, part, counters, s);
        default: return run_dp<128>(q, k, v, out, t, n_heads, head_dim, part, counters, s);
    }
}

}  // namespace rt_hip
