// Fused paged encode: Hadamard-128 + norm + nearest centroid + pack + scatter
// into the paged slot layout (gfx950).
//
// Reference contract: cda_paged_encode_fused as bound by
// cda/kernels_cuda/wrappers.py:127-156; arithmetic of Compressor.encode
// (cda/algorithm/compression.py:287-335) and pack_4bit / pack_2bit
// (:163-179, :375-386).  The result is bit-identical to the reference's CPU
// path, which fixes three orders:
//
//  * rotation (compression.py:290-291): x_rot_j = fp16(acc_j) with acc_j the
//    fp32 fused-multiply-add chain over k = 0..127 in order,
//    acc = fma(x_k, H[k][j], acc), H[k][j] = (-1)^popcount(k & j) * h,
//    h = fp32(1/sqrt(128)) (the order of the MKL sgemm behind torch.matmul);
//  * norm (:328): eight lane sums a_l = sq_l + sq_{8+l} + ... + sq_{120+l}
//    with sq_j = fp32(x_j * x_j), then a_0 + ... + a_7 in order, a correctly
//    rounded fp32 square root, clamp_min(1e-12);
//  * x_unit = fp32(x_rot / norm), clamp to [-1, 1], then the bucketize +
//    neighbour compare of quantize_unit (:298-313) in fp32.
//
// Work layout.  The rotation runs on the fp32 matrix cores:
// v_mfma_f32_16x16x4_f32 adds its four products to the accumulator in ascending
// k, each with one rounding (checked bit for bit against the fmaf chain), so a
// sequence of them is exactly the reference's chain.  A operand: 16 output
// rows j of H, B operand: 16 vectors; lane (q4, r16) then holds outputs j = 16 *
// blk + 4 * q4 + i (i = 0..3) of vector r16 for each of the eight row blocks.
// Chains that agree in the low bits of j agree in their first steps:
// (-1)^popcount(k & j) depends only on the bits of j below the highest set bit
// of k, so for k < 16 * 2^t the blocks blk and blk + 2^t are equal.  One block
// runs k < 16, two 16 <= k < 32, four k < 64 and eight the rest: 172 MFMAs for
// 16 vectors instead of 256.
//
// What bounds it: 172 MFMAs of 32 cycles and about 900 other vector instructions
// per 16 vectors (fp16 round trip, norm, quantiser), 9100 cycles of a SIMD in
// all: no vector instruction of another wave issues while an fp32 MFMA runs.
// The vector form of the same chains (2731 fmas per lane, four lanes to a
// vector) has the same rate but longer waves: 8 heads, K and V, 1000 tokens
// 12.6 -> 9.2 us a call, 3000 20.8 -> 17.4, 8002 42.8 -> 41.8 (2-bit codes 40.7
// -> 37.4).
//
// Quantisation without a division.  For a sorted codebook the reference's
// index is monotone in u = RN32(x / n): it equals #{i in 1..L-1 : u >= th_i}
// where th_i is the smallest fp32 in (cb[i-1], cb[i]] for which
// |RN(cb[i] - u)| < |RN(u - cb[i-1])| (found once per block by bisection over
// the ordered fp32 bit patterns).  RN32(x / n) >= th holds exactly when
// x / n >= beta (th even) or x / n > beta (th odd), beta the midpoint of th
// and its fp32 predecessor; x / n >= beta <=> x >= n * beta, and n * beta
// (24 x 25 significant bits) is exact in float64.  So each vector gets L-1
// thresholds in the x domain (rounded up to fp32, where every fp16 x lives)
// and each element a four-step bisection of compares.  Non-finite norms
// (an fp16 overflow in x_rot, or NaN input) take the reference's formula
// with a true division.
#include "cda_common.h"

namespace cda {

namespace {

struct EncodeParams {
    const uint16_t *k;
    const uint16_t *v;
    int64_t k_stride;      // elements between tokens
    int64_t v_stride;
    const int32_t *slot_mapping;
    int64_t num_tokens;
    uint8_t *cache;
    int64_t num_slots;
    int64_t row_bytes;     // H_kv * slot_bytes
    int slot_bytes;
    int H_kv;
    const float *cb_k;
    const float *cb_v;
};

constexpr int kEncWaves = 4;          // waves 2q, 2q+1: K and V of item group q

// Ordered-integer image of an fp32 value (monotone in the value; -0 < +0).
__device__ __forceinline__ uint32_t f2key(float f) {
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key2f(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// The neighbour compare of quantize_unit for u in bucket i (lo < u <= hi):
// true picks the upper centroid.
__device__ __forceinline__ bool pick_upper(float u, float lo, float hi) {
    return fabsf(__fsub_rn(hi, u)) < fabsf(__fsub_rn(u, lo));
}

// Decision threshold i (1 <= i < L) of a sorted codebook in the u domain,
// expressed as (beta, strict): clamp(u) selects at least level i exactly when
// u >= beta (u > beta when strict), for every u = RN32(v) with v real.
// Thresholds at or below -1 always hold after the clamp (beta = -inf);
// thresholds above 1 never do (beta = +inf).
//
// kSearch lanes (j = 0..7, aligned in the wave) search one threshold together:
// each tests one of eight points, which cuts the interval of ordered bit patterns
// by eight a turn, 11 turns where one lane's bisection took 31 (2.5 us before the
// first vector could be quantised).  Every lane of the wave has to call; those
// without a threshold pass live = false.
constexpr int kSearch = 64 * kEncWaves / 32;          // a block's lanes, 16 thresholds a role
static_assert(kSearch == 8, "lanes per threshold");
__device__ void codebook_threshold(const float *cb, int i, int j, bool live, double *beta,
                                   int *strict) {
    constexpr int K = kSearch;
    const float lo = live ? cb[i - 1] : 0.0f, hi = live ? cb[i] : 0.0f;
    uint32_t a = f2key(lo) + 1u, b = f2key(hi);
    // The answer lies in [a, b].  The largest point tested is never below b,
    // which counts as an upper pick without a test.
    while (__builtin_amdgcn_ballot_w64(live && a < b)) {
        const bool open = live && a < b;
        const uint32_t step = ((b - a) / K) + 1u;
        const uint64_t end = (uint64_t)a + (uint64_t)(j + 1) * step - 1u;   // of part j
        const bool lower = open && end < b && !pick_upper(key2f((uint32_t)end), lo, hi);
        const uint64_t m = __builtin_amdgcn_ballot_w64(lower) >> ((threadIdx.x & 63) & ~(K - 1));
        const uint32_t below = (uint32_t)__popcll(m & ((1ull << K) - 1));   // parts wholly below
        if (open) {
            const uint64_t last = (uint64_t)a + (uint64_t)(below + 1) * step - 1u;
            b = last < b ? (uint32_t)last : b;
            a += below * step;
        }
    }
    if (!live || j != 0) return;
    // a: the smallest fp32 above lo that selects i (an empty bucket, lo == hi,
    // gives nextup(hi): only values above hi select it, as in the reference).
    const float th = key2f(a);
    if (th <= -1.0f) { *beta = -__builtin_inf(); *strict = 0; return; }
    if (th > 1.0f) { *beta = __builtin_inf(); *strict = 0; return; }
    uint32_t pk = a - 1u;
    if (__float_as_uint(key2f(pk)) == 0x80000000u && __float_as_uint(th) == 0u) pk -= 1u;  // pred(+0)
    *beta = ((double)key2f(pk) + (double)th) * 0.5;
    *strict = (int)(__float_as_uint(th) & 1u);
}

// Both codebooks' thresholds, by the whole block.
template <int LK, int LV>
__device__ __forceinline__ void codebook_thresholds(const EncodeParams &p, double (&beta)[2][16],
                                                    int (&strict)[2][16], float (&s_cb)[2][16]) {
    constexpr int K = kSearch;
    const int at = (int)threadIdx.x / K, r = at >> 4, i = at & 15;
    const float *cb = r ? p.cb_v : p.cb_k;
    const int j = (int)threadIdx.x & (K - 1);
    const bool in = i < (r ? LV : LK);
    if (in && j == 0) s_cb[r][i] = cb[i];
    codebook_threshold(cb, i, j, in && i > 0, &beta[r][i], &strict[r][i]);
}

// Smallest fp32 >= t (t finite or infinite).
__device__ __forceinline__ float round_up_f32(double t) {
    float f = (float)t;
    if ((double)f < t) f = __uint_as_float(__float_as_uint(f) + (f >= 0.0f ? 1u : 0xFFFFFFFFu));
    return f;
}

// Next float64 above t (t finite, non-zero).
__device__ __forceinline__ double next_up(double t) {
    const long long b = __double_as_longlong(t);
    return __longlong_as_double(t > 0.0 ? b + 1 : b - 1);
}

// The reference's quantize_unit on one fp32 value (compression.py:298-313):
// only used for vectors with a non-finite norm.
template <int L>
__device__ uint32_t quantize_ref(float u, const float *cb) {
    int upper = 0;
#pragma unroll
    for (int i = 0; i < L; ++i) upper += !(cb[i] >= u) ? 1 : 0;
    upper = upper > L - 1 ? L - 1 : upper;
    const int lower = upper - 1 < 0 ? 0 : upper - 1;
    const float du = fabsf(__fsub_rn(cb[upper], u));
    const float dl = fabsf(__fsub_rn(u, cb[lower]));
    return (uint32_t)(du < dl ? upper : lower);
}

// L - 1 - #{i : x >= thr[i]} for the sorted thresholds thr[1..L-1] of this
// vector, by bisection, for all of a lane's elements level by level (their
// reads of one level are in flight together).  A level appends the sign of x -
// threshold: one subtraction and one v_alignbit, where a compare into VCC and
// its use need two wait states between them.  The thresholds are stored by
// level in the order of those (inverted) bits, t[2^level + c], a zero as -0 so
// that x = -0 is not below it.
template <int L, int N>
__device__ __forceinline__ void count_below_lds(const float (&x)[N], const float *t,
                                                uint32_t (&c)[N]) {
    static_assert(L == 4 || L == 16, "4 or 16 levels");
    const float tmid = t[1];
#pragma unroll
    for (int e = 0; e < N; ++e) c[e] = __float_as_uint(__fsub_rn(x[e], tmid)) >> 31;
#pragma unroll
    for (int n = 2; n < L; n *= 2) {
        float th[N];
#pragma unroll
        for (int e = 0; e < N; ++e) th[e] = t[n + c[e]];
#pragma unroll
        for (int e = 0; e < N; ++e)
            c[e] = __builtin_amdgcn_alignbit(c[e], __float_as_uint(__fsub_rn(x[e], th[e])), 31);
    }
}

// Position of threshold i (1 <= i < L) in that order.
template <int L>
__device__ __forceinline__ int thr_pos(int i) {
    const int z = __builtin_ctz((unsigned)i);              // level = log2(L / 2) - z
    const int n = (L / 2) >> z;
    return n + ((n - 1) ^ (i >> (z + 1)));
}

typedef float floatx4 __attribute__((ext_vector_type(4)));

// The pair (a, b) after rows 2, 3 of a (16 lanes each) trade places with rows
// 0, 1 of b (swap32), or row 1 of a with row 0 of b and row 3 with row 2
// (swap16).
__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// 4 x 4 transpose over the four 16-lane rows: d[p] of row q <-> d[q] of row p.
__device__ __forceinline__ void transpose_rows(uint32_t (&d)[4]) {
    swap32(d[0], d[2]);
    swap32(d[1], d[3]);
    swap16(d[0], d[1]);
    swap16(d[2], d[3]);
}

constexpr int kThrPitch = 17;         // thresholds of one vector in LDS (bank spread)

template <int LK, int LV>
__global__ void __launch_bounds__(64 * kEncWaves)
paged_encode_kernel(EncodeParams p) {
    // Slot: [K codes KBK | V codes KBV | K norm | V norm | pad].
    constexpr int KBK = kD * (LK == 16 ? 4 : 2) / 8;
    constexpr int KBV = kD * (LV == 16 ? 4 : 2) / 8;
    __shared__ double s_beta[2][16];
    __shared__ int s_strict[2][16];
    __shared__ float s_cb[2][16];
    __shared__ float s_thr[kEncWaves][16 * kThrPitch];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int role = wave & 1;                        // wave-uniform: 0 = K, 1 = V
    const int r16 = lane & 15, q4 = lane >> 4;

    // (token, head) item of this lane's vector; fewer than 2^31 items (host check).
    const uint32_t items = (uint32_t)(p.num_tokens * p.H_kv);
    const uint32_t item = (blockIdx.x * (uint32_t)(kEncWaves / 2) + (uint32_t)(wave >> 1)) * 16u +
                          (uint32_t)r16;
    const bool valid = item < items;
    const uint32_t t32 = valid ? item / (uint32_t)p.H_kv : 0u;
    const int h = valid ? (int)(item - t32 * (uint32_t)p.H_kv) : 0;
    const int64_t t = t32;

    // ---- load the vector: elements 32g + 8 * q4 .. + 7 of it per lane (lanes
    // past the last item read the first and store nothing).  The loads go out
    // before the codebook's thresholds are worked out.
    uint4 xw[4];
    {
        const uint16_t *src = role == 0 ? p.k + t * p.k_stride + (int64_t)h * kD
                                        : p.v + t * p.v_stride + (int64_t)h * kD;
#pragma unroll
        for (int g = 0; g < 4; ++g)
            xw[g] = reinterpret_cast<const uint4 *>(src)[4 * g + q4];
    }
    const int64_t slot_of_t = p.slot_mapping[t];
    const int64_t slot = valid ? slot_of_t : -1;

    codebook_thresholds<LK, LV>(p, s_beta, s_strict, s_cb);
    __syncthreads();

    // ---- rotation ------------------------------------------------------------
    // The four lanes of a vector exchange their elements so that lane q4 gets
    // x[4m + q4] for every m (the k slot it feeds), widened to fp32: pairs
    // (0, 1) / (2, 3) of a block of four change rows in the first swap, single
    // elements in the second.
    float x[kD / 4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const uint32_t w[4] = {xw[g].x, xw[g].y, xw[g].z, xw[g].w};
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            uint32_t a = w[2 * e], b = w[2 * e + 1];
            swap32(a, b);
            uint32_t lo = __builtin_amdgcn_perm(b, a, 0x05040100u);
            uint32_t hi = __builtin_amdgcn_perm(b, a, 0x07060302u);
            swap16(lo, hi);
            x[8 * g + 0 + e] = h2f((uint16_t)(lo & 0xFFFFu));
            x[8 * g + 4 + e] = h2f((uint16_t)(lo >> 16));
            x[8 * g + 2 + e] = h2f((uint16_t)(hi & 0xFFFFu));
            x[8 * g + 6 + e] = h2f((uint16_t)(hi >> 16));
        }
    }
    // H[16 * blk + r16][4m + q4]: the sign from bits 0-3 of j and k per lane (hp
    // and its negative hn, by m & 3), that from bits 4-6 below.
    const float hval = __int_as_float(0x3db504f3);    // fp32(1/sqrt(128))
    float hp[4], hn[4];
#pragma unroll
    for (int mm = 0; mm < 4; ++mm) {
        hp[mm] = (__popc((uint32_t)((4 * mm + q4) & r16)) & 1) ? -hval : hval;
        hn[mm] = -hp[mm];
    }
    floatx4 ch[8];
    ch[0] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < 4; ++m)
        ch[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(hp[m], x[m], ch[0], 0, 0, 0);
#pragma unroll
    for (int half = 1; half < 8; half *= 2) {         // blocks so far
#pragma unroll
        for (int blk = 0; blk < half; ++blk) ch[blk + half] = ch[blk];
#pragma unroll
        for (int m = 4 * half; m < 8 * half; ++m)
#pragma unroll
            for (int blk = 0; blk < 2 * half; ++blk) {
                const bool neg = (__builtin_popcount((unsigned)((m >> 2) & blk)) & 1) != 0;
                ch[blk] = __builtin_amdgcn_mfma_f32_16x16x4f32(neg ? hn[m & 3] : hp[m & 3], x[m],
                                                               ch[blk], 0, 0, 0);
            }
    }

    // ---- fp16 rounding, squares, norm (reference order) ---------------------
    // The reference rounds its fp32 matmul output to the input dtype, squares
    // it and adds eight lane sums a_l = sq_l + sq_{8 + l} + ..., then a_0 + ... + a_7.
    float xr[32];                                     // element i of block blk at 4 * blk + i
    uint32_t sq[32];
#pragma unroll
    for (int e = 0; e < 32; ++e) {
        xr[e] = h2f(f2h_after_f32(ch[e >> 2][e & 3]));
        sq[e] = __float_as_uint(__fmul_rn(xr[e], xr[e]));
    }
    // Square j = 8c + l is in lane row (l >> 2) + 2 * (c & 1), register i = l & 3 of
    // block c >> 1, so the sum over c of one l alternates between two rows.  A
    // swap brings both parts to one lane: rows 0, 1 sum l with i = 0, 1 and
    // rows 2, 3 those with i = 2, 3.
    float a01[2];
#pragma unroll
    for (int blk = 0; blk < 8; ++blk)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            uint32_t &a = sq[4 * blk + i], &b = sq[4 * blk + i + 2];
            swap32(a, b);                             // now c = 2 * blk, then 2 * blk + 1
            a01[i] = blk ? __fadd_rn(a01[i], __uint_as_float(a)) : __uint_as_float(a);
            a01[i] = __fadd_rn(a01[i], __uint_as_float(b));
        }
    // a_0 .. a_7 of the vector in every lane of it: first, the lane rows' pairs.
    float ss;
    {
        uint32_t lo[2], hi[2];                         // rows 0, 1 and rows 2, 3 of a01[i]
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            lo[i] = hi[i] = __float_as_uint(a01[i]);
            swap32(lo[i], hi[i]);
        }
        uint32_t e[4] = {lo[0], lo[1], hi[0], hi[1]}, o[4] = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
        for (int l = 0; l < 4; ++l) swap16(e[l], o[l]);
        // Rows 0, 2, 1, 3 hold l = 0-1, 2-3, 4-5, 6-7.
        ss = __uint_as_float(e[0]);
#pragma unroll
        for (int l = 1; l < 4; ++l) ss = __fadd_rn(ss, __uint_as_float(e[l]));
#pragma unroll
        for (int l = 0; l < 4; ++l) ss = __fadd_rn(ss, __uint_as_float(o[l]));
    }
    float n = sqrt_f64_to_f32_rn((double)ss);
    n = (n < 1e-12f) ? 1e-12f : n;                    // clamp_min(1e-12); NaN passes

    // ---- thresholds, quantisation, packing and the store, for this role's
    // codebook (K: LK levels, V: LV levels; wave-uniform branch).
    auto finish = [&](auto levels) CDA_INLINE {
        constexpr int L = decltype(levels)::value;
        // ---- per-vector thresholds in the x domain --------------------------
        const bool finite_n = fabsf(n) < __builtin_inff();
        float *thr = s_thr[wave] + r16 * kThrPitch;
#pragma unroll
        for (int i0 = 1; i0 < L; i0 += 4) {
            const int i = i0 + q4;
            if (i < L) {
                const double beta = s_beta[role][i];
                double tt = (double)n * beta;         // exact: 24 x 25 significant bits
                if (s_strict[role][i] && finite_n) tt = next_up(tt);
                const float th = round_up_f32(tt);
                thr[thr_pos<L>(i)] = th == 0.0f ? -0.0f : th;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

        // ---- quantise.  A non-finite norm has garbage thresholds (the
        // bisection's indices stay in range); its lanes then take the
        // reference's formula.
        uint32_t c[32];
        count_below_lds<L>(xr, thr, c);
        if (__builtin_expect(!finite_n, 0)) {
#pragma unroll
            for (int e = 0; e < 32; ++e) {
                float u = __fdiv_rn(xr[e], n);
                u = u < -1.0f ? -1.0f : (u > 1.0f ? 1.0f : u);
                c[e] = (uint32_t)(L - 1) - quantize_ref<L>(u, s_cb[role]);
            }
        }
        // ---- pack: four consecutive codes of a block make two bytes (4-bit
        // codes) or one (2-bit), the first in the high bits (inverted up to
        // the store).
        uint32_t part[8];
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint32_t *cc = c + 4 * b;
            part[b] = L == 16 ? (cc[0] << 4) | cc[1] | (cc[2] << 12) | (cc[3] << 8)
                              : (cc[0] << 6) | (cc[1] << 4) | (cc[2] << 2) | cc[3];
        }
        // Lane row q takes blocks 2q and 2q + 1 of all four rows: dims [32q, +32).
        uint32_t d[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) d[q] = part[2 * q] | part[2 * q + 1] << 16;
        transpose_rows(d);
        if (slot < 0 || slot >= p.num_slots) return;  // also the lanes past the last item
        uint8_t *dst = p.cache + slot * p.row_bytes + (int64_t)h * p.slot_bytes;
        uint32_t *cw = reinterpret_cast<uint32_t *>(dst + (role ? KBK : 0)) + (L == 16 ? 4 : 2) * q4;
        if constexpr (L == 16) {
            cw[0] = ~__builtin_amdgcn_perm(d[1], d[0], 0x05040100u);
            cw[1] = ~__builtin_amdgcn_perm(d[3], d[2], 0x05040100u);
            cw[2] = ~__builtin_amdgcn_perm(d[1], d[0], 0x07060302u);
            cw[3] = ~__builtin_amdgcn_perm(d[3], d[2], 0x07060302u);
        } else {
            cw[0] = ~((d[0] & 0xFFu) | (d[1] & 0xFFu) << 8 | (d[2] & 0xFFu) << 16 | d[3] << 24);
            cw[1] = ~(d[0] >> 16 | d[1] >> 16 << 8 | (d[2] & 0xFF0000u) | d[3] >> 16 << 24);
        }
        if (q4 == 0) *reinterpret_cast<float *>(dst + KBK + KBV + 4 * role) = n;
    };
    if (role == 0) finish(std::integral_constant<int, LK>{});
    else finish(std::integral_constant<int, LV>{});
}

// Small batches: 16 lanes share a vector, and lane r of them runs the chains of
// outputs r + 16m as a tree of fp32 fmas (688 a lane).  That ends sooner than the
// 172 MFMAs of a wave above while a SIMD has only a wave or two to run.
constexpr int kSmallLanes = 16;               // per vector
constexpr int kSmallVecs = 64 / kSmallLanes;  // vectors per wave
constexpr int kSmallPitch = kD + kSmallLanes; // floats per vector row in LDS (bank spread)

template <int LK, int LV>
__global__ void __launch_bounds__(64 * kEncWaves)
paged_encode_small_kernel(EncodeParams p) {
    constexpr int P = kSmallLanes, V = kSmallVecs, M = kD / P;   // M: outputs per lane
    // Slot: [K codes KBK | V codes KBV | K norm | V norm | pad].
    constexpr int KBK = kD * (LK == 16 ? 4 : 2) / 8;
    constexpr int KBV = kD * (LV == 16 ? 4 : 2) / 8;
    __shared__ double s_beta[2][16];
    __shared__ int s_strict[2][16];
    __shared__ float s_cb[2][16];
    // Per wave: V rows of sq / idx, then V x 16 thresholds, V x 8 lane sums.
    __shared__ __align__(16) float s_w[kEncWaves][V * (kSmallPitch + kThrPitch + 8)];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int role = wave & 1;                        // wave-uniform: 0 = K, 1 = V
    const int g = lane / P, r = lane % P;
    float *sq_row = s_w[wave] + g * kSmallPitch;      // this vector's 128 floats
    float *thr = s_w[wave] + V * kSmallPitch + g * kThrPitch;
    float *lsum = s_w[wave] + V * (kSmallPitch + kThrPitch) + g * 8;

    // (token, head) item of this lane group; fewer than 2^31 items (host check).
    const uint32_t items = (uint32_t)(p.num_tokens * p.H_kv);
    const uint32_t item = blockIdx.x * (uint32_t)(V * kEncWaves / 2) +
                          (uint32_t)(wave >> 1) * (uint32_t)V + (uint32_t)g;
    const bool valid = item < items;
    const uint32_t t32 = valid ? item / (uint32_t)p.H_kv : 0u;
    const int h = valid ? (int)(item - t32 * (uint32_t)p.H_kv) : 0;
    const int64_t t = t32;

    // ---- load the vector (lanes past the last item read the first and store
    // nothing; the 16 lanes of a vector read the same 256 B) ----
    // Kept as packed fp16 pairs; each x_k is widened to fp32 once, where the
    // chains use it (xf below).
    uint32_t xw[kD / 2];
    {
        const uint16_t *src = role == 0 ? p.k + t * p.k_stride + (int64_t)h * kD
                                        : p.v + t * p.v_stride + (int64_t)h * kD;
        const uint4 *s4 = reinterpret_cast<const uint4 *>(src);
#pragma unroll
        for (int q = 0; q < kD / 8; ++q) {
            const uint4 w = s4[q];
            xw[4 * q + 0] = w.x;
            xw[4 * q + 1] = w.y;
            xw[4 * q + 2] = w.z;
            xw[4 * q + 3] = w.w;
        }
    }
    const int64_t slot_of_t = p.slot_mapping[t];
    // The loads above go out before the codebook's thresholds are worked out.
    codebook_thresholds<LK, LV>(p, s_beta, s_strict, s_cb);
    __syncthreads();
    // x_k in fp32 (exact).  The empty asm makes the widened value opaque, so
    // the compiler cannot fold the conversion into every fma that uses it
    // (v_fma_mix_f32, about twice the issue cost of v_fma_f32 on gfx950).
    auto xf = [&](int k) CDA_INLINE -> float {
        float v = h2f((uint16_t)((k & 1) ? (xw[k >> 1] >> 16) : (xw[k >> 1] & 0xFFFFu)));
        asm volatile("" : "+v"(v));
        return v;
    };

    // ---- rotation: the fma chains as a tree ---------------------------------
    const float hval = __int_as_float(0x3db504f3);    // fp32(1/sqrt(128))
    float hs[P];                                      // s(k & r) * h for k mod P
#pragma unroll
    for (int q = 0; q < P; ++q) hs[q] = (__popc((uint32_t)(q & r)) & 1) ? -hval : hval;
    float ch[M];
    {
        float c = 0.0f;
#pragma unroll
        for (int k = 0; k < P; ++k) c = fmaf(xf(k), hs[k], c);
        ch[0] = c;
    }
#pragma unroll
    for (int lvl = 0; (P << lvl) < kD; ++lvl) {
        const int cnt = 1 << lvl;                     // chains so far (m mod cnt)
        const int k0 = P << lvl;                      // steps k0 .. 2 k0 - 1
#pragma unroll
        for (int m = 0; m < cnt; ++m) ch[m + cnt] = ch[m];
#pragma unroll
        for (int k = k0; k < 2 * k0; ++k) {
            const float xk = xf(k);
#pragma unroll
            for (int m = 0; m < 2 * cnt; ++m) {
                const bool neg = (__builtin_popcount((unsigned)(k & (P * m))) & 1) != 0;
                ch[m] = fmaf(xk, neg ? -hs[k % P] : hs[k % P], ch[m]);
            }
        }
    }

    // ---- fp16 rounding, squares, norm (reference order) ---------------------
    float xr[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        // The fp32 chain value is rounded on its own, then to fp16 (the
        // reference rounds its fp32 matmul output to the input dtype); the
        // empty asm keeps the compiler from fusing the last fma with the fp16
        // conversion into one rounding (v_fma_mixlo_f16).
        asm volatile("" : "+v"(ch[m]));
        xr[m] = __half2float(__float2half_rn(ch[m]));
        sq_row[r + P * m] = __fmul_rn(xr[m], xr[m]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (r < 8) {
        float a = sq_row[r];
#pragma unroll
        for (int c = 1; c < kD / 8; ++c) a = __fadd_rn(a, sq_row[8 * c + r]);
        lsum[r] = a;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float ss = lsum[0];
#pragma unroll
    for (int l = 1; l < 8; ++l) ss = __fadd_rn(ss, lsum[l]);
    float n = sqrt_f64_to_f32_rn((double)ss);
    n = (n < 1e-12f) ? 1e-12f : n;                    // clamp_min(1e-12); NaN passes

    // ---- thresholds, quantisation, packing and the store, for this role's
    // codebook (K: LK levels, V: LV levels; wave-uniform branch).
    auto finish = [&](auto levels) CDA_INLINE {
        constexpr int L = decltype(levels)::value;
        // ---- per-vector thresholds in the x domain ------------------------------
        const bool finite_n = fabsf(n) < __builtin_inff();
        if (r > 0 && r < L) {                             // lane r: threshold r
            const double beta = s_beta[role][r];
            double tt = (double)n * beta;                 // exact: 24 x 25 significant bits
            if (s_strict[role][r] && finite_n) tt = next_up(tt);
            const float th = round_up_f32(tt);
            thr[thr_pos<L>(r)] = th == 0.0f ? -0.0f : th;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

        // ---- quantise; codes go through LDS (the sq row is free again) ----------
        uint8_t *idx_row = reinterpret_cast<uint8_t *>(sq_row);
        uint32_t code[M];
        count_below_lds<L>(xr, thr, code);
        if (__builtin_expect(!finite_n, 0)) {
    #pragma unroll
            for (int m = 0; m < M; ++m) {
                float u = __fdiv_rn(xr[m], n);
                u = u < -1.0f ? -1.0f : (u > 1.0f ? 1.0f : u);
                code[m] = (uint32_t)(L - 1) - quantize_ref<L>(u, s_cb[role]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();                  // lane sums read before the row is reused
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    #pragma unroll
        for (int m = 0; m < M; ++m) idx_row[r + P * m] = (uint8_t)((L - 1) - code[m]);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

        if (!valid) return;
        const int64_t slot = slot_of_t;
        if (slot < 0 || slot >= p.num_slots) return;
        uint8_t *dst = p.cache + slot * p.row_bytes + (int64_t)h * p.slot_bytes;
        uint8_t *codes = dst + (role ? KBK : 0);
        // Lane r packs the codes of dims [8r, 8r + 8): four bytes of 4-bit codes,
        // two of 2-bit codes.
        const uint2 e = *reinterpret_cast<const uint2 *>(idx_row + 8 * r);
        auto code_at = [&](int i) CDA_INLINE { return ((i < 4 ? e.x : e.y) >> (8 * (i & 3))) & 0xFFu; };
        uint32_t packed = 0;
    #pragma unroll
        for (int i = 0; i < 8; ++i)
            packed |= L == 16 ? code_at(i) << (8 * (i / 2) + 4 * (1 - i % 2))
                              : code_at(i) << (8 * (i / 4) + 2 * (3 - i % 4));
        if constexpr (L == 16)
            reinterpret_cast<uint32_t *>(codes)[r] = packed;
        else
            reinterpret_cast<uint16_t *>(codes)[r] = (uint16_t)packed;
        if (r == 0) *reinterpret_cast<float *>(dst + KBK + KBV + 4 * role) = n;
    };
    if (role == 0) finish(std::integral_constant<int, LK>{});
    else finish(std::integral_constant<int, LV>{});
}

// Items up to which the 16-lane form is taken: two of its waves per SIMD.
// Measured us a call, 16-lane / MFMA form, 8 heads: 32 tokens 6.7 / 9.0, 256
// 6.8 / 9.0, 500 8.4 / 9.1, 1000 11.7 / 9.2, 1500 16.5 / 13.2.
constexpr int64_t kSmallItems = 4096;

template <int LK, int LV>
void launch_encode(const EncodeParams &p, int64_t items, hipStream_t st) {
    if (items <= kSmallItems) {
        constexpr int per_block = kSmallVecs * kEncWaves / 2;
        paged_encode_small_kernel<LK, LV>
            <<<dim3((unsigned)((items + per_block - 1) / per_block)), 64 * kEncWaves, 0, st>>>(p);
    } else {
        constexpr int per_block = 16 * kEncWaves / 2;
        paged_encode_kernel<LK, LV>
            <<<dim3((unsigned)((items + per_block - 1) / per_block)), 64 * kEncWaves, 0, st>>>(p);
    }
}

}  // namespace

}  // namespace cda

using namespace cda;

namespace cda {
namespace {
int encode_impl(const void *k, const void *v, int64_t k_stride, int64_t v_stride,
                const int32_t *slot_mapping, int64_t num_tokens, void *flat_cache,
                int64_t num_slots, int slot_bytes, int H_kv, const float *cb_k, const float *cb_v,
                int levels_k, int levels_v, void *stream, const char *fn) {
    const std::string f(fn);
    CDA_REQUIRE(num_tokens >= 0, f + ": num_tokens must be >= 0");
    if (num_tokens == 0) return CDA_OK;
    CDA_REQUIRE(k && v && slot_mapping && flat_cache && cb_k && cb_v, f + ": null pointer argument");
    CDA_REQUIRE(H_kv > 0 && num_slots > 0, f + ": H_kv and num_slots must be > 0");
    const int kbk = kD * (levels_k == 16 ? 4 : 2) / 8;
    const int kbv = kD * (levels_v == 16 ? 4 : 2) / 8;
    CDA_REQUIRE(slot_bytes >= kbk + kbv + 8, f + ": slot_bytes too small for the layout");
    CDA_REQUIRE(k_stride >= (int64_t)H_kv * kD && v_stride >= (int64_t)H_kv * kD,
                f + ": token stride smaller than H_kv * 128");
    CDA_REQUIRE(((uintptr_t)k & 3) == 0 && ((uintptr_t)v & 3) == 0 && slot_bytes % 4 == 0 &&
                    ((uintptr_t)flat_cache & 3) == 0,
                f + ": k, v, cache must be 4-byte aligned");
    EncodeParams p;
    p.k = static_cast<const uint16_t *>(k);
    p.v = static_cast<const uint16_t *>(v);
    p.k_stride = k_stride;
    p.v_stride = v_stride;
    p.slot_mapping = slot_mapping;
    p.num_tokens = num_tokens;
    p.cache = static_cast<uint8_t *>(flat_cache);
    p.num_slots = num_slots;
    p.row_bytes = (int64_t)H_kv * slot_bytes;
    p.slot_bytes = slot_bytes;
    p.H_kv = H_kv;
    p.cb_k = cb_k;
    p.cb_v = cb_v;
    const int64_t items = num_tokens * H_kv;
    CDA_REQUIRE(items < ((int64_t)1 << 31), f + ": too many tokens x heads");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (levels_k == 16 && levels_v == 16)
        launch_encode<16, 16>(p, items, st);
    else if (levels_k == 4 && levels_v == 4)
        launch_encode<4, 4>(p, items, st);
    else
        launch_encode<16, 4>(p, items, st);
    CDA_LAUNCH_CHECK(f + ": paged_encode_kernel");
    return CDA_OK;
}
}  // namespace
}  // namespace cda

extern "C" int cda_paged_encode_fused(const void *k, const void *v, int64_t k_stride,
                                      int64_t v_stride, const int32_t *slot_mapping,
                                      int64_t num_tokens, void *flat_cache, int64_t num_slots,
                                      int slot_bytes, int H_kv, const float *cb_k,
                                      const float *cb_v, int levels, void *stream) {
    CDA_REQUIRE(levels == 16 || levels == 4, "cda_paged_encode_fused: levels must be 16 or 4");
    return encode_impl(k, v, k_stride, v_stride, slot_mapping, num_tokens, flat_cache, num_slots,
                       slot_bytes, H_kv, cb_k, cb_v, levels, levels, stream,
                       "cda_paged_encode_fused");
}

extern "C" int cda_paged_encode_fused_k4v2(const void *k, const void *v, int64_t k_stride,
                                           int64_t v_stride, const int32_t *slot_mapping,
                                           int64_t num_tokens, void *flat_cache,
                                           int64_t num_slots, int slot_bytes, int H_kv,
                                           const float *cb_k, const float *cb_v, void *stream) {
    return encode_impl(k, v, k_stride, v_stride, slot_mapping, num_tokens, flat_cache, num_slots,
                       slot_bytes, H_kv, cb_k, cb_v, 16, 4, stream, "cda_paged_encode_fused_k4v2");
}
