// Packed decode attention for many query rows per kv head (several new tokens, wide GQA groups),
// matrix cores: the layout of decode_mfma.hip (head_dim 128, page = Key group = 128 tokens, one
// Value group, int2 Values), 2-byte rows of one dtype.
//
// Reference: src/logitfill/packed/reference.py:18-56 (the right-aligned causal mask over the new
// tokens; the reference sends several new tokens to its dense path, reference.py:62).
//
// decode_mfma.hip serves 8 rows per workgroup and unpacks every page again for each 8.  Here one
// workgroup of 8 waves per (split item, kv head, tile of 16 * WR rows) unpacks a page once into LDS
// as matrix operands -- the Key codes as fp16 integers and the fp16 tier's values as stored
// [token][slot], the Value codes as fp16 (code - 1.5) [32 tokens][channel][token], transposed -- and
// every wave multiplies them with its own 16 rows: WR = 8 row groups, or 4 of them with WT = 2 waves
// sharing a row group's tokens.  A page's bytes arrive by LDS-DMA, one page ahead of the one being
// computed.
//
// Scores S^T = Codes . Qs^T, Qs = q * (scale * scaling * log2 e) as fp16 hi + lo made in registers
// from the wave's q (kept packed there).  Qs carries a power of two per page that brings the largest
// |q| times the largest scale just below fp16's largest number, so the lo parts stay clear of its
// smallest (unscaled, an int8 channel's lo lost up to 8e-6 of a score); the sums are divided by it in
// fp32.  It is never below 1, so Qs holds what decode_mfma.hip's unscaled Qs holds: |q| * scale *
// scaling * log2 e below 65 504, and no bit fewer.  Values O^T = (code - 1.5)^T . P'^T, P' = p * vscale
// as fp16 hi + lo, in decode_mfma.hip's range.  A query row is a lane (lane % 16) throughout, so the running max, its rescale and the sums
// stay in the lane.  The codes enter as they are (decode_mfma.hip adds an offset to each and takes it
// out of the sums again), so the sums carry no cancelling part.  The tail page and the new tokens
// follow as dense chunks of 128 tokens through the same buffers.
//
// What bounds it: the LDS reads of the operands (12 of 1 KB per K-step and wave) and the VALU work
// beside them (Qs 6.5 operations per slot and row, softmax and P' split about 14 per score).  Counters of 512
// new tokens x 28 q / 4 kv heads over 16 384 tokens (224 workgroups of 64 pages, one per CU): a wave runs
// 77 200 VALU operations, 11 400 products and 10 000 LDS instructions in 1.0 M cycles; over the chip the
// VALU is 52 % and the matrix cores 30 % busy, and a cycle of LDS activity comes with 2.4 of bank conflicts.
// The call takes 975 us a layer with decode_mfma.hip's 448 tiles of 8 rows, here 473 (470 before the factor
// of Qs was the page's own).  Against float64 (float32 output) 0.2-1.1e-6, decode_mfma.hip 1-6e-5.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "decode_common.hpp"

namespace lf {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kD = 128, kPage = 128;
constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kMaxSteps = 10;  // K-steps of 32 slots a wave keeps its q for
constexpr int kMaxDma = 4;     // 1 KB DMA instructions of a page per wave
constexpr int kVtBytes = kPage * kD * 2;
constexpr int kDenseStride = 2 * kD + 16;  // bytes of a token's row of the dense Key chunk

struct RowsLayout {
    int steps;       // K-steps, integer tiers then fp16
    int nb_int, nb;  // 8-slot blocks of the integer tiers, of all
    int step1, step2, step3;  // first step of tiers 1, 2, 3
    int end[8];      // ends of a page's regions in 16-byte chunks: the Key tiers' rows, Value codes, scales,
                     // mins, the k_sm_page block
    int stride;      // bytes of a token's row in the Key operand buffer (16 more than its blocks)
    int off_v, off_s, off_raw, raw_bytes, lds_bytes;  // two raw pages at off_raw
};

struct RowsParams {
    DecodeParams p;
    RowsLayout y;
};

__device__ __forceinline__ uint32_t fresh(uint32_t x) {
    asm volatile("" : "+v"(x));
    return x;
}
__device__ __forceinline__ half8 as_half8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(half8, u32x4{a, b, c, d});
}
__device__ __forceinline__ uint32_t pack_half(float a, float b) {
    return __builtin_bit_cast(uint32_t, half2v{static_cast<_Float16>(a), static_cast<_Float16>(b)});
}

// Two 2-bit codes in bits 8-9 and 24-25 of s as fp16 (the high byte from a table; the low one is 0).
__device__ __forceinline__ uint32_t code_pair(uint32_t s, uint32_t table, uint32_t mask, uint32_t zero) {
    return __builtin_amdgcn_perm(0u, table, (s & mask) | zero);
}

// 8 floats as fp16 hi + lo.  x is pinned: the compiler may otherwise form hi from the product behind
// x in one rounding and the hi that lo completes from x in two, which differ by a unit of hi now and
// then (rows off by 1e-3).
struct Split2 {
    half8 hi, lo;
};
__device__ __forceinline__ Split2 split2(const float (&x)[8]) {
    Split2 r;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float v = x[e];
        asm("" : "+v"(v));
        const _Float16 h = static_cast<_Float16>(v);
        r.hi[e] = h;
        r.lo[e] = static_cast<_Float16>(v - static_cast<float>(h));
    }
    return r;
}

// The largest of x over the wave.
template <int Ctrl>
__device__ __forceinline__ float dpp_max(float x) {
    const int xi = __builtin_bit_cast(int, x);
    return fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(xi, xi, Ctrl, 0xf, 0xf, false)));
}
__device__ __forceinline__ float wave_top(float x) {
    x = dpp_max<0xB1>(x);   // lanes ^ 1
    x = dpp_max<0x4E>(x);   // ^ 2
    x = dpp_max<0x141>(x);  // half rows mirrored
    x = dpp_max<0x140>(x);  // rows mirrored
    return rows_max(x);
}
// Larger 16-bit halves of two words of them (as unsigned numbers).
__device__ __forceinline__ uint32_t pair_max(uint32_t a, uint32_t b) {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

// Exponent of a page's factor on Qs: brings ``top`` (kTopMargin times a bound of |Qs|) into [2^15, 2^16),
// the bound itself then below 65 504; none below 1, and none past 2^24 (tiny or no q).
constexpr float kTopMargin = 1.001f;
__device__ __forceinline__ int qs_exponent(float top) {
    return min(max(142 - static_cast<int>(__float_as_uint(top) >> 23), 0), 24);
}
__device__ __forceinline__ float exp_of_2(int k) { return __uint_as_float(static_cast<uint32_t>(127 + k) << 23); }

template <bool Bf>
__device__ __forceinline__ float4v mfma16(u32x4 a, u32x4 b, float4v c) {
    if constexpr (Bf) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
}

// Byte address of 16 bytes (8 tokens of quarter q4) of ``channel`` in 32-token step ks of the
// transposed Value buffer; the quarters are rotated by channel group, which spreads the unpack's
// stores over the banks.
__device__ __forceinline__ int vt_at(int ks, int channel, int q4) {
    return ((ks * kD + channel) * 4 + ((q4 + (channel >> 2)) & 3)) * 16;
}

// Bf: rows are bf16 (else fp16).  WT: waves that share a row group's tokens.
template <bool Bf, int WT>
__global__ __launch_bounds__(kThreads, 2) void decode_rows_kernel(RowsParams rp) {
    constexpr int kWR = kWaves / WT;   // row groups of 16
    constexpr int kTT = 8 / WT;        // 16-token tiles of a wave per page
    constexpr int kKS = kTT / 2;       // 32-token steps of a wave per page
    const DecodeParams& p = rp.p;
    const RowsLayout& y = rp.y;
    const lf_packed_layer& L = p.L;
    const lf_decode_args& A = p.A;
    const int h = blockIdx.y, item = blockIdx.z;
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, q4 = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave % kWR, wt = wave / kWR;  // this wave's row group and token group
    typedef const __attribute__((address_space(4))) i32x4 ci32x4;
    const i32x4 rec = ((ci32x4*)A.work)[item];
    const int b = rec[0], pbeg = rec[1], pend = rec[2], kind = rec[3] & 0xff;
    const int part_slot = static_cast<unsigned>(rec[3] >> 8) - 1u < static_cast<unsigned>(A.n_work) ? (rec[3] >> 8) - 1 : item;
    const int row_first = 16 * kWR * static_cast<int>(blockIdx.x);   // the workgroup's rows
    const int row_end = min(p.g, row_first + 16 * kWR);
    const int row = row_first + 16 * wr + n;                         // this lane's row
    const int row_safe = min(row, p.g - 1);                          // (lanes past the rows repeat the last)
    const int64_t bh = static_cast<int64_t>(b) * L.n_kv + h;

    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char* kbuf = smem;
    unsigned char* vbuf = smem + y.off_v;
    float* sbuf = reinterpret_cast<float*>(smem + y.off_s);  // Key scales [nb * 8], mins [nb * 8]
    float* vsb = sbuf + 16 * y.nb;                            // Value scales [128], scaled middles [128],
                                                              // 1 / the page's factor

    const uint16_t* qrow = static_cast<const uint16_t*>(A.query) + (static_cast<int64_t>(b) * A.n_q + h * p.g + row_safe) * kD;
    auto widen = [](uint32_t u) { return Bf ? bf16_to_f32(static_cast<uint16_t>(u)) : f16_to_f32(static_cast<uint16_t>(u)); };

    float m = -__builtin_inff(), l = 0.f, csum = 0.f;
    float4v o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = float4v{0.f, 0.f, 0.f, 0.f};

    // New scores of the lane's kTT * 4 tokens: moves the reference point when one exceeds it by more
    // than 8 (log2), then turns the scores into weights and adds them to l.
    auto softmax = [&](float (&s)[kTT * 4]) {
        float mx = s[0];
#pragma unroll
        for (int e = 1; e < kTT * 4; ++e) mx = fmaxf(mx, s[e]);
        if (__any(mx > m + 8.f || m == -__builtin_inff())) {
            const float mnew = fmaxf(m, rows_max(mx));
            const float alpha = mnew == m ? 1.f : __builtin_amdgcn_exp2f(m - mnew);
            m = mnew;
            l *= alpha;
            csum *= alpha;
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] *= alpha;
        }
        const float mref = m == -__builtin_inff() ? 0.f : m;
#pragma unroll
        for (int e = 0; e < kTT * 4; ++e) {
            s[e] = __builtin_amdgcn_exp2f(s[e] - mref);
            l += s[e];
        }
    };

    if (kind != 1 && pbeg < pend) {
        // ---- the wave's q, in block order, packed ----
        const int steps = in_sgpr(y.steps), stride = in_sgpr(y.stride);
        const int st1 = in_sgpr(y.step1), st2 = in_sgpr(y.step2), st3 = in_sgpr(y.step3);
        const int cnt0 = L.k_width[0] > 0 ? L.tier_count[0][h] : 0, cnt1 = L.k_width[1] > 0 ? L.tier_count[1][h] : 0;
        const int cnt2 = L.k_width[2] > 0 ? L.tier_count[2][h] : 0, cnt3 = L.k_width[3] > 0 ? L.tier_count[3][h] : 0;
        const int32_t *ti0 = in_sgpr(L.tier_index[0] + h * L.k_width[0]), *ti1 = in_sgpr(L.tier_index[1] + h * L.k_width[1]);
        const int32_t *ti2 = in_sgpr(L.tier_index[2] + h * L.k_width[2]), *ti3 = in_sgpr(L.tier_index[3] + h * L.k_width[3]);
        // The rows' q and the channel of every position go through LDS (a gather from memory per
        // position and row took the prologue 18 us).
        constexpr int kQStride = 2 * kD + 16;
        int16_t* chan = reinterpret_cast<int16_t*>(vbuf);
        uint32_t qtop = 0;  // largest |q| bits of the thread's elements, even and odd ones
        for (int i = tid; i < 16 * kWR * 16; i += kThreads) {
            const int r = min(row_first + (i >> 4), p.g - 1);
            const u32x4 q = *reinterpret_cast<const u32x4*>(
                static_cast<const uint16_t*>(A.query) + (static_cast<int64_t>(b) * A.n_q + h * p.g + r) * kD + 8 * (i & 15));
            *reinterpret_cast<u32x4*>(kbuf + (i >> 4) * kQStride + 16 * (i & 15)) = q;
#pragma unroll
            for (int k = 0; k < 4; ++k) qtop = pair_max(qtop, q[k] & 0x7fff7fffu);
        }
        // (a NaN counts as an infinity: the factor is then 1 and the bound holds for the other rows)
        qtop = max(qtop & 0xffffu, qtop >> 16);
        const float top = wave_top(fminf(fabsf(widen(qtop)), __builtin_inff()));
        if (lane == 0) vsb[wave] = top;
        if (tid < 8 * y.nb) {
            const int s = tid >> 5;
            const bool in1 = s >= st1, in2 = s >= st2, in3 = s >= st3;
            const int slot = sm_slot(in1 + in2 + in3, (tid >> 3) - 4 * pick4(in1, in2, in3, 0, st1, st2, st3), tid & 7);
            int c = -1;
            if (slot < pick4(in1, in2, in3, cnt0, cnt1, cnt2, cnt3)) c = pick4(in1, in2, in3, ti0, ti1, ti2, ti3)[slot];
            chan[tid] = static_cast<int16_t>(c);
        }
        __syncthreads();
        float qbound = vsb[0];
#pragma unroll
        for (int k = 1; k < kWaves; ++k) qbound = fmaxf(qbound, vsb[k]);
        qbound *= fabsf(p.qscale) * kTopMargin;  // of |Qs| / scale
        u32x4 qr[kMaxSteps];
#pragma unroll
        for (int s = 0; s < kMaxSteps; ++s) {
            qr[s] = u32x4{0, 0, 0, 0};
            if (s >= steps) continue;
            const u32x4 cc = *reinterpret_cast<const u32x4*>(chan + (4 * s + q4) * 8);
            const uint16_t* qs = reinterpret_cast<const uint16_t*>(kbuf + (16 * wr + n) * kQStride);
            uint32_t x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int c = static_cast<int16_t>(cc[e >> 1] >> (16 * (e & 1)));
                x[e] = c >= 0 ? qs[max(c, 0)] : 0u;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) qr[s][k] = x[2 * k] | x[2 * k + 1] << 16;
        }
        __syncthreads();  // (the buffers change hands)

        // ---- a page's bytes, by LDS-DMA: chunk 64 (8 i + wave) + lane of the regions laid end to end ----
        const int64_t tok0 = bh * L.cap_tokens + static_cast<int64_t>(pbeg) * kPage;
        auto bytes = [](const void* q, int64_t off) { return in_sgpr(static_cast<const unsigned char*>(q) + off); };
        const int w0 = in_sgpr(L.k_words[0]), w1 = in_sgpr(L.k_words[1]), w2 = in_sgpr(L.k_words[2]), w16 = in_sgpr(L.k_width[3]);
        const int e0 = in_sgpr(y.end[0]), e1 = in_sgpr(y.end[1]), e2 = in_sgpr(y.end[2]), e3 = in_sgpr(y.end[3]);
        const int e4 = in_sgpr(y.end[4]), e5 = in_sgpr(y.end[5]), e6 = in_sgpr(y.end[6]), e7 = in_sgpr(y.end[7]);
        const unsigned char *k0 = bytes(L.k_code[0], tok0 * w0 * 4), *k1 = bytes(L.k_code[1], tok0 * w1 * 4);
        const unsigned char *k2 = bytes(L.k_code[2], tok0 * w2 * 4), *k3 = bytes(L.k_value16, tok0 * w16 * 2);
        const unsigned char *vc = bytes(L.v_code, tok0 * 32), *vsp = bytes(L.v_scale, tok0 * 2), *vmp = bytes(L.v_min, tok0 * 2);
        const unsigned char* smp = bytes(L.k_sm_page, (bh * L.cap_kgroups + pbeg) * 32 * y.nb_int);
        const unsigned char* src[kMaxDma];
        uint32_t step[kMaxDma];  // bytes to the same chunk of the next page
#pragma unroll
        for (int i = 0; i < kMaxDma; ++i) {
            const int c = min(64 * (kWaves * i + wave) + lane, e7 - 1);  // (past the end: the last chunk again)
            const bool v0 = c >= e3, v1 = c >= e4, v2 = c >= e5, v3 = c >= e6;
            const int first = v0 ? pick4(v1, v2, v3, e3, e4, e5, e6) : pick4(c >= e0, c >= e1, c >= e2, 0, e0, e1, e2);
            src[i] = (v0 ? pick4(v1, v2, v3, vc, vsp, vmp, smp) : pick4(c >= e0, c >= e1, c >= e2, k0, k1, k2, k3)) + 16 * (c - first);
            step[i] = v0 ? pick4(v1, v2, v3, 32 * kPage, 2 * kPage, 2 * kPage, 32 * y.nb_int)
                         : pick4(c >= e0, c >= e1, c >= e2, 4 * w0, 4 * w1, 4 * w2, 2 * w16) * kPage;
        }
        const uint32_t raw_lds = lds_addr(smem + y.off_raw) + 1024 * wave;
        auto load_page = [&](int buffer) {  // the next page, into raw buffer 0 or 1
#pragma unroll
            for (int i = 0; i < kMaxDma; ++i)
                if (64 * (kWaves * i + wave) < e7) {
                    dma16(src[i], raw_lds + buffer * y.raw_bytes + 1024 * kWaves * i);
                    src[i] += step[i];
                }
        };
        // idx / w as idx * r >> 20, r = ceil(2^20 / w): exact for idx < 128 w, w < 90
        auto reciprocal = [](int w) { return in_sgpr(w > 0 ? static_cast<int>(((1u << 20) + w - 1) / w) : 0); };
        const uint32_t r0 = reciprocal(w0), r1 = reciprocal(w1), r2 = reciprocal(w2), r16 = reciprocal(w16);
        const uint32_t pairs = fresh(0x03000300u), zero = fresh(0x000c000cu);
        const uint32_t key_table = fresh(0x42403C00u);    // high bytes of fp16 0, 1, 2, 3
        const uint32_t value_table = fresh(0x3E38B8BEu);  // ... and of -1.5, -0.5, 0.5, 1.5
        auto unpack_page = [&](const unsigned char* raw) {
            // (fresh: addresses are computed here, not kept in registers over the page loop)
            const int tid = static_cast<int>(fresh(threadIdx.x));
            // Scales and mins: every wave that needs the page's largest scale (1 for the fp16 tier) finds
            // it itself
            if (__builtin_amdgcn_readfirstlane(tid) < 8 * y.nb) {
                const unsigned char* sm = raw + 16 * e6;
                uint32_t t2 = w16 > 0 ? 0x3C00u : 0u;
                if (lane < y.nb_int) {
                    const u32x4 w = *reinterpret_cast<const u32x4*>(sm + 32 * lane);
                    t2 = pair_max(pair_max(t2, w[0]), pair_max(w[1], pair_max(w[2], w[3])));
                }
                const float top = wave_top(f16_to_f32(static_cast<uint16_t>(max(t2 & 0xffffu, t2 >> 16)))) * qbound;
                const int k = qs_exponent(top);
                const float unit = p.qscale * exp_of_2(k);
                if (tid < 8 * y.nb_int) {
                    const uint16_t* at = reinterpret_cast<const uint16_t*>(sm) + (tid >> 3) * 16 + (tid & 7);
                    sbuf[tid] = f16_to_f32(at[0]) * unit;
                    sbuf[8 * y.nb + tid] = f16_to_f32(at[8]) * p.qscale;
                } else if (tid < 8 * y.nb) {  // (their mins stay 0)
                    sbuf[tid] = unit;
                }
                if (tid == 0) vsb[2 * kPage] = exp_of_2(-k);
            }
            for (int c = tid; c < e3; c += kThreads) {
                const u32x4 w4 = *reinterpret_cast<const u32x4*>(raw + 16 * c);
                if (c < e0) {  // int2: 16 codes a word, block halves (j, j + 8), j = 0..3 and 4..7
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const uint32_t w = w4[k], idx = 4 * c + k, tok = idx * r0 >> 20, word = idx - tok * w0;
                        unsigned char* at = kbuf + tok * stride + (8 * (word >> 2) + (word & 3)) * 16;
                        *reinterpret_cast<half8*>(at) = as_half8(code_pair(w << 8, key_table, pairs, zero), code_pair(w << 6, key_table, pairs, zero),
                                                                 code_pair(w << 4, key_table, pairs, zero), code_pair(w << 2, key_table, pairs, zero));
                        *reinterpret_cast<half8*>(at + 64) = as_half8(code_pair(w, key_table, pairs, zero), code_pair(w >> 2, key_table, pairs, zero),
                                                                      code_pair(w >> 4, key_table, pairs, zero), code_pair(w >> 6, key_table, pairs, zero));
                    }
                } else if (c < e2) {
                    // int4 and int8: the code's bits under the exponent of 1 024, less that (exact)
                    const bool four = c < e1;
                    const uint32_t words = four ? w1 : w2, rec_w = four ? r1 : r2;
                    auto ints = [](uint32_t x, uint32_t mask) {
                        const _Float16 z = static_cast<_Float16>(1024.f);
                        return __builtin_bit_cast(half2v, (x & mask) | 0x64006400u) - half2v{z, z};
                    };
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const uint32_t w = w4[k], idx = 4 * (c - (four ? e0 : e1)) + k, tok = idx * rec_w >> 20, word = idx - tok * words;
                        if (four) {
                            unsigned char* at = kbuf + tok * stride + (4 * st1 + word) * 16;
                            half2v x[4];
#pragma unroll
                            for (int r = 0; r < 4; ++r) x[r] = ints(w >> (4 * r), 0x000f000fu);
                            *reinterpret_cast<half8*>(at) = half8{x[0][0], x[0][1], x[1][0], x[1][1], x[2][0], x[2][1], x[3][0], x[3][1]};
                        } else {
                            typedef _Float16 half4 __attribute__((ext_vector_type(4)));
                            unsigned char* at = kbuf + tok * stride + (4 * st2 + (word >> 1)) * 16 + (word & 1) * 8;
                            const half2v x = ints(w, 0x00ff00ffu), z = ints(w >> 8, 0x00ff00ffu);
                            *reinterpret_cast<half4*>(at) = half4{x[0], x[1], z[0], z[1]};
                        }
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        const uint32_t idx = 8 * (c - e2) + k, tok = idx * r16 >> 20, j = idx - tok * w16;
                        *reinterpret_cast<uint16_t*>(kbuf + tok * stride + 4 * st3 * 16 + j * 2) =
                            static_cast<uint16_t>(w4[k >> 1] >> (16 * (k & 1)));
                    }
                }
            }
            // Values: byte (tid & 3) of the octet's words: 4 channels x 8 tokens
            const int oct = tid >> 5, word = (tid >> 2) & 7, by = tid & 3;
            const uint32_t sel = 0x04040000u + 0x01010101u * by;
            uint32_t vraw[8], pr[4];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int tok = 32 * (oct >> 2) + 16 * (e >> 2) + 4 * (oct & 3) + (e & 3);
                vraw[e] = *reinterpret_cast<const uint32_t*>(raw + 16 * e3 + tok * 32 + word * 4);
            }
            // pr: two tokens' byte, each twice
#pragma unroll
            for (int k = 0; k < 4; ++k) pr[k] = __builtin_amdgcn_perm(vraw[2 * k + 1], vraw[2 * k], sel);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                *reinterpret_cast<half8*>(vbuf + vt_at(oct >> 2, 16 * word + 4 * by + j, oct & 3)) =
                    as_half8(code_pair(pr[0] >> (2 * j), value_table, pairs, zero), code_pair(pr[1] >> (2 * j), value_table, pairs, zero),
                             code_pair(pr[2] >> (2 * j), value_table, pairs, zero), code_pair(pr[3] >> (2 * j), value_table, pairs, zero));
            if (tid < kPage) {
                const float s = f16_to_f32(reinterpret_cast<const uint16_t*>(raw + 16 * e4)[tid]);
                vsb[tid] = s;
                vsb[kPage + tid] = fmaf(1.5f, s, f16_to_f32(reinterpret_cast<const uint16_t*>(raw + 16 * e5)[tid]));
            }
        };

        // blocks of padding words stay 0, as do the fp16 tier's mins
        for (int i = tid; i < kPage * y.stride / 16; i += kThreads) reinterpret_cast<u32x4*>(kbuf)[i] = u32x4{0, 0, 0, 0};
        for (int i = 8 * y.nb_int + tid; i < 8 * y.nb; i += kThreads) sbuf[8 * y.nb + i] = 0.f;
        load_page(0);
        for (int page = pbeg; page < pend; ++page) {
            const int buffer = (page - pbeg) & 1;
            // the page has landed, the one before it is computed
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (page + 1 < pend) load_page(buffer ^ 1);
            unpack_page(smem + y.off_raw + buffer * y.raw_bytes);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (the DMA stays in flight)

            // ---- scores of the wave's tokens ----
            float4v acc[kTT];
#pragma unroll
            for (int T = 0; T < kTT; ++T) acc[T] = float4v{0.f, 0.f, 0.f, 0.f};
            float bias = 0.f;
            const unsigned char* krow = kbuf + (16 * kTT * wt + n) * stride + q4 * 16;
            // (the count is laundered: ten conditions kept over the page loop cost SGPR spills)
            int n_steps = steps;
            asm volatile("" : "+s"(n_steps));
#pragma unroll
            for (int s = 0; s < kMaxSteps; ++s) {
                if (s >= n_steps) continue;
                const float4v* sp = reinterpret_cast<const float4v*>(sbuf + (4 * s + q4) * 8);
                const float4v* mp = reinterpret_cast<const float4v*>(sbuf + 8 * y.nb + (4 * s + q4) * 8);
                const float4v sa = sp[0], sb = sp[1], ma = mp[0], mb = mp[1];
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float q = widen(qr[s][e >> 1] >> (16 * (e & 1)));
                    x[e] = q * (e < 4 ? sa[e & 3] : sb[e & 3]);
                    bias = fmaf(q, e < 4 ? ma[e & 3] : mb[e & 3], bias);
                }
                const Split2 B = split2(x);
                half8 a[kTT];
#pragma unroll
                for (int T = 0; T < kTT; ++T) a[T] = *reinterpret_cast<const half8*>(krow + 16 * T * stride + s * 64);
#pragma unroll
                for (int T = 0; T < kTT; ++T) acc[T] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[T], B.lo, acc[T], 0, 0, 0);
#pragma unroll
                for (int T = 0; T < kTT; ++T) acc[T] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[T], B.hi, acc[T], 0, 0, 0);
            }
            const float inv = vsb[2 * kPage];
            bias = rows_sum(bias);
            float s[kTT * 4];
#pragma unroll
            for (int e = 0; e < kTT * 4; ++e) s[e] = fmaf(acc[e >> 2][e & 3], inv, bias);
            softmax(s);

            // ---- Values ----
#pragma unroll
            for (int u = 0; u < kKS; ++u) {
                const int ks = kKS * wt + u;
                float x[8];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int tok = 32 * ks + 16 * t + 4 * q4;
                    const float4v vs = *reinterpret_cast<const float4v*>(vsb + tok);
                    const float4v vm = *reinterpret_cast<const float4v*>(vsb + kPage + tok);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float pr = s[8 * u + 4 * t + i];
                        x[4 * t + i] = pr * vs[i];
                        csum = fmaf(pr, vm[i], csum);
                    }
                }
                const Split2 B = split2(x);
                half8 a[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) a[j] = *reinterpret_cast<const half8*>(vbuf + vt_at(ks, 16 * j + n, q4));
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j], B.lo, o[j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j], B.hi, o[j], 0, 0, 0);
            }
        }
    }

    if (kind != 0) {
        // ---- residual: the tail page, then the new tokens, 128 dense tokens at a time ----
        const int q_len = p.q_len;
        const int tl = min(max(A.tail_len[b], 0), min(A.tail_cap, kPage - 1));
        const int n_res = tl + (A.k_new != nullptr ? q_len : 0);
        // new tokens beyond every row's own are masked for all of the workgroup's rows
        int last = q_len - 1;
        if (row_first / q_len == (row_end - 1) / q_len) last = (row_end - 1) % q_len;
        const int n_vis = min(n_res, tl + last + 1);
        const int own = row_safe % q_len;
        u32x4 qd[4];  // the row's q by channel
#pragma unroll
        for (int s = 0; s < 4; ++s) qd[s] = *reinterpret_cast<const u32x4*>(qrow + 32 * s + 8 * q4);
        auto row_ptr = [&](const void* tail, const void* fresh_rows, int t) {
            t = min(t, n_res - 1);
            return t < tl ? static_cast<const uint16_t*>(tail) + (bh * A.tail_cap + t) * kD
                          : static_cast<const uint16_t*>(fresh_rows) + (bh * q_len + t - tl) * kD;
        };
        for (int t0 = 0; t0 < n_vis; t0 += kPage) {
            const int cnt = min(kPage, n_vis - t0);
            __syncthreads();  // the buffers are free
            // rows past the visible ones are zeros: they weigh nothing, and 0 * 0 stays 0
            u32x4 kr[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int idx = tid + kThreads * i, t = idx >> 4, c = idx & 15;
                kr[i] = u32x4{0, 0, 0, 0};
                if (t < cnt) kr[i] = *reinterpret_cast<const u32x4*>(row_ptr(A.tail_k, A.k_new, t0 + t) + 8 * c);
            }
            uint32_t vr[2][8];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int idx = tid + kThreads * i, oct = idx >> 6, pair = idx & 63;  // octet, channel pair
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int t = 32 * (oct >> 2) + 16 * (e >> 2) + 4 * (oct & 3) + (e & 3);
                    vr[i][e] = 0;
                    if (t < cnt) vr[i][e] = *reinterpret_cast<const uint32_t*>(row_ptr(A.tail_v, A.v_new, t0 + t) + 2 * pair);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int idx = tid + kThreads * i;
                *reinterpret_cast<u32x4*>(kbuf + (idx >> 4) * kDenseStride + 16 * (idx & 15)) = kr[i];
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int idx = tid + kThreads * i, oct = idx >> 6, pair = idx & 63;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    u32x4 w;
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        w[k] = __builtin_amdgcn_perm(vr[i][2 * k + 1], vr[i][2 * k], c ? 0x07060302u : 0x05040100u);
                    *reinterpret_cast<u32x4*>(vbuf + vt_at(oct >> 2, 2 * pair + c, oct & 3)) = w;
                }
            }
            __syncthreads();
            if (16 * kTT * wt >= cnt) continue;  // none of this wave's tokens

            float4v acc[kTT];
#pragma unroll
            for (int T = 0; T < kTT; ++T) acc[T] = float4v{0.f, 0.f, 0.f, 0.f};
            const unsigned char* krow = kbuf + (16 * kTT * wt + n) * kDenseStride + q4 * 16;
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int T = 0; T < kTT; ++T)
                    acc[T] = mfma16<Bf>(*reinterpret_cast<const u32x4*>(krow + 16 * T * kDenseStride + s * 64), qd[s], acc[T]);
            float s[kTT * 4];
#pragma unroll
            for (int e = 0; e < kTT * 4; ++e) {
                const int t = t0 + 16 * (kTT * wt + (e >> 2)) + 4 * q4 + (e & 3);
                s[e] = t >= n_res || t - tl > own ? -__builtin_inff() : acc[e >> 2][e & 3] * p.qscale;
            }
            softmax(s);
#pragma unroll
            for (int u = 0; u < kKS; ++u) {
                const int ks = kKS * wt + u;
                // p in parts of the rows' type: fp16 two, bf16 three (by truncation, exact)
                u32x4 part[3];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float pa = s[8 * u + 2 * k], pb = s[8 * u + 2 * k + 1];
                    if constexpr (Bf) {
                        auto top = [](float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); };
                        auto pair = [](float x, float z) { return __builtin_amdgcn_perm(__float_as_uint(z), __float_as_uint(x), 0x07060302u); };
                        const float ra = pa - top(pa), rb = pb - top(pb);
                        part[0][k] = pair(ra - top(ra), rb - top(rb));
                        part[1][k] = pair(ra, rb);
                        part[2][k] = pair(pa, pb);
                    } else {
                        const float ha = static_cast<float>(static_cast<_Float16>(pa)), hb = static_cast<float>(static_cast<_Float16>(pb));
                        part[0][k] = 0;
                        part[1][k] = pack_half(pa - ha, pb - hb);
                        part[2][k] = pack_half(pa, pb);
                    }
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const u32x4 a = *reinterpret_cast<const u32x4*>(vbuf + vt_at(ks, 16 * j + n, q4));
#pragma unroll
                    for (int k = Bf ? 0 : 1; k < 3; ++k) o[j] = mfma16<Bf>(a, part[k], o[j]);
                }
            }
        }
    }

    // ---- the row's partial: over the lane quarters, then over the waves that share its tokens ----
    l = rows_sum(l);
    csum = rows_sum(csum);
    if constexpr (WT > 1) {
        constexpr int kLd = kD + 4;  // row stride of the merge slots
        float* slots = reinterpret_cast<float*>(smem);               // [wave][16 rows][kLd]
        float* stat = slots + kWaves * 16 * kLd;                     // [wave][16 rows]: m, then l
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; ++j) *reinterpret_cast<float4v*>(slots + (wave * 16 + n) * kLd + 16 * j + 4 * q4) = o[j] + csum;
        if (q4 == 0) {
            stat[wave * 16 + n] = m;
            stat[(kWaves + wave) * 16 + n] = l;
        }
        __syncthreads();
        for (int e = tid; e < 16 * kWR * kD; e += kThreads) {
            const int r = e / kD, c = e % kD;  // row of the workgroup
            if (row_first + r >= row_end) break;
            float mw[WT], M = -__builtin_inff(), lo = 0.f, oo = 0.f;
#pragma unroll
            for (int w = 0; w < WT; ++w) { mw[w] = stat[(w * kWR + r / 16) * 16 + r % 16]; M = fmaxf(M, mw[w]); }
#pragma unroll
            for (int w = 0; w < WT; ++w) {
                const int at = (w * kWR + r / 16) * 16 + r % 16;
                const float f = M == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(mw[w] - M);
                lo = fmaf(f, stat[kWaves * 16 + at], lo);
                oo = fmaf(f, slots[at * kLd + c], oo);
            }
            float* out = part_rec(p, part_slot, h, row_first + r);
            out[c] = oo;
            if (c == 0) { out[kD] = M; out[kD + 1] = lo; }
        }
    } else if (row < row_end) {
        float* out = part_rec(p, part_slot, h, row);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float4v v = o[j] + csum;
            __builtin_memcpy(out + 16 * j + 4 * q4, &v, 16);
        }
        if (q4 == 0) { out[kD] = m; out[kD + 1] = l; }
    }
    if (A.commit_new && kind != 0 && blockIdx.x == 0) commit_new_rows(p, b, h, tid, kThreads);
}

bool aligned(const void* ptr, uintptr_t a) { return (reinterpret_cast<uintptr_t>(ptr) & (a - 1)) == 0; }

// Host: LDS layout for this layer; false when it is outside this kernel.
bool plan_rows(const lf_packed_layer& L, RowsLayout& y) {
    if (L.head_dim != kD || L.page_size != kPage || L.k_group != kPage || L.bit_v != 2 || L.v_group != kD) return false;
    if (L.k_sm_page == nullptr) return false;
    const SmPage sp = sm_page(L.k_words);
    y.nb_int = sp.nb;
    y.step1 = sp.blk0[1] / 4;
    y.step2 = sp.blk0[2] / 4;
    y.step3 = sp.nb / 4;
    y.steps = y.step3 + (L.k_width[3] + 31) / 32;
    if (y.steps == 0 || y.steps > kMaxSteps) return false;
    y.nb = 4 * y.steps;
    int c = 0;
    for (int i = 0; i < 8; ++i) {
        c += i < 3 ? kPage / 4 * L.k_words[i] : i == 3 ? kPage / 8 * L.k_width[3] : i == 4 ? kPage * 2 : i < 7 ? kPage / 8 : 2 * y.nb_int;
        y.end[i] = c;
    }
    if (c > 64 * kWaves * kMaxDma || 8 * y.nb > kThreads) return false;
    for (int t = 0; t < 3; ++t)
        if (L.k_width[t] && (!aligned(L.k_code[t], 16) || L.k_words[t] >= 90)) return false;
    if (L.k_width[3] && (!aligned(L.k_value16, 16) || L.k_width[3] >= 90)) return false;
    if (!aligned(L.v_code, 16) || !aligned(L.v_scale, 16) || !aligned(L.v_min, 16) || !aligned(L.k_sm_page, 16)) return false;
    if (L.cap_tokens % kPage) return false;
    y.stride = 16 * y.nb + 16;
    y.off_v = kPage * std::max(y.stride, kDenseStride);
    y.off_s = y.off_v + kVtBytes;
    y.off_raw = y.off_s + (16 * y.nb + 2 * kPage + 4) * 4;
    y.raw_bytes = 1024 * ((c + 63) / 64);
    y.lds_bytes = y.off_raw + 2 * y.raw_bytes;
    const int merge = kWaves * 16 * (kD + 4) * 4 + 2 * kWaves * 16 * 4;
    y.lds_bytes = std::max(y.lds_bytes, merge);
    return y.lds_bytes <= 160 * 1024;
}

template <bool Bf, int WT>
int launch_rows(const RowsParams& rp, hipStream_t stream) {
    const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(&decode_rows_kernel<Bf, WT>), rp.y.lds_bytes);
    if (rc != LF_OK) return rc;
    constexpr int kRowsWg = 16 * kWaves / WT;
    const dim3 grid((rp.p.g + kRowsWg - 1) / kRowsWg, rp.p.L.n_kv, rp.p.A.n_work);
    hipLaunchKernelGGL((decode_rows_kernel<Bf, WT>), grid, dim3(kThreads), rp.y.lds_bytes, stream, rp);
    return LF_OK;
}

bool serves(const DecodeParams& p, int64_t pages, RowsLayout& y) {
    const int tiles = (p.g + 7) / 8;
    if (tiles < kRowsTiles || p.A.n_work > 65535 || p.L.n_kv > 65535) return false;
    if (pages * p.L.n_kv * tiles < kRowsWork) return false;
    // 2-byte rows of one dtype, read in 16-byte pieces
    const int dt = p.A.q_dtype;
    if (dt == LF_FP32 || !aligned(p.A.query, 16)) return false;
    if (p.A.k_new && (p.A.new_dtype != dt || !aligned(p.A.k_new, 16) || !aligned(p.A.v_new, 16))) return false;
    if (p.A.tail_cap > 0 && (p.A.tail_dtype != dt || !aligned(p.A.tail_k, 16) || !aligned(p.A.tail_v, 16))) return false;
    return plan_rows(p.L, y);
}

}  // namespace

bool decode_rows_serves(const DecodeParams& p, int64_t pages) {
    RowsLayout y;
    return serves(p, pages, y);
}

int launch_decode_rows(const DecodeParams& p, hipStream_t stream, bool* handled) {
    RowsParams rp;
    rp.p = p;
    int64_t pages = 0;
    for (int i = 0; p.A.work_host && i < p.A.n_work; ++i) pages += p.A.work_host[4 * i + 2] - p.A.work_host[4 * i + 1];
    *handled = serves(p, pages, rp.y);
    if (!*handled) return LF_OK;
    const bool bf = p.A.q_dtype == LF_BF16;
    int rc;
    if (p.g > 64) rc = bf ? launch_rows<true, 1>(rp, stream) : launch_rows<false, 1>(rp, stream);
    else rc = bf ? launch_rows<true, 2>(rp, stream) : launch_rows<false, 2>(rp, stream);
    if (rc != LF_OK) return rc;
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return static_cast<int>(err);
    return launch_decode_reduce(p, stream);
}

}  // namespace lf
