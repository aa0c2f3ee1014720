// Packed decode attention, matrix-core variant for the layouts outside decode_mfma.hip: head_dim
// 64, 128 or 256, any page of whole 32-token tiles, Key groups of whole 32-token tiles, Value
// groups of 16 * 2^k channels, any row dtype (with several new tokens as well).  Everything else
// runs the VALU kernel, whose fp32 precision this kernel keeps.
//
// Reference: src/logitfill/packed/kernel.cu:112-190 and reference.py:30-56, as decode_valu.hip.
//
// Work: one workgroup of 4 waves per (split item, kv head, tile of 8 query rows).  The item's
// tokens are cut into four contiguous shares of whole 32-token tiles; each wave walks its share in
// runs of 64 tokens on its own (own LDS buffers, own running softmax, no barrier until the merge
// of the four partials).  The run's packed rows arrive by LDS-DMA: the Key rows of run r + 1 are
// issued once run r's scores have read theirs and land behind its Value product, the Value rows
// behind run r + 1's scores.
//
// Scores: S^T = Codes . Qs^T on v_mfma_f32_16x16x32_bf16, A = 16 tokens x 32 slots of integer
// codes (exact in bf16), B = 32 slots x 8 query rows of Qs = q * scaling * log2(e) * scale, once for
// the Key group of the run's first 32 tokens (columns 0-7) and once for that of its last 32 (columns
// 8-15), cut into three bf16 parts that add up to the fp32 value exactly: every product is exact and the sums
// are the matrix cores' fp32, so nothing is held in fewer bits than the VALU kernel holds it, and
// bf16's exponent range leaves no scale out of range.  The K dimension is the tiers' slots in
// steps of 32 (four 8-slot blocks, block = lane / 16), in the order the codes unpack in
// (block_rank).  The fp16 tier's values are two bf16 parts each; a run that holds a non-finite one
// takes that tier in fp32 FMAs instead (the parts of an infinity do not add up).
//
// Values: O^T = (code - 1.5) . P'^T, P' = p * vscale per Value group in three bf16 parts.  A column
// (lane % 16) is a query row and half of the run from the scores to the output -- sixteen softmax
// streams a workgroup merges at the end --, so the running max, its rescale and the sums l = sum p,
// sum p * vmin and sum P' (the centre) stay in that lane and no lane works on another's tokens.
// The products of each half of the run's tokens go to accumulators of their own, whose columns of
// the other half are never read.  The channels of
// a Value group go to its 16-channel tiles so that a lane's codes of one token lie in one or two
// bytes of one word.
//
// What bounds it: VALU work (unpacking codes, 1.5 operations each; the three-part splits of Qs and P') at
// one or two waves per SIMD, and in short items the dependent loads before the first run (argument block,
// tier tables, q).  Counters of the two calls below: 5 700 VALU operations and 290 products per wave (two
// runs of 64 tokens, prologue, residual, merge) at 38 % of the VALU and 8 % of the matrix cores busy;
// 2 700 and 140 (one run) at 13 % and 3 %.  Registers: 256 VGPRs; head_dim 128 spills 9 to 28 of them, 256
// (whose accumulators alone are 128) 72 to 322, and still takes 1 / 2.6 to 1 / 81 of the general kernel's
// time (plan_tiled).  Measured with the general kernel before it (us per layer-step, decode and merge): 8 sequences of
// 3K-8K tokens, 28 q / 4 kv heads, head_dim 128, Key and Value groups of 32 at Key 4.0 bits
// 1 490 -> 35; 8 of 1.5K-5K, 14 / 2 heads, head_dim 64, 64-token pages and groups 124 -> 21.  Against
// float64 (float32 output) 1.6e-6 and 1.5e-6 where the general kernel has 2.2e-6 and 2.0e-6.
#include <algorithm>
#include <cstddef>
#include <cstring>
#include <type_traits>

#include "decode_common.hpp"

namespace lf {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kRows = 8;     // query rows per workgroup
constexpr int kStreams = 2 * kWaves;  // softmax streams of a row: (wave, half of the run)
constexpr int kRun = 64;     // tokens a wave takes at a time
constexpr int kWindow = 4;   // Key groups whose scales and mins are staged at a time

struct TiledLayout {
    int kst[4];      // K-steps of each tier
    int n_int;       // positions (32 per step) of the integer tiers
    int n_pos;       // ... and of the fp16 tier
    int rb[4];       // bytes of a token's row in each tier
    int cend[4];     // end of each tier's 16-byte chunks of a run
    int nk;          // DMA instructions of a run's Key rows
    int off_stat, off_q, off_buf, wave_bytes, sm_off;  // sm_off: scales inside a wave's buffer
    int lds_bytes;
};

struct TiledParams {
    DecodeParams p;
    TiledLayout y;
    int res_vec;      // the residual's rows are 16-byte aligned and of one dtype
    int inline_work;  // 1: work_inline holds the plan (n_work <= LF_INLINE_WORK)
    int32_t work_inline[4 * LF_INLINE_WORK];
};
static_assert(sizeof(TiledParams) <= 4096, "kernel arguments are limited to 4 KB");

// Rank inside its tier of element e (0..7) of lane group q's block in the tier's K-step j.
__device__ __forceinline__ int block_rank(int tier, int j, int q, int e) {
    const int pr = e >> 1, odd = e & 1;
    if (tier == 0) return 16 * (4 * (j >> 1) + q) + 8 * (j & 1) + pr + 4 * odd;
    if (tier == 1) return 8 * (4 * j + q) + 4 * (pr & 1) + (pr >> 1) + 2 * odd;
    if (tier == 2) return 8 * (4 * j + q) + e;
    return 32 * j + 4 * e + q;
}

// (tier, rank) of position pos of the K dimension; k1, k2, k3: the first K-steps of tiers 1 to 3.
__device__ __forceinline__ void pos_slot(int k1, int k2, int k3, int pos, int& tier, int& rank) {
    const int step = pos >> 5;
    const bool in1 = step >= k1, in2 = step >= k2, in3 = step >= k3;
    tier = (in1 ? 1 : 0) + (in2 ? 1 : 0) + (in3 ? 1 : 0);
    rank = block_rank(tier, step - pick4(in1, in2, in3, 0, k1, k2, k3), (pos >> 3) & 3, pos & 7);
}

__device__ __forceinline__ uint32_t fbits(float x) { return __float_as_uint(x); }
// bf16 pairs (lo half first): the upper halves of two floats, or of (code) table entries
__device__ __forceinline__ uint32_t upper_pair(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

// Lookup tables of a 2-bit code as bf16 (low and high bytes of its four values) and the selector's
// constants, held in VGPRs: VOP3 takes no literal and one SGPR, so each lookup is one and_or and
// one perm only with register operands.
struct CodeTable {
    uint32_t lo, hi, mask, high;
};
__device__ __forceinline__ uint32_t in_vgpr(uint32_t x) {
    asm volatile("" : "+v"(x));
    return x;
}
// x again, opaque to the compiler: what is derived from it is computed where it is used instead of
// being hoisted out of the token loop into registers (and spilled).
__device__ __forceinline__ int fresh(int x) {
    asm volatile("" : "+v"(x));
    return x;
}
__device__ __forceinline__ CodeTable code_table(uint32_t lo, uint32_t hi) {
    return {in_vgpr(lo), in_vgpr(hi), in_vgpr(0x03030303u), in_vgpr(0x04000400u)};
}
// 0, 1, 2, 3 (Key codes) and -1.5, -0.5, 0.5, 1.5 (Value codes about their middle)
__device__ __forceinline__ CodeTable key_table() { return code_table(0x40008000u, 0x40403F00u); }
__device__ __forceinline__ CodeTable value_table() { return code_table(0xC00000C0u, 0x3F3FBFBFu); }

__device__ __forceinline__ bf16x8 as_bf16x8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(bf16x8, u32x4{a, b, c, d});
}

// Eight 2-bit codes as bf16: s holds one byte of codes in bytes 0, 1 and another in bytes 2, 3;
// element pairs are (first byte's code j, second byte's code j).
__device__ __forceinline__ uint32_t code_pair(uint32_t s, const CodeTable& t) {
    return __builtin_amdgcn_perm(t.hi, t.lo, (s & t.mask) | t.high);
}
__device__ __forceinline__ bf16x8 codes8(uint32_t s, const CodeTable& t) {
    return as_bf16x8(code_pair(s, t), code_pair(s >> 2, t), code_pair(s >> 4, t), code_pair(s >> 6, t));
}

// The byte of a word as a float (exact), pairs packed to bf16.
template <int B>
__device__ __forceinline__ uint32_t byte_f32(uint32_t w) { return fbits(static_cast<float>((w >> (8 * B)) & 0xffu)); }

// 8 floats as three bf16 parts by truncation: x = hi + mid + lo exactly for finite x.
struct Split3 {
    bf16x8 hi, mid, lo;
};
__device__ __forceinline__ Split3 split3(const float (&x)[8]) {
    uint32_t h[4], m[4], l[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float a = x[2 * k], b = x[2 * k + 1];
        h[k] = upper_pair(fbits(a), fbits(b));
        const float ra = a - __uint_as_float(fbits(a) & 0xffff0000u), rb = b - __uint_as_float(fbits(b) & 0xffff0000u);
        m[k] = upper_pair(fbits(ra), fbits(rb));
        const float la = ra - __uint_as_float(fbits(ra) & 0xffff0000u), lb = rb - __uint_as_float(fbits(rb) & 0xffff0000u);
        l[k] = upper_pair(fbits(la), fbits(lb));
    }
    return {as_bf16x8(h[0], h[1], h[2], h[3]), as_bf16x8(m[0], m[1], m[2], m[3]), as_bf16x8(l[0], l[1], l[2], l[3])};
}

__device__ __forceinline__ float4v mfma3(bf16x8 a, const Split3& b, float4v c) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b.lo, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b.mid, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b.hi, c, 0, 0, 0);
}

// The same for the four token tiles of a run, part by part: a dependent product waits for the one
// before it, four independent ones in between cover that.
__device__ __forceinline__ void mfma3x4(const bf16x8 (&a)[4], const Split3& b, float4v (&c)[4]) {
#pragma unroll
    for (int T = 0; T < 4; ++T) c[T] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[T], b.lo, c[T], 0, 0, 0);
#pragma unroll
    for (int T = 0; T < 4; ++T) c[T] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[T], b.mid, c[T], 0, 0, 0);
#pragma unroll
    for (int T = 0; T < 4; ++T) c[T] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[T], b.hi, c[T], 0, 0, 0);
}

// This wave's DMA and LDS reads so far are done, except the newest N DMA instructions.
template <int N>
__device__ __forceinline__ void wait_dma() {
    if constexpr (N == 0) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// Keeps the compiler from starting the memory reads after it before the sums in x are done.
__device__ __forceinline__ void fence8(float (&x)[8]) {
    asm volatile("" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]), "+v"(x[6]), "+v"(x[7]) :: "memory");
}

// Eight consecutive elements as floats; ``Dt`` an lf_dtype.
template <int Dt>
__device__ __forceinline__ void widen8(const u32x4* raw, float (&x)[8]) {
    if constexpr (Dt == LF_FP32) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = __uint_as_float(raw[e >> 2][e & 3]);
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint16_t u = static_cast<uint16_t>(raw[0][e >> 1] >> (16 * (e & 1)));
            x[e] = Dt == LF_BF16 ? bf16_to_f32(u) : f16_to_f32(u);
        }
    }
}

// The residual -- the tail page, then the new tokens -- in plain fp32 FMAs (any row dtype, and
// infinities as fp32 arithmetic has them): 32 tokens per wave and pass.  Scores with lane =
// (token, half of the channels), the Value product with lane = D / 64 channels.  Row i (token
// i % q_len) sees new tokens 0 .. i % q_len; the tail length is clamped as in the other kernels.
// ``Dt``: the dtype of every row, read in 16-byte pieces that are all in flight at once, or -1
// (mixed dtypes, unaligned rows): element by element.
template <int D, int Dt>
__device__ __forceinline__ void residual_rows(const DecodeParams& p, int b, int h, int row0, int g, const float* qc, float* pb,
                                              int wave, int lane, float (&m)[kRows], float (&l)[kRows],
                                              float (&o)[D / 64][kRows]) {
    constexpr int CPL = D / 64;
    const lf_packed_layer& L = p.L;
    const lf_decode_args& A = p.A;
    const int64_t bh = static_cast<int64_t>(b) * L.n_kv + h;
    const int q_len = p.q_len;
    const int tl = min(max(A.tail_len[b], 0), min(A.tail_cap, L.page_size - 1));
    const int n_res = tl + (A.k_new != nullptr ? q_len : 0);
    const int tk = lane & 31, half = lane >> 5;
    for (int t0 = 32 * wave; t0 < n_res; t0 += 32 * kWaves) {
        const int tt = t0 + tk;
        const bool active = tt < n_res;
        float s[kRows];
#pragma unroll
        for (int i = 0; i < kRows; ++i) s[i] = 0.f;
        auto add = [&](int c, float k) {
            const float4v* q = reinterpret_cast<const float4v*>(qc + c * kRows);
            const float4v qa = q[0], qb = q[1];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[i] = fmaf(qa[i], k, s[i]);
                s[4 + i] = fmaf(qb[i], k, s[4 + i]);
            }
        };
        // row of token u (clamped to a stored one), as an element index of its tensor
        auto row_of = [&](int u, bool& tail) {
            u = min(u, n_res - 1);
            tail = u < tl;
            return tail ? (bh * A.tail_cap + u) * D : (bh * q_len + u - tl) * D;
        };
        bool tail;
        const int64_t kb = row_of(tt, tail) + half * (D / 2);
        if constexpr (Dt >= 0) {
            constexpr int kSize = Dt == LF_FP32 ? 4 : 2, kRaw = kSize / 2;      // 16-byte pieces per 8 elements
            constexpr int kGroups = D / 16, kBatch = kGroups * kRaw > 16 ? 16 / kRaw : kGroups;
            const unsigned char* base = static_cast<const unsigned char*>(tail ? A.tail_k : A.k_new) + kb * kSize;
#pragma unroll
            for (int c0 = 0; c0 < kGroups; c0 += kBatch) {
                u32x4 raw[kBatch * kRaw];
#pragma unroll
                for (int k = 0; k < kBatch * kRaw; ++k) raw[k] = *reinterpret_cast<const u32x4*>(base + 16 * (c0 * kRaw + k));
#pragma unroll
                for (int k = 0; k < kBatch; ++k) {
                    float x[8];
                    widen8<Dt>(raw + k * kRaw, x);
#pragma unroll
                    for (int e = 0; e < 8; ++e) add(half * (D / 2) + 8 * (c0 + k) + e, x[e]);
                    fence8(s);  // eight channels' q rows in registers at a time (all of them would spill)
                }
            }
        } else {
            for (int c = 0; c < D / 2; ++c)
                add(half * (D / 2) + c, load_as_f32(tail ? A.tail_k : A.k_new, kb + c, tail ? A.tail_dtype : A.new_dtype));
        }
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            float x = s[i] + __shfl_xor(s[i], 32, kWave);
            if (!active || (q_len > 1 && tt - tl > (row0 + i) % q_len)) x = -__builtin_inff();
            const float mnew = fmaxf(m[i], wave_max(x));
            const float alpha = mnew == -__builtin_inff() ? 1.f : __builtin_amdgcn_exp2f(m[i] - mnew);
            const float pr = mnew == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(x - mnew);
            m[i] = mnew;
            l[i] = fmaf(l[i], alpha, half ? 0.f : pr);
#pragma unroll
            for (int cc = 0; cc < CPL; ++cc) o[cc][i] *= alpha;
            if (half == 0) pb[tk * kRows + i] = pr;
        }
        __builtin_amdgcn_wave_barrier();
        // tokens past the residual carry p = 0 over a stored row's values; a non-finite one of
        // those must not enter
        const int cnt = min(32, n_res - t0);
        auto accumulate = [&](int j, int cc, float v) {
            const float4v* pr = reinterpret_cast<const float4v*>(pb + j * kRows);
            const float4v pa = pr[0], pc = pr[1];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                o[cc][i] = fmaf(pa[i], v, o[cc][i]);
                o[cc][4 + i] = fmaf(pc[i], v, o[cc][4 + i]);
            }
        };
        if constexpr (Dt >= 0) {
            constexpr int kSize = Dt == LF_FP32 ? 4 : 2, kTok = CPL * kSize > 8 ? 8 : 16;
#pragma unroll
            for (int j0 = 0; j0 < 32; j0 += kTok) {
                if (j0 >= cnt) break;
                float v[kTok][CPL];
#pragma unroll
                for (int j = 0; j < kTok; ++j) {
                    bool vt;
                    const int64_t at = row_of(t0 + j0 + j, vt) + CPL * lane;
                    const unsigned char* src = static_cast<const unsigned char*>(vt ? A.tail_v : A.v_new) + at * kSize;
                    if constexpr (Dt == LF_FP32) {
                        __builtin_memcpy(v[j], __builtin_assume_aligned(src, 4 * CPL), 4 * CPL);
                    } else {
                        uint16_t raw[CPL];
                        __builtin_memcpy(raw, __builtin_assume_aligned(src, 2 * CPL), 2 * CPL);
#pragma unroll
                        for (int cc = 0; cc < CPL; ++cc) v[j][cc] = Dt == LF_BF16 ? bf16_to_f32(raw[cc]) : f16_to_f32(raw[cc]);
                    }
                }
#pragma unroll
                for (int j = 0; j < kTok; ++j) {
#pragma unroll
                    for (int cc = 0; cc < CPL; ++cc) accumulate(j0 + j, cc, j0 + j < cnt ? v[j][cc] : 0.f);
                    if (j % 4 == 3) fence8(o[CPL - 1]);
                }
            }
        } else {
            for (int j = 0; j < cnt; ++j) {
                bool vt;
                const int64_t at = row_of(t0 + j, vt) + CPL * lane;
#pragma unroll
                for (int cc = 0; cc < CPL; ++cc)
                    accumulate(j, cc, load_as_f32(vt ? A.tail_v : A.v_new, at + cc, vt ? A.tail_dtype : A.new_dtype));
            }
        }
    }
}

// The residual's partials, one stream per wave, into ``slots`` and ``stat`` (q by channel and the
// probabilities behind the slots).
template <int D>
__device__ __forceinline__ void residual_pass(const TiledParams& tp, int b, int h, int row0, int g, float* slots, float* stat, int tid) {
    constexpr int CPL = D / 64, kLd = D + 1;
    const DecodeParams& p = tp.p;
    const lf_decode_args& A = p.A;
    const int lane = tid & 63, wave = tid >> 6;
    float* qc = slots + kStreams * kRows * kLd;     // [channel][row]
    float* pb = qc + D * kRows + wave * 32 * kRows; // [32 tokens][row]
    for (int idx = tid; idx < kRows * D; idx += kThreads) {
        const int i = idx / D, c = idx % D;
        float v = 0.f;
        if (i < g) v = load_as_f32(A.query, (static_cast<int64_t>(b) * A.n_q + h * p.g + row0 + i) * D + c, A.q_dtype) * p.qscale;
        qc[c * kRows + i] = v;
    }
    __syncthreads();
    float m[kRows], l[kRows], o[CPL][kRows];
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        m[i] = -__builtin_inff();
        l[i] = 0.f;
#pragma unroll
        for (int cc = 0; cc < CPL; ++cc) o[cc][i] = 0.f;
    }
    const int dt = A.tail_cap > 0 ? A.tail_dtype : A.new_dtype;
    if (!tp.res_vec) residual_rows<D, -1>(p, b, h, row0, g, qc, pb, wave, lane, m, l, o);
    else if (dt == LF_BF16) residual_rows<D, LF_BF16>(p, b, h, row0, g, qc, pb, wave, lane, m, l, o);
    else if (dt == LF_FP16) residual_rows<D, LF_FP16>(p, b, h, row0, g, qc, pb, wave, lane, m, l, o);
    else residual_rows<D, LF_FP32>(p, b, h, row0, g, qc, pb, wave, lane, m, l, o);
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
#pragma unroll
        for (int cc = 0; cc < CPL; ++cc) slots[(wave * kRows + i) * kLd + CPL * lane + cc] = o[cc][i];
        const float lt = wave_sum(l[i]);
        if (lane == 0) {
            stat[i * kStreams + wave] = m[i];
            stat[(kRows + i) * kStreams + wave] = lt;
        }
    }
}

// G: 32-bit words of a Value group's codes (16 channels each); D / 16 / G Value groups.
template <int D, int G>
__global__ __launch_bounds__(kThreads, 2) void decode_tiled_kernel(TiledParams tp) {
    constexpr int kVG = D / 16 / G;             // Value groups
    constexpr int kVChunks = D + 16 * kVG;      // 16-byte chunks of a run's Value rows: codes, scales, mins
    constexpr int kNV = (kVChunks + 63) / 64;   // DMA instructions
    constexpr int kTiles = D / 16;              // 16-channel output tiles
    constexpr int kEl = kRows * D / kThreads;   // merged outputs per thread
    constexpr int kLd = D + 1;                  // row stride of the merge slots
    // the argument block and this workgroup's inline work record, in one round of loads
    const i32x4 rec_arg = prefetch_args_rec4<offsetof(TiledParams, work_inline)>(
        static_cast<uint32_t>(offsetof(TiledParams, work_inline)) + 16u * min(blockIdx.y, LF_INLINE_WORK - 1u));
    const DecodeParams& p = tp.p;
    const TiledLayout& y = tp.y;
    const lf_packed_layer& L = p.L;
    const lf_decode_args& A = p.A;
    const int h = blockIdx.x, item = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, q4 = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row0 = kRows * static_cast<int>(blockIdx.z);
    const int g = min(kRows, p.g - row0);
    typedef const __attribute__((address_space(4))) i32x4 ci32x4;
    const i32x4 rec = tp.inline_work ? rec_arg : ((ci32x4*)A.work)[item];
    const int b = rec[0], pbeg = rec[1], pend = rec[2], kind = rec[3] & 0xff;
    const int part_slot = static_cast<unsigned>(rec[3] >> 8) - 1u < static_cast<unsigned>(A.n_work) ? (rec[3] >> 8) - 1 : item;

    extern __shared__ __align__(16) unsigned char smem[];
    float* stat = reinterpret_cast<float*>(smem + y.off_stat);  // [m, l][row][stream]
    float* qs = reinterpret_cast<float*>(smem + y.off_q);       // [block][half][row][4]
    unsigned char* buf = smem + y.off_buf + wave * y.wave_bytes;
    unsigned char* vbuf = buf + 1024 * y.nk;
    unsigned char* smbuf = buf + y.sm_off;                      // [window][block][8 scales, 8 mins] fp16
    const int64_t bh = static_cast<int64_t>(b) * L.n_kv + h;

    float om[kEl], Mm[kEl], Lm[kEl];  // merged partials: element tid + 256 k of [row][channel]
#pragma unroll
    for (int k = 0; k < kEl; ++k) { om[k] = 0.f; Lm[k] = 0.f; Mm[k] = -__builtin_inff(); }
    float* slots = reinterpret_cast<float*>(smem + y.off_buf);  // [stream][row][kLd], once the buffers are free

    // Merge the first ``ns`` streams' slots and statistics into the running (om, Mm, Lm).
    auto merge = [&](auto ns) {
        constexpr int kN = decltype(ns)::value;
#pragma unroll
        for (int k = 0; k < kEl; ++k) {
            const int e = tid + kThreads * k, row = e / D, c = e % D;
            if (row >= g) continue;
            float mw[kN], lw[kN], ow[kN], M = Mm[k];
#pragma unroll
            for (int w = 0; w < kN; w += 4) {
                const float4v a = *reinterpret_cast<const float4v*>(stat + row * kStreams + w);
                const float4v c4 = *reinterpret_cast<const float4v*>(stat + (kRows + row) * kStreams + w);
#pragma unroll
                for (int i = 0; i < 4; ++i) { mw[w + i] = a[i]; lw[w + i] = c4[i]; }
            }
#pragma unroll
            for (int w = 0; w < kN; ++w) { ow[w] = slots[(w * kRows + row) * kLd + c]; M = fmaxf(M, mw[w]); }
            const float w0 = M == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(Mm[k] - M);
            float o = om[k] * w0, l = Lm[k] * w0;
#pragma unroll
            for (int w = 0; w < kN; ++w) {
                const float ww = M == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(mw[w] - M);
                o = fmaf(ww, ow[w], o);
                l = fmaf(ww, lw[w], l);
            }
            om[k] = o; Lm[k] = l; Mm[k] = M;
        }
    };

    if (kind != 1) {
        const int64_t tok0 = static_cast<int64_t>(pbeg) * L.page_size;
        const int nt = (pend - pbeg) * L.page_size;
        const int share = (nt + 32 * kWaves - 1) / (32 * kWaves) * 32;
        const int t_lo = min(nt, wave * share), t_hi = min(nt, t_lo + share);

        // ---- the channel of a position (-1: none), its load ahead of the DMA it does not wait for ----
        const unsigned char* ti0 = in_sgpr(reinterpret_cast<const unsigned char*>(L.tier_index[0] + h * L.k_width[0]));
        const unsigned char* ti1 = in_sgpr(reinterpret_cast<const unsigned char*>(L.tier_index[1] + h * L.k_width[1]));
        const unsigned char* ti2 = in_sgpr(reinterpret_cast<const unsigned char*>(L.tier_index[2] + h * L.k_width[2]));
        const unsigned char* ti3 = in_sgpr(reinterpret_cast<const unsigned char*>(L.tier_index[3] + h * L.k_width[3]));
        const int cnt0 = L.k_width[0] > 0 ? L.tier_count[0][h] : 0, cnt1 = L.k_width[1] > 0 ? L.tier_count[1][h] : 0;
        const int cnt2 = L.k_width[2] > 0 ? L.tier_count[2][h] : 0, cnt3 = L.k_width[3] > 0 ? L.tier_count[3][h] : 0;
        const int k1 = in_sgpr(y.kst[0]), k2 = in_sgpr(k1 + y.kst[1]), k3 = in_sgpr(k2 + y.kst[2]);
        auto pos_channel = [&](int pos) {
            int t, rank;
            pos_slot(k1, k2, k3, pos, t, rank);
            const bool in1 = t >= 1, in2 = t >= 2, in3 = t >= 3;
            typedef const __attribute__((address_space(1))) int32_t global_i32;
            if (rank >= pick4(in1, in2, in3, L.k_width[0], L.k_width[1], L.k_width[2], L.k_width[3])) return -1;
            const int c = ((global_i32*)pick4(in1, in2, in3, ti0, ti1, ti2, ti3))[rank];
            return rank < pick4(in1, in2, in3, cnt0, cnt1, cnt2, cnt3) ? c : -1;
        };
        const int channel0 = tid < y.n_pos ? pos_channel(tid) : -1;

        // ---- DMA sources ----
        const int64_t row0k = bh * L.cap_tokens + tok0;
        const unsigned char* kb0 = in_sgpr(reinterpret_cast<const unsigned char*>(L.k_code[0]) + row0k * y.rb[0]);
        const unsigned char* kb1 = in_sgpr(reinterpret_cast<const unsigned char*>(L.k_code[1]) + row0k * y.rb[1]);
        const unsigned char* kb2 = in_sgpr(reinterpret_cast<const unsigned char*>(L.k_code[2]) + row0k * y.rb[2]);
        const unsigned char* kb3 = in_sgpr(reinterpret_cast<const unsigned char*>(L.k_value16) + row0k * y.rb[3]);
        const int rb0 = in_sgpr(y.rb[0]), rb1 = in_sgpr(y.rb[1]), rb2 = in_sgpr(y.rb[2]), rb3 = in_sgpr(y.rb[3]);
        const int ce0 = in_sgpr(y.cend[0]), ce1 = in_sgpr(y.cend[1]), ce2 = in_sgpr(y.cend[2]);
        const unsigned char* vcode = in_sgpr(reinterpret_cast<const unsigned char*>(L.v_code) + (bh * L.cap_tokens + tok0) * (D / 4));
        const unsigned char* vscale = in_sgpr(reinterpret_cast<const unsigned char*>(L.v_scale) + (bh * L.cap_tokens + tok0) * (2 * kVG));
        const unsigned char* vmin = in_sgpr(reinterpret_cast<const unsigned char*>(L.v_min) + (bh * L.cap_tokens + tok0) * (2 * kVG));
        const uint32_t kdst = lds_addr(buf), vdst = lds_addr(vbuf);
        // Run at token t (ntok = 32 or 64 of it valid): chunk c of the run's Key rows, tier by tier;
        // chunks past a tier's valid rows re-read its last valid chunk.
        auto dma_k = [&](int t, int ntok) {
            const int ln = fresh(lane);
            for (int i = 0; i < y.nk; ++i) {
                const int c = min(64 * i + ln, y.cend[3] - 1);
                const bool in1 = c >= ce0, in2 = c >= ce1, in3 = c >= ce2;
                const int first = pick4(in1, in2, in3, 0, ce0, ce1, ce2);
                const int rb = pick4(in1, in2, in3, rb0, rb1, rb2, rb3);
                const unsigned char* base = pick4(in1, in2, in3, kb0, kb1, kb2, kb3);
                const int lc = min(c - first, ntok * rb / 16 - 1);
                dma16(base + static_cast<int64_t>(t) * rb + 16 * lc, kdst + 1024 * i);
            }
        };
        auto dma_v = [&](int t, int ntok) {
            const int ln = fresh(lane);
#pragma unroll
            for (int i = 0; i < kNV; ++i) {
                const int c = min(64 * i + ln, kVChunks - 1);
                const bool in1 = c >= D, in2 = c >= D + 8 * kVG;
                const int64_t row = static_cast<int64_t>(t) * pick3(in1, in2, D / 4, 2 * kVG, 2 * kVG);
                const int lc = min(c - pick3(in1, in2, 0, D, D + 8 * kVG), (in1 ? ntok * kVG / 8 : ntok * D / 64) - 1);
                dma16(pick3(in1, in2, vcode, vscale, vmin) + row + 16 * lc, vdst + 1024 * i);
            }
        };
        if (t_lo < t_hi) {
            dma_k(t_lo, min(kRun, t_hi - t_lo));
            dma_v(t_lo, min(kRun, t_hi - t_lo));
        }

        // ---- Key scales and mins: windows of kWindow groups, the rows of a slot are contiguous ----
        const int kg = L.k_group;
        const int64_t grp0 = tok0 / kg;
        const int kgroups = in_sgpr(L.cap_kgroups);
        auto slot_rows = [&](const uint16_t* a, int width) {  // the (b, h) rows of a tier, from the item's first group
            return in_sgpr(reinterpret_cast<const unsigned char*>(a + bh * width * L.cap_kgroups + grp0));
        };
        const unsigned char *sc0 = slot_rows(L.k_scale[0], L.k_width[0]), *mn0 = slot_rows(L.k_min[0], L.k_width[0]);
        const unsigned char *sc1 = slot_rows(L.k_scale[1], L.k_width[1]), *mn1 = slot_rows(L.k_min[1], L.k_width[1]);
        const unsigned char *sc2 = slot_rows(L.k_scale[2], L.k_width[2]), *mn2 = slot_rows(L.k_min[2], L.k_width[2]);
        int win0 = t_lo / kg, win1 = 0;  // staged groups, relative to the item's first
        constexpr int kBatch = 4;        // positions of a lane loaded at once
        uint64_t ws[kBatch], wm[kBatch];  // kWindow halves each
        auto window_size = [&](int g0) { return min(kWindow, (t_hi - 1) / kg - g0 + 1); };
        auto window_load = [&](int g0, int p0) {
            p0 = fresh(p0);
            const int nw = window_size(g0);
            const bool wide = grp0 + g0 + kWindow <= kgroups;  // past the window's end, but inside the slot's row
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                int tier, rank;
                pos_slot(k1, k2, k3, min(p0 + 64 * k, y.n_int - 1), tier, rank);
                const bool in1 = tier >= 1, in2 = tier >= 2;
                const int live = pick3(in1, in2, cnt0, cnt1, cnt2);
                const int64_t at = 2 * (static_cast<int64_t>(rank) * kgroups + g0);
                typedef const __attribute__((address_space(1))) uint16_t global_u16;
                typedef uint64_t u64_any __attribute__((aligned(2)));
                typedef const __attribute__((address_space(1))) u64_any global_u64;
                global_u16* sp = (global_u16*)(pick3(in1, in2, sc0, sc1, sc2) + at);
                global_u16* mp = (global_u16*)(pick3(in1, in2, mn0, mn1, mn2) + at);
                ws[k] = wm[k] = 0;
                if (rank < live) {
                    if (wide) {
                        ws[k] = *reinterpret_cast<global_u64*>(sp);
                        wm[k] = *reinterpret_cast<global_u64*>(mp);
                    } else {
                        for (int w = 0; w < nw; ++w) {
                            ws[k] |= static_cast<uint64_t>(sp[w]) << (16 * w);
                            wm[k] |= static_cast<uint64_t>(mp[w]) << (16 * w);
                        }
                    }
                }
            }
        };
        auto window_store = [&](int g0, int p0) {
            p0 = fresh(p0);
            const int nw = window_size(g0);
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const int pos = p0 + 64 * k;
                if (pos < y.n_int) {
                    unsigned char* d = smbuf + (pos >> 3) * 32 + (pos & 7) * 2;
#pragma unroll
                    for (int w = 0; w < kWindow; ++w)
                        if (w < nw) {
                            *reinterpret_cast<uint16_t*>(d + 4 * w * y.n_int) = static_cast<uint16_t>(ws[k] >> (16 * w));
                            *reinterpret_cast<uint16_t*>(d + 4 * w * y.n_int + 16) = static_cast<uint16_t>(wm[k] >> (16 * w));
                        }
                }
            }
        };
        // the loaded positions, then any past the first 64 * kBatch
        auto window_finish = [&](int g0) {
            window_store(g0, lane);
            for (int p0 = lane + 64 * kBatch; p0 - lane < y.n_int; p0 += 64 * kBatch) {
                window_load(g0, p0);
                window_store(g0, p0);
            }
            win0 = g0;
            win1 = g0 + window_size(g0);
        };
        if (y.n_int > 0 && t_lo < t_hi) window_load(win0, lane);

        // ---- q in the K dimension's order, log2 domain ----
        for (int pos = tid; pos < y.n_pos; pos += kThreads) {
            float v[kRows];
#pragma unroll
            for (int i = 0; i < kRows; ++i) v[i] = 0.f;
            const int c = pos == tid ? channel0 : pos_channel(pos);
            if (c >= 0) {
                const int64_t at = (static_cast<int64_t>(b) * A.n_q + h * p.g + row0) * D + c;
                if (A.q_dtype == LF_FP32) {
#pragma unroll
                    for (int i = 0; i < kRows; ++i) v[i] = static_cast<const float*>(A.query)[at + D * min(i, g - 1)];
                } else {
                    uint16_t x[kRows];
#pragma unroll
                    for (int i = 0; i < kRows; ++i) x[i] = static_cast<const uint16_t*>(A.query)[at + D * min(i, g - 1)];
#pragma unroll
                    for (int i = 0; i < kRows; ++i) v[i] = A.q_dtype == LF_BF16 ? bf16_to_f32(x[i]) : f16_to_f32(x[i]);
                }
            }
#pragma unroll
            for (int i = 0; i < kRows; ++i) qs[((pos >> 2) * kRows + i) * 4 + (pos & 3)] = i < g ? v[i] * p.qscale : 0.f;
        }
        __syncthreads();

        // ---- per-lane state: query row n % 8, half n / 8 of the run ----
        float m = -__builtin_inff(), l = 0.f, cmin[kVG], cmid[kVG];
        float4v o[2][kTiles];  // by half of the run's tokens
#pragma unroll
        for (int v = 0; v < kVG; ++v) { cmin[v] = 0.f; cmid[v] = 0.f; }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int j = 0; j < kTiles; ++j) o[u][j] = float4v{0.f, 0.f, 0.f, 0.f};
        const int row = n & 7;
        const bool second = n >= 8;
        const CodeTable kt = key_table(), vt = value_table();
        if (y.n_int > 0 && t_lo < t_hi) window_finish(win0);

        for (int t = t_lo; t < t_hi; t += kRun) {
            const int ntok = min(kRun, t_hi - t);
            const int ga = t / kg, gb = ntok > 32 ? (t + 32) / kg : ga;  // groups of the two 32-token halves
            const unsigned char* sm = smbuf + ((second ? gb : ga) - win0) * y.n_int * 4 + 32 * q4;

            // ---- scores ----
            wait_dma<kNV>();  // the Key rows have landed (the Value rows may still be in flight)
            float4v acc[4];
#pragma unroll
            for (int T = 0; T < 4; ++T) acc[T] = float4v{0.f, 0.f, 0.f, 0.f};
            float bias = 0.f;
            const bool full = ntok > 32;

            auto load_q = [&](int step, float (&qv)[8]) {
                const float4v x = *reinterpret_cast<const float4v*>(qs + (((step * 4 + q4) * 2 + 0) * kRows + row) * 4);
                const float4v z = *reinterpret_cast<const float4v*>(qs + (((step * 4 + q4) * 2 + 1) * kRows + row) * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) { qv[e] = x[e]; qv[4 + e] = z[e]; }
            };
            // one K-step of an integer tier: code(T) unpacks token tile T's operand
            auto int_step = [&](int step, auto&& code) {
                float qv[8], x[8];
                load_q(step, qv);
                const u32x4 sc = *reinterpret_cast<const u32x4*>(sm + 128 * step);
                const u32x4 mn = *reinterpret_cast<const u32x4*>(sm + 128 * step + 16);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    x[e] = qv[e] * f16_to_f32(static_cast<uint16_t>(sc[e >> 1] >> (16 * (e & 1))));
                    bias = fmaf(qv[e], f16_to_f32(static_cast<uint16_t>(mn[e >> 1] >> (16 * (e & 1)))), bias);
                }
                const Split3 B = split3(x);
                bf16x8 a[4];
#pragma unroll
                for (int T = 0; T < 4; ++T) a[T] = code(T);
                mfma3x4(a, B, acc);
            };
            int step = 0;
            for (int j = 0; j < y.kst[0]; j += 2, step += 2) {
                uint32_t w[4];
                const unsigned char* src = buf + n * rb0 + 4 * (2 * j + q4);
#pragma unroll
                for (int T = 0; T < 4; ++T) w[T] = *reinterpret_cast<const uint32_t*>(src + 16 * T * rb0);
                int_step(step, [&](int T) { return codes8(__builtin_amdgcn_perm(w[T], w[T], 0x01010000u), kt); });
                int_step(step + 1, [&](int T) { return codes8(__builtin_amdgcn_perm(w[T], w[T], 0x03030202u), kt); });
            }
            for (int j = 0; j < y.kst[1]; ++j, ++step) {
                const unsigned char* src = buf + 16 * ce0 + n * rb1 + 4 * (4 * j + q4);
                uint32_t w[4];
#pragma unroll
                for (int T = 0; T < 4; ++T) w[T] = *reinterpret_cast<const uint32_t*>(src + 16 * T * rb1);
                int_step(step, [&](int T) {
                    const uint32_t e = w[T] & 0x0f0f0f0fu, d = (w[T] >> 4) & 0x0f0f0f0fu;
                    return as_bf16x8(upper_pair(byte_f32<0>(e), byte_f32<1>(e)), upper_pair(byte_f32<2>(e), byte_f32<3>(e)),
                                     upper_pair(byte_f32<0>(d), byte_f32<1>(d)), upper_pair(byte_f32<2>(d), byte_f32<3>(d)));
                });
            }
            for (int j = 0; j < y.kst[2]; ++j, ++step) {
                const unsigned char* src = buf + 16 * ce1 + n * rb2 + 8 * (4 * j + q4);
                uint32_t w[4][2];
#pragma unroll
                for (int T = 0; T < 4; ++T) {
                    const uint32_t* at = reinterpret_cast<const uint32_t*>(src + 16 * T * rb2);
                    w[T][0] = at[0];
                    w[T][1] = at[1];
                }
                int_step(step, [&](int T) {
                    const uint32_t e = w[T][0], d = w[T][1];
                    return as_bf16x8(upper_pair(byte_f32<0>(e), byte_f32<1>(e)), upper_pair(byte_f32<2>(e), byte_f32<3>(e)),
                                     upper_pair(byte_f32<0>(d), byte_f32<1>(d)), upper_pair(byte_f32<2>(d), byte_f32<3>(d)));
                });
            }
            if (y.kst[3] > 0) {
                const unsigned char* base = buf + 16 * ce2;
                const int w16 = L.k_width[3];
                auto half_step = [&](int j, auto ne) {
                    // elements the lane groups hold in this step: values past the tier read as 0
                    constexpr int kNe = decltype(ne)::value;
                    uint16_t raw[4][kNe];
                    uint32_t bad = 0;
#pragma unroll
                    for (int T = 0; T < 4; ++T)
#pragma unroll
                        for (int e = 0; e < kNe; ++e)
                            raw[T][e] = reinterpret_cast<const uint16_t*>(base)[(16 * T + n) * w16 + min(32 * j + 4 * e + q4, w16 - 1)];
#pragma unroll
                    for (int T = 0; T < 4; ++T)
#pragma unroll
                        for (int e = 0; e < kNe; ++e) {
                            if (32 * j + 4 * e + q4 >= w16 || 16 * T >= ntok) raw[T][e] = 0;
                            bad |= (raw[T][e] & 0x7c00u) == 0x7c00u;
                        }
                    if (__builtin_expect(__any(bad != 0), 0)) {
                        // the parts of an infinity do not add up to it: this step in fp32 FMAs
                        for (int r = 32 * j; r < min(32 * j + 32, cnt3); ++r) {
                            const int pos = y.n_int + 32 * j + 8 * (r & 3) + ((r & 31) >> 2);
                            const float qv = qs[((pos >> 2) * kRows + row) * 4 + (pos & 3)];
#pragma unroll
                            for (int T = 0; T < 4; ++T)
#pragma unroll
                                for (int i = 0; i < 4; ++i)
                                    if (16 * T < ntok) acc[T][i] = fmaf(qv, f16_to_f32(reinterpret_cast<const uint16_t*>(base)[(16 * T + 4 * q4 + i) * w16 + r]), acc[T][i]);
                        }
                        return;
                    }
                    float qv[8];
                    load_q(step + j, qv);
                    const Split3 B = split3(qv);
                    bf16x8 ah[4], al[4];
#pragma unroll
                    for (int T = 0; T < 4; ++T) {
                        // 11 significant bits: two parts
                        uint32_t hi[4] = {}, lo[4] = {};
#pragma unroll
                        for (int k = 0; k < kNe / 2; ++k) {
                            const float u = f16_to_f32(raw[T][2 * k]), v = f16_to_f32(raw[T][2 * k + 1]);
                            hi[k] = upper_pair(fbits(u), fbits(v));
                            lo[k] = upper_pair(fbits(u - __uint_as_float(fbits(u) & 0xffff0000u)),
                                               fbits(v - __uint_as_float(fbits(v) & 0xffff0000u)));
                        }
                        al[T] = as_bf16x8(lo[0], lo[1], lo[2], lo[3]);
                        ah[T] = as_bf16x8(hi[0], hi[1], hi[2], hi[3]);
                    }
                    mfma3x4(al, B, acc);
                    mfma3x4(ah, B, acc);
                };
                for (int j = 0; j < y.kst[3]; ++j) {
                    if (w16 - 32 * j <= 8) half_step(j, std::integral_constant<int, 2>{});
                    else half_step(j, std::integral_constant<int, 8>{});
                }
            }
            bias = rows_sum(bias);

            wait_dma<0>();  // the Value rows have landed; the Key rows are read
            bool more = false;  // the next run needs the next window
            if (t + kRun < t_hi) {
                const int next = min(kRun, t_hi - t - kRun);
                dma_k(t + kRun, next);
                more = y.n_int > 0 && (t + kRun + next - 1) / kg >= win1;
                if (more) window_load((t + kRun) / kg, lane);
            }

            // ---- online softmax of this lane's stream: tokens 32 second + 16 k + 4 q4 + i ----
            float s[8], mx = -__builtin_inff();
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x = second ? acc[2 + (e >> 2)][e & 3] : acc[e >> 2][e & 3];
                s[e] = second && !full ? -__builtin_inff() : x + bias;
                mx = fmaxf(mx, s[e]);
            }
            // the reference point moves only when a score exceeds it by more than 8 (log2)
            if (__any(mx > m + 8.f || m == -__builtin_inff())) {
                const float mnew = fmaxf(m, rows_max(mx));
                const float alpha = mnew == m ? 1.f : __builtin_amdgcn_exp2f(m - mnew);
                m = mnew;
                l *= alpha;
#pragma unroll
                for (int v = 0; v < kVG; ++v) { cmin[v] *= alpha; cmid[v] *= alpha; }
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int j = 0; j < kTiles; ++j) o[u][j] *= alpha;
            }
            const float mref = m == -__builtin_inff() ? 0.f : m;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                s[e] = __builtin_amdgcn_exp2f(s[e] - mref);
                l += s[e];
            }

            // ---- Values ----
            const unsigned char* vs_l = vbuf + 16 * D;
            const unsigned char* vm_l = vs_l + 128 * kVG;
#pragma unroll
            for (int v = 0; v < kVG; ++v) {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int tok = 32 * (second ? 1 : 0) + 16 * (e >> 2) + 4 * q4 + (e & 3);
                    x[e] = s[e] * f16_to_f32(reinterpret_cast<const uint16_t*>(vs_l)[tok * kVG + v]);
                    cmin[v] = fmaf(s[e], f16_to_f32(reinterpret_cast<const uint16_t*>(vm_l)[tok * kVG + v]), cmin[v]);
                    cmid[v] += x[e];
                }
                const Split3 B = split3(x);
                // lane n holds channels 16 (n % G) + (n / G) G + j of the group, j = 0 .. G - 1
                const unsigned char* src = vbuf + (v * G + n % G) * 4;
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    // the lane's codes of its 8 tokens of half u: the bytes that hold them
                    uint32_t c[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const unsigned char* at = src + (32 * u + 16 * (e >> 2) + 4 * q4 + (e & 3)) * (D / 4);
                        if constexpr (G <= 4) c[e] = at[2 * G * (n / G) / 8];
                        else if constexpr (G == 8) c[e] = *reinterpret_cast<const uint16_t*>(at + 2 * (n / G));
                        else c[e] = *reinterpret_cast<const uint32_t*>(at);
                    }
                    constexpr int kBytes = G <= 4 ? 1 : G / 4, kPer = G <= 4 ? G : 4;  // bytes of codes, tiles per byte
#pragma unroll
                    for (int by = 0; by < kBytes; ++by) {
                        uint32_t w[4];  // two tokens' byte, each twice
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            w[k] = __builtin_amdgcn_perm(c[2 * k + 1], c[2 * k], 0x04040000u + 0x01010101u * by);
                            if constexpr (G < 4) w[k] >>= 2 * G * (n / G) % 8;
                        }
#pragma unroll
                        for (int j = 0; j < kPer; ++j) {
                            float4v& acc_o = o[u][v * G + kPer * by + j];
                            acc_o = mfma3(as_bf16x8(code_pair(w[0] >> (2 * j), vt), code_pair(w[1] >> (2 * j), vt),
                                                    code_pair(w[2] >> (2 * j), vt), code_pair(w[3] >> (2 * j), vt)), B, acc_o);
                        }
                    }
                }
            }
            if (more) window_finish((t + kRun) / kg);
            if (t + kRun < t_hi) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the Value rows are read
                dma_v(t + kRun, min(kRun, t_hi - t - kRun));
            }
        }

        // ---- the wave's two streams per row, in [row][channel] order ----
        l = rows_sum(l);
#pragma unroll
        for (int v = 0; v < kVG; ++v) cmin[v] = rows_sum(fmaf(1.5f, cmid[v], cmin[v]));
        __syncthreads();  // every wave is done with its buffers
        const int stream = 2 * wave + (second ? 1 : 0);
        float* slot = slots + (stream * kRows + row) * kLd;
#pragma unroll
        for (int v = 0; v < kVG; ++v)
#pragma unroll
            for (int j = 0; j < G; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = 4 * q4 + i;
                    slot[16 * (v * G + r % G) + (r / G) * G + j] = (second ? o[1] : o[0])[v * G + j][i] + cmin[v];
                }
        if (q4 == 0) {
            stat[row * kStreams + stream] = m;
            stat[(kRows + row) * kStreams + stream] = l;
        }
        __syncthreads();
        merge(std::integral_constant<int, kStreams>{});
        if (kind != 0) __syncthreads();  // the residual reuses the slots
    }

    if (kind != 0) {
        residual_pass<D>(tp, b, h, row0, g, slots, stat, tid);
        __syncthreads();
        merge(std::integral_constant<int, kWaves>{});
        if (A.commit_new && blockIdx.z == 0) commit_new_rows(p, b, h, tid, kThreads);
    }

#pragma unroll
    for (int k = 0; k < kEl; ++k) {
        const int e = tid + kThreads * k, row = e / D, c = e % D;
        if (row >= g) continue;
        float* r = part_rec(p, part_slot, h, row0 + row);
        r[c] = om[k];
        if (c == 0) { r[D] = Mm[k]; r[D + 1] = Lm[k]; }
    }
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

// LDS of a workgroup for this layer; false when the layout is outside this kernel.  Every layout inside goes to
// it: 4 500 drawn calls (any page, Key and Value group, 1 to 16 sequences of 40 to 8 000 tokens, 1 to 17 new
// tokens, all row types) take 1 / 2.0 to 1 / 43 of the general kernel's time at head_dim 64, 1 / 2.6 to 1 / 49
// at 128 and 1 / 2.6 to 1 / 81 at 256.
bool plan_tiled(const lf_packed_layer& L, TiledLayout& y) {
    const int D = L.head_dim;
    if (D != 64 && D != 128 && D != 256) return false;
    if (L.page_size % 32 || L.k_group % 32 || L.cap_tokens % 32) return false;
    if (L.bit_v != 2 || L.v_group < 16 || L.v_group > D || (L.v_group & (L.v_group - 1))) return false;
    for (int t = 0; t < 3; ++t)
        if (L.k_width[t] && !aligned16(L.k_code[t])) return false;
    if (L.k_width[3] && !aligned16(L.k_value16)) return false;
    if (!aligned16(L.v_code) || !aligned16(L.v_scale) || !aligned16(L.v_min)) return false;
    y.kst[0] = 2 * ((L.k_words[0] + 3) / 4);
    y.kst[1] = (L.k_words[1] + 3) / 4;
    y.kst[2] = (L.k_words[2] + 7) / 8;
    y.kst[3] = (L.k_width[3] + 31) / 32;
    y.n_int = 32 * (y.kst[0] + y.kst[1] + y.kst[2]);
    y.n_pos = y.n_int + 32 * y.kst[3];
    int c = 0;
    for (int t = 0; t < 4; ++t) {
        y.rb[t] = t < 3 ? 4 * L.k_words[t] : 2 * L.k_width[3];
        c += kRun * y.rb[t] / 16;
        y.cend[t] = c;
    }
    if (c == 0) return false;
    y.nk = (c + 63) / 64;
    // A lane reads whole K-steps of a row, past the row's own words and, in the last rows, past
    // its tier's region: at most 16 * 8 bytes, kept inside the wave's buffer by the Value rows
    // that follow the Key rows (1 KB or more).
    const int vg = D / L.v_group;
    const int nv = (D + 16 * vg + 63) / 64;
    y.sm_off = 1024 * (y.nk + nv);
    y.wave_bytes = y.sm_off + kWindow * y.n_int * 4;
    y.off_stat = 0;
    y.off_q = 2 * kStreams * kRows * 4;
    y.off_buf = y.off_q + y.n_pos * kRows * 4;
    // merge slots, q by channel and probabilities of the residual pass, over the wave buffers
    const int alias = (kStreams * (D + 1) + D + kWaves * 32) * kRows * 4;
    y.lds_bytes = y.off_buf + std::max(kWaves * y.wave_bytes, alias);
    return y.lds_bytes <= 160 * 1024;
}

template <int D, int G>
int launch_tiled_dg(const TiledParams& tp, hipStream_t stream) {
    const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(&decode_tiled_kernel<D, G>), tp.y.lds_bytes);
    if (rc != LF_OK) return rc;
    const dim3 grid(tp.p.L.n_kv, tp.p.A.n_work, (tp.p.g + kRows - 1) / kRows);
    hipLaunchKernelGGL((decode_tiled_kernel<D, G>), grid, dim3(kThreads), tp.y.lds_bytes, stream, tp);
    return LF_OK;
}

template <int D>
int launch_tiled_d(const TiledParams& tp, hipStream_t stream) {
    switch (tp.p.L.v_group / 16) {
        case 1: return launch_tiled_dg<D, 1>(tp, stream);
        case 2: return launch_tiled_dg<D, 2>(tp, stream);
        case 4: return launch_tiled_dg<D, 4>(tp, stream);
        case 8: if constexpr (D >= 128) return launch_tiled_dg<D, 8>(tp, stream); break;
        case 16: if constexpr (D >= 256) return launch_tiled_dg<D, 16>(tp, stream); break;
    }
    return LF_E_UNSUPPORTED;
}

bool serves(const DecodeParams& p, TiledLayout& y) {
    return plan_tiled(p.L, y) && p.A.n_work <= 65535 && (p.g + kRows - 1) / kRows <= 65535;
}

}  // namespace

bool decode_tiled_serves(const DecodeParams& p) {
    TiledLayout y;
    return serves(p, y);
}

int launch_decode_tiled(const DecodeParams& p, hipStream_t stream, bool* handled) {
    TiledParams tp;
    tp.p = p;
    *handled = serves(p, tp.y);
    if (!*handled) return LF_OK;
    const bool has_tail = p.A.tail_cap > 0, has_new = p.A.k_new != nullptr;
    tp.res_vec = (!has_tail || (aligned16(p.A.tail_k) && aligned16(p.A.tail_v))) &&
                 (!has_new || (aligned16(p.A.k_new) && aligned16(p.A.v_new))) &&
                 (!has_tail || !has_new || p.A.tail_dtype == p.A.new_dtype);
    tp.inline_work = p.A.work_host != nullptr && p.A.n_work <= LF_INLINE_WORK;
    if (tp.inline_work) std::memcpy(tp.work_inline, p.A.work_host, sizeof(int32_t) * 4 * p.A.n_work);
    const int D = p.L.head_dim;
    const int rc = D == 64 ? launch_tiled_d<64>(tp, stream) : D == 128 ? launch_tiled_d<128>(tp, stream) : launch_tiled_d<256>(tp, stream);
    if (rc != LF_OK) return rc;
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return static_cast<int>(err);
    return launch_decode_reduce(p, stream);
}

}  // namespace lf
