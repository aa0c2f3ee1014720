// Dense float32 reconstruction of one sequence's packed history.
//
// Reference: dequantize_key / dequantize_value, src/logitfill/packed/layout.py:132-182
// (restored = code * scale + min with float16 scale/min upcast; the fp16 tier
// upcast as stored).  The product of code and scale and the add of min are
// separately rounded, as in the reference's torch arithmetic.
//
// One workgroup per (run of tokens, kv head, Key or Value).  A Key workgroup turns the head's tier
// tables into a map channel -> (tier, rank) in LDS once; a thread then keeps its V consecutive
// channels (V = 4, a 16-byte store, where head_dim, the pointers and the Value grouping allow it) for
// every token it takes, with their address, shift, scale and min in registers, so an element costs one
// 16-bit load (no code crosses 16 bits, and an fp16 value is 16) and its arithmetic, without a branch.
// Bound: the float32 writes (8 bytes per token and channel against about one read).
// The kernel before it looked each element's channel up in the tier tables by a linear scan, V loads
// and four integer divisions per element: 6 200 tokens x 8 heads x 128 took 279 us, now 26
// (1.9 TB/s of writes; about 10 of them are the launch and the dependent loads before the first store).
#pragma clang fp contract(off)

#include <algorithm>

#include "decode_common.hpp"

namespace lf {
namespace {

struct DequantArgs {
    lf_packed_layer L;
    int b;
    int tokens;
    int run;   // tokens per workgroup
    int both;  // Key and Value: workgroups of each (blockIdx.z & 1)
    float* k_out;
    float* v_out;
    char pad[96];  // (whole lines for prefetch_args)
};
static_assert(sizeof(DequantArgs) > 320 && sizeof(DequantArgs) <= 640, "prefetch_args takes 6 to 10 lines");

constexpr int kThreads = 256;
constexpr int kSlab = 4096;  // channels of a workgroup (its map: 16 KB of LDS)

template <int V>
__device__ __forceinline__ void store_row(float* dst, const float (&x)[V]) {
    if constexpr (V == 4) *reinterpret_cast<float4*>(dst) = float4{x[0], x[1], x[2], x[3]};
    else dst[0] = x[0];
}

// Channels c .. c + V - 1 of tokens t0, t0 + step, ... below t1, for Key or Value.
template <int V>
__device__ __forceinline__ void key_rows(const DequantArgs& a, const uint32_t* map, int c0, int h, int c, int t0, int t1, int step) {
    const lf_packed_layer& L = a.L;
    const int64_t row0 = tok_row(L, a.b, h, 0), bh = static_cast<int64_t>(a.b) * L.n_kv + h;
    // row 0 and the (b, h) rows of the group arrays, per tier
    auto bytes = [](const void* p, int64_t off) { return in_sgpr(static_cast<const unsigned char*>(p) + off); };
    const int w0 = in_sgpr(L.k_words[0]), w1 = in_sgpr(L.k_words[1]), w2 = in_sgpr(L.k_words[2]), w16 = in_sgpr(L.k_width[3]);
    const unsigned char *c_0 = bytes(L.k_code[0], row0 * w0 * 4), *c_1 = bytes(L.k_code[1], row0 * w1 * 4);
    const unsigned char *c_2 = bytes(L.k_code[2], row0 * w2 * 4), *c_3 = bytes(L.k_value16, row0 * w16 * 2);
    const int64_t g0 = bh * L.k_width[0] * L.cap_kgroups * 2, g1 = bh * L.k_width[1] * L.cap_kgroups * 2;
    const int64_t g2 = bh * L.k_width[2] * L.cap_kgroups * 2;
    const unsigned char *s_0 = bytes(L.k_scale[0], g0), *s_1 = bytes(L.k_scale[1], g1), *s_2 = bytes(L.k_scale[2], g2);
    const unsigned char *m_0 = bytes(L.k_min[0], g0), *m_1 = bytes(L.k_min[1], g1), *m_2 = bytes(L.k_min[2], g2);
    const int groups = in_sgpr(L.cap_kgroups);
    // Per channel: the address in row 0 of the 16 bits that hold its code or its fp16 value, the
    // row's stride in bytes, the code's shift, and where its group scales and mins are.  A channel
    // of no tier reads a row of the output and restores 0.
    const unsigned char* base[V];
    const uint16_t *sc[V], *mn[V];
    int stride[V], shift[V];
    uint32_t mask[V];
    bool half[V];
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const uint32_t e = map[c - c0 + k];
        const int t = static_cast<int>(e >> 28), j = static_cast<int>(e & 0xfffffffu);
        half[k] = t == 3;
        const bool live = e != 0xffffffffu, in1 = t >= 1, in2 = t >= 2, in3 = t >= 3;
        const int bits = 2 << (in3 ? 3 : t), bit = j * bits;  // an fp16 value: 16
        shift[k] = bit % 16;
        mask[k] = live && !in3 ? (1u << bits) - 1u : 0u;
        stride[k] = live ? pick4(in1, in2, in3, 4 * w0, 4 * w1, 4 * w2, 2 * w16) : 0;
        base[k] = live ? pick4(in1, in2, in3, c_0, c_1, c_2, c_3) + bit / 16 * 2 : reinterpret_cast<const unsigned char*>(a.k_out);
        const int64_t g = 2 * static_cast<int64_t>(j) * groups;
        sc[k] = live && !in3 ? reinterpret_cast<const uint16_t*>(pick3(in1, in2, s_0, s_1, s_2) + g) : nullptr;
        mn[k] = live && !in3 ? reinterpret_cast<const uint16_t*>(pick3(in1, in2, m_0, m_1, m_2) + g) : nullptr;
    }
    float* out = a.k_out + static_cast<int64_t>(h) * a.tokens * L.head_dim + c;
    float s[V], m[V];
    for (int t = t0; t < t1;) {
        // the tokens of one Key group
        const int g = t / L.k_group, end = min(t1, (g + 1) * L.k_group);
#pragma unroll
        for (int k = 0; k < V; ++k) {
            s[k] = sc[k] ? f16_to_f32(sc[k][g]) : 0.f;
            m[k] = mn[k] ? f16_to_f32(mn[k][g]) : 0.f;
        }
#pragma unroll 4
        for (; t < end; t += step) {
            float x[V];
#pragma unroll
            for (int k = 0; k < V; ++k) {
                const uint16_t raw = *reinterpret_cast<const uint16_t*>(base[k] + static_cast<int64_t>(t) * stride[k]);
                const float prod = static_cast<float>(static_cast<uint32_t>(raw) >> shift[k] & mask[k]) * s[k];
                x[k] = half[k] ? f16_to_f32(raw) : prod + m[k];
            }
            store_row<V>(out + static_cast<int64_t>(t) * L.head_dim, x);
        }
    }
}

template <int V>
__device__ __forceinline__ void value_rows(const DequantArgs& a, int h, int c, int t0, int t1, int step) {
    const lf_packed_layer& L = a.L;
    const int D = L.head_dim;
    const int64_t row0 = tok_row(L, a.b, h, 0);
    float* out = a.v_out + static_cast<int64_t>(h) * a.tokens * D + c;
    if (L.bit_v >= 16) {
#pragma unroll 4
        for (int t = t0; t < t1; t += step) {
            float x[V];
            const uint16_t* src = L.v_value16 + (row0 + t) * D + c;
#pragma unroll
            for (int k = 0; k < V; ++k) x[k] = f16_to_f32(src[k]);
            store_row<V>(out + static_cast<int64_t>(t) * D, x);
        }
        return;
    }
    // V = 4: the channels share a word (c is a multiple of 4, a word holds 4, 8 or 16 codes) and,
    // the Value group being a multiple of 4, a scale and min
    const int bits = L.bit_v, per = 32 / bits;
    const int shift = c % per * bits;
    const uint32_t mask = (1u << bits) - 1u;
    const int32_t* code = L.v_code + row0 * L.v_words + c / per;
    const int64_t g0 = row0 * L.v_groups + c / L.v_group;
#pragma unroll 4
    for (int t = t0; t < t1; t += step) {
        const uint32_t w = static_cast<uint32_t>(code[static_cast<int64_t>(t) * L.v_words]) >> shift;
        const int64_t g = g0 + static_cast<int64_t>(t) * L.v_groups;
        const float s = f16_to_f32(L.v_scale[g]), m = f16_to_f32(L.v_min[g]);
        float x[V];
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const float prod = static_cast<float>(w >> (k * bits) & mask) * s;
            x[k] = prod + m;
        }
        store_row<V>(out + static_cast<int64_t>(t) * D, x);
    }
}

template <int V>
__global__ __launch_bounds__(kThreads) void dequant_kernel(DequantArgs a) {
    prefetch_args<sizeof(DequantArgs)>();
    extern __shared__ uint32_t map[];  // [channel - c0]: tier << 28 | rank, all ones: no tier
    const lf_packed_layer& L = a.L;
    const int h = blockIdx.y, tid = threadIdx.x;
    const int z = blockIdx.z, slab = a.both ? z >> 1 : z;
    const bool key = a.both ? (z & 1) == 0 : a.k_out != nullptr;
    const int c0 = slab * kSlab, D = min(kSlab, L.head_dim - c0);  // this slab
    const int t0 = static_cast<int>(blockIdx.x) * a.run, t1 = min(a.tokens, t0 + a.run);
    if (key) {
        const int w0 = L.k_width[0], w1 = w0 + L.k_width[1], w2 = w1 + L.k_width[2], w3 = w2 + L.k_width[3];
        const int n0 = L.k_width[0] ? L.tier_count[0][h] : 0, n1 = L.k_width[1] ? L.tier_count[1][h] : 0;
        const int n2 = L.k_width[2] ? L.tier_count[2][h] : 0, n3 = L.k_width[3] ? L.tier_count[3][h] : 0;
        const int32_t *i0 = in_sgpr(L.tier_index[0] + h * L.k_width[0]), *i1 = in_sgpr(L.tier_index[1] + h * L.k_width[1]);
        const int32_t *i2 = in_sgpr(L.tier_index[2] + h * L.k_width[2]), *i3 = in_sgpr(L.tier_index[3] + h * L.k_width[3]);
        for (int c = tid; c < D; c += kThreads) map[c] = 0xffffffffu;
        __syncthreads();
        // every tier's slots in one pass
        for (int i = tid; i < w3; i += kThreads) {
            const bool in1 = i >= w0, in2 = i >= w1, in3 = i >= w2;
            const int t = in1 + in2 + in3;
            const int j = i - pick4(in1, in2, in3, 0, w0, w1, w2);
            const int c = pick4(in1, in2, in3, i0, i1, i2, i3)[j];  // (with the counts in flight)
            if (j < pick4(in1, in2, in3, n0, n1, n2, n3) && c >= c0 && c < c0 + D) atomicMin(&map[c - c0], static_cast<uint32_t>(t) << 28 | static_cast<uint32_t>(j));
        }
        __syncthreads();
    }
    const int per_tok = D / V;  // threads of a token
    if (per_tok <= kThreads) {
        const int rows = kThreads / per_tok;  // tokens at once
        const int r = tid / per_tok, c = c0 + tid % per_tok * V;
        if (r >= rows) return;
        if (key) key_rows<V>(a, map, c0, h, c, t0 + r, t1, rows);
        else value_rows<V>(a, h, c, t0 + r, t1, rows);
    } else {
        for (int c = c0 + tid * V; c < c0 + D; c += kThreads * V) {
            if (key) key_rows<V>(a, map, c0, h, c, t0, t1, 1);
            else value_rows<V>(a, h, c, t0, t1, 1);
        }
    }
}

}  // namespace

int launch_dequantize(const lf_packed_layer& L, int b, int tokens, float* k_out, float* v_out,
                      hipStream_t stream) {
    // As many tokens a workgroup as make two rounds of five workgroups per CU, Key and Value, in
    // steps of 8, at most 512: one round leaves the last stores without company, more rounds repeat
    // the dependent loads before a workgroup's first store (us at 2 012 and 6 200 tokens x 8 heads x
    // 128, runs of 8 and 32: 20.0 and 25.3; of 32 and 80: 15.0 and 27.5; of 16 and 40: 13.9 and 26.3)
    int run = static_cast<int>(std::min<int64_t>(512, std::max<int64_t>(8, (static_cast<int64_t>(tokens) * L.n_kv * 2 / 2560 + 7) / 8 * 8)));
    while (static_cast<int64_t>(tokens) / run > (1 << 23)) run *= 2;  // the grid's limit
    DequantArgs a{L, b, tokens, run, k_out && v_out, k_out, v_out, {}};
    const bool out16 = ((reinterpret_cast<uintptr_t>(k_out) | reinterpret_cast<uintptr_t>(v_out)) & 15) == 0;
    const bool vec = L.head_dim % 4 == 0 && out16 && (!v_out || L.bit_v >= 16 || L.v_group % 4 == 0);
    const dim3 grid((tokens + run - 1) / run, L.n_kv, (L.head_dim + kSlab - 1) / kSlab * (a.both ? 2 : 1));
    const size_t lds = sizeof(uint32_t) * (L.head_dim < kSlab ? L.head_dim : kSlab);
    if (vec) hipLaunchKernelGGL(dequant_kernel<4>, grid, dim3(kThreads), lds, stream, a);
    else hipLaunchKernelGGL(dequant_kernel<1>, grid, dim3(kThreads), lds, stream, a);
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? LF_OK : static_cast<int>(err);
}

}  // namespace lf
