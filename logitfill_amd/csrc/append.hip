// Single-token append to the residual pages, on the device: the one-token commit of a decode
// step (reference src/logitfill/packed/cache.py:48-62 while the page is not full) without a
// host round trip for the write position.  Workgroup b copies sequence b's new Key and Value
// rows of every kv head into row tail_len[b] of its residual page (converted to the residual
// dtype) and then advances tail_len[b]; a full residual page is left untouched (the caller
// flushes full pages before appending).  fill_tail_kernel below is the same for several tokens at
// positions the host knows.
#include <cstring>

#include "lf_common.hpp"

namespace lf {
namespace {

struct AppendArgs {
    void* tail_k;
    void* tail_v;
    int tail_dtype, tail_cap;
    int32_t* tail_len;
    const void* k_new;
    const void* v_new;
    int new_dtype;
    int n_kv, head_dim;
};

__global__ __launch_bounds__(256) void append_token_kernel(AppendArgs a) {
    const int b = blockIdx.x;
    const int row = a.tail_len[b];
    __syncthreads();  // every thread has read the position before thread 0 advances it
    if (row < 0 || row >= a.tail_cap) return;
    const int D = a.head_dim;
    for (int e = threadIdx.x; e < a.n_kv * D; e += blockDim.x) {
        const int h = e / D, c = e - h * D;
        const int64_t src = (static_cast<int64_t>(b) * a.n_kv + h) * D + c;
        const int64_t dst = ((static_cast<int64_t>(b) * a.n_kv + h) * a.tail_cap + row) * D + c;
        store_from_f32(a.tail_k, dst, a.tail_dtype, load_as_f32(a.k_new, src, a.new_dtype));
        store_from_f32(a.tail_v, dst, a.tail_dtype, load_as_f32(a.v_new, src, a.new_dtype));
    }
    if (threadIdx.x == 0) a.tail_len[b] = row + 1;
}

// Rows of new tokens into the residual pages: segment (sequence, first source token, first page
// row, tokens) of a commit, for every kv head, Key and Value, in one launch (a copy each took the
// commit two launches per sequence and fill level).  Bound by the launch for a few sequences, by
// memory for many: 64 sequences x 4 heads x 128 tokens (16.8 MB read, as much written) 9.6 us, 3.5 TB/s.
constexpr int kInlineSegs = 160;

struct FillArgs {
    void* tail[2];            // K, V [batch][n_kv][tail_cap][head_dim]
    const void* src[2];
    int64_t sb[2], sh[2], st[2];  // source strides in elements
    int esize;                // bytes per element
    int tail_cap, n_kv, head_dim;
    int vec;                  // every row starts on 16 bytes and has a whole number of them
    int every;                // 1: segs[0] for every sequence (blockIdx.x)
    int32_t segs[4 * kInlineSegs];
};
static_assert(sizeof(FillArgs) <= 4096, "kernel arguments are limited to 4 KB");

__global__ __launch_bounds__(256) void fill_tail_kernel(FillArgs a) {
    const int seg = a.every ? 0 : blockIdx.x, h = blockIdx.y, w = blockIdx.z;
    const int b = a.every ? static_cast<int>(blockIdx.x) : a.segs[4 * seg];
    const int tok = a.segs[4 * seg + 1], row = a.segs[4 * seg + 2], n = a.segs[4 * seg + 3];
    const int64_t rb = static_cast<int64_t>(a.head_dim) * a.esize;  // bytes of a row
    const int64_t sb = w ? a.sb[1] : a.sb[0], sh = w ? a.sh[1] : a.sh[0], st = w ? a.st[1] : a.st[0];
    const char* src = static_cast<const char*>(w ? a.src[1] : a.src[0]) + (b * sb + h * sh + tok * st) * a.esize;
    char* dst = static_cast<char*>(w ? a.tail[1] : a.tail[0]) + ((static_cast<int64_t>(b) * a.n_kv + h) * a.tail_cap + row) * rb;
    const int64_t step = st * a.esize;  // bytes between source rows
    if (a.vec) {
        const int per = static_cast<int>(rb / 16);
#pragma unroll 4
        for (int i = threadIdx.x; i < n * per; i += 256) {
            const int t = i / per, c = i - t * per;
            *reinterpret_cast<uint4*>(dst + t * rb + 16 * c) = *reinterpret_cast<const uint4*>(src + t * step + 16 * c);
        }
    } else if (a.esize == 2) {
        for (int i = threadIdx.x; i < n * a.head_dim; i += 256) {
            const int t = i / a.head_dim, c = i - t * a.head_dim;
            reinterpret_cast<uint16_t*>(dst + t * rb)[c] = reinterpret_cast<const uint16_t*>(src + t * step)[c];
        }
    } else {
        for (int i = threadIdx.x; i < n * a.head_dim; i += 256) {
            const int t = i / a.head_dim, c = i - t * a.head_dim;
            reinterpret_cast<uint32_t*>(dst + t * rb)[c] = reinterpret_cast<const uint32_t*>(src + t * step)[c];
        }
    }
}

}  // namespace

int launch_fill_tail(void* tail_k, void* tail_v, const void* k_src, const void* v_src, int dtype,
                     const int64_t* k_strides, const int64_t* v_strides, int tail_cap, const int32_t* segs, int n_segs,
                     int every, int n_kv, int head_dim, hipStream_t stream) {
    FillArgs a;
    a.tail[0] = tail_k; a.tail[1] = tail_v;
    a.src[0] = k_src; a.src[1] = v_src;
    a.esize = dtype == LF_FP32 ? 4 : 2;
    bool vec = static_cast<int64_t>(head_dim) * a.esize % 16 == 0;
    for (int w = 0; w < 2; ++w) {
        const int64_t* s = w ? v_strides : k_strides;
        a.sb[w] = s[0]; a.sh[w] = s[1]; a.st[w] = s[2];
        for (int i = 0; i < 3; ++i) vec = vec && s[i] * a.esize % 16 == 0;
        vec = vec && ((reinterpret_cast<uintptr_t>(a.src[w]) | reinterpret_cast<uintptr_t>(a.tail[w])) & 15) == 0;
    }
    a.vec = vec;
    a.tail_cap = tail_cap; a.n_kv = n_kv; a.head_dim = head_dim;
    a.every = every > 0;
    for (int i = 0; i < n_segs; i += kInlineSegs) {
        const int n = n_segs - i < kInlineSegs ? n_segs - i : kInlineSegs;
        std::memcpy(a.segs, segs + 4 * i, sizeof(int32_t) * 4 * n);
        hipLaunchKernelGGL(fill_tail_kernel, dim3(every > 0 ? every : n, n_kv, 2), dim3(256), 0, stream, a);
    }
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? LF_OK : static_cast<int>(err);
}

int launch_append_token(void* tail_k, void* tail_v, int tail_dtype, int tail_cap, int32_t* tail_len,
                        const void* k_new, const void* v_new, int new_dtype, int batch, int n_kv, int head_dim,
                        hipStream_t stream) {
    AppendArgs a{tail_k, tail_v, tail_dtype, tail_cap, tail_len, k_new, v_new, new_dtype, n_kv, head_dim};
    hipLaunchKernelGGL(append_token_kernel, dim3(batch), dim3(256), 0, stream, a);
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? LF_OK : static_cast<int>(err);
}

}  // namespace lf
