// Sums over the partial matrices that a product in several ranges of its contraction leaves, in range order whoever computes them.
#pragma once
#include "rdb_tile.hpp"

namespace rdb {

// part[0] + part[stride] + ... in split order, eight loads in flight: one at a time the sum is a chain of `splits` memory latencies
// (4097 tokens x 1001 -> 999 in bf16, k = 100: step 97 -> 91 us, three of these launches)
template <typename V> __device__ __forceinline__ V sum_in_order(const float *__restrict__ part, int64_t stride, int splits)
{
    V v = *reinterpret_cast<const V *>(part);
    for (int s0 = 1; s0 < splits; s0 += 8) {
        V u[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) u[j] = *reinterpret_cast<const V *>(part + (int64_t)min(s0 + j, splits - 1) * stride);   // clamped: loaded, not added
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (s0 + j < splits) v += u[j];
    }
    return v;
}

// out[i] = part[0][i] + part[1][i] + ... in split order, four values per thread (n4 groups of four, then the n % 4 last values
// one thread each); out fp32, or bf16 (rounded once); bias: NULL, or fp32, added to rows of cols values.
struct FgSum {
    void *out;
    const float *part;
    int64_t n, stride;   // values, floats between the partial matrices
    int out_bf16, splits, vec;
    int blocks;          // 0: no such sum
    const float *bias;
    uint32_t cols;
};
// block of q.blocks, of 256 threads
__device__ __forceinline__ void f32_sum_block(const FgSum &q, int block, int thread)
{
    const int64_t i = (int64_t)block * 256 + thread, n4 = q.vec ? q.n / 4 : 0;
    if (i < n4) {
        f32x4 v = sum_in_order<f32x4>(q.part + i * 4, q.stride, q.splits);
        if (q.bias) {
            uint32_t c = (uint32_t)(i * 4) % q.cols;   // n is below 2^29
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[j] += q.bias[c];
                if (++c == q.cols) c = 0;
            }
        }
        if (q.out_bf16) store4<bf16_t>(static_cast<bf16_t *>(q.out) + i * 4, v[0], v[1], v[2], v[3]);
        else *reinterpret_cast<f32x4 *>(static_cast<float *>(q.out) + i * 4) = v;
    } else if (n4 * 4 + (i - n4) < q.n) {
        const int64_t e = n4 * 4 + (i - n4);
        const float v = sum_in_order<float>(q.part + e, q.stride, q.splits) + (q.bias ? q.bias[(uint32_t)e % q.cols] : 0.0f);
        if (q.out_bf16) static_cast<bf16_t *>(q.out)[e] = f32_to_bf16(v);
        else static_cast<float *>(q.out)[e] = v;
    }
}

// dW of a vector-coef layer as its product leaves it: partial matrices, out_f x in_f each, `stride` floats apart
struct VectorDW {
    const float *part;
    int64_t stride;
    int parts;
};
constexpr int VECTOR_DW_PARTS = 8;   // what the contraction with the noise holds on the way
// rdb_f32.hip
int64_t vector_products_workspace(int64_t tokens, int64_t in_f, int64_t out_f, bool want_dx);
int vector_dw_ranges(int64_t tokens, int64_t in_f, int64_t out_f);   // of dW's product without dx beside it; 0: not taken
int vector_products(float *dx, const float *dy, int64_t lddy, const float *x, int64_t ldx, const float *W, int64_t tokens, int64_t in_f, int64_t out_f,
                    void *workspace, FgSum *dx_sum, VectorDW *dw, hipStream_t s);
}  // namespace rdb
