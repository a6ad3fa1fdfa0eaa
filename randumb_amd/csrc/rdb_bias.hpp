// Gradient of a pseudorandom bias from a small dy, in blocks that every launch may carry (rdb_noise.hip says what it computes).
#pragma once
#include "rdb_tile.hpp"
#include <algorithm>

namespace rdb {

constexpr int BIAS_M = 4;   // coefficients to a block
__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return bf16_to_f32(v); }

// What a block of the gradient does with a column's sum g (block b: coefficients b * BIAS_M .. + 3; the block behind the last
// coefficient: the scale), and at the end with its threads' shares (sh: BIAS_M * THREADS / 64 floats).
__device__ __forceinline__ void bias_contract(float (&acc)[BIAS_M], float g, uint32_t o, int64_t m0, bool scale, uint32_t seed)
{
    if (scale) {
        acc[0] = fmaf(g, noise1d(o, seed), acc[0]);
    } else {
        const uint32_t f = sq5_first(o, (uint32_t)m0, seed);
#pragma unroll
        for (int j = 0; j < BIAS_M; ++j) acc[j] = fmaf(g, sq5_unit(sq5_tail(f + (uint32_t)j * SQ5_N1)), acc[j]);
    }
}
template <int THREADS> __device__ __forceinline__ void bias_finish(float (&acc)[BIAS_M], float *dcoef, float *ds, int64_t m0, int64_t k, bool scale, float *sh)
{
    constexpr int WAVES = THREADS / 64;
#pragma unroll
    for (int j = 0; j < BIAS_M; ++j) {
#pragma unroll
        for (int w = 32; w >= 1; w >>= 1) acc[j] += __shfl_xor(acc[j], w);
        if ((threadIdx.x & 63) == 0) sh[j * WAVES + (threadIdx.x >> 6)] = acc[j];
    }
    __syncthreads();
    const int j = threadIdx.x;
    if (j >= BIAS_M) return;
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; w += 4) v += (sh[j * WAVES + w] + sh[j * WAVES + w + 1]) + (sh[j * WAVES + w + 2] + sh[j * WAVES + w + 3]);
    if (scale) {
        if (j == 0) ds[0] = v;
    } else if (m0 + j < k) {
        dcoef[m0 + j] = v;
    }
}

// The whole gradient in one launch, for a dy so small that every block may read it: blocks of 1024 threads, as many of them side by side
// on a column's rows as its outputs leave room for, sixteen rows in flight each.  3.3 us and 1.3 for every sixteen rows of a thread, against
// 8.2 (and a launch more on the host) for the two: 128 rows x 256 5.9, 128 x 10 4.6, 512 x 128 8.5; 250 x 262, six turns, 11.0.  Only while a
// compute unit has one block, which reads all of dy, whichever gradients are wanted (512 x 128: k = 1016 8.7, 1024 13.2, 4096 29.5, 16384 94, and the two
// launches there 6.0, 6.0, 6.3 and 10 behind one another).
constexpr int64_t BIAS_DIRECT_BYTES = 256 << 10, BIAS_DIRECT_TURNS = 4;
constexpr int BIAS_AHEAD = 16;
struct BiasGrad {
    float *dcoef, *ds;   // NULL where not wanted
    const void *dy;
    int64_t ldy, k;
    int rows, n, bf16;
    uint32_t seed;
    int blocks;          // 0: nothing to do
};
inline int bias_wide(int64_t n, int threads) { return n < threads ? (int)cdiv(n, 64) * 64 : threads; }   // threads along the outputs
inline bool bias_direct(int64_t rows, int64_t n, int es, int64_t k, int num_cus, int threads = 1024)
{
    if (rows <= 0 || n <= 0 || rows * n * es > BIAS_DIRECT_BYTES || cdiv(k, BIAS_M) + 1 > num_cus) return false;
    const int wide = bias_wide(n, threads);
    return cdiv(rows, BIAS_AHEAD * (threads / wide)) * cdiv(n, wide) <= BIAS_DIRECT_TURNS;
}
template <typename T, int THREADS> __device__ __forceinline__ void bias_direct_block(const BiasGrad &q, int block, float *sh)
{
    const T *const dy = static_cast<const T *>(q.dy);
    const int64_t m0 = (int64_t)block * BIAS_M;
    const bool scale = !q.dcoef || m0 >= q.k;
    const int wide = q.n < THREADS ? (q.n + 63) / 64 * 64 : THREADS, beside = THREADS / wide, first = (int)threadIdx.x / wide;
    float acc[BIAS_M] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int o = (int)threadIdx.x - first * wide; o < q.n && first < beside; o += wide) {
        float g = 0.0f;
        for (int r0 = first; r0 < q.rows; r0 += BIAS_AHEAD * beside) {
            float v[BIAS_AHEAD];
#pragma unroll
            for (int i = 0; i < BIAS_AHEAD; ++i) v[i] = to_f32(dy[(int64_t)min(r0 + i * beside, q.rows - 1) * q.ldy + o]);   // clamped: loaded, not added
#pragma unroll
            for (int i = 0; i < BIAS_AHEAD; ++i) g += r0 + i * beside < q.rows ? v[i] : 0.0f;
        }
        bias_contract(acc, g, (uint32_t)o, m0, scale, q.seed);
    }
    bias_finish<THREADS>(acc, q.dcoef, q.ds, m0, q.k, scale, sh);
}
int bias_direct_launch(const BiasGrad &q, hipStream_t s);   // rdb_noise.hip

}  // namespace rdb
