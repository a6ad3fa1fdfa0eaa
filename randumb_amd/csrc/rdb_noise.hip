// Noise probes, materialise forward/backward, random-bias gradient and embedding gather for gfx950.
// These are the HBM-facing ops of the pseudorandom tensor (the fused linear kernels live in rdb_linear.hip).
#include "rdb_common.hpp"
#include "rdb_bias.hpp"
#include "rdb_sums.hpp"
#include <algorithm>
#include <type_traits>

namespace rdb {

int num_compute_units();   // rdb_error.hip

constexpr int NT = 256;  // threads per block for every kernel in this file

// =============================================================================================== probes
// out[n*M + m] = noise(PRIME*n + m).  Reference: RandumbTensor.py:78-105.
template <typename IM>   // type of the column index: uint32_t where M < 2^31, else int64_t
__global__ __launch_bounds__(NT) void sq5_fill_2d_kernel(float *__restrict__ out, int64_t N, int64_t M, uint32_t seed)
{
    // No division and no multiplication per element: the first round's value of the thread's first element, first(n, m) =
    // n * PN1 + m * N1 + seed (mod 2^32), then a step of (S / M, S % M) elements with a carry, S = the grid's stride
    const int64_t total = N * M, S = (int64_t)gridDim.x * NT, sn = S / M;
    const IM sm = (IM)(S - sn * M), MM = (IM)M;
    int64_t e = (int64_t)blockIdx.x * NT + threadIdx.x;
    // (the one division: in 32 bits where the operands fit, a fifth of the instructions of the 64-bit one)
    const int64_t n0 = (total < (1ll << 32)) ? (int64_t)((uint32_t)e / (uint32_t)M) : e / M;
    IM m = (IM)(e - n0 * M);
    uint32_t f = sq5_first((uint32_t)n0, (uint32_t)m, seed);
    const uint32_t step = (uint32_t)sn * PN1 + (uint32_t)sm * SQ5_N1, carry = PN1 - (uint32_t)M * SQ5_N1;
    for (; e < total; e += S) {
        out[e] = sq5_unit(sq5_tail(f));
        f += step;
        m += sm;
        if (m >= MM) {
            m -= MM;
            f += carry;
        }
    }
}

// out[n] = noise(n).  Reference: RandumbTensor.py:108-126, 204-232.
__global__ __launch_bounds__(NT) void sq5_fill_1d_kernel(float *__restrict__ out, int64_t N, uint32_t seed)
{
    for (int64_t e = (int64_t)blockIdx.x * NT + threadIdx.x; e < N; e += (int64_t)gridDim.x * NT)
        out[e] = noise1d((uint32_t)e, seed);
}

// =============================================================================================== forward
// Vector-coef materialise / embedding gather: one thread per output element, coef broadcast from LDS, serial fp32 FMA over m (the
// order the reference's CUDA kernel uses, rten.cu:101-104).  Bound by the hash on the vector ALU.
// GATHER = false: a = (n % Q)*sQ + (n / Q)*sP                       (RandumbTensor.py:264)
// GATHER = true : a = idx[n / Q]*Q + n % Q   (Q = rowsize)          (RandumbTensor.py:1029)
// A thread's terms are one chain, four of them hashed side by side, in the order of instructions that lets two waves issue together (sq5_four_terms):
// 768 x 3072 elements, k = 256: 189 -> 171 us; 524288 elements, k = 4096: 681 -> 590 (3.64 Thash/s; one term after the other, as the compiler orders it, 3.15).
// Also measured, before that: the terms as bytes of an 8-bit matrix operand, without conversion and multiplication on the vector ALU
// (v_mfma_i32_16x16x64_i8): 229 us.
constexpr int COEF_CHUNK = 2048;
// Coefficients below this in magnitude: 2^31 times their terms stays finite, and so do sums of them; others (and NaNs) get the factor 2^-31
// term by term.  Without it a term takes two vector instructions less.  A turn of the loop is MAT_UNROLL terms, whose coefficients were read the turn before (turns of
// 8: 43.2 clocks a hash, of 16: 42.2).  What is left of a chunk goes by fours.  The look at the coefficients costs a launch about
// a microsecond, which up to MAT_SHORT terms are not paid back: those get the factor term by term.  768 x 3072 elements, term by term
// and otherwise: k = 8 11.8 and 13.9 us, 23 22.9 and 24.5, 48 41.2 and 42.1, 64 52.9 and 53.6, 96 76.6 and 76.5, 256 194 and 190; 300 x 800
// elements: 48 8.5 both, 64 9.1 and 8.7.
constexpr float MAT_LARGE = 3.777893186295716e22f;   // 2^75
constexpr int MAT_UNROLL = 16;
constexpr int MAT_SHORT = 48;

struct MatVecParams {
    float *out;
    const void *coef, *scale_bias;
    const int64_t *idx;
    int64_t k, Nw, Q, sP, sQ;
    int coef_dtype, narrow, contiguous;   // narrow: element numbers fit 32 bits; contiguous: element n has offset n
    uint32_t seed;
    unsigned blocks;   // of NT / LANES elements
};

// LANES > 1: that many neighbouring lanes share an element, lane l its terms l, l + LANES, .. (then added up across the lanes, nearest
// first): with few elements the chip is not full, and the chain's length is what a launch takes (3072 elements, k = 256: 16.5 ->
// 4 us).  SHORT: at most MAT_SHORT terms.
// fill: the coefficients are not in cs yet, or do not fit all at once; one_factor: what a call that fills it says of them, for those that do not
template <bool GATHER, int LANES, bool SHORT>
__device__ __forceinline__ void materialize_vec_block(const MatVecParams &p, float *__restrict__ cs, unsigned block, bool fill, bool &one_factor)
{
    const int64_t n = ((int64_t)block * NT + threadIdx.x) / LANES;
    const int part = threadIdx.x % LANES;
    const bool live = n < p.Nw;
    uint32_t a = (uint32_t)n;
    if (live && (GATHER || !p.contiguous)) {
        const int64_t r = p.narrow ? (int64_t)((uint32_t)n / (uint32_t)p.Q) : n / p.Q, q = n - r * p.Q;
        a = GATHER ? (uint32_t)(p.idx[r] * p.Q + q) : (uint32_t)(q * p.sQ + r * p.sP);
    }
    uint32_t first = a * PN1 + p.seed + (uint32_t)part * SQ5_N1;  // first-round value for m = part; +N1 per step of m
    float acc = 0.0f;
    int large = 0;   // stays so for the chunks that follow: the sum is large then
    for (int64_t m0 = 0; m0 < p.k; m0 += COEF_CHUNK) {   // a multiple of LANES
        const int cnt = (int)((p.k - m0) < COEF_CHUNK ? (p.k - m0) : COEF_CHUNK);
        if (fill) {
            __syncthreads();
            for (int j = threadIdx.x; j < cnt; j += NT) {
                const float c = load_as_f32(p.coef, p.coef_dtype, m0 + j);
                cs[j] = c;
                large |= !(fabsf(c) < MAT_LARGE);
            }
            if (SHORT) __syncthreads();
            else one_factor = !__syncthreads_or(large);
        }
        if (SHORT || !one_factor) {
            if (live)
                for (int j = part; j < cnt; j += LANES) {
                    acc = fmaf(sq5_unit(sq5_tail_apart(first)), cs[j], acc);
                    first += LANES * SQ5_N1;
                }
            continue;
        }
        if (live) {
            // 2^31 times the sum: the terms' common factor is taken out of the loop (a power of two: the same roundings)
            float sum = acc * 2147483648.0f;
            int j = part;
            if (LANES == 1 && cnt >= MAT_UNROLL) {
                // coefficients are read a turn ahead
                uint32_t at = 0;
                asm("" : "+v"(at));   // an address in a vector register: moving it there costs a slot a read
                auto read = [&](int e) { return *reinterpret_cast<const f32x4 *>(reinterpret_cast<const char *>(cs) + at + e * 4); };
                f32x4 c[MAT_UNROLL / 4];
#pragma unroll
                for (int q = 0; q < MAT_UNROLL / 4; ++q) c[q] = read(q * 4);
                for (; j + MAT_UNROLL <= cnt; j += MAT_UNROLL) {
#pragma unroll
                    for (int q = 0; q < MAT_UNROLL / 4; ++q) {
                        sq5_four_terms(first, sum, c[q]);
                        c[q] = read(MAT_UNROLL + q * 4);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    at += MAT_UNROLL * 4;
                }
            }
            if (LANES == 1)
                for (; j + 4 <= cnt; j += 4) sq5_four_terms(first, sum, *reinterpret_cast<const f32x4 *>(cs + j));
            for (; j < cnt; j += LANES) {
                sum = fmaf((float)(int32_t)sq5_tail_apart(first), cs[j], sum);
                first += LANES * SQ5_N1;
            }
            acc = sum * 4.656612873077392578125e-10f;
        }
    }
#pragma unroll
    for (int w = 1; w < LANES; w *= 2) acc += __shfl_xor(acc, w);
    if (live && part == 0) {
        if (p.scale_bias) acc += load_as_f32(p.scale_bias, p.coef_dtype, 0) * noise1d(a, p.seed);
        p.out[n] = acc;
    }
}
// TURNS: blocks take several turns (p.blocks of them in all); without, the kernel is one turn and nothing else: with the loop around it a short launch, which is all latency, takes
// 0.4 us more (40 x 5 elements, k = 3: 2.2 -> 2.65 us)
template <bool GATHER, int LANES, bool SHORT, bool TURNS>
__device__ __forceinline__ void materialize_vec_turns(const MatVecParams &p, float *__restrict__ cs, unsigned first, unsigned blocks)
{
    bool one_factor = false;
    if constexpr (TURNS) {
        for (unsigned block = first; block < p.blocks; block += blocks)
            materialize_vec_block<GATHER, LANES, SHORT>(p, cs, block, block == first || p.k > COEF_CHUNK, one_factor);
    } else {
        materialize_vec_block<GATHER, LANES, SHORT>(p, cs, first, true, one_factor);
    }
}
template <bool GATHER, int LANES, bool SHORT, bool TURNS> __global__ __launch_bounds__(NT) void materialize_vec_kernel(MatVecParams p)
{
    __shared__ __align__(16) float cs[COEF_CHUNK + MAT_UNROLL];   // reads run a turn ahead
    materialize_vec_turns<GATHER, LANES, SHORT, TURNS>(p, cs, blockIdx.x, TURNS ? gridDim.x : 0);
}
// A weight and its bias, contiguous both: the bias's blocks (16 lanes an element) first.
template <int LANES, bool SHORT, bool TURNS> __global__ __launch_bounds__(NT) void materialize_vec_pair_kernel(MatVecParams weight, MatVecParams bias, unsigned bias_blocks)
{
    __shared__ __align__(16) float cs[COEF_CHUNK + MAT_UNROLL];   // reads run a turn ahead
    if (blockIdx.x < bias_blocks) materialize_vec_turns<false, 16, false, false>(bias, cs, blockIdx.x, 0);
    else materialize_vec_turns<false, LANES, SHORT, TURNS>(weight, cs, blockIdx.x - bias_blocks, TURNS ? gridDim.x - bias_blocks : 0);
}

// Matrix-coef materialise, arbitrary view: one thread per output element (no sharing of noise between rows).
__global__ __launch_bounds__(NT) void materialize_mat_generic_kernel(float *__restrict__ out, const void *__restrict__ coef,
                                                                     int coef_dtype, int64_t k, int64_t row_len,
                                                                     int64_t Nw, int64_t Q, int64_t sP, int64_t sQ,
                                                                     uint32_t seed, const void *__restrict__ scale_bias)
{
    const int64_t n = (int64_t)blockIdx.x * NT + threadIdx.x;
    if (n >= Nw) return;
    const int64_t p = n / Q, q = n - p * Q;
    const int64_t a = q * sQ + p * sP;
    const int64_t o = a / row_len, i = a - o * row_len;
    uint32_t first = (uint32_t)i * PN1 + seed;
    float acc = 0.0f;
    for (int64_t m = 0; m < k; ++m) {
        acc = fmaf(sq5_unit(sq5_tail(first)), load_as_f32(coef, coef_dtype, o * k + m), acc);
        first += SQ5_N1;
    }
    if (scale_bias) acc += load_as_f32(scale_bias, coef_dtype, 0) * noise1d((uint32_t)a, seed);
    out[n] = acc;
}

// Matrix-coef materialise of the base tensor or its transpose: W[o, i] = sum_m C[o, m] * noise(i, m).
// A block owns a 16 (o) x 64 (i) tile and walks m in chunks of 32; the noise chunk is hashed once per block
// and shared by the 16 rows through LDS.  out[o*ooS + i*oiS].
constexpr int MT_O = 16, MT_I = 64, MT_M = 32;
__global__ __launch_bounds__(NT) void materialize_mat_tiled_kernel(float *__restrict__ out, const void *__restrict__ coef,
                                                                   int coef_dtype, int64_t rows, int64_t k, int64_t row_len,
                                                                   int64_t ooS, int64_t oiS, uint32_t seed,
                                                                   const void *__restrict__ scale_bias)
{
    __shared__ float Ns[MT_M][MT_I];
    __shared__ float Cs[MT_O][MT_M + 1];
    const int t = threadIdx.x;
    const int64_t i0 = (int64_t)blockIdx.x * MT_I, o0 = (int64_t)blockIdx.y * MT_O;
    const int il = t % MT_I, og = t / MT_I;  // thread owns column il, rows og*4 .. og*4+3
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int64_t m0 = 0; m0 < k; m0 += MT_M) {
        __syncthreads();
        // hash the noise chunk: Ns[mm][ii] = noise(i0+ii, m0+mm); 2048 values, 8 per thread
#pragma unroll
        for (int r = 0; r < (MT_M * MT_I) / NT; ++r) {
            const int e = r * NT + t;
            const int mm = e / MT_I, ii = e % MT_I;
            Ns[mm][ii] = noise2d((uint32_t)(i0 + ii), (uint32_t)(m0 + mm), seed);
        }
        for (int e = t; e < MT_O * MT_M; e += NT) {
            const int oo = e / MT_M, mm = e % MT_M;
            const int64_t o = o0 + oo, m = m0 + mm;
            Cs[oo][mm] = (o < rows && m < k) ? load_as_f32(coef, coef_dtype, o * k + m) : 0.0f;
        }
        __syncthreads();
#pragma unroll 8
        for (int mm = 0; mm < MT_M; ++mm) {
            const float nv = Ns[mm][il];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] = fmaf(nv, Cs[og * 4 + j][mm], acc[j]);
        }
    }
    const int64_t i = i0 + il;
    if (i >= row_len) return;
    const float sb = scale_bias ? load_as_f32(scale_bias, coef_dtype, 0) : 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t o = o0 + og * 4 + j;
        if (o >= rows) continue;
        float v = acc[j];
        if (scale_bias) v += sb * noise1d((uint32_t)(o * row_len + i), seed);
        out[o * ooS + i * oiS] = v;
    }
}

// =============================================================================================== backward
// ----------------------------------------------------------------------------------------------- sums over elements on the matrix cores
// The gradient's terms noise(a, m) d[a] are summed over the elements a: with a lane per coefficient every term would fetch its d
// and its first-round value from LDS (2.1 - 2.4 Thash/s, as a plain chain or interleaved).  Taken off the vector ALU instead: a
// hashed 32-bit integer is, as it lies in its register, four bytes of an 8-bit matrix operand.  d becomes an integer q of 39 bits
// relative to the largest of the block's span (below 2^-39 of it is dropped; fp32 sums drop more at every addition), in five
// signed base-256 digits, and
//     sum n q = sum over s of 256^s . sum over (element, byte j of n) of byte_j(n) . digit_(s-j)(q)
// is one matrix instruction per 32 elements x 16 coefficients: columns = coefficients, contraction = (element, byte), rows = s (0 .. 7) for
// the lower two bytes of an element and again for the upper two.  Two of a row's four bytes an element are zeros then, always the same, so
// it is the sparse one (v_smfmac_i32_16x16x128_i8), with twice the contraction of the dense one in the same time (16 M elements, k = 256: 1252 -> 1178 us).  The 32-bit sums are exact for up to 2^14 elements; they are put together in fp64 and rounded once.  (Bytes 0 .. 2 of n
// are unsigned where the instruction takes signed ones: n ^ 0x00808080 gives n - 128 (1 + 2^8 + 2^16), and 8421504 . sum q is
// added back.)  13 vector instructions a term and no LDS read: 768 x 3072 elements, k = 256: 250 -> 204 us (2.95 Thash/s), and
// 33 -> 4 for the partial rows' sum; with the order of instructions of sq5_eight_masked, the operands of a step read ahead and those of the
// next 256 elements fetched while these are hashed 208 -> 174 (3.47 Thash/s), 16 M elements 1449 -> 1190.
typedef int q8x4 __attribute__((ext_vector_type(4)));
typedef int q8x8 __attribute__((ext_vector_type(8)));
constexpr double Q_OFFSET = 8421504.0;   // 128 (1 + 2^8 + 2^16)
constexpr uint32_t Q_MASK = 0x00808080u;

// p with which values of at most the magnitude behind `top` (the largest |v| as bits, finite), times 2^p, stay below 2^38
__device__ __forceinline__ int q8_exponent(uint32_t top)
{
    if (top == 0) return 0;
    const int e = (int)(top >> 23);
    return e ? 38 - (e - 126) : 38 - (-117 - __clz((int)top));   // |v| < 2^(e - 126); denormals: 2^(32 - clz - 149)
}
__device__ __forceinline__ double pow2(int p) { return __longlong_as_double((long long)(p + 1023) << 52); }

// q = v 2^p and the eight windows of its digits: byte j of win[s] is digit s - j
__device__ __forceinline__ long long q8_windows(float v, double scale, uint32_t (&win)[8])
{
    const long long q = __double2ll_rn((double)v * scale);
    const unsigned long long w = ((unsigned long long)q + 0x8080808080ull) ^ 0x8080808080ull;
    const uint32_t lo = __builtin_bswap32((uint32_t)w), hi = (uint32_t)(w >> 32) << 24;
    win[7] = hi;
    win[6] = __builtin_amdgcn_alignbyte(lo, hi, 1);
    win[5] = __builtin_amdgcn_alignbyte(lo, hi, 2);
    win[4] = __builtin_amdgcn_alignbyte(lo, hi, 3);
    win[3] = lo;
    win[2] = lo >> 8;
    win[1] = lo >> 16;
    win[0] = lo >> 24;
    return q;
}

// A result's rows are 4 (lane / 16) + j; r and r + 8 belong together.  Lanes 0 .. 31 take the columns of one accumulator, lanes 32 .. 63 those of
// the other; the two halves of a column meet across 16 lanes.
__device__ __forceinline__ double q8_total(const q8x4 &low, const q8x4 &high)
{
    double v = 0.0;
#pragma unroll
    for (int j = 3; j >= 0; --j) {
        const auto s = __builtin_amdgcn_permlane32_swap((uint32_t)low[j], (uint32_t)high[j], false, false);
        v = v * 256.0 + (double)(int)(s[0] + s[1]);
    }
    if (threadIdx.x & 16) v *= 4294967296.0;
    const long long bits = __double_as_longlong(v);
    const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)bits, (uint32_t)bits, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(bits >> 32), (uint32_t)(bits >> 32), false, false);
    return __longlong_as_double(((long long)hi[0] << 32) | lo[0]) + __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}

// Largest |v| (as bits) of the block, and the sum of a 64-bit integer; `scratch` holds four of each.
__device__ __forceinline__ uint32_t block_max_bits(uint32_t v, uint32_t *scratch)
{
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, m, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
    __syncthreads();
    return max(max(scratch[0], scratch[1]), max(scratch[2], scratch[3]));
}
__device__ __forceinline__ double block_sum_ll(long long v, long long *scratch)
{
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
    __syncthreads();
    return (double)(scratch[0] + scratch[1] + scratch[2] + scratch[3]);
}

// ----------------------------------------------------------------------------------------------- column sums
constexpr int BIAS_MAX_CHUNKS = 16;
static int bias_chunks(int64_t rows) { return (int)std::min<int64_t>(BIAS_MAX_CHUNKS, std::max<int64_t>(1, cdiv(rows, 32))); }

// block (bx, by): 64 V columns of a chunk of rows; sh: 256 V floats
template <typename T, int V>
__device__ __forceinline__ void column_sums_block(float *__restrict__ part, const T *__restrict__ dy, int64_t ldy, int64_t rows, int64_t n, int64_t per_chunk, int bx, int by,
                                                  float (*sh)[64 * V])
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t c = ((int64_t)bx * 64 + lane) * V, r0 = (int64_t)by * per_chunk, r1 = r0 + per_chunk < rows ? r0 + per_chunk : rows;
    float sum[V];
#pragma unroll
    for (int j = 0; j < V; ++j) sum[j] = 0.0f;
    if (c < n) {
        constexpr int AHEAD = 8;   // rows in flight
        for (int64_t r = r0 + wave; r < r1; r += 4 * AHEAD) {
            float v[AHEAD][V];
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) {
                const int64_t row = r + 4 * i;
                const bool in = row < r1;
                const T *src = dy + (in ? row : r) * ldy + c;
                if constexpr (V == 1) {
                    v[i][0] = to_f32(src[0]);
                } else {
                    T raw[V];
                    __builtin_memcpy(raw, __builtin_assume_aligned(src, 16), sizeof raw);
#pragma unroll
                    for (int j = 0; j < V; ++j) v[i][j] = to_f32(raw[j]);
                }
#pragma unroll
                for (int j = 0; j < V; ++j) v[i][j] = in ? v[i][j] : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < AHEAD; ++i)
#pragma unroll
                for (int j = 0; j < V; ++j) sum[j] += v[i][j];
        }
    }
#pragma unroll
    for (int j = 0; j < V; ++j) sh[wave][lane * V + j] = sum[j];
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * V; i += NT) {
        const int64_t o = (int64_t)bx * 64 * V + i;
        if (o < n) part[(int64_t)by * n + o] = (sh[0][i] + sh[1][i]) + (sh[2][i] + sh[3][i]);
    }
}
template <typename T, int V> __global__ __launch_bounds__(NT) void column_sums_kernel(float *__restrict__ part, const T *__restrict__ dy, int64_t ldy, int64_t rows, int64_t n,
                                                                                    int64_t per_chunk)
{
    __shared__ float sh[4][64 * V];
    column_sums_block<T, V>(part, dy, ldy, rows, n, per_chunk, blockIdx.x, blockIdx.y, sh);
}

// Vector-coef coefficient gradient / embedding gradient.
//   dcoef[m] = sum_e noise(PRIME*a(e) + m) * d[e],  a(e) = e  or  idx[e / Q]*Q + e % Q.
// A block owns a span of elements, whose digits go through LDS 256 at a time (their scale found in a pass of its own over the span),
// and 16 MT WM coefficients, 16 MT a wave, with WM of the four waves side by side along the coefficients and 4 / WM along the
// elements (few coefficients).  Each block writes 4 / WM partial rows; reduce_rows_kernel adds the rows in a fixed order, so the
// result is reproducible.
// Reference: RandumbTensor.py:304-359 (split-N + relaxed atomics there), 1059-1108.
struct GradVecParams {
    float *partial;
    const void *d;
    const int64_t *idx;
    int64_t k, Nw, span, Q;
    int d_dtype, narrow;
    uint32_t seed;
};
// LAYER: d is the sum of `parts` matrices, fp32, part_stride floats apart; the grid is one-dimensional, mblocks along the coefficients, and behind
// the gradient's blocks come those that add up dx, and those of the column sums of dy (col_x along its columns).  A type of its own: a launch waits for what it is given (an embedding's
// step of 3 x 9 values, k = 3 7.6 us, 7.7 with these)
struct GradLayerParams : GradVecParams {
    int parts, mblocks, main_blocks;
    int64_t part_stride;
    FgSum sum;
    float *col_part;
    const float *dy;
    int64_t lddy, rows, n, per_chunk;
    int col_x, col_vec;
};

template <bool GATHER> __device__ __forceinline__ uint32_t gradvec_offset(const GradVecParams &p, int64_t e)
{
    if (!GATHER) return (uint32_t)e;
    const int64_t j = p.narrow ? (int64_t)((uint32_t)e / (uint32_t)p.Q) : e / p.Q;
    return (uint32_t)(p.idx[j] * p.Q + (e - j * p.Q));
}

template <bool GATHER, int MT, int WM, bool LAYER> __global__ __launch_bounds__(NT) void coef_grad_vec_kernel(std::conditional_t<LAYER, GradLayerParams, GradVecParams> p)
{
    constexpr int WE = 4 / WM, MBLOCK = 16 * MT * WM, LD = NT + 8;   // LD: 16 bytes of padding, so that 16 rows' pieces lie in different banks
    __shared__ __align__(16) unsigned short win[16][LD];   // rows 0 .. 7: the windows' lower halves, 8 .. 15: their upper halves
    __shared__ __align__(16) uint32_t as[NT];
    __shared__ uint32_t tops[4];
    __shared__ long long sums[4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, grp = lane >> 4;
    int bx = blockIdx.x, by = blockIdx.y;
    if constexpr (LAYER) {
        const int b = blockIdx.x;
        if (b >= p.main_blocks + p.sum.blocks) {
            const int c = b - p.main_blocks - p.sum.blocks, cy = c / p.col_x, cx = c - cy * p.col_x;
            if (p.col_vec) column_sums_block<float, 4>(p.col_part, p.dy, p.lddy, p.rows, p.n, p.per_chunk, cx, cy, reinterpret_cast<float (*)[256]>(win));
            else column_sums_block<float, 1>(p.col_part, p.dy, p.lddy, p.rows, p.n, p.per_chunk, cx, cy, reinterpret_cast<float (*)[64]>(win));
            return;
        }
        if (b >= p.main_blocks) {
            f32_sum_block(p.sum, b - p.main_blocks, t);
            return;
        }
        by = b / p.mblocks;
        bx = b - by * p.mblocks;
    }
    constexpr int RAW = LAYER ? VECTOR_DW_PARTS : 1;
    auto raw_d = [&](int64_t e, float (&v)[RAW]) {
        if constexpr (LAYER) {
#pragma unroll
            for (int r = 0; r < RAW; ++r) v[r] = r < p.parts ? static_cast<const float *>(p.d)[r * p.part_stride + e] : 0.0f;   // uniform
        } else {
            v[0] = load_as_f32(p.d, p.d_dtype, e);
        }
    };
    auto sum_d = [&](const float (&v)[RAW]) {   // in range order
        float s = v[0];
        if constexpr (LAYER) {
#pragma unroll
            for (int r = 1; r < RAW; ++r)
                if (r < p.parts) s += v[r];
        }
        return s;
    };
    auto load_d = [&](int64_t e) {
        float v[RAW];
        raw_d(e, v);
        return sum_d(v);
    };
    const int64_t e_begin = (int64_t)by * p.span, e_end = (e_begin + p.span < p.Nw) ? e_begin + p.span : p.Nw;
    const int64_t m_block = (int64_t)bx * MBLOCK, m0 = m_block + (wave % WM) * (16 * MT) + (lane & 15);
    float *row = p.partial + ((int64_t)by * WE + wave / WM) * p.k;
    uint32_t top = 0;
    for (int64_t e = e_begin + t; e < e_end; e += NT) top = max(top, __float_as_uint(load_d(e)) & 0x7fffffffu);
    top = block_max_bits(top, tops);
    if (top >= 0x7f800000u) {   // infinities or NaNs, which have to come out where they belong: a term at a time in fp32
        const int64_t m_end = m_block + MBLOCK < p.k ? m_block + MBLOCK : p.k;
        for (int64_t m = m_block + t; m < m_end; m += NT) {
            float acc = 0.0f;
            for (int64_t e = e_begin; e < e_end; ++e)
                acc = fmaf(noise2d(gradvec_offset<GATHER>(p, e), (uint32_t)m, p.seed), load_d(e), acc);
            for (int r = 0; r < WE; ++r) p.partial[((int64_t)by * WE + r) * p.k + m] = r ? 0.0f : acc;
        }
        return;
    }
    const int ex = q8_exponent(top);
    const double scale = pow2(ex), back = pow2(-ex) * 4.656612873077392578125e-10;
    q8x4 acc[MT];
    uint32_t mterm[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        acc[i] = q8x4{0, 0, 0, 0};
        mterm[i] = (uint32_t)(m0 + i * 16) * SQ5_N1 + p.seed;
    }
    long long q = 0;
    uint32_t mask = Q_MASK;
    asm("" : "+v"(mask));   // stays in a vector register
    const int pairs = lane & 8 ? (int)0xeeeeeeeeu : 0x44444444;   // which two of an element's bytes this lane's row has: 2 and 3, or 0 and 1
    float next_d[RAW];
    uint32_t next_a;
    auto fetch = [&](int64_t e0) {
        const int64_t e = e0 + t;
#pragma unroll
        for (int r = 0; r < RAW; ++r) next_d[r] = 0.0f;   // zero beyond the span, so the tail adds nothing
        next_a = 0;
        if (e < e_end) {
            raw_d(e, next_d);
            next_a = gradvec_offset<GATHER>(p, e);
        }
    };
    fetch(e_begin);
    for (int64_t e0 = e_begin; e0 < e_end; e0 += NT) {
        const float dv = sum_d(next_d);
        const uint32_t a = next_a;
        fetch(e0 + NT);   // while this one is hashed
        uint32_t w[8];
        q += q8_windows(dv, scale, w);
        __syncthreads();
        as[t] = a * PN1;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            win[s][t] = (unsigned short)w[s];
            win[s + 8][t] = (unsigned short)(w[s] >> 16);
        }
        __syncthreads();
        const int steps = (int)((e_end - e0 < NT ? e_end - e0 : NT) + 31) / 32;
        // A step is 32 elements: of the hashed operand, lane group g of a column has 4 g .. 4 g + 3 of each half of them; of the other one, lane group g of a
        // row has 8 g .. 8 g + 7.  A step's operands are read while the one before is hashed.
        auto read = [&](int st, q8x4 &d, q8x4 &f, q8x4 &g) __attribute__((always_inline)) {
            st = min(st, NT / 32 - 1);
            d = *reinterpret_cast<const q8x4 *>(&win[lane & 15][st * 32 + grp * 8]);
            f = *reinterpret_cast<const q8x4 *>(&as[st * 32 + grp * 4]);
            g = *reinterpret_cast<const q8x4 *>(&as[st * 32 + 16 + grp * 4]);
        };
        auto step = [&](const q8x4 &d, const q8x4 &f, const q8x4 &g) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                q8x8 h;
                sq5_eight_masked(f, g, mterm[i], mask, h);
                acc[i] = __builtin_amdgcn_smfmac_i32_16x16x128_i8(d, h, acc[i], pairs, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        q8x4 d0, f0, g0, d1, f1, g1;
        int st = wave / WM;
        read(st, d0, f0, g0);
        for (; st < steps; st += 2 * WE) {
            read(st + WE, d1, f1, g1);
            __builtin_amdgcn_sched_barrier(0);
            step(d0, f0, g0);
            if (st + WE >= steps) break;
            read(st + 2 * WE, d0, f0, g0);
            __builtin_amdgcn_sched_barrier(0);
            step(d1, f1, g1);
        }
    }
    __builtin_amdgcn_s_setprio(0);
    double offset = block_sum_ll(q, sums) * Q_OFFSET;
    if (wave / WM) offset = 0.0;   // once per block
#pragma unroll
    for (int i = 0; i < MT; i += 2) {   // lanes 0 .. 15: tile i, lanes 32 .. 47: tile i + 1
        const double r = (q8_total(acc[i], acc[MT > 1 ? i + 1 : i]) + offset) * back;
        const int64_t m = m0 + (i + (MT > 1 ? lane >> 5 : 0)) * 16;
        if (!(grp & 1) && (MT > 1 || lane < 16) && m < p.k) row[m] = (float)r;
    }
}

// out[c] = sum_r partial[r*cols + c] in a fixed order: 32 columns a block, 32 threads a column that take every 32nd row each (the
// rows of a gradient's thousand blocks: one thread a column took 60 us), their sums added in thread order.
__device__ __forceinline__ void reduce_rows_block(float *__restrict__ out, const float *__restrict__ partial, int64_t rows, int64_t cols, int block)
{
    __shared__ float part[32][33];
    const int cl = threadIdx.x & 31, rg = threadIdx.x >> 5;
    const int64_t c = (int64_t)block * 32 + cl;
    float s = 0.0f;
    if (c < cols) {
#pragma unroll 8
        for (int64_t r = rg; r < rows; r += 32) s += partial[r * cols + c];
    }
    part[rg][cl] = s;
    __syncthreads();
    if (rg || c >= cols) return;
#pragma unroll
    for (int j = 1; j < 32; ++j) s += part[j][cl];
    out[c] = s;
}
__global__ __launch_bounds__(1024) void reduce_rows_kernel(float *__restrict__ out, const float *__restrict__ partial, int64_t rows, int64_t cols)
{
    reduce_rows_block(out, partial, rows, cols, blockIdx.x);
}

// Matrix-coef coefficient gradient: dC[o, m] = sum_i noise(i, m) * dW[o, i].
// A block owns a 16 (o) x 64 (m) tile and walks the whole row in chunks of 32 columns (no split: reproducible).
constexpr int GB_O = 16, GB_M = 64, GB_I = 32;
__global__ __launch_bounds__(NT) void coef_grad_mat_kernel(float *__restrict__ dcoef, const void *__restrict__ dW, int dw_dtype,
                                                           int64_t rows, int64_t k, int64_t row_len, uint32_t seed)
{
    __shared__ float Ns[GB_I][GB_M];
    __shared__ float Ds[GB_O][GB_I + 1];
    const int t = threadIdx.x;
    const int64_t m0 = (int64_t)blockIdx.x * GB_M, o0 = (int64_t)blockIdx.y * GB_O;
    const int ml = t % GB_M, og = t / GB_M;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int64_t i0 = 0; i0 < row_len; i0 += GB_I) {
        __syncthreads();
#pragma unroll
        for (int r = 0; r < (GB_I * GB_M) / NT; ++r) {
            const int e = r * NT + t;
            const int ii = e / GB_M, mm = e % GB_M;
            Ns[ii][mm] = noise2d((uint32_t)(i0 + ii), (uint32_t)(m0 + mm), seed);
        }
        for (int e = t; e < GB_O * GB_I; e += NT) {
            const int oo = e / GB_I, ii = e % GB_I;
            const int64_t o = o0 + oo, i = i0 + ii;
            Ds[oo][ii] = (o < rows && i < row_len) ? load_as_f32(dW, dw_dtype, o * row_len + i) : 0.0f;
        }
        __syncthreads();
#pragma unroll 8
        for (int ii = 0; ii < GB_I; ++ii) {
            const float nv = Ns[ii][ml];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] = fmaf(nv, Ds[og * 4 + j][ii], acc[j]);
        }
    }
    const int64_t m = m0 + ml;
    if (m >= k) return;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t o = o0 + og * 4 + j;
        if (o < rows) dcoef[o * k + m] = acc[j];
    }
}

// Random-bias gradient, stage 1: partial[b] = sum over the block's span of d[e]*noise(e).
// Reference: RandumbTensor.py:399-420.
__global__ __launch_bounds__(NT) void scale_bias_grad_kernel(float *__restrict__ partial, const void *__restrict__ d, int d_dtype,
                                                             int64_t Nw, int64_t span, uint32_t seed)
{
    __shared__ float red[NT];
    const int64_t b = (int64_t)blockIdx.x * span;
    const int64_t e_end = (b + span < Nw) ? b + span : Nw;
    float acc = 0.0f;
    for (int64_t e = b + threadIdx.x; e < e_end; e += NT) acc = fmaf(load_as_f32(d, d_dtype, e), noise1d((uint32_t)e, seed), acc);
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = NT / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// =============================================================================================== host side
static inline int grid_for(int64_t n, int64_t cap = 1 << 20) { return (int)(cdiv(n, NT) < cap ? cdiv(n, NT) : cap); }
static bool dtype_ok(int d) { return d == RDB_F32 || d == RDB_BF16; }

// Coefficients a block of the gradient takes: the fewest of 16, 32, 64, 128 that hold them all (then with fewer waves along them), and
// beyond that 64 or as many of 128 and 256 as leave no block half empty; and the partial rows a block writes.
static int grad_block(int64_t k)
{
    if (k <= 32) return k <= 16 ? 16 : 32;
    const int64_t tiles = cdiv(k, 64);
    return tiles % 4 == 0 ? 256 : tiles % 2 == 0 ? 128 : 64;
}
static int grad_rows(int64_t k) { return k <= 16 ? 4 : k <= 32 ? 2 : 1; }

// splits: partial rows in all
static void split_plan(int64_t Nw, int64_t k, int64_t *splits, int64_t *span)
{
    // about four blocks a compute unit (16 waves), of a multiple of 32 elements, 256 to 2^14 (six of a multiple of 256: 2.1 M elements, k = 256 174 -> 156 us, 0.8 M
    // 77 -> 67; six of a multiple of 32: 160 and 70; three: 172 and 72; 2.4 M 174 each)
    const int64_t mblocks = cdiv(k, grad_block(k));
    int64_t s = cdiv(Nw, NT), want = cdiv(1024, mblocks);
    if (s > want) s = want;
    int64_t sp = cdiv(cdiv(Nw, s < 1 ? 1 : s), 32) * 32;
    if (sp < NT) sp = NT;
    if (sp > (1 << 14)) sp = 1 << 14;
    *span = sp;
    *splits = (cdiv(Nw, sp) > 0 ? cdiv(Nw, sp) : 1) * grad_rows(k);
}

// lanes per element of a tensor of n values by k terms: as many as fill the chip's 8192 wave slots, of 1, 4, 16
static int mat_lanes(int64_t n, int64_t k) { return k < 8 ? 1 : n <= (1 << 15) ? 16 : n <= (1 << 17) ? 4 : 1; }
// as many blocks as are resident at once, which take the elements in turns: their coefficients are read once, and no unit is left with a block more
// than others (blocks in turn -> so: 2.4 M elements, k = 256 173.7 -> 170.5 us; 0.8 M 65.6 -> 62.6; 1.5 M 113.6 -> 107.8; 2.9 M 215.0 -> 210.7; at most 0.5 M: even).  Not
// with few terms, where a turn is short and the loop around it costs more than new blocks do: 0.6 M, k = 9 4.9 us in turn, 5.5 so; 2.4 M, k = 23 25.3, 26.7; 4 M, k = 48 77.9, 82.7, k = 49 79.1, 71.3;
// 16 M, k = 2 33.5, 29.9, k = 7 59.3, 59.9 (a grid's threads stay below 2^32).  Several lanes to an element: few elements.
static unsigned mat_blocks(unsigned all, int lanes, int64_t k) { return lanes > 1 || (k <= MAT_SHORT && all < (1u << 24)) ? all : std::min(all, 8u * (unsigned)num_compute_units()); }
template <class F> static void mat_variant(int lanes, int64_t k, bool turns, F &&f)
{
    auto with_terms = [&](auto lanes_) {
        if (k <= MAT_SHORT) f(lanes_, std::true_type{}, std::false_type{});
        else f(lanes_, std::false_type{}, std::false_type{});
    };
    if (lanes == 16) with_terms(std::integral_constant<int, 16>{});
    else if (lanes == 4) with_terms(std::integral_constant<int, 4>{});
    else if (turns) f(std::integral_constant<int, 1>{}, std::false_type{}, std::true_type{});
    else with_terms(std::integral_constant<int, 1>{});
}
static int launch_materialize_vec(float *out, const void *coef, int coef_dtype, int64_t k, int64_t Nw, int64_t Q, int64_t sP, int64_t sQ, uint32_t seed,
                                  const void *scale_bias, const int64_t *idx, hipStream_t s)
{
    const int lanes = mat_lanes(Nw, k);
    const MatVecParams p = {out, coef, scale_bias, idx, k, Nw, Q, sP, sQ, coef_dtype, Nw < (1ll << 32) && Q < (1ll << 32), sQ == 1 && (sP == Q || Nw == Q), seed,
                            (unsigned)cdiv(Nw * lanes, NT)};
    const unsigned blocks = mat_blocks(p.blocks, lanes, k);
    mat_variant(lanes, k, blocks < p.blocks, [&](auto lanes_, auto short_, auto turns) {
        constexpr int L = decltype(lanes_)::value;
        constexpr bool SHORT = decltype(short_)::value, TURNS = decltype(turns)::value;
        if (idx) materialize_vec_kernel<true, L, SHORT, TURNS><<<blocks, NT, 0, s>>>(p);
        else materialize_vec_kernel<false, L, SHORT, TURNS><<<blocks, NT, 0, s>>>(p);
    });
    return check_launch("materialize_vec_kernel");
}

template <bool GATHER, bool LAYER = false> static void launch_grad_vec(const std::conditional_t<LAYER, GradLayerParams, GradVecParams> &p, dim3 grid, hipStream_t s)
{
    switch (grad_block(p.k)) {
    case 16: coef_grad_vec_kernel<GATHER, 1, 1, LAYER><<<grid, NT, 0, s>>>(p); break;
    case 32: coef_grad_vec_kernel<GATHER, 1, 2, LAYER><<<grid, NT, 0, s>>>(p); break;
    case 64: coef_grad_vec_kernel<GATHER, 1, 4, LAYER><<<grid, NT, 0, s>>>(p); break;
    case 128: coef_grad_vec_kernel<GATHER, 2, 4, LAYER><<<grid, NT, 0, s>>>(p); break;
    default: coef_grad_vec_kernel<GATHER, 4, 4, LAYER><<<grid, NT, 0, s>>>(p); break;
    }
}
static int launch_reduce_rows(float *out, const float *partial, int64_t rows, int64_t cols, hipStream_t s)
{
    reduce_rows_kernel<<<(unsigned)cdiv(cols, 32), 1024, 0, s>>>(out, partial, rows, cols);
    return check_launch("reduce_rows_kernel");
}

// rdb_error.hip, rdb_f32.hip
int num_compute_units();
int materialize_mat_f32(float *out, const void *coef, int coef_dtype, int64_t coef_rows, int64_t k, int64_t row_len, bool transposed, uint32_t seed,
                        const void *scale_bias, int num_cus, hipStream_t s);
int64_t coef_grad_mat_f32_workspace(int64_t coef_rows, int64_t k, int64_t row_len, int num_cus);
int coef_grad_mat_f32(float *dcoef, const void *dW, int dw_dtype, int64_t coef_rows, int64_t k, int64_t row_len, uint32_t seed, void *workspace,
                      int64_t workspace_bytes, int num_cus, hipStream_t s);

}  // namespace rdb

using namespace rdb;

extern "C" int rdb_sq5_fill_2d(float *out, int64_t N, int64_t M, uint32_t seed, void *stream)
{
    if (N < 0 || M < 0) return set_error(RDB_E_SHAPE, "rdb_sq5_fill_2d: negative size N=%lld M=%lld", (long long)N, (long long)M);
    if (N == 0 || M == 0) return RDB_OK;
    if (!out) return set_error(RDB_E_NULL, "rdb_sq5_fill_2d: out is NULL");
    if (M < (1ll << 31)) sq5_fill_2d_kernel<uint32_t><<<grid_for(N * M, 8192), NT, 0, (hipStream_t)stream>>>(out, N, M, seed);
    else sq5_fill_2d_kernel<int64_t><<<grid_for(N * M, 8192), NT, 0, (hipStream_t)stream>>>(out, N, M, seed);
    return check_launch("sq5_fill_2d_kernel");
}

extern "C" int rdb_sq5_fill_1d(float *out, int64_t N, uint32_t seed, void *stream)
{
    if (N < 0) return set_error(RDB_E_SHAPE, "rdb_sq5_fill_1d: negative size N=%lld", (long long)N);
    if (N == 0) return RDB_OK;
    if (!out) return set_error(RDB_E_NULL, "rdb_sq5_fill_1d: out is NULL");
    sq5_fill_1d_kernel<<<grid_for(N, 8192), NT, 0, (hipStream_t)stream>>>(out, N, seed);
    return check_launch("sq5_fill_1d_kernel");
}

extern "C" int rdb_materialize_fwd(float *out, const void *coef, int coef_dtype, int64_t coef_rows, int64_t k, int64_t row_len,
                                   int64_t P, int64_t Q, int64_t sP, int64_t sQ, uint32_t seed, const void *scale_bias,
                                   void *stream)
{
    if (P < 0 || Q < 0 || k < 0 || coef_rows < 0)
        return set_error(RDB_E_SHAPE, "rdb_materialize_fwd: negative size P=%lld Q=%lld k=%lld rows=%lld", (long long)P,
                         (long long)Q, (long long)k, (long long)coef_rows);
    if (!dtype_ok(coef_dtype)) return set_error(RDB_E_DTYPE, "rdb_materialize_fwd: unknown coef dtype %d", coef_dtype);
    const int64_t Nw = P * Q;
    if (Nw == 0) return RDB_OK;
    if (!out || (!coef && k > 0)) return set_error(RDB_E_NULL, "rdb_materialize_fwd: out or coef is NULL");
    if (Nw > ((int64_t)1 << 38)) return set_error(RDB_E_SHAPE, "rdb_materialize_fwd: %lld elements is too many", (long long)Nw);
    hipStream_t s = (hipStream_t)stream;
    if (coef_rows == 0) {
        return launch_materialize_vec(out, coef, coef_dtype, k, Nw, Q, sP, sQ, seed, scale_bias, nullptr, s);
    }
    if (row_len <= 0) return set_error(RDB_E_SHAPE, "rdb_materialize_fwd: matrix-coef needs row_len > 0");
    // every addressed offset must fall inside the (coef_rows, row_len) base tensor
    const int64_t max_a = (P - 1) * sP + (Q - 1) * sQ;
    if (sP < 0 || sQ < 0 || max_a >= coef_rows * row_len)
        return set_error(RDB_E_SHAPE, "rdb_materialize_fwd: view (%lld,%lld)/(%lld,%lld) leaves the (%lld,%lld) base tensor",
                         (long long)P, (long long)Q, (long long)sP, (long long)sQ, (long long)coef_rows, (long long)row_len);
    const bool base = (P == coef_rows && Q == row_len && sP == row_len && sQ == 1);
    const bool transposed = (P == row_len && Q == coef_rows && sP == 1 && sQ == row_len);
    if (base || transposed) {
        // from some tens of millions of multiply-adds on: C . N on the fp32 matrix cores, the noise hashed as an operand
        const int rc = materialize_mat_f32(out, coef, coef_dtype, coef_rows, k, row_len, transposed, seed, scale_bias, num_compute_units(), s);
        if (rc != RDB_E_UNSUPPORTED) return rc;
        dim3 grid((unsigned)cdiv(row_len, MT_I), (unsigned)cdiv(coef_rows, MT_O));
        materialize_mat_tiled_kernel<<<grid, NT, 0, s>>>(out, coef, coef_dtype, coef_rows, k, row_len, base ? row_len : 1,
                                                         base ? 1 : coef_rows, seed, scale_bias);
        return check_launch("materialize_mat_tiled_kernel");
    }
    materialize_mat_generic_kernel<<<(unsigned)cdiv(Nw, NT), NT, 0, s>>>(out, coef, coef_dtype, k, row_len, Nw, Q, sP, sQ, seed,
                                                                         scale_bias);
    return check_launch("materialize_mat_generic_kernel");
}

extern "C" int rdb_materialize_weight_and_bias(float *weight, int64_t n, const float *coef, int64_t k, uint32_t seed, const float *scale, const rdb_pseudo_bias *bias,
                                               int64_t bias_n, void *stream)
{
    const char *who = "rdb_materialize_weight_and_bias";
    if (!bias) return set_error(RDB_E_NULL, "%s: bias is NULL", who);
    if (n < 0 || k < 0 || bias_n < 0 || bias->k < 0 || n > ((int64_t)1 << 38) || bias_n > ((int64_t)1 << 38))
        return set_error(RDB_E_SHAPE, "%s: n=%lld k=%lld, bias n=%lld k=%lld", who, (long long)n, (long long)k, (long long)bias_n, (long long)bias->k);
    if ((n > 0 && (!weight || (!coef && k > 0))) || (bias_n > 0 && (!bias->values || (!bias->coef && bias->k > 0)))) return set_error(RDB_E_NULL, "%s: an output or its coefficients are NULL", who);
    hipStream_t s = (hipStream_t)stream;
    // side by side, but for biases that get another number of lanes
    if (n > 0 && bias_n > 0 && mat_lanes(bias_n, bias->k) == 16) {
        const auto params = [](float *out, const float *c, const float *sc, int64_t terms, int64_t len, uint32_t sd) {
            return MatVecParams{out, c, sc, nullptr, terms, len, len, 0, 1, RDB_F32, len < (1ll << 32), 1, sd, (unsigned)cdiv(len * mat_lanes(len, terms), NT)};
        };
        const MatVecParams w = params(weight, coef, scale, k, n, seed), b = params(bias->values, bias->coef, bias->scale, bias->k, bias_n, bias->seed);
        const int lanes = mat_lanes(n, k);
        const unsigned blocks = mat_blocks(w.blocks, lanes, k);
        mat_variant(lanes, k, blocks < w.blocks, [&](auto lanes_, auto short_, auto turns) {
            materialize_vec_pair_kernel<decltype(lanes_)::value, decltype(short_)::value, decltype(turns)::value><<<b.blocks + blocks, NT, 0, s>>>(w, b, b.blocks);
        });
        return check_launch("materialize_vec_pair_kernel");
    }
    if (n > 0)
        if (int rc = launch_materialize_vec(weight, coef, RDB_F32, k, n, n, 0, 1, seed, scale, nullptr, s)) return rc;
    return bias_n > 0 ? launch_materialize_vec(bias->values, bias->coef, RDB_F32, bias->k, bias_n, bias_n, 0, 1, bias->seed, bias->scale, nullptr, s) : RDB_OK;
}

extern "C" int64_t rdb_materialize_bwd_workspace_bytes(int64_t coef_rows, int64_t k, int64_t row_len, int64_t Nw)
{
    if (coef_rows != 0) return coef_grad_mat_f32_workspace(coef_rows, k, row_len, num_compute_units());   // matrix-coef: the ranges' sums
    if (k <= 0 || Nw <= 0) return 0;
    int64_t splits, span;
    split_plan(Nw, k, &splits, &span);
    return splits > 1 ? splits * k * (int64_t)sizeof(float) : 0;
}

static int coef_grad_vec(float *dcoef, const void *d, int d_dtype, int64_t k, int64_t Nw, int64_t Q, uint32_t seed,
                         const int64_t *idx, void *workspace, int64_t workspace_bytes, hipStream_t s, const char *who)
{
    int64_t splits, span;
    split_plan(Nw, k, &splits, &span);
    float *partial = dcoef;
    if (splits > 1) {
        if (!workspace || workspace_bytes < splits * k * (int64_t)sizeof(float))
            return set_error(RDB_E_WORKSPACE, "%s: workspace of %lld bytes needed, %lld given", who,
                             (long long)(splits * k * sizeof(float)), (long long)workspace_bytes);
        partial = (float *)workspace;
    }
    const dim3 grid((unsigned)cdiv(k, grad_block(k)), (unsigned)(splits / grad_rows(k)));
    const GradVecParams p = {partial, d, idx, k, Nw, span, Q, d_dtype, Nw < (1ll << 32) && Q < (1ll << 32), seed};
    if (idx) launch_grad_vec<true>(p, grid, s);
    else launch_grad_vec<false>(p, grid, s);
    int rc = check_launch("coef_grad_vec_kernel");
    if (rc || splits == 1) return rc;
    return launch_reduce_rows(dcoef, partial, splits, k, s);
}

extern "C" int rdb_materialize_bwd(float *dcoef, const void *dW, int dw_dtype, int64_t coef_rows, int64_t k, int64_t row_len,
                                   int64_t Nw, uint32_t seed, void *workspace, int64_t workspace_bytes, void *stream)
{
    if (k < 0 || Nw < 0 || coef_rows < 0)
        return set_error(RDB_E_SHAPE, "rdb_materialize_bwd: negative size k=%lld Nw=%lld rows=%lld", (long long)k, (long long)Nw,
                         (long long)coef_rows);
    if (!dtype_ok(dw_dtype)) return set_error(RDB_E_DTYPE, "rdb_materialize_bwd: unknown dW dtype %d", dw_dtype);
    if (k == 0) return RDB_OK;
    if (!dcoef) return set_error(RDB_E_NULL, "rdb_materialize_bwd: dcoef is NULL");
    hipStream_t s = (hipStream_t)stream;
    if (coef_rows == 0) {
        if (Nw == 0) {  // empty sum
            return launch_reduce_rows(dcoef, dcoef, 0, k, s);
        }
        if (!dW) return set_error(RDB_E_NULL, "rdb_materialize_bwd: dW is NULL");
        return coef_grad_vec(dcoef, dW, dw_dtype, k, Nw, 1, seed, nullptr, workspace, workspace_bytes, s, "rdb_materialize_bwd");
    }
    if (row_len < 0 || coef_rows * row_len != Nw)
        return set_error(RDB_E_SHAPE, "rdb_materialize_bwd: Nw=%lld is not rows*row_len=%lld*%lld", (long long)Nw,
                         (long long)coef_rows, (long long)row_len);
    if (!dW && Nw > 0) return set_error(RDB_E_NULL, "rdb_materialize_bwd: dW is NULL");
    {   // large enough: dW . N^T on the fp32 matrix cores
        const int rc = coef_grad_mat_f32(dcoef, dW, dw_dtype, coef_rows, k, row_len, seed, workspace, workspace_bytes, num_compute_units(), s);
        if (rc != RDB_E_UNSUPPORTED) return rc;
    }
    dim3 grid((unsigned)cdiv(k, GB_M), (unsigned)cdiv(coef_rows, GB_O));
    coef_grad_mat_kernel<<<grid, NT, 0, s>>>(dcoef, dW, dw_dtype, coef_rows, k, row_len, seed);
    return check_launch("coef_grad_mat_kernel");
}

static void sb_plan(int64_t Nw, int64_t *blocks, int64_t *span)
{
    int64_t b = cdiv(Nw, 4096);
    if (b > 1024) b = 1024;
    if (b < 1) b = 1;
    *span = cdiv(cdiv(Nw, b), NT) * NT;
    if (*span < NT) *span = NT;
    *blocks = cdiv(Nw, *span) > 0 ? cdiv(Nw, *span) : 1;
}

extern "C" int64_t rdb_scale_bias_bwd_workspace_bytes(int64_t Nw)
{
    if (Nw <= 0) return 0;
    int64_t blocks, span;
    sb_plan(Nw, &blocks, &span);
    return blocks > 1 ? blocks * (int64_t)sizeof(float) : 0;
}

extern "C" int rdb_scale_bias_bwd(float *ds, const void *dW, int dw_dtype, int64_t Nw, uint32_t seed, void *workspace,
                                  int64_t workspace_bytes, void *stream)
{
    if (Nw < 0) return set_error(RDB_E_SHAPE, "rdb_scale_bias_bwd: negative size %lld", (long long)Nw);
    if (!dtype_ok(dw_dtype)) return set_error(RDB_E_DTYPE, "rdb_scale_bias_bwd: unknown dW dtype %d", dw_dtype);
    if (!ds) return set_error(RDB_E_NULL, "rdb_scale_bias_bwd: ds is NULL");
    hipStream_t s = (hipStream_t)stream;
    if (Nw == 0) {
        return launch_reduce_rows(ds, ds, 0, 1, s);
    }
    if (!dW) return set_error(RDB_E_NULL, "rdb_scale_bias_bwd: dW is NULL");
    int64_t blocks, span;
    sb_plan(Nw, &blocks, &span);
    float *partial = ds;
    if (blocks > 1) {
        if (!workspace || workspace_bytes < blocks * (int64_t)sizeof(float))
            return set_error(RDB_E_WORKSPACE, "rdb_scale_bias_bwd: workspace of %lld bytes needed, %lld given",
                             (long long)(blocks * sizeof(float)), (long long)workspace_bytes);
        partial = (float *)workspace;
    }
    scale_bias_grad_kernel<<<(unsigned)blocks, NT, 0, s>>>(partial, dW, dw_dtype, Nw, span, seed);
    int rc = check_launch("scale_bias_grad_kernel");
    if (rc || blocks == 1) return rc;
    return launch_reduce_rows(ds, partial, blocks, 1, s);
}

extern "C" int rdb_embed_fwd(float *out, const int64_t *idx, int64_t n_idx, const void *coef, int coef_dtype, int64_t k,
                             int64_t rowsize, uint32_t seed, void *stream)
{
    if (n_idx < 0 || rowsize < 0 || k < 0)
        return set_error(RDB_E_SHAPE, "rdb_embed_fwd: negative size n_idx=%lld rowsize=%lld k=%lld", (long long)n_idx,
                         (long long)rowsize, (long long)k);
    if (!dtype_ok(coef_dtype)) return set_error(RDB_E_DTYPE, "rdb_embed_fwd: unknown coef dtype %d", coef_dtype);
    const int64_t Nw = n_idx * rowsize;
    if (Nw == 0) return RDB_OK;
    if (!out || !idx || (!coef && k > 0)) return set_error(RDB_E_NULL, "rdb_embed_fwd: out, idx or coef is NULL");
    return launch_materialize_vec(out, coef, coef_dtype, k, Nw, rowsize, 0, 0, seed, nullptr, idx, (hipStream_t)stream);
}

extern "C" int64_t rdb_embed_bwd_workspace_bytes(int64_t n_idx, int64_t rowsize, int64_t k)
{
    return rdb_materialize_bwd_workspace_bytes(0, k, 0, n_idx * rowsize);
}

extern "C" int rdb_embed_bwd(float *dcoef, const int64_t *idx, int64_t n_idx, const void *dout, int dout_dtype, int64_t k,
                             int64_t rowsize, uint32_t seed, void *workspace, int64_t workspace_bytes, void *stream)
{
    if (n_idx < 0 || rowsize < 0 || k < 0)
        return set_error(RDB_E_SHAPE, "rdb_embed_bwd: negative size n_idx=%lld rowsize=%lld k=%lld", (long long)n_idx,
                         (long long)rowsize, (long long)k);
    if (!dtype_ok(dout_dtype)) return set_error(RDB_E_DTYPE, "rdb_embed_bwd: unknown dout dtype %d", dout_dtype);
    if (k == 0) return RDB_OK;
    if (!dcoef) return set_error(RDB_E_NULL, "rdb_embed_bwd: dcoef is NULL");
    hipStream_t s = (hipStream_t)stream;
    const int64_t Nw = n_idx * rowsize;
    if (Nw == 0) {
        return launch_reduce_rows(dcoef, dcoef, 0, k, s);
    }
    if (!idx || !dout) return set_error(RDB_E_NULL, "rdb_embed_bwd: idx or dout is NULL");
    return coef_grad_vec(dcoef, dout, dout_dtype, k, Nw, rowsize, seed, idx, workspace, workspace_bytes, s, "rdb_embed_bwd");
}

// ----------------------------------------------------------------------------------------------- gradient of a pseudorandom bias
// b[o] = sum_m noise(PRIME*o + m) coef[m] + s noise1d(o), added to every row of y: with g[o] = sum_t dy[t, o],
// dcoef[m] = sum_o g[o] noise(PRIME*o + m) and ds = sum_o g[o] noise1d(o).
// A small dy: one launch (bias_grad_direct_kernel) or blocks of a layer's (rdb_bias.hpp).  Otherwise two.  First launch: the column sums of dy, a chunk of rows per block (memory-bound: dy is read once, 16 bytes a lane where its rows
// allow), partial sums [chunks x n].  Second launch: every block adds the chunks up again for itself (a few rows out of L2)
// and contracts them with the noise of its own BIAS_M coefficients; the n * k hashes are few.  Fixed orders throughout.
// Replaces a column sum by the library, its cast, the contraction and the sum over its splits: 128 tokens x 256, k = 64: 12.6 ->
// 6.0 us; 1024 tokens x 3072, k = 256: 19 -> 12 us.
namespace rdb {

template <typename T> __global__ __launch_bounds__(1024) void bias_grad_direct_kernel(BiasGrad q)
{
    __shared__ float sh[BIAS_M * 1024 / 64];
    bias_direct_block<T, 1024>(q, blockIdx.x, sh);
}
int bias_direct_launch(const BiasGrad &q, hipStream_t s)
{
    if (q.bf16) bias_grad_direct_kernel<bf16_t><<<(unsigned)q.blocks, 1024, 0, s>>>(q);
    else bias_grad_direct_kernel<float><<<(unsigned)q.blocks, 1024, 0, s>>>(q);
    return check_launch("bias_grad_direct_kernel");
}

// The second launch.  THREADS: a thread's outputs are a chain of
// memory latencies, so long biases take blocks of 1024 (3072 outputs, k = 256: 15.7 us with 256 threads, 12 turns of the loop; vector-coef layer step 561 -> 540).
template <int THREADS>
__device__ __forceinline__ void bias_grad_block(float *__restrict__ dcoef, float *__restrict__ ds, const float *__restrict__ part, int chunks, int64_t n, int64_t k, uint32_t seed,
                                                int block)
{
    const int64_t m0 = (int64_t)block * BIAS_M;
    const bool scale = !dcoef || m0 >= k;
    float acc[BIAS_M] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int64_t o = threadIdx.x; o < n; o += THREADS) {
        float g = 0.0f;
        for (int c0 = 0; c0 < chunks; c0 += 8) {   // eight loads in flight
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = part[(int64_t)(c0 + i < chunks ? c0 + i : chunks - 1) * n + o];
#pragma unroll
            for (int i = 0; i < 8; ++i) g += c0 + i < chunks ? v[i] : 0.0f;
        }
        bias_contract(acc, g, (uint32_t)o, m0, scale, seed);
    }
    __shared__ float sh[BIAS_M * THREADS / 64];
    bias_finish<THREADS>(acc, dcoef, ds, m0, k, scale, sh);
}
template <int THREADS> __global__ __launch_bounds__(THREADS) void bias_grad_kernel(float *__restrict__ dcoef, float *__restrict__ ds, const float *__restrict__ part, int chunks, int64_t n, int64_t k,
                                                       uint32_t seed)
{
    bias_grad_block<THREADS>(dcoef, ds, part, chunks, n, k, seed, blockIdx.x);
}
// The end of a vector-coef layer's backward pass: the partial rows of its coefficients' gradient, and behind them its bias's blocks
__global__ __launch_bounds__(1024) void layer_grads_kernel(float *__restrict__ dcoef, const float *__restrict__ partial, int64_t rows, int64_t k, int row_blocks,
                                                           float *__restrict__ db, const float *__restrict__ part, int chunks, int64_t n, int64_t bias_k, uint32_t bias_seed)
{
    if ((int)blockIdx.x < row_blocks) reduce_rows_block(dcoef, partial, rows, k, blockIdx.x);
    else bias_grad_block<1024>(db, nullptr, part, chunks, n, bias_k, bias_seed, (int)blockIdx.x - row_blocks);
}

}  // namespace rdb

extern "C" int64_t rdb_bias_bwd_workspace_bytes(int64_t rows, int64_t n) { return rows >= 0 && n > 0 ? bias_chunks(rows) * n * (int64_t)sizeof(float) : 0; }

extern "C" int rdb_bias_bwd(float *dcoef, float *ds, const void *dy, int dtype, int64_t ldy, int64_t rows, int64_t n, int64_t k, uint32_t seed, void *workspace,
                            int64_t workspace_bytes, void *stream)
{
    if (rows < 0 || n < 0 || k < 0 || ldy < n || n >= (1ll << 31))
        return set_error(RDB_E_SHAPE, "rdb_bias_bwd: rows=%lld n=%lld k=%lld ldy=%lld", (long long)rows, (long long)n, (long long)k, (long long)ldy);
    if (!dtype_ok(dtype)) return set_error(RDB_E_DTYPE, "rdb_bias_bwd: unknown dtype %d", dtype);
    if (k == 0) dcoef = nullptr;
    if (!dcoef && !ds) return RDB_OK;
    if (rows > 0 && n > 0 && !dy) return set_error(RDB_E_NULL, "rdb_bias_bwd: dy is NULL");
    hipStream_t s = (hipStream_t)stream;
    float *part = static_cast<float *>(workspace);
    int chunks = bias_chunks(rows);
    const int64_t blocks = (dcoef ? cdiv(k, BIAS_M) : 0) + (ds ? 1 : 0);
    // asked for whichever kernels run
    if (n > 0 && (!workspace || ((uintptr_t)workspace & 3) || workspace_bytes < rdb_bias_bwd_workspace_bytes(rows, n)))
        return set_error(RDB_E_WORKSPACE, "rdb_bias_bwd: workspace of %lld bytes needed, %lld given", (long long)rdb_bias_bwd_workspace_bytes(rows, n),
                         (long long)workspace_bytes);
    if (bias_direct(rows, n, dtype == RDB_BF16 ? 2 : 4, k, num_compute_units()))
        return bias_direct_launch({dcoef, ds, dy, ldy, k, (int)rows, (int)n, dtype == RDB_BF16, seed, (int)blocks}, s);
    if (n > 0) {
        const int64_t per = cdiv(rows, chunks);
        const int es = dtype == RDB_BF16 ? 2 : 4, V = 16 / es;
        const bool vec = ((uintptr_t)dy & 15) == 0 && ldy % V == 0 && n % V == 0;
        const dim3 grid((unsigned)cdiv(n, 64 * (vec ? V : 1)), (unsigned)chunks);
        if (dtype == RDB_BF16) {
            if (vec) column_sums_kernel<bf16_t, 8><<<grid, NT, 0, s>>>(part, static_cast<const bf16_t *>(dy), ldy, rows, n, per);
            else column_sums_kernel<bf16_t, 1><<<grid, NT, 0, s>>>(part, static_cast<const bf16_t *>(dy), ldy, rows, n, per);
        } else {
            if (vec) column_sums_kernel<float, 4><<<grid, NT, 0, s>>>(part, static_cast<const float *>(dy), ldy, rows, n, per);
            else column_sums_kernel<float, 1><<<grid, NT, 0, s>>>(part, static_cast<const float *>(dy), ldy, rows, n, per);
        }
        if (int rc = check_launch("column_sums_kernel")) return rc;
    }
    if (n > 512) bias_grad_kernel<1024><<<(unsigned)blocks, 1024, 0, s>>>(dcoef, ds, part, chunks, n, k, seed);
    else bias_grad_kernel<NT><<<(unsigned)blocks, NT, 0, s>>>(dcoef, ds, part, chunks, n, k, seed);
    return check_launch("bias_grad_kernel");
}

// ----------------------------------------------------------------------------------------------- backward pass of a vector-coef layer
// As calls of their own: dx and dW, a product and a sum of its ranges each, dW's contraction with the noise and the sum of its partial rows, the
// column sums of dy and the bias's contraction, eight launches of which six are 5 to 8 us and a gap behind each.  Here three: the two products side by
// side, the contraction, which adds dW's ranges up on the way and has dx's sums and the column sums beside it (it is the vector ALU's, they are the memory's), and the
// small ends together; more than VECTOR_DW_PARTS ranges of dW, many tokens of a small layer, are added up by a fourth.  Step of 1024 tokens x 768 -> 3072, k = 256: 481 -> 466 us (1.3 % of it for the bias's values formed beside W's in the forward pass); 1024 x 512 ->
// 1024, k = 200: 131 -> 118; steps that wait for the host, 2048 x 256 -> 512, k = 100: 100 -> 81; 32 x 64 -> 64, k = 16: 90 -> 79.
namespace rdb {

struct VectorBwdPlan {
    int64_t products, rows_at, cols_at, bytes, splits, span;
    int chunks;
};
static bool vector_bwd_plan(VectorBwdPlan &v, int64_t tokens, int64_t in_f, int64_t out_f, int64_t k, bool want_dx, bool bias)
{
    if (tokens <= 0 || in_f <= 0 || out_f <= 0 || k <= 0 || out_f * in_f >= (1ll << 31)) return false;
    v.products = vector_products_workspace(tokens, in_f, out_f, want_dx);
    if (!v.products) return false;
    split_plan(out_f * in_f, k, &v.splits, &v.span);
    auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
    v.rows_at = v.products;
    v.cols_at = v.rows_at + (v.splits > 1 ? up(v.splits * k * 4) : 0);
    v.chunks = bias_chunks(tokens);
    v.bytes = v.cols_at + (bias ? up((int64_t)v.chunks * out_f * 4) : 0);
    return true;
}

}  // namespace rdb

extern "C" int64_t rdb_vector_linear_bwd_workspace_bytes(int64_t tokens, int64_t in_f, int64_t out_f, int64_t k, int want_dx, int want_bias)
{
    VectorBwdPlan v;
    return vector_bwd_plan(v, tokens, in_f, out_f, k, want_dx != 0, want_bias != 0) ? v.bytes : 0;
}

// Of dcoef alone: only where the contraction adds up dW's ranges on its way, which saves a launch.  With one range, or more than it adds up, the launches are as many, and its kernel, which could carry more, takes 1 to
// 3 us longer: on the device, a step, calls of their own and this one: 29 tokens x 8 -> 10, k = 4 14.0, 15.0; 59 x 78 -> 1915, k = 4 26.2, 27.4; 2 x 769 -> 314, k = 14 30.7, 32.4; 13448 x 1031 -> 73, k = 4
// 88.8, 91.8; two ranges to eight: 333 x 84 -> 23, k = 12 30.0, 21.0; 443 x 42 -> 287, k = 4 24.9, 22.6; 594 x 781 -> 743, k = 3 57.6, 55.2.
extern "C" int rdb_vector_linear_bwd_pays(int64_t tokens, int64_t in_f, int64_t out_f, int want_dx, int want_bias)
{
    VectorBwdPlan v;
    if (!vector_bwd_plan(v, tokens, in_f, out_f, 1, want_dx != 0, want_bias != 0)) return 0;
    const int ranges = vector_dw_ranges(tokens, in_f, out_f);
    return want_dx || want_bias || (ranges > 1 && ranges <= VECTOR_DW_PARTS) ? 1 : 0;
}

extern "C" int rdb_vector_linear_bwd(float *dx, float *dcoef, float *dbias_coef, const float *dy, int64_t lddy, const float *x, int64_t ldx, const float *W, int64_t tokens,
                                     int64_t in_f, int64_t out_f, int64_t k, uint32_t seed, int64_t bias_k, uint32_t bias_seed, void *workspace, int64_t workspace_bytes,
                                     void *stream)
{
    const char *who = "rdb_vector_linear_bwd";
    if (tokens < 0 || in_f < 0 || out_f < 0 || k < 0 || bias_k < 0 || lddy < out_f || ldx < in_f)
        return set_error(RDB_E_SHAPE, "%s: tokens=%lld in_f=%lld out_f=%lld k=%lld bias k=%lld lddy=%lld ldx=%lld", who, (long long)tokens, (long long)in_f, (long long)out_f,
                         (long long)k, (long long)bias_k, (long long)lddy, (long long)ldx);
    if (!dcoef || !dy || !x || (dx && !W)) return set_error(RDB_E_NULL, "%s: dcoef, dy, x or (with dx) W is NULL", who);
    VectorBwdPlan v;
    const bool bias = dbias_coef && bias_k > 0;
    if (!vector_bwd_plan(v, tokens, in_f, out_f, k, dx != nullptr, bias))
        return set_error(RDB_E_UNSUPPORTED, "%s: needs non-empty sizes, matrices of less than 2^29 elements and the split products (rdb_set_f32_split)", who);
    if (!workspace || ((uintptr_t)workspace & 15) || workspace_bytes < v.bytes)
        return set_error(RDB_E_WORKSPACE, "%s: workspace of %lld bytes needed, %lld given", who, (long long)v.bytes, (long long)workspace_bytes);
    hipStream_t s = (hipStream_t)stream;
    char *ws = static_cast<char *>(workspace);
    GradLayerParams p = {};
    VectorDW dw;
    int rc = vector_products(dx, dy, lddy, x, ldx, W, tokens, in_f, out_f, ws, &p.sum, &dw, s);
    if (rc == RDB_E_UNSUPPORTED) return set_error(rc, "%s: matrices of less than 2^29 elements", who);
    if (rc) return rc;
    float *rows = v.splits > 1 ? reinterpret_cast<float *>(ws + v.rows_at) : dcoef, *cols = reinterpret_cast<float *>(ws + v.cols_at);
    p.partial = rows;
    p.d = dw.part;
    p.parts = dw.parts;
    p.part_stride = dw.stride;
    p.k = k;
    p.Nw = out_f * in_f;
    p.span = v.span;
    p.Q = 1;
    p.d_dtype = RDB_F32;
    p.narrow = 1;
    p.seed = seed;
    p.mblocks = (int)cdiv(k, grad_block(k));
    p.main_blocks = p.mblocks * (int)(v.splits / grad_rows(k));
    unsigned blocks = (unsigned)(p.main_blocks + p.sum.blocks);
    if (bias) {
        p.col_part = cols;
        p.dy = dy;
        p.lddy = lddy;
        p.rows = tokens;
        p.n = out_f;
        p.per_chunk = cdiv(tokens, v.chunks);
        p.col_vec = ((uintptr_t)dy & 15) == 0 && lddy % 4 == 0 && out_f % 4 == 0;
        p.col_x = (int)cdiv(out_f, p.col_vec ? 256 : 64);
        blocks += (unsigned)(p.col_x * v.chunks);
    }
    launch_grad_vec<false, true>(p, dim3(blocks), s);
    if ((rc = check_launch("coef_grad_vec_kernel"))) return rc;
    const int row_blocks = v.splits > 1 ? (int)cdiv(k, 32) : 0, bias_blocks = bias ? (int)cdiv(bias_k, BIAS_M) : 0;
    if (!(row_blocks + bias_blocks)) return RDB_OK;
    layer_grads_kernel<<<(unsigned)(row_blocks + bias_blocks), 1024, 0, s>>>(dcoef, rows, v.splits, k, row_blocks, dbias_coef, cols, v.chunks, out_f, bias_k, bias_seed);
    return check_launch("layer_grads_kernel");
}
