// Products at fp32 accuracy on the matrix cores: the kernel template of rdb_f32.hip, how a product is planned and how it is
// launched.  Each rdb_f32_*.hip compiles the kernels of some pairs of operand sources (they build in parallel).
#pragma once
#include "rdb_bias.hpp"
#include "rdb_gemm.hpp"
#include "rdb_sums.hpp"
#include <algorithm>
#include <type_traits>

namespace rdb {

constexpr int FG_BN = 128;        // B rows (output columns) per block
constexpr int FG_BK = 16;         // contraction values per stage
constexpr int FG_THREADS = 256;   // threads of a group: four waves, 2 x 2
constexpr uint32_t FG_OOB = 0x80000000u;   // a byte offset past the end of any matrix these kernels take (below 2^31 bytes)

// Where an operand's tile [rows x FG_BK] comes from.  In LDS every tile is [FG_BK][rows + 4]: an MFMA operand is 32
// consecutive floats of each of two contraction values.
enum FgSource {
    FG_KCONT = 0,    // src[row * ld + kk]: a row-major matrix whose rows are the tile's rows
    FG_MCONT = 1,    // src[kk * ld + row]: a row-major matrix whose rows are contraction values
    FG_NOISE_M = 2,  // 2-D noise (feature kk, coefficient row): the rows are coefficients, the contraction runs over features
    FG_NOISE_I = 3,  // 2-D noise (feature row, coefficient kk): the rows are features, the contraction runs over coefficients
    FG_NOISE_1D = 4  // 1-D noise at index row * sR + kk * sK: the random-bias matrix R, read along or across its rows
};
// What a block does with its accumulators.
enum FgEpilogue {
    FG_STORE = 0,       // out = acc
    FG_STORE_BIAS = 1,  // out = acc + bias[column]
    FG_ADD_SCALED = 2,  // out += scale[0] * acc; with dotm also the sums of FG_DOT
    FG_DOT = 3,         // dot_part[block] = sum over the tile of acc * dotm (nothing is stored to out)
    FG_STORE_RBIAS = 4  // out = acc + scale[0] * noise1d(row * nsR + column * nsK): materialising W = C . N + s . R
};

// Values of a contiguous vector-coef tensor in fp32, by blocks of their own beside a product's: out[e] = sum_m noise(e, m) coef[m] (+ scale[0]
// noise1d(e)), sixteen lanes an element, added up as the kernel that forms such tensors does.
struct FgValues {
    float *out;
    const float *coef, *scale;   // scale: NULL, or one value
    int n, k;                    // n: 0: no such blocks
    uint32_t seed;
    int slices;                  // of the launch's grid along z, behind the product's
};
__device__ __forceinline__ void fg_values(const FgValues &v, int thread, int threads)
{
    constexpr int LANES = 16;
    const int part = thread % LANES;
    for (int e = thread / LANES; e < v.n; e += threads / LANES) {
        uint32_t first = sq5_first((uint32_t)e, (uint32_t)part, v.seed);
        float acc = 0.0f;
        for (int m = part; m < v.k; m += LANES) {
            acc = fmaf(sq5_unit(sq5_tail(first)), v.coef[m], acc);
            first += LANES * SQ5_N1;
        }
#pragma unroll
        for (int w = 1; w < LANES; w *= 2) acc += __shfl_xor(acc, w);
        if (part == 0) v.out[e] = v.scale ? acc + v.scale[0] * noise1d((uint32_t)e, v.seed) : acc;
    }
}

// As many blocks as leave a thread 16 hashes, or one element's: the product's tiles may be a single one, and with one block for each of them 64 tokens x
// 4096 -> 4096, k = 64, a bias of 64 coefficients took 57 us (now 19.3, without a bias 18.8), -> 32768 518 (now 15.9, without 15.2).  32 hashes: 17.9 -> 19.2 for
// 128 x 2048 -> 2048, and 64 24.6; 8: the same.
constexpr int FG_VALUE_HASHES = 16;
inline int fg_value_slices(const FgValues &v, int64_t tiles, int threads)
{
    if (!v.n) return 0;
    const int64_t each = std::max<int64_t>(1, FG_VALUE_HASHES / std::max<int64_t>(1, cdiv(v.k, 16)));   // elements of sixteen lanes
    return (int)cdiv(cdiv(cdiv(v.n, each) * 16, threads), tiles);
}
// Beside the projection up to 64 hashes a lane in turn: more are longer than its blocks run, and a launch of its own, with more waves to a unit, ends sooner
// (us, beside and apart: 128 x 2048 -> 2048 with 64 coefficients 17.9, 20.3; 1024 22.4, 23.9; 1536 26.8, 26.0; 4096 47.4, 37.1; 64 x 784 -> 32768 with 1024 33.4,
// 34.3); n: of the tensors that a launch of their own adds up in the same order.
constexpr int FG_VALUES_K = 1024, FG_VALUES_N = 1 << 15;

struct FgParams {
    const float *a;   // A operand's matrix (FG_KCONT / FG_MCONT)
    int64_t lda;
    const float *b;   // B operand's matrix; not used by the noise sources
    int64_t ldb;
    float *out;       // [M x N], leading dimension ldo; split s of the contraction writes out + s * split_stride
    int64_t ldo, split_stride;
    const float *bias;   // [N] or NULL
    int M, N, K;
    int kchunk;          // contraction values per split (a multiple of FG_BK); K when there is one split
    int64_t a_bytes, b_bytes;   // extent of the matrices, for the bounds check of the loads (< 2^31)
    uint32_t seed;
    int a_es, b_es;             // bytes per element of the A and B matrices: 4, or 2 (bf16)
    int out_bf16;               // out, bias and dotm are bf16 (the activations' dtype)
    int scale_bf16;             // scale is bf16 (the coefficients' dtype)
    uint32_t nsR, nsK;          // FG_NOISE_1D: index steps per row and per contraction value
    const float *scale;         // FG_ADD_SCALED: one device value
    const float *dotm;          // FG_DOT, FG_ADD_SCALED (or NULL): [M x N] matrix, leading dimension lddot
    int64_t lddot;
    float *dot_part;            // with dotm: one value per block, in block order (x fastest, then y)
    FgValues values;            // FG_NOISE_M on the B side: formed by the last blocks along z
};
// ... of a launch that carries more than its product: a type of its own, since every launch waits for what it is given (150 bytes more in each of the five of a step: +1 us)
struct FgCarried : FgParams {
    FgSum sum;                  // FG_NOISE_I on the B side: a sum that an earlier launch left to do, by the last blocks along z
    int sum_slices;
    BiasGrad bias_grad;         // by the blocks before those
    int bias_slices;
};

// fp32 products on the bf16 matrix cores.  v = h + m + l exactly, each part a bf16: v rounded to the nearest, what is left rounded to
// the nearest, and what is left of that (both differences are exact).  A product a . b is then the sum of the nine products of the
// parts, each exact in the matrix core's fp32 accumulation, of which the six largest are computed: ah bh + ah bm + am bh + ah bl +
// al bh + am bm.  The three left out, am bl + al bm + al bl, are of either sign and at most 1.01 * 2^-24 |a b|, what one rounding of the
// product does (|m| <= 2^-8 |v|, |l| <= 2^-17 |v|), 2^-28 |a b| on average over normally distributed values.  (Parts cut off instead of
// rounded leave out up to 1.01 * 2^-21 |a b|, always of the product's sign, and are no faster.)  Six bf16 matrix instructions of
// 32 x 32 x 16 do the work of eight fp32 ones of 32 x 32 x 2 in 3/8 of the time.  fg_split3: two values at a time, the parts packed.
__device__ __forceinline__ void fg_split3(float v0, float v1, uint32_t &h, uint32_t &m, uint32_t &l)
{
    h = f32x2_to_bf16x2(v0, v1);
    v0 -= __uint_as_float(h << 16);
    v1 -= __uint_as_float(h & 0xffff0000u);
    m = f32x2_to_bf16x2(v0, v1);
    l = f32x2_to_bf16x2(v0 - __uint_as_float(m << 16), v1 - __uint_as_float(m & 0xffff0000u));
}
// The same where a value may be infinite, or round to an infinity.  An infinity becomes (largest bf16, largest bf16, infinity), so
// that its products are what an infinity's are: inf by nonzero and by infinite values, NaN by zero.  For that the parts are cut off
// and not rounded: all of one sign, so that none of a product's terms overflows to the other side.  A NaN stays a NaN.  This takes two
// v_med3 a value, 3 % of a step (2048 tokens x 768 -> 3072, k = 256, fp32: 107 -> 110 us, and 112 with a look at each stage's
// values instead), so it is not done at first: an infinity then gives NaN wherever it is met, and a block whose sums are not all
// finite runs its stages once more with it, for those (104.4 us, against 103.4 without any of it in the same run).  A value that comes from
// a bf16 matrix has one part, and an infinite one gives NaN where its partner's lower parts are zero: the products of bf16
// layers do without the second run.
__device__ __forceinline__ void fg_split3_any(float v, uint32_t &h, uint32_t &m, uint32_t &l)
{
    constexpr float top = 3.40282346638528859812e38f;
    h = __float_as_uint(__builtin_amdgcn_fmed3f(v, -top, top)) & 0xffff0000u;
    const float r1 = v - __uint_as_float(h);
    m = __float_as_uint(__builtin_amdgcn_fmed3f(r1, -top, top)) & 0xffff0000u;
    const float r2 = r1 - __uint_as_float(m);
    l = __float_as_uint(r2) & 0xffff0000u;
}

// One operand's way from its source into LDS: load(stage) requests / hashes the stage's values into registers, store() puts
// them into a tile.  Rows past `rows` and contraction values past `kend` are zeros.
// VEC: the matrix is read in pieces of four values (16 bytes of fp32, 8 bytes of bf16; 16-byte aligned base, leading dimension a
// multiple of 4, and the extent that runs along a piece a multiple of 4, so that a piece lies inside or outside as a whole);
// otherwise four values at a time at any address, see load4u.
// SPLIT: the tile goes to LDS as three bf16 planes (see fg_split3): planes of [2 halves of the stage's 16 contraction values]
// [rows][8] for the sources read along the contraction (a lane's MFMA operand is 16 consecutive bytes), of [16][rows + 32] for
// FG_MCONT (read back with the LDS transpose read).  The noise sources then give a thread consecutive contraction values.
// ES: bytes per element of the matrix, 4 or 2 (bf16).  Known to the compiler, because a load whose width is chosen by a branch has to
// be widened inside the branch, and so waited for where it is requested: every stage of a product with a bf16 matrix cost a memory
// latency (4097 tokens x 1001 -> 999 in bf16, k = 100: t = dy . C 21.0 -> 11.2 us, dC 17.5 -> 14.3, z 17.1 -> 15.7, step 91.8 -> 80.9).
// bf16 values stay as they are until they reach their one plane.  0: known per launch (es; not SPLIT).
template <int ROWS, int SRC, bool VEC, bool SPLIT = false, int ES = 4> struct FgOperand {
    static_assert(SPLIT ? ES == 4 || ES == 2 : ES == 0, "the fp32 matrix instructions' kernels learn the element's size at run time");
    static constexpr int LD = ROWS + 4, TILE = FG_BK * LD, NV = ROWS * FG_BK / FG_THREADS / 4;   // float4 per thread and stage
    static_assert(NV >= 1, "a stage is at least one float4 per thread");
    static constexpr bool HASHED = SRC == FG_NOISE_M || SRC == FG_NOISE_I || SRC == FG_NOISE_1D;
    static constexpr bool ONE = ES == 2 && !HASHED;   // values that are their own first part: only the first plane is written and read
    static constexpr int LDM = ROWS + 32;                                            // FG_MCONT plane: elements per contraction value
    static constexpr int PLANE = SRC == FG_MCONT ? FG_BK * LDM : 2 * ROWS * 8;       // bf16 elements of one plane
    static constexpr int TILE_BYTES = SPLIT ? (ONE ? 1 : 3) * PLANE * 2 : TILE * 4;
    static constexpr int KPT = NV * 4;                                               // SPLIT, noise: consecutive contraction values per thread
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef std::conditional_t<ONE, u32x2, f32x4> Piece;   // four values as they are on their way to LDS
    __amdgpu_buffer_rsrc_t rs;
    uint32_t off[NV];   // byte offset of the thread's pieces at stage 0
    bool ok[NV];        // ... and whether the piece's (first) row exists
    uint32_t step;      // bytes per stage
    uint32_t first;     // noise: first-round value of the thread's first element at stage 0
    int kk0, kend, k_begin;
    int rows_left[NV];  // FG_MCONT without VEC: how many of the piece's four rows exist
    bool edge, tiny;    // without VEC, the same for the whole block: some piece is not whole; some row has fewer than four values
    Piece r[NV];

    uint32_t inc;       // noise: first-round step per contraction value
    const char *base;   // the matrix, for load4u
    int es;             // bytes per element of the matrix
    // VEC: four consecutive elements at byte offset o, zeros when outside
    __device__ __forceinline__ Piece load4(uint32_t o, bool in) const
    {
        if constexpr (ONE) {
            return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, in ? (int)o : (int)FG_OOB, 0, 0));
        } else {
            if (ES == 0 && es == 2) {
                const u32x2 h = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, in ? (int)o : (int)FG_OOB, 0, 0));
                return f32x4{__uint_as_float(h[0] << 16), __uint_as_float(h[0] & 0xffff0000u), __uint_as_float(h[1] << 16), __uint_as_float(h[1] & 0xffff0000u)};
            }
            return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, in ? (int)o : (int)FG_OOB, 0, 0));
        }
    }
    // not VEC: four consecutive elements at any element's address (the hardware takes loads of 8 and 16 bytes at any address; 4097 tokens
    // x 1001 features in bf16, k = 100: z = x . N^T 20.8 us with a load per value, 14.4 us with these).  Where only the first n of
    // the four exist, the last four that do are loaded, from 4 - n elements before, and moved down by whole() when the piece
    // is stored: no branch that would have to wait for its loads.
    __device__ __forceinline__ Piece load4u(uint32_t o) const
    {
        typedef uint32_t pair_any __attribute__((ext_vector_type(2), aligned(2)));
        typedef float quad_any __attribute__((ext_vector_type(4), aligned(4)));
        if constexpr (ONE) {
            const pair_any h = *reinterpret_cast<const pair_any *>(base + o);
            return u32x2{h[0], h[1]};
        } else {
            if (ES == 0 && es == 2) {
                const pair_any h = *reinterpret_cast<const pair_any *>(base + o);
                return f32x4{__uint_as_float(h[0] << 16), __uint_as_float(h[0] & 0xffff0000u), __uint_as_float(h[1] << 16), __uint_as_float(h[1] & 0xffff0000u)};
            }
            const quad_any v = *reinterpret_cast<const quad_any *>(base + o);
            return f32x4{v[0], v[1], v[2], v[3]};
        }
    }
    // the first n (any number) of four elements, one by one: rows of fewer than four values
    __device__ __forceinline__ Piece load_first(uint32_t o, int n) const
    {
        Piece v = {};
        const bool b16 = ES == 2 || (ES == 0 && es == 2);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int at = j < n ? (int)(o + (b16 ? 2 : 4) * j) : (int)FG_OOB;
            if (b16) {
                const uint32_t h = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(rs, at, 0, 0);
                if constexpr (ONE) v[j / 2] |= h << (16 * (j & 1));
                else v[j] = __uint_as_float(h << 16);
            } else if constexpr (!ONE) {
                v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, at, 0, 0));
            }
        }
        return v;
    }
    // not VEC: how many of the values of piece h of a stage exist (any number: none when below 1, all when above 3)
    __device__ __forceinline__ int existing(int stage, int h) const
    {
        const int kk = k_begin + stage * FG_BK + kk0;
        if (SRC == FG_KCONT) return ok[h] ? kend - kk : 0;
        return ok[h] && kk + h * (FG_THREADS / (ROWS / 4)) < kend ? rows_left[h] : 0;
    }
    __device__ __forceinline__ Piece request(int stage, int h) const
    {
        const uint32_t o = off[h] + (uint32_t)stage * step;
        const int n = existing(stage, h);
        if (tiny) return load_first(o, n);
        const uint32_t e = ES ? (uint32_t)ES : (uint32_t)es;
        return load4u(n >= 4 ? o : n > 0 ? o - (uint32_t)(4 - n) * e : 0u);
    }
    // ... and the piece as it belongs: the values that exist first, zeros behind them
    __device__ __forceinline__ Piece whole(int stage, int h) const
    {
        Piece v = r[h];
        if (VEC || HASHED || !edge) return v;
        const int n = existing(stage, h);
        if (tiny || n >= 4) return v;
        if constexpr (ONE) {
            const uint64_t w = n > 0 ? (((uint64_t)v[1] << 32) | v[0]) >> (16 * (4 - n)) : 0;
            v = u32x2{(uint32_t)w, (uint32_t)(w >> 32)};
        } else {
            if (n <= 2) v = f32x4{v[2], v[3], 0.0f, 0.0f};
            if (n & 1) v = f32x4{v[1], v[2], v[3], 0.0f};
            if (n <= 0) v = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        return v;
    }
    __device__ __forceinline__ void init(const float *src, int64_t ld, int64_t bytes, int row0, int rows, int K, int k_begin_, int kend_, int nstage, uint32_t seed,
                                         uint32_t sR, uint32_t sK, int es_)
    {
        const int t = threadIdx.x & (FG_THREADS - 1);
        k_begin = k_begin_;
        kend = kend_;
        es = ES ? ES : es_;
        base = reinterpret_cast<const char *>(src);
        if (SRC == FG_KCONT) {
            rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(src), 0, (int)bytes, 0x00020000);
            step = (uint32_t)(FG_BK * es);
#pragma unroll
            for (int h = 0; h < NV; ++h) {
                const int idx = h * FG_THREADS + t, row = idx >> 2, kq = idx & 3;
                ok[h] = row0 + row < rows;
                off[h] = ok[h] ? (uint32_t)(((int64_t)(row0 + row) * ld + k_begin + kq * 4) * es) : 0u;
            }
            kk0 = (t & 3) * 4;
            tiny = K < 4;
            edge = row0 + ROWS > rows || kend_ - k_begin_ != nstage * FG_BK;
        } else if (SRC == FG_MCONT) {
            rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(src), 0, (int)bytes, 0x00020000);
            step = (uint32_t)(FG_BK * ld * es);
#pragma unroll
            for (int h = 0; h < NV; ++h) {
                const int idx = h * FG_THREADS + t, kk = idx / (ROWS / 4), r4 = (idx % (ROWS / 4)) * 4;
                ok[h] = row0 + r4 < rows;
                off[h] = ok[h] ? (uint32_t)(((int64_t)(k_begin + kk) * ld + row0 + r4) * es) : 0u;
                rows_left[h] = rows - (row0 + r4);
            }
            kk0 = t / (ROWS / 4);
            tiny = rows < 4;
            edge = row0 + ROWS > rows || kend_ - k_begin_ != nstage * FG_BK;
        } else {
            const int row = t % ROWS;
            kk0 = SPLIT ? (t / ROWS) * KPT : t / ROWS;
            if (SRC == FG_NOISE_1D) {
                first = ((uint32_t)(row0 + row) * sR + (uint32_t)(k_begin + kk0) * sK) * SQ5_N1 + seed;
                inc = sK * SQ5_N1;
            } else {
                first = SRC == FG_NOISE_M ? sq5_first((uint32_t)(k_begin + kk0), (uint32_t)(row0 + row), seed)
                                          : sq5_first((uint32_t)(row0 + row), (uint32_t)(k_begin + kk0), seed);
                inc = SRC == FG_NOISE_M ? PN1 : SQ5_N1;
            }
        }
    }
    __device__ __forceinline__ void load(int stage)
    {
        if constexpr (HASHED) {
#pragma unroll
            for (int j = 0; j < NV * 4; ++j) hash_piece(stage, j);
        } else if constexpr (VEC) {   // all inside or all outside
            // a thread's four values are consecutive contraction values (FG_KCONT) or consecutive rows (FG_MCONT)
            const int kk = k_begin + stage * FG_BK + kk0;
#pragma unroll
            for (int h = 0; h < NV; ++h)
                r[h] = load4(off[h] + (uint32_t)stage * step, ok[h] && kk + (SRC == FG_MCONT ? h * (FG_THREADS / (ROWS / 4)) : 0) < kend);
        } else {
#pragma unroll
            for (int h = 0; h < NV; ++h) r[h] = request(stage, h);
        }
    }
    // Noise sources: element j of the thread's NV * 4 values of a stage (contraction value kk0 + j * (FG_THREADS / ROWS), one add
    // apart in the first round).  The main loop calls this between the matrix instructions of the stage before.  Rows and contraction
    // values past the end are hashed as well: such rows' results are not stored, and such contraction values meet zeros of the other
    // side, which is a matrix.  A condition here is a branch around every hash, and no two hashes overlap (1660 tokens x 3902 -> 3361 in
    // bf16, k = 82, random bias: dy . R 320 -> 287 us, x . R^T 295 -> 263; 616 x 288 -> 1464, k = 40, fp32: z 7.0 -> 6.3).  Where k is a quarter of a
    // tile's 128 columns and less, the condition had spared whole waves their hashes, and z is up to 5 % longer (5417 x 1784, k = 10, bf16: 21.7 -> 22.9).
    __device__ __forceinline__ void hash_piece(int stage, int j)
    {
        if constexpr (HASHED) {
            constexpr int KSTEP = SPLIT ? 1 : FG_THREADS / ROWS;
            const uint32_t f = first + (uint32_t)(stage * FG_BK + j * KSTEP) * inc;
            r[j >> 2][j & 3] = sq5_unit(sq5_tail(f));
        }
    }
    __device__ __forceinline__ void store(int stage, float *__restrict__ tile) const
    {
        const int t = threadIdx.x & (FG_THREADS - 1);
        if (SRC == FG_KCONT) {
#pragma unroll
            for (int h = 0; h < NV; ++h) {
                const int idx = h * FG_THREADS + t, row = idx >> 2, kq = idx & 3;
                const Piece v = whole(stage, h);
#pragma unroll
                for (int j = 0; j < 4; ++j) tile[(kq * 4 + j) * LD + row] = v[j];
            }
        } else if (SRC == FG_MCONT) {
#pragma unroll
            for (int h = 0; h < NV; ++h) {
                const int idx = h * FG_THREADS + t, kk = idx / (ROWS / 4), r4 = (idx % (ROWS / 4)) * 4;
                *reinterpret_cast<Piece *>(tile + kk * LD + r4) = whole(stage, h);
            }
        } else {
            constexpr int KSTEP = FG_THREADS / ROWS;
            const int row = t % ROWS;
#pragma unroll
            for (int j = 0; j < NV * 4; ++j) tile[(kk0 + j * KSTEP) * LD + row] = r[j >> 2][j & 3];
        }
    }
    // SPLIT: four of the thread's values into the planes, 8 bytes each, at element offset `at` of a plane.
    template <bool FINITE> __device__ __forceinline__ void put4(bf16_t *__restrict__ tile, int at, const Piece &v) const
    {
        if constexpr (ONE) {
            *reinterpret_cast<u32x2 *>(tile + at) = v;
        } else {
            uint2 h, m, l;
            if (FINITE) {
                fg_split3(v[0], v[1], h.x, m.x, l.x);
                fg_split3(v[2], v[3], h.y, m.y, l.y);
            } else {
                uint32_t p[4][3];
#pragma unroll
                for (int j = 0; j < 4; ++j) fg_split3_any(v[j], p[j][0], p[j][1], p[j][2]);
                h = make_uint2(p[1][0] | (p[0][0] >> 16), p[3][0] | (p[2][0] >> 16));
                m = make_uint2(p[1][1] | (p[0][1] >> 16), p[3][1] | (p[2][1] >> 16));
                l = make_uint2(p[1][2] | (p[0][2] >> 16), p[3][2] | (p[2][2] >> 16));
            }
            *reinterpret_cast<uint2 *>(tile + at) = h;
            *reinterpret_cast<uint2 *>(tile + PLANE + at) = m;
            *reinterpret_cast<uint2 *>(tile + 2 * PLANE + at) = l;
        }
    }
    template <bool FINITE> __device__ __forceinline__ void store_split(int stage, bf16_t *__restrict__ tile) const
    {
        const int t = threadIdx.x & (FG_THREADS - 1);
        if (SRC == FG_KCONT) {
#pragma unroll
            for (int h = 0; h < NV; ++h) {   // contraction values 4 kq .. 4 kq + 3 of a row
                const int idx = h * FG_THREADS + t, row = idx >> 2, kq = idx & 3;
                put4<FINITE>(tile, ((kq >> 1) * ROWS + row) * 8 + (kq & 1) * 4, whole(stage, h));
            }
        } else if (SRC == FG_MCONT) {
#pragma unroll
            for (int h = 0; h < NV; ++h) {   // four consecutive rows at one contraction value
                const int idx = h * FG_THREADS + t, kk = idx / (ROWS / 4), r4 = (idx % (ROWS / 4)) * 4;
                put4<FINITE>(tile, kk * LDM + r4, whole(stage, h));
            }
        } else {
            const int row = t % ROWS;
#pragma unroll
            for (int h = 0; h < NV; ++h) {   // contraction values kk0 + 4 h .. + 3 of a row
                const int kk = kk0 + 4 * h;
                put4<FINITE>(tile, ((kk >> 3) * ROWS + row) * 8 + (kk & 7), r[h]);
            }
        }
    }
    // SPLIT: the MFMA operand of the 32 rows from rb of one plane: lane (r, g) gets contraction values 8 g .. 8 g + 7 of row rb + r
    __device__ static __forceinline__ bf16x8 frag(const bf16_t *__restrict__ plane, int rb, int lane)
    {
        const int r = lane & 31, g = lane >> 5;
        if (SRC != FG_MCONT) return *reinterpret_cast<const bf16x8 *>(plane + (g * ROWS + rb + r) * 8);
        // 16-lane group q covers rows rb + 16 q .. + 15; source lane s of the group addresses contraction value 8 g + s / 4,
        // rows 4 (s % 4) .. + 3; result lane c receives the rows' column c for four contraction values
        Frag8 f;
        const int sl = lane & 15, q = (lane >> 4) & 1;
        const bf16_t *src = plane + (g * 8 + (sl >> 2)) * LDM + rb + q * 16 + (sl & 3) * 4;
        f.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(src));
        f.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(src + 4 * LDM));
        return f.v;
    }
};

// out[M x N] (+)= A . B^T over one split of the contraction.  Block: BM x 128 of the output, G groups of four waves as 2 x 2, a
// wave owns (BM / 2) x 64 in BM / 64 x 2 accumulator tiles.  Two LDS buffers, one barrier per stage: while a stage is multiplied
// the next one is on its way from memory (or being hashed) in registers.
// G groups cut the block's contraction into G runs of stages, each with its own LDS buffers, and add their accumulators up
// through LDS in group order at the end.  One group is one wave to a SIMD, and its stages are a serial chain of about 1 us (load,
// split, barrier, LDS read, products, hash): a product with fewer blocks than compute units is bound by that chain, and G of
// them run side by side.  2048 tokens x 768 -> 3072, k = 256, fp32: z = x . N^T 14.6 us (64 rows, 6 ranges) -> 10.3 (G = 4, 4
// ranges), dx = t . N 19.5 -> 11.7 (G = 4), t = dy . C 27.4 us in 16 ranges -> 23.4 in 8 (G = 2: half the partial sums).  With
// blocks enough the chip's power is the bound (1.75 GHz under y = z . C^T, 3 groups a unit), and how the groups are arranged
// matters little.
// Results leave with streaming stores: they would be written back from L2 at the end of the kernel otherwise, after the last
// block (y of that layer, 25 MB: 26.4 -> 24.8 us).  Not so where rows are not whole lines of 128 bytes: a streaming store of part of
// a line goes to memory as such, where L2 puts a line's parts together (y of 3899 tokens x 5603, k = 199: 107 -> 75 us; 1500 x 5245, k =
// 156: 36 -> 24.6; 4096 x 999, k = 100: 16.7 -> 15.3; the step of 4096 x 1024 -> 8190, k = 128: 275 -> 267).
// AES, BES: bytes per element of the two matrices (SPLIT: 4, or 2, bf16; otherwise 0, see FgOperand).
// f32_gemm_block: what block (bx, by, bz) of a product does (gx: how many there are along x).  `lds`: FgBlock::LDS floats; not_finite: a
// word of LDS.
template <int BM, int G, int ASRC, int BSRC, bool VEC, bool SPLIT, int AES, int BES> struct FgBlock {
    typedef FgOperand<BM, ASRC, VEC, SPLIT, AES> PA;
    typedef FgOperand<FG_BN, BSRC, VEC, SPLIT, BES> PB;
    static constexpr int MI = BM / 64, NI = 2, STAGE = (PA::TILE_BYTES + PB::TILE_BYTES) / 4;   // floats
    static constexpr int UNITS = MI * NI * 2;   // a wave's accumulators in units of 8 registers: what the groups share out at the end
    static constexpr int EXCHANGE = (G - 1) * UNITS * 4 * 512;
    static constexpr int LDS = 2 * STAGE * G > EXCHANGE ? 2 * STAGE * G : EXCHANGE;
    static_assert(G == 1 || SPLIT, "groups: the bf16 matrix instructions only");
};
template <int BM, int G, int ASRC, int BSRC, int EPI, bool VEC, bool SPLIT, int AES, int BES>
__device__ __forceinline__ void f32_gemm_block(const FgParams &p, const int bx, const int by, const int bz, const int gx, float *__restrict__ lds_all, int &not_finite)
{
    typedef FgBlock<BM, G, ASRC, BSRC, VEC, SPLIT, AES, BES> Block;
    typedef typename Block::PA PA;
    typedef typename Block::PB PB;
    constexpr bool ANY16 = PA::ONE || PB::ONE, AGAIN = SPLIT && !ANY16;   // AGAIN: sums that are not finite are looked for
    constexpr int MI = Block::MI, NI = Block::NI, STAGE = Block::STAGE, UNITS = Block::UNITS;
    const int group = G == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / FG_THREADS);
    float *lds = lds_all + group * 2 * STAGE;
    const int t = threadIdx.x & (FG_THREADS - 1), wave = t >> 6, lane = t & 63, r = lane & 31, g = lane >> 5, wm = wave >> 1, wn = wave & 1;
    const int m0 = bx * BM, n0 = by * FG_BN;   // the long extent (tokens, as a rule) on the grid's x
    const int k_first = bz * p.kchunk, k_last = min(p.K, k_first + p.kchunk);
    const int nstage = ((k_last - k_first + FG_BK - 1) / FG_BK + G - 1) / G;   // of every group: the last one's may be empty
    const int k_begin = k_first + group * nstage * FG_BK, kend = min(k_last, k_begin + nstage * FG_BK);
    PA pa;
    PB pb;
    pa.init(p.a, p.lda, p.a_bytes, m0, p.M, p.K, k_begin, kend, nstage, p.seed, p.nsR, p.nsK, p.a_es);
    pb.init(p.b, p.ldb, p.b_bytes, n0, p.N, p.K, k_begin, kend, nstage, p.seed, p.nsR, p.nsK, p.b_es);
    // The five smaller products of the parts in sums of their own (low), where registers allow it: the large sum is then rounded once a
    // stage and not six times.  Distance from 64 bits, 13 layers of 32 to 1024 tokens with k <= 64, input gradient: 0.60 times that of
    // fp32 multiplications and additions one after the other, as the vector-ALU kernels do them (1.01 times with one sum, 1.15 with
    // one sum and parts cut off); outputs 0.68, coefficient gradients 0.46.  With it the 64-row kernels of one group would lose a
    // quarter of their waves (2048 tokens x 768 -> 3072, k = 256: step 106.5 us against 104.4); their contractions are short.
    constexpr bool APART = SPLIT && BM == 64 && G > 1 && !ANY16;
    f32x16 acc[MI][NI], low[MI][NI];
    if (AGAIN && threadIdx.x == 0) not_finite = 0;   // seen by everybody behind the first stage's barrier
    // The stage loop; for fp32 matrices once more for sums that are not finite (fg_split3).  A side that comes from a bf16 matrix has one
    // plane.
    auto stages = [&](auto finite) __attribute__((always_inline)) {
        constexpr int AP = PA::ONE ? 1 : 3, BP = PB::ONE ? 1 : 3;
        constexpr bool FINITE = decltype(finite)::value;
        for (int s = 0; s < nstage; ++s) {
            float *As = lds + (s & 1) * STAGE, *Bs = As + PA::TILE_BYTES / 4;
            if (SPLIT) {
                pa.template store_split<PA::HASHED || FINITE>(s, reinterpret_cast<bf16_t *>(As));
                pb.template store_split<PB::HASHED || FINITE>(s, reinterpret_cast<bf16_t *>(Bs));
            } else {
                pa.store(s, As);
                pb.store(s, Bs);
            }
            __syncthreads();   // also: every wave is done reading the other buffer (the stage before this one)
            const bool more = s + 1 < nstage;
            if (more) {
                if (!PA::HASHED) pa.load(s + 1);
                if (!PB::HASHED) pb.load(s + 1);
            }
            if (SPLIT) {
                // the stage is one k-step of the bf16 matrix instruction: three planes a side, six products a tile pair, the small
                // ones first (a side that comes from a bf16 matrix has one plane: three products, or one); the next stage's noise
                // values are hashed between the tile pairs
                const bf16_t *ap = reinterpret_cast<const bf16_t *>(As), *bp = reinterpret_cast<const bf16_t *>(Bs);
                {
                    bf16x8 fa[MI][AP], fb[NI][BP];
#pragma unroll
                    for (int pl = 0; pl < 3; ++pl) {
#pragma unroll
                        for (int mi = 0; mi < MI; ++mi)
                            if (pl < AP) fa[mi][pl] = PA::frag(ap + pl * PA::PLANE, wm * (BM / 2) + mi * 32, lane);
#pragma unroll
                        for (int ni = 0; ni < NI; ++ni)
                            if (pl < BP) fb[ni][pl] = PB::frag(bp + pl * PB::PLANE, wn * 64 + ni * 32, lane);
                    }
#pragma unroll
                    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                        for (int ni = 0; ni < NI; ++ni) {
                            f32x16 c = APART ? low[mi][ni] : acc[mi][ni];
                            if constexpr (AP == 3 && BP == 3) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi][1], fb[ni][1], c, 0, 0, 0);
                            if constexpr (AP == 3) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi][2], fb[ni][0], c, 0, 0, 0);
                            if constexpr (BP == 3) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi][0], fb[ni][2], c, 0, 0, 0);
                            if constexpr (AP == 3) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi][1], fb[ni][0], c, 0, 0, 0);
                            if constexpr (BP == 3) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi][0], fb[ni][1], c, 0, 0, 0);
                            if (APART) low[mi][ni] = c;
                            acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[mi][0], fb[ni][0], APART ? acc[mi][ni] : c, 0, 0, 0);
                            constexpr int GROUPS = MI * NI;
                            const int grp = mi * NI + ni;
                            if (PB::HASHED && more) {
                                constexpr int PER = (PB::NV * 4 + GROUPS - 1) / GROUPS;
#pragma unroll
                                for (int j = grp * PER; j < (grp + 1) * PER && j < PB::NV * 4; ++j) pb.hash_piece(s + 1, j);
                            }
                            if (PA::HASHED && more) {
                                constexpr int PER = (PA::NV * 4 + GROUPS - 1) / GROUPS;
#pragma unroll
                                for (int j = grp * PER; j < (grp + 1) * PER && j < PA::NV * 4; ++j) pa.hash_piece(s + 1, j);
                            }
                        }
                }
                continue;
            }
            const float *ap = As + g * PA::LD + wm * (BM / 2) + r, *bp = Bs + g * PB::LD + wn * 64 + r;
#pragma unroll
            for (int ks = 0; ks < FG_BK / 2; ++ks) {
                float fa[MI], fb[NI];
#pragma unroll
                for (int mi = 0; mi < MI; ++mi) fa[mi] = ap[ks * 2 * PA::LD + mi * 32];
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) fb[ni] = bp[ks * 2 * PB::LD + ni * 32];
#pragma unroll
                for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                    for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[mi], fb[ni], acc[mi][ni], 0, 0, 0);
                // the next stage's noise values are hashed in the shadow of these matrix instructions, a share per k-step
                if (PB::HASHED && more) {
                    constexpr int PER = (PB::NV * 4 + FG_BK / 2 - 1) / (FG_BK / 2);
#pragma unroll
                    for (int j = ks * PER; j < (ks + 1) * PER && j < PB::NV * 4; ++j) pb.hash_piece(s + 1, j);
                }
                if (PA::HASHED && more) {
                    constexpr int PER = (PA::NV * 4 + FG_BK / 2 - 1) / (FG_BK / 2);
#pragma unroll
                    for (int j = ks * PER; j < (ks + 1) * PER && j < PA::NV * 4; ++j) pa.hash_piece(s + 1, j);
                }
            }
        }
    };
    auto product = [&](auto finite) __attribute__((always_inline)) {
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[mi][ni][e] = low[mi][ni][e] = 0.0f;
        pa.load(0);
        pb.load(0);
        stages(finite);
        if (APART) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[mi][ni][e] += low[mi][ni][e];
        }
    };
    product(std::true_type{});
    bool again = false;
    if (AGAIN) {
        float zero = 0.0f;   // stays so as long as every sum is finite
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                for (int e = 0; e < 16; ++e) zero = fmaf(acc[mi][ni][e], 0.0f, zero);
        if (zero != 0.0f) not_finite = 1;
        __syncthreads();   // also: the stage buffers are free
        again = __builtin_amdgcn_readfirstlane(not_finite) != 0;
    }
    // The groups' sums: unit u (registers 8 (u % 2) .. of tile u / 2) is finished by group u * G / UNITS; the others hand theirs over.  Behind a
    // barrier: the stage buffers are free
    auto exchange = [&]() __attribute__((always_inline)) {
        auto slot = [&](int u, int from, int owner) { return lds_all + ((u * (G - 1) + (from < owner ? from : from - 1)) * 4 + wave) * 512 + lane; };
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            const int owner = u * G / UNITS;
            if (group == owner) continue;
            float *dst = slot(u, group, owner);
#pragma unroll
            for (int j = 0; j < 8; ++j) dst[j * 64] = acc[u / 2 / NI][u / 2 % NI][(u & 1) * 8 + j];
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            const int owner = u * G / UNITS;
            if (group != owner) continue;
#pragma unroll
            for (int from = 0; from < G; ++from) {
                if (from == owner) continue;
                const float *src = slot(u, from, owner);
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[u / 2 / NI][u / 2 % NI][(u & 1) * 8 + j] += src[j * 64];
            }
        }
    };
    if constexpr (G > 1) {
        if (!AGAIN) __syncthreads();
        exchange();
    }
    // accumulator j of lane (r, g): row 8 (j / 4) + 4 g + j % 4 of the A side, column r of the B side
    float *out = p.out + (int64_t)bz * p.split_stride;
    bf16_t *out16 = reinterpret_cast<bf16_t *>(p.out);   // bf16 outputs are never the ranges' partial matrices
    const bool o16 = p.out_bf16 != 0;
    const float scale = (EPI != FG_ADD_SCALED && EPI != FG_STORE_RBIAS) ? 0.0f
                        : p.scale_bf16 ? bf16_to_f32(reinterpret_cast<const bf16_t *>(p.scale)[0]) : p.scale[0];
    float dot = 0.0f;
    // KIND: how the results leave, where that is known outside of the loops (a branch per store costs 4 us of the fp32 step above).
    // Sums that are not finite come from the stages run once more (fg_split3_any), and only those: the others leave as they do without
    // these beside them.  WHICH: all; or, from the second run, those in whose place the first one left a value that is not finite.
    // What is added to an output is not seen there: the first run then leaves out the sums that are not finite, `bad`, for the second.
    enum { STREAM, PLAIN, NARROW, ANY };
    enum { ALL, REPAIR, GOOD, BAD };
    uint32_t bad[MI * NI / 2];
    auto results = [&](auto kind, auto which) __attribute__((always_inline)) {
        constexpr int KIND = decltype(kind)::value, WHICH = decltype(which)::value;
        const bool to16 = KIND == NARROW || (KIND == ANY && o16);
        int r_ = r, g_ = g;
        if (WHICH != ALL) asm volatile("" : "+v"(r_), "+v"(g_));   // addresses are made here and not kept in registers over the stages
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
            const int n = n0 + wn * 64 + ni * 32 + r_;
            if (n >= p.N) continue;
            const float bv = EPI != FG_STORE_BIAS ? 0.0f : to16 ? bf16_to_f32(reinterpret_cast<const bf16_t *>(p.bias)[n]) : p.bias[n];
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    if (G > 1 && group != ((mi * NI + ni) * 2 + j / 8) * G / UNITS) continue;
                    const int m = m0 + wm * (BM / 2) + mi * 32 + 8 * (j >> 2) + 4 * g_ + (j & 3);
                    if (m >= p.M) continue;
                    if ((WHICH == GOOD || WHICH == BAD) && (bad[(mi * NI + ni) / 2] >> ((mi * NI + ni) % 2 * 16 + j) & 1) != (WHICH == BAD)) continue;
                    const float a = acc[mi][ni][j];
                    if (EPI == FG_DOT || (EPI == FG_ADD_SCALED && p.dotm)) {
                        const int64_t e = (int64_t)m * p.lddot + n;
                        dot = fmaf(a, to16 ? bf16_to_f32(reinterpret_cast<const bf16_t *>(p.dotm)[e]) : p.dotm[e], dot);
                    }
                    if (EPI != FG_DOT) {
                        const int64_t e = (int64_t)m * p.ldo + n;
                        if (WHICH == REPAIR && (to16 ? bf16_to_f32(out16[e]) : out[e]) * 0.0f == 0.0f) continue;
                        if (EPI == FG_STORE_RBIAS) out[e] = fmaf(scale, noise1d((uint32_t)m * p.nsR + (uint32_t)n * p.nsK, p.seed), a);
                        else if (to16) out16[e] = f32_to_bf16(EPI == FG_ADD_SCALED ? fmaf(scale, a, bf16_to_f32(out16[e])) : a + bv);
                        else if (EPI == FG_ADD_SCALED) out[e] = fmaf(scale, a, out[e]);
                        else if (KIND == STREAM) __builtin_nontemporal_store(a + bv, out + e);
                        else out[e] = a + bv;
                    }
                }
        }
    };
    typedef std::integral_constant<int, ANY> Any;
    typedef std::integral_constant<int, ALL> All;
    auto second_run = [&]() __attribute__((always_inline)) {
        __syncthreads();   // the groups' sums have been read
        product(std::false_type{});
        if constexpr (G > 1) {
            __syncthreads();
            exchange();
        }
    };
    if constexpr (EPI == FG_ADD_SCALED || EPI == FG_DOT) {
        if (again) {
#pragma unroll
            for (int i = 0; i < MI * NI / 2; ++i) {
                bad[i] = 0;
#pragma unroll
                for (int e = 0; e < 32; ++e) bad[i] |= acc[(2 * i + e / 16) / NI][(2 * i + e / 16) % NI][e % 16] * 0.0f != 0.0f ? 1u << e : 0u;
                asm volatile("" : "+v"(bad[i]));   // a word, not 32 comparisons
            }
            results(Any{}, std::integral_constant<int, GOOD>{});
        } else {
            results(Any{}, All{});
        }
        if constexpr (AGAIN) {
            if (again) {
                second_run();
                results(Any{}, std::integral_constant<int, BAD>{});
            }
        }
    } else {
        if constexpr (EPI == FG_STORE_RBIAS) results(Any{}, All{});
        else if (o16) results(std::integral_constant<int, NARROW>{}, All{});
        else if (p.ldo % 32 == 0) results(std::integral_constant<int, STREAM>{}, All{});   // rows of whole lines
        else results(std::integral_constant<int, PLAIN>{}, All{});
        if constexpr (AGAIN) {
            if (again) {
                second_run();
                results(Any{}, std::integral_constant<int, REPAIR>{});
            }
        }
    }
    if (EPI == FG_DOT || (EPI == FG_ADD_SCALED && p.dotm)) {
        // lanes, then waves, in a fixed order
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) dot += __shfl_xor(dot, o);
        __syncthreads();   // the stage buffers are free
        if (lane == 0) lds_all[group * 4 + wave] = dot;
        __syncthreads();
        if (threadIdx.x == 0) {
            float sum = 0.0f;
#pragma unroll
            for (int i = 0; i < 4 * G; ++i) sum += lds_all[i];
            p.dot_part[(int64_t)by * gx + bx] = sum;
        }
    }
}

// Waves a SIMD that registers have to leave room for.  Hashing without a condition per value takes 4 to 8 registers more, which two kinds of tiles do not have
// to spare: 128 rows of x . R^T, 170 instead of 164 registers, two blocks to a unit instead of three (7028 tokens x 1240 -> 1248 in fp32: 218 us with the
// condition, 250 without, 208 so), and 64 rows in two groups, 134 instead of 126, one block instead of two.  Asked for, they are found without spills.
template <int BM, int G, int BSRC> constexpr int fg_min_waves()
{
    if (G == 1) return BM == 128 && BSRC == FG_NOISE_1D ? 3 : 2;
    return G == 2 && BM == 64 && (BSRC == FG_NOISE_M || BSRC == FG_NOISE_I) ? 4 : 1;
}
// The last launch of a backward pass, dx = t . N or dC = dy^T . z alone, carries the gradient of a pseudorandom bias where dy is small: a launch of its own is 6 us
// of kernel and as much on the host (128 images through 784 -> 256 -> 10, k = 64, fp32: 18 launches a step, 16 without).
constexpr bool fg_carries_bias(int asrc, int bsrc) { return bsrc == FG_NOISE_I || (asrc == FG_MCONT && bsrc == FG_MCONT); }
template <int BM, int G, int ASRC, int BSRC, int EPI, bool VEC, bool SPLIT, int AES, int BES, bool CARRY = false>
__global__ __launch_bounds__(FG_THREADS * G, (fg_min_waves<BM, G, BSRC>())) void f32_gemm_kernel(std::conditional_t<CARRY, FgCarried, FgParams> p)
{
    __shared__ __align__(16) float lds[FgBlock<BM, G, ASRC, BSRC, VEC, SPLIT, AES, BES>::LDS];
    __shared__ int not_finite;   // some thread's sum is an infinity or a NaN
    if constexpr (BSRC == FG_NOISE_M) {
        const unsigned products = gridDim.z - (unsigned)p.values.slices;
        if (blockIdx.z >= products) {
            constexpr int THREADS = FG_THREADS * G;
            const int tiles = (int)(gridDim.x * gridDim.y), block = (int)(blockIdx.z - products) * tiles + (int)(blockIdx.y * gridDim.x + blockIdx.x);
            fg_values(p.values, block * THREADS + (int)threadIdx.x, p.values.slices * tiles * THREADS);
            return;
        }
    }
    if constexpr (CARRY) {
        const unsigned sums = gridDim.z - (unsigned)p.sum_slices, products = sums - (unsigned)p.bias_slices;
        if (blockIdx.z >= products) {
            const bool sum = BSRC == FG_NOISE_I && blockIdx.z >= sums;
            const int tiles = (int)(gridDim.x * gridDim.y), block = (int)(blockIdx.z - (sum ? sums : products)) * tiles + (int)(blockIdx.y * gridDim.x + blockIdx.x);
            if (sum) {
                const int mine = block * G + (int)threadIdx.x / FG_THREADS;
                if (mine < p.sum.blocks) f32_sum_block(p.sum, mine, threadIdx.x & (FG_THREADS - 1));
            } else if (block < p.bias_grad.blocks) {
                if (p.bias_grad.bf16) bias_direct_block<bf16_t, FG_THREADS * G>(p.bias_grad, block, lds);
                else bias_direct_block<float, FG_THREADS * G>(p.bias_grad, block, lds);
            }
            return;
        }
    }
    f32_gemm_block<BM, G, ASRC, BSRC, EPI, VEC, SPLIT, AES, BES>(p, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.x, lds, not_finite);
}

// ----------------------------------------------------------------------------------------------- host side
inline bool fg_aligned16(const void *q) { return ((uintptr_t)q & 15) == 0; }
inline int64_t up256(int64_t n) { return (n + 255) / 256 * 256; }

int f32_split_mode();   // rdb_f32.hip

// How a product [M x N] over K runs: tile height, groups per block, contraction ranges.  Each range leaves a partial matrix,
// added up in range order afterwards, so the result does not depend on which block finishes first.
struct FgPlan {
    int bm, ranges, groups;
};
// Room for partial matrices: what a workspace holds.  128-row tiles, two blocks per compute unit at a time, unless even in ranges
// they would leave half of the compute units without a block; 64-row tiles then.  A product with fewer tiles than that is cut
// into ranges of the contraction, at least min_range values each, at most max_ranges.
inline FgPlan fg_room(int64_t M, int64_t N, int64_t K, int num_cus, int64_t min_range, int max_ranges)
{
    const int64_t slots = 2 * (int64_t)num_cus;
    const int64_t t128 = cdiv(M, 128) * cdiv(N, FG_BN), t64 = cdiv(M, 64) * cdiv(N, FG_BN);
    int64_t cap = K / min_range;
    if (cap > max_ranges) cap = max_ranges;
    if (cap < 1) cap = 1;
    auto ranges = [&](int64_t tiles) {
        int64_t r = slots / tiles;
        if (r > cap) r = cap;
        return r < 1 ? (int64_t)1 : r;
    };
    const int64_t r128 = ranges(t128), r64 = ranges(t64);
    if (t128 * r128 * 2 < slots) return {64, (int)r64, 1};
    return {128, (int)r128, 1};
}
// The plan with the least modelled time, of those with at most max_ranges ranges.  The model is measured (22 products of this
// file's kinds, [258 .. 7520] x [100 .. 7520] over [100 .. 7520], some 380 plans; what it picks is within 1 % of the best of
// them on average, 3 % at most): a stage of a group takes `chain` us when it has the compute unit to itself, the groups that
// share a unit take `unit` us of its throughput each, a launch `base` us and every further round of blocks 2.6; outputs leave at 4.8 TB/s; adding ranges up is one more
// launch, whose 14 TB/s say that the partial matrices come back out of the caches.  `host_us`: what that launch counts
// for besides: a step whose kernels are shorter than the host's work on it (50 to 70 us for a layer) pays for the launch as well, so where the
// product is short (FG_SHORT_US, and less and less up to FG_LONG_US) ranges have to gain more than both, and 4 % where it
// is long: a product that fills the chip a little better slows the kernels beside it, which share its power (a vector-coef step of 696 tokens x 856
// -> 3069, k = 74: y 41.7 -> 39.1 us in three ranges, 3.7 % by the model, the hashing kernels 190 -> 204; dW of 1024 x 768 -> 3072, 4.7 %: 45.5 -> 41.0 and
// the others as they were: the line lies between these two, no other product near it was measured).  `resident`, the groups that take turns on a unit's
// time, was fitted with the others and is not what registers and LDS leave room for.  The products measured had fp32 matrices; a
// side that comes from a bf16 matrix takes less LDS and fewer registers (four to seven blocks of 256 threads fit a unit), and hashing
// is not told apart: for those the constants are what they are for fp32.
struct FgKind {
    int bm, groups, resident;
    double chain, unit, base;
};
constexpr FgKind FG_KINDS[] = {{128, 1, 3, 0.51, 0.36, 5.4}, {128, 2, 1, 0.51, 0.36, 5.4}, {64, 1, 4, 0.46, 0.26, 3.7},
                               {64, 2, 2, 0.46, 0.26, 3.7},  {64, 4, 1, 0.46, 0.26, 3.7}};
// contraction values of each of r ranges; 0 where a range would hold nothing, or less than four stages
inline int64_t fg_chunk(int64_t K, int r)
{
    const int64_t chunk = cdiv(cdiv(K, r), FG_BK) * FG_BK;
    return r > 1 && (cdiv(K, chunk) != r || chunk < 64) ? 0 : chunk;
}
constexpr double FG_HOST_US = 3.8, FG_SHORT_US = 16.0, FG_LONG_US = 24.0, FG_HEAT = 0.04;
inline FgPlan fg_plan(int64_t M, int64_t N, int64_t K, int num_cus, int max_ranges, bool groups4, double host_us = 0.0, bool split = f32_split_mode() != 0)
{
    const double out_mb = (double)M * N * 4e-6;
    FgPlan best = {128, 1, 1};
    double best_us = 1e30;
    // the ranges that fg_chunk allows and the stages of each, once for all kinds: a step makes five plans, and this is host time (1.2 us a plan of 32
    // ranges with a chunk and three 64-bit divisions per range and kind, 0.4 so)
    constexpr uint32_t CAP = 64;
    uint32_t count = 0, ranges[CAP], stages_of[CAP];
    const uint32_t all = (uint32_t)cdiv(K, FG_BK), most = (uint32_t)(max_ranges < (int)CAP ? max_ranges : (int)CAP);
    for (uint32_t r = 1; r <= most; ++r) {
        const uint32_t n = (all + r - 1) / r;
        if (r > 1 && n < 4) break;
        if (r > 1 && (all + n - 1) / n != r) continue;
        ranges[count] = r;
        stages_of[count++] = n;
    }
    auto tiles = [&](int bm) { return (uint32_t)std::min<int64_t>(cdiv(M, bm) * cdiv(N, FG_BN), 1 << 25); };
    const uint32_t t128 = tiles(128), t64 = tiles(64);
    for (uint32_t i = 0; i < count; ++i) {
        const uint32_t r = ranges[i];
        const double more = r > 1 ? 4.2 + out_mb * r * 0.28 : out_mb * 0.21;
        for (const FgKind &kd : FG_KINDS) {
            if (kd.groups > 1 && (!split || (kd.groups == 4 && !groups4))) continue;
            const uint32_t per_cu = ((kd.bm == 128 ? t128 : t64) * r + (uint32_t)num_cus - 1) / (uint32_t)num_cus, rounds = (per_cu + (uint32_t)kd.resident - 1) / (uint32_t)kd.resident;
            const uint32_t stages = (stages_of[i] + (uint32_t)kd.groups - 1) / (uint32_t)kd.groups;
            double us = kd.base + 2.6 * (rounds - 1) + stages * (rounds * kd.chain + per_cu * kd.groups * kd.unit) + more;
            if (r > 1 && host_us > 0.0) us += std::max(FG_HEAT * us, us < FG_SHORT_US ? host_us : host_us * (FG_LONG_US - us) / (FG_LONG_US - FG_SHORT_US));
            if (us < best_us) {
                best_us = us;
                best = {kd.bm, (int)r, kd.groups};
            }
        }
    }
    return best;
}
// Two products side by side in one launch, blocks of one kind (rdb_f32_pair.hip).  The same model with constants of its own, fitted to
// 14 layers of 256 to 8000 tokens ([300 .. 3001] -> [256 .. 8192], k 40 to 700), some 100 plans each: what it picks is within 5 % of
// the backward pass of the best of them (1 % on average).  chain, unit: as above; a unit's blocks are of both products, so the mean of
// their stages counts; out, sum: us per MB of partial matrices written, and read back; resident: fitted as the others are (of 128 rows
// and two groups one block fits a unit whatever the matrices, 132 registers and 512 threads in bf16; two say that rounds cost less).
struct FgPairPlan {
    int bm, groups, ranges[2];
};
inline FgPairPlan fg_plan_pair(const int64_t (&M)[2], const int64_t (&N)[2], const int64_t (&K)[2], int num_cus, const int (&max_ranges)[2], bool b16)
{
    constexpr int CAP = 64;
    struct Kind {
        int bm, groups;
        double resident, chain, unit;
    };
    struct Model {
        Kind kinds[3];
        double round, out, sum, sums;
    };
    static const Model wide = {{{128, 1, 2, 0.438, 0.082}, {128, 2, 1, 0.375, 0.275}, {64, 2, 1, 0.074, 0.223}}, 0.34, 0.33, 0.0, 2.9};
    static const Model narrow = {{{128, 1, 3, 0.656, 0.084}, {128, 2, 2, 0.219, 0.342}, {64, 2, 2, 0.476, 0.107}}, 0.0, 0.0, 0.29, 0.15};
    const Model &m = b16 ? narrow : wide;
    const double per_unit = 1.0 / num_cus;
    FgPairPlan best = {128, 1, {1, 1}};
    double best_us = 1e30;
    for (const Kind &kd : m.kinds) {
        struct Option {
            int r;
            double blocks, stages, out;
        } opt[2][CAP];
        int n[2] = {0, 0};
        for (int i = 0; i < 2; ++i)
            for (int r = 1; r <= max_ranges[i] && r <= CAP; ++r) {
                const int64_t chunk = fg_chunk(K[i], r);
                if (!chunk) continue;
                const double mb = (double)M[i] * N[i] * 4e-6 * r;
                opt[i][n[i]++] = {r, (double)(cdiv(M[i], kd.bm) * cdiv(N[i], FG_BN) * r), (double)cdiv(chunk / FG_BK, kd.groups), mb * (r > 1 ? m.out + m.sum : m.out)};
            }
        for (int i = 0; i < n[0]; ++i)
            for (int j = 0; j < n[1]; ++j) {
                const Option &a = opt[0][i], &b = opt[1][j];
                const double blocks = a.blocks + b.blocks, mean = (a.blocks * a.stages + b.blocks * b.stages) / blocks, longest = a.stages > b.stages ? a.stages : b.stages;
                // units that hold several blocks are not filled to the last one: 510 blocks in 512 places ran as two rounds
                const double fill = blocks * per_unit, per_cu = (double)(int64_t)(fill + 0.999);
                const double rounds = (double)(int64_t)(fill * (kd.resident > 1.0 ? 1.02 : 1.0) / kd.resident + 0.999);
                const double alone = longest * (kd.chain + kd.groups * kd.unit);   // a unit with one block
                const double busy = (rounds > 1.0 ? rounds * mean : longest) * kd.chain + per_cu * mean * kd.groups * kd.unit;
                const double us = m.round * (rounds - 1.0) + (alone > busy ? alone : busy) + a.out + b.out + (a.r > 1 || b.r > 1 ? m.sums : 0.0);
                if (us < best_us) {
                    best_us = us;
                    best = {kd.bm, kd.groups, {a.r, b.r}};
                }
            }
    }
    return best;
}
struct FgProduct {
    const float *a;
    int64_t lda, a_elems;
    const float *b;
    int64_t ldb, b_elems;
    float *out;
    int64_t ldo;
    const float *bias;
    int64_t M, N, K;
    int bm;                 // tile height: 128 or 64; 0: fg_launch plans it, and the groups
    int groups;             // per block: 1, 2 or (64-row tiles) 4
    int64_t kchunk;         // contraction values per range (a multiple of FG_BK); 0: one range
    int64_t split_stride;   // floats between the ranges' outputs
    uint32_t seed;
    // the random-bias products (FG_NOISE_1D on the B side): index steps, and what the epilogue does
    uint32_t nsR, nsK;
    const float *scale;     // out += scale[0] * product
    const float *dotm;      // and / or: dot_part[block] = <product tile, dotm tile>
    int64_t lddot;
    float *dot_part;
    // bytes per element of the A and B matrices (2: bf16), and whether out / bias / dotm and scale are bf16
    int a_es = 4, b_es = 4, out_bf16 = 0, scale_bf16 = 0;
    // the products as six bf16 matrix instructions on three-way splits of the operands (fg_split3); materialising stays on the
    // fp32 matrix instructions (its unit-coefficient results are compared bit for bit)
    bool split = f32_split_mode() != 0;
    FgValues values = {};
    FgSum sum = {};
    BiasGrad bias_grad = {};   // bias_direct holds for it
};

#define FG_LAUNCH_GROUPS(BM_, G_, EPI_)                                                                               \
    do {                                                                                                            \
        const int nt = FG_THREADS * G_;                                                                             \
        auto of = [&](auto aes_, auto bes_) {                                                                       \
            constexpr int AES = decltype(aes_)::value, BES = decltype(bes_)::value;                                 \
            if constexpr (fg_carries_bias(ASRC, BSRC) && EPI_ == FG_STORE)                                          \
                if (more) {                                                                                         \
                    if (vec) f32_gemm_kernel<BM_, G_, ASRC, BSRC, EPI_, true, true, AES, BES, true><<<grid, nt, 0, s>>>(carried); \
                    else f32_gemm_kernel<BM_, G_, ASRC, BSRC, EPI_, false, true, AES, BES, true><<<grid, nt, 0, s>>>(carried);    \
                    return;                                                                                         \
                }                                                                                                   \
            if (vec) f32_gemm_kernel<BM_, G_, ASRC, BSRC, EPI_, true, true, AES, BES><<<grid, nt, 0, s>>>(p);       \
            else f32_gemm_kernel<BM_, G_, ASRC, BSRC, EPI_, false, true, AES, BES><<<grid, nt, 0, s>>>(p);          \
        };                                                                                                          \
        typedef std::integral_constant<int, 4> Wide;                                                                \
        typedef std::integral_constant<int, 2> Narrow;                                                              \
        if (a16) {                                                                                                  \
            if constexpr (Groups::a16_b16) { if (b16) { of(Narrow{}, Narrow{}); break; } }                          \
            if constexpr (Groups::a16_b32) of(Narrow{}, Wide{});                                                    \
        } else if (b16) {                                                                                           \
            if constexpr (Groups::a32_b16) of(Wide{}, Narrow{});                                                    \
        } else {                                                                                                    \
            of(Wide{}, Wide{});                                                                                     \
        }                                                                                                           \
    } while (0)
#define FG_LAUNCH(BM_, EPI_)                                                                                        \
    do {                                                                                                            \
        if (q.split) FG_LAUNCH_GROUPS(BM_, 1, EPI_);                                                                \
        else if (vec) f32_gemm_kernel<BM_, 1, ASRC, BSRC, EPI_, true, false, 0, 0><<<grid, FG_THREADS, 0, s>>>(p);  \
        else f32_gemm_kernel<BM_, 1, ASRC, BSRC, EPI_, false, false, 0, 0><<<grid, FG_THREADS, 0, s>>>(p);          \
    } while (0)
// What is built for a pair of sources: four groups per block (their buffers do not fit in LDS where a side is read
// across its rows: its planes are padded), and the epilogues that add a bias and a random-bias share.
template <int ASRC, int BSRC> struct FgGroups {
    static constexpr bool four = ASRC != FG_MCONT && BSRC != FG_MCONT;
    // which sides may be bf16 matrices: x and dy are as the coefficients are, z and t are fp32
    static constexpr bool matrices = ASRC != FG_NOISE_I && (BSRC == FG_KCONT || BSRC == FG_MCONT);
    static constexpr bool a16_b16 = matrices && BSRC == FG_MCONT;                               // t = dy . C, dW = dy^T . x
    static constexpr bool a16_b32 = ASRC == FG_MCONT || (ASRC == FG_KCONT && !matrices);        // dC = dy^T . z, z = x . N^T, W = C . N
    static constexpr bool a32_b16 = BSRC == FG_KCONT;                                           // y = z . C^T, W^T = N^T . C^T
    static constexpr bool biased = ASRC == FG_KCONT && BSRC == FG_KCONT, scaled = ASRC == FG_NOISE_I || BSRC == FG_NOISE_I;
};
inline bool fg_fits(const FgProduct &q)
{
    return q.a_elems < (1ll << 29) && q.b_elems < (1ll << 29) && q.M < (1ll << 30) && q.N < (1ll << 30) && q.K < (1ll << 30) && cdiv(q.N, FG_BN) <= 65535;
}
inline FgParams fg_params(const FgProduct &q)
{
    FgParams p = {};
    p.a = q.a;
    p.lda = q.lda;
    p.b = q.b;
    p.ldb = q.ldb;
    p.out = q.out;
    p.ldo = q.ldo;
    p.split_stride = q.split_stride;
    p.bias = q.bias;
    p.M = (int)q.M;
    p.N = (int)q.N;
    p.K = (int)q.K;
    p.kchunk = (int)(q.kchunk > 0 ? q.kchunk : cdiv(q.K, FG_BK) * FG_BK);
    p.a_bytes = q.a_elems * q.a_es;
    p.b_bytes = q.b_elems * q.b_es;
    p.a_es = q.a_es;
    p.b_es = q.b_es;
    p.out_bf16 = q.out_bf16;
    p.scale_bf16 = q.scale_bf16;
    p.seed = q.seed;
    p.nsR = q.nsR;
    p.nsK = q.nsK;
    p.scale = q.scale;
    p.dotm = q.dotm;
    p.lddot = q.lddot;
    p.dot_part = q.dot_part;
    p.values = q.values;
    return p;
}
// 16-byte pieces (8 of a bf16 matrix: four values) when both matrices allow them: aligned bases and leading dimensions, and the extent
// along a piece a multiple of 4 (along the rows of a matrix: the contraction; across them: the rows of the tile)
inline bool fg_vec(const FgProduct &q, int asrc, int bsrc)
{
    auto ok = [&](int src, const float *m, int64_t ld, int64_t rows) {
        if (src != FG_KCONT && src != FG_MCONT) return true;
        return fg_aligned16(m) && ld % 4 == 0 && (src == FG_KCONT ? q.K % 4 == 0 : rows % 4 == 0);
    };
    return ok(asrc, q.a, q.lda, q.M) && ok(bsrc, q.b, q.ldb, q.N);
}
template <int ASRC, int BSRC> int fg_launch(FgProduct q, int num_cus, hipStream_t s, const char *name)
{
    typedef FgGroups<ASRC, BSRC> Groups;
    if (!q.bm) {
        const FgPlan pl = !(Groups::scaled && q.scale) ? fg_plan(q.M, q.N, q.K, num_cus, 1, Groups::four) : fg_room(q.M, q.N, q.K, num_cus, q.K, 1);
        q.bm = pl.bm;
        q.groups = pl.groups;
    }
    if (!fg_fits(q)) return RDB_E_UNSUPPORTED;
    if constexpr (BSRC == FG_NOISE_M) q.values.slices = fg_value_slices(q.values, cdiv(q.M, q.bm) * cdiv(q.N, FG_BN), FG_THREADS * (q.split ? q.groups : 1));
    const FgParams p = fg_params(q);
    FgCarried carried = {};
    const int splits = (int)cdiv(q.K, p.kchunk);
    const int64_t tiles = cdiv(q.M, q.bm) * cdiv(q.N, FG_BN);
    const int groups = q.split ? q.groups : 1;
    if (BSRC == FG_NOISE_I) carried.sum_slices = (int)cdiv(cdiv(q.sum.blocks, groups), tiles);
    if (fg_carries_bias(ASRC, BSRC) && q.bias_grad.blocks) {
        const BiasGrad &g = q.bias_grad;
        if (q.split && bias_direct(g.rows, g.n, g.bf16 ? 2 : 4, g.k, num_cus, FG_THREADS * groups)) carried.bias_slices = (int)cdiv(g.blocks, tiles);
        else if (int rc = bias_direct_launch(g, s)) return rc;   // too few threads to a block, or fp32 matrix instructions (rdb_set_f32_split), whose kernels carry nothing
    }
    const int more = carried.sum_slices + carried.bias_slices;
    if (more) {
        static_cast<FgParams &>(carried) = p;
        carried.sum = q.sum;
        carried.bias_grad = q.bias_grad;
    }
    const bool vec = fg_vec(q, ASRC, BSRC);
    const bool a16 = (ASRC == FG_KCONT || ASRC == FG_MCONT) && q.a_es == 2, b16 = (BSRC == FG_KCONT || BSRC == FG_MCONT) && q.b_es == 2;
    if (q.split && ((a16 && b16) ? !Groups::a16_b16 : a16 ? !Groups::a16_b32 : b16 && !Groups::a32_b16)) return RDB_E_UNSUPPORTED;
    const dim3 grid((unsigned)cdiv(q.M, q.bm), (unsigned)cdiv(q.N, FG_BN), (unsigned)(splits + (BSRC == FG_NOISE_M ? q.values.slices : 0) + more));
    auto run = [&](auto epi_) {
        constexpr int EPI = decltype(epi_)::value;
        if (q.bm == 128 && q.groups == 2) FG_LAUNCH_GROUPS(128, 2, EPI);
        else if (q.bm == 128) FG_LAUNCH(128, EPI);
        else if (q.groups == 1) FG_LAUNCH(64, EPI);
        else if (q.groups == 2) FG_LAUNCH_GROUPS(64, 2, EPI);
        else if constexpr (Groups::four) FG_LAUNCH_GROUPS(64, 4, EPI);
    };
    if constexpr (BSRC == FG_NOISE_1D) {   // the random-bias products: added on top of an output, and / or reduced against a matrix
        if (q.scale) run(std::integral_constant<int, FG_ADD_SCALED>{});
        else if (q.dotm) run(std::integral_constant<int, FG_DOT>{});
        else run(std::integral_constant<int, FG_STORE>{});   // a range's share, for f32_rbias_sum_kernel
    } else if (Groups::scaled && q.scale) {   // materialising W with its random-bias share
        if constexpr (Groups::scaled) {
            if (q.bm == 128) FG_LAUNCH(128, FG_STORE_RBIAS);
            else FG_LAUNCH(64, FG_STORE_RBIAS);
        }
    } else {
        if constexpr (Groups::biased) {
            if (q.bias) run(std::integral_constant<int, FG_STORE_BIAS>{});
            else run(std::integral_constant<int, FG_STORE>{});
        } else {
            run(std::integral_constant<int, FG_STORE>{});
        }
    }
    return check_launch(name);
}

#undef FG_LAUNCH
#undef FG_LAUNCH_GROUPS

#define FG_PAIR(A_, B_) template int fg_launch<A_, B_>(FgProduct, int, hipStream_t, const char *)
#ifndef RDB_F32_INSTANTIATE
extern FG_PAIR(FG_KCONT, FG_KCONT);
extern FG_PAIR(FG_KCONT, FG_MCONT);
extern FG_PAIR(FG_MCONT, FG_MCONT);
extern FG_PAIR(FG_KCONT, FG_NOISE_M);
extern FG_PAIR(FG_KCONT, FG_NOISE_I);
extern FG_PAIR(FG_NOISE_I, FG_KCONT);
extern FG_PAIR(FG_KCONT, FG_NOISE_1D);
#endif

}  // namespace rdb
