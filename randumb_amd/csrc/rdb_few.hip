// Forward pass of a matrix-coef layer for few tokens (a served model generating, short prompts): z = x . N^T, y = z . C^T (+ bias) on
// the matrix cores with 16 x 16 tiles, at fp32 accuracy whatever the operands' type, in one to three launches.
//
// What bounds it is latency: 16 tokens x 4096 -> 11008, k = 256 move 6 MB and multiply next to nothing.  Contracting blocks (16 coefficients
// x a chunk of in_f x up to 32 tokens, each noise value hashed once for all of them) leave partial sums of z; expanding blocks (64
// output features x 16 tokens, or 32 where there are more blocks than the chip runs at once) have their rows of C in registers by
// the time these are there, add them up in chunk order, and multiply.  In one launch the contracting blocks come first and publish
// a tag each (rdb_common.hpp); where the partial sums are so many that reading them around the dies' L2 caches costs more than a
// launch, the two kinds of block are two launches of the same kernel.
// us per call, three launches on the vector ALU (or the kernels for many tokens) -> here: 16 tokens x 4096 -> 11008, k = 256, bf16 14.5 ->
// 11.5; 1 x 7512 -> 2376, k = 512, bf16 34.6 -> 14.0; 5 x 1001 -> 999, k = 99, bf16 17.1 -> 7.5; 22 x 264 -> 352, k = 64, fp32 17.7 -> 8.6;
// 1 x 4096 -> 4096, k = 16, fp32: even (8.6 to 9.0 either way); 64 x 4096 -> 11008, k = 256, bf16 29.2 -> 17.9; 128 x 8192 -> 1024, k = 128, bf16 28.0 -> 15.2;
// 256 x 512 -> 512, k = 128, fp32 17.4 -> 9.8.  What is left is launches and memory round trips: x in, partial sums out and in, y out.
// Tokens split finer than they were (48 to a block of either kind): 48 x 768 -> 3072, k = 256, bf16 15.5 -> 10.7, 32 tokens 13.6 -> 10.6.
//
// fp32 accuracy: a noise value is exactly three bf16 parts, so its products with bf16 activations are exact in three matrix instructions;
// so are those of z (fp32) with bf16 coefficients.  fp32 activations and coefficients are split as well: the six largest of the nine
// products (rdb_f32.hpp says what is left out).  Infinities come out as they do of fp32 products: an infinite fp32 value is split into
// (largest, largest, infinity), an infinite bf16 value meets its partner's lower parts as the largest finite one, and sums of y that
// are not finite are done again with parts of one sign.
#include "rdb_common.hpp"
#include <algorithm>
#include <type_traits>

namespace rdb {

int f32_split_mode();   // rdb_f32.hip
int num_compute_units();   // rdb_error.hip

constexpr int FEW_ROWS = 64;       // output features of an expanding block: 16 a wave
constexpr int FEW_COEFS = 16;      // coefficients of a contracting block
constexpr int FEW_TOKENS = 256, FEW_K = 512;   // z's three parts of 32 tokens in LDS: at most 100 KB

struct FewParams {
    void *y;
    const void *x, *coef, *bias;
    int64_t ldx, ldy;
    float *part;   // [chunks][tiles of 16 tokens, or fewer if there are no more][ranges of 16 coefficients][tokens of a tile][16]
    int T, in_f, out_f, k, chunks, ranges;
    int tile, tiles;     // tokens of a tile, tiles
    int c_groups;        // groups of tokens of the contracting blocks
    int wave_values;     // contraction values per wave and chunk: a multiple of 32
    int x_vec, c_vec, y_vec;   // 16-byte pieces of x and C, 4 values of y at a time
    uint32_t seed;
    int c_blocks;        // contracting blocks of this launch: they come first
    int e_blocks;        // expanding blocks of a group of tokens
    unsigned long long *slots;   // NULL, or one tag per contracting block
    unsigned long long tag;
    int tags;
    SyncWait wait;
    unsigned int *count;
    int consumers;
};

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));

// eight values as three bf16 fragments
struct Split8 {
    bf16x8 h, m, l;
};
__device__ __forceinline__ void few_split2(float v0, float v1, uint32_t &h, uint32_t &m, uint32_t &l)
{
    constexpr float top = 3.3895313892515355e38f;   // the largest bf16: nothing below an infinity rounds to one
    h = f32x2_to_bf16x2(__builtin_amdgcn_fmed3f(v0, -top, top), __builtin_amdgcn_fmed3f(v1, -top, top));
    v0 -= __uint_as_float(h << 16);
    v1 -= __uint_as_float(h & 0xffff0000u);
    m = f32x2_to_bf16x2(__builtin_amdgcn_fmed3f(v0, -top, top), __builtin_amdgcn_fmed3f(v1, -top, top));
    l = f32x2_to_bf16x2(v0 - __uint_as_float(m << 16), v1 - __uint_as_float(m & 0xffff0000u));
}
__device__ __forceinline__ Split8 few_split8(const f32x8 &v)
{
    u32x4_t h, m, l;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint32_t a, b, c;
        few_split2(v[2 * e], v[2 * e + 1], a, b, c);
        h[e] = a;
        m[e] = b;
        l[e] = c;
    }
    return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}
// The same with the parts cut off and not rounded, all of one sign: no two of a product's terms overflow to different sides.  What is
// left out of a product of two such splits is up to 2^-21 of it and of its sign, so only sums that came out not finite are taken from it.
__device__ __forceinline__ Split8 few_split8_any(const f32x8 &v)
{
    constexpr float top = 3.40282346638528859812e38f;
    u32x4_t p[3];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float rest = v[e];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const uint32_t part = __float_as_uint(q < 2 ? __builtin_amdgcn_fmed3f(rest, -top, top) : rest) & 0xffff0000u;
            rest -= __uint_as_float(part);
            p[q][e / 2] = e & 1 ? p[q][e / 2] | part : part >> 16;
        }
    }
    return {__builtin_bit_cast(bf16x8, p[0]), __builtin_bit_cast(bf16x8, p[1]), __builtin_bit_cast(bf16x8, p[2])};
}
// eight values back from their parts (exactly)
__device__ __forceinline__ f32x8 few_join8(const Split8 &z)
{
    const u32x4_t h = __builtin_bit_cast(u32x4_t, z.h), m = __builtin_bit_cast(u32x4_t, z.m), l = __builtin_bit_cast(u32x4_t, z.l);
    f32x8 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        v[2 * e] = (__uint_as_float(h[e] << 16) + __uint_as_float(m[e] << 16)) + __uint_as_float(l[e] << 16);
        v[2 * e + 1] = (__uint_as_float(h[e] & 0xffff0000u) + __uint_as_float(m[e] & 0xffff0000u)) + __uint_as_float(l[e] & 0xffff0000u);
    }
    return v;
}
// infinities as the largest finite value of their sign, for the products with the lower parts of the other side
__device__ __forceinline__ bf16x8 few_finite(const bf16x8 &v)
{
    u32x4_t w = __builtin_bit_cast(u32x4_t, v);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t lo = w[e] & 0x7fffu, hi = (w[e] >> 16) & 0x7fffu;
        w[e] = (w[e] & 0x80008000u) | min(lo, 0x7f7fu) | (min(hi, 0x7f7fu) << 16);
    }
    return __builtin_bit_cast(bf16x8, w);
}
__device__ __forceinline__ f32x4 few_mma(const bf16x8 &a, const bf16x8 &b, const f32x4 &c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// Eight consecutive values of a row as they are in memory; a fragment lane's share of a matrix operand
template <typename E> struct FewRaw;
template <> struct FewRaw<bf16_t> {
    u32x4_t w;
};
template <> struct FewRaw<float> {
    f32x4 lo, hi;
};
// values at .. at + 7 of the row at `row`, zeros from n on and where !ok
template <typename E> __device__ __forceinline__ FewRaw<E> few_load(const E *row, int at, int n, bool ok, int vec)
{
    FewRaw<E> r;
    if (vec) {   // n is a multiple of 8: a piece lies inside or outside
        const bool in = ok && at < n;
        const E *src = in ? row + at : row;
        if constexpr (sizeof(E) == 2) {
            r.w = *reinterpret_cast<const u32x4_t *>(src);
            if (!in) r.w = u32x4_t{0, 0, 0, 0};
        } else {
            r.lo = *reinterpret_cast<const f32x4 *>(src);
            r.hi = *reinterpret_cast<const f32x4 *>(src + 4);
            if (!in) r.lo = r.hi = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        return r;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const bool in = ok && at + e < n;
        const E v = row[in ? at + e : 0];
        if constexpr (sizeof(E) == 2) {
            const uint32_t b = in ? (uint32_t)v << (16 * (e & 1)) : 0u;
            r.w[e / 2] = e & 1 ? r.w[e / 2] | b : b;
        } else {
            (e < 4 ? r.lo : r.hi)[e & 3] = in ? v : 0.0f;
        }
    }
    return r;
}

// acc (the large products) and low (the small ones) += A . B^T, A from memory, B in three parts
template <typename E> struct FewSide;
template <> struct FewSide<bf16_t> {
    bf16x8 v, f;
    template <bool ANY = false> __device__ __forceinline__ void set(const FewRaw<bf16_t> &r)
    {
        v = __builtin_bit_cast(bf16x8, r.w);
        f = few_finite(v);
    }
    // the side from memory as the A operand (rows of the result)
    __device__ __forceinline__ void mma_a(f32x4 &acc, f32x4 &low, const Split8 &b) const
    {
        low = few_mma(f, b.l, low);
        low = few_mma(f, b.m, low);
        acc = few_mma(v, b.h, acc);
    }
};
template <> struct FewSide<float> {
    Split8 s;
    template <bool ANY = false> __device__ __forceinline__ void set(const FewRaw<float> &r)
    {
        const f32x8 v = {r.lo[0], r.lo[1], r.lo[2], r.lo[3], r.hi[0], r.hi[1], r.hi[2], r.hi[3]};
        s = ANY ? few_split8_any(v) : few_split8(v);
    }
    __device__ __forceinline__ void mma_a(f32x4 &acc, f32x4 &low, const Split8 &b) const
    {
        low = few_mma(s.m, b.m, low);
        low = few_mma(s.l, b.h, low);
        low = few_mma(s.h, b.l, low);
        low = few_mma(s.m, b.h, low);
        low = few_mma(s.h, b.m, low);
        acc = few_mma(s.h, b.h, acc);
    }
};

// Block (range, chunk, group) of WAVES waves: z[TT tiles of tokens][16 coefficients] over the chunk, each wave its share of it.
template <typename E, int TT, int WAVES> __device__ __forceinline__ void few_contract(const FewParams &p, int b, float *__restrict__ lds)
{
    constexpr int FEW_STEPS = 16 / WAVES;   // steps of 32 contraction values a wave hashes ahead of its products
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r = lane & 15, g = lane >> 4;
    int range = b % p.ranges, ch = b / p.ranges, group = 0;
    if (TT > 1) {   // a group's chunk is read by blocks of one die where that comes out even
        const int pieces = p.chunks * p.c_groups;
        range = b / pieces;
        ch = (b - range * pieces) / p.c_groups;
        group = b - range * pieces - ch * p.c_groups;
    }
    const int m = range * FEW_COEFS + r, tile0 = group * TT, t0 = tile0 * 16, T = min(TT * 16, p.T - t0);
    const int i_begin = (ch * WAVES + wave) * p.wave_values;
    const E *const x = static_cast<const E *>(p.x) + (int64_t)t0 * p.ldx;
    const E *row[TT];
    bool live[TT];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
        live[tt] = tt * 16 + r < T;
        row[tt] = x + (int64_t)(live[tt] ? tt * 16 + r : 0) * p.ldx;
    }
    f32x4 acc[TT], low[TT];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) acc[tt] = low[tt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int i0 = 0; i0 < p.wave_values; i0 += 32 * FEW_STEPS) {
        FewRaw<E> raw[FEW_STEPS];
        auto request = [&](int tt) {
#pragma unroll
            for (int s = 0; s < FEW_STEPS; ++s)
                if (i0 + s * 32 < p.wave_values) raw[s] = few_load<E>(row[tt], i_begin + i0 + s * 32 + g * 8, p.in_f, live[tt], p.x_vec);
        };
        request(0);
        // values past in_f meet zeros of x
        Split8 noise[FEW_STEPS];
#pragma unroll
        for (int s = 0; s < FEW_STEPS; ++s)
            if (i0 + s * 32 < p.wave_values) {
                const uint32_t first = sq5_first((uint32_t)(i_begin + i0 + s * 32 + g * 8), (uint32_t)m, p.seed);
                f32x8 v;
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = sq5_unit(sq5_tail(first + (uint32_t)e * PN1));
                noise[s] = few_split8(v);
            }
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
            if (tt * 16 >= T) break;   // uniform
            FewSide<E> a[FEW_STEPS];
#pragma unroll
            for (int s = 0; s < FEW_STEPS; ++s)
                if (i0 + s * 32 < p.wave_values) a[s].set(raw[s]);
            if (tt + 1 < TT && (tt + 1) * 16 < T) request(tt + 1);
#pragma unroll
            for (int s = 0; s < FEW_STEPS; ++s)
                if (i0 + s * 32 < p.wave_values) a[s].mma_a(acc[tt], low[tt], noise[s]);
        }
    }
    // result element j of lane (r, g): token 4 g + j, coefficient r; the waves' sums meet in LDS
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int j = 0; j < 4; ++j) lds[((wave * TT + tt) * 16 + g * 4 + j) * 16 + r] = acc[tt][j] + low[tt][j];
    __syncthreads();
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
        const int t = tt * 16 + (tid >> 4);
        if (t < T && (WAVES <= 4 || tid < 256)) {
            float *const out = p.part + (((int64_t)ch * p.tiles + tile0 + tt) * p.ranges + range) * p.tile * 16;
            float v = lds[tt * 256 + tid];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) v += lds[(w * TT + tt) * 256 + tid];
            __hip_atomic_store(out + tid, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// Block: 64 output features, TT tiles of tokens.  MANY: tiles have 16 tokens.  Waves behind the first four (a block as large as a contracting one) add z up and leave
template <typename E, int KS, int TT, bool MANY, int WAVES> __device__ __forceinline__ void few_expand(const FewParams &p, int b, unsigned char *__restrict__ smem)
{
    constexpr int THREADS = WAVES * 64, KW = KS * 32, LD = KW + 8;   // 16 bytes of padding: 16 rows' pieces lie in different banks
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int tile = MANY ? 16 : p.tile, tile0 = MANY ? b / p.e_blocks * TT : 0, t0 = tile0 * 16, T = min(TT * 16, p.T - t0), ob = MANY ? b % p.e_blocks : b, o0 = ob * FEW_ROWS + wave * 16;
    bf16_t *const planes = reinterpret_cast<bf16_t *>(smem);
    const int PLANE = (T + 15) / 16 * 16 * LD;
    E *const y = static_cast<E *>(p.y) + (int64_t)t0 * p.ldy;
    // the wave's rows of C, before anything is waited for
    FewRaw<E> c[KS];
    {
        const bool ok = (WAVES <= 4 || wave < 4) && o0 + r < p.out_f;
        const E *const row = static_cast<const E *>(p.coef) + (int64_t)(ok ? o0 + r : 0) * p.k;
#pragma unroll
        for (int s = 0; s < KS; ++s) c[s] = few_load<E>(row, s * 32 + g * 8, p.k, ok, p.c_vec);
    }
    if (p.slots) {
        __shared__ int verdict;
        const int n = p.tags;
        if (tid < 64) {
            bool there = false;
            for (int it = 0; it < p.wait.polls && !there; ++it) {
                bool mine = true;
                for (int i = lane; i < n; i += 64) mine &= __hip_atomic_load(p.slots + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == p.tag;
                there = __all(mine);
                if (!there) __builtin_amdgcn_s_sleep(10);
            }
            if (there) {   // the last of the consumers clears the slots (a recorded launch runs again with the same tag)
                unsigned int old = 0;
                if (lane == 0) old = __hip_atomic_fetch_add(p.count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                old = (unsigned int)__builtin_amdgcn_readfirstlane((int)old);
                if (old == (unsigned int)(p.consumers - 1))
                    for (int i = lane; i < n; i += 64) __hip_atomic_store(p.slots + i, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else if (lane == 0) {
                if (p.wait.err) atomicOr(p.wait.err, 2u);
                atomicAdd(p.wait.giveups, 1u);
            }
            if (tid == 0) verdict = there ? 1 : 0;
        }
        __syncthreads();
        if (verdict == 0) {   // gave up: the block's share of the output becomes NaN, never a sum of whatever is in memory
            for (int i = tid; i < T * FEW_ROWS; i += THREADS) {
                const int t = i / FEW_ROWS, o = ob * FEW_ROWS + i % FEW_ROWS;
                if (o < p.out_f) elem<E>::store(y + (int64_t)t * p.ldy + o, __uint_as_float(0x7fc00000u));
            }
            return;
        }
    }
    // z: four coefficients of a token at a time, the chunks' sums in chunk order, then its three parts
    const int per = p.ranges * tile, n4 = min(TT, p.tiles - tile0) * per * 4;
    const int64_t stride = (int64_t)p.tiles * per * 16, first = (int64_t)tile0 * per * 16;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(p.part, 0, (int)(stride * p.chunks * 4), 0x00020000);
    // IB entries of CB chunks in flight
    auto add_up = [&](auto ib_, auto cb_) __attribute__((always_inline)) {
        constexpr int IB = decltype(ib_)::value, CB = decltype(cb_)::value;
        for (int i0 = tid; i0 < n4; i0 += THREADS * IB) {
            f32x4 v[IB];
            for (int c0 = 0; c0 < p.chunks; c0 += CB) {
                f32x4 u[IB][CB];
#pragma unroll
                for (int i = 0; i < IB; ++i)
#pragma unroll
                    for (int q = 0; q < CB; ++q) {
                        const int at = (int)(((int64_t)min(c0 + q, p.chunks - 1) * stride + first + (int64_t)min(i0 + i * THREADS, n4 - 1) * 4) * 4);
                        u[i][q] = __builtin_bit_cast(f32x4, p.slots ? __builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, SCOPE_DEVICE) : __builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, 0));
                    }
#pragma unroll
                for (int i = 0; i < IB; ++i)
#pragma unroll
                    for (int q = 0; q < CB; ++q) {
                        if (c0 + q >= p.chunks) continue;
                        v[i] = c0 + q == 0 ? u[i][q] : v[i] + u[i][q];
                    }
            }
#pragma unroll
            for (int i = 0; i < IB; ++i) {
                const int e = i0 + i * THREADS;
                if (e >= n4) continue;
                const int sub = TT > 1 && (e >> 2) >= per ? 1 : 0, rt = (e >> 2) - sub * per, range = rt / tile, t = sub * 16 + rt - range * tile, m = range * FEW_COEFS + (e & 3) * 4;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (m + j >= p.k) v[i][j] = 0.0f;
                uint2 h, mm, l;
                few_split2(v[i][0], v[i][1], h.x, mm.x, l.x);
                few_split2(v[i][2], v[i][3], h.y, mm.y, l.y);
                bf16_t *const dst = planes + t * LD + m;
                *reinterpret_cast<uint2 *>(dst) = h;
                *reinterpret_cast<uint2 *>(dst + PLANE) = mm;
                *reinterpret_cast<uint2 *>(dst + 2 * PLANE) = l;
            }
        }
    };
    if (p.chunks == 1) add_up(std::integral_constant<int, 16>{}, std::integral_constant<int, 1>{});
    else if (p.chunks <= 4) add_up(std::integral_constant<int, 4>{}, std::integral_constant<int, 4>{});
    else add_up(std::integral_constant<int, 2>{}, std::integral_constant<int, 8>{});
    // coefficients beyond the last range meet zeros of C: they must be finite
    const int tail4 = (KW - p.ranges * FEW_COEFS) / 4;
    if (tail4 > 0)
        for (int e = tid; e < 3 * T * tail4; e += THREADS) {
            const int row = e / tail4, pl = row / T;
            *reinterpret_cast<uint2 *>(planes + pl * PLANE + (row - pl * T) * LD + p.ranges * FEW_COEFS + (e - row * tail4) * 4) = make_uint2(0u, 0u);
        }
    __syncthreads();
    if (WAVES > 4 && wave >= 4) return;
    f32x4 acc[TT], low[TT];
    auto product = [&](auto any) __attribute__((always_inline)) {
        constexpr bool ANY = decltype(any)::value;
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) acc[tt] = low[tt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            if (s * 32 >= p.k) break;   // uniform
            FewSide<E> a;
            a.template set<ANY>(c[s]);
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
                if (tt * 16 >= T) break;
                const bf16_t *const src = planes + (tt * 16 + r) * LD + s * 32 + g * 8;   // tokens from T on: whatever lies there, in columns nobody stores
                Split8 z = {*reinterpret_cast<const bf16x8 *>(src), *reinterpret_cast<const bf16x8 *>(src + PLANE), *reinterpret_cast<const bf16x8 *>(src + 2 * PLANE)};
                if (ANY) z = few_split8_any(few_join8(z));
                a.mma_a(acc[tt], low[tt], z);
            }
        }
    };
    product(std::false_type{});
    float zero = 0.0f;   // stays so as long as every sum is finite
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int j = 0; j < 4; ++j) zero = tt * 16 + r < T ? fmaf(acc[tt][j] + low[tt][j], 0.0f, zero) : zero;
    if (__any(zero != 0.0f)) {   // once more, for the sums that are not finite: the others stay as they would be without these beside them
        f32x4 sum[TT];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) sum[tt] = acc[tt] + low[tt];
        product(std::true_type{});
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (sum[tt][j] * 0.0f == 0.0f) {
                    acc[tt][j] = sum[tt][j];
                    low[tt][j] = -0.0f;
                }
    }
    // result element j of lane (r, g): output feature o0 + 4 g + j, token r
    const int o = o0 + g * 4;
    float bv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) bv[j] = p.bias && o + j < p.out_f ? elem<E>::load(static_cast<const E *>(p.bias) + o + j) : 0.0f;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
        const int t = tt * 16 + r;
        if (t >= T || o >= p.out_f) continue;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = acc[tt][j] + low[tt][j] + bv[j];
        E *const dst = y + (int64_t)t * p.ldy + o;
        if (p.y_vec) {   // out_f is a multiple of 4
            if constexpr (sizeof(E) == 2) *reinterpret_cast<uint2 *>(dst) = make_uint2(f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3]));
            else *reinterpret_cast<f32x4 *>(dst) = f32x4{v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (o + j < p.out_f) elem<E>::store(dst + j, v[j]);
        }
    }
}

// the chunks' sums, in chunk order, into chunk 0's place
__global__ __launch_bounds__(256) void few_sum_kernel(float *__restrict__ part, int64_t n4, int chunks)
{
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n4) return;
    f32x4 *const at = reinterpret_cast<f32x4 *>(part) + e;
    f32x4 v = *at;
    for (int c0 = 1; c0 < chunks; c0 += 8) {
        f32x4 u[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) u[q] = at[(int64_t)min(c0 + q, chunks - 1) * n4];
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (c0 + q < chunks) v += u[q];
    }
    *at = v;
}

// TC, TE: tiles of tokens of a contracting and of an expanding block
template <typename E, int KS, int TC, int TE, int WAVES> __global__ __launch_bounds__(WAVES * 64, 1) void few_fwd_kernel(FewParams p)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int b = blockIdx.x;
    if (b >= p.c_blocks) {
        few_expand<E, KS, TE, TC == 2, WAVES>(p, b - p.c_blocks, smem);
        return;
    }
    if (p.slots && threadIdx.x == 0) __hip_atomic_store(p.slots + b, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // a replay may find its tag
    few_contract<E, TC, WAVES>(p, b, reinterpret_cast<float *>(smem));
    if (!p.slots) return;
    if (b == 0 && threadIdx.x == 0) __hip_atomic_store(p.count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    publish_tag(p.slots + b, p.tag);
}

// the contracting blocks of the form in two launches
template <typename E, int TC, int WAVES> __global__ __launch_bounds__(WAVES * 64, 1) void few_contract_kernel(FewParams p)
{
    __shared__ __align__(16) float lds[WAVES * TC * 256];
    few_contract<E, TC, WAVES>(p, blockIdx.x, lds);
}

// ----------------------------------------------------------------------------------------------- host side
// Chunks: about eight of them (sixteen where there is one range of coefficients), of 128 to 512 values (a contracting block hashes a chunk for 16 coefficients: 128 values cost it 0.6 us;
// an expanding block reads eight at a time: 1 x 4096 -> 4096, k = 16: chunks of 128, 256, 512, 1024: 8.9, 8.0, 8.2, 10.9 us).
// waves: a wave hashes 32 contraction values for its 16 coefficients, which a SIMD with a single wave does at half its rate, and the blocks are fewer than the chip holds; so
// a chunk of 512 is 16 waves, or 8 where an expanding block is as large (more have no registers for that; k > 256: four).  us per call, four waves -> so: 16 x 4096 -> 11008, k = 256,
// bf16 11.3 -> 10.7 to 11.2; 64 tokens 18.6 -> 17.3; 8 x 8192 -> 8192, k = 512 21.9 -> 19.9; in one launch: 1 x 4096 -> 4096, k = 16, fp32 8.9 -> 8.1; 4 x 2000 -> 5000, k = 100 9.5 -> 8.7;
// 16 x 4096 -> 4096, k = 128 11.1 -> 10.6.  (Chunks of 1024 and 2048 in 16 waves, half and a quarter of the partial sums: 11.8 and 15.1 for the first.  Expanding blocks of eight waves in
// a launch of their own: 64 tokens 20.7.)  In one launch four again where eight cost more.  Of eight waves a unit has one block: contracting
// blocks of fp32 that are more than the units, 460 x 1862 -> 164, k = 40, 360 blocks 16.8, four 15.4; 511 x 5005 -> 267, k = 47 24.9, 22.7 (bf16 either way: 106 x 1923 -> 371, k = 136 16.7, 15.9; 242 x 8261 -> 92, k = 27 18.8, 20.9; fewer
// blocks: 235 x 3014 -> 491, k = 57, 192 and 120 14.8, 17.6), and, of one tile of tokens, k > 128 that is no multiple of 8, whose rows of C are read a value at a time, with more blocks in all than
// units, 1 x 7728 -> 273, k = 255, 261 of them, 15.2, 12.5; 4 x 1833 -> 9483, k = 213 14.0, 12.2 (k = 192, 2 x 5225 -> 7979 13.2, 14.8), or chunks of 256, one step a wave, up to 8 tokens: 3 x 1425 -> 4496, k = 187, fp32 11.2, 10.6; 74
// and 87 sizes, bf16 and fp32, 0.98 and 0.965 times eight's, but 1.03 and 1.055 where k is a multiple of 8 (5 x 1775 -> 6639, k = 176, bf16 10.2, 11.0), and 15 x 1202 -> 460, k = 208 10.4, 11.8.
// The number depends on the layer and its tokens alone, so that the same sums come out in one launch and in two.
// te: tiles of an expanding block.  Finer is sooner ready while the blocks run side by side, two (of k > 128: one) to a compute unit: 64 x
// 768 -> 3072, k = 64: 8.2 us, two tiles 9.1; 80 x 8192 -> 8192, k = 64, 640 blocks of one tile: 18.7, two tiles 15.1.
// sum: beyond 200 KB of partial sums for a block they are added up once, by a launch of its own, and not by every expanding block
// (48 to a block, 32 tokens x 4096 -> 11008, k = 256: 15.6 -> 14.9 us; 16 tokens, 131 KB: 11.5, and 12.7 with it).
// one: a single launch where the expanding blocks are few and the partial sums of each small; tags and reads that go around L2 cost many
// blocks more than a launch does (16 x 4096 -> 11008, k = 256: two launches 11.5, one 13.5), but a program's host takes 9.0 to 11.7 us (by
// the machine and by what the program does between calls) to issue two, and those calls then take that.  us of a call in one launch, which
// the host does not hold up: 5 x 1001 -> 999, k = 99: 7.8; 48 x 768 -> 768, k = 64: 8.3; 100 x 264 -> 352, k = 64: 8.7; 32 x 1024 -> 2048,
// k = 128, 64 blocks of 64 KB: 9.2; 4 x 2048 -> 10000, k = 32, 157 blocks: 9.0; 64 x 768 -> 2048, k = 64, 128 blocks: 9.9.  At the line the
// two are about even, whichever the host: 256 x 512 -> 640, k = 128, 160 blocks of 32 KB and 256 tags: 10.7 in bf16 and 11.6 in fp32, two launches
// 9.3 and 9.7 on the fastest host, 11.7 and 11.5 in a program; 224 x 512 -> 640, k = 96, 140 blocks, 168 tags, bf16: 12.2, and 9.5 or 11.3.
// More blocks, up to 192 of 16 KB and 32 tags: of one tile of tokens, where two launches wait for the host and one is mostly sooner than that (on the device, two and one, and two called in a loop: 8 x 515 -> 10437, k = 14 8.0,
// 9.0, 10.4; 4 x 448 -> 10988, k = 5 7.9, 8.7, 9.7; 1 x 267 -> 10914, k = 48 7.4, 9.6, 9.8); of several only for sizes that are other kernels' in two launches (few_one_or_none): 48 x 237 -> 3841, k = 116 15.5, 10.6; 107 x 226 -> 1452,
// k = 21 13.5, 10.2, but 97 x 91 -> 1616, k = 18 9.8, 10.6; others: 51 x 327 -> 2944, k = 32 8.9, 10.9; 20 x 1840 -> 5285, k = 8 9.1, 11.2.
struct FewPlan {
    int wave_values, waves, chunks, ranges;   // waves: of a contracting block, and of both kinds where they are one launch
    int tile, tiles, tc, te;
    int c_blocks, e_blocks;
    bool sum, one;
    int64_t part_bytes;
};
// short contractions in bf16, which are other kernels' in two launches (few_pays)
static bool few_one_or_none(const rdb_linear_desc *d)
{
    return d->act_dtype == RDB_BF16 && d->in_f < 512 && (d->k > 64 || (d->tokens > 96 && d->in_f > 128));
}
static FewPlan few_plan(const rdb_linear_desc *d)
{
    FewPlan f;
    f.ranges = (int)cdiv(d->k, FEW_COEFS);
    f.tile = (int)std::min<int64_t>(d->tokens, 16);
    f.tiles = (int)cdiv(d->tokens, f.tile);
    f.tc = f.tiles > 1 ? 2 : 1;
    const int64_t rows = cdiv(d->out_f, FEW_ROWS), c_groups = cdiv(f.tiles, f.tc);
    f.te = f.tiles > 1 && rows * f.tiles > (d->k <= 128 ? 512 : 256) ? 2 : 1;
    int64_t chunk = 128;
    while (chunk < 512 && chunk * (f.ranges == 1 ? 16 : 8) < d->in_f) chunk *= 2;
    if (c_groups > 1)
        while ((chunk < 1024 && cdiv(d->in_f, chunk) * f.ranges * c_groups > 512) || cdiv(d->in_f, chunk) > 64) chunk *= 2;   // two blocks a compute unit; the workspace
    const int64_t per_chunk = (int64_t)f.ranges * f.tile * FEW_COEFS * 4;   // of a tile
    f.sum = cdiv(d->in_f, chunk) * per_chunk * std::min(f.te, f.tiles) > 200 * 1024;
    if (f.sum && chunk > 256 && c_groups == 1) chunk = 256;
    f.chunks = (int)cdiv(d->in_f, chunk);
    f.part_bytes = f.chunks * per_chunk * f.tiles;
    f.c_blocks = (int)(f.chunks * f.ranges * c_groups);
    f.e_blocks = (int)(rows * cdiv(f.tiles, f.te));
    const int64_t block_bytes = f.chunks * per_chunk * std::min(f.te, f.tiles);   // what an expanding block reads
    f.one = !f.sum && ((f.e_blocks <= 64 && block_bytes <= 100 * 1024) || (f.e_blocks <= 160 && block_bytes <= 32 * 1024) ||
                       ((f.tc == 1 || few_one_or_none(d)) && f.e_blocks <= 192 && block_bytes <= 16 * 1024 && f.c_blocks <= 32));
    const bool four = d->k > 256 || (f.tc == 1 ? d->k > 128 && d->k % 8 && (f.c_blocks + f.e_blocks > num_compute_units() || (chunk <= 256 && f.tile <= 8))
                                               : d->act_dtype == RDB_F32 && f.c_blocks > num_compute_units());
    f.waves = (int)std::min<int64_t>(f.one ? (four ? 4 : 8) : 16, chunk / 32);
    f.wave_values = (int)chunk / f.waves;
    return f;
}

// Where these kernels are ahead of those of rdb_smallk.hip, rdb_factored.hip and rdb_f32.hip.  `units` are the expanding blocks of one
// tile of tokens: each splits its tokens' z again, so the more of them there are, and the larger k, the sooner the kernels that
// make z once for wide tiles win; fp32 multiplies twice as much.  us per call, those kernels -> here:
//   k <= 64    128 x 2048 -> 2048, k = 64: bf16 16.1 -> 9.1, fp32 17.1 -> 10.0; 128 x 3000 -> 11008, k = 64 (1376 units): 18.9 ->
//              14.1 and 19.6 -> 16.8; 256 x 8192 -> 8192 (2048): fp32 24.4 -> 27.9
//   k <= 128   128 x 8192 -> 8192: bf16 25.8 -> 18.3, fp32 25.1 -> 22.3 (1024 units); 192 (1536): 29.7 -> 23.1, fp32 26.1 -> 30.0
//   k <= 256   128 x 4096 -> 4096: bf16 20.9 -> 18.5, fp32 24.6 -> 22.2 (512 units); 160 (640): 22.4 -> 23.0 and 25.6 -> 30.5;
//              96 x 4096 -> 11008: 39 -> 22.3 and 39.4 -> 32.1; fp32 48 x 5000 -> 600, k = 200: 16.6 -> 19.1
//   beyond     64 x 1024 -> 4096, k = 512: bf16 17.8 -> 16.0; 64 x 1504 -> 6000, k = 304 (376 units): 17.1 -> 18.5;
//              fp32 32 x 8192 -> 11008, k = 512: 39 -> 33, 48 tokens 33 -> 50
// bf16 contractions of at most 512 are short for the kernels of rdb_factored.hip too, which take one launch where a program's host needs 10.7 us
// for two (no gradients wanted; 128 x 320 -> 640, k = 160: 10.2 -> 11.0): 160 x 384 -> 8000, k = 24 (1250 units): 10.7 -> 11.1;
// 128 x 512 -> 4096, k = 256 (512 units): 12.8 -> 13.1; 64 tokens (256): 12.4 -> 10.1.
// Beyond 256 tokens only contractions of 512 and more, where the other kernels' one block a tile takes longest: 512 x 2048 -> 2048, k = 64: 19.0 ->
// 13.2, fp32 18.5 -> 15.1; 512 x 8192 -> 512, k = 16: 30.9 -> 11.5 and 21.1 -> 13.0; 512 x 4096 -> 512, k = 128: 28.7 -> 18.9, fp32 24.0 -> 24.6; 512 x
// 520 -> 2000, k = 64: 12.0 -> 11.2; 640 tokens x 1001 -> 999, k = 60: 16.2 -> 17.4.  In bf16 y is not bit for bit that of the forms that keep z
// for a backward pass (rounded to bf16, and multiplied as it is kept): z stays in fp32 here, and y is nearer to 64 bits.
// The factored form is taken as far as everywhere: up to 16 times the products of one with a stored weight.
static bool few_pays(const rdb_linear_desc *d)
{
    const int64_t T = d->tokens, k = d->k, units = cdiv(d->out_f, FEW_ROWS) * cdiv(T, 16);
    const bool b16 = d->act_dtype == RDB_BF16;
    if (T > 2 * FEW_TOKENS) return false;
    if (b16 && d->in_f < 512 && (T > 96 || k > 64) && !few_plan(d).one) return false;
    if (T <= 16) return true;
    if (T > (d->in_f >= 512 && (k <= 64 || (b16 && k <= 128)) ? 2 * FEW_TOKENS : FEW_TOKENS)) return false;
    if (b16 && d->in_f <= 512 && units > (k <= 128 ? 512 : 256)) return false;
    if (k <= 128) return units <= (b16 || k <= 64 ? 1536 : 1024);
    if (k > 256) return T <= 32 || (b16 && T <= 96 && units <= 300);
    return b16 ? T <= 96 || units <= 512 : (T <= 96 || (T <= 192 && units <= 512)) && d->in_f <= 4 * d->out_f;
}
static bool few_ok(const rdb_linear_desc *d)
{
    const bool f32 = d->act_dtype == RDB_F32 && d->coef_dtype == RDB_F32, b16 = d->act_dtype == RDB_BF16 && d->coef_dtype == RDB_BF16;
    if (!f32_split_mode() && !(b16 && d->in_f % 8 == 0 && d->out_f % 8 == 0 && d->k % 8 == 0)) return false;   // fp32 products are asked for (rdb_set_f32_split)
    return (f32 || b16) && d->algo == RDB_ALGO_AUTO && d->coef_rows != 0 && d->k > 0 && d->k <= FEW_K && d->tokens > 0 && d->in_f > 0 &&
           d->out_f > 0 && d->in_f < (1 << 20) && d->out_f < (1 << 24) && few_pays(d) && d->k * (d->in_f + d->out_f) < 16 * d->in_f * d->out_f;
}
int64_t linear_few_workspace(const rdb_linear_desc *d)
{
    if (!few_ok(d)) return 0;
    const FewPlan f = few_plan(d);
    return f.part_bytes + (int64_t)f.c_blocks * 8 + 8;   // ... the tags, and the consumers' counter
}

template <typename E, int KS, int TC, int TE> static int few_launch(FewParams p, const FewPlan &f, int c_blocks, bool one, hipStream_t s)
{
    const size_t smem_y = (size_t)3 * TE * 16 * (KS * 32 + 8) * 2;
    const auto fused = [&](auto waves_, size_t smem, unsigned blocks, const char *name) {
        constexpr int WAVES = decltype(waves_)::value;
        const auto kernel = few_fwd_kernel<E, KS, TC, TE, WAVES>;
        if (int rc = reserve_lds(reinterpret_cast<const void *>(kernel), std::max((size_t)WAVES * TC * 1024, smem_y), name)) return rc;
        kernel<<<blocks, WAVES * 64, smem, s>>>(p);
        return check_launch(name);
    };
    typedef std::integral_constant<int, 4> W4;
    typedef std::integral_constant<int, 8> W8;
    p.c_blocks = c_blocks;
    if (one) {
        const unsigned blocks = (unsigned)(c_blocks + f.e_blocks);
        const size_t smem = std::max((size_t)f.waves * TC * 1024, smem_y);
        return f.waves == 8 ? fused(W8{}, smem, blocks, "few_fwd_kernel") : fused(W4{}, smem, blocks, "few_fwd_kernel");
    }
    if (f.waves == 16) few_contract_kernel<E, TC, 16><<<(unsigned)c_blocks, 1024, 0, s>>>(p);
    else if (f.waves == 8) few_contract_kernel<E, TC, 8><<<(unsigned)c_blocks, 512, 0, s>>>(p);
    else few_contract_kernel<E, TC, 4><<<(unsigned)c_blocks, 256, 0, s>>>(p);
    if (int rc = check_launch("few_contract_kernel")) return rc;
    if (f.sum) {
        const int64_t n4 = (int64_t)p.tiles * p.ranges * p.tile * 4;
        few_sum_kernel<<<(unsigned)cdiv(n4, 256), 256, 0, s>>>(p.part, n4, p.chunks);
        if (int rc = check_launch("few_sum_kernel")) return rc;
        p.chunks = 1;
    }
    p.c_blocks = 0;
    return fused(W4{}, smem_y, (unsigned)f.e_blocks, "few_fwd_kernel (y)");
}
template <typename E> static int few_dispatch(const FewParams &p, const FewPlan &f, int c_blocks, bool one, hipStream_t s)
{
    auto of = [&](auto ks_) {
        constexpr int KS = decltype(ks_)::value;
        if (f.tc == 1) return few_launch<E, KS, 1, 1>(p, f, c_blocks, one, s);
        if (f.te == 1) return few_launch<E, KS, 2, 1>(p, f, c_blocks, one, s);
        return few_launch<E, KS, 2, 2>(p, f, c_blocks, one, s);
    };
    if (p.k <= 128) return of(std::integral_constant<int, 4>{});
    if (p.k <= 256) return of(std::integral_constant<int, 8>{});
    return of(std::integral_constant<int, 16>{});
}

static FewParams few_params(const rdb_linear_desc *d, const FewPlan &f, void *y, int64_t ldy, const void *x, int64_t ldx, const void *coef, const void *bias,
                            void *workspace)
{
    const int es = d->act_dtype == RDB_BF16 ? 2 : 4;
    FewParams p = {};
    p.y = y;
    p.x = x;
    p.coef = coef;
    p.bias = bias;
    p.ldx = ldx;
    p.ldy = ldy;
    p.part = static_cast<float *>(workspace);
    p.T = (int)d->tokens;
    p.in_f = (int)d->in_f;
    p.out_f = (int)d->out_f;
    p.k = (int)d->k;
    p.chunks = f.chunks;
    p.ranges = f.ranges;
    p.tile = f.tile;
    p.tiles = f.tiles;
    p.c_groups = (int)cdiv(f.tiles, f.tc);
    p.e_blocks = (int)cdiv(d->out_f, FEW_ROWS);
    p.wave_values = f.wave_values;
    p.x_vec = d->in_f % 8 == 0 && ldx * es % 16 == 0 && ((uintptr_t)x & 15) == 0;
    p.c_vec = d->k % 8 == 0 && ((uintptr_t)coef & 15) == 0;
    p.y_vec = d->out_f % 4 == 0 && ldy % 4 == 0 && ((uintptr_t)y & (4 * es - 1)) == 0;
    p.seed = d->seed;
    return p;
}
static int few_tags(FewParams &p, const FewPlan &f, int polls)
{
    p.slots = reinterpret_cast<unsigned long long *>(reinterpret_cast<char *>(p.part) + f.part_bytes);
    p.tag = next_sync_tag();
    p.wait = {nullptr, nullptr, polls};
    p.tags = f.c_blocks;
    p.count = reinterpret_cast<unsigned int *>(p.slots + f.c_blocks);
    p.consumers = f.e_blocks;
    return sync_giveups_ptr(&p.wait.giveups);
}

// Returns RDB_E_UNSUPPORTED, without setting an error, when the request does not fit.
int linear_fwd_few(void *y, int64_t ldy, const void *x, int64_t ldx, const void *coef, const void *scale_bias, const void *bias, const rdb_linear_desc *d,
                   void *workspace, int64_t workspace_bytes, hipStream_t s)
{
    if (scale_bias || !few_ok(d) || !workspace || ((uintptr_t)workspace & 15) || workspace_bytes < linear_few_workspace(d)) return RDB_E_UNSUPPORTED;
    const FewPlan f = few_plan(d);
    FewParams p = few_params(d, f, y, ldy, x, ldx, coef, bias, workspace);
    const bool one = f.one && one_launch_mode();
    if (one) {
        if (int rc = few_tags(p, f, SYNC_SPIN_LIMIT)) return rc;
    }
    return d->act_dtype == RDB_BF16 ? few_dispatch<bf16_t>(p, f, f.c_blocks, one, s) : few_dispatch<float>(p, f, f.c_blocks, one, s);
}

// Test hook: only the expanding blocks of the one-launch form, waiting (at most `polls` polls each) for tags that nobody publishes.
int selftest_giveup_few(void *y, int64_t ldy, const void *coef, const rdb_linear_desc *d, void *workspace, int64_t workspace_bytes, int polls, hipStream_t s)
{
    if (!few_ok(d) || ((uintptr_t)workspace & 15) || workspace_bytes < linear_few_workspace(d)) return RDB_E_UNSUPPORTED;
    const FewPlan f = few_plan(d);
    if (!f.one) return RDB_E_UNSUPPORTED;
    FewParams p = few_params(d, f, y, ldy, nullptr, 0, coef, nullptr, workspace);
    if (int rc = few_tags(p, f, polls)) return rc;
    return d->act_dtype == RDB_BF16 ? few_dispatch<bf16_t>(p, f, 0, true, s) : few_dispatch<float>(p, f, 0, true, s);
}

}  // namespace rdb
