// Causal self-attention of a transformer block in bf16, head dimension 64, from the output of its qkv linear to the input of its
// output projection, forwards and back: RMS normalisation and rotary embedding of q and k, softmax(q.k^T / 8).v, and the gradient
// of all of it (modded-nanogpt/gpt_models.py:29-49, 201-232, with plain causal attention).
//
//   attn_prep_kernel     qkv [tokens][3][heads][64] -> q, k normalised and rotated, [batch * heads][T][64]; the rotary table
//   attn_fwd_kernel      y [tokens][heads * 64] and log2 of every row's sum
//   attn_bwd_dq_kernel   the q part of dqkv, through rotation and normalisation; <dy, y> per row for the next kernel
//   attn_bwd_dkv_kernel  the k and v parts of dqkv
//
// Scores: |q| and |k| are at most 8 (1 + 2^-7) after the normalisation, so q.k / 8 stays below 8.2 in magnitude and exp needs no
// running maximum: no rescaling of the accumulators, no reduction inside the loop, the row sum is added up once at the end.
//
// Every product is taken transposed, D^T[kv][q] = K . Q^T with the wave's own 32 rows as the columns, so that a lane holds 16
// values of one q row (or of one kv row in the dk / dv kernel): the softmax needs no data from other lanes, and the rounded
// probabilities are, as they lie in the registers, the right operand of the next product.  (Its contraction runs over kv in
// another order, 4 g + {0..3, 8..11} of every 16 for lane half g, which the left operand's transposing LDS reads follow.)
//
// A block owns 128 rows, 32 a wave, or (HALVES) 64, two waves to 32 rows that take the two halves of every tile of the other side and
// add up at the end.  The longest block is then half as long and there are twice as many, but each stages its tiles for half the
// rows: for grids that do not keep the compute units busy (at_halves).
//
// Measured at 8 sequences x 12 heads x 1024 tokens, us: forward 34.7 (13.5 of them prep), backward 79 (the stock operators they
// replace: attention 81 forward, 267 backward, normalisation and rotation some 450).  13 GFLOP forward and 45 backward.  No pipe is
// full (SQ counters, shares of a compute unit's time): matrix cores 28 to 30 %, vector ALU 40 to 51 % (29 % of the
// forward pass in exponentials, 16 a lane for 16 matrix instructions), LDS 36 to 43 % without bank conflicts; two waves a SIMD and a
// barrier per 64 rows put them one after the other.  The preparing kernel is the vector ALU's (94 %;
// without its 64-bit divisions by T and with one call for sine and cosine it is 1 us shorter, which no step showed).
#include "rdb_gemm.hpp"

namespace rdb {

constexpr int HD = 64;              // head dimension
constexpr int AT_TILE = 64;         // rows of the other side a step takes
constexpr float AT_SCALE = 0.125f;  // 1 / sqrt(HD)
constexpr float AT_EXP2 = 0.125f * 1.44269504088896340736f;

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float at_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float at_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ float at_round(float v) { return bf16_to_f32(f32_to_bf16(v)); }

// ----------------------------------------------------------------------------------------------- normalisation and rotation
struct PrepParams {
    bf16_t *q, *k;          // [B * H][T][64]
    float *table;           // [T][32] pairs (cos, sin)
    const bf16_t *qkv;      // [B * T][3][H][64]
    const void *inv_freq;   // [32]
    int inv_bf16, B, T, H;
    float eps;
};

// A block takes four tokens: 128 threads compute their rotary pairs, then eight lanes each take one head's row (16 bytes a lane).
// A frequency in bf16 makes position, angle, cosine and sine bf16 too, as the stock operators' type promotion does.
__global__ __launch_bounds__(256) void attn_prep_kernel(PrepParams p)
{
    __shared__ float cs[4][32], sn[4][32];
    const int t = threadIdx.x;
    const int64_t tok0 = (int64_t)blockIdx.x * 4, ntok = (int64_t)p.B * p.T;
    if (t < 128) {
        const int64_t tok = tok0 + (t >> 5);
        if (tok < ntok) {
            const int pos = (int)(tok % p.T), i = t & 31;
            float a, c, s;
            if (p.inv_bf16) {
                a = at_round(at_round((float)pos) * bf16_to_f32(static_cast<const bf16_t *>(p.inv_freq)[i]));
                c = at_round(cosf(a));
                s = at_round(sinf(a));
            } else {
                a = (float)pos * static_cast<const float *>(p.inv_freq)[i];
                c = cosf(a);
                s = sinf(a);
            }
            cs[t >> 5][i] = c;
            sn[t >> 5][i] = s;
            if (tok < p.T) {
                p.table[((int64_t)pos * 32 + i) * 2] = c;
                p.table[((int64_t)pos * 32 + i) * 2 + 1] = s;
            }
        }
    }
    __syncthreads();
    const int part = t & 7, rows = 8 * p.H;   // 4 tokens x (q, k) x heads
    for (int v = t >> 3; v < rows; v += 32) {
        const int tl = v / (2 * p.H), w = v - tl * 2 * p.H, kind = w >= p.H ? 1 : 0, h = w - kind * p.H;
        const int64_t tok = tok0 + tl;
        const bool live = tok < ntok;
        const int64_t tk = live ? tok : ntok - 1;
        const u32x4 x = *reinterpret_cast<const u32x4 *>(p.qkv + ((tk * 3 + kind) * p.H + h) * HD + part * 8);
        float f[8], s = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            f[2 * e] = at_lo(x[e]);
            f[2 * e + 1] = at_hi(x[e]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) s = fmaf(f[e], f[e], s);
        s += __shfl_xor(s, 1, 64);
        s += __shfl_xor(s, 2, 64);
        s += __shfl_xor(s, 4, 64);
        const float r = rsqrtf(s * (1.0f / HD) + p.eps);
        u32x4 o;
        float g[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            f[e] = at_round(f[e] * r);
            g[e] = __shfl_xor(f[e], 4, 64);   // the other half of the rotated pair
        }
        const float *c = cs[tl] + (part & 3) * 8, *sv = sn[tl] + (part & 3) * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = part < 4 ? f[e] * c[e] + g[e] * sv[e] : f[e] * c[e] - g[e] * sv[e];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = f32x2_to_bf16x2(f[2 * e], f[2 * e + 1]);
        if (live) {
            const int64_t b = tok / p.T, pos = tok - b * p.T;
            *reinterpret_cast<u32x4 *>((kind ? p.k : p.q) + ((b * p.H + h) * p.T + pos) * HD + part * 8) = o;
        }
    }
}

// ----------------------------------------------------------------------------------------------- tiles in LDS
// 64 rows of 64 values, 128 bytes each without padding, 16-byte chunk c of a row at position c ^ at_swz(row).  The fragment reads
// along the rows take one chunk from each of 16 consecutive rows (eight different positions in either half of the banks), the
// transposing reads four chunks from each of 4 consecutive rows (two rows of a half apart in bit 2): both free of conflicts, so
// one copy of a tile serves as an operand in both directions.
__device__ __forceinline__ int at_swz(int row) { return (((row >> 1) & 1) << 2) | ((row >> 2) & 3); }

struct TileSource {   // rows of one (batch, head) in memory; rows from `rows` on read as zeros
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t ld;   // bytes
    __device__ __forceinline__ TileSource(const bf16_t *base, int64_t ld_elems, int rows)
    {
        ld = (uint32_t)(ld_elems * 2);
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(base), 0, (int)(((int64_t)(rows - 1) * ld_elems + HD) * 2), 0x00020000);
    }
    __device__ __forceinline__ f32x4 load(int row, int chunk) const
    {
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)((uint32_t)row * ld + (uint32_t)chunk * 16u), 0, 0));
    }
    __device__ __forceinline__ void tile(f32x4 (&r)[2], int row0) const
    {
#pragma unroll
        for (int p = 0; p < 2; ++p) r[p] = load(row0 + p * 32 + (threadIdx.x >> 3), threadIdx.x & 7);
    }
    // the wave's 32 rows as the right operand of a product that contracts over the head dimension
    __device__ __forceinline__ void frags(bf16x8 (&f)[4], int row0) const
    {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) f[ks] = __builtin_bit_cast(bf16x8, load(row0 + (lane & 31), ks * 2 + (lane >> 5)));
    }
};
__device__ __forceinline__ void at_store_tile(bf16_t *lds, const f32x4 (&r)[2])
{
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int row = p * 32 + (threadIdx.x >> 3), c = threadIdx.x & 7;
        *reinterpret_cast<f32x4 *>(lds + row * HD + ((c ^ at_swz(row)) * 8)) = r[p];
    }
}
// rows rb .. rb + 31, contraction values ks * 16 + g * 8 .. + 7 (along the row)
__device__ __forceinline__ bf16x8 at_row_frag(const bf16_t *lds, int rb, int ks, int lane)
{
    const int r = lane & 31, g = lane >> 5;
    return *reinterpret_cast<const bf16x8 *>(lds + (rb + r) * HD + (((ks * 2 + g) ^ at_swz(r)) * 8));
}
// columns cb .. cb + 31 as rows, contraction over the tile's rows st * 16 + 4 g + {0 .. 3, 8 .. 11}
__device__ __forceinline__ bf16x8 at_col_frag(const bf16_t *lds, int cb, int st, int lane)
{
    const int s = lane & 15, row = st * 16 + (lane >> 5) * 4 + (s >> 2), col = cb + ((lane >> 4) & 1) * 16 + (s & 3) * 4;
    Frag8 f;
    f.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(lds + row * HD + (((col >> 3) ^ at_swz(row)) * 8) + (col & 7)));
    f.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (s16x4 __attribute__((address_space(3))) *)(lds + (row + 8) * HD + (((col >> 3) ^ at_swz(row + 8)) * 8) + (col & 7)));
    return f.v;
}
// 16 values of a 32-row block in the accumulators' order -> the right operand's fragments of its two k-steps
__device__ __forceinline__ void at_pack(bf16x8 (&f)[2], const float (&v)[16])
{
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        Frag8 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o.u[e] = f32x2_to_bf16x2(v[s * 8 + 2 * e], v[s * 8 + 2 * e + 1]);
        f[s] = o.v;
    }
}
__device__ __forceinline__ f32x16 at_mma(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
// The loads behind these registers are waited for here.  Operands that a loop only reads: their loads may be scheduled behind those of the
// first tiles, and loads return in order, so a first use inside the loop waits in every turn for the next tile's loads, which that turn has
// just requested (forward with preparation, us: 1 x 12 x 1024 21.2 -> 17.5, 4 x 12 x 1024 26.6 -> 24.3, 8 x 12 x 1024 36.7 -> 34.7, 3 x 8 x 200 9.8 ->
// 9.0; with the tiles requested two steps ahead as well 18.4, 24.1, 36.1, 9.4).
template <int N> __device__ __forceinline__ void at_arrived(bf16x8 (&f)[N])
{
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(f[i]));
}
// one accumulator (32 x 32) of a wave in LDS, for the other wave of its rows
__device__ __forceinline__ void at_put(float *lds, const f32x16 &v, int lane)
{
#pragma unroll
    for (int j = 0; j < 16; ++j) lds[j * 64 + lane] = v[j];
}
__device__ __forceinline__ void at_add(f32x16 &v, const float *lds, int lane)
{
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] += lds[j * 64 + lane];
}
// row (0 .. 31) of accumulator element j in lane half g
__device__ __forceinline__ int at_row(int j, int g) { return 8 * (j >> 2) + 4 * g + (j & 3); }

struct AttnParams {
    const bf16_t *q, *k;     // [B * H][T][64], normalised and rotated
    const bf16_t *qkv;       // [B * T][3][H][64]
    bf16_t *y;               // [B * T][H * 64]
    float *lsum;             // [B * H][T]: log2 of the row sums
    const bf16_t *dy;        // [B * T][H * 64]
    float *delta;            // [B * H][T]
    const float *table;
    bf16_t *dqkv;
    int T, H, BH, nb;        // nb: blocks per head
    float eps;
};

// Blocks are numbered with the longest first (causal: a block's work grows with its rows' index, or falls with it for dk / dv),
// all heads of a block index before the next: with a multiple of 8 heads, a head's blocks all run on the die that holds its k and v in its L2.
// Every second 256 of them, one for each compute unit, come in the opposite order, eights of them so that the dies stay: a
// compute unit's first two blocks are a long one and a short one.  us in order -> so: 8 x 12 heads x 1024, forward with preparation
// 38.3 -> 36.7, backward 83.4 -> 79.0; 7 x 12 x 900: 31.3 -> 31.3, 68.5 -> 64.9.
__device__ __forceinline__ void at_block(const AttnParams &p, int &bh, int &b, int &h, int &rank)
{
    const int first = (int)blockIdx.x & ~255, at = (int)blockIdx.x & 255, len = min(256, (int)gridDim.x - first) & ~7;
    const int x = (first & 256) && at < len ? first + len - 8 - (at & ~7) + (at & 7) : (int)blockIdx.x;
    rank = x / p.BH;
    bh = x - rank * p.BH;
    b = bh / p.H;
    h = bh - b * p.H;
}

// ----------------------------------------------------------------------------------------------- forward
template <bool HALVES> __global__ __launch_bounds__(256, 3) void attn_fwd_kernel(AttnParams p)
{
    __shared__ __align__(16) bf16_t tiles[4][AT_TILE * HD];   // K, K, V, V
    __shared__ float ls_[4][64];
    bf16_t *const ks_ = tiles[0], *const vs_ = tiles[2];
    constexpr int TILE = AT_TILE * HD;
    int bh, b, h, rank;
    at_block(p, bh, b, h, rank);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = HALVES ? wave >> 1 : 0, r = lane & 31, g = lane >> 5;
    constexpr int ROWS = HALVES ? 64 : 128;
    const int m0 = (p.nb - 1 - rank) * ROWS, q0 = m0 + (HALVES ? wave & 1 : wave) * 32, T = p.T;
    const int64_t ld3 = (int64_t)3 * p.H * HD;
    const TileSource qs(p.q + (int64_t)bh * T * HD, HD, T), kg(p.k + (int64_t)bh * T * HD, HD, T);
    const TileSource vg(p.qkv + (int64_t)b * T * ld3 + (2 * p.H + h) * HD, ld3, T);
    bf16x8 qf[4];
    qs.frags(qf, q0);
    const int last = (m0 + ROWS < T ? m0 + ROWS : T), nt = (last + AT_TILE - 1) / AT_TILE;
    f32x4 kr[2], vr[2];
    kg.tile(kr, 0);
    vg.tile(vr, 0);
    at_store_tile(ks_, kr);
    at_store_tile(vs_, vr);
    at_arrived(qf);
    __syncthreads();
    f32x16 o[2] = {zero16(), zero16()};
    float l = 0.0f;
    for (int t = 0; t < nt; ++t) {
        const bf16_t *K = ks_ + (t & 1) * TILE, *V = vs_ + (t & 1) * TILE;
        const bool more = t + 1 < nt;
        const int n0 = t * AT_TILE;
        if (more) {
            kg.tile(kr, n0 + AT_TILE);
            vg.tile(vr, n0 + AT_TILE);
        }
#pragma unroll
        for (int i = 0; i < (HALVES ? 1 : 2); ++i) {
            const int kb = HALVES ? half : i;
            if (n0 + kb * 32 > q0 + 31) continue;   // past the diagonal
            f32x16 s = zero16();
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) s = at_mma(at_row_frag(K, kb * 32, ks, lane), qf[ks], s);
            float e[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) e[j] = __builtin_amdgcn_exp2f(s[j] * AT_EXP2);
            if (n0 + kb * 32 + 31 > q0) {   // reaches past the diagonal
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    if (n0 + kb * 32 + at_row(j, g) > q0 + r) e[j] = 0.0f;
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) l += e[j];
            bf16x8 f[2];
            at_pack(f, e);
#pragma unroll
            for (int st = 0; st < 2; ++st)
#pragma unroll
                for (int db = 0; db < 2; ++db) o[db] = at_mma(at_col_frag(V, db * 32, kb * 2 + st, lane), f[st], o[db]);
        }
        if (more) {
            at_store_tile(ks_ + ((t + 1) & 1) * TILE, kr);
            at_store_tile(vs_ + ((t + 1) & 1) * TILE, vr);
        }
        __syncthreads();
    }
    l += __shfl_xor(l, 32, 64);
    if constexpr (HALVES) {   // the two waves of a row: each finishes half of the dimensions
        float *const acc = reinterpret_cast<float *>(tiles);
        ls_[wave][lane] = l;
        at_put(acc + wave * 1024, half ? o[0] : o[1], lane);
        __syncthreads();
        l += ls_[wave ^ 2][lane];
        if (half) o[0] = o[1];
        at_add(o[0], acc + (wave ^ 2) * 1024, lane);
    }
    const int row = q0 + r;
    if (row >= T) return;
    const float inv = 1.0f / l;
    if (g == 0 && half == 0) p.lsum[(int64_t)bh * T + row] = log2f(l);
    bf16_t *out = p.y + ((int64_t)b * T + row) * p.H * HD + h * HD + half * 32;
#pragma unroll
    for (int db = 0; db < (HALVES ? 1 : 2); ++db)
#pragma unroll
        for (int jq = 0; jq < 4; ++jq) {
            const u32x2 w = {f32x2_to_bf16x2(o[db][jq * 4] * inv, o[db][jq * 4 + 1] * inv), f32x2_to_bf16x2(o[db][jq * 4 + 2] * inv, o[db][jq * 4 + 3] * inv)};
            *reinterpret_cast<u32x2 *>(out + db * 32 + 8 * jq + 4 * g) = w;
        }
}

// ----------------------------------------------------------------------------------------------- backward
// Gradient of a q or k row behind the rotation and the normalisation: d holds the gradient of the rotated row (a lane: dimensions
// at_row(j, g) and 32 + at_row(j, g), the two of a rotated pair), x the row of qkv it came from.
__device__ __forceinline__ void at_row_grad(bf16_t *out, const bf16_t *x, const float *table, const f32x16 (&d)[2], float eps, int g)
{
    float n[2][16], v[2][16], ss = 0.0f;
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) {
        const int i = 8 * jq + 4 * g;
        const u32x2 a = *reinterpret_cast<const u32x2 *>(x + i), c = *reinterpret_cast<const u32x2 *>(x + 32 + i);
        const f32x4 t0 = *reinterpret_cast<const f32x4 *>(table + i * 2), t1 = *reinterpret_cast<const f32x4 *>(table + i * 2 + 4);
        const float co[4] = {t0.x, t0.z, t1.x, t1.z}, si[4] = {t0.y, t0.w, t1.y, t1.w};
        v[0][jq * 4] = at_lo(a.x);
        v[0][jq * 4 + 1] = at_hi(a.x);
        v[0][jq * 4 + 2] = at_lo(a.y);
        v[0][jq * 4 + 3] = at_hi(a.y);
        v[1][jq * 4] = at_lo(c.x);
        v[1][jq * 4 + 1] = at_hi(c.x);
        v[1][jq * 4 + 2] = at_lo(c.y);
        v[1][jq * 4 + 3] = at_hi(c.y);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int j = jq * 4 + e;
            const float g1 = at_round(d[0][j] * AT_SCALE), g2 = at_round(d[1][j] * AT_SCALE);
            n[0][j] = at_round(g1 * co[e] - g2 * si[e]);
            n[1][j] = at_round(g1 * si[e] + g2 * co[e]);
            ss = fmaf(v[0][j], v[0][j], fmaf(v[1][j], v[1][j], ss));
        }
    }
    ss += __shfl_xor(ss, 32, 64);
    const float rs = rsqrtf(ss * (1.0f / HD) + eps);
    float m = 0.0f;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int j = 0; j < 16; ++j) m = fmaf(n[db][j], v[db][j] * rs, m);
    m += __shfl_xor(m, 32, 64);
    m *= 1.0f / HD;
    if (!out) return;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int jq = 0; jq < 4; ++jq) {
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (n[db][jq * 4 + e] - v[db][jq * 4 + e] * rs * m) * rs;
            *reinterpret_cast<u32x2 *>(out + db * 32 + 8 * jq + 4 * g) = u32x2{f32x2_to_bf16x2(o[0], o[1]), f32x2_to_bf16x2(o[2], o[3])};
        }
}

template <bool HALVES> __global__ __launch_bounds__(256, 2) void attn_bwd_dq_kernel(AttnParams p)
{
    __shared__ __align__(16) bf16_t tiles[4][AT_TILE * HD];   // K, K, V, V
    bf16_t *const ks_ = tiles[0], *const vs_ = tiles[2];
    constexpr int TILE = AT_TILE * HD;
    int bh, b, h, rank;
    at_block(p, bh, b, h, rank);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = HALVES ? wave >> 1 : 0, r = lane & 31, g = lane >> 5;
    constexpr int ROWS = HALVES ? 64 : 128;
    const int m0 = (p.nb - 1 - rank) * ROWS, q0 = m0 + (HALVES ? wave & 1 : wave) * 32, T = p.T;
    const int64_t ld3 = (int64_t)3 * p.H * HD, ld1 = (int64_t)p.H * HD;
    const TileSource qs(p.q + (int64_t)bh * T * HD, HD, T), kg(p.k + (int64_t)bh * T * HD, HD, T);
    const TileSource vg(p.qkv + (int64_t)b * T * ld3 + (2 * p.H + h) * HD, ld3, T);
    const TileSource ds(p.dy + (int64_t)b * T * ld1 + h * HD, ld1, T), ys(p.y + (int64_t)b * T * ld1 + h * HD, ld1, T);
    bf16x8 qf[4], df[4];
    qs.frags(qf, q0);
    ds.frags(df, q0);
    float delta = 0.0f;
    {   // <dy, y> of the row
        bf16x8 yf[4];
        ys.frags(yf, q0);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            Frag8 a, c;
            a.v = df[ks];
            c.v = yf[ks];
#pragma unroll
            for (int e = 0; e < 4; ++e) delta = fmaf(at_lo(a.u[e]), at_lo(c.u[e]), fmaf(at_hi(a.u[e]), at_hi(c.u[e]), delta));
        }
        delta += __shfl_xor(delta, 32, 64);
    }
    const int row = q0 + r;
    const float l2 = row < T ? p.lsum[(int64_t)bh * T + row] : 0.0f;
    if (g == 0 && half == 0 && row < T) p.delta[(int64_t)bh * T + row] = delta;
    const int last = (m0 + ROWS < T ? m0 + ROWS : T), nt = (last + AT_TILE - 1) / AT_TILE;
    f32x4 kr[2], vr[2];
    kg.tile(kr, 0);
    vg.tile(vr, 0);
    at_store_tile(ks_, kr);
    at_store_tile(vs_, vr);
    __syncthreads();
    f32x16 dq[2] = {zero16(), zero16()};
    for (int t = 0; t < nt; ++t) {
        const bf16_t *K = ks_ + (t & 1) * TILE, *V = vs_ + (t & 1) * TILE;
        const bool more = t + 1 < nt;
        const int n0 = t * AT_TILE;
        if (more) {
            kg.tile(kr, n0 + AT_TILE);
            vg.tile(vr, n0 + AT_TILE);
        }
#pragma unroll
        for (int i = 0; i < (HALVES ? 1 : 2); ++i) {
            const int kb = HALVES ? half : i;
            if (n0 + kb * 32 > q0 + 31) continue;   // past the diagonal
            f32x16 s = zero16(), d = zero16();
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                s = at_mma(at_row_frag(K, kb * 32, ks, lane), qf[ks], s);
                d = at_mma(at_row_frag(V, kb * 32, ks, lane), df[ks], d);
            }
            float e[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) e[j] = __builtin_amdgcn_exp2f(fmaf(s[j], AT_EXP2, -l2));
            if (n0 + kb * 32 + 31 > q0) {
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    if (n0 + kb * 32 + at_row(j, g) > q0 + r) e[j] = 0.0f;
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) e[j] *= d[j] - delta;
            bf16x8 f[2];
            at_pack(f, e);
#pragma unroll
            for (int st = 0; st < 2; ++st)
#pragma unroll
                for (int db = 0; db < 2; ++db) dq[db] = at_mma(at_col_frag(K, db * 32, kb * 2 + st, lane), f[st], dq[db]);
        }
        if (more) {
            at_store_tile(ks_ + ((t + 1) & 1) * TILE, kr);
            at_store_tile(vs_ + ((t + 1) & 1) * TILE, vr);
        }
        __syncthreads();
    }
    if constexpr (HALVES) {   // the two waves of a row: the first one adds up and goes on
        float *const acc = reinterpret_cast<float *>(tiles) + (wave & 1) * 2048;
        if (half) {
            at_put(acc, dq[0], lane);
            at_put(acc + 1024, dq[1], lane);
        }
        __syncthreads();
        if (half) return;
        at_add(dq[0], acc, lane);
        at_add(dq[1], acc + 1024, lane);
    }
    const int64_t at = ((int64_t)b * T + (row < T ? row : T - 1)) * ld3 + h * HD;
    at_row_grad(row < T ? p.dqkv + at : nullptr, p.qkv + at, p.table + (int64_t)(row < T ? row : T - 1) * 64, dq, p.eps, g);
}

template <bool HALVES> __global__ __launch_bounds__(256, 2) void attn_bwd_dkv_kernel(AttnParams p)
{
    __shared__ __align__(16) bf16_t tiles[4][AT_TILE * HD];   // Q, Q, dY, dY
    bf16_t *const qs_ = tiles[0], *const ds_ = tiles[2];
    constexpr int TILE = AT_TILE * HD;
    __shared__ __align__(16) float ls_[2][AT_TILE], dl_[2][AT_TILE];
    int bh, b, h, rank;
    at_block(p, bh, b, h, rank);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = HALVES ? wave >> 1 : 0, r = lane & 31, g = lane >> 5;
    constexpr int ROWS = HALVES ? 64 : 128;
    const int m0 = rank * ROWS, n0 = m0 + (HALVES ? wave & 1 : wave) * 32, T = p.T;   // n0: the wave's first kv row
    const int64_t ld3 = (int64_t)3 * p.H * HD, ld1 = (int64_t)p.H * HD;
    const TileSource qg(p.q + (int64_t)bh * T * HD, HD, T), kg(p.k + (int64_t)bh * T * HD, HD, T);
    const TileSource vg(p.qkv + (int64_t)b * T * ld3 + (2 * p.H + h) * HD, ld3, T), dg(p.dy + (int64_t)b * T * ld1 + h * HD, ld1, T);
    bf16x8 kf[4], vf[4];
    kg.frags(kf, n0);
    vg.frags(vf, n0);
    const int t0 = m0 / AT_TILE, nt = (T + AT_TILE - 1) / AT_TILE;
    f32x4 qr[2], dr[2];
    float lr = 0.0f;
    // threads 0 .. 63: the tile's log sums (rows past the end: so large that their probabilities are zero), 64 .. 127: its deltas
    auto load_row = [&](int t) {
        const int row = t * AT_TILE + (threadIdx.x & 63);
        if (threadIdx.x < 128) lr = row < T ? (threadIdx.x < 64 ? p.lsum : p.delta)[(int64_t)bh * T + row] : (threadIdx.x < 64 ? 1e30f : 0.0f);
    };
    auto store_row = [&](int buf) {
        if (threadIdx.x < 128) (threadIdx.x < 64 ? ls_ : dl_)[buf][threadIdx.x & 63] = lr;
    };
    qg.tile(qr, t0 * AT_TILE);
    dg.tile(dr, t0 * AT_TILE);
    load_row(t0);
    at_store_tile(qs_ + (t0 & 1) * TILE, qr);
    at_store_tile(ds_ + (t0 & 1) * TILE, dr);
    store_row(t0 & 1);
    __syncthreads();
    f32x16 dk[2] = {zero16(), zero16()}, dv[2] = {zero16(), zero16()};
    for (int t = t0; t < nt; ++t) {
        const bf16_t *Q = qs_ + (t & 1) * TILE, *D = ds_ + (t & 1) * TILE;
        const float *L = ls_[t & 1], *E = dl_[t & 1];
        const bool more = t + 1 < nt;
        const int q0 = t * AT_TILE;
        if (more) {
            qg.tile(qr, q0 + AT_TILE);
            dg.tile(dr, q0 + AT_TILE);
            load_row(t + 1);
        }
#pragma unroll
        for (int i = 0; i < (HALVES ? 1 : 2); ++i) {
            const int qb = HALVES ? half : i;
            if (q0 + qb * 32 + 31 < n0) continue;   // past the diagonal
            f32x16 s = zero16(), d = zero16();
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                s = at_mma(at_row_frag(Q, qb * 32, ks, lane), kf[ks], s);
                d = at_mma(at_row_frag(D, qb * 32, ks, lane), vf[ks], d);
            }
            float e[16], u[16];
#pragma unroll
            for (int jq = 0; jq < 4; ++jq) {
                const f32x4 l4 = *reinterpret_cast<const f32x4 *>(L + qb * 32 + 8 * jq + 4 * g);
                const f32x4 e4 = *reinterpret_cast<const f32x4 *>(E + qb * 32 + 8 * jq + 4 * g);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int j = jq * 4 + c;
                    e[j] = __builtin_amdgcn_exp2f(fmaf(s[j], AT_EXP2, -l4[c]));
                    u[j] = d[j] - e4[c];
                }
            }
            if (q0 + qb * 32 < n0 + 31) {   // reaches past the diagonal
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    if (q0 + qb * 32 + at_row(j, g) < n0 + r) e[j] = 0.0f;
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) u[j] *= e[j];
            bf16x8 f[2], w[2];
            at_pack(f, e);
            at_pack(w, u);
#pragma unroll
            for (int st = 0; st < 2; ++st)
#pragma unroll
                for (int db = 0; db < 2; ++db) {
                    dv[db] = at_mma(at_col_frag(D, db * 32, qb * 2 + st, lane), f[st], dv[db]);
                    dk[db] = at_mma(at_col_frag(Q, db * 32, qb * 2 + st, lane), w[st], dk[db]);
                }
        }
        if (more) {
            at_store_tile(qs_ + ((t + 1) & 1) * TILE, qr);
            at_store_tile(ds_ + ((t + 1) & 1) * TILE, dr);
            store_row((t + 1) & 1);
        }
        __syncthreads();
    }
    if constexpr (HALVES) {   // the two waves of a row: one finishes dk, the other one dv
        float *const acc = reinterpret_cast<float *>(tiles);
#pragma unroll
        for (int db = 0; db < 2; ++db) at_put(acc + wave * 2048 + db * 1024, half ? dk[db] : dv[db], lane);
        __syncthreads();
        const float *const other = acc + (wave ^ 2) * 2048;
        if (half) {
            at_add(dv[0], other, lane);
            at_add(dv[1], other + 1024, lane);
        } else {
            at_add(dk[0], other, lane);
            at_add(dk[1], other + 1024, lane);
        }
    }
    const int row = n0 + r;
    const int64_t at = ((int64_t)b * T + (row < T ? row : T - 1)) * ld3 + (p.H + h) * HD;
    if (!HALVES || half == 0) at_row_grad(row < T ? p.dqkv + at : nullptr, p.qkv + at, p.table + (int64_t)(row < T ? row : T - 1) * 64, dk, p.eps, g);
    if (row >= T || (HALVES && half == 0)) return;
    bf16_t *out = p.dqkv + at + (int64_t)p.H * HD;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int jq = 0; jq < 4; ++jq)
            *reinterpret_cast<u32x2 *>(out + db * 32 + 8 * jq + 4 * g) =
                u32x2{f32x2_to_bf16x2(dv[db][jq * 4], dv[db][jq * 4 + 1]), f32x2_to_bf16x2(dv[db][jq * 4 + 2], dv[db][jq * 4 + 3])};
}

// ----------------------------------------------------------------------------------------------- host side
static int check_attn(const char *who, int64_t B, int64_t T, int64_t H)
{
    if (B <= 0 || T <= 0 || H <= 0) return set_error(RDB_E_SHAPE, "%s: sizes must be positive", who);
    if (T > (1 << 20) || H > 1024 || T * 3 * H * HD * 2 >= (1ll << 30) || B * H * cdiv(T, 128) >= (1ll << 31))
        return set_error(RDB_E_UNSUPPORTED, "%s: a sequence's qkv must stay below 2^30 bytes", who);
    return RDB_OK;
}
// us with blocks of 128 rows -> of 64, batch x heads x tokens: forward with preparation 1 x 12 x 1024 25.2 -> 21.3, 8 x 10 x 1024 (640
// blocks of 128) 34.0 -> 32.8, 8 x 12 x 1024 (768) 36.7 -> 39.0; backward 1 x 12 x 1024 49.6 -> 33.1, 4 x 12 x 1024 (384) 54.3 -> 47.3, 7 x 8 x 1024
// (448) 54.7 -> 57.3.
static bool at_halves(const AttnParams &p, bool backward) { return cdiv(p.T, 128) * p.BH <= (backward ? 384 : 640); }
static bool at16(const void *p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace rdb

using namespace rdb;

// floats of scratch: the rotary table, and log sum and delta per row and head
extern "C" int64_t rdb_causal_attention_scratch_floats(int64_t batch, int64_t T, int64_t heads) { return T * 64 + 2 * batch * heads * T; }

extern "C" int rdb_causal_attention_fwd(void *y, void *q, void *k, float *scratch, const void *qkv, const void *inv_freq, int inv_freq_dtype, int64_t batch,
                                        int64_t T, int64_t heads, float eps, void *stream)
{
    if (int rc = check_attn("rdb_causal_attention_fwd", batch, T, heads)) return rc;
    if (!y || !q || !k || !scratch || !qkv || !inv_freq) return set_error(RDB_E_NULL, "rdb_causal_attention_fwd: an argument is NULL");
    if (inv_freq_dtype != RDB_F32 && inv_freq_dtype != RDB_BF16) return set_error(RDB_E_DTYPE, "rdb_causal_attention_fwd: unknown dtype %d", inv_freq_dtype);
    if (!at16(y) || !at16(q) || !at16(k) || !at16(scratch) || !at16(qkv)) return set_error(RDB_E_ALIGN, "rdb_causal_attention_fwd: pointers must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    const PrepParams pp = {static_cast<bf16_t *>(q), static_cast<bf16_t *>(k), scratch, static_cast<const bf16_t *>(qkv), inv_freq,
                           inv_freq_dtype == RDB_BF16, (int)batch, (int)T, (int)heads, eps};
    attn_prep_kernel<<<(unsigned)cdiv(batch * T, 4), 256, 0, s>>>(pp);
    if (int rc = check_launch("attn_prep_kernel")) return rc;
    AttnParams p = {};
    p.q = pp.q;
    p.k = pp.k;
    p.qkv = pp.qkv;
    p.y = static_cast<bf16_t *>(y);
    p.lsum = scratch + T * 64;
    p.T = (int)T;
    p.H = (int)heads;
    p.BH = (int)(batch * heads);
    const bool halves = at_halves(p, false);
    p.nb = (int)cdiv(T, halves ? 64 : 128);
    if (halves) attn_fwd_kernel<true><<<(unsigned)(p.nb * p.BH), 256, 0, s>>>(p);
    else attn_fwd_kernel<false><<<(unsigned)(p.nb * p.BH), 256, 0, s>>>(p);
    return check_launch("attn_fwd_kernel");
}

extern "C" int rdb_causal_attention_bwd(void *dqkv, const void *dy, const void *y, const void *q, const void *k, float *scratch, const void *qkv,
                                        int64_t batch, int64_t T, int64_t heads, float eps, void *stream)
{
    if (int rc = check_attn("rdb_causal_attention_bwd", batch, T, heads)) return rc;
    if (!dqkv || !dy || !y || !q || !k || !scratch || !qkv) return set_error(RDB_E_NULL, "rdb_causal_attention_bwd: an argument is NULL");
    if (!at16(dqkv) || !at16(dy) || !at16(y) || !at16(q) || !at16(k) || !at16(scratch) || !at16(qkv))
        return set_error(RDB_E_ALIGN, "rdb_causal_attention_bwd: pointers must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    AttnParams p = {};
    p.q = static_cast<const bf16_t *>(q);
    p.k = static_cast<const bf16_t *>(k);
    p.qkv = static_cast<const bf16_t *>(qkv);
    p.y = static_cast<bf16_t *>(const_cast<void *>(y));
    p.lsum = scratch + T * 64;
    p.delta = p.lsum + batch * heads * T;
    p.dy = static_cast<const bf16_t *>(dy);
    p.table = scratch;
    p.dqkv = static_cast<bf16_t *>(dqkv);
    p.T = (int)T;
    p.H = (int)heads;
    p.BH = (int)(batch * heads);
    const bool halves = at_halves(p, true);
    p.nb = (int)cdiv(T, halves ? 64 : 128);
    p.eps = eps;
    const unsigned grid = (unsigned)(p.nb * p.BH);
    if (halves) attn_bwd_dq_kernel<true><<<grid, 256, 0, s>>>(p);
    else attn_bwd_dq_kernel<false><<<grid, 256, 0, s>>>(p);
    if (int rc = check_launch("attn_bwd_dq_kernel")) return rc;
    if (halves) attn_bwd_dkv_kernel<true><<<grid, 256, 0, s>>>(p);
    else attn_bwd_dkv_kernel<false><<<grid, 256, 0, s>>>(p);
    return check_launch("attn_bwd_dkv_kernel");
}
