// Input gradient of the fused linear layer, matrix-coef + bf16, "factored" algorithm:
//
//   dx = dy . W = dy . (C . N) = (dy . C) . N
//
// With k < in*out/(in+out) the right-hand grouping needs 2*T*k*(out+in) flops instead of 2*T*out*in + 2*out*in*k and
// forms no weight tile at all.  Two kernels on the tile engine:
//   1. t[tok, m] = sum_o dy[tok, o] * C[o, m]            (dense; t is a bf16 [tokens x k] scratch in the workspace)
//   2. dx[tok, i] = sum_m t[tok, m] * noise(PRIME*i + m)  (the noise operand is hashed straight into the pipeline's
//                                                          registers, stage by stage, interleaved with the MFMAs)
// Replaces autograd's MmBackward on the re-materialised weight (materialize() + dense product,
// src/rten_cpp/RandumbTensor.py:942-946).
#include "rdb_blocks.hpp"
#include "rdb_stationary.hpp"
#include <algorithm>
#include <type_traits>

namespace rdb {

int num_compute_units();   // rdb_error.hip

constexpr int X_BK = 64;

// ----------------------------------------------------------------------------------------------- kernel 1: t = dy . C
// tile: 128 coefficient columns (engine rows "a") x 64 tokens (engine rows "b"), contraction over out_f.  The output is
// small (tokens x k), so the token tile is kept short to have a block for every compute unit; loads run two stages ahead.
constexpr int K1_BC = 128, K1_BT = 64;
// pipeline shape of the dy.C blocks that take C^T straight into registers: contraction per stage, stages per unrolled trip,
// how many stages ahead dy is loaded, wave priority
#ifndef RDB_DYC_BKD
#define RDB_DYC_BKD 128
#endif
#ifndef RDB_DYC_TRIP
#define RDB_DYC_TRIP 2
#endif
#ifndef RDB_DYC_DSTG
#define RDB_DYC_DSTG 2
#endif
#ifndef RDB_DYC_PRIO
#define RDB_DYC_PRIO 2
#endif

struct DyCParams {
    const bf16_t *dy;
    const bf16_t *coef;
    const bf16_t *ctf;      // NULL, or C transposed in fragment order (rows = coefficients), valid when *ctf_flag != 0
    const uint32_t *ctf_flag;
    int osteps, kpad;       // of ctf: k-steps per row block (out_f rounded up to 64, / 16), k rounded up to 64
    bf16_t *t;
    float *zero;     // NULL, or an array this launch clears on the side (16-byte aligned, zero_n a multiple of 4)
    int64_t zero_n;
    int64_t lddy;
    int tokens, out_f, k;
    int tiles_c, tiles_t;
    // the contraction is added up in `ranges` ranges of range_len output features, range by range, whoever computes them.  part == NULL:
    // every block runs its tile's ranges one after the other; else a block per tile and range, whose sums go to
    // part[range][token][coefficient] for dyc_sum_kernel
    float *part;
    int ranges, range_len;
    int frag_ksteps;  // 0: t row-major [tokens x k]; else t in fragment order with this many k-steps per 32 tokens and scaled
                      // by 2^-31, for the kernel that keeps it in registers (rdb_stationary.hpp)
};

// A range's sums, waves as WM x (4 / WM): four consecutive coefficients of a token a lane and store
template <int MI, int NI, int WM>
__device__ __forceinline__ void dyc_store_part(const DyCParams &p, const f32x16 (&acc)[MI][NI], int range, int m0, int tok0)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 31, g = lane >> 5, wm = wave / (4 / WM), wn = wave % (4 / WM);
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
        const int tok = tok0 + wn * NI * 32 + ni * 32 + r;
        if (tok >= p.tokens) continue;
        float *row = p.part + ((int64_t)range * p.tokens + tok) * p.k;
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int jq = 0; jq < 4; ++jq) {
                const int m = m0 + wm * MI * 32 + mi * 32 + 8 * jq + 4 * g;
                if (m < p.k)   // k is a multiple of 8
                    *reinterpret_cast<f32x4 *>(row + m) = f32x4{acc[mi][ni][jq * 4], acc[mi][ni][jq * 4 + 1], acc[mi][ni][jq * 4 + 2], acc[mi][ni][jq * 4 + 3]};
            }
    }
}

// `block`: index of this block among the blocks that run this body.
__device__ __forceinline__ void dyc_block(const DyCParams &p, bf16_t *lds, int block)
{
    // work item = (range, token tile, coefficient tile), coefficient tile fastest: neighbours share the dy tile
    const int tiles = p.tiles_c * p.tiles_t, items = p.part ? tiles * p.ranges : tiles, wr = xcd_work_item(block, items);
    if (wr >= items) return;
    const int range = wr / tiles, w = wr - range * tiles, last = p.part ? range : p.ranges - 1;
    const int m0 = (w % p.tiles_c) * K1_BC, tok0 = (w / p.tiles_c) * K1_BT;
    f32x16 acc[K1_BC / 64][K1_BT / 64], sum[K1_BC / 64][K1_BT / 64];
    for (int rg = range; rg <= last; ++rg) {
        const int o_begin = rg * p.range_len, o_end = min(p.out_f, o_begin + p.range_len);
#pragma unroll
        for (int mi = 0; mi < K1_BC / 64; ++mi)
#pragma unroll
            for (int ni = 0; ni < K1_BT / 64; ++ni) acc[mi][ni] = zero16();
        // "A": C[o][m], tile rows = m (contiguous in memory), contraction index = o
        GlobalOperand<K1_BC, X_BK, M_CONT> opc = {p.coef, (int64_t)p.k, m0, p.k, o_end, (int64_t)p.out_f * p.k};
        // "B": dy[tok][o], contraction index contiguous
        GlobalOperand<K1_BT, X_BK, K_CONT> opdy = {p.dy, p.lddy, tok0, p.tokens, o_end, (int64_t)(p.tokens - 1) * p.lddy + p.out_f};
        gemm_mainloop<K1_BC, K1_BT, X_BK, 2, 2>(acc, lds, opc, opdy, o_begin, (o_end - o_begin + X_BK - 1) / X_BK);
        if (last == range) break;
        __syncthreads();   // the next range begins by writing the stage buffers
#pragma unroll
        for (int mi = 0; mi < K1_BC / 64; ++mi)
#pragma unroll
            for (int ni = 0; ni < K1_BT / 64; ++ni) {
                if (rg > range) sum[mi][ni] += acc[mi][ni];
                else sum[mi][ni] = acc[mi][ni];
                acc[mi][ni] = sum[mi][ni];
            }
    }
    if (p.part)
        dyc_store_part<K1_BC / 64, K1_BT / 64, 2>(p, acc, range, m0, tok0);
    else if (p.frag_ksteps)
        store_tile_bf16_frag<K1_BC, K1_BT>(acc, lds, p.t, p.frag_ksteps, m0, p.frag_ksteps * 16, tok0, (p.tokens + 31) / 32 * 32,
                                           4.656612873077392578125e-10f);
    else
        store_tile_bf16<K1_BC, K1_BT>(acc, lds, p.t, p.k, m0, p.k, tok0, p.tokens, 1.0f, nullptr);
    RDB_STAMP(3);
}

// The same block with C taken from its transposed, fragment-ordered copy: only dy passes through LDS.  The four waves split
// the coefficient rows (one 32-row block each, no fragment loaded twice) and share the 64 tokens.  RD: how many stages ahead C's fragments are
// loaded (bwd_dc_dyc_kernel).
template <int RD> __device__ __forceinline__ void dyc_block_direct(const DyCParams &p, bf16_t *lds, int block)
{
    const int tiles = p.tiles_c * p.tiles_t, items = p.part ? tiles * p.ranges : tiles, wr = xcd_work_item(block, items);
    if (wr >= items) return;
    const int range = wr / tiles, w = wr - range * tiles, last = p.part ? range : p.ranges - 1;
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int m0 = (w % p.tiles_c) * K1_BC, tok0 = (w / p.tiles_c) * K1_BT;
    f32x16 acc[1][K1_BT / 32], sum[K1_BT / 32];
    // stages of 128: half as many barriers (and waits for the first fragments after them) as with 64, for the same LDS
    constexpr int BKD = RDB_DYC_BKD;
    FragSource fc;
    fc.init(p.ctf, (int64_t)p.kpad * p.osteps * 16, p.osteps, (m0 >> 5) + wave, lane);
    // these blocks are the longer ones of the launch they share with the coefficient-gradient blocks: their waves issue first
    __builtin_amdgcn_s_setprio(RDB_DYC_PRIO);
    for (int rg = range; rg <= last; ++rg) {
        const int o_begin = rg * p.range_len, o_end = min(p.out_f, o_begin + p.range_len);
#pragma unroll
        for (int ni = 0; ni < K1_BT / 32; ++ni) acc[0][ni] = zero16();
        GlobalOperand<K1_BT, BKD, K_CONT> opdy = {p.dy, p.lddy, tok0, p.tokens, o_end, (int64_t)(p.tokens - 1) * p.lddy + p.out_f};
        direct_mainloop<K1_BT / 32, 1, BKD / 16, false, RDB_DYC_TRIP, RDB_DYC_DSTG, RD>(acc, lds, opdy, fc, o_begin, (o_end - o_begin + BKD - 1) / BKD, 0,
                                                                                               lane);
        if (last == range) break;
        __syncthreads();   // the next range begins by writing the stage buffers
#pragma unroll
        for (int ni = 0; ni < K1_BT / 32; ++ni) {
            if (rg > range) sum[ni] += acc[0][ni];
            else sum[ni] = acc[0][ni];
            acc[0][ni] = sum[ni];
        }
    }
    if (p.part)
        dyc_store_part<1, K1_BT / 32, 4>(p, acc, range, m0, tok0);
    else if (p.frag_ksteps)
        store_tile_bf16_frag<K1_BC, K1_BT, 4>(acc, lds, p.t, p.frag_ksteps, m0, p.frag_ksteps * 16, tok0, (p.tokens + 31) / 32 * 32,
                                              4.656612873077392578125e-10f);
    else
        store_tile_bf16<K1_BC, K1_BT, 4>(acc, lds, p.t, p.k, m0, p.k, tok0, p.tokens, 1.0f, nullptr);
    RDB_STAMP(3);
}

// t from the ranges' sums, added in range order: eight coefficients of a token a thread, row-major or in fragment order (as store_tile_bf16_frag
// writes it: tokens padded to 32 and coefficients to a multiple of 64 with zeros, times 2^-31)
__global__ __launch_bounds__(256) void dyc_sum_kernel(DyCParams p, int pieces, int k8)
{
    const int e = (int)blockIdx.x * 256 + threadIdx.x;
    if (e >= pieces) return;
    const int tok = e / k8, m = (e - tok * k8) * 8;
    f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = lo;
    if (tok < p.tokens && m < p.k) {
        const float *src = p.part + (int64_t)tok * p.k + m;
        const int64_t stride = (int64_t)p.tokens * p.k;
        f32x4 a[8], b[8];   // at most eight ranges, all in flight
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float *q = src + (int64_t)min(i, p.ranges - 1) * stride;
            a[i] = *reinterpret_cast<const f32x4 *>(q);
            b[i] = *reinterpret_cast<const f32x4 *>(q + 4);
        }
        lo = a[0];
        hi = b[0];
#pragma unroll
        for (int i = 1; i < 8; ++i)
            if (i < p.ranges) {
                lo += a[i];
                hi += b[i];
            }
    }
    bf16_t *dst = p.t + (int64_t)tok * p.k + m;
    if (p.frag_ksteps) {
        lo *= 4.656612873077392578125e-10f;
        hi *= 4.656612873077392578125e-10f;
        dst = p.t + ((int64_t)(tok >> 5) * p.frag_ksteps + (m >> 4)) * 512 + (((m >> 3) & 1) * 32 + (tok & 31)) * 8;
    }
    const i32x4 h = {(int)f32x2_to_bf16x2(lo[0], lo[1]), (int)f32x2_to_bf16x2(lo[2], lo[3]), (int)f32x2_to_bf16x2(hi[0], hi[1]),
                     (int)f32x2_to_bf16x2(hi[2], hi[3])};
    *reinterpret_cast<i32x4 *>(dst) = h;
}

__global__ __launch_bounds__(256, 2) void dx_dyc_kernel(DyCParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    if (p.zero) {  // a kernel later in the stream accumulates into this array with atomics
        const f32x4 z4 = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < p.zero_n / 4; e += (int64_t)gridDim.x * 256)
            reinterpret_cast<f32x4 *>(p.zero)[e] = z4;
    }
    dyc_block(p, reinterpret_cast<bf16_t *>(smem_raw), blockIdx.x);
}

// ----------------------------------------------------------------------------------------------- kernel 2: dx = t . N
// body in rdb_blocks.hpp (tn_block)
__global__ __launch_bounds__(256, 1) void dx_tn_kernel(TNParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    tn_block(p, reinterpret_cast<bf16_t *>(smem_raw), blockIdx.x);
}

// ----------------------------------------------------------------------------------------------- dC and dx = t . N in one launch
// The coefficient-gradient blocks (LDS- and matrix-core-bound) and the dx = t.N blocks (bound by the integer hash on the
// vector ALU) are independent once t, z and a zeroed dcoef exist, and lean on different units: launched as one grid, two
// blocks per compute unit, they overlap instead of queueing.  Both bodies use exactly 80 KB of LDS.
struct BwdParams {
    DcParams dc;
    TNParams tn;
    int dc_blocks;  // multiple of 8, so both parts keep their die assignment
};

__global__ __launch_bounds__(256, 2) void bwd_dc_tn_kernel(BwdParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    bf16_t *lds = reinterpret_cast<bf16_t *>(smem_raw);
    if ((int)blockIdx.x < p.dc_blocks)
        dc_block_direct(p.dc, lds, blockIdx.x);
    else
        tn_block(p.tn, lds, blockIdx.x - p.dc_blocks);
}

// ----------------------------------------------------------------------------------------------- the backward pass regrouped
// With room for the coefficient gradient's partial sums in the workspace nothing has to be zeroed first, so the two long
// contractions over dy, t = dy.C and dC = dy^T.z, can share a launch: both run the tile engine with four waves a block and
// wait on memory much of the time, and two blocks per compute unit fill each other's gaps (they also read the same dy).
// The second launch runs the dx = t.N blocks and, beside them, the blocks that add the partial sums up in split order.
struct BwdAParams {
    DcParams dc;
    DyCParams dyc;
    int dc_blocks;  // multiple of 8, so both parts keep their die assignment
};

// RD: see dyc_block_direct.  Where the blocks of t = dy . C take half the compute units or fewer, each is a chain of stages that wait for C's
// fragments, and two stages ahead shorten it (528 tokens x 384 -> 1536, k = 112, 9 blocks of 12 stages: 14.2 us -> 11.7; 700 x 2000 -> 1000, k = 128:
// 10.0 -> 8.6; 5000 x 1000 -> 1000, k = 64: 10.6 -> 9.4); with a block or more a unit the others' work fills the waits, and the 24 registers are missed
// (8192 x 768 -> 3072, k = 256: 34.5 -> 36.5; 4096 tokens: 27.7 -> 28.2).
// NOISE: blocks behind those write the tables that the second launch reads: N, and with a fused random bias R (big_dx_kernel).
struct BwdTables {
    NoiseTable r, n;
    int first;   // their first block
};
template <int RD, bool NOISE> __global__ __launch_bounds__(256, 2) void bwd_dc_dyc_kernel(BwdAParams p, std::conditional_t<NOISE, BwdTables, int> tables)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    bf16_t *lds = reinterpret_cast<bf16_t *>(smem_raw);
    if constexpr (NOISE) {
        if ((int)blockIdx.x >= tables.first) {
            const uint32_t at = (blockIdx.x - (uint32_t)tables.first) * 256u + threadIdx.x, step = (gridDim.x - (uint32_t)tables.first) * 256u;
            noise_table(tables.n, at, step);
            noise_table(tables.r, at, step);
            return;
        }
    }
    if ((int)blockIdx.x < p.dc_blocks) {
        dc_block_direct(p.dc, lds, blockIdx.x);
    } else {
        if (p.dyc.ctf && *p.dyc.ctf_flag)   // the forward pass left the transposed coefficients in the state
            dyc_block_direct<RD>(p.dyc, lds, blockIdx.x - p.dc_blocks);
        else
            dyc_block(p.dyc, lds, blockIdx.x - p.dc_blocks);
    }
}

struct BwdBParams {
    TNParams tn;
    RedParams red;
    int tn_blocks;
};

__global__ __launch_bounds__(256, 2) void bwd_tn_red_kernel(BwdBParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    if ((int)blockIdx.x < p.tn_blocks)
        tn_block(p.tn, reinterpret_cast<bf16_t *>(smem_raw), blockIdx.x);
    else
        red_block(p.red, blockIdx.x - p.tn_blocks, gridDim.x - p.tn_blocks);
}

// dx = t . N for k <= 256 with t held in registers (rdb_stationary.hpp), alone and beside the reduction blocks.
template <int KG, int AUX> __global__ __launch_bounds__(ST_THREADS, 1) void dx_tns_kernel(StParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    stationary_block<KG, false, true, AUX, true>(p, smem_raw, blockIdx.x);
}

struct BwdBsParams {
    StParams tn;
    RedParams red;
    int tn_blocks;
};

template <int KG, int AUX, bool TABLE, int SIDE = ST_ALONE> __global__ __launch_bounds__(ST_THREADS, 1) void bwd_tns_red_kernel(BwdBsParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    if ((int)blockIdx.x < p.tn_blocks)
        stationary_block<KG, false, !TABLE, AUX, true, TABLE, SIDE>(p.tn, smem_raw, blockIdx.x);
    else
        red_block(p.red, blockIdx.x - p.tn_blocks, gridDim.x - p.tn_blocks);
}

// ----------------------------------------------------------------------------------------------- host side
void dc_params_from_state(DcParams &p, const void *state, const rdb_linear_desc *d);   // rdb_factored.hip

static bool dx_factored_ok(const rdb_linear_desc *d)
{
    return d->act_dtype == RDB_BF16 && d->coef_dtype == RDB_BF16 && d->coef_rows != 0 && d->k % 8 == 0 && d->in_f % 8 == 0 &&
           d->out_f % 8 == 0 && d->k > 0 && d->tokens > 0 && d->tokens < (1 << 30) && d->in_f < (1 << 30) && d->out_f < (1 << 30) &&
           d->k < (1 << 24) && d->tokens * d->k < (1ll << 29) && d->out_f * d->k < (1ll << 29);
}

// t = dy.C: [tokens x k] bf16, or, for the kernel that keeps t in registers, tokens padded to 32 and k to 64
int64_t linear_dx_factored_workspace(const rdb_linear_desc *d)
{
    if (!dx_factored_ok(d)) return 0;
    if (d->k <= ST_KMAX && cdiv(d->tokens, 32) * 32 * cdiv(d->k, 64) * 64 < (1ll << 29))
        return cdiv(d->tokens, 32) * 32 * cdiv(d->k, 64) * 64 * (int64_t)sizeof(bf16_t);
    return d->tokens * d->k * (int64_t)sizeof(bf16_t);
}

static int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }

// Workspace of the regrouped backward pass: t, then the partial sums of the coefficient gradient.
// force_partial: also with a single token range (the call adds to dcoef instead of overwriting it).
int64_t linear_bwd_projected_workspace(const rdb_linear_desc *d, int num_cus, bool force_partial)
{
    if (!dx_factored_ok(d)) return 0;
    DcParams dc;
    make_dc_params(dc, nullptr, nullptr, d->out_f, d, num_cus);
    if (dc.splits == 1 && !force_partial) return linear_dx_factored_workspace(d);   // a single token range is stored straight into dcoef
    return align256(linear_dx_factored_workspace(d)) + (int64_t)dc.splits * d->out_f * d->k * (int64_t)sizeof(float);
}

// Ranges of t = dy . C where its tiles are half the compute units or fewer and each contracts 2048 output features or more (k > 256: 2560): a
// block walks through them at 0.75 to 1 us a stage of 128 while the launch's other blocks are long done (the two launches, and the one without:
// 300 tokens x 512 -> 2560, k = 64: 11.1 us, 13.7; 2000, k = 256: 19.4, 20.3; 300 x 512 -> 3584, k = 512: 15.9, 27.7; at 2048 features, k = 64, 200
// and 256: 10.9, 11.4; 14.2, 13.0; 17.5, 19.7; with k = 304 16.6, 14.1).  At least 512 output features a range, four stages (with 1024: 446 x 792 -> 4168, k = 64: 16.4 us, now 12.1; 1056 x 768 -> 3072, k =
// 240: 19.0, now 16.7; 384 gains nothing more), at most eight ranges.  Up to five eighths of the units and from 4096 features on, two ranges still
// pay (3010 x 1024 -> 7736, k = 272, 144 tiles: 68 -> 54 us; 158 tiles: 76 either way; 192: 59 -> 69, and 142 tiles of 3072 features 30 -> 36).
// Not where the 256-wide tiles take the layer when they are switched on: those contract in one range, and both give the same bits.  The rule
// knows nothing of workspaces: without room for the ranges' sums a block adds its tile's ranges up itself, to the same bits.
static int dyc_ranges(const rdb_linear_desc *d, int num_cus, int *range_len)
{
    const int64_t tiles = cdiv(d->k, K1_BC) * cdiv(d->tokens, K1_BT);
    int64_t r = std::min<int64_t>(std::min<int64_t>(num_cus / tiles, d->out_f / 512), 8);
    if (r < 2 && tiles * 8 <= num_cus * 5 && d->out_f >= 4096) r = 2;
    if (r < 2 || d->out_f < (d->k <= ST_KMAX ? 2048 : 2560) || big_bwd_enough(d, num_cus)) r = 1;
    *range_len = (int)(cdiv(cdiv(d->out_f, r), 128) * 128);
    return (int)cdiv(d->out_f, *range_len);
}
static void make_dyc_params(DyCParams &p1, const void *dy, int64_t lddy, const void *coef, void *t, const rdb_linear_desc *d)
{
    p1.dy = (const bf16_t *)dy;
    p1.coef = (const bf16_t *)coef;
    p1.ctf = nullptr;
    p1.ctf_flag = nullptr;
    p1.osteps = 0;
    p1.kpad = 0;
    p1.t = (bf16_t *)t;
    p1.zero = nullptr;
    p1.zero_n = 0;
    p1.lddy = lddy;
    p1.tokens = (int)d->tokens;
    p1.out_f = (int)d->out_f;
    p1.k = (int)d->k;
    p1.tiles_c = (int)cdiv(d->k, K1_BC);
    p1.tiles_t = (int)cdiv(d->tokens, K1_BT);
    p1.part = nullptr;
    p1.ranges = dyc_ranges(d, num_compute_units(), &p1.range_len);
    p1.frag_ksteps = 0;
}

// Scratch for N^T where dx = t . N with t in registers takes it from memory, written by the first launch beside its products; 0: where it is hashed
// under the matrix instructions.  Those hide the hash of a unit of up to 128 coefficients, no more: from 136 up each step of a block is the vector
// ALU's.  Not where a block takes one unit (nothing is hashed under anything, and the units come from memory a round trip later), nor below 12 token
// tiles (every value is hashed once a tile), nor with two units where adding up a large dC beside them takes as long.  us of the backward call,
// hashed and from memory: 8192 tokens x 3072 -> 768, k = 256, 192, 128 and 64: 44.9, 37.5; 40.0, 36.5; 35.6, 36.1; 27.6, 29.7; 8192 x 768 -> 768,
// k = 256 (two units): 24.9, 24.4; 3072 x 8192 -> 1024, k = 136: 45.5, 36.0; 6000 x 1000 -> 1000, k = 192: 25.3, 23.5; 3072 x 3072 -> 4096, k = 256:
// 39.3, 39.6; one unit: 4096 x 768 -> 768, k = 256: 20.6, 21.2; two and a large dC: 8192 x 768 -> 3072, k = 256: 42.6, 43.0; 9 tiles: 2304 x 3072 ->
// 768, k = 256: 20.0, 20.5; 3 tiles: 600 x 4096 -> 512, k = 256: 12.5, 13.7.
static int64_t tns_table_bytes(const rdb_linear_desc *d, int num_cus)
{
    const int64_t bytes = cdiv(d->in_f, 32) * 32 * cdiv(d->k, 64) * 64 * (int64_t)sizeof(bf16_t);
    if (d->k <= 128 || d->k > ST_KMAX || bytes >= (1ll << 30)) return 0;
    StParams q;
    make_stationary_grid(q, d->tokens, d->in_f, num_cus);
    return q.tiles_t >= 12 && q.units_per_split >= (d->out_f <= 2 * d->in_f ? 2 : 3) ? bytes : 0;
}
// Scratch of the regrouped backward pass that it can do without: the ranges' sums and behind them, or later in their place (k > 256), N^T for dx = t . N
// (table false: for the random bias's form, which has room for N^T of its own)
int64_t linear_bwd_projected_extra(const rdb_linear_desc *d, int num_cus, bool table)
{
    if (!dx_factored_ok(d)) return 0;
    int len;
    const int ranges = dyc_ranges(d, num_cus, &len);
    const int64_t part = ranges > 1 ? align256(ranges * d->tokens * d->k * (int64_t)sizeof(float)) : 0;
    return table ? std::max<int64_t>(part + tns_table_bytes(d, num_cus), dx_big_table_bytes(d, num_cus)) : part;
}

// t . N with t in registers applies when k is short enough and dx fits a buffer descriptor.
static bool tn_stationary_ok(const rdb_linear_desc *d, int64_t lddx)
{   // dx and the padded, fragment-ordered t must each fit a buffer descriptor
    return d->k <= ST_KMAX && d->tokens * lddx < (1ll << 29) && cdiv(d->tokens, 32) * 32 * cdiv(d->k, 64) * 64 < (1ll << 29);
}

static int make_tns_params(StParams &q, void *dx, int64_t lddx, const void *t, const rdb_linear_desc *d, int num_cus)
{
    q.z = (const bf16_t *)t;
    q.coef = nullptr;
    q.bias = nullptr;
    q.y = (bf16_t *)dx;
    q.ldy = lddx;
    q.k = (int)d->k;
    q.seed = d->seed;
    return make_stationary_grid(q, d->tokens, d->in_f, num_cus);
}

// Returns RDB_E_UNSUPPORTED (without setting an error) when the request does not fit this algorithm.
int linear_dx_factored(void *dx, int64_t lddx, const void *dy, int64_t lddy, const void *coef, const void *scale_bias,
                       const rdb_linear_desc *d, int num_cus, void *workspace, int64_t workspace_bytes, hipStream_t s)
{
    if (!dx_factored_ok(d) || scale_bias) return RDB_E_UNSUPPORTED;  // the random-bias term is not low rank
    if (!workspace || workspace_bytes < linear_dx_factored_workspace(d) || ((uintptr_t)workspace & 15)) return RDB_E_UNSUPPORTED;
    if (d->tokens * lddy >= (1ll << 29)) return RDB_E_UNSUPPORTED;
    if (lddy % 8 || lddx % 8 || ((uintptr_t)dy & 15) || ((uintptr_t)coef & 15) || ((uintptr_t)dx & 15)) return RDB_E_UNSUPPORTED;
    // AUTO: up to 16 times the flops of one product on a stored W (the same bound as the forward's: see cheaper_factored there)
    if (d->algo == RDB_ALGO_AUTO && d->k * (d->in_f + d->out_f) >= 16 * d->in_f * d->out_f) return RDB_E_UNSUPPORTED;

    DyCParams p1;
    make_dyc_params(p1, dy, lddy, coef, workspace, d);
    const bool stationary = tn_stationary_ok(d, lddx);
    const int kg = (int)cdiv(d->k, 64);
    if (stationary) p1.frag_ksteps = kg * 4;
    int rc = launch_engine(dx_dyc_kernel, p1, p1.tiles_c * p1.tiles_t, engine_smem<K1_BC, K1_BT, X_BK, M_CONT, K_CONT>(), s, "dx_dyc_kernel");
    if (rc) return rc;
    if (stationary) {
        StParams q;
        const int items = make_tns_params(q, dx, lddx, workspace, d, num_cus);
        return with_stationary_variant(q, [&](auto kgc, auto aux) {
            return launch_stationary(dx_tns_kernel<decltype(kgc)::value, decltype(aux)::value>, q, items, stationary_smem(kgc), s, "dx_tns_kernel");
        });
    }
    TNParams p2;
    const int items = make_tn_params(p2, dx, lddx, workspace, d);
    return launch_engine(dx_tn_kernel, p2, items, engine_smem<K2_BI, K2_BT, X_BK, K_CONT, K_CONT>(), s, "dx_tn_kernel");
}

// Whether dx may leave through the gradient of a squared ReLU: where t stays in registers and rows are whole lines (the other kernels are not built for it)
bool linear_bwd_projected_gates(const rdb_linear_desc *d, const void *dx, int64_t lddx, const void *gate)
{
    return dx_factored_ok(d) && tn_stationary_ok(d, lddx) && lddx % 64 == 0 && ((uintptr_t)dx & 127) == 0 && ((uintptr_t)gate & 15) == 0;
}

// Which of the two launches linear_bwd_projected enqueues: bit 0 the first, bit 1 the second (3: both).  Timing tools launch one
// of them alone (rdb_linear_bwd_projected_part); the mask is the calling thread's.
static thread_local int g_bwd_parts = 3;
void set_bwd_projected_parts(int mask) { g_bwd_parts = mask & 3; }

// Blocks that write the tables, behind the others: short ones, so that every unit that is done with the products finds one.  They take a product's
// registers and LDS and so run mostly as the launch's tail: what they save is launches and passes over memory, not the hash (34.4 us without tables and 39.8
// with N and R, 2.6 M values, at 8192 tokens x 768 -> 3072, k = 256).  us of the step with 32,
// 128, 512 and 1024 of them on 256 units: 8192 tokens x 768 -> 3072, k = 256: 176.4, 167.6, 164.8, 164.4; 4096 x 1536 -> 4096, k = 128: 197.5, 177.1,
// 169.8, 170.0; 4096 x 4096 -> 8192, k = 256: 856, 727, 707, 717; 8192 x 2048 -> 768, k = 64: 116.8, 113.5, 113.4, 113.5.
static int table_blocks(uint32_t pieces, int num_cus) { return (int)std::min<int64_t>(cdiv(pieces, 256), 2 * num_cus); }

// Whole backward pass of the layer from the saved projection z: dx = (dy.C).N and dcoef = dy^T.z in two launches.
// Returns RDB_E_UNSUPPORTED (without setting an error) when the request does not fit.
// accumulate: dcoef += instead of dcoef = (a later chunk of tokens of a layer whose activations are passed in chunks).
// dc_bf16: dcoef is bf16 [out_f x k], the fp32 sums rounded once by the blocks that add them up (needs the workspace with room
// for the sums, linear_bwd_projected_workspace(d, num_cus, true), and is not combined with accumulate).
// rb: NULL, or the fused random bias's share, for layers whose t stays in registers otherwise (tn_stationary_ok).
// gate: NULL, or a matrix as dx is: dx = (dy.C).N * 2 relu(gate), where linear_bwd_projected_gates.
int linear_bwd_projected(void *dx, int64_t lddx, float *dcoef, const void *dy, int64_t lddy, const void *z, const void *coef,
                         const rdb_linear_desc *d, int num_cus, void *workspace, int64_t workspace_bytes, bool accumulate, bool dc_bf16,
                         hipStream_t s, const RBiasDx *rb, const void *gate)
{
    if (!dx_factored_ok(d)) return RDB_E_UNSUPPORTED;
    if (gate && (rb || accumulate || !linear_bwd_projected_gates(d, dx, lddx, gate) || workspace_bytes < linear_bwd_projected_workspace(d, num_cus, dc_bf16)))
        return RDB_E_UNSUPPORTED;
    if (rb && (accumulate || !tn_stationary_ok(d, lddx) || workspace_bytes < linear_bwd_projected_workspace(d, num_cus, dc_bf16))) return RDB_E_UNSUPPORTED;
    if (dc_bf16 && (accumulate || workspace_bytes < linear_bwd_projected_workspace(d, num_cus, true))) return RDB_E_UNSUPPORTED;
    if (!workspace || workspace_bytes < linear_dx_factored_workspace(d) || ((uintptr_t)workspace & 15)) return RDB_E_UNSUPPORTED;
    if (d->tokens * lddy >= (1ll << 29) || lddy % 8 || lddx % 8) return RDB_E_UNSUPPORTED;
    if (((uintptr_t)dy & 15) || ((uintptr_t)coef & 15) || ((uintptr_t)dx & 15) || ((uintptr_t)z & 15) || ((uintptr_t)dcoef & 15))
        return RDB_E_UNSUPPORTED;
    DyCParams p1;
    make_dyc_params(p1, dy, lddy, coef, workspace, d);
    const size_t smem_dc = engine_smem<KD_BO, KD_BM, X_BK, M_CONT, M_CONT>(), smem_tn = engine_smem<K2_BI, K2_BT, X_BK, K_CONT, K_CONT>();
    const size_t smem_dyc = engine_smem<K1_BC, K1_BT, X_BK, M_CONT, K_CONT>();
    if (workspace_bytes >= linear_bwd_projected_workspace(d, num_cus, accumulate || dc_bf16)) {
        BwdAParams a;
        const int dc_items = make_dc_params(a.dc, dcoef, dy, lddy, d, num_cus);
        dc_params_from_state(a.dc, z, d);
        // one token range only (the 256-wide tiles always have one): its sums are the result, stored straight into dcoef, and
        // nothing is left to add up
        const bool big = big_bwd_applies(d, num_cus) && !tn_stationary_ok(d, lddx) && p1.ranges == 1;   // more than one: only when they are forced on
        const bool direct = !accumulate && (big || (a.dc.splits == 1 && !dc_bf16));
        a.dc.partial = direct ? dcoef : reinterpret_cast<float *>(static_cast<char *>(workspace) + align256(linear_dx_factored_workspace(d)));
        a.dyc = p1;
        {   // the transposed coefficients, if the forward pass left them in the state (its header says so)
            const ProjLayout L = proj_layout(d);
            a.dyc.ctf = reinterpret_cast<const bf16_t *>(static_cast<const char *>(z) + L.ctf_off);
            a.dyc.ctf_flag = static_cast<const uint32_t *>(z);
            a.dyc.osteps = (int)(L.out64 / 16);
            a.dyc.kpad = L.kpad;
        }
        if (tn_stationary_ok(d, lddx)) a.dyc.frag_ksteps = (int)cdiv(d->k, 64) * 4;   // the t.N kernel below keeps t in registers
        const int64_t base = align256(linear_bwd_projected_workspace(d, num_cus, accumulate || dc_bf16));
        if (a.dyc.ranges > 1 && workspace_bytes >= base + align256(a.dyc.ranges * d->tokens * d->k * (int64_t)sizeof(float)))
            a.dyc.part = reinterpret_cast<float *>(static_cast<char *>(workspace) + base);
        const int64_t table_at = base + (a.dyc.part ? align256(a.dyc.ranges * d->tokens * d->k * (int64_t)sizeof(float)) : 0), table_n = tns_table_bytes(d, num_cus);
        bf16_t *n = rb ? rb->n : nullptr;   // N^T in memory, or none
        if (!rb && table_n && tn_stationary_ok(d, lddx) && workspace_bytes >= table_at + table_n)
            n = reinterpret_cast<bf16_t *>(static_cast<char *>(workspace) + table_at);
        a.dc_blocks = xcd_grid_size(dc_items);
        int rc = RDB_OK;
        const int red_splits = big ? 1 : a.dc.splits;
        if (!(g_bwd_parts & 1)) {
        } else if (big) {
            // long coefficient dimension and many tiles: both products on 256-wide tiles; a dC tile contracts all tokens, so
            // there is one set of sums, stored into dcoef or, when it is to be added to, where the first split's would go
            rc = linear_bwd_big(workspace, a.dc.partial, direct && dc_bf16, dy, lddy, z, coef, d, num_cus, true, true, s);
        } else {
            size_t smem = smem_dc > smem_dyc ? smem_dc : smem_dyc;
            const int dyc_items = p1.tiles_c * p1.tiles_t * (a.dyc.part ? a.dyc.ranges : 1);
            const int blocks = a.dc_blocks + xcd_grid_size(dyc_items);
            if (n) {
                const BwdTables tables = {rb ? rbias_dx_table(*rb, d) : NoiseTable{}, noise_dx_table(n, d), blocks};
                auto kernel = dyc_items * 2 <= num_cus ? bwd_dc_dyc_kernel<2, true> : bwd_dc_dyc_kernel<1, true>;
                if (int rl = reserve_lds(reinterpret_cast<const void *>(kernel), smem, "bwd_dc_dyc_kernel")) return rl;
                kernel<<<blocks + table_blocks(tables.r.pieces + tables.n.pieces, num_cus), 256, smem, s>>>(a, tables);
            } else {
                auto kernel = dyc_items * 2 <= num_cus ? bwd_dc_dyc_kernel<2, false> : bwd_dc_dyc_kernel<1, false>;
                if (int rl = reserve_lds(reinterpret_cast<const void *>(kernel), smem, "bwd_dc_dyc_kernel")) return rl;
                kernel<<<blocks, 256, smem, s>>>(a, 0);
            }
            rc = check_launch("bwd_dc_dyc_kernel");
            if (!rc && a.dyc.part) {
                const int k8 = a.dyc.frag_ksteps ? a.dyc.frag_ksteps * 2 : (int)d->k / 8;
                const int pieces = (int)(a.dyc.frag_ksteps ? cdiv(d->tokens, 32) * 32 : d->tokens) * k8;
                dyc_sum_kernel<<<(unsigned)cdiv(pieces, 256), 256, 0, s>>>(a.dyc, pieces, k8);
                rc = check_launch("dyc_sum_kernel");
            }
        }
        if (rc) return rc;
        if (!(g_bwd_parts & 2)) return RDB_OK;
        RedParams red;
        red.partial = a.dc.partial;
        red.out = dcoef;
        red.n = d->out_f * d->k;
        red.splits = red_splits;
        red.accumulate = accumulate ? 1 : 0;
        red.out_bf16 = dc_bf16 ? 1 : 0;
        if (rb) return linear_dx_rbias_big(dx, lddx, workspace, dy, lddy, *rb, direct ? nullptr : &red, d, num_cus, s);
        if (tn_stationary_ok(d, lddx)) {
            BwdBsParams bs;
            const int items = make_tns_params(bs.tn, dx, lddx, workspace, d, num_cus);
            bs.red = red;
            bs.tn_blocks = xcd_grid_size(items);
            // One element (of all splits) a thread while there are units for it: a turn is a round trip to memory of 1.5 us, and with 16 loads
            // a thread a few blocks were still adding when the product was done (528 tokens x 384 -> 1536, k = 112: 16 blocks 7.6 us, 84
            // blocks 3.6; 3008 x 768 -> 2304, k = 96: 5.7 -> 4.1).
            int rblocks = (int)std::min<int64_t>(cdiv(red.n / 4, ST_THREADS), num_cus);
            // A block of this kernel has a compute unit to itself: where the product's blocks leave units free, no more reduction
            // blocks than those, so that the launch is one round of blocks (8192 tokens x 768 -> 3072, k = 256, 64 units: 9.8 us against
            // 11.2 with 128 blocks).  Less than a quarter of the chip would still be adding long after the product is done, and a second
            // round is cheaper: 6784 x 576 -> 1728, k = 256, 8 units: 10.5 against 50.4; 4000 x 960 -> 4096, k = 128, 32 units: 8.6
            // against 20.0; 8192 x 448 -> 4096, k = 256, 32 units: 11.6 against 18.4.
            const int spare = num_cus - bs.tn_blocks;
            if (spare > 0 && rblocks > spare && std::min(rblocks, num_cus / 2) <= 2 * spare) rblocks = spare;
            if (rblocks < 1) rblocks = 1;
            if (direct) rblocks = 0;
            bs.tn.coef = n;
            bs.tn.side = static_cast<bf16_t *>(const_cast<void *>(gate));   // read
            return with_stationary_variant(bs.tn, [&](auto kg, auto aux) {
                constexpr int KG = decltype(kg)::value, AUX = decltype(aux)::value;
                auto kernel = n ? bwd_tns_red_kernel<KG, AUX, (KG > 2)> : bwd_tns_red_kernel<KG, AUX, false>;   // no table up to k = 128
                if constexpr (AUX == Y_STREAM)
                    if (gate) kernel = n ? bwd_tns_red_kernel<KG, AUX, (KG > 2), ST_GATE> : bwd_tns_red_kernel<KG, AUX, false, ST_GATE>;
                const size_t smem_s = stationary_smem(kg);
                if (int rl = reserve_lds(reinterpret_cast<const void *>(kernel), smem_s, "bwd_tns_red_kernel")) return rl;
                kernel<<<bs.tn_blocks + rblocks, ST_THREADS, smem_s, s>>>(bs);
                return check_launch("bwd_tns_red_kernel");
            });
        }
        const int64_t table = dx_big_table_bytes(d, num_cus);
        if (direct && table && workspace_bytes >= base + table) {   // nothing to add up, and room for N^T
            rc = linear_tn_big(dx, lddx, workspace, static_cast<char *>(workspace) + base, d, num_cus, s);
            if (rc != RDB_E_UNSUPPORTED) return rc;
        }
        BwdBParams b;
        const int tn_items = make_tn_params(b.tn, dx, lddx, workspace, d);
        b.tn_blocks = xcd_grid_size(tn_items);
        b.red = red;
        int red_blocks = (int)cdiv(b.red.n / 4 * b.red.splits, 256 * 16);   // two blocks a unit: no gain from more
        if (red_blocks > num_cus) red_blocks = num_cus;
        if (red_blocks < 1) red_blocks = 1;
        if (direct) red_blocks = 0;
        if (int rl = reserve_lds(reinterpret_cast<const void *>(bwd_tn_red_kernel), smem_tn, "bwd_tn_red_kernel")) return rl;
        bwd_tn_red_kernel<<<b.tn_blocks + red_blocks, 256, smem_tn, s>>>(b);
        return check_launch("bwd_tn_red_kernel");
    }
    // workspace for t only: dy.C first (clearing dcoef on the side), then the coefficient gradient with atomics beside t.N
    p1.zero = accumulate ? nullptr : dcoef;
    p1.zero_n = d->out_f * d->k;
    int rc = launch_engine(dx_dyc_kernel, p1, p1.tiles_c * p1.tiles_t, smem_dyc, s, "dx_dyc_kernel");
    if (rc) return rc;
    BwdParams p;
    const int dc_items = make_dc_params(p.dc, dcoef, dy, lddy, d, num_cus);
    dc_params_from_state(p.dc, z, d);
    const int tn_items = make_tn_params(p.tn, dx, lddx, workspace, d);
    p.dc_blocks = xcd_grid_size(dc_items);
    const size_t smem = smem_dc > smem_tn ? smem_dc : smem_tn;
    if (int rl = reserve_lds(reinterpret_cast<const void *>(bwd_dc_tn_kernel), smem, "bwd_dc_tn_kernel")) return rl;
    bwd_dc_tn_kernel<<<p.dc_blocks + xcd_grid_size(tn_items), 256, smem, s>>>(p);
    return check_launch("bwd_dc_tn_kernel");
}

}  // namespace rdb
