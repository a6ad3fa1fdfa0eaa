// The factored algorithm's dense products on 256-wide tiles, for layers with a long coefficient dimension (k > 256) and
// enough tiles to give every compute unit one:
//   big_y_kernel    y[tok, o]  = sum_m z[tok, m] * C[o, m] (+ bias[o])          256 (o) x 256 (tok) tiles
//   big_bwd_kernel  t[tok, m]  = sum_o dy[tok, o] * C[o, m]                       256 (m) x 128 (tok) tiles, and in the same launch
//                   dC[o, m]   = sum_tok dy[tok, o] * z[tok, m]                   256 (o) x 256 (m) tiles over all tokens
//   big_z_kernel    z[tok, m]  = sum_i x[tok, i] * N[m, i]                        256 (m) x 128 (tok) tiles, N from memory
//   big_yr_kernel   y[tok, o]  = z . C^T + s * x . R^T (any k)                    256 (o) x 128 (tok) tiles, R from memory
//   big_rbias_kernel  y += s * x . R^T,  dx += s * dy . R (any k)                 256 (features) x 128 (tok) tiles, R from memory
//   big_y_kernel    dx[tok, i] = sum_m t[tok, m] * N[m, i]                        256 (i) x 256 (tok) tiles, N from memory
// z, z^T and C^T come from the projection state in fragment order (rdb_direct.hpp: ProjLayout).  One persistent block per
// compute unit (rdb_big.hpp).  Replaces materialize() + dense product and MmBackward's two products
// (src/rten_cpp/RandumbTensor.py:942-946, 979-990) for such layers, as the 128-wide kernels of rdb_factored.hip / rdb_dx.hip do
// for all others.
#include "rdb_big.hpp"
#include "rdb_blocks.hpp"
#include <atomic>
#include <type_traits>

namespace rdb {

constexpr int BG = 256;   // tile edge

// Work item w of the forward product -> (output tile, token tile).  Neighbouring items run at the same time on one die: they
// are numbered so that 32 of them cover 8 output tiles x 4 token tiles (6 MB of operands, which a die's L2 holds) rather
// than 32 x 1 (16.5 MB): groups of 4 token tiles, walked through output tile by output tile.
constexpr int BY_GROUP_T = 4;
__device__ __forceinline__ void big_y_decode(int w, int tiles_o, int tiles_t, int &to, int &tt)
{
    const int per_group = BY_GROUP_T * tiles_o, group = w / per_group, in_group = w - group * per_group;
    const int first_t = group * BY_GROUP_T, gsize = tiles_t - first_t < BY_GROUP_T ? tiles_t - first_t : BY_GROUP_T;
    to = in_group / gsize;
    tt = first_t + in_group - to * gsize;
}

// 0: never use these kernels, 1: when the layer has enough tiles (default), 2: whenever the shapes allow (tests)
static std::atomic<int> g_big_mode{1};
void set_big_tiles_mode(int mode) { g_big_mode.store(mode < 0 ? 0 : mode > 2 ? 2 : mode); }
int big_tiles_mode() { return g_big_mode.load(); }

static bool enough_tiles(int64_t tiles, int num_cus)
{
    const int mode = g_big_mode.load();
    return mode == 2 || (mode == 1 && tiles * 2 >= num_cus);
}

// Rows row0 .. of a [rows x cols] matrix in fragment order, rows padded to 32 and columns to 64
template <int ROWS> __device__ __forceinline__ void frag_rows(FragOperand<ROWS, 64> &op, const bf16_t *src, int rows, int cols, int row0)
{
    op.src = src;
    op.ksteps = ((cols + 63) >> 6) * 4;
    op.nrb = (rows + 31) >> 5;
    op.rb0 = row0 >> 5;
    op.klim_steps = op.ksteps;
}

// ----------------------------------------------------------------------------------------------- y = z . C^T
// Also dx = t . N, with N^T [in_f x k] in fragment order in the place of C and t row-major: a noise value of a 64 x 256 tile's product is hashed again
// for every 256 tokens, and at k > 256 that, not the matrix cores, is what the product waits for (4096 tokens x 4096, k = 1024: 57 us
// for 34 GFLOP).  Written once (in_f * k values, 6 us) and read back the same product takes 39.
struct BigYParams {
    const bf16_t *zf;   // FRAG: fragment order, rows = tokens (tok32 / 32 row blocks), kpad / 16 k-steps; else [tokens x k] row-major
    const bf16_t *coef;
    const bf16_t *bias;
    bf16_t *y;
    int64_t ldy, y_elems;
    int tokens, out_f, k, kpad, tok32;
    int tiles_o, tiles_t;
};

// Tiles are dealt out in rounds of one per block.  A last round that would occupy at most half of the blocks is dealt out as
// half tiles (256 output features x 128 tokens) instead, two blocks to a tile, so that no block idles through a whole tile.
constexpr int BY_HALF = 128;

template <int ROWS, bool FRAG> struct BigTokens {   // z (or t): rows = tokens
    typedef typename std::conditional<FRAG, FragOperand<ROWS, 64>, GlobalOperand<ROWS, 64, K_CONT>>::type Operand;
    static __device__ __forceinline__ void set(Operand &pb, const BigYParams &p, int tok0)
    {
        if constexpr (FRAG) {
            pb.src = p.zf;
            pb.ksteps = p.kpad >> 4;
            pb.nrb = p.tok32 >> 5;
            pb.rb0 = tok0 >> 5;
            pb.klim_steps = p.kpad >> 4;
        } else {
            pb = Operand{p.zf, (int64_t)p.k, tok0, p.tokens, p.k, (int64_t)p.tokens * p.k};
        }
    }
};

template <bool BIAS, bool FRAG = true> __global__ __launch_bounds__(256, 1) void big_y_kernel(BigYParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    bf16_t *lds = reinterpret_cast<bf16_t *>(smem_raw);
    typedef typename std::conditional<FRAG, GlobalOperand<BG, 64, K_CONT>, FragOperand<BG, 64>>::type PA;   // C (N^T): rows = output features
    typedef typename BigTokens<BG, FRAG>::Operand PB;
    typedef typename BigTokens<BY_HALF, FRAG>::Operand PH;   // the tokens of a half tile
    const int total = p.tiles_o * p.tiles_t, vtotal = (total + 7) / 8 * 8, nblk = gridDim.x, nstage = (p.k + 63) / 64;
    const int full_rounds = vtotal / nblk, rest = vtotal - full_rounds * nblk;
    const bool halves = rest > 0 && 2 * rest <= nblk;
    const int my_rounds = full_rounds + ((!halves && (int)blockIdx.x < rest) ? 1 : 0);
    // this block's r-th tile: virtual index v -> work item w (a die's items are neighbours: they share z tiles and C)
    int r = 0;
#ifdef RDB_STAMPS
    int rdb_stamp_seq = 0;   // a timing harness records the block's tiles one after the other
#endif
    auto next = [&]() {
        for (; r < my_rounds; ++r) {
            const int w = xcd_work_item(r * nblk + (int)blockIdx.x, total);
            if (w < total) { ++r; return w; }
        }
        return -1;
    };
    PA pa;
    auto init_a = [&](int to) {
        if constexpr (FRAG) pa = PA{p.coef, (int64_t)p.k, to * BG, p.out_f, p.k, (int64_t)p.out_f * p.k};
        else frag_rows(pa, p.coef, p.out_f, p.k, to * BG);
    };
    int w = next();
    if (w >= 0) {
        PB pb;
        BigRegs<PA, PB> regs;
        auto request = [&](int w) {
            int to, tt;
            big_y_decode(w, p.tiles_o, p.tiles_t, to, tt);
            init_a(to);
            BigTokens<BG, FRAG>::set(pb, p, tt * BG);
            big_prefetch(regs, pa, pb, 0);
        };
        request(w);
        while (true) {
            int to, tt;
            big_y_decode(w, p.tiles_o, p.tiles_t, to, tt);
            const int o0 = to * BG, tok0 = tt * BG;
            f32x16 acc[BG / 64][BG / 64];
            RDB_STAMP(0);
            big_zero<BG, BG>(acc);
            big_mainloop<BG, BG>(acc, lds, regs, pa, pb, nstage);
            RDB_STAMP(1);
            BigBias<BG> bias;   // requested ahead of the next tile's first stages, which the epilogue does not wait for
            if (BIAS) big_load_bias<BG>(bias, p.bias, o0, p.out_f);
            const int wn = next();
            if (wn >= 0) request(wn);   // on its way while this tile leaves
            __builtin_amdgcn_sched_barrier(0);
            RDB_STAMP(2);
            big_store_bf16<BG, BG, BIAS, true>(acc, lds, p.y, p.ldy, p.y_elems, o0, p.out_f, tok0, p.tokens, bias, opaque_tid());
            RDB_STAMP(3);
#ifdef RDB_STAMPS
            ++rdb_stamp_seq;
#endif
            if (wn < 0) break;
            w = wn;
        }
    }
    if (!halves || (int)blockIdx.x >= 2 * rest) return;
    w = xcd_work_item(full_rounds * nblk + ((int)blockIdx.x >> 1), total);
    if (w >= total) return;
    {
        int to, tt;
        big_y_decode(w, p.tiles_o, p.tiles_t, to, tt);
        const int o0 = to * BG, tok0 = tt * BG + ((int)blockIdx.x & 1) * BY_HALF;
        PH pb;
        BigRegs<PA, PH> regs;
        init_a(to);
        BigTokens<BY_HALF, FRAG>::set(pb, p, tok0);
        big_prefetch(regs, pa, pb, 0);
        f32x16 acc[BG / 64][BY_HALF / 64];
        big_zero<BG, BY_HALF>(acc);
        RDB_STAMP(0);
        big_mainloop<BG, BY_HALF>(acc, lds, regs, pa, pb, nstage);
        RDB_STAMP(1);
        BigBias<BG> bias;
        if (BIAS) big_load_bias<BG>(bias, p.bias, o0, p.out_f);
        RDB_STAMP(2);
        big_store_bf16<BG, BY_HALF, BIAS, true>(acc, lds, p.y, p.ldy, p.y_elems, o0, p.out_f, tok0, p.tokens, bias, opaque_tid());
        RDB_STAMP(3);
    }
}

// ----------------------------------------------------------------------------------------------- t = dy . C and dC = dy^T . z
constexpr int BT_TOK = 128;   // token edge of a t tile

struct BigBwdParams {
    const bf16_t *dy;
    int64_t lddy;
    const bf16_t *coef;
    const bf16_t *ctf;            // C transposed in fragment order (rows = coefficients), valid when *ctf_flag != 0
    const uint32_t *ctf_flag;
    const bf16_t *ztf;            // z transposed in fragment order (rows = coefficients)
    bf16_t *t;                    // [tokens x k] row-major
    void *dc;                     // [out_f x k], fp32 or bf16: dcoef itself, or the fp32 area a reduction adds to dcoef
    int tokens, out_f, k, kpad;
    int osteps, tsteps;           // k-steps per row block of ctf (out_f rounded up to 64, / 16) and of ztf (tokens likewise)
    int t_tiles_m, t_tiles_t;     // t tiles: 256 coefficients x 128 tokens; 0 tiles: the launch computes dC only
    int c_tiles_o, c_tiles_m;     // dC tiles: 256 output features x 256 coefficients; 0 tiles: t only
    int t_first;                  // the t tiles come first in the list (they are the longer ones), else the dC tiles
};

// t tiles of one block.  CT: C^T from its fragment-ordered copy; otherwise C itself, staged as an M_CONT operand.
template <bool CT> __device__ __forceinline__ void big_t_items(const BigBwdParams &p, bf16_t *lds, int &r, int base, int n1)
{
    const int n1v = (n1 + 7) / 8 * 8;
    typedef typename std::conditional<CT, FragOperand<BG, 64>, GlobalOperand<BG, 64, M_CONT>>::type PA;   // rows = coefficients
    typedef GlobalOperand<BT_TOK, 64, K_CONT> PB;                                                          // dy: rows = tokens
    const int nblk = gridDim.x, nstage = (p.out_f + 63) / 64;
    auto next = [&]() {
        for (;; ++r) {
            const int v = big_item(blockIdx.x, r, nblk) - base;
            if (v >= n1v) return -1;   // r stays at the first round past the t tiles
            const int w = xcd_work_item(v, n1);
            if (w < n1) { ++r; return w; }
        }
    };
    PA pa;
    PB pb;
    BigRegs<PA, PB> regs;
    auto request = [&](int w) {
        const int m0 = (w % p.t_tiles_m) * BG, tok0 = (w / p.t_tiles_m) * BT_TOK;
        if constexpr (CT) {
            pa.src = p.ctf;
            pa.ksteps = p.osteps;
            pa.nrb = p.kpad >> 5;
            pa.rb0 = m0 >> 5;
            pa.klim_steps = p.osteps;
        } else {
            pa = PA{p.coef, (int64_t)p.k, m0, p.k, p.out_f, (int64_t)p.out_f * p.k};
        }
        pb = PB{p.dy, p.lddy, tok0, p.tokens, p.out_f, (int64_t)(p.tokens - 1) * p.lddy + p.out_f};
        big_prefetch(regs, pa, pb, 0);
    };
    int w = next();
    if (w < 0) return;
    request(w);
    while (true) {
        const int m0 = (w % p.t_tiles_m) * BG, tok0 = (w / p.t_tiles_m) * BT_TOK;
        f32x16 acc[BG / 64][BT_TOK / 64];
        big_zero<BG, BT_TOK>(acc);
        big_mainloop<BG, BT_TOK>(acc, lds, regs, pa, pb, nstage);
        const int wn = next();
        if (wn >= 0) request(wn);
        __builtin_amdgcn_sched_barrier(0);
        big_store_bf16<BG, BT_TOK, false>(acc, lds, p.t, p.k, (int64_t)p.tokens * p.k, m0, p.k, tok0, p.tokens, BigBias<BG>(), opaque_tid());
        if (wn < 0) break;
        w = wn;
    }
}

// dC tiles of one block, from the block's round r on; `base`: index of the first dC tile in the launch's list.
template <typename E> __device__ __forceinline__ void big_dc_items(const BigBwdParams &p, bf16_t *lds, int &r, int base, int n2)
{
    typedef GlobalOperand<BG, 64, M_CONT> PA;   // dy: rows = output features, contraction = tokens
    typedef FragOperand<BG, 64> PB;             // z^T: rows = coefficients
    const int nblk = gridDim.x, nstage = (p.tokens + 63) / 64, n2v = (n2 + 7) / 8 * 8;
    auto next = [&]() {
        for (;; ++r) {
            const int v = big_item(blockIdx.x, r, nblk) - base;
            if (v >= n2v) return -1;
            const int w = xcd_work_item(v, n2);
            if (w < n2) { ++r; return w; }
        }
    };
    PA pa;
    PB pb;
    BigRegs<PA, PB> regs;
    auto request = [&](int w) {
        pa = PA{p.dy, p.lddy, (w / p.c_tiles_m) * BG, p.out_f, p.tokens, (int64_t)(p.tokens - 1) * p.lddy + p.out_f};
        pb.src = p.ztf;
        pb.ksteps = p.tsteps;
        pb.nrb = p.kpad >> 5;
        pb.rb0 = (w % p.c_tiles_m) * (BG / 32);
        pb.klim_steps = p.tsteps;
        big_prefetch(regs, pa, pb, 0);
    };
    int w = next();
    if (w < 0) return;
    request(w);
    while (true) {
        const int m0 = (w % p.c_tiles_m) * BG, o0 = (w / p.c_tiles_m) * BG;
        f32x16 acc[BG / 64][BG / 64];
        big_zero<BG, BG>(acc);
        big_mainloop<BG, BG>(acc, lds, regs, pa, pb, nstage);
        const int wn = next();
        if (wn >= 0) request(wn);
        __builtin_amdgcn_sched_barrier(0);
        big_store_rows<BG, BG, E>(acc, lds, static_cast<E *>(p.dc), p.k, (int64_t)p.out_f * p.k, o0, p.out_f, m0, p.k, opaque_tid());
        if (wn < 0) break;
        w = wn;
    }
}

// The launch's list holds the tiles of the longer kind first (a t tile contracts out_f with half-size stages, a dC tile the
// tokens) and is dealt out to the blocks in rows of alternating direction (big_item): the blocks that got a long tile in
// one row get the later, shorter ones of the next.  A block's rounds walk through the list in order, so it finishes its
// tiles of the first kind before it starts on the second.  E: dC's type.  A bf16 gradient leaves rounded from here: as fp32 sums
// for the second launch to round it was 118 MB more through memory at 4096 -> 14336, k = 1024, and that launch waited for it
// (125 us where its product takes 57).
template <typename E> __global__ __launch_bounds__(256, 1) void big_bwd_kernel(BigBwdParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    bf16_t *lds = reinterpret_cast<bf16_t *>(smem_raw);
    const int n1 = p.t_tiles_m * p.t_tiles_t, n1v = (n1 + 7) / 8 * 8, n2 = p.c_tiles_o * p.c_tiles_m, n2v = (n2 + 7) / 8 * 8;
    const bool ct = n1 && p.ctf && *p.ctf_flag;
    int r = 0;
    if (p.t_first) {
        if (n1) {
            if (ct) big_t_items<true>(p, lds, r, 0, n1);
            else big_t_items<false>(p, lds, r, 0, n1);
        }
        if (n2) big_dc_items<E>(p, lds, r, n1v, n2);
    } else {
        if (n2) big_dc_items<E>(p, lds, r, 0, n2);
        if (n1) {
            if (ct) big_t_items<true>(p, lds, r, n2v, n1);
            else big_t_items<false>(p, lds, r, n2v, n1);
        }
    }
}

// ----------------------------------------------------------------------------------------------- z = x . N^T
// For layers with as many tiles as half the compute units.  The kernel that hashes (factored_z_kernel) has 32 x 256 tiles: every noise
// value hashed again for every 256 tokens, x read again for every 32 coefficients, 2 KB out of LDS per matrix instruction (4096 tokens x
// 4096, k = 1024: 96 us for 34 GFLOP).  Blocks past the tiles transpose C for the backward pass, 64 x 256 of it at a time.
struct BigZParams {
    const bf16_t *noise;   // N [k x in_f] in fragment order
    const bf16_t *x;
    int64_t ldx;
    bf16_t *zf, *ztf;      // z and z^T in fragment order (ProjLayout)
    uint32_t *flag;        // header of the state
    const bf16_t *coef;    // NULL, or C [out_f x k], to leave transposed in ctf
    bf16_t *ctf;
    int tokens, in_f, out_f, k, kpad, tok32, tok64, out64;
    int tiles_m, tiles_t, tile_blocks;
};
constexpr int BZ_TOK = 128;

// 16 rows (the contraction) x 32 columns of an LDS matrix with row stride LD, as the fragment whose rows are those columns
template <int LD> __device__ __forceinline__ f32x4 transposed_frag(const bf16_t *src, int lane)
{
    const int sl = lane & 15, qq = (lane >> 4) & 1, g = lane >> 5;
    const bf16_t *p = src + (g * 8 + (sl >> 2)) * LD + qq * 16 + (sl & 3) * 4;
    Frag8 f;
    f.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(p));
    f.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(p + 4 * LD));
    return f.f4;
}

__device__ __forceinline__ void transpose_coef(const BigZParams &p, bf16_t *lds, int block, int nblocks)
{
    constexpr int LD = BG + 32;   // 64 bytes of padding: the four rows of a transposing read cover all banks
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63, osteps = p.out64 >> 4, mt = (p.kpad + BG - 1) / BG;
    for (int w = block; w < (p.out64 >> 6) * mt; w += nblocks) {
        const int o0 = (w / mt) * 64, m0 = (w % mt) * BG;
        f32x4 v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int o = o0 + q * 8 + (t >> 5), m = m0 + (t & 31) * 8;
            v[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (o < p.out_f && m < p.k) v[q] = *reinterpret_cast<const f32x4 *>(p.coef + (int64_t)o * p.k + m);   // k is a multiple of 8
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) *reinterpret_cast<f32x4 *>(lds + (q * 8 + (t >> 5)) * LD + (t & 31) * 8) = v[q];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int mb = wave * 2 + (q >> 2), ks = q & 3;
            const f32x4 f = transposed_frag<LD>(lds + ks * 16 * LD + mb * 32, lane);
            if (m0 + mb * 32 < p.kpad)
                store_stream(reinterpret_cast<f32x4 *>(p.ctf + ((int64_t)((m0 >> 5) + mb) * osteps + (o0 >> 4) + ks) * 512 + lane * 8), f);
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(256, 1) void big_z_kernel(BigZParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    bf16_t *lds = reinterpret_cast<bf16_t *>(smem_raw);
    if ((int)blockIdx.x >= p.tile_blocks) {
        transpose_coef(p, lds, (int)blockIdx.x - p.tile_blocks, (int)gridDim.x - p.tile_blocks);
        return;
    }
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63, r = lane & 31, g = lane >> 5, wm = wave >> 1, wn = wave & 1;
    if (blockIdx.x == 0 && t == 0) {
        p.flag[0] = p.coef ? 1u : 0u;
        p.flag[1] = 0u;
    }
    const int total = p.tiles_m * p.tiles_t, w = xcd_work_item(blockIdx.x, total);   // coefficient tile fastest: neighbours share the x tile
    if (w >= total) return;
    const int m0 = (w % p.tiles_m) * BG, tok0 = (w / p.tiles_m) * BZ_TOK;
    typedef FragOperand<BG, 64> PA;
    typedef GlobalOperand<BZ_TOK, 64, K_CONT> PB;
    PA pa;
    frag_rows(pa, p.noise, p.k, p.in_f, m0);
    PB pb = {p.x, p.ldx, tok0, p.tokens, p.in_f, (int64_t)(p.tokens - 1) * p.ldx + p.in_f};
    BigRegs<PA, PB> regs;
    big_prefetch(regs, pa, pb, 0);
    constexpr int MI = BG / 64, NI = BZ_TOK / 64, LD = BG + 8;
    f32x16 acc[MI][NI];
    big_zero<BG, BZ_TOK>(acc);
    big_mainloop<BG, BZ_TOK>(acc, lds, regs, pa, pb, (p.in_f + 63) / 64);
    // D[a = coefficient][b = token] to LDS once, as bf16 rows of tokens; from there in both orders.  Coefficients past k and tokens
    // past the end are zeros.
    acc_settle<MI, NI>(acc);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni)
#pragma unroll
            for (int jq = 0; jq < 4; ++jq)
                store4<bf16_t>(lds + (wn * NI * 32 + ni * 32 + r) * LD + wm * MI * 32 + mi * 32 + 8 * jq + 4 * g, acc_read(acc[mi][ni][jq * 4 + 0]),
                               acc_read(acc[mi][ni][jq * 4 + 1]), acc_read(acc[mi][ni][jq * 4 + 2]), acc_read(acc[mi][ni][jq * 4 + 3]));
    __syncthreads();
    const int ksteps = p.kpad >> 4, tsteps = p.tok64 >> 4;
#pragma unroll
    for (int q = 0; q < BG * BZ_TOK / 8 / 256; ++q) {   // rows = tokens: a piece is 8 coefficients of one token
        const int idx = q * 256 + t, b = idx % BZ_TOK, a = (idx / BZ_TOK) * 8, gb = tok0 + b, ga = m0 + a;
        if (gb < p.tok32 && ga < p.kpad)
            *reinterpret_cast<f32x4 *>(p.zf + (((int64_t)(gb >> 5) * ksteps + (ga >> 4)) * 512 + (((ga >> 3) & 1) * 32 + (gb & 31)) * 8)) =
                *reinterpret_cast<const f32x4 *>(lds + b * LD + a);
    }
#pragma unroll
    for (int q = 0; q < BG / 32 * (BZ_TOK / 16) / 4; ++q) {   // rows = coefficients
        const int u = wave * (BG / 32 * (BZ_TOK / 16) / 4) + q, mb = u / (BZ_TOK / 16), ks = u % (BZ_TOK / 16);
        const f32x4 f = transposed_frag<LD>(lds + ks * 16 * LD + mb * 32, lane);
        if (tok0 + ks * 16 < p.tok64 && m0 + mb * 32 < p.kpad)
            store_stream(reinterpret_cast<f32x4 *>(p.ztf + ((int64_t)((m0 >> 5) + mb) * tsteps + (tok0 >> 4) + ks) * 512 + lane * 8), f);
    }
}

// ----------------------------------------------------------------------------------------------- out += s * src . R^T (or R)
// The fused random bias's share alone (rdb_rbias.hip) with R written once as bf16 and read back: layers that have no product of both shares
// (backward with more than 256 coefficients, chunks of tokens) and calls for this share.  Hashed into the product it costs its hash for every 512 tokens
// on tiles of 64 features: 63 us forward and 71 backward for 38.6 GFLOP at 8192 tokens x 768 -> 3072; here 52 forward (3072 features: 768 tiles of 256,
// three a block, each with 64 KB of dst to read and to write) and 46 backward (768 features: 256 tiles of 192, one of 48 stages a block), and 5 to 7 for R.
// Tiles of 256 features x 128 tokens or of 192 x 128 (rbias_big_rows); one persistent block a compute unit.  What the epilogue adds to is requested
// before a tile's main loop, the next tile's first stages before its epilogue.
struct BigRBiasParams {
    const bf16_t *noise;    // [cols x contraction] in fragment order
    const bf16_t *src;      // [tokens x contraction]
    bf16_t *dst;            // [tokens x cols]
    const bf16_t *scale;    // one value
    const bf16_t *other;    // DOT: [tokens x cols], what the product without s is reduced against: one sum a tile, in tile order
    BlockSum dscale;
    int64_t ld_src, ld_dst, ld_other;
    int tokens, cols, contraction, tiles_a, tiles_t;
};
constexpr int BR_TOK = 128, BR_LOW = 192;   // tokens of a tile; features of the lower kind (rbias_big_rows)

template <int BA, bool DOT> __global__ __launch_bounds__(256, 1) void big_rbias_kernel(BigRBiasParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    bf16_t *lds = reinterpret_cast<bf16_t *>(smem_raw);
    typedef FragOperand<BA, 64> PA;                 // R: rows = columns of dst
    typedef GlobalOperand<BR_TOK, 64, K_CONT> PB;   // src: rows = tokens
    constexpr int MI = BA / 64, NI = BR_TOK / 64, LDP = BA / 2 + 4;
    constexpr int LPT = BA / 16, PIECES = 32 * LPT / 64;   // 16-byte pieces of a token's features in a wave's share of the tile; pieces of a lane per 32 tokens
    const int total = p.tiles_a * p.tiles_t, vtotal = (total + 7) / 8 * 8, nblk = gridDim.x, nstage = (p.contraction + 63) / 64;
    int rd = 0;
    auto next = [&]() {
        for (; rd * nblk + (int)blockIdx.x < vtotal; ++rd) {
            const int w = xcd_work_item(rd * nblk + (int)blockIdx.x, total);
            if (w < total) { ++rd; return w; }
        }
        return -1;
    };
    PA pa;
    PB pb;
    BigRegs<PA, PB> regs;
    auto request = [&](int w) {   // feature tile fastest: neighbours share the tokens
        frag_rows(pa, p.noise, p.cols, p.contraction, (w % p.tiles_a) * BA);
        pb = PB{p.src, p.ld_src, (w / p.tiles_a) * BR_TOK, p.tokens, p.contraction, (int64_t)(p.tokens - 1) * p.ld_src + p.contraction};
        big_prefetch(regs, pa, pb, 0);
    };
    auto add_up = [&]() { sum_shares(p.dscale, total, 1, 0, nblk, reinterpret_cast<float *>(lds)); };
    int w = next();
    if (w < 0) {   // the grid is rounded up to a multiple of 8: blocks without a tile are counted too
        if (DOT) add_up();
        return;
    }
    request(w);
    const float sval = bf16_to_f32(*p.scale);
    const __amdgpu_buffer_rsrc_t rs_d = __builtin_amdgcn_make_buffer_rsrc(p.dst, 0, (int)(((int64_t)(p.tokens - 1) * p.ld_dst + p.cols) * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t rs_o =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(DOT ? p.other : p.dst), 0, DOT ? (int)(((int64_t)(p.tokens - 1) * p.ld_other + p.cols) * 2) : 0, 0x00020000);
    while (true) {
        const int a0 = (w % p.tiles_a) * BA, tok0 = (w / p.tiles_a) * BR_TOK;
        // the thread's pieces of the tile: 8 features of a token; LPT pieces cover a wave's features
        auto at = [&](int t, int ni, int q, int64_t ld) {
            const int wave = t >> 6, e = q * 64 + (t & 63), tok = tok0 + (wave & 1) * NI * 32 + ni * 32 + e / LPT;
            const int a = a0 + (wave >> 1) * MI * 32 + e % LPT * 8;   // cols is a multiple of 8: a piece lies inside or outside
            return tok < p.tokens && a < p.cols ? (uint32_t)(((int64_t)tok * ld + a) * 2) : BUFFER_OOB;
        };
        Frag8 old[NI][PIECES];
        {
            const int t = opaque_tid();
#pragma unroll
            for (int ni = 0; ni < NI; ++ni)
#pragma unroll
                for (int q = 0; q < PIECES; ++q)
                    old[ni][q].f4 = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_d, (int)at(t, ni, q, p.ld_dst), 0, 0));
        }
        f32x16 acc[MI][NI];
        big_zero<BA, BR_TOK>(acc);
        big_mainloop<BA, BR_TOK>(acc, lds, regs, pa, pb, nstage);
        const int wn = next();
        if (wn >= 0) request(wn);
        __builtin_amdgcn_sched_barrier(0);
        acc_settle<MI, NI>(acc);
        const int t = opaque_tid(), wave = t >> 6, lane = t & 63, r = lane & 31, g = lane >> 5;
        float *patch = reinterpret_cast<float *>(lds) + wave * 32 * LDP;   // 32 tokens x the wave's features
        float dot = 0.0f;
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
            Frag8 ot[PIECES];
            if (DOT) {
#pragma unroll
                for (int q = 0; q < PIECES; ++q) ot[q].f4 = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_o, (int)at(t, ni, q, p.ld_other), 0, 0));
            }
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int jq = 0; jq < 4; ++jq)
                    *reinterpret_cast<f32x4 *>(patch + r * LDP + mi * 32 + 8 * jq + 4 * g) =
                        f32x4{acc_read(acc[mi][ni][jq * 4]), acc_read(acc[mi][ni][jq * 4 + 1]), acc_read(acc[mi][ni][jq * 4 + 2]), acc_read(acc[mi][ni][jq * 4 + 3])};
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_wave_barrier();   // LDS serves a wave's instructions in order: the reads see these writes
#pragma unroll
            for (int q = 0; q < PIECES; ++q) {
                const float *src = patch + (q * 64 + lane) / LPT * LDP + (q * 64 + lane) % LPT * 8;
                const f32x4 lo = *reinterpret_cast<const f32x4 *>(src), hi = *reinterpret_cast<const f32x4 *>(src + 4);
                const uint32_t off = at(t, ni, q, p.ld_dst);
                if (DOT) {   // outside the matrix `ot` reads as zeros
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        dot = fmaf(lo[2 * e], __uint_as_float(ot[q].u[e] << 16), dot);
                        dot = fmaf(lo[2 * e + 1], __uint_as_float(ot[q].u[e] & 0xffff0000u), dot);
                        dot = fmaf(hi[2 * e], __uint_as_float(ot[q].u[2 + e] << 16), dot);
                        dot = fmaf(hi[2 * e + 1], __uint_as_float(ot[q].u[2 + e] & 0xffff0000u), dot);
                    }
                }
                const Frag8 o = old[ni][q];
                const i32x4 nw = {(int)f32x2_to_bf16x2(__uint_as_float(o.u[0] << 16) + sval * lo[0], __uint_as_float(o.u[0] & 0xffff0000u) + sval * lo[1]),
                                  (int)f32x2_to_bf16x2(__uint_as_float(o.u[1] << 16) + sval * lo[2], __uint_as_float(o.u[1] & 0xffff0000u) + sval * lo[3]),
                                  (int)f32x2_to_bf16x2(__uint_as_float(o.u[2] << 16) + sval * hi[0], __uint_as_float(o.u[2] & 0xffff0000u) + sval * hi[1]),
                                  (int)f32x2_to_bf16x2(__uint_as_float(o.u[3] << 16) + sval * hi[2], __uint_as_float(o.u[3] & 0xffff0000u) + sval * hi[3])};
                __builtin_amdgcn_raw_buffer_store_b128(nw, rs_d, (int)off, 0, 0);
            }
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();   // the patches lie where the next tile's first stage goes
        if (DOT) {   // lanes, then waves, in a fixed order
            float *wsum = reinterpret_cast<float *>(lds);
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) dot += __shfl_xor(dot, o, 64);
            if (lane == 0) wsum[wave] = dot;
            __syncthreads();
            if (t == 0) leave_share(p.dscale, w, (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]));
            __syncthreads();
        }
        if (wn < 0) break;
        w = wn;
    }
    if (DOT) add_up();
}

// ----------------------------------------------------------------------------------------------- y = z . C^T + s * x . R^T (+ bias)
// A forward pass with the fused random bias in one product: the tile's accumulators contract in_f (x with R), are scaled, and go on with
// k (z with C), so that y is written once, rounded once, and never read back (8192 tokens x 768 -> 3072, k = 256: y = z . C^T beside the
// projection and y += s x . R^T: 98 us; z, R and this: 84).  Tiles of 256 output features x 128 tokens, one persistent block a compute
// unit (256 x 256: 75 us instead of 66, the second pair of operands does not fit in registers beside 256 accumulators).
struct BigYRParams {
    const bf16_t *noise;   // R [out_f x in_f] in fragment order
    const bf16_t *x;
    const bf16_t *zf;      // fragment order, rows = tokens
    const bf16_t *coef;    // [out_f x k]
    const bf16_t *scale;   // one value
    const bf16_t *bias;
    bf16_t *y;
    int64_t ldx, ldy;
    int tokens, in_f, out_f, k, tiles_o, tiles_t;
};

template <bool BIAS> __global__ __launch_bounds__(256, 1) void big_yr_kernel(BigYRParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    bf16_t *lds = reinterpret_cast<bf16_t *>(smem_raw);
    typedef FragOperand<BG, 64> PR;                  // R: rows = output features
    typedef GlobalOperand<BR_TOK, 64, K_CONT> PX;    // x: rows = tokens
    typedef GlobalOperand<BG, 64, K_CONT> PC;        // C: rows = output features
    typedef FragOperand<BR_TOK, 64> PZ;              // z: rows = tokens
    constexpr int MI = BG / 64, NI = BR_TOK / 64;
    const int total = p.tiles_o * p.tiles_t, vtotal = (total + 7) / 8 * 8, nblk = gridDim.x;
    int rd = 0;
    auto next = [&]() {
        for (; rd * nblk + (int)blockIdx.x < vtotal; ++rd) {
            const int w = xcd_work_item(rd * nblk + (int)blockIdx.x, total);
            if (w < total) { ++rd; return w; }
        }
        return -1;
    };
    PR pr;
    PX px;
    BigRegs<PR, PX> regs;
    auto request = [&](int w) {   // output tile fastest: neighbours share the tokens
        frag_rows(pr, p.noise, p.out_f, p.in_f, (w % p.tiles_o) * BG);
        px = PX{p.x, p.ldx, (w / p.tiles_o) * BR_TOK, p.tokens, p.in_f, (int64_t)(p.tokens - 1) * p.ldx + p.in_f};
        big_prefetch(regs, pr, px, 0);
    };
    int w = next();
    if (w < 0) return;
    request(w);
    const float sval = bf16_to_f32(*p.scale);
    while (true) {
        const int o0 = (w % p.tiles_o) * BG, tok0 = (w / p.tiles_o) * BR_TOK;
        PC pc = {p.coef, (int64_t)p.k, o0, p.out_f, p.k, (int64_t)p.out_f * p.k};
        PZ pz;
        frag_rows(pz, p.zf, p.tokens, p.k, tok0);
        BigRegs<PC, PZ> regs2;
        big_prefetch(regs2, pc, pz, 0);
        f32x16 acc[MI][NI];
        big_zero<BG, BR_TOK>(acc);
        big_mainloop<BG, BR_TOK>(acc, lds, regs, pr, px, (p.in_f + 63) / 64);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) acc[mi][ni] *= sval;
        big_mainloop<BG, BR_TOK>(acc, lds, regs2, pc, pz, (p.k + 63) / 64);
        BigBias<BG> bias;
        if (BIAS) big_load_bias<BG>(bias, p.bias, o0, p.out_f);
        const int wn = next();
        if (wn >= 0) request(wn);
        __builtin_amdgcn_sched_barrier(0);
        big_store_bf16<BG, BR_TOK, BIAS, true>(acc, lds, p.y, p.ldy, (int64_t)(p.tokens - 1) * p.ldy + p.out_f, o0, p.out_f, tok0, p.tokens, bias, opaque_tid());
        if (wn < 0) break;
        w = wn;
    }
}

// ----------------------------------------------------------------------------------------------- dx = t . N + s * dy . R
// The backward pass of a layer with a fused random bias, second launch: a tile contracts dy with R, its sums times x are its share of the scale's
// gradient; scaled by s they go on with t and N, so that dx is written once, rounded once, and never read back, and N, written down by the launch
// before like R, is not hashed once a row tile.  Blocks behind the tiles' add up the coefficient gradient's token ranges: they take a tile's
// registers, one wave a SIMD, and start where a tile is done or a unit has none.  41.9 GFLOP at 8192 tokens x 768 -> 3072, k = 256, 256 tiles for 256 units: 51 us
// by itself, 46 (0.91 PFLOP/s) without those sums, 50 to 64 within a step; 4096 x 1536 -> 4096, k = 128: 56 and 54; 8192 x 1024 -> 2048, k = 256: 45 and 43.
// A tile is big_rbias_kernel's.  Where the rest goes above the 36 us of the best large products is not measured: with one tile a block nothing
// covers its start and its epilogue.  x is read as the accumulators lie, half a cache line a piece, all of it on its way before the main loop.  us of the layer's step with the random bias in launches of its own (the table, dx +=) and with this: 8192 tokens x
// 768 -> 3072, k = 256: 165.6, 160.2; 4096 x 1536 -> 4096, k = 128: 173.5, 167.3; 8192 x 2048 -> 768, k = 64: 120.7, 111.3; 8192 x 1024 -> 2048,
// k = 256: 146.8, 138.1; 5000 x 3072 -> 2000, k = 64: 212.1, 202.6; 4096 x 4096 -> 8192, k = 256: 724, 709; no size measured got slower, so all
// layers take it whose t the first launch leaves in fragment order (k <= 256; for the row-major t of longer contractions it is not built) and whose R is
// written to memory at all (rbias_big_table_bytes).
struct BigDxParams {
    const bf16_t *r, *n;    // R [in_f x out_f] and N^T [in_f x k], fragment order
    const bf16_t *dy;       // [tokens x out_f]
    const bf16_t *t;        // fragment order, rows = tokens, times 2^-31
    const bf16_t *scale;    // one value
    const bf16_t *x;        // DOT: [tokens x in_f]
    bf16_t *dx;
    BlockSum dscale;
    RedParams red;
    int64_t lddy, ldx, lddx;
    int tokens, in_f, out_f, k, tiles_a, tiles_t, tile_blocks;
};

template <int BA, bool DOT, bool STREAM> __global__ __launch_bounds__(256, 1) void big_dx_kernel(BigDxParams p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    bf16_t *lds = reinterpret_cast<bf16_t *>(smem_raw);
    if ((int)blockIdx.x >= p.tile_blocks) {
        red_block(p.red, (int)blockIdx.x - p.tile_blocks, (int)gridDim.x - p.tile_blocks);
        return;
    }
    typedef FragOperand<BA, 64> PR;                  // R, and N^T: rows = features
    typedef GlobalOperand<BR_TOK, 64, K_CONT> PY;    // dy: rows = tokens
    typedef FragOperand<BR_TOK, 64> PT;              // t: rows = tokens
    constexpr int MI = BA / 64, NI = BR_TOK / 64, LDP = BA / 2 + 4;
    constexpr int LPT = BA / 16, PIECES = 32 * LPT / 64;   // as in big_rbias_kernel
    const int total = p.tiles_a * p.tiles_t, vtotal = (total + 7) / 8 * 8, nblk = p.tile_blocks;
    int rd = 0;
    auto next = [&]() {
        for (; rd * nblk + (int)blockIdx.x < vtotal; ++rd) {
            const int w = xcd_work_item(rd * nblk + (int)blockIdx.x, total);
            if (w < total) { ++rd; return w; }
        }
        return -1;
    };
    PR pr;
    PY py;
    BigRegs<PR, PY> regs;
    auto request = [&](int w) {   // feature tile fastest: neighbours share the tokens
        frag_rows(pr, p.r, p.in_f, p.out_f, (w % p.tiles_a) * BA);
        py = PY{p.dy, p.lddy, (w / p.tiles_a) * BR_TOK, p.tokens, p.out_f, (int64_t)(p.tokens - 1) * p.lddy + p.out_f};
        big_prefetch(regs, pr, py, 0);
    };
    auto add_up = [&]() { sum_shares(p.dscale, total, 1, 0, nblk, reinterpret_cast<float *>(lds)); };
    int w = next();
    if (w < 0) {   // the grid is rounded up to a multiple of 8: blocks without a tile are counted too
        if (DOT) add_up();
        return;
    }
    request(w);
    const float sval = bf16_to_f32(*p.scale);
    const __amdgpu_buffer_rsrc_t rs_d = __builtin_amdgcn_make_buffer_rsrc(p.dx, 0, (int)(((int64_t)(p.tokens - 1) * p.lddx + p.in_f) * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t rs_x =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(DOT ? p.x : p.dx), 0, DOT ? (int)(((int64_t)(p.tokens - 1) * p.ldx + p.in_f) * 2) : 0, 0x00020000);
    while (true) {
        const int a0 = (w % p.tiles_a) * BA, tok0 = (w / p.tiles_a) * BR_TOK;
        PR pn;
        frag_rows(pn, p.n, p.in_f, p.k, a0);
        PT pt;
        frag_rows(pt, p.t, p.tokens, p.k, tok0);
        BigRegs<PR, PT> regs2;
        // x as the accumulators lie: four features of a token a lane (in_f is a multiple of 8: all inside or all outside, which reads as zeros).  A token
        // behind the last has no offset of its own: with rows far apart the 32-bit product would come round and lie between rows of x.
        uint2 xv[NI][MI][4];
        auto load_x = [&](int ni) __attribute__((always_inline)) {
            const int t = opaque_tid(), wave = t >> 6, lane = t & 63;
            const int tok = tok0 + (wave & 1) * NI * 32 + ni * 32 + (lane & 31), f = a0 + (wave >> 1) * MI * 32 + 4 * (lane >> 5);
            const uint32_t at = tok < p.tokens ? ((uint32_t)tok * (uint32_t)p.ldx + (uint32_t)f) * 2u : BUFFER_OOB;
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int jq = 0; jq < 4; ++jq) {
                    const int a = mi * 32 + 8 * jq;
                    xv[ni][mi][jq] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rs_x, (int)(f + a < p.in_f ? at + 2u * a : BUFFER_OOB), 0, 0));
                }
        };
        // x is requested ahead of the main loop, and what registers still hold: the second contraction's first stage with 192 features or without x
        constexpr bool BOTH = !DOT || BA == BR_LOW;
        if (DOT) {
#pragma unroll
            for (int ni = 0; ni < NI; ++ni) load_x(ni);
        }
        if (BOTH) big_prefetch(regs2, pn, pt, 0);
        f32x16 acc[MI][NI];
        big_zero<BA, BR_TOK>(acc);
        big_mainloop<BA, BR_TOK>(acc, lds, regs, pr, py, (p.out_f + 63) / 64);
        if (!BOTH) big_prefetch(regs2, pn, pt, 0);
        float dot = 0.0f;
        acc_settle<MI, NI>(acc);
        // one accumulator tile at a time, back in its registers and part of the sum before the next is read (see acc_read; with the sum left to the
        // compiler all values wait for it, 46 of them in scratch)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) {
#pragma unroll
                for (int jq = 0; jq < 4; ++jq) {
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = acc_read(acc[mi][ni][jq * 4 + e]);
                    if (DOT) {
                        const uint2 h = xv[ni][mi][jq];
                        dot = fmaf(v[0], __uint_as_float(h.x << 16), dot);
                        dot = fmaf(v[1], __uint_as_float(h.x & 0xffff0000u), dot);
                        dot = fmaf(v[2], __uint_as_float(h.y << 16), dot);
                        dot = fmaf(v[3], __uint_as_float(h.y & 0xffff0000u), dot);
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[mi][ni][jq * 4 + e] = v[e] * sval;
                }
                asm volatile("" : "+a"(acc[mi][ni]), "+v"(dot));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        big_mainloop<BA, BR_TOK>(acc, lds, regs2, pn, pt, (p.k + 63) / 64);
        const int wn = next();
        if (wn >= 0) request(wn);
        __builtin_amdgcn_sched_barrier(0);
        acc_settle<MI, NI>(acc);
        const int t = opaque_tid(), wave = t >> 6, lane = t & 63, r = lane & 31, g = lane >> 5;
        float *patch = reinterpret_cast<float *>(lds) + wave * 32 * LDP;   // 32 tokens x the wave's features
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int jq = 0; jq < 4; ++jq)
                    *reinterpret_cast<f32x4 *>(patch + r * LDP + mi * 32 + 8 * jq + 4 * g) =
                        f32x4{acc_read(acc[mi][ni][jq * 4]), acc_read(acc[mi][ni][jq * 4 + 1]), acc_read(acc[mi][ni][jq * 4 + 2]), acc_read(acc[mi][ni][jq * 4 + 3])};
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_wave_barrier();   // LDS serves a wave's instructions in order: the reads see these writes
#pragma unroll
            for (int q = 0; q < PIECES; ++q) {
                const int e = q * 64 + lane, tok = tok0 + (wave & 1) * NI * 32 + ni * 32 + e / LPT, a = a0 + (wave >> 1) * MI * 32 + e % LPT * 8;
                const float *src = patch + e / LPT * LDP + e % LPT * 8;
                const f32x4 lo = *reinterpret_cast<const f32x4 *>(src), hi = *reinterpret_cast<const f32x4 *>(src + 4);
                const i32x4 h = {(int)f32x2_to_bf16x2(lo[0], lo[1]), (int)f32x2_to_bf16x2(lo[2], lo[3]), (int)f32x2_to_bf16x2(hi[0], hi[1]), (int)f32x2_to_bf16x2(hi[2], hi[3])};
                __builtin_amdgcn_raw_buffer_store_b128(h, rs_d, (int)(tok < p.tokens && a < p.in_f ? (uint32_t)(((int64_t)tok * p.lddx + a) * 2) : BUFFER_OOB), 0,
                                                      STREAM ? 2 : 0);
            }
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();   // the patches lie where the next tile's first stage goes
        if (DOT) {   // lanes, then waves, in a fixed order
            float *wsum = reinterpret_cast<float *>(lds);
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) dot += __shfl_xor(dot, o, 64);
            if (lane == 0) wsum[wave] = dot;
            __syncthreads();
            if (t == 0) leave_share(p.dscale, w, (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]));
            __syncthreads();
        }
        if (wn < 0) break;
        w = wn;
    }
    if (DOT) add_up();
}

// ----------------------------------------------------------------------------------------------- host side
static bool big_aligned16(const void *q) { return ((uintptr_t)q & 15) == 0; }

// Do these kernels apply to the layer's forward product / backward pass?  (The shape conditions of the 128-wide kernels are
// checked by the callers, which fall back to those kernels when the answer is no.)
bool big_fwd_applies(const rdb_linear_desc *d, int num_cus)
{
    const ProjLayout L = proj_layout(d);
    return L.ok && !L.fits_regs && enough_tiles(cdiv(d->out_f, BG) * cdiv(d->tokens, BG), num_cus);
}
// every dC tile contracts all tokens (no partial sums over token ranges), so the tiles alone must fill the chip; and the t
// tiles, each of which contracts all of out_f, must not be so few that a handful of blocks is left with all of that work
static int64_t bwd_tiles(const rdb_linear_desc *d)
{
    return std::min<int64_t>(cdiv(d->out_f, BG) * cdiv(d->k, BG), 2 * cdiv(d->k, BG) * cdiv(d->tokens, BT_TOK));
}
bool big_bwd_applies(const rdb_linear_desc *d, int num_cus)
{
    const ProjLayout L = proj_layout(d);
    return L.ok && !L.fits_regs && enough_tiles(bwd_tiles(d), num_cus);
}
// ... by their sizes, whether or not these kernels are switched on
bool big_bwd_enough(const rdb_linear_desc *d, int num_cus)
{
    const ProjLayout L = proj_layout(d);
    return L.ok && !L.fits_regs && bwd_tiles(d) * 2 >= num_cus;
}

template <class K, class P> static int launch_big(K kernel, const P &p, int items, int num_cus, size_t smem, hipStream_t s, const char *name)
{
    if (int rl = reserve_lds(reinterpret_cast<const void *>(kernel), smem, name)) return rl;
    int blocks = num_cus / 8 * 8;   // a multiple of 8: a block's tiles stay on one die's share of the list
    if (blocks < 8) blocks = 8;
    const int vitems = (items + 7) / 8 * 8;
    if (blocks > vitems) blocks = vitems;
    kernel<<<blocks, 256, smem, s>>>(p);
    return check_launch(name);
}

int linear_fwd_big(void *y, int64_t ldy, const void *state, const void *coef, const void *bias, const rdb_linear_desc *d, int num_cus, hipStream_t s)
{
    const ProjLayout L = proj_layout(d);
    if (!L.ok || d->coef_dtype != RDB_BF16 || ldy % 8 || !big_aligned16(y) || !big_aligned16(state) || !big_aligned16(coef)) return RDB_E_UNSUPPORTED;
    if (((uintptr_t)bias & 7) || d->tokens * ldy >= (1ll << 29)) return RDB_E_UNSUPPORTED;
    BigYParams p;
    p.zf = reinterpret_cast<const bf16_t *>(static_cast<const char *>(state) + L.zf_off);
    p.coef = (const bf16_t *)coef;
    p.bias = (const bf16_t *)bias;
    p.y = (bf16_t *)y;
    p.ldy = ldy;
    p.y_elems = (d->tokens - 1) * ldy + d->out_f;
    p.tokens = (int)d->tokens;
    p.out_f = (int)d->out_f;
    p.k = (int)d->k;
    p.kpad = L.kpad;
    p.tok32 = (int)L.tok32;
    p.tiles_o = (int)cdiv(d->out_f, BG);
    p.tiles_t = (int)cdiv(d->tokens, BG);
    typedef OperandTile<BG, 64, K_CONT> TA;
    typedef FragTile<BG, 64> TB;
    if (bias) return launch_big(big_y_kernel<true>, p, p.tiles_o * p.tiles_t, num_cus, big_smem<BG, BG, TA, TB>(), s, "big_y_kernel<bias>");
    return launch_big(big_y_kernel<false>, p, p.tiles_o * p.tiles_t, num_cus, big_smem<BG, BG, TA, TB>(), s, "big_y_kernel");
}

// noise_table (rdb_direct.hpp) in a launch of its own, a piece a thread
__global__ __launch_bounds__(256) void noise_frag_bf16_kernel(NoiseTable table)
{
    noise_table(table, blockIdx.x * 256u + threadIdx.x, gridDim.x * 256u);
}
// rows rounded up to 32, columns to 64
static int64_t noise_frag_bytes(int64_t rows, int64_t cols) { return cdiv(rows, 32) * 32 * cdiv(cols, 64) * 64 * (int64_t)sizeof(bf16_t); }
static NoiseTable noise_frag_table(void *out, int64_t rows, int64_t cols, uint32_t row_step, uint32_t col_step, uint32_t seed, unsigned int *cleared = nullptr,
                                   float scale = 4.656612873077392578125e-10f)
{
    return {static_cast<bf16_t *>(out), (uint32_t)(noise_frag_bytes(rows, cols) / 16), (uint32_t)(cdiv(cols, 64) * 4), (uint32_t)rows, (uint32_t)cols, row_step, col_step,
            seed, cleared, scale};
}
static int launch_noise_frag(const NoiseTable &table, hipStream_t s)
{
    noise_frag_bf16_kernel<<<(unsigned)cdiv(table.pieces, 256), 256, 0, s>>>(table);
    return check_launch("noise_frag_bf16_kernel");
}
// R [out_f x in_f] of a layer's fused random bias, R[o, i] = noise1d(o * in_f + i)
NoiseTable rbias_fwd_table(void *out, const rdb_linear_desc *d)
{
    return noise_frag_table(out, d->out_f, d->in_f, (uint32_t)d->in_f * SQ5_N1, SQ5_N1, d->seed);
}

// R for dx += s * dy . R, R[i, o] = noise1d(o * in_f + i), and N^T for t . N with a t that has the 2^-31 already
NoiseTable rbias_dx_table(const RBiasDx &rb, const rdb_linear_desc *d)
{
    return noise_frag_table(rb.r, d->in_f, d->out_f, SQ5_N1, (uint32_t)d->in_f * SQ5_N1, d->seed, rb.arrived);
}
NoiseTable noise_dx_table(bf16_t *n, const rdb_linear_desc *d) { return noise_frag_table(n, d->in_f, d->k, PN1, SQ5_N1, d->seed, nullptr, 1.0f); }

// Scratch for N^T where dx = t . N takes it from memory; 0: where it does not.
int64_t dx_big_table_bytes(const rdb_linear_desc *d, int num_cus)
{
    const ProjLayout L = proj_layout(d);
    if (!L.ok || L.fits_regs || noise_frag_bytes(d->in_f, d->k) >= (1ll << 30) || !enough_tiles(cdiv(d->in_f, BG) * cdiv(d->tokens, BG), num_cus)) return 0;
    return noise_frag_bytes(d->in_f, d->k);
}

// dx = t . N with t [tokens x k] row-major and room for N^T at `table`
int linear_tn_big(void *dx, int64_t lddx, const void *t, void *table, const rdb_linear_desc *d, int num_cus, hipStream_t s)
{
    if (!dx_big_table_bytes(d, num_cus) || lddx % 8 || d->tokens * lddx >= (1ll << 29) || !big_aligned16(dx) || !big_aligned16(t) || !big_aligned16(table))
        return RDB_E_UNSUPPORTED;
    if (int rc = launch_noise_frag(noise_frag_table(table, d->in_f, d->k, PN1, SQ5_N1, d->seed), s)) return rc;   // N^T[i, m] = noise(PRIME * i + m)
    BigYParams p = {};
    p.zf = static_cast<const bf16_t *>(t);
    p.coef = static_cast<const bf16_t *>(table);
    p.y = static_cast<bf16_t *>(dx);
    p.ldy = lddx;
    p.y_elems = (d->tokens - 1) * lddx + d->in_f;
    p.tokens = (int)d->tokens;
    p.out_f = (int)d->in_f;
    p.k = (int)d->k;
    p.tiles_o = (int)cdiv(d->in_f, BG);
    p.tiles_t = (int)cdiv(d->tokens, BG);
    typedef OperandTile<BG, 64, K_CONT> TA;
    return launch_big(big_y_kernel<false, false>, p, p.tiles_o * p.tiles_t, num_cus, big_smem<BG, BG, FragTile<BG, 64>, TA>(), s, "big_y_kernel (dx = t . N)");
}

// state <- z (and C transposed, with coef), N in `room` (room_bytes of it; the rows of the forward product to come will do)
int linear_z_big(void *state, const void *x, int64_t ldx, const void *coef, void *room, int64_t room_bytes, const rdb_linear_desc *d, int num_cus,
                 hipStream_t s)
{
    const ProjLayout L = proj_layout(d);
    const int64_t tiles = cdiv(d->k, BG) * cdiv(d->tokens, BZ_TOK);
    if (!L.ok || L.fits_regs || !enough_tiles(tiles, num_cus) || noise_frag_bytes(d->k, d->in_f) >= (1ll << 30) || !room || room_bytes < noise_frag_bytes(d->k, d->in_f))
        return RDB_E_UNSUPPORTED;
    if (ldx % 8 || d->tokens * ldx >= (1ll << 29) || !big_aligned16(x) || !big_aligned16(state) || !big_aligned16(coef) || !big_aligned16(room))
        return RDB_E_UNSUPPORTED;
    if (int rc = launch_noise_frag(noise_frag_table(room, d->k, d->in_f, SQ5_N1, PN1, d->seed), s)) return rc;   // N[m, i] = noise(PRIME * i + m)
    char *st = static_cast<char *>(state);
    BigZParams p;
    p.noise = static_cast<const bf16_t *>(room);
    p.x = static_cast<const bf16_t *>(x);
    p.ldx = ldx;
    p.zf = reinterpret_cast<bf16_t *>(st + L.zf_off);
    p.ztf = reinterpret_cast<bf16_t *>(st + L.ztf_off);
    p.flag = reinterpret_cast<uint32_t *>(st);
    p.coef = static_cast<const bf16_t *>(coef);
    p.ctf = reinterpret_cast<bf16_t *>(st + L.ctf_off);
    p.tokens = (int)d->tokens;
    p.in_f = (int)d->in_f;
    p.out_f = (int)d->out_f;
    p.k = (int)d->k;
    p.kpad = L.kpad;
    p.tok32 = (int)L.tok32;
    p.tok64 = (int)L.tok64;
    p.out64 = (int)L.out64;
    p.tiles_m = (int)cdiv(d->k, BG);
    p.tiles_t = (int)cdiv(d->tokens, BZ_TOK);
    p.tile_blocks = xcd_grid_size((int)tiles);
    const size_t smem = big_smem<BG, BZ_TOK, FragTile<BG, 64>, OperandTile<BZ_TOK, 64, K_CONT>>();
    if (int rl = reserve_lds(reinterpret_cast<const void *>(big_z_kernel), smem, "big_z_kernel")) return rl;
    // the transposing blocks: the compute units that the tiles leave free, or as many as there are
    int c_blocks = coef ? num_cus - p.tile_blocks : 0;
    if (coef && c_blocks < num_cus / 4) c_blocks = num_cus;
    big_z_kernel<<<p.tile_blocks + c_blocks, 256, smem, s>>>(p);
    return check_launch("big_z_kernel");
}

// Scratch for R where the random bias's share of [tokens x cols] takes it from memory; 0: where it does not (too few tiles, or more
// than the activations of the pass take).
int64_t rbias_big_table_bytes(const rdb_linear_desc *d, int64_t cols, int num_cus)
{
    const int64_t n = d->in_f * d->out_f, bytes = noise_frag_bytes(cols, cols == d->in_f ? d->out_f : d->in_f);
    if (d->act_dtype != RDB_BF16 || d->in_f % 8 || d->out_f % 8 || d->in_f < 8 || d->out_f < 8 || bytes >= (1ll << 30) ||
        n > d->tokens * (d->in_f + d->out_f) || !enough_tiles(cdiv(cols, BG) * cdiv(d->tokens, BR_TOK), num_cus))
        return 0;
    return bytes;
}

// Features of a tile of the product above: 192 where as many rounds of tiles as with 256 do, which are more tiles then, for compute units
// that stood idle.  A round takes 0.93 of one with 256 features, so another round is never worth it.  us of the step with
// 256 and with 192 features a tile: 8192 tokens x 768 -> 3072, k = 256, 192 and 256 tiles 179.6, 176.2; 4096 x 1536 -> 4096, k = 128, the same
// 186.6, 182.4; 8192 x 1024 -> 2048, 256 and 384: 152.9, 166.0; 5000 x 3072 -> 2000, 480 and 640: 222.2, 239.3.  us of the forward share alone (y of the
// second figure's features), the same: 8192 x 3072 -> 768, 192 and 256 tiles 52.2, 49.7; 4096 x 4096 -> 1536 65.9, 62.6; 12000 x 1024 -> 960, 376 and 470: 44.7,
// 41.1; 16384 x 2048 -> 136, 128 of either: 34.4, 33.8; another round: 8192 x 768 -> 3072, 768 and 1024: 65.3, 71.0; 8192 x 2048 -> 1024, 256 and 384: 42.0, 61.4.
static int rbias_big_rows(int64_t cols, int64_t tokens, int num_cus)
{
    auto rounds = [&](int rows) { return cdiv(cdiv(cols, rows) * cdiv(tokens, BR_TOK), num_cus); };
    return rounds(BR_LOW) <= rounds(BG) ? BR_LOW : BG;
}
int64_t rbias_big_tiles(int64_t cols, int64_t tokens, int num_cus) { return cdiv(cols, rbias_big_rows(cols, tokens, num_cus)) * cdiv(tokens, BR_TOK); }

// dst[t, a] += s * sum_c src[t, c] * noise1d(a * sR + c * sK); with `other` also the sum of the product's elements times its, to dscale, with one
// share per tile in dot_part and a word behind the table.  The caller has checked alignments and extents.
int linear_rbias_big(void *dst, int64_t ld_dst, int64_t cols, const void *src, int64_t ld_src, int64_t contraction, uint32_t sR, uint32_t sK,
                     const void *scale, const rdb_linear_desc *d, void *table, const void *other, int64_t ld_other, float *dot_part, void *dscale, int dscale_dtype,
                     int num_cus, hipStream_t s)
{
    BigRBiasParams p;
    const int ba = rbias_big_rows(cols, d->tokens, num_cus);
    p.tiles_a = (int)cdiv(cols, ba);
    p.tiles_t = (int)cdiv(d->tokens, BR_TOK);
    const int tiles = p.tiles_a * p.tiles_t;
    p.dscale = {dot_part, other ? reinterpret_cast<unsigned int *>(static_cast<char *>(table) + noise_frag_bytes(cols, contraction)) : nullptr, dscale,
                dscale_dtype == RDB_BF16};
    if (int rc = launch_noise_frag(noise_frag_table(table, cols, contraction, sR * SQ5_N1, sK * SQ5_N1, d->seed, p.dscale.arrived), s)) return rc;
    p.noise = static_cast<const bf16_t *>(table);
    p.src = static_cast<const bf16_t *>(src);
    p.dst = static_cast<bf16_t *>(dst);
    p.scale = static_cast<const bf16_t *>(scale);
    p.other = static_cast<const bf16_t *>(other);
    p.ld_src = ld_src;
    p.ld_dst = ld_dst;
    p.ld_other = ld_other;
    p.tokens = (int)d->tokens;
    p.cols = (int)cols;
    p.contraction = (int)contraction;
    auto run = [&](auto rows, auto dot) {
        constexpr int BA = decltype(rows)::value;
        constexpr size_t stages = big_smem<BA, BR_TOK, FragTile<BA, 64>, OperandTile<BR_TOK, 64, K_CONT>>();
        static_assert((size_t)4 * 32 * (BA / 2 + 4) * sizeof(float) <= stages, "the epilogue's patches fit the pipeline's LDS");
        return launch_big(big_rbias_kernel<BA, decltype(dot)::value>, p, tiles, num_cus, stages, s, "big_rbias_kernel");
    };
    auto with = [&](auto rows) { return other ? run(rows, std::true_type{}) : run(rows, std::false_type{}); };
    return ba == BG ? with(std::integral_constant<int, BG>{}) : with(std::integral_constant<int, BR_LOW>{});
}

// y = z . C^T + s * x . R^T (+ bias) from the state, R in `table` (rbias_big_table_bytes of out_f columns), where it is already if `written`
int linear_fwd_rbias_big(void *y, int64_t ldy, const void *x, int64_t ldx, const void *state, const void *coef, const void *scale, const void *bias,
                         const rdb_linear_desc *d, void *table, bool written, int num_cus, hipStream_t s)
{
    const ProjLayout L = proj_layout(d);
    if (!L.ok || d->coef_dtype != RDB_BF16 || ldx % 8 || ldy % 8 || d->tokens * ldx >= (1ll << 29) || d->tokens * ldy >= (1ll << 29)) return RDB_E_UNSUPPORTED;
    if (!big_aligned16(y) || !big_aligned16(x) || !big_aligned16(state) || !big_aligned16(coef) || !big_aligned16(table) || ((uintptr_t)bias & 7))
        return RDB_E_UNSUPPORTED;
    if (!written) {
        if (int rc = launch_noise_frag(rbias_fwd_table(table, d), s)) return rc;
    }
    BigYRParams p;
    p.noise = static_cast<const bf16_t *>(table);
    p.x = static_cast<const bf16_t *>(x);
    p.zf = reinterpret_cast<const bf16_t *>(static_cast<const char *>(state) + L.zf_off);
    p.coef = static_cast<const bf16_t *>(coef);
    p.scale = static_cast<const bf16_t *>(scale);
    p.bias = static_cast<const bf16_t *>(bias);
    p.y = static_cast<bf16_t *>(y);
    p.ldx = ldx;
    p.ldy = ldy;
    p.tokens = (int)d->tokens;
    p.in_f = (int)d->in_f;
    p.out_f = (int)d->out_f;
    p.k = (int)d->k;
    p.tiles_o = (int)cdiv(d->out_f, BG);
    p.tiles_t = (int)cdiv(d->tokens, BR_TOK);
    typedef OperandTile<BG, 64, K_CONT> TC;
    typedef OperandTile<BR_TOK, 64, K_CONT> TX;
    constexpr size_t one = big_smem<BG, BR_TOK, FragTile<BG, 64>, TX>(), two = big_smem<BG, BR_TOK, TC, FragTile<BR_TOK, 64>>(), smem = one > two ? one : two;
    if (bias) return launch_big(big_yr_kernel<true>, p, p.tiles_o * p.tiles_t, num_cus, smem, s, "big_yr_kernel<bias>");
    return launch_big(big_yr_kernel<false>, p, p.tiles_o * p.tiles_t, num_cus, smem, s, "big_yr_kernel");
}

// dx = t . N + s * dy . R and the scale's gradient, from the tables of rbias_dx_table and noise_dx_table; red: NULL, or sums to be added up behind its tiles
int linear_dx_rbias_big(void *dx, int64_t lddx, const void *t, const void *dy, int64_t lddy, const RBiasDx &rb, const RedParams *red, const rdb_linear_desc *d,
                        int num_cus, hipStream_t s)
{
    BigDxParams p = {};
    const int ba = rbias_big_rows(d->in_f, d->tokens, num_cus);
    p.r = rb.r;
    p.n = rb.n;
    p.dy = static_cast<const bf16_t *>(dy);
    p.t = static_cast<const bf16_t *>(t);
    p.scale = static_cast<const bf16_t *>(rb.scale);
    p.x = static_cast<const bf16_t *>(rb.x);
    p.dx = static_cast<bf16_t *>(dx);
    p.dscale = {rb.dots, rb.arrived, rb.dscale, rb.dscale_dtype == RDB_BF16};
    p.lddy = lddy;
    p.ldx = rb.ldx;
    p.lddx = lddx;
    p.tokens = (int)d->tokens;
    p.in_f = (int)d->in_f;
    p.out_f = (int)d->out_f;
    p.k = (int)d->k;
    p.tiles_a = (int)cdiv(d->in_f, ba);
    p.tiles_t = (int)cdiv(d->tokens, BR_TOK);
    const int vtiles = (p.tiles_a * p.tiles_t + 7) / 8 * 8;
    p.tile_blocks = std::min(std::max(num_cus / 8 * 8, 8), vtiles);
    int rblocks = 0;
    if (red) {
        p.red = *red;
        rblocks = (int)std::max<int64_t>(1, std::min<int64_t>(cdiv(red->n / 4, 256), num_cus));
        const int spare = num_cus - p.tile_blocks;
        if (spare > 0 && rblocks > spare && std::min(rblocks, num_cus / 2) <= 2 * spare) rblocks = spare;   // as beside t . N (linear_bwd_projected)
    }
    const bool stream = lddx % 64 == 0 && ((uintptr_t)dx & 127) == 0;   // rows of whole lines (Y_STREAM): 163.8 us a step at 8192 x 768 -> 3072 with plain stores, 162.4
    auto run = [&](auto rows, auto dot) {
        constexpr int BA = decltype(rows)::value;
        constexpr bool DOT = decltype(dot)::value;
        auto kernel = stream ? big_dx_kernel<BA, DOT, true> : big_dx_kernel<BA, DOT, false>;
        constexpr size_t one = big_smem<BA, BR_TOK, FragTile<BA, 64>, OperandTile<BR_TOK, 64, K_CONT>>();
        static_assert((size_t)4 * 32 * (BA / 2 + 4) * sizeof(float) <= one && big_smem<BA, BR_TOK, FragTile<BA, 64>, FragTile<BR_TOK, 64>>() <= one,
                      "the second contraction's stages and the epilogue's patches fit the first one's LDS");
        if (int rl = reserve_lds(reinterpret_cast<const void *>(kernel), one, "big_dx_kernel")) return rl;
        kernel<<<p.tile_blocks + rblocks, 256, one, s>>>(p);
        return check_launch("big_dx_kernel");
    };
    auto with = [&](auto rows) { return rb.dscale ? run(rows, std::true_type{}) : run(rows, std::false_type{}); };
    return ba == BG ? with(std::integral_constant<int, BG>{}) : with(std::integral_constant<int, BR_LOW>{});
}

// First launch of the backward pass: t (row-major, for the t . N kernel of the tile engine) and dC.  `dc`: where the
// coefficient gradient's sums go (dcoef, fp32 or, with dc_bf16, bf16; or the area a reduction adds to dcoef).  want_t / want_dc: which of the two
// (t alone needs no state, dC alone no coefficients).
int linear_bwd_big(void *t, void *dc, bool dc_bf16, const void *dy, int64_t lddy, const void *state, const void *coef, const rdb_linear_desc *d,
                   int num_cus, bool want_t, bool want_dc, hipStream_t s)
{
    const ProjLayout L = proj_layout(d);
    if (!L.ok || d->tokens * lddy >= (1ll << 29) || lddy % 8) return RDB_E_UNSUPPORTED;
    if ((want_t && (d->coef_dtype != RDB_BF16 || !coef || !t)) || (want_dc && (!state || !dc))) return RDB_E_UNSUPPORTED;
    if (!big_aligned16(dy) || !big_aligned16(state) || !big_aligned16(coef) || !big_aligned16(t) || !big_aligned16(dc)) return RDB_E_UNSUPPORTED;
    BigBwdParams p;
    p.dy = (const bf16_t *)dy;
    p.lddy = lddy;
    p.coef = (const bf16_t *)coef;
    // without a state (the input gradient called on its own) C is staged from its row-major form
    p.ctf = state ? reinterpret_cast<const bf16_t *>(static_cast<const char *>(state) + L.ctf_off) : nullptr;
    p.ctf_flag = static_cast<const uint32_t *>(state);
    p.ztf = state ? reinterpret_cast<const bf16_t *>(static_cast<const char *>(state) + L.ztf_off) : nullptr;
    p.t = (bf16_t *)t;
    p.dc = dc;
    p.tokens = (int)d->tokens;
    p.out_f = (int)d->out_f;
    p.k = (int)d->k;
    p.kpad = L.kpad;
    p.osteps = (int)(L.out64 / 16);
    p.tsteps = (int)(L.tok64 / 16);
    p.t_tiles_m = want_t ? (int)cdiv(d->k, BG) : 0;
    p.t_tiles_t = want_t ? (int)cdiv(d->tokens, BT_TOK) : 0;
    p.c_tiles_o = want_dc ? (int)cdiv(d->out_f, BG) : 0;
    p.c_tiles_m = want_dc ? (int)cdiv(d->k, BG) : 0;
    typedef OperandTile<BG, 64, M_CONT> TM;
    typedef FragTile<BG, 64> TF;
    typedef OperandTile<BT_TOK, 64, K_CONT> TD;
    constexpr size_t smem_dc = big_smem<BG, BG, TM, TF>(), smem_t = big_smem<BG, BT_TOK, TM, TD>();
    p.t_first = d->out_f >= 2 * d->tokens;   // stages of 64 at half the matrix work against stages of 64 over the tokens
    const int items = (p.t_tiles_m * p.t_tiles_t + 7) / 8 * 8 + (p.c_tiles_o * p.c_tiles_m + 7) / 8 * 8;
    const size_t smem = smem_dc > smem_t ? smem_dc : smem_t;
    if (dc_bf16) return launch_big(big_bwd_kernel<bf16_t>, p, items, num_cus, smem, s, "big_bwd_kernel<bf16>");
    return launch_big(big_bwd_kernel<float>, p, items, num_cus, smem, s, "big_bwd_kernel");
}

}  // namespace rdb
