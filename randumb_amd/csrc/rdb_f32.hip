// Fused linear layer, matrix-coef + fp32, any coefficient dimension and many tokens: the factored algorithm on the matrix
// cores at fp32 accuracy.  By default every operand value is split exactly into three bf16 parts on its way into LDS and a
// product runs as six bf16 matrix instructions (v_mfma_f32_32x32x16_bf16; see fg_split3): gfx950's bf16 matrix rate is 16 times
// its fp32 one, so six of them cost 3/8 of the eight fp32 instructions (v_mfma_f32_32x32x2_f32) they replace; the fp32
// instructions remain as the other mode of rdb_set_f32_split.
//
//   forward  z = x . N^T [T x k],  y = z . C^T (+ bias)
//   dx       t = dy . C  [T x k],  dx = t . N
//   dcoef    z as above,           dC = dy^T . z     (token ranges summed in a fixed order: bit-reproducible)
//
// N[m, i] = noise(PRIME*i + m) is hashed into the pipeline's LDS tiles and never stored; W = C . N is never formed.  All
// five products run on one kernel template that differs in where its two operands come from (a row-major matrix read along
// or across its rows, or the hash).  Operands, intermediate matrices and sums are fp32 in memory and in the accumulators.  (bf16 layers whose sizes keep them off
// the bf16 kernels, which want multiples of 8, run here too: a bf16 value is its own first part, z and t stay
// fp32, y and dx are rounded to bf16 once.)
// With scale_bias (W = C . N + s . R, R[o, i] = noise1d(o*in_f + i), full rank: src/rten_cpp/RandumbTensor.py:286-289) the
// random-bias share is one more product with R as the hashed operand, added on top:  y += s * x . R^T,  dx += s * dy . R,  and
// the gradient of s is <dy, x . R^T>, summed tile by tile in the epilogue of that product and block by block afterwards.
// Replaces materialize() + dense product (src/rten_cpp/RandumbTensor.py:942-946) and MmBackward's dW followed by
// materialize_bwd (RandumbTensor.py:979-990, 304-359) for fp32 layers beyond the few-token regime of rdb_smallk.hip.
#include "rdb_f32.hpp"
#include "rdb_sums.hpp"

namespace rdb {

int num_compute_units();   // rdb_error.hip

// out[0] = part[0] + part[1] + ... : one block, every thread a strided share in index order, then the shares in thread order
__global__ __launch_bounds__(256) void f32_sum_scalars_kernel(float *__restrict__ out, const float *__restrict__ part, int n)
{
    __shared__ float sh[256];
    float v = 0.0f;
    for (int i = threadIdx.x; i < n; i += 256) v += part[i];
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int w = 128; w >= 1; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = sh[0];
}

// One or two sums a launch: the second one's blocks follow.
__global__ __launch_bounds__(256) void f32_sum_splits_kernel(FgSum a, FgSum b)
{
    const bool second = (int)blockIdx.x >= a.blocks;
    f32_sum_block(second ? b : a, (int)blockIdx.x - (second ? a.blocks : 0), threadIdx.x);
}
static FgSum fg_sum(void *out, int out_bf16, const float *part, int64_t n, int64_t stride, int splits, const float *bias = nullptr, int64_t cols = 0)
{
    if (splits <= 1 && !bias) return {};
    const int vec = fg_aligned16(out) ? 1 : 0;   // the partial matrices are 256-byte aligned
    return {out, part, n, stride, out_bf16, splits, vec, (int)cdiv(vec ? n / 4 + n % 4 : n, 256), bias, (uint32_t)cols};
}
static int fg_launch_sums(const FgSum &a, const FgSum &b, hipStream_t s)
{
    if (!(a.blocks + b.blocks)) return RDB_OK;
    f32_sum_splits_kernel<<<(unsigned)(a.blocks + b.blocks), 256, 0, s>>>(a, b);
    return check_launch("f32_sum_splits_kernel");
}

// 1 (default): the linear layers' products run as six bf16 matrix instructions on three-way splits of their operands
// (fg_split3); 0: as fp32 matrix instructions.  Process-wide (rdb_set_f32_split).
static int g_f32_split = 1;
int f32_split_mode() { return g_f32_split; }
int set_f32_split_mode(int mode)
{
    const int old = g_f32_split;
    g_f32_split = mode ? 1 : 0;
    return old;
}

// The shapes these kernels take: matrix-coef fp32, matrices below 2^31 bytes.  Extents, leading dimensions and pointers that are
// multiples of 4 elements / 16 bytes get the kernels that read aligned pieces, everything else those that read four values at any address.
static bool fg_ok(const rdb_linear_desc *d)
{
    const bool f32 = d->act_dtype == RDB_F32 && d->coef_dtype == RDB_F32, b16 = d->act_dtype == RDB_BF16 && d->coef_dtype == RDB_BF16;
    return (f32 || b16) && d->coef_rows != 0 && d->k > 0 && d->tokens > 0 && d->in_f > 0 && d->out_f > 0 &&
           d->tokens * d->k < (1ll << 29) && d->out_f * d->k < (1ll << 29) && d->in_f < (1 << 30) && d->out_f < (1 << 30);
}
static int fg_es(int dtype) { return dtype == RDB_BF16 ? 2 : 4; }
// Wanted whenever the shapes fit: what AUTO would run instead is the general kernel, which forms W tiles on the vector ALU at a
// few TFLOP/s, so the factored form on the matrix cores wins also where it is more flops than a product on a stored W.
static bool fg_wanted(const rdb_linear_desc *) { return true; }

// z = x . N^T and t = dy . C, [tokens x k] over in_f and out_f; dC = dy^T . z, [out_f x k] over the tokens: ranges there is room for.  The
// two of the backward pass run side by side or alone, with the same sums: short contractions take one range either way.
static int z_room(const rdb_linear_desc *d, int num_cus)
{
    return fg_room(d->tokens, d->k, d->in_f, num_cus, d->tokens < 32 ? 128 : 64, 32).ranges;   // fewer tokens: only what rdb_few.hip leaves
}
static int t_room(const rdb_linear_desc *d, int num_cus) { return fg_room(d->tokens, d->k, d->out_f, num_cus, 128, 32).ranges; }
static int dc_room(const rdb_linear_desc *d, int num_cus) { return fg_room(d->out_f, d->k, d->tokens, num_cus, 256, 64).ranges; }

// z's ranges that a workspace is asked for: those that pay, whichever products are on (rdb_set_f32_split).  All that z_room allows is up to twice that
// (2048 x 768, k = 256: 27.3 MB instead of 14.7).
static int z_ranges(const rdb_linear_desc *d, int num_cus)
{
    const int room = z_room(d, num_cus);
    if (room <= 1 || d->tokens < 32) return room;
    auto ranges = [&](bool split) { return fg_plan(d->tokens, d->k, d->in_f, num_cus, room, FgGroups<FG_KCONT, FG_NOISE_M>::four, 0.0, split).ranges; };
    return std::max(ranges(true), ranges(false));
}
static int64_t with_parts(const rdb_linear_desc *d, int ranges) { return up256(d->tokens * d->k * 4) * (ranges > 1 ? 1 + ranges : 1); }

// scratch: z or t [tokens x k] and its partial matrices; for the coefficient gradient also one [out_f x k] matrix per token range
int64_t linear_f32_workspace(int op, const rdb_linear_desc *d, int num_cus)
{
    rdb_linear_desc dd = *d;
    if (op == RDB_OP_LINEAR_BWD_DCOEF) dd.coef_dtype = dd.act_dtype;   // reads no coefficients
    if (!fg_ok(&dd)) return 0;
    if (op == RDB_OP_LINEAR_FWD) return with_parts(d, z_ranges(d, num_cus));
    if (op == RDB_OP_LINEAR_BWD_DX) return with_parts(d, t_room(d, num_cus));
    if (op != RDB_OP_LINEAR_BWD_DCOEF) return 0;
    const int r = dc_room(d, num_cus);
    // ... and, for the gradient of the random bias's scale, one value per 64 x 128 tile of [tokens x out_f]
    return with_parts(d, z_ranges(d, num_cus)) + (r > 1 ? (int64_t)r * up256(d->out_f * d->k * 4) : 0) + up256(cdiv(d->tokens, 64) * cdiv(d->out_f, FG_BN) * 4);
}

// The forward pass runs with room for ranges of 128 values and more, in as many as there is room for: shorter ones may pay, and are not needed.
int64_t linear_f32_fwd_workspace_least(const rdb_linear_desc *d, int num_cus)
{
    if (!fg_ok(d)) return 0;
    return with_parts(d, std::min(z_ranges(d, num_cus), fg_room(d->tokens, d->k, d->in_f, num_cus, 128, 32).ranges));
}

static bool fg_ws_ok(int op, const rdb_linear_desc *d, int num_cus, const void *ws, int64_t bytes)
{
    return ws && fg_aligned16(ws) && bytes >= linear_f32_workspace(op, d, num_cus);
}

// A product whose dense output [M x N] (ldo = N) may be computed in up to `room` ranges of the contraction: the ranges' partial
// matrices go to `part` (stride floats apart) and are added up into q.out in range order.
template <int ASRC, int BSRC>
static int fg_launch_ranges(FgProduct q, int room, float *part, int64_t stride, int num_cus, hipStream_t s, const char *name, double host_us = 0.0)
{
    const FgPlan plan = fg_plan(q.M, q.N, q.K, num_cus, room, FgGroups<ASRC, BSRC>::four, host_us);
    q.bm = plan.bm;
    q.groups = plan.groups;
    q.kchunk = 0;
    q.split_stride = 0;
    float *const out = q.out;
    const float *const bias = q.bias;   // fp32, as out is then
    const int out_bf16 = q.out_bf16;
    const int64_t n = q.M * q.N;
    if (plan.ranges <= 1) {
        if (int rc = fg_launch<ASRC, BSRC>(q, num_cus, s, name)) return rc;
        // the kernels that read a matrix across its rows are not built with a bias: it is added in place
        return FgGroups<ASRC, BSRC>::biased ? RDB_OK : fg_launch_sums(fg_sum(out, out_bf16, out, n, 0, 1, bias, q.N), FgSum{}, s);
    }
    q.out = part;
    q.out_bf16 = 0;
    q.kchunk = cdiv(cdiv(q.K, plan.ranges), FG_BK) * FG_BK;   // every range holds something (fg_plan)
    q.split_stride = stride;
    q.bias = nullptr;
    if (int rc = fg_launch<ASRC, BSRC>(q, num_cus, s, name)) return rc;
    return fg_launch_sums(fg_sum(out, out_bf16, part, n, stride, plan.ranges, bias, q.N), FgSum{}, s);
}

// Two such products that do not need each other, in one launch, and their sums in one: t = dy . C and dC = dy^T . z.
int fg_launch_pair(const FgProduct &t, const FgProduct &dc, hipStream_t s);   // rdb_f32_pair.hip
// dc_sum: dC's sum where it is left to the launch that comes next, dx = t . N: where t's ranges are one, so that no launch of sums is left, or that product's tiles leave compute
// units free and dC's partial matrices are long, 8 MB.  2048 tokens x 768 -> 3072, k = 256, 192 tiles, 16 MB: sums 7.6 -> 4.8 us, dx 12.5 -> 13.2, step 98.3 -> 96.1; 512 tiles, 4096 x
// 1024 -> 8192, k = 128: sums 8.1 -> 5.3, dx 17.4 -> 20.0, step 208.6 -> 210.7; 256 tiles, 1024 x 4096 -> 4096, k = 256: 106.6 -> 108.0; 6 MB, 4097 x 1001 -> 999, k = 100 in bf16: sums 4.5 ->
// 4.2, dx 15.6 -> 16.7.
static int fg_launch_pair_ranges(FgProduct t, int t_room, float *t_part, int64_t t_stride, FgProduct dc, int dc_room, float *dc_part, int64_t dc_stride,
                                 int num_cus, hipStream_t s, const rdb_linear_desc *d, FgSum &dc_sum)
{
    const FgPairPlan plan = fg_plan_pair({t.M, dc.M}, {t.N, dc.N}, {t.K, dc.K}, num_cus, {t_room, dc_room}, t.a_es == 2);
    FgProduct *const q[2] = {&t, &dc};
    float *const part[2] = {t_part, dc_part};
    const int64_t stride[2] = {t_stride, dc_stride};
    FgSum sum[2];
    for (int i = 0; i < 2; ++i) {
        FgProduct &p = *q[i];
        const int r = plan.ranges[i];
        p.bm = plan.bm;
        p.groups = plan.groups;
        p.kchunk = fg_chunk(p.K, r);
        sum[i] = fg_sum(p.out, p.out_bf16, part[i], p.M * p.N, stride[i], r);
        if (r > 1) {
            p.out = part[i];
            p.out_bf16 = 0;
            p.split_stride = stride[i];
        }
    }
    if (int rc = fg_launch_pair(t, dc, s)) return rc;
    bool beside = !sum[0].blocks;
    if (!beside && sum[1].n * sum[1].splits * 4 >= (8 << 20)) {
        const FgPlan dx = fg_plan(d->tokens, d->in_f, d->k, num_cus, 1, FgGroups<FG_KCONT, FG_NOISE_I>::four);
        beside = cdiv(d->tokens, dx.bm) * cdiv(d->in_f, FG_BN) < num_cus;
    }
    dc_sum = beside ? sum[1] : FgSum{};
    return fg_launch_sums(sum[0], beside ? FgSum{} : sum[1], s);
}

// What z's launch of sums counts for on the host in a training step, which has 60 to 70 us of host work (a forward pass alone has 10, and its kernels are what
// it waits for: 4700 tokens x 496 -> 32, k = 16 16.2 us a pass, 20.6 with z in one range): nothing where the step's products, z, y, t, dC and dx at 1.16 PFLOP/s, take 40 us and more (with as much
// again for what they wait, the kernels then outlast the host's 60 to 70: 2859 tokens x 584 -> 7920, k = 208, step 219 us, 222 with z in one range).  Both sides, us a step in six
// processes each, weighed and not: 207 x 392 -> 1440, k = 56 65.4 to 67.9, 68.1 to 72.5; 181 x 410 -> 3589, k = 293 in bf16 95 to 104, 99 to 104; 1024 x 1024 ->
// 1024, k = 128 68 to 71 either way.  A process whose host takes 40 a step, one of the twelve, waits for kernels that are 2 to 5 longer instead.
static double z_host_us(const rdb_linear_desc *d)
{
    const double parts = d->act_dtype == RDB_BF16 ? 3.0 : 6.0;   // bf16 products per product
    return parts * 2.0 * d->tokens * d->k * (2.0 * d->in_f + 3.0 * d->out_f) / 1.16e9 < 40.0 ? FG_HOST_US : 0.0;
}
// z[T x k] = src[T x in_f] . N^T; the partial matrices of its ranges go to `part` (room for max_ranges of them, up256(T k 4)
// bytes apart; NULL: right behind z, as many as there is room for)
static int fg_project(float *z, const float *x, int64_t ldx, const rdb_linear_desc *d, int num_cus, hipStream_t s, float *part = nullptr,
                      int max_ranges = 1 << 30, double host_us = 0.0, const FgValues &values = {})
{
    FgProduct q = {x, ldx, (d->tokens - 1) * ldx + d->in_f, nullptr, 0, 0, z, d->k, nullptr, d->tokens, d->k, d->in_f, 0, 0, 0, 0, d->seed};
    q.a_es = fg_es(d->act_dtype);
    q.values = values;
    const int64_t zt = up256(d->tokens * d->k * 4) / 4;
    return fg_launch_ranges<FG_KCONT, FG_NOISE_M>(q, std::max(1, std::min(z_room(d, num_cus), max_ranges)), part ? part : z + zt, zt, num_cus, s,
                                                  "f32_gemm_kernel (z = x . N^T)", host_us);
}

// Where the forward pass puts the partial matrices of z's ranges: into y, which is written last, or, where y holds less than a third of those that pay, into
// scratch of the call's own (32 MB at most: ranges times tiles are at most two to a compute unit, a tile 64 KB), no part of what is kept.  With the ranges that y holds instead,
// z of 492 tokens x 3184 -> 273, k = 118 in bf16, one range: 80 us, now 12.1 and 4 for the sums; 300 x 4000 -> 301, k = 100: 99, 9.2; 700 x 4000 -> 256, k =
// 120 in fp32: 63, 13.9.  Where it holds more, scratch is not asked for the 3 to 5 us
// that are left (433 x 3320 -> 1288, k = 144: 18.3, 15.0; 128 x 784 -> 256, k = 64: four ranges, nine would pay).
static int64_t z_scratch(const rdb_linear_desc *d)
{
    const int num_cus = num_compute_units();
    const int64_t zt = up256(d->tokens * d->k * 4), in_y = std::max<int64_t>(1, d->tokens * d->out_f * fg_es(d->act_dtype) / zt);
    const int most = z_room(d, num_cus);
    if (most < 3 * in_y) return 0;
    // by the layer alone, whatever products are asked for (rdb_set_f32_split): it may be larger than they need, never smaller
    const int want = fg_plan(d->tokens, d->k, d->in_f, num_cus, std::max(1, most), FgGroups<FG_KCONT, FG_NOISE_M>::four, z_host_us(d), true).ranges;
    return want >= 3 * in_y ? want * zt : 0;
}
// z into `z`, y (or NULL) to come; scratch: NULL, or scratch_bytes (less than z_scratch, or not aligned: y's room, as without)
static int fg_project_kept(float *z, const void *x, int64_t ldx, void *y, int64_t ldy, const rdb_linear_desc *d, int num_cus, void *scratch, int64_t scratch_bytes,
                           hipStream_t s, const FgValues &values)
{
    const int64_t zt = up256(d->tokens * d->k * 4), asked = scratch && fg_aligned16(scratch) ? z_scratch(d) : 0;
    float *part = z;
    int64_t room = 0;
    if (asked > 0 && scratch_bytes >= asked) part = static_cast<float *>(scratch), room = asked;
    else if (y && ldy == d->out_f && fg_aligned16(y)) part = static_cast<float *>(y), room = d->tokens * d->out_f * fg_es(d->act_dtype);
    return fg_project(z, static_cast<const float *>(x), ldx, d, num_cus, s, part, (int)std::min<int64_t>(32, room / zt), z_host_us(d), values);
}

// The three entry points return RDB_E_UNSUPPORTED, without setting an error, when the request does not fit.
int linear_fwd_f32(void *y, int64_t ldy, const void *x, int64_t ldx, const void *coef, const void *scale_bias, const void *bias,
                   const rdb_linear_desc *d, int num_cus, void *workspace, int64_t workspace_bytes, hipStream_t s)
{
    if (!fg_ok(d) || !fg_wanted(d) || !workspace || !fg_aligned16(workspace) || workspace_bytes < linear_f32_fwd_workspace_least(d, num_cus)) return RDB_E_UNSUPPORTED;
    if (d->tokens * ldx >= (1ll << 29) || d->tokens * ldy >= (1ll << 29)) return RDB_E_UNSUPPORTED;
    float *z = (float *)workspace;
    const int64_t parts = workspace_bytes / up256(d->tokens * d->k * 4) - 1;
    if (int rc = fg_project(z, (const float *)x, ldx, d, num_cus, s, nullptr, (int)std::min<int64_t>(parts, z_ranges(d, num_cus)))) return rc;
    FgProduct q = {z, d->k, d->tokens * d->k, (const float *)coef, d->k, d->out_f * d->k, (float *)y, ldy, (const float *)bias,
                   d->tokens, d->out_f, d->k, 0, 0, 0, 0, d->seed};
    const int b16 = d->act_dtype == RDB_BF16;
    q.b_es = fg_es(d->coef_dtype);
    q.out_bf16 = b16;
    if (int rc = fg_launch<FG_KCONT, FG_KCONT>(q, num_cus, s, "f32_gemm_kernel (y = z . C^T)")) return rc;
    if (!scale_bias) return RDB_OK;
    // y += s * x . R^T: the B side's rows are output features, index o * in_f + i
    FgProduct qr = {(const float *)x, ldx, (d->tokens - 1) * ldx + d->in_f, nullptr, 0, 0, (float *)y, ldy, nullptr, d->tokens, d->out_f, d->in_f,
                    0, 0, 0, 0, d->seed, (uint32_t)d->in_f, 1u, (const float *)scale_bias,
                    nullptr, 0, nullptr};
    qr.a_es = fg_es(d->act_dtype);
    qr.out_bf16 = b16;
    qr.scale_bf16 = d->coef_dtype == RDB_BF16;
    return fg_launch<FG_KCONT, FG_NOISE_1D>(qr, num_cus, s, "f32_gemm_kernel (y += s x . R^T)");
}

// t[T x k] = dy[T x out_f] . C: the B side's rows are coefficients, read across the rows of C
static FgProduct fg_t(float *t, const void *dy, int64_t lddy, const void *coef, const rdb_linear_desc *d)
{
    FgProduct q = {(const float *)dy, lddy, (d->tokens - 1) * lddy + d->out_f, (const float *)coef, d->k, d->out_f * d->k, t, d->k, nullptr,
                   d->tokens, d->k, d->out_f, 0, 0, 0, 0, d->seed};
    q.a_es = fg_es(d->act_dtype);
    q.b_es = fg_es(d->coef_dtype);
    return q;
}
// dx[T x in_f] = t . N: the B side's rows are input features, hashed
// sum, bias: what is still to be done, beside the product
static int fg_dx_from_t(void *dx, int64_t lddx, const float *t, const rdb_linear_desc *d, int num_cus, hipStream_t s, const FgSum &sum = {}, const BiasGrad &bias = {})
{
    FgProduct q = {t, d->k, d->tokens * d->k, nullptr, 0, 0, (float *)dx, lddx, nullptr, d->tokens, d->in_f, d->k, 0, 0, 0, 0, d->seed};
    q.out_bf16 = d->act_dtype == RDB_BF16;
    q.sum = sum;
    if (sum.blocks) q.split = true;   // as it was when the sum was left
    q.bias_grad = bias;
    return fg_launch<FG_KCONT, FG_NOISE_I>(q, num_cus, s, "f32_gemm_kernel (dx = t . N)");
}
// dC[out_f x k] = dy^T . z: both sides are read across their rows (the contraction runs over the tokens)
static FgProduct fg_dc(void *dcoef, int dcoef_dtype, const void *dy, int64_t lddy, const float *z, const rdb_linear_desc *d)
{
    FgProduct q = {(const float *)dy, lddy, (d->tokens - 1) * lddy + d->out_f, z, d->k, d->tokens * d->k, (float *)dcoef, d->k, nullptr,
                   d->out_f, d->k, d->tokens, 0, 0, 0, 0, d->seed};
    q.a_es = fg_es(d->act_dtype);
    q.out_bf16 = dcoef_dtype == RDB_BF16;
    return q;
}
int linear_dx_f32(void *dx, int64_t lddx, const void *dy, int64_t lddy, const void *coef, const void *scale_bias, const rdb_linear_desc *d,
                  int num_cus, void *workspace, int64_t workspace_bytes, hipStream_t s);
// dx and / or dC (each NULL where it is not wanted) from dy, z and C; dc_part: room for dC's partial matrices; bias: a gradient from dy that the last launch carries
static int fg_backward(void *dx, int64_t lddx, void *dcoef, int dcoef_dtype, const void *dy, int64_t lddy, const float *z, const void *coef,
                       const rdb_linear_desc *d, int num_cus, void *workspace, int64_t workspace_bytes, float *dc_part, hipStream_t s, const BiasGrad &bias = {})
{
    const int room = dc_room(d, num_cus);
    const int64_t dc_stride = up256(d->out_f * d->k * 4) / 4;
    if (dx && dcoef && f32_split_mode()) {
        float *t = (float *)workspace;
        const int64_t zt = up256(d->tokens * d->k * 4) / 4;
        FgSum dc_sum;
        if (int rc = fg_launch_pair_ranges(fg_t(t, dy, lddy, coef, d), t_room(d, num_cus), t + zt, zt, fg_dc(dcoef, dcoef_dtype, dy, lddy, z, d),
                                           room, dc_part, dc_stride, num_cus, s, d, dc_sum))
            return rc;
        return fg_dx_from_t(dx, lddx, t, d, num_cus, s, dc_sum, bias);
    }
    if (dx) {
        if (int rc = linear_dx_f32(dx, lddx, dy, lddy, coef, nullptr, d, num_cus, workspace, workspace_bytes, s)) return rc;
    }
    if (!dcoef) return bias.blocks ? bias_direct_launch(bias, s) : RDB_OK;
    FgProduct dc = fg_dc(dcoef, dcoef_dtype, dy, lddy, z, d);
    dc.bias_grad = bias;
    return fg_launch_ranges<FG_MCONT, FG_MCONT>(dc, room, dc_part, dc_stride, num_cus, s, "f32_gemm_kernel (dC = dy^T . z)");
}

int linear_dx_f32(void *dx, int64_t lddx, const void *dy, int64_t lddy, const void *coef, const void *scale_bias, const rdb_linear_desc *d,
                  int num_cus, void *workspace, int64_t workspace_bytes, hipStream_t s)
{
    if (!fg_ok(d) || !fg_wanted(d) || !fg_ws_ok(RDB_OP_LINEAR_BWD_DX, d, num_cus, workspace, workspace_bytes)) return RDB_E_UNSUPPORTED;
    if (d->tokens * lddx >= (1ll << 29) || d->tokens * lddy >= (1ll << 29)) return RDB_E_UNSUPPORTED;
    float *t = (float *)workspace;
    const int b16 = d->act_dtype == RDB_BF16;
    const int64_t zt = up256(d->tokens * d->k * 4) / 4;
    if (int rc = fg_launch_ranges<FG_KCONT, FG_MCONT>(fg_t(t, dy, lddy, coef, d), t_room(d, num_cus), t + zt, zt, num_cus, s, "f32_gemm_kernel (t = dy . C)"))
        return rc;
    if (int rc = fg_dx_from_t(dx, lddx, t, d, num_cus, s)) return rc;
    if (!scale_bias) return RDB_OK;
    // dx += s * dy . R: the B side's rows are input features, index o * in_f + i
    FgProduct qr = {(const float *)dy, lddy, (d->tokens - 1) * lddy + d->out_f, nullptr, 0, 0, (float *)dx, lddx, nullptr, d->tokens, d->in_f, d->out_f,
                    0, 0, 0, 0, d->seed, 1u, (uint32_t)d->in_f, (const float *)scale_bias,
                    nullptr, 0, nullptr};
    qr.a_es = fg_es(d->act_dtype);
    qr.out_bf16 = b16;
    qr.scale_bf16 = d->coef_dtype == RDB_BF16;
    return fg_launch<FG_KCONT, FG_NOISE_1D>(qr, num_cus, s, "f32_gemm_kernel (dx += s dy . R)");
}

// dcoef is overwritten (no zero fill needed).
// d_scale_bias: NULL, or where the gradient of the random bias's scale goes: <dy, x . R^T>.
int linear_dcoef_f32(float *dcoef, float *d_scale_bias, const void *dy, int64_t lddy, const void *x, int64_t ldx, const rdb_linear_desc *d, int num_cus,
                     void *workspace, int64_t workspace_bytes, hipStream_t s)
{
    rdb_linear_desc dd = *d;
    dd.coef_dtype = dd.act_dtype;   // no coefficients are read here
    if (!fg_ok(&dd) || !fg_wanted(&dd) || !fg_ws_ok(RDB_OP_LINEAR_BWD_DCOEF, &dd, num_cus, workspace, workspace_bytes)) return RDB_E_UNSUPPORTED;
    if (d->tokens * ldx >= (1ll << 29) || d->tokens * lddy >= (1ll << 29)) return RDB_E_UNSUPPORTED;
    float *z = (float *)workspace;
    const int zs = z_ranges(&dd, num_cus);
    if (int rc = fg_project(z, (const float *)x, ldx, &dd, num_cus, s, nullptr, zs)) return rc;
    float *part = reinterpret_cast<float *>(static_cast<char *>(workspace) + up256(d->tokens * d->k * 4) * (zs > 1 ? 1 + zs : 1));
    const int dcr = dc_room(&dd, num_cus);
    if (int rc = fg_launch_ranges<FG_MCONT, FG_MCONT>(fg_dc(dcoef, RDB_F32, dy, lddy, z, &dd), dcr, part, up256(d->out_f * d->k * 4) / 4, num_cus, s, "f32_gemm_kernel (dC = dy^T . z)")) return rc;
    if (!d_scale_bias) return RDB_OK;
    // <dy, x . R^T>: the random-bias product once more, each block reducing its tile against dy's; then the blocks in order
    float *dots = part + (dcr > 1 ? (int64_t)dcr * (up256(d->out_f * d->k * 4) / 4) : 0);
    FgProduct qr = {(const float *)x, ldx, (d->tokens - 1) * ldx + d->in_f, nullptr, 0, 0, nullptr, 0, nullptr, d->tokens, d->out_f, d->in_f,
                    fg_room(d->tokens, d->out_f, d->in_f, num_cus, d->in_f, 1).bm, 1, 0, 0, d->seed, (uint32_t)d->in_f, 1u, nullptr,
                    (const float *)dy, lddy, dots};
    qr.a_es = fg_es(d->act_dtype);
    qr.out_bf16 = d->act_dtype == RDB_BF16;   // dy, the matrix the product is reduced against
    if (int rc = fg_launch<FG_KCONT, FG_NOISE_1D>(qr, num_cus, s, "f32_gemm_kernel (<dy, x . R^T>)")) return rc;
    const int nblocks = (int)(cdiv(d->tokens, qr.bm) * cdiv(d->out_f, FG_BN));
    f32_sum_scalars_kernel<<<1, 256, 0, s>>>(d_scale_bias, dots, nblocks);
    return check_launch("f32_sum_scalars_kernel");
}

// ----------------------------------------------------------------------------------------------- or the few-token kernels
// fp32 with k <= 64: where the kernels above are ahead of the vector-ALU kernels of rdb_smallk.hip.  Microseconds of one direction
// (contraction over J, expansion to E columns), fitted to 252 measured calls (k 16, 32, 64; 32 to 1024 tokens; 128 -> 256 to
// 4096 -> 11008): what it picks is 0.2 us behind the faster of the two on average.  The vector-ALU kernels' hash costs a wave 0.2 us a
// coefficient whatever the tokens (0.16 since they fetch all their coefficients at once: up to 3 us less at k = 64 than the model
// says, so a call near the line may now be 2 us behind), and their time grows with the products; the matrix cores' grows with
// the contraction a block walks through alone.  1024 tokens x 4096 -> 11008, k = 64: forward 134 -> 41 us, dx 93 -> 45; 128 tokens x 784 -> 256,
// k = 64: 20.4 -> 18.8, 20.8 -> 15.8; k = 16 stays (10.5 against 16.2).
static double few_token_us(const rdb_linear_desc *d)
{
    return 7.0 + 0.21 * d->k + (double)d->tokens * (d->in_f + d->out_f) * (1.7e-6 + 0.9e-7 * d->k);
}
static double f32_products_us(const rdb_linear_desc *d, bool dx)
{
    const int64_t J = dx ? d->out_f : d->in_f, E = dx ? d->in_f : d->out_f;
    return (dx ? 11.7 : 11.0) + 0.0034 * std::min<int64_t>(J, 5200) + 0.04 * d->k + 0.5e-6 * d->tokens * E;
}
bool f32_products_first(const rdb_linear_desc *d, bool dx)
{
    return d->algo == RDB_ALGO_AUTO && d->act_dtype == RDB_F32 && d->coef_dtype == RDB_F32 && d->k <= 64 && d->tokens >= 32 &&
           f32_products_us(d, dx) < few_token_us(d);
}

// ----------------------------------------------------------------------------------------------- z kept from forward to backward
// For the layers that have no projection state of their own (bf16 with sizes that are not multiples of 8, fp32 in the few-token
// regime): the forward pass leaves z = x . N^T, [tokens x k] in fp32, and the backward pass takes it from there instead of
// projecting x again.  Only while that is at most twice the size of x, which the caller keeps too.  Few tokens (in bf16 up to 96,
// in fp32 below 32 and where the vector-ALU kernels' three calls take less: their coefficient gradient projects x again, 5 us more
// than their forward pass, against 10 here) stay with the kernels of rdb_smallk.hip.  4097 tokens x 1001 -> 999, k = 100 in bf16, forward and backward:
// 122 -> 98 us; 128 tokens x 784 -> 256, k = 64 in fp32: 22.7 + 11.1 + 27.8 us of few-token kernels -> 17 + 6.
int64_t linear_kept_f32_bytes(const rdb_linear_desc *d)
{
    if (!fg_ok(d) || d->algo != RDB_ALGO_AUTO || d->tokens * std::max(d->in_f, d->out_f) >= (1ll << 28) || d->sO != d->in_f || d->sI != 1) return 0;
    const bool b16 = d->act_dtype == RDB_BF16;
    if (b16 ? (d->tokens <= 96 || !(d->in_f % 8 || d->out_f % 8 || d->k % 8) || d->k > d->in_f) : (d->tokens < 32 || d->k > 2 * d->in_f)) return 0;
    if (!b16 && d->k <= 64 && f32_products_us(d, false) + f32_products_us(d, true) + 10.0 > 3.0 * few_token_us(d) + 5.0) return 0;
    return up256(d->tokens * d->k * 4);
}
int64_t linear_kept_f32_scratch(const rdb_linear_desc *d) { return linear_kept_f32_bytes(d) ? z_scratch(d) : 0; }

static int fg_rbias(FgProduct q, const void *scale, const rdb_linear_desc *d, int num_cus, hipStream_t s, const char *name)
{
    q.a_es = fg_es(d->act_dtype);
    q.out_bf16 = d->act_dtype == RDB_BF16;
    q.scale = static_cast<const float *>(scale);
    q.scale_bf16 = d->coef_dtype == RDB_BF16;
    return fg_launch<FG_KCONT, FG_NOISE_1D>(q, num_cus, s, name);
}

// values: NULL, or a pseudorandom bias whose values the launch of the projection forms on the side, or one of their own (an fp32 layer's; then `bias`)
int linear_fwd_kept_f32(void *y, int64_t ldy, void *kept, const void *x, int64_t ldx, const void *coef, const void *scale_bias, const void *bias,
                        const rdb_pseudo_bias *values, const rdb_linear_desc *d, int num_cus, void *scratch, int64_t scratch_bytes, hipStream_t s)
{
    if (!linear_kept_f32_bytes(d) || !fg_aligned16(kept) || d->tokens * ldx >= (1ll << 29) || d->tokens * ldy >= (1ll << 29)) return RDB_E_UNSUPPORTED;
    FgValues v = {};
    if (values) {
        bias = values->values;
        if (values->k <= FG_VALUES_K && d->out_f <= FG_VALUES_N)
            v = {values->values, values->coef, values->scale, (int)d->out_f, (int)values->k, values->seed, 0};
        else if (int rc = rdb_materialize_fwd(values->values, values->coef, RDB_F32, 0, values->k, 0, 1, d->out_f, 0, 1, values->seed, values->scale, (void *)s))
            return rc;
    }
    float *z = static_cast<float *>(kept);
    if (int rc = fg_project_kept(z, x, ldx, y, ldy, d, num_cus, scratch, scratch_bytes, s, v)) return rc;
    FgProduct q = {z, d->k, d->tokens * d->k, (const float *)coef, d->k, d->out_f * d->k, (float *)y, ldy, (const float *)bias, d->tokens, d->out_f, d->k,
                   0, 0, 0, 0, d->seed};
    q.b_es = fg_es(d->coef_dtype);
    q.out_bf16 = d->act_dtype == RDB_BF16;
    if (int rc = fg_launch<FG_KCONT, FG_KCONT>(q, num_cus, s, "f32_gemm_kernel (y = z . C^T)")) return rc;
    if (!scale_bias) return RDB_OK;
    FgProduct qr = {(const float *)x, ldx, (d->tokens - 1) * ldx + d->in_f, nullptr, 0, 0, (float *)y, ldy, nullptr, d->tokens, d->out_f, d->in_f,
                    0, 0, 0, 0, d->seed, (uint32_t)d->in_f, 1u};
    return fg_rbias(qr, scale_bias, d, num_cus, s, "f32_gemm_kernel (y += s x . R^T)");
}

// t = dy . C and its partial matrices, those of dC = dy^T . z, and one value per tile of dy . R (at most 64 x 128 of [tokens x in_f] or
// [tokens x out_f])
int64_t linear_bwd_kept_f32_workspace(const rdb_linear_desc *d, int num_cus)
{
    if (!linear_kept_f32_bytes(d)) return 0;
    const int r = dc_room(d, num_cus);
    return linear_f32_workspace(RDB_OP_LINEAR_BWD_DX, d, num_cus) + (r > 1 ? (int64_t)r * up256(d->out_f * d->k * 4) : 0) +
           up256(cdiv(d->tokens, 64) * cdiv(std::max(d->in_f, d->out_f), FG_BN) * 4);
}

// dx += s * (the ranges' sums of dy . R, [rows x cols] each, `stride` floats apart, added in range order), all in bf16 but the sums; dots: NULL, or a
// value per block, its share of their product with x.  One element a thread and turn: rows are of any length.
__global__ __launch_bounds__(256) void f32_rbias_sum_kernel(bf16_t *__restrict__ dx, int64_t lddx, const float *__restrict__ part, int64_t stride, int ranges,
                                                            const bf16_t *__restrict__ scale, const bf16_t *__restrict__ x, int64_t ldx, float *__restrict__ dots,
                                                            uint32_t n, uint32_t cols)
{
    const float s = bf16_to_f32(*scale);
    float dot = 0.0f;
    for (uint32_t e = blockIdx.x * 256u + threadIdx.x; e < n; e += gridDim.x * 256u) {
        const uint32_t row = e / cols, col = e - row * cols;
        bf16_t *const to = dx + row * lddx + col;
        const float old = bf16_to_f32(*to), other = dots ? bf16_to_f32(x[row * ldx + col]) : 0.0f;
        float v = part[e];
        for (int r0 = 1; r0 < ranges; r0 += 4) {   // four ranges' loads in flight
            float u[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) u[j] = part[min(r0 + j, ranges - 1) * stride + e];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (r0 + j < ranges) v += u[j];
        }
        dot = fmaf(v, other, dot);
        *to = f32_to_bf16(fmaf(s, v, old));
    }
    if (!dots) return;
    __shared__ float wsum[4];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) dot += __shfl_xor(dot, o, 64);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = dot;
    __syncthreads();
    if (threadIdx.x == 0) dots[blockIdx.x] = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
}

// dx, dcoef (fp32 or bf16) and d_scale_bias: each NULL where it is not wanted.  With dx wanted, the gradient of the scale, <dy . R, x>,
// comes out of the random-bias product that dx needs anyway.
int linear_bwd_kept_f32(void *dx, int64_t lddx, void *dcoef, int dcoef_dtype, float *d_scale_bias, const void *dy, int64_t lddy, const void *x, int64_t ldx,
                        const void *kept, const void *coef, const void *scale_bias, const rdb_linear_desc *d, int num_cus, void *workspace,
                        int64_t workspace_bytes, hipStream_t s, const BiasGrad &bias)
{
    if (!linear_kept_f32_bytes(d) || !fg_aligned16(kept) || !workspace || !fg_aligned16(workspace) ||
        workspace_bytes < linear_bwd_kept_f32_workspace(d, num_cus) || d->tokens * lddy >= (1ll << 29) || (dx && d->tokens * lddx >= (1ll << 29)) ||
        (d_scale_bias && d->tokens * ldx >= (1ll << 29)))
        return RDB_E_UNSUPPORTED;
    char *const dc_part = static_cast<char *>(workspace) + linear_f32_workspace(RDB_OP_LINEAR_BWD_DX, d, num_cus);
    const int r = dc_room(d, num_cus);
    float *const dots = reinterpret_cast<float *>(dc_part + (r > 1 ? (int64_t)r * up256(d->out_f * d->k * 4) : 0));
    if (int rc = fg_backward(dx, lddx, dcoef, dcoef_dtype, dy, lddy, static_cast<const float *>(kept), coef, d, num_cus, workspace, workspace_bytes,
                             reinterpret_cast<float *>(dc_part), s, bias))
        return rc;
    if (!scale_bias || (!dx && !d_scale_bias)) return RDB_OK;
    FgProduct q;
    if (dx) {   // dx += s * dy . R, and <dy . R, x> on the way
        q = {(const float *)dy, lddy, (d->tokens - 1) * lddy + d->out_f, nullptr, 0, 0, (float *)dx, lddx, nullptr, d->tokens, d->in_f, d->out_f,
             0, 0, 0, 0, d->seed, 1u, (uint32_t)d->in_f};
        if (d_scale_bias) q.dotm = (const float *)x, q.lddot = ldx;
    } else {    // <x . R^T, dy>
        q = {(const float *)x, ldx, (d->tokens - 1) * ldx + d->in_f, nullptr, 0, 0, nullptr, 0, nullptr, d->tokens, d->out_f, d->in_f,
             0, 0, 0, 0, d->seed, (uint32_t)d->in_f, 1u};
        q.dotm = (const float *)dy, q.lddot = lddy;
    }
    // dx of bf16 layers (the kernel that adds the ranges up takes bf16 rows; fp32 layers and the forward share have not been tried in ranges) in as many ranges of the output features as pay and as the workspace, whose t and partial matrices are used up, holds: few
    // tokens are a handful of tiles otherwise, each with all of out_f to hash, split and multiply (us, with the sums: 502 x 527 -> 2918, k = 251: 87 -> 28;
    // 942 x 729 -> 6529, k = 92: 179 -> 59; 1346 x 289 -> 5636, k = 48: 143 -> 38; 1494 x 2739 -> 8065, k = 105: 667 -> 396)
    const int64_t stride = up256(q.M * q.N * 4) / 4, room = (reinterpret_cast<char *>(dots) - static_cast<char *>(workspace)) / (stride * 4);
    const FgPlan rp = fg_plan(q.M, q.N, q.K, num_cus, dx && d->act_dtype == RDB_BF16 ? (int)std::max<int64_t>(1, std::min<int64_t>(room, 32)) : 1, true, FG_HOST_US);
    if (rp.ranges > 1) {
        FgProduct p = q;
        p.a_es = fg_es(d->act_dtype);
        p.bm = rp.bm;
        p.groups = rp.groups;
        p.out = static_cast<float *>(workspace);
        p.ldo = q.N;
        p.kchunk = fg_chunk(q.K, rp.ranges);
        p.split_stride = stride;
        p.dotm = nullptr;
        if (int rc = fg_launch<FG_KCONT, FG_NOISE_1D>(p, num_cus, s, "f32_gemm_kernel (dy . R in ranges)")) return rc;
        const int blocks = (int)std::min<int64_t>(cdiv(d->tokens, 64) * cdiv(std::max(d->in_f, d->out_f), FG_BN), cdiv(q.M * q.N, 256));   // of room for dots
        f32_rbias_sum_kernel<<<blocks, 256, 0, s>>>(static_cast<bf16_t *>(dx), lddx, p.out, stride, rp.ranges, static_cast<const bf16_t *>(scale_bias),
                                                    static_cast<const bf16_t *>(x), ldx, d_scale_bias ? dots : nullptr, (uint32_t)(q.M * q.N), (uint32_t)q.N);
        if (int rc = check_launch("f32_rbias_sum_kernel")) return rc;
        if (!d_scale_bias) return RDB_OK;
        f32_sum_scalars_kernel<<<1, 256, 0, s>>>(d_scale_bias, dots, blocks);
        return check_launch("f32_sum_scalars_kernel");
    }
    const FgPlan pl = fg_plan(q.M, q.N, q.K, num_cus, 1, true);
    q.bm = pl.bm;
    q.groups = pl.groups;
    q.dot_part = d_scale_bias ? dots : nullptr;
    if (int rc = fg_rbias(q, dx ? scale_bias : nullptr, d, num_cus, s, "f32_gemm_kernel (dx += s dy . R)")) return rc;
    if (!d_scale_bias) return RDB_OK;
    f32_sum_scalars_kernel<<<1, 256, 0, s>>>(d_scale_bias, dots, (int)(cdiv(q.M, q.bm) * cdiv(q.N, FG_BN)));
    return check_launch("f32_sum_scalars_kernel");
}

// ----------------------------------------------------------------------------------------------- dW = dy^T . x on its own
// For the vector-coef coefficient gradient: every element of dW meets k hashed values, so that gradient is bound by the hash
// whatever is fused into it, and a kernel that forms dW tile by tile per block of tokens repeats the k hashes per element for
// every block.  With room for dW (fp32, [out_f x in_f]) in the caller's workspace it is formed once, by this product, and
// contracted once by the kernels of rdb_materialize_bwd.  Scratch behind dW: one more [out_f x in_f] matrix per token range.
static int dw_room(const rdb_linear_desc *d, int num_cus) { return fg_room(d->out_f, d->in_f, d->tokens, num_cus, 256, 64).ranges; }
int64_t linear_dw_f32_workspace(const rdb_linear_desc *d, int num_cus)
{
    if (d->out_f * d->in_f >= (1ll << 29) || d->tokens <= 0) return 0;
    const int r = dw_room(d, num_cus);
    return up256(d->out_f * d->in_f * 4) * (1 + (r > 1 ? r : 0));
}
int linear_dw_f32(float *dW, const void *dy, int64_t lddy, const void *x, int64_t ldx, const rdb_linear_desc *d, int num_cus, hipStream_t s)
{
    if (d->tokens * lddy >= (1ll << 29) || d->tokens * ldx >= (1ll << 29) || d->out_f * d->in_f >= (1ll << 29)) return RDB_E_UNSUPPORTED;
    FgProduct q = {(const float *)dy, lddy, (d->tokens - 1) * lddy + d->out_f, (const float *)x, ldx, (d->tokens - 1) * ldx + d->in_f, dW, d->in_f, nullptr,
                   d->out_f, d->in_f, d->tokens, 0, 0, 0, 0, d->seed};
    q.a_es = q.b_es = fg_es(d->act_dtype);
    const int64_t stride = up256(d->out_f * d->in_f * 4) / 4;
    return fg_launch_ranges<FG_MCONT, FG_MCONT>(q, dw_room(d, num_cus), dW + stride, stride, num_cus, s, "f32_gemm_kernel (dW = dy^T . x)");
}

// ----------------------------------------------------------------------------------------------- projected form in fp32
// What a training step keeps from the forward to the backward pass (all that the latter needs of x): z = x . N^T in fp32, [tokens x k] row-major,
// behind a 256-byte header (the same role as the bf16 state of rdb_direct.hpp; no fragment orders, no transposed copies: these
// kernels stage both operands through LDS).  fp32 activations and coefficients, one launch's worth of tokens.
static bool fg_state_ok(const rdb_linear_desc *d)
{
    return d->act_dtype == RDB_F32 && d->coef_dtype == RDB_F32 && fg_ok(d) && d->tokens * std::max(d->in_f, d->out_f) < (1ll << 28);
}
int64_t linear_f32_state_bytes(const rdb_linear_desc *d) { return fg_state_ok(d) ? 256 + up256(d->tokens * d->k * 4) : 0; }
int64_t linear_project_f32_scratch(const rdb_linear_desc *d) { return fg_state_ok(d) ? z_scratch(d) : 0; }
static float *fg_state_z(const void *state) { return reinterpret_cast<float *>(static_cast<char *>(const_cast<void *>(state)) + 256); }

// workspace of the backward pass from the state: t = dy . C with the partial matrices of its ranges, then the partial matrices
// of dC = dy^T . z
int64_t linear_f32_bwd_projected_workspace(const rdb_linear_desc *d, int num_cus)
{
    if (!fg_state_ok(d)) return 0;
    const int r = dc_room(d, num_cus);
    return linear_f32_workspace(RDB_OP_LINEAR_BWD_DX, d, num_cus) + (r > 1 ? (int64_t)r * up256(d->out_f * d->k * 4) : 0);
}

static int fg_fwd_from_z(void *y, int64_t ldy, const float *z, const void *coef, const void *bias, const rdb_linear_desc *d, int num_cus, hipStream_t s)
{
    FgProduct q = {z, d->k, d->tokens * d->k, (const float *)coef, d->k, d->out_f * d->k, (float *)y, ldy, (const float *)bias,
                   d->tokens, d->out_f, d->k, 0, 0, 0, 0, d->seed};
    return fg_launch<FG_KCONT, FG_KCONT>(q, num_cus, s, "f32_gemm_kernel (y = z . C^T)");
}

// state <- z.  The partial matrices of the projection's contraction ranges lie in y's memory, which is written last (only when y is
// contiguous, and as many ranges as fit there; without y the contraction runs in one range), or in scratch where y is too narrow for them.
int linear_project_f32(void *state, void *y, int64_t ldy, const void *x, int64_t ldx, const void *coef, const void *bias, const rdb_linear_desc *d,
                       int num_cus, void *scratch, int64_t scratch_bytes, hipStream_t s)
{
    if (!fg_state_ok(d) || !fg_aligned16(state) || d->tokens * ldx >= (1ll << 29)) return RDB_E_UNSUPPORTED;
    if (y && (d->tokens * ldy >= (1ll << 29))) return RDB_E_UNSUPPORTED;
    float *z = fg_state_z(state);
    if (int rc = fg_project_kept(z, x, ldx, y, ldy, d, num_cus, scratch, scratch_bytes, s, {})) return rc;
    if (!y) return RDB_OK;
    return fg_fwd_from_z(y, ldy, z, coef, bias, d, num_cus, s);
}

int linear_fwd_projected_f32(void *y, int64_t ldy, const void *state, const void *coef, const void *bias, const rdb_linear_desc *d, int num_cus,
                             hipStream_t s)
{
    if (!fg_state_ok(d) || d->tokens * ldy >= (1ll << 29)) return RDB_E_UNSUPPORTED;
    return fg_fwd_from_z(y, ldy, fg_state_z(state), coef, bias, d, num_cus, s);
}

// dx (NULL: not wanted) and dcoef from dy, the state and C.
int linear_bwd_projected_f32(void *dx, int64_t lddx, float *dcoef, const void *dy, int64_t lddy, const void *state, const void *coef,
                             const rdb_linear_desc *d, int num_cus, void *workspace, int64_t workspace_bytes, hipStream_t s)
{
    if (!fg_state_ok(d) || !workspace || !fg_aligned16(workspace) || workspace_bytes < linear_f32_bwd_projected_workspace(d, num_cus))
        return RDB_E_UNSUPPORTED;
    if (d->tokens * lddy >= (1ll << 29) || (dx && d->tokens * lddx >= (1ll << 29))) return RDB_E_UNSUPPORTED;
    float *part = reinterpret_cast<float *>(static_cast<char *>(workspace) + linear_f32_workspace(RDB_OP_LINEAR_BWD_DX, d, num_cus));
    return fg_backward(dx, lddx, dcoef, RDB_F32, dy, lddy, fg_state_z(state), coef, d, num_cus, workspace, workspace_bytes, part, s);
}

// ----------------------------------------------------------------------------------------------- materialise on the matrix cores
// W = C . N (+ s . R) written to memory as fp32, matrix-coef, the (coef_rows, row_len) base tensor or its transpose
// (src/rten_cpp/RandumbTensor.py:235-290), and its adjoint dcoef = dW . N^T (RandumbTensor.py:304-359): the same products as
// the factored layer's, with the other operand being C or dW.  Worth it from some tens of millions of multiply-adds on; below
// that the caller's vector-ALU kernels are as fast.
constexpr int64_t FG_MATERIALIZE_MIN_MACS = (int64_t)1 << 26, FG_COEF_GRAD_MIN_MACS = (int64_t)1 << 23;

static bool fg_mat_ok(int64_t coef_rows, int64_t k, int64_t row_len, int64_t min_macs)
{
    return coef_rows > 0 && k > 0 && row_len > 0 && coef_rows * k < (1ll << 29) && coef_rows * row_len < (1ll << 29) && row_len < (1 << 30) &&
           coef_rows * k * row_len >= min_macs;
}

int materialize_mat_f32(float *out, const void *coef, int coef_dtype, int64_t coef_rows, int64_t k, int64_t row_len, bool transposed, uint32_t seed,
                        const void *scale_bias, int num_cus, hipStream_t s)
{
    if (!fg_mat_ok(coef_rows, k, row_len, FG_MATERIALIZE_MIN_MACS)) return RDB_E_UNSUPPORTED;
    const float *C = (const float *)coef;
    if (!transposed) {
        // W[o, i] = sum_m C[o, m] noise(i, m): rows = o from C, columns = i hashed; the random bias at index o * row_len + i
        FgProduct q = {C, k, coef_rows * k, nullptr, 0, 0, out, row_len, nullptr, coef_rows, row_len, k,
                       0, 0, 0, 0, seed, (uint32_t)row_len, 1u, (const float *)scale_bias, nullptr, 0, nullptr};
        q.a_es = fg_es(coef_dtype);
        q.scale_bf16 = coef_dtype == RDB_BF16;
        return fg_launch<FG_KCONT, FG_NOISE_I>(q, num_cus, s, "f32_gemm_kernel (W = C . N)");
    }
    // W^T[i, o]: rows = i hashed, columns = o from C; the random bias at index o * row_len + i
    FgProduct q = {nullptr, 0, 0, C, k, coef_rows * k, out, coef_rows, nullptr, row_len, coef_rows, k,
                   0, 0, 0, 0, seed, 1u, (uint32_t)row_len, (const float *)scale_bias, nullptr, 0, nullptr};
    q.b_es = fg_es(coef_dtype);
    q.scale_bf16 = coef_dtype == RDB_BF16;
    return fg_launch<FG_NOISE_I, FG_KCONT>(q, num_cus, s, "f32_gemm_kernel (W^T = N^T . C^T)");
}

static int mat_bwd_room(int64_t coef_rows, int64_t k, int64_t row_len, int num_cus) { return fg_room(coef_rows, k, row_len, num_cus, 256, 64).ranges; }

// scratch of the adjoint: one [coef_rows x k] matrix per range of the row (none with a single range)
int64_t coef_grad_mat_f32_workspace(int64_t coef_rows, int64_t k, int64_t row_len, int num_cus)
{
    if (!fg_mat_ok(coef_rows, k, row_len, FG_COEF_GRAD_MIN_MACS)) return 0;
    const int r = mat_bwd_room(coef_rows, k, row_len, num_cus);
    return r > 1 ? (int64_t)r * up256(coef_rows * k * 4) : 0;
}

// dcoef[o, m] = sum_i dW[o, i] noise(i, m); dcoef is overwritten
int coef_grad_mat_f32(float *dcoef, const void *dW, int dw_dtype, int64_t coef_rows, int64_t k, int64_t row_len, uint32_t seed, void *workspace,
                      int64_t workspace_bytes, int num_cus, hipStream_t s)
{
    if (!fg_mat_ok(coef_rows, k, row_len, FG_COEF_GRAD_MIN_MACS)) return RDB_E_UNSUPPORTED;
    const int64_t need = coef_grad_mat_f32_workspace(coef_rows, k, row_len, num_cus);
    if (need > 0 && (!workspace || !fg_aligned16(workspace) || workspace_bytes < need)) return RDB_E_UNSUPPORTED;
    FgProduct q = {(const float *)dW, row_len, coef_rows * row_len, nullptr, 0, 0, dcoef, k, nullptr, coef_rows, k, row_len, 0, 0, 0, 0, seed};
    q.a_es = fg_es(dw_dtype);
    return fg_launch_ranges<FG_KCONT, FG_NOISE_M>(q, mat_bwd_room(coef_rows, k, row_len, num_cus), (float *)workspace, up256(coef_rows * k * 4) / 4, num_cus,
                                                  s, "f32_gemm_kernel (dcoef = dW . N^T)");
}

// ----------------------------------------------------------------------------------------------- a dense product
// ranges of 64 values and more: 216 tokens x 966 -> 198 took 30 us in one, 14 with the sums; dW of 497 tokens x 797 -> 410 22 -> 15
static int product_room(int64_t M, int64_t N, int64_t K, int num_cus) { return fg_room(M, N, K, num_cus, 64, 64).ranges; }
static bool product_ok(int64_t M, int64_t N, int64_t K) { return M > 0 && N > 0 && K > 0 && M * N < (1ll << 29) && K < (1 << 30); }

// The products of a vector-coef layer's backward pass, dx = dy . W and dW = dy^T . x, side by side in one launch where both are wanted; what is left to
// add up is left to a launch that comes anyway: dx's ranges (dx_sum, blocks 0: there are none), and up to VECTOR_DW_PARTS of dW's, as partial matrices (dw).
static bool vector_products_ok(int64_t tokens, int64_t in_f, int64_t out_f)
{
    return product_ok(tokens, in_f, out_f) && product_ok(out_f, in_f, tokens) && tokens * out_f < (1ll << 29) && tokens * in_f < (1ll << 29) && f32_split_mode();
}
// dW's ranges: its partial matrices are added up where dW is contracted with the noise, which is the vector ALU's, so they cost memory traffic and its power: at most 16 MB
// of them.  Vector-coef steps, us, with one, two, four, eight ranges at most: 1024 tokens x 512 -> 1024, k = 200 130, 118, 117, 118; 1500 x 300 -> 3000, k = 60 146,
// 147, 130, 131; 2048 x 1024 -> 1024, k = 256 256, 245, 245, 244; 1024 x 768 -> 3072, k = 256, kept up for a second: 464, 475, 475, 477.
// Many tokens of a small layer are more ranges than the contraction holds on the way (VECTOR_DW_PARTS): they and dx's are added up by a launch of their own then.  Eight at most
// and so, us: 30138 x 111 -> 331, k = 111 217, 131 (eight launches 145); 13811 x 135 -> 211, k = 52 96, 80 (85); 9080 x 280 -> 560, k = 18 130, 109 (118).
// Without dx beside it, whose tiles fill its last round, a product of dW that is not short (1280 tokens and more) loses more to that round: 32 MB there.  No dx, 16 and 32 MB: 8192 x 768 -> 3072, k = 8
// 539, 442 (469 as calls of their own); 19876 x 1288 -> 680, k = 4 539, 486 (501); 16384 x 1024 -> 1024, k = 8 384, 386; 1722 x 1388 -> 1566, k = 8 217, 191 (199); 1024 x 768 -> 3072, k = 256 447, 452; with dx
// 16384 x 1024 -> 1024 514, 551, 32768 x 512 -> 512, k = 8 313, 334.
// With dx one range of dW is tiles that run as long as the whole launch, each beside others on its unit, where they are less than two to three units: two ranges there.  Steps with one and two: 8192 x 1388 -> 1566, k = 8
// 993, 813 (892 as calls of their own); 8192 x 1771 -> 1463 1042, 956 (962); 4096 x 768 -> 3072, k = 256 778, 726 (831); 1400 tokens of it 527, 531, 1250 493, 501; 8192 x 2000 -> 2000, 256 tiles, one range: 1199 (1211).
static int vector_dw_room(int64_t tokens, int64_t in_f, int64_t out_f, bool dx, int num_cus)
{
    const bool few_tiles = 3 * cdiv(out_f, 128) * cdiv(in_f, 128) < 2 * num_cus;
    const int64_t most = std::max<int64_t>(few_tiles && tokens >= 1280 ? 2 : 1, (dx || tokens < 1280 ? 16 << 20 : 32 << 20) / (out_f * in_f * 4));
    return (int)std::min<int64_t>(product_room(out_f, in_f, tokens, num_cus), most);
}
// scratch: dx's partial matrices and dW's (or dW); 0: not taken
int64_t vector_products_workspace(int64_t tokens, int64_t in_f, int64_t out_f, bool want_dx)
{
    if (!vector_products_ok(tokens, in_f, out_f)) return 0;
    const int num_cus = num_compute_units(), r = want_dx ? product_room(tokens, in_f, out_f, num_cus) : 1;
    const int dw = vector_dw_room(tokens, in_f, out_f, want_dx, num_cus);
    return (r > 1 ? r : 0) * up256(tokens * in_f * 4) + (dw > VECTOR_DW_PARTS ? dw + 1 : dw) * up256(out_f * in_f * 4);
}
static FgPlan vector_dw_plan(int64_t tokens, int64_t in_f, int64_t out_f, bool dx, int num_cus)
{
    return fg_plan(out_f, in_f, tokens, num_cus, vector_dw_room(tokens, in_f, out_f, dx, num_cus), FgGroups<FG_MCONT, FG_MCONT>::four);
}
int vector_dw_ranges(int64_t tokens, int64_t in_f, int64_t out_f)
{
    return vector_products_ok(tokens, in_f, out_f) ? vector_dw_plan(tokens, in_f, out_f, false, num_compute_units()).ranges : 0;
}
int vector_products(float *dx, const float *dy, int64_t lddy, const float *x, int64_t ldx, const float *W, int64_t tokens, int64_t in_f, int64_t out_f,
                    void *workspace, FgSum *dx_sum, VectorDW *dw, hipStream_t s)
{
    if (!vector_products_ok(tokens, in_f, out_f) || tokens * lddy >= (1ll << 29) || tokens * ldx >= (1ll << 29)) return RDB_E_UNSUPPORTED;
    const int num_cus = num_compute_units(), room = dx ? product_room(tokens, in_f, out_f, num_cus) : 1, dw_room = vector_dw_room(tokens, in_f, out_f, dx != nullptr, num_cus);
    const int64_t dx_stride = up256(tokens * in_f * 4) / 4, dw_stride = up256(out_f * in_f * 4) / 4;
    float *dx_part = static_cast<float *>(workspace), *dw_part = dx_part + (room > 1 ? room : 0) * dx_stride;
    FgProduct qx = {dy, lddy, (tokens - 1) * lddy + out_f, W, in_f, out_f * in_f, dx, in_f, nullptr, tokens, in_f, out_f, 0, 0, 0, 0, 0u};
    FgProduct qw = {dy, lddy, (tokens - 1) * lddy + out_f, x, ldx, (tokens - 1) * ldx + in_f, dw_part, in_f, nullptr, out_f, in_f, tokens, 0, 0, 0, 0, 0u};
    *dx_sum = {};
    // what the contraction does not add up on its way
    auto done = [&](int parts) {
        *dw = {dw_part, dw_stride, parts};
        if (parts <= VECTOR_DW_PARTS) return (int)RDB_OK;
        float *const sum = dw_part + dw_room * dw_stride;
        const int rc = fg_launch_sums(*dx_sum, fg_sum(sum, 0, dw_part, qw.M * qw.N, dw_stride, parts), s);
        *dx_sum = {};
        *dw = {sum, 0, 1};
        return rc;
    };
    auto ranges = [](FgProduct &q, int r, float *part, int64_t stride) {
        q.kchunk = r > 1 ? fg_chunk(q.K, r) : 0;
        if (r > 1) {
            q.out = part;
            q.split_stride = stride;
        }
    };
    if (dx) {
        const FgPairPlan plan = fg_plan_pair({qx.M, qw.M}, {qx.N, qw.N}, {qx.K, qw.K}, num_cus, {room, dw_room}, false);
        FgProduct tx = qx, tw = qw;
        tx.bm = tw.bm = plan.bm;
        tx.groups = tw.groups = plan.groups;
        ranges(tx, plan.ranges[0], dx_part, dx_stride);
        ranges(tw, plan.ranges[1], dw_part, dw_stride);
        const int rc = fg_launch_pair(tx, tw, s);
        if (rc != RDB_E_UNSUPPORTED) {
            *dx_sum = fg_sum(dx, 0, dx_part, qx.M * qx.N, dx_stride, plan.ranges[0]);
            return rc ? rc : done(plan.ranges[1]);
        }
        const FgPlan px = fg_plan(qx.M, qx.N, qx.K, num_cus, room, FgGroups<FG_KCONT, FG_MCONT>::four);
        qx.bm = px.bm;
        qx.groups = px.groups;
        ranges(qx, px.ranges, dx_part, dx_stride);
        if (int rx = fg_launch<FG_KCONT, FG_MCONT>(qx, num_cus, s, "f32_gemm_kernel (dx = dy . W)")) return rx;
        *dx_sum = fg_sum(dx, 0, dx_part, qx.M * qx.N, dx_stride, px.ranges);
    }
    const FgPlan pw = vector_dw_plan(tokens, in_f, out_f, dx != nullptr, num_cus);
    qw.bm = pw.bm;
    qw.groups = pw.groups;
    ranges(qw, pw.ranges, dw_part, dw_stride);
    const int rc = fg_launch<FG_MCONT, FG_MCONT>(qw, num_cus, s, "f32_gemm_kernel (dW = dy^T . x)");
    return rc ? rc : done(pw.ranges);
}

}  // namespace rdb

using namespace rdb;

extern "C" int64_t rdb_product_f32_workspace_bytes(int64_t M, int64_t N, int64_t K)
{
    if (!product_ok(M, N, K)) return 0;
    const int r = product_room(M, N, K, num_compute_units());
    return r > 1 ? (int64_t)r * up256(M * N * 4) : 0;
}

extern "C" int rdb_product_f32(float *out, const float *a, int64_t lda, int a_across, const float *b, int64_t ldb, int b_across, const float *bias, int64_t M,
                               int64_t N, int64_t K, void *workspace, int64_t workspace_bytes, void *stream)
{
    if (M < 0 || N < 0 || K < 0) return set_error(RDB_E_SHAPE, "rdb_product_f32: negative size %lld x %lld x %lld", (long long)M, (long long)N, (long long)K);
    if (!product_ok(M, N, K) || (a_across && !b_across))
        return set_error(RDB_E_UNSUPPORTED, "rdb_product_f32: needs non-empty sizes, M * N below 2^29 and not (a_across without b_across)");
    if (!out || !a || !b) return set_error(RDB_E_NULL, "rdb_product_f32: out, a or b is NULL");
    if (lda < (a_across ? M : K) || ldb < (b_across ? N : K)) return set_error(RDB_E_SHAPE, "rdb_product_f32: leading dimension smaller than the row");
    if (lda * (a_across ? K : M) >= (1ll << 29) || ldb * (b_across ? K : N) >= (1ll << 29))
        return set_error(RDB_E_UNSUPPORTED, "rdb_product_f32: matrices of less than 2^29 elements");
    const int num_cus = num_compute_units();
    FgProduct q = {a, lda, a_across ? (K - 1) * lda + M : (M - 1) * lda + K, b, ldb, b_across ? (K - 1) * ldb + N : (N - 1) * ldb + K, out, N, bias, M, N, K,
                   0, 0, 0, 0, 0u};
    const int64_t stride = up256(M * N * 4);
    int room = product_room(M, N, K, num_cus);
    if (!workspace || !fg_aligned16(workspace)) room = 1;
    else if (room * stride > workspace_bytes) room = (int)std::max<int64_t>(1, workspace_bytes / stride);
    float *part = static_cast<float *>(workspace);
    hipStream_t s = (hipStream_t)stream;
    const char *name = "f32_gemm_kernel (dense product)";
    if (a_across) return fg_launch_ranges<FG_MCONT, FG_MCONT>(q, room, part, stride / 4, num_cus, s, name, FG_HOST_US);
    if (b_across) return fg_launch_ranges<FG_KCONT, FG_MCONT>(q, room, part, stride / 4, num_cus, s, name, FG_HOST_US);
    return fg_launch_ranges<FG_KCONT, FG_KCONT>(q, room, part, stride / 4, num_cus, s, name, FG_HOST_US);
}
