// The row-wise and element-wise passes of a transformer block around its pseudorandom linears, in bf16 with fp32 arithmetic:
// RMS normalisation (with the residual addition in front of it), the squared ReLU, and the cross entropy of the output head.
// Each is one pass over memory where a chain of stock operators makes several and converts to fp32 and back in between; the
// values are rounded to bf16 at the same places as there (src: modded-nanogpt/gpt_models.py:186-257, F.rms_norm,
// F.relu(x).square(), F.cross_entropy(logits.float(), target)).  All are bound by memory; measured, us, against the stock chain:
// 8192 x 768: normalisation 6.1 (38), with the addition 10.2 (46), backward 8.6 (69), with the second gradient 9.8 (76);
// 8192 x 3072: squared ReLU 19 (43), backward 26 (47); cross entropy of 8192 x 50304 logits 152 forward and 324 backward, 5.4 and
// 5.1 TB/s (with the conversion to fp32 and back 1800 and 2000).
#include "rdb_common.hpp"

namespace rdb {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));


__device__ __forceinline__ float wave_sum(float v)
{
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}

// ----------------------------------------------------------------------------------------------- RMS normalisation
// Memory bound: a wave owns a row and holds it in registers (NV pieces of 4 values a lane), so x is read once and the reduction
// costs no second pass; four rows a block.
struct NormParams {
    bf16_t *y;            // normalised rows
    bf16_t *sum;          // ADD: x + delta, rounded to bf16 (what is normalised)
    float *rstd;          // [rows]
    const bf16_t *x, *delta;
    int rows, dim;
    float eps;
};

template <int NV, bool ADD> __global__ __launch_bounds__(256) void rms_norm_kernel(NormParams p)
{
    const int row = (int)blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= p.rows) return;
    const int64_t base = (int64_t)row * p.dim;
    float v[NV][4];
    u32x2 in[NV], de[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 64 + lane) * 4;
        in[i] = u32x2{0, 0};
        de[i] = u32x2{0, 0};
        if (c < p.dim) {
            in[i] = *reinterpret_cast<const u32x2 *>(p.x + base + c);
            if (ADD) de[i] = *reinterpret_cast<const u32x2 *>(p.delta + base + c);
        }
    }
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 64 + lane) * 4;
        if (ADD) {
            in[i].x = f32x2_to_bf16x2(lo_f32(in[i].x) + lo_f32(de[i].x), hi_f32(in[i].x) + hi_f32(de[i].x));
            in[i].y = f32x2_to_bf16x2(lo_f32(in[i].y) + lo_f32(de[i].y), hi_f32(in[i].y) + hi_f32(de[i].y));
            if (c < p.dim) *reinterpret_cast<u32x2 *>(p.sum + base + c) = in[i];
        }
        v[i][0] = lo_f32(in[i].x);
        v[i][1] = hi_f32(in[i].x);
        v[i][2] = lo_f32(in[i].y);
        v[i][3] = hi_f32(in[i].y);
#pragma unroll
        for (int e = 0; e < 4; ++e) s = fmaf(v[i][e], v[i][e], s);
    }
    const float r = rsqrtf(wave_sum(s) / (float)p.dim + p.eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 64 + lane) * 4;
        if (c >= p.dim) continue;
        const u32x2 o = {f32x2_to_bf16x2(v[i][0] * r, v[i][1] * r), f32x2_to_bf16x2(v[i][2] * r, v[i][3] * r)};
        *reinterpret_cast<u32x2 *>(p.y + base + c) = o;
    }
    if (lane == 0) p.rstd[row] = r;
}

// dx = rstd (dy - xhat <dy, xhat> / dim) (+ dsum: the gradient that reaches the sum past the normalisation), xhat = x rstd
struct NormBwdParams {
    bf16_t *dx;
    const bf16_t *dy, *x, *dsum;
    const float *rstd;
    int rows, dim;
};

template <int NV, bool ADD> __global__ __launch_bounds__(256) void rms_norm_bwd_kernel(NormBwdParams p)
{
    const int row = (int)blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= p.rows) return;
    const int64_t base = (int64_t)row * p.dim;
    u32x2 d[NV], x[NV], a[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 64 + lane) * 4;
        d[i] = x[i] = a[i] = u32x2{0, 0};
        if (c < p.dim) {
            d[i] = *reinterpret_cast<const u32x2 *>(p.dy + base + c);
            x[i] = *reinterpret_cast<const u32x2 *>(p.x + base + c);
            if (ADD) a[i] = *reinterpret_cast<const u32x2 *>(p.dsum + base + c);
        }
    }
    const float r = p.rstd[row];
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        s = fmaf(lo_f32(d[i].x), lo_f32(x[i].x) * r, s);
        s = fmaf(hi_f32(d[i].x), hi_f32(x[i].x) * r, s);
        s = fmaf(lo_f32(d[i].y), lo_f32(x[i].y) * r, s);
        s = fmaf(hi_f32(d[i].y), hi_f32(x[i].y) * r, s);
    }
    const float m = wave_sum(s) / (float)p.dim;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 64 + lane) * 4;
        if (c >= p.dim) continue;
        u32x2 o = {f32x2_to_bf16x2((lo_f32(d[i].x) - lo_f32(x[i].x) * r * m) * r, (hi_f32(d[i].x) - hi_f32(x[i].x) * r * m) * r),
                   f32x2_to_bf16x2((lo_f32(d[i].y) - lo_f32(x[i].y) * r * m) * r, (hi_f32(d[i].y) - hi_f32(x[i].y) * r * m) * r)};
        if (ADD) {   // the two gradients are bf16 tensors that autograd would add
            o.x = f32x2_to_bf16x2(lo_f32(o.x) + lo_f32(a[i].x), hi_f32(o.x) + hi_f32(a[i].x));
            o.y = f32x2_to_bf16x2(lo_f32(o.y) + lo_f32(a[i].y), hi_f32(o.y) + hi_f32(a[i].y));
        }
        *reinterpret_cast<u32x2 *>(p.dx + base + c) = o;
    }
}

// ----------------------------------------------------------------------------------------------- squared ReLU
// y = relu(x)^2;  dx = dy * 2 relu(x).  Memory bound: 16 bytes a lane and step, two steps in flight.
template <bool GRAD> __global__ __launch_bounds__(256) void relu_square_kernel(bf16_t *__restrict__ out, const bf16_t *__restrict__ x,
                                                                               const bf16_t *__restrict__ dy, int64_t n)
{
    const int64_t nvec = n / 8, stride = (int64_t)gridDim.x * 256;
    const u32x4 *xv = reinterpret_cast<const u32x4 *>(x), *dv = reinterpret_cast<const u32x4 *>(dy);
    u32x4 *ov = reinterpret_cast<u32x4 *>(out);
#pragma unroll 2
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nvec; e += stride) {
        const u32x4 w = xv[e];
        u32x4 o;
        if (GRAD) {
            const u32x4 d = dv[e];
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = relu2_grad_pair(w[i], d[i]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = relu2_pair(w[i]);
        }
        ov[e] = o;
    }
    const int64_t e = nvec * 8 + (int64_t)threadIdx.x;
    if (blockIdx.x == 0 && e < n) {
        const uint32_t w = x[e];
        out[e] = (bf16_t)((GRAD ? relu2_grad_pair(w, dy[e]) : relu2_pair(w)) & 0xffffu);
    }
}

// ----------------------------------------------------------------------------------------------- cross entropy
// Per row of bf16 logits: lse = log sum exp, nll = lse - logit[target]; rows whose target is ignore_index count for nothing, a
// target outside the classes gives NaN.  One block a row, one pass: every thread keeps a running maximum and a sum scaled to it
// (the exponentials of 8192 x 50304 logits cost the vector ALU less time than reading them), which the block merges at the end.
constexpr float LOG2E = 1.44269504088896340736f;

__global__ __launch_bounds__(256) void cross_entropy_kernel(float *__restrict__ lse, float *__restrict__ nll, const bf16_t *__restrict__ logits,
                                                            const int64_t *__restrict__ target, int64_t V, int64_t ignore)
{
    __shared__ float ms[4], ss[4];
    const int64_t row = blockIdx.x;
    const bf16_t *r = logits + row * V;
    const u32x4 *rv = reinterpret_cast<const u32x4 *>(r);
    const int nvec = (int)(V / 8), t = threadIdx.x;
    float m = -INFINITY, s = 0.0f;
#pragma unroll 4
    for (int i = t; i < nvec; i += 256) {
        const u32x4 w = rv[i];
        float f[8], top = m;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f[2 * j] = lo_f32(w[j]);
            f[2 * j + 1] = hi_f32(w[j]);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) top = fmaxf(top, f[j]);
        const float ref = top == -INFINITY ? 0.0f : top;   // nothing but -inf so far: every term is exp2(-inf) = 0
        s *= __builtin_amdgcn_exp2f((m - ref) * LOG2E);
#pragma unroll
        for (int j = 0; j < 8; ++j) s += __builtin_amdgcn_exp2f((f[j] - ref) * LOG2E);
        m = top;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float m2 = __shfl_xor(m, o, 64), s2 = __shfl_xor(s, o, 64), top = fmaxf(m, m2), ref = top == -INFINITY ? 0.0f : top;
        s = s * __builtin_amdgcn_exp2f((m - ref) * LOG2E) + s2 * __builtin_amdgcn_exp2f((m2 - ref) * LOG2E);
        m = top;
    }
    if ((t & 63) == 0) {
        ms[t >> 6] = m;
        ss[t >> 6] = s;
    }
    __syncthreads();
    if (t == 0) {
        const float top = fmaxf(fmaxf(ms[0], ms[1]), fmaxf(ms[2], ms[3])), ref = top == -INFINITY ? 0.0f : top;
        float sum = 0.0f;
        for (int w = 0; w < 4; ++w) sum += ss[w] * __builtin_amdgcn_exp2f((ms[w] - ref) * LOG2E);
        const float l = logf(sum) + ref;
        const int64_t c = target[row];
        lse[row] = l;
        nll[row] = c == ignore ? 0.0f : (c < 0 || c >= V) ? NAN : l - bf16_to_f32(r[c]);
    }
}

// loss = sum of nll / number of rows that count; count[0] is kept for the backward pass.  One block, fixed order.
__global__ __launch_bounds__(1024) void cross_entropy_mean_kernel(float *__restrict__ loss, float *__restrict__ count, const float *__restrict__ nll,
                                                                  const int64_t *__restrict__ target, int64_t rows, int64_t ignore)
{
    __shared__ float s[16], n[16];
    float a = 0.0f, c = 0.0f;
#pragma unroll 4
    for (int64_t i = threadIdx.x; i < rows; i += 1024) {
        a += nll[i];
        c += target[i] == ignore ? 0.0f : 1.0f;
    }
    a = wave_sum(a);
    c = wave_sum(c);
    if ((threadIdx.x & 63) == 0) {
        s[threadIdx.x >> 6] = a;
        n[threadIdx.x >> 6] = c;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        a = c = 0.0f;
        for (int w = 0; w < 16; ++w) {
            a += s[w];
            c += n[w];
        }
        loss[0] = a / c;
        count[0] = c;
    }
}

// dlogits = (exp(logit - lse) - [class == target]) * dloss / count, 0 in ignored rows, NaN in rows whose target is outside the
// classes (their loss is NaN too: a program that does not look at the loss must not train on them)
__global__ __launch_bounds__(256) void cross_entropy_bwd_kernel(bf16_t *__restrict__ dlogits, const bf16_t *__restrict__ logits,
                                                                const int64_t *__restrict__ target, const float *__restrict__ lse,
                                                                const float *__restrict__ dloss, const float *__restrict__ count, int64_t V, int64_t ignore)
{
    const int64_t row = blockIdx.x, c = target[row];
    const u32x4 *rv = reinterpret_cast<const u32x4 *>(logits + row * V);
    u32x4 *ov = reinterpret_cast<u32x4 *>(dlogits + row * V);
    const float l = lse[row] * LOG2E, g = c == ignore ? 0.0f : c < 0 || c >= V ? __uint_as_float(0x7fc00000u) : dloss[0] / count[0];
    const int nvec = (int)(V / 8);
#pragma unroll 4
    for (int i = threadIdx.x; i < nvec; i += 256) {
        const u32x4 w = rv[i];
        u32x4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = i * 8 + 2 * j;
            float a = __builtin_amdgcn_exp2f(fmaf(lo_f32(w[j]), LOG2E, -l)), b = __builtin_amdgcn_exp2f(fmaf(hi_f32(w[j]), LOG2E, -l));
            if (k == c) a -= 1.0f;
            if (k + 1 == c) b -= 1.0f;
            o[j] = g == 0.0f ? 0u : f32x2_to_bf16x2(a * g, b * g);
        }
        store_stream(ov + i, o);
    }
}

static bool a16(const void *p) { return ((uintptr_t)p & 15) == 0; }
static bool a8(const void *p) { return ((uintptr_t)p & 7) == 0; }

template <bool ADD> static int launch_norm(const NormParams &p, hipStream_t s)
{
    const dim3 grid((unsigned)cdiv(p.rows, 4));
    const int nv = (int)cdiv(p.dim, 256);
    if (nv <= 1) rms_norm_kernel<1, ADD><<<grid, 256, 0, s>>>(p);
    else if (nv <= 2) rms_norm_kernel<2, ADD><<<grid, 256, 0, s>>>(p);
    else if (nv <= 3) rms_norm_kernel<3, ADD><<<grid, 256, 0, s>>>(p);
    else if (nv <= 4) rms_norm_kernel<4, ADD><<<grid, 256, 0, s>>>(p);
    else if (nv <= 8) rms_norm_kernel<8, ADD><<<grid, 256, 0, s>>>(p);
    else rms_norm_kernel<16, ADD><<<grid, 256, 0, s>>>(p);
    return check_launch("rms_norm_kernel");
}
template <bool ADD> static int launch_norm_bwd(const NormBwdParams &p, hipStream_t s)
{
    const dim3 grid((unsigned)cdiv(p.rows, 4));
    const int nv = (int)cdiv(p.dim, 256);
    if (nv <= 1) rms_norm_bwd_kernel<1, ADD><<<grid, 256, 0, s>>>(p);
    else if (nv <= 2) rms_norm_bwd_kernel<2, ADD><<<grid, 256, 0, s>>>(p);
    else if (nv <= 3) rms_norm_bwd_kernel<3, ADD><<<grid, 256, 0, s>>>(p);
    else if (nv <= 4) rms_norm_bwd_kernel<4, ADD><<<grid, 256, 0, s>>>(p);
    else if (nv <= 8) rms_norm_bwd_kernel<8, ADD><<<grid, 256, 0, s>>>(p);
    else rms_norm_bwd_kernel<16, ADD><<<grid, 256, 0, s>>>(p);
    return check_launch("rms_norm_bwd_kernel");
}

}  // namespace rdb

using namespace rdb;

static int check_rows(const char *who, int64_t rows, int64_t dim)
{
    if (rows < 0 || dim <= 0 || rows >= (1ll << 31)) return set_error(RDB_E_SHAPE, "%s: bad size %lld x %lld", who, (long long)rows, (long long)dim);
    if (dim % 4 || dim > 4096) return set_error(RDB_E_UNSUPPORTED, "%s: rows of up to 4096 values, a multiple of 4", who);
    return RDB_OK;
}

extern "C" int rdb_rms_norm_fwd(void *y, void *sum, float *rstd, const void *x, const void *delta, int64_t rows, int64_t dim, float eps, void *stream)
{
    if (int rc = check_rows("rdb_rms_norm_fwd", rows, dim)) return rc;
    if (rows == 0) return RDB_OK;
    if (!y || !rstd || !x || (delta && !sum)) return set_error(RDB_E_NULL, "rdb_rms_norm_fwd: y, rstd, x or sum is NULL");
    if (!a8(y) || !a8(x) || !a8(delta) || (delta && !a8(sum))) return set_error(RDB_E_ALIGN, "rdb_rms_norm_fwd: rows must be 8-byte aligned");
    const NormParams p = {static_cast<bf16_t *>(y), static_cast<bf16_t *>(sum), rstd, static_cast<const bf16_t *>(x), static_cast<const bf16_t *>(delta),
                          (int)rows, (int)dim, eps};
    return delta ? launch_norm<true>(p, (hipStream_t)stream) : launch_norm<false>(p, (hipStream_t)stream);
}

extern "C" int rdb_rms_norm_bwd(void *dx, const void *dy, const void *x, const void *dsum, const float *rstd, int64_t rows, int64_t dim, void *stream)
{
    if (int rc = check_rows("rdb_rms_norm_bwd", rows, dim)) return rc;
    if (rows == 0) return RDB_OK;
    if (!dx || !dy || !x || !rstd) return set_error(RDB_E_NULL, "rdb_rms_norm_bwd: dx, dy, x or rstd is NULL");
    if (!a8(dx) || !a8(dy) || !a8(x) || !a8(dsum)) return set_error(RDB_E_ALIGN, "rdb_rms_norm_bwd: rows must be 8-byte aligned");
    const NormBwdParams p = {static_cast<bf16_t *>(dx), static_cast<const bf16_t *>(dy), static_cast<const bf16_t *>(x), static_cast<const bf16_t *>(dsum),
                             rstd, (int)rows, (int)dim};
    return dsum ? launch_norm_bwd<true>(p, (hipStream_t)stream) : launch_norm_bwd<false>(p, (hipStream_t)stream);
}

extern "C" int rdb_relu_square(void *out, const void *x, const void *dy, int64_t n, void *stream)
{
    if (n < 0) return set_error(RDB_E_SHAPE, "rdb_relu_square: negative size");
    if (n == 0) return RDB_OK;
    if (!out || !x) return set_error(RDB_E_NULL, "rdb_relu_square: out or x is NULL");
    if (!a16(out) || !a16(x) || !a16(dy)) return set_error(RDB_E_ALIGN, "rdb_relu_square: pointers must be 16-byte aligned");
    const int64_t blocks = cdiv(cdiv(n, 8), 512);
    const unsigned grid = (unsigned)(blocks < 1 ? 1 : blocks < 8192 ? blocks : 8192);
    hipStream_t s = (hipStream_t)stream;
    if (dy) relu_square_kernel<true><<<grid, 256, 0, s>>>(static_cast<bf16_t *>(out), static_cast<const bf16_t *>(x), static_cast<const bf16_t *>(dy), n);
    else relu_square_kernel<false><<<grid, 256, 0, s>>>(static_cast<bf16_t *>(out), static_cast<const bf16_t *>(x), nullptr, n);
    return check_launch("relu_square_kernel");
}

static int check_ce(const char *who, int64_t rows, int64_t V, const void *logits)
{
    if (rows <= 0 || V <= 0 || rows >= (1ll << 31) || V >= (1ll << 30)) return set_error(RDB_E_SHAPE, "%s: bad size %lld x %lld", who, (long long)rows, (long long)V);
    if (V % 8 || !a16(logits)) return set_error(RDB_E_UNSUPPORTED, "%s: a multiple of 8 classes and 16-byte aligned logits", who);
    return RDB_OK;
}

// scratch: 2 * rows + 1 floats, of which the backward pass needs lse (the first `rows`) and the count behind them
extern "C" int rdb_cross_entropy_fwd(float *loss, float *scratch, const void *logits, const int64_t *target, int64_t rows, int64_t classes, int64_t ignore_index,
                                     void *stream)
{
    if (int rc = check_ce("rdb_cross_entropy_fwd", rows, classes, logits)) return rc;
    if (!loss || !scratch || !logits || !target) return set_error(RDB_E_NULL, "rdb_cross_entropy_fwd: loss, scratch, logits or target is NULL");
    hipStream_t s = (hipStream_t)stream;
    cross_entropy_kernel<<<(unsigned)rows, 256, 0, s>>>(scratch, scratch + rows + 1, static_cast<const bf16_t *>(logits), target, classes, ignore_index);
    if (int rc = check_launch("cross_entropy_kernel")) return rc;
    cross_entropy_mean_kernel<<<1, 1024, 0, s>>>(loss, scratch + rows, scratch + rows + 1, target, rows, ignore_index);
    return check_launch("cross_entropy_mean_kernel");
}

extern "C" int rdb_cross_entropy_bwd(void *dlogits, const void *logits, const int64_t *target, const float *scratch, const float *dloss, int64_t rows,
                                     int64_t classes, int64_t ignore_index, void *stream)
{
    if (int rc = check_ce("rdb_cross_entropy_bwd", rows, classes, logits)) return rc;
    if (!dlogits || !logits || !target || !scratch || !dloss) return set_error(RDB_E_NULL, "rdb_cross_entropy_bwd: an argument is NULL");
    if (!a16(dlogits)) return set_error(RDB_E_ALIGN, "rdb_cross_entropy_bwd: dlogits must be 16-byte aligned");
    cross_entropy_bwd_kernel<<<(unsigned)rows, 256, 0, (hipStream_t)stream>>>(static_cast<bf16_t *>(dlogits), static_cast<const bf16_t *>(logits), target, scratch,
                                                                              dloss, scratch + rows, classes, ignore_index);
    return check_launch("cross_entropy_bwd_kernel");
}
