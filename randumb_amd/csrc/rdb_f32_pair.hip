// Two products of rdb_f32.hpp in one launch: t = dy . C and dC = dy^T . z of a layer's backward pass, which both read dy and do not need
// each other.  As launches of their own each pays for the start of its blocks (operands come from memory for all of them at
// once), for the end (all outputs leave at once) and for the gap behind; side by side one product's stages run under the other's.
// Backward pass of 2048 tokens x 768 -> 3072, k = 256, fp32: 72.2 -> 61.2 us (t and dC 25 + 25 -> 36, one sum fewer); 4097 tokens x 1001 ->
// 999, k = 100, bf16: 50.4 -> 38.8; 8000 x 3001 -> 601, k = 201, bf16: 130 -> 116; 300 x 2048 -> 2048, k = 512, fp32: 46.8 -> 37.4.
#include "rdb_f32.hpp"

namespace rdb {

struct FgPair {
    FgParams p[2];      // t = dy . C, dC = dy^T . z
    int x[2], y[2];     // blocks along the outputs' rows and columns
    int first;          // which of them has the lower block numbers: the one with the longer contraction per block
    int split;          // ... and how many they are
};

template <int BM, int G, bool VEC, int ES> __global__ __launch_bounds__(FG_THREADS * G, G == 1 ? 2 : 1) void f32_pair_kernel(FgPair q)
{
    constexpr int LT = FgBlock<BM, G, FG_KCONT, FG_MCONT, VEC, true, ES, ES>::LDS, LD = FgBlock<BM, G, FG_MCONT, FG_MCONT, VEC, true, ES, 4>::LDS;
    __shared__ __align__(16) float lds[LT > LD ? LT : LD];
    __shared__ int not_finite;
    const int b = (int)blockIdx.x, second = b >= q.split, which = q.first ^ second, at = b - (second ? q.split : 0);
    const int gx = q.x[which], xy = gx * q.y[which], bz = at / xy, in = at - bz * xy, by = in / gx, bx = in - by * gx;
    if (which == 0) f32_gemm_block<BM, G, FG_KCONT, FG_MCONT, FG_STORE, VEC, true, ES, ES>(q.p[0], bx, by, bz, gx, lds, not_finite);
    else f32_gemm_block<BM, G, FG_MCONT, FG_MCONT, FG_STORE, VEC, true, ES, 4>(q.p[1], bx, by, bz, gx, lds, not_finite);
}

// t: FG_KCONT x FG_MCONT, dc: FG_MCONT x FG_MCONT (its B side fp32); both with their plan (bm and groups the same), kchunk and out set.
int fg_launch_pair(const FgProduct &t, const FgProduct &dc, hipStream_t s)
{
    if (!fg_fits(t) || !fg_fits(dc) || t.bm != dc.bm || t.groups != dc.groups || (t.bm == 64 && t.groups != 2) || t.a_es != t.b_es || t.a_es != dc.a_es || dc.b_es != 4) return RDB_E_UNSUPPORTED;
    FgPair q;
    q.p[0] = fg_params(t);
    q.p[1] = fg_params(dc);
    const FgProduct *const of[2] = {&t, &dc};
    int64_t blocks[2];
    for (int i = 0; i < 2; ++i) {
        q.x[i] = (int)cdiv(of[i]->M, t.bm);
        q.y[i] = (int)cdiv(of[i]->N, FG_BN);
        blocks[i] = (int64_t)q.x[i] * q.y[i] * cdiv(of[i]->K, q.p[i].kchunk);
    }
    if (blocks[0] + blocks[1] >= (1ll << 31)) return RDB_E_UNSUPPORTED;
    q.first = q.p[1].kchunk > q.p[0].kchunk ? 1 : 0;
    q.split = (int)blocks[q.first];
    const unsigned grid = (unsigned)(blocks[0] + blocks[1]);
    const bool vec = fg_vec(t, FG_KCONT, FG_MCONT) && fg_vec(dc, FG_MCONT, FG_MCONT);
    auto run = [&](auto bm_, auto g_) {
        constexpr int BM = decltype(bm_)::value, G = decltype(g_)::value;
        if (t.a_es == 2) {
            if (vec) f32_pair_kernel<BM, G, true, 2><<<grid, FG_THREADS * G, 0, s>>>(q);
            else f32_pair_kernel<BM, G, false, 2><<<grid, FG_THREADS * G, 0, s>>>(q);
        } else {
            if (vec) f32_pair_kernel<BM, G, true, 4><<<grid, FG_THREADS * G, 0, s>>>(q);
            else f32_pair_kernel<BM, G, false, 4><<<grid, FG_THREADS * G, 0, s>>>(q);
        }
    };
    typedef std::integral_constant<int, 1> I1;
    typedef std::integral_constant<int, 2> I2;
    typedef std::integral_constant<int, 64> I64;
    typedef std::integral_constant<int, 128> I128;
    if (t.bm == 128 && t.groups == 2) run(I128{}, I2{});
    else if (t.bm == 128) run(I128{}, I1{});
    else run(I64{}, I2{});
    return check_launch("f32_pair_kernel (t = dy . C, dC = dy^T . z)");
}

}  // namespace rdb
