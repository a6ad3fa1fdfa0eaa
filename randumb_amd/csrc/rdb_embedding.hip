// Gradient of a dense embedding table in bf16, dW[v] = sum of dy over the positions that looked v up, rows that nobody looked up zero: one launch, bound by
// writing the table (50304 x 768: 77 MB), where the stock operator sorts the indices, clears the table and adds up in a dozen launches.  A block owns up to 128 rows
// of the table, two blocks to a compute unit, and looks through all indices itself, out of L2: nothing has to be sorted, cleared or counted by an earlier launch.
// Its eight waves take an eighth of the positions each, so that their lists, one behind the other, are in the order of the positions: fixed sums, in fp32,
// rounded once.  The block's lists together are mostly shorter than a wave, and then lie in one register.  A row of up to 64 positions is one wave's; one of more,
// a chain of that many loads, is all waves', each the positions of its own list, sixteen rows of dy in flight.  us, kernel alone, and the stock call with its launches:
// 50304 x 768, 8192 positions 27, 112; 1024 24, 77; 16384 31, 146 (48 with one block to a compute unit); half of 8192 at one row 181, 204; all of them 206, 304; 50304 x 256,
// 64 positions 19, 26.
#include "rdb_common.hpp"
#include <algorithm>
#include <type_traits>

namespace rdb {

int num_compute_units();   // rdb_error.hip
constexpr int EG_ROW_BITS = 7, EG_ROWS = 1 << EG_ROW_BITS, EG_WAVES = 8, EG_THREADS = EG_WAVES * 64, EG_PIECE = 512, EG_LIGHT = 64, EG_AHEAD = 8;
constexpr int64_t EG_POSITIONS = 16384;   // as many as the lists of two blocks have room for in a compute unit's LDS, 4 bytes each
constexpr int64_t EG_SUMS_BYTES = (EG_WAVES - 1) * EG_PIECE * (int64_t)sizeof(float);
static_assert(2 * (EG_SUMS_BYTES + EG_POSITIONS * 4 + (EG_ROWS + EG_WAVES) * 4) <= 160 * 1024, "two blocks to a compute unit");

template <typename I> __global__ __launch_bounds__(EG_THREADS) void embedding_grad_kernel(bf16_t *__restrict__ dw, const I *__restrict__ idx, const bf16_t *__restrict__ dy,
                                                                                          int positions, int each, int64_t vocab, int dim, int block_rows)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int hist[EG_ROWS], count[EG_WAVES];
    float *const sums = reinterpret_cast<float *>(smem);                                    // [EG_WAVES - 1][EG_PIECE]: those of wave 0 stay in its registers
    uint32_t *const lists = reinterpret_cast<uint32_t *>(sums + (EG_WAVES - 1) * EG_PIECE);   // [EG_WAVES][each]: position << EG_ROW_BITS | row of the block
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row0 = (int64_t)blockIdx.x * block_rows;
    if (threadIdx.x < EG_ROWS) hist[threadIdx.x] = 0;
    __syncthreads();
    uint32_t *const mine = lists + wave * each;
    const int first = wave * each, last = min(first + each, positions);
    int n = 0;
    for (int p0 = first; p0 < last; p0 += 64 * EG_AHEAD) {
        int64_t v[EG_AHEAD];
#pragma unroll
        for (int i = 0; i < EG_AHEAD; ++i) v[i] = (int64_t)idx[min(p0 + i * 64 + lane, last - 1)];   // clamped: loaded, not looked at
#pragma unroll
        for (int i = 0; i < EG_AHEAD; ++i) {
            const int p = p0 + i * 64 + lane;
            const int64_t r = v[i] - row0;
            const bool here = (p < last) & ((uint64_t)r < (uint64_t)block_rows);
            const uint64_t mask = __ballot(here);
            if (here) {
                mine[n + __popcll(mask & ((1ull << lane) - 1ull))] = (uint32_t)p << EG_ROW_BITS | (uint32_t)r;
                atomicAdd(&hist[r], 1);
            }
            n += __popcll(mask);
        }
    }
    if (lane == 0) count[wave] = n;
    __syncthreads();

    float acc[8];
    // adds the rows of dy that the lanes of `mask` have in `entry`, columns `col` and on, to acc, A rows in flight
    auto gather = [&](auto ahead, uint32_t entry, uint64_t mask, int col) {
        constexpr int A = decltype(ahead)::value;
        const bf16_t *const from = dy + (col < dim ? col : 0);   // loaded, not stored
        while (mask) {
            u32x4 d[A];
            const int took = __popcll(mask);
            int at = 0;
#pragma unroll
            for (int i = 0; i < A; ++i) {
                at = mask ? __builtin_ctzll(mask) : at;   // none left: the last one again, not added
                asm volatile("" : "+s"(at));              // a select, and not a branch around the load
                mask &= mask - 1;
                d[i] = *reinterpret_cast<const u32x4 *>(from + (int64_t)(__builtin_amdgcn_readlane((int)entry, at) >> EG_ROW_BITS) * dim);
            }
            // zeros for what was not there: under a condition the compiler moves each load behind it, one at a time (8192 positions of one row 205 -> 670 us)
#pragma unroll
            for (int i = 0; i < A; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t v = i < took ? d[i][j] : 0u;
                    acc[2 * j] += lo_f32(v);
                    acc[2 * j + 1] += hi_f32(v);
                }
        }
    };
    // ... that list w has of row r
    auto add = [&](auto ahead, int w, int r, int col) {
        const int entries = count[w];
        for (int e0 = 0; e0 < entries; e0 += 64) {
            const uint32_t entry = e0 + lane < entries ? lists[w * each + e0 + lane] : 0u;
            gather(ahead, entry, __ballot(e0 + lane < entries && (int)(entry & (EG_ROWS - 1)) == r), col);
        }
    };
    // all lists in the lanes of one register, where they fit
    int all = 0;
    uint32_t one = 0u;
    for (int w = 0; w < EG_WAVES; ++w) {
        const int entries = count[w], e = lane - all;
        if (e >= 0 && e < entries) one = lists[w * each + e];
        all += entries;
    }
    auto clear = [&]() {
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
    };
    auto store = [&](int r, int col) {
        if (col < dim)
            *reinterpret_cast<u32x4 *>(dw + (row0 + r) * dim + col) =
                u32x4{f32x2_to_bf16x2(acc[0], acc[1]), f32x2_to_bf16x2(acc[2], acc[3]), f32x2_to_bf16x2(acc[4], acc[5]), f32x2_to_bf16x2(acc[6], acc[7])};
    };
    const int rows = (int)min((int64_t)block_rows, vocab - row0);
    for (int r = wave; r < rows; r += EG_WAVES) {
        const int looked_up = hist[r];
        if (looked_up > EG_LIGHT) continue;
        for (int col = lane * 8; col < (dim + EG_PIECE - 1) / EG_PIECE * EG_PIECE; col += EG_PIECE) {
            clear();
            if (looked_up && all <= 64) gather(std::integral_constant<int, 4>{}, one, __ballot(lane < all && (int)(one & (EG_ROWS - 1)) == r), col);
            else if (looked_up)
                for (int w = 0; w < EG_WAVES; ++w) add(std::integral_constant<int, 4>{}, w, r, col);
            store(r, col);
        }
    }
    for (int r = 0; r < rows; ++r) {
        if (hist[r] <= EG_LIGHT) continue;   // the same for all waves
        for (int col = lane * 8; col < (dim + EG_PIECE - 1) / EG_PIECE * EG_PIECE; col += EG_PIECE) {
            clear();
            add(std::integral_constant<int, 16>{}, wave, r, col);
            if (wave) {
#pragma unroll
                for (int j = 0; j < 8; ++j) sums[(wave - 1) * EG_PIECE + j * 64 + lane] = acc[j];
            }
            __syncthreads();
            if (wave == 0) {
#pragma unroll
                for (int j = 0; j < 8; ++j)
#pragma unroll
                    for (int w = 1; w < EG_WAVES; ++w) acc[j] += sums[(w - 1) * EG_PIECE + j * 64 + lane];
                store(r, col);
            }
            __syncthreads();
        }
    }
}

}  // namespace rdb

using namespace rdb;

// what one launch can do: the grid's threads stay below 2^32
static bool embedding_fits(int64_t positions, int64_t vocab, int64_t dim)
{
    return positions > 0 && positions <= EG_POSITIONS && vocab > 0 && vocab <= (1ll << 29) && dim > 0 && dim % 8 == 0 && dim <= (1 << 20);
}

// Where that is the faster way.  Every block looks through all indices and writes its rows one by one, so a table costs rounds of blocks, some 12 us each, however few its columns; the stock call
// adds up positions one after the other, 50 ns each up to 3072 of them, sorts more than that, 55 us, and clears the table, which is faster than rows one by one.  us on the device, this one and the
// stock one, on either side of each line (256 compute units: a round is 65536 rows):
//   one round, few positions for the rows: 16384 x 64, 64 positions 8.3, 6.9; 128 8.3, 10.0; 50304 x 256, 256 18.6, 20.2; 128 18.5, 13.6; 65536 x 8, 256 20.5, 16.8; 400 20.6, 24.2; x 768, 128 28.1, 24.1;
//   256 28.4, 32.3; 32768 x 768, 64 16.6, 14.4; 128 16.8, 18.1
//   few rows, where a block's eight have most positions: 10 x 384, 1024 positions 33, 48; 10 x 768 60, 48; 30 x 1600, 2048 115, 90; 65 x 1600 29, 88; sorted ones: 65 x 768, 4096 54, 55; 8192 83, 73;
//   100 x 768, 8192 70, 72; 16384 89, 84; 100 x 1600, 4096 33, 62; 8192 148, 84
//   rounds against positions: two, x 64 columns: 512 positions 38.1, 32.2; 1024 38.0, 57.8; three: 1024 55.1, 59.8; four: 1024 72.3, 70.6; 2048 73.0, 132
//   rounds, 4096 positions: four, x 256 74, 95; five 91, 97; seven 112, 100; eight 142, 98; x 768, whose writing takes longer than the indices: eight 187, 198; thirteen 265, 261; a million rows x 8:
//   246, 99
extern "C" int rdb_embedding_bwd_takes(int64_t positions, int64_t vocab, int64_t dim)
{
    if (!embedding_fits(positions, vocab, dim)) return 0;
    const int64_t round = 2 * (int64_t)EG_ROWS * num_compute_units(), rounds = (vocab + round - 1) / round;
    if (rounds > 1) return rounds <= (dim >= 768 ? 8 : 4) && positions >= 512 * rounds ? 1 : 0;
    if (positions * (dim >= 512 ? 320 : 192) < vocab) return 0;
    const int64_t pieces = std::min<int64_t>(8, vocab) * ((dim + EG_PIECE - 1) / EG_PIECE);   // of a position in every row of a block, of vocab blocks' worth
    return positions <= 3072 ? pieces <= vocab : positions * pieces <= 1600 * vocab;
}

extern "C" int rdb_embedding_bwd(void *dweight, const void *idx, int idx_bytes, const void *dy, int64_t positions, int64_t vocab, int64_t dim, void *stream)
{
    if (positions < 0 || vocab < 0 || dim < 0) return set_error(RDB_E_SHAPE, "rdb_embedding_bwd: negative size");
    if (!embedding_fits(positions, vocab, dim))
        return set_error(RDB_E_UNSUPPORTED, "rdb_embedding_bwd: 1 to %lld positions, up to 2^29 rows and a multiple of 8 columns", (long long)EG_POSITIONS);
    if (!dweight || !idx || !dy) return set_error(RDB_E_NULL, "rdb_embedding_bwd: dweight, idx or dy is NULL");
    if (idx_bytes != 4 && idx_bytes != 8) return set_error(RDB_E_DTYPE, "rdb_embedding_bwd: indices of 4 or 8 bytes");
    if (((uintptr_t)dweight & 15) || ((uintptr_t)dy & 15) || ((uintptr_t)idx & (uintptr_t)(idx_bytes - 1)))
        return set_error(RDB_E_ALIGN, "rdb_embedding_bwd: dweight and dy must be 16-byte aligned");
    const int each = (int)((positions + EG_WAVES - 1) / EG_WAVES);
    const int64_t cus = num_compute_units(), block_rows = std::min<int64_t>(EG_ROWS, std::max<int64_t>(8, (vocab + 2 * cus - 1) / (2 * cus)));
    const size_t smem = (size_t)EG_SUMS_BYTES + (size_t)EG_WAVES * each * sizeof(uint32_t);
    auto launch = [&](auto zero) {
        typedef decltype(zero) I;
        if (int rl = reserve_lds(reinterpret_cast<const void *>(embedding_grad_kernel<I>), smem, "embedding_grad_kernel")) return rl;
        embedding_grad_kernel<I><<<(unsigned)((vocab + block_rows - 1) / block_rows), EG_THREADS, smem, (hipStream_t)stream>>>(
            static_cast<bf16_t *>(dweight), static_cast<const I *>(idx), static_cast<const bf16_t *>(dy), (int)positions, each, vocab, (int)dim, (int)block_rows);
        return check_launch("embedding_grad_kernel");
    };
    return idx_bytes == 4 ? launch((int32_t)0) : launch((int64_t)0);
}
