// Kernels of rdb_f32.hpp: z = x . N^T, dcoef = dW . N^T.
#define RDB_F32_INSTANTIATE
#include "rdb_f32.hpp"

namespace rdb {
FG_PAIR(FG_KCONT, FG_NOISE_M);
}  // namespace rdb
