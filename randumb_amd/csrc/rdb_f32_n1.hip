// Kernels of rdb_f32.hpp: the random-bias products.
#define RDB_F32_INSTANTIATE
#include "rdb_f32.hpp"

namespace rdb {
FG_PAIR(FG_KCONT, FG_NOISE_1D);
}  // namespace rdb
