// Kernels of rdb_f32.hpp: dx = t . N, W = C . N and its transpose.
#define RDB_F32_INSTANTIATE
#include "rdb_f32.hpp"

namespace rdb {
FG_PAIR(FG_KCONT, FG_NOISE_I);
FG_PAIR(FG_NOISE_I, FG_KCONT);
}  // namespace rdb
