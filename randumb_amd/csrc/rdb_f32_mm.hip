// Kernels of rdb_f32.hpp: both sides read across their rows: dC = dy^T . z, dW = dy^T . x.
#define RDB_F32_INSTANTIATE
#include "rdb_f32.hpp"

namespace rdb {
FG_PAIR(FG_MCONT, FG_MCONT);
}  // namespace rdb
