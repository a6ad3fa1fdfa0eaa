// Kernels of rdb_f32.hpp: both sides read along their rows: y = z . C^T, y = x . W^T.
#define RDB_F32_INSTANTIATE
#include "rdb_f32.hpp"

namespace rdb {
FG_PAIR(FG_KCONT, FG_KCONT);
}  // namespace rdb
