// Kernels of rdb_f32.hpp: B read across its rows: t = dy . C, dx = dy . W.
#define RDB_F32_INSTANTIATE
#include "rdb_f32.hpp"

namespace rdb {
FG_PAIR(FG_KCONT, FG_MCONT);
}  // namespace rdb
