// FP32-bulk specialisations of the q1-line stage kernel.
#define BX_QL_INSTANTIATE
#include "ql_launch.h"

namespace bx {
template void ql_launch<float>(const QLParams&, bool, int, int, int, int, hipStream_t);
template int ql_blocks_per_cu<float>(int, bool, int, int, int);
}
