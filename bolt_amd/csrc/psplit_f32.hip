// FP32-bulk instances of the two-kernel stage with p-advection.
#define BX_PSPLIT_INSTANTIATE
#include "psplit_launch.h"

namespace bx {
template int psplit_stage<float>(const StageParams&, int, int, int, void*, double*, double*, bool, hipStream_t);
template int psplit_currents<float>(const StageParams&, int, int, void*, double*, double*, hipStream_t);
template int qmarch_stage<float>(const StageParams&, int, int, void*, double*, hipStream_t);
}
