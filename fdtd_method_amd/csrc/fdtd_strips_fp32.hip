// Strip passes, FP32.
#include "fdtd_strips.hpp"

namespace fdtd::rt {
template int launch_strip<float>(fdtd_grid*, bool, bool, int, int, int, void* const*, void* const*);
template int strip_occupancy_s<float>(const BlockTuning&, int);
template const void* batch_strip_kernel<float>(int, int, int, int, bool, int, bool);
}  // namespace fdtd::rt
