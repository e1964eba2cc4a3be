// Strip passes, FP64.
#include "fdtd_strips.hpp"

namespace fdtd::rt {
template int launch_strip<double>(fdtd_grid*, bool, bool, int, int, int, void* const*, void* const*);
template int strip_occupancy_s<double>(const BlockTuning&, int);
template const void* batch_strip_kernel<double>(int, int, int, int, bool, int, bool);
}  // namespace fdtd::rt
