// Strip passes, FP16 storage.
#include "fdtd_strips.hpp"

namespace fdtd::rt {
template int launch_strip<_Float16>(fdtd_grid*, bool, bool, int, int, int, void* const*, void* const*);
template int strip_occupancy_s<_Float16>(const BlockTuning&, int);
template const void* batch_strip_kernel<_Float16>(int, int, int, int, bool, int, bool);
}  // namespace fdtd::rt
