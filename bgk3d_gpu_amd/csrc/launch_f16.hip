#include "launch.hpp"

template void bgk::eng::launch_step<f16_t>(bgk_handle&, bool);
