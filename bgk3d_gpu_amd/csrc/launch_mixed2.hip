#include "launch.hpp"

template void bgk::eng::launch_step<mix32_t>(bgk_handle&, bool);
