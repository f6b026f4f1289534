#include "launch.hpp"

template void bgk::eng::launch_step<f16r_t>(bgk_handle&, bool);
