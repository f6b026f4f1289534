#include "launch.hpp"

template void bgk::eng::launch_step<bf16_t>(bgk_handle&, bool);
