#include "launch.hpp"

template void bgk::eng::launch_step<float>(bgk_handle&, bool);
