#include "launch.hpp"

template void bgk::eng::launch_step<double>(bgk_handle&, bool);
