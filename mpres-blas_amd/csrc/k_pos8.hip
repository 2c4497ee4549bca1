// Kernel instantiation: positional reduction chains, 8 moduli.
#include "launch_pos.hpp"

MPH_INSTANTIATE_POS(8)
