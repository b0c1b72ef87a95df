// Instantiations of the two-step march for the f32 storage kind.
#include "flb_march.hpp"

FLB_DEFINE_MARCH(f32, StoreF32)
