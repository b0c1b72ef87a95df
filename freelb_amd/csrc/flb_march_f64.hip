// Instantiations of the two-step march for the f64 storage kind.
#include "flb_march.hpp"

FLB_DEFINE_MARCH(f64, StoreF64)
