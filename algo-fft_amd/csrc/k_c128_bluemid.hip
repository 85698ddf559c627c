// Middle passes (c128) of the Bluestein chains beyond LDS.
#include "inst.hpp"

AFFT_POW2_SMALL(double, ::afft::VAR_BLUEMID)
