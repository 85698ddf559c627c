// Middle passes (c64) of the Bluestein chains beyond LDS.
#include "inst.hpp"

AFFT_POW2_SMALL(float, ::afft::VAR_BLUEMID)
AFFT_POW2_16K(float, ::afft::VAR_BLUEMID)
