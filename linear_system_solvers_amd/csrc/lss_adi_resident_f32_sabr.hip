// Resident ADI loop (float, sabr coefficient pattern); the kernel is in lss_adi_resident.hpp.
#include "lss_adi_resident.hpp"

LSS_INST_RES(float, 2)
