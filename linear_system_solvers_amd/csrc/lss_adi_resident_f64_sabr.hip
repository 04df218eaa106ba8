// Resident ADI loop (double, sabr coefficient pattern); the kernel is in lss_adi_resident.hpp.
#include "lss_adi_resident.hpp"

LSS_INST_RES(double, 2)
