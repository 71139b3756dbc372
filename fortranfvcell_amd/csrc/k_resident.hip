// k_resident.hip -- instantiates the on-chip PCG and BiCGSTAB (fvc_resident.h)
// for the formats and rows per thread listed in fvc_instances.h.
#define FVC_INSTANTIATE
#include "fvc_instances.h"

FVCI_FORMATS_RES(FVCI_RES, template)
