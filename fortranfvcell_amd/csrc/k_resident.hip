// k_resident.hip -- instantiates the on-chip PCG, BiCGSTAB, mixed PCG and GMRES
// and the batches of PCG and mixed PCG (fvc_resident.h) for the formats and rows
// per thread listed in fvc_instances.h.
#define FVC_INSTANTIATE
#include "fvc_instances.h"

FVCI_FORMATS_RES(FVCI_RES, template)
