// Matrix-core stage kernels for cutoffs 6..8 (see mstage_impl.h).
#include "mstage_impl.h"

SFAMD_MST_DEFINE_D(6)
SFAMD_MST_DEFINE_D(7)
SFAMD_MST_DEFINE_D(8)
