// Matrix-core stage kernels for cutoffs 17..20 (see mstage_impl.h).
#include "mstage_impl.h"

SFAMD_MST_DEFINE_D(17)
SFAMD_MST_DEFINE_D(18)
SFAMD_MST_DEFINE_D(19)
SFAMD_MST_DEFINE_D(20)
