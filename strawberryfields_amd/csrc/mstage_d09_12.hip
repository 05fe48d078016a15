// Matrix-core stage kernels for cutoffs 9..12 (see mstage_impl.h).
#include "mstage_impl.h"

SFAMD_MST_DEFINE_D(9)
SFAMD_MST_DEFINE_D(10)
SFAMD_MST_DEFINE_D(11)
SFAMD_MST_DEFINE_D(12)
