// Matrix-core stage kernels for cutoffs 2..5 (see mstage_impl.h).
#include "mstage_impl.h"

SFAMD_MST_DEFINE_D(2)
SFAMD_MST_DEFINE_D(3)
SFAMD_MST_DEFINE_D(4)
SFAMD_MST_DEFINE_D(5)
