// Matrix-core stage kernels for cutoffs 13..16 (see mstage_impl.h).
#include "mstage_impl.h"

SFAMD_MST_DEFINE_D(13)
SFAMD_MST_DEFINE_D(14)
SFAMD_MST_DEFINE_D(15)
SFAMD_MST_DEFINE_D(16)
