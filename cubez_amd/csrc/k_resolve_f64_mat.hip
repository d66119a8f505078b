// k_resolve_f64_mat.hip — the FP64 resolver kernel, kind KIND_MAT (cbz_islands.h, cbz_resolve.h).
#define CBZ_RESOLVE_INSTANTIATE
#include "cbz_islands.h"

namespace cbz {
CBZ_RESOLVE_KIND(, double, KIND_MAT)
}  // namespace cbz
