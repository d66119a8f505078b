// k_resolve_f32_plain.hip — the FP32 resolver kernel, kind KIND_PLAIN (cbz_islands.h, cbz_resolve.h).
#define CBZ_RESOLVE_INSTANTIATE
#include "cbz_islands.h"

namespace cbz {
CBZ_RESOLVE_KIND(, float, KIND_PLAIN)
}  // namespace cbz
