// Prefill GEMM instances (prefill_tile.h).
#include "prefill_tile.h"

namespace lf::prefill {
template int launch_rows<4>(const PrefillParams&, int64_t, bool, bool, hipStream_t);
template int launch_rows<3>(const PrefillParams&, int64_t, bool, bool, hipStream_t);
}  // namespace lf::prefill
