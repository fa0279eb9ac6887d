// Prefill GEMM instances (prefill_tile.h).
#define LF_PREFILL_Z_KERNEL  // (the z producers' own launch lives in this unit)
#include "prefill_tile.h"

namespace lf::prefill {
template int launch_rows<8>(const PrefillParams&, int64_t, bool, bool, hipStream_t);
}  // namespace lf::prefill
