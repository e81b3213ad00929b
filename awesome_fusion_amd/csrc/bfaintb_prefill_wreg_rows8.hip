// bfaintb_prefill_wreg_kernel over 8-bit codes in rows (one of four such files, compiled side by side).
#include "bfaintb_prefill_wreg.hpp"

namespace bfaintb {
hipError_t launch_wreg_rows8(const GemmParams& p, hipStream_t stream) { return launch_wreg_scales<8, false>(p, stream); }
}  // namespace bfaintb
