// Which of the four builds of bfaintb_prefill_wreg_kernel (bfaintb_prefill_wreg.hpp) serves a launch.
#include "bfaintb_device.hpp"

namespace bfaintb {

hipError_t launch_wreg_rows8(const GemmParams& p, hipStream_t stream);
hipError_t launch_wreg_rows4(const GemmParams& p, hipStream_t stream);
hipError_t launch_wreg_packed8(const GemmParams& p, hipStream_t stream);
hipError_t launch_wreg_packed4(const GemmParams& p, hipStream_t stream);

// Whether that kernel can serve a launch: this library's own arithmetic (either order of the weights).
bool prefill_wreg_serves(const GemmParams& p) { return !p.reference_arith; }

// packed: p.b is the buffer in the packed order (p.ldb_bytes is unused)
hipError_t launch_prefill_wreg(const GemmParams& p, int bits, bool packed, hipStream_t stream)
{
    if (packed) return bits == 8 ? launch_wreg_packed8(p, stream) : launch_wreg_packed4(p, stream);
    return bits == 8 ? launch_wreg_rows8(p, stream) : launch_wreg_rows4(p, stream);
}

}  // namespace bfaintb
