// pk_chain4_f32.hip - instantiates the four-deep chain tiles for W_F32 weights.
#include "pk_chain4.h"

namespace pkgpu {
namespace chain4 {

hipError_t launch_f32(int tile, const KArgs& a, hipStream_t s) { return launch<W_F32>(tile, a, s); }

}  // namespace chain4
}  // namespace pkgpu
