// pk_chain4_i8.hip - instantiates the four-deep chain tiles for W_I8 weights.
#include "pk_chain4.h"

namespace pkgpu {
namespace chain4 {

hipError_t launch_i8(int tile, const KArgs& a, hipStream_t s) { return launch<W_I8>(tile, a, s); }

}  // namespace chain4
}  // namespace pkgpu
