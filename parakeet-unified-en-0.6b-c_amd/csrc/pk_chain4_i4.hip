// pk_chain4_i4.hip - instantiates the four-deep chain tiles for W_I4 weights.
#include "pk_chain4.h"

namespace pkgpu {
namespace chain4 {

hipError_t launch_i4(int tile, const KArgs& a, hipStream_t s) { return launch<W_I4>(tile, a, s); }

}  // namespace chain4
}  // namespace pkgpu
