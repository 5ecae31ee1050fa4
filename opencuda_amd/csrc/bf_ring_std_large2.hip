// bf_ring_std_large2.hip -- instances of the unrolled STD kernels (bf_ring.h).
#include "bf_ring.h"

namespace bfimpl {
BF_RING_STD_LARGE()
}  // namespace bfimpl
