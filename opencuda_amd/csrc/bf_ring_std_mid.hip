// bf_ring_std_mid.hip -- instances of the unrolled STD kernels (bf_ring.h).
#include "bf_ring.h"

namespace bfimpl {
BF_RING_MID(, 1)
}  // namespace bfimpl
