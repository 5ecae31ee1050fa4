// bf_ring_std_small.hip -- instances of the unrolled STD kernels (bf_ring.h).
#include "bf_ring.h"

namespace bfimpl {
BF_RING_SMALL(, 1)
}  // namespace bfimpl
