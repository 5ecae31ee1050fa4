// bf_ring_std_large.hip -- instances of the unrolled STD kernels (bf_ring.h).
#include "bf_ring.h"

namespace bfimpl {
BF_RING_LARGE(, 1)
}  // namespace bfimpl
