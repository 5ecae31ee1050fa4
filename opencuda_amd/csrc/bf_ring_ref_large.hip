// bf_ring_ref_large.hip -- instances of the unrolled REF kernels (bf_ring.h).
#include "bf_ring.h"

namespace bfimpl {
BF_RING_LARGE(, 0)
}  // namespace bfimpl
