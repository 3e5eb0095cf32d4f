// The kernels of ehip_wino_ring.hpp for tile size 6 (a file each: they compile side by side).
#include "ehip_wino_ring.hpp"

namespace ehip {

RingForm wino_ring_form6(int form, int nks) { return ring_form<6>(form, nks); }

}  // namespace ehip
