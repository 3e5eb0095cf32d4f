// The kernels of ehip_wino_ring.hpp for tile size 4 (a file each: they compile side by side).
#include "ehip_wino_ring.hpp"

namespace ehip {

RingForm wino_ring_form4(int form, int nks) { return ring_form<4>(form, nks); }

}  // namespace ehip
