// The kernels of ehip_wino_ring.hpp for tile size 5 (a file each: they compile side by side).
#include "ehip_wino_ring.hpp"

namespace ehip {

RingForm wino_ring_form5(int form, int nks) { return ring_form<5>(form, nks); }

}  // namespace ehip
