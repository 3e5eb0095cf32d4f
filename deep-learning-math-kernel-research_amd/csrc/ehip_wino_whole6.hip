// The kernels of ehip_wino_whole.hpp for tile size 6 (a file each: they compile side by side).
#include "ehip_wino_whole.hpp"

namespace ehip {

WholeForm wino_whole_form6(int nks, int nw, int out_type, bool sum) { return whole_form<6>(nks, nw, out_type, sum); }

}  // namespace ehip
