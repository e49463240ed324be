// line_pass_f64.hip -- the natural-order line passes in FP64.
#include "line_pass_inst.hpp"

namespace zm {
namespace lp {

//       T      LN radix16 | rows: ept lines small mode | tiles: ept lines small mode
ZM_SPLIT(double, 4, false, 2, 4, -1, ONCE, 2, 4, -1, ONCE)
ZM_SPLIT(double, 5, false, 3, 4, -1, ONCE, 3, 4, -1, ONCE)
ZM_SPLIT(double, 6, false, 3, 4, 3, ONCE, 3, 4, 3, ONCE)
ZM_SPLIT(double, 7, false, 3, 4, 2, ONCE, 3, 4, 2, ONCE)
ZM_SPLIT(double, 8, false, 3, 3, 1, ONCE, 3, 4, 2, ONCE)
ZM_SPLIT(double, 8, true, 4, 3, 2, ONCE, 4, 4, 2, ONCE)
ZM_SPLIT(double, 9, false, 3, 3, 1, ONCE, 4, 3, 1, ONCE)
ZM_SPLIT(double, 10, false, 4, 1, 0, ONCE, 4, 3, 2, LOOP)
ZM_SPLIT(double, 11, false, 4, 1, 0, LOOP, 4, 2, -1, LOOP)
ZM_SPLIT(double, 12, false, 4, 0, -1, ONCE, 4, -1, -1, ONCE)
ZM_SPLIT(double, 13, false, 4, 0, -1, ONCE, 4, -1, -1, ONCE)

}  // namespace lp

template LinePassInfo line_pass_info<double>(LinePass, const LinePassSize&);
template int line_pass_occupancy<double>(LinePass, const LinePassSize&);
template hipError_t launch_line_pass<double>(LinePass, const LinePassSize&, const double2*, double2*, const LinePassArgs&, const double2*, double,
                                                const SpectralArgs&, int, hipStream_t);

}  // namespace zm
