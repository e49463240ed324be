// line_pass_f32.hip -- the natural-order line passes in FP32.
#include "line_pass_inst.hpp"

namespace zm {
namespace lp {

//       T     LN radix16 | rows: ept lines small mode | tiles: ept lines small mode
ZM_SPLIT(float, 4, false, 2, 4, -1, ONCE, 2, 4, -1, ONCE)
ZM_SPLIT(float, 5, false, 3, 4, -1, ONCE, 3, 4, -1, ONCE)
ZM_SPLIT(float, 6, false, 3, 4, 3, ONCE, 3, 4, 3, ONCE)
ZM_SPLIT(float, 7, false, 3, 4, 2, ONCE, 3, 4, 2, ONCE)
ZM_SPLIT(float, 8, false, 3, 3, 1, ONCE, 3, 4, 2, ONCE)
ZM_SPLIT(float, 9, false, 4, 3, 1, ONCE, 4, 4, 2, ONCE)
ZM_SPLIT(float, 10, false, 4, 2, 0, ONCE, 4, 4, 2, LOOP)
ZM_SPLIT(float, 11, false, 4, 1, 0, ONCE, 5, 3, -1, LOOP)
ZM_SPLIT(float, 12, false, 4, 0, -1, ONCE, 4, -1, -1, ONCE)
ZM_SPLIT(float, 13, false, 4, 0, -1, ONCE, 4, -1, -1, ONCE)

}  // namespace lp

template LinePassInfo line_pass_info<float>(LinePass, const LinePassSize&);
template int line_pass_occupancy<float>(LinePass, const LinePassSize&);
template hipError_t launch_line_pass<float>(LinePass, const LinePassSize&, const float2*, float2*, const LinePassArgs&, const float2*, double,
                                               const SpectralArgs&, int, hipStream_t);

}  // namespace zm
