// lutgemm_mx_kernel.h making its rows itself: its variants, one per tile height (kMxExpandUnits).
#include "lutgemm_mx_kernel.h"

namespace axc {

hipError_t launch_dense_mx_expand(const MxParams &p, hipStream_t stream)
{
    switch (p.plan.units) {
    case 2: return launch_mx_units<2, true>(p, stream);
    case 3: return launch_mx_units<3, true>(p, stream);
    case 4: return launch_mx_units<4, true>(p, stream);
    case 6: return launch_mx_units<6, true>(p, stream);
    case 8: return launch_mx_units<8, true>(p, stream);
    case 10: return launch_mx_units<10, true>(p, stream);
    case 12: return launch_mx_units<12, true>(p, stream);
    case 13: return launch_mx_units<13, true>(p, stream);
    case 14: return launch_mx_units<14, true>(p, stream);
    case 16: return launch_mx_units<16, true>(p, stream);
    case 18: return launch_mx_units<18, true>(p, stream);
    }
    return hipErrorInvalidValue;
}

} // namespace axc
