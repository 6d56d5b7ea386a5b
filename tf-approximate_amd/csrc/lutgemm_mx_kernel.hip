// lutgemm_mx_kernel.h out of pre-expanded rows: its variants, one per tile height.
#include "lutgemm_mx_kernel.h"

namespace axc {

hipError_t launch_dense_mx(const MxParams &p, hipStream_t stream)
{
    switch (p.plan.units) {
    case 2: return launch_mx_units<2, false>(p, stream);
    case 3: return launch_mx_units<3, false>(p, stream);
    case 4: return launch_mx_units<4, false>(p, stream);
    case 6: return launch_mx_units<6, false>(p, stream);
    case 8: return launch_mx_units<8, false>(p, stream);
    case 10: return launch_mx_units<10, false>(p, stream);
    case 13: return launch_mx_units<13, false>(p, stream);
    case 16: return launch_mx_units<16, false>(p, stream);
    case 20: return launch_mx_units<20, false>(p, stream);
    case 25: return launch_mx_units<25, false>(p, stream);
    }
    return hipErrorInvalidValue;
}

} // namespace axc
