// The EXACT kernels of the plane stages by row residue (pf_resid.hip), in a
// translation unit of their own.
#include "pf_resid_kern.h"

namespace pf {

int dispatch_resid_exact(const Fft3D& f, const FusedArgs& a, const ResSplit& sp, int which,
                         int nplanes, int zr, hipStream_t s) {
    return dispatch_resid<true>(f, a, sp, which, nplanes, zr, s);
}

}  // namespace pf
