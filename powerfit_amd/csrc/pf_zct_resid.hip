// The register z stage with the residues' part of the y transform
// (pf_resid.hip, pf_zct_kern.h), one kernel per z length and kind of residue
// transform.
#include "pf_zct_kern.h"

namespace pf {

namespace {

// Register plan: one per length.  The alternative (at most 8 slots) where the
// default has one or two threads a column (as the plain z stage), where it has 14
// or 15 slots over 8 threads and the alternative 16 threads (z 70: 2.71 against
// 2.60 us per rotation, 75: 4.21 against 3.79, 84: 4.84 against 4.40; not so at 16
// slots, 112: 6.7 against 12.1), and where the general sums over residues spill at
// 16 slots (120 x 150 x 210: 49.6 against 29.5).
template <int L, int RES>
constexpr bool res_alt() {
    using D = ZF<L, kFlexZSlots>;
    if constexpr (!flex_zalt_ok(L)) {
        return false;
    } else {
        return D::T <= 2 ||
               ((D::E == 14 || D::E == 15) && D::T == 8 && ZF<L, kFlexZSlotsAlt>::T == 16) ||
               (RES == 3 && D::E == 16);
    }
}

template <int L, int RES>
int launch_res(const Fft3D& f, const FusedArgs& a, int zr, hipStream_t s) {
    return launch_zct_kernel<L, res_alt<L, RES>() ? kFlexZSlotsAlt : kFlexZSlots, RES>(f, a, zr, s);
}

}  // namespace

int launch_zcorr_resid(const Fft3D& f, const FusedArgs& a, int zr, hipStream_t s) {
    switch (f.nz) {
#define PF_ZCASE(L)                                                 \
    case L:                                                         \
        if (a.rmap.rb == 2) return launch_res<L, 2>(f, a, zr, s);   \
        if (a.rmap.rb == 4) return launch_res<L, 4>(f, a, zr, s);   \
        return launch_res<L, 3>(f, a, zr, s);
        PF_CT_COL_LENGTHS(PF_ZCASE)
#undef PF_ZCASE
        default:
            set_error("z stage: no compiled transform for length %d", f.nz);
            return kErrUnsupported;
    }
}

}  // namespace pf
