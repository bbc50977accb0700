// z stage of the run-time planned fused pipeline with the z length fixed at
// compile time (one kernel per 2,3,5,7-smooth length from 16 to 256; other
// lengths use the LDS-planned k_zcorr_rt in pf_planes.hip).
//
// k_zcorr_ct: one block per (tile of TQ (ky,kx) columns, rotation chunk); the
// column's L points live in the registers of T threads (pf_ct_fft.h Flex).
// Per rotation: forward z FFT of the P and W (and W^2) xy-spectra, the
// products conj(X) F1 / conj(X) F2 with the F tiles held in registers for the
// whole chunk, inverse z FFT, written back in place.  The forward transform
// leaves each thread holding exactly the elements the inverse starts from, so
// product and inverse need no exchange; each transform exchanges through LDS
// once per stage boundary.
//
// Bound by HBM: s d + 3 half spectra per rotation (s forward grids, d the share
// of planes in the support).  The columns of the next transform are loaded while
// the current one runs; addresses are one 32-bit offset per slot into a buffer
// resource, whose bounds check also supplies the zeros of idle slots and of planes
// beyond the support; blocks of neighbouring tiles share an XCD.  With padded
// planes (WorkLayout) 120^3 takes 6.6 us per rotation (9.4 before: 64-bit
// addresses, loads waited for, packed planes), 75 x 81 x 105 2.9 (4.0),
// 70 x 72 x 98 2.0 (2.3), 216 x 225 x 240 61 (88).
#include "pf_zct_kern.h"

namespace pf {

bool zcorr_ct_supported(int nz) {
    switch (nz) {
#define PF_ZCASE(L) case L:
        PF_CT_COL_LENGTHS(PF_ZCASE)
#undef PF_ZCASE
        return true;
        default: return false;
    }
}

int launch_zcorr_ct(const Fft3D& f, const FusedArgs& a, int zr, hipStream_t s) {
    if (a.nrot <= 0) return kOk;
    if (a.nrot > 65535 || a.chunk_z < 1) {
        set_error("z stage: invalid batch or chunk size");
        return kErrArg;
    }
    if (a.rmap.rb > 1) return launch_zcorr_resid(f, a, zr, s);
    // schedule bit 0: the alternative register plan where the length has one,
    // which is also the default's where that has one or two threads a column
    // (blocks of a wavefront or less; z length 16 0.52 against 0.31 us per
    // rotation, 24 0.76 against 0.67, 30 0.97 against 0.83)
    const bool alt = a.zsched & 1;
    switch (f.nz) {
#define PF_ZCASE(L)                                                          \
    case L:                                                                  \
        if constexpr (flex_zalt_ok(L))                                       \
            if (alt || ZF<L, kFlexZSlots>::T <= 2)                           \
                return launch_zct_kernel<L, kFlexZSlotsAlt, 0>(f, a, zr, s);      \
        return launch_zct_kernel<L, kFlexZSlots, 0>(f, a, zr, s);
        PF_CT_COL_LENGTHS(PF_ZCASE)
#undef PF_ZCASE
        default:
            set_error("z stage: no compiled transform for length %d", f.nz);
            return kErrUnsupported;
    }
}

}  // namespace pf
