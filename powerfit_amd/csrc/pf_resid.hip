// Plane stages of the run-time planned pipeline by row residue.
//
// With ny = RA RB, the rows y = RB a + b of one residue b (RA of them) go
// through the y transform's first RA-point part by themselves, and the other
// part, RB-point transforms over the residues, joins the z stage
// (pf_zct.hip), where the residues of a column sit in neighbouring lanes:
//
//   X[ka + RA kb] = sum_b w_RB^(b kb) w_ny^(b ka) sum_a x[RB a + b] w_RA^(a ka)
//
// and the same backwards.  So a block of the plane stages holds RA rows instead
// of a plane, of all grids at once: a few small blocks per compute unit whose
// barriers overlap, in place of one that fills its LDS.
//
//   k_fwd_resid  block per (plane, residue, rotation): gathers the rotated
//                template and mask of the rows, x transforms, RA-point y
//                transforms and twiddles of P, W (and W^2) together;
//   k_inv_resid  block per (plane, residue, rotation chunk): RA-point inverse y
//                and inverse x transforms of B, A and G together, the LCC in the
//                registers of the last x stage, and the running best of the
//                chunk in registers, merged with one atomicMax per improved voxel.
//
// Per rotation, forward / z / inverse stage, against the plane kernels
// (k_fwd_plane_rt, k_inv_plane_rt): 120^3 4.7 / 7.4 / 8.9 us (7.9 / 6.6 / 15.5),
// 75 x 81 x 105 1.8 / 3.6 / 3.2 (3.9 / 2.9 / 8.8), 70 x 72 x 98 1.4 / 2.5 / 2.6
// (2.4 / 2.0 / 4.9), 32^3 0.64 / 0.39 / 0.54 at 24 rotations (1.23 / 0.44 / 1.6).
// The plane kernels spend their time at barriers: fifteen a rotation, behind one or
// two blocks a unit; here five, behind two to four, and vector arithmetic issues
// two thirds of the time (120^3).
//
// Work layout (ResidMap): 16 columns of the z stage are one 128-byte line: TK =
// 16 / RB kx of each of the RB residues, [z][ka][kx / TK][b][kx % TK].  (With the
// residues innermost the z stage's exchanges are cheaper, but single complex
// numbers at a distance cost the plane stages more: 120^3 inverse 8.8 -> 9.4 us.)
#include "pf_resid_kern.h"

namespace pf {

namespace {

constexpr bool res_row_length(int nx) {
#define PF_XCASE(L) case L:
    if (nx % 2) {
        switch (nx) {
            PF_CT_ODD_LENGTHS(PF_XCASE)
            return true;
            default: return false;
        }
    }
    switch (nx / 2) {
        PF_CT_ROW_LENGTHS(PF_XCASE)
        return true;
        default: return false;
    }
#undef PF_XCASE
}

// Residues 1, 2, 4 (cross-lane steps in the z stage are single instructions),
// 3, 5: the first whose rows of three grids take at most lds_max bytes.  The z
// stage pays for residues (z length 60: 1.25, 1.45 and 1.7 us with 1, 2 and 4), the
// plane stages for large blocks.
ResSplit res_split(int ny, int nx, size_t lds_max) {
    const bool odd = nx % 2;
    const int rl = odd ? nx : nx / 2, nxh = nx / 2 + 1;
    const ResPlan xp = res_plan(rl);
    if (!xp.ns) return {};
    for (int rb : {1, 2, 4, 3, 5}) {
        if (ny % rb) continue;
        const int ra = ny / rb;
        if (res_lds(rl, odd, ra, 3) > lds_max) continue;
        // balanced radices (at most 10 and 8), the larger one first; one up to 8
        int r1 = 0, r2 = 0;
        for (int a = 2; a <= 10; ++a)
            if (ra % a == 0 && ra / a <= a && (ra / a > 1 ? ra / a <= 8 : a <= 8) && !r1) {
                r1 = a;
                r2 = ra / a;
            }
        if (!r1) continue;
        const int nrow = odd ? (ra + 1) / 2 : ra, rz = xp.r[xp.ns - 1];
        const int own = nrow * (rl / rz);          // items of the last x stage: one a thread
        int best = 0;
        int64_t best_cost = 0;
        // (wavefronts in multiples of the SIMDs: 320 threads against 256 at 75 x 81 x
        // 105 took 5.2 for 3.6 us)
        for (int n = 256; n <= kResThreads; n += 256) {
            // (k_fwd_resid holds two columns a thread)
            if (own > n || (odd ? r2 * nxh > 2 * n : r2 * (rl / 2 + 1) > n)) continue;
            // lanes x (work + a fixed charge) of every pass of k_inv_resid
            auto pass = [&](int64_t items, int work) { return (items + n - 1) / n * n * (work + 6); };
            int64_t cost = pass(3 * r2 * nxh, r1) + pass(own, 3 * rz + 2 * rz);
            if (r2 > 1) cost += pass(3 * r1 * nxh, r2);
            for (int s = 0; s + 1 < xp.ns; ++s) {
                const int nb = rl / xp.r[s], per = n / nb;
                cost += (int64_t)((3 * nrow + per - 1) / per) * n * (2 * xp.r[s] + 6);
            }
            if (!best || cost < best_cost) {
                best = n;
                best_cost = cost;
            }
        }
        if (best) return {rb, r1, r2, best};
    }
    return {};
}

ResSplit res_choose(int ny, int nx) {
    // three blocks a compute unit, else two
    ResSplit s = res_split(ny, nx, 52 * 1024);
    return s.rb ? s : res_split(ny, nx, 78 * 1024);
}

}  // namespace

ResidMap resid_map(int nz, int ny, int nx) {
    ResidMap m{};
    if (nz < 2 || ny < 2 || nx < 3 || !zcorr_ct_supported(nz) || !res_row_length(nx)) return m;
    // (spectra of at most 256 x 256 rows, voxels in 32-bit indices)
    if (ny > 256) return m;
    const ResSplit s = res_choose(ny, nx);
    if (!s.rb) return m;
    m.rb = s.rb;
    m.ra = ny / s.rb;
    m.tk = 16 / s.rb;
    m.magic = (65536 + m.tk - 1) / m.tk;
    m.nkg = (nx / 2 + 1 + m.tk - 1) / m.tk;
    m.rp = s.rb == 1 ? nx / 2 + 1 : 16 * m.nkg;
    // whole lines, an odd number of them a plane (WorkLayout)
    const int lines = (m.ra * m.rp + 15) / 16;
    m.ps = (lines | 1) * 16;
    return m;
}

int launch_resid_stage(const Fft3D& f, const FusedArgs& a, int which, hipStream_t s) {
    if (a.nrot <= 0) return kOk;
    if (a.rmap.rb == 0) {
        set_error("residue stages not available for grid (%d, %d, %d)", f.nz, f.ny, f.nx);
        return kErrUnsupported;
    }
    if (a.nrot > 65535 || a.chunk_z < 1 || a.chunk_lcc < 1) {
        set_error("fused: invalid batch or chunk sizes");
        return kErrArg;
    }
    // planes |z| <= zr only (rotation sphere and support), the z stage reading
    // the others as zero
    const int zr = std::max(0, std::min(std::min(a.zr, a.rmax), f.nz / 2));
    const int nplanes = std::min(2 * zr + 1, f.nz);
    if (which == 1) return launch_zcorr_ct(f, a, nplanes < f.nz ? zr : f.nz, s);
    const ResSplit sp = res_choose(f.ny, f.nx);
    if (a.exact) return dispatch_resid_exact(f, a, sp, which, nplanes, zr, s);
    return dispatch_resid<false>(f, a, sp, which, nplanes, zr, s);
}

int prepare_resid(int nx) {
    Fft3D f{};
    f.nx = nx;
    PF_CHECK_STATUS(dispatch_resid<false>(f, {}, {}, -1, 0, 0, nullptr));
    return dispatch_resid_exact(f, {}, {}, -1, 0, 0, nullptr);
}

}  // namespace pf
