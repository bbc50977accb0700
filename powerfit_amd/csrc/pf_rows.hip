// Row and column stages of the LCC search for grids whose z-planes do not fit
// the plane kernels' LDS or voxels-per-thread limits (pf_fused.hip,
// pf_planes.hip) nor split into residues that do (pf_resid.hip): any grid whose y and z lengths have a compiled register
// transform (pf_ct_fft.h), e.g. 216 x 225 x 240.
//
// Five kernels per batch of rotations, all on the half spectra of the work
// buffer ([rotation][3][z][y][kx], WorkLayout):
//
//   k_rows_fwd   block per (rows of one plane, rotation): gathers the rotated
//                template and mask of the rows and runs their x transforms
//                (P, W and, for weighted masks, W^2 together);
//   k_cols<-1>   block per (16 kx columns of one plane, rotation): y transform
//                with the columns in registers;
//   k_zcorr_ct   the z stage of the run-time planned pipeline (pf_zct.hip);
//   k_cols<1>    inverse y transform of the three correlation spectra;
//   k_rows_inv   block per (rows of one plane, rotation chunk): inverse x
//                transforms of B, A and G of the rows together, the LCC, and
//                the running best of the chunk in registers.
//
// Only rows and planes that the rotated template can reach are gathered,
// written and read in the forward half.  Bound by HBM: per rotation the
// stages move (in half spectra of 8 H bytes, s forward grids, f the share of
// live rows, d of live planes) s f + s (f + d) + (s d + 3) + 6 + 3, against
// about 50 for the unfused kernels.  Measured per rotation at 216 x 225 x 240,
// 0/1 mask: forward rows 32 us, columns 24 us, z 57 us (88 before its
// loads ran ahead), inverse columns 64 us
// (4.4 TB/s), inverse rows 50 us, against 1,318 us unfused; 150 x 168 x 180
// core-weighted 93 against 370 us.  The row kernels are compiled per row
// length: with one switch over all lengths in the kernel the inverse rows
// took 248 registers (or spilled 500) and 176-220 us.
#include <algorithm>

#include "pf_planes_kern.h"

namespace pf {

namespace {

constexpr int kRowThreads = 256;   // largest block of the row kernels
constexpr int kRowVox = 8;         // voxels a thread of k_rows_inv owns, at most
constexpr int kRowMax = 32;        // rows per block, at most
constexpr int kRowPairs = 7;       // input pairs a thread of k_rows_inv loads, at most
constexpr size_t kRowLds = 60 * 1024;
constexpr int kColTmax = 32;       // threads per column of k_cols
constexpr int kColTq = 16;         // columns per block

// Rows of the x transform in one block: `rpb` rows (a power of two, lg its
// logarithm) of rl points of each of `ng` grids, twice (ping-pong), and the
// twiddles.
constexpr size_t row_lds_bytes(int rl, bool odd, int rpb, int ng) {
    return sizeof(float2) * ((size_t)2 * ng * rpb * rl + rl + (odd ? 0 : 2 * rl));
}

// log2 of the rows per block: the most (up to kRowMax) whose LDS leaves several
// blocks per compute unit and whose voxels and input pairs fit the threads'
// slots; -1 when none do.
constexpr int row_log(int rl, bool odd, int ng) {
    const int pairs = rl / 2 + 1;   // of one packed row or half-length row
    int lg = -1;
    for (int l = 0; (1 << l) <= kRowMax; ++l)
        if (row_lds_bytes(rl, odd, 1 << l, ng) <= kRowLds &&
            (int64_t)2 * (1 << l) * rl <= (int64_t)kRowVox * kRowThreads &&
            (int64_t)3 * (1 << l) * pairs <= (int64_t)kRowPairs * kRowThreads)
            lg = l;
    return lg;
}

// nfft transforms of a block's rows: the pass of length RL, or (RL = 0) the
// run-time planned one.
template <int DIR, int RL>
__device__ __forceinline__ float2* rows_fft(float2* a, float2* b, const PlanRt& p,
                                            const float2* tw, int nfft, int rl) {
    if constexpr (RL > 0) return ct_run<RL, DIR, false>(a, b, nfft, RL, tw);
    else return lds_fft_rt<DIR>(a, b, p, tw, nfft, rl, 1);
}

// Forward x transforms of rows [row0, row0 + rpb) (packed rows for odd nx) of
// one plane, ng grids at once.  rg2: squared radius of the voxels gathered;
// rows wholly outside it are zero and are neither transformed nor written.
template <bool ODD, int RL>
__global__ __launch_bounds__(kRowThreads) void k_rows_fwd(
    const float2* __restrict__ tm, const uint32_t* __restrict__ occ,
    const double* __restrict__ rots, RtGeo g, int r, int rg2, int zlo, int nplanes, int ng, int lgr,
    float2* __restrict__ out, PlanRt px, const float2* __restrict__ twx_g,
    const float2* __restrict__ twf_g) {
    extern __shared__ float2 lds[];
    const int rl = RL > 0 ? RL : g.rl;
    const int rpb = 1 << lgr, tile = rpb * rl;
    float2* const A = lds;
    float2* const B = lds + ng * tile;
    float2* const twx = B + ng * tile;
    float2* const twfull = twx + rl;
    // neighbouring rows and planes of a rotation on one XCD: they gather from
    // neighbouring parts of the template
    const int nblk = (g.nr + rpb - 1) / rpb;
    const int blk = xcd_order(blockIdx.x, gridDim.x);
    const int pl = blk / nblk, b = pl / nplanes;
    const int iz = (pl - b * nplanes + zlo + g.nz) % g.nz;
    const int sz = scoord(iz, r, g.nz);
    const int row0 = (blk - pl * nblk) * rpb, nrow = min(rpb, g.nr - row0);
    // a row of the grid holds a voxel of the sphere
    auto live = [&](int y) -> bool {
        const int sy = scoord(y, r, g.ny);
        return y < g.ny && sz * sz + sy * sy <= rg2;
    };
    {
        bool any = false;
        for (int f = 0; f < nrow; ++f)
            any |= ODD ? live(2 * (row0 + f)) || live(2 * (row0 + f) + 1) : live(row0 + f);
        if (!any) return;   // uniform over the block
    }
    stage_tw(twx, twx_g, rl);
    if (!ODD) stage_tw(twfull, twf_g, 2 * rl);
    double R[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) R[i] = rots[9 * b + i];
    {
        Step2 it(rl);
        for (int u = threadIdx.x; u < tile; u += blockDim.x, it.next()) {
            // even nx: voxels (y, 2m), (y, 2m + 1); odd nx: (2p, x), (2p + 1, x)
            const int row = row0 + it.r;
            float2 p2 = c2(0.f, 0.f), w2 = c2(0.f, 0.f);
            if (it.r < nrow) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int y = ODD ? 2 * row + h : row;
                    const int sy = scoord(y, r, g.ny);
                    const int sx = scoord(ODD ? it.c : 2 * it.c + h, r, ODD ? rl : 2 * rl);
                    float p = 0.f, w = 0.f;
                    if (y < g.ny && sz * sz + sy * sy + sx * sx <= rg2)
                        gather_pw_f64(tm, occ, g.nz, g.ny, g.nx, R, sz, sy, sx, &p, &w);
                    if (h) {
                        p2.y = p;
                        w2.y = w;
                    } else {
                        p2.x = p;
                        w2.x = w;
                    }
                }
            }
            A[u] = p2;
            A[tile + u] = w2;
            if (ng == 3) A[2 * tile + u] = c2(w2.x * w2.x, w2.y * w2.y);
        }
    }
    __syncthreads();
    const float2* Z = rows_fft<-1, RL>(A, B, px, twx, ng * rpb, rl);
    // R2C post-processing on the way out (as k_fwd_plane_rt)
    float2* const dst = out + (int64_t)b * 3 * g.H + (int64_t)iz * g.ps;
    const int M = rl, nx = ODD ? rl : 2 * rl, nxh = nx / 2 + 1;
    const int orow = ODD ? 2 * rpb : rpb, y0 = ODD ? 2 * row0 : row0;
    for (int gi = 0; gi < ng; ++gi) {
        const float2* zg = Z + gi * tile;
        float2* const o = dst + (int64_t)gi * g.H;
        Step2 ip(nxh);
        for (int u = threadIdx.x; u < orow * nxh; u += blockDim.x, ip.next()) {
            const int k = ip.c;
            if (!live(y0 + ip.r)) continue;
            float2 X;
            if constexpr (!ODD) {
                const float2* z = zg + ip.r * M;
                if (k == 0 || k == M) {
                    const float2 z0 = z[0];
                    X = c2(k == 0 ? z0.x + z0.y : z0.x - z0.y, 0.f);
                } else {
                    const float2 zk = z[k], zm = cconj(z[M - k]);
                    const float2 E = cscale(cadd(zk, zm), 0.5f);
                    const float2 O = mul_si<-1>(cscale(csub(zk, zm), 0.5f));
                    X = cadd(E, cmul(twfull[k], O));
                }
            } else {
                const float2* z = zg + (ip.r >> 1) * nx;
                const float2 zk = z[k], zm = cconj(z[k ? nx - k : 0]);
                X = (ip.r & 1) ? mul_si<-1>(cscale(csub(zk, zm), 0.5f))
                               : cscale(cadd(zk, zm), 0.5f);
            }
            o[(y0 + ip.r) * g.rp + k] = X;
        }
    }
}

// In-place y transforms of 16 kx columns of one plane, ng grids in turn, each
// column in the registers of T threads.  Forward (DIR -1): rows outside the
// sphere (rg2) were not written by k_rows_fwd and are zero.
template <int L, int DIR>
__global__ __launch_bounds__((kColTq * Flex<L, kFlexZSlots, kColTmax, false, true>::T)) void k_cols(
    float2* __restrict__ X, int nz, int nxh, int rp, int ps, int nplanes, int nrot, int ng, int r,
    int rg2, int zlo, const float2* __restrict__ tw) {
    using FX = Flex<L, kFlexZSlots, kColTmax, false, true>;
    constexpr int T = FX::T, E = FX::E;
    __shared__ float2 ex[L * kColTq];
    __shared__ float2 stw[L];
    for (int i = threadIdx.x; i < L; i += blockDim.x) stw[i] = tw[i];
    __syncthreads();
    const int c = threadIdx.x % kColTq, t = threadIdx.x / kColTq;
    // blocks of neighbouring tiles and planes on one XCD: rows of nxh complex
    // are not multiples of a cache line, so neighbouring tiles share lines
    const int ntiles = (nxh + kColTq - 1) / kColTq;
    const int blk = xcd_order(blockIdx.x, ntiles * nplanes * nrot);
    const int pl = blk / ntiles, b = pl / nplanes;
    const int q = (blk - pl * ntiles) * kColTq + c;
    const bool active = q < nxh;
    const int iz = (pl - b * nplanes + zlo + nz) % nz;
    const int sz = scoord(iz, r, nz);
    const int lim = rg2 - sz * sz;
    const int64_t H = (int64_t)nz * ps;
    float2* col = X + (int64_t)b * 3 * H + (int64_t)iz * ps + q;
    for (int gi = 0; gi < ng; ++gi, col += H) {
        float2 v[E];
#pragma unroll
        for (int s = 0; s < E; ++s) v[s] = c2(0.f, 0.f);
#pragma unroll
        for (int s = 0; s < FX::in_slots(); ++s) {
            const int p = FX::in_pos(t, s);
            bool ok = active && p >= 0;
            if (DIR < 0) {
                const int sy = scoord(p, r, L);
                ok = ok && sy * sy <= lim;
            }
            if (ok) v[s] = col[p * rp];
        }
        flex_fft<L, kFlexZSlots, kColTmax, false, DIR, true>(v, ex + c, kColTq, t, stw, active);
        if (active) {
#pragma unroll
            for (int s = 0; s < FX::out_slots(); ++s) {
                const int p = FX::out_pos(t, s);
                if (p >= 0) col[p * rp] = v[s];
            }
        }
    }
}

// Inverse x transforms of rows [row0, row0 + rpb) of one plane for B, A and G
// of each rotation of the chunk, and the LCC.  Thread t owns voxels u = t + j
// blockDim of the block's rows (odd nx: float u of the packed rows) and holds
// their best (score, index) over the chunk, starting from the stored result,
// which it replaces with one atomicMax per improved voxel.  The score decides
// in FP32; a score within a few roundings of the best, or above it, is formed
// in FP64 as the unfused kernel does.
template <bool ODD, int RL>
__global__ __launch_bounds__(kRowThreads) void k_rows_inv(
    const float2* __restrict__ X, const uint8_t* __restrict__ lmask,
    unsigned long long* __restrict__ keys, RtGeo g, int nrot, int chunk, int64_t first,
    double norm, int lgr, PlanRt px, const float2* __restrict__ twx_g,
    const float2* __restrict__ twf_g) {
    extern __shared__ float2 lds[];
    const int rl = RL > 0 ? RL : g.rl;
    const int lg = RL > 0 ? row_log(RL > 0 ? RL : 1, ODD, 3) : lgr;
    const int rpb = 1 << lg, tile = rpb * rl;
    float2* const A = lds;
    float2* const B = lds + 3 * tile;
    float2* const twx = B + 3 * tile;
    float2* const twfull = twx + rl;
    stage_tw(twx, twx_g, rl);
    if (!ODD) stage_tw(twfull, twf_g, 2 * rl);
    const int iz = blockIdx.y, row0 = blockIdx.x * rpb;
    const int b0 = blockIdx.z * chunk, b1 = min(nrot, b0 + chunk);
    const int M = rl, nx = ODD ? rl : 2 * rl, nxh = nx / 2 + 1, ny = g.ny;
    const double nv = norm * ((double)g.nz * ny * nx);   // N V (exact)
    // float u of the block's transformed rows -> voxel, or -1
    auto voxel = [&](int u) -> int64_t {
        if (u >= 2 * tile) return -1;
        int y, x;
        if constexpr (!ODD) {
            y = u / nx;
            x = u - y * nx;
            y += row0;
        } else {
            const int e = u >> 1, p = e / nx;
            x = e - p * nx;
            y = 2 * (row0 + p) + (u & 1);
        }
        return y < ny ? ((int64_t)iz * ny + y) * nx + x : -1;
    };
    float bv[kRowVox];
    int32_t bi[kRowVox];
    uint32_t mbits = 0, won = 0;
#pragma unroll
    for (int j = 0; j < kRowVox; ++j) {
        const int64_t v = voxel(threadIdx.x + j * kRowThreads);
        bv[j] = 0.f;
        bi[j] = 0;
        if (v >= 0 && lmask[v]) {
            mbits |= 1u << j;
            lcc_unkey(keys[v], &bv[j], &bi[j]);
        }
    }
    // Input pairs of the x transforms: even nx, X[k] and X[M - k] of a row give
    // z[k] and z[M - k] (C2R pre-processing, as k_inv_plane_rt); odd nx, X[k] of
    // rows 2p and 2p + 1 give the packed row's z[k] and z[nx - k].  Slot j of a
    // thread is pair u = t + j blockDim: transform f = u / P (grid f / rpb, row
    // f % rpb), k = u % P.  A rotation's pairs are loaded while the one before
    // is transformed.
    // The slots' indices pass through an empty asm so that they are computed
    // again for every rotation instead of being held in registers.
    const int P = ODD ? nxh : M / 2 + 1, np = 3 * rpb * P;
    float2 xa[kRowPairs], xb[kRowPairs];
    auto load = [&](int b) {
        const float2* src = X + (int64_t)b * 3 * g.H + (int64_t)iz * g.ps;
        const uint32_t H = (uint32_t)g.H;
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
#pragma unroll
        for (int j = 0; j < kRowPairs; ++j) {
            const int u = t + j * kRowThreads, f = u / P, k = u - f * P;
            const int row = row0 + (f & (rpb - 1));
            xa[j] = c2(0.f, 0.f);
            xb[j] = c2(0.f, 0.f);
            const uint32_t at = (f >> lg) * H + (uint32_t)((ODD ? 2 * row : row) * g.rp + k);
            if constexpr (!ODD) {
                if (u < np && row < ny) {
                    xa[j] = src[at];
                    xb[j] = src[at + (uint32_t)(M - 2 * k)];
                }
            } else {
                if (u < np && 2 * row < ny) xa[j] = src[at];
                if (u < np && 2 * row + 1 < ny) xb[j] = src[at + (uint32_t)g.rp];
            }
        }
    };
    if (b0 < b1) load(b0);
    __syncthreads();   // the twiddles are in LDS
    for (int b = b0; b < b1; ++b) {
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
#pragma unroll
        for (int j = 0; j < kRowPairs; ++j) {
            const int u = t + j * kRowThreads, f = u / P, k = u - f * P;
            if (u >= np) continue;
            float2* z = A + f * rl;
            float2 a = xa[j], c = xb[j];
            if constexpr (!ODD) {
                if (k == 0) {
                    // X[0] and X[M] are real
                    z[0] = c2(a.x + c.x, a.x - c.x);
                } else {
                    // i w^-k (X[k] - conj X[M-k]), and its mirror image at M - k
                    const float2 s = cadd(a, cconj(c)), d = csub(a, cconj(c));
                    const float2 e = mul_si<1>(cmul(d, cconj(twfull[k])));
                    z[k] = cadd(s, e);
                    z[M - k] = cconj(csub(s, e));
                }
            } else {
                if (k == 0) {
                    z[0] = c2(a.x, c.x);   // the DC bins are real
                } else {
                    z[k] = c2(a.x - c.y, a.y + c.x);
                    z[nx - k] = c2(a.x + c.y, c.x - a.y);
                }
            }
        }
        if (b + 1 < b1) load(b + 1);
        __syncthreads();
        const float2* Z = rows_fft<1, RL>(A, B, px, twx, 3 * rpb, rl);
        const float* zf = reinterpret_cast<const float*>(Z);
#pragma unroll
        for (int j = 0; j < kRowVox; ++j) {
            if (!((mbits >> j) & 1u)) continue;
            const int u = threadIdx.x + j * kRowThreads;
            const float gr = zf[u], ar = zf[2 * tile + u], br = zf[4 * tile + u];
            const double ad = (double)ar;
            const double var = fma(-ad, ad, (double)br * nv);
            const float s32 = gr * __builtin_amdgcn_rsqf((float)var);
            // only S > 0 can beat the initial (0, 0); NaN never wins
            if (s32 > 0.f && s32 >= bv[j] * (1.f - 1e-6f)) {
                const float s = (float)((double)gr / sqrt(var));
                const int32_t idx = (int32_t)(first + b);
                if (s > bv[j] || (s == bv[j] && idx < bi[j])) {
                    bv[j] = s;
                    bi[j] = idx;
                    won |= 1u << j;
                }
            }
        }
        __syncthreads();   // the rows are read: the next rotation may overwrite them
    }
#pragma unroll
    for (int j = 0; j < kRowVox; ++j)
        if ((won >> j) & 1u)
            atomicMax(keys + voxel(threadIdx.x + j * kRowThreads), lcc_key(bv[j], (uint32_t)bi[j]));
}

template <int L, int DIR>
int launch_cols(const Fft3D& f, const FusedArgs& a, int nplanes, int ng, int rg2, int zlo,
                hipStream_t s) {
    using FX = Flex<L, kFlexZSlots, kColTmax, false, true>;
    const int64_t blocks = (int64_t)((f.nxh + kColTq - 1) / kColTq) * nplanes * a.nrot;
    if (blocks > 0x7fffffffLL) {
        set_error("column stage: grid too large");
        return kErrUnsupported;
    }
    hipLaunchKernelGGL((k_cols<L, DIR>), dim3((unsigned)blocks), dim3(kColTq * FX::T), 0, s,
                       a.work, f.nz, f.nxh, a.rp, a.ps, nplanes, a.nrot, ng, a.rmax, rg2, zlo,
                       f.twy);
    return launched("k_cols");
}

template <int DIR>
int dispatch_cols(const Fft3D& f, const FusedArgs& a, int nplanes, int ng, int rg2, int zlo,
                  hipStream_t s) {
    switch (f.ny) {
#define PF_YCASE(L) \
    case L: return launch_cols<L, DIR>(f, a, nplanes, ng, rg2, zlo, s);
        PF_CT_COL_LENGTHS(PF_YCASE)
#undef PF_YCASE
        default:
            set_error("column stage: no compiled transform for length %d", f.ny);
            return kErrUnsupported;
    }
}

// The row kernels of stage `which` with row length RL compiled in (0: planned
// at run time).
template <bool ODD, int RL>
int launch_row_kernel(const Fft3D& f, const FusedArgs& a, int which, int nplanes, int zr,
                      hipStream_t s) {
    const RtGeo g = make_geo(f.nz, f.ny, f.nx, a.rp, a.ps);
    PlanRt px;
    const int ng = which == 0 ? (a.binary_mask ? 2 : 3) : 3;
    const int lg = row_log(g.rl, ODD, ng);
    if (!pack_plan(f.px, &px) || lg < 0) {
        set_error("row stages not available for x length %d", f.nx);
        return kErrUnsupported;
    }
    const int rpb = 1 << lg;
    const unsigned blocks = (unsigned)((g.nr + rpb - 1) / rpb);
    const size_t lds = row_lds_bytes(g.rl, ODD, rpb, ng);
    if (which == 0) {
        const int zlo = nplanes < f.nz ? -zr : 0;
        hipLaunchKernelGGL((k_rows_fwd<ODD, RL>), dim3(blocks * nplanes * a.nrot),
                           dim3(kRowThreads), lds, s, a.tm, a.occ, a.rots, g, a.rmax, zr * zr,
                           zlo, nplanes, ng, lg, a.work, px, f.twx, f.twfull);
        return launched("k_rows_fwd");
    }
    hipLaunchKernelGGL((k_rows_inv<ODD, RL>),
                       dim3(blocks, f.nz, (a.nrot + a.chunk_lcc - 1) / a.chunk_lcc),
                       dim3(kRowThreads), lds, s, a.work, a.lcc_mask, a.keys, g, a.nrot,
                       a.chunk_lcc, a.first, a.norm, lg, px, f.twx, f.twfull);
    return launched("k_rows_inv");
}

int launch_rows(const Fft3D& f, const FusedArgs& a, int which, int nplanes, int zr,
                hipStream_t s) {
    if (f.nx % 2) {
        switch (f.nx) {
#define PF_XCASE(L)     case L: return launch_row_kernel<true, L>(f, a, which, nplanes, zr, s);
            PF_CT_ODD_LENGTHS(PF_XCASE)
#undef PF_XCASE
            default: return launch_row_kernel<true, 0>(f, a, which, nplanes, zr, s);
        }
    }
    switch (f.nx / 2) {
#define PF_XCASE(L)     case L: return launch_row_kernel<false, L>(f, a, which, nplanes, zr, s);
        PF_CT_ROW_LENGTHS(PF_XCASE)
#undef PF_XCASE
        default: return launch_row_kernel<false, 0>(f, a, which, nplanes, zr, s);
    }
}

}  // namespace

bool rows_supported(int nz, int ny, int nx) {
    if (nz < 2 || ny < 2 || nx < 3 || nz > 65535 || ny > 65535) return false;
    if (!zcorr_ct_supported(ny) || !zcorr_ct_supported(nz)) return false;
    const RtGeo g = make_geo(nz, ny, nx);
    PlanRt p;
    return plan_rt(g.rl, &p) && row_log(g.rl, g.odd, 3) >= 0;
}

int launch_rows_stage(const Fft3D& f, const FusedArgs& a, int which, hipStream_t s) {
    if (a.nrot <= 0) return kOk;
    if (!rows_supported(f.nz, f.ny, f.nx)) {
        set_error("row stages not available for grid (%d, %d, %d)", f.nz, f.ny, f.nx);
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
    if (which == 0) {
        PF_CHECK_STATUS(launch_rows(f, a, 0, nplanes, zr, s));
        return dispatch_cols<-1>(f, a, nplanes, a.binary_mask ? 2 : 3, zr * zr,
                                 nplanes < f.nz ? -zr : 0, s);
    }
    PF_CHECK_STATUS(dispatch_cols<1>(f, a, f.nz, 3, 0, 0, s));
    return launch_rows(f, a, 2, f.nz, 0, s);
}

}  // namespace pf
