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
#include <algorithm>

#include "pf_ct_fft.h"
#include "pf_internal.h"

namespace pf {

namespace {

constexpr int kZTmax = 32;   // threads per transform
constexpr int kZTq = 16;     // columns per block

// power-of-two threads per column: a block is 16 T threads, whole wavefronts
// from T = 4 up.  EMAX: register slots per thread and transform (the default
// kFlexZSlots, or the alternative kFlexZSlotsAlt plan of more threads with
// fewer registers each, where one exists).
template <int L, int EMAX>
using ZF = Flex<L, EMAX, kZTmax, false, true>;
template <int L, int EMAX>
using ZB = Flex<L, EMAX, kZTmax, true, true>;

// Wavefronts per SIMD the registers of E slots leave room for: four (128
// registers) where that spills nothing that matters, and for the 512-thread
// blocks of T = 32, which otherwise fit a compute unit once.
constexpr int z_waves(int E, int T) { return E <= 9 || (T == 32 && E == 10) ? 4 : 2; }

// An offset beyond the end of any spectrum (at most 256 x 256 x 144 complex).
constexpr uint32_t kBeyond = 0xfffffff0u;

__device__ __forceinline__ float2 buffer_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}

__device__ __forceinline__ void buffer_store(float2 v, __amdgpu_buffer_rsrc_t r, uint32_t off) {
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, (int)off, 0, 0);
}

template <int L, bool BIN, int EMAX>
__global__ __launch_bounds__((kZTq * ZF<L, EMAX>::T), z_waves(ZF<L, EMAX>::E, ZF<L, EMAX>::T)) void k_zcorr_ct(
    float2* __restrict__ X, const float2* __restrict__ F1, const float2* __restrict__ F2,
    int ny, int nxh, int rp, int ps, int nrot, int chunk, int zr,
    const float2* __restrict__ twz) {
    using ZF = pf::ZF<L, EMAX>;
    using ZB = pf::ZB<L, EMAX>;
    constexpr int T = ZF::T, E = ZF::E;
    constexpr int EI = ZF::in_slots(), EO = ZF::out_slots();
    static_assert(ZB::T == T && ZB::E == E, "same threads and slots both ways");
    __shared__ float2 ex[L * kZTq];
    __shared__ float2 stw[L];
    for (int i = threadIdx.x; i < L; i += blockDim.x) stw[i] = twz[i];
    __syncthreads();
    const int c = threadIdx.x % kZTq, t = threadIdx.x / kZTq;
    // neighbouring tiles on one XCD: they share cache lines where planes or
    // rows are not whole lines
    const int ntiles = (ny * rp + kZTq - 1) / kZTq, nch = (nrot + chunk - 1) / chunk;
    const int blk = xcd_order(blockIdx.x, ntiles * nch);
    // column q of the work planes, kx = q mod rp of row y = q / rp
    const int q = (blk % ntiles) * kZTq + c;
    const int y = q / rp, kx = q - y * rp;
    const bool active = y < ny && kx < nxh;
    const int64_t H = (int64_t)L * ps;
    const int b0 = blk / ntiles * chunk;
    const int b1 = min(nrot, b0 + chunk);
    // byte offsets of this thread's input-pattern elements in a spectrum; idle
    // slots lie beyond its end, where buffer loads give 0 and stores are dropped
    uint32_t off[EI], in[EI];
#pragma unroll
    for (int s = 0; s < EI; ++s) {
        const int p = ZF::in_pos(t, s);
        const int sz = p <= L / 2 ? p : p - L;
        off[s] = active && p >= 0 ? (uint32_t)(p * ps + q) * 8u : kBeyond;
        // planes beyond the support were not written: they are zero
        in[s] = sz >= -zr && sz <= zr ? off[s] : kBeyond;
    }
    const int bytes = (int)(H * 8);
    auto spectrum = [&](int b, int g) {
        return __builtin_amdgcn_make_buffer_rsrc(X + ((int64_t)b * 3 + g) * H, 0, bytes,
                                                 0x00020000);
    };
    // target spectra at this thread's output-pattern elements
    float2 f1[EO], f2[EO];
#pragma unroll
    for (int s = 0; s < EO; ++s) {
        const int p = ZF::out_pos(t, s);
        const bool ok = active && p >= 0;
        const int fq = (p * ny + y) * nxh + kx;
        f1[s] = ok ? F1[fq] : c2(0.f, 0.f);
        f2[s] = ok ? F2[fq] : c2(0.f, 0.f);
    }
    float2* const exc = ex + c;
    // columns are loaded one transform ahead
    float2 nx[EI];
    auto load = [&](int b, int g) {
        const __amdgpu_buffer_rsrc_t r = spectrum(b, g);
#pragma unroll
        for (int s = 0; s < EI; ++s) nx[s] = buffer_load(r, in[s]);
    };
    auto store = [&](const float2 (&v)[E], int b, int g) {
        const __amdgpu_buffer_rsrc_t r = spectrum(b, g);
#pragma unroll
        for (int s = 0; s < EI; ++s) buffer_store(v[s], r, off[s]);
    };
    constexpr int NG = BIN ? 2 : 3;
    constexpr bool AHEAD = !(T == 32 && E > 8);
    if (AHEAD && b0 < b1) load(b0, 0);
    for (int b = b0; b < b1; ++b) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            if (!AHEAD) load(b, g);
            float2 v[E];
#pragma unroll
            for (int s = 0; s < E; ++s) v[s] = s < EI ? nx[s] : c2(0.f, 0.f);
            if (AHEAD && g + 1 < NG) load(b, g + 1);
            else if (AHEAD && b + 1 < b1) load(b + 1, 0);
            flex_fft<L, EMAX, kZTmax, false, -1, true>(v, exc, kZTq, t, stw, true);
            if (BIN && g == 1) {
                // W's spectrum feeds both A (with F1) and B (with F2)
                float2 u[E];
#pragma unroll
                for (int s = 0; s < E; ++s) {
                    u[s] = s < EO ? cmul(cconj(v[s]), f2[s]) : c2(0.f, 0.f);
                    v[s] = s < EO ? cmul(cconj(v[s]), f1[s]) : c2(0.f, 0.f);
                }
                flex_fft<L, EMAX, kZTmax, true, 1, true>(v, exc, kZTq, t, stw, true);
                store(v, b, 1);
                flex_fft<L, EMAX, kZTmax, true, 1, true>(u, exc, kZTq, t, stw, true);
                store(u, b, 2);
            } else {
#pragma unroll
                for (int s = 0; s < E; ++s)
                    v[s] = s < EO ? cmul(cconj(v[s]), g == 2 ? f2[s] : f1[s]) : c2(0.f, 0.f);
                flex_fft<L, EMAX, kZTmax, true, 1, true>(v, exc, kZTq, t, stw, true);
                store(v, b, g);
            }
        }
    }
}

template <int L, int EMAX>
int launch_zct(const Fft3D& f, const FusedArgs& a, int zr, hipStream_t s) {
    const dim3 grid((f.ny * a.rp + kZTq - 1) / kZTq * ((a.nrot + a.chunk_z - 1) / a.chunk_z));
    const dim3 block(kZTq * ZF<L, EMAX>::T);
    if (a.binary_mask)
        hipLaunchKernelGGL((k_zcorr_ct<L, true, EMAX>), grid, block, 0, s, a.work, a.F1, a.F2,
                           f.ny, f.nxh, a.rp, a.ps, a.nrot, a.chunk_z, zr, f.twz);
    else
        hipLaunchKernelGGL((k_zcorr_ct<L, false, EMAX>), grid, block, 0, s, a.work, a.F1, a.F2,
                           f.ny, f.nxh, a.rp, a.ps, a.nrot, a.chunk_z, zr, f.twz);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("launch of k_zcorr_ct failed: %s", hipGetErrorString(e));
        return kErrHip;
    }
    return kOk;
}

}  // namespace

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
                return launch_zct<L, kFlexZSlotsAlt>(f, a, zr, s);      \
        return launch_zct<L, kFlexZSlots>(f, a, zr, s);
        PF_CT_COL_LENGTHS(PF_ZCASE)
#undef PF_ZCASE
        default:
            set_error("z stage: no compiled transform for length %d", f.nz);
            return kErrUnsupported;
    }
}

}  // namespace pf
