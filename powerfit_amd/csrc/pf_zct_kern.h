// Kernel of the register z stage (pf_zct.hip; the residue forms are instantiated
// in pf_zct_resid.hip).  Internal linkage in each unit that includes it.
#pragma once
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

// Lane exchanges within the 16 lanes of a tile: the value of lane ^ 8, lane ^ 4.
__device__ __forceinline__ float lane_xor8(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
        0, __builtin_bit_cast(int, x), 0x128, 0xf, 0xf, false));   // row_ror:8
}
__device__ __forceinline__ float lane_xor4(float x) {
    // row_half_mirror (lane ^ 7), then quad_perm 3,2,1,0 (lane ^ 3)
    const int m = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x141, 0xf, 0xf, false);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, m, 0x1b, 0xf, 0xf, false));
}

// RB-point transforms over the residues of a column, which lie TK = 16 / RB
// lanes apart in a tile (pf_resid.hip).  Forward: residue b in, kb out; inverse
// the other way.  RB 2 and 4 (RES 2, 4) as butterflies between lanes, RB 4
// leaving kb in bit-reversed order; RB 3 and 5 (RES 3) as sums over the lanes of a
// column with the powers of w_RB.
template <int RES>
struct ResidDft {
    float s8, s4;        // -1 in the upper lane of a butterfly, else 1
    bool turn;           // RB 4: this lane's value takes the factor w_4

    __device__ __forceinline__ ResidDft(const ResidMap&, int c, const float2*) {
        s8 = c & 8 ? -1.f : 1.f;
        s4 = c & 4 ? -1.f : 1.f;
        turn = c >= 12;
    }
    static __device__ __forceinline__ float2 step8(float2 x, float s) {
        return c2(fmaf(s, x.x, lane_xor8(x.x)), fmaf(s, x.y, lane_xor8(x.y)));
    }
    static __device__ __forceinline__ float2 step4(float2 x, float s) {
        return c2(fmaf(s, x.x, lane_xor4(x.x)), fmaf(s, x.y, lane_xor4(x.y)));
    }
    template <int DIR, int E>
    __device__ __forceinline__ void run(float2 (&v)[E]) const {
#pragma unroll
        for (int s = 0; s < E; ++s) {
            if constexpr (RES == 2) {
                v[s] = step8(v[s], s8);
            } else if constexpr (RES == 4) {
                float2 x = DIR < 0 ? step8(v[s], s8) : step4(v[s], s4);
                // times -i (forward) or i
                const float2 q = DIR < 0 ? c2(x.y, -x.x) : c2(-x.y, x.x);
                x = turn ? q : x;
                v[s] = DIR < 0 ? step4(x, s4) : step8(x, s8);
            }
        }
    }
};

template <>
struct ResidDft<3> {
    int rb, src[4];      // residues; byte addresses of the other lanes of the column
    const float2* w;     // this lane's powers of w_RB, by the other lane's order

    __device__ __forceinline__ ResidDft(const ResidMap& m, int c, const float2* wrb) {
        rb = m.rb;
        // (a lane past the last residue stands by itself)
        const int b = c / m.tk, lane = (int)(threadIdx.x & 63);
        w = wrb + (b < rb ? b : 0) * 5;
#pragma unroll
        for (int j = 1; j < 5; ++j)
            src[j - 1] = 4 * (b < rb && j < rb ? lane + ((b + j) % rb - b) * m.tk : lane);
    }
    template <int DIR, int E>
    __device__ __forceinline__ void run(float2 (&v)[E]) const {
        if (rb == 3) sum<DIR, 3>(v);
        else sum<DIR, 5>(v);
    }
    template <int DIR, int RB, int E>
    __device__ __forceinline__ void sum(float2 (&v)[E]) const {
        float2 f[RB];
#pragma unroll
        for (int j = 0; j < RB; ++j) f[j] = DIR < 0 ? w[j] : cconj(w[j]);
#pragma unroll
        for (int s = 0; s < E; ++s) {
            float2 x = cmul(v[s], f[0]);
#pragma unroll
            for (int j = 1; j < RB; ++j) {
                const float2 o = c2(lane_get(src[j - 1], v[s].x), lane_get(src[j - 1], v[s].y));
                x = cadd(x, cmul(o, f[j]));
            }
            v[s] = x;
        }
    }
    static __device__ __forceinline__ float lane_get(int at, float x) {
        return __builtin_bit_cast(float,
                                  __builtin_amdgcn_ds_bpermute(at, __builtin_bit_cast(int, x)));
    }
};

template <int L, bool BIN, int EMAX, int RES>
__global__ __launch_bounds__((kZTq * ZF<L, EMAX>::T), z_waves(ZF<L, EMAX>::E, ZF<L, EMAX>::T)) void k_zcorr_ct(
    float2* __restrict__ X, const float2* __restrict__ F1, const float2* __restrict__ F2,
    int ny, int nxh, int rp, int ps, ResidMap m, int nrot, int chunk, int zr,
    const float2* __restrict__ twz, const float2* __restrict__ twy) {
    using ZF = pf::ZF<L, EMAX>;
    using ZB = pf::ZB<L, EMAX>;
    constexpr int T = ZF::T, E = ZF::E;
    constexpr int EI = ZF::in_slots(), EO = ZF::out_slots();
    static_assert(ZB::T == T && ZB::E == E, "same threads and slots both ways");
    __shared__ float2 ex[L * kZTq];
    __shared__ float2 stw[L];
    __shared__ float2 wrb[RES == 3 ? 25 : 1];
    for (int i = threadIdx.x; i < L; i += blockDim.x) stw[i] = twz[i];
    if (RES == 3 && threadIdx.x < 25) {
        // lane of residue b, other lane's residue (b + j) mod RB: w_RB^(b ((b + j) mod
        // RB)), w_RB^i = w_ny^(RA i)
        const int b = threadIdx.x / 5, j = threadIdx.x - 5 * b;
        if (b < m.rb && j < m.rb) wrb[threadIdx.x] = twy[b * ((b + j) % m.rb) % m.rb * m.ra];
    }
    __syncthreads();
    const int c = threadIdx.x % kZTq, t = threadIdx.x / kZTq;
    // neighbouring tiles on one XCD: they share cache lines where planes or
    // rows are not whole lines
    const int ntiles = RES ? m.ra * m.nkg : (ny * rp + kZTq - 1) / kZTq;
    const int nch = (nrot + chunk - 1) / chunk;
    const int blk = xcd_order(blockIdx.x, ntiles * nch);
    const int tl = blk % ntiles, q = tl * kZTq + c;
    // column q of the work planes: row y and kx; with residues the tile holds TK
    // kx of row ka of each residue, which the cross-lane transforms turn into rows
    // ka + RA kb
    int y, kx;
    bool active;
    const ResidDft<RES> dft(m, c, wrb);
    if constexpr (RES > 0) {
        const int ka = tl / m.nkg;
        const int b = c / m.tk;
        kx = (tl - ka * m.nkg) * m.tk + c - b * m.tk;
        y = ka + m.ra * (RES == 4 ? (b >> 1) | ((b & 1) << 1) : b);
        active = b < m.rb && kx < nxh;
    } else {
        y = q / rp;
        kx = q - y * rp;
        active = y < ny && kx < nxh;
    }
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
        // (the unused lanes of a residue tile are stored too: whole lines)
        off[s] = (RES || active) && p >= 0 ? (uint32_t)(p * ps + q) * 8u : kBeyond;
        // planes beyond the support were not written: they are zero
        in[s] = active && sz >= -zr && sz <= zr ? off[s] : kBeyond;
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
            if (RES) dft.template run<-1>(v);
            if (BIN && g == 1) {
                // W's spectrum feeds both A (with F1) and B (with F2)
                float2 u[E];
#pragma unroll
                for (int s = 0; s < E; ++s) {
                    u[s] = s < EO ? cmul(cconj(v[s]), f2[s]) : c2(0.f, 0.f);
                    v[s] = s < EO ? cmul(cconj(v[s]), f1[s]) : c2(0.f, 0.f);
                }
                if (RES) dft.template run<1>(v);
                flex_fft<L, EMAX, kZTmax, true, 1, true>(v, exc, kZTq, t, stw, true);
                store(v, b, 1);
                if (RES) dft.template run<1>(u);
                flex_fft<L, EMAX, kZTmax, true, 1, true>(u, exc, kZTq, t, stw, true);
                store(u, b, 2);
            } else {
#pragma unroll
                for (int s = 0; s < E; ++s)
                    v[s] = s < EO ? cmul(cconj(v[s]), g == 2 ? f2[s] : f1[s]) : c2(0.f, 0.f);
                if (RES) dft.template run<1>(v);
                flex_fft<L, EMAX, kZTmax, true, 1, true>(v, exc, kZTq, t, stw, true);
                store(v, b, g);
            }
        }
    }
}

template <int L, int EMAX, int RES>
int launch_zct_kernel(const Fft3D& f, const FusedArgs& a, int zr, hipStream_t s) {
    const ResidMap& m = a.rmap;
    const int tiles = RES ? m.ra * m.nkg : (f.ny * a.rp + kZTq - 1) / kZTq;
    const dim3 grid(tiles * ((a.nrot + a.chunk_z - 1) / a.chunk_z));
    const dim3 block(kZTq * ZF<L, EMAX>::T);
    if (a.binary_mask)
        hipLaunchKernelGGL((k_zcorr_ct<L, true, EMAX, RES>), grid, block, 0, s, a.work, a.F1, a.F2,
                           f.ny, f.nxh, a.rp, a.ps, m, a.nrot, a.chunk_z, zr, f.twz, f.twy);
    else
        hipLaunchKernelGGL((k_zcorr_ct<L, false, EMAX, RES>), grid, block, 0, s, a.work, a.F1, a.F2,
                           f.ny, f.nxh, a.rp, a.ps, m, a.nrot, a.chunk_z, zr, f.twz, f.twy);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("launch of k_zcorr_ct failed: %s", hipGetErrorString(e));
        return kErrHip;
    }
    return kOk;
}

}  // namespace

// Residue forms (pf_zct_resid.hip).
int launch_zcorr_resid(const Fft3D& f, const FusedArgs& a, int zr, hipStream_t s);

}  // namespace pf
