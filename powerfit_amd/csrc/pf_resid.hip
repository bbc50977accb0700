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
// (k_fwd_plane_rt, k_inv_plane_rt): 120^3 5.4 / 7.5 / 8.6 us (7.9 / 6.6 / 15.5),
// 75 x 81 x 105 2.3 / 3.5 / 5.2 (3.9 / 2.9 / 8.8), 70 x 72 x 98 1.8 / 2.3 / 2.5
// (2.4 / 2.0 / 4.9), 32^3 0.83 / 0.39 / 0.57 at 24 rotations (1.23 / 0.44 / 1.6).
// The plane kernels spend their time at barriers: fifteen a rotation, behind one or
// two blocks a unit; here five, behind two to four.
//
// Work layout (ResidMap): 16 columns of the z stage are one 128-byte line: TK =
// 16 / RB kx of each of the RB residues, [z][ka][kx / TK][b][kx % TK].
#include <algorithm>

#include "pf_planes_kern.h"

namespace pf {

namespace {

constexpr int kResThreads = 512;

// x plan of a row: two stages (three where the length needs them), the last
// radix at most 10 (its outputs are the voxels a thread owns).
struct ResPlan {
    int ns = 0;
    int r[3] = {1, 1, 1};
};
constexpr ResPlan res_plan(int L) {
    ResPlan best;
    int cost = 1 << 30;
    for (int a = 2; a <= 16; ++a) {
        if (L % a) continue;
        const int b = L / a;
        if (b >= 2 && b <= 10) {
            const int c = 2 * a > 3 * b ? 2 * a : 3 * b;
            if (c < cost) {
                cost = c;
                best.ns = 2;
                best.r[0] = a;
                best.r[1] = b;
            }
        }
    }
    if (best.ns) return best;
    for (int a = 2; a <= 16; ++a)
        for (int b = 2; b <= 16; ++b) {
            if (L % (a * b)) continue;
            const int d = L / (a * b);
            if (d < 2 || d > 10) continue;
            const int c = a + b + d;
            if (c < cost) {
                cost = c;
                best.ns = 3;
                best.r[0] = a;
                best.r[1] = b;
                best.r[2] = d;
            }
        }
    return best;
}

template <int RL>
struct XPlan {
    static constexpr ResPlan P = res_plan(RL);
    static constexpr int radix(int s) { return P.r[s]; }
    static constexpr int span(int s) {
        int n = 1;
        for (int i = 0; i < s; ++i) n *= P.r[i];
        return n;
    }
};

// Inputs, twiddles and DFT of butterfly j of x stage S; element e of the row
// through ld(e).
template <int RL, int DIR, int S, class LD>
__device__ __forceinline__ void x_bfly(float2 (&v)[XPlan<RL>::radix(S)], int j, const float2* tw,
                                       const LD& ld) {
    using X = XPlan<RL>;
    constexpr int R = X::radix(S), Ns = X::span(S), NB = RL / R, STEP = RL / (Ns * R);
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = ld(j + r * NB);
    if constexpr (Ns > 1) {
        const int k = j % Ns;
#pragma unroll
        for (int r = 1; r < R; ++r) v[r] = cmul(v[r], twid<DIR>(tw, r * k * STEP));
    }
    dft_any<R, DIR>(v);
}

// Output position r of butterfly j of x stage S.
template <int RL, int S>
__device__ __forceinline__ int x_out(int j, int r) {
    using X = XPlan<RL>;
    constexpr int R = X::radix(S), Ns = X::span(S);
    const int k = j % Ns;
    return (j - k) * R + k + r * Ns;
}

// The thread index as a value the compiler does not carry over from an earlier use.
__device__ __forceinline__ int fresh_tid() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// Stage S over `rows` rows (row f at base + f pitch) in place: a pass takes as
// many whole rows as the block's threads cover, reads, waits, writes.  The
// last stage of two reads and writes the same positions and needs no wait
// between.
template <int RL, int DIR, int S, class LD>
__device__ __forceinline__ void x_stage(float2* base, int pitch, int rows, const float2* tw,
                                        const LD& ld) {
    using X = XPlan<RL>;
    constexpr int R = X::radix(S), NB = RL / R;
    constexpr bool own = X::P.ns == 2 && S == 1;
    const int per = (int)blockDim.x / NB;
    const int t = fresh_tid(), f0 = t / NB, j = t - f0 * NB;
#pragma unroll 1
    for (int at = 0; at < rows; at += per) {
        const int f = at + f0;
        const bool act = f0 < per && f < rows;
        float2 v[R];
        if (act) x_bfly<RL, DIR, S>(v, j, tw, [&](int e) { return ld(f, e); });
        if constexpr (!own) __syncthreads();
        if (act) {
#pragma unroll
            for (int r = 0; r < R; ++r) base[f * pitch + x_out<RL, S>(j, r)] = v[r];
        }
    }
    __syncthreads();
}

// Calls f with the radix R as a constant.
template <class F>
__device__ __forceinline__ void with_radix(int R, const F& f) {
    switch (R) {
        case 2: f(std::integral_constant<int, 2>()); break;
        case 3: f(std::integral_constant<int, 3>()); break;
        case 4: f(std::integral_constant<int, 4>()); break;
        case 5: f(std::integral_constant<int, 5>()); break;
        case 6: f(std::integral_constant<int, 6>()); break;
        case 7: f(std::integral_constant<int, 7>()); break;
        case 8: f(std::integral_constant<int, 8>()); break;
        case 9: f(std::integral_constant<int, 9>()); break;
        default: f(std::integral_constant<int, 10>()); break;
    }
}

struct ResArgs {
    int nz, ny, nx;
    int r1, r2;          // RA = r1 r2
    ResidMap m;
    int64_t H;           // work spectrum stride
};

// Offset of (residue b, row ka, kx) within a work plane.
__device__ __forceinline__ int res_at(const ResidMap& m, int b, int ka, int kx) {
    if (m.rb == 1) return ka * m.rp + kx;
    const int g = (kx * m.magic) >> 16;
    return (ka * m.nkg + g) * 16 + b * m.tk + kx - g * m.tk;
}

// LDS: rows of all grids (pitch NXH; odd x: packed row pairs, pitch 2 NXH), x
// twiddles, R2C twiddles (even x), w_RA, w_ny^(b ka).
constexpr int res_rows(int ra, bool odd) { return odd ? (ra + 1) / 2 * 2 : ra; }
constexpr size_t res_lds(int rl, bool odd, int ra, int ng) {
    return sizeof(float2) * ((size_t)ng * res_rows(ra, odd) * (odd ? rl / 2 + 1 : rl + 1) + rl +
                             (odd ? 0 : rl) + 2 * (size_t)ra);
}

template <bool ODD, int RL>
__global__ __launch_bounds__(kResThreads, 4) void k_fwd_resid(
    const float2* __restrict__ tm, const uint32_t* __restrict__ occ,
    const double* __restrict__ rots, ResArgs g, int rad, int rg2, int zlo, int nplanes, int ng,
    float2* __restrict__ out, const float2* __restrict__ twx_g, const float2* __restrict__ twy_g,
    const float2* __restrict__ twf_g) {
    constexpr int nx = ODD ? RL : 2 * RL, NXH = nx / 2 + 1, M = RL;
    constexpr int PZ = ODD ? 2 * NXH : NXH;   // pitch of a transformed (packed) row
    extern __shared__ float2 lds[];
    const int ra = g.m.ra, rb = g.m.rb, nrow = ODD ? (ra + 1) / 2 : ra;
    const int tile = res_rows(ra, ODD) * NXH;
    float2* const A = lds;
    float2* const twx = lds + ng * tile;
    float2* const twf = twx + RL;
    float2* const twa = twf + (ODD ? 0 : RL);
    float2* const twb = twa + ra;
    // residues of a plane and neighbouring planes of a rotation on one XCD
    const int blk = xcd_order(blockIdx.x, gridDim.x);
    const int pl = blk / rb, b = blk - pl * rb, rot = pl / nplanes;
    const int iz = (pl - rot * nplanes + zlo + g.nz) % g.nz;
    const int sz = scoord(iz, rad, g.nz);
    stage_tw(twx, twx_g, RL);
    if (!ODD) stage_tw(twf, twf_g, RL);
    for (int i = threadIdx.x; i < ra; i += blockDim.x) {
        twa[i] = twy_g[i * rb];
        twb[i] = twy_g[i * b];
    }
    double R[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) R[i] = rots[9 * rot + i];
#pragma unroll 1
    for (int u = threadIdx.x; u < nrow * RL; u += blockDim.x) {
        // even nx: voxels 2m, 2m + 1 of row a; odd nx: voxel x of rows 2p, 2p + 1
        const int f = u / RL, e = u - f * RL;
        float2 p2 = c2(0.f, 0.f), w2 = c2(0.f, 0.f);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int a = ODD ? 2 * f + h : f;
            const int sy = scoord(a * rb + b, rad, g.ny);
            const int sx = scoord(ODD ? e : 2 * e + h, rad, nx);
            float p = 0.f, w = 0.f;
            if (a < ra && sz * sz + sy * sy + sx * sx <= rg2)
                gather_pw_rt(tm, occ, g.nz, g.ny, nx, R, sz, sy, sx, &p, &w);
            if (h) {
                p2.y = p;
                w2.y = w;
            } else {
                p2.x = p;
                w2.x = w;
            }
        }
        A[f * PZ + e] = p2;
        A[tile + f * PZ + e] = w2;
        if (ng == 3) A[2 * tile + f * PZ + e] = c2(w2.x * w2.x, w2.y * w2.y);
    }
    __syncthreads();
    // x transforms of all rows of all grids
    const int rows = ng * nrow;
    static_assert(XPlan<RL>::P.ns >= 2, "x plan");
    auto ldrow = [&](int f, int e) { return A[f * PZ + e]; };
    x_stage<RL, -1, 0>(A, PZ, rows, twx, ldrow);
    x_stage<RL, -1, 1>(A, PZ, rows, twx, ldrow);
    if constexpr (XPlan<RL>::P.ns == 3) x_stage<RL, -1, 2>(A, PZ, rows, twx, ldrow);
    // X[a][k] of grid gi from the transformed rows
    auto post = [&](const float2* G, int a, int k) -> float2 {
        if constexpr (!ODD) {
            const float2* z = G + a * PZ;
            if (k == 0 || k == M) {
                const float2 z0 = z[0];
                return c2(k == 0 ? z0.x + z0.y : z0.x - z0.y, 0.f);
            }
            const float2 zk = z[k], zm = cconj(z[M - k]);
            const float2 E = cscale(cadd(zk, zm), 0.5f);
            const float2 O = mul_si<-1>(cscale(csub(zk, zm), 0.5f));
            return cadd(E, cmul(twf[k], O));
        } else {
            const float2* z = G + (a >> 1) * PZ;
            const float2 zk = z[k], zm = cconj(z[k ? nx - k : 0]);
            return (a & 1) ? mul_si<-1>(cscale(csub(zk, zm), 0.5f)) : cscale(cadd(zk, zm), 0.5f);
        }
    };
    float2* const dst = out + (int64_t)rot * 3 * g.H + (int64_t)iz * g.m.ps;
    const int r1 = g.r1, r2 = g.r2;
    for (int gi = 0; gi < ng; ++gi) {
        float2* const G = A + gi * tile;
        float2* const o = dst + (int64_t)gi * g.H;
        // first y stage: inputs a = j + r r2, outputs j r1 + r (held over the
        // wait: two items a thread at most)
        with_radix(r1, [&](auto rc) {
            constexpr int Q = rc();
            float2 v[2][Q];
            const int t = fresh_tid();
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int u = t + s * (int)blockDim.x, j = u / NXH, k = u - j * NXH;
                if (j >= r2) continue;
#pragma unroll
                for (int r = 0; r < Q; ++r) v[s][r] = post(G, j + r * r2, k);
                dft_any<Q, -1>(v[s]);
            }
            if (r2 > 1) __syncthreads();
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int u = t + s * (int)blockDim.x, j = u / NXH, k = u - j * NXH;
                if (j >= r2) continue;
#pragma unroll
                for (int r = 0; r < Q; ++r) {
                    const int a = j * Q + r;
                    if (r2 > 1) G[a * NXH + k] = v[s][r];
                    else o[res_at(g.m, b, a, k)] = cmul(v[s][r], twb[a]);
                }
            }
        });
    }
    if (r2 == 1) return;
    __syncthreads();
    // last y stage, with the twiddles of the residue, out to the work buffer
    with_radix(r2, [&](auto rc) {
        constexpr int Q = rc();
#pragma unroll 1
        for (int u = fresh_tid(); u < ng * r1 * NXH; u += blockDim.x) {
            const int gj = u / NXH, k = u - gj * NXH, gi = gj / r1, j = gj - gi * r1;
            const float2* G = A + gi * tile + k;
            float2 v[Q];
#pragma unroll
            for (int r = 0; r < Q; ++r) v[r] = G[(j + r * r1) * NXH];
#pragma unroll
            for (int r = 1; r < Q; ++r) v[r] = cmul(v[r], twa[r * j]);
            dft_any<Q, -1>(v);
            float2* const o = dst + (int64_t)gi * g.H;
#pragma unroll
            for (int r = 0; r < Q; ++r) {
                const int ka = j + r * r1;
                o[res_at(g.m, b, ka, k)] = cmul(v[r], twb[ka]);
            }
        }
    });
}

template <bool ODD, int RL>
__global__ __launch_bounds__(kResThreads, 4) void k_inv_resid(
    const float2* __restrict__ X, const uint8_t* __restrict__ lmask,
    unsigned long long* __restrict__ keys, ResArgs g, int nrot, int chunk, int64_t first,
    double norm, const float2* __restrict__ twx_g, const float2* __restrict__ twy_g,
    const float2* __restrict__ twf_g) {
    constexpr int nx = ODD ? RL : 2 * RL, NXH = nx / 2 + 1, M = RL;
    constexpr int PZ = ODD ? 2 * NXH : NXH;
    using XP = XPlan<RL>;
    constexpr int SL = XP::P.ns - 1, RZ = XP::radix(SL), NBZ = RL / RZ;   // last x stage
    extern __shared__ float2 lds[];
    const int ra = g.m.ra, rb = g.m.rb, nrow = ODD ? (ra + 1) / 2 : ra;
    const int tile = res_rows(ra, ODD) * NXH;
    float2* const A = lds;
    float2* const twx = lds + 3 * tile;
    float2* const twf = twx + RL;
    float2* const twa = twf + (ODD ? 0 : RL);
    float2* const twb = twa + ra;
    const int blk = xcd_order(blockIdx.x, gridDim.x);
    const int pl = blk / rb, b = blk - pl * rb, ch = pl / g.nz;
    const int iz = pl - ch * g.nz;
    const int b0 = ch * chunk, b1 = min(nrot, b0 + chunk);
    stage_tw(twx, twx_g, RL);
    if (!ODD) stage_tw(twf, twf_g, RL);
    for (int i = threadIdx.x; i < ra; i += blockDim.x) {
        twa[i] = twy_g[i * rb];
        twb[i] = twy_g[i * b];
    }
    const double nv = norm * ((double)g.nz * g.ny * nx);   // N V (exact)
    const int r1 = g.r1, r2 = g.r2;
    // owned voxels: item (row f, butterfly j) of the last x stage, outputs r
    const bool own = (int)threadIdx.x / NBZ < nrow;
    auto voxel = [&](int t, int r, int h) -> int {   // -1: none
        const int f = t / NBZ, e = x_out<RL, SL>(t - f * NBZ, r);
        const int a = ODD ? 2 * f + h : f, x = ODD ? e : 2 * e + h;
        return own && a < ra ? (iz * g.ny + a * rb + b) * nx + x : -1;
    };
    // their best score and its rotation within the chunk
    float bv[2 * RZ];
    int bi[2 * RZ];
#pragma unroll
    for (int q = 0; q < 2 * RZ; ++q) {
        bv[q] = 0.f;
        bi[q] = 0;
    }
    __syncthreads();   // the twiddles are in LDS
#pragma unroll 1
    for (int rot = b0; rot < b1; ++rot) {
        // first y stage, from the work buffer: item (gj = grid r2 + j, k), inputs
        // ka = j + r r2
        const float2* const src = X + (int64_t)rot * 3 * g.H + (int64_t)iz * g.m.ps;
        with_radix(r1, [&](auto rc) {
            constexpr int Q = rc();
#pragma unroll 1
            for (int u = fresh_tid(); u < 3 * r2 * NXH; u += blockDim.x) {
                const int gj = u / NXH, k = u - gj * NXH, gi = gj / r2, j = gj - gi * r2;
                const float2* const sg = src + gi * g.H;
                float2 v[Q];
#pragma unroll
                for (int r = 0; r < Q; ++r) v[r] = sg[res_at(g.m, b, j + r * r2, k)];
#pragma unroll
                for (int r = 0; r < Q; ++r) v[r] = cmul(v[r], cconj(twb[j + r * r2]));
                dft_any<Q, 1>(v);
                float2* const G = A + gi * tile + k;
#pragma unroll
                for (int r = 0; r < Q; ++r) G[(j * Q + r) * NXH] = v[r];
            }
        });
        __syncthreads();
        if (r2 > 1) {
            with_radix(r2, [&](auto rc) {
                constexpr int Q = rc();
#pragma unroll 1
                for (int u = fresh_tid(); u < 3 * r1 * NXH; u += blockDim.x) {
                    const int gj = u / NXH, k = u - gj * NXH, gi = gj / r1, j = gj - gi * r1;
                    float2* const G = A + gi * tile + k;
                    float2 v[Q];
#pragma unroll
                    for (int r = 0; r < Q; ++r) v[r] = G[(j + r * r1) * NXH];
#pragma unroll
                    for (int r = 1; r < Q; ++r) v[r] = cmul(v[r], cconj(twa[r * j]));
                    dft_any<Q, 1>(v);
#pragma unroll
                    for (int r = 0; r < Q; ++r) G[(j + r * r1) * NXH] = v[r];
                }
            });
            __syncthreads();
        }
        // C2R pre-processing while the first x stage reads
        auto pre = [&](int f, int k) -> float2 {
            if constexpr (!ODD) {
                const float2* xr = A + f * PZ;
                float2 xk = xr[k], xm = xr[M - k];
                if (k == 0) {
                    xk.y = 0.f;
                    xm.y = 0.f;
                }
                const float2 xmc = cconj(xm);
                const float2 d = cmul(csub(xk, xmc), cconj(twf[k]));
                return cadd(cadd(xk, xmc), mul_si<1>(d));
            } else {
                // rows 2p and 2p + 1 as one complex row; the DC bins are real
                const float2* x0 = A + f * PZ;
                const bool two = 2 * (f % nrow) + 1 < ra;
                const int kk = k < NXH ? k : nx - k;
                float2 a = x0[kk], c = two ? x0[NXH + kk] : c2(0.f, 0.f);
                if (k == 0) {
                    a.y = 0.f;
                    c.y = 0.f;
                }
                if (k >= NXH) {
                    a.y = -a.y;
                    c.y = -c.y;
                }
                return c2(a.x - c.y, a.y + c.x);
            }
        };
        x_stage<RL, 1, 0>(A, PZ, 3 * nrow, twx, pre);
        auto ldrow = [&](int f, int e) { return A[f * PZ + e]; };
        if constexpr (XP::P.ns == 3) x_stage<RL, 1, 1>(A, PZ, 3 * nrow, twx, ldrow);
        if (own) {
            // last x stage of B, A, G of the owned voxels, then the LCC (as
            // k_inv_plane_rt)
            float isd[2 * RZ];
            float2 v[RZ];
            auto last = [&](int gi) {
                const int t = fresh_tid(), f = t / NBZ, j = t - f * NBZ;
                x_bfly<RL, 1, SL>(v, j, twx, [&](int e) { return A[gi * tile + f * PZ + e]; });
            };
            last(2);
#pragma unroll
            for (int r = 0; r < RZ; ++r) {
                isd[2 * r] = v[r].x;
                isd[2 * r + 1] = v[r].y;
            }
            last(1);
#pragma unroll
            for (int q = 0; q < 2 * RZ; ++q) {
                const double ad = (double)(q & 1 ? v[q >> 1].y : v[q >> 1].x);
                isd[q] = __builtin_amdgcn_rsqf((float)fma(-ad, ad, (double)isd[q] * nv));
            }
            last(0);
            // only S > 0 can beat the initial (0, 0); NaN never wins; ties keep the
            // earlier rotation.  Selects, for voxels outside the lcc mask too (a
            // branch per voxel makes the compiler copy all the held values around
            // each one: 1,400 spilled registers)
#pragma unroll
            for (int q = 0; q < 2 * RZ; ++q) {
                const float s = (q & 1 ? v[q >> 1].y : v[q >> 1].x) * isd[q];
                const bool better = s > bv[q];
                bv[q] = better ? s : bv[q];
                bi[q] = better ? rot : bi[q];
            }
        }
        __syncthreads();   // the rows are read: the next rotation may overwrite them
    }
    const int t = fresh_tid();
#pragma unroll
    for (int q = 0; q < 2 * RZ; ++q) {
        const int vox = voxel(t, q >> 1, q & 1);
        if (vox >= 0 && bv[q] > 0.f && lmask[vox])
            atomicMax(keys + vox, lcc_key(bv[q], (uint32_t)(first + bi[q])));
    }
}

// The y split of a grid: RB and RA = r1 r2, and the blocks' threads.
struct ResSplit {
    int rb = 0, r1 = 0, r2 = 0, nthr = 0;
};

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
        // balanced radices; the larger one first
        int r1 = 0, r2 = 0;
        for (int a = 2; a <= 10; ++a)
            if (ra % a == 0 && ra / a <= a && ra / a <= 8 && !r1) {
                r1 = a;
                r2 = ra / a;
            }
        if (!r1) continue;
        const int nrow = odd ? (ra + 1) / 2 : ra, rz = xp.r[xp.ns - 1];
        const int own = nrow * (rl / rz);          // items of the last x stage: one a thread
        int best = 0;
        int64_t best_cost = 0;
        for (int n = 128; n <= kResThreads; n += 64) {
            if (own > n || r2 * nxh > 2 * n) continue;   // k_fwd_resid's held items
            // lanes x (work + a fixed charge) of every pass of k_inv_resid
            auto pass = [&](int64_t items, int work) { return (items + n - 1) / n * n * (work + 6); };
            int64_t cost = pass(3 * r2 * nxh, r1) + (r2 > 1 ? pass(3 * r1 * nxh, r2) : 0) +
                           pass(own, 3 * rz + 2 * rz);
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

template <bool ODD, int RL>
int launch_resid(const Fft3D& f, const FusedArgs& a, int which, int nplanes, int zr,
                 hipStream_t s) {
    const ResSplit sp = res_choose(f.ny, f.nx);
    ResArgs g{f.nz, f.ny, f.nx, sp.r1, sp.r2, a.rmap, (int64_t)f.nz * a.rmap.ps};
    const int ng = which == 0 ? (a.binary_mask ? 2 : 3) : 3;
    const size_t lds = res_lds(RL, ODD, g.m.ra, ng);
    if (which == 0) {
        const int zlo = nplanes < f.nz ? -zr : 0;
        hipLaunchKernelGGL((k_fwd_resid<ODD, RL>), dim3((unsigned)(g.m.rb * nplanes * a.nrot)),
                           dim3(sp.nthr), lds, s, a.tm, a.occ, a.rots, g, a.rmax, zr * zr, zlo,
                           nplanes, ng, a.work, f.twx, f.twy, f.twfull);
        return launched("k_fwd_resid");
    }
    const int nch = (a.nrot + a.chunk_lcc - 1) / a.chunk_lcc;
    hipLaunchKernelGGL((k_inv_resid<ODD, RL>), dim3((unsigned)(g.m.rb * f.nz * nch)),
                       dim3(sp.nthr), lds, s, a.work, a.lcc_mask, a.keys, g, a.nrot, a.chunk_lcc,
                       a.first, a.norm, f.twx, f.twy, f.twfull);
    return launched("k_inv_resid");
}

template <bool ODD, int RL>
int allow_resid() {
    PF_CHECK_STATUS(allow_lds((const void*)k_fwd_resid<ODD, RL>, 80 * 1024));
    return allow_lds((const void*)k_inv_resid<ODD, RL>, 80 * 1024);
}

}  // namespace

ResidMap resid_map(int nz, int ny, int nx) {
    ResidMap m{};
    if (!plane_rt_supported(nz, ny, nx) || !zcorr_ct_supported(nz) || !res_row_length(nx)) return m;
    const ResSplit s = res_choose(ny, nx);
    if (!s.rb) return m;
    m.rb = s.rb;
    m.ra = ny / s.rb;
    m.tk = 16 / s.rb;
    m.magic = (65536 + m.tk - 1) / m.tk;
    m.nkg = (nx / 2 + 1 + m.tk - 1) / m.tk;
    m.rp = nx / 2 + 1;
    // whole lines, an odd number of them a plane (WorkLayout)
    const int lines = s.rb == 1 ? (ny * m.rp + 15) / 16 : m.ra * m.nkg;
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
    if (f.nx % 2) {
        switch (f.nx) {
#define PF_XCASE(L) \
    case L: return launch_resid<true, L>(f, a, which, nplanes, zr, s);
            PF_CT_ODD_LENGTHS(PF_XCASE)
#undef PF_XCASE
        }
    }
    switch (f.nx / 2) {
#define PF_XCASE(L) \
    case L: return launch_resid<false, L>(f, a, which, nplanes, zr, s);
        PF_CT_ROW_LENGTHS(PF_XCASE)
#undef PF_XCASE
    }
    set_error("residue stages: no compiled transform for x length %d", f.nx);
    return kErrUnsupported;
}

int prepare_resid(int nx) {
    if (!res_row_length(nx)) return kOk;
    if (nx % 2) {
        switch (nx) {
#define PF_XCASE(L) \
    case L: return allow_resid<true, L>();
            PF_CT_ODD_LENGTHS(PF_XCASE)
#undef PF_XCASE
        }
    }
    switch (nx / 2) {
#define PF_XCASE(L) \
    case L: return allow_resid<false, L>();
        PF_CT_ROW_LENGTHS(PF_XCASE)
#undef PF_XCASE
    }
    return kOk;
}

}  // namespace pf
