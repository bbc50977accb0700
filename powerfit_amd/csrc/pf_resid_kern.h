// Kernels of the plane stages by row residue (pf_resid.hip), shared by its two
// translation units.  Internal linkage in each unit that includes it.
#pragma once
#include <algorithm>

#include "pf_planes_kern.h"

namespace pf {

// The y split of a grid: RB and RA = r1 r2, and the blocks' threads.
struct ResSplit {
    int rb = 0, r1 = 0, r2 = 0, nthr = 0;
};

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

// x twiddles in LDS: of a two-stage plan w^(r k) of the second stage at (r - 1) Ns
// + k, so that a butterfly's are at constant distances; of three stages w^m at m.
template <int RL>
__device__ __forceinline__ void stage_twx(float2* dst, const float2* __restrict__ src) {
    using X = XPlan<RL>;
    if constexpr (X::P.ns == 2) {
        constexpr int Ns = X::span(1);
        for (int i = threadIdx.x; i < RL - Ns; i += blockDim.x)
            dst[i] = src[(i / Ns + 1) * (i % Ns)];
    } else {
        stage_tw(dst, src, RL);
    }
}

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
        for (int r = 1; r < R; ++r)
            v[r] = cmul(v[r], twid<DIR>(tw, X::P.ns == 2 ? (r - 1) * Ns + k : r * k * STEP));
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

// Stage S over `rows` rows in place, the f-th at base + at(f), element e of its
// input ld(at(f), e): a pass takes as many whole rows as the block's threads
// cover, reads, waits, writes.  The last stage of two reads and writes the same
// positions and needs no wait between.
template <int RL, int DIR, int S, class AT, class LD>
__device__ __forceinline__ void x_stage(float2* base, int rows, const float2* tw, const AT& row_at,
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
        const int o = act ? row_at(f) : 0;
        float2 v[R];
        if (act) x_bfly<RL, DIR, S>(v, j, tw, [&](int e) { return ld(o, e); });
        if constexpr (!own) __syncthreads();
        if (act) {
#pragma unroll
            for (int r = 0; r < R; ++r) base[o + x_out<RL, S>(j, r)] = v[r];
        }
    }
    __syncthreads();
}

// Calls f with the radix R (2 to MAXR) as a constant.
template <int MAXR, class F>
__device__ __forceinline__ void with_radix(int R, const F& f) {
    switch (R) {
        case 2: f(std::integral_constant<int, 2>()); break;
        case 3: f(std::integral_constant<int, 3>()); break;
        case 4: f(std::integral_constant<int, 4>()); break;
        case 5: f(std::integral_constant<int, 5>()); break;
        case 6: f(std::integral_constant<int, 6>()); break;
        case 7: f(std::integral_constant<int, 7>()); break;
        case 8: f(std::integral_constant<int, 8>()); break;
        case 9: if constexpr (MAXR >= 9) f(std::integral_constant<int, 9>()); break;
        default: if constexpr (MAXR >= 10) f(std::integral_constant<int, 10>()); break;
    }
}

struct ResArgs {
    int nz, ny, nx;
    int r1, r2;          // RA = r1 r2
    ResidMap m;
    int64_t H;           // work spectrum stride
};

// Offset of (residue b, kx) within a row ka of a work plane (rows of m.rp).
__device__ __forceinline__ int res_col(const ResidMap& m, int b, int kx) {
    const int g = (kx * m.magic) >> 16;
    return m.rb == 1 ? kx : g * 16 + b * m.tk + kx - g * m.tk;
}

// LDS: rows of all grids (pitch NXH; odd x: packed row pairs, pitch 2 NXH), x
// twiddles, R2C twiddles (even x), w_RA, w_ny^(b ka).
constexpr int res_rows(int ra, bool odd) { return odd ? (ra + 1) / 2 * 2 : ra; }
constexpr size_t res_lds(int rl, bool odd, int ra, int ng) {
    return sizeof(float2) * ((size_t)ng * res_rows(ra, odd) * (odd ? rl / 2 + 1 : rl + 1) + rl +
                             (odd ? 0 : rl) + 2 * (size_t)ra);
}

// EXACT: for grids whose other path is the unfused kernels, their FP64 blend of the
// template, and 1 / sqrt(variance) rounded from FP64.
template <bool ODD, int RL, bool EXACT>
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
    stage_twx<RL>(twx, twx_g);
    if (!ODD) stage_tw(twf, twf_g, RL);
    for (int i = threadIdx.x; i < ra; i += blockDim.x) {
        twa[i] = twy_g[i * rb];
        twb[i] = twy_g[i * b];
    }
    double R[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) R[i] = rots[9 * rot + i];
    // rows that hold a voxel of the sphere: the first n1 and the last n2; the
    // others are zero and are not transformed
    int n1 = 0, n2 = 0;
    {
        const int y2 = rg2 - sz * sz;   // (planes within the support: not negative)
        int yl = (int)sqrtf((float)y2);
        while (yl * yl > y2) --yl;
        while ((yl + 1) * (yl + 1) <= y2) ++yl;
        n1 = yl >= b ? min(ra, (yl - b) / rb + 1) : 0;
        const int lo = g.ny - yl - b;   // rows from y = ny - yl up
        n2 = lo <= 0 ? ra : max(0, ra - (lo + rb - 1) / rb);
        if (ODD) {
            n1 = (n1 + 1) / 2;
            n2 = nrow - (ra - n2) / 2;
        }
        if (n1 + n2 >= nrow) {
            n1 = nrow;
            n2 = 0;
        }
    }
    const int nlive = n1 + n2;
    auto live_at = [&](int i) { return (i < n1 ? i : i - n1 + nrow - n2) * PZ; };
    // zero rows (with the columns that only the spectra use)
    for (int gi = 0; gi < ng; ++gi)
        for (int u = n1 * PZ + (int)threadIdx.x; u < (nrow - n2) * PZ; u += blockDim.x)
            A[gi * tile + u] = c2(0.f, 0.f);
#pragma unroll 1
    for (int u = threadIdx.x; u < nlive * RL; u += blockDim.x) {
        // even nx: voxels 2m, 2m + 1 of row a; odd nx: voxel x of rows 2p, 2p + 1
        const int i = u / RL, e = u - i * RL;
        const int at = live_at(i) + e, f = i < n1 ? i : i - n1 + nrow - n2;
        float2 p2 = c2(0.f, 0.f), w2 = c2(0.f, 0.f);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int a = ODD ? 2 * f + h : f;
            const int sy = scoord(a * rb + b, rad, g.ny);
            const int sx = scoord(ODD ? e : 2 * e + h, rad, nx);
            float p = 0.f, w = 0.f;
            if (a < ra && sz * sz + sy * sy + sx * sx <= rg2) {
                if (EXACT) gather_pw_f64(tm, occ, g.nz, g.ny, nx, R, sz, sy, sx, &p, &w);
                else gather_pw_rt(tm, occ, g.nz, g.ny, nx, R, sz, sy, sx, &p, &w);
            }
            // halved (exact), for the half sums of the spectra
            if (h) {
                p2.y = 0.5f * p;
                w2.y = w;
            } else {
                p2.x = 0.5f * p;
                w2.x = w;
            }
        }
        A[at] = p2;
        A[tile + at] = cscale(w2, 0.5f);
        if (ng == 3) A[2 * tile + at] = c2(0.5f * w2.x * w2.x, 0.5f * w2.y * w2.y);
    }
    __syncthreads();
    // x transforms of the live rows of all grids
    static_assert(XPlan<RL>::P.ns >= 2, "x plan");
    auto row_at = [&](int f) {
        const int gi = (f >= nlive) + (f >= 2 * nlive);
        return gi * tile + live_at(f - gi * nlive);
    };
    auto ldrow = [&](int o, int e) { return A[o + e]; };
    x_stage<RL, -1, 0>(A, ng * nlive, twx, row_at, ldrow);
    x_stage<RL, -1, 1>(A, ng * nlive, twx, row_at, ldrow);
    if constexpr (XPlan<RL>::P.ns == 3) x_stage<RL, -1, 2>(A, ng * nlive, twx, row_at, ldrow);
    float2* const dst = out + (int64_t)rot * 3 * g.H + (int64_t)iz * g.m.ps;
    const int r1 = g.r1, r2 = g.r2;
    const int rp = g.m.rp;
    // rows ka = base + r step of column k out to the work buffer, with the
    // residue's twiddles
    auto emit = [&](float2* o, int base, int step, int k, auto& v) {
        constexpr int Q = sizeof(v) / sizeof(float2);
        float2* const c = o + res_col(g.m, b, k);
        if (b) {
#pragma unroll
            for (int r = 0; r < Q; ++r) v[r] = cmul(v[r], twb[base + r * step]);
        }
#pragma unroll
        for (int r = 0; r < Q; ++r) c[(base + r * step) * rp] = v[r];
    };
    for (int gi = 0; gi < ng; ++gi) {
        float2* const G = A + gi * tile;
        float2* const o = dst + (int64_t)gi * g.H;
        // spectra of the rows (R2C post-processing) and first y stage: inputs a = j
        // + r r2, outputs j r1 + r, held over the wait.  Even nx: columns k and M -
        // k together, which come from the same pair of values,
        //   X[k] = E + w^k O, X[M - k] = conj(E - w^k O);
        // odd nx: rows 2p and 2p + 1 from the packed row, (z[k] + conj z[-k]) / 2
        // and (z[k] - conj z[-k]) / 2i.
        with_radix<10>(r1, [&](auto rc) {
            constexpr int Q = rc();
            constexpr int NC = ODD ? NXH : M / 2 + 1;
            float2 v[2][Q];
            const int t = fresh_tid();
            if constexpr (!ODD) {
                const int j = t / NC, k = t - j * NC;
                if (j < r2) {
                    const float2 wk = twf[k];
#pragma unroll
                    for (int r = 0; r < Q; ++r) {
                        const float2* z = G + (j + r * r2) * PZ;
                        if (k == 0) {
                            const float2 z0 = cscale(z[0], 2.f);
                            v[0][r] = c2(z0.x + z0.y, 0.f);
                            v[1][r] = c2(z0.x - z0.y, 0.f);
                        } else {
                            const float2 zk = z[k], zm = cconj(z[M - k]);
                            const float2 E = cadd(zk, zm);
                            const float2 O = cmul(wk, mul_si<-1>(csub(zk, zm)));
                            v[0][r] = cadd(E, O);
                            v[1][r] = cconj(csub(E, O));
                        }
                    }
                    dft_any<Q, -1>(v[0]);
                    dft_any<Q, -1>(v[1]);
                }
            } else {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const int u = t + s * (int)blockDim.x, j = u / NC, k = u - j * NC;
                    if (j >= r2) continue;
#pragma unroll
                    for (int r = 0; r < Q; ++r) {
                        const int a = j + r * r2;
                        const float2* z = G + (a >> 1) * PZ;
                        const float2 zk = z[k], zm = cconj(z[k ? nx - k : 0]);
                        v[s][r] = (a & 1) ? mul_si<-1>(csub(zk, zm)) : cadd(zk, zm);
                    }
                    dft_any<Q, -1>(v[s]);
                }
            }
            if (r2 > 1) __syncthreads();
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int u = ODD ? t + s * (int)blockDim.x : t;
                const int j = u / NC, kc = u - j * NC;
                if (j >= r2 || (!ODD && s && 2 * kc == M)) continue;
                const int k = !ODD && s ? M - kc : kc;
                if (r2 > 1) {
#pragma unroll
                    for (int r = 0; r < Q; ++r) G[(j * Q + r) * NXH + k] = v[s][r];
                } else {
                    emit(o, 0, 1, k, v[s]);
                }
            }
        });
    }
    if (r2 == 1) return;
    __syncthreads();
    // last y stage, with the twiddles of the residue, out to the work buffer
    with_radix<8>(r2, [&](auto rc) {
        constexpr int Q = rc();
#pragma unroll 1
        for (int u = fresh_tid(); u < ng * r1 * NXH; u += blockDim.x) {
            const int gj = u / NXH, k = u - gj * NXH;
            const int gi = (gj >= r1) + (gj >= 2 * r1), j = gj - gi * r1;
            const float2* G = A + gi * tile + k;
            float2 v[Q];
#pragma unroll
            for (int r = 0; r < Q; ++r) v[r] = G[(j + r * r1) * NXH];
#pragma unroll
            for (int r = 1; r < Q; ++r) v[r] = cmul(v[r], twa[r * j]);
            dft_any<Q, -1>(v);
            emit(dst + (int64_t)gi * g.H, j, r1, k, v);
        }
    });
}

template <bool ODD, int RL, bool EXACT>
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
    stage_twx<RL>(twx, twx_g);
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
        // First y stage, from the work buffer: inputs ka = j + r r2, outputs j r1 + r;
        // last y stage in place: inputs and outputs j + r r1.  (Taking columns k and
        // M - k together here, with the C2R pre-processing of both, saves a tenth of
        // the instructions but takes 128 registers for 80: 120^3 8.8 -> 10.8 us.)
        const float2* const src = X + (int64_t)rot * 3 * g.H + (int64_t)iz * g.m.ps;
        const int rp = g.m.rp;
        // rows ka = base + r step of column k of a spectrum, with the residue's
        // twiddles
        auto in = [&](const float2* sg, int base, int step, int k, auto& v) {
            constexpr int Q = sizeof(v) / sizeof(float2);
            const float2* const c = sg + res_col(g.m, b, k);
#pragma unroll
            for (int r = 0; r < Q; ++r) v[r] = c[(base + r * step) * rp];
            if (b) {
#pragma unroll
                for (int r = 0; r < Q; ++r) v[r] = cmul(v[r], cconj(twb[base + r * step]));
            }
        };
        with_radix<10>(r1, [&](auto rc) {
            constexpr int Q = rc();
#pragma unroll 1
            for (int u = fresh_tid(); u < 3 * r2 * NXH; u += blockDim.x) {
                const int gj = u / NXH, k = u - gj * NXH;
                const int gi = (gj >= r2) + (gj >= 2 * r2), j = gj - gi * r2;
                const float2* const sg = src + gi * g.H;
                float2 v[Q];
                in(sg, j, r2, k, v);
                dft_any<Q, 1>(v);
                float2* const G = A + gi * tile + k;
#pragma unroll
                for (int r = 0; r < Q; ++r) G[(j * Q + r) * NXH] = v[r];
            }
        });
        __syncthreads();
        if (r2 > 1) {
            with_radix<8>(r2, [&](auto rc) {
                constexpr int Q = rc();
#pragma unroll 1
                for (int u = fresh_tid(); u < 3 * r1 * NXH; u += blockDim.x) {
                    const int gj = u / NXH, k = u - gj * NXH;
                    const int gi = (gj >= r1) + (gj >= 2 * r1), j = gj - gi * r1;
                    float2* const G = A + gi * tile + j * NXH + k;
                    float2 v[Q];
#pragma unroll
                    for (int r = 0; r < Q; ++r) v[r] = G[r * r1 * NXH];
#pragma unroll
                    for (int r = 1; r < Q; ++r) v[r] = cmul(v[r], cconj(twa[r * j]));
                    dft_any<Q, 1>(v);
#pragma unroll
                    for (int r = 0; r < Q; ++r) G[r * r1 * NXH] = v[r];
                }
            });
            __syncthreads();
        }
        // C2R pre-processing while the first x stage reads: even nx z[k] = X[k] + conj
        // X[M - k] + i w^-k (X[k] - conj X[M - k]); odd nx rows 2p and 2p + 1 as one
        // complex row.  The DC (and Nyquist) bins are real
        auto pre = [&](int o, int k) -> float2 {
            if constexpr (!ODD) {
                float2 xk = A[o + k], xm = A[o + M - k];
                if (k == 0) {
                    xk.y = 0.f;
                    xm.y = 0.f;
                }
                const float2 xmc = cconj(xm);
                const float2 d = cmul(csub(xk, xmc), cconj(twf[k]));
                return cadd(cadd(xk, xmc), mul_si<1>(d));
            }
            const bool two = o % tile + NXH < ra * NXH;
            const int kk = k < NXH ? k : nx - k;
            float2 a = A[o + kk], c = two ? A[o + NXH + kk] : c2(0.f, 0.f);
            if (k == 0) {
                a.y = 0.f;
                c.y = 0.f;
            }
            if (k >= NXH) {
                a.y = -a.y;
                c.y = -c.y;
            }
            return c2(a.x - c.y, a.y + c.x);
        };
        auto row_at = [&](int f) { return f * PZ; };
        x_stage<RL, 1, 0>(A, 3 * nrow, twx, row_at, pre);
        auto ldrow = [&](int o, int e) { return A[o + e]; };
        if constexpr (XP::P.ns == 3) x_stage<RL, 1, 1>(A, 3 * nrow, twx, row_at, ldrow);
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
                const double var = fma(-ad, ad, (double)isd[q] * nv);
                const float r = __builtin_amdgcn_rsqf((float)var);
                isd[q] = r;
                if (EXACT) {
                    // one Newton step, its correction formed in FP64 (0: r stays inf)
                    const float c = (float)fma(-0.5 * var * (double)r, (double)r, 0.5);
                    isd[q] = var == 0.0 ? r : fmaf(r, c, r);
                }
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

template <bool ODD, int RL, bool EXACT>
int launch_resid(const Fft3D& f, const FusedArgs& a, const ResSplit& sp, int which, int nplanes,
                 int zr, hipStream_t s) {
    ResArgs g{f.nz, f.ny, f.nx, sp.r1, sp.r2, a.rmap, (int64_t)f.nz * a.rmap.ps};
    const int ng = which == 0 ? (a.binary_mask ? 2 : 3) : 3;
    const size_t lds = res_lds(RL, ODD, g.m.ra, ng);
    if (which == 0) {
        const int zlo = nplanes < f.nz ? -zr : 0;
        hipLaunchKernelGGL((k_fwd_resid<ODD, RL, EXACT>), dim3((unsigned)(g.m.rb * nplanes * a.nrot)),
                           dim3(sp.nthr), lds, s, a.tm, a.occ, a.rots, g, a.rmax, zr * zr, zlo,
                           nplanes, ng, a.work, f.twx, f.twy, f.twfull);
        return launched("k_fwd_resid");
    }
    const int nch = (a.nrot + a.chunk_lcc - 1) / a.chunk_lcc;
    hipLaunchKernelGGL((k_inv_resid<ODD, RL, EXACT>), dim3((unsigned)(g.m.rb * f.nz * nch)),
                       dim3(sp.nthr), lds, s, a.work, a.lcc_mask, a.keys, g, a.nrot, a.chunk_lcc,
                       a.first, a.norm, f.twx, f.twy, f.twfull);
    return launched("k_inv_resid");
}

template <bool ODD, int RL, bool EXACT>
int allow_resid() {
    PF_CHECK_STATUS(allow_lds((const void*)k_fwd_resid<ODD, RL, EXACT>, 80 * 1024));
    return allow_lds((const void*)k_inv_resid<ODD, RL, EXACT>, 80 * 1024);
}

// Stage `which` with the kernels of the x length (its LDS allowance when which < 0).
template <bool EXACT>
int dispatch_resid(const Fft3D& f, const FusedArgs& a, const ResSplit& sp, int which, int nplanes,
                   int zr, hipStream_t s) {
#define PF_XCASE(ODD, L) \
    case L:              \
        return which < 0 ? allow_resid<ODD, L, EXACT>() \
                         : launch_resid<ODD, L, EXACT>(f, a, sp, which, nplanes, zr, s);
#define PF_XODD(L) PF_XCASE(true, L)
#define PF_XEVEN(L) PF_XCASE(false, L)
    if (f.nx % 2) {
        switch (f.nx) { PF_CT_ODD_LENGTHS(PF_XODD) }
    } else {
        switch (f.nx / 2) { PF_CT_ROW_LENGTHS(PF_XEVEN) }
    }
#undef PF_XEVEN
#undef PF_XODD
#undef PF_XCASE
    set_error("residue stages: no compiled transform for x length %d", f.nx);
    return kErrUnsupported;
}

}  // namespace

// EXACT kernels (pf_resid_exact.hip).
int dispatch_resid_exact(const Fft3D& f, const FusedArgs& a, const ResSplit& sp, int which,
                         int nplanes, int zr, hipStream_t s);

}  // namespace pf
