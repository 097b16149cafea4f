// Adjoint kernels for gfx950: the two passes of the discrete adjoint step
// (capaz_adjoint.h) and the observation gathers of the history-matching
// objective.  One thread per cell, x fastest: a wavefront reads rows of 64 (the
// tiles of pass 2: 32) consecutive doubles of every field it touches, as the
// forward kernels do.
#include <hip/hip_runtime.h>

#include "capaz_adjoint.h"
#include "capaz_adjoint_launch.h"
#include "capaz_fused.h"
#include "capaz_launch.h"

namespace capaz {

namespace {

constexpr int kAdjBlock = 64;

template <int IT>
__global__ void __launch_bounds__(kAdjBlock) k_adj_newton(DevParams p, AdjIO a) {
    const int i = (int)blockIdx.x * kAdjBlock + (int)threadIdx.x, j = (int)blockIdx.y, k = (int)blockIdx.z;
    if (i >= p.Nx || !interior3(p, i, j, k)) return;
    adj_newton_cell<IT>(p, a, i, j, k, (int64_t)i + (int64_t)j * p.sy + (int64_t)k * p.sz);
}

// Interior cells, densely numbered (every lane of a wavefront has a cell).
template <int IT>
__global__ void __launch_bounds__(256) k_adj_newton_rec(DevParams p, AdjIO a, const double* div, int64_t stride,
                                                        uint32_t ni, uint32_t nj, uint32_t total) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t >= total) return;
    int i, j, k;
    box_cell(t, ni, nj, p.Nx >= 3 ? 1 : 0, 1, p.Nz >= 3 ? 1 : 0, i, j, k);
    adj_newton_recorded<IT>(p, a, i, j, k, (int64_t)i + (int64_t)j * p.sy + (int64_t)k * p.sz, div, stride);
}

// Every cell, in memory order.  Four waves per SIMD (128 VGPRs; the
// compiler's own choice of 130 allows three) hide more of the neighbours'
// load latency, at the cost of a 12-byte spill.
// The grid is a multiple of the 8 XCDs; each XCD takes a contiguous run of
// cells (workgroups go to the XCDs round robin), so the z neighbours a cell
// gathers from were read by the same XCD and hit its L2.
// CL: the closure (1 Corey, 0 the reference's van Genuchten).
template <int CL>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_adj_coef(DevParams p, AdjIO a) {
    const uint32_t b = (blockIdx.x % 8u) * (gridDim.x / 8u) + blockIdx.x / 8u;
    const uint32_t t = b * 256u + threadIdx.x;
    if (t >= (uint32_t)p.n) return;
    int i, j, k;
    box_cell(t, (uint32_t)p.Nx, (uint32_t)p.Ny, 0, 0, 0, i, j, k);
    adj_coef_cell<CL>(p, a, i, j, k, (int64_t)t);
}

// Two phases: pass 1 over the interior cells (dense numbering), pass 2 over
// every cell (XCD-contiguous runs, as k_adj_coef).
template <int IT>
__global__ void __launch_bounds__(256) k_adj2_newton_rec(DevParams p, AdjIO a, const double* div, int64_t stride,
                                                         uint32_t ni, uint32_t nj, uint32_t total) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t >= total) return;
    int i, j, k;
    box_cell(t, ni, nj, 1, 1, p.Nz >= 3 ? 1 : 0, i, j, k);
    adj2_newton_recorded<IT>(p, a, i, j, k, (int64_t)i + (int64_t)j * p.sy + (int64_t)k * p.sz, div, stride);
}

template <bool N2>
__global__ void __launch_bounds__(256) k_adj2_coef(DevParams p, AdjIO a) {
    const uint32_t b = (blockIdx.x % 8u) * (gridDim.x / 8u) + blockIdx.x / 8u;
    const uint32_t t = b * 256u + threadIdx.x;
    if (t >= (uint32_t)p.n) return;
    int i, j, k;
    box_cell(t, (uint32_t)p.Nx, (uint32_t)p.Ny, 0, 0, 0, i, j, k);
    adj2_coef_cell<N2>(p, a, i, j, k, (int64_t)t);
}

// Tangent-linear step: interior cells (dense numbering), then the faces.
__global__ void __launch_bounds__(256) k_tan_interior(DevParams p, TanIO a, uint32_t ni, uint32_t nj, uint32_t total) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t >= total) return;
    int i, j, k;
    box_cell(t, ni, nj, p.Nx >= 3 ? 1 : 0, 1, p.Nz >= 3 ? 1 : 0, i, j, k);
    tan_cell<0>(p, a, i, j, k, (int64_t)i + (int64_t)j * p.sy + (int64_t)k * p.sz);
}

__global__ void __launch_bounds__(256) k_tan_faces(DevParams p, TanIO a) {
    int i, j, k;
    if (!face_cell(p, (int64_t)blockIdx.x * 256 + threadIdx.x, i, j, k)) return;
    tan_boundary(p, a, i, j, k);
}

// out_w[c] = S_w[cells[c]], out_n[c] = S_n[cells[c]]; Sw == NULL (two
// phases): S_w = 1 - S_n.
__global__ void k_obs_gather(const double* Sw, const double* Sn, const int64_t* cells, int64_t ncells, double* out_w,
                             double* out_n) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= ncells) return;
    const double sn = Sn[cells[c]];
    out_w[c] = Sw ? Sw[cells[c]] : 1. - sn;
    out_n[c] = sn;
}

// lam_S[cells[c]] += seen[c] - want[c] (cells distinct); lSw == NULL (two
// phases, S_w = 1 - S_n): the S_w mismatch goes to lam_S_n with a minus sign.
__global__ void k_obs_adjoint(double* lSw, double* lSn, const int64_t* cells, int64_t ncells, const double* seen_w,
                              const double* seen_n, const double* want_w, const double* want_n) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= ncells) return;
    const int64_t l = cells[c];
    if (lSw) {
        lSw[l] += seen_w[c] - want_w[c];
        lSn[l] += seen_n[c] - want_n[c];
    } else {
        lSn[l] += (seen_n[c] - want_n[c]) - (seen_w[c] - want_w[c]);
    }
}

// ---- tiled passes: the z-marching tiles of the fused step -------------------

// Pass 1 as the fused step's epilogue: the tile computes the cell's
// coefficients and flux divergence exactly as the step does, then runs the
// Newton iteration backwards instead of forwards.
template <int IT>
struct AdjNewtonStore {
    AdjIO a;
    static constexpr bool kLeaves = false;
    __device__ __forceinline__ int none() const { return 0; }
    template <class At>
    __device__ __forceinline__ int prefetch(const At&) const { return 0; }
    template <class At>
    __device__ __forceinline__ void cell(const DevParams& p, const DevParams&, int i, int j, int k, const At& at,
                                         const CellState<3>& s, const double* div, int, uint32_t&, uint32_t) const {
        adj_newton_tail<IT>(p, a, i, j, k, at.l(), s.ro, s.P, s.Sw, s.Sn, div);
    }
};

constexpr int kTX = 64, kTY = 8;

template <int CLOSURE, int IT>
__global__ void __launch_bounds__(kTX * kTY) k_adj_newton_z(DevParams p, StepIO io, AdjIO a, int kchunk) {
    __shared__ FusedLds<3, CLOSURE, kTX, kTY, kAxesAny> lds;
    fused_z_tile<3, CLOSURE, kTX, kTY, kAxesAny>(p, kernel_params(), kernel_io(), io, kchunk, (int)blockIdx.x, (int)blockIdx.y,
                                              (int)blockIdx.z, lds, AdjNewtonStore<IT>{a});
}

// Pass 2 on tiles of 32 x 8 columns (every cell, boundary included) marching
// kchunk planes: each cell's pressures, L = -Xi ro, ro and mu are formed once
// (and once more where another tile's ring holds it) and staged in LDS with a
// one-cell ring for the x and y neighbours; a z face's driving force and upwind L
// are carried from the plane below.  The values of adj_coef_cell, with its terms
// in its order: a neighbour that is not interior, or does not exist, counts with
// mu = 0 (the cells past the grid repeat the one before them).
//
// Bound by VALU issue and, at three waves per SIMD, by latency; the cell-by-cell
// pass forms each cell's coefficients seven times (1608 instructions per cell):
// 96^3, Corey-2, 42 us against 54.  159 VGPRs; four waves spill 31 of them (58
// us), 32 x 16 workgroups, one per CU, 116.  One plane's LDS and two barriers per
// plane; the next plane's loads are issued before this plane's terms.
struct AdjRaw {
    double Pw[1], Sw[1], Sn[1], K[1], Pn[1], Pg[1], mu[3];  // arrays of one, as coef_v reads them
};
struct AdjCell {
    double P[3], L[3], ro[3], mu[3];
};
template <class At>
__device__ __forceinline__ void adj_load(const AdjIO& a, const At& at, bool inner, AdjRaw& r) {
    r.Pw[0] = ld(a.Pw, at);
    r.Sw[0] = ld(a.Sw, at);
    r.Sn[0] = ld(a.Sn, at);
    r.K[0] = ld(a.K, at);
    if (inner) {
        r.mu[0] = ld(a.mu_w, at);
        r.mu[1] = ld(a.mu_n, at);
        r.mu[2] = ld(a.mu_g, at);
    } else {
        r.Pn[0] = ld(a.Pn, at);
        r.Pg[0] = ld(a.Pg, at);
        r.mu[0] = r.mu[1] = r.mu[2] = 0.;
    }
}
template <int CL>
__device__ __forceinline__ void adj_cell(const DevParams& p, const AdjRaw& r, bool inner, AdjCell& c) {
    const Coef v = coef_v<CL>(p, r, 0, inner);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        c.P[a] = v.P[a];
        c.L[a] = -v.Xi[a] * v.ro[a];
        c.ro[a] = v.ro[a];
        c.mu[a] = r.mu[a];
    }
}
// The upwind L of a face whose driving force is x: Lm of its minus side for x >
// 0, Lp of its plus side for x < 0, their mean else (upwind_w).
__device__ __forceinline__ double upwind_L(double x, double Lm, double Lp) {
    const double t = 0.5 * Lm + 0.5 * Lp;
    return x > 0. ? Lm : (x < 0. ? Lp : t);
}
// adj_coef_axis's terms of one phase from the driving forces and upwind Ls of the
// own flux's faces (x1, T1, x2, T2) and of the two neighbours' fluxes there.
__device__ __forceinline__ void adj_terms(double x1, double T1, double x2, double T2, double xm, double Tm, double xq,
                                          double Tq, double mu, double mum, double muq, double rh, double& lP,
                                          double& lL) {
    const double d1 = -(T1 * rh), d2 = T2 * rh;
    lP += mu * (d2 - d1) * rh;
    lL += mu * ((pos_part(x2) - neg_part(x1)) * rh);
    lP += muq * -(Tq * rh) * rh;
    lL += muq * (-pos_part(xq) * rh);
    lP += mum * (-(Tm * rh) * rh);
    lL += mum * (neg_part(xm) * rh);
}

template <int CL, int TX, int TY>
__global__ void __launch_bounds__(TX * TY) __attribute__((amdgpu_waves_per_eu(CL == 0 ? 2 : 3)))
k_adj_coef_z(DevParams p, AdjIO a, int kchunk) {
    static_assert((TX == 32 || TX == 64) && TX >= 2 * TY && TY >= 3, "whole rows per wavefront; ring cells of three rows");
    constexpr int NV = 13, ROW = (TX + 2) * NV;  // an odd count: a row's reads of one value on distinct banks
    __shared__ double lds[TY + 2][TX + 2][NV];
    int bx, by, bz;
    xcd_tile(bx, by, bz);
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int i0 = TX * bx, j0 = TY * by, k0 = kchunk * bz, k1 = min(p.Nz - 1, k0 + kchunk - 1);
    const int i = i0 + tx, j = j0 + ty;
    const bool own = i < p.Nx && j < p.Ny, hasx = p.Nx >= 2, hasz = p.Nz >= 2;
    const int ic = min(i, p.Nx - 1), jc = min(j, p.Ny - 1);
    const int jw = __builtin_amdgcn_readfirstlane(jc);
    CellAt at{(int64_t)i0 + (int64_t)jw * p.sy + (int64_t)k0 * p.sz, 8u * (uint32_t)(ic - i0)};
    if (TX < 64) at.off += 8u * (uint32_t)(jc - jw) * (uint32_t)p.sy;
    const bool own_ij = own && inner_ij<3>(p, ic, jc);
    // ring cell of this thread, clamped into the grid
    int hi = 0, hj = 0, hx = 0, hy = 0;
    if (ty == 0) { hi = i; hj = j0 - 1; hx = tx + 1; hy = 0; }
    else if (ty == 1) { hi = i; hj = j0 + TY; hx = tx + 1; hy = TY + 1; }
    else { hi = tx < TY ? i0 - 1 : i0 + TX; hj = j0 + (tx & (TY - 1)); hx = tx < TY ? 0 : TX + 1; hy = (tx & (TY - 1)) + 1; }
    const bool halo = ty < 2 || (ty == 2 && tx < 2 * TY);
    const bool halo_ij = hi >= 0 && hi < p.Nx && hj >= 0 && hj < p.Ny && inner_ij<3>(p, hi, hj);
    hi = min(max(hi, 0), p.Nx - 1);
    hj = min(max(hj, 0), p.Ny - 1);
    const int64_t hcol = (int64_t)hi + (int64_t)hj * p.sy;

    const LdsDouble v0 = (LdsDouble)&lds[ty + 1][tx + 1][0], vh = (LdsDouble)&lds[hy][hx][0];
    auto stage = [&](LdsDouble w, const AdjCell& c) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            w[q] = c.P[q];
            w[3 + q] = c.L[q];
            w[6 + q] = c.ro[q];
            w[9 + q] = c.mu[q];
        }
    };

    AdjRaw r;
    // the face between this plane and the one below: its driving force and
    // upwind L, and the mu below
    double x1[3] = {0., 0., 0.}, T1[3] = {0., 0., 0.}, mum[3] = {0., 0., 0.};
    bool inner = own_ij && inner_k(p, k0);
    adj_load(a, at, inner, r);
    {
        AdjRaw rm, rh;
        AdjCell c, m;
        const bool inner_m = own_ij && k0 >= 1 && inner_k(p, k0 - 1), inner_h = halo_ij && inner_k(p, k0);
        if (k0 >= 1) adj_load(a, CellAt{at.base - p.sz, at.off}, inner_m, rm);
        if (halo) adj_load(a, CellIndex{hcol + (int64_t)k0 * p.sz}, inner_h, rh);
        adj_cell<CL>(p, r, inner, c);
        stage(v0, c);
        if (k0 >= 1) {
            adj_cell<CL>(p, rm, inner_m, m);
#pragma unroll
            for (int ph = 0; ph < 3; ++ph) {
                x1[ph] = -((c.P[ph] - m.P[ph]) * p.r_hz);
                T1[ph] = upwind_L(x1[ph], m.L[ph], c.L[ph]);
                mum[ph] = m.mu[ph];
            }
        }
        if (halo) {
            adj_cell<CL>(p, rh, inner_h, m);
            stage(vh, m);
        }
    }
    __syncthreads();
    for (int k = k0; k <= k1; ++k) {
        const bool next = k < k1, zp = hasz && k + 1 < p.Nz;
        const bool inner_q = own_ij && zp && inner_k(p, k + 1), inner_h = halo_ij && inner_k(p, k + 1);
        renew(at);
        AdjRaw rq, rh;
        if (zp) adj_load(a, CellAt{at.base + p.sz, at.off}, inner_q, rq);
        double lP[3], lL[3], lro[3];
        // the own cell's row of values and the rows below and above it, from x - 1 on
        LdsDouble row[3];
#pragma unroll
        for (int y = 0; y < 3; ++y) {
            row[y] = v0 + (y - 1) * ROW - NV;
            asm("" : "+v"(row[y]));
        }
        auto nb = [&](int q, int y, int x) { return row[y][x * NV + q]; };
#pragma unroll
        for (int ph = 0; ph < 3; ++ph) {
            lP[ph] = lL[ph] = lro[ph] = 0.;
            const double P = nb(ph, 1, 1), L = nb(3 + ph, 1, 1), mu = nb(9 + ph, 1, 1);
            if (hasx) {
                const double xa = -((P - nb(ph, 1, 0)) * p.r_hx), xb = -((nb(ph, 1, 2) - P) * p.r_hx);
                const double Ta = upwind_L(xa, nb(3 + ph, 1, 0), L), Tb = upwind_L(xb, L, nb(3 + ph, 1, 2));
                adj_terms(xa, Ta, xb, Tb, xa, Ta, xb, Tb, mu, nb(9 + ph, 1, 0), nb(9 + ph, 1, 2), p.r_hx, lP[ph], lL[ph]);
            }
            const double da = -((P - nb(ph, 0, 1)) * p.r_hy), db = -((nb(ph, 2, 1) - P) * p.r_hy);
            const double La = nb(3 + ph, 0, 1), Lb = nb(3 + ph, 2, 1), gc = p.g * nb(6 + ph, 1, 1);
            const double xa = da + gc, xb = db + gc, xm = da + p.g * nb(6 + ph, 0, 1), xq = db + p.g * nb(6 + ph, 2, 1);
            const double Ta = upwind_L(xa, La, L), Tb = upwind_L(xb, L, Lb);
            adj_terms(xa, Ta, xb, Tb, xm, upwind_L(xm, La, L), xq, upwind_L(xq, L, Lb), mu, nb(9 + ph, 0, 1),
                      nb(9 + ph, 2, 1), p.r_hy, lP[ph], lL[ph]);
            lro[ph] += mu * (-(Ta * p.r_hy) + Tb * p.r_hy) * p.g;
            // one phase's values in registers at a time: its sums are done here
            asm volatile("" : "+v"(lP[ph]), "+v"(lL[ph]), "+v"(lro[ph])::"memory");
        }
        if (next && halo) adj_load(a, CellIndex{hcol + (int64_t)(k + 1) * p.sz}, inner_h, rh);
        AdjCell q;
        if (zp) adj_cell<CL>(p, rq, inner_q, q);
        if (hasz) {
#pragma unroll
            for (int ph = 0; ph < 3; ++ph) {
                const double mu = nb(9 + ph, 1, 1);
                double x2 = 0., T2 = 0.;
                if (zp) {
                    x2 = -((q.P[ph] - nb(ph, 1, 1)) * p.r_hz);
                    T2 = upwind_L(x2, nb(3 + ph, 1, 1), q.L[ph]);
                }
                adj_terms(x1[ph], T1[ph], x2, T2, x1[ph], T1[ph], x2, T2, mu, mum[ph], zp ? q.mu[ph] : 0., p.r_hz,
                          lP[ph], lL[ph]);
                x1[ph] = x2;
                T1[ph] = T2;
                mum[ph] = mu;
            }
        }
        if (own) {
            const CoefD cd = coef_d<CL>(p, r, 0, inner);
            CellAt to = at;
            renew(to);
            adj_coef_finish(p, a, to.l(), cd, lP, lL, lro);
        }
        if (next) {
            r = rq;
            inner = inner_q;
            at.base += p.sz;
            __syncthreads();
            stage(v0, q);
            if (halo) {
                AdjCell h;
                adj_cell<CL>(p, rh, inner_h, h);
                stage(vh, h);
            }
            __syncthreads();
        }
    }
}

template <int CL>
hipError_t launch_adj_coef_tile(const DevParams& p, const AdjIO& a, hipStream_t s) {
    constexpr int TX = 32, TY = 8;
    constexpr auto kernel = k_adj_coef_z<CL, TX, TY>;
    const int kchunk = fused_kchunk(p, 0, TY, resident_groups<kernel>(TX * TY), TX);
    const dim3 grid((p.Nx + TX - 1) / TX, (p.Ny + TY - 1) / TY, (p.Nz + kchunk - 1) / kchunk);
    hipLaunchKernelGGL(kernel, grid, dim3(TX, TY), 0, s, p, a, kchunk);
    return hipGetLastError();
}
hipError_t launch_adj_coef_z(const DevParams& p, const AdjIO& a, hipStream_t s) {
    if (p.closure == 0) return launch_adj_coef_tile<0>(p, a, s);
    return p.corey_n == 2. ? launch_adj_coef_tile<2>(p, a, s) : launch_adj_coef_tile<1>(p, a, s);
}

// Planes per tile: enough workgroups to fill the GPU several times over,
// at most 16 planes (the fused step's default) and at least 2.
int adj_kchunk(int nz, int64_t tiles_xy) {
    int64_t kc = (nz * tiles_xy + 2047) / 2048;
    return (int)(kc < 2 ? 2 : (kc > 16 ? 16 : kc));
}

}  // namespace

hipError_t launch_adjoint_step_tiled(const DevParams& p, const AdjIO& a, hipStream_t s) {
    StepIO io{};
    io.Pw = a.Pw;
    io.Sw = a.Sw;
    io.Sn = a.Sn;
    io.Pn = a.Pn;
    io.Pg = a.Pg;
    io.m = a.m;
    io.K = a.K;
    io.dtm = a.dtm;
    const int nx = p.Nx >= 3 ? p.Nx - 2 : 1, ny = p.Ny - 2, nz = p.Nz >= 3 ? p.Nz - 2 : 1;
    const int64_t txy = (int64_t)((nx + kTX - 1) / kTX) * ((ny + kTY - 1) / kTY);
    const int kc1 = adj_kchunk(nz, txy);
    const dim3 g1((unsigned)((nx + kTX - 1) / kTX), (unsigned)((ny + kTY - 1) / kTY), (unsigned)((nz + kc1 - 1) / kc1));
    const int closure = p.closure == 0 ? 0 : (p.corey_n == 2. ? 2 : 1);
#define CAPAZ_ADJ1(IT)                                                                                         \
    do {                                                                                                       \
        if (closure == 2)                                                                                      \
            hipLaunchKernelGGL((k_adj_newton_z<2, IT>), g1, dim3(kTX, kTY), 0, s, p, io, a, kc1);             \
        else if (closure == 1)                                                                                 \
            hipLaunchKernelGGL((k_adj_newton_z<1, IT>), g1, dim3(kTX, kTY), 0, s, p, io, a, kc1);             \
        else                                                                                                   \
            hipLaunchKernelGGL((k_adj_newton_z<0, IT>), g1, dim3(kTX, kTY), 0, s, p, io, a, kc1);             \
    } while (0)
    switch (p.iterations) {
        case 1: CAPAZ_ADJ1(1); break;
        case 2: CAPAZ_ADJ1(2); break;
        case 3: CAPAZ_ADJ1(3); break;
        case 4: CAPAZ_ADJ1(4); break;
        default: CAPAZ_ADJ1(0); break;
    }
#undef CAPAZ_ADJ1
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_adj_coef_z(p, a, s);
}

hipError_t launch_adjoint_coef(const DevParams& p, const AdjIO& a, hipStream_t s) {
    const dim3 grid((unsigned)((p.n + 255) / 256 + 7) / 8 * 8);
    if (p.closure == 0)
        hipLaunchKernelGGL(k_adj_coef<0>, grid, dim3(256), 0, s, p, a);
    else if (p.corey_n == 2.)
        hipLaunchKernelGGL(k_adj_coef<2>, grid, dim3(256), 0, s, p, a);
    else
        hipLaunchKernelGGL(k_adj_coef<1>, grid, dim3(256), 0, s, p, a);
    return hipGetLastError();
}

hipError_t launch_adjoint_step_recorded(const DevParams& p, const AdjIO& a, const double* div, int64_t stride,
                                        hipStream_t s) {
    const uint32_t ni = p.Nx >= 3 ? p.Nx - 2 : 1, nj = p.Ny - 2, nk = p.Nz >= 3 ? p.Nz - 2 : 1;
    const uint32_t total = ni * nj * nk;
    if (p.model == 2) {
        hipLaunchKernelGGL(k_adj2_newton_rec<0>, dim3((total + 255) / 256), dim3(256), 0, s, p, a, div, stride, ni, nj,
                           total);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const dim3 grid((unsigned)((p.n + 255) / 256 + 7) / 8 * 8);
        if (p.corey_n == 2.)
            hipLaunchKernelGGL(k_adj2_coef<true>, grid, dim3(256), 0, s, p, a);
        else
            hipLaunchKernelGGL(k_adj2_coef<false>, grid, dim3(256), 0, s, p, a);
        return hipGetLastError();
    }
    // the run-time iteration count: its loop holds fewer live registers
    // (144 VGPRs) than the fully unrolled fixed counts, without scratch
    hipLaunchKernelGGL(k_adj_newton_rec<0>, dim3((total + 255) / 256), dim3(256), 0, s, p, a, div, stride, ni, nj,
                       total);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_adj_coef_z(p, a, s);
}

hipError_t launch_adjoint_step(const DevParams& p, const AdjIO& a, hipStream_t s) {
    const dim3 grid((unsigned)((p.Nx + kAdjBlock - 1) / kAdjBlock), (unsigned)p.Ny, (unsigned)p.Nz);
    // the common iteration counts keep the Newton iterates in registers
    switch (p.iterations) {
        case 1: hipLaunchKernelGGL(k_adj_newton<1>, grid, dim3(kAdjBlock), 0, s, p, a); break;
        case 2: hipLaunchKernelGGL(k_adj_newton<2>, grid, dim3(kAdjBlock), 0, s, p, a); break;
        case 3: hipLaunchKernelGGL(k_adj_newton<3>, grid, dim3(kAdjBlock), 0, s, p, a); break;
        case 4: hipLaunchKernelGGL(k_adj_newton<4>, grid, dim3(kAdjBlock), 0, s, p, a); break;
        default: hipLaunchKernelGGL(k_adj_newton<0>, grid, dim3(kAdjBlock), 0, s, p, a); break;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_adjoint_coef(p, a, s);
}

hipError_t launch_tangent_step(const DevParams& p, const TanIO& a, hipStream_t s) {
    const uint32_t ni = p.Nx >= 3 ? p.Nx - 2 : 1, nj = p.Ny - 2, nk = p.Nz >= 3 ? p.Nz - 2 : 1;
    const uint32_t total = ni * nj * nk;
    hipLaunchKernelGGL(k_tan_interior, dim3((total + 255) / 256), dim3(256), 0, s, p, a, ni, nj, total);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int64_t nf = fused_face_cells(p);
    hipLaunchKernelGGL(k_tan_faces, dim3((unsigned)((nf + 255) / 256)), dim3(256), 0, s, p, a);
    return hipGetLastError();
}

hipError_t launch_obs_gather(const double* Sw, const double* Sn, const int64_t* cells, int64_t ncells, double* out_w,
                             double* out_n, hipStream_t s) {
    if (ncells <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_obs_gather, dim3((unsigned)((ncells + 255) / 256)), dim3(256), 0, s, Sw, Sn, cells, ncells,
                       out_w, out_n);
    return hipGetLastError();
}

hipError_t launch_obs_adjoint(double* lSw, double* lSn, const int64_t* cells, int64_t ncells, const double* seen_w,
                              const double* seen_n, const double* want_w, const double* want_n, hipStream_t s) {
    if (ncells <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_obs_adjoint, dim3((unsigned)((ncells + 255) / 256)), dim3(256), 0, s, lSw, lSn, cells, ncells,
                       seen_w, seen_n, want_w, want_n);
    return hipGetLastError();
}

}  // namespace capaz
