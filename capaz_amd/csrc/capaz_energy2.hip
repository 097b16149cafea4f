// The two-phase energy model's fused time step for gfx950 (the
// configurations' energy closure): one pass over the primary state (P_w,
// S_n, T) per step, reading the current arrays and writing the second ones.
//
// Per interior cell the step of the entry-point sequence is
//   roS (the 7-point upwind mass flux, cpu.cpp:619-731) from the closure
//       coefficients (P, Xi, ro) of the cell and its six neighbours,
//   E   (assign_E_current) of the cell,
//   E_new = E + dt (T_flow - E_flow): the conduction of T over the six
//       neighbours and the central difference of (ro H) u at them, where u
//       at a neighbour is its Darcy velocity (assign_u), a difference of P
//       at the cells on either side of it -- two cells from the centre;
//   the 4 x 4 Newton in (S_w, S_n, P_w, T) in registers,
// and the boundary cells take their new state from their inward cell
// (Border_S, Border_P, Border_T) in the same thread.
//
// Mapping.  A workgroup owns a TX x TY block of interior columns and marches a
// chunk of planes along z.  Per plane each thread stages its cell's
// coefficients in LDS; the ring of cells around the block (x and y
// neighbours of the edge cells) is staged too, and a second ring of
// pressures only (the far points of the neighbours' velocities).  Two planes'
// buffers and one barrier per plane: the next plane's loads are issued first,
// this plane's x and y terms cover them, then the next plane is staged, and
// the z terms and the Newton end the turn.  Along z each thread carries the
// minus face's flux parts and the (ro H) u_z products of planes k-1 and k, so
// each plane's u_z is computed once.  Every value is formed by the per-cell
// bodies' operations in their order, so the step has the bits of the
// entry-point sequence (capaz_bodies.h).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "capaz_fused.h"
#include "capaz_launch.h"

namespace capaz {

namespace {

struct E2IO {
    const double *Pw, *Sn, *T, *m, *K;  // current state and parameters
    double *Pw1, *Sn1, *T1;             // next state
};

// The parameters of a part of a plane's work (fresh()); ecfg as a constant.
template <int CLOSURE>
__device__ __forceinline__ DevParams e2_coef_params(ConstParams* q) {
    DevParams p = coef_params<2, CLOSURE>(q);
    p.ecfg = 1;
    p.mu_T_a = q->mu_T_a, p.mu_T_ref = q->mu_T_ref;
    p.H0_w = q->H0_w, p.H0_n = q->H0_n;
    p.lam_eff = q->lam_eff;
    return p;
}
__device__ __forceinline__ DevParams e2_flux_params(ConstParams* q) {
    DevParams p = flux_params(q);
    p.hx2 = q->hx2, p.r_hx2 = q->r_hx2, p.hy2 = q->hy2, p.r_hy2 = q->r_hy2, p.hz2 = q->hz2, p.r_hz2 = q->r_hz2;
    return p;
}
__device__ __forceinline__ DevParams e2_newton_params(ConstParams* q) {
    DevParams p;
    p.ecfg = 1;
    p.iterations = q->iterations;
    p.dt = q->dt;
    p.P_atm = q->P_atm;
    p.ro0_w = q->ro0_w, p.beta_w = q->beta_w;
    p.ro0_n = q->ro0_n, p.beta_n = q->beta_n;
    p.H0_w = q->H0_w, p.H0_n = q->H0_n, p.H0_r = q->H0_r;
    p.c_r = q->c_r, p.ro_r = q->ro_r;
    return p;
}

// A cell's values as read (loaded ahead of their use) and the coefficients
// that a neighbour reads: Xi, density and density * enthalpy of the phases,
// lambda_eff * T, and the pressures (one but for a capillary pressure).
struct E2Raw {
    double Pw, Sn, T, K;
};
template <int CLOSURE>
constexpr int kE2P = CLOSURE == 0 ? 2 : 1;
template <int CLOSURE>
struct E2Coef {
    double P[kE2P<CLOSURE>], Xi[2], ro[2], roH[2], LT;
};

template <class At>
__device__ __forceinline__ void e2_load(const E2IO& io, const At& at, E2Raw& r) {
    r.Pw = ld(io.Pw, at);
    r.Sn = ld(io.Sn, at);
    r.T = ld(io.T, at);
    r.K = ld(io.K, at);
}
// The pressures of a cell: P_w and, with a capillary pressure, P_w + P_k
// (two-phase.cpp:4-23).
template <int CLOSURE, class At>
__device__ __forceinline__ void e2_pressures(const DevParams& p, const E2IO& io, const At& at, double* P) {
    P[0] = ld(io.Pw, at);
    if constexpr (CLOSURE == 0) {
        double kw, kn, Pk;
        relperm2(p, ld(io.Sn, at), kw, kn, Pk);
        P[1] = P[0] + Pk;
    }
}

// assign_P_Xi + assign_ro + assign_H of a cell (body_P_Xi_ro, body_HE).
template <int CLOSURE>
__device__ __forceinline__ void e2_coef(const DevParams& p, const E2Raw& r, E2Coef<CLOSURE>& c) {
    double mKw, mKn;  // -K k_r
    c.P[0] = r.Pw;
    if constexpr (CLOSURE >= 1) {
        const double se = exact_div(1. - r.Sn - p.S_wr, p.den2c, p.r_den2c);
        mKw = corey_mK<CLOSURE>(p, r.K, se);
        mKn = corey_mK<CLOSURE>(p, r.K, 1. - se);
    } else {
        double kw, kn, Pk;
        relperm2(p, r.Sn, kw, kn, Pk);
        mKw = (-1.) * r.K * kw;
        mKn = (-1.) * r.K * kn;
        c.P[kE2P<CLOSURE> - 1] = r.Pw + Pk;
    }
    const double decay = exp_t(-p.mu_T_a * (r.T - p.mu_T_ref));  // mu_cfg's factor
    c.Xi[0] = mKw / (p.mu_w * decay);
    c.Xi[1] = mKn / (p.mu_n * decay);
    c.ro[0] = ro_w_T(p, r.Pw, r.T);
    c.ro[1] = ro_n_T(p, c.P[kE2P<CLOSURE> - 1], r.T);
    c.roH[0] = c.ro[0] * H_w_of(p, r.T);
    c.roH[1] = c.ro[1] * H_n_T(p, r.T);
    c.LT = p.lam_eff * r.T;
}

// Boundary cell (bi, bj, bk) from its inward cell's new state (Border_S and
// Border_P, two-phase.cpp:163-215, with the fixed bottom pressure; Border_T
// with the configuration's face temperatures).
__device__ __forceinline__ void e2_write_boundary(const DevParams& p, const E2IO& io, int bi, int bj, int bk,
                                                  double Pw, double Sn, double T, double ro_eff) {
    const int64_t lb = (int64_t)bi + (int64_t)bj * p.sy + (int64_t)bk * p.sz;
    double Snb = Sn;
    if (bj == 0 && p.source > 0 && in_source_window(p, bi, bk)) Snb = p.S_n_gr;
    io.Sn1[lb] = Snb;
    double Pb;
    if ((bj != 0) && (bj != p.Ny - 1))
        Pb = Pw;
    else if (bj == 0)
        Pb = p.P_atm;
    else if (p.P_bottom > 0)
        Pb = p.P_bottom;
    else
        Pb = Pw + ro_eff;
    io.Pw1[lb] = Pb;
    io.T1[lb] = border_T_cfg(p, bj, T);
}

// The boundary cells whose inward cell is the interior cell (i, j, k), from its
// new state; the cell's previous one still stands in the arrays read.
template <int CLOSURE>
__device__ __forceinline__ void e2_store_faces(const DevParams& p, const E2IO& io, int i, int j, int k) {
    const bool hasz = p.Nz >= 3;
    const bool xl = i == 1, xh = i == p.Nx - 2;
    const bool yl = j == 1, yh = j == p.Ny - 2;
    const bool zl = hasz && k == 1, zh = hasz && k == p.Nz - 2;
    const CellIndex at{(int64_t)i + (int64_t)j * p.sy + (int64_t)k * p.sz};
    const double Pw = ld(io.Pw1, at), Sn = ld(io.Sn1, at), T = ld(io.T1, at);
    double ro_eff = 0.;
    if (yh && !(p.P_bottom > 0)) {
        // ro_eff_gdy (main.cpp:255-267): this step's densities of the cell
        // (from its previous state), its new saturation
        double P0[2];
        e2_pressures<CLOSURE>(p, io, at, P0);
        const double T0 = ld(io.T, at);
        const double ro_w = ro_w_T(p, P0[0], T0), ro_n = ro_n_T(p, P0[kE2P<CLOSURE> - 1], T0);
        ro_eff = (ro_n * Sn + ro_w * (1 - Sn)) * ld(io.m, at) * p.g * p.hy;
    }
    // 0, -1 next to a low face, +1 next to a high one
    for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b)
            for (int d = 0; d < 3; ++d) {
                if ((a == 1 && !xl) || (a == 2 && !xh) || (b == 1 && !yl) || (b == 2 && !yh) || (d == 1 && !zl) ||
                    (d == 2 && !zh) || !(a || b || d))
                    continue;
                e2_write_boundary(p, io, i + (a == 2) - (a == 1), j + (b == 2) - (b == 1), k + (d == 2) - (d == 1), Pw,
                                  Sn, T, ro_eff);
            }
}

// LDS of a tile, for the plane being read and the one being staged: the
// pressures of the block and two rings, the other coefficients of the block
// and one ring, a cell's values together (7: an odd count puts a row's reads
// of one value on distinct banks).
template <int CLOSURE, int TX, int TY>
struct E2Lds {
    double P[2][TY + 4][TX + 4][kE2P<CLOSURE>];
    double C[2][TY + 2][TX + 2][7];  // Xi_w, Xi_n, ro_w, ro_n, roH_w, roH_n, lambda_eff * T
};

// One tile.  Bound by VALU issue (FP64), 1290 instructions per cell at 4 Newton
// iterations, 840 of them the Newton's.  256 x 256 x 128, Corey-2: 381 us per
// step (408 with S_n, T and lambda_eff * T kept across the Newton, whose loop
// then spilled) against 866 for one workgroup per CU with 215 VGPRs, a called Newton
// and parameters in vector-register lanes (2510 instructions).  Blocks of
// 32 x 16: their two planes' LDS (80 KB) lets two workgroups share a CU and
// their rings re-evaluate 20% of the cells; 64 x 8 (87 KB, 29%) takes 499 us.
// Cells whose Newton needs the pivot search leave its right side in their
// place of the next state and are done after the planes, with no register
// held for them; so are the boundary cells, from what their inward cells then
// hold.  kchunk <= kMaxPlanes.
// cp: p in constant memory (fresh()).  HASZ: Nz >= 3 (else one plane without z
// terms).
template <int CLOSURE, int TX, int TY, bool HASZ>
__device__ __forceinline__ void e2_tile(const DevParams& p, ConstParams* cp, const E2IO& io, int kchunk,
                                        E2Lds<CLOSURE, TX, TY>& lds) {
    static_assert(TX == 32 || TX == 64, "whole rows per wavefront");
    static_assert(TY >= 7 && TX >= 2 * TY, "ring cells of six rows of the workgroup");
    constexpr int NP = kE2P<CLOSURE>;
    constexpr int ROW = (TX + 2) * 7, PLANE = (TY + 2) * ROW, PROW = (TX + 4) * NP, PPLANE = (TY + 4) * PROW;
    int bx, by, bz;
    xcd_tile(bx, by, bz);
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int klo = HASZ ? 1 : 0, khi = HASZ ? p.Nz - 2 : 0;
    const int i0 = 1 + TX * bx, j0 = 1 + TY * by;
    const int k0 = klo + kchunk * bz;
    const int k1 = min(khi, k0 + kchunk - 1);
    const int i = i0 + tx, j = j0 + ty;
    const bool active = i <= p.Nx - 2 && j <= p.Ny - 2;
    // the own column, clamped into the grid (lanes past it stage values that
    // no active lane reads); jw: the wavefront's first row
    const int ic = min(i, p.Nx - 1), jc = min(j, p.Ny - 1);
    const int jw = __builtin_amdgcn_readfirstlane(jc);
    CellAt own{(int64_t)i0 + (int64_t)jw * p.sy + (int64_t)k0 * p.sz, 8u * (uint32_t)(ic - i0)};
    if (TX < 64) own.off += 8u * (uint32_t)(jc - jw) * (uint32_t)p.sy;

    // This thread's ring cell of each plane, if any: ring 1 (coefficients)
    // for ty 0-2, ring 2 (pressures) for ty 4-6; (hx, hy) its place in the
    // pressure plane, whose origin is (i0 - 2, j0 - 2).
    int hi = -1, hj = -1;
    const bool ring1 = ty < 3;
    {
        const int d = ring1 ? 1 : 2, t = ring1 ? ty : ty - 4;
        if (t == 0) { hi = i; hj = j0 - d; }
        else if (t == 1) { hi = i; hj = j0 + TY - 1 + d; }
        else if (t == 2 && tx < TY) { hi = i0 - d; hj = j0 + tx; }
        else if (t == 2 && tx < 2 * TY) { hi = i0 + TX - 1 + d; hj = j0 + tx - TY; }
    }
    const bool halo = hi >= 0 && hi < p.Nx && hj >= 0 && hj < p.Ny;
    const int hx = hi - i0 + 2, hy = hj - j0 + 2;
    const HaloAt hat(p, i0 - 1, j0 - 1, hi, hj);

    // LDS places in the buffers of plane 0: the own and the ring cell
    const LdsDouble c0 = (LdsDouble)&lds.C[0][ty + 1][tx + 1][0], p0 = (LdsDouble)&lds.P[0][ty + 2][tx + 2][0];
    const LdsDouble ch = (LdsDouble)&lds.C[0][0][0][0] + (halo && ring1 ? (hy - 1) * ROW + (hx - 1) * 7 : 0);
    const LdsDouble ph = (LdsDouble)&lds.P[0][0][0][0] + (halo ? hy * PROW + hx * NP : 0);
    // assign_u's difference of P at the x and y neighbours (cpu.cpp:346-477):
    // over two cells, P at the cell beyond the neighbour against the own one;
    // over one, against the neighbour, at a face -- there twice the difference
    // is divided by 2 h, whose quotient has the same bits
    const int fxm = i == 1, fxp = i == p.Nx - 2, fym = j == 1, fyp = j == p.Ny - 2;
    const int oxm = (fxm - 2) * NP, oxp = (2 - fxp) * NP, oym = (fym - 2) * PROW, oyp = (2 - fyp) * PROW;

    auto stage_p = [&](LdsDouble w, const double* P) {
#pragma unroll
        for (int a = 0; a < NP; ++a) w[a] = P[a];
    };
    auto stage = [&](int k, LdsDouble w, LdsDouble wp, const E2Coef<CLOSURE>& c) {
        w += (k & 1) * PLANE;
        stage_p(wp + (k & 1) * PPLANE, c.P);
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            w[a] = c.Xi[a];
            w[2 + a] = c.ro[a];
            w[4 + a] = c.roH[a];
        }
        w[6] = c.LT;
    };
    // the difference of P that assign_u takes at plane k + 1 of the own column
    auto dPz = [&](const DevParams& pf, int k, double Pm, double Pc, double Pp) {
        if (k == 0) return exact_div(Pp - Pc, pf.hz, pf.r_hz);
        if (k == p.Nz - 1) return exact_div(Pc - Pm, pf.hz, pf.r_hz);
        return exact_div(Pp - Pm, pf.two_hz, pf.r_two_hz);
    };

    // carried along z: the minus face (directed()'s neg_part(x1) and t2) and the
    // (ro H) u_z products of planes k - 1 (gm) and k (gc); lambda_eff * T of plane
    // k - 1 stands in the own cell's place of the other buffer until plane k + 1
    // is staged there
    double zneg[NP], zt2[2] = {0., 0.}, gm[2] = {0., 0.}, gc[2] = {0., 0.};
#pragma unroll
    for (int a = 0; a < NP; ++a) zneg[a] = 0.;
    uint32_t undone = 0;
    {
        E2Raw r, rm, rh;
        double P2[NP] = {}, P1[NP] = {}, Ph[NP] = {};
        const DevParams pc = e2_coef_params<CLOSURE>(cp), pf = e2_flux_params(cp);
        e2_load(io, own, r);
        if (HASZ) {
            e2_load(io, CellAt{own.base - p.sz, own.off}, rm);
            e2_pressures<CLOSURE>(pc, io, CellAt{own.base + p.sz, own.off}, P1);
            if (k0 >= 2) e2_pressures<CLOSURE>(pc, io, CellAt{own.base - 2 * p.sz, own.off}, P2);
        }
        if (halo) {
            if (ring1) hat.with(p, k0, [&](const auto& at) { e2_load(io, at, rh); });
            else hat.with(p, k0, [&](const auto& at) { e2_pressures<CLOSURE>(pc, io, at, Ph); });
        }
        E2Coef<CLOSURE> c, m;
        e2_coef(pc, r, c);
        stage(k0, c0, p0, c);
        if (HASZ) {
            e2_coef(pc, rm, m);
            (c0 + ((k0 + 1) & 1) * PLANE)[6] = m.LT;
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                const double d = exact_div(c.P[q] - m.P[q], pf.hz, pf.r_hz);
                const double um = dPz(pf, k0 - 1, P2[q], m.P[q], c.P[q]), uc = dPz(pf, k0, m.P[q], c.P[q], P1[q]);
                zneg[q] = neg_part(-1. * d);
#pragma unroll
                for (int a = q; a < (NP == 1 ? 2 : q + 1); ++a) {
                    zt2[a] = directed_t2(-1. * d, m.Xi[a], m.ro[a]);
                    gm[a] = m.roH[a] * (m.Xi[a] * um);
                    gc[a] = c.roH[a] * (c.Xi[a] * uc);
                }
            }
        }
        if (halo) {
            if (ring1) {
                e2_coef(pc, rh, c);
                stage(k0, ch, ph, c);
            } else {
                stage_p(ph + (k0 & 1) * PPLANE, Ph);
            }
        }
    }
    __syncthreads();

    for (int k = k0; k <= k1; ++k) {
        const bool next = k < k1;
        renew(own);
        E2Raw r, rh;
        double P2 = 0., Sn2 = 0.;
        if (HASZ) {
            e2_load(io, CellAt{own.base + p.sz, own.off}, r);
            if (k + 1 != p.Nz - 1) {
                P2 = ld(io.Pw, CellAt{own.base + 2 * p.sz, own.off});
                if constexpr (NP == 2) Sn2 = ld(io.Sn, CellAt{own.base + 2 * p.sz, own.off});
            }
        }
        if (next && halo) {
            hat.with(p, k + 1, [&](const auto& at) {
                rh.Pw = ld(io.Pw, at);
                if (ring1 || NP == 2) rh.Sn = ld(io.Sn, at);
                if (ring1) {
                    rh.T = ld(io.T, at);
                    rh.K = ld(io.K, at);
                }
            });
        }
        // read again rather than kept from the plane before: registers
        const double m_c = ld(io.m, own), Sn_c = ld(io.Sn, own), T_c = ld(io.T, own);

        const DevParams pf = e2_flux_params(fresh(cp));
        // the own cell's row of coefficients and the rows below and above it, from
        // the cell at x - 1 on, and the own cell's pressure: one register each
        LdsDouble row[3], pp = p0 + (k & 1) * PPLANE;
#pragma unroll
        for (int y = 0; y < 3; ++y) {
            row[y] = c0 + (k & 1) * PLANE + (y - 1) * ROW - 7;
            asm("" : "+v"(row[y]));
        }
        asm("" : "+v"(pp));
        auto C_at = [&](int q, int y, int x) { return row[y][x * 7 + q]; };
        double div[2], T_flow = 0., E_flow = 0.;
        const double zLT = HASZ ? (c0 + ((k + 1) & 1) * PLANE)[6] : 0.;
        if (active) {
            double e[2][2];  // (ro H) u of the minus and plus neighbours
            const double LT2 = 2. * C_at(6, 1, 1);
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                const double P = pp[q], Pm = pp[q - NP], Pp = pp[q + NP];
                const double x1 = -1. * exact_div(P - Pm, pf.hx, pf.r_hx), x2 = -1. * exact_div(Pp - P, pf.hx, pf.r_hx);
                const double um = exact_div(__builtin_amdgcn_ldexp(P - pp[q + oxm], fxm), pf.two_hx, pf.r_two_hx);
                const double up = exact_div(__builtin_amdgcn_ldexp(pp[q + oxp] - P, fxp), pf.two_hx, pf.r_two_hx);
                const double s1 = (pos_part(x2) - neg_part(x1)) * (-1.), s2 = pos_part(x1) * (-1.),
                             s3 = neg_part(x2) * (-1.);
#pragma unroll
                for (int a = q; a < (NP == 1 ? 2 : q + 1); ++a) {
                    const double Xm = C_at(a, 1, 0), Xp = C_at(a, 1, 2);
                    const double t1 = s1 * C_at(a, 1, 1) * C_at(2 + a, 1, 1);
                    const double t2 = s2 * Xm * C_at(2 + a, 1, 0), t3 = s3 * Xp * C_at(2 + a, 1, 2);
                    div[a] = exact_div(t1 - t2 + t3, pf.hx, pf.r_hx);
                    e[a][0] = C_at(4 + a, 1, 0) * (Xm * um);
                    e[a][1] = C_at(4 + a, 1, 2) * (Xp * up);
                }
            }
            T_flow = exact_div(C_at(6, 1, 2) - LT2 + C_at(6, 1, 0), pf.hx2, pf.r_hx2);
            E_flow = exact_div(e[0][1] - e[0][0] + e[1][1] - e[1][0], pf.two_hx, pf.r_two_hx);
            // the x neighbours' values are done with before the y ones are read
            asm volatile("" ::: "memory");
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                const double P = pp[q], Pm = pp[q - PROW], Pp = pp[q + PROW];
                const double dm = exact_div(P - Pm, pf.hy, pf.r_hy), dp = exact_div(Pp - P, pf.hy, pf.r_hy);
                const double um = exact_div(__builtin_amdgcn_ldexp(P - pp[q + oym], fym), pf.two_hy, pf.r_two_hy);
                const double up = exact_div(__builtin_amdgcn_ldexp(pp[q + oyp] - P, fyp), pf.two_hy, pf.r_two_hy);
#pragma unroll
                for (int a = q; a < (NP == 1 ? 2 : q + 1); ++a) {
                    const double Xm = C_at(a, 0, 1), Xp = C_at(a, 2, 1), rm = C_at(2 + a, 0, 1), rp = C_at(2 + a, 2, 1);
                    div[a] = div[a] + flux_y(pf, dm, dp, C_at(a, 1, 1), C_at(2 + a, 1, 1), Xm, rm, Xp, rp);
                    e[a][0] = C_at(4 + a, 0, 1) * (Xm * (um - rm * pf.g));
                    e[a][1] = C_at(4 + a, 2, 1) * (Xp * (up - rp * pf.g));
                }
            }
            T_flow += exact_div(C_at(6, 2, 1) - LT2 + C_at(6, 0, 1), pf.hy2, pf.r_hy2);
            E_flow += exact_div(e[0][1] - e[0][0] + e[1][1] - e[1][0], pf.two_hy, pf.r_two_hy);
        }

        // the next plane: coefficients, staged in the other buffer
        asm volatile("" ::: "memory");
        E2Coef<CLOSURE> zp;
        double P2n[2] = {P2, 0.};
        {
            const DevParams pc = e2_coef_params<CLOSURE>(fresh(cp));
            if (HASZ) {
                e2_coef(pc, r, zp);
                if (next) stage(k + 1, c0, p0, zp);
                if constexpr (NP == 2) {
                    double kw, kn, Pk;
                    relperm2(pc, Sn2, kw, kn, Pk);
                    P2n[1] = P2 + Pk;
                }
            }
            if (next && halo) {
                if (ring1) {
                    E2Coef<CLOSURE> h;
                    e2_coef(pc, rh, h);
                    stage(k + 1, ch, ph, h);
                } else {
                    double Ph[2] = {rh.Pw, 0.};
                    if constexpr (NP == 2) {
                        double kw, kn, Pk;
                        relperm2(pc, rh.Sn, kw, kn, Pk);
                        Ph[1] = rh.Pw + Pk;
                    }
                    stage_p(ph + ((k + 1) & 1) * PPLANE, Ph);
                }
            }
        }
        asm volatile("" ::: "memory");
        double gp[2] = {0., 0.};
        if (active) {
            double Xi[2], ro[2];
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                Xi[a] = C_at(a, 1, 1);
                ro[a] = C_at(2 + a, 1, 1);
            }
            if (HASZ) {
                const double LT_c = C_at(6, 1, 1);
#pragma unroll
                for (int q = 0; q < NP; ++q) {
                    const double P = pp[q];
                    const double x2 = -1. * exact_div(zp.P[q] - P, pf.hz, pf.r_hz);
                    const double n2 = neg_part(x2), p2 = pos_part(x2);
                    const double s1 = (p2 - zneg[q]) * (-1.), s3 = n2 * (-1.), s2 = p2 * (-1.);
                    const double u = dPz(pf, k + 1, P, zp.P[q], P2n[q]);
#pragma unroll
                    for (int a = q; a < (NP == 1 ? 2 : q + 1); ++a) {
                        const double t1 = s1 * Xi[a] * ro[a], t3 = s3 * zp.Xi[a] * zp.ro[a];
                        div[a] = div[a] + exact_div(t1 - zt2[a] + t3, pf.hz, pf.r_hz);
                        zt2[a] = s2 * Xi[a] * ro[a];  // the next plane's minus face
                        gp[a] = zp.roH[a] * (zp.Xi[a] * u);
                    }
                    zneg[q] = n2;
                }
                T_flow += exact_div(zp.LT - 2. * LT_c + zLT, pf.hz2, pf.r_hz2);
                E_flow += exact_div(gp[0] - gm[0] + gp[1] - gm[1], pf.two_hz, pf.r_two_hz);
            } else {
                div[0] = div[0] + 0.;
                div[1] = div[1] + 0.;
            }
            // mass: roS = ro S - dt/m * div; energy: E (assign_E_current) and
            // E_new (assign_E_new); the 4 x 4 Newton
            const DevParams pn = e2_newton_params(fresh(cp));
            const double dtm = pn.dt / m_c;
            const double Sw_c = 1. - Sn_c;  // S_calculation
            const double roSw = ro[0] * (1. - Sn_c) - dtm * div[0];
            const double roSn = ro[1] * Sn_c - dtm * div[1];
            const double E = (m_c * (Sw_c * (C_at(4, 1, 1) - pp[0]) + Sn_c * (C_at(5, 1, 1) - pp[NP - 1])) +
                              (1. - m_c) * (pn.ro_r * H_r_of(pn, T_c) - pp[0]));
            const double Q_hw = 0, Q_hr = 0;
            const double E_new = E + pn.dt * (T_flow + Q_hw + Q_hr - E_flow);
            double Sw = Sw_c, Sn = Sn_c, P = pp[0], T = T_c;
            const bool done = newton_energy2_fast(pn, Sw, Sn, P, T, m_c, roSw, roSn, E_new);
            CellAt to = own;
            renew(to);
            // a cell left undone: its Newton's right side, for after the planes
            if (__builtin_expect(!done, 0)) {
                P = roSw;
                Sn = roSn;
                T = E_new;
                undone |= 1u << (k - k0);
            }
            st(io.Pw1, to, P);
            st(io.Sn1, to, Sn);
            st(io.T1, to, T);
        }
        if (next) {
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                gm[a] = gc[a];
                gc[a] = gp[a];
            }
            own.base += p.sz;
            __syncthreads();
        }
    }

    if (!active) return;
    // the cells whose inverse needs the pivot search
    while (__builtin_expect(undone != 0, 0)) {
        const int k = k0 + __ffs(undone) - 1;
        undone &= undone - 1;
        const CellIndex at{(int64_t)i + (int64_t)j * p.sy + (int64_t)k * p.sz};
        const double roSw = ld(io.Pw1, at), roSn = ld(io.Sn1, at), E_new = ld(io.T1, at);
        double Sn = ld(io.Sn, at), P = ld(io.Pw, at), T = ld(io.T, at), Sw = 1. - Sn;
        double Hw = H_w_of(p, T), Hn = H_n_T(p, T), Hr = H_r_of(p, T);
        newton_energy2_t<false>(p, Sw, Sn, P, T, Hw, Hn, Hr, ld(io.m, at), roSw, roSn, E_new);
        st(io.Pw1, at, P);
        st(io.Sn1, at, Sn);
        st(io.T1, at, T);
    }
    const bool side = i == 1 || i == p.Nx - 2 || j == 1 || j == p.Ny - 2;
    for (int k = k0; k <= k1; ++k)
        if (side || (HASZ && (k == 1 || k == p.Nz - 2))) e2_store_faces<CLOSURE>(p, io, i, j, k);
}

// Two workgroups per CU (LDS and, at 4 waves per SIMD, 128 VGPRs), but for the
// closure with a capillary pressure, whose LDS (91.6 KB) allows one.
template <int CLOSURE>
constexpr int kE2Waves = CLOSURE == 0 ? 2 : 4;

template <int CLOSURE, int TX, int TY, bool HASZ>
__global__ void __launch_bounds__(TX * TY) __attribute__((amdgpu_waves_per_eu(kE2Waves<CLOSURE>)))
k_energy2_z(DevParams p, E2IO io, int kchunk) {
    __shared__ E2Lds<CLOSURE, TX, TY> lds;
    e2_tile<CLOSURE, TX, TY, HASZ>(p, kernel_params(), io, kchunk, lds);
}

template <int CLOSURE, bool HASZ>
hipError_t launch_e2(const DevParams& p, const E2IO& io, int kchunk, hipStream_t s, const KernelEvents* ev) {
    constexpr int TX = 32, TY = 512 / TX;
    const int nx = p.Nx - 2, ny = p.Ny - 2, nz = HASZ ? p.Nz - 2 : 1;
    constexpr auto kernel = k_energy2_z<CLOSURE, TX, TY, HASZ>;
    kchunk = fused_kchunk(p, kchunk, TY, resident_groups<kernel>(TX * TY), TX);
    const dim3 grid((nx + TX - 1) / TX, (ny + TY - 1) / TY, (nz + kchunk - 1) / kchunk);
    hipError_t e;
    if (ev && (e = hipEventRecord(ev->begin, s)) != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, grid, dim3(TX, TY), 0, s, p, io, kchunk);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    return ev ? hipEventRecord(ev->end, s) : hipSuccess;
}

template <int CLOSURE>
hipError_t launch_e2(const DevParams& p, const E2IO& io, int kchunk, hipStream_t s, const KernelEvents* ev) {
    return p.Nz >= 3 ? launch_e2<CLOSURE, true>(p, io, kchunk, s, ev) : launch_e2<CLOSURE, false>(p, io, kchunk, s, ev);
}

}  // namespace

hipError_t launch_energy2_step(const DevParams& p, const double* const* cur, double* const* next, int kchunk,
                               hipStream_t s, const KernelEvents* ev) {
    if (p.model != 2 || !p.energy || p.Nx < 3) return hipErrorInvalidValue;
    E2IO io{cur[0], cur[1], cur[2], cur[3], cur[4], next[0], next[1], next[2]};
    if (p.closure == 1 && p.corey_n == 2.) return launch_e2<2>(p, io, kchunk, s, ev);
    if (p.closure == 1) return launch_e2<1>(p, io, kchunk, s, ev);
    return launch_e2<0>(p, io, kchunk, s, ev);
}

}  // namespace capaz
