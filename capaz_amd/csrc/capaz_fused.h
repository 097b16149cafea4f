// The fused time-step kernel for gfx950: one pass over the primary state per
// time step (two- and three-phase models without the energy equation).
//
// Mapping.  A workgroup owns a TX x TY block of interior columns (x fastest,
// so each wavefront row streams TX consecutive doubles of every field) and a
// chunk of planes along z, which it walks plane by plane.  For the current
// plane the closure coefficients of each cell -- phase pressures, Xi and
// densities, the values the upwind flux reads from a neighbour -- are computed
// once and staged in LDS together with a one-cell halo ring, so the x and y
// neighbours come from LDS; the z face's flux terms are carried over from the
// previous plane (the same bits as recomputing them).
// After the divergence each thread solves its cell's Newton system in
// registers and writes the new state.  The boundary cells take theirs from
// their inward neighbours' new state (Border_S/Border_P, two-phase.cpp:163-215,
// three-phase.cpp:345-427): in the tiles for two phases and for three-phase
// grids whose workgroups all fit at once, else in an O(N^2) pass afterwards
// (k_fused_faces), which keeps the face logic out of the interior kernel's
// registers.
//
// Arithmetic is that of capaz_cell.h / capaz_bodies.h, so the kernel gives
// the entry-point sequence's bits.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "capaz_bodies.h"

namespace capaz {

// -K k_r of a phase with the Corey closure: exponent 2 (CLOSURE 2) or read
// from p (1).  For exponent 2 the clip to [0, 1] is one instruction (the clamp
// modifier, which makes a NaN 0), and a NaN s comes back through K: 0 * s + K
// is K for every finite s, and the quotient s is finite or NaN.
template <int CLOSURE>
__device__ __forceinline__ double corey_mK(const DevParams& p, double K, double s) {
    if constexpr (CLOSURE == 2) {
        const double c = fmin(fmax(s, 0.), 1.);
        return (-1.) * fma(0., s, K) * (c * c);
    } else {
        return (-1.) * K * corey_kr(p, s);
    }
}

// The two phases' densities of a cell in the state a step reads (body_P_Xi_ro).
template <int CLOSURE>
__device__ __forceinline__ void densities2(const DevParams& p, const StepIO& io, int64_t l, double* ro) {
    const double Pw = io.Pw[l];
    double Pn = Pw;
    if constexpr (CLOSURE == 0) {
        double kw, kn, Pk;
        relperm2(p, io.Sn[l], kw, kn, Pk);
        Pn = Pw + Pk;
    }
    ro[0] = ro_w_of(p, Pw);
    ro[1] = ro_n_of(p, Pn);
}

// Whether a cell is interior (interior_newton2, interior3), split into its (i, j)
// and k factors: a tile column evaluates the (i, j) factor once, so only one lane
// mask per column stays live across the planes.
template <int MODEL>
__device__ __forceinline__ bool inner_ij(const DevParams& p, int i, int j) {
    const bool ii = (i != 0) && (i != p.Nx - 1);
    return (MODEL == 2 ? ii : (ii || p.Nx < 2)) && (j != 0) && (j != p.Ny - 1);
}
__device__ __forceinline__ bool inner_k(const DevParams& p, int k) {
    return ((k != 0) && (k != p.Nz - 1)) || (p.Nz < 2);
}

// The new state (P_w, S_w, S_n, P_n, P_g) of boundary cell (bi, bj, bk) from
// its inward neighbour's new state (two phases: v[0] = P_w, v[2] = S_n).
template <int MODEL>
__device__ __forceinline__ void boundary_values(const DevParams& p, int bi, int bj, int bk, double Pw, double Sw,
                                                double Sn, double ro_eff, double* v) {
    if constexpr (MODEL == 2) {
        double Snb = Sn;
        if (bj == 0 && p.source > 0 && in_source_window(p, bi, bk)) Snb = p.S_n_gr;
        double Pb;
        if ((bj != 0) && (bj != p.Ny - 1))
            Pb = Pw;
        else if (bj == 0)
            Pb = p.P_atm;
        else if (p.P_bottom > 0)  // the configurations' fixed bottom pressure
            Pb = p.P_bottom;
        else
            Pb = Pw + ro_eff;
        v[0] = Pb;
        v[2] = Snb;
    } else {
        (void)bi;
        (void)bk;
        if (bj == 0 && p.source > 0) {
            v[1] = p.S_w_gr;
            v[2] = p.S_n_gr;
        } else {
            v[1] = Sw;
            v[2] = Sn;
        }
        border_p3(p, bj, Pw, v[0], v[3], v[4]);
    }
}

// Boundary cell (bi, bj, bk) from its inward neighbour's new state.
template <int MODEL>
__device__ __forceinline__ void write_boundary(const DevParams& p, const StepIO& io, int bi, int bj, int bk,
                                               double Pw, double Sw, double Sn, double ro_eff) {
    const int64_t lb = (int64_t)bi + (int64_t)bj * p.sy + (int64_t)bk * p.sz;
    double v[5];
    boundary_values<MODEL>(p, bi, bj, bk, Pw, Sw, Sn, ro_eff, v);
    io.Pw1[lb] = v[0];
    io.Sn1[lb] = v[2];
    if constexpr (MODEL == 3) {
        io.Sw1[lb] = v[1];
        io.Pn1[lb] = v[3];
        io.Pg1[lb] = v[4];
    }
}

// An epilogue with kWantsU = true also receives the cell's Darcy velocities
// u[phase][axis] (assign_u's central differences, cpu.cpp:346-477), from the
// neighbours' pressures the tile already holds.
template <class E, class = void>
struct EpiWantsU : std::false_type {};
template <class E>
struct EpiWantsU<E, std::void_t<decltype(E::kWantsU)>> : std::bool_constant<E::kWantsU> {};

// Pressures staged per cell: the phases' pressures are one value except where
// a closure has a capillary pressure (two phases, Brooks-Corey) and in the roS
// entry point (CLOSURE 3), which takes P_n and P_g of every cell as a caller set
// them.  Three phases otherwise: P_n = P_g = P_w in the interior and, once
// Border_P has run, on the x and z faces; the top and bottom rows' own P_n and
// P_g are staged apart.
template <int MODEL, int CLOSURE>
constexpr int kStagedP = MODEL == 2 ? (CLOSURE == 0 ? 2 : 1) : (CLOSURE == 3 ? 3 : 1);

// LDS of a tile: two planes' coefficients (P, Xi, ro) of the tile and its
// one-cell ring, the plane being read and the one being staged.  A cell's
// values lie together, so that a neighbour's are one address and constant
// offsets that a paired read reaches (an array per value needed ~20 address
// additions per cell); their number is odd, which puts 64 lanes' reads of one
// value on distinct banks.  Three phases with one staged pressure: edge[.][0 / 1]
// = P_n, P_g of the top / bottom row (j = 0 / Ny - 1) where the tile touches it,
// side[.][0 / 1] of the x face cells (i = 0 / Nx - 1), odd[.][row] = the plane k in
// which such a cell of that row has a P_n or P_g that is not its P_w (else any
// value, k too: side holds them whether they differ or not).
// The axes of the grids a kernel is compiled for: any; Nx, Ny, Nz >= 3 (no axis
// tests in the plane's code); one plane (Nz = 1: nothing carried along z, one
// plane's LDS, 52 to 88 VGPRs and no spills instead of 94 to 150, and what the
// epilogue reads is loaded before the barrier, whose latency is all such a grid
// waits for: us per step, one plane / any axes, 512 x 512 x 1 three phases Corey-2
// 13.0 / 18.2, van Genuchten 21.1 / 27.0, two phases Corey-2 6.8 / 9.3).
enum Axes { kAxesAny, kAxesAll, kAxesOnePlane };
template <int MODEL, int CLOSURE, int TX, int TY, int AXES>
struct FusedLds {
    static constexpr int kNP = kStagedP<MODEL, CLOSURE>, kNV = (kNP + 2 * MODEL) | 1;
    static constexpr bool kApart = MODEL == 3 && kNP == 1;
    static constexpr int kPlanes = AXES == kAxesOnePlane ? 1 : 2;
    double v[kPlanes][TY + 2][TX + 2][kNV];
    double edge[kPlanes][kApart ? 2 : 0][2][TX + 2], side[kPlanes][kApart ? 2 : 0][2][TY + 2];
    int odd[kPlanes][kApart ? TY + 2 : 0];
};

// A cell of a field array: a wave-uniform index (scalar registers) and the
// lane's own offset in bytes, which a load or store then takes as they are.
struct CellAt {
    int64_t base;
    uint32_t off;
    __device__ __forceinline__ int64_t l() const { return base + off / 8u; }
};
// The row's address in a scalar register pair and the lane's offset in one
// vector register, the two operands of a global access: left to itself the
// compiler adds the lane's offset to the field's address outside the plane
// loop (two vector registers per field) and the row to that for every access
// (a 64-bit add).  renew(): to be called in each block of code that accesses
// the cell, so that the offset is known to be a 32-bit value there.
__device__ __forceinline__ __attribute__((address_space(1))) char* row_of(const double* f, int64_t base) {
    auto* r = (__attribute__((address_space(1))) char*)(f + base);
    asm("" : "+s"(r));
    return r;
}
__device__ __forceinline__ void renew(CellAt& a) { asm volatile("" : "+v"(a.off)); }
__device__ __forceinline__ double ld(const double* f, const CellAt& a) {
    return *(__attribute__((address_space(1))) const double*)(row_of(f, a.base) + a.off);
}
// A cell by its own index alone.
struct CellIndex {
    int64_t i;
    __device__ __forceinline__ int64_t l() const { return i; }
};
__device__ __forceinline__ void renew(CellIndex&) {}
__device__ __forceinline__ double ld(const double* f, const CellIndex& a) { return f[a.i]; }
__device__ __forceinline__ void st(double* f, const CellIndex& a, double v) { f[a.i] = v; }
__device__ __forceinline__ void st(double* f, const CellAt& a, double v) {
    *(__attribute__((address_space(1))) double*)(row_of(f, a.base) + a.off) = v;
}

// A value compared in rarely taken code: the compiler otherwise makes the
// comparison's lane mask outside the plane loop and keeps it there, in scalar
// registers that the closures' constants need (van Genuchten: 8 more lane reads per
// closure evaluation, 1.2% of the step's VALU instructions).
__device__ __forceinline__ int seldom(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// A tile's halo cell (hi, hj) of a plane: from the cell below and left of the
// tile's first (i0, j0), whose index is uniform, a lane offset of up to 19
// rows, below 2^32 bytes for rows of at most kMaxRow32 cells (which leaves a
// factor of 25); with(k, f) calls f with the cell of plane k, by its own 64-bit index
// in wider grids.
constexpr int kMaxRow32 = 1 << 20;
struct HaloAt {
    int64_t base;
    uint32_t off;
    int i, j;
    __device__ __forceinline__ HaloAt(const DevParams& p, int i0, int j0, int hi, int hj)
        : base((int64_t)(i0 - 1) + (int64_t)(j0 - 1) * p.sy),
          off(8u * ((uint32_t)(hi - i0 + 1) + (uint32_t)(hj - j0 + 1) * (uint32_t)p.Nx)), i(hi), j(hj) {}
    template <class F>
    __device__ __forceinline__ void with(const DevParams& p, int k, const F& f) const {
        if (__builtin_expect(p.Nx <= kMaxRow32, 1)) {
            CellAt at{base + (int64_t)k * p.sz, off};
            renew(at);
            f(at);
        } else {
            f(CellIndex{(int64_t)i + (int64_t)j * p.sy + (int64_t)k * p.sz});
        }
    }
};

// The parameter block in constant memory.  The tiles hold more parameters
// than there are scalar registers; kept across the plane loop, the rest lived
// in lanes of vector registers, one v_readlane (a VALU slot) per word and use:
// some 45 per cell of the 256^3 Corey-2 step's 795.  fresh() makes the compiler
// read the ones a part of a plane's work needs where it begins (scalar loads).
using ConstParams = const __attribute__((address_space(4))) DevParams;
__device__ __forceinline__ ConstParams* fresh(ConstParams* p) {
    asm volatile("" : "+s"(p));
    return p;
}
// The kernel's first argument.
__device__ __forceinline__ ConstParams* kernel_params() {
    return (ConstParams*)__builtin_amdgcn_kernarg_segment_ptr();
}
// The field pointers in constant memory (the kernel's second argument), read again
// in every plane by the reference's closures, whose constants need the scalar
// registers: van Genuchten 256^3 455 M -> 449 M VALU instructions, 160 x 144 x 130
// 195.3 -> 193.3 us.
using ConstIO = const __attribute__((address_space(4))) StepIO;
__device__ __forceinline__ ConstIO* fresh(ConstIO* q) {
    asm volatile("" : "+s"(q));
    return q;
}
static_assert(sizeof(DevParams) % alignof(StepIO) == 0, "the second argument follows the first");
__device__ __forceinline__ ConstIO* kernel_io() { return (ConstIO*)(kernel_params() + 1); }
template <int CLOSURE>
__device__ __forceinline__ StepIO state_arrays(const StepIO& io, ConstIO* q) {
    StepIO now = io;
    if constexpr (CLOSURE == 0) {
        q = fresh(q);
        now.Pw = q->Pw, now.Sw = q->Sw, now.Sn = q->Sn, now.Pn = q->Pn, now.Pg = q->Pg, now.K = q->K;
    }
    return now;
}
// The parameters that coef_of / the fluxes / the Newton solves read.
template <int MODEL, int CLOSURE>
__device__ __forceinline__ DevParams coef_params(ConstParams* q) {
    DevParams p;
    if constexpr (CLOSURE == 3) return p;
    if constexpr (CLOSURE == 4) {
        p.P_atm = q->P_atm, p.r_P_atm = q->r_P_atm;
        p.ro0_w = q->ro0_w, p.beta_w = q->beta_w;
        p.ro0_n = q->ro0_n, p.beta_n = q->beta_n;
        p.ro0_g = q->ro0_g;
        return p;
    }
    p.closure = CLOSURE == 0 ? 0 : 1;
    if constexpr (CLOSURE == 0) p.pow_fast = q->pow_fast;
    p.P_atm = q->P_atm;
    p.mu_w = q->mu_w, p.r_mu_w = q->r_mu_w;
    p.mu_n = q->mu_n, p.r_mu_n = q->r_mu_n;
    p.ro0_w = q->ro0_w, p.beta_w = q->beta_w;
    p.ro0_n = q->ro0_n, p.beta_n = q->beta_n;
    p.S_wr = q->S_wr;
    if constexpr (CLOSURE == 1) p.corey_n = q->corey_n;
    if constexpr (MODEL == 2) {
        if constexpr (CLOSURE == 0) {
            p.den2 = q->den2, p.r_den2 = q->r_den2;
            p.bc_ew = q->bc_ew, p.bc_en = q->bc_en, p.bc_epk = q->bc_epk, p.P_d = q->P_d;
        } else {
            p.den2c = q->den2c, p.r_den2c = q->r_den2c;
        }
    } else {
        p.S_nr = q->S_nr, p.den3 = q->den3, p.r_den3 = q->r_den3;
        p.mu_g = q->mu_g, p.r_mu_g = q->r_mu_g;
        p.ro0_g = q->ro0_g, p.r_P_atm = q->r_P_atm;
        if constexpr (CLOSURE == 0) p.vg_a = q->vg_a, p.vg_b = q->vg_b, p.vg_c = q->vg_c;
    }
    return p;
}
__device__ __forceinline__ DevParams flux_params(ConstParams* q) {
    DevParams p;
    p.hx = q->hx, p.r_hx = q->r_hx, p.hy = q->hy, p.r_hy = q->r_hy, p.hz = q->hz, p.r_hz = q->r_hz, p.g = q->g;
    p.two_hx = q->two_hx, p.r_two_hx = q->r_two_hx, p.two_hy = q->two_hy, p.r_two_hy = q->r_two_hy;
    p.two_hz = q->two_hz, p.r_two_hz = q->r_two_hz;
    return p;
}
template <int MODEL, int CLOSURE>
__device__ __forceinline__ DevParams newton_params(ConstParams* q) {
    DevParams p;
    p.closure = CLOSURE == 0 ? 0 : 1;
    p.iterations = q->iterations;
    p.P_atm = q->P_atm;
    p.ro0_w = q->ro0_w, p.beta_w = q->beta_w;
    p.ro0_n = q->ro0_n, p.beta_n = q->beta_n;
    if constexpr (MODEL == 3) {
        p.ro0_g = q->ro0_g, p.r_P_atm = q->r_P_atm;
        p.c_wb = q->c_wb, p.c_nb = q->c_nb;
    } else if constexpr (CLOSURE == 0) {
        p.pow_fast = q->pow_fast;
        p.S_wr = q->S_wr, p.den2 = q->den2, p.r_den2 = q->r_den2, p.P_d = q->P_d;
        p.bc_epk = q->bc_epk, p.bc_eaaa = q->bc_eaaa, p.bc_pks_den = q->bc_pks_den, p.r_bc_pks_den = q->r_bc_pks_den;
    }
    return p;
}

// The values of a cell that its coefficients are made of, as read (loaded
// ahead of their use), and the coefficients themselves.
template <int MODEL, int CLOSURE>
struct CellRaw {
    double Pw, Sw, Sn, K, Pn, Pg, Xi[MODEL], ro[MODEL], T;
};
template <int MODEL, int CLOSURE>
struct CellCoef {
    double P[kStagedP<MODEL, CLOSURE>], Xi[MODEL], ro[MODEL];
};

template <int MODEL, int CLOSURE, class At>
__device__ __forceinline__ void load_raw(const StepIO& io, const At& at, bool inner, CellRaw<MODEL, CLOSURE>& r) {
    r.Pw = ld(io.Pw, at);
    r.Sn = ld(io.Sn, at);
    if constexpr (MODEL == 3) r.Sw = ld(io.Sw, at);
    if constexpr (CLOSURE >= 3) {
#pragma unroll
        for (int a = 0; a < MODEL; ++a) {
            r.Xi[a] = ld(io.Xi[a], at);
            if constexpr (CLOSURE == 3) r.ro[a] = ld(io.ro[a], at);
        }
        if constexpr (CLOSURE == 4) r.T = ld(io.T, at);
    } else {
        r.K = ld(io.K, at);
    }
    if constexpr (MODEL == 3) {
        if (!inner) {
            r.Pn = ld(io.Pn, at);
            r.Pg = ld(io.Pg, at);
        }
    }
}

// assign_P_Xi + assign_ro of one cell with the model and closure fixed at compile
// time (cpu.cpp:143-169; two-phase.cpp:4-23; three-phase.cpp:198-240) from what
// load_raw read.  CLOSURE 3 (three phases): the values of the P_n, P_g, Xi and ro
// arrays; 4, the energy step: Xi as its first pass stored it, ro from P and T.  The
// return value tells a cell whose P_n or P_g is not its P_w (three phases with one staged pressure,
// boundary cells).
template <int MODEL, int CLOSURE>
__device__ __forceinline__ bool coef_of(const DevParams& p, const CellRaw<MODEL, CLOSURE>& r, bool inner,
                                        CellCoef<MODEL, CLOSURE>& c) {
    c.P[0] = r.Pw;
    if constexpr (CLOSURE >= 3) {
        if constexpr (CLOSURE == 3) {
            c.P[1] = r.Pn;
            c.P[2] = r.Pg;
        }
#pragma unroll
        for (int a = 0; a < MODEL; ++a) {
            c.Xi[a] = r.Xi[a];
            if constexpr (CLOSURE == 3) c.ro[a] = r.ro[a];
        }
        if constexpr (CLOSURE == 4) {
            c.ro[0] = ro_w_T(p, r.Pw, r.T);
            c.ro[1] = ro_n_T(p, inner ? r.Pw : r.Pn, r.T);
            c.ro[2] = ro_g_T(p, inner ? r.Pw : r.Pg, r.T);
        }
    } else if constexpr (MODEL == 2) {
        double mKw, mKn;  // -K k_r
        if constexpr (CLOSURE >= 1) {
            const double se = exact_div(1. - r.Sn - p.S_wr, p.den2c, p.r_den2c);
            mKw = corey_mK<CLOSURE>(p, r.K, se);
            mKn = corey_mK<CLOSURE>(p, r.K, 1. - se);
        } else {
            double kw, kn, Pk;
            relperm2(p, r.Sn, kw, kn, Pk);
            mKw = (-1.) * r.K * kw;
            mKn = (-1.) * r.K * kn;
            c.P[1] = r.Pw + Pk;
        }
        c.Xi[0] = exact_div(mKw, p.mu_w, p.r_mu_w);
        c.Xi[1] = exact_div(mKn, p.mu_n, p.r_mu_n);
        c.ro[0] = ro_w_of(p, r.Pw);
        c.ro[1] = ro_n_of(p, CLOSURE >= 1 ? r.Pw : c.P[kStagedP<MODEL, CLOSURE> - 1]);
    } else {
        double mKw, mKn, mKg;  // -K k_r
        if constexpr (CLOSURE >= 1) {
            const double Swe = exact_div(r.Sw - p.S_wr, p.den3, p.r_den3);
            const double Sne = exact_div(r.Sn - p.S_nr, p.den3, p.r_den3);
            const double Sge = 1. - Swe - Sne;
            mKw = corey_mK<CLOSURE>(p, r.K, Swe);
            mKn = corey_mK<CLOSURE>(p, r.K, Sne);
            mKg = corey_mK<CLOSURE>(p, r.K, Sge);
        } else {
            double kw, kn, kg;
            relperm3(p, r.Sw, r.Sn, kw, kn, kg);
            mKw = (-1.) * r.K * kw;
            mKn = (-1.) * r.K * kn;
            mKg = (-1.) * r.K * kg;
        }
        c.Xi[0] = exact_div(mKw, p.mu_w, p.r_mu_w);
        c.Xi[1] = exact_div(mKn, p.mu_n, p.r_mu_n);
        c.Xi[2] = exact_div(mKg, p.mu_g, p.r_mu_g);
        c.ro[0] = ro_w_of(p, r.Pw);
        c.ro[1] = ro_n_of(p, r.Pw);
        c.ro[2] = ro_g_of(p, r.Pw);
    }
    if constexpr (MODEL == 3 && CLOSURE != 3) {
        if (!inner) {
            if constexpr (CLOSURE < 3) {
                c.ro[1] = ro_n_of(p, r.Pn);
                c.ro[2] = ro_g_of(p, r.Pg);
            }
            return r.Pn != r.Pw || r.Pg != r.Pw;
        }
    }
    return false;
}

using LdsDouble = __attribute__((address_space(3))) double*;

// What an epilogue reads of the cell it finishes.
template <int MODEL>
struct CellState {
    double P, Sw, Sn, ro[MODEL];
};

// One tile of the fused step: interior columns i0 .. i0+TX-1 (i0 = first
// interior i + TX*bx), j0 .. j0+TY-1 (j0 = 1 + TY*by), planes k0 .. k0+kchunk-1
// (k0 = first interior k + kchunk*bz), on a TX x TY workgroup (TY >= 3,
// TX >= 2*TY: rows 0-2 of the workgroup also load the halo ring; TX 32 or 64,
// so that a wavefront holds whole rows).
//
// What bounds it: VALU issue (FP64).  The 256^3 three-phase Corey-2 step went
// from 850 to 715 VALU instructions per cell and from 571 to 475 us, the
// two-phase one from 336 to 266 us, against tiles with two barriers and one LDS
// buffer per plane, every phase's pressure staged, calls and branches in the
// Newton and parameters in vector-register lanes.
//
// A plane's turn: issue the loads of the next plane (own cell and ring) and
// of what the epilogue reads; the x and y fluxes of this plane from LDS,
// which cover those loads; the next plane's coefficients, staged in the
// other LDS buffer; the z flux; the epilogue; one barrier.  The closures that
// raise powers (EARLY) take the coefficients first, while few values are
// live, and read the own ones back from LDS for the z flux.  Across planes a
// thread keeps two pressure parts, the minus z face's flux terms and its
// saturations; its own coefficients come back from LDS.
//
// Epi: what happens at an interior cell once its state and flux divergence
// are known -- the Newton solve and store of the step (FusedStore) or the
// adjoint's backward Newton (AdjNewtonStore).  prefetch() loads what it needs;
// with kLeaves, cell() may leave the cell undone, with its plane's bit set in
// `undone` and its right side in the cell's place of the next state, which nothing
// else in the launch reads: late() does it after the last plane, so that the
// planes' code holds no call and no registers for it (kchunk <= kMaxPlanes, one
// bit per plane).
//
// P_n or P_g apart from P_w in an x or z face cell (values a caller set, or an
// exchange of faces: Border_P gives those faces P_n = P_g = P_w, P_Xi_ro every
// interior cell): the x face's stand in LDS as the top and bottom rows' do, the z
// face's are read again; the wavefronts next to such a cell take each phase's own
// differences in that plane.
// cp, ci: p and io in constant memory (fresh()).
constexpr int kMaxPlanes = 32;
template <int MODEL, int CLOSURE, int TX, int TY, int AXES, class Epi>
__device__ __forceinline__ void fused_z_tile(const DevParams& p, ConstParams* cp, ConstIO* ci, const StepIO& io, int kchunk, int bx, int by, int bz,
                                             FusedLds<MODEL, CLOSURE, TX, TY, AXES>& lds, const Epi& epi) {
    static_assert(TY >= 3 && TX >= 2 * TY, "halo ring needs TY >= 3 and TX >= 2*TY");
    static_assert(TX == 32 || TX == 64, "whole rows per wavefront");
    constexpr int NPH = MODEL, NPR = kStagedP<MODEL, CLOSURE>, NV = FusedLds<MODEL, CLOSURE, TX, TY, AXES>::kNV;
    constexpr int ROW = (TX + 2) * NV, PLANE = (TY + 2) * ROW;  // LDS pitch of a row, of a plane
    constexpr bool U = EpiWantsU<Epi>::value;
    constexpr bool EARLY = CLOSURE == 0 || CLOSURE == 1;
    // three phases: P_n and P_g apart from the staged pressure, where they differ
    constexpr bool APART = FusedLds<MODEL, CLOSURE, TX, TY, AXES>::kApart;

    const int tx = threadIdx.x, ty = threadIdx.y;
    constexpr bool FLAT = AXES == kAxesOnePlane;
    const bool hasx = AXES == kAxesAll || p.Nx >= 3, hasz = AXES == kAxesAll || (!FLAT && p.Nz >= 3);
    const int ilo = hasx ? 1 : 0, ihi = hasx ? p.Nx - 2 : 0;
    const int klo = hasz ? 1 : 0, khi = hasz ? p.Nz - 2 : 0;
    const int i0 = ilo + TX * bx, j0 = 1 + TY * by;
    const int k0 = FLAT ? 0 : klo + kchunk * bz;
    const int k1 = FLAT ? 0 : min(khi, k0 + kchunk - 1);
    const int i = i0 + tx, j = j0 + ty;
    const bool active = i <= ihi && j <= p.Ny - 2;
    // the own column, clamped into the grid (lanes past it stage values that
    // no active lane reads); jw: the wavefront's first row
    const int ic = min(i, p.Nx - 1), jc = min(j, p.Ny - 1);
    const int jw = __builtin_amdgcn_readfirstlane(jc);
    const bool own_ij = CLOSURE != 3 && inner_ij<MODEL>(p, ic, jc);
    CellAt own{(int64_t)i0 + (int64_t)jw * p.sy + (int64_t)k0 * p.sz, 8u * (uint32_t)(ic - i0)};
    if (TX < 64) own.off += 8u * (uint32_t)(jc - jw) * (uint32_t)p.sy;

    // This thread's halo cell of each plane, if any (ty 0 / 1: the y rows
    // below / above the block, ty 2: the x columns left / right of it).
    int hi = -1, hj = -1, hx = 0, hy = 0;
    if (ty == 0) { hi = i; hj = j0 - 1; hx = tx + 1; hy = 0; }
    else if (ty == 1) { hi = i; hj = j0 + TY; hx = tx + 1; hy = TY + 1; }
    else if (ty == 2 && tx < TY) { hi = i0 - 1; hj = j0 + tx; hx = 0; hy = tx + 1; }
    else if (ty == 2 && tx >= TY && tx < 2 * TY) { hi = i0 + TX; hj = j0 + tx - TY; hx = TX + 1; hy = tx - TY + 1; }
    const bool halo = hi >= 0 && hi < p.Nx && hj >= 0 && hj < p.Ny && (hasx || hi == i0 + tx);
    const bool halo_ij = CLOSURE != 3 && inner_ij<MODEL>(p, hi, hj);
    const HaloAt hat(p, i0, j0, hi, hj);

    // LDS places in the buffer of plane 0: the own and the halo cell
    auto buffer = [](int k) { return FLAT ? 0 : (k & 1) * PLANE; };
    const LdsDouble v0 = (LdsDouble)&lds.v[0][ty + 1][tx + 1][0], vh = (LdsDouble)&lds.v[0][hy][hx][0];
    auto stage = [&](int k, LdsDouble w, int row, int x, int ii, int jj, const CellRaw<MODEL, CLOSURE>& r, bool inner,
                     const CellCoef<MODEL, CLOSURE>& c, bool odd) {
#pragma unroll
        for (int a = 0; a < NPR; ++a) w[a] = c.P[a];
#pragma unroll
        for (int a = 0; a < NPH; ++a) {
            w[NPR + a] = c.Xi[a];
            w[NPR + NPH + a] = c.ro[a];
        }
        if constexpr (APART) {
            if (!inner) {
                if (jj == 0 || jj == p.Ny - 1) {
                    lds.edge[k & 1][jj == 0 ? 0 : 1][0][x] = r.Pn;
                    lds.edge[k & 1][jj == 0 ? 0 : 1][1][x] = r.Pg;
                } else {
                    // an x face cell (a z face's plane is not read from LDS)
                    const int s = seldom(ii) == 0 ? 0 : 1;
                    lds.side[k & 1][s][0][row] = r.Pn;
                    lds.side[k & 1][s][1][row] = r.Pg;
                    if (odd) lds.odd[k & 1][row] = k;
                }
            }
        }
    };

    // the minus z face (directed()'s neg_part(x1) and t2) and the own
    // saturations, carried from plane to plane
    double zneg[NPR], zt2[NPH], zmP[NPR], Sw = 0., Sn = 0.;
    // the lanes whose cell below (k - 1) has a P_n or P_g of its own: a boundary
    // plane's, below the tile's first one
    uint64_t zodd = 0;
    uint32_t undone = 0;
#pragma unroll
    for (int a = 0; a < NPR; ++a) zneg[a] = zmP[a] = 0.;
#pragma unroll
    for (int a = 0; a < NPH; ++a) zt2[a] = 0.;
    auto pre = epi.none();
    {
        CellRaw<MODEL, CLOSURE> r, rm, rh;
        const bool inner = own_ij && inner_k(p, k0), inner_m = own_ij && inner_k(p, k0 - 1);
        const bool inner_h = halo_ij && inner_k(p, k0);
        load_raw(io, own, inner, r);
        if (hasz) load_raw(io, CellAt{own.base - p.sz, own.off}, inner_m, rm);
        if (halo) hat.with(p, k0, [&](const auto& at) { load_raw(io, at, inner_h, rh); });
        if constexpr (FLAT) pre = epi.prefetch(own);
        CellCoef<MODEL, CLOSURE> c, m;
        const DevParams pc = coef_params<MODEL, CLOSURE>(cp);
        const bool odd = coef_of(pc, r, inner, c);
        stage(k0, v0 + buffer(k0), ty + 1, tx + 1, ic, jc, r, inner, c, odd);
        Sn = r.Sn;
        if constexpr (MODEL == 3) Sw = r.Sw;
        if (hasz) {
            const bool apart = coef_of(pc, rm, inner_m, m);
            if constexpr (APART) zodd = __ballot(apart);
#pragma unroll
            for (int a = 0; a < NPR; ++a) {
                zmP[a] = m.P[a];
                const double d = exact_div(c.P[a] - m.P[a], p.hz, p.r_hz);
                zneg[a] = neg_part(-1. * d);
#pragma unroll
                for (int b = a; b < (NPR == 1 ? NPH : a + 1); ++b) zt2[b] = directed_t2(-1. * d, m.Xi[b], m.ro[b]);
            }
            if constexpr (APART) {
                if (apart) {
                    zt2[1] = directed_t2(-1. * exact_div(c.P[0] - rm.Pn, p.hz, p.r_hz), m.Xi[1], m.ro[1]);
                    zt2[2] = directed_t2(-1. * exact_div(c.P[0] - rm.Pg, p.hz, p.r_hz), m.Xi[2], m.ro[2]);
                }
            }
        }
        if (halo) {
            const bool oddh = coef_of(pc, rh, inner_h, c);
            stage(k0, vh + buffer(k0), hy, hx, hi, hj, rh, inner_h, c, oddh);
        }
    }
    __syncthreads();

    for (int k = k0; k <= k1; ++k) {
        const bool next = k < k1;  // another plane follows in this tile
        renew(own);
        CellRaw<MODEL, CLOSURE> r, rh;
        const bool inner = own_ij && inner_k(p, k + 1), inner_h = halo_ij && inner_k(p, k + 1);
        const StepIO now = state_arrays<CLOSURE>(io, ci);
        if (hasz) load_raw(now, CellAt{own.base + p.sz, own.off}, inner, r);
        if (next && halo) hat.with(p, k + 1, [&](const auto& at) { load_raw(now, at, inner_h, rh); });
        if constexpr (!FLAT) pre = epi.prefetch(own);
        // the next plane: coefficients, staged in the other buffer
        CellCoef<MODEL, CLOSURE> zp;
        uint64_t odd = 0;
        auto next_plane = [&]() {
            const DevParams pc = coef_params<MODEL, CLOSURE>(fresh(cp));
            if (hasz) {
                const bool mine = coef_of(pc, r, inner, zp);
                if constexpr (APART) odd = __ballot(mine);
                if (next || EARLY) stage(k + 1, v0 + buffer(k + 1), ty + 1, tx + 1, ic, jc, r, inner, zp, mine);
            }
            if (next && halo) {
                CellCoef<MODEL, CLOSURE> h;
                const bool oddh = coef_of(pc, rh, inner_h, h);
                stage(k + 1, vh + buffer(k + 1), hy, hx, hi, hj, rh, inner_h, h, oddh);
            }
        };
        if constexpr (EARLY) next_plane();

        // the own cell's row and the rows below and above it, from the cell at
        // x - 1 on; one register each, every value a constant offset away
        LdsDouble row[3];
#pragma unroll
        for (int y = 0; y < 3; ++y) {
            row[y] = v0 + buffer(k) + (y - 1) * ROW - NV;
            asm("" : "+v"(row[y]));
        }
        auto P_at = [&](int a, int y, int x) { return row[y][x * NV + a]; };
        auto Xi_at = [&](int a, int y, int x) { return row[y][x * NV + NPR + a]; };
        auto ro_at = [&](int a, int y, int x) { return row[y][x * NV + NPR + NPH + a]; };
        double div[NPH], u[NPH][3];
        CellCoef<MODEL, CLOSURE> c;
        const DevParams pf = flux_params(fresh(cp));
        if (active) {
            // order as cpu.cpp:651-708: z, x, y, then (-q + fx + fy + fz)
#pragma unroll
            for (int a = 0; a < NPR; ++a) c.P[a] = P_at(a, 1, 1);
#pragma unroll
            for (int a = 0; a < NPH; ++a) {
                c.Xi[a] = Xi_at(a, 1, 1);
                c.ro[a] = ro_at(a, 1, 1);
                div[a] = 0.;
            }
            if (hasx) {
                // the phases from a0 to a1, whose pressure is one
                auto x_flux = [&](double P, double Pm, double Pp, int a0, int a1) {
                    const double x1 = -1. * exact_div(P - Pm, pf.hx, pf.r_hx);
                    const double x2 = -1. * exact_div(Pp - P, pf.hx, pf.r_hx);
                    const double s1 = (pos_part(x2) - neg_part(x1)) * (-1.), s2 = pos_part(x1) * (-1.),
                                 s3 = neg_part(x2) * (-1.);
#pragma unroll
                    for (int a = a0; a < a1; ++a) {
                        const double t1 = s1 * c.Xi[a] * c.ro[a];
                        const double t2 = s2 * Xi_at(a, 1, 0) * ro_at(a, 1, 0);
                        const double t3 = s3 * Xi_at(a, 1, 2) * ro_at(a, 1, 2);
                        const double fx = exact_div(t1 - t2 + t3, pf.hx, pf.r_hx);
                        div[a] = a == 2 ? 0. + fx : fx;
                        if constexpr (U) u[a][0] = c.Xi[a] * exact_div(Pp - Pm, pf.two_hx, pf.r_two_hx);
                    }
                };
#pragma unroll
                for (int q = 0; q < NPR; ++q)
                    x_flux(c.P[q], P_at(q, 1, 0), P_at(q, 1, 2), q, NPR == 1 ? NPH : q + 1);
                if constexpr (APART) {
                    // n and g again, each from its own pressures
                    if (__builtin_expect(__ballot(lds.odd[k & 1][ty + 1] == k) != 0, 0)) {
                        const int is = seldom(i);
#pragma unroll
                        for (int a = 1; a < NPH; ++a)
                            x_flux(c.P[0], is == 1 ? lds.side[k & 1][0][a - 1][ty + 1] : P_at(0, 1, 0),
                                   is == p.Nx - 2 ? lds.side[k & 1][1][a - 1][ty + 1] : P_at(0, 1, 2), a, a + 1);
                    }
                }
            } else if constexpr (U) {
#pragma unroll
                for (int a = 0; a < NPH; ++a) u[a][0] = 0.;
            }
            // the x neighbours' values are done with before the y ones are read
            asm volatile("" ::: "memory");
            // the face differences dm, dp and their sum's dd of phase a's pressure
            auto y_flux = [&](int a, double dm, double dp, double dd) {
                div[a] = div[a] + flux_y(pf, dm, dp, c.Xi[a], c.ro[a], Xi_at(a, 0, 1), ro_at(a, 0, 1), Xi_at(a, 2, 1),
                                         ro_at(a, 2, 1));
                if constexpr (U) u[a][1] = c.Xi[a] * (exact_div(dd, pf.two_hy, pf.r_two_hy) - c.ro[a] * pf.g);
            };
            // three phases, next to the top and bottom rows: their own P_n and P_g
            const int jr = TX == 64 ? jw : j;
            if (APART && (jr == 1 || jr == p.Ny - 2)) {
#pragma unroll
                for (int a = 0; a < NPH; ++a) {
                    double Pm = P_at(0, 0, 1), Pp = P_at(0, 2, 1);
                    if constexpr (APART) {
                        if (a > 0 && jr == 1) Pm = lds.edge[k & 1][0][a - 1][tx + 1];
                        if (a > 0 && jr == p.Ny - 2) Pp = lds.edge[k & 1][1][a - 1][tx + 1];
                    }
                    y_flux(a, exact_div(c.P[0] - Pm, pf.hy, pf.r_hy), exact_div(Pp - c.P[0], pf.hy, pf.r_hy), Pp - Pm);
                }
            } else {
#pragma unroll
                for (int q = 0; q < NPR; ++q) {
                    const double Pm = P_at(q, 0, 1), Pp = P_at(q, 2, 1);
                    const double dm = exact_div(c.P[q] - Pm, pf.hy, pf.r_hy), dp = exact_div(Pp - c.P[q], pf.hy, pf.r_hy);
#pragma unroll
                    for (int a = q; a < (NPR == 1 ? NPH : q + 1); ++a) y_flux(a, dm, dp, Pp - Pm);
                }
            }
        }
        if constexpr (!EARLY) next_plane();
        if constexpr (EARLY) {
            // own values staged above, read back where they are used
            const LdsDouble w = v0 + buffer(k + 1);
#pragma unroll
            for (int a = 0; a < NPR; ++a) zp.P[a] = w[a];
#pragma unroll
            for (int a = 0; a < NPH; ++a) {
                zp.Xi[a] = w[NPR + a];
                zp.ro[a] = w[NPR + NPH + a];
            }
        }
        if (active) {
            if (hasz) {
                // the phases from a0 to a1, of one pressure; the plus face's neg_part
                auto z_flux = [&](double zn, double Pm, double P, double Pp, int a0, int a1) {
                    const double x2 = -1. * exact_div(Pp - P, pf.hz, pf.r_hz);
                    const double n2 = neg_part(x2), p2 = pos_part(x2);
                    const double s1 = (p2 - zn) * (-1.), s3 = n2 * (-1.), s2 = p2 * (-1.);
#pragma unroll
                    for (int a = a0; a < a1; ++a) {
                        const double t1 = s1 * c.Xi[a] * c.ro[a];
                        const double t3 = s3 * zp.Xi[a] * zp.ro[a];
                        div[a] = div[a] + exact_div(t1 - zt2[a] + t3, pf.hz, pf.r_hz);
                        zt2[a] = s2 * c.Xi[a] * c.ro[a];  // the next plane's minus face
                        if constexpr (U) u[a][2] = c.Xi[a] * exact_div(Pp - Pm, pf.two_hz, pf.r_two_hz);
                    }
                    return n2;
                };
                if (APART && __builtin_expect((zodd | odd) != 0, 0)) {
                    const uint64_t lane = 1ull << ((ty * TX + tx) & 63);
                    const double zn = zneg[0];
                    const StepIO now = state_arrays<CLOSURE>(io, ci);
                    zneg[0] = z_flux(zn, zmP[0], c.P[0], zp.P[0], 0, 1);
#pragma unroll
                    for (int a = 1; a < NPH; ++a) {
                        const double* P = a == 1 ? now.Pn : now.Pg;
                        double zna = zn, Pm = zmP[0], Pp = zp.P[0];
                        if (zodd & lane) {
                            Pm = ld(P, CellAt{own.base - p.sz, own.off});
                            zna = neg_part(-1. * exact_div(c.P[0] - Pm, pf.hz, pf.r_hz));
                        }
                        if (odd & lane) Pp = ld(P, CellAt{own.base + p.sz, own.off});
                        z_flux(zna, Pm, c.P[0], Pp, a, a + 1);
                    }
                } else {
#pragma unroll
                    for (int q = 0; q < NPR; ++q)
                        zneg[q] = z_flux(zneg[q], zmP[q], c.P[q], zp.P[q], q, NPR == 1 ? NPH : q + 1);
                }
                if constexpr (U) {
#pragma unroll
                    for (int q = 0; q < NPR; ++q) zmP[q] = c.P[q];
                }
            } else {
#pragma unroll
                for (int a = 0; a < NPH; ++a) {
                    div[a] = div[a] + 0.;
                    if constexpr (U) u[a][2] = 0.;
                }
            }
            CellState<MODEL> s;
            s.P = c.P[0];
            s.Sw = Sw;
            s.Sn = Sn;
#pragma unroll
            for (int a = 0; a < NPH; ++a) s.ro[a] = c.ro[a];
            if constexpr (U) epi.store_u(own, u);
            epi.cell(p, newton_params<MODEL, CLOSURE>(fresh(cp)), i, j, k, own, s, div, pre, undone, 1u << (k - k0));
        }
        if (next) {
            zodd = 0;
            Sn = r.Sn;
            if constexpr (MODEL == 3) Sw = r.Sw;
            own.base += p.sz;
            __syncthreads();
        }
    }

    if constexpr (Epi::kLeaves) {
        while (__builtin_expect(undone != 0, 0)) {
            epi.late(p, newton_params<MODEL, CLOSURE>(fresh(cp)), i, j, k0 + __ffs(undone) - 1);
            undone &= undone - 1;
        }
    }
}

// Tile of workgroup (blockIdx): workgroups go to the 8 XCDs round robin, so
// when the grid divides by 8 each XCD takes one contiguous run of tiles (x
// fastest, then y, then z) and the halo rows its tiles share stay in its L2.
__device__ __forceinline__ void xcd_tile(int& bx, int& by, int& bz) {
    const uint32_t gx = gridDim.x, gy = gridDim.y;
    const uint32_t nb = gx * gy * gridDim.z;
    uint32_t id = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    if (nb % 8u == 0u) id = (id % 8u) * (nb / 8u) + id / 8u;
    bx = (int)(id % gx);
    const uint32_t r = id / gx;
    by = (int)(r % gy);
    bz = (int)(r / gy);
}

// The boundary cells whose inward neighbour (set_boundary_basic_coordinate,
// cpu.cpp:107-141) is the interior cell (i, j, k), from its new state: the
// cell's offsets along each axis are 0 and -1 next to the low face, +1 next to
// the high face.  On the supported grids every boundary cell has exactly one
// interior inward neighbour, so this writes each boundary cell once, with the
// values k_fused_faces would write.
template <int MODEL>
__device__ __forceinline__ void store_faces(const DevParams& p, const StepIO& io, int i, int j, int k, int64_t l,
                                            const double* ro, double Pw, double Sw, double Sn) {
    const bool hasx = p.Nx >= 3, hasz = p.Nz >= 3;
    const bool xl = hasx && i == 1, xh = hasx && i == p.Nx - 2;
    const bool yl = j == 1, yh = j == p.Ny - 2;
    const bool zl = hasz && k == 1, zh = hasz && k == p.Nz - 2;
    if (!(xl || xh || yl || yh || zl || zh)) return;
    double ro_eff = 0.;
    if constexpr (MODEL == 2) {
        // ro_eff_gdy (main.cpp:255-267) for the bottom face: this step's
        // densities of the cell (from its previous state), its new saturation
        if (yh) ro_eff = (ro[1] * Sn + ro[0] * (1 - Sn)) * io.m[l] * p.g * p.hy;
    }
    int xo[3] = {0, 0, 0}, yo[3] = {0, 0, 0}, zo[3] = {0, 0, 0};
    int nx = 1, ny = 1, nz = 1;
    if (xl) xo[nx++] = -1;
    if (xh) xo[nx++] = 1;
    if (yl) yo[ny++] = -1;
    if (yh) yo[ny++] = 1;
    if (zl) zo[nz++] = -1;
    if (zh) zo[nz++] = 1;
    for (int a = 0; a < nx; ++a)
        for (int b = 0; b < ny; ++b)
            for (int d = 0; d < nz; ++d)
                if (a || b || d) write_boundary<MODEL>(p, io, i + xo[a], j + yo[b], k + zo[d], Pw, Sw, Sn, ro_eff);
}

// The step's epilogue: A = roS - dt/m * div, the Newton solve, the new state;
// FACES: also the boundary cells this cell is the inward neighbour of (else
// k_fused_faces writes them after the kernel).  The two-phase kernels write
// their faces here (the strided x faces cost a separate pass more than the
// epilogue costs); in the three-phase kernels the extra registers would cost
// a wave per SIMD, so but for small grids they keep the face pass.  CLOSURE: the kernel's
// (the two-phase Newton then carries only its closure's code).
template <int MODEL, bool FACES = false, int CLOSURE = -1>
struct FusedStore {
    StepIO io;
    // dt / m, computed once per porosity field
    __device__ __forceinline__ double none() const { return 0.; }
    template <class At>
    __device__ __forceinline__ double prefetch(const At& at) const { return ld(io.dtm, at); }
    static constexpr bool kLeaves = true;
    template <class At>
    __device__ __forceinline__ void cell(const DevParams& p, const DevParams& pn, int i, int j, int k, const At& at,
                                         const CellState<MODEL>& s, const double* div, double dtm, uint32_t& undone,
                                         uint32_t bit) const {
        (void)i; (void)j; (void)k;
        double Pw = s.P, Sn = s.Sn, Sw = s.Sw;
        bool done;
        if constexpr (MODEL == 2) {
            const double A1 = s.ro[0] * (1. - Sn) - dtm * div[0];
            const double A2 = s.ro[1] * Sn - dtm * div[1];
            done = newton2_fast<CLOSURE>(pn, Pw, Sn, A1, A2);
            if (__builtin_expect(!done, 0)) {
                Pw = A1;
                Sn = A2;
                undone |= bit;
            }
        } else {
            const double A1 = s.ro[0] * Sw - dtm * div[0];
            const double A2 = s.ro[1] * Sn - dtm * div[1];
            const double A3 = s.ro[2] * (1. - Sw - Sn) - dtm * div[2];
            done = newton3_fast(pn, Pw, Sw, Sn, A1, A2, A3);
            if (__builtin_expect(!done, 0)) {
                Pw = A1;
                Sw = A3;
                Sn = A2;
                undone |= bit;
            }
        }
        At to = at;
        renew(to);
        st(io.Pw1, to, Pw);
        if constexpr (MODEL == 3) st(io.Sw1, to, Sw);
        st(io.Sn1, to, Sn);
        if constexpr (FACES)
            if (done) store_faces<MODEL>(p, io, i, j, k, at.l(), s.ro, Pw, Sw, Sn);
    }
    // The cell from its state and the right side that cell() left.
    __device__ __forceinline__ void late(const DevParams& p, const DevParams& pn, int i, int j, int k) const {
        const int64_t l = (int64_t)i + (int64_t)j * p.sy + (int64_t)k * p.sz;
        const double A1 = io.Pw1[l], A2 = io.Sn1[l];
        double Pw = io.Pw[l], Sn = io.Sn[l], Sw = 0., ro[MODEL] = {};
        if constexpr (MODEL == 2) {
            if constexpr (FACES) densities2<CLOSURE>(p, io, l, ro);
            newton2_ieee<CLOSURE>(pn, Pw, Sn, A1, A2);
        } else {
            const double A3 = io.Sw1[l];
            Sw = io.Sw[l];
            newton3_general(pn, Pw, Sw, Sn, A1, A2, A3);
            io.Sw1[l] = Sw;
        }
        io.Pw1[l] = Pw;
        io.Sn1[l] = Sn;
        if constexpr (FACES) store_faces<MODEL>(p, io, i, j, k, l, ro, Pw, Sw, Sn);
    }
};

// Two phases: boundary cells included (kFusedFaces); three phases: followed
// by k_fused_faces (but for small grids, k_fused_z).
template <int MODEL>
constexpr bool kFusedFaces = MODEL == 2;

// FusedStore that also records the cell's flux divergence div_a (field a at
// div + a*stride), for the adjoint's backward Newton.
template <int MODEL, int CLOSURE = -1>
struct FusedStoreRecord {
    FusedStore<MODEL, kFusedFaces<MODEL>, CLOSURE> step;
    double* div;
    int64_t stride;
    __device__ __forceinline__ double none() const { return 0.; }
    template <class At>
    __device__ __forceinline__ double prefetch(const At& at) const { return step.prefetch(at); }
    static constexpr bool kLeaves = true;
    template <class At>
    __device__ __forceinline__ void cell(const DevParams& p, const DevParams& pn, int i, int j, int k, const At& at,
                                         const CellState<MODEL>& s, const double* d, double dtm, uint32_t& undone,
                                         uint32_t bit) const {
        At to = at;
        renew(to);
#pragma unroll
        for (int a = 0; a < MODEL; ++a) st(div + a * stride, to, d[a]);
        step.cell(p, pn, i, j, k, at, s, d, dtm, undone, bit);
    }
    __device__ __forceinline__ void late(const DevParams& p, const DevParams& pn, int i, int j, int k) const { step.late(p, pn, i, j, k); }
};

// assign_roS_nr (cpu.cpp:619-731) on the z tiles (three phases): roS_old and
// roS of the cell from the stored coefficients (CLOSURE 3, the roS entry point,
// every cell's P_n and P_g as they stand) or (U, CLOSURE 4) the energy step's roS +
// u pass, with the cell's velocities (assign_u) from the same neighbours.  Arrays
// that are NULL are not stored.
template <bool U>
struct RoSStore {
    static constexpr bool kWantsU = U, kLeaves = false;
    const double* dtm;
    double *roS[3], *roS_old[3];
    double* u[3][3];  // [phase][axis]: ux_w, uy_w, uz_w, ux_n, ... (U only)
    __device__ __forceinline__ double none() const { return 0.; }
    template <class At>
    __device__ __forceinline__ double prefetch(const At& at) const { return ld(dtm, at); }
    template <class At>
    __device__ __forceinline__ void store_u(const At& at, const double (&v)[3][3]) const {
        At to = at;
        renew(to);
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int x = 0; x < 3; ++x)
                if (x < 2 || u[a][2]) st(u[a][x], to, v[a][x]);
    }
    template <class At>
    __device__ __forceinline__ void cell(const DevParams& p, const DevParams& pn, int i, int j, int k, const At& at,
                                         const CellState<3>& s, const double* div, double d, uint32_t&, uint32_t) const {
        (void)p; (void)pn; (void)i; (void)j; (void)k;
        const double old[3] = {s.ro[0] * s.Sw, s.ro[1] * s.Sn, s.ro[2] * (1. - s.Sw - s.Sn)};
        At to = at;
        renew(to);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (!U || roS_old[a]) st(roS_old[a], to, old[a]);
            st(roS[a], to, old[a] - d * div[a]);
        }
    }
};

template <int TX, int TY, int AXES, bool U>
__global__ void __launch_bounds__(TX * TY) k_roS_z(DevParams p, StepIO io, int kchunk, RoSStore<U> st) {
    __shared__ FusedLds<3, U ? 4 : 3, TX, TY, AXES> lds;
    int bx, by, bz;
    xcd_tile(bx, by, bz);
    fused_z_tile<3, U ? 4 : 3, TX, TY, AXES>(p, kernel_params(), kernel_io(), io, kchunk, bx, by, bz, lds, st);
}

// The energy step's E pass (assign_E_new, energy.cpp:235-340, as body_E_with)
// on z-marching TX x TY tiles: each cell's lambda_eff * T and its advected
// products (ro_a * H_a) * u_a are formed once (and once more where another
// tile's ring holds the cell), staged in LDS with a one-cell halo ring for the
// x and y neighbours and carried in registers for the z ones.  Each term is
// the product the per-cell body forms, so E_new has its bits.
//
// Bound by memory (14 fields read and one written per cell; with STEP 10 and one): the next plane's
// loads are issued before this plane's sums and one barrier ends a plane (two
// LDS buffers).  160 x 128 x 96: 92 us against 115 for tiles that read the
// fields again for the z neighbours (32 x 16 tiles, whose threads cover the 158
// columns without the sixth that 64 x 8 leave idle: 88, and roS 98 against 95).
//
// STEP: ro and H from P and T, as the step's first pass has them, instead of
// from their arrays.  LAM, where lambda_eff comes from: kLamStored (STEP), lam as
// that pass stored it; kLamEvaluated (the entry point), from m, S_w, S_n, S_g and
// T; kLamConstant, lam_cfg: the configurations' energy closure, whose z term
// advects with uz (the reference's with uy, energy.cpp:300-305) and whose z
// conduction adds to the x and y terms.
enum { kLamStored, kLamEvaluated, kLamConstant };
struct EnergyEIO {
    const double *lam, *T, *E;
    const double *m, *Sw, *Sn, *Sg;
    const double *ro[3], *H[3], *ux[3], *uy[3], *uz[3];
    const double *P[3];
    double* E_new;
    double lam_cfg;
};

template <bool STEP, int LAM>
struct EnergyRaw {
    double lam, m, Sw, Sn, Sg, T, P[3], ro[3], H[3], ux[3], uy[3], uz[3];
};
template <bool STEP, int LAM, class At>
__device__ __forceinline__ void load_energy(const EnergyEIO& a, const At& at, bool inner, EnergyRaw<STEP, LAM>& r) {
    r.T = ld(a.T, at);
    if constexpr (LAM == kLamStored) r.lam = ld(a.lam, at);
    if constexpr (LAM == kLamEvaluated) {
        r.m = ld(a.m, at);
        r.Sw = ld(a.Sw, at);
        r.Sn = ld(a.Sn, at);
        r.Sg = ld(a.Sg, at);
    }
    if constexpr (STEP) {
        r.P[0] = ld(a.P[0], at);
        if (!inner) {
            r.P[1] = ld(a.P[1], at);
            r.P[2] = ld(a.P[2], at);
        }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        if constexpr (!STEP) {
            r.ro[q] = ld(a.ro[q], at);
            r.H[q] = ld(a.H[q], at);
        }
        r.ux[q] = ld(a.ux[q], at);
        r.uy[q] = ld(a.uy[q], at);
        if constexpr (LAM == kLamConstant) r.uz[q] = ld(a.uz[q], at);
    }
}
// v[0] = lambda_eff * T, v[1 + a] = (ro_a H_a) ux_a, v[4 + a] = (ro_a H_a) uy_a;
// z[a]: the product that the z term advects
template <bool STEP, int LAM>
__device__ __forceinline__ void energy_vals(const DevParams& p, const EnergyEIO& a, const EnergyRaw<STEP, LAM>& r,
                                            bool inner, double* v, double* z) {
    double lam;
    if constexpr (LAM == kLamStored) lam = r.lam;
    if constexpr (LAM == kLamEvaluated) lam = lambda_eff(r.m, r.Sw, r.Sn, r.Sg, r.T);
    if constexpr (LAM == kLamConstant) lam = a.lam_cfg;
    v[0] = lam * r.T;
    double rh[3];
    if constexpr (STEP) {
        rh[0] = ro_w_T(p, r.P[0], r.T) * H_w_of(p, r.T);
        rh[1] = ro_n_T(p, inner ? r.P[0] : r.P[1], r.T) * H_n_T(p, r.T);
        rh[2] = ro_g_T(p, inner ? r.P[0] : r.P[2], r.T) * H_g_T(p, r.T);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        if constexpr (!STEP) rh[q] = r.ro[q] * r.H[q];
        v[1 + q] = rh[q] * r.ux[q];
        v[4 + q] = rh[q] * r.uy[q];
        z[q] = LAM == kLamConstant ? rh[q] * r.uz[q] : v[4 + q];
    }
}

// advection's (((X_w+ - X_w-) + X_n+) - X_n-) + X_g+) - X_g- (the body's order)
__device__ __forceinline__ double energy_adv(double wp, double wm, double np_, double nm, double gp, double gm) {
    return wp - wm + np_ - nm + gp - gm;
}

template <bool STEP, int LAM, int TX, int TY>
__global__ void __launch_bounds__(TX * TY) __attribute__((amdgpu_waves_per_eu(4)))
k_energy_e_z(DevParams p, EnergyEIO a, int kchunk) {
    static_assert(TY >= 3 && TX == 64, "halo ring and whole rows per wavefront");
    constexpr int NV = 7, ROW = (TX + 2) * NV, PLANE = (TY + 2) * ROW;
    __shared__ double lds[2][TY + 2][TX + 2][NV];
    int bx, by, bz;
    xcd_tile(bx, by, bz);
    const int tx = threadIdx.x, ty = threadIdx.y;
    const bool hasx = p.Nx >= 3, hasz = p.Nz >= 3;
    const int ilo = hasx ? 1 : 0, ihi = hasx ? p.Nx - 2 : 0;
    const int klo = hasz ? 1 : 0, khi = hasz ? p.Nz - 2 : 0;
    const int i0 = ilo + TX * bx, j0 = 1 + TY * by;
    const int k0 = klo + kchunk * bz;
    const int k1 = min(khi, k0 + kchunk - 1);
    const int i = i0 + tx, j = j0 + ty;
    const bool active = i <= ihi && j <= p.Ny - 2;
    // the own column, clamped into the grid, and the halo cell, as in fused_z_tile
    const int ic = min(i, p.Nx - 1), jw = __builtin_amdgcn_readfirstlane(min(j, p.Ny - 1));
    CellAt own{(int64_t)i0 + (int64_t)jw * p.sy + (int64_t)k0 * p.sz, 8u * (uint32_t)(ic - i0)};
    int hi = -1, hj = -1, hx = 0, hy = 0;
    if (ty == 0) { hi = i; hj = j0 - 1; hx = tx + 1; hy = 0; }
    else if (ty == 1) { hi = i; hj = j0 + TY; hx = tx + 1; hy = TY + 1; }
    else if (ty == 2 && tx < TY) { hi = i0 - 1; hj = j0 + tx; hx = 0; hy = tx + 1; }
    else if (ty == 2 && tx >= TY && tx < 2 * TY) { hi = i0 + TX; hj = j0 + tx - TY; hx = TX + 1; hy = tx - TY + 1; }
    const bool halo = hi >= 0 && hi < p.Nx && hj >= 0 && hj < p.Ny && (hasx || hi == i0 + tx);
    const bool own_ij = inner_ij<3>(p, ic, min(j, p.Ny - 1)), halo_ij = inner_ij<3>(p, hi, hj);
    const HaloAt hat(p, i0, j0, hi, hj);
    const LdsDouble v0 = (LdsDouble)&lds[0][ty + 1][tx + 1][0], vh = (LdsDouble)&lds[0][hy][hx][0];
    auto stage = [&](LdsDouble w, const double* v) {
#pragma unroll
        for (int q = 0; q < NV; ++q) w[q] = v[q];
    };

    // lambda_eff * T and the z products of the planes k - 1 and k
    double lm = 0., zm[3] = {}, lc, zc[3];
    {
        EnergyRaw<STEP, LAM> r, rh;
        double v[NV], z[3];
        if (hasz) {
            const bool inner = own_ij && inner_k(p, k0 - 1);
            load_energy(a, CellAt{own.base - p.sz, own.off}, inner, r);
            energy_vals(p, a, r, inner, v, zm);
            lm = v[0];
        }
        asm volatile("" ::: "memory");  // one plane's values in registers at a time
        const bool inner = own_ij && inner_k(p, k0), inner_h = halo_ij && inner_k(p, k0);
        load_energy(a, own, inner, r);
        if (halo) hat.with(p, k0, [&](const auto& at) { load_energy(a, at, inner_h, rh); });
        energy_vals(p, a, r, inner, v, zc);
        lc = v[0];
        stage(v0 + (k0 & 1) * PLANE, v);
        if (halo) {
            energy_vals(p, a, rh, inner_h, v, z);
            stage(vh + (k0 & 1) * PLANE, v);
        }
    }
    __syncthreads();
    for (int k = k0; k <= k1; ++k) {
        const bool next = k < k1;
        renew(own);
        EnergyRaw<STEP, LAM> r, rh;
        const bool inner = own_ij && inner_k(p, k + 1), inner_h = halo_ij && inner_k(p, k + 1);
        if (hasz) load_energy(a, CellAt{own.base + p.sz, own.off}, inner, r);
        if (next && halo) hat.with(p, k + 1, [&](const auto& at) { load_energy(a, at, inner_h, rh); });
        const double E = ld(a.E, own);
        const LdsDouble c = v0 + (k & 1) * PLANE;
        double T_flow = 0, E_flow = 0;
        if (p.Nx > 2) {
            const LdsDouble m = c - NV, q = c + NV;
            T_flow += exact_div(q[0] - 2 * lc + m[0], p.hx2, p.r_hx2);
            E_flow += exact_div(energy_adv(q[1], m[1], q[2], m[2], q[3], m[3]), p.two_hx, p.r_two_hx);
        }
        {
            const LdsDouble m = c - ROW, q = c + ROW;
            T_flow += exact_div(q[0] - 2 * lc + m[0], p.hy2, p.r_hy2);
            E_flow += exact_div(energy_adv(q[4], m[4], q[5], m[5], q[6], m[6]), p.two_hy, p.r_two_hy);
        }
        double zp[3], lp = 0.;
        if (hasz) {
            double v[NV];
            energy_vals(p, a, r, inner, v, zp);
            lp = v[0];
            if (next) stage(v0 + ((k + 1) & 1) * PLANE, v);
        }
        if (next && halo) {
            double v[NV], z[3];
            energy_vals(p, a, rh, inner_h, v, z);
            stage(vh + ((k + 1) & 1) * PLANE, v);
        }
        if (hasz) {
            const double tz = exact_div(lp - 2 * lc + lm, p.hz2, p.r_hz2);
            if constexpr (LAM == kLamConstant)
                T_flow += tz;
            else
                T_flow = tz;  // '=' as energy.cpp:257
            E_flow += exact_div(energy_adv(zp[0], zm[0], zp[1], zm[1], zp[2], zm[2]), p.two_hz, p.r_two_hz);
        }
        if (active) {
            double Q_hw = 0, Q_hr = 0;
            CellAt to = own;
            renew(to);
            st(a.E_new, to, E + p.dt * (T_flow + Q_hw + Q_hr - E_flow));
        }
        if (next) {
            lm = lc;
            lc = lp;
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                zm[q] = zc[q];
                zc[q] = zp[q];
            }
            own.base += p.sz;
            __syncthreads();
        }
    }
}

// The step that also records each interior cell's flux divergence.  Four waves
// per SIMD, two workgroups per CU: 96^3 three phases 38 us where the 142 VGPRs that
// the compiler takes by itself gave 45; 36.5 now.
template <int MODEL, int CLOSURE, int TX, int TY, int AXES>
__global__ void __launch_bounds__(TX * TY) __attribute__((amdgpu_waves_per_eu(4))) k_fused_z_record(DevParams p, StepIO io, int kchunk, double* div,
                                                           int64_t stride) {
    __shared__ FusedLds<MODEL, CLOSURE, TX, TY, AXES> lds;
    int bx, by, bz;
    xcd_tile(bx, by, bz);
    fused_z_tile<MODEL, CLOSURE, TX, TY, AXES>(p, kernel_params(), kernel_io(), io, kchunk, bx, by, bz, lds,
                                               FusedStoreRecord<MODEL, CLOSURE>{
                                                   FusedStore<MODEL, kFusedFaces<MODEL>, CLOSURE>{io}, div, stride});
}

// Waves per SIMD of the step's tiles, and their shapes per model and closure: a
// wide one, 64 x kWideTY, and a narrow one, 32 x kNarrowTY, of which the launch
// takes the one whose workgroups cover the grid's columns with fewer threads,
// and 64 x 4 for grids so small that its workgroups all fit at once.  us per
// step, wide / narrow, and per thread and plane of the covering workgroups (ps):
//   three phases, Corey-2   256^3 479 / 475 (28.8 / 28.5), 203 x 117 x 83 72.5 / 65.6 (29.1 / 28.2)
//     van Genuchten         160 x 144 x 130 236 / 193 (66.6 / 65.3)
//     run-time exponent     160 x 144 x 130 144 / 120
//   two phases, Corey-2     256^3 273 / 266, 96^3 25.4 / 20.0
//     Brooks-Corey          190 x 150 x 110 186 / 206, 160^3 282 / 240
//     run-time exponent     256^3 386 / 378
// the other shapes of 256 and 512 threads are slower or equal, but in small
// grids, where a workgroup's latency counts: three phases (with k_fused_faces)
// 24^3 64 x 4 9.7, 64 x 8 11.3, 32 x 16 11.3; 48^3 13.9, 16.8, 16.3.  Registers:
// 128 VGPRs at 4 waves (32 to 64 B spilled for three phases, nearly all of it
// outside the plane loop's usual path), 88 at 5, 168 at 3.
template <int MODEL, int CLOSURE, int TX, int TY>
constexpr int kFusedWaves = TX * TY == 512 ? 4 : (MODEL == 2 && CLOSURE == 2 ? 5 : 3);
template <int MODEL, int CLOSURE>
constexpr int kWideTY = MODEL == 2 && CLOSURE != 1 ? 4 : 8;
template <int MODEL, int CLOSURE>
constexpr int kNarrowTY = MODEL == 2 && CLOSURE == 2 ? 8 : 16;

// FACES: the boundary cells too, for three phases in grids that take the 64 x 4
// tiles for being small: there a launch counts, not the registers (24^3 8.4 us per
// step against 9.7 with k_fused_faces, 48^3 12.2 against 13.9; 256^3 579 against
// 475 with the tiles and pass that large grids take).
template <int MODEL, int CLOSURE, int TX, int TY, int AXES, bool FACES>
__global__ void __launch_bounds__(TX * TY) __attribute__((amdgpu_waves_per_eu(kFusedWaves<MODEL, CLOSURE, TX, TY>)))
k_fused_z(DevParams p, StepIO io, int kchunk) {
    __shared__ FusedLds<MODEL, CLOSURE, TX, TY, AXES> lds;
    int bx, by, bz;
    xcd_tile(bx, by, bz);
    fused_z_tile<MODEL, CLOSURE, TX, TY, AXES>(p, kernel_params(), kernel_io(), io, kchunk, bx, by, bz, lds,
                                               FusedStore<MODEL, FACES, CLOSURE>{io});
}

// Cell number t of a box of ni x nj cells per plane starting at (i0, j0, k0),
// x fastest (32-bit index arithmetic: grids of < 2^31 cells).
__device__ __forceinline__ void box_cell(uint32_t t, uint32_t ni, uint32_t nj, int i0, int j0, int k0, int& i, int& j,
                                         int& k) {
    const uint32_t a = t / ni, b = a / nj;
    i = i0 + (int)(t - a * ni);
    j = j0 + (int)(a - b * nj);
    k = k0 + (int)b;
}

// Coordinates of boundary cell number t (t enumerates the j faces (all i,
// k), then the x faces (j interior, all k), then the z faces (i, j
// interior)); false for t past the last face cell.  32-bit index
// arithmetic: the face cells of a grid of < 2^31 cells.
__device__ __forceinline__ bool face_cell(const DevParams& p, int64_t t64, int& i, int& j, int& k) {
    const bool hasx = p.Nx >= 3, hasz = p.Nz >= 3;
    const uint32_t Nx = (uint32_t)p.Nx, Ny2 = (uint32_t)(p.Ny - 2);
    const uint32_t nj = 2u * Nx * (uint32_t)p.Nz;
    const uint32_t nx = hasx ? 2u * Ny2 * (uint32_t)p.Nz : 0u;
    const uint32_t ni = hasx ? Nx - 2u : Nx;
    const uint32_t nzf = hasz ? 2u * ni * Ny2 : 0u;
    if (t64 >= (int64_t)nj + nx + nzf) return false;
    uint32_t t = (uint32_t)t64;
    if (t < nj) {
        j = (t & 1u) ? p.Ny - 1 : 0;
        t >>= 1;
        const uint32_t q = t / Nx;
        i = (int)(t - q * Nx);
        k = (int)q;
    } else if ((t -= nj) < nx) {
        i = (t & 1u) ? p.Nx - 1 : 0;
        t >>= 1;
        const uint32_t q = t / Ny2;
        j = 1 + (int)(t - q * Ny2);
        k = (int)q;
    } else {
        t -= nx;
        k = (t & 1u) ? p.Nz - 1 : 0;
        t >>= 1;
        const uint32_t q = t / ni;
        i = (hasx ? 1 : 0) + (int)(t - q * ni);
        j = 1 + (int)q;
    }
    return true;
}

// Boundary cell number t of the step after the interior tiles (face_cell's
// numbering); nothing for t past the last face cell.
template <int MODEL, int CLOSURE>
__device__ __forceinline__ void fused_face(const DevParams& p, const StepIO& io, int64_t t64) {
    int i, j, k;
    if (!face_cell(p, t64, i, j, k)) return;
    const int64_t l1 = inward(p, i, j, k);
    const double Pw = io.Pw1[l1], Sn = io.Sn1[l1];
    const double Sw = MODEL == 3 ? io.Sw1[l1] : 0.;
    double ro_eff = 0.;
    if constexpr (MODEL == 2) {
        // ro_eff_gdy (main.cpp:255-267), read by the bottom face only: this
        // step's densities of the inward cell (from its previous state) with
        // its new saturation
        if (j == p.Ny - 1) {
            double ro[2];
            densities2<CLOSURE>(p, io, l1, ro);
            ro_eff = (ro[1] * Sn + ro[0] * (1 - Sn)) * io.m[l1] * p.g * p.hy;
        }
    }
    write_boundary<MODEL>(p, io, i, j, k, Pw, Sw, Sn, ro_eff);
}

template <int MODEL, int CLOSURE>
__global__ void __launch_bounds__(256) k_fused_faces(DevParams p, StepIO io) {
    fused_face<MODEL, CLOSURE>(p, io, (int64_t)blockIdx.x * 256 + threadIdx.x);
}

inline int64_t fused_face_cells(const DevParams& p) {
    const bool hasx = p.Nx >= 3, hasz = p.Nz >= 3;
    const int64_t ni = hasx ? p.Nx - 2 : p.Nx;
    return 2LL * p.Nx * p.Nz + (hasx ? 2LL * (p.Ny - 2) * p.Nz : 0) + (hasz ? 2LL * ni * (p.Ny - 2) : 0);
}

// The halo pack of a z-slab exchange written by the step itself: cell c of
// side s (plane 1, or plane Nz - 2) of the new state into io.pack at
// (f * 2 + s) * Nx * Ny + c for the state fields f (three phases: P_w, S_w,
// S_n, P_n, P_g; two: P_w, S_n) -- capaz_load_faces' layout for axis 2.
// Interior cells give their new values (P_n = P_g = P_w, as the step takes
// them), the plane's x / y boundary cells the Border values of their inward
// cell, computed here rather than read, so the pack needs no second launch
// after the boundary writes.
template <int MODEL, int CLOSURE>
__device__ __forceinline__ void fused_pack(const DevParams& p, const StepIO& io, int64_t t) {
    const int64_t plane = (int64_t)p.Nx * p.Ny;
    if (t >= 2 * plane) return;
    const int s = t >= plane ? 1 : 0;
    const int64_t c = t - s * plane;
    const int k = s ? p.Nz - 2 : 1;
    const int j = (int)(c / p.Nx), i = (int)(c - (int64_t)j * p.Nx);
    const bool interior = (p.Nx < 3 || (i != 0 && i != p.Nx - 1)) && j != 0 && j != p.Ny - 1;
    const int64_t l = (int64_t)i + (int64_t)j * p.sy + (int64_t)k * p.sz;
    double v[5];
    if (interior) {
        v[0] = io.Pw1[l];
        v[2] = io.Sn1[l];
        if constexpr (MODEL == 3) {
            v[1] = io.Sw1[l];
            v[3] = v[4] = v[0];
        }
    } else {
        const int64_t l1 = inward(p, i, j, k);
        const double Pw = io.Pw1[l1], Sn = io.Sn1[l1];
        const double Sw = MODEL == 3 ? io.Sw1[l1] : 0.;
        double ro_eff = 0.;
        if constexpr (MODEL == 2) {
            if (j == p.Ny - 1) {
                double ro[2];
                densities2<CLOSURE>(p, io, l1, ro);
                ro_eff = (ro[1] * Sn + ro[0] * (1 - Sn)) * io.m[l1] * p.g * p.hy;
            }
        }
        boundary_values<MODEL>(p, i, j, k, Pw, Sw, Sn, ro_eff, v);
    }
    if constexpr (MODEL == 3) {
#pragma unroll
        for (int f = 0; f < 5; ++f) io.pack[(f * 2 + s) * plane + c] = v[f];
    } else {
        io.pack[s * plane + c] = v[0];
        io.pack[(2 + s) * plane + c] = v[2];
    }
}

// k_fused_faces followed, in the same launch, by the halo pack (threads past
// the face cells).
template <int MODEL, int CLOSURE>
__global__ void __launch_bounds__(256) k_fused_faces_pack(DevParams p, StepIO io, int64_t nfaces) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t < nfaces)
        fused_face<MODEL, CLOSURE>(p, io, t);
    else
        fused_pack<MODEL, CLOSURE>(p, io, t - nfaces);
}

// Workgroups of a kernel resident at once on the device (cached per kernel;
// one device type per process).
template <auto Kernel>
int resident_groups(int threads) {
    static int cached = 0;
    if (cached) return cached;
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, Kernel, threads, 0) != hipSuccess || per_cu < 1)
        return 512;
    cached = cus * per_cu;
    return cached;
}

}  // namespace capaz
