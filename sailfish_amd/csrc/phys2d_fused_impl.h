// phys2d_fused_impl.h -- kernels of the physics-mode barotropic substep (ROMS LF-AM3
// in 2D form, obsolete/step2d_LF_AM3.h.py:917-2780) as ONE launch per substep, for a
// single basin (k_phys_fused) and for an ensemble of basins (k_phys_ensemble).
// Included by phys2d_fused.hip (FP64 instances, C ABI) and phys2d_fused_f32.hip
// (FP32 instances).
//
// Each workgroup owns an output tile of TI x TJ points (all fields: zeta, ubar,
// vbar, their right-hand sides and the FP64 time averages of the tile's points).
// It loads a frame of (TI+5) x (TJ+5) points (3 to the low side, 2 to the high
// side) and evaluates the four stages of the substep on shrinking regions, so that
// no intermediate state ever goes to HBM:
//
//   stage  region (frame coords, core = [3, 3+T))   writes (LDS plane)
//   L      [0, T+5)    z1                               Z1
//   A      [1, T+5)    DU1 = D*u*on_u, DV1 = D*v*om_v   DU, DV
//   P1     [1, T+4)    predicted zeta zs, its RHS rz    ZS
//   P2     [2, T+4)    predicted ubar us, vbar vs       US, VS
//   C0     [2, T+4)    DUs, DVs of the predicted state  DU, DV (reused)
//   C1     [2, T+3)    corrected zeta z2 (+ averages)   Z1 (reused as Z2)
//   C2     [3, T+3)    corrected ubar, vbar             -
//
// Ten planes of (TI+5)(TJ+5) values: Z1, DU, DV, ZS, US, VS and ubar, vbar (t1), pm, pn over
// the whole frame, filled in stage L, so that every stencil neighbour of those fields is an
// LDS read; some instances add h, fomn and zeta(t0).  RZ stays with its thread (core) or in a
// row and a column of C1's ring.  The core points come first in every stage with the same
// thread mapping, so a thread keeps its core points' values (z1, u1, v1, zs, the predictor
// right-hand sides, metric factors) in registers from stage to stage.  The other read-only
// fields (fomn, the stresses, the old time level, the history right-hand sides) are read
// from global memory where they are used.
//
// Small grids are bound by the chain of six load, barrier and divide latencies, not by any
// rate: one wave per SIMD walks it.  There (NR > 0) the ring points get waves of their own,
// which run beside the core's instead of after them, and every global load of the tile is
// issued before the first barrier.
//
// Closed-basin boundary: a ghost rho point takes the value of its clamped interior source; u
// = 0 at i <= 1 and i = L, v = 0 at j <= 1 and j = M; the remaining ghost rows/columns of u
// and v copy their inward neighbour.  The source's thread writes its ghosts along with its own
// value (to LDS and to global memory), so no thread evaluates a formula at a ghost: against
// evaluating it there from fresh loads this saves 6 (FP32 64 x 8) to 31 (FP32 64 x 4)
// registers and up to four dependent load latencies in boundary tiles (128 x 64 FP64: 10.8 ->
// 9.1 us a substep).  The tile origin is shifted by one point when sz % T == 1 so that the
// source of every ghost point of a tile's core is a core point of the same tile.
//
// Expression order is the one of phys2d_kernels.hip: the FP64 instances (contraction
// off) equal the oracle and the four-launch form bit for bit; the FP32 instances are
// compiled with contraction on and agree with the four-launch FP32 form to rounding.
#pragma once

#include "mlp_net.h"
#include "sf_internal.h"

#include <type_traits>
#include <vector>

// the learned closure of a fused substep: the network and its Coriolis field
struct ClosureIn {
    const sf_mlp *mlp;
    const void *f;
};

// shape (xi, eta) of a tile
struct PhysTile {
    int ti, tj;
};

namespace {

template <typename T>
struct PFA {
    const T *h, *pm, *pn, *fomn, *sustr, *svstr;
    const T *z0, *z1, *u0, *u1, *v0, *v1;
    T *z2, *u2, *v2;
    const T *rz0, *ru0, *rv0;
    T *rz1, *ru1, *rv1;
    double *Zt, *DUa, *DVa;
    int szI, szJ, tiles_i, tiles_j, off_i, off_j;
    T g, rdrg, dt;
    int first;
    int nts;   // streaming (non-temporal) stores and average loads: set when one substep's
               // bytes exceed what the 256 MB last-level cache keeps for the next substep
    double w1;
    sf_couple_fields c;   // coupling with the baroclinic step (CPL instances only)
    // the learned closure evaluated in the tile (CLO instances only): network operands,
    // input normalisation {mu[45], 1/sd[45]}, output de-normalisation, Coriolis field
    const uint16_t *cl_wpk;
    const float *cl_w, *cl_norm;
    const T *cl_f;
    float cl_ynorm[4];
};

// FP64 closure instances of 64-wide tiles keep the network's feature tiles in frame planes
// 1..5, written only from stage A on, and one more (a barrier ends the closure phase): 27 KB
// less LDS, so two 64 x 4 workgroups fit a CU.  Smaller planes cannot hold the tiles; they
// get their own array.
template <typename T, bool CLO, int TI>
constexpr bool cl_tiles_in_frame = CLO && sizeof(T) == 8 && TI == 64;

// Registers against LDS reads: LEAN instances keep h in a plane too and read the core points'
// statics and t1 state from LDS where they are used; the others hold them in registers.
//  - FP64: at 122 VGPRs 64 x 8 tiles on 512 threads fit two workgroups, 16 waves, a CU where
//    256 threads of 209 VGPRs fit 8 (4096 x 4096: 970 us a substep against 1030; 2048 x 1024:
//    120 / 128); the coupled split form drops from 142 to 126 (768 x 384: 26 / 34 us).
//  - FP32 at streaming sizes (4096 x 4096: 547 us against 568); in the last-level cache the
//    registers are faster (2048 x 1024: 57.3 against 59.1).
template <typename T, int NT, int NR, bool CPL, bool NTS>
constexpr bool lean_regs = NR > 0 ? (CPL && sizeof(T) == 8) : (NT == 512 && (sizeof(T) == 8 || NTS));

// LDS planes of a tile's frame: the ten listed above.  NR > 0 (core and ring on different
// waves): h, fomn and zeta(t0) over the frame as well, so that every stencil neighbour of a
// static field is an LDS read and all global loads of the tile are issued together at its
// start.
template <typename T, int TI, int TJ, int NT, int NR, bool NTS, bool CPL, bool CLO>
struct PhysLds {
    static constexpr int FN = (TI + 5) * (TJ + 5);
    static constexpr int SP = cl_tiles_in_frame<T, CLO, TI> ? 1 : 0;   // spare plane of the feature tiles
    static constexpr bool HP = NR > 0 || CLO || lean_regs<T, NT, NR, CPL, NTS>;
    static constexpr int PLANES = 10 + SP + (NR > 0 ? 3 : (HP ? 1 : 0));
};

// Element (f + d) of p, given the byte offset boff of element f: the address is the
// array's scalar base plus a 32-bit vector offset (global_load saddr form).  The
// neighbour offset boff + d*sizeof(T) is computed in 32-bit arithmetic, so it is one
// vector add per neighbour and point, shared by every array read at that neighbour.
// All field pointers point to global memory; the explicit address space keeps the
// global_load/global_store forms also for pointers read from a member table.
#define SF_GLOBAL __attribute__((address_space(1)))
#define SF_CONST __attribute__((address_space(4)))
template <typename T>
__device__ __forceinline__ T ldo(const T *p, long long d, uint32_t boff)
{
    const uint32_t o = boff + (uint32_t)(d * (long long)sizeof(T));
    return *(const SF_GLOBAL T *)((const SF_GLOBAL char *)p + o);
}
// The outputs of a substep are read by no other workgroup of the launch, and the FP64
// averages are read once per point.  When a substep moves more bytes than the last-level
// cache keeps between launches, streaming (non-temporal) stores and average loads keep L2
// for the halo reads; below that size plain ones let the next substep find its inputs in
// that cache.  NTS is a template parameter: a runtime choice between the two store forms
// would be merged into one plain store by the compiler.
template <bool NTS>
__device__ __forceinline__ double ldavg(const double *p, uint32_t boff)
{
    if constexpr (NTS) return __builtin_nontemporal_load((const SF_GLOBAL double *)((const SF_GLOBAL char *)p + boff));
    return ldo(p, 0, boff);
}
template <bool NTS, typename T>
__device__ __forceinline__ void sto(T *p, uint32_t boff, T v)
{
    if constexpr (NTS) __builtin_nontemporal_store(v, (SF_GLOBAL T *)((SF_GLOBAL char *)p + boff));
    else *(SF_GLOBAL T *)((SF_GLOBAL char *)p + boff) = v;
}

// Workgroup barrier that orders LDS only: global loads issued before it stay in
// flight (the stages exchange data through LDS exclusively).
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Map ring index t of region [3-LO, 3+TI+HI) x [3-LO, 3+TJ+HI) minus the core to (a, b).
template <int TI, int TJ, int LO, int HI>
__device__ __forceinline__ void ring_point(int t, int &a, int &b)
{
    constexpr int W = TI + LO + HI, NBOT = LO * W, WROW = LO + HI, NMID = TJ * WROW;
    if (t < NBOT) {
        b = 3 - LO + t / W;
        a = 3 - LO + t % W;
    } else if (t < NBOT + NMID) {
        const int s = t - NBOT;
        b = 3 + s / WROW;
        const int c = s % WROW;
        a = c < LO ? 3 - LO + c : 3 + TI + (c - LO);
    } else {
        const int s = t - NBOT - NMID;
        b = 3 + TJ + s / W;
        a = 3 - LO + s % W;
    }
}
template <int TI, int TJ, int LO, int HI>
constexpr int ring_size() { return (TI + LO + HI) * (TJ + LO + HI) - TI * TJ; }

// inputs of the ubar / vbar right-hand side at a u / v point
template <typename T>
struct UVIn {
    T m1, m2, cff;              // u: onu, omu ; v: omv, onv
    T pmc, pmb, pnc, pnb;       // raw pm, pn at the point and the back neighbour (generic path)
    T hb, hc;                   // h at the back neighbour (i-1 / j-1) and the point
    T xb, xc, xf, yf, yb;       // same-component velocity: back, centre, forward, cross+, cross-
    T fc, fb;                   // fomn at the point and the back neighbour
    T oc, of, ob, obf;          // other component for Coriolis (see rhs_u / rhs_v)
    T st;                       // surface stress
    T x0, z0c, z0b;             // predictor "before" velocity and zeta (t0) at point / back
};

// The tile's arguments.  Closure instances (launched only as k_phys_fused, whose one kernel
// argument is P) read them through the kernel-argument segment pointer, which an empty asm
// statement re-derives after the closure phase; other instances use P itself.
template <typename T, bool CLO>
__device__ __forceinline__ auto arg_ptr(const PFA<T> &P)
{
    if constexpr (CLO) return (const __attribute__((address_space(4))) PFA<T> *)__builtin_amdgcn_kernarg_segment_ptr();
    else return &P;
}

// Which points a call of phys_tile computes: every thread its core points and then its
// share of the ring, or (NR > 0) the core points only / the ring only.
enum TileRole { ROLE_ALL, ROLE_CORE, ROLE_RING };

template <typename T, int TI, int TJ, int NT, int NR, TileRole ROLE, bool FIRST, bool NTS, bool CPL = false,
          bool CLO = false>
__device__ __forceinline__ void phys_tile(const PFA<T> &P, int ti, int tj, T (*sm)[(TI + 5) * (TJ + 5)], T *rzl,
                                          uint32_t *clX = nullptr, float *clN = nullptr, T *clF = nullptr)
{
    // the arguments through a pointer that the closure instances re-derive after the closure
    // phase, so that pointers first needed from stage A on are loaded there again instead of
    // being held across the phase
    auto Pp = arg_ptr<T, CLO>(P);
    constexpr bool XP = NR > 0;              // h, fomn, zeta(t0) planes; all loads issued first
    constexpr bool CORE = ROLE != ROLE_RING, RINGS = ROLE != ROLE_CORE;
    static_assert(XP == (ROLE != ROLE_ALL), "core and ring roles go with their own ring threads");
    constexpr int RT = XP ? NR : NT;         // threads that share the ring
    constexpr int FW = TI + 5;
    constexpr int KC = CORE ? TI * TJ / NT : 1;
    constexpr uint32_t ES = sizeof(T);
    T *const sZ1 = sm[0], *const sZ2 = sm[0];
    T *const sDU = sm[1], *const sDV = sm[2];
    T *const sZS = sm[3], *const sUS = sm[4], *const sVS = sm[5];
    // read-only after L: ubar, vbar at t1, pm, pn; HP: h; XP: fomn, zeta at t0
    using Lds = PhysLds<T, TI, TJ, NT, NR, NTS, CPL, CLO>;
    constexpr bool HP = Lds::HP, LEAN = lean_regs<T, NT, NR, CPL, NTS>;
    constexpr int S0 = 6 + Lds::SP;
    T *const sU1 = sm[S0], *const sV1 = sm[S0 + 1];
    T *const sPM = sm[S0 + 2], *const sPN = sm[S0 + 3];
    T *const sH = sm[HP ? S0 + 4 : 0];
    T *const sFO = sm[XP ? S0 + 5 : 0], *const sZ0 = sm[XP ? S0 + 6 : 0];

    const int szI = Pp->szI, szJ = Pp->szJ, L = szI - 1, M = szJ - 1;
    const long long W = szI;
    const int fi0 = ti * TI - Pp->off_i - 3, fj0 = tj * TJ - Pp->off_j - 3;   // frame origin
    const int tid = threadIdx.x, rtid = XP ? tid - NT : tid;
    const T dt = Pp->dt;
    constexpr bool first = FIRST;

    auto inside = [&](int i, int j) { return i >= 0 && i <= L && j >= 0 && j <= M; };
    auto off = [&](int i, int j) { return (uint32_t)(j * szI + i) * ES; };
    auto offd = [&](int i, int j) { return (uint32_t)(j * szI + i) * 8u; };
    auto core_ab = [&](int k, int &a, int &b) {
        const int idx = tid + k * NT;
        a = 3 + idx % TI;
        b = 3 + idx / TI;
    };
    auto rho_int = [&](int i, int j) { return i >= 1 && i <= L - 1 && j >= 1 && j <= M - 1; };
    auto u_int = [&](int i, int j) { return i >= 2 && i <= L - 1 && j >= 1 && j <= M - 1; };
    auto v_int = [&](int i, int j) { return i >= 1 && i <= L - 1 && j >= 2 && j <= M - 1; };

    // Closed-basin ghosts: a ghost point is written by the thread of its interior source,
    // together with the source's own value.  di (dj): step from a source in the outermost
    // interior column (row) to its ghost, else 0.
    auto ghost_di = [&](int i) { return i == 1 ? -1 : (i == L - 1 ? 1 : 0); };
    auto ghost_dj = [&](int j) { return j == 1 ? -1 : (j == M - 1 ? 1 : 0); };
    auto put_rho = [&](T *p, int o, int i, int j, T v) {
        const int di = ghost_di(i), dj = ghost_dj(j) * FW;
        p[o] = v;
        if (di) p[o + di] = v;
        if (dj) {
            p[o + dj] = v;
            if (di) p[o + dj + di] = v;
        }
    };
    auto put_u = [&](T *p, int o, int j, T v) {   // ghost rows
        const int dj = ghost_dj(j) * FW;
        p[o] = v;
        if (dj) p[o + dj] = v;
    };
    auto put_v = [&](T *p, int o, int i, T v) {   // ghost columns
        const int di = ghost_di(i);
        p[o] = v;
        if (di) p[o + di] = v;
    };
    // u is 0 at i <= 1 and i = L (v likewise), written by the point itself
    auto u_wall = [&](int i) { return i < 2 || i > L - 1; };
    auto v_wall = [&](int j) { return j < 2 || j > M - 1; };

    // metric factors of u / v inputs
    auto metrics_u = [&](UVIn<T> &x) {
        x.m1 = T(2) * sf::recip(x.pnb + x.pnc);
        x.m2 = T(2) * sf::recip(x.pmb + x.pmc);
        x.cff = (x.pmc + x.pmb) * (x.pnc + x.pnb);
    };
    auto metrics_v = [&](UVIn<T> &x) {
        x.m1 = T(2) * sf::recip(x.pmb + x.pmc);
        x.m2 = T(2) * sf::recip(x.pnb + x.pnc);
        x.cff = (x.pmc + x.pmb) * (x.pnc + x.pnb);
    };
    // face fluxes DU, DV of a ring point of state (z, u, v) at LDS index o; h at the point and
    // its west / south neighbour from the plane or (no plane) rh, rhw, rhs
    auto flux = [&](const T *z, const T *u, const T *v, int i, int j, int o, T rh, T rhw, T rhs) {
        T du = T(0), dv = T(0);
        if (inside(i, j)) {
            const T hc = HP ? sH[o] : rh;
            if (i >= 1) {
                const T onu = T(2) * sf::recip(sPN[o - 1] + sPN[o]);
                du = ((T(0.5) * (((HP ? sH[o - 1] : rhw) + z[o - 1]) + (hc + z[o]))) * u[o]) * onu;
            }
            if (j >= 1) {
                const T omv = T(2) * sf::recip(sPM[o - FW] + sPM[o]);
                dv = ((T(0.5) * (((HP ? sH[o - FW] : rhs) + z[o - FW]) + (hc + z[o]))) * v[o]) * omv;
            }
        }
        sDU[o] = du;
        sDV[o] = dv;
    };
    // h of ring point (i, j): loaded ahead of the core's work where no plane holds it
    auto load_h = [&](int i, int j, T &hc, T &hw, T &hs) {
        if constexpr (!HP) {
            if (inside(i, j)) {
                const uint32_t f = off(i, j);
                hc = ldo(Pp->h, 0, f);
                if (i >= 1) hw = ldo(Pp->h, -1, f);
                if (j >= 1) hs = ldo(Pp->h, -W, f);
            }
        }
    };
    // inputs of the u / v right-hand side of a ring point: the values that come from global
    // memory (offset f) and those in the frame's planes (LDS index q)
    auto load_u_global = [&](UVIn<T> &x, uint32_t f) {
        if constexpr (!HP) {
            x.hb = ldo(Pp->h, -1, f);
            x.hc = ldo(Pp->h, 0, f);
        }
        if constexpr (!XP) {
            x.fc = ldo(Pp->fomn, 0, f);
            x.fb = ldo(Pp->fomn, -1, f);
            x.z0c = first ? T(0) : ldo(Pp->z0, 0, f);
            x.z0b = first ? T(0) : ldo(Pp->z0, -1, f);
        }
        x.st = ldo(Pp->sustr, 0, f);
        if (!first) x.x0 = ldo(Pp->u0, 0, f);
    };
    auto load_u_lds = [&](UVIn<T> &x, int q) {
        x.pmc = sPM[q];
        x.pmb = sPM[q - 1];
        x.pnc = sPN[q];
        x.pnb = sPN[q - 1];
        if constexpr (HP) {
            x.hb = sH[q - 1];
            x.hc = sH[q];
        }
        if constexpr (XP) {
            x.fc = sFO[q];
            x.fb = sFO[q - 1];
            x.z0c = first ? T(0) : sZ0[q];
            x.z0b = first ? T(0) : sZ0[q - 1];
        }
        x.xb = sU1[q - 1];
        x.xc = sU1[q];
        x.xf = sU1[q + 1];
        x.yf = sU1[q + FW];
        x.yb = sU1[q - FW];
        x.oc = sV1[q];
        x.of = sV1[q + FW];
        x.ob = sV1[q - 1];
        x.obf = sV1[q + FW - 1];
        if (first) x.x0 = x.xc;
    };
    auto load_v_global = [&](UVIn<T> &x, uint32_t f) {
        if constexpr (!HP) {
            x.hb = ldo(Pp->h, -W, f);
            x.hc = ldo(Pp->h, 0, f);
        }
        if constexpr (!XP) {
            x.fc = ldo(Pp->fomn, 0, f);
            x.fb = ldo(Pp->fomn, -W, f);
            x.z0c = first ? T(0) : ldo(Pp->z0, 0, f);
            x.z0b = first ? T(0) : ldo(Pp->z0, -W, f);
        }
        x.st = ldo(Pp->svstr, 0, f);
        if (!first) x.x0 = ldo(Pp->v0, 0, f);
    };
    auto load_v_lds = [&](UVIn<T> &x, int q) {
        x.pmc = sPM[q];
        x.pmb = sPM[q - FW];
        x.pnc = sPN[q];
        x.pnb = sPN[q - FW];
        if constexpr (HP) {
            x.hb = sH[q - FW];
            x.hc = sH[q];
        }
        if constexpr (XP) {
            x.fc = sFO[q];
            x.fb = sFO[q - FW];
            x.z0c = first ? T(0) : sZ0[q];
            x.z0b = first ? T(0) : sZ0[q - FW];
        }
        x.xb = sV1[q - FW];
        x.xc = sV1[q];
        x.xf = sV1[q + FW];
        x.yf = sV1[q + 1];
        x.yb = sV1[q - 1];
        x.oc = sU1[q];
        x.of = sU1[q + 1];
        x.ob = sU1[q - FW];
        x.obf = sU1[q + 1 - FW];
        if (first) x.x0 = x.xc;
    };

    // CPL: forcing of the predictor right-hand side r of a u (v) point: the first substep
    // forms F = rufrc - r and adds its Adams-Bashforth extrapolation over the baroclinic
    // steps, the others add F (as pred_forcing of the four-launch form); F is returned in Fk
    struct Forcing { double f0, f1, f2; };
    auto load_forcing = [&](bool vdir, uint32_t fd) {
        Forcing q{0.0, 0.0, 0.0};
        if constexpr (FIRST) {
            q.f0 = ldo(vdir ? Pp->c.rvfrc : Pp->c.rufrc, 0, fd);
            if (Pp->c.ab > 0) q.f1 = ldo(vdir ? Pp->c.Fv1 : Pp->c.Fu1, 0, fd);
            if (Pp->c.ab > 1) q.f2 = ldo(vdir ? Pp->c.Fv2 : Pp->c.Fu2, 0, fd);
        } else {
            q.f0 = ldo(vdir ? Pp->c.Fv : Pp->c.Fu, 0, fd);
        }
        return q;
    };
    auto pred_forcing = [&](const Forcing &q, T r, double &Fk) {
        if constexpr (FIRST) {
            const double F = q.f0 - (double)r;
            Fk = F;
            return r + T(sf::ab_extrapolate(Pp->c.ab, F, q.f1, q.f2));
        } else {
            Fk = q.f0;
            return r + T(Fk);
        }
    };

    // ---- predictor momentum at LDS index q from inputs x (returns rhs in r) ----------
    const T cff4 = T(4.0 / 25.0), cff5 = T(1) - T(2) * cff4;
    const T c1dt = first ? T(0.5) * dt : dt;
    auto gzp = [&](int o, T z0) { return first ? T(0.5) * (sZ1[o] + sZS[o]) : cff5 * sZ1[o] + cff4 * (z0 + sZS[o]); };
    auto Dbp = [&](int o, T h, T z0) { return first ? h + sZ1[o] : h + z0; };
    auto pred_u = [&](int q, const UVIn<T> &x, T &r, const Forcing &fq, double &Fk) {
        const T onu = x.m1, omu = x.m2;
        const T g0 = gzp(q - 1, x.z0b), g1 = gzp(q, x.z0c);
        r = ((T(0.5) * Pp->g) * onu) * ((x.hb + x.hc) * (g0 - g1) + (g0 * g0 - g1 * g1));
        const T UFx1 = T(0.25) * (sDU[q] + sDU[q + 1]) * (x.xc + x.xf);
        const T UFx0 = T(0.25) * (sDU[q - 1] + sDU[q]) * (x.xb + x.xc);
        const T UFe1 = T(0.25) * (sDV[q + FW] + sDV[q + FW - 1]) * (x.yf + x.xc);
        const T UFe0 = T(0.25) * (sDV[q] + sDV[q - 1]) * (x.xc + x.yb);
        r = r - ((UFx1 - UFx0) + (UFe1 - UFe0));
        const T cr1 = ((T(0.5) * (x.hc + sZ1[q])) * x.fc) * (x.oc + x.of);
        const T cr0 = ((T(0.5) * (x.hb + sZ1[q - 1])) * x.fb) * (x.ob + x.obf);
        r = r + T(0.5) * (cr1 + cr0);
        r = r - ((Pp->rdrg * x.xc) * omu) * onu;
        r = r + (x.st * omu) * onu;
        if constexpr (CPL) r = pred_forcing(fq, r, Fk);
        const T fac = sf::recip((x.hc + sZS[q]) + (x.hb + sZS[q - 1]));
        return (x.x0 * (Dbp(q, x.hc, x.z0c) + Dbp(q - 1, x.hb, x.z0b)) + (x.cff * c1dt) * r) * fac;
    };
    auto pred_v = [&](int q, const UVIn<T> &x, T &r, const Forcing &fq, double &Fk) {
        const T omv = x.m1, onv = x.m2;
        const T g0 = gzp(q - FW, x.z0b), g1 = gzp(q, x.z0c);
        r = ((T(0.5) * Pp->g) * omv) * ((x.hb + x.hc) * (g0 - g1) + (g0 * g0 - g1 * g1));
        const T VFx1 = T(0.25) * (sDU[q + 1] + sDU[q + 1 - FW]) * (x.yf + x.xc);
        const T VFx0 = T(0.25) * (sDU[q] + sDU[q - FW]) * (x.xc + x.yb);
        const T VFe1 = T(0.25) * (sDV[q] + sDV[q + FW]) * (x.xc + x.xf);
        const T VFe0 = T(0.25) * (sDV[q - FW] + sDV[q]) * (x.xb + x.xc);
        r = r - ((VFx1 - VFx0) + (VFe1 - VFe0));
        const T cr1 = ((T(0.5) * (x.hc + sZ1[q])) * x.fc) * (x.oc + x.of);
        const T cr0 = ((T(0.5) * (x.hb + sZ1[q - FW])) * x.fb) * (x.ob + x.obf);
        r = r - T(0.5) * (cr1 + cr0);
        r = r - ((Pp->rdrg * x.xc) * omv) * onv;
        r = r + (x.st * omv) * onv;
        if constexpr (CPL) r = pred_forcing(fq, r, Fk);
        const T fac = sf::recip((x.hc + sZS[q]) + (x.hb + sZS[q - FW]));
        return (x.x0 * (Dbp(q, x.hc, x.z0c) + Dbp(q - FW, x.hb, x.z0b)) + (x.cff * c1dt) * r) * fac;
    };

    // ============ core-point registers ============
    bool cin[KC];
    uint32_t cf[KC];
    T z1c[KC], u1c[KC], v1c[KC], hc_[KC], hw_[KC], hs_[KC];
    T clf0[CLO ? KC : 1];                            // CLO: f at the core point
    T clsu[CLO ? KC : 1], clsv[CLO ? KC : 1];       // CLO: wind stress at the core point
    T pm_[KC], pn_[KC];
    T onuc[KC], omuc[KC], cffuc[KC], omvc[KC], onvc[KC], cffvc[KC], pmnc[KC];
    T zsc[KC], rzc[KC], ruc[KC], rvc[KC], duc[KC], dvc[KC];
    // G1 (predictor) and G2 (corrector) prefetch
    T z0c_[KC], z0w_[KC], z0s_[KC], u0c_[KC], v0c_[KC], fo_[KC], fow_[KC], fos_[KC], su_[KC], sv_[KC];
    T rz0_[KC], ru0_[KC], rv0_[KC], z1w_[KC], z1s_[KC];
    double zt_[KC], dua_[KC], dva_[KC];
    // core values at slot k, LDS index o: held in registers, or (LEAN) read where used
    auto h_c = [&](int k, int o) { if constexpr (LEAN) return sH[o]; else return hc_[k]; };
    auto h_w = [&](int k, int o) { if constexpr (LEAN) return sH[o - 1]; else return hw_[k]; };
    auto h_s = [&](int k, int o) { if constexpr (LEAN) return sH[o - FW]; else return hs_[k]; };
    auto u1_c = [&](int k, int o) { if constexpr (LEAN) return sU1[o]; else return u1c[k]; };
    auto v1_c = [&](int k, int o) { if constexpr (LEAN) return sV1[o]; else return v1c[k]; };
    auto cff_u = [&](int o) { return (sPM[o] + sPM[o - 1]) * (sPN[o] + sPN[o - 1]); };
    auto cff_v = [&](int o) { return (sPM[o] + sPM[o - FW]) * (sPN[o] + sPN[o - FW]); };
    // CPL: stage-A fluxes of the core points, their forcing F and DU_avg2 / DV_avg2
    T du1c[KC], dv1c[KC], fuc[KC], fvc[KC];
    double du2_[KC], dv2_[KC];
    Forcing fqu[KC], fqv[KC];

    // core: the predictor's inputs (G1)
    auto issue_pred = [&](int k) {
        int a, b;
        core_ab(k, a, b);
        const int i = fi0 + a, j = fj0 + b;
        const uint32_t f = cf[k];
        const bool ui = cin[k] && u_int(i, j), vi = cin[k] && v_int(i, j), ri_ = cin[k] && rho_int(i, j);
        if constexpr (!XP) {
            if (ri_) {   // holds every u and v point
                if (!first) z0c_[k] = ldo(Pp->z0, 0, f);
                fo_[k] = ldo(Pp->fomn, 0, f);
            }
        }
        if (ui) {
            if constexpr (!XP) {
                if (!first) z0w_[k] = ldo(Pp->z0, -1, f);
                fow_[k] = ldo(Pp->fomn, -1, f);
            }
            if (!first) u0c_[k] = ldo(Pp->u0, 0, f);
            su_[k] = ldo(Pp->sustr, 0, f);
            if constexpr (CPL && XP) fqu[k] = load_forcing(false, offd(i, j));
        }
        if (vi) {
            if constexpr (!XP) {
                if (!first) z0s_[k] = ldo(Pp->z0, -W, f);
                fos_[k] = ldo(Pp->fomn, -W, f);
            }
            if (!first) v0c_[k] = ldo(Pp->v0, 0, f);
            sv_[k] = ldo(Pp->svstr, 0, f);
            if constexpr (CPL && XP) fqv[k] = load_forcing(true, offd(i, j));
        }
    };
    // core: the averages of an interior point, issued in C0: the ring of P2 needs the registers
    auto issue_avg = [&](int k, uint32_t fd) {
        zt_[k] = ldavg<NTS>(Pp->Zt, fd);
        dua_[k] = ldavg<NTS>(Pp->DUa, fd);
        dva_[k] = ldavg<NTS>(Pp->DVa, fd);
        if constexpr (CPL) {
            du2_[k] = FIRST ? 0.0 : ldavg<NTS>(Pp->c.DU_avg2, fd);
            dv2_[k] = FIRST ? 0.0 : ldavg<NTS>(Pp->c.DV_avg2, fd);
        }
    };
    // core: the corrector's inputs (G2); LEAN: issued in C0, with the Coriolis factors, the
    // stress and the forcing read again rather than held across the ring of P2
    auto issue_corr = [&](int k, bool avg) {
        int a, b;
        core_ab(k, a, b);
        const int i = fi0 + a, j = fj0 + b;
        const uint32_t f = cf[k], fd = offd(i, j);
        constexpr bool again = LEAN && !XP;
        if (rho_int(i, j)) {
            if (!first) rz0_[k] = ldo(Pp->rz0, 0, f);
            if (avg) issue_avg(k, fd);
            if constexpr (again) fo_[k] = ldo(Pp->fomn, 0, f);
        }
        if (u_int(i, j)) {
            if (!first) ru0_[k] = ldo(Pp->ru0, 0, f);
            if constexpr (again) {
                fow_[k] = ldo(Pp->fomn, -1, f);
                su_[k] = ldo(Pp->sustr, 0, f);
                if constexpr (CPL && !FIRST) fuc[k] = T(ldo(Pp->c.Fu, 0, fd));
            }
        }
        if (v_int(i, j)) {
            if (!first) rv0_[k] = ldo(Pp->rv0, 0, f);
            if constexpr (again) {
                fos_[k] = ldo(Pp->fomn, -W, f);
                sv_[k] = ldo(Pp->svstr, 0, f);
                if constexpr (CPL && !FIRST) fvc[k] = T(ldo(Pp->c.Fv, 0, fd));
            }
        }
    };

    // ring slots of each stage
    constexpr int RSL = (ring_size<TI, TJ, 3, 2>() + RT - 1) / RT;
    constexpr int RSP2 = (ring_size<TI, TJ, 1, 1>() + RT - 1) / RT;
    constexpr int RSC1 = (ring_size<TI, TJ, 1, 0>() + RT - 1) / RT;
    // XP: inputs of the ring's later stages, loaded with the frame
    UVIn<T> xu[XP ? RSP2 : 1], xv[XP ? RSP2 : 1];
    Forcing xfu[XP ? RSP2 : 1], xfv[XP ? RSP2 : 1];
    T xrz0[XP ? RSC1 : 1];

    if constexpr (CLO && CORE)   // input normalisation of the closure (read after L's barrier)
        if (tid < 2 * NIN) clN[tid] = Pp->cl_norm[tid];

    // ---- G0 + L: z1 over the frame; core statics -----------------------------------------
    if constexpr (CORE) {
        T z0f[KC], fof[KC];
#pragma unroll
        for (int k = 0; k < KC; k++) {
            int a, b;
            core_ab(k, a, b);
            const int i = fi0 + a, j = fj0 + b;
            cin[k] = inside(i, j);
            cf[k] = cin[k] ? off(i, j) : 0u;
            const uint32_t f = cf[k];
            // values below are read only under the predicate they are loaded under
            z1c[k] = u1c[k] = v1c[k] = hc_[k] = pm_[k] = pn_[k] = T(0);
            if constexpr (XP) z0f[k] = fof[k] = T(0);
            if (cin[k]) {
                z1c[k] = ldo(Pp->z1, 0, f);
                u1c[k] = ldo(Pp->u1, 0, f);
                v1c[k] = ldo(Pp->v1, 0, f);
                hc_[k] = ldo(Pp->h, 0, f);
                pm_[k] = ldo(Pp->pm, 0, f);
                pn_[k] = ldo(Pp->pn, 0, f);
                if constexpr (XP) {
                    fof[k] = ldo(Pp->fomn, 0, f);
                    if (!first) z0f[k] = ldo(Pp->z0, 0, f);
                } else if constexpr (!LEAN) {
                    if (i >= 1) hw_[k] = ldo(Pp->h, -1, f);
                    if (j >= 1) hs_[k] = ldo(Pp->h, -W, f);
                }
            }
            if constexpr (CLO) {   // the closure's f and wind stress, in flight with the frame loads
                clf0[k] = cin[k] ? ldo(Pp->cl_f, 0, f) : T(0);
                clsu[k] = u_int(i, j) ? ldo(Pp->sustr, 0, f) : T(0);
                clsv[k] = v_int(i, j) ? ldo(Pp->svstr, 0, f) : T(0);
            }
        }
        if constexpr (XP) {
#pragma unroll
            for (int k = 0; k < KC; k++) issue_pred(k);
#pragma unroll
            for (int k = 0; k < KC; k++) issue_corr(k, true);
#pragma unroll
            for (int k = 0; k < KC; k++) {
                int a, b;
                core_ab(k, a, b);
                const int o = b * FW + a;
                sFO[o] = fof[k];
                if (!first) sZ0[o] = z0f[k];
            }
        }
    }
    {
        T rz[RSL], ru[RSL], rv[RSL], rm[RSL], rn[RSL], rfo[XP ? RSL : 1], rz0[XP ? RSL : 1];
        T rh[HP ? RSL : 1], rf[CLO ? RSL : 1];   // CLO: f of the ring for the closure's stencils
        int ro[RSL];
        if constexpr (RINGS) {
            constexpr int RING = ring_size<TI, TJ, 3, 2>();
#pragma unroll
            for (int s = 0; s < RSL; s++) {
                const int t = rtid + s * RT;
                rz[s] = ru[s] = rv[s] = rm[s] = rn[s] = T(0);
                if constexpr (HP) rh[s] = T(0);
                if constexpr (XP) rfo[s] = rz0[s] = T(0);
                if constexpr (CLO) rf[s] = T(0);
                ro[s] = -1;
                if (t < RING) {
                    int a, b;
                    ring_point<TI, TJ, 3, 2>(t, a, b);
                    const int i = fi0 + a, j = fj0 + b;
                    ro[s] = b * FW + a;
                    if (inside(i, j)) {
                        const uint32_t f = off(i, j);
                        rz[s] = ldo(Pp->z1, 0, f);
                        ru[s] = ldo(Pp->u1, 0, f);
                        rv[s] = ldo(Pp->v1, 0, f);
                        rm[s] = ldo(Pp->pm, 0, f);
                        rn[s] = ldo(Pp->pn, 0, f);
                        if constexpr (HP) rh[s] = ldo(Pp->h, 0, f);
                        if constexpr (XP) {
                            rfo[s] = ldo(Pp->fomn, 0, f);
                            if (!first) rz0[s] = ldo(Pp->z0, 0, f);
                        }
                        if constexpr (CLO) rf[s] = ldo(Pp->cl_f, 0, f);
                    }
                }
            }
            if constexpr (XP) {   // the later stages' global inputs, in flight behind the frame
#pragma unroll
                for (int s = 0; s < RSP2; s++) {
                    const int t = rtid + s * RT;
                    if (t < ring_size<TI, TJ, 1, 1>()) {
                        int a, b;
                        ring_point<TI, TJ, 1, 1>(t, a, b);
                        const int i = fi0 + a, j = fj0 + b;
                        if (u_int(i, j)) {
                            load_u_global(xu[s], off(i, j));
                            if constexpr (CPL) xfu[s] = load_forcing(false, offd(i, j));
                        }
                        if (v_int(i, j)) {
                            load_v_global(xv[s], off(i, j));
                            if constexpr (CPL) xfv[s] = load_forcing(true, offd(i, j));
                        }
                    }
                }
#pragma unroll
                for (int s = 0; s < RSC1; s++) {
                    const int t = rtid + s * RT;
                    if (t < ring_size<TI, TJ, 1, 0>()) {
                        int a, b;
                        ring_point<TI, TJ, 1, 0>(t, a, b);
                        if (!first && rho_int(fi0 + a, fj0 + b)) xrz0[s] = ldo(Pp->rz0, 0, off(fi0 + a, fj0 + b));
                    }
                }
            }
        }
        if constexpr (CORE) {
#pragma unroll
            for (int k = 0; k < KC; k++) {
                int a, b;
                core_ab(k, a, b);
                const int o = b * FW + a;
                sZ1[o] = z1c[k];
                sU1[o] = u1c[k];
                sV1[o] = v1c[k];
                sPM[o] = pm_[k];
                sPN[o] = pn_[k];
                if constexpr (HP) sH[o] = hc_[k];
                if constexpr (CLO) clF[o] = clf0[k];
            }
        }
        if constexpr (RINGS) {
#pragma unroll
            for (int s = 0; s < RSL; s++)
                if (ro[s] >= 0) {
                    sZ1[ro[s]] = rz[s];
                    sU1[ro[s]] = ru[s];
                    sV1[ro[s]] = rv[s];
                    sPM[ro[s]] = rm[s];
                    sPN[ro[s]] = rn[s];
                    if constexpr (HP) sH[ro[s]] = rh[s];
                    if constexpr (XP) {
                        sFO[ro[s]] = rfo[s];
                        if (!first) sZ0[ro[s]] = rz0[s];
                    }
                    if constexpr (CLO) clF[ro[s]] = rf[s];
                }
        }
    }
    lds_barrier();

    // ---- CL: the learned closure's corrector-stage stresses at the core points ----------
    // Each wave evaluates the network on its core points, 64 at a time (features from the
    // t1 frame planes and the h, f planes staged with them) and keeps
    // sustr + R_u D_u / svstr + R_v D_v of its points for C2.  The same arithmetic as
    // sf_closure_stress.
    T csu[KC], csv[KC];
    if constexpr (CLO && CORE) {
#pragma clang fp contract(off)   // the same roundings as sf_closure_stress in both precisions
        Fwd Wn;
        load_fwd(Wn, Pp->cl_wpk, Pp->cl_w);
        uint32_t *X = clX + (tid >> 6) * (64 * XS);
#pragma unroll
        for (int k = 0; k < KC; k++) {
            int a, b;
            core_ab(k, a, b);
            const int i = fi0 + a, j = fj0 + b, o = b * FW + a;
            float xvv[NIN];
#pragma unroll
            for (int kk = 0; kk < NIN; kk++) {
                const int fld = kk / 9, dj = (kk % 9) / 3 - 1, di = kk % 3 - 1;
                const int d = dj * FW + di;
                const T *pl = fld == 0 ? sU1 : fld == 1 ? sV1 : fld == 2 ? sZ1 : fld == 3 ? sH : clF;
                const T cv = pl[o], nv = pl[o + d];
                xvv[kk] = (dj == 0 && di == 0) ? (float)cv : (float)(nv - cv);
            }
            closure_row(X, tid & 63, xvv, clN);
            float zu, zv;
            closure_eval(Wn, X, zu, zv);
            csu[k] = csv[k] = T(0);   // read in C2 only at u / v interior points
            if (u_int(i, j)) {
                const T Du = T(0.5) * ((sH[o - 1] + sZ1[o - 1]) + (sH[o] + sZ1[o]));
                csu[k] = clsu[k] + T(zu * Pp->cl_ynorm[1] + Pp->cl_ynorm[0]) * Du;
            }
            if (v_int(i, j)) {
                const T Dv = T(0.5) * ((sH[o - FW] + sZ1[o - FW]) + (sH[o] + sZ1[o]));
                csv[k] = clsv[k] + T(zv * Pp->cl_ynorm[3] + Pp->cl_ynorm[2]) * Dv;
            }
        }
    }

    if constexpr (cl_tiles_in_frame<T, CLO, TI>) lds_barrier();   // feature tiles read; planes 1..6 free
    if constexpr (CLO && CORE) asm volatile("" : "+s"(Pp));

    // ---- A: DU1 at u points, DV1 at v points ---------------------------------------------
    {
        constexpr int RING = ring_size<TI, TJ, 2, 2>();
        constexpr int RS = (RING + RT - 1) / RT;
        T rh[RS], rhw[RS], rhs[RS];
        if constexpr (RINGS) {
#pragma unroll
            for (int s = 0; s < RS; s++) {
                int a, b;
                ring_point<TI, TJ, 2, 2>(rtid + s * RT, a, b);
                if (rtid + s * RT < RING) load_h(fi0 + a, fj0 + b, rh[s], rhw[s], rhs[s]);
            }
        }
        // core: metric factors, fluxes
        if constexpr (CORE) {
#pragma unroll
            for (int k = 0; k < KC; k++) {
                int a, b;
                core_ab(k, a, b);
                const int i = fi0 + a, j = fj0 + b, o = b * FW + a;
                if constexpr (XP && !LEAN) {
                    hw_[k] = sH[o - 1];
                    hs_[k] = sH[o - FW];
                }
                T du = T(0), dv = T(0);
                if (cin[k]) {
                    const T pmc = LEAN ? sPM[o] : pm_[k], pnc = LEAN ? sPN[o] : pn_[k];
                    if constexpr (!LEAN) pmnc[k] = pmc * pnc;
                    if (i >= 1) {
                        const T pmw = sPM[o - 1], pnw = sPN[o - 1];
                        onuc[k] = T(2) * sf::recip(pnw + pnc);
                        omuc[k] = T(2) * sf::recip(pmw + pmc);
                        if constexpr (!LEAN) cffuc[k] = (pmc + pmw) * (pnc + pnw);
                        du = ((T(0.5) * ((h_w(k, o) + sZ1[o - 1]) + (h_c(k, o) + sZ1[o]))) * u1_c(k, o)) * onuc[k];
                    }
                    if constexpr (CPL) du1c[k] = du;
                    if (j >= 1) {
                        const T pms = sPM[o - FW], pns = sPN[o - FW];
                        omvc[k] = T(2) * sf::recip(pms + pmc);
                        onvc[k] = T(2) * sf::recip(pns + pnc);
                        if constexpr (!LEAN) cffvc[k] = (pmc + pms) * (pnc + pns);
                        dv = ((T(0.5) * ((h_s(k, o) + sZ1[o - FW]) + (h_c(k, o) + sZ1[o]))) * v1_c(k, o)) * omvc[k];
                    }
                    if constexpr (CPL) dv1c[k] = dv;
                }
                sDU[o] = du;
                sDV[o] = dv;
            }
        }
        // ring fluxes
        if constexpr (RINGS) {
#pragma unroll
            for (int s = 0; s < RS; s++) {
                if (rtid + s * RT >= RING) continue;
                int a, b;
                ring_point<TI, TJ, 2, 2>(rtid + s * RT, a, b);
                flux(sZ1, sU1, sV1, fi0 + a, fj0 + b, b * FW + a, rh[s], rhw[s], rhs[s]);
            }
        }
    }
    if constexpr (!XP) {
#pragma unroll
        for (int k = 0; k < KC; k++) issue_pred(k);
    }
    lds_barrier();

    // ---- P1: predicted zeta and its right-hand side -----------------------------------
    {
        constexpr int RING = ring_size<TI, TJ, 2, 1>();
        constexpr int RS = (RING + RT - 1) / RT;
        T rz0[RS];
        int ro[RS], ri[RS], rj[RS];
        if constexpr (RINGS) {
#pragma unroll
            for (int s = 0; s < RS; s++) {
                const int t = rtid + s * RT;
                ro[s] = -1;
                ri[s] = rj[s] = -1;
                if (t < RING) {
                    int a, b;
                    ring_point<TI, TJ, 2, 1>(t, a, b);
                    const int i = fi0 + a, j = fj0 + b;
                    ro[s] = b * FW + a;
                    if (rho_int(i, j)) {
                        ri[s] = i;
                        rj[s] = j;
                        if (!first) rz0[s] = XP ? sZ0[ro[s]] : ldo(Pp->z0, 0, off(i, j));
                    } else if (inside(i, j)) {
                        ro[s] = -1;           // a ghost: its source writes it
                    } else {
                        ro[s] = -2 - ro[s];   // outside: store zeros
                    }
                }
            }
        }
        auto zs_of = [&](int qo, T pmn, T z0, T &r) {
            r = (sDU[qo] - sDU[qo + 1]) + (sDV[qo] - sDV[qo + FW]);
            if (first) return sZ1[qo] + (pmn * dt) * r;
            return z0 + (pmn * (T(2) * dt)) * r;
        };
        if constexpr (CORE) {
#pragma unroll
            for (int k = 0; k < KC; k++) {
                int a, b;
                core_ab(k, a, b);
                const int i = fi0 + a, j = fj0 + b, o = b * FW + a;
                T zs = T(0), r = T(0);
                if (cin[k]) {
                    if (rho_int(i, j)) {
                        if constexpr (XP) z0c_[k] = first ? T(0) : sZ0[o];
                        const T pmn = LEAN ? sPM[o] * sPN[o] : pmnc[k];
                        zs = zs_of(o, pmn, z0c_[k], r);
                        sto<NTS>(Pp->rz1, cf[k], r);
                        put_rho(sZS, o, i, j, zs);
                    }
                } else {
                    sZS[o] = zs;
                }
                if constexpr (!LEAN) zsc[k] = zs;
                rzc[k] = r;
            }
        }
        if constexpr (RINGS) {
#pragma unroll
            for (int s = 0; s < RS; s++) {
                if (ro[s] == -1) continue;
                if (ro[s] < -1) {
                    sZS[-2 - ro[s]] = T(0);
                    continue;
                }
                T r;
                const T zs = zs_of(ro[s], sPM[ro[s]] * sPN[ro[s]], rz0[s], r);
                put_rho(sZS, ro[s], ri[s], rj[s], zs);
                const int a = ri[s] - fi0, b = rj[s] - fj0;
                if (b == 2) {   // the low row and column of C1's ring
                    if (a >= 2 && a < 3 + TI) rzl[a - 2] = r;
                } else if (a == 2 && b >= 3 && b < 3 + TJ) {
                    rzl[TI + 1 + b - 3] = r;
                }
            }
        }
    }
    lds_barrier();

    // ---- P2: predicted ubar / vbar --------------------------------------------------
    if constexpr (CORE) {
#pragma unroll
        for (int k = 0; k < KC; k++) {
            int a, b;
            core_ab(k, a, b);
            const int i = fi0 + a, j = fj0 + b, o = b * FW + a;
            if constexpr (XP) {
                fo_[k] = sFO[o];
                fow_[k] = sFO[o - 1];
                fos_[k] = sFO[o - FW];
                z0w_[k] = first ? T(0) : sZ0[o - 1];
                z0s_[k] = first ? T(0) : sZ0[o - FW];
            }
            if (u_int(i, j)) {
                UVIn<T> x;
                x.m1 = onuc[k];
                x.m2 = omuc[k];
                x.cff = LEAN ? cff_u(o) : cffuc[k];
                x.hb = h_w(k, o);
                x.hc = h_c(k, o);
                x.xb = sU1[o - 1];
                x.xc = u1_c(k, o);
                x.xf = sU1[o + 1];
                x.yf = sU1[o + FW];
                x.yb = sU1[o - FW];
                x.fc = fo_[k];
                x.fb = fow_[k];
                x.oc = v1_c(k, o);
                x.of = sV1[o + FW];
                x.ob = sV1[o - 1];
                x.obf = sV1[o + FW - 1];
                x.st = su_[k];
                x.x0 = first ? x.xc : u0c_[k];
                x.z0c = z0c_[k];
                x.z0b = z0w_[k];
                T r;
                double F = 0.0;
                Forcing fq{};
                if constexpr (CPL) fq = XP ? fqu[k] : load_forcing(false, offd(i, j));
                const T us = pred_u(o, x, r, fq, F);
                put_u(sUS, o, j, us);
                sto<NTS>(Pp->ru1, cf[k], r);
                ruc[k] = r;
                if constexpr (CPL) {
                    if constexpr (FIRST || !LEAN || XP) fuc[k] = T(F);
                    if constexpr (FIRST) sto<NTS>(Pp->c.Fu, offd(i, j), F);
                }
            } else if (!cin[k] || u_wall(i)) {
                sUS[o] = T(0);
            }
            if (v_int(i, j)) {
                UVIn<T> x;
                x.m1 = omvc[k];
                x.m2 = onvc[k];
                x.cff = LEAN ? cff_v(o) : cffvc[k];
                x.hb = h_s(k, o);
                x.hc = h_c(k, o);
                x.xb = sV1[o - FW];
                x.xc = v1_c(k, o);
                x.xf = sV1[o + FW];
                x.yf = sV1[o + 1];
                x.yb = sV1[o - 1];
                x.fc = fo_[k];
                x.fb = fos_[k];
                x.oc = u1_c(k, o);
                x.of = sU1[o + 1];
                x.ob = sU1[o - FW];
                x.obf = sU1[o + 1 - FW];
                x.st = sv_[k];
                x.x0 = first ? x.xc : v0c_[k];
                x.z0c = z0c_[k];
                x.z0b = z0s_[k];
                T r;
                double F = 0.0;
                Forcing fq{};
                if constexpr (CPL) fq = XP ? fqv[k] : load_forcing(true, offd(i, j));
                const T vs = pred_v(o, x, r, fq, F);
                put_v(sVS, o, i, vs);
                sto<NTS>(Pp->rv1, cf[k], r);
                rvc[k] = r;
                if constexpr (CPL) {
                    if constexpr (FIRST || !LEAN || XP) fvc[k] = T(F);
                    if constexpr (FIRST) sto<NTS>(Pp->c.Fv, offd(i, j), F);
                }
            } else if (!cin[k] || v_wall(j)) {
                sVS[o] = T(0);
            }
        }
        // core: issue the corrector inputs (G2)
#pragma unroll
        for (int k = 0; k < KC; k++) {
            int a, b;
            core_ab(k, a, b);
            const int i = fi0 + a, j = fj0 + b, o = b * FW + a;
            if constexpr (!XP && !LEAN) issue_corr(k, false);
            if constexpr (!LEAN) {   // the Z1 plane holds z1 until C1
                if (cin[k] && u_int(i, j)) z1w_[k] = sZ1[o - 1];
                if (cin[k] && v_int(i, j)) z1s_[k] = sZ1[o - FW];
            }
        }
    }
    if constexpr (RINGS) {
        constexpr int RING = ring_size<TI, TJ, 1, 1>();
#pragma unroll
        for (int s = 0; s < RSP2; s++) {
            const int t = rtid + s * RT;
            if (t >= RING) continue;
            int a, b;
            ring_point<TI, TJ, 1, 1>(t, a, b);
            const int i = fi0 + a, j = fj0 + b, o = b * FW + a;
            const bool in = inside(i, j);
            T r;
            double F;
            if (u_int(i, j)) {
                UVIn<T> x;
                Forcing fq{};
                if constexpr (XP) {
                    x = xu[s];
                    if constexpr (CPL) fq = xfu[s];
                } else {
                    load_u_global(x, off(i, j));
                    if constexpr (CPL) fq = load_forcing(false, offd(i, j));
                }
                load_u_lds(x, o);
                metrics_u(x);
                put_u(sUS, o, j, pred_u(o, x, r, fq, F));
            } else if (!in || u_wall(i)) {
                sUS[o] = T(0);
            }
            if (v_int(i, j)) {
                UVIn<T> x;
                Forcing fq{};
                if constexpr (XP) {
                    x = xv[s];
                    if constexpr (CPL) fq = xfv[s];
                } else {
                    load_v_global(x, off(i, j));
                    if constexpr (CPL) fq = load_forcing(true, offd(i, j));
                }
                load_v_lds(x, o);
                metrics_v(x);
                put_v(sVS, o, i, pred_v(o, x, r, fq, F));
            } else if (!in || v_wall(j)) {
                sVS[o] = T(0);
            }
        }
    }
    lds_barrier();

    // ---- C0: fluxes DUs, DVs of the predicted state ------------------------------------
    {
        constexpr int RING = ring_size<TI, TJ, 1, 1>();
        if constexpr (!XP && !LEAN && CORE) {
#pragma unroll
            for (int k = 0; k < KC; k++) {
                int a, b;
                core_ab(k, a, b);
                if (rho_int(fi0 + a, fj0 + b)) issue_avg(k, offd(fi0 + a, fj0 + b));
            }
        }
        T rh[RSP2], rhw[RSP2], rhs[RSP2];
        if constexpr (RINGS) {
#pragma unroll
            for (int s = 0; s < RSP2; s++) {
                int a, b;
                ring_point<TI, TJ, 1, 1>(rtid + s * RT, a, b);
                if (rtid + s * RT < RING) load_h(fi0 + a, fj0 + b, rh[s], rhw[s], rhs[s]);
            }
        }
        if constexpr (CORE) {
#pragma unroll
            for (int k = 0; k < KC; k++) {
                int a, b;
                core_ab(k, a, b);
                const int i = fi0 + a, j = fj0 + b, o = b * FW + a;
                if constexpr (LEAN) {
                    if constexpr (!XP) issue_corr(k, true);
                    z1w_[k] = sZ1[o - 1];   // the Z1 plane holds z1 until C1
                    z1s_[k] = sZ1[o - FW];
                }
                T du = T(0), dv = T(0);
                if (cin[k]) {
                    const T hc = h_c(k, o);
                    if (i >= 1) du = ((T(0.5) * ((h_w(k, o) + sZS[o - 1]) + (hc + sZS[o]))) * sUS[o]) * onuc[k];
                    if (j >= 1) dv = ((T(0.5) * ((h_s(k, o) + sZS[o - FW]) + (hc + sZS[o]))) * sVS[o]) * omvc[k];
                }
                sDU[o] = du;
                sDV[o] = dv;
                duc[k] = du;
                dvc[k] = dv;
            }
        }
        if constexpr (RINGS) {
#pragma unroll
            for (int s = 0; s < RSP2; s++) {
                if (rtid + s * RT >= RING) continue;
                int a, b;
                ring_point<TI, TJ, 1, 1>(rtid + s * RT, a, b);
                flux(sZS, sUS, sVS, fi0 + a, fj0 + b, b * FW + a, rh[s], rhw[s], rhs[s]);
            }
        }
    }
    lds_barrier();

    // ---- C1: corrected zeta, time averages ------------------------------------------
    const T a1 = dt * T(5.0) / T(12.0), a2 = dt * T(8.0) / T(12.0), a3 = dt * T(1.0) / T(12.0);
    {
        auto z2_of = [&](int qo, T pmn, T z1q, T rz1, T rz0) {
            const T r = (sDU[qo] - sDU[qo + 1]) + (sDV[qo] - sDV[qo + FW]);
            if (first) return z1q + pmn * (dt * r);
            return z1q + pmn * ((a1 * r + a2 * rz1) - a3 * rz0);
        };
        constexpr int RING = ring_size<TI, TJ, 1, 0>();
        T rrz0[RSC1];
        int ro[RSC1], ri[RSC1], rj[RSC1];
        if constexpr (RINGS) {
#pragma unroll
            for (int s = 0; s < RSC1; s++) {
                const int t = rtid + s * RT;
                ro[s] = -1;
                ri[s] = rj[s] = -1;
                if (t < RING) {
                    int a, b;
                    ring_point<TI, TJ, 1, 0>(t, a, b);
                    const int i = fi0 + a, j = fj0 + b;
                    ro[s] = b * FW + a;
                    if (rho_int(i, j)) {
                        ri[s] = i;
                        rj[s] = j;
                        if (!first) rrz0[s] = XP ? xrz0[s] : ldo(Pp->rz0, 0, off(i, j));
                    } else if (inside(i, j)) {
                        ro[s] = -1;
                    } else {
                        ro[s] = -2 - ro[s];
                    }
                }
            }
        }
        // Z2 reuses the Z1 plane: after the last barrier a point's z1 is read by its own
        // thread only (a ghost's, which its source overwrites, by none)
        if constexpr (CORE) {
#pragma unroll
            for (int k = 0; k < KC; k++) {
                int a, b;
                core_ab(k, a, b);
                const int i = fi0 + a, j = fj0 + b, o = b * FW + a;
                if (rho_int(i, j)) {
                    const T z2 = z2_of(o, LEAN ? sPM[o] * sPN[o] : pmnc[k], z1c[k], rzc[k], rz0_[k]);
                    const double w = Pp->w1;
                    const uint32_t fd = offd(i, j);
                    sto<NTS>(Pp->Zt, fd, zt_[k] + w * (double)(LEAN ? sZS[o] : zsc[k]));
                    sto<NTS>(Pp->DUa, fd, dua_[k] + w * (double)duc[k]);
                    sto<NTS>(Pp->DVa, fd, dva_[k] + w * (double)dvc[k]);
                    if constexpr (CPL) {
                        sto<NTS>(Pp->c.DU_avg2, fd, (du2_[k] + Pp->c.w2p * (double)du1c[k]) + Pp->c.w2c * (double)duc[k]);
                        sto<NTS>(Pp->c.DV_avg2, fd, (dv2_[k] + Pp->c.w2p * (double)dv1c[k]) + Pp->c.w2c * (double)dvc[k]);
                    }
                    const int di = ghost_di(i), dj = ghost_dj(j);
                    sto<NTS>(Pp->z2, cf[k], z2);
                    if (di) sto<NTS>(Pp->z2, off(i + di, j), z2);
                    if (dj) {
                        sto<NTS>(Pp->z2, off(i, j + dj), z2);
                        if (di) sto<NTS>(Pp->z2, off(i + di, j + dj), z2);
                    }
                    put_rho(sZ2, o, i, j, z2);
                } else if (!cin[k]) {
                    sZ2[o] = T(0);
                }
            }
        }
        if constexpr (RINGS) {
#pragma unroll
            for (int s = 0; s < RSC1; s++) {
                if (ro[s] == -1) continue;
                if (ro[s] < -1) {
                    sZ2[-2 - ro[s]] = T(0);
                    continue;
                }
                const int o = ro[s];
                const T rz1 = rj[s] - fj0 == 2 ? rzl[ri[s] - fi0 - 2] : rzl[TI + 1 + rj[s] - fj0 - 3];
                put_rho(sZ2, o, ri[s], rj[s], z2_of(o, sPM[o] * sPN[o], sZ1[o], rz1, rrz0[s]));
            }
        }
    }
    lds_barrier();

    // ---- C2: corrected ubar / vbar on the core -----------------------------------------
    if constexpr (CORE) {
        const T cf4 = T(2.0 / 5.0), cf5 = T(1) - cf4;
        const T b1 = T(0.5) * dt * T(5.0) / T(12.0), b2 = T(0.5) * dt * T(8.0) / T(12.0),
                b3 = T(0.5) * dt * T(1.0) / T(12.0);
        auto gzc = [&](int o) { return cf5 * sZ2[o] + cf4 * sZS[o]; };
        // corrected ubar at LDS index q: metrics m1 = onu, m2 = omu; statics hb/hc, fc/fb, st
        auto corr_u = [&](int q, T onu, T omu, T cff, T hb, T hc, T fc, T fb, T st, T ru1, T ru0, T z1c_, T z1b,
                          T u1c_, T F) {
            const T g0 = gzc(q - 1), g1 = gzc(q);
            T r = ((T(0.5) * Pp->g) * onu) * ((hb + hc) * (g0 - g1) + (g0 * g0 - g1 * g1));
            const T uc = sUS[q];
            const T UFx1 = T(0.25) * (sDU[q] + sDU[q + 1]) * (uc + sUS[q + 1]);
            const T UFx0 = T(0.25) * (sDU[q - 1] + sDU[q]) * (sUS[q - 1] + uc);
            const T UFe1 = T(0.25) * (sDV[q + FW] + sDV[q + FW - 1]) * (sUS[q + FW] + uc);
            const T UFe0 = T(0.25) * (sDV[q] + sDV[q - 1]) * (uc + sUS[q - FW]);
            r = r - ((UFx1 - UFx0) + (UFe1 - UFe0));
            const T cr1 = ((T(0.5) * (hc + sZS[q])) * fc) * (sVS[q] + sVS[q + FW]);
            const T cr0 = ((T(0.5) * (hb + sZS[q - 1])) * fb) * (sVS[q - 1] + sVS[q - 1 + FW]);
            r = r + T(0.5) * (cr1 + cr0);
            r = r - ((Pp->rdrg * uc) * omu) * onu;
            r = r + (st * omu) * onu;
            if constexpr (CPL) r = r + F;
            const T fac = sf::recip((hc + sZ2[q]) + (hb + sZ2[q - 1]));
            T tend;
            if (first) tend = (T(0.5) * dt) * r;
            else tend = (b1 * r + b2 * ru1) - b3 * ru0;
            return (u1c_ * ((hc + z1c_) + (hb + z1b)) + cff * tend) * fac;
        };
        auto corr_v = [&](int q, T omv, T onv, T cff, T hb, T hc, T fc, T fb, T st, T rv1, T rv0, T z1c_, T z1b,
                          T v1c_, T F) {
            const T g0 = gzc(q - FW), g1 = gzc(q);
            T r = ((T(0.5) * Pp->g) * omv) * ((hb + hc) * (g0 - g1) + (g0 * g0 - g1 * g1));
            const T vc = sVS[q];
            const T VFx1 = T(0.25) * (sDU[q + 1] + sDU[q + 1 - FW]) * (sVS[q + 1] + vc);
            const T VFx0 = T(0.25) * (sDU[q] + sDU[q - FW]) * (vc + sVS[q - 1]);
            const T VFe1 = T(0.25) * (sDV[q] + sDV[q + FW]) * (vc + sVS[q + FW]);
            const T VFe0 = T(0.25) * (sDV[q - FW] + sDV[q]) * (sVS[q - FW] + vc);
            r = r - ((VFx1 - VFx0) + (VFe1 - VFe0));
            const T cr1 = ((T(0.5) * (hc + sZS[q])) * fc) * (sUS[q] + sUS[q + 1]);
            const T cr0 = ((T(0.5) * (hb + sZS[q - FW])) * fb) * (sUS[q - FW] + sUS[q - FW + 1]);
            r = r - T(0.5) * (cr1 + cr0);
            r = r - ((Pp->rdrg * vc) * omv) * onv;
            r = r + (st * omv) * onv;
            if constexpr (CPL) r = r + F;
            const T fac = sf::recip((hc + sZ2[q]) + (hb + sZ2[q - FW]));
            T tend;
            if (first) tend = (T(0.5) * dt) * r;
            else tend = (b1 * r + b2 * rv1) - b3 * rv0;
            return (v1c_ * ((hc + z1c_) + (hb + z1b)) + cff * tend) * fac;
        };
#pragma unroll
        for (int k = 0; k < KC; k++) {
            int a, b;
            core_ab(k, a, b);
            const int i = fi0 + a, j = fj0 + b, o = b * FW + a;
            if (!cin[k]) continue;
            if (u_int(i, j)) {
                const T cff = LEAN ? cff_u(o) : cffuc[k];
                const T u2 = corr_u(o, onuc[k], omuc[k], cff, h_w(k, o), h_c(k, o), fo_[k], fow_[k],
                                    CLO ? csu[k] : su_[k], ruc[k], ru0_[k], z1c[k], z1w_[k], u1_c(k, o),
                                    CPL ? fuc[k] : T(0));
                sto<NTS>(Pp->u2, cf[k], u2);
                const int dj = ghost_dj(j);
                if (dj) sto<NTS>(Pp->u2, off(i, j + dj), u2);
            } else if (u_wall(i)) {
                sto<NTS>(Pp->u2, cf[k], T(0));
            }
            if (v_int(i, j)) {
                const T cff = LEAN ? cff_v(o) : cffvc[k];
                const T v2 = corr_v(o, omvc[k], onvc[k], cff, h_s(k, o), h_c(k, o), fo_[k], fos_[k],
                                    CLO ? csv[k] : sv_[k], rvc[k], rv0_[k], z1c[k], z1s_[k], v1_c(k, o),
                                    CPL ? fvc[k] : T(0));
                sto<NTS>(Pp->v2, cf[k], v2);
                const int di = ghost_di(i);
                if (di) sto<NTS>(Pp->v2, off(i + di, j), v2);
            } else if (v_wall(j)) {
                sto<NTS>(Pp->v2, cf[k], T(0));
            }
        }
    }
}

// Block id -> tile: each XCD (block id mod 8) walks a contiguous band of tiles so that
// neighbouring tiles share that XCD's L2.
__device__ __forceinline__ int xcd_band(int nblk)
{
    int b = blockIdx.x;
    if ((nblk & 7) == 0) b = (blockIdx.x & 7) * (nblk >> 3) + (blockIdx.x >> 3);
    return b;
}

template <typename T, int TI, int TJ, int NT, int NR, bool FIRST, bool NTS, bool CPL = false, bool CLO = false>
__global__ __launch_bounds__(NT + NR) void k_phys_fused(PFA<T> P)
{
    constexpr bool IN_FRAME = cl_tiles_in_frame<T, CLO, TI>;
    using Lds = PhysLds<T, TI, TJ, NT, NR, NTS, CPL, CLO>;
    __shared__ T sm[Lds::PLANES][Lds::FN];
    __shared__ T rzl[TI + TJ + 1];
    static_assert(!IN_FRAME || 6 * Lds::FN * sizeof(T) >= (NT / 64) * 64 * XS * sizeof(uint32_t),
                  "frame planes 1..6 hold the feature tiles");
    __shared__ __attribute__((aligned(16))) uint32_t clX[CLO && !IN_FRAME ? (NT / 64) * 64 * XS : 1];
    __shared__ float clN[CLO ? 2 * NIN : 1];
    __shared__ T clF[CLO ? Lds::FN : 1];   // f over the frame
    const int b = xcd_band(P.tiles_i * P.tiles_j), ti = b % P.tiles_i, tj = b / P.tiles_i;
    uint32_t *X = IN_FRAME ? (uint32_t *)sm[1] : clX;
    if constexpr (NR == 0) {
        phys_tile<T, TI, TJ, NT, NR, ROLE_ALL, FIRST, NTS, CPL, CLO>(P, ti, tj, sm, rzl, X, clN, clF);
    } else {
        // whole waves of one role each: the branch is on a scalar, and both sides meet the
        // same number of barriers
        if (__builtin_amdgcn_readfirstlane((int)threadIdx.x) < NT)
            phys_tile<T, TI, TJ, NT, NR, ROLE_CORE, FIRST, NTS, CPL, CLO>(P, ti, tj, sm, rzl, X, clN, clF);
        else
            phys_tile<T, TI, TJ, NT, NR, ROLE_RING, FIRST, NTS, CPL, CLO>(P, ti, tj, sm, rzl, X, clN, clF);
    }
}


template <typename T, int TI, int TJ, int NT, int NR = 0>
int launch_fused(const sf_phys_fields *x, double dt, int first, double w1, void *stream,
                 const sf_couple_fields *cp = nullptr, const ClosureIn *cl = nullptr)
{
    PFA<T> a;
    a.c = cp ? *cp : sf_couple_fields{};
    a.cl_wpk = cl ? cl->mlp->wpk : nullptr;
    a.cl_w = cl ? cl->mlp->w : nullptr;
    a.cl_norm = cl ? cl->mlp->norm : nullptr;
    a.cl_f = cl ? (const T *)cl->f : nullptr;
    for (int k = 0; k < 4; k++) a.cl_ynorm[k] = cl ? cl->mlp->ynorm[k] : 0.0f;
    a.h = (const T *)x->h;
    a.pm = (const T *)x->pm;
    a.pn = (const T *)x->pn;
    a.fomn = (const T *)x->fomn;
    a.sustr = (const T *)x->sustr;
    a.svstr = (const T *)x->svstr;
    a.z0 = (const T *)x->zeta[0];
    a.z1 = (const T *)x->zeta[1];
    a.z2 = (T *)x->zeta[2];
    a.u0 = (const T *)x->ubar[0];
    a.u1 = (const T *)x->ubar[1];
    a.u2 = (T *)x->ubar[2];
    a.v0 = (const T *)x->vbar[0];
    a.v1 = (const T *)x->vbar[1];
    a.v2 = (T *)x->vbar[2];
    a.rz0 = (const T *)x->rzeta[0];
    a.rz1 = (T *)x->rzeta[1];
    a.ru0 = (const T *)x->rubar[0];
    a.ru1 = (T *)x->rubar[1];
    a.rv0 = (const T *)x->rvbar[0];
    a.rv1 = (T *)x->rvbar[1];
    a.Zt = x->Zt_avg1;
    a.DUa = x->DU_avg1;
    a.DVa = x->DV_avg1;
    a.szI = x->szI;
    a.szJ = x->szJ;
    a.off_i = (x->szI % TI == 1) ? 1 : 0;
    a.off_j = (x->szJ % TJ == 1) ? 1 : 0;
    a.tiles_i = (x->szI + a.off_i + TI - 1) / TI;
    a.tiles_j = (x->szJ + a.off_j + TJ - 1) / TJ;
    a.g = T(x->g);
    a.rdrg = T(x->rdrg);
    a.dt = T(dt);
    a.first = first;
    a.nts = (double)x->szI * x->szJ * (3.0 * sizeof(T) * 7 + 8.0 * 6) > sf::kStreamingBytes ? 1 : 0;
    a.w1 = w1;
    SF_REQUIRE((long long)x->szI * x->szJ < (1LL << 29), "sf_phys_substep_fused: grid of %dx%d points exceeds 2^29",
               x->szI, x->szJ);
    const long long nb = (long long)a.tiles_i * a.tiles_j;
    SF_REQUIRE(nb < (1LL << 31), "sf_phys_substep_fused: grid too large");
    const dim3 grid((unsigned)nb), block(NT + NR);
    hipStream_t s = sf::as_stream(stream);
    // one launch of the instance <FIRST, streaming>; split tiles run on small grids only and
    // never stream
    auto launch = [&](auto cpl, auto clo, const char *name) {
        constexpr bool CPL = decltype(cpl)::value, CLO = decltype(clo)::value, S = NR == 0;
        if (first && S && a.nts) hipLaunchKernelGGL((k_phys_fused<T, TI, TJ, NT, NR, true, S, CPL, CLO>), grid, block, 0, s, a);
        else if (first) hipLaunchKernelGGL((k_phys_fused<T, TI, TJ, NT, NR, true, false, CPL, CLO>), grid, block, 0, s, a);
        else if (S && a.nts) hipLaunchKernelGGL((k_phys_fused<T, TI, TJ, NT, NR, false, S, CPL, CLO>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_phys_fused<T, TI, TJ, NT, NR, false, false, CPL, CLO>), grid, block, 0, s, a);
        return sf::check_launch(name);
    };
    using Yes = std::true_type;
    using No = std::false_type;
    if (cl) {
        SF_REQUIRE(!cp, "sf_phys_substep_closure_fused: coupling and closure together are not supported");
        if constexpr (NT == 256) return launch(No{}, Yes{}, "sf_phys_substep_closure_fused");
    } else if (cp) {
        if constexpr (NT <= 256) return launch(Yes{}, No{}, "sf_phys_substep_coupled_fused");
    } else {
        if constexpr (NT == 512 || TJ == 4 || NR > 0) return launch(No{}, No{}, "sf_phys_substep_fused");
    }
    sf::set_error("%s: tile height %d (4 or 8)",
                  cp ? "sf_phys_substep_coupled_fused" : "sf_phys_substep_closure_fused", TJ);
    return SF_ERR_ARG;
}

// The tile of a substep that names none (microseconds per substep, graph replays):
//  - grids of at most one 16 x 8 tile per CU: core and ring on different waves, all loads at
//    the start of the tile (128 x 64: FP64 6.4 against 9.1 with 64 x 4 tiles, FP32 5.6 / 7.7);
//  - the same form with 32 x 8 tiles while all of them are resident (by their registers two a
//    CU, FP32 without coupling three) and their number divides by eight, so that they go to
//    the XCDs in bands (xcd_band): FP64 512 x 256 (512 tiles) 11.5 against 11.8 with 64 x 8,
//    but 544 x 256 (544, a second round) 15.3 against 14.3 with 64 x 4; FP32 768 x 256 (768)
//    9.7 against 10.4, 640 x 320 (800) 12.3 against 10.4; coupled FP32 512 x 256 8.9 against
//    10.4 with 64 x 4, 544 x 256 12.5 against 11.1;
//  - without bands they lose earlier: FP64 keeps them up to one a CU (352 x 184, 253 tiles,
//    8.9 against 10.9; 480 x 168, 315, 11.2 against 10.7), FP32 up to two where the tiles they
//    replace have no bands either (544 x 240, 510 tiles, 8.9 against 10.3 with 270 64 x 8;
//    475 x 245, 465, 10.7 against 9.0 with 248; 672 x 248, 651, 12.2 against 11.4; coupled
//    663 x 166, 441, 11.0 against 11.9 with 462 64 x 4; 475 x 245 11.2 against 10.5 with 496);
//  - coupled FP64 gains from them up to 1024 64 x 8 tiles (768 x 384: 25.0 against 28.1), but
//    without bands not past two a CU while 64 x 8 tiles are all resident, two a CU
//    (640 x 184, 460 tiles, 15.1 either way; 640 x 296, 740, 20.9 against 19.2 with 370;
//    832 x 344, 1118, 28.4 against 29.7 with 559).  The closure needs the registers of a whole
//    CU: one tile per CU (343 x 129: 11.0 / 12.6; 512 x 256: 18.4 / 14.5);
//  - else 64 x 8 tiles, or 64 x 4 where one of those a CU leaves none idle and one of these
//    more than fills it: FP64 with more than one 64 x 8 tile per CU and at most three 64 x 4
//    (513 x 255: 14.3 against 16.3; 640 x 272: 14.8 / 16.8; 480 x 248, one per CU: 12.6 / 11.3);
//    coupled FP32 below four 64 x 8 tiles per CU (768 x 384: 15.5 against 16.8); the closure
//    (its 64 x 8 instances exceed two waves per SIMD).
inline PhysTile phys_tile_of(bool f64, bool coupled, bool closure, int szI, int szJ)
{
    constexpr long long CU = sf::kCUs;
    auto tiles = [&](int TI, int TJ) {
        const int oi = szI % TI == 1 ? 1 : 0, oj = szJ % TJ == 1 ? 1 : 0;
        return (long long)((szI + oi + TI - 1) / TI) * ((szJ + oj + TJ - 1) / TJ);
    };
    const bool few8 = tiles(64, 8) < 4 * CU;
    const long long t32 = tiles(32, 8);
    const bool banded = t32 % 8 == 0;
    if (closure) return t32 <= CU ? PhysTile{32, 8} : PhysTile{64, 4};
    if (tiles(16, 8) <= CU) return PhysTile{16, 8};
    const long long alt = tiles(64, coupled ? 4 : 8);   // of FP32, where 32 x 8 are not taken
    bool small;
    if (coupled && f64) small = few8 && (banded || t32 <= 2 * CU || tiles(64, 8) > 2 * CU);
    else if (banded) small = t32 <= (f64 || coupled ? 2 : 3) * CU;
    else small = t32 <= CU || (!f64 && t32 <= 2 * CU && alt % 8 != 0);
    if (small) return PhysTile{32, 8};
    if (coupled) return PhysTile{64, !f64 && few8 ? 4 : 8};
    return PhysTile{64, f64 && tiles(64, 8) > CU && tiles(64, 4) <= 3 * CU ? 4 : 8};
}

// Tile height tj: 4, 8 or 16 (64-wide tiles), or 0 for phys_tile_of's choice.
template <typename T>
int dispatch_tj(const sf_phys_fields *x, double dt, int first, double w1, int tj, void *stream,
                const sf_couple_fields *cp = nullptr, const ClosureIn *cl = nullptr)
{
    if (tj == 0) {
        const PhysTile t = phys_tile_of(sizeof(T) == 8, cp, cl, x->szI, x->szJ);
        if (t.ti == 16) return launch_fused<T, 16, 8, 128, 192>(x, dt, first, w1, stream, cp);
        if (t.ti == 32) return launch_fused<T, 32, 8, 256, 256>(x, dt, first, w1, stream, cp, cl);
        tj = t.tj;
    }
    switch (tj) {
    case 4: return launch_fused<T, 64, 4, 256>(x, dt, first, w1, stream, cp, cl);
    case 8:
        // 512 threads: one core point per thread; the coupled and closure instances need too
        // many registers for that
        if (cp || cl) return launch_fused<T, 64, 8, 256>(x, dt, first, w1, stream, cp, cl);
        return launch_fused<T, 64, 8, 512>(x, dt, first, w1, stream);
    case 16: return launch_fused<T, 64, 16, 512>(x, dt, first, w1, stream, cp, cl);
    default: break;
    }
    sf::set_error("sf_phys_substep_fused: unsupported tile height %d (4, 8 or 16)", tj);
    return SF_ERR_ARG;
}


// ---------------------------------------------------------------------------------
// Ensembles: many basins of uneven size advance in ONE launch per substep.  The
// launch walks a device-side list of (member, tile) pairs; each workgroup takes
// tiles from the list in one of two orders and runs the same per-tile function as
// the single-grid kernel, so a member's result equals its solo run bit for bit.
// ---------------------------------------------------------------------------------
// The member table holds, for every member, its kernel arguments for each of the
// three time rotations (index 3*member + rot): no runtime indexing of slot pointers
// inside the kernel.
// order 0: block b takes list entries b, b + G, b + 2G, ...
// order 1: block b (after the XCD band remap) takes a contiguous chunk of the list
template <typename T, int TI, int TJ, int NT, bool FIRST, bool NTS>
__global__ __launch_bounds__(NT) void k_phys_ensemble(const PFA<T> *__restrict__ members,
                                                      const int2 *__restrict__ list, int ntiles, int order,
                                                      int rot, double w1)
{
    using Lds = PhysLds<T, TI, TJ, NT, 0, NTS, false, false>;
    __shared__ T sm[Lds::PLANES][Lds::FN];
    __shared__ T rzl[TI + TJ + 1];
    const int G = gridDim.x;
    int t0, t1, step;
    if (order == 0) {
        t0 = blockIdx.x;
        t1 = ntiles;
        step = G;
    } else {
        const int b = xcd_band(G);
        t0 = (int)((long long)ntiles * b / G);
        t1 = (int)((long long)ntiles * (b + 1) / G);
        step = 1;
    }
    // the tables are read-only for the whole launch: scalar loads through the constant
    // address space keep every member pointer in scalar registers
    const SF_CONST int *clist = (const SF_CONST int *)list;
    const SF_CONST PFA<T> *cmem = (const SF_CONST PFA<T> *)members;
    for (int t = t0; t < t1; t += step) {
        const int ex = clist[2 * t], ey = clist[2 * t + 1];
        PFA<T> P;
        {
            static_assert(sizeof(PFA<T>) % 4 == 0, "argument block of whole words");
            const SF_CONST uint32_t *src = (const SF_CONST uint32_t *)(cmem + 3 * ex + rot);
            uint32_t *dst = reinterpret_cast<uint32_t *>(&P);
#pragma unroll
            for (int w = 0; w < (int)(sizeof(PFA<T>) / 4); w++) dst[w] = src[w];
        }
        P.w1 = w1;
        phys_tile<T, TI, TJ, NT, 0, ROLE_ALL, FIRST, NTS>(P, ey % P.tiles_i, ey / P.tiles_i, sm, rzl);
        lds_barrier();   // the next tile overwrites the LDS planes
    }
}

// One workgroup per list entry (grid = number of tiles): no tile loop, so the tile
// code is register-allocated as in the single-basin kernel.  order 0 takes entry b,
// order 1 the XCD-banded entry of block b.
template <typename T, int TI, int TJ, int NT, bool FIRST, bool NTS>
__global__ __launch_bounds__(NT) void k_phys_ensemble1(const PFA<T> *__restrict__ members,
                                                       const int2 *__restrict__ list, int order, int rot,
                                                       double w1)
{
    using Lds = PhysLds<T, TI, TJ, NT, 0, NTS, false, false>;
    __shared__ T sm[Lds::PLANES][Lds::FN];
    __shared__ T rzl[TI + TJ + 1];
    const int t = order == 0 ? (int)blockIdx.x : xcd_band(gridDim.x);
    const SF_CONST int *clist = (const SF_CONST int *)list;
    const SF_CONST PFA<T> *cmem = (const SF_CONST PFA<T> *)members;
    const int ex = clist[2 * t], ey = clist[2 * t + 1];
    PFA<T> P;
    {
        const SF_CONST uint32_t *src = (const SF_CONST uint32_t *)(cmem + 3 * ex + rot);
        uint32_t *dst = reinterpret_cast<uint32_t *>(&P);
#pragma unroll
        for (int w = 0; w < (int)(sizeof(PFA<T>) / 4); w++) dst[w] = src[w];
    }
    P.w1 = w1;
    phys_tile<T, TI, TJ, NT, 0, ROLE_ALL, FIRST, NTS>(P, ey % P.tiles_i, ey / P.tiles_i, sm, rzl);
}
}  // namespace


// ---------------------------------------------------------------------------------
// Ensemble C ABI
// ---------------------------------------------------------------------------------
struct sf_ens {
    int n, precision, device;
    int tile_j, order, grid;
    int ntiles, rot;
    int nts;                    // streaming stores (see PFA::nts), set by ens_build
    void *members;              // device PFA<T>[3 n]: arguments of member k for rotation r at 3k + r
    int2 *list;                 // device (member, tile) list for tile_j
    std::vector<sf_phys_fields> host;
    std::vector<double> dt;
    hipGraph_t graph;
    hipGraphExec_t exec;
    int graph_nsub;
};

namespace {

template <int TJ>
int ens_tiles(const sf_phys_fields &x, int &ti, int &tj, int &oi, int &oj)
{
    constexpr int TI = 64;
    oi = (x.szI % TI == 1) ? 1 : 0;
    oj = (x.szJ % TJ == 1) ? 1 : 0;
    ti = (x.szI + oi + TI - 1) / TI;
    tj = (x.szJ + oj + TJ - 1) / TJ;
    return ti * tj;
}

template <typename T>
int ens_build(sf_ens *e)
{
    std::vector<PFA<T>> hm(3 * e->n);
    std::vector<int2> list;
    double bytes = 0.0;   // one substep of the whole ensemble (see PFA::nts)
    for (int k = 0; k < e->n; k++)
        bytes += (double)e->host[k].szI * e->host[k].szJ * (3.0 * sizeof(T) * 7 + 8.0 * 6);
    const int nts = bytes > sf::kStreamingBytes ? 1 : 0;
    e->nts = nts;
    for (int k = 0; k < e->n; k++) {
        const sf_phys_fields &x = e->host[k];
        int ti = 0, tj = 0, oi = 0, oj = 0, nt = 0;
        switch (e->tile_j) {
        case 4: nt = ens_tiles<4>(x, ti, tj, oi, oj); break;
        case 8: nt = ens_tiles<8>(x, ti, tj, oi, oj); break;
        default: nt = ens_tiles<16>(x, ti, tj, oi, oj); break;
        }
        for (int rot = 0; rot < 3; rot++) {
            // level t_l lives in slot (l + rot) % 3
            const int s0 = rot % 3, s1 = (rot + 1) % 3, s2 = (rot + 2) % 3;
            PFA<T> &a = hm[3 * k + rot];
            a.h = (const T *)x.h;
            a.pm = (const T *)x.pm;
            a.pn = (const T *)x.pn;
            a.fomn = (const T *)x.fomn;
            a.sustr = (const T *)x.sustr;
            a.svstr = (const T *)x.svstr;
            a.z0 = (const T *)x.zeta[s0];
            a.z1 = (const T *)x.zeta[s1];
            a.z2 = (T *)x.zeta[s2];
            a.u0 = (const T *)x.ubar[s0];
            a.u1 = (const T *)x.ubar[s1];
            a.u2 = (T *)x.ubar[s2];
            a.v0 = (const T *)x.vbar[s0];
            a.v1 = (const T *)x.vbar[s1];
            a.v2 = (T *)x.vbar[s2];
            a.rz0 = (const T *)x.rzeta[s0];
            a.rz1 = (T *)x.rzeta[s1];
            a.ru0 = (const T *)x.rubar[s0];
            a.ru1 = (T *)x.rubar[s1];
            a.rv0 = (const T *)x.rvbar[s0];
            a.rv1 = (T *)x.rvbar[s1];
            a.Zt = x.Zt_avg1;
            a.DUa = x.DU_avg1;
            a.DVa = x.DV_avg1;
            a.szI = x.szI;
            a.szJ = x.szJ;
            a.tiles_i = ti;
            a.tiles_j = tj;
            a.off_i = oi;
            a.off_j = oj;
            a.g = T(x.g);
            a.rdrg = T(x.rdrg);
            a.dt = T(e->dt[k]);
            a.first = 0;
            a.nts = nts;
            a.w1 = 0.0;
        }
        for (int t = 0; t < nt; t++) list.push_back(make_int2(k, t));
    }
    e->ntiles = (int)list.size();
    hipError_t r = hipFree(e->members);
    if (r == hipSuccess) r = hipFree(e->list);
    e->members = nullptr;
    e->list = nullptr;
    if (r == hipSuccess) r = hipMalloc(&e->members, sizeof(PFA<T>) * hm.size());
    if (r == hipSuccess) r = hipMalloc((void **)&e->list, sizeof(int2) * list.size());
    if (r == hipSuccess) r = hipMemcpy(e->members, hm.data(), sizeof(PFA<T>) * hm.size(), hipMemcpyHostToDevice);
    if (r == hipSuccess) r = hipMemcpy(e->list, list.data(), sizeof(int2) * list.size(), hipMemcpyHostToDevice);
    if (r != hipSuccess) return sf::hip_fail(r, "sf_ens: device tables");
    return SF_OK;
}

template <typename T, int TJ>
void ens_launch_tj(sf_ens *e, int first, double w1, int rot, hipStream_t s)
{
    constexpr int TI = 64, NT = TJ == 4 ? 256 : 512;
    const int G = e->grid > 0 ? (e->grid < e->ntiles ? e->grid : e->ntiles) : e->ntiles;
    const PFA<T> *m = (const PFA<T> *)e->members;
    if (G == e->ntiles) {   // one workgroup per tile
        if (first && e->nts)
            hipLaunchKernelGGL((k_phys_ensemble1<T, TI, TJ, NT, true, true>), dim3(G), dim3(NT), 0, s, m, e->list,
                               e->order, rot, w1);
        else if (first)
            hipLaunchKernelGGL((k_phys_ensemble1<T, TI, TJ, NT, true, false>), dim3(G), dim3(NT), 0, s, m, e->list,
                               e->order, rot, w1);
        else if (e->nts)
            hipLaunchKernelGGL((k_phys_ensemble1<T, TI, TJ, NT, false, true>), dim3(G), dim3(NT), 0, s, m, e->list,
                               e->order, rot, w1);
        else
            hipLaunchKernelGGL((k_phys_ensemble1<T, TI, TJ, NT, false, false>), dim3(G), dim3(NT), 0, s, m,
                               e->list, e->order, rot, w1);
        return;
    }
    // The tile loop's own registers take FP64's one-point-a-thread form (512 threads) past 128:
    // one workgroup a CU where two of 256 threads fit.  21 basins of 256 x 128 to 1024 x 512, a
    // grid of 512: 5.76 ms for twelve substeps with 512 threads, 4.51 with 256.
    constexpr int NP = sizeof(T) == 8 && TJ == 8 ? 256 : NT;
    if (first && e->nts)
        hipLaunchKernelGGL((k_phys_ensemble<T, TI, TJ, NP, true, true>), dim3(G), dim3(NP), 0, s, m, e->list,
                           e->ntiles, e->order, rot, w1);
    else if (first)
        hipLaunchKernelGGL((k_phys_ensemble<T, TI, TJ, NP, true, false>), dim3(G), dim3(NP), 0, s, m, e->list,
                           e->ntiles, e->order, rot, w1);
    else if (e->nts)
        hipLaunchKernelGGL((k_phys_ensemble<T, TI, TJ, NP, false, true>), dim3(G), dim3(NP), 0, s, m, e->list,
                           e->ntiles, e->order, rot, w1);
    else
        hipLaunchKernelGGL((k_phys_ensemble<T, TI, TJ, NP, false, false>), dim3(G), dim3(NP), 0, s, m, e->list,
                           e->ntiles, e->order, rot, w1);
}

template <typename T>
void ens_launch(sf_ens *e, int first, double w1, int rot, hipStream_t s)
{
    switch (e->tile_j) {
    case 4: ens_launch_tj<T, 4>(e, first, w1, rot, s); break;
    case 8: ens_launch_tj<T, 8>(e, first, w1, rot, s); break;
    default: ens_launch_tj<T, 16>(e, first, w1, rot, s); break;
    }
}

}  // namespace

// FP32 instances, compiled in phys2d_fused_f32.hip with contraction on
int sf_phys_fused_dispatch_f32(const sf_phys_fields *x, double dt, int first, double w1, int tj, void *stream,
                               const sf_couple_fields *cp = nullptr, const ClosureIn *cl = nullptr);
void sf_ens_launch_f32(sf_ens *e, int first, double w1, int rot, hipStream_t s);
