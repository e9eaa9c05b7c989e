// baroclinic.hip -- the baroclinic terms the reference names but leaves out: the linear
// equation of state (utility/test.in:2130-2160), the baroclinic pressure gradient
// (nonlinear/rhs.py:31-32, "prsgrd()" commented out) and the tracer step
// (nonlinear/step3d_t.py, Fortran text).  One thread per water column (pressure
// gradient, tracer) or per cell (state equation); flat layout of the 3D kernels (level
// stride S2 = szI*szJ, xi fastest).  FP64 instances follow the oracle
// (oracle/sf_oracle3d.c) operation by operation; FP32 bulk instances read and write FP32
// fields and form each column's pressure-gradient and volume-flux sums in FP64.
#include "sf_internal.h"

namespace {

struct Col {
    int szI, szJ, N;
    long long S2;
    const double *pm, *pn;
    bool band;   // columns in XCD bands (sf::column_block)
};

// elem: bytes of a 3D field's element
inline Col col_of(const sf_ctx *c, size_t elem)
{
    const bool band = (c->szK + 1.0) * (double)c->S2 * (double)elem <= sf::kBandBytes;
    return Col{c->szI, c->szJ, c->szK, c->S2, c->pm, c->pn, band};
}

// ---- linear equation of state: rho = ((R0 - 1000) - R0 Tcoef (T - T0)) + R0 Scoef (S - S0)
template <class T>
__global__ __launch_bounds__(256) void k_rho_eos(long long n, const T *t, const T *s, double a, double bt,
                                                 double bs, double T0, double S0, T *rho)
{
    const long long b = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= n) return;
    rho[b] = T((a - bt * ((double)t[b] - T0)) + bs * ((double)s[b] - S0));
}

// ---- baroclinic pressure gradient, standard density Jacobian (Song 1998), added to ru/rv.
// Per interior u (v) column with neighbour p = f-1 (f-szI), from the top level down:
//   phi(N-1) = fac1 drho (dz_top + dz_top_p) + (fac2 + fac1 (rho + rho_p)) (z_w(N) - z_w_p(N))
//   phi(k)   = phi(k+1) + fac3 (C1 C3 - C2 C4)       (gamma-weighted Jacobian of rho and z_r)
//   r(k)    += (-0.5 (Hz + Hz_p) phi(k)) * (2 / (pn + pn_p))      [v: 2 / (pm + pm_p)]
// The difference phi(k) - phi(k+1) from rho (r) and z_r (z) at the column f and its
// neighbour p, levels k (0) and k + 1 (1).
__device__ __forceinline__ double pgf_diff(double r0f, double r1f, double r0p, double r1p, double z0f, double z1f,
                                           double z0p, double z1p, double fac3)
{
    const double dzf = z1f - z0f, dzp = z1p - z0p;
    const double a2 = (z0f - z0p) + (z1f - z1p);
    const double a3 = dzf - dzp;
    const double gam = ((0.125 * a2) * a3) / (dzf * dzp);
    const double C1 = (1.0 + gam) * (r1f - r1p) + (1.0 - gam) * (r0f - r0p);
    const double C2 = (r1f + r1p) - (r0f + r0p);
    const double C3 = (z1f + z1p) - (z0f + z0p);
    const double C4 = (1.0 + gam) * (z1f - z1p) + (1.0 - gam) * (z0f - z0p);
    return fac3 * (C1 * C3 - C2 * C4);
}

// A block is 256 / NW columns by NW level waves (NW by sf::level_waves).  Per round, from the
// top, each wave takes LB levels of both directions: their loads go out together, the
// differences of phi meet in LDS, and every wave runs the columns' sums over the round (one
// level wave: from its registers).  Against a thread that walked its column twice, once per
// direction: FP32 1024 x 512 x 32 (seven fields, 470 MB, without the density's 23 us) 167 ->
// 148 us (the FP64 differences take about 60 us of that), 386 x 258 x 40 48 -> 36, 90 x 60 x 20
// 19 -> 8, 3000 x 1500 x 4 (one level wave) 180 -> 165; FP64 1024 x 512 x 32 310 -> 250.
template <class T, int LB, int NW>
__global__ __launch_bounds__(256) void k_prsgrd(Col g, const T *rho, const T *z_r, const T *z_w, const T *Hz,
                                                double grav, double rho0, T *ru, T *rv)
{
    constexpr int ROUND = NW * LB, COLS = 256 / NW;
    __shared__ double sP[2][2][ROUND][NW > 1 ? COLS : 1];   // by buffer, direction, level of the round, column
    const int col = threadIdx.x % COLS;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / COLS);
    const long long f = (long long)sf::column_block(g.band) * COLS + col;
    const long long S2 = g.S2, W = g.szI;
    const int N = g.N, i = (int)(f % W), j = (int)(f / W), L = g.szI - 1, M = g.szJ - 1;
    const bool un = f < S2 && i >= 2 && i <= L - 1 && j >= 1 && j <= M - 1;
    const bool vn = f < S2 && j >= 2 && j <= M - 1 && i >= 1 && i <= L - 1;
    const bool on = un || vn;   // i, j >= 1: both neighbours exist
    const double fac1 = 0.5 * grav / rho0, fac2 = 1000.0 * grav / rho0, fac3 = 0.25 * grav / rho0;
    double metu = 0.0, metv = 0.0, phiu = 0.0, phiv = 0.0;
    if (on) {
        metu = 2.0 / (g.pn[f - 1] + g.pn[f]);
        metv = 2.0 / (g.pm[f - W] + g.pm[f]);
        const long long t = (long long)(N - 1) * S2 + f;
        const double r = rho[t], ru_ = rho[t - 1], rv_ = rho[t - W];
        const double z = z_r[t], zu = z_r[t - 1], zv = z_r[t - W];
        const double w = z_w[t + S2], wu = z_w[t + S2 - 1], wv = z_w[t + S2 - W];
        phiu = (fac1 * (r - ru_)) * ((w - z) + (wu - zu));
        phiu = phiu + (fac2 + fac1 * (r + ru_)) * (w - wu);
        phiv = (fac1 * (r - rv_)) * ((w - z) + (wv - zv));
        phiv = phiv + (fac2 + fac1 * (r + rv_)) * (w - wv);
        if (wave == 0) {   // the top level itself
            if (un) ru[t] = T((double)ru[t] + ((-0.5 * ((double)Hz[t] + (double)Hz[t - 1])) * phiu) * metu);
            if (vn) rv[t] = T((double)rv[t] + ((-0.5 * ((double)Hz[t] + (double)Hz[t - W])) * phiv) * metv);
        }
    }
    // a round: levels top, top - 1, ...; the wave's are hi, hi - 1, ... (LB of them)
    for (int top = N - 2, buf = 0; top >= 0; top -= ROUND, buf ^= 1) {
        const int hi = top - wave * LB;
        const bool mine = on && hi >= 0;   // the last round may end above the wave
        auto level = [&](int k) { return (long long)(k < 0 ? 0 : k) * S2 + f; };
        T hz[LB], hu[LB], hv[LB], xu[LB], xv[LB];
        double pu[LB], pv[LB];
        if (mine) {
            T r[LB + 1], rw[LB + 1], rs[LB + 1], z[LB + 1], zw[LB + 1], zs[LB + 1];
#pragma unroll
            for (int q = 0; q <= LB; q++) {
                const long long b = level(hi + 1 - q);
                r[q] = rho[b];
                rw[q] = rho[b - 1];
                rs[q] = rho[b - W];
                z[q] = z_r[b];
                zw[q] = z_r[b - 1];
                zs[q] = z_r[b - W];
            }
#pragma unroll
            for (int q = 0; q < LB; q++) {
                const long long b = level(hi - q);
                hz[q] = Hz[b];
                hu[q] = Hz[b - 1];
                hv[q] = Hz[b - W];
                xu[q] = ru[b];
                xv[q] = rv[b];
            }
#pragma unroll
            for (int q = 0; q < LB; q++) {
                pu[q] = pgf_diff(r[q + 1], r[q], rw[q + 1], rw[q], z[q + 1], z[q], zw[q + 1], zw[q], fac3);
                pv[q] = pgf_diff(r[q + 1], r[q], rs[q + 1], rs[q], z[q + 1], z[q], zs[q + 1], zs[q], fac3);
                if constexpr (NW > 1) {
                    sP[buf][0][wave * LB + q][col] = pu[q];
                    sP[buf][1][wave * LB + q][col] = pv[q];
                }
            }
        }
        if constexpr (NW > 1) __syncthreads();   // the next round fills the other buffer
        if (!mine) continue;
        if constexpr (NW > 1) {
#pragma unroll
            for (int m = 0; m < ROUND; m++) {
                phiu = phiu + sP[buf][0][m][col];
                phiv = phiv + sP[buf][1][m][col];
#pragma unroll
                for (int q = 0; q < LB; q++)
                    if (m == wave * LB + q) {
                        pu[q] = phiu;
                        pv[q] = phiv;
                    }
            }
        } else {
#pragma unroll
            for (int q = 0; q < LB; q++) {
                phiu = phiu + pu[q];
                phiv = phiv + pv[q];
                pu[q] = phiu;
                pv[q] = phiv;
            }
        }
#pragma unroll
        for (int q = 0; q < LB; q++) {
            if (hi - q < 0) break;
            const long long b = level(hi - q);
            if (un) ru[b] = T((double)xu[q] + ((-0.5 * ((double)hz[q] + (double)hu[q])) * pu[q]) * metu);
            if (vn) rv[b] = T((double)xv[q] + ((-0.5 * ((double)hz[q] + (double)hv[q])) * pv[q]) * metv);
        }
    }
}

// ---- tracer step: flux form, first-order upstream faces, forward in time, with the
// vertical volume flux of each cell's top formed from the horizontal volume fluxes and
// the thickness change (a uniform tracer stays uniform).  Interior columns; the thread of
// a column next to the boundary also writes its ghost columns (zero gradient).
// A block is 64 columns by four waves.  Per round each wave takes LB levels: their loads
// go out together, the divergences and thickness changes meet in LDS, and every wave runs
// the column's sum W over the round.  The NTR tracers share the fluxes and thicknesses.
// Two tracers with the copy back to the old arrays, against a launch per tracer that walked
// its columns and two ghost launches each: FP32 1024 x 512 x 32 (eight fields, 537 MB, and
// 268 MB copied) 318 -> 212 us, 386 x 258 x 40 171 -> 51, 90 x 60 x 20 68 -> 14; FP64
// 386 x 258 x 40 158 -> 88.  Two levels a wave hold 104 (FP32) or 126 VGPRs, four 159 or 211.
template <class T>
struct Tracers2 {
    const T *t[2];
    T *tn[2];
};

template <class T, int NTR, int LB>
__global__ __launch_bounds__(256) void k_step3d_t(Col g, Tracers2<T> x, const T *Huon, const T *Hvom,
                                                  const T *Hz_old, const T *Hz_new, double dt)
{
    constexpr int NW = 4, ROUND = NW * LB;
    __shared__ double sD[2][ROUND][64], sC[2][ROUND][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long f = (long long)sf::column_block(g.band) * 64 + lane;
    const long long S2 = g.S2, W = g.szI;
    const int N = g.N, i = (int)(f % W), j = (int)(f / W), L = g.szI - 1, M = g.szJ - 1;
    const bool on = f < S2 && i >= 1 && i <= L - 1 && j >= 1 && j <= M - 1;
    const bool edge = on && (i == 1 || i == L - 1 || j == 1 || j == M - 1);
    const double mn = on ? g.pm[f] * g.pn[f] : 0.0;
    double Wlow = 0.0;   // W below the round
    for (int k0 = 0, buf = 0; k0 < N; k0 += ROUND, buf ^= 1) {
        const int lo = k0 + wave * LB;
        auto level = [&](int k) { return (long long)(k < 0 ? 0 : (k < N ? k : N - 1)) * S2 + f; };
        T hu0[LB], hu1[LB], hv0[LB], hv1[LB], hzo[LB], hzn[LB];
        T c[NTR][LB + 2], e[NTR][LB], w[NTR][LB], n[NTR][LB], s[NTR][LB];
        const bool mine = on && lo < N;   // the last round may end below the wave
        if (mine) {
#pragma unroll
            for (int q = 0; q < LB; q++) {
                const long long b = level(lo + q);
                hu0[q] = Huon[b];
                hu1[q] = Huon[b + 1];
                hv0[q] = Hvom[b];
                hv1[q] = Hvom[b + W];
                hzo[q] = Hz_old[b];
                hzn[q] = Hz_new[b];
            }
#pragma unroll
            for (int m = 0; m < NTR; m++) {
#pragma unroll
                for (int q = 0; q < LB + 2; q++) c[m][q] = x.t[m][level(lo + q - 1)];
#pragma unroll
                for (int q = 0; q < LB; q++) {
                    const long long b = level(lo + q);
                    w[m][q] = x.t[m][b - 1];
                    e[m][q] = x.t[m][b + 1];
                    s[m][q] = x.t[m][b - W];
                    n[m][q] = x.t[m][b + W];
                }
            }
#pragma unroll
            for (int q = 0; q < LB; q++) {
                sD[buf][wave * LB + q][lane] =
                    mn * (((double)hu1[q] - (double)hu0[q]) + ((double)hv1[q] - (double)hv0[q]));
                sC[buf][wave * LB + q][lane] = ((double)hzn[q] - (double)hzo[q]) / dt;
            }
        }
        __syncthreads();   // the next round fills the other buffer
        if (!mine) continue;
        double Wk[LB + 1], Wr = Wlow;   // W at the tops of levels lo-1 .. lo+LB-1
        Wk[0] = Wlow;
#pragma unroll
        for (int r = 0; r < ROUND; r++) {
            Wr = (Wr - sD[buf][r][lane]) - sC[buf][r][lane];
            if (r == wave * LB - 1) Wk[0] = Wr;
#pragma unroll
            for (int q = 0; q < LB; q++)
                if (r == wave * LB + q) Wk[q + 1] = Wr;
        }
        Wlow = Wr;
#pragma unroll
        for (int m = 0; m < NTR; m++) {
            T *tn = x.tn[m];
            double FClow = lo > 0 ? Wk[0] * (Wk[0] > 0.0 ? (double)c[m][0] : (double)c[m][1]) : 0.0;
#pragma unroll
            for (int q = 0; q < LB; q++) {
                if (lo + q >= N) break;
                const double u0 = hu0[q], u1 = hu1[q], v0 = hv0[q], v1 = hv1[q], zo = hzo[q], zn = hzn[q];
                const double tc = c[m][q + 1];
                const double FX0 = u0 * (u0 > 0.0 ? (double)w[m][q] : tc);
                const double FX1 = u1 * (u1 > 0.0 ? tc : (double)e[m][q]);
                const double FE0 = v0 * (v0 > 0.0 ? (double)s[m][q] : tc);
                const double FE1 = v1 * (v1 > 0.0 ? tc : (double)n[m][q]);
                const double FCk =
                    lo + q < N - 1 ? Wk[q + 1] * (Wk[q + 1] > 0.0 ? tc : (double)c[m][q + 2]) : Wk[q + 1] * tc;
                const double div = mn * ((FX1 - FX0) + (FE1 - FE0)) + (FCk - FClow);
                const T r = T((zo * tc - dt * div) / zn);
                FClow = FCk;
                const long long b = (long long)(lo + q) * S2 + f;
                tn[b] = r;
                if (edge) {
                    const long long row = j == 1 ? -W : (j == M - 1 ? W : 0), row2 = j == 1 && j == M - 1 ? W : row;
                    const bool west = i == 1, east = i == L - 1;
                    if (west) tn[b - 1] = r;
                    if (east) tn[b + 1] = r;
                    if (row != 0) {
                        tn[b + row] = r;
                        if (west) tn[b + row - 1] = r;
                        if (east) tn[b + row + 1] = r;
                    }
                    if (row2 != row) {   // a single interior row
                        tn[b + row2] = r;
                        if (west) tn[b + row2 - 1] = r;
                        if (east) tn[b + row2 + 1] = r;
                    }
                }
            }
        }
    }
}

template <class T>
int eos_launch(sf_ctx *c, const void *t, const void *s, double R0, double T0, double S0, double Tcoef,
               double Scoef, void *rho, void *stream)
{
    const long long n = (long long)c->szK * c->S2;
    hipLaunchKernelGGL(k_rho_eos<T>, dim3(sf::grid1d(n)), dim3(256), 0, sf::as_stream(stream), n, (const T *)t,
                       (const T *)s, R0 - 1000.0, R0 * Tcoef, R0 * Scoef, T0, S0, (T *)rho);
    return sf::check_launch("sf_rho_eos");
}

template <class T>
int prsgrd_launch(sf_ctx *c, const void *rho, const void *z_r, const void *z_w, const void *Hz, double g,
                  double rho0, void *ru, void *rv, void *stream)
{
    auto go = [&](auto kernel, int cols) {
        hipLaunchKernelGGL(kernel, sf::wide_grid(sf::column_grid(c->S2, cols), 256), dim3(256), 0, sf::as_stream(stream),
                           col_of(c, sizeof(T)), (const T *)rho, (const T *)z_r, (const T *)z_w, (const T *)Hz, g, rho0,
                           (T *)ru, (T *)rv);
    };
    if (sf::level_waves(c, 16) == 4) go(k_prsgrd<T, 2, 4>, 64);
    else go(k_prsgrd<T, 2, 1>, 256);
    return sf::check_launch("sf_prsgrd");
}

template <class T>
int tracer_launch(sf_ctx *c, int ntr, const void *const *t, void *const *tn, const void *Huon, const void *Hvom,
                  const void *Hz_old, const void *Hz_new, double dt, void *stream)
{
    constexpr int LB = 2;
    Tracers2<T> x{};
    for (int m = 0; m < ntr; m++) {
        x.t[m] = (const T *)t[m];
        x.tn[m] = (T *)tn[m];
    }
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, sf::wide_grid(sf::column_grid(c->S2, 64), 256), dim3(256), 0, sf::as_stream(stream),
                           col_of(c, sizeof(T)), x, (const T *)Huon, (const T *)Hvom, (const T *)Hz_old,
                           (const T *)Hz_new, dt);
    };
    if (ntr == 2) go(k_step3d_t<T, 2, LB>);
    else go(k_step3d_t<T, 1, LB>);
    return sf::check_launch("sf_step3d_t");
}

int tracer_step(sf_ctx *c, int32_t precision, int ntr, const void *const *t, void *const *tn, const void *Huon,
                const void *Hvom, const void *Hz_old, const void *Hz_new, double dt, void *stream)
{
    SF_REQUIRE(c && Huon && Hvom && Hz_old && Hz_new, "sf_step3d_t: null argument");
    for (int m = 0; m < ntr; m++) {
        SF_REQUIRE(t[m] && tn[m], "sf_step3d_t: null argument");
        for (int k = 0; k < ntr; k++)
            SF_REQUIRE(t[k] != tn[m] && (k == m || tn[k] != tn[m]),
                       "sf_step3d_t: the new tracer must not alias the old one");
    }
    SF_REQUIRE(dt > 0.0, "sf_step3d_t: dt=%g", dt);
    if (precision == SF_FP64) return tracer_launch<double>(c, ntr, t, tn, Huon, Hvom, Hz_old, Hz_new, dt, stream);
    if (precision == SF_FP32) return tracer_launch<float>(c, ntr, t, tn, Huon, Hvom, Hz_old, Hz_new, dt, stream);
    sf::set_error("sf_step3d_t: unknown precision %d", precision);
    return SF_ERR_ARG;
}

}  // namespace

extern "C" int sf_rho_eos(sf_ctx *c, int32_t precision, const void *t, const void *s, double R0, double T0,
                          double S0, double Tcoef, double Scoef, void *rho, void *stream)
{
    SF_REQUIRE(c && t && s && rho, "sf_rho_eos: null argument");
    if (precision == SF_FP64) return eos_launch<double>(c, t, s, R0, T0, S0, Tcoef, Scoef, rho, stream);
    if (precision == SF_FP32) return eos_launch<float>(c, t, s, R0, T0, S0, Tcoef, Scoef, rho, stream);
    sf::set_error("sf_rho_eos: unknown precision %d", precision);
    return SF_ERR_ARG;
}

extern "C" int sf_prsgrd(sf_ctx *c, int32_t precision, const void *rho, const void *z_r, const void *z_w,
                         const void *Hz, double g, double rho0, void *ru, void *rv, void *stream)
{
    SF_REQUIRE(c && rho && z_r && z_w && Hz && ru && rv, "sf_prsgrd: null argument");
    SF_REQUIRE(c->szK >= 2, "sf_prsgrd: needs at least 2 levels (N=%d)", c->szK);
    if (precision == SF_FP64) return prsgrd_launch<double>(c, rho, z_r, z_w, Hz, g, rho0, ru, rv, stream);
    if (precision == SF_FP32) return prsgrd_launch<float>(c, rho, z_r, z_w, Hz, g, rho0, ru, rv, stream);
    sf::set_error("sf_prsgrd: unknown precision %d", precision);
    return SF_ERR_ARG;
}

extern "C" int sf_step3d_t(sf_ctx *c, int32_t precision, const void *t, void *tn, const void *Huon,
                           const void *Hvom, const void *Hz_old, const void *Hz_new, double dt, void *stream)
{
    return tracer_step(c, precision, 1, &t, &tn, Huon, Hvom, Hz_old, Hz_new, dt, stream);
}

extern "C" int sf_step3d_ts(sf_ctx *c, int32_t precision, const void *t, void *tn, const void *s, void *sn,
                            const void *Huon, const void *Hvom, const void *Hz_old, const void *Hz_new, double dt,
                            void *stream)
{
    const void *const old[2] = {t, s};
    void *const now[2] = {tn, sn};
    return tracer_step(c, precision, 2, old, now, Huon, Hvom, Hz_old, Hz_new, dt, stream);
}
