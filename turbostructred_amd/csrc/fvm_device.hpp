// fvm_device.hpp -- device-side physics of the explicit finite-volume step (gfx950).
//
// Point-wise pieces used by the fused stage kernels: boundary images, cell reconstruction and
// the Riemann fluxes, templated on the arithmetic type R (double, or float for the
// FP32-residual form).  Each function cites the reference routine whose result it reproduces;
// the arithmetic is written for CDNA (fused multiply-add, reciprocal instead of division where
// the result stays within a few ulp), not transcribed.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tsd {

constexpr int NV = 5;

// A flow without momentum out of the grid's axes (a 1-D tube, a plane 2-D flow) keeps those
// momenta at exactly zero: no flux, limiter or boundary image makes any.  The kernels are
// templated on the number N of variables they carry (density, the first N - 2 momenta,
// energy): N = 3 in 1-D and N = 4 in 2-D when the state and the boundary conditions have none, and
// N = 5 otherwise.  The other variables' arithmetic is the same operation for operation.
template <int N>
__device__ __host__ constexpr int plane_of(int v) { return v == N - 1 ? NV - 1 : v; }

// Sums over the components are written with explicit fused operations: left to itself the compiler chooses
// which products of a sum it fuses, and chose differently for three components than for two.
__device__ inline double madd(double a, double b, double s) { return __builtin_fma(a, b, s); }
__device__ inline float madd(float a, float b, float s) { return __builtin_fmaf(a, b, s); }
template <typename R, int M>
__device__ __forceinline__ R dot(const R (&a)[M], const R (&b)[M]) {
#pragma clang fp contract(off)
    R s = a[0] * b[0];
#pragma unroll
    for (int i = 1; i < M; i++) s = madd(a[i], b[i], s);
    return s;
}
// |momentum|^2
template <typename R, int N>
__device__ __forceinline__ R momentum2(const R (&u)[N]) {
#pragma clang fp contract(off)
    R s = u[1] * u[1];
#pragma unroll
    for (int i = 2; i < N - 1; i++) s = madd(u[i], u[i], s);
    return s;
}

// ---- boundary conditions -------------------------------------------------------------------
// Values of BoundaryConditionType (src/BoundaryConditions/BoundaryConditionConfiguration.h:12-19)
enum : int { BC_WALL = 0, BC_SYMMETRY = 1, BC_MOVING_WALL = 2, BC_SUBSONIC_INLET = 3,
             BC_SUBSONIC_OUTLET = 4, BC_NATURAL = 5 };

struct BCDev {
    int type;
    double vel[3];
    double p;
    double rho;
};

// ---- fast reciprocal / square root ---------------------------------------------------------
// Hardware estimates (good to about 2^-23 in double) refined by the shortest chain that reaches
// working precision, or used directly (float).  Results are within an ulp or two of the correctly
// rounded value; the parity tolerance is 1e-12.  Only for operands well inside the normal range
// (densities, sound speeds, mass fluxes): the estimate overflows for subnormal divisors.
//   reciprocal: one cubic step r (1 + e + e^2), e = 1 - x r, leaves e^3 ~ 2^-69 (4 instructions;
//               two quadratic steps take 5 and a longer chain);
//   quotient:   one quadratic step on the reciprocal (2^-46), then the residual correction of the
//               quotient itself, whose error is the product of both (6 instructions against 8);
//   root:       one Goldschmidt step (2^-45), then one residual correction.
__device__ inline double frcp(double x) {
    const double r = __builtin_amdgcn_rcp(x);
    const double e = __builtin_fma(-x, r, 1.0);
    return __builtin_fma(r, __builtin_fma(e, e, e), r);
}
__device__ inline float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ inline double fdiv(double a, double b) {
    double r = __builtin_amdgcn_rcp(b);
    r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}
__device__ inline float fdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
// for normal-range arguments and zero; negative arguments give NaN.  The addend keeps the
// estimate of a zero finite (its root comes out as 1e-150) and leaves every other argument as it is,
// in one instruction where selecting the zero took three.
__device__ inline double fsqrt(double x) {
    x += 1e-300;
    const double r = __builtin_amdgcn_rsq(x);
    double y = x * r;
    const double h = 0.5 * r;
    y = __builtin_fma(y, __builtin_fma(-h, y, 0.5), y);
    return __builtin_fma(__builtin_fma(-y, y, x), h, y);
}
__device__ inline float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }

// one-instruction maximum / minimum in the arithmetic type (v_max_f64 / v_max_f32, no
// conversion to double for float operands)
__device__ inline double vmax(double a, double b) { return __builtin_fmax(a, b); }
__device__ inline float vmax(float a, float b) { return __builtin_fmaxf(a, b); }
__device__ inline double vmin(double a, double b) { return __builtin_fmin(a, b); }
__device__ inline float vmin(float a, float b) { return __builtin_fminf(a, b); }
__device__ inline double vabs(double a) { return __builtin_fabs(a); }
__device__ inline float vabs(float a) { return __builtin_fabsf(a); }

// The same on values that come straight from memory: the compiler would first pass each of them
// through a maximum with itself, in case it is a signalling NaN (25 extra instructions per row of a
// 2-D reconstruction); v_max_f64 and v_min_f64 quiet those by themselves.
__device__ inline double vmax_mem(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ inline double vmin_mem(double a, double b) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ inline float vmax_mem(float a, float b) { return __builtin_fmaxf(a, b); }
__device__ inline float vmin_mem(float a, float b) { return __builtin_fminf(a, b); }

// smallest divisor the limiter uses: well inside the normal range, where the reciprocal
// estimate and its Newton steps are accurate
template <typename R> __device__ inline R tiny_divisor();
template <> __device__ inline double tiny_divisor<double>() { return 1e-290; }
template <> __device__ inline float tiny_divisor<float>() { return 1e-35f; }

// ---- equation of state (generalEOS.h:6-23; ideal gas, idealGasEOS.h:7-46) -------------------
// The reference's GeneralEOS interface as a device functor: pressure, sound speed and specific
// internal energy, and the two pressure derivatives, as functions of the density and the
// specific internal energy e (these five follow the reference's formulas operation for
// operation, with IEEE division and square root).  The kernels work on conserved variables, so
// the functor also gives the volumetric forms they evaluate: the pressure of an internal energy
// density rho e, the sound speed from p and 1/rho, and rho e of a pressure -- each the
// reference's method with the density factor folded in (for an ideal gas
// GetPressure(rho, rho e / rho) = (gamma - 1) rho e, with no division).  HLLC, its dt
// eigenvalues, the boundary images and the exact solver's pressures and face energy go through
// it.  The Roe flux and the exact solver's wave relations are the reference's perfect-gas
// formulas (RoeSolverPerfectGasEOS.h, GodunovSolverPerfectGasEOS.h) and use gamma directly.
__device__ inline double ieee_sqrt(double x) { return __builtin_sqrt(x); }
__device__ inline float ieee_sqrt(float x) { return __builtin_sqrtf(x); }

template <typename R>
struct IdealGasEOS {
    R gamma;
    __device__ explicit IdealGasEOS(R g) : gamma(g) {}
    // GeneralEOS (generalEOS.h:9-21) as IdealGasEOS implements it (idealGasEOS.h:22-44)
    __device__ R GetPressure(R ro, R e) const { return (gamma - R(1)) * ro * e; }
    __device__ R GetSoundSpeed(R ro, R e) const {
        const R pressure = (gamma - R(1)) * ro * e;
        return ieee_sqrt(gamma * pressure / ro);
    }
    __device__ R GetInternalEnergy(R ro, R pressure) const { return pressure / ((gamma - R(1)) * ro); }
    __device__ R GetPressureEnergyDerivative(R ro, R) const { return (gamma - R(1)) * ro; }
    __device__ R GetPressureDensityDerivative(R, R e) const { return (gamma - R(1)) * e; }
    // volumetric forms of the kernels (rho_e = rho e; inv_ro = 1/rho from the caller's reciprocal)
    __device__ R PressureOfEnergyDensity(R rho_e) const { return (gamma - R(1)) * rho_e; }
    __device__ R SoundSpeedOfPressure(R p, R inv_ro) const { return fsqrt(gamma * p * inv_ro); }
    __device__ R EnergyDensityOfPressure(R p) const { return p / (gamma - R(1)); }
};

// Image state of a boundary condition across a face normal to `axis` (getDummyValues,
// BCGeneral.h:186-268).  Every condition in the reference is even in the normal's sign, so the
// ghost fill (normal -e_axis on both sides, kernel.h:743,760) and the boundary-face states
// (normal +e_axis, ExplicitRungeKuttaFVM.h:1202,1208) share this one function.
template <typename R, int N>
__device__ __forceinline__ void bc_image(const BCDev& bc, R gamma, int axis, const R (&u)[N], R (&o)[N]) {
    switch (bc.type) {
    case BC_SYMMETRY:
        // U - 2 (n.m) n: only the normal momentum changes sign
#pragma unroll
        for (int v = 0; v < N; v++) o[v] = u[v];
        o[1 + axis] = -u[1 + axis];
        break;
    case BC_WALL:
        o[0] = u[0];
#pragma unroll
        for (int v = 1; v < N - 1; v++) o[v] = -u[v];
        o[N - 1] = u[N - 1];
        break;
    case BC_MOVING_WALL: {
        const R rho = u[0];
        const R ir = R(1) / rho;
        R in = R(0), out = R(0);
        o[0] = rho;
#pragma unroll
        for (int v = 1; v < N - 1; v++) {
            const R vel = u[v] * ir, img = R(2) * R(bc.vel[v - 1]) - vel;
            in += vel * vel;
            out += img * img;
            o[v] = rho * img;
        }
        const R rhoe = u[N - 1] - R(0.5) * rho * in;
        o[N - 1] = rhoe + R(0.5) * rho * out;
        break;
    }
    case BC_SUBSONIC_INLET: {
        const R r = R(bc.rho);
        R q = R(0);
        o[0] = r;
#pragma unroll
        for (int v = 1; v < N - 1; v++) {
            const R vel = R(bc.vel[v - 1]);
            q += vel * vel;
            o[v] = r * vel;
        }
        o[N - 1] = IdealGasEOS<R>(gamma).EnergyDensityOfPressure(R(bc.p)) + R(0.5) * r * q;
        break;
    }
    default:  // Natural, SubsonicOutlet: copy
#pragma unroll
        for (int v = 0; v < N; v++) o[v] = u[v];
    }
}

template <typename R> __device__ inline R tiny_spread();
template <> __device__ inline double tiny_spread<double>() { return 3.0 * 2.2250738585072014e-308; }
template <> __device__ inline float tiny_spread<float>() { return 3.0f * 1.17549435e-38f; }

// ---- reconstruction ------------------------------------------------------------------------
// Values of Reconstruction / LimiterType (src/Methods/MethodConfiguration.h:5-21)
enum : int { RC_PWC = 0, RC_LINEAR = 1, RC_ENO2 = 2, RC_LINLIM = 3 };
enum : int { LIM_BJ = 0, LIM_VENKAT = 1 };

// Geometry of one cell along its ND axes: half sizes and slope denominators.
template <int ND, typename R>
struct CellGeo {
    R hh[ND];   // 0.5 * h (face sample offset, Linear2psLim.h:77-89, ERK:1194-1195)
    R rc[ND];   // 1 / (x_{i+1} - x_{i-1})  (Linear2PointsStencil.h:72)
    R rl[ND];   // 1 / (x_i - x_{i-1})      (ENO2PointsStencil.h:28)
    R rr[ND];   // 1 / (x_{i+1} - x_i)      (ENO2PointsStencil.h:29)
    R eps2;     // Venkatakrishnan (K dx)^3 (Limiters.h:93-96)
};

// Reconstruct one cell: its state on the minus face of axis a is c - t[a], on the plus face c + t[a].
// nb[2a], nb[2a+1] are the axis neighbours (x-,x+,y-,y+,z-,z+), the stencil of
// ComputeSolutionReconstruction (ERK:897-916).
template <int ND, int RECON, int LIM, typename R, int N>
__device__ inline void face_offsets(const R (&c)[N], const R (&nb)[2 * ND][N], const CellGeo<ND, R>& geo, R (&t)[ND][N]) {
#pragma unroll
    for (int v = 0; v < N; v++) {
        if constexpr (RECON == RC_PWC) {  // PiecewiseConstant.h:15
#pragma unroll
            for (int a = 0; a < ND; a++) t[a][v] = R(0);
        } else if constexpr (RECON == RC_LINLIM && LIM == LIM_BJ) {
            // Limited linear with Barth-Jespersen (Linear2psLim.h:64-96, Limiters.h:28-67,80-82).
            // Along each axis the two face projections are +-d_a, d_a = g_a h_a / 2 with the
            // central slope g_a (Linear2PointsStencil.h:66-97); one is bounded by umax and the
            // other by umin, so the minimum over the faces of min(1, (u_m - u_i)/d2) is
            // min(umax - c, c - umin) / max_a |d_a| when that is below 1.  The projection is
            // formed as (u_+ - u_-) (h_a / (2 (x_+ - x_-))) rather than the reference's
            // (c + g.p) - c: the two differ by an ulp of c, and so do the face values.  A
            // variable without spread has d_a = 0 and keeps its cell value, as the reference's
            // spread test (Limiters.h:50) gives.
            // The largest |d_a| starts at a floor, so that the divisor of a variable that is
            // constant up to round-off stays in the reciprocal's range; its face values move by
            // less than the floor.
            R d[ND], dmax = tiny_divisor<R>();
#pragma unroll
            for (int a = 0; a < ND; a++) {
                d[a] = (nb[2 * a + 1][v] - nb[2 * a][v]) * (geo.rc[a] * geo.hh[a]);
                dmax = vmax(dmax, vabs(d[a]));
            }
            R umax = c[v], umin = c[v];
#pragma unroll
            for (int n = 0; n < 2 * ND; n++) {
                umax = vmax_mem(umax, nb[n][v]);
                umin = vmin_mem(umin, nb[n][v]);
            }
            const R hi = umax - c[v], lo = c[v] - umin;
            const R lim = vmin(fdiv(vmin(hi, lo), dmax), R(1));
#pragma unroll
            for (int a = 0; a < ND; a++) t[a][v] = lim * d[a];
        } else {
            R g[ND];
#pragma unroll
            for (int a = 0; a < ND; a++) {
                if constexpr (RECON == RC_ENO2) {  // ENO2PointsStencil.h:21-58
                    R gl = (c[v] - nb[2 * a][v]) * geo.rl[a];
                    R gr = (nb[2 * a + 1][v] - c[v]) * geo.rr[a];
                    g[a] = (__builtin_fabs(gl) < __builtin_fabs(gr)) ? gl : gr;
                } else {  // Linear2PointsStencil.h:66-97
                    g[a] = (nb[2 * a + 1][v] - nb[2 * a][v]) * geo.rc[a];
                }
            }
            R lim = R(1);
            if constexpr (RECON == RC_LINLIM) {
                // Limiter::ComputeLimiterValues (Limiters.h:28-67).  The minimum over the
                // faces of min(1, l_j) is found by comparing fractions A/D, then divided once.
                R umax = c[v], umin = c[v];
#pragma unroll
                for (int n = 0; n < 2 * ND; n++) {
                    umax = __builtin_fmax(umax, nb[n][v]);
                    umin = __builtin_fmin(umin, nb[n][v]);
                }
                if (!(umax - umin < tiny_spread<R>())) {
                    {  // Venkatakrishnan (Barth-Jespersen takes the branch above)
                        R bestA = R(1), bestD = R(1);
                        R inv_un = frcp(R(0.5) * (umax - umin));
#pragma unroll
                        for (int a = 0; a < ND; a++) {
#pragma unroll
                            for (int s = 0; s < 2; s++) {
                                R pt = s ? geo.hh[a] : -geo.hh[a];
                                R d2;
                                {
#pragma clang fp contract(off)
                                    R fv = c[v] + g[a] * pt;
                                    d2 = fv - c[v];
                                }
                                if (d2 > R(0) || d2 < R(0)) {
                                    // Venkatakrishnan (Limiters.h:102-115), normalised by
                                    // (umax - umin)/2
                                    R um = (d2 > R(0)) ? umax : umin;
                                    R dm = um * inv_un - c[v] * inv_un;
                                    R dn = d2 * inv_un;
                                    R A = (dm * dm + geo.eps2) + R(2) * dn * dm;
                                    R D = dm * dm + R(2) * dn * dn + dm * dn + geo.eps2;
                                    if (A * bestD < bestA * D) { bestA = A; bestD = D; }
                                }
                            }
                        }
                        lim = (bestA == bestD) ? R(1) : bestA / bestD;
                    }
                }
            }
#pragma unroll
            for (int a = 0; a < ND; a++) {
                t[a][v] = g[a] * geo.hh[a];  // Linear2PointsStencil.h:26-30
                if constexpr (RECON == RC_LINLIM) t[a][v] *= lim;  // Linear2psLim.h:17-21
            }
        }
    }
}

// whether a state has no real sound speed (rho <= 0 or 2 rho E <= |m|^2)
template <typename R, int N>
__device__ __forceinline__ bool no_sound_speed(const R (&u)[N]) {
    return !(u[0] > R(0) && R(2) * u[0] * u[N - 1] - momentum2(u) > R(0));
}

// The face states themselves, face[2a] on the minus face of axis a and face[2a+1] on the plus face.
// With POS set (the HLLC and exact-Godunov paths), a face state without a real sound speed falls
// back to the cell value.
template <int ND, int RECON, int LIM, typename R, bool POS = false, int N>
__device__ inline void reconstruct(const R (&c)[N], const R (&nb)[2 * ND][N],
                                   const CellGeo<ND, R>& geo, R (&face)[2 * ND][N]) {
    {
        R t[ND][N];
        face_offsets<ND, RECON, LIM>(c, nb, geo, t);
#pragma unroll
        for (int a = 0; a < ND; a++)
#pragma unroll
            for (int v = 0; v < N; v++) {
                face[2 * a][v] = c[v] - t[a][v];
                face[2 * a + 1][v] = c[v] + t[a][v];
            }
    }
    if constexpr (POS && RECON != RC_PWC) {
        bool bad[2 * ND];
        bool any = false;
#pragma unroll
        for (int f = 0; f < 2 * ND; f++) {
            bad[f] = no_sound_speed(face[f]);
            any = any || bad[f];
        }
        // rare: a branch the wavefront skips when none of its lanes needs the fallback
        if (__builtin_expect(any, 0)) {
#pragma unroll
            for (int f = 0; f < 2 * ND; f++)
                if (bad[f]) {
#pragma unroll
                    for (int v = 0; v < N; v++) face[f][v] = c[v];
                }
        }
    }
}

// ---- Riemann solvers -------------------------------------------------------------------------
enum : int { FX_GODUNOV = 0, FX_ROE = 1, FX_HLLC = 3 };

// Internal energy density E - rho|v|^2/2 from the conserved state.  In the FP32 form the
// difference is redone in double when it is a small part of E (near vacuum, where the float
// subtraction loses most of its digits).
template <int N>
__device__ inline float checked_energy(float e, const float (&U)[N]) {
    if (e < 0.01f * U[N - 1]) {
        double m2 = double(U[1]) * U[1];
#pragma unroll
        for (int i = 2; i < N - 1; i++) m2 = __builtin_fma(double(U[i]), double(U[i]), m2);
        e = float(double(U[N - 1]) - 0.5 * m2 / double(U[0]));
    }
    return e;
}
template <int N>
__device__ inline double checked_energy(double e, const double (&)[N]) { return e; }
template <typename R, int N>
__device__ inline R internal_energy(R E, R rho_ke, const R (&U)[N]) { return checked_energy(E - rho_ke, U); }

// Roe-Pike flux with Harten's entropy fix (RoeSolverPerfectGasEOS.h:48-134) across a face with
// normal +e_D.  lam receives |u.n| + c of the Roe average (RoeSolverPerfectGasEOS.h:88,128).
template <int D, typename R, int N>
__device__ inline void roe_flux(R gamma, R eps, const R (&UL)[N], const R (&UR)[N], R (&F)[N],
                                R& lam) {
    constexpr int NM = N - 2;  // velocity components
    const R gm1 = gamma - R(1);
    R il = frcp(UL[0]), ir = frcp(UR[0]);
    R vl[NM], vr[NM];
#pragma unroll
    for (int i = 0; i < NM; i++) {
        vl[i] = UL[1 + i] * il;
        vr[i] = UR[1 + i] * ir;
    }
    const R kl = R(0.5) * dot(vl, vl), kr = R(0.5) * dot(vr, vr);
    R el = UL[N - 1] * il, er = UR[N - 1] * ir;
    // physical fluxes (RoeSolverPerfectGasEOS.h:15-32)
    R pl = gm1 * internal_energy(UL[N - 1], UL[0] * kl, UL);
    R pr = gm1 * internal_energy(UR[N - 1], UR[0] * kr, UR);
    R hl = (el - kl) * gamma + kl;
    R hr = (er - kr) * gamma + kr;
    R sl = fsqrt(UL[0]), sr = fsqrt(UR[0]);
    R isum = frcp(sl + sr);
    R ql = sl * isum, qr = sr * isum;
    R v[NM];
#pragma unroll
    for (int i = 0; i < NM; i++) v[i] = ql * vl[i] + qr * vr[i];
    const R vv = dot(v, v), vvl = dot(v, vl), vvr = dot(v, vr);
    R h = ql * hl + qr * hr;
    R phi2 = R(0.5) * gm1 * vv;
    R c = fsqrt(gm1 * h - phi2);
    R uw = v[D];
    R eig = __builtin_fabs(uw) + c;
    R e = eps * eig;
    R a1 = __builtin_fabs(uw), a3 = __builtin_fabs(uw + c), a4 = __builtin_fabs(uw - c);
    if (a1 < e) a1 = (a1 * a1 / e + e) * R(0.5);  // Harten (RoeSolverPerfectGasEOS.h:35-40)
    if (a3 < e) a3 = (a3 * a3 / e + e) * R(0.5);
    if (a4 < e) a4 = (a4 * a4 / e + e) * R(0.5);
    R ic = frcp(c);
    R Eig1 = a1;
    R Eiga = (a3 - a4) * R(0.5) * ic;
    R Eigb = (a3 + a4) * R(0.5) - a1;
    R R1 = phi2 * UR[0] - gm1 * UR[0] * (vvr - er);
    R R2 = phi2 * UL[0] - gm1 * UL[0] * (vvl - el);
    R D1 = UR[0] * (vr[D] - v[D]);
    R D2 = UL[0] * (vl[D] - v[D]);
    R C2 = ic * ic;
    // dissipation (RoeSolverPerfectGasEOS.h:96-125) with Qa = (0, n, u.n), Qb = (1, v, h)
    R vnl = vl[D], vnr = vr[D];
    R FL[N], FR[N], Qb[N];
    FL[0] = UL[0] * vnl; FR[0] = UR[0] * vnr;
    Qb[0] = R(1);
#pragma unroll
    for (int i = 0; i < NM; i++) {
        FL[1 + i] = FL[0] * vl[i];
        FR[1 + i] = FR[0] * vr[i];
        Qb[1 + i] = v[i];
    }
    FL[1 + D] += pl; FR[1 + D] += pr;
    FL[N - 1] = vnl * (UL[N - 1] + pl); FR[N - 1] = vnr * (UR[N - 1] + pr);
    Qb[N - 1] = h;
#pragma unroll
    for (int i = 0; i < N; i++) {
        R qa = (i == N - 1) ? uw : ((i == 1 + D) ? R(1) : R(0));
        R diss = Eig1 * (UL[i] - UR[i]) + Eiga * ((R2 - R1) * qa + (D2 - D1) * Qb[i]) +
                 Eigb * ((R2 - R1) * Qb[i] * C2 + (D2 - D1) * qa);
        F[i] = R(0.5) * (FL[i] + FR[i] + diss);
    }
    lam = eig;
}

// The same from the momenta, 1 / rho and the velocity along D, with rho |u|^2 formed as momentum times velocity:
// its range is that of the energy itself, where the momenta's squares leave a float's for densities of
// 1e-21 or 1e21.
template <int D, typename R, int N>
__device__ __forceinline__ R internal_energy_along(const R (&u)[N], R ir, R un) {
#pragma clang fp contract(off)
    R s = un * u[1 + D];
#pragma unroll
    for (int i = 1; i < N - 1; i++)
        if (i != 1 + D) s = madd(u[i] * ir, u[i], s);
    const R e = madd(R(-0.5), s, u[N - 1]);
    return checked_energy(e, u);
}

// HLLC flux (Toro, Riemann Solvers and Numerical Methods for Fluid Dynamics, 3rd ed.,
// sec. 10.4, eqs. 10.37-10.39) with Davis wave-speed bounds (eq. 10.48); lam = max(|SL|,|SR|).
// Extension with no counterpart in the reference.  Branch-free: the upwind side K of the contact is
// selected first, then the flux of the state the face lies in is formed once.  With w = S_K - u_K
// and r = 1 / (S_K - S*), the star state's density is rho_K w r, its tangential momentum m_t w r, its
// pressure p* = p_K + rho_K w (S* - u_K) and its energy (w E_K - p_K u_K + p* S*) r (the jump
// conditions across S_K), and its flux needs no more than that: (rho, m_t) S*, rho S*^2 + p*,
// S* (E + p*).  A supersonic side takes its own velocity, pressure and energy in the places of
// the star's.  (Against F_K + S_K (U* - U_K), which needs the whole flux of side K and
// its velocities first: about 50 instructions fewer per face in double.)
template <int D, typename R, int N>
__device__ inline void hllc_flux(R gamma, const R (&UL)[N], const R (&UR)[N], R (&F)[N],
                                 R& lam) {
    // every fused operation is written out, so that a plane flow's kernels and those with all variables, and
    // the dt pass, form the same bits
#pragma clang fp contract(off)
    const IdealGasEOS<R> eos(gamma);
    const R il = frcp(UL[0]), ir = frcp(UR[0]);
    const R ul = UL[1 + D] * il, ur = UR[1 + D] * ir;
    const R pl = eos.PressureOfEnergyDensity(internal_energy_along<D>(UL, il, ul));
    const R pr = eos.PressureOfEnergyDensity(internal_energy_along<D>(UR, ir, ur));
    const R al = eos.SoundSpeedOfPressure(pl, il), ar = eos.SoundSpeedOfPressure(pr, ir);
    const R SL = vmin(ul - al, ur - ar);
    const R SR = vmax(ul + al, ur + ar);
    lam = vmax(vabs(SL), vabs(SR));
    const R wl = SL - ul, wr = SR - ur;
    const R ml = UL[0] * wl, mr = UR[0] * wr;
    const R Ss = fdiv(madd(-ur, mr, madd(ul, ml, pr - pl)), ml - mr);
    const bool left = Ss >= R(0);
    const R S = left ? SL : SR, w = left ? wl : wr, m = left ? ml : mr;
    const R rho = left ? UL[0] : UR[0], un = left ? ul : ur, p = left ? pl : pr, E = left ? UL[N - 1] : UR[N - 1];
    const bool supersonic = left ? (S >= R(0)) : (S <= R(0));
    // on a subsonic side S - S* is not zero (S < 0 <= S*, or the mirror case)
    const R r = frcp(supersonic ? R(1) : S - Ss);
    const R ps = madd(m, Ss - un, p);
    const R Es = madd(ps, Ss, madd(w, E, -(p * un))) * r;
    const R c = supersonic ? R(1) : w * r;
    const R uf = supersonic ? un : Ss, pf = supersonic ? p : ps, Ef = supersonic ? E : Es;
    const R q = c * uf;
    F[0] = rho * q;
#pragma unroll
    for (int i = 1; i < N - 1; i++)
        if (i != 1 + D) F[i] = (left ? UL[i] : UR[i]) * q;
    F[1 + D] = madd(F[0], uf, pf);
    F[N - 1] = uf * (Ef + pf);
}

// ---- exact Riemann solver (always double) -----------------------------------------------------
// Powers x^y = exp(y ln x) of the exact solver's bases (pressure ratios, the two-rarefaction
// guess, the fan's C_K), all non-negative, with positive exponents, evaluated in line:
//   ln x: x = m 2^e with m in [1/sqrt2, sqrt2), ln m = 2 atanh s = 2 s (1 + s^2/3 + s^4/5 + ...)
//         with s = (m - 1)/(m + 1), |s| <= 0.172, summed to s^21 (the next term is below 1e-18);
//   exp t: t = k ln2 + r with k = rint(t / ln2), |r| <= 0.347, ln2 split in a high part with 32
//         significant bits (k ln2_hi exact) and the rest, and e^r by its Taylor series to r^13
//         (remainder below 5e-18), scaled by 2^k.
// On 2e6 bases in [1e-12, 1e4] with the solver's exponents this is within 2e-15 of the correctly
// rounded power for y <= 1 and 1.5e-14 for y up to 7 (the rounding of t = y ln x), the same as
// exp(y ln x) with the library's ln and exp, in 101 VALU instructions against their 139 (and 223
// for the library's correctly rounded pow).  One out-of-line copy: inlined at each call site the
// kernels outgrew the instruction cache.
// x = 0 gives 0; x < 0 or NaN gives NaN; x = +inf gives +inf.
static __device__ __noinline__ double dpow(double x, double y) {
    if (!(x > 0.0)) return x == 0.0 ? 0.0 : __builtin_nan("");
    if (x == __builtin_inf()) return x;
    constexpr double LN2_HI = 0.6931471803691238, LN2_LO = 1.9082149292705877e-10;
    int e;
    double m = __builtin_frexp(x, &e);
    if (m < 0.7071067811865476) {
        m *= 2.0;
        e -= 1;
    }
    const double s = fdiv(m - 1.0, m + 1.0);
    const double w = s * s;
    double p = 1.0 / 21.0;
    p = __builtin_fma(p, w, 1.0 / 19.0);
    p = __builtin_fma(p, w, 1.0 / 17.0);
    p = __builtin_fma(p, w, 1.0 / 15.0);
    p = __builtin_fma(p, w, 1.0 / 13.0);
    p = __builtin_fma(p, w, 1.0 / 11.0);
    p = __builtin_fma(p, w, 1.0 / 9.0);
    p = __builtin_fma(p, w, 1.0 / 7.0);
    p = __builtin_fma(p, w, 1.0 / 5.0);
    p = __builtin_fma(p, w, 1.0 / 3.0);
    p = __builtin_fma(p, w, 1.0);
    const double lnm = 2.0 * s * p;
    const double de = double(e);
    const double lnx = de * LN2_HI + __builtin_fma(de, LN2_LO, lnm);
    const double t = y * lnx;
    const double k = __builtin_rint(t * 1.4426950408889634);
    const double r = __builtin_fma(-k, LN2_LO, __builtin_fma(-k, LN2_HI, t));
    // 1/j! for j = 13 .. 2, then 1, 1
    double q = 1.6059043836821613e-10;
    q = __builtin_fma(q, r, 2.08767569878681e-09);
    q = __builtin_fma(q, r, 2.505210838544172e-08);
    q = __builtin_fma(q, r, 2.755731922398589e-07);
    q = __builtin_fma(q, r, 2.7557319223985893e-06);
    q = __builtin_fma(q, r, 2.48015873015873e-05);
    q = __builtin_fma(q, r, 0.0001984126984126984);
    q = __builtin_fma(q, r, 0.001388888888888889);
    q = __builtin_fma(q, r, 0.008333333333333333);
    q = __builtin_fma(q, r, 0.041666666666666664);
    q = __builtin_fma(q, r, 0.16666666666666666);
    q = __builtin_fma(q, r, 0.5);
    q = __builtin_fma(q, r, 1.0);
    q = __builtin_fma(q, r, 1.0);
    return __builtin_ldexp(q, int(k));
}

// The side-K constants of f_K (GodunovSolverPerfectGasEOS.h:58-97), formed once per face
// instead of once per Newton iteration.
struct SideDev {
    double pk, ak;
    double A, B;  // 2 / ((g+1) rho_K), p_K (g-1)/(g+1): the shock branch
    double ipk;   // 1 / p_K
    double ira;   // 1 / (rho_K a_K)
    double c2a;   // 2 a_K / (g-1)
};
// cA = 2/(g+1), cB = (g-1)/(g+1), c2 = 2/(g-1)
__device__ inline SideDev side_dev(double cA, double cB, double c2, double ir, double pk, double ak, double r) {
    SideDev s;
    s.pk = pk;
    s.ak = ak;
    s.A = cA * ir;
    s.B = pk * cB;
    s.ipk = frcp(pk);
    s.ira = frcp(r * ak);
    s.c2a = c2 * ak;
    return s;
}

// f_K(p) and its derivative (GodunovSolverPerfectGasEOS.h:58-97; derivative Toro eq. 4.37);
// z = (g-1)/2g.  The reciprocals and the square root are the refined estimates (a few ulps).
// `pzk` = (p/pK)^z, used on the rarefaction side.
__device__ inline double fk_dev(const SideDev& s, double p, double pzk, double& d, double& pz) {
    if (p > s.pk) {
        const double ipb = frcp(p + s.B);
        const double q = fsqrt(s.A * ipb);
        d = q * (1.0 - 0.5 * (p - s.pk) * ipb);
        pz = 0.0;
        return (p - s.pk) * q;
    }
    // rarefaction: the power (p/pK)^z gives f, f' = (p/pK)^(z-1)/(r aK) and the tail speed of
    // the fan (the sampler reuses pz)
    const double pr = p * s.ipk;
    pz = pzk;
    d = pz * frcp(pr) * s.ira;
    return (pz - 1.0) * s.c2a;
}
// (p/pL)^z and (p/pR)^z with one power: (p/pR)^z = (p/pL)^z (pL/pR)^z, the last factor formed
// once per face; skipped when neither side is a rarefaction at p
__device__ inline void side_powers(const SideDev& l, const SideDev& r, double z, double rho_lr, double p, double& pzl,
                                   double& pzr) {
    pzl = pzr = 0.0;
    if (!(p > l.pk) || !(p > r.pk)) {
        pzl = dpow(p * l.ipk, z);
        pzr = pzl * rho_lr;
    }
}

// Star pressure and velocity, wave speeds and smax; the star densities are formed by the sampler,
// for the sampled side only.
struct StarDev {
    double p, u, SL, SHL, STL, SR, SHR, STR, smax;
    bool shock_l, shock_r, vacuum;
};

// Star state by Newton-Raphson from Toro's adaptive initial guess (Toro sec. 4.3, 9.5.1); the
// reference uses ALGLIB's bounded Levenberg-Marquardt for the same root
// (GodunovSolverPerfectGasEOS.h:143-185).  Divergent lanes simply run a masked loop, so a
// wavefront pays for its slowest lane: what bounds the exact solver is the number of evaluations
// of f_K (a power, two branches, about 190 instructions) and, in a short grid, their serial chain.
//   - The loop ends after a step D with |D| <= 1e-8 p: f is concave with |f''| < f' / p, so the error
//     after that step is below (D/p)^2 / 2 = 5e-17 p, and the evaluation that would confirm it is
//     not made.
//   - f_K and (p/p_K)^z at the final p come from the last evaluation, one such step away, to
//     first order: the next term is as small.
//   - Pressures within a factor of two start from the primitive-variable guess wherever that is
//     not far below both: Newton takes no more steps from it than from the two-rarefaction formula,
//     whose three powers every lane of the wavefront would wait for.
__device__ inline StarDev star_state_dev(double g, double rl, double ul, double pl, double rr,
                                         double ur, double pr, double al, double irl, double irr) {
    StarDev s;
    const double ar = fsqrt(g * pr * irr);  // (and al, the left side's)
    const double du = ur - ul;
    const double ig = frcp(g), igp = frcp(g + 1.0), c2 = 2.0 * frcp(g - 1.0);
    s.vacuum = c2 * (al + ar) <= du;
    const double z = 0.5 * (g - 1.0) * ig;
    const double cA = 2.0 * igp, cB = (g - 1.0) * igp;
    const SideDev sl = side_dev(cA, cB, c2, irl, pl, al, rl), sr = side_dev(cA, cB, c2, irr, pr, ar, rr);
    const double rho_lr = dpow(pl * sr.ipk, z);  // (pL/pR)^z
    double p = 0.0;
    double f1 = 0.0, f2 = 0.0, pzl = 0.0, pzr = 0.0;
    bool known = false;  // f_L, f_R and the powers at p are formed
    // Inputs that are not a physical state (zero, negative or NaN density or pressure) give a
    // NaN star pressure straight away.  Such inputs reach the solver on halo lanes, which are
    // fed by a cross-lane shift and whose flux is discarded; iterating on them to the cap would
    // hold the whole wavefront.  (For a face whose flux is used they give NaN either way.)
    const bool physical = rl > 0.0 && pl > 0.0 && rr > 0.0 && pr > 0.0;
    if (!physical) {
        p = __builtin_nan("");
    } else if (!s.vacuum) {
        const double pmin = __builtin_fmin(pl, pr), pmax = __builtin_fmax(pl, pr);
        double ppv = 0.5 * (pl + pr) - 0.125 * du * (rl + rr) * (al + ar);
        ppv = __builtin_fmax(0.0, ppv);
        if (pmax <= 2.0 * pmin && ppv >= 0.5 * pmin && ppv <= pmax) {
            p = ppv;
        } else if (ppv < pmin) {
            const double plz = dpow(pl, z), prz = dpow(pr, z);
            const double t = fdiv(al + ar - 0.5 * (g - 1.0) * du, fdiv(al, plz) + fdiv(ar, prz));
            p = dpow(t, g * c2);
        } else {
            const double gl = fsqrt(sl.A * frcp(ppv + sl.B));
            const double gr = fsqrt(sr.A * frcp(ppv + sr.B));
            p = fdiv(gl * pl + gr * pr - du, gl + gr);
        }
        if (!(p > 0.0)) p = 1e-12 * pmin;
        for (int it = 1; it <= 60; it++) {
            double dl, dr, zl, zr;
            double ql, qr;
            side_powers(sl, sr, z, rho_lr, p, ql, qr);
            const double fl = fk_dev(sl, p, ql, dl, zl), fr = fk_dev(sr, p, qr, dr, zr);
            const double f = fl + fr + du;
            double pn = p - fdiv(f, dl + dr);
            if (!(pn > 0.0)) pn = 0.01 * p;
            const double dp = pn - p;
            if (__builtin_fabs(dp) <= 1e-8 * p) {
                known = true;
                f1 = fl + dl * dp;
                f2 = fr + dr * dp;
                // on a shock's side at the last evaluation the power was not formed; where the step
                // leads to that side's own pressure it is next to 1
                const double zp = z * fdiv(dp, p);
                pzl = p > pl ? 1.0 + z * (pn * sl.ipk - 1.0) : zl + zl * zp;
                pzr = p > pr ? 1.0 + z * (pn * sr.ipk - 1.0) : zr + zr * zp;
                p = pn;
                break;
            }
            p = pn;
        }
    }
    s.p = p;
    if (!known) {  // vacuum, a non-physical input, or the iteration cap
        double d1, d2;
        double ql, qr;
        side_powers(sl, sr, z, rho_lr, p, ql, qr);
        f1 = fk_dev(sl, p, ql, d1, pzl);
        f2 = fk_dev(sr, p, qr, d2, pzr);
    }
    s.u = 0.5 * (ul + ur) + 0.5 * (f2 - f1);
    s.smax = 0.0;
    s.SL = s.SHL = s.STL = s.SR = s.SHR = s.STR = 0.0;
    const double gs = 0.5 * (g + 1.0) * ig;
    if (p > pl) {
        s.shock_l = true;
        s.SL = ul - al * fsqrt(gs * (p * sl.ipk) + z);
        s.smax = __builtin_fmax(s.smax, __builtin_fabs(s.SL));
    } else {
        s.shock_l = false;
        s.SHL = ul - al;
        s.STL = s.u - al * pzl;  // (p/pL)^((g-1)/2g), from f_L
        s.smax = __builtin_fmax(s.smax, __builtin_fabs(s.SHL));
    }
    if (p > pr) {
        s.shock_r = true;
        s.SR = ur + ar * fsqrt(gs * (p * sr.ipk) + z);
        s.smax = __builtin_fmax(s.smax, __builtin_fabs(s.SR));
    } else {
        s.shock_r = false;
        s.SHR = ur + ar;
        s.STR = s.u + ar * pzr;
        s.smax = __builtin_fmax(s.smax, __builtin_fabs(s.SHR));
    }
    if (s.vacuum) {  // the fan tails bound the vacuum (Toro sec. 4.6)
        s.STL = ul + c2 * al;
        s.STR = ur - c2 * ar;
    }
    return s;
}

// Exact Godunov flux: the solution sampled at x/t = 0 (GodunovSolverPerfectGasEOS.h:276-433),
// tangential velocity from the upwind side of the contact.  Computed in double for both
// arithmetic forms.
template <int D, typename R, int N>
__device__ inline void godunov_flux(R gammaR, const R (&ULr)[N], const R (&URr)[N], R (&F)[N],
                                    R& lam) {
    constexpr int NM = N - 2;  // velocity components
    const double g = double(gammaR);
    const IdealGasEOS<double> eos(g);
    double UL[N], UR[N];
#pragma unroll
    for (int i = 0; i < N; i++) { UL[i] = double(ULr[i]); UR[i] = double(URr[i]); }
    const double il = frcp(UL[0]), ir = frcp(UR[0]);
    double vL[NM], vR[NM];
#pragma unroll
    for (int i = 0; i < NM; i++) {
        vL[i] = UL[1 + i] * il;
        vR[i] = UR[1 + i] * ir;
    }
    const double kL = dot(vL, vL), kR = dot(vR, vR);
    double pL = eos.GetPressure(UL[0], UL[N - 1] * il - kL / 2.0);
    double pR = eos.GetPressure(UR[0], UR[N - 1] * ir - kR / 2.0);
    double uL = vL[D], uR = vR[D];
    // Ahead of the waves a tube is constant, half of it on average over a run, and its faces have the
    // same state on both sides: a wavefront of nothing else skips the star state and the sampling, about 900
    // instructions.  (All lanes or none: with a single other face among them the wavefront runs the
    // whole solver anyway.)  Batch of 1024 tubes 346 -> 304 ms, a 1000-cell tube 38 -> 32 ms.  Such a face
    // has the flux and the speed of its state in either case, lane by lane: the two cells beside a face may
    // ask two wavefronts for it.
    const double S = 0.0;
    bool same = UL[0] > 0.0 && pL > 0.0;
#pragma unroll
    for (int i = 0; i < N; i++) same = same && UL[i] == UR[i];
    const double aL = fsqrt(g * pL * il);
    double ro, u, p;
    bool left = true;
    if (__all(same)) {
        ro = UL[0];
        u = uL;
        p = pL;
        lam = R(__builtin_fabs(uL) + aL);
    } else {
        const StarDev st = star_state_dev(g, UL[0], uL, pL, UR[0], uR, pR, aL, il, ir);
        lam = R(same ? __builtin_fabs(uL) + aL : st.smax);
        left = st.vacuum ? (S <= 0.5 * (st.STL + st.STR)) : (st.u >= S);
        // The side of the contact the sample lies on, then one of four cases for that side K:
        // 0 its initial state, 1 its star state, 2 inside its rarefaction fan, 3 vacuum.  The
        // conditions are the reference's with the right side mirrored by sgn = -1 (exact), so one
        // fan evaluation serves both sides.
        const double sgn = left ? 1.0 : -1.0;
        const bool shockK = left ? st.shock_l : st.shock_r;
        const double SK = left ? st.SL : st.SR, SHK = left ? st.SHL : st.SHR, STK = left ? st.STL : st.STR;
        const double rK = left ? UL[0] : UR[0], uK = left ? uL : uR, pK = left ? pL : pR;
        int cs;
        if (shockK && !st.vacuum) cs = (sgn * (SK - S) >= 0.0) ? 0 : 1;
        else if (sgn * (SHK - S) > 0.0) cs = 0;
        else if (sgn * (S - STK) > 0.0) cs = st.vacuum ? 3 : 1;
        else cs = 2;
        if (cs == 0) { ro = rK; u = uK; p = pK; }
        else if (cs == 1) {
            // star density behind a shock (Toro eq. 4.50) or a rarefaction (eq. 4.53)
            const double prK = fdiv(st.p, pK);
            if (shockK) {
                const double C = (g - 1.0) * frcp(g + 1.0);
                ro = fdiv(prK + C, C * prK + 1.0) * rK;
            } else {
                ro = rK * dpow(prK, frcp(g));
            }
            u = st.u;
            p = st.p;
        }
        else if (cs == 3) { ro = 0; u = 0; p = 0; }
        else {
            // inside the fan (Toro eq. 4.56): C^(2/(g-1)) scales the density, and the pressure by
            // C^(2g/(g-1)) = C^(2/(g-1)) C^2
            const double aK = fsqrt(fdiv(g * pK, rK)), igp = frcp(g + 1);
            const double C = igp * (2.0 + sgn * (g - 1) * fdiv(uK - S, aK));
            const double w = dpow(C, 2.0 * frcp(g - 1));
            ro = w * rK;
            u = (sgn * aK + 0.5 * (g - 1) * uK + S) * (2 * igp);
            p = w * C * C * pK;
        }
        ro = same ? UL[0] : ro;
        u = same ? uL : u;
        p = same ? pL : p;
    }
    double Vf[NM];
#pragma unroll
    for (int i = 0; i < NM; i++) Vf[i] = left ? vL[i] : vR[i];
    Vf[D] = Vf[D] + (u - Vf[D]);
    double Fd[N];
    if (ro == 0.0) {
#pragma unroll
        for (int i = 0; i < N; i++) Fd[i] = 0.0;
    } else {
        // the flux of the sampled state (GodunovSolverPerfectGasEOS.h:416-427), with its fused operations
        // written out: the compiler may form it once for each way here, and has to form the same bits
#pragma clang fp contract(off)
        double k = Vf[0] * Vf[0];
#pragma unroll
        for (int i = 1; i < NM; i++) k = __builtin_fma(Vf[i], Vf[i], k);
        const double un = Vf[D];
        Fd[0] = ro * un;
#pragma unroll
        for (int i = 0; i < NM; i++) Fd[1 + i] = i == D ? __builtin_fma(Fd[0], un, p) : Fd[0] * Vf[i];
        Fd[N - 1] = un * __builtin_fma(0.5 * ro, k, __builtin_fma(p, frcp(g - 1.0), p));
    }
#pragma unroll
    for (int i = 0; i < N; i++) F[i] = R(Fd[i]);
}

// Face eigenvalue only (the dt pass needs no flux).
template <int FLUX, int D, typename R, int N>
__device__ inline R face_eigen(R gamma, const R (&UL)[N], const R (&UR)[N]) {
    if constexpr (FLUX == FX_ROE) {
        // |u.n| + c of the Roe average (RoeSolverPerfectGasEOS.h:60-88)
        constexpr int NM = N - 2;
        const R gm1 = gamma - R(1);
        R il = frcp(UL[0]), ir = frcp(UR[0]);
        R vl[NM], vr[NM];
#pragma unroll
        for (int i = 0; i < NM; i++) {
            vl[i] = UL[1 + i] * il;
            vr[i] = UR[1 + i] * ir;
        }
        const R kl = R(0.5) * dot(vl, vl), kr = R(0.5) * dot(vr, vr);
        R hl = (UL[N - 1] * il - kl) * gamma + kl;
        R hr = (UR[N - 1] * ir - kr) * gamma + kr;
        R sl = fsqrt(UL[0]), sr = fsqrt(UR[0]);
        R isum = frcp(sl + sr);
        R ql = sl * isum, qr = sr * isum;
        R v[NM];
#pragma unroll
        for (int i = 0; i < NM; i++) v[i] = ql * vl[i] + qr * vr[i];
        const R vv = dot(v, v), vn = v[D];
        R h = ql * hl + qr * hr;
        R phi2 = R(0.5) * gm1 * vv;
        return __builtin_fabs(vn) + fsqrt(gm1 * h - phi2);
    } else if constexpr (FLUX == FX_HLLC) {
#pragma clang fp contract(off)
        const IdealGasEOS<R> eos(gamma);
        const R il = frcp(UL[0]), ir = frcp(UR[0]);
        const R ul = UL[1 + D] * il, ur = UR[1 + D] * ir;
        const R al = eos.SoundSpeedOfPressure(eos.PressureOfEnergyDensity(internal_energy_along<D>(UL, il, ul)), il);
        const R ar = eos.SoundSpeedOfPressure(eos.PressureOfEnergyDensity(internal_energy_along<D>(UR, ir, ur)), ir);
        return vmax(vabs(vmin(ul - al, ur - ar)), vabs(vmax(ul + al, ur + ar)));
    } else {
        R F[N], lam;
        godunov_flux<D, R>(gamma, UL, UR, F, lam);
        return lam;
    }
}

template <int FLUX, int D, typename R, int N>
__device__ inline void face_flux(R gamma, R eps, const R (&UL)[N], const R (&UR)[N], R (&F)[N],
                                 R& lam) {
    if constexpr (FLUX == FX_ROE) roe_flux<D, R>(gamma, eps, UL, UR, F, lam);
    else if constexpr (FLUX == FX_HLLC) hllc_flux<D, R>(gamma, UL, UR, F, lam);
    else godunov_flux<D, R>(gamma, UL, UR, F, lam);
}

}  // namespace tsd
