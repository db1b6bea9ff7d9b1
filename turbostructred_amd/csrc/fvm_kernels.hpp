// fvm_kernels.hpp -- fused finite-volume stage kernels for gfx950 (1-D and 2-D marching form).
//
// One wavefront owns a strip of 64 columns along x (60 output columns plus a halo of two
// lanes on each side) and marches along y over `ty` output rows.  In 2-D it keeps a three-row
// window of the state, and the values carried from one row to the next, in its own LDS slots
// (no other lane reads them, so there are no barriers), with the next row in flight in
// registers (prefetched one iteration ahead).  In 2-D, x-neighbours are read from the same LDS
// rows at the adjacent lanes (1-D and 3-D use DPP wave shifts); every face flux is evaluated
// once, by the lane on its plus side, and the residual of a cell is accumulated from its x
// faces, then its y faces (ERK:1232,1312) before the stage update is applied and the row is
// stored with coalesced SoA writes.
//
// Modes
//   MODE_DT  spectral radius of every cell from the face eigenvalues, min(V/SR) over the grid
//            (one stored minimum per workgroup); a one-workgroup kernel launched
//            after it turns the minima into dt (ERK:1427-1437).  Used before forward Euler.
//   MODE_S1  U1 = U + dt L(U)          forward Euler (kernel.h:319-331) / SSP stage 1
//   MODE_S2  U2 = 3/4 Un + 1/4 (U1 + dt L(U1))
//   MODE_S3  U  = 1/3 Un + 2/3 (U2 + dt L(U2))   (written in place over Un: Un is read
//            point-wise by the thread that overwrites it)
//   MODE_F1  SSP stage 1 with the dt pass fused in: writes L(Un) = R/V and does the dt
//            reduction of MODE_DT from the same face eigenvalues.
//   MODE_F2  SSP stage 2 reading Un and L(Un): its stencil values are U1 = Un + dt L(Un)
//            formed on the fly, so U1 never goes to HBM.
//   MODE_RN  residual norms sum(V |R|) per variable of UpdateSolution (kernel.h:326) over the
//            interior, writing nothing else: per-block partial sums, and the last block adds
//            them in block order (a deterministic sum).  Launched after the dt pass of every
//            step when the norms are asked for, it runs only in the step that ends the
//            ts_step call (the norms reported), so a call costs one extra residual pass.
#pragma once

#include <type_traits>

#include "fvm_device.hpp"

namespace tsd {

enum : int { MODE_DT = 0, MODE_S1 = 1, MODE_S2 = 2, MODE_S3 = 3, MODE_F1 = 4, MODE_F2 = 5, MODE_RN = 6 };
constexpr int STRIP = 60;   // output columns per wavefront
// Wavefronts (z-planes) per 3-D workgroup; all but two produce output.  In double, whose kernels
// hold 200 to 250 registers, a SIMD takes two.  In float four fit, with a few registers spilled (HLLC: up to 4
// of 128 with Barth-Jespersen and 20 with the other reconstructions; Roe: 25 and 37; the exact solver,
// which works in double, more than a hundred), but stage 2 then spills 15 more of its two
// prefetched rows: three (256^3: 899 us against 1078 with four).
template <typename R, int VIS, int MODE>
constexpr int z_waves = sizeof(R) == 8 ? 8 : (MODE == MODE_F2 ? 12 : 16);
// output planes of stage 2 and of the others (which set the number of dt minima)
constexpr int z_out_of(int real_bytes, bool stage2) { return (real_bytes == 8 ? 8 : stage2 ? 12 : 16) - 2; }
constexpr int MAX_BC = 8;

// Device-resident control block of one solve: the step bookkeeping of StepInfo (kernel.h:56) and
// the termination rule of Kernel::Run (kernel.h:1834-1846), evaluated on the device so that a
// chunk of steps can be issued without host round trips.
struct StepCtl {
    double time, dt, t_max, next_snap;
    long long iter;
    int max_steps, steps_done;
    int active;  // 1 while steps remain to be taken
    int go;      // 1 if the current step runs (set by the dt pass)
    int error;   // 1 = dt not finite and positive
    int out_of_grid;  // set by an upload that finds momentum out of the grid's axes
    double* dt_log;
    long long dt_log_base, dt_log_cap;  // dt of iteration `it` goes to dt_log[it - base]
    double rnorm[5];                    // residual norms of the last step (MODE_RN)
    unsigned int rn_done, pad2;
};

struct GridArgs {
    int nd;
    int n[3];
    int periodic[3];
    const double* h[3];   // cell sizes, ghost layer included (n + 2 entries)
    const double* rc[3];  // 1/(x_{i+1} - x_{i-1}), interior cells
    const double* rl[3];  // 1/(x_i - x_{i-1})
    const double* rr[3];  // 1/(x_{i+1} - x_i)
    const double* ih[3];  // 1/h, ghost layer included
    double eps2;          // Venkatakrishnan eps^2 of every cell (uniform grids)
    // non-uniform grids: eps^2 of cell (i, j, k) = ev[0][i] * ev[1][j] * ev[2][k], the per-axis
    // factors (K h_a)^(3/nd) of (K (hx hy hz)^(1/nd))^3 (Limiters.h:93-96); null when uniform
    const double* ev[3];
    double gamma, eps, cfl;
    BCDev bc[MAX_BC];
    int side_marker[6];
    const uint8_t* face_marker[6];
};

// Viscous terms and body forces (ERK:79-874, kernel.h:941-989), read only by the VIS instances
// of the stage kernels and by the viscous pre-pass.
struct VisArgs {
    const double* x[3];  // cell-centre coordinates, ghost layer included (n + 2 entries)
    double* grad;        // (1-D, 3-D pre-pass) velocity gradients of the interior cells: plane d*nd + e = d vel_d / d x_e
    double* fv[3];       // (1-D, 3-D pre-pass) viscous fluxes of the faces normal to axis a: 4 planes (momentum x, y, z,
                         // energy), faces numbered like cells with n_a + 1 along a
    unsigned nface[3];   // faces normal to axis a (the plane size of fv[a])
    double mu;           // gas viscosity (viscous fluxes and the spectral-radius term)
    double sigma[3];     // potential force (IsExternalForceRequared)
    double accel[3];     // uniform acceleration (IsUnifromAccelerationRequared)
    int viscous, force, accel_on;
    int gate_go;         // pre-pass: runs when the step runs (1) or while steps remain (0)
};

struct KArgs {
    GridArgs g;
    VisArgs v;
    const void* uin;   // stencil input planes (TIn)
    const void* lin;   // L(Un) planes (TOut type), MODE_F2
    const double* un;  // U^n planes (SSP stages 2, 3)
    void* uout;        // output planes (TOut)
    void* dout;        // FP32-residual stage 2: the increment U2 - U^n (float planes), or null
    const void* din;   // FP32-residual stage 3: that increment (float planes), or null
    size_t plane;      // cells per plane
    StepCtl* ctl;
    int ty;            // output rows per tile
    int ty2;           // the same for 3-D fused stage 2, whose workgroups output other planes in float
    int nstrips;       // strips along x
    int ntiles;        // strips * row blocks
    double* rn_part;   // per-block partial residual norms, 5 per block (MODE_RN)
    double* dt_part;   // single solves: each workgroup's minimum of V/SR (dt passes, fused stage 1)
    int dt_minima;     // fused stages 2 and 3: number of those minima where they apply the step's dt
                       // themselves (see step_dt); 0 where dt_finalize_kernel has done it
};

// ---- wave-level helpers -------------------------------------------------------------------------
// lane i receives lane i-1 (wave_shr:1) / lane i+1 (wave_shl:1); the end lanes are halo lanes
// and receive 0 (bound_ctrl), which needs no copy of an "old" value before each move.
__device__ inline double dpp_from_left(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_mov_dpp(lo, 0x138, 0xF, 0xF, true);
    hi = __builtin_amdgcn_mov_dpp(hi, 0x138, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
__device__ inline double dpp_from_right(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_mov_dpp(lo, 0x130, 0xF, 0xF, true);
    hi = __builtin_amdgcn_mov_dpp(hi, 0x130, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
__device__ inline float dpp_from_left(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x138, 0xF, 0xF, true));
}
__device__ inline float dpp_from_right(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x130, 0xF, 0xF, true));
}

// Blocks are dispatched round-robin over the 8 XCDs; give each XCD a contiguous range of
// tiles so that neighbouring tiles (which share halo rows/columns) share an L2.
__device__ inline int xcd_remap(int b, int nb) {
    int q = nb >> 3, r = nb & 7;
    int x = b & 7, l = b >> 3;
    return x * q + (x < r ? x : r) + l;
}

// Map a possibly out-of-range index to its source cell: periodic wrap, or the mirror image
// of the ghost fill (ghost i = -l takes cell l-1, kernel.h:734-735, 751-752).
__device__ inline void map_index(int x, int n, int periodic, int& xs, int& side) {
    side = 0;
    if (periodic) {
        xs = x % n;
        if (xs < 0) xs += n;
        return;
    }
    if (x < 0) {
        xs = -x - 1;
        side = -1;
    } else if (x >= n) {
        xs = 2 * n - 1 - x;
        side = 1;
    } else {
        xs = x;
    }
    xs = xs < 0 ? 0 : (xs >= n ? n - 1 : xs);
}

__device__ inline int bc_marker(const GridArgs& g, int side, int face_index) {
    const uint8_t* fm = g.face_marker[side];
    return fm ? int(fm[face_index]) : g.side_marker[side];
}

// Variable v of an SoA state array at a cell: a wave-uniform 64-bit plane base plus a 32-bit
// per-lane byte offset -- the global load/store form with a scalar base address, so that each
// access needs one VGPR of address and no 64-bit address arithmetic.  A plane stays below
// 4 GiB (checked when a context is created).  (Casting the base to the global address space
// explicitly changed nothing for the 1-D / 2-D stages and made the viscous stages 10-25% slower.)
template <typename T>
__device__ __forceinline__ T ld_plane(const T* base, size_t P, int v, unsigned cell) {
    const char* b = reinterpret_cast<const char*>(base + (size_t)v * P);
    return *reinterpret_cast<const T*>(b + cell * unsigned(sizeof(T)));
}
template <typename T>
__device__ __forceinline__ void st_plane(T* base, size_t P, int v, unsigned cell, T x) {
    char* b = reinterpret_cast<char*>(base + (size_t)v * P);
    *reinterpret_cast<T*>(b + cell * unsigned(sizeof(T))) = x;
}

// The same store with the non-temporal hint, for the 1-D / 2-D stage outputs: each value is
// written once and is next read by the following launch, so keeping it out of the way of the
// stencil rows still being re-read from L2 pays (about 3 % per 2-D step in FP64); the 3-D kernel
// keeps the plain store, which measured faster there.
template <typename T>
__device__ __forceinline__ void st_plane_stream(T* base, size_t P, int v, unsigned cell, T x) {
    char* b = reinterpret_cast<char*>(base + (size_t)v * P);
    __builtin_nontemporal_store(x, reinterpret_cast<T*>(b + cell * unsigned(sizeof(T))));
}

// The batched kernel reads its descriptors, and so every state and geometry pointer, from memory:
// as generic pointers their accesses became flat instructions (which also wait on the scalar
// loads' counter) and the wave-uniform row geometry came from vector loads, whose waits also
// waited for the stencil prefetch.  Its instances (GP) address the state planes and per-lane
// geometry as global memory and the row geometry, read-only for the whole run, as constant
// memory (scalar loads).  The single-solve kernels take their pointers from kernel arguments,
// where the compiler infers as much, and keep the generic forms (the explicit casts slowed the
// viscous stages).
#define TS_AS_GLOBAL __attribute__((address_space(1)))
#define TS_AS_CONST __attribute__((address_space(4)))
template <bool GP, typename T>
__device__ __forceinline__ T ld_state(const T* base, size_t P, int v, unsigned cell) {
    if constexpr (GP) {
        const TS_AS_GLOBAL char* b = (const TS_AS_GLOBAL char*)(base + (size_t)v * P);
        return *(const TS_AS_GLOBAL T*)(b + cell * unsigned(sizeof(T)));
    } else {
        return ld_plane(base, P, v, cell);
    }
}
template <bool GP, typename T>
__device__ __forceinline__ void st_state_stream(T* base, size_t P, int v, unsigned cell, T x) {
    if constexpr (GP) {
        TS_AS_GLOBAL char* b = (TS_AS_GLOBAL char*)(base + (size_t)v * P);
        __builtin_nontemporal_store(x, (TS_AS_GLOBAL T*)(b + cell * unsigned(sizeof(T))));
    } else {
        st_plane_stream(base, P, v, cell, x);
    }
}
// per-lane geometry
template <bool GP, typename T>
__device__ __forceinline__ T ld_geo(const T* p, int i) {
    if constexpr (GP) return ((const TS_AS_GLOBAL T*)p)[i];
    else return p[i];
}
// wave-uniform geometry (row sizes and slope factors)
template <bool GP, typename T>
__device__ __forceinline__ T ld_geo_uniform(const T* p, int i) {
    if constexpr (GP) return ((const TS_AS_CONST T*)p)[i];
    else return p[i];
}


// V/SR of one cell; a NaN or negative spectral radius (non-physical state) becomes 0 so that
// the step fails with dt = 0 instead of silently skipping the cell in the minimum.  A cell whose
// spectral radius is zero (or below the reciprocal's range) bounds nothing.
__device__ inline double dt_candidate(double vol, double sr) {
    const double q = (sr >= 0.0 && sr < 1e-290) ? __builtin_inf() : fdiv(vol, sr);
    return (q > 0.0) ? q : 0.0;
}

// dt = min(V/SR) * CFL (ERK:1430) from the grid minimum mn, clamped to the next snapshot
// (ERK:1433); false where it is not finite and positive
__device__ inline bool dt_rule(const StepCtl* ctl, double cfl, double mn, double& dtn) {
    dtn = mn * cfl;
    const double t0 = ctl->time;
    if (ctl->next_snap > 0 && ctl->next_snap < t0 + dtn) dtn = ctl->next_snap - t0;
    return dtn > 0.0 && dtn < __builtin_inf();
}
__device__ inline void step_fails(StepCtl* ctl) {
    ctl->error = 1;
    ctl->go = 0;
    ctl->active = 0;
}
// advances Time / Iteration, logs dt and evaluates the stop rule of Kernel::Run
// (kernel.h:1834-1846).  One thread.
__device__ inline void step_advances(StepCtl* ctl, double dtn) {
    const double t1 = ctl->time + dtn;
    ctl->time = t1;
    long long it = ctl->iter;
    ctl->iter = it + 1;
    int sd = ctl->steps_done + 1;
    ctl->steps_done = sd;
    long long li = it - ctl->dt_log_base;
    if (ctl->dt_log && li >= 0 && li < ctl->dt_log_cap) ctl->dt_log[li] = dtn;
    bool stop = (t1 >= ctl->t_max) || (ctl->next_snap > 0 && t1 == ctl->next_snap) || (sd >= ctl->max_steps);
    ctl->active = stop ? 0 : 1;
}
// the step's dt from the grid minimum.  One thread.
__device__ inline void dt_apply(StepCtl* ctl, double cfl, double mn) {
    double dtn;
    if (!dt_rule(ctl, cfl, mn, dtn)) {
        step_fails(ctl);
        return;
    }
    ctl->dt = dtn;
    ctl->go = 1;
    step_advances(ctl, dtn);
}

// minimum over the wavefront, in lane 63 (row shifts, then row broadcasts)
__device__ inline double wave_min_lane63(double v) {
#define TS_MIN_STEP(ctrl)                                                              \
    {                                                                                  \
        const int lo = __double2loint(v), hi = __double2hiint(v);                      \
        v = __builtin_fmin(v, __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, ctrl, 0xF, 0xF, false), \
                                               __builtin_amdgcn_update_dpp(lo, lo, ctrl, 0xF, 0xF, false))); \
    }
    TS_MIN_STEP(0x111) TS_MIN_STEP(0x112) TS_MIN_STEP(0x114) TS_MIN_STEP(0x118)  // row_shr 1, 2, 4, 8
    TS_MIN_STEP(0x142) TS_MIN_STEP(0x143)                                        // row_bcast 15, 31
#undef TS_MIN_STEP
    return v;
}
// the same lane's value in every lane
__device__ inline double read_lane63(double v) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63), __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// A launch between stage 1 and stage 2 for one reduction costs 4 to 5 us, a tenth of the step of a
// small grid.  Where the minima are few, every wavefront of stage 2 reduces them itself and so
// knows the step's dt (the minimum is exact: all get the same); `first` marks the one that writes
// what stage 3 reads, dt and go.  Time, the step count and the stop rule, which the other wavefronts
// of stage 2 still read, are advanced by stage 3.  False where the step does not run.
__device__ inline bool step_dt(StepCtl* ctl, double cfl, const double* part, int n, int lane, bool first, double& dt) {
    // up to 640 minima in one round trip to memory, and 576 more in each further one: all loads of a trip
    // are in flight together (one load at a time, 385 minima took most of what the launch does)
    double m = part[lane < n ? lane : n - 1];
    for (int i = 64; i < n; i += 576) {
        double q[9];
#pragma unroll
        for (int k = 0; k < 9; k++) {
            const int j = i + 64 * k + lane;
            q[k] = part[j < n ? j : n - 1];
        }
#pragma unroll
        for (int k = 0; k < 9; k++) m = __builtin_fmin(m, q[k]);
    }
    if (!ctl->active) return false;  // stage 1 has cleared go
    m = read_lane63(wave_min_lane63(m));
    const bool ok = dt_rule(ctl, cfl, m, dt);
    if (first && lane == 0) {
        if (ok) {
            ctl->dt = dt;
            ctl->go = 1;
        } else {
            step_fails(ctl);
        }
    }
    return ok;
}

// Single solves: the step's dt from the `n` per-workgroup minima of V/SR that a dt pass or fused
// stage 1 stored, launched right after it.  Plain stores and one workgroup's reduction instead of
// one same-address atomic per wavefront: those serialise where the wavefronts finish together,
// at the end of the launch (a 1-D stage 1 with 70k strips spent most of its time in them).  The
// minimum is exact, so its order does not matter.  Skipped when no step is running.  (A template
// only so that the translation units including this header share one definition.)
template <int = 0>
__global__ void __launch_bounds__(1024) dt_finalize_kernel(StepCtl* ctl, double cfl, const double* part, int n) {
    if (!ctl->active) return;  // the same for every thread: before the barrier
    double m = __builtin_inf();
    for (int i = threadIdx.x; i < n; i += blockDim.x) m = __builtin_fmin(m, part[i]);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = __builtin_fmin(m, __shfl_xor(m, o));
    __shared__ double red[16];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (unsigned w = 1; w < (blockDim.x >> 6); w++) m = __builtin_fmin(m, red[w]);
        dt_apply(ctl, cfl, m);
    }
}

// Batched solves whose stage 2 does not do it (2-D, and 1-D of many work items): the dt of each from its
// work items' minima of V/SR, which fused stage 1 stored by table entry (a solve's entries are
// contiguous: `ranges` holds the descriptor slot, first entry and count of each such member).  One wavefront per member, launched
// right after stage 1; skipped for a solve whose run has ended.  Per-item atomics on the solve's
// control block serialised on a lone large solve (2 x 3000 same-address atomics per stage 1 at
// 2048^2), and their ordering needed either a fence, which writes back the L2, or waiting for a
// returned value.
template <int = 0>
__global__ void __launch_bounds__(256) dt_finalize_batched(const KArgs* __restrict__ descs, const int4* __restrict__ ranges,
                                                           const int* __restrict__ nmem_p, const double* __restrict__ part) {
    const int lane = threadIdx.x & 63;
    const int nm = __builtin_amdgcn_readfirstlane(*nmem_p);
    const int stride = gridDim.x * (blockDim.x >> 6);
    for (int i = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)); i < nm; i += stride) {
        const int4 r = ranges[i];  // slot, first entry, entries
        const KArgs& a = descs[r.x];
        StepCtl* ctl = a.ctl;
        if (!ctl->active) continue;
        double m = __builtin_inf();
        for (int j = lane; j < r.z; j += 64) m = __builtin_fmin(m, part[r.y + j]);
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) m = __builtin_fmin(m, __shfl_xor(m, o));
        if (lane == 0) dt_apply(ctl, a.g.cfl, m);
    }
}

// Block sum of the per-lane residual norms (wave shuffle tree, then the waves in order), one
// partial per block, and the last block to finish adds the partials in block order.
__device__ inline void rn_reduce_finalize(StepCtl* ctl, double* part, const double (&rn)[NV], double* red,
                                          int lane, int wave, int nwaves) {
#pragma unroll
    for (int v = 0; v < NV; v++) {
        double x = rn[v];
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) x += __shfl_xor(x, o);
        if (lane == 0) red[wave * NV + v] = x;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int v = 0; v < NV; v++) {
            double x = red[v];
            for (int w = 1; w < nwaves; w++) x += red[w * NV + v];
            part[(size_t)blockIdx.x * NV + v] = x;
        }
        __threadfence();
        unsigned prev = atomicAdd(&ctl->rn_done, 1u);
        if (prev == gridDim.x - 1) {
            __threadfence();
            for (int v = 0; v < NV; v++) {
                double x = 0.0;
                for (unsigned b = 0; b < gridDim.x; b++) x += part[(size_t)b * NV + v];
                ctl->rnorm[v] = x;
            }
            atomicExch(&ctl->rn_done, 0u);
        }
    }
}

template <int MODE> struct ModeTraits {
    static constexpr bool sr = MODE == MODE_DT || MODE == MODE_F1;  // needs V/SR and dt
    static constexpr bool flux = MODE != MODE_DT;                    // needs fluxes
    static constexpr bool use_un = MODE == MODE_S2 || MODE == MODE_S3 || MODE == MODE_F2;
    static constexpr double ca = (MODE == MODE_S3) ? 1.0 / 3.0 : 0.75;
    static constexpr double cb = (MODE == MODE_S3) ? 2.0 / 3.0 : 0.25;
};

// ---- one tile of the 1-D / 2-D stage: a strip of 60 columns marching over ty rows ----------------
// block_min receives the tile's min(V/SR) (sr modes).  `tile` < 0 marks a wavefront without work
// that still has to take part in a block reduction.
// max(4/(3 rho_f), gamma/rho_f) mu fS^2 / V: the viscous part of a cell's spectral radius from
// one face, rho_f = sqrt(rho_L rho_R) of the face states (ERK:1239-1248)
__device__ inline double viscous_sr(double rho_l, double rho_r, double gamma, double mu, double fS, double vol) {
    const double k = (4.0 / 3.0 < gamma) ? gamma : 4.0 / 3.0;
    return fdiv(k * mu * (fS * fS), fsqrt(rho_l * rho_r) * vol);
}

// Differences of fluxes, with every flux (and its product with a face's area) rounded to R first.  Left to
// itself the compiler fuses the product that a flux ends in into the subtraction: one side is then rounded
// and the other is not, equal fluxes leave half an ulp of theirs, always of the same sign, and what one cell
// gains its neighbour does not lose.  (A uniform FP32 flow drifted, and the density of a 2048^2
// run with the FP32 residual was off by 1.1e-8 in L1 after 20 steps; now 1.5e-10.)  The rounded values are
// needed anyway, for the neighbour or for the next row: 512^2 to 2048^2 take the same time either way.
template <typename R>
__device__ __forceinline__ R flux_difference(R plus, R minus) {
#pragma clang fp contract(off)
    return plus - minus;
}
template <typename R>
__device__ __forceinline__ R through(R flux, R area) {
#pragma clang fp contract(off)
    return flux * area;
}

// residual += force and acceleration sources of a cell (kernel.h:941-989)
template <typename R, int N>
__device__ inline void add_sources(const VisArgs& v, const R (&u)[N], double vol, R (&res)[N]) {
    const double ro = double(u[0]);
    double vel[N - 2];
#pragma unroll
    for (int i = 0; i < N - 2; i++) vel[i] = double(u[1 + i]) / ro;
    if (v.force) {
        double w = 0.0;
#pragma unroll
        for (int i = 0; i < N - 2; i++) {
            res[1 + i] = R(double(res[1 + i]) + vol * v.sigma[i]);
            w += v.sigma[i] * vel[i];
        }
        res[N - 1] = R(double(res[N - 1]) + w * vol);
    }
    if (v.accel_on) {
        double w = 0.0;
#pragma unroll
        for (int i = 0; i < N - 2; i++) {
            res[1 + i] = R(double(res[1 + i]) + ro * vol * v.accel[i]);
            w += ro * v.accel[i] * vel[i];
        }
        res[N - 1] = R(double(res[N - 1]) + w * vol);
    }
}

// ---- viscous face fluxes of the 2-D stage ------------------------------------------------------
// Flux of x momentum, y momentum, (z momentum) and energy through a face normal to axis D
// (ComputeViscousFluxes, ERK:668-874): normal derivatives from the two cell velocities vl, vr,
// tangential ones tan[] (of the first two components) already weighted, l = h_L / dx and r = h_R / dx.
template <int D, int NM>
__device__ __forceinline__ void vis_flux2(double mu, double idx, double l, double r, const double (&vl)[NM], const double (&vr)[NM],
                                          const double (&tan)[2], double (&t)[NM + 1]) {
    constexpr int T = 1 - D;
    double dn[NM];
#pragma unroll
    for (int d = 0; d < NM; d++) dn[d] = (vr[d] - vl[d]) * idx;
    t[D] = mu * ((-2.0 / 3.0) * (dn[D] + tan[T]) + 2.0 * dn[D]);
    t[T] = mu * (dn[T] + tan[D]);
    if constexpr (NM == 3) t[2] = mu * dn[2];
    double e = 0.0;
#pragma unroll
    for (int d = 0; d < NM; d++) e += 0.5 * (l * vr[d] + r * vl[d]) * t[d];
    t[NM] = e;
}

// Tangential derivative of the dummy cell across a boundary face (ComputeDummyCellGradients, ERK:303-665,
// GradientComputer.h:19-53): 2 g_face - g_in, with g_face the least-squares gradient at the face centre
// over the boundary cell, its two transverse neighbours and the dummy cell, anchored at the
// face value; solved from the 2 x 2 normal equations.  rn, rd: distances along the normal from
// the boundary cell and from the dummy cell to the face centre; rp, rm: along the face from the
// transverse neighbours.
struct FaceLsq {
    double rn, rd, rp, rm;
    __device__ __forceinline__ double operator()(double face, double in, double plus, double minus, double dummy, double g_in) const {
        const double mnn = 3.0 * rn * rn + rd * rd, mnt = rn * (rp + rm), mtt = rp * rp + rm * rm;
        const double dp = face - plus, dm = face - minus;
        const double bn = rn * ((face - in) + dp + dm) + rd * (face - dummy), bt = rp * dp + rm * dm;
        return 2.0 * fdiv(mnn * bt - mnt * bn, mnn * mtt - mnt * mnt) - g_in;
    }
};

// VIS instances (FP64) subtract the viscous face fluxes from the convective ones before these are
// differenced (ERK:1221-1222), add the viscous spectral-radius term after each plus face's eigenvalue,
// and the body-force sources after the flux sweeps.  1-D takes the viscous fluxes from the pre-pass.
// 2-D forms them here, from the velocities of the window that the march holds anyway: a lane keeps those
// of its column in three rows and takes its x neighbours' by lane shifts, a dummy cell's gradient is
// formed by the lane of its face.  (A pre-pass of three launches wrote 6 gradients per cell and 8
// values per cell for the faces, and the stages read the latter back: 72 us of a 164 us forward-Euler
// step at 1024^2.  The stage costs as much as it did with those reads, 54 us, so the step is at 87 us, of
// which leaving out the momentum out of the plane is 7; it is bound by VALU issue.)
// DT_ARG instances take the step's dt from `dt_arg` instead of the control block in memory.
template <int DIM, int RECON, int LIM, int FLUX, int MODE, typename R, typename TIn, typename TOut, int N = NV,
          int VIS = 0, bool DT_ARG = false, bool GP = false>
__device__ __forceinline__ void stage_tile(const KArgs& a, int tile, int lane, double& block_min,
                                           double* rn = nullptr, double dt_arg = 0.0) {
    using MT = ModeTraits<MODE>;
    constexpr bool VIN = VIS != 0 && DIM == 2 && MT::flux;  // viscous fluxes formed here
    constexpr int NM = N - 2;                               // velocity components
    const GridArgs& g = a.g;
    const StepCtl* ctl = a.ctl;
    const bool tile_ok = tile >= 0 && tile < a.ntiles;
    const int strip = tile_ok ? tile % a.nstrips : 0;
    const int yb = tile_ok ? tile / a.nstrips : 0;

    const int nx = g.n[0];
    const int ny = (DIM > 1) ? g.n[1] : 1;
    const int xg = strip * STRIP - 2 + lane;
    int xs, xside;
    map_index(xg, nx, g.periodic[0], xs, xside);
    const bool out_lane = tile_ok && lane >= 2 && lane < 2 + STRIP && xg < nx;
    // lane holding the right ghost column: its minus-face flux is the right boundary face
    const bool ghost_x_lane = tile_ok && xg == nx && lane >= 2 && lane <= 62;

    const R gamma = R(g.gamma), eps = R(g.eps);
    const double dt = MT::sr ? 0.0 : (DT_ARG ? dt_arg : ctl->dt);

    CellGeo<DIM, R> geo;
    const double hx = ld_geo<GP>(g.h[0], xs + 1);
    const double ihx = ld_geo<GP>(g.ih[0], xs + 1);
    geo.hh[0] = R(0.5 * hx);
    geo.rc[0] = R(ld_geo<GP>(g.rc[0], xs));
    geo.rl[0] = R(ld_geo<GP>(g.rl[0], xs));
    geo.rr[0] = R(ld_geo<GP>(g.rr[0], xs));
    geo.eps2 = R(g.eps2);
    constexpr bool VENKAT = RECON == RC_LINLIM && LIM == LIM_VENKAT;
    // per-cell eps^2 on non-uniform grids (a wave-uniform branch, Venkatakrishnan instances only)
    const bool ev_cells = VENKAT && g.ev[0] != nullptr;
    const double ev_x = ev_cells ? ld_geo<GP>(g.ev[0], xs) : 0.0;
    if (ev_cells && DIM == 1) geo.eps2 = R(ev_x);

    const TIn* __restrict__ uin = (const TIn*)a.uin;
    const TOut* __restrict__ lin = (const TOut*)a.lin;
    TOut* uo = (TOut*)a.uout;
    const size_t P = a.plane;
    auto store = [&](int v, unsigned off, TOut x) {
        st_state_stream<GP>(uo, P, v, off, x);
    };

    // One stencil value, the input state at a (possibly ghost) cell of row r, in two steps: the
    // loads (issue_row), and the value formed from them with its ghost image (complete_row).  The
    // prefetched row is completed one iteration after its loads are issued, so that no arithmetic
    // on the loaded values (stage 2's U^n + dt L, a ghost image) makes the wavefront wait for them
    // early.
    struct RawRow {
        TIn u[N];
        TOut l[MODE == MODE_F2 ? N : 1];
        int rs, yside;
    };
    auto issue_row = [&](int r, RawRow& q) {
        int rs = 0, yside = 0;
        if constexpr (DIM > 1) map_index(r, ny, g.periodic[1], rs, yside);
        q.rs = rs;
        q.yside = yside;
        const unsigned off = unsigned(rs) * unsigned(nx) + unsigned(xs);
#pragma unroll
        for (int v = 0; v < N; v++) q.u[v] = ld_state<GP>(uin, P, plane_of<N>(v), off);
        if constexpr (MODE == MODE_F2) {
#pragma unroll
            for (int v = 0; v < N; v++) q.l[v] = ld_state<GP>(lin, P, plane_of<N>(v), off);
        }
    };
    auto complete_row = [&](const RawRow& q, R (&u)[N]) {
        if constexpr (MODE == MODE_F2) {
#pragma unroll
            for (int v = 0; v < N; v++) u[v] = R(double(q.u[v]) + dt * double(q.l[v]));
        } else {
#pragma unroll
            for (int v = 0; v < N; v++) u[v] = R(q.u[v]);
        }
        if (xside != 0) {
            // one branch per side, so that the side (and, along a row, the condition) is
            // wave-uniform and its data come from scalar loads
            R t[N];
            if (xside < 0) bc_image(g.bc[bc_marker(g, 0, q.rs)], gamma, 0, u, t);
            else bc_image(g.bc[bc_marker(g, 1, q.rs)], gamma, 0, u, t);
#pragma unroll
            for (int v = 0; v < N; v++) u[v] = t[v];
        } else if (q.yside != 0) {
            R t[N];
            bc_image(g.bc[bc_marker(g, q.yside < 0 ? 2 : 3, xs)], gamma, 1, u, t);
#pragma unroll
            for (int v = 0; v < N; v++) u[v] = t[v];
        }
    };
    auto load_row = [&](int r, R (&u)[N]) {
        RawRow q;
        issue_row(r, q);
        complete_row(q, u);
    };

    // FP32-residual SSP stages with the state kept in double: stage 2 also writes the increment
    // D = U2 - U^n = dt/4 (L(U^n) + L(U1)), and stage 3 forms U^{n+1} = U^n + 2/3 (D + dt L(U2))
    // from it, so U^n is never rounded to float.  The centre value of L(U^n) (stage 2) or of D
    // (stage 3) is loaded with the centre U^n, ahead of the finalize that uses it.
    constexpr bool INC_F2 = MODE == MODE_F2 && sizeof(TOut) == 4, INC_S3 = MODE == MODE_S3 && sizeof(TIn) == 4;
    const bool inc = (INC_F2 && a.dout != nullptr) || (INC_S3 && a.din != nullptr);
    using IncT = typename std::conditional<MODE == MODE_F2, TOut, TIn>::type;
    const IncT* incsrc = (MODE == MODE_F2) ? (const IncT*)a.lin : (const IncT*)a.din;
    auto load_inc = [&](unsigned off, IncT (&d)[N]) {
        if (inc) {
#pragma unroll
            for (int v = 0; v < N; v++) d[v] = ld_state<GP>(incsrc, P, plane_of<N>(v), off);
        }
    };

    // write the result for a finalized cell: the stage update, or L = R/V (MODE_F1)
    auto finish = [&](unsigned off, const R (&u)[N], const R (&res0)[N], const double (&un)[N],
                      const IncT (&dc)[N], double ivol, double vol) {
        R res[N];
#pragma unroll
        for (int v = 0; v < N; v++) res[v] = res0[v];
        if constexpr (VIS) add_sources(a.v, u, vol, res);
#pragma unroll
        for (int v = 0; v < N; v++) {
            if constexpr (MODE == MODE_RN) {
                if (out_lane) rn[v] += vol * __builtin_fabs(double(res[v]));
            } else if constexpr (MODE == MODE_F1) {
                if (out_lane) store(plane_of<N>(v), off, TOut(double(res[v]) * ivol));
            } else {
                if (inc && MODE == MODE_F2) {
                    const double d = 0.25 * dt * (double(dc[v]) + double(res[v]) * ivol);
                    if (out_lane) {
                        st_state_stream<GP>((TOut*)a.dout, P, plane_of<N>(v), off, TOut(d));
                        store(plane_of<N>(v), off, TOut(un[v] + d));
                    }
                } else if (inc && MODE == MODE_S3) {
                    const double d = double(dc[v]);
                    const double q = un[v] + (2.0 / 3.0) * (d + dt * (double(res[v]) * ivol));
                    if (out_lane) store(plane_of<N>(v), off, TOut(q));
                } else {
                    double q = double(u[v]) + dt * (double(res[v]) * ivol);
                    if constexpr (MT::use_un) q = MT::ca * un[v] + MT::cb * q;
                    if (out_lane) store(plane_of<N>(v), off, TOut(q));
                }
            }
        }
    };


    if constexpr (DIM == 1) {
        // ---- one row ----
        R c[N], nb[2][N], face[2][N];
        load_row(0, c);
        double un[N];
#pragma unroll
        for (int v = 0; v < N; v++) un[v] = MT::use_un ? ld_state<GP>(a.un, P, plane_of<N>(v), unsigned(xs)) : 0.0;
        IncT dc[N];
        load_inc(unsigned(xs), dc);
#pragma unroll
        for (int v = 0; v < N; v++) {
            nb[0][v] = dpp_from_left(c[v]);
            nb[1][v] = dpp_from_right(c[v]);
        }
        reconstruct<1, RECON, LIM, R, FLUX != FX_ROE>(c, nb, geo, face);
        R UL[N], UR[N];
#pragma unroll
        for (int v = 0; v < N; v++) {
            UL[v] = dpp_from_left(face[1][v]);
            UR[v] = face[0][v];
        }
        // the end lanes lack a neighbour (the fluxes of lanes 0, 1 and 63 are not used): nothing in them
        // may keep the exact solver from finding the strip constant
        if (FLUX == FX_GODUNOV && (lane < 2 || lane == 63)) {
#pragma unroll
            for (int v = 0; v < N; v++) UL[v] = UR[v];
        }
        if (!g.periodic[0]) {
            if (xg == 0) bc_image(g.bc[bc_marker(g, 0, 0)], gamma, 0, UR, UL);
            if (xg == nx) bc_image(g.bc[bc_marker(g, 1, 0)], gamma, 0, UL, UR);
        }
        const R Sx = R(1);
        R lam;
        R F[N];
        if constexpr (MT::flux) face_flux<FLUX, 0, R>(gamma, eps, UL, UR, F, lam);
        else lam = face_eigen<FLUX, 0, R>(gamma, UL, UR);
        if constexpr (VIS && MT::flux) {
            if (a.v.viscous) {
                const unsigned fi = unsigned(xg < 0 ? 0 : (xg > nx ? nx : xg));
#pragma unroll
                for (int v = 1; v < N; v++) F[v] -= R(ld_plane(a.v.fv[0], a.v.nface[0], v - 1, fi));
            }
        }
        if constexpr (MT::sr) {
            R lam_r = dpp_from_right(lam);
            double sr;
            {
#pragma clang fp contract(off)
                sr = double(Sx * lam) + double(Sx * lam_r);
            }
            if constexpr (VIS) {
                const double rl = dpp_from_right(double(UL[0])), rr = dpp_from_right(double(UR[0]));
                sr = sr + viscous_sr(rl, rr, g.gamma, a.v.mu, double(Sx), hx);
            }
            if (out_lane) block_min = dt_candidate(hx, sr);
            if (ghost_x_lane) block_min = __builtin_fmin(block_min, dt_candidate(ld_geo_uniform<GP>(g.h[0], nx + 1), double(Sx * lam)));
        }
        if constexpr (MT::flux) {
            R res[N];
#pragma unroll
            for (int v = 0; v < N; v++) {
                res[v] = -(flux_difference(dpp_from_right(F[v]), F[v]) * Sx);
            }
            finish(unsigned(xs), c, res, un, dc, ihx, hx);
        }
    } else {
        // ---- march along y ----
        const int y0 = yb * a.ty;
        const int yend = (y0 + a.ty < ny) ? y0 + a.ty : ny;
        RawRow Pn;              // prefetched stencil row (completed and entered into the window one
                                // iteration later)
        double Nc[N];          // U^n of the row finalized in this iteration (SSP stages 2, 3)
        IncT Dc[N];            // its L(U^n) or increment (FP32-residual stages 2, 3)
        R ytop[N];             // +y face state of the previously reconstructed row
        // The three-row window (rows rc-1, rc, rc+1) and the values carried to the next row live
        // in LDS, one set per wavefront; no other lane reads them, so no barrier is needed.  The
        // window rotates by slot index instead of register moves, and out of the register file
        // these 20 doubles per lane (40 KB per 4-wavefront block in FP64) leave the occupancy to
        // the register count.
        __shared__ R ring[4][3][N][64];  // [wavefront][slot][variable][lane]
        // residual carried to the pending row: its x part plus S_y times the y-flux through its
        // bottom face; the finalize subtracts S_y times the flux through its top face
        __shared__ R carry[4][N][64];
        const int wl = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
        R (&cy)[N][64] = carry[wl];
        int sm = 0, s0 = 1, sp = 2;  // slots of rows rc-1, rc, rc+1
        // x-neighbours are read from the same LDS rows at lane -+ 1 (the end lanes, halo lanes
        // whose results are discarded, read themselves): LDS reads instead of VALU lane shifts
        const int lm = lane > 0 ? lane - 1 : 0, lp = lane < 63 ? lane + 1 : 63;
        // velocities of this lane's column in rows rc-1, rc, rc+1; x derivatives of the first two of them
        // in rows rc-1 and rc, y derivatives in row rc; of the face on the minus x side: 1/dx and the
        // weights h_L/dx, h_R/dx
        const bool vin = VIN && a.v.viscous;
        double vm[NM], v0[NM], vp[NM], gxm[2], gx[2], gy[2], vdx = 0.0, vhl = 0.0, vhr = 0.0;
        if constexpr (VIN) {
            if (vin) {
                const int f = xg < 0 ? 0 : (xg > nx ? nx : xg);
                vdx = fdiv(1.0, a.v.x[0][f + 1] - a.v.x[0][f]);
                vhl = g.h[0][f] * vdx;
                vhr = g.h[0][f + 1] * vdx;
            }
        }
        auto velocity = [&](const R (&u)[N], double (&vel)[NM]) {
            const double ir = frcp(double(u[0]));
#pragma unroll
            for (int d = 0; d < NM; d++) vel[d] = double(u[1 + d]) * ir;
        };
        double srp = 0.0;       // spectral radius of the pending row without its top face
        R lam_gb = R(0);
        {
            R t0[N], t1[N];
            load_row(y0 - 2, t0);
            load_row(y0 - 1, t1);
#pragma unroll
            for (int v = 0; v < N; v++) {
                ring[wl][sm][v][lane] = t0[v];
                ring[wl][s0][v][lane] = t1[v];
            }
            if constexpr (VIN) {
                if (vin) {
                    velocity(t0, vm);
                    velocity(t1, v0);
                }
            }
        }
        issue_row(y0, Pn);
#pragma unroll
        for (int v = 0; v < N; v++) Nc[v] = 0.0;
        const int nit = yend - y0 + 2;
        for (int t = 0; t < nit; t++) {
            const int rc = y0 - 1 + t;  // row being reconstructed
            {
                R un1[N];
                complete_row(Pn, un1);
#pragma unroll
                for (int v = 0; v < N; v++) ring[wl][sp][v][lane] = un1[v];
                if constexpr (VIN) {
                    if (vin) velocity(un1, vp);
                }
            }
            if (t + 1 < nit) issue_row(rc + 2, Pn);
            if constexpr (MT::use_un) {
                // U^n of the row finalized below, loaded now: the reconstruction and the y-face
                // flux cover its latency (it was read three iterations ago as a stencil row, so
                // it is normally an L2 hit), and only one buffer is live
                if (t >= 2) {
                    const unsigned offn = unsigned(rc - 1) * unsigned(nx) + unsigned(xs);
#pragma unroll
                    for (int v = 0; v < N; v++) Nc[v] = ld_state<GP>(a.un, P, plane_of<N>(v), offn);
                    load_inc(offn, Dc);
                }
            }
            int rcs, rcside;
            map_index(rc, ny, g.periodic[1], rcs, rcside);
            const double hy = ld_geo_uniform<GP>(g.h[1], rcs + 1);
            geo.hh[1] = R(0.5 * hy);
            geo.rc[1] = R(ld_geo_uniform<GP>(g.rc[1], rcs));
            geo.rl[1] = R(ld_geo_uniform<GP>(g.rl[1], rcs));
            geo.rr[1] = R(ld_geo_uniform<GP>(g.rr[1], rcs));
            if (ev_cells) geo.eps2 = R(ev_x * ld_geo_uniform<GP>(g.ev[1], rcs));
            if constexpr (VIN) {
                if (vin) {
#pragma unroll
                    for (int d = 0; d < 2; d++) {
                        gx[d] = (dpp_from_right(v0[d]) - dpp_from_left(v0[d])) * double(geo.rc[0]);
                        gy[d] = (vp[d] - vm[d]) * double(geo.rc[1]);
                    }
                }
            }
            R nb[4][N], face[4][N];
            {
                R U0[N];
#pragma unroll
                for (int v = 0; v < N; v++) {
                    U0[v] = ring[wl][s0][v][lane];
                    nb[0][v] = ring[wl][s0][v][lm];
                    nb[1][v] = ring[wl][s0][v][lp];
                    nb[2][v] = ring[wl][sm][v][lane];
                    nb[3][v] = ring[wl][sp][v][lane];
                }
                reconstruct<2, RECON, LIM, R, FLUX != FX_ROE>(U0, nb, geo, face);
            }
            if (t >= 1) {
                // face between rows rc-1 and rc
                R GL[N], GR[N];
#pragma unroll
                for (int v = 0; v < N; v++) { GL[v] = ytop[v]; GR[v] = face[2][v]; }
                if (!g.periodic[1]) {
                    if (rc == 0) bc_image(g.bc[bc_marker(g, 2, xs)], gamma, 1, GR, GL);
                    if (rc == ny) bc_image(g.bc[bc_marker(g, 3, xs)], gamma, 1, GL, GR);
                }
                const R Sy = R(hx);  // face area of a y-face (ERK:1268)
                R G[N], lam;
                if constexpr (MT::flux) face_flux<FLUX, 1, R>(gamma, eps, GL, GR, G, lam);
                else lam = face_eigen<FLUX, 1, R>(gamma, GL, GR);
                if constexpr (VIN) {
                    if (vin) {
                        const double yl = a.v.x[1][rc], yr = a.v.x[1][rc + 1], hl = g.h[1][rc], hr = g.h[1][rc + 1];
                        const double idy = fdiv(1.0, yr - yl), l = hl * idy, r = hr * idy;
                        double gl[2] = {gxm[0], gxm[1]}, gr[2] = {gx[0], gx[1]};
                        if (!g.periodic[1] && (rc == 0 || rc == ny)) {
                            // the dummy cell is below (rc = 0) or above the face, the boundary cell on the
                            // other side
                            const bool below = rc == 0;
                            const int si = below ? s0 : sm, sd = below ? sm : s0;
                            const double yf = below ? yr - 0.5 * hr : yl + 0.5 * hl;
                            const double xc = a.v.x[0][xs + 1];
                            const FaceLsq lsq{yf - (below ? yr : yl), yf - (below ? yl : yr), xc - a.v.x[0][xs + 2], xc - a.v.x[0][xs]};
                            const double ir = frcp(0.5 * double(ring[wl][si][0][lane] + ring[wl][sd][0][lane]));
#pragma unroll
                            for (int d = 0; d < 2; d++) {
                                const double in = below ? v0[d] : vm[d], dummy = below ? vm[d] : v0[d];
                                const double face = 0.5 * double(ring[wl][si][1 + d][lane] + ring[wl][sd][1 + d][lane]) * ir;
                                const double g_in = below ? gx[d] : gxm[d];
                                const double gd = lsq(face, in, dpp_from_right(in), dpp_from_left(in), dummy, g_in);
                                if (below) gl[d] = gd;
                                else gr[d] = gd;
                            }
                        }
                        const double tan[2] = {0.5 * (r * gl[0] + l * gr[0]), 0.5 * (r * gl[1] + l * gr[1])};
                        double tv[NM + 1];
                        vis_flux2<1, NM>(a.v.mu, idy, l, r, vm, v0, tan, tv);
#pragma unroll
                        for (int v = 1; v < N; v++) G[v] -= R(tv[v - 1]);
                    }
                }
                if constexpr (MT::sr) {
                    if (t >= 2) {
                        double sr;
                        {
#pragma clang fp contract(off)
                            sr = srp + double(Sy * lam);
                        }
                        if constexpr (VIS)
                            sr = sr + viscous_sr(double(GL[0]), double(GR[0]), g.gamma, a.v.mu, double(Sy), hx * g.h[1][rc]);
                        if (out_lane) block_min = __builtin_fmin(block_min, dt_candidate(hx * ld_geo_uniform<GP>(g.h[1], rc), sr));
                    }
                    if (rc == ny && out_lane)  // top ghost row: only this face (ERK:1305)
                        block_min = __builtin_fmin(block_min, dt_candidate(hx * ld_geo_uniform<GP>(g.h[1], ny + 1), double(Sy * lam)));
                    lam_gb = lam;
                }
                if constexpr (MT::flux) {
                    if (t >= 2) {
                        // finalize row rc-1 = the row in slot sm
                        const int rf = rc - 1;
                        const double ivol = ihx * ld_geo_uniform<GP>(g.ih[1], rf + 1);
                        R res[N], Um[N];
#pragma unroll
                        for (int v = 0; v < N; v++) {
                            res[v] = flux_difference(cy[v][lane], through(G[v], Sy));
                            Um[v] = ring[wl][sm][v][lane];
                        }
                        finish(unsigned(rf) * unsigned(nx) + unsigned(xs), Um, res, Nc, Dc, ivol, hx * ld_geo_uniform<GP>(g.h[1], rf + 1));
                    }
#pragma unroll
                    for (int v = 0; v < N; v++) cy[v][lane] = through(G[v], Sy);
                }
                if (rc < yend) {
                    // x-faces of row rc: each lane evaluates its minus face.  The plus-face
                    // states of the left neighbours, then the fluxes and eigenvalues of the right
                    // neighbours, pass through the LDS slot of row rc-1, free after its finalize
                    // (LDS operations of one wavefront complete in order).
                    R (&xch)[N][64] = ring[wl][sm];
                    R UL[N], UR[N];
#pragma unroll
                    for (int v = 0; v < N; v++) xch[v][lane] = face[1][v];
#pragma unroll
                    for (int v = 0; v < N; v++) {
                        UL[v] = xch[v][lm];
                        UR[v] = face[0][v];
                    }
                    if (!g.periodic[0]) {
                        if (xg == 0) bc_image(g.bc[bc_marker(g, 0, rcs)], gamma, 0, UR, UL);
                        if (xg == nx) bc_image(g.bc[bc_marker(g, 1, rcs)], gamma, 0, UL, UR);
                    }
                    const R Sx = R(hy);  // face area of an x-face (ERK:1189)
                    R F[N], lamx;
                    if constexpr (MT::flux) face_flux<FLUX, 0, R>(gamma, eps, UL, UR, F, lamx);
                    else lamx = face_eigen<FLUX, 0, R>(gamma, UL, UR);
                    if constexpr (VIN) {
                        if (vin) {
                            double gl[2], gr[2], vl[NM];
#pragma unroll
                            for (int d = 0; d < NM; d++) vl[d] = dpp_from_left(v0[d]);
#pragma unroll
                            for (int d = 0; d < 2; d++) {
                                gl[d] = dpp_from_left(gy[d]);
                                gr[d] = gy[d];
                            }
                            double pl[2], ml[2];  // lane shifts outside the lanes' branch: they read every lane
                            if (!g.periodic[0] && (strip == 0 || strip == a.nstrips - 1)) {
#pragma unroll
                                for (int d = 0; d < 2; d++) {
                                    pl[d] = dpp_from_left(vp[d]);
                                    ml[d] = dpp_from_left(vm[d]);
                                }
                                if (xg == 0 || xg == nx) {
                                    // the dummy cell is on the left (xg = 0, the boundary cell this lane's) or
                                    // this lane's own (xg = nx, the boundary cell the left neighbour's)
                                    const bool west = xg == 0;
                                    const int f = west ? 0 : nx;
                                    const double xl = a.v.x[0][f], xr = a.v.x[0][f + 1], hb = g.h[0][west ? 1 : nx];
                                    const double xf = west ? xr - 0.5 * hb : xl + 0.5 * hb;
                                    const double yc = a.v.x[1][rc + 1];
                                    const FaceLsq lsq{xf - (west ? xr : xl), xf - (west ? xl : xr), yc - a.v.x[1][rc + 2], yc - a.v.x[1][rc]};
                                    const double ir = frcp(0.5 * double(ring[wl][s0][0][lm] + ring[wl][s0][0][lane]));
#pragma unroll
                                    for (int d = 0; d < 2; d++) {
                                        const double face = 0.5 * double(ring[wl][s0][1 + d][lm] + ring[wl][s0][1 + d][lane]) * ir;
                                        const double gd = west ? lsq(face, v0[d], vp[d], vm[d], vl[d], gr[d])
                                                               : lsq(face, vl[d], pl[d], ml[d], v0[d], gl[d]);
                                        if (west) gl[d] = gd;
                                        else gr[d] = gd;
                                    }
                                }
                            }
                            const double tan[2] = {0.5 * (vhr * gl[0] + vhl * gr[0]), 0.5 * (vhr * gl[1] + vhl * gr[1])};
                            double tv[NM + 1];
                            vis_flux2<0, NM>(a.v.mu, vdx, vhl, vhr, vl, v0, tan, tv);
#pragma unroll
                            for (int v = 1; v < N; v++) F[v] -= R(tv[v - 1]);
                        }
                    }
                    if constexpr (MT::flux) {
#pragma unroll
                        for (int v = 0; v < N; v++) xch[v][lane] = F[v];
#pragma unroll
                        for (int v = 0; v < N; v++) cy[v][lane] = cy[v][lane] - flux_difference(xch[v][lp], F[v]) * Sx;
                    }
                    if constexpr (MT::sr) {
                        xch[0][lane] = lamx;
                        const R lam_r = xch[0][lp];
                        {
#pragma clang fp contract(off)
                            srp = double(Sx * lamx) + double(Sx * lam_r);
                        }
                        if constexpr (VIS) {
                            const double rl = dpp_from_right(double(UL[0])), rr = dpp_from_right(double(UR[0]));
                            srp = srp + viscous_sr(rl, rr, g.gamma, a.v.mu, double(Sx), hx * hy);
                        }
                        {
#pragma clang fp contract(off)
                            srp = srp + double(Sy * lam_gb);
                        }
                        if (ghost_x_lane)  // right ghost column (ERK:1225)
                            block_min = __builtin_fmin(block_min, dt_candidate(ld_geo_uniform<GP>(g.h[0], nx + 1) * hy, double(Sx * lamx)));
                    }
                }
            }
#pragma unroll
            for (int v = 0; v < N; v++) ytop[v] = face[3][v];
            if constexpr (VIN) {
#pragma unroll
                for (int d = 0; d < NM; d++) {
                    vm[d] = v0[d];
                    v0[d] = vp[d];
                }
#pragma unroll
                for (int d = 0; d < 2; d++) gxm[d] = gx[d];
            }
            const int st = sm;
            sm = s0;
            s0 = sp;
            sp = st;
        }
    }

}

// ---- single-solve kernel: one wavefront per tile, block-level dt reduction ----------------------
template <int DIM, int RECON, int LIM, int FLUX, int MODE, typename R, typename TIn, typename TOut, int N = NV, int VIS = 0>
__global__ void __launch_bounds__(256) fvm_stage(KArgs a) {
    static_assert(DIM == 1 || DIM == 2, "3-D uses its own kernel");
    using MT = ModeTraits<MODE>;
    StepCtl* ctl = a.ctl;
    if constexpr (MT::sr) {
        if (!ctl->active) {
            if (blockIdx.x == 0 && threadIdx.x == 0) ctl->go = 0;
            return;
        }
    } else {
        // stage 2 that applies the step's dt itself is the one that sets go
        if (!(MODE == MODE_F2 && a.dt_minima) && !ctl->go) return;
        if constexpr (MODE == MODE_RN) {
            if (ctl->active) return;  // not the last step of this call
        }
    }
    const int lane = threadIdx.x & 63;
    // the wavefront index is the same in all its lanes: readfirstlane lets the compiler keep the
    // tile, its rows and every row's geometry in scalar registers (scalar loads, whose waits do
    // not also wait for the vector loads of the stencil prefetch)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    const int tile = xcd_remap(blockIdx.x, gridDim.x) * nwaves + wave;
    if constexpr (MODE != MODE_RN && !MT::sr) {
        if (tile >= a.ntiles) return;  // the norms and the minima are reduced across the block
    }
    double block_min = __builtin_inf();
    double rn[N] = {};
    if constexpr (MODE == MODE_F2) {
        double dt = 0.0;
        if (a.dt_minima) {
            if (!step_dt(ctl, a.g.cfl, a.dt_part, a.dt_minima, lane, tile == 0, dt)) return;
        } else {
            dt = ctl->dt;
        }
        stage_tile<DIM, RECON, LIM, FLUX, MODE, R, TIn, TOut, N, VIS, true>(a, tile, lane, block_min, rn, dt);
    } else if (MODE == MODE_RN || tile < a.ntiles) {
        stage_tile<DIM, RECON, LIM, FLUX, MODE, R, TIn, TOut, N, VIS>(a, tile < a.ntiles ? tile : -1, lane, block_min, rn);
    }
    if constexpr (MODE == MODE_S3) {
        if (a.dt_minima && tile == 0 && lane == 0) step_advances(ctl, ctl->dt);
    }
    if constexpr (MT::sr) {
        // store the workgroup's minimum; stage 2 or dt_finalize_kernel turns these into dt after this
        // launch.  (One for each wavefront was four times as many: with the 1539 of a 512^2 grid stage 2
        // lost more by reducing them itself than the launch between them takes.)
        __shared__ double wave_min[4];
        block_min = wave_min_lane63(block_min);  // +inf without a tile
        if (lane == 63) wave_min[wave] = block_min;
        __syncthreads();
        if (threadIdx.x == 0) {
            const double m = __builtin_fmin(__builtin_fmin(wave_min[0], wave_min[1]), __builtin_fmin(wave_min[2], wave_min[3]));
            st_plane(a.dt_part, 0, 0, blockIdx.x, m);
        }
    }
    if constexpr (MODE == MODE_RN) {
        __shared__ double rred[4 * NV];
        double rn5[NV] = {};
#pragma unroll
        for (int v = 0; v < N; v++) rn5[plane_of<N>(v)] = rn[v];
        rn_reduce_finalize(ctl, a.rn_part, rn5, rred, lane, wave, nwaves);
    }
}

// ---- small 1-D forward-Euler solves: a chunk of steps in one workgroup -------------------------
// A grid of a few strips is launch-bound (two short kernels per step).  One workgroup runs up to
// `cap` steps of a ts_step call instead.  Every wavefront leaves the loop together: after a step
// that ends the run (stop rule, error) or after `cap` steps.
//
// Grids that fit keep the whole problem in LDS, a thread to each cell and to the face on its
// minus side (strided where the cells outnumber the threads): the state, the face fluxes and
// eigenvalues and the cell sizes; with a reconstruction also the plus-face states (the minus-face
// ones wait in the places of the fluxes).  A face is evaluated once, for its eigenvalue and its
// flux, and a step is the face pass, the minimum of V/SR, and the update, with three barriers (four
// with a reconstruction).  What bounds it is the latency of that chain; each thread keeps time, dt
// and the step count itself, so that no bookkeeping passes through memory.  (The former kernel walked
// 60-cell strips twice per step, first for the eigenvalues and then for the fluxes, and 1000
// cells are 17 strips: two rounds for 16 wavefronts.  1000 cells, first-order Roe:
// 5.1 us per step, now 2.7.)
template <int FLUX>
constexpr int euler1d_threads = FLUX == FX_GODUNOV ? 512 : 1024;  // Godunov: over 128 registers
constexpr int EULER1D_LDS = 20000;                               // doubles of the state and face arrays
template <int RECON, int N>
constexpr int euler1d_cells = EULER1D_LDS / (2 * N + 3 + (RECON == RC_PWC ? 0 : N)) - 1;

// a0: input buffer 0 -> output buffer 1 of the ping-pong; the final state goes to buffer 0 after an
// even number of steps and to buffer 1 after an odd one.  n <= euler1d_cells<RECON, N>.
template <int RECON, int LIM, int FLUX, int N>
__global__ void __launch_bounds__(euler1d_threads<FLUX>) fvm_euler1d_lds(KArgs a, int cap) {
    const GridArgs& g = a.g;
    const int n = g.n[0], T = blockDim.x, tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6, nwaves = T >> 6;
    const bool per = g.periodic[0] != 0;
    const int S = n + 1;  // plane stride: a plane holds the faces 0..n
    __shared__ double pool[EULER1D_LDS];
    __shared__ double red[16];
    double* U = pool;           // [N][S] cells
    double* F = U + N * S;      // [N][S] minus-face states, then fluxes, of faces 0..n
    double* lam = F + N * S;    // [S] eigenvalues of the faces
    double* h = lam + S;        // [S] sizes of cells 0..n (n: the right ghost)
    double* ih = h + S;         // [S]
    double* FP = ih + S;        // [N][S] plus-face states (RECON != PWC)
    StepCtl* ctl = a.ctl;
    const double* u0 = (const double*)a.uin;
    for (int c = tid; c <= n; c += T) {
        h[c] = g.h[0][c + 1];
        ih[c] = g.ih[0][c + 1];
        if (c < n)
#pragma unroll
            for (int v = 0; v < N; v++) U[v * S + c] = ld_plane(u0, a.plane, plane_of<N>(v), unsigned(c));
    }
    double time = ctl->time, dt = ctl->dt;
    const double t_max = ctl->t_max, next_snap = ctl->next_snap;
    const long long iter0 = ctl->iter;
    const int sd0 = ctl->steps_done, max_steps = ctl->max_steps;
    bool active = ctl->active != 0, failed = false;
    int done = 0;
    __syncthreads();
    while (active && done < cap) {
        if constexpr (RECON != RC_PWC) {
            for (int c = tid; c < n; c += T) {
                double u[N], nb[2][N], face[2][N];
                const int l = c > 0 ? c - 1 : (per ? n - 1 : 0), r = c < n - 1 ? c + 1 : (per ? 0 : n - 1);
#pragma unroll
                for (int v = 0; v < N; v++) {
                    u[v] = U[v * S + c];
                    nb[0][v] = U[v * S + l];
                    nb[1][v] = U[v * S + r];
                }
                if (!per && c == 0) bc_image(g.bc[bc_marker(g, 0, 0)], g.gamma, 0, u, nb[0]);
                if (!per && c == n - 1) bc_image(g.bc[bc_marker(g, 1, 0)], g.gamma, 0, u, nb[1]);
                CellGeo<1, double> geo;
                geo.hh[0] = 0.5 * h[c];
                geo.rc[0] = g.rc[0][c];
                geo.rl[0] = g.rl[0][c];
                geo.rr[0] = g.rr[0][c];
                geo.eps2 = (RECON == RC_LINLIM && LIM == LIM_VENKAT && g.ev[0]) ? g.ev[0][c] : g.eps2;
                reconstruct<1, RECON, LIM, double, FLUX != FX_ROE>(u, nb, geo, face);
#pragma unroll
                for (int v = 0; v < N; v++) {
                    F[v * S + c] = face[0][v];
                    FP[v * S + c] = face[1][v];
                    if (per && c == 0) F[v * S + n] = face[0][v];
                }
            }
            __syncthreads();
        }
        // faces: the state on the minus side, the state on the plus side, eigenvalue and flux
        for (int c = tid; c <= n; c += T) {
            const double* L = RECON == RC_PWC ? U : FP;
            const double* R = RECON == RC_PWC ? U : F;
            const int l = c > 0 ? c - 1 : (per ? n - 1 : 0);
            const int r = (RECON == RC_PWC && c == n) ? (per ? 0 : n - 1) : c;
            double UL[N], UR[N], Fx[N], lx;
#pragma unroll
            for (int v = 0; v < N; v++) {
                UL[v] = L[v * S + l];
                UR[v] = R[v * S + r];
            }
            if (!per && c == 0) bc_image(g.bc[bc_marker(g, 0, 0)], g.gamma, 0, UR, UL);
            if (!per && c == n) bc_image(g.bc[bc_marker(g, 1, 0)], g.gamma, 0, UL, UR);
            face_flux<FLUX, 0, double>(g.gamma, g.eps, UL, UR, Fx, lx);
            lam[c] = lx;
#pragma unroll
            for (int v = 0; v < N; v++) F[v * S + c] = Fx[v];
        }
        __syncthreads();
        double m = __builtin_inf();
        for (int c = tid; c <= n; c += T) {
            const double sr = c < n ? lam[c] + lam[c + 1] : lam[n];  // the right ghost cell has one face
            m = __builtin_fmin(m, dt_candidate(h[c], sr));
        }
        m = wave_min_lane63(m);
        if (lane == 63) red[wave] = m;
        __syncthreads();
        m = read_lane63(wave_min_lane63(red[lane < nwaves ? lane : 0]));
        // dt_apply's rule, by every thread
        double dtn = m * g.cfl;
        if (next_snap > 0 && next_snap < time + dtn) dtn = next_snap - time;
        if (!(dtn > 0.0) || !(dtn < __builtin_inf())) {
            failed = true;
            break;  // the state of the last good step stays in place
        }
        dt = dtn;
        time += dtn;
        for (int c = tid; c < n; c += T) {
            const double iv = ih[c];
#pragma unroll
            for (int v = 0; v < N; v++) U[v * S + c] += dtn * ((F[v * S + c] - F[v * S + c + 1]) * iv);
        }
        if (tid == 0 && ctl->dt_log) {
            const long long li = iter0 + done - ctl->dt_log_base;
            if (li >= 0 && li < ctl->dt_log_cap) ctl->dt_log[li] = dtn;
        }
        done++;
        active = !((time >= t_max) || (next_snap > 0 && time == next_snap) || (sd0 + done >= max_steps));
        __syncthreads();
    }
    double* out = (done & 1) ? (double*)a.uout : (double*)const_cast<void*>(a.uin);
    for (int c = tid; c < n; c += T)
#pragma unroll
        for (int v = 0; v < N; v++) st_plane(out, a.plane, plane_of<N>(v), unsigned(c), U[v * S + c]);
    if (tid == 0) {
        ctl->time = time;
        ctl->dt = dt;
        ctl->iter = iter0 + done;
        ctl->steps_done = sd0 + done;
        ctl->active = active && !failed ? 1 : 0;
        ctl->go = active && !failed ? 1 : 0;
        if (failed) ctl->error = 1;
    }
}

// Larger grids (up to 64 strips) keep the state in memory: the dt pass over the workgroup's strips
// (each wavefront takes strips w, w + W, ...), the workgroup minimum in LDS, the finalize by one
// thread, a barrier, the forward-Euler stage into the other state buffer and a barrier before the
// next dt pass reads it.  The two directions of the state ping-pong come as two kernel arguments
// (a0: buffer 0 -> 1, a1: 1 -> 0), so that nothing is copied per step; the control block lives in
// LDS for the chunk (thread 0 copies it in at the start and back at the end).  The exact
// solver's registers do not fit the 128 per lane of a 1024-thread workgroup, so Godunov has 8
// wavefronts instead of 16.
template <int FLUX>
constexpr int wg1d_waves = FLUX == FX_GODUNOV ? 8 : 16;

// one step; false when the loop has to end
template <int RECON, int LIM, int FLUX, int N>
__device__ __forceinline__ bool euler1d_step(const KArgs& a, StepCtl* ctl, double* red, int* run, int lane, int wave) {
    if (threadIdx.x == 0) *run = ctl->active;
    __syncthreads();
    if (!*run) {
        if (threadIdx.x == 0) ctl->go = 0;
        return false;
    }
    double m = __builtin_inf();
    for (int tile = wave; tile < a.ntiles; tile += wg1d_waves<FLUX>) {
        double mt = __builtin_inf();
        stage_tile<1, RECON, LIM, FLUX, MODE_DT, double, double, double, N>(a, tile, lane, mt);
        m = __builtin_fmin(m, mt);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = __builtin_fmin(m, __shfl_xor(m, o));
    if (lane == 0) red[wave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        double bmin = red[0];
        for (int w = 1; w < wg1d_waves<FLUX>; w++) bmin = __builtin_fmin(bmin, red[w]);
        // the whole grid is this workgroup: no atomics on the control block
        dt_apply(ctl, a.g.cfl, bmin);
        *run = ctl->go;
    }
    __syncthreads();
    if (!*run) return false;  // non-physical step: the state of the last good step stays in place
    const double dt = ctl->dt;
    for (int tile = wave; tile < a.ntiles; tile += wg1d_waves<FLUX>) {
        double unused = 0.0;
        stage_tile<1, RECON, LIM, FLUX, MODE_S1, double, double, double, N, 0, true>(a, tile, lane, unused, nullptr, dt);
    }
    __syncthreads();
    return true;
}

template <int RECON, int LIM, int FLUX, int N>
__global__ void __launch_bounds__(64 * wg1d_waves<FLUX>) fvm_euler1d_workgroup(KArgs a0, KArgs a1, int cap) {
    __shared__ double red[wg1d_waves<FLUX>];
    __shared__ int run;
    __shared__ StepCtl ctl;  // a0.ctl and a1.ctl are the same block
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x == 0) ctl = *a0.ctl;  // read only by thread 0 until the first barrier
    for (int it = 0; it < cap; it += 2) {
        if (!euler1d_step<RECON, LIM, FLUX, N>(a0, &ctl, red, &run, lane, wave)) break;
        if (it + 1 >= cap) break;
        if (!euler1d_step<RECON, LIM, FLUX, N>(a1, &ctl, red, &run, lane, wave)) break;
    }
    if (threadIdx.x == 0) *a0.ctl = ctl;  // the other threads only ever read the LDS copy
}

// ---- batched kernel: a persistent grid over a table of (problem, tile) pairs -----------------
// Every problem of the batch keeps its own KArgs (state, geometry, control block).  Wavefront w of
// the persistent grid takes tiles w, w + W, w + 2W, ... of the table (W = wavefronts in the grid):
// no claim atomics, which serialise at one address at tens of ns each, and every wavefront's
// loop ends after at most ceil(ntiles / W) tiles.  Neighbouring wavefront ids sit on one XCD, so
// neighbouring tiles of a problem share an L2.  Stage 1 stores each table entry's wavefront-level
// minimum of V/SR in `part` (by entry), and dt_finalize_batched or stage 2 turns each problem's entries
// into its dt.  A cell's arithmetic depends only on its own problem, and the minimum is exact, so a
// result is the same alone or in a mix.

template <int DIM, int RECON, int LIM, int FLUX, int MODE, typename R, typename TIn, typename TOut, int N = NV>
__global__ void __launch_bounds__(256) fvm_stage_batched(const KArgs* __restrict__ descs,
                                                         const int2* __restrict__ table,
                                                         const int* __restrict__ ntiles_p,
                                                         double* __restrict__ part) {
    using MT = ModeTraits<MODE>;
    const int lane = threadIdx.x & 63;
    // loop control in SGPRs: every quantity below is uniform over the wavefront
    const int ntiles = __builtin_amdgcn_readfirstlane(*ntiles_p);
    const int nwpb = blockDim.x >> 6;
    const int stride = gridDim.x * nwpb;
    const int w0 = __builtin_amdgcn_readfirstlane(xcd_remap(blockIdx.x, gridDim.x) * nwpb + (threadIdx.x >> 6));
    for (int t = w0; t < ntiles; t += stride) {
        const int2 e = table[t];
        const KArgs& a = descs[e.x];
        StepCtl* ctl = a.ctl;
        if constexpr (MT::sr) {
            if (!ctl->active) {
                if (e.y == 0 && lane == 0) ctl->go = 0;
                continue;
            }
        } else {
            // (stage 2 that applies the step's dt itself is the one that sets go)
            if (!(DIM == 1 && MODE == MODE_F2 && a.dt_minima) && !ctl->go) continue;
        }
        double m = __builtin_inf();
        // A 1-D solve of few entries applies dt itself in stage 2 (see step_dt).  A solve's entries are
        // contiguous, so its first one is this entry's index less its place in the solve.
        double dt = 0.0;
        if constexpr (DIM == 1 && MODE == MODE_F2) {
            if (!a.dt_minima) dt = ctl->dt;
            else if (!step_dt(ctl, a.g.cfl, part + (t - e.y), a.dt_minima, lane, e.y == 0, dt)) continue;
        }
        if constexpr (DIM == 1) {
            // a 1-D work item is a group of a.ty consecutive strips, walked by one wavefront
            const int s0 = e.y * a.ty;
            const int s1 = (s0 + a.ty < a.ntiles) ? s0 + a.ty : a.ntiles;
            for (int sidx = s0; sidx < s1; sidx++) {
                double ms = __builtin_inf();
                stage_tile<DIM, RECON, LIM, FLUX, MODE, R, TIn, TOut, N, 0, MODE == MODE_F2, true>(a, sidx, lane, ms, nullptr, dt);
                m = __builtin_fmin(m, ms);
            }
        } else {
            stage_tile<DIM, RECON, LIM, FLUX, MODE, R, TIn, TOut, N, 0, false, true>(a, e.y, lane, m);
        }
        if constexpr (DIM == 1 && MODE == MODE_S3) {
            if (a.dt_minima && e.y == 0 && lane == 0) step_advances(ctl, ctl->dt);
        }
        if constexpr (MT::sr) {
            // the entry's minimum; stage 2 or dt_finalize_batched reduces each solve's entries
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) m = __builtin_fmin(m, __shfl_xor(m, o));
            if (lane == 0) part[t] = m;
        }
    }
}

}  // namespace tsd
