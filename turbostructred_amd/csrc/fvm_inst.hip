// fvm_inst.hip -- instantiates the stage kernels of one (dimension, flux) pair.  Compiled once
// per pair with -DTS_DIM=<1|2|3> -DTS_FLUX=<0 Godunov|1 Roe|3 HLLC> so that the kernel families
// build in parallel.
#include "fvm_dispatch.hpp"
#include "fvm_viscous.hpp"
#if TS_DIM == 3 && __has_include("fvm_kernels3d.hpp")
#include "fvm_kernels3d.hpp"
#define TS_HAVE_3D 1
#endif

#ifndef TS_DIM
#error "TS_DIM must be defined"
#endif
#ifndef TS_FLUX
#error "TS_FLUX must be defined"
#endif

#define TS_CAT2(a, b, c, d) a##b##c##d
#define TS_CAT(a, b, c, d) TS_CAT2(a, b, c, d)
#define TS_GETTER TS_CAT(get_kernels_d, TS_DIM, _f, TS_FLUX)

namespace tsd {

#if !(TS_DIM == 3 && !defined(TS_HAVE_3D))
#if TS_DIM == 3
// one workgroup per tile: strips, row blocks, and blocks of the z-planes the instance outputs
template <typename R, int VIS, int MODE>
static dim3 grid3d(const KArgs& a) {
    constexpr int zout = z_waves<R, VIS, MODE> - 2;
    return dim3(a.nstrips * ((a.g.n[1] + a.ty - 1) / a.ty) * ((a.g.n[2] + zout - 1) / zout));
}
#endif
template <int RC, int LM, int N, int MODE, typename R, typename TIn, typename TOut>
static void launch(const KArgs& a, dim3 g, dim3 b, hipStream_t s) {
#if TS_DIM == 3
    KArgs b3 = a;
    if (MODE == MODE_F2) b3.ty = a.ty2;
    hipLaunchKernelGGL((fvm_stage3d<RC, LM, TS_FLUX, MODE, R, TIn, TOut>), (grid3d<R, 0, MODE>(b3)), dim3(64 * (z_waves<R, 0, MODE>)), 0, s, b3);
#else
    hipLaunchKernelGGL((fvm_stage<TS_DIM, RC, LM, TS_FLUX, MODE, R, TIn, TOut, N>), g, b, 0, s, a);
#endif
    if constexpr (ModeTraits<MODE>::sr) {
        if (!a.dt_minima) hipLaunchKernelGGL(dt_finalize_kernel<0>, dim3(1), dim3(1024), 0, s, a.ctl, a.g.cfl, a.dt_part, int(g.x));
    }
}

// resident workgroups per CU of the single-solve stage kernels (the minimum over the kernels of
// one precision): sets how many tiles run in one round
template <typename K> static int blocks_per_cu(K kernel, int threads) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, 0) != hipSuccess) return 1;
    return n > 0 ? n : 1;
}
template <int RC, int LM, int N, typename R, typename S, typename E>
static int single_occupancy() {
#if TS_DIM == 3
#define TS_T(MODE) 64 * z_waves<R, 0, MODE>
#define TS_K(MODE, A, B, C) fvm_stage3d<RC, LM, TS_FLUX, MODE, A, B, C>
#else
#define TS_T(MODE) 256
#define TS_K(MODE, A, B, C) fvm_stage<TS_DIM, RC, LM, TS_FLUX, MODE, A, B, C, N>
#endif
    int m = blocks_per_cu(TS_K(MODE_F1, R, double, S), TS_T(MODE_F1));
    int v[] = {blocks_per_cu(TS_K(MODE_F2, R, double, S), TS_T(MODE_F2)), blocks_per_cu(TS_K(MODE_S3, R, S, double), TS_T(MODE_S3)),
               blocks_per_cu(TS_K(MODE_DT, R, double, double), TS_T(MODE_DT)), blocks_per_cu(TS_K(MODE_S1, R, double, E), TS_T(MODE_S1))};
#undef TS_K
#undef TS_T
    for (int x : v) m = x < m ? x : m;
    return m;
}

#if TS_DIM != 3
template <int RC, int LM, int N, int MODE, typename R, typename TIn, typename TOut>
static void launch_batched(const KArgs* d, const int2* t, const int* ntiles, double* part, int nblk, hipStream_t s) {
    hipLaunchKernelGGL((fvm_stage_batched<TS_DIM, RC, LM, TS_FLUX, MODE, R, TIn, TOut, N>), dim3(nblk), dim3(256), 0, s,
                       d, t, ntiles, part);
}
template <int RC, int LM, int N, typename R, typename S>
static int batched_occupancy() {
    int a = 0, b = 0, c = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, fvm_stage_batched<TS_DIM, RC, LM, TS_FLUX, MODE_F1, R, double, S, N>, 256, 0) != hipSuccess) return 1;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, fvm_stage_batched<TS_DIM, RC, LM, TS_FLUX, MODE_F2, R, double, S, N>, 256, 0) != hipSuccess) return 1;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&c, fvm_stage_batched<TS_DIM, RC, LM, TS_FLUX, MODE_S3, R, S, double, N>, 256, 0) != hipSuccess) return 1;
    int m = a < b ? a : b;
    m = m < c ? m : c;
    return m > 0 ? m : 1;
}
#endif

#if TS_DIM != 2
// viscous pre-pass: gradients of the interior cells, then the faces of every axis
static void launch_vis_prepass(const KArgs& a, dim3, dim3, hipStream_t s) {
    const unsigned nb = unsigned((a.plane + 255) / 256);
    hipLaunchKernelGGL(vis_gradients<TS_DIM>, dim3(nb), dim3(256), 0, s, a);
    hipLaunchKernelGGL((vis_face_flux<TS_DIM, 0>), dim3((a.v.nface[0] + 255) / 256), dim3(256), 0, s, a);
#if TS_DIM > 2
    hipLaunchKernelGGL((vis_face_flux<TS_DIM, 1>), dim3((a.v.nface[1] + 255) / 256), dim3(256), 0, s, a);
    hipLaunchKernelGGL((vis_face_flux<TS_DIM, 2>), dim3((a.v.nface[2] + 255) / 256), dim3(256), 0, s, a);
#endif
}
#endif
template <int RC, int LM, int N, int MODE>
static void launch_vis(const KArgs& a, dim3 g, dim3 b, hipStream_t s) {
#if TS_DIM == 3
    hipLaunchKernelGGL((fvm_stage3d<RC, LM, TS_FLUX, MODE, double, double, double, 1>), (grid3d<double, 1, MODE>(a)),
                       dim3(64 * (z_waves<double, 1, MODE>)), 0, s, a);
#else
    hipLaunchKernelGGL((fvm_stage<TS_DIM, RC, LM, TS_FLUX, MODE, double, double, double, N, 1>), g, b, 0, s, a);
#endif
    if constexpr (ModeTraits<MODE>::sr) hipLaunchKernelGGL(dt_finalize_kernel<0>, dim3(1), dim3(1024), 0, s, a.ctl, a.g.cfl, a.dt_part, int(g.x));
}

#if TS_DIM == 1
template <int RC, int LM, int N>
static void launch_euler1d_chunk(const KArgs& a, int steps, hipStream_t s) {
    if (a.g.n[0] <= euler1d_cells<RC, N>) {
        // a thread per face (faces 0..n), whole wavefronts
        const int threads = (a.g.n[0] + 64) / 64 * 64;
        hipLaunchKernelGGL((fvm_euler1d_lds<RC, LM, TS_FLUX, N>), dim3(1),
                           dim3(threads < euler1d_threads<TS_FLUX> ? threads : euler1d_threads<TS_FLUX>), 0, s, a, steps);
        return;
    }
    KArgs b = a;  // the other direction of the ping-pong
    b.uin = a.uout;
    b.uout = const_cast<void*>(a.uin);
    hipLaunchKernelGGL((fvm_euler1d_workgroup<RC, LM, TS_FLUX, N>), dim3(1), dim3(64 * wg1d_waves<TS_FLUX>), 0, s, a, b, steps);
}
#endif

// the instances that carry N variables; the ones with every variable also cover the unfused SSP
// sequence, and they and the 2-D ones the viscous terms
template <int RC, int LM, int N>
static void fill(int precision, KernelSet* ks) {
    if (precision == 0) {
        ks->dt = launch<RC, LM, N, MODE_DT, double, double, double>;
        ks->s1e = launch<RC, LM, N, MODE_S1, double, double, double>;
        ks->s3 = launch<RC, LM, N, MODE_S3, double, double, double>;
        ks->f1 = launch<RC, LM, N, MODE_F1, double, double, double>;
        ks->f2 = launch<RC, LM, N, MODE_F2, double, double, double>;
        ks->rn = launch<RC, LM, N, MODE_RN, double, double, double>;
        ks->socc = single_occupancy<RC, LM, N, double, double, double>;
#if TS_DIM != 3
        ks->bf1 = launch_batched<RC, LM, N, MODE_F1, double, double, double>;
        ks->bf2 = launch_batched<RC, LM, N, MODE_F2, double, double, double>;
        ks->bs3 = launch_batched<RC, LM, N, MODE_S3, double, double, double>;
        ks->bocc = batched_occupancy<RC, LM, N, double, double>;
#endif
        if constexpr (N == NV) {
            ks->s1r = ks->s1e;
            ks->s2 = launch<RC, LM, N, MODE_S2, double, double, double>;
        }
        if constexpr (N == NV || TS_DIM == 2) {
#if TS_DIM != 2
            ks->vpre = launch_vis_prepass;
#endif
            ks->vdt = launch_vis<RC, LM, N, MODE_DT>;
            ks->vs1 = launch_vis<RC, LM, N, MODE_S1>;
            ks->vs2 = launch_vis<RC, LM, N, MODE_S2>;
            ks->vs3 = launch_vis<RC, LM, N, MODE_S3>;
            ks->vrn = launch_vis<RC, LM, N, MODE_RN>;
        }
#if TS_DIM == 1
        ks->euler1d_chunk = launch_euler1d_chunk<RC, LM, N>;
#endif
    } else {
        ks->dt = launch<RC, LM, N, MODE_DT, float, double, double>;
        ks->s1e = launch<RC, LM, N, MODE_S1, float, double, double>;
        ks->s3 = launch<RC, LM, N, MODE_S3, float, float, double>;
        ks->f1 = launch<RC, LM, N, MODE_F1, float, double, float>;
        ks->f2 = launch<RC, LM, N, MODE_F2, float, double, float>;
        ks->rn = launch<RC, LM, N, MODE_RN, float, double, float>;
        ks->socc = single_occupancy<RC, LM, N, float, float, double>;
#if TS_DIM != 3
        ks->bf1 = launch_batched<RC, LM, N, MODE_F1, float, double, float>;
        ks->bf2 = launch_batched<RC, LM, N, MODE_F2, float, double, float>;
        ks->bs3 = launch_batched<RC, LM, N, MODE_S3, float, float, double>;
        ks->bocc = batched_occupancy<RC, LM, N, float, float>;
#endif
        if constexpr (N == NV) {
            ks->s1r = launch<RC, LM, N, MODE_S1, float, double, float>;
            ks->s2 = launch<RC, LM, N, MODE_S2, float, float, float>;
        }
    }
}
#endif

#if TS_DIM == 3 && !defined(TS_HAVE_3D)
bool TS_GETTER(int, int, bool, KernelSet*) { return false; }
#else
template <int N>
static bool fill_variant(int rv, int precision, KernelSet* ks) {
    switch (rv) {
    case 0: fill<RC_PWC, LIM_BJ, N>(precision, ks); return true;
    case 1: fill<RC_LINEAR, LIM_BJ, N>(precision, ks); return true;
    case 2: fill<RC_ENO2, LIM_BJ, N>(precision, ks); return true;
    case 3: fill<RC_LINLIM, LIM_BJ, N>(precision, ks); return true;
    case 4: fill<RC_LINLIM, LIM_VENKAT, N>(precision, ks); return true;
    }
    return false;
}
bool TS_GETTER(int rv, int precision, bool in_grid, KernelSet* ks) {
#if TS_DIM < 3
    if (in_grid) return fill_variant<TS_DIM + 2>(rv, precision, ks);
#endif
    return fill_variant<NV>(rv, precision, ks);
}
#endif

}  // namespace tsd
