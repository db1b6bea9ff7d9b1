// fvm_kernels3d.hpp -- fused finite-volume stage kernel for 3-D grids (gfx950).
//
// A workgroup is ZW wavefronts, one per z-plane k = k0-1+w; wavefronts 1..ZW-2 produce output and the
// two edge wavefronts only supply reconstructions (each loads the one extra centre row its outer
// z-neighbour needs).  Inside a plane the scheme is the 2-D one: 64 lanes along x (60 output
// columns) and a three-row window marching along y in the wavefront's own LDS slots, from which
// the z-neighbours of its centre row are read too.  The z+ face state travels to the plane
// above through the slot of the row just finalized, and the z-face flux back to the plane below
// through a slot of its own, read one row later: two barriers per row.  Each z-face flux is
// evaluated once, by the wavefront above it.
//
// What bounds it is VALU issue and the latency of the row's serial chain, so registers and LDS are
// spent to have wavefronts: 20 values per lane and wavefront in LDS (window 15, z-flux 5) and, where
// they do not fit into registers, 10 that are carried to the next row; the face states as the cell and
// its offsets.  In float 16 wavefronts share a CU, four per SIMD, and 14 of 16 planes produce output
// (stage 2: 12, three, 10 of 12).  In double 220 to 250 registers allow two per SIMD, 8 and 6 of 8; 12 wavefronts
// at 168 registers spilled (stage 2 of 256^3 3.0 ms).  With the window in registers and copies of the centre
// row, the carried fluxes and both z exchanges in LDS (42 values) the float kernels ran at two per
// SIMD: 150x141x133 step 507 us, now 363; 256^3 double step 3.37 ms, now 2.96.
//
// The residual of a cell is the sum of the flux differences of x, y and z, and its spectral radius that of
// x-, x+, y-, y+, z-, z+ (ERK:1225-1248, 1305-1328, 1385-1408).  (Adding the fluxes one by one rounds
// at the size of a flux, not of the difference: a uniform float flow drifted.)  VIS instances add the viscous face fluxes of the
// pre-pass, the viscous spectral-radius term after each plus face (the z-face part travels through
// LDS with the z eigenvalue) and the body-force sources.
#pragma once

#include "fvm_kernels.hpp"

namespace tsd {

// geometry of one row, the same for the whole workgroup; loaded a row ahead
struct RowGeo {
    double h, ih, rc, rl, rr, ev;
};

template <int RECON, int LIM, int FLUX, int MODE, typename R, typename TIn, typename TOut, int VIS = 0>
__global__ void __launch_bounds__(64 * (z_waves<R, VIS, MODE>)) fvm_stage3d(KArgs a) {
    using MT = ModeTraits<MODE>;
    constexpr int ZW = z_waves<R, VIS, MODE>, ZOUT = ZW - 2;
    StepCtl* ctl = a.ctl;
    __shared__ R ring[ZW][3][NV][64];                  // [wavefront][slot][variable][lane]
    // What is carried to the next row, of the row that is pending then: the x part of its residual and the
    // fluxes through its faces below, in y and z.  In double all 15 values fit into the registers with the
    // HLLC flux (247 of 256 at most; 256^3 step 2.96 ms, 3.04 with the x part in LDS, 3.16 with
    // none) and with Roe's, whose stage 2 spills little (128^3 611 us, 637 with the x part in LDS) but for
    // ENO2 (650 against 631), and in first order also with the exact solver (128^3 step 1137 us, 1189 in LDS);
    // with a reconstruction that one and the float kernels would spill.
    constexpr bool X_REGS = sizeof(R) == 8 && (FLUX == FX_HLLC || RECON == RC_PWC || (FLUX == FX_ROE && RECON != RC_ENO2));
    constexpr bool YZ_REGS = sizeof(R) == 8 && (FLUX != FX_GODUNOV || RECON == RC_PWC);
    __shared__ R carry_x[MT::flux && !X_REGS ? ZW : 1][NV][64];
    __shared__ R carry_y[MT::flux && !YZ_REGS ? ZW : 1][NV][64];
    __shared__ R lds_h[MT::flux ? ZW : 1][NV][64];     // flux through the z-face below every plane
    __shared__ R lds_l[MT::sr ? ZW : 1][64];           // eigenvalue of that face
    __shared__ double lds_vz[VIS && MT::sr ? ZW : 1][64];  // its viscous spectral-radius term before / V
    __shared__ double red[ZW];
    if constexpr (MT::sr) {
        if (!ctl->active) {
            if (blockIdx.x == 0 && threadIdx.x == 0) ctl->go = 0;
            return;
        }
    } else {
        if (!ctl->go) return;
        if constexpr (MODE == MODE_RN) {
            if (ctl->active) return;  // only in the step that ends the ts_step call
        }
    }
    const GridArgs& g = a.g;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: scalar plane indices
    const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
    const int nyb = (ny + a.ty - 1) / a.ty;
    const int tile = xcd_remap(blockIdx.x, gridDim.x);  // one tile per workgroup
    const int strip = tile % a.nstrips;
    const int yb = (tile / a.nstrips) % nyb;
    const int zb = tile / (a.nstrips * nyb);
    const int k = zb * ZOUT - 1 + w;  // this wavefront's plane (may be a ghost plane)
    int ks, kside;
    map_index(k, nz, g.periodic[2], ks, kside);
    const bool out_plane = w >= 1 && w <= ZOUT && k < nz;
    const bool edge = (w == 0) || (w == ZW - 1);

    const int xg = strip * STRIP - 2 + lane;
    int xs, xside;
    map_index(xg, nx, g.periodic[0], xs, xside);
    const bool x_out = lane >= 2 && lane < 2 + STRIP && xg < nx;
    const bool out_lane = out_plane && x_out;
    const bool ghost_x_lane = out_plane && xg == nx && lane >= 2 && lane <= 62;

    const R gamma = R(g.gamma), eps = R(g.eps);
    const double dt = MT::sr ? 0.0 : ctl->dt;

    CellGeo<3, R> geo;
    const double hx = g.h[0][xs + 1], ihx = g.ih[0][xs + 1];
    const double hz = g.h[2][ks + 1], ihz = g.ih[2][ks + 1];
    geo.hh[0] = R(0.5 * hx);
    geo.rc[0] = R(g.rc[0][xs]);
    geo.rl[0] = R(g.rl[0][xs]);
    geo.rr[0] = R(g.rr[0][xs]);
    geo.hh[2] = R(0.5 * hz);
    geo.rc[2] = R(g.rc[2][ks]);
    geo.rl[2] = R(g.rl[2][ks]);
    geo.rr[2] = R(g.rr[2][ks]);
    geo.eps2 = R(g.eps2);
    // per-cell Venkatakrishnan eps^2 on non-uniform grids (see GridArgs::ev)
    const bool ev_cells = RECON == RC_LINLIM && LIM == LIM_VENKAT && g.ev[0] != nullptr;
    const double ev_xz = ev_cells ? g.ev[0][xs] * g.ev[2][ks] : 0.0;
    auto row_geo = [&](int r) {
        int rs, side;
        map_index(r, ny, g.periodic[1], rs, side);
        RowGeo q;
        q.h = g.h[1][rs + 1];
        q.ih = g.ih[1][rs + 1];
        q.rc = g.rc[1][rs];
        if constexpr (RECON == RC_ENO2) {
            q.rl = g.rl[1][rs];
            q.rr = g.rr[1][rs];
        }
        if (ev_cells) q.ev = g.ev[1][rs];
        return q;
    };

    const TIn* __restrict__ uin = (const TIn*)a.uin;
    const TOut* __restrict__ lin = (const TOut*)a.lin;
    TOut* uo = (TOut*)a.uout;
    const size_t P = a.plane;
    // FP32-residual stages 2 and 3 with the increment form (see stage_tile)
    constexpr bool INC_F2 = MODE == MODE_F2 && sizeof(TOut) == 4, INC_S3 = MODE == MODE_S3 && sizeof(TIn) == 4;
    const bool inc = (INC_F2 && a.dout != nullptr) || (INC_S3 && a.din != nullptr);
    // the centre L(U^n) (stage 2) or increment (stage 3) is loaded with the centre U^n
    using IncT = typename std::conditional<MODE == MODE_F2, TOut, TIn>::type;
    const IncT* incsrc = (MODE == MODE_F2) ? (const IncT*)a.lin : (const IncT*)a.din;

    // Stencil input at (xg, row r, plane kk), in two steps: the loads (issue_cell), and the
    // value formed from them with its ghost image (complete_cell).  Prefetched cells are
    // completed one iteration after their loads are issued, so that no arithmetic on the loaded
    // values makes the wavefront wait for them early.
    struct RawCell {
        TIn u[NV];
        TOut l[MODE == MODE_F2 ? NV : 1];
    };
    auto issue_cell = [&](int r, int kk, RawCell& q) {
        int rs, kks, side;
        map_index(r, ny, g.periodic[1], rs, side);
        map_index(kk, nz, g.periodic[2], kks, side);
        const unsigned off = (unsigned(kks) * unsigned(ny) + unsigned(rs)) * unsigned(nx) + unsigned(xs);
#pragma unroll
        for (int v = 0; v < NV; v++) q.u[v] = ld_plane(uin, P, v, off);
        if constexpr (MODE == MODE_F2) {
#pragma unroll
            for (int v = 0; v < NV; v++) q.l[v] = ld_plane(lin, P, v, off);
        }
    };
    auto complete_cell = [&](const RawCell& q, int r, int kk, R (&u)[NV]) {
        if constexpr (MODE == MODE_F2) {
#pragma unroll
            for (int v = 0; v < NV; v++) u[v] = R(double(q.u[v]) + dt * double(q.l[v]));
        } else {
#pragma unroll
            for (int v = 0; v < NV; v++) u[v] = R(q.u[v]);
        }
        // one call per axis, so that the axis is a constant inside bc_image (a run-time axis
        // would index the state arrays dynamically and put them in scratch memory)
        int rs, kks, yside, zside;
        map_index(r, ny, g.periodic[1], rs, yside);
        map_index(kk, nz, g.periodic[2], kks, zside);
        R t[NV];
        bool img = true;
        if (xside != 0) bc_image(g.bc[bc_marker(g, xside < 0 ? 0 : 1, kks * ny + rs)], gamma, 0, u, t);
        else if (yside != 0) bc_image(g.bc[bc_marker(g, yside < 0 ? 2 : 3, kks * nx + xs)], gamma, 1, u, t);
        else if (zside != 0) bc_image(g.bc[bc_marker(g, zside < 0 ? 4 : 5, rs * nx + xs)], gamma, 2, u, t);
        else img = false;
        if (img) {
#pragma unroll
            for (int v = 0; v < NV; v++) u[v] = t[v];
        }
    };
    auto load_cell = [&](int r, int kk, R (&u)[NV]) {
        RawCell q;
        issue_cell(r, kk, q);
        complete_cell(q, r, kk, u);
    };

    double block_min = __builtin_inf();
    double rn[NV] = {0.0, 0.0, 0.0, 0.0, 0.0};
    const int y0 = yb * a.ty;
    const int yend = (y0 + a.ty < ny) ? y0 + a.ty : ny;
    R Db[X_REGS ? NV : 1], Gb[YZ_REGS ? NV : 1], Hb[YZ_REGS ? NV : 1];
    auto dfx = [&](int v) -> R& {
        if constexpr (X_REGS) return Db[v];
        else return carry_x[MT::flux ? w : 0][v][lane];
    };
    auto gbot = [&](int v) -> R& {
        if constexpr (YZ_REGS) return Gb[v];
        else return carry_y[MT::flux ? w : 0][v][lane];
    };
    auto hbot = [&](int v) -> R {
        if constexpr (YZ_REGS) return Hb[v];
        else return lds_h[w][v][lane];
    };
    int sm = 0, s0 = 1, sp = 2;  // slots of rows rc-1, rc, rc+1
    RawCell Pn;                  // prefetched stencil row, completed one iteration later
    // The centre row of the z-neighbour that no wavefront holds (edge wavefronts, prefetched), or U^n
    // of the row finalized in this iteration (output wavefronts, SSP stages 2, 3): a wavefront needs
    // one or the other, in the same registers.
    RawCell Zq;
    constexpr bool SHARED_REGS = sizeof(TIn) == 8;
    double Ns[SHARED_REGS ? 1 : NV];
    auto nc = [&](int v) -> double& {
        if constexpr (SHARED_REGS) return Zq.u[v];
        else return Ns[v];
    };
    IncT Dc[NV];            // its L(U^n) or increment (FP32-residual stages 2, 3)
    R ytop[NV];             // +y face state of the previous row
    double srp = 0.0;       // x terms + bottom y term of the pending row's spectral radius
    R lzb = R(0);           // eigenvalue of its bottom z-face
    R lam_gb = R(0);
    R Szb = R(0);           // z-face area of the pending row (its y size differs from the current row's)
    {
        R t0[NV], t1[NV];
        load_cell(y0 - 2, k, t0);
        load_cell(y0 - 1, k, t1);
#pragma unroll
        for (int v = 0; v < NV; v++) {
            ring[w][sm][v][lane] = t0[v];
            ring[w][s0][v][lane] = t1[v];
        }
    }
    issue_cell(y0, k, Pn);
    const int zoff = (w == 0) ? -1 : 1;  // the z-neighbour an edge wavefront loads itself
    if (edge) issue_cell(y0 - 1, k + zoff, Zq);
    RowGeo gc = row_geo(y0 - 1);
    double hyp = gc.h, ihyp = gc.ih;  // of the row above which the window moves on
    const int lm = lane > 0 ? lane - 1 : 0, lp = lane < 63 ? lane + 1 : 63;
    // The next row's loads go out at the start of an iteration where the registers allow (double,
    // stages that read one array: 256^3 stage 1 988 us against 1041), else after the second barrier,
    // where the z and x faces still cover most of their latency and they do not add to the registers of
    // the reconstruction and the y-face (stage 2 1058 us against 1190).
    constexpr bool EARLY = sizeof(R) == 8 && !MT::use_un;
    const int nit = yend - y0 + 2;
    __syncthreads();  // the first rows of the neighbouring planes
    for (int t = 0; t < nit; t++) {
        const int rc = y0 - 1 + t;  // row being reconstructed
        const bool row_out = rc >= y0 && rc < yend;
        const RowGeo gn = row_geo(rc + 1);
        R Up[NV], Zx[NV];
        complete_cell(Pn, rc + 1, k, Up);
        if (EARLY && t + 1 < nit) issue_cell(rc + 2, k, Pn);
        if (edge) {
            complete_cell(Zq, rc, k + zoff, Zx);
            if (EARLY && t + 1 < nit) issue_cell(rc + 1, k + zoff, Zq);
        } else if (MT::use_un && out_plane && t >= 2) {
            // U^n of the row finalized in this iteration (read earlier as a stencil row)
            const unsigned offn = (unsigned(ks) * unsigned(ny) + unsigned(rc - 1)) * unsigned(nx) + unsigned(xs);
#pragma unroll
            for (int v = 0; v < NV; v++) nc(v) = ld_plane(a.un, P, v, offn);
            if (inc) {
#pragma unroll
                for (int v = 0; v < NV; v++) Dc[v] = ld_plane(incsrc, P, v, offn);
            }
        }
        int rcs, rcside;
        map_index(rc, ny, g.periodic[1], rcs, rcside);
        const double hy = gc.h;
        geo.hh[1] = R(0.5 * hy);
        geo.rc[1] = R(gc.rc);
        if constexpr (RECON == RC_ENO2) {
            geo.rl[1] = R(gc.rl);
            geo.rr[1] = R(gc.rr);
        }
        if (ev_cells) geo.eps2 = R(ev_xz * gc.ev);

        // Face states are kept as the cell and its offset per axis (20 values instead of 30) and formed
        // where they are used; `bad` marks the faces that fall back to the cell value.
        R U0[NV], off[3][NV];
        unsigned bad = 0;
        {
            R nb[6][NV];
#pragma unroll
            for (int v = 0; v < NV; v++) {
                U0[v] = ring[w][s0][v][lane];
                nb[0][v] = ring[w][s0][v][lm];
                nb[1][v] = ring[w][s0][v][lp];
                nb[2][v] = ring[w][sm][v][lane];
                nb[3][v] = Up[v];
                nb[4][v] = (w == 0) ? Zx[v] : ring[w - 1][s0][v][lane];
                nb[5][v] = (w == ZW - 1) ? Zx[v] : ring[w + 1][s0][v][lane];
            }
            face_offsets<3, RECON, LIM>(U0, nb, geo, off);
        }
        auto face_state = [&](int f, R (&u)[NV]) {
#pragma unroll
            for (int v = 0; v < NV; v++) u[v] = (f & 1) ? U0[v] + off[f >> 1][v] : U0[v] - off[f >> 1][v];
        };
        constexpr bool POS = FLUX != FX_ROE && RECON != RC_PWC;
        if constexpr (POS) {
#pragma unroll
            for (int f = 0; f < 6; f++) {
                R u[NV];
                face_state(f, u);
                bad |= no_sound_speed(u) ? 1u << f : 0u;
            }
        }
        auto face_of = [&](int f, R (&u)[NV]) {
            face_state(f, u);
            if constexpr (POS) {
                if (__builtin_expect(bad & (1u << f), 0)) {
#pragma unroll
                    for (int v = 0; v < NV; v++) u[v] = U0[v];
                }
            }
        };
        // y-face between rows rc-1 and rc
        R G[NV], lamy = R(0), GL0 = R(0), GR0 = R(0);
        const R Sy = R(hx * hz);  // face area of a y-face (ERK:1269)
        if (out_plane && t >= 1) {
            R GL[NV], GR[NV];
#pragma unroll
            for (int v = 0; v < NV; v++) GL[v] = ytop[v];
            face_of(2, GR);
            if (!g.periodic[1]) {
                if (rc == 0) bc_image(g.bc[bc_marker(g, 2, ks * nx + xs)], gamma, 1, GR, GL);
                if (rc == ny) bc_image(g.bc[bc_marker(g, 3, ks * nx + xs)], gamma, 1, GL, GR);
            }
            if constexpr (MT::flux) face_flux<FLUX, 1, R>(gamma, eps, GL, GR, G, lamy);
            else lamy = face_eigen<FLUX, 1, R>(gamma, GL, GR);
            GL0 = GL[0];
            GR0 = GR[0];
            if constexpr (VIS && MT::flux) {
                if (a.v.viscous) {
                    const unsigned fi = (unsigned(ks) * unsigned(ny + 1) + unsigned(rc)) * unsigned(nx) + unsigned(xs);
#pragma unroll
                    for (int v = 1; v < NV; v++) G[v] -= R(ld_plane(a.v.fv[1], a.v.nface[1], v - 1, fi));
                }
            }
        }
        face_of(3, ytop);
        // (1) the previous row's z-fluxes are written, and its z+ face states (in slot sp) are read
        __syncthreads();
#pragma unroll
        for (int v = 0; v < NV; v++) ring[w][sp][v][lane] = Up[v];
        if (out_plane && t >= 1) {
            if constexpr (MT::sr) {
                if (t >= 2) {
                    double sr;
                    {
#pragma clang fp contract(off)
                        sr = srp + double(Sy * lamy);
                    }
                    if constexpr (VIS)
                        sr = sr + viscous_sr(double(GL0), double(GR0), g.gamma, a.v.mu, double(Sy), hx * hyp * hz);
                    {
#pragma clang fp contract(off)
                        sr = sr + double(Szb * lzb);
                        sr = sr + double(Szb * lds_l[w + 1][lane]);
                        if constexpr (VIS) sr = sr + lds_vz[w + 1][lane] / (hx * hyp * hz);
                    }
                    if (out_lane) block_min = __builtin_fmin(block_min, dt_candidate(hx * hyp * hz, sr));
                }
                if (rc == ny && out_lane)  // top ghost row (ERK:1305)
                    block_min = __builtin_fmin(block_min, dt_candidate(hx * g.h[1][ny + 1] * hz, double(Sy * lamy)));
                lam_gb = lamy;
            }
            if constexpr (MT::flux) {
                if (t >= 2) {
                    // finalize row rc-1, in slot sm
                    const int rf = rc - 1;
                    const double ivol = ihx * ihyp * ihz;
                    const unsigned off = (unsigned(ks) * unsigned(ny) + unsigned(rf)) * unsigned(nx) + unsigned(xs);
                    R resv[NV], Um[NV];
#pragma unroll
                    for (int v = 0; v < NV; v++) {
                        resv[v] = (dfx(v) - flux_difference(G[v], gbot(v)) * Sy) -
                                  flux_difference(lds_h[w + 1][v][lane], hbot(v)) * Szb;
                        Um[v] = ring[w][sm][v][lane];
                    }
                    if constexpr (VIS) add_sources(a.v, Um, hx * hyp * hz, resv);
#pragma unroll
                    for (int v = 0; v < NV; v++) {
                        R res = resv[v];
                        if constexpr (MODE == MODE_RN) {
                            if (out_lane) rn[v] += hx * hyp * hz * __builtin_fabs(double(res));
                        } else if constexpr (MODE == MODE_F1) {
                            if (out_lane) st_plane(uo, P, v, off, TOut(double(res) * ivol));
                        } else if (inc && MODE == MODE_F2) {
                            // FP32-residual stage 2: the increment dt/4 (L(U^n) + L(U1)) in float
                            // beside U2 (stage 3 accumulates U^n + 2/3 (D + dt L(U2)) in double)
                            const double d = 0.25 * dt * (double(Dc[v]) + double(res) * ivol);
                            if (out_lane) {
                                st_plane((TOut*)a.dout, P, v, off, TOut(d));
                                st_plane(uo, P, v, off, TOut(nc(v) + d));
                            }
                        } else if (inc && MODE == MODE_S3) {
                            const double d = double(Dc[v]);
                            const double q = nc(v) + (2.0 / 3.0) * (d + dt * (double(res) * ivol));
                            if (out_lane) st_plane(uo, P, v, off, TOut(q));
                        } else {
                            double q = double(Um[v]) + dt * (double(res) * ivol);
                            if constexpr (MT::use_un) q = MT::ca * nc(v) + MT::cb * q;
                            if (out_lane) st_plane(uo, P, v, off, TOut(q));
                        }
                    }
                }
#pragma unroll
                for (int v = 0; v < NV; v++) gbot(v) = G[v];
            }
        }
        // the z+ face state goes up through the slot of the finalized row
        {
            R up[NV];
            face_of(5, up);
#pragma unroll
            for (int v = 0; v < NV; v++) ring[w][sm][v][lane] = up[v];
        }
        __syncthreads();  // (2)
        if (!EARLY && t + 1 < nit) issue_cell(rc + 2, k, Pn);
        const R Sz = R(hx * hy);  // face area of a z-face (ERK:1349)
        R lamz = R(0);
        if (w >= 1 && row_out) {
            // the wavefront above each z-face evaluates it
            R ZL[NV], ZR[NV], H[NV];
#pragma unroll
            for (int v = 0; v < NV; v++) ZL[v] = ring[w - 1][sm][v][lane];
            face_of(4, ZR);
            if (!g.periodic[2]) {
                if (k == 0) bc_image(g.bc[bc_marker(g, 4, rcs * nx + xs)], gamma, 2, ZR, ZL);
                if (k == nz) bc_image(g.bc[bc_marker(g, 5, rcs * nx + xs)], gamma, 2, ZL, ZR);
            }
            if constexpr (MT::flux) face_flux<FLUX, 2, R>(gamma, eps, ZL, ZR, H, lamz);
            else lamz = face_eigen<FLUX, 2, R>(gamma, ZL, ZR);
            if constexpr (VIS && MT::flux) {
                if (a.v.viscous) {
                    const int kf = k < 0 ? 0 : (k > nz ? nz : k);
                    const unsigned fi = (unsigned(kf) * unsigned(ny) + unsigned(rcs)) * unsigned(nx) + unsigned(xs);
#pragma unroll
                    for (int v = 1; v < NV; v++) H[v] -= R(ld_plane(a.v.fv[2], a.v.nface[2], v - 1, fi));
                }
            }
            if constexpr (VIS && MT::sr) {
                // max(4/(3 rho_f), gamma/rho_f) mu Sz^2; the plane below divides by its volume
                const double ro = __builtin_sqrt(double(ZL[0]) * double(ZR[0]));
                const double va = 4.0 / (3.0 * ro), vb = g.gamma / ro;
                double vz = (va < vb) ? vb : va;
                vz *= a.v.mu / 1.0;
                vz *= double(Sz) * double(Sz);
                lds_vz[w][lane] = vz;
            }
            if constexpr (MT::flux) {
#pragma unroll
                for (int v = 0; v < NV; v++) {
                    lds_h[w][v][lane] = H[v];
                    if constexpr (YZ_REGS) Hb[v] = H[v];
                }
            }
            if constexpr (MT::sr) {
                lds_l[w][lane] = lamz;
                // top ghost plane: only the face below it (ERK:1385)
                if (k == nz && x_out)
                    block_min = __builtin_fmin(block_min, dt_candidate(hx * hy * g.h[2][nz + 1], double(Sz * lamz)));
            }
        }
        lzb = lamz;
        Szb = Sz;
        hyp = gc.h;
        ihyp = gc.ih;
        if (out_plane && row_out) {
            // x-faces of row rc
            R UL[NV], UR[NV];
            face_of(1, UL);
            face_of(0, UR);
#pragma unroll
            for (int v = 0; v < NV; v++) {
                UL[v] = dpp_from_left(UL[v]);
                // lane 0 has no left neighbour and its flux is not used: as in the 1-D stage
                if (FLUX == FX_GODUNOV && lane == 0) UL[v] = UR[v];
            }
            if (!g.periodic[0]) {
                if (xg == 0) bc_image(g.bc[bc_marker(g, 0, ks * ny + rcs)], gamma, 0, UR, UL);
                if (xg == nx) bc_image(g.bc[bc_marker(g, 1, ks * ny + rcs)], gamma, 0, UL, UR);
            }
            const R Sx = R(hy * hz);  // face area of an x-face (ERK:1190)
            R F[NV], lamx;
            if constexpr (MT::flux) face_flux<FLUX, 0, R>(gamma, eps, UL, UR, F, lamx);
            else lamx = face_eigen<FLUX, 0, R>(gamma, UL, UR);
            if constexpr (VIS && MT::flux) {
                if (a.v.viscous) {
                    const unsigned fi = (unsigned(ks) * unsigned(ny) + unsigned(rcs)) * unsigned(nx + 1) +
                                        unsigned(xg < 0 ? 0 : (xg > nx ? nx : xg));
#pragma unroll
                    for (int v = 1; v < NV; v++) F[v] -= R(ld_plane(a.v.fv[0], a.v.nface[0], v - 1, fi));
                }
            }
            if constexpr (MT::sr) {
                R lam_r = dpp_from_right(lamx);
                {
#pragma clang fp contract(off)
                    srp = double(Sx * lamx) + double(Sx * lam_r);
                }
                if constexpr (VIS) {
                    const double rl = dpp_from_right(double(UL[0])), rr = dpp_from_right(double(UR[0]));
                    srp = srp + viscous_sr(rl, rr, g.gamma, a.v.mu, double(Sx), hx * hy * hz);
                }
                {
#pragma clang fp contract(off)
                    srp = srp + double(Sy * lam_gb);
                }
                if (ghost_x_lane)  // right ghost column (ERK:1225)
                    block_min = __builtin_fmin(block_min, dt_candidate(g.h[0][nx + 1] * hy * hz, double(Sx * lamx)));
            }
            if constexpr (MT::flux) {
#pragma unroll
                for (int v = 0; v < NV; v++) dfx(v) = -(flux_difference(dpp_from_right(F[v]), F[v]) * Sx);
            }
        }
        if (!EARLY && edge && t + 1 < nit) issue_cell(rc + 1, k + zoff, Zq);  // (these have no x-faces)
        gc = gn;
        const int st = sm;
        sm = s0;
        s0 = sp;
        sp = st;
    }
    if constexpr (MT::sr) {
        // the workgroup's minimum, stored for its tile; dt_finalize_kernel follows the launch
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) block_min = __builtin_fmin(block_min, __shfl_xor(block_min, o));
        if (lane == 0) red[w] = block_min;
        __syncthreads();
        if (threadIdx.x == 0) {
            double m = red[0];
            for (int q = 1; q < ZW; q++) m = __builtin_fmin(m, red[q]);
            st_plane(a.dt_part, 0, 0, unsigned(tile), m);
        }
    }
    if constexpr (MODE == MODE_RN) {
        __shared__ double rred[ZW * NV];
        rn_reduce_finalize(ctl, a.rn_part, rn, rred, lane, w, ZW);
    }
}

}  // namespace tsd
