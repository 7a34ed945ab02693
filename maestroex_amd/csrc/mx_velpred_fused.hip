// mx_velpred_fused.hip -- fused 3-D VelPred: PPM of the three velocity
// components, the interface, transverse and final states and the Riemann
// solve of the MAC velocities in one z-marching kernel
// (MaestroVelPred.cpp:5-292 with VelPredInterface :735-1128,
// VelPredTransverse :1130-1595 and VelPredVelocities :1597-1915).
//
// Two kernels.  k_vp_fused_comp, the one in use: one velocity component per block,
// upwind first, three phases a plane (described above its code).  k_vp_fused: all
// three components per block, both sides of every face, for FABs whose rows the
// other's 32-bit offsets do not reach, and as the choice "velpred_fused_comp" 0.
//
// In both a block owns a TX x TY tile of cell columns of one box, grown by one cell
// in x and y (one thread per column), and marches up a chunk [z0, z1] of the
// box's planes, one cell plane q per step (plus q = z0 - 1 and q = z1 + 1).
// Nothing goes through HBM between the stages: the reference's sixteen
// temporaries (Ip/Im per component, the interface and upwind states, the six
// transverse states) live in LDS and registers.
//
// Names: iface(D, n) are the left/right interface states of velocity
// component n on D-faces, uimh(T, n) their upwind state by utrans; the
// transverse state pair (D, T) is component O = 3 - D - T on D-faces
// corrected by direction T (uimhyz = (1, 2), uimhzy = (2, 1), vimhxz =
// (0, 2), vimhzx = (2, 0), wimhxy = (0, 1), wimhyx = (1, 0)); umac on
// D-faces is corrected by the pairs (T, 3 - D - T), T != D.
//
// The reference formulas are regrouped, not changed: a transverse correction
// (dt/6h_T)(utrans_T(+) + utrans_T(-))(uimh_T(+) - uimh_T(-)) depends only on
// the cell it is taken across; the final corrections (dt/4h_T) likewise.  Each is
// the reference's expression in the reference's operand order, so the
// results are bit-identical to the per-point kernels.  PPM boundary stencils
// (ext_dir / hoextrap within three cells of a domain side) use the full
// per-cell routine of mx_device.H; the tracing velocity is ufull at the cell
// (is_umac = 0).
//
// k_vp_fused evaluates a correction once per cell for the faces on both sides.  Per
// step q, phases separated by barriers:
//   A  stage plane q of the three components and of utrans_x, utrans_y;
//      shift the column's z windows; issue the loads of plane q + 1;
//   B1 face values of plane q (x, y, three components); PPM of cell q in z
//      (register windows) and the z-face q interface / upwind states;
//   B2 PPM of plane q in x and y;
//   C  interface and upwind states on the x- and y-faces of plane q;
//   D1 per-cell transverse corrections: x, y of plane q, z of plane q - 1;
//   D2 transverse states wimhxy, wimhyx (plane q), vimhxz, uimhyz (plane
//      q - 1), vimhzx, uimhzy (z-face q, registers);
//   E1 per-cell final corrections: plane q - 1 (x, y faces), plane q (z);
//   E2 umac, vmac on the faces of plane q - 1 and wmac on z-face q.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "mx_internal.H"
#include "mx_march.H"

using namespace mxd;
using namespace mxh;

namespace {

__host__ __device__ constexpr int vf_nt(int tx, int ty) {
    return ((tx + 2) * (ty + 2) + 63) / 64 * 64;
}

struct VFBox {
    int lo[3], hi[3];
    DA ut, uf, fo, w0c;
    DA tr[3], um[3], w0m[3];
    double dx[3];
    int domlo[3], domhi[3];
    // plane strides in bytes: utilde, force, ufull, utrans x / y / z, umac x / y /
    // z, w0mac x / y / z, w0_cart; the cell widths as divisors
    long long ks[13];
    DivBy h[3];
    const double* w0a;  // Addw0 at the store of umac: the planar w0
    int add;
    int pad_ = 0;  // explicit, so that equal tables are equal byte for byte
};

struct VFTile {
    int box, tx, ty, tzc;
};

struct VFArgs {
    int bclo[3][3], bchi[3][3];  // bcs_u[n].lo/hi[dir] (BCType)
    int plo[3], phi[3];          // phys_bc lo/hi (PhysBCType)
    int spherical;
    int tz;
    double dt, rel_eps, dt4, dt6;
};

// VelPredInterface overrides of the (l, r) pair of a component on a face at
// `pos` (3-D; MaestroVelPred.cpp:790-875): `normal` when the component is the
// face's normal velocity, ulo / uhi the cell values below / above the face
__device__ __forceinline__ void vf_iface_bc(int pos, int dlo, int dhi, int bclo, int bchi,
                                            bool normal, double ulo, double uhi, double& l,
                                            double& r) {
    if (pos == dlo) {
        switch (bclo) {
            case MX_PHYS_INFLOW:
                l = ulo;
                r = l;
                break;
            case MX_PHYS_SLIPWALL:
            case MX_PHYS_SYMMETRY:
                if (normal) {
                    l = 0.0;
                    r = 0.0;
                } else {
                    l = r;
                }
                break;
            case MX_PHYS_NOSLIPWALL:
                l = 0.0;
                r = 0.0;
                break;
            case MX_PHYS_OUTFLOW:
                if (normal) r = dmin(r, 0.0);
                l = r;
                break;
            default:
                break;
        }
    } else if (pos == dhi + 1) {
        switch (bchi) {
            case MX_PHYS_INFLOW:
                l = uhi;
                r = l;
                break;
            case MX_PHYS_SLIPWALL:
            case MX_PHYS_SYMMETRY:
                if (normal) {
                    l = 0.0;
                    r = 0.0;
                } else {
                    r = l;
                }
                break;
            case MX_PHYS_NOSLIPWALL:
                l = 0.0;
                r = 0.0;
                break;
            case MX_PHYS_OUTFLOW:
                if (normal) l = dmax(l, 0.0);
                r = l;
                break;
            default:
                break;
        }
    }
}

// VelPredTransverse overrides after the correction (MaestroVelPred.cpp:1183-1230)
__device__ __forceinline__ void vf_trans_bc(int pos, int dlo, int dhi, int bclo, int bchi,
                                            double ulo, double uhi, double& l, double& r) {
    if (pos == dlo) {
        switch (bclo) {
            case MX_PHYS_INFLOW:
                l = ulo;
                r = l;
                break;
            case MX_PHYS_SLIPWALL:
            case MX_PHYS_SYMMETRY:
            case MX_PHYS_OUTFLOW:
                l = r;
                break;
            case MX_PHYS_NOSLIPWALL:
                l = 0.0;
                r = 0.0;
                break;
            default:
                break;
        }
    } else if (pos == dhi + 1) {
        switch (bchi) {
            case MX_PHYS_INFLOW:
                l = uhi;
                r = l;
                break;
            case MX_PHYS_SLIPWALL:
            case MX_PHYS_SYMMETRY:
            case MX_PHYS_OUTFLOW:
                r = l;
                break;
            case MX_PHYS_NOSLIPWALL:
                l = 0.0;
                r = 0.0;
                break;
            default:
                break;
        }
    }
}

// upwind by a transverse velocity, averaging below rel_eps (MaestroVelPred.cpp:887-896)
__device__ __forceinline__ double vf_upwind(double l, double r, double t, double rel_eps) {
    double res = t > 0.0 ? l : r;
    res = dabs(t) < rel_eps ? 0.5 * (l + r) : res;
    return res;
}

// the Riemann solve of VelPredVelocities, with w0 where it acts
// (MaestroVelPred.cpp:1690-1715)
__device__ __forceinline__ double vf_riemann(double umacl, double umacr, bool has_w, double w,
                                             double rel_eps) {
    if (has_w) {
        const bool test = (umacl + w <= 0.0 && umacr + w >= 0.0) ||
                          (dabs(umacl + umacr + 2.0 * w) < rel_eps);
        const double res = 0.5 * (umacl + umacr) + w > 0.0 ? umacl : umacr;
        return test ? 0.0 : res;
    }
    const bool test = (umacl <= 0.0 && umacr >= 0.0) || (dabs(umacl + umacr) < rel_eps);
    const double res = 0.5 * (umacl + umacr) > 0.0 ? umacl : umacr;
    return test ? 0.0 : res;
}

// the overrides after the Riemann solve (MaestroVelPred.cpp:1717-1750)
__device__ __forceinline__ double vf_vel_bc(double res, int pos, int dlo, int dhi, int bclo,
                                            int bchi, double ulo, double uhi, double umacl,
                                            double umacr) {
    if (pos == dlo) {
        switch (bclo) {
            case MX_PHYS_INFLOW: res = ulo; break;
            case MX_PHYS_SLIPWALL:
            case MX_PHYS_SYMMETRY:
            case MX_PHYS_NOSLIPWALL: res = 0.0; break;
            case MX_PHYS_OUTFLOW: res = dmin(umacr, 0.0); break;
            default: break;
        }
    } else if (pos == dhi + 1) {
        switch (bchi) {
            case MX_PHYS_INFLOW: res = uhi; break;
            case MX_PHYS_SLIPWALL:
            case MX_PHYS_SYMMETRY:
            case MX_PHYS_NOSLIPWALL: res = 0.0; break;
            case MX_PHYS_OUTFLOW: res = dmax(umacl, 0.0); break;
            default: break;
        }
    }
    return res;
}

// PPM edge values of a cell from its face values (type 1) or its stencil and
// face values (type 2), with the boundary stencils where they act
template <int PPM, int D>
__device__ __forceinline__ void vf_cell_edges(const double* w9, const double* F, int fst, int pos,
                                              int dlo, int dhi, int bclo, int bchi,
                                              bool check_bc, double& sm, double& sp) {
    if (PPM == 1) {
        sm = F[0];
        sp = F[fst];
        cw_limit(w9[4], sm, sp);
    } else {
        cs_cell(w9, F[-fst], F[0], F[fst], F[2 * fst], 1.e-10, sm, sp);
    }
    if (check_bc && ppm_special<PPM>(pos, dlo, dhi, bclo, bchi))
        ppm_edges<PPM, D>(w9, pos, dlo, dhi, bclo, bchi, sm, sp);
}

// XYF: no x- or y-boundary condition acts on the tile (no PPM boundary
// stencil and no physical-boundary override within the tile's reach)
template <int PPM, int TX, int TY, bool XYF, int WPE>
__global__ void __launch_bounds__(vf_nt(TX, TY)) __attribute__((amdgpu_waves_per_eu(WPE)))
    k_vp_fused(const VFBox* __restrict__ boxes, const VFTile* __restrict__ tiles, KGeom g,
               VFArgs A) {
    constexpr int NT = vf_nt(TX, TY);
    constexpr int G = PPM == 2 ? 3 : 2;
    constexpr int W = TX + 2;
    constexpr int H = TY + 2;
    constexpr int NE = W * H;
    constexpr int SW = W + 2 * G;
    constexpr int SH = H + 2 * G;
    constexpr int UW = W + 1;  // x-faces per row of the utrans_x plane
    constexpr int VH = H + 1;  // y-faces per column of the utrans_y plane
    constexpr int FO = PPM == 2 ? 1 : 0;
    constexpr int FXW = W + 1 + 2 * FO;  // x-face values per row
    constexpr int FYH = H + 1 + 2 * FO;  // y-face values per column
    constexpr int NF = FXW * H > W * FYH ? FXW * H : W * FYH;
    static_assert(NE <= NT, "tile too large for the block");

    __shared__ double S[3][SW * SH];
    __shared__ double UL[3][UW * H];
    __shared__ double VL[3][W * VH];
    __shared__ double FX[3][NF];   // x-face values; later phases reuse it
    __shared__ double FY[3][NF];   // y-face values; later phases reuse it
    __shared__ double P[12][NE];   // Ipx, Imx, Ipy, Imy per component
    __shared__ double SC[3][NE];   // plane q - 1 cell values (inflow overrides)
    __shared__ double FL[2][NE];   // plane q - 1 forces, x and y components

    const VFTile tl = tiles[blockIdx.x];
    const VFBox& B = boxes[tl.box];
    const int bhi0 = B.hi[0], bhi1 = B.hi[1], bhi2 = B.hi[2];
    const int X0 = B.lo[0] + tl.tx * TX;
    const int Y0 = B.lo[1] + tl.ty * TY;
    const int nx = min(TX, bhi0 - X0 + 1);
    const int ny = min(TY, bhi1 - Y0 + 1);
    const int z0 = B.lo[2] + tl.tzc * A.tz;
    const int z1 = min(z0 + A.tz - 1, bhi2);
    const bool last_x = (X0 + nx - 1 == bhi0);
    const bool last_y = (Y0 + ny - 1 == bhi1);
    const bool last_z = (z1 == bhi2);
    const int dlx = B.domlo[0], dhx = B.domhi[0];
    const int dly = B.domlo[1], dhy = B.domhi[1];
    const int dlz = B.domlo[2], dhz = B.domhi[2];
    const int pxl = A.plo[0], pxh = A.phi[0], pyl = A.plo[1], pyh = A.phi[1];
    const int pzl = A.plo[2], pzh = A.phi[2];
    const bool sph = A.spherical != 0;

    const DA utv = B.ut, ufv = B.uf, fov = B.fo;
    const DA trx = B.tr[0], tryv = B.tr[1], trz = B.tr[2];
    const DA umx = B.um[0], umy = B.um[1], umz = B.um[2];
    const int sjs = (int)utv.js, sks = (int)utv.ks, sns = (int)utv.ns;
    const int xjs = (int)trx.js, xks = (int)trx.ks;
    const int yjs = (int)tryv.js, yks = (int)tryv.ks;

    const int tid = threadIdx.x;
    const int a = tid % W;  // local column: cell (X0 + a - 1, Y0 + b - 1)
    const int b = tid / W;
    const bool col = (tid < NE) && (a <= nx + 1) && (b <= ny + 1);
    const int I = X0 + a - 1;
    const int J = Y0 + b - 1;
    const int si = (a + G) + (b + G) * SW;
    const int ui = a + b * UW;
    const int vi = a + b * W;

    const double dt = g.dt;
    const double rel_eps = g.rel_eps;
    const double dt2 = 0.5 * dt;
    const double dt4 = 0.25 * dt;
    const double dt6 = dt / 6.0;
    const double hx = B.dx[0], hy = B.dx[1], hz = B.dx[2];
    const double t6x = dt6 / hx, t6y = dt6 / hy, t6z = dt6 / hz;
    const double t4x = dt4 / hx, t4y = dt4 / hy, t4z = dt4 / hz;

    // plane pointers (block-uniform) at plane z0 - 1
    gcd* sPl = (gcd*)utv.p + utv.off(X0 - 1 - G, Y0 - 1 - G, z0 - 1);
    gcd* xPl = (gcd*)trx.p + trx.off(X0 - 1, Y0 - 1, z0 - 1);
    gcd* yPl = (gcd*)tryv.p + tryv.off(X0 - 1, Y0 - 1, z0 - 1);
    // column pointers
    gcd* sCol = (gcd*)utv.p;
    gcd* ufCol = (gcd*)ufv.p;
    gcd* foCol = (gcd*)fov.p;
    gcd* zCol = (gcd*)trz.p;
    gd* oxCol = (gd*)umx.p;
    gd* oyCol = (gd*)umy.p;
    gd* ozCol = (gd*)umz.p;
    if (col) {
        sCol += utv.off(I, J, z0 - 1 + G);  // next z-window load: s(q + G)
        ufCol += ufv.off(I, J, z0 - 1);
        foCol += fov.off(I, J, z0 - 1);
        zCol += trz.off(I, J, z0 - 1);
        oxCol += umx.off(I, J, z0 - 1);
        oyCol += umy.off(I, J, z0 - 1);
        ozCol += umz.off(I, J, z0 - 1);
    }
    const int ufks = (int)ufv.ks, ufns = (int)ufv.ns;
    const int foks = (int)fov.ks, fons = (int)fov.ns;
    const int zks = (int)trz.ks;
    const int oxks = (int)umx.ks, oyks = (int)umy.ks, ozks = (int)umz.ks;

    // column state
    double v[3][9];
#pragma unroll
    for (int n = 0; n < 3; ++n)
#pragma unroll
        for (int jj = 0; jj < 9; ++jj) v[n][jj] = 0.0;
    double zf0[3] = {0.0, 0.0, 0.0}, zf1[3] = {0.0, 0.0, 0.0}, zf2[3] = {0.0, 0.0, 0.0};
    double zsl[3] = {0.0, 0.0, 0.0};
    double Ipz_prev[3] = {0.0, 0.0, 0.0};
    double zl[3] = {0.0, 0.0, 0.0}, zr[3] = {0.0, 0.0, 0.0};  // iface(2, n) on z-face q
    double uz_q[2] = {0.0, 0.0}, uz_p[2] = {0.0, 0.0};        // uimh(2, 0), uimh(2, 1)
    double xl0_p = 0.0, xr0_p = 0.0, xl1_p = 0.0, xr1_p = 0.0;  // iface(0, 0/1), plane p
    double yl1_p = 0.0, yr1_p = 0.0, yl0_p = 0.0, yr0_p = 0.0;  // iface(1, 1/0), plane p
    double xl[3] = {0.0, 0.0, 0.0}, xr[3] = {0.0, 0.0, 0.0};
    double yl[3] = {0.0, 0.0, 0.0}, yr[3] = {0.0, 0.0, 0.0};
    double t01_q = 0.0, t01_p = 0.0, t10_q = 0.0, t10_p = 0.0;  // own-column corrections
    double p201_q = 0.0, p201_p = 0.0, p210_q = 0.0, p210_p = 0.0;  // vimhzx, uimhzy
    double ez0_q = 0.0, ez0_p = 0.0, ez1_q = 0.0, ez1_p = 0.0;  // wmac corrections
    double trz_q = 0.0, trz_p = 0.0;
    double uf_q[3] = {0.0, 0.0, 0.0};
    double fo_q[3] = {0.0, 0.0, 0.0}, foz_p = 0.0;
    if (col) {
#pragma unroll
        for (int n = 0; n < 3; ++n)
            for (int jj = 5 - G; jj <= 4 + G; ++jj) v[n][jj] = utv(I, J, z0 - 6 + jj, n);
    }
    int slot_q = 0, slot_p = 2;

    // plane q + 1's loads are issued during step q (the barriers wait for LDS
    // traffic only); each thread owns fixed slots of the staged planes
    constexpr int NS = (SW * SH + NT - 1) / NT;
    constexpr int NU = (UW * H + NT - 1) / NT;
    constexpr int NV = (W * VH + NT - 1) / NT;
    bool okS[NS], okU[NU], okV[NV];
    int offS[NS], offU[NU], offV[NV];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int idx = tid + k * NT;
        const int sx = idx % SW, sy = idx / SW;
        okS[k] = idx < SW * SH && sx <= nx + 1 + 2 * G && sy <= ny + 1 + 2 * G;
        offS[k] = sx + sy * sjs;
    }
#pragma unroll
    for (int k = 0; k < NU; ++k) {
        const int idx = tid + k * NT;
        const int f = idx % UW, r = idx / UW;
        okU[k] = idx < UW * H && f <= nx + 2 && r <= ny + 1;
        offU[k] = f + r * xjs;
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int idx = tid + k * NT;
        const int cc = idx % W, r = idx / W;
        okV[k] = idx < W * VH && cc <= nx + 1 && r <= ny + 2;
        offV[k] = cc + r * yjs;
    }
    double pS[3][NS], pU[NU], pV[NV];
    double pcs[3] = {0.0, 0.0, 0.0}, puf[3] = {0.0, 0.0, 0.0}, pfo[3] = {0.0, 0.0, 0.0};
    double pz = 0.0;
#pragma unroll
    for (int k = 0; k < NS; ++k)
#pragma unroll
        for (int n = 0; n < 3; ++n) pS[n][k] = okS[k] ? sPl[offS[k] + n * sns] : 0.0;
#pragma unroll
    for (int k = 0; k < NU; ++k) pU[k] = okU[k] ? xPl[offU[k]] : 0.0;
#pragma unroll
    for (int k = 0; k < NV; ++k) pV[k] = okV[k] ? yPl[offV[k]] : 0.0;
    if (col) {
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            pcs[n] = sCol[n * sns];
            puf[n] = ufCol[n * ufns];
            pfo[n] = foCol[n * fons];
        }
        pz = *zCol;
    }

    for (int q = z0 - 1; q <= z1 + 1; ++q) {
        const bool zface = q >= z0;        // z-face q is in the chunk's range
        const bool pplane = q >= z0 + 1;   // plane p = q - 1 is a chunk plane
        const bool first = q == z0 - 1;
        double* ULq = UL[slot_q];
        double* VLq = VL[slot_q];
        const double* ULp = UL[slot_p];
        const double* VLp = VL[slot_p];

        // ---- A: stage plane q; shift the column windows; issue the loads
        //      of plane q + 1
#pragma unroll
        for (int k = 0; k < NS; ++k)
            if (okS[k]) {
#pragma unroll
                for (int n = 0; n < 3; ++n) S[n][tid + k * NT] = pS[n][k];
            }
#pragma unroll
        for (int k = 0; k < NU; ++k)
            if (okU[k]) ULq[tid + k * NT] = pU[k];
#pragma unroll
        for (int k = 0; k < NV; ++k)
            if (okV[k]) VLq[tid + k * NT] = pV[k];
        double flx = 0.0, fly = 0.0;  // plane q - 1 forces, x and y
        if (col) {
#pragma unroll
            for (int n = 0; n < 3; ++n) {
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) v[n][jj] = v[n][jj + 1];
                v[n][4 + G] = pcs[n];
            }
            flx = fo_q[0];
            fly = fo_q[1];
            foz_p = fo_q[2];
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                uf_q[n] = puf[n];
                fo_q[n] = pfo[n];
            }
            trz_p = trz_q;
            trz_q = pz;
        }
        if (q <= z1) {
            sPl += sks;
            xPl += xks;
            yPl += yks;
#pragma unroll
            for (int k = 0; k < NS; ++k)
                if (okS[k]) {
#pragma unroll
                    for (int n = 0; n < 3; ++n) pS[n][k] = sPl[offS[k] + n * sns];
                }
#pragma unroll
            for (int k = 0; k < NU; ++k)
                if (okU[k]) pU[k] = xPl[offU[k]];
#pragma unroll
            for (int k = 0; k < NV; ++k)
                if (okV[k]) pV[k] = yPl[offV[k]];
            if (col) {
                sCol += sks;
                ufCol += ufks;
                foCol += foks;
                zCol += zks;
#pragma unroll
                for (int n = 0; n < 3; ++n) {
                    pcs[n] = sCol[n * sns];
                    puf[n] = ufCol[n * ufns];
                    pfo[n] = foCol[n * fons];
                }
                pz = *zCol;
            }
        }
        __syncthreads();

        // plane q - 1's cell values and forces, which D2 and E2 read across
        // columns: stored after the barrier above, which no thread passes
        // before every thread is done with the previous plane's E2
        if (col) {
#pragma unroll
            for (int n = 0; n < 3; ++n) SC[n][tid] = v[n][3];
            FL[0][tid] = flx;
            FL[1][tid] = fly;
        }

        // ---- B1: face values of plane q; PPM of cell q in z
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            const double* Sn = S[n];
            for (int idx = tid; idx < FXW * H; idx += NT) {
                const int f = idx % FXW - FO, r = idx / FXW;  // face f: cells f-1 | f
                if (f <= nx + 2 + FO && r <= ny + 1) {
                    const double* sr = Sn + (f + G) + (r + G) * SW;
                    if (PPM == 1) {
                        const double sa2 = sr[-2], sa = sr[-1], sb = sr[0], sb2 = sr[1];
                        FX[n][idx] = face1(sa, sb, vl_slope(sa2, sa, sb), vl_slope(sa, sb, sb2));
                    } else {
                        FX[n][idx] = cs_face(sr[-2], sr[-1], sr[0], sr[1]);
                    }
                }
            }
            for (int idx = tid; idx < W * FYH; idx += NT) {
                const int c = idx % W, f = idx / W - FO;  // face f: cells f-1 | f
                if (c <= nx + 1 && f <= ny + 2 + FO) {
                    const double* sr = Sn + (c + G) + (f + G) * SW;
                    if (PPM == 1) {
                        const double sa2 = sr[-2 * SW], sa = sr[-SW], sb = sr[0], sb2 = sr[SW];
                        FY[n][idx] = face1(sa, sb, vl_slope(sa2, sa, sb), vl_slope(sa, sb, sb2));
                    } else {
                        FY[n][idx] = cs_face(sr[-2 * SW], sr[-SW], sr[0], sr[SW]);
                    }
                }
            }
        }
        if (col) {
            const double sgz = dabs(uf_q[2]) * dt / hz;
            double Ipz[3], Imz[3];
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                double* vn = v[n];
                double sm, sp;
                if (PPM == 1) {
                    if (first) {
                        const double d0 = vl_slope(vn[2], vn[3], vn[4]);
                        zsl[n] = vl_slope(vn[3], vn[4], vn[5]);
                        zf0[n] = face1(vn[3], vn[4], d0, zsl[n]);
                    }
                    const double d1 = vl_slope(vn[4], vn[5], vn[6]);
                    zf1[n] = face1(vn[4], vn[5], zsl[n], d1);
                    zsl[n] = d1;
                    sm = zf0[n];
                    sp = zf1[n];
                    cw_limit(vn[4], sm, sp);
                } else {
                    if (first) {
                        zf0[n] = cs_face(vn[1], vn[2], vn[3], vn[4]);
                        zf1[n] = cs_face(vn[2], vn[3], vn[4], vn[5]);
                        zf2[n] = cs_face(vn[3], vn[4], vn[5], vn[6]);
                    }
                    const double f3 = cs_face(vn[4], vn[5], vn[6], vn[7]);
                    cs_cell(vn, zf0[n], zf1[n], zf2[n], f3, 1.e-10, sm, sp);
                    zf0[n] = zf1[n];
                    zf1[n] = zf2[n];
                    zf2[n] = f3;
                }
                if (ppm_special<PPM>(q, dlz, dhz, A.bclo[n][2], A.bchi[n][2]))
                    ppm_edges<PPM, 2>(vn, q, dlz, dhz, A.bclo[n][2], A.bchi[n][2], sm, sp);
                if (PPM == 1) zf0[n] = zf1[n];
                trace_sig(vn[4], sm, sp, uf_q[2], uf_q[2], sgz, sgz, rel_eps, Ipz[n], Imz[n]);
            }
            if (zface) {
#pragma unroll
                for (int n = 0; n < 3; ++n) {
                    zl[n] = Ipz_prev[n];
                    zr[n] = Imz[n];
                    vf_iface_bc(q, dlz, dhz, pzl, pzh, n == 2, v[n][3], v[n][4], zl[n], zr[n]);
                }
                uz_q[0] = vf_upwind(zl[0], zr[0], trz_q, rel_eps);
                uz_q[1] = vf_upwind(zl[1], zr[1], trz_q, rel_eps);
            }
#pragma unroll
            for (int n = 0; n < 3; ++n) Ipz_prev[n] = Ipz[n];
        }
        __syncthreads();

        // ---- B2: PPM of plane q in x and y
        if (col) {
            const double sgx = dabs(uf_q[0]) * dt / hx;
            const double sgy = dabs(uf_q[1]) * dt / hy;
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                double sm, sp, Ip, Im;
                double w9[9];
#pragma unroll
                for (int o = -4; o <= 4; ++o)
                    w9[4 + o] = (o >= -G && o <= G) ? S[n][si + o] : 0.0;
                vf_cell_edges<PPM, 0>(w9, FX[n] + (a + FO) + b * FXW, 1, I, dlx, dhx,
                                      A.bclo[n][0], A.bchi[n][0], !XYF, sm, sp);
                trace_sig(w9[4], sm, sp, uf_q[0], uf_q[0], sgx, sgx, rel_eps, Ip, Im);
                P[4 * n][tid] = Ip;
                P[4 * n + 1][tid] = Im;
#pragma unroll
                for (int o = -4; o <= 4; ++o)
                    w9[4 + o] = (o >= -G && o <= G) ? S[n][si + o * SW] : 0.0;
                vf_cell_edges<PPM, 1>(w9, FY[n] + a + (b + FO) * W, W, J, dly, dhy,
                                      A.bclo[n][1], A.bchi[n][1], !XYF, sm, sp);
                trace_sig(w9[4], sm, sp, uf_q[1], uf_q[1], sgy, sgy, rel_eps, Ip, Im);
                P[4 * n + 2][tid] = Ip;
                P[4 * n + 3][tid] = Im;
            }
        }
        __syncthreads();

        // ---- C: interface and upwind states on the x- and y-faces of plane q
        //      (FX[0..1] <- uimh(0, 1), uimh(0, 2); FY[0..1] <- uimh(1, 0), uimh(1, 2))
        if (col && a >= 1) {
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                xl[n] = P[4 * n][tid - 1];
                xr[n] = P[4 * n + 1][tid];
                if (!XYF)
                    vf_iface_bc(I, dlx, dhx, pxl, pxh, n == 0, S[n][si - 1], S[n][si], xl[n],
                                xr[n]);
            }
            const double t = ULq[ui];
            FX[0][tid] = vf_upwind(xl[1], xr[1], t, rel_eps);
            FX[1][tid] = vf_upwind(xl[2], xr[2], t, rel_eps);
        }
        if (col && b >= 1) {
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                yl[n] = P[4 * n + 2][tid - W];
                yr[n] = P[4 * n + 3][tid];
                if (!XYF)
                    vf_iface_bc(J, dly, dhy, pyl, pyh, n == 1, S[n][si - SW], S[n][si], yl[n],
                                yr[n]);
            }
            const double t = VLq[vi];
            FY[0][tid] = vf_upwind(yl[0], yr[0], t, rel_eps);
            FY[1][tid] = vf_upwind(yl[2], yr[2], t, rel_eps);
        }
        __syncthreads();

        // ---- D1: per-cell transverse corrections
        //      P[0] <- (y; w) plane q, P[1] <- (x; w) plane q,
        //      P[2] <- (z; v) plane p, P[3] <- (z; u) plane p
        if (col) {
            if (a >= 1 && a <= nx) {
                const double s = ULq[ui + 1] + ULq[ui];
                t01_q = t6x * s * (FX[0][tid + 1] - FX[0][tid]);       // (x; v)
                P[1][tid] = t6x * s * (FX[1][tid + 1] - FX[1][tid]);  // (x; w)
            }
            if (b >= 1 && b <= ny) {
                const double s = VLq[vi + W] + VLq[vi];
                t10_q = t6y * s * (FY[0][tid + W] - FY[0][tid]);       // (y; u)
                P[0][tid] = t6y * s * (FY[1][tid + W] - FY[1][tid]);  // (y; w)
            }
            if (pplane) {
                const double s = trz_q + trz_p;
                P[2][tid] = t6z * s * (uz_q[1] - uz_p[1]);  // (z; v)
                P[3][tid] = t6z * s * (uz_q[0] - uz_p[0]);  // (z; u)
            }
        }
        __syncthreads();

        // ---- D2: transverse states
        //      FX[2] <- wimhxy (x-faces, plane q), FY[2] <- wimhyx (y-faces, q),
        //      P[4] <- vimhxz (x-faces, plane p), P[5] <- uimhyz (y-faces, p)
        if (col && a >= 1 && b >= 1 && b <= ny) {  // wimhxy: w on x-faces, by y
            double l = xl[2] - P[0][tid - 1];
            double r = xr[2] - P[0][tid];
            if (!XYF) vf_trans_bc(I, dlx, dhx, pxl, pxh, S[2][si - 1], S[2][si], l, r);
            FX[2][tid] = vf_upwind(l, r, ULq[ui], rel_eps);
        }
        if (col && b >= 1 && a >= 1 && a <= nx) {  // wimhyx: w on y-faces, by x
            double l = yl[2] - P[1][tid - W];
            double r = yr[2] - P[1][tid];
            if (!XYF) vf_trans_bc(J, dly, dhy, pyl, pyh, S[2][si - SW], S[2][si], l, r);
            FY[2][tid] = vf_upwind(l, r, VLq[vi], rel_eps);
        }
        if (pplane && col && a >= 1) {  // vimhxz: v on x-faces of plane p, by z
            double l = xl1_p - P[2][tid - 1];
            double r = xr1_p - P[2][tid];
            if (!XYF) vf_trans_bc(I, dlx, dhx, pxl, pxh, SC[1][tid - 1], SC[1][tid], l, r);
            P[4][tid] = vf_upwind(l, r, ULp[ui], rel_eps);
        }
        if (pplane && col && b >= 1) {  // uimhyz: u on y-faces of plane p, by z
            double l = yl0_p - P[3][tid - W];
            double r = yr0_p - P[3][tid];
            if (!XYF) vf_trans_bc(J, dly, dhy, pyl, pyh, SC[0][tid - W], SC[0][tid], l, r);
            P[5][tid] = vf_upwind(l, r, VLp[vi], rel_eps);
        }
        if (zface && col && a >= 1 && a <= nx) {  // vimhzx: v on z-face q, by x
            double l = zl[1] - t01_p;
            double r = zr[1] - t01_q;
            vf_trans_bc(q, dlz, dhz, pzl, pzh, v[1][3], v[1][4], l, r);
            p201_q = vf_upwind(l, r, trz_q, rel_eps);
        }
        if (zface && col && b >= 1 && b <= ny) {  // uimhzy: u on z-face q, by y
            double l = zl[0] - t10_p;
            double r = zr[0] - t10_q;
            vf_trans_bc(q, dlz, dhz, pzl, pzh, v[0][3], v[0][4], l, r);
            p210_q = vf_upwind(l, r, trz_q, rel_eps);
        }
        __syncthreads();

        // ---- E1: per-cell final corrections
        //      P[6], P[7] <- umac's (y), (z) of plane p; P[8], P[9] <- vmac's (x), (z)
        if (col && a >= 1 && a <= nx && b >= 1 && b <= ny) {  // wmac's, plane q
            ez0_q = t4x * (ULq[ui + 1] + ULq[ui]) * (FX[2][tid + 1] - FX[2][tid]);
            ez1_q = t4y * (VLq[vi + W] + VLq[vi]) * (FY[2][tid + W] - FY[2][tid]);
        }
        if (pplane && col) {
            const double s = trz_q + trz_p;
            if (b >= 1 && b <= ny) {  // umac's: uimhyz across y, uimhzy across z
                P[6][tid] = t4y * (VLp[vi + W] + VLp[vi]) * (P[5][tid + W] - P[5][tid]);
                P[7][tid] = t4z * s * (p210_q - p210_p);
            }
            if (a >= 1 && a <= nx) {  // vmac's: vimhxz across x, vimhzx across z
                P[8][tid] = t4x * (ULp[ui + 1] + ULp[ui]) * (P[4][tid + 1] - P[4][tid]);
                P[9][tid] = t4z * s * (p201_q - p201_p);
            }
        }
        __syncthreads();

        // ---- E2: MAC velocities
        if (pplane && col && a >= 1 && b >= 1 && b <= ny && (a <= nx || last_x)) {  // umac, p
            double vl = xl0_p - P[6][tid - 1];
            vl = vl - P[7][tid - 1];
            double vr = xr0_p - P[6][tid];
            vr = vr - P[7][tid];
            const double umacl = vl + dt2 * FL[0][tid - 1];
            const double umacr = vr + dt2 * FL[0][tid];
            const double w = sph ? B.w0m[0](I, J, q - 1) : 0.0;
            double res = vf_riemann(umacl, umacr, sph, w, rel_eps);
            if (!XYF)
                res = vf_vel_bc(res, I, dlx, dhx, pxl, pxh, SC[0][tid - 1], SC[0][tid], umacl,
                                umacr);
            oxCol[-oxks] = res;  // plane p
        }
        if (pplane && col && b >= 1 && a >= 1 && a <= nx && (b <= ny || last_y)) {  // vmac, p
            double vl = yl1_p - P[8][tid - W];
            vl = vl - P[9][tid - W];
            double vr = yr1_p - P[8][tid];
            vr = vr - P[9][tid];
            const double umacl = vl + dt2 * FL[1][tid - W];
            const double umacr = vr + dt2 * FL[1][tid];
            const double w = sph ? B.w0m[1](I, J, q - 1) : 0.0;
            double res = vf_riemann(umacl, umacr, sph, w, rel_eps);
            if (!XYF)
                res = vf_vel_bc(res, J, dly, dhy, pyl, pyh, SC[1][tid - W], SC[1][tid], umacl,
                                umacr);
            oyCol[-oyks] = res;  // plane p
        }
        if (((zface && q <= z1) || (q == z1 + 1 && last_z)) && col && a >= 1 && a <= nx &&
            b >= 1 && b <= ny) {  // wmac, z-face q
            double vl = zl[2] - ez0_p;
            vl = vl - ez1_p;
            double vr = zr[2] - ez0_q;
            vr = vr - ez1_q;
            const double umacl = vl + dt2 * foz_p;
            const double umacr = vr + dt2 * fo_q[2];
            // planar: w0_cart of the cell at the face's index (MaestroVelPred.cpp:1880)
            const double w = sph ? B.w0m[2](I, J, q) : B.w0c(I, J, q, 2);
            double res = vf_riemann(umacl, umacr, true, w, rel_eps);
            res = vf_vel_bc(res, q, dlz, dhz, pzl, pzh, v[2][3], v[2][4], umacl, umacr);
            *ozCol = res;  // z-face q
        }

        // ---- advance the column state to the next plane
        xl0_p = xl[0];
        xr0_p = xr[0];
        xl1_p = xl[1];
        xr1_p = xr[1];
        yl0_p = yl[0];
        yr0_p = yr[0];
        yl1_p = yl[1];
        yr1_p = yr[1];
        uz_p[0] = uz_q[0];
        uz_p[1] = uz_q[1];
        t01_p = t01_q;
        t10_p = t10_q;
        p201_p = p201_q;
        p210_p = p210_q;
        ez0_p = ez0_q;
        ez1_p = ez1_q;
        oxCol += oxks;
        oyCol += oyks;
        ozCol += ozks;
        slot_p = slot_q;
        slot_q = slot_q == 2 ? 0 : slot_q + 1;
    }
}

// ---------------------------------------------------------------------------
// One velocity component per block.  umac on N-faces depends on component N
// alone: its interface states iface(N, N), the transverse states of
// component N (pairs (T, 3 - N - T)), their corrections (uimh(T', N)) and
// the N-component force.  So the blocks of blockIdx.z = N compute the chain
// of component N only and write umac_N.
//   N = 0: uimhyz (y-faces of plane q - 1, by z) and uimhzy (z-face q, by y);
//          umac on x-faces;
//   N = 1: vimhxz (x-faces of plane q - 1, by z) and vimhzx (z-face q, by x);
//          vmac on y-faces;
//   N = 2: wimhxy (x-faces of plane q, by y) and wimhyx (y-faces of plane q,
//          by x); wmac on z-faces.
//
// On the transverse faces (T != N) a state is selected by utrans_T, so each is
// evaluated on its upwind cell only (predict of mx_march.H with the cell's
// own tracing velocity, which the columns exchange through LDS); a face with
// |utrans| < rel_eps averages both sides and carries the other one along.  The
// Riemann solve needs both sides of the N-faces: there the cell's one traced
// state (its velocity points at one of its faces) is exchanged through LDS.
//
// Per step q three phases separated by barriers, straight-line code in which
// columns past the tile take clamped loads and neighbouring LDS slots:
//   1  umac_N of step q - 1; the PPM face values of plane q;
//   2  traces of plane q (x, y, z); the z transverse term of plane q - 1;
//   3  the transverse states and the z edge terms; plane q + 1 goes to LDS.
//
// What bounds it: like the edge kernel, VALU issue and the latency of its
// dependent chains.  Against evaluating both sides of every face in seven
// phases, per launch: 256^3 ppm_type 1 1.20 ms (1.60), ppm_type 2 1.72 ms (2.28),
// a 192^3 star in 27 boxes, ppm_type 2, 0.72 ms (1.30, in two launches); with the
// chunks of pick_chunks one 32^3 box 0.019 ms (0.122).
struct VPTile {
    int box, x0, y0, z0;
    int nx, ny, nz;
    int zgen;  // bits: a z side (0 low, 1 high) in reach that is not open
};

// the block's LDS, one set for the three component bodies, every array at a
// multiple of 512 bytes from S
template <int PPM, int TX, int TY>
struct VPLayout {
    static constexpr int NT = vf_nt(TX, TY);
    static constexpr int G = PPM == 2 ? 3 : 2;
    static constexpr int W = TX + 2;
    static constexpr int H = TY + 2;
    static constexpr int SW = W + 2 * G;
    static constexpr int SH = H + 2 * G;
    static constexpr int FO = PPM == 2 ? 1 : 0;
    static constexpr int FXW = W + 1 + 2 * FO;
    static constexpr int FYH = H + 1 + 2 * FO;
    static constexpr int NS = (SW * SH + NT - 1) / NT;
    static constexpr int NFX = (FXW * H + NT - 1) / NT;
    static constexpr int NFY = (W * FYH + NT - 1) / NT;
    static constexpr int oU = (SW * SH + 63) / 64 * 64;  // utrans_x (or _y), 3 planes
    static constexpr int oFX = oU + 3 * NT;
    static constexpr int oFY = oFX + NFX * NT;
    static constexpr int oHA = oFY + NFY * NT;  // uimh(T, N)
    static constexpr int oUA = oHA + NT;        // tracing velocity along T
    static constexpr int oPA = oUA + NT;        // transverse states
    static constexpr int oC = oPA + NT;
    // N < 2: the traced N-state, the z term, the z edge term, the force
    static constexpr int oIP = oC, oTZ = oIP + NT, oEZ = oTZ + NT, oFL = oEZ + NT;
    // N = 2: the second in-plane direction
    static constexpr int oV = oC, oHB = oV + 3 * NT, oUB = oHB + NT, oPB = oUB + NT;
    static constexpr int oEnd = oPB + NT + W + 2;
};

typedef __attribute__((address_space(4))) const VFBox cvbox;
typedef __attribute__((address_space(4))) const double cd4;
__device__ __forceinline__ cvbox* vfresh(const VFBox* p) {
    unsigned long long a = (unsigned long long)p;
    asm("" : "+s"(a));
    return (cvbox*)a;
}

// a component's side at a face: `in`: the inside cell's state (lo, hi which
// side); fixed: the outside cell's value, or zero
struct VSide {
    bool lo, hi, fixed, zero;
    __device__ __forceinline__ VSide(int pos, int dlo, int dhi, int plo, int phi, bool normal) {
        lo = plo != MX_PHYS_INTERIOR && pos == dlo;
        hi = phi != MX_PHYS_INTERIOR && pos == dhi + 1;
        const int p = lo ? plo : phi;
        const bool wall = p == MX_PHYS_SLIPWALL || p == MX_PHYS_SYMMETRY;
        fixed = (lo || hi) && (p == MX_PHYS_INFLOW || p == MX_PHYS_NOSLIPWALL || (normal && wall));
        zero = fixed && p != MX_PHYS_INFLOW;
    }
};

// a transverse face's upwind choice by utrans (vf_upwind)
struct VFace {
    bool left, both;
    __device__ __forceinline__ VFace(double t, double eps, bool lo, bool hi) {
        left = ((t > 0.0) | hi) & !lo;
        both = (dabs(t) < eps) & !(lo | hi);
    }
};

// MODE, the sides in the tile's reach: 0 interior or outflow; 1 any z side may be
// another; 2 any side may be
template <int PPM, int TX, int TY, int MODE, int N>
__device__ __forceinline__ void vp_comp(const VFBox& B, const VPTile& tl, const VFArgs& A,
                                        double* lds) {
    using L = VPLayout<PPM, TX, TY>;
    constexpr int NT = L::NT, G = L::G, W = L::W, H = L::H, SW = L::SW, SH = L::SH;
    constexpr int FO = L::FO, FXW = L::FXW, FYH = L::FYH, NS = L::NS, NFX = L::NFX, NFY = L::NFY;
    constexpr bool GEN = MODE == 2;
    // the in-plane transverse direction of N < 2 and its steps in a column
    // plane and in S; the N direction's
    constexpr int T = N == 0 ? 1 : 0;
    constexpr int TS = T == 0 ? 1 : W, TSS = T == 0 ? 1 : SW;
    constexpr int DS = N == 0 ? 1 : W, DSS = N == 0 ? 1 : SW;
    double* S = lds;
    double* FX = lds + L::oFX;
    double* FY = lds + L::oFY;
    double* HA = lds + L::oHA;
    double* UA = lds + L::oUA;
    double* PA = lds + L::oPA;
    double* IP = lds + L::oIP;
    double* TZ = lds + L::oTZ;
    double* EZ = lds + L::oEZ;
    double* FL = lds + L::oFL;
    double* HB = lds + L::oHB;
    double* UB = lds + L::oUB;
    double* PB = lds + L::oPB;

    const int X0 = tl.x0, Y0 = tl.y0, nx = tl.nx, ny = tl.ny;
    const int z0 = tl.z0, z1 = tl.z0 + tl.nz - 1;
    const bool last_x = X0 + nx - 1 == B.hi[0];
    const bool last_y = Y0 + ny - 1 == B.hi[1];
    const bool last_z = z1 == B.hi[2];
    const bool sph = A.spherical != 0;
    const int* bcl = A.bclo[N];
    const int* bch = A.bchi[N];

    const double dt = A.dt, eps = A.rel_eps, dt2 = 0.5 * dt;
    const double t6x = uniform(A.dt6 / B.h[0].d), t6y = uniform(A.dt6 / B.h[1].d),
                 t6z = uniform(A.dt6 / B.h[2].d);
    const double t4x = uniform(A.dt4 / B.h[0].d), t4y = uniform(A.dt4 / B.h[1].d),
                 t4z = uniform(A.dt4 / B.h[2].d);

    const int tid = threadIdx.x;
    const int a = tid % W;  // local column: cell (X0 + a - 1, Y0 + b - 1)
    const int b = tid / W;
    const int I = X0 + a - 1;
    const int J = Y0 + b - 1;
    const int si = (a + G) + (b + G) * SW;
    const bool inx = a >= 1 && a <= nx, iny = b >= 1 && b <= ny;
    const bool store = N == 0 ? a >= 1 && iny && (a <= nx || (last_x && a == nx + 1))
                              : N == 1 ? b >= 1 && inx && (b <= ny || (last_y && b == ny + 1))
                                       : inx && iny;
    const VSide dx(I, B.domlo[0], B.domhi[0], A.plo[0], A.phi[0], N == 0);
    const VSide dy(J, B.domlo[1], B.domhi[1], A.plo[1], A.phi[1], N == 1);
    const int zlo = A.plo[2] != MX_PHYS_INTERIOR ? B.domlo[2] : INT_MIN;
    const int zhi = A.phi[2] != MX_PHYS_INTERIOR ? B.domhi[2] + 1 : INT_MIN;
    const bool zgl = tl.zgen & 1, zgh = tl.zgen & 2;
    auto z_general = [&](int q) {
        return MODE > 0 && ((zgl && q <= B.domlo[2] + 3) || (zgh && q >= B.domhi[2] - 2));
    };
    auto side_z = [&](int q) {
        cvbox* Bf = vfresh(&B);
        return VSide(q, Bf->domlo[2], Bf->domhi[2], A.plo[2], A.phi[2], N == 2);
    };

    // byte offsets within a plane; a column past the tile takes its last one
    const DA sv = B.ut, fv = B.fo, ufv = B.uf, ov = B.um[N], tzv = B.tr[2];
    const int ac = min(a, nx + 1), bc = min(b, ny + 1);
    const unsigned sjs = (unsigned)sv.js * 8u;
    const unsigned oCol = (unsigned)(ac + G) * 8u + (unsigned)(bc + G) * sjs;
    const unsigned oF = (unsigned)ac * 8u + (unsigned)bc * (unsigned)fv.js * 8u;
    const unsigned oUf = (unsigned)ac * 8u + (unsigned)bc * (unsigned)ufv.js * 8u;
    const unsigned oTr = (unsigned)ac * 8u + (unsigned)bc * (unsigned)tzv.js * 8u;
    const unsigned oO = (unsigned)ac * 8u + (unsigned)bc * (unsigned)ov.js * 8u;
    const unsigned oUx = (unsigned)ac * 8u + (unsigned)bc * (unsigned)B.tr[0].js * 8u;
    const unsigned oUy = (unsigned)ac * 8u + (unsigned)bc * (unsigned)B.tr[1].js * 8u;
    // w on the N-faces: w0mac (spherical), w0_cart (planar, N = 2); else unused
    // (utrans_N stands in, so that the load is unconditional).  It has no ghosts
    // that the tile's own faces do not lie in.
    const bool has_w = sph || N == 2;
    const bool add_m = sph && B.add, add_p = !sph && B.add;
    cd4* const w0_z = (cd4*)B.w0a;
    const DA wv = sph ? B.w0m[N] : (N == 2 ? B.w0c : B.tr[N]);
    const int aw = min(max(a, 1), N == 0 ? nx + 1 : nx), bw = min(max(b, 1), N == 1 ? ny + 1 : ny);
    const unsigned oWv = (unsigned)(aw - 1) * 8u + (unsigned)(bw - 1) * (unsigned)wv.js * 8u;
    unsigned offS[NS];
    int slS[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int idx = tid + k * NT < SW * SH ? tid + k * NT : tid;
        slS[k] = idx;
        offS[k] = (unsigned)min(idx % SW, nx + 1 + 2 * G) * 8u +
                  (unsigned)min(idx / SW, ny + 1 + 2 * G) * sjs;
    }
    int fxi[NFX], fyi[NFY];
#pragma unroll
    for (int k = 0; k < NFX; ++k) {
        const int idx = min(tid + k * NT, FXW * H - 1);
        fxi[k] = (idx % FXW - FO + G) + (idx / FXW + G) * SW;
    }
#pragma unroll
    for (int k = 0; k < NFY; ++k) {
        const int idx = min(tid + k * NT, W * FYH - 1);
        fyi[k] = (idx % W + G) + (idx / W - FO + G) * SW;
    }

    // plane bases: the next plane to load; w of the faces phase 1 solves; the
    // output plane
    gcc* sN = (gcc*)sv.p + 8 * sv.off(X0 - 1 - G, Y0 - 1 - G, z0 - 1, N);
    gcc* sC = sN + G * B.ks[0];
    gcc* fN = (gcc*)fv.p + 8 * fv.off(X0 - 1, Y0 - 1, z0 - 1, N);
    gcc* xN = (gcc*)B.tr[0].p + 8 * B.tr[0].off(X0 - 1, Y0 - 1, z0 - 1);
    gcc* yN = (gcc*)B.tr[1].p + 8 * B.tr[1].off(X0 - 1, Y0 - 1, z0 - 1);
    gcc* zN = (gcc*)tzv.p + 8 * tzv.off(X0 - 1, Y0 - 1, z0 - 1);
    gcc* ux = (gcc*)ufv.p + 8 * ufv.off(X0 - 1, Y0 - 1, z0 - 1, 0);
    gcc* uy = (gcc*)ufv.p + 8 * ufv.off(X0 - 1, Y0 - 1, z0 - 1, 1);
    gcc* uz = (gcc*)ufv.p + 8 * ufv.off(X0 - 1, Y0 - 1, z0 - 1, 2);
    gcc* wN = (gcc*)wv.p + 8 * wv.off(X0, Y0, z0, sph || N < 2 ? 0 : 2);
    gc* oP = (gc*)ov.p + 8 * ov.off(X0 - 1, Y0 - 1, z0 - (N < 2 ? 3 : 2));

    // column state of step q (see k_es_fused); v[jj] = s(q - 4 + jj)
    double v[9];
#pragma unroll
    for (int jj = 0; jj < 9; ++jj) v[jj] = 0.0;
#pragma unroll
    for (int jj = 4 - G; jj < 4 + G; ++jj) v[jj + 1] = gload(sN + (jj - 4) * B.ks[0], oCol);
    double pcs = gload(sC, oCol), pf = gload(fN, oF), pt = gload(zN, oTr);
    double pux = gload(ux, oUf), puy = gload(uy, oUf), puz = gload(uz, oUf);
    double pw = 0.0, w_r = 0.0;
    double fo_p = 0.0, fo_q = 0.0, tr_p = 0.0, tr_q = 0.0, ufx = 0.0, ufy = 0.0, ufz = 0.0;
    double zf0 = 0.0, zf1 = 0.0, zf2 = 0.0, zsl = 0.0, Ipz_prev = 0.0;
    double zl = 0.0, zr = 0.0, hz = 0.0, hz_p = 0.0;
    double sa = 0.0, sa_o = 0.0, sa_p = 0.0, sa_po = 0.0;  // T state, its other side
    double sb = 0.0, sb_o = 0.0;
    double nl = 0.0, nr = 0.0, nl_p = 0.0, nr_p = 0.0;  // iface(N, N) (N < 2)
    double tc_p = 0.0, pz_p = 0.0, ez0_p = 0.0, ez1_p = 0.0;
    if (PPM == 1) {
        const double d0 = vl_slope(v[3], v[4], v[5]);
        zsl = vl_slope(v[4], v[5], v[6]);
        zf1 = face1(v[4], v[5], d0, zsl);  // face z0 - 1
    } else {
        zf0 = cs_face(v[2], v[3], v[4], v[5]);
        zf1 = cs_face(v[3], v[4], v[5], v[6]);
        zf2 = cs_face(v[4], v[5], v[6], v[7]);
    }

    double pS[NS], pU = 0.0, pV = 0.0;
    auto load_planes = [&]() {
#pragma unroll
        for (int k = 0; k < NS; ++k) pS[k] = gload(sN, offS[k]);
        if (N != 0) pU = gload(xN, oUx);
        if (N != 1) pV = gload(yN, oUy);
    };
    auto stage_planes = [&](int slot) {
#pragma unroll
        for (int k = 0; k < NS; ++k) S[(k + 1) * NT <= SW * SH ? tid + k * NT : slS[k]] = pS[k];
        lds[L::oU + slot * NT + tid] = N != 0 ? pU : pV;
        if (N == 2) lds[L::oV + slot * NT + tid] = pV;
    };
    auto s_plane = [&](int k) {  // rare paths
        cvbox* Bf = vfresh(&B);
        return (gcc*)Bf->ut.p + 8 * ((long long)(X0 - 1 - G - Bf->ut.b0) +
                                     (long long)(Y0 - 1 - G - Bf->ut.b1) * Bf->ut.js +
                                     (long long)(k - Bf->ut.b2) * Bf->ut.ks +
                                     (long long)N * Bf->ut.ns);
    };
    load_planes();
    stage_planes(0);
    int slot_q = 0, slot_p = 2, slot_o = 1;  // planes q, q - 1, q - 2 (then q + 1)
    // loads stay at plane z1 + 1 (w: at the last face), see k_es_fused
    auto advance = [&](bool more, bool wmore) {
        __attribute__((address_space(4))) const long long* ks = vfresh(&B)->ks;
        if (more) {
            sN += ks[0];
            sC += ks[0];
            fN += ks[1];
            ux += ks[2];
            uy += ks[2];
            uz += ks[2];
            xN += ks[3];
            yN += ks[4];
            zN += ks[5];
        }
        if (wmore) wN += sph ? ks[9 + N] : (N == 2 ? ks[12] : ks[3 + N]);
        oP += ks[6 + N];
    };
    // umac_N of step r = q - 1: plane r - 1 (N < 2) or z-face r
    auto solve = [&](int q) {
        const double* Uo = lds + L::oU + slot_o * NT;  // utrans_T, plane r - 1
        const double* Ur = lds + L::oU + slot_p * NT;  // N = 2: utrans_x, _y, plane r
        const double* Vr = lds + L::oV + slot_p * NT;
        double l, r;
        if (N < 2) {
            const double tt = N == 0 ? t4y : t4x;
            auto side = [&](double s, int t) {
                double x = s - tt * (Uo[t + TS] + Uo[t]) * (PA[t + TS] - PA[t]);
                x = x - EZ[t];
                return x + dt2 * FL[t];
            };
            l = side(nl_p, tid - DS);
            r = side(nr_p, tid);
        } else {
            const double ez0 = t4x * (Ur[tid + 1] + Ur[tid]) * (PA[tid + 1] - PA[tid]);
            const double ez1 = t4y * (Vr[tid + W] + Vr[tid]) * (PB[tid + W] - PB[tid]);
            l = zl - ez0_p;
            l = l - ez1_p;
            r = zr - ez0;
            r = r - ez1;
            l = l + dt2 * fo_p;
            r = r + dt2 * fo_q;
            ez0_p = ez0;
            ez1_p = ez1;
        }
        double res = vf_riemann(l, r, has_w, w_r, eps);
        if (N == 2) {
            if (q - 1 == zlo) res = dmin(r, 0.0);
            if (q - 1 == zhi) res = dmax(l, 0.0);
            if (z_general(q - 1)) {
                const VSide d = side_z(q - 1);
                if (d.fixed) res = d.zero ? 0.0 : (d.lo ? v[3] : v[4]);
            }
        } else {
            const VSide& d = N == 0 ? dx : dy;
            if (d.lo | d.hi) {
                res = d.lo ? dmin(r, 0.0) : dmax(l, 0.0);
                if (GEN && d.fixed) {
                    const unsigned st = N == 0 ? 8u : sjs;
                    res = d.zero ? 0.0 : gload(s_plane(q - 2), d.lo ? oCol - st : oCol);
                }
            }
        }
        const bool now = N < 2 ? q >= z0 + 2 : q > z0 && (q <= z1 + 1 || last_z);
        // Addw0: w0mac, or the planar w0 of z-face q - 1
        if (add_m) res = res + w_r;
        if (N == 2 && add_p) res = res + w0_z[now ? q - 1 : z0];
        if (now && store) gstore(oP, oO, res);
    };
    sN += B.ks[0];
    sC += B.ks[0];
    fN += B.ks[1];
    ux += B.ks[2];
    uy += B.ks[2];
    uz += B.ks[2];
    xN += B.ks[3];
    yN += B.ks[4];
    zN += B.ks[5];
    __syncthreads();

    for (int q = z0 - 1; q <= z1 + 1; ++q) {
        const double* Uq = lds + L::oU + slot_q * NT;  // utrans_x (N = 0: _y)
        const double* Vq = lds + L::oV + slot_q * NT;  // N = 2: utrans_y
        const double* Up = lds + L::oU + slot_p * NT;
        load_planes();

        // ---- 1: umac of step q - 1; the column state moves on; face values
        w_r = pw;
        solve(q);
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) v[jj] = v[jj + 1];
        v[4 + G] = pcs;
        fo_p = fo_q;
        fo_q = pf;
        tr_p = tr_q;
        tr_q = pt;
        ufx = pux;
        ufy = puy;
        ufz = puz;
        sa_p = sa;
        sa_po = sa_o;
        nl_p = nl;
        nr_p = nr;
        hz_p = hz;
        pcs = gload(sC, oCol);
        pf = gload(fN, oF);
        pt = gload(zN, oTr);
        pux = gload(ux, oUf);
        puy = gload(uy, oUf);
        puz = gload(uz, oUf);
        pw = gload(wN, oWv);
        UA[tid] = N == 0 ? ufy : ufx;
        if (N == 2) UB[tid] = ufy;
#pragma unroll
        for (int k = 0; k < NFX; ++k) {
            const double* s = S + fxi[k];  // face between s[-1] and s[0]
            FX[tid + k * NT] = PPM == 1 ? face1(s[-1], s[0], vl_slope(s[-2], s[-1], s[0]),
                                                vl_slope(s[-1], s[0], s[1]))
                                        : cs_face(s[-2], s[-1], s[0], s[1]);
        }
#pragma unroll
        for (int k = 0; k < NFY; ++k) {
            const double* s = S + fyi[k];
            FY[tid + k * NT] =
                PPM == 1 ? face1(s[-SW], s[0], vl_slope(s[-2 * SW], s[-SW], s[0]),
                                 vl_slope(s[-SW], s[0], s[SW]))
                         : cs_face(s[-2 * SW], s[-SW], s[0], s[SW]);
        }
        cvbox* Bq = vfresh(&B);
        const DivBy hx{Bq->h[0].d, Bq->h[0].r, Bq->h[0].rl}, hy{Bq->h[1].d, Bq->h[1].r, Bq->h[1].rl},
            hzd{Bq->h[2].d, Bq->h[2].r, Bq->h[2].rl};
        __syncthreads();

        // ---- 2: traces of plane q
        const double* FXc = FX + (a + FO) + b * FXW;
        const double* FYc = FY + a + (b + FO) * W;
        const double ta = Uq[tid], tb = N == 2 ? Vq[tid] : 0.0;
        const VSide& da = T == 0 ? dx : dy;  // the first transverse direction's side
        const VFace fa(ta, eps, da.lo, da.hi), fb(tb, eps, dy.lo, dy.hi);
        // the T state of one side: the traced state of that side's cell
        auto state = [&](auto dir, bool left) {
            constexpr int D = decltype(dir)::value;
            constexpr int FST = D == 0 ? 1 : W, SST = D == 0 ? 1 : SW;
            const double u = (N == 2 && D == 1 ? UB : UA)[tid + (left ? -FST : 0)];
            const bool tr = (left & (u > eps)) | (!left & (u < -eps));
            const double sig = div_by(dabs(u) * dt, D == 0 ? hx : hy);
            double x = predict<PPM, FST, SST>(S + si, D == 0 ? FXc : FYc, left, tr, sig);
            if (GEN) {
                const int pos = D == 0 ? I : J;
                if ((D == 0 ? a : b) >= 1 && ppm_special<PPM>(pos - (left ? 1 : 0), B.domlo[D],
                                                              B.domhi[D], bcl[D], bch[D]))
                    x = predict_special<PPM, D, SST>(S + si, left, tr, sig, pos, B.domlo[D],
                                                     B.domhi[D], bcl[D], bch[D]);
            }
            return x;
        };
        using DirT = std::integral_constant<int, T>;
        using DirY = std::integral_constant<int, 1>;
        sa = state(DirT{}, fa.left);
        if (N == 2) sb = state(DirY{}, fb.left);
        double ipn = 0.0;
        if (N < 2) {  // the cell's state traced along N, at its downwind face
            const double u = N == 0 ? ufx : ufy;
            const double sig = div_by(dabs(u) * dt, N == 0 ? hx : hy);
            const double* F = N == 0 ? FXc : FYc;
            constexpr int FST = DS;
            const bool up = u > 0.0, off = dabs(u) > eps;
            double x;
            if (PPM == 1) {
                x = cw_trace(v[4], F[up ? FST : 0], F[up ? 0 : FST], sig);
            } else {
                double w9[9], sm, sp;
#pragma unroll
                for (int o = -4; o <= 4; ++o)
                    w9[4 + o] = (o >= -2 && o <= 2) ? S[si + o * DSS] : 0.0;
                cs_cell(w9, F[-FST], F[0], F[FST], F[2 * FST], 1.e-10, sm, sp);
                x = trace_face(v[4], up ? sp : sm, up ? sm : sp, sig);
            }
            if (GEN) {
                constexpr int D = N == 0 ? 0 : 1;
                const int pos = D == 0 ? I : J;
                // (S holds the stencil of the tile's cells and the ones beside)
                if (a <= nx + 1 && b <= ny + 1 &&
                    ppm_special<PPM>(pos, B.domlo[D], B.domhi[D], bcl[D], bch[D])) {
                    double w9[9], sm, sp;
#pragma unroll
                    for (int o = -4; o <= 4; ++o)
                        w9[4 + o] = (o >= -1 - PPM && o <= 1 + PPM) ? S[si + o * DSS] : 0.0;
                    ppm_edges<PPM, D>(w9, pos, B.domlo[D], B.domhi[D], bcl[D], bch[D], sm, sp);
                    x = trace_face(v[4], up ? sp : sm, up ? sm : sp, sig);
                }
            }
            ipn = off && up ? x : v[4];
            nr = off && !up ? x : v[4];
            IP[tid] = ipn;
        }
        {  // z: the cell's states at its two z-faces
            const double sig = div_by(dabs(ufz) * dt, hzd);
            const bool up = ufz > 0.0, off = dabs(ufz) > eps;
            double x, sm = 0.0, sp = 0.0;
            if (PPM == 1) {
                const double d1 = vl_slope(v[4], v[5], v[6]);
                zf2 = face1(v[4], v[5], zsl, d1);
                zsl = d1;
                x = cw_trace(v[4], up ? zf2 : zf1, up ? zf1 : zf2, sig);
                zf1 = zf2;
            } else {
                const double f3 = cs_face(v[4], v[5], v[6], v[7]);
                cs_cell(v, zf0, zf1, zf2, f3, 1.e-10, sm, sp);
                zf0 = zf1;
                zf1 = zf2;
                zf2 = f3;
                x = trace_face(v[4], up ? sp : sm, up ? sm : sp, sig);
            }
            if (z_general(q)) {
                cvbox* Bf = vfresh(&B);
                const int dl = Bf->domlo[2], dh = Bf->domhi[2];
                if (ppm_special<PPM>(q, dl, dh, bcl[2], bch[2])) {
                    double w9[9];
#pragma unroll
                    for (int o = 0; o < 9; ++o)
                        w9[o] = o >= 3 - PPM && o <= 5 + PPM ? gload(s_plane(q - 4 + o), oCol) : 0.0;
                    ppm_edges<PPM, 2>(w9, q, dl, dh, bcl[2], bch[2], sm, sp);
                    x = trace_face(v[4], up ? sp : sm, up ? sm : sp, sig);
                }
            }
            zl = Ipz_prev;
            zr = off && !up ? x : v[4];
            Ipz_prev = off && up ? x : v[4];
        }
        const VFace fz(tr_q, eps, q == zlo, q == zhi);
        double sz = 0.0;
        if (N < 2) {
            sz = fz.left ? zl : zr;
            hz = fz.both ? 0.5 * (zl + zr) : sz;
        } else {
            if (q == zlo) zr = dmin(zr, 0.0);
            if (q == zhi) zl = dmax(zl, 0.0);
        }
        double ha = sa, hb = sb;
        if (fa.both | fb.both) {
            if (fa.both) {
                sa_o = state(DirT{}, !fa.left);
                ha = 0.5 * (sa + sa_o);
            }
            if (N == 2 && fb.both) {
                sb_o = state(DirY{}, !fb.left);
                hb = 0.5 * (sb + sb_o);
            }
        }
        if (GEN) {  // fixed sides
            if (da.fixed) ha = sa = da.zero ? 0.0 : (da.lo ? S[si - TSS] : S[si]);
            if (N == 2 && dy.fixed) hb = sb = dy.zero ? 0.0 : (dy.lo ? S[si - SW] : S[si]);
        }
        if (N < 2 && z_general(q)) {
            const VSide d = side_z(q);
            if (d.fixed) hz = sz = d.zero ? 0.0 : (d.lo ? v[3] : v[4]);
        }
        HA[tid] = ha;
        if (N == 2) HB[tid] = hb;
        if (N < 2) TZ[tid] = t6z * (tr_q + tr_p) * (hz - hz_p);
        __syncthreads();

        // ---- 3: transverse states of component N
        if (N == 2) {
            auto ycell = [&](int t) { return t6y * (Vq[t + W] + Vq[t]) * (HB[t + W] - HB[t]); };
            auto xcell = [&](int t) { return t6x * (Uq[t + 1] + Uq[t]) * (HA[t + 1] - HA[t]); };
            double xy = sa - ycell(tid + (fa.left ? -1 : 0));
            double yx = sb - xcell(tid + (fb.left ? -W : 0));
            if (fa.both | fb.both) {
                const double al = fa.left ? sa : sa_o, ar = fa.left ? sa_o : sa;
                const double bl = fb.left ? sb : sb_o, br = fb.left ? sb_o : sb;
                if (fa.both) xy = 0.5 * ((al - ycell(tid - 1)) + (ar - ycell(tid)));
                if (fb.both) yx = 0.5 * ((bl - xcell(tid - W)) + (br - xcell(tid)));
            }
            if (GEN) {
                if (dx.fixed) xy = sa;
                if (dy.fixed) yx = sb;
            }
            PA[tid] = xy;
            PB[tid] = yx;
        } else {
            const double tt = N == 0 ? t6y : t6x;
            const double tc_q = tt * (Uq[tid + TS] + Uq[tid]) * (HA[tid + TS] - HA[tid]);
            const VFace fp(Up[tid], eps, da.lo, da.hi);  // plane q - 1
            double pa = sa_p - TZ[tid + (fp.left ? -TS : 0)];
            double pz = sz - (fz.left ? tc_p : tc_q);
            if (fp.both | fz.both) {
                const double pl = fp.left ? sa_p : sa_po, pr = fp.left ? sa_po : sa_p;
                if (fp.both) pa = 0.5 * ((pl - TZ[tid - TS]) + (pr - TZ[tid]));
                if (fz.both) pz = 0.5 * ((zl - tc_p) + (zr - tc_q));
            }
            if (GEN && da.fixed) pa = sa_p;
            if (z_general(q) && side_z(q).fixed) pz = sz;
            PA[tid] = pa;
            EZ[tid] = t4z * (tr_q + tr_p) * (pz - pz_p);
            FL[tid] = fo_p;
            pz_p = pz;
            tc_p = tc_q;
            nl = IP[tid - DS];
            const VSide& d = N == 0 ? dx : dy;
            if (d.lo | d.hi) {
                if (d.lo) nr = dmin(nr, 0.0);
                if (d.hi) nl = dmax(nl, 0.0);
            }
        }
        stage_planes(slot_o);
        __syncthreads();

        advance(q < z1, N < 2 ? q > z0 && q <= z1 : q >= z0 && q <= z1);
        const int s_new = slot_o;
        slot_o = slot_p;
        slot_p = slot_q;
        slot_q = s_new;
    }
    w_r = pw;
    solve(z1 + 2);
}

// xmode 1, 2: the XCD-aware orders of xcd_tile over a 1-D grid; 0: tile
// blockIdx.x and component blockIdx.z
template <int PPM, int TX, int TY, int MODE, int WPE>
__global__ void __launch_bounds__(vf_nt(TX, TY)) __attribute__((amdgpu_waves_per_eu(WPE)))
    k_vp_fused_comp(const VFBox* __restrict__ boxes, const VPTile* __restrict__ tiles, VFArgs A,
                    int ntile, int xmode) {
    __shared__ double lds[VPLayout<PPM, TX, TY>::oEnd];
    int t = blockIdx.x, n = blockIdx.z;
    if (xmode != 0 && !xcd_tile(ntile, 3, xmode, t, n)) return;
    const VPTile tl = tiles[t];
    const VFBox& B = boxes[tl.box];
    if (n == 0)
        vp_comp<PPM, TX, TY, MODE, 0>(B, tl, A, lds);
    else if (n == 1)
        vp_comp<PPM, TX, TY, MODE, 1>(B, tl, A, lds);
    else
        vp_comp<PPM, TX, TY, MODE, 2>(B, tl, A, lds);
}

}  // namespace

namespace mxh {

bool velpred_fused_ok(const mx_adv_ctx* c) {
    return c->p.dim == 3 && (c->p.ppm_type == 1 || c->p.ppm_type == 2) &&
           c->p.ppm_trace_forces == 0 && c->vp_fused;
}

namespace {

bool phys_acts(int bc) { return bc != MX_PHYS_INTERIOR; }

bool bc_type_acts(int bc) { return bc == MX_BC_EXT_DIR || bc == MX_BC_HOEXTRAP; }

// x/y-free: in x and in y each domain side either carries nothing that acts
// (no physical override, no PPM boundary stencil) or lies beyond the tile's
// reach (cells [X0 - 1, X0 + nx], faces [X0, X0 + nx]; stencils act within
// three cells of a side)
bool vf_tile_free(int lo0, int n, int dlo, int dhi, bool act_lo, bool act_hi) {
    const bool free_lo = !act_lo || lo0 - 1 > dlo + 2;
    const bool free_hi = !act_hi || lo0 + n < dhi - 2;
    return free_lo && free_hi;
}

// does a side need more than its inside cell's state and a clamp of the normal
// component (everything but outflow), or a PPM boundary stencil?
bool vp_side_general(const mx_adv_ctx* c, int d, bool hi) {
    const int p = hi ? c->p.phys_bc_hi[d] : c->p.phys_bc_lo[d];
    bool g = p != MX_PHYS_INTERIOR && p != MX_PHYS_OUTFLOW;
    for (int n = 0; n < 3; ++n)
        g = g || bc_type_acts(hi ? c->bcs_u[n].hi[d] : c->bcs_u[n].lo[d]);
    return g;
}

int vf_boxes(mx_adv_ctx* c, const std::vector<VpLevel>& levs, std::vector<VFBox>& boxes) {
    const long long lim = 0x7fffffffLL;
    const bool sph = c->p.spherical != 0;
    for (const VpLevel& L : levs) {
        const auto& grids = c->grids[L.lev];
        for (size_t b = 0; b < grids.size(); ++b) {
            VFBox B;
            HBox g = hbox(grids[b]);
            for (int q = 0; q < 3; ++q) {
                B.lo[q] = g.lo[q];
                B.hi[q] = g.hi[q];
                B.dx[q] = c->p.dx[L.lev][q];
                B.h[q] = div_const(B.dx[q]);
                B.domlo[q] = c->p.domain_lo[L.lev][q];
                B.domhi[q] = c->p.domain_hi[L.lev][q];
            }
            B.ut = to_da(L.utilde->fab[b]);
            B.uf = to_da(L.ufull->fab[b]);
            B.fo = to_da(L.force->fab[b]);
            B.w0c = (!sph && L.w0_cart) ? to_da(L.w0_cart->fab[b]) : null_da();
            for (int d = 0; d < 3; ++d) {
                B.tr[d] = to_da(L.utrans->dir[d].fab[b]);
                B.um[d] = to_da(L.umac->dir[d].fab[b]);
                B.w0m[d] = sph ? to_da(L.w0mac->dir[d].fab[b]) : null_da();
            }
            const DA* views[] = {&B.ut,    &B.fo,    &B.uf,     &B.tr[0],  &B.tr[1],  &B.tr[2], &B.um[0],
                                 &B.um[1], &B.um[2], &B.w0m[0], &B.w0m[1], &B.w0m[2], &B.w0c};
            B.w0a = L.add.w0;
            B.add = L.add.umac;
            for (int q = 0; q < 13; ++q) B.ks[q] = 8 * views[q]->ks;
            for (int q = 0; q < 9; ++q)
                if (views[q]->js > lim || views[q]->ks > lim || views[q]->ns > lim)
                    return MX_ERR_UNSUPPORTED;
            boxes.push_back(B);
        }
    }
    return MX_OK;
}

VFArgs vf_args(const mx_adv_ctx* c, int tz) {
    VFArgs A;
    for (int n = 0; n < 3; ++n)
        for (int d = 0; d < 3; ++d) {
            A.bclo[n][d] = c->bcs_u[n].lo[d];
            A.bchi[n][d] = c->bcs_u[n].hi[d];
        }
    for (int d = 0; d < 3; ++d) {
        A.plo[d] = c->p.phys_bc_lo[d];
        A.phi[d] = c->p.phys_bc_hi[d];
    }
    A.spherical = c->p.spherical != 0 ? 1 : 0;
    A.tz = tz;
    A.dt = c->p.dt;
    A.rel_eps = c->p.rel_eps;
    A.dt4 = 0.25 * c->p.dt;
    A.dt6 = c->p.dt / 6.0;
    return A;
}

// all three components per block
template <int TX, int TY, int WPE>
int vf_launch(mx_adv_ctx* c, const std::vector<VFBox>& boxes, int tz, int lev) {
    std::vector<VFTile> tiles, btiles;
    bool act[2][2] = {{false, false}, {false, false}};
    for (int d = 0; d < 2; ++d) {
        act[d][0] = phys_acts(c->p.phys_bc_lo[d]);
        act[d][1] = phys_acts(c->p.phys_bc_hi[d]);
        for (int n = 0; n < 3; ++n) {
            act[d][0] = act[d][0] || bc_type_acts(c->bcs_u[n].lo[d]);
            act[d][1] = act[d][1] || bc_type_acts(c->bcs_u[n].hi[d]);
        }
    }
    for (size_t id = 0; id < boxes.size(); ++id) {
        const VFBox& B = boxes[id];
        const int ntx = (B.hi[0] - B.lo[0] + TX) / TX;
        const int nty = (B.hi[1] - B.lo[1] + TY) / TY;
        const int nzc = (B.hi[2] - B.lo[2] + tz) / tz;
        for (int z = 0; z < nzc; ++z)
            for (int y = 0; y < nty; ++y)
                for (int x = 0; x < ntx; ++x) {
                    const int x0 = B.lo[0] + x * TX, y0 = B.lo[1] + y * TY;
                    const int nx = std::min(TX, B.hi[0] - x0 + 1);
                    const int ny = std::min(TY, B.hi[1] - y0 + 1);
                    const bool f =
                        vf_tile_free(x0, nx, B.domlo[0], B.domhi[0], act[0][0], act[0][1]) &&
                        vf_tile_free(y0, ny, B.domlo[1], B.domhi[1], act[1][0], act[1][1]);
                    (f ? tiles : btiles).push_back({(int)id, x, y, z});
                }
    }
    const size_t nfree = tiles.size();
    tiles.insert(tiles.end(), btiles.begin(), btiles.end());
    if (tiles.empty()) return MX_OK;
    if (tiles.size() > 0x7fffffffULL) return MX_ERR_UNSUPPORTED;
    const VFArgs A = vf_args(c, tz);
    Table tab(c);
    const size_t ob = tab.add(boxes);
    const size_t ot = tab.add(tiles);
    int rc = tab.upload();
    if (rc) return rc;
    const VFBox* db = tab.dev<VFBox>(ob);
    const VFTile* dt = tab.dev<VFTile>(ot);
    const KGeom kg = kgeom(c, lev);
    const dim3 block(vf_nt(TX, TY));
    auto launch = [&](auto xyf, const VFTile* d, size_t n) -> int {
        constexpr bool XYF = decltype(xyf)::value;
        if (n == 0) return MX_OK;
        if (c->p.ppm_type == 1)
            MX_LAUNCH(c, "k_vp_fused", (k_vp_fused<1, TX, TY, XYF, WPE>), dim3((unsigned)n), block,
                      db, d, kg, A);
        else
            MX_LAUNCH(c, "k_vp_fused", (k_vp_fused<2, TX, TY, XYF, WPE>), dim3((unsigned)n), block,
                      db, d, kg, A);
        return MX_OK;
    };
    rc = launch(std::true_type{}, dt, nfree);
    return rc ? rc : launch(std::false_type{}, dt + nfree, tiles.size() - nfree);
}

// blocks of the kernel a CU holds; WPE as in vp_launch
template <int PPM, int TX, int TY, int MODE, int WPE>
int vp_blocks() {
    constexpr int W = MODE == 0 ? WPE : 3;
    static const int n = [] {
        int v = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, k_vp_fused_comp<PPM, TX, TY, MODE, W>,
                                                         vf_nt(TX, TY), 0) != hipSuccess) {
            (void)hipGetLastError();
            v = 0;
        }
        return v > 0 ? v : W;
    }();
    return n;
}
template <int TX, int TY, int MODE, int WPE>
int vp_blocks(int ppm) {
    return ppm == 1 ? vp_blocks<1, TX, TY, MODE, WPE>() : vp_blocks<2, TX, TY, MODE, WPE>();
}

// one component per block.  WPE: the register budget (waves per SIMD) of the
// kernel without the rules of general sides; the others take 3
template <int TX, int TY, int WPE>
int vp_launch(mx_adv_ctx* c, const std::vector<VFBox>& boxes, int tz, bool one_level) {
    bool act[3][2], zgen = false;
    for (int d = 0; d < 3; ++d)
        for (int s = 0; s < 2; ++s) act[d][s] = vp_side_general(c, d, s == 1);
    auto clear_xy = [&](const VFBox& B, int x, int nx, int y, int ny) {
        return vf_tile_free(x, nx, B.domlo[0], B.domhi[0], act[0][0], act[0][1]) &&
               vf_tile_free(y, ny, B.domlo[1], B.domhi[1], act[1][0], act[1][1]);
    };
    if (tz <= 0) {
        std::vector<ChunkCols> cols;
        for (const VFBox& B : boxes) {
            ChunkCols col{B.hi[2] - B.lo[2] + 1, {0, 0}};
            for (int y = B.lo[1]; y <= B.hi[1]; y += TY)
                for (int x = B.lo[0]; x <= B.hi[0]; x += TX)
                    ++col.tiles[clear_xy(B, x, std::min(TX, B.hi[0] - x + 1), y,
                                         std::min(TY, B.hi[1] - y + 1))
                                    ? 0
                                    : 1];
            cols.push_back(col);
            zgen = zgen || (col.tiles[0] && !vf_tile_free(B.lo[2], col.nz, B.domlo[2], B.domhi[2],
                                                          act[2][0], act[2][1]));
        }
        // of the kernels that the launches take (a query loads its kernel)
        bool any[2] = {false, false};
        for (const ChunkCols& col : cols)
            for (int l = 0; l < 2; ++l) any[l] = any[l] || col.tiles[l];
        const int ppm = c->p.ppm_type;
        const int blocks[2] = {!any[0] ? 1
                               : zgen  ? vp_blocks<TX, TY, 1, WPE>(ppm)
                                       : vp_blocks<TX, TY, 0, WPE>(ppm),
                               any[1] ? vp_blocks<TX, TY, 2, WPE>(ppm) : 1};
        tz = pick_chunks(cols, 3, blocks);
    }
    std::vector<VPTile> tiles, btiles;  // clear of general x/y sides, the others
    for (size_t id = 0; id < boxes.size(); ++id) {
        const VFBox& B = boxes[id];
        const int nz = B.hi[2] - B.lo[2] + 1, nch = chunk_count(nz, tz);
        for (int ch = 0; ch < nch; ++ch)
            for (int y = B.lo[1]; y <= B.hi[1]; y += TY)
                for (int x = B.lo[0]; x <= B.hi[0]; x += TX) {
                    const int z = chunk_start(nz, nch, ch), ze = chunk_start(nz, nch, ch + 1);
                    VPTile T{(int)id,
                             x,
                             y,
                             B.lo[2] + z,
                             std::min(TX, B.hi[0] - x + 1),
                             std::min(TY, B.hi[1] - y + 1),
                             ze - z,
                             0};
                    const bool f = clear_xy(B, x, T.nx, y, T.ny);
                    for (int s = 0; s < 2; ++s)
                        if (!vf_tile_free(T.z0, T.nz, B.domlo[2], B.domhi[2], s == 0 && act[2][0],
                                          s == 1 && act[2][1]))
                            T.zgen |= 1 << s;
                    (f ? tiles : btiles).push_back(T);
                    zgen = zgen || (f && T.zgen);
                }
    }
    const size_t nfree = tiles.size();
    tiles.insert(tiles.end(), btiles.begin(), btiles.end());
    if (tiles.empty()) return MX_OK;
    if (tiles.size() > 0x7fffffffULL) return MX_ERR_UNSUPPORTED;
    const VFArgs A = vf_args(c, 0);
    Table tab(c);
    const size_t ob = tab.add(boxes);
    const size_t ot = tab.add(tiles);
    int rc = tab.upload();
    if (rc) return rc;
    const VFBox* db = tab.dev<VFBox>(ob);
    const VPTile* dt = tab.dev<VPTile>(ot);
    // the block order: -1 (the default) takes contiguous tile ranges per XCD
    // (2) for one level of equal boxes, whose tiles cost alike, and the
    // round robin (1) otherwise, where contiguous ranges of unequal tiles
    // unbalance the XCDs
    int xm = c->vp_fused_xcd;
    if (xm < 0) {
        bool equal = one_level;
        for (size_t b = 1; equal && b < boxes.size(); ++b)
            for (int q = 0; q < 3; ++q)
                equal = equal && boxes[b].hi[q] - boxes[b].lo[q] == boxes[0].hi[q] - boxes[0].lo[q];
        xm = equal ? 2 : 1;
    }
    auto launch = [&](auto mode, const VPTile* d, size_t n) -> int {
        constexpr int MODE = decltype(mode)::value;
        constexpr int W = MODE == 0 ? WPE : 3;
        if (n == 0) return MX_OK;
        const dim3 grid = xm ? dim3(xcd_tile_blocks((long long)n, 3)) : dim3((unsigned)n, 1, 3);
        const dim3 block(vf_nt(TX, TY));
        const int nt = (int)n;
        if (c->p.ppm_type == 1)
            MX_LAUNCH(c, "k_vp_fused", (k_vp_fused_comp<1, TX, TY, MODE, W>), grid, block, db, d, A,
                      nt, xm);
        else
            MX_LAUNCH(c, "k_vp_fused", (k_vp_fused_comp<2, TX, TY, MODE, W>), grid, block, db, d, A,
                      nt, xm);
        return MX_OK;
    };
    // a general z side puts every clear tile in the kernel with the z rules, as
    // in the edge kernel's launch
    rc = zgen ? launch(std::integral_constant<int, 1>{}, dt, nfree)
              : launch(std::integral_constant<int, 0>{}, dt, nfree);
    return rc ? rc : launch(std::integral_constant<int, 2>{}, dt + nfree, tiles.size() - nfree);
}

}  // namespace

int velpred_fused(mx_adv_ctx* c, const std::vector<VpLevel>& levs, bool* added) {
    if (added) *added = false;
    if (levs.empty()) return MX_OK;
    int rc = check_phys(c);
    if (rc) return rc;
    std::vector<VFBox> boxes;
    if ((rc = vf_boxes(c, levs, boxes))) return rc;
    const int tz = c->vp_fused_tz;
    // rows past the per-component kernel's unsigned 32-bit byte offsets (a tile
    // and its stencil span at most 25 rows), or that run downwards
    bool rows = true;
    for (const VFBox& B : boxes) {
        const DA* views[] = {&B.ut,    &B.fo,    &B.uf,     &B.tr[0],  &B.tr[1],  &B.tr[2], &B.um[0],
                             &B.um[1], &B.um[2], &B.w0m[0], &B.w0m[1], &B.w0m[2], &B.w0c};
        for (const DA* d : views) rows = rows && d->js >= 0 && d->js <= 0x7fffffffLL / (8 * 26);
    }
    // all three components per block: 16 x 11 columns at 2 waves per SIMD
    // (256 VGPRs); one component per block: the tile shape (cell columns)
    // and register budget (waves per SIMD) of `velpred_fused_tile`
    if (!c->vp_fused_comp || !rows) return vf_launch<16, 11, 2>(c, boxes, tz > 0 ? tz : 32, levs[0].lev);
    if (added) *added = true;
    const bool one = levs.size() == 1;
    // 16 x 11 columns: ppm_type 1 at 4 waves per SIMD (1.20 ms per 256^3 launch
    // against 1.21 at 3), ppm_type 2 at 3, where 4 spill 67 VGPRs (1.72 against
    // 2.46 ms)
    const int tile = c->vp_fused_tile >= 0 ? c->vp_fused_tile : (c->p.ppm_type == 1 ? 2 : 0);
    switch (tile) {
        case 1: return vp_launch<16, 8, 3>(c, boxes, tz, one);
        case 2: return vp_launch<16, 11, 4>(c, boxes, tz, one);
        case 3: return vp_launch<32, 8, 3>(c, boxes, tz, one);
        case 4: return vp_launch<16, 8, 4>(c, boxes, tz, one);
        case 5: return vp_launch<16, 12, 4>(c, boxes, tz, one);
        default: return vp_launch<16, 11, 3>(c, boxes, tz, one);
    }
}

}  // namespace mxh
