// mx_edge_fused.hip -- fused 3-D MakeEdgeScal: PPM, predictor, transverse
// and edge states of one scalar in a single z-marching kernel.
//
// A block owns a tile of cell columns of one box (16 x 11 by default), grown
// by one cell in x and y (18 x 13 columns, one thread each), and marches up a
// chunk [z0, z1] of the box's planes, one cell plane q per step (plus
// q = z0 - 1 and q = z1 + 1, whose states the chunk's first and last faces
// need).
//
// The reference formulas (MaestroMakeEdgeScalars.cpp: Predictor :662-863,
// Transverse :865-1359, Edges :1361-1667; MaestroPPM.cpp) are evaluated upwind
// first:
//   * a face's predictor, corner-coupled and edge states are selected by the
//     sign of the face velocity, so a face evaluates the PPM limiter, the
//     trace, the transverse and the edge corrections of its upwind cell only
//     (the cell's LDS slot is the face's own or its low neighbour's).  The
//     reference forms both sides and selects; the selected value is the same
//     expression with the same operands in the same order;
//   * a face with |u| <= rel_eps averages both sides.  Its two states are the
//     plain cell values (the trace is off), so the rare path re-reads them;
//   * domain sides: an extrapolating or even side takes the inside cell's
//     state, ext_dir the outside value, an odd side zero, at every stage, so a
//     side fixes the face's upwind cell or its value;
//   * a PPM face value (type 1: the limited 4th-order interpolant; type 2: the
//     Colella-Sekora face value) is computed once per face and read by the
//     faces whose upwind cell it bounds.
// PPM boundary stencils (ext_dir / hoextrap within two or three cells of the
// domain edge) fall back to the full per-cell routine of mx_device.H.
//
// Per step q a block runs three phases separated by barriers:
//   1  the edge states of step q - 1 (x and y faces of plane q - 2, z-face
//      q - 1); the PPM face values of plane q;
//   2  limiter, trace and upwind state of the x, y and z faces of cell q; the z
//      transverse term of plane q - 1;
//   3  corner-coupled states simhxy, simhyx (plane q), simhxz, simhyz (plane
//      q - 1), simhzx, simhzy (z-face q, in registers) and the z edge terms;
//      plane q + 1 (loaded into registers since phase 1) goes to LDS.
// A phase is straight-line code: every thread evaluates it, columns past the
// tile on clamped loads and neighbouring LDS slots, and only stores and the rare
// paths are predicated.
//
// What bounds it: VALU issue and the latency of the dependent FP64 chains
// between barriers, then HBM.  A 256^3 launch of 5 scalars (ppm_type 1, 2.73 ms)
// issues VALU for 1.66 ms (56 to 61%), its waves wait for half of their cycles,
// and 9.8 GB move (7.2 read, 2.6 written), 3.6 TB/s, 70% of what a copy reaches.
// One wave alone takes 10.7 thousand cycles a step for 510 VALU instructions,
// so waves in flight decide: the advective ppm_type 1 kernel is held to 128
// VGPRs and 40 KB of LDS, 4 blocks a CU (3.11 ms at 3 blocks, 2.68 ms at 4).
// Measured per 256^3 launch against evaluating both sides of every face in
// seven phases: ppm_type 1 2.68 ms (3.74); ppm_type 2 4.51 ms (5.48);
// conservative, 128^3 and 3 species, 0.38 ms (0.46).
#include <algorithm>
#include <climits>

#include "mx_internal.H"
#include "mx_march.H"

using namespace mxd;
using namespace mxh;

namespace {

// threads of a block: the tile's columns grown by one cell on each side,
// rounded up to whole waves
__host__ __device__ constexpr int fused_nt(int tx, int ty) {
    return ((tx + 2) * (ty + 2) + 63) / 64 * 64;
}

// the register budget, as waves per SIMD: 4 (128 VGPRs) where the advective
// ppm_type 1 kernel fits it and 4 blocks' LDS fit a CU, else 3 (168)
constexpr int fused_wpe(int ppm, bool cons, int tx, int ty, int mode) {
    return ppm == 1 && !cons && mode == 0 && tx * ty == 16 * 11 ? 4 : 3;
}

struct FBox {
    int hi[3];
    int pad_ = 0;  // explicit, so that equal tables are equal byte for byte
    DA s, fo;
    DA um[3], se[3];
    // plane strides in bytes: s, force, umac x / y / z, sedge x / y / z
    long long ks[8];
    // the box's level: its domain and, per direction, the cell width
    int domlo[3], domhi[3];
    DivBy h[3];
    // the flux epilogue (FComp::flux): the fluxes and the level's base
    // state at cell heights (bc_a, bc_b: old, new) and at edges (be_a, be_b)
    DA sf[3];
    const double *bc_a, *bc_b, *be_a, *be_b;
};

// one block's work: nx x ny columns and nz planes of one box from (x0, y0, z0)
struct FTile {
    int box, x0, y0, z0;
    int nx, ny, nz;
    int zgen;  // bits: a z side (0 low, 1 high) in reach needs more than the upwind cell
};

struct FComp {
    int bclo[3], bchi[3];
    int comp;  // state / edge-state component
    // flux epilogue of this component (MakeRhoHFlux's planar branches,
    // MaestroMakeFlux.cpp:557-620): 0 none; 1 umac (rhoh0_edge + sedge)
    // (enthalpy_pred_type 1, 3); 2 umac sedge (enthalpy_pred_type 0)
    int flux;
};

struct FArgs {
    double dt, rel_eps, dt2, dt3, tf, ef;  // tf, ef: h x the factors of the
                                           // transverse and edge terms
    int num_comp;
    int is_vel;
};

// The table's pointer, behind the optimiser's back: what is read from it is
// read (by scalar loads, from the constant address space) where it is used, not
// kept in scalar registers over the whole loop (which overflow into vector
// lanes, two vector instructions per use).
typedef __attribute__((address_space(4))) const FBox cbox;
__device__ __forceinline__ cbox* fresh(const FBox* p) {
    unsigned long long a = (unsigned long long)p;
    asm("" : "+s"(a));
    return (cbox*)a;
}

// the flux of edge state `se` on d-face (i, j, k) (MakeRhoHFlux, planar,
// MaestroMakeFlux.cpp:557-620: umac (rhoh0_edge + sedge), the base state at
// the face's height, averaged over old and new, from the edge-centred state on
// vertical faces)
__device__ __forceinline__ void flux_store(const FBox& B, int d, int i, int j, int k, int comp,
                                           int kind, double um, double se) {
    double f;
    if (kind == 1) {
        gcd* a = (gcd*)(d == 2 ? B.be_a : B.bc_a);
        gcd* b = (gcd*)(d == 2 ? B.be_b : B.bc_b);
        f = um * (0.5 * (a[k] + b[k]) + se);
    } else {
        f = um * se;
    }
    ((gd*)B.sf[d].p)[B.sf[d].off(i, j, k, comp)] = f;
}

// What an acting boundary condition makes of the face on a domain side
// (MaestroMakeEdgeScalars.cpp:709-738, 931-961, 1446-1480): foextrap, hoextrap
// and reflect_even take the inside cell's state at every stage, ext_dir the
// outside cell's value, reflect_odd zero.
enum { kInside = 1, kOutside = 2, kZero = 3 };
__device__ __forceinline__ int side_kind(int bc) {
    if (bc == MX_BC_EXT_DIR) return kOutside;
    if (bc == MX_BC_REFLECT_ODD) return kZero;
    return bc == MX_BC_FOEXTRAP || bc == MX_BC_HOEXTRAP || bc == MX_BC_REFLECT_EVEN ? kInside : 0;
}

// one direction's domain sides as the faces at `pos` see them
struct Side {
    bool lo, hi;  // on an acting low / high side: the upwind cell is the inside one
    bool fixed;   // its value is not computed (ext_dir, reflect_odd)
    bool zero;    // reflect_odd
    bool clamp;   // the normal velocity does not enter through it
    __device__ __forceinline__ Side(int pos, int dlo, int dhi, int bclo, int bchi, bool normal) {
        const int kl = side_kind(bclo), kh = side_kind(bchi);
        lo = kl && pos == dlo;
        hi = kh && pos == dhi + 1;
        const int k = lo ? kl : (hi ? kh : 0);
        const int bc = lo ? bclo : bchi;
        fixed = k >= kOutside;
        zero = k == kZero;
        clamp = normal && k == kInside && bc != MX_BC_REFLECT_EVEN;
    }
    // a stage's state x, s being the predictor's state (final on a fixed side)
    __device__ __forceinline__ double set(double x, double s) const {
        if (clamp) x = lo ? dmin(x, 0.0) : dmax(x, 0.0);
        return fixed ? s : x;
    }
};

// a face's upwind choice: `left` its low cell, `both` the average (|u| <=
// rel_eps); `traced`: the cell's state is traced to it (ppm_trace: u > rel_eps
// from the left, u < -rel_eps from the right)
struct Face {
    bool left, both, traced;
    __device__ __forceinline__ Face(double u, double eps, bool lo, bool hi) {
        const bool up = u > 0.0, off = dabs(u) > eps;
        left = (up | hi) & !lo;
        both = !(off | lo | hi);
        traced = off & !(left ^ up);
    }
};

// MODE, the boundary conditions of the domain sides in the tile's reach: 0: each
// side is free of overrides or extrapolates to first order (or evenly), which
// only picks the face's upwind cell; 1: a z side may carry any; 2: any side may.
template <int PPM, bool CONS, int TX, int TY, int MODE>
__global__ void __launch_bounds__(fused_nt(TX, TY))
    __attribute__((amdgpu_waves_per_eu(fused_wpe(PPM, CONS, TX, TY, MODE))))
    k_es_fused(const FBox* __restrict__ boxes, const FTile* __restrict__ tiles,
               const FComp* __restrict__ comps, FArgs A, int ntile, int xmode) {
    constexpr bool GEN = MODE == 2;
    constexpr int NT = fused_nt(TX, TY);
    constexpr int G = PPM == 2 ? 3 : 2;
    constexpr int W = TX + 2;
    constexpr int H = TY + 2;
    constexpr int SW = W + 2 * G;
    constexpr int SH = H + 2 * G;
    // x-faces per row of the x-velocity plane, y-faces per column of the
    // y-velocity plane: the low faces of the grown tile's cells; the
    // conservative form's divergence reads the high faces too
    constexpr int UW = W + (CONS ? 1 : 0);
    constexpr int VH = H + (CONS ? 1 : 0);
    constexpr int FO = PPM == 2 ? 1 : 0;
    constexpr int FXW = W + 1 + 2 * FO;  // x-face values per row
    constexpr int FYH = H + 1 + 2 * FO;  // y-face values per column
    static_assert(W * H <= NT, "tile too large for the block");
    constexpr int NS = (SW * SH + NT - 1) / NT;
    constexpr int NU = (UW * H + NT - 1) / NT;
    constexpr int NV = (W * VH + NT - 1) / NT;
    constexpr int NFX = (FXW * H + NT - 1) / NT;
    constexpr int NFY = (W * FYH + NT - 1) / NT;

    // One block of LDS, so that the slots a column past the tile reads as its
    // neighbours' lie in it: S first, whose rows keep tid - W in bounds.  Every
    // array starts at a multiple of 512 bytes from the first, so that one
    // two-address read reaches the same column of two of them.
    constexpr int UP = NU * NT, VP = NV * NT;
    constexpr int oS = 0, oU = oS + (SW * SH + 63) / 64 * 64, oV = oU + 3 * UP, oFX = oV + 3 * VP,
                  oFY = oFX + NFX * NT, oHX = oFY + NFY * NT, oHY = oHX + NT, oTZ = oHY + NT,
                  oXY = oTZ + NT, oYX = oXY + NT, oXZ = oYX + NT, oYZ = oXZ + NT, oEX = oYZ + NT,
                  oEY = oEX + NT, oFL = oEY + NT, oBB = oFL + NT, oSC = oBB + (CONS ? 2 * NT : 0),
                  oCZ = oSC + (CONS ? 2 * NT : 0), oEnd = oCZ + (CONS ? NT : 0) + W + 2;
    __shared__ double lds[oEnd];
    double* S = lds + oS;
    double* FX = lds + oFX;
    double* FY = lds + oFY;
    double* HX = lds + oHX;
    double* HY = lds + oHY;
    double* TZ = lds + oTZ;
    double* XY = lds + oXY;
    double* YX = lds + oYX;
    double* XZ = lds + oXZ;
    double* YZ = lds + oYZ;
    double* EX = lds + oEX;
    double* EY = lds + oEY;
    double* FL = lds + oFL;
    double* CZ = lds + oCZ;

    // xmode 1, 2: the XCD-aware orders of xcd_tile over a 1-D grid; 0: tile
    // blockIdx.x and component blockIdx.z
    int tix = blockIdx.x, vc = blockIdx.z;
    if (xmode != 0 && !xcd_tile(ntile, A.num_comp, xmode, tix, vc)) return;
    const FTile tl = tiles[tix];
    const FBox& B = boxes[tl.box];
    const int X0 = tl.x0, Y0 = tl.y0, nx = tl.nx, ny = tl.ny;
    const int z0 = tl.z0, z1 = tl.z0 + tl.nz - 1;
    const bool last_x = X0 + nx - 1 == B.hi[0];
    const bool last_y = Y0 + ny - 1 == B.hi[1];
    const bool last_z = z1 == B.hi[2];

    const int comp = comps[vc].comp;
    const int flux = comps[vc].flux;
    const int* bcl = comps[vc].bclo;
    const int* bch = comps[vc].bchi;

    const double dt = A.dt, eps = A.rel_eps, dt2 = A.dt2, dt3 = A.dt3;
    const double tfx = uniform(A.tf / B.h[0].d), tfy = uniform(A.tf / B.h[1].d),
                 tfz = uniform(A.tf / B.h[2].d);
    const double efx = uniform(A.ef / B.h[0].d), efy = uniform(A.ef / B.h[1].d),
                 efz = uniform(A.ef / B.h[2].d);
    double dt2hx = 0.0, dt2hy = 0.0, dt2hz = 0.0;
    if (CONS) {
        dt2hx = uniform(dt2 / B.h[0].d);
        dt2hy = uniform(dt2 / B.h[1].d);
        dt2hz = uniform(dt2 / B.h[2].d);
    }

    const int tid = threadIdx.x;
    const int a = tid % W;  // local column: cell (X0 + a - 1, Y0 + b - 1)
    const int b = tid / W;
    const int I = X0 + a - 1;
    const int J = Y0 + b - 1;
    const int si = (a + G) + (b + G) * SW;
    const int ui = CONS ? a + b * UW : tid;
    const bool inx = a >= 1 && a <= nx, iny = b >= 1 && b <= ny;
    const bool st_x = a >= 1 && iny && (a <= nx || (last_x && a == nx + 1));
    const bool st_y = b >= 1 && inx && (b <= ny || (last_y && b == ny + 1));
    const bool st_z = inx && iny;
    const Side dx(I, B.domlo[0], B.domhi[0], bcl[0], bch[0], A.is_vel && comp == 0);
    const Side dy(J, B.domlo[1], B.domhi[1], bcl[1], bch[1], A.is_vel && comp == 1);
    // the z-faces on acting sides
    const int zlo = side_kind(bcl[2]) ? B.domlo[2] : INT_MIN;
    const int zhi = side_kind(bch[2]) ? B.domhi[2] + 1 : INT_MIN;
    // z-face q may need more than its upwind cell: a boundary stencil, a fixed
    // value or a clamp.  Uniform, and rare: the branches it guards read the
    // table and the column's cells again.
    const bool zgl = tl.zgen & 1, zgh = tl.zgen & 2;
    auto z_general = [&](int q) {
        return MODE > 0 && ((zgl && q <= B.domlo[2] + 3) || (zgh && q >= B.domhi[2] - 2));
    };
    auto side_z = [&](int q) {
        cbox* Bf = fresh(&B);
        return Side(q, Bf->domlo[2], Bf->domhi[2], bcl[2], bch[2], A.is_vel && comp == 2);
    };

    // byte offsets within a plane of the tile's arrays; a column past the
    // tile takes the tile's last one
    const DA sv = B.s, fv = B.fo, uv = B.um[0], vv = B.um[1], wv = B.um[2];
    const int ac = min(a, nx + 1), bc = min(b, ny + 1);
    const unsigned sjs = (unsigned)sv.js * 8u;
    const unsigned oCol = (unsigned)(ac + G) * 8u + (unsigned)(bc + G) * sjs;
    const unsigned oF = (unsigned)ac * 8u + (unsigned)bc * (unsigned)fv.js * 8u;
    const unsigned oW = (unsigned)ac * 8u + (unsigned)bc * (unsigned)wv.js * 8u;
    const unsigned oE0 = (unsigned)ac * 8u + (unsigned)bc * (unsigned)B.se[0].js * 8u;
    const unsigned oE1 = (unsigned)ac * 8u + (unsigned)bc * (unsigned)B.se[1].js * 8u;
    const unsigned oE2 = (unsigned)ac * 8u + (unsigned)bc * (unsigned)B.se[2].js * 8u;
    // each thread's slots of the staged planes (an item past the plane is the
    // thread's first again)
    unsigned offS[NS], offU[NU], offV[NV];
    int slS[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int idx = tid + k * NT < SW * SH ? tid + k * NT : tid;
        slS[k] = idx;
        offS[k] = (unsigned)min(idx % SW, nx + 1 + 2 * G) * 8u +
                  (unsigned)min(idx / SW, ny + 1 + 2 * G) * sjs;
    }
#pragma unroll
    for (int k = 0; k < NU; ++k) {
        const int idx = tid + k * NT;
        offU[k] = (unsigned)min(idx % UW, nx + 2) * 8u +
                  (unsigned)min(idx / UW, ny + 1) * (unsigned)uv.js * 8u;
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int idx = tid + k * NT;
        offV[k] = (unsigned)min(idx % W, nx + 1) * 8u +
                  (unsigned)min(idx / W, ny + 2) * (unsigned)vv.js * 8u;
    }
    // S slot of this thread's x- and y-face items
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

    // Plane bases (block-uniform).  Loads: s, u, v, w and the force of the
    // next plane to load, s also G planes further for the column window; stores: the edge
    // states' plane.
    gcc* sN = (gcc*)sv.p + 8 * sv.off(X0 - 1 - G, Y0 - 1 - G, z0 - 1, comp);
    gcc* uN = (gcc*)uv.p + 8 * uv.off(X0 - 1, Y0 - 1, z0 - 1);
    gcc* vN = (gcc*)vv.p + 8 * vv.off(X0 - 1, Y0 - 1, z0 - 1);
    gcc* wN = (gcc*)wv.p + 8 * wv.off(X0 - 1, Y0 - 1, z0 - 1);
    gcc* fN = (gcc*)fv.p + 8 * fv.off(X0 - 1, Y0 - 1, z0 - 1, comp);
    gcc* sC = sN + G * B.ks[0];
    gc* e0P = (gc*)B.se[0].p + 8 * B.se[0].off(X0 - 1, Y0 - 1, z0 - 3, comp);
    gc* e1P = (gc*)B.se[1].p + 8 * B.se[1].off(X0 - 1, Y0 - 1, z0 - 3, comp);
    gc* e2P = (gc*)B.se[2].p + 8 * B.se[2].off(X0 - 1, Y0 - 1, z0 - 2, comp);

    // column state of step q, moved on to q + 1 in phase 1: v[jj] =
    // s(q - 4 + jj); w_p, w_q, w_hi: w on z-faces q - 1, q, q + 1; p..: loaded
    // for the next step
    double v[9];
#pragma unroll
    for (int jj = 0; jj < 9; ++jj) v[jj] = 0.0;
#pragma unroll
    for (int jj = 4 - G; jj < 4 + G; ++jj) v[jj + 1] = gload(sN + (jj - 4) * B.ks[0], oCol);
    double w_p = 0.0, w_q = 0.0, w_hi = gload(wN, oW), fo_p = 0.0, fo_q = 0.0;
    double pcs = gload(sC, oCol), pw = gload(wN + B.ks[4], oW), pf = gload(fN, oF);
    // z face values q - 1, q, q + 1 at phase 2, and the slope of cell q
    double zf0 = 0.0, zf1 = 0.0, zf2 = 0.0, zsl = 0.0;
    double sig_lo = 0.0, Ipz_prev = 0.0;
    double sx = 0.0, sy = 0.0, sz = 0.0, sx_p = 0.0, sy_p = 0.0, sz_p = 0.0;
    double tx_p = 0.0, ty_p = 0.0, cx_p = 0.0, cy_p = 0.0, bp = 0.0;
    double tzx_p = 0.0, tzy_p = 0.0, exy_p = 0.0, eyx_p = 0.0;
    if (PPM == 1) {
        const double d0 = vl_slope(v[3], v[4], v[5]);
        zsl = vl_slope(v[4], v[5], v[6]);
        zf1 = face1(v[4], v[5], d0, zsl);  // face z0 - 1
    } else {
        zf0 = cs_face(v[2], v[3], v[4], v[5]);
        zf1 = cs_face(v[3], v[4], v[5], v[6]);
        zf2 = cs_face(v[4], v[5], v[6], v[7]);
        sig_lo = div_by(dabs(w_hi) * dt, B.h[2]);
    }

    // Plane q + 1's loads are issued at the start of step q and land in
    // registers (the barriers wait for LDS traffic only); phase 3 puts them
    // in LDS.  Each thread owns fixed slots of the staged planes.
    double pS[NS], pU[NU], pV[NV];
    auto load_planes = [&](gcc* s, gcc* u, gcc* vp) {
#pragma unroll
        for (int k = 0; k < NS; ++k) pS[k] = gload(s, offS[k]);
#pragma unroll
        for (int k = 0; k < NU; ++k) pU[k] = gload(u, offU[k]);
#pragma unroll
        for (int k = 0; k < NV; ++k) pV[k] = gload(vp, offV[k]);
    };
    auto stage_planes = [&](int slot) {
#pragma unroll
        for (int k = 0; k < NS; ++k) S[(k + 1) * NT <= SW * SH ? tid + k * NT : slS[k]] = pS[k];
#pragma unroll
        for (int k = 0; k < NU; ++k) lds[oU + slot * UP + tid + k * NT] = pU[k];
#pragma unroll
        for (int k = 0; k < NV; ++k) lds[oV + slot * VP + tid + k * NT] = pV[k];
    };
    // plane k of s (rare paths)
    auto s_plane = [&](int k) {
        cbox* Bf = fresh(&B);
        return (gcc*)Bf->s.p + 8 * ((long long)(X0 - 1 - G - Bf->s.b0) +
                                    (long long)(Y0 - 1 - G - Bf->s.b1) * Bf->s.js +
                                    (long long)(k - Bf->s.b2) * Bf->s.ks +
                                    (long long)comp * Bf->s.ns);
    };
    load_planes(sN, uN, vN);
    stage_planes(0);
    int slot_q = 0, slot_p = 2, slot_o = 1;  // planes q, q - 1, q - 2 (then q + 1)
    // on to the next plane; the loads stay at plane z1 + 1 (a step past it loads
    // it again: conditional loads would leave the compiler's wait counters open
    // and stall on every load in flight)
    auto advance = [&](bool more) {
        __attribute__((address_space(4))) const long long* ks = fresh(&B)->ks;
        if (more) {
            sN += ks[0];
            sC += ks[0];
            fN += ks[1];
            uN += ks[2];
            vN += ks[3];
            wN += ks[4];
        }
        e0P += ks[5];
        e1P += ks[6];
        e2P += ks[7];
    };
    // The edge states of step r = q - 1: x- and y-faces of plane r - 1, z-face
    // r, from the column state of step r (at the first two steps, with nothing to
    // store, of whatever LDS holds).
    auto edges = [&](int q) {
        const double* ULp = lds + oU + slot_p * UP;  // plane r
        const double* VLp = lds + oV + slot_p * VP;
        const double* ULo = lds + oU + slot_o * UP;  // plane r - 1
        const double* VLo = lds + oV + slot_o * VP;
        const double* SCo = lds + oSC + (CONS ? (q & 1) * NT : 0);  // s, plane r - 1
        const double u0 = ULo[ui], v0 = VLo[tid];
        const Face fx(u0, eps, dx.lo, dx.hi), fy(v0, eps, dy.lo, dy.hi),
            fz(w_q, eps, q - 1 == zlo, q - 1 == zhi);
        auto edge_x = [&](double s, int o) {
            const int t = tid + o;
            const double y1 = VLo[t + W], y0 = VLo[t], h1 = YZ[t + W], h0 = YZ[t];
            double x = s - (CONS ? efy * (h1 * y1 - h0 * y0) : efy * (y1 + y0) * (h1 - h0));
            x = x - EY[t];
            if (CONS) x = x - dt2hx * SCo[t] * (ULo[ui + o + 1] - ULo[ui + o]);
            return x + dt2 * FL[t];
        };
        auto edge_y = [&](double s, int n) {
            const int t = tid + n * W, u = ui + n * UW;
            const double x1 = ULo[u + 1], x0 = ULo[u], h1 = XZ[t + 1], h0 = XZ[t];
            double x = s - (CONS ? efx * (h1 * x1 - h0 * x0) : efx * (x1 + x0) * (h1 - h0));
            x = x - EX[t];
            if (CONS) x = x - dt2hy * SCo[t] * (VLo[t + W] - VLo[t]);
            return x + dt2 * FL[t];
        };
        const double a1 = ULp[ui + 1], a0 = ULp[ui], b1 = VLp[tid + W], b0 = VLp[tid];
        const double x1 = XY[tid + 1], x0 = XY[tid], y1 = YX[tid + W], y0 = YX[tid];
        const double exy = CONS ? efx * (x1 * a1 - x0 * a0) : efx * (a1 + a0) * (x1 - x0);
        const double eyx = CONS ? efy * (y1 * b1 - y0 * b0) : efy * (b1 + b0) * (y1 - y0);
        auto edge_z = [&](double s, bool left) {
            double x = s - (left ? exy_p : exy);
            x = x - (left ? eyx_p : eyx);
            if (CONS) x = x - dt2hz * (left ? v[3] : v[4]) * (left ? w_q - w_p : w_hi - w_q);
            return x + dt2 * (left ? fo_p : fo_q);
        };
        double rx = edge_x(sx_p, fx.left ? -1 : 0);
        double ry = edge_y(sy_p, fy.left ? -1 : 0);
        double rz = edge_z(sz, fz.left);
        if (fx.both | fy.both | fz.both) {
            gcc* row = s_plane(q - 2);
            if (fx.both)
                rx = 0.5 * (edge_x(gload(row, oCol - 8u), -1) + edge_x(gload(row, oCol), 0));
            if (fy.both)
                ry = 0.5 * (edge_y(gload(row, oCol - sjs), -1) + edge_y(gload(row, oCol), 0));
            if (fz.both) rz = 0.5 * (edge_z(v[3], true) + edge_z(v[4], false));
        }
        if (GEN) {
            rx = dx.set(rx, sx_p);
            ry = dy.set(ry, sy_p);
        }
        if (z_general(q - 1)) rz = side_z(q - 1).set(rz, sz);
        exy_p = exy;
        eyx_p = eyx;
        if (q >= z0 + 2) {
            if (st_x) gstore(e0P, oE0, rx);
            if (st_y) gstore(e1P, oE1, ry);
            if (flux) {
                if (st_x) flux_store(B, 0, I, J, q - 2, comp, flux, u0, rx);
                if (st_y) flux_store(B, 1, I, J, q - 2, comp, flux, v0, ry);
            }
        }
        if (q > z0 && (q <= z1 + 1 || last_z) && st_z) {
            gstore(e2P, oE2, rz);
            if (flux) flux_store(B, 2, I, J, q - 1, comp, flux, w_q, rz);
        }
    };
    // w and s of plane z0 are loaded: step z0 - 1 loads the planes after
    sN += B.ks[0];
    sC += B.ks[0];
    fN += B.ks[1];
    uN += B.ks[2];
    vN += B.ks[3];
    wN += 2 * B.ks[4];
    __syncthreads();

    for (int q = z0 - 1; q <= z1 + 1; ++q) {
        const double* ULq = lds + oU + slot_q * UP;
        const double* VLq = lds + oV + slot_q * VP;
        const double* ULp = lds + oU + slot_p * UP;
        const double* VLp = lds + oV + slot_p * VP;
        load_planes(sN, uN, vN);

        // ---- 1a: the edge states of step q - 1; the column state moves on
        edges(q);
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) v[jj] = v[jj + 1];
        v[4 + G] = pcs;
        sx_p = sx;
        sy_p = sy;
        sz_p = sz;
        w_p = w_q;
        w_q = w_hi;
        w_hi = pw;
        fo_p = fo_q;
        fo_q = pf;
        pcs = gload(sC, oCol);
        pw = gload(wN, oW);
        pf = gload(fN, oF);

        // ---- 1b: PPM face values of plane q
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
        cbox* Bq = fresh(&B);
        const DivBy hx{Bq->h[0].d, Bq->h[0].r, Bq->h[0].rl}, hy{Bq->h[1].d, Bq->h[1].r, Bq->h[1].rl},
            hz{Bq->h[2].d, Bq->h[2].r, Bq->h[2].rl};
        __syncthreads();

        // ---- 2: the predictor's upwind states on the low faces of cell q
        const double ux = ULq[ui], vy = VLq[tid];
        const Face fx(ux, eps, dx.lo, dx.hi), fy(vy, eps, dy.lo, dy.hi),
            fz(w_q, eps, q == zlo, q == zhi);
        {
            const bool px = fx.traced, py = fy.traced, pz = fz.traced;
            const double gx = div_by(dabs(ux) * dt, hx), gy = div_by(dabs(vy) * dt, hy);
            sx = predict<PPM, 1, 1>(S + si, FX + (a + FO) + b * FXW, fx.left, px, gx);
            sy = predict<PPM, W, SW>(S + si, FY + a + (b + FO) * W, fy.left, py, gy);
            if (PPM == 1) {
                const double d1 = vl_slope(v[4], v[5], v[6]);
                zf2 = face1(v[4], v[5], zsl, d1);
                zsl = d1;
                const double s0 = fz.left ? v[3] : v[4];
                const double gz = div_by(dabs(w_q) * dt, hz);
                const double t = cw_trace(s0, zf1, fz.left ? zf0 : zf2, gz);
                sz = pz ? t : s0;
                zf0 = zf1;
                zf1 = zf2;
                // (face z0 - 1 enters nothing that is stored, and its low cell's
                // stencil would reach a plane past the ghosts of a box that
                // starts two or three planes above the domain's low side)
                if (q >= z0 && z_general(q)) {
                    cbox* Bf = fresh(&B);
                    const int dl = Bf->domlo[2], dh = Bf->domhi[2];
                    const int pos = q - (fz.left ? 1 : 0);
                    if (ppm_special<PPM>(pos, dl, dh, bcl[2], bch[2])) {
                        double w9[9], sm, sp;
#pragma unroll
                        for (int o = 0; o < 9; ++o)
                            w9[o] = o >= 2 && o <= 6
                                        ? (fz.left ? gload(s_plane(q - 5 + o), oCol)
                                                   : gload(s_plane(q - 4 + o), oCol))
                                        : 0.0;
                        ppm_edges<PPM, 2>(w9, pos, dl, dh, bcl[2], bch[2], sm, sp);
                        const double x =
                            trace_face(s0, fz.left ? sp : sm, fz.left ? sm : sp, gz);
                        sz = pz ? x : s0;
                    }
                }
            } else {
                double sm, sp, Ipz, Imz;
                const double f3 = cs_face(v[4], v[5], v[6], v[7]);
                cs_cell(v, zf0, zf1, zf2, f3, 1.e-10, sm, sp);
                zf0 = zf1;
                zf1 = zf2;
                zf2 = f3;
                if (z_general(q)) {
                    cbox* Bf = fresh(&B);
                    const int dl = Bf->domlo[2], dh = Bf->domhi[2];
                    if (ppm_special<PPM>(q, dl, dh, bcl[2], bch[2]))
                        ppm_edges<PPM, 2>(v, q, dl, dh, bcl[2], bch[2], sm, sp);
                }
                const double sig_hi = div_by(dabs(w_hi) * dt, hz);
                trace_sig(v[4], sm, sp, w_hi, w_q, sig_hi, sig_lo, eps, Ipz, Imz);
                sig_lo = sig_hi;
                sz = fz.left ? Ipz_prev : Imz;
                Ipz_prev = Ipz;
            }
            if (GEN) {
                // boundary stencils of the tile's own faces (another's may
                // reach past S)
                const int pI = I - (fx.left ? 1 : 0), pJ = J - (fy.left ? 1 : 0);
                if (a >= 1 && ppm_special<PPM>(pI, B.domlo[0], B.domhi[0], bcl[0], bch[0]))
                    sx = predict_special<PPM, 0, 1>(S + si, fx.left, px, gx, I, B.domlo[0],
                                                    B.domhi[0], bcl[0], bch[0]);
                if (b >= 1 && ppm_special<PPM>(pJ, B.domlo[1], B.domhi[1], bcl[1], bch[1]))
                    sy = predict_special<PPM, 1, SW>(S + si, fy.left, py, gy, J, B.domlo[1],
                                                     B.domhi[1], bcl[1], bch[1]);
            }
            if (fx.both | fy.both | fz.both) {  // u == 0 averages the cells
                if (fx.both && !(dabs(ux) > 0.0)) sx = 0.5 * (S[si - 1] + S[si]);
                if (fy.both && !(dabs(vy) > 0.0)) sy = 0.5 * (S[si - SW] + S[si]);
                if (fz.both && !(dabs(w_q) > 0.0)) sz = 0.5 * (v[3] + v[4]);
            }
            if (GEN) {
                if (dx.fixed || dx.clamp)
                    sx = dx.set(sx, dx.zero ? 0.0 : (dx.lo ? S[si - 1] : S[si]));
                if (dy.fixed || dy.clamp)
                    sy = dy.set(sy, dy.zero ? 0.0 : (dy.lo ? S[si - SW] : S[si]));
            }
            if (z_general(q)) {
                const Side dz = side_z(q);
                if (dz.fixed || dz.clamp) sz = dz.set(sz, dz.zero ? 0.0 : (dz.lo ? v[3] : v[4]));
            }
        }
        HX[tid] = sx;
        HY[tid] = sy;
        TZ[tid] = CONS ? tfz * (sz * w_q - sz_p * w_p) : tfz * (w_q + w_p) * (sz - sz_p);
        double* BBq = lds + oBB + (CONS ? (q & 1) * NT : 0);  // planes q and q - 1
        double* SCq = lds + oSC + (CONS ? (q & 1) * NT : 0);
        const double* BBp = lds + oBB + (CONS ? (~q & 1) * NT : 0);
        double bq = 0.0;
        if (CONS) {
            double dv = ULq[ui + 1] - ux + VLq[tid + W] - vy + w_hi - w_q;
            dv = div_by(dv, hx);
            bq = dt3 * v[4] * dv;
            BBq[tid] = bq;
            SCq[tid] = v[4];
            CZ[tid] = tfz * v[3] * (w_q - w_p);
        }
        __syncthreads();

        // ---- 3: corner-coupled states
        {
            const double up = ULp[ui], vp = VLp[tid];  // plane q - 1
            const Face gx(up, eps, dx.lo, dx.hi), gy(vp, eps, dy.lo, dy.hi);
            // the transverse y term of the cell at column t and the state s
            // after it (simhxy); then the same along x (simhyx), and by the z
            // term of plane q - 1 (simhxz, simhyz)
            auto ycell = [&](int t, double& tt, double& cc) {
                const double y1 = VLq[t + W], y0 = VLq[t], h1 = HY[t + W], h0 = HY[t];
                tt = CONS ? tfy * (h1 * y1 - h0 * y0) : tfy * (y1 + y0) * (h1 - h0);
                cc = CONS ? tfy * SCq[t] * (y1 - y0) : 0.0;
            };
            auto xcell = [&](int t, int u, double& tt, double& cc) {
                const double x1 = ULq[u + 1], x0 = ULq[u], h1 = HX[t + 1], h0 = HX[t];
                tt = CONS ? tfx * (h1 * x1 - h0 * x0) : tfx * (x1 + x0) * (h1 - h0);
                cc = CONS ? tfx * SCq[t] * (x1 - x0) : 0.0;
            };
            auto corner_x = [&](double s, int o) {
                double tt, cc;
                ycell(tid + o, tt, cc);
                return CONS ? ((s - tt) - BBq[tid + o]) + cc : s - tt;
            };
            auto corner_y = [&](double s, int n) {
                double tt, cc;
                xcell(tid + n * W, ui + n * UW, tt, cc);
                return CONS ? ((s - tt) - BBq[tid + n * W]) + cc : s - tt;
            };
            auto corner_z = [&](double s, int t) {
                return CONS ? ((s - TZ[t]) - BBp[t]) + CZ[t] : s - TZ[t];
            };
            double tx_q, ty_q, cx_q, cy_q;
            ycell(tid, ty_q, cy_q);
            xcell(tid, ui, tx_q, cx_q);
            auto corner_f = [&](double s, bool left, double tp, double tq, double cp, double cq) {
                const double x = s - (left ? tp : tq);
                return CONS ? (x - (left ? bp : bq)) + (left ? cp : cq) : x;
            };
            double xy = corner_x(sx, fx.left ? -1 : 0);
            double yx = corner_y(sy, fy.left ? -1 : 0);
            double xz = corner_z(sx_p, tid + (gx.left ? -1 : 0));
            double yz = corner_z(sy_p, tid + (gy.left ? -W : 0));
            double zx = corner_f(sz, fz.left, tx_p, tx_q, cx_p, cx_q);
            double zy = corner_f(sz, fz.left, ty_p, ty_q, cy_p, cy_q);
            if (fx.both | fy.both | fz.both | gx.both | gy.both) {
                gcc* sq = s_plane(q);
                gcc* sp = s_plane(q - 1);
                if (fx.both)
                    xy = 0.5 * (corner_x(gload(sq, oCol - 8u), -1) + corner_x(v[4], 0));
                if (fy.both)
                    yx = 0.5 * (corner_y(gload(sq, oCol - sjs), -1) + corner_y(v[4], 0));
                if (gx.both)
                    xz = 0.5 * (corner_z(gload(sp, oCol - 8u), tid - 1) +
                                corner_z(v[3], tid));
                if (gy.both)
                    yz = 0.5 * (corner_z(gload(sp, oCol - sjs), tid - W) +
                                corner_z(v[3], tid));
                if (fz.both) {
                    zx = 0.5 * (corner_f(v[3], true, tx_p, tx_q, cx_p, cx_q) +
                                corner_f(v[4], false, tx_p, tx_q, cx_p, cx_q));
                    zy = 0.5 * (corner_f(v[3], true, ty_p, ty_q, cy_p, cy_q) +
                                corner_f(v[4], false, ty_p, ty_q, cy_p, cy_q));
                }
            }
            if (GEN) {
                xy = dx.set(xy, sx);
                yx = dy.set(yx, sy);
                xz = dx.set(xz, sx_p);
                yz = dy.set(yz, sy_p);
            }
            if (z_general(q)) {
                const Side dz = side_z(q);
                zx = dz.set(zx, sz);
                zy = dz.set(zy, sz);
            }
            XY[tid] = xy;
            YX[tid] = yx;
            XZ[tid] = xz;
            YZ[tid] = yz;
            // the z edge terms of plane q - 1
            EX[tid] = CONS ? efz * (zx * w_q - tzx_p * w_p) : efz * (w_q + w_p) * (zx - tzx_p);
            EY[tid] = CONS ? efz * (zy * w_q - tzy_p * w_p) : efz * (w_q + w_p) * (zy - tzy_p);
            FL[tid] = fo_p;
            tzx_p = zx;
            tzy_p = zy;
            tx_p = tx_q;
            ty_p = ty_q;
            cx_p = cx_q;
            cy_p = cy_q;
            bp = bq;
        }
        // plane q + 1 takes plane q - 2's slots
        stage_planes(slot_o);
        __syncthreads();

        advance(q < z1);
        const int s_new = slot_o;
        slot_o = slot_p;
        slot_p = slot_q;
        slot_q = s_new;
    }
    edges(z1 + 2);
}

}  // namespace

namespace mxh {

bool fused_edge_scal_ok(const mx_adv_ctx* c, int is_conservative) {
    (void)is_conservative;
    return c->p.dim == 3 && (c->p.ppm_type == 1 || c->p.ppm_type == 2) &&
           c->p.ppm_trace_forces == 0 && c->fused_edge;
}

// unsigned 32-bit byte offsets in a plane: a tile and its stencil span at most 25
// rows, which follow each other upwards
bool fused_edge_rows_ok(const EdgeLevel& L) {
    const long long lim = 0x7fffffffLL / (8 * 26);
    const long long max = 0x7fffffffLL;  // past which the launch refuses them
    auto ok = [&](const mx_multifab* m) {
        for (int b = 0; b < m->nfab; ++b) {
            const long long js = m->fab[b].jstride;
            if (js > max || m->fab[b].kstride > max) continue;
            if (js < 0 || js > lim) return false;
        }
        return true;
    };
    bool r = ok(L.state) && ok(L.force);
    for (int d = 0; d < 3; ++d) r = r && ok(&L.umac->dir[d]) && ok(&L.sedge->dir[d]);
    return r;
}

namespace {

// does boundary code `bc` override anything (everything but INT_DIR)?
bool bc_acts(int bc) {
    return bc == MX_BC_EXT_DIR || bc == MX_BC_HOEXTRAP || bc == MX_BC_FOEXTRAP ||
           bc == MX_BC_REFLECT_EVEN || bc == MX_BC_REFLECT_ODD;
}

// does it do more than pick the inside cell's state on the side's face?
// (hoextrap has PPM boundary stencils; extrapolation clamps a normal velocity)
bool bc_general(int bc, int is_vel) {
    return bc_acts(bc) && bc != MX_BC_REFLECT_EVEN && (bc != MX_BC_FOEXTRAP || is_vel);
}

// A tile's chunk is out of reach of a direction's sides when each either
// carries no such condition for any component or lies beyond it: the kernel
// evaluates cells [lo0 - 1, lo0 + n] (PPM boundary stencils act within three
// cells of a side) and faces [lo0, lo0 + n] (face overrides act on the side's
// face).
bool tile_clear(const int lo0, int n, int dlo, int dhi, bool act_lo, bool act_hi) {
    const bool clear_lo = !act_lo || lo0 - 1 > dlo + 2;
    const bool clear_hi = !act_hi || lo0 + n < dhi - 2;
    return clear_lo && clear_hi;
}

template <int TX, int TY, int MODE>
int launch_one(mx_adv_ctx* c, const FBox* db, const FTile* dtl, size_t ntile, const FComp* dc,
               const FArgs& A, int num_comp, bool cons) {
    if (ntile == 0) return MX_OK;
    const int xm = c->es_fused_xcd;
    const dim3 grid = xm ? dim3(xcd_tile_blocks((long long)ntile, num_comp))
                         : dim3((unsigned)ntile, 1, (unsigned)num_comp);
    const int nt = (int)ntile;
    dim3 block(fused_nt(TX, TY));
    if (c->p.ppm_type == 1) {
        if (cons)
            MX_LAUNCH(c, "k_es_fused", (k_es_fused<1, true, TX, TY, MODE>), grid, block, db, dtl, dc, A, nt, xm);
        else
            MX_LAUNCH(c, "k_es_fused", (k_es_fused<1, false, TX, TY, MODE>), grid, block, db, dtl, dc, A, nt, xm);
    } else {
        if (cons)
            MX_LAUNCH(c, "k_es_fused", (k_es_fused<2, true, TX, TY, MODE>), grid, block, db, dtl, dc, A, nt, xm);
        else
            MX_LAUNCH(c, "k_es_fused", (k_es_fused<2, false, TX, TY, MODE>), grid, block, db, dtl, dc, A, nt, xm);
    }
    return MX_OK;
}

// blocks of the kernel a CU holds
template <int PPM, bool CONS, int TX, int TY, int MODE>
int fused_blocks() {
    static const int n = [] {
        int v = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, k_es_fused<PPM, CONS, TX, TY, MODE>,
                                                         fused_nt(TX, TY), 0) != hipSuccess) {
            (void)hipGetLastError();
            v = 0;
        }
        return v > 0 ? v : 3;
    }();
    return n;
}
template <int TX, int TY, int MODE>
int fused_blocks(int ppm, bool cons) {
    if (ppm == 1)
        return cons ? fused_blocks<1, true, TX, TY, MODE>() : fused_blocks<1, false, TX, TY, MODE>();
    return cons ? fused_blocks<2, true, TX, TY, MODE>() : fused_blocks<2, false, TX, TY, MODE>();
}

template <int TX, int TY>
int launch_fused(mx_adv_ctx* c, const std::vector<EdgeLevel>& levs, int tz, int is_vel,
                 const mx_bcrec* bcs, const std::vector<int>& scomps,
                 const std::vector<int>& bccomps, int is_conservative) {
    const int num_comp = (int)scomps.size();
    std::vector<FBox> boxes;
    bool zgen = false;
    std::vector<HBox> hb;
    std::vector<ChunkCols> cols;
    std::vector<FTile> tiles, btiles;  // tiles clear of general x/y sides, then the others
    bool act[3][2] = {{false, false}, {false, false}, {false, false}};
    for (int vc = 0; vc < num_comp; ++vc)
        for (int d = 0; d < 3; ++d) {
            act[d][0] = act[d][0] || bc_general(bcs[bccomps[vc]].lo[d], is_vel);
            act[d][1] = act[d][1] || bc_general(bcs[bccomps[vc]].hi[d], is_vel);
        }
    auto clear_xy = [&](const FBox& B, int x, int nx, int y, int ny) {
        return tile_clear(x, nx, B.domlo[0], B.domhi[0], act[0][0], act[0][1]) &&
               tile_clear(y, ny, B.domlo[1], B.domhi[1], act[1][0], act[1][1]);
    };
    const double dt = c->p.dt, dt2 = 0.5 * dt, dt3 = dt / 3.0, dt4 = 0.25 * dt, dt6 = dt / 6.0;
    const bool cons = is_conservative != 0;
    for (const EdgeLevel& L : levs) {
        const auto& grids = c->grids[L.lev];
        for (size_t b = 0; b < grids.size(); ++b) {
            if (L.box >= 0 && (size_t)L.box != b) continue;
            FBox B;
            HBox g = hbox(grids[b]);
            for (int q = 0; q < 3; ++q) {
                B.hi[q] = g.hi[q];
                B.h[q] = div_const(c->p.dx[L.lev][q]);
                B.domlo[q] = c->p.domain_lo[L.lev][q];
                B.domhi[q] = c->p.domain_hi[L.lev][q];
            }
            B.s = to_da(L.state->fab[b]);
            B.fo = to_da(L.force->fab[b]);
            for (int d = 0; d < 3; ++d) {
                B.um[d] = to_da(L.umac->dir[d].fab[b]);
                B.se[d] = to_da(L.sedge->dir[d].fab[b]);
                B.sf[d] = L.sflux ? to_da(L.sflux->dir[d].fab[b]) : null_da();
            }
            B.bc_a = L.bc_a;
            B.bc_b = L.bc_b;
            B.be_a = L.be_a;
            B.be_b = L.be_b;
            const DA* strided[] = {&B.s,     &B.fo,    &B.um[0], &B.um[1],
                                   &B.um[2], &B.se[0], &B.se[1], &B.se[2]};
            for (int q = 0; q < 8; ++q) B.ks[q] = 8 * strided[q]->ks;
            for (const DA* d : strided)
                if (d->js > 0x7fffffffLL || d->ks > 0x7fffffffLL) return MX_ERR_UNSUPPORTED;
            boxes.push_back(B);
            hb.push_back(g);
            ChunkCols col{g.hi[2] - g.lo[2] + 1, {0, 0}};
            for (int y = g.lo[1]; y <= g.hi[1]; y += TY)
                for (int x = g.lo[0]; x <= g.hi[0]; x += TX)
                    ++col.tiles[clear_xy(B, x, std::min(TX, g.hi[0] - x + 1), y,
                                         std::min(TY, g.hi[1] - y + 1))
                                    ? 0
                                    : 1];
            cols.push_back(col);
            zgen = zgen || (col.tiles[0] && !tile_clear(g.lo[2], col.nz, B.domlo[2], B.domhi[2],
                                                        act[2][0], act[2][1]));
        }
    }
    if (tz <= 0) {
        // of the kernels that the launches take (a query loads its kernel)
        bool any[2] = {false, false};
        for (const ChunkCols& col : cols)
            for (int l = 0; l < 2; ++l) any[l] = any[l] || col.tiles[l];
        const int ppm = c->p.ppm_type;
        const int blocks[2] = {!any[0] ? 1
                               : zgen  ? fused_blocks<TX, TY, 1>(ppm, cons)
                                       : fused_blocks<TX, TY, 0>(ppm, cons),
                               any[1] ? fused_blocks<TX, TY, 2>(ppm, cons) : 1};
        tz = pick_chunks(cols, num_comp, blocks);
    }
    for (size_t id = 0; id < boxes.size(); ++id) {
        const HBox& g = hb[id];
        const FBox& B = boxes[id];
        const int nz = g.hi[2] - g.lo[2] + 1, nch = chunk_count(nz, tz);
        for (int ch = 0; ch < nch; ++ch)
            for (int y = g.lo[1]; y <= g.hi[1]; y += TY)
                for (int x = g.lo[0]; x <= g.hi[0]; x += TX) {
                    const int z = chunk_start(nz, nch, ch), ze = chunk_start(nz, nch, ch + 1);
                    FTile T{(int)id,
                            x,
                            y,
                            g.lo[2] + z,
                            std::min(TX, g.hi[0] - x + 1),
                            std::min(TY, g.hi[1] - y + 1),
                            ze - z,
                            0};
                    const bool f = clear_xy(B, x, T.nx, y, T.ny);
                    for (int s = 0; s < 2; ++s)
                        if (!tile_clear(T.z0, T.nz, B.domlo[2], B.domhi[2], s == 0 && act[2][0],
                                        s == 1 && act[2][1]))
                            T.zgen |= 1 << s;
                    (f ? tiles : btiles).push_back(T);
                }
    }
    const size_t nfree = tiles.size();
    tiles.insert(tiles.end(), btiles.begin(), btiles.end());
    if (tiles.empty()) return MX_OK;
    if (tiles.size() > 0x7fffffffULL) return MX_ERR_UNSUPPORTED;
    std::vector<FComp> comps(num_comp);
    for (int vc = 0; vc < num_comp; ++vc) {
        for (int d = 0; d < 3; ++d) {
            comps[vc].bclo[d] = bcs[bccomps[vc]].lo[d];
            comps[vc].bchi[d] = bcs[bccomps[vc]].hi[d];
        }
        comps[vc].comp = scomps[vc];
        comps[vc].flux = (levs[0].sflux && scomps[vc] == levs[0].flux_comp) ? levs[0].flux_kind : 0;
    }
    const FArgs A{dt,     c->p.rel_eps,      dt2,      dt3, cons ? dt3 : dt6, cons ? dt2 : dt4,
                  num_comp, is_vel};
    Table tab(c);
    size_t ob = tab.add(boxes);
    size_t ot = tab.add(tiles);
    size_t oc = tab.add(comps);
    int rc = tab.upload();
    if (rc) return rc;
    const FBox* db = tab.dev<FBox>(ob);
    const FTile* dtl = tab.dev<FTile>(ot);
    const FComp* dc = tab.dev<FComp>(oc);
    // a z side that needs more than the upwind cell puts every clear tile in the
    // kernel with the z rules (3 waves per SIMD): apart, the chunks at the side
    // and the others would each leave the chip half empty
    rc = zgen ? launch_one<TX, TY, 1>(c, db, dtl, nfree, dc, A, num_comp, cons)
              : launch_one<TX, TY, 0>(c, db, dtl, nfree, dc, A, num_comp, cons);
    if (rc) return rc;
    return launch_one<TX, TY, 2>(c, db, dtl + nfree, tiles.size() - nfree, dc, A, num_comp, cons);
}

// the tile shape of `fused_tile`, with the block size (columns rounded up to
// whole waves) and the register budget (waves per SIMD):
//   0: 32 x 8 (384 threads), 1: 16 x 16 (384), 2: 16 x 12 (256), 3: 16 x 8 (192),
//   4: 16 x 11 (256)
// -1 (the default) is 16 x 11: with ppm_type 1 its face values (19 x 13
// x-faces, 18 x 14 y-faces) are one item per thread of 256, and its LDS is the
// largest of which a CU holds four blocks
int fused_tile_of(const mx_adv_ctx* c) {
    if (c->fused_tile >= 0) return c->fused_tile;
    return 4;
}
int launch_tile(mx_adv_ctx* c, const std::vector<EdgeLevel>& levs, int tz, int is_vel,
                const mx_bcrec* bcs, const std::vector<int>& sc, const std::vector<int>& bc,
                int cons) {
    switch (fused_tile_of(c)) {
        case 1: return launch_fused<16, 16>(c, levs, tz, is_vel, bcs, sc, bc, cons);
        case 2: return launch_fused<16, 12>(c, levs, tz, is_vel, bcs, sc, bc, cons);
        case 3: return launch_fused<16, 8>(c, levs, tz, is_vel, bcs, sc, bc, cons);
        case 4: return launch_fused<16, 11>(c, levs, tz, is_vel, bcs, sc, bc, cons);
        default: return launch_fused<32, 8>(c, levs, tz, is_vel, bcs, sc, bc, cons);
    }
}

}  // namespace

int make_edge_scal_fused_list(mx_adv_ctx* c, const std::vector<EdgeLevel>& levs, int is_vel,
                              const mx_bcrec* bcs, const std::vector<int>& scomps,
                              const std::vector<int>& bccomps, int is_conservative) {
    if (levs.empty() || scomps.empty()) return MX_OK;
    if (scomps.size() != bccomps.size()) return MX_ERR_ARG;
    const int tz = c->fused_tz;
    if (c->fused_per_box) {
        // comparison mode: the same work as one launch per box
        std::vector<EdgeLevel> one(1);
        for (const EdgeLevel& L : levs)
            for (size_t b = 0; b < c->grids[L.lev].size(); ++b) {
                one[0] = L;
                one[0].box = (int)b;
                int rc = launch_tile(c, one, tz, is_vel, bcs, scomps, bccomps, is_conservative);
                if (rc) return rc;
            }
        return MX_OK;
    }
    return launch_tile(c, levs, tz, is_vel, bcs, scomps, bccomps, is_conservative);
}

int make_edge_scal_fused_levels(mx_adv_ctx* c, const std::vector<EdgeLevel>& levs, int is_vel,
                                const mx_bcrec* bcs, int start_scomp, int start_bccomp,
                                int num_comp, int is_conservative) {
    std::vector<int> sc(num_comp), bc(num_comp);
    for (int vc = 0; vc < num_comp; ++vc) {
        sc[vc] = start_scomp + vc;
        bc[vc] = start_bccomp + vc;
    }
    return make_edge_scal_fused_list(c, levs, is_vel, bcs, sc, bc, is_conservative);
}

int make_edge_scal_fused(mx_adv_ctx* c, int lev, const mx_multifab* state,
                         const mx_face_multifab* sedge, const mx_face_multifab* umac,
                         const mx_multifab* force, int is_vel, const mx_bcrec* bcs,
                         int start_scomp, int start_bccomp, int num_comp, int is_conservative) {
    std::vector<EdgeLevel> levs(1);
    levs[0] = {lev, state, sedge, umac, force};
    return make_edge_scal_fused_levels(c, levs, is_vel, bcs, start_scomp, start_bccomp, num_comp,
                                       is_conservative);
}

}  // namespace mxh
