// mx_march.H -- what the z-marching kernels (mx_edge_fused.hip,
// mx_velpred_fused.hip) share: memory access and the one-sided trace.
#ifndef MX_MARCH_H
#define MX_MARCH_H

#include "mx_device.H"

namespace mxd {

typedef __attribute__((address_space(1))) const double gcd;
typedef __attribute__((address_space(1))) double gd;
typedef __attribute__((address_space(1))) const char gcc;
typedef __attribute__((address_space(1))) char gc;

// a double at a uniform base plus a 32-bit byte offset.  The empty asm keeps
// the offset's widening beside the access, where the compiler folds it into
// the addressing mode (one VGPR per address, no 64-bit add).
__device__ __forceinline__ double gload(gcc* base, unsigned off) {
    asm("" : "+v"(off));
    return *(gcd*)(base + off);
}
__device__ __forceinline__ void gstore(gc* base, unsigned off, double v) {
    asm("" : "+v"(off));
    *(gd*)(base + off) = v;
}

// trace of the upwind cell to its face (ppm_trace of mx_device.H for one
// side): A the edge value at the face, B the cell's other edge value.
// sp - h (sp - sm - c s6) and sm + h (sp - sm + c s6) are both
// A + h ((B - A) + c s6).
__device__ __forceinline__ double trace_face(double s0, double A, double B, double sig) {
    // 3 x and 6 x rounded once, by inline constants: 2 x + x, twice that
    const double s3 = fma(2.0, s0, s0), ab = A + B;
    const double s6 = 2.0 * s3 - fma(2.0, ab, ab);
    return A + 0.5 * sig * ((B - A) + (1.0 - 2.0 / 3.0 * sig) * s6);
}

// the CW84 limiter (cw_limit of mx_device.H, symmetric in its two edges)
// and the trace
__device__ __forceinline__ double cw_trace(double s0, double A, double B, double sig) {
    const double a = A - s0, b = s0 - B;
    const bool flat = a * b <= 0.0;
    const bool ca = dabs(a) >= 2.0 * dabs(b);
    const bool cb = dabs(b) >= 2.0 * dabs(a);
    const double s3 = fma(2.0, s0, s0);  // 3 s0
    const double A2 = s3 - 2.0 * B, B2 = s3 - 2.0 * A;
    const double A1 = ca ? A2 : A;
    const double B1 = (cb && !ca) ? B2 : B;
    return trace_face(s0, flat ? s0 : A1, flat ? s0 : B1, sig);
}

// The predictor's upwind state on the low face of a cell along a direction, s
// the cell's S slot and F its low face value's (FST, SST: one cell along the
// direction in the face and the S plane).
template <int PPM, int FST, int SST>
__device__ __forceinline__ double predict(const double* s, const double* F, bool left, bool traced,
                                          double sig) {
    const double* c = s + (left ? -SST : 0);
    const double s0 = c[0];
    double x;
    if (PPM == 1) {
        x = cw_trace(s0, F[0], F[left ? -FST : FST], sig);
    } else {
        const double* Fc = F + (left ? -FST : 0);
        double w9[9], sm, sp;
#pragma unroll
        for (int o = -4; o <= 4; ++o) w9[4 + o] = (o >= -2 && o <= 2) ? c[o * SST] : 0.0;
        cs_cell(w9, Fc[-FST], Fc[0], Fc[FST], Fc[2 * FST], 1.e-10, sm, sp);
        x = trace_face(s0, left ? sp : sm, left ? sm : sp, sig);
    }
    return traced ? x : s0;
}
// the same with the upwind cell's boundary stencil
template <int PPM, int D, int SST>
__device__ __forceinline__ double predict_special(const double* s, bool left, bool traced,
                                                  double sig, int pos, int dlo, int dhi, int bclo,
                                                  int bchi) {
    const double* c = s + (left ? -SST : 0);
    double w9[9], sm, sp;
#pragma unroll
    for (int o = -4; o <= 4; ++o) w9[4 + o] = (o >= -1 - PPM && o <= 1 + PPM) ? c[o * SST] : 0.0;
    ppm_edges<PPM, D>(w9, pos - (left ? 1 : 0), dlo, dhi, bclo, bchi, sm, sp);
    const double x = trace_face(c[0], left ? sp : sm, left ? sm : sp, sig);
    return traced ? x : c[0];
}

}  // namespace mxd

#endif
