// amx_free.hip -- method 2 (FREE): element contributions computed from node
// coordinates at every application; no element matrices are stored.
//
// The reference's FREE method calls a user function that builds K_e from the
// element's coordinates before each element GEMV (aMat::set_element_matrix_
// function, include/aMat.hpp:114-116, called from aMatFree.hpp:2449-2476;
// the examples pass ke_hex20_iso through computeElemMat,
// examples/src/example07a.cpp:54-70).  Here the element kinds of the examples
// are built in and applied without forming K_e, with the quadrature, shape
// functions and constitutive matrix of ke_hex8 / ke_tet10 / ke_hex20_iso
// (examples/src/ke_matrix.cpp), so f = s_e K_e u_e up to rounding:
//
//   J[k][d] = sum_a x_ak dN_ad,  inv = J^-1 (inv[d][k] = dxi_d/dx_k),
//   w = |J| w_q s_e,  dN_ad = dN_a/dxi_d at the quadrature point.
//   Laplace (one DoF per node):
//     h_d = sum_a u_a dN_ad,  p_d = w sum_k inv[d][k] (sum_d' h_d' inv[d'][k]),
//     f_a += sum_d dN_ad p_d.
//   Isotropic elasticity (DoF 3a+i, Voigt xx,yy,zz,xy,yz,xz, engineering shear):
//     H_id = sum_a u_ai dN_ad,  grad u = H inv,  sigma = w C eps(u),
//     P_di = sum_k inv[d][k] sigma_ik,  f_ai += sum_d dN_ad P_di.
//
// Outputs go to the element rows of the deterministic scatter (or atomics), so
// the maps, BC forms and gather are those of the stored-matrix kernels.  With
// DIAG the kernels write diag(s_e K_e) instead (Jacobi, penalty, trace).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "amx_device.hpp"
#include "amx_internal.hpp"
#include "amx_kernels.hpp"

namespace amx {

namespace {

constexpr uint32_t kFlag = 0x80000000u, kMask = 0x7fffffffu;
constexpr int kMaxDevices = 64;

// det J and inv[d][k] = cofactor(J)[k][d] / det (cofactors as in the host
// element routines, amx_fem.cpp jacobian; one division)
template <typename RT> __device__ __forceinline__ RT jac_inv_r(const RT J[3][3], RT inv[3][3])
{
    const RT c00 = J[1][1] * J[2][2] - J[2][1] * J[1][2];
    const RT c10 = J[2][1] * J[0][2] - J[0][1] * J[2][2];
    const RT c20 = J[0][1] * J[1][2] - J[1][1] * J[0][2];
    const RT det = J[0][0] * c00 + J[1][0] * c10 + J[2][0] * c20;
    const RT r = RT(1) / det;
    inv[0][0] = c00 * r;
    inv[0][1] = c10 * r;
    inv[0][2] = c20 * r;
    inv[1][0] = (J[1][2] * J[2][0] - J[2][2] * J[1][0]) * r;
    inv[1][1] = (J[2][2] * J[0][0] - J[0][2] * J[2][0]) * r;
    inv[1][2] = (J[0][2] * J[1][0] - J[1][2] * J[0][0]) * r;
    inv[2][0] = (J[2][1] * J[1][0] - J[1][1] * J[2][0]) * r;
    inv[2][1] = (J[0][1] * J[2][0] - J[2][1] * J[0][0]) * r;
    inv[2][2] = (J[1][1] * J[0][0] - J[0][1] * J[1][0]) * r;
    return det;
}

// ---- Laplace elements: one lane per element slot ------------------------
// xe: [NN*3][stride] (coordinate-major, slot fastest), qp: [nq][NN*3+1]
// (dN_ad at 3a+d, weight last; uniform across lanes -> scalar loads).
// RT: compute, coordinate and vector type (FP64; FP32 for the inner solves of
// the mixed-precision solvers, reading an FP32 copy of the coordinates).
// Factors and the table stay FP64 in memory and are rounded on load.
template <int NN, typename RT, bool MASKED, bool ATOMIC, bool DIAG>
__global__ __launch_bounds__(256) void free_laplace_kernel(const RT* __restrict__ xe, const double* __restrict__ scale,
                                                          const uint32_t* __restrict__ map, const RT* __restrict__ u,
                                                          RT* __restrict__ out, uint64_t ve_base, uint32_t rs,
                                                          uint32_t ss, uint32_t slot_begin, uint32_t n_slots,
                                                          uint32_t stride, const double* __restrict__ qp, uint32_t nq,
                                                          const uint32_t* __restrict__ skip)
{
    if (skip && *skip) return;
    const uint32_t sl = blockIdx.x * blockDim.x + threadIdx.x;
    if (sl >= n_slots) return;
    const uint64_t slot = (uint64_t)slot_begin + sl;
    RT x[NN * 3], ue[NN], f[NN];
    uint32_t m[NN];
#pragma unroll
    for (int i = 0; i < NN * 3; i++) x[i] = (RT)xe[(uint64_t)i * stride + slot];
#pragma unroll
    for (int a = 0; a < NN; a++) {
        m[a] = map[slot * NN + a];
        ue[a] = RT(0);
        if constexpr (!DIAG) {
            const RT v = u[m[a] & kMask];
            ue[a] = (MASKED && (m[a] & kFlag)) ? RT(0) : v;
        }
        f[a] = RT(0);
    }
    const RT sc = (RT)scale[slot];
    for (uint32_t q = 0; q < nq; q++) {
        const double* t = qp + (uint64_t)q * (NN * 3 + 1);
        RT J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, h[3] = {0, 0, 0};
#pragma unroll
        for (int a = 0; a < NN; a++)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const RT dn = (RT)t[3 * a + d];
#pragma unroll
                for (int k = 0; k < 3; k++) J[k][d] += x[3 * a + k] * dn;
                if constexpr (!DIAG) h[d] += ue[a] * dn;
            }
        RT inv[3][3];
        const RT det = jac_inv_r(J, inv);
        RT w = det * (RT)t[NN * 3] * sc;
        if constexpr (DIAG) {
            // a non-positive Jacobian at any point marks the element (NaN diagonal);
            // finalize rejects it, as the element routines do
            if (!(det > RT(0))) w = (RT)__builtin_nan("");
#pragma unroll
            for (int a = 0; a < NN; a++) {
                RT s = RT(0);
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    const RT g = (RT)t[3 * a] * inv[0][k] + (RT)t[3 * a + 1] * inv[1][k] + (RT)t[3 * a + 2] * inv[2][k];
                    s += g * g;
                }
                f[a] += s * w;
            }
        } else {
            RT gu[3], p[3];
#pragma unroll
            for (int k = 0; k < 3; k++) gu[k] = (h[0] * inv[0][k] + h[1] * inv[1][k] + h[2] * inv[2][k]) * w;
#pragma unroll
            for (int d = 0; d < 3; d++) p[d] = inv[d][0] * gu[0] + inv[d][1] * gu[1] + inv[d][2] * gu[2];
#pragma unroll
            for (int a = 0; a < NN; a++) f[a] += (RT)t[3 * a] * p[0] + (RT)t[3 * a + 1] * p[1] + (RT)t[3 * a + 2] * p[2];
        }
    }
#pragma unroll
    for (int a = 0; a < NN; a++) {
        if constexpr (ATOMIC) unsafeAtomicAdd(&out[m[a] & kMask], f[a]);
        else out[ve_base + (uint64_t)a * rs + slot * ss] = f[a];
    }
}

// ---- tet10 Laplacian: one lane per element slot --------------------------
// The derivatives of the quadratic interpolant are linear in xi:
//   df/dxi_d = A_d + sum_k xi_k D_dk,  D symmetric, with vertices v0 (origin),
//   v_d, and mid-edge nodes e_d (v0, v_d), e_dk (v_d, v_k):
//   A_d  = 4 (e_d - v0) - (v_d - v0),  D_dd = 4 ((v_d - e_d) + (v0 - e_d)),
//   D_dk = 4 ((e_dk - e_k) - (e_d - v0)).
// A point then costs 9 multiply-adds per field instead of 30, and the output
// needs the sums M_d = sum p_d, M_dd = sum xi_d p_d, S_dk = sum xi_k p_d + xi_d p_k
// only.  p = w inv inv^T h is formed from the cofactors, one division per point.
// Coordinates as in free_laplace_kernel; rule: [point][xi, weight].
//
// What bounds it: memory (41^3 cubes of 6, FP64: 153 MB at 5 TB/s; VGPRs allow 4
// waves per SIMD).  Against sums over the 10 nodes at every point, at ngt = 2:
// element kernel 38.5 -> 30.9 us, matvec FP64 56.5 -> 44.4 us (4 of it the gather),
// FP32 41 -> 31 us;
// relative L2 error 7.1e-16 -> 4.9e-16 (9^3 cubes), FP32 3.9e-7 -> 2.9e-7.
template <typename RT> struct Tet10 {
    RT A[3], D[3], S[3];  // S: D_12, D_23, D_31
    __device__ __forceinline__ explicit Tet10(const RT (&f)[10])
    {
        const RT v0 = f[0], e[3] = {f[4], f[6], f[7]}, c[3] = {f[5], f[9], f[8]};  // c: (1,2) (2,3) (3,1)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const RT r = e[d] - v0;
            A[d] = RT(4) * r - (f[1 + d] - v0);
            D[d] = RT(4) * ((f[1 + d] - e[d]) - r);
            S[d] = RT(4) * ((c[d] - e[(d + 1) % 3]) - r);
        }
    }
    __device__ __forceinline__ void at(const RT (&x)[3], RT (&g)[3]) const
    {
        g[0] = A[0] + x[0] * D[0] + x[1] * S[0] + x[2] * S[2];
        g[1] = A[1] + x[1] * D[1] + x[2] * S[1] + x[0] * S[0];
        g[2] = A[2] + x[2] * D[2] + x[0] * S[2] + x[1] * S[1];
    }
};

template <typename RT, bool MASKED, bool ATOMIC>
__global__ __launch_bounds__(256) void free_tet10_kernel(const RT* __restrict__ xe, const double* __restrict__ scale,
                                                        const uint32_t* __restrict__ map, const RT* __restrict__ u,
                                                        RT* __restrict__ out, uint64_t ve_base, uint32_t rs,
                                                        uint32_t ss, uint32_t slot_begin, uint32_t n_slots,
                                                        uint32_t stride, const double* __restrict__ rule, uint32_t nq,
                                                        const uint32_t* __restrict__ skip)
{
    if (skip && *skip) return;
    const uint32_t sl = blockIdx.x * blockDim.x + threadIdx.x;
    if (sl >= n_slots) return;
    const uint64_t slot = (uint64_t)slot_begin + sl;
    uint32_t m[10];
#pragma unroll
    for (int a = 0; a < 10; a++) m[a] = map[slot * 10 + a];
    RT v[3][10];
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int a = 0; a < 10; a++) v[k][a] = xe[(uint64_t)(3 * a + k) * stride + slot];
    const RT sc = (RT)scale[slot];
    RT w[10];
#pragma unroll
    for (int a = 0; a < 10; a++) {
        w[a] = u[m[a] & kMask];
        if (MASKED && (m[a] & kFlag)) w[a] = RT(0);
    }
    const Tet10<RT> X[3] = {Tet10<RT>(v[0]), Tet10<RT>(v[1]), Tet10<RT>(v[2])}, U(w);
    RT M[3] = {0, 0, 0}, Md[3] = {0, 0, 0}, S[3] = {0, 0, 0};
    for (uint32_t q = 0; q < nq; q++) {
        const RT x[3] = {(RT)rule[4 * q], (RT)rule[4 * q + 1], (RT)rule[4 * q + 2]};
        RT J[3][3], h[3], C[3][3], p[3];
#pragma unroll
        for (int k = 0; k < 3; k++) X[k].at(x, J[k]);
        U.at(x, h);
        // C[d][k]: cofactor of J[k][d]
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
            for (int k = 0; k < 3; k++)
                C[d][k] = J[(k + 1) % 3][(d + 1) % 3] * J[(k + 2) % 3][(d + 2) % 3] -
                          J[(k + 1) % 3][(d + 2) % 3] * J[(k + 2) % 3][(d + 1) % 3];
        const RT det = J[0][0] * C[0][0] + J[0][1] * C[1][0] + J[0][2] * C[2][0];
        const RT f = (RT)rule[4 * q + 3] * sc / det;
        RT g[3];
#pragma unroll
        for (int k = 0; k < 3; k++) g[k] = (h[0] * C[0][k] + h[1] * C[1][k] + h[2] * C[2][k]) * f;
#pragma unroll
        for (int d = 0; d < 3; d++) p[d] = C[d][0] * g[0] + C[d][1] * g[1] + C[d][2] * g[2];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            M[d] += p[d];
            Md[d] += x[d] * p[d];
            S[d] += x[d] * p[(d + 1) % 3] + x[(d + 1) % 3] * p[d];
        }
    }
    // transposed: r_d is the weight of e_d - v0, S_d of e_(d,d+1) - e_(d+1)
    RT o[10];
    constexpr int E[3] = {4, 6, 7}, C2[3] = {5, 9, 8};
    o[0] = RT(0);
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const RT r = RT(4) * (M[d] - (Md[d] + S[d]));
        o[1 + d] = RT(4) * Md[d] - M[d];
        o[0] += M[d] - r;
        o[E[d]] = r - RT(4) * (Md[d] + S[(d + 2) % 3]);
        o[C2[d]] = RT(4) * S[d];
    }
#pragma unroll
    for (int a = 0; a < 10; a++) {
        if constexpr (ATOMIC) unsafeAtomicAdd(&out[m[a] & kMask], o[a]);
        else out[ve_base + (uint64_t)a * rs + slot * ss] = o[a];
    }
}

// ---- hex20 isotropic elasticity -----------------------------------------
// The serendipity interpolant is a polynomial with few terms per direction, so
// its derivatives need not be summed node by node at every point.  With a the
// direction of the derivative and b, c the other two (cyclic), signs s_b, s_c
// of the four node lines along a (end values f-, f+, middle f0), and
//   D = f+ - f-,  S = f+ + f- - 2 f0  of a line, D00 = sum D, D10 = sum s_b D,
//   D01 = sum s_c D, D11 = sum s_b s_c D (S alike), E_b0, E_b1 the sum and
//   difference over s_c of f+ - f- of the b-edge middles, E_c0, E_c1 alike:
//   df/da = A(b, c) + a B(b, c)
//   A = al + be b^2 + ga c^2 + de bc + ep c + ze b^2 c + et b + th bc^2
//   B = s00 + s10 b + s01 c + s11 bc
//   al = (E_b0 + E_c0)/4 - D00/8, be = D00/8 - E_b0/4, ga = D00/8 - E_c0/4,
//   de = D11/8, ep = E_b1/4, ze = D01/8 - E_b1/4, et = E_c1/4,
//   th = D10/8 - E_c1/4, sxx = Sxx/4.
// At the ngt^3 points of a tensor rule that is about 5 operations per value
// instead of 20, and the transposed sums of the output likewise.
//
// A wave takes EW elements at a time, the values passed through its LDS region
// between the stages:
//   1  lane (element, coordinate, direction), 9 per element: 20 node values ->
//      12 coefficients -> the derivative at all points;
//   2  lane (element, point): J -> inverse and weight, kept in registers;
//   3  stage 1 on u in place of the coordinates;
//   4  lane (element, point): H -> stress -> P, 9 values in place of H;
//   5  lane (element, component, direction): the points' P -> 12 coefficients
//      -> 20 node contributions; then the sum over directions.
// EW = 7 fills 63 lanes in stages 1, 3 and 5 (and 189 = 2.95 waves of points at
// ngt = 3).  Coordinates and u in turn, so that a region holds the derivatives
// of three fields and not of six (both at once: 27 KB per wave at ngt = 3, 5
// waves per CU, 126 us on 48^3).  LDS rows have odd strides: lanes of stages
// 1, 3 and 5 hit distinct banks.
//
// What bounds it: the chain of stages with 8 (FP64, ngt = 3) to 16 waves per CU
// in flight (VGPRs; 4 waves per SIMD asked for in FP64 spill, 132 us).  Against
// node-by-node sums (60 per point and direction, 440 LDS values per lane),
// element kernel FP64 / matvec FP64 / matvec FP32:
//   48^3, ngt = 3   160 -> 68 us   182 -> 87 us   134 -> 59 us
//   48^3, ngt = 2    48 -> 47 us    71 -> 66 us    56 -> 47 us
//   24^3, ngt = 3    29 -> 15 us    32 -> 16 us    23 -> 13 us
//   24^3, ngt = 4    64 -> 36 us    67 -> 38 us    49 -> 23 us
// Relative L2 error of the FP64 product against 64 bits with the same rule (12^3,
// ngt = 2, 3, 4): 3.2e-15, 1.8e-15, 2.5e-15 -> 1.7e-16, 1.5e-16, 1.5e-16.  The
// digits of the rule's weights put the product 5.7e-16, 1.06e-14 and 2.5e-14 off that
// of an exact rule, whatever kernel forms it.
constexpr uint32_t kH20Node[3][5] = {  // byte j: 8 * node of entry j (per line f-, f+, f0; then the edge pairs)
    {0x18400800u, 0x28205010u, 0x70303860u, 0x68784858u, 0x90988880u},
    {0x20581800u, 0x10087838u, 0x68302848u, 0x90889880u, 0x70605040u},
    {0x08802000u, 0x38188828u, 0x90301098u, 0x70506040u, 0x68487858u}};

template <int NG> struct H20 {
    static constexpr int EW = NG == 4 ? 3 : 7;      // elements per wave
    static constexpr int PTS = NG * NG * NG;
    static constexpr int TS = PTS | 1;              // values of one (field, direction), odd
    static constexpr int GS = 9 * TS;               // derivatives of one element's three fields
    static constexpr int CS = 181, IS = 61;         // node contributions [direction][60], node values [field][20]
    static constexpr int WAVE = EW * (GS > CS ? GS : CS);
    static constexpr int P2 = (EW * PTS + 63) / 64; // passes over the points
};

// 12 coefficients of a (field, direction) from its 20 node values
template <typename RT> struct H20Coef {
    RT al, be, ga, de, ep, ze, et, th, s00, s10, s01, s11;

    static __device__ __forceinline__ void fly(const RT x[4], RT& q00, RT& q10, RT& q01, RT& q11)
    {
        const RT a0 = x[0] + x[1], a1 = x[1] - x[0], b0 = x[2] + x[3], b1 = x[3] - x[2];
        q00 = a0 + b0, q01 = b0 - a0, q10 = a1 + b1, q11 = b1 - a1;
    }
    __device__ __forceinline__ void from_nodes(const RT (&v)[20])
    {
        RT D[4], S[4], d00, d10, d01, d11;
#pragma unroll
        for (int l = 0; l < 4; l++) {
            D[l] = v[3 * l + 1] - v[3 * l];
            S[l] = (v[3 * l + 1] - v[3 * l + 2]) + (v[3 * l] - v[3 * l + 2]);
        }
        fly(D, d00, d10, d01, d11);
        fly(S, s00, s10, s01, s11);
        s00 *= RT(0.25), s10 *= RT(0.25), s01 *= RT(0.25), s11 *= RT(0.25);
        const RT e0 = v[13] - v[12], e1 = v[15] - v[14], g0 = v[17] - v[16], g1 = v[19] - v[18];
        const RT eb0 = RT(0.25) * (e0 + e1), eb1 = RT(0.25) * (e1 - e0);
        const RT ec0 = RT(0.25) * (g0 + g1), ec1 = RT(0.25) * (g1 - g0);
        be = RT(0.125) * d00 - eb0, ga = RT(0.125) * d00 - ec0, al = eb0 - ga;
        de = RT(0.125) * d11;
        ep = eb1, ze = RT(0.125) * d01 - eb1;
        et = ec1, th = RT(0.125) * d10 - ec1;
    }
    // derivative at the points (b, c, a), a fastest
    template <int NG> __device__ __forceinline__ void evaluate(const RT (&x)[NG], RT* g) const
    {
#pragma unroll
        for (int b = 0; b < NG; b++) {
            const RT xb = x[b];
            const RT a0 = al + xb * (et + xb * be), a1 = ep + xb * (de + xb * ze), a2 = ga + xb * th;
            const RT b0 = s00 + xb * s10, b1 = s01 + xb * s11;
#pragma unroll
            for (int c = 0; c < NG; c++) {
                const RT A = a0 + x[c] * (a1 + x[c] * a2), B = b0 + x[c] * b1;
#pragma unroll
                for (int a = 0; a < NG; a++) g[(b * NG + c) * NG + a] = A + x[a] * B;
            }
        }
    }
    // the transposed sums: coefficients of the points' values p
    template <int NG> __device__ __forceinline__ void collect(const RT (&x)[NG], const RT* p)
    {
        al = be = ga = de = ep = ze = et = th = s00 = s10 = s01 = s11 = RT(0);
#pragma unroll
        for (int b = 0; b < NG; b++) {
            RT r0 = RT(0), r1 = RT(0), r2 = RT(0), t0 = RT(0), t1 = RT(0);
#pragma unroll
            for (int c = 0; c < NG; c++) {
                RT q0 = RT(0), q1 = RT(0);
#pragma unroll
                for (int a = 0; a < NG; a++) {
                    const RT v = p[(b * NG + c) * NG + a];
                    q0 += v;
                    q1 += x[a] * v;
                }
                const RT cq = x[c] * q0;
                r0 += q0, r1 += cq, r2 += x[c] * cq;
                t0 += q1, t1 += x[c] * q1;
            }
            const RT xb = x[b], br0 = xb * r0, br1 = xb * r1;
            al += r0, et += br0, be += xb * br0;
            ep += r1, de += br1, ze += xb * br1;
            ga += r2, th += xb * r2;
            s00 += t0, s10 += xb * t0, s01 += t1, s11 += xb * t1;
        }
    }
    // node contributions (the order of from_nodes)
    __device__ __forceinline__ void to_nodes(RT (&v)[20]) const
    {
        const RT d00 = RT(0.125) * (be + ga - al), d11 = RT(0.125) * de, d01 = RT(0.125) * ze, d10 = RT(0.125) * th;
        const RT q00 = RT(0.25) * s00, q10 = RT(0.25) * s10, q01 = RT(0.25) * s01, q11 = RT(0.25) * s11;
#pragma unroll
        for (int l = 0; l < 4; l++) {
            const RT sb = (l & 1) ? RT(1) : RT(-1), sc = (l & 2) ? RT(1) : RT(-1);
            const RT D = (d00 + sb * d10) + sc * (d01 + sb * d11), S = (q00 + sb * q10) + sc * (q01 + sb * q11);
            v[3 * l] = S - D;
            v[3 * l + 1] = S + D;
            v[3 * l + 2] = RT(-2) * S;
        }
        const RT eb0 = RT(0.25) * (al - be), eb1 = RT(0.25) * (ep - ze);
        const RT ec0 = RT(0.25) * (al - ga), ec1 = RT(0.25) * (et - th);
        v[13] = eb0 - eb1, v[15] = eb0 + eb1, v[17] = ec0 - ec1, v[19] = ec0 + ec1;
        v[12] = -v[13], v[14] = -v[15], v[16] = -v[17], v[18] = -v[19];
    }
};

// P = inv . sigma at a point (w: |J|, weight and factor): H becomes P, [i][d]
template <typename RT>
__device__ __forceinline__ void h20_point(const RT (&inv)[3][3], RT w, RT (&H)[3][3], RT k1, RT k2, RT k3)
{
    RT g[3][3], sg[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int k = 0; k < 3; k++) g[i][k] = H[i][0] * inv[0][k] + H[i][1] * inv[1][k] + H[i][2] * inv[2][k];
    const RT exx = g[0][0] * w, eyy = g[1][1] * w, ezz = g[2][2] * w;
    sg[0][0] = k1 * exx + k2 * eyy + k2 * ezz;
    sg[1][1] = k2 * exx + k1 * eyy + k2 * ezz;
    sg[2][2] = k2 * exx + k2 * eyy + k1 * ezz;
    sg[0][1] = sg[1][0] = (k3 * w) * (g[0][1] + g[1][0]);
    sg[1][2] = sg[2][1] = (k3 * w) * (g[1][2] + g[2][1]);
    sg[0][2] = sg[2][0] = (k3 * w) * (g[0][2] + g[2][0]);
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int d = 0; d < 3; d++) H[i][d] = inv[d][0] * sg[i][0] + inv[d][1] * sg[i][1] + inv[d][2] * sg[i][2];
}

// the derivatives of an element group's three fields at the points, from the
// node values in W (overlaid)
template <int NG, typename RT>
__device__ __forceinline__ void h20_derivatives(RT* W, uint32_t lane, const RT (&x)[NG])
{
    using T = H20<NG>;
    const uint32_t t = min(lane, 9u * T::EW - 1u), e = t / 9u, r = t - 9u * e, f = r / 3u, d = r - 3u * f;
    const char* in = reinterpret_cast<const char*>(W + e * T::IS + f * 20u);
    RT v[20];
#pragma unroll
    for (int w = 0; w < 5; w++) {
        const uint32_t pk = d == 0 ? kH20Node[0][w] : d == 1 ? kH20Node[1][w] : kH20Node[2][w];
#pragma unroll
        for (int b = 0; b < 4; b++)
            v[4 * w + b] = *reinterpret_cast<const RT*>(in + ((pk >> (8 * b)) & 0xffu) * sizeof(RT) / 8u);
    }
    H20Coef<RT> co;
    co.from_nodes(v);
    lds_sync_wave();  // every lane's node values are read before the derivatives overlay them
    if (lane < 9u * T::EW) co.template evaluate<NG>(x, W + t * T::TS);
    lds_sync_wave();
}

// where point t of a group finds the derivatives of a field in direction d
template <int NG> struct H20At {
    uint32_t base, at[3];
    __device__ __forceinline__ explicit H20At(uint32_t t)
    {
        const uint32_t e = t / H20<NG>::PTS, q = t - e * H20<NG>::PTS;
        const uint32_t ix = q / (NG * NG), iy = q / NG % NG, iz = q % NG;
        base = e * H20<NG>::GS;
        at[0] = base + (iy * NG + iz) * NG + ix;
        at[1] = base + (iz * NG + ix) * NG + iy;
        at[2] = base + (ix * NG + iy) * NG + iz;
    }
};

// rule: the NG points, then the NG weights, of the one-dimensional rule
template <int NG, typename RT, bool MASKED, bool ATOMIC>
__global__ __launch_bounds__(64, sizeof(RT) == 4 && NG <= 3 ? 4 : 1) void free_hex20_kernel(const RT* __restrict__ xe, const double* __restrict__ scale,
                                                       const uint32_t* __restrict__ map, const RT* __restrict__ u,
                                                       RT* __restrict__ out, uint64_t ve_base, uint32_t rs,
                                                       uint32_t ss, uint32_t slot_begin, uint32_t n_slots,
                                                       const double* __restrict__ rule, double c1, double c2,
                                                       double c3, const uint32_t* __restrict__ skip)
{
    using T = H20<NG>;
    constexpr int EW = T::EW, PTS = T::PTS, TS = T::TS;
    __shared__ RT W[T::WAVE];
    if (skip && *skip) return;
    const RT k1 = (RT)c1, k2 = (RT)c2, k3 = (RT)c3;
    RT x[NG], wq[T::P2];
#pragma unroll
    for (int i = 0; i < NG; i++) x[i] = (RT)rule[i];
#pragma unroll
    for (int j = 0; j < T::P2; j++) {
        const uint32_t q = (threadIdx.x + 64u * j) % PTS;
        wq[j] = (RT)(rule[NG + q % NG] * rule[NG + q / NG % NG] * rule[NG + q / (NG * NG)]);
    }
    const uint32_t n_groups = (n_slots + EW - 1) / EW;

    // the next group's coordinates, map entries, node values and factors are
    // loaded into registers while the current group is computed: lane value j
    // is entry idx = lane + 64 j of the group's EW x 60 block
    constexpr int NL = (EW * 60 + 63) / 64;
    RT px[NL], pu[NL], ps[T::P2];
    uint32_t pm[NL];
    auto issue = [&](uint32_t grp) {
        const uint32_t lane = threadIdx.x, first = grp * EW, n_here = min((uint32_t)EW, n_slots - first);
        const uint64_t src0 = ((uint64_t)slot_begin + first) * 60u;
        // branch-free: entries past the group's elements repeat its last entry
        const uint32_t last = n_here * 60u - 1u;
#pragma unroll
        for (int j = 0; j < NL; j++) {
            const uint64_t src = src0 + min(lane + 64u * j, last);
            px[j] = xe[src];
            pm[j] = map[src];
        }
#pragma unroll
        for (int j = 0; j < T::P2; j++)
            ps[j] = (RT)scale[(uint64_t)slot_begin + first + min((lane + 64u * j) / PTS, n_here - 1u)];
    };
    auto gather = [&]() {
#pragma unroll
        for (int j = 0; j < NL; j++) {
            RT v = u[pm[j] & kMask];
            if (MASKED && (pm[j] & kFlag)) v = RT(0);
            pu[j] = v;
        }
    };
    // node values of the three fields, [element][field][node]
    auto put = [&](uint32_t lane, const RT (&v)[NL]) {
#pragma unroll
        for (int j = 0; j < NL; j++) {
            const uint32_t idx = lane + 64u * j;
            if (idx < EW * 60u) {
                const uint32_t e = idx / 60u, r = idx - e * 60u, a = r / 3u, k = r - 3u * a;
                W[e * T::IS + k * 20u + a] = v[j];
            }
        }
        lds_sync_wave();
    };

    uint32_t base = 0, grp = xcd_block(blockIdx.x, gridDim.x);  // consecutive groups on one XCD
    if (grp < n_groups) {
        issue(grp);
        gather();
    }
    for (; grp < n_groups; base += gridDim.x, grp = base + xcd_block(blockIdx.x, gridDim.x)) {
        const uint32_t first = grp * EW, n_here = min((uint32_t)EW, n_slots - first);
        const uint32_t next = base + gridDim.x + xcd_block(blockIdx.x, gridDim.x);
        // the lane's LDS addresses are formed anew for every group: kept over the
        // loop they take 80 registers, and with them a third of the waves
        uint32_t lane = threadIdx.x;
        asm volatile("" : "+v"(lane));
        put(lane, px);
        h20_derivatives<NG, RT>(W, lane, x);
        RT inv[T::P2][3][3], w[T::P2];
#pragma unroll
        for (int j = 0; j < T::P2; j++) {
            const H20At<NG> g(min(lane + 64u * j, (uint32_t)EW * PTS - 1u));
            RT J[3][3];
#pragma unroll
            for (int k = 0; k < 3; k++)
#pragma unroll
                for (int d = 0; d < 3; d++) J[k][d] = W[g.at[d] + (3 * k + d) * TS];
            w[j] = jac_inv_r(J, inv[j]) * wq[j] * ps[j];
        }
        lds_sync_wave();
        put(lane, pu);
        if (next < n_groups) issue(next);
        h20_derivatives<NG, RT>(W, lane, x);
#pragma unroll
        for (int j = 0; j < T::P2; j++) {
            const uint32_t t = lane + 64u * j;
            const H20At<NG> g(min(t, (uint32_t)EW * PTS - 1u));
            RT H[3][3];
#pragma unroll
            for (int i = 0; i < 3; i++)
#pragma unroll
                for (int d = 0; d < 3; d++) H[i][d] = W[g.at[d] + (3 * i + d) * TS];
            h20_point<RT>(inv[j], w[j], H, k1, k2, k3);
            if (t < (uint32_t)EW * PTS) {
#pragma unroll
                for (int i = 0; i < 3; i++)
#pragma unroll
                    for (int d = 0; d < 3; d++) W[g.at[d] + (3 * i + d) * TS] = H[i][d];
            }
        }
        lds_sync_wave();
        if (next < n_groups) gather();
        {
            const uint32_t t = min(lane, 9u * EW - 1u), e = t / 9u, r = t - 9u * e, i = r / 3u, d = r - 3u * i;
            H20Coef<RT> co;
            co.template collect<NG>(x, W + t * TS);
            lds_sync_wave();  // every lane's reads of P precede the contributions that overlay it
            RT v[20];
            co.to_nodes(v);
            char* o = reinterpret_cast<char*>(W + e * T::CS + d * 60u + i);
            if (lane < 9u * EW) {
#pragma unroll
                for (int k = 0; k < 5; k++) {
                    const uint32_t pk = d == 0 ? kH20Node[0][k] : d == 1 ? kH20Node[1][k] : kH20Node[2][k];
#pragma unroll
                    for (int b = 0; b < 4; b++)
                        *reinterpret_cast<RT*>(o + ((pk >> (8 * b)) & 0xffu) * 3u * sizeof(RT) / 8u) = v[4 * k + b];
                }
            }
        }
        lds_sync_wave();
#pragma unroll
        for (int j = 0; j < NL; j++) {
            const uint32_t idx = lane + 64u * j, e = idx / 60u, r = idx - e * 60u;
            if (idx < n_here * 60u) {
                const RT* c = W + e * T::CS + r;
                const RT f = c[0] + c[60] + c[120];
                const uint64_t slot = (uint64_t)slot_begin + first + e;
                if constexpr (ATOMIC) unsafeAtomicAdd(&out[map[slot * 60u + r] & kMask], f);
                else out[ve_base + (uint64_t)r * rs + slot * ss] = f;
            }
        }
        lds_sync_wave();  // the contributions are read before the next group's node values
    }
}

// diag(s_e K_e) of hex20 elements: lane l = e*QP + q of a wave holds element e at
// point q and leaves inv and w in LDS, then lane 3a+i sums the points.  qp:
// [nq][61] (dN_ad at 3a+d, weight).  Set-up only.
template <int QP>
__global__ __launch_bounds__(64) void free_hex20_diag_kernel(const double* __restrict__ xe,
                                                            const double* __restrict__ scale,
                                                            double* __restrict__ out, uint64_t ve_base, uint32_t rs,
                                                            uint32_t ss, uint32_t n_slots,
                                                            const double* __restrict__ qp, uint32_t nq, double c1,
                                                            double c3)
{
    constexpr int EW = 64 / QP;
    __shared__ double S[64][11];  // inv[d][k] at 3k + d, w at 9 (odd row stride)
    const uint32_t lane = threadIdx.x, slot0 = blockIdx.x * EW;
    {
        const uint32_t e = lane / QP, q = lane % QP, slot = min(slot0 + e, n_slots - 1u);
        const double* t = qp + (uint64_t)q * 61u;  // padded with rows of weight 0
        double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, inv[3][3];
        for (int a = 0; a < 20; a++)
            for (int k = 0; k < 3; k++)
                for (int d = 0; d < 3; d++) J[k][d] += xe[(uint64_t)slot * 60u + 3 * a + k] * t[3 * a + d];
        const double det = jac_inv_r(J, inv);
        double w = det * t[60] * scale[slot];
        // a non-positive Jacobian at a real point marks the element (NaN diagonal)
        if (q < nq && !(det > 0.0)) w = __builtin_nan("");
        for (int k = 0; k < 3; k++)
            for (int d = 0; d < 3; d++) S[lane][3 * k + d] = inv[d][k];
        S[lane][9] = w;
    }
    lds_sync_wave();
    if (lane >= 60u) return;
    const uint32_t a = lane / 3u, i = lane - 3u * a;
    for (uint32_t e = 0; e < EW && slot0 + e < n_slots; e++) {
        double f = 0.0;
        for (uint32_t q = 0; q < nq; q++) {
            const double* t = qp + (uint64_t)q * 61u + 3u * a;
            const double* s = S[e * QP + q];
            double g[3];
            for (int k = 0; k < 3; k++) g[k] = t[0] * s[3 * k] + t[1] * s[3 * k + 1] + t[2] * s[3 * k + 2];
            const double gi = i == 0 ? g[0] : (i == 1 ? g[1] : g[2]);
            const double gg = g[0] * g[0] + g[1] * g[1] + g[2] * g[2];
            f += (c1 * gi * gi + c3 * (gg - gi * gi)) * s[9];
        }
        out[ve_base + (uint64_t)lane * rs + (uint64_t)(slot0 + e) * ss] = f;
    }
}

// coordinates in the compute type: FP64, or the FP32 copy built at finalize
template <typename RT> const RT* coords(const FreeArgs& a)
{
    if constexpr (std::is_same<RT, float>::value) {
        AMX_REQUIRE(a.xe32 != nullptr, AMX_INVALID_STATE, "no FP32 coordinates");
        return a.xe32;
    } else {
        return a.xe;
    }
}

template <int NG, typename RT> void launch_hex20(bool masked, bool atomic, const FreeArgs& a, hipStream_t s)
{
    constexpr uint32_t EW = H20<NG>::EW;
    // resident waves per device: CUs x blocks per CU (the LDS bounds it); a
    // benign race between threads computes the same value
    static std::atomic<int> resident[kMaxDevices];
    int dev = 0;
    AMX_HIP(hipGetDevice(&dev));
    AMX_REQUIRE(dev >= 0 && dev < kMaxDevices, AMX_NOT_IMPLEMENTED, "device ordinal beyond the supported range");
    int res = resident[dev].load(std::memory_order_relaxed);
    if (res == 0) {
        int cus = 0, per_cu = 0;
        AMX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        AMX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, free_hex20_kernel<NG, RT, false, false>, 64, 0));
        res = std::max(1, cus * std::max(per_cu, 1));
        resident[dev].store(res, std::memory_order_relaxed);
    }
    const uint32_t need = (a.n_slots + EW - 1) / EW;
    const dim3 grid(std::min<uint32_t>(need, (uint32_t)res)), block(64);
    const RT* x = coords<RT>(a);
    const RT* u = static_cast<const RT*>(a.u);
    RT* out = static_cast<RT*>(a.out);
#define AMX_H20(M, A)                                                                                              \
    free_hex20_kernel<NG, RT, M, A><<<grid, block, 0, s>>>(x, a.scale, a.map, u, out, a.ve_base, a.ve_rs, a.ve_ss,  \
                                                           a.slot_begin, a.n_slots, a.rule, a.c1, a.c2, a.c3,       \
                                                           a.skip)
    if (masked) { if (atomic) AMX_H20(true, true); else AMX_H20(true, false); }
    else { if (atomic) AMX_H20(false, true); else AMX_H20(false, false); }
#undef AMX_H20
}

template <int QP> void launch_hex20_diag(const FreeArgs& a, hipStream_t s)
{
    AMX_REQUIRE(a.slot_begin == 0, AMX_INVALID_STATE, "the diagonal covers every slot");
    constexpr uint32_t EW = 64 / QP;
    free_hex20_diag_kernel<QP><<<(a.n_slots + EW - 1) / EW, 64, 0, s>>>(
        a.xe, a.scale, static_cast<double*>(a.out), a.ve_base, a.ve_rs, a.ve_ss, a.n_slots, a.qp, a.nq, a.c1, a.c3);
}

template <int NN, typename RT>
void launch_laplace(bool masked, bool atomic, bool diag, const FreeArgs& a, hipStream_t s)
{
    const dim3 grid((a.n_slots + 255) / 256), block(256);
    const RT* x = coords<RT>(a);
    const RT* u = static_cast<const RT*>(a.u);
    RT* out = static_cast<RT*>(a.out);
#define AMX_LAP(M, A, D)                                                                                           \
    free_laplace_kernel<NN, RT, M, A, D><<<grid, block, 0, s>>>(x, a.scale, a.map, u, out, a.ve_base, a.ve_rs,  \
                                                                a.ve_ss, a.slot_begin, a.n_slots, a.stride, a.qp,   \
                                                                a.nq, a.skip)
    if constexpr (std::is_same<RT, double>::value) {
        if (diag) {
            AMX_LAP(false, false, true);
            return;
        }
    }
    if constexpr (NN == 8) {  // (tet10: launch_tet10)
        if (masked) { if (atomic) AMX_LAP(true, true, false); else AMX_LAP(true, false, false); }
        else { if (atomic) AMX_LAP(false, true, false); else AMX_LAP(false, false, false); }
    }
#undef AMX_LAP
}

template <typename RT> void launch_tet10(bool masked, bool atomic, const FreeArgs& a, hipStream_t s)
{
    const dim3 grid((a.n_slots + 255) / 256), block(256);
    const RT* x = coords<RT>(a);
    const RT* u = static_cast<const RT*>(a.u);
    RT* out = static_cast<RT*>(a.out);
#define AMX_TET(M, A)                                                                                              \
    free_tet10_kernel<RT, M, A><<<grid, block, 0, s>>>(x, a.scale, a.map, u, out, a.ve_base, a.ve_rs, a.ve_ss,      \
                                                       a.slot_begin, a.n_slots, a.stride, a.rule, a.nq, a.skip)
    if (masked) { if (atomic) AMX_TET(true, true); else AMX_TET(true, false); }
    else { if (atomic) AMX_TET(false, true); else AMX_TET(false, false); }
#undef AMX_TET
}

template <typename RT>
void launch_free_t(int kind, bool masked, bool atomic, bool diag, const FreeArgs& a, hipStream_t s)
{
    switch (kind) {
    case AMX_ELEM_HEX8_LAPLACE: launch_laplace<8, RT>(masked, atomic, diag, a, s); break;
    case AMX_ELEM_TET10_LAPLACE:
        if (diag) launch_laplace<10, RT>(false, false, true, a, s);
        else launch_tet10<RT>(masked, atomic, a, s);
        break;
    case AMX_ELEM_HEX20_ELASTIC: {
        AMX_REQUIRE(a.nq <= 64, AMX_NOT_IMPLEMENTED, "hex20: at most 64 quadrature points");
        if (diag) {
            const uint32_t qp = free_padded_points(kind, a.nq);
            if (qp == 8) launch_hex20_diag<8>(a, s);
            else if (qp == 32) launch_hex20_diag<32>(a, s);
            else launch_hex20_diag<64>(a, s);
        } else if (a.nq == 1) {
            launch_hex20<1, RT>(masked, atomic, a, s);
        } else if (a.nq == 8) {
            launch_hex20<2, RT>(masked, atomic, a, s);
        } else if (a.nq == 27) {
            launch_hex20<3, RT>(masked, atomic, a, s);
        } else {
            launch_hex20<4, RT>(masked, atomic, a, s);
        }
        break;
    }
    default: fail(AMX_INVALID_ARGUMENT, "unknown element kind " + std::to_string(kind));
    }
}

}  // namespace

uint32_t free_padded_points(int kind, uint32_t nq)
{
    if (kind != AMX_ELEM_HEX20_ELASTIC) return nq;
    return nq <= 8 ? 8 : (nq <= 32 ? 32 : 64);
}

void launch_free(int kind, bool masked, bool atomic, bool diag, const FreeArgs& a, hipStream_t s)
{
    if (a.n_slots == 0) return;
    AMX_REQUIRE(!(diag && a.f32), AMX_INVALID_ARGUMENT, "the FREE diagonal is computed in FP64");
    if (a.f32) launch_free_t<float>(kind, masked, atomic, diag, a, s);
    else launch_free_t<double>(kind, masked, atomic, diag, a, s);
    AMX_HIP(hipGetLastError());
}

}  // namespace amx
