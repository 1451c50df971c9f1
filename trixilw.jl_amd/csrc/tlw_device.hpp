// tlw_device.hpp -- gfx950 kernels of the TreeMesh Lax-Wendroff / MDRK step.
//
// Work decomposition: one thread per GLL node; a volume workgroup owns EB
// consecutive elements (with Z-ordered meshes, 16 consecutive elements form
// a 4x4 block of the tree).  Fluxes and flux time derivatives are exchanged
// through LDS for the derivative-matrix contractions; Taylor states, Ũ and F̃
// stay in registers.
//
// One step is three launches:
//   volume    uⁿ -> approximate LW procedure, volume term D̂F̃, then the
//             Rusanov flux of every interface whose two elements belong to
//             the workgroup (both face records are in LDS), the lifted
//             surface terms, the Jacobian and the update of every node.
//             Faces leaving the workgroup write a 10-double face record.
//   surface   the remaining faces: Rusanov flux from the two face records
//             (or the time-averaged Dirichlet state on a domain boundary),
//             lifted correction of those face nodes.
//   finalize  CFL reduction and compute_dt / set_dt! / set_t_and_iter! /
//             isfinished on the device state.
// The reference computes the same quantities in
//   lw_volume_kernel_3!/4!         src/solvers/dgsem_tree/dg_2d.jl:674-1267
//   prolong2interfaces!            src/solvers/dgsem_tree/dg_2d.jl:1269-1326
//   calc_interface_flux!           src/solvers/dgsem_tree/dg_2d.jl:1903-1946
//   calc_boundary_flux!            src/solvers/dgsem_tree/dg_2d.jl:1379-1454
//   Trixi calc_surface_integral!, apply_jacobian!, max_dt
//   update_soln!/set_dt!/set_t_and_iter!  src/solvers/lwfr.jl:70-103
//   mdrk_kernel_1!/2!              src/solvers/dgsem_tree/multi_derivative_2d.jl:263-555
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tlw_sincos.hpp"

namespace tlw {

constexpr int kBcSlipWall = 4;  // boundary kind of the reflecting wall (TLW_BV_SLIP_WALL)
constexpr int kBcTable = 5;     // caller-defined boundary data (TLW_BV_TABLE)
constexpr int kBcConvergenceTest = 6;  // the convergence test's state (TLW_BV_CONVERGENCE_TEST)
constexpr int kBcOutflow = 7;          // the normal flux of uⁿ (TLW_BV_OUTFLOW, curvilinear mesh)
constexpr int kBcSlipWallApprox = 8;   // Rusanov with uⁿ's reflection (TLW_BV_SLIP_WALL_APPROXIMATE, curvilinear)
constexpr int kTraceQ = 10;  // face record: jump state (4), normal flux (4), |v_n|, c
// shock-capturing face record: + fn_low (4), blending factor, padding
constexpr int kTraceQSC = 16;
template <bool SC> constexpr int kRQ = SC ? kTraceQSC : kTraceQ;
constexpr int kSurfBlock = 128;

// Row stride of an n x n operator kept in LDS: rounded up to a pair of doubles,
// so that a row is read in 16-byte loads.
constexpr int op_stride(int n) { return (n + 1) & ~1; }

// Volume workgroup geometry: EB elements, NT threads (a multiple of 64).
template <int N, int EB> struct VGeo {
    static constexpr int n = N + 1;
    static constexpr int NN = n * n;
    static constexpr int S = EB * NN;  // nodes of a workgroup: LDS stride of one exchanged pair of variables
    static constexpr int NT = ((EB * NN + 63) / 64) * 64;
    static constexpr int LDS = 3 * 8 * S;  // three exchange buffers
    // two exchange buffers, the second large enough for the face records
    static constexpr int LDS2 = 8 * S + (EB * 4 * n * kTraceQ > 8 * S ? EB * 4 * n * kTraceQ : 8 * S);
    static constexpr int MS = op_stride(n), M = n * MS;  // row stride and size of an operator in LDS
};
// Surface / reduction workgroup geometry: 128 threads.
template <int N> struct SGeo {
    static constexpr int n = N + 1;
    static constexpr int NN = n * n;
    static constexpr int EB = kSurfBlock / NN;
    static constexpr int S = EB * NN;
};

// Basis and boundary data, uploaded once per context.
struct DevConst {
    double D[8][8];      // derivative_matrix, row-major D[i][k]
    double Dhat[8][8];   // derivative_dhat
    double nodes[8], weights[8];
    double bnd_lo, bnd_hi;  // boundary_interpolation[1,1], [n,2]
    double gamma;
    double bc_par[24];
    int bc_kind;
    int flux_order;
    // shock capturing (IndicatorHennemannGassner on density_pressure)
    double Vinv[8][8];  // inverse normalised-Legendre Vandermonde, row-major
    double alpha_max, alpha_min;
    int alpha_smooth;
    double hg_threshold, hg_sharpness;  // 0.5·10^(-1.8 n^0.25), ln((1-1e-4)/1e-4)
    // positivity limiter thresholds for density and pressure
    double pos_threshold[2];
    // CompressibleNavierStokesDiffusion2D (conservative gradient variables):
    // dynamic viscosity, Prandtl number, κ = γ/((γ-1) Pr)
    double visc_mu, visc_Pr, visc_kappa;
    // no-slip adiabatic walls of the Navier-Stokes path on every boundary face:
    // wall velocity (v1, v2) per face 0..3 (x_neg, x_pos, y_neg, y_pos)
    int ns_walls;
    double wall_v[8];
    // per direction: 1 for Isothermal(wall_T) (NoSlip with a wall temperature), 0 Adiabatic(0)
    int wall_iso[4];
    double wall_T[4];
    // MUSCL-Hancock subcell geometry per node i (compute_subcells): spacings
    // to the neighbouring nodes, the centred-difference weights, the distances
    // from the node to its subcell faces, and hw[k] = xs[k+2] - xs[k+1], the
    // width the half-step divides by for subcell k
    int recon;  // TLW_RECON_*
    double mh_dx1[8], mh_dx2[8], mh_fa[8], mh_fb[8], mh_fc[8], mh_xl[8], mh_xr[8], mh_hw[8];
    int src_kind;  // SrcKind
    // L2 mortar operators of a TreeMesh with refined cells (LobattoLegendreMortarL2),
    // row-major [output node][input node]: [0] lower half, [1] upper half
    double mfwd[2][8][8];  // large face -> the half's GLL nodes
    double mrev[2][8][8];  // the half's fluxes -> large face (L2 projection)
};

// Device-resident integrator state (LWIntegrator fields t, dt, iter and the
// isfinished test), updated by the finalize kernel.
struct DevState {
    double t, dt, t_final, cfl;
    double invJ0;   // interface inverse Jacobian of compute_alp: the instance's first element
    double query;   // Trixi max_dt result of a query reduction
    int finished;
    int cur;        // state buffer holding uⁿ
    int bad_state;  // set when a non-admissible state was met
    long long iter;
    // Adaptive time stepping (src/solvers/adaptive.jl): the error estimates
    // epsilon[-1], epsilon[0], epsilon[1], tolerances, the instance's Trixi ndofs,
    // the retry count of the current step and the accumulated rejections
    double eps[3];
    double abstol, reltol, ndofs;
    int adaptive, nfail;
    long long nreject;
};

// Both structs as the kernels read them: constant for the whole launch (a kernel
// that changes the state writes through the plain pointer, and to fields it does
// not read), so that their fields come by scalar loads.  Through plain pointers
// each one after a store is a vector load the wave waits for, with every load
// in flight before it.
using DevC = const __attribute__((address_space(4))) DevConst*;
using DevS = const __attribute__((address_space(4))) DevState*;
__device__ __forceinline__ DevC dev_const(const DevConst* p) { return (DevC)(uintptr_t)p; }
__device__ __forceinline__ DevS dev_state(const DevState* p) { return (DevS)(uintptr_t)p; }
// an array of the same kind (workgroup tables, neighbours)
template <class T> using ConstArr = const __attribute__((address_space(4))) T*;
template <class T> __device__ __forceinline__ ConstArr<T> const_arr(const T* p) { return (ConstArr<T>)(uintptr_t)p; }

// a face whose two elements share a volume workgroup (KArgs::link)
constexpr int kResolved = -0x7fffffff;

enum BufSel { SEL_EXPLICIT = 0, SEL_CUR = 1, SEL_OTHER = 2 };
// RED_ADAPT: adaptive step (per-workgroup sums of the temporal errors and the
// admissibility test of the updated state instead of CFL maxima)
enum Reduce { RED_NONE = 0, RED_STEP = 1, RED_INIT = 2, RED_QUERY = 3, RED_ADAPT = 4 };
// VOL_LW_ADAPT: the LW kernel with the temporal-error estimate of adaptive steps
// (a separate instantiation, so the plain LW kernel carries none of its registers)
// VOL_LW_WALL, VOL_MDRK1_WALL, VOL_MDRK2_WALL: the Navier-Stokes LW and MDRK
// kernels that also keep the viscous time average of boundary face nodes
// (no-slip walls)
// VOL_*_SRC: the Euler LW and MDRK kernels with source terms (separate
// instantiations, VOL_LW_SRC + the plain kind)
enum VolKind {
    VOL_LW = 0, VOL_MDRK1 = 1, VOL_MDRK2 = 2, VOL_LW_ADAPT = 3, VOL_LW_WALL = 4,
    VOL_LW_SRC = 5, VOL_MDRK1_SRC = 6, VOL_MDRK2_SRC = 7, VOL_MDRK1_WALL = 8, VOL_MDRK2_WALL = 9,
    VOL_LW_ADAPT_WALL = 10
};
constexpr bool vol_is_src(int k) { return k >= VOL_LW_SRC && k <= VOL_MDRK2_SRC; }
constexpr bool vol_is_wall(int k) {
    return k == VOL_LW_WALL || k == VOL_MDRK1_WALL || k == VOL_MDRK2_WALL || k == VOL_LW_ADAPT_WALL;
}
// the plain kind of a source-term or wall instantiation
constexpr int vol_base(int k) {
    return vol_is_src(k)           ? k - VOL_LW_SRC
           : k == VOL_LW_WALL      ? (int)VOL_LW
           : k == VOL_MDRK1_WALL   ? (int)VOL_MDRK1
           : k == VOL_MDRK2_WALL   ? (int)VOL_MDRK2
           : k == VOL_LW_ADAPT_WALL ? (int)VOL_LW_ADAPT
                                   : k;
}
// source-term kinds of DevConst::src_kind
enum SrcKind { SRC_NONE = 0, SRC_CONVERGENCE_TEST = 1, SRC_NS_CONVERGENCE_TEST = 2 };

struct KArgs {
    int E;
    const double* u;      // uⁿ (explicit)
    const double* us;     // MDRK stage state
    double* out;          // volume: result; surface: corrected in place
    double* bufs[2];      // ping-pong state buffers for the device-resident loop
    int in_sel, out_sel;  // BufSel (the surface kernel reads the input at curvilinear boundary faces)
    double* trace;        // [E][4][n][kTraceQ], written for faces leaving a volume workgroup
    const int* nbr;       // [E][4]
    const double* inv_jac;
    const double* center;  // [E][2]
    const double* length;  // [E]
    const DevConst* c;
    DevState* st;
    double* auxU;      // optional full Ũ
    double* auxF;      // optional full F̃
    double* partial;   // the volume workgroups' temporal-error sums (adaptive steps)
    // Workgroup tables: {first element, elements, instance, 0} per workgroup of the
    // volume grid (vblk) and of the node-per-lane grids (sblk).  Workgroups never
    // straddle two instances of a batch, so each reads one instance's state.
    const int4* vblk;
    const int4* sblk;
    const int* link;   // [E][4] nbr for the faces that leave a volume workgroup, kResolved for the others
    const double* alpha_tmp;  // indicator values before smoothing [E]
    double* alpha_out;        // smoothed blending factors [E] (optional)
    // hyperbolic-parabolic: the CFL reduction takes the maximum of the viscous bound
    // J⁻² max(4μ/(3ρ), μκ/(ρ Pr)) too
    int parabolic;
    // curvilinear StructuredMesh (null on a TreeMesh): per node the contravariant
    // vectors (Ja11, Ja12, Ja21, Ja22) [E][n²][4] and inverse Jacobian [E][n²],
    // per face node the shared face normal (n1, n2, |n|, 0) [E][4][n][4]
    const double* Ja;
    const double* ijn;
    const double* fnorm;
    const double* fxy;  // boundary face-node coordinates [E][4][n][2] (curvilinear mesh with boundaries)
    const double* nxy;  // node coordinates [E][n*n][2] (curvilinear mesh with source terms)
    double* slots;      // per instance: kSlots CFL maxima, then kSlots viscous maxima (k_finalize resets them)
    // Navier-Stokes walls: per boundary face node the time-averaged viscous flux
    // of the face's orientation (momentum x, momentum y, energy), then the same
    // components at uⁿ [E][4][n][6]
    double* fvb;
    // curvilinear shock capturing: per node the subcell normals of its lower ξ
    // and η subcell faces [E][n²][4], and the calc_fn_low! normals of subcell
    // face n-1 per row (ξ) and column (η) [E][n][4]
    const double* snrm;
    const double* sqrk;
    // caller-defined Dirichlet data (bc_kind kBcTable): per element face the
    // boundary face index or -1 [E][4], and the state at every boundary face node
    // [face][n][levels][4]: levels 1 (steady) or n + 1 (GLL time levels, then t)
    const int* bidx;
    const double* btab;
    int btab_levels;
    double t_arg, dt_arg;
    int use_state_dt;  // 1: t, dt from DevState (device loop); 0: from t_arg/dt_arg
    int step_mode;     // 1: out = u + dt * rhs; 0: out = rhs
    int reduce;        // Reduce
    double bc_scale;   // scaling_factor of the Dirichlet time average
    // L2 mortars of a TreeMesh with refined cells: a face on mortar m in role r
    // (0 lower, 1 upper small element, 2 large element) has neighbour
    // -2 - (3 m + r).  Per mortar (orientation 1|2, large_side 1|2); per role and
    // face node the volume kernel's (jump state, normal flux, λ state) [M][3][n][12]
    // and the mortar kernel's fluxes [M][3][n][4]
    int n_mortars;
    const int2* mort;
    double* mrec;
    double* mflux;
    // P4estMesh (null otherwise): per element face its interface partner (element,
    // face, flipped node order, 1 if this element is the interface's primary);
    // interface faces carry neighbour code -3, so every face record goes to HBM
    const int4* plink;
};

// ---------------------------------------------------------------------------
// 1/x from the hardware reciprocal estimate r and one third-order step
// r <- r + r (e + e²), e = 1 - x r: the estimate's relative error is below
// 2^-24, so the step leaves e³ < 2^-72 and the result is rounded once, within
// an ulp for the normal densities it is applied to.  Three FMAs on top of the
// estimate (itself the time of four), where two Newton steps take four.
__device__ __forceinline__ double rcp_nr(double x) {
    const double r = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

// Euler flux, both directions (Trixi flux(u, 1|2, CompressibleEulerEquations2D)).
// The velocities use one reciprocal of ρ instead of two divisions.
__device__ __forceinline__ void euler_fluxes(const double* u, double gm1, double* f, double* g) {
    const double rho = u[0], m1 = u[1], m2 = u[2], E = u[3];
    const double ir = rcp_nr(rho);
    const double v1 = m1 * ir, v2 = m2 * ir;
    const double p = gm1 * (E - 0.5 * (m1 * v1 + m2 * v2));
    f[0] = m1;
    f[1] = m1 * v1 + p;
    f[2] = m1 * v2;
    f[3] = (E + p) * v1;
    g[0] = m2;
    g[1] = m2 * v1;
    g[2] = m2 * v2 + p;
    g[3] = (E + p) * v2;
}

// The quadratic parts of both Euler fluxes,
// q = (ρv1², ρv1v2, ρv2², (ρe+p)v1, (ρe+p)v2): the mass flux and the ρe inside p
// are linear in u, so a flux difference over Taylor states needs these five
// sums only (8 for two whole flux vectors), and its linear part is the time
// derivative of u itself, free of cancellation.  kh = -(γ-1)/2.
__device__ __forceinline__ void euler_q(const double* u, double gamma, double kh, double* q) {
    const double ir = rcp_nr(u[0]);
    const double v1 = u[1] * ir, v2 = u[2] * ir;
    q[0] = u[1] * v1;
    q[1] = u[1] * v2;
    q[2] = u[2] * v2;
    const double H = fma(gamma, u[3], kh * (q[0] + q[2]));  // ρe + p
    q[3] = H * v1;
    q[4] = H * v2;
}
// The flux pair of the sums q and the linear parts (l1, l2, lE) of ρv1, ρv2, ρe.
__device__ __forceinline__ void euler_join(const double* q, double l1, double l2, double lE, double gm1, double kh,
                                           double* f, double* g) {
    const double p = fma(kh, q[0] + q[2], gm1 * lE);
    f[0] = l1;
    f[1] = q[0] + p;
    f[2] = q[1];
    f[3] = q[3];
    g[0] = l2;
    g[1] = q[1];
    g[2] = q[2] + p;
    g[3] = q[4];
}

// The Taylor states of the LW procedure, u(t + s dt) for s = 1, -1, 2, -2
// (rows): level m adds kTaylor[s][m-1] = s^m/m! times the m-th derivative.
__device__ constexpr double kTaylor[4][4] = {{1.0, 0.5, 1.0 / 6.0, 1.0 / 24.0},
                                             {-1.0, 0.5, -1.0 / 6.0, 1.0 / 24.0},
                                             {2.0, 2.0, 4.0 / 3.0, 2.0 / 3.0},
                                             {-2.0, 2.0, -4.0 / 3.0, 2.0 / 3.0}};
// The k-th time difference of the flux: Σ_s c[s] f(state s) + c[4] f(uⁿ), times
// scale (calc_time_differences of kernels 3 and 4: five points for f_t, f_tt at
// N = 4 and f_ttt, three for f_tt at N = 3; the 0.5 of f_tttt is the
// reference's, dg_2d.jl:1203-1206).  The coefficients are integers or powers of
// two, so that equal states cancel exactly (a rounded 2/3 leaves an ulp of the
// flux, which the next levels' derivatives amplify); a division by 12 comes last.
// linear: what the stencil gives of a linear function, times its derivative.
struct TimeDiff {
    double c[5], scale, linear;
};
template <int N> __device__ constexpr TimeDiff time_diff(int k) {
    if (k == 1) return {{8.0, -8.0, -1.0, 1.0, 0.0}, 1.0 / 12.0, 1.0};
    if (k == 2 && N == 4) return {{16.0, 16.0, -1.0, -1.0, -30.0}, 1.0 / 12.0, 1.0};
    if (k == 2) return {{1.0, 1.0, 0.0, 0.0, -2.0}, 1.0, 1.0};
    if (k == 3) return {{-1.0, 1.0, 0.5, -0.5, 0.0}, 1.0, 1.0};
    return {{-2.0, -2.0, 0.5, 0.5, 3.0}, 1.0, 0.5};
}
// weight of the k-th derivative in Ũ and F̃: 1/(k+1)!
__device__ constexpr double lw_weight(int k) {
    return k == 0 ? 1.0 : k == 1 ? 0.5 : k == 2 ? 1.0 / 6.0 : k == 3 ? 1.0 / 24.0 : 1.0 / 120.0;
}

// ---------------------------------------------------------------------------
// Source terms of the LW procedure (dg_2d.jl:89-176).  The device's source is
// Trixi's source_terms_convergence_test for CompressibleEulerEquations2D, the
// residual ∂t u + ∇·f(u) of the manufactured state ρ = ρv1 = ρv2 = φ, ρe = φ²,
// φ = 2 + 0.1 sin(π(x + y - t)): with φ' = 0.1π cos(π(x + y - t)) and
// τ = (2φ - 1)(γ - 1), s = (φ', φ'(1 + τ), φ'(1 + τ), 2φ'(φ + τ)).  It depends
// on (x, t) only, so every time difference of s the reference forms at its
// stencil states is a combination of s(x, t + k dt), k = -2..2, and the order
// in which the reference passes those states does not change it.
struct SrcPt {
    double x, y, t, gamma;
};
__device__ __forceinline__ void src_eval(const SrcPt& p, double toff, double* s) {
    const double w = 3.141592653589793;
    double si, co;
    sincos_cw(w * (p.x + p.y - (p.t + toff)), &si, &co);
    const double rho = 2.0 + 0.1 * si;
    const double rho_x = w * 0.1 * co;
    const double tmp = (2.0 * rho - 1.0) * (p.gamma - 1.0);
    s[0] = rho_x;
    s[1] = rho_x * (1.0 + tmp);
    s[2] = s[1];
    s[3] = 2.0 * rho_x * (rho + tmp);
}
// dt-scaled time differences about p.t + t0 (calc_source_t_N34,
// calc_source_tt_N23, calc_source_ttt_N34, calc_source_tttt_N4)
__device__ __forceinline__ void src_t5(const SrcPt& p, double t0, double dt, double* o) {
    double a[4], b[4];
    src_eval(p, t0 + 2.0 * dt, a);
    src_eval(p, t0 + dt, b);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = 8.0 * b[v] - a[v];
    src_eval(p, t0 - dt, a);
    src_eval(p, t0 - 2.0 * dt, b);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = (1.0 / 12.0) * (o[v] - 8.0 * a[v] + b[v]);
}
__device__ __forceinline__ void src_tt3(const SrcPt& p, double dt, double* o) {
    double a[4], b[4];
    src_eval(p, dt, a);
    src_eval(p, 0.0, b);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = a[v] - 2.0 * b[v];
    src_eval(p, -dt, a);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] += a[v];
}
__device__ __forceinline__ void src_ttt5(const SrcPt& p, double dt, double* o) {
    double a[4], b[4];
    src_eval(p, 2.0 * dt, a);
    src_eval(p, dt, b);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = a[v] - 2.0 * b[v];
    src_eval(p, -dt, a);
    src_eval(p, -2.0 * dt, b);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = 0.5 * (o[v] + 2.0 * a[v] - b[v]);
}
__device__ __forceinline__ void src_tttt5(const SrcPt& p, double dt, double* o) {
    double a[4], b[4];
    src_eval(p, 2.0 * dt, a);
    src_eval(p, dt, b);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = a[v] - 4.0 * b[v];
    src_eval(p, 0.0, a);
    src_eval(p, -dt, b);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = o[v] + 6.0 * a[v] - 4.0 * b[v];
    src_eval(p, -2.0 * dt, a);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] += a[v];
}

// s_tt of calc_source_tt_N4 (five points), which the StructuredMesh kernel 4
// takes: (-s(t+2dt) + 16 s(t+dt) - 30 s(t) + 16 s(t-dt) - s(t-2dt))/12
__device__ __forceinline__ void src_tt5(const SrcPt& p, double dt, double* o) {
    double a[4], b[4];
    src_eval(p, 2.0 * dt, a);
    src_eval(p, dt, b);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = 16.0 * b[v] - a[v];
    src_eval(p, 0.0, a);
    src_eval(p, -dt, b);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = o[v] - 30.0 * a[v] + 16.0 * b[v];
    src_eval(p, -2.0 * dt, a);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = (1.0 / 12.0) * (o[v] - a[v]);
}
// Source level k of the StructuredMesh LW kernels (structured/dg_2d.jl:1440-1666,
// 1750-2058): s^(k) about t into sk (s; s_t of N34; s_tt five-point at polydeg
// 4, three-point at 3; s_ttt of N34; s_tttt of N4), and S += weight·s^(k)
// (S = s at k = 0)
__device__ __forceinline__ void src_level_c(const SrcPt& p, double dt, int k, bool five_tt, double* sk, double* S,
                                            double weight) {
    if (k == 0) src_eval(p, 0.0, sk);
    else if (k == 1) src_t5(p, 0.0, dt, sk);
    else if (k == 2 && five_tt) src_tt5(p, dt, sk);
    else if (k == 2) src_tt3(p, dt, sk);
    else if (k == 3) src_ttt5(p, dt, sk);
    else src_tttt5(p, dt, sk);
#pragma unroll
    for (int v = 0; v < 4; ++v) S[v] = k == 0 ? weight * sk[v] : fma(weight, sk[v], S[v]);
}

// The Navier-Stokes convergence source (the source_terms of
// examples/tree_2d_dgsem/elixir_navierstokes_convergence.jl:49-205): the
// residual ∂t u + ∇·f_a - ∇·f_v of ρ = 2 + ½ sin πx cos πy cos πt,
// v1 = v2 = sin πx g(y) cos πt with g = log(y + 2)(1 - e^{-(y-1)/2}), p = ρ²,
// under Trixi's viscous fluxes (Stokes' hypothesis, heat flux μκ∇T with
// κ = γ/((γ-1)Pr), T = p/ρ), by the product rule from the closed-form
// derivatives.  The node's spatial factors are formed once (NsSrcPt), each
// time level then needs sin and cos of πt only.  It does not depend on u.
struct NsSrcPt {
    double sx, cx, sy, cy, g, g1, g2, t, gamma, mu, prandtl;
};
__device__ __forceinline__ NsSrcPt ns_src_point(double x, double y, double t, DevC c) {
    constexpr double pi = 3.141592653589793, A = 0.5;
    NsSrcPt p;
    sincos_cw(pi * x, &p.sx, &p.cx);
    sincos_cw(pi * y, &p.sy, &p.cy);
    const double e = exp(-A * (y - 1.0)), L = log(y + 2.0), q = 1.0 / (y + 2.0);
    p.g = L * (1.0 - e);
    p.g1 = (1.0 - e) * q + A * L * e;
    p.g2 = -(1.0 - e) * q * q + 2.0 * A * e * q - A * A * L * e;
    p.t = t;
    p.gamma = c->gamma;
    p.mu = c->visc_mu;
    p.prandtl = c->visc_Pr;
    return p;
}
__device__ __forceinline__ void ns_src_eval(const NsSrcPt& p, double toff, double* s) {
    constexpr double pi = 3.141592653589793, A = 0.5;
    double st, ct;
    sincos_cw(pi * (p.t + toff), &st, &ct);
    const double sx = p.sx, cx = p.cx, sy = p.sy, cy = p.cy;
    const double r = 2.0 + A * sx * cy * ct;
    const double r_t = -pi * A * sx * cy * st;
    const double r_x = pi * A * cx * cy * ct;
    const double r_y = -pi * A * sx * sy * ct;
    const double r_xx = -pi * pi * A * sx * cy * ct, r_yy = r_xx;
    const double v = sx * p.g * ct, v_t = -pi * sx * p.g * st;
    const double v_x = pi * cx * p.g * ct, v_y = sx * p.g1 * ct;
    const double v_xx = -pi * pi * sx * p.g * ct, v_xy = pi * cx * p.g1 * ct, v_yy = sx * p.g2 * ct;
    const double pr = r * r, p_x = 2.0 * r * r_x, p_y = 2.0 * r * r_y;
    const double p_xx = 2.0 * (r_x * r_x + r * r_xx), p_yy = 2.0 * (r_y * r_y + r * r_yy);
    const double ig = 1.0 / (p.gamma - 1.0), k2 = v * v + v * v;
    const double E = pr * ig + 0.5 * r * k2;
    const double E_t = 2.0 * r * r_t * ig + 0.5 * r_t * k2 + r * (v * v_t + v * v_t);
    const double E_x = p_x * ig + 0.5 * r_x * k2 + r * (v * v_x + v * v_x);
    const double E_y = p_y * ig + 0.5 * r_y * k2 + r * (v * v_y + v * v_y);
    const double t11 = (4.0 / 3.0) * v_x - (2.0 / 3.0) * v_y, t12 = v_y + v_x;
    const double t22 = (4.0 / 3.0) * v_y - (2.0 / 3.0) * v_x;
    const double t11_x = (4.0 / 3.0) * v_xx - (2.0 / 3.0) * v_xy, t12_x = v_xy + v_xx;
    const double t12_y = v_yy + v_xy, t22_y = (4.0 / 3.0) * v_yy - (2.0 / 3.0) * v_xy;
    const double ir3 = 1.0 / (r * r * r);
    const double T_xx = (p_xx * r * r - 2.0 * p_x * r * r_x + 2.0 * pr * r_x * r_x - pr * r * r_xx) * ir3;
    const double T_yy = (p_yy * r * r - 2.0 * p_y * r * r_y + 2.0 * pr * r_y * r_y - pr * r * r_yy) * ir3;
    const double kappa = p.gamma * ig / p.prandtl, mu = p.mu;
    s[0] = r_t + r_x * v + r * v_x + r_y * v + r * v_y;
    s[1] = r_t * v + r * v_t + r_x * v * v + 2.0 * r * v * v_x + p_x + r_y * v * v + r * v_y * v + r * v * v_y -
           mu * (t11_x + t12_y);
    s[2] = r_t * v + r * v_t + r_x * v * v + r * v_x * v + r * v * v_x + r_y * v * v + 2.0 * r * v * v_y + p_y -
           mu * (t12_x + t22_y);
    const double work_x = v_x * t11 + v * t11_x + v_x * t12 + v * t12_x;
    const double work_y = v_y * t12 + v * t12_y + v_y * t22 + v * t22_y;
    s[3] = E_t + (E_x + p_x) * v + (E + pr) * v_x + (E_y + p_y) * v + (E + pr) * v_y -
           mu * (work_x + work_y + kappa * (T_xx + T_yy));
}
// s_t of calc_source_t_N34 about t: (-s(t+2dt) + 8 s(t+dt) - 8 s(t-dt) + s(t-2dt))/12
__device__ __forceinline__ void ns_src_t5(const NsSrcPt& p, double dt, double* o) {
    double a[4];
    ns_src_eval(p, 2.0 * dt, a);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = -a[v];
    ns_src_eval(p, dt, a);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = fma(8.0, a[v], o[v]);
    ns_src_eval(p, -dt, a);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = fma(-8.0, a[v], o[v]);
    ns_src_eval(p, -2.0 * dt, a);
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = (1.0 / 12.0) * (o[v] + a[v]);
}

// The time difference of order k of the source at the node about t, as the
// reference's LW kernels form it (calc_source / _t_N34 / _tt_N4 (five_tt) or
// _tt_N23 / _ttt_N34 / _tttt_N4, dg_2d.jl:89-176).
__device__ __forceinline__ void ns_src_diff(const NsSrcPt& p, double dt, int order, bool five_tt, double* o) {
    double a[4], b[4], z[4], c[4], d[4];
    ns_src_eval(p, 0.0, z);
    if (order == 0) {
#pragma unroll
        for (int v = 0; v < 4; ++v) o[v] = z[v];
        return;
    }
    ns_src_eval(p, 2.0 * dt, a);
    ns_src_eval(p, dt, b);
    ns_src_eval(p, -dt, c);
    ns_src_eval(p, -2.0 * dt, d);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        if (order == 1) o[v] = (1.0 / 12.0) * (-a[v] + 8.0 * b[v] - 8.0 * c[v] + d[v]);
        else if (order == 2 && five_tt) o[v] = (1.0 / 12.0) * (-a[v] + 16.0 * b[v] - 30.0 * z[v] + 16.0 * c[v] - d[v]);
        else if (order == 2) o[v] = b[v] - 2.0 * z[v] + c[v];
        else if (order == 3) o[v] = 0.5 * (a[v] - 2.0 * b[v] + 2.0 * c[v] - d[v]);
        else o[v] = a[v] - 4.0 * b[v] + 6.0 * z[v] - 4.0 * c[v] + d[v];
    }
}

__device__ __forceinline__ void euler_flux_dir(const double* u, double gm1, int orientation, double* f) {
    double ff[4], gg[4];
    euler_fluxes(u, gm1, ff, gg);
    for (int v = 0; v < 4; ++v) f[v] = orientation == 1 ? ff[v] : gg[v];
}

__device__ __forceinline__ double dmax(double x, double y) { return (y > x) ? y : x; }

// The CFL maxima of the node-per-lane workgroups meet in kSlots slots per
// instance by an integer atomic maximum: non-negative doubles order like their
// bit patterns, and a maximum does not depend on the order, so the reduction is
// deterministic.  NaN and 0 leave a slot as dmax would.
constexpr int kSlots = 256;
__device__ __forceinline__ void slot_max(double* slots, int inst, int which, double v) {
    if (v > 0.0)
        atomicMax(reinterpret_cast<unsigned long long*>(slots + ((size_t)inst * 2 + which) * kSlots +
                                                        (blockIdx.x & (kSlots - 1))),
                  (unsigned long long)__double_as_longlong(v));
}

// v of the lane that the DPP control picks (a lane of the same row of 16).
template <int CTRL> __device__ __forceinline__ double dpp_f64(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double readlane_f64(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// maximum over the 8 lanes of a group, over a row's two groups, over the rows
// (non-negative operands; a NaN loses against any of them, as in dmax(m, NaN))
__device__ __forceinline__ double max_group8(double v) {
    v = fmax(v, dpp_f64<0xB1>(v));   // quad_perm 1 0 3 2
    v = fmax(v, dpp_f64<0x4E>(v));   // quad_perm 2 3 0 1
    return fmax(v, dpp_f64<0x141>(v));  // row_half_mirror
}
__device__ __forceinline__ double max_groups(double v) {
    v = fmax(v, dpp_f64<0x128>(v));  // row_ror 8
    return fmax(fmax(readlane_f64(v, 0), readlane_f64(v, 16)), fmax(readlane_f64(v, 32), readlane_f64(v, 48)));
}

// The CFL maxima of a node-per-lane workgroup of nel elements into its slots:
// J⁻¹ (max λ1 + max λ2) over its elements (with `scaled`, a curvilinear mesh,
// the speeds carry the node's |J⁻¹| and invJ is not used), and with par the
// maximum of the viscous bounds lv.  Every lane of the workgroup calls it, with
// the node's values where act.  One barrier, then the first wave takes eight
// lanes per element.  One lane per element walking its 25 nodes was most of the
// instructions of the kernels that end with it: at 1024², N=4, the surface
// kernel went from 548 to 411 us (2.7 GB, now at HBM speed), the initial dt's
// k_max_speed from 415 to 169 us (0.84 GB).
template <int N>
__device__ __forceinline__ void cfl_maxima(double* slots, int inst, int tid, int nel, int sidx, bool act, bool first,
                                           double l1, double l2, double lv, double invJ, bool scaled, bool par) {
    using G_ = SGeo<N>;
    constexpr int NN = G_::NN, EB = G_::EB;
    static_assert(EB <= 8, "eight lanes per element in one wave");
    __shared__ double2 s_l[G_::S];
    __shared__ double s_v[G_::S], s_j[EB];
    if (act) {
        s_l[sidx] = make_double2(l1, l2);
        if (par) s_v[sidx] = lv;
        if (first) s_j[sidx / NN] = invJ;
    }
    __syncthreads();
    if (tid >= 64) return;
    const int el = tid >> 3, q = tid & 7;
    double m1 = 0.0, m2 = 0.0, mv = 0.0;
    if (el < nel) {
#pragma unroll
        for (int k = 0; k < NN; k += 8) {
            if (k + q >= NN) continue;
            const double2 x = s_l[el * NN + k + q];
            m1 = fmax(m1, x.x);
            m2 = fmax(m2, x.y);
            if (par) mv = fmax(mv, s_v[el * NN + k + q]);
        }
    }
    m1 = max_group8(m1);
    m2 = max_group8(m2);
    double bm = 0.0;
    if (el < nel) bm = scaled ? m1 + m2 : s_j[el] * (m1 + m2);
    bm = max_groups(bm);
    if (par) mv = max_groups(max_group8(mv));
    if (tid == 0) {
        slot_max(slots, inst, 0, bm);
        if (par) slot_max(slots, inst, 1, mv);
    }
}

// Square root of a positive normal argument: the hardware reciprocal
// square-root estimate refined by two steps of Goldschmidt's iteration and a
// final Newton correction (P. Markstein, "IA-64 and Elementary Functions",
// 2000, ch. 8), within an ulp or two of the rounded root.  Zero, negative and
// NaN arguments give NaN; callers apply it to sound speeds, whose states are
// checked for ρ > 0 and p > 0.
__device__ __forceinline__ double sqrt_gs(double x) {
    const double r = __builtin_amdgcn_rsq(x);
    double g = x * r, h = 0.5 * r;
    double e = fma(-g, h, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    e = fma(-g, h, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    const double d = fma(-g, g, x);
    return fma(d, h, g);
}

// |v_n| and the sound speed: the per-side ingredients of Trixi's
// max_abs_speed_naive (λ = max(|v_n,L|,|v_n,R|) + max(c_L, c_R)).
__device__ __forceinline__ void speed_parts(const double* s, double gamma, int orientation, double& a, double& c) {
    const double ir = rcp_nr(s[0]);
    const double v1 = s[1] * ir, v2 = s[2] * ir;
    const double p = (gamma - 1.0) * (s[3] - 0.5 * (s[1] * v1 + s[2] * v2));
    a = fabs(orientation == 1 ? v1 : v2);
    c = sqrt_gs(gamma * p * ir);
}

// |v1|, |v2| and the sound speed of one state: the λ ingredients of both
// orientations with one reciprocal of ρ and one square root.
__device__ __forceinline__ void speed_parts2(const double* s, double gamma, double& a1, double& a2, double& c) {
    const double ir = rcp_nr(s[0]);
    const double v1 = s[1] * ir, v2 = s[2] * ir;
    const double p = (gamma - 1.0) * (s[3] - 0.5 * (s[1] * v1 + s[2] * v2));
    a1 = fabs(v1);
    a2 = fabs(v2);
    c = sqrt_gs(gamma * p * ir);
}



// Julia's x ≈ y for Float64 (atol = 0, rtol = sqrt(eps)): equal, or both
// finite and |x - y| <= rtol max(|x|, |y|).  isfinished (lwfr.jl:146-148).
__device__ __forceinline__ int julia_isapprox(double x, double y) {
    if (x == y) return 1;
    if (!isfinite(x) || !isfinite(y)) return 0;
    return fabs(x - y) <= 1.4901161193847656e-08 * dmax(fabs(x), fabs(y));
}

// Boundary value functions of the time-averaged Dirichlet condition.
__device__ inline void boundary_value(DevC c, double x, double y, double t, double* u) {
    const auto* par = c->bc_par;
    double rho, v1, v2, p, gamma;
    if (c->bc_kind == kBcConvergenceTest) {
        // Trixi's initial_condition_convergence_test: ρ = ρv1 = ρv2 = φ, ρe = φ²
        double si, co;
        sincos_cw(3.141592653589793 * (x + y - t), &si, &co);
        const double phi = 2.0 + 0.1 * si;
        u[0] = u[1] = u[2] = phi;
        u[3] = phi * phi;
        return;
    }
    if (c->bc_kind == 1) {  // isentropic vortex
        const double eps = par[0], mach = par[1], Lx = par[4], Ly = par[5];
        gamma = par[6];
        const double vinf = mach * sqrt(gamma) / sqrt(2.0);
        double dx = x - (par[2] + vinf * t), dy = y - (par[3] + vinf * t);
        dx -= Lx * floor(dx / Lx + 0.5);
        dy -= Ly * floor(dy / Ly + 0.5);
        const double r2 = dx * dx + dy * dy;
        const double pi = 3.141592653589793;
        const double du = eps / (2 * pi) * exp(0.5 * (1 - r2));
        const double T = 1 - (gamma - 1) * eps * eps / (8 * gamma * pi * pi) * exp(1 - r2);
        rho = pow(T, 1 / (gamma - 1));
        v1 = vinf - du * dy;
        v2 = vinf + du * dx;
        p = rho * T;
    } else if (c->bc_kind == 2) {  // constant state
        rho = par[0]; v1 = par[1]; v2 = par[2]; p = par[3]; gamma = par[4];
    } else {  // four-quadrant Riemann data, quadrants NE, NW, SW, SE
        gamma = par[2];
        int q;
        if (x >= par[0]) q = (y >= par[1]) ? 0 : 3;
        else q = (y >= par[1]) ? 1 : 2;
        rho = par[3 + 4 * q]; v1 = par[4 + 4 * q]; v2 = par[5 + 4 * q]; p = par[6 + 4 * q];
    }
    u[0] = rho;
    u[1] = rho * v1;
    u[2] = rho * v2;
    u[3] = p / (gamma - 1) + 0.5 * rho * (v1 * v1 + v2 * v2);
}

// Exchange buffers in LDS hold the variables of every node of the workgroup in
// pairs, [pair][node][2], so that each access moves 16 bytes.  An LDS access
// takes about 4.5 cycles of a CU per wave instruction for 8 and for 16 bytes a
// lane alike, and the contractions are bound by it: with 8-byte accesses LW N=4
// at 1024² spent 1.50 ms in the volume kernel at 10 elements per workgroup.
template <int S> __device__ __forceinline__ void put4(double* s, int idx, const double* w) {
    double2* p = reinterpret_cast<double2*>(s);
    p[idx] = make_double2(w[0], w[1]);
    p[S + idx] = make_double2(w[2], w[3]);
}
template <int S> __device__ __forceinline__ void get4(const double* s, int idx, double* w) {
    const double2* p = reinterpret_cast<const double2*>(s);
    const double2 a = p[idx], b = p[S + idx];
    w[0] = a.x; w[1] = a.y; w[2] = b.x; w[3] = b.y;
}
// f (variables 0..3) in the first two pairs, g in the last two
template <int S> __device__ __forceinline__ void put8(double* s, int idx, const double* f, const double* g) {
    put4<S>(s, idx, f);
    put4<S>(s + 4 * S, idx, g);
}
// row i of an operator in LDS
template <int n> __device__ __forceinline__ void op_row(const double* M, int i, double* r) {
    const double* q = M + i * op_stride(n);
#pragma unroll
    for (int k = 0; k + 1 < n; k += 2) {
        const double2 x = *reinterpret_cast<const double2*>(q + k);
        r[k] = x.x;
        r[k + 1] = x.y;
    }
    if constexpr (n & 1) r[n - 1] = q[n - 1];
}

// Derivative contraction of one element: out[v] = Σ_k M[i,k] f[v](k, j) + Σ_k M[j,k] g[v](i, k)
// with f and g of every node of the workgroup in s (put8) and M (n x n, rows
// of op_stride(n)) in LDS.
template <int n, int S>
__device__ __forceinline__ void contract_rows(const double* s, int base, int i, int j, const double* Di,
                                              const double* Dj, double* out) {
    const double2* p = reinterpret_cast<const double2*>(s);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        double a = 0.0, b = 0.0;
#pragma unroll
        for (int k = 0; k < n; ++k) {
            const double2 x = p[h * S + base + j * n + k];
            a = fma(Di[k], x.x, a);
            b = fma(Di[k], x.y, b);
        }
#pragma unroll
        for (int k = 0; k < n; ++k) {
            const double2 x = p[(2 + h) * S + base + k * n + i];
            a = fma(Dj[k], x.x, a);
            b = fma(Dj[k], x.y, b);
        }
        out[2 * h] = a;
        out[2 * h + 1] = b;
    }
}

__device__ __forceinline__ void load4(const double* p, double* u) {
    const double2* p2 = reinterpret_cast<const double2*>(p);
    const double2 a = p2[0], b = p2[1];
    u[0] = a.x; u[1] = a.y; u[2] = b.x; u[3] = b.y;
}

template <int n, int S>
__device__ __forceinline__ void contract(const double* s, int base, int i, int j, const double* M, double* out) {
    double Di[n], Dj[n];
    op_row<n>(M, i, Di);
    op_row<n>(M, j, Dj);
    contract_rows<n, S>(s, base, i, j, Di, Dj, out);
}

// Boundary state of face node l of element e's face at GLL time level q (q = n:
// the time t itself): the caller's table (kBcTable) or a built-in function.
template <int n>
__device__ __forceinline__ void boundary_state(DevC c, const int* bidx, const double* btab, int levels,
                                               int e, int face, int l, int q, double x, double y, double t,
                                               double* u) {
    if (c->bc_kind == kBcTable) {
        const size_t row = ((size_t)bidx[4 * (size_t)e + face] * n + l) * levels + (levels == 1 ? 0 : q);
        load4(btab + 4 * row, u);
    } else {
        boundary_value(c, x, y, t, u);
    }
}

__device__ __forceinline__ void store4(double* p, const double* u) {
    double2* p2 = reinterpret_cast<double2*>(p);
    p2[0] = make_double2(u[0], u[1]);
    p2[1] = make_double2(u[2], u[3]);
}

template <int RQ = kTraceQ> __device__ __forceinline__ void load_record(const double* p, double* r) {
    const double2* p2 = reinterpret_cast<const double2*>(p);
#pragma unroll
    for (int k = 0; k < RQ / 2; ++k) {
        const double2 x = p2[k];
        r[2 * k] = x.x;
        r[2 * k + 1] = x.y;
    }
}
template <int RQ = kTraceQ> __device__ __forceinline__ void store_record(double* p, const double* r) {
    double2* p2 = reinterpret_cast<double2*>(p);
#pragma unroll
    for (int k = 0; k < RQ / 2; ++k) p2[k] = make_double2(r[2 * k], r[2 * k + 1]);
}

// Pair p of variables of face record `slot` in LDS.  The shock-capturing records
// are 128 bytes apart, half a cycle of the banks: their pairs are permuted by the
// slot, so that neighbouring lanes reading one pair meet different banks.
template <int RQ> __device__ __forceinline__ double2* rec_pair(double* rec, int slot, int p) {
    double2* q = reinterpret_cast<double2*>(rec + slot * RQ);
    return q + (RQ == kTraceQSC ? (p ^ ((slot >> 1) & 7)) : p);
}
template <int RQ> __device__ __forceinline__ void get_record(double* rec, int slot, double* r) {
#pragma unroll
    for (int k = 0; k < RQ / 2; ++k) {
        const double2 x = *rec_pair<RQ>(rec, slot, k);
        r[2 * k] = x.x;
        r[2 * k + 1] = x.y;
    }
}
// pairs [first, last) of the record
template <int RQ, int first = 0, int last = RQ / 2>
__device__ __forceinline__ void put_record(double* rec, int slot, const double* r) {
#pragma unroll
    for (int k = first; k < last; ++k) *rec_pair<RQ>(rec, slot, k) = make_double2(r[2 * k], r[2 * k + 1]);
}

// Buffer selection by integer arithmetic on the loaded pointers: a select
// between fields of the argument struct would be folded into a load from a
// computed offset, which moves the whole struct to private memory.
__device__ __forceinline__ uintptr_t pick_addr(uintptr_t p0, uintptr_t p1, bool second) {
    const uintptr_t m = (uintptr_t)0 - (uintptr_t)second;
    return p0 ^ ((p0 ^ p1) & m);
}
__device__ __forceinline__ const double* sel_in(const KArgs& a, int cur) {
    const uintptr_t b0 = (uintptr_t)a.bufs[0], b1 = (uintptr_t)a.bufs[1], ue = (uintptr_t)a.u;
    const int sel = a.in_sel;
    const bool second = (sel == SEL_CUR) != (cur == 0);
    return (const double*)pick_addr(pick_addr(b0, b1, second), ue, sel == SEL_EXPLICIT);
}
__device__ __forceinline__ double* sel_out(const KArgs& a, int cur) {
    const uintptr_t b0 = (uintptr_t)a.bufs[0], b1 = (uintptr_t)a.bufs[1], ue = (uintptr_t)a.out;
    const int sel = a.out_sel;
    const bool second = (sel == SEL_CUR) != (cur == 0);
    return (double*)pick_addr(pick_addr(b0, b1, second), ue, sel == SEL_EXPLICIT);
}

// A workgroup-table entry, read once per workgroup into scalar registers.
// bid is the workgroup's index in its own table (blockIdx.x, or the index
// within its half of a two-context launch).
__device__ __forceinline__ int4 load_blk_at(const int4* t, int bid) {
    const ConstArr<int> q = const_arr(reinterpret_cast<const int*>(t + bid));
    return make_int4(__builtin_amdgcn_readfirstlane(q[0]), __builtin_amdgcn_readfirstlane(q[1]),
                     __builtin_amdgcn_readfirstlane(q[2]), 0);
}
__device__ __forceinline__ int4 load_blk(const int4* t) { return load_blk_at(t, blockIdx.x); }

// Rusanov flux of one face node from the two face records (left = -side):
// F* = ½(F̃n_L + F̃n_R) − ½ λ (q_R − q_L), λ = max(|v_n|) + max(c)
// (FluxPlusDissipation with flux_central and DissipationLocalLaxFriedrichs,
// src/equations/numerical_fluxes.jl:7-38).
__device__ __forceinline__ void face_numflux(const double* L, const double* R, double* Fs) {
    const double lam = dmax(L[8], R[8]) + dmax(L[9], R[9]);
#pragma unroll
    for (int v = 0; v < 4; ++v) Fs[v] = 0.5 * (L[4 + v] + R[4 + v]) + (-0.5 * lam) * (R[v] - L[v]);
}

// Trixi flux_lax_friedrichs (Rusanov with max_abs_speed_naive) of two states.
__device__ __forceinline__ void rusanov(const double* ul, const double* ur, double gamma, int orientation, double* out) {
    const double gm1 = gamma - 1.0;
    double fl[4], fr[4], al, cl, ar, cr;
    euler_flux_dir(ul, gm1, orientation, fl);
    euler_flux_dir(ur, gm1, orientation, fr);
    speed_parts(ul, gamma, orientation, al, cl);
    speed_parts(ur, gamma, orientation, ar, cr);
    const double lam = dmax(al, ar) + dmax(cl, cr);
#pragma unroll
    for (int v = 0; v < 4; ++v) out[v] = 0.5 * (fl[v] + fr[v]) + (-0.5 * lam) * (ur[v] - ul[v]);
}

__device__ __forceinline__ bool admissible(const double* u, double gamma) {
    const double rho = u[0];
    const double v1 = u[1] / rho, v2 = u[2] / rho;
    const double p = (gamma - 1.0) * (u[3] - 0.5 * (u[1] * v1 + u[2] * v2));
    return rho > 0.0 && p > 0.0;
}

// ---------------------------------------------------------------------------
// MUSCL-Hancock subcell reconstruction of a blended element (calcflux_mh!,
// src/solvers/dgsem_structured/dg_2d.jl:313-538, on the TreeMesh's Cartesian
// metric: unit normals, the element's J⁻¹ at every node).

// minmod(a, b, c, β, 0) (structured/dg_2d.jl:83-95) of finite arguments:
// s·min(β|a|, |b|, β|c|) if a, b, c have one sign, else 0
__device__ __forceinline__ double minmod3(double a, double b, double c, double beta) {
    const double m = fmin(fmin(beta * fabs(a), fabs(b)), beta * fabs(c));
    const double sa = (a > 0.0) ? 1.0 : ((a < 0.0) ? -1.0 : 0.0);
    const double sb = (b > 0.0) ? 1.0 : ((b < 0.0) ? -1.0 : 0.0);
    const double sc = (c > 0.0) ? 1.0 : ((c < 0.0) ? -1.0 : 0.0);
    return (sa != sb || sb != sc) ? 0.0 : sa * m;
}

// limit_variable_slope (equations.jl:262-287) for density (var 0) or pressure
// (var 1): when a doubled extrapolation u* drops below 1e-10, the slope is
// scaled by θ = min(|0.1 v - v| / (|v* - v| + 1e-13), 1) and u* recomputed
// with 2θ and the scaled slope.
__device__ __forceinline__ void mh_limit_var(int var, double* s, double* usl, double* usr, const double* u, double xl,
                                             double xr, double gm1) {
    auto val = [&](const double* q) {
        return var == 0 ? q[0] : gm1 * (q[3] - 0.5 * (q[1] * q[1] + q[2] * q[2]) / q[0]);
    };
    const double vll = val(usl), vrr = val(usr), vlow = val(u);
    if (vll < 1e-10 || vrr < 1e-10) {
        const double thr = 0.1 * vlow;
        const double rll = fabs(thr - vlow) / (fabs(vll - vlow) + 1e-13);
        const double rrr = fabs(thr - vlow) / (fabs(vrr - vlow) + 1e-13);
        const double th = fmin(fmin(rll, rrr), 1.0);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            s[v] *= th;
            usl[v] = u[v] + (2.0 * th) * (xl * s[v]);
            usr[v] = u[v] + (2.0 * th) * (xr * s[v]);
        }
    }
}

// limit_slope (compressible_euler_2d.jl:9-21): density then pressure, face values u + s x
__device__ __forceinline__ void mh_face_pair(double* s, const double* u, double xl, double xr, double gm1, double* qlo,
                                             double* qhi) {
    double usl[4], usr[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        usl[v] = u[v] + 2.0 * s[v] * xl;
        usr[v] = u[v] + 2.0 * s[v] * xr;
    }
    mh_limit_var(0, s, usl, usr, u, xl, xr, gm1);
    mh_limit_var(1, s, usl, usr, u, xl, xr, gm1);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        qlo[v] = u[v] + s[v] * xl;
        qhi[v] = u[v] + s[v] * xr;
    }
}

// Face values of node (i, j) after the Hancock half-step.  s1 holds the
// element's uⁿ (put4).  End nodes (ξ = ±1) keep zero
// slope: the reference's one-sided differences there are 0/0.  Half-step
// terms (all added to the four face values, in the reference's order):
// +Δt/2 J⁻¹ f(left) / hw[i] for 0 < i < n-1, -Δt/2 J⁻¹ f(right) / hw[i] for
// i < n-1, then the same in y.
template <int N, int S>
__device__ __forceinline__ void mh_faces(const double* s1, int sidx, int i, int j, const double* u, DevC c,
                                         double beta, double dtmh, double invJ, double gm1, double* ql, double* qr,
                                         double* qd, double* qu) {
    constexpr int n = N + 1;
    double sx[4] = {0.0, 0.0, 0.0, 0.0}, sy[4] = {0.0, 0.0, 0.0, 0.0};
    double lo[4], hi[4];
    if (i > 0 && i < n - 1) {
        get4<S>(s1, sidx - 1, lo);
        get4<S>(s1, sidx + 1, hi);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double ul = lo[v], ur = hi[v];
            const double back = (u[v] - ul) / c->mh_dx1[i], fwd = (ur - u[v]) / c->mh_dx2[i];
            const double cent = fma(c->mh_fc[i], ur, fma(c->mh_fa[i], ul, c->mh_fb[i] * u[v]));
            sx[v] = minmod3(back, cent, fwd, beta);
        }
    }
    if (j > 0 && j < n - 1) {
        get4<S>(s1, sidx - n, lo);
        get4<S>(s1, sidx + n, hi);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double ud = lo[v], uu = hi[v];
            const double back = (u[v] - ud) / c->mh_dx1[j], fwd = (uu - u[v]) / c->mh_dx2[j];
            const double cent = fma(c->mh_fc[j], uu, fma(c->mh_fa[j], ud, c->mh_fb[j] * u[v]));
            sy[v] = minmod3(back, cent, fwd, beta);
        }
    }
    mh_face_pair(sx, u, c->mh_xl[i], c->mh_xr[i], gm1, ql, qr);
    mh_face_pair(sy, u, c->mh_xl[j], c->mh_xr[j], gm1, qd, qu);
    double fl[4], fr[4], fd[4], fu[4];
    euler_flux_dir(ql, gm1, 1, fl);
    euler_flux_dir(qr, gm1, 1, fr);
    euler_flux_dir(qd, gm1, 2, fd);
    euler_flux_dir(qu, gm1, 2, fu);
    const double hm = (-0.5 * dtmh) * invJ, hp = (0.5 * dtmh) * invJ;
    auto add = [&](double coef, const double* f) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double r = coef * f[v];
            ql[v] += r;
            qr[v] += r;
            qd[v] += r;
            qu[v] += r;
        }
    };
    if (i > 0 && i < n - 1) add(hp / c->mh_hw[i], fl);
    if (i < n - 1) add(hm / c->mh_hw[i], fr);
    if (j > 0 && j < n - 1) add(hp / c->mh_hw[j], fd);
    if (j < n - 1) add(hm / c->mh_hw[j], fu);
}

// Shock-capturing interface flux (dg_2d.jl:1879-1946): the LW flux blended
// with the first-order Rusanov flux of uⁿ by the average blending factor of
// the two elements, falling back to the first-order flux when the low-order
// update of an adjacent node with the blended flux is not admissible.
// Records: [0..3] uⁿ, [4..7] F̃n, [8] |v_n|(Ũ), [9] c(Ũ), [10..13] fn_low, [14] α.
__device__ __forceinline__ void face_numflux_sc(const double* L, const double* R, int orientation, double gamma,
                                                double J, double dt, double w_n, double w_1, double* Fs) {
    double Fh[4], fn[4], Fb[4], low[4];
    face_numflux(L, R, Fh);
    rusanov(L, R, gamma, orientation, fn);
    double alp = 0.5 * (L[14] + R[14]);
#pragma unroll
    for (int v = 0; v < 4; ++v) Fb[v] = (1.0 - alp) * Fh[v] + alp * fn[v];
    const double cl = dt * J / (w_n * 0.5), cr = dt * J / (w_1 * 0.5);
#pragma unroll
    for (int v = 0; v < 4; ++v) low[v] = L[v] - cl * (Fb[v] - L[10 + v]);
    bool ok = admissible(low, gamma);
#pragma unroll
    for (int v = 0; v < 4; ++v) low[v] = R[v] - cr * (R[10 + v] - Fb[v]);
    ok = ok && admissible(low, gamma);
    if (!ok) alp = 1.0;
#pragma unroll
    for (int v = 0; v < 4; ++v) Fs[v] = alp * fn[v] + (1.0 - alp) * Fh[v];
}

// Rusanov flux with a normal direction n (Trixi flux_lax_friedrichs(u_l, u_r,
// n)): Trixi's normal flux (ρv_n, ρv_n v1 + p n1, ρv_n v2 + p n2, (ρe + p) v_n)
// and λ = max|v·n| + max(c)|n|.
__device__ __forceinline__ void rusanov_normal(const double* ul, const double* ur, double gamma, double n1, double n2,
                                               double nn, double* out) {
    const double gm1 = gamma - 1.0;
    double fl[4], fr[4], vl, cl, vr, cr;
    auto side = [&](const double* q, double* f, double& vabs, double& c) {
        const double ir = rcp_nr(q[0]);
        const double v1 = q[1] * ir, v2 = q[2] * ir;
        const double p = gm1 * (q[3] - 0.5 * (q[1] * v1 + q[2] * v2));
        const double vn = fma(v1, n1, v2 * n2), rvn = q[0] * vn;
        f[0] = rvn;
        f[1] = fma(rvn, v1, p * n1);
        f[2] = fma(rvn, v2, p * n2);
        f[3] = (q[3] + p) * vn;
        vabs = fabs(vn);
        c = sqrt_gs(gamma * p * ir) * nn;
    };
    side(ul, fl, vl, cl);
    side(ur, fr, vr, cr);
    const double lam = dmax(vl, vr) + dmax(cl, cr);
#pragma unroll
    for (int v = 0; v < 4; ++v) out[v] = 0.5 * (fl[v] + fr[v]) + (-0.5 * lam) * (ur[v] - ul[v]);
}

// Shock-capturing interface flux on a curvilinear mesh (calc_interface_flux!
// and compute_alp for StructuredMesh, structured/dg_2d.jl:2169-2288).  Records
// (16 doubles): [0..3] Ũ, [4..7] F̃·n, [8..11] uⁿ, [12..15] fn_low.  The LW flux
// takes λ from uⁿ and the jump on Ũ; the low-order flux is the Rusanov flux of
// uⁿ with the same normal; the admissibility test of compute_alp uses each
// side's own node J⁻¹.
__device__ __forceinline__ void face_numflux_sc_curved(const double* L, const double* R, const double* nf, double JL,
                                                       double JR, double aL, double aR, double gamma, double dt,
                                                       double w_n, double w_1, double* Fs) {
    double fn[4], Fh[4], Fb[4], low[4];
    rusanov_normal(L + 8, R + 8, gamma, nf[0], nf[1], nf[2], fn);
    // λ of uⁿ with the normal, as in the Rusanov flux above
    double lam;
    {
        const double gm1 = gamma - 1.0;
        double va[2], ca[2];
        const double* q2[2] = {L + 8, R + 8};
        for (int k = 0; k < 2; ++k) {
            const double* q = q2[k];
            const double ir = rcp_nr(q[0]);
            const double v1 = q[1] * ir, v2 = q[2] * ir;
            const double p = gm1 * (q[3] - 0.5 * (q[1] * v1 + q[2] * v2));
            va[k] = fabs(fma(v1, nf[0], v2 * nf[1]));
            ca[k] = sqrt_gs(gamma * p * ir) * nf[2];
        }
        lam = dmax(va[0], va[1]) + dmax(ca[0], ca[1]);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) Fh[v] = 0.5 * (L[4 + v] + R[4 + v]) + (-0.5 * lam) * (R[v] - L[v]);
    double alp = 0.5 * (aL + aR);
#pragma unroll
    for (int v = 0; v < 4; ++v) Fb[v] = (1.0 - alp) * Fh[v] + alp * fn[v];
    const double cl = dt * JL / (w_n * 0.5), cr = dt * JR / (w_1 * 0.5);
#pragma unroll
    for (int v = 0; v < 4; ++v) low[v] = L[8 + v] - cl * (Fb[v] - L[12 + v]);
    bool ok = admissible(low, gamma);
#pragma unroll
    for (int v = 0; v < 4; ++v) low[v] = R[8 + v] - cr * (R[12 + v] - Fb[v]);
    ok = ok && admissible(low, gamma);
    if (!ok) alp = 1.0;
#pragma unroll
    for (int v = 0; v < 4; ++v) Fs[v] = alp * fn[v] + (1.0 - alp) * Fh[v];
}

// Face record of a face node: jump state, normal component of F̃ and the λ
// ingredients |v_n| and c of the λ state (TreeMesh order: λ from Ũ, jump on uⁿ).
// A face node on a mortar (neighbour code -2 - (3 m + role)): the jump state,
// the normal flux and the λ state the mortar kernel interpolates or pairs.
__device__ __forceinline__ void mortar_side(const KArgs& a, int code, int n, int l, const double* jump,
                                            const double* Fn, const double* lam) {
    double* q = a.mrec + ((size_t)(-2 - code) * n + l) * 12;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        q[v] = jump[v];
        q[4 + v] = Fn[v];
        q[8 + v] = lam[v];
    }
}

__device__ __forceinline__ void make_record(double* r, const double* jump, const double* Fn, double vn_abs, double c) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        r[v] = jump[v];
        r[4 + v] = Fn[v];
    }
    r[8] = vn_abs;
    r[9] = c;
}

// Per-node maxima λ1 = |v1| + c, λ2 = |v2| + c (Trixi max_abs_speeds).
__device__ __forceinline__ void node_speeds(const double* un, double gamma, double& l1, double& l2, bool& bad) {
    const double ir = rcp_nr(un[0]);
    const double v1 = un[1] * ir, v2 = un[2] * ir;
    const double p = (gamma - 1.0) * (un[3] - 0.5 * (un[1] * v1 + un[2] * v2));
    bad = !(un[0] > 0.0) || !(p > 0.0);
    const double cs = sqrt_gs(gamma * p * ir);
    l1 = fabs(v1) + cs;
    l2 = fabs(v2) + cs;
}

// ---------------------------------------------------------------------------
// Element volume computations.  Each fills uN (state), Uc (Ũ), F, G (F̃) and
// vol (D̂F̃ contraction) for the calling node; sD and sDh hold D and D̂, and
// sc = -dt J⁻¹ turns a D contraction into the next time derivative.  Exchanges alternate between two
// LDS buffers A and B, one barrier each: a buffer is rewritten two exchanges
// later, when every lane has passed its contraction.

// Contravariant fluxes of a Cartesian pair: Ja¹·(f, g), Ja²·(f, g)
// (contravariant_flux, structured/dg_2d.jl:550-556).
__device__ __forceinline__ void to_contravariant(const double* J, const double* f, const double* g, double* fc,
                                                 double* gc) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        fc[v] = fma(J[0], f[v], J[1] * g[v]);
        gc[v] = fma(J[2], f[v], J[3] * g[v]);
    }
}
// The node's flux pair into an exchange buffer, contravariant on a curvilinear mesh.
template <int S, bool CURV>
__device__ __forceinline__ void put_fluxes(double* s, int sidx, bool act, const double* J, const double* f,
                                           const double* g) {
    if constexpr (CURV) {
        double cx[4], cy[4];
        to_contravariant(J, f, g, cx, cy);
        if (act) put8<S>(s, sidx, cx, cy);
    } else {
        if (act) put8<S>(s, sidx, f, g);
    }
}

// lw_volume_kernel_3!/4!, dg_2d.jl:674-916, 918-1267, and on a curvilinear mesh
// (CURV) structured/dg_2d.jl:1379-2105: the same procedure with the node's
// contravariant vectors J = (Ja11, Ja12, Ja21, Ja22) turning each Cartesian
// flux derivative for the contractions, while the Cartesian time averages F̃, G̃
// feed the face records.  The last exchange is in A (N = 4) or B (N = 3).
// Bound by FP64 issue with the LDS contractions beside it: per node and level
// four euler_q with five sums each (22 issue slots + 4 for the estimate of 1/ρ),
// 20 LDS loads and 4 stores.  LW N=4 1024², 10 elements per workgroup: whole
// flux vectors, three buffers and plain loads of the constants 1283 us, this form
// with the early loads of volume_body 1138 us.
// With KEEP, tder receives the time derivatives ut, utt, ... (4 per order),
// the intermediates an adjoint sweep needs.
// With terr, the temporal error of the node for the adaptive controller
// (dg_2d.jl:1183-1199, 1251-1265; structured/dg_2d.jl:1595-1681, 1983-2077):
// u_np1 = u - dt J⁻¹ D F̃ and u_np1_low, the same with F̃ before the last flux
// derivative's term, compared variable by variable as
// ((u_np1 - u_np1_low) / (abstol + reltol max(|u_np1|, |u_np1_low|)))², summed.
// terr must be uniformly null or non-null over the workgroup (it adds barriers).
// With SRC, the source terms of the node (*sp) enter every time derivative as
// dt times the source's own difference (dg_2d.jl:980-987, 1033-1045, 1093-1103,
// 1148-1160; five-point s_tt in the curvilinear kernel 4) and Ssrc receives
// S = s + s_t/2 + s_tt/6 + ... (1228-1247), which the caller adds to the residual.
// Without FLUXES it ends with Ũ and tder, which need neither the last level's
// stencil nor F̃.
template <int N, int EB, bool CURV = false, bool KEEP = false, bool SRC = false, bool FLUXES = true>
__device__ __forceinline__ void lw_element(const double* uN, const double* J, double dt, double sc, double gamma,
                                           int i, int j, bool act, int sidx, int sbase, double* A, double* B,
                                           const double* sD, const double* sDh, double* Uc, double* F, double* G,
                                           double* vol, double* tder = nullptr, double* terr = nullptr,
                                           double abstol = 0.0, double reltol = 0.0, const SrcPt* sp = nullptr,
                                           double* Ssrc = nullptr) {
    using G_ = VGeo<N, EB>;
    constexpr int n = G_::n, S = G_::S;
    const double gm1 = gamma - 1.0, kh = -0.5 * gm1;
    double q0[5], sum[5], st[4][4], w[4], sk[4] = {0.0, 0.0, 0.0, 0.0};
    double Di[n], Dj[n];
    euler_q(uN, gamma, kh, q0);
    euler_join(q0, uN[1], uN[2], uN[3], gm1, kh, F, G);
#pragma unroll
    for (int m = 0; m < 5; ++m) sum[m] = q0[m];
#pragma unroll
    for (int k = 1; k <= N; ++k) {
        // F, G: the (k-1)-th time difference of the flux pair
        double* buf = (k & 1) ? A : B;
        put_fluxes<S, CURV>(buf, sidx, act, J, F, G);
        __syncthreads();
        if (k == 1) {  // read once: 20 LDS loads a level instead of 26 (1.3% of a step at 1024², N=4)
            op_row<n>(sD, i, Di);
            op_row<n>(sD, j, Dj);
        }
        contract_rows<n, S>(buf, sbase, i, j, Di, Dj, w);
        if constexpr (SRC) src_level_c(*sp, dt, k - 1, CURV && N == 4, sk, Ssrc, lw_weight(k - 1));
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            w[v] *= sc;
            if constexpr (SRC) w[v] = fma(dt, sk[v], w[v]);
            if constexpr (KEEP) tder[4 * (k - 1) + v] = w[v];
            Uc[v] = fma(lw_weight(k), w[v], k == 1 ? uN[v] : Uc[v]);
#pragma unroll
            for (int s = 0; s < 4; ++s) st[s][v] = fma(kTaylor[s][k - 1], w[v], k == 1 ? uN[v] : st[s][v]);
        }
        if (!FLUXES && k == N) return;
        constexpr TimeDiff tds[5] = {{}, time_diff<N>(1), time_diff<N>(2), time_diff<N>(3), time_diff<N>(4)};
        const TimeDiff td = tds[k];
        double d[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, q[5];
        // in the order of time, uⁿ between u(t + dt) and u(t - dt): small partial sums
#pragma unroll
        for (int r = 0; r < 5; ++r) {
            const int s = r == 0 ? 2 : r == 1 ? 0 : r == 2 ? 4 : r == 3 ? 1 : 3;
            if (td.c[s] == 0.0) continue;
            if (s < 4) euler_q(st[s & 3], gamma, kh, q);
#pragma unroll
            for (int m = 0; m < 5; ++m) d[m] = fma(td.c[s], s < 4 ? q[m] : q0[m], d[m]);
        }
#pragma unroll
        for (int m = 0; m < 5; ++m) {
            if (td.scale != 1.0) d[m] *= td.scale;
            sum[m] = fma(lw_weight(k), d[m], sum[m]);
        }
        if (k < N || terr)
            euler_join(d, td.linear * w[1], td.linear * w[2], td.linear * w[3], gm1, kh, F, G);
    }
    // the source's last difference enters S only
    if constexpr (SRC) src_level_c(*sp, dt, N, CURV && N == 4, sk, Ssrc, lw_weight(N));
    double* last = (N & 1) ? B : A;   // the exchange of F̃
    double* other = (N & 1) ? A : B;
    if (terr) {
        __syncthreads();  // the last contraction has read this buffer
        put_fluxes<S, CURV>(other, sidx, act, J, F, G);
    }
    // the linear parts of F̃: those of Ũ, up to the factor the last stencil puts on them
    constexpr double miss = lw_weight(N) * (1.0 - time_diff<N>(N).linear);
    double l[4];
#pragma unroll
    for (int v = 1; v < 4; ++v) l[v] = miss == 0.0 ? Uc[v] : fma(-miss, w[v], Uc[v]);
    euler_join(sum, l[1], l[2], l[3], gm1, kh, F, G);
    put_fluxes<S, CURV>(last, sidx, act, J, F, G);
    __syncthreads();
    contract<n, S>(last, sbase, i, j, sDh, vol);
    if (terr) {
        // one contraction at a time: interleaved, their loads spill 23 registers
        double a1[4], a2[4];
        __builtin_amdgcn_sched_barrier(0);
        contract<n, S>(last, sbase, i, j, sD, a1);  // D F̃
        __builtin_amdgcn_sched_barrier(0);
        contract<n, S>(other, sbase, i, j, sD, a2);  // D of the last flux derivative
        // u_np1 - u_np1_low is formed as the contraction of the last term itself,
        // not as a difference of the two updates (which cancels to ~1e-7 relative)
        double e = 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double d = sc * (lw_weight(N) * a2[v]);
            const double hi = fma(sc, a1[v], uN[v]);
            const double lo = hi - d;
            const double r = d / (abstol + reltol * dmax(fabs(hi), fabs(lo)));
            e = fma(r, r, e);
        }
        *terr = e;
        __syncthreads();  // both buffers are reused for the face records
    }
}

// acc += weight · f_t of the two-level Taylor states u ± ut, u ± 2ut
// (five euler_q sums; the linear part of f_t is ut)
__device__ __forceinline__ void mdrk_ft(const double* u, const double* ut, double gamma, double kh, double weight,
                                        double* acc) {
    constexpr TimeDiff td = time_diff<4>(1);
    double d[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, q[5], w[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int s = r == 0 ? 2 : r == 1 ? 0 : r == 2 ? 1 : 3;
#pragma unroll
        for (int v = 0; v < 4; ++v) w[v] = fma(kTaylor[s][0], ut[v], u[v]);
        euler_q(w, gamma, kh, q);
#pragma unroll
        for (int m = 0; m < 5; ++m) d[m] = fma(td.c[s], q[m], d[m]);
    }
#pragma unroll
    for (int m = 0; m < 5; ++m) acc[m] = fma(weight * td.scale, d[m], acc[m]);
}

// mdrk_kernel_1!, tree/multi_derivative_2d.jl:263-420 and (CURV)
// structured/multi_derivative_2d.jl:82-243: F̃ = f/2 + f_t/8, Ũ = u/2 + ut/8, ut
// from the contravariant fluxes on a curvilinear mesh.  F2 = f + f_t/6 and
// U2 = u + ut/6 are recomputed by the stage-2 kernel instead of being stored.
// With SRC (323-379; structured 146-200): ut gets dt s(t), and
// Ssrc = s/2 + s_t/8.  The last exchange is in B.
template <int N, int EB, bool CURV = false, bool SRC = false>
__device__ __forceinline__ void mdrk1_element(const double* uN, const double* J, double dt, double sc, double gamma,
                                              int i, int j, bool act, int sidx, int sbase, double* A, double* B,
                                              const double* sD, const double* sDh, double* Uc, double* F, double* G,
                                              double* vol, const SrcPt* sp = nullptr, double* Ssrc = nullptr) {
    using G_ = VGeo<N, EB>;
    constexpr int n = G_::n, S = G_::S;
    const double gm1 = gamma - 1.0, kh = -0.5 * gm1;
    double q[5], ut[4];
    euler_q(uN, gamma, kh, q);
    euler_join(q, uN[1], uN[2], uN[3], gm1, kh, F, G);
    put_fluxes<S, CURV>(A, sidx, act, J, F, G);
    __syncthreads();
    contract<n, S>(A, sbase, i, j, sD, ut);
#pragma unroll
    for (int v = 0; v < 4; ++v) ut[v] *= sc;
    if constexpr (SRC) {
        double s[4], sd[4];
        src_eval(*sp, 0.0, s);
        src_t5(*sp, 0.0, dt, sd);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            ut[v] = fma(dt, s[v], ut[v]);
            Ssrc[v] = fma(0.125, sd[v], 0.5 * s[v]);
        }
    }
#pragma unroll
    for (int m = 0; m < 5; ++m) q[m] *= 0.5;
    mdrk_ft(uN, ut, gamma, kh, 0.125, q);
#pragma unroll
    for (int v = 0; v < 4; ++v) Uc[v] = fma(0.125, ut[v], 0.5 * uN[v]);
    euler_join(q, Uc[1], Uc[2], Uc[3], gm1, kh, F, G);
    put_fluxes<S, CURV>(B, sidx, act, J, F, G);
    __syncthreads();
    contract<n, S>(B, sbase, i, j, sDh, vol);
}

// mdrk_kernel_2!, tree/multi_derivative_2d.jl:423-555 and (CURV)
// structured/multi_derivative_2d.jl:245-445: F̃ = F2 + f_t(us)/3, Ũ = U2 + ust/3
// with F2, U2 recomputed from uⁿ.  With SRC on a TreeMesh (487-522): the
// recomputed stage-1 ut gets dt s(t) and S2 = s + s_t/6; ust gets dt s(t + dt/2),
// and Ssrc = S2 + s_t(t + dt/2)/3.  On a StructuredMesh (326-339, 358-385): ut
// and ust += dt s(t); Ssrc = s + s_t/3 about t, the reference's stage 2
// overwriting the S2 it loads (stage 1's s + s_t/6) with s.  The last exchange
// is in A, behind a barrier of its own (both buffers have just been read).
template <int N, int EB, bool CURV = false, bool SRC = false>
__device__ __forceinline__ void mdrk2_element(const double* uN, const double* usn, const double* J, double dt,
                                              double sc, double gamma, int i, int j, bool act, int sidx, int sbase,
                                              double* A, double* B, const double* sD, const double* sDh, double* Uc,
                                              double* F, double* G, double* vol, const SrcPt* sp = nullptr,
                                              double* Ssrc = nullptr) {
    using G_ = VGeo<N, EB>;
    constexpr int n = G_::n, S = G_::S;
    const double gm1 = gamma - 1.0, kh = -0.5 * gm1;
    double q[5], qs[5], ut[4], ust[4];
    euler_q(uN, gamma, kh, q);
    euler_join(q, uN[1], uN[2], uN[3], gm1, kh, F, G);
    put_fluxes<S, CURV>(A, sidx, act, J, F, G);
    euler_q(usn, gamma, kh, qs);
    euler_join(qs, usn[1], usn[2], usn[3], gm1, kh, F, G);
    put_fluxes<S, CURV>(B, sidx, act, J, F, G);
    __syncthreads();
    contract<n, S>(A, sbase, i, j, sD, ut);
    contract<n, S>(B, sbase, i, j, sD, ust);
#pragma unroll
    for (int v = 0; v < 4; ++v) { ut[v] *= sc; ust[v] *= sc; }
    if constexpr (SRC && CURV) {
        double s[4], sd[4];
        src_eval(*sp, 0.0, s);
        src_t5(*sp, 0.0, dt, sd);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            ut[v] = fma(dt, s[v], ut[v]);
            ust[v] = fma(dt, s[v], ust[v]);
            Ssrc[v] = fma(1.0 / 3.0, sd[v], s[v]);
        }
    } else if constexpr (SRC) {
        double sk[4], sh[4];
        src_eval(*sp, 0.0, sk);
        src_eval(*sp, 0.5 * dt, sh);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            ut[v] = fma(dt, sk[v], ut[v]);
            ust[v] = fma(dt, sh[v], ust[v]);
            Ssrc[v] = sk[v];
        }
        src_t5(*sp, 0.0, dt, sk);
        src_t5(*sp, 0.5 * dt, dt, sh);
#pragma unroll
        for (int v = 0; v < 4; ++v) Ssrc[v] = fma(1.0 / 3.0, sh[v], fma(1.0 / 6.0, sk[v], Ssrc[v]));
    }
    mdrk_ft(uN, ut, gamma, kh, 1.0 / 6.0, q);    // F2
    mdrk_ft(usn, ust, gamma, kh, 1.0 / 3.0, q);
#pragma unroll
    for (int v = 0; v < 4; ++v) Uc[v] = fma(1.0 / 3.0, ust[v], fma(1.0 / 6.0, ut[v], uN[v]));
    euler_join(q, Uc[1], Uc[2], Uc[3], gm1, kh, F, G);
    __syncthreads();
    put_fluxes<S, CURV>(A, sidx, act, J, F, G);
    __syncthreads();
    contract<n, S>(A, sbase, i, j, sDh, vol);
}

// ---------------------------------------------------------------------------
// Hyperbolic-parabolic element procedures (compressible Navier-Stokes with
// conservative gradient variables).  The BR1 gradient of the input state is
// formed in the volume workgroup itself (weak-form D̂ volume term, central
// face value ½(u + u_neighbour) lifted by 1/w at the end nodes, ×J⁻¹), so no
// gradient array goes through HBM.  The LW procedure then runs on the total
// flux f_a(u) - f_v(u, ∇u) with Taylor states of u and of ∇u, the time
// derivatives' gradients being element-local (J⁻¹ D ∂ₜᵏu).  Only the total
// F̃ = F̃a - F̃v is kept: the interface flux of the reference,
// LW-Rusanov(F̃a) - ½(F̃v_L + F̃v_R), equals ½(F̃_L + F̃_R) - ½λ(u_R - u_L),
// so the face records and the surface kernel are those of the Euler path.
// Reference: lw_volume_kernel_3!/4!, dg_2d_parabolic.jl:725-1860;
// calc_interface_flux_hyperbolic_parabolic!, dg_2d_parabolic.jl:1911-1948;
// mdrk_kernel_1!/2!, multi_derivative_2d_parabolic.jl:221-711.

// Separate x and y contractions of the 4 variables in s (put4):
// ox[v] = Σ_k M[i,k] s[v](k, j), oy[v] = Σ_k M[j,k] s[v](i, k).
template <int n, int S>
__device__ __forceinline__ void contract_xy(const double* s, int base, int i, int j, const double* M, double* ox,
                                            double* oy) {
    double Mi[n], Mj[n];
    op_row<n>(M, i, Mi);
    op_row<n>(M, j, Mj);
    const double2* p = reinterpret_cast<const double2*>(s);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        double ax = 0.0, bx = 0.0, ay = 0.0, by = 0.0;
#pragma unroll
        for (int k = 0; k < n; ++k) {
            const double2 x = p[h * S + base + j * n + k], y = p[h * S + base + k * n + i];
            ax = fma(Mi[k], x.x, ax);
            bx = fma(Mi[k], x.y, bx);
            ay = fma(Mj[k], y.x, ay);
            by = fma(Mj[k], y.y, by);
        }
        ox[2 * h] = ax;
        ox[2 * h + 1] = bx;
        oy[2 * h] = ay;
        oy[2 * h + 1] = by;
    }
}

// Viscous fluxes of CompressibleNavierStokesDiffusion2D from the conservative
// state and conservative gradients (convert_derivative_to_primitive,
// compressible_navier_stokes_2d.jl:37-57; Trixi flux(u, ∇u, orientation)).
__device__ __forceinline__ void ns_visc_fluxes(const double* u, const double* gx, const double* gy, double gm1,
                                               DevC c, double* fx, double* fy) {
    const double ir = rcp_nr(u[0]);
    const double v1 = u[1] * ir, v2 = u[2] * ir;
    const double p = gm1 * (u[3] - 0.5 * (u[1] * v1 + u[2] * v2));
    const double T = p * ir;
    const double vv = v1 * v1 + v2 * v2;
    auto prim = [&](const double* W, double& v1d, double& v2d, double& Td) {
        const double rd = W[0];
        v1d = (W[1] - rd * v1) * ir;
        v2d = (W[2] - rd * v2) * ir;
        const double pd = (W[3] - 0.5 * rd * vv - u[0] * (v1 * v1d + v2 * v2d)) * gm1;
        Td = (pd - rd * T) * ir;
    };
    double v1x, v2x, Tx, v1y, v2y, Ty;
    prim(gx, v1x, v2x, Tx);
    prim(gy, v1y, v2y, Ty);
    const double mu = c->visc_mu, kappa = c->visc_kappa;
    const double t11 = (4.0 / 3.0) * v1x - (2.0 / 3.0) * v2y;
    const double t12 = v1y + v2x;
    const double t22 = (4.0 / 3.0) * v2y - (2.0 / 3.0) * v1x;
    fx[0] = 0.0;
    fx[1] = t11 * mu;
    fx[2] = t12 * mu;
    fx[3] = (v1 * t11 + v2 * t12 + kappa * Tx) * mu;
    fy[0] = 0.0;
    fy[1] = t12 * mu;
    fy[2] = t22 * mu;
    fy[3] = (v1 * t12 + v2 * t22 + kappa * Ty) * mu;
}

// The total flux pair f_a(u) - f_v(u, ∇u) as the five values the stencils sum:
// q = (f2, f3 = g2, f4, g3, g4), the mass fluxes ρv1, ρv2 being linear and
// without a viscous part (euler_q keeps p out of its sums; here the stresses sit
// on top of it).  The primitive gradients stay multiplied by ρ and 1/ρ enters
// the viscosity once: 52 instructions against 77 for the two flux vectors.
__device__ __forceinline__ void ns_q(const double* u, const double* gx, const double* gy, double gm1, DevC c,
                                     double* q) {
    const double ir = rcp_nr(u[0]);
    const double v1 = u[1] * ir, v2 = u[2] * ir;
    const double q11 = u[1] * v1, q12 = u[1] * v2, q22 = u[2] * v2;
    const double hk = 0.5 * (q11 + q22);
    const double p = gm1 * (u[3] - hk);
    const double T = p * ir, hv = hk * ir;
    // ρ ∂v1, ρ ∂v2 and ρ ∂T of one direction
    auto prim = [&](const double* W, double& a1, double& a2, double& rT) {
        a1 = fma(-W[0], v1, W[1]);
        a2 = fma(-W[0], v2, W[2]);
        const double pd = fma(-v2, a2, fma(-v1, a1, fma(-W[0], hv, W[3])));
        rT = fma(gm1, pd, -(W[0] * T));
    };
    double a1x, a2x, Tx, a1y, a2y, Ty;
    prim(gx, a1x, a2x, Tx);
    prim(gy, a1y, a2y, Ty);
    const double mi = c->visc_mu * ir, ki = mi * c->visc_kappa;
    const double t11 = mi * fma(4.0 / 3.0, a1x, (-2.0 / 3.0) * a2y);
    const double t12 = mi * (a1y + a2x);
    const double t22 = mi * fma(4.0 / 3.0, a2y, (-2.0 / 3.0) * a1x);
    const double H = u[3] + p;
    q[0] = (q11 + p) - t11;
    q[1] = q12 - t12;
    q[2] = fma(H, v1, -fma(v1, t11, fma(v2, t12, ki * Tx)));
    q[3] = (q22 + p) - t22;
    q[4] = fma(H, v2, -fma(v1, t12, fma(v2, t22, ki * Ty)));
}
// the flux pair of the sums q and the linear parts of the mass fluxes
__device__ __forceinline__ void ns_join(const double* q, double l1, double l2, double* f, double* g) {
    f[0] = l1;
    f[1] = q[0];
    f[2] = q[1];
    f[3] = q[2];
    g[0] = l2;
    g[1] = q[1];
    g[2] = q[3];
    g[3] = q[4];
}

// Viscous time-step bound of one node, J⁻² max(4μ/(3ρ), μκ/(ρ Pr))
// (compressible_navier_stokes_2d.jl:230-237), with IEEE divisions.
__device__ __forceinline__ double lam_visc(const double* u, double invJ, DevC c) {
    const double mu = c->visc_mu, rho = u[0];
    return invJ * invJ * dmax(4.0 * mu / (3.0 * rho), mu * c->visc_kappa / (rho * c->visc_Pr));
}
// The same with the node's J⁻¹ of a curvilinear mesh in place of J⁻² (the 2-D
// Jacobian already scales as h²)
__device__ __forceinline__ double lam_visc_curved(const double* u, double invJ, DevC c) {
    const double mu = c->visc_mu, rho = u[0];
    return invJ * dmax(4.0 * mu / (3.0 * rho), mu * c->visc_kappa / (rho * c->visc_Pr));
}

// Reference-space gradient (w_ξ, w_η) → Cartesian with the transposed
// contravariant vectors J = (Ja11, Ja12, Ja21, Ja22) and the node's J⁻¹
// (compute_local_grad_u!, p4est/dg_2d_parabolic.jl:51-104).
__device__ __forceinline__ void grad_to_cartesian(const double* J, double invJ, double* gx, double* gy) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const double g1 = gx[v], g2 = gy[v];
        gx[v] = fma(J[0], g1, J[2] * g2) * invJ;
        gy[v] = fma(J[1], g1, J[3] * g2) * invJ;
    }
}

// BR1 gradient of the node's state: s holds the element's state (put4 before
// the barrier), src the state array the face neighbours are read from.
template <int N, int EB, bool CURV = false>
__device__ __forceinline__ void br1_gradient(const double* s, const double* src, int nbx, int nby, DevC c,
                                             int i, int j, int sbase, double invJ, const double* sDh,
                                             const double* uown, double* gx, double* gy, const double* Jn = nullptr) {
    using G_ = VGeo<N, EB>;
    constexpr int n = G_::n, NN = G_::NN, S = G_::S;
    contract_xy<n, S>(s, sbase, i, j, sDh, gx, gy);
    // at a no-slip wall the interface value is the wall state prim2cons(ρ, v_wall, p)
    // of the node (Trixi calc_boundary_flux_by_direction_gradient! with
    // compressible_navier_stokes_2d.jl:113-124)
    // the gradient's boundary value at a no-slip wall: prim2cons(ρ, v_wall, p) with the
    // node's pressure (Adiabatic) or p = ρ T_wall (Isothermal, the reference's R = 1;
    // compressible_navier_stokes_2d.jl:93-101)
    auto wall_state = [&](int f, double* uo) {
        const double vw1 = c->wall_v[2 * f], vw2 = c->wall_v[2 * f + 1];
        const double rho = uown[0];
        const double p = c->wall_iso[f] ? rho * c->wall_T[f]
                                        : (c->gamma - 1.0) * (uown[3] - 0.5 * (uown[1] * uown[1] + uown[2] * uown[2]) / rho);
        uo[0] = rho;
        uo[1] = rho * vw1;
        uo[2] = rho * vw2;
        uo[3] = p / (c->gamma - 1.0) + 0.5 * rho * (vw1 * vw1 + vw2 * vw2);
    };
    if (i == 0 || i == n - 1) {
        const int f = (i == 0) ? 0 : 1;
        const int nb = nbx;
        const double wf = f ? c->bnd_hi : -c->bnd_lo;
        if (nb >= 0) {
            double un[4];
            load4(src + ((size_t)nb * NN + j * n + (n - 1 - i)) * 4, un);
#pragma unroll
            for (int v = 0; v < 4; ++v) gx[v] = fma(0.5 * (uown[v] + un[v]), wf, gx[v]);
        } else if (c->ns_walls) {
            double uo[4];
            wall_state(f, uo);
#pragma unroll
            for (int v = 0; v < 4; ++v) gx[v] = fma(uo[v], wf, gx[v]);
        }
    }
    if (j == 0 || j == n - 1) {
        const int f = (j == 0) ? 2 : 3;
        const int nb = nby;
        const double wf = (f & 1) ? c->bnd_hi : -c->bnd_lo;
        if (nb >= 0) {
            double un[4];
            load4(src + ((size_t)nb * NN + (n - 1 - j) * n + i) * 4, un);
#pragma unroll
            for (int v = 0; v < 4; ++v) gy[v] = fma(0.5 * (uown[v] + un[v]), wf, gy[v]);
        } else if (c->ns_walls) {
            double uo[4];
            wall_state(f, uo);
#pragma unroll
            for (int v = 0; v < 4; ++v) gy[v] = fma(uo[v], wf, gy[v]);
        }
    }
    if constexpr (CURV) {
        // curvilinear BR1 (Trixi calc_gradient! for P4estMesh): the reference-space
        // volume and lifted interface terms above, turned with the transposed
        // metric; the face terms of the element's own outward normal ±Ja are the
        // same linear map
        grad_to_cartesian(Jn, invJ, gx, gy);
        return;
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        gx[v] *= invJ;
        gy[v] *= invJ;
    }
}

// Taylor states of u and ∇u: q = 0..3 for u+, u-, u++, u--.
struct ParStates {
    double u[4][4], x[4][4], y[4][4];
    __device__ __forceinline__ void init(const double* w, const double* wx, const double* wy) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                u[q][v] = w[v];
                x[q][v] = wx[v];
                y[q][v] = wy[v];
            }
    }
    // states += c[q] · (w, wx, wy)
    __device__ __forceinline__ void add(double c0, double c1, double c2, double c3, const double* w,
                                        const double* wx, const double* wy) {
        const double cq[4] = {c0, c1, c2, c3};
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                u[q][v] = fma(cq[q], w[v], u[q][v]);
                x[q][v] = fma(cq[q], wx[v], x[q][v]);
                y[q][v] = fma(cq[q], wy[v], y[q][v]);
            }
    }
    __device__ __forceinline__ void flux(int s, double gm1, DevC c, double* q) const {
        ns_q(u[s], x[s], y[s], gm1, c, q);
    }
    // components 1..3 of the viscous fluxes of state q: (fx1, fx2, fx3, fy1, fy2, fy3)
    __device__ __forceinline__ void visc6(int q, double gm1, DevC c, double* out) const {
        double fx[4], fy[4];
        ns_visc_fluxes(u[q], x[q], y[q], gm1, c, fx, fy);
        out[0] = fx[1];
        out[1] = fx[2];
        out[2] = fx[3];
        out[3] = fy[1];
        out[4] = fy[2];
        out[5] = fy[3];
    }
};

// Time derivative of the next level and its element-local gradient:
// w = sc D · (dx, dy), sc = -dt J⁻¹, (+ add, the level's source term dt·s) through sa,
// then (wx, wy) = J⁻¹ D w through sg.
template <int N, int EB, bool CURV = false>
__device__ __forceinline__ void par_level(bool act, int sidx, int sbase, int i, int j, double invJ, double sc,
                                          double* sa, double* sg, const double* sD, const double* dx,
                                          const double* dy, double* w, double* wx, double* wy,
                                          const double* Jn = nullptr, const double* add = nullptr) {
    using G_ = VGeo<N, EB>;
    constexpr int n = G_::n, S = G_::S;
    if constexpr (CURV) {
        // contravariant pair for the derivative contraction
        double cx[4], cy[4];
        to_contravariant(Jn, dx, dy, cx, cy);
        if (act) put8<S>(sa, sidx, cx, cy);
    } else {
        if (act) put8<S>(sa, sidx, dx, dy);
    }
    __syncthreads();
    contract<n, S>(sa, sbase, i, j, sD, w);
#pragma unroll
    for (int v = 0; v < 4; ++v) w[v] *= sc;
    if (add) {
#pragma unroll
        for (int v = 0; v < 4; ++v) w[v] += add[v];
    }
    if (act) put4<S>(sg, sidx, w);
    __syncthreads();
    contract_xy<n, S>(sg, sbase, i, j, sD, wx, wy);
    if constexpr (CURV) {
        grad_to_cartesian(Jn, invJ, wx, wy);
    } else {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            wx[v] *= invJ;
            wy[v] *= invJ;
        }
    }
}

// lw_volume_kernel_3!/4! with viscous terms (dg_2d_parabolic.jl:725-1189,
// 1191-1860): the Euler procedure of lw_element on the total
// flux, with the states of ∇u advanced by the same Taylor coefficients.
// Buffer use: s0 keeps f(uⁿ) for the 5- and 3-point stencils, s1 takes each
// flux derivative, s2 each time derivative; the final F̃ exchange is in s2.
template <int N, int EB, bool CURV = false, bool WALL = false>
__device__ __forceinline__ void lwp_element(const double* uN, const double* gxN, const double* gyN, double invJ,
                                            double sc, double gm1, DevC c, int i, int j, bool act, int sidx,
                                            int sbase, double* s0, double* s1, double* s2, const double* sD,
                                            const double* sDh, double* Uc, double* F, double* G,
                                            double* vol, const double* Jn = nullptr, double* const* wq = nullptr,
                                            double* terr = nullptr, double abstol = 0.0, double reltol = 0.0,
                                            bool has_src = false, const NsSrcPt& sp = NsSrcPt{},
                                            double* Ssrc = nullptr, double dtv = 0.0) {
    using G_ = VGeo<N, EB>;
    constexpr int n = G_::n, S = G_::S;
    double q0[5], sum[5];
    ns_q(uN, gxN, gyN, gm1, c, q0);
    ns_join(q0, uN[1], uN[2], F, G);
#pragma unroll
    for (int m = 0; m < 5; ++m) sum[m] = q0[m];
    // the Navier-Stokes convergence source (the wall instantiation, has_src;
    // dg_2d_parabolic.jl:725-1860): level k of the Taylor procedure gets dt·s^(k)
    // before its gradient is formed, S the same weights as F̃ (s^(k) the time
    // difference of ns_src_diff; kernel 4 takes the five-point s_tt)
    auto src_lvl = [&](int order, double weight, double* ds) {
        if constexpr (WALL) {
            double v4[4] = {0.0, 0.0, 0.0, 0.0};
            if (has_src) ns_src_diff(sp, dtv, order, N == 4, v4);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (ds) ds[v] = dtv * v4[v];
                if (has_src) Ssrc[v] = order == 0 ? weight * v4[v] : fma(weight, v4[v], Ssrc[v]);
            }
        }
    };
    // with walls: the time average of the viscous flux of a wall face node in the
    // face's orientation, alongside F̃, accumulated in the node's wall record
    // wq[o] (o = 0: its x face, 1: its y face; null where that face is no wall):
    // [time average (3), value at uⁿ (3)].  Only wall lanes touch memory here.
    if constexpr (WALL) {
        double fx[4], fy[4];
        ns_visc_fluxes(uN, gxN, gyN, gm1, c, fx, fy);
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            double* q = wq[o];
            if (!q) continue;
            const double* f = o ? fy : fx;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                q[k] = f[1 + k];
                q[3 + k] = f[1 + k];
            }
        }
    }
    // one stage of the wall average: weight · scale · (cv v(uⁿ) + Σ c_s v(state s)),
    // the states u+, u-, u++, u-- one at a time, both orientations from one
    // viscous-flux evaluation; only wall lanes enter
    auto wall_stage = [&](const ParStates& Ps, double c0, double c1, double c2, double c3, double cv, double scale,
                          double weight, bool outer) {
        if constexpr (WALL) {
            if (!wq[0] && !wq[1]) return;
            double d[6], a6[6];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                d[k] = wq[0] ? cv * wq[0][3 + k] : 0.0;
                d[3 + k] = wq[1] ? cv * wq[1][3 + k] : 0.0;
            }
            Ps.visc6(0, gm1, c, a6);
#pragma unroll
            for (int k = 0; k < 6; ++k) d[k] = fma(c0, a6[k], d[k]);
            Ps.visc6(1, gm1, c, a6);
#pragma unroll
            for (int k = 0; k < 6; ++k) d[k] = fma(c1, a6[k], d[k]);
            if (outer) {
                Ps.visc6(2, gm1, c, a6);
#pragma unroll
                for (int k = 0; k < 6; ++k) d[k] = fma(c2, a6[k], d[k]);
                Ps.visc6(3, gm1, c, a6);
#pragma unroll
                for (int k = 0; k < 6; ++k) d[k] = fma(c3, a6[k], d[k]);
            }
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                double* q = wq[o];
                if (!q) continue;
#pragma unroll
                for (int k = 0; k < 3; ++k) q[k] = fma(weight, scale * d[3 * o + k], q[k]);
            }
        }
    };
    double w[4], wx[4], wy[4];
    ParStates P;
    P.init(uN, gxN, gyN);
#pragma unroll
    for (int k = 1; k <= N; ++k) {
        // F, G: the (k-1)-th time difference of the total flux pair
        double* sa = k == 1 ? s0 : s1;
        if constexpr (WALL) {
            double ds[4];
            src_lvl(k - 1, lw_weight(k - 1), ds);
            par_level<N, EB, CURV>(act, sidx, sbase, i, j, invJ, sc, sa, s2, sD, F, G, w, wx, wy, Jn, ds);
        } else {
            par_level<N, EB, CURV>(act, sidx, sbase, i, j, invJ, sc, sa, s2, sD, F, G, w, wx, wy, Jn);
        }
        // s0 keeps the node's own Cartesian f(uⁿ) for the centred stencils: on a
        // curvilinear mesh written once every lane has passed its contraction
        if constexpr (CURV) {
            if (k == 1 && act) put8<S>(s0, sidx, F, G);
        }
        P.add(kTaylor[0][k - 1], kTaylor[1][k - 1], kTaylor[2][k - 1], kTaylor[3][k - 1], w, wx, wy);
#pragma unroll
        for (int v = 0; v < 4; ++v) Uc[v] = fma(lw_weight(k), w[v], k == 1 ? uN[v] : Uc[v]);
        constexpr TimeDiff tds[5] = {{}, time_diff<N>(1), time_diff<N>(2), time_diff<N>(3), time_diff<N>(4)};
        const TimeDiff td = tds[k];
        double d[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, q[5];
#pragma unroll
        for (int r = 0; r < 5; ++r) {
            const int s = r == 0 ? 2 : r == 1 ? 0 : r == 2 ? 4 : r == 3 ? 1 : 3;
            if (td.c[s] == 0.0) continue;
            if (s < 4) {
                P.flux(s & 3, gm1, c, q);
            } else {
                double f0[4], g0[4];
                get4<S>(s0, sidx, f0);
                get4<S>(s0 + 4 * S, sidx, g0);
                q[0] = f0[1];
                q[1] = f0[2];
                q[2] = f0[3];
                q[3] = g0[2];
                q[4] = g0[3];
            }
#pragma unroll
            for (int m = 0; m < 5; ++m) d[m] = fma(td.c[s], q[m], d[m]);
        }
#pragma unroll
        for (int m = 0; m < 5; ++m) {
            if (td.scale != 1.0) d[m] *= td.scale;
            sum[m] = fma(lw_weight(k), d[m], sum[m]);
        }
        ns_join(d, td.linear * w[1], td.linear * w[2], F, G);
        // the viscous part of this difference into the wall records
        wall_stage(P, td.c[0], td.c[1], td.c[2], td.c[3], td.c[4], td.scale, lw_weight(k), td.c[2] != 0.0);
    }
    // s0 is read only at the own node since the first contraction: it takes
    // the total f_tttt for the temporal error
    if constexpr (N == 4) {
        if (terr && act) put8<S>(s0, sidx, F, G);
    }
    // the source's last difference enters S only: s_tttt/120 (kernel 4), s_ttt/24 (kernel 3)
    src_lvl(N, lw_weight(N), nullptr);
    // the linear parts of F̃: those of Ũ, up to the factor the last stencil puts on them
    constexpr double miss = lw_weight(N) * (1.0 - time_diff<N>(N).linear);
    ns_join(sum, fma(-miss, w[1], Uc[1]), fma(-miss, w[2], Uc[2]), F, G);
    __syncthreads();  // every thread has finished reading s2 before it is reused
    if constexpr (CURV) {
        double Fc[4], Gc[4];
        to_contravariant(Jn, F, G, Fc, Gc);
        if (act) put8<S>(s2, sidx, Fc, Gc);
    } else {
        if (act) put8<S>(s2, sidx, F, G);
    }
    __syncthreads();
    contract<n, S>(s2, sbase, i, j, sDh, vol);
    if (terr) {
        // temporal error of kernel 4 (dg_2d_parabolic.jl:1749-1775, 1841-1855): as in
        // lw_element, with the total F̃ and f_tttt
        double a1[4], a2[4];
        contract<n, S>(s2, sbase, i, j, sD, a1);  // D F̃
        contract<n, S>(s0, sbase, i, j, sD, a2);  // D f_tttt
        double e = 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double d = sc * ((1.0 / 120.0) * a2[v]);
            const double hi = fma(sc, a1[v], uN[v]);
            const double lo = hi - d;
            const double r = d / (abstol + reltol * dmax(fabs(hi), fabs(lo)));
            e = fma(r, r, e);
        }
        *terr = e;
        __syncthreads();  // s0 is reused for the face records
    }
}

// acc += weight · f_t of the states w ± wt, w ± 2wt (and their gradients) for
// the MDRK stages (the five ns_q sums; the mass fluxes' part of f_t is ut);
// WALL: also f_t of components 1..3 of the viscous fluxes in v6 (x, then y)
template <bool WALL = false>
__device__ __forceinline__ void mdrkp_ft(const double* u, const double* ut, const double* gx, const double* gtx,
                                         const double* gy, const double* gty, double gm1, DevC c, double weight,
                                         double* acc, double* v6 = nullptr) {
    constexpr TimeDiff td = time_diff<4>(1);
    double d[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, a6[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    constexpr int kUnroll = WALL ? 1 : 4;  // the wall kernels spill the interleaved states
#pragma unroll kUnroll
    for (int r = 0; r < 4; ++r) {
        // the states u + 2ut, u + ut, u - ut, u - 2ut (selects, as the loop may stay one)
        const double off = r == 0 ? 2.0 : r == 1 ? 1.0 : r == 2 ? -1.0 : -2.0;
        const double ck = r == 0 ? td.c[2] : r == 1 ? td.c[0] : r == 2 ? td.c[1] : td.c[3];
        double s[4], sx[4], sy[4], q[5];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            s[v] = fma(off, ut[v], u[v]);
            sx[v] = fma(off, gtx[v], gx[v]);
            sy[v] = fma(off, gty[v], gy[v]);
        }
        ns_q(s, sx, sy, gm1, c, q);
#pragma unroll
        for (int m = 0; m < 5; ++m) d[m] = fma(ck, q[m], d[m]);
        if constexpr (WALL) {
            double fx[4], fy[4];
            ns_visc_fluxes(s, sx, sy, gm1, c, fx, fy);
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                a6[m] = fma(ck, fx[1 + m], a6[m]);
                a6[3 + m] = fma(ck, fy[1 + m], a6[3 + m]);
            }
        }
    }
#pragma unroll
    for (int m = 0; m < 5; ++m) acc[m] = fma(weight * td.scale, d[m], acc[m]);
    if constexpr (WALL) {
#pragma unroll
        for (int m = 0; m < 6; ++m) v6[m] = a6[m] * td.scale;
    }
}

// No-slip walls: the wall records of a face node, wq[o] (o = 0: its x face,
// 1: its y face; null where that face is no wall), take the time average of
// components 1..3 of the viscous flux in the face's orientation: q = w·v6
// (first term) or q += w·v6.  Only wall lanes touch memory.
__device__ __forceinline__ void wall_acc(double* const* wq, double w, const double* v6, bool first) {
#pragma unroll
    for (int o = 0; o < 2; ++o) {
        double* q = wq[o];
        if (!q) continue;
#pragma unroll
        for (int k = 0; k < 3; ++k) q[k] = first ? w * v6[3 * o + k] : fma(w, v6[3 * o + k], q[k]);
    }
}
// components 1..3 of the viscous fluxes of a wall face node's state into its
// wall records with weight w (the first term of the average)
__device__ __forceinline__ void wall_first(double* const* wq, double w, const double* u, const double* gx,
                                           const double* gy, double gm1, DevC c) {
    if (!wq[0] && !wq[1]) return;
    double fx[4], fy[4], v6[6];
    ns_visc_fluxes(u, gx, gy, gm1, c, fx, fy);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        v6[k] = fx[1 + k];
        v6[3 + k] = fy[1 + k];
    }
    wall_acc(wq, w, v6, true);
}

// mdrk_kernel_1! with viscous terms (multi_derivative_2d_parabolic.jl:221-464):
// F̃ = f/2 + f_t/8, Ũ = u/2 + ut/8 on the total flux.  WALL: the wall records
// of the node take the stage's viscous average f_v/2 + f_v,t/8 (the Fv the
// reference's prolong2boundaries_visc_lw! reads).  With the Navier-Stokes
// convergence source (has_src; 290-300, 380-392, 441-446): ut += dt s(t) before
// its gradient, and Ssrc = s/2 + s_t/8 for the residual.
template <int N, int EB, bool CURV = false, bool WALL = false>
__device__ __forceinline__ void mdrkp1_element(const double* uN, const double* gxN, const double* gyN, double invJ,
                                               double sc, double gm1, DevC c, int i, int j, bool act, int sidx,
                                               int sbase, double* s0, double* s1, double* s2, const double* sD,
                                               const double* sDh, double* Uc, double* F,
                                               double* G, double* vol, const double* Jn = nullptr,
                                               double* const* wq = nullptr, bool has_src = false,
                                               const NsSrcPt& sp = NsSrcPt{}, double dt = 0.0,
                                               double* Ssrc = nullptr) {
    using G_ = VGeo<N, EB>;
    constexpr int n = G_::n, S = G_::S;
    double f[4], g[4], q[5];
    ns_q(uN, gxN, gyN, gm1, c, q);
    ns_join(q, uN[1], uN[2], f, g);
    if constexpr (WALL) wall_first(wq, 0.5, uN, gxN, gyN, gm1, c);
    double ut[4], utx[4], uty[4];
    if (has_src) {
        double s[4], st[4], ds[4];
        ns_src_eval(sp, 0.0, s);
        ns_src_t5(sp, dt, st);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            ds[v] = dt * s[v];
            Ssrc[v] = fma(0.125, st[v], 0.5 * s[v]);
        }
        par_level<N, EB, CURV>(act, sidx, sbase, i, j, invJ, sc, s0, s2, sD, f, g, ut, utx, uty, Jn, ds);
    } else {
        par_level<N, EB, CURV>(act, sidx, sbase, i, j, invJ, sc, s0, s2, sD, f, g, ut, utx, uty, Jn);
    }
#pragma unroll
    for (int m = 0; m < 5; ++m) q[m] *= 0.5;
    if constexpr (WALL) {
        double v6[6];
        mdrkp_ft<true>(uN, ut, gxN, utx, gyN, uty, gm1, c, 0.125, q, v6);
        wall_acc(wq, 0.125, v6, false);
    } else {
        mdrkp_ft(uN, ut, gxN, utx, gyN, uty, gm1, c, 0.125, q);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) Uc[v] = fma(0.125, ut[v], 0.5 * uN[v]);
    ns_join(q, Uc[1], Uc[2], F, G);
    __syncthreads();  // every thread has finished reading s2 before it is reused
    if constexpr (CURV) {
        double Fc[4], Gc[4];
        to_contravariant(Jn, F, G, Fc, Gc);
        if (act) put8<S>(s2, sidx, Fc, Gc);
    } else {
        if (act) put8<S>(s2, sidx, F, G);
    }
    __syncthreads();
    contract<n, S>(s2, sbase, i, j, sDh, vol);
}

// mdrk_kernel_2! with viscous terms (multi_derivative_2d_parabolic.jl:506-711):
// F̃ = F2 + f_t(us)/3, Ũ = U2 + ust/3, with F2 = f + f_t/6 and U2 = u + ut/6
// recomputed from uⁿ and its BR1 gradient.  WALL: the wall records take the
// stage's viscous average f_v + f_v,t/6 + f_v,t(us)/3.  With the Navier-Stokes
// convergence source (has_src; 576-601, 668-674): ut and ust both += dt s(t)
// before their gradients (the reference evaluates stage 2's source at the
// call's t), Ssrc = S2 + s_t/3 with S2 = s + s_t/6.
template <int N, int EB, bool CURV = false, bool WALL = false>
__device__ __forceinline__ void mdrkp2_element(const double* uN, const double* gxN, const double* gyN,
                                               const double* usn, const double* gxS, const double* gyS,
                                               double invJ, double sc, double gm1, DevC c, int i, int j, bool act,
                                               int sidx, int sbase, double* s0, double* s1, double* s2,
                                               const double* sD, const double* sDh, double* Uc,
                                               double* F, double* G, double* vol, const double* Jn = nullptr,
                                               double* const* wq = nullptr, bool has_src = false,
                                               const NsSrcPt& sp = NsSrcPt{}, double dt = 0.0,
                                               double* Ssrc = nullptr) {
    using G_ = VGeo<N, EB>;
    constexpr int n = G_::n, S = G_::S;
    double f[4], g[4], fs[4], gs[4], q[5], qs[5];
    ns_q(uN, gxN, gyN, gm1, c, q);
    ns_join(q, uN[1], uN[2], f, g);
    if constexpr (WALL) wall_first(wq, 1.0, uN, gxN, gyN, gm1, c);
    ns_q(usn, gxS, gyS, gm1, c, qs);
    ns_join(qs, usn[1], usn[2], fs, gs);
    if constexpr (CURV) {
        double cx[4], cy[4];
        to_contravariant(Jn, f, g, cx, cy);
        if (act) put8<S>(s0, sidx, cx, cy);
        to_contravariant(Jn, fs, gs, cx, cy);
        if (act) put8<S>(s1, sidx, cx, cy);
    } else if (act) {
        put8<S>(s0, sidx, f, g);
        put8<S>(s1, sidx, fs, gs);
    }
    __syncthreads();
    double ut[4], ust[4];
    contract<n, S>(s0, sbase, i, j, sD, ut);
    contract<n, S>(s1, sbase, i, j, sD, ust);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        ut[v] *= sc;
        ust[v] *= sc;
    }
    if (has_src) {
        double s[4], st[4];
        ns_src_eval(sp, 0.0, s);
        ns_src_t5(sp, dt, st);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            ut[v] = fma(dt, s[v], ut[v]);
            ust[v] = fma(dt, s[v], ust[v]);
            Ssrc[v] = fma(1.0 / 3.0, st[v], fma(1.0 / 6.0, st[v], s[v]));
        }
    }
    if (act) {
        put4<S>(s2, sidx, ut);
        put4<S>(s2 + 4 * S, sidx, ust);
    }
    __syncthreads();
    double utx[4], uty[4], stx[4], sty[4];
    contract_xy<n, S>(s2, sbase, i, j, sD, utx, uty);
    contract_xy<n, S>(s2 + 4 * S, sbase, i, j, sD, stx, sty);
    if constexpr (CURV) {
        grad_to_cartesian(Jn, invJ, utx, uty);
        grad_to_cartesian(Jn, invJ, stx, sty);
    } else {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            utx[v] *= invJ;
            uty[v] *= invJ;
            stx[v] *= invJ;
            sty[v] *= invJ;
        }
    }
    if constexpr (WALL) {
        double v6[6];
        mdrkp_ft<true>(uN, ut, gxN, utx, gyN, uty, gm1, c, 1.0 / 6.0, q, v6);
        wall_acc(wq, 1.0 / 6.0, v6, false);
        mdrkp_ft<true>(usn, ust, gxS, stx, gyS, sty, gm1, c, 1.0 / 3.0, q, v6);
        wall_acc(wq, 1.0 / 3.0, v6, false);
    } else {
        mdrkp_ft(uN, ut, gxN, utx, gyN, uty, gm1, c, 1.0 / 6.0, q);
        mdrkp_ft(usn, ust, gxS, stx, gyS, sty, gm1, c, 1.0 / 3.0, q);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) Uc[v] = fma(1.0 / 3.0, ust[v], fma(1.0 / 6.0, ut[v], uN[v]));
    ns_join(q, Uc[1], Uc[2], F, G);
    __syncthreads();  // every thread has finished reading s2 before it is reused
    if constexpr (CURV) {
        double Fc[4], Gc[4];
        to_contravariant(Jn, F, G, Fc, Gc);
        if (act) put8<S>(s2, sidx, Fc, Gc);
    } else {
        if (act) put8<S>(s2, sidx, F, G);
    }
    __syncthreads();
    contract<n, S>(s2, sbase, i, j, sDh, vol);
}

// Curvilinear CFL speeds of a node (Trixi max_dt for curvilinear meshes): the
// speeds transformed to the reference element, |Ja^k · (λ1, λ2)| |J⁻¹|.
__device__ __forceinline__ void curved_speeds(const double* u, const double* J, double invJ, double gamma, double& m1,
                                              double& m2, bool& bad) {
    double l1, l2;
    node_speeds(u, gamma, l1, l2, bad);
    const double aj = fabs(invJ);
    m1 = fabs(fma(J[0], l1, J[1] * l2)) * aj;
    m2 = fabs(fma(J[2], l1, J[3] * l2)) * aj;
}

// ---------------------------------------------------------------------------
// Volume kernel: element computation, then the interfaces inside the
// workgroup, the lifted surface terms (weak form, ℓ̂ = 1/w at the end nodes),
// the Jacobian and the update.  Faces leaving the workgroup write their face
// record for the surface kernel.  The CFL reduction of a step is left to the
// surface kernel, which reads every node once after its corrections (a
// reduction here costs barriers and LDS passes worth 15% of this kernel).
// Waves per SIMD the register budget is sized for: 3 (168 VGPRs) for the
// plain scheme (TLW_VOL_WAVES at build time); 2 (256 VGPRs) with shock
// capturing, which takes 157 on a TreeMesh (and so runs 3 waves all the same)
// but 172 on a curvilinear mesh, and with source terms (the source's time
// differences at every stage).
#ifndef TLW_VOL_WAVES
#define TLW_VOL_WAVES 3
#endif
template <bool TWO> constexpr int kVolWaves = TWO ? 2 : TLW_VOL_WAVES;
template <bool SC, bool PAR> constexpr bool vol_two_buffers = !SC && !PAR;

// pure_and_blended_element_ids!: an element without subcell FV
__device__ __forceinline__ bool pure_dg(double alpha) { return fabs(alpha) <= 1e-12; }

// What a lane of a volume workgroup reads of its tile before the element procedure.
template <bool CURV, bool US> struct TileIn {
    double u[4];               // uⁿ of the lane's node
    double us[US ? 4 : 1];     // the MDRK stage state
    double J[CURV ? 4 : 1];    // Ja11, Ja12, Ja21, Ja22 of the node
    double invJ;               // per element on a TreeMesh, per node on a curvilinear mesh
    int nbx, nby;              // neighbours across the node's x and y face (where it lies on one)
    int slot;                  // neighbour across the lane's face slot (element, face, node)
};

// PAR: hyperbolic-parabolic (compressible Navier-Stokes) element procedures,
// same register budget as shock capturing.
// One tile (blk) of a's table, number bid, with its LDS: lds [G_::LDS2 or LDS],
// sDh and sD [G_::M] (D̂ and D, rows of G_::MS) and s_alpha [EB + 1] (smoothed
// blending factors, and whether any of them blends).
template <int N, int EB, int KIND, bool SC, bool PAR, bool CURV>
__device__ __forceinline__ void volume_tile(const KArgs& a, int bid, const int4& blk,
                                            const TileIn<CURV, vol_base(KIND) == VOL_MDRK2>& in, double* lds,
                                            double* sDh, double* sD, double* s_alpha) {
    static_assert(!(SC && PAR), "shock capturing has no hyperbolic-parabolic form");
    static_assert(!CURV || !PAR || KIND != VOL_LW_ADAPT, "adaptive steps: Euler LW, or Navier-Stokes LW on a TreeMesh");
    static_assert(!PAR || vol_base(KIND) != VOL_LW_ADAPT || N == 4, "the parabolic temporal error is kernel 4's");
    static_assert(!vol_is_wall(KIND) || (PAR && !CURV && !SC), "walls: the TreeMesh Navier-Stokes kernels");
    static_assert(!(CURV && PAR && SC), "no shock capturing with parabolic terms");
    using G_ = VGeo<N, EB>;
    constexpr int n = G_::n, NN = G_::NN, S = G_::S, NT = G_::NT;
    // The plain Euler kernels exchange through two buffers: F̃ last in the first of
    // them, where the interface fluxes go later, and the face records in the
    // second.  Shock capturing and the Navier-Stokes kernels use three: s2 takes F̃;
    // then s0 and s1 the records and s2 the interface fluxes, or with shock capturing
    // s1 and s2 the records and s0, which holds uⁿ before, the fluxes.
    constexpr bool TWO = vol_two_buffers<SC, PAR>;
    double* s0 = lds;
    double* s1 = lds + 8 * S;
    double* s2 = TWO ? lds : lds + 16 * S;
    constexpr int KB = vol_base(KIND);
    // (A, B) of the element procedures, whose last exchange goes to s2
    constexpr bool last_is_a = KB == VOL_MDRK2 || (N == 4 && (KB == VOL_LW || KB == VOL_LW_ADAPT));
    double* bufA = last_is_a ? s2 : s1;
    double* bufB = last_is_a ? s1 : s2;
    const DevS st = dev_state(a.st + blk.z);
    if (a.use_state_dt && st->finished) return;
    const int tid = threadIdx.x;
    if constexpr (SC) {
        // the tile's blending factors, smoothed over the face neighbours (Trixi
        // apply_smoothing!), by one lane an element of the first wave: read early,
        // and published by the first barrier of the element procedure
        static_assert(EB < 64, "one wave's lanes");
        if (tid < 64) {
            double al = 0.0;
            if (tid < blk.y) {
                const int es = blk.x + tid;
                al = a.alpha_tmp[es];
                if (dev_const(a.c)->alpha_smooth) {
                    const int4 nb = *reinterpret_cast<const int4*>(a.nbr + 4 * es);
                    if (nb.x >= 0) al = dmax(al, 0.5 * a.alpha_tmp[nb.x]);
                    if (nb.y >= 0) al = dmax(al, 0.5 * a.alpha_tmp[nb.y]);
                    if (nb.z >= 0) al = dmax(al, 0.5 * a.alpha_tmp[nb.z]);
                    if (nb.w >= 0) al = dmax(al, 0.5 * a.alpha_tmp[nb.w]);
                }
                s_alpha[tid] = al;
                if (a.alpha_out) a.alpha_out[es] = al;
            }
            const bool any = __any(!pure_dg(al));
            if (tid == 0) s_alpha[EB] = any ? 1.0 : 0.0;
        }
    }
    const int le = tid / NN, node = tid - (tid / NN) * NN;
    const int i = node % n, j = node / n;
    const int e0 = blk.x;
    const int nel = blk.y;
    const bool act = le < nel;
    const int lec = le < nel ? le : nel - 1;
    const int e = e0 + lec;
    const int sidx = lec * NN + node, sbase = lec * NN;
    const int cur = a.use_state_dt ? st->cur : 0;
    const double* uin = sel_in(a, cur);
    double* out = sel_out(a, cur);
    const double dt = a.use_state_dt ? st->dt : a.dt_arg;
    const DevC c = dev_const(a.c);
    const double gamma = c->gamma, gm1 = gamma - 1.0;
    const double invJ = in.invJ;
    const double sc = -dt * invJ;
    const size_t off = ((size_t)e * NN + node) * 4;
    // source terms: separate instantiations (KIND = VOL_LW_SRC + the plain kind);
    // the node's coordinates from the element's centre and edge length, the
    // time of the call; Ssrc = S, added to the residual at the end
    constexpr bool SRC = vol_is_src(KIND);
    constexpr bool WALL = vol_is_wall(KIND);
    static_assert(!SRC || (!SC && !PAR), "source terms: the Euler kernels");
    double Ssrc[4] = {0.0, 0.0, 0.0, 0.0};
    SrcPt sp{0.0, 0.0, 0.0, gamma};
    if constexpr (SRC && CURV) {  // the node's coordinates of the curvilinear mesh
        sp.x = a.nxy[((size_t)e * NN + node) * 2];
        sp.y = a.nxy[((size_t)e * NN + node) * 2 + 1];
        sp.t = a.use_state_dt ? st->t : a.t_arg;
    } else if constexpr (SRC) {
        const double hh = 0.5 * a.length[e];
        sp.x = a.center[2 * e] + hh * c->nodes[i];
        sp.y = a.center[2 * e + 1] + hh * c->nodes[j];
        sp.t = a.use_state_dt ? st->t : a.t_arg;
    }

    double Uc[4], F[4], G[4], vol[4];
    double terr = 0.0;  // temporal error of the node (adaptive steps, LW N=4)
    const double* uN = in.u;
    const double* Jn = in.J;
    // walls: the node's wall records (its x face, its y face; null where that face is no wall)
    double* wq[2] = {nullptr, nullptr};
    if constexpr (WALL) {
        const int wfx = (i == 0) ? 0 : ((i == n - 1) ? 1 : -1), wfy = (j == 0) ? 2 : ((j == n - 1) ? 3 : -1);
        if (act && wfx >= 0 && in.nbx == -1) wq[0] = a.fvb + (((size_t)e * 4 + wfx) * n + j) * 6;
        if (act && wfy >= 0 && in.nby == -1) wq[1] = a.fvb + (((size_t)e * 4 + wfy) * n + i) * 6;
    }
    if constexpr (!PAR) {
        const bool adapt = KB == VOL_LW_ADAPT;
        if constexpr (KB == VOL_LW || KB == VOL_LW_ADAPT) {
            lw_element<N, EB, CURV, false, SRC>(uN, Jn, dt, sc, gamma, i, j, act, sidx, sbase, bufA, bufB, sD, sDh,
                                                Uc, F, G, vol, nullptr, adapt ? &terr : nullptr,
                                                adapt ? st->abstol : 0.0, adapt ? st->reltol : 0.0, &sp, Ssrc);
        } else if constexpr (KB == VOL_MDRK1) {
            mdrk1_element<N, EB, CURV, SRC>(uN, Jn, dt, sc, gamma, i, j, act, sidx, sbase, bufA, bufB, sD, sDh, Uc,
                                            F, G, vol, &sp, Ssrc);
        } else {
            mdrk2_element<N, EB, CURV, SRC>(uN, in.us, Jn, dt, sc, gamma, i, j, act, sidx, sbase, bufA, bufB, sD,
                                            sDh, Uc, F, G, vol, &sp, Ssrc);
        }
    } else if constexpr (PAR) {
        // BR1 gradients of uⁿ (and of us in MDRK stage 2), exchanged through a
        // buffer the element procedure writes only after its first barrier
        double* sg = (KB == VOL_MDRK2) ? s2 : s1;
        double gxN[4], gyN[4];
        if (act) put4<S>(sg, sidx, uN);
        // the Navier-Stokes convergence source (MDRK on the TreeMesh): the node's
        // spatial factors once, at the call's t
        NsSrcPt nsp{};
        bool nsrc = false;
        if constexpr (!CURV && (KB == VOL_MDRK1 || KB == VOL_MDRK2 || (WALL && KB == VOL_LW))) {
            nsrc = c->src_kind == SRC_NS_CONVERGENCE_TEST;
            if (nsrc) {
                const double hh = 0.5 * a.length[e];
                nsp = ns_src_point(a.center[2 * e] + hh * c->nodes[i], a.center[2 * e + 1] + hh * c->nodes[j],
                                   a.use_state_dt ? st->t : a.t_arg, c);
            }
        }
        if constexpr (KB == VOL_MDRK2) {
            const double* usn = in.us;
            double gxS[4], gyS[4];
            if (act) put4<S>(sg + 4 * S, sidx, usn);
            __syncthreads();
            br1_gradient<N, EB, CURV>(sg, uin, in.nbx, in.nby, c, i, j, sbase, invJ, sDh, uN, gxN, gyN, Jn);
            br1_gradient<N, EB, CURV>(sg + 4 * S, a.us, in.nbx, in.nby, c, i, j, sbase, invJ, sDh, usn, gxS, gyS, Jn);
            mdrkp2_element<N, EB, CURV, WALL>(uN, gxN, gyN, usn, gxS, gyS, invJ, sc, gm1, c, i, j, act, sidx, sbase, s0,
                                              s1, s2, sD, sDh, Uc, F, G, vol, Jn, wq, nsrc, nsp, dt, Ssrc);
        } else {
            __syncthreads();
            br1_gradient<N, EB, CURV>(sg, uin, in.nbx, in.nby, c, i, j, sbase, invJ, sDh, uN, gxN, gyN, Jn);
            if constexpr (KB == VOL_LW)
                lwp_element<N, EB, CURV, WALL>(uN, gxN, gyN, invJ, sc, gm1, c, i, j, act, sidx, sbase, s0, s1, s2, sD,
                                               sDh, Uc, F, G, vol, Jn, wq, nullptr, 0.0, 0.0, nsrc, nsp, Ssrc,
                                               dt);
            else if constexpr (KB == VOL_LW_ADAPT)
                lwp_element<N, EB, CURV, WALL>(uN, gxN, gyN, invJ, sc, gm1, c, i, j, act, sidx, sbase, s0, s1, s2, sD,
                                               sDh, Uc, F, G, vol, Jn, wq, &terr, st->abstol, st->reltol);
            else
                mdrkp1_element<N, EB, CURV, WALL>(uN, gxN, gyN, invJ, sc, gm1, c, i, j, act, sidx, sbase, s0, s1, s2, sD,
                                                  sDh, Uc, F, G, vol, Jn, wq, nsrc, nsp, dt, Ssrc);
        }
    }
    if (act && a.auxU) {
        store4(a.auxU + off, Uc);
        store4(a.auxF + ((size_t)e * NN + node) * 8, F);
        store4(a.auxF + ((size_t)e * NN + node) * 8 + 4, G);
    }

    const int fx = (i == 0) ? 0 : ((i == n - 1) ? 1 : -1);
    const int fy = (j == 0) ? 2 : ((j == n - 1) ? 3 : -1);
    constexpr int RQ = kRQ<SC>;
    double fnlx[4] = {0, 0, 0, 0}, fnly[4] = {0, 0, 0, 0};
    double alpha_e = 0.0;
    bool subcells = false;  // the workgroup has a blended element
    if constexpr (SC) {
        // Away from shocks a workgroup has no blended element, and what is left of
        // the subcell FV is one Rusanov flux a face node (below) in place of two a
        // node and two barriers fewer.  256², N=4, tile 10, one workgroup in ten
        // blended: 168 us (234 VGPRs) with the subcell FV of every element and the
        // blending factors read here, now 130 (157 VGPRs).
        alpha_e = s_alpha[lec];
        subcells = __builtin_amdgcn_readfirstlane(s_alpha[EB] != 0.0);
        if (subcells) {
            const bool blended = !pure_dg(alpha_e);
            // subcell FV (fv_kernel!, dg_2d.jl:251-324): Rusanov fluxes between the
            // face values of neighbouring subcells, zero at the element faces.  First
            // order (Trixi calcflux_fv!): the face values are the node values.  A
            // blended element away from the domain boundary with MUSCL-Hancock takes
            // the reconstructed, half-step-evolved face values (mh_faces).
            if (act) put4<S>(s1, sidx, uN);
            __syncthreads();
            double ql[4], qr[4], qd[4], qu[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) ql[v] = qr[v] = qd[v] = qu[v] = uN[v];
            if (!CURV && c->recon == 1 && blended && a.nbr[4 * e] >= 0 && a.nbr[4 * e + 1] >= 0 && a.nbr[4 * e + 2] >= 0 &&
                a.nbr[4 * e + 3] >= 0) {
                const double dtmh = (KIND == VOL_MDRK1) ? 0.5 * dt : dt;  // tree/multi_derivative_2d.jl:199
                mh_faces<N, S>(s1, sidx, i, j, uN, c, 2.0 - alpha_e, dtmh, invJ, gm1, ql, qr, qd, qu);
            }
            // the right and upper face values go to the neighbouring subcells
            if (act) put8<S>(s0, sidx, qr, qu);
            __syncthreads();
            double fxl[4] = {0, 0, 0, 0}, gyl[4] = {0, 0, 0, 0}, w[4];
            if (i > 0) {
                get4<S>(s0, sidx - 1, w);
                if constexpr (CURV) {
                    // Trixi's subcell normal, or for a pure-DG element at subcell face n-1 the
                    // normal of the reference's calc_fn_low! (structured/dg_2d.jl:111-173)
                    const double* nq = (!blended && i == n - 1) ? a.sqrk + ((size_t)e * n + j) * 4
                                                                 : a.snrm + ((size_t)e * NN + node) * 4;
                    rusanov_normal(w, ql, gamma, nq[0], nq[1], sqrt(fma(nq[0], nq[0], nq[1] * nq[1])), fxl);
                } else {
                    rusanov(w, ql, gamma, 1, fxl);
                }
            }
            if (j > 0) {
                get4<S>(s0 + 4 * S, sidx - n, w);
                if constexpr (CURV) {
                    const double* nq = (!blended && j == n - 1) ? a.sqrk + ((size_t)e * n + i) * 4 + 2
                                                                 : a.snrm + ((size_t)e * NN + node) * 4 + 2;
                    rusanov_normal(w, qd, gamma, nq[0], nq[1], sqrt(fma(nq[0], nq[0], nq[1] * nq[1])), gyl);
                } else {
                    rusanov(w, qd, gamma, 2, gyl);
                }
            }
            if (act) put8<S>(s2, sidx, fxl, gyl);
            __syncthreads();
            const double iwi = 1.0 / c->weights[i], iwj = 1.0 / c->weights[j];
            double fxr4[4] = {0.0, 0.0, 0.0, 0.0}, gyr4[4] = {0.0, 0.0, 0.0, 0.0};
            if (i < n - 1) get4<S>(s2, sidx + 1, fxr4);
            if (j < n - 1) get4<S>(s2 + 4 * S, sidx + n, gyr4);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const double fxr = fxr4[v], gyr = gyr4[v];
                const double fv = iwi * (fxr - fxl[v]) + iwj * (gyr - gyl[v]);
                vol[v] = (1.0 - alpha_e) * vol[v] + (blended ? alpha_e * fv : 0.0);
                // fn_low: the subcell fluxes next to the element faces (load_fn_low!)
                fnlx[v] = (fx == 0) ? fxr : fxl[v];
                fnly[v] = (fy == 2) ? gyr : gyl[v];
            }
            __syncthreads();  // s1 and s2 are reused for the face records
        } else {
            if (act) put4<S>(s0, sidx, uN);
            __syncthreads();
#pragma unroll
            for (int v = 0; v < 4; ++v) vol[v] = (1.0 - alpha_e) * vol[v];
        }
    }
    // --- face records into LDS (s0, s1 are free), one per face the node lies on.
    // λ ingredients: |v1|, |v2| and c of the λ state, once per node.
    double* rec = (TWO || SC) ? s1 : lds;  // [EB][4][n][RQ]
    const bool tree = c->flux_order == 0;
    const double* jump = tree ? uN : Uc;
    const double* lamst = tree ? Uc : uN;
    const int nbx = in.nbx, nby = in.nby;
    constexpr int NSLOT = EB * 4 * n;
    static_assert(NSLOT <= NT, "one face slot per lane");
    constexpr int FN = CURV ? 12 : 10;  // fn_low in a record: variables [FN, FN + 4)
    auto put_face = [&](int f, int l, const double* r) {
        const int slot = (lec * 4 + f) * n + l;
        if constexpr (SC) {
            put_record<RQ, 0, FN / 2>(rec, slot, r);
            if (subcells) put_record<RQ, FN / 2, FN / 2 + 2>(rec, slot, r);
            put_record<RQ, FN / 2 + 2>(rec, slot, r);
        } else {
            put_record<RQ>(rec, slot, r);
        }
    };
    if constexpr (SC) {
        // without a blended element only fn_low is left of the subcell FV: the flux
        // between the face's node and the next one inwards, by the lane of the slot
        if (!subcells && tid < NSLOT && tid / (4 * n) < nel) {
            const int ls = tid / (4 * n), f = (tid / n) % 4, l = tid % n;
            const int k = (f & 1) ? n - 1 : 1;  // upper node of the two, along the face's direction
            const int hi = (f < 2) ? l * n + k : k * n + l;
            double ul[4], ur[4], r[RQ];
            get4<S>(s0, ls * NN + hi - (f < 2 ? 1 : n), ul);
            get4<S>(s0, ls * NN + hi, ur);
            if constexpr (CURV) {
                const size_t es = e0 + ls;
                const double* nq = ((f & 1) ? a.sqrk + (es * n + l) * 4 : a.snrm + (es * NN + hi) * 4) + (f < 2 ? 0 : 2);
                rusanov_normal(ul, ur, gamma, nq[0], nq[1], sqrt(fma(nq[0], nq[0], nq[1] * nq[1])), r + FN);
            } else {
                rusanov(ul, ur, gamma, f < 2 ? 1 : 2, r + FN);
            }
            put_record<RQ, FN / 2, FN / 2 + 2>(rec, tid, r);
        }
    }
    if constexpr (CURV) {
        // structured order with the interface's normal n (shared by both
        // elements): F̃·n, |v(uⁿ)·n| and c(uⁿ)|n| (dg_2d.jl:2229-2264)
        const double ir = rcp_nr(uN[0]);
        const double v1 = uN[1] * ir, v2 = uN[2] * ir;
        const double p = gm1 * (uN[3] - 0.5 * (uN[1] * v1 + uN[2] * v2));
        const double cs = sqrt_gs(gamma * p * ir);
        // (a domain-boundary face is rewritten to the TreeMesh order of the
        // Dirichlet call by the surface kernel, which has uⁿ at hand)
        // with shock capturing: Ũ, F̃·n, uⁿ and fn_low (face_numflux_sc_curved)
        auto face = [&](int f, int l, const double* fnl) {
            double nf[4], Fn[4], r[RQ];
            load4(a.fnorm + (((size_t)e * 4 + f) * n + l) * 4, nf);
#pragma unroll
            for (int v = 0; v < 4; ++v) Fn[v] = fma(F[v], nf[0], G[v] * nf[1]);
            if constexpr (SC) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    r[v] = Uc[v];
                    r[4 + v] = Fn[v];
                    r[8 + v] = uN[v];
                    r[12 + v] = fnl[v];
                }
            } else {
                make_record(r, Uc, Fn, fabs(fma(v1, nf[0], v2 * nf[1])), cs * nf[2]);
            }
            put_face(f, l, r);
        };
        if (act && fx >= 0) face(fx, j, fnlx);
        if (act && fy >= 0) face(fy, i, fnly);
    } else {
        double av1, av2, cs;
        speed_parts2(lamst, gamma, av1, av2, cs);
        auto fill = [&](double* r, const double* fnl) {
            if constexpr (SC) {
#pragma unroll
                for (int v = 0; v < 4; ++v) r[10 + v] = fnl[v];
                r[14] = alpha_e;
                r[15] = 0.0;
            }
        };
        if (act && fx >= 0) {
            double r[RQ];
            make_record(r, jump, F, av1, cs);
            fill(r, fnlx);
            put_face(fx, j, r);
            if (nbx <= -2) mortar_side(a, nbx, n, j, jump, F, lamst);
        }
        if (act && fy >= 0) {
            double r[RQ];
            make_record(r, jump, G, av2, cs);
            fill(r, fnly);
            put_face(fy, i, r);
            if (nby <= -2) mortar_side(a, nby, n, i, jump, G, lamst);
        }
    }
    __syncthreads();
    // --- one lane per face slot (element, face, node).  An interface inside the
    // workgroup is evaluated once, by the slot of its left element's + face, and
    // its flux goes to both adjacent nodes (accx for x faces, accy for y faces);
    // the record of a face leaving the workgroup goes to HBM for the surface kernel.
    double* accx = SC ? s0 : s2;  // pairs of variables (put4); free after the last contraction
    double* accy = accx + 4 * S;
    static_assert(TWO || EB * 4 * n * RQ <= 16 * S, "records fit in two buffers");
    if (tid < NSLOT) {
        const int ls = tid / (4 * n), f = (tid / n) % 4, l = tid % n;
        if (ls < nel) {
            const int es = e0 + ls;
            const int ne = in.slot;
            if (!(ne >= e0 && ne < e0 + nel)) {
                double r[RQ];
                get_record<RQ>(rec, tid, r);
                store_record<RQ>(a.trace + ((size_t)es * 4 * n + f * n + l) * RQ, r);
            } else if (f & 1) {
                double Lr[RQ], Rr[RQ], Fs[4];
                get_record<RQ>(rec, tid, Lr);
                get_record<RQ>(rec, ((ne - e0) * 4 + (f ^ 1)) * n + l, Rr);
                // + face of ls: node (n-1, l) or (l, n-1); - face of ne: node (0, l) or (l, 0)
                const int nodeL = (f == 1) ? l * n + (n - 1) : (n - 1) * n + l;
                const int nodeR = (f == 1) ? l * n : l;
                if constexpr (SC && CURV) {
                    double nf[4];
                    load4(a.fnorm + (((size_t)es * 4 + f) * n + l) * 4, nf);
                    face_numflux_sc_curved(Lr, Rr, nf, a.ijn[(size_t)es * NN + nodeL], a.ijn[(size_t)ne * NN + nodeR],
                                           s_alpha[ls], s_alpha[ne - e0], gamma, dt, c->weights[n - 1], c->weights[0],
                                           Fs);
                } else if constexpr (SC) {
                    face_numflux_sc(Lr, Rr, f < 2 ? 1 : 2, gamma, st->invJ0, dt, c->weights[n - 1], c->weights[0], Fs);
                } else {
                    face_numflux(Lr, Rr, Fs);
                }
                double* acc = (f == 1) ? accx : accy;
                put4<S>(acc, ls * NN + nodeL, Fs);
                put4<S>(acc, (ne - e0) * NN + nodeR, Fs);
            }
        }
    }
    __syncthreads();
    // --- lifted internal fluxes, Jacobian, output
    const bool intx = fx >= 0 && nbx >= e0 && nbx < e0 + nel;
    const bool inty = fy >= 0 && nby >= e0 && nby < e0 + nel;
    double surf[4] = {0.0, 0.0, 0.0, 0.0};
    if (intx) {
        const double wf = (fx & 1) ? c->bnd_hi : -c->bnd_lo;
        double Fs[4];
        get4<S>(accx, sidx, Fs);
#pragma unroll
        for (int v = 0; v < 4; ++v) surf[v] = Fs[v] * wf;
    }
    if (inty) {
        const double wf = (fy & 1) ? c->bnd_hi : -c->bnd_lo;
        double Fs[4];
        get4<S>(accy, sidx, Fs);
#pragma unroll
        for (int v = 0; v < 4; ++v) surf[v] = fma(Fs[v], wf, surf[v]);
    }
    // du = -J⁻¹ (vol + surf) + S, or u + dt du rounded once
    constexpr bool ADD_SRC =
        SRC || (PAR && !CURV && (KB == VOL_MDRK1 || KB == VOL_MDRK2 || (WALL && KB == VOL_LW)));
    const double fac = a.step_mode ? sc : -invJ;
    double val[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        val[v] = a.step_mode ? uN[v] : 0.0;
        if constexpr (ADD_SRC) val[v] = fma(a.step_mode ? dt : 1.0, Ssrc[v], val[v]);
        val[v] = fma(fac, vol[v] + surf[v], val[v]);
    }
    if (act) store4(out + off, val);
    if constexpr (KB == VOL_LW_ADAPT) {
        if (a.reduce != RED_ADAPT) return;
        // the workgroup's sum of its elements' temporal errors (adaptive.jl:48-64), in
        // the records' place: the interface fluxes may still be read by other lanes
        double* se = rec;
        double* rs = se + S;
        double* es = rs + EB * n;
        if (act) se[sidx] = terr;
        __syncthreads();
        if (act && i == 0) {
            double r = 0.0;
#pragma unroll
            for (int k = 0; k < n; ++k) r += se[sbase + j * n + k];
            rs[lec * n + j] = r;
        }
        __syncthreads();
        if (act && node == 0) {
            double r = 0.0;
#pragma unroll
            for (int k = 0; k < n; ++k) r += rs[lec * n + k];
            es[lec] = r;
        }
        __syncthreads();
        if (tid == 0) {
            double r = 0.0;
            for (int k = 0; k < nel; ++k) r += es[k];
            a.partial[bid] = r;
        }
    }
    // the CFL reduction of a step (and the admissibility test) is the surface
    // kernel's: it reads every node once after the last correction
}

// The volume workgroup `bid` of a's table.  The loads of a lane's tile data go
// out together at the start, the neighbours among them, which are first needed
// after the element procedure (the Navier-Stokes kernels: for the BR1 gradient).
template <int N, int EB, int KIND, bool SC, bool PAR, bool CURV>
__device__ __forceinline__ void volume_body(const KArgs& a, int bid, double* lds, double* sDh, double* sD,
                                            double* s_alpha) {
    using G_ = VGeo<N, EB>;
    constexpr int n = G_::n, NN = G_::NN, NSLOT = EB * 4 * n;
    const int4 blk = load_blk_at(a.vblk, bid);
    const int tid = threadIdx.x;
    const int le = tid / NN, node = tid - (tid / NN) * NN;
    const int i = node % n, j = node / n;
    const int lec = le < blk.y ? le : blk.y - 1;
    const int e = blk.x + lec;
    const size_t off = ((size_t)e * NN + node) * 4;
    TileIn<CURV, vol_base(KIND) == VOL_MDRK2> in;
    load4(sel_in(a, a.use_state_dt ? dev_state(a.st + blk.z)->cur : 0) + off, in.u);
    if constexpr (vol_base(KIND) == VOL_MDRK2) load4(a.us + off, in.us);
    if constexpr (CURV) load4(a.Ja + off, in.J);
    in.invJ = CURV ? a.ijn[(size_t)e * NN + node] : a.inv_jac[e];
    in.nbx = in.nby = in.slot = -1;
    if (i == 0 || i == n - 1) in.nbx = a.nbr[4 * e + (i == 0 ? 0 : 1)];
    if (j == 0 || j == n - 1) in.nby = a.nbr[4 * e + (j == 0 ? 2 : 3)];
    const int ls = tid / (4 * n);
    if (tid < NSLOT && ls < blk.y) in.slot = a.nbr[4 * (blk.x + ls) + (tid / n) % 4];
    if (tid < NN) {  // published by the first barrier of the element procedure
        const int q = (tid / n) * G_::MS + tid % n;
        sDh[q] = dev_const(a.c)->Dhat[tid / n][tid % n];
        sD[q] = dev_const(a.c)->D[tid / n][tid % n];
    }
    volume_tile<N, EB, KIND, SC, PAR, CURV>(a, bid, blk, in, lds, sDh, sD, s_alpha);
}

// the Navier-Stokes LW and MDRK stage-2 wall kernels (a rarely used
// configuration: the lid-driven cavity's walls) run at one wave per SIMD, so
// their extra wall terms live in the accumulation registers instead of private
// memory; the stage-1 wall kernel fits two waves
template <int KIND, bool SC, bool PAR>
constexpr int kVolWavesOf =
    (KIND == VOL_LW_WALL || KIND == VOL_MDRK2_WALL || KIND == VOL_LW_ADAPT_WALL)
        ? 1
        : kVolWaves<SC || PAR || vol_is_src(KIND)>;
template <int N, int EB, int KIND, bool SC, bool PAR = false, bool CURV = false>
__global__ __launch_bounds__((VGeo<N, EB>::NT), (kVolWavesOf<KIND, SC, PAR>)) void k_volume(KArgs a) {
    using G_ = VGeo<N, EB>;
    __shared__ alignas(16) double lds[vol_two_buffers<SC, PAR> ? G_::LDS2 : G_::LDS];
    __shared__ alignas(16) double sDh[G_::M], sD[G_::M];
    __shared__ double s_alpha[SC ? EB + 1 : 1];
    volume_body<N, EB, KIND, SC, PAR, CURV>(a, blockIdx.x, lds, sDh, sD, s_alpha);
}

// Outer record of a domain-boundary face node: time average of the boundary
// value over the step with the GLL rule (equations.jl:6-37).
template <int N>
__device__ inline void boundary_record(const KArgs& a, int e, int face, int l, double t, double dt, double* r) {
    constexpr int n = N + 1;
    const DevC c = dev_const(a.c);
    const int orientation = face < 2 ? 1 : 2;
    const double half = 0.5 * a.length[e];
    double x, y;
    if (orientation == 1) {
        x = a.center[2 * e] + half * c->nodes[face == 0 ? 0 : n - 1];
        y = a.center[2 * e + 1] + half * c->nodes[l];
    } else {
        x = a.center[2 * e] + half * c->nodes[l];
        y = a.center[2 * e + 1] + half * c->nodes[face == 2 ? 0 : n - 1];
    }
    const double sf = a.bc_scale;
    const double dts = sf * dt;
    const double gm1 = c->gamma - 1.0;
    double Uo[4] = {0, 0, 0, 0}, Fo[4] = {0, 0, 0, 0}, uo[4];
    for (int q = 0; q < n; ++q) {
        const double ts = t + 0.5 * dts * (c->nodes[q] + 1.0);
        double ub[4], fb[4];
        boundary_state<n>(c, a.bidx, a.btab, a.btab_levels, e, face, l, q, x, y, ts, ub);
        euler_flux_dir(ub, gm1, orientation, fb);
        for (int v = 0; v < 4; ++v) {
            Uo[v] += 0.5 * sf * ub[v] * c->weights[q];
            Fo[v] += 0.5 * sf * fb[v] * c->weights[q];
        }
    }
    boundary_state<n>(c, a.bidx, a.btab, a.btab_levels, e, face, l, n, x, y, t, uo);
    const bool tree = c->flux_order == 0;
    double av1, av2, cs;
    speed_parts2(tree ? Uo : uo, c->gamma, av1, av2, cs);
    make_record(r, tree ? uo : Uo, Fo, orientation == 1 ? av1 : av2, cs);
}

// Outer record of a domain-boundary face node of a curvilinear mesh
// (calc_boundary_flux_by_direction!, structured/dg_2d.jl:2352-2391, into the
// Dirichlet call of equations.jl:6-37): the GLL time averages (over
// [t, t + s dt], s = a.bc_scale: 1 on a StructuredMesh, 0.5 in MDRK stage 1 of
// a P4estMesh) of the boundary value and of its flux in the normal direction
// (Trixi flux(u, n): (ρv_n, ρv_n v1 + p n1, ρv_n v2 + p n2, (ρe + p) v_n)) with
// the element's own face normal, and λ's parts of the average.  The record's
// jump state is u_outer(t) (the StructuredMesh call: TreeMesh order, jump on
// uⁿ, λ from Ũ) or, with p4est_form, the time average itself (the P4est
// method, equations.jl:66-93).
template <int N>
__device__ inline void boundary_record_curved(const KArgs& a, int e, int face, int l, double t, double dt, double* r,
                                              bool p4est_form = false) {
    constexpr int n = N + 1;
    const DevC c = dev_const(a.c);
    const size_t fo = ((size_t)e * 4 + face) * n + l;
    const double x = a.fxy[2 * fo], y = a.fxy[2 * fo + 1];
    double nf[4];
    load4(a.fnorm + 4 * fo, nf);
    const double gm1 = c->gamma - 1.0;
    const double sf = a.bc_scale, dts = sf * dt;
    double Uo[4] = {0, 0, 0, 0}, Fo[4] = {0, 0, 0, 0}, uo[4];
    for (int q = 0; q < n; ++q) {
        const double ts = t + 0.5 * dts * (c->nodes[q] + 1.0);
        double ub[4];
        boundary_state<n>(c, a.bidx, a.btab, a.btab_levels, e, face, l, q, x, y, ts, ub);
        const double rho = ub[0], v1 = ub[1] / rho, v2 = ub[2] / rho;
        const double p = gm1 * (ub[3] - 0.5 * (ub[1] * v1 + ub[2] * v2));
        const double vn = v1 * nf[0] + v2 * nf[1], rvn = rho * vn;
        const double fb[4] = {rvn, rvn * v1 + p * nf[0], rvn * v2 + p * nf[1], (ub[3] + p) * vn};
        for (int v = 0; v < 4; ++v) {
            Uo[v] += 0.5 * sf * ub[v] * c->weights[q];
            Fo[v] += 0.5 * sf * fb[v] * c->weights[q];
        }
    }
    if (!p4est_form) boundary_state<n>(c, a.bidx, a.btab, a.btab_levels, e, face, l, n, x, y, t, uo);
    const double ir = rcp_nr(Uo[0]);
    const double b1 = Uo[1] * ir, b2 = Uo[2] * ir;
    const double pb = gm1 * (Uo[3] - 0.5 * (Uo[1] * b1 + Uo[2] * b2));
    make_record(r, p4est_form ? Uo : uo, Fo, fabs(fma(b1, nf[0], b2 * nf[1])), sqrt_gs(c->gamma * pb * ir) * nf[2]);
}

// Surface kernel: the faces that leave a volume workgroup.
// Each interface is evaluated by both neighbours from identical inputs, so
// both see the same bits.  In step mode every lane then takes its node's
// final value (corrected here or finalised by the volume kernel) into the
// CFL maxima and the admissibility test.
// BC: the mesh has domain-boundary faces; MORT: it has faces on L2 mortars (a
// mesh with mortars and no boundary face compiles no boundary code).
// RED: the launch reduces (a.reduce is not RED_NONE) and reads every node's value,
// which goes out together with the faces' links.  One that does not (a rhs, MDRK
// stage 1, a step with the limiter) reads only what it corrects: a rhs at 256² then
// takes 103.5 us instead of 105.9 (N=4) and 58.9 instead of 60.3 (N=3), MDRK stage 2
// alone at 512² 206 instead of 211 (N=3) and 326 instead of 331 (N=4).  A kernel of
// its own, as the choice at run time costs a step of a 32² mesh 1.5 %.
template <int N, bool BC, bool SC, bool CURV, bool MORT, bool RED>
__device__ __forceinline__ void surface_body(const KArgs& a, int bid) {
    using G_ = SGeo<N>;
    constexpr int n = G_::n, NN = G_::NN, EB = G_::EB, S = G_::S;
    const int4 blk = load_blk_at(a.sblk, bid);
    const DevS st = dev_state(a.st + blk.z);
    if (a.use_state_dt && st->finished) return;
    const int tid = threadIdx.x;
    const int le = tid / NN, node = tid - (tid / NN) * NN;
    const int i = node % n, j = node / n;
    const int e0 = blk.x;
    const int nel = blk.y;
    const bool act = le < nel;
    const int lec = le < nel ? le : nel - 1;
    const int e = e0 + lec;
    const int cur = a.use_state_dt ? st->cur : 0;
    double* out = sel_out(a, cur);
    const double dt = a.use_state_dt ? st->dt : a.dt_arg;
    const double t = a.use_state_dt ? st->t : a.t_arg;
    const DevC c = dev_const(a.c);
    const double invJ = CURV ? a.ijn[(size_t)e * NN + node] : a.inv_jac[e];
    const int fx = (i == 0) ? 0 : ((i == n - 1) ? 1 : -1);
    const int fy = (j == 0) ? 2 : ((j == n - 1) ? 3 : -1);
    const size_t off = ((size_t)e * NN + node) * 4;
    int nbx = kResolved, nby = kResolved;
    if (fx >= 0) nbx = a.link[4 * e + fx];
    if (fy >= 0) nby = a.link[4 * e + fy];
    double val[4];
    if constexpr (RED) load4(out + off, val);
    const bool extx = nbx != kResolved, exty = nby != kResolved;
    if (act && (extx || exty)) {
        if constexpr (!RED) load4(out + off, val);
        double surf[4] = {0.0, 0.0, 0.0, 0.0};
        constexpr int RQ = kRQ<SC>;
        auto do_face = [&](int f, int l, int nb) {
            double own[RQ], oth[RQ], Fs[4];
            load_record<RQ>(a.trace + (((size_t)e * 4 + f) * n + l) * RQ, own);
            const double* Lr = (f & 1) ? own : oth;
            const double* Rr = (f & 1) ? oth : own;
            if ((!BC && !MORT) || nb >= 0) {
                load_record<RQ>(a.trace + (((size_t)nb * 4 + (f ^ 1)) * n + l) * RQ, oth);
                if constexpr (SC && CURV) {
                    // the neighbour's mirrored face node and the element-wise blending factors
                    const int nnode = (f == 0) ? l * n + (n - 1) : (f == 1) ? l * n : (f == 2) ? (n - 1) * n + l : l;
                    const double Jo = a.ijn[(size_t)e * NN + node], Jn = a.ijn[(size_t)nb * NN + nnode];
                    const double ao = a.alpha_out[e], an = a.alpha_out[nb];
                    double nf[4];
                    load4(a.fnorm + (((size_t)e * 4 + f) * n + l) * 4, nf);
                    if (f & 1)
                        face_numflux_sc_curved(Lr, Rr, nf, Jo, Jn, ao, an, c->gamma, dt, c->weights[n - 1],
                                               c->weights[0], Fs);
                    else
                        face_numflux_sc_curved(Lr, Rr, nf, Jn, Jo, an, ao, c->gamma, dt, c->weights[n - 1],
                                               c->weights[0], Fs);
                } else if constexpr (SC) {
                    face_numflux_sc(Lr, Rr, f < 2 ? 1 : 2, c->gamma, st->invJ0, dt, c->weights[n - 1], c->weights[0],
                                    Fs);
                } else {
                    face_numflux(Lr, Rr, Fs);
                }
            } else if (MORT && nb <= -2) {
                // a face on an L2 mortar: the mortar kernel's flux of this element's role
                load4(a.mflux + ((size_t)(-2 - nb) * n + l) * 4, Fs);
            } else if constexpr (BC) {
                // domain boundary: time-averaged Dirichlet state, no blending
                // (calc_boundary_flux!, dg_2d.jl:1379-1454; structured/dg_2d.jl:2297-2391)
                if constexpr (CURV) {
                    // the volume kernel's record holds Ũ and F̃·n (and uⁿ with shock
                    // capturing); the Dirichlet call takes the TreeMesh order: jump on
                    // uⁿ, λ from Ũ; no blending (structured/dg_2d.jl:2352-2391)
                    double nf[4], in10[kTraceQ], out10[kTraceQ];
                    load4(a.fnorm + (((size_t)e * 4 + f) * n + l) * 4, nf);
                    if (nb == -3) {
                        // P4estMesh interface (prolong2interfaces!/calc_interface_flux!,
                        // p4est/dg_2d.jl:8-192): each record holds F̃ in its element's +ξ/+η
                        // direction (F̃·Ja of its own node); in the primary's outward
                        // direction that is s_p·F̃_p and -s_s·F̃_s (s = +1 on + faces, -1 on
                        // - faces); λ's parts from uⁿ, the jump on Ũ.  Both elements form
                        // the same primary-outward flux; each keeps its +ξ/+η version.
                        const int4 pl = a.plink[4 * e + f];
                        const int lp = pl.z ? n - 1 - l : l;
                        load_record<RQ>(a.trace + (((size_t)pl.x * 4 + pl.y) * n + lp) * RQ, oth);
                        const double so = (f & 1) ? 1.0 : -1.0, sq = (pl.y & 1) ? 1.0 : -1.0;
                        const double* P = pl.w ? own : oth;
                        const double* Q = pl.w ? oth : own;
                        const double sP = pl.w ? so : sq, sQ = pl.w ? sq : so;
                        double Lq[kTraceQ], Rq[kTraceQ], Fo_[4];
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            Lq[v] = P[v];
                            Rq[v] = Q[v];
                            Lq[4 + v] = sP * P[4 + v];
                            Rq[4 + v] = -sQ * Q[4 + v];
                        }
                        Lq[8] = P[8];
                        Lq[9] = P[9];
                        Rq[8] = Q[8];
                        Rq[9] = Q[9];
                        face_numflux(Lq, Rq, Fo_);
#pragma unroll
                        for (int v = 0; v < 4; ++v) Fs[v] = pl.w ? so * Fo_[v] : -so * Fo_[v];
                        const double wf = (f & 1) ? c->bnd_hi : -c->bnd_lo;
#pragma unroll
                        for (int v = 0; v < 4; ++v) surf[v] = fma(Fs[v], wf, surf[v]);
                        return;
                    }
                    if (a.plink) {
                        // P4estMesh boundary with the time-averaged Dirichlet value (the
                        // P4est method, equations.jl:66-93): the volume kernel's record as
                        // the inner state (jump on Ũ, λ from uⁿ), the outer record with the
                        // time average as both jump state and λ state; inner first along
                        // the outward normal, i.e. the outer record on the - side in +ξ/+η
                        if (c->bc_kind != kBcOutflow && c->bc_kind != kBcSlipWallApprox) {
                            boundary_record_curved<N>(a, e, f, l, t, dt, out10, true);
                            if (f & 1) face_numflux(own, out10, Fs);
                            else face_numflux(out10, own, Fs);
                            const double wf = (f & 1) ? c->bnd_hi : -c->bnd_lo;
#pragma unroll
                            for (int v = 0; v < 4; ++v) surf[v] = fma(Fs[v], wf, surf[v]);
                            return;
                        }
                    }
                    if (c->bc_kind == kBcOutflow || c->bc_kind == kBcSlipWallApprox) {
                        // conditions on uⁿ with the node's contravariant vector as normal
                        // (boundary_condition_outflow, slip_wall_approximate,
                        // equations.jl:185-197, 251-260): the normal flux of uⁿ, or the
                        // Rusanov flux between uⁿ and its reflection with the reflected
                        // state on the side of the boundary
                        double un[4], ur[4];
                        if constexpr (SC) {
#pragma unroll
                            for (int v = 0; v < 4; ++v) un[v] = own[8 + v];
                        } else {
                            load4(sel_in(a, cur) + ((size_t)e * NN + node) * 4, un);
                        }
                        if (c->bc_kind == kBcOutflow) {
                            rusanov_normal(un, un, c->gamma, nf[0], nf[1], nf[2], Fs);
                        } else {
                            const double ir = rcp_nr(un[0]);
                            const double v1 = un[1] * ir, v2 = un[2] * ir;
                            const double p = (c->gamma - 1.0) * (un[3] - 0.5 * (un[1] * v1 + un[2] * v2));
                            const double vn = fma(v1, nf[0], v2 * nf[1]) / (nf[2] * nf[2]);
                            const double w1 = v1 - 2.0 * vn * nf[0], w2 = v2 - 2.0 * vn * nf[1];
                            ur[0] = un[0];
                            ur[1] = un[0] * w1;
                            ur[2] = un[0] * w2;
                            ur[3] = p / (c->gamma - 1.0) + 0.5 * un[0] * (w1 * w1 + w2 * w2);
                            if (f & 1) rusanov_normal(un, ur, c->gamma, nf[0], nf[1], nf[2], Fs);
                            else rusanov_normal(ur, un, c->gamma, nf[0], nf[1], nf[2], Fs);
                        }
                        const double wf = (f & 1) ? c->bnd_hi : -c->bnd_lo;
#pragma unroll
                        for (int v = 0; v < 4; ++v) surf[v] = fma(Fs[v], wf, surf[v]);
                        return;
                    }
                    const double ir = rcp_nr(own[0]);
                    const double b1 = own[1] * ir, b2 = own[2] * ir;
                    const double pb = (c->gamma - 1.0) * (own[3] - 0.5 * (own[1] * b1 + own[2] * b2));
                    if constexpr (SC) {
#pragma unroll
                        for (int v = 0; v < 4; ++v) in10[v] = own[8 + v];
                    } else {
                        load4(sel_in(a, cur) + ((size_t)e * NN + node) * 4, in10);
                    }
#pragma unroll
                    for (int v = 0; v < 4; ++v) in10[4 + v] = own[4 + v];
                    in10[8] = fabs(fma(b1, nf[0], b2 * nf[1]));
                    in10[9] = sqrt_gs(c->gamma * pb * ir) * nf[2];
                    boundary_record_curved<N>(a, e, f, l, t, dt, out10);
                    if (f & 1) face_numflux(in10, out10, Fs);
                    else face_numflux(out10, in10, Fs);
                } else if (c->bc_kind == kBcSlipWall) {
                    // reflecting wall (equations.jl:95-139): the mirrored record, whatever
                    // the flux order (both states are mirrored, the speeds kept)
                    const int m = (f < 2) ? 1 : 2;
                    double fvw[3] = {0.0, 0.0, 0.0};
                    if (c->ns_walls) {
                        // Navier-Stokes: the record holds F̃a - F̃v; the wall flux is built
                        // from F̃a (its normal-momentum component: the others cancel against
                        // their mirror images), then the wall's viscous flux is subtracted
                        const double* q = a.fvb + (((size_t)e * 4 + f) * n + l) * 6;
                        fvw[0] = q[0];
                        fvw[1] = q[1];
                        fvw[2] = q[2];
                        own[4 + m] += fvw[m - 1];
                    }
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        oth[v] = (v == m) ? -own[v] : own[v];
                        oth[4 + v] = (v == m) ? own[4 + v] : -own[4 + v];
                    }
                    oth[8] = own[8];
                    oth[9] = own[9];
                    face_numflux(Lr, Rr, Fs);
                    if (c->ns_walls) {
                        // NoSlip/Adiabatic (compressible_navier_stokes_2d.jl:81-91):
                        // (F̃v1, F̃v2, F̃v3, v_wall · (F̃v2, F̃v3)), F̃v1 = 0; NoSlip/Isothermal
                        // (103-109): the inner viscous flux itself
                        Fs[1] -= fvw[0];
                        Fs[2] -= fvw[1];
                        Fs[3] -= c->wall_iso[f] ? fvw[2]
                                                : fma(c->wall_v[2 * f], fvw[0], c->wall_v[2 * f + 1] * fvw[1]);
                    }
                } else {
                    boundary_record<N>(a, e, f, l, t, dt, oth);
                    face_numflux(Lr, Rr, Fs);
                }
            }
            const double wf = (f & 1) ? c->bnd_hi : -c->bnd_lo;
#pragma unroll
            for (int v = 0; v < 4; ++v) surf[v] = fma(Fs[v], wf, surf[v]);
        };
        if (extx) do_face(fx, j, nbx);
        if (exty) do_face(fy, i, nby);
        const double fac = a.step_mode ? -dt * invJ : -invJ;
#pragma unroll
        for (int v = 0; v < 4; ++v) val[v] = fma(fac, surf[v], val[v]);
        store4(out + off, val);
    }
    if constexpr (!RED) return;
    // Every node's final value, corrected here or finalised by the volume kernel:
    // CFL maxima (Trixi max_dt) and the admissibility test of the updated state
    // cover all nodes here.
    if (a.reduce == RED_ADAPT) {  // test_updated_solution (adaptive.jl:30-46)
        if (act && !admissible(val, c->gamma)) a.st[blk.z].bad_state = 1;
        return;
    }
    const bool par = a.parabolic != 0;
    double l1, l2;
    bool bad;
    if constexpr (CURV) {
        double Jn[4];
        load4(a.Ja + off, Jn);
        curved_speeds(val, Jn, invJ, c->gamma, l1, l2, bad);
    } else {
        node_speeds(val, c->gamma, l1, l2, bad);
    }
    if (act && bad) a.st[blk.z].bad_state = 1;
    const double lv = par ? (CURV ? lam_visc_curved(val, invJ, c) : lam_visc(val, invJ, c)) : 0.0;
    cfl_maxima<N>(a.slots, blk.z, tid, nel, lec * NN + node, act, node == 0, l1, l2, lv, invJ, CURV, par);
}

template <int N, bool BC, bool SC, bool CURV, bool MORT, bool RED>
__global__ __launch_bounds__(kSurfBlock) void k_surface(KArgs a) {
    surface_body<N, BC, SC, CURV, MORT, RED>(a, blockIdx.x);
}

// KArgs::link of one volume workgroup's elements, when the tile is set.
__global__ __launch_bounds__(64) void k_link(const int4* vblk, const int* nbr, int* link) {
    const int4 b = vblk[blockIdx.x];
    for (int q = 4 * b.x + (int)threadIdx.x; q < 4 * (b.x + b.y); q += 64) {
        const int nb = nbr[q];
        link[q] = (nb >= b.x && nb < b.x + b.y) ? kResolved : nb;
    }
}

// AMR solution transfer between two TreeMesh leaf sets (Trixi's refine! and
// coarsen! of the DG solution, src/callbacks_step/amr_dg2d.jl in Trixi.jl,
// which the reference's AMR callback runs before resizing its caches,
// src/callbacks/amr.jl:2-20): one lane per node of the new mesh.  Plan
// [E_new][5]: (0, e) copies leaf e; (1, p, child) interpolates parent p to its
// child (0 lower left, 1 lower right, 2 upper left, 3 upper right) with the
// forward mortar operators in x, then y; (2, c0, c1, c2, c3) projects four
// children onto their parent with the reverse operators, summed over children.
constexpr int kTransferBlock = 256;
template <int N>
__global__ __launch_bounds__(kTransferBlock) void k_transfer(const double* __restrict__ uold, double* __restrict__ unew,
                                                            const int* __restrict__ plan, int E_new,
                                                            const DevConst* dc) {
    const DevC c = dev_const(dc);
    constexpr int n = N + 1, NN = n * n;
    const long long gid = (long long)blockIdx.x * kTransferBlock + threadIdx.x;
    if (gid >= (long long)E_new * NN) return;
    const int e = (int)(gid / NN), node = (int)(gid - (long long)e * NN);
    const int i = node % n, j = node / n;
    const int* p = plan + 5 * (size_t)e;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if (p[0] == 0) {
        load4(uold + ((size_t)p[1] * NN + node) * 4, acc);
    } else {
        const int nsrc = (p[0] == 1) ? 1 : 4;
        for (int q = 0; q < nsrc; ++q) {
            const int src = (p[0] == 1) ? p[1] : p[1 + q];
            const int child = (p[0] == 1) ? p[2] : q;
            const auto* Mx = (p[0] == 1) ? c->mfwd[child & 1][i] : c->mrev[child & 1][i];
            const auto* My = (p[0] == 1) ? c->mfwd[child >> 1][j] : c->mrev[child >> 1][j];
            const double* us = uold + (size_t)src * NN * 4;
            for (int l = 0; l < n; ++l) {
                double t[4] = {0.0, 0.0, 0.0, 0.0};
                for (int k = 0; k < n; ++k) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) t[v] = fma(Mx[k], us[((size_t)l * n + k) * 4 + v], t[v]);
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[v] = fma(My[l], t[v], acc[v]);
            }
        }
    }
    store4(unew + ((size_t)e * NN + node) * 4, acc);
}

// L2 mortars of a TreeMesh with refined cells (prolong2mortars! and
// calc_mortar_flux!, dg_2d.jl:1456-1646, with Trixi's
// mortar_fluxes_to_elements!): one lane per mortar and face node.  On each
// half the large element's jump state, normal flux and λ state are
// interpolated to the node (forward operator of the half) and paired with
// the small element's, the LW flux taken in the interface order (the large
// element on the left when large_side is 1) and kept for the small element;
// the large element's flux at the node is reverse_upper·F*_upper +
// reverse_lower·F*_lower.  The surface kernel lifts both.
constexpr int kMortarBlock = 64;
template <int N>
__global__ __launch_bounds__(kMortarBlock) void k_mortar(KArgs a) {
    constexpr int n = N + 1, MPB = kMortarBlock / n;
    __shared__ double fs[MPB][2][n][4];
    if (a.use_state_dt && a.st[0].finished) return;
    const DevC c = dev_const(a.c);
    const int tid = threadIdx.x, lm = tid / n, l = tid - lm * n;
    const int m = blockIdx.x * MPB + lm;
    const bool act = lm < MPB && m < a.n_mortars;
    if (act) {
        const int2 mo = a.mort[m];
        const double* base = a.mrec + (size_t)m * 3 * n * 12;
        const double* lg = base + 2 * n * 12;
        for (int half = 0; half < 2; ++half) {
            double jl[4] = {0, 0, 0, 0}, Fl[4] = {0, 0, 0, 0}, Ul[4] = {0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < n; ++k) {
                const double p = c->mfwd[half][l][k];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    jl[v] = fma(p, lg[k * 12 + v], jl[v]);
                    Fl[v] = fma(p, lg[k * 12 + 4 + v], Fl[v]);
                    Ul[v] = fma(p, lg[k * 12 + 8 + v], Ul[v]);
                }
            }
            const double* sm = base + ((size_t)half * n + l) * 12;
            double rL[kTraceQ], rS[kTraceQ], Fs[4];
            double aL, cL, aS, cS;
            speed_parts(Ul, c->gamma, mo.x, aL, cL);
            speed_parts(sm + 8, c->gamma, mo.x, aS, cS);
            make_record(rL, jl, Fl, aL, cL);
            make_record(rS, sm, sm + 4, aS, cS);
            if (mo.y == 1) face_numflux(rL, rS, Fs);
            else face_numflux(rS, rL, Fs);
            store4(a.mflux + (((size_t)m * 3 + half) * n + l) * 4, Fs);
#pragma unroll
            for (int v = 0; v < 4; ++v) fs[lm][half][l][v] = Fs[v];
        }
    }
    __syncthreads();
    if (act) {
        double Fb[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            double acc = 0.0;
#pragma unroll
            for (int k = 0; k < n; ++k) acc = fma(c->mrev[1][l][k], fs[lm][1][k][v], acc);
#pragma unroll
            for (int k = 0; k < n; ++k) acc = fma(c->mrev[0][l][k], fs[lm][0][k][v], acc);
            Fb[v] = acc;
        }
        store4(a.mflux + (((size_t)m * 3 + 2) * n + l) * 4, Fb);
    }
}

// CFL reduction over a whole state (Trixi max_dt) without an update: first dt
// of a solve (RED_INIT) or a max_dt query (RED_QUERY).
template <int N>
__global__ __launch_bounds__(kSurfBlock) void k_max_speed(KArgs a) {
    using G_ = SGeo<N>;
    constexpr int NN = G_::NN;
    const int4 blk = load_blk(a.sblk);
    const int tid = threadIdx.x;
    const int le = tid / NN, node = tid - (tid / NN) * NN;
    const int nel = blk.y;
    const bool act = le < nel;
    const int lec = le < nel ? le : nel - 1;
    const int e = blk.x + lec;
    const DevC c = dev_const(a.c);
    const size_t off = ((size_t)e * NN + node) * 4;
    const double* uin = sel_in(a, dev_state(a.st + blk.z)->cur);
    double val[4];
    load4(uin + off, val);
    const bool curv = a.Ja != nullptr;  // speeds in reference space, |J⁻¹| included
    const double invJ = curv ? a.ijn[(size_t)e * NN + node] : a.inv_jac[e];
    double l1, l2;
    bool bad;
    if (curv) {
        double Jn[4];
        load4(a.Ja + off, Jn);
        curved_speeds(val, Jn, invJ, c->gamma, l1, l2, bad);
    } else {
        node_speeds(val, c->gamma, l1, l2, bad);
    }
    if (act && bad) a.st[blk.z].bad_state = 1;
    const bool par = a.parabolic != 0;
    const double lv = par ? (curv ? lam_visc_curved(val, invJ, c) : lam_visc(val, invJ, c)) : 0.0;
    cfl_maxima<N>(a.slots, blk.z, tid, nel, lec * NN + node, act, node == 0, l1, l2, lv, invJ, curv, par);
}

// Hennemann-Gassner indicator (Trixi IndicatorHennemannGassner, Hennemann et
// al., JCP 426, 2021) on density_pressure, before smoothing: modal energy of
// the highest and second-highest modes, logistic blending with threshold
// 0.5·10^(-1.8 n^0.25) and sharpness ln((1-1e-4)/1e-4), clipped below
// alpha_min to 0, above 1-alpha_min to 1, capped at alpha_max.
template <int N>
__global__ __launch_bounds__(kSurfBlock) void k_indicator(KArgs a, double* alpha_tmp) {
    using G_ = SGeo<N>;
    constexpr int n = G_::n, NN = G_::NN, EB = G_::EB, S = G_::S;
    constexpr int NP = NN + (NN & 1);  // element stride: pairs of doubles
    __shared__ double s_a[S], s_b[S];
    __shared__ alignas(16) double s_e[EB * NP];
    const int tid = threadIdx.x;
    const int le = tid / NN, node = tid - (tid / NN) * NN;
    const int i = node % n, j = node / n;
    const int4 blk = load_blk(a.sblk);
    const DevState* st = a.st + blk.z;
    const int e0 = blk.x;
    const int nel = blk.y;
    const bool act = le < nel;
    const int lec = le < nel ? le : nel - 1;
    const int e = e0 + lec;
    const DevC c = dev_const(a.c);
    const double* uin = sel_in(a, a.use_state_dt ? st->cur : 0);
    if (a.use_state_dt && st->finished) return;
    double un[4];
    load4(uin + ((size_t)e * NN + node) * 4, un);
    const double rp = (c->gamma - 1.0) * (un[0] * un[3] - 0.5 * (un[1] * un[1] + un[2] * un[2]));
    if (act) s_a[lec * NN + node] = rp;
    __syncthreads();
    double acc = 0.0;  // x transform: tmp[j][i] = Σ_ii Vinv[i][ii] ind[j][ii]
#pragma unroll
    for (int k = 0; k < n; ++k) acc = fma(c->Vinv[i][k], s_a[lec * NN + j * n + k], acc);
    if (act) s_b[lec * NN + node] = acc;
    __syncthreads();
    double m = 0.0;  // y transform: modal[j][i] = Σ_jj Vinv[j][jj] tmp[jj][i]
#pragma unroll
    for (int k = 0; k < n; ++k) m = fma(c->Vinv[j][k], s_b[lec * NN + k * n + i], m);
    if (act) s_e[lec * NP + node] = m * m;
    __syncthreads();
    // the energies in node order (the reference's: their differences cancel), by
    // one lane per element of the first wave from pairs of modes in registers;
    // 75 single reads by a lane of every element before: 23.0 us at 256², N=4, now 17.8
    if (tid < nel) {
        double q[NP];
#pragma unroll
        for (int k = 0; k < NP; k += 2) {
            const double2 x = *reinterpret_cast<const double2*>(s_e + tid * NP + k);
            q[k] = x.x;
            q[k + 1] = x.y;
        }
        double tot = 0.0, c1 = 0.0, c2 = 0.0;
#pragma unroll
        for (int k = 0; k < NN; ++k) {
            const int a1 = k % n, a2 = k / n;
            tot += q[k];
            if (a1 < n - 1 && a2 < n - 1) c1 += q[k];
            if (a1 < n - 2 && a2 < n - 2) c2 += q[k];
        }
        const double f1 = tot != 0.0 ? (tot - c1) / tot : 0.0;
        const double f2 = c1 != 0.0 ? (c1 - c2) / c1 : 0.0;
        const double energy = dmax(f1, f2);
        const double threshold = c->hg_threshold, par_s = c->hg_sharpness;
        double al = 1.0 / (1.0 + exp(-par_s / threshold * (energy - threshold)));
        if (al < c->alpha_min) al = 0.0;
        if (al > 1.0 - c->alpha_min) al = 1.0;
        alpha_tmp[e0 + tid] = al < c->alpha_max ? al : c->alpha_max;
    }
}

// Zhang-Shu positivity limiter on (density, pressure), in that order
// (my_limiter_zhang_shu!, src/callbacks/callbacks_stage/positivity_zhang_shu_dg2d.jl:8-45,
// positivity_zhang_shu.jl:26-41): where the variable's minimum over an
// element's nodes is below its threshold, u <- θ u + (1-θ) ū with
// θ = (var(ū) - threshold) / (var(ū) - min var) and ū = Σ u w_i w_j / 4 summed
// in the reference's node order.  Limits a.out (explicit) or the new state of
// the device loop in place and, in the loop, takes the CFL reduction of the
// limited state (the next step's compute_dt).
template <int N>
__global__ __launch_bounds__(kSurfBlock) void k_limiter(KArgs a) {
    using G_ = SGeo<N>;
    constexpr int n = G_::n, NN = G_::NN, EB = G_::EB, S = G_::S;
    __shared__ double s_var[S], s_q[4][S];
    __shared__ double s_theta[EB], s_mean[EB][4];
    __shared__ int s_flag[EB];
    const int4 blk = load_blk(a.sblk);
    DevState* st = a.st + blk.z;
    if (a.use_state_dt && st->finished) return;
    const int tid = threadIdx.x;
    const int le = tid / NN, node = tid - (tid / NN) * NN;
    const int i = node % n, j = node / n;
    const int e0 = blk.x;
    const int nel = blk.y;
    const bool act = le < nel;
    const int lec = le < nel ? le : nel - 1;
    const int e = e0 + lec;
    const int sidx = lec * NN + node, sbase = lec * NN;
    const int cur = a.use_state_dt ? st->cur : 0;
    double* u = sel_out(a, cur);
    const DevC c = dev_const(a.c);
    const double gm1 = c->gamma - 1.0;
    const size_t off = ((size_t)e * NN + node) * 4;
    double un[4];
    load4(u + off, un);
    bool changed = false;
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        const double thr = c->pos_threshold[pass];
        const double var = pass == 0 ? un[0] : gm1 * (un[3] - 0.5 * (un[1] * un[1] + un[2] * un[2]) / un[0]);
        if (act) {
            s_var[sidx] = var;
#pragma unroll
            for (int v = 0; v < 4; ++v) s_q[v][sidx] = un[v] * c->weights[i] * c->weights[j];
        }
        __syncthreads();
        if (act && node == 0) {
            double vmin = s_var[sbase];
            for (int k = 1; k < NN; ++k) vmin = s_var[sbase + k] < vmin ? s_var[sbase + k] : vmin;
            int flag = vmin < thr;
            if (flag) {
                double m[4] = {0.0, 0.0, 0.0, 0.0};
                for (int k = 0; k < NN; ++k)
#pragma unroll
                    for (int v = 0; v < 4; ++v) m[v] += s_q[v][sbase + k];
#pragma unroll
                for (int v = 0; v < 4; ++v) m[v] = m[v] / 4.0;
                const double vmean = pass == 0 ? m[0] : gm1 * (m[3] - 0.5 * (m[1] * m[1] + m[2] * m[2]) / m[0]);
                s_theta[le] = (vmean - thr) / (vmean - vmin);
#pragma unroll
                for (int v = 0; v < 4; ++v) s_mean[le][v] = m[v];
            }
            s_flag[le] = flag;
        }
        __syncthreads();
        if (s_flag[lec]) {
            const double th = s_theta[lec];
#pragma unroll
            for (int v = 0; v < 4; ++v) un[v] = th * un[v] + (1.0 - th) * s_mean[lec][v];
            changed = true;
        }
        __syncthreads();  // s_var, s_q, s_flag are rewritten by the next pass
    }
    if (act && changed) store4(u + off, un);
    if (a.reduce == RED_NONE) return;
    // CFL maxima of the limited state (curvilinear speeds carry the node's |J⁻¹|;
    // Navier-Stokes adds the viscous bound)
    const bool curv = a.Ja != nullptr, par = a.parabolic != 0;
    const double invJ = curv ? a.ijn[(size_t)e * NN + node] : a.inv_jac[e];
    double l1, l2;
    bool bad;
    if (curv) {
        double Jn[4];
        load4(a.Ja + off, Jn);
        curved_speeds(un, Jn, invJ, c->gamma, l1, l2, bad);
    } else {
        node_speeds(un, c->gamma, l1, l2, bad);
    }
    if (act && bad) st->bad_state = 1;
    const double lv = par ? (curv ? lam_visc_curved(un, invJ, c) : lam_visc(un, invJ, c)) : 0.0;
    cfl_maxima<N>(a.slots, blk.z, tid, nel, sidx, act, node == 0, l1, l2, lv, invJ, curv, par);
}

// Step control of the adaptive LW loop (perform_step! for Adaptive and LW,
// adaptive.jl:48-64, 95-173): total error sqrt(Σ temporal_errors / ndofs),
// epsilon shift on a first attempt, factor 1 + atan(ε1^(β1/k) ε0^(β2/k) ε-1^(β3/k) - 1)
// with (β1, β2, β3) = (0.6, -0.2, 0) (lwfr.jl:162) and k = nnodes; the step is
// rejected when the updated state is not admissible or factor <= 0.81 (retry
// from uⁿ with min(factor, 0.95)·dt), else accepted with next dt min(factor, 1.5)·dt.
// A non-finite factor on a rejected step shrinks dt by 0.95.
__device__ inline void adaptive_control(DevState* st, double total, double k) {
    const double err = sqrt(total / st->ndofs);
    if (st->nfail == 0) {
        st->eps[0] = st->eps[1];
        st->eps[1] = st->eps[2];
    }
    st->eps[2] = 1.0 / (err + 1e-12);
    const double fac = pow(st->eps[2], 0.6 / k) * pow(st->eps[1], -0.2 / k) * pow(st->eps[0], 0.0 / k);
    const double factor = 1.0 + atan(fac - 1.0);
    const double t = st->t, tf = st->t_final;
    double dt = st->dt;
    if (st->bad_state || !(factor > 0.81)) {
        st->nfail = st->nfail + 1;
        dt = (factor < 0.95 ? factor : 0.95) * dt;
        if (t + dt > tf) dt = tf - t;  // set_dt!
        st->dt = dt;
        st->bad_state = 0;
        return;
    }
    st->nreject = st->nreject + st->nfail;
    st->nfail = 0;
    double dtn = (factor < 1.5 ? factor : 1.5) * dt;
    double dts = dt;
    if (t + dts > tf) dts = tf - t;  // set_t_and_iter!
    const double t1 = t + dts;
    st->t = t1;
    st->iter = st->iter + 1;
    st->cur = 1 - st->cur;
    if (t1 + dtn > tf) dtn = tf - t1;  // set_dt!
    st->dt = dtn;
    st->finished = julia_isapprox(t1, tf);
}

constexpr int kFinalizeBlock = 1024;  // adaptive steps
constexpr int kFinalizeWave = 64;
// Per-step dt record and prescription of a single-instance device loop: the dt
// of step k (k = the iteration count since the last solve_init) is written to
// log[k] while k < log_cap, and taken from presc[k] instead of cfl · max_dt
// while k < presc_n (the truncation at the final time still applies).
struct DtLog {
    double* log;
    long long log_cap;
    const double* presc;
    long long presc_n;
};
// The arguments of one context's finalize launch; reduce is RED_QUERY, RED_INIT or
// RED_STEP, or RED_ADAPT for k_finalize_adaptive, which reads partial and rng (the range
// of each instance's volume workgroups).
struct FinArgs {
    DevState* st_all;
    const double* partial;
    const int2* rng;
    int reduce, parabolic;
    double* slots;
    DtLog dl;
};

// The end of an adaptive step, one workgroup per instance: the sum of the volume
// workgroups' temporal-error partials (rng[inst].x to .y), then the controller.
template <int N>
__global__ __launch_bounds__(kFinalizeBlock) void k_finalize_adaptive(FinArgs f) {
    __shared__ double s[kFinalizeBlock];
    const double* partial = f.partial;
    DevState* st = f.st_all + blockIdx.x;
    const int2 r = f.rng[blockIdx.x];
    if (st->finished) return;
    double m[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    int k = r.x + (int)threadIdx.x;
    for (; k + 7 * kFinalizeBlock < r.y; k += 8 * kFinalizeBlock) {
#pragma unroll
        for (int q = 0; q < 8; ++q) m[q] += partial[k + q * kFinalizeBlock];
    }
    for (; k < r.y; k += kFinalizeBlock) m[0] += partial[k];
    s[threadIdx.x] = ((m[0] + m[1]) + (m[2] + m[3])) + ((m[4] + m[5]) + (m[6] + m[7]));
    __syncthreads();
    for (int w = kFinalizeBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) adaptive_control(st, s[0], N + 1.0);
}

// The maximum over the CFL slots of instance `bid` (reset for the next reduction),
// then compute_dt / set_dt! / set_t_and_iter! / isfinished on the instance's state
// (lwfr.jl:76-103, 146-148, 176-190; Trixi max_dt).  The viscous maxima give the
// parabolic bound 1/((λa + λv)·2(2N+1)), λv = 2(2N+1)·max J⁻² max(4μ/(3ρ), μκ/(ρPr)),
// and max_dt is the smaller of the two (compute_dt for
// SemidiscretizationHyperbolicParabolic, lwfr.jl:192-210).
// A step of a small mesh waits for this kernel's chain of memory latencies, so one
// wave does it, four slots a lane, with every load sent out at the start and the
// maximum taken across lanes: 1.76 us of a 32² step of 13.7 us (N=4), where 1024
// lanes and a tree in LDS took 2.96.
template <int N> __device__ __forceinline__ void finalize_body(const FinArgs& f, int bid) {
    constexpr int n = N + 1, Q = kSlots / kFinalizeWave;
    const int lane = threadIdx.x;
    DevState* st = f.st_all + bid;
    double* sl = f.slots + (size_t)bid * 2 * kSlots + lane;
    const bool par = f.parabolic != 0;
    double m[Q], mv[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        m[q] = sl[q * kFinalizeWave];
        mv[q] = par ? sl[kSlots + q * kFinalizeWave] : 0.0;
    }
    double t = st->t;
    const double dt_step = st->dt, tf = st->t_final, cfl = st->cfl;
    const int cur = st->cur;
    long long it = st->iter;
    if (f.reduce == RED_STEP && st->finished) return;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        sl[q * kFinalizeWave] = 0.0;
        if (par) sl[kSlots + q * kFinalizeWave] = 0.0;
    }
    auto wave_max = [](const double* x) {
        double v = x[0];
#pragma unroll
        for (int q = 1; q < Q; ++q) v = fmax(v, x[q]);
        return max_groups(max_group8(v));
    };
    const double tiny = 4.9406564584124654e-324;  // nextfloat(0.0), Trixi's start value
    const double M = dmax(tiny, wave_max(m));
    double max_dt = 2.0 / (n * M);
    if (par) {
        const double lam_v = dmax(tiny, wave_max(mv)) * (2.0 * (2.0 * N + 1.0));
        const double dtv = 1.0 / ((M + lam_v) * (2 * (2.0 * N + 1.0)));
        if (dtv < max_dt) max_dt = dtv;
    }
    if (lane != 0) return;
    if (f.reduce == RED_QUERY) {
        st->query = max_dt;
        return;
    }
    if (f.reduce == RED_STEP) {
        t = t + dt_step;  // set_t_and_iter!
        it = it + 1;
        st->t = t;
        st->iter = it;
        st->cur = 1 - cur;
    }
    const DtLog& dl = f.dl;
    double dt = cfl * max_dt;  // compute_dt
    if (dl.presc && it < dl.presc_n) dt = dl.presc[it];  // prescribed dt of step `it`
    if (t + dt > tf) dt = tf - t;  // set_dt!
    st->dt = dt;
    if (dl.log && it < dl.log_cap) dl.log[it] = dt;
    st->finished = julia_isapprox(t, tf);
}

template <int N> __global__ __launch_bounds__(kFinalizeWave) void k_finalize(FinArgs f) {
    finalize_body<N>(f, blockIdx.x);
}

// Two contexts advanced by the same launches (tlw_create_ensemble): one of
// polydeg 3 (workgroups [0, g3) of each launch) and one of polydeg 4, plain LW
// on periodic meshes; each half runs its own context's kernel body on its own
// tables, so every instance gets the bits of its own context's launches.
template <int EB3, int EB4>
__global__ __launch_bounds__((VGeo<4, EB4>::NT), kVolWaves<false>) void k_volume_pair(KArgs a3, KArgs a4, int g3) {
    static_assert(VGeo<3, EB3>::NT == VGeo<4, EB4>::NT, "one block size for both halves");
    constexpr int L = VGeo<3, EB3>::LDS2 > VGeo<4, EB4>::LDS2 ? VGeo<3, EB3>::LDS2 : VGeo<4, EB4>::LDS2;
    constexpr int M = VGeo<4, EB4>::M;
    static_assert(M >= VGeo<3, EB3>::M, "operators of both degrees");
    __shared__ alignas(16) double lds[L];
    __shared__ alignas(16) double sDh[M], sD[M];
    __shared__ double s_alpha[1];
    if ((int)blockIdx.x < g3)
        volume_body<3, EB3, VOL_LW, false, false, false>(a3, blockIdx.x, lds, sDh, sD, s_alpha);
    else
        volume_body<4, EB4, VOL_LW, false, false, false>(a4, blockIdx.x - g3, lds, sDh, sD, s_alpha);
}

__global__ __launch_bounds__(kSurfBlock) void k_surface_pair(KArgs a3, KArgs a4, int g3) {
    if ((int)blockIdx.x < g3)
        surface_body<3, false, false, false, false, true>(a3, blockIdx.x);
    else
        surface_body<4, false, false, false, false, true>(a4, blockIdx.x - g3);
}

__global__ __launch_bounds__(kFinalizeWave) void k_finalize_pair(FinArgs f3, FinArgs f4, int n3) {
    if ((int)blockIdx.x < n3)
        finalize_body<3>(f3, blockIdx.x);
    else
        finalize_body<4>(f4, blockIdx.x - n3);
}

// Initialisation of the device integrator state of every instance.
// adaptive: dt_initial, tolerances and epsilon = (1, 1, 1) of the adaptive loop
// (solve_lwfr's set_dt!(integrator, dt_initial); LWIntegrator, lwfr.jl:162-168)
__global__ void k_init_state(DevState* st_all, int ninst, double t0, double tf, double cfl, const int* cur,
                             int adaptive, double dt0, double abstol, double reltol) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= ninst) return;
    DevState* st = st_all + k;
    st->t = t0;
    st->dt = 0.0;
    st->adaptive = adaptive;
    st->nfail = 0;
    st->nreject = 0;
    st->eps[0] = st->eps[1] = st->eps[2] = 1.0;
    st->abstol = abstol;
    st->reltol = reltol;
    if (adaptive) st->dt = (t0 + dt0 > tf) ? tf - t0 : dt0;
    st->t_final = tf;
    st->cfl = cfl;
    st->query = 0.0;
    st->finished = julia_isapprox(t0, tf);
    st->cur = cur[k];
    st->bad_state = 0;
    st->iter = 0;
}

__global__ void k_clear_bad_state(DevState* st_all, int ninst) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < ninst) st_all[k].bad_state = 0;
}

}  // namespace tlw
