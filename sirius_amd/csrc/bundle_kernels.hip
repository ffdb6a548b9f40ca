// bundle_kernels.hip — ray bundles: each pixel's ray with its geodesic deviation.
//
// The reference follows two deviation vectors xi_1, xi_2 (seeded along the camera's right and
// up axes) beside the central ray with D^2 xi / dlam^2 = R^mu_{nu rho sigma} k^nu xi^rho k^sigma,
// either with a tidal approximation or a finite-difference Riemann tensor
// (RDOP002A.cu:4239-4354, 5014-5047, 5364-5439), and reads the beam's ellipse off their Gram
// matrix. Here the deviation is the linearisation of the ray's own flow: in Hamiltonian form
// the geodesic deviation equation is the tangent (variational) equation of
// (dx/dlam, dp/dlam) = (dH/dp, -dH/dx), so the two deviation vectors are the derivatives of
// the state (x^mu, p_mu) with respect to the image coordinates (u, v) of the ray's pixel. They
// are carried by dual numbers: the camera, the initial state and every DP45 step run on
// Dual<double, 1> values seeded with d/du, and again with d/dv, so each accepted step advances the
// deviation by the exact derivative of that step's map (its length held; the length is chosen
// on the central ray alone). At the end the derivative of the outcome follows: of the escape
// direction (theta, phi) for an escaped ray (rad per pixel), or of the equatorial hit point
// (X, Y) for a ray ending on the thin disk (M per pixel), the deviation there projected along
// the ray onto the plane.
//
// Two lanes per ray, one per image axis, FP64 values and tangents.
#include <hip/hip_runtime.h>

#include "../../include/sirius_hip.h"
#include "geodesic.hpp"
#include "sirius_bundle.hpp"

namespace sirius {

namespace {

SIRIUS_HD __forceinline__ int find_cam(const CamConst* cams, int n_cam, int64_t id) {
    int c = 0;
    while (c + 1 < n_cam && cams[c + 1].offset <= id) ++c;
    return c;
}

// Escape angles of the final state (x, p) of the ray through the image point (u, v), as the
// trace's outputs define them (the wormhole's orbital plane depends on the pixel).
template <int FAM>
SIRIUS_HD __forceinline__ void escape_angles(const CamConst& c, const Spacetime<double>& s, double u, double v,
                                             const double x[4], const double p[4], double& th, double& ph) {
    double k[4];
    raise_index<double, FAM>(s, x, p, k);
    double dir[3];
    if constexpr (FAM == 1) {
        double ns[3];
        camera_dir_uv<double>(c, u, v, ns);
        double nt = sqrt(ns[1] * ns[1] + ns[2] * ns[2]);
        double e2[3];
        for (int i = 0; i < 3; ++i) e2[i] = nt > 1e-300 ? (ns[1] * c.et[i] + ns[2] * c.ep[i]) / nt : c.et[i];
        double l = x[1], psi = x[2], r = sqrt(l * l + c.b0 * c.b0);
        double drdl = (l / r) * k[1], rdpsi = p[2] / r;
        double cp = cos(psi), sp = sin(psi);
        for (int i = 0; i < 3; ++i) {
            double e = cp * c.er[i] + sp * e2[i], t = -sp * c.er[i] + cp * e2[i];
            dir[i] = drdl * e + rdpsi * t;
        }
    } else {
        dir[0] = k[1];
        dir[1] = k[2];
        dir[2] = k[3];
    }
    double n = sqrt(dir[0] * dir[0] + dir[1] * dir[1] + dir[2] * dir[2]);
    th = acos(fmin(1.0, fmax(-1.0, dir[2] / n)));
    ph = atan2(dir[1], dir[0]);
}

// Difference scale for the escape direction along a deviation t at state y: a perturbation of
// 1e-4 pixel, or less where the deviation has grown, so that eps |t| stays below 1e-6 of the
// state's scale.
SIRIUS_HD __forceinline__ double fd_eps(const double x[4], const double p[4], const double t[8]) {
    double ys = 1.0, tn = 0.0;
    for (int i = 1; i < 4; ++i) ys = fmax(ys, fabs(x[i]));
    for (int i = 0; i < 8; ++i) tn = fmax(tn, fabs(t[i]));
    double eps = 1e-4;
    if (tn * eps > 1e-6 * ys) eps = 1e-6 * ys / tn;
    return eps;
}

// Footprint of a 2x2 Jacobian m (rows: the two outcome coordinates in an orthonormal frame;
// columns: d/du, d/dv) for a circle of radius `size` pixels: semi-axes and the major axis's
// angle from the frame's first axis.
SIRIUS_HD __forceinline__ void ellipse_of(const double m[2][2], double size, float* beam3) {
    const double g00 = size * size * (m[0][0] * m[0][0] + m[0][1] * m[0][1]);
    const double g11 = size * size * (m[1][0] * m[1][0] + m[1][1] * m[1][1]);
    const double g01 = size * size * (m[0][0] * m[1][0] + m[0][1] * m[1][1]);
    const double tr = g00 + g11, det = g00 * g11 - g01 * g01;
    const double disc = sqrt(fmax(0.0, tr * tr - 4.0 * det));
    beam3[0] = (float)sqrt(fmax(0.5 * (tr + disc), 0.0));
    beam3[1] = (float)sqrt(fmax(0.5 * (tr - disc), 0.0));
    beam3[2] = (float)(0.5 * atan2(2.0 * g01, g00 - g11));
}

}  // namespace

// One pair of neighbouring lanes per ray: lane 0 of the pair carries the deviation d/du, lane 1 d/dv,
// in one Dual<double, 1> state each. The value parts of both lanes are the same instructions on the
// same numbers, so the pair takes the same decisions and stays together; what the pair does twice
// is the values' third of a dual step. Both axes in one lane, one pass after the other, spilled
// 212-364 bytes per lane (the state, two tangents and their derivatives beside seven stages).
// A wave's rays that end on the disk are landed together, and the escape angles differenced
// together, after its last ray has ended. Bound by FP64 issue and by the longest ray's steps: 641x361
// Kerr rays at the FP32 path's tolerances take 1.18 ms in squares with the near-critical rays first (1.83 in rows
// and raster order, 2.15 also with the Lambda terms; spill-free at one wave per SIMD); one lane per
// ray took 4.74 (5.89 also with IEEE roots and divisions).
template <int FAM, int EMIT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_trace_bundle(
    const CamConst* __restrict__ cams, int n_cam, TraceParams tp, BundleParams bp, BundleOut bo,
    const int32_t* __restrict__ order, const int32_t* __restrict__ first, const uint32_t* __restrict__ first_count) {
    int64_t id = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 1;
    const int axis = threadIdx.x & 1;
    if (id >= bo.n) return;
    if (order) {
        const int64_t nf = *first_count;
        id = id < nf ? first[id] : order[id - nf];
    }
    const CamConst& c = cams[find_cam(cams, n_cam, id)];
    if (!traces_camera<double, FAM>(c)) return;
    const int64_t pix = order ? id - c.offset : tile_pixel(c.width, c.height, TILE_SQUARE, id - c.offset);
    id = c.offset + pix;
    const double u0 = (double)(pix % c.width) + 0.5, v0 = (double)(pix / c.width) + 0.5;
    using D = Dual<double, 1>;
    const Spacetime<double> s = make_spacetime<double>(c);
    D X[4], P[4];
    Der<D> dA;  // FSAL derivative at the step's start
    {
        D u(u0), v(v0);
        u.d[0] = axis == 0 ? 1.0 : 0.0;
        v.d[0] = axis == 1 ? 1.0 : 0.0;
        init_state_uv<D>(c, s, u, v, X, P);
        X[0].d[0] = 0.0;  // nothing depends on t: its tangent is not carried (here and below)
        eval<D, FAM>(s, X, P, dA);
    }
    auto values = [](const D a[4], double o[4]) {
        for (int i = 0; i < 4; ++i) o[i] = a[i].v;
    };
    double h = tp.h_init, r0;
    {
        double x[4];
        values(X, x);
        r0 = event_radius(s, x);
    }
    if (tp.far_slope > 0) h = fmax(h, fmax(tp.h_max, r0 * tp.far_slope));
    int cls = SIRIUS_RAY_MAX_STEPS;
    double th_land = 0.0;  // fraction of the step at which a disk ray ends
    uint32_t attempts = 0;
    while (attempts < (uint32_t)tp.max_steps) {
        double hmax = tp.h_max;
        if (tp.far_slope > 0) hmax = fmax(hmax, r0 * tp.far_slope);
        D X1[4], P1[4], err[4];
        Der<D> d1;
        dp45_step<D, FAM, true>(s, X, P, dA, h, X1, P1, d1, err, true);
        ++attempts;
        double e = 0;
        for (int i = 0; i < 4; ++i) {
            const double q = err[i].v * rcp_t(fmax(tp.atol, 1e-70) + tp.rtol * fabs(X1[i].v));
            e += q * q;
        }
        e = sqrt(0.25 * e);
        if (!(e <= 1.0)) {
            h = next_step(h, e, tp.h_min, hmax);
            if (!sfinite(e) || h <= tp.h_min) { cls = SIRIUS_RAY_FAILED; break; }
            continue;
        }
        double x1[4];
        values(X1, x1);
        bool bad = false;
        for (int i = 0; i < 4; ++i) bad |= !sfinite(x1[i]) || !sfinite(P1[i].v);
        if (bad) { cls = SIRIUS_RAY_FAILED; break; }
        // thin disk: first crossing inside [r_in, r_out]
        if constexpr (is_ks(FAM) && EMIT == SIRIUS_EMISSION_THIN_DISK) {
            if (X[3].v * x1[3] < 0) {
                double x[4], k0[4], k1[4], xc[4];
                values(X, x);
                values(dA.k, k0);
                values(d1.k, k1);
                const double th = locate_event(s, EV_Z, 0.0, x, k0, x1, k1, h);
                hermite(x, k0, x1, k1, h, th, xc);
                const double rc = kerr_r(s, xc[1], xc[2], xc[3]);
                if (rc >= c.r_in && rc <= c.r_out) {
                    th_land = th;
                    cls = SIRIUS_RAY_DISK;
                    break;
                }
            }
        }
        double r1;
        if constexpr (FAM == FAM_KS_FLAT) r1 = d1.r.v;
        else r1 = event_radius(s, x1);
        if (is_ks(FAM) && r1 < c.r_cap) { cls = SIRIUS_RAY_CAPTURED; break; }
        // accepted: the state, its tangent and the FSAL derivative advance
        for (int i = 0; i < 4; ++i) { X[i] = X1[i]; P[i] = P1[i]; }
        X[0].d[0] = 0.0;
        dA = d1;
        r0 = r1;
        if (r1 > tp.r_escape) {
            const double radial = (FAM == 1) ? x1[1] * d1.k[1].v : x1[1] * d1.k[1].v + x1[2] * d1.k[2].v + x1[3] * d1.k[3].v;
            if (radial > 0) { cls = SIRIUS_RAY_ESCAPED; break; }
        }
        h = next_step(h, e, tp.h_min, hmax);
    }
    // derivative of the outcome along this lane's axis
    double j0 = 0.0, j1 = 0.0;
    double x[4], p[4];
    values(X, x);
    values(P, p);
    if (EMIT == SIRIUS_EMISSION_THIN_DISK && cls == SIRIUS_RAY_DISK) {
        // landed with a DP45 step to the plane; the deviation of the hit point goes along the ray
        // onto the plane z = 0
        D XL[4], PL[4], el[4];
        Der<D> dl;
        dp45_step<D, FAM, true>(s, X, P, dA, th_land * h, XL, PL, dl, el, false);
        const double kz = dl.k[3].v;
        const double dz = fabs(kz) > 1e-300 ? XL[3].d[0] / kz : 0.0;
        j0 = XL[1].d[0] - dz * dl.k[1].v;
        j1 = XL[2].d[0] - dz * dl.k[2].v;
    } else if (cls == SIRIUS_RAY_ESCAPED) {
        // the escape direction (a closed-form function of the final state and, for the wormhole, of
        // the image point) differentiated along the deviation
        double t[8];
        for (int i = 0; i < 4; ++i) { t[i] = X[i].d[0]; t[4 + i] = P[i].d[0]; }
        const double eps = fd_eps(x, p, t);
        double ang[2][2];
        for (int sg = 0; sg < 2; ++sg) {
            const double e3 = sg ? -eps : eps;
            double xs[4], ps[4];
            for (int i = 0; i < 4; ++i) {
                xs[i] = x[i] + e3 * t[i];
                ps[i] = p[i] + e3 * t[4 + i];
            }
            escape_angles<FAM>(c, s, u0 + (axis == 0 ? e3 : 0.0), v0 + (axis == 1 ? e3 : 0.0), xs, ps, ang[sg][0],
                               ang[sg][1]);
        }
        double dph = ang[0][1] - ang[1][1];
        dph = remainder(dph, 2.0 * M_PI);
        j0 = (ang[0][0] - ang[1][0]) / (2.0 * eps);
        j1 = dph / (2.0 * eps);
    }
    // both lanes hold the whole Jacobian; lane 0 of the pair writes the ray's outputs
    const double o0 = __shfl_xor(j0, 1), o1 = __shfl_xor(j1, 1);
    if (axis) return;
    const double jac[4] = {j0, o0, j1, o1};
    bo.cls[id] = (uint8_t)cls;
    uint8_t flags = 0;
    float beam[3] = {0.f, 0.f, 0.f};
    if (cls == SIRIUS_RAY_ESCAPED || cls == SIRIUS_RAY_DISK) {
        double m[2][2] = {{jac[0], jac[1]}, {jac[2], jac[3]}};
        if (cls == SIRIUS_RAY_ESCAPED) {
            // (theta, phi) -> the orthonormal sky frame (e_theta, e_phi)
            double th, ph;
            escape_angles<FAM>(c, s, u0, v0, x, p, th, ph);
            m[1][0] *= sin(th);
            m[1][1] *= sin(th);
        }
        ellipse_of(m, bp.size, beam);
        bool fin = true;
        for (int i = 0; i < 4; ++i) fin &= sfinite(jac[i]);
        if (!fin || !(beam[0] >= bp.min_size) || !(beam[0] <= bp.max_ratio * fmax(beam[1], 1e-30f)))
            flags |= SIRIUS_BUNDLE_TERMINATED;
    } else {
        flags |= SIRIUS_BUNDLE_TERMINATED;
    }
    bo.flags[id] = flags;
    for (int i = 0; i < 4; ++i) bo.jac[(int64_t)i * bo.n + id] = (float)jac[i];
    for (int i = 0; i < 3; ++i) bo.beam[(int64_t)i * bo.n + id] = beam[i];
}

hipError_t launch_trace_bundle(int family, int emission, const CamConst* cams, int n_cam, const TraceParams& tp,
                               const BundleParams& bp, const BundleOut& bo, const int32_t* order, const int32_t* first,
                               const uint32_t* first_count, hipStream_t st) {
    if (bo.n <= 0) return hipSuccess;
    const dim3 grid((unsigned)((2 * bo.n + 63) / 64)), block(64);  // two lanes per ray
    const bool disk = emission == SIRIUS_EMISSION_THIN_DISK;
    if (family == 1)
        hipLaunchKernelGGL((k_trace_bundle<1, 0>), grid, block, 0, st, cams, n_cam, tp, bp, bo, order, first, first_count);
    else if (family == 2)
        hipLaunchKernelGGL((k_trace_bundle<2, 0>), grid, block, 0, st, cams, n_cam, tp, bp, bo, order, first, first_count);
    else if (family == FAM_KS_FLAT && disk)
        hipLaunchKernelGGL((k_trace_bundle<FAM_KS_FLAT, SIRIUS_EMISSION_THIN_DISK>), grid, block, 0, st, cams, n_cam, tp, bp, bo, order, first, first_count);
    else if (family == FAM_KS_FLAT)
        hipLaunchKernelGGL((k_trace_bundle<FAM_KS_FLAT, 0>), grid, block, 0, st, cams, n_cam, tp, bp, bo, order, first, first_count);
    else if (disk)
        hipLaunchKernelGGL((k_trace_bundle<0, SIRIUS_EMISSION_THIN_DISK>), grid, block, 0, st, cams, n_cam, tp, bp, bo, order, first, first_count);
    else
        hipLaunchKernelGGL((k_trace_bundle<0, 0>), grid, block, 0, st, cams, n_cam, tp, bp, bo, order, first, first_count);
    return hipGetLastError();
}

}  // namespace sirius
