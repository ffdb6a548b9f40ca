// Host build of the event locator of the FP64 paths and of the FP32 symplectic integrator
// (sirius_amd/csrc/geodesic.hpp, locate_event) against bisection of the same cubic Hermite interpolant
// to the last bit: random steps over the plane z = 0 and over spheres of the
// event radius, and steps on which Newton's iteration is slow or runs in circles (triple roots, nearly
// flat crossings, pairs of iterates that map to each other). An event is in place if the function changes
// sign within 1e-11 of the step of it (the iteration ends on a step of 1e-12, whose error is the square
// where it converges fast; slower, it halves the bracket; FP32: 1e-6 and 2e-7), or if the function there
// is rounding: below 64 units of 2^-53 (2^-24) of its terms. Prints the cases and "OK".
#include "../../sirius_amd/csrc/geodesic.hpp"

#include <cmath>
#include <cstdio>
#include <random>

using namespace sirius;

template <class T>
static Spacetime<T> spacetime(double a) {
    CamConst c{};
    c.M = 1.0;
    c.a = a;
    return make_spacetime<T>(c);
}

template <class T>
struct Step {
    T x0[4] = {}, k0[4] = {}, x1[4] = {}, k1[4] = {}, h = 1;
    // component i: the cubic c0 + c1 t + c2 t^2 + c3 t^3 of the step's fraction
    void set(int i, double c0, double c1, double c2, double c3) {
        x0[i] = (T)c0;
        x1[i] = (T)(c0 + c1 + c2 + c3);
        k0[i] = (T)(c1 / h);
        k1[i] = (T)((c1 + 2 * c2 + 3 * c3) / h);
    }
};

template <class T>
static T value(const Spacetime<T>& s, int kind, T target, const Step<T>& q, T th) {
    T x[4];
    hermite(q.x0, q.k0, q.x1, q.k1, q.h, th, x);
    return event_value(s, kind, x, target);
}

static long cases = 0;
template <class T>
static bool in_place(const Spacetime<T>& s, int kind, T target, const Step<T>& q, const char* what) {
    const T f0 = value(s, kind, target, q, T(0)), f1 = value(s, kind, target, q, T(1));
    if (!(f0 < 0 != f1 < 0) || f0 == 0 || f1 == 0) return true;
    ++cases;
    const T th = locate_event(s, kind, target, q.x0, q.k0, q.x1, q.k1, q.h);
    T scale = std::fabs(target);
    for (int i = 1; i < 4; ++i)
        scale = std::fmax(scale, std::fabs(q.x0[i]) + std::fabs(q.x1[i]) + q.h * (std::fabs(q.k0[i]) + std::fabs(q.k1[i])));
    const T f = value(s, kind, target, q, th), eps = sizeof(T) == 8 ? T(1e-11) : T(1e-6);
    if (std::fabs(f) <= 64 * std::ldexp(scale, sizeof(T) == 8 ? -53 : -24)) return true;
    const T lo = std::fmax(T(0), th - eps), hi = std::fmin(T(1), th + eps);
    if (th >= 0 && th <= 1 && (value(s, kind, target, q, lo) < 0) != (value(s, kind, target, q, hi) < 0)) return true;
    T a = 0, b = 1;
    for (int it = 0; it < 60; ++it) {
        const T m = T(0.5) * (a + b);
        if ((value(s, kind, target, q, m) < 0) == (f0 < 0)) a = m; else b = m;
    }
    std::printf("%s (%zu bytes): located at %.17g (value %.3g), bisection %.17g\n", what, sizeof(T), (double)th, (double)f, (double)a);
    return false;
}

template <class T>
static bool all_in_place() {
    std::mt19937_64 g(7);
    std::uniform_real_distribution<double> u(-1.0, 1.0);
    const Spacetime<T> flat = spacetime<T>(0.0), kerr = spacetime<T>(0.9);
    bool ok = true;
    for (int i = 0; i < 200000; ++i) {  // any cubic that changes sign
        Step<T> q;
        q.h = std::exp(3 * u(g));
        q.set(3, u(g), 2 * u(g), 3 * u(g), 3 * u(g));
        ok = ok && in_place(flat, EV_Z, T(0), q, "plane");
    }
    for (int i = 0; i < 20000; ++i) {  // (t - r)^3 + e (t - r): flat at the root
        const double r = 0.5 + 0.49 * u(g), e = i % 2 ? 0.0 : std::exp(10 * u(g) - 12), c = std::exp(8 * u(g));
        Step<T> q;
        q.set(3, c * (-r * r * r - e * r), c * (3 * r * r + e), c * (-3 * r), c);
        ok = ok && in_place(flat, EV_Z, T(0), q, "flat root");
    }
    for (int i = 0; i < 20000; ++i) {  // 2 t^3 - ... around a point: Newton's two-cycles of t^3 - 2 t + 2 and its relatives
        const double p = 0.5 + 0.4 * u(g), w = 0.05 + 0.2 * std::fabs(u(g)), b = 1.9 + 0.2 * u(g), d = 2 + 0.2 * u(g);
        // y = (t - p) / w; f = y^3 - b y + d
        const double y0 = -p / w, iw = 1 / w;
        Step<T> q;
        q.set(3, y0 * y0 * y0 - b * y0 + d, iw * (3 * y0 * y0 - b), 3 * y0 * iw * iw, iw * iw * iw);
        ok = ok && in_place(flat, EV_Z, T(0), q, "two-cycle");
    }
    for (int i = 0; i < 100000; ++i) {  // spheres: curved, nearly tangential and radial steps
        const Spacetime<T>& s = i % 2 ? kerr : flat;
        const double target = std::exp(2.5 + 2.5 * u(g)), len = target * std::exp(2 * u(g) - 1);
        Step<T> q;
        q.h = std::exp(2 * u(g));
        for (int k = 1; k < 4; ++k) q.set(k, target * 1.5 * u(g), len * u(g), len * u(g), 0.5 * len * u(g));
        ok = ok && in_place(s, EV_R, T(target), q, "sphere");
        Step<T> t;  // straight past the sphere at almost its radius
        const double bb = target * (1 - std::exp(6 * u(g) - 8));
        t.set(1, bb, 0, 0, 0);
        t.set(2, -target * std::fabs(u(g)) * 0.5, 2 * target, 0, 0);
        t.set(3, 0.1 * target * u(g), 0, 0, 0);
        ok = ok && in_place(s, EV_R, T(target), t, "tangent");
    }
    return ok;
}

int main() {
    const bool ok = all_in_place<double>() && all_in_place<float>();
    std::printf("%ld events\n", cases);
    if (ok) std::puts("OK");
    return ok ? 0 : 1;
}
