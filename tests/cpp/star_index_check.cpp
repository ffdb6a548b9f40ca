// The celestial spheres' star index (sirius_amd/csrc/starfield.cpp, star_cell_index) on the host, as the library
// holds it. Catalogues of many sizes and spreads, uniform, about the poles and about the phi = +-pi seam.
// For an index: its offsets and lists are in order, and for directions over the whole sphere, at the
// poles, on the seam, and inside and at the edge of the stars' cuts, every star that passes its cut by
// the device's float cosine is in the list of the cell that the device's float arithmetic picks. And
// which catalogues have one: none whose lists would hold more than a sixteenth of the catalogue on
// average, all of those well below. Prints the catalogues and "OK".
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

namespace sirius {
std::vector<int32_t> star_cell_index(const std::vector<float>& rec, int n);
}

constexpr int REC = 12, NT = 128, NP = 256;

static int cell_of(float th, float ph) {
    int it = (int)(th * (float)(NT / 3.141592653589793));
    int ip = (int)((ph + 3.14159265f) * (float)(NP / 6.283185307179586));
    return std::min(std::max(it, 0), NT - 1) * NP + std::min(std::max(ip, 0), NP - 1);
}

int main() {
    std::mt19937_64 g(3);
    std::uniform_real_distribution<double> u(-1.0, 1.0);
    long checked = 0, lit = 0, indexed = 0, walked = 0;
    for (int where = 0; where < 3; ++where)
        for (int n : {1, 2, 7, 100, 1000, 4096})
            for (double cut : {5e-6, 1e-3, 0.02, 0.1, 0.2, 0.3, 0.8, 1.6, 4.0}) {
                std::vector<float> rec((size_t)n * REC, 0.f);
                for (int i = 0; i < n; ++i) {
                    double z = u(g), ph = M_PI * u(g);
                    if (where == 1) z = (i % 2 ? 1 : -1) * std::cos(i < 2 ? 0.0 : 0.4 * u(g));
                    if (where == 2) ph = i ? M_PI + 0.02 * u(g) : M_PI;
                    const double s = std::sqrt(std::max(0.0, 1 - z * z));
                    float* r = rec.data() + (size_t)i * REC;
                    r[0] = (float)(s * std::cos(ph)); r[1] = (float)(s * std::sin(ph)); r[2] = (float)z;
                    r[3] = cut >= M_PI ? -2.0f : (float)std::cos(cut);
                    r[4] = (float)(cut * cut / 28);
                }
                const std::vector<int32_t> idx = sirius::star_cell_index(rec, n);
                if (idx.empty()) {
                    ++walked;
                    if (cut <= 0.1 && where != 1) return std::printf("no index: place %d, %d stars, cut %g\n", where, n, cut), 1;
                    continue;
                }
                ++indexed;
                const int32_t *list = idx.data() + NT * NP + 1, total = idx[NT * NP];
                if (idx.size() != (size_t)(NT * NP + 1 + total) || idx[0] != 0) return std::puts("layout"), 1;
                if (16LL * total > (long long)n * NT * NP) return std::printf("long lists: place %d, %d stars, cut %g: %d entries\n", where, n, cut, total), 1;
                for (int c = 0; c < NT * NP; ++c) {
                    if (idx[c + 1] < idx[c]) return std::puts("offsets"), 1;
                    for (int j = idx[c]; j < idx[c + 1]; ++j)
                        if (list[j] < 0 || list[j] >= n || (j > idx[c] && list[j] <= list[j - 1])) return std::puts("order"), 1;
                }
                auto look = [&](float th, float ph) {
                    const double t = th, p = ph;
                    const float vx = (float)(std::sin(t) * std::cos(p)), vy = (float)(std::sin(t) * std::sin(p)), vz = (float)std::cos(t);
                    const int c = cell_of(th, ph);
                    ++checked;
                    for (int i = 0; i < n; ++i) {
                        const float* r = rec.data() + (size_t)i * REC;
                        const float m0 = vx * r[0], m1 = vy * r[1], m2 = vz * r[2];
                        if ((m0 + m1) + m2 < r[3]) continue;
                        ++lit;
                        if (!std::binary_search(list + idx[c], list + idx[c + 1], i)) {
                            std::printf("place %d, %d stars, cut %g: star %d missing from the cell of (%.9g, %.9g)\n", where, n, cut, i, th, ph);
                            return false;
                        }
                    }
                    return true;
                };
                const int any = n <= 100 ? 20000 : 400;
                for (int k = 0; k < any; ++k)
                    if (!look((float)std::acos(u(g)), (float)(M_PI * u(g)))) return 1;
                for (float th : {0.f, 1e-7f, 1e-3f, 1.5707964f, 3.1405926f, 3.1415925f, 3.1415927f})
                    for (float ph : {-3.1415927f, -3.1415925f, -1e-7f, 0.f, 1.f, 3.1415925f, 3.1415927f})
                        if (!look(th, ph)) return 1;
                for (int k = 0; k < 400; ++k) {  // around a star, inside its cut and at its edge
                    const float* r = rec.data() + (size_t)(g() % n) * REC;
                    const double a = std::min(cut, M_PI) * (k % 2 ? 1.0 + 1e-6 * u(g) : std::fabs(u(g))), b = M_PI * u(g);
                    const double st = std::hypot(r[0], r[1]), ct = r[2], cp = st > 0 ? r[0] / st : 1, sp = st > 0 ? r[1] / st : 0;
                    const double lx = std::sin(a) * std::cos(b), ly = std::sin(a) * std::sin(b), lz = std::cos(a);
                    const double x0 = ct * lx + st * lz, z = -st * lx + ct * lz, x = cp * x0 - sp * ly, y = sp * x0 + cp * ly;
                    if (!look((float)std::atan2(std::hypot(x, y), z), (float)std::atan2(y, x))) return 1;
                }
            }
    std::printf("%ld catalogues with an index, %ld without, %ld directions, %ld stars in them\n", indexed, walked, checked, lit);
    if (indexed > 60 && walked > 40 && lit > 100000) std::puts("OK");
    return 0;
}
