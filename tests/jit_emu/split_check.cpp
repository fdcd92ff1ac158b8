// CPU check of the factors that 2x2 gates are split into: their product against
// the gate in extended precision, and its norm, over random gates; no worse than
// the factors by angles (split_1q_rotations with keep_grouping). Test
// infrastructure.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "lq_gates.hpp"
#include "lq_plan.hpp"

using namespace lqamd;
using cl = std::complex<long double>;
struct M2 {
    cl a[4];
};

static M2 times(const M2 &x, const M2 &y) {
    M2 r;
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) r.a[2 * i + j] = x.a[2 * i] * y.a[j] + x.a[2 * i + 1] * y.a[2 + j];
    return r;
}

static M2 of(const LOp &o) {
    if (o.kind == TOP_DIAG) return {{cl(o.coef[0]), 0.0L, 0.0L, cl(o.coef[1])}};
    return {{cl(o.coef[0]), cl(o.coef[1]), cl(o.coef[2]), cl(o.coef[3])}};
}

int main() {
    const std::vector<GateId> families[] = {{GateId::Rot},
                                            {GateId::RX},
                                            {GateId::RZ, GateId::RY, GateId::RZ},
                                            {GateId::RX, GateId::RY, GateId::RZ},
                                            {GateId::Hadamard, GateId::RX, GateId::RZ, GateId::RY}};
    int failures = 0;
    for (size_t f = 0; f < sizeof(families) / sizeof(families[0]); ++f) {
        long double err[2] = {0, 0}, norm[2] = {0, 0};
        const int N = 20000;
        for (int keep = 0; keep < 2; ++keep) {
            std::mt19937 rng(11 + static_cast<unsigned>(f));
            std::uniform_real_distribution<double> U(-3.14, 3.14);
            for (int i = 0; i < N; ++i) {
                std::vector<LOp> q;
                for (GateId g : families[f]) {
                    const uint32_t w = 0;
                    const double v[3] = {U(rng), U(rng), U(rng)};
                    LOp o = lower_gate(2, g, &w, 1, nullptr, nullptr, 0, false, v);
                    if (!try_merge_1q(q, o)) q.push_back(o);
                }
                if (q.size() != 1) {
                    std::printf("family %zu: not one gate\n", f);
                    return 2;
                }
                const M2 gate = of(q[0]);
                split_1q_rotations(q, keep != 0);
                M2 m = {{1.0L, 0.0L, 0.0L, 1.0L}};
                for (const LOp &o : q) m = times(of(o), m);
                long double e = 0, n = 0;
                for (int k = 0; k < 4; ++k) {
                    e += std::norm(m.a[k] - gate.a[k]);
                    n += std::norm(m.a[k]);
                }
                err[keep] += e;
                norm[keep] += (n / 2 - 1) * (n / 2 - 1);
            }
        }
        const bool ok = err[0] <= err[1] && norm[0] <= norm[1];
        std::printf("family %zu: from the gate %.3Le (by angles %.3Le), norm %.3Le (%.3Le)%s\n", f, sqrtl(err[0] / N),
                    sqrtl(err[1] / N), sqrtl(norm[0] / N), sqrtl(norm[1] / N), ok ? "" : " WORSE");
        failures += !ok;
    }
    // a phase of a few units in the last place stays
    for (double a : {1.6e-15, -1.6e-15}) {
        const uint32_t w = 0;
        std::vector<LOp> q;
        const double th = 0.7;
        q.push_back(lower_gate(2, GateId::RY, &w, 1, nullptr, nullptr, 0, false, &th));
        LOp p = lower_gate(2, GateId::RZ, &w, 1, nullptr, nullptr, 0, false, &a);
        if (!try_merge_1q(q, p)) return 2;
        const M2 gate = of(q[0]);
        split_1q_rotations(q);
        M2 m = {{1.0L, 0.0L, 0.0L, 1.0L}};
        for (const LOp &o : q) m = times(of(o), m);
        if (std::fabs(static_cast<double>(m.a[2].imag() - gate.a[2].imag())) > 0.3 * std::fabs(static_cast<double>(gate.a[2].imag()))) {
            std::printf("phase %.1e lost: %.3Le of %.3Le\n", a, m.a[2].imag(), gate.a[2].imag());
            ++failures;
        }
    }
    std::printf("%d failures\n", failures);
    return failures ? 1 : 0;
}
