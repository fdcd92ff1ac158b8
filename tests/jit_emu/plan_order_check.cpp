// CPU check of the order in which plans run their ops: random programs of gates
// and dots are planned as the engine plans them, the passes interpreted op by
// op on the host, and the states and every dot compared with the ops applied
// one after the other. Test infrastructure.
//
//   plan_order_check FAMILY SEEDS
//   words:      rotations, CNOT and CRX, then words of X, Y and Z on neighbouring wires
//   cz:         the same with runs of CZ in either order of its wires, CCZ and phases
//   nonunitary: operators that are not unitary among the gates (one to three wires, with
//               and without controls, zeroing generators), dots after and between them
//   long:       8000 gates in one pass, on a few wires and on all; planning takes at most
//               24 times as long as for 1000 gates (8 times the ops; 64 if pair by pair)
//   partial:    two and three states, gates on some of them only, dots between them
// Each program is planned on 12 to 14 qubits, with one to three states, plain and with
// split rotations, and with the grouping of either precision. Exit status 0 when nothing
// is off by more than 1e-10 of the states' norms: a split gate is exact to 1e-13 of its
// amplitudes, and no program has more than 200 gates.
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "lq_gates.hpp"
#include "lq_plan.hpp"

using namespace lqamd;
using State = std::vector<cd>;

// One op by its targets, controls and table, whatever form it came in.
struct Action {
    std::vector<int> bits;         // dense: targets, the first the local MSB
    const cd *m = nullptr;         // dense: 2^k x 2^k
    uint64_t cmask = 0, cval = 0;  // amplitudes it acts on
    bool zero = false;             // zero the others
    bool dense = false;
    std::vector<cd> factor;        // otherwise: one factor per amplitude
};

static void act(std::vector<State> &S, const Action &a, bool dot, uint32_t smask, uint32_t sa, uint32_t sb, cd *out) {
    const uint64_t N = S[0].size();
    auto image = [&](const State &v) {
        State r(N, cd(0.0));
        if (!a.dense) {
            for (uint64_t i = 0; i < N; ++i)
                if ((i & a.cmask) == a.cval) r[i] = a.factor[i] * v[i];
            return r;
        }
        const int k = static_cast<int>(a.bits.size()), K = 1 << k;
        for (uint64_t i = 0; i < N; ++i) {
            if ((i & a.cmask) != a.cval) continue;
            int row = 0;
            uint64_t base = i;
            for (int j = 0; j < k; ++j) {
                row |= static_cast<int>((i >> a.bits[j]) & 1) << (k - 1 - j);
                base &= ~(1ull << a.bits[j]);
            }
            cd s(0.0);
            for (int c = 0; c < K; ++c) {
                uint64_t at = base;
                for (int j = 0; j < k; ++j)
                    if ((c >> (k - 1 - j)) & 1) at |= 1ull << a.bits[j];
                s += a.m[row * K + c] * v[at];
            }
            r[i] = s;
        }
        return r;
    };
    if (dot) {
        const State r = image(S[sa]);
        cd s(0.0);
        for (uint64_t i = 0; i < N; ++i) s += std::conj(S[sb][i]) * r[i];
        *out = s;
        return;
    }
    for (size_t s = 0; s < S.size(); ++s) {
        if (!((smask >> s) & 1u)) continue;
        State r = image(S[s]);
        if (!a.zero)
            for (uint64_t i = 0; i < N; ++i)
                if ((i & a.cmask) != a.cval) r[i] = S[s][i];
        S[s].swap(r);
    }
}

static void program_order(std::vector<State> &S, const std::vector<LOp> &prog, std::vector<cd> &dots) {
    const uint64_t N = S[0].size();
    for (const LOp &o : prog) {
        Action a;
        a.cmask = o.cmask;
        a.cval = o.cval & o.cmask;
        a.zero = (o.flags & TF_ZERO_UNCTRL) != 0;
        if (o.kind == TOP_DENSE1 || o.kind == TOP_DENSE2 || o.kind == TOP_DENSEK) {
            a.dense = true;
            a.bits.assign(o.bits, o.bits + o.k);
            a.m = o.coef.data();
        } else {
            a.factor.resize(N);
            for (uint64_t i = 0; i < N; ++i) {
                uint64_t idx = 0;
                for (int j = 0; j < o.k; ++j) idx |= ((i >> o.bits[j]) & 1ull) << (o.k - 1 - j);
                if (o.kind == TOP_PARITY) idx = static_cast<uint64_t>(__builtin_popcountll(i & o.pmask) & 1);
                else if (o.kind == TOP_PCPHASE) idx = idx < o.pc_dim ? 0 : 1;
                a.factor[i] = o.coef[idx];
            }
        }
        act(S, a, o.is_dot(), o.smask, o.sa, o.sb, o.is_dot() ? &dots[static_cast<size_t>(o.slot)] : nullptr);
    }
}

static void planned_order(std::vector<State> &S, int n, const std::vector<PassPlan> &plan, std::vector<cd> &dots) {
    const uint64_t N = 1ull << n;
    for (const PassPlan &p : plan) {
        auto spread = [&](uint32_t local) {
            uint64_t g = 0;
            for (size_t b = 0; b < p.tbits.size(); ++b)
                if ((local >> b) & 1u) g |= 1ull << p.tbits[b];
            return g;
        };
        auto run = [&](const TileOp &t, const TileStage *st) {
            Action a;
            a.zero = (t.flags & TF_ZERO_UNCTRL) != 0;
            if (st || p.dense) {
                a.cmask = t.gcmask;
                a.cval = t.gcval;
            } else {
                a.cmask = spread(t.lcmask) | t.ocmask;
                a.cval = spread(t.lcval) | t.ocval;
            }
            const cd *c = p.coef.data() + t.coef_off;
            if (t.kind == TOP_DENSE1 || t.kind == TOP_DENSE2 || t.kind == TOP_DENSEK) {
                a.dense = true;
                a.bits.assign(t.gpos, t.gpos + t.k);
                a.m = c;
            } else {
                const uint64_t pm = st ? t.gpmask : spread(t.lxmask) | t.omask;
                a.factor.resize(N);
                for (uint64_t i = 0; i < N; ++i) {
                    uint64_t idx = 0;
                    for (uint32_t j = 0; j < t.k && t.kind != TOP_RPHASE; ++j) idx |= ((i >> t.gpos[j]) & 1ull) << (t.k - 1 - j);
                    cd f(1.0);
                    switch (t.kind) {
                    case TOP_DIAG: f = c[idx]; break;
                    case TOP_PCPHASE: f = c[idx < t.pc_dim ? 0 : 1]; break;
                    case TOP_PARITY: f = c[__builtin_popcountll(i & pm) & 1]; break;
                    case TOP_SIGN: f = -1.0; break;
                    case TOP_CZSET: {
                        int flips = 0;
                        for (uint32_t z = 0; z < t.nz; ++z) flips += __builtin_popcountll(i & (i >> t.sd[z]) & t.sm[z]);
                        f = (flips & 1) ? -1.0 : 1.0;
                        break;
                    }
                    case TOP_TPHASE:
                        for (uint32_t j = 0; j < t.k; ++j) f *= c[2 * j + ((i >> t.gpos[j]) & 1ull)];
                        break;
                    case TOP_RPHASE: {
                        uint32_t e = 0;
                        for (uint32_t j = 0; j < t.k; ++j) e |= static_cast<uint32_t>((i >> p.tbits[static_cast<size_t>(st->rbits[j])]) & 1ull) << j;
                        f = c[e];
                        break;
                    }
                    default: std::printf("unexpected op kind %u\n", t.kind); std::exit(2);
                    }
                    a.factor[i] = f;
                }
            }
            const bool dot = (t.flags & TF_DOT) != 0;
            act(S, a, dot, t.smask, t.sa, t.sb, dot ? &dots[static_cast<size_t>(p.slot_ids[t.slot])] : nullptr);
        };
        if (!p.reg) {
            for (const TileOp &t : p.ops) run(t, nullptr);
            continue;
        }
        for (const TileStage &st : p.stages)
            for (uint32_t i = st.op_begin; i < st.op_end; ++i) run(p.ops[i], st.kind == STAGE_REG ? &st : nullptr);
    }
}

struct Builder {
    int n, ns;
    std::mt19937 rng;
    std::vector<LOp> prog, queue; // gates wait in a queue, merged there, until dots read the state
    int slots = 0;
    Builder(int n_, int ns_, unsigned seed) : n(n_), ns(ns_), rng(seed) {}
    uint32_t below(uint32_t m) { return rng() % m; }
    double angle() { return std::uniform_real_distribution<double>(0.0, 6.28)(rng); }
    uint32_t all() const { return (1u << ns) - 1u; }
    std::vector<uint32_t> wires(int k) {
        std::vector<uint32_t> w;
        while (static_cast<int>(w.size()) < k) {
            const uint32_t x = below(static_cast<uint32_t>(n));
            bool seen = false;
            for (uint32_t y : w) seen |= y == x;
            if (!seen) w.push_back(x);
        }
        return w;
    }
    void push(LOp op, uint32_t smask) {
        op.smask = smask;
        if (!try_merge_1q(queue, op)) queue.push_back(std::move(op));
    }
    void flush() {
        for (LOp &o : queue) prog.push_back(std::move(o));
        queue.clear();
    }
    void gate(GateId g, const std::vector<uint32_t> &w, uint32_t smask, const std::vector<uint32_t> &ctrl = {}) {
        std::vector<double> p(4);
        for (double &x : p) x = angle();
        const std::vector<uint8_t> cv(ctrl.size(), 1);
        push(lower_gate(n, g, w.data(), static_cast<int>(w.size()), ctrl.data(), cv.data(), static_cast<int>(ctrl.size()),
                        false, p.data()), smask);
    }
    void matrix(std::vector<cd> m, const std::vector<uint32_t> &w, uint32_t smask, uint32_t ctrl = ~0u) {
        std::vector<int> tb;
        for (uint32_t x : w) tb.push_back(phys_bit(n, x));
        const uint64_t cm = ctrl == ~0u ? 0ull : 1ull << phys_bit(n, ctrl);
        push(lower_matrix(std::move(m), tb, cm, cm, false), smask);
    }
    void add_dot(LOp d, uint32_t sa, uint32_t sb) {
        flush();
        d.flags = (d.flags & ~TF_ZERO_UNCTRL) | TF_DOT;
        d.sa = sa;
        d.sb = sb;
        d.slot = slots++;
        prog.push_back(std::move(d));
    }
    // <sb| P_a P_b |sa> with a letter on each of two neighbouring wires
    void word(uint32_t w, int a, int b, uint32_t sa, uint32_t sb) {
        const cd I(0.0, 1.0);
        const std::vector<cd> P[3] = {{0, 1, 1, 0}, {0, -I, I, 0}, {1, 0, 0, -1}};
        std::vector<cd> m(16);
        for (int r = 0; r < 4; ++r)
            for (int c = 0; c < 4; ++c) m[4 * r + c] = P[a][2 * (r >> 1) + (c >> 1)] * P[b][2 * (r & 1) + (c & 1)];
        add_dot(lower_matrix(m, {phys_bit(n, w), phys_bit(n, w + 1)}, 0, 0, true), sa, sb);
    }
    void generator(GateId g, uint32_t w, uint32_t sa, uint32_t sb) {
        double s;
        add_dot(lower_generator(n, g, &w, 1, nullptr, nullptr, 0, &s), sa, sb);
    }
};

static void gates(Builder &b, int count, bool cz, bool partial) {
    const GateId one[] = {GateId::RX, GateId::RY, GateId::RZ, GateId::Rot, GateId::Hadamard, GateId::PhaseShift};
    for (int i = 0; i < count; ++i) {
        uint32_t sm = b.all();
        if (partial && b.below(3) == 0) sm = 1u + b.below(b.all());
        const uint32_t pick = b.below(cz ? 12u : 8u);
        if (pick < 5) b.gate(one[b.below(6)], b.wires(1), sm);
        else if (pick < 7) b.gate(GateId::CNOT, b.wires(2), sm);
        else if (pick < 8) b.gate(GateId::CRX, b.wires(2), sm);
        else if (pick < 11) {
            const std::vector<uint32_t> w = b.wires(2);
            b.gate(GateId::CZ, w, sm);
            if (b.below(2)) b.gate(GateId::CZ, b.below(2) ? std::vector<uint32_t>{w[1], w[0]} : b.wires(2), sm);
            if (b.below(3) == 0) b.gate(GateId::CZ, {w[1], w[0]}, sm);
        } else {
            const std::vector<uint32_t> w = b.wires(3);
            b.gate(GateId::PauliZ, {w[0]}, sm, {w[1], w[2]});
        }
    }
}

static void not_unitary(Builder &b, uint32_t sm) {
    const cd I(0.0, 1.0);
    switch (b.below(5)) {
    case 0: b.matrix({0.5, 0, 0, 1.3 * I}, b.wires(1), sm); break;
    case 1: b.matrix({0.7, 0.4, -0.2 * I, 1.1}, b.wires(1), sm); break;
    case 2: {
        const std::vector<uint32_t> w = b.wires(2);
        b.matrix({0.9, 0.2, 0.1, 1.2}, {w[0]}, sm, w[1]);
        break;
    }
    case 3: {
        const int K = b.below(2) ? 4 : 8;
        std::vector<cd> m(static_cast<size_t>(K) * K);
        for (int r = 0; r < K; ++r)
            for (int c = 0; c < K; ++c) m[static_cast<size_t>(r) * K + c] = (r == c ? 0.9 : 0.0) + 0.1 * std::polar(1.0, b.angle());
        b.matrix(m, b.wires(K == 4 ? 2 : 3), sm);
        break;
    }
    default: {
        // a controlled gate's generator: zero outside its control's subspace
        const std::vector<uint32_t> w = b.wires(2);
        const uint8_t one = 1;
        double s;
        b.push(lower_generator(b.n, GateId::RX, &w[0], 1, &w[1], &one, 1, &s), sm);
    }
    }
}

// Gates of a program for the family "long".
static std::vector<LOp> long_program(int n, int wires, int count) {
    Builder b(n, 1, 41);
    b.n = wires; // gates on the first wires, lowered for n qubits below
    std::vector<LOp> prog;
    const GateId one[] = {GateId::RX, GateId::RZ, GateId::Rot};
    while (static_cast<int>(prog.size()) < count) {
        const bool two = b.below(2) != 0;
        const std::vector<uint32_t> w = b.wires(two ? 2 : 1);
        const double p[3] = {b.angle(), b.angle(), b.angle()};
        LOp op = lower_gate(n, two ? GateId::CNOT : one[b.below(3)], w.data(), static_cast<int>(w.size()), nullptr, nullptr,
                            0, false, p);
        if (!try_merge_1q(prog, op)) prog.push_back(std::move(op));
    }
    return prog;
}

static int long_passes() {
    int wrong = 0;
    for (int wires : {4, 12}) {
        PlanConfig cfg;
        cfg.n = 12;
        cfg.kt_max = 12;
        cfg.reg_rb = 4;
        cfg.max_dots = 32;
        cfg.budget = 1e9;
        double best[2] = {1e9, 1e9};
        std::vector<PassPlan> plan;
        for (int k = 0; k < 2; ++k) {
            const std::vector<LOp> prog = long_program(12, wires, k ? 8000 : 1000);
            for (int r = 0; r < 5; ++r) {
                const auto t = std::chrono::steady_clock::now();
                plan = plan_passes(prog, cfg);
                best[k] = std::min(best[k], std::chrono::duration<double>(std::chrono::steady_clock::now() - t).count());
            }
            std::vector<State> ref(1, State(1ull << 12)), got;
            ref[0][5] = 1.0;
            got = ref;
            std::vector<cd> none;
            program_order(ref, prog, none);
            planned_order(got, 12, plan, none);
            double err = 0.0;
            for (size_t i = 0; i < ref[0].size(); ++i) err = std::max(err, std::abs(ref[0][i] - got[0][i]));
            const bool ok = err <= 1e-10 && plan.size() == 1;
            std::printf("%d wires, %zu gates: %zu passes, off by %.1e, planned in %.2f ms\n", wires, prog.size(), plan.size(),
                        err, best[k] * 1e3);
            wrong += !ok;
        }
        if (!(best[1] <= 24.0 * best[0])) {
            std::printf("%d wires: planning is not linear in the gates\n", wires);
            ++wrong;
        }
    }
    std::printf("long: 4 plans, %d wrong\n", wrong);
    return wrong ? 1 : 0;
}

int main(int argc, char **argv) {
    const std::string family = argc > 1 ? argv[1] : "words";
    const unsigned seeds = argc > 2 ? static_cast<unsigned>(std::atoi(argv[2])) : 100;
    if (family == "long") return long_passes();
    int wrong = 0, plans = 0;
    double worst = 0.0;
    for (unsigned seed = 0; seed < seeds; ++seed) {
        Builder b(12 + static_cast<int>(seed % 5 == 3) + 2 * static_cast<int>(seed % 10 == 7),
                  family == "partial" ? 2 + static_cast<int>(seed & 1) : 1 + static_cast<int>(seed & 1), 977 * seed + 3);
        const uint32_t bra = b.ns > 1 ? 1u : 0u;
        const bool cz = family == "cz", partial = family == "partial";
        auto words = [&](int count) {
            for (int i = 0; i < count; ++i) {
                const uint32_t w = b.below(static_cast<uint32_t>(b.n - 1)), s = 1 + b.below(static_cast<uint32_t>(b.ns));
                b.word(w, static_cast<int>(b.below(3)), static_cast<int>(b.below(3)), 0, s <= bra ? s : bra);
            }
        };
        if (family == "words" || cz) {
            gates(b, 40 + static_cast<int>(b.below(60)), cz, false);
            // dots one after the other, or with phases and a few gates between them
            for (int i = 0; i < 12; ++i) {
                words(1);
                if (seed % 3 == 1) b.gate(GateId::RZ, b.wires(1), b.all());
                if (seed % 6 == 1 && i % 3 == 2) gates(b, 2, cz, false);
            }
            if (seed % 3 == 0) {
                gates(b, 30, cz, false);
                for (uint32_t w = 0; w < 6; ++w) b.generator(w % 2 ? GateId::RX : GateId::RZ, w, 0, bra);
            }
        } else if (family == "nonunitary") {
            for (int part = 0; part < 3; ++part) {
                gates(b, 15, false, false);
                not_unitary(b, b.all());
                if (part != 1) words(5);
            }
        } else if (partial) {
            for (int part = 0; part < 4; ++part) {
                gates(b, 12, false, true);
                words(4);
                b.generator(GateId::RY, b.below(static_cast<uint32_t>(b.n)), 0, b.below(static_cast<uint32_t>(b.ns)));
            }
        } else {
            std::printf("unknown family %s\n", family.c_str());
            return 2;
        }
        b.flush();
        std::vector<State> start(static_cast<size_t>(b.ns), State(1ull << b.n));
        for (State &s : start) {
            double norm = 0.0;
            for (cd &v : s) {
                v = cd(std::normal_distribution<double>()(b.rng), std::normal_distribution<double>()(b.rng));
                norm += std::norm(v);
            }
            for (cd &v : s) v /= std::sqrt(norm);
        }
        std::vector<State> ref = start;
        std::vector<cd> ref_dots(static_cast<size_t>(b.slots));
        program_order(ref, b.prog, ref_dots);
        for (int form = 0; form < 4; ++form) {
            const bool split = form & 1, keep = form & 2;
            PlanConfig cfg;
            cfg.n = b.n;
            cfg.ns = b.ns;
            cfg.dense_passes = true;
            cfg.keep_grouping = keep;
            // tiles of 12 bits with one or two states, of 11 with three (specialised passes)
            cfg.kt_max = b.ns > 2 ? 11 : 12;
            cfg.reg_rb = cfg.kt_max - 8;
            cfg.max_dots = 32;
            cfg.low_bits = 4;
            cfg.budget = seed % 4 == 0 ? 1e9 : split ? 52.0 : 24.0;
            cfg.lookahead = split;
            cfg.scale_rotations = split;
            if (keep) cfg.max_scale_growth = 1e20;
            std::vector<LOp> prog = b.prog;
            if (split) split_1q_rotations(prog, keep);
            std::vector<State> got = start;
            std::vector<cd> got_dots(static_cast<size_t>(b.slots), cd(1e9));
            planned_order(got, b.n, plan_passes(prog, cfg), got_dots);
            double state_err = 0.0, dot_err = 0.0, norm = 1.0;
            for (size_t s = 0; s < ref.size(); ++s) {
                double q = 0.0;
                for (const cd &v : ref[s]) q += std::norm(v);
                norm = std::max(norm, q);
                for (size_t i = 0; i < ref[s].size(); ++i) state_err = std::max(state_err, std::abs(ref[s][i] - got[s][i]));
            }
            for (size_t d = 0; d < ref_dots.size(); ++d) dot_err = std::max(dot_err, std::abs(ref_dots[d] - got_dots[d]));
            const double err = std::max(state_err, dot_err) / norm;
            ++plans;
            worst = std::max(worst, err);
            if (!(err <= 1e-10)) {
                ++wrong;
                if (wrong <= 12)
                    std::printf("%s seed %u, %d qubits, %d states, split %d, keep %d: states off by %.1e, dots by %.1e\n",
                                family.c_str(), seed, b.n, b.ns, split, keep, state_err, dot_err);
            }
        }
    }
    std::printf("%s: %d plans, %d wrong, worst %.1e\n", family.c_str(), plans, wrong, worst);
    return wrong ? 1 : 0;
}
