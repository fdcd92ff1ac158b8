// Lowering and pass planning (host).
//
// Gate semantics follow the reference: controls select the subspace
// ctrl == value (GateImplementationsLM.hpp:407-440); generators zero the
// non-control subspace (:2181-2228); MultiRZ is a parity phase (:1988-2010);
// PCPhase is a threshold phase on the local index (:2113-2162).
//
// Planning: ops form a DAG in which two ops commute when every bit they share
// is acted on diagonally by both (controls, diagonal targets), or when both
// are read-only dots. A pass greedily takes ready ops whose non-diagonal bits
// fit in its tile (at most kt_max bits, the low bits always included), up to
// a compute budget; diagonal ops fit any pass. A dot passes only unitary ops,
// whatever their bits: it reads every amplitude of its states.
#include "lq_kernels.hpp"
#include "lq_plan.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <queue>
#include <set>

namespace lqamd {

namespace {
inline int popc(uint64_t x) { return __builtin_popcountll(x); }

bool all_zero(const std::vector<cd> &m) {
    for (const auto &x : m)
        if (x != cd(0.0)) return false;
    return true;
}
bool is_identity(const std::vector<cd> &m, int d) {
    for (int r = 0; r < d; ++r)
        for (int c = 0; c < d; ++c)
            if (m[static_cast<size_t>(r) * d + c] != (r == c ? cd(1.0) : cd(0.0))) return false;
    return true;
}
bool is_diagonal(const std::vector<cd> &m, int d) {
    for (int r = 0; r < d; ++r)
        for (int c = 0; c < d; ++c)
            if (r != c && m[static_cast<size_t>(r) * d + c] != cd(0.0)) return false;
    return true;
}
} // namespace

uint64_t LOp::target_mask() const {
    uint64_t m = 0;
    for (int j = 0; j < k; ++j) m |= 1ull << bits[j];
    return m;
}

uint64_t LOp::nmask() const {
    switch (kind) {
    case TOP_DENSE1:
    case TOP_DENSE2:
    case TOP_DENSEK: return target_mask();
    case TOP_PAULI: return xmask;
    default: return 0;
    }
}

uint64_t LOp::dmask() const {
    uint64_t m = cmask;
    switch (kind) {
    case TOP_DIAG:
    case TOP_PCPHASE: m |= target_mask(); break;
    case TOP_PARITY: m |= pmask; break;
    case TOP_PAULI: m |= yzmask & ~xmask; break;
    default: break;
    }
    return m;
}

bool LOp::is_swap() const {
    static const cd kX[4] = {0.0, 1.0, 1.0, 0.0};
    static const cd kSwap[16] = {1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 1.0};
    if (kind == TOP_DENSE1) return coef.size() == 4 && std::equal(coef.begin(), coef.end(), kX);
    return kind == TOP_DENSE2 && coef.size() == 16 && std::equal(coef.begin(), coef.end(), kSwap);
}

uint32_t LOp::dot_class() const {
    if (!is_dot()) return 0;
    const cd one(1.0), zero(0.0), im(0.0, 1.0);
    if (kind == TOP_DENSE1 && coef.size() == 4 && coef[0] == zero && coef[3] == zero) {
        if (coef[1] == one && coef[2] == one) return TF_DOT_X;
        if (coef[1] == -im && coef[2] == im) return TF_DOT_Y;
    }
    if (((kind == TOP_DIAG && k == 1) || kind == TOP_PARITY) && coef.size() == 2 && coef[0] == one && coef[1] == -one)
        return TF_DOT_Z;
    if (kind == TOP_DIAG && k == 0 && coef.size() == 1 && coef[0] == one) return TF_DOT_Z; // no bits: the identity
    return 0;
}

bool LOp::is_unitary(double tol, int max_k) const {
    if (flags & TF_ZERO_UNCTRL) return false;
    switch (kind) {
    case TOP_DIAG:
    case TOP_PARITY:
    case TOP_PCPHASE:
    case TOP_PAULI:
        for (const cd &v : coef)
            if (!(std::fabs(std::norm(v) - 1.0) <= tol)) return false;
        return true;
    case TOP_DENSE1:
    case TOP_DENSE2:
    case TOP_DENSEK: break;
    default: return false;
    }
    const size_t d = static_cast<size_t>(1) << k;
    if (k > max_k || k > 6 || coef.size() != d * d) return false;
    // rows against rows; those without a column that both fill need no product
    // (a gate that leaves most basis states alone has rows of one entry)
    uint64_t filled[64];
    for (size_t a = 0; a < d; ++a) {
        filled[a] = 0;
        for (size_t c = 0; c < d; ++c)
            if (coef[a * d + c] != cd(0.0)) filled[a] |= 1ull << c; // NaN too
    }
    typedef double v2 __attribute__((vector_size(16))); // (re, im)
    auto load = [&](size_t i) {
        v2 x;
        std::memcpy(&x, &coef[i], sizeof(x));
        return x;
    };
    for (size_t a = 0; a < d; ++a)
        for (size_t b = a; b < d; ++b) {
            if (!(filled[a] & filled[b]) && a != b) continue;
            v2 p[2] = {}, q[2] = {}; // u v, and u times v with its parts exchanged
            for (size_t c = 0; c < d; c += 2)
                for (size_t j = 0; j < 2; ++j) {
                    const v2 u = load(a * d + c + j), v = load(b * d + c + j);
                    p[j] += u * v;
                    q[j] += u * v2{v[1], v[0]};
                }
            const v2 ps = p[0] + p[1], qs = q[0] + q[1];
            const double re = ps[0] + ps[1] - (a == b ? 1.0 : 0.0), im = qs[0] - qs[1];
            if (!(re * re + im * im <= tol * tol)) return false;
        }
    return true;
}

double LOp::cost() const {
    double c = 0.5;
    switch (kind) {
    case TOP_DENSE1: c = (flags & TF_REAL) ? 0.5 : 1.0; break; // real rotations take half the arithmetic
    case TOP_DENSE2: c = 2.5; break;
    case TOP_DENSEK: c = static_cast<double>(1 << k) / 2.0; break;
    case TOP_DIAG: c = (k == 1 && cmask == 0) ? 0.15 : 0.5; break; // one-bit phases share a table per stage
    case TOP_PARITY: c = 0.4; break;
    case TOP_PCPHASE: c = 0.5; break;
    case TOP_PAULI: c = 0.6; break;
    default: break;
    }
    if (is_dot()) return c + 0.5;
    return c * std::max(1, popc(smask));
}

LOp lower_matrix(std::vector<cd> mat, std::vector<int> tbits, uint64_t cmask, uint64_t cval, bool gen) {
    int k = static_cast<int>(tbits.size());
    LQ_ABORT_IF(mat.size() != (static_cast<size_t>(1) << (2 * k)), "The size of matrix does not match with the given number of wires");
    bool changed = true;
    while (changed && k > 0) {
        changed = false;
        for (int j = 0; j < k && !changed; ++j) {
            const int d = 1 << k, h = d / 2, lb = k - 1 - j;
            bool offzero = true;
            for (int r = 0; r < d && offzero; ++r)
                for (int c = 0; c < d; ++c)
                    if ((((r >> lb) ^ (c >> lb)) & 1) && mat[static_cast<size_t>(r) * d + c] != cd(0.0)) {
                        offzero = false;
                        break;
                    }
            if (!offzero) continue;
            std::vector<cd> A(static_cast<size_t>(h) * h), B(static_cast<size_t>(h) * h);
            auto ins = [lb](int x, int v) { return ((x >> lb) << (lb + 1)) | (v << lb) | (x & ((1 << lb) - 1)); };
            for (int r = 0; r < h; ++r)
                for (int c = 0; c < h; ++c) {
                    A[static_cast<size_t>(r) * h + c] = mat[static_cast<size_t>(ins(r, 0)) * d + ins(c, 0)];
                    B[static_cast<size_t>(r) * h + c] = mat[static_cast<size_t>(ins(r, 1)) * d + ins(c, 1)];
                }
            int ctrl = -1;
            std::vector<cd> *keep = nullptr;
            if (A == B) {
                keep = &A;
            } else if (!gen && is_identity(A, h)) {
                keep = &B;
                ctrl = 1;
            } else if (!gen && is_identity(B, h)) {
                keep = &A;
                ctrl = 0;
            } else if (gen && all_zero(A)) {
                keep = &B;
                ctrl = 1;
            } else if (gen && all_zero(B)) {
                keep = &A;
                ctrl = 0;
            }
            if (!keep) continue;
            if (ctrl >= 0) {
                cmask |= 1ull << tbits[j];
                if (ctrl) cval |= 1ull << tbits[j];
            }
            mat = *keep;
            tbits.erase(tbits.begin() + j);
            --k;
            changed = true;
        }
    }
    LOp op;
    op.cmask = cmask;
    op.cval = cval;
    op.k = k;
    for (int j = 0; j < k; ++j) op.bits[j] = tbits[j];
    const int d = 1 << k;
    if (k == 0 || is_diagonal(mat, d)) {
        LQ_ABORT_IF(k > kMaxTileOpTargets, "diagonal operator on too many wires");
        op.kind = TOP_DIAG;
        op.coef.resize(d);
        for (int i = 0; i < d; ++i) op.coef[i] = mat[static_cast<size_t>(i) * d + i];
        return op;
    }
    LQ_ABORT_IF(k > 10, "dense operators are supported on at most 10 wires");
    op.kind = k == 1 ? TOP_DENSE1 : k == 2 ? TOP_DENSE2 : TOP_DENSEK;
    op.coef = std::move(mat);
    return op;
}

namespace {
void controls_to_mask(int n, const uint32_t *ctrls, const uint8_t *cvals, int nc, uint64_t *cm, uint64_t *cv) {
    *cm = 0;
    *cv = 0;
    for (int i = 0; i < nc; ++i) {
        const int b = phys_bit(n, ctrls[i]);
        *cm |= 1ull << b;
        if (cvals == nullptr || cvals[i]) *cv |= 1ull << b;
    }
}
} // namespace

namespace {
// Lowered forms of the gates without parameters and of the generators, made
// once on bits 0..nw-1 (wires[j] on bit nw-1-j): lowering one of them is then a
// copy with its bits put in place.
struct Template {
    bool known = false;
    LOp op;
    double scale = 0.0;
};
constexpr int kGates = static_cast<int>(GateId::Count);

LOp place_template(const LOp &t, const int *tb, int nw, uint64_t cm, uint64_t cv) {
    LOp op = t;
    for (int j = 0; j < op.k; ++j) op.bits[j] = tb[nw - 1 - t.bits[j]];
    op.cmask = cm;
    op.cval = cv;
    for (int j = 0; j < nw; ++j) {
        const uint64_t from = 1ull << (nw - 1 - j), to = 1ull << tb[j];
        if (t.cmask & from) op.cmask |= to;
        if (t.cval & from) op.cval |= to;
    }
    return op;
}

const Template &gate_template(GateId g, bool inverse) {
    static const std::vector<Template> table = [] {
        std::vector<Template> t(2 * kGates);
        for (int i = 0; i < kGates; ++i) {
            const GateInfo &info = gate_info(static_cast<GateId>(i));
            if (info.nparams != 0 || info.nwires < 1 || info.nwires > 4 || static_cast<GateId>(i) == GateId::Identity)
                continue;
            std::vector<int> tb;
            for (int j = 0; j < info.nwires; ++j) tb.push_back(info.nwires - 1 - j);
            for (int inv = 0; inv < 2; ++inv) {
                Template &x = t[2 * i + inv];
                x.op = lower_matrix(gate_matrix(static_cast<GateId>(i), nullptr, inv != 0, info.nwires), tb, 0, 0, false);
                x.known = true;
            }
        }
        return t;
    }();
    return table[2 * static_cast<size_t>(g) + (inverse ? 1 : 0)];
}

const Template &generator_template(GateId g) {
    static const std::vector<Template> table = [] {
        std::vector<Template> t(kGates);
        for (int i = 0; i < kGates; ++i) {
            const GateInfo &info = gate_info(static_cast<GateId>(i));
            if (!info.has_generator || info.nwires < 1 || info.nwires > 4) continue;
            std::vector<int> tb;
            for (int j = 0; j < info.nwires; ++j) tb.push_back(info.nwires - 1 - j);
            Generator gen = gate_generator(static_cast<GateId>(i), info.nwires);
            t[i].op = lower_matrix(gen.g, tb, 0, 0, true);
            t[i].scale = gen.scale;
            t[i].known = true;
        }
        return t;
    }();
    return table[static_cast<size_t>(g)];
}
} // namespace

LOp lower_gate(int n, GateId g, const uint32_t *wires, int nw, const uint32_t *ctrls, const uint8_t *cvals, int nc,
               bool inverse, const double *params) {
    if (const Template &t = gate_template(g, inverse); t.known && nw == gate_info(g).nwires) {
        uint64_t cm, cv;
        controls_to_mask(n, ctrls, cvals, nc, &cm, &cv);
        int tb[4];
        for (int j = 0; j < nw; ++j) tb[j] = phys_bit(n, wires[j]);
        return place_template(t.op, tb, nw, cm, cv);
    }
    uint64_t cm, cv;
    controls_to_mask(n, ctrls, cvals, nc, &cm, &cv);
    std::vector<int> tb(nw);
    for (int j = 0; j < nw; ++j) tb[j] = phys_bit(n, wires[j]);
    const cd I1(0.0, 1.0);
    if (g == GateId::MultiRZ) {
        LOp op;
        op.kind = TOP_PARITY;
        op.cmask = cm;
        op.cval = cv;
        for (int b : tb) op.pmask |= 1ull << b;
        const cd first = std::exp(-I1 * (params[0] / 2)), second = std::exp(I1 * (params[0] / 2));
        op.coef = {inverse ? std::conj(first) : first, inverse ? std::conj(second) : second};
        return op;
    }
    if (g == GateId::PCPhase) {
        LQ_ABORT_IF(nw > kMaxTileOpTargets, "PCPhase is supported on at most 12 wires");
        const double dim = std::round(params[1]);
        LQ_ABORT_IF(dim < 0 || dim > std::ldexp(1.0, n),
                    "The dimension of the PCPhase gate must be a positive integer and less than or equal to statevector size.");
        LOp op;
        op.kind = TOP_PCPHASE;
        op.cmask = cm;
        op.cval = cv;
        op.k = nw;
        for (int j = 0; j < nw; ++j) op.bits[j] = tb[j];
        op.pc_dim = static_cast<uint64_t>(dim);
        const double ph = inverse ? -params[0] : params[0];
        op.coef = {std::exp(I1 * ph), std::exp(-I1 * ph)};
        return op;
    }
    if (g == GateId::GlobalPhase) {
        LOp op;
        op.kind = TOP_DIAG;
        op.k = 0;
        op.cmask = cm;
        op.cval = cv;
        op.coef = {std::exp(cd(0.0, inverse ? params[0] : -params[0]))};
        return op;
    }
    std::vector<cd> m = gate_matrix(g, params, inverse, nw);
    if (nw == 1 && m.size() == 4 && m[1] != cd(0.0) && m[2] != cd(0.0)) {
        // nothing for lower_matrix to take apart
        LOp op;
        op.kind = TOP_DENSE1;
        op.k = 1;
        op.bits[0] = tb[0];
        op.cmask = cm;
        op.cval = cv;
        op.coef = std::move(m);
        return op;
    }
    if (nw == 1 && m.size() == 4 && m[1] == cd(0.0) && m[2] == cd(0.0) && m[0] != m[3] && m[0] != cd(1.0) &&
        m[3] != cd(1.0)) {
        LOp op; // RZ
        op.kind = TOP_DIAG;
        op.k = 1;
        op.bits[0] = tb[0];
        op.cmask = cm;
        op.cval = cv;
        op.coef = {m[0], m[3]};
        return op;
    }
    return lower_matrix(std::move(m), tb, cm, cv, false);
}

LOp lower_generator(int n, GateId g, const uint32_t *wires, int nw, const uint32_t *ctrls, const uint8_t *cvals,
                    int nc, double *scale) {
    uint64_t cm, cv;
    controls_to_mask(n, ctrls, cvals, nc, &cm, &cv);
    if (const Template &t = generator_template(g); t.known && nw == gate_info(g).nwires) {
        int tb4[4];
        for (int j = 0; j < nw; ++j) tb4[j] = phys_bit(n, wires[j]);
        LOp op = place_template(t.op, tb4, nw, cm, cv);
        op.flags |= TF_ZERO_UNCTRL;
        *scale = t.scale;
        return op;
    }
    std::vector<int> tb(nw);
    for (int j = 0; j < nw; ++j) tb[j] = phys_bit(n, wires[j]);
    LOp op;
    if (g == GateId::MultiRZ) {
        op.kind = TOP_PARITY;
        op.cmask = cm;
        op.cval = cv;
        for (int b : tb) op.pmask |= 1ull << b;
        op.coef = {1.0, -1.0};
        *scale = -0.5;
    } else if (g == GateId::GlobalPhase) {
        op.kind = TOP_DIAG;
        op.k = 0;
        op.cmask = cm;
        op.cval = cv;
        op.coef = {1.0};
        *scale = -1.0;
    } else {
        Generator gen = gate_generator(g, nw);
        op = lower_matrix(gen.g, tb, cm, cv, true);
        *scale = gen.scale;
    }
    op.flags |= TF_ZERO_UNCTRL;
    return op;
}

namespace {
uint64_t touch_mask(const LOp &o) { return o.target_mask() | o.cmask | o.pmask | o.xmask | o.yzmask; }

bool single_bit_1q(const LOp &o) {
    return !o.is_dot() && !(o.flags & TF_ZERO_UNCTRL) && o.k == 1 && (o.kind == TOP_DENSE1 || o.kind == TOP_DIAG);
}

std::vector<cd> as_2x2(const LOp &o) {
    if (o.kind == TOP_DENSE1) return o.coef;
    return {o.coef[0], 0.0, 0.0, o.coef[1]};
}
} // namespace

size_t absorb_into_product(std::vector<LOp> &prog, std::vector<cd> &f) {
    const int nq = static_cast<int>(f.size() / 2);
    LQ_ABORT_IF(nq < 1 || nq > 64, "product state of unsupported size");
    const uint64_t all = nq == 64 ? ~0ull : ((1ull << nq) - 1ull);
    uint64_t blocked = 0;
    size_t folded = 0, i = 0;
    std::vector<LOp> rest;
    rest.reserve(prog.size());
    for (; i < prog.size() && blocked != all; ++i) {
        LOp &o = prog[i];
        const bool own = !o.is_dot() && !(o.flags & TF_ZERO_UNCTRL) && o.cmask == 0 && o.smask == 1u;
        if (own && o.kind == TOP_DIAG && o.k == 0 && o.coef.size() == 1) {
            f[0] *= o.coef[0];
            f[1] *= o.coef[0];
            ++folded;
            continue;
        }
        if (own && single_bit_1q(o) && o.bits[0] < nq && !((blocked >> o.bits[0]) & 1ull)) {
            const size_t q = static_cast<size_t>(o.bits[0]);
            const std::vector<cd> m = as_2x2(o);
            const cd a = f[2 * q], b = f[2 * q + 1];
            f[2 * q] = m[0] * a + m[1] * b;
            f[2 * q + 1] = m[2] * a + m[3] * b;
            ++folded;
            continue;
        }
        blocked |= o.is_dot() ? all : touch_mask(o);
        rest.push_back(std::move(o));
    }
    for (; i < prog.size(); ++i) rest.push_back(std::move(prog[i]));
    prog.swap(rest);
    return folded;
}

void split_1q_rotations(std::vector<LOp> &prog, bool keep_grouping) {
    std::vector<LOp> out;
    out.reserve(prog.size() * 3);
    for (auto &o : prog) {
        const bool candidate = (o.kind == TOP_DENSE1 || o.kind == TOP_DENSEK) && o.k == 1 && o.cmask == 0 &&
                               !o.is_dot() && !(o.flags & TF_ZERO_UNCTRL) && o.coef.size() == 4 &&
                               (keep_grouping || !o.is_swap());
        if (!candidate) {
            out.push_back(std::move(o));
            continue;
        }
        const cd u00 = o.coef[0], u01 = o.coef[1], u10 = o.coef[2], u11 = o.coef[3];
        // U = D2 R D1 with R = [[c, -s], [s, c]] from the entries of U, without
        // angles; D1 = diag(1, .) unless an entry vanishes. The signs go to c
        // and s (phases from one half of the plane), so that which phases are
        // exactly 1 or -1 depends on the kind of gate, not on its angles.
        // Formed in extended precision and rounded once: a phase taken as u / |u|
        // in double precision is off modulus one by its rounding. Over random Rot
        // gates the factors' product is 0.8e-16 off the gate and its norm 1.4e-16
        // off one; with phases in double precision 1.9e-16 and 1.9e-16, by angles
        // 2.0e-16 and 1.9e-16.
        double c = 0.0, sn = 0.0;
        cd d1_0(1.0), d1_1, d2_0, d2_1;
        using cl = std::complex<long double>;
        // one rounding next to 1, -1, i, -i does not count
        auto snap = [](cl ph) {
            constexpr long double kOne = 2.3e-16L;
            if (std::fabs(ph.imag()) <= kOne) return cl(ph.real() < 0.0L ? -1.0L : 1.0L, 0.0L);
            if (std::fabs(ph.real()) <= kOne) return cl(0.0L, ph.imag() < 0.0L ? -1.0L : 1.0L);
            return ph;
        };
        auto phase_of = [&](const cl &u, long double &m) {
            m = std::sqrt(std::norm(u));
            cl ph = snap(u / m);
            if (ph.real() < 0.0L || (ph.real() == 0.0L && ph.imag() < 0.0L)) {
                ph = -ph;
                m = -m;
            }
            return ph;
        };
        auto rounded = [](const cl &v) { return cd(static_cast<double>(v.real()), static_cast<double>(v.imag())); };
        auto size = [](const cd &u) { return std::max(std::fabs(u.real()), std::fabs(u.imag())); };
        if (!keep_grouping && size(u00) > 1e-100 && size(u10) > 1e-100 && size(u11) > 1e-100) {
            long double lc, ls, l11;
            const cl p0 = phase_of(cl(u00), lc), p1 = phase_of(cl(u10), ls);
            const cl p11 = phase_of(cl(u11), l11);
            const cl q = snap(p11 * std::conj(p1));
            c = static_cast<double>(lc);
            sn = static_cast<double>(ls);
            d2_0 = rounded(p0);
            d2_1 = rounded(p1);
            d1_1 = rounded((lc < 0.0L) != (l11 < 0.0L) ? -q : q);
        } else {
            const double gamma = std::arg(u00 * u11 - u01 * u10) / 2.0;
            const cd eg = std::polar(1.0, -gamma);
            const cd a = eg * u00, b = eg * u10;
            c = std::abs(a);
            sn = std::abs(b);
            const double pa = c > 1e-300 ? std::arg(a) : 0.0, pb = sn > 1e-300 ? std::arg(b) : 0.0;
            const double alpha = pb - pa, delta = -pa - pb;
            d1_0 = std::polar(1.0, -delta / 2);
            d1_1 = std::polar(1.0, delta / 2);
            d2_0 = std::polar(1.0, gamma - alpha / 2);
            d2_1 = std::polar(1.0, gamma + alpha / 2);
        }
        const cd r00 = d2_0 * c * d1_0, r01 = d2_0 * (-sn) * d1_1, r10 = d2_1 * sn * d1_0, r11 = d2_1 * c * d1_1;
        const double err = std::max(std::max(std::abs(r00 - u00), std::abs(r01 - u01)),
                                    std::max(std::abs(r10 - u10), std::abs(r11 - u11)));
        if (!(err <= 1e-13)) {
            out.push_back(std::move(o));
            continue;
        }
        LOp p1;
        p1.kind = TOP_DIAG;
        p1.k = 1;
        p1.bits[0] = o.bits[0];
        p1.coef = {d1_0, d1_1};
        p1.smask = o.smask;
        LOp rot = o;
        rot.kind = TOP_DENSE1;
        rot.flags |= TF_REAL;
        rot.coef = {cd(c), cd(-sn), cd(sn), cd(c)};
        LOp p2 = p1;
        p2.coef = {d2_0, d2_1};
        const cd one(1.0);
        if (keep_grouping || d1_0 != one || d1_1 != one) out.push_back(std::move(p1)); // RY has none
        out.push_back(std::move(rot));
        if (keep_grouping || d2_0 != one || d2_1 != one) out.push_back(std::move(p2));
    }
    // Move each one-bit phase later past the ops it commutes with (anything
    // acting diagonally on its bit or on other states) and fold it into the
    // next one-bit phase on the same bit, so that consecutive rotations on a
    // wire share one phase between them.
    auto is_phase = [](const LOp &o) {
        return o.kind == TOP_DIAG && o.k == 1 && o.cmask == 0 && !o.is_dot() && o.coef.size() == 2;
    };
    auto unit_phase = [](const LOp &o) {
        return std::fabs(std::norm(o.coef[0]) - 1.0) <= 1e-12 && std::fabs(std::norm(o.coef[1]) - 1.0) <= 1e-12;
    };
    // Walking backwards, a phase only has to look at the next op on its bit
    // that acts non-diagonally there or is a phase, and at what acts on other
    // states: per bit, the next op that a phase on it can meet.
    std::vector<char> gone(out.size(), 0);
    constexpr size_t kNone = static_cast<size_t>(-1);
    size_t next_on[64];
    size_t next_any = kNone; // next op or dot that stops phases of the common state set on every bit
    std::fill(next_on, next_on + 64, kNone);
    uint32_t common = 0;     // the states of the phases tracked
    std::vector<size_t> link(out.size(), kNone); // the op that phase i meets first
    for (size_t i = out.size(); i-- > 0;) {
        const LOp &o = out[i];
        if (is_phase(o)) {
            if (o.smask != common) {
                // phases on other states: nothing is known about the ops after it
                std::fill(next_on, next_on + 64, kNone);
                next_any = i + 1 < out.size() ? i + 1 : kNone;
                common = o.smask;
            }
            link[i] = std::min(next_on[o.bits[0]], next_any);
            next_on[o.bits[0]] = i;
            continue;
        }
        if (o.is_dot()) {
            const uint32_t ab = (1u << o.sa) | (1u << o.sb);
            if ((common & ab) != ab || keep_grouping) {
                if (common) next_any = i;
                continue;
            }
        } else if (o.smask != common) {
            if (common & o.smask) next_any = i;
            continue;
        }
        for (uint64_t m = o.nmask(); m; m &= m - 1) next_on[__builtin_ctzll(m)] = i;
    }
    for (size_t i = 0; i < out.size(); ++i) {
        if (!is_phase(out[i])) continue;
        size_t j = link[i];
        if (j == kNone || !is_phase(out[j]) || out[j].bits[0] != out[i].bits[0] || out[j].smask != out[i].smask) continue;
        if (keep_grouping && j - i >= 4096) continue;
        // past a dot only when unitary
        if (!unit_phase(out[i]) && std::any_of(out.begin() + static_cast<long>(i), out.begin() + static_cast<long>(j),
                                               [](const LOp &o) { return o.is_dot(); }))
            continue;
        out[j].coef[0] *= out[i].coef[0];
        out[j].coef[1] *= out[i].coef[1];
        gone[i] = 1;
    }
    prog.clear();
    for (size_t i = 0; i < out.size(); ++i)
        if (!gone[i]) prog.push_back(std::move(out[i]));
}

bool try_merge_1q(std::vector<LOp> &queue, const LOp &op) {
    if (!single_bit_1q(op)) return false;
    const uint64_t mine = touch_mask(op);
    const int lim = std::max(0, static_cast<int>(queue.size()) - 256);
    for (int i = static_cast<int>(queue.size()) - 1; i >= lim; --i) {
        LOp &q = queue[i];
        if (!(touch_mask(q) & mine)) continue;
        if (!single_bit_1q(q) || q.bits[0] != op.bits[0] || q.cmask != op.cmask || q.cval != op.cval ||
            q.smask != op.smask)
            return false;
        const auto a = as_2x2(op), b = as_2x2(q);
        std::vector<cd> m = {a[0] * b[0] + a[1] * b[2], a[0] * b[1] + a[1] * b[3], a[2] * b[0] + a[3] * b[2],
                             a[2] * b[1] + a[3] * b[3]};
        if (m[1] == cd(0.0) && m[2] == cd(0.0)) {
            q.kind = TOP_DIAG;
            q.coef = {m[0], m[3]};
        } else {
            q.kind = TOP_DENSE1;
            q.coef = m;
        }
        return true;
    }
    return false;
}

namespace {
// Ops of one stage of a register-kernel pass.
struct StagePlan {
    bool reg = false;
    uint32_t R = 0;       // tile-local register bits (register stages)
    std::vector<int> ops; // indices into the program
};

// Whether a dot may be taken before or after an op that it shares no
// non-diagonal bit with: <b|U^dagger G U|a> = <b|G|a> takes a unitary that acts
// on both states (an op on neither does not matter to it).
bool passes_dot(const LOp &op, bool unitary, const LOp &dot) {
    const uint32_t ab = (1u << dot.sa) | (1u << dot.sb);
    return !(op.smask & ab) || (unitary && (op.smask & ab) == ab);
}

// The ops ops[sel[0]], ops[sel[1]], ... that must come before others: two must
// keep their order when a bit they share is acted on non-diagonally by one of
// them, or when one is a dot that the other does not leave as it is; read-only
// dots commute with each other. Indices are places in sel; what follows from
// other pairs is left out, so the pairs are few. nm, dm: bits acted on
// non-diagonally and diagonally; unitary: of all ops, read where there are dots.
struct OpOrder {
    std::vector<std::vector<int>> succ;
    std::vector<int> indeg;
};

OpOrder order_ops(const std::vector<LOp> &ops, const std::vector<int> &sel, const std::vector<uint64_t> &nm,
                  const std::vector<uint64_t> &dm, const std::vector<char> &unitary, int n, int ns) {
    const int N = static_cast<int>(sel.size());
    OpOrder o;
    o.succ.resize(static_cast<size_t>(N));
    o.indeg.assign(static_cast<size_t>(N), 0);
    std::vector<int> mark(static_cast<size_t>(N), -1);
    struct BitDeps {
        int lastN = -1;
        std::vector<int> D, RN, RD;
    };
    std::vector<BitDeps> bd(static_cast<size_t>(n));
    // ops that a dot may not change places with on any bits, and the dots so far
    const bool has_dots = std::any_of(sel.begin(), sel.end(), [&](int i) { return ops[i].is_dot(); });
    const uint32_t all_states = (1u << ns) - 1u;
    std::vector<int> barriers, dots;
    for (int j = 0; j < N; ++j) {
        const LOp &op = ops[sel[j]];
        const bool dot = op.is_dot();
        auto dep = [&](int i) {
            if (i >= 0 && mark[i] != j) {
                mark[i] = j;
                o.succ[i].push_back(j);
                ++o.indeg[j];
            }
        };
        for (int b = 0; b < n; ++b) {
            const uint64_t bit = 1ull << b;
            BitDeps &s = bd[b];
            if (nm[sel[j]] & bit) {
                dep(s.lastN);
                if (!dot) {
                    for (int i : s.D) dep(i);
                    for (int i : s.RN) dep(i);
                    for (int i : s.RD) dep(i);
                    s.lastN = j;
                    s.D.clear();
                    s.RN.clear();
                    s.RD.clear();
                } else {
                    for (int i : s.D) dep(i);
                    s.RN.push_back(j);
                }
            } else if (dm[sel[j]] & bit) {
                dep(s.lastN);
                if (!dot) {
                    for (int i : s.RN) dep(i);
                    s.D.push_back(j);
                } else {
                    s.RD.push_back(j);
                }
            }
        }
        if (!has_dots) continue;
        if (dot) {
            for (int i : barriers)
                if (!passes_dot(ops[sel[i]], unitary[sel[i]], op)) dep(i);
            dots.push_back(j);
        } else if (!unitary[sel[j]] || (op.smask & all_states) != all_states) {
            for (int i : dots)
                if (!passes_dot(op, unitary[sel[j]], ops[sel[i]])) dep(i);
            barriers.push_back(j);
        }
    }
    return o;
}

// Ops of one register stage: within a stage they are compared pair by pair
// (stage_levels_order). A longer run goes on in a stage of the same register
// bits, which costs the kernels nothing. 8000 gates on four wires of a 12-qubit
// state, one pass, are planned in 18 ms; in 820 with one stage and the order of
// the pass's ops found pair by pair as well.
constexpr size_t kMaxStageOps = 512;

bool reg_capable(const LOp &o) {
    if (o.flags & TF_ZERO_UNCTRL) return false;
    switch (o.kind) {
    case TOP_DENSE1:
    case TOP_DENSE2:
    case TOP_PARITY:
    case TOP_PCPHASE: return true;
    case TOP_DIAG: return o.k <= 2;
    default: return false;
    }
}

// Split a pass's ops into register stages (each with at most rb register
// bits among its non-diagonal targets) and LDS stages, respecting the order
// constraints between ops. Register bits of a stage are padded with the
// previous stage's bits so that unchanged mappings need no transpose.
template <typename LocalF>
std::vector<StagePlan> plan_stages(const std::vector<LOp> &ops, OpOrder order, const std::vector<int> &sel,
                                   LocalF local, int rb, int kt) {
    const int m = static_cast<int>(sel.size());
    std::vector<std::vector<int>> &succ = order.succ;
    std::vector<int> &indeg = order.indeg;
    std::vector<uint32_t> nl(m);
    std::vector<char> rc(m);
    for (int i = 0; i < m; ++i) {
        nl[i] = local(ops[sel[i]].nmask());
        rc[i] = reg_capable(ops[sel[i]]) ? 1 : 0;
    }
    std::set<int> ready;
    for (int i = 0; i < m; ++i)
        if (indeg[i] == 0) ready.insert(i);
    int left = m;
    auto take = [&](int i) {
        ready.erase(i);
        --left;
        for (int s : succ[i])
            if (--indeg[s] == 0) ready.insert(s);
    };
    uint32_t prevR = ((1u << kt) - 1u) & ~0xFFu; // the load mapping's register bits
    std::vector<StagePlan> out;
    while (left > 0) {
        StagePlan sp;
        uint32_t U = 0;
        while (sp.ops.size() < kMaxStageOps) {
            int pick = -1;
            for (int i : ready)
                if (rc[i] && (nl[i] & ~U) == 0) {
                    pick = i;
                    break;
                }
            if (pick < 0)
                for (int i : ready)
                    if (rc[i] && popc(U | nl[i]) <= rb) {
                        pick = i;
                        break;
                    }
            if (pick < 0) break;
            U |= nl[pick];
            sp.ops.push_back(sel[pick]);
            take(pick);
        }
        if (!sp.ops.empty()) {
            sp.reg = true;
            uint32_t R = U;
            for (int b = 0; b < kt && popc(R) < rb; ++b)
                if ((prevR >> b) & 1u) R |= 1u << b;
            for (int b = kt - 1; b >= 0 && popc(R) < rb; --b) R |= 1u << b;
            sp.R = R;
            prevR = R;
        } else {
            while (true) {
                int pick = -1;
                for (int i : ready)
                    if (!rc[i]) {
                        pick = i;
                        break;
                    }
                if (pick < 0) break;
                sp.ops.push_back(sel[pick]);
                take(pick);
            }
            LQ_ABORT_IF(sp.ops.empty(), "stage planning made no progress");
        }
        out.push_back(std::move(sp));
    }
    return out;
}

// Targets as register-index bits, controls and diagonal bits as global masks;
// a diagonal +-1 table becomes a sign flip.
void to_register_form(TileOp &t, const LOp &o, const TileStage &st, const int *pos, int rb) {
    auto ridx = [&](int lb) -> int {
        for (int i = 0; i < rb; ++i)
            if (st.rbits[i] == lb) return i;
        LQ_ABORT("register bit not found");
    };
    t.gcmask = o.cmask;
    t.gcval = o.cval & o.cmask;
    if (o.kind == TOP_DENSE1) {
        t.lpos[0] = ridx(pos[o.bits[0]]);
    } else if (o.kind == TOP_DENSE2) {
        t.lpos[0] = ridx(pos[o.bits[0]]);
        t.lpos[1] = ridx(pos[o.bits[1]]);
    } else if (o.kind == TOP_PARITY) {
        t.gpmask = o.pmask;
    } else if (o.kind == TOP_DIAG && !o.is_dot()) {
        const cd one(1.0), mone(-1.0);
        if (o.k == 1 && o.coef[0] == one && o.coef[1] == mone) {
            t.kind = TOP_SIGN;
            t.gcmask |= 1ull << o.bits[0];
            t.gcval |= 1ull << o.bits[0];
        } else if (o.k == 1 && o.coef[0] == mone && o.coef[1] == one) {
            t.kind = TOP_SIGN;
            t.gcmask |= 1ull << o.bits[0];
        } else if (o.k == 0 && o.coef[0] == mone) {
            t.kind = TOP_SIGN;
        }
    }
}

bool diagonal_kind(uint32_t k) {
    return k == TOP_DIAG || k == TOP_SIGN || k == TOP_CZSET || k == TOP_PARITY || k == TOP_PCPHASE ||
           k == TOP_RPHASE || k == TOP_TPHASE;
}

// Whether a dot (register form, one or two targets) and an op may change
// places: the op is unitary, acts on both of the dot's states, and acts
// non-diagonally on no bit the dot touches (and the dot on none of the op's).
bool dot_commutes(const TileOp &dot, const TileOp &op) {
    const uint32_t ab = (1u << dot.sa) | (1u << dot.sb);
    if (!(op.flags & TF_UNITARY) || (op.smask & ab) != ab) return false;
    auto bits = [](const TileOp &t, uint64_t *nd, uint64_t *dg) {
        *nd = 0;
        *dg = t.gcmask;
        uint64_t m = 0;
        for (uint32_t j = 0; j < t.k && j < static_cast<uint32_t>(kMaxTileOpTargets); ++j) m |= 1ull << t.gpos[j];
        switch (t.kind) {
        case TOP_DENSE1:
        case TOP_DENSE2: *nd = m; return true;
        case TOP_DIAG:
        case TOP_PCPHASE: *dg |= m; return true;
        case TOP_PARITY: *dg |= t.gpmask; return true;
        case TOP_SIGN: return true;
        default: return false;
        }
    };
    uint64_t na, da, nb, db;
    if (!bits(dot, &na, &da) || !bits(op, &nb, &db)) return false;
    return !(na & (nb | db)) && !(nb & da);
}

// A one-bit phase on a register bit: it can stand anywhere between the ops
// that block it, from lo (before rest[lo]) to hi.
struct RegPhase {
    int lo, hi, r;
    uint32_t sm;
    cd d0, d1;
    int at; // it stood before rest[at]
    uint64_t src;
    bool unit;
};

bool blocks_phase(const TileOp &l, const RegPhase &ph) {
    if (l.flags & TF_DOT) {
        // <b|D^dagger G D|a> = <b|G|a> for a unitary phase D on both states and
        // a bit that G acts on diagonally or not at all
        const uint32_t ab = (1u << l.sa) | (1u << l.sb);
        if (!ph.unit || (ph.sm & ab) != ab) return true;
    } else if (!(l.smask & ph.sm)) {
        return false;
    }
    if (diagonal_kind(l.kind)) return false;
    if (l.kind == TOP_DENSE1) return l.lpos[0] == ph.r;
    if (l.kind == TOP_DENSE2) return l.lpos[0] == ph.r || l.lpos[1] == ph.r;
    return true;
}

// Order of a register stage's ops by earliest level: an op's level is one
// more than that of the latest earlier op it does not commute with. Ops
// commute when they act on different states, or when neither acts
// non-diagonally on a bit the other touches; dots commute with each other and
// with the ops of dot_commutes, unless a phase stands between two of them that
// neither may pass. Ops without a known bit set keep their place relative to
// everything.
std::vector<int> stage_levels_order(const std::vector<TileOp> &ops, const std::vector<RegPhase> &phases) {
    const int M = static_cast<int>(ops.size());
    const uint64_t ALL = ~0ull;
    std::vector<uint64_t> nd(static_cast<size_t>(M)), dg(static_cast<size_t>(M));
    for (int x = 0; x < M; ++x) {
        const TileOp &t = ops[x];
        uint64_t a = 0, d = t.gcmask;
        if (t.flags & TF_DOT) {
            a = ALL;
        } else if (t.kind == TOP_DENSE1) {
            a = 1ull << t.gpos[0];
        } else if (t.kind == TOP_DENSE2) {
            a = (1ull << t.gpos[0]) | (1ull << t.gpos[1]);
        } else if (t.kind == TOP_DIAG || t.kind == TOP_PCPHASE || t.kind == TOP_TPHASE) {
            for (uint32_t j = 0; j < t.k; ++j) d |= 1ull << t.gpos[j];
        } else if (t.kind == TOP_PARITY) {
            d |= t.gpmask;
        } else if (t.kind == TOP_SIGN) {
        } else {
            a = ALL;
        }
        nd[x] = a;
        dg[x] = d;
    }
    auto commute = [&](int x, int y) {
        const bool dx = ops[x].flags & TF_DOT, dy = ops[y].flags & TF_DOT;
        if (dx && dy) return true;
        if (dx) return dot_commutes(ops[x], ops[y]);
        if (dy) return dot_commutes(ops[y], ops[x]);
        if (nd[x] == ALL || nd[y] == ALL) return false;
        if (!(ops[x].smask & ops[y].smask)) return true;
        return !(nd[x] & (nd[y] | dg[y])) && !(nd[y] & (nd[x] | dg[x]));
    };
    std::vector<int> level(static_cast<size_t>(M), 0);
    // of each phase, the highest level among the ops before it that block it:
    // no op after it that blocks it may get a lower one (ops of one level keep
    // their order)
    std::vector<int> floor(phases.size(), 0);
    size_t passed = 0; // phases before op y (they are in the order of their places)
    for (int y = 0; y < M; ++y) {
        for (; passed < phases.size() && phases[passed].at <= y; ++passed)
            for (int x = 0; x < phases[passed].at; ++x)
                if (level[x] > floor[passed] && blocks_phase(ops[x], phases[passed])) floor[passed] = level[x];
        for (int x = 0; x < y; ++x)
            if (!commute(x, y)) level[y] = std::max(level[y], level[x] + 1);
        for (size_t j = 0; j < passed; ++j)
            if (floor[j] > level[y] && blocks_phase(ops[y], phases[j])) level[y] = floor[j];
    }
    std::vector<int> perm(static_cast<size_t>(M));
    for (int x = 0; x < M; ++x) perm[x] = x;
    std::stable_sort(perm.begin(), perm.end(), [&](int x, int y) { return level[x] < level[y]; });
    return perm;
}

// In a register stage the non-diagonal ops act on register bits only, so a
// one-bit phase on any other bit (a thread or outside bit: fixed per thread)
// commutes with every op of the stage but one of unknown action and, where it
// is not unitary or acts on one of the dot's states only, a dot.
// Between two such blockers, the phases of one state set become one
// TOP_TPHASE op at the first one's place: each thread forms the product of
// their factors once and multiplies its amplitudes once, instead of once per
// phase. Coefficients are copied (pairs d0, d1 per phase) with their sources.
void group_thread_phases(PassPlan &p, std::vector<TileOp> &ops, const int *ridx) {
    auto is_tphase = [&](const TileOp &t) {
        return t.kind == TOP_DIAG && t.k == 1 && t.gcmask == 0 && !(t.flags & TF_DOT) && t.gpos[0] >= 0 &&
               t.gpos[0] < 64 && ridx[t.gpos[0]] < 0;
    };
    auto blocker = [&](const TileOp &t) {
        return !(t.flags & TF_DOT) && !diagonal_kind(t.kind) && t.kind != TOP_DENSE1 && t.kind != TOP_DENSE2;
    };
    int count = 0;
    for (const TileOp &t : ops) count += is_tphase(t);
    if (count < 2) return;
    std::vector<TileOp> out;
    struct Group {
        uint32_t sm;
        size_t at;      // index into out
        bool past_dot;  // a dot stands after it
    };
    std::vector<Group> open;
    for (const TileOp &t : ops) {
        if (blocker(t)) open.clear();
        if (t.flags & TF_DOT) {
            // phases on thread bits commute with a dot whose states they both
            // act on (its non-diagonal bits are register bits): the group
            // stays open for unitary ones
            const uint32_t ab = (1u << t.sa) | (1u << t.sb);
            open.erase(std::remove_if(open.begin(), open.end(), [&](const Group &g) { return (g.sm & ab) != ab; }),
                       open.end());
            for (Group &g : open) g.past_dot = true;
        }
        if (!is_tphase(t)) {
            out.push_back(t);
            continue;
        }
        size_t at = out.size();
        bool found = false;
        for (const Group &g : open)
            if (g.sm == t.smask && out[g.at].k < static_cast<uint32_t>(kMaxTileOpTargets) &&
                (!g.past_dot || (t.flags & TF_UNITARY))) {
                at = g.at;
                found = true;
            }
        if (!found) {
            TileOp n{};
            n.kind = TOP_TPHASE;
            n.smask = t.smask;
            n.k = 0;
            for (int j = 0; j < kMaxTileOpTargets; ++j) n.lpos[j] = n.gpos[j] = -1;
            n.coef_off = p.coef.size();
            // room for a full op: coefficients of one op are contiguous
            p.coef.insert(p.coef.end(), 2 * kMaxTileOpTargets, cd(1.0));
            p.coef_src.insert(p.coef_src.end(), 2 * kMaxTileOpTargets, PassPlan::CoefSrc{PassPlan::kNoSrc, 0});
            out.push_back(n);
            open.push_back({t.smask, at, false});
        }
        TileOp &g = out[at];
        const uint64_t dst = g.coef_off + 2 * static_cast<uint64_t>(g.k);
        for (int c = 0; c < 2; ++c) {
            p.coef[dst + c] = p.coef[t.coef_off + c];
            p.coef_src[dst + c] = p.coef_src[t.coef_off + c];
        }
        g.gpos[g.k] = t.gpos[0];
        ++g.k;
    }
    ops.swap(out);
}

// In each register stage, one-bit phases on register bits commute with
// diagonal ops and with dense ops on other register bits, so each can sit
// anywhere between the ops that block it (blocks_phase: a dense op or dot on
// its bit, any dot for a phase that is not unitary, any other non-diagonal op). Choose the fewest points that every phase's range
// contains (interval stabbing, greedy by right end) and replace the phases at
// each point by one table over the stage's register index.
void group_register_phases(PassPlan &p, int rb) {
    std::vector<TileOp> out;
    const int E = 1 << rb;
    for (auto &st : p.stages) {
        const uint32_t begin = static_cast<uint32_t>(out.size());
        std::vector<TileOp> ops(p.ops.begin() + st.op_begin, p.ops.begin() + st.op_end);
        if (st.kind == STAGE_REG) {
            int ridx[64];
            for (int b = 0; b < 64; ++b) ridx[b] = -1;
            for (int i = 0; i < rb; ++i) ridx[p.tbits[st.rbits[i]]] = i;
            group_thread_phases(p, ops, ridx);
            auto is_phase = [&](const TileOp &t) {
                return t.kind == TOP_DIAG && t.k == 1 && t.gcmask == 0 && !(t.flags & TF_DOT) && t.gpos[0] >= 0 &&
                       t.gpos[0] < 64 && ridx[t.gpos[0]] >= 0;
            };
            std::vector<TileOp> rest;      // non-phase ops; gap g sits before rest[g]
            std::vector<RegPhase> ph;
            for (const TileOp &t : ops) {
                if (is_phase(t)) {
                    ph.push_back({0, 0, ridx[t.gpos[0]], t.smask, p.coef[t.coef_off], p.coef[t.coef_off + 1],
                                  static_cast<int>(rest.size()), t.coef_off, (t.flags & TF_UNITARY) != 0});
                } else {
                    rest.push_back(t);
                }
            }
            const int M = static_cast<int>(rest.size());
            // Reorder the other ops by their earliest level (ops that commute
            // may pass each other), so that ops on different bits at the same
            // depth sit together and the phases between them share one point.
            std::vector<int> perm = stage_levels_order(rest, ph);
            std::vector<int> newpos(static_cast<size_t>(M));
            for (int x = 0; x < M; ++x) newpos[perm[x]] = x;
            // a phase's range is bounded by every op that blocks it: commuting
            // ones (two dots) may have changed places, so the nearest in program
            // order need not be the nearest now
            for (RegPhase &q : ph) {
                q.lo = 0;
                q.hi = M;
                for (int x = 0; x < M; ++x) {
                    if (!blocks_phase(rest[x], q)) continue;
                    if (x < q.at) q.lo = std::max(q.lo, newpos[x] + 1);
                    else q.hi = std::min(q.hi, newpos[x]);
                }
                LQ_ABORT_IF(q.lo > q.hi, "a phase between ops that changed places");
            }
            {
                std::vector<TileOp> re(static_cast<size_t>(M));
                for (int x = 0; x < M; ++x) re[x] = rest[perm[x]];
                rest.swap(re);
            }
            std::vector<int> order(ph.size());
            for (size_t i = 0; i < ph.size(); ++i) order[i] = static_cast<int>(i);
            std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return ph[x].hi < ph[y].hi; });
            std::vector<int> point(ph.size(), -1);
            for (int i : order) {
                if (point[i] >= 0) continue;
                const int g = ph[i].hi;
                for (size_t j = 0; j < ph.size(); ++j)
                    if (point[j] < 0 && ph[j].sm == ph[i].sm && ph[j].lo <= g && g <= ph[j].hi) point[j] = g;
            }
            std::vector<TileOp> merged;
            for (int g = 0; g <= M; ++g) {
                std::vector<uint32_t> sms;
                for (size_t j = 0; j < ph.size(); ++j)
                    if (point[j] == g && std::find(sms.begin(), sms.end(), ph[j].sm) == sms.end()) sms.push_back(ph[j].sm);
                for (uint32_t sm : sms) {
                    std::vector<cd> table(static_cast<size_t>(E), cd(1.0));
                    TileOp t{};
                    PassPlan::PhaseTable rec;
                    rec.off = p.coef.size();
                    rec.rb = rb;
                    for (size_t j = 0; j < ph.size(); ++j) {
                        if (point[j] != g || ph[j].sm != sm) continue;
                        for (int e = 0; e < E; ++e) table[e] *= ((e >> ph[j].r) & 1) ? ph[j].d1 : ph[j].d0;
                        rec.phases.emplace_back(ph[j].src, ph[j].r);
                    }
                    t.kind = TOP_RPHASE;
                    t.k = static_cast<uint32_t>(rb);
                    t.smask = sm;
                    for (int j = 0; j < kMaxTileOpTargets; ++j) t.lpos[j] = t.gpos[j] = -1;
                    t.coef_off = p.coef.size();
                    p.coef.insert(p.coef.end(), table.begin(), table.end());
                    p.coef_src.insert(p.coef_src.end(), table.size(), PassPlan::CoefSrc{PassPlan::kNoSrc, 0});
                    p.tables.push_back(std::move(rec));
                    merged.push_back(t);
                }
                if (g < M) merged.push_back(rest[g]);
            }
            ops.swap(merged);
        }
        out.insert(out.end(), ops.begin(), ops.end());
        st.op_begin = begin;
        st.op_end = static_cast<uint32_t>(out.size());
    }
    p.ops.swap(out);
}

// Merge runs of CZ sign flips into popcount-parity ops and set how each
// stage's register mapping is reached.
void finish_reg_pass(PassPlan &p, int kt) {
    group_register_phases(p, kt - 8);
    std::vector<TileOp> merged;
    for (auto &st : p.stages) {
        const uint32_t begin = static_cast<uint32_t>(merged.size());
        TileOp cur{};
        bool open = false;
        auto flush = [&]() {
            if (open) merged.push_back(cur);
            open = false;
        };
        for (uint32_t i = st.op_begin; i < st.op_end; ++i) {
            const TileOp &t = p.ops[i];
            const bool cz = st.kind == STAGE_REG && t.kind == TOP_SIGN && !(t.flags & TF_DOT) &&
                            popc(t.gcmask) == 2 && t.gcval == t.gcmask;
            if (!cz) {
                flush();
                merged.push_back(t);
                continue;
            }
            const int lo = __builtin_ctzll(t.gcmask), hi = 63 - __builtin_clzll(t.gcmask);
            const uint32_t d = static_cast<uint32_t>(hi - lo);
            int slot = -1;
            if (open && cur.smask == t.smask) {
                for (uint32_t z = 0; z < cur.nz; ++z)
                    if (cur.sd[z] == d) slot = static_cast<int>(z);
                if (slot < 0 && cur.nz < 4) slot = static_cast<int>(cur.nz++);
            }
            if (slot < 0) {
                flush();
                cur = t;
                cur.kind = TOP_CZSET;
                cur.gcmask = cur.gcval = 0;
                cur.nz = 1;
                cur.sd[0] = d;
                cur.sm[0] = 0;
                for (int z = 1; z < 4; ++z) {
                    cur.sd[z] = 0;
                    cur.sm[z] = 0;
                }
                open = true;
                slot = 0;
            }
            cur.sd[slot] = d;
            cur.sm[slot] ^= 1ull << lo; // a pair that comes twice cancels
        }
        flush();
        st.op_begin = begin;
        st.op_end = static_cast<uint32_t>(merged.size());
    }
    p.ops.swap(merged);

    const uint32_t m0 = ((1u << kt) - 1u) & ~0xFFu;
    uint32_t prevR = m0;
    bool prev_lds = false;
    for (auto &st : p.stages) {
        if (st.kind != STAGE_REG) {
            prev_lds = true;
            continue;
        }
        uint32_t R = 0;
        for (int i = 0; i < kt - 8; ++i) R |= 1u << st.rbits[i];
        st.entry = prev_lds ? ENTRY_FROM_LDS : (R == prevR ? ENTRY_NONE : ENTRY_TRANSPOSE);
        prevR = R;
        prev_lds = false;
    }
    p.end_transpose = (!prev_lds && prevR != m0) ? 1u : 0u;
}
} // namespace

TileGeom make_geom(int n, const std::vector<int> &tbits) {
    TileGeom g{};
    g.n = n;
    g.kt = static_cast<int>(tbits.size());
    g.nout = n - g.kt;
    LQ_ABORT_IF(g.kt > 16 || g.nout > kMaxOutsideBits, "tile geometry out of range");
    uint64_t tm = 0;
    for (int j = 0; j < g.kt; ++j) {
        g.tb[j] = tbits[j];
        tm |= 1ull << tbits[j];
    }
    g.c = 0;
    while (g.c < g.kt && g.tb[g.c] == g.c) ++g.c;
    int o = 0;
    for (int b = 0; b < n; ++b)
        if (!((tm >> b) & 1ull)) g.ob[o++] = b;
    return g;
}

namespace {
constexpr double kMinCos = 1e-100;

// Convert the recorded (or, at plan time, the eligible) real rotations of a
// pass to [[1, -t], [t, 1]] and multiply the product of their cosines into
// the pass's scale table. Returns false if the recorded choice no longer
// holds for the current angles (a cosine too small for the stored form, or
// the growth bound now crossed in either direction).
bool apply_rotation_scaling(PassPlan &p, bool at_plan_time, int rb, double max_growth) {
    if (at_plan_time) {
        p.scaled.clear();
        p.scale_dropped.clear();
        p.scale_table = -1;
        if (!p.reg || p.load_mask != 1u || p.store_mask != 1u || !p.slot_ids.empty() || p.stages.empty() ||
            p.stages.back().kind != STAGE_REG)
            return true;
        for (const TileStage &st : p.stages) {
            if (st.kind != STAGE_REG) continue;
            for (uint32_t i = st.op_begin; i < st.op_end; ++i) {
                TileOp &t = p.ops[i];
                if (t.kind != TOP_DENSE1 || !(t.flags & TF_REAL) || (t.flags & TF_DOT) || t.smask != 1u ||
                    t.gcmask != 0 || t.lcmask != 0 || t.ocmask != 0)
                    continue;
                if (std::fabs(p.coef[t.coef_off].real()) < kMinCos) continue;
                t.flags |= TF_SCALED;
                p.scaled.push_back(t.coef_off);
            }
        }
        if (p.scaled.empty()) return true;
        p.scale_growth_limit = max_growth;
        double growth = 1.0;
        for (uint64_t off : p.scaled) growth /= std::fabs(p.coef[off].real());
        if (!(growth <= max_growth)) {
            // too much growth for these angles: the full form throughout; a
            // refresh whose angles would allow the scaled form asks for a new plan
            for (const TileStage &st : p.stages)
                for (uint32_t i = st.op_begin; i < st.op_end; ++i) p.ops[i].flags &= ~static_cast<uint32_t>(TF_SCALED);
            p.scale_dropped.swap(p.scaled);
            return true;
        }
        // the carrier: the last one-state phase table, or a new one at the end
        for (const TileStage &st : p.stages) {
            if (st.kind != STAGE_REG) continue;
            for (uint32_t i = st.op_begin; i < st.op_end; ++i)
                if (p.ops[i].kind == TOP_RPHASE && p.ops[i].smask == 1u) p.scale_table = static_cast<int64_t>(p.ops[i].coef_off);
        }
        if (p.scale_table < 0) {
            TileOp t{};
            t.kind = TOP_RPHASE;
            t.k = static_cast<uint32_t>(rb);
            t.smask = 1u;
            for (int j = 0; j < kMaxTileOpTargets; ++j) t.lpos[j] = t.gpos[j] = -1;
            t.coef_off = p.coef.size();
            const size_t E = static_cast<size_t>(1) << rb;
            p.coef.insert(p.coef.end(), E, cd(1.0));
            p.coef_src.insert(p.coef_src.end(), E, PassPlan::CoefSrc{PassPlan::kNoSrc, 0});
            PassPlan::PhaseTable rec;
            rec.off = t.coef_off;
            rec.rb = rb;
            p.tables.push_back(rec);
            p.scale_table = static_cast<int64_t>(t.coef_off);
            LQ_ABORT_IF(p.stages.back().op_end != p.ops.size(), "last stage does not end the pass");
            p.ops.push_back(t);
            p.stages.back().op_end = static_cast<uint32_t>(p.ops.size());
        }
    }
    auto growth_of = [&](const std::vector<uint64_t> &offs) {
        double g = 1.0;
        for (uint64_t off : offs) g /= std::fabs(p.coef[off].real());
        return g;
    };
    if (!p.scale_dropped.empty() && growth_of(p.scale_dropped) <= p.scale_growth_limit) return false;
    if (p.scaled.empty()) return true;
    if (!(growth_of(p.scaled) <= p.scale_growth_limit)) return false;
    double prod = 1.0;
    for (uint64_t off : p.scaled) {
        const double c = p.coef[off].real(), s = p.coef[off + 2].real();
        if (std::fabs(c) < kMinCos) return false;
        const double t = s / c;
        p.coef[off] = cd(1.0);
        p.coef[off + 1] = cd(-t);
        p.coef[off + 2] = cd(t);
        p.coef[off + 3] = cd(1.0);
        prod *= c;
    }
    // the table's size from its record
    int trb = 0;
    for (const auto &tb : p.tables)
        if (static_cast<int64_t>(tb.off) == p.scale_table) trb = tb.rb;
    LQ_ABORT_IF(trb <= 0, "scale table not found");
    for (int e = 0; e < (1 << trb); ++e) p.coef[static_cast<size_t>(p.scale_table) + static_cast<size_t>(e)] *= prod;
    return true;
}
} // namespace

namespace {
constexpr double kSwapCost = 0.25; // of a 2x2 dense op's 1.0

// Tile bits of an operator that runs in a pass of its own, 0 when it does not:
// its targets and the lowest other bits. Controls stay outside the tile (a
// tile they rule out is not visited) except on the four low bits, which every
// tile holds so that HBM is read in runs of 16 amplitudes.
uint64_t dense_pass_bits(const LOp &o, int n) {
    if (o.kind != TOP_DENSEK || o.is_dot() || (o.flags & TF_ZERO_UNCTRL) || o.k < 3 || o.k > 6) return 0;
    uint64_t T = o.target_mask();
    for (int b = 0; b < n && popc(T) < kDenseTileBits; ++b)
        if (b < 4 || !((o.cmask >> b) & 1ull)) T |= 1ull << b;
    return popc(T) == kDenseTileBits ? T : 0;
}

PassPlan dense_pass(const LOp &o, int index, int n) {
    PassPlan p;
    p.dense = true;
    const uint64_t T = dense_pass_bits(o, n);
    for (int b = 0; b < n; ++b)
        if ((T >> b) & 1ull) p.tbits.push_back(b);
    TileOp t{};
    t.kind = o.kind;
    t.flags = o.flags;
    t.k = static_cast<uint32_t>(o.k);
    t.smask = o.smask;
    t.gcmask = o.cmask;
    t.gcval = o.cval & o.cmask;
    for (int j = 0; j < o.k; ++j) t.gpos[j] = o.bits[j];
    p.ops.push_back(t);
    p.coef = o.coef;
    for (size_t c = 0; c < o.coef.size(); ++c)
        p.coef_src.push_back({static_cast<uint32_t>(index), static_cast<uint32_t>(c)});
    p.load_mask = p.store_mask = o.smask;
    return p;
}
} // namespace

DenseTileArgs dense_tile_args(const PassPlan &p, int n) {
    LQ_ABORT_IF(!p.dense || p.ops.size() != 1 || p.tbits.size() != kDenseTileBits, "not a dense pass");
    const TileOp &o = p.ops[0];
    const int k = static_cast<int>(o.k), cl = kDenseTileBits - k;
    DenseTileArgs a{};
    uint64_t T = 0;
    int col = 0;
    for (int b = 0; b < kDenseTileBits; ++b) {
        const int g = p.tbits[b];
        T |= 1ull << g;
        a.tb[b] = g;
        a.lp[b] = -1;
        for (int j = 0; j < k; ++j)
            if (o.gpos[j] == g) a.lp[b] = cl + k - 1 - j;
        if (a.lp[b] >= 0) continue;
        a.lp[b] = col;
        if ((o.gcmask >> g) & 1ull) {
            a.ccmask |= 1u << col;
            if ((o.gcval >> g) & 1ull) a.ccval |= 1u << col;
        }
        ++col;
    }
    LQ_ABORT_IF(col != cl, "dense pass targets outside its tile");
    a.ocval = o.gcval & ~T;
    for (int b = 0; b < n; ++b)
        if (!((T >> b) & 1ull) && !((o.gcmask >> b) & 1ull)) a.ob[a.nout++] = b;
    a.ntiles = 1ull << a.nout;
    return a;
}

std::vector<PassPlan> plan_passes(const std::vector<LOp> &ops, const PlanConfig &cfg) {
    const int N = static_cast<int>(ops.size());
    const int n = cfg.n;
    std::vector<uint64_t> nm(N), dm(N);
    std::vector<double> cost_of(N);
    const bool has_dots = std::any_of(ops.begin(), ops.end(), [](const LOp &o) { return o.is_dot(); });
    std::vector<char> unitary(N, 0);
    std::vector<int> all(N);
    for (int j = 0; j < N; ++j) {
        all[j] = j;
        nm[j] = ops[j].nmask();
        dm[j] = ops[j].dmask() & ~nm[j];
        // specialised passes swap the amplitudes of an X or SWAP: a select per
        // word where a control is a thread bit, nothing otherwise
        cost_of[j] = ops[j].cost();
        if (cfg.lookahead && !cfg.keep_grouping && !ops[j].is_dot() && ops[j].is_swap()) cost_of[j] *= kSwapCost / (ops[j].k == 1 ? 1.0 : 2.5);
        LQ_ABORT_IF(((nm[j] | dm[j]) >> n) != 0, "operation acts on a wire outside the state");
        if (has_dots && !ops[j].is_dot()) unitary[j] = ops[j].is_unitary(cfg.unitary_tol(), cfg.max_unitary_test());
    }
    OpOrder whole = order_ops(ops, all, nm, dm, unitary, n, cfg.ns);
    std::vector<std::vector<int>> &succ = whole.succ;
    std::vector<int> &indeg = whole.indeg;

    std::set<int> ready;
    for (int j = 0; j < N; ++j)
        if (indeg[j] == 0) ready.insert(j);
    // operators that run in passes of their own; everything else that is
    // ready goes first, so they split as few tile passes as possible
    std::vector<char> alone(N, 0);
    for (int j = 0; j < N; ++j) alone[j] = cfg.dense_passes && dense_pass_bits(ops[j], n) != 0;

    const int ktmax = std::min(cfg.kt_max, n);
    const int low = std::max(0, std::min(cfg.low_bits, ktmax));
    const uint64_t low_mask = (low >= 64) ? ~0ull : ((1ull << low) - 1);

    // Lookahead choice of a pass's tile bits. run_with(T) replays, without
    // committing, the schedule the pass would make with tile bits T (ready ops
    // in program order, within the cost budget and dot slots) and returns the
    // cost it fits; ops held back only by bits outside T are collected as the
    // frontier. Starting from the low bits, the missing bits of the frontier
    // op whose addition lets the most work run per added bit are added until
    // the tile is full or the budget is met. On a chain of two-qubit gates
    // this grows contiguous blocks of wires, which advance several layers per
    // pass, where adding the first ready op's bits picks every other wire and
    // advances two.
    std::vector<int> touched;
    double budget = cfg.budget; // this pass's
    auto run_with = [&](uint64_t T, std::vector<int> *frontier, bool *full) {
        std::priority_queue<int, std::vector<int>, std::greater<int>> q(ready.begin(), ready.end());
        double cost = 0.0;
        int dots = 0, done = 0;
        *full = false;
        while (!q.empty()) {
            const int i = q.top();
            q.pop();
            if (alone[i]) continue;
            if ((nm[i] & ~T) != 0 || (dots >= cfg.max_dots && ops[i].is_dot())) {
                if (frontier) frontier->push_back(i);
                continue;
            }
            if (done > 0 && cost + cost_of[i] > budget) {
                *full = true;
                break;
            }
            cost += cost_of[i];
            dots += ops[i].is_dot() ? 1 : 0;
            ++done;
            for (int s2 : succ[i]) {
                touched.push_back(s2);
                if (--indeg[s2] == 0) q.push(s2);
            }
        }
        for (int s2 : touched) ++indeg[s2];
        touched.clear();
        return cost;
    };
    auto choose_bits = [&]() {
        uint64_t T = low_mask;
        std::vector<int> frontier;
        while (popc(T) < ktmax) {
            frontier.clear();
            bool full = false;
            const double base = run_with(T, &frontier, &full);
            if (full) break;
            uint64_t best = 0;
            double best_score = 0.0;
            int best_bits = 0;
            std::vector<uint64_t> seen;
            for (int i : frontier) {
                const uint64_t m = nm[i] & ~T;
                if (m == 0 || popc(T | m) > ktmax || std::find(seen.begin(), seen.end(), m) != seen.end()) continue;
                seen.push_back(m);
                bool f2 = false;
                const double score = (run_with(T | m, nullptr, &f2) - base) / popc(m);
                if (score > best_score + 1e-12 || (best != 0 && std::fabs(score - best_score) <= 1e-12 && popc(m) < best_bits)) {
                    best = m;
                    best_score = score;
                    best_bits = popc(m);
                }
            }
            if (best == 0) break;
            T |= best;
        }
        return T;
    };

    std::vector<PassPlan> passes;
    int remaining = N;
    while (remaining > 0) {
        if (std::all_of(ready.begin(), ready.end(), [&](int i) { return alone[i]; })) {
            const int i = *ready.begin();
            ready.erase(ready.begin());
            --remaining;
            for (int s : succ[i])
                if (--indeg[s] == 0) ready.insert(s);
            passes.push_back(dense_pass(ops[i], i, n));
            continue;
        }
        std::vector<int> sel;
        uint64_t T = 0;
        budget = (passes.empty() && cfg.first_budget > 0) ? cfg.first_budget : cfg.budget;
        const uint64_t T0 = cfg.lookahead ? choose_bits() : low_mask;
        for (int attempt = 0; attempt < 2 && sel.empty(); ++attempt) {
            T = attempt == 0 ? T0 : 0ull;
            double cost = 0.0;
            int dots = 0;
            while (true) {
                int pick = -1;
                const bool dots_full = dots >= cfg.max_dots;
                for (int i : ready)
                    if (!alone[i] && (nm[i] & ~T) == 0 && !(dots_full && ops[i].is_dot())) {
                        pick = i;
                        break;
                    }
                if (pick < 0)
                    for (int i : ready)
                        if (!alone[i] && popc(T | nm[i]) <= ktmax && !(dots_full && ops[i].is_dot())) {
                            pick = i;
                            break;
                        }
                if (pick < 0) break;
                if (!sel.empty() && cost + cost_of[pick] > budget) break;
                T |= nm[pick];
                cost += cost_of[pick];
                dots += ops[pick].is_dot() ? 1 : 0;
                sel.push_back(pick);
                ready.erase(pick);
                --remaining;
                for (int s : succ[pick])
                    if (--indeg[s] == 0) ready.insert(s);
            }
        }
        LQ_ABORT_IF(sel.empty(), "operation needs more tile bits than fit in LDS");
        // pad the tile with the lowest free bits
        for (int b = 0; b < n && popc(T) < ktmax; ++b) T |= 1ull << b;

        PassPlan p;
        int pos[64];
        for (int b = 0; b < 64; ++b) pos[b] = -1;
        for (int b = 0; b < n; ++b)
            if ((T >> b) & 1ull) {
                pos[b] = static_cast<int>(p.tbits.size());
                p.tbits.push_back(b);
            }
        auto local = [&](uint64_t m) {
            uint32_t r = 0;
            for (int b = 0; b < n; ++b)
                if (((m >> b) & 1ull) && pos[b] >= 0) r |= 1u << pos[b];
            return r;
        };
        const int kt = static_cast<int>(p.tbits.size());
        p.reg = cfg.reg_rb > 0 && kt == 8 + cfg.reg_rb && cfg.ns <= kMaxStates;
        std::vector<int> order = sel;
        std::vector<StagePlan> stages;
        if (p.reg) {
            stages = plan_stages(ops, order_ops(ops, sel, nm, dm, unitary, n, cfg.ns), sel, local, cfg.reg_rb, kt);
            order.clear();
            for (const auto &st : stages) order.insert(order.end(), st.ops.begin(), st.ops.end());
        }
        std::vector<int> op_stage;
        for (size_t si = 0; si < stages.size(); ++si)
            for (size_t k2 = 0; k2 < stages[si].ops.size(); ++k2) op_stage.push_back(static_cast<int>(si));
        size_t stage_cursor = 0;
        for (size_t oi = 0; oi < order.size(); ++oi) {
            const int idx = order[oi];
            const LOp &o = ops[idx];
            if (p.reg) {
                const int si = op_stage[oi];
                if (p.stages.size() <= static_cast<size_t>(si)) {
                    // open the stage
                    TileStage ts{};
                    ts.kind = stages[si].reg ? STAGE_REG : STAGE_LDS;
                    ts.op_begin = ts.op_end = static_cast<uint32_t>(p.ops.size());
                    int r = 0, h = 0;
                    for (int b = 0; b < kt; ++b) {
                        if ((stages[si].R >> b) & 1u) {
                            if (r < kMaxRegBits) ts.rbits[r++] = b;
                        } else if (h < 8) {
                            ts.hbits[h++] = b;
                        }
                    }
                    p.stages.push_back(ts);
                    stage_cursor = static_cast<size_t>(si);
                }
            }
            TileOp t{};
            t.kind = o.kind;
            t.flags = o.flags;
            if (!o.is_dot() && o.is_swap()) t.flags |= TF_SWAP;
            if (has_dots) t.flags |= o.is_dot() ? o.dot_class() : !cfg.keep_grouping && unitary[idx] ? TF_UNITARY : 0u;
            t.k = static_cast<uint32_t>(o.k);
            t.smask = o.smask;
            t.sa = o.sa;
            t.sb = o.sb;
            t.lcmask = local(o.cmask);
            t.lcval = local(o.cval & o.cmask);
            t.ocmask = o.cmask & ~T;
            t.ocval = o.cval & o.cmask & ~T;
            for (int j = 0; j < kMaxTileOpTargets; ++j) {
                t.lpos[j] = j < o.k ? pos[o.bits[j]] : -1;
                t.gpos[j] = j < o.k ? o.bits[j] : 0;
            }
            if (o.kind == TOP_PARITY) {
                t.lxmask = local(o.pmask);
                t.omask = o.pmask & ~T;
            } else if (o.kind == TOP_PAULI) {
                t.lxmask = local(o.xmask);
                t.lzmask = local(o.yzmask);
                t.omask = o.yzmask & ~T;
                t.ny = static_cast<uint32_t>(o.ny);
            }
            t.pc_dim = o.pc_dim;
            t.coef_off = p.coef.size();
            p.coef.insert(p.coef.end(), o.coef.begin(), o.coef.end());
            for (size_t c = 0; c < o.coef.size(); ++c)
                p.coef_src.push_back({static_cast<uint32_t>(idx), static_cast<uint32_t>(c)});
            if (o.is_dot()) {
                t.slot = static_cast<uint32_t>(p.slot_ids.size());
                p.slot_ids.push_back(o.slot);
                p.load_mask |= (1u << o.sa) | (1u << o.sb);
            } else {
                p.load_mask |= o.smask;
                p.store_mask |= o.smask;
            }
            if (p.reg && p.stages[stage_cursor].kind == STAGE_REG)
                to_register_form(t, o, p.stages[stage_cursor], pos, cfg.reg_rb);
            p.ops.push_back(t);
            if (p.reg) p.stages[stage_cursor].op_end = static_cast<uint32_t>(p.ops.size());
        }
        if (p.reg) finish_reg_pass(p, kt);
        if (p.reg && cfg.scale_rotations) apply_rotation_scaling(p, true, kt - 8, cfg.max_scale_growth);
        passes.push_back(std::move(p));
    }
    return passes;
}

std::string plan_structure_key(const std::vector<LOp> &ops, const PlanConfig &cfg) {
    std::string key;
    key.reserve(ops.size() * 32 + 128);
    auto put = [&key](const void *p, size_t n) { key.append(static_cast<const char *>(p), n); };
    const double b = cfg.budget;
    const int32_t hdr[10] = {cfg.n, cfg.ns, cfg.kt_max, cfg.low_bits, cfg.reg_rb, cfg.max_dots,
                             cfg.scale_rotations ? 1 : 0, cfg.lookahead ? 1 : 0, cfg.dense_passes ? 1 : 0,
                             cfg.keep_grouping ? 1 : 0};
    put(hdr, sizeof(hdr));
    put(&b, sizeof(b));
    put(&cfg.first_budget, sizeof(cfg.first_budget));
    put(&cfg.max_scale_growth, sizeof(cfg.max_scale_growth));
    const cd one(1.0), mone(-1.0);
    const bool has_dots = std::any_of(ops.begin(), ops.end(), [](const LOp &o) { return o.is_dot(); });
    for (const LOp &o : ops) {
        // value tests made while planning (to_register_form)
        uint32_t vflags = 0;
        if (!o.is_dot() && o.is_swap()) vflags = 5;
        else if (o.kind == TOP_DENSE1 && (o.flags & TF_REAL) && o.coef.size() == 4 && std::fabs(o.coef[0].real()) < kMinCos)
            vflags = 4;
        if (o.kind == TOP_DIAG && !o.is_dot()) {
            if (o.k == 1 && o.coef.size() == 2 && o.coef[0] == one && o.coef[1] == mone) vflags = 1;
            else if (o.k == 1 && o.coef.size() == 2 && o.coef[0] == mone && o.coef[1] == one) vflags = 2;
            else if (o.k == 0 && o.coef.size() == 1 && o.coef[0] == mone) vflags = 3;
        }
        if (has_dots) vflags |= o.is_dot() ? o.dot_class() : o.is_unitary(cfg.unitary_tol(), cfg.max_unitary_test()) ? TF_UNITARY : 0u;
        // fields that are zero for most ops are written only where they are
        // not, behind a byte that says which
        const uint64_t m[8] = {o.cmask, o.cval, o.xmask, o.yzmask, o.pmask, o.pc_dim, static_cast<uint64_t>(o.ny),
                               (static_cast<uint64_t>(o.sa) << 32) | o.sb};
        uint32_t present = 0;
        for (int j = 0; j < 8; ++j) present |= (m[j] != 0 ? 1u : 0u) << j;
        const uint32_t w[5] = {o.kind | (static_cast<uint32_t>(o.k) << 8) | (o.smask << 16) | (present << 24), o.flags,
                               vflags, static_cast<uint32_t>(o.slot), static_cast<uint32_t>(o.coef.size())};
        put(w, sizeof(w));
        int8_t b8[kMaxTileOpTargets];
        const int nb = std::max(0, std::min(o.k, kMaxTileOpTargets));
        for (int j = 0; j < nb; ++j) b8[j] = static_cast<int8_t>(o.bits[j]);
        put(b8, static_cast<size_t>(nb));
        for (int j = 0; j < 8; ++j)
            if (m[j]) put(&m[j], sizeof(uint64_t));
    }
    return key;
}

bool refresh_plan_coefs(std::vector<PassPlan> &passes, const std::vector<LOp> &ops) {
    for (PassPlan &p : passes) {
        LQ_ABORT_IF(p.coef_src.size() != p.coef.size(), "plan without coefficient sources");
        for (size_t i = 0; i < p.coef.size(); ++i) {
            const PassPlan::CoefSrc &s = p.coef_src[i];
            if (s.op == PassPlan::kNoSrc) continue;
            p.coef[i] = ops[s.op].coef[s.idx];
        }
        for (const PassPlan::PhaseTable &t : p.tables) {
            const int E = 1 << t.rb;
            for (int e = 0; e < E; ++e) {
                cd v(1.0);
                for (const auto &ph : t.phases) v *= p.coef[ph.first + (((e >> ph.second) & 1) ? 1 : 0)];
                p.coef[t.off + static_cast<uint64_t>(e)] = v;
            }
        }
        if (!apply_rotation_scaling(p, false, 0, p.scale_growth_limit)) return false;
    }
    return true;
}

} // namespace lqamd
