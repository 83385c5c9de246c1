// Circuit passes, host side (see pass.hpp).
#include "pass.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <iterator>
#include <stdexcept>

namespace qcore
{
    namespace
    {
        uint64_t bit(int q) { return uint64_t(1) << q; }

        const cd kOne(1.0);

        cl times(cl a, cl b) { return {a.real() * b.real() - a.imag() * b.imag(), a.real() * b.imag() + a.imag() * b.real()}; }
        // a / b for phases b of modulus 1
        cl over(cl a, cl b) { return times(a, std::conj(b)); }
        cl unit(cl z)
        {
            const long double r = std::sqrt(std::norm(z));
            return r == 0 ? cl(1.0) : cl(z.real() / r, z.imag() / r);
        }

        // The shears of [[c, -s], [s, c]]: -t and 2t / (1 + t^2) with t = s / (1 + c) rounded
        // first, so that the three shears stay orthogonal to the rounding of the second.
        void shears(long double c, long double s, double *m)
        {
            const double t = double(s / (1 + c));
            const long double x = t;
            m[0] = -t;
            m[1] = double(2 * x / (1 + x * x));
        }

        // M = e [[1, 0], [0, p]] [[c, -s], [s, c]] [[1, 0], [0, l]] with c, s >= 0; m: the
        // rotation's shears.  The phases come from the larger entries (those of a small one
        // hold only rounding).
        struct Euler
        {
            cl e, p, l;
            double m[2];
        };
        Euler euler(const cl *M)
        {
            const long double cc = std::norm(M[0]), ss = std::norm(M[2]), r = std::sqrt(cc + ss);
            const long double c = std::sqrt(cc), s = std::sqrt(ss);
            Euler u;
            u.e = cc == 0 ? cl(1.0) : cl(M[0].real() / c, M[0].imag() / c);
            const cl ep = ss == 0 ? cl(1.0) : cl(M[2].real() / s, M[2].imag() / s);
            u.p = over(ep, u.e);
            u.l = c >= s ? over(unit(M[3]), ep) : over(unit(-M[1]), u.e);
            shears(c / r, s / r, u.m);
            return u;
        }
    } // namespace

    // ---- lowering ----
    // M_q <- [[a, b], [c, d]] M_q
    void PassLowering::mul(int q, cl a, cl b, cl c, cl d)
    {
        One &o = one_[q];
        if (!o.any)
        {
            o.any = true;
            o.m[0] = a, o.m[1] = b, o.m[2] = c, o.m[3] = d;
            return;
        }
        const cl e[4] = {times(a, o.m[0]) + times(b, o.m[2]), times(a, o.m[1]) + times(b, o.m[3]), times(c, o.m[0]) + times(d, o.m[2]), times(c, o.m[1]) + times(d, o.m[3])};
        std::copy(e, e + 4, o.m);
    }

    // Before an operation that is diagonal in q: writes q's pending gates up to a phase of |1>,
    // which stays pending (as [[1, 0], [0, p]]).
    void PassLowering::touch_z(int q)
    {
        One &o = one_[q];
        if (!o.any)
            return;
        cl *m = o.m;
        const cl zero(0.0), one(1.0);
        if (m[1] == zero && m[2] == zero)
        { // m00 [[1, 0], [0, m11 / m00]]
            if (m[0] != one)
            {
                global_ = times(global_, m[0]);
                m[3] = unit(over(m[3], m[0]));
                m[0] = 1.0;
            }
        }
        else if (m[0] == zero && m[3] == zero)
        { // [[0, b], [c, 0]] = b [[1, 0], [0, c / b]] X
            out_.push_back(PassGate{q, qsv::kPassFlip, 0, 0, {}});
            global_ = times(global_, m[1]);
            m[3] = unit(over(m[2], m[1]));
            m[0] = 1.0;
            m[1] = m[2] = 0.0;
        }
        else if (m[0] == m[1] && m[0] == m[2] && m[3] == -m[0] && m[0].imag() == 0.0)
        {
            out_.push_back(PassGate{q, qsv::kPassHad, 0, 0, {double(m[0].real())}});
            o.any = false;
            return;
        }
        else if (m[0] == m[3] && m[1] == m[2] && m[0].imag() == 0.0 && m[1].real() == 0.0)
        { // [[c, -is], [-is, c]]; a negative c as -[[-c, is], [is, -c]]
            long double c = m[0].real(), sn = -m[1].imag();
            if (c < 0)
                c = -c, sn = -sn, global_ = -global_;
            PassGate g{q, qsv::kPassCross, 0, 0, {}};
            shears(c, sn, g.m);
            g.m[0] = -g.m[0];
            out_.push_back(g);
            o.any = false;
            return;
        }
        else
        {
            const Euler u = euler(m);
            PassGate g{q, qsv::kPassRot, 0, 0, {u.m[0], u.m[1]}};
            g.pre = cd(u.l);
            out_.push_back(g);
            global_ = times(global_, u.e);
            m[3] = u.p;
            m[0] = 1.0;
            m[1] = m[2] = 0.0;
        }
        o.any = m[3] != one;
    }

    // Before an operation on q that is not diagonal: nothing stays pending; returns the phase
    // of |1> that the operation has to apply first.
    cd PassLowering::touch_x(int q)
    {
        touch_z(q);
        One &o = one_[q];
        const cd p = o.any ? cd(o.m[3]) : kOne;
        o.any = false;
        return p;
    }

    void PassLowering::phase(uint64_t cmask, uint64_t cval, cl p)
    {
        // Entries of a gate lie off the unit circle by their rounding to double.  A ratio of several
        // of them would add that up (RZZ as the phase of both its qubits' |1>: four times); scaled
        // to modulus 1 it keeps their angles' errors only, as the gate has them.
        p = unit(p);
        if (p == cl(1.0))
            return;
        if (!cmask)
        {
            global_ = times(global_, p);
            return;
        }
        if (!(cmask & (cmask - 1)))
        { // one qubit: joins its pending gates
            const int q = __builtin_ctzll(cmask);
            cval ? mul(q, 1.0, 0.0, 0.0, p) : mul(q, p, 0.0, 0.0, 1.0);
            return;
        }
        for (uint64_t b = cmask; b; b &= b - 1)
            touch_z(__builtin_ctzll(b));
        out_.push_back(PassGate{-1, qsv::kPassPhase, cmask, cval, {double(p.real()), double(p.imag())}});
    }

    void PassLowering::two_by_two(int t, uint64_t cmask, uint64_t cval, cd a, cd b, cd c, cd d)
    {
        if (!cmask)
        {
            mul(t, a, b, c, d);
            return;
        }
        for (uint64_t q = cmask; q; q &= q - 1)
            touch_z(__builtin_ctzll(q));
        PassGate g{t, qsv::kPassRot, cmask, cval, {}};
        const cd zero(0.0);
        const bool re = a.imag() == 0.0 && b.imag() == 0.0 && c.imag() == 0.0 && d.imag() == 0.0;
        double sign = 1.0;
        if (a == zero && d == zero && b == kOne && c == kOne)
            g.kind = qsv::kPassFlip;
        else if (re && a == b && a == c && d == -a)
        {
            g.kind = qsv::kPassHad;
            g.m[0] = a.real();
        }
        else if (re && a == d && b == -c)
        { // [[c, -s], [s, c]]; a negative c as -[[-c, s], [-s, -c]] on the controlled part
            sign = a.real() < 0 ? -1.0 : 1.0;
            shears(sign * a.real(), sign * c.real(), g.m);
        }
        else if (a == d && b == c && a.imag() == 0.0 && b.real() == 0.0)
        {
            sign = a.real() < 0 ? -1.0 : 1.0;
            g.kind = qsv::kPassCross;
            shears(sign * a.real(), -sign * b.imag(), g.m);
            g.m[0] = -g.m[0];
        }
        else
        { // controlled phases around a controlled rotation
            const cl m[4] = {a, b, c, d};
            const Euler u = euler(m);
            phase(cmask | bit(t), cval | bit(t), u.l);
            if (u.m[1] != 0.0)
            {
                g.m[0] = u.m[0];
                g.m[1] = u.m[1];
                g.pre = touch_x(t);
                out_.push_back(g);
            }
            phase(cmask | bit(t), cval | bit(t), u.p);
            phase(cmask, cval, u.e);
            return;
        }
        g.pre = touch_x(t);
        out_.push_back(g);
        if (sign < 0)
            phase(cmask, cval, -1.0);
    }

    std::vector<PassGate> PassLowering::finish()
    {
        for (int q = 0; q < (int)one_.size(); ++q)
        {
            touch_z(q);
            if (one_[q].any)
                out_.push_back(PassGate{-1, qsv::kPassPhase, bit(q), bit(q), {double(one_[q].m[3].real()), double(one_[q].m[3].imag())}});
            one_[q].any = false;
        }
        global_ = unit(global_); // a product of phases: only rounding takes it off the circle
        if (global_ != cl(1.0))
            out_.push_back(PassGate{-1, qsv::kPassPhase, 0, 0, {double(global_.real()), double(global_.imag())}});
        global_ = 1.0;
        return std::move(out_);
    }

    static bool finite(const GateSpec &s)
    {
        double zero = 0.0;
        auto look = [&](const cd *z, int count) {
            for (int i = 0; i < count; ++i)
                zero += 0.0 * z[i].real() + 0.0 * z[i].imag();
        };
        look(s.phase, 4);
        look(s.m, s.kind == Kind::Dense4 ? 16 : 4);
        look(s.coef, s.nrows);
        return zero == 0.0;
    }

    bool PassLowering::add(const ResolvedGate &g)
    {
        const GateSpec &s = g.spec;
        // multiplied into others, an angle that is no number would reach amplitudes that its gate
        // leaves alone
        if (g.mmask || !finite(s))
            return false;
        uint64_t c1 = 0, c0 = 0;
        for (int q : g.pphys)
            c1 |= bit(q);
        for (int q : g.nphys)
            c0 |= bit(q);
        const uint64_t cm = c0 | c1, cv = c1;
        const auto &t = g.tphys;
        // a 4x4 on (t0, t1) whose nonzeros pair the indices that agree on one bit, or on their
        // parity
        auto dense4 = [&](const cd *M) {
            const int a = t[0], b = t[1];
            for (int pre = 0; pre < 3; ++pre) // M = M' X on nothing, t0 or t1
            {
                const int x = pre == 0 ? 0 : pre == 1 ? 1 : 2;
                auto n = [&](int r, int c) { return M[4 * r + (c ^ x)]; };
                auto closed = [&](auto same) {
                    for (int r = 0; r < 4; ++r)
                        for (int c = 0; c < 4; ++c)
                            if (!same(r, c) && n(r, c) != cd(0.0))
                                return false;
                    return true;
                };
                const bool by0 = closed([](int r, int c) { return (r & 1) == (c & 1); });
                const bool by1 = !by0 && closed([](int r, int c) { return (r & 2) == (c & 2); });
                const bool par = !by0 && !by1 && closed([](int r, int c) { return (((r ^ c) & 1) ^ (((r ^ c) >> 1) & 1)) == 0; });
                if (!by0 && !by1 && !par)
                    continue;
                if (pre)
                    flip(pre == 1 ? a : b, cm, cv);
                if (by0) // t0 picks a 2x2 on t1
                    for (int v = 0; v < 2; ++v)
                        two_by_two(b, cm | bit(a), cv | (v ? bit(a) : 0), n(v, v), n(v, v + 2), n(v + 2, v), n(v + 2, v + 2));
                else if (by1)
                    for (int v = 0; v < 2; ++v)
                        two_by_two(a, cm | bit(b), cv | (v ? bit(b) : 0), n(2 * v, 2 * v), n(2 * v, 2 * v + 1), n(2 * v + 1, 2 * v), n(2 * v + 1, 2 * v + 1));
                else
                {
                    // after a CNOT t0 -> t1, t1 holds the parity: even indices (0, 3), odd (2, 1)
                    flip(b, bit(a), bit(a));
                    two_by_two(a, cm | bit(b), cv, n(0, 0), n(0, 3), n(3, 0), n(3, 3));
                    two_by_two(a, cm | bit(b), cv | bit(b), n(2, 2), n(2, 1), n(1, 2), n(1, 1));
                    flip(b, bit(a), bit(a));
                }
                return true;
            }
            return false;
        };
        switch (s.kind)
        {
        case Kind::Identity:
            return true;
        case Kind::GlobalPhase:
            phase(cm, cv, s.phase[0]);
            return true;
        case Kind::PhaseOne:
            phase(cm | bit(t[0]), cv | bit(t[0]), s.phase[1]);
            return true;
        case Kind::Diag1:
            if (!cm)
                mul(t[0], s.phase[0], 0.0, 0.0, s.phase[1]);
            else
            {
                phase(cm, cv, s.phase[0]);
                phase(cm | bit(t[0]), cv | bit(t[0]), over(s.phase[1], s.phase[0]));
            }
            return true;
        case Kind::Diag2:
        {
            const uint64_t a = bit(t[0]), b = bit(t[1]);
            phase(cm, cv, s.phase[0]);
            phase(cm | a, cv | a, over(s.phase[1], s.phase[0]));
            phase(cm | b, cv | b, over(s.phase[2], s.phase[0]));
            phase(cm | a | b, cv | a | b, over(times(s.phase[3], s.phase[0]), times(s.phase[1], s.phase[2])));
            return true;
        }
        case Kind::Pair1:
            two_by_two(t[0], cm, cv, s.m[0], s.m[1], s.m[2], s.m[3]);
            return true;
        case Kind::PairSub:
        {
            const int a = t[0], b = t[1];
            const bool odd = s.pat[0] == 1 && s.pat[1] == 2, even = s.pat[0] == 0 && s.pat[1] == 3;
            if (!odd && !even)
                return false;
            // after the CNOT, t1 holds the parity of the pattern; for 1 and 2, t0 = 1 is pattern
            // 1 and t0 = 0 pattern 2; for 0 and 3, t0 = 0 is pattern 0 and t0 = 1 pattern 3
            flip(b, bit(a), bit(a));
            if (odd)
                two_by_two(a, cm | bit(b), cv | bit(b), s.m[3], s.m[2], s.m[1], s.m[0]);
            else
                two_by_two(a, cm | bit(b), cv, s.m[0], s.m[1], s.m[2], s.m[3]);
            flip(b, bit(a), bit(a));
            return true;
        }
        case Kind::Dense4:
            return dense4(s.m);
        case Kind::Mono:
        {
            if (s.ntargets == 2)
            { // dcx: CNOT t0 -> t1, then t1 -> t0
                if (s.nrows != 3 || s.row[0] != 1 || s.src[0] != 3 || s.row[1] != 2 || s.src[1] != 1 || s.row[2] != 3 || s.src[2] != 2)
                    return false;
                for (int k = 0; k < 3; ++k)
                    if (s.coef[k] != kOne)
                        return false;
                flip(t[1], cm | bit(t[0]), cv | bit(t[0]));
                flip(t[0], cm | bit(t[1]), cv | bit(t[1]));
                return true;
            }
            // rows in place, and pairs of rows one bit apart that exchange
            uint64_t tm = 0;
            for (int q : t)
                tm |= bit(q);
            auto pattern = [&](int k) {
                uint64_t v = 0;
                for (int j = 0; j < s.ntargets; ++j)
                    if ((k >> j) & 1)
                        v |= bit(t[j]);
                return v;
            };
            auto partner = [&](int k) {
                for (int j = 0; j < s.nrows; ++j)
                    if (s.row[j] == s.src[k] && s.src[j] == s.row[k])
                        return j;
                return -1;
            };
            for (int k = 0; k < s.nrows; ++k)
                if (s.row[k] != s.src[k] && (__builtin_popcount(s.row[k] ^ s.src[k]) != 1 || partner(k) < 0))
                    return false;
            for (int k = 0; k < s.nrows; ++k)
            {
                const int r = s.row[k], c = s.src[k];
                if (r == c)
                    phase(cm | tm, cv | pattern(r), s.coef[k]);
                else if (r < c)
                {
                    const int q = t[__builtin_ctz(unsigned(r ^ c))];
                    two_by_two(q, cm | (tm & ~bit(q)), cv | (pattern(r) & ~bit(q)), 0.0, s.coef[k], s.coef[partner(k)], 0.0);
                }
            }
            return true;
        }
        }
        return false;
    }

    // Small states are one tile in one workgroup, larger ones want several workgroups a CU more
    // than few passes.  Kernel time of whole circuits in us, by tile bits (10 / 11 / 12 / 13):
    // 11 qubits, 6 RY RZ CNOT layers 51 / 54; 12 qubits 63 / 60 / 62 (4 / 2 / 1 passes); 13 qubits
    // - / 67 / - / 90; 18 qubits, GHZ and 10 U3 CZ layers 139 / 127 / 135; 20 qubits, 20 layers
    // - / 430 / 389 / 438; 26 qubits, brick depth 6 - / - / 2523 / 2661; 30 qubits, depth 3
    // - / - / 27168 / 29108.
    int pass_tile_bits(int n)
    {
        if (n <= 12)
            return std::max(n, qsv::kPassMinBits);
        return n <= 18 ? 11 : 12;
    }

    namespace
    {
        // Gates still to be planned, by index and in order.  They are taken from the front part that
        // a scan covers: what stays of it moves up to the rest, so that a round costs what it scans
        // and not what is left of the circuit.
        class Remaining
        {
        public:
            Remaining() = default;
            explicit Remaining(const std::vector<PassGate> &gates) : Remaining(gates, all(gates.size())) {}
            Remaining(const std::vector<PassGate> &gates, std::vector<int> indices) : v_(std::move(indices))
            {
                for (int i : v_)
                    count(gates[i], 1);
            }
            const int *data() const { return v_.data() + head_; }
            size_t size() const { return v_.size() - head_; }
            bool empty() const { return size() == 0; }
            // qubits that a remaining 2x2 has as its target; a scan need not wait for others
            uint64_t targets() const { return targets_; }
            bool phases_only() const { return targets_ == 0; }

            // Goes through the gates until more(gate) is false; those that ok(gate) chooses are
            // appended to taken, the others stay.
            template <class Ok, class More>
            void take(const std::vector<PassGate> &gates, std::vector<int> &taken, Ok ok, More more)
            {
                stay_.clear();
                size_t i = head_;
                for (bool go = true; go && i < v_.size(); ++i)
                {
                    const PassGate &g = gates[v_[i]];
                    if (ok(g))
                    {
                        taken.push_back(v_[i]);
                        count(g, -1);
                    }
                    else
                        stay_.push_back(v_[i]);
                    go = more(g);
                }
                head_ = i - stay_.size();
                std::copy(stay_.begin(), stay_.end(), v_.begin() + long(head_));
            }
            // the first ones, phases or not
            void take_front(const std::vector<PassGate> &gates, std::vector<int> &taken, size_t most)
            {
                for (; most > 0 && !empty(); --most, ++head_)
                {
                    taken.push_back(*data());
                    count(gates[*data()], -1);
                }
            }
            // takes gates back in, `back` in order
            void put_back(const std::vector<PassGate> &gates, const std::vector<int> &back)
            {
                for (int i : back)
                    count(gates[i], 1);
                if (back.size() > head_)
                {
                    std::vector<int> merged;
                    merged.reserve(size() + back.size());
                    std::merge(v_.begin() + long(head_), v_.end(), back.begin(), back.end(), std::back_inserter(merged));
                    v_.swap(merged);
                    head_ = 0;
                    return;
                }
                size_t to = head_ - back.size(), from = head_;
                head_ = to;
                for (int b : back)
                {
                    while (from < v_.size() && v_[from] < b)
                        v_[to++] = v_[from++];
                    v_[to++] = b;
                }
            }

        private:
            std::vector<int> v_, stay_;
            size_t head_ = 0;
            uint64_t targets_ = 0;
            int left_[64] = {}; // 2x2s by target

            static std::vector<int> all(size_t n)
            {
                std::vector<int> v(n);
                for (size_t i = 0; i < n; ++i)
                    v[i] = int(i);
                return v;
            }
            void count(const PassGate &g, int by)
            {
                if (g.t < 0)
                    return;
                left_[g.t] += by;
                targets_ = left_[g.t] ? targets_ | bit(g.t) : targets_ & ~bit(g.t);
            }
        };

        // Which gates of `rem` can be applied with 2x2 targets in `targets` only; `no_control`: qubits
        // that a 2x2 other than a flip may not be controlled by.  Scans stop once no target is left
        // that a later 2x2 could use, or `most` 2x2s are taken.
        struct Frontier
        {
            uint64_t x = 0, z = 0; // qubits with a deferred 2x2 target, a deferred control or phase
            bool free(const PassGate &g) const
            {
                const uint64_t tb = g.t >= 0 ? bit(g.t) : 0;
                return !(tb & (x | z)) && !(g.cmask & x);
            }
            void defer(const PassGate &g)
            {
                if (g.t >= 0)
                    x |= bit(g.t);
                z |= g.cmask;
            }
        };

        bool is_dense(const PassGate &g) { return g.t >= 0 && g.kind != qsv::kPassFlip; }
        // instructions per pair of amplitudes, roughly
        int weight(const PassGate &g)
        {
            if (g.t < 0)
                return 1;
            return g.kind == qsv::kPassFlip ? 6 : g.pre == kOne ? 6 : 10;
        }

        // weight of the 2x2s of rem that a fixed target set takes
        int count_take(const std::vector<PassGate> &gates, const Remaining &rem, uint64_t targets, uint64_t no_control, size_t most = ~size_t(0))
        {
            Frontier f;
            int w = 0;
            const int *at = rem.data();
            targets &= rem.targets();
            for (size_t i = 0; i < rem.size(); ++i)
            {
                const PassGate &g = gates[at[i]];
                const bool ok = f.free(g) && (g.t < 0 || ((targets >> g.t) & 1)) && !(is_dense(g) && (g.cmask & no_control));
                if (!ok)
                {
                    f.defer(g);
                    if (!(targets & ~(f.x | f.z)))
                        break;
                }
                else if (g.t >= 0)
                {
                    w += weight(g);
                    if (--most == 0)
                        break;
                }
            }
            return w;
        }

        // a target set of at most `room` more qubits, grown over the gates in order
        uint64_t grow(const std::vector<PassGate> &gates, const Remaining &rem, uint64_t allowed, uint64_t start, int room, bool avoid_controls, uint64_t &avoid, size_t most = ~size_t(0))
        {
            Frontier f;
            uint64_t set = start;
            avoid = 0;
            const int *at = rem.data();
            for (size_t i = 0; i < rem.size(); ++i)
            {
                const PassGate &g = gates[at[i]];
                bool ok = f.free(g);
                if (ok && g.t >= 0)
                {
                    const bool in = (set >> g.t) & 1;
                    if (!in && (room == 0 || !((allowed >> g.t) & 1) || ((avoid >> g.t) & 1)))
                        ok = false;
                    else if (avoid_controls && is_dense(g) && ((g.cmask & set) || __builtin_popcountll(allowed & ~(avoid | g.cmask)) < 4))
                        ok = false;
                    else
                    {
                        if (!in)
                        {
                            set |= bit(g.t);
                            --room;
                        }
                        if (avoid_controls && is_dense(g))
                            avoid |= g.cmask;
                    }
                }
                if (!ok)
                {
                    f.defer(g);
                    if (!((room > 0 ? set | (allowed & ~avoid) : set) & rem.targets() & ~(f.x | f.z)))
                        break;
                }
                else if (g.t >= 0 && --most == 0)
                    break;
            }
            return set;
        }

        // moves the gates that the target set takes from rem to taken
        void take(const std::vector<PassGate> &gates, Remaining &rem, uint64_t targets, uint64_t no_control, std::vector<int> &taken, size_t most = ~size_t(0))
        {
            Frontier f;
            targets &= rem.targets();
            rem.take(
                gates, taken,
                [&](const PassGate &g) {
                    const bool ok = f.free(g) && (g.t < 0 || ((targets >> g.t) & 1)) && !(is_dense(g) && (g.cmask & no_control));
                    if (!ok)
                        f.defer(g);
                    else if (g.t >= 0)
                        --most;
                    return ok;
                },
                // with every target blocked nothing but phases could follow
                [&](const PassGate &) { return most > 0 && (targets & ~(f.x | f.z)); });
        }

        // A phase can wait until a 2x2 needs one of its qubits: of the gates just taken, the phases
        // that no later taken 2x2 waits for go back to rem (in order), unless only phases are
        // left.  They then join that 2x2's own phase instead of being multiplied in at the end
        // of each round.
        void put_back_phases(const std::vector<PassGate> &gates, std::vector<int> &taken, Remaining &rem)
        {
            if (rem.phases_only())
            {
                rem.take_front(gates, taken, rem.size());
                return;
            }
            uint64_t needed = 0;
            std::vector<int> keep, back;
            for (size_t i = taken.size(); i-- > 0;)
            {
                const PassGate &g = gates[taken[i]];
                if (g.t >= 0)
                    needed |= bit(g.t);
                (g.t >= 0 || (g.cmask & needed) ? keep : back).push_back(taken[i]);
            }
            if (back.empty())
                return;
            std::reverse(keep.begin(), keep.end());
            std::reverse(back.begin(), back.end());
            taken.swap(keep);
            rem.put_back(gates, back);
        }

        // Gates of a round: bounds its operations (at most two a gate, and the last flushes), so
        // that a round always fits the memory that programs pass through.
        constexpr size_t kRoundGates = (kProgramRoundOps - 2) / 2;

        // Of more gates taken than a round holds, those past its end go back to rem.
        void put_back_rest(const std::vector<PassGate> &gates, std::vector<int> &taken, Remaining &rem)
        {
            if (taken.size() <= kRoundGates)
                return;
            std::vector<int> back(taken.begin() + kRoundGates, taken.end());
            taken.resize(kRoundGates);
            std::sort(back.begin(), back.end()); // the circuit's order again
            rem.put_back(gates, back);
        }

        // Emits one round: register qubits reg[0..3] (ascending tile bits), the gates `taken`.
        void emit_round(PassPlan &P, const std::vector<PassGate> &gates, const uint8_t *tq, int m, uint32_t regbits, const std::vector<int> &taken)
        {
            qsv::PassRound R{};
            int nr = 0, nt = 0;
            int reg_of[64];
            std::fill(reg_of, reg_of + 64, -1);
            uint64_t regmask = 0;
            for (int b = 0; b < m; ++b)
            {
                if ((regbits >> b) & 1)
                {
                    R.rq[nr] = tq[b];
                    R.rl[nr] = 8 * qsv::pass_slot(1u << b);
                    reg_of[tq[b]] = nr++;
                    regmask |= bit(tq[b]);
                }
                else
                {
                    R.tq[nt] = tq[b];
                    R.tl[nt] = 8 * qsv::pass_slot(1u << b);
                    ++nt;
                }
            }
            if (nr != 4)
                throw std::runtime_error("pass: a round needs 4 register bits");
            R.first = uint32_t(P.ops.size());
            auto op = [&](uint32_t kind, uint32_t sel, uint64_t cmask, uint64_t cval, const double *mm) {
                qsv::PassOp o{};
                o.kind = kind;
                o.sel = sel;
                o.cmask = cmask;
                o.cval = cval;
                if (mm)
                    std::memcpy(o.m, mm, sizeof o.m);
                P.ops.push_back(o);
            };
            // register indices that match the register part of (cmask, cval)
            auto select = [&](uint64_t cmask, uint64_t cval) {
                uint32_t sel = 0;
                for (int r = 0; r < 16; ++r)
                {
                    bool on = true;
                    for (int j = 0; j < 4; ++j)
                        if ((cmask >> R.rq[j]) & 1)
                            on = on && ((r >> j) & 1) == int((cval >> R.rq[j]) & 1);
                    sel |= uint32_t(on) << r;
                }
                return sel;
            };
            bool pending = false;
            int pending_bit = -1;
            auto flush_bit = [&] {
                if (pending_bit >= 0)
                    op(qsv::kPassFlushBit + pending_bit, 0, 0, 0, nullptr), P.work += 16;
                pending_bit = -1;
            };
            // phases between two 2x2s commute: those on one register bit are taken together
            std::vector<const PassGate *> run[4];
            auto close_run = [&] {
                const int start = std::max(pending_bit, 0); // the open bit's first
                for (int j0 = 0; j0 < 4; ++j0)
                {
                    const int j = (start + j0) & 3;
                    if (run[j].empty())
                        continue;
                    if (pending_bit >= 0 && pending_bit != j)
                        flush_bit();
                    for (const PassGate *g : run[j])
                        op(qsv::kPassPhaseBit, 0, g->cmask & ~regmask, g->cval & ~regmask, g->m), P.work += 2;
                    pending_bit = j;
                }
                for (auto &v : run)
                    v.clear();
            };
            for (int gi : taken)
            {
                const PassGate &g = gates[gi];
                const uint64_t cm = g.cmask & ~regmask, cv = g.cval & ~regmask, rm = g.cmask & regmask;
                if (g.t < 0)
                {
                    if (!rm)
                        op(qsv::kPassPhase, 0, cm, cv, g.m), pending = true, P.work += 2;
                    else if (!(rm & (rm - 1)) && (g.cval & rm))
                        run[reg_of[__builtin_ctzll(rm)]].push_back(&g);
                    else
                    {
                        const uint32_t sel = select(g.cmask, g.cval);
                        uint32_t kind = qsv::kPassPhaseSel;
                        if (__builtin_popcountll(rm) == 2 && (g.cval & rm) == rm)
                        { // pairs 01 02 03 12 13 23
                            const int a = reg_of[__builtin_ctzll(rm)], b = reg_of[63 - __builtin_clzll(rm)];
                            kind = qsv::kPassPhasePair + (a == 0 ? b - 1 : a == 1 ? b + 1 : 5);
                        }
                        op(kind, sel, cm, cv, g.m), P.work += 2 * __builtin_popcount(sel);
                    }
                    continue;
                }
                close_run();
                const int j = reg_of[g.t];
                if (j < 0 || (is_dense(g) && rm))
                    throw std::runtime_error("pass: a 2x2 outside its round's registers");
                double m[4];
                std::memcpy(m, g.m, sizeof m);
                const uint32_t sel = is_dense(g) ? 0xffffu : select(g.cmask, g.cval);
                uint32_t kind = g.kind == qsv::kPassFlip && sel != 0xffffu ? uint32_t(qsv::kPassFlipSel) : g.kind;
                if (g.pre != kOne)
                {
                    const double pre[4] = {g.pre.real(), g.pre.imag()};
                    if (pending_bit == j) // joins the pending phase
                        op(qsv::kPassPhaseBit, 0, 0, 0, pre), P.work += 2;
                    else if (kind == qsv::kPassRot && !g.cmask)
                    {
                        kind = qsv::kPassTurnRot;
                        m[2] = pre[0];
                        m[3] = pre[1];
                    }
                    else
                        op(qsv::kPassTurnBit + j, 0, 0, 0, pre), P.work += 16;
                }
                if (pending_bit == j)
                    flush_bit();
                op(kind + j, sel, cm, cv, m);
                P.work += 4 * weight(g);
            }
            close_run();
            flush_bit();
            if (pending)
                op(qsv::kPassFlush, 0, 0, 0, nullptr), P.work += 32;
            R.count = uint32_t(P.ops.size()) - R.first;
            P.rounds.push_back(R);
            P.work += 16; // the exchange
        }

        // the rounds of one sweep over the tile tq[0..m-1]
        void plan_rounds(PassPlan &P, const std::vector<PassGate> &gates, Remaining rem, const uint8_t *tq, int n, int m, int line_bits)
        {
            uint64_t tile = 0;
            for (int b = 0; b < m; ++b)
                tile |= bit(tq[b]);
            auto bits_of = [&](uint64_t qubits) {
                uint32_t r = 0;
                for (int b = 0; b < m; ++b)
                    if ((qubits >> tq[b]) & 1)
                        r |= 1u << b;
                return r;
            };
            // fill a register set to 4 with the highest tile qubits outside `avoid`; 0: no room
            auto fill = [&](uint64_t set, uint64_t avoid) {
                for (int b = m - 1; b >= 0 && __builtin_popcountll(set) < 4; --b)
                    if (!(avoid & bit(tq[b])))
                        set |= bit(tq[b]);
                return __builtin_popcountll(set) == 4 ? set : 0;
            };
            const uint64_t low = line_bits ? (bit(line_bits) - 1) : 0; // kept out of first and last rounds
            const uint64_t top = fill(0, 0);
            uint64_t last = 0;
            bool first = true;
            std::vector<int> taken;
            while (!rem.empty())
            {
                taken.clear();
                uint64_t best = 0;
                int best_w = -1;
                const bool phases_only = rem.phases_only();
                auto consider = [&](uint64_t set) {
                    if (!set)
                        return;
                    int w = 4 * count_take(gates, rem, set, set, kRoundGates);
                    if (w == 0 && !phases_only)
                        return;
                    if (first && !(set & low))
                        w += 24; // saves an exchange
                    if (set == last)
                        w -= 1;
                    if (w > best_w)
                        best_w = w, best = set;
                };
                uint64_t avoid = 0;
                const uint64_t g0 = grow(gates, rem, tile, 0, 4, true, avoid, kRoundGates);
                consider(fill(g0, avoid));
                for (int b = 0; b + 4 <= std::min(m, n); ++b)
                    consider(bit(tq[b]) | bit(tq[b + 1]) | bit(tq[b + 2]) | bit(tq[b + 3]));
                if (best_w <= 0 && !fill(g0, avoid))
                    throw std::runtime_error("pass: no register set for a gate");
                take(gates, rem, best, best, taken, kRoundGates);
                if (taken.empty())
                    throw std::runtime_error("pass: planning does not advance");
                put_back_phases(gates, taken, rem);
                put_back_rest(gates, taken, rem);
                if (first && (best & low))
                    emit_round(P, gates, tq, m, bits_of(top), {});
                emit_round(P, gates, tq, m, bits_of(best), taken);
                last = best;
                first = false;
            }
            if (last & low)
                emit_round(P, gates, tq, m, bits_of(top), {});
        }
    } // namespace

    namespace
    {
        // a target set filled up to a tile of m qubits with the lowest others
        uint64_t fill_tile(uint64_t set, int n, int m)
        {
            for (int q = 0; q < n && __builtin_popcountll(set) < m; ++q)
                set |= bit(q);
            return set;
        }
    } // namespace

    std::vector<uint64_t> search_tiles(const std::vector<PassGate> &gates, int n, int m, int low_least, int low_most, int width, int count)
    {
        struct Kept
        {
            Remaining rem;
            std::vector<uint64_t> tiles;
            long left = 0; // weight of rem
        };
        std::vector<Kept> kept(1, Kept{Remaining(gates), {}, 0}), next;
        if (n <= m || width < 1 || count < 1 || low_least < 3 || low_most > 4)
            return {};
        std::vector<int> taken;
        std::vector<std::pair<int, uint64_t>> tries;
        while (!gates.empty())
        {
            next.clear();
            for (const Kept &k : kept)
            {
                tries.clear();
                auto add = [&](uint64_t set) {
                    set = fill_tile(set, n, m);
                    if (std::none_of(tries.begin(), tries.end(), [&](auto &t) { return t.second == set; }))
                        tries.push_back({count_take(gates, k.rem, set, 0), set});
                };
                for (int low_bits = low_least; low_bits <= low_most; ++low_bits)
                {
                    const uint64_t low = bit(low_bits) - 1;
                    uint64_t avoid;
                    add(grow(gates, k.rem, bit(n) - 1, low, m - low_bits, false, avoid));
                    for (int a = low_bits; a + (m - low_bits) <= n; ++a)
                        add(low | ((bit(m - low_bits) - 1) << a));
                }
                std::stable_sort(tries.begin(), tries.end(), [](auto &a, auto &b) { return a.first > b.first; });
                for (size_t t = 0; t < tries.size() && t < size_t(count); ++t)
                {
                    Kept x{k.rem, k.tiles, 0};
                    taken.clear();
                    take(gates, x.rem, tries[t].second, 0, taken);
                    if (taken.empty())
                        continue;
                    put_back_phases(gates, taken, x.rem);
                    x.tiles.push_back(tries[t].second);
                    if (x.rem.empty())
                        return x.tiles;
                    for (size_t i = 0; i < x.rem.size(); ++i)
                        x.left += weight(gates[x.rem.data()[i]]);
                    // one of those that leave as much: mostly the same tiles in another order
                    if (std::none_of(next.begin(), next.end(), [&](auto &o) { return o.left == x.left && o.rem.size() == x.rem.size(); }))
                        next.push_back(std::move(x));
                }
            }
            if (next.empty())
                return {};
            std::stable_sort(next.begin(), next.end(), [](auto &a, auto &b) { return a.left < b.left; });
            if (next.size() > size_t(width))
                next.resize(size_t(width));
            kept.swap(next);
        }
        return {};
    }

    PassPlan plan_passes(const std::vector<PassGate> &gates, int n, int m, int amp_bytes, int low_bits, const std::function<void(const PassPlan &, bool)> &planned, const std::vector<uint64_t> &tiles)
    {
        if (n < 1 || n > qsv::kMaxQubits || m < qsv::kPassMinBits || m > qsv::kPassMaxBits || (n < m && m != qsv::kPassMinBits) || low_bits < (amp_bytes == 16 ? 3 : 4) || low_bits > 4)
            throw std::runtime_error("passes: state or tile size out of range");
        PassPlan P;
        P.m = m;
        Remaining rem(gates);
        const int line_bits = n < 18 ? 0 : amp_bytes == 16 ? 3 : 4;
        std::vector<int> taken;
        while (!rem.empty())
        {
            PassPlan::Pass ps{};
            if (n <= m)
            {
                for (int b = 0; b < m; ++b)
                    ps.tq[b] = uint8_t(b);
                taken.clear();
                rem.take_front(gates, taken, rem.size());
            }
            else
            {
                // the low qubits (contiguous runs of amplitudes) and m - low_bits others: those of
                // the 2x2s in order, or the run of qubits that takes most
                const uint64_t low = bit(low_bits) - 1, all = (bit(n) - 1);
                uint64_t avoid, best = P.passes.size() < tiles.size() ? tiles[P.passes.size()] : grow(gates, rem, all, low, m - low_bits, false, avoid);
                if (tiles.empty())
                {
                    int best_w = count_take(gates, rem, best, 0);
                    for (int a = low_bits; a + (m - low_bits) <= n; ++a)
                    {
                        const uint64_t w = low | ((bit(m - low_bits) - 1) << a);
                        const int c = count_take(gates, rem, w, 0);
                        if (c > best_w)
                            best_w = c, best = w;
                    }
                    best = fill_tile(best, n, m);
                }
                int b = 0;
                for (int q = 0; q < n; ++q)
                    if ((best >> q) & 1)
                        ps.tq[b++] = uint8_t(q);
                taken.clear();
                take(gates, rem, best, 0, taken);
                if (taken.empty())
                    throw std::runtime_error("passes: planning does not advance");
                put_back_phases(gates, taken, rem);
            }
            ps.first_round = uint32_t(P.rounds.size());
            plan_rounds(P, gates, Remaining(gates, taken), ps.tq, n, m, line_bits);
            ps.nrounds = uint32_t(P.rounds.size()) - ps.first_round;
            P.passes.push_back(ps);
            if (planned)
                planned(P, rem.empty());
        }
        P.ops.resize(P.ops.size() + qsv::kPassOpPad, qsv::PassOp{});
        return P;
    }

    ProgramPart program_part(const PassPlan &P, uint32_t first, size_t room, bool split)
    {
        auto fits = [&](uint32_t end) { return ProgramPart{first, end}.bytes(P) + qsv::kPassOpPad * sizeof(qsv::PassOp) <= room; };
        ProgramPart part{first, first};
        for (const auto &ps : P.passes)
            if (const uint32_t end = ps.first_round + ps.nrounds; end > first)
            {
                if (!fits(end))
                    break;
                part.end = end;
            }
        if (part.end == first && split) // not even one pass: as many of its rounds
            while (part.end < P.rounds.size() && fits(part.end + 1))
                ++part.end;
        return part;
    }

    size_t ProgramPart::bytes(const PassPlan &P) const
    {
        return end == first ? 0 : qsv::pass_rounds_bytes(end - first) + (P.rounds[end - 1].first + P.rounds[end - 1].count - P.rounds[first].first) * sizeof(qsv::PassOp);
    }

    void ProgramPart::write(const PassPlan &P, char *to) const
    {
        const uint32_t first_op = P.rounds[first].first;
        for (uint32_t r = first; r < end; ++r)
        {
            qsv::PassRound R = P.rounds[r];
            R.first -= first_op;
            std::memcpy(to + (r - first) * sizeof R, &R, sizeof R);
        }
        const size_t at = qsv::pass_rounds_bytes(end - first);
        std::memcpy(to + at, P.ops.data() + first_op, bytes(P) - at);
    }
} // namespace qcore
