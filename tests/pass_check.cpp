// Circuit passes on the CPU: random circuits over the whole gate table are lowered and planned
// by the library (PassLowering, plan_passes), the resulting program is run by an interpreter of
// its operations written from their definitions, and the state is compared with the gates'
// matrices applied one by one.  Also checked: every round's layout is a bijection of the tile,
// operations stay inside their round's registers, and the first and last round of a sweep of a
// large state keep the low qubits in the thread index.
#include "pass.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>

using namespace qcore;

static uint64_t mix(uint64_t &s)
{
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
static double unif(uint64_t &s) { return double(mix(s) >> 11) * 0x1.0p-53; }

static void fail(const char *what, int c)
{
    std::printf("FAIL case %d: %s\n", c, what);
    std::exit(1);
}

static const char *kNames[] = {"h", "x", "y", "z", "s", "sdg", "t", "tdg", "sx", "sxdg", "id", "rx", "ry", "rz", "u1", "p", "u2", "r", "u3", "u", "u4",
                               "swap", "iswap", "dcx", "ecr", "rxx", "ryy", "rzz", "rzx", "xx_plus_yy", "xx_minus_yy", "rccx", "rcccx", "global_phase"};

static void apply_direct(std::vector<cd> &psi, int n, const ResolvedGate &g)
{
    const auto U = dense_matrix(g.spec);
    const int t = g.spec.ntargets, T = 1 << t;
    uint64_t c1 = 0, c0 = 0, tm = 0;
    for (int q : g.pphys)
        c1 |= 1ull << q;
    for (int q : g.nphys)
        c0 |= 1ull << q;
    for (int q : g.tphys)
        tm |= 1ull << q;
    auto at = [&](uint64_t i, int k) {
        for (int j = 0; j < t; ++j)
            if ((k >> j) & 1)
                i |= 1ull << g.tphys[j];
        return i;
    };
    for (uint64_t i = 0; i < (1ull << n); ++i)
    {
        if ((i & tm) || (i & c1) != c1 || (i & c0))
            continue;
        cd in[16], out[16];
        for (int k = 0; k < T; ++k)
            in[k] = psi[at(i, k)];
        for (int r = 0; r < T; ++r)
        {
            out[r] = 0.0;
            for (int k = 0; k < T; ++k)
                out[r] += U[r * T + k] * in[k];
        }
        for (int k = 0; k < T; ++k)
            psi[at(i, k)] = out[k];
    }
}

static void run_program(std::vector<cd> &psi, int n, const PassPlan &P, int amp_bytes, int c)
{
    const uint64_t N = 1ull << n;
    const int line_bits = n < 18 ? 0 : amp_bytes == 16 ? 3 : 4;
    for (const auto &ps : P.passes)
    {
        uint64_t tile = 0;
        for (int b = 0; b < P.m; ++b)
            tile |= 1ull << ps.tq[b];
        if (ps.nrounds < 1)
            fail("a pass without rounds", c);
        for (uint32_t ri = 0; ri < ps.nrounds; ++ri)
        {
            const qsv::PassRound &R = P.rounds[ps.first_round + ri];
            uint64_t seen = 0, regs = 0;
            uint32_t slots = 0;
            for (int j = 0; j < 4; ++j)
            {
                seen |= 1ull << R.rq[j];
                regs |= 1ull << R.rq[j];
            }
            for (int j = 0; j < P.m - 4; ++j)
            {
                if ((seen >> R.tq[j]) & 1)
                    fail("a tile qubit twice in a layout", c);
                seen |= 1ull << R.tq[j];
            }
            if (seen != tile)
                fail("a layout does not cover the tile", c);
            // slot weights: the XOR of all of them over any subset is a bijection iff they are
            // independent; check by enumeration
            std::vector<char> hit(1u << P.m, 0);
            for (uint32_t x = 0; x < (1u << P.m); ++x)
            {
                slots = 0;
                for (int j = 0; j < 4; ++j)
                    if ((x >> j) & 1)
                        slots ^= R.rl[j];
                for (int j = 0; j < P.m - 4; ++j)
                    if ((x >> (4 + j)) & 1)
                        slots ^= R.tl[j];
                if (slots % 8 || slots / 8 >= (1u << P.m) || hit[slots / 8])
                    fail("LDS slots of a layout are not a bijection", c);
                hit[slots / 8] = 1;
            }
            if ((ri == 0 || ri + 1 == ps.nrounds) && (regs & ((1ull << line_bits) - 1)))
                fail("a line's qubits in the registers at a load or store", c);
            auto reg = [&](uint64_t i) {
                int r = 0;
                for (int j = 0; j < 4; ++j)
                    r |= int((i >> R.rq[j]) & 1) << j;
                return r;
            };
            std::vector<cd> pend(N, 1.0), pendb(N, 1.0);
            bool dirty = false, dirtyb = false;
            for (uint32_t k = 0; k < R.count; ++k)
            {
                const qsv::PassOp &o = P.ops[R.first + k];
                if (o.cmask & regs)
                    fail("a control mask on a register qubit", c);
                const cd z(o.m[0], o.m[1]);
                for (uint64_t i = 0; i < N; ++i)
                {
                    if ((i & o.cmask) != o.cval)
                        continue;
                    const int r = reg(i);
                    if (o.kind == qsv::kPassPhase)
                        pend[i] *= z, dirty = true;
                    else if (o.kind == qsv::kPassPhaseBit)
                        pendb[i] *= z, dirtyb = true;
                    else if (o.kind == qsv::kPassPhaseSel)
                    {
                        if ((o.sel >> r) & 1)
                            psi[i] *= z;
                    }
                    else if (o.kind >= qsv::kPassPhasePair && o.kind < qsv::kPassKinds)
                    {
                        const int lo[] = {0, 0, 0, 1, 1, 2}, hi[] = {1, 2, 3, 2, 3, 3}, k2 = int(o.kind) - qsv::kPassPhasePair;
                        if (((r >> lo[k2]) & 1) && ((r >> hi[k2]) & 1))
                            psi[i] *= z;
                    }
                    else if (o.kind == qsv::kPassFlush)
                        psi[i] *= pend[i], pend[i] = 1.0, dirty = false;
                    else if (o.kind >= qsv::kPassFlushBit && o.kind < qsv::kPassFlushBit + 4)
                    {
                        if ((r >> (o.kind - qsv::kPassFlushBit)) & 1)
                            psi[i] *= pendb[i];
                        pendb[i] = 1.0, dirtyb = false;
                    }
                    else
                    {
                        const int j = o.kind & 3;
                        if ((r >> j) & 1)
                            continue;
                        const uint64_t i1 = i | (1ull << R.rq[j]);
                        const cd a = psi[i], b = psi[i1];
                        // shears in real arithmetic, on the parts that they act on
                        auto shear = [&](double &u, double &v, double s0, double s1) {
                            u += s0 * v;
                            v += s1 * u;
                            u += s0 * v;
                        };
                        double ux = a.real(), uy = a.imag(), vx = b.real(), vy = b.imag();
                        switch (o.kind & ~3u)
                        {
                        case qsv::kPassFlip:
                            std::swap(psi[i], psi[i1]);
                            break;
                        case qsv::kPassFlipSel:
                            if ((o.sel >> r) & 1)
                                std::swap(psi[i], psi[i1]);
                            break;
                        case qsv::kPassTurnRot:
                        {
                            const cd w = b * cd(o.m[2], o.m[3]);
                            vx = w.real(), vy = w.imag();
                        }
                        [[fallthrough]];
                        case qsv::kPassRot:
                            shear(ux, vx, o.m[0], o.m[1]);
                            shear(uy, vy, o.m[0], o.m[1]);
                            psi[i] = cd(ux, uy), psi[i1] = cd(vx, vy);
                            break;
                        case qsv::kPassCross:
                            shear(ux, vy, o.m[0], -o.m[1]);
                            shear(uy, vx, -o.m[0], o.m[1]);
                            psi[i] = cd(ux, uy), psi[i1] = cd(vx, vy);
                            break;
                        case qsv::kPassHad:
                            psi[i] = o.m[0] * (a + b), psi[i1] = o.m[0] * (a - b);
                            break;
                        case qsv::kPassTurnBit:
                            psi[i1] = b * z;
                            break;
                        default:
                            fail("unknown operation", c);
                        }
                    }
                }
            }
            if (dirty || dirtyb)
                fail("a pending phase is left at the end of a round", c);
        }
    }
}

int main(int argc, char **argv)
{
    const int cases = argc > 1 ? std::atoi(argv[1]) : 20;
    uint64_t seed = argc > 2 ? std::strtoull(argv[2], nullptr, 10) : 1;
    for (int c = 0; c < cases; ++c)
    {
        // 1 .. 14 qubits with tiles of 2^10 amplitudes; every 8th case larger, on bigger tiles
        const bool big = c % 8 == 7;
        const int n = big ? 18 : 1 + int(mix(seed) % 14);
        const int m = big ? 11 + int(mix(seed) % 2) : (n == 11 || n == 12) && (mix(seed) & 1) ? n : 10;
        const int amp_bytes = (mix(seed) & 1) ? 16 : 8;
        const int ngates = big ? 24 : 1 + int(mix(seed) % 80);
        std::vector<ResolvedGate> gates;
        PassLowering lowering(n);
        for (int i = 0; i < ngates; ++i)
        {
            double prm[4];
            for (double &p : prm)
                p = 6.283 * unif(seed) - 3.14;
            ResolvedGate g;
            g.spec = make_gate(kNames[mix(seed) % (sizeof kNames / sizeof *kNames)], prm);
            const int t = g.spec.ntargets;
            int nc = int(mix(seed) % 8) < 4 ? 0 : int(mix(seed) % 4);
            if (t > n)
                continue;
            nc = std::min(nc, n - t);
            std::vector<int> qs(n);
            for (int q = 0; q < n; ++q)
                qs[q] = q;
            for (int q = n - 1; q > 0; --q)
                std::swap(qs[q], qs[mix(seed) % uint64_t(q + 1)]);
            g.tphys.assign(qs.begin(), qs.begin() + t);
            for (int j = 0; j < nc; ++j)
                ((mix(seed) & 1) ? g.pphys : g.nphys).push_back(qs[t + j]);
            if (!lowering.add(g))
                fail("a gate of the table was not lowered", c);
            gates.push_back(g);
        }
        const std::vector<PassGate> low = lowering.finish();
        const int low_bits = amp_bytes == 16 && (mix(seed) & 1) ? 3 : 4;
        const std::vector<uint64_t> tiles = mix(seed) & 1 ? search_tiles(low, n, m, low_bits, 4, 1 + int(mix(seed) % 4), 1 + int(mix(seed) % 6)) : std::vector<uint64_t>();
        const PassPlan P = plan_passes(low, n, m, amp_bytes, low_bits, {}, tiles);
        if (!tiles.empty() && P.passes.size() != tiles.size())
            fail("the plan does not follow its tiles", c);
        std::vector<cd> a(1ull << n);
        for (auto &z : a)
            z = cd(unif(seed) - 0.5, unif(seed) - 0.5);
        std::vector<cd> b = a;
        for (const auto &g : gates)
            apply_direct(a, n, g);
        run_program(b, n, P, amp_bytes, c);
        double err = 0;
        for (size_t i = 0; i < a.size(); ++i)
            err = std::max(err, std::abs(a[i] - b[i]));
        std::printf("case %d: n %d m %d, %zu gates, %zu operations, %zu passes, %zu rounds, max|d| %.1e\n", c, n, m, gates.size(), P.ops.size() - qsv::kPassOpPad, P.passes.size(), P.rounds.size(), err);
        // amplitudes of order 1, at most 80 gates of a few roundings each
        if (!(err <= 80 * 16 * 2.3e-16))
            fail("the program's state differs from the gates'", c);
    }
    std::printf("ok\n");
    return 0;
}
