// Pass programs in parts on the CPU: long circuits whose programs go to the device through areas
// of several sizes.  The parts have to hold every round once, in order, with its own operations,
// fit their area, and cut passes only where asked to; and rounds of more gates than one holds
// have to leave the state that the gates leave (the interpreter of pass_check.cpp).
#define main pass_check_main
#include "pass_check.cpp"
#undef main

static void check_parts(const PassPlan &P, size_t room, bool split, int c)
{
    const size_t pad = qsv::kPassOpPad * sizeof(qsv::PassOp);
    std::vector<char> area(room);
    uint32_t at = 0;
    while (at < P.rounds.size())
    {
        const ProgramPart part = program_part(P, at, room, split);
        if (part.first != at || part.end < at || part.end > P.rounds.size())
            fail("a part is out of order", c);
        if (part.end == at)
        { // no room for the next pass; a round always has
            if (split)
                fail("a round does not fit", c);
            size_t need = 0;
            for (const auto &ps : P.passes)
                if (ps.first_round <= at && at < ps.first_round + ps.nrounds)
                    need = ProgramPart{at, ps.first_round + ps.nrounds}.bytes(P) + pad;
            if (need <= room)
                fail("a pass that fits was left out", c);
            return;
        }
        bool whole = false;
        for (const auto &ps : P.passes)
            whole = whole || part.end == ps.first_round + ps.nrounds;
        if (!whole && !split)
            fail("a pass was cut unasked", c);
        const size_t bytes = part.bytes(P);
        if (bytes + pad > room || bytes % 64)
            fail("a part's size", c);
        std::memset(area.data(), 0x55, room);
        part.write(P, area.data());
        const auto *ops = reinterpret_cast<const qsv::PassOp *>(area.data() + qsv::pass_rounds_bytes(part.end - part.first));
        for (uint32_t r = part.first; r < part.end; ++r)
        {
            qsv::PassRound R;
            std::memcpy(&R, area.data() + (r - part.first) * sizeof R, sizeof R);
            if (R.count > kProgramRoundOps)
                fail("a round of too many operations", c);
            if (reinterpret_cast<const char *>(ops + R.first + R.count) > area.data() + bytes || std::memcmp(ops + R.first, &P.ops[P.rounds[r].first], R.count * sizeof *ops))
                fail("a round's operations", c);
            R.first = P.rounds[r].first;
            if (std::memcmp(&R, &P.rounds[r], sizeof R))
                fail("a round", c);
        }
        at = part.end;
    }
}

int main(int argc, char **argv)
{
    uint64_t seed = argc > 1 ? std::strtoull(argv[1], nullptr, 10) : 1;
    struct Case
    {
        int n, m, gates;
        enum { Any, Phases, Flips, PhasesFirst } kind;
    };
    // one tile and many; any gates, doubly controlled phases, and Hadamards
    // and CNOTs, which all run in one round where 4 qubits are all there are; 400 phases before 100
    // other gates, and 400 after them
    for (const Case &k : {Case{4, 10, 1500, Case::Flips}, {4, 10, 1500, Case::Any}, {9, 10, 2500, Case::Any}, {5, 10, 1400, Case::Phases}, {12, 12, 1200, Case::Any}, {12, 12, 6000, Case::Flips}, {13, 11, 1500, Case::Any}, {14, 11, 700, Case::Phases}, {6, 10, 900, Case::PhasesFirst}, {14, 11, 900, Case::PhasesFirst}})
    {
        const int c = k.n;
        PassLowering lowering(k.n);
        std::vector<ResolvedGate> gates;
        for (int i = 0; i < k.gates; ++i)
        {
            double prm[4];
            for (double &p : prm)
                p = 6.283 * unif(seed) - 3.14;
            ResolvedGate g;
            const bool phase = k.kind == Case::Phases || (k.kind == Case::PhasesFirst && (i < 400 || i >= 500));
            const int nc = phase ? 2 : int(mix(seed) % 2);
            g.spec = make_gate(phase ? "p" : k.kind == Case::Flips ? (nc ? "x" : "h") : kNames[mix(seed) % 21], prm);
            int qs[64];
            for (int q = 0; q < k.n; ++q)
                qs[q] = q;
            for (int q = k.n - 1; q > 0; --q)
                std::swap(qs[q], qs[mix(seed) % uint64_t(q + 1)]);
            g.tphys = {qs[0]};
            for (int j = 0; j < nc; ++j)
                g.pphys.push_back(qs[1 + j]);
            if (!lowering.add(g))
                fail("a gate was not lowered", c);
            gates.push_back(g);
        }
        const std::vector<PassGate> low = lowering.finish();
        const PassPlan P = plan_passes(low, k.n, k.m, 16, 3);
        size_t longest = 0;
        for (const auto &R : P.rounds)
            longest = std::max<size_t>(longest, R.count);
        for (size_t room : {kProgramRoundOps * 64 + 144 + 48 + 128, size_t(40000), size_t(64) << 10, size_t(512) << 10})
            for (bool split : {true, false})
                check_parts(P, room, split, c);
        if (program_part(P, 0, 200, true).end != 0)
            fail("a part in no room", c);
        std::vector<cd> a(1ull << k.n);
        for (auto &z : a)
            z = cd(unif(seed) - 0.5, unif(seed) - 0.5);
        std::vector<cd> b = a;
        for (const auto &g : gates)
            apply_direct(a, k.n, g);
        run_program(b, k.n, P, 16, c);
        double err = 0;
        for (size_t i = 0; i < a.size(); ++i)
            err = std::max(err, std::abs(a[i] - b[i]));
        std::printf("n %d: %zu gates, %zu operations, %zu passes, %zu rounds of at most %zu, max|d| %.1e\n", k.n, gates.size(), P.ops.size(), P.passes.size(), P.rounds.size(), longest, err);
        if (!(err <= k.gates * 16 * 2.3e-16))
            fail("the program's state differs from the gates'", c);
        if (k.n == 4 && k.kind == Case::Flips && longest < 255)
            fail("the case's rounds are not full", c);
    }
    std::printf("ok\n");
    return 0;
}
