// Planning takes time in proportion to the circuit, also where a circuit uses few of the tile's
// qubits: microseconds a gate of 16 times the gates against those of a short list, the best of
// five each.  (Scans that run to the circuit's end take 16 times as long a gate.)
#include "pass.hpp"

#include <algorithm>
#include <chrono>
#include <cstdio>

using namespace qcore;

static double us_per_gate(int n, int used, int count)
{
    uint64_t s = 7;
    auto next = [&](int k) {
        s = s * 6364136223846793005ull + 1442695040888963407ull;
        return int((s >> 33) % uint64_t(k));
    };
    PassLowering lowering(n);
    for (int i = 0; i < count; ++i)
    {
        const double prm[3] = {0.3 + i, 0.2, 0.1 * i};
        ResolvedGate g;
        const int t = next(used), c = next(used);
        g.spec = make_gate(c == t ? "u3" : "x", prm);
        g.tphys = {t};
        if (c != t)
            g.pphys = {c};
        lowering.add(g);
    }
    const std::vector<PassGate> low = lowering.finish();
    const int m = pass_tile_bits(n);
    double best = 1e30;
    for (int k = 0; k < 5; ++k)
    {
        const auto t0 = std::chrono::steady_clock::now();
        const PassPlan P = plan_passes(low, n, m, 16, 3);
        best = std::min(best, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count());
        if (P.ops.empty())
            return 1e30;
    }
    return best / count;
}

int main()
{
    for (const auto &[n, used] : {std::pair{4, 4}, {9, 6}, {13, 5}, {20, 8}})
    {
        const double a = us_per_gate(n, used, 1000), b = us_per_gate(n, used, 16000);
        std::printf("n %d, %d qubits used: %.2f us a gate of 1000, %.2f of 16000\n", n, used, a, b);
        if (b > 4 * a)
            return 1;
    }
    std::printf("ok\n");
    return 0;
}
