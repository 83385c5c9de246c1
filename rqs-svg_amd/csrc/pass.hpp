// Circuit passes, host side: gates lowered to controlled 2x2 and phase operations, grouped
// into sweeps of the state (pass_kernels.hpp) and into the rounds of each sweep.
#pragma once
#include "pass_kernels.hpp"
#include "simulator.hpp"

#include <functional>
#include <vector>

namespace qcore
{
    // What the lowering multiplies together is rounded to double once, when it is written.
    using cl = std::complex<long double>;

    // An operation on qubit t, or (t < 0) a phase, on the amplitudes whose index matches
    // (cmask, cval); physical qubits.  kind: kPassRot, kPassFlip, kPassCross or kPassHad.
    // pre: a phase of qubit t's |1> that comes first, on every amplitude.
    struct PassGate
    {
        int t;
        uint32_t kind;
        uint64_t cmask, cval;
        double m[4]; // as the kind's PassOp, or the phase in m[0..1]
        cd pre = 1.0;
    };

    // Lowers a gate list to PassGates.  Uncontrolled 1-qubit gates are multiplied together per
    // qubit (80-bit) and written as phase * rotation * phase only when another gate needs the
    // qubit; the trailing phase waits on, since it commutes with controls and phases.  A
    // 2-target gate becomes 2x2s between CNOTs (its matrix mixes amplitudes in pairs).
    class PassLowering
    {
    public:
        explicit PassLowering(int n) : one_(n) {}
        // false, with nothing changed, for a gate that has no such form (or holds no numbers)
        bool add(const ResolvedGate &g);
        // the operations of every gate added
        std::vector<PassGate> finish();

    private:
        struct One
        {
            bool any = false;
            cl m[4];
        };
        std::vector<One> one_; // pending 1-qubit gates, per qubit
        cl global_ = 1.0;
        std::vector<PassGate> out_;

        void mul(int q, cl a, cl b, cl c, cl d);
        void touch_z(int q);
        cd touch_x(int q);
        void phase(uint64_t cmask, uint64_t cval, cl p);
        void two_by_two(int t, uint64_t cmask, uint64_t cval, cd a, cd b, cd c, cd d);
        void flip(int t, uint64_t cmask, uint64_t cval) { two_by_two(t, cmask, cval, 0.0, 1.0, 1.0, 0.0); }
    };

    struct PassPlan
    {
        struct Pass
        {
            uint8_t tq[16];
            uint32_t first_round, nrounds;
        };
        int m = 0;
        std::vector<Pass> passes;
        std::vector<qsv::PassRound> rounds;
        std::vector<qsv::PassOp> ops; // the rounds' operations, then kPassOpPad unused ones
        // rough cost in FP64 instructions per amplitude and lane (for choosing a path)
        double work = 0;
    };

    // Tile bits of a pass over a state of n qubits.
    int pass_tile_bits(int n);

    // Sweeps that apply `gates` in an order equivalent to theirs: a gate may pass a deferred
    // one only if on every shared qubit both act as a control or a phase.  A 2x2's target has
    // to be a tile qubit; controls and phases need not be.  amp_bytes: 16 or 8 (complex64),
    // which decides the low qubits that the first and last round of a sweep keep in the
    // thread index, so that loads and stores cover whole lines.  low_bits: qubits 0 .. low_bits - 1
    // are in every tile (4, or 3 for complex128: one line of 128 bytes).  planned: called after each
    // pass with the plan so far and whether that is all of it.
    PassPlan plan_passes(const std::vector<PassGate> &gates, int n, int m, int amp_bytes, int low_bits = 4, const std::function<void(const PassPlan &, bool)> &planned = {}, const std::vector<uint64_t> &tiles = {});
    // Tiles (masks of m qubits) of a plan of few passes, for plan_passes: after each of the
    // `width` sequences kept, the `count` tiles that take most are tried (with the low_least to
    // low_most low qubits), and the sequences kept that leave least.  Empty if none is found.
    std::vector<uint64_t> search_tiles(const std::vector<PassGate> &gates, int n, int m, int low_least, int low_most, int width, int count);

    // Programs reach the device in parts: consecutive rounds with their operations, numbered
    // from the part's first.  Each round carries everything it needs, so a pass may be cut
    // between two of its rounds into sweeps of their own.
    struct ProgramPart
    {
        uint32_t first, end; // rounds
        size_t bytes(const PassPlan &P) const;
        void write(const PassPlan &P, char *to) const;
    };
    constexpr size_t kProgramRoundOps = 512; // operations of a round, at most
    // The rounds of P from `first` on that fit `room` bytes with the padding behind them: whole
    // passes, or (split) some rounds of one that does not fit; none if there is no room.
    ProgramPart program_part(const PassPlan &P, uint32_t first, size_t room, bool split);
} // namespace qcore
