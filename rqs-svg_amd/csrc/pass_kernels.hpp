// Launch interface of the circuit-pass kernel (pass_kernels.hip).
#pragma once
#include "sv_kernels.hpp"

namespace qsv
{
    // What one operation of a round does.  "Registers": the 4 tile bits whose 16 amplitudes a
    // thread holds.  Every operation acts on the threads whose amplitude index matches (cmask,
    // cval), bits outside the registers, inside the tile or not.
    enum PassKind : uint32_t
    {
        // + register bit t; u, v: the amplitudes with bit t 0 and 1.  Rotations run as three
        // shears (6 FP64 instructions a pair, where a complex 2x2 takes 16).
        kPassTurnRot = 0,   // v *= (m[2], m[3]), then kPassRot
        kPassRot = 4,       // u += m[0] v, v += m[1] u, u += m[0] v: [[c, -s], [s, c]] with m[0] = -s / (1 + c), m[1] = s
        kPassFlip = 8,      // u <-> v
        kPassPhase = 12,    // the thread's pending phase times (m[0], m[1])
        kPassPhaseBit = 13, // the pending phase of one register bit times (m[0], m[1])
        kPassPhaseSel = 14, // the amplitudes selected by sel times (m[0], m[1])
        kPassFlush = 15,    // the thread's pending phase into its amplitudes
        kPassFlushBit = 16, // + register bit: the pending phase into the amplitudes with it set
        kPassTurnBit = 20,  // + register bit: v *= (m[0], m[1])
        kPassCross = 24,    // + register bit: [[c, -is], [-is, c]] with m[0] = s / (1 + c), m[1] = s, as shears
        kPassHad = 28,      // + register bit: m[0] [[1, 1], [1, -1]]
        kPassFlipSel = 32,  // + register bit: u <-> v on the pairs selected by sel
        kPassPhasePair = 36, // + pair of register bits (01 02 03 12 13 23): amplitudes with both set times (m[0], m[1])
        kPassKinds = 42,
    };

    // One cache line, read by one scalar load.
    struct alignas(64) PassOp
    {
        uint32_t kind;
        uint32_t sel; // bit r: register index r (of a pair: its index with the bit 0)
        uint64_t cmask, cval;
        double m[4];
        uint32_t pad[2];
    };

    // A round: which tile bits are register bits (4) and which the thread-index bits, each
    // with its physical qubit and its LDS byte offset (8 pass_slot); the operations
    // ops[first .. first+count).
    struct PassRound
    {
        uint32_t rq[4], rl[4];
        uint32_t tq[12], tl[12];
        uint32_t first, count;
        uint32_t pad[2];
    };

    // operations that the kernel may read past a program's last one (it reads ahead)
    constexpr int kPassOpPad = 2;

    constexpr int kPassMinBits = 10, kPassMaxBits = 12;
    // LDS slot (8 B) of tile index i: bits 0..4 XOR the higher groups of 5 bits, linear over
    // GF(2), so that the 32 lanes of a half wave fall in different banks for most layouts.
    constexpr uint32_t pass_slot(uint32_t i) { return i ^ ((i >> 5) & 31u) ^ ((i >> 10) & 31u); }

    // One sweep of a 2^n-amplitude state: every tile of 2^m amplitudes (m = kPassMinBits ..
    // kPassMaxBits; tile qubits tq[0..m-1] ascending; for n < m the whole state, tile qubits
    // 0..m-1) goes through the rounds.  rounds and ops are device memory (nrounds rounds, kPassOpPad
    // operations past the last round's).
    template <class A>
    void launch_pass(hipStream_t s, A *state, int n, int m, const uint8_t *tq, const PassRound *rounds, int nrounds, const PassOp *ops);
} // namespace qsv
