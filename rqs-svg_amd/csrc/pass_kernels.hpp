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

    // Half a line, read by scalar loads of its own 64 bytes: programs place the operations, after
    // the rounds, on a multiple of that.
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
    struct alignas(16) PassRound
    {
        uint32_t rq[4], rl[4];
        uint32_t tq[12], tl[12];
        uint32_t first, count;
        uint32_t pad[2];
    };

    // bytes of `count` rounds with the padding to the operations behind them
    constexpr size_t pass_rounds_bytes(size_t count) { return (count * sizeof(PassRound) + alignof(PassOp) - 1) / alignof(PassOp) * alignof(PassOp); }

    // operations that the kernel may read past a program's last one (it reads ahead)
    constexpr int kPassOpPad = 2;

    constexpr int kPassMinBits = 10, kPassMaxBits = 12;
    // LDS slot (8 B) of tile index i: bits 0..4 XOR the higher groups of 5 bits, linear over
    // GF(2), so that the 32 lanes of a half wave fall in different banks for most layouts.
    constexpr uint32_t pass_slot(uint32_t i) { return i ^ ((i >> 5) & 31u) ^ ((i >> 10) & 31u); }

    // One sweep of a 2^n-amplitude state: every tile of 2^m amplitudes (m = kPassMinBits ..
    // kPassMaxBits; tile qubits tq[0..m-1] ascending; for n < m the whole state, tile qubits
    // 0..m-1) goes through the rounds.  rounds and ops are device memory (nrounds rounds, kPassOpPad
    // operations past the last round's), each aligned as its type.
    template <class A>
    void launch_pass(hipStream_t s, A *state, int n, int m, const uint8_t *tq, const PassRound *rounds, int nrounds, const PassOp *ops);

    // Copies a program (16-byte units) from pinned host memory to device memory.
    void launch_program_copy(hipStream_t s, void *dst, const void *src, size_t bytes);

    // One pass of one circuit among several (the batching form), complex64 states: tiles
    // tile_begin .. of the launch.  The first pass may start from |0...0> without reading, the
    // last one write its tiles' sums (kPassSums doubles each: all probabilities, then per
    // tile bit those with the bit 0 less those with it 1) in place of the amplitudes.  A circuit
    // of one tile does both (its amplitudes past 2^n stay zero), and its differences are its <Z>:
    // with its qubit count in flags from kPassQubits on, sums is where they go, qubit 0 first.
    constexpr uint32_t kPassZeroState = 1, kPassExpectZ = 2, kPassQubits = 8;
    constexpr int kPassSums = 16;
    struct alignas(16) PassTask
    {
        c64 *state;
        double *sums;
        uint32_t tile_begin, first_round, nrounds, flags;
        uint32_t tq[4]; // tile qubits, ascending, a byte each (words: they become scalar loads)
        uint8_t zb[16]; // tile bit of the last round's 4 register bits and its thread bits
    };
    // tasks in device memory, tile_begin ascending from 0; tiles: those of all tasks.
    void launch_pass_tasks(hipStream_t s, int m, bool nt, const PassTask *tasks, int ntasks, uint32_t tiles, const PassRound *rounds, const PassOp *ops);

    // <Z_q> of one qubit: the sum over tiles of sums[slot], negative where tile & sign.
    struct alignas(16) PassZ
    {
        const double *sums;
        double *out;
        uint32_t ntiles, slot, sign, pad;
    };
    void launch_pass_z(hipStream_t s, const PassZ *qubits, uint32_t count);
} // namespace qsv
