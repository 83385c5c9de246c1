// Circuit passes: many gates applied to a state in one sweep, gate by gate in FP64.
//
// A workgroup takes a tile of 2^M amplitudes (the amplitudes that agree on every qubit
// outside the tile) into the registers of 2^(M-4) threads, 16 amplitudes each, and applies a
// list of rounds.  In a round the 16 amplitudes of a thread differ in 4 tile bits, the
// round's register bits: a gate whose target is one of them is 8 independent 2x2 products
// per thread with its matrix in scalar registers.  Controls and diagonal gates need no
// register bit: they test the amplitude index, on qubits inside or outside the tile alike.
// Phases that depend on no register bit, or on one, are collected per thread (one product)
// and multiplied into the amplitudes once.  Between rounds the tile is exchanged through LDS,
// real parts and then imaginary parts, so that 2^12 amplitudes take 32 KiB and 4 workgroups
// share a CU: one loads or stores while others compute.
//
// What bounds it.  A pass reads and writes the state once (30 qubits complex128: 34.4 GB,
// 5.5 ms at the pair kernel's rate); a gate costs 48 to 80 FP64 instructions per 1024
// amplitudes: 1-qubit gates run as phase * rotation * phase, the rotation as three in-place
// shears of 2 instructions a pair, the phases joined with those of controlled phases where a
// later gate flushes them (a complex 2x2 would take 128, and brick passes at 26 qubits then
// issued VALU instructions in all of their cycles, 3.19 ms for 4 passes; now 2.52 ms, VALU 78 %
// busy).  Passes of few gates run at the memory rate.  Measured, one kernel per gate -> passes:
// 30 qubits, brick depth 3 (138 gates) 577 -> 27 ms; 26 qubits, QFT (364 gates) in 2.5 ms; 20
// qubits, 20 U3 CZ layers (620 gates) 3.3 -> 0.39 ms; 6 qubits (42 gates) 16 us, there by
// 0.14-0.2 us an operation (instruction fetch and branches), not by arithmetic.
#include "pass_kernels.hpp"

#include <stdexcept>
#include <string>

#ifndef QSV_PASS_WAVES
#define QSV_PASS_WAVES 4 // waves per SIMD the register allocation leaves room for
#endif

namespace qsv
{
    namespace
    {
        typedef double v2d __attribute__((ext_vector_type(2)));
        typedef float v2f __attribute__((ext_vector_type(2)));

        template <bool NT>
        __device__ __forceinline__ v2d pload(const c128 *p)
        {
            const v2d *q = reinterpret_cast<const v2d *>(p);
            return NT ? __builtin_nontemporal_load(q) : *q;
        }
        template <bool NT>
        __device__ __forceinline__ v2d pload(const c64 *p)
        {
            const v2f *q = reinterpret_cast<const v2f *>(p);
            const v2f f = NT ? __builtin_nontemporal_load(q) : *q;
            return v2d{double(f.x), double(f.y)};
        }
        template <bool NT>
        __device__ __forceinline__ void pstore(c128 *p, v2d v)
        {
            v2d *q = reinterpret_cast<v2d *>(p);
            if (NT)
                __builtin_nontemporal_store(v, q);
            else
                *q = v;
        }
        template <bool NT>
        __device__ __forceinline__ void pstore(c64 *p, v2d v)
        {
            v2f *q = reinterpret_cast<v2f *>(p);
            const v2f f{float(v.x), float(v.y)};
            if (NT)
                __builtin_nontemporal_store(f, q);
            else
                *q = f;
        }

        // rounds and ops through the constant address space: uniform loads become scalar loads
        typedef const __attribute__((address_space(4))) PassRound *RoundPtr;
        typedef const __attribute__((address_space(4))) PassOp *OpPtr;

        struct OpRegs
        {
            uint32_t kind, sel;
            uint64_t cmask, cval;
            double m[4];
            __device__ __forceinline__ void load(OpPtr o)
            {
                kind = o->kind;
                sel = o->sel;
                cmask = o->cmask;
                cval = o->cval;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    m[j] = o->m[j];
            }
            __device__ __forceinline__ void arrived() const
            {
                asm volatile("s_waitcnt lgkmcnt(0)" ::"s"(kind), "s"(sel), "s"(cmask), "s"(cval), "s"(m[0]), "s"(m[1]), "s"(m[2]), "s"(m[3]));
            }
        };

        struct PassTile
        {
            uint8_t tq[16]; // physical qubits of the tile bits, ascending
            int n;
            int nrounds;
        };

        // One operation on a thread's 16 amplitudes (x0, y0) .. (x15, y15), in place.  It is one
        // block of instructions with its own uniform branches because every path has to leave
        // each amplitude in the register it came in: as C++ paths the joins copied and spilled
        // them (199 registers, or 150 spills at 128), as one block the kernel takes 116 and
        // spills none.
        // %[m0] .. %[m7]: the operation's numbers in scalar registers.
#define QSV_T0 "%[t0]"
#define QSV_T1 "%[t1]"
#define QSV_X(i) "%[x" #i "]"
#define QSV_Y(i) "%[y" #i "]"
#define QSV_M(i) "%[m" #i "]"
#define QSV_MUL(d, a, b) "v_mul_f64 " d ", " a ", " b "\n\t"
#define QSV_FMA(d, a, b, c) "v_fma_f64 " d ", " a ", " b ", " c "\n\t"
        // Two pairs at a time (u, v and w, z), interleaved: an instruction then waits for one
        // four before it, which covers the FP64 latency when a SIMD holds a single wave.
        // [[c, -s], [s, c]] as shears
#define QSV_ROT(u, v, w, z)                         \
    QSV_FMA(QSV_X(u), QSV_M(0), QSV_X(v), QSV_X(u)) \
    QSV_FMA(QSV_Y(u), QSV_M(0), QSV_Y(v), QSV_Y(u)) \
    QSV_FMA(QSV_X(w), QSV_M(0), QSV_X(z), QSV_X(w)) \
    QSV_FMA(QSV_Y(w), QSV_M(0), QSV_Y(z), QSV_Y(w)) \
    QSV_FMA(QSV_X(v), QSV_M(1), QSV_X(u), QSV_X(v)) \
    QSV_FMA(QSV_Y(v), QSV_M(1), QSV_Y(u), QSV_Y(v)) \
    QSV_FMA(QSV_X(z), QSV_M(1), QSV_X(w), QSV_X(z)) \
    QSV_FMA(QSV_Y(z), QSV_M(1), QSV_Y(w), QSV_Y(z)) \
    QSV_FMA(QSV_X(u), QSV_M(0), QSV_X(v), QSV_X(u)) \
    QSV_FMA(QSV_Y(u), QSV_M(0), QSV_Y(v), QSV_Y(u)) \
    QSV_FMA(QSV_X(w), QSV_M(0), QSV_X(z), QSV_X(w)) \
    QSV_FMA(QSV_Y(w), QSV_M(0), QSV_Y(z), QSV_Y(w))
#define QSV_TURN_ROT(u, v, w, z)                                                         \
    QSV_TURN_BY(QSV_X(v), QSV_Y(v), QSV_X(z), QSV_Y(z), QSV_M(2), QSV_M(3)) \
    QSV_ROT(u, v, w, z)
        // [[c, -is], [-is, c]]: the rotations of (re u, im v) and (im u, re v)
#define QSV_CROSS(u, v, w, z)                           \
    QSV_FMA(QSV_X(u), QSV_M(0), QSV_Y(v), QSV_X(u))     \
    QSV_FMA(QSV_Y(u), "-" QSV_M(0), QSV_X(v), QSV_Y(u)) \
    QSV_FMA(QSV_X(w), QSV_M(0), QSV_Y(z), QSV_X(w))     \
    QSV_FMA(QSV_Y(w), "-" QSV_M(0), QSV_X(z), QSV_Y(w)) \
    QSV_FMA(QSV_Y(v), "-" QSV_M(1), QSV_X(u), QSV_Y(v)) \
    QSV_FMA(QSV_X(v), QSV_M(1), QSV_Y(u), QSV_X(v))     \
    QSV_FMA(QSV_Y(z), "-" QSV_M(1), QSV_X(w), QSV_Y(z)) \
    QSV_FMA(QSV_X(z), QSV_M(1), QSV_Y(w), QSV_X(z))     \
    QSV_FMA(QSV_X(u), QSV_M(0), QSV_Y(v), QSV_X(u))     \
    QSV_FMA(QSV_Y(u), "-" QSV_M(0), QSV_X(v), QSV_Y(u)) \
    QSV_FMA(QSV_X(w), QSV_M(0), QSV_Y(z), QSV_X(w))     \
    QSV_FMA(QSV_Y(w), "-" QSV_M(0), QSV_X(z), QSV_Y(w))
        // m0 [[1, 1], [1, -1]]
#define QSV_HAD1(u, v)                                  \
    QSV_MUL(QSV_T0, QSV_M(0), QSV_X(v))                 \
    QSV_MUL(QSV_T1, QSV_M(0), QSV_Y(v))                 \
    QSV_FMA(QSV_X(v), QSV_M(0), QSV_X(u), "-" QSV_T0)   \
    QSV_FMA(QSV_Y(v), QSV_M(0), QSV_Y(u), "-" QSV_T1)   \
    QSV_FMA(QSV_X(u), QSV_M(0), QSV_X(u), QSV_T0)       \
    QSV_FMA(QSV_Y(u), QSV_M(0), QSV_Y(u), QSV_T1)
#define QSV_HAD(u, v, w, z) QSV_HAD1(u, v) QSV_HAD1(w, z)
        // exchange
#define QSV_SWAP1(u, v)                               \
    "v_mov_b64 " QSV_T0 ", " QSV_X(u) "\n\t"          \
    "v_mov_b64 " QSV_T1 ", " QSV_Y(u) "\n\t"          \
    "v_mov_b64 " QSV_X(u) ", " QSV_X(v) "\n\t"        \
    "v_mov_b64 " QSV_Y(u) ", " QSV_Y(v) "\n\t"        \
    "v_mov_b64 " QSV_X(v) ", " QSV_T0 "\n\t"          \
    "v_mov_b64 " QSV_Y(v) ", " QSV_T1 "\n\t"
#define QSV_SWAP(u, v, w, z) QSV_SWAP1(u, v) QSV_SWAP1(w, z)
        // (x, y) and (p, q) times (re, im)
#define QSV_TURN_BY(x, y, p, q, re, im)               \
    QSV_MUL(QSV_T0, im, y)                            \
    QSV_MUL(QSV_T1, im, q)                            \
    QSV_MUL(y, re, y)                                 \
    QSV_MUL(q, re, q)                                 \
    QSV_FMA(y, im, x, y)                              \
    QSV_FMA(q, im, p, q)                              \
    QSV_FMA(x, re, x, "-" QSV_T0)                     \
    QSV_FMA(p, re, p, "-" QSV_T1)
#define QSV_TURN1_BY(x, y, re, im)                    \
    QSV_MUL(QSV_T0, im, y)                            \
    QSV_MUL(y, re, y)                                 \
    QSV_FMA(y, im, x, y)                              \
    QSV_FMA(x, re, x, "-" QSV_T0)
#define QSV_ONE(x, y) "v_mov_b64 " x ", 1.0\n\tv_mov_b64 " y ", 0\n\t"
#define QSV_TURN1(i) QSV_TURN1_BY(QSV_X(i), QSV_Y(i), QSV_M(0), QSV_M(1))
#define QSV_TURN(i, j) QSV_TURN_BY(QSV_X(i), QSV_Y(i), QSV_X(j), QSV_Y(j), QSV_M(0), QSV_M(1))
#define QSV_TURN_P(i, j) QSV_TURN_BY(QSV_X(i), QSV_Y(i), QSV_X(j), QSV_Y(j), "%[px]", "%[py]")
#define QSV_TURN_B(i, j) QSV_TURN_BY(QSV_X(i), QSV_Y(i), QSV_X(j), QSV_Y(j), "%[bx]", "%[by]")
        // the 8 pairs of a register bit
#define QSV_PAIRS0(F) F(0, 1, 2, 3) F(4, 5, 6, 7) F(8, 9, 10, 11) F(12, 13, 14, 15)
#define QSV_PAIRS1(F) F(0, 2, 1, 3) F(4, 6, 5, 7) F(8, 10, 9, 11) F(12, 14, 13, 15)
#define QSV_PAIRS2(F) F(0, 4, 1, 5) F(2, 6, 3, 7) F(8, 12, 9, 13) F(10, 14, 11, 15)
#define QSV_PAIRS3(F) F(0, 8, 1, 9) F(2, 10, 3, 11) F(4, 12, 5, 13) F(6, 14, 7, 15)
        // the amplitudes with a register bit set, with two set, all
#define QSV_SET0(F) F(1, 3) F(5, 7) F(9, 11) F(13, 15)
#define QSV_SET1(F) F(2, 3) F(6, 7) F(10, 11) F(14, 15)
#define QSV_SET2(F) F(4, 5) F(6, 7) F(12, 13) F(14, 15)
#define QSV_SET3(F) F(8, 9) F(10, 11) F(12, 13) F(14, 15)
#define QSV_BOTH01(F) F(3, 7) F(11, 15)
#define QSV_BOTH02(F) F(5, 7) F(13, 15)
#define QSV_BOTH03(F) F(9, 11) F(13, 15)
#define QSV_BOTH12(F) F(6, 7) F(14, 15)
#define QSV_BOTH13(F) F(10, 11) F(14, 15)
#define QSV_BOTH23(F) F(12, 13) F(14, 15)
#define QSV_ALL(F) F(0, 1) F(2, 3) F(4, 5) F(6, 7) F(8, 9) F(10, 11) F(12, 13) F(14, 15)
        // a conditional exchange or phase: skipped where the operation's mask of register
        // indices (%[sel], bit = register index of the amplitude or of the pair's first) is clear
#define QSV_SWAP1_IF(u, v)                            \
    "s_bitcmp1_b32 %[sel], " #u "\n\t"                \
    "s_cbranch_scc0 .Lqsv_sw" #u "_" #v "_%=\n\t"     \
    QSV_SWAP1(u, v)                                   \
    ".Lqsv_sw" #u "_" #v "_%=:\n\t"
#define QSV_SWAP_IF(u, v, w, z) QSV_SWAP1_IF(u, v) QSV_SWAP1_IF(w, z)
#define QSV_TURN1_IF(i)                               \
    "s_bitcmp1_b32 %[sel], " #i "\n\t"                \
    "s_cbranch_scc0 .Lqsv_tu" #i "_%=\n\t"            \
    QSV_TURN1(i)                                      \
    ".Lqsv_tu" #i "_%=:\n\t"
#define QSV_TURN_IF(i, j) QSV_TURN1_IF(i) QSV_TURN1_IF(j)
        // Each operation begins a line of instructions: a wave that is alone on its SIMD waits for
        // their fetch, and without this its time changes with the length of the code before (8
        // circuits of 4-6 qubits and 150 layers, the touch above written three ways: 570, 576 and
        // 605 us, on lines 547 and 562).
#define QSV_CASE(n, body)                             \
    ".p2align 6\n.Lqsv_c" #n "_%=:\n\t"               \
    body                                              \
    "s_branch .Lqsv_end_%=\n\t"
#define QSV_CASES(n0, n1, n2, n3, F)                                                      \
    QSV_CASE(n0, QSV_PAIRS0(F)) QSV_CASE(n1, QSV_PAIRS1(F)) QSV_CASE(n2, QSV_PAIRS2(F)) \
    QSV_CASE(n3, QSV_PAIRS3(F))
#define QSV_JUMP(n) "s_branch .Lqsv_c" #n "_%=\n\t"

        struct Amps
        {
            double x[16], y[16];
            double px, py; // pending phase of the thread
            double bx, by; // pending phase of one register bit
        };

        // An operation of kind k on the lanes of `mine`.
        __device__ __forceinline__ void apply_op(Amps &a, uint32_t k, uint32_t sel, uint64_t mine, double m0, double m1, double m2, double m3)
        {
            double t0, t1;
            // jump through a table of branches, one per kind: entry k is 12 + 4 k bytes past the
            // program counter that s_getpc returns
            const uint32_t jump = 4 * k + 12;
            asm("s_mov_b64 s[98:99], exec\n\t"
                "s_and_b64 exec, exec, %[mine]\n\t"
                "s_getpc_b64 s[96:97]\n\t"
                "s_add_u32 s96, s96, %[jump]\n\t"
                "s_addc_u32 s97, s97, 0\n\t"
                "s_setpc_b64 s[96:97]\n\t"
                QSV_JUMP(0) QSV_JUMP(1) QSV_JUMP(2) QSV_JUMP(3) QSV_JUMP(4) QSV_JUMP(5)
                QSV_JUMP(6) QSV_JUMP(7) QSV_JUMP(8) QSV_JUMP(9) QSV_JUMP(10) QSV_JUMP(11)
                QSV_JUMP(12) QSV_JUMP(13) QSV_JUMP(14) QSV_JUMP(15) QSV_JUMP(16) QSV_JUMP(17)
                QSV_JUMP(18) QSV_JUMP(19) QSV_JUMP(20) QSV_JUMP(21) QSV_JUMP(22) QSV_JUMP(23)
                QSV_JUMP(24) QSV_JUMP(25) QSV_JUMP(26) QSV_JUMP(27) QSV_JUMP(28) QSV_JUMP(29)
                QSV_JUMP(30) QSV_JUMP(31) QSV_JUMP(32) QSV_JUMP(33) QSV_JUMP(34) QSV_JUMP(35)
                QSV_JUMP(36) QSV_JUMP(37) QSV_JUMP(38) QSV_JUMP(39) QSV_JUMP(40) QSV_JUMP(41)
                QSV_CASES(0, 1, 2, 3, QSV_TURN_ROT)
                QSV_CASES(4, 5, 6, 7, QSV_ROT)
                QSV_CASES(8, 9, 10, 11, QSV_SWAP)
                QSV_CASE(12, QSV_TURN1_BY("%[px]", "%[py]", QSV_M(0), QSV_M(1)))
                QSV_CASE(13, QSV_TURN1_BY("%[bx]", "%[by]", QSV_M(0), QSV_M(1)))
                QSV_CASE(14, QSV_ALL(QSV_TURN_IF))
                QSV_CASE(15, QSV_ALL(QSV_TURN_P) QSV_ONE("%[px]", "%[py]"))
                QSV_CASE(16, QSV_SET0(QSV_TURN_B) QSV_ONE("%[bx]", "%[by]"))
                QSV_CASE(17, QSV_SET1(QSV_TURN_B) QSV_ONE("%[bx]", "%[by]"))
                QSV_CASE(18, QSV_SET2(QSV_TURN_B) QSV_ONE("%[bx]", "%[by]"))
                QSV_CASE(19, QSV_SET3(QSV_TURN_B) QSV_ONE("%[bx]", "%[by]"))
                QSV_CASE(20, QSV_SET0(QSV_TURN)) QSV_CASE(21, QSV_SET1(QSV_TURN)) QSV_CASE(22, QSV_SET2(QSV_TURN)) QSV_CASE(23, QSV_SET3(QSV_TURN))
                QSV_CASES(24, 25, 26, 27, QSV_CROSS)
                QSV_CASES(28, 29, 30, 31, QSV_HAD)
                QSV_CASES(32, 33, 34, 35, QSV_SWAP_IF)
                QSV_CASE(36, QSV_BOTH01(QSV_TURN)) QSV_CASE(37, QSV_BOTH02(QSV_TURN)) QSV_CASE(38, QSV_BOTH03(QSV_TURN))
                QSV_CASE(39, QSV_BOTH12(QSV_TURN)) QSV_CASE(40, QSV_BOTH13(QSV_TURN)) QSV_CASE(41, QSV_BOTH23(QSV_TURN))
                ".Lqsv_end_%=:\n\t"
                "s_mov_b64 exec, s[98:99]"
                : [x0] "+v"(a.x[0]), [x1] "+v"(a.x[1]), [x2] "+v"(a.x[2]), [x3] "+v"(a.x[3]), [x4] "+v"(a.x[4]), [x5] "+v"(a.x[5]), [x6] "+v"(a.x[6]), [x7] "+v"(a.x[7]),
                  [x8] "+v"(a.x[8]), [x9] "+v"(a.x[9]), [x10] "+v"(a.x[10]), [x11] "+v"(a.x[11]), [x12] "+v"(a.x[12]), [x13] "+v"(a.x[13]), [x14] "+v"(a.x[14]), [x15] "+v"(a.x[15]),
                  [y0] "+v"(a.y[0]), [y1] "+v"(a.y[1]), [y2] "+v"(a.y[2]), [y3] "+v"(a.y[3]), [y4] "+v"(a.y[4]), [y5] "+v"(a.y[5]), [y6] "+v"(a.y[6]), [y7] "+v"(a.y[7]),
                  [y8] "+v"(a.y[8]), [y9] "+v"(a.y[9]), [y10] "+v"(a.y[10]), [y11] "+v"(a.y[11]), [y12] "+v"(a.y[12]), [y13] "+v"(a.y[13]), [y14] "+v"(a.y[14]), [y15] "+v"(a.y[15]),
                  [px] "+v"(a.px), [py] "+v"(a.py), [bx] "+v"(a.bx), [by] "+v"(a.by), [t0] "=&v"(t0), [t1] "=&v"(t1)
                : [m0] "s"(m0), [m1] "s"(m1), [m2] "s"(m2), [m3] "s"(m3), [jump] "s"(jump), [sel] "s"(sel), [mine] "s"(mine)
                : "scc", "s96", "s97", "s98", "s99");
        }

        template <int M>
        __device__ __forceinline__ void pass_sync()
        {
            if (M == 10) // one wave
            {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
            else
            {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            }
        }

        // The amplitude index of tile amplitude 0 of tile `t`: the bits of t at the qubits that
        // are not tile qubits.
        template <int M, class Qubit>
        __device__ __forceinline__ uint64_t tile_base(uint64_t t, Qubit tq)
        {
            for (int b = 0; b < M; ++b)
            {
                const uint64_t lo = t & ((uint64_t(1) << tq(b)) - 1);
                t = lo | ((t ^ lo) << 1);
            }
            return t;
        }

        // A thread's place in the current round's layout.
        struct Place
        {
            uint64_t idx;   // its amplitude index with the register bits 0
            uint64_t ro[4]; // the register bits' index offsets
            __device__ __forceinline__ uint64_t at(int r) const
            {
                uint64_t o = idx;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if ((r >> j) & 1)
                        o |= ro[j];
                return o;
            }
        };

        // The rounds on one tile.  load(i): amplitude i of the state; x: 2^M doubles of LDS.
        template <int M, class Load>
        __device__ __forceinline__ void run_rounds(Amps &a, Place &at_, double *x, uint64_t base, const PassRound *__restrict__ rounds_, int nrounds, const PassOp *__restrict__ ops_, Load load)
        {
            constexpr int TB = M - 4; // thread-index bits
            const RoundPtr rounds = (RoundPtr)rounds_;
            const OpPtr ops = (OpPtr)ops_;
            const uint32_t tid = threadIdx.x;
            uint32_t slot = 0; // the LDS address of the thread's slot, register bits 0
            uint32_t rl[4];    // the register bits' slot offsets
            auto layout = [&](RoundPtr R) {
                at_.idx = base;
                slot = 0;
#pragma unroll
                for (int i = 0; i < TB; ++i)
                {
                    const uint32_t bit = (tid >> i) & 1;
                    at_.idx |= uint64_t(bit) << R->tq[i];
                    slot ^= uint32_t(-int(bit)) & R->tl[i];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    at_.ro[j] = uint64_t(1) << R->rq[j];
                    rl[j] = R->rl[j];
                }
            };
            auto rslot = [&](int r) {
                uint32_t o = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if ((r >> j) & 1)
                        o ^= rl[j];
                return o;
            };
            auto at = [&](uint32_t address) -> double & { return *reinterpret_cast<double *>(reinterpret_cast<char *>(x) + address); };
            uint32_t adr[16]; // LDS addresses of the thread's amplitudes in the current layout
            layout(rounds);
#pragma unroll
            for (int r = 0; r < 16; ++r)
                adr[r] = slot ^ rslot(r);
#pragma unroll
            for (int r = 0; r < 16; ++r)
            {
                const v2d v = load(at_.at(r));
                a.x[r] = v.x;
                a.y[r] = v.y;
            }
            // The program's lines into this XCD's L2 while the tile's loads are in flight: each
            // first touch by a scalar load would cost a memory round trip (13 qubits, one tile of
            // 388 operations: 235 -> 121 us).
            {
                const uint32_t first = rounds[0].first, last = rounds[nrounds - 1].first + rounds[nrounds - 1].count;
                auto touch = [&](const void *p, uint32_t bytes) {
                    uint32_t v = 0;
                    // one step past the end falls on the last word: p need not begin a line
                    for (uint32_t b = tid * 128; b < bytes + 124; b += (128u << TB))
                        v |= *reinterpret_cast<const uint32_t *>(static_cast<const char *>(p) + (b < bytes ? b : bytes - 4));
                    asm volatile("" ::"v"(v));
                };
                touch(ops_ + first, (last - first + 1) * uint32_t(sizeof(PassOp)));
                touch(rounds_, uint32_t(nrounds) * uint32_t(sizeof(PassRound)));
            }
            for (int rd = 0; rd < nrounds; ++rd)
            {
                const RoundPtr R = rounds + rd;
                if (rd > 0)
                {
                    // the tile to the next round's layout
                    pass_sync<M>(); // the last exchange's reads are done
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        at(adr[r]) = a.x[r];
                    layout(R);
                    pass_sync<M>();
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        a.x[r] = at(slot ^ rslot(r));
                    pass_sync<M>();
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        at(adr[r]) = a.y[r];
                    pass_sync<M>();
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                    {
                        adr[r] = slot ^ rslot(r);
                        a.y[r] = at(adr[r]);
                    }
                }
                a.px = a.bx = 1.0;
                a.py = a.by = 0.0;
                const OpPtr first = ops + R->first;
                const uint32_t nops = R->count;
                if (nops == 0) // a layout only
                    continue;
                // the first load and the exchange's LDS reads done here (they share a counter):
                // otherwise the wait for them stands inside the loop, after the next load
                OpRegs cur;
                cur.load(first);
                cur.arrived();
                for (uint32_t i = 0; i < nops; ++i)
                {
                    // the next operation's load is issued before this one's arithmetic
                    OpRegs nxt;
                    nxt.load(first + (i + 1));
                    const uint64_t mine = __builtin_amdgcn_ballot_w64((at_.idx & cur.cmask) == cur.cval);
                    __builtin_amdgcn_sched_barrier(0);
                    apply_op(a, cur.kind, cur.sel, mine, cur.m[0], cur.m[1], cur.m[2], cur.m[3]);
                    __builtin_amdgcn_sched_barrier(0);
                    cur = nxt;
                }
            }
        }

        // GUARD: the state is smaller than the tile; indices past it read as zero and are not
        // written.  One tile per workgroup.
        template <class A, int M, bool NT, bool GUARD>
        __global__ __launch_bounds__(1 << (M - 4), QSV_PASS_WAVES) void k_pass(A *__restrict__ s, PassTile tile, const PassRound *__restrict__ rounds, const PassOp *__restrict__ ops)
        {
            __shared__ double x[1 << M];
            const uint64_t count = uint64_t(1) << tile.n;
            Amps a;
            Place at;
            run_rounds<M>(a, at, x, tile_base<M>(blockIdx.x, [&](int b) { return tile.tq[b]; }), rounds, tile.nrounds, ops,
                          [&](uint64_t i) { return !GUARD || i < count ? pload<NT>(s + i) : v2d{0.0, 0.0}; });
#pragma unroll
            for (int r = 0; r < 16; ++r)
            {
                const uint64_t i = at.at(r);
                if (!GUARD || i < count)
                    pstore<NT>(s + i, v2d{a.x[r], a.y[r]});
            }
        }

        // Sum of the tile's probabilities (out[0]) and, per tile bit b, the sum over the half with
        // the bit 0 less the one with it 1 (out[1 + b]): 4 register bits, 6 lane bits (each
        // step of the wave's butterfly yields its bit's difference), then the waves through LDS.
        // zb: the tile bit of each register bit and thread bit.  qubits > 0: only the differences of
        // that many tile bits, from out[0] on.
        template <int M>
        __device__ __forceinline__ void tile_z(const Amps &a, double *x, const uint8_t *zb, double *out, uint32_t qubits)
        {
            constexpr int W = 1 << (M - 10); // waves
            double v[11];
            double p[16];
#pragma unroll
            for (int r = 0; r < 16; ++r)
                p[r] = __builtin_fma(a.x[r], a.x[r], a.y[r] * a.y[r]);
#pragma unroll
            for (int j = 0; j < 4; ++j)
            { // halve p, keeping the differences of the bit
                double d = 0.0;
#pragma unroll
                for (int r = 0; r < (8 >> j); ++r)
                {
                    const double lo = p[2 * r], hi = p[2 * r + 1];
                    d += lo - hi;
                    p[r] = lo + hi;
                }
                v[1 + j] = d;
            }
            v[0] = p[0];
#pragma unroll
            for (int k = 0; k < 6; ++k)
            {
                const double t = v[0], o = __shfl_xor(t, 1 << k);
                v[0] = t + o;
#pragma unroll
                for (int j = 1; j < 5 + k; ++j)
                    v[j] += __shfl_xor(v[j], 1 << k);
                v[5 + k] = (threadIdx.x >> k) & 1 ? o - t : t - o;
            }
            pass_sync<M>(); // the last exchange's reads are done
            const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
            if (lane == 0)
#pragma unroll
                for (int j = 0; j < 11; ++j)
                    x[11 * wave + j] = v[j];
            pass_sync<M>();
            if (threadIdx.x <= M)
            { // thread 0: the sum; thread 1 + i: register bit i, or thread bit i - 4
                const int j = threadIdx.x;
                double sum = 0.0;
                for (int w = 0; w < W; ++w)
                {
                    const double y = x[11 * w + (j < 11 ? j : 0)];
                    sum += j >= 11 && ((w >> (j - 11)) & 1) ? -y : y;
                }
                const uint32_t b = j == 0 ? 0 : zb[j - 1];
                if (qubits == 0)
                    out[j == 0 ? 0 : 1 + b] = sum;
                else if (j > 0 && b < qubits)
                    out[b] = sum;
            }
        }

        // One tile of one of several circuits per workgroup (PassTask).  Bound by FP64 arithmetic
        // like k_pass: 96 circuits of 10-20 qubits run 8 rounds of up to 4172 tiles, 35 to 400 us
        // each, and the whole circuits of up to 12 qubits beside the first; the batch takes 1.14
        // ms where per-block launches, stage rounds and the LDS kernel took 2.7.
        template <int M, bool NT>
        __global__ __launch_bounds__(1 << (M - 4), QSV_PASS_WAVES) void k_pass_tasks(const PassTask *__restrict__ tasks_, int ntasks, const PassRound *__restrict__ rounds, const PassOp *__restrict__ ops)
        {
            __shared__ double x[1 << M];
            const auto tasks = (const __attribute__((address_space(4))) PassTask *)tasks_;
            int lo = 0, hi = ntasks - 1; // the last task that begins at or before this workgroup
            while (lo < hi)
            {
                const int mid = (lo + hi + 1) >> 1;
                if (tasks[mid].tile_begin <= blockIdx.x)
                    lo = mid;
                else
                    hi = mid - 1;
            }
            const auto &T = tasks[lo];
            const uint32_t t = blockIdx.x - T.tile_begin, flags = T.flags;
            c64 *const s = T.state;
            Amps a;
            Place at;
            run_rounds<M>(a, at, x, tile_base<M>(t, [&](int b) { return (T.tq[b >> 2] >> (8 * (b & 3))) & 255u; }), rounds + T.first_round, int(T.nrounds), ops,
                          [&](uint64_t i) { return flags & kPassZeroState ? v2d{i == 0 ? 1.0 : 0.0, 0.0} : pload<NT>(s + i); });
            if (flags & kPassExpectZ)
                tile_z<M>(a, x, reinterpret_cast<const uint8_t *>(tasks_[lo].zb), T.sums + uint64_t(t) * kPassSums, flags >> kPassQubits);
            else
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    pstore<NT>(s + at.at(r), v2d{a.x[r], a.y[r]});
        }

        // A program from pinned host memory to the device.  A kernel because the copy engine and
        // the passes that follow wait for each other (13 qubits, 228 gates: 220 -> 209 us a call).
        __global__ __launch_bounds__(256) void k_program_copy(uint4 *__restrict__ dst, const uint4 *__restrict__ src, uint64_t count)
        {
            const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
            if (i < count)
                dst[i] = src[i];
        }

        // <Z_q> of a circuit from its tiles' sums: one wave per qubit; lane l adds tiles l,
        // l + 64, ... in order, then a fixed tree.
        __global__ __launch_bounds__(64) void k_pass_z(const PassZ *__restrict__ qubits)
        {
            const PassZ Q = qubits[blockIdx.x];
            double acc = 0.0;
            for (uint32_t t = threadIdx.x; t < Q.ntiles; t += 64)
            {
                const double v = Q.sums[uint64_t(t) * kPassSums + Q.slot];
                acc += (t & Q.sign) ? -v : v;
            }
#pragma unroll
            for (int k = 32; k >= 1; k /= 2)
                acc += __shfl_down(acc, k);
            if (threadIdx.x == 0)
                *Q.out = acc;
        }
    } // namespace

    namespace
    {
        void check_program(const PassRound *rounds, const PassOp *ops)
        {
            if (reinterpret_cast<uintptr_t>(rounds) % alignof(PassRound) || reinterpret_cast<uintptr_t>(ops) % alignof(PassOp))
                throw std::runtime_error("pass: rounds or operations are not aligned");
        }
    } // namespace

    template <class A>
    void launch_pass(hipStream_t st, A *state, int n, int m, const uint8_t *tq, const PassRound *rounds, int nrounds, const PassOp *ops)
    {
        if (n < 1 || n > kMaxQubits || m < kPassMinBits || m > kPassMaxBits)
            throw std::runtime_error("pass: state or tile size out of range");
        if (state == nullptr || rounds == nullptr || ops == nullptr || nrounds < 1)
            throw std::runtime_error("pass: no state or no rounds");
        check_program(rounds, ops);
        PassTile tile{};
        for (int b = 0; b < m; ++b)
        {
            // a state smaller than the tile: tile bit b is index bit b
            if ((n >= m && tq[b] >= n) || (n < m && tq[b] != b) || (b > 0 && tq[b] <= tq[b - 1]))
                throw std::runtime_error("pass: tile qubits must be ascending and inside the state");
            tile.tq[b] = tq[b];
        }
        tile.n = n;
        tile.nrounds = nrounds;
        if (n < m && m != kPassMinBits)
            throw std::runtime_error("pass: only the smallest tile may exceed the state");
        const uint64_t grid = n > m ? uint64_t(1) << (n - m) : 1;
        if (grid > (uint64_t(1) << 30))
            throw std::runtime_error("pass: too many tiles");
        // states within the 256 MB memory-side cache keep cached accesses, as the gate kernels do
        const bool nt = (uint64_t(sizeof(A)) << n) > (uint64_t(256) << 20);
        auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(grid), dim3(1 << (m - 4)), 0, st, state, tile, rounds, ops); };
        if (n < m)
            go(k_pass<A, 10, false, true>);
        else if (m == 10)
            nt ? go(k_pass<A, 10, true, false>) : go(k_pass<A, 10, false, false>);
        else if (m == 11)
            nt ? go(k_pass<A, 11, true, false>) : go(k_pass<A, 11, false, false>);
        else
            nt ? go(k_pass<A, 12, true, false>) : go(k_pass<A, 12, false, false>);
        check(hipGetLastError(), "pass kernel");
    }

    void launch_program_copy(hipStream_t st, void *dst, const void *src, size_t bytes)
    {
        if (dst == nullptr || src == nullptr || bytes == 0 || bytes % 16 || (reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) % 16)
            throw std::runtime_error("pass: program is not in 16-byte units");
        const uint64_t count = bytes / 16;
        hipLaunchKernelGGL(k_program_copy, dim3(unsigned((count + 255) / 256)), dim3(256), 0, st, static_cast<uint4 *>(dst), static_cast<const uint4 *>(src), count);
        check(hipGetLastError(), "pass program copy");
    }

    void launch_pass_tasks(hipStream_t st, int m, bool nt, const PassTask *tasks, int ntasks, uint32_t tiles, const PassRound *rounds, const PassOp *ops)
    {
        if (tasks == nullptr || rounds == nullptr || ops == nullptr || ntasks < 1 || tiles < uint32_t(ntasks))
            throw std::runtime_error("pass: no tasks");
        check_program(rounds, ops);
        auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(tiles), dim3(1 << (m - 4)), 0, st, tasks, ntasks, rounds, ops); };
        if (m == 10)
            nt ? go(k_pass_tasks<10, true>) : go(k_pass_tasks<10, false>);
        else if (m == 11)
            nt ? go(k_pass_tasks<11, true>) : go(k_pass_tasks<11, false>);
        else if (m == 12)
            nt ? go(k_pass_tasks<12, true>) : go(k_pass_tasks<12, false>);
        else
            throw std::runtime_error("pass: tile size out of range");
        check(hipGetLastError(), "pass kernel");
    }

    void launch_pass_z(hipStream_t st, const PassZ *qubits, uint32_t count)
    {
        if (qubits == nullptr || count < 1)
            throw std::runtime_error("pass: no qubits");
        hipLaunchKernelGGL(k_pass_z, dim3(count), dim3(64), 0, st, qubits);
        check(hipGetLastError(), "pass <Z> kernel");
    }

    template void launch_pass<c128>(hipStream_t, c128 *, int, int, const uint8_t *, const PassRound *, int, const PassOp *);
    template void launch_pass<c64>(hipStream_t, c64 *, int, int, const uint8_t *, const PassRound *, int, const PassOp *);
} // namespace qsv
