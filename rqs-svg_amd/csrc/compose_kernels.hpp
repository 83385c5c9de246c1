// Launch interface of the kernel that composes block matrices (compose_kernels.hip).
#pragma once
#include "sv_kernels.hpp"

namespace qsv
{
    // A gate of a block: targets at block bits tpos[0..t-1] (ascending copy in tmask), controls
    // inside the block as masks of block bits; its 2^t x 2^t matrix (row-major, interleaved
    // doubles, local bit j = target j) is `coef` complex numbers into the launch's coefficients.
    struct alignas(16) ComposeGate
    {
        uint32_t coef;
        uint8_t t, tmask, need1, need0;
        uint8_t tpos[4];
        uint32_t pad;
    };
    // A diagonal of 2^kq entries at `coef`, its bit j the tile index bit bpos[j].
    struct alignas(16) ComposeDiagonal
    {
        uint32_t coef;
        uint8_t bpos[8];
        uint32_t pad;
    };
    enum ComposeKind : uint32_t
    {
        kComposeX3 = 0,    // real form R as bfloat16 high parts, then low parts
        kComposeThree = 1, // Re M, Im M, Re M + Im M in FP32
        kComposeReal = 2,  // real form R in FP32
        kComposeTable = 3, // product of diagonals over 2^kComposeTableBits tile indices from `first` on
    };
    constexpr int kComposeTableBits = 10;
    // One matrix, or a part of one table, written `dst` floats into the launch's buffer: the
    // product of gates (diagonals) first_gate .. first_gate + count - 1 in that order.
    struct alignas(16) ComposeJob
    {
        uint32_t kind, kq, first_gate, count;
        uint32_t dst, first, pad[2];
    };
    // One workgroup per job; everything in device memory.
    void launch_compose(hipStream_t s, float *base, const ComposeJob *jobs, uint32_t njobs, const ComposeGate *gates, const ComposeDiagonal *diagonals, const double *coefs);
} // namespace qsv
