// Composition of block matrices on the device: the gates of a block multiplied together in
// FP64 and written in the form that the block and stage kernels read.
//
// Why here: a flush of 250 gates composes 30 matrices of 32 x 32 complex entries, 10 gates each.
// On one host thread that took 1 to 2 ms with the GPU idle; here each matrix is one workgroup's,
// in LDS, and the 36 of a 30-qubit circuit take 41 us.  Bound by latency: the gates of a block
// follow one another, 512 pairs of entries each and a barrier.  One flush of 4 RY/RZ/CNOT layers
// in BF16x3 products: 14 qubits 374 -> 131 us, 20 qubits 1494 -> 423 us.
//
// The operations and their order are those of the host's composition, with no contraction, so
// that the matrices have the same bits wherever they are composed.
#include "compose_kernels.hpp"

#include <stdexcept>

#pragma clang fp contract(off)

namespace qsv
{
    namespace
    {
        constexpr int kThreads = 256;
        constexpr int kChunkGates = 32, kChunkCoefs = 512; // a gate has at most 4^4 coefficients
        typedef double v2d __attribute__((ext_vector_type(2)));
        typedef float v2f __attribute__((ext_vector_type(2)));

        __device__ __forceinline__ v2d times(v2d a, v2d b) { return v2d{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }

        // float -> bfloat16 bits, round to nearest even (NaN stays NaN)
        __device__ __forceinline__ uint16_t bf16_bits(float f)
        {
            uint32_t u = __float_as_uint(f);
            if ((u & 0x7fffffffu) > 0x7f800000u)
                return uint16_t((u >> 16) | 0x40u);
            u += 0x7fffu + ((u >> 16) & 1u);
            return uint16_t(u >> 16);
        }
        __device__ __forceinline__ float bf16_value(uint16_t b) { return __uint_as_float(uint32_t(b) << 16); }

        // M <- G M on a 2^kq x 2^kq matrix in LDS: every column's groups of 2^t entries that
        // differ in the targets, one group a thread at a time.
        template <int T>
        __device__ __forceinline__ void apply_gate(v2d *M, int kq, const ComposeGate &g, const v2d *U)
        {
            const int K = 1 << kq, groups = K >> g.t;
            for (int i = threadIdx.x; i < groups * K; i += kThreads)
            {
                const int c = i & (K - 1);
                int x = i >> kq;
                for (int b = 0; b < kq; ++b)
                    if ((g.tmask >> b) & 1)
                    {
                        const int lo = x & ((1 << b) - 1);
                        x = lo | ((x ^ lo) << 1);
                    }
                if ((x & g.need1) != g.need1 || (x & g.need0))
                    continue;
                int at[T];
                v2d in[T];
#pragma unroll
                for (int r = 0; r < T; ++r)
                {
                    int y = x;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if ((1 << j) < T && ((r >> j) & 1))
                            y |= 1 << g.tpos[j];
                    at[r] = (y << kq) + c;
                    in[r] = M[at[r]];
                }
#pragma unroll
                for (int r = 0; r < T; ++r)
                {
                    v2d acc{0.0, 0.0};
#pragma unroll
                    for (int k = 0; k < T; ++k)
                        acc += times(U[r * T + k], in[k]);
                    M[at[r]] = acc;
                }
            }
        }

        __global__ __launch_bounds__(kThreads) void k_compose(float *__restrict__ base, const ComposeJob *__restrict__ jobs, const ComposeGate *__restrict__ gates, const ComposeDiagonal *__restrict__ diagonals, const v2d *__restrict__ coefs)
        {
            __shared__ v2d M[32 * 32], u[kChunkCoefs];
            __shared__ ComposeGate chunk[kChunkGates];
            const ComposeJob J = jobs[blockIdx.x];
            const int kq = int(J.kq), K = 1 << kq;
            if (J.kind == kComposeTable)
            {
                v2f *out = reinterpret_cast<v2f *>(base + J.dst);
                for (uint32_t i = J.first + threadIdx.x; i < J.first + (1u << kComposeTableBits); i += kThreads)
                {
                    v2d v{1.0, 0.0};
                    for (uint32_t d = 0; d < J.count; ++d)
                    {
                        const ComposeDiagonal &D = diagonals[J.first_gate + d];
                        uint32_t e = 0;
                        for (int j = 0; j < kq; ++j)
                            e |= ((i >> D.bpos[j]) & 1u) << j;
                        v = times(v, coefs[D.coef + e]);
                    }
                    out[i] = v2f{float(v.x), float(v.y)};
                }
                return;
            }
            for (int i = threadIdx.x; i < K * K; i += kThreads)
                M[i] = v2d{(i >> kq) == (i & (K - 1)) ? 1.0 : 0.0, 0.0};
            // gates and their coefficients (contiguous) come to LDS a chunk at a time
            for (uint32_t k = 0; k < J.count;)
            {
                const int n = int(J.count - k) < kChunkGates ? int(J.count - k) : kChunkGates;
                __syncthreads();
                if (int(threadIdx.x) < n)
                    chunk[threadIdx.x] = gates[J.first_gate + k + threadIdx.x];
                __syncthreads();
                const uint32_t from = chunk[0].coef;
                int m = 0, count = 0;
                while (m < n && int(chunk[m].coef - from) + (1 << (2 * chunk[m].t)) <= kChunkCoefs)
                {
                    count = int(chunk[m].coef - from) + (1 << (2 * chunk[m].t));
                    ++m;
                }
                for (int i = threadIdx.x; i < count; i += kThreads)
                    u[i] = coefs[from + i];
                for (int i = 0; i < m; ++i)
                {
                    __syncthreads();
                    const ComposeGate g = chunk[i];
                    const v2d *U = u + (g.coef - from);
                    switch (g.t)
                    {
                    case 0:
                        apply_gate<1>(M, kq, g, U);
                        break;
                    case 1:
                        apply_gate<2>(M, kq, g, U);
                        break;
                    case 2:
                        apply_gate<4>(M, kq, g, U);
                        break;
                    case 3:
                        apply_gate<8>(M, kq, g, U);
                        break;
                    default:
                        apply_gate<16>(M, kq, g, U);
                    }
                }
                k += uint32_t(m);
            }
            __syncthreads();
            const int D = 2 * K, per = D * D;
            if (J.kind == kComposeThree)
            {
                float *out = base + J.dst;
                for (int i = threadIdx.x; i < K * K; i += kThreads)
                {
                    const v2d z = M[i];
                    out[i] = float(z.x);
                    out[K * K + i] = float(z.y);
                    out[2 * K * K + i] = float(z.x + z.y);
                }
                return;
            }
            uint16_t *half = reinterpret_cast<uint16_t *>(base + J.dst);
            for (int i = threadIdx.x; i < per; i += kThreads)
            {
                const int r = i >> (kq + 1), c = i & (D - 1);
                const v2d z = M[((r >> 1) << kq) + (c >> 1)];
                const double v = (r & 1) == (c & 1) ? z.x : (r & 1) ? z.y : -z.y;
                if (J.kind == kComposeReal)
                    base[J.dst + i] = float(v);
                else
                {
                    const uint16_t hi = bf16_bits(float(v));
                    half[i] = hi;
                    half[per + i] = bf16_bits(float(v - double(bf16_value(hi))));
                }
            }
        }
    } // namespace

    void launch_compose(hipStream_t s, float *base, const ComposeJob *jobs, uint32_t njobs, const ComposeGate *gates, const ComposeDiagonal *diagonals, const double *coefs)
    {
        if (base == nullptr || jobs == nullptr || gates == nullptr || diagonals == nullptr || coefs == nullptr || njobs < 1)
            throw std::runtime_error("compose: no jobs");
        hipLaunchKernelGGL(k_compose, dim3(njobs), dim3(kThreads), 0, s, base, jobs, gates, diagonals, reinterpret_cast<const v2d *>(coefs));
        check(hipGetLastError(), "compose kernel");
    }
} // namespace qsv
