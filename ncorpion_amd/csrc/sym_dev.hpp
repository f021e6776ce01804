// Frame of the symmetric pair kernels (gravity_sym.hip, adjoint.hip): every
// unordered pair of bodies once, its term added to both bodies.
//
// The bodies are cut into chunks of C (columns) and row groups of W.  A
// workgroup of SY_WAVES wavefronts takes one (row group, chunk) with the
// chunk's records in LDS.  A wavefront holds NI bodies i in scalar registers
// with their sums in its lanes' registers, walks the chunk's blocks of 64
// bodies j (one per lane), and adds the block's terms to the j sums in LDS.
// The wavefronts start at different blocks and step together, so that no two
// meet in a block and the order of every sum is fixed.  A sum over lanes ends
// a row; the j sums of the chunk and the i sums of the row group go to memory
// once each, packed to the triangle that exists, and a last kernel adds them
// in a fixed order.
#pragma once
#include "ncg_internal.hpp"

namespace {

constexpr int SY_WAVES = 8;
constexpr int SY_T = 64 * SY_WAVES;

// Shape for n bodies: nb blocks of 64 bodies j a wavefront takes per step, ni
// bodies i of a wavefront, reps rows of wavefronts per row group.
struct SymShape {
    int n, np;        // bodies, padded to whole chunks
    int C;            // bodies of a chunk
    int chunks, rowg; // columns, row groups
    int W;            // bodies of a row group (at most C, and a divisor of it)
    // Slots of the partial sums: chunk c holds the i sums of slots below its
    // end, row group r the j sums of the slots from its start.
    __host__ __device__ long ioff(int c) const { return (long)C * c * (c + 1) / 2; }
    __host__ __device__ long joff(int r) const { return (long)r * np - (long)W * r * (r - 1) / 2; }
    long islots() const { return ioff(chunks); }
    long jslots() const { return joff(rowg); }
    // Workgroups: per chunk, the row groups that start below its end.
    __host__ __device__ int rows_of(int c) const
    {
        const int r = (c + 1) * (C / W);
        return r < rowg ? r : rowg;
    }
    long workgroups() const
    {
        long g = 0;
        for (int c = 0; c < chunks; ++c) g += rows_of(c);
        return g;
    }
};

inline SymShape sym_shape(int n, int nb, int ni, int reps)
{
    SymShape s;
    s.n = n;
    s.C = SY_T * nb;
    s.chunks = (int)cdiv(n, s.C);
    s.np = s.chunks * s.C;
    s.W = SY_WAVES * ni * reps;
    s.rowg = (int)cdiv(n, s.W);
    return s;
}

// Row group and chunk of workgroup g.
__device__ inline void sym_place(const SymShape &S, int g, int &r, int &c)
{
    c = 0;
    r = g;
    while (r >= S.rows_of(c)) r -= S.rows_of(c++);
}

// Sum of v over the 64 lanes, in every lane.
__device__ inline double lanes_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

template <int CTRL>
__device__ inline double dpp_get64(double v)
{
    union {
        double d;
        int i[2];
    } a, b;
    a.d = v;
    b.i[0] = __builtin_amdgcn_mov_dpp(a.i[0], CTRL, 0xf, 0xf, true);
    b.i[1] = __builtin_amdgcn_mov_dpp(a.i[1], CTRL, 0xf, 0xf, true);
    return b.d;
}

// One halving of 2 N values: lanes with `up` keep the upper N, the others the
// lower N, each added to its partner's.
template <int N, int CTRL>
__device__ inline void halve64(double *a, bool up)
{
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const double keep = up ? a[q + N] : a[q], give = up ? a[q] : a[q + N];
        a[q] = keep + dpp_get64<CTRL>(give);
    }
}

// Sums over the lanes of 4 M values: after it a[0..M) of lane l hold the sums
// of values m + M (bits 3, 2 of l), m < M.  The partners (row mirror, half-row
// mirror) differ in the bit that selects and agree in the bit used before it.
template <int M>
__device__ inline int lanes_sum4(double *a, int lane)
{
    halve64<2 * M, 0x140>(a, (lane & 8) != 0);
    halve64<M, 0x141>(a, (lane & 4) != 0);
#pragma unroll
    for (int m = 0; m < M; ++m) {
        a[m] += dpp_get64<0x1b>(a[m]);  // quad [3, 2, 1, 0]
        a[m] += dpp_get64<0xb1>(a[m]);  // quad [1, 0, 3, 2]
        a[m] += __shfl_xor(a[m], 16);
        a[m] += __shfl_xor(a[m], 32);
    }
    return (lane & 8 ? 2 : 0) + (lane & 4 ? 1 : 0);
}

// Sum of the partials at(k), k = k0, k0 + FQ, ... below k1, four reads in flight.
template <int FQ, class At>
__device__ inline double share_sum(int k0, int k1, At at)
{
    double a = 0.0, b = 0.0;
    int k = k0;
    for (; k + 3 * FQ < k1; k += 4 * FQ) {
        const double x0 = at(k), x1 = at(k + FQ), x2 = at(k + 2 * FQ), x3 = at(k + 3 * FQ);
        a += x0 + x1;
        b += x2 + x3;
    }
    for (; k < k1; k += FQ) a += at(k);
    return a + b;
}

}  // namespace
