// FP64-fast all-pairs gravity, every unordered pair once.
//
// The same field as the split kernel of gravity_tiled.hip (k_pairs), in body
// order (existing bodies first): a_i += G m_j d / D^3, a_j -= G m_i d / D^3
// with one separation, one 1/D and one D^-3 for both.  A pair is 22 FP64
// instructions (20 without softening) and one v_rsq_f64 (17 clocks a wavefront,
// as much as 3.5 others), where the split kernel takes 18 (16) and one v_rsq_f64
// for each of the two: 123 against 206 clocks of issue, of which 165 are reached
// (the rest: barriers, the j sums in LDS, the sums over lanes).  50,021 bodies:
// 1.87 ms a call with the split kernel, 1.35 here; 100,003: 6.12 and 4.8; 16,384:
// 0.32 and 0.19.  Eight bodies i a wavefront spilled or left two wavefronts a
// SIMD (2.0 ms at 50,021); their records read from LDS bound it by LDS (1.44).
#include <algorithm>

#include "ncg_internal.hpp"
#include "sym_dev.hpp"
#include "tiled_dev.hpp"

namespace {

constexpr int GI = 4;          // bodies i of a wavefront
constexpr int GROW = SY_WAVES * GI;
constexpr int SY_NB = 2;       // blocks of 64 bodies j a wavefront takes per step
constexpr int SY_C = SY_T * SY_NB;

// One block: lane's body j against the wavefront's GI bodies i.  DIAG: only
// pairs with j above i (slots); the others' masses are zeroed (1/D of a body
// against itself is finite, TINY2).
template <bool SOFT, bool DIAG>
__device__ inline void sym_block(const double4 *ri, const double *rs, int i0, int j, double xj,
                                 double yj, double zj, double mj, double sj, double (*acc)[GI],
                                 double &bx, double &by, double &bz)
{
#pragma unroll
    for (int u = 0; u < GI; ++u) {
        const double4 p = ri[u];
        const double dx = xj - p.x, dy = yj - p.y, dz = zj - p.z;
        double seed = TINY2;
        if (SOFT) {
            const double e = sj + rs[u];
            seed = fma(e, e, TINY2);
        }
        const double r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, seed)));
        double y = __builtin_amdgcn_rsq(r2);
        y = y * fma(-0.5 * r2, y * y, 1.5);
        const double y3 = y * (y * y);
        double a = mj, b = p.w;
        if (DIAG && j <= i0 + u) a = b = 0.0;
        a *= y3;
        b *= y3;
        acc[0][u] = fma(a, dx, acc[0][u]);
        acc[1][u] = fma(a, dy, acc[1][u]);
        acc[2][u] = fma(a, dz, acc[2][u]);
        bx = fma(-b, dx, bx);
        by = fma(-b, dy, by);
        bz = fma(-b, dz, bz);
    }
}

template <bool SOFT>
__global__ __launch_bounds__(SY_T, 4) void k_pairs_sym(const double4 *__restrict__ jd,
                                                       const double *__restrict__ jsig,
                                                       const int *__restrict__ nvalid, SymShape S,
                                                       double *__restrict__ pi,
                                                       double *__restrict__ pj)
{
    __shared__ double4 rec[SY_C];
    __shared__ double sig[SOFT ? SY_C : 1];
    __shared__ double js[3][SY_C];
    // This workgroup's chunk and row group.
    int r, c;
    sym_place(S, blockIdx.x, r, c);
    const int nv = nvalid ? *nvalid : S.n;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j0 = c * SY_C;
    const int row0 = r * S.W;
    if (j0 >= nv || row0 >= nv) return;
#pragma unroll
    for (int h = 0; h < SY_NB; ++h) {
        const int k = h * SY_T + tid, j = min(j0 + k, nv - 1);
        double4 q = jd[j];
        if (j0 + k >= nv) q.w = 0.0;
        rec[k] = q;
        if (SOFT) sig[k] = jsig[j];
        js[0][k] = js[1][k] = js[2][k] = 0.0;
    }
    __syncthreads();
    for (int row = row0; row < row0 + S.W; row += GROW) {
        if (row >= nv || row >= j0 + SY_C) break;
        // The wavefront's bodies i (uniform addresses: scalar loads).
        const int i0 = row + w * GI;
        double4 ri[GI];
        double rs[GI];
#pragma unroll
        for (int u = 0; u < GI; ++u) {
            const int i = min(i0 + u, nv - 1);
            ri[u] = jd[i];
            if (i0 + u >= nv) ri[u].w = 0.0;
            rs[u] = SOFT ? jsig[i] : 0.0;
        }
        double acc[3][GI];
#pragma unroll
        for (int u = 0; u < GI; ++u) acc[0][u] = acc[1][u] = acc[2][u] = 0.0;
        for (int s = 0; s < SY_WAVES; ++s) {
#pragma unroll
            for (int h = 0; h < SY_NB; ++h) {
                const int kb = (((w + s) & (SY_WAVES - 1)) * SY_NB + h) * 64;  // in the chunk
                const int k = kb + lane, jb = j0 + kb;
                // Blocks wholly at or below the wavefront's first body have no
                // pair.
                if (jb + 63 <= i0) continue;
                const double4 q = rec[k];
                const double sj = SOFT ? sig[k] : 0.0;
                double bx = js[0][k], by = js[1][k], bz = js[2][k];
                if (jb >= i0 + GI)
                    sym_block<SOFT, false>(ri, rs, i0, jb + lane,
                                           q.x, q.y, q.z, q.w, sj, acc, bx, by, bz);
                else
                    sym_block<SOFT, true>(ri, rs, i0, jb + lane,
                                          q.x, q.y, q.z, q.w, sj, acc, bx, by, bz);
                js[0][k] = bx;
                js[1][k] = by;
                js[2][k] = bz;
            }
            __syncthreads();
        }
        // Value 3 u + d, so that a lane ends with the three sums of one body.
        double v[3 * GI];
#pragma unroll
        for (int u = 0; u < GI; ++u)
            for (int d = 0; d < 3; ++d) v[3 * u + d] = acc[d][u];
        const int u = lanes_sum4<3>(v, lane);
        if ((lane & ~12) == 0 && i0 + u < nv) {
            double *o = pi + 3 * (S.ioff(c) + i0 + u);
            o[0] = v[0];
            o[1] = v[1];
            o[2] = v[2];
        }
    }
    double *o = pj + 3 * (S.joff(r) + (j0 - row0));
#pragma unroll
    for (int h = 0; h < SY_NB; ++h) {
        const int k = h * SY_T + tid;
        if (j0 + k >= row0)
            for (int d = 0; d < 3; ++d) o[3 * (long)k + d] = js[d][k];
    }
}

// Sums of a slot over chunks and row groups in a fixed order, the central term,
// and the block's share of CM_acc.  FS slots a workgroup: phase 1 adds their
// components in FQ interleaved shares (coalesced reads, four in flight), phase
// 2 one slot per lane.  Bound by the reads' latency: 64 slots and 4 shares a
// workgroup took 62 us at 16,384 bodies, this 11.
constexpr int FT = 256, FS = 16, FQ = 16;

__global__ __launch_bounds__(FT) void k_sym_finish(const DBody *__restrict__ b,
                                                   const int *__restrict__ perm,
                                                   const int *__restrict__ nvalid, SymShape S,
                                                   const double *__restrict__ pi,
                                                   const double *__restrict__ pj, int cp, double cx,
                                                   double cy, double cz, double mu,
                                                   const double *__restrict__ dcen, double G,
                                                   double *__restrict__ acc,
                                                   double *__restrict__ cmpart)
{
    __shared__ double sh[FQ][3 * FS];
    const int nv = nvalid ? *nvalid : S.n;
    const int s0 = blockIdx.x * FS, tid = threadIdx.x;
    for (int item = tid; item < FQ * 3 * FS; item += FT) {
        const int q = item / (3 * FS), e = item % (3 * FS);
        const int s = s0 + e / 3;
        double a = 0.0;
        if (s < nv) {
            const int c1 = (nv + SY_C - 1) / SY_C, r1 = s / S.W + 1;
            a = share_sum<FQ>(s / SY_C + q, c1, [&](int c) { return pi[3 * (S.ioff(c) + s0) + e]; });
            a += share_sum<FQ>(q, r1,
                           [&](int r) { return pj[3 * (S.joff(r) + s0 - (long)r * S.W) + e]; });
        }
        sh[q][e] = a;
    }
    __syncthreads();
    if (tid >= 64) return;
    double ct[3] = {0.0, 0.0, 0.0};
    const int s = s0 + tid;
    if (dcen) {  // central body state {x, y, z, vx, vy, vz, M, present} on the device
        cx = dcen[0];
        cy = dcen[1];
        cz = dcen[2];
        mu = G * dcen[6];
        cp = dcen[7] != 0.0;
    }
    if (tid < FS && s < nv) {
        const int k = perm ? perm[s] : s;
        double a[3];
        for (int d = 0; d < 3; ++d) {
            const int e = 3 * tid + d;
            a[d] = 0.0;
            for (int q = 0; q < FQ; ++q) a[d] += sh[q][e];
        }
        if (cp) {
            const DBody q = b[k];
            const double DX = q.x - cx, DY = q.y - cy, DZ = q.z - cz;
            const double rk = sqrt(DX * DX + DY * DY + DZ * DZ);
            const double r3 = rk * rk * rk;
            a[0] += -mu * DX / r3;
            a[1] += -mu * DY / r3;
            a[2] += -mu * DZ / r3;
            ct[0] = G * q.mass * DX / r3;
            ct[1] = G * q.mass * DY / r3;
            ct[2] = G * q.mass * DZ / r3;
        }
        for (int d = 0; d < 3; ++d) acc[3 * (size_t)k + d] = a[d];
    }
    if (!cmpart) return;
    for (int d = 0; d < 3; ++d) {
        const double t = lanes_sum(ct[d]);
        if (tid == 0) cmpart[3 * (size_t)blockIdx.x + d] = t;
    }
}

// Records {x, y, z, G m} and s R in slot order.
__global__ __launch_bounds__(FT) void k_sym_records(const DBody *__restrict__ b, int n,
                                                    const int *__restrict__ perm,
                                                    const int *__restrict__ nvalid, double G,
                                                    double soft, double4 *__restrict__ jd,
                                                    double *__restrict__ jsig)
{
    const int s = blockIdx.x * FT + threadIdx.x;
    if (s >= (nvalid ? *nvalid : n)) return;
    const DBody q = b[perm ? perm[s] : s];
    jd[s] = make_double4(q.x, q.y, q.z, G * q.mass);
    jsig[s] = soft * q.radius;
}

// CM_acc from the partials of k_sym_finish.
__global__ __launch_bounds__(FT) void k_sym_cm(const double *__restrict__ part, int np,
                                               double *__restrict__ out)
{
    __shared__ double sh[FT / 64][3];
    double a[3] = {0.0, 0.0, 0.0};
    for (int q = threadIdx.x; q < np; q += FT)
        for (int d = 0; d < 3; ++d) a[d] += part[3 * (size_t)q + d];
    for (int d = 0; d < 3; ++d) {
        const double t = lanes_sum(a[d]);
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6][d] = t;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int d = threadIdx.x;
        out[d] = (sh[0][d] + sh[1][d]) + (sh[2][d] + sh[3][d]);
    }
}

}  // namespace

// Rows of 32 bodies per row group: few enough for workgroups to fill the chip
// some rounds (512 at a time; n = 16,384: 2176), and as many as keep the j sums a
// small share of the traffic (per call at 16,384 bodies 0.199, 0.192, 0.199 ms
// with 1, 2, 4; at 50,021 1.66, 1.46, 1.35).
static int sym_reps(int32_t n) { return n <= 20000 ? 2 : n <= 65536 ? 4 : n <= 131072 ? 8 : 16; }

ncg_status ncg_gravity_sym(ncg_ctx *ctx, const DBody *d_b, int32_t n, const int *d_perm,
                           const int *d_nvalid, const ncg_central *c, const double *d_central,
                           double G, double soft, double *d_acc, double *d_cm_acc, hipStream_t st)
{
    const SymShape S = sym_shape(n, SY_NB, GI, sym_reps(n));
    double4 *jd = dbuf<double4>(ctx, "y_jd", n);
    double *jsig = dbuf<double>(ctx, "y_jsig", n);
    double *pi = dbuf<double>(ctx, "y_pi", 3 * (size_t)S.islots());
    double *pj = dbuf<double>(ctx, "y_pj", 3 * (size_t)S.jslots());
    const int nb = (int)cdiv(n, FS);
    double *cmpart = d_cm_acc ? dbuf<double>(ctx, "y_cm", 3 * (size_t)nb) : nullptr;
    if (!jd || !jsig || !pi || !pj || (d_cm_acc && !cmpart)) return NCG_ERR_NOMEM;
    hipLaunchKernelGGL(k_sym_records, dim3(cdiv(n, FT)), dim3(FT), 0, st, d_b, (int)n, d_perm,
                       d_nvalid, G, soft, jd, jsig);
    NCG_CHECK_LAUNCH();
    const long wgs = S.workgroups();
    {
        ProfScope ps(ctx, st, "pairs_fast64");
        if (soft != 0.0)
            hipLaunchKernelGGL(k_pairs_sym<true>, dim3((unsigned)wgs), dim3(SY_T), 0, st, jd, jsig,
                               d_nvalid, S, pi, pj);
        else
            hipLaunchKernelGGL(k_pairs_sym<false>, dim3((unsigned)wgs), dim3(SY_T), 0, st, jd, jsig,
                               d_nvalid, S, pi, pj);
        NCG_CHECK_LAUNCH();
    }
    const int cp = (c && c->present) ? 1 : 0;
    hipLaunchKernelGGL(k_sym_finish, dim3(nb), dim3(FT), 0, st, d_b, d_perm, d_nvalid, S, pi, pj, cp,
                       cp ? c->x : 0.0, cp ? c->y : 0.0, cp ? c->z : 0.0, cp ? G * c->mass : 0.0,
                       d_central, G, d_acc, cmpart);
    if (d_cm_acc)
        hipLaunchKernelGGL(k_sym_cm, dim3(1), dim3(FT), 0, st, cmpart, nb, d_cm_acc);
    NCG_CHECK_LAUNCH();
    return NCG_OK;
}
