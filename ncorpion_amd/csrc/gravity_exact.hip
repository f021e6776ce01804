// Brute-force gravity in the reference's FP64 expression tree and order.
//
// Restates vector_field's brute-force and central branches (NcorpiON
// physics.c:63-82, 120-202, 263-266) so that each acceleration is bit-identical.
// In the reference, body k starts from the central term, subtracts
// G*m_p*(X_k-X_p)/D^3 for p < k while k is the outer body, and later receives
// += G*m_q*(X_q-X_k)/D^3 from every q > k as they become the outer body.  For
// body k that is one sequential sum over j ascending, j != k.  A workgroup holds
// four bodies: lanes of three wavefronts form the terms, one j each, and one lane
// per component of the fourth adds them in that order; the p < k terms are
// formed exactly as the reference forms them (X_k - X_p, then subtracted) and
// the q > k terms likewise (X_q - X_k, then added), so signed zeros match too.
// This translation unit is compiled with -ffp-contract=off: no FMA fusion.
#include "ncg_internal.hpp"
#include "exact_div.hpp"
#include "exact_term.hpp"

#pragma clang fp contract(off)

namespace {

// physics.c:186-201 for body k at (X, Y, Z) and body j: D = sqrt(DX*DX +
// DY*DY + DZ*DZ + soft*soft), D3 = D*D*D, term G m_j DX / D3, with DX formed
// as the reference forms it for j < k (X_k - X_j) and j > k (X_j - X_k).
__device__ inline void exact_term(double X, double Y, double Z, double Rk, double xj, double yj,
                                  double zj, double Rj, double gmj, double s, bool lower,
                                  double &tX, double &tY, double &tZ)
{
    const double dx = lower ? X - xj : xj - X;
    const double dy = lower ? Y - yj : yj - Y;
    const double dz = lower ? Z - zj : zj - Z;
    const double soft = s * (lower ? (Rk + Rj) : (Rj + Rk));
    const double D = sqrt(dx * dx + dy * dy + dz * dz + soft * soft);
    const double D3 = D * D * D;
    {
        double q0, q1, q2;
        div3(gmj * dx, gmj * dy, gmj * dz, D3, q0, q1, q2);
        tX = q0;
        tY = q1;
        tZ = q2;
    }
}

// A workgroup takes EXP_B bodies k.  Waves 1..3 form the
// terms of 192 bodies j at a time (one j per lane, EXP_B terms each) into LDS;
// lanes 0 .. 3 EXP_B - 1 of wave 0 add the previous 192 terms, one component
// of one body each, in j order.  A term to subtract is stored negated and a
// skipped one as -0.0, so the sums are runs of additions: a - t and a + (-t)
// are one operation, and a + (-0.0) is a for every a.  Block 0 forms CM_acc
// the same way from the per-body reaction terms (physics.c:141-146 adds them
// body by body), beside the other blocks.
//
// What bounds it: from ~5000 bodies the FP64 issue of the terms (44 instructions
// when the operands are in the window of exact_term.hpp).  Below that neither half
// alone: of 21 us at 2000 bodies the chain of dependent additions (5.7 clocks each)
// takes 5 and the issue of the terms about 9 (85 instructions a wavefront of them);
// a wavefront lives 40,000 clocks (counters), 16,000 of them waiting, with two
// wavefronts a SIMD.  EXP_B = 4 makes the two halves of a chunk about equal (192
// additions ~1100 clocks, 4 terms ~900).
// One wavefront per body, its three summing lanes idle during the terms and
// the other 61 during the sums, took 40 us at 2000 bodies and 2.27 ms at 20,011
// (and CM_acc 13 and 101 us after it); this form takes 21 us and 1.13 ms with
// CM_acc.  One body per lane, the form above 32,768 bodies before, took 25.7 ms
// at 65,536 and 212 ms at 262,144, this one 10.9 and 171.  EXP_B = 2 takes 1.66 ms
// at 20,011 (the summing wavefronts' share), 8 (two workgroups a CU by LDS) 1.17.
constexpr int EXP_B = 4;
constexpr int EXP_ACROSS_MAX = 8192; // bodies
constexpr int EXP_CH = 192;          // bodies j of a chunk
constexpr int EXP_G = 8;             // pairs of terms the summing lanes read ahead
constexpr int EXP_RS = EXP_CH + 2;   // row stride: the summing lanes read different banks

// Body j of a term as read (skip: absent, or past n).
struct ExpJ {
    double x, y, z, m, R;
    int skip;
};

__device__ inline ExpJ exp_load(const DBody *__restrict__ b, int n, const int32_t *__restrict__ ex,
                                int j)
{
    ExpJ r;
    const int jj = min(j, n - 1);
    const DBody &q = b[jj];
    r.x = q.x;
    r.y = q.y;
    r.z = q.z;
    r.m = q.mass;
    r.R = q.radius;
    r.skip = j >= n;
    if (ex) r.skip |= ex[jj] == 0;
    return r;
}

// The window form for EXP_B bodies at once (their chains overlap): for a wavefront
// of j below all of them (negated), above, or ACROSS, with the bodies themselves
// among its j.  False, with nothing written, when an operand is outside the window.  SOFT
// false: s is zero; with finite radii the softening is then zero and adds nothing
// to r2.
enum ExpSide { EXP_BELOW, EXP_ABOVE, EXP_ACROSS };

template <bool SOFT, ExpSide SIDE>
__device__ inline bool exp_window(const ExpJ &q, bool ok, double gm, const double *X,
                                  const double *Y, const double *Z, const double *R, double s,
                                  double (*row)[EXP_RS], int jl, int jk /* j - k0 */)
{
    double t[3][EXP_B], r2[EXP_B];
#pragma unroll
    for (int u = 0; u < EXP_B; ++u) {
        const bool low = SIDE == EXP_BELOW || (SIDE == EXP_ACROSS && jk < u);
        t[0][u] = low ? X[u] - q.x : q.x - X[u];
        t[1][u] = low ? Y[u] - q.y : q.y - Y[u];
        t[2][u] = low ? Z[u] - q.z : q.z - Z[u];
        r2[u] = t[0][u] * t[0][u] + t[1][u] * t[1][u] + t[2][u] * t[2][u];
        if (SOFT) {
            const double soft = s * (R[u] + q.R);
            r2[u] = r2[u] + soft * soft;
        }
        ok = ok && (r2_ok(r2[u]) || (SIDE == EXP_ACROSS && jk == u));
    }
    if (!__all(ok || q.skip)) return false;
    const bool holes = __any(q.skip);
#pragma unroll
    for (int u = 0; u < EXP_B; ++u) {
        double v[3] = {gm * t[0][u], gm * t[1][u], gm * t[2][u]};
        window_quotients<SIDE == EXP_BELOW>(v, r2[u]);
        if (SIDE == EXP_ACROSS)
            for (int d = 0; d < 3; ++d) v[d] = jk < u ? -v[d] : jk == u ? -0.0 : v[d];
        if (holes && q.skip) v[0] = v[1] = v[2] = -0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) row[3 * u + d][jl] = v[d];
    }
    return true;
}

// ACROSS: the one wavefront of terms with the bodies themselves among its j takes the
// window form too (64 bodies: 4.7 us a call, 5.6 with the form with branches; 2000: a
// resident step 2 % less).  With many other wavefronts it gains nothing, and the
// larger loop costs (32,000 bodies: 2.97 ms against 2.94).
template <bool SOFT, bool ACROSS>
__global__ __launch_bounds__(256) void k_grav_exact_p(const DBody *__restrict__ b, int n,
                                                      const int32_t *__restrict__ ex, int cp,
                                                      double cx, double cy, double cz, double mu,
                                                      const double *__restrict__ dcen, double G,
                                                      double s, const double *__restrict__ init,
                                                      double *__restrict__ acc, int cmblk,
                                                      double *__restrict__ cm, NcgKickTail tail)
{
    __shared__ __align__(16) double st[2][3 * EXP_B][EXP_RS];
    if (dcen) {
        cp = dcen[7] != 0.0;
        cx = dcen[0];
        cy = dcen[1];
        cz = dcen[2];
        mu = G * dcen[6];  // physics.c:131
    }
    // Role of the wavefront (0: the summing one).  It turns with the block, so
    // that the summing wavefronts of a CU's blocks are not all on one SIMD.
    const int turn = (int)((blockIdx.x >> 3) + (blockIdx.x >> 8));
    const int w = __builtin_amdgcn_readfirstlane(((threadIdx.x >> 6) + turn) & 3);
    const int lane = threadIdx.x & 63, tid = w * 64 + lane;
    const bool sums = cmblk && blockIdx.x == 0;  // this block forms CM_acc
    const int k0 = ((int)blockIdx.x - cmblk) * EXP_B;
    const int nch = (n + EXP_CH - 1) / EXP_CH;
    if (sums && tail.zero && tid == 0) *tail.zero = 0ull;
    if (sums && !cp) {
        if (tid < 3) cm[tid] = 0.0;
        return;
    }
    if (w > 0) {
        const int jl = tid - 64;
        // The workgroup's bodies k (uniform).
        double X[EXP_B], Y[EXP_B], Z[EXP_B], R[EXP_B];
        bool kok = true;
        if (!sums) {
#pragma unroll
            for (int u = 0; u < EXP_B; ++u) {
                const DBody &q = b[min(k0 + u, n - 1)];
                X[u] = q.x;
                Y[u] = q.y;
                Z[u] = q.z;
                R[u] = q.radius;
                kok = kok && coord_ok(X[u]) && coord_ok(Y[u]) && coord_ok(Z[u]) &&
                      (SOFT || fabs(R[u]) < 1e100);
            }
        }
        // The next chunk's records are in flight during the current terms.
        ExpJ q = exp_load(b, n, ex, jl);
        for (int c = 0; c < nch; ++c) {
            const int j = c * EXP_CH + jl;
            const ExpJ now = q;
            if (c + 1 < nch) q = exp_load(b, n, ex, j + EXP_CH);
            double(*row)[EXP_RS] = st[c & 1];
            const double gm = G * now.m;  // the reference's G*mp (physics.c:192)
            if (sums) {
                double t[3] = {-0.0, -0.0, -0.0};
                if (!now.skip) {
                    // physics.c:121-146
                    const double DX = now.x - cx, DY = now.y - cy, DZ = now.z - cz;
                    const double rk = sqrt(DX * DX + DY * DY + DZ * DZ);
                    const double r3 = rk * rk * rk;
                    t[0] = gm * DX / r3;
                    t[1] = gm * DY / r3;
                    t[2] = gm * DZ / r3;
                }
                for (int d = 0; d < 3; ++d) row[d][jl] = t[d];
            } else {
                const int j0 = c * EXP_CH + (w - 1) * 64;
                // Zeros are looked for only where there is something else (1 % of the
                // kernel at 20,011 bodies).
                bool ok = kok && coord_big(now.x) && coord_big(now.y) && coord_big(now.z) &&
                          gm_big(gm) && (SOFT || fabs(now.R) < 1e100);
                if (!__all(ok || now.skip))
                    ok = kok && coord_ok(now.x) && coord_ok(now.y) && coord_ok(now.z) && gm_ok(gm) &&
                         (SOFT || fabs(now.R) < 1e100);
                bool done = false;
                if (j0 + 63 < k0)
                    done = exp_window<SOFT, EXP_BELOW>(now, ok, gm, X, Y, Z, R, s, row, jl, j - k0);
                else if (j0 >= k0 + EXP_B)
                    done = exp_window<SOFT, EXP_ABOVE>(now, ok, gm, X, Y, Z, R, s, row, jl, j - k0);
                else if (ACROSS)
                    done = exp_window<SOFT, EXP_ACROSS>(now, ok, gm, X, Y, Z, R, s, row, jl, j - k0);
                if (!done) {
#pragma nounroll
                    for (int u = 0; u < EXP_B; ++u) {
                        const int k = k0 + u;
                        const DBody &me = b[min(k, n - 1)];
                        double t[3] = {-0.0, -0.0, -0.0};
                        if (!now.skip && j != k) {
                            exact_term(me.x, me.y, me.z, me.radius, now.x, now.y, now.z, now.R, gm,
                                       s, j < k, t[0], t[1], t[2]);
                            if (j < k)
                                for (int d = 0; d < 3; ++d) t[d] = -t[d];
                        }
                        for (int d = 0; d < 3; ++d) row[3 * u + d][jl] = t[d];
                    }
                }
            }
            __syncthreads();
        }
        __syncthreads();
        return;
    }
    const int u = lane / 3, d = lane - 3 * u;  // body and component of a summing lane
    const int k = k0 + u;
    const bool on = sums ? lane < 3 : u < EXP_B && k < n && (!ex || ex[k] != 0);
    double a = 0.0;
    if (!sums && on) {
        if (init) {
            a = init[3 * (size_t)k + d];
        } else if (cp) {
            // physics.c:121-146
            const DBody me = b[k];
            const double DX = me.x - cx, DY = me.y - cy, DZ = me.z - cz;
            const double rk = sqrt(DX * DX + DY * DY + DZ * DZ);
            const double r3 = rk * rk * rk;
            const double D = d == 0 ? DX : d == 1 ? DY : DZ;
            a = -mu * D / r3;
        }
    }
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
        if (on) {
            const double2 *row = reinterpret_cast<const double2 *>(st[c & 1][sums ? lane : 3 * u + d]);
            // 2 EXP_G terms are read while as many before them are added (all
            // of a chunk: those past n are -0.0).
            double2 x[EXP_G], y[EXP_G];
#pragma unroll
            for (int m = 0; m < EXP_G; ++m) x[m] = row[m];
#pragma unroll
            for (int i = EXP_G; i < EXP_CH / 2; i += 2 * EXP_G) {
#pragma unroll
                for (int m = 0; m < EXP_G; ++m) y[m] = row[i + m];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int m = 0; m < EXP_G; ++m) {
                    a += x[m].x;
                    a += x[m].y;
                }
                __builtin_amdgcn_sched_barrier(0);
                if (i + EXP_G < EXP_CH / 2) {
#pragma unroll
                    for (int m = 0; m < EXP_G; ++m) x[m] = row[i + EXP_G + m];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int m = 0; m < EXP_G; ++m) {
                    a += y[m].x;
                    a += y[m].y;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
    }
    if (!on) return;
    if (sums) {
        cm[lane] = a;
        if (tail.kcen) tail.kcen[3 + lane] += tail.h * a;
    } else {
        acc[3 * (size_t)k + d] = a;
        if (tail.kb) (&tail.kb[k].vx)[d] += tail.h * a;
    }
}

}  // namespace

// The field, and with cm (null: not wanted) CM_acc summed in body order.
static ncg_status exact_launch(ncg_ctx *ctx, const DBody *d_b, int32_t n, const int32_t *d_ex,
                               const ncg_central *c, const double *d_cen, double G, double soft,
                               const double *d_init, double *d_acc, double *d_cm_acc,
                               const NcgKickTail &tail, hipStream_t st)
{
    const int cp = (c && c->present) ? 1 : 0;
    const double cx = cp ? c->x : 0.0, cy = cp ? c->y : 0.0, cz = cp ? c->z : 0.0;
    const double mu = cp ? G * c->mass : 0.0;  // physics.c:131
    const int cmblk = d_cm_acc ? 1 : 0;
    const dim3 grid(cmblk + cdiv(n, EXP_B));
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, d_b, (int)n, d_ex, cp, cx, cy, cz, mu,
                           d_cen, G, soft, d_init, d_acc, cmblk, d_cm_acc, tail);
    };
    if (n <= EXP_ACROSS_MAX) soft != 0.0 ? launch(k_grav_exact_p<true, true>)
                                         : launch(k_grav_exact_p<false, true>);
    else soft != 0.0 ? launch(k_grav_exact_p<true, false>) : launch(k_grav_exact_p<false, false>);
    NCG_CHECK_LAUNCH();
    return NCG_OK;
}

ncg_status ncg_grav_exact_launch(ncg_ctx *ctx, const DBody *d_b, int32_t n, const int32_t *d_ex,
                                 const ncg_central *c, double G, double soft, double *d_acc,
                                 double *d_cm_acc, hipStream_t st, const double *d_init)
{
    return exact_launch(ctx, d_b, n, d_ex, c, nullptr, G, soft, d_init, d_acc, d_cm_acc,
                        NcgKickTail{}, st);
}

// The same with the central body in a device record (8 doubles).
ncg_status ncg_grav_exact_dev(ncg_ctx *ctx, const DBody *d_b, int32_t n, const int32_t *d_ex,
                              const double *d_cen, double G, double soft, double *d_acc,
                              double *d_cm_acc, const NcgKickTail &tail, hipStream_t st)
{
    ProfScope ps(ctx, st, "exact");
    return exact_launch(ctx, d_b, n, d_ex, nullptr, d_cen, G, soft, nullptr, d_acc, d_cm_acc, tail,
                        st);
}
