// FP64-fast all-pairs gravity, every unordered pair once.
//
// The same field as the split kernel of gravity_tiled.hip (k_pairs), in body
// order (existing bodies first): a_i += G m_j d / D^3, a_j -= G m_i d / D^3
// with one separation, one 1/D and one D^-3 for both.  A pair is 22 FP64
// instructions (20 without softening) and one v_rsq_f64 (17 clocks a wavefront,
// as much as 3.5 others), where the split kernel takes 18 (16) and one v_rsq_f64
// for each of the two: 123 against 206 clocks of issue a wavefront of pairs, which
// takes 154 (counters at 50,021 bodies; the rest: 29 instructions issued in all,
// barriers, the j sums in LDS, the sums over lanes).  50,021 bodies: 1.76 ms a call
// with the split kernel, 1.30 here; 100,003: 6.4 and 5.0; 16,384: 0.28 and 0.17.
// Eight bodies i a wavefront spilled or left two wavefronts a SIMD (2.0 ms at
// 50,021); their records read from LDS bound it by LDS (1.44).
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
                                                   const double *__restrict__ near, int nnear,
                                                   const int *__restrict__ far,
                                                   const Scal *__restrict__ scal,
                                                   double *__restrict__ acc,
                                                   double *__restrict__ cmpart)
{
    __shared__ double sh[FQ][3 * FS];
    const int nv = nvalid ? *nvalid : S.n;
    const int s0 = blockIdx.x * FS, tid = threadIdx.x;
    const bool pairs = !far || *far;  // the pair kernel wrote sums
    for (int item = tid; item < FQ * 3 * FS; item += FT) {
        const int q = item / (3 * FS), e = item % (3 * FS);
        const int s = s0 + e / 3;
        double a = 0.0;
        if (s < nv) {
            const int c1 = (nv + SY_C - 1) / SY_C, r1 = s / S.W + 1;
            if (pairs) {
                a = share_sum<FQ>(s / SY_C + q, c1,
                                  [&](int c) { return pi[3 * (S.ioff(c) + s0) + e]; });
                a += share_sum<FQ>(q, r1, [&](int r) {
                    return pj[3 * (S.joff(r) + s0 - (long)r * S.W) + e];
                });
            }
            // The mixed form's near terms.
            if (q < nnear) a += near[3 * ((size_t)q * S.n + s0) + e];
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
        if (scal) {  // the mixed form's powers of two
            const int ex = mass_exp(*scal, G) - 2 * scal->lexp;
            for (int d = 0; d < 3; ++d) a[d] = ldexp(a[d], ex);
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

// ---- mixed form ---------------------------------------------------------------
// The bodies are in Hilbert order, cut into groups of 64.  For two groups a
// decision from their boxes (near_pair, one bit, the same for both orders)
// picks the form of their pairs:
//   near: FP64, ordered, by k_mix_near;
//   far:  FP32, unordered, by k_pairs_mix: separations d = W_j - v_i of positions
//         taken from the box centre of i's group in FP64 and rounded once; 16
//         instructions and a v_rsq_f32 a pair, where the scaled far term of the
//         split kernel takes 11 and one for each of the two: 51 against 76
//         clocks of issue a wavefront of pairs, which takes 67 at 262,144 bodies
//         and 72 at 100,003 (counters; the rest: 19.5 instructions issued in all, j
//         records and sums in LDS, barriers).  Operands are vector registers (a
//         scalar one takes the issue from 2.6 to 4.4 clocks).
// A lane's FP32 sums are 16 terms of a body j, or 16 of a body i, and i's over 8
// lanes; all after that are FP64.  Positions and G m are scaled by powers of two
// (the box's edge and the largest G m about 1), so that no system of units over-
// or underflows FP32 (the FP64 terms are unchanged by it, but for results at the
// ends of its range).
// Calls of 262,144 bodies: 19.4 ms with the split kernel, 16.1 here; 100,003:
// 3.17 and 2.66; 32,800: 0.49 and 0.42; the field's error against FP64 is that
// of the split kernel or less (norm 2.3e-9 and 2.0e-9, 1.5e-9 and 1.5e-9, 1.6e-9
// and 1.1e-9).
// Eight bodies i a wavefront: 21.2 ms at 262,144 (the j records and sums come
// twice as often); sums over all lanes in FP32: error +10 %.
constexpr int MI = 16;            // bodies i of a wavefront
constexpr int MG = 64;            // bodies of a group: half a row of wavefronts
constexpr int MNEAR = 16;         // partial sums of a body's near terms
constexpr int NW = 4;             // wavefronts that form one
static_assert(MNEAR <= FQ && MNEAR * NW == 64, "one share of k_sym_finish, one bit of a word each");
constexpr int MROW = SY_WAVES * MI;
static_assert(MROW == 2 * MG, "a row of wavefronts is two groups");

__global__ __launch_bounds__(64) void k_mix_records(const DBody *__restrict__ b,
                                                    const int *__restrict__ perm,
                                                    const Scal *__restrict__ scal, double G,
                                                    double soft, double4 *__restrict__ jd,
                                                    double *__restrict__ jsig,
                                                    TileHdr *__restrict__ hdr, int *__restrict__ far)
{
    const Scal S = *scal;
    const int g = blockIdx.x, lane = threadIdx.x, s = g * MG + lane;
    if (g == 0 && lane == 0) *far = 0;
    if (g * MG >= S.nvalid) return;
    const DBody q = b[perm[min(s, S.nvalid - 1)]];
    const double gm = G * q.mass;
    const double p[3] = {ldexp(q.x, -S.lexp), ldexp(q.y, -S.lexp), ldexp(q.z, -S.lexp)};
    const double sg = ldexp(gm, -mass_exp(S, G));
    // Slots past the last body repeat it without mass.
    jd[s] = make_double4(p[0], p[1], p[2], s < S.nvalid ? sg : 0.0);
    jsig[s] = ldexp(soft * q.radius, -S.lexp);
    // Negative, not finite, or a term of it could leave FP32's normal range
    // (near_pair bounds the distances).
    const bool bad = __any(!(sg == 0.0 || (sg >= 0x1p-96 && sg <= 2.0)));
    double A[3];
    float H[3];
    for (int c = 0; c < 3; ++c) {
        double lo = p[c], hi = p[c];
        for (int o = 32; o > 0; o >>= 1) {
            lo = fmin(lo, __shfl_xor(lo, o));
            hi = fmax(hi, __shfl_xor(hi, o));
        }
        A[c] = 0.5 * (lo + hi);
        const double h = fmax(hi - A[c], A[c] - lo);
        H[c] = (float)h;
        if ((double)H[c] < h) H[c] = nextafterf(H[c], 3.0e38f);
    }
    if (lane == 0) {
        TileHdr th;
        th.ax = A[0];
        th.ay = A[1];
        th.az = A[2];
        th.hx = H[0];
        th.hy = H[1];
        th.hz = H[2];
        th.count = 0;
        th.smax = bad ? INFINITY : 0.f;
        th.smin = 0.f;
        hdr[g] = th;
    }
}

// Near unless the box distance is at least theta times (anchor distance + half
// extents), beyond FP32 resolution of the largest softening length, and the
// distances are in the range that FP32 terms are safe in (scaled units; bodies
// may have left the box that set the scale); a group with an unfit G m (smax
// set) is near to all, as is any whose box is NaN.
__device__ inline bool near_pair(const TileHdr &a, const TileHdr &b, double theta, double eps2x)
{
    const double Cx = fabs(a.ax - b.ax), Cy = fabs(a.ay - b.ay), Cz = fabs(a.az - b.az);
    const double gx = fmax(0.0, Cx - ((double)a.hx + b.hx));
    const double gy = fmax(0.0, Cy - ((double)a.hy + b.hy));
    const double gz = fmax(0.0, Cz - ((double)a.hz + b.hz));
    const double dmin2 = gx * gx + gy * gy + gz * gz;
    const double ha = sqrt((double)a.hx * a.hx + (double)a.hy * a.hy + (double)a.hz * a.hz);
    const double hb = sqrt((double)b.hx * b.hx + (double)b.hy * b.hy + (double)b.hz * b.hz);
    const double size = sqrt(Cx * Cx + Cy * Cy + Cz * Cz) + (ha + hb);
    const bool far = dmin2 >= theta * theta * size * size && dmin2 > eps2x && dmin2 >= 0x1p-50 &&
                     size <= 0x1p4 && a.smax == 0.f && b.smax == 0.f;
    return !far;
}

// Bit h of group g's row: g and h are far; *any: some two groups are.
__global__ __launch_bounds__(64) void k_mix_mask(const TileHdr *__restrict__ hdr,
                                                 const Scal *__restrict__ scal, int nw, double theta,
                                                 double soft, unsigned long long *__restrict__ mask,
                                                 int *__restrict__ any)
{
    const int ng = (scal->nvalid + MG - 1) / MG;
    const int g = blockIdx.x, h = blockIdx.y * 64 + (int)threadIdx.x;
    bool far = false;
    if (g < ng && h < ng) {
        // In this order for both bits of the pair, which must be one.
        const TileHdr a = hdr[min(g, h)], b = hdr[max(g, h)];
        const double eps = ldexp(2.0 * soft * scal->rmax, -scal->lexp);
        far = !near_pair(a, b, theta, eps * eps * 67108864.0 /* 2^26 */);
    }
    const unsigned long long bits = __ballot(far);
    if (threadIdx.x == 0) {
        mask[(size_t)g * nw + blockIdx.y] = bits;
        if (bits) *any = 1;
    }
}

// Near terms: body i per lane, the near groups h = share modulo 64 with
// wave-uniform addresses.  FP64 issue.  So many shares because a few groups (the
// sparse rim of a disk) are near to most others and last (8 shares: 2.32 ms at
// 262,144 bodies and 0.98 at 65,536, 32: 1.29 and 0.28), and because fewer leave
// compute units idle at the end where all groups are near to all (softening
// lengths above some 1e-4 of the system; 45,983 bodies: 1.64 ms with 32 shares in
// workgroups of 8 wavefronts, 1.58 so).
template <bool SOFT>
__global__ __launch_bounds__(64 * NW) void k_mix_near(const double4 *__restrict__ jd,
                                                 const double *__restrict__ jsig,
                                                 const Scal *__restrict__ scal, int nw, int nslots,
                                                 const unsigned long long *__restrict__ mask,
                                                 double *__restrict__ part)
{
    __shared__ double sum[NW][3][MG];
    const int nv = scal->nvalid, ng = (nv + MG - 1) / MG;
    const int g = blockIdx.x, lane = threadIdx.x & 63, i = g * MG + lane;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int share = blockIdx.y * NW + wv;
    if (g >= ng) return;
    const double4 me = jd[i];
    const double si = SOFT ? jsig[i] : 0.0;
    double ax = 0.0, ay = 0.0, az = 0.0;
    const unsigned long long *row = mask + (size_t)g * nw;
    for (int h = share; h < ng; h += 64) {
        if ((row[h >> 6] >> share) & 1) continue;
        const int jb = h * MG, cnt = min(MG, nv - jb);
        if (h == g) {
            for (int jj = 0; jj < cnt; ++jj)
                near_term_self<1, SOFT>(jd[jb + jj], SOFT ? jsig[jb + jj] : 0.0, jb + jj, i, MG, &me.x,
                                        &me.y, &me.z, &si, &ax, &ay, &az);
        } else if (cnt == MG) {
#pragma unroll 4
            for (int jj = 0; jj < MG; ++jj)
                near_term<1, SOFT>(jd[jb + jj], SOFT ? jsig[jb + jj] : 0.0, &me.x, &me.y, &me.z, &si,
                                   &ax, &ay, &az);
        } else {
            for (int jj = 0; jj < cnt; ++jj)
                near_term<1, SOFT>(jd[jb + jj], SOFT ? jsig[jb + jj] : 0.0, &me.x, &me.y, &me.z, &si,
                                   &ax, &ay, &az);
        }
    }
    sum[wv][0][lane] = ax;
    sum[wv][1][lane] = ay;
    sum[wv][2][lane] = az;
    __syncthreads();
    for (int e = threadIdx.x; e < 3 * MG; e += 64 * NW) {
        const int s = e / 3, d = e - 3 * s;
        double v = 0.0;
        for (int q = 0; q < NW; ++q) v += sum[q][d][s];
        if (g * MG + s < nv) part[3 * ((size_t)blockIdx.y * nslots + g * MG) + e] = v;
    }
}

template <int CTRL>
__device__ inline float dpp_get32(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}

template <int N, int CTRL>
__device__ inline void halve32(float *a, bool up)
{
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const float keep = up ? a[q + N] : a[q], give = up ? a[q] : a[q + N];
        a[q] = keep + dpp_get32<CTRL>(give);
    }
}

// One workgroup per (row group r, chunk c) with pairs j > i, as k_pairs_sym.
__global__ __launch_bounds__(SY_T, 4) void k_pairs_mix(const double4 *__restrict__ jd,
                                                       const TileHdr *__restrict__ hdr,
                                                       const Scal *__restrict__ scal, int nw,
                                                       const unsigned long long *__restrict__ mask,
                                                       const int *__restrict__ far, SymShape S,
                                                       double *__restrict__ pi,
                                                       double *__restrict__ pj)
{
    __shared__ double4 rec[SY_C];
    __shared__ double js[3][SY_C];
    int r, c;
    sym_place(S, blockIdx.x, r, c);
    const int nv = scal->nvalid, tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j0 = c * SY_C, row0 = r * S.W, h0 = j0 / MG;
    // Without two far groups there is nothing to form or to add (the flag's load
    // is one latency with nv's: before the others it cost 1.6 % at 65,536 bodies).
    if (!*far || j0 >= nv || row0 >= nv) return;
#pragma unroll
    for (int h = 0; h < SY_NB; ++h) {
        const int k = h * SY_T + tid;
        // Slots up to the end of the last group hold records.
        rec[k] = jd[min(j0 + k, (nv + MG - 1) / MG * MG - 1)];
        js[0][k] = js[1][k] = js[2][k] = 0.0;
    }
    __syncthreads();
    const int ng = (nv + MG - 1) / MG;
    for (int row = row0; row < row0 + S.W; row += MROW) {
        if (row >= nv || row >= j0 + SY_C) break;
        const int i0 = row + w * MI, g = min(i0 / MG, ng - 1);
        // The chunk's groups (a power of two of them, within one word) that are
        // far from g and above it.
        unsigned bits = 0, any = 0;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int f = row / MG + e;
            if (f >= ng) continue;
            unsigned v = (unsigned)(mask[(size_t)f * nw + (h0 >> 6)] >> (h0 & 63)) &
                         ((1u << (SY_C / MG)) - 1u);
            if (f >= h0) v &= ~((2u << (f - h0)) - 1u);
            any |= v;
            if (f == i0 / MG) bits = v;
        }
        double sum[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        float acc[3 * MI];
#pragma unroll
        for (int q = 0; q < 3 * MI; ++q) acc[q] = 0.f;
        if (any) {  // uniform in the workgroup
            const TileHdr th = hdr[g];
            float vx[MI], vy[MI], vz[MI], mi[MI];
#pragma unroll
            for (int u = 0; u < MI; ++u) {
                const double4 p = jd[min(i0 + u, ng * MG - 1)];
                vx[u] = (float)(p.x - th.ax);
                vy[u] = (float)(p.y - th.ay);
                vz[u] = (float)(p.z - th.az);
                mi[u] = (float)p.w;
                asm("" : "+v"(vx[u]), "+v"(vy[u]), "+v"(vz[u]), "+v"(mi[u]));
            }
            for (int s = 0; s < SY_WAVES; ++s) {
#pragma unroll
                for (int h = 0; h < SY_NB; ++h) {
                    const int blk = ((w + s) & (SY_WAVES - 1)) * SY_NB + h;
                    if (!((bits >> blk) & 1u)) continue;
                    const int k = blk * 64 + lane;
                    const double4 q = rec[k];
                    const float wx = (float)(q.x - th.ax), wy = (float)(q.y - th.ay),
                                wz = (float)(q.z - th.az), mj = (float)q.w;
                    float bx = 0.f, by = 0.f, bz = 0.f;
#pragma unroll
                    for (int u = 0; u < MI; ++u) {
                        const float dx = wx - vx[u], dy = wy - vy[u], dz = wz - vz[u];
                        const float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                        const float y = __builtin_amdgcn_rsqf(r2);
                        const float y3 = (y * y) * y;
                        const float a = mj * y3, b = mi[u] * y3;
                        acc[3 * u] = fmaf(a, dx, acc[3 * u]);
                        acc[3 * u + 1] = fmaf(a, dy, acc[3 * u + 1]);
                        acc[3 * u + 2] = fmaf(a, dz, acc[3 * u + 2]);
                        bx = fmaf(b, dx, bx);
                        by = fmaf(b, dy, by);
                        bz = fmaf(b, dz, bz);
                    }
                    js[0][k] -= (double)bx;
                    js[1][k] -= (double)by;
                    js[2][k] -= (double)bz;
                }
                __syncthreads();
            }
            // Value 3 u + d; a lane ends with the sums of body u = bits 3, 2, 1
            // of its number (partners as in lanes_sum4).
            halve32<24, 0x140>(acc, (lane & 8) != 0);
            halve32<12, 0x141>(acc, (lane & 4) != 0);
            halve32<6, 0x1b>(acc, (lane & 2) != 0);
#pragma unroll
            for (int d = 0; d < 6; ++d) sum[d] = (double)acc[d];
            halve64<3, 0xb1>(sum, (lane & 1) != 0);
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                sum[d] += __shfl_xor(sum[d], 16);
                sum[d] += __shfl_xor(sum[d], 32);
            }
        }
        const int u = lane & 15;
        if (lane < 16 && i0 + u < nv) {
            double *o = pi + 3 * (S.ioff(c) + i0 + u);
            o[0] = sum[0];
            o[1] = sum[1];
            o[2] = sum[2];
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

static SymShape fast64_shape(int32_t n) { return sym_shape(n, SY_NB, GI, sym_reps(n)); }

// Rows a row group: few where workgroups are few (32,800 bodies, 2 / 8: 0.44
// and 0.50 ms), many where the partial sums weigh (262,144: 17.8 and 16.9).
static SymShape mixed_shape(int32_t n)
{
    return sym_shape(n, SY_NB, MI, n <= 65536 ? 2 : n <= 131072 ? 4 : 8);
}

bool ncg_sym_room(ncg_ctx *ctx, int32_t n, ncg_precision prec, bool make)
{
    const SymShape S = prec == NCG_MIXED ? mixed_shape(n) : fast64_shape(n);
    return ncg_pair_scratch(ctx, "y_pi", 24 * (size_t)S.islots(), "y_pj", 24 * (size_t)S.jslots(),
                            make);
}

// Callers have ncg_sym_room's word for the partial sums.
ncg_status ncg_gravity_sym(ncg_ctx *ctx, const DBody *d_b, int32_t n, const int *d_perm,
                           const int *d_nvalid, const ncg_central *c, const double *d_central,
                           double G, double soft, double *d_acc, double *d_cm_acc, hipStream_t st)
{
    const SymShape S = fast64_shape(n);
    double4 *jd = dbuf<double4>(ctx, "y_jd", n);
    double *jsig = dbuf<double>(ctx, "y_jsig", n);
    double *pi = static_cast<double *>(ctx->bufs["y_pi"].ptr);
    double *pj = static_cast<double *>(ctx->bufs["y_pj"].ptr);
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
                       d_central, G, (const double *)nullptr, 0, (const int *)nullptr,
                       (const Scal *)nullptr, d_acc, cmpart);
    if (d_cm_acc)
        hipLaunchKernelGGL(k_sym_cm, dim3(1), dim3(FT), 0, st, cmpart, nb, d_cm_acc);
    NCG_CHECK_LAUNCH();
    return NCG_OK;
}

ncg_status ncg_gravity_mixed_sym(ncg_ctx *ctx, const DBody *d_b, int32_t n, const int *d_perm,
                                 const void *d_scal, const ncg_central *c, const double *d_central,
                                 double G, double soft, double theta, double *d_acc,
                                 double *d_cm_acc, hipStream_t st)
{
    const Scal *scal = static_cast<const Scal *>(d_scal);
    const SymShape S = mixed_shape(n);
    const int ng = (int)cdiv(n, MG), nw = (int)cdiv(ng, 64);
    double4 *jd = dbuf<double4>(ctx, "y_jd", (size_t)ng * MG);
    double *jsig = dbuf<double>(ctx, "y_jsig", (size_t)ng * MG);
    TileHdr *hdr = dbuf<TileHdr>(ctx, "y_hdr", ng);
    unsigned long long *mask = dbuf<unsigned long long>(ctx, "y_mask", (size_t)ng * nw);
    double *near = dbuf<double>(ctx, "y_near", 3 * (size_t)MNEAR * n);
    int *far = dbuf<int>(ctx, "y_far", 1);
    double *pi = static_cast<double *>(ctx->bufs["y_pi"].ptr);
    double *pj = static_cast<double *>(ctx->bufs["y_pj"].ptr);
    const int nb = (int)cdiv(n, FS);
    double *cmpart = d_cm_acc ? dbuf<double>(ctx, "y_cm", 3 * (size_t)nb) : nullptr;
    if (!jd || !jsig || !hdr || !mask || !near || !far || !pi || !pj || (d_cm_acc && !cmpart))
        return NCG_ERR_NOMEM;
    hipLaunchKernelGGL(k_mix_records, dim3(ng), dim3(64), 0, st, d_b, d_perm, scal, G, soft, jd, jsig,
                       hdr, far);
    hipLaunchKernelGGL(k_mix_mask, dim3(ng, nw), dim3(64), 0, st, hdr, scal, nw, theta, soft, mask,
                       far);
    NCG_CHECK_LAUNCH();
    {
        ProfScope ps(ctx, st, "pairs_mixed");
        if (soft != 0.0)
            hipLaunchKernelGGL(k_mix_near<true>, dim3(ng, MNEAR), dim3(64 * NW), 0, st, jd, jsig, scal,
                               nw, (int)n, mask, near);
        else
            hipLaunchKernelGGL(k_mix_near<false>, dim3(ng, MNEAR), dim3(64 * NW), 0, st, jd, jsig, scal,
                               nw, (int)n, mask, near);
        hipLaunchKernelGGL(k_pairs_mix, dim3((unsigned)S.workgroups()), dim3(SY_T), 0, st, jd, hdr,
                           scal, nw, mask, far, S, pi, pj);
        NCG_CHECK_LAUNCH();
    }
    const int cp = (c && c->present) ? 1 : 0;
    hipLaunchKernelGGL(k_sym_finish, dim3(nb), dim3(FT), 0, st, d_b, d_perm, &scal->nvalid, S, pi, pj,
                       cp, cp ? c->x : 0.0, cp ? c->y : 0.0, cp ? c->z : 0.0,
                       cp ? G * c->mass : 0.0, d_central, G, near, MNEAR, far, scal, d_acc, cmpart);
    if (d_cm_acc)
        hipLaunchKernelGGL(k_sym_cm, dim3(1), dim3(FT), 0, st, cmpart, nb, d_cm_acc);
    NCG_CHECK_LAUNCH();
    return NCG_OK;
}
