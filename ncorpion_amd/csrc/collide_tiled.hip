// Brute-force collision pass over spatial tiles, for one system of NCG_CP_MIN
// bodies and more (the search alone, for host calls, from NCG_CP_HOST_MIN).
//
// The pass has brute_force's results (NcorpiON collision.c:425-456): every
// pair i < j is a candidate exactly when closest_approach's predicate accepts
// it (collide_allpairs.hip tests all of them), but a pair can only meet within
// dt when its distance is at most R + |dv| |dt|.  The bodies are put into the
// cells of a Hilbert grid by a counting sort, cut into tiles of 64, and a tile
// pair whose boxes (of positions, of velocities, and the largest |radius|) are
// farther apart than that is skipped, then each body of a tile pair left that
// is too far from the other tile's box.  What remains is tested with the same
// predicate, so the candidates are the same set whatever the order of the
// bodies in the tiles.
//
// 65,536 bodies, R = 2e-4, dt = 2 pi / 256: the tests of all pairs took 2.39 ms;
// here the order, boxes and tests of a pass take 0.09 ms (the tests 0.043), most
// of it the seven launches' latency.
//
// The replay decides the candidates in brute_force's order with one workgroup
// (k_cp_replay): a resolved pair changes two bodies, and the pairs they may
// take part in later in the pass are found at once by testing both new states
// against every tile box, then the bodies of the tiles within reach.  The
// replay of rows by one wavefront (k_bf_replay) reads every body for each
// changed one and walks the rows between: 13.2 ms for 25 collisions among
// 65,536 bodies against 0.16 ms here (about 6 us a collision: a chain of dependent
// loads, the bounce and the two scans).
//
// Where every pair is within reach (a timestep in which bodies cross the system)
// nothing is skipped, and the search takes 1.5 to 1.7 times the tests of all pairs.
//
// Nothing here is a library sort or a memset, so the pass can be captured in a
// graph.
#include <algorithm>

#include "ncg_internal.hpp"
#include "collide_dev.hpp"
#include "tiled_dev.hpp"

#pragma clang fp contract(off)

namespace {

constexpr int CT = 256;        // threads of the order kernels
constexpr int CPT = 64;        // bodies of a tile
constexpr int CBIN = 1024;     // cells of one block of the scan
constexpr int CPARTS = 256;    // partial sums of the frame
constexpr int CSTAT = 13;      // per axis: min, max, sum, sum of squares; count

// Body of a tile (id: its slot).
struct alignas(64) CpRec {
    double x, y, z, vx, vy, vz, R;
    int id, pad;
};

// Boxes of the tiles, one array of `ntiles` values per bound: positions lo
// and hi, velocities lo and hi (three each), largest |radius| (the predicate
// takes the square of a sum of radii, of any sign).
constexpr int CBOX = 13;

__device__ inline double wave_min(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o));
    return v;
}

__device__ inline double wave_max(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    return v;
}

__device__ inline double wave_sum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Partial statistics of the existing bodies' positions (bodies with a
// coordinate that is not finite left out: they are in no candidate), and the
// cell counts zeroed.
__global__ __launch_bounds__(CT) void k_cp_stats(const DBody *__restrict__ b, int n,
                                                 const int32_t *__restrict__ ex,
                                                 double *__restrict__ part,
                                                 unsigned *__restrict__ hist, int bins)
{
    __shared__ double sh[CT / 64][CSTAT];
    for (int q = blockIdx.x * CT + threadIdx.x; q < bins; q += gridDim.x * CT) hist[q] = 0u;
    double mn[3], mx[3], s1[3], s2[3], cnt = 0.0;
    for (int c = 0; c < 3; ++c) {
        mn[c] = 1e300;
        mx[c] = -1e300;
        s1[c] = s2[c] = 0.0;
    }
    for (int k = blockIdx.x * CT + threadIdx.x; k < n; k += gridDim.x * CT) {
        if (ex && !ex[k]) continue;
        const double p[3] = {b[k].x, b[k].y, b[k].z};
        if (!(fabs(p[0]) < 1e150 && fabs(p[1]) < 1e150 && fabs(p[2]) < 1e150)) continue;
        for (int c = 0; c < 3; ++c) {
            mn[c] = fmin(mn[c], p[c]);
            mx[c] = fmax(mx[c], p[c]);
            s1[c] += p[c];
            s2[c] += p[c] * p[c];
        }
        cnt += 1.0;
    }
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double v[CSTAT];
    for (int c = 0; c < 3; ++c) {
        v[c] = wave_min(mn[c]);
        v[3 + c] = wave_max(mx[c]);
        v[6 + c] = wave_sum(s1[c]);
        v[9 + c] = wave_sum(s2[c]);
    }
    v[12] = wave_sum(cnt);
    if (lane == 0)
        for (int c = 0; c < CSTAT; ++c) sh[w][c] = v[c];
    __syncthreads();
    if (threadIdx.x < CSTAT) {
        const int c = threadIdx.x;
        double a = sh[0][c];
        for (int q = 1; q < CT / 64; ++q)
            a = c < 3 ? fmin(a, sh[q][c]) : c < 6 ? fmax(a, sh[q][c]) : a + sh[q][c];
        part[blockIdx.x * CSTAT + c] = a;
    }
}

// Cell of every existing body and its rank among the cell's bodies.  The grid
// spans the bounding box cut at 2.5 standard deviations around the mean, so
// that one body far out does not leave the others in a few cells (bodies
// outside go to the border cells; the tile boxes are those of the bodies).
__global__ __launch_bounds__(CT) void k_cp_cells(const DBody *__restrict__ b, int n,
                                                 const int32_t *__restrict__ ex,
                                                 const double *__restrict__ part, int nparts,
                                                 int bits, unsigned *__restrict__ hist,
                                                 unsigned *__restrict__ cell,
                                                 unsigned *__restrict__ rank)
{
    __shared__ double sh[CT / 64][CSTAT], fr[CSTAT];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    {
        const bool on = (int)threadIdx.x < nparts;
        const double *p = part + (on ? threadIdx.x : 0) * CSTAT;
        for (int c = 0; c < CSTAT; ++c) {
            const double x = on ? p[c] : c < 3 ? 1e300 : c < 6 ? -1e300 : 0.0;
            const double v = c < 3 ? wave_min(x) : c < 6 ? wave_max(x) : wave_sum(x);
            if (lane == 0) sh[w][c] = v;
        }
        __syncthreads();
        if (threadIdx.x < CSTAT) {
            const int c = threadIdx.x;
            double a = sh[0][c];
            for (int q = 1; q < CT / 64; ++q)
                a = c < 3 ? fmin(a, sh[q][c]) : c < 6 ? fmax(a, sh[q][c]) : a + sh[q][c];
            fr[c] = a;
        }
        __syncthreads();
    }
    const int k = blockIdx.x * CT + threadIdx.x;
    if (k >= n) return;
    if (ex && !ex[k]) {
        cell[k] = 0xffffffffu;
        return;
    }
    double lo[3], width = 0.0;
    const double cnt = fmax(fr[12], 1.0);
    for (int c = 0; c < 3; ++c) {
        const double mean = fr[6 + c] / cnt;
        const double dev = 2.5 * sqrt(fmax(fr[9 + c] / cnt - mean * mean, 0.0));
        const double l = fmax(fr[c], mean - dev), h = fmin(fr[3 + c], mean + dev);
        width = fmax(width, h - l);
        lo[c] = 0.5 * (l + h);
    }
    const double p[3] = {b[k].x, b[k].y, b[k].z};
    const int side = 1 << bits;
    unsigned q[3];
    for (int c = 0; c < 3; ++c) {
        const double f = width > 0.0 ? ((p[c] - lo[c]) / width + 0.5) * side : 0.0;
        q[c] = f >= side - 1 ? (unsigned)(side - 1) : f > 0.0 ? (unsigned)f : 0u;
    }
    const unsigned key = bits == 6 ? hilbert<6>(q[0], q[1], q[2]) : hilbert<7>(q[0], q[1], q[2]);
    cell[k] = key;
    rank[k] = atomicAdd(&hist[key], 1u);
}

// Exclusive prefix of each block of CBIN cells, and the block's total.
__global__ __launch_bounds__(CT) void k_cp_scan(unsigned *__restrict__ hist,
                                                unsigned *__restrict__ tot)
{
    __shared__ unsigned ws[CT / 64];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    uint4 *h4 = reinterpret_cast<uint4 *>(hist + (size_t)blockIdx.x * CBIN);
    const uint4 v = h4[t];
    const unsigned sum = v.x + v.y + v.z + v.w;
    unsigned inc = sum;
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned u = __shfl_up(inc, o);
        if (lane >= o) inc += u;
    }
    if (lane == 63) ws[w] = inc;
    __syncthreads();
    unsigned base = inc - sum;
    for (int q = 0; q < w; ++q) base += ws[q];
    uint4 r;
    r.x = base;
    r.y = r.x + v.x;
    r.z = r.y + v.y;
    r.w = r.z + v.z;
    h4[t] = r;
    if (t == CT - 1) tot[blockIdx.x] = base + sum;
}

// The bodies in cell order; *nvalid: existing bodies.  Every block forms the
// prefix of the block totals it needs (at most 2048 of them).
__global__ __launch_bounds__(CT) void k_cp_place(const DBody *__restrict__ b, int n,
                                                 const unsigned *__restrict__ hist,
                                                 const unsigned *__restrict__ tot, int nblk,
                                                 const unsigned *__restrict__ cell,
                                                 const unsigned *__restrict__ rank,
                                                 CpRec *__restrict__ rec, int *__restrict__ nvalid)
{
    __shared__ unsigned pre[2048], ws[CT / 64];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    unsigned v[8], sum = 0;
    for (int q = 0; q < 8; ++q) {
        const int k = t * 8 + q;
        v[q] = k < nblk ? tot[k] : 0u;
        sum += v[q];
    }
    unsigned inc = sum;
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned u = __shfl_up(inc, o);
        if (lane >= o) inc += u;
    }
    if (lane == 63) ws[w] = inc;
    __syncthreads();
    unsigned base = inc - sum;
    for (int q = 0; q < w; ++q) base += ws[q];
    if (blockIdx.x == 0 && t == CT - 1) *nvalid = (int)(base + sum);
    for (int q = 0; q < 8; ++q) {
        pre[t * 8 + q] = base;
        base += v[q];
    }
    __syncthreads();
    const int k = blockIdx.x * CT + t;
    if (k >= n) return;
    const unsigned c = cell[k];
    if (c == 0xffffffffu) return;
    const unsigned slot = pre[c / CBIN] + hist[c] + rank[k];
    const DBody q = b[k];
    CpRec r;
    r.x = q.x;
    r.y = q.y;
    r.z = q.z;
    r.vx = q.vx;
    r.vy = q.vy;
    r.vz = q.vz;
    r.R = q.radius;
    r.id = k;
    r.pad = 0;
    rec[slot] = r;
}

// One wavefront per tile.
__global__ __launch_bounds__(CT) void k_cp_boxes(const CpRec *__restrict__ rec,
                                                 const int *__restrict__ nvalid, int ntiles,
                                                 double *__restrict__ box)
{
    const int t = blockIdx.x * (CT / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nv = *nvalid;
    if (t >= ntiles || t * CPT >= nv) return;
    const CpRec r = rec[min(t * CPT + lane, nv - 1)];
    const double v[7] = {r.x, r.y, r.z, r.vx, r.vy, r.vz, fabs(r.R)};
    double o[CBOX];
    for (int c = 0; c < 3; ++c) {
        o[c] = wave_min(v[c]);
        o[3 + c] = wave_max(v[c]);
        o[6 + c] = wave_min(v[3 + c]);
        o[9 + c] = wave_max(v[3 + c]);
    }
    o[12] = wave_max(v[6]);
    if (lane == 0)
        for (int c = 0; c < CBOX; ++c) box[(size_t)c * ntiles + t] = o[c];
}

struct CpBox {
    double lo[3], hi[3], vlo[3], vhi[3], rmax;
};

__device__ inline CpBox load_box(const double *__restrict__ box, int ntiles, int t)
{
    CpBox o;
    for (int c = 0; c < 3; ++c) {
        o.lo[c] = box[(size_t)c * ntiles + t];
        o.hi[c] = box[(size_t)(3 + c) * ntiles + t];
        o.vlo[c] = box[(size_t)(6 + c) * ntiles + t];
        o.vhi[c] = box[(size_t)(9 + c) * ntiles + t];
    }
    o.rmax = box[(size_t)12 * ntiles + t];
    return o;
}

// Whether a body of one box may be accepted with a body of the other: the
// predicate needs |d| <= R + |dv| t with t <= dt (t < 0: the bodies overlap,
// |d| < R), up to the rounding of its own operations, at most ~1e-7 of |d|
// (a discriminant rounded to a positive value); (1 + 1e-6) covers it.  Any NaN
// keeps the pair.  A body alone is the box with equal bounds.
__device__ inline bool may_meet(const CpBox &a, const CpBox &c, double adt)
{
    double d2 = 0.0, v2 = 0.0;
    for (int k = 0; k < 3; ++k) {
        const double g = fmax(0.0, fmax(a.lo[k] - c.hi[k], c.lo[k] - a.hi[k]));
        d2 += g * g;
        const double v = fmax(fabs(a.vhi[k] - c.vlo[k]), fabs(c.vhi[k] - a.vlo[k]));
        v2 += v * v;
    }
    const double reach = ((a.rmax + c.rmax) + sqrt(v2) * adt) * (1.0 + 1e-6);
    return !(d2 > reach * reach);
}

__device__ inline CpBox body_box(const double *v /* x, y, z, vx, vy, vz, R */)
{
    CpBox o;
    for (int c = 0; c < 3; ++c) {
        o.lo[c] = o.hi[c] = v[c];
        o.vlo[c] = o.vhi[c] = v[3 + c];
    }
    o.rmax = fabs(v[6]);
    return o;
}

// Which tiles J >= I the tiles I of a slab (rows row0 ..) may meet: one bit
// each, rows of nw words.  One wavefront per (64 tiles J, CPI tiles I): the J
// boxes stay in registers.
constexpr int CPI = 8;

__global__ __launch_bounds__(64) void k_cp_near(const int *__restrict__ nvalid, int ntiles,
                                                const double *__restrict__ box, double adt,
                                                int row0, int rows, int nw,
                                                unsigned long long *__restrict__ mask)
{
    const int lane = threadIdx.x, nt = (*nvalid + CPT - 1) / CPT;
    const int J = blockIdx.y * 64 + lane;
    const int i0 = row0 + blockIdx.x * CPI, i1 = min(min(i0 + CPI, row0 + rows), nt);
    if (i0 >= nt) return;
    const bool on = J < nt;
    const CpBox bj = load_box(box, ntiles, on ? J : 0);
    for (int I = i0; I < i1; ++I) {
        unsigned long long m = 0ull;
        if ((int)blockIdx.y * 64 + 63 >= I)
            m = __ballot(on && J >= I && may_meet(load_box(box, ntiles, I), bj, adt));
        if (lane == 0) mask[(size_t)(I - row0) * nw + blockIdx.y] = m;
    }
}

// One wavefront per (tile I, share of the tiles J that k_cp_near found): the
// bodies of each tile that reach the other's box, and those of the tile with
// fewer, each against the other tile's 64 (one per lane).  A tile across a gap
// of the curve has a box as large as the system and meets every tile, with all
// of their bodies but almost none of its own: taking the shorter side brought
// 65,536 bodies from 421 to 43 us.
__global__ __launch_bounds__(64) void k_cp_pairs(const CpRec *__restrict__ rec,
                                                 const int *__restrict__ nvalid, int ntiles,
                                                 const double *__restrict__ box, double dt,
                                                 int row0, int nw,
                                                 const unsigned long long *__restrict__ mask,
                                                 int2 *__restrict__ out, unsigned long long cap,
                                                 unsigned long long *__restrict__ count)
{
    __shared__ double sv[2][7][CPT];
    __shared__ int sid[2][CPT];
    const int lane = threadIdx.x, I = row0 + blockIdx.x;
    const int nv = *nvalid, nt = (nv + CPT - 1) / CPT;
    if (I >= nt) return;
    const double adt = fabs(dt);
    const CpBox bi = load_box(box, ntiles, I);
    const bool iv = I * CPT + lane < nv;
    const CpRec a = rec[min(I * CPT + lane, nv - 1)];
    const double va[7] = {a.x, a.y, a.z, a.vx, a.vy, a.vz, a.R};
    for (int k = 0; k < 7; ++k) sv[0][k][lane] = va[k];
    sid[0][lane] = a.id;
    const unsigned long long *row = mask + (size_t)blockIdx.x * nw;
    unsigned turn = 0;  // tiles found so far: shares take them in turn
    for (int c0 = I / 64; c0 < (nt + 63) / 64; c0 += 64) {
        const unsigned long long mine = c0 + lane < (nt + 63) / 64 ? row[c0 + lane] : 0ull;
        unsigned long long words = __ballot(mine != 0ull);
        while (words) {
            const int wl = __ffsll((long long)words) - 1;
            words &= words - 1;
            unsigned long long m = __shfl(mine, wl);
            while (m) {
                const int j = (c0 + wl) * 64 + __ffsll((long long)m) - 1;
                m &= m - 1;
                if ((turn++ & (gridDim.y - 1)) != blockIdx.y) continue;
                const bool jv = j * CPT + lane < nv;
                const CpRec q = rec[min(j * CPT + lane, nv - 1)];
                const double v[7] = {q.x, q.y, q.z, q.vx, q.vy, q.vz, q.R};
                const unsigned long long jm = __ballot(jv && may_meet(body_box(v), bi, adt));
                const unsigned long long im =
                    __ballot(iv && may_meet(body_box(va), load_box(box, ntiles, j), adt));
                if (!jm || !im) continue;
                // Ordered after the reads of the previous tile and before the
                // reads below.
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
                for (int k = 0; k < 7; ++k) sv[1][k][lane] = v[k];
                sid[1][lane] = q.id;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
                const bool turned = __popcll(im) < __popcll(jm);
                const int side = turned ? 0 : 1;
                const CpRec &l = turned ? q : a;
                const bool on = turned ? jv : iv;
                for (unsigned long long um = turned ? im : jm; um; um &= um - 1) {
                    const int u = __ffsll((long long)um) - 1;
                    if (!on || (j == I && u <= lane)) continue;
                    const double(*o)[CPT] = sv[side];
                    if (approach_hit(l.x, l.y, l.z, l.vx, l.vy, l.vz, l.R, o[0][u], o[1][u],
                                     o[2][u], o[3][u], o[4][u], o[5][u], o[6][u], dt)) {
                        const unsigned long long slot = atomicAdd(count, 1ull);
                        const int id = sid[side][u];
                        if (slot < cap) out[slot] = make_int2(min(l.id, id), max(l.id, id));
                    }
                }
            }
        }
    }
}

// ---- replay ------------------------------------------------------------------
constexpr int RPT = 1024;     // threads of the replay
constexpr int RP_EV = NCG_CP_EVENTS;
constexpr int RP_DYN = NCG_CP_FOUND;
constexpr int RP_CH = NCG_CP_CHANGED;

__device__ inline unsigned long long pair_key(int a, int c)
{
    return ((unsigned long long)(unsigned)min(a, c) << 32) | (unsigned)max(a, c);
}

// brute_force's order is that of the key (i, j), i < j.  Wavefront 0 takes the
// smallest key not yet decided among the candidates (sorted) and the pairs
// that scans added, decides it at the current states and resolves a hit; then
// all wavefronts scan for the pairs after it that the two changed bodies may
// take part in.  A pair is decided with the states it has when its turn comes
// (NcorpiON's rule), and every pair that can be accepted then is listed: its
// bodies' last changes were followed by a scan at those states.  did_collide
// and holes as in k_bf_replay.  err: 1 more candidates than cap, 2 than RP_EV
// (both with nothing changed), 4 more changed bodies or found pairs than fit (in
// the middle of the pass): the caller restores the state and replays on the host.
__global__ __launch_bounds__(RPT) void k_cp_replay(
    DBody *__restrict__ b, const int32_t *__restrict__ ex, int32_t *__restrict__ dc, int one_coll,
    const CpRec *__restrict__ rec, const int *__restrict__ nvalid, int ntiles,
    const double *__restrict__ box, const int2 *__restrict__ cand,
    const unsigned long long *__restrict__ count, unsigned cap, double dt, double f,
    unsigned *__restrict__ ncoll, unsigned *__restrict__ err)
{
    __shared__ unsigned long long ev[RP_EV], dyn[RP_DYN];
    __shared__ int ch[RP_CH], tl[RPT];
    __shared__ int s_nd, s_ndyn, s_nt, s_i, s_j, s_known;
    __shared__ unsigned long long s_cur;
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const unsigned long long total = *count;
    if (total == 0ull) return;
    if (total > cap || total > RP_EV) {
        if (tid == 0) atomicOr(err, total > cap ? 1u : 2u);
        return;
    }
    const int m = (int)total;
    int P = 2;
    while (P < m) P <<= 1;
    for (int q = tid; q < P; q += RPT) {
        unsigned long long k = ~0ull;
        if (q < m) {
            const int2 c = cand[q];
            k = pair_key(c.x, c.y);
        }
        ev[q] = k;
    }
    if (tid == 0) {
        s_nd = 0;
        s_ndyn = 0;
    }
    __syncthreads();
    for (int k = 2; k <= P; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int q = tid; q < P / 2; q += RPT) {
                const int lo = 2 * q - (q & (j - 1));  // index with bit j clear
                const int hi = lo + j;
                const unsigned long long x = ev[lo], y = ev[hi];
                if ((x > y) == ((lo & k) == 0)) {
                    ev[lo] = y;
                    ev[hi] = x;
                }
            }
            __syncthreads();
        }
    const int nv = *nvalid, nt = (nv + CPT - 1) / CPT;
    const double adt = fabs(dt);
    unsigned hits = 0;             // wavefront 0
    unsigned long long cur = 0ull; // wavefront 0: the key decided last
    int ptr = 0;
    while (true) {
        if (w == 0) {
            int i = -1, j = -1;
            while (true) {
                unsigned long long best = ~0ull;
                for (int q = lane; q < s_ndyn; q += 64) {
                    const unsigned long long v = dyn[q];
                    if (v > cur && v < best) best = v;
                }
                for (int o = 32; o > 0; o >>= 1) {
                    const unsigned long long v = __shfl_xor(best, o);
                    best = v < best ? v : best;
                }
                while (ptr < m && ev[ptr] <= cur) ++ptr;
                if (ptr < m && ev[ptr] < best) best = ev[ptr];
                if (best == ~0ull) break;
                cur = best;
                i = (int)(best >> 32);
                j = (int)(best & 0xffffffffu);
                double ap[6], tc;
                const bool hit = bf_hit(b, ex, dc, i, j, dt, ap, &tc);
                if (!hit) {
                    i = -1;
                    continue;
                }
                if (lane == 0) {
                    bf_bounce(b, i, j, f, ap, tc);
                    if (dc) {
                        dc[i] = one_coll;
                        dc[j] = one_coll;
                    }
                }
                ++hits;
                break;
            }
            if (lane == 0) {
                s_i = i;
                s_j = j;
                s_cur = cur;
                s_known = 0;
            }
            __threadfence_block();
        }
        __syncthreads();
        const int i = s_i, j = s_j;
        if (i < 0) break;
        if (dc && one_coll) {  // neither body takes part in a later pair
            __syncthreads();
            continue;
        }
        const unsigned long long now = s_cur;
        const DBody A = b[i], B = b[j];
        const double va[7] = {A.x, A.y, A.z, A.vx, A.vy, A.vz, A.radius};
        const double vb[7] = {B.x, B.y, B.z, B.vx, B.vy, B.vz, B.radius};
        const CpBox ba = body_box(va), bb = body_box(vb);
        auto found = [&](int q, const DBody &X, int o, double x, double y, double z, double vx,
                         double vy, double vz, double R) {
            const unsigned long long key = pair_key(q, o);
            if (key <= now || q == o) return;
            if (approach_hit(X.x, X.y, X.z, X.vx, X.vy, X.vz, X.radius, x, y, z, vx, vy, vz, R, dt)) {
                const int slot = atomicAdd(&s_ndyn, 1);
                if (slot < RP_DYN) dyn[slot] = key;
            }
        };
        for (int t0 = 0; t0 < nt; t0 += RPT) {
            if (tid == 0) s_nt = 0;
            __syncthreads();
            const int t = t0 + tid;
            if (t < nt) {
                const CpBox c = load_box(box, ntiles, t);
                const int fl = (may_meet(ba, c, adt) ? 1 : 0) | (may_meet(bb, c, adt) ? 2 : 0);
                if (fl) tl[atomicAdd(&s_nt, 1)] = t * 4 + fl;
            }
            __syncthreads();
            const int nl = s_nt;
            for (int e = w; e < nl; e += RPT / 64) {
                const int tt = tl[e] >> 2, fl = tl[e] & 3;
                if (tt * CPT + lane < nv) {
                    const CpRec q = rec[tt * CPT + lane];
                    if (fl & 1) found(i, A, q.id, q.x, q.y, q.z, q.vx, q.vy, q.vz, q.R);
                    if (fl & 2) found(j, B, q.id, q.x, q.y, q.z, q.vx, q.vy, q.vz, q.R);
                }
            }
            __syncthreads();
        }
        // The bodies changed earlier, at their own states (their tiles hold
        // the old ones).
        const int nd = s_nd;
        for (int q = tid; q < nd; q += RPT) {
            const int o = ch[q];
            if (o == i) atomicOr(&s_known, 1);
            if (o == j) atomicOr(&s_known, 2);
            const DBody X = b[o];
            found(i, A, o, X.x, X.y, X.z, X.vx, X.vy, X.vz, X.radius);
            found(j, B, o, X.x, X.y, X.z, X.vx, X.vy, X.vz, X.radius);
        }
        __syncthreads();
        const int known = s_known;
        if (s_ndyn > RP_DYN || nd + 2 - __popc(known) > RP_CH) {
            if (tid == 0) atomicOr(err, 4u);
            break;
        }
        if (tid == 0) {
            int m2 = nd;
            if (!(known & 1)) ch[m2++] = i;
            if (!(known & 2)) ch[m2++] = j;
            s_nd = m2;
        }
        __syncthreads();
    }
    if (tid == 0 && hits) atomicAdd(ncoll, hits);
}

struct CpWork {
    double *part, *box;
    unsigned *hist, *tot, *cell, *rank;
    CpRec *rec;
    int *nvalid;
    unsigned long long *mask;
    int bits, bins, nblk, ntiles;
    int nw, slab;  // words of a row of tile bits, rows of a slab
};

ncg_status cp_work(ncg_ctx *ctx, int32_t n, CpWork &w)
{
    // Cells smaller than a tile on a thin disk: 64 cells an axis up to 16,384
    // bodies (some 1.1e3 of them hold a disk around the origin), 128 above.
    w.bits = n <= (1 << 14) ? 6 : 7;
    w.bins = 1 << (3 * w.bits);
    w.nblk = w.bins / CBIN;
    w.ntiles = (int)cdiv(n, CPT);
    w.part = dbuf<double>(ctx, "cp_part", CPARTS * CSTAT);
    w.hist = dbuf<unsigned>(ctx, "cp_hist", (size_t)w.bins);
    w.tot = dbuf<unsigned>(ctx, "cp_tot", (size_t)w.nblk);
    w.cell = dbuf<unsigned>(ctx, "cp_cell", (size_t)n);
    w.rank = dbuf<unsigned>(ctx, "cp_rank", (size_t)n);
    w.rec = dbuf<CpRec>(ctx, "cp_rec", (size_t)n);
    w.box = dbuf<double>(ctx, "cp_box", (size_t)CBOX * w.ntiles);
    w.nvalid = dbuf<int>(ctx, "cp_nvalid", 1);
    // The tile bits of a slab of rows: 64 MiB (all rows up to 1.4M bodies).
    w.nw = (int)cdiv(w.ntiles, 64);
    w.slab = (int)std::max<long>(CPI, std::min<long>(w.ntiles, (8L << 20) / w.nw));
    w.mask = dbuf<unsigned long long>(ctx, "cp_mask", (size_t)w.slab * w.nw);
    if (!w.mask || !w.part || !w.hist || !w.tot || !w.cell || !w.rank || !w.rec || !w.box || !w.nvalid)
        return NCG_ERR_NOMEM;
    return NCG_OK;
}

}  // namespace

ncg_status ncg_cp_candidates_launch(ncg_ctx *ctx, const DBody *d_b, int32_t n, const int32_t *d_ex,
                                    double dt, int2 *d_out, unsigned long long cap,
                                    unsigned long long *d_count, hipStream_t st)
{
    CpWork w;
    ncg_status r = cp_work(ctx, n, w);
    if (r != NCG_OK) return r;
    const int nparts = (int)std::min<long>(CPARTS, cdiv(n, CT));
    hipLaunchKernelGGL(k_cp_stats, dim3(nparts), dim3(CT), 0, st, d_b, (int)n, d_ex, w.part, w.hist,
                       w.bins);
    hipLaunchKernelGGL(k_cp_cells, dim3(cdiv(n, CT)), dim3(CT), 0, st, d_b, (int)n, d_ex, w.part,
                       nparts, w.bits, w.hist, w.cell, w.rank);
    hipLaunchKernelGGL(k_cp_scan, dim3(w.nblk), dim3(CT), 0, st, w.hist, w.tot);
    hipLaunchKernelGGL(k_cp_place, dim3(cdiv(n, CT)), dim3(CT), 0, st, d_b, (int)n, w.hist, w.tot,
                       w.nblk, w.cell, w.rank, w.rec, w.nvalid);
    hipLaunchKernelGGL(k_cp_boxes, dim3(cdiv(w.ntiles, CT / 64)), dim3(CT), 0, st, w.rec, w.nvalid,
                       w.ntiles, w.box);
    NCG_CHECK_LAUNCH();
    // Shares of a tile's neighbours for at least 8192 wavefronts (8 per SIMD).
    int share = 1;
    while (share < 64 && share * w.ntiles < 8192) share *= 2;
    ProfScope ps(ctx, st, "candidates");
    for (int row0 = 0; row0 < w.ntiles; row0 += w.slab) {
        const int rows = std::min(w.slab, w.ntiles - row0);
        hipLaunchKernelGGL(k_cp_near, dim3(cdiv(rows, CPI), w.nw), dim3(64), 0, st, w.nvalid,
                           w.ntiles, w.box, fabs(dt), row0, rows, w.nw, w.mask);
        hipLaunchKernelGGL(k_cp_pairs, dim3(rows, share), dim3(64), 0, st, w.rec, w.nvalid,
                           w.ntiles, w.box, dt, row0, w.nw, w.mask, d_out, cap, d_count);
        NCG_CHECK_LAUNCH();
    }
    return NCG_OK;
}

ncg_status ncg_cp_replay_launch(ncg_ctx *ctx, DBody *d_b, int32_t n, const int32_t *d_ex,
                                int32_t *d_dc, int one_collision_only, const int2 *d_cand,
                                const unsigned long long *d_count, unsigned cap, double dt,
                                double f, unsigned *d_stat, hipStream_t st)
{
    CpWork w;
    ncg_status r = cp_work(ctx, n, w);
    if (r != NCG_OK) return r;
    hipLaunchKernelGGL(k_cp_replay, dim3(1), dim3(RPT), 0, st, d_b, d_ex, d_dc, one_collision_only,
                       w.rec, w.nvalid, w.ntiles, w.box, d_cand, d_count, cap, dt, f, d_stat,
                       d_stat + 1);
    NCG_CHECK_LAUNCH();
    return NCG_OK;
}
