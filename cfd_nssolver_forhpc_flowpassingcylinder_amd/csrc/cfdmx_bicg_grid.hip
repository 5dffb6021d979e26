// cfdmx_bicg_grid.hip -- the BiCGSTAB iteration of small grids as one resident kernel
// (bicgstabRe2.hpp:82-180): grids whose workgroups the device holds all at once.  On 256 CUs
// that is up to 128 march blocks of tiles over 512 cells (a million cells, two workgroups each),
// or 256 of smaller ones.
//
// Launched phase by phase, such a grid's iteration is bound by latency: a march block takes
// its 8 planes one after the other (phases A, B, C 13, 12 and 6 us at 128x64x4, 19, 17 and
// 18 us at 256x128x32), whatever it computes, and there are fewer blocks than CUs.  Here
// every march block is one workgroup that stays on its CU for the whole solve and keeps its
// cells' vectors with it: a thread owns one column of the tile, the block's 8 planes, with r,
// q or p, Ap and As in registers and r0 in LDS.  Memory is used for x, which only its owner
// reads, and for what the blocks tell each other:
//   - the cells along a block's faces (r and q after phase C, Ap after phase A), written
//     through to memory and read from there;
//   - each phase's partial sums.  A block writes its partials once its faces are written, and
//     every block waits for all of them, so the sums are also the barrier between the phases.
// A partial's slot holds kEmpty until it is written.  A block empties its slot of a phase
// after it has seen every partial of the next phase, which a block writes only when it has
// read all of this one; and it does so before its own partials of the phase after that, which
// every block waits for before it looks at the slot again.
// The sums keep the march order and the folds of the launched phases: same bits.
//
// A tile of more than 512 cells takes two workgroups, each with half the planes of its march
// block (two columns a thread): the first half in march order hands its running sums to the
// second.  With whole blocks of two columns the vectors spilled (49 us an iteration at
// 256x128x32 against 26), and only half the CUs had one.
//
// Measured, us an iteration, launched phases -> resident: 128x64x4 32.6 -> 11.5, 112x104x4
// 37 -> 14.9, 63x41x15 42 -> 19, 197x93x31 56 -> 25, 256x128x8 48 -> 21, 256x128x32 56 -> 26
// (PRE = 1: 62 -> 31).  What is left is the three waits, about 2 us each, and the arithmetic
// of a block's cells on one CU.
//
// All blocks have to be resident at once.  bicg_grid_cus takes no grid whose blocks the device
// cannot hold, and the caller has no more resident kernels of a process on a device than leave
// every block of each a CU of its own, so that a block that is not placed yet finds a CU without
// one; other kernels end by themselves.  (A cooperative launch would ask for the same, but the
// runtime has one queue for those: four contexts' 300 iterations at 64x40x8 take 17.6 ms so, 8.9
// by ordinary launches.)  Every wait is bounded all the same (kMaxPolls, seconds): a block that
// gives up raises `failed` and returns, as then do all others, and the caller solves again by
// launched phases.
#include "cfdmx_bicg.hpp"

#include <algorithm>

namespace cfdmx {

// a quiet NaN that no arithmetic produces (its payload is set); a partial that is this very
// value is written as the plain NaN
constexpr unsigned long long kEmpty = 0x7ff8dead5eed0001ull;
// looks at a slot before a block gives up (about a microsecond each, of waits that take two or
// three)
constexpr int kMaxPolls = 1 << 21;
constexpr int kGridHalo = 2; // cells of the rows beside the tile that one thread holds

__device__ __forceinline__ void put_through(double *p, double v)
{
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(p),
                       (unsigned long long)__double_as_longlong(v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double get_through(const double *p)
{
    return __longlong_as_double((long long)__hip_atomic_load(
        reinterpret_cast<const unsigned long long *>(p), __ATOMIC_RELAXED,
        __HIP_MEMORY_SCOPE_AGENT));
}

// before the launch: all slots empty; before a solve's first also the solver state kept aside
__global__ void k_grid_slots(int n, unsigned long long *slots, const KState *st, KState *keep)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) slots[q] = kEmpty;
    if (q == 0 && keep) *keep = *st;
}

// T threads a block, NC columns of the plane tile each (T * NC is at least the tile's cells).
// UNI (bicg_grid_uni): every block holds 8 planes and a whole tile, and every row has the same
// coefficients (a uniform grid), so that they are scalars and a row's diagonal is one of three
// values per column.
//
// A column or plane that does not exist holds zeros throughout: its coefficients towards the
// others are zeros, so that it takes part in the arithmetic without a branch, and only the
// writes and the sums leave it out.
template <int PRE, int T, int NC, int PL, bool UNI>
__global__ void __launch_bounds__(T)
k_bicg_grid(Geo g, BicgBuffers B, double *__restrict__ x, double *partC,
            unsigned long long *slots, KState *st, int *failed, int give_up, int m0, int count)
{
    static_assert(PL == kChunk || 2 * PL == kChunk, "whole or half march blocks");
    extern __shared__ double lds[];
    __shared__ double red[2][4];
    __shared__ int gave_up;
    __shared__ double cx[2][PL]; // x coefficients of the block's planes
    if (st->done) return; // the same for every block: nothing in this launch has written it
    constexpr int TN = T * NC;
    const int nb = g.nmarch, tid = threadIdx.x;
    // march block b; of two halves the first and the second in march order, the last of
    // which has the block's sums
    constexpr bool halves = PL < kChunk;
    const int b = halves ? (int)blockIdx.x >> 1 : (int)blockIdx.x;
    const bool second = halves && (blockIdx.x & 1), last = !halves || second;
    const int tile = b % g.ntile, chunk = b / g.ntile;
    int ib, d, all;
    march_span(g, chunk, ib, d, all);
    // the block's planes: len of them from i0
    const int head = min(PL, all), len = second ? all - head : head;
    int i0 = chunk * kChunk;
    if (d > 0 && second) i0 += head;                   // marching up, the second half is above
    if (d < 0 && !second) i0 += all - head;            // marching down, the first
    if (len == 0) i0 = 0; // holds nothing; any address inside will do
    const int q0 = tile * kTile, qn = min(kTile, g.cyz - q0);
    // an LDS plane: the tile's cells between the rows beside it, then one zero that stands
    // for a neighbour beyond a z wall
    const int H = g.nzc, WP = TN + 2 * H + 1;
    double *Z = lds + PL * WP; // r0, plane by plane
    // slots of phase A (1 sum), B and C (2 sums), by block
    unsigned long long *slotA = slots, *slotB = slots + nb, *slotC = slots + 3 * nb;
    if (tid == 0) gave_up = give_up;
    if (tid < PL) {
        cx[0][tid] = tid < len ? g.pa[0].m[i0 + tid] : 0.0;
        cx[1][tid] = tid < len ? g.pa[0].p[i0 + tid] : 0.0;
    }
    __syncthreads();
    // planes beyond the block's in x
    const bool xlo = len > 0 && i0 > 0, xhi = len > 0 && i0 + len < g.nxc;
    const unsigned step = (unsigned)g.cyz * 8u;
    // UNI: the coefficients of every row
    const double uxm = g.pa[0].m[0], uxp = g.pa[0].p[0], uym = g.pa[1].m[0], uyp = g.pa[1].p[0],
                 uzm = g.pa[2].m[0], uzp = g.pa[2].p[0];
    const unsigned back = xlo ? step : 0u, ahead = xhi ? step * (unsigned)len : 0u;
    struct Col {
        bool ok, yrow;                // the cell exists; other blocks read it as a row
        unsigned own;                 // byte offset of element (i0, q)
        int so, zmo, zpo;             // LDS index of plane 0, and of its z neighbours from there
        double ym, yp, zm, zp;        // y and z coefficients
        double eym, eyp, ezm, ezp;    // what the diagonal leaves out of them
        double dg[3];                 // UNI: diagonal (PRE = 1: its reciprocal) of the block's
                                      // first, inner and last plane
    } col[NC];
    auto at = [&](auto *v, int c, int s) {
        using D = decltype(v);
        return (D)((const char *)v + (col[c].own + (unsigned)s * step));
    };
    double r[NC][PL] = {}, p[NC][PL] = {}; // p: q between phases C and A
    double ap[NC][PL] = {}, as[NC][PL] = {};
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        Col &w = col[c];
        const int tq = c * T + tid;
        w.ok = UNI || tq < qn;
        // (all of a block that ends below its last plane but not at the grid's end)
        w.yrow = w.ok && ((tile > 0 && tq < H) || (tile < g.ntile - 1 && tq >= qn - H) ||
                          (xhi && len < PL));
        const int q = q0 + (w.ok ? tq : 0);
        const int j = (int)fdiv((unsigned)q, g.dz), k = q - j * g.nzc;
        w.own = (unsigned)(i0 * g.cyz + q) * 8u;
        w.so = H + tq;
        w.zmo = k > 0 ? -1 : (g.zper ? g.nzc - 1 : WP - 1 - w.so);
        w.zpo = k < g.nzc - 1 ? 1 : (g.zper ? -(g.nzc - 1) : WP - 1 - w.so);
        w.ym = w.ok ? g.pa[1].m[j] : 0.0, w.yp = w.ok ? g.pa[1].p[j] : 0.0;
        w.zm = w.ok ? g.pa[2].m[k] : 0.0, w.zp = w.ok ? g.pa[2].p[k] : 0.0;
        w.eym = j == 0 ? w.ym : 0.0;
        w.eyp = j == g.nyc - 1 ? w.yp : 0.0;
        w.ezm = !g.zper && k == 0 ? w.zm : 0.0;
        w.ezp = !g.zper && k == g.nzc - 1 ? w.zp : 0.0;
        if (UNI) {
#pragma unroll
            for (int z = 0; z < 3; ++z) {
                const RowEnds end = {z == 0 && !xlo ? uxm : 0.0, z == 2 && !xhi ? uxp : 0.0,
                                     w.eym, w.eyp, w.ezm, w.ezp};
                w.dg[z] = march_diag<PRE>(end, uxm, uxp, uym, uyp, uzm, uzp);
                if (PRE) w.dg[z] = 1.0 / w.dg[z];
            }
        }
#pragma unroll
        for (int s = 0; s < PL; ++s) {
            const int z = s < len ? s : 0;
            const bool in = w.ok && s < len;
            const double rv = *at(B.r, c, z), qv = *at(B.q, c, z), zv = *at(B.r0, c, z);
            r[c][s] = in ? rv : 0.0;
            p[c][s] = in ? qv : 0.0;
            Z[s * TN + tq] = in ? zv : 0.0;
        }
    }
    // cells of the rows beside the tile: element e is cell e % 2H of plane e / 2H
    int hn[kGridHalo], ht[kGridHalo];
#pragma unroll
    for (int h = 0; h < kGridHalo; ++h) {
        const int e = tid + h * T, s = e / (2 * H), z = e - s * 2 * H;
        const int qh = z < H ? q0 - H + z : q0 + qn + z - H;
        const bool in = s < len && qh >= 0 && qh < g.cyz;
        hn[h] = in ? (i0 + s) * g.cyz + qh : -1;
        ht[h] = s < PL ? s * WP + (z < H ? z : qn + z) : -1;
    }
    // the solve's scalars, the same in every thread
    double alpha = st->alpha, omega = st->omega, beta = st->beta, res = st->res;
    double rho = m0 == 0 ? st->rho[0] : st->rho[(m0 - 1) & 1];
    int mode = st->mode, restarts = st->restarts, done = 0, iter = st->iter, m = m0;

    // Addresses and row coefficients are formed again where they are used: held from
    // iteration to iteration they would not fit the registers
    auto fresh = [&]() {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            asm volatile("" : "+v"(col[c].own), "+v"(col[c].so), "+v"(col[c].zmo), "+v"(col[c].zpo));
            if (!UNI)
                asm volatile("" : "+v"(col[c].ym), "+v"(col[c].yp), "+v"(col[c].zm), "+v"(col[c].zp));
        }
#pragma unroll
        for (int h = 0; h < kGridHalo; ++h) asm volatile("" : "+v"(hn[h]), "+v"(ht[h]));
    };
    // f(c, s) for every cell of the thread; stored: for every one that exists
    auto cells = [&](auto &&f) {
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int s = 0; s < PL; ++s) f(c, s);
    };
    auto stored = [&](auto &&f) {
#pragma unroll
        for (int c = 0; c < NC; ++c)
            if (UNI || col[c].ok) {
#pragma unroll
                for (int s = 0; s < PL; ++s)
                    if (UNI || s < len) f(c, s);
            }
    };
    // the cells along the block's faces
    auto publish = [&](double *v, const double (&u)[NC][PL]) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if ((UNI || col[c].ok) && xlo) put_through(at(v, c, 0), u[c][0]);
            if ((UNI || col[c].ok) && xhi && (UNI || len == PL)) put_through(at(v, c, PL - 1), u[c][PL - 1]);
            if (col[c].yrow) {
#pragma unroll
                for (int s = 0; s < PL; ++s)
                    if (UNI || s < len) put_through(at(v, c, s), u[c][s]);
            }
        }
    };
    auto tell = [&](unsigned long long *slot, double v) {
        unsigned long long u = (unsigned long long)__double_as_longlong(v);
        if (u == kEmpty) u = 0x7ff8000000000000ull;
        __hip_atomic_store(slot, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto empty = [&](unsigned long long *slot) {
        __hip_atomic_store(slot, kEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    // what a thread wrote through has reached memory
    auto written = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
    // One sum's partial from the block's terms, in march order; thread 0 of the last half has
    // it.  The first half of a march block hands its 256 running sums to the second half,
    // which goes on from them: slot k of five (phase A, B, B, C, C).  `faces`: the block has
    // written cells that others read, which have to arrive before its sums do.
    unsigned long long *chain = slots + 5 * nb + (size_t)b * 5 * kThreads;
    auto block_sum = [&](int k, bool faces, auto &&term) -> double {
        int w = tid;
        asm volatile("" : "+v"(w));
        __syncthreads();
        cells([&](int c, int s) {
            lds[s * TN + c * T + w] = UNI ? term(c, s) : keep_if(term(c, s), col[c].ok ? 1 : 0);
        });
        if (faces) written();
        __syncthreads();
        if (tid < kThreads) {
            const int first = d > 0 ? 0 : len - 1;
            double acc = 0.0;
            if (second) {
                unsigned long long v = kEmpty;
                for (int q = 0; q < kMaxPolls && v == kEmpty; ++q)
                    v = __hip_atomic_load(chain + k * kThreads + w, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
                if (v == kEmpty) gave_up = 1;
                acc = __longlong_as_double((long long)v);
            }
#pragma unroll
            for (int u = 0; u < PL; ++u) {
                if (!UNI && u >= len) break;
                const double *z = lds + ((first + d * u) * TN + w);
#pragma unroll
                for (int c = 0; c < TN / kThreads; ++c) acc += z[c * kThreads];
            }
            if (last) {
                acc = wave_fold(acc);
                if ((tid & 63) == 0) red[0][tid >> 6] = acc;
            } else {
                tell(chain + k * kThreads + w, acc);
            }
        }
        __syncthreads();
        return (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
    };
    // empty the chain's slot k again (its next writer waits for this block's next partials)
    auto rest = [&](int k) {
        if (tid < kThreads) empty(chain + k * kThreads + tid);
    };
    // wait for every block's partials of a phase and fold them as fold_partials does
    auto gather = [&](unsigned long long *slot, int ns, double (&t)[2]) -> bool {
        __syncthreads(); // red has been read
        if (tid < kThreads) {
            unsigned long long v[2] = {0, 0};
            if (tid < nb) {
                for (int w = 0; w < kMaxPolls; ++w) {
                    v[0] = __hip_atomic_load(slot + ns * tid, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
                    if (ns == 2)
                        v[1] = __hip_atomic_load(slot + 2 * tid + 1, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
                    if (v[0] != kEmpty && v[1] != kEmpty) break;
                }
                if (v[0] == kEmpty || v[1] == kEmpty) gave_up = 1;
            }
            for (int s = 0; s < ns; ++s) {
                double acc = 0.0;
                acc += __longlong_as_double((long long)v[s]);
                acc = wave_fold(acc);
                if ((tid & 63) == 0) red[s][tid >> 6] = acc;
            }
        }
        __syncthreads();
        t[0] = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
        t[1] = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
        return !gave_up;
    };
    // a vector's plane by plane LDS copy for the stencil: the own cells (e), the rows beside
    // the tile (halo) and the zeros beyond the z walls
    auto stage = [&](auto &&e, auto &&halo) {
#pragma unroll
        for (int c = 0; c < NC; ++c)
            if (UNI || col[c].ok) {
#pragma unroll
                for (int s = 0; s < PL; ++s) lds[col[c].so + s * WP] = e(c, s);
            }
#pragma unroll
        for (int h = 0; h < kGridHalo; ++h)
            if (ht[h] >= 0) lds[ht[h]] = hn[h] >= 0 ? halo(h) : 0.0;
        if (tid < PL) lds[tid * WP + WP - 1] = 0.0;
        __syncthreads();
    };
    // the 7-point sums of the staged vector e (k_march's expression); em, ep: its values on
    // the planes beside the block, zero where there is none.  A missing neighbour is a zero,
    // and its coefficient times it adds a zero: an identity, as the sum starts at +0.0
    auto stencil = [&](auto &&e, const double (&em)[NC], const double (&ep)[NC],
                       double (&out)[NC][PL]) {
        cells([&](int c, int s) {
            const Col &w = col[c];
            const double xm = UNI ? uxm : cx[0][s], xp = UNI ? uxp : cx[1][s];
            const double ym = UNI ? uym : w.ym, yp = UNI ? uyp : w.yp;
            const double zm = UNI ? uzm : w.zm, zp = UNI ? uzp : w.zp;
            double v[7];
            if (UNI) {
                const double dg = w.dg[s == 0 ? 0 : (s == PL - 1 ? 2 : 1)];
                if (PRE) {
                    const RowEnds end = {s == 0 && !xlo ? xm : 0.0,
                                         s == PL - 1 && !xhi ? xp : 0.0,
                                         w.eym, w.eyp, w.ezm, w.ezp};
                    march_offdiag<PRE>(xm, xp, ym, yp, zm, zp, dg, v);
                    v[3] = march_diag<PRE>(end, xm, xp, ym, yp, zm, zp) * dg;
                } else {
                    march_offdiag<PRE>(xm, xp, ym, yp, zm, zp, 0.0, v);
                    v[3] = dg;
                }
            } else {
                const RowEnds end = {s == 0 && !xlo ? xm : 0.0, s == len - 1 && !xhi ? xp : 0.0,
                                     w.eym, w.eyp, w.ezm, w.ezp};
                march_row<PRE>(end, xm, xp, ym, yp, zm, zp, v);
            }
            const double *S = lds + (w.so + s * WP);
            const double n0 = s > 0 ? e(c, s > 0 ? s - 1 : 0) : em[c];
            double n6 = s < PL - 1 ? e(c, s < PL - 1 ? s + 1 : s) : ep[c];
            if (!UNI && s < PL - 1) n6 = s == len - 1 ? ep[c] : n6;
            double z = 0.0;
            z += v[0] * n0;
            z += v[1] * S[-H];
            z += v[2] * S[w.zmo];
            z += v[3] * e(c, s);
            z += v[4] * S[w.zpo];
            z += v[5] * S[H];
            z += v[6] * n6;
            out[c][s] = z;
        });
    };

    double t[2];
    bool fine = true;
    for (;; ++m) {
        fresh();
        // ---- end of iteration m-1, scalars of iteration m
        if (m == 0) {
            mode = 2; // p = r0 (bicgstabRe2.hpp:101-102)
            beta = 0.0;
        } else {
            if (m == m0) {
                if (tid < kThreads) {
                    for (int s = 0; s < 2; ++s) {
                        double acc = 0.0;
                        if (tid < nb) acc += partC[s * nb + tid];
                        acc = wave_fold(acc);
                        if ((tid & 63) == 0) red[s][tid >> 6] = acc;
                    }
                }
                __syncthreads();
                t[0] = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
                t[1] = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
            } else {
                if (!(fine = gather(slotC, 2, t))) break;
                if (last && tid == 0) empty(slotB + 2 * b), empty(slotB + 2 * b + 1);
            }
            if (m == m0 + count) break;
            BicgNext o;
            if (!bicg_next(t, st->norm0, st->tol, st->restart_factor, st->maxit, st->timestep, m,
                           alpha, omega, rho, o)) {
                res = o.res;
                iter = m - 1;
                done = res < st->tol ? 1 : 2;
                break;
            }
            res = o.res;
            iter = m;
            beta = o.beta;
            mode = o.mode;
            rho = t[1];
            if (mode == 1) ++restarts;
        }
        // ---- phase A: p = r + beta q (or r), Ap, (Ap, r0)
        auto form_p = [&](double rv, double qv) { return mode == 0 ? rv + beta * qv : rv; };
        double rm[NC], rp[NC], em[NC], ep[NC], rh[kGridHalo], qh[kGridHalo];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            rm[c] = get_through((const double *)((const char *)B.r + (col[c].own - back)));
            em[c] = get_through((const double *)((const char *)B.q + (col[c].own - back)));
            rp[c] = get_through((const double *)((const char *)B.r + (col[c].own + ahead)));
            ep[c] = get_through((const double *)((const char *)B.q + (col[c].own + ahead)));
        }
#pragma unroll
        for (int h = 0; h < kGridHalo; ++h) {
            rh[h] = get_through(B.r + max(hn[h], 0));
            qh[h] = get_through(B.q + max(hn[h], 0));
        }
        if (mode == 0) cells([&](int c, int s) { p[c][s] = r[c][s] + beta * p[c][s]; });
        else cells([&](int c, int s) { p[c][s] = r[c][s]; });
        if (mode == 1) // restart: r0 = r
            cells([&](int c, int s) { Z[s * TN + c * T + tid] = r[c][s]; });
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            em[c] = xlo ? form_p(rm[c], em[c]) : 0.0;
            ep[c] = xhi ? form_p(rp[c], ep[c]) : 0.0;
        }
        auto pv = [&](int c, int s) { return p[c][s]; };
        stage(pv, [&](int h) { return form_p(rh[h], qh[h]); });
        stencil(pv, em, ep, ap);
        publish(B.ap, ap);
        if (second) rest(3), rest(4); // phase C's of the iteration before
        {
            const double v = block_sum(
                0, true, [&](int c, int s) { return ap[c][s] * Z[s * TN + c * T + tid]; });
            if (last && tid == 0) tell(slotA + b, v);
        }
        if (!(fine = gather(slotA, 1, t))) break;
        if (last && tid == 0 && m > m0) empty(slotC + 2 * b), empty(slotC + 2 * b + 1);
        alpha = rho / t[0]; // a = r1r0 / dot(ap, r0)
        // ---- phase B: s = r - alpha Ap, As, (As, s), (As, As)
        fresh();
        double ah[kGridHalo];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            em[c] = get_through((const double *)((const char *)B.ap + (col[c].own - back)));
            ep[c] = get_through((const double *)((const char *)B.ap + (col[c].own + ahead)));
        }
#pragma unroll
        for (int h = 0; h < kGridHalo; ++h) ah[h] = get_through(B.ap + max(hn[h], 0));
        auto sv = [&](int c, int s) { return r[c][s] - alpha * ap[c][s]; };
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            em[c] = xlo ? rm[c] - alpha * em[c] : 0.0;
            ep[c] = xhi ? rp[c] - alpha * ep[c] : 0.0;
        }
        stage(sv, [&](int h) { return rh[h] - alpha * ah[h]; });
        stencil(sv, em, ep, as);
        {
            const double v0 = block_sum(1, false, [&](int c, int s) { return as[c][s] * sv(c, s); });
            const double v1 = block_sum(2, false, [&](int c, int s) { return as[c][s] * as[c][s]; });
            if (last && tid == 0) {
                written(); // the emptied slot of phase C
                tell(slotB + 2 * b, v0), tell(slotB + 2 * b + 1, v1);
            }
        }
        fresh();
        double xv[NC][PL];
        cells([&](int c, int s) { xv[c][s] = *at(x, c, UNI || s < len ? s : 0); });
        if (!(fine = gather(slotB, 2, t))) break;
        if (last && tid == 0) empty(slotA + b);
        omega = t[0] / t[1]; // w = dot(as, s) / dot(as, as)
        // ---- phase C: x, r, q = p - omega Ap, (r, r), (r, r0)
        cells([&](int c, int s) {
            const double s1 = sv(c, s);
            xv[c][s] = xv[c][s] + (alpha * p[c][s] + omega * s1);
            r[c][s] = s1 - omega * as[c][s];
            p[c][s] = p[c][s] - omega * ap[c][s];
        });
        stored([&](int c, int s) { *at(x, c, s) = xv[c][s]; });
        publish(B.r, r);
        publish(B.q, p);
        if (second) rest(0), rest(1), rest(2);
        {
            const double v0 = block_sum(3, true, [&](int c, int s) { return r[c][s] * r[c][s]; });
            const double v1 = block_sum(
                4, false, [&](int c, int s) { return r[c][s] * Z[s * TN + c * T + tid]; });
            if (last && tid == 0) {
                tell(slotC + 2 * b, v0), tell(slotC + 2 * b + 1, v1);
                partC[b] = v0, partC[nb + b] = v1; // for a launch that goes on from here
            }
        }
    }
    if (!fine) {
        if (tid == 0) *failed = 1;
        return;
    }
    if (m == m0 + count) {
        // the launch's last iteration is m-1: its convergence test (k_bicg_check)
        res = sqrt(t[0]) / st->norm0;
        if (res < st->tol || m - 1 >= st->maxit) {
            done = res < st->tol ? 1 : 2;
            iter = m - 1;
        }
    }
    // the vectors a launch that goes on reads
    stored([&](int c, int s) {
        *at(B.r, c, s) = r[c][s];
        *at(B.q, c, s) = p[c][s];
        *at(B.r0, c, s) = Z[s * TN + c * T + tid];
    });
    if (b == 0 && tid == 0) {
        st->rho[(m - 1) & 1] = rho;
        st->alpha = alpha;
        st->omega = omega;
        st->beta = beta;
        st->mode = mode;
        st->res = res;
        st->iter = iter;
        st->restarts = restarts;
        st->done = done;
    }
}

// ---- launchers ----
// a tile of at most 512 cells: one column a thread, whole march blocks; a larger one: two
// columns of half the planes
static bool grid_halves(const Geo &g) { return g.cyz > 2 * kThreads; }
static int grid_threads(const Geo &g) { return g.cyz <= kThreads ? kThreads : 2 * kThreads; }
static int grid_blocks_of(const Geo &g) { return grid_halves(g) ? 2 * g.nmarch : g.nmarch; }
template <int PRE, bool UNI> static const void *grid_kernel_of(const Geo &g)
{
    if (grid_halves(g)) return (const void *)k_bicg_grid<PRE, 2 * kThreads, 2, kChunk / 2, UNI>;
    if (grid_threads(g) == 2 * kThreads)
        return (const void *)k_bicg_grid<PRE, 2 * kThreads, 1, kChunk, UNI>;
    return (const void *)k_bicg_grid<PRE, kThreads, 1, kChunk, UNI>;
}
static const void *grid_kernel(const Geo &g, int pre, int uni)
{
    if (uni) return pre ? grid_kernel_of<1, true>(g) : grid_kernel_of<0, true>(g);
    return pre ? grid_kernel_of<1, false>(g) : grid_kernel_of<0, false>(g);
}
static size_t grid_lds(const Geo &g)
{
    const int TN = grid_halves(g) ? kTile : grid_threads(g), PL = grid_halves(g) ? kChunk / 2 : kChunk;
    return (size_t)PL * (TN + 2 * g.nzc + 1 + TN) * sizeof(double);
}

int bicg_grid_slots(const Geo &g) { return 5 * g.nmarch * (1 + (grid_halves(g) ? kThreads : 0)); }

// UNI: every row has the same coefficients (element 0 of each axis's), every march block holds
// 8 planes, and every thread's column exists
int bicg_grid_uni(const Geo &g, const double *const (&coef)[3][2])
{
    const int n[3] = {g.nxc, g.nyc, g.nzc};
    for (int a = 0; a < 3; ++a)
        for (int q = 0; q < 2; ++q)
            for (int i = 0; i < n[a]; ++i)
                if (coef[a][q][i] != coef[a][q][0]) return 0;
    return g.nxc % kChunk == 0 &&
           (g.cyz % kTile == 0 || g.cyz == kThreads || g.cyz == 2 * kThreads);
}

int bicg_grid_cus(const Geo &g, int pre, int uni, int &cus)
{
    // one partial per polling thread, the rows beside the tile in kGridHalo cells a thread
    const int PL = grid_halves(g) ? kChunk / 2 : kChunk;
    if (g.nmarch > kThreads || 2 * PL * g.nzc > kGridHalo * grid_threads(g)) return 0;
    int dev = 0, per = 0;
    const void *k = grid_kernel(g, pre, uni);
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, grid_threads(g), grid_lds(g)) !=
            hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    const int blocks = grid_blocks_of(g);
    if ((long long)per * cus < blocks) return 0;
    // workgroups are dealt to the 8 XCDs in turn, so the blocks of one count as those of the
    // fullest; more than one a CU leave no room beside them
    return std::min((blocks + 7) / 8 * 8, cus);
}

hipError_t launch_bicg_grid(const Geo &g, hipStream_t s, int pre, int uni, BicgBuffers &B,
                            double *x, double *partC, unsigned long long *slots, KState *st,
                            KState *keep, int *failed, int give_up, int m0, int count)
{
    const int n = bicg_grid_slots(g);
    hipLaunchKernelGGL(k_grid_slots, dim3((n + 255) / 256), dim3(256), 0, s, n, slots,
                       (const KState *)st, m0 == 0 ? keep : nullptr);
    Geo geo = g;
    BicgBuffers buf = B;
    void *args[] = {&geo, &buf, &x, &partC, &slots, &st, &failed, &give_up, &m0, &count};
    return hipLaunchKernel(grid_kernel(g, pre, uni), dim3(grid_blocks_of(g)),
                           dim3(grid_threads(g)), args, grid_lds(g), s);
}

} // namespace cfdmx
