// cfdmx_sor.hip -- red-black SOR of the uniform grid, two sweeps in one pass over memory.
#include "cfdmx_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace cfdmx {

static inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// ---------------------------------------------------------------------------
// Two sweeps (red, black, red, black) of SorPipeLine_seq (SorPipeLine.seq.hpp:40-123) on
// p's natural ghosted order, from src to dst (the ghosts of both hold the last boundary
// values, fixed during the solve).  A block owns a tile of rows by pairs of k of a span of
// planes i and marches along i; a thread holds one column of pairs (k, k + 1), one cell of
// each colour.  In step t it takes plane t in and runs the four half sweeps one plane
// behind each other: red on plane t - 1, black on t - 2, red on t - 3, black on t - 4, which
// is then done and written.  The x neighbours are the thread's own registers, the y and z
// neighbours other threads' values of the step before (LDS, two buffers, one barrier a
// step).  Around the tile four rows, two pairs and four planes are computed again, each half
// sweep as far out as the next needs it.
//
// The values, operations and their order are k_sor_half's, and max |dp| of each sweep is
// exact in any order, so the results are the same bits.
//
// Bound by memory at the large end: by the counters a pass moves 33 bytes a cell at 512x256x64
// (25 read, of which 16 are p and the right-hand side and the rest the planes around the tiles;
// 8 written) where four half sweeps moved 65.  A sweep of a solve of 401, half sweeps and then
// passes: 512x256x64 52.9 and 27.1 us (a pass 53, 5.3 TB/s), 420x210x72 48.7 and 24.3, 256x128x128 30.7 and 19.7, 256x128x32 20.9 and
// 10.8, 64x40x8 12.3 and 6.4, 40x24x4 13.1 and 5.7 us (twelve steps of 0.5 us and a launch).
// 1024 threads (102 registers): tiles of 32 rows lose a quarter to the halo, of 16 rows a half.
// All neighbours read ahead of the four half sweeps spill (128 registers): 27.5 us at
// 512x256x64.  The pass before is counted by each block of the next one: a launch of its own
// for that cost 1.0 us a sweep at 64x40x8.
// ---------------------------------------------------------------------------
constexpr int kSorThreads = 1024;

__device__ __forceinline__ double sor_pick(bool c, double a, double b) { return c ? a : b; }

// the state after a pass: its two sweeps' max |dp|, from the blocks' in part, counted one
// after the other (all threads of the block; red: two values a wave)
__device__ __forceinline__ SorState sor_advance(SorState st, const double *part, int nb,
                                                double *red)
{
    const int t = threadIdx.x, T = blockDim.x, waves = T >> 6;
    double m1 = 0.0, m2 = 0.0;
    for (int m = t; m < nb; m += T) {
        m1 = part[m] > m1 ? part[m] : m1;
        m2 = part[nb + m] > m2 ? part[nb + m] : m2;
    }
    m1 = wave_max(m1);
    m2 = wave_max(m2);
    if ((t & 63) == 0) {
        red[t >> 6] = m1;
        red[waves + (t >> 6)] = m2;
    }
    __syncthreads();
    for (int s = 0; s < 2 && !st.done; ++s) {
        double m = red[s * waves];
        for (int w = 1; w < waves; ++w) m = red[s * waves + w] > m ? red[s * waves + w] : m;
        st.residual = m;
        st.iters += 1;
        st.done = !(m > st.tol && st.iters < st.itmax);
    }
    __syncthreads();
    return st;
}

__global__ void __launch_bounds__(kSorThreads)
k_sor_pass(Geo g, SorPlan pl, double omega, SorCoef sc, const double *__restrict__ rhs,
           const double *__restrict__ src, double *__restrict__ dst, SorTurn turn)
{
    const int L = logical_block(g);
    if (L >= pl.blocks) return;
    extern __shared__ double lds[];
    const int sweeps = turn.sweeps;
    const int T = blockDim.x, t = threadIdx.x;
    const int tz = L % pl.ntz, ty = (L / pl.ntz) % pl.nty, tx = L / (pl.ntz * pl.nty);
    const int hz = g.nzc >> 1;
    const int x0 = tx * pl.xlen, x1 = min(x0 + pl.xlen, g.nxc);
    const int y0 = ty * pl.yown, y1 = min(y0 + pl.yown, g.nyc);
    const int rlo = max(y0 - 4, -1), rhi = min(y1 + 4, g.nyc + 1);
    const int c0 = tz * pl.cown, c1 = min(c0 + pl.cown, hz);
    const bool whole = pl.ntz == 1;
    const int clo = whole ? (g.zper ? 0 : -1) : c0 - 2;

    const int r = t / pl.width, c = t - r * pl.width;
    const int row = rlo + r, rows = rhi - rlo;
    int col = clo + c;
    const bool own_col = col >= c0 && col < c1;
    if (g.zper) col = col < 0 ? col + hz : col >= hz ? col - hz : col;
    const bool inner =
        r < rows && row >= 0 && row < g.nyc && col >= 0 && col < hz;
    const bool own = inner && own_col && row >= y0 && row < y1;
    bool need[5];
#pragma unroll
    for (int s = 1; s <= 4; ++s)
        need[s] = inner && row >= y0 - (4 - s) && row < y1 + (4 - s);
    int offP = t, offM = t, offN = t, offS = t;
    if (r < rows) {
        const bool circ = whole && g.zper;
        offP = c + 1 < pl.width ? t + 1 : circ ? t - c : t;
        offM = c > 0 ? t - 1 : circ ? t + pl.width - 1 : t;
        offN = r + 1 < rows ? t + pl.width : t;
        offS = r > 0 ? t - pl.width : t;
    }
    // threads beside the tile read (and drop) the nearest value there is
    const int rowc = min(max(row, -1), g.nyc), colc = min(max(col, -1), hz);
    const int rowi = min(max(row, 0), g.nyc - 1), coli = min(max(col, 0), hz - 1);
    const double *pin = src + (rowc + kGC) * g.sy + 2 * colc + kGC;
    const double *fin = rhs + rowi * g.nzc + 2 * coli;
    double *pout = dst + (rowc + kGC) * g.sy + 2 * colc + kGC;

    double2 pp[3], pf[3];
    double B0[3], R0[3], R1[3], B1[3], R2[3], rr[3], rb[3];
#pragma unroll
    for (int u = 0; u < 3; ++u)
        B0[u] = R0[u] = R1[u] = B1[u] = R2[u] = rr[u] = rb[u] = 0.0;
    const auto load = [&](int u, int i) { // plane i of p and plane i - 1 of the right-hand side
        const int ip = min(max(i, -1), g.nxc) + kGC;
        const int ir = min(max(i - 1, 0), g.nxc - 1);
        pp[u] = *reinterpret_cast<const double2 *>(pin + ip * g.sx);
        pf[u] = *reinterpret_cast<const double2 *>(fin + ir * g.cyz);
    };
    double mx1 = 0.0, mx2 = 0.0;
    // one half sweep of plane i: the new value of a cell of value v
    const auto half = [&](int s, int i, const double *sh, int zoff, bool q, double E, double o,
                          double W, double v, double f, double &mx) -> double {
        if (i < max(0, x0 - (4 - s)) || i >= min(g.nxc, x1 + (4 - s))) return v;
        if (s > 2 && sweeps == 1) return v;
        if (!need[s]) return v;
        const double N = sh[offN], S = sh[offS], z = sh[zoff];
        const double pT = sor_pick(q, z, o), pB = sor_pick(q, o, z);
        const double pNEW = (-E * sc.c[0] - W * sc.c[1] - N * sc.c[2] - S * sc.c[3] -
                             pT * sc.c[4] - pB * sc.c[5] + f) *
                            sc.c[6];
        if (i >= x0 && i < x1) {
            const double d = fabs(pNEW - v);
            mx = d > mx ? d : mx;
        }
        return v + omega * (pNEW - v);
    };
    const auto step = [&](auto U, int i) {
        constexpr int p0 = U, p1 = (U + 2) % 3, p2 = (U + 1) % 3; // planes i, i - 1, i - 2
        const bool q0 = ((i + row) & 1) != 0, q = !q0;
        const double *was = lds + ((i - 1) & 1) * 4 * T;
        double *now = lds + (i & 1) * 4 * T;
        const int zoff = q ? offP : offM;
        R0[p0] = sor_pick(q0, pp[p0].y, pp[p0].x);
        B0[p0] = sor_pick(q0, pp[p0].x, pp[p0].y);
        const double rb4 = rb[p1]; // the black right-hand side of plane i - 4
        rr[p1] = sor_pick(q, pf[p0].y, pf[p0].x);
        rb[p1] = sor_pick(q, pf[p0].x, pf[p0].y);
        load(p0, i + 3);
        R1[p1] = half(1, i - 1, was, zoff, q, B0[p0], B0[p1], B0[p2], R0[p1], rr[p1], mx1);
        B1[p2] = half(2, i - 2, was + T, zoff, q, R1[p1], R1[p2], R1[p0], B0[p2], rb[p2], mx1);
        R2[p0] = half(3, i - 3, was + 2 * T, zoff, q, B1[p2], B1[p0], B1[p1], R1[p0], rr[p0],
                      mx2);
        const double B2 =
            half(4, i - 4, was + 3 * T, zoff, q, R2[p0], R2[p1], R2[p2], B1[p1], rb4, mx2);
        if (i >= x0 + 4 && own)
            *reinterpret_cast<double2 *>(pout + (i - 4 + kGC) * g.sx) =
                make_double2(sor_pick(q0, B2, R2[p1]), sor_pick(q0, R2[p1], B2));
        now[t] = B0[p0];
        now[T + t] = R1[p1];
        now[2 * T + t] = B1[p2];
        now[3 * T + t] = R2[p0];
        __syncthreads();
    };
    const int first = max(x0 - 4, -1), last = x1 + 3;
#pragma unroll
    for (int u = 0; u < 3; ++u) load(u, first + u);
    // every block counts the pass before this one, the first block for the passes to come
    if (sweeps == 2) {
        SorState st = *turn.in;
        if (st.done == 0 && turn.was) st = sor_advance(st, turn.was, pl.blocks, lds);
        if (L == 0 && t == 0) *turn.out = st;
        if (st.done) return;
    }
    for (int i = first; i <= last; i += 3) {
        step(std::integral_constant<int, 0>{}, i);
        if (i + 1 > last) break;
        step(std::integral_constant<int, 1>{}, i + 1);
        if (i + 2 > last) break;
        step(std::integral_constant<int, 2>{}, i + 2);
    }

    mx1 = wave_max(own ? mx1 : 0.0);
    mx2 = wave_max(own ? mx2 : 0.0);
    if ((t & 63) == 0) {
        lds[t >> 6] = mx1;
        lds[16 + (t >> 6)] = mx2;
    }
    __syncthreads();
    if (t < 2) {
        double m = 0.0;
        for (int w = 0; w < T >> 6; ++w) m = lds[16 * t + w] > m ? lds[16 * t + w] : m;
        turn.part[t * pl.blocks + L] = m;
    }
}

__global__ void __launch_bounds__(kThreads)
k_sor_pass_fin(const SorState *in, const double *part, int nb, SorState *out)
{
    __shared__ double red[2 * kThreads / 64];
    SorState st = *in;
    if (!st.done) st = sor_advance(st, part, nb, red);
    if (threadIdx.x == 0) *out = st;
}

// Tiles for grids of one spacing an axis (other grids' coefficients cost seven divisions a cell,
// which the half sweeps do once a sweep and the halo would do again) and an even nz;
// on these the pass was 1.5 to 2.3 times as fast as the half sweeps at every size measured
// (40x24x4 to 512x256x64).  Rows of pairs are cut where that leaves the least to do: all
// threads of all rounds of blocks, times their steps.
SorPlan sor_plan(const Geo &g, const SorCoef &sc, int cus)
{
    SorPlan best = {};
    if (!sc.constant || g.nzc % 2) return best;
    const int hz = g.nzc >> 1;
    long long least = 0;
    for (int n = 1; n <= (hz + 7) / 8; ++n) { // pieces of a row's pairs
        SorPlan p = {};
        p.ntz = n;
        p.cown = cdiv(hz, n);
        if ((n - 1) * p.cown >= hz) continue;
        p.width = n > 1 ? p.cown + 4 : g.zper ? hz : hz + 2;
        const int most = kSorThreads / p.width; // rows of a block
        if (most < 12 && most < g.nyc + 2) continue;
        p.nty = g.nyc + 2 <= most ? 1 : cdiv(g.nyc, most - 8);
        p.yown = cdiv(g.nyc, p.nty);
        p.nty = cdiv(g.nyc, p.yown);
        const int rows = p.nty == 1 ? g.nyc + 2 : std::min(p.yown + 8, g.nyc + 2);
        p.threads = cdiv(rows * p.width, 64) * 64;
        const int tiles = p.nty * p.ntz, room = cus * (kSorThreads / p.threads);
        p.ntx = std::max(1, std::min(room / tiles, cdiv(g.nxc, 4)));
        p.xlen = std::max(4, cdiv(g.nxc, p.ntx));
        p.ntx = cdiv(g.nxc, p.xlen);
        p.blocks = tiles * p.ntx;
        // steps of the blocks that share a CU, one round after the other
        const long long cost = (long long)cdiv(p.blocks, room) * (p.xlen + 8) *
                               (kSorThreads / p.threads) * p.threads;
        if (!best.blocks || cost < least) {
            best = p;
            least = cost;
        }
    }
    return best;
}

void launch_sor_pass(const Geo &g, hipStream_t s, const SorPlan &pl, double omega,
                     const SorCoef &sc, const double *rhs, const double *src, double *dst,
                     const SorTurn &turn)
{
    const int grid = g.xcd_remap ? (pl.blocks + 7) / 8 * 8 : pl.blocks;
    hipLaunchKernelGGL(k_sor_pass, dim3(grid), dim3(pl.threads),
                       (size_t)8 * pl.threads * sizeof(double), s, g, pl, omega, sc, rhs, src,
                       dst, turn);
}

void launch_sor_pass_fin(hipStream_t s, const SorPlan &pl, const SorState *in,
                         const double *part, SorState *out)
{
    hipLaunchKernelGGL(k_sor_pass_fin, dim3(1), dim3(kThreads), 0, s, in, part, pl.blocks, out);
}

} // namespace cfdmx
