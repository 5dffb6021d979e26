// cfdmx_mg_sweep.hpp -- the two halves of a V(2,2) cycle on one multigrid level with even
// nz, each as one kernel that passes over the level once.
//
// Down: the first red-black sweep from u = 0, the second sweep, the residual and its
// restriction.  Up: the coarse correction added, then two red-black sweeps.  Four half
// sweeps each depend on the other colour's neighbours one cell away, so a pass over the
// level in x can carry all of them at once, one plane apart: while plane i gets its first
// half sweep, plane i-1 gets the second, i-2 the third, i-3 the fourth and i-4 its residual.
// A block owns `ty` rows of y (whole rows of z, or `tz` pairs of long ones) on `cxl` planes
// of x and forms again the cells of the 4 rows, 4 planes and 2 pairs around them that its own
// depend on, so no block waits for another and every value is the one the separate half
// sweeps would give.
//
// A thread keeps P z-pairs (cells 2kk and 2kk+1) of one row through all planes.  Its x
// neighbours are its own values of the planes before and after, one of its two z
// neighbours is the other cell of its pair; the y neighbours and the other z neighbour
// come from LDS, where each half sweep leaves its half plane (one colour) in one of two
// slots: a step reads the slots written the step before, so one barrier per plane orders
// all of it.  Rows and planes outside the level hold zeros, which stand for the missing
// neighbours (weight 0): adding +0 changes no sum, since every sum starts at +0.
//
// What bounds it: the separate kernels moved 8 half sweeps of the level through memory per
// cycle and half, at a launch each; here the down half reads f and writes the black half of
// u (the red half is formed again by the up half without being read) and the coarse f, the
// up half reads those and writes u.  The arithmetic (about 20 instructions a cell and half
// sweep, the halo's on top) then takes longer than the memory does.
#pragma once
#include "cfdmx_internal.hpp"

#include <type_traits>

namespace cfdmx {

constexpr int kMGHalo = 4;          // rows and planes a block forms again on each side
constexpr int kMGSweepThreads = 512; // largest block of the sweep kernels

// a / b from r = RN(1/b), correctly rounded (see divr) where the corrections' residuals and
// the quotient have no subnormal part; r = 0 gives 0
__device__ __forceinline__ double mg_quot(double a, double b, double r)
{
    double q = a * r;
    double t = __builtin_fma(q, b, -a);
    q = __builtin_fma(-t, r, q);
    t = __builtin_fma(q, b, -a);
    return __builtin_fma(-t, r, q);
}
__device__ __forceinline__ float mg_quot(float a, float b, float r)
{
    float q = a * r;
    float t = __builtin_fmaf(q, b, -a);
    q = __builtin_fmaf(-t, r, q);
    t = __builtin_fmaf(q, b, -a);
    return __builtin_fmaf(-t, r, q);
}

// P values moved as one vector (all addresses are multiples of P values)
template <typename T, int P> struct alignas(sizeof(T) * P <= 16 ? sizeof(T) * P : 16) MGVec {
    T v[P];
};
template <typename T, int P>
__device__ __forceinline__ void mg_get(const T *s, T (&u)[P])
{
    const MGVec<T, P> v = *reinterpret_cast<const MGVec<T, P> *>(s);
#pragma unroll
    for (int q = 0; q < P; ++q) u[q] = v.v[q];
}
template <typename T, int P>
__device__ __forceinline__ void mg_put(T *s, const T (&u)[P])
{
    MGVec<T, P> v;
#pragma unroll
    for (int q = 0; q < P; ++q) v.v[q] = u[q];
    *reinterpret_cast<MGVec<T, P> *>(s) = v;
}

// LDS row: the pairs of one colour and a zero entry behind them for the z walls
template <int P> __host__ __device__ inline int mg_lds_row(int pairs) { return pairs + P; }

// pairs a block forms again on each side of a part of a row: 4 cells, in whole columns
template <int P> __host__ __device__ constexpr int mg_zhalo() { return P > 2 ? P : 2; }

// threads of a block: those of the even rows, then those of the odd rows, each a multiple
// of a wave, so that a wave's cells of one colour and plane have k of one parity
__host__ __device__ inline int mg_half_block(int rows, int tpr)
{
    return (rows / 2 * tpr + 63) / 64 * 64;
}

// the diagonal d of a plane's cells, r = RN(1/d); walls: dz, rz with one z neighbour
// missing.  r = 0 outside the level, which makes every value there 0
template <typename T> struct MGDiag {
    T d, r, dz, rz;
};

// What a thread knows of its block and of its P z-pairs of one row.
template <typename T, int P, bool ZPER> struct MGCol {
    int x0, x1;           // planes of the block
    int j, jc, row;       // row of the level (jc: held inside it) and of the block
    int kk0, lk;          // first pair, in the level's row and in the block's
    // has a row of the block; its cells are cells of the level; its results leave the block
    bool live, in_level, mine;
    int own, ym, yp;      // LDS offsets: own pairs, the rows beside
    int zoff[2];          // LDS offset of the z neighbour outside its pairs, by parity of k
    bool zlo, zhi;        // walls: its pairs touch k = 0 / k = nz - 1
    MGDiag<T> in, edge;   // planes with both x neighbours / with one (or none: nx = 1)
    int par0;             // parity of k of the red cells of plane x0 - kMGHalo (wave-uniform)

    __device__ __forceinline__ bool init(const MGSweepT<T> &a)
    {
        // consecutive blocks (neighbouring row tiles of one chunk) on one XCD, whose L2
        // then serves the rows that both read
        const int per = (a.nblk + 7) >> 3;
        const int b = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
        if (b >= a.nblk) return false;
        const int rest = b / a.nkt, kt = b - rest * a.nkt;
        const int chunk = rest / a.njt, jt = rest - chunk * a.njt;
        x0 = chunk * a.cxl;
        x1 = min(x0 + a.cxl, a.nx);
        const int H = mg_half_block(a.rows, a.tpr), t = threadIdx.x;
        const int odd = t >= H ? 1 : 0, th = t - odd * H;
        const int rr = th / a.tpr;
        live = rr < a.rows / 2;
        row = live ? 2 * rr + odd : odd;
        lk = live ? (th - rr * a.tpr) * P : 0;
        j = jt * a.ty - kMGHalo + row;
        jc = min(max(j, 0), a.ny - 1);
        in_level = live && j == jc;
        mine = in_level && row >= kMGHalo && row < kMGHalo + a.ty;
        const int W = mg_lds_row<P>(a.pairs);
        own = row * W + lk;
        ym = (row > 0 ? row - 1 : row) * W + lk;
        yp = (row < a.rows - 1 ? row + 1 : row) * W + lk;
        if (a.nkt == 1) {
            const int zero = a.pairs;
            kk0 = lk;
            zoff[0] = kk0 > 0 ? own - 1 : (ZPER ? row * W + a.half - 1 : zero);
            zoff[1] = kk0 + P < a.half ? own + P : (ZPER ? row * W : zero);
        } else {
            // part of a row: beyond its ends the pairs of the wrapped row, or none (zeros)
            constexpr int Z = mg_zhalo<P>();
            const int k = kt * a.tz - Z + lk;
            if (ZPER) {
                kk0 = k < 0 ? k + a.half : k % a.half;
            } else {
                kk0 = min(max(k, 0), a.half - P);
                in_level = in_level && kk0 == k;
            }
            mine = mine && lk >= Z && lk < Z + a.tz && k < a.half;
            zoff[0] = lk > 0 ? own - 1 : own;
            zoff[1] = lk + P < a.pairs ? own + P : own;
        }
        const bool jin = in_level;
        zlo = kk0 == 0;
        zhi = kk0 + P == a.half;
        // jt * ty and kMGHalo are even, so j and row have the same parity
        par0 = (x0 - kMGHalo + odd) & 1;
        // the diagonal in the order of mg_diag
        auto diag = [&](int nxn, bool zmiss) {
            T d = (T)0;
            for (int q = 0; q < nxn; ++q) d += a.cx;
            if (j > 0) d += a.cy;
            if (j < a.ny - 1) d += a.cy;
            if (ZPER) {
                d += (T)2 * a.cz;
            } else {
                d += a.cz;
                if (!zmiss) d += a.cz;
            }
            return d;
        };
        auto both = [&](int nxn) {
            MGDiag<T> m;
            m.d = diag(nxn, false);
            m.r = jin ? (T)1 / m.d : (T)0;
            m.dz = ZPER ? (T)0 : diag(nxn, true);
            m.rz = ZPER || !jin ? (T)0 : (T)1 / m.dz;
            return m;
        };
        in = both(2);
        edge = both(a.nx > 1 ? 1 : 0);
        return true;
    }

    __device__ __forceinline__ MGDiag<T> plane(const MGSweepT<T> &a, int i) const
    {
        const bool inside = i > 0 && i < a.nx - 1, some = i >= 0 && i < a.nx;
        const T d0 = in.d, d1 = edge.d, r0 = in.r, r1 = some ? edge.r : (T)0;
        MGDiag<T> m;
        m.d = inside ? d0 : d1;
        m.r = inside ? r0 : r1;
        if (ZPER) {
            m.dz = m.rz = (T)0;
        } else {
            const T dz0 = in.dz, dz1 = edge.dz, rz0 = in.rz, rz1 = some ? edge.rz : (T)0;
            m.dz = inside ? dz0 : dz1;
            m.rz = inside ? rz0 : rz1;
        }
        return m;
    }

    // (f + s) / d at pair q for a cell of parity PAR; d is returned too.  EXACT: by division;
    // else `least` takes the magnitude of a dividend other than zero (as ordered bits, float)
    template <int PAR, bool EXACT>
    __device__ __forceinline__ T quot(const MGDiag<T> &m, int q, T v, T &d, unsigned &least) const
    {
        T r = m.r;
        d = m.d;
        if (!ZPER && ((PAR == 0 && q == 0) || (PAR == 1 && q == P - 1))) {
            const bool miss = PAR == 0 ? zlo : zhi;
            const T rz = m.rz, dz = m.dz;
            r = miss ? rz : r;
            d = miss ? dz : d;
        }
        if constexpr (EXACT) return r != (T)0 ? v / d : (T)0;
        if constexpr (std::is_same<T, float>::value)
            least = min(least, 2u * __float_as_uint(v) - 1u);
        return mg_quot(v, d, r);
    }

    // The neighbour sums of a plane at a thread's cells of one colour, in the order -x, +x,
    // -y, +y, -z, +z of mg_nbsum.  S: the slot with the other colour's half plane; xm, xp:
    // cx times the x neighbours; mate: the other colour's cells of the same pairs; PAR:
    // parity of k of the cells.
    template <int PAR>
    __device__ __forceinline__ void sum(const MGSweepT<T> &a, const T *S, const T (&xm)[P],
                                        const T (&xp)[P], const T (&mate)[P], T (&s)[P]) const
    {
        T vm[P], vp[P];
        mg_get(S + ym, vm);
        mg_get(S + yp, vp);
        const T l = S[zoff[PAR]];
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const T zm = PAR ? mate[q] : (q > 0 ? mate[q > 0 ? q - 1 : 0] : l);
            const T zp = PAR ? (q < P - 1 ? mate[q < P - 1 ? q + 1 : q] : l) : mate[q];
            T t = xm[q] + xp[q];
            t += a.cy * vm[q];
            t += a.cy * vp[q];
            t += a.cz * zm;
            t += a.cz * zp;
            s[q] = t;
        }
    }
};

// planes that the inputs are loaded ahead: three, or one where a plane's are so many that
// more would spill registers (P = 4 in float and P = 2 in double at 512x256x64: three
// planes ahead the up kernel spilled and took 62 and 112 us, one plane ahead 24 and 36 us; what
// still spills at one plane is in the comment of mg_pairs)
template <typename T, int P> __host__ __device__ constexpr int mg_ahead()
{
    return sizeof(T) * P >= 16 ? 1 : 3;
}

template <int V> struct MGInt {
    static constexpr int v = V;
};

#define MG_INLINE __attribute__((always_inline))

// A float dividend below a.tiny gives mg_quot a subnormal part.  A right-hand side of ordinary
// size has none, so a block divides only in a second pass over its cells, if one of its threads
// met such a dividend in the first; the results are then written again.  Steps of 39 grids took
// 4% less to 3% more with the look at the dividends (nothing in the mean), 3 to 11% more with a
// branch at every quotient.  In double such a value is 2^-400 times the largest of a residual
// whose norm does not underflow, and is not looked for.
template <typename T, class Pass> __device__ __forceinline__ void mg_exactly(Pass &&pass)
{
    if (!pass(std::false_type())) return;
    __syncthreads(); // the flag has been read
    pass(std::true_type());
}
// whether a thread of the block met a small dividend.  flag: an entry of LDS that the last step
// of a pass, which no barrier follows, neither reads nor writes; its zero is the zero behind a
// row.  (Four bytes of LDS of its own took a CU's second block from the largest tiles: a step of
// 1024x512x128 cells 21.4 -> 28.0 ms.)
template <typename T, bool EXACT>
__device__ __forceinline__ bool mg_small(const MGSweepT<T> &a, unsigned least, T *flag)
{
    if constexpr (EXACT || !std::is_same<T, float>::value) return false;
    if (least < 2u * __float_as_uint((float)a.tiny) - 1u) *flag = (T)1;
    __syncthreads();
    return *flag != (T)0;
}

// GEN: 0 = z-only coarsening (fx = fy = 1, fz = 2); 1 = any other, by the factors in a
template <typename T, int P, bool ZPER, int GEN, bool EXACT>
__device__ __forceinline__ bool mg_down(const MGSweepT<T> &a, const MGCol<T, P, ZPER> &c)
{
    extern __shared__ double mg_lds[];
    unsigned least = ~0u;
    const int SL = a.rows * mg_lds_row<P>(a.pairs);
    // half planes of the four half sweeps, two slots each: first red and black, second red
    // and black
    T *const L1 = reinterpret_cast<T *>(mg_lds), *const L2 = L1 + 2 * SL, *const L3 = L2 + 2 * SL,
            *const L4 = L3 + 2 * SL;
    T *const E = L4 + 2 * SL; // GEN: residuals of the odd rows, two slots
    const int EW = 2 * a.pairs, EL = a.rows * EW;
    for (int q = threadIdx.x; q < 8 * SL; q += blockDim.x) L1[q] = (T)0;
    const int fplane = a.ny * a.nz, foff = c.jc * a.nz + 2 * c.kk0;
    // the planes a step still needs, by plane index modulo 4 (mod 2): f as loaded (three
    // planes ahead) and by colour, diagonals, cx times the half sweeps' results
    T fl[4][2 * P], fr[4][P] = {}, fb[4][P] = {};
    MGDiag<T> dg[4] = {};
    T xr1[2][P] = {}, xb1[2][P] = {}, xr2[2][P] = {}, xb2[2][P] = {};
    // results of the step before: each the pair mates of the next half sweep's cells
    T r1m[P] = {}, b1m[P] = {}, r2m[P] = {}, b2m[P] = {}, r2o[P] = {}, rb[P] = {};
    T rz[2 * P] = {}, acc[2 * P] = {}; // GEN: residuals of the plane before, restriction sums
    auto load = [&](int i, T (&v)[2 * P]) MG_INLINE {
        const int ic = min(max(i, 0), a.nx - 1);
        mg_get(a.f + (size_t)ic * fplane + foff, v);
    };
    const int first = c.x0 - kMGHalo, steps = c.x1 - c.x0 + 2 * kMGHalo + (GEN ? 1 : 0);
    constexpr int D = mg_ahead<T, P>();
#pragma unroll
    for (int q = 0; q < D; ++q) load(first + q, fl[q]);
    __syncthreads();
    // step S (modulo 4) of plane i; PAR: parity of k of plane i's red cells, which is also
    // that of plane i-1's black ones, plane i-2's red ones and so on
    auto step = [&](auto S_, auto PAR_, int i) MG_INLINE {
        constexpr int S = decltype(S_)::v, PAR = decltype(PAR_)::v;
        constexpr int e = S & 1, o = e ^ 1;
        constexpr int m1 = (S + 3) & 3, m2 = (S + 2) & 3, m3 = (S + 1) & 3;
        const MGDiag<T> d4 = dg[S];
        T f4[P];
#pragma unroll
        for (int q = 0; q < P; ++q) {
            f4[q] = fr[S][q];
            fr[S][q] = fl[S][2 * q + PAR];
            fb[S][q] = fl[S][2 * q + 1 - PAR];
        }
        load(i + D, fl[(S + D) & 3]);
        dg[S] = c.plane(a, i);
        T d, s[P];
        // plane i: red = f / d
        T r1[P], x1[P];
#pragma unroll
        for (int q = 0; q < P; ++q) {
            r1[q] = c.template quot<PAR, EXACT>(dg[S], q, fr[S][q], d, least);
            x1[q] = a.cx * r1[q];
        }
        if (c.live) mg_put(L1 + e * SL + c.own, r1);
        // plane i-1: black
        T b1[P], x2[P];
        c.template sum<PAR>(a, L1 + o * SL, xr1[e], x1, r1m, s);
#pragma unroll
        for (int q = 0; q < P; ++q) {
            b1[q] = c.template quot<PAR, EXACT>(dg[m1], q, fb[m1][q] + s[q], d, least);
            x2[q] = a.cx * b1[q];
            xr1[e][q] = x1[q];
            r1m[q] = r1[q];
        }
        if (c.live) mg_put(L2 + o * SL + c.own, b1);
        // plane i-2: red
        T r2[P], x3[P];
        c.template sum<PAR>(a, L2 + e * SL, xb1[o], x2, b1m, s);
#pragma unroll
        for (int q = 0; q < P; ++q) {
            r2[q] = c.template quot<PAR, EXACT>(dg[m2], q, fr[m2][q] + s[q], d, least);
            x3[q] = a.cx * r2[q];
            xb1[o][q] = x2[q];
            b1m[q] = b1[q];
        }
        if (c.live) mg_put(L3 + e * SL + c.own, r2);
        // plane i-3: black, and its residual f - (d u - s) from the same sum
        T b2[P], x4[P], rbn[P];
        c.template sum<PAR>(a, L3 + o * SL, xr2[e], x3, r2m, s);
#pragma unroll
        for (int q = 0; q < P; ++q) {
            b2[q] = c.template quot<PAR, EXACT>(dg[m3], q, fb[m3][q] + s[q], d, least);
            x4[q] = a.cx * b2[q];
            rbn[q] = fb[m3][q] - (d * b2[q] - s[q]);
            xr2[e][q] = x3[q];
        }
        if (c.live) mg_put(L4 + o * SL + c.own, b2);
        const int i3 = i - 3, i4 = i - 4;
        if (c.mine && i3 >= c.x0 && i3 < c.x1)
            mg_put(a.ub + (size_t)i3 * (a.ny * a.half) + (c.j * a.half + c.kk0), b2);
        // plane i-4: residual of the red cells, restriction
        T rzn[2 * P];
        if (c.mine && i4 >= c.x0 && i4 < c.x1) {
            c.template sum<PAR>(a, L4 + e * SL, xb2[o], x4, b2m, s);
#pragma unroll
            for (int q = 0; q < P; ++q) {
                const T dz4 = d4.dz;
                T dd = d4.d;
                if (!ZPER && ((PAR == 0 && q == 0) || (PAR == 1 && q == P - 1)))
                    dd = (PAR == 0 ? c.zlo : c.zhi) ? dz4 : dd;
                rzn[2 * q + PAR] = f4[q] - (dd * r2o[q] - s[q]);
                rzn[2 * q + 1 - PAR] = rb[q];
            }
            if (GEN == 0) {
                T out[P];
#pragma unroll
                for (int q = 0; q < P; ++q) out[q] = (((T)0 + rzn[2 * q]) + rzn[2 * q + 1]) / (T)2;
                mg_put(a.fc + (size_t)i4 * (a.ny * a.half) + (c.j * a.half + c.kk0), out);
            } else if (a.fy == 2 && (c.j & 1)) {
                mg_put(E + e * EL + c.row * EW + 2 * c.lk, rzn);
            }
        }
        if (GEN) {
            // plane i-5, whose odd rows' residuals were left in LDS the step before:
            // children in the order x, y, z
            const int ie = i - 5;
            if (c.mine && (a.fy == 1 || !(c.j & 1)) && ie >= c.x0 && ie < c.x1) {
                if (a.fx == 1 || !(ie & 1)) {
#pragma unroll
                    for (int q = 0; q < 2 * P; ++q) acc[q] = (T)0;
                }
                auto add = [&](const T (&v)[2 * P]) MG_INLINE {
#pragma unroll
                    for (int q = 0; q < P; ++q) {
                        acc[2 * q] += v[2 * q];
                        if (a.fz == 2) acc[2 * q] += v[2 * q + 1];
                        else acc[2 * q + 1] += v[2 * q + 1];
                    }
                };
                add(rz);
                if (a.fy == 2) {
                    T v[2 * P];
                    mg_get(E + o * EL + (c.row + 1) * EW + 2 * c.lk, v);
                    add(v);
                }
                if (a.fx == 1 || (ie & 1)) {
                    const T w = (T)(a.fx * a.fy * a.fz); // a power of two
                    const size_t ro =
                        ((size_t)(ie >> (a.fx >> 1)) * a.cny + (c.j >> (a.fy >> 1))) * a.cnz;
                    if (a.fz == 2) {
                        T out[P];
#pragma unroll
                        for (int q = 0; q < P; ++q) out[q] = acc[2 * q] / w;
                        mg_put(a.fc + ro + c.kk0, out);
                    } else {
                        T out[2 * P];
#pragma unroll
                        for (int q = 0; q < 2 * P; ++q) out[q] = acc[q] / w;
                        mg_put(a.fc + ro + 2 * c.kk0, out);
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < 2 * P; ++q) rz[q] = rzn[q];
        }
#pragma unroll
        for (int q = 0; q < P; ++q) {
            xb2[o][q] = x4[q];
            r2o[q] = r2m[q];
            r2m[q] = r2[q];
            b2m[q] = b2[q];
            rb[q] = rbn[q];
        }
    };
    auto march = [&](auto PAR_) MG_INLINE {
        constexpr int A = decltype(PAR_)::v;
        for (int t = 0;;) {
            step(MGInt<0>(), MGInt<A>(), first + t);
            if (++t >= steps) break;
            __syncthreads();
            step(MGInt<1>(), MGInt<1 - A>(), first + t);
            if (++t >= steps) break;
            __syncthreads();
            step(MGInt<2>(), MGInt<A>(), first + t);
            if (++t >= steps) break;
            __syncthreads();
            step(MGInt<3>(), MGInt<1 - A>(), first + t);
            if (++t >= steps) break;
            __syncthreads();
        }
    };
    // a wave's parity is one value, and every wave takes the same number of steps (and so
    // of barriers) on either side
    if (__builtin_amdgcn_readfirstlane(c.par0)) march(MGInt<1>());
    else march(MGInt<0>());
    // the slot of L1 that the last step writes is read by none
    return mg_small<T, EXACT>(a, least, L1 + ((steps - 1) & 1) * SL + a.pairs);
}
template <typename T, int P, bool ZPER, int GEN>
__global__ void __launch_bounds__(kMGSweepThreads) k_mg_down(MGSweepT<T> a)
{
    MGCol<T, P, ZPER> c;
    if (!c.init(a)) return;
    mg_exactly<T>([&](auto exact) {
        return mg_down<T, P, ZPER, GEN, decltype(exact)::value>(a, c);
    });
}

// FZ2: the level was coarsened in z (a pair's cells have one parent)
template <typename T, int P, bool ZPER, bool FZ2, bool EXACT>
__device__ __forceinline__ bool mg_up(const MGSweepT<T> &a, const MGCol<T, P, ZPER> &c)
{
    extern __shared__ double mg_lds[];
    unsigned least = ~0u;
    const int SL = a.rows * mg_lds_row<P>(a.pairs);
    // half planes: corrected black, first red and black, second red
    T *const L1 = reinterpret_cast<T *>(mg_lds), *const L2 = L1 + 2 * SL, *const L3 = L2 + 2 * SL,
            *const L4 = L3 + 2 * SL;
    for (int q = threadIdx.x; q < 8 * SL; q += blockDim.x) L1[q] = (T)0;
    const int fplane = a.ny * a.nz, foff = c.jc * a.nz + 2 * c.kk0;
    const int shx = a.fx >> 1, shy = a.fy >> 1;
    constexpr int PE = FZ2 ? P : 2 * P;
    const int eoff = (c.jc >> shy) * a.cnz + (FZ2 ? c.kk0 : 2 * c.kk0);
    T fl[4][2 * P], ul[4][P], el[4][PE], fr[4][P] = {}, fb[4][P] = {};
    MGDiag<T> dg[4] = {};
    T xw[2][P] = {}, xr1[2][P] = {}, xb1[2][P] = {}, xr2[2][P] = {};
    T wm[P] = {}, r1m[P] = {}, b1m[P] = {}, r2m[P] = {};
    auto load = [&](int i, T (&f)[2 * P], T (&u)[P], T (&e)[PE]) MG_INLINE {
        const int ic = min(max(i, 0), a.nx - 1);
        mg_get(a.f + (size_t)ic * fplane + foff, f);
        mg_get(a.ub + (size_t)ic * (a.ny * a.half) + (c.jc * a.half + c.kk0), u);
        mg_get(a.e + (size_t)(ic >> shx) * (a.cny * a.cnz) + eoff, e);
    };
    const int first = c.x0 - kMGHalo, steps = c.x1 - c.x0 + 2 * kMGHalo;
    constexpr int D = mg_ahead<T, P>();
#pragma unroll
    for (int q = 0; q < D; ++q) load(first + q, fl[q], ul[q], el[q]);
    __syncthreads();
    // PAR: parity of k of plane i's black cells, plane i-1's red ones, and so on
    auto step = [&](auto S_, auto PAR_, int i) MG_INLINE {
        constexpr int S = decltype(S_)::v, PAR = decltype(PAR_)::v;
        constexpr int e = S & 1, o = e ^ 1;
        constexpr int m1 = (S + 3) & 3, m2 = (S + 2) & 3, m3 = (S + 1) & 3;
        const MGDiag<T> d4 = dg[S];
        const bool ok = c.in_level && i >= 0 && i < a.nx;
        T f4[P], w[P], x0[P], d, s[P];
#pragma unroll
        for (int q = 0; q < P; ++q) {
            f4[q] = fb[S][q];
            fr[S][q] = fl[S][2 * q + 1 - PAR];
            fb[S][q] = fl[S][2 * q + PAR];
            // a black cell's own value plus its parent's
            const T v = ul[S][q] + el[S][FZ2 ? q : 2 * q + PAR];
            w[q] = ok ? v : (T)0;
            x0[q] = a.cx * w[q];
        }
        load(i + D, fl[(S + D) & 3], ul[(S + D) & 3], el[(S + D) & 3]);
        dg[S] = c.plane(a, i);
        if (c.live) mg_put(L1 + e * SL + c.own, w);
        // plane i-1: red
        T r1[P], x1[P];
        c.template sum<PAR>(a, L1 + o * SL, xw[e], x0, wm, s);
#pragma unroll
        for (int q = 0; q < P; ++q) {
            r1[q] = c.template quot<PAR, EXACT>(dg[m1], q, fr[m1][q] + s[q], d, least);
            x1[q] = a.cx * r1[q];
            xw[e][q] = x0[q];
            wm[q] = w[q];
        }
        if (c.live) mg_put(L2 + o * SL + c.own, r1);
        // plane i-2: black
        T b1[P], x2[P];
        c.template sum<PAR>(a, L2 + e * SL, xr1[o], x1, r1m, s);
#pragma unroll
        for (int q = 0; q < P; ++q) {
            b1[q] = c.template quot<PAR, EXACT>(dg[m2], q, fb[m2][q] + s[q], d, least);
            x2[q] = a.cx * b1[q];
            xr1[o][q] = x1[q];
            r1m[q] = r1[q];
        }
        if (c.live) mg_put(L3 + e * SL + c.own, b1);
        // plane i-3: red
        T r2[P], x3[P];
        c.template sum<PAR>(a, L3 + o * SL, xb1[e], x2, b1m, s);
#pragma unroll
        for (int q = 0; q < P; ++q) {
            r2[q] = c.template quot<PAR, EXACT>(dg[m3], q, fr[m3][q] + s[q], d, least);
            x3[q] = a.cx * r2[q];
            xb1[e][q] = x2[q];
            b1m[q] = b1[q];
        }
        if (c.live) mg_put(L4 + o * SL + c.own, r2);
        // plane i-4: black, and both colours out
        const int i4 = i - 4;
        if (c.mine && i4 >= c.x0 && i4 < c.x1) {
            T out[2 * P];
            c.template sum<PAR>(a, L4 + e * SL, xr2[o], x3, r2m, s);
#pragma unroll
            for (int q = 0; q < P; ++q) {
                out[2 * q + PAR] = c.template quot<PAR, EXACT>(d4, q, f4[q] + s[q], d, least);
                out[2 * q + 1 - PAR] = r2m[q];
            }
            mg_put(a.u + (size_t)i4 * fplane + (c.j * a.nz + 2 * c.kk0), out);
        }
#pragma unroll
        for (int q = 0; q < P; ++q) {
            xr2[o][q] = x3[q];
            r2m[q] = r2[q];
        }
    };
    auto march = [&](auto PAR_) MG_INLINE {
        constexpr int A = decltype(PAR_)::v;
        for (int t = 0;;) {
            step(MGInt<0>(), MGInt<A>(), first + t);
            if (++t >= steps) break;
            __syncthreads();
            step(MGInt<1>(), MGInt<1 - A>(), first + t);
            if (++t >= steps) break;
            __syncthreads();
            step(MGInt<2>(), MGInt<A>(), first + t);
            if (++t >= steps) break;
            __syncthreads();
            step(MGInt<3>(), MGInt<1 - A>(), first + t);
            if (++t >= steps) break;
            __syncthreads();
        }
    };
    // as in mg_down; plane i's black cells have the other parity
    if (__builtin_amdgcn_readfirstlane(c.par0)) march(MGInt<0>());
    else march(MGInt<1>());
    // the slot of L1 that the last step writes is read by none
    return mg_small<T, EXACT>(a, least, L1 + ((steps - 1) & 1) * SL + a.pairs);
}
template <typename T, int P, bool ZPER, bool FZ2>
__global__ void __launch_bounds__(kMGSweepThreads) k_mg_up(MGSweepT<T> a)
{
    MGCol<T, P, ZPER> c;
    if (!c.init(a)) return;
    mg_exactly<T>([&](auto exact) {
        return mg_up<T, P, ZPER, FZ2, decltype(exact)::value>(a, c);
    });
}

} // namespace cfdmx
