// cfdmx_mg.hip -- geometric multigrid preconditioner and the preconditioned BiCGSTAB of
// the multigrid pressure solves (no reference counterpart), in T = float (the
// mixed-precision inner solve) or T = double (the same algorithm in FP64).
//
// The SPE operator on the uniform grid (SPE_sparseMatrix.hpp:42-106) is the 7-point
// Laplacian (A u)_c = sum over existing neighbours of c_d (u_c - u_nb), c_d = 1/h_d^2,
// with the Neumann faces folded into the diagonal and, with periodic z, the z
// neighbours wrapped.  Each coarser level halves the directions whose spacing is within
// a factor 2 of the smallest (z first on the flat cells of the cylinder grids), down to
// at most 512 cells or no even size left; its operator is the same Laplacian on the
// coarse spacings.  Cycle: V(2,2) with red-black Gauss-Seidel, restriction = mean of the
// children's residuals, prolongation = the parent's value; the coarsest level is solved
// exactly by fast diagonalisation (the 1-D eigenbases of its three axes, computed on the
// host).  Every inner product accumulates in double.
//
// Every level is stored in natural order.  A level with even nz takes two kernels a cycle,
// one on the way down and one on the way up, each passing over the level once with all its
// half sweeps (cfdmx_mg_sweep.hpp).  The smallest levels run in one workgroup, in LDS.
// Levels with odd nz above those take a launch per half sweep, one thread per cell.  The
// arithmetic of every cell update (terms, weights, order) is the same in each form.
//
// Measured, a V-cycle before (a launch per half sweep, colours stored apart) and after:
// 350 -> 173 us in float and 508 -> 238 us in double at 512x256x64, 2.4 ms -> 660 us in
// float at 1024x512x128.
#include "cfdmx_internal.hpp"
#include "cfdmx_mg_sweep.hpp"

namespace cfdmx {

static inline int cdiv(int a, int b) { return (a + b - 1) / b; }

template <typename T>
__device__ __forceinline__ void mg_coords(const MGLevelT<T> &L, int n, int &i, int &j, int &k)
{
    const unsigned t = fdiv((unsigned)n, L.dz);
    k = n - (int)t * L.nz;
    i = (int)fdiv(t, L.dy);
    j = (int)t - i * L.ny;
}

template <typename T>
__device__ __forceinline__ T mg_diag(const MGLevelT<T> &L, int i, int j, int k)
{
    T d = (T)0;
    if (i > 0) d += L.cx;
    if (i < L.nx - 1) d += L.cx;
    if (j > 0) d += L.cy;
    if (j < L.ny - 1) d += L.cy;
    if (L.nz > 1) {
        if (L.zper) {
            d += (T)2 * L.cz;
        } else {
            if (k > 0) d += L.cz;
            if (k < L.nz - 1) d += L.cz;
        }
    }
    return d;
}

// sum of c_d * v(nb) over the existing neighbours nb of cell n, in the order
// -x, +x, -y, +y, -z, +z; v(m, a, b, c) gives the value of cell m = (a, b, c).  A
// missing neighbour is taken as the cell itself with weight 0 (adding +0 changes no
// sum), so that every value is fetched without a branch and the loads overlap.
template <typename T, class V>
__device__ __forceinline__ T mg_nbsum(const MGLevelT<T> &L, int n, int i, int j, int k, V &&v)
{
    const int sx = L.ny * L.nz, sy = L.nz;
    const bool xm = i > 0, xp = i < L.nx - 1, ym = j > 0, yp = j < L.ny - 1;
    T s = (T)0;
    s += (xm ? L.cx : (T)0) * v(xm ? n - sx : n, xm ? i - 1 : i, j, k);
    s += (xp ? L.cx : (T)0) * v(xp ? n + sx : n, xp ? i + 1 : i, j, k);
    s += (ym ? L.cy : (T)0) * v(ym ? n - sy : n, i, ym ? j - 1 : j, k);
    s += (yp ? L.cy : (T)0) * v(yp ? n + sy : n, i, yp ? j + 1 : j, k);
    if (L.nz > 1) {
        const bool zm = L.zper || k > 0, zp = L.zper || k < L.nz - 1;
        const int km = k > 0 ? k - 1 : (zm ? L.nz - 1 : k);
        const int kp = k < L.nz - 1 ? k + 1 : (zp ? 0 : k);
        s += (zm ? L.cz : (T)0) * v(n + (km - k), i, j, km);
        s += (zp ? L.cz : (T)0) * v(n + (kp - k), i, j, kp);
    }
    return s;
}

// ---- a launch per half sweep, one thread per cell ----

// half sweep; zero_first: u starts at zero (the other colour is written 0).  With
// periodic z and odd nz > 1 the planes k = 0 and k = nz-1 hold the same colour and are
// neighbours, so a half sweep there runs in two launches, planes = 1 (k < nz-1) and then
// planes = 2 (k = nz-1): the first reads the old k = nz-1 values, the second the new
// k = 0 values, and no cell is read while another thread writes it.  planes = 0: all.
template <typename T>
__global__ void __launch_bounds__(256) k_mg_smooth_cell(MGLevelT<T> L, int colour, int zero_first,
                                                        int planes)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= L.n) return;
    int i, j, k;
    mg_coords(L, n, i, j, k);
    if (((i + j + k) & 1) != colour) {
        if (zero_first) L.u[n] = (T)0;
        return;
    }
    if ((planes == 1 && k == L.nz - 1) || (planes == 2 && k != L.nz - 1)) return;
    const T *u = L.u;
    const T s = zero_first ? (T)0 : mg_nbsum(L, n, i, j, k, [&](int q, int, int, int) { return u[q]; });
    L.u[n] = (L.f[n] + s) / mg_diag(L, i, j, k);
}

template <typename T>
__device__ __forceinline__ void mg_prolong_at(const MGLevelT<T> &F, const MGLevelT<T> &C, int n)
{
    int i, j, k;
    mg_coords(F, n, i, j, k);
    F.u[n] += C.u[((i >> (C.fx >> 1)) * C.ny + (j >> (C.fy >> 1))) * C.nz + (k >> (C.fz >> 1))];
}

template <typename T>
__global__ void __launch_bounds__(256) k_mg_prolong(MGLevelT<T> F, MGLevelT<T> C)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= F.n) return;
    mg_prolong_at(F, C, n);
}

// coarse right-hand side: mean over the children of the fine residual f - A u
// (LDS: their loads need no overlap, and absent children are left out)
template <bool LDS = false, typename T>
__device__ __forceinline__ void mg_restrict_at(const MGLevelT<T> &F, const MGLevelT<T> &C, int m)
{
    int I, J, K;
    mg_coords(C, m, I, J, K);
    const T *u = F.u;
    T acc = (T)0;
    // at most 2 x 2 x 2 children in the order (a, b, c), unrolled and branch-free so that
    // their loads are in flight together: a child that does not exist evaluates child
    // (0, 0, 0) and adds +0, an identity (the sum starts at +0 and so never holds -0)
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int a = q >> 2, b = (q >> 1) & 1, c = q & 1;
        const bool ok = a < C.fx && b < C.fy && c < C.fz;
        if (LDS && !ok) continue;
        const int i = I * C.fx + (ok ? a : 0), j = J * C.fy + (ok ? b : 0),
                  k = K * C.fz + (ok ? c : 0);
        const int n = (i * F.ny + j) * F.nz + k;
        const T s = mg_nbsum(F, n, i, j, k, [&](int x, int, int, int) { return u[x]; });
        const T r = F.f[n] - (mg_diag(F, i, j, k) * u[n] - s);
        acc += ok ? r : (T)0;
    }
    C.f[m] = acc / (T)(C.fx * C.fy * C.fz);
}

template <typename T>
__global__ void __launch_bounds__(256) k_mg_restrict(MGLevelT<T> F, MGLevelT<T> C)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= C.n) return;
    mg_restrict_at(F, C, m);
}

// coarsest level: the exact solve by fast diagonalisation.  The level's operator is the
// Kronecker sum of three 1-D chains with orthonormal eigenvectors Qx, Qy, Qz, so
// u = Q diag(1 / lambda) Q^T f with Q = Qx (x) Qy (x) Qz and lambda = lx + ly + lz; the
// constant mode (lambda = 0) is dropped, which returns the mean-free solution of A u = f
// for the mean-free part of f.  One workgroup: the six 1-D transforms run through LDS,
// a barrier apart.
constexpr int kMGCoarseThreads = 1024;
// sum over q < n of Q[q * sq] * a[q * sa], in order; the loads of eight terms overlap
template <typename T>
__device__ __forceinline__ T mg_dot(const T *Q, int sq, const T *a, int sa, int n)
{
    T acc = (T)0;
    int q = 0;
    for (; q + 8 <= n; q += 8) {
        T x[8], y[8];
#pragma unroll
        for (int w = 0; w < 8; ++w) x[w] = Q[(q + w) * sq], y[w] = a[(q + w) * sa];
#pragma unroll
        for (int w = 0; w < 8; ++w) acc += x[w] * y[w];
    }
    for (; q < n; ++q) acc += Q[q * sq] * a[q * sa];
    return acc;
}

// Qx: the eigenvectors and eigenvalues (MGLevelT::fd or its copy in LDS); L.f may be b, and
// L.u is written last, from b
template <typename T>
__device__ __forceinline__ void mg_coarse_solve(const MGLevelT<T> &L, const T *Qx, T *a, T *b)
{
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const T *Qy = Qx + nx * nx, *Qz = Qy + ny * ny;
    const T *lx = Qz + nz * nz, *ly = lx + nx, *lz = ly + ny;
    const int tid = threadIdx.x, nt = blockDim.x;
    for (int n = tid; n < L.n; n += nt) a[n] = L.f[n];
    __syncthreads();
    // forward: coefficients along x, then y, then z (divided by the eigenvalue)
    for (int n = tid; n < L.n; n += nt) {
        int m, j, k;
        mg_coords(L, n, m, j, k);
        b[n] = mg_dot(Qx + m * nx, 1, a + j * nz + k, ny * nz, nx);
    }
    __syncthreads();
    for (int n = tid; n < L.n; n += nt) {
        int mx, m, k;
        mg_coords(L, n, mx, m, k);
        a[n] = mg_dot(Qy + m * ny, 1, b + mx * ny * nz + k, nz, ny);
    }
    __syncthreads();
    for (int n = tid; n < L.n; n += nt) {
        int mx, my, m;
        mg_coords(L, n, mx, my, m);
        const T acc = mg_dot(Qz + m * nz, 1, a + (mx * ny + my) * nz, 1, nz);
        const T lam = lx[mx] + ly[my] + lz[m];
        b[n] = (mx == 0 && my == 0 && m == 0) ? (T)0 : acc / lam;
    }
    __syncthreads();
    // inverse: back along z, y, x
    for (int n = tid; n < L.n; n += nt) {
        int mx, my, k;
        mg_coords(L, n, mx, my, k);
        a[n] = mg_dot(Qz + k, nz, b + (mx * ny + my) * nz, 1, nz);
    }
    __syncthreads();
    for (int n = tid; n < L.n; n += nt) {
        int mx, j, k;
        mg_coords(L, n, mx, j, k);
        b[n] = mg_dot(Qy + j, ny, a + mx * ny * nz + k, nz, ny);
    }
    __syncthreads();
    for (int n = tid; n < L.n; n += nt) {
        int i, j, k;
        mg_coords(L, n, i, j, k);
        L.u[n] = mg_dot(Qx + i, nx, b + j * nz + k, ny * nz, nx);
    }
}

// values of the exact solve's tables; they are copied to LDS where they are this few
constexpr int kMGTableLds = 4096;
template <typename T> __host__ __device__ inline int mg_table(const MGLevelT<T> &B)
{
    return B.nx * B.nx + B.ny * B.ny + B.nz * B.nz + B.nx + B.ny + B.nz;
}

// The tail of the hierarchy in one workgroup: its first level (see kMGTailCells) and all
// below it, from that level's first sweep to its last, the exact solve included.
// These levels hold a few thousand cells, where a launch per half sweep costs more than
// the sweep.  Every level's u and f stay in LDS, the steps a barrier apart; only the first
// level's f comes from global memory and its u goes back.
template <typename T>
struct MGTail {
    MGLevelT<T> L[kMGTailLevels];
    int nlev;
};

// half sweep of colour c over a level in LDS.  The threads count cells of the colour: nz / 2 of
// each row (below the top plane where nz is odd), then every other row's cell of that plane.
// Counted over all cells, with half of the threads idle, k_mg_tail took 37.7 us for 48x24x3 and
// below in FP32, now 28.1: one CU, about a microsecond a half sweep of the first level (cheaper index divisions
// and one copy of the sweeps' code, 3168 lines in place of 6039, changed nothing or cost 3 us).
template <typename T>
__device__ __forceinline__ void mg_tail_sweep(const MGLevelT<T> &L, int c)
{
    const int tid = threadIdx.x, nt = blockDim.x;
    const T *u = L.u;
    auto cell = [&](int row, int i, int j, int k) {
        const int n = row * L.nz + k;
        const T s = mg_nbsum(L, n, i, j, k, [&](int q, int, int, int) { return u[q]; });
        L.u[n] = (L.f[n] + s) / mg_diag(L, i, j, k);
    };
    const int half = L.nz >> 1, rows = L.nx * L.ny;
    for (int m = tid; m < rows * half; m += nt) {
        const int row = (int)fdiv((unsigned)m, L.dzh);
        const int i = (int)fdiv((unsigned)row, L.dy), j = row - i * L.ny;
        cell(row, i, j, 2 * (m - row * half) + ((i + j + c) & 1));
    }
    if (L.nz & 1) {
        // periodic z joins two cells of one colour: their planes in turn (k_mg_smooth_cell)
        if (L.zper && L.nz > 1) __syncthreads();
        const int top = L.nz - 1; // even: the colour's rows are those of i + j of c's parity
        for (int m = tid; m < (rows + 1) >> 1; m += nt) {
            int row = 2 * m, i = (int)fdiv((unsigned)row, L.dy);
            // i + j runs with the row number where ny is odd; else row 2m and the next share i
            row += L.ny & 1 ? c : (i + c) & 1;
            if (row >= rows) continue;
            i = (int)fdiv((unsigned)row, L.dy);
            cell(row, i, row - i * L.ny, top);
        }
    }
    __syncthreads();
}

template <typename T>
__global__ void __launch_bounds__(kMGCoarseThreads) k_mg_tail(MGTail<T> t)
{
    extern __shared__ double coarse_lds[];
    const int tid = threadIdx.x, nt = blockDim.x, nl = t.nlev;
    const int table = mg_table(t.L[nl - 1]);
    T *tab = reinterpret_cast<T *>(coarse_lds);
    T *mem = tab + (table <= kMGTableLds ? (table + 1) / 2 * 2 : 0);
    for (int n = tid; n < t.L[0].n; n += nt) mem[t.L[0].n + n] = t.L[0].f[n];
    if (table <= kMGTableLds)
        for (int n = tid; n < table; n += nt) tab[n] = t.L[nl - 1].fd[n];
    __syncthreads();
    T *at = mem;
    for (int l = 0; l < nl - 1; ++l) {
        MGLevelT<T> F = t.L[l], C = t.L[l + 1];
        F.u = at;
        F.f = at + F.n;
        at += 2 * F.n;
        C.f = at + C.n;
        // first red sweep from u = 0
        for (int n = tid; n < F.n; n += nt) {
            int i, j, k;
            mg_coords(F, n, i, j, k);
            F.u[n] = ((i + j + k) & 1) ? (T)0 : F.f[n] / mg_diag(F, i, j, k);
        }
        __syncthreads();
        mg_tail_sweep(F, 1);
        mg_tail_sweep(F, 0);
        mg_tail_sweep(F, 1);
        for (int m = tid; m < C.n; m += nt) mg_restrict_at<true>(F, C, m);
        __syncthreads();
    }
    {
        MGLevelT<T> B = t.L[nl - 1];
        B.f = at + B.n;
        B.u = at;
        if (table <= kMGTableLds) mg_coarse_solve(B, (const T *)tab, at, at + B.n);
        else mg_coarse_solve(B, B.fd, at, at + B.n);
        __syncthreads();
    }
    for (int l = nl - 2; l >= 0; --l) {
        MGLevelT<T> F = t.L[l], C = t.L[l + 1];
        C.u = at;
        at -= 2 * F.n;
        F.u = at;
        F.f = at + F.n;
        for (int n = tid; n < F.n; n += nt) mg_prolong_at(F, C, n);
        __syncthreads();
        mg_tail_sweep(F, 0);
        mg_tail_sweep(F, 1);
        mg_tail_sweep(F, 0);
        mg_tail_sweep(F, 1);
    }
    for (int n = tid; n < t.L[0].n; n += nt) t.L[0].u[n] = mem[n];
}

// ---- preconditioned BiCGSTAB pieces (linear cell order, canonical block sums) ----
// out = A in on level 0 (double accumulation of the 7 terms); partials of (out, w) and,
// with NS = 2, (out, out)
template <int NS, typename T>
__global__ void __launch_bounds__(kThreads)
k_pb_spmv(Geo g, MGLevelT<T> L, const T *__restrict__ in, T *__restrict__ out,
          const T *__restrict__ w, double *part, const PBState *st)
{
    if (st->done) return;
    const int B = logical_block(g);
    if (B >= g.nblocks) return;
    double acc[NS];
    for (int q = 0; q < NS; ++q) acc[q] = 0.0;
    auto cell = [&](int n) {
        {
            int i, j, k;
            mg_coords(L, n, i, j, k);
            // branch-free: a missing neighbour reads the cell itself with weight 0
            const int sx = L.ny * L.nz, sy = L.nz;
            const bool xm = i > 0, xp = i < L.nx - 1, ym = j > 0, yp = j < L.ny - 1;
            const bool zm = L.zper || k > 0, zp = L.zper || k < L.nz - 1;
            const double cx = L.cx, cy = L.cy, cz = L.cz;
            const double wxm = xm ? cx : 0.0, wxp = xp ? cx : 0.0, wym = ym ? cy : 0.0,
                         wyp = yp ? cy : 0.0, wzm = zm ? cz : 0.0, wzp = zp ? cz : 0.0;
            const int km = k > 0 ? n - 1 : (L.zper ? n + L.nz - 1 : n);
            const int kp = k < L.nz - 1 ? n + 1 : (L.zper ? n - (L.nz - 1) : n);
            double s = 0.0;
            s += wxm * (double)in[xm ? n - sx : n];
            s += wxp * (double)in[xp ? n + sx : n];
            s += wym * (double)in[ym ? n - sy : n];
            s += wyp * (double)in[yp ? n + sy : n];
            s += wzm * (double)in[km];
            s += wzp * (double)in[kp];
            const double d = wxm + wxp + wym + wyp + wzm + wzp;
            const T o = (T)(d * (double)in[n] - s);
            out[n] = o;
            acc[0] += (double)o * (double)w[n];
            if (NS == 2) acc[NS - 1] += (double)o * (double)o;
        }
    };
    // a full block has no bounds test, so its cells' loads overlap
    if ((B + 1) * kPerBlock <= g.N) {
#pragma unroll
        for (int c = 0; c < kCells; ++c) cell(B * kPerBlock + c * kThreads + threadIdx.x);
    } else {
        for (int c = 0; c < kCells; ++c) {
            const int n = B * kPerBlock + c * kThreads + threadIdx.x;
            if (n < g.N) cell(n);
        }
    }
    block_sums<NS>(acc, part, g.nblocks, B);
}

// The same product with four consecutive cells of a z-row per thread (nz a multiple of
// 4): their centres, x and y neighbours are read as one vector each and their z
// neighbours are each other, so a thread issues 7 loads for 4 cells instead of 28.
// Each cell's terms, weights and order are k_pb_spmv's, so out is the same; the dot
// partials add a thread's cells in another order.
template <typename T> struct Vec4;
template <> struct Vec4<float> {
    float v[4];
    __device__ __forceinline__ void load(const float *p)
    {
        const float4 a = *reinterpret_cast<const float4 *>(p);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
    }
    __device__ __forceinline__ void store(float *p) const
    {
        *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
    }
};
template <> struct Vec4<double> {
    double v[4];
    __device__ __forceinline__ void load(const double *p)
    {
        const double2 a = reinterpret_cast<const double2 *>(p)[0];
        const double2 b = reinterpret_cast<const double2 *>(p)[1];
        v[0] = a.x, v[1] = a.y, v[2] = b.x, v[3] = b.y;
    }
    __device__ __forceinline__ void store(double *p) const
    {
        reinterpret_cast<double2 *>(p)[0] = make_double2(v[0], v[1]);
        reinterpret_cast<double2 *>(p)[1] = make_double2(v[2], v[3]);
    }
};

template <int NS, typename T>
__global__ void __launch_bounds__(kThreads)
k_pb_spmv4(Geo g, MGLevelT<T> L, const T *__restrict__ in, T *__restrict__ out,
           const T *__restrict__ w, double *part, const PBState *st)
{
    if (st->done) return;
    const int B = logical_block(g);
    if (B >= g.nblocks) return;
    double acc[NS];
    for (int q = 0; q < NS; ++q) acc[q] = 0.0;
    const int n0 = B * kPerBlock + 4 * threadIdx.x;
    if (n0 < g.N) {
        int i, j, k0;
        mg_coords(L, n0, i, j, k0);
        const int sx = L.ny * L.nz, sy = L.nz;
        const bool xm = i > 0, xp = i < L.nx - 1, ym = j > 0, yp = j < L.ny - 1;
        const double cx = L.cx, cy = L.cy, cz = L.cz;
        const double wxm = xm ? cx : 0.0, wxp = xp ? cx : 0.0, wym = ym ? cy : 0.0,
                     wyp = yp ? cy : 0.0;
        Vec4<T> c, vxm, vxp, vym, vyp, vw;
        c.load(in + n0);
        vxm.load(in + (xm ? n0 - sx : n0));
        vxp.load(in + (xp ? n0 + sx : n0));
        vym.load(in + (ym ? n0 - sy : n0));
        vyp.load(in + (yp ? n0 + sy : n0));
        vw.load(w + n0);
        const int klo = k0 > 0 ? n0 - 1 : (L.zper ? n0 + L.nz - 1 : n0);
        const int khi = k0 + 3 < L.nz - 1 ? n0 + 4 : (L.zper ? n0 + 4 - L.nz : n0 + 3);
        const T zlo = in[klo], zhi = in[khi];
        Vec4<T> o;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = k0 + q;
            const bool zm = L.zper || k > 0, zp = L.zper || k < L.nz - 1;
            const double wzm = zm ? cz : 0.0, wzp = zp ? cz : 0.0;
            const T zmv = q > 0 ? c.v[q - 1] : zlo, zpv = q < 3 ? c.v[q + 1] : zhi;
            double s = 0.0;
            s += wxm * (double)vxm.v[q];
            s += wxp * (double)vxp.v[q];
            s += wym * (double)vym.v[q];
            s += wyp * (double)vyp.v[q];
            s += wzm * (double)zmv;
            s += wzp * (double)zpv;
            const double d = wxm + wxp + wym + wyp + wzm + wzp;
            o.v[q] = (T)(d * (double)c.v[q] - s);
            acc[0] += (double)o.v[q] * (double)vw.v[q];
            if (NS == 2) acc[NS - 1] += (double)o.v[q] * (double)o.v[q];
        }
        o.store(out + n0);
    }
    block_sums<NS>(acc, part, g.nblocks, B);
}

// p = r (first iteration) or r + beta (p - omega v)
template <typename T>
__global__ void k_pb_update_p(Geo g, int first, const T *r, const T *v, T *p, const PBState *st)
{
    if (st->done) return;
    const T beta = (T)st->beta, om = (T)st->omega;
    for (int n = blockIdx.x * blockDim.x + threadIdx.x; n < g.N; n += gridDim.x * blockDim.x)
        p[n] = first ? r[n] : r[n] + beta * (p[n] - om * v[n]);
}

// Up to this many partials every block of the kernel that uses a scalar folds them itself
// (a block and all of them in flight together: 1 to 2 us); above, a kernel of one block does
// it once.  Steps of 16 to 1024 partials measured 5 to 16 us less so, of 2048 the same, of 4096
// up to 2% more and of 8192 (512x256x64, each block would read 64 KiB) 3 to 7% more.
constexpr int kPBFoldEach = 1024;
// alpha = rho / (v, r0)
template <int U>
__device__ __forceinline__ double pb_alpha(const Geo &g, const double *part, const PBState *st)
{
    double t[1];
    fold_partials<1, U>(part, g.nblocks, g.nblocks, t);
    return st->rho / t[0];
}
__global__ void __launch_bounds__(kThreads) k_pb_alpha(Geo g, const double *part, PBState *st)
{
    if (st->done) return;
    const double alpha = pb_alpha<kFoldAlone>(g, part, st);
    if (threadIdx.x == 0) st->alpha = alpha;
}

// omega = (t, s) / (t, t)
template <int U>
__device__ __forceinline__ double pb_omega(const Geo &g, const double *part)
{
    double t[2];
    fold_partials<2, U>(part, g.nblocks, g.nblocks, t);
    return t[0] / t[1];
}
__global__ void __launch_bounds__(kThreads) k_pb_omega(Geo g, const double *part, PBState *st)
{
    if (st->done) return;
    const double omega = pb_omega<kFoldAlone>(g, part);
    if (threadIdx.x == 0) st->omega = omega;
}

// s = r - alpha v; FOLD: alpha from the partials of (v, r0), for the kernels to come too
template <typename T, bool FOLD>
__global__ void __launch_bounds__(kThreads)
k_pb_update_s(Geo g, const double *part, const T *r, const T *v, T *s, PBState *st)
{
    if (st->done) return;
    double alpha;
    if constexpr (FOLD) {
        alpha = pb_alpha<8>(g, part, st);
        if (blockIdx.x == 0 && threadIdx.x == 0) st->alpha = alpha;
    } else {
        alpha = st->alpha;
    }
    const T a = (T)alpha;
    for (int n = blockIdx.x * blockDim.x + threadIdx.x; n < g.N; n += gridDim.x * blockDim.x)
        s[n] = r[n] - a * v[n];
}

// e += alpha p^ + omega s^; r = s - omega t; partials (r, r), (r, r0).  The correction e
// and its increments are FP64 in both modes: in FP32 its own rounding (6e-8 of e),
// multiplied by the operator's condition number (~1e5 here), would leave a true residual
// near 1e-2 of the pass's start, whatever the inner tolerance; in FP64 the pass's floor is
// the FP32 recursion's drift from the true residual, ~1e-6.  FIRST (the solve's first
// iteration, e = 0): e is written as +0.0 plus the increment without being read, which is
// the sum the zeroed vector would give, -0.0 turning to +0.0 included.
// FOLD: omega from the partials of (t, s), (t, t).
template <typename T, bool FIRST, bool FOLD>
__global__ void __launch_bounds__(kThreads)
k_pb_update_xr(Geo g, const double *part_in, const T *__restrict__ ph, const T *__restrict__ sh,
               const T *__restrict__ s, const T *__restrict__ t, const T *__restrict__ r0,
               double *__restrict__ e, T *__restrict__ r, double *part_out, PBState *st)
{
    if (st->done) return;
    const int B = logical_block(g);
    if (B >= g.nblocks) return;
    const double ad = st->alpha;
    double omd;
    if constexpr (FOLD) {
        omd = pb_omega<8>(g, part_in);
        if (B == 0 && threadIdx.x == 0) st->omega = omd;
    } else {
        omd = st->omega;
    }
    const T om = (T)omd;
    double acc[2] = {0.0, 0.0};
    auto cell = [&](int n) {
        const double inc = ad * (double)ph[n] + omd * (double)sh[n];
        if constexpr (FIRST) e[n] = 0.0 + inc;
        else e[n] += inc;
        const T rn = s[n] - om * t[n];
        r[n] = rn;
        acc[0] += (double)rn * (double)rn;
        acc[1] += (double)rn * (double)r0[n];
    };
    if ((B + 1) * kPerBlock <= g.N) {
#pragma unroll
        for (int c = 0; c < kCells; ++c) cell(B * kPerBlock + c * kThreads + threadIdx.x);
    } else {
        for (int c = 0; c < kCells; ++c) {
            const int n = B * kPerBlock + c * kThreads + threadIdx.x;
            if (n < g.N) cell(n);
        }
    }
    block_sums<2>(acc, part_out, g.nblocks, B);
}

// end of an iteration: residual test, rho and beta for the next one.  host: the host's copy of
// the state in pinned memory, written here (a copy after the kernel is a kernel of its own)
__global__ void __launch_bounds__(kThreads)
k_pb_end(Geo g, const double *part, PBState *st, PBState *host)
{
    if (st->done) return;
    double t[2];
    fold_partials<2, kFoldAlone>(part, g.nblocks, g.nblocks, t);
    if (threadIdx.x == 0) {
        const double res = sqrt(t[0]) / st->norm0;
        st->res = res;
        st->iter += 1;
        const double rho = t[1];
        st->beta = (rho / st->rho) * (st->alpha / st->omega);
        st->rho = rho;
        if (res < st->tol) st->done = 1;
        else if (st->iter >= st->maxit || !(res == res)) st->done = 2;
        *host = *st;
    }
}

// ---- launchers ----
template <typename T, int P> static size_t sweep_lds(const MGSweepT<T> &a);

template <typename T, int P, bool ZPER>
static void launch_sweep(hipStream_t s, const MGSweepT<T> &a, bool down)
{
    const int threads = 2 * mg_half_block(a.rows, a.tpr);
    const size_t lds = sweep_lds<T, P>(a);
    const dim3 grid((a.nblk + 7) / 8 * 8);
    if (!down) {
        if (a.fz == 2)
            hipLaunchKernelGGL((k_mg_up<T, P, ZPER, true>), grid, dim3(threads), lds, s, a);
        else
            hipLaunchKernelGGL((k_mg_up<T, P, ZPER, false>), grid, dim3(threads), lds, s, a);
    } else if (a.fx == 1 && a.fy == 1 && a.fz == 2) {
        hipLaunchKernelGGL((k_mg_down<T, P, ZPER, 0>), grid, dim3(threads), lds, s, a);
    } else {
        hipLaunchKernelGGL((k_mg_down<T, P, ZPER, 1>), grid, dim3(threads), lds, s, a);
    }
}

// Whether a thread may take P z-pairs of a level.  In double with walls two spill up to 157
// registers: a step of 384x192x96 cells took 5.58 ms, 4.85 with one and 5.03 with separate half
// sweeps, one of 128x128x128 7.24, 5.53 and 6.58.  With periodic z two spill at most 32
// (coarsening in all directions) and are up to 10% slower or 7% faster than one by the grid;
// float's four with walls spill 29 and are level with two or up to 9% faster.
template <typename T> constexpr bool mg_pairs(int P, bool zper)
{
    return std::is_same<T, float>::value || P == 1 || (P == 2 && zper);
}

// The tiling of a level for the one-pass kernels, from an estimate of a block's step: a CU
// with W waves resident takes lat + add W us for a plane, or W issue us where the
// instructions bound it (fitted to both kernels over 15 level shapes from 96x48x6 to
// 1024x512x128, every P, ty and cxl: the choice is within 0.3% of the best measured one in
// the mean of these).  More rows and planes a block mean fewer formed twice; more blocks fill the CUs.
struct SweepCost {
    double lat, add, issue;
    int waves; // of this kernel a CU holds (registers)
};
template <typename T, int P> static SweepCost sweep_cost()
{
    if (std::is_same<T, float>::value)
        return P == 1 ? SweepCost{0.45, 0.012, 0.054, 16}
                      : (P == 2 ? SweepCost{0.63, 0.008, 0.070, 8}
                                : SweepCost{0.86, 0.020, 0.133, 8});
    return P == 1 ? SweepCost{0.45, 0.035, 0.060, 8} : SweepCost{0.74, 0.039, 0.134, 8};
}

template <typename T, int P>
static size_t sweep_lds(const MGSweepT<T> &a)
{
    return 8 * (size_t)a.rows * mg_lds_row<P>(a.pairs) * sizeof(T) +
           (a.fy == 2 ? 4 * (size_t)a.rows * a.pairs * sizeof(T) : 0);
}

template <typename T, int P>
static void sweep_tiles(MGSweepT<T> &a, int ty, int tz, int cxl)
{
    a.ty = ty;
    a.rows = ty + 2 * kMGHalo;
    a.tz = tz;
    a.nkt = cdiv(a.half, tz);
    a.pairs = a.nkt == 1 ? a.half : tz + 2 * mg_zhalo<P>();
    a.tpr = a.pairs / P;
    a.cxl = cxl;
    a.njt = cdiv(a.ny, ty);
    a.nblk = a.njt * a.nkt * cdiv(a.nx, cxl);
}

template <typename T, int P>
static void sweep_try(const MGSweepT<T> &base, double &best, MGLevelT<T> &F)
{
    if (base.half % P) return;
    const SweepCost c = sweep_cost<T, P>();
    MGSweepT<T> a = base;
    for (int tz : {base.half, 64, 32}) {
        if (tz < base.half && base.half <= kMGLongRow) break;
        if (tz > base.half) continue;
        for (int ty : {2, 4, 8, 16, 24, 32, 40, 56, 64, 120}) {
            if (ty > 2 && ty - 8 >= base.ny) break;
            sweep_tiles<T, P>(a, ty, tz, 2);
            const int waves = 2 * mg_half_block(a.rows, a.tpr) / 64;
            const size_t lds = sweep_lds<T, P>(a);
            if (waves * 64 > kMGSweepThreads || lds > kMGSweepLds) break;
            const int fit = std::max(1, std::min(c.waves / waves, (int)(kMGSweepLds / lds)));
            auto step = [&](int blocks) {
                const double w = (double)blocks * waves;
                return std::max(c.lat + c.add * w, c.issue * w);
            };
            for (int cxl : {2, 4, 6, 8, 12, 16, 20, 24, 28, 32, 48, 64, 96, 128, 256, 512}) {
                if (cxl > 2 && cxl >= 2 * base.nx) break;
                sweep_tiles<T, P>(a, ty, tz, cxl);
                const int per_cu = cdiv(a.nblk, 256), full = per_cu / fit, rest = per_cu % fit;
                const double t =
                    (cxl + 2 * kMGHalo) * (full * step(fit) + (rest ? step(rest) : 0.0));
                if (t < best) {
                    best = t;
                    F.sp = P, F.sty = ty, F.stz = tz, F.scx = cxl;
                }
            }
        }
    }
}

template <typename T>
static MGSweepT<T> sweep_args(const MGLevelT<T> &F, const MGLevelT<T> &C)
{
    MGSweepT<T> a = {};
    a.nx = F.nx, a.ny = F.ny, a.nz = F.nz, a.half = F.nz >> 1;
    a.fx = C.fx, a.fy = C.fy, a.fz = C.fz, a.cny = C.ny, a.cnz = C.nz;
    a.cx = F.cx, a.cy = F.cy, a.cz = F.cz;
    // from here on a float dividend's quotient by any diagonal of the level is normal and the
    // products that correct it are exact (2^-102)
    a.tiny = std::max((T)0x1p-100, (T)0x1p-120 * (F.cx + F.cy + F.cz));
    a.f = F.f, a.e = C.u, a.ub = F.ub, a.fc = C.f, a.u = F.u;
    return a;
}

template <typename T>
void mg_plan(MGLevelT<T> *L, int nlev)
{
    for (int l = 0; l + 1 < nlev; ++l) {
        L[l].sp = 0;
        if (L[l].nz & 1) continue; // odd nz: a launch per half sweep
        const MGSweepT<T> a = sweep_args(L[l], L[l + 1]);
        double best = 1e30;
        sweep_try<T, 1>(a, best, L[l]);
        if (mg_pairs<T>(2, L[l].zper)) sweep_try<T, 2>(a, best, L[l]);
        if (mg_pairs<T>(4, L[l].zper)) sweep_try<T, 4>(a, best, L[l]);
    }
}

template <typename T>
static void launch_half_cycle(hipStream_t s, const MGLevelT<T> &F, const MGSweepT<T> &a, int P,
                              bool down)
{
    auto go = [&](auto zper) {
        constexpr bool Z = decltype(zper)::value;
        if constexpr (mg_pairs<T>(4, Z)) {
            if (P == 4) return launch_sweep<T, 4, Z>(s, a, down);
        }
        if constexpr (mg_pairs<T>(2, Z)) {
            if (P == 2) return launch_sweep<T, 2, Z>(s, a, down);
        }
        launch_sweep<T, 1, Z>(s, a, down);
    };
    if (F.zper) go(std::true_type());
    else go(std::false_type());
}

// LDS of the tail from level l on; 0 where level l does not start it
template <typename T>
static size_t tail_lds(const MGLevelT<T> *L, int nlev, int l)
{
    if (l < nlev - 1 && (L[l].n > ((L[l].nz & 1) ? kMGTailCellsOdd : kMGTailCells) ||
                         nlev - l > kMGTailLevels))
        return 0;
    const int table = mg_table(L[nlev - 1]);
    size_t n = table <= kMGTableLds ? (table + 1) / 2 * 2 : 0;
    for (int q = l; q < nlev; ++q) n += 2 * (size_t)L[q].n;
    return n * sizeof(T);
}

template <typename T>
void launch_mg_vcycle(hipStream_t s, const MGLevelT<T> *L, int nlev, int l)
{
    const MGLevelT<T> &F = L[l];
    if (const size_t lds = tail_lds(L, nlev, l)) {
        MGTail<T> t;
        t.nlev = nlev - l;
        for (int q = l; q < nlev; ++q) t.L[q - l] = L[q];
        hipLaunchKernelGGL(k_mg_tail<T>, dim3(1), dim3(kMGCoarseThreads), lds, s, t);
        return;
    }
    const MGLevelT<T> &C = L[l + 1];
    if (F.sp) {
        MGSweepT<T> a = sweep_args(F, C);
        if (F.sp == 4) sweep_tiles<T, 4>(a, F.sty, F.stz, F.scx);
        else if (F.sp == 2) sweep_tiles<T, 2>(a, F.sty, F.stz, F.scx);
        else sweep_tiles<T, 1>(a, F.sty, F.stz, F.scx);
        launch_half_cycle(s, F, a, F.sp, true);
        launch_mg_vcycle(s, L, nlev, l + 1);
        launch_half_cycle(s, F, a, F.sp, false);
        return;
    }
    const int nb = cdiv(F.n, 256);
    // a half sweep that reads neighbours; two launches where the periodic z wrap joins
    // two cells of one colour (see k_mg_smooth_cell)
    const bool wrap_same = F.zper && F.nz > 1;
    auto half_sweep = [&](int colour) {
        if (wrap_same) {
            hipLaunchKernelGGL(k_mg_smooth_cell<T>, dim3(nb), dim3(256), 0, s, F, colour, 0, 1);
            hipLaunchKernelGGL(k_mg_smooth_cell<T>, dim3(nb), dim3(256), 0, s, F, colour, 0, 2);
        } else {
            hipLaunchKernelGGL(k_mg_smooth_cell<T>, dim3(nb), dim3(256), 0, s, F, colour, 0, 0);
        }
    };
    hipLaunchKernelGGL(k_mg_smooth_cell<T>, dim3(nb), dim3(256), 0, s, F, 0, 1, 0);
    half_sweep(1);
    half_sweep(0);
    half_sweep(1);
    hipLaunchKernelGGL(k_mg_restrict<T>, dim3(cdiv(C.n, 256)), dim3(256), 0, s, F, C);
    launch_mg_vcycle(s, L, nlev, l + 1);
    hipLaunchKernelGGL(k_mg_prolong<T>, dim3(nb), dim3(256), 0, s, F, C);
    for (int q = 0; q < 2; ++q) {
        half_sweep(0);
        half_sweep(1);
    }
}

static inline int lin_blocks(const Geo &g)
{
    return g.xcd_remap ? ((g.nblocks + 7) / 8) * 8 : g.nblocks;
}

template <typename T>
void launch_pb_spmv(const Geo &g, hipStream_t s, const MGLevelT<T> &L0, int ns, const T *in,
                    T *out, const T *w, double *part, const PBState *st)
{
    // four cells of a z-row per thread when rows hold whole fours (kPerBlock = 4 * 256,
    // so each block still covers the same 1024 cells)
    const bool by4 = (L0.nz % 4) == 0 && kPerBlock == 4 * kThreads;
    if (ns == 1) {
        if (by4)
            hipLaunchKernelGGL((k_pb_spmv4<1, T>), dim3(lin_blocks(g)), dim3(kThreads), 0, s, g,
                               L0, in, out, w, part, st);
        else
            hipLaunchKernelGGL((k_pb_spmv<1, T>), dim3(lin_blocks(g)), dim3(kThreads), 0, s, g,
                               L0, in, out, w, part, st);
    } else {
        if (by4)
            hipLaunchKernelGGL((k_pb_spmv4<2, T>), dim3(lin_blocks(g)), dim3(kThreads), 0, s, g,
                               L0, in, out, w, part, st);
        else
            hipLaunchKernelGGL((k_pb_spmv<2, T>), dim3(lin_blocks(g)), dim3(kThreads), 0, s, g,
                               L0, in, out, w, part, st);
    }
}

template <typename T>
void launch_pb_update_p(const Geo &g, hipStream_t s, int first, const T *r, const T *v, T *p,
                        const PBState *st)
{
    hipLaunchKernelGGL(k_pb_update_p<T>, dim3(std::min(2048, cdiv(g.N, 256))), dim3(256), 0, s, g,
                       first, r, v, p, st);
}

template <typename T>
void launch_pb_update_s(const Geo &g, hipStream_t s, const double *part, const T *r, const T *v,
                        T *sv, PBState *st)
{
    if (g.nblocks <= kPBFoldEach) {
        hipLaunchKernelGGL((k_pb_update_s<T, true>), dim3(std::min(2048, cdiv(g.N, kThreads))),
                           dim3(kThreads), 0, s, g, part, r, v, sv, st);
        return;
    }
    hipLaunchKernelGGL(k_pb_alpha, dim3(1), dim3(kThreads), 0, s, g, part, st);
    hipLaunchKernelGGL((k_pb_update_s<T, false>), dim3(2048), dim3(kThreads), 0, s, g, part, r, v,
                       sv, st);
}

template <typename T>
void launch_pb_update_xr(const Geo &g, hipStream_t s, int first, const double *part_in,
                         const T *ph, const T *sh, const T *sv, const T *t, const T *r0,
                         double *e, T *r, double *part_out, PBState *st)
{
    const bool fold = g.nblocks <= kPBFoldEach;
    if (!fold) hipLaunchKernelGGL(k_pb_omega, dim3(1), dim3(kThreads), 0, s, g, part_in, st);
    auto run = [&](auto k) {
        hipLaunchKernelGGL(k, dim3(lin_blocks(g)), dim3(kThreads), 0, s, g, part_in, ph, sh, sv,
                           t, r0, e, r, part_out, st);
    };
    if (first) run(fold ? k_pb_update_xr<T, true, true> : k_pb_update_xr<T, true, false>);
    else run(fold ? k_pb_update_xr<T, false, true> : k_pb_update_xr<T, false, false>);
}

void launch_pb_end(const Geo &g, hipStream_t s, const double *part, PBState *st, PBState *host)
{
    hipLaunchKernelGGL(k_pb_end, dim3(1), dim3(kThreads), 0, s, g, part, st, host);
}

#define CFDMX_MG_INSTANCES(T)                                                                 \
    template void mg_plan<T>(MGLevelT<T> *, int);                                             \
    template void launch_mg_vcycle<T>(hipStream_t, const MGLevelT<T> *, int, int);            \
    template void launch_pb_spmv<T>(const Geo &, hipStream_t, const MGLevelT<T> &, int,       \
                                    const T *, T *, const T *, double *, const PBState *);    \
    template void launch_pb_update_p<T>(const Geo &, hipStream_t, int, const T *, const T *,  \
                                        T *, const PBState *);                                \
    template void launch_pb_update_s<T>(const Geo &, hipStream_t, const double *, const T *,  \
                                        const T *, T *, PBState *);                           \
    template void launch_pb_update_xr<T>(const Geo &, hipStream_t, int, const double *,       \
                                         const T *, const T *, const T *, const T *,          \
                                         const T *, double *, T *, double *, PBState *);
CFDMX_MG_INSTANCES(float)
CFDMX_MG_INSTANCES(double)
#undef CFDMX_MG_INSTANCES

} // namespace cfdmx
