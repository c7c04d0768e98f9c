// SPME reciprocal space (ewald_spole.F90:244-477, ewald_general.F90:517-869,
// bspline.F90:192-306, ewald_spole.F90:1257-1386) on the GPU.
//
//  k_spread_cells  one workgroup per link cell: B-splines of its atoms go to
//               LDS and each wavefront adds one atom's S^3 charge weights into
//               an LDS window of the grid (lanes over the (x, y) plane), which
//               is then added to the global grid.
//  k_splines, k_spread_tiles  the splines of every atom, then one workgroup per
//               mesh tile that sums the atoms of its list with FP64 matrix
//               instructions and stores each grid point once.
//  (fft.hip)    Q <- FFT-(theta . FFT+(Q)); theta(m) on the half spectrum
//               with the spherical cutoff 0.525 min_d K_d w*_d, and the
//               reciprocal stress.
//  k_gather     B-splines of a block's atoms staged in LDS; a group of lanes
//               per atom (lane = x column) reads the potential grid, a group
//               reduction gives the atom's energy and force.
//  k_finish     subtracts the mean reciprocal force (ewald_general.F90:857-864),
//               scales by 2*scale and adds into the total force.
// FP64 or FP32 (mixed) arithmetic; sums across lanes and atoms in FP64.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "common.h"
#include "device_util.h"

namespace dlpx {

struct SpmeParams {
    int K[3];
    float invK[3];          // 1/K (fast wrapping of grid indices)
    int K1h;
    int S;
    double kr[3];           // K as real
    double rcell[9];        // inverse cell (numerics.F90 invert)
    double rk[3];           // Matmul(reshape(rcell,[3,3]), K) (ewald_general.F90:770-771)
};

// bspline_splines_gen (bspline.F90:192-306) for one coordinate: order-S
// values M[t] and first derivatives D[t] at the S grid points
// floor(u) - S + 1 + t, t = 0..S-1, evaluated with the reference's recursion
// (S even in 4..16; the reference forces an even order, control.F90:1651-1675).
template <typename R, int S, bool DERIV2 = false>
__device__ __forceinline__ void bspline_low(R w, R *z, R *D2 = nullptr)
{
    R zd[S + 2];
#pragma unroll
    for (int j = 0; j < S + 2; j++) zd[j] = (R)0;
    // 1-based indices as in the reference: zd[1..S], zd[S+1] == 0
    zd[S] = w;
    zd[S - 1] = (R)1 - w;
#pragma unroll
    for (int k = S - 2; k >= 3; k--) {
        const R k_r = (R)(S - k + 1);
        const R km1_rr = (R)1 / (R)(S - k);
#pragma unroll
        for (int j = k; j <= S - 1; j++) {
            const R pt = w + (R)(S - j);
            zd[j] = (pt * zd[j] + (k_r - pt) * zd[j + 1]) * km1_rr;
        }
        zd[S] = zd[S] * w * km1_rr;
    }
    // l = 2 stage: second derivatives from order S-2 (z_j - 2 z_j+1 + z_j+2,
    // zd[S+1] = 0), then raise to order S-1
    {
        const R k_r = (R)(S - 1);
        const R km1_rr = (R)1 / (R)(S - 2);
#pragma unroll
        for (int j = 1; j <= S - 1; j++) {
            if (DERIV2) D2[j - 1] = (zd[j] - (R)2 * zd[j + 1]) + zd[j + 2];
            const R pt = w + (R)(S - j);
            zd[j] = (pt * zd[j] + (k_r - pt) * zd[j + 1]) * km1_rr;
        }
        if (DERIV2) D2[S - 1] = zd[S];
        zd[S] = zd[S] * w * km1_rr;
    }
#pragma unroll
    for (int j = 1; j <= S; j++) z[j - 1] = zd[j];
}
// l = 1 stage: first derivatives from the order S-1 values z, then order S
template <typename R, int S, bool DERIV>
__device__ __forceinline__ void bspline_top(const R *z, R w, R *M, R *D)
{
    const R k_r = (R)S;
    const R km1_rr = (R)1 / (R)(S - 1);
#pragma unroll
    for (int k = 0; k < S; k++) {
        if (DERIV) D[k] = k < S - 1 ? z[k] - z[k + 1] : z[k];
        const R pt = w + (R)(S - 1 - k);
        M[k] = k < S - 1 ? (pt * z[k] + (k_r - pt) * z[k + 1]) * km1_rr : z[k] * w * km1_rr;
    }
}
template <typename R, bool DERIV, int S, bool DERIV2 = false>
__device__ __forceinline__ void bspline(R w, R *M, R *D, R *D2 = nullptr)
{
    R z[S];
    bspline_low<R, S, DERIV2>(w, z, D2);
    bspline_top<R, S, DERIV>(z, w, M, D);
}

// Fractional grid coordinate of one axis, folded into [0, K) so an atom that
// drifted out of the cell is represented by its periodic image
// (ewald_spole.F90:364-387).
__device__ __forceinline__ void grid_coord(const SpmeParams &sp, int d, double x, double y, double z, int &idx,
                                           double &w)
{
    double u = sp.kr[d] * (sp.rcell[d] * x + sp.rcell[d + 3] * y + sp.rcell[d + 6] * z + 0.5);
    if (u < 0.0 || u >= sp.kr[d]) u -= sp.kr[d] * floor(u / sp.kr[d]);
    int i = (int)u;
    if (i >= sp.K[d]) i = sp.K[d] - 1;  // u rounded up to K after folding
    if (!(i >= 0)) i = 0;               // non-finite coordinates stay inside the grid
    idx = i;
    w = u - (double)i;
}

// Unwrapped fractional grid coordinate of one axis (no folding): the base
// grid point floor(u) - S + 1 may be negative or >= K; callers fold indices.
__device__ __forceinline__ double grid_u(const SpmeParams &sp, int d, double x, double y, double z)
{
    return sp.kr[d] * (sp.rcell[d] * x + sp.rcell[d + 3] * y + sp.rcell[d + 6] * z + 0.5);
}

// floor(u) for the spreading window, held within +-2^20: a coordinate far
// outside the cell (a diverging run) then still gives window bounds whose
// integer arithmetic cannot overflow (an overflowed bound passed the window's
// one-period test and indexed the grid out of range); such a window exceeds
// the mesh and takes the direct path, which wraps every index.  NaN maps to
// the lower bound (fmax returns the non-NaN operand).
__device__ __forceinline__ double spread_floor(double u)
{
    return fmin(fmax(floor(u), -1048576.0), 1048576.0);
}

// A value every lane of the wavefront holds, moved to scalar registers.
__device__ __forceinline__ float uniform_value(float v)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ double uniform_value(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffll)), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ int wrapk(int v, int K)
{
    v %= K;
    return v < 0 ? v + K : v;
}

constexpr int kSlabBytes = 32768;

// Charge spreading by link cell (one workgroup per cell of the sorted atom
// order): the cell's atoms touch a compact window of grid points, which is
// accumulated in LDS in z-slabs with LDS atomics and then added to the global
// grid with one atomic per window point, instead of S^3 global atomics per
// atom.  A window too large for LDS (very large cells, or atoms far outside
// their cell) falls back to per-atom global atomics for that cell.
//
// The window accumulates in FP64 at either precision: FP64 LDS atomic adds
// (ds_add_f64) sustain several times the rate of FP32 ones (ds_add_f32) on
// gfx950, and the FP32 grid then receives one rounding per window point.
// One workgroup per link cell gives only ~730 workgroups at 64k ions, so each
// needs many wavefronts to keep the LDS atomics busy: 512 threads in FP32;
// the FP64 build's register use makes 256 the better trade there (measured).
//
// The B-splines of up to spread_atoms() atoms are staged in LDS once and
// serve every z-slab; a cell with more atoms restages them per slab.  Each
// wavefront adds one atom at a time, lanes over the (x, y) points, with the
// atom's S z-weights held in registers so the S atomic adds of a lane issue
// back to back.
template <typename R>
constexpr int spread_threads()
{
    return sizeof(R) == 4 ? 512 : 256;
}
template <typename R, int S>
constexpr int spread_atoms()
{
    // 12 KB (FP32) or 18 KB (FP64) of staged splines: with the 32 KB slab,
    // three workgroups fit in a CU's LDS
    return (sizeof(R) == 8 ? 18432 : 12288) / (3 * S * (int)sizeof(R));
}
template <typename R>
struct SpreadArgs {
    const double4 *pos;
    const int32_t *cell_start;
    int ncell;
    SpmeParams sp;
    R *Q;
};
template <typename R, int S>
__device__ __forceinline__ void spread_body(const SpreadArgs<R> &sa, int c)
{
    constexpr int kCap = kSlabBytes / (int)sizeof(double);
    constexpr int NA = spread_atoms<R, S>();
    constexpr int NT = spread_threads<R>();
    __shared__ double slab[kCap];
    __shared__ R sM[3][NA][S];
    __shared__ int sB[3][NA];
    __shared__ R sQ[NA];
    __shared__ int wlo[3], whi[3];
    const double4 *__restrict__ pos = sa.pos;
    const int32_t *__restrict__ cell_start = sa.cell_start;
    const SpmeParams &sp = sa.sp;
    R *__restrict__ Q = sa.Q;
    const int t = threadIdx.x, wid = t >> 6, lane = t & 63;
    if (c >= sa.ncell) return;
    const int s0 = cell_start[c], n = cell_start[c + 1] - s0;
    if (n <= 0) return;
    if (t < 3) {
        wlo[t] = 0x7fffffff;
        whi[t] = -0x7fffffff;
    }
    __syncthreads();
    // window bounds; a cell whose atoms all fit the staging arrays has their
    // B-splines, base points and charges staged in the same pass (one read of
    // the positions)
    const bool once = n <= NA;
    // per-thread bounds, reduced across the wavefront before one LDS atomic
    // per wavefront: atomics of every atom on the same six LDS words
    // serialise (measured: 9 us of the kernel at 64k ions)
    int bmin[3] = {0x7fffffff, 0x7fffffff, 0x7fffffff}, bmax[3] = {-0x7fffffff, -0x7fffffff, -0x7fffffff};
    for (int k = t; k < n; k += NT) {
        const double4 p = pos[s0 + k];
        for (int d = 0; d < 3; d++) {
            const double u = grid_u(sp, d, p.x, p.y, p.z);
            const double fl = spread_floor(u);
            const int b = (int)fl - S + 1;
            bmin[d] = min(bmin[d], b);
            bmax[d] = max(bmax[d], b);
            if (once) {
                R M[S];
                bspline<R, false, S>((R)(u - fl), M, nullptr);
#pragma unroll
                for (int m = 0; m < S; m++) sM[d][k][m] = M[m];
                sB[d][k] = b;
            }
        }
        if (once) sQ[k] = (R)p.w;
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            bmin[d] = min(bmin[d], __shfl_xor(bmin[d], o, 64));
            bmax[d] = max(bmax[d], __shfl_xor(bmax[d], o, 64));
        }
        if (lane == 0 && bmin[d] <= bmax[d]) {
            atomicMin(&wlo[d], bmin[d]);
            atomicMax(&whi[d], bmax[d]);
        }
    }
    __syncthreads();
    const int lo0 = wlo[0], lo1 = wlo[1], lo2 = wlo[2];
    // window extents in 64-bit so that non-finite coordinates cannot overflow
    const long ex = (long)whi[0] - lo0 + S, ey = (long)whi[1] - lo1 + S, ez = (long)whi[2] - lo2 + S;
    const bool tile = ex <= sp.K[0] && ey <= sp.K[1] && ez <= sp.K[2] && ex * ey <= kCap;
    const int Wx = tile ? (int)ex : 0, Wy = tile ? (int)ey : 0, Wz = tile ? (int)ez : 1;
    const int Dz = tile ? min(Wz, kCap / (Wx * Wy)) : Wz;
    const int plane = Wx * Wy;
    // B-splines, base points and charges of atoms a0 .. a0+NA-1 into LDS
    auto stage = [&](int a0) {
        for (int k = t; k < 3 * NA; k += NT) {
            const int d = k / NA, a = k % NA;
            if (a0 + a < n) {
                const double4 p = pos[s0 + a0 + a];
                const double u = grid_u(sp, d, p.x, p.y, p.z);
                const double fl = spread_floor(u);
                R M[S];
                bspline<R, false, S>((R)(u - fl), M, nullptr);
#pragma unroll
                for (int m = 0; m < S; m++) sM[d][a][m] = M[m];
                sB[d][a] = (int)fl - S + 1;
                if (d == 0) sQ[a] = (R)p.w;
            }
        }
    };
    for (int z0 = 0; z0 < Wz; z0 += Dz) {
        if (tile) {
            if (z0 > 0) __syncthreads();  // the previous slab's flush has read the slab
            for (int k = t; k < plane * Dz; k += NT) slab[k] = 0.0;
        }
        for (int a0 = 0; a0 < n; a0 += NA) {
            __syncthreads();
            if (!once) {
                stage(a0);
                __syncthreads();
            }
            const int na = min(NA, n - a0);
            for (int a = wid; a < na; a += NT / 64) {
                // the atom's charge as a wavefront-uniform value: the skip below
                // is then a scalar branch
                const R q = uniform_value(sQ[a]);
                if (fabs((double)q) <= kZeroPlus) continue;
                // one atom per wavefront: its base point and z-range are scalars,
                // so the per-z tests below are scalar branches, not exec masks
                const int bx = __builtin_amdgcn_readfirstlane(sB[0][a]);
                const int by = __builtin_amdgcn_readfirstlane(sB[1][a]);
                const int bz = __builtin_amdgcn_readfirstlane(sB[2][a]);
                // spline points of this atom inside the current z-slab
                const int tz0 = tile ? max(0, z0 + lo2 - bz) : 0;
                const int tz1 = tile ? min(S, z0 + lo2 + Dz - bz) : S;
                if (tz0 >= tz1) continue;
                R mz[S];
#pragma unroll
                for (int m = 0; m < S; m++) mz[m] = q * sM[2][a][m];
                for (int pp = lane; pp < S * S; pp += 64) {
                    const int tx = pp % S, ty = pp / S;
                    const R mxy = sM[0][a][tx] * sM[1][a][ty];
                    if (tile) {
                        // slab index of spline point tz = 0 (points outside the slab are skipped);
                        // the slab's spline points as a scalar bit mask, one bit test per point
                        const int l0 = (bz - lo2 - z0) * plane + (by + ty - lo1) * Wx + (bx + tx - lo0);
                        const unsigned zm = ((1u << tz1) - 1u) & ~((1u << tz0) - 1u);
#pragma unroll
                        for (int tz = 0; tz < S; tz++)
                            if (zm & (1u << tz)) atomicAdd(&slab[l0 + tz * plane], (double)(mz[tz] * mxy));
                    } else {
                        const int gx = wrapk(bx + tx, sp.K[0]), gy = wrapk(by + ty, sp.K[1]);
#pragma unroll
                        for (int tz = 0; tz < S; tz++) {
                            const int gz = wrapk(bz + tz, sp.K[2]);
                            unsafeAtomicAdd(&Q[((size_t)gz * sp.K[1] + gy) * sp.K[0] + gx], mz[tz] * mxy);
                        }
                    }
                }
            }
        }
        __syncthreads();
        if (!tile) break;  // the direct path did every z at once
        const int dz = min(Dz, Wz - z0);
        // window coordinates within one period of the grid (always, for
        // positions near the cell) wrap with one compare
        const bool near = lo0 >= -sp.K[0] && lo1 >= -sp.K[1] && lo2 >= -sp.K[2] && lo0 + Wx <= 2 * sp.K[0] &&
                          lo1 + Wy <= 2 * sp.K[1] && lo2 + Wz <= 2 * sp.K[2];
        if (near && Wx <= 64) {
            // one (y, z) row of the slab per group of 32 or 64 lanes, lanes over x
            const int LW = Wx <= 32 ? 32 : 64, lx = lane & (LW - 1);
            auto fold = [](int v, int K) { return v < 0 ? v + K : (v >= K ? v - K : v); };
            const int gx = fold(lo0 + lx, sp.K[0]);
            for (int row = wid * (64 / LW) + lane / LW; row < Wy * dz; row += NT / LW) {
                const int lz = row / Wy, ly = row - lz * Wy;
                const R v = lx < Wx ? (R)slab[row * Wx + lx] : (R)0;
                if (v == (R)0) continue;
                const int gy = fold(lo1 + ly, sp.K[1]), gz = fold(lo2 + z0 + lz, sp.K[2]);
                unsafeAtomicAdd(&Q[((size_t)gz * sp.K[1] + gy) * sp.K[0] + gx], v);
            }
            continue;
        }
        const float iWx = 1.0f / (float)Wx, iWy = 1.0f / (float)Wy;
        // the float-reciprocal wrap is exact for window coordinates below 2^20
        // in magnitude
        const bool small = abs(lo0) < (1 << 19) && abs(lo1) < (1 << 19) && abs(lo2) < (1 << 19);
        for (int k = t; k < plane * dz; k += NT) {
            const R v = (R)slab[k];
            if (v == (R)0) continue;
            int lx, ly, gx, gy, gz;
            const int lz = fdiv_floor(fdiv_floor(k, Wx, iWx, lx), Wy, iWy, ly);
            if (small) {
                (void)fdiv_floor(lo0 + lx, sp.K[0], sp.invK[0], gx);
                (void)fdiv_floor(lo1 + ly, sp.K[1], sp.invK[1], gy);
                (void)fdiv_floor(lo2 + z0 + lz, sp.K[2], sp.invK[2], gz);
            } else {
                gx = wrapk(lo0 + lx, sp.K[0]);
                gy = wrapk(lo1 + ly, sp.K[1]);
                gz = wrapk(lo2 + z0 + lz, sp.K[2]);
            }
            unsafeAtomicAdd(&Q[((size_t)gz * sp.K[1] + gy) * sp.K[0] + gx], v);
        }
    }
}

template <typename R, int S>
__global__ void __launch_bounds__(spread_threads<R>()) k_spread_cells(SpreadArgs<R> a)
{
    spread_body<R, S>(a, xcd_block(blockIdx.x, gridDim.x));
}
template <typename R, int S>
__global__ void __launch_bounds__(spread_threads<R>()) k_spread_cells_batch(const SpreadArgs<R> *__restrict__ av,
                                                                            const int32_t *__restrict__ boff,
                                                                            int nsys)
{
    BatchPos bp;
    if (!batch_pos(boff, nsys, bp)) return;
    const SpreadArgs<R> &a = av[bp.s];
    spread_body<R, S>(a, bp.b);
}

// The spline data of every atom, once per evaluation, for the spreading by
// tiles (where an atom is met in about four tiles): per axis
// the order S-1 values z[0..S-1] that the last step of the recursion
// (bspline) turns into the values and first derivatives of order S,
//   M[t] = (pt z[t] + (S - pt) z[t+1]) / (S - 1), pt = w + S - 1 - t,
//   D[t] = z[t] - z[t+1]   (z[S] = 0),
// in [atom][axis][S]; {w_x, w_y, w_z, charge}; and the folded grid points
// {floor(u_x), floor(u_y), floor(u_z), whether the atom has a charge}.
//
// When an atom has moved further than the tiles' lists allow for (F_STRAY), the
// lists are not used.  Up to kStrayTest atoms every tile then tests every atom;
// with more, each charged atom is put here on the lists of the tiles that it
// reaches, by an atomic count per tile (which the upload has cleared), in any
// order.  A force call on such positions, tested and listed: 4,096 ions, mixed,
// 127 and 167 us (the counts' atomics, and lists without y order), 21,952 272 and
// 286, 27,000 286 and 281, 46,656 478 and 375; 1,728,000 ions 116 and 11.1 ms.
template <typename R> struct R4T;
template <> struct R4T<double> { using type = double4; };
template <> struct R4T<float> { using type = float4; };
template <typename R>
struct SplineArgs {
    const double4 *pos;
    int n;
    SpmeParams sp;
    R *z, *wq;
    ushort4 *base;
    const int32_t *flags;
    int32_t no;                 // upload whose strays matter (F_STRAY), 0: none
    int32_t *list, *found;      // the tiles' lists and, for strays, the atoms found for each
    int cap, tiles[3];
};
constexpr int kTileX = 16, kTileY = 8, kTileZ = 16;
template <typename R, int S, bool STRAYS>
__device__ __forceinline__ void splines_body(const SplineArgs<R> &a, int bid)
{
    const int k = bid * 256 + threadIdx.x, i = k / 3, d = k - 3 * i;
    if (i >= a.n) return;
    const double4 p = a.pos[i];
    int idx;
    double w;
    grid_coord(a.sp, d, p.x, p.y, p.z, idx, w);
    R z[S];
    bspline_low<R, S>((R)w, z);
    R *out = a.z + (size_t)k * S;
#pragma unroll
    for (int m = 0; m < S; m++) out[m] = z[m];
    a.wq[4 * (size_t)i + d] = (R)w;
    unsigned short *b = (unsigned short *)(a.base + i);
    b[d] = (unsigned short)idx;
    if (d == 0) {
        a.wq[4 * (size_t)i + 3] = (R)p.w;
        b[3] = fabs(p.w) > kZeroPlus ? 1 : 0;
        if (STRAYS && a.no != 0 && a.flags[F_STRAY] == a.no && b[3]) {
            // the tiles of the atom's S points from floor(u) - S + 1 on, per axis
            constexpr int T[3] = {kTileX, kTileY, kTileZ}, MT = 2 + (S + 6) / 8;
            int tl[3][MT], nt[3];
#pragma unroll
            for (int x = 0; x < 3; x++) {
                int g = idx;
                if (x > 0) grid_coord(a.sp, x, p.x, p.y, p.z, g, w);
                g -= S - 1;
                if (g < 0) g += a.sp.K[x];
                nt[x] = 0;
                for (int left = S; left > 0 && nt[x] < MT;) {
                    const int tile = g / T[x], step = min((tile + 1) * T[x], a.sp.K[x]) - g;
                    tl[x][nt[x]++] = tile;
                    left -= step;
                    g += step;
                    if (g >= a.sp.K[x]) g = 0;
                }
            }
            for (int q2 = 0; q2 < nt[2]; q2++)
                for (int q1 = 0; q1 < nt[1]; q1++)
                    for (int q0 = 0; q0 < nt[0]; q0++) {
                        const int tile = (tl[2][q2] * a.tiles[1] + tl[1][q1]) * a.tiles[0] + tl[0][q0];
                        const int slot = atomicAdd(&a.found[tile], 1);
                        if (slot < a.cap) a.list[(size_t)tile * a.cap + slot] = i;
                    }
        }
    }
}
template <typename R, int S>
__global__ void __launch_bounds__(256) k_splines(SplineArgs<R> a) { splines_body<R, S, true>(a, blockIdx.x); }
template <typename R, int S>
__global__ void __launch_bounds__(256) k_splines_batch(const SplineArgs<R> *__restrict__ av,
                                                       const int32_t *__restrict__ boff, int nsys)
{
    const int lb = blockIdx.x;
    if (lb >= boff[nsys]) return;
    const int s = batch_find(boff, nsys, lb);
    splines_body<R, S, false>(av[s], lb - boff[s]);  // a resident run's atoms never stray
}
// Charge spreading by mesh tiles: one workgroup per tile of kTileX x kTileY x
// kTileZ grid points sums every atom that reaches into it and stores each
// point once, so the grid needs no atomics and no clearing.  Over the atoms,
// a y plane of the tile is a product of matrices,
//   Q[z][x] = sum_a (q_a Mz_a[z]) (Mx_a[x] My_a[y]),
// 16 x 16 outputs with the atoms as the contracted index: one FP64 matrix
// instruction adds four atoms to a plane (FP64 in both precision modes, as
// the LDS window of k_spread_cells is).  Each wavefront holds kTilePlanes.
//
// The atoms come from the tile's own list, made when the Verlet list is: every
// atom of the bins in reach that comes within half the Verlet padding of the
// tile's reach (its points and S - 1 below them); no atom moves further
// without a rebuild.  A host that evaluates such positions all the same, or in
// another cell, is noticed at the upload, which holds every atom's displacement
// against the same bound (F_STRAY), and then the lists are not used (k_splines).
// The splines of a chunk of kTileChunk atoms are laid out in LDS over the tile's points
// with zeros outside, while the next chunk's are being loaded; each chunk of
// the list is in y order, so that a wavefront only meets the groups of four
// that reach its planes.
//
// Bound by instruction issue: an FP64 matrix instruction takes the FP64
// vector unit's time (64 cycles for 1024 multiply-adds, the rate of the vector
// unit), about a tenth of them useful (an atom's 8 x 8 points of a 16 x 16
// plane, 2.1 tile columns an atom at S = 8), 8 us at 64,000 ions; laying out
// a chunk costs about as much.  With the splines' own kernel, against
// k_spread_cells (LDS atomics, one atom per wavefront at a time):
// 64,000 ions, 128^3, S = 8 mixed 29 against 50 us, FP64 35 against 75;
// 1,728,000 ions mixed 532 against 894; 10,296 ions, S = 6 FP64 14 against
// 31; 1,000 ions, 32^3 mixed 14 against 38.  One wavefront per 16 atoms with
// all eight planes, no barriers and a last exchange of planes: 38 against 29
// (190 registers); 16 planes to a tile: 40 against 34; a wavefront's bounds of
// 5 per SIMD keep the list making's registers off the rest (1,728,000 ions
// 593 -> 546).
constexpr int kTileThreads = 256, kTileChunk = 64;
constexpr int kTilePlanes = kTileY / (kTileThreads / 64);
constexpr int kTileScan = 2;     // candidates a thread tests per round of a list's making
constexpr int kTileBins = 1024;  // most bins within a tile's reach
constexpr int kStrayTest = 24576; // most atoms that every tile tests when some have strayed (k_splines)
template <typename R>
struct TileArgs {
    const R *z, *wq;        // the atoms' splines and grid points (k_splines)
    const ushort4 *base;
    int n;
    const int32_t *start;   // first atom of each bin
    CellGrid g;             // sub: 1 bins are link cells, 2 subcells
    int bins[3], tiles[3];
    int32_t *list, *count;  // cap atoms per tile; their number, -1 none
    const int32_t *found;   // of strays, the atoms k_splines found for each tile; null: it looked for none
    int cap;
    const double4 *xref;    // the positions of the list build, in a cell of
    double invL0[3];        // these reciprocal edges
    double drift_k[3];      // grid points an atom moves from there at most
    int slack[3];           // and floor(u) changes by
    const int32_t *upd;     // nonzero: the Verlet list is new (may be null)
    int fresh;              // so it is
    const int32_t *flags;
    int32_t no;             // upload whose strays matter (F_STRAY), 0: none
    SpmeParams sp;
    R *Q;
};
// Barrier for data exchanged through LDS: global loads stay in flight.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
__device__ __forceinline__ int lanes_before(unsigned long long mask)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}
template <typename R, int S, bool STRAYS>
__device__ __forceinline__ void spread_tile_body(const TileArgs<R> &a, int b)
{
    typedef double double4v __attribute__((ext_vector_type(4)));
    constexpr int T[3] = {kTileX, kTileY, kTileZ}, NW = kTileThreads / 64, PW = kTilePlanes;
    // a chunk's splines over the tile's points, an atom per row: z, x, y (the
    // odd stride puts a column's rows on distinct banks)
    constexpr int OX = 16, OY = 32, RS = OY + kTileY + 1;
    static_assert(kTileX == 16 && kTileZ == 16, "planes of 16 x 16");
    __shared__ double rows[kTileChunk * RS];
    __shared__ int sOy[kTileChunk];
    __shared__ int s_start[kTileBins], s_off[kTileBins];  // the making of a list
    __shared__ int wcnt[kTileScan][NW];
    const SpmeParams &sp = a.sp;
    const int t = threadIdx.x, lane = t & 63, wid = __builtin_amdgcn_readfirstlane(t >> 6);
    const int tc[3] = {b % a.tiles[0], (b / a.tiles[0]) % a.tiles[1], b / (a.tiles[0] * a.tiles[1])};
    int t0[3], reach[3];  // first point; largest floor(u) - t0 of an atom that reaches the tile
#pragma unroll
    for (int d = 0; d < 3; d++) {
        t0[d] = tc[d] * T[d];
        reach[d] = min(T[d], sp.K[d] - t0[d]) + S - 2;
    }
    int32_t *const list = a.list + (size_t)b * a.cap;
    double4v acc[PW];
#pragma unroll
    for (int p = 0; p < PW; p++) acc[p] = (double4v){0.0, 0.0, 0.0, 0.0};

    // wavefronts 0-2 hold one axis each of a chunk's atoms, an atom per lane
    const int d = wid < 3 ? wid : 0;
    const int td = d == 0 ? t0[0] : d == 1 ? t0[1] : t0[2], rd = d == 0 ? reach[0] : d == 1 ? reach[1] : reach[2];
    const int kd = d == 0 ? sp.K[0] : d == 1 ? sp.K[1] : sp.K[2], sd = d == 0 ? a.slack[0] : d == 1 ? a.slack[1] : a.slack[2];
    // first point of an atom's spline relative to the tile's, the image in reach
    auto offset = [](int idx, int t, int r, int K, int slack) {
        int rel = idx - t;
        if (rel < -slack) rel += K;
        else if (rel > r + slack) rel -= K;
        return rel - (S - 1);
    };
    R z[S], w = (R)0, q = (R)0;
    int id = 0;
    auto fetch = [&](int j) {  // the splines of atom j
        if (wid < 3) {
            const R *zp = a.z + ((size_t)j * 3 + d) * S;
#pragma unroll
            for (int k = 0; k < S; k++) z[k] = zp[k];
            w = a.wq[4 * (size_t)j + d];
            q = a.wq[4 * (size_t)j + 3];
            id = ((const unsigned short *)(a.base + j))[d];
        }
    };
    // the splines of the m fetched atoms over the tile's points
    double *const row = rows + lane * RS + (d == 0 ? OX : d == 1 ? OY : 0);
    auto lay = [&](int m) {
        if (wid < 3) {
            const bool on = lane < m;
            const int od = offset(id, td, rd, kd, sd);
            const unsigned len = d == 1 ? kTileY : 16;
#pragma unroll
            for (int k = 0; k < 16; k++)
                if (d != 1 || k < kTileY) row[k] = 0.0;
            if (d == 1) sOy[lane] = on ? od : 1 << 20;
            R M[S];
            bspline_top<R, S, false>(z, w, M, nullptr);
            const R f = d == 2 ? q : (R)1;
            // points outside the tile go to the row's padding: a select, not a branch
            const unsigned lim = on ? len : 0u;
            double *const pad = rows + lane * RS + RS - 1;
#pragma unroll
            for (int k = 0; k < S; k++) {
                double *const out = (unsigned)(od + k) < lim ? row + od + k : pad;
                *out = (double)(f * M[k]);
            }
        }
    };
    // the laid-out atoms into this wavefront's planes: the groups of four from
    // the first to the last that reach one of them (a chunk is in y order), the
    // next group's values read while the matrix unit adds the present one's
    const double *const pzx = rows + (lane >> 4) * RS + (lane & 15), *const py = rows + (lane >> 4) * RS + OY + PW * wid;
    struct Group {
        double z, x, y[PW];
    };
    auto add = [&]() {
        const int oy = sOy[lane], y0 = PW * wid;
        const unsigned long long any = __ballot(oy <= y0 + PW - 1 && oy + S - 1 >= y0);
        if (any == 0) return;
        const int first = __builtin_ctzll(any) >> 2, last = (63 - __builtin_clzll(any)) >> 2;
        auto read = [&](int g, Group &v) {
            const int h = 4 * min(g, kTileChunk / 4 - 1) * RS;
            v.z = pzx[h];
            v.x = pzx[h + OX];
#pragma unroll
            for (int p = 0; p < PW; p++) v.y[p] = py[h + p];
            __builtin_amdgcn_sched_barrier(0);  // not sunk to their use
        };
        auto mul = [&](const Group &v) {
            double dy[PW];
#pragma unroll
            for (int p = 0; p < PW; p++) dy[p] = v.x * v.y[p];
#pragma unroll
            for (int p = 0; p < PW; p++) acc[p] = __builtin_amdgcn_mfma_f64_16x16x4f64(v.z, dy[p], acc[p], 0, 0, 0);
        };
        Group va, vb;
        read(first, va);
        for (int g = first; g <= last; g += 2) {
            read(g + 1, vb);
            mul(va);
            if (g + 1 > last) break;
            read(g + 2, va);
            mul(vb);
        }
    };
    // the n atoms of the list into the tile
    auto sum = [&](int n) {
        int jn = lane < n ? list[lane] : 0;
        if (n > 0) fetch(jn);
        if (n > kTileChunk) jn = list[min(kTileChunk + lane, n - 1)];
        for (int h = 0; h < n; h += kTileChunk) {
            lay(min(kTileChunk, n - h));
            if (h + kTileChunk < n) {
                fetch(jn);
                jn = list[min(h + 2 * kTileChunk + lane, n - 1)];
            }
            lds_barrier();
            add();
            lds_barrier();
        }
    };

    // each chunk of the list put in y order, as its atoms are placed now, so
    // that the four atoms of a matrix instruction reach about the same planes
    auto order = [&](int n) {
        for (int h = wid * kTileChunk; h < n; h += NW * kTileChunk) {
            const bool on = h + lane < n;
            const int j = on ? list[h + lane] : 0;
            const int oy = offset(a.base[j].y, t0[1], reach[1], sp.K[1], a.slack[1]);
            // the atom's place, from the lanes with a smaller key and the
            // earlier ones with the same (lanes past n last)
            const int key = on ? min(max(oy + S, 0), 62) : 63;
            unsigned long long less = 0, same = ~0ull;
#pragma unroll
            for (int bit = 5; bit >= 0; bit--) {
                const bool one = key >> bit & 1;
                const unsigned long long m1 = __ballot(one);
                less |= one ? same & ~m1 : 0ull;
                same &= one ? m1 : ~m1;
            }
            if (on) list[h + __popcll(less) + lanes_before(same)] = j;
        }
        __syncthreads();
    };

    // strays: the lists k_splines made, and every atom tested for a tile whose
    // list they outgrew
    const bool all = STRAYS && a.no != 0 && a.flags[F_STRAY] == a.no;
    const bool fresh = a.fresh != 0 || (a.upd && *a.upd != 0);
    const int have = all ? (a.found ? a.found[b] : -1) : fresh ? -1 : a.count[b];
    if (have >= 0 && (!STRAYS || have <= a.cap)) {
        if (all && t == 0) a.count[b] = -1;
        sum(have);
    } else {
        // the list made anew, from the bins within reach
        int ncand = a.n, nq = 0;  // candidates; entries of s_off
        if (!all) {
            int nb[3], b0[3];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const double per = (double)a.bins[k] / (double)sp.K[k];
                const int lo = (int)floor((t0[k] - a.drift_k[k]) * per);
                const int hi = (int)floor((t0[k] + reach[k] + 1 + a.drift_k[k]) * per);
                nb[k] = min(hi - lo + 1, a.bins[k]);
                b0[k] = lo;
            }
            // bin q of the reach, y fastest, so that a chunk holds every y (a
            // thread takes bins U t .. U t + U-1, U as small as holds them)
            constexpr int UM = kTileBins / kTileThreads;
            const int nreg = nb[0] * nb[1] * nb[2], U = (nreg + kTileThreads - 1) / kTileThreads;
            const float iby = 1.0f / (float)nb[1], ibx = 1.0f / (float)nb[0];
            int cnt[UM], tot = 0;
#pragma unroll
            for (int u = 0; u < UM; u++) {
                cnt[u] = 0;
                const int qb = U * t + u;
                if (u < U && qb < nreg) {
                    int o[3];
                    o[2] = fdiv_floor(fdiv_floor(qb, nb[1], iby, o[1]), nb[0], ibx, o[0]);
#pragma unroll
                    for (int k = 0; k < 3; k++) {
                        o[k] += b0[k];
                        if (o[k] < 0) o[k] += a.bins[k];
                        if (o[k] >= a.bins[k]) o[k] -= a.bins[k];
                    }
                    const int key = a.g.sub == 2 ? subcell_key(a.g, o[0], o[1], o[2])
                                                 : (o[2] * a.g.nc[1] + o[1]) * a.g.nc[0] + o[0];
                    const int st = a.start[key];
                    cnt[u] = a.start[key + 1] - st;
                    s_start[qb] = st;
                }
                tot += cnt[u];
            }
            int incl = tot;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(incl, o, 64);
                if (lane >= o) incl += y;
            }
            if (lane == 63) wcnt[0][wid] = incl;
            __syncthreads();
            int run = incl - tot;
            for (int v = 0; v < wid; v++) run += wcnt[0][v];
            ncand = 0;
            for (int v = 0; v < NW; v++) ncand += wcnt[0][v];
#pragma unroll
            for (int u = 0; u < UM; u++)
                if (u < U) {
                    s_off[U * t + u] = run;
                    run += cnt[u];
                }
            nq = U * kTileThreads;
            __syncthreads();
        }
        int fill = 0;
        bool whole = !all;  // the list so far holds every atom found
        for (int c0 = 0; c0 < ncand; c0 += kTileScan * kTileThreads) {
            int j[kTileScan];
            double at[kTileScan][3];  // where the atom was at the list build, or is if it is looked for anywhere
#pragma unroll
            for (int u = 0; u < kTileScan; u++) {
                j[u] = min(c0 + u * kTileThreads + t, ncand - 1);
                if (!all) {
                    int lo = 0;  // the last bin with off[lo] <= j
#pragma unroll
                    for (int s = kTileBins / 2; s > 0; s >>= 1)
                        if (lo + s < nq && s_off[lo + s] <= j[u]) lo += s;
                    j[u] = s_start[lo] + (j[u] - s_off[lo]);
                }
            }
#pragma unroll
            for (int u = 0; u < kTileScan; u++) {
                if (all) {
                    const ushort4 pb = a.base[j[u]];
                    const R *w = a.wq + 4 * (size_t)j[u];
                    at[u][0] = pb.x + (double)w[0];
                    at[u][1] = pb.y + (double)w[1];
                    at[u][2] = pb.z + (double)w[2];
                } else {
                    const double4 p = a.xref[j[u]];
                    at[u][0] = p.x;
                    at[u][1] = p.y;
                    at[u][2] = p.z;
                }
            }
            unsigned long long mask[kTileScan];
#pragma unroll
            for (int u = 0; u < kTileScan; u++) {
                bool in = c0 + u * kTileThreads + t < ncand;
#pragma unroll
                for (int x = 0; x < 3; x++) {
                    double rel = (all ? at[u][x] : sp.kr[x] * (at[u][x] * a.invL0[x] + 0.5)) - t0[x];
                    if (rel < -a.drift_k[x]) rel += sp.K[x];
                    else if (rel >= sp.K[x] - a.drift_k[x]) rel -= sp.K[x];  // just below the tile's first point
                    in = in && !(rel >= reach[x] + 1 + a.drift_k[x]);
                }
                mask[u] = __ballot(in);
                if (lane == 0) wcnt[u][wid] = __popcll(mask[u]);
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kTileScan; u++)
#pragma unroll
                for (int v = 0; v < NW; v++) {
                    if (v == wid && (mask[u] >> lane & 1)) list[fill + lanes_before(mask[u])] = j[u];
                    fill += wcnt[u][v];
                }
            __syncthreads();
            if (fill + kTileScan * kTileThreads > a.cap && c0 + kTileScan * kTileThreads < ncand) {
                // no room for another round: what is there goes into the tile now
                order(fill);
                sum(fill);
                fill = 0;
                whole = false;
            }
        }
        if (t == 0) a.count[b] = whole ? fill : -1;
        order(fill);
        sum(fill);
    }
    // lane l of plane y holds x = l % 16 and z = 4 r + l / 16, r = 0..3
    const int gx = t0[0] + (lane & 15);
#pragma unroll
    for (int p = 0; p < PW; p++) {
        const int gy = t0[1] + PW * wid + p;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int gz = t0[2] + 4 * r + (lane >> 4);
            if (gx < sp.K[0] && gy < sp.K[1] && gz < sp.K[2])
                a.Q[((size_t)gz * sp.K[1] + gy) * sp.K[0] + gx] = (R)acc[p][r];
        }
    }
}
template <typename R, int S>
__global__ void __launch_bounds__(kTileThreads, 5) k_spread_tiles(TileArgs<R> a)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    if (b < a.tiles[0] * a.tiles[1] * a.tiles[2]) spread_tile_body<R, S, true>(a, b);
}
template <typename R, int S>
__global__ void __launch_bounds__(kTileThreads, 5) k_spread_tiles_batch(const TileArgs<R> *__restrict__ av,
                                                                     const int32_t *__restrict__ boff, int nsys)
{
    BatchPos bp;
    if (!batch_pos(boff, nsys, bp)) return;
    spread_tile_body<R, S, false>(av[bp.s], bp.b);
}

// Lanes per atom in the gather: the next power of two >= S, lane tx < S
// taking the grid column x = base + tx.
constexpr int gather_lanes(int S) { return S <= 4 ? 4 : S <= 8 ? 8 : 16; }

// Force interpolation (ewald_general.F90:776-855).  A group of gather_lanes(S)
// lanes serves one atom: lane tx reads the S x S (y, z) potential values of
// its grid column, so one wavefront load instruction covers 64/G atoms with
// runs of S contiguous x points each, and the cross-lane reduction spans only
// the group.  z and y sums are separable:
//   E  = sum_y M_y sum_z M_z Phi,  Fy = sum_y dM_y sum_z M_z Phi,
//   Fz = sum_y M_y sum_z dM_z Phi,
// then e = M_x E, fx = dM_x E, fy = M_x Fy, fz = M_x Fz per lane.  The z sums
// run in R, everything after them in FP64.
template <typename R>
struct GatherArgs {
    const double4 *pos;
    int n;
    SpmeParams sp;
    const R *Phi;
    double4 *frc_recip;
    double *red;
    // batched runs: the energy and net-force totals are also added into
    // acc[4 (bid % kAccSlots) + 0..3] (zero before the launch), one atomic
    // each per workgroup, so the velocity stage needs no reduction launch to
    // subtract the mean reciprocal force (null: rows only)
    double *acc;
};
template <typename R, int S>
__device__ __forceinline__ void gather_body(const GatherArgs<R> &ga, int bid)
{
    constexpr int G = gather_lanes(S), APB = 256 / G;
    __shared__ R sM[3][APB][S];
    __shared__ R sD[3][APB][S];
    __shared__ int sB[3][APB];
    __shared__ double sQ[APB];
    __shared__ double lred[4 * 4];
    const double4 *__restrict__ pos = ga.pos;
    const int n = ga.n;
    const SpmeParams &sp = ga.sp;
    const R *__restrict__ Phi = ga.Phi;
    double4 *__restrict__ frc_recip = ga.frc_recip;
    const int a0 = bid * APB;
    const int t = threadIdx.x;
    if (t < 3 * APB) {
        const int d = t / APB, a = t % APB;
        const int i = a0 + a;
        if (i < n) {
            const double4 p = pos[i];
            int idx;
            double w;
            grid_coord(sp, d, p.x, p.y, p.z, idx, w);
            R M[S], D[S];
            bspline<R, true, S>((R)w, M, D);
#pragma unroll
            for (int k = 0; k < S; k++) {
                sM[d][a][k] = M[k];
                sD[d][a][k] = D[k];
            }
            // first grid point of the stencil, in [0, K)
            int b = idx - S + 1;
            if (b < 0) b += sp.K[d];
            sB[d][a] = b;
            if (d == 0) sQ[a] = p.w;
        }
    }
    __syncthreads();
    const int a = t / G, tx = t % G, i = a0 + a;
    double acc[4] = {0, 0, 0, 0};  // energy, fx, fy, fz (unscaled, summed over atoms)
    double e = 0.0, fx = 0.0, fy = 0.0, fz = 0.0;
    const double q = i < n ? sQ[a] : 0.0;
    if (i < n && tx < S && fabs(q) > kZeroPlus) {
        int gx = sB[0][a] + tx;
        if (gx >= sp.K[0]) gx -= sp.K[0];
        const int by = sB[1][a], bz = sB[2][a];
        const size_t plane = (size_t)sp.K[0] * sp.K[1];
        // z planes of the stencil, wrapped once
        size_t zoff[S];
#pragma unroll
        for (int tz = 0; tz < S; tz++) {
            int gz = bz + tz;
            if (gz >= sp.K[2]) gz -= sp.K[2];
            zoff[tz] = (size_t)gz * plane + gx;
        }
        double E = 0.0, Fy = 0.0, Fz = 0.0;
        // y rows per iteration (a divisor of S, which is even), their RY*S
        // grid values in flight together
        constexpr int RY = S % 4 == 0 ? 4 : 2;
        for (int ty = 0; ty < S; ty += RY) {
            size_t yo[RY];
#pragma unroll
            for (int r = 0; r < RY; r++) {
                int gy = by + ty + r;
                if (gy >= sp.K[1]) gy -= sp.K[1];
                yo[r] = (size_t)gy * sp.K[0];
            }
            R ph[RY][S];
#pragma unroll
            for (int tz = 0; tz < S; tz++)
#pragma unroll
                for (int r = 0; r < RY; r++) ph[r][tz] = Phi[zoff[tz] + yo[r]];
#pragma unroll
            for (int r = 0; r < RY; r++) {
                R se = (R)0, sz = (R)0;
#pragma unroll
                for (int tz = 0; tz < S; tz++) {
                    se += sM[2][a][tz] * ph[r][tz];
                    sz += sD[2][a][tz] * ph[r][tz];
                }
                const double my = (double)sM[1][a][ty + r], dy = (double)sD[1][a][ty + r];
                E += my * (double)se;
                Fy += dy * (double)se;
                Fz += my * (double)sz;
            }
        }
        const double mx = (double)sM[0][a][tx], dx = (double)sD[0][a][tx];
        e = mx * E;
        fx = dx * E;
        fy = mx * Fy;
        fz = mx * Fz;
    }
    e = group_sum<G>(e);
    fx = group_sum<G>(fx);
    fy = group_sum<G>(fy);
    fz = group_sum<G>(fz);
    if (i < n && tx == 0) {
        // ewald_general.F90:800-855: F_i = -q sum dM.M.M.Phi * recip_kmax
        const double Fx_ = -q * fx * sp.rk[0], Fy_ = -q * fy * sp.rk[1], Fz_ = -q * fz * sp.rk[2];
        frc_recip[i] = make_double4(Fx_, Fy_, Fz_, q * e);  // w: the atom's energy (ewald_general.F90:852)
        acc[0] = q * e;
        acc[1] = Fx_;
        acc[2] = Fy_;
        acc[3] = Fz_;
    }
    const double tot = block_sum<4>(acc, lred, ga.red + (size_t)bid * kReduceSlots + R_ERECIP);
    if (ga.acc && t < 4 && tot != 0.0) atomicAdd(&ga.acc[4 * (bid % kAccSlots) + t], tot);
}
template <typename R, int S>
__global__ void __launch_bounds__(256) k_gather(GatherArgs<R> a)
{
    gather_body<R, S>(a, xcd_block(blockIdx.x, gridDim.x));
}
template <typename R, int S>
__global__ void __launch_bounds__(256) k_gather_batch(const GatherArgs<R> *__restrict__ av,
                                                      const int32_t *__restrict__ boff, int nsys)
{
    BatchPos bp;
    if (!batch_pos(boff, nsys, bp)) return;
    const GatherArgs<R> &a = av[bp.s];
    gather_body<R, S>(a, bp.b);
}

// Per-particle reciprocal stress (spme_calc_stress, ewald_general.F90:871-
// 1009) from the stress grid G (the charge grid convolved with the stress
// kernel): S_ab = -q sum (d_a d_b M_x M_y M_z) G kmax_a kmax_b / (4 pi alpha)
// with second derivatives of the splines, for ab = 11, 21, 31, 22, 32, 33.
// The lane layout of k_gather: lane tx takes grid column x; the (y, z) sums
//   A = sum My Mz G, B = sum dMy Mz G, C = sum My dMz G,
//   D = sum d2My Mz G, E = sum dMy dMz G, F = sum My d2Mz G
// give S11 ~ d2Mx A, S21 ~ dMx B, S31 ~ dMx C, S22 ~ Mx D, S32 ~ Mx E,
// S33 ~ Mx F.  Writes pp[i*kPPStride + 8..13] and the block sums of the six
// components into R_RS11..R_RS33: with per-particle collection the reference
// takes the reciprocal stress from these sums (ewald_general.F90:963,1002).
template <typename R, int S>
__global__ void __launch_bounds__(256) k_gather_stress(const double4 *__restrict__ pos, int n, SpmeParams sp,
                                                       double c_fac, const R *__restrict__ Gs,
                                                       double *__restrict__ pp, double *red)
{
    constexpr int G = gather_lanes(S), APB = 256 / G;
    __shared__ R sM[3][APB][S];
    __shared__ R sD[3][APB][S];
    __shared__ R sD2[3][APB][S];
    __shared__ int sB[3][APB];
    __shared__ double sQ[APB];
    __shared__ double lred[6 * 4];
    const int a0 = xcd_block(blockIdx.x, gridDim.x) * APB;
    const int t = threadIdx.x;
    if (t < 3 * APB) {
        const int d = t / APB, a = t % APB;
        const int i = a0 + a;
        if (i < n) {
            const double4 p = pos[i];
            int idx;
            double w;
            grid_coord(sp, d, p.x, p.y, p.z, idx, w);
            R M[S], D[S], D2[S];
            bspline<R, true, S, true>((R)w, M, D, D2);
#pragma unroll
            for (int k = 0; k < S; k++) {
                sM[d][a][k] = M[k];
                sD[d][a][k] = D[k];
                sD2[d][a][k] = D2[k];
            }
            int b = idx - S + 1;
            if (b < 0) b += sp.K[d];
            sB[d][a] = b;
            if (d == 0) sQ[a] = p.w;
        }
    }
    __syncthreads();
    const int a = t / G, tx = t % G, i = a0 + a;
    double v[6] = {0, 0, 0, 0, 0, 0};
    if (i < n && tx < S) {
        int gx = sB[0][a] + tx;
        if (gx >= sp.K[0]) gx -= sp.K[0];
        const int by = sB[1][a], bz = sB[2][a];
        const size_t plane = (size_t)sp.K[0] * sp.K[1];
        double A = 0, B = 0, C = 0, D = 0, E = 0, F = 0;
        for (int tz = 0; tz < S; tz++) {
            int gz = bz + tz;
            if (gz >= sp.K[2]) gz -= sp.K[2];
            const double mz = (double)sM[2][a][tz], dz = (double)sD[2][a][tz], d2z = (double)sD2[2][a][tz];
            double a_ = 0, b_ = 0, d_ = 0;  // sum over y of My G, dMy G, d2My G
            for (int ty = 0; ty < S; ty++) {
                int gy = by + ty;
                if (gy >= sp.K[1]) gy -= sp.K[1];
                const double g = (double)Gs[(size_t)gz * plane + (size_t)gy * sp.K[0] + gx];
                a_ += (double)sM[1][a][ty] * g;
                b_ += (double)sD[1][a][ty] * g;
                d_ += (double)sD2[1][a][ty] * g;
            }
            A += mz * a_;
            B += mz * b_;
            C += dz * a_;
            D += mz * d_;
            E += dz * b_;
            F += d2z * a_;
        }
        const double mx = (double)sM[0][a][tx], dx = (double)sD[0][a][tx], d2x = (double)sD2[0][a][tx];
        v[0] = d2x * A;
        v[1] = dx * B;
        v[2] = dx * C;
        v[3] = mx * D;
        v[4] = mx * E;
        v[5] = mx * F;
    }
#pragma unroll
    for (int k = 0; k < 6; k++) v[k] = group_sum<G>(v[k]);
    double acc[6] = {0, 0, 0, 0, 0, 0};
    if (i < n && tx == 0) {
        const double q = sQ[a];
        const int ab[6][2] = {{0, 0}, {1, 0}, {2, 0}, {1, 1}, {2, 1}, {2, 2}};
#pragma unroll
        for (int k = 0; k < 6; k++) {
            acc[k] = -(q * v[k]) * sp.rk[ab[k][0]] * sp.rk[ab[k][1]] * c_fac;
            pp[(size_t)i * kPPStride + 8 + k] = acc[k];
        }
    }
    block_sum<6>(acc, lred, red + (size_t)blockIdx.x * kReduceSlots + R_RS11);
}

int gather_blocks(const Ctx *c)
{
    return xcd_grid(ceil_div(c->natms, 256 / gather_lanes(c->prm.nsplines)));
}

// total force += 2 scale (F_recip - mean F_recip) (ewald_general.F90:857-864,
// ewald_spole.F90:430)
__global__ void k_finish(double4 *__restrict__ frc, const double4 *__restrict__ frc_recip, int n, double two_scale,
                         const double *__restrict__ red_out, double inv_n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double mx = red_out[R_FNETX] * inv_n, my = red_out[R_FNETY] * inv_n, mz = red_out[R_FNETZ] * inv_n;
    const double4 r = frc_recip[i];
    double4 f = frc[i];
    f.x += (r.x - mx) * two_scale;
    f.y += (r.y - my) * two_scale;
    f.z += (r.z - mz) * two_scale;
    frc[i] = f;
}

// Sum the partial rows of every column into red_out.
struct RedRows {
    int rows[kReduceSlots];
};
// one workgroup per column; fixed summation order (deterministic)
__device__ __forceinline__ void reduce_body(const double *__restrict__ red, const int *rows, double *out, int col,
                                            double *rec)
{
    __shared__ double part[256];
    const double v = column_sum<256>(red, rows[col], kReduceSlots, col, part);
    if (threadIdx.x == 0) {
        out[col] = v;
        if (rec) rec[col] = v;
    }
}
__global__ void __launch_bounds__(256) k_reduce(const double *__restrict__ red, RedRows rr, double *out, double *rec)
{
    reduce_body(red, rr.rows, out, blockIdx.x, rec);
}

int ensure_red_rows(Ctx *c, int rows)
{
    if (rows <= c->red_cap) return 0;
    if (c->red) (void)hipFree(c->red);
    c->red = nullptr;
    DLPX_HIP(c, hipMalloc((void **)&c->red, sizeof(double) * kReduceSlots * (size_t)rows));
    c->red_cap = rows;
    return 0;
}

int reduce_partials(Ctx *c, double *rec)
{
    RedRows rr;
    for (int k = 0; k < kReduceSlots; k++) rr.rows[k] = c->red_rows[k];
    hipLaunchKernelGGL(k_reduce, dim3(kReduceSlots), dim3(256), 0, c->stream, c->red, rr, c->red_out, rec);
    DLPX_HIP(c, hipGetLastError());
    return 0;
}

static SpmeParams spme_params(const Ctx *c)
{
    SpmeParams sp;
    for (int d = 0; d < 3; d++) {
        sp.K[d] = c->K[d];
        sp.kr[d] = (double)c->K[d];
        sp.invK[d] = 1.0f / (float)c->K[d];
    }
    sp.K1h = c->K1h;
    sp.S = c->prm.nsplines;
    for (int k = 0; k < 9; k++) sp.rcell[k] = c->rcell[k];
    for (int d = 0; d < 3; d++)
        sp.rk[d] = c->rcell[d] * sp.kr[0] + c->rcell[d + 3] * sp.kr[1] + c->rcell[d + 6] * sp.kr[2];
    return sp;
}

int spme_setup(Ctx *c)
{
    const int S = c->prm.nsplines;
    if (S < 4 || S > kMaxSplines || (S & 1))
        return fail(c, DLPX_ERR_UNSUPPORTED, "spline order must be even and in 4..16");
    for (int d = 0; d < 3; d++) {
        int k = c->prm.kvec[d];
        if (k < S) return fail(c, DLPX_ERR_BAD_ARG, "kvec must be >= the spline order");
        for (int p : {2, 3, 5})
            while (k % p == 0) k /= p;
        if (k != 1) return fail(c, DLPX_ERR_BAD_ARG, "kvec entries must be 2^a 3^b 5^c");
        c->K[d] = c->prm.kvec[d];
    }
    c->K1h = c->K[0] / 2 + 1;
    c->nreal = (size_t)c->K[0] * c->K[1] * c->K[2];
    c->K1hp = (c->K1h + 15) / 16 * 16;  // row stride of the half spectrum (128-byte aligned runs)
    c->nhalf = (size_t)c->K1hp * c->K[1] * c->K[2];
    const size_t rs = c->prm.precision == DLPX_MIXED ? sizeof(float) : sizeof(double);
    DLPX_HIP(c, hipMalloc(&c->Q, rs * c->nreal));
    DLPX_HIP(c, dev_zero(c->stream, c->Q, rs * c->nreal));  // kept zero from here on by the forward x pass
    DLPX_HIP(c, hipMalloc(&c->Phi, rs * c->nreal));
    DLPX_HIP(c, hipMalloc(&c->H, 2 * rs * c->nhalf));
    DLPX_HIP(c, hipMalloc(&c->theta, 2 * rs * c->nhalf));
    DLPX_HIP(c, dev_zero(c->stream, c->theta, 2 * rs * c->nhalf));  // the row padding stays zero
    c->theta_valid = false;
    const int ksum = c->K[0] + c->K[1] + c->K[2];
    std::vector<double> n2(ksum);
    bspline_norm2(c->K[0], S, n2.data());
    bspline_norm2(c->K[1], S, n2.data() + c->K[0]);
    bspline_norm2(c->K[2], S, n2.data() + c->K[0] + c->K[1]);
    DLPX_HIP(c, hipMalloc((void **)&c->bsp_n2, sizeof(double) * ksum));
    DLPX_HIP(c, dev_upload(c->stream, c->bsp_n2, n2.data(), sizeof(double) * ksum));
    // twiddles exp(+2 pi i m/K) per axis, in the grid precision
    std::vector<double> twd(2 * (size_t)ksum);
    size_t o = 0;
    for (int d = 0; d < 3; d++)
        for (int m = 0; m < c->K[d]; m++, o++) {
            const double a = 2.0 * kPi * (double)m / (double)c->K[d];
            twd[2 * o] = std::cos(a);
            twd[2 * o + 1] = std::sin(a);
        }
    if (c->prm.precision == DLPX_MIXED) {
        std::vector<float> twf(twd.begin(), twd.end());
        DLPX_HIP(c, hipMalloc(&c->tw, sizeof(float) * twf.size()));
        DLPX_HIP(c, dev_upload(c->stream, c->tw, twf.data(), sizeof(float) * twf.size()));
    } else {
        DLPX_HIP(c, hipMalloc(&c->tw, sizeof(double) * twd.size()));
        DLPX_HIP(c, dev_upload(c->stream, c->tw, twd.data(), sizeof(double) * twd.size()));
    }
    return 0;
}

// ewald_spole.F90:1296-1306 cutoff and convergence factors
InflParams infl_params(const Ctx *c)
{
    InflParams ip;
    for (int d = 0; d < 3; d++) ip.K[d] = c->K[d];
    ip.K1h = c->K1h;
    for (int k = 0; k < 9; k++) ip.rcell[k] = c->rcell[k];
    double rcp[10];
    dcell(c->rcell, rcp);
    ip.rcf = kPi / c->prm.alpha;
    ip.test_fac = std::pow(1.0e-6 / ip.rcf, 2);
    const double m = std::min(std::min((double)c->K[0] * rcp[6], (double)c->K[1] * rcp[7]), (double)c->K[2] * rcp[8]);
    const double cut_off = 0.5 * 1.05 * m;
    ip.cut2 = cut_off * cut_off;
    ip.alpha = c->prm.alpha;
    ip.mode = 0;
    return ip;
}

template <typename R>
static SpreadArgs<R> spread_args(const Ctx *c)
{
    return SpreadArgs<R>{c->pos, c->cell_start, c->ncell, spme_params(c), (R *)c->Q};
}
// How far along axis d an atom of a tile's list may be from its place at the
// list build, in grid points: half the padding, and 1e-4 points of which the
// upload's test leaves half to the rounding of either side.
static double tile_drift(const Ctx *c, int d)
{
    return 0.5 * c->prm.padding * c->K[d] / c->list_L[d] * (1.0 + 1.0e-6) + 1.0e-4;
}
// The largest displacement since then that passes that test, as a fraction of the cell.
double tile_reach(const Ctx *c, int d) { return (tile_drift(c, d) - 0.5e-4) / c->K[d]; }
static int tile_slack(const Ctx *c, int d) { return (int)std::ceil(tile_drift(c, d)) + 1; }
int tile_blocks(const Ctx *c)
{
    return ceil_div(c->K[0], kTileX) * ceil_div(c->K[1], kTileY) * ceil_div(c->K[2], kTileZ);
}
// After the tiles' lists: the number of atoms of each, and of those found for each among strays.
static int32_t *tile_count(const Ctx *c) { return c->tile_list + (size_t)tile_blocks(c) * c->tile_cap; }
int32_t *tile_found(const Ctx *c) { return tile_count(c) + tile_blocks(c); }
// Mesh tiles need a mesh that holds a tile and an atom's reach without
// meeting itself (an atom then has one image in reach of a tile), and bins
// not much finer than a tile (kTileBins of them in reach).
static bool tiles_fit(const Ctx *c)
{
    if (!c->prm.electrostatics || c->spread_tiles == 0) return false;
    const int T[3] = {kTileX, kTileY, kTileZ}, S = c->prm.nsplines;
    long bins = 1;
    for (int d = 0; d < 3; d++) {
        if (c->K[d] < T[d] + S - 1 + 2 * tile_slack(c, d)) return false;
        const int nb = (c->list_coded ? 2 : 1) * c->nc[d];
        bins *= std::min<long>(nb, (long)((T[d] + S - 1 + 2.0 * tile_drift(c, d)) * nb / c->K[d]) + 2);
    }
    return bins <= kTileBins;
}
// A host that asks for one evaluation of a Verlet list has no use for the
// tiles' lists, whose making costs more than they save in one: its first
// evaluation spreads by link cells, the next by tiles (4,000 atoms of three
// species on 36^3: 14 us by cells, 32 by tiles with the making of the lists).
bool spread_by_tiles(const Ctx *c) { return c->tile_cap > 0 && (c->resident || c->tile_lists || c->list_evals > 0); }
// How much denser than the mean the atoms are where they are densest, from the
// largest neighbour count of the list build: 1 for fluids and solids that fill
// the cell, more for slabs and droplets.
static double crowding(const Ctx *c)
{
    const double rc = c->prm.cutoff + c->prm.padding, mean = c->natms / (c->L[0] * c->L[1] * c->L[2]);
    const double r = (c->h_flags[F_IBIG] + 1) / (4.0 / 3.0 * kPi * rc * rc * rc * mean);
    return r <= 1.3 ? 1.0 : r;
}
// Estimated times (us) of the spreading by mesh tiles (atoms: in the densest
// tile's reach) and by link cells: a start; what the busiest workgroup takes
// (a tile for each chunk of its atoms; a cell for each of its atoms, over the
// 64-lane passes of an atom's S x S columns and again for each further slab of its
// window, and for its window's points); and the whole's throughput.  Fitted to
// 4,447 measured pairs of systems of 400 to 150,000 ions at every spline order, on
// meshes of 0.35 to 1.8 points to the A, cutoffs of 8 to 12 A, filling the cell or
// as slabs and droplets: nine of ten within 0.75 to 1.17 of the time measured by
// tiles and 0.64 to 1.27 of that by cells.  A tile's chunk is then charged 0.015 S^2
// us more (mixed 0.4 + 0.008 S^2), for its share of the lists' making (1.5 us a chunk
// at each rebuild) and of the CUs beside the pair kernel.
static double tiles_us(const Ctx *c, double atoms)
{
    const bool mixed = c->prm.precision == DLPX_MIXED;
    const double S = c->prm.nsplines, chunks = std::ceil(atoms / kTileChunk), perCU = tile_blocks(c) / 256.0;
    return mixed ? 11.0 + 1.31e-5 * S * std::sqrt(S) * c->natms + (0.43 + 0.032 * S) * perCU +
                       (1.44 + 0.0109 * S * S) * chunks
                 : 11.0 + 1.58e-5 * S * std::sqrt(S) * c->natms + (0.51 + 0.056 * S) * perCU +
                       (0.87 + 0.0208 * S * S) * chunks;
}
static double cells_us(const Ctx *c, double crowd)
{
    const bool mixed = c->prm.precision == DLPX_MIXED;
    const double S = c->prm.nsplines, passes = std::ceil(S * S / 64.0);
    double ext[3];
    for (int d = 0; d < 3; d++) ext[d] = (double)c->K[d] / c->nc[d] + S;
    const double window = ext[0] * ext[1] * ext[2];
    const double planes = std::max(1.0, std::floor(kSlabBytes / sizeof(double) / (ext[0] * ext[1])));
    const double slabs = std::ceil(ext[2] / std::min(planes, ext[2]));
    const double atoms = (double)c->natms / c->ncell * crowd, perCU = c->ncell / 256.0;
    const double points = perCU / crowd * window, each = S * passes * c->natms / 256.0;
    return mixed ? 5.75 + 0.0175 * S * passes * atoms + 0.308e-3 * window + 0.0051 * S * atoms * (slabs - 1.0) +
                       0.0085 * each + 0.464e-3 * points + passes * perCU * (0.503 + 0.75 / crowd)
                 : 6.8 + 0.0250 * S * passes * atoms + 0.410e-3 * window + 0.0109 * S * atoms * (slabs - 1.0) +
                       0.0083 * each + 0.571e-3 * points + passes * perCU * (0.55 + 1.63 / crowd);
}
// After a list build: whether the charges are spread by tiles, and room for
// the tiles' lists: 1.3 times the mean where the atoms are densest (a list that
// outgrows its room is made anew at every evaluation: 7,200 ions in an eighth of
// their cell, 72 x 60 x 72, S = 8 FP64, 70 us instead of 46), in steps of sqrt(2)
// so that the configurations of one system get the same room and captured
// graphs, and one round of their making.
// Where the mesh allows, by tiles unless cells are a fifth faster by these
// estimates (beside the other systems of a batch, which fill the GPU, tiles are the
// better choice a little longer): over the resident steps of 667 more such systems
// with either, 0.26 % of the time is lost to the faster choice (1.9 % without the
// order, the precision and the crowding in it), and 12 steps instead of 77 are more
// than 3 % (9 % at most, 40 %) slower by tiles than by cells.  Few atoms to a tile (fine
// meshes) are the tiles': 64,000 ions on 128^3 at order 4, 8 and 16, mixed, 33, 52
// and 474 us by cells and 22, 34 and 81 by tiles.  Many, or a part of the cell
// crowded, are the cells': the same on 64^3 20, 35 and 292 and 35, 75 and 226; 8,000
// ions on 36^3 at order 8 in FP64 32 and 56; the 7,200 ions above 31 and 46.
// The room, and that of the splines, is taken when the tiles first need it (332 MB
// at 1,728,000 ions in FP64 at order 8); without memory for it the cells are there.
void tile_room(Ctx *c)
{
    auto room = [](auto **p, size_t bytes) {
        if (!*p && hipMalloc((void **)p, bytes) != hipSuccess) {
            *p = nullptr;
            (void)hipGetLastError();
        }
        return *p != nullptr;
    };
    c->tile_cap = 0;
    c->tile_lists = false;
    c->list_evals = 0;
    if (!tiles_fit(c)) return;
    const int T[3] = {kTileX, kTileY, kTileZ};
    double mean = c->natms;
    for (int d = 0; d < 3; d++)
        mean *= std::min(1.0, (T[d] + c->prm.nsplines - 1 + 2.0 * tile_drift(c, d)) / c->K[d]);
    const double crowd = crowding(c), most = std::min<double>(c->natms, mean * crowd);
    if (c->spread_tiles < 0 && tiles_us(c, most) > 1.2 * cells_us(c, crowd)) return;
    const double steps = crowd > 1.0 ? std::exp2(0.5 * std::ceil(2.0 * std::log2(crowd))) : 1.0;
    const int cap = kTileScan * kTileThreads + (int)(1.3 * std::min<double>(c->natms, mean * steps) / 64.0 + 1.0) * 64;
    const size_t words = (size_t)tile_blocks(c) * (cap + 2);
    if (words > c->tile_words) {
        if (c->tile_list) (void)hipFree(c->tile_list);
        c->tile_list = nullptr;
        c->tile_words = 0;
        if (!room(&c->tile_list, sizeof(int32_t) * words)) return;
        c->tile_words = words;
    }
    const size_t rs = c->prm.precision == DLPX_MIXED ? sizeof(float) : sizeof(double), n = c->cap;
    if (room(&c->spl_z, rs * 3 * c->prm.nsplines * n) && room(&c->spl_wq, rs * 4 * n) &&
        room(&c->spl_base, sizeof(ushort4) * n))
        c->tile_cap = cap;
}
template <typename R>
static SplineArgs<R> spline_args(const Ctx *c, int32_t no)
{
    SplineArgs<R> a{c->pos, c->natms, spme_params(c), (R *)c->spl_z, (R *)c->spl_wq, c->spl_base};
    a.flags = c->flags;
    a.no = c->natms > kStrayTest ? no : 0;
    a.list = c->tile_list;
    a.found = tile_found(c);
    a.cap = c->tile_cap;
    const int T[3] = {kTileX, kTileY, kTileZ};
    for (int d = 0; d < 3; d++) a.tiles[d] = ceil_div(c->K[d], T[d]);
    return a;
}
static int spline_blocks(const Ctx *c) { return ceil_div(3L * c->natms, 256); }
template <typename R>
static TileArgs<R> tile_args(const Ctx *c, int32_t no, const int32_t *upd)
{
    const int T[3] = {kTileX, kTileY, kTileZ};
    TileArgs<R> a{};
    a.z = (const R *)c->spl_z;
    a.wq = (const R *)c->spl_wq;
    a.base = c->spl_base;
    a.n = c->natms;
    a.g.sub = c->list_coded ? 2 : 1;
    a.start = c->list_coded ? c->key_start : c->cell_start;
    a.list = c->tile_list;
    a.cap = c->tile_cap;
    a.count = tile_count(c);
    a.found = c->natms > kStrayTest ? tile_found(c) : nullptr;
    a.xref = c->xref;
    a.upd = upd;
    a.fresh = c->tile_lists ? 0 : 1;
    a.flags = c->flags;
    a.no = no;
    for (int d = 0; d < 3; d++) {
        a.g.nc[d] = c->nc[d];
        a.bins[d] = a.g.sub * c->nc[d];
        a.tiles[d] = ceil_div(c->K[d], T[d]);
        a.invL0[d] = 1.0 / c->list_L[d];
        a.drift_k[d] = tile_drift(c, d);
        a.slack[d] = tile_slack(c, d);
    }
    a.sp = spme_params(c);
    a.Q = (R *)c->Q;
    return a;
}
template <typename R>
static GatherArgs<R> gather_args(const Ctx *c)
{
    return GatherArgs<R>{c->pos, c->natms, spme_params(c), (const R *)c->Phi, c->frc_recip, c->red, nullptr};
}

#define DLPX_S_SWITCH(S, CALL)                                                                             \
    switch (S) {                                                                                           \
        case 4: CALL(4); break;                                                                            \
        case 6: CALL(6); break;                                                                            \
        case 8: CALL(8); break;                                                                            \
        case 10: CALL(10); break;                                                                          \
        case 12: CALL(12); break;                                                                          \
        case 14: CALL(14); break;                                                                          \
        case 16: CALL(16); break;                                                                          \
        default: return fail(c, DLPX_ERR_UNSUPPORTED, "spline order must be even and in 4..16");           \
    }

template <typename R>
__global__ void __launch_bounds__(256) k_zero(R *p, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = (R)0;
}
// The charge grid zero for a spreading by link cells, after one by tiles.
template <typename R>
static int grid_zero(Ctx *c, hipStream_t s)
{
    if (!c->grid_used) return 0;
    hipLaunchKernelGGL((k_zero<R>), dim3(std::min<size_t>((c->nreal + 255) / 256, 2048)), dim3(256), 0, s, (R *)c->Q,
                       c->nreal);
    DLPX_HIP(c, hipGetLastError());
    c->grid_used = false;
    return 0;
}

template <typename R>
static int spme_run(Ctx *c)
{
    const int n = c->natms;
    hipStream_t s = c->sp;  // the evaluation's reciprocal-space stream
    const SpmeParams sp = spme_params(c);
    const int nb = gather_blocks(c);  // evaluate() has sized the partial-sum rows
    int r;
    // ewald_general.F90:517-576 charge spreading into the charge grid
    const bool tiles = spread_by_tiles(c);
    c->list_evals++;
    if (tiles) {
        const SplineArgs<R> sa = spline_args<R>(c, c->stray_no);
#define DLPX_SPLINES(SS) hipLaunchKernelGGL((k_splines<R, SS>), dim3(spline_blocks(c)), dim3(256), 0, s, sa)
        DLPX_S_SWITCH(sp.S, DLPX_SPLINES)
#undef DLPX_SPLINES
        const TileArgs<R> ta = tile_args<R>(c, c->stray_no, nullptr);
#define DLPX_TILES(SS) \
    hipLaunchKernelGGL((k_spread_tiles<R, SS>), dim3(xcd_grid(tile_blocks(c))), dim3(kTileThreads), 0, s, ta)
        DLPX_S_SWITCH(sp.S, DLPX_TILES)
#undef DLPX_TILES
        c->grid_used = true;
        c->tile_lists = true;
    } else {
        // onto a grid that is zero here: set at allocation, and cleared by
        // the forward x pass of each convolution after reading it
        if ((r = grid_zero<R>(c, s))) return r;
        const SpreadArgs<R> spa = spread_args<R>(c);
#define DLPX_SPREAD(SS) \
    hipLaunchKernelGGL((k_spread_cells<R, SS>), dim3(xcd_grid(c->ncell)), dim3(spread_threads<R>()), 0, s, spa)
        DLPX_S_SWITCH(sp.S, DLPX_SPREAD)
#undef DLPX_SPREAD
    }
    if (c->timing) DLPX_HIP(c, hipEventRecord(c->ev[2], s));
    InflParams ip = infl_params(c);
    if (c->pp_now) {
        // keep the charge grid for the per-particle stress convolution
        const size_t bytes = (c->prm.precision == DLPX_MIXED ? sizeof(float) : sizeof(double)) * c->nreal;
        DLPX_HIP(c, hipMemcpyAsync(c->Q2, c->Q, bytes, hipMemcpyDeviceToDevice, s));
    }
    if ((r = fft_convolve(c, ip, c->Q, c->Phi, !tiles))) return r;
    if (c->timing) DLPX_HIP(c, hipEventRecord(c->ev[3], s));
    const GatherArgs<R> ga = gather_args<R>(c);
#define DLPX_GATHER(SS) hipLaunchKernelGGL((k_gather<R, SS>), dim3(nb), dim3(256), 0, s, ga)
    DLPX_S_SWITCH(sp.S, DLPX_GATHER)
#undef DLPX_GATHER
    for (int k = R_ERECIP; k <= R_FNETZ; k++) c->red_rows[k] = nb;
    if (c->pp_now) {
        // per-particle stresses: the saved charge grid convolved with the
        // stress kernel, then gathered with second spline derivatives
        InflParams ips = ip;
        ips.mode = 1;
        if ((r = fft_convolve(c, ips, c->Q2, c->Q2, false))) return r;
        const double c_fac = 1.0 / (2.0 * 2.0 * kPi * c->prm.alpha);  // ewald_general.F90:932-933
#define DLPX_GSTRESS(SS)                                                                                        \
    hipLaunchKernelGGL((k_gather_stress<R, SS>), dim3(nb), dim3(256), 0, s, c->pos, n, sp, c_fac,              \
                       (const R *)c->Q2, c->pp, c->red)
        DLPX_S_SWITCH(sp.S, DLPX_GSTRESS)
#undef DLPX_GSTRESS
        for (int k = R_RS11; k <= R_RS33; k++) c->red_rows[k] = nb;
    }
    if (c->timing) DLPX_HIP(c, hipEventRecord(c->ev[4], s));
    DLPX_HIP(c, hipGetLastError());
    return 0;
}

int gather_blocks_exact(const Ctx *c) { return ceil_div(c->natms, 256 / gather_lanes(c->prm.nsplines)); }

// Batched reciprocal space over the systems with electrostatics: spreading,
// the convolution passes and the gather, one launch each.  Every system of
// the batch must have the same spline order.
template <typename R>
static int spme_prepare_t(const std::vector<Ctx *> &cs, SpmeBatch &sb)
{
    std::vector<SpreadArgs<R>> spa;
    std::vector<SplineArgs<R>> sa;
    std::vector<TileArgs<R>> ta;
    std::vector<GatherArgs<R>> ga;
    std::vector<InflParams> ips;
    std::vector<int> nbp, nbs, nbt, nbg;
    int r, S = 0;
    for (Ctx *c : cs) {
        const bool on = c->prm.electrostatics != 0;
        if (on) {
            if (S && c->prm.nsplines != S)
                return fail(c, DLPX_ERR_UNSUPPORTED, "systems of one batch must share the spline order");
            S = c->prm.nsplines;
        }
        const bool tiles = on && spread_by_tiles(c);
        if (tiles) c->grid_used = true;
        else if (on) {
            if ((r = grid_zero<R>(c, c->stream))) return r;
            DLPX_HIP(c, hipStreamSynchronize(c->stream));
        }
        sa.push_back(tiles ? spline_args<R>(c, 0) : SplineArgs<R>{});
        nbp.push_back(tiles ? spline_blocks(c) : 0);
        spa.push_back(on && !tiles ? spread_args<R>(c) : SpreadArgs<R>{});
        ta.push_back(tiles ? tile_args<R>(c, 0, c->flags + F_UPD) : TileArgs<R>{});
        ga.push_back(on ? gather_args<R>(c) : GatherArgs<R>{});
        ga.back().acc = on ? c->acc : nullptr;
        ips.push_back(on ? infl_params(c) : InflParams{});
        nbs.push_back(on && !tiles ? c->ncell : 0);
        nbt.push_back(tiles ? tile_blocks(c) : 0);
        nbg.push_back(on ? gather_blocks_exact(c) : 0);
    }
    sb.S = S;
    if ((r = batch_upload(cs[0], sb.spread, spa.data(), sizeof(SpreadArgs<R>), nbs, true)) ||
        (r = batch_upload(cs[0], sb.splines, sa.data(), sizeof(SplineArgs<R>), nbp, false)) ||
        (r = batch_upload(cs[0], sb.tiles, ta.data(), sizeof(TileArgs<R>), nbt, true)) ||
        (r = batch_upload(cs[0], sb.gather, ga.data(), sizeof(GatherArgs<R>), nbg, true)))
        return r;
    sb.gather_rows = nbg;
    return fft_prepare(cs, ips, sb.fft);
}

int spme_prepare(const std::vector<Ctx *> &cs, SpmeBatch &sb)
{
    if (cs[0]->prm.precision == DLPX_MIXED) return spme_prepare_t<float>(cs, sb);
    return spme_prepare_t<double>(cs, sb);
}

template <typename R>
static int spme_launch_t(Ctx *c, hipStream_t s, const SpmeBatch &sb, hipEvent_t *marks)
{
    if (sb.S == 0) return 0;
    const BatchLaunch &bp = sb.splines, &bs = sb.spread, &bt = sb.tiles, &bg = sb.gather;
#define DLPX_SPLINESB(SS)                                                                                        \
    hipLaunchKernelGGL((k_splines_batch<R, SS>), dim3(bp.total), dim3(256), 0, s, (const SplineArgs<R> *)bp.args, \
                       bp.boff, bp.nsys)
    if (bp.total > 0) {
        DLPX_S_SWITCH(sb.S, DLPX_SPLINESB)
    }
#undef DLPX_SPLINESB
#define DLPX_TILESB(SS)                                                                                          \
    hipLaunchKernelGGL((k_spread_tiles_batch<R, SS>), dim3(bt.total), dim3(kTileThreads), 0, s,                  \
                       (const TileArgs<R> *)bt.args, bt.boff, bt.nsys)
    if (bt.total > 0) {
        DLPX_S_SWITCH(sb.S, DLPX_TILESB)
    }
#undef DLPX_TILESB
#define DLPX_SPREADB(SS)                                                                                         \
    hipLaunchKernelGGL((k_spread_cells_batch<R, SS>), dim3(bs.total), dim3(spread_threads<R>()), 0, s,          \
                       (const SpreadArgs<R> *)bs.args, bs.boff, bs.nsys)
    if (bs.total > 0) {
        DLPX_S_SWITCH(sb.S, DLPX_SPREADB)
    }
#undef DLPX_SPREADB
    if (marks && marks[0]) DLPX_HIP(c, hipEventRecord(marks[0], s));
    int r;
    if ((r = fft_launch(c, s, sb.fft))) return r;
    if (marks && marks[1]) DLPX_HIP(c, hipEventRecord(marks[1], s));
#define DLPX_GATHERB(SS)                                                                                         \
    hipLaunchKernelGGL((k_gather_batch<R, SS>), dim3(bg.total), dim3(256), 0, s, (const GatherArgs<R> *)bg.args, \
                       bg.boff, bg.nsys)
    DLPX_S_SWITCH(sb.S, DLPX_GATHERB)
#undef DLPX_GATHERB
    if (marks && marks[2]) DLPX_HIP(c, hipEventRecord(marks[2], s));
    DLPX_HIP(c, hipGetLastError());
    return 0;
}

int spme_launch(Ctx *c, hipStream_t s, const SpmeBatch &sb, hipEvent_t *marks)
{
    if (c->prm.precision == DLPX_MIXED) return spme_launch_t<float>(c, s, sb, marks);
    return spme_launch_t<double>(c, s, sb, marks);
}

int spme_forces(Ctx *c)
{
    if (c->prm.precision == DLPX_MIXED) return spme_run<float>(c);
    return spme_run<double>(c);
}

int spme_finish(Ctx *c, double two_scale)
{
    hipLaunchKernelGGL(k_finish, dim3(ceil_div(c->natms, 256)), dim3(256), 0, c->stream, c->frc, c->frc_recip,
                       c->natms, two_scale, c->red_out, 1.0 / (double)c->natms);
    DLPX_HIP(c, hipGetLastError());
    return 0;
}

}  // namespace dlpx
