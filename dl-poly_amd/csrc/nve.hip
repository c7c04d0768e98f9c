// Velocity-Verlet NVE integration on the device (nve.F90:127-215) and the
// host-order <-> cell-order transfers of per-atom data.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "common.h"
#include "device_util.h"

namespace dlpx {

// Stage 1: v += dt/2 F/m ; x += dt v  (atoms of mass <= 1e-6 stay frozen),
// fused with the displacement test of vnl_check (neighbours.F90:150-178):
// the largest minimum-image |x - x_ref|^2 goes to *dmax (as the bit pattern
// of a non-negative double).  The last workgroup to finish copies it to host
// memory (host_dmax: the host decides the rebuild) and resets *dmax and
// *done for the next step.  Host-decided runs only; a batched run decides on
// the device (k_step_batch).
struct Box {
    double L[3], invL[3];
};
struct Vv1Args {
    double4 *pos, *vel;
    const double4 *frc, *xref;
    int n;
    double dt;
    Box b;
    unsigned long long *dmax;
    unsigned int *done;
    unsigned long long *host_dmax;
};
// 1024-thread workgroups: the maximum is reduced in LDS first, so only one
// atomic per workgroup (63 at 64k atoms) meets the single device word.
constexpr int kVv1Threads = 1024;
__device__ __forceinline__ void vv1_body(const Vv1Args &a, int bid, int nb)
{
    __shared__ double wmax[kVv1Threads / 64];
    __shared__ bool last;
    const int i = bid * blockDim.x + threadIdx.x;
    double r2 = 0.0;
    if (i < a.n) {
        double4 v = a.vel[i];
        double4 p = a.pos[i];
        if (v.w > 1.0e-6) {
            const double4 f = a.frc[i];
            const double tmp = (0.5 * a.dt) / v.w;
            v.x += tmp * f.x;
            v.y += tmp * f.y;
            v.z += tmp * f.z;
            p.x += a.dt * v.x;
            p.y += a.dt * v.y;
            p.z += a.dt * v.z;
            a.vel[i] = v;
            a.pos[i] = p;
        }
        const double4 q = a.xref[i];
        const double dx = min_image_1(p.x, q.x, a.b.L[0], a.b.invL[0]);
        const double dy = min_image_1(p.y, q.y, a.b.L[1], a.b.invL[1]);
        const double dz = min_image_1(p.z, q.z, a.b.L[2], a.b.invL[2]);
        r2 = dx * dx + dy * dy + dz * dz;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) r2 = fmax(r2, __shfl_xor(r2, o, 64));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = r2;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) m = fmax(m, wmax[w]);
        atomicMax(a.dmax, (unsigned long long)__double_as_longlong(m));
        __threadfence();
        last = atomicAdd(a.done, 1u) == (unsigned)nb - 1;
    }
    __syncthreads();
    if (last && threadIdx.x == 0) {
        __threadfence();
        *a.host_dmax = atomicAdd(a.dmax, 0ull);
        __threadfence_system();
        *a.dmax = 0ull;
        *a.done = 0u;
    }
}
__global__ void __launch_bounds__(kVv1Threads) k_vv1(Vv1Args a) { vv1_body(a, blockIdx.x, gridDim.x); }
// Stage 2: v += dt/2 F/m, and sum m v^2 per block.  With fin the
// reciprocal forces are first added to the total force as k_finish does:
// frc += 2 scale (frc_recip - mean frc_recip) (ewald_general.F90:857-864).
// Frozen atoms (frz[gid[i]] /= 0; frz may be null) get zero force and
// velocity, as freeze_atoms does after each force evaluation
// (configuration.F90:3240-3258), so they neither move nor add kinetic energy.
struct Vv2Args {
    double4 *vel, *frc;
    int n;
    double dt;
    double *red;
    const double4 *frc_recip;  // fin only
    double two_scale;
    const double *red_out;
    double inv_n;
    const int32_t *gid, *frz;
    int fin;
};
__device__ __forceinline__ void vv2_body(const Vv2Args &a, int bid)
{
    __shared__ double lred[4];
    const int i = bid * blockDim.x + threadIdx.x;
    double acc[1] = {0.0};
    if (i < a.n) {
        double4 v = a.vel[i];
        double4 f = a.frc[i];
        if (a.fin) {
            const double mx = a.red_out[R_FNETX] * a.inv_n, my = a.red_out[R_FNETY] * a.inv_n,
                         mz = a.red_out[R_FNETZ] * a.inv_n;
            const double4 r = a.frc_recip[i];
            f.x += (r.x - mx) * a.two_scale;
            f.y += (r.y - my) * a.two_scale;
            f.z += (r.z - mz) * a.two_scale;
            a.frc[i] = f;
        }
        if (a.frz && a.frz[a.gid[i]] != 0) {
            f.x = f.y = f.z = 0.0;
            v.x = v.y = v.z = 0.0;
            a.frc[i] = f;
            a.vel[i] = v;
        }
        if (v.w > 1.0e-6) {
            const double tmp = (0.5 * a.dt) / v.w;
            v.x += tmp * f.x;
            v.y += tmp * f.y;
            v.z += tmp * f.z;
            a.vel[i] = v;
            acc[0] = v.w * (v.x * v.x + v.y * v.y + v.z * v.z);
        }
    }
    block_sum<1>(acc, lred, a.red + (size_t)bid * kReduceSlots + R_KIN);
}
__global__ void __launch_bounds__(256) k_vv2(Vv2Args a) { vv2_body(a, blockIdx.x); }
// freeze_atoms (configuration.F90:3240-3258): zero force and velocity of
// frozen atoms (frz[gid[i]] /= 0)
__global__ void k_freeze(double4 *vel, double4 *frc, int n, const int32_t *__restrict__ gid,
                         const int32_t *__restrict__ frz)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || frz[gid[i]] == 0) return;
    double4 v = vel[i], f = frc[i];
    v.x = v.y = v.z = 0.0;
    f.x = f.y = f.z = 0.0;
    vel[i] = v;
    frc[i] = f;
}

int freeze_atoms(Ctx *c)
{
    if (c->nfrozen == 0) return 0;
    hipLaunchKernelGGL(k_freeze, dim3(ceil_div(c->natms, 256)), dim3(256), 0, c->stream, c->vel, c->frc, c->natms,
                       c->gid, c->frz);
    DLPX_HIP(c, hipGetLastError());
    return 0;
}

// The test of an upload onto an existing list: whether each atom is still as
// near its place at the list build as the tiles' lists of the spreading allow
// for (tile_drift, spme.hip), per axis in fractions of the cell, so that a
// change of the cell counts too.
struct StrayArgs {
    const double4 *xref;
    double invL0[3], invL[3]; // the cell of the list build; the present one
    double reach[3];
    int32_t *flag;            // null: no list to hold them to
    int32_t no;
};
__device__ __forceinline__ bool strayed(const StrayArgs &a, const double (&x)[3], const double (&x0)[3])
{
    bool out = false;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        double f = x[d] * a.invL[d] - x0[d] * a.invL0[d];
        f -= rint(f);
        out = out || !(fabs(f) <= a.reach[d]);  // a coordinate that is no number strays
    }
    return out;
}

// Host order -> cell order, from pinned host memory (4 doubles per atom, x y z
// q, or 8 with vx vy vz m; and its type from 1).  disp, when not null, gets
// the largest minimum-image displacement squared since the list build of each
// workgroup's atoms, as the bit pattern of a non-negative double (vnl_check,
// neighbours.F90:150-178).
//
// Bound by the host link (36 B an atom without velocities), and in a small
// system by the number of operations: the kernel reads the host's rows and
// writes the displacements to the host itself, one launch where copies to
// staging, a load, a clear, a displacement kernel and a copy back were six.
// 64,000 atoms 54 us (43 GB/s of the link); a list check of 256 atoms, with the
// wait, 58 -> 30 us.
struct LoadArgs {
    const double *st;
    const int32_t *st_t;
    int n, row;
    const int32_t *slot;  // null: the order as given
    double4 *pos, *vel;
    int32_t *typ, *gid;
    unsigned long long *disp;
    Box b;
    StrayArgs stray;
    int32_t *clear;  // words zeroed for the spreading (k_splines); null: none
    int nclear;
};
constexpr int kLoadThreads = 256;
__global__ void __launch_bounds__(kLoadThreads) k_load(LoadArgs a)
{
    __shared__ double wmax[kLoadThreads / 64];
    const int h = blockIdx.x * kLoadThreads + threadIdx.x;
    double r2 = 0.0;
    for (int k = h; k < a.nclear; k += gridDim.x * kLoadThreads) a.clear[k] = 0;
    if (h < a.n) {
        const int s = a.slot ? a.slot[h] : h;
        const double4 *r = (const double4 *)(a.st + (size_t)a.row * h);
        const double4 p = r[0];
        a.typ[s] = a.st_t[h] - 1;
        a.pos[s] = p;
        if (!a.slot) a.gid[s] = h;
        if (a.row == 8) a.vel[s] = r[1];
        if (a.slot) {
            const double4 q = a.stray.xref[s];
            const double x[3] = {p.x, p.y, p.z}, x0[3] = {q.x, q.y, q.z};
            if (a.stray.flag && strayed(a.stray, x, x0)) *a.stray.flag = a.stray.no;
            const double dx = min_image_1(p.x, q.x, a.b.L[0], a.b.invL[0]);
            const double dy = min_image_1(p.y, q.y, a.b.L[1], a.b.invL[1]);
            const double dz = min_image_1(p.z, q.z, a.b.L[2], a.b.invL[2]);
            r2 = dx * dx + dy * dy + dz * dz;
        }
    }
    if (!a.disp) return;  // uniform
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) r2 = fmax(r2, __shfl_xor(r2, o, 64));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = r2;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long m = 0;
        for (int w = 0; w < kLoadThreads / 64; w++)
            m = max(m, (unsigned long long)__double_as_longlong(wmax[w]));
        a.disp[blockIdx.x] = m;
    }
}

// Cell order -> host order, into pinned host memory: W = 3, the forces; W =
// 9, x y z | vx vy vz | fx fy fz.  frc_recip, when not null, is added first
// (total force += 2 scale (F_recip - mean F_recip), ewald_general.F90:857-864,
// ewald_spole.F90:430), here and in frc.  Bound by the host link (8 W bytes an
// atom): threads take the atoms in host order, gathering from the card's own
// memory, and a workgroup's rows go out through LDS as whole lines.
// Forces of 64,000 atoms 32 us (48 GB/s), 1,728,000 atoms with W = 9 2.4 ms
// (52 GB/s).
struct StoreArgs {
    double *out;
    int n;
    const int32_t *slot;
    const double4 *pos, *vel;
    double4 *frc;
    const double4 *frc_recip;
    const double *red_out;
    double two_scale, inv_n;
};
constexpr int kStoreThreads = 256;
template <int W>
__global__ void __launch_bounds__(kStoreThreads) k_store(StoreArgs a)
{
    __shared__ double row[kStoreThreads * W];
    const int t = threadIdx.x, h = blockIdx.x * kStoreThreads + t;
    if (h < a.n) {
        const int s = a.slot[h];
        double4 f = a.frc[s];
        if (a.frc_recip) {
            const double4 r = a.frc_recip[s];
            f.x += (r.x - a.red_out[R_FNETX] * a.inv_n) * a.two_scale;
            f.y += (r.y - a.red_out[R_FNETY] * a.inv_n) * a.two_scale;
            f.z += (r.z - a.red_out[R_FNETZ] * a.inv_n) * a.two_scale;
            a.frc[s] = f;
        }
        double *o = row + W * t;
        if (W == 9) {
            const double4 p = a.pos[s], v = a.vel[s];
            o[0] = p.x; o[1] = p.y; o[2] = p.z;
            o[3] = v.x; o[4] = v.y; o[5] = v.z;
        }
        o[W - 3] = f.x; o[W - 2] = f.y; o[W - 1] = f.z;
    }
    __syncthreads();
    const size_t base = (size_t)blockIdx.x * kStoreThreads * W, end = (size_t)a.n * W;
#pragma unroll
    for (int k = 0; k < W; k++)
        if (base + k * kStoreThreads + t < end) a.out[base + k * kStoreThreads + t] = row[k * kStoreThreads + t];
}

// Per-particle output to the host: of each atom, in host order, the energy
// without the shared parts and the six stress elements, real-space part plus
// scale times the reciprocal one (frc_recip null: none).  As k_store, in place
// of copies of the raw rows (16 doubles an atom) and a loop over them on the
// host: a heat-flux evaluation of 4,000 atoms 284 -> 234 us, with 32 lanes to
// an atom in its pair kernel.
__global__ void __launch_bounds__(kStoreThreads) k_store_pp(double *__restrict__ out, int n,
                                                            const int32_t *__restrict__ slot,
                                                            const double *__restrict__ pp,
                                                            const double4 *__restrict__ frc_recip, double scale)
{
    constexpr int W = 7;
    __shared__ double row[kStoreThreads * W];
    const int t = threadIdx.x, h = blockIdx.x * kStoreThreads + t;
    if (h < n) {
        const int s = slot[h];
        const double *p = pp + (size_t)s * kPPStride;
        double *o = row + W * t;
        o[0] = p[0] + (frc_recip ? frc_recip[s].w * scale : 0.0);
#pragma unroll
        for (int k = 0; k < 6; k++) o[1 + k] = p[1 + k] + (frc_recip ? p[8 + k] * scale : 0.0);
    }
    __syncthreads();
    const size_t base = (size_t)blockIdx.x * kStoreThreads * W, end = (size_t)n * W;
#pragma unroll
    for (int k = 0; k < W; k++)
        if (base + k * kStoreThreads + t < end) out[base + k * kStoreThreads + t] = row[k * kStoreThreads + t];
}

static Vv1Args vv1_args(Ctx *c, double dt)
{
    Vv1Args a;
    a.pos = c->pos;
    a.vel = c->vel;
    a.frc = c->frc;
    a.xref = c->xref;
    a.n = c->natms;
    a.dt = dt;
    for (int d = 0; d < 3; d++) {
        a.b.L[d] = c->L[d];
        a.b.invL[d] = c->invL[d];
    }
    // device words F_DMAX (maximum) and F_DONE (workgroup count) are zero
    // between launches
    a.dmax = (unsigned long long *)(c->flags + F_DMAX);
    a.done = (unsigned int *)(c->flags + F_DONE);
    a.host_dmax = (unsigned long long *)(c->h_flags_dev + 8);
    return a;
}
int vv1_blocks(const Ctx *c) { return ceil_div(c->natms, kVv1Threads); }

int nve_first(Ctx *c, double dt)
{
    // the result lands in host word h_flags[8..9]
    hipLaunchKernelGGL(k_vv1, dim3(vv1_blocks(c)), dim3(kVv1Threads), 0, c->stream, vv1_args(c, dt));
    DLPX_HIP(c, hipGetLastError());
    return 0;
}

double nve_first_displacement(Ctx *c)
{
    double r2;
    memcpy(&r2, c->h_flags + 8, sizeof(r2));
    return std::sqrt(r2);
}

static Vv2Args vv2_args(Ctx *c, double dt, bool fin)
{
    Vv2Args a;
    a.vel = c->vel;
    a.frc = c->frc;
    a.n = c->natms;
    a.dt = dt;
    a.red = c->red;
    a.fin = fin ? 1 : 0;
    a.frc_recip = fin ? c->frc_recip : nullptr;
    a.two_scale = fin ? 2.0 * recip_scale(c) : 0.0;
    a.red_out = fin ? c->red_out : nullptr;
    a.inv_n = 1.0 / (double)c->natms;
    a.gid = c->gid;
    a.frz = c->nfrozen > 0 ? c->frz : nullptr;
    return a;
}
int vv2_blocks(const Ctx *c) { return ceil_div(c->natms, 256); }

int nve_second(Ctx *c, double dt, bool /*kinetic*/)
{
    const int nb = vv2_blocks(c);
    int r;
    if ((r = ensure_red_rows(c, nb))) return r;
    hipLaunchKernelGGL(k_vv2, dim3(nb), dim3(256), 0, c->stream, vv2_args(c, dt, c->finish_in_vv2));
    c->finish_in_vv2 = false;
    c->red_rows[R_KIN] = nb;
    DLPX_HIP(c, hipGetLastError());
    return 0;
}

// One launch per step of a resident batched run (every system of the batch):
// S2, stage 2 of the step just evaluated: the reciprocal finish (frc +=
// 2 scale (frc_recip - mean), the mean from the gather's atomic totals in
// acc), frozen atoms, the second half-kick and m v^2; when records are kept,
// the step's partial sums reduced into its record (one wavefront per column);
// and
// S1, stage 1 of the next step: half-kick, drift, and the displacement test,
// whose largest value the last workgroup to finish turns into the rebuild
// decision (as k_vv1).  With both stages the total force is not stored: the
// next pair kernel overwrites it, and a run's last step has no stage 1.
//
// Bound by HBM at many atoms (224 B each), by latency at few.  Atomics on one
// word complete about every 25 ns whatever the load, so a workgroup issues
// exactly one (the count of finished workgroups): its kinetic-energy and
// displacement partials go to its own slot of part[], and a launch has at
// most kStepBlocks workgroups per system, each striding over the atoms with
// the next atom's loads in flight.  Against three atomics from each of
// ceil(n / 256) workgroups, the column sums ahead of the atoms and the force
// stored every step: 1,728,000 ions 596 -> 150 us (2.6 TB/s), 64,000 ions
// 14.2 -> 12.4 us, 4,000 atoms 8.5 -> 6.0 us.
struct StepArgs {
    double4 *pos, *vel, *frc;
    const double4 *frc_recip;  // null: no reciprocal part
    const double4 *xref;
    const int32_t *gid, *frz;  // frz may be null
    int n;
    double dt, two_scale, inv_n, half_pad;
    Box b;
    const double *red;
    double *part;              // kStepBlocks x {m v^2, largest displacement squared}
    double *acc;               // the gather's kAccSlots x 4 totals (null: no reciprocal part)
    int rows[kReduceSlots];    // partial rows per column of the step
    double *energies;          // per-step records (kReduceSlots each) or null
    int ecap;
    int32_t *flags;
};
__device__ __forceinline__ bool atomic_column(int col) { return col == R_KIN || (col >= R_ERECIP && col <= R_FNETZ); }
// 256 threads: workgroups small enough to spread a 64k-atom system over
// every CU
constexpr int kStepThreads = 256;
// workgroups beside the atoms' that sum the record's columns, one column per
// wavefront (23 columns of partial rows)
constexpr int kStepColumnBlocks = 6;
template <bool S2, bool S1>
__device__ __forceinline__ void step_body(const StepArgs &a, int bid, int nb)
{
    constexpr int NW = kStepThreads / 64;
    __shared__ double wke[NW], wr2[NW];
    __shared__ bool last;
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    static_assert(kAccSlots == 64, "a wavefront reads one accumulator slot per lane");
    // this thread's first atom is loaded before anything waits; each later one
    // while its predecessor is computed
    struct Atom {
        double4 v, f, r, p, q;
    } cur, nxt;
    auto load = [&](int i, Atom &m) {
        m.v = a.vel[i];
        m.f = a.frc[i];
        if (S2 && a.frc_recip) m.r = a.frc_recip[i];
        if (S1) {
            m.p = a.pos[i];
            m.q = a.xref[i];
        }
    };
    const int ncb = S2 && a.energies ? kStepColumnBlocks : 0;  // the last workgroups take the columns
    const int stride = (nb - ncb) * kStepThreads;
    int i = bid < nb - ncb ? bid * kStepThreads + t : a.n;
    if (i < a.n) load(i, cur);
    // reciprocal energy and net force (unscaled): the gather's slot totals,
    // summed in a fixed order by every wavefront
    double recip[4] = {0.0, 0.0, 0.0, 0.0};
    if (S2 && a.acc) {
#pragma unroll
        for (int k = 0; k < 4; k++) recip[k] = a.acc[4 * lane + k];
#pragma unroll
        for (int k = 0; k < 4; k++) recip[k] = wave_sum(recip[k]);
    }
    // the step's record index (the last workgroup advances it after every
    // workgroup has read it)
    const int rec = (S2 && a.energies) ? a.flags[F_STEP] : a.ecap;
    double *record = rec < a.ecap ? a.energies + (size_t)rec * kReduceSlots : nullptr;
    if (S2 && record && bid >= nb - ncb) {
        // the columns the step's kernels filled with partial rows, in a fixed
        // order, eight rows of a lane in flight
        for (int col = (bid - (nb - ncb)) * NW + wid; col < kReduceSlots; col += kStepColumnBlocks * NW) {
            if (atomic_column(col)) continue;
            const int rows = a.rows[col];
            constexpr int U = 8;
            double s[U];
#pragma unroll
            for (int u = 0; u < U; u++) s[u] = 0.0;
            for (int r = lane; r < rows; r += 64 * U)
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (r + 64 * u < rows) s[u] += a.red[(size_t)(r + 64 * u) * kReduceSlots + col];
            const double v = wave_sum(((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7])));
            if (lane == 0) record[col] = v;
        }
    }
    double ke = 0.0, r2 = 0.0;
    const double mx = recip[1] * a.inv_n, my = recip[2] * a.inv_n, mz = recip[3] * a.inv_n;
    for (; i < a.n; i += stride) {
        if (i + stride < a.n) load(i + stride, nxt);
        double4 v = cur.v, f = cur.f;
        if (S2) {
            if (a.frc_recip) {
                f.x += (cur.r.x - mx) * a.two_scale;
                f.y += (cur.r.y - my) * a.two_scale;
                f.z += (cur.r.z - mz) * a.two_scale;
            }
            if (a.frz && a.frz[a.gid[i]] != 0) {
                f.x = f.y = f.z = 0.0;
                v.x = v.y = v.z = 0.0;
            }
            if (!S1) a.frc[i] = f;
            if (v.w > 1.0e-6) {
                const double tmp = (0.5 * a.dt) / v.w;
                v.x += tmp * f.x;
                v.y += tmp * f.y;
                v.z += tmp * f.z;
                ke += v.w * (v.x * v.x + v.y * v.y + v.z * v.z);
            }
        }
        if (S1) {
            double4 p = cur.p;
            if (v.w > 1.0e-6) {
                const double tmp = (0.5 * a.dt) / v.w;
                v.x += tmp * f.x;
                v.y += tmp * f.y;
                v.z += tmp * f.z;
                p.x += a.dt * v.x;
                p.y += a.dt * v.y;
                p.z += a.dt * v.z;
                a.pos[i] = p;
            }
            const double dx = min_image_1(p.x, cur.q.x, a.b.L[0], a.b.invL[0]);
            const double dy = min_image_1(p.y, cur.q.y, a.b.L[1], a.b.invL[1]);
            const double dz = min_image_1(p.z, cur.q.z, a.b.L[2], a.b.invL[2]);
            r2 = fmax(r2, dx * dx + dy * dy + dz * dz);
        }
        a.vel[i] = v;
        cur = nxt;
    }
    auto wave_max = [](double x) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) x = fmax(x, __shfl_xor(x, o, 64));
        return x;
    };
    if (S2) ke = wave_sum(ke);
    if (S1) r2 = wave_max(r2);
    if (lane == 0) {
        wke[wid] = ke;
        wr2[wid] = r2;
    }
    __syncthreads();
    if (t == 0) {
        double k = 0.0, m = 0.0;
        for (int w = 0; w < NW; w++) {
            k += wke[w];
            m = fmax(m, wr2[w]);
        }
        __hip_atomic_store(&a.part[2 * bid], k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&a.part[2 * bid + 1], m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        wait_memory();
        last = atomicAdd((unsigned int *)(a.flags + F_DONE), 1u) == (unsigned)nb - 1;
    }
    __syncthreads();
    if (!last) return;
    // the last workgroup: every other one has read acc and F_STEP and its
    // partials are in part[]
    if (S2 && a.acc && t < 4 * kAccSlots)  // the gather's slots cleared for the next step
        __hip_atomic_store(&a.acc[t], 0.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (wid != 0) return;
    ke = r2 = 0.0;
    for (int b = lane; b < nb; b += 64) {
        if (S2 && record) ke += load_coherent(&a.part[2 * b]);
        if (S1) r2 = fmax(r2, load_coherent(&a.part[2 * b + 1]));
    }
    if (S2 && record) ke = wave_sum(ke);
    if (S1) r2 = wave_max(r2);
    if (lane != 0) return;
    if (S2 && a.energies) {
        if (record) {
            record[R_KIN] = ke;
#pragma unroll
            for (int k = 0; k < 4; k++) record[R_ERECIP + k] = recip[k];
        }
        a.flags[F_STEP] = rec + 1;
    }
    if (S1) {
        const int upd = (a.half_pad <= 0.0 || sqrt(r2) >= a.half_pad) ? 1 : 0;
        a.flags[F_UPD] = upd;
        if (upd) {
            a.flags[F_OVF] = 0;
            a.flags[F_IBIG] = 0;
            a.flags[F_PAIRS] = 0;
            a.flags[F_NREB] += 1;
        }
    }
    __hip_atomic_store((unsigned int *)(a.flags + F_DONE), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool S2, bool S1>
__global__ void __launch_bounds__(kStepThreads) k_step_batch(const StepArgs *__restrict__ av,
                                                            const int32_t *__restrict__ boff, int nsys)
{
    const int lb = blockIdx.x;  // atoms in order: no XCD renumbering
    if (lb >= boff[nsys]) return;
    const int s = batch_find(boff, nsys, lb);
    step_body<S2, S1>(av[s], lb - boff[s], boff[s + 1] - boff[s]);
}

static int step_blocks(const Ctx *c, bool energies)
{
    const int cols = energies ? kStepColumnBlocks : 0;
    return std::min(ceil_div(c->natms, kStepThreads), kStepBlocks - cols) + cols;
}

int step_prepare(const std::vector<Ctx *> &cs, const std::vector<RedRowsHost> &rows, bool energies,
                 BatchLaunch &bl)
{
    std::vector<StepArgs> av;
    std::vector<int> nb;
    for (size_t k = 0; k < cs.size(); k++) {
        Ctx *c = cs[k];
        StepArgs a{};
        a.pos = c->pos;
        a.vel = c->vel;
        a.frc = c->frc;
        a.frc_recip = c->prm.electrostatics ? c->frc_recip : nullptr;
        a.xref = c->xref;
        a.gid = c->gid;
        a.frz = c->nfrozen > 0 ? c->frz : nullptr;
        a.n = c->natms;
        a.dt = c->run_dt;
        a.two_scale = c->prm.electrostatics ? 2.0 * recip_scale(c) : 0.0;
        a.inv_n = 1.0 / (double)c->natms;
        a.half_pad = kHalfMinus * c->prm.padding;
        for (int d = 0; d < 3; d++) {
            a.b.L[d] = c->L[d];
            a.b.invL[d] = c->invL[d];
        }
        a.red = c->red;
        a.part = c->step_part;
        a.acc = c->prm.electrostatics ? c->acc : nullptr;
        for (int q = 0; q < kReduceSlots; q++) a.rows[q] = rows[k].rows[q];
        a.energies = energies ? c->energies_dev : nullptr;
        a.ecap = c->energies_cap;
        a.flags = c->flags;
        av.push_back(a);
        nb.push_back(step_blocks(c, energies));
    }
    return batch_upload(cs[0], bl, av.data(), sizeof(StepArgs), nb, false);
}

int step_launch(Ctx *c, hipStream_t s, const BatchLaunch &bl, bool stage2, bool stage1)
{
    const dim3 g(bl.total), b(kStepThreads);
    const StepArgs *av = (const StepArgs *)bl.args;
    if (stage2 && stage1) hipLaunchKernelGGL((k_step_batch<true, true>), g, b, 0, s, av, bl.boff, bl.nsys);
    else if (stage2) hipLaunchKernelGGL((k_step_batch<true, false>), g, b, 0, s, av, bl.boff, bl.nsys);
    else if (stage1) hipLaunchKernelGGL((k_step_batch<false, true>), g, b, 0, s, av, bl.boff, bl.nsys);
    DLPX_HIP(c, hipGetLastError());
    return 0;
}

int load_blocks(const Ctx *c) { return ceil_div(c->natms, kLoadThreads); }

int load_atoms(Ctx *c, bool identity, bool with_vel, bool disp)
{
    LoadArgs a{};
    if (!identity) {
        StrayArgs &sa = a.stray;
        sa.xref = c->xref;
        if (c->tile_cap > 0) {
            for (int d = 0; d < 3; d++) {
                sa.invL0[d] = 1.0 / c->list_L[d];
                sa.invL[d] = c->invL[d];
                sa.reach[d] = tile_reach(c, d);
            }
            sa.flag = c->flags + F_STRAY;
            a.clear = tile_found(c);
            a.nclear = tile_blocks(c);
        }
        c->upload_no = c->upload_no == INT32_MAX ? 1 : c->upload_no + 1;
        sa.no = c->upload_no;
    }
    c->stray_no = a.stray.no;
    a.st = c->h_st_dev;
    a.st_t = c->h_t_dev;
    a.n = c->natms;
    a.row = with_vel ? 8 : 4;
    a.slot = identity ? nullptr : c->slot;
    a.pos = c->pos;
    a.vel = c->vel;
    a.typ = c->typ;
    a.gid = c->gid;
    a.disp = disp ? (unsigned long long *)c->h_disp_dev : nullptr;
    for (int d = 0; d < 3; d++) {
        a.b.L[d] = c->L[d];
        a.b.invL[d] = c->invL[d];
    }
    c->rows_busy = true;
    hipLaunchKernelGGL(k_load, dim3(load_blocks(c)), dim3(kLoadThreads), 0, c->stream, a);
    DLPX_HIP(c, hipGetLastError());
    return 0;
}

int store_atoms(Ctx *c, bool with_state, bool finish)
{
    StoreArgs a{};
    a.out = c->h_st_dev;
    a.n = c->natms;
    a.slot = c->slot;
    a.pos = c->pos;
    a.vel = c->vel;
    a.frc = c->frc;
    a.frc_recip = finish ? c->frc_recip : nullptr;
    a.red_out = c->red_out;
    a.two_scale = finish ? 2.0 * recip_scale(c) : 0.0;
    a.inv_n = 1.0 / (double)c->natms;
    const dim3 grid(ceil_div(c->natms, kStoreThreads));
    c->rows_busy = true;
    if (with_state) hipLaunchKernelGGL(k_store<9>, grid, dim3(kStoreThreads), 0, c->stream, a);
    else hipLaunchKernelGGL(k_store<3>, grid, dim3(kStoreThreads), 0, c->stream, a);
    DLPX_HIP(c, hipGetLastError());
    return 0;
}

int store_per_particle(Ctx *c, double scale)
{
    c->rows_busy = true;
    hipLaunchKernelGGL(k_store_pp, dim3(ceil_div(c->natms, kStoreThreads)), dim3(kStoreThreads), 0, c->stream,
                       c->h_st_dev, c->natms, c->slot, c->pp, c->prm.electrostatics ? c->frc_recip : nullptr, scale);
    DLPX_HIP(c, hipGetLastError());
    return 0;
}

}  // namespace dlpx
