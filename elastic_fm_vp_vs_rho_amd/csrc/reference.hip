// Reference-style adjoint and imaging, for drop-in parity with
// Elastic3D.backwardFields (M:2056-2082) and
// Elastic3D.backwardFields_FowardFieldsRemake (M:1929-2054).
//
// The reference runs the forward operator (+dt) on a zeroed adjoint state with
// the residual injected time-reversed into v (kernel_add_adjoint_source,
// M:310-322), rebuilds the forward wavefield in reverse time from the last
// state with the saved CPML boundaries (kernel_set_border, M:422-462), zeroes
// the x/y/bottom CPML zones (kernel_setZero_CPMLzone, M:466-499), and forms
// continuous-adjoint imaging conditions (kernel_Gradients_Rho/_Lambda/_Mu,
// M:191-294; kernel_Gradients_Mij, M:337-372).  It keeps an extra copy of v
// (kernel_DTD_copy, M:501-511); here the reverse velocity sweep writes
// out of place and the two v buffers swap roles, so no copy is made.
//
// An iteration is two launches instead of eight (see backward_remake_ref): the adjoint
// sweep and the reconstruction's sweep of one kind share a launch, the adjoint stress
// sweep forms the images of the iteration before (it holds the cell's v, τ and moduli),
// and the velocity sweeps inject the residual and restore the borders.
#include <string>
#include <utility>

#include "sweeps.hpp"

namespace efm {

__global__ void k_inject_ref(Geo g, ShotPtrs sh, StatePtrs a, const float *res, int it) {
    const int s = g.s0 + blockIdx.x;
    const int nts = sh.nt[s];
    const int n = nts - it - 1;
    if (n < 0 || n >= nts) return;
    for (int r = threadIdx.x; r < g.nrec; r += blockDim.x) {
        const int cell = sh.rec[(long long)s * g.nrec + r];
        if (cell < 0) continue;
        const long long t = (long long)s * g.N + cell;
        const long long base = ((long long)s * 3 * g.ntmax + n) * g.nrec + r;
        const long long cs = (long long)g.ntmax * g.nrec;
        atomicAdd(&a.v[0][t], res[base]);
        atomicAdd(&a.v[1][t], res[base + cs]);
        atomicAdd(&a.v[2][t], res[base + 2 * cs]);
    }
}

// Single thread per shot, like the reference (which uses thread 0 of one block);
// the reference evaluates this with double literals, so it is done in double.
__global__ void k_image_mt_ref(Geo g, const float *lam, const float *mu, ShotPtrs sh, StatePtrs a,
                               double *gm6, int it) {
    const int s = g.s0 + blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.s0 + g.S) return;
    const int nts = sh.nt[s];
    if (it >= nts) return;
    const int *sp = sh.src + 3 * s;
    const long long nx = g.nx, sxz = g.sxz;
    const long long lc = sp[0] + sp[2] * nx + sp[1] * sxz;
    const long long t = (long long)s * g.N + lc;
    const double Mu = mu[lc], L = lam[lc];
    const double Mi = mu[lc + 1], Mk = mu[lc + nx], Mj = mu[lc + sxz];
    const double Mik = mu[lc + 1 + nx], Mjk = mu[lc + nx + sxz], Mij = mu[lc + 1 + sxz];
    const double mxz = 1.0 / (0.25 / Mu + 0.25 / Mi + 0.25 / Mk + 0.25 / Mik);
    const double mxy = 1.0 / (0.25 / Mu + 0.25 / Mi + 0.25 / Mj + 0.25 / Mij);
    const double myz = 1.0 / (0.25 / Mu + 0.25 / Mj + 0.25 / Mk + 0.25 / Mjk);
    const double w = sh.wav[(long long)s * g.ntmax + (nts - it - 1)];
    const double txx = a.t[0][t], tyy = a.t[1][t], tzz = a.t[2][t];
    const double txy = a.t[3][t], txz = a.t[4][t], tyz = a.t[5][t];
    const double k = 1.0 / (2.0 * Mu * (3.0 * L + 2.0 * Mu));
    double *o = gm6 + 6 * s;
    // each term is stored to float in the reference before the host sum
    o[0] += (float)(w * k * (2.0 * (L + Mu) * txx - L * tyy - L * tzz));
    o[1] += (float)(w * k * (2.0 * (L + Mu) * tyy - L * txx - L * tzz));
    o[2] += (float)(w * k * (2.0 * (L + Mu) * tzz - L * txx - L * tyy));
    o[3] += (float)(w * (1.0 / mxy) * txy);
    o[4] += (float)(w * (1.0 / mxz) * txz);
    o[5] += (float)(w * (1.0 / myz) * tyz);
}

// What the images of an iteration take besides the adjoint state: the reconstruction's
// velocities after and before the iteration, and where the images go (glam null: none).
struct ImageRef {
    const float *f[3], *fp[3];
    float idt, idx, idy, idz;
    float *glam, *gmu, *grho;
};

// λ/μ/ρ imaging conditions of cell i of the shot at offset so, `o` the adjoint's cell,
// accumulated in float32 (the reference adds the
// per-step device volumes on the host in float32).  Divisions by the medium
// use the hardware reciprocal (1 ulp) and those by dt, dx, dy, dz the
// reciprocals of the steps: the images move by a few ulp, far inside the
// 1e-4 the gradients are held to.  Index arithmetic is 32-bit (N < 2^31).
__device__ __forceinline__ void image_cell(const Geo &g, const ImageRef &im, CellOld o, long long so, int i) {
    const int nx = g.nx, sxz = g.sxz32;
    const float *__restrict__ vx = im.fp[0] + so, *__restrict__ vy = im.fp[1] + so, *__restrict__ vz = im.fp[2] + so;
    const float *__restrict__ fx = im.f[0] + so, *__restrict__ fy = im.f[1] + so, *__restrict__ fz = im.f[2] + so;
    // M:206
    const float r = -((o.vx * (vx[i] - fx[i]) * im.idt) + (o.vy * (vy[i] - fy[i]) * im.idt) +
                      (o.vz * (vz[i] - fz[i]) * im.idt));
    const float L = o.lam, M = o.mu;
    // M:234-238
    const float dvx = 0.5f * (vx[i] - vx[i - 1]) * im.idx + 0.5f * (vx[i - 1] - vx[i - 2]) * im.idx;
    const float dvy = 0.5f * (vy[i] - vy[i - sxz]) * im.idy + 0.5f * (vy[i - sxz] - vy[i - 2 * sxz]) * im.idy;
    const float dvz = 0.5f * (vz[i] - vz[i - nx]) * im.idz + 0.5f * (vz[i - nx] - vz[i - 2 * nx]) * im.idz;
    const float k3 = frcp(3.f * L + 2.f * M);
    const float gl = (o.txx + o.tyy + o.tzz) * (dvx + dvy + dvz) * k3;
    // M:262-291: 1/μ̄ for the three shear planes (the reference inverts the
    // harmonic mean and then inverts it back; here the sum of quarter
    // reciprocals is used directly)
    const float q0 = 0.25f * o.r0, qi = 0.25f * o.ri, qk = 0.25f * o.rk, qj = 0.25f * o.rj;
    const float imxz = q0 + qi + qk + 0.25f * o.rik;
    const float imxy = q0 + qi + qj + 0.25f * o.rij;
    const float imyz = q0 + qj + qk + 0.25f * o.rjk;
    const float ex = vx[i] - vx[i - 1], ey = vy[i] - vy[i - sxz], ez = vz[i] - vz[i - nx];
    const float dvx_dz = vx[i + nx] - vx[i], dvx_dy = vx[i + sxz] - vx[i];
    const float dvy_dx = vy[i + 1] - vy[i], dvy_dz = vy[i + nx] - vy[i];
    const float dvz_dx = vz[i + 1] - vz[i], dvz_dy = vz[i + sxz] - vz[i];
    const float k = o.r0 * k3;
    const float gm = k * (2.f * (L + M) * o.txx - L * o.tyy - L * o.tzz) * ex
                   + k * (2.f * (L + M) * o.tyy - L * o.txx - L * o.tzz) * ey
                   + k * (2.f * (L + M) * o.tzz - L * o.txx - L * o.tyy) * ez
                   + imxy * o.txy * (dvy_dx + dvx_dy)
                   + imxz * o.txz * (dvx_dz + dvz_dx)
                   + imyz * o.tyz * (dvz_dy + dvy_dz);
    im.glam[so + i] += gl;
    im.gmu[so + i] += gm;
    im.grho[so + i] += r;
}

// Jobs of a shared launch: the adjoint's sweep and the reconstruction's, as shots
// s0 .. s0+S-1 of the first and then of the second (job0: the first job present).
__device__ __forceinline__ int split_job(const Geo &g, int job0, int &s) {
    const int j = (s - g.s0) / g.S;
    s -= j * g.S;
    return job0 + j;
}
__host__ __device__ inline Geo with_jobs(Geo g, int njobs) {
    g.S *= njobs;
    return g;
}
__device__ __forceinline__ Geo reversed(Geo g) {
    g.c = -g.c;
    return g;
}
constexpr int kAdjoint = 0, kRemake = 1;

// Adjoint stress sweep of iteration `it` with the images of iteration it - 1, and the
// reconstruction's stress sweep of iteration it - 1 (c = -ga.c) outside the x, y and
// bottom CPML zones: τ there only reaches velocities that the restored borders
// and the zeroing replace.  100^3, W = 10: 27 us for both, against 15 + 15 + 17 us
// of the sweeps and the images alone (each about 4 us of launch, and the images read
// again what the sweep holds).  Without `step` the adjoint's job forms the images alone
// (behind a range's last iteration).
template <int BX, int BZ, int NYC, int MAP>
__global__ EFM_KERNEL_ATTRS(BX, BZ, MAP) void k_ref_stress(Geo g, Med m, ShotPtrs sh, StatePtrs a, StatePtrs f, int it,
                                                           int step, ImageRef im, int W, int job0, int njobs) {
    int x, z, s, yb;
    if (!tile_coords<BX, BZ, NYC, MAP>(with_jobs(g, njobs), x, z, s, yb)) return;
    if (x < H || x >= g.nx - H || z < H || z >= g.nz - H) return;
    const int y0 = H + yb * NYC, y1 = min(y0 + NYC, g.ny - H);
    if (split_job(g, job0, s) == kAdjoint) {
        const long long sa = (long long)s * g.N;
        const bool write = step && it < sh.nt[s];
        if (!write && !im.glam) return;
        stress_cells<NYC>(g, m, sh, a, a, it, 0, x, z, s, yb, write, [&](int t, CellOld o) EFM_INLINE {
            if (im.glam) image_cell(g, im, o, sa, t);
        });
    } else {
        if (x < W || x >= g.nx - W || z >= g.nz - W || y1 <= W || y0 >= g.ny - W) return;
        if (it - 1 >= sh.nt[s]) return;
        stress_cells<NYC>(reversed(g), m, sh, f, f, it - 1, -1, x, z, s, yb, true, [](int, CellOld) {});
    }
}

// Border element of an interior cell outside the zeroed zones, or -1.
__device__ __forceinline__ long long border_of(const Geo &g, const BorderLayout &L, int W, int x, int y, int z) {
    const long long yz = (long long)y * g.nz + z, yh = (long long)y * H + z;
    if (x < W + H) return L.left + yz * H + x - W;
    if (x >= g.nx - W - H) return L.right + yz * H + x - (g.nx - W - H);
    if (z < 2 * H) return L.top + (yh - H) * g.nx + x;
    if (z >= g.nz - W - H) return L.bottom + (yh - (g.nz - W - H)) * g.nx + x;
    if (y < W + H) return L.front + ((long long)(y - W) * g.nz + z) * g.nx + x;
    if (y >= g.ny - W - H) return L.back + ((long long)(y - (g.ny - W - H)) * g.nz + z) * g.nx + x;
    return -1;
}

// Border elements of a component in the two guard rows at the top of the left, right,
// front and back faces, the only ones outside the interior and the zones (W >= H).
__host__ __device__ inline int guard_borders(const Geo &g) { return 4 * H * (g.nx + g.ny); }
__device__ __forceinline__ void restore_guard(const Geo &g, const BorderLayout &L, const float *slot, int W, float *v,
                                              int i) {
    const int per = i < 4 * H * g.ny ? g.ny : g.nx;
    const int k = i < 4 * H * g.ny ? i : i - 4 * H * g.ny;
    const int along = k % per, q = k / per, h = q % H, z = q / H % H, side = q / (H * H);
    int x, y;
    long long e;
    if (per == g.ny && i < 4 * H * g.ny) {
        y = along;
        x = side ? g.nx - W - H + h : W + h;
        e = L.left + side * (L.right - L.left) + ((long long)y * g.nz + z) * H + h;
    } else {
        x = along;
        y = side ? g.ny - W - H + h : W + h;
        e = L.front + side * (L.back - L.front) + ((long long)h * g.nz + z) * g.nx + x;
    }
    if (x < W || x >= g.nx - W || y < W || y >= g.ny - W) return;       // zeroed
    v[x + z * g.nx + y * g.sxz32] = slot[e];
}

// Adjoint velocity sweep of iteration `it`, with the residual added at its receivers
// (res null: not here), and the reconstruction's velocity sweep of the iteration, from
// cur to nxt, whose border cells take the saved values of step `slot` and whose x, y and
// bottom CPML zones stay zero.  Blocks behind the sweeps serve receivers and border
// elements in the guard rows.  100^3: 22.5 us, against 12 + 12 + 8 + 5 + 7 us of two sweeps,
// injection, border and zeroing.
template <int BX, int BZ, int NYC, int MAP>
__global__ EFM_KERNEL_ATTRS(BX, BZ, MAP) void k_ref_velocity(Geo g, Med m, ShotPtrs sh, StatePtrs a, StatePtrs cur,
                                                             StatePtrs nxt, int it, const float *res,
                                                             const float *borders, int W, int slot, int njobs,
                                                             long long nsweep) {
    const BorderLayout L = border_layout(g.nx, g.ny, g.nz);
    const long long cs = (long long)g.ntmax * g.nrec;
    const long long extra = block_number() - nsweep;
    if (extra >= 0) {
        long long k = extra * (BX * BZ) + threadIdx.y * BX + threadIdx.x;
        if (res) {
            if (k < (long long)g.S * g.nrec) {
                const int s = g.s0 + (int)(k / g.nrec), r = (int)(k % g.nrec);
                const int cell = sh.rec[(long long)s * g.nrec + r], n = sh.nt[s] - it - 1;
                if (cell < 0 || n < 0) return;
                const int row = cell / g.nx, y = row / g.nz;
                if (interior(cell - row * g.nx, y, row - y * g.nz, g)) return;
                const long long t = (long long)s * g.N + cell, base = ((long long)s * 3 * g.ntmax + n) * g.nrec + r;
                atomicAdd(&a.v[0][t], res[base]);
                atomicAdd(&a.v[1][t], res[base + cs]);
                atomicAdd(&a.v[2][t], res[base + 2 * cs]);
                return;
            }
            k -= (long long)g.S * g.nrec;
        }
        const long long per = 3LL * guard_borders(g), sl = k / per;
        if (njobs < 2 || sl >= g.S) return;
        const int s = g.s0 + (int)sl, i = (int)(k - sl * per), c = i / guard_borders(g);
        restore_guard(g, L, borders + (((long long)s * g.ntmax + slot) * 3 + c) * L.comp, W,
                      (c == 0 ? nxt.v[0] : c == 1 ? nxt.v[1] : nxt.v[2]) + (long long)s * g.N, i - c * guard_borders(g));
        return;
    }
    int x, z, s, yb;
    if (!tile_coords<BX, BZ, NYC, MAP>(with_jobs(g, njobs), x, z, s, yb)) return;
    if (x < H || x >= g.nx - H || z < H || z >= g.nz - H) return;
    if (split_job(g, kAdjoint, s) == kAdjoint) {
        const int n = sh.nt[s] - it - 1;
        if (n < 0) return;
        velocity_cells<NYC>(g, m, sh, a, a, x, z, s, yb, [&](int, int t, float &v0, float &v1, float &v2) EFM_INLINE {
            if (res) inject_wave(g, sh, s, t, res, n, v0, v1, v2);
        }, [](int, float, float, float) {});
    } else {
        const int y0 = H + yb * NYC, y1 = min(y0 + NYC, g.ny - H);
        if (x < W || x >= g.nx - W || z >= g.nz - W || y1 <= W || y0 >= g.ny - W) return;
        const float *buf = borders + ((long long)s * g.ntmax + slot) * 3 * L.comp;
        auto restore = [&](int y, int, float &v0, float &v1, float &v2) EFM_INLINE {
            if (y < W || y >= g.ny - W) { v0 = v1 = v2 = 0.f; return; }
            const long long e = border_of(g, L, W, x, y, z);
            if (e < 0) return;
            v0 = buf[e];
            v1 = buf[e + L.comp];
            v2 = buf[e + 2 * L.comp];
        };
        if (it >= sh.nt[s]) {
            // the shot's record is over: its borders are restored all the same
            for (int y = y0; y < y1; ++y) {
                const long long t = (long long)s * g.N + x + z * g.nx + y * g.sxz32;
                float v0 = nxt.v[0][t], v1 = nxt.v[1][t], v2 = nxt.v[2][t];
                restore(y, 0, v0, v1, v2);
                nxt.v[0][t] = v0; nxt.v[1][t] = v1; nxt.v[2][t] = v2;
            }
            return;
        }
        velocity_cells<NYC>(reversed(g), m, sh, cur, nxt, x, z, s, yb, restore, [](int, float, float, float) {});
    }
}

__global__ void k_zero_cpml(Geo g, StatePtrs f, int W) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int s = g.s0 + blockIdx.y;
    if (i >= g.N) return;
    const int row = i / g.nx;
    const int x = i - row * g.nx;
    const int y = row / g.nz;
    const int z = row - y * g.nz;
    if (!(x < W || x >= g.nx - W || z >= g.nz - W || y < W || y >= g.ny - W)) return;
    const long long t = (long long)s * g.N + i;
    for (int k = 0; k < 3; ++k) f.v[k][t] = 0.f;
    for (int k = 0; k < 6; ++k) f.t[k][t] = 0.f;
}

}  // namespace efm

using namespace efm;

static inline unsigned nblk(long long n, int b) { return (unsigned)((n + b - 1) / b); }

static int check_common(const EfmDims *d, const EfmMedium *m, const EfmShots *sh) {
    return validate(d, m, sh);
}

extern "C" int efm_inject_residual(const EfmDims *d, const EfmShots *sh, const EfmState *st,
                                   const float *res, int it, void *stream) {
    if (!d || !sh || !st || (!res && d->nrec > 0))
        return fail(EFM_E_ARG, "efm_inject_residual: null argument");
    if (int rc = check_dims(d)) return rc;
    if (int rc = validate_shots(d, sh)) return rc;
    if (int rc = validate_state(d, st)) return rc;
    const Geo g = make_geo(*d);
    if (g.nrec <= 0) return EFM_OK;
    hipLaunchKernelGGL(k_inject_ref, dim3(g.S), dim3(64), 0, (hipStream_t)stream, g,
                       make_shots(*sh), make_state(*st), res, it);
    return check_launch("inject residual");
}

extern "C" int efm_image_mt_ref(const EfmDims *d, const EfmMedium *m, const EfmShots *sh,
                                const EfmState *adj, double *gm6, int it, void *stream) {
    int rc = check_common(d, m, sh);
    if (rc) return rc;
    if (!adj || !gm6) return fail(EFM_E_ARG, "efm_image_mt_ref: null argument");
    if ((rc = validate_state(d, adj))) return rc;
    const Geo g = make_geo(*d);
    hipLaunchKernelGGL(k_image_mt_ref, dim3(nblk(g.S, 64)), dim3(64), 0, (hipStream_t)stream, g,
                       m->lam, m->mu, make_shots(*sh), make_state(*adj), gm6, it);
    return check_launch("image mt");
}

extern "C" int efm_backward_mt_ref(const EfmDims *d, const EfmMedium *m, const EfmShots *sh,
                                   const EfmState *adj, const float *res, double *gm6, int nsteps,
                                   void *stream) {
    int rc = check_common(d, m, sh);
    if (rc) return rc;
    if (!adj || (!res && d->nrec > 0) || !gm6)
        return fail(EFM_E_ARG, "efm_backward_mt_ref: null argument");
    if ((rc = validate_state(d, adj))) return rc;
    if (nsteps < 0 || nsteps > d->ntmax) return fail(EFM_E_ARG, "efm_backward_mt_ref: nsteps out of range");
    Geo g = make_geo(*d);
    if (g.c < 0) g.c = -g.c;  // the adjoint runs the forward operator with +dt (M:2066-2068)
    hipStream_t st = (hipStream_t)stream;
    const ShotPtrs shp = make_shots(*sh);
    const StatePtrs a = make_state(*adj);
    for (int it = 0; it < nsteps; ++it) {
        if ((rc = launch_stress_src(g, *m, shp, a, a, it, 0, st))) return rc;
        if ((rc = launch_velocity(g, *m, shp, a, a, it, st))) return rc;
        if (g.nrec > 0) {
            hipLaunchKernelGGL(k_inject_ref, dim3(g.S), dim3(64), 0, st, g, shp, a, res, it);
            if ((rc = check_launch("inject residual"))) return rc;
        }
        hipLaunchKernelGGL(k_image_mt_ref, dim3(nblk(g.S, 64)), dim3(64), 0, st, g, m->lam, m->mu,
                           shp, a, gm6, it);
        if ((rc = check_launch("image mt"))) return rc;
    }
    return EFM_OK;
}

extern "C" long long efm_border_floats(const EfmDims *d, int W) {
    if (!d || check_dims(d)) return -1;
    return border_floats(make_geo(*d), W);
}

// Whether the sweeps of njobs jobs, and `extra` blocks, fit one dispatch (< 2^32
// work-items, 65535 blocks along z).
static bool jobs_fit(const Geo &g, int njobs, const Tile &t, long long extra) {
    const dim3 d = sweep_grid_plus(with_jobs(g, njobs), t, extra);
    return grid_blocks(d) * t.bx * t.bz <= (long long)UINT32_MAX && d.z <= 65535;
}

static int launch_ref_stress(const Geo &g, const Med &md, const ShotPtrs &sh, const StatePtrs &a, const StatePtrs &f,
                             int it, bool step, const ImageRef &im, int W, int job0, int njobs, hipStream_t st) {
    const Tile t = get_tile(0);
    if (njobs == 2 && !jobs_fit(g, 2, t, 0)) {
        if (int rc = launch_ref_stress(g, md, sh, a, f, it, step, im, W, kAdjoint, 1, st)) return rc;
        return launch_ref_stress(g, md, sh, a, f, it, step, im, W, kRemake, 1, st);
    }
    const dim3 grid = sweep_grid(with_jobs(g, njobs), t);
    bool launched = false;
#define X(a_, b_, c_, o_) \
    EFM_LAUNCH_GRID_IF(a_, b_, c_, o_, grid, k_ref_stress, g, md, sh, a, f, it, step, im, W, job0, njobs)
    EFM_TILE_LIST(X)
#undef X
    if (!launched) return fail(EFM_E_UNSUPPORTED, "unsupported stress tile");
    return check_launch("reverse stress sweeps");
}

// njobs 1: the adjoint's sweep alone; the residual then takes a launch of its own where the
// blocks for its receivers would pass a dispatch's limit.
static int launch_ref_velocity(const Geo &g, const Med &md, const ShotPtrs &sh, const StatePtrs &a,
                               const StatePtrs &cur, const StatePtrs &nxt, int it, const float *res,
                               const float *borders, int W, int slot, int njobs, hipStream_t st) {
    const Tile t = get_tile(1);
    const auto blocks = [&](long long n) { return (n + t.bx * t.bz - 1) / (t.bx * t.bz); };
    const bool fused = sh.recmask && g.nrec > 0 && (njobs == 2 || jobs_fit(g, 1, t, blocks((long long)g.S * g.nrec)));
    const long long n = (fused ? (long long)g.S * g.nrec : 0) + (njobs == 2 ? 3LL * guard_borders(g) * g.S : 0);
    const long long extra = blocks(n);
    const Geo gj = with_jobs(g, njobs);
    const dim3 grid = sweep_grid_plus(gj, t, extra);
    const long long nsweep = grid_blocks(sweep_grid(gj, t));
    bool launched = false;
#define X(a_, b_, c_, o_)                                                                                  \
    EFM_LAUNCH_GRID_IF(a_, b_, c_, o_, grid, k_ref_velocity, g, md, sh, a, cur, nxt, it,                   \
                       fused ? res : nullptr, borders, W, slot, njobs, nsweep)
    EFM_TILE_LIST(X)
#undef X
    if (!launched) return fail(EFM_E_UNSUPPORTED, "unsupported velocity tile");
    if (int rc = check_launch("reverse velocity sweeps")) return rc;
    if (fused || g.nrec <= 0) return EFM_OK;
    hipLaunchKernelGGL(k_inject_ref, dim3(g.S), dim3(64), 0, st, g, sh, a, res, it);
    return check_launch("inject residual");
}

// Iterations it0 .. it0+nsteps-1 of the reverse loop.  The present velocity
// alternates between the forward state's v and vpres (swapped every
// iteration), so iteration `it` finds it in fwd.v when it is even and in vpres
// when it is odd.
//
// Iteration it: [adjoint stress, images of it-1 | reconstruction's stress of it-1],
// [adjoint velocity, residual | reconstruction's velocity, borders].  The
// reconstruction's stress sweep and the images of an iteration need what both of its
// velocity sweeps wrote and nothing after them, so they wait for the next launch; the
// last iteration's get one of their own.  The zones of both velocity buffers are
// zeroed, guard cells included, behind a range's first two iterations; no later one
// writes them.  Every iteration's sweeps and images are the same kernels wherever a
// range starts or ends, so a run split into ranges leaves the bits of one run over all
// nt-1 iterations.  A CPML narrower than the guard layer has the reconstruction's
// velocity sweep, the borders and the zeroing as separate launches throughout, as does
// a batch whose two sweeps exceed one dispatch.
static int backward_remake_ref(const EfmDims *d, const EfmMedium *m, const EfmShots *sh,
                               const EfmState *fwd, float *vpres, const float *borders, int W,
                               const EfmState *adj, const float *res, float dt, float dx, float dy,
                               float dz, float *glam, float *gmu, float *grho, int it0, int nsteps,
                               void *stream, const char *who) {
    int rc = check_common(d, m, sh);
    if (rc) return rc;
    if (!fwd || !vpres || !borders || !adj || (!res && d->nrec > 0) || !glam || !gmu || !grho)
        return fail(EFM_E_ARG, std::string(who) + ": null argument");
    if ((rc = validate_state(d, fwd)) || (rc = validate_state(d, adj))) return rc;
    if (W + H + 1 > d->nx / 2 || W + H + 1 > d->ny / 2 || W + H + 1 > d->nz / 2)
        return fail(EFM_E_ARG, std::string(who) + ": CPML too wide for the grid");
    const int nt = d->ntmax;
    if (it0 < 0 || nsteps < 0 || it0 + nsteps > nt - 1)
        return fail(EFM_E_ARG, std::string(who) + ": iterations outside [0, nt-1)");
    Geo ga = make_geo(*d);
    if (ga.c < 0) ga.c = -ga.c;
    Geo gf = ga;
    gf.c = -ga.c;  // flagMode = 1 reverse stepping (M:1951, 1964)
    hipStream_t st = (hipStream_t)stream;
    const Med md{m->lam, m->mu, m->rho};
    const ShotPtrs shp = make_shots(*sh);
    const StatePtrs a = make_state(*adj);
    StatePtrs cur = make_state(*fwd);           // v buffers: cur = present
    StatePtrs nxt = cur;                         // nxt.v = the other buffer
    const long long vol = (long long)ga.S * ga.N;
    nxt.v[0] = vpres; nxt.v[1] = vpres + vol; nxt.v[2] = vpres + 2 * vol;
    if (it0 & 1) std::swap(cur.v, nxt.v);
    const bool fits = W >= H && jobs_fit(ga, 2, get_tile(1), (long long)ga.S * (ga.nrec + 3LL * guard_borders(ga)));
    // cur and nxt after an iteration's swap: the reconstruction's new and old velocities
    auto images = [&]() {
        return ImageRef{{cur.v[0], cur.v[1], cur.v[2]}, {nxt.v[0], nxt.v[1], nxt.v[2]}, 1.f / dt, 1.f / dx, 1.f / dy,
                        1.f / dz, glam, gmu, grho};
    };
    for (int it = it0; it < it0 + nsteps; ++it) {
        const bool first = it == it0;
        if ((rc = launch_ref_stress(ga, md, shp, a, cur, it, true, first ? ImageRef{} : images(), W, kAdjoint,
                                    first ? 1 : 2, st)))
            return rc;
        const int slot = nt - it - 2;
        if ((rc = launch_ref_velocity(ga, md, shp, a, cur, nxt, it, res, borders, W, slot, fits ? 2 : 1, st)))
            return rc;
        if (!fits) {
            if ((rc = launch_velocity(gf, *m, shp, cur, nxt, it, st))) return rc;
            if ((rc = launch_border(gf, shp, nxt, const_cast<float *>(borders), W, slot, 0, -1, st))) return rc;
        }
        if (!fits || it < it0 + 2) {
            hipLaunchKernelGGL(k_zero_cpml, dim3(nblk(ga.N, 256), ga.S), dim3(256), 0, st, ga, nxt, W);
            if ((rc = check_launch("zero cpml"))) return rc;
        }
        std::swap(cur.v, nxt.v);
    }
    if (nsteps == 0) return EFM_OK;
    return launch_ref_stress(ga, md, shp, a, cur, it0 + nsteps, false, images(), W, kAdjoint, 2, st);
}

extern "C" int efm_backward_remake_ref(const EfmDims *d, const EfmMedium *m, const EfmShots *sh,
                                       const EfmState *fwd, float *vpres, const float *borders,
                                       int W, const EfmState *adj, const float *res, float dt,
                                       float dx, float dy, float dz, float *glam, float *gmu,
                                       float *grho, void *stream) {
    if (!d) return fail(EFM_E_ARG, "efm_backward_remake_ref: null dims");
    return backward_remake_ref(d, m, sh, fwd, vpres, borders, W, adj, res, dt, dx, dy, dz, glam, gmu,
                               grho, 0, d->ntmax - 1, stream, "efm_backward_remake_ref");
}

extern "C" int efm_backward_remake_ref_steps(const EfmDims *d, const EfmMedium *m, const EfmShots *sh,
                                             const EfmState *fwd, float *vpres, const float *borders,
                                             int W, const EfmState *adj, const float *res, float dt,
                                             float dx, float dy, float dz, float *glam, float *gmu,
                                             float *grho, int it0, int nsteps, void *stream) {
    return backward_remake_ref(d, m, sh, fwd, vpres, borders, W, adj, res, dt, dx, dy, dz, glam, gmu,
                               grho, it0, nsteps, stream, "efm_backward_remake_ref_steps");
}
