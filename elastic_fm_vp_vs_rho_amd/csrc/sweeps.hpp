// Cell updates of the forward sweeps, for the kernels of forward.hip and reference.hip.
//
// Reference: kernel_Tau (mainPropElastic3D_MT.py M:59-128), addSource
// (M:1728-1734), kernel_Vx_Vy_Vz (M:133-188).
//
// Addressing: per-shot base pointers are wave-uniform (scalar registers) and
// every per-lane offset is a 32-bit int, so loads use the base+offset form.
#pragma once
#include "common.hpp"

// For the sweeps' closures: one that stays a call keeps its captures in scratch memory.
#define EFM_INLINE __attribute__((always_inline))

namespace efm {

struct Med {
    const float *lam, *mu, *rho;
};

// What the stress sweep holds of a cell before it updates it: v, τ, the moduli and
// the reciprocals of μ at the corners of its shear planes.
struct CellOld {
    float vx, vy, vz, txx, tyy, tzz, txy, txz, tyz, lam, mu, r0, ri, rk, rj, rik, rjk, rij;
};

// Stress update of the column (x, z), rows y of chunk yb, of shot s.
// src_mode: 1 adds M·w[it] (forward), -1 subtracts M·w[nt-1-it] (reverse-time
// reconstruction, flagMode = 1 in M:1964), 0 injects nothing (adjoint runs).
// before(t, old) sees each cell before its update; without `write` that is all.
template <int NYC, typename F>
__device__ __forceinline__ void stress_cells(const Geo &g, const Med &m, const ShotPtrs &sh, const StatePtrs &in,
                                             const StatePtrs &out, int it, int src_mode, int x, int z, int s, int yb,
                                             bool write, F before) {
    const int y0 = H + yb * NYC;
    const int y1 = min(y0 + NYC, g.ny - H);
    const int nx = g.nx, sxz = g.sxz32;
    const long long so = (long long)s * g.N;
    const float c = g.c;

    const int sxs = slab_coord(x, g.nx, g.wxl, g.wxh);
    const int szs = slab_coord(z, g.nz, g.wzl, g.wzh);
    float ax = 0.f, bx = 0.f, az = 0.f, bz = 0.f;
    if (sxs >= 0) { ax = sh.ax[s * g.nx + x]; bx = sh.bx[s * g.nx + x]; }
    if (szs >= 0) { az = sh.az[s * g.nz + z]; bz = sh.bz[s * g.nz + z]; }
    const int *sp = sh.src + 3 * s;
    const bool src_col = (src_mode != 0) && (x == sp[0]) && (z == sp[2]);
    const int srcy = sp[1];

    const float *__restrict__ vx = in.v[0] + so;
    const float *__restrict__ vy = in.v[1] + so;
    const float *__restrict__ vz = in.v[2] + so;
    const float *__restrict__ mu = m.mu;
    const float *__restrict__ lam = m.lam;
    const float *pxi = in.px + px_shot(g, s), *pyi = in.py + py_shot(g, s), *pzi = in.pz + pz_shot(g, s);
    float *pxo = out.px + px_shot(g, s), *pyo = out.py + py_shot(g, s), *pzo = out.pz + pz_shot(g, s);
    // τ in/out may alias (in-place update): no restrict on them
    const float *ti0 = in.t[0] + so, *ti1 = in.t[1] + so, *ti2 = in.t[2] + so;
    const float *ti3 = in.t[3] + so, *ti4 = in.t[4] + so, *ti5 = in.t[5] + so;
    float *to0 = out.t[0] + so, *to1 = out.t[1] + so, *to2 = out.t[2] + so;
    float *to3 = out.t[3] + so, *to4 = out.t[4] + so, *to5 = out.t[5] + so;

    for (int y = y0; y < y1; ++y) {
        const int t = x + z * nx + y * sxz;
        const float vxc = vx[t], vyc = vy[t], vzc = vz[t];
        const float dvx_dx = vxc - vx[t - 1];
        const float dvy_dy = vyc - vy[t - sxz];
        const float dvz_dz = vzc - vz[t - nx];
        const float dvx_dz = vx[t + nx] - vxc;
        const float dvx_dy = vx[t + sxz] - vxc;
        const float dvy_dx = vy[t + 1] - vyc;
        const float dvy_dz = vy[t + nx] - vyc;
        const float dvz_dx = vz[t + 1] - vzc;
        const float dvz_dy = vz[t + sxz] - vzc;
        // strain-like terms e = Δ + ψ(new)   (ψ = b·ψ + a·Δ, updated then used)
        float exx = dvx_dx, eyx = dvy_dx, ezx = dvz_dx;
        float exy = dvx_dy, eyy = dvy_dy, ezy = dvz_dy;
        float exz = dvx_dz, eyz = dvy_dz, ezz = dvz_dz;
        if (sxs >= 0) {
            const int pi = px_off(g, y, z, sxs), cs = g.pxc;
            const float p0 = bx * pxi[pi] + ax * dvx_dx;
            const float p1 = bx * pxi[pi + cs] + ax * dvy_dx;
            const float p2 = bx * pxi[pi + 2 * cs] + ax * dvz_dx;
            if (write) { pxo[pi] = p0; pxo[pi + cs] = p1; pxo[pi + 2 * cs] = p2; }
            exx += p0; eyx += p1; ezx += p2;
        }
        const int sys = slab_coord(y, g.ny, g.wyl, g.wyh);
        if (sys >= 0) {
            const float ay = sh.ay[s * g.ny + y], by = sh.by[s * g.ny + y];
            const int pi = py_off(g, sys, z, x), cs = g.pyc;
            const float p0 = by * pyi[pi] + ay * dvx_dy;
            const float p1 = by * pyi[pi + cs] + ay * dvy_dy;
            const float p2 = by * pyi[pi + 2 * cs] + ay * dvz_dy;
            if (write) { pyo[pi] = p0; pyo[pi + cs] = p1; pyo[pi + 2 * cs] = p2; }
            exy += p0; eyy += p1; ezy += p2;
        }
        if (szs >= 0) {
            const int pi = pz_off(g, y, szs, x), cs = g.pzc;
            const float p0 = bz * pzi[pi] + az * dvx_dz;
            const float p1 = bz * pzi[pi + cs] + az * dvy_dz;
            const float p2 = bz * pzi[pi + 2 * cs] + az * dvz_dz;
            if (write) { pzo[pi] = p0; pzo[pi + cs] = p1; pzo[pi + 2 * cs] = p2; }
            exz += p0; eyz += p1; ezz += p2;
        }
        // moduli: λ, μ and the three 4-point harmonic means of μ (M:80-89)
        const float L = lam[t];
        const float Mu = mu[t];
        const float r0 = frcp(Mu);
        const float ri = frcp(mu[t + 1]);
        const float rk = frcp(mu[t + nx]);
        const float rj = frcp(mu[t + sxz]);
        const float rik = frcp(mu[t + 1 + nx]);
        const float rjk = frcp(mu[t + nx + sxz]);
        const float rij = frcp(mu[t + 1 + sxz]);
        const float mxz = 4.f * frcp(r0 + ri + rk + rik);
        const float mxy = 4.f * frcp(r0 + ri + rj + rij);
        const float myz = 4.f * frcp(r0 + rj + rk + rjk);
        const float l2m = L + 2.f * Mu;
        const float o0 = ti0[t], o1 = ti1[t], o2 = ti2[t], o3 = ti3[t], o4 = ti4[t], o5 = ti5[t];
        before(t, CellOld{vxc, vyc, vzc, o0, o1, o2, o3, o4, o5, L, Mu, r0, ri, rk, rj, rik, rjk, rij});
        float txx = o0 + c * (l2m * exx + L * (eyy + ezz));
        float tyy = o1 + c * (l2m * eyy + L * (exx + ezz));
        float tzz = o2 + c * (l2m * ezz + L * (exx + eyy));
        float txy = o3 + c * mxy * (exy + eyx);
        float txz = o4 + c * mxz * (exz + ezx);
        float tyz = o5 + c * myz * (eyz + ezy);
        if (src_col && y == srcy) {
            const int iw = src_mode > 0 ? it : sh.nt[s] - 1 - it;
            const float w0 = sh.wav[(long long)s * g.ntmax + iw];
            const float w = src_mode > 0 ? w0 : -w0;
            const float *m6 = sh.m6 + 6 * s;
            txx += m6[0] * w; tyy += m6[1] * w; tzz += m6[2] * w;
            txy += m6[3] * w; txz += m6[4] * w; tyz += m6[5] * w;
        }
        if (!write) continue;
        to0[t] = txx; to1[t] = tyy; to2[t] = tzz;
        to3[t] = txy; to4[t] = txz; to5[t] = tyz;
    }
}

// Velocity update of the column; change(y, t, vx, vy, vz) may change the values written,
// done(t, vx, vy, vz) sees them.
template <int NYC, typename F, typename G>
__device__ __forceinline__ void velocity_cells(const Geo &g, const Med &m, const ShotPtrs &sh, const StatePtrs &in,
                                               const StatePtrs &out, int x, int z, int s, int yb, F change,
                                               G done) {
    const int y0 = H + yb * NYC;
    const int y1 = min(y0 + NYC, g.ny - H);
    const int nx = g.nx, sxz = g.sxz32;
    const long long so = (long long)s * g.N;
    const float c = g.c;

    const int sxs = slab_coord(x, g.nx, g.wxl, g.wxh);
    const int szs = slab_coord(z, g.nz, g.wzl, g.wzh);
    float ax = 0.f, bx = 0.f, az = 0.f, bz = 0.f;
    if (sxs >= 0) { ax = sh.ax[s * g.nx + x]; bx = sh.bx[s * g.nx + x]; }
    if (szs >= 0) { az = sh.az[s * g.nz + z]; bz = sh.bz[s * g.nz + z]; }

    // τ is read from `out` (the stress sweep of this step wrote it there)
    const float *__restrict__ txx = out.t[0] + so;
    const float *__restrict__ tyy = out.t[1] + so;
    const float *__restrict__ tzz = out.t[2] + so;
    const float *__restrict__ txy = out.t[3] + so;
    const float *__restrict__ txz = out.t[4] + so;
    const float *__restrict__ tyz = out.t[5] + so;
    const float *__restrict__ rho = m.rho;
    const float *pxi = in.px + px_shot(g, s), *pyi = in.py + py_shot(g, s), *pzi = in.pz + pz_shot(g, s);
    float *pxo = out.px + px_shot(g, s), *pyo = out.py + py_shot(g, s), *pzo = out.pz + pz_shot(g, s);
    // v in/out may alias (in-place update)
    const float *vi0 = in.v[0] + so, *vi1 = in.v[1] + so, *vi2 = in.v[2] + so;
    float *vo0 = out.v[0] + so, *vo1 = out.v[1] + so, *vo2 = out.v[2] + so;

    for (int y = y0; y < y1; ++y) {
        const int t = x + z * nx + y * sxz;
        const float dtxx_dx = txx[t + 1] - txx[t];
        const float dtzz_dz = tzz[t + nx] - tzz[t];
        const float dtyy_dy = tyy[t + sxz] - tyy[t];
        const float txyc = txy[t], txzc = txz[t], tyzc = tyz[t];
        const float dtxy_dy = txyc - txy[t - sxz];
        const float dtxy_dx = txyc - txy[t - 1];
        const float dtxz_dz = txzc - txz[t - nx];
        const float dtxz_dx = txzc - txz[t - 1];
        const float dtyz_dz = tyzc - tyz[t - nx];
        const float dtyz_dy = tyzc - tyz[t - sxz];
        float fxx = dtxx_dx, fyx = dtxy_dx, fzx = dtxz_dx;
        float fxy = dtxy_dy, fyy = dtyy_dy, fzy = dtyz_dy;
        float fxz = dtxz_dz, fyz = dtyz_dz, fzz = dtzz_dz;
        if (sxs >= 0) {
            const int cs = g.pxc, pi = px_off(g, y, z, sxs) + 3 * cs;
            const float p0 = bx * pxi[pi] + ax * dtxx_dx;
            const float p1 = bx * pxi[pi + cs] + ax * dtxy_dx;
            const float p2 = bx * pxi[pi + 2 * cs] + ax * dtxz_dx;
            pxo[pi] = p0; pxo[pi + cs] = p1; pxo[pi + 2 * cs] = p2;
            fxx += p0; fyx += p1; fzx += p2;
        }
        const int sys = slab_coord(y, g.ny, g.wyl, g.wyh);
        if (sys >= 0) {
            const float ay = sh.ay[s * g.ny + y], by = sh.by[s * g.ny + y];
            const int cs = g.pyc, pi = py_off(g, sys, z, x) + 3 * cs;
            const float p0 = by * pyi[pi] + ay * dtxy_dy;
            const float p1 = by * pyi[pi + cs] + ay * dtyy_dy;
            const float p2 = by * pyi[pi + 2 * cs] + ay * dtyz_dy;
            pyo[pi] = p0; pyo[pi + cs] = p1; pyo[pi + 2 * cs] = p2;
            fxy += p0; fyy += p1; fzy += p2;
        }
        if (szs >= 0) {
            const int cs = g.pzc, pi = pz_off(g, y, szs, x) + 3 * cs;
            const float p0 = bz * pzi[pi] + az * dtxz_dz;
            const float p1 = bz * pzi[pi + cs] + az * dtyz_dz;
            const float p2 = bz * pzi[pi + 2 * cs] + az * dtzz_dz;
            pzo[pi] = p0; pzo[pi + cs] = p1; pzo[pi + 2 * cs] = p2;
            fxz += p0; fyz += p1; fzz += p2;
        }
        // averaged buoyancy b̄ = 2bb'/(b+b') = 2/(ρ+ρ')  (M:153-159)
        const float r = rho[t];
        const float bbx = 2.f * frcp(r + rho[t + 1]);
        const float bby = 2.f * frcp(r + rho[t + sxz]);
        const float bbz = 2.f * frcp(r + rho[t + nx]);
        float n0 = vi0[t] + c * bbx * (fxx + fxy + fxz);
        float n1 = vi1[t] + c * bby * (fyx + fyy + fyz);
        float n2 = vi2[t] + c * bbz * (fzx + fzy + fzz);
        change(y, t, n0, n1, n2);
        vo0[t] = n0;
        vo1[t] = n1;
        vo2[t] = n2;
        done(t, n0, n1, n2);
    }
}

// ---------------------------------------------------------------------------
// reference boundary save / restore of v (2 layers inside the CPML on x, y,
// bottom; z in [2,4) at the top)
// ---------------------------------------------------------------------------
struct BorderLayout {
    long long left, right, top, bottom, front, back, comp;  // offsets, comp = floats per component
};
__host__ __device__ inline BorderLayout border_layout(int nx, int ny, int nz) {
    BorderLayout b;
    const long long lr = (long long)ny * nz * H, tb = (long long)ny * H * nx, fb = (long long)H * nz * nx;
    b.left = 0; b.right = lr; b.top = 2 * lr; b.bottom = 2 * lr + tb; b.front = 2 * lr + 2 * tb;
    b.back = 2 * lr + 2 * tb + fb; b.comp = 2 * lr + 2 * tb + 2 * fb;
    return b;
}

// Element i of shot s's 3·comp border values of one step: its component, its place in
// the component and its cell.
struct BorderCell {
    int comp, x, y, z;
    long long e;
};
__device__ __forceinline__ BorderCell border_cell(const Geo &g, const BorderLayout &L, int W, long long i) {
    BorderCell c;
    c.comp = (int)(i / L.comp);
    c.e = i - c.comp * L.comp;
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    if (c.e < L.top) {                   // left / right: (ny, nz, H)
        const int side = c.e >= L.right;
        long long k = c.e - (side ? L.right : 0);
        const int h = (int)(k % H); k /= H;
        c.z = (int)(k % nz); c.y = (int)(k / nz);
        c.x = side ? nx - W - H + h : W + h;
    } else if (c.e < L.front) {          // top / bottom: (ny, H, nx)
        const int side = c.e >= L.bottom;
        long long k = c.e - (side ? L.bottom : L.top);
        c.x = (int)(k % nx); k /= nx;
        const int h = (int)(k % H); c.y = (int)(k / H);
        c.z = side ? nz - W - H + h : H + h;
    } else {                             // front / back: (H, nz, nx)
        const int side = c.e >= L.back;
        long long k = c.e - (side ? L.back : L.front);
        c.x = (int)(k % nx); k /= nx;
        c.z = (int)(k % nz); const int h = (int)(k / nz);
        c.y = side ? ny - W - H + h : W + h;
    }
    return c;
}

// Index of the calling block in launch order (the extra blocks some sweeps carry
// follow those of the sweep).
__device__ __forceinline__ long long block_number() {
    return blockIdx.x + (long long)gridDim.x * (blockIdx.y + (long long)gridDim.y * blockIdx.z);
}

// The sweep's grid with at least `extra` blocks behind it.
inline dim3 sweep_grid_plus(const Geo &g, const Tile &t, long long extra) {
    dim3 d = sweep_grid(g, t);
    if (t.map > 0) d.x += (unsigned)extra;
    else d.z += (unsigned)((extra + (long long)d.x * d.y - 1) / ((long long)d.x * d.y));
    return d;
}
inline long long grid_blocks(const dim3 &d) { return (long long)d.x * d.y * d.z; }

}  // namespace efm
