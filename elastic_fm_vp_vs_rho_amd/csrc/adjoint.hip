// Exact discrete adjoint of the forward recurrence in forward.hip, plus the
// model maps.  The reference has no exact adjoint (its backwardFields re-uses
// the forward operator, M:2056-2082); these kernels are the transpose of the
// two sweeps, derived by hand:
//
//   forward step n     τ' = τ + c·S(λ,μ)·e(v,ψv),  τ'' = τ' + M·w[n]δ_src,
//                      v' = v + c·B̄(ρ)·F(τ'',ψτ),  d[n] = R v'
//   ψ recurrences      ψ' = bψ + aΔ,  e = Δ + ψ'   (likewise for ψτ)
//
//   reverse step n     R1 v̄[rec] += r[n]
//                      R2 u = c·b̄·v̄;  h̄ = u + a(C+u);  C ← b(C+u);  τ̄ += D_τᵀ h̄
//                      R3 M̄ += w[n]·τ̄(src)
//                      R4 ē = c·Sᵀτ̄;  ḡ = ē + a(C+ē);  C ← b(C+ē);  v̄ += D_vᵀ ḡ
//   images             λ/μ sums += τ̄·(∂S/∂λ,μ)e (by R2, with the τ̄ it writes);
//                      ρ sums += v̄·(v^{n+1} - v^n) (= v̄·c·b̄·F; by R4, with the v̄ it reads)
//
// D_ᵀ are applied in gather form (each thread writes only its own cell), which
// needs h̄/ḡ at the ±1 neighbours; C is read at neighbours while its owner
// rewrites it, so C is ping-ponged between two buffers.  The derived medium
// (μ̄, b̄) is zero outside the interior and τ̄, v̄, C are only ever written on
// the interior, so neighbour terms vanish there without branches.
#include <mutex>
#include <string>
#include <utility>

#include "common.hpp"

namespace efm {

// Streaming (nontemporal) load of a stored forward value: the hint keeps the
// reused adjoint state, medium and accumulators cached.
#define LDF(p) __builtin_nontemporal_load(p)

struct AdjArgs {
    const float *lam, *mu;
    const float *mbar, *bbar;      // (3, N) each
    StatePtrs fn, fn1;             // forward S^n, S^{n+1}
    const float *vm1[3];           // forward velocities before step n - 1 (R4's two-step ρ sums)
    StatePtrs a, a2;               // adjoint: a = live (v̄, τ̄, C in), a2 = C out
    float *acc;                    // per shot 8 padded components: λ, μ, μ_xy, μ_xz sums
                                   // interleaved (one float4 per cell) in components 0-3, the
                                   // ρ sums of the x, y, z faces in 4-6, μ_yz in 7 (8 components
                                   // keep every shot's float4 base 16-byte aligned for any N)
    ShotPtrs sh;
    const float *resid;            // ∂J/∂gathers, used by R4 when the shots carry a receiver mask
    double *gm6;                   // ∂J/∂M, likewise
    int n0, n1;                    // step range of the call: n0 <= n < n1
};

// The reverse sweep images two steps at a time, so that the accumulators cross
// memory every other step: of each pair (n odd, n - 1) R2 of step n - 1 holds τ̄
// before and after its update and adds the λ/μ products of both steps, and R4 of
// step n holds v̄ before and after its update and adds the ρ products of both.  A
// step whose partner is outside the call's range or past the shot's record is
// imaged alone, by R2 with the new τ̄ and by R4 with the old v̄.
//   older: the products of step n + 1 (R2) / of step n (R4) from the value read
//   newer: the products of step n (R2) / of step n - 1 (R4) from the value written
struct Pairing {
    bool older, newer;
};
__device__ __forceinline__ Pairing image_r2(const AdjArgs &A, int nts, int n) {
    const int end = min(A.n1, nts);
    return n & 1 ? Pairing{false, n == A.n0} : Pairing{n + 1 < end, true};
}
__device__ __forceinline__ Pairing image_r4(const AdjArgs &A, int nts, int n) {
    const int end = min(A.n1, nts);
    // without a receiver mask the residual of step n - 1 joins v̄ in a kernel of its
    // own after this sweep: every step is imaged alone
    if (!A.sh.recmask) return Pairing{true, false};
    return n & 1 ? Pairing{true, n > A.n0} : Pairing{n + 1 >= end, false};
}

// The five λ/μ sums of a cell, fed by the adjoint stress τ̄ and the forward strain
// e = Δ + ψ' of a step (from the velocities and the ψ_v before the step).
struct ImageSums {
    float lam, mu, xy, xz, yz;
};
template <bool STREAM>
static __device__ __forceinline__ float ldf(const float *p) {
    return STREAM ? LDF(p) : *p;
}
struct StrainLoads {
    float v0, v1, v2, v0mx, v1my, v2mz, v0pz, v0py, v1px, v1pz, v2px, v2py;
    float fx0, fx1, fx2, fy0, fy1, fy2, fz0, fz1, fz2;
};
struct Slabs {
    int ix, iy, iz;                // own offsets of component 0 in the three slabs (-1 outside)
    float ax, bx, ay, by, az, bz;  // own coefficients (0 outside)
};
template <bool STREAM>
static __device__ __forceinline__ StrainLoads strain_loads(const Geo &g, const StatePtrs &f, int s, int t,
                                                           const Slabs &q) {
    const long long so = (long long)s * g.N;
    const float *__restrict__ V0 = f.v[0] + so, *__restrict__ V1 = f.v[1] + so, *__restrict__ V2 = f.v[2] + so;
    const int nx = g.nx, sxz = g.sxz32;
    StrainLoads l;
    l.v0 = ldf<STREAM>(&V0[t]); l.v1 = ldf<STREAM>(&V1[t]); l.v2 = ldf<STREAM>(&V2[t]);
    l.v0mx = ldf<STREAM>(&V0[t - 1]); l.v1my = ldf<STREAM>(&V1[t - sxz]); l.v2mz = ldf<STREAM>(&V2[t - nx]);
    l.v0pz = ldf<STREAM>(&V0[t + nx]); l.v0py = ldf<STREAM>(&V0[t + sxz]); l.v1px = ldf<STREAM>(&V1[t + 1]);
    l.v1pz = ldf<STREAM>(&V1[t + nx]); l.v2px = ldf<STREAM>(&V2[t + 1]); l.v2py = ldf<STREAM>(&V2[t + sxz]);
    l.fx0 = l.fx1 = l.fx2 = l.fy0 = l.fy1 = l.fy2 = l.fz0 = l.fz1 = l.fz2 = 0.f;
    if (q.ix >= 0) {
        const float *F = f.px + px_shot(g, s);
        l.fx0 = ldf<STREAM>(&F[q.ix]); l.fx1 = ldf<STREAM>(&F[q.ix + g.pxc]); l.fx2 = ldf<STREAM>(&F[q.ix + 2 * g.pxc]);
    }
    if (q.iy >= 0) {
        const float *F = f.py + py_shot(g, s);
        l.fy0 = ldf<STREAM>(&F[q.iy]); l.fy1 = ldf<STREAM>(&F[q.iy + g.pyc]); l.fy2 = ldf<STREAM>(&F[q.iy + 2 * g.pyc]);
    }
    if (q.iz >= 0) {
        const float *F = f.pz + pz_shot(g, s);
        l.fz0 = ldf<STREAM>(&F[q.iz]); l.fz1 = ldf<STREAM>(&F[q.iz + g.pzc]); l.fz2 = ldf<STREAM>(&F[q.iz + 2 * g.pzc]);
    }
    return l;
}
// a += the products of one step.  Every rounding is spelled out: a pair's two steps
// then give the same bits added in one sweep or in two.
static __device__ __forceinline__ void image_add(ImageSums &a, const StrainLoads &l, const Slabs &q, float txx,
                                                 float tyy, float tzz, float txy, float txz, float tyz) {
#pragma clang fp contract(off)
    const float d_xx = l.v0 - l.v0mx, d_yy = l.v1 - l.v1my, d_zz = l.v2 - l.v2mz;
    const float d_xz = l.v0pz - l.v0, d_xy = l.v0py - l.v0, d_yx = l.v1px - l.v1, d_yz = l.v1pz - l.v1;
    const float d_zx = l.v2px - l.v2, d_zy = l.v2py - l.v2;
    // e = Δ + (bψ + aΔ); a = b = 0 outside the slabs
    const float fxx = d_xx + fmaf(q.bx, l.fx0, q.ax * d_xx);
    const float fyx = d_yx + fmaf(q.bx, l.fx1, q.ax * d_yx);
    const float fzx = d_zx + fmaf(q.bx, l.fx2, q.ax * d_zx);
    const float fxy = d_xy + fmaf(q.by, l.fy0, q.ay * d_xy);
    const float fyy = d_yy + fmaf(q.by, l.fy1, q.ay * d_yy);
    const float fzy = d_zy + fmaf(q.by, l.fy2, q.ay * d_zy);
    const float fxz = d_xz + fmaf(q.bz, l.fz0, q.az * d_xz);
    const float fyz = d_yz + fmaf(q.bz, l.fz1, q.az * d_yz);
    const float fzz = d_zz + fmaf(q.bz, l.fz2, q.az * d_zz);
    a.lam = fmaf(txx + tyy + tzz, fxx + fyy + fzz, a.lam);
    a.mu = fmaf(2.f, fmaf(txx, fxx, fmaf(tyy, fyy, tzz * fzz)), a.mu);
    a.xy = fmaf(txy, fxy + fyx, a.xy);
    a.xz = fmaf(txz, fxz + fzx, a.xz);
    a.yz = fmaf(tyz, fyz + fzy, a.yz);
}

// ---------------------------------------------------------------------------
// R2: transpose of the velocity sweep, λ/μ imaging
// ---------------------------------------------------------------------------
template <int BX, int BZ, int NYC, int MAP, bool IMAGE, bool STREAM>
static __device__ __forceinline__ void adj_velocity_cells(const Geo &g, const AdjArgs &A, int n) {
    int x, z, s, yb;
    if (!tile_coords<BX, BZ, NYC, MAP>(g, x, z, s, yb)) return;
    if (x < H || x >= g.nx - H || z < H || z >= g.nz - H) return;
    const int nts = A.sh.nt[s];
    if (n >= nts) return;
    const Pairing im = image_r2(A, nts, n);
    const int y0 = H + yb * NYC;
    const int y1 = min(y0 + NYC, g.ny - H);
    const int nx = g.nx, sxz = g.sxz32;
    const long long so = (long long)s * g.N;
    const float c = g.c;
    const ShotPtrs &sh = A.sh;

    // slab coordinates of this column and its x/z neighbours
    const int sx0 = slab_coord(x, g.nx, g.wxl, g.wxh);
    const int sxm = slab_coord(x - 1, g.nx, g.wxl, g.wxh);
    const int sxp = slab_coord(x + 1, g.nx, g.wxl, g.wxh);
    const int sz0 = slab_coord(z, g.nz, g.wzl, g.wzh);
    const int szm = slab_coord(z - 1, g.nz, g.wzl, g.wzh);
    const int szp = slab_coord(z + 1, g.nz, g.wzl, g.wzh);
    const float *axs = sh.ax + (long long)s * g.nx, *bxs = sh.bx + (long long)s * g.nx;
    const float *ays = sh.ay + (long long)s * g.ny, *bys = sh.by + (long long)s * g.ny;
    const float *azs = sh.az + (long long)s * g.nz, *bzs = sh.bz + (long long)s * g.nz;
    const int csx = g.pxc, csy = g.pyc, csz = g.pzc;

    const float *__restrict__ bbx = A.bbar;
    const float *__restrict__ bby = A.bbar + g.ps;
    const float *__restrict__ bbz = A.bbar + 2 * g.ps;
    const float *__restrict__ vbx = A.a.v[0] + so;
    const float *__restrict__ vby = A.a.v[1] + so;
    const float *__restrict__ vbz = A.a.v[2] + so;
    float *__restrict__ tb0 = A.a.t[0] + so;
    float *__restrict__ tb1 = A.a.t[1] + so;
    float *__restrict__ tb2 = A.a.t[2] + so;
    float *__restrict__ tb3 = A.a.t[3] + so;
    float *__restrict__ tb4 = A.a.t[4] + so;
    float *__restrict__ tb5 = A.a.t[5] + so;
    const float *__restrict__ Cx = A.a.px + px_shot(g, s);
    const float *__restrict__ Cy = A.a.py + py_shot(g, s);
    const float *__restrict__ Cz = A.a.pz + pz_shot(g, s);
    float *__restrict__ Cxo = A.a2.px + px_shot(g, s);
    float *__restrict__ Cyo = A.a2.py + py_shot(g, s);
    float *__restrict__ Czo = A.a2.pz + pz_shot(g, s);
    float4 *__restrict__ acc4v = reinterpret_cast<float4 *>(A.acc + (long long)s * 8 * g.ps);
    float *__restrict__ accyz = A.acc + ((long long)s * 8 + 7) * g.ps;

    for (int y = y0; y < y1; ++y) {
        const int t = x + z * nx + y * sxz;
        const int sy0 = slab_coord(y, g.ny, g.wyl, g.wyh);
        const int sym = slab_coord(y - 1, g.ny, g.wyl, g.wyh);
        const int syp = slab_coord(y + 1, g.ny, g.wyl, g.wyh);

        // Every load of the cell is issued before the first use or store.  The slab
        // loads above all: a slab cell used to wait for each neighbour's ψ in turn.
        const float tbo0 = tb0[t], tbo1 = tb1[t], tbo2 = tb2[t];
        const float tbo3 = tb3[t], tbo4 = tb4[t], tbo5 = tb5[t];
        const float wx0 = vbx[t], wy0 = vby[t], wz0 = vbz[t];
        const float wx_mx = vbx[t - 1], wy_my = vby[t - sxz], wz_mz = vbz[t - nx];
        const float wx_py = vbx[t + sxz], wy_px = vby[t + 1], wx_pz = vbx[t + nx];
        const float wz_px = vbz[t + 1], wy_pz = vby[t + nx], wz_py = vbz[t + sxz];
        const float gx0 = bbx[t], gy0 = bby[t], gz0 = bbz[t];
        const float gx_mx = bbx[t - 1], gy_my = bby[t - sxz], gz_mz = bbz[t - nx];
        const float gx_py = bbx[t + sxz], gy_px = bby[t + 1], gx_pz = bbx[t + nx];
        const float gz_px = bbz[t + 1], gy_pz = bby[t + nx], gz_py = bbz[t + sxz];
        // x-slab components 3 txx_x, 4 txy_x, 5 txz_x; y: 3 txy_y, 4 tyy_y, 5 tyz_y;
        // z: 3 txz_z, 4 tyz_z, 5 tzz_z.  a = 0 outside the slab.
        Slabs q{-1, -1, -1, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        float axm = 0.f, axp = 0.f, aym = 0.f, ayp = 0.f, azm = 0.f, azp = 0.f;
        float cxm = 0.f, cxp1 = 0.f, cxp2 = 0.f, cx0 = 0.f, cx1 = 0.f, cx2 = 0.f;
        float cym = 0.f, cyp0 = 0.f, cyp2 = 0.f, cy0 = 0.f, cy1 = 0.f, cy2 = 0.f;
        float czm = 0.f, czp0 = 0.f, czp1 = 0.f, cz0 = 0.f, cz1 = 0.f, cz2 = 0.f;
        if (sxm >= 0) { axm = axs[x - 1]; cxm = Cx[px_off(g, y, z, sxm) + 3 * csx]; }
        if (sxp >= 0) {
            const int pi = px_off(g, y, z, sxp) + 4 * csx;
            axp = axs[x + 1]; cxp1 = Cx[pi]; cxp2 = Cx[pi + csx];
        }
        if (sx0 >= 0) {
            q.ix = px_off(g, y, z, sx0);
            q.ax = axs[x]; q.bx = bxs[x];
            cx0 = Cx[q.ix + 3 * csx]; cx1 = Cx[q.ix + 4 * csx]; cx2 = Cx[q.ix + 5 * csx];
        }
        if (sym >= 0) { aym = ays[y - 1]; cym = Cy[py_off(g, sym, z, x) + 4 * csy]; }
        if (syp >= 0) {
            const int pi = py_off(g, syp, z, x) + 3 * csy;
            ayp = ays[y + 1]; cyp0 = Cy[pi]; cyp2 = Cy[pi + 2 * csy];
        }
        if (sy0 >= 0) {
            q.iy = py_off(g, sy0, z, x);
            q.ay = ays[y]; q.by = bys[y];
            cy0 = Cy[q.iy + 3 * csy]; cy1 = Cy[q.iy + 4 * csy]; cy2 = Cy[q.iy + 5 * csy];
        }
        if (szm >= 0) { azm = azs[z - 1]; czm = Cz[pz_off(g, y, szm, x) + 5 * csz]; }
        if (szp >= 0) {
            const int pi = pz_off(g, y, szp, x) + 3 * csz;
            azp = azs[z + 1]; czp0 = Cz[pi]; czp1 = Cz[pi + csz];
        }
        if (sz0 >= 0) {
            q.iz = pz_off(g, y, sz0, x);
            q.az = azs[z]; q.bz = bzs[z];
            cz0 = Cz[q.iz + 3 * csz]; cz1 = Cz[q.iz + 4 * csz]; cz2 = Cz[q.iz + 5 * csz];
        }

        // u = c·b̄·v̄ at p and at the neighbours the transposes need (b̄ = 0 off the interior)
        const float ux = c * gx0 * wx0, uy = c * gy0 * wy0, uz = c * gz0 * wz0;
        const float ux_mx = c * gx_mx * wx_mx;        // txx_x at p-x
        const float uy_my = c * gy_my * wy_my;        // tyy_y at p-y
        const float uz_mz = c * gz_mz * wz_mz;        // tzz_z at p-z
        const float ux_py = c * gx_py * wx_py;        // txy_y at p+y
        const float uy_px = c * gy_px * wy_px;        // txy_x at p+x
        const float ux_pz = c * gx_pz * wx_pz;        // txz_z at p+z
        const float uz_px = c * gz_px * wz_px;        // txz_x at p+x
        const float uy_pz = c * gy_pz * wy_pz;        // tyz_z at p+z
        const float uz_py = c * gz_py * wz_py;        // tyz_y at p+y
        // h̄ = u + a(C + u) with C read from the "in" buffer
        cx0 += ux; cx1 += uy; cx2 += uz;
        cy0 += ux; cy1 += uy; cy2 += uz;
        cz0 += ux; cz1 += uy; cz2 += uz;
        const float hb_xx = (ux_mx + axm * (cxm + ux_mx)) - (ux + q.ax * cx0);
        const float hb_yy = (uy_my + aym * (cym + uy_my)) - (uy + q.ay * cy1);
        const float hb_zz = (uz_mz + azm * (czm + uz_mz)) - (uz + q.az * cz2);
        const float hb_xyy = (ux + q.ay * cy0) - (ux_py + ayp * (cyp0 + ux_py));
        const float hb_xyx = (uy + q.ax * cx1) - (uy_px + axp * (cxp1 + uy_px));
        const float hb_xzz = (ux + q.az * cz0) - (ux_pz + azp * (czp0 + ux_pz));
        const float hb_xzx = (uz + q.ax * cx2) - (uz_px + axp * (cxp2 + uz_px));
        const float hb_yzz = (uy + q.az * cz1) - (uy_pz + azp * (czp1 + uy_pz));
        const float hb_yzy = (uz + q.ay * cy2) - (uz_py + ayp * (cyp2 + uz_py));
        // τ̄ += D_τᵀ h̄
        const float n0 = tbo0 + hb_xx, n1 = tbo1 + hb_yy, n2 = tbo2 + hb_zz;
        const float n3 = tbo3 + (hb_xyy + hb_xyx);
        const float n4 = tbo4 + (hb_xzz + hb_xzx);
        const float n5 = tbo5 + (hb_yzz + hb_yzy);
        if (IMAGE && im.newer) {
            const float4 a = acc4v[t];
            ImageSums sum{a.x, a.y, a.z, a.w, accyz[t]};
            const StrainLoads l = strain_loads<STREAM>(g, A.fn, s, t, q);
            if (im.older) {
                const StrainLoads l1 = strain_loads<STREAM>(g, A.fn1, s, t, q);
                image_add(sum, l1, q, tbo0, tbo1, tbo2, tbo3, tbo4, tbo5);
            }
            image_add(sum, l, q, n0, n1, n2, n3, n4, n5);
            acc4v[t] = make_float4(sum.lam, sum.mu, sum.xy, sum.xz);
            accyz[t] = sum.yz;
        }
        tb0[t] = n0; tb1[t] = n1; tb2[t] = n2;
        tb3[t] = n3; tb4[t] = n4; tb5[t] = n5;
        if (sx0 >= 0) {
            const int pi = q.ix + 3 * csx;
            Cxo[pi] = q.bx * cx0; Cxo[pi + csx] = q.bx * cx1; Cxo[pi + 2 * csx] = q.bx * cx2;
        }
        if (sy0 >= 0) {
            const int pi = q.iy + 3 * csy;
            Cyo[pi] = q.by * cy0; Cyo[pi + csy] = q.by * cy1; Cyo[pi + 2 * csy] = q.by * cy2;
        }
        if (sz0 >= 0) {
            const int pi = q.iz + 3 * csz;
            Czo[pi] = q.bz * cz0; Czo[pi + csz] = q.bz * cz1; Czo[pi + 2 * csz] = q.bz * cz2;
        }
    }
}

// Three instances.  The steps that no shot images (one of every pair) run without
// the imaging's registers (78 VGPRs against 98): 28 against 65 us at 128^3, where one
// instance for both took 53 on average of either.  The imaging instances differ in
// the streaming hint on the forward state (see launch_adj_velocity).
template <int BX, int BZ, int NYC, int MAP>
__global__ EFM_KERNEL_ATTRS(BX, BZ, MAP) void k_adj_velocity(Geo g, AdjArgs A, int n) {
    adj_velocity_cells<BX, BZ, NYC, MAP, false, false>(g, A, n);
}
template <int BX, int BZ, int NYC, int MAP>
__global__ EFM_KERNEL_ATTRS(BX, BZ, MAP) void k_adj_velocity_image(Geo g, AdjArgs A, int n) {
    adj_velocity_cells<BX, BZ, NYC, MAP, true, false>(g, A, n);
}
template <int BX, int BZ, int NYC, int MAP>
__global__ EFM_KERNEL_ATTRS(BX, BZ, MAP) void k_adj_velocity_image_stream(Geo g, AdjArgs A, int n) {
    adj_velocity_cells<BX, BZ, NYC, MAP, true, true>(g, A, n);
}

// ---------------------------------------------------------------------------
// R4: transpose of the stress sweep, ρ imaging
// ---------------------------------------------------------------------------
template <int BX, int BZ, int NYC, int MAP>
__global__ EFM_KERNEL_ATTRS(BX, BZ, MAP) void k_adj_stress(Geo g, AdjArgs A, int n) {
    int x, z, s, yb;
    if (!tile_coords<BX, BZ, NYC, MAP>(g, x, z, s, yb)) return;
    if (x < H || x >= g.nx - H || z < H || z >= g.nz - H) return;
    const int nts = A.sh.nt[s];
    const int y0 = H + yb * NYC;
    const int y1 = min(y0 + NYC, g.ny - H);
    const int nx = g.nx, sxz = g.sxz32;
    const long long so = (long long)s * g.N;
    const float c = g.c;
    const ShotPtrs &sh = A.sh;
    // with a receiver mask this sweep also injects the residual of step n-1 (R1
    // of the next reverse step) and sums ∂J/∂M of step n (R3)
    const bool fused = sh.recmask != nullptr;
    if (n >= nts) {
        // the shot's record ends at step nts - 1: its first residual is injected here
        if (fused && n == nts && n >= 1 && g.nrec > 0)
            for (int y = y0; y < y1; ++y) {
                const int t = x + z * nx + y * sxz;
                float v0 = A.a.v[0][so + t], v1 = A.a.v[1][so + t], v2 = A.a.v[2][so + t];
                inject_wave(g, sh, s, t, A.resid, n - 1, v0, v1, v2);
                if (!is_receiver(g, sh, s, t)) continue;
                A.a.v[0][so + t] = v0;
                A.a.v[1][so + t] = v1;
                A.a.v[2][so + t] = v2;
            }
        return;
    }
    const Pairing im = image_r4(A, nts, n);
    const int *sp = sh.src + 3 * s;
    const int tsrc = sp[0] + sp[2] * nx + sp[1] * sxz;
    const bool inject = fused && n >= 1 && g.nrec > 0;

    const int sx0 = slab_coord(x, g.nx, g.wxl, g.wxh);
    const int sxm = slab_coord(x - 1, g.nx, g.wxl, g.wxh);
    const int sxp = slab_coord(x + 1, g.nx, g.wxl, g.wxh);
    const int sz0 = slab_coord(z, g.nz, g.wzl, g.wzh);
    const int szm = slab_coord(z - 1, g.nz, g.wzl, g.wzh);
    const int szp = slab_coord(z + 1, g.nz, g.wzl, g.wzh);
    const float *axs = sh.ax + (long long)s * g.nx, *bxs = sh.bx + (long long)s * g.nx;
    const float *ays = sh.ay + (long long)s * g.ny, *bys = sh.by + (long long)s * g.ny;
    const float *azs = sh.az + (long long)s * g.nz, *bzs = sh.bz + (long long)s * g.nz;
    const int csx = g.pxc, csy = g.pyc, csz = g.pzc;

    const float *__restrict__ mxy = A.mbar;
    const float *__restrict__ mxz = A.mbar + g.ps;
    const float *__restrict__ myz = A.mbar + 2 * g.ps;
    const float *__restrict__ lam = A.lam;
    const float *__restrict__ mu = A.mu;
    const float *__restrict__ Txx = A.a.t[0] + so;
    const float *__restrict__ Tyy = A.a.t[1] + so;
    const float *__restrict__ Tzz = A.a.t[2] + so;
    const float *__restrict__ Txy = A.a.t[3] + so;
    const float *__restrict__ Txz = A.a.t[4] + so;
    const float *__restrict__ Tyz = A.a.t[5] + so;
    float *__restrict__ vb0 = A.a.v[0] + so;
    float *__restrict__ vb1 = A.a.v[1] + so;
    float *__restrict__ vb2 = A.a.v[2] + so;
    const float *__restrict__ Cx = A.a.px + px_shot(g, s);
    const float *__restrict__ Cy = A.a.py + py_shot(g, s);
    const float *__restrict__ Cz = A.a.pz + pz_shot(g, s);
    float *__restrict__ Cxo = A.a2.px + px_shot(g, s);
    float *__restrict__ Cyo = A.a2.py + py_shot(g, s);
    float *__restrict__ Czo = A.a2.pz + pz_shot(g, s);
    float *__restrict__ accr = A.acc + ((long long)s * 8 + 4) * g.ps;

    for (int y = y0; y < y1; ++y) {
        const int t = x + z * nx + y * sxz;
        const int sy0 = slab_coord(y, g.ny, g.wyl, g.wyh);
        const int sym = slab_coord(y - 1, g.ny, g.wyl, g.wyh);
        const int syp = slab_coord(y + 1, g.ny, g.wyl, g.wyh);

        const float txx = Txx[t], tyy = Tyy[t], tzz = Tzz[t];
        const float txy = Txy[t], txz = Txz[t], tyz = Tyz[t];
        const float L0 = lam[t], M0 = mu[t];
        const float kxy = mxy[t], kxz = mxz[t], kyz = myz[t];
        const float vo0 = vb0[t], vo1 = vb1[t], vo2 = vb2[t];
        // x-slab components 0 vx_x, 1 vy_x, 2 vz_x; y: 0 vx_y, 1 vy_y, 2 vz_y;
        // z: 0 vx_z, 1 vy_z, 2 vz_z.  a = 0 outside the slab; all loads before the first use.
        float ax0 = 0.f, bx0 = 0.f, ay0 = 0.f, by0 = 0.f, az0 = 0.f, bz0 = 0.f;
        float axm = 0.f, axp = 0.f, aym = 0.f, ayp = 0.f, azm = 0.f, azp = 0.f;
        float cxp = 0.f, cxm1 = 0.f, cxm2 = 0.f, cx0 = 0.f, cx1 = 0.f, cx2 = 0.f;
        float cyp = 0.f, cym0 = 0.f, cym2 = 0.f, cy0 = 0.f, cy1 = 0.f, cy2 = 0.f;
        float czp = 0.f, czm0 = 0.f, czm1 = 0.f, cz0 = 0.f, cz1 = 0.f, cz2 = 0.f;
        if (sxp >= 0) { axp = axs[x + 1]; cxp = Cx[px_off(g, y, z, sxp)]; }
        if (sxm >= 0) {
            const int pi = px_off(g, y, z, sxm) + csx;
            axm = axs[x - 1]; cxm1 = Cx[pi]; cxm2 = Cx[pi + csx];
        }
        if (sx0 >= 0) {
            const int pi = px_off(g, y, z, sx0);
            ax0 = axs[x]; bx0 = bxs[x];
            cx0 = Cx[pi]; cx1 = Cx[pi + csx]; cx2 = Cx[pi + 2 * csx];
        }
        if (syp >= 0) { ayp = ays[y + 1]; cyp = Cy[py_off(g, syp, z, x) + csy]; }
        if (sym >= 0) {
            const int pi = py_off(g, sym, z, x);
            aym = ays[y - 1]; cym0 = Cy[pi]; cym2 = Cy[pi + 2 * csy];
        }
        if (sy0 >= 0) {
            const int pi = py_off(g, sy0, z, x);
            ay0 = ays[y]; by0 = bys[y];
            cy0 = Cy[pi]; cy1 = Cy[pi + csy]; cy2 = Cy[pi + 2 * csy];
        }
        if (szp >= 0) { azp = azs[z + 1]; czp = Cz[pz_off(g, y, szp, x) + 2 * csz]; }
        if (szm >= 0) {
            const int pi = pz_off(g, y, szm, x);
            azm = azs[z - 1]; czm0 = Cz[pi]; czm1 = Cz[pi + csz];
        }
        if (sz0 >= 0) {
            const int pi = pz_off(g, y, sz0, x);
            az0 = azs[z]; bz0 = bzs[z];
            cz0 = Cz[pi]; cz1 = Cz[pi + csz]; cz2 = Cz[pi + 2 * csz];
        }
        // ē at the neighbours
        float exx_px, eyy_py, ezz_pz;
        {
            const int o = t + 1;
            const float L = lam[o], M = mu[o];
            exx_px = c * ((L + 2.f * M) * Txx[o] + L * (Tyy[o] + Tzz[o]));   // vx_x at p+x
        }
        {
            const int o = t + sxz;
            const float L = lam[o], M = mu[o];
            eyy_py = c * ((L + 2.f * M) * Tyy[o] + L * (Txx[o] + Tzz[o]));   // vy_y at p+y
        }
        {
            const int o = t + nx;
            const float L = lam[o], M = mu[o];
            ezz_pz = c * ((L + 2.f * M) * Tzz[o] + L * (Txx[o] + Tyy[o]));   // vz_z at p+z
        }
        const float exz_mz = c * mxz[t - nx] * Txz[t - nx];     // vx_z at p-z
        const float exy_my = c * mxy[t - sxz] * Txy[t - sxz];   // vx_y at p-y
        const float exy_mx = c * mxy[t - 1] * Txy[t - 1];       // vy_x at p-x
        const float eyz_mz = c * myz[t - nx] * Tyz[t - nx];     // vy_z at p-z
        const float exz_mx = c * mxz[t - 1] * Txz[t - 1];       // vz_x at p-x
        const float eyz_my = c * myz[t - sxz] * Tyz[t - sxz];   // vz_y at p-y
        // ē at p
        const float e_xx = c * ((L0 + 2.f * M0) * txx + L0 * (tyy + tzz));
        const float e_yy = c * ((L0 + 2.f * M0) * tyy + L0 * (txx + tzz));
        const float e_zz = c * ((L0 + 2.f * M0) * tzz + L0 * (txx + tyy));
        const float e_xy = c * kxy * txy;
        const float e_xz = c * kxz * txz;
        const float e_yz = c * kyz * tyz;
        // ḡ = ē + a(C + ē)
        cx0 += e_xx; cx1 += e_xy; cx2 += e_xz;
        cy0 += e_xy; cy1 += e_yy; cy2 += e_yz;
        cz0 += e_xz; cz1 += e_yz; cz2 += e_zz;
        const float g_vxx = (e_xx + ax0 * cx0) - (exx_px + axp * (cxp + exx_px));
        const float g_vyy = (e_yy + ay0 * cy1) - (eyy_py + ayp * (cyp + eyy_py));
        const float g_vzz = (e_zz + az0 * cz2) - (ezz_pz + azp * (czp + ezz_pz));
        const float g_vxz = (exz_mz + azm * (czm0 + exz_mz)) - (e_xz + az0 * cz0);
        const float g_vxy = (exy_my + aym * (cym0 + exy_my)) - (e_xy + ay0 * cy0);
        const float g_vyx = (exy_mx + axm * (cxm1 + exy_mx)) - (e_xy + ax0 * cx1);
        const float g_vyz = (eyz_mz + azm * (czm1 + eyz_mz)) - (e_yz + az0 * cz1);
        const float g_vzx = (exz_mx + axm * (cxm2 + exz_mx)) - (e_xz + ax0 * cx2);
        const float g_vzy = (eyz_my + aym * (cym2 + eyz_my)) - (e_yz + ay0 * cy2);
        // v̄ += D_vᵀ ḡ
        float nv0 = vo0 + (g_vxx + g_vxz + g_vxy);
        float nv1 = vo1 + (g_vyy + g_vyx + g_vyz);
        float nv2 = vo2 + (g_vzz + g_vzx + g_vzy);
        // R1 of step n-1 at this cell's receivers
        if (inject) inject_wave(g, sh, s, t, A.resid, n - 1, nv0, nv1, nv2);
        if (im.older) {
            // ρ: each of the cell's own faces sums v̄·Δv over the steps (k_combine puts in
            // c·b̄ and gathers the six faces of a cell)
            float a0 = accr[t], a1 = accr[t + g.ps], a2 = accr[t + 2 * g.ps];
            const float q0 = LDF(&A.fn.v[0][so + t]), q1 = LDF(&A.fn.v[1][so + t]), q2 = LDF(&A.fn.v[2][so + t]);
            a0 = fmaf(vo0, LDF(&A.fn1.v[0][so + t]) - q0, a0);
            a1 = fmaf(vo1, LDF(&A.fn1.v[1][so + t]) - q1, a1);
            a2 = fmaf(vo2, LDF(&A.fn1.v[2][so + t]) - q2, a2);
            if (im.newer) {
                a0 = fmaf(nv0, q0 - LDF(&A.vm1[0][so + t]), a0);
                a1 = fmaf(nv1, q1 - LDF(&A.vm1[1][so + t]), a1);
                a2 = fmaf(nv2, q2 - LDF(&A.vm1[2][so + t]), a2);
            }
            accr[t] = a0;
            accr[t + g.ps] = a1;
            accr[t + 2 * g.ps] = a2;
        }
        vb0[t] = nv0;
        vb1[t] = nv1;
        vb2[t] = nv2;
        if (sx0 >= 0) {
            const int pi = px_off(g, y, z, sx0);
            Cxo[pi] = bx0 * cx0; Cxo[pi + csx] = bx0 * cx1; Cxo[pi + 2 * csx] = bx0 * cx2;
        }
        if (sy0 >= 0) {
            const int pi = py_off(g, sy0, z, x);
            Cyo[pi] = by0 * cy0; Cyo[pi + csy] = by0 * cy1; Cyo[pi + 2 * csy] = by0 * cy2;
        }
        if (sz0 >= 0) {
            const int pi = pz_off(g, y, sz0, x);
            Czo[pi] = bz0 * cz0; Czo[pi + csz] = bz0 * cz1; Czo[pi + 2 * csz] = bz0 * cz2;
        }
        if (fused && t == tsrc) {                       // R3 of step n: ∂J/∂M += w[n]·τ̄(src)
            const double w = sh.wav[(long long)s * g.ntmax + n];
            double *gm = A.gm6 + 6 * s;
            gm[0] += w * (double)txx; gm[1] += w * (double)tyy; gm[2] += w * (double)tzz;
            gm[3] += w * (double)txy; gm[4] += w * (double)txz; gm[5] += w * (double)tyz;
        }
    }
}

// ---------------------------------------------------------------------------
// R1 + R3 (one block per shot): moment-tensor sum of step n+1, residual of step n
// ---------------------------------------------------------------------------
__global__ void k_adj_points(Geo g, ShotPtrs sh, StatePtrs a, const float *resid, double *gm6,
                             int n, int n_m) {
    const int s = g.s0 + blockIdx.x;
    const int nts = sh.nt[s];
    if (threadIdx.x == 0 && n_m >= 0 && n_m < nts) {
        const int *sp = sh.src + 3 * s;
        const long long t = (long long)s * g.N + sp[0] + (long long)sp[2] * g.nx + (long long)sp[1] * g.sxz;
        const double w = sh.wav[(long long)s * g.ntmax + n_m];
        for (int k = 0; k < 6; ++k) gm6[6 * s + k] += w * (double)a.t[k][t];
    }
    if (n < 0 || n >= nts) return;
    for (int r = threadIdx.x; r < g.nrec; r += blockDim.x) {
        const int cell = sh.rec[(long long)s * g.nrec + r];
        if (cell < 0) continue;
        const long long t = (long long)s * g.N + cell;
        const long long base = ((long long)s * 3 * g.ntmax + n) * g.nrec + r;
        const long long cs = (long long)g.ntmax * g.nrec;
        atomicAdd(&a.v[0][t], resid[base]);
        atomicAdd(&a.v[1][t], resid[base + cs]);
        atomicAdd(&a.v[2][t], resid[base + 2 * cs]);
    }
}

// ---------------------------------------------------------------------------
// derived medium, gradient combine, model maps
// ---------------------------------------------------------------------------
__global__ void k_derived(Geo g, const float *mu, const float *rho, float *mbar, float *bbar) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= g.N) return;
    const int x = (int)(i % g.nx);
    const int z = (int)((i / g.nx) % g.nz);
    const int y = (int)(i / g.sxz);
    float mxy = 0.f, mxz = 0.f, myz = 0.f, bx = 0.f, by = 0.f, bz = 0.f;
    if (interior(x, y, z, g)) {
        const long long nx = g.nx, sxz = g.sxz;
        // the forward sweeps' own operations (forward.hip), so that the adjoint
        // is the transpose of the forward operator as implemented
        const float q0 = frcp(mu[i]), qi = frcp(mu[i + 1]), qk = frcp(mu[i + nx]);
        const float qj = frcp(mu[i + sxz]), qik = frcp(mu[i + 1 + nx]);
        const float qjk = frcp(mu[i + nx + sxz]), qij = frcp(mu[i + 1 + sxz]);
        mxz = 4.f * frcp(q0 + qi + qk + qik);
        mxy = 4.f * frcp(q0 + qi + qj + qij);
        myz = 4.f * frcp(q0 + qj + qk + qjk);
        const float r = rho[i];
        bx = 2.f * frcp(r + rho[i + 1]);
        by = 2.f * frcp(r + rho[i + sxz]);
        bz = 2.f * frcp(r + rho[i + nx]);
    }
    mbar[i] = mxy; mbar[i + g.ps] = mxz; mbar[i + 2 * g.ps] = myz;
    bbar[i] = bx; bbar[i + g.ps] = by; bbar[i + 2 * g.ps] = bz;
}

__global__ void k_combine(Geo g, const float *mu, const float *mbar, const float *bbar,
                          const float *acc, float *glam, float *gmu, float *grho) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= g.N) return;
    const int x = (int)(i % g.nx);
    const int z = (int)((i / g.nx) % g.nz);
    const int y = (int)(i / g.sxz);
    const long long N = g.ps, nx = g.nx, sxz = g.sxz;   // N: padded component stride
    const float c = g.c;
    const float *mxy = mbar, *mxz = mbar + N, *myz = mbar + 2 * N;
    const float *bx = bbar, *by = bbar + N, *bz = bbar + 2 * N;
    float sl = 0.f, sm = 0.f, shear = 0.f, sr = 0.f;
    for (int s = 0; s < g.S; ++s) {
        const float *A = acc + (long long)s * 8 * N;
        // component k of cell j: 0-3 interleaved at the base, 4 (μ_yz) at 7·N; the ρ sums
        // of the x, y, z faces at 4·N, 5·N, 6·N
        auto AC = [&](int k, long long j) -> float { return k < 4 ? A[4 * j + k] : A[7 * N + j]; };
        sl += AC(0, i);
        sm += AC(1, i);
        auto sh4 = [&](int comp, const float *mb, long long o1, bool v1, long long o2, bool v2) {
            float r = AC(comp, i) * mb[i] * mb[i];
            if (v1) r += AC(comp, i - o1) * mb[i - o1] * mb[i - o1];
            if (v2) r += AC(comp, i - o2) * mb[i - o2] * mb[i - o2];
            if (v1 && v2) r += AC(comp, i - o1 - o2) * mb[i - o1 - o2] * mb[i - o1 - o2];
            return r;
        };
        shear += sh4(2, mxy, 1, x > 0, sxz, y > 0);
        shear += sh4(3, mxz, 1, x > 0, nx, z > 0);
        shear += sh4(4, myz, sxz, y > 0, nx, z > 0);
        // a face's sum is Σ v̄·Δv (Δv = c·b̄·F); per face of the cell
        // ∂J/∂ρ = -(c/2)·b̄²·v̄·F = -½·b̄·(v̄·Δv)
        const float *R = A + 4 * N;
        sr += bx[i] * R[i] + by[i] * R[N + i] + bz[i] * R[2 * N + i];
        if (x > 0) sr += bx[i - 1] * R[i - 1];
        if (y > 0) sr += by[i - sxz] * R[N + i - sxz];
        if (z > 0) sr += bz[i - nx] * R[2 * N + i - nx];
    }
    const float m = mu[i];
    glam[i] = c * sl;
    gmu[i] = c * (sm + (m != 0.f ? 0.25f * shear / (m * m) : 0.f));
    grho[i] = -0.5f * sr;
}

// r = mod - obs and J += ½Σr² (block partial sums in double, one atomic per block)
__global__ void k_residual(const float *mod, const float *obs, float *res, double *J, long long n) {
    __shared__ double part[256];
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (i < n) {
        const float r = mod[i] - obs[i];
        res[i] = r;
        v = 0.5 * (double)r * (double)r;
    }
    part[threadIdx.x] = v;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(J, part[0]);
}

__global__ void k_lame(const float *vp, const float *vs, const float *rho, float *lam, float *mu,
                       long long n) {
#pragma clang fp contract(off)
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float m = vs[i] * vs[i] * rho[i];
    mu[i] = m;
    lam[i] = vp[i] * vp[i] * rho[i] - 2.0f * m;
}

__global__ void k_lame_adjoint(const float *vp, const float *vs, const float *rho,
                               const float *glam, const float *gmu, const float *grho_in,
                               float *gvp, float *gvs, float *grho_out, long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float p = vp[i], s = vs[i], r = rho[i], gl = glam[i], gm = gmu[i];
    gvp[i] = 2.f * r * p * gl;
    gvs[i] = 2.f * r * s * (gm - 2.f * gl);
    grho_out[i] = (p * p - 2.f * s * s) * gl + s * s * gm + (grho_in ? grho_in[i] : 0.f);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
int launch_adj_velocity(const Geo &g, const AdjArgs &A, int n, hipStream_t st) {
    const Tile t = get_tile(2);
    bool launched = false;
#define X_PLAIN(a, b, c, o) EFM_LAUNCH_IF(a, b, c, o, k_adj_velocity, g, A, n)
#define X_IMAGE(a, b, c, o) EFM_LAUNCH_IF(a, b, c, o, k_adj_velocity_image, g, A, n)
#define X_STREAM(a, b, c, o) EFM_LAUNCH_IF(a, b, c, o, k_adj_velocity_image_stream, g, A, n)
    const bool stream = stream_forward_state(g);
    if (n % 2 && n != A.n0) {          // image_r2 images nothing in this step
        EFM_TILE_LIST(X_PLAIN)
    } else if (stream) {
        EFM_TILE_LIST(X_STREAM)
    } else {
        EFM_TILE_LIST(X_IMAGE)
    }
#undef X_PLAIN
#undef X_IMAGE
#undef X_STREAM
    if (!launched) return fail(EFM_E_UNSUPPORTED, "unsupported adjoint-velocity tile");
    return check_launch("adjoint velocity sweep");
}

int launch_adj_stress(const Geo &g, const AdjArgs &A, int n, hipStream_t st) {
    const Tile t = get_tile(3);
    bool launched = false;
#define X(a, b, c, o) EFM_LAUNCH_IF(a, b, c, o, k_adj_stress, g, A, n)
    EFM_TILE_LIST(X)
#undef X
    if (!launched) return fail(EFM_E_UNSUPPORTED, "unsupported adjoint-stress tile");
    return check_launch("adjoint stress sweep");
}

}  // namespace efm

using namespace efm;

static inline unsigned blocks_for(long long n, int b) { return (unsigned)((n + b - 1) / b); }

extern "C" int efm_derived_medium(const EfmDims *d, const EfmMedium *m, float *mbar, float *bbar,
                                  void *stream) {
    if (!d || !m || !mbar || !bbar || !m->mu || !m->rho)
        return fail(EFM_E_ARG, "efm_derived_medium: null argument");
    if (int rc = check_dims(d)) return rc;
    const Geo g = make_geo(*d);
    hipLaunchKernelGGL(k_derived, dim3(blocks_for(g.N, 256)), dim3(256), 0, (hipStream_t)stream, g,
                       m->mu, m->rho, mbar, bbar);
    return check_launch("derived medium");
}

namespace efm {

// The reverse sweep of steps n1-1 .. n0 (the body of efm_adjoint, shared with
// efm_gradient_static).  `copy_back` leaves the live ψ adjoint in adj's
// buffers when the ping-pong ended in adj2's.
static int run_adjoint(const EfmDims *d, const Geo &g, AdjArgs A, const EfmState *const *fwd,
                       const EfmState *adj, const EfmState *adj2, int n0, int n1, int last,
                       bool copy_back, hipStream_t st) {
    StatePtrs live = make_state(*adj), other = make_state(*adj2);
    const float *resid = A.resid;
    double *gm6 = A.gm6;
    const bool fused = A.sh.recmask != nullptr;
    if (fused && n1 == d->ntmax) {
        // first residual injection of the run; the sweeps do the rest
        hipLaunchKernelGGL(k_adj_points, dim3(g.S), dim3(64), 0, st, g, A.sh, live, resid, gm6,
                           n1 - 1, -1);
        int rc = check_launch("adjoint points");
        if (rc) return rc;
    }
    for (int n = n1 - 1; n >= n0; --n) {
        int rc = EFM_OK;
        if (!fused) {
            hipLaunchKernelGGL(k_adj_points, dim3(g.S), dim3(64), 0, st, g, A.sh, live, resid, gm6,
                               n, n + 1 < d->ntmax ? n + 1 : -1);
            if ((rc = check_launch("adjoint points"))) return rc;
        }
        A.fn = make_state(*fwd[n - n0]);
        A.fn1 = make_state(*fwd[n - n0 + 1]);
        const StatePtrs fm1 = make_state(*fwd[n > n0 ? n - n0 - 1 : 0]);
        for (int k = 0; k < 3; ++k) A.vm1[k] = fm1.v[k];
        A.a = live;
        A.a2 = other;
        A.a2.v[0] = live.v[0]; A.a2.v[1] = live.v[1]; A.a2.v[2] = live.v[2];
        for (int k = 0; k < 6; ++k) A.a2.t[k] = live.t[k];
        if ((rc = launch_adj_velocity(g, A, n, st))) return rc;
        // R4 reads the τ̄-side C from `other` (just written) and its own v̄-side C from `live`:
        // the two sweeps touch disjoint ψ components, so swap only after both.
        if ((rc = launch_adj_stress(g, A, n, st))) return rc;
        std::swap(live.px, other.px); std::swap(live.py, other.py); std::swap(live.pz, other.pz);
    }
    if (!fused && last && n0 == 0) {
        hipLaunchKernelGGL(k_adj_points, dim3(g.S), dim3(64), 0, st, g, A.sh, live, resid, gm6, -1, 0);
        int rc = check_launch("adjoint points");
        if (rc) return rc;
    }
    // leave the live ψ adjoint in adj's buffers (copy back when they were swapped)
    if (copy_back && live.px != adj->psi_x) {
        const long long fx = (long long)g.S * 6 * g.ny * g.nz * g.Lx;
        const long long fy = (long long)g.S * 6 * g.Ly * g.nz * g.nx;
        const long long fz = (long long)g.S * 6 * g.ny * g.Lz * g.nx;
        if (fx && hipMemcpyAsync(adj->psi_x, live.px, fx * 4, hipMemcpyDeviceToDevice, st))
            return fail(EFM_E_HIP, "efm_adjoint: psi copy");
        if (fy && hipMemcpyAsync(adj->psi_y, live.py, fy * 4, hipMemcpyDeviceToDevice, st))
            return fail(EFM_E_HIP, "efm_adjoint: psi copy");
        if (fz && hipMemcpyAsync(adj->psi_z, live.pz, fz * 4, hipMemcpyDeviceToDevice, st))
            return fail(EFM_E_HIP, "efm_adjoint: psi copy");
    }
    return EFM_OK;
}

}  // namespace efm

extern "C" int efm_adjoint(const EfmDims *d, const EfmMedium *m, const float *mbar,
                           const float *bbar, const EfmShots *sh, const EfmState *const *fwd,
                           const EfmState *adj, const EfmState *adj2, const float *resid,
                           float *acc, double *gm6, int n0, int n1, int last, void *stream) {
    if (!d || !m || !mbar || !bbar || !sh || !fwd || !adj || !adj2 || (!resid && d->nrec > 0) ||
        !acc || !gm6)
        return fail(EFM_E_ARG, "efm_adjoint: null argument");
    if (int rc = validate(d, m, sh)) return rc;
    if (n0 < 0 || n1 <= n0 || n1 > d->ntmax) return fail(EFM_E_ARG, "efm_adjoint: bad step range");
    if (int rc = validate_state(d, adj)) return rc;
    // adj2 carries only the second ψ buffer
    if ((d->wx_lo + d->wx_hi > 0 && !adj2->psi_x) || (d->wy_lo + d->wy_hi > 0 && !adj2->psi_y) ||
        (d->wz_lo + d->wz_hi > 0 && !adj2->psi_z))
        return fail(EFM_E_ARG, "efm_adjoint: adj2 psi slab pointer is null");
    for (int k = 0; k <= n1 - n0; ++k)
        if (int rc = validate_state(d, fwd[k])) return rc;
    const Geo g = make_geo(*d);
    AdjArgs A;
    A.lam = m->lam; A.mu = m->mu; A.mbar = mbar; A.bbar = bbar; A.acc = acc;
    A.sh = make_shots(*sh);
    A.resid = resid;
    A.gm6 = gm6;
    A.n0 = n0;
    A.n1 = n1;
    return run_adjoint(d, g, A, fwd, adj, adj2, n0, n1, last, true, (hipStream_t)stream);
}

extern "C" int efm_gradient_combine(const EfmDims *d, const EfmMedium *m, const float *mbar,
                                    const float *bbar, const float *acc, float *glam, float *gmu,
                                    float *grho, void *stream) {
    if (!d || !m || !m->mu || !mbar || !bbar || !acc || !glam || !gmu || !grho)
        return fail(EFM_E_ARG, "efm_gradient_combine: null argument");
    if (int rc = check_dims(d)) return rc;
    const Geo g = make_geo(*d);
    hipLaunchKernelGGL(k_combine, dim3(blocks_for(g.N, 256)), dim3(256), 0, (hipStream_t)stream, g,
                       m->mu, mbar, bbar, acc, glam, gmu, grho);
    return check_launch("gradient combine");
}

extern "C" int efm_residual(const float *mod, const float *obs, float *res, double *J, long long n,
                            void *stream) {
    if (n == 0) return EFM_OK;                   // no receivers: nothing to compare
    if (!mod || !obs || !res || !J || n < 0) return fail(EFM_E_ARG, "efm_residual: bad argument");
    hipLaunchKernelGGL(k_residual, dim3(blocks_for(n, 256)), dim3(256), 0, (hipStream_t)stream, mod,
                       obs, res, J, n);
    return check_launch("residual");
}

extern "C" int efm_model_lame(const float *vp, const float *vs, const float *rho, float *lam,
                              float *mu, long long n, void *stream) {
    if (!vp || !vs || !rho || !lam || !mu || n < 0) return fail(EFM_E_ARG, "efm_model_lame: bad argument");
    if (n == 0) return EFM_OK;
    hipLaunchKernelGGL(k_lame, dim3(blocks_for(n, 256)), dim3(256), 0, (hipStream_t)stream, vp, vs,
                       rho, lam, mu, n);
    return check_launch("model lame");
}

extern "C" int efm_model_lame_adjoint(const float *vp, const float *vs, const float *rho,
                                      const float *glam, const float *gmu, const float *grho_in,
                                      float *gvp, float *gvs, float *grho_out, long long n,
                                      void *stream) {
    if (!vp || !vs || !rho || !glam || !gmu || !gvp || !gvs || !grho_out || n < 0)
        return fail(EFM_E_ARG, "efm_model_lame_adjoint: bad argument");
    if (n == 0) return EFM_OK;
    hipLaunchKernelGGL(k_lame_adjoint, dim3(blocks_for(n, 256)), dim3(256), 0, (hipStream_t)stream,
                       vp, vs, rho, glam, gmu, grho_in, gvp, gvs, grho_out, n);
    return check_launch("model lame adjoint");
}

// ---------------------------------------------------------------------------
// Allocation-free whole gradient (no reference counterpart): the derived medium,
// the adjoint accumulators and the second ψ-adjoint buffer live in a
// file-scope device array instead of caller workspaces.
// ---------------------------------------------------------------------------
namespace efm {

constexpr long long kScratchFloats = 16LL << 20;   // 64 MiB per device
static __device__ __align__(256) float scratch[kScratchFloats];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static float *g_scratch_dev[kMaxDevices];   // device address of `scratch`, per device

// The calling thread's current device's copy of `scratch` (looked up once per
// device, with that device current).
static int scratch_address(float **out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
        return fail(EFM_E_HIP, "efm_gradient_static: no current device");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(EFM_E_HIP, std::string("efm_gradient_static: hipGetSymbolAddress: ") +
                                       hipGetErrorString(e));
        g_scratch_dev[dev] = static_cast<float *>(p);
    }
    *out = g_scratch_dev[dev];
    return EFM_OK;
}

template <typename T>
__global__ void k_fill_zero(T *p, long long n) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = T(0);
}

template <typename T>
static int zero_fill(T *p, long long n, hipStream_t st) {
    if (n <= 0 || !p) return EFM_OK;
    const long long b = (n + 255) / 256;
    hipLaunchKernelGGL(k_fill_zero<T>, dim3((unsigned)(b < 65536 ? b : 65536)), dim3(256), 0, st, p, n);
    return check_launch("zero fill");
}

}  // namespace efm

extern "C" int efm_gradient_static(const EfmDims *d, const EfmMedium *m, const EfmShots *sh,
                                   const EfmState *const *fwd, const EfmState *adj,
                                   const float *resid, float *glam, float *gmu, float *grho,
                                   double *gm6, void *stream) {
    if (!d || !m || !sh || !fwd || !adj || (!resid && d->nrec > 0) || !glam || !gmu || !grho || !gm6)
        return fail(EFM_E_ARG, "efm_gradient_static: null argument");
    if (int rc = validate(d, m, sh)) return rc;
    if (int rc = validate_state(d, adj)) return rc;
    for (int k = 0; k <= d->ntmax; ++k)
        if (int rc = validate_state(d, fwd[k])) return rc;
    const Geo g = make_geo(*d);
    const long long psi = (long long)g.S * 6 * ((long long)g.pxc + g.pyc + g.pzc);
    const long long need = (6 + 8LL * g.S) * g.ps + psi;
    if (need > kScratchFloats)
        return fail(EFM_E_ARG, "efm_gradient_static: the batch needs " + std::to_string(need * 4) +
                                   " bytes of scratch, above the library's static " +
                                   std::to_string(kScratchFloats * 4) + " (use efm_adjoint with "
                                   "caller workspaces)");
    float *base = nullptr;
    if (int rc = scratch_address(&base)) return rc;
    hipStream_t st = (hipStream_t)stream;
    float *mbar = base, *bbar = base + 3 * g.ps, *acc = base + 6 * g.ps;
    float *psi2 = acc + 8LL * g.S * g.ps;
    // what must start at zero: accumulators, the second ψ buffer, the adjoint
    // state and ∂J/∂M (fill kernels, no memset: callers may capture this call)
    int rc = zero_fill(acc, 8LL * g.S * g.ps + psi, st);
    const long long vol = (long long)g.S * g.N;
    float *fields[9] = {adj->vx, adj->vy, adj->vz, adj->txx, adj->tyy, adj->tzz, adj->txy, adj->txz, adj->tyz};
    for (int k = 0; k < 9 && !rc; ++k) rc = zero_fill(fields[k], vol, st);
    if (!rc) rc = zero_fill(adj->psi_x, (long long)g.S * 6 * g.pxc, st);
    if (!rc) rc = zero_fill(adj->psi_y, (long long)g.S * 6 * g.pyc, st);
    if (!rc) rc = zero_fill(adj->psi_z, (long long)g.S * 6 * g.pzc, st);
    if (!rc) rc = zero_fill(gm6, 6LL * g.S, st);
    if (rc) return rc;
    hipLaunchKernelGGL(k_derived, dim3(blocks_for(g.N, 256)), dim3(256), 0, st, g, m->mu, m->rho, mbar, bbar);
    if ((rc = check_launch("derived medium"))) return rc;
    EfmState second = *adj;
    second.psi_x = psi2;
    second.psi_y = psi2 + (long long)g.S * 6 * g.pxc;
    second.psi_z = second.psi_y + (long long)g.S * 6 * g.pyc;
    AdjArgs A;
    A.lam = m->lam; A.mu = m->mu; A.mbar = mbar; A.bbar = bbar; A.acc = acc;
    A.sh = make_shots(*sh);
    A.resid = resid;
    A.gm6 = gm6;
    A.n0 = 0;
    A.n1 = d->ntmax;
    if ((rc = run_adjoint(d, g, A, fwd, adj, &second, 0, d->ntmax, 1, false, st))) return rc;
    hipLaunchKernelGGL(k_combine, dim3(blocks_for(g.N, 256)), dim3(256), 0, st, g, m->mu, mbar, bbar,
                       acc, glam, gmu, grho);
    return check_launch("gradient combine");
}
