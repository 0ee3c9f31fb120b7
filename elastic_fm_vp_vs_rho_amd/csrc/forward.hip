// Forward sweeps of the 3-D elastic velocity-stress staggered-grid FDTD
// (O(2,2), CPML), written for gfx950.
//
// Reference: kernel_Tau (mainPropElastic3D_MT.py M:59-128), addSource
// (M:1728-1734), kernel_Vx_Vy_Vz (M:133-188), kernel_get_Station (M:324-335),
// kernel_get_border / kernel_set_border (M:378-462).
//
// Mapping: a block is BX (x) × BZ (z) threads and each thread owns NYC cells along y; the
// compact mapping (the default) deals a plane's cells to the lanes in memory order.  x is
// the contiguous axis, so every wave issues coalesced row loads; a cell's ±1 neighbours are
// other lanes' cells and come from the CU's vector cache or the XCD's L2.  ψ memory
// variables live only in CPML slabs (identically zero elsewhere, where a = b = 0).  The
// moment-tensor source is added by the thread that owns the source cell right after it
// writes τ (the reference adds it with six separate gpuarray launches).
#include "sweeps.hpp"

namespace efm {

// ---------------------------------------------------------------------------
// stress sweep
// ---------------------------------------------------------------------------
template <int BX, int BZ, int NYC, int MAP>
__global__ EFM_KERNEL_ATTRS(BX, BZ, MAP) void k_stress(Geo g, Med m, ShotPtrs sh, StatePtrs in,
                                                       StatePtrs out, int it, int src_mode) {
    if (g.itp) it += *g.itp;
    int x, z, s, yb;
    if (!tile_coords<BX, BZ, NYC, MAP>(g, x, z, s, yb)) return;
    if (x < H || x >= g.nx - H || z < H || z >= g.nz - H) return;
    if (it >= sh.nt[s]) return;
    stress_cells<NYC>(g, m, sh, in, out, it, src_mode, x, z, s, yb, true, [](int, CellOld) {});
}

// ---------------------------------------------------------------------------
// velocity sweep
// ---------------------------------------------------------------------------
// 8 waves to a SIMD: at 82 to 86 SGPRs, which the compiler takes by itself, 7 fit (16 more
// belong to the trap handler), at 78 or fewer 8, and none is spilled; a launch of 3585 to 4096
// blocks of 128 then takes one round of them, not two.  Forward step: 52x124x78 17.8 -> 16.8 us,
// 64x132x64 18.1 -> 17.0, 128x27x55 x 6 28.0 -> 27.1, 128^3 50.6 -> 50.0, in row tiles (64, 4)
// 64x132x64 18.9 -> 17.7.  The XCD-aware row tiles gain nothing and would spill.
template <int BX, int BZ, int NYC, int MAP>
__global__ EFM_KERNEL_ATTRS(BX, BZ, MAP) __attribute__((amdgpu_waves_per_eu(NYC == 1 && MAP != 8 ? 8 : 1, 8))) void
k_velocity(Geo g, Med m, ShotPtrs sh, StatePtrs in, StatePtrs out, int it, float *gathers) {
    if (g.itp) it += *g.itp;
    int x, z, s, yb;
    if (!tile_coords<BX, BZ, NYC, MAP>(g, x, z, s, yb)) return;
    if (x < H || x >= g.nx - H || z < H || z >= g.nz - H) return;
    if (it >= sh.nt[s]) return;
    auto keep = [](int, int, float, float, float) {};
    velocity_cells<NYC>(g, m, sh, in, out, x, z, s, yb, keep, [&](int t, float n0, float n1, float n2) EFM_INLINE {
        // receiver sampling from the cells' own lanes (kernel_get_Station, M:324-335)
        if (!gathers || !__any(is_receiver(g, sh, s, t))) return;
        const long long cs = (long long)g.ntmax * g.nrec;
        const long long base = ((long long)s * 3 * g.ntmax + it) * g.nrec;
        wave_receivers(g, sh, s, t, [&](int r, int owner, bool hit) EFM_INLINE {
            const float v0 = __shfl(n0, owner), v1 = __shfl(n1, owner), v2 = __shfl(n2, owner);
            if (!hit) return;
            gathers[base + r] = v0;
            gathers[base + cs + r] = v1;
            gathers[base + 2 * cs + r] = v2;
        });
    });
}

// ---------------------------------------------------------------------------
// receivers
// ---------------------------------------------------------------------------
__global__ void k_record(Geo g, ShotPtrs sh, StatePtrs st, float *gathers, int it) {
    if (g.itp) it += *g.itp;
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    const int s = g.s0 + blockIdx.y;
    if (r >= g.nrec || it >= sh.nt[s]) return;
    const int cell = sh.rec[(long long)s * g.nrec + r];
    if (cell < 0) return;
    const long long t = (long long)s * g.N + cell;
    const long long base = ((long long)s * 3 * g.ntmax + it) * g.nrec + r;
    const long long cstride = (long long)g.ntmax * g.nrec;
    gathers[base] = st.v[0][t];
    gathers[base + cstride] = st.v[1][t];
    gathers[base + 2 * cstride] = st.v[2][t];
}

// ---------------------------------------------------------------------------
// reference boundary save / restore of v
// ---------------------------------------------------------------------------
long long border_floats(const Geo &g, int W) {
    (void)W;
    return 3 * border_layout(g.nx, g.ny, g.nz).comp;
}

// borders: (S, nslot, 3, comp)
__device__ __forceinline__ float *border_slot(float *borders, const BorderLayout &L, int s, int slot, int nslot) {
    return borders + ((long long)s * nslot + slot) * 3 * L.comp;
}

// One thread per (component, face element).
__global__ void k_border(Geo g, ShotPtrs sh, StatePtrs st, float *borders, int W, int slot,
                         int nslot, int save, int it_gate) {
    const BorderLayout L = border_layout(g.nx, g.ny, g.nz);
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int s = g.s0 + blockIdx.y;
    if (i >= 3 * L.comp) return;
    if (it_gate >= 0 && it_gate >= sh.nt[s]) return;
    const BorderCell c = border_cell(g, L, W, i);
    const long long t = (long long)s * g.N + c.x + (long long)c.z * g.nx + (long long)c.y * g.sxz;
    float *buf = border_slot(borders, L, s, slot, nslot) + i;
    if (save) *buf = st.v[c.comp][t];
    else st.v[c.comp][t] = *buf;
}

// The stress sweep of step `it` with the border save of step it - 1 in the blocks behind
// it: both only read v.  A launch of its own took the save 4.7 us of a step's 32 at 100^3,
// nearly all of it the launch; here it adds 0.5.
template <int BX, int BZ, int NYC, int MAP>
__global__ EFM_KERNEL_ATTRS(BX, BZ, MAP) void k_stress_save(Geo g, Med m, ShotPtrs sh, StatePtrs in, StatePtrs out,
                                                            int it, float *borders, int W, long long nsweep) {
    const long long extra = block_number() - nsweep;
    if (extra >= 0) {
        const BorderLayout L = border_layout(g.nx, g.ny, g.nz);
        const long long k = extra * (BX * BZ) + threadIdx.y * BX + threadIdx.x;
        const long long sl = k / (3 * L.comp), i = k - sl * 3 * L.comp;
        const int s = g.s0 + (int)sl;
        if (sl >= g.S || it - 1 >= sh.nt[s]) return;
        const BorderCell c = border_cell(g, L, W, i);
        border_slot(borders, L, s, it - 1, g.ntmax)[i] =
            in.v[c.comp][(long long)s * g.N + c.x + (long long)c.z * g.nx + (long long)c.y * g.sxz];
        return;
    }
    int x, z, s, yb;
    if (!tile_coords<BX, BZ, NYC, MAP>(g, x, z, s, yb)) return;
    if (x < H || x >= g.nx - H || z < H || z >= g.nz - H) return;
    if (it >= sh.nt[s]) return;
    stress_cells<NYC>(g, m, sh, in, out, it, 1, x, z, s, yb, true, [](int, CellOld) {});
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
int launch_stress_src(const Geo &g, const EfmMedium &m, const ShotPtrs &sh, const StatePtrs &in,
                      const StatePtrs &out, int it, int src_mode, hipStream_t st) {
    const Tile t = get_tile(0);
    Med md{m.lam, m.mu, m.rho};
    bool launched = false;
#define X(a, b, c, o) EFM_LAUNCH_IF(a, b, c, o, k_stress, g, md, sh, in, out, it, src_mode)
    EFM_TILE_LIST(X)
#undef X
    if (!launched) return fail(EFM_E_UNSUPPORTED, "unsupported stress tile");
    return check_launch("stress sweep");
}

// Whether a sweep's blocks and `extra` more make a legal dispatch (< 2^32 work-items).
static bool dispatch_fits(const dim3 &grid, const Tile &t) {
    return grid_blocks(grid) * t.bx * t.bz <= (long long)UINT32_MAX && grid.z <= 65535 && grid.x <= 0x7fffffffu;
}

// Saves step it - 1's borders beside the stress sweep of step `it`; false where the
// dispatch would be too large.
static bool launch_stress_save(const Geo &g, const EfmMedium &m, const ShotPtrs &sh, const StatePtrs &in,
                               const StatePtrs &out, int it, float *borders, int W, hipStream_t st, int &rc) {
    const Tile t = get_tile(0);
    const long long n = 3 * border_layout(g.nx, g.ny, g.nz).comp * g.S;
    const dim3 grid = sweep_grid_plus(g, t, (n + t.bx * t.bz - 1) / (t.bx * t.bz));
    if (!dispatch_fits(grid, t)) return false;
    const long long nsweep = grid_blocks(sweep_grid(g, t));
    Med md{m.lam, m.mu, m.rho};
    bool launched = false;
#define X(a, b, c, o) EFM_LAUNCH_GRID_IF(a, b, c, o, grid, k_stress_save, g, md, sh, in, out, it, borders, W, nsweep)
    EFM_TILE_LIST(X)
#undef X
    rc = launched ? check_launch("stress sweep") : fail(EFM_E_UNSUPPORTED, "unsupported stress tile");
    return true;
}

int launch_stress(const Geo &g, const EfmMedium &m, const ShotPtrs &sh, const StatePtrs &in,
                  const StatePtrs &out, int it, hipStream_t st) {
    return launch_stress_src(g, m, sh, in, out, it, 1, st);
}

int launch_velocity(const Geo &g, const EfmMedium &m, const ShotPtrs &sh, const StatePtrs &in,
                    const StatePtrs &out, int it, hipStream_t st, float *gathers) {
    const Tile t = get_tile(1);
    Med md{m.lam, m.mu, m.rho};
    bool launched = false;
    // the sweep samples the receivers only when the shots carry a receiver bitmask
    float *gat = (sh.recmask && g.nrec > 0) ? gathers : nullptr;
#define X(a, b, c, o) EFM_LAUNCH_IF(a, b, c, o, k_velocity, g, md, sh, in, out, it, gat)
    EFM_TILE_LIST(X)
#undef X
    if (!launched) return fail(EFM_E_UNSUPPORTED, "unsupported velocity tile");
    return check_launch("velocity sweep");
}

int launch_record(const Geo &g, const ShotPtrs &sh, const StatePtrs &s, float *gathers, int it,
                  hipStream_t st) {
    if (g.nrec <= 0) return EFM_OK;
    dim3 grid((g.nrec + 63) / 64, g.S);
    hipLaunchKernelGGL(k_record, grid, dim3(64), 0, st, g, sh, s, gathers, it);
    return check_launch("record");
}

int launch_border(const Geo &g, const ShotPtrs &sh, const StatePtrs &s, float *borders, int W,
                  int slot, int save, int it_gate, hipStream_t st) {
    const long long n = 3 * border_layout(g.nx, g.ny, g.nz).comp;
    dim3 grid((unsigned)((n + 255) / 256), g.S);
    hipLaunchKernelGGL(k_border, grid, dim3(256), 0, st, g, sh, s, borders, W, slot, g.ntmax,
                       save, it_gate);
    return check_launch("border");
}

int run_forward(const Geo &g0, const EfmMedium &m, const ShotPtrs &sh, const EfmState *const *states,
                bool in_place, float *gathers, float *borders, int W, int it0, int nsteps,
                hipStream_t st) {
    const int group = forward_group(g0, nsteps);
    Geo gd = g0;
    gd.dense |= dense_walk(g0);
    return for_shot_groups(gd, group, [&](const Geo &g) {
        bool unsaved = false;       // the borders of the step before
        for (int k = 0; k < nsteps; ++k) {
            const int it = it0 + k;
            const StatePtrs in = make_state(*states[in_place ? 0 : k]);
            const StatePtrs out = make_state(*states[in_place ? 0 : k + 1]);
            int rc = EFM_OK;
            if (!unsaved || !launch_stress_save(g, m, sh, in, out, it, borders, W, st, rc)) {
                if (unsaved && (rc = launch_border(g, sh, in, borders, W, it - 1, 1, it - 1, st))) return rc;
                rc = launch_stress_src(g, m, sh, in, out, it, 1, st);
            }
            if (rc || (rc = launch_velocity(g, m, sh, in, out, it, st, gathers))) return rc;
            if (gathers && !sh.recmask)
                if ((rc = launch_record(g, sh, out, gathers, it, st))) return rc;
            unsaved = borders != nullptr;
            if (unsaved && k == nsteps - 1)
                if ((rc = launch_border(g, sh, out, borders, W, it, 1, it, st))) return rc;
        }
        return (int)EFM_OK;
    });
}

}  // namespace efm
