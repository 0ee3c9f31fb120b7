// Internal header shared by the gfx950 kernels of libefm.so.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <string>

#include "efm.h"

namespace efm {

constexpr int H = 2;  // interior guard: 2 <= x,y,z < n-2 (reference M:54, 77, 152)
constexpr int kLine = 32;  // floats of a 128-byte cache line

// Everything a sweep kernel needs, passed by value (kernel-argument memory).
struct Geo {
    int nx, ny, nz, S;
    int s0;                            // first shot of this launch (it covers shots s0 .. s0+S-1)
    int wxl, wxh, wyl, wyh, wzl, wzh;  // CPML widths per face
    int Lx, Ly, Lz;                    // slab extents wxl+wxh, ...
    int ntmax, nrec;
    float c;                           // signed dt/dx
    long long N;                       // nx*ny*nz
    long long sxz;                     // nx*nz (y stride)
    long long ps;                      // padded component stride N + EFM_PAD (acc, mbar, bbar)
    int sxz32;                         // nx*nz as int (per-shot offsets are 32-bit)
    int pxc, pyc, pzc;                 // per-component strides of the ψ slabs
    const int *itp;                    // device time-step counter added to `it` (graph replay), or null
    int recw;                          // words per shot of the receiver bitmask, ceil(N/32)
    int dense;                         // compact sweeps walk the interior cells only (see tile_coords)
};

struct StatePtrs {
    float *v[3];    // vx vy vz
    float *t[6];    // txx tyy tzz txy txz tyz
    float *px, *py, *pz;
};

struct ShotPtrs {
    const float *ax, *bx, *ay, *by, *az, *bz;
    const int *src;
    const float *m6;
    const float *wav;
    const int *nt;
    const int *rec;
    const unsigned *recmask;   // (S, recw) receiver bitmask, or null
};

inline Geo make_geo(const EfmDims &d) {
    Geo g;
    g.nx = d.nx; g.ny = d.ny; g.nz = d.nz; g.S = d.nshot; g.s0 = 0;
    g.wxl = d.wx_lo; g.wxh = d.wx_hi; g.wyl = d.wy_lo; g.wyh = d.wy_hi;
    g.wzl = d.wz_lo; g.wzh = d.wz_hi;
    g.Lx = d.wx_lo + d.wx_hi; g.Ly = d.wy_lo + d.wy_hi; g.Lz = d.wz_lo + d.wz_hi;
    g.ntmax = d.ntmax; g.nrec = d.nrec; g.c = d.dtdx;
    g.sxz = (long long)d.nx * d.nz;
    g.N = g.sxz * d.ny;
    g.ps = g.N + EFM_PAD;
    g.sxz32 = d.nx * d.nz;
    g.pxc = d.ny * d.nz * g.Lx;
    g.pyc = g.Ly * d.nz * d.nx;
    g.pzc = d.ny * g.Lz * d.nx;
    g.itp = nullptr;
    g.recw = (int)((g.N + 31) / 32);
    // the line-aligned walk takes the guard cells of its rows along: a batch that would pass a
    // dispatch's 2^32 work-items with them (bound for blocks of up to 256 cells, 8 runs of
    // blocks a shot) walks the interior cells only
    const long long per_plane = (long long)(d.nz - 2 * H) * d.nx + kLine + 255;
    g.dense = g.S * (per_plane * (d.ny - 2 * H) + 7 * 256) > (long long)UINT32_MAX;
    return g;
}

inline StatePtrs make_state(const EfmState &s) {
    StatePtrs p;
    p.v[0] = s.vx; p.v[1] = s.vy; p.v[2] = s.vz;
    p.t[0] = s.txx; p.t[1] = s.tyy; p.t[2] = s.tzz;
    p.t[3] = s.txy; p.t[4] = s.txz; p.t[5] = s.tyz;
    p.px = s.psi_x; p.py = s.psi_y; p.pz = s.psi_z;
    return p;
}

inline ShotPtrs make_shots(const EfmShots &s) {
    ShotPtrs p;
    p.ax = s.ax; p.bx = s.bx; p.ay = s.ay; p.by = s.by; p.az = s.az; p.bz = s.bz;
    p.src = s.src; p.m6 = s.m6; p.wav = s.wavelet; p.nt = s.nt; p.rec = s.rec;
    p.recmask = s.recmask;
    return p;
}

// Per-shot ψ slab bases: comp c of shot s starts at base + c*pxc (int offsets below).
__device__ __forceinline__ long long px_shot(const Geo &g, int s) { return (long long)s * 6 * g.pxc; }
__device__ __forceinline__ long long py_shot(const Geo &g, int s) { return (long long)s * 6 * g.pyc; }
__device__ __forceinline__ long long pz_shot(const Geo &g, int s) { return (long long)s * 6 * g.pzc; }
__device__ __forceinline__ int px_off(const Geo &g, int y, int z, int sx) { return (y * g.nz + z) * g.Lx + sx; }
__device__ __forceinline__ int py_off(const Geo &g, int sy, int z, int x) { return (sy * g.nz + z) * g.nx + x; }
__device__ __forceinline__ int pz_off(const Geo &g, int y, int sz, int x) { return (y * g.Lz + sz) * g.nx + x; }

// ---- slab addressing (ψ lives only in the CPML slabs) ----------------------
// Returns the slab coordinate along an axis of length n with widths lo/hi, or -1.
__device__ __forceinline__ int slab_coord(int i, int n, int lo, int hi) {
    if (i < lo) return i;
    if (i >= n - hi) return lo + (i - (n - hi));
    return -1;
}
// psi_x (S, 6, ny, nz, Lx)
__device__ __forceinline__ long long px_index(const Geo &g, int s, int comp, int y, int z, int sx) {
    return ((((long long)s * 6 + comp) * g.ny + y) * g.nz + z) * g.Lx + sx;
}
__device__ __forceinline__ long long px_cstride(const Geo &g) { return (long long)g.ny * g.nz * g.Lx; }
// psi_y (S, 6, Ly, nz, nx)
__device__ __forceinline__ long long py_index(const Geo &g, int s, int comp, int sy, int z, int x) {
    return ((((long long)s * 6 + comp) * g.Ly + sy) * g.nz + z) * g.nx + x;
}
__device__ __forceinline__ long long py_cstride(const Geo &g) { return (long long)g.Ly * g.nz * g.nx; }
// psi_z (S, 6, ny, Lz, nx)
__device__ __forceinline__ long long pz_index(const Geo &g, int s, int comp, int y, int sz, int x) {
    return ((((long long)s * 6 + comp) * g.ny + y) * g.Lz + sz) * g.nx + x;
}
__device__ __forceinline__ long long pz_cstride(const Geo &g) { return (long long)g.ny * g.Lz * g.nx; }

__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }

// Whether cell t (per-shot linear index) of shot s holds a receiver.
__device__ __forceinline__ bool is_receiver(const Geo &g, const ShotPtrs &sh, int s, int t) {
    return (sh.recmask[(long long)s * g.recw + (t >> 5)] >> (t & 31)) & 1u;
}

// The receivers among a wave's cells, which follow one another in memory (or, in a dense
// walk, among the interior cells of their plane): t is the lane's cell.  The active lanes
// take the list one receiver each; f(r, lane, hit) is called by all of them for each
// share of the list, with the lane that owns the cell of this lane's receiver r where there
// is one (hit).  A lane with a receiver that walked the list by itself kept its wave, and
// with it the sweep, for 6.5 us per 100 receivers: velocity sweep of 100^3 with 200
// receivers 25.7 -> 13.0 us, 64^3 with 16 receivers 6.2 -> 5.7.
template <typename F>
__device__ __forceinline__ void wave_receivers(const Geo &g, const ShotPtrs &sh, int s, int t, F f) {
    const unsigned long long on = __ballot(1);
    const int lane = __lane_id(), n = __popcll(on), rank = __popcll(on & ((1ull << lane) - 1));
    const int *rs = sh.rec + (long long)s * g.nrec;
    // place of cell c in the walk; another plane's or a guard cell of a dense walk: far away
    const int y0 = g.dense ? t / g.sxz32 : 0;
    auto place = [&](int c) {
        if (!g.dense) return c;
        const int p = c - y0 * g.sxz32, z = p / g.nx, x = p - z * g.nx;
        const bool in = p >= 0 && p < g.sxz32 && x >= H && x < g.nx - H && z >= H && z < g.nz - H;
        return in ? (z - H) * (g.nx - 2 * H) + x - H : -(1 << 30);
    };
    const int first = place(t) - lane;
    for (int r0 = 0; r0 < g.nrec; r0 += n) {
        const int r = r0 + rank;
        const int j = place(r < g.nrec ? rs[r] : -1) - first;
        f(r, j & 63, (unsigned)j < 64u && (on >> (j & 63) & 1));
    }
}

// Adds the residual of sample n, res (S, 3, ntmax, nrec), to v at the receivers among the
// wave's cells, in the order of the list where several share a cell.
__device__ __forceinline__ void inject_wave(const Geo &g, const ShotPtrs &sh, int s, int t, const float *res, int n,
                                            float &v0, float &v1, float &v2) {
    if (!__any(is_receiver(g, sh, s, t))) return;
    const long long cs = (long long)g.ntmax * g.nrec, base = ((long long)s * 3 * g.ntmax + n) * g.nrec;
    wave_receivers(g, sh, s, t, [&](int r, int owner, bool hit) __attribute__((always_inline)) {
        unsigned long long todo = __ballot(hit);
        if (!todo) return;
        float q0 = 0.f, q1 = 0.f, q2 = 0.f;
        if (hit) { q0 = res[base + r]; q1 = res[base + cs + r]; q2 = res[base + 2 * cs + r]; }
        for (; todo; todo &= todo - 1) {
            const int i = __ffsll(todo) - 1;
            const float a0 = __shfl(q0, i), a1 = __shfl(q1, i), a2 = __shfl(q2, i);
            if ((int)__lane_id() == __shfl(owner, i)) { v0 += a0; v1 += a1; v2 += a2; }
        }
    });
}

__device__ __forceinline__ bool interior(int x, int y, int z, const Geo &g) {
    return x >= H && x < g.nx - H && y >= H && y < g.ny - H && z >= H && z < g.nz - H;
}

// Four consecutive floats read or written with one instruction; 4-byte alignment is
// enough for global memory.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// ---- error plumbing ---------------------------------------------------------
void set_error(const std::string &msg);
int fail(int code, const std::string &msg);
int check_launch(const char *what);
// Grid, CPML widths, record length and the size limits of the sweep kernels
// (32-bit offsets inside a shot, one dispatch of < 2^32 work-items per sweep).
int check_dims(const EfmDims *d);
// Null checks of the C-ABI structs (EFM_E_ARG with a message): the shot
// description's arrays, dims + medium + shots, and one state (ψ slab pointers
// are required for every axis that has a CPML layer).
int validate_shots(const EfmDims *d, const EfmShots *sh);
int validate(const EfmDims *d, const EfmMedium *m, const EfmShots *sh);
int validate_state(const EfmDims *d, const EfmState *s);

// ---- tile configuration chosen by the autotuner ------------------------------
struct Tile {
    int bx, bz, ny;  // threads in x, threads in z, cells per thread along y
    int map;         // block mapping: 0 = linear 3-D grid; 8 = XCD-aware over 8 XCDs;
                     // 16 = XCD-aware over the plane's cells in memory order (see tile_coords)
};

// Compiled tile variants (bx, bz, ny, map).  Whole 64-lane waves along x.
#define EFM_TILE_LIST(X) \
    X(64, 1, 1, 0)       \
    X(64, 2, 1, 0)       \
    X(64, 4, 1, 0)       \
    X(128, 1, 1, 0)      \
    X(128, 2, 1, 0)      \
    X(64, 4, 2, 0)       \
    X(64, 1, 1, 8)       \
    X(64, 2, 1, 8)       \
    X(64, 4, 1, 8)       \
    X(64, 8, 1, 8)       \
    X(128, 1, 1, 8)      \
    X(128, 2, 1, 8)      \
    X(256, 1, 1, 8)      \
    X(64, 4, 2, 8)       \
    X(64, 1, 1, 16)      \
    X(128, 1, 1, 16)     \
    X(256, 1, 1, 16)     \
    X(128, 1, 2, 16)

// XCDs the blocks of an XCD-aware mapping are dealt over.
__host__ __device__ constexpr int map_xcds(int map) { return map == 16 ? 8 : map; }

// The cells a compact sweep walks in a plane: from the line of the first interior cell to
// the last interior cell, or the interior ones.
__host__ __device__ inline int plane_span(const Geo &g) {
    return g.dense ? (g.nz - 2 * H) * (g.nx - 2 * H) : (g.nz - 2 * H) * g.nx - 2 * H + kLine - 1;
}

// Number of tiles (blocks × y-chunks × shots) of a sweep: x-blocks × z-blocks,
// or, for the compact mapping, blocks of bx·bz consecutive cells of the plane.
inline long long sweep_tiles(const Geo &g, int bx, int bz, int ny, int map) {
    const long long nyc = (g.ny - 2 * H + ny - 1) / ny;
    if (map == 16) {
        const long long q = plane_span(g);
        return (q + bx * bz - 1) / (bx * bz) * nyc * g.S;
    }
    const long long nbx = (g.nx + bx - 1) / bx, nbz = (g.nz + bz - 1) / bz;
    return nbx * nbz * nyc * g.S;
}

// Whether a forward step walks the interior cells only (Geo::dense) and not the cells of
// whole lines.  Its shorter index arithmetic gives the aligned walk the launches whose blocks
// the chip holds at once (the stress sweep: 14 of 128 lanes a CU); a few blocks more take a
// second round, and without the four guard cells of each row they often fit.  Aligned and dense
// walks, us per step, with the aligned walk's blocks: 64x122x64 (3658) 15.8 and 15.7,
// 64x126x64 (3782) 16.7 and 16.0, 76x90x76 (3698) 16.5 and 16.0, 68x40x70 x 3 (3888) 18.5 and 17.5,
// 52x124x78 (3720) 16.6 and 15.7; below, 130x60x64 (3472) 15.5 and 16.4, 61x47x53 x 3 (3096) 15.8
// and 16.3, 45x100x100 (3264) 15.0 and 15.7, 48^3 (748) 9.7 and 10.0.  Beyond one round rows under
// 64 cells keep the dense walk, since the guard cells are a larger share: 1.4 % shorter over
// 40 batches (28x100x100 x 3 22.6 and 21.4, 36x138x89 x 10 109.4 and 107.8; runs differ by 0.3 %),
// 3.3 % longer at worst (60x200x200 x 4, 257 and 266).  From 64 cells on the walks are within 1-2 %
// of each other until memory binds them, where whole lines count (128^3 and up).
constexpr int kDenseRow = 64;
constexpr long long kRoundLanes = 14LL * 128 * 256;
inline bool dense_walk(Geo g) {
    const auto lanes = [&](int dense) { g.dense = dense; return 128 * sweep_tiles(g, 128, 1, 1, 16); };
    return lanes(0) > kRoundLanes && (g.nx < kDenseRow || lanes(1) <= kRoundLanes);
}

// Blocks of an XCD-aware sweep: each shot's tiles are dealt over the k XCDs in
// runs of ceil(tiles/k) (see tile_coords), so a shot takes k·ceil(tiles/k).
inline long long xcd_blocks(const Geo &g, const Tile &t) {
    const long long per_shot = sweep_tiles(g, t.bx, t.bz, t.ny, t.map) / g.S;
    const int k = map_xcds(t.map);
    return k * ((per_shot + k - 1) / k) * g.S;
}

inline dim3 sweep_grid(const Geo &g, const Tile &t) {
    if (t.map > 0) return dim3((unsigned)xcd_blocks(g, t));
    const int nyc = (g.ny - 2 * H + t.ny - 1) / t.ny;
    return dim3((g.nx + t.bx - 1) / t.bx, (g.nz + t.bz - 1) / t.bz, g.S * nyc);
}

// Tile coordinates of the calling block.  MAP = 0: the 3-D grid as launched.
// MAP = k: workgroups are dealt to the k XCDs round-robin (w mod k), each with
// its own L2, so block w is given a tile of its XCD's contiguous run: every XCD
// walks a run of a shot's tiles (x fastest, then z, then y), and the ±z rows and
// ±y planes a tile reads were fetched into the same L2 by its neighbours.  The
// runs are per shot (XCD k takes the k-th run of shot 0, then of shot 1, ...), so
// all XCDs work on the same shot at a time and a batch's sweep keeps one shot's
// working set in the Infinity Cache, as a one-shot sweep does.
// MAP = 16: the same XCD order over blocks of BX·BZ consecutive cells of the plane's
// memory, rows wrapped, from the 128-byte line of its first interior cell: waves are
// full but for the four guard cells of each row whatever nx is (the other mappings
// leave part-empty waves where nx is not a multiple of 64), and each wave's row of
// 64 floats is two whole cache lines in every array whose base is line-aligned.
// Walking the interior cells only (124 of 128 lanes more useful at 128^3, but waves
// that straddle three lines) was slower: adjoint step 107 against 97 us at 128^3, 226
// against 204 at 200x200x100; forward step 979 against 906 us for four shots of
// 256x256x128, 728 against 704 for 32 of 96^3, the same at 128^3.
// The kernels return on lanes outside the interior.
// Returns false for the padding blocks past the last tile.
template <int BX, int BZ, int NYC, int MAP>
__device__ __forceinline__ bool tile_coords(const Geo &g, int &x, int &z, int &s, int &yb) {
    const int nyc = (g.ny - 2 * H + NYC - 1) / NYC;
    if (MAP == 16) {
        const int nqb = (plane_span(g) + BX * BZ - 1) / (BX * BZ);
        const int per_shot = nqb * nyc;
        const int run = (per_shot + 7) / 8;
        const int w = blockIdx.x;
        const int j = w / 8;
        const int sl = j / run;
        const int gi = (w % 8) * run + (j - sl * run);
        if (sl >= g.S || gi >= per_shot) return false;
        s = g.s0 + sl;
        const int qb = gi % nqb;
        yb = gi / nqb;
        if (g.dense) {
            const int q = qb * (BX * BZ) + threadIdx.y * BX + threadIdx.x, w = g.nx - 2 * H;
            z = H + q / w;
            x = H + q - (z - H) * w;
            return z < g.nz - H;
        }
        // position in the plane of the line-aligned cell the plane's walk starts at
        const int row0 = (H + yb * NYC) * g.sxz32;
        const int p = ((row0 + H * g.nx + H) & ~(kLine - 1)) - row0 + qb * (BX * BZ) + threadIdx.y * BX + threadIdx.x;
        z = p / g.nx;
        x = p - z * g.nx;
        return true;
    }
    if (MAP == 0) {
        x = blockIdx.x * BX + threadIdx.x;
        z = blockIdx.y * BZ + threadIdx.y;
        const int sl = blockIdx.z / nyc;
        s = g.s0 + sl;
        yb = blockIdx.z - sl * nyc;
        return true;
    }
    const int nbx = (g.nx + BX - 1) / BX, nbz = (g.nz + BZ - 1) / BZ;
    constexpr int K = MAP > 0 ? MAP : 1;
    const int per_shot = nbx * nbz * nyc;
    const int run = (per_shot + K - 1) / K;
    const int w = blockIdx.x;
    const int j = w / K;
    const int sl = j / run;
    const int gi = (w % K) * run + (j - sl * run);
    if (sl >= g.S || gi >= per_shot) return false;
    s = g.s0 + sl;
    const int xb = gi % nbx;
    const int r = gi / nbx;
    const int zb = r % nbz;
    yb = r / nbz;
    x = xb * BX + threadIdx.x;
    z = zb * BZ + threadIdx.y;
    return true;
}

// Launch KER<bx,bz,ny,map> for the selected tile; sets `launched`.
#define EFM_LAUNCH_GRID_IF(BX_, BZ_, NY_, MAP_, GRID, KER, ...)                                       \
    if (!launched && t.bx == BX_ && t.bz == BZ_ && t.ny == NY_ && t.map == MAP_) {                    \
        hipLaunchKernelGGL((KER<BX_, BZ_, NY_, MAP_>), GRID, dim3(BX_, BZ_), 0, st, __VA_ARGS__);     \
        launched = true;                                                                             \
    }
#define EFM_LAUNCH_IF(BX_, BZ_, NY_, MAP_, KER, ...) \
    EFM_LAUNCH_GRID_IF(BX_, BZ_, NY_, MAP_, sweep_grid(g, t), KER, __VA_ARGS__)
#define EFM_KERNEL_ATTRS(BX, BZ, MAP) __launch_bounds__(BX *BZ)

Tile get_tile(int kernel);  // 0 stress, 1 velocity, 2 adjoint-velocity, 3 adjoint-stress
int set_tile(int kernel, Tile t);

// ---- shot groups ---------------------------------------------------------------
// The forward loop takes the shots of a batch through all its steps a group at a
// time, each group as many shots as fit the 256 MB Infinity Cache with the medium,
// so that a group's fields come from HBM once per loop and not once per step.
// Measured on the two sweeps, ns per thousand interior cell-steps by shots per
// launch: 96^3 25.6 at 4 shots (190 MB), 25.8 at 5 (237 MB), 32.1 at 6 (281 MB), 35.0
// at 32; 64^3 29.0 at 16 (248 MB), 42.0 at 24 (371 MB); 128^3 22.7 at 2 (223 MB),
// 34.2 at 3.  32 shots of 96^3 went from 872 to 682 us per step.  The line lies at the
// cache's own size, 256 MiB: over 24 grids of 50 thousand to 1.1 million cells, all and
// part of the steps recorded, whole and in two groups (us per step): 64^3 106.5 and 115.2 at 263
// MB, 130.2 and 121.5 at 279; 48^3 105.9 and 112.7 at 260, 119.2 and 121.1 at 280; 73x64x37 98.8
// and 108.4 at 263, 106.3 and 111.7 at 272, 126.5 and 119.0 at 290; 57x169x47 98.6 and 105.7 at
// 248, 134.9 and 115.7 at 271; 36x138x89 123.0 and 120.2 at 266.  Bytes do not tell all:
// the sides cross between 255 and 280 MB by grid (33x150x60 already 131.3 and 117.7 at
// 263), and a line anywhere from 265 to 277 MB loses 0.3 % to the better side on
// average (12 % at worst from here, 17 % from 272 on), at 260 or 280 MB 0.7 %.  Where even one shot exceeds the cache all
// shots stay in one launch (fewer, longer launches).  The adjoint sweeps gain nothing from
// groups (96^3: 71 ns with 8 shots in a launch, 74-83 in groups of 2 or 1), so they take
// the whole batch.
constexpr long long kCacheBytes = 268LL * 1000 * 1000;

// Bytes of one shot's nine fields and of its ψ slabs.
inline long long field_bytes(const Geo &g) { return 36 * g.N; }
inline long long psi_bytes(const Geo &g) { return 24LL * ((long long)g.pxc + g.pyc + g.pzc); }

// Whether the imaging adjoint sweep reads the forward state with the streaming hint.  It pays
// as long as the adjoint's own working set (9 fields, 8 sums and two sets of ψ slabs a shot, 8
// volumes of the medium) stays largely in the Infinity Cache; beyond, the hint only drops lines
// that the neighbouring cells still read.  Adjoint step without and with it, us, by that set:
// 64^3 x 4 (119 MB) 56.8 and 56.2, 96^3 x 2 (193) 85.5 and 83.4, 128^3 (249) 102.7 and 93.7, 64^3 x 9
// (257) 114.7 and 109.2, 160x150x100 (281) 118.4 and 112.2, 48^3 x 24 (290) 124.6 and 120.7,
// 140x136x136 (304) 131.1 and 128.6, 48^3 x 28 (338) 149.3 and 148.0, 144^3 (348) 142.5 and 144.7,
// 200x200x100 (458) 181.3 and 184.1.
constexpr long long kStreamBytes = 320LL * 1000 * 1000;
inline bool stream_forward_state(const Geo &g) {
    return 68 * g.S * g.N + 32 * g.N + 2 * g.S * psi_bytes(g) <= kStreamBytes;
}

// Shots per group for a loop that touches `per_shot` bytes of each shot and
// `shared` bytes of the medium in every step: as many groups as the cache asks for, equal
// ones but for the last, which takes what is left.
inline int group_shots(const Geo &g, long long per_shot, long long shared) {
    const long long fit = (kCacheBytes - shared) / (per_shot > 0 ? per_shot : 1);
    if (fit < 1 || fit >= g.S) return g.S;
    const int groups = (int)((g.S + fit - 1) / fit);
    return (g.S + groups - 1) / groups;
}

// Shots per group of nsteps steps of the forward loop.  A group's first step brings its
// fields from HBM as the whole batch's steps do, so a call of one step gains nothing and
// pays the further launches: over 52 batches of 1 to 2.5 times the line, with full and with
// uneven records, groups took 6.3 % longer than the whole batch at one step a call (10 % at
// worst, 96^3 x 32 831.7 against 773.7 us), 1.4 % less at two (from 8 % longer to 10 %
// less), 4.6 % less at three, 6.4 % at four, 12 % at 24.  Kept states take a second state's
// velocities and slabs along, which these bytes leave out; whole and in groups, us per step:
// 64^3 x 20 147.0 and 143.0, 96^3 x 8 205.0 and 189.5, 128^3 x 3 163.0 and 163.2, 36x138x89 x 16
// 222.1 and 190.5.  Counting both states shortens some (57x169x47 x 12 144.5 -> 134.8) and lengthens
// others (64^3 x 12 84.5 -> 90.4).
constexpr int kGroupSteps = 3;
inline int forward_group(const Geo &g, int nsteps) {
    return nsteps < kGroupSteps ? g.S : group_shots(g, field_bytes(g) + psi_bytes(g), 12 * g.N);
}

// Calls f(geo) for each group (geo.s0, geo.S name its shots); f returns an error code.
template <typename F>
int for_shot_groups(const Geo &g, int group, F f) {
    for (int s = 0; s < g.S; s += group) {
        Geo gg = g;
        gg.s0 = g.s0 + s;
        gg.S = g.S - s < group ? g.S - s : group;
        if (int rc = f(gg)) return rc;
    }
    return EFM_OK;
}

// ---- launchers (defined in the .hip files) ------------------------------------
int launch_stress_src(const Geo &g, const EfmMedium &m, const ShotPtrs &sh, const StatePtrs &in,
                      const StatePtrs &out, int it, int src_mode, hipStream_t st);
int launch_stress(const Geo &g, const EfmMedium &m, const ShotPtrs &sh, const StatePtrs &in,
                  const StatePtrs &out, int it, hipStream_t st);
int launch_velocity(const Geo &g, const EfmMedium &m, const ShotPtrs &sh, const StatePtrs &in,
                    const StatePtrs &out, int it, hipStream_t st, float *gathers = nullptr);
int launch_record(const Geo &g, const ShotPtrs &sh, const StatePtrs &s, float *gathers, int it,
                  hipStream_t st);
int launch_border(const Geo &g, const ShotPtrs &sh, const StatePtrs &s, float *borders, int W,
                  int slot, int save, int it_gate, hipStream_t st);
long long border_floats(const Geo &g, int W);
// Steps it0 .. it0+nsteps-1 of the forward loop.  `states`: nsteps + 1 states, step
// it0 + k reading state k and writing state k + 1, or (in_place) one state advanced
// in place.  Receivers are sampled when `gathers` is set, the reference's border
// layers saved when `borders` is set.
int run_forward(const Geo &g, const EfmMedium &m, const ShotPtrs &sh, const EfmState *const *states,
                bool in_place, float *gathers, float *borders, int W, int it0, int nsteps,
                hipStream_t st);

}  // namespace efm
