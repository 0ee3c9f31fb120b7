// Gradient conditioning and model maps of the FWI driver, on the device.
//
// Reference: fwi_Vp_Vs_Rho (mainPropElastic3D_MT.py M:2349-2719) smooths the
// summed λ/μ/ρ images with scipy.ndimage.gaussian_filter(σ = 1; defaults
// mode='reflect', truncate=4.0) and zeroes the top 10 cells and the CPML+2
// zones (M:2479-2504), then updates λ and μ, maps them back to Vp and Vs
// (Model.compute_Vp_Vs, M:1200-1202), ρ from Vp by the Nafe-Drake polynomial
// (Model.compute_Rho, M:1204-1206) and restores ρ in the top 10 cells
// (M:2580-2583, 2656-2661, 2688-2694).  The reference does all of this with
// numpy/scipy on the host; here the volumes stay in HBM.
//
// Smoothing: one pass per axis in scipy's order (axis 0 = y, 1 = z, 2 = x of
// the (ny, nz, nx) volume), each output cell summed in double over its
// 2r+1 neighbours in scipy's order (centre first, then the symmetric pairs
// from the outermost inwards) and rounded to float32 per pass, as
// scipy.ndimage.correlate1d does for float32 arrays; 'reflect' extends a line
// as (d c b a | a b c d | d c b a).  The masks are applied while the last pass
// writes.  For the driver's radius the three passes are one kernel (k_gauss4); any other
// takes a streaming pass per axis (8 B per cell and pass; the neighbours come from the
// caches).
#include <algorithm>
#include <cmath>

#include "common.hpp"

namespace efm {

constexpr int kMaxRadius = 64;

struct GaussTaps {
    double w[kMaxRadius + 1];   // w[j] for j = 0 .. r (symmetric kernel)
    int r;
};

// scipy.ndimage 'reflect' index for a line of length n (any j).
__device__ __forceinline__ int reflect_index(int j, int n) {
    const int p = 2 * n;
    int m = j % p;
    if (m < 0) m += p;
    return m >= n ? p - 1 - m : m;
}

struct Margins {
    int xl, xh, yl, yh, zl, zh;
};

__device__ __forceinline__ bool masked(const Margins &mg, int x, int y, int z, int nx, int ny, int nz) {
    return x < mg.xl || x >= nx - mg.xh || y < mg.yl || y >= ny - mg.yh || z < mg.zl || z >= nz - mg.zh;
}

// The same for -n <= j < 2n (one reflection), without the modulo.
__device__ __forceinline__ int reflect_once(int j, int n) {
    return j < 0 ? -1 - j : (j >= n ? 2 * n - 1 - j : j);
}

// The sum of one output cell from its 2R+1 values, in scipy's order (products not rounded).
template <int R>
__device__ __forceinline__ float gauss_sum(const float *v, const GaussTaps &taps) {
#pragma clang fp contract(off)
    double acc = (double)v[R] * taps.w[0];
#pragma unroll
    for (int j = R; j >= 1; --j) acc = fma((double)v[R - j] + (double)v[R + j], taps.w[j], acc);
    return (float)acc;
}

// One separable pass along AXIS (0 = y, 1 = z, 2 = x); mask applied when
// `mask` is set (the last pass).  Threads are (x, z), the blocks' third index is y, so
// coordinates cost no division.  Any radius, any line.
template <int AXIS>
__global__ __launch_bounds__(256) void k_gauss_pass(const float *__restrict__ in, float *__restrict__ out,
                                                    int nx, int ny, int nz, GaussTaps taps, int mask,
                                                    Margins mg) {
#pragma clang fp contract(off)
    const int x = blockIdx.x * blockDim.x + threadIdx.x, r = taps.r;
    if (x >= nx) return;
    const long long stride = AXIS == 0 ? (long long)nx * nz : AXIS == 1 ? nx : 1;
    const int n = AXIS == 0 ? ny : AXIS == 1 ? nz : nx;
    for (int y = blockIdx.z; y < ny; y += gridDim.z)
        for (int z = blockIdx.y * blockDim.y + threadIdx.y; z < nz; z += gridDim.y * blockDim.y) {
            const int c = AXIS == 0 ? y : AXIS == 1 ? z : x;
            const long long i = ((long long)y * nz + z) * nx + x;
            if (mask && masked(mg, x, y, z, nx, ny, nz)) {
                out[i] = 0.f;
                continue;
            }
            const float *line = in + (i - c * stride);
            double acc = (double)line[c * stride] * taps.w[0];
            if (n >= r) {
#pragma unroll 4
                for (int j = r; j >= 1; --j)
                    acc += ((double)line[reflect_once(c - j, n) * stride] +
                            (double)line[reflect_once(c + j, n) * stride]) * taps.w[j];
            } else {
                for (int j = r; j >= 1; --j)
                    acc += ((double)line[reflect_index(c - j, n) * stride] +
                            (double)line[reflect_index(c + j, n) * stride]) * taps.w[j];
            }
            out[i] = (float)acc;
        }
}

// All three passes for radius 4 on lines of at least 4 cells (σ = 1 with scipy's truncate,
// the driver's rule).  A block makes 64 x TZ x 8 cells (x, z, y): its columns of 16 values
// along y from memory, 8 sums of each into LDS with the 4 cells on either side in x and z,
// then the z sums in place (a column of a plane belongs to one thread) and the x sums,
// four a thread, to memory.  An image is read 2·(TZ + 8)/TZ·72/64 times, mostly from the
// caches, and written once; three passes moved 8 bytes a cell each and paid three launches
// of about 4 us.  200x200x100 under the driver's margins: 37.4 us in
// three passes (13.9 + 10.5 + 13), 24 here, bound by the double sums (about 17 operations
// for each of 3.1 sums a cell; 16 rows a tile halve the surplus but leave fewer waves: 28).
constexpr int kTX = 64, kTY = 8, kTZ = 8, kR4 = 4, kGaussThreads = 576;
__global__ __launch_bounds__(kGaussThreads) void k_gauss4(const float *__restrict__ in, float *__restrict__ out,
                                                          int nx, int ny, int nz, int ntx, int ntz, GaussTaps taps,
                                                          Margins mg) {
    constexpr int W = kTX + 2 * kR4, D = kTZ + 2 * kR4, M = kTY + 2 * kR4;
    __shared__ __attribute__((aligned(16))) float A[kTY][D][W];
    const int tile = blockIdx.x, tx = tile % ntx, tz = tile / ntx % ntz, ty = tile / (ntx * ntz);
    const int x0 = tx * kTX, z0 = tz * kTZ, y0 = ty * kTY;
    const long long plane = (long long)nx * nz;
    // a tile the mask covers is only cleared
    const bool clear = x0 + kTX <= mg.xl || x0 >= nx - mg.xh || y0 + kTY <= mg.yl || y0 >= ny - mg.yh ||
                       z0 + kTZ <= mg.zl || z0 >= nz - mg.zh;
    for (int k = threadIdx.x; !clear && k < D * W; k += kGaussThreads) {
        const int zr = k / W, xr = k - zr * W;
        const int x = reflect_once(min(x0 + xr - kR4, nx - 1 + kR4), nx);
        const int z = reflect_once(min(z0 + zr - kR4, nz - 1 + kR4), nz);
        const float *p = in + ((long long)z * nx + x);
        float v[M];
#pragma unroll
        for (int j = 0; j < M; ++j) v[j] = p[reflect_once(min(y0 + j - kR4, ny - 1 + kR4), ny) * plane];
#pragma unroll
        for (int j = 0; j < kTY; ++j) A[j][zr][xr] = gauss_sum<kR4>(v + j, taps);
    }
    __syncthreads();
    for (int k = threadIdx.x; !clear && k < kTY * W; k += kGaussThreads) {
        const int y = k / W, xr = k - y * W;
        float v[D];
#pragma unroll
        for (int j = 0; j < D; ++j) v[j] = A[y][j][xr];
#pragma unroll
        for (int j = 0; j < kTZ; ++j) A[y][j][xr] = gauss_sum<kR4>(v + j, taps);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kTY * kTZ * (kTX / 4); k += kGaussThreads) {
        const int q = k % (kTX / 4), zr = k / (kTX / 4) % kTZ, yr = k / (kTX / 4 * kTZ);
        const int x = x0 + 4 * q, y = y0 + yr, z = z0 + zr;
        if (x >= nx || y >= ny || z >= nz) continue;
        float v[4 + 2 * kR4], o[4];
#pragma unroll
        for (int j = 0; j < 4 + 2 * kR4; j += 4)
            *reinterpret_cast<float4 *>(v + j) = *reinterpret_cast<const float4 *>(&A[yr][zr][4 * q + j]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            o[j] = masked(mg, x + j, y, z, nx, ny, nz) ? 0.f : gauss_sum<kR4>(v + j, taps);
        float *d = out + (y * plane + (long long)z * nx + x);
        if (x + 4 <= nx) {
            *reinterpret_cast<f32x4u *>(d) = f32x4u{o[0], o[1], o[2], o[3]};
        } else {
            for (int j = 0; j < nx - x; ++j) d[j] = o[j];
        }
    }
}

__global__ void k_mask_copy(const float *__restrict__ in, float *__restrict__ out, int nx, int ny,
                            int nz, Margins mg) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long N = (long long)nx * ny * nz;
    if (i >= N) return;
    const int x = (int)(i % nx);
    const int z = (int)((i / nx) % nz);
    const int y = (int)(i / ((long long)nx * nz));
    out[i] = masked(mg, x, y, z, nx, ny, nz) ? 0.f : in[i];
}

// Model.compute_Rho (M:1204-1206) in the reference's float32 numpy arithmetic:
// v = vp/1e3, the five terms each a float32 product with the powers of v
// (v² as v·v, v³..v⁵ rounded once from exact double products, as a correctly
// rounded powf gives), summed left to right in float32, times 1e3.
__device__ __forceinline__ float nafe_drake_f32(float vp) {
#pragma clang fp contract(off)
    const float v = vp / 1000.0f;
    const double vd = (double)v;
    const float v2 = v * v;
    const float v3 = (float)(vd * vd * vd);
    const float v4 = (float)((vd * vd) * (vd * vd));
    const float v5 = (float)((vd * vd) * (vd * vd) * vd);
    float r = 1.6612f * v - 0.4712f * v2;
    r = r + 0.0671f * v3;
    r = r - 0.0043f * v4;
    r = r + 0.000106f * v5;
    return r * 1000.0f;
}

// lam = f32(lam0 + α_λ·dlam), mu likewise (double, one rounding: the
// reference's float32 model plus a float64 step); vp, vs from (lam, mu, rho_in) in
// float32 (compute_Vp_Vs); rho = Nafe-Drake(vp) (compute_Rho) except at
// z < top, where rho_keep is kept.
__global__ void k_model_update(const float *lam0, const float *dlam, double alam, const float *mu0,
                               const float *dmu, double amu, const float *rho_in,
                               const float *rho_keep, int top, int nx, int nz, long long N,
                               float *lam, float *mu, float *vp, float *vs, float *rho) {
#pragma clang fp contract(off)
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const float L = dlam ? (float)((double)lam0[i] + alam * (double)dlam[i]) : lam0[i];
    const float M = dmu ? (float)((double)mu0[i] + amu * (double)dmu[i]) : mu0[i];
    const float R = rho_in[i];
    const float p = sqrtf((L + 2.0f * M) / R);
    const float s = sqrtf(M / R);
    lam[i] = L;
    mu[i] = M;
    vp[i] = p;
    vs[i] = s;
    if (rho) {
        const int z = (int)((i / nx) % nz);
        if (z < top && rho_keep) {
            rho[i] = rho_keep[i];
        } else {
            rho[i] = nafe_drake_f32(p);
        }
    }
}

__global__ void k_rho_nafe_drake(const float *vp, float *rho, long long n) {
#pragma clang fp contract(off)
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    rho[i] = nafe_drake_f32(vp[i]);
}

__global__ void k_axpy(float a, const float *x, float *y, long long n) {
#pragma clang fp contract(off)
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = y[i] + a * x[i];
}

// Cross-correlation residual (computeResidualCrossCorrelation, M:2145-2179).  A
// block takes G receivers of one (shot, component): thread (t, r) = (tid / G, tid % G)
// walks every (threads / G)-th sample, the three sums of a trace (in double) are
// reduced over its threads, and a second walk writes the residual (its reads come
// from the caches).  J += the traces' 1 - a/(|m||o|), one atomic per block.  One
// thread per trace walking all its samples left 48 wavefronts for 16 shots' 3072 traces
// and waited for memory 5000 times in a row: 1540 us for 16 x 2500 samples x 64
// receivers, where the bytes need 19; now 39 (two walks, the second from the caches).
constexpr int kXcorrThreads = 1024;
__global__ __launch_bounds__(kXcorrThreads) void k_xcorr(const float *__restrict__ mod,
                                                         const float *__restrict__ obs,
                                                         float *__restrict__ res, double *J, int ntmax,
                                                         int nrec, int G, long long nsc, long long nblk) {
    __shared__ double part[3][kXcorrThreads];
    const int tid = threadIdx.x, rl = tid & (G - 1);
    const int t0 = tid / G, dt = kXcorrThreads / G;
    const int ngr = (nrec + G - 1) / G;
    for (long long blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
        // workgroups are dealt to the 8 XCDs in turn: an XCD takes all receiver groups of a
        // (shot, component), which share cache lines
        const long long q = (blk >> 3) / ngr, sc = 8 * q + (blk & 7);
        if (sc >= nsc) continue;
        const long long r = ((blk >> 3) - q * ngr) * G + rl;
        const long long base = sc * ntmax * nrec + r;
        const bool on = r < nrec;
        double mm = 0.0, oo = 0.0, mo = 0.0;
        if (on) {
#pragma unroll 8
            for (int t = t0; t < ntmax; t += dt) {
                const double m = mod[base + (long long)t * nrec], o = obs[base + (long long)t * nrec];
                mm += m * m;
                oo += o * o;
                mo += m * o;
            }
        }
        part[0][tid] = mm; part[1][tid] = oo; part[2][tid] = mo;
        __syncthreads();
        for (int w = kXcorrThreads / 2; w >= G; w >>= 1) {
            if (tid < w)
                for (int k = 0; k < 3; ++k) part[k][tid] += part[k][tid + w];
            __syncthreads();
        }
        mm = part[0][rl]; oo = part[1][rl]; mo = part[2][rl];
        double nm = sqrt(mm), no = sqrt(oo);
        if (nm == 0.0) nm = 1.0;
        if (no == 0.0) no = 1.0;
        const double ag = mo == 0.0 ? 1.0 : mo;
        const double k1 = ag / (no * nm * nm * nm), k2 = 1.0 / (nm * no);
        __syncthreads();
        if (tid < G) part[0][tid] = on ? 1.0 - mo / (nm * no) : 0.0;
        __syncthreads();
        if (tid == 0) {
            double sum = 0.0;
            for (int k = 0; k < G; ++k) sum += part[0][k];
            atomicAdd(J, sum);
        }
        if (on) {
#pragma unroll 8
            for (int t = t0; t < ntmax; t += dt) {
                const long long i = base + (long long)t * nrec;
                res[i] = (float)((double)mod[i] * k1 - (double)obs[i] * k2);
            }
        }
        __syncthreads();
    }
}

static inline unsigned nblocks(long long n) { return (unsigned)((n + 255) / 256); }

}  // namespace efm

using namespace efm;

extern "C" int efm_condition_gradient(const EfmSmooth *p, int nx, int ny, int nz, const float *in,
                                      float *out, float *work, void *stream) {
    if (!p || !in || !out) return fail(EFM_E_ARG, "efm_condition_gradient: null argument");
    if (nx < 1 || ny < 1 || nz < 1) return fail(EFM_E_ARG, "efm_condition_gradient: empty volume");
    if (in == out) return fail(EFM_E_ARG, "efm_condition_gradient: in and out must differ");
    if (!(p->sigma >= 0.f) || !(p->truncate >= 0.f))
        return fail(EFM_E_ARG, "efm_condition_gradient: sigma and truncate must be >= 0");
    for (int k = 0; k < 6; ++k)
        if (p->margin[k] < 0) return fail(EFM_E_ARG, "efm_condition_gradient: negative margin");
    const long long N = (long long)nx * ny * nz;
    const Margins mg{p->margin[0], p->margin[1], p->margin[2], p->margin[3], p->margin[4],
                     p->margin[5]};
    hipStream_t st = (hipStream_t)stream;
    // scipy: radius = int(truncate·σ + 0.5); no filtering when σ is (nearly) zero
    const int r = p->sigma > 1e-15f ? (int)((double)p->truncate * (double)p->sigma + 0.5) : 0;
    if (r > kMaxRadius) return fail(EFM_E_UNSUPPORTED, "efm_condition_gradient: kernel radius above 64");
    if (p->sigma <= 1e-15f || r == 0) {
        // a radius-0 Gaussian is the identity (its single weight normalises to 1)
        hipLaunchKernelGGL(k_mask_copy, dim3(nblocks(N)), dim3(256), 0, st, in, out, nx, ny, nz, mg);
        return check_launch("gradient mask");
    }
    if (!work || work == in || work == out)
        return fail(EFM_E_ARG, "efm_condition_gradient: a separate work volume is required");
    GaussTaps taps{};
    taps.r = r;
    // scipy.ndimage._gaussian_kernel1d: exp(-x²/(2σ²)) over x = -r..r, normalised
    const double s2 = (double)p->sigma * (double)p->sigma;
    double phi[2 * kMaxRadius + 1], sum = 0.0;
    for (int j = -r; j <= r; ++j) sum += (phi[j + r] = std::exp(-0.5 / s2 * (double)j * (double)j));
    for (int j = 0; j <= r; ++j) taps.w[j] = phi[j + r] / sum;
    const Margins none{0, 0, 0, 0, 0, 0};
    if (r == kR4 && nx >= r && ny >= r && nz >= r) {
        const long long ntx = (nx + kTX - 1) / kTX, ntz = (nz + kTZ - 1) / kTZ, nty = (ny + kTY - 1) / kTY;
        if (ntx * ntz * nty <= (long long)UINT32_MAX / kGaussThreads) {
            hipLaunchKernelGGL(k_gauss4, dim3((unsigned)(ntx * ntz * nty)), dim3(kGaussThreads), 0, st, in, out, nx, ny,
                               nz, (int)ntx, (int)ntz, taps, mg);
            return check_launch("gaussian smoothing");
        }
    }
    auto pass = [&](auto kernel, const float *src, float *dst, int mask, const Margins &m, const char *what) {
        // rows of 32 lanes where that leaves fewer of them idle than 64
        const int bx = (nx + 31) / 32 % 2 ? 32 : 64, bz = 256 / bx;
        hipLaunchKernelGGL(kernel, dim3((nx + bx - 1) / bx, std::min((nz + bz - 1) / bz, 65535), std::min(ny, 65535)),
                           dim3(bx, bz), 0, st, src, dst, nx, ny, nz, taps, mask, m);
        return check_launch(what);
    };
    if (int rc = pass(k_gauss_pass<0>, in, out, 0, none, "gaussian pass y")) return rc;
    if (int rc = pass(k_gauss_pass<1>, out, work, 0, none, "gaussian pass z")) return rc;
    return pass(k_gauss_pass<2>, work, out, 1, mg, "gaussian pass x");
}

extern "C" int efm_model_update(const float *lam0, const float *dlam, double alpha_lam,
                                const float *mu0, const float *dmu, double alpha_mu,
                                const float *rho_in,
                                const float *rho_keep, int top, int nx, int ny, int nz, float *lam,
                                float *mu, float *vp, float *vs, float *rho, void *stream) {
    if (!lam0 || !mu0 || !rho_in || !lam || !mu || !vp || !vs)
        return fail(EFM_E_ARG, "efm_model_update: null argument");
    if (nx < 1 || ny < 1 || nz < 1 || top < 0) return fail(EFM_E_ARG, "efm_model_update: bad size");
    if (rho && (rho == rho_in || (rho_keep && rho == rho_keep)))
        return fail(EFM_E_ARG, "efm_model_update: rho must not alias rho_in or rho_keep");
    const long long N = (long long)nx * ny * nz;
    hipLaunchKernelGGL(k_model_update, dim3(nblocks(N)), dim3(256), 0, (hipStream_t)stream, lam0,
                       dlam, alpha_lam, mu0, dmu, alpha_mu, rho_in, rho_keep, top, nx, nz, N, lam, mu, vp, vs, rho);
    return check_launch("model update");
}

extern "C" int efm_model_rho_nafe_drake(const float *vp, float *rho, long long n, void *stream) {
    if (!vp || !rho || n < 0) return fail(EFM_E_ARG, "efm_model_rho_nafe_drake: bad argument");
    if (n == 0) return EFM_OK;
    hipLaunchKernelGGL(k_rho_nafe_drake, dim3(nblocks(n)), dim3(256), 0, (hipStream_t)stream, vp, rho, n);
    return check_launch("rho nafe-drake");
}

extern "C" int efm_volume_axpy(float a, const float *x, float *y, long long n, void *stream) {
    if (!x || !y || n < 0) return fail(EFM_E_ARG, "efm_volume_axpy: bad argument");
    if (n == 0) return EFM_OK;
    hipLaunchKernelGGL(k_axpy, dim3(nblocks(n)), dim3(256), 0, (hipStream_t)stream, a, x, y, n);
    return check_launch("axpy");
}

extern "C" int efm_xcorr_residual(const float *mod, const float *obs, float *res, double *J,
                                  int nshot, int ntmax, int nrec, void *stream) {
    if (nshot < 0 || ntmax < 0 || nrec < 0) return fail(EFM_E_ARG, "efm_xcorr_residual: bad size");
    const long long ntr = 3LL * nshot * nrec;
    if (ntr == 0 || ntmax == 0) return EFM_OK;
    if (!mod || !obs || !res || !J) return fail(EFM_E_ARG, "efm_xcorr_residual: null argument");
    // 8 receivers to a block: enough blocks for the chip at a few shots, and 128 samples of a
    // trace in flight at a time
    int G = 8;
    while (G > 1 && G / 2 >= nrec) G /= 2;
    const long long nsc = 3LL * nshot, nblk = (nsc + 7) / 8 * 8 * ((nrec + G - 1) / G);
    hipLaunchKernelGGL(k_xcorr, dim3((unsigned)std::min(nblk, 1LL << 20)), dim3(kXcorrThreads), 0, (hipStream_t)stream,
                       mod, obs, res, J, ntmax, nrec, G, nsc, nblk);
    return check_launch("cross-correlation residual");
}
