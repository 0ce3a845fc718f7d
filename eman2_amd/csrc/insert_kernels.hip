// Fourier-space gridding kernels of the "fourier" reconstructor path.
//
// Per-pixel semantics restate FourierReconstructor::do_insert_slice_work
// (libEM/reconstructor.cpp:1122-1210), FourierInserter3DMode2 / Mode2l
// ::insert_pixel (libEM/reconstructor_tools.cpp:128-239), Util::fast_exp /
// hypot3sq (libEM/util.cpp:788-800, util.h:816-819) and
// EMData::add_complex_at_fast (libEM/emdata_core.h:368-413).  The float
// arithmetic of coordinates and weights is evaluated in the reference's
// order with contraction off, so a weight is the reference's bit for bit; the
// brick scatters fuse a value's last product into its FP32 sum, and the order
// of the sums differs.  The 6-cell Gaussians multiply value and weight first
// and take gauss_var's width by Newton steps (k_scatter_gauss6).
//
//  k_insert_corners  one launch per (slice, symmetry op), one thread per pixel
//                    and corner, global atomics per contribution (the plain
//                    form; k_insert_plain for the wide modes).
//  k_bin_*           bins (slice, brick) pairs over the unfolded frequency
//                    grid [-P/2, P/2]^3 cut into 8^3 bricks, keyed by brick
//                    and the slice's dominant normal axis.
//  k_scatter_insert  one wave per work item holds the brick's accumulator in
//                    LDS and adds the stencils of the slice pixels reaching
//                    the brick with plain read-modify-writes (lanes sharing
//                    a stencil origin take turns, elected by an LDS tag).
//                    Each item writes its partial brick to HBM.
//  k_reduce_items    the items of a brick summed into its first one, where
//                    the batch has an item per brick of the grid or more.
//  k_merge_partials  one thread per half-volume voxel sums the partial
//                    bricks of its unfolded source cells under the Hermitian
//                    fold of add_complex_at_fast and adds them with plain
//                    stores (each voxel has one owner: no atomics).
#pragma clang fp contract(off)
#include <climits>
#include "fh_device.hpp"

namespace fh {

#define EXPN 400  // fast_exp entries reachable by a 2x2x2 stencil (r^2 <= 3)

__device__ __forceinline__ void gadd(float *p, float v) { unsafeAtomicAdd(p, v); }

// ------------------------------------------------------------ compose
// t3d[q] = R[p] * S[s] with q = p*nsym + s (Transform operator*,
// libEM/transform.cpp:1384-1395, FP32 in source order).
__global__ void k_compose(const float *__restrict__ rots, const float *__restrict__ weights, int n,
                          const float *__restrict__ syms, int nsym, float *__restrict__ t3d,
                          float *__restrict__ wq)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n * nsym) return;
    const int p = q / nsym, s = q - p * nsym;
    const float *a = rots + 9 * (size_t)p;
    const float *b = syms + 9 * s;
    float *r = t3d + 9 * (size_t)q;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) r[3 * i + j] = a[3 * i + 0] * b[0 * 3 + j] + a[3 * i + 1] * b[1 * 3 + j] + a[3 * i + 2] * b[2 * 3 + j];
    wq[q] = weights[p];
}

// The "xform" processor's resampling (xform_sample) of n particles (edge means or null) into P x P images.
__global__ void __launch_bounds__(256) k_xform2d(const float *__restrict__ imgs, int B, int P, int off,
                                                 const float *__restrict__ means, const float *__restrict__ xf,
                                                 float *__restrict__ out)
{
    const int p = blockIdx.y;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= P * P) return;
    const int i = idx % P, j = idx / P;
    out[(size_t)p * P * P + idx] =
        xform_sample(imgs + (size_t)p * B * B, B, P, off, means ? means[p] : 0.f, xf + 6 * (size_t)p, i, j);
}

hipError_t launch_xform2d(const float *imgs, int n, int B, int P, const float *means, const float *xf, float *out,
                          hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const int d = B - P;
    const int fl = d >= 0 ? d / 2 : -((-d + 1) / 2);  // clip_inplace Region((B-P)//2, ...)
    hipLaunchKernelGGL(k_xform2d, dim3((P * P + 255) / 256, n), dim3(256), 0, s, imgs, B, P, -fl, means, xf, out);
    return hipGetLastError();
}

hipError_t launch_compose(const float *rots, const float *weights, int n, const float *syms, int nsym,
                          float *t3d, float *wq, hipStream_t s)
{
    const int tot = n * nsym;
    if (tot <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_compose, dim3((tot + 255) / 256), dim3(256), 0, s, rots, weights, n, syms, nsym, t3d, wq);
    return hipGetLastError();
}

// ------------------------------------------------------------ per-pixel math
// (rx, ry, 0) * t3d, then x (nx-2, ny, nz) = P (libEM/reconstructor.cpp:1171-1196)
__device__ __forceinline__ void pixel_coords(int x, int y, const float *m, const float *rtab, int H, float Pf,
                                             float &xx, float &yy, float &zz)
{
    const float rx = rtab[x + H], ry = rtab[y + H];
    xx = (rx * m[0] + ry * m[3]) * Pf;
    yy = (rx * m[1] + ry * m[4]) * Pf;
    zz = (rx * m[2] + ry * m[5]) * Pf;
}

// slice.get_complex_at(x, y) for x >= 0 (libEM/emdata_core.cpp:126-132);
// the x=0, y<0 pixel is read as the conjugate of (0, -y).
__device__ __forceinline__ float2 slice_value(const float2 *__restrict__ S, int x, int y, int P, int H)
{
    const bool cj = x == 0 && y < 0;
    const int row = cj ? -y : (y < 0 ? P + y : y);
    float2 v = S[row * (H + 1) + x];  // P (P/2 + 1) < 2^31
    if (cj) v.y = -v.y;
    return v;
}

// gauss_2 / trilinear weight of corner (i,j,k) for a pixel at (xx,yy,zz).
__device__ __forceinline__ float corner_weight(int mode, int i, int j, int k, float xx, float yy, float zz, float h,
                                               float weight, const float *etab)
{
    const float dx = (float)i - xx, dy = (float)j - yy, dz = (float)k - zz;
    if (mode == 0) {
        const float r = dx * dx + dy * dy + dz * dz;  // Util::hypot3sq
        const float f = r * h;                          // -(-r*h)
        const int g = (int)__builtin_fma((double)f, 50.0, 0.5);  // Util::fast_exp index: f*50 is exact in double
        return etab[g] * weight;
    }
    return (float)((1.0 - (double)fabsf(dx)) * (1.0 - (double)fabsf(dy)) * (1.0 - (double)fabsf(dz)) *
                   (double)weight);
}

__device__ __forceinline__ size_t cidx(int xs, int ys, int zs, int P, int H)
{
    return ((size_t)zs * P + ys) * (size_t)(H + 1) + xs;
}

// EMData::add_complex_at_fast with the weight update norm[off/2] += gg of
// insert_pixel, as device atomics.  (x,y,z) unfolded, value v, weight gg.
__device__ __forceinline__ void add_complex_atomic(float2 *data, float *norm, int P, int H, int x, int y, int z,
                                                   float vr, float vi, float gg)
{
    if (abs(x) >= H + 1 || abs(y) > H || abs(z) > H) return;
    float *d = reinterpret_cast<float *>(data);
    const int wy = y < 0 ? P + y : y, wz = z < 0 ? P + z : z;
    const int ny = y <= 0 ? -y : P - y, nz = z <= 0 ? -z : P - z;
    if (x == 0) {
        if (y == 0 && z == 0) {
            gadd(&d[0], vr);
            d[1] = 0.f;
            gadd(&norm[0], gg);
            return;
        }
        const size_t i2 = cidx(0, ny, nz, P, H);
        gadd(&d[2 * i2], vr);
        gadd(&d[2 * i2 + 1], -vi);
    }
    if (abs(x) == H) {
        if (y == 0 && z == 0) {
            gadd(&d[2 * H], vr);
            d[2 * H + 1] = 0.f;
            gadd(&norm[H], gg);
            return;
        }
        const size_t i2 = cidx(H, ny, nz, P, H);
        gadd(&d[2 * i2], vr);
        gadd(&d[2 * i2 + 1], -vi);
    }
    if (x < 0) {
        const size_t i = cidx(-x, ny, nz, P, H);
        gadd(&d[2 * i], vr);
        gadd(&d[2 * i + 1], -vi);
        gadd(&norm[i], gg);
        return;
    }
    const size_t i = cidx(x, wy, wz, P, H);
    gadd(&d[2 * i], vr);
    gadd(&d[2 * i + 1], vi);
    gadd(&norm[i], gg);
}

// ------------------------------------------------------------ other inserter modes
// Util::fast_exp (util.cpp:788-800) with its full 1000-entry table
__device__ __forceinline__ float fast_exp_full(float f, const float *__restrict__ etab)
{
    return (f > 0 || f < -19.98) ? expf(f) : etab[(int)(-(double)f * 50.0 + 0.5)];
}

// e^-|x| I0(x), the exponentially scaled modified Bessel function of order 0
// that kaiser_bessel takes from GSL (gsl_sf_bessel_i0_scaled): the
// polynomial approximations of Abramowitz & Stegun 9.8.1 (|x| <= 3.75,
// |error| < 1.6e-7 of I0) and 9.8.2 (x > 3.75, |error| < 1.9e-7 of
// sqrt(x) e^-x I0(x)), evaluated in double.
__host__ __device__ inline double bessel_i0_scaled(double x)
{
    const double ax = fabs(x);
    if (ax <= 3.75) {
        const double t = (ax / 3.75) * (ax / 3.75);
        const double i0 = 1.0 + t * (3.5156229 + t * (3.0899424 + t * (1.2067492 + t * (0.2659732 +
                          t * (0.0360768 + t * 0.0045813)))));
        return i0 * exp(-ax);
    }
    const double u = 3.75 / ax;
    return (0.39894228 + u * (0.01328592 + u * (0.00225319 + u * (-0.00157565 + u * (0.00916281 +
            u * (-0.02057706 + u * (0.02635537 + u * (-0.01647633 + u * 0.00392377)))))))) / sqrt(ax);
}

// The inserters the brick scatter does not take, in the global-atomic form
// (libEM/reconstructor_tools.cpp):
//   mode 2 gauss_var (Mode6, :382-433): 6x6x6 stencil from floor(p - 2.5),
//     h = 1 / (|p|^2 / 4000 + 0.15) at least 0.1, weight fast_exp(-r h) w;
//   mode 3 gauss_5 (Mode5): the same stencil with h = 1 / I5G;
//   mode 4 nearest_neighbor (Mode1, :113-126): the voxel floor(p + 0.5);
//   mode 5 gauss_3 (Mode3): 3x3x3 from floor(p - 0.5), h = 32 / ((8 + |p|) I3G),
//     weight fast_exp(-r h) w / (1 + 6 e^-h + 12 e^-2h + 8 e^-3h);
//   mode 10 fourier_iter (FourierIterReconstructor::insert_slice,
//     libEM/reconstructor.cpp:520-637): gauss_var's stencil and width with x
//     clamped to |x| <= P/2 - 1 (nx2 = nx/2 - 2); mode 11 the same
//     reconstructor with a reference volume: value dt + ref(i,j,k) -
//     trilinear ref(p), h = 1/2, cells inside i^2 + j^2 + k^2 <= P^2/4.
// Stencils are clamped to [-P/2, P/2] per axis; subnormal weights are
// dropped (flush-to-zero: the reference's -ffast-math build and the float
// atomics do not keep them).
__device__ void insert_wide(int mode, float2 dt, float xx, float yy, float zz, float w, int P, int H,
                            const float *__restrict__ etab, float2 *data, float *norm, const float2 *ref);

// ------------------------------------------------------------ plain form
// Util::hypot_fast_int(x, y) (libEM/util.cpp:764-785): round(hypot(x, y)),
// exact for 0 <= x^2 + y^2 < 2^24 (sqrt of an integer is never a half-integer).
__device__ __forceinline__ int hypot_int(int x, int y)
{
    const int n = x * x + y * y;
    int r = (int)__builtin_amdgcn_sqrtf((float)n);
    r -= (r * r > n);
    r += ((r + 1) * (r + 1) <= n);
    return r + (n > r * r + r);
}

// The wide modes: one thread per pixel.
__global__ void __launch_bounds__(256) k_insert_plain(const float2 *__restrict__ S, InsertConst c, Mat9 m,
                                                      float weight, float2 *data, float *norm,
                                                      const float *__restrict__ exptab,
                                                      const float *__restrict__ rtab_g,
                                                      const float *__restrict__ rw)
{
    const int H = c.H, P = c.P;
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = (int)blockIdx.y - H;
    if (x > H) return;
    if (!c.corners && x * x + y * y > c.rcut * c.rcut + c.rcut) return;  // hypot_fast_int(x,y) > rcut
    // class_ssnr weighting (reconstructor.cpp:1170-1184): the weight of radius r
    if (rw) weight = rw[hypot_int(x, y)];
    float xx, yy, zz;
    pixel_coords(x, y, m.m, rtab_g, H, c.Pf, xx, yy, zz);
    insert_wide(c.mode, slice_value(S, x, y, P, H), xx, yy, zz, weight, P, H, exptab, data, norm, c.ref);
}

// gauss_2 and trilinear: one thread per (pixel, corner), 32 pixels of a row
// per block.  One slice is bound by latency: with a thread per pixel each
// corner's table read waited for the atomics of the corner before it: 10.3 us
// for a slice of pad 96, 33 at 256 and 171 at 600, now 6.8, 21 and 98.
__global__ void __launch_bounds__(256) k_insert_corners(const float2 *__restrict__ S, InsertConst c, Mat9 m,
                                                        float weight, float2 *data, float *norm,
                                                        const float *__restrict__ exptab,
                                                        const float *__restrict__ rtab_g,
                                                        const float *__restrict__ rw)
{
    const int H = c.H, P = c.P;
    const int x = blockIdx.x * 32 + (threadIdx.x >> 3), corner = threadIdx.x & 7;
    const int y = (int)blockIdx.y - H;
    if (x > H) return;
    if (!c.corners && x * x + y * y > c.rcut * c.rcut + c.rcut) return;  // hypot_fast_int(x,y) > rcut
    // class_ssnr weighting (reconstructor.cpp:1170-1184): the weight of radius r
    if (rw) weight = rw[hypot_int(x, y)];
    float xx, yy, zz;
    pixel_coords(x, y, m.m, rtab_g, H, c.Pf, xx, yy, zz);
    const int x0 = (int)floorf(xx), y0 = (int)floorf(yy), z0 = (int)floorf(zz);
    if (x0 < -H - 1 || y0 < -H - 1 || z0 < -H - 1 || x0 > H || y0 > H || z0 > H) return;
    const float2 dt = slice_value(S, x, y, P, H);
    const int i = x0 + (corner & 1), j = y0 + ((corner >> 1) & 1), k = z0 + (corner >> 2);
    const float gg = corner_weight(c.mode, i, j, k, xx, yy, zz, c.h, weight, exptab);
    add_complex_atomic(data, norm, P, H, i, j, k, dt.x * gg, dt.y * gg, gg);
}

// The plain (global-atomic) form over every slice of a batch in one launch:
// block (xb, q) covers pixels x in [64 xb, 64 xb + 64) of rows y of slice q
// = p nsym + s, with t3d[q] and weight wq[q] (or the particle's class_ssnr
// radial weights).  For the wide modes where a batch has more tiles than a grid
// of k_insert_wide_tiles holds (2^31).
__global__ void __launch_bounds__(64) k_insert_plain_batch(const float2 *__restrict__ slices, int nsym, int nxb,
                                                           const float *__restrict__ t3d, const float *__restrict__ wq,
                                                           InsertConst c, float2 *data, float *norm,
                                                           const float *__restrict__ exptab,
                                                           const float *__restrict__ rtab_g,
                                                           const float *__restrict__ rw)
{
    const int H = c.H, P = c.P;
    const int q = blockIdx.x / nxb;
    const int x = (blockIdx.x - q * nxb) * 64 + threadIdx.x;
    const int y = (int)blockIdx.y - H;
    const float wgt = wq[q];
    if (x > H || wgt == 0.0f) return;
    if (!c.corners && x * x + y * y > c.rcut * c.rcut + c.rcut) return;  // hypot_fast_int(x,y) > rcut
    const int p = q / nsym;
    const float weight = rw ? rw[(size_t)p * (H + 1) + hypot_int(x, y)] : wgt;
    const float2 *S = slices + (size_t)p * P * (H + 1);
    const float *m = t3d + 9 * (size_t)q;
    float xx, yy, zz;
    pixel_coords(x, y, m, rtab_g, H, c.Pf, xx, yy, zz);
    insert_wide(c.mode, slice_value(S, x, y, P, H), xx, yy, zz, weight, P, H, exptab, data, norm, c.ref);
}

// The wide modes with LDS accumulation: a workgroup takes an 8 x 8 tile of
// one slice's pixels (4 threads per pixel, 54 of the 216 stencil cells each),
// adds every contribution into an LDS window of 17^3 unfolded cells with LDS
// float atomics, then adds each touched cell to the volume once through the
// add_complex_at_fast fold (global atomics): about ten times fewer global
// atomics than one per contribution.  Each contribution's value and weight
// are computed exactly as in insert_wide.  Across an 8 x 8 tile a pixel
// coordinate moves by at most 7 sqrt 2 (orthonormal slice axes), so the
// stencil origins of a tile span at most 10 cells per axis and the stencils
// 10 + (n - 1) cells for an n-cell stencil: within the 17-cell window for
// n <= 7 (gauss_var, gauss_5, gauss_3, kaiser_bessel, gridding_5,
// gridding_7); kaiser_bessel_derived's 9-cell stencil can reach 18, and the
// cells of a tile beyond the window go straight to the volume with global
// atomics (same result, less of the window's saving).  The window (59 KB)
// and the pixel records stay within 64 KB of LDS per workgroup.
constexpr int WT_TILE = 8;
constexpr int WT_WIN = 17;
constexpr int WT_CELLS = WT_WIN * WT_WIN * WT_WIN;

// gridding_5 / gridding_7 kernels, 3x oversampled (reconstructor_tools.cpp:455, :817)
#include "gridding_tables.inc"
__constant__ float c_grid5[9 * 9 * 9] = {FH_GRIDDING5_VALUES};
__constant__ float c_grid7[12 * 12 * 12] = {FH_GRIDDING7_VALUES};

// Util::fast_floor (libEM/util.h:874-880): one less than floor at negative integers
__device__ __forceinline__ int ref_fast_floor(float x) { return x < 0 ? (int)x - 1 : (int)x; }

// table index of one axis: |fast_floor((i - p) * 3 + 0.5)|, the 0.5 added in double as in the reference
__device__ __forceinline__ int grid_index(int i, float p, int n)
{
    const int t = abs(ref_fast_floor((float)((double)(((float)i - p) * 3.0f) + 0.5)));
    return min(t, n - 1);  // <= n - 1 for every finite p (the stencil spans |i - p| <= n / 3 - 0.5)
}

struct WidePix {
    float xx, yy, zz, dre, dim, w, h, ww;
    float nre, nim;        // fourier_iter with a reference: the reference trilinear at p
    int lo[3], hi[3];      // stencil cells, clamped to the volume
    int a[3];              // stencil origin before the clamp
    int H;
    const float2 *ref;
};

// EMData::get_complex_at(x, y, z) of a reference volume in the reconstructor's
// layout (libEM/emdata_core.cpp:135-144): 0 outside, conjugate for x < 0
__device__ __forceinline__ float2 ref_get(const float2 *__restrict__ ref, int x, int y, int z, int H)
{
    const int P = 2 * H;
    if (abs(x) >= H + 1 || abs(y) > H || abs(z) > H) return make_float2(0.f, 0.f);
    if (x < 0) {
        const float2 v = ref[cidx(-x, y <= 0 ? -y : P - y, z <= 0 ? -z : P - z, P, H)];
        return make_float2(v.x, -v.y);
    }
    return ref[cidx(x, y < 0 ? P + y : y, z < 0 ? P + z : z, P, H)];
}

// Util::trilinear_interpolate_complex (libEM/util.h:645-654) of a reference volume at floor(p)
__device__ __forceinline__ void ref_trilinear(const float2 *__restrict__ ref, float xx, float yy, float zz, int H,
                                              float &re, float &im)
{
    const float xx0 = floorf(xx), yy0 = floorf(yy), zz0 = floorf(zz);
    const int x0 = (int)xx0, y0 = (int)yy0, z0 = (int)zz0;
    const float t = xx - xx0, u = yy - yy0, v = zz - zz0;
    re = im = 0.f;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const float2 q = ref_get(ref, x0 + (c & 1), y0 + ((c >> 1) & 1), z0 + (c >> 2), H);
        const float a = (c & 1) ? t : 1 - t, b = (c & 2) ? u : 1 - u, e = (c & 4) ? v : 1 - v;
        const float wc = a * b * e;
        if (c == 0) {
            re = wc * q.x;
            im = wc * q.y;
        } else {
            re = re + wc * q.x;
            im = im + wc * q.y;
        }
    }
}

// stencil range (clamped to [-P/2, P/2]) and width of one pixel; false if the
// reference's range check rejects it (insert_wide's first half)
__device__ __forceinline__ bool wide_setup(int mode, float xx, float yy, float zz, float w, int H,
                                           const float *__restrict__ etab, WidePix &px,
                                           const float2 *ref = nullptr)
{
    px.xx = xx;
    px.yy = yy;
    px.zz = zz;
    px.w = w;
    px.ww = w;
    px.h = 0.f;
    px.H = H;
    px.ref = ref;
    px.nre = px.nim = 0.f;
    if (mode >= 10) {
        // FourierIterReconstructor::insert_slice: floor(p - 2.5) + [0, 5]; rejected when the
        // origin is below -n2 - 4 or above n2 + 3, n2 = P/2 - 1 for x and P/2 for y, z; clamped to [-n2, n2]
        const float pp[3] = {xx, yy, zz};
        for (int d = 0; d < 3; d++) {
            const int n2 = d == 0 ? H - 1 : H;
            const int a = (int)floor((double)pp[d] - 2.5);
            if (a < -n2 - 4 || a > n2 + 3) return false;
            px.a[d] = a;
            px.lo[d] = max(a, -n2);
            px.hi[d] = min(a + 5, n2);
            if (px.hi[d] < px.lo[d]) return false;
        }
        if (mode == 10) {
            float h = (float)(1.0f / ((double)((xx * xx + yy * yy + zz * zz) / 4000) + .15));
            px.h = h < 0.1 ? (float)0.1 : h;
            return true;
        }
        px.h = 1.0f / 2.0f;
        ref_trilinear(ref, xx, yy, zz, H, px.nre, px.nim);
        return true;
    }
    if (mode == 4) {
        const int c0 = (int)floor((double)(xx + 0.5f)), c1 = (int)floor((double)(yy + 0.5f));
        const int c2 = (int)floor((double)(zz + 0.5f));
        px.lo[0] = px.hi[0] = px.a[0] = c0;
        px.lo[1] = px.hi[1] = px.a[1] = c1;
        px.lo[2] = px.hi[2] = px.a[2] = c2;
        return true;
    }
    if (mode == 9) {
        // kaiser_bessel_derived: floor(p - 4) + [0, 8]; h = ws[0..2] = I0s(0) / I0s(32 pi) (ws[3..4] = 1),
        // ww = their float sum in the reference's order
        const float pp[3] = {xx, yy, zz};
        for (int d = 0; d < 3; d++) {
            const int a = (int)floorf(pp[d] - 4.0f);
            if (a < -H - 7 || a > H + 6) return false;
            px.a[d] = a;
            px.lo[d] = max(a, -H);
            px.hi[d] = min(a + 8, H);
            if (px.hi[d] < px.lo[d]) return false;
        }
        const float w0 = (float)(bessel_i0_scaled(0.0) / bessel_i0_scaled(M_PI * 32.0));
        px.h = w0;
        px.ww = w0 + w0 + w0 + 1.0f + 1.0f;
        return true;
    }
    if (mode == 7 || mode == 8) {
        // gridding_5: fast_floor(p - 1.5) + [0, 4]; gridding_7: fast_floor(p - 2.5) + [0, 6]
        const double sh = mode == 8 ? 2.5 : 1.5;
        const int span = mode == 8 ? 6 : 4, lo = mode == 8 ? 6 : 4, hi = mode == 8 ? 5 : 3;
        const float pp[3] = {xx, yy, zz};
        for (int d = 0; d < 3; d++) {
            const int a = ref_fast_floor((float)((double)pp[d] - sh));
            if (a < -H - lo || a > H + hi) return false;
            px.a[d] = a;
            px.lo[d] = max(a, -H);
            px.hi[d] = min(a + span, H);
            if (px.hi[d] < px.lo[d]) return false;
        }
        return true;
    }
    // gauss_3: floor(p - .5) + [0, 2]; kaiser_bessel: floor(p - 2) + [0, 4]; else floor(p - 2.5) + [0, 5]
    const double off = mode == 5 ? 0.5 : 2.5;
    const int span = mode == 5 ? 2 : mode == 6 ? 4 : 5, lo = mode == 5 ? 2 : mode == 6 ? 7 : 4;
    const int hi = mode == 5 ? 1 : mode == 6 ? 6 : 3;
    const float pp[3] = {xx, yy, zz};
    for (int d = 0; d < 3; d++) {
        const int a = mode == 6 ? (int)floor((double)(pp[d] - 2.0f)) : (int)floor((double)pp[d] - off);
        if (a < -H - lo || a > H + hi) return false;
        px.a[d] = a;
        px.lo[d] = max(a, -H);
        px.hi[d] = min(a + span, H);
        if (px.hi[d] < px.lo[d]) return false;  // an empty loop in the reference
    }
    if (mode == 6) {
        px.h = (float)(H - 1);  // nx2 - 1 of the kaiser_bessel radius scaling
    } else if (mode == 2) {
        float h = (float)(1.0f / ((double)((xx * xx + yy * yy + zz * zz) / 4000) + .15));
        px.h = h < 0.1 ? (float)0.1 : h;
    } else if (mode == 3) {
        px.h = 1.0f / (float)(10.4 / (M_PI * M_PI));
    } else {
        const float I3G = (float)(6.4 / (M_PI * M_PI));
        px.h = 32.0f / ((8.0f + sqrt_rn(xx * xx + yy * yy + zz * zz)) * I3G);
        px.ww = w / (1.0f + 6.0f * fast_exp_full(-px.h, etab) + 12 * fast_exp_full(-px.h * 2.0f, etab) +
                     8 * fast_exp_full(-px.h * 3.0f, etab));
    }
    return true;
}

// value and weight of cell (i, j, k) for the pixel (insert_wide's loop body);
// false when the contribution is dropped
__device__ __forceinline__ bool wide_term(int mode, const WidePix &px, int i, int j, int k,
                                          const float *__restrict__ etab, float &vr, float &vi, float &g)
{
    if (mode == 4) {
        vr = px.dre * px.w;
        vi = px.dim * px.w;
        g = px.w;
        return true;
    }
    if (mode == 11) {
        // updt = dt + ref(i,j,k) - ref~(p) under fast_exp(-r / 2), inside the sphere of radius P/2
        if ((long long)i * i + (long long)j * j + (long long)k * k > (long long)(2 * px.H) * (2 * px.H) / 4)
            return false;
        const float2 nt = ref_get(px.ref, i, j, k, px.H);
        const float ur = (px.dre + nt.x) - px.nre, ui = (px.dim + nt.y) - px.nim;
        const float dx = (float)i - px.xx, dy = (float)j - px.yy, dz = (float)k - px.zz;
        const float gg = fast_exp_full(-(dx * dx + dy * dy + dz * dz) * px.h, etab);
        if (fabsf(gg * px.w) < FLT_MIN) return false;
        vr = ur * gg * px.w;
        vi = ui * gg * px.w;
        g = gg * px.w;
        return true;
    }
    if (mode == 9) {
        // Mode10 (reconstructor_tools.cpp:759-812): kb = ws[0] + ... + ws[q], q <= min(r, 4) with r the
        // squared distance; value dt sqrt(kb / sum ws) w, weight w
        const float dx = (float)i - px.xx, dy = (float)j - px.yy, dz = (float)k - px.zz;
        const float r = dx * dx + dy * dy + dz * dz;
        const float lim = r < 4.0f ? r : 4.0f;
        float kb = 0.0f;
        for (int q = 0; q <= 4 && (float)q <= lim; q++) kb += q < 3 ? px.h : 1.0f;
        const float dn = sqrt_rn(__fdiv_rn(kb, px.ww));
        vr = px.dre * dn * px.w;
        vi = px.dim * dn * px.w;
        g = px.w;
        return true;
    }
    if (mode == 7 || mode == 8) {
        // Mode7 / Mode11: value dt gg w, weight w (reconstructor_tools.cpp:539-576, 964-1001)
        const int n = mode == 8 ? 12 : 9;
        const float *tab = mode == 8 ? c_grid7 : c_grid5;
        const float gg = tab[(grid_index(i, px.xx, n) * n + grid_index(j, px.yy, n)) * n + grid_index(k, px.zz, n)];
        vr = px.dre * gg * px.w;
        vi = px.dim * gg * px.w;
        g = px.w;
        return true;
    }
    const float dx = (float)i - px.xx, dy = (float)j - px.yy, dz = (float)k - px.zz;
    if (mode == 6) {
        // Mode9 (reconstructor_tools.cpp): kb = I0s(pi a sqrt(1 - (r / (nx2 - 1) - 1)^2)) / I0s(pi a),
        // a = 15, r the squared distance; value dt * kb * w, weight w
        const float r = dx * dx + dy * dy + dz * dz;
        const float t = r / px.h - 1;
        const float a = 15.0f;
        const float kb = (float)(bessel_i0_scaled(M_PI * a * (double)sqrt_rn(1.0f - t * t)) /
                                 bessel_i0_scaled(M_PI * a));
        vr = px.dre * kb * px.w;
        vi = px.dim * kb * px.w;
        g = px.w;
        return true;
    }
    const float gg = fast_exp_full(-(dx * dx + dy * dy + dz * dz) * px.h, etab);
    if (mode == 5) {
        g = gg * px.ww;
        if (fabsf(g) < FLT_MIN) return false;
        vr = px.dre * g;
        vi = px.dim * g;
        return true;
    }
    if (fabsf(gg * px.ww) < FLT_MIN) return false;
    vr = px.dre * gg * px.ww;
    vi = px.dim * gg * px.ww;
    g = gg * px.ww;
    return true;
}

// one pixel's stencil straight into the volume (the single-slice and
// fallback form of the wide modes), the same terms as the LDS-window form
__device__ void insert_wide(int mode, float2 dt, float xx, float yy, float zz, float w, int P, int H,
                            const float *__restrict__ etab, float2 *data, float *norm, const float2 *ref)
{
    WidePix px;
    if (!wide_setup(mode, xx, yy, zz, w, H, etab, px, ref)) return;
    px.dre = dt.x;
    px.dim = dt.y;
    for (int k = px.lo[2]; k <= px.hi[2]; k++)
        for (int j = px.lo[1]; j <= px.hi[1]; j++)
            for (int i = px.lo[0]; i <= px.hi[0]; i++) {
                float vr, vi, g;
                if (wide_term(mode, px, i, j, k, etab, vr, vi, g)) add_complex_atomic(data, norm, P, H, i, j, k, vr, vi, g);
            }
}

__global__ void __launch_bounds__(256) k_insert_wide_tiles(const float2 *__restrict__ slices, int nsym, int ntx,
                                                           int nty, const float *__restrict__ t3d,
                                                           const float *__restrict__ wq, InsertConst c, float2 *data,
                                                           float *norm, const float *__restrict__ exptab,
                                                           const float *__restrict__ rtab_g,
                                                           const float *__restrict__ rw)
{
    extern __shared__ float win[];  // re, im, weight: 3 x WT_CELLS
    __shared__ WidePix pix[WT_TILE * WT_TILE];
    __shared__ int okp[WT_TILE * WT_TILE];
    __shared__ int wlo[3], nvalid;
    const int H = c.H, P = c.P;
    const int tiles = ntx * nty;
    const int q = blockIdx.x / tiles;
    const int tt = blockIdx.x - q * tiles;
    const int tx0 = (tt % ntx) * WT_TILE, ty0 = (tt / ntx) * WT_TILE - H;
    const int p = q / nsym;
    const float wgt = wq[q];
    if (threadIdx.x < 3) wlo[threadIdx.x] = INT_MAX;
    if (threadIdx.x == 0) nvalid = 0;
    __syncthreads();
    if (threadIdx.x < WT_TILE * WT_TILE) {
        const int x = tx0 + (threadIdx.x % WT_TILE), y = ty0 + (threadIdx.x / WT_TILE);
        bool ok = wgt != 0.0f && x <= H && y <= H - 1 && (c.corners || x * x + y * y <= c.rcut * c.rcut + c.rcut);
        if (ok) {
            const float weight = rw ? rw[(size_t)p * (H + 1) + hypot_int(x, y)] : wgt;
            float xx, yy, zz;
            pixel_coords(x, y, t3d + 9 * (size_t)q, rtab_g, H, c.Pf, xx, yy, zz);
            WidePix px;
            ok = wide_setup(c.mode, xx, yy, zz, weight, H, exptab, px, c.ref);
            if (ok) {
                const float2 dt = slice_value(slices + (size_t)p * P * (H + 1), x, y, P, H);
                px.dre = dt.x;
                px.dim = dt.y;
                pix[threadIdx.x] = px;
                for (int d = 0; d < 3; d++) atomicMin(&wlo[d], px.lo[d]);
                atomicAdd(&nvalid, 1);
            }
        }
        okp[threadIdx.x] = ok;
    }
    __syncthreads();
    if (nvalid == 0) return;  // block-uniform
    for (int i = threadIdx.x; i < 3 * WT_CELLS; i += blockDim.x) win[i] = 0.f;
    __syncthreads();
    const int pi = threadIdx.x >> 2, part = threadIdx.x & 3;
    if (okp[pi]) {
        const WidePix px = pix[pi];
        const int nx = px.hi[0] - px.lo[0] + 1, ny = px.hi[1] - px.lo[1] + 1;
        const int ncell = nx * ny * (px.hi[2] - px.lo[2] + 1);
        for (int ci = part; ci < ncell; ci += 4) {
            const int kk = ci / (nx * ny), rem = ci - kk * nx * ny, jj = rem / nx, ii = rem - jj * nx;
            const int i = px.lo[0] + ii, j = px.lo[1] + jj, k = px.lo[2] + kk;
            float vr, vi, g;
            if (!wide_term(c.mode, px, i, j, k, exptab, vr, vi, g)) continue;
            const int a = i - wlo[0], b = j - wlo[1], e = k - wlo[2];
            if ((unsigned)a < (unsigned)WT_WIN && (unsigned)b < (unsigned)WT_WIN && (unsigned)e < (unsigned)WT_WIN) {
                const int cell = (e * WT_WIN + b) * WT_WIN + a;
                atomicAdd(&win[cell], vr);
                atomicAdd(&win[WT_CELLS + cell], vi);
                atomicAdd(&win[2 * WT_CELLS + cell], g);
            } else {
                add_complex_atomic(data, norm, P, H, i, j, k, vr, vi, g);
            }
        }
    }
    __syncthreads();
    for (int cell = threadIdx.x; cell < WT_CELLS; cell += blockDim.x) {
        const float g = win[2 * WT_CELLS + cell];
        if (g == 0.f) continue;
        const int a = cell % WT_WIN, b = (cell / WT_WIN) % WT_WIN, e = cell / (WT_WIN * WT_WIN);
        add_complex_atomic(data, norm, P, H, wlo[0] + a, wlo[1] + b, wlo[2] + e, win[cell], win[WT_CELLS + cell], g);
    }
}

hipError_t launch_insert_plain_batch(const float2 *slices, int nslices, int nsym, const float *t3d, const float *wq,
                                     InsertConst c, float2 *data, float *norm, const float *exptab, const float *rtab,
                                     const float *rw, hipStream_t s)
{
    if (nslices <= 0) return hipSuccess;
    if (c.mode < 2) return hipErrorInvalidValue;
    const int ntx = (c.H + 1 + WT_TILE - 1) / WT_TILE, nty = (c.P + WT_TILE - 1) / WT_TILE;
    const long long blocks = (long long)ntx * nty * nslices;
    if (blocks < INT32_MAX) {
        hipLaunchKernelGGL(k_insert_wide_tiles, dim3((unsigned)blocks), dim3(256), sizeof(float) * 3 * WT_CELLS, s,
                           slices, nsym, ntx, nty, t3d, wq, c, data, norm, exptab, rtab, rw);
        return hipGetLastError();
    }
    const int nxb = (c.H + 1 + 63) / 64;
    hipLaunchKernelGGL(k_insert_plain_batch, dim3(nxb * nslices, c.P), dim3(64), 0, s, slices, nsym, nxb, t3d, wq, c,
                       data, norm, exptab, rtab, rw);
    return hipGetLastError();
}

hipError_t launch_insert_plain(const float2 *slice, InsertConst c, const float *t3d9, float weight, float2 *data,
                               float *norm, const float *exptab, const float *rtab, const float *rw, hipStream_t s)
{
    Mat9 m;
    for (int i = 0; i < 9; i++) m.m[i] = t3d9[i];
    if (c.mode >= 2)
        hipLaunchKernelGGL(k_insert_plain, dim3((c.H + 1 + 63) / 64, c.P), dim3(64), 0, s, slice, c, m, weight, data, norm,
                           exptab, rtab, rw);
    else
        hipLaunchKernelGGL(k_insert_corners, dim3((c.H + 1 + 31) / 32, c.P), dim3(256), 0, s, slice, c, m, weight, data,
                           norm, exptab, rtab, rw);
    return hipGetLastError();
}

// ------------------------------------------------------------ slice agreement
// FourierReconstructor::do_compare_slice_work (libEM/reconstructor.cpp:1259-1381)
// with pixel_at (:1448-1461): nearest-voxel value/weight at each slice pixel
// x in [0, P/2+1] (the x = P/2+1 column reads the next row's x = 0 element,
// and past the last row 0), eight double sums per (slice, block).
__device__ __forceinline__ int round_ref(float v) { return v < 0 ? (int)(v - 0.5f) : (int)(v + 0.5f); }

__global__ void __launch_bounds__(256) k_agree(const float2 *__restrict__ slices, int nsym, const float *__restrict__ t3d,
                                               InsertConst c, float rmax, const float2 *__restrict__ data,
                                               const float *__restrict__ norm, const float *__restrict__ rtab,
                                               double *__restrict__ partial)
{
    const int H = c.H, P = c.P;
    const int q = blockIdx.y;
    const int pidx = blockIdx.x * blockDim.x + threadIdx.x;
    const int W = H + 2;
    double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // dot vweight power power2 dotlow dlpow dlpow2 nval
    if (pidx < W * P) {
        const int x = pidx % W, y = pidx / W - H;
        const float *m = t3d + 9 * (size_t)q;
        if (!(x == 0 && y == 0)) {
            const float rx = rtab[x + H], ry = rtab[y + H];
            const float c0 = rx * m[0] + ry * m[3];
            const float c1 = rx * m[1] + ry * m[4];
            const float c2 = rx * m[2] + ry * m[5];
            if (!(fabsf(c0) > 0.5f || fabsf(c1) >= 0.5f || fabsf(c2) >= 0.5f)) {
                const float xx = c0 * c.Pf, yy = c1 * c.Pf, zz = c2 * c.Pf;
                const float *Sf = reinterpret_cast<const float *>(slices + (size_t)(q / nsym) * P * (H + 1));
                const int slen = (P + 2) * P;
                const int fidx = 2 * x + (P + 2) * (y < 0 ? P + y : y);
                const float d20 = fidx < slen ? Sf[fidx] : 0.f;
                const float d21 = fidx + 1 < slen ? Sf[fidx + 1] : 0.f;
                const int x0 = round_ref(xx), y0 = round_ref(yy), z0 = round_ref(zz);
                float vr = 0.f, vi = 0.f;
                size_t ci;
                if (x0 < 0) ci = cidx(-x0, y0 <= 0 ? -y0 : P - y0, z0 <= 0 ? -z0 : P - z0, P, H);
                else ci = cidx(x0, y0 < 0 ? P + y0 : y0, z0 < 0 ? P + z0 : z0, P, H);
                if (!(abs(x0) >= H + 1 || abs(y0) > H || abs(z0) > H)) {
                    const float2 v = data[ci];
                    vr = v.x;
                    vi = x0 < 0 ? -v.y : v.y;
                }
                const float nv = norm[ci];
                if (nv != 0.f) {
                    const float dt0 = __fdiv_rn(vr, nv), dt1 = __fdiv_rn(vi, nv), dt2 = nv;
                    const float r = sqrt_int_rn(x * x + y * y);  // Util::hypot_fast
                    const float dotv = (dt0 * d20 + dt1 * d21) * dt2;
                    const float pw = (dt0 * dt0 + dt1 * dt1) * dt2;
                    const float pw2 = (d20 * d20 + d21 * d21) * dt2;
                    if (r > 3 && r < rmax) {
                        acc[4] += dotv;
                        acc[5] += pw;
                        acc[6] += pw2;
                    }
                    acc[1] += dt2;
                    acc[0] += dotv;
                    acc[2] += pw;
                    acc[3] += pw2;
                    acc[7] += 1.0;
                }
            }
        }
    }
    __shared__ double red[8][256];
#pragma unroll
    for (int k = 0; k < 8; k++) red[k][threadIdx.x] = acc[k];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s)
#pragma unroll
            for (int k = 0; k < 8; k++) red[k][threadIdx.x] += red[k][threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x < 8) partial[((size_t)q * gridDim.x + blockIdx.x) * 8 + threadIdx.x] = red[threadIdx.x][0];
}

int agree_blocks(int P) { return ((P / 2 + 2) * P + 255) / 256; }

// ---- batched agreement: compare against V - own(p) without mutating V ----
// own(p) at a storage voxel is what determine_slice_agreement's
// do_insert_slice_work(slice, R, -w) would subtract there
// (libEM/reconstructor.cpp:1236): the gauss_2 / trilinear contributions of
// all symmetry copies of particle p whose stencil cell folds onto the voxel.
// Unfolded sources of storage voxel (xs, ys, zs), following
// add_complex_at_fast: direct cells (xs, j, k) with wrap(j)=ys, wrap(k)=zs,
// conjugate cells (-xs, j, k) with wrapneg(j)=ys, wrapneg(k)=zs, and on the
// x=0 / x=P/2 planes the conjugate copies of the double insertion.

// contributions of slice copy m (t3d rows) of particle S to unfolded cell c
__device__ __forceinline__ void gather_cell(const float2 *__restrict__ S, const float *m, int ci, int cj, int ck,
                                            const InsertConst &c, float weight, const float *etab,
                                            const float *rtab, float &re, float &im, float &w)
{
    const int H = c.H, P = c.P;
    const float n0 = m[1] * m[5] - m[2] * m[4], n1 = m[2] * m[3] - m[0] * m[5], n2 = m[0] * m[4] - m[1] * m[3];
    const float dist = n0 * ci + n1 * cj + n2 * ck;
    if (fabsf(dist) > 1.7330f) return;  // |p - c|_inf < 1 on the plane => |n.c| < sqrt(3)
    const float s = m[0] * ci + m[1] * cj + m[2] * ck;
    const float t = m[3] * ci + m[4] * cj + m[5] * ck;
    const int xa = max(0, (int)ceilf(s - 1.7330f)), xb = min(H, (int)floorf(s + 1.7330f));
    const int ya = max(-H, (int)ceilf(t - 1.7330f)), yb = min(H - 1, (int)floorf(t + 1.7330f));
    for (int y = ya; y <= yb; y++)
        for (int x = xa; x <= xb; x++) {
            if (x * x + y * y > H * H + H) continue;  // radius cut (corners=false)
            float xx, yy, zz;
            pixel_coords(x, y, m, rtab, H, c.Pf, xx, yy, zz);
            const int x0 = (int)floorf(xx), y0 = (int)floorf(yy), z0 = (int)floorf(zz);
            if (x0 < -H - 1 || y0 < -H - 1 || z0 < -H - 1 || x0 > H || y0 > H || z0 > H) continue;
            if ((unsigned)(ci - x0) > 1u || (unsigned)(cj - y0) > 1u || (unsigned)(ck - z0) > 1u) continue;
            const float gg = corner_weight(c.mode, ci, cj, ck, xx, yy, zz, c.h, weight, etab);
            const float2 dt = slice_value(S, x, y, P, H);
            re += dt.x * gg;
            im += dt.y * gg;
            w += gg;
        }
}

__device__ __forceinline__ void gather_cell_all(const float2 *S, const float *t3dp, int nsym, int ci, int cj, int ck,
                                                const InsertConst &c, float weight, const float *etab,
                                                const float *rtab, float &re, float &im, float &w)
{
    for (int s = 0; s < nsym; s++) gather_cell(S, t3dp + 9 * s, ci, cj, ck, c, weight, etab, rtab, re, im, w);
}

// own(p) at storage voxel (xs, ys, zs): value (ore, oim) and weight ow
__device__ void own_contribution(const float2 *S, const float *t3dp, int nsym, int xs, int ys, int zs,
                                 const InsertConst &c, float weight, const float *etab, const float *rtab,
                                 float &ore, float &oim, float &ow)
{
    const int H = c.H, P = c.P;
    ore = oim = ow = 0.f;
    int jd[2], njd = 0, jn[2], njn = 0, kd[2], nkd = 0, kn[2], nkn = 0;
    if (ys <= H) jd[njd++] = ys;
    if (ys >= H) jd[njd++] = ys - P;
    if (ys <= H) jn[njn++] = -ys;
    if (ys >= H && P - ys <= H && P - ys != -ys) jn[njn++] = P - ys;
    if (zs <= H) kd[nkd++] = zs;
    if (zs >= H) kd[nkd++] = zs - P;
    if (zs <= H) kn[nkn++] = -zs;
    if (zs >= H && P - zs <= H && P - zs != -zs) kn[nkn++] = P - zs;
    if (ys == 0 && zs == 0 && (xs == 0 || xs == H)) {
        float r = 0, i = 0, w = 0;
        gather_cell_all(S, t3dp, nsym, xs, 0, 0, c, weight, etab, rtab, r, i, w);
        if (xs == H) gather_cell_all(S, t3dp, nsym, -H, 0, 0, c, weight, etab, rtab, r, i, w);
        ore = r;
        ow = w;
        return;
    }
    for (int a = 0; a < njd; a++)
        for (int b = 0; b < nkd; b++) {  // direct: value and weight
            float r = 0, i = 0, w = 0;
            gather_cell_all(S, t3dp, nsym, xs, jd[a], kd[b], c, weight, etab, rtab, r, i, w);
            ore += r;
            oim += i;
            ow += w;
        }
    for (int a = 0; a < njn; a++)
        for (int b = 0; b < nkn; b++) {
            float r = 0, i = 0, w = 0;
            if (xs == 0 || xs == H) {
                // conjugate copy of the double insertion: value only
                gather_cell_all(S, t3dp, nsym, xs, jn[a], kn[b], c, weight, etab, rtab, r, i, w);
                ore += r;
                oim -= i;
                if (xs == H) {  // x = -P/2 cells: conjugate added twice, weight once
                    float r2 = 0, i2 = 0, w2 = 0;
                    gather_cell_all(S, t3dp, nsym, -H, jn[a], kn[b], c, weight, etab, rtab, r2, i2, w2);
                    ore += 2.f * r2;
                    oim -= 2.f * i2;
                    ow += w2;
                }
            } else {
                gather_cell_all(S, t3dp, nsym, -xs, jn[a], kn[b], c, weight, etab, rtab, r, i, w);
                ore += r;
                oim -= i;
                ow += w;
            }
        }
}

// Tiles of compare pixels: each workgroup takes a tile of one (particle,
// symmetry op) slice, 32 x 32 pixels without symmetry and 32 x 16 with it, and
// stages the slice around it (2-pixel halo: the sources of a compare pixel's
// nearest cell lie within 2 pixels of it) in LDS -- pixel positions, values
// and the insertion loop's pixel filters -- so that the own-contribution
// gather of the slice's own plane reads LDS; the other symmetry planes and
// windows that leave the patch take the global gather.
constexpr int AT_X = 32, AT_HALO = 2;
constexpr int AT_PX = AT_X + 2 * AT_HALO;
constexpr int AT_MX = 7;
// Sizes for tiles of AY rows.  Mirror patch of the x = 0 tiles: pixels x in
// [-4, 2], y in [-ty0 - AY - 1, -ty0 + 2], the sources of the mirrored cells of
// compare pixels x < 3 (around (-x, -y)).
template <int AY>
struct AgreeTile {
    static constexpr int PY = AY + 2 * AT_HALO, PATCH = AT_PX * PY, MY = AY + 4, MPATCH = AT_MX * MY;
    static constexpr int THREADS = 16 * AY, WAVES = THREADS / 64;
};

// Patch entries carry the floors of their position packed as
// (x0 + 512) | (y0 + 512) << 10 | (z0 + 512) << 20, or
// AP_NOKEY for pixels the insertion loop skips (radius cut, origin range).
// For a cell key kc, kc - key has every 10-bit digit in {0, 1} exactly when
// the cell is a corner of the pixel's 2x2x2 stencil; the digits are
// differences of at most a few units between neighbouring pixels, so the
// packed difference is unambiguous, and AP_NOKEY makes it negative.
constexpr int AP_NOKEY = (int)0x80000000u;
constexpr unsigned AP_DIGITS = 0x100401u;
__device__ __forceinline__ int ap_key(int x0, int y0, int z0)
{
    return x0 + (y0 << 10) + (z0 << 20) + (512 + (512 << 10) + (512 << 20));  // digits of 10 bits, none negative
}

// A patch entry: pixel position, packed floors (AP_NOKEY: skipped by the
// insertion loop) and slice_value.
struct AgreePx {
    float x, y, z;
    int key;
    float2 v;
};

struct AgreePatch {
    const AgreePx *px;
    int x0, y0;          // pixel of patch entry 0
    int py;              // patch rows
};

__device__ __forceinline__ void gather_cell_patch(const float2 *__restrict__ S, const float *m, const AgreePatch &pt,
                                                  int ci, int cj, int ck, const InsertConst &c, float weight,
                                                  const float *etab, const float *rtab, float &re, float &im,
                                                  float &w)
{
    const int H = c.H;
    const float n0 = m[1] * m[5] - m[2] * m[4], n1 = m[2] * m[3] - m[0] * m[5], n2 = m[0] * m[4] - m[1] * m[3];
    const float dist = n0 * ci + n1 * cj + n2 * ck;
    if (fabsf(dist) > 1.7330f) return;  // |p - c|_inf < 1 on the plane => |n.c| < sqrt(3)
    const float s = m[0] * ci + m[1] * cj + m[2] * ck;
    const float t = m[3] * ci + m[4] * cj + m[5] * ck;
    const int xa = max(0, (int)ceilf(s - 1.7330f)), xb = min(H, (int)floorf(s + 1.7330f));
    const int ya = max(-H, (int)ceilf(t - 1.7330f)), yb = min(H - 1, (int)floorf(t + 1.7330f));
    if (xa < pt.x0 || xb >= pt.x0 + AT_PX || ya < pt.y0 || yb >= pt.y0 + pt.py) {
        gather_cell(S, m, ci, cj, ck, c, weight, etab, rtab, re, im, w);
        return;
    }
    for (int y = ya; y <= yb; y++)
        for (int x = xa; x <= xb; x++) {
            const int e = (y - pt.y0) * AT_PX + (x - pt.x0);
            const AgreePx q = pt.px[e];
            if (q.key == AP_NOKEY) continue;  // radius cut / origin out of range
            const int x0 = (int)floorf(q.x), y0 = (int)floorf(q.y), z0 = (int)floorf(q.z);
            if ((unsigned)(ci - x0) > 1u || (unsigned)(cj - y0) > 1u || (unsigned)(ck - z0) > 1u) continue;
            const float gg = corner_weight(c.mode, ci, cj, ck, q.x, q.y, q.z, c.h, weight, etab);
            re += q.v.x * gg;
            im += q.v.y * gg;
            w += gg;
        }
}

// Own-plane contributions to unfolded cell (ci, cj, ck), the nearest cell of
// patch entry e, or its mirror -(ci, cj, ck) gathered around the mirrored
// pixel.  A stencil that holds the cell starts
// within 1 of it on every axis, and the cell lies within 0.5 of entry e's
// position, so the source pixel sits less than 1.5 from that position on
// every axis: only the in-plane offsets (ox, oy) in [-2, 2]^2 of
// own_offset_mask can hold it.  Lane k of `list` holds the k-th of the n
// offsets, in patch entries times 24 bytes; taken four at a time, so that
// their reads are in flight together.
// gauss_2's table index (int)((double)f 50 + 0.5) is read off the sum's bits:
// with 2^18 added the double's high word ends in the index and two fraction
// bits, so that word & 0xffc is the entry's byte offset (the sum is exact
// wherever it could reach the next integer: f 50 is a multiple of 2^-29 from
// f = 2^-7 on).  Misses read the table too, up to byte 0xffc of the LDS, which
// the table starts.
template <int MODE, int N>
__device__ __forceinline__ void gather_some_offsets(const AgreePx *px, int list, int k0, int kc, float cx, float cy, float cz,
                                                    float h, float weight, float &re, float &im, float &w)
{
    AgreePx q[N];
    float g[N];
#pragma unroll
    for (int k = 0; k < N; k++)
        q[k] = *reinterpret_cast<const AgreePx *>(reinterpret_cast<const char *>(px) +
                                                  __builtin_amdgcn_readlane(list, k0 + k));
#pragma unroll
    for (int k = 0; k < N; k++) {
        const float dx = cx - q[k].x, dy = cy - q[k].y, dz = cz - q[k].z;
        if (MODE == 0) {
            const float f = (dx * dx + dy * dy + dz * dz) * h;
            const unsigned b = (unsigned)__double2hiint(__builtin_fma((double)f, 50.0, 262144.5)) & 0xffcu;
            g[k] = *(const __attribute__((address_space(3))) float *)b * weight;
        } else {
            g[k] = (float)((1.0 - (double)fabsf(dx)) * (1.0 - (double)fabsf(dy)) * (1.0 - (double)fabsf(dz)) *
                           (double)weight);
        }
    }
    // each term as the insertion adds it, so that a voxel that only this particle reached, through one or two
    // terms, cancels to 0 (the order of more than two is not the insertion's)
#pragma unroll
    for (int k = 0; k < N; k++) {
        const float gg = ((unsigned)(kc - q[k].key) & ~AP_DIGITS) == 0u ? g[k] : 0.f;
        re += q[k].v.x * gg;
        im += q[k].v.y * gg;
        w += gg;
    }
}

template <int MODE>
__device__ __forceinline__ void gather_own_offsets(const AgreePx *px, int list, int n, int ci, int cj, int ck, float h,
                                                   float weight, float &re, float &im, float &w)
{
    const int kc = ap_key(ci, cj, ck);
    const float cx = (float)ci, cy = (float)cj, cz = (float)ck;
    int k = 0;
    for (; k + 4 <= n; k += 4) gather_some_offsets<MODE, 4>(px, list, k, kc, cx, cy, cz, h, weight, re, im, w);
    if (n & 2) gather_some_offsets<MODE, 2>(px, list, k, kc, cx, cy, cz, h, weight, re, im, w);
    if (n & 1) gather_some_offsets<MODE, 1>(px, list, n - 1, kc, cx, cy, cz, h, weight, re, im, w);
}

// Offsets (ox, oy) in [-2, 2]^2 whose step ox * row0 + oy * row1 of slice
// rows m stays under 1.5 (plus rounding slack) on every axis: lane k < 25
// tests offset k, the wave's ballot is the mask (the whole wave active).
__device__ __forceinline__ unsigned own_offset_mask(const float *m)
{
    const int k = threadIdx.x & 63;
    bool ok = false;
    if (k < 25) {
        const float ox = (float)(k % 5 - 2), oy = (float)(k / 5 - 2);
        const float d0 = ox * m[0] + oy * m[3], d1 = ox * m[1] + oy * m[4], d2 = ox * m[2] + oy * m[5];
        ok = fmaxf(fabsf(d0), fmaxf(fabsf(d1), fabsf(d2))) < 1.51f;
    }
    return (unsigned)__ballot(ok);
}

// Lane k: the k-th set bit's offset in patch entries of row pitch `pitch`, times 24 bytes.
__device__ __forceinline__ int own_offset_list(unsigned mask, int pitch)
{
    const int b = threadIdx.x & 63;
    const int o = (int)sizeof(AgreePx) * ((b / 5 - 2) * pitch + (b % 5 - 2));
    // lane b < 25 with its bit set sends its offset to lane (bits below b), the others to lane 63
    const int to = b < 25 && (mask >> b & 1u) ? __popc(mask & ((1u << b) - 1u)) : 63;
    return __builtin_amdgcn_ds_permute(to << 2, o);
}

// own_contribution() with the slice's own plane gathered from the patch.
__device__ void own_contribution_tile(const float2 *S, const float *t3dp, int nsym, int own, const AgreePatch &pt,
                                      int xs, int ys, int zs, const InsertConst &c, float weight, const float *etab,
                                      const float *rtab, float &ore, float &oim, float &ow)
{
    const int H = c.H, P = c.P;
    auto cell_all = [&](int ci, int cj, int ck, float &r, float &i, float &w) {
        for (int sop = 0; sop < nsym; sop++) {
            if (sop == own) gather_cell_patch(S, t3dp + 9 * sop, pt, ci, cj, ck, c, weight, etab, rtab, r, i, w);
            else gather_cell(S, t3dp + 9 * sop, ci, cj, ck, c, weight, etab, rtab, r, i, w);
        }
    };
    ore = oim = ow = 0.f;
    int jd[2], njd = 0, jn[2], njn = 0, kd[2], nkd = 0, kn[2], nkn = 0;
    if (ys <= H) jd[njd++] = ys;
    if (ys >= H) jd[njd++] = ys - P;
    if (ys <= H) jn[njn++] = -ys;
    if (ys >= H && P - ys <= H && P - ys != -ys) jn[njn++] = P - ys;
    if (zs <= H) kd[nkd++] = zs;
    if (zs >= H) kd[nkd++] = zs - P;
    if (zs <= H) kn[nkn++] = -zs;
    if (zs >= H && P - zs <= H && P - zs != -zs) kn[nkn++] = P - zs;
    if (ys == 0 && zs == 0 && (xs == 0 || xs == H)) {
        float r = 0, i = 0, w = 0;
        cell_all(xs, 0, 0, r, i, w);
        if (xs == H) cell_all(-H, 0, 0, r, i, w);
        ore = r;
        ow = w;
        return;
    }
    for (int a = 0; a < njd; a++)
        for (int b = 0; b < nkd; b++) {  // direct: value and weight
            float r = 0, i = 0, w = 0;
            cell_all(xs, jd[a], kd[b], r, i, w);
            ore += r;
            oim += i;
            ow += w;
        }
    for (int a = 0; a < njn; a++)
        for (int b = 0; b < nkn; b++) {
            float r = 0, i = 0, w = 0;
            if (xs == 0 || xs == H) {
                // conjugate copy of the double insertion: value only
                cell_all(xs, jn[a], kn[b], r, i, w);
                ore += r;
                oim -= i;
                if (xs == H) {  // x = -P/2 cells: conjugate added twice, weight once
                    float r2 = 0, i2 = 0, w2 = 0;
                    cell_all(-H, jn[a], kn[b], r2, i2, w2);
                    ore += 2.f * r2;
                    oim -= 2.f * i2;
                    ow += w2;
                }
            } else {
                cell_all(-xs, jn[a], kn[b], r, i, w);
                ore += r;
                oim -= i;
                ow += w;
            }
        }
}

// Voxel (x, y, z) of the packed volume: cubes of 2^3 voxels, 128 bytes, so that the nearest voxels of a
// slice's plane fall in few cache lines.  (P even; fewer than 2^30 entries for P <= 1024.)
__device__ __forceinline__ unsigned pack_index(unsigned x, unsigned y, unsigned z, int P)
{
    const unsigned H = P / 2;
    return (((z >> 1) * H + (y >> 1)) * (H / 2 + 1) + (x >> 1)) * 8 + ((z & 1) << 2 | (y & 1) << 1 | (x & 1));
}

// One workgroup per (compare-pixel tile, particle x symmetry op slice); eight
// double sums per particle accumulated with float64 atomics into acc[p][8].
// vol: the volume as float4 (re, im, weight, 0) per voxel, or null, then data
// and norm are read.  n3: the low-resolution band is 9 < x^2 + y^2 < n3.
// Bound: latency.  At pad 600 0.24 VALU instructions per SIMD and clock, 0.48
// of the published vector rate (k_scatter_gauss6 reaches 0.70), the LDS busy
// 38 %, 5.2 waves per SIMD resident: a gather is a chain of patch read, table
// read and sum.  With symmetry 0.14 at 2.6 waves.  8,000 slices at pad 600:
// 36.5 ms before, 23.7 now.  What it took: the voxels read before the patch is
// staged and at most 80 registers (3 workgroups of 8 waves per CU; 34 ms with
// 2), the packed volume in 2^3 cubes (0.60 G instead of 0.92 G line misses;
// data and weights read apart: 33.4 ms), offsets in groups of four so that
// their LDS reads overlap, 32 x 32 tiles (halo 1.27 instead of 1.41).  1,500
// particles of d2 at pad 192: 7.1 -> 5.5 ms, the other planes' gather by full
// waves.  The whole call 5.8 ms with their sums in double; 5.9 with float
// atomics, whose order showed in the results; 7.6 plane by plane without
// atomics, the waves half empty (300 particles of d7: 7.0, 7.7 and 13.6).
template <int MODE, bool SYM, bool PACKED>
__global__ void __launch_bounds__(AgreeTile<SYM ? 16 : 32>::THREADS) __attribute__((amdgpu_waves_per_eu(SYM ? 5 : 6)))
    k_agree_batch(const float2 *__restrict__ slices, int nsym, const float *__restrict__ t3d, const float *__restrict__ wq,
                  InsertConst c, int n3, int sub, int qcap, const float2 *__restrict__ data, const float *__restrict__ norm,
                  const float4 *__restrict__ vol, const float *__restrict__ exptab, const float *__restrict__ rtab_g,
                  double *__restrict__ acc_out)
{
    constexpr int AY = SYM ? 16 : 32;
    using AT = AgreeTile<AY>;
    const int H = c.H, P = c.P;
    const int q = blockIdx.y, p = q / nsym, own = q - p * nsym;
    const int W = H + 2;
    const int ntx = (W + AT_X - 1) / AT_X;
    const int tx0 = (blockIdx.x % ntx) * AT_X, ty0 = (int)(blockIdx.x / ntx) * AY - H;
    const float2 *S = slices + (size_t)p * P * (H + 1);
    const float *t3dp = t3d + 9 * (size_t)p * nsym;
    const float *m = t3d + 9 * (size_t)q;
    const float weight = wq[q];
    // dynamic LDS, from address 0: fast_exp table, patch, mirror patch; with symmetry the near planes; counters;
    // with symmetry the sums of the other planes, fl(i/P), the pixels' cells (keys) and the other planes' queue
    // of qcap entries; the queued compare pixels
    extern __shared__ float4 agree_lds[];
    float *etab = reinterpret_cast<float *>(agree_lds);
    AgreePx *ppx = reinterpret_cast<AgreePx *>(etab + EXPN);
    AgreePx *mpx = ppx + AT::PATCH;
    unsigned long long *near_ops = reinterpret_cast<unsigned long long *>(mpx + AT::MPATCH);  // a bit per plane
    const int nwords = (nsym + 63) / 64;  // symmetries of more than 4096 operators take every plane
    int *dn = reinterpret_cast<int *>(near_ops + (SYM ? min(nwords, 64) : 0));
    constexpr int NPX = AT_X * AY;
    double *osum = reinterpret_cast<double *>(dn + 4);
    float *rtab_l = reinterpret_cast<float *>(osum + (SYM ? 3 * NPX : 0));
    int *cell = reinterpret_cast<int *>(rtab_l + (SYM ? P + 2 : 0));
    unsigned short *queue = reinterpret_cast<unsigned short *>(cell + (SYM ? NPX : 0));
    unsigned short *dq = queue;  // at most NPX compare pixels (tile index), after the other planes are through
    const float *rtab = SYM ? rtab_l : rtab_g;
    if (SYM) {
        for (int i = threadIdx.x; i < P + 2; i += AT::THREADS) rtab_l[i] = rtab_g[i];
        for (int i = threadIdx.x; i < 3 * NPX; i += AT::THREADS) osum[i] = 0.0;
    }
    for (int i = threadIdx.x; i < EXPN; i += AT::THREADS) etab[i] = exptab[i];
    AgreePatch pt{ppx, tx0 - AT_HALO, ty0 - AT_HALO, AT::PY};
    if (threadIdx.x == 0) dn[0] = dn[1] = 0;
    // packed floor keys need |x0|, |y0|, |z0| <= 511
    const bool fastkeys = sub && H <= 510;
    const unsigned omask = fastkeys ? own_offset_mask(m) : 0u;
    const int olist = own_offset_list(omask, AT_PX), on = __popc(omask);
    auto stage = [&](int x, int y, AgreePx &e) {
        AgreePx o{0.f, 0.f, 0.f, AP_NOKEY, make_float2(0.f, 0.f)};
        // the insertion loop's pixels: x in [0, P/2], y in [-P/2, P/2), radius cut (corners off here; it
        // bounds |x| and |y| by P/2)
        if (x >= 0 && y < H && x * x + y * y <= H * H + H) {
            pixel_coords(x, y, m, rtab_g, H, c.Pf, o.x, o.y, o.z);
            // origins in [-P/2 - 1, P/2]
            if (fmaxf(fabsf(o.x), fmaxf(fabsf(o.y), fabsf(o.z))) < (float)(H + 1)) {
                o.key = ap_key((int)floorf(o.x), (int)floorf(o.y), (int)floorf(o.z));
                const bool cj = x == 0 && y < 0;  // slice_value
                o.v = S[(unsigned)(cj ? -y : (y < 0 ? P + y : y)) * (unsigned)(H + 1) + (unsigned)x];
                if (cj) o.v.y = -o.v.y;
            }
        }
        e = o;
    };
    // own contributions reach compare pixels within the insertion radius plus sqrt(3) (a stencil) plus
    // sqrt(3) / 2 (the nearest cell): beyond, the tile's patch is not needed
    const int rown2 = (H + 4) * (H + 4);
    const int ny0 = ty0 > 0 ? ty0 : (ty0 + AY - 1 < 0 ? ty0 + AY - 1 : 0);  // the tile's row nearest 0
    const bool inner = sub && tx0 * tx0 + ny0 * ny0 <= rown2;
    const int my0 = -ty0 - AY - 1;
    const bool mirror = fastkeys && tx0 == 0;
    // the other symmetry planes that pass within reach of the tile's nearest cells: |n . p| <= sqrt(3)
    // (gather_cell's bound) + sqrt(3) / 2
    const int lane = threadIdx.x & 63;
    if (SYM && fastkeys && nwords <= 64) {
        for (int wd = threadIdx.x >> 6; wd < nwords; wd += AT::WAVES) {
            const int sop = 64 * wd + lane;
            bool hit = false;
            if (sop < nsym && sop != own) {
                const float *o = t3dp + 9 * sop;
                const float n0 = o[1] * o[5] - o[2] * o[4], n1 = o[2] * o[3] - o[0] * o[5], n2 = o[0] * o[4] - o[1] * o[3];
                const float a = n0 * m[0] + n1 * m[1] + n2 * m[2], b = n0 * m[3] + n1 * m[4] + n2 * m[5];
                const float xa = a * (float)tx0, xb = a * (float)(tx0 + AT_X - 1);
                const float ya = b * (float)ty0, yb = b * (float)(ty0 + AY - 1);
                hit = fminf(xa, xb) + fminf(ya, yb) <= 2.62f && fmaxf(xa, xb) + fmaxf(ya, yb) >= -2.62f;
            }
            const unsigned long long hm = __ballot(hit);
            if (lane == 0) near_ops[wd] = hm;
        }
    }
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    int nval = 0;
    // One compare pixel: load() takes its voxel and slice value, compare() its own contribution and the
    // sums.  Outside the general pass a pixel whose voxel needs the general own-contribution enumeration is
    // left for later (the few such pixels of a tile, voxels on the x = P/2 and y, z = P/2 planes, then share
    // waves instead of holding back every wave they fall in).
    struct Pixel {
        int l, x, y, x0, y0, z0;
        bool now, later;
        float vr, vi, nv;
        float2 d;
    };
    auto load = [&](Pixel &a, bool valid, int x, int y, bool general) {
        a.x = x;
        a.y = y;
        const float rx = valid ? rtab_g[x + H] : 0.f, ry = valid ? rtab_g[y + H] : 0.f;
        const float c0 = rx * m[0] + ry * m[3];
        const float c1 = rx * m[1] + ry * m[4];
        const float c2 = rx * m[2] + ry * m[5];
        valid = valid && !(fabsf(c0) > 0.5f || fabsf(c1) >= 0.5f || fabsf(c2) >= 0.5f);
        // Util::round: half away from zero
        a.x0 = (int)(c0 * c.Pf + copysignf(0.5f, c0));
        a.y0 = (int)(c1 * c.Pf + copysignf(0.5f, c1));
        a.z0 = (int)(c2 * c.Pf + copysignf(0.5f, c2));
        const int x0 = a.x0, y0 = a.y0, z0 = a.z0;
        // Common voxel: |x0|, |y0|, |z0| < P/2 leave one direct and one
        // mirrored source cell, +-(x0, y0, z0) (on x0 = 0 the mirrored one
        // through the double insertion's conjugate copy, value only).  From
        // x >= 3 on, the own plane (pixels x >= 0) cannot reach the mirrored
        // cell, whose in-plane distance exceeds sqrt(3) + sqrt(3)/2; below,
        // its sources lie around (-x, -y), in the mirror patch.
        const bool common = fastkeys && (x >= 3 || mirror) && abs(x0) < H && abs(y0) < H && abs(z0) < H;
        a.later = valid && sub && !general && !common;
        a.now = valid && !a.later;
        a.vr = a.vi = a.nv = 0.f;
        a.d = make_float2(0.f, 0.f);
        if (a.now) {
            // the slice's floats 2x, 2x + 1 of row y; x = P/2 + 1 reads the next row's first, past the last row 0
            const unsigned fidx = (unsigned)(y < 0 ? P + y : y) * (unsigned)(H + 1) + (unsigned)x;
            if (fidx < (unsigned)P * (unsigned)(H + 1)) a.d = S[fidx];
            const int sg = x0 < 0 ? -1 : 1;
            const int ys = sg * y0, zs = sg * z0;
            const unsigned zi = (unsigned)(zs < 0 ? P + zs : zs), yi = (unsigned)(ys < 0 ? P + ys : ys);
            const unsigned xi = (unsigned)(sg * x0);
            if (PACKED) {
                const float4 v = vol[pack_index(xi, yi, zi, P)];
                a.vr = v.x;
                a.vi = v.y;
                a.nv = v.z;
            } else {
                const unsigned ci = (zi * P + yi) * (unsigned)(H + 1) + xi;  // P^2 (P/2 + 1) < 2^30
                const float2 v = data[ci];
                a.vr = v.x;
                a.vi = v.y;
                a.nv = norm[ci];
            }
        }
    };
    auto compare = [&](Pixel &a, bool general) {
        const int x0 = a.x0, y0 = a.y0, z0 = a.z0, r2d = a.x * a.x + a.y * a.y;
        const bool reach = a.now && r2d <= rown2;
        if (sub) {
            float ore = 0.f, oim = 0.f, ow = 0.f;
            if (general) {
                if (reach) {
                    const int sg = x0 < 0 ? -1 : 1, ys = sg * y0, zs = sg * z0;
                    own_contribution_tile(S, t3dp, nsym, own, pt, sg * x0, ys < 0 ? P + ys : ys, zs < 0 ? P + zs : zs, c,
                                          weight, etab, rtab, ore, oim, ow);
                }
            } else {
                float r = 0.f, i = 0.f, w = 0.f, r2 = 0.f, i2 = 0.f, w2 = 0.f;
                if (__ballot(reach)) {
                    // lanes without a pixel in reach gather around entry 0, in bounds, and drop the sums
                    const int e = reach ? (a.y - pt.y0) * AT_PX + (a.x - pt.x0) : 2 * AT_PX + 2;
                    gather_own_offsets<MODE>(ppx + e, olist, on, x0, y0, z0, c.h, weight, r, i, w);
                    const bool low = reach && a.x < 3;
                    if (__ballot(low)) {  // mirror patch entry of (-x, -y)
                        const int e2 = low ? 4 - a.x + (-a.y - my0) * AT_MX : 2 * AT_MX + 2;
                        gather_own_offsets<MODE>(mpx + e2, own_offset_list(omask, AT_MX), on, -x0, -y0, -z0, c.h, weight, r2, i2,
                                                 w2);
                    }
                    if (!reach) r = i = w = 0.f;
                    if (!low) r2 = i2 = w2 = 0.f;
                }
                // direct cell (x0, y0, z0) and mirrored -(x0, y0, z0), the volume's voxel being the mirrored
                // one of a cell with x0 < 0
                ore = r + r2;
                oim = i - i2;
                ow = x0 == 0 ? w : w + w2;
                if (SYM && reach) {
                    ore += (float)osum[a.l];
                    oim += (float)osum[NPX + a.l];
                    ow += (float)osum[2 * NPX + a.l];
                }
                oim = x0 >= 0 ? oim : -oim;
            }
            a.vr = a.vr - ore;
            a.vi = a.vi - oim;
            a.nv = a.nv - ow;
        }
        const float vr = a.vr, vi = x0 < 0 ? -a.vi : a.vi, nv = a.nv;  // get_complex_at conjugate for x<0
        if (a.now && nv != 0.f) {
            // value v over weight nv against d: dot and powers weighted by nv, nv cancelled once.  |v|^2 / nv with
            // nv = m 2^e, m in [1/2, 1): the exponent goes to one factor before the product (squares of v leave
            // the float range for weights from about 1e19 on and below 1e-19), 1 / m by a Newton step.
            const float dotv = vr * a.d.x + vi * a.d.y;
            const int e = __builtin_amdgcn_frexp_expf(nv);
            const float mn = __builtin_amdgcn_frexp_mantf(nv);
            float rm = __builtin_amdgcn_rcpf(mn);
            rm = __builtin_fmaf(__builtin_fmaf(-mn, rm, 1.0f), rm, rm);
            const float pw = __builtin_fmaf(vr, ldexpf(vr, -e), vi * ldexpf(vi, -e)) * rm;
            const float pw2 = (a.d.x * a.d.x + a.d.y * a.d.y) * nv;
            if (r2d > 9 && r2d < n3) {  // 3 < hypot_fast(x, y) < rmax
                acc[4] += dotv;
                acc[5] += pw;
                acc[6] += pw2;
            }
            acc[1] += nv;
            acc[0] += dotv;
            acc[2] += pw;
            acc[3] += pw2;
            nval++;
        }
    };
    // tile slot l -> pixel; in the x = 0 tiles the first slots are the columns
    // x < 3 of all rows, so that few waves run their mirrored gather
    auto slot = [&](int l, int &x, int &y) {
        if (tx0 == 0) {
            if (l < 3 * AY) {
                x = l % 3;
                y = ty0 + l / 3;
            } else {
                x = 3 + (l - 3 * AY) % (AT_X - 3);
                y = ty0 + (l - 3 * AY) / (AT_X - 3);
            }
        } else {
            x = tx0 + l % AT_X;
            y = ty0 + l / AT_X;
        }
    };
    // the voxels are read before the patch is staged: their latency runs beside it
    constexpr int NP = AY * AT_X / AT::THREADS;
    Pixel px[NP];
#pragma unroll
    for (int it = 0; it < NP; it++) {
        int x, y;
        slot(threadIdx.x + it * AT::THREADS, x, y);
        px[it].l = threadIdx.x + it * AT::THREADS;
        load(px[it], x < W && y < H && !(x == 0 && y == 0), x, y, false);
        if (SYM) cell[px[it].l] = ap_key(px[it].x0, px[it].y0, px[it].z0);
    }
    if (inner)
        for (int e = threadIdx.x; e < AT::PATCH; e += AT::THREADS)
            stage(pt.x0 + e % AT_PX, pt.y0 + e / AT_PX, ppx[e]);
    if (mirror && inner)
        for (int e = threadIdx.x; e < AT::MPATCH; e += AT::THREADS)
            stage(e % AT_MX - 4, my0 + e / AT_MX, mpx[e]);
    __syncthreads();
    if (SYM && fastkeys && inner) {
        // The other planes' contributions to the pixels' nearest cells and their mirrors, 64 planes at a time:
        // the (pixel, sign, plane) triples whose cell lies within the plane's reach are queued, so that full
        // waves run the gather for the few pixels along the planes' intersections, and summed per pixel: value
        // of the cell minus the conjugate of its mirror's, weights (the mirror's not on x0 = 0).  What the queue
        // does not hold is gathered at once.  The lanes come to a pixel in any order: summed in double and
        // rounded to float once, the sum does not show it (two terms give their float sum).
        for (int wd = 0; wd < nwords; wd++) {
            int *count = dn + 1 + (wd & 1);  // the other one is cleared before the barrier
            auto gather = [&](int e) {
                const int l = e & (NPX - 1), kc = cell[l], is = e >> 9 & 1 ? -1 : 1;
                const int x0 = (kc & 1023) - 512, y0 = (kc >> 10 & 1023) - 512, z0 = (kc >> 20) - 512;
                float a = 0.f, b = 0.f, g = 0.f;
                gather_cell(S, t3dp + 9 * (64 * wd + (e >> 10)), is * x0, is * y0, is * z0, c, weight, etab, rtab, a, b, g);
                if (a != 0.f || b != 0.f || g != 0.f) {
                    atomicAdd(&osum[l], (double)a);
                    atomicAdd(&osum[NPX + l], (double)(is < 0 ? -b : b));
                    if (is > 0 || x0 != 0) atomicAdd(&osum[2 * NPX + l], (double)g);
                }
            };
            for (unsigned long long ops = nwords <= 64 ? near_ops[wd] : ~0ull; ops; ops &= ops - 1) {
                const int k = __builtin_ctzll(ops), sop = 64 * wd + k;
                if (sop >= nsym) break;
                if (sop == own) continue;
                const float *o = t3dp + 9 * sop;
                const float n0 = o[1] * o[5] - o[2] * o[4], n1 = o[2] * o[3] - o[0] * o[5], n2 = o[0] * o[4] - o[1] * o[3];
#pragma unroll
                for (int it = 0; it < NP; it++) {
                    const Pixel &a = px[it];
                    const bool slab = a.now && a.x * a.x + a.y * a.y <= rown2 &&
                                      !(fabsf(n0 * a.x0 + n1 * a.y0 + n2 * a.z0) > 1.7330f);
                    const float s = o[0] * a.x0 + o[1] * a.y0 + o[2] * a.z0;  // gather_cell's x range is not empty
#pragma unroll
                    for (int sgn = 0; sgn < 2; sgn++) {
                        const bool hit = slab && (sgn ? s <= 1.74f : s >= -1.74f);
                        const unsigned long long hm = __ballot(hit);
                        if (!hm) continue;
                        int base = 0;
                        if (lane == 0) base = atomicAdd(count, __popcll(hm));
                        base = __builtin_amdgcn_readfirstlane(base) + __popcll(hm & ((1ull << lane) - 1ull));
                        if (hit) {
                            const int e = a.l | sgn << 9 | k << 10;
                            if (base < qcap) queue[base] = (unsigned short)e;
                            else gather(e);
                        }
                    }
                }
            }
            if (threadIdx.x == 0) dn[1 + ((wd + 1) & 1)] = 0;
            __syncthreads();
            const int n = min(*count, qcap);
            for (int k = threadIdx.x; k < n; k += AT::THREADS) gather(queue[k]);
            __syncthreads();
        }
    }
#pragma unroll
    for (int it = 0; it < NP; it++) {
        compare(px[it], false);
        if (px[it].later) dq[atomicAdd(dn, 1)] = (unsigned short)(threadIdx.x + it * AT::THREADS);
    }
    __syncthreads();
    for (int j = threadIdx.x; j < *dn; j += AT::THREADS) {
        int x, y;
        slot(dq[j], x, y);
        Pixel a;
        load(a, true, x, y, true);
        compare(a, true);
    }
    // block sums through LDS (the patch's space, no longer read): a wave per sum, or two sums per wave
    __syncthreads();
    static_assert(sizeof(AgreePx) * (AT::PATCH + AT::MPATCH) >= 8 * AT::THREADS * sizeof(double), "block sums");
    double *red = reinterpret_cast<double *>(ppx);  // 8 x THREADS doubles within the patches' bytes
#pragma unroll
    for (int k = 0; k < 7; k++) red[k * AT::THREADS + threadIdx.x] = acc[k];
    red[7 * AT::THREADS + threadIdx.x] = (double)nval;
    __syncthreads();
    constexpr int PER = AT::THREADS / 8;  // threads per sum: 64 or 32
    const int k = threadIdx.x / PER, l = threadIdx.x % PER;
    double v = 0.0;
#pragma unroll
    for (int i = 0; i < 8; i++) v += red[k * AT::THREADS + l + PER * i];
#pragma unroll
    for (int o = PER / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (l == 0) unsafeAtomicAdd(&acc_out[(size_t)p * 8 + k], v);
}

// One thread per entry, the 8 of a cube consecutive; cubes past x = P/2 (P/2 even) are half filled.
__global__ void __launch_bounds__(256) k_pack_volume(const float2 *__restrict__ data, const float *__restrict__ norm, int P,
                                                     float4 *__restrict__ vol)
{
    const unsigned H = P / 2, nbx = H / 2 + 1, n = nbx * H * H * 8;
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const unsigned b = i >> 3, x = 2 * (b % nbx) + (i & 1), yz = b / nbx;
        const unsigned y = 2 * (yz % H) + (i >> 1 & 1), z = 2 * (yz / H) + (i >> 2 & 1);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (x <= H) {
            const unsigned ci = (z * P + y) * (H + 1) + x;
            const float2 d = data[ci];
            v = make_float4(d.x, d.y, norm[ci], 0.f);
        }
        vol[i] = v;
    }
}

size_t pack_elems(int P) { return (size_t)(P / 4 + 1) * (P / 2) * (P / 2) * 8; }

hipError_t launch_pack_volume(const float2 *data, const float *norm, int P, float4 *vol, hipStream_t s)
{
    hipLaunchKernelGGL(k_pack_volume, dim3(8192), dim3(256), 0, s, data, norm, P, vol);
    return hipGetLastError();
}

hipError_t launch_agree_batch(const float2 *slices, int nsym, const float *t3d, const float *wq, int nslices,
                              InsertConst c, float rmax, int sub, const float2 *data, const float *norm,
                              const float4 *vol, const float *exptab, const float *rtab, double *acc, hipStream_t s)
{
    if (nslices <= 0) return hipSuccess;
    c.corners = 0;
    // the first n whose root, rounded to float, is not below rmax
    int n3 = std::max(0, (int)((double)rmax * rmax) - 2);
    while ((float)sqrt((double)n3) < rmax) n3++;
    const bool sym = nsym > 1;
    const int AY = sym ? 16 : 32;
    const int ntx = (c.P / 2 + 2 + AT_X - 1) / AT_X, nty = (c.P + AY - 1) / AY;
    const size_t patch = sym ? AgreeTile<16>::PATCH + AgreeTile<16>::MPATCH : AgreeTile<32>::PATCH + AgreeTile<32>::MPATCH;
    // With symmetry the other planes' queue takes what four workgroups per CU leave: 1,792 entries at pad 192, 976
    // at 600, the fewest (the compare pixels share it) from about pad 830 on.  Three workgroups: 7.2 ms instead of
    // 5.8 for 1,500 particles of d2 at pad 192.
    const int npx = AT_X * AY;
    const size_t fixed = sizeof(float) * EXPN + sizeof(AgreePx) * patch + 16 +
                         (sym ? 8 * std::min((nsym + 63) / 64, 64) + sizeof(float) * (c.P + 2) + (4 + 3 * 8) * npx : 0);
    const int qcap = sym ? (int)std::max<long long>(npx, ((40 << 10) - (long long)fixed) / 2) : npx;
    const size_t lds = fixed + sizeof(short) * qcap;
#define FH_AGREE(M, S, K)                                                                                               \
    if (c.mode == M && sym == S && (vol != nullptr) == K) {                                                             \
        hipLaunchKernelGGL((k_agree_batch<M, S, K>), dim3(ntx * nty, nslices), dim3(16 * AY), lds, s, slices, nsym, t3d, \
                           wq, c, n3, sub, qcap, data, norm, vol, exptab, rtab, acc);                                         \
        return hipGetLastError();                                                                                       \
    }
    FH_AGREE(0, false, false)
    FH_AGREE(0, false, true)
    FH_AGREE(0, true, false)
    FH_AGREE(0, true, true)
    FH_AGREE(1, false, false)
    FH_AGREE(1, false, true)
    FH_AGREE(1, true, false)
    FH_AGREE(1, true, true)
#undef FH_AGREE
    return hipErrorInvalidValue;
}

// ------------------------------------------------------------ projection
// FourierReconstructor::projection (libEM/reconstructor.cpp:1383-1445): the
// slice pixel (x, y) takes the nearest voxel's value over its weight
// (pixel_at, :1448-1461) when the weight is at least 0.005, halved on the
// x = 0 column.  The result is what set_complex_at (emdata_core.cpp:171-205)
// leaves in the (P+2) x P image after the reference's loop: on the x = 0 and
// x = P/2 columns each pixel also writes its conjugate at -y, so a stored
// row holds the later of the two iterations that write it (y > 0 comes after
// y < 0), rows 0 and P/2 keep the real part only.
__device__ __forceinline__ bool project_pixel(int x, int y, const Mat9 &m, const InsertConst &c,
                                              const float *__restrict__ rtab, const float2 *__restrict__ data,
                                              const float *__restrict__ norm, float &re, float &im)
{
    const int H = c.H, P = c.P;
    const float rx = rtab[x + H], ry = rtab[y + H];
    const float c0 = rx * m.m[0] + ry * m.m[3];
    const float c1 = rx * m.m[1] + ry * m.m[4];
    const float c2 = rx * m.m[2] + ry * m.m[5];
    if (fabsf(c0) > 0.5f || fabsf(c1) >= 0.5f || fabsf(c2) >= 0.5f) return false;
    const int x0 = round_ref(c0 * c.Pf), y0 = round_ref(c1 * c.Pf), z0 = round_ref(c2 * c.Pf);
    size_t ci;
    if (x0 < 0) ci = cidx(-x0, y0 <= 0 ? -y0 : P - y0, z0 <= 0 ? -z0 : P - z0, P, H);
    else ci = cidx(x0, y0 < 0 ? P + y0 : y0, z0 < 0 ? P + z0 : z0, P, H);
    const float nv = norm[ci];
    if ((double)nv < 0.005) return false;  // dt[2] < 0.005, a double comparison
    const float2 v = data[ci];
    re = __fdiv_rn(v.x, nv);
    im = __fdiv_rn(x0 < 0 ? -v.y : v.y, nv);
    if (x == 0 && y != 0 && y != -H) {
        re /= 2;
        im /= 2;
    }
    return true;
}

// shift: the translation's phase ramp of the "xform" processor's complex
// branch (libEM/processor.cpp:11081-11176; with no rotation its bilinear
// weights are exactly 1, 0, 0, 0), the reference's long double pi
// arithmetic restated in double.  center: xform.phaseorigin.tocenter on the
// complex image, x (-1)^(x + row) (sparx/emdata_sparx.cpp:8451-8460).
__global__ void __launch_bounds__(256) k_project(const float2 *__restrict__ data, const float *__restrict__ norm,
                                                 InsertConst c, Mat9 m, const float *__restrict__ rtab, float xshift,
                                                 float yshift, int shift, int center, float2 *__restrict__ out)
{
    const int H = c.H, P = c.P;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= P * (H + 1)) return;
    const int x = idx % (H + 1), r = idx / (H + 1);
    float re = 0.f, im = 0.f, pr, pim;
    if (x != 0 && x != H) {
        if (!project_pixel(x, r < H ? r : r - P, m, c, rtab, data, norm, re, im)) re = im = 0.f;
    } else if (r == 0 || r == H) {
        if (project_pixel(x, r == 0 ? 0 : -H, m, c, rtab, data, norm, pr, pim)) re = pr;
    } else {
        const int a = r < H ? r : P - r;
        if (project_pixel(x, a, m, c, rtab, data, norm, pr, pim)) {
            re = pr;
            im = r < H ? pim : -pim;
        } else if (project_pixel(x, -a, m, c, rtab, data, norm, pr, pim)) {
            re = pr;
            im = r < H ? -pim : pim;
        }
    }
    if (shift) {
        const double pi = 3.141592653589793238462643383279502884;
        const int ky = r >= H + 1 ? r - P : r;
        const float phaseY = (float)(-2 * pi * ky * (double)yshift / P);
        const float phase = (float)((double)phaseY - 2 * pi * x * (double)xshift / P);
        const double cp = cos((double)phase), sp = sin((double)phase);
        const float rb = (float)((double)re * cp - (double)im * sp);
        const float ib = (float)((double)re * sp + (double)im * cp);
        re = rb;
        im = ib;
    }
    if (center && ((x + r) & 1)) {
        re = -re;
        im = -im;
    }
    out[idx] = make_float2(re, im);
}

hipError_t launch_project(const float2 *data, const float *norm, InsertConst c, const float *rot9, const float *rtab,
                          float xshift, float yshift, int center, float2 *out, hipStream_t s)
{
    Mat9 m;
    for (int i = 0; i < 9; i++) m.m[i] = rot9[i];
    const int n = c.P * (c.H + 1);
    const int shift = xshift != 0.0f || yshift != 0.0f;
    hipLaunchKernelGGL(k_project, dim3((n + 255) / 256), dim3(256), 0, s, data, norm, c, m, rtab, xshift, yshift, shift,
                       center, out);
    return hipGetLastError();
}

// ------------------------------------------------------------ gauss_fft projector
// GaussFFTProjector::project3d (libEM/projector.cpp:69-212) and interp_ft_3d
// (:216-295) for modes 0-2 on the map's transform kept in the volume layout
// (phase origin at the corner, rows and planes in wrap order).  The
// reference interpolates the complex volume with its Fourier origin moved
// to the centre in y and z and reads it by linear float index
// 2 x + y (P+2) + z (P+2) P; pv_lin maps such an index (0 outside the array)
// back to the wrap-ordered storage.  Per projection q: rec[12 q ..] =
// inverse rotation rows (9), scale, tx, ty.  Output element (x, r) of
// projection q is the slice pixel (x, row (r + P/2) mod P of the centred
// slice): the Fourier origin back in the corner.
__device__ __forceinline__ float pv_lin(const float2 *__restrict__ pv, long long L, int P, int H)
{
    const int nx = P + 2;
    if (L < 0 || L >= (long long)nx * P * P) return 0.f;
    const int xr = (int)(L % nx);
    const long long q = L / nx;
    const int y = (int)(q % P), z = (int)(q / P);
    const float2 v = pv[cidx(xr >> 1, y + H < P ? y + H : y + H - P, z + H < P ? z + H : z + H - P, P, H)];
    return (xr & 1) ? v.y : v.x;
}

__device__ __forceinline__ float agauss_f(float a, float dx, float dy, float dz, float d)
{
    return a * expf(-(dx * dx + dy * dy + dz * dz) / d);  // Util::agauss (util.h:912-915)
}

__device__ bool gfft_interp(int mode, const float2 *__restrict__ pv, int P, int H, float x, float y, float z,
                            float &d0, float &d1, float gw)
{
    const int nx = P + 2, ny = P, nz = P;
    if (mode == 0) {
        const int x0 = (int)floor(x), y0 = (int)floor(y), z0 = (int)floor(z);
        float a0 = 0.f, a1 = 0.f, nrm = 0.f;
        for (int ix = x0; ix <= x0 + 1; ix++)
            for (int iy = y0; iy <= y0 + 1; iy++)
                for (int iz = z0; iz <= z0 + 1; iz++) {
                    const float w = (float)((1.0 - (double)fabsf((float)ix - x)) * (1.0 - (double)fabsf((float)iy - y)) *
                                            (1.0 - (double)fabsf((float)iz - z)));
                    const long long L = 2LL * ix + (long long)iy * nx + (long long)iz * nx * ny;
                    a0 += w * pv_lin(pv, L, P, H);
                    a1 += w * pv_lin(pv, L + 1, P, H);
                    nrm += w;
                }
        d0 = a0 / nrm;
        d1 = a1 / nrm;
        return true;
    }
    if (mode == 1) {
        const int x0 = 2 * (int)floor(x + 0.5f), y0 = (int)floor(y + 0.5f), z0 = (int)floor(z + 0.5f);
        const long long L = (long long)x0 + (long long)y0 * nx + (long long)z0 * nx * ny;
        d0 = pv_lin(pv, L, P, H);
        d1 = pv_lin(pv, L + 1, P, H);
        return true;
    }
    const int x0 = (int)floor(x), y0 = (int)floor(y), z0 = (int)floor(z);
    const float dx = x - x0, dy = y - y0, dz = z - z0;
    if (!(x0 <= nx / 2 - 2 && y0 <= ny - 1 && z0 <= nz - 1)) return false;
    const long long i0 = (long long)x0 * 2 + (long long)y0 * nx + (long long)z0 * nx * ny;
    const float n = agauss_f(1, dx, dy, dz, gw) + agauss_f(1, 1 - dx, dy, dz, gw) + agauss_f(1, dx, 1 - dy, dz, gw) +
                    agauss_f(1, 1 - dx, 1 - dy, dz, gw) + agauss_f(1, dx, dy, 1 - dz, gw) +
                    agauss_f(1, 1 - dx, dy, 1 - dz, gw) + agauss_f(1, dx, 1 - dy, 1 - dz, gw) +
                    agauss_f(1, 1 - dx, 1 - dy, 1 - dz, gw);
    float d[2];
    for (int c = 0; c < 2; c++) {
        const long long i = i0 + c;
        const long long nxy = (long long)nx * ny;
        // the reference divides its last term only by n (operator precedence)
        d[c] = agauss_f(pv_lin(pv, i, P, H), dx, dy, dz, gw) + agauss_f(pv_lin(pv, i + 2, P, H), 1 - dx, dy, dz, gw) +
               agauss_f(pv_lin(pv, i + nx, P, H), dx, 1 - dy, dz, gw) +
               agauss_f(pv_lin(pv, i + nx + 2, P, H), 1 - dx, 1 - dy, dz, gw) +
               agauss_f(pv_lin(pv, i + nxy, P, H), dx, dy, 1 - dz, gw) +
               agauss_f(pv_lin(pv, i + 2 + nxy, P, H), 1 - dx, dy, 1 - dz, gw) +
               agauss_f(pv_lin(pv, i + nx + nxy, P, H), dx, 1 - dy, 1 - dz, gw) +
               agauss_f(pv_lin(pv, i + 2 + nx + nxy, P, H), 1 - dx, 1 - dy, 1 - dz, gw) / n;
    }
    d0 = d[0];
    d1 = d[1];
    return true;
}

// ramp: the translation's phase ramp (the "xform" processor's complex
// branch, as in k_project), for the Fourier-slice output
__global__ void __launch_bounds__(256) k_gauss_fft(const float2 *__restrict__ pv, int P, int mode, float gw,
                                                   const float *__restrict__ rec, int ramp, float2 *__restrict__ out)
{
    const int H = P / 2;
    const int q = blockIdx.y;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= P * (H + 1)) return;
    const int x = idx % (H + 1), r = idx / (H + 1);
    const int yc = r + H < P ? r + H : r + H - P;  // the centred slice's row
    const float *m = rec + 12 * (size_t)q;
    float re = 0.f, im = 0.f;
    const int yy_i = yc - P / 2;
    if ((long long)x * x + (long long)yy_i * yy_i < (long long)(P / 2 - 1) * (P / 2 - 1)) {
        const float cx = (float)x, cy = (float)yy_i, cz = 0.0f;
        float xx = m[0] * cx + m[1] * cy + m[2] * cz + 0.0f;
        float yy = m[3] * cx + m[4] * cy + m[5] * cz + 0.0f;
        float zz = m[6] * cx + m[7] * cy + m[8] * cz + 0.0f;
        int cc = 1;
        if (xx < 0) {
            xx = -xx;
            yy = -yy;
            zz = -zz;
            cc = -1;
        }
        const float scale = m[9];
        if (scale != 1.0f) {
            xx *= scale;
            yy *= scale;
            zz *= scale;
        }
        yy += (float)(P / 2);
        zz += (float)(P / 2);
        if (!(yy < 0 || xx < 0 || zz < 0)) {
            float d0, d1;
            if (gfft_interp(mode, pv, P, H, xx, yy, zz, d0, d1, gw)) {
                re = d0;
                im = d1 * (float)cc;
            }
        }
    }
    const float xshift = m[10], yshift = m[11];
    if (ramp && (xshift != 0.0f || yshift != 0.0f)) {
        const double pi = 3.141592653589793238462643383279502884;
        const int ky = r >= H + 1 ? r - P : r;
        const float phaseY = (float)(-2 * pi * ky * (double)yshift / P);
        const float phase = (float)((double)phaseY - 2 * pi * x * (double)xshift / P);
        const double cp = cos((double)phase), sp = sin((double)phase);
        const float rb = (float)((double)re * cp - (double)im * sp);
        const float ib = (float)((double)re * sp + (double)im * cp);
        re = rb;
        im = ib;
    }
    out[(size_t)q * P * (H + 1) + idx] = make_float2(re, im);
}

// math.gausskernelfix on n P x P images (MaskGaussInvProcessor,
// processor.h:4131-4176): each pixel over exp(-dist sv), dist the squared
// distance from (P/2, P/2), sv = gauss_width / P^2
__global__ void k_gausskernelfix2d(float *__restrict__ img, int P, int n, float sv)
{
    const size_t tot = (size_t)n * P * P;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < tot; i += (size_t)gridDim.x * blockDim.x) {
        const int x = (int)(i % P), y = (int)((i / P) % P);
        const float xc = (float)(P / 2), yc = (float)(P / 2);
        const float dist = ((float)x - xc) * ((float)x - xc) + ((float)y - yc) * ((float)y - yc) + 0.0f;
        img[i] = img[i] / expf(-dist * sv);
    }
}

hipError_t launch_gauss_fft(const float2 *pv, int P, int n, int mode, float gw, const float *rec, int ramp,
                            float2 *out, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const int m = P * (P / 2 + 1);
    hipLaunchKernelGGL(k_gauss_fft, dim3((m + 255) / 256, n), dim3(256), 0, s, pv, P, mode, gw, rec, ramp, out);
    return hipGetLastError();
}

hipError_t launch_gausskernelfix2d(float *img, int P, int n, float gauss_width, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const float sv = gauss_width / (float)(P * P);
    const unsigned blocks = (unsigned)std::min<size_t>(((size_t)n * P * P + 255) / 256, 65536);
    hipLaunchKernelGGL(k_gausskernelfix2d, dim3(blocks), dim3(256), 0, s, img, P, n, sv);
    return hipGetLastError();
}

hipError_t launch_agree(const float2 *slices, int nsym, const float *t3d, int nslices, InsertConst c, float rmax,
                        const float2 *data, const float *norm, const float *rtab, double *partial, hipStream_t s)
{
    if (nslices <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_agree, dim3(agree_blocks(c.P), nslices), dim3(256), 0, s, slices, nsym, t3d, c, rmax, data,
                       norm, rtab, partial);
    return hipGetLastError();
}

// ------------------------------------------------------------ binning
// Brick b = (bx, by, bz) owns the stencil origins [lo, lo + bs) per axis,
// lo = ow + bs*b: a pixel is added by the one brick holding its stencil
// origin, i.e. p in [po + bs*b, po + bs*(b+1)) on every axis (for gauss_2
// the origin is floor(p), po = ow = -H-1, and the 8 corners land in the
// brick's (bs+1)^3 cells [lo, lo+bs]^3).  Pixel positions lie on the
// plane n.p = 0 (n = u x v of the slice's t3d rows), so per brick column
// along the dominant normal axis at most 4 bricks qualify.  A slice is
// binned under key 3 * brick + (its dominant normal axis), so that every
// work item's slices share one column direction.
//
// The binning is owned by brick columns: one workgroup per (column, axis)
// runs over the slices of that dominant axis and counts / lists the
// column's bricks in LDS, so no (slice, brick) pair touches a global atomic.

// Per slice: the plane record, appended to the segment of its dominant axis
// (one atomic per wave and axis).  Weight-0 slices are skipped
// (reconstructor.cpp:1088).
__global__ void __launch_bounds__(256) k_slice_recs(const float *__restrict__ t3d, const float *__restrict__ wq,
                                                    int nslices, BinBuffers bb)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    int a = -1;
    SliceRec r;
    if (q < nslices && wq[q] != 0.0f) {
        const float *m = t3d + 9 * (size_t)q;
        double u[3], v[3];
        for (int d = 0; d < 3; d++) {
            r.u[d] = m[d];
            r.v[d] = m[3 + d];
            u[d] = m[d];
            v[d] = m[3 + d];
        }
        const double n[3] = {u[1] * v[2] - u[2] * v[1], u[2] * v[0] - u[0] * v[2], u[0] * v[1] - u[1] * v[0]};
        const double a0 = fabs(n[0]), a1 = fabs(n[1]), a2 = fabs(n[2]);
        a = (a0 >= a1 && a0 >= a2) ? 0 : (a1 >= a2 ? 1 : 2);
        const int b1 = a == 0 ? 1 : 0, b2 = a == 2 ? 1 : 2;
        r.r1 = -n[b1] / n[a];
        r.r2 = -n[b2] / n[a];
        r.q = q;
        r.pad = 0;
    }
#pragma unroll
    for (int ax = 0; ax < 3; ax++) {
        const unsigned long long m = __ballot(a == ax);
        if (m == 0) continue;
        const int leader = __ffsll((long long)m) - 1;
        int base = 0;
        if (lane == leader) base = atomicAdd(&bb.ctl[4 + ax], __popcll(m));
        base = __shfl(base, leader, 64);
        if (a == ax) {
            const int rank = __popcll(m & ((1ull << lane) - 1ull));
            bb.recs[(size_t)ax * bb.rec_cap + base + rank] = r;
        }
    }
}

constexpr int BIN_COLS = 2;  // brick columns per workgroup
// One workgroup per (brick columns (c1 .. c1 + BIN_COLS - 1, c2), axis a): MODE 0 counts the
// slices of each brick of the column, MODE 1 lists them from the key
// offsets on.  LDS: one counter per brick of the column.
// Bound by the slice records, read once per workgroup (48 bytes times
// bricks per plane), and the double-precision work on them: two columns share
// a read, a slice's range along the column takes the reciprocal of the brick
// edge, its distance from a brick's centre one FMA from the column's part.
// Both modes together 1.97 -> 1.14 ms for 112,000 slices at pad 288 (1.50 with
// one column), 1.32 -> 0.72 for 8,000 of gauss_var at 384 (3 x 3 x 5 bricks;
// 1.02); four columns take as long there and 24 instead of 16 us for 2,000
// slices at pad 96.
template <int MODE>
__global__ void __launch_bounds__(256) k_bin_cols(InsertConst c, BrickGeom g, BinBuffers bb)
{
    extern __shared__ int colcnt[];
    const int nb = g.nb, H = c.H;
    const double po = g.po;
    const int A = blockIdx.y, cols = (nb + BIN_COLS - 1) / BIN_COLS;
    const int c1 = (blockIdx.x % cols) * BIN_COLS, c2 = blockIdx.x / cols;
    const int b1 = A == 0 ? 1 : 0, b2 = A == 2 ? 1 : 2;
    const int bs[3] = {g.bs, g.bs, g.bsz};
    const int na = A == 2 ? g.nbz : nb;  // bricks of a column
    const int nc = min(BIN_COLS, nb - c1);
    if (c2 >= (b2 == 2 ? g.nbz : nb)) return;
    auto key = [&](int i) {  // of entry i of the columns' bricks, column after column
        int bc[3];
        bc[b1] = c1 + i / na;
        bc[b2] = c2;
        bc[A] = i % na;
        return 3 * ((bc[2] * nb + bc[1]) * nb + bc[0]) + A;
    };
    for (int i = threadIdx.x; i < nc * na; i += blockDim.x) colcnt[i] = MODE == 0 ? 0 : bb.offsets[key(i)];
    __syncthreads();
    const double dlt = 1e-3;
    const double L2 = po + bs[b2] * c2 - dlt, U2 = po + bs[b2] * c2 + bs[b2] + dlt;
    // does the slice's pixel domain (half-disk x >= 0 of radius sqrt(H^2+H), or
    // the half-square with corners) come within reach of the brick?
    const double rh = 0.5 * sqrt((double)(2 * g.bs * g.bs + g.bsz * g.bsz)) + 0.01;  // its half diagonal and a margin
    const double rr = sqrt((double)c.rcut * c.rcut + c.rcut) + rh, rr2 = rr * rr;
    const double e2 = po + bs[b2] * c2 + 0.5 * bs[b2];  // the bricks' centres
    const double ea = po + 0.5 * bs[A], ba = bs[A], inv = 1.0 / bs[A];
    const int n = bb.ctl[4 + A];
    const SliceRec *recs = bb.recs + (size_t)A * bb.rec_cap;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const SliceRec f = recs[i];
        const double l2 = f.r2 * L2, u2 = f.r2 * U2, min2 = fmin(l2, u2) - dlt - po, max2 = fmax(l2, u2) + dlt - po;
        const double ua = A == 0 ? f.u[0] : A == 1 ? f.u[1] : f.u[2], va = A == 0 ? f.v[0] : A == 1 ? f.v[1] : f.v[2];
        const double ub = A == 0 ? f.u[1] : f.u[0], vb = A == 0 ? f.v[1] : f.v[0];
        const double s2 = e2 * (double)(A == 2 ? f.u[1] : f.u[2]), t2 = e2 * (double)(A == 2 ? f.v[1] : f.v[2]);
#pragma unroll
        for (int k = 0; k < BIN_COLS; k++) {
            if (k >= nc) break;
            const double org = po + bs[b1] * (c1 + k), e1 = org + 0.5 * bs[b1];
            const double l1 = f.r1 * (org - dlt), u1 = f.r1 * (org + bs[b1] + dlt);
            int lo = (int)floor((fmin(l1, u1) + min2) * inv);
            int hi = (int)floor((fmax(l1, u1) + max2) * inv);
            if (lo < 0) lo = 0;
            if (hi > na - 1) hi = na - 1;
            const double s0 = __builtin_fma(e1, ub, s2), t0 = __builtin_fma(e1, vb, t2);
            for (int ca = lo; ca <= hi; ca++) {
                const double cen = __builtin_fma(ba, (double)ca, ea);
                const double sd = __builtin_fma(cen, ua, s0), td = __builtin_fma(cen, va, t0);
                if (sd < -rh) continue;
                if (c.corners ? (sd > H + rh || td < -H - rh || td > H - 1 + rh) : sd * sd + td * td > rr2) continue;
                const int pos = atomicAdd(&colcnt[k * na + ca], 1);
                if (MODE == 1) {
                    if (pos < bb.list_cap) bb.list[pos] = f.q;
                    else bb.ctl[3] = 1;
                }
            }
        }
    }
    if (MODE == 0) {
        __syncthreads();
        for (int i = threadIdx.x; i < nc * na; i += blockDim.x) bb.counts[key(i)] = colcnt[i];
    }
}

// Exclusive scans of the key counts (-> list offsets) and of the work items
// per key (ceil(count / K) -> item offsets) in three passes: per-tile sums,
// a scan of the tile sums with the totals, and the per-key offsets.  With
// per_brick the items of a brick span its three axis keys (whose lists are
// consecutive): key 3b holds ceil((c[3b] + c[3b+1] + c[3b+2]) / K) items,
// keys 3b+1 and 3b+2 none.
constexpr int SCAN_TILE = 1024;  // keys per tile: 256 threads x 4

__device__ __forceinline__ int key_items(const int *__restrict__ counts, int k, int nkeys, int ck, int K,
                                         int per_brick)
{
    if (!per_brick) return (ck + K - 1) / K;
    if (k % 3) return 0;
    const int c = ck + (k + 1 < nkeys ? counts[k + 1] : 0) + (k + 2 < nkeys ? counts[k + 2] : 0);
    return (c + K - 1) / K;
}

__device__ __forceinline__ int4 load_counts4(const int *counts, int k, int n)
{
    if (k + 3 < n) return *reinterpret_cast<const int4 *>(counts + k);
    int4 v;
    v.x = k < n ? counts[k] : 0;
    v.y = k + 1 < n ? counts[k + 1] : 0;
    v.z = k + 2 < n ? counts[k + 2] : 0;
    v.w = 0;
    return v;
}

// 256-thread exclusive scan of (a, b); returns the block totals
__device__ __forceinline__ void block_scan2(int &a, int &b, int &ta, int &tb)
{
    __shared__ int sa[4], sb[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int ia = a, ib = b;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int va = __shfl_up(ia, off, 64), vb = __shfl_up(ib, off, 64);
        if (lane >= off) {
            ia += va;
            ib += vb;
        }
    }
    if (lane == 63) {
        sa[wave] = ia;
        sb[wave] = ib;
    }
    __syncthreads();
    int pa = 0, pb = 0;
    for (int w = 0; w < wave; w++) {
        pa += sa[w];
        pb += sb[w];
    }
    ta = sa[0] + sa[1] + sa[2] + sa[3];
    tb = sb[0] + sb[1] + sb[2] + sb[3];
    a = pa + ia - a;
    b = pb + ib - b;
}

__global__ void __launch_bounds__(256) k_scan_tiles(BrickGeom g, BinBuffers bb, int K)
{
    const int k = blockIdx.x * SCAN_TILE + threadIdx.x * 4;
    const int4 c = load_counts4(bb.counts, k, g.nkeys);
    const int cv[4] = {c.x, c.y, c.z, c.w};
    int a = c.x + c.y + c.z + c.w;
    int b = 0;
#pragma unroll
    for (int t = 0; t < 4; t++)
        if (k + t < g.nkeys) b += key_items(bb.counts, k + t, g.nkeys, cv[t], K, g.per_brick);
    int ta, tb;
    block_scan2(a, b, ta, tb);
    if (threadIdx.x == 0) {
        bb.tile[2 * blockIdx.x] = ta;
        bb.tile[2 * blockIdx.x + 1] = tb;
    }
}

__global__ void __launch_bounds__(1024) k_scan_top(BrickGeom g, BinBuffers bb, int ntiles)
{
    const int tid = threadIdx.x;
    const int per = (ntiles + 1023) / 1024;
    const int t0 = tid * per, t1 = min(ntiles, t0 + per);
    long long sc = 0, si = 0;
    for (int t = t0; t < t1; t++) {
        sc += bb.tile[2 * t];
        si += bb.tile[2 * t + 1];
    }
    __shared__ long long s_c[1024], s_i[1024];
    s_c[tid] = sc;
    s_i[tid] = si;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const long long vc = tid >= off ? s_c[tid - off] : 0;
        const long long vi = tid >= off ? s_i[tid - off] : 0;
        __syncthreads();
        s_c[tid] += vc;
        s_i[tid] += vi;
        __syncthreads();
    }
    long long ec = s_c[tid] - sc, ei = s_i[tid] - si;
    for (int t = t0; t < t1; t++) {
        const int a = bb.tile[2 * t], b = bb.tile[2 * t + 1];
        bb.tile[2 * t] = (int)ec;
        bb.tile[2 * t + 1] = (int)ei;
        ec += a;
        ei += b;
    }
    if (tid == 1023) {
        const long long tc = s_c[1023], ti = s_i[1023];
        bb.offsets[g.nkeys] = (int)tc;
        bb.item_off[g.nkeys] = (int)ti;
        bb.ctl[0] = 0;
        bb.ctl[1] = (int)(ti < bb.item_cap ? ti : bb.item_cap);
        bb.ctl[2] = (int)(tc < bb.list_cap ? tc : bb.list_cap);
        if (tc > bb.list_cap || ti > bb.item_cap) bb.ctl[3] = 1;
    }
}

__global__ void __launch_bounds__(256) k_scan_apply(BrickGeom g, BinBuffers bb, int K)
{
    const int k = blockIdx.x * SCAN_TILE + threadIdx.x * 4;
    const int4 c = load_counts4(bb.counts, k, g.nkeys);
    const int cv[4] = {c.x, c.y, c.z, c.w};
    int iv[4];
#pragma unroll
    for (int t = 0; t < 4; t++) iv[t] = k + t < g.nkeys ? key_items(bb.counts, k + t, g.nkeys, cv[t], K, g.per_brick) : 0;
    int a = c.x + c.y + c.z + c.w;
    int b = iv[0] + iv[1] + iv[2] + iv[3];
    int ta, tb;
    block_scan2(a, b, ta, tb);
    a += bb.tile[2 * blockIdx.x];
    b += bb.tile[2 * blockIdx.x + 1];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        if (k + t < g.nkeys) {
            bb.offsets[k + t] = a;
            bb.item_off[k + t] = b;
        }
        a += cv[t];
        b += iv[t];
    }
}

int scan_tiles(const BrickGeom &g) { return (g.nkeys + SCAN_TILE - 1) / SCAN_TILE; }

__global__ void k_bin_items(BrickGeom g, BinBuffers bb, int K)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= g.nkeys) return;
    if (g.per_brick && b % 3) return;  // the brick's items are listed under key 3 * brick
    const int cnt = g.per_brick ? bb.counts[b] + (b + 1 < g.nkeys ? bb.counts[b + 1] : 0) +
                                      (b + 2 < g.nkeys ? bb.counts[b + 2] : 0)
                                : bb.counts[b];
    const int base = bb.item_off[b];
    const int off = bb.offsets[b];
    for (int i = 0; i * K < cnt; i++) {
        if ((long long)base + i >= bb.item_cap) break;
        WorkItem w;
        w.key = b;
        w.start = off + i * K;
        w.count = min(K, cnt - i * K);
        if ((long long)w.start + w.count > bb.list_cap) w.count = (int)max(0LL, bb.list_cap - w.start);
        w.pad = 0;
        bb.items[base + i] = w;
    }
}

hipError_t launch_bin(const float *t3d, const float *wq, int nslices, InsertConst c, BrickGeom g, BinBuffers b,
                      int K, hipStream_t s)
{
    hipError_t e;
    if (nslices > b.rec_cap) return hipErrorInvalidValue;
    if ((e = launch_fill_i32(b.counts, 0, g.nkeys, s)) != hipSuccess) return e;
    if ((e = launch_fill_i32(b.ctl, 0, 8, s)) != hipSuccess) return e;
    const dim3 cgrid((g.nb + BIN_COLS - 1) / BIN_COLS * std::max(g.nb, g.nbz), 3);
    const size_t clds = sizeof(int) * BIN_COLS * std::max(g.nb, g.nbz);
    if (nslices > 0) {
        hipLaunchKernelGGL(k_slice_recs, dim3((nslices + 255) / 256), dim3(256), 0, s, t3d, wq, nslices, b);
        hipLaunchKernelGGL(k_bin_cols<0>, cgrid, dim3(256), clds, s, c, g, b);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    const int nt = scan_tiles(g);
    hipLaunchKernelGGL(k_scan_tiles, dim3(nt), dim3(256), 0, s, g, b, K);
    hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, s, g, b, nt);
    hipLaunchKernelGGL(k_scan_apply, dim3(nt), dim3(256), 0, s, g, b, K);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (nslices > 0) {
        hipLaunchKernelGGL(k_bin_cols<1>, cgrid, dim3(256), clds, s, c, g, b);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_bin_items, dim3((g.nkeys + 255) / 256), dim3(256), 0, s, g, b, K);
    return hipGetLastError();
}

// ------------------------------------------------------------ brick scatter insertion
// A work item is (brick of 8^3 stencil origins, axis A, up to K slices whose
// dominant normal axis is A).  Its wave owns a private accumulator of the
// brick's 9^3 cells in LDS and walks the slice pixels whose stencil origin
// lies in the brick in windows of 64 (one pixel per lane), adding each
// pixel's 8 corners with plain LDS read-modify-writes; every pixel is added
// by exactly one brick, and the cells on a brick's high faces are summed
// with the next bricks' in the merge:
//  - two lanes whose pixels share a stencil origin cell would race on all
//    eight corners; an LDS tag per origin cell elects one lane per cell, the
//    others stay pending for the next window (no atomics);
//  - two lanes with different origins can still meet on a cell through
//    different corners, so the corners are processed one after another with
//    a wave-level ordering point between them.
// The accumulator is three float arrays (re, im, w) over the cells in
// [A][B2][B1] order (B1 < B2 the other axes): one corner's cells of a slice
// with dominant axis A fall in distinct (B1, B2) columns, so the lanes of an
// access spread over the 32 banks.
constexpr int ACC_N = HALO_CELLS;                      // cells per field
constexpr int TAG_N = BRICK * BRICK * BRICK;           // stencil origins in [lo, lo+7]^3
constexpr int ACC_BYTES = (12 * ACC_N + 15) & ~15;     // re, im, w
constexpr int REC_OFF = ACC_BYTES;                     // slice records: 2 float4 per slice of a group
constexpr int MARK_OFF = REC_OFF + 16 * 8;             // 64 row marks
constexpr int TAG_OFF = MARK_OFF + 4 * 64;             // one byte per origin
constexpr int WAVE_LDS_BYTES = TAG_OFF + TAG_N;
#define SC_DLT 2e-3f   // margin on p: the FP32 position error is < 3e-4 for P <= 1024
#define SC_EPS 1e-3f   // margin on enumeration bounds
#define SC_RAD 6.95f   // 4 sqrt(3) + margin: |p - brick centre| for an origin in [lo, lo+7]^3

template <int A>
__device__ __forceinline__ int acc_slot(int i, int j, int k)
{
    return A == 0 ? (i * HALO + k) * HALO + j : (A == 1 ? (j * HALO + k) * HALO + i : (k * HALO + j) * HALO + i);
}

// Wave64 inclusive scans on DPP (GFX9 row shifts and row broadcasts): no
// LDS traffic.  Lanes without a source keep the identity.
#define DPP_ROW_SHR(n) (0x110 + (n))
#define DPP_ROW_BCAST15 0x142
#define DPP_ROW_BCAST31 0x143
__device__ __forceinline__ int wave_scan_add(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR(1), 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR(2), 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR(4), 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR(8), 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_BCAST15, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_BCAST31, 0xc, 0xf, false);
    return v;
}
__device__ __forceinline__ int wave_scan_max(int v)
{
    const int lo = -2147483647 - 1;
    v = max(v, __builtin_amdgcn_update_dpp(lo, v, DPP_ROW_SHR(1), 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(lo, v, DPP_ROW_SHR(2), 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(lo, v, DPP_ROW_SHR(4), 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(lo, v, DPP_ROW_SHR(8), 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(lo, v, DPP_ROW_BCAST15, 0xa, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(lo, v, DPP_ROW_BCAST31, 0xc, 0xf, false));
    return v;
}

// floor(sqrt(n)) for 0 <= n < 2^24
__device__ __forceinline__ int isqrt24(int n)
{
    int r = (int)__builtin_amdgcn_sqrtf((float)n);
    r -= (r * r > n);
    r += ((r + 1) * (r + 1) <= n);
    return r;
}

// gauss_2 / trilinear weights of the 8 corners (floor(p) + (di, dj, dk)),
// corner index di + 2 dj + 4 dk; each equals corner_weight() bit for bit.
// gauss_2's table index is read off the bits of one FMA rounded toward zero
// (see g6_entries); the table starts the kernel's LDS.
__device__ __forceinline__ void corner_weights8(int mode, float xx, float yy, float zz, float h, float weight, float wg[8])
{
    const float fx = floorf(xx), fy = floorf(yy), fz = floorf(zz);
    const float dx[2] = {fx - xx, (fx + 1.0f) - xx};
    const float dy[2] = {fy - yy, (fy + 1.0f) - yy};
    const float dz[2] = {fz - zz, (fz + 1.0f) - zz};
    if (mode == 0) {
        float f[8];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const float sxy = dx[b & 1] * dx[b & 1] + dy[b >> 1] * dy[b >> 1];
#pragma unroll
            for (int dk = 0; dk < 2; dk++) f[b + 4 * dk] = (sxy + dz[dk] * dz[dk]) * h;  // Util::hypot3sq, times h
        }
        asm("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 3\n\t"
            "v_fma_f32 %0, %0, %8, %9\n\t"
            "v_fma_f32 %1, %1, %8, %9\n\t"
            "v_fma_f32 %2, %2, %8, %9\n\t"
            "v_fma_f32 %3, %3, %8, %9\n\t"
            "v_fma_f32 %4, %4, %8, %9\n\t"
            "v_fma_f32 %5, %5, %8, %9\n\t"
            "v_fma_f32 %6, %6, %8, %9\n\t"
            "v_fma_f32 %7, %7, %8, %9\n\t"
            "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0"
            : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7])
            : "s"(50.0f), "v"(2097152.5f));
#pragma unroll
        for (int k = 0; k < 8; k++)
            wg[k] = *(const __attribute__((address_space(3))) float *)((unsigned)__float_as_int(f[k]) & 0xffcu) * weight;
    } else {
        double ax[2], ay[2], az[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            ax[t] = 1.0 - (double)fabsf(dx[t]);
            ay[t] = 1.0 - (double)fabsf(dy[t]);
            az[t] = 1.0 - (double)fabsf(dz[t]);
        }
#pragma unroll
        for (int cI = 0; cI < 8; cI++)
            wg[cI] = (float)(ax[cI & 1] * ay[(cI >> 1) & 1] * az[cI >> 2] * (double)weight);
    }
}

// A pixel waiting for its turn to add into the brick accumulator: value,
// position and weight (the corner weights are recomputed from these in the
// window that adds it).  Non-pending lanes hold a finite position, so the
// weight computation they run along with the wave stays inside the tables.
struct PendPix {
    float re, im, px, py, pz, pw;
    int org;    // stencil origin: tag index in [0, BRICK^3), accumulator slot << 16
    bool pend;
};

// Election of a window: one lane per stencil origin among the pending
// pixels wins the right to add its 8 corners; pixels carried over from
// earlier windows take precedence over the window's new ones (`fresh`), so a
// carried pixel is added in the next window it takes part in unless it
// collides with another carried pixel.  The losers stay pending.
__device__ __forceinline__ bool scatter_elect(const PendPix &st, bool fresh, int lane, unsigned char *tag)
{
    const int ti = st.org & 0xffff;
    if (st.pend && fresh) tag[ti] = (unsigned char)lane;
    wave_sync_lds();
    if (st.pend && !fresh) tag[ti] = (unsigned char)lane;
    wave_sync_lds();
    const bool win = st.pend && tag[ti] == (unsigned char)lane;
    wave_sync_lds();
    return win;
}

// The winners add their 8 corners: lanes with different origins can still
// meet on a cell through different corners, so the corners go one after
// another with a wave-level ordering point between them.
template <int A>
__device__ __forceinline__ void scatter_add(const PendPix &st, bool win, const InsertConst &c, float *acc)
{
    float wg[8];
    corner_weights8(c.mode, st.px, st.py, st.pz, c.h, st.pw, wg);
    float *const p_re = acc + (st.org >> 16), *const p_im = p_re + ACC_N, *const p_w = p_re + 2 * ACC_N;
#pragma unroll
    for (int cI = 0; cI < 8; cI++) {
        const int di = cI & 1, dj = (cI >> 1) & 1, dk = cI >> 2;
        if (win) {
            const int a = acc_slot<A>(di, dj, dk);
            p_re[a] = __builtin_fmaf(st.re, wg[cI], p_re[a]);
            p_im[a] = __builtin_fmaf(st.im, wg[cI], p_im[a]);
            p_w[a] += wg[cI];
        }
        wave_sync_lds();
    }
}

// Up to GROUP slices of an item in one stream of 64-pixel windows: lane
// (g, r) = (lane / 16, lane % 16) sets up row r of slice g (a stencil origin
// in [lo, lo+7]^3 puts p within 4 sqrt(3) of the brick centre, i.e. at most
// 14 rows), the rows' pixel counts are scanned over the wave, and each
// window gives the next pixels of the stream, whatever slice they belong to,
// to the lanes that hold no pending pixel.
constexpr int GROUP = 4;

// The slice of lane (g, r) in a group: index, t3d rows 0-1, weight.  Loaded
// one group ahead, so the reads are in flight while the previous group's
// windows run.
struct GroupSlice {
    int q;  // -1: no slice
    float mm[6];
    float wgt;
};

// Slice record of lane (g, r) for the group starting at item slice s: the
// index from the 64 list entries held in qbuf (entries qbase .. qbase+63).
__device__ __forceinline__ void fetch_group_slice(GroupSlice &gs, int s, int count, int qbuf, int qbase, int lane,
                                                  int nslices, const float *__restrict__ t3d,
                                                  const float *__restrict__ wq)
{
    const int idx = s + (lane >> 4);
    const int qi = __builtin_amdgcn_ds_bpermute((idx - qbase) << 2, qbuf);
    const int q = idx < count ? qi : -1;
    const bool qv = q >= 0 && q < nslices;  // never written list entries are skipped
    gs.q = qv ? q : -1;
#pragma unroll
    for (int d = 0; d < 6; d++) gs.mm[d] = qv ? t3d[9 * (size_t)q + d] : 0.f;
    gs.wgt = qv ? wq[q] : 0.f;
}

template <int A, bool SSNR>
__device__ __forceinline__ void scatter_group(const float2 *__restrict__ slices, int nsym, const GroupSlice &gs,
                                              const InsertConst &c, const int lo[3], int lane, float *acc,
                                              unsigned char *tag, int *mark, float4 *rec, const float *rtab,
                                              const float *__restrict__ rw, PendPix &st, bool &fresh)
{
    const int H = c.H, P = c.P;
    const unsigned slice_elems = (unsigned)P * (unsigned)(H + 1);
    const int g = lane >> 4, r = lane & 15;
    const int q = gs.q;
    const bool qv = q >= 0;
    float mm[6];
#pragma unroll
    for (int d = 0; d < 6; d++) mm[d] = gs.mm[d];
    const float wgt = gs.wgt;
    if (r == 0) {
        rec[2 * g] = make_float4(mm[0], mm[1], mm[2], mm[3]);
        rec[2 * g + 1] = make_float4(mm[4], mm[5], wgt, __int_as_float(qv ? q / nsym : 0));  // particle
    }
    // the pixel nearest the brick centre's projection; bounds are relative to it
    const float cx = (float)lo[0] + 4.0f, cy = (float)lo[1] + 4.0f, cz = (float)lo[2] + 4.0f;
    const float sc = cx * mm[0] + cy * mm[1] + cz * mm[2];
    const float tc = cx * mm[3] + cy * mm[4] + cz * mm[5];
    const int xc0 = (int)rintf(sc), yc0 = (int)rintf(tc);
    const int dya = (int)ceilf(tc - (float)yc0 - SC_RAD), dyb = (int)floorf(tc - (float)yc0 + SC_RAD);
    const int dxa = (int)ceilf(sc - (float)xc0 - SC_RAD), dxb = (int)floorf(sc - (float)xc0 + SC_RAD);
    // row dy: x range where p[d] in [lo, lo+8) (+- margin) on every axis
    int cnt = 0, xs = 0;
    const int y = yc0 + dya + r;
    if (qv && dya + r <= dyb && y >= -H && y <= H - 1) {
        const float dyf = (float)(dya + r);
        float xl = (float)dxa, xh = (float)dxb;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const float ud = mm[d], vd = mm[3 + d];
            if (fabsf(ud) >= 0.05f) {
                const float P0 = (float)xc0 * ud + (float)yc0 * vd;
                const float iu = __builtin_amdgcn_rcpf(ud);
                const float t0 = ((float)lo[d] - P0 - SC_DLT - dyf * vd) * iu;
                const float t1 = ((float)(lo[d] + BRICK) - P0 + SC_DLT - dyf * vd) * iu;
                xl = fmaxf(xl, fminf(t0, t1));
                xh = fminf(xh, fmaxf(t0, t1));
            }
        }
        int a = max((int)ceilf(xl - SC_EPS), -xc0);
        int b = min((int)floorf(xh + SC_EPS), H - xc0);
        if (!c.corners) b = min(b, isqrt24(H * H + H - y * y) - xc0);  // hypot_fast_int(x,y) <= P/2
        xs = xc0 + a;
        cnt = max(0, b - a + 1);
    }
    const int incl = wave_scan_add(cnt);
    const int total = __builtin_amdgcn_readlane(incl, 63);
    const int excl = incl - cnt;
    // row record read by the slots of this row: (x - slot, y) as two int16
    const int rowrec = (int)(((unsigned)(xs - excl) & 0xffffu) | ((unsigned)y << 16));
    // Software-pipelined windows: the election of the pending pixels comes
    // first, then the lanes that will be free after this window load their
    // next pixels (slots next, next+1, ... in lane order), and the winners'
    // corner updates run while those slice reads are in flight.
    for (int next = 0; next < total;) {
        const bool win = scatter_elect(st, fresh, lane, tag);
        const bool freed = !st.pend || win;
        const unsigned long long fm = __ballot(freed);
        const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(fm >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)fm, 0u));
        // row of slot next+lane: the last non-empty row starting at or before it
        mark[lane] = -1;
        wave_sync_lds();
        if (cnt > 0 && excl >= next && excl < next + 64) mark[excl - next] = lane;
        if (cnt > 0 && excl < next && excl + cnt > next) mark[0] = lane;
        wave_sync_lds();
        const int rk = wave_scan_max(mark[lane]) & 63;
        const int rl = __builtin_amdgcn_ds_bpermute(rank << 2, rk);  // row of slot next+rank
        const int rr = __builtin_amdgcn_ds_bpermute(rl << 2, rowrec);
        const int s = next + rank;
        PendPix ns;
        ns.pend = false;
        bool ncj = false;
        if (freed && s < total) {
            const float4 ra = rec[2 * (rl >> 4)], rb = rec[2 * (rl >> 4) + 1];
            const int x = (int)(short)(rr & 0xffff) + s, ry = rr >> 16;
            const float pm[6] = {ra.x, ra.y, ra.z, ra.w, rb.x, rb.y};
            float px, py, pz;
            pixel_coords(x, ry, pm, rtab, H, c.Pf, px, py, pz);
            const int i0 = (int)floorf(px) - lo[0], i1 = (int)floorf(py) - lo[1], i2 = (int)floorf(pz) - lo[2];
            // x in [0, P/2] holds by construction; origins lie in [-P/2-1, ...): the
            // ones past P/2 only reach cells that are never merged
            if ((unsigned)x <= (unsigned)H && (unsigned)i0 < (unsigned)BRICK && (unsigned)i1 < (unsigned)BRICK &&
                (unsigned)i2 < (unsigned)BRICK) {
                // slice_value() with the conjugation applied after the corner
                // updates, so that nothing waits for the read before then
                const bool cj = x == 0 && ry < 0;
                const int row = cj ? -ry : (ry < 0 ? P + ry : ry);
                const float2 dt = (slices + (unsigned long long)(unsigned)__float_as_int(rb.w) *
                                                slice_elems)[row * (H + 1) + x];
                ns.re = dt.x;
                ns.im = dt.y;
                ncj = cj;
                ns.px = px;
                ns.py = py;
                ns.pz = pz;
                ns.org = i0 + BRICK * (i1 + BRICK * i2) + (acc_slot<A>(i0, i1, i2) << 16);
                // class_ssnr weighting: the particle's weight at radius hypot_fast_int(x, y)
                ns.pw = SSNR ? rw[(unsigned long long)(unsigned)__float_as_int(rb.w) * (unsigned)(H + 1) +
                                  (unsigned)hypot_int(x, ry)]
                             : rb.z;
                ns.pend = true;
            }
        }
        wave_sync_lds();  // rec reads before the next group rewrites them
        if (__ballot(win)) scatter_add<A>(st, win, c, acc);
        if (freed) {
            st.pend = ns.pend;
            if (ns.pend) {
                st = ns;
                if (ncj) st.im = -st.im;
            }
        }
        fresh = freed && ns.pend;
        next += __popcll(fm);
    }
}

// Partial brick layout in HBM: [field re/im/w][z][y][x] of the brick's 9^3 cells.
template <int A, bool SSNR>
__device__ __forceinline__ void scatter_item(const float2 *__restrict__ slices, int nslices, int nsym,
                                             const float *__restrict__ t3d, const float *__restrict__ wq,
                                             const InsertConst &c, const int *__restrict__ list, const WorkItem &w,
                                             const int lo[3], int lane, float *acc, unsigned char *tag, int *mark,
                                             float4 *rec, const float *rtab, const float *__restrict__ rw, float *out)
{
    PendPix st;
    st.re = st.im = st.pw = 0.f;
    st.px = (float)lo[0];
    st.py = (float)lo[1];
    st.pz = (float)lo[2];
    st.org = 0;
    st.pend = false;
    bool fresh = false;
    // list entries 64 at a time; each group's slice records fetched one group ahead
    int qbase = 0;
    int qbuf = lane < w.count ? list[w.start + lane] : -1;
    GroupSlice nxt;
    fetch_group_slice(nxt, 0, w.count, qbuf, qbase, lane, nslices, t3d, wq);
    for (int s0 = 0; s0 < w.count; s0 += GROUP) {
        const GroupSlice cur = nxt;
        const int s1 = s0 + GROUP;
        if (s1 < w.count) {
            if (s1 + GROUP > qbase + 64) {
                qbase = s1;
                qbuf = qbase + lane < w.count ? list[w.start + qbase + lane] : -1;
            }
            fetch_group_slice(nxt, s1, w.count, qbuf, qbase, lane, nslices, t3d, wq);
        }
        scatter_group<A, SSNR>(slices, nsym, cur, c, lo, lane, acc, tag, mark, rec, rtab, rw, st, fresh);
    }
    while (__ballot(st.pend)) {
        const bool win = scatter_elect(st, fresh, lane, tag);
        scatter_add<A>(st, win, c, acc);
        st.pend = st.pend && !win;
        fresh = false;
    }
    wave_sync_lds();
#pragma unroll
    for (int wv = 0; wv < (ACC_N + 63) / 64; wv++) {
        const int cc = lane + 64 * wv;
        if (cc < ACC_N) {
            const int z = cc / (HALO * HALO), yx = cc - z * HALO * HALO, y = yx / HALO, x = yx - y * HALO;
            const int a = acc_slot<A>(x, y, z);
            out[cc] = acc[a];
            out[ACC_N + cc] = acc[ACC_N + a];
            out[2 * ACC_N + cc] = acc[2 * ACC_N + a];
        }
    }
    wave_sync_lds();
}

// Bound by the random read-modify-writes into LDS (24 per pixel, about 0.73
// of the rate at which the LDS serves them alone), the VALU work next to it.
// Stencil origins kept as a tag and slot index from the bounds test on, table
// indexes read off the bits of one FMA, and the table at a constant address:
// 49.0 -> 47.8 ms for 8,000 particles of D7 at pad 288, 18.9 -> 18.5 ms for
// 24,000 slices at pad 384.
// SSNR: per-pixel weights from the particles' radial class_ssnr tables rw
// ((P/2+1) floats per particle) instead of the slice weight.
template <bool SSNR>
__global__ void __launch_bounds__(256) k_scatter_insert(const float2 *__restrict__ slices, int nslices, int nsym,
                                                        const float *__restrict__ t3d, const float *__restrict__ wq,
                                                        InsertConst c, BrickGeom g, BinBuffers bb,
                                                        const float *__restrict__ exptab_g,
                                                        const float *__restrict__ rtab_g,
                                                        const float *__restrict__ rw)
{
    extern __shared__ float4 lds4[];
    float *etab = reinterpret_cast<float *>(lds4);  // from LDS address 0
    char *base = reinterpret_cast<char *>(etab + EXPN);
    const int lane = threadIdx.x & 63;
    char *mine = base + (size_t)(threadIdx.x >> 6) * WAVE_LDS_BYTES;
    float *acc = reinterpret_cast<float *>(mine);
    float4 *rec = reinterpret_cast<float4 *>(mine + REC_OFF);
    int *mark = reinterpret_cast<int *>(mine + MARK_OFF);
    unsigned char *tag = reinterpret_cast<unsigned char *>(mine + TAG_OFF);
    float *rtab = reinterpret_cast<float *>(base + (size_t)(blockDim.x >> 6) * WAVE_LDS_BYTES);  // P+2 entries: fl(i/P)
    for (int i = threadIdx.x; i < EXPN; i += blockDim.x) etab[i] = exptab_g[i];
    for (int i = threadIdx.x; i < c.P + 2; i += blockDim.x) rtab[i] = rtab_g[i];
    __syncthreads();
    const int H = c.H, nb = g.nb;
    const int total = bb.ctl[1];
    for (;;) {
        int it = 0;
        if (lane == 0) it = atomicAdd(&bb.ctl[0], 1);
        it = __shfl(it, 0, 64);
        if (it >= total) break;
        const WorkItem w = bb.items[it];
        const int brick = w.key / 3, A = w.key - 3 * brick;
        const int lo[3] = {-H - 1 + BRICK * (brick % nb), -H - 1 + BRICK * ((brick / nb) % nb),
                           -H - 1 + BRICK * (brick / (nb * nb))};
#pragma unroll
        for (int wv = 0; wv < (3 * ACC_N + 63) / 64; wv++)
            if (lane + 64 * wv < 3 * ACC_N) acc[lane + 64 * wv] = 0.f;
        wave_sync_lds();
        float *out = bb.part + (size_t)it * PART_FLOATS;
        if (A == 0) scatter_item<0, SSNR>(slices, nslices, nsym, t3d, wq, c, bb.list, w, lo, lane, acc, tag, mark, rec, rtab, rw, out);
        else if (A == 1) scatter_item<1, SSNR>(slices, nslices, nsym, t3d, wq, c, bb.list, w, lo, lane, acc, tag, mark, rec, rtab, rw, out);
        else scatter_item<2, SSNR>(slices, nslices, nsym, t3d, wq, c, bb.list, w, lo, lane, acc, tag, mark, rec, rtab, rw, out);
    }
}

size_t scatter_lds_bytes(int P, int waves_per_block)
{
    return (size_t)waves_per_block * WAVE_LDS_BYTES + sizeof(float) * (EXPN + P + 2);
}

hipError_t launch_scatter_insert(const float2 *slices, int nslices, int nsym, const float *t3d, const float *wq,
                                 InsertConst c, BrickGeom g, BinBuffers b, const float *exptab, const float *rtab,
                                 const float *rw, int grid, int waves_per_block, hipStream_t s)
{
    if (waves_per_block < 1 || waves_per_block > 4) return hipErrorInvalidValue;
    if (rw)
        hipLaunchKernelGGL(k_scatter_insert<true>, dim3(grid), dim3(64 * waves_per_block),
                           scatter_lds_bytes(c.P, waves_per_block), s, slices, nslices, nsym, t3d, wq, c, g, b, exptab,
                           rtab, rw);
    else
        hipLaunchKernelGGL(k_scatter_insert<false>, dim3(grid), dim3(64 * waves_per_block),
                           scatter_lds_bytes(c.P, waves_per_block), s, slices, nslices, nsym, t3d, wq, c, g, b, exptab,
                           rtab, rw);
    return hipGetLastError();
}

// ------------------------------------------------------------ wide-stencil brick scatter
// The inserters with stencils of S = 3 to 9 cells per axis other than the
// 6-cell Gaussians (gauss_3, kaiser_bessel, kaiser_bessel_derived,
// gridding_5, gridding_7) on bricks of 4^3 stencil origins, binned like
// gauss_2's on the origin grid of the mode.  A work item's wave
// owns the brick's (3 + S)^3 cells in LDS.  For each slice of the item it
// tests the 8 x 8 pixels around the projection of the brick's centre (a
// pixel whose origin lies in the brick is within 2 sqrt 3 of that centre in
// p, so within 7 pixels per axis in the slice), then adds the stencils of the
// pixels whose origin lies in the brick one pixel after another, all 64 lanes
// over the pixel's S^3 cells.  The cells of one stencil are distinct and the
// pixels of a wave follow one another in program order, so plain LDS
// read-modify-writes suffice: no atomics and no election.  Each contribution
// is computed by wide_setup / wide_term, as in every other form.
#define WR_CAND 3.4691f  // 2 sqrt 3 + margin for the FP32 position and origin rounding

__device__ __forceinline__ float bcast_f(float v, int j)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}

template <int MODE>
__global__ void __launch_bounds__(256) k_scatter_wide(const float2 *__restrict__ slices, int nslices, int nsym,
                                                      const float *__restrict__ t3d, const float *__restrict__ wq,
                                                      InsertConst c, BrickGeom g, BinBuffers bb,
                                                      const float *__restrict__ exptab_g,
                                                      const float *__restrict__ rtab, const float *__restrict__ rw)
{
    constexpr int S = wide_cells(MODE), HL = WBS + S - 1, HC = HL * HL * HL;
    constexpr int NC = S * S * S, NIT = (NC + 63) / 64;
    extern __shared__ float lds_w[];
    float *etab = lds_w;  // the 1000 fast_exp entries
    float *acc = lds_w + 1024 + (size_t)(threadIdx.x >> 6) * 3 * HC;  // re, im, w over [z][y][x] of the cells
    const int lane = threadIdx.x & 63;
    for (int i = threadIdx.x; i < 1000; i += blockDim.x) etab[i] = exptab_g[i];
    __syncthreads();
    const int H = c.H, P = c.P, nb = g.nb;
    // this lane's stencil cell in pass t: offsets oi | oj << 4 | ok << 8 (-1 past S^3) and its LDS offset
    int oc[NIT], off[NIT];
#pragma unroll
    for (int t = 0; t < NIT; t++) {
        const int ci = lane + 64 * t;
        const int oi = ci % S, oj = (ci / S) % S, ok = ci / (S * S);
        const bool in = ci < NC;
        oc[t] = in ? (oi | (oj << 4) | (ok << 8)) : -1;
        off[t] = in ? (ok * HL + oj) * HL + oi : 0;
    }
    const int total = bb.ctl[1];
    for (;;) {
        int it = 0;
        if (lane == 0) it = atomicAdd(&bb.ctl[0], 1);
        it = __shfl(it, 0, 64);
        if (it >= total) break;
        const WorkItem w = bb.items[it];
        const int brick = w.key / 3;
        const int bc[3] = {brick % nb, (brick / nb) % nb, brick / (nb * nb)};
        int lo[3];
        float pc[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            lo[d] = g.ow + WBS * bc[d];
            pc[d] = g.po + (float)(WBS * bc[d]) + 0.5f * WBS;  // exact: half-integers of magnitude < 2^20
        }
        for (int i = lane; i < 3 * HC; i += 64) acc[i] = 0.f;
        wave_sync_lds();
        int qbuf = -1;
        for (int s = 0; s < w.count; s++) {
            if ((s & 63) == 0) qbuf = s + lane < w.count ? bb.list[w.start + s + lane] : -1;
            const int q = __builtin_amdgcn_readlane(qbuf, s & 63);
            if (q < 0 || q >= nslices) continue;  // never written list entries are skipped
            const float wgt = wq[q];
            if (wgt == 0.0f) continue;
            float mm[6];
#pragma unroll
            for (int d = 0; d < 6; d++) mm[d] = t3d[9 * (size_t)q + d];
            const float sc = pc[0] * mm[0] + pc[1] * mm[1] + pc[2] * mm[2];
            const float tc = pc[0] * mm[3] + pc[1] * mm[4] + pc[2] * mm[5];
            const int x = (int)ceilf(sc - WR_CAND) + (lane & 7), y = (int)ceilf(tc - WR_CAND) + (lane >> 3);
            bool ok = x >= 0 && x <= H && y >= -H && y <= H - 1 &&
                      (c.corners || x * x + y * y <= c.rcut * c.rcut + c.rcut);  // hypot_fast_int(x, y) <= rcut
            WidePix px;
            int pk = 0;
            if (ok) {
                const int p = q / nsym;
                const float weight = rw ? rw[(size_t)p * (H + 1) + hypot_int(x, y)] : wgt;
                float xx, yy, zz;
                pixel_coords(x, y, mm, rtab, H, c.Pf, xx, yy, zz);
                ok = wide_setup(MODE, xx, yy, zz, weight, H, etab, px);
                if (ok) {
#pragma unroll
                    for (int d = 0; d < 3; d++) ok = ok && (unsigned)(px.a[d] - lo[d]) < (unsigned)WBS;
                }
                if (ok) {
                    const float2 dt = slice_value(slices + (size_t)p * P * (H + 1), x, y, P, H);
                    px.dre = dt.x;
                    px.dim = dt.y;
#pragma unroll
                    for (int d = 0; d < 3; d++)
                        pk |= ((px.a[d] - lo[d]) | ((px.lo[d] - px.a[d]) << 2) | ((px.hi[d] - px.a[d]) << 6))
                              << (10 * d);
                }
            }
            unsigned long long hits = __ballot(ok);
            while (hits) {
                const int j = (int)__builtin_ctzll(hits);
                hits &= hits - 1;
                WidePix u;
                u.xx = bcast_f(px.xx, j);
                u.yy = bcast_f(px.yy, j);
                u.zz = bcast_f(px.zz, j);
                u.w = bcast_f(px.w, j);
                u.ww = bcast_f(px.ww, j);
                u.h = bcast_f(px.h, j);
                u.dre = bcast_f(px.dre, j);
                u.dim = bcast_f(px.dim, j);
                u.nre = u.nim = 0.f;
                u.H = H;
                u.ref = nullptr;
                const int pkj = __builtin_amdgcn_readlane(pk, j);
                bool full = true;
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    const int f = pkj >> (10 * d);
                    u.a[d] = lo[d] + (f & 3);
                    u.lo[d] = u.a[d] + ((f >> 2) & 15);
                    u.hi[d] = u.a[d] + ((f >> 6) & 15);
                    full = full && u.lo[d] == u.a[d] && u.hi[d] == u.a[d] + S - 1;
                }
                const int base = ((u.a[2] - lo[2]) * HL + (u.a[1] - lo[1])) * HL + (u.a[0] - lo[0]);
                // the pixel's cells are distinct: every lane reads its cells first (lanes past the
                // stencil read cell `base`, in bounds) and the lanes with a contribution write them
                // back after the terms are computed
                float ar[NIT], ai[NIT], aw[NIT];
#pragma unroll
                for (int t = 0; t < NIT; t++) {
                    ar[t] = acc[base + off[t]];
                    ai[t] = acc[HC + base + off[t]];
                    aw[t] = acc[2 * HC + base + off[t]];
                }
                float vr[NIT], vi[NIT], vg[NIT];
                bool on[NIT];
#pragma unroll
                for (int t = 0; t < NIT; t++) {
                    const int o = oc[t];
                    const int i = u.a[0] + (o & 15), jj = u.a[1] + ((o >> 4) & 15), k = u.a[2] + ((o >> 8) & 15);
                    on[t] = o >= 0 && (full || (i >= u.lo[0] && i <= u.hi[0] && jj >= u.lo[1] && jj <= u.hi[1] &&
                                                k >= u.lo[2] && k <= u.hi[2]));
                    if (on[t]) on[t] = wide_term(MODE, u, i, jj, k, etab, vr[t], vi[t], vg[t]);
                }
#pragma unroll
                for (int t = 0; t < NIT; t++)
                    if (on[t]) {
                        acc[base + off[t]] = ar[t] + vr[t];
                        acc[HC + base + off[t]] = ai[t] + vi[t];
                        acc[2 * HC + base + off[t]] = aw[t] + vg[t];
                    }
            }
        }
        wave_sync_lds();
        float *out = bb.part + (size_t)it * g.part_floats;
        for (int i = lane; i < 3 * HC; i += 64) out[i] = acc[i];
        wave_sync_lds();
    }
}

// ------------------------------------------------------------ 6-cell Gaussian scatter
// gauss_var (e2make3dpar's default), gauss_5 and fourier_iter with or without
// a reference (modes 2, 3, 10, 11): 6^3 cells per pixel with weights
// fast_exp(-r^2 h) w.  A work item is a brick of 3 x 3 x 5 stencil origins and
// up to K slices; its 8 x 8 x 10 cells are kept in registers, lane (x, y) =
// (lane & 7, lane >> 3) owning the column of 10 cells at (x, y).  A pixel
// takes 6 passes, one per z plane of its stencil, over the 36 of the 64 lanes
// whose column lies in the stencil: x and y distances are computed once per
// pixel, the six z distances come from the lane that tested the pixel, and
// the sums are three FMAs into fixed registers (one copy of the passes per
// z offset of the origin).
//
// Bound: VALU, 0.35 instructions per SIMD and clock (0.70 of the published
// vector rate), 50 per pixel in the passes that stay within the table, 70 in
// all; the LDS is busy 83 % of the cycles with table reads and records.  The form
// before kept the cells in LDS (54 lanes per pass, 4 passes, 6 LDS operations
// and 28 VALU instructions each; an 8 x 8 window of candidate pixels tested
// per slice): 142 VALU instructions per pixel, 116 ms for 8,000 x pad 384
// gauss_var, now 41 ms; for 2,000 x pad 160 of fourier_iter with a reference
// (its cells read from memory for every term before, kept in the lanes'
// registers now) 37.3 ms, now 3.3 ms.  Taking the pixels' values by readlane
// instead of through LDS: 68 ms.  At 4 waves per SIMD, without spills: 43.5.
// The table index floor(f 50 + 1/2), f = r^2 h, which the reference takes in
// double, is one FMA rounded toward zero with 2^21 + 1/2 added: the sum's low
// mantissa bits are floor(4 (f 50 + 1/2)), so that its bits & 0xffc are 4
// times the index, the byte offset of the table entry.
#define G6_CAND 3.2838f  // half diagonal of 3 x 3 x 5 + margin for the FP32 position and origin rounding

// The byte offsets of the table entries of f[0..5], or'ed with `out`: 0 on the
// lanes of the pixel's window (f in [0, 20) there), 0xffc, the table's last
// entry, a zero, elsewhere.  A mode switch to rounding toward zero around the
// six FMAs.
__device__ __forceinline__ void g6_entries(const float f[6], unsigned out, unsigned e[6])
{
    float t[6];
#pragma unroll
    for (int k = 0; k < 6; k++) t[k] = f[k];
    asm("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 3\n\t"
        "v_fma_f32 %0, %0, %6, %7\n\t"
        "v_fma_f32 %1, %1, %6, %7\n\t"
        "v_fma_f32 %2, %2, %6, %7\n\t"
        "v_fma_f32 %3, %3, %6, %7\n\t"
        "v_fma_f32 %4, %4, %6, %7\n\t"
        "v_fma_f32 %5, %5, %6, %7\n\t"
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0"
        : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3]), "+v"(t[4]), "+v"(t[5])
        : "s"(50.0f), "v"(2097152.5f));
#pragma unroll
    for (int k = 0; k < 6; k++) e[k] = ((unsigned)__float_as_int(t[k]) & 0xffcu) | out;
}

// One pixel's values, uniform over the wave.
struct G6Pix {
    float xx, yy, h, re, im, w, nre, nim;  // re, im: times the weight w (mode 11: without it)
    float dz2[6];                          // squared z distances (1e30 on clipped planes)
};

// table entry at byte offset e: the table starts the kernel's LDS (dynamic, with no static LDS before it)
__device__ __forceinline__ float g6_table(unsigned e)
{
    return *(const __attribute__((address_space(3))) float *)e;
}

// The passes of a pixel whose origin lies OZ above the brick's in z; `in`: the
// lanes of its (x, y) window.  No lane is switched off: the others add zeros.
template <int MODE, int OZ>
__device__ __forceinline__ void g6_add(const G6Pix &u, float cx, float cy, bool in, const float2 (&rf)[G6_HZ],
                                       float (&ar)[G6_HZ], float (&ai)[G6_HZ], float (&aw)[G6_HZ])
{
    const float dx = cx - u.xx, dy = cy - u.yy;
    const float s = dx * dx + dy * dy;
    float f[6];
    unsigned e[6];
#pragma unroll
    for (int k = 0; k < 6; k++) f[k] = (s + u.dz2[k]) * u.h;  // hypot3sq in the reference's order, times h
    g6_entries(f, in ? 0u : 0xffcu, e);
    float g[6];
#pragma unroll
    for (int k = 0; k < 6; k++) g[k] = g6_table(e[k]);
#pragma unroll
    for (int k = 0; k < 6; k++) {
        const int z = OZ + k;
        if (MODE == 11) {
            // updt = dt + ref(i, j, k) - ref~(p)
            const float gw = g[k] * u.w;
            ar[z] = __builtin_fmaf((u.re + rf[z].x) - u.nre, gw, ar[z]);
            ai[z] = __builtin_fmaf((u.im + rf[z].y) - u.nim, gw, ai[z]);
            aw[z] += gw;
        } else {
            ar[z] = __builtin_fmaf(u.re, g[k], ar[z]);
            ai[z] = __builtin_fmaf(u.im, g[k], ai[z]);
            aw[z] = __builtin_fmaf(u.w, g[k], aw[z]);
        }
    }
}

// The same where terms past the table (f > 19.98, by expf) can occur.  ANY:
// also dropped ones (below FLT_MIN), cells outside fourier_iter's sphere and
// values that are not finite: what is not added leaves the sum as it is.
template <int MODE, int OZ, bool ANY>
__device__ __forceinline__ void g6_add_far(const G6Pix &u, float cx, float cy, bool in, unsigned inside,
                                           const float2 (&rf)[G6_HZ], float (&ar)[G6_HZ], float (&ai)[G6_HZ],
                                           float (&aw)[G6_HZ])
{
    const float dx = cx - u.xx, dy = cy - u.yy;
    const float s = dx * dx + dy * dy;
    float f[6], fc[6];
    unsigned e[6];
#pragma unroll
    for (int k = 0; k < 6; k++) {
        f[k] = (s + u.dz2[k]) * u.h;
        fc[k] = fminf(f[k], 19.98f);
    }
    g6_entries(fc, in ? 0u : 0xffcu, e);
    float g[6];
#pragma unroll
    for (int k = 0; k < 6; k++) g[k] = g6_table(e[k]);
#pragma unroll
    for (int k = 0; k < 6; k++) {
        const int z = OZ + k;
        const bool big = in && f[k] > 19.98f;  // the same floats as the reference's (double)f > 19.98
        if (__ballot(big)) {
            asm volatile("");  // a branch, not a select: most passes have no such lane
            const float t = expf(-f[k]);
            g[k] = big ? t : g[k];
        }
        bool on = in;
        if (ANY) on = on && !(fabsf(g[k] * u.w) < FLT_MIN);
        float re, im, wg;
        if (MODE == 11) {
            if (ANY) on = on && (inside >> z & 1u);
            wg = g[k] * u.w;
            re = __builtin_fmaf((u.re + rf[z].x) - u.nre, wg, ar[z]);
            im = __builtin_fmaf((u.im + rf[z].y) - u.nim, wg, ai[z]);
            wg += aw[z];
        } else {
            re = __builtin_fmaf(u.re, g[k], ar[z]);
            im = __builtin_fmaf(u.im, g[k], ai[z]);
            wg = __builtin_fmaf(u.w, g[k], aw[z]);
        }
        ar[z] = on || !ANY ? re : ar[z];
        ai[z] = on || !ANY ? im : ai[z];
        aw[z] = on || !ANY ? wg : aw[z];
    }
}

// the width of the modes where it is the same for every pixel: gauss_5, fourier_iter with a reference
template <int MODE>
__device__ constexpr float g6_width()
{
    return MODE == 3 ? 1.0f / (float)(10.4 / (M_PI * M_PI)) : 1.0f / 2.0f;
}

// The lane that tests a pixel leaves its values in LDS (G6_REC float4 per
// lane), all lanes read them back for the pixel's passes: one address for the
// wave, no bank conflicts, where 13 readlanes cost a fifth of the passes'
// VALU time.
constexpr int G6_REC = 4;
constexpr int G6_WAVE = 16 + 16 + 64 * G6_REC;  // float4 of LDS per wave

template <int MODE>
__device__ __forceinline__ void g6_put(float4 *r, const G6Pix &px)
{
    r[0] = make_float4(px.xx, px.yy, px.w, px.re);
    r[1] = make_float4(px.im, MODE == 11 ? px.nre : px.h, px.dz2[0], px.dz2[1]);
    r[2] = make_float4(px.dz2[2], px.dz2[3], px.dz2[4], px.dz2[5]);
    if (MODE == 11) r[3].x = px.nim;
}

template <int MODE>
__device__ __forceinline__ void g6_get(const float4 *r, G6Pix &u)
{
    const float4 a = r[0], b = r[1], d = r[2];
    u.xx = a.x;
    u.yy = a.y;
    u.w = a.z;
    u.re = a.w;
    u.im = b.x;
    u.h = MODE == 2 || MODE == 10 ? b.y : g6_width<MODE>();
    u.nre = MODE == 11 ? b.y : 0.f;
    u.nim = MODE == 11 ? r[3].x : 0.f;
    u.dz2[0] = b.z;
    u.dz2[1] = b.w;
    u.dz2[2] = d.x;
    u.dz2[3] = d.y;
    u.dz2[4] = d.z;
    u.dz2[5] = d.w;
}

// the window of lanes of the pixel tested by lane j: bits [x0, x0 + nx) of bytes [y0, y0 + ny)
__device__ __forceinline__ bool g6_window(int pk, int j)
{
    const unsigned b = (unsigned)__builtin_amdgcn_readlane(pk, j);
    const unsigned row = (((1u << (b >> 3 & 7)) - 1u) << (b & 7)) * 0x01010101u;
    return __builtin_amdgcn_inverse_ballot_w64(((unsigned long long)row << 32 | row) &
                                               (((1ull << (b >> 9 & 7) * 8) - 1ull) << (b >> 6 & 7) * 8));
}

// gauss_var's width of the pixel at p, (float)(1 / ((double)(|p|^2 / 4000) + 0.15)) and at least 0.1: |p|^2 / 4000
// by the reciprocal with one exact-residual step, which rounds correctly; the double reciprocal by two Newton steps.
__device__ __forceinline__ float g6_width_at(float x, float y, float z)
{
    const float n = x * x + y * y + z * z, inv = 1.0f / 4000.0f;
    const float v = n * inv;
    const double t = (double)__builtin_fmaf(__builtin_fmaf(-v, 4000.0f, n), inv, v) + 0.15;
    double r = __builtin_amdgcn_rcp(t);
    r = __builtin_fma(__builtin_fma(-t, r, 1.0), r, r);
    r = __builtin_fma(__builtin_fma(-t, r, 1.0), r, r);
    return fmaxf((float)r, 0.1f);  // the same floats as the reference's double comparison with 0.1
}

// The slice of lane (i, r) in a group of 8: index (-1: none), t3d rows 0 and 1, weight; loaded one group ahead.
struct G6Slice {
    int q;
    float mm[6];
    float wgt;
};

__device__ __forceinline__ void g6_fetch(G6Slice &gs, int s, int count, int qbuf, int qbase, int lane, int nslices,
                                         const float *__restrict__ t3d, const float *__restrict__ wq)
{
    const int idx = s + (lane >> 3);
    const int qi = __builtin_amdgcn_ds_bpermute((idx - qbase) << 2, qbuf);
    const int q = idx < count ? qi : -1;
    const bool qv = q >= 0 && q < nslices;  // never written list entries are skipped
    gs.q = qv ? q : -1;
#pragma unroll
    for (int d = 0; d < 6; d++) gs.mm[d] = qv ? t3d[9 * (size_t)q + d] : 0.f;
    gs.wgt = qv ? wq[q] : 0.f;
}

template <int MODE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MODE == 11 ? 4 : 5))) k_scatter_gauss6(const float2 *__restrict__ slices, int nslices, int nsym,
                                                        const float *__restrict__ t3d, const float *__restrict__ wq,
                                                        InsertConst c, BrickGeom g, BinBuffers bb,
                                                        const float *__restrict__ exptab_g,
                                                        const float *__restrict__ rtab_g,
                                                        const float *__restrict__ rw)
{
    extern __shared__ float4 lds_g6[];
    float *etab = reinterpret_cast<float *>(lds_g6);  // the 1000 fast_exp entries, then zeros
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // per wave: 8 slice records (2 float4 each), 64 row marks and 64 pixels
    float4 *rec = lds_g6 + 256 + wave * G6_WAVE;
    int *mark = reinterpret_cast<int *>(rec + 16);
    float4 *pix = rec + 32;
    float *rtab = reinterpret_cast<float *>(lds_g6 + 256 + (blockDim.x >> 6) * G6_WAVE);  // P + 2 entries: fl(i/P)
    const int H = c.H, P = c.P, nb = g.nb;
    for (int i = threadIdx.x; i < 1024; i += blockDim.x) etab[i] = i < 1000 ? exptab_g[i] : 0.f;
    for (int i = threadIdx.x; i < P + 2; i += blockDim.x) rtab[i] = rtab_g[i];
    __syncthreads();
    const int n2x = MODE >= 10 ? H - 1 : H;  // stencils are clamped to [-n2, n2], fourier_iter's in x to P/2 - 1
    const int total = bb.ctl[1];
    for (;;) {
        int it = 0;
        if (lane == 0) it = atomicAdd(&bb.ctl[0], 1);
        it = __builtin_amdgcn_readfirstlane(it);
        if (it >= total) break;
        const WorkItem w = bb.items[it];
        const int brick = w.key / 3;
        const int bc[3] = {brick % nb, (brick / nb) % nb, brick / (nb * nb)};
        const int lo[3] = {g.ow + G6_BX * bc[0], g.ow + G6_BX * bc[1], g.ow + G6_BZ * bc[2]};
        // p-space centre of the brick (exact: half-integers of magnitude < 2^20)
        const float pc[3] = {g.po + (float)(G6_BX * bc[0]) + 0.5f * G6_BX, g.po + (float)(G6_BX * bc[1]) + 0.5f * G6_BX,
                             g.po + (float)(G6_BZ * bc[2]) + 0.5f * G6_BZ};
        const float pl[3] = {g.po + (float)(G6_BX * bc[0]), g.po + (float)(G6_BX * bc[1]), g.po + (float)(G6_BZ * bc[2])};
        // a cell of the brick lies outside the volume: the stencils are clamped
        const bool edge = lo[0] < -n2x || lo[0] + G6_HX - 1 > n2x || lo[1] < -H || lo[1] + G6_HX - 1 > H ||
                          lo[2] < -H || lo[2] + G6_HZ - 1 > H;
        // the table may end within a stencil: not for h <= 1/2 (farthest corner 3 * 3.5^2), which
        // gauss_var's width stays below beyond |p| = 87 (the brick's pixels lie within 3.3 of its centre)
        const bool near = MODE == 3 || (MODE != 11 && pc[0] * pc[0] + pc[1] * pc[1] + pc[2] * pc[2] < 90.5f * 90.5f);
        const int ix = lo[0] + (lane & 7), iy = lo[1] + (lane >> 3);  // this lane's column of cells
        const float cx = (float)ix, cy = (float)iy;
        float ar[G6_HZ], ai[G6_HZ], aw[G6_HZ];
        float2 rf[G6_HZ];
        unsigned inside = 0;
        bool cut = false;  // a cell of the brick lies outside fourier_iter's sphere, or its value is not finite
#pragma unroll
        for (int z = 0; z < G6_HZ; z++) {
            ar[z] = ai[z] = aw[z] = 0.f;
            rf[z] = make_float2(0.f, 0.f);
            if (MODE == 11) {
                const int iz = lo[2] + z;
                rf[z] = ref_get(c.ref, ix, iy, iz, H);
                if (ix * ix + iy * iy + iz * iz <= H * H) inside |= 1u << z;
                cut = cut || !(fabsf(rf[z].x) + fabsf(rf[z].y) < FLT_MAX);
            }
        }
        if (MODE == 11) cut = __ballot(cut || inside != (1u << G6_HZ) - 1u) != 0;
        // 8 slices at a time: lane (i, r) = (lane / 8, lane % 8) sets up row r of slice i, the rows of
        // the slice's pixels around the projection of the brick's centre (a pixel whose origin lies in the
        // brick is within the half diagonal of that centre in p: at most 7 rows), with the range of x
        // where p lies in the brick's box, margins as in scatter_group; the rows' pixels then form one
        // stream of which each window gives 64 to the lanes.
        int qbase = 0;
        int qbuf = lane < w.count ? bb.list[w.start + lane] : -1;
        G6Slice nxt;
        g6_fetch(nxt, 0, w.count, qbuf, qbase, lane, nslices, t3d, wq);
        for (int s0 = 0; s0 < w.count; s0 += 8) {
            const G6Slice gs = nxt;
            const int s1 = s0 + 8;
            if (s1 < w.count) {
                if (s1 + 8 > qbase + 64) {
                    qbase = s1;
                    qbuf = qbase + lane < w.count ? bb.list[w.start + qbase + lane] : -1;
                }
                g6_fetch(nxt, s1, w.count, qbuf, qbase, lane, nslices, t3d, wq);
            }
            if ((lane & 7) == 0) {
                rec[2 * (lane >> 3)] = make_float4(gs.mm[0], gs.mm[1], gs.mm[2], gs.mm[3]);
                rec[2 * (lane >> 3) + 1] = make_float4(gs.mm[4], gs.mm[5], gs.wgt,
                                                       __int_as_float(gs.q >= 0 ? gs.q / nsym : 0));  // particle
            }
            int cnt = 0, xs = 0, y = 0;
            {
                const float sc = pc[0] * gs.mm[0] + pc[1] * gs.mm[1] + pc[2] * gs.mm[2];
                const float tc = pc[0] * gs.mm[3] + pc[1] * gs.mm[4] + pc[2] * gs.mm[5];
                const int xc0 = (int)rintf(sc), yc0 = (int)rintf(tc);
                const float fs = sc - (float)xc0, ft = tc - (float)yc0;
                const int dy = (int)ceilf(ft - G6_CAND) + (lane & 7);
                y = yc0 + dy;
                if (gs.q >= 0 && gs.wgt != 0.0f && (float)dy <= ft + G6_CAND && y >= -H && y <= H - 1) {
                    float xl = fs - G6_CAND, xh = fs + G6_CAND;
#pragma unroll
                    for (int d = 0; d < 3; d++) {
                        const float ud = gs.mm[d], vd = gs.mm[3 + d];
                        if (fabsf(ud) >= 0.05f) {
                            const float b0 = pl[d] - ((float)xc0 * ud + (float)yc0 * vd) - (float)dy * vd;
                            const float iu = __builtin_amdgcn_rcpf(ud);
                            const float t0 = (b0 - SC_DLT) * iu;
                            const float t1 = (b0 + (float)(d == 2 ? G6_BZ : G6_BX) + SC_DLT) * iu;
                            xl = fmaxf(xl, fminf(t0, t1));
                            xh = fminf(xh, fmaxf(t0, t1));
                        }
                    }
                    const int a = max((int)ceilf(xl - SC_EPS), -xc0);
                    int b = min((int)floorf(xh + SC_EPS), H - xc0);
                    // hypot_fast_int(x, y) <= rcut
                    if (!c.corners) b = min(b, isqrt24(c.rcut * c.rcut + c.rcut - y * y) - xc0);
                    xs = xc0 + a;
                    cnt = max(0, b - a + 1);
                }
            }
            const int incl = wave_scan_add(cnt);
            const int rows = __builtin_amdgcn_readlane(incl, 63);
            const int excl = incl - cnt;
            // row record read by the slots of this row: (x - slot, y) as two int16
            const int rowrec = (int)(((unsigned)(xs - excl) & 0xffffu) | ((unsigned)y << 16));
            for (int next = 0; next < rows; next += 64) {
                // row of slot next + lane: the last non-empty row starting at or before it
                mark[lane] = -1;
                wave_sync_lds();
                if (cnt > 0 && excl >= next && excl < next + 64) mark[excl - next] = lane;
                if (cnt > 0 && excl < next && excl + cnt > next) mark[0] = lane;
                wave_sync_lds();
                const int rl = wave_scan_max(mark[lane]) & 63;
                const int rr = __builtin_amdgcn_ds_bpermute(rl << 2, rowrec);
                const int slot = next + lane;
                bool ok = slot < rows, med = false, any = false;
                G6Pix px;
                px.xx = px.yy = px.h = px.re = px.im = px.w = px.nre = px.nim = 0.f;
#pragma unroll
                for (int k = 0; k < 6; k++) px.dz2[k] = 0.f;
                int pk = 0, oz = 0;
                if (ok) {
                    const float4 ra = rec[2 * (rl >> 3)], rb = rec[2 * (rl >> 3) + 1];
                    const int x = (int)(short)(rr & 0xffff) + slot, ry = rr >> 16;
                    const float pm[6] = {ra.x, ra.y, ra.z, ra.w, rb.x, rb.y};
                    float pp[3];
                    pixel_coords(x, ry, pm, rtab, H, c.Pf, pp[0], pp[1], pp[2]);
                    int a[3];
                    ok = (unsigned)x <= (unsigned)H;
#pragma unroll
                    for (int d = 0; d < 3; d++) {
                        // floor((double)p - 2.5): the fraction p - floor(p) is below 1/2 or not
                        const float fl = floorf(pp[d]);
                        a[d] = (int)fl - (pp[d] - fl >= 0.5f ? 2 : 3);
                        ok = ok && (unsigned)(a[d] - lo[d]) < (unsigned)(d == 2 ? G6_BZ : G6_BX);
                    }
                    pk = (a[0] - lo[0]) | 6 << 3 | (a[1] - lo[1]) << 6 | 6 << 9;
                    oz = a[2] - lo[2];
#pragma unroll
                    for (int k = 0; k < 6; k++) {
                        const float dz = (float)(a[2] + k) - pp[2];
                        px.dz2[k] = dz * dz;
                    }
                    if (edge) {
                        // the stencil clamped to the volume: window of columns and planes of the cells inside
                        int l[3], n[3];
#pragma unroll
                        for (int d = 0; d < 3; d++) {
                            const int n2 = d == 0 ? n2x : H;
                            l[d] = max(a[d], -n2);
                            n[d] = min(a[d] + 5, n2) - l[d] + 1;
                            ok = ok && a[d] >= -n2 - 4 && a[d] <= n2 + 3 && n[d] > 0;
                        }
                        pk = (l[0] - lo[0]) | n[0] << 3 | (l[1] - lo[1]) << 6 | n[1] << 9;
#pragma unroll
                        for (int k = 0; k < 6; k++)
                            if (a[2] + k < l[2] || a[2] + k >= l[2] + n[2]) {
                                px.dz2[k] = 1e30f;  // weight 0
                                any = true;
                            }
                    }
                    if (ok) {
                        const unsigned p = (unsigned)__float_as_int(rb.w);
                        const float2 dt = slice_value(slices + (size_t)p * P * (H + 1), x, ry, P, H);
                        const float wt = rw ? rw[(size_t)p * (H + 1) + hypot_int(x, ry)] : rb.z;
                        px.xx = pp[0];
                        px.yy = pp[1];
                        px.w = wt;
                        px.h = MODE == 2 || MODE == 10 ? g6_width_at(pp[0], pp[1], pp[2]) : g6_width<MODE>();
                        if (MODE == 11) ref_trilinear(c.ref, pp[0], pp[1], pp[2], H, px.nre, px.nim);
                        px.re = MODE == 11 ? dt.x : dt.x * wt;
                        px.im = MODE == 11 ? dt.y : dt.y * wt;
                        any = any || cut || !(fabsf(wt) > 1e-25f) ||
                              !(fabsf(px.re) + fabsf(px.im) + fabsf(px.nre) + fabsf(px.nim) + fabsf(wt) < FLT_MAX);
                        if (near) {
                            float far = 0.f;  // squared distance of the stencil's farthest corner
#pragma unroll
                            for (int d = 0; d < 3; d++) {
                                const float e = fmaxf(pp[d] - (float)a[d], (float)(a[d] + 5) - pp[d]);
                                far += e * e;
                            }
                            med = far * px.h > 19.9f;
                            // exp(-80) / 100 is above FLT_MIN
                            any = any || far * px.h > 80.f || (med && !(fabsf(wt) > 1e-2f));
                        }
                    }
                }
                if (ok) g6_put<MODE>(pix + G6_REC * lane, px);
                wave_sync_lds();
                // the pixels one after another, by the z offset of their origin: each offset's loop adds
                // into registers of its own choice
#define G6_LOOP(Z, COND, ADD)                                                              \
    for (unsigned long long left = __ballot((COND) && oz == Z); left; left &= left - 1) {   \
        const int j = (int)__builtin_ctzll(left);                                           \
        G6Pix u;                                                                            \
        g6_get<MODE>(pix + G6_REC * j, u);                                                  \
        const bool in = g6_window(pk, j);                                                   \
        ADD;                                                                                \
    }
#define G6_LOOPS(COND, ADD) \
    G6_LOOP(0, COND, ADD(0)) G6_LOOP(1, COND, ADD(1)) G6_LOOP(2, COND, ADD(2)) G6_LOOP(3, COND, ADD(3)) G6_LOOP(4, COND, ADD(4))
#define G6_NEAR(Z) g6_add<MODE, Z>(u, cx, cy, in, rf, ar, ai, aw)
#define G6_FAR(Z) g6_add_far<MODE, Z, false>(u, cx, cy, in, inside, rf, ar, ai, aw)
#define G6_ANY(Z) g6_add_far<MODE, Z, true>(u, cx, cy, in, inside, rf, ar, ai, aw)
                G6_LOOPS(ok && !med && !any, G6_NEAR)
                if (MODE != 11 && __ballot(ok && med && !any)) { G6_LOOPS(ok && med && !any, G6_FAR) }
                if (__ballot(ok && any)) { G6_LOOPS(ok && any, G6_ANY) }
#undef G6_LOOP
#undef G6_LOOPS
#undef G6_NEAR
#undef G6_FAR
#undef G6_ANY
                wave_sync_lds();  // the pixels' and slices' records are read before the next ones are written
            }
        }
        float *out = bb.part + (size_t)it * g.part_floats + lane;  // [field][z][y][x]
#pragma unroll
        for (int z = 0; z < G6_HZ; z++) {
            out[64 * z] = ar[z];
            out[64 * (G6_HZ + z)] = ai[z];
            out[64 * (2 * G6_HZ + z)] = aw[z];
        }
    }
}

static size_t scatter_wide_lds_bytes(InsertConst c, int waves_per_block)
{
    if (gauss6(c.mode)) return sizeof(float) * (1024 + 4 * G6_WAVE * (size_t)waves_per_block + c.P + 2);
    const int HL = WBS + wide_cells(c.mode) - 1;
    return sizeof(float) * (1024 + (size_t)waves_per_block * 3 * HL * HL * HL);
}

hipError_t launch_scatter_wide(const float2 *slices, int nslices, int nsym, const float *t3d, const float *wq,
                               InsertConst c, BrickGeom g, BinBuffers b, const float *exptab, const float *rtab,
                               const float *rw, int items, int cus, hipStream_t s)
{
    const int S = wide_cells(c.mode);
    const bool g6 = gauss6(c.mode);
    if (S == 0 || g.bs != (g6 ? G6_BX : WBS) || g.bsz != (g6 ? G6_BZ : WBS) || g.halo != g.bs + S - 1 ||
        g.haloz != g.bsz + S - 1)
        return hipErrorInvalidValue;
    // one wave per item: 4 waves per workgroup (2 for 9-cell stencils), as many workgroups as fit
    // the compute units
    const int ww = S > 7 ? 2 : 4;
    const size_t lds = scatter_wide_lds_bytes(c, ww);
    if (lds > 65536) return hipErrorInvalidValue;
#define FH_WIDE(KERNEL)                                                                                                  \
    {                                                                                                                    \
        int per = 0;                                                                                                     \
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, KERNEL, 64 * ww, lds) != hipSuccess || per < 1) per = 1;   \
        hipLaunchKernelGGL((KERNEL), dim3(std::min(cus * per, (items + ww - 1) / ww)), dim3(64 * ww), lds, s, slices,     \
                           nslices, nsym, t3d, wq, c, g, b, exptab, rtab, rw);                                           \
        return hipGetLastError();                                                                                        \
    }
    switch (c.mode) {
    case 2: FH_WIDE(k_scatter_gauss6<2>)
    case 3: FH_WIDE(k_scatter_gauss6<3>)
    case 5: FH_WIDE(k_scatter_wide<5>)
    case 6: FH_WIDE(k_scatter_wide<6>)
    case 7: FH_WIDE(k_scatter_wide<7>)
    case 8: FH_WIDE(k_scatter_wide<8>)
    case 9: FH_WIDE(k_scatter_wide<9>)
    case 10: FH_WIDE(k_scatter_gauss6<10>)
    case 11: FH_WIDE(k_scatter_gauss6<11>)
    default: return hipErrorInvalidValue;
    }
#undef FH_WIDE
}

// ------------------------------------------------------------ merge of partial bricks
// Items per brick from which they are summed before the merge reads them: 2
// where the batch has an item per brick of the grid (bricks outside the
// sphere of slices, about half, have none), else never.  A batch that overran
// the item list (bb.ctl[3], an internal error that the host reports, in a
// captured sequence after the merge) has offsets past the partial bricks:
// both kernels leave it alone.
__device__ __forceinline__ int reduce_least(const int *__restrict__ item_off, int nbricks)
{
    return item_off[3 * nbricks] >= nbricks ? 2 : INT_MAX;
}

// The items of every such brick summed into its first one's partial brick.
// A unit is 256 floats of a brick; the units go round the blocks, and the
// waves of a block share the ones of its turn that have work.  Read in whole
// runs here, the items cost their bytes; the merge, whose lanes read rows of 9
// floats out of neighbouring bricks, and one item after the other, took 1.08
// ms (24,000 slices at pad 384, 2.6 items per brick), 1.19 (112,000 at 288,
// 11) and 0.11 (2,000 at 96, 6): now 1.02, 0.59 and 0.033, this pass
// included.  Below an item per brick of the grid nothing is gained (8,000
// gauss_var slices at pad 384, 0.5: 4.6 ms, and 4.7 with a pass over all).
__global__ void __launch_bounds__(256) k_reduce_items(float *__restrict__ part, const int *__restrict__ item_off,
                                                      const int *__restrict__ ctl, int nbricks, int pf)
{
    __shared__ int q[256][3];  // first item, items, segment
    __shared__ int nq;
    const int least = reduce_least(item_off, nbricks);
    if (least == INT_MAX || ctl[3]) return;
    const int segs = (pf + 255) / 256, lane = threadIdx.x & 63;
    const long long units = (long long)nbricks * segs;
    for (long long r = 0; r * 256 * gridDim.x < units; r++) {
        if (threadIdx.x == 0) nq = 0;
        __syncthreads();
        const long long u = (r * 256 + threadIdx.x) * gridDim.x + blockIdx.x;
        if (u < units) {
            const int b = (int)(u / segs), i0 = item_off[3 * b], n = item_off[3 * b + 3] - i0;
            if (n >= least) {
                const int slot = atomicAdd(&nq, 1);
                q[slot][0] = i0;
                q[slot][1] = n;
                q[slot][2] = (int)(u - (long long)b * segs);
            }
        }
        __syncthreads();
        const int m = nq;
        for (int e = threadIdx.x >> 6; e < m; e += 4) {
            const int n = __builtin_amdgcn_readfirstlane(q[e][1]);
            const int c0 = 256 * __builtin_amdgcn_readfirstlane(q[e][2]) + lane;
            float *p = part + (size_t)__builtin_amdgcn_readfirstlane(q[e][0]) * pf;
            float sum[4] = {0.f, 0.f, 0.f, 0.f};
            for (int it = 0; it < n; it += 4) {
                float v[4][4];
#pragma unroll
                for (int k = 0; k < 4; k++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        v[k][j] = it + k < n && c0 + 64 * j < pf ? p[(size_t)(it + k) * pf + c0 + 64 * j] : 0.f;
#pragma unroll
                for (int k = 0; k < 4; k++)
#pragma unroll
                    for (int j = 0; j < 4; j++) sum[j] += v[k][j];
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (c0 + 64 * j < pf) p[c0 + 64 * j] = sum[j];
        }
        __syncthreads();  // the queue is read before the next turn fills it
    }
}

// Sum over the work items of the bricks whose cells include unfolded cell
// (i, j, k): brick b covers cells [ow + BS*b, ow + BS*b + HL) per axis (z:
// BZ, HZ), so a cell lies in the bricks floor(u / BS) down to
// ceil((u - HL + 1) / BS), u = cell - ow (for gauss_2, BS 8 and HL 9: the
// brick owning the origin and, on each axis where the cell is a brick's
// first, also the previous brick).
template <int BS, int HL, int BZ, int HZ>
__device__ __forceinline__ void partial_sum(const float *__restrict__ part, const int *__restrict__ item_off, int nb,
                                            int nbz, int ow, int pf, int least, int i, int j, int k, float &re,
                                            float &im, float &w)
{
    constexpr int HC = HL * HL * HZ;
    const int ui = i - ow, uj = j - ow, uk = k - ow;  // >= 0 for cells >= -H
    const int bi1 = min(ui / BS, nb - 1), bj1 = min(uj / BS, nb - 1), bk1 = min(uk / BZ, nbz - 1);
    const int bi0 = ui < HL ? 0 : (ui - HL + BS) / BS, bj0 = uj < HL ? 0 : (uj - HL + BS) / BS;
    const int bk0 = uk < HZ ? 0 : (uk - HZ + BZ) / BZ;
    re = im = w = 0.f;
    for (int bk = bk1; bk >= bk0; bk--)
        for (int bj = bj1; bj >= bj0; bj--)
            for (int bi = bi1; bi >= bi0; bi--) {
                const int b = (bk * nb + bj) * nb + bi;
                const int cc = ((uk - BZ * bk) * HL + (uj - BS * bj)) * HL + (ui - BS * bi);
                const int i0 = item_off[3 * b], n = item_off[3 * b + 3] - i0;
                const int i1 = i0 + (n >= least ? 1 : n);  // summed into the first one
                for (int it = i0; it < i1; it++) {
                    const float *p = part + (size_t)it * pf + cc;
                    re += p[0];
                    im += p[HC];
                    w += p[2 * HC];
                }
            }
}

// Storage voxel (xs, ys, zs) of the half volume receives, per
// add_complex_at_fast (libEM/emdata_core.h:368-413): the direct cells
// (xs, j, k) with wrap(j) = ys, wrap(k) = zs; the conjugate cells (-xs, j, k)
// with wrapneg(j) = ys, wrapneg(k) = zs; on the x = 0 and x = P/2 planes the
// conjugate copies of the double insertion (value only) and, at x = P/2,
// the x = -P/2 cells added twice with their weight once; at (0,0,0) and
// (P/2,0,0) the real part and weight with the imaginary part set to 0.
// PATCH: a wave takes 8 x 8 voxels of a plane and an XCD whole planes (blocks
// go round the 8 XCDs), so that the lines of a partial brick's plane, read
// for each of the many bricks over a voxel, meet in one L1 and L2.  It pays
// where those planes are whole lines, the 8 x 8 of the 6-cell Gaussians (some
// 14 bricks over a voxel; bound by those lines): 4.6 -> 3.2 ms for 700,000
// items at pad 384, 0.47 -> 0.36 for 61,000 at 160.  With 9 x 9 planes and
// 1.4 bricks over a voxel (gauss_2) whole planes per XCD took 0.70 instead of
// 0.59 ms at pad 384, and with the 10 x 10 of gridding_7 both took 0.89
// instead of 0.65 at 192.
template <int BS, int HL, int BZ, int HZ, bool PATCH>
__global__ void __launch_bounds__(256) k_merge_partials(const float *__restrict__ part, const int *__restrict__ item_off,
                                                        const int *__restrict__ ctl, BrickGeom g, InsertConst c,
                                                        float2 *data, float *norm)
{
    if (ctl[3]) return;
    const int least = reduce_least(item_off, g.nb * g.nb * g.nbz);
    const int H = c.H, P = c.P, nb = g.nb, nbz = g.nbz, ow = g.ow, pf = g.part_floats;
    int xs, ys, zs;
    if (PATCH) {
        const int nx = (H + 32) / 32, per = nx * ((P + 7) / 8), m = blockIdx.x / 8, in = m % per;
        zs = m / per * 8 + blockIdx.x % 8;
        ys = in / nx * 8 + (threadIdx.x >> 3) % 8;
        xs = in % nx * 32 + (threadIdx.x >> 6) * 8 + threadIdx.x % 8;
        if (zs >= P || ys >= P || xs > H) return;
    } else {
        const long long n = (long long)blockIdx.x * 256 + threadIdx.x, rest = n / (H + 1);
        if (rest >= (long long)P * P) return;
        xs = (int)(n - rest * (H + 1));
        ys = (int)(rest % P);
        zs = (int)(rest / P);
    }
    const size_t idx = ((size_t)zs * P + ys) * (H + 1) + xs;
    float r, i, w;
    if (ys == 0 && zs == 0 && (xs == 0 || xs == H)) {
        partial_sum<BS, HL, BZ, HZ>(part, item_off, nb, nbz, ow, pf, least, xs, 0, 0, r, i, w);
        if (xs == H) {
            float r2, i2, w2;
            partial_sum<BS, HL, BZ, HZ>(part, item_off, nb, nbz, ow, pf, least, -H, 0, 0, r2, i2, w2);
            r += r2;
            i += i2;
            w += w2;
        }
        if (r == 0.f && i == 0.f && w == 0.f) return;
        float2 d = data[idx];
        d.x += r;
        d.y = 0.f;
        data[idx] = d;
        norm[idx] += w;
        return;
    }
    int jd[2], njd = 0, jn[2], njn = 0, kd[2], nkd = 0, kn[2], nkn = 0;
    if (ys <= H) jd[njd++] = ys;
    if (ys >= H) jd[njd++] = ys - P;
    if (ys <= H) jn[njn++] = -ys;
    if (ys >= H && P - ys <= H && P - ys != -ys) jn[njn++] = P - ys;
    if (zs <= H) kd[nkd++] = zs;
    if (zs >= H) kd[nkd++] = zs - P;
    if (zs <= H) kn[nkn++] = -zs;
    if (zs >= H && P - zs <= H && P - zs != -zs) kn[nkn++] = P - zs;
    float dre = 0.f, dim = 0.f, dw = 0.f;
    for (int a = 0; a < njd; a++)
        for (int b = 0; b < nkd; b++) {
            partial_sum<BS, HL, BZ, HZ>(part, item_off, nb, nbz, ow, pf, least, xs, jd[a], kd[b], r, i, w);
            dre += r;
            dim += i;
            dw += w;
        }
    for (int a = 0; a < njn; a++)
        for (int b = 0; b < nkn; b++) {
            if (xs == 0 || xs == H) {
                partial_sum<BS, HL, BZ, HZ>(part, item_off, nb, nbz, ow, pf, least, xs, jn[a], kn[b], r, i, w);
                dre += r;
                dim -= i;
                if (xs == H) {
                    partial_sum<BS, HL, BZ, HZ>(part, item_off, nb, nbz, ow, pf, least, -H, jn[a], kn[b], r, i, w);
                    dre += 2.f * r;
                    dim -= 2.f * i;
                    dw += w;
                }
            } else {
                partial_sum<BS, HL, BZ, HZ>(part, item_off, nb, nbz, ow, pf, least, -xs, jn[a], kn[b], r, i, w);
                dre += r;
                dim -= i;
                dw += w;
            }
        }
    if (dre == 0.f && dim == 0.f && dw == 0.f) return;
    float2 d = data[idx];
    d.x += dre;
    d.y += dim;
    data[idx] = d;
    norm[idx] += dw;
}

hipError_t launch_merge_partials(BrickGeom g, BinBuffers b, InsertConst c, float2 *data, float *norm, hipStream_t s)
{
    const unsigned linear = (unsigned)(((long long)c.P * c.P * (c.H + 1) + 255) / 256);
    const unsigned patches = (unsigned)((c.H + 32) / 32 * ((c.P + 7) / 8) * ((c.P + 7) / 8 * 8));
    const int nbricks = g.nb * g.nb * g.nbz;
    const long long units = (long long)nbricks * ((g.part_floats + 255) / 256);
    hipLaunchKernelGGL(k_reduce_items, dim3((unsigned)std::min(2048LL, (units + 3) / 4)), dim3(256), 0, s, b.part,
                       b.item_off, b.ctl, nbricks, g.part_floats);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
#define FH_MERGE(BS, HL, BZ, HZ, PATCH)                                                                                \
    if (g.bs == BS && g.halo == HL && g.bsz == BZ && g.haloz == HZ) {                                                  \
        hipLaunchKernelGGL((k_merge_partials<BS, HL, BZ, HZ, PATCH>), dim3(PATCH ? patches : linear), dim3(256), 0, s, \
                           b.part, b.item_off, b.ctl, g, c, data, norm);                                                      \
        return hipGetLastError();                                                                                      \
    }
    FH_MERGE(BRICK, HALO, BRICK, HALO, false)
    FH_MERGE(G6_BX, G6_HX, G6_BZ, G6_HZ, true)
    FH_MERGE(WBS, WBS + 2, WBS, WBS + 2, false)
    FH_MERGE(WBS, WBS + 4, WBS, WBS + 4, false)
    FH_MERGE(WBS, WBS + 6, WBS, WBS + 6, false)
    FH_MERGE(WBS, WBS + 8, WBS, WBS + 8, false)
#undef FH_MERGE
    return hipErrorInvalidValue;
}

}  // namespace fh
