// Particle prep (edge mean, pad, phase origin, r2c FFT, CTF sign, scale) and
// finish (weight normalisation, 3-D c2r FFT, depad, phase origin) kernels.
//
// Prep follows programs/e2make3dpar.py:630-654,704-716 and
// FourierReconstructor::preprocess_slice (libEM/reconstructor.cpp:1022-1061);
// finish follows libEM/reconstructor.cpp:315-388,1552-1641.  All FFTs are
// LDS Stockham transforms (fh_device.hpp) over tiles of T transforms.
#include "fh_device.hpp"

namespace fh {

// ---------------------------------------------------------------- plans
bool make_plan(int N, FftPlan *p)
{
    p->N = N;
    p->npass = 0;
    int m = N;
    while (m % 8 == 0 && p->npass < 16) { p->radix[p->npass++] = 8; m /= 8; }
    while (m % 6 == 0 && p->npass < 16) { p->radix[p->npass++] = 6; m /= 6; }
    while (m % 4 == 0 && p->npass < 16) { p->radix[p->npass++] = 4; m /= 4; }
    while (m % 2 == 0 && p->npass < 16) { p->radix[p->npass++] = 2; m /= 2; }
    while (m % 3 == 0 && p->npass < 16) { p->radix[p->npass++] = 3; m /= 3; }
    while (m % 5 == 0 && p->npass < 16) { p->radix[p->npass++] = 5; m /= 5; }
    while (m % 7 == 0 && p->npass < 16) { p->radix[p->npass++] = 7; m /= 7; }
    while (m % 11 == 0 && p->npass < 16) { p->radix[p->npass++] = 11; m /= 11; }
    while (m % 13 == 0 && p->npass < 16) { p->radix[p->npass++] = 13; m /= 13; }
    if (m != 1 || N <= 1 || N >= 65536) return false;
    int ns = 1;
    for (int i = 0; i < p->npass; i++) {
        p->ns[i] = ns;
        p->mag[i] = ns == 1 ? 0u : (unsigned)((((uint64_t)1 << 32) + ns - 1) / ns);
        p->twm[i] = N / (ns * p->radix[i]);
        ns *= p->radix[i];
    }
    return true;
}

// ---------------------------------------------------------------- edge mean
// EMData::get_edge_mean, 2-D branch (libEM/emdata_metadata.cpp:713-736):
// float pair sums of opposite edge pixels accumulated in double.
__global__ void __launch_bounds__(256) k_edge_mean(const float *__restrict__ imgs, int B, float *__restrict__ means)
{
    const float *d = imgs + (size_t)blockIdx.x * B * B;
    double acc = 0.0;
    for (int i = threadIdx.x; i < 2 * B; i += blockDim.x) {
        float pair;
        if (i < B) pair = d[i] + d[(size_t)(B - 1) * B + i];
        else {
            int r = i - B;
            pair = d[(size_t)r * B] + d[(size_t)r * B + B - 1];
        }
        acc += (double)pair;
    }
    __shared__ double red[256];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) means[blockIdx.x] = (float)red[0] / (float)(B * 2 + B * 2);
}

hipError_t launch_edge_mean(const float *imgs, int n, int B, float *means, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_edge_mean, dim3(n), dim3(256), 0, s, imgs, B, means);
    return hipGetLastError();
}

// ---------------------------------------------------------------- launch shapes
// Compute units of the current device (persistent grids), cached per device.
static int device_cus()
{
    static int cus[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cus[dev] == 0) {
        int v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
        cus[dev] = v;
    }
    return cus[dev];
}

// Every transform pass below is one kernel family: T interleaved transforms of
// length P per tile in LDS, 256 threads, E tile elements per thread, the next
// tile read into registers while the current one is transformed.  E is a
// template bound (T P <= 256 E), so that the register arrays and the
// butterflies per thread are sized to the length's class and not to the
// longest one.  T = 8 (64-byte runs of adjacent columns) up to P = 400 where
// the passes walk along columns, 4 above and for the passes along rows.
#define FH_ROW_CLASS(P, CALL)             \
    do {                                  \
        if ((P) <= 256) { CALL(4, 4); }   \
        else if ((P) <= 512) { CALL(4, 8); } \
        else if ((P) <= 640) { CALL(4, 10); } \
        else { CALL(4, 16); }             \
    } while (0)
#define FH_COL_CLASS(P, CALL)             \
    do {                                  \
        if ((P) <= 128) { CALL(8, 4); }   \
        else if ((P) <= 256) { CALL(8, 8); } \
        else if ((P) <= 400) { CALL(8, 13); } \
        else if ((P) <= 512) { CALL(4, 8); } \
        else if ((P) <= 640) { CALL(4, 10); } \
        else { CALL(4, 16); }             \
    } while (0)

// Pads with a compile-time plan; others take the runtime plan.
#define FIXED_PADS(X) X(96) X(192) X(288) X(384) X(480) X(600)

// Waves per SIMD the register allocation of the runtime-plan passes must
// allow (none of them spills; the compile-time ones are left alone, held to
// 3-4 waves they spill at 600 and take 1.67 instead of 1.12 ms).
constexpr int tile_waves(int nf, int E) { return nf ? 1 : E <= 4 ? 5 : E <= 8 ? 4 : E < 16 ? 3 : 2; }

// twiddles + one tile
static size_t tile_lds(int P, int T) { return sizeof(float2) * (size_t)P * (T + 1); }

// Persistent blocks: the tiles of XCD x (blocks b = x mod 8) are the
// contiguous range [x ntiles / 8, (x + 1) ntiles / 8), so the tiles that share
// cache lines meet in the same L2.
struct TileWalk {
    int t, end, step;
    __device__ TileWalk(int ntiles)
    {
        const int G8 = gridDim.x / 8, x = blockIdx.x % 8, lb = blockIdx.x / 8;
        const int lo = (int)((long long)ntiles * x / 8), hi = (int)((long long)ntiles * (x + 1) / 8);
        t = lo + lb;
        end = hi;
        step = G8;
    }
};

// Their grid: resident blocks per CU times the CUs, a multiple of 8 (one
// share per XCD), at most the tiles rounded up to 8.
template <typename K>
static int persistent_grid(K kernel, size_t lds, int ntiles)
{
    const int cus = device_cus();
    if (ntiles <= cus) return (ntiles + 7) / 8 * 8;
    int per = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, 256, lds) != hipSuccess || per < 1) per = 1;
    const int g = std::min(cus * per, (ntiles + 7) / 8 * 8);
    return std::max(8, g / 8 * 8);
}

// fixed plan (NF, compile time) or the runtime plan
template <int T, int NF, int E>
__device__ __forceinline__ void fft_run(float2 *A, const FftPlan &plan, const float2 *tw)
{
    if constexpr (NF != 0) fft_fixed<T, NF>(A, tw);
    else fft_lds_inplace<T, E>(A, plan, tw);
}

// The spectra a, c (k = 0..P/2) of two real signals A, C as the conjugate of
// A + iC, element k and its mirror P - k: a forward transform of it is the
// conjugate of the pair's inverse transform.
template <int T>
__device__ __forceinline__ void store_pair(float2 *A, int k, int t, int P, float4 v)
{
    const int H = P / 2;
    const bool self = k == 0 || k == H;
    if (self) v.y = v.w = 0.f;
    A[k * T + t] = make_float2(v.x - v.w, -(v.y + v.z));
    if (!self) A[(P - k) * T + t] = make_float2(v.x + v.w, v.y - v.z);
}

// ---------------------------------------------------------------- CTF sign
// CTF_SIGN of EMAN2Ctf::compute_2d_complex (libEM/ctf.cpp:1076-1090) at
// the Fourier pixel of radius hyp = Util::hypot_fast(x, y).  Evaluated with the reference's float
// operation order (no contraction); the sign of cos is taken in double.
// cos(t) < 0 exactly when floor(t / pi - 1/2) is even; away from the
// zeros of cos (|frac| > 1e-9, far above the ~1e-13 error of u) the parity
// decides, next to them cos itself is evaluated.  The single-precision
// u_f = fma(t, fl(1/pi), -1/2) is within 2 |u| 2^-24 < 5e-4 of u for
// |u| < 4096, so a fraction of u_f more than 1e-3 from an integer already
// fixes floor(u); only the rest take the double-precision test.
__device__ __forceinline__ float ctf_sign(float hyp, float defocus, const CtfConst &cc)
{
#pragma clang fp contract(off)
    const float s = hyp * cc.ds;
    const float gam = -cc.g1 * s * s * s * s + cc.g2 * defocus * s * s;
    const float tf = gam - cc.acac;
    const float uf = __fmaf_rn(tf, 0.318309886f, -0.5f);
    const float flf = floorf(uf);
    const float frf = uf - flf;
    if (fabsf(uf) < 4096.f && frf > 1e-3f && frf < 1.f - 1e-3f) return (((int)flf) & 1) == 0 ? -1.0f : 1.0f;
    const double t = (double)tf;
    const double u = t * 0.31830988618379067154 - 0.5;
    const double fl = floor(u);
    const double fr = u - fl;
    if (fr > 1e-9 && fr < 1.0 - 1e-9) return (((long long)fl) & 1) == 0 ? -1.0f : 1.0f;
    return cos(t) < 0 ? -1.0f : 1.0f;
}

// ---------------------------------------------------------------- 2-D prep
// The 2-D r2c transform runs columns first, so that the larger second pass
// reads and writes whole rows.
// Pass 1 (k_prep_ycols): 2T image columns per block, packed pairwise into T
// complex transforms along y (padded row ys = (b + off + P/2) mod P of image
// row b, edge mean subtracted, zero outside the image); the half spectrum
// ky = 0..P/2 of each real column is split out of the pair and stored to the
// intermediate I[p][ky][c] (row pitch IP, c = image column), 2T columns of a
// row per store run.
// Pass 2 (k_prep_xrows): T intermediate rows per block, transformed along x
// (padded column xs = (c + off + P/2) mod P); slice row ky takes
// kx = 0..P/2 and, for 0 < ky < P/2, row P - ky takes the conjugates of
// kx' = (P - kx) mod P (F(kx, -ky) = conj F(-kx, ky) for a real image), both
// times the CTF sign and scale of (kx, |ky|), evaluated once for the pair.
// XF: the image of pass 1 is the "xform" processor's resampling of the
// source (xform_sample), taken where it is read, all P x P of it.
// FLIP: pass 2 of the flip back to real space: the row's spectrum times the
// sign goes through the inverse x transform in the same tile, and row ky of
// J[p][ky][x] (pitch P, the slice's own memory) is written; pass 3
// (k_flip_ycols) takes J back along y to the flipped P x P image.
// Bound by memory where the plan is a compile-time one (2.0 and 3.0 GB per
// 3,000 particles of 256 px at pad 384 in 0.54 and 0.78 ms, 3.8 TB/s; a copy
// reaches 4.9), by address and twiddle arithmetic where it is not: the same
// through the runtime plan 0.58 and 1.03 ms.  5,000 particles of 169 px at pad
// 256, flipped, resampled and transformed again: 5.1 ms, 8.9 by rows, then
// columns in place, columns back, rows back and a resampling pass.
template <int T, int NF, int E, bool XF>
__global__ void __launch_bounds__(256, tile_waves(NF, E))
    k_prep_ycols(const float *__restrict__ imgs, int B, int Pr, int off, int n, const float *__restrict__ means,
                 const float *__restrict__ xf, float2 *__restrict__ inter, int IP, FftPlan plan,
                 const float2 *__restrict__ twg)
{
    const int P = NF ? NF : Pr, H = P / 2;
    constexpr int EL = NF ? (T * NF + 255) / 256 : E;
    const int Bv = XF ? P : B, offv = XF ? 0 : off;  // the image that is transformed
    extern __shared__ float2 smem[];
    float2 *tw = smem;
    float2 *A = tw + P;
    load_twiddles(tw, twg, P);
    const int ng = (Bv + 2 * T - 1) / (2 * T);
    TileWalk w(ng * n);
    // element e of the thread: (ys, t) = ((tid + 256 e) / T, (tid + 256 e) % T), image columns c, c + 1
    // of padded row ys; slots outside the image hold the mean (zero after the subtraction)
    float2 v[EL];
    float vmean = 0.f;
    auto fetch = [&](int tile) {
        const int tid = NF ? (int)threadIdx.x : opaque_tid();
        const int p = tile / ng, c0 = (tile - p * ng) * 2 * T;
        const float mean = means ? means[p] : 0.f;
        const float *img = imgs + (size_t)p * B * B;
        vmean = XF ? 0.f : mean;
#pragma unroll
        for (int e = 0; e < EL; e++) {
            const int idx = tid + 256 * e;
            const int t = idx % T, ys = idx / T;
            int b = ys - offv - H;  // image row of padded row ys, in [-P, P/2)
            if (b < 0) b += P;
            const int c = c0 + 2 * t;
            const bool in = idx < T * P && b < Bv;
            if constexpr (XF) {
                v[e].x = in && c < Bv ? xform_sample(img, B, P, off, mean, xf + 6 * (size_t)p, c, b) : 0.f;
                v[e].y = in && c + 1 < Bv ? xform_sample(img, B, P, off, mean, xf + 6 * (size_t)p, c + 1, b) : 0.f;
            } else {
                v[e].x = in && c < Bv ? img[(size_t)b * B + c] : mean;
                v[e].y = in && c + 1 < Bv ? img[(size_t)b * B + c + 1] : mean;
            }
        }
    };
    if (w.t < w.end) fetch(w.t);
    for (; w.t < w.end; w.t += w.step) {
        const int tid = NF ? (int)threadIdx.x : opaque_tid();
        const int p = w.t / ng, c0 = (w.t - p * ng) * 2 * T;
        const float mean = vmean;
#pragma unroll
        for (int e = 0; e < EL; e++) {
            const int idx = tid + 256 * e;
            if (idx < T * P) A[idx] = make_float2(v[e].x - mean, v[e].y - mean);  // A[ys T + t]
        }
        __syncthreads();
        if (w.t + w.step < w.end) fetch(w.t + w.step);
        fft_run<T, NF, E>(A, plan, tw);
        float2 *I = inter + (size_t)p * (H + 1) * IP;
        for (int idx = tid; idx < T * (H + 1); idx += 256) {
            const int t = idx % T;
            const int k = idx / T;
            const int c = c0 + 2 * t;
            if (c >= Bv) continue;
            const float2 z1 = A[k * T + t];
            const float2 z2 = A[(k == 0 ? 0 : P - k) * T + t];
            // columns c and c + 1 (for odd B the last pair's second column is
            // zero and lands in the row padding, IP > B)
            *reinterpret_cast<float4 *>(I + (size_t)k * IP + c) = make_float4(
                0.5f * (z1.x + z2.x), 0.5f * (z1.y - z2.y), 0.5f * (z1.y + z2.y), -0.5f * (z1.x - z2.x));
        }
        __syncthreads();  // the tile is read before the next one is stored
    }
}

// defocus2 (optional): a second defocus per particle; the flip is then the
// product of the two signs (the dfdf flip of e2make3dpar.py:698-709)
template <int T, int NF, int E, bool FLIP>
__global__ void __launch_bounds__(256, tile_waves(NF, E))
    k_prep_xrows(int B, int Pr, int off, int n, const float2 *__restrict__ inter, int IP, float2 *__restrict__ slices,
                 const float *__restrict__ defocus, const float *__restrict__ defocus2, CtfConst cc, float scale,
                 FftPlan plan, const float2 *__restrict__ twg)
{
    const int P = NF ? NF : Pr, H = P / 2, NG = (H + T) / T;
    constexpr int EL = NF ? (T * NF + 255) / 256 : E;
    extern __shared__ float2 smem[];
    float2 *tw = smem;
    float2 *A = tw + P;
    load_twiddles(tw, twg, P);
    TileWalk w(NG * n);
    // element e of the thread: (xs, t) = ((tid + 256 e) / T, (tid + 256 e) % T): a wave reads runs of
    // 64 / T columns of T intermediate rows and writes LDS without bank conflicts
    float2 v[EL];
    auto fetch = [&](int tile) {
        const int tid = NF ? (int)threadIdx.x : opaque_tid();
        const int p = tile / NG, k0 = (tile - p * NG) * T;
        const float2 *I = inter + (size_t)p * (H + 1) * IP;
#pragma unroll
        for (int e = 0; e < EL; e++) {
            const int idx = tid + 256 * e;
            const int t = idx % T, xs = idx / T;
            const int k = k0 + t;
            int c = xs - off - H;  // image column of padded column xs
            if (c < 0) c += P;
            v[e] = (idx < T * P && k <= H && c < B) ? I[(size_t)k * IP + c] : make_float2(0.f, 0.f);
        }
    };
    if (w.t < w.end) fetch(w.t);
    for (; w.t < w.end; w.t += w.step) {
        const int tid = NF ? (int)threadIdx.x : opaque_tid();
        const int p = w.t / NG, k0 = (w.t - p * NG) * T;
#pragma unroll
        for (int e = 0; e < EL; e++) {
            const int idx = tid + 256 * e;
            if (idx < T * P) A[idx] = v[e];  // A[xs T + t]
        }
        __syncthreads();
        if (w.t + w.step < w.end) fetch(w.t + w.step);
        fft_run<T, NF, E>(A, plan, tw);
        const float df = defocus ? defocus[p] : 0.f;
        const float df2 = defocus2 ? defocus2[p] : 0.f;
        auto flip = [&](int kx, int ky) {  // sign times scale
            const float hyp = defocus ? sqrt_int_rn(kx * kx + ky * ky) : 0.f;  // Util::hypot_fast(x, y)
            float ss = defocus ? ctf_sign(hyp, df, cc) * scale : scale;
            if (defocus2) ss = ss * ctf_sign(hyp, df2, cc);
            return ss;
        };
        float2 *sl = slices + (size_t)p * P * (H + 1);
        if constexpr (FLIP) {
            for (int idx = tid; idx < T * (H + 1); idx += 256) {
                const int t = idx % T, k = idx / T;
                const float ss = flip(k, k0 + t);
                float2 *a = A + k * T + t;
                *a = make_float2(a->x * ss, -(a->y * ss));
                if (k > 0 && k < H) {
                    a = A + (P - k) * T + t;
                    *a = make_float2(a->x * ss, -(a->y * ss));
                }
            }
            __syncthreads();
            fft_run<T, NF, E>(A, plan, tw);
#pragma unroll
            for (int e = 0; e < EL; e++) {
                const int idx = tid + 256 * e;
                const int t = idx % T, xs = idx / T;
                if (idx < T * P && k0 + t <= H) sl[(size_t)(k0 + t) * P + xs] = make_float2(A[idx].x, -A[idx].y);
            }
        } else {
            // two rows per lane (one 16-byte LDS read per column), lanes along the
            // rows: whole-row store runs
            static_assert(T % 2 == 0, "row pairs");
            constexpr int TH = 256 / (T / 2);  // threads per row pair
            const int t0 = 2 * (tid / TH);
            for (int kx = tid % TH; kx <= H; kx += TH) {
                const float4 u2 = *reinterpret_cast<const float4 *>(A + kx * T + t0);
                const float4 q2 = *reinterpret_cast<const float4 *>(A + (kx == 0 ? 0 : P - kx) * T + t0);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int ky = k0 + t0 + h;
                    if (ky > H) continue;
                    const float ss = flip(kx, ky);
                    const float ux = h ? u2.z : u2.x, uy = h ? u2.w : u2.y;
                    const float qx = h ? q2.z : q2.x, qy = h ? q2.w : q2.y;
                    sl[(size_t)ky * (H + 1) + kx] = make_float2(ux * ss, uy * ss);
                    if (ky > 0 && ky < H) sl[(size_t)(P - ky) * (H + 1) + kx] = make_float2(qx * ss, -qy * ss);
                }
            }
        }
        __syncthreads();  // the tile is read before the next one is stored
    }
}

// J[p][ky][x] (k_prep_xrows<FLIP>) along y to real P x P images times scale,
// phase origin to the centre: pairs of real columns per complex transform
template <int T, int E>
__global__ void __launch_bounds__(256, tile_waves(0, E))
    k_flip_ycols(const float2 *__restrict__ J, int P, int n, float *__restrict__ out, float scale, FftPlan plan,
                 const float2 *__restrict__ twg)
{
    const int H = P / 2, ng = (P + 2 * T - 1) / (2 * T);
    constexpr int EH = E / 2 + 1;
    extern __shared__ float2 smem[];
    float2 *tw = smem;
    float2 *A = tw + P;
    load_twiddles(tw, twg, P);
    TileWalk w(ng * n);
    float4 v[EH];
    auto fetch = [&](int tile) {
        const int tid = opaque_tid();
        const int p = tile / ng, c0 = (tile - p * ng) * 2 * T;
        const float2 *src = J + (size_t)p * P * (H + 1);
#pragma unroll
        for (int e = 0; e < EH; e++) {
            const int idx = tid + 256 * e;
            const int c = c0 + 2 * (idx % T), k = idx / T;
            v[e] = k <= H && c < P ? *reinterpret_cast<const float4 *>(src + (size_t)k * P + c)
                                   : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    if (w.t < w.end) fetch(w.t);
    for (; w.t < w.end; w.t += w.step) {
        const int tid = opaque_tid();
        const int p = w.t / ng, c0 = (w.t - p * ng) * 2 * T;
#pragma unroll
        for (int e = 0; e < EH; e++) {
            const int idx = tid + 256 * e;
            if (idx / T <= H) store_pair<T>(A, idx / T, idx % T, P, v[e]);
        }
        __syncthreads();
        if (w.t + w.step < w.end) fetch(w.t + w.step);
        fft_run<T, 0, E>(A, plan, tw);
        float *o = out + (size_t)p * P * P;
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int idx = tid + 256 * e;
            const int c = c0 + 2 * (idx % T), y = idx / T;
            if (y >= P || c >= P) continue;
            const float2 r = A[idx];
            float *row = o + (size_t)(y + H < P ? y + H : y + H - P) * P;
            row[c + H < P ? c + H : c + H - P] = r.x * scale;
            row[c + 1 + H < P ? c + 1 + H : c + 1 + H - P] = -r.y * scale;
        }
        __syncthreads();  // the tile is read before the next one is stored
    }
}

// Intermediate row pitch of box B (a multiple of 16 columns: 128-byte rows,
// and one padding column for odd B).
int prep_inter_pitch(int B) { return (B + 16) & ~15; }

// n particles through the two passes, in sub-batches of the intermediate's
// room (inter_n particles of box P).  xf: resample by these inverse 2-D
// transforms first; flip_back: leave J instead of slices.
static hipError_t prep2d_passes(const float *imgs, int n, int B, int P, const float *means, const float *xf,
                                bool flip_back, float2 *slices, float2 *inter, int inter_n, const float *defocus,
                                const float *defocus2, CtfConst cc, float scale, const FftPlan &plan, const float2 *tw,
                                hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const int d = B - P;
    const int fl = d >= 0 ? d / 2 : -((-d + 1) / 2);  // clip_inplace Region((B-P)//2, ...), e2make3dpar.py:651-652
    const int off = -fl;
    const int Bt = xf ? P : B, offt = xf ? 0 : off;  // what is transformed
    const int H = P / 2, IP = prep_inter_pitch(Bt);
    const long long room = (long long)inter_n * prep_inter_pitch(P);
    const int sub = (int)std::max(1LL, room / IP);
    for (int i0 = 0; i0 < n; i0 += sub) {
        const int m = std::min(sub, n - i0);
        const float *im = imgs + (size_t)i0 * B * B;
        const float *mn = means ? means + i0 : nullptr;
        const float *xm = xf ? xf + 6 * (size_t)i0 : nullptr;
        float2 *sl = slices + (size_t)i0 * P * (H + 1);
        const float *df = defocus ? defocus + i0 : nullptr;
        const float *df2 = defocus2 ? defocus2 + i0 : nullptr;
#define FH_Y(TT, EE, NN, XX)                                                                                      \
        {                                                                                                         \
            const auto k = k_prep_ycols<TT, NN, EE, XX>;                                                          \
            const size_t l = tile_lds(P, TT);                                                                     \
            hipLaunchKernelGGL(k, dim3(persistent_grid(k, l, (Bt + 2 * TT - 1) / (2 * TT) * m)), dim3(256), l, s, im, \
                               B, P, off, m, mn, xm, inter, IP, plan, tw);                                        \
        }
#define FH_X(TT, EE, NN, FF)                                                                                      \
        {                                                                                                         \
            const auto k = k_prep_xrows<TT, NN, EE, FF>;                                                          \
            const size_t l = tile_lds(P, TT);                                                                     \
            hipLaunchKernelGGL(k, dim3(persistent_grid(k, l, (H + TT) / TT * m)), dim3(256), l, s, Bt, P, offt, m, \
                               inter, IP, sl, df, df2, cc, scale, plan, tw);                                      \
        }
#define FH_Y_PLAIN(TT, EE) FH_Y(TT, EE, 0, false)
#define FH_Y_XF(TT, EE) FH_Y(TT, EE, 0, true)
#define FH_X_PLAIN(TT, EE) FH_X(TT, EE, 0, false)
#define FH_X_FLIP(TT, EE) FH_X(TT, EE, 0, true)
#define FH_FIXED(NN)                                                        \
        if (!xf && !flip_back && P == NN) {                                 \
            FH_Y(8, 0, NN, false)                                           \
            FH_X(4, 0, NN, false)                                           \
        } else
        FIXED_PADS(FH_FIXED)
        {
            if (xf) FH_COL_CLASS(P, FH_Y_XF);
            else FH_COL_CLASS(P, FH_Y_PLAIN);
            if (flip_back) FH_ROW_CLASS(P, FH_X_FLIP);
            else FH_ROW_CLASS(P, FH_X_PLAIN);
        }
#undef FH_FIXED
#undef FH_Y_PLAIN
#undef FH_Y_XF
#undef FH_X_PLAIN
#undef FH_X_FLIP
#undef FH_Y
#undef FH_X
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// The whole prep of n particles into their slices.
hipError_t launch_prep2d(const float *imgs, int n, int B, int P, const float *means, float2 *slices,
                         float2 *inter, int inter_n, const float *defocus, const float *defocus2, CtfConst cc,
                         float scale, const FftPlan &plan, const float2 *tw, hipStream_t s)
{
    return prep2d_passes(imgs, n, B, P, means, nullptr, false, slices, inter, inter_n, defocus, defocus2, cc, scale,
                         plan, tw, s);
}

// The prep of n particles (box B, edge means or null) resampled by the
// inverse 2-D transforms xf (6 floats each), without a flip.
hipError_t launch_prep2d_xform(const float *imgs, int n, int B, int P, const float *means, const float *xf,
                               float2 *slices, float2 *inter, int inter_n, float scale, const FftPlan &plan,
                               const float2 *tw, hipStream_t s)
{
    return prep2d_passes(imgs, n, B, P, means, xf, false, slices, inter, inter_n, nullptr, nullptr, CtfConst{}, scale,
                         plan, tw, s);
}

// The padded particles flipped in Fourier space and back in real space: P x P
// images, phase origin at the centre, times scale.  work: n slices of memory.
hipError_t launch_flip2d(const float *imgs, int n, int B, int P, const float *means, float2 *work, float2 *inter,
                         int inter_n, const float *defocus, const float *defocus2, CtfConst cc, float scale,
                         float *out, const FftPlan &plan, const float2 *tw, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipError_t e = prep2d_passes(imgs, n, B, P, means, nullptr, true, work, inter, inter_n, defocus, defocus2, cc, 1.0f,
                                 plan, tw, s);
    if (e != hipSuccess) return e;
#define FH_CALL(TT, EE)                                                                                           \
    {                                                                                                             \
        const auto k = k_flip_ycols<TT, EE>;                                                                      \
        const size_t l = tile_lds(P, TT);                                                                         \
        hipLaunchKernelGGL(k, dim3(persistent_grid(k, l, (P + 2 * TT - 1) / (2 * TT) * n)), dim3(256), l, s, work, P, \
                           n, out, scale, plan, tw);                                                              \
    }
    FH_COL_CLASS(P, FH_CALL);
#undef FH_CALL
    return hipGetLastError();
}

// ---------------------------------------------------------------- normalise
// ReconstructorVolumeData::normalize_threed (libEM/reconstructor.cpp:315-388).
// The conjugate-plane loop pairs each weight on the x=0 and x=P/2 planes
// with its partner at (-y,-z); the pairing is an involution, so each fixed
// weight is norm[self] + norm[partner] except for self-paired cells, of which
// five are doubled.  Step 1 writes the fixed planes to plane_tmp [2][P][P].
__global__ void k_norm_planes(const float *__restrict__ norm, int P, float *__restrict__ plane_tmp)
{
    const int H = P / 2;
    const size_t nnx = H + 1;
    const int ys = blockIdx.x * blockDim.x + threadIdx.x;
    const int zs = blockIdx.y;
    const int pl = blockIdx.z;  // 0: x=0, 1: x=H
    if (ys >= P) return;
    const int xs = pl ? H : 0;
    const int yp = (P - ys) % P, zp = (P - zs) % P;
    const float self = norm[((size_t)zs * P + ys) * nnx + xs];
    float v;
    if (yp == ys && zp == zs) {
        bool dbl;
        if (pl == 0) dbl = (ys == 0 && zs == H) || (ys == H && zs == 0) || (ys == H && zs == H);
        else dbl = (ys == 0 && zs == H) || (ys == H && zs == 0);
        v = dbl ? self * 2 : self;
    } else {
        v = self + norm[((size_t)zp * P + yp) * nnx + xs];
    }
    plane_tmp[((size_t)pl * P + zs) * P + ys] = v;
}

__global__ void k_normalize(float2 *__restrict__ data, float *__restrict__ norm, int P, int sqrtnorm,
                            const float *__restrict__ plane_tmp)
{
    const int H = P / 2;
    const size_t nnx = H + 1;
    const size_t total = nnx * P * P;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const int xs = (int)(i % nnx);
        const size_t yz = i / nnx;
        float d;
        if (xs == 0 || xs == H) {
            const int ys = (int)(yz % P), zs = (int)(yz / P);
            d = plane_tmp[((size_t)(xs == 0 ? 0 : 1) * P + zs) * P + ys];
            norm[i] = d;
        } else {
            d = norm[i];
        }
        if (sqrtnorm) d = sqrt_rn(d);
        float2 v = data[i];
        if (d == 0) v = make_float2(0.f, 0.f);
        else v = make_float2(__fdiv_rn(v.x, d), __fdiv_rn(v.y, d));
        data[i] = v;
    }
}

hipError_t launch_normalize(float2 *data, float *norm, int P, int sqrtnorm, float *plane_tmp, hipStream_t s)
{
    hipLaunchKernelGGL(k_norm_planes, dim3((P + 127) / 128, P, 2), dim3(128), 0, s, norm, P, plane_tmp);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_normalize, dim3(4096), dim3(256), 0, s, data, norm, P, sqrtnorm, plane_tmp);
    return hipGetLastError();
}

// ---------------------------------------------------------------- 3-D inverse
// Bound by memory: 0.46 GB per pass at 384^3 in 0.13 ms (3.5 TB/s); by blocks
// of one tile each, whose reads nothing covers, 0.31 along an axis and 0.27 to
// real rows.
// In-place inverse complex transform of length P along one axis (stride
// axis_stride) for tiles of T consecutive x; inverse = conj o forward o conj.
// FWD: the forward transform instead (no conjugation), each output n times
// (-1)^n: the axis's phase origin moved to the corner
template <int T, int E, int FWD>
__global__ void __launch_bounds__(256, tile_waves(0, E))
    k_fft_axis(float2 *__restrict__ data, int P, size_t axis_stride, size_t outer_stride, int outer, FftPlan plan,
               const float2 *__restrict__ twg)
{
    extern __shared__ float2 smem[];
    float2 *tw = smem;
    float2 *A = tw + P;
    const int H = P / 2, ng = (H + T) / T;
    load_twiddles(tw, twg, P);
    TileWalk w(ng * outer);
    float2 v[E];
    auto fetch = [&](int tile) {
        const int tid = opaque_tid();
        const int o = tile / ng, x0 = (tile - o * ng) * T;
        const float2 *base = data + (size_t)o * outer_stride;
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int idx = tid + 256 * e;
            const int x = x0 + idx % T, j = idx / T;
            v[e] = j < P && x <= H ? base[(size_t)j * axis_stride + x] : make_float2(0.f, 0.f);
        }
    };
    if (w.t < w.end) fetch(w.t);
    for (; w.t < w.end; w.t += w.step) {
        const int tid = opaque_tid();
        const int o = w.t / ng, x0 = (w.t - o * ng) * T;
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int idx = tid + 256 * e;
            if (idx < T * P) A[idx] = FWD ? v[e] : conjf2(v[e]);
        }
        __syncthreads();
        if (w.t + w.step < w.end) fetch(w.t + w.step);
        fft_lds_inplace<T, E>(A, plan, tw);
        float2 *base = data + (size_t)o * outer_stride;
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int idx = tid + 256 * e;
            const int x = x0 + idx % T, j = idx / T;
            if (j < P && x <= H) {
                const float2 r = A[idx];
                base[(size_t)j * axis_stride + x] = FWD ? ((j & 1) ? make_float2(-r.x, -r.y) : r) : conjf2(r);
            }
        }
        __syncthreads();  // the tile is read before the next one is stored
    }
}

template <int FWD>
static hipError_t fft_axis(float2 *data, int P, size_t axis_stride, size_t outer_stride, int outer,
                           const FftPlan &plan, const float2 *tw, hipStream_t s)
{
    const int H = P / 2;
#define FH_CALL(TT, EE)                                                                                           \
    {                                                                                                             \
        const auto k = k_fft_axis<TT, EE, FWD>;                                                                   \
        const size_t l = tile_lds(P, TT);                                                                         \
        hipLaunchKernelGGL(k, dim3(persistent_grid(k, l, (H + TT) / TT * outer)), dim3(256), l, s, data, P,       \
                           axis_stride, outer_stride, outer, plan, tw);                                           \
    }
    FH_COL_CLASS(P, FH_CALL);
#undef FH_CALL
    return hipGetLastError();
}

hipError_t launch_fft3d_inverse_zy(float2 *data, int P, const FftPlan &plan, const float2 *tw, hipStream_t s)
{
    const size_t row = P / 2 + 1, plane = (size_t)P * row;
    hipError_t e = fft_axis<0>(data, P, plane, row, P, plan, tw, s);  // along z, at fixed y
    if (e != hipSuccess) return e;
    return fft_axis<0>(data, P, row, plane, P, plan, tw, s);  // along y, at fixed z
}

// c2r along x for row pairs, x 1/P^3 (do_ift_inplace, emdata_transform.cpp:392-425),
// depad, and phase origin to centre (fftshift) on the write.
// nz planes of P rows; shift 1: fftshift of the written volume (3-D finish),
// shift 2: fftshift of each plane (a batch of 2-D images), 0: rows written
// in place (2-D projection).
template <int T, int E>
__global__ void __launch_bounds__(256, tile_waves(0, E))
    k_c2r_x(const float2 *__restrict__ data, int P, int nz, int shift, float *__restrict__ out, float scale,
            FftPlan plan, const float2 *__restrict__ twg)
{
    constexpr int EH = E / 2 + 1;
    extern __shared__ float2 smem[];
    float2 *tw = smem;
    float2 *A = tw + P;
    const int H = P / 2;
    const size_t nrows = (size_t)nz * P;  // even: P is
    load_twiddles(tw, twg, P);
    TileWalk w((int)((nrows + 2 * T - 1) / (2 * T)));
    float4 v[EH];
    auto fetch = [&](int tile) {
        const int tid = opaque_tid();
#pragma unroll
        for (int e = 0; e < EH; e++) {
            const int idx = tid + 256 * e;
            const size_t r = (size_t)tile * 2 * T + 2 * (idx % T);
            const int k = idx / T;
            v[e] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (k <= H && r < nrows) {
                const float2 a = data[r * (H + 1) + k], c = data[(r + 1) * (H + 1) + k];
                v[e] = make_float4(a.x, a.y, c.x, c.y);
            }
        }
    };
    if (w.t < w.end) fetch(w.t);
    for (; w.t < w.end; w.t += w.step) {
        const int tid = opaque_tid();
#pragma unroll
        for (int e = 0; e < EH; e++) {
            const int idx = tid + 256 * e;
            if (idx / T <= H) store_pair<T>(A, idx / T, idx % T, P, v[e]);
        }
        __syncthreads();
        if (w.t + w.step < w.end) fetch(w.t + w.step);
        fft_lds_inplace<T, E>(A, plan, tw);
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int idx = tid + 256 * e;
            const size_t r = (size_t)w.t * 2 * T + 2 * (idx % T);
            const int x = idx / T;
            if (x >= P || r >= nrows) continue;
            const float2 z = A[idx];
            const int xc = !shift ? x : x + H < P ? x + H : x + H - P;
            const int zz = (int)(r / P), y = (int)(r - (size_t)zz * P);
            const int zc = shift != 1 ? zz : zz + H < P ? zz + H : zz + H - P;
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int yq = y + q, yc = !shift ? yq : yq + H < P ? yq + H : yq + H - P;
                out[((size_t)zc * P + yc) * P + xc] = (q == 0 ? z.x : -z.y) * scale;
            }
        }
        __syncthreads();  // the tile is read before the next one is stored
    }
}

static hipError_t c2r_rows(const float2 *data, int P, int nz, int shift, float *out, float scale,
                           const FftPlan &plan, const float2 *tw, hipStream_t s)
{
    const int nrows = nz * P;
#define FH_CALL(TT, EE)                                                                                           \
    {                                                                                                             \
        const auto k = k_c2r_x<TT, EE>;                                                                           \
        const size_t l = tile_lds(P, TT);                                                                         \
        hipLaunchKernelGGL(k, dim3(persistent_grid(k, l, (nrows + 2 * TT - 1) / (2 * TT))), dim3(256), l, s, data, P, \
                           nz, shift, out, scale, plan, tw);                                                      \
    }
    FH_ROW_CLASS(P, FH_CALL);
#undef FH_CALL
    return hipGetLastError();
}

hipError_t launch_c2r_x(const float2 *data, int P, float *out, float scale, const FftPlan &plan, const float2 *tw,
                        hipStream_t s)
{
    return c2r_rows(data, P, P, 1, out, scale, plan, tw, s);
}

// 2-D do_ift of one (P+2) x P complex image (emdata_transform.cpp:330-375):
// inverse FFT along y of the P/2+1 columns, c2r along x, x 1/P^2.
hipError_t launch_ift2d(float2 *data, int P, float *out, const FftPlan &plan, const float2 *tw, hipStream_t s)
{
    hipError_t e = fft_axis<0>(data, P, P / 2 + 1, 0, 1, plan, tw, s);
    if (e != hipSuccess) return e;
    return c2r_rows(data, P, 1, 0, out, 1.0f / ((float)P * (float)P), plan, tw, s);
}

// do_ift of n complex images (P x (P/2+1) each, in place: overwritten) into n
// real P x P images with scale, phase origin to the centre
hipError_t launch_ift2d_batch(float2 *data, int n, int P, float *out, float scale, const FftPlan &plan,
                              const float2 *tw, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const size_t row = P / 2 + 1;
    hipError_t e = fft_axis<0>(data, P, row, (size_t)P * row, n, plan, tw, s);
    if (e != hipSuccess) return e;
    return c2r_rows(data, P, n, 2, out, scale, plan, tw, s);
}

// ---------------------------------------------------------------- forward 3-D
// do_fft of a real P^3 volume with the phase origin moved to the corner (the
// Fourier-space xform.phaseorigin.tocorner, center_origin_fft): the particle
// prep's passes over the P z planes (their load index applies the x and y
// shift), then the z transform, each output times (-1)^z.  vol: P^3 floats,
// out: P x P x (P/2+1) complex.
hipError_t launch_fft3d_forward_corner(const float *vol, int P, float2 *out, float2 *inter, int inter_n,
                                       const FftPlan &plan, const float2 *tw, hipStream_t s)
{
    hipError_t e = launch_prep2d(vol, P, P, P, nullptr, out, inter, inter_n, nullptr, nullptr, CtfConst{}, 1.0f, plan,
                                 tw, s);
    if (e != hipSuccess) return e;
    const size_t row = P / 2 + 1;
    return fft_axis<1>(out, P, (size_t)P * row, row, P, plan, tw, s);
}

// ---------------------------------------------------------------- task merge
// e2spa_make3d.py:180-184: a task's normalised volume times its normout
// ("math.multamplitude": both floats of a voxel times its weight), added to
// the sum; the normout added to the summed weights
__global__ void k_merge_add(float2 *__restrict__ data, float *__restrict__ norm, const float2 *__restrict__ threed,
                            const float *__restrict__ normv, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float w = normv[i];
        const float2 t = threed[i];
        const float2 d = data[i];
        data[i] = make_float2(d.x + t.x * w, d.y + t.y * w);
        norm[i] = norm[i] + w;
    }
}

// e2spa_make3d.py:186-187: the summed weights' reciprocal ("math.reciprocal",
// 0 where the weight is 0), times the summed volume
__global__ void k_merge_scale(float2 *__restrict__ data, const float *__restrict__ norm, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float w = norm[i];
        const float r = w == 0.0f ? 0.0f : 1.0f / w;
        const float2 d = data[i];
        data[i] = make_float2(d.x * r, d.y * r);
    }
}

hipError_t launch_merge_add(float2 *data, float *norm, const float2 *threed, const float *normv, size_t n,
                            hipStream_t s)
{
    const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(k_merge_add, dim3(blocks), dim3(256), 0, s, data, norm, threed, normv, n);
    return hipGetLastError();
}

hipError_t launch_merge_scale(float2 *data, const float *norm, size_t n, hipStream_t s)
{
    const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(k_merge_scale, dim3(blocks), dim3(256), 0, s, data, norm, n);
    return hipGetLastError();
}

// ---------------------------------------------------------------- fills
// Fill kernels instead of hipMemsetAsync so the sequences stay capturable.
__global__ void k_fill_f32(float *p, float v, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}
__global__ void k_fill_i32(int *p, int v, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}
__global__ void k_scale_f32(float *p, float v, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = p[i] * v;
}

static unsigned fill_grid(size_t n)
{
    size_t g = (n + 255) / 256;
    return (unsigned)(g < 8192 ? (g ? g : 1) : 8192);
}

hipError_t launch_fill_f32(float *p, float v, size_t n, hipStream_t s)
{
    hipLaunchKernelGGL(k_fill_f32, dim3(fill_grid(n)), dim3(256), 0, s, p, v, n);
    return hipGetLastError();
}
hipError_t launch_fill_i32(int *p, int v, size_t n, hipStream_t s)
{
    hipLaunchKernelGGL(k_fill_i32, dim3(fill_grid(n)), dim3(256), 0, s, p, v, n);
    return hipGetLastError();
}
hipError_t launch_scale_f32(float *p, float v, size_t n, hipStream_t s)
{
    hipLaunchKernelGGL(k_scale_f32, dim3(fill_grid(n)), dim3(256), 0, s, p, v, n);
    return hipGetLastError();
}

// setup_seed weights (libEM/reconstructor.cpp:870-904): seed weight
// everywhere, halved on the x=0 and x=P/2 planes except four cells.
__global__ void k_seed_weights(float *norm, int P, float w)
{
    const int H = P / 2;
    const size_t nnx = H + 1;
    const size_t total = nnx * P * P;
    const float half = (float)(w / 2.0);
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const int xs = (int)(i % nnx);
        const size_t yz = i / nnx;
        const int ys = (int)(yz % P), zs = (int)(yz / P);
        float v = w;
        if (xs == 0 || xs == H) {
            v = half;
            if ((ys == H && zs == 0) || (ys == 0 && zs == H)) v = w;
        }
        norm[i] = v;
    }
}

hipError_t launch_seed_weights(float *norm, int P, float w, hipStream_t s)
{
    hipLaunchKernelGGL(k_seed_weights, dim3(4096), dim3(256), 0, s, norm, P, w);
    return hipGetLastError();
}

}  // namespace fh
