/*
 * accel_gpu.hip -- HIP kernels for the accelsearch hot path on MI355X
 * (gfx950) and the thin C ABI (agpu.h) that the C host calls.
 *
 *   k_resp_z / k_template_dft : FP64 z-response templates, FFT'd to the
 *       correlation length in FP64 and kept resident as FP32
 *       (src/accel_utils.c:153-170, src/responses.c:228-316).
 *   k_block_norms_wave / k_block_norms : exact block medians (one
 *       wavefront per window by ballot counts for windows of <= 1024
 *       bins, a workgroup radix select in LDS above) and the block-median
 *       normalisation of src/accel_utils.c:1087-1099.
 *   k_corr : fused overlap-save correlation -- spectrum
 *       segment -> Stockham FFT in LDS -> multiply by each
 *       template -> inverse FFT -> |.|^2 -> raw plane row
 *       (the template loop of src/accel_utils.c:1141-1190).
 *   k_harmsum : harmonic summing with the reference's index rules and
 *       per-block normalisation, and the threshold of search_ffdotpows
 *       (src/accel_utils.c:1261-1452); k_harmbound : the same hits from
 *       bounds of the powers, the sums formed only where a bound crosses.
 */
#include <hip/hip_runtime.h>
#include <pthread.h>
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "agpu.h"

static thread_local char g_err[512];   /* per host thread */

#define AGPU_CHECK(call)                                                          \
    do {                                                                          \
        hipError_t e_ = (call);                                                   \
        if (e_ != hipSuccess) {                                                   \
            snprintf(g_err, sizeof(g_err), "%s:%d %s: %s", __FILE__, __LINE__,    \
                     #call, hipGetErrorString(e_));                               \
            return -1;                                                            \
        }                                                                         \
    } while (0)

void agpu_set_error(const char *msg)
{
    snprintf(g_err, sizeof(g_err), "%s", msg);
}

static int fail(const char *msg)
{
    snprintf(g_err, sizeof(g_err), "%s", msg);
    return -2;
}

#include "dev_fresnel.h"
#define ACCEL_SIGMA_FN __device__ static
#define ACCEL_SIGMA_TOL 1e-15
#include "accel_sigma.h"

#define CORR_N 4096   /* half-bins per correlation segment */

/* One tap of the z-response kernel with roffset = 0 and numbetween = 2
 * (src/responses.c:159-225 for |z| < 1e-4, :228-316 otherwise). */
__global__ void k_resp_z(const int *zs, const int *nks, int nkmax, double2 *resp)
{
    const double PI = 3.14159265358979323846;
    const int t = blockIdx.y;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int nk = nks[t];
    if (k >= nkmax)
        return;
    double2 out = make_double2(0.0, 0.0);
    if (k < nk) {
        const double z = (double) zs[t];
        if (fabs(z) < 1e-4) {
            /* exp(-i pi f) sinc(f), f = k/2 - nk/4 */
            double f = 0.5 * k - 0.25 * nk;
            double r = -PI * f;
            double sv, cv;
            sincospi(-f, &sv, &cv);
            double sinc = (f == 0.0) ? 1.0 : sv / r;
            out = make_double2(cv * sinc, sv * sinc);
        } else {
            int signz = (z < 0.0) ? -1 : 1;
            double zd = signz * 1.41421356237309504880 / sqrt(fabs(z));
            double cons = zd / 2.0;
            double r = -0.5 * z + 0.25 * nk - 0.5 * k;   /* exact on this grid */
            double yy = r * zd;
            double zz = yy + z * zd;
            double sv, cv;
            sincospi(r * r / z, &sv, &cv);               /* cos/sin(pi r^2 / z) */
            double fsy, fcy, fsz, fcz;
            d_fresnl(yy, &fsy, &fcy);
            d_fresnl(zz, &fsz, &fcz);
            double tre = signz * (fcz - fcy);
            double tim = fsy - fsz;
            out = make_double2((tre * cv - tim * sv) * cons, -(tre * sv + tim * cv) * cons);
        }
    }
    resp[(size_t) t * nkmax + k] = out;
}

/* Jerk template (|w| >= 1e-4), src/responses.c:333-418: the reference
 * samples a chirp of npts points into FP32, zero-pads it to 2 npts and
 * real-FFTs it, keeping numkern bins around 2 fbar.  Here: the same FP32
 * samples (phase in FP64, rounded like the reference's data[] array), then
 * the FP64 DFT at exactly the kept bins.  One workgroup per template. */
__global__ __launch_bounds__(256) void k_resp_w(const int *zs, const int *ws, const int *nks,
                                                const int *npts_arr, const int *tlist,
                                                int nkmax, double2 *resp)
{
    extern __shared__ float xs[];
    const double TWOPI = 6.28318530717958647692;
    const int t = tlist[blockIdx.x];
    const double z = (double) zs[t], w = (double) ws[t];
    const int nk = nks[t], npts = npts_arr[t];
    const double dt = 1.0 / (double) npts;
    const double amp = 2.0 * dt;
    const int fbar = npts / 4;
    const double f = (double) fbar - 0.5 * z + w / 12.0;
    const double fd = (z - 0.5 * w) / 2.0;
    const double fdd = w / 6.0;
    for (int ii = threadIdx.x; ii < npts; ii += blockDim.x) {
        const double tt = ii * dt;
        const double phase = TWOPI * (tt * (tt * (tt * fdd + fd) + f));
        xs[ii] = (float) (amp * cos(phase));
    }
    __syncthreads();
    const long long ntot = 2LL * npts;
    const long long first = 2LL * fbar - nk / 2;
    for (int k = threadIdx.x; k < nk; k += blockDim.x) {
        const long long m = first + k;
        double ws_, wc_;
        sincospi(-2.0 * (double) (m % ntot) / (double) ntot, &ws_, &wc_);
        double ar = 0.0, ai = 0.0, cr = 1.0, ci = 0.0;
        for (int i = 0; i < npts; i++) {
            if ((i & 511) == 0 && i) {   /* re-seed the rotation exactly */
                sincospi(-2.0 * (double) ((m * i) % ntot) / (double) ntot, &ci, &cr);
            }
            const double x = (double) xs[i];
            ar += x * cr;
            ai += x * ci;
            const double nr = cr * wc_ - ci * ws_;
            ci = cr * ws_ + ci * wc_;
            cr = nr;
        }
        resp[(size_t) t * nkmax + k] = make_double2(ar, ai);
    }
}

/* Correlation templates for segments of L = 4096 half-bins whose odd
 * half-bins are zero.  With T[f] = conj(sum_m resp[nk/2+m]
 * e^{-2 pi i f m / L}) / L, the even and the odd half-bins of the
 * correlation are inverse transforms of half the length, of
 *   Te[f] = T[f] + T[f + L/2]                       (the even taps)
 *   To[f] = (T[f] - T[f + L/2]) e^{2 pi i f / L}    (the odd taps)
 * times the data's transform.  Both in FP64, rounded to FP32, stored in
 * the order in which k_corr reads them: a thread's pairs f = j + 128 p,
 * f + 1024 side by side. */
__global__ void k_template_dft(const double2 *resp, const int *nks, int nkmax, float2 *T)
{
    const int L = CORR_N;
    const int t = blockIdx.y;
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= L / 2)
        return;
    const int nk = nks[t], half = nk / 2;   /* half is even */
    const double2 *rp = resp + (size_t) t * nkmax;
    double ws, wc, s0, c0, s1, c1;
    sincospi(-4.0 * (double) f / (double) L, &ws, &wc);    /* two taps on */
    sincospi(2.0 * (double) f / (double) L, &s1, &c1);
    const int e0 = (int) (((long long) f * half) % L);     /* m = -half */
    sincospi(2.0 * (double) e0 / (double) L, &s0, &c0);
    double cr = c0, ci = s0, er = 0.0, ei = 0.0, odr = 0.0, odi = 0.0;
    for (int m = 0; m < nk; m += 2) {
        const double2 v = rp[m], u = rp[m + 1];
        er += v.x * cr - v.y * ci;
        ei += v.x * ci + v.y * cr;
        odr += u.x * cr - u.y * ci;   /* without the odd tap's own e^{-2 pi i f / L} */
        odi += u.x * ci + u.y * cr;
        const double nr = cr * wc - ci * ws;
        ci = cr * ws + ci * wc;
        cr = nr;
    }
    /* conj(sum_odd e^{-2 pi i f / L}) e^{2 pi i f / L} = conj(sum_odd) e^{4 pi i f / L} */
    const double inv = 2.0 / (double) L;
    const int j = f & 127, r = f >> 7;
    float2 *o = T + (size_t) t * L + (r & 7) * 256 + 2 * j + (r >> 3);
    o[0] = make_float2((float) (er * inv), (float) (-ei * inv));
    const double tr = c1 * c1 - s1 * s1, ti = 2.0 * c1 * s1;
    o[L / 2] = make_float2((float) ((odr * tr + odi * ti) * inv),
                           (float) ((odr * ti - odi * tr) * inv));
}

/* ------------------------------------------------------------------ */
/* Exact block medians: radix select over the FP32 power bit patterns  */
/* ------------------------------------------------------------------ */
#define NORM_MAXN 15360   /* keys in LDS: 60 KiB, with the 1 KiB histogram under 64 KiB */

/* Inclusive prefix sum of hist[0..255] by a 256-thread block (one bucket
 * per thread); returns the sum up to and including this thread's bucket. */
__device__ static unsigned block_scan256(unsigned v, unsigned *wsum)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        unsigned o = __shfl_up(v, d, 64);
        if (lane >= d)
            v += o;
    }
    if (lane == 63)
        wsum[wv] = v;
    __syncthreads();
    unsigned add = 0;
    for (int w = 0; w < wv; w++)
        add += wsum[w];
    __syncthreads();
    return v + add;
}

/* k-th smallest (0-based) of keys[0..n) by 4 passes of 8-bit buckets */
__device__ static unsigned radix_select(const unsigned *keys, int n, int k, unsigned *hist,
                                        unsigned *sh)
{
    unsigned prefix = 0, mask = 0;
    for (int shift = 24; shift >= 0; shift -= 8) {
        hist[threadIdx.x] = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += 256) {
            unsigned key = keys[i];
            if ((key & mask) == prefix)
                atomicAdd(&hist[(key >> shift) & 255u], 1u);
        }
        __syncthreads();
        unsigned h = hist[threadIdx.x];
        unsigned incl = block_scan256(h, sh + 2);
        unsigned excl = incl - h;
        if ((unsigned) k >= excl && (unsigned) k < incl) {
            sh[0] = prefix | ((unsigned) threadIdx.x << shift);
            sh[1] = (unsigned) k - excl;
        }
        __syncthreads();
        prefix = sh[0];
        k = (int) sh[1];
        mask |= 255u << shift;
        __syncthreads();
    }
    return prefix;
}

/* Exact median of the FP32 powers |x|^2 of spectrum bins [lo, lo+n)
 * (lo relative to the array; bins outside [0, numbins) count as 0), as
 * PRESTO's median(): the middle order statistic, or for even n the mean of
 * the two middle ones formed in FP64 and rounded to FP32.  Called by the
 * whole workgroup; keys holds n entries of dynamic LDS. */
__device__ static float block_median(const float2 *spec, long long numbins, long long lo, int n,
                                     unsigned *keys, unsigned *hist, unsigned *sh)
{
    /* the reference forms r*r + i*i with two roundings (no FMA) */
#pragma clang fp contract(off)
    for (int i = threadIdx.x; i < n; i += 256) {
        long long b = lo + i;
        float p = 0.0f;
        if (b >= 0 && b < numbins) {
            float2 v = spec[b];
            p = v.x * v.x + v.y * v.y;
        }
        keys[i] = __float_as_uint(p);
    }
    __syncthreads();
    const int lhs = (n - 1) / 2, rhs = n / 2;
    const unsigned ka = radix_select(keys, n, lhs, hist, sh);
    float med = __uint_as_float(ka);
    if (lhs != rhs) {
        /* the (lhs+1)-th key: ka again if more than lhs+1 keys are <= ka,
         * else the smallest key above ka */
        unsigned cnt = 0, mn = 0xffffffffu;
        for (int i = threadIdx.x; i < n; i += 256) {
            unsigned key = keys[i];
            cnt += (key <= ka);
            if (key > ka && key < mn)
                mn = key;
        }
        if (threadIdx.x == 0) {
            sh[4] = 0;
            sh[5] = 0xffffffffu;
        }
        __syncthreads();
        atomicAdd(&sh[4], cnt);
        atomicMin(&sh[5], mn);
        __syncthreads();
        const unsigned kb = (sh[4] >= (unsigned) rhs + 1) ? ka : sh[5];
        med = (float) (0.5 * ((double) __uint_as_float(ka) + (double) __uint_as_float(kb)));
    }
    __syncthreads();
    return med;
}

__global__ __launch_bounds__(256) void k_block_norms(const float2 *spec, long long numbins,
                                                     long long lobin_file,
                                                     const agpu_window *win, double *norm,
                                                     float *nsq)
{
    extern __shared__ unsigned keys[];
    __shared__ unsigned hist[256];
    __shared__ unsigned sh[8];
    const agpu_window w = win[blockIdx.x];
    const float med = block_median(spec, numbins, w.lobin - lobin_file, w.numdata, keys, hist, sh);
    if (threadIdx.x == 0) {
        double nv = 1.0 / sqrt((double) med / 0.69314718055994530942);
        norm[blockIdx.x] = nv;
        nsq[blockIdx.x] = (float) (nv * nv);
    }
}

/* Windows of at most NW_KPL * 64 bins: one wavefront per window, four
 * windows per workgroup, and no workgroup barrier.  Each lane keeps KPL
 * power bit patterns in registers, 4, 8, 12 or 16 by the window's length (the
 * work is proportional: 1.05 million bins in blocks of <= 200, 32 us with 16,
 * 13 with 4); bins past the window hold 0xffffffff, above every power.  The
 * k-th smallest pattern is built
 * bit by bit from the top: a bit is kept when fewer than k + 1 patterns
 * lie below the value with it set, the counts coming from wave ballots.
 * The selected patterns, hence the medians and norms, are those of
 * k_block_norms. */
#define NW_KPL 16

template <int KPL>
__device__ static unsigned wave_select(const unsigned *key, unsigned k)
{
    unsigned v = 0;
    for (int bit = 31; bit >= 0; bit--) {
        const unsigned c = v | (1u << bit);
        unsigned below = 0;
#pragma unroll
        for (int j = 0; j < KPL; j++)
            below += (unsigned) __popcll(__ballot(key[j] < c));
        if (below <= k)
            v = c;
    }
    return v;
}

/* The exact median of window [lo, lo+n) (n <= KPL * 64) by one wavefront;
 * every lane returns it. */
template <int KPL>
__device__ static float wave_median(const float2 *spec, long long numbins, long long lo,
                                          int n, int lane)
{
#pragma clang fp contract(off)
    unsigned key[KPL];
#pragma unroll
    for (int j = 0; j < KPL; j++) {
        const int i = lane + 64 * j;
        unsigned kv = 0xffffffffu;
        if (i < n) {
            const long long b = lo + i;
            float p = 0.0f;
            if (b >= 0 && b < numbins) {
                const float2 v = spec[b];
                p = v.x * v.x + v.y * v.y;
            }
            kv = __float_as_uint(p);
        }
        key[j] = kv;
    }
    const unsigned lhs = (unsigned) (n - 1) / 2, rhs = (unsigned) n / 2;
    const unsigned ka = wave_select<KPL>(key, lhs);
    if (lhs == rhs)
        return __uint_as_float(ka);
    /* the (lhs+1)-th pattern: ka again if more than lhs + 1 patterns are
     * <= ka, else the smallest pattern above ka */
    unsigned le = 0, mn = 0xffffffffu;
#pragma unroll
    for (int j = 0; j < KPL; j++) {
        le += (unsigned) __popcll(__ballot(key[j] <= ka));
        if (key[j] > ka && key[j] < mn)
            mn = key[j];
    }
    for (int d = 32; d >= 1; d >>= 1) {
        const unsigned o = __shfl_xor(mn, d, 64);
        mn = o < mn ? o : mn;
    }
    const unsigned kb = le >= rhs + 1 ? ka : mn;
    return (float) (0.5 * ((double) __uint_as_float(ka) + (double) __uint_as_float(kb)));
}

/* n <= NW_KPL * 64, the same for all lanes */
__device__ static float wave_block_median(const float2 *spec, long long numbins, long long lo,
                                          int n, int lane)
{
    const int kpl = (__builtin_amdgcn_readfirstlane(n) + 255) >> 8;
    switch (kpl) {
    case 0:
    case 1: return wave_median<4>(spec, numbins, lo, n, lane);
    case 2: return wave_median<8>(spec, numbins, lo, n, lane);
    case 3: return wave_median<12>(spec, numbins, lo, n, lane);
    default: return wave_median<16>(spec, numbins, lo, n, lane);
    }
}

__global__ __launch_bounds__(256) void k_block_norms_wave(const float2 *spec, long long numbins,
                                                          long long lobin_file,
                                                          const agpu_window *win, int nwin,
                                                          double *norm, float *nsq)
{
    const int wid = (int) blockIdx.x * 4 + (int) (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (wid >= nwin)
        return;
    const agpu_window w = win[wid];
    const float med = wave_block_median(spec, numbins, w.lobin - lobin_file, w.numdata, lane);
    if (lane == 0) {
        const double nv = 1.0 / sqrt((double) med / 0.69314718055994530942);
        norm[wid] = nv;
        nsq[wid] = (float) (nv * nv);
    }
}

/* One window given by value (the accel.h surface normalises one block
 * per subharm_fderivs_vol call). */
__global__ __launch_bounds__(256) void k_block_norm1(const float2 *spec, long long numbins,
                                                     long long lobin_file, long long lobin,
                                                     int numdata, double *norm, float *nsq)
{
    extern __shared__ unsigned keys[];
    __shared__ unsigned hist[256];
    __shared__ unsigned sh[8];
    const float med = block_median(spec, numbins, lobin - lobin_file, numdata, keys, hist, sh);
    if (threadIdx.x == 0) {
        double nv = 1.0 / sqrt((double) med / 0.69314718055994530942);
        norm[0] = nv;
        nsq[0] = (float) (nv * nv);
    }
}

/* De-reddening (src/misc_utils.c:912-1067), block medians: mean_b =
 * median(|x|^2 of block b) / ln 2, rounded to FP32 as the reference. */
__global__ __launch_bounds__(256) void k_dered_means(const float2 *spec, long long numbins,
                                                     const agpu_window *blk, float *mean)
{
    extern __shared__ unsigned keys[];
    __shared__ unsigned hist[256];
    __shared__ unsigned sh[8];
    const agpu_window w = blk[blockIdx.x];
    const float med = block_median(spec, numbins, w.lobin, w.numdata, keys, hist, sh);
    if (threadIdx.x == 0)
        mean[blockIdx.x] = (float) ((double) med / 0.69314718055994530942);
}

/* The same block means, one wavefront per block (blocks of at most
 * NW_KPL * 64 bins, as the de-reddening's always are). */
__global__ __launch_bounds__(256) void k_dered_means_wave(const float2 *spec, long long numbins,
                                                          const agpu_window *blk, int nblk,
                                                          float *mean)
{
    const int wid = (int) blockIdx.x * 4 + (int) (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (wid >= nblk)
        return;
    const agpu_window w = blk[wid];
    const float med = wave_block_median(spec, numbins, w.lobin, w.numdata, lane);
    if (lane == 0)
        mean[wid] = (float) ((double) med / 0.69314718055994530942);
}

/* invsqrtf of src/misc_utils.c:291-302: one Newton step from the
 * 0x5f3759df estimate, in FP32 without fused operations. */
__device__ static float dered_invsqrt(float x)
{
#pragma clang fp contract(off)
    float y = __int_as_float(0x5f3759df - (__float_as_int(x) >> 1));
    return y * (1.5f - 0.5f * x * y * y);
}

/* De-reddening, scaling: bin 0 -> (1, im0); the first half of block 0 by
 * invsqrt(mean_0); then each span [middle of block b, middle of block
 * b+1) by invsqrt(mean_b + dslope_b ii), ii counted from the span start,
 * dslope_b = (mean_{b+1} - mean_b) / ((n_b + n_{b+1}) / 2); the last
 * half-block continues with the last slope (1 if there is one block).  A
 * wave per span (~200 bins): its constants once, no search for the span of
 * a bin (1.05 million bins: 16.5 us with one, 7.7 without). */
__global__ __launch_bounds__(256) void k_dered_apply(float2 *spec, long long numbins,
                                                     const agpu_window *blk, const float *mean,
                                                     int nblk, float im0)
{
#pragma clang fp contract(off)
    /* span 0: bins [1, mid_0); span b + 1: [mid_b, mid_{b+1}) */
    const int span = (int) blockIdx.x * 4 + (int) (threadIdx.x >> 6), b = span - 1;
    const int lane = threadIdx.x & 63;
    if (span > nblk)
        return;
    const long long first = b < 0 ? 1 : blk[b].lobin + blk[b].numdata / 2;
    long long end = b + 1 < nblk ? blk[b + 1].lobin + blk[b + 1].numdata / 2 : numbins;
    end = end < numbins ? end : numbins;
    const float m = mean[b < 0 ? 0 : b];
    float dslope = 0.0f;
    if (b >= 0) {
        if (b + 1 < nblk)
            dslope = (float) ((mean[b + 1] - m) / (0.5 * (blk[b].numdata + blk[b + 1].numdata)));
        else if (nblk > 1)
            dslope = (float) ((m - mean[b - 1]) / (0.5 * (blk[b - 1].numdata + blk[b].numdata)));
        else
            dslope = 1.0f;
    }
    if (span == 0 && lane == 0 && numbins > 0)
        spec[0] = make_float2(1.0f, im0);
    for (long long k = first + lane; k < end; k += 64) {
        const int ii = (int) (k - first);
        const float norm = dered_invsqrt(b < 0 ? m : m + dslope * (float) ii);
        const float2 v = spec[k];
        spec[k] = make_float2(v.x * norm, v.y * norm);
    }
}

int agpu_deredden(void *d_spec, long long numbins, const agpu_window *d_blk, int nblk,
                  int maxn, float *d_mean, float im0, void *stream)
{
    hipStream_t st = (hipStream_t) stream;
    if (nblk <= 0 || maxn <= 0 || maxn > NORM_MAXN)
        return fail("agpu_deredden: bad block table");
    if (maxn <= NW_KPL * 64)
        hipLaunchKernelGGL(k_dered_means_wave, dim3((unsigned) ((nblk + 3) / 4)), dim3(256), 0,
                           st, (const float2 *) d_spec, numbins, d_blk, nblk, d_mean);
    else
        hipLaunchKernelGGL(k_dered_means, dim3(nblk), dim3(256), sizeof(unsigned) * maxn, st,
                           (const float2 *) d_spec, numbins, d_blk, d_mean);
    AGPU_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_dered_apply, dim3((unsigned) (nblk / 4 + 1)), dim3(256), 0, st,
                       (float2 *) d_spec, numbins, d_blk, (const float *) d_mean, nblk, im0);
    AGPU_CHECK(hipGetLastError());
    return 0;
}

/* In-memory path: norm^2 of the fundamental block that last wrote each
 * half-bin -- main blocks from rh0 on, pre-population blocks from half-bin
 * 16 (r = 8) on, nothing below (src/accelsearch.c:166-205). */
__global__ void k_inmem_nsq_table(const float *nsq, int npre, int nblocks, long long rh0,
                                  int cu, long long hb_end, float *out)
{
    long long hb = (long long) blockIdx.x * blockDim.x + threadIdx.x;
    if (hb >= hb_end)
        return;
    float v = 0.0f;
    if (hb >= rh0) {
        long long b = (hb - rh0) / cu;
        if (b < nblocks)
            v = nsq[npre + b];
    } else if (hb >= 16 && npre > 0) {
        long long b = (hb - 16) / cu;
        if (b < npre)
            v = nsq[b];
    }
    out[hb] = v;
}

/* ------------------------------------------------------------------ */
/* Overlap-save correlation                                             */
/* ------------------------------------------------------------------ */

/* Butterflies (a, b) -> (a + t b, a - t b), the twiddle product fused into
 * the sum: four multiply-adds give a + t b, two more 2 a - (a + t b). */
__device__ __forceinline__ void bfly(float2 &a, float2 &b, float2 t)
{
    const float x = __builtin_fmaf(-b.y, t.y, __builtin_fmaf(b.x, t.x, a.x));
    const float y = __builtin_fmaf(b.x, t.y, __builtin_fmaf(b.y, t.x, a.y));
    b = make_float2(__builtin_fmaf(2.0f, a.x, -x), __builtin_fmaf(2.0f, a.y, -y));
    a = make_float2(x, y);
}

/* the twiddle i t */
__device__ __forceinline__ void bfly_i(float2 &a, float2 &b, float2 t)
{
    const float x = __builtin_fmaf(-b.x, t.y, __builtin_fmaf(-b.y, t.x, a.x));
    const float y = __builtin_fmaf(-b.y, t.y, __builtin_fmaf(b.x, t.x, a.y));
    b = make_float2(__builtin_fmaf(2.0f, a.x, -x), __builtin_fmaf(2.0f, a.y, -y));
    a = make_float2(x, y);
}

/* the twiddles 1 and i */
__device__ __forceinline__ void bfly1(float2 &a, float2 &b)
{
    const float2 d = make_float2(a.x - b.x, a.y - b.y);
    a = make_float2(a.x + b.x, a.y + b.y);
    b = d;
}
__device__ __forceinline__ void bfly1_i(float2 &a, float2 &b)
{
    const float2 d = make_float2(a.x + b.y, a.y - b.x);
    a = make_float2(a.x - b.y, a.y + b.x);
    b = d;
}

/* Inverse-sign DFTs of v[r] w^r, radix 2, decimation in time, in place:
 * X[k] ends in slot bitrev(k).  The twiddles of every stage come from a
 * few powers of w (the factors i are free). */
#define REV8(k) ((((k) & 1) << 2) | ((k) & 2) | (((k) >> 2) & 1))
#define REV16(k) ((((k) & 1) << 3) | (((k) & 2) << 1) | (((k) >> 1) & 2) | (((k) >> 3) & 1))

/* w = 1, after the first stage (the pairs r, r + 8) */
__device__ __forceinline__ void dft16_rest(float2 *v)
{
    const float2 w1 = make_float2(0.92387953251128675613f, 0.38268343236508977173f);
    const float2 w2 = make_float2(0.70710678118654752440f, 0.70710678118654752440f);
    const float2 w3 = make_float2(0.38268343236508977173f, 0.92387953251128675613f);
#pragma unroll
    for (int r = 0; r < 4; r++) {
        bfly1(v[r], v[r + 4]);
        bfly1_i(v[r + 8], v[r + 12]);
    }
#pragma unroll
    for (int r = 0; r < 2; r++) {
        bfly1(v[r], v[r + 2]);
        bfly(v[r + 8], v[r + 10], w2);
        bfly1_i(v[r + 4], v[r + 6]);
        bfly_i(v[r + 12], v[r + 14], w2);
    }
    bfly1(v[0], v[1]);
    bfly(v[8], v[9], w1);
    bfly(v[4], v[5], w2);
    bfly(v[12], v[13], w3);
    bfly1_i(v[2], v[3]);
    bfly_i(v[10], v[11], w1);
    bfly_i(v[6], v[7], w2);
    bfly_i(v[14], v[15], w3);
}

/* t: w^8, w^4, w^2, w^2 W8, w, w W16, w W8, w W16^3 */
__device__ __forceinline__ void dft16_tw(float2 *v, const float2 *t)
{
#pragma unroll
    for (int r = 0; r < 8; r++)
        bfly(v[r], v[r + 8], t[0]);
#pragma unroll
    for (int r = 0; r < 4; r++) {
        bfly(v[r], v[r + 4], t[1]);
        bfly_i(v[r + 8], v[r + 12], t[1]);
    }
#pragma unroll
    for (int r = 0; r < 2; r++) {
        bfly(v[r], v[r + 2], t[2]);
        bfly(v[r + 8], v[r + 10], t[3]);
        bfly_i(v[r + 4], v[r + 6], t[2]);
        bfly_i(v[r + 12], v[r + 14], t[3]);
    }
    bfly(v[0], v[1], t[4]);
    bfly(v[8], v[9], t[5]);
    bfly(v[4], v[5], t[6]);
    bfly(v[12], v[13], t[7]);
    bfly_i(v[2], v[3], t[4]);
    bfly_i(v[10], v[11], t[5]);
    bfly_i(v[6], v[7], t[6]);
    bfly_i(v[14], v[15], t[7]);
}

/* t: w^4, w^2, w, w W8 */
__device__ __forceinline__ void dft8_tw(float2 *v, const float2 *t)
{
#pragma unroll
    for (int r = 0; r < 4; r++)
        bfly(v[r], v[r + 4], t[0]);
#pragma unroll
    for (int r = 0; r < 2; r++) {
        bfly(v[r], v[r + 2], t[1]);
        bfly_i(v[r + 4], v[r + 6], t[1]);
    }
    bfly(v[0], v[1], t[2]);
    bfly(v[4], v[5], t[3]);
    bfly_i(v[2], v[3], t[2]);
    bfly_i(v[6], v[7], t[3]);
}

/* e^{2 pi i a / n}, FP64 rounded to FP32 */
__device__ static float2 unit_root(int a, int n)
{
    double s, c;
    sincospi(2.0 * (double) a / (double) n, &s, &c);
    return make_float2((float) c, (float) s);
}

/* Stores through a buffer descriptor: a 32-bit byte offset from a base that
 * all lanes share, and the offset OFF_NONE is out of range, so the hardware
 * drops that lane's store. */
#define OFF_NONE 0xffffffffu
typedef unsigned v2u __attribute__((ext_vector_type(2)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(float *p)
{
    return __builtin_amdgcn_make_buffer_rsrc(p, 0, (int) 0xfffffff0u, 0x00027000);
}
__device__ __forceinline__ void store_pair(__amdgpu_buffer_rsrc_t r, unsigned off, float2 v)
{
    const v2u u = {__float_as_uint(v.x), __float_as_uint(v.y)};
    __builtin_amdgcn_raw_buffer_store_b64(u, r, (int) off, 0, 0);
}
__device__ __forceinline__ void store_bound(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned v)
{
    __builtin_amdgcn_raw_buffer_store_b16((unsigned short) v, r, (int) off, 0, 0);
}

/* LDS slot of point i: one slot of padding every 16.  LPR(i, r): of point
 * i + r, r a multiple of 16 (an immediate offset from i's slot) */
#define LP(i) ((i) + ((i) >> 4))
#define LPR(i, r) (LP(i) + (r) + (r) / 16)
#define FFT_HALF (CORR_N / 2)
#define FFT_LDS (FFT_HALF + FFT_HALF / 16)

/* The two exchanges of an inverse FFT of 2048 points by 128 threads (16
 * points each, radix 16, 16, 8): v holds the first radix-16 DFT's output
 * in REV16 order; on return buf holds the input of the radix-8 pass.
 * Called by the whole workgroup, each half on its own buf. */
__device__ __forceinline__ void fft2048_mid(float2 *v, float2 *buf, int j, const float4 *tw2)
{
#pragma unroll
    for (int r = 0; r < 16; r++)
        buf[LP(16 * j) + r] = v[REV16(r)];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; r++)
        v[r] = buf[LPR(j, 128 * r)];
    float2 tw[8];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const float4 w = tw2[r];
        tw[2 * r] = make_float2(w.x, w.y);
        tw[2 * r + 1] = make_float2(w.z, w.w);
    }
    __syncthreads();
    dft16_tw(v, tw);
    const int base = (j >> 4) * 256 + (j & 15);
#pragma unroll
    for (int r = 0; r < 16; r++)
        buf[LPR(base, 16 * r)] = v[REV16(r)];
    __syncthreads();
}

/* Fused correlation for segments of 4096 half-bins.  The segment's odd
 * half-bins are zero, so its transform D repeats after 2048 points and the
 * even and the odd half-bins of D T's inverse transform are two transforms
 * of 2048 points (k_template_dft): waves 0-1 run the even one, waves 2-3
 * the odd one (radix 16 and 16, 16 points per thread), and the last,
 * radix-8, pass gives each thread two adjacent half-bins 8 times, stored
 * as one float2.  A workgroup keeps D in registers over its group's
 * templates.
 *
 * Bound: FP32 VALU issue.  ~570 vector instructions per thread and
 * template (196 for the template product and the first radix 16, 192, 144,
 * 32 for the powers) and ~80 for the stores, against ~760 for one
 * 4096-point transform with separate twiddle products: 2.0 ms of issue for
 * the 2^23-sample, zmax 200 search, measured 2.7 ms beside the norms
 * (3.91 ms before; 2^20 samples, 201 x 31 templates: 10.6 ms, 14.1 ms).
 * 124 VGPRs and 35 KB of LDS: four workgroups per CU, against two. */
template <bool BOUNDS>
__global__ __launch_bounds__(256, 4) void k_corr(const float2 *spec, long long numbins,
                                                 long long lobin_file, const float2 *T, int nt,
                                                 int hw, int uselen, long long hb_end,
                                                 float *plane, int groups, int tpg,
                                                 long long seg0, long long nsr)
{
    __shared__ float2 lds[2 * FFT_LDS];
    const int tid = threadIdx.x, j = tid & 127;
    const int odd = __builtin_amdgcn_readfirstlane(tid >> 7);
    float2 *buf = lds + odd * FFT_LDS;
    /* XCD x (block ids x, x + 8, ...) takes the template groups x, x + 8,
     * ... one after another, each over all nsr segments, so the workgroups
     * resident on an XCD share one group's templates in its L2 (a jerk
     * bank is ~200 MB; with 8 groups this is one group per XCD) */
    const int g = (int) (blockIdx.x & 7) + 8 * (int) ((blockIdx.x >> 3) / nsr);
    const long long seg = seg0 + (long long) (blockIdx.x >> 3) % nsr;
    const long long seg_hb = seg * (long long) uselen;
    const long long lobin = seg_hb / 2 - hw;
    const int t0 = g * tpg;
    if (t0 >= nt)
        return;
    const int t1 = min(nt, t0 + tpg);
    /* pass-2 twiddles of the 16 values of j % 16: read from LDS by every
     * template (8 of 16 apart would cost 16 registers); rows 5 float4 apart
     * keep 16-byte reads of the 16 rows on distinct banks */
    __shared__ float4 tw2l[16 * 5];
    if (tid < 128) {
        static const int off[8] = {0, 0, 0, 32, 0, 16, 32, 48}, mul[8] = {8, 4, 2, 2, 1, 1, 1, 1};
        const int m = tid >> 3, k = tid & 7;
        ((float2 *) (tw2l + 5 * m))[k] = unit_root(mul[k] * m + off[k], 256);
    }
    const float4 *tw2 = tw2l + 5 * (j & 15);
    float2 tw3[4];
    {
        tw3[0] = unit_root(4 * tid, 2048);
        tw3[1] = unit_root(2 * tid, 2048);
        tw3[2] = unit_root(tid, 2048);
        tw3[3] = unit_root(tid + 256, 2048);
    }

    /* D = conj(inverse FFT of the conjugated bins), by both halves */
    float2 D[16];
    {
        float2 v[16];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            v[r] = make_float2(0.0f, 0.0f);
            const long long bin = lobin + j + 128 * r - lobin_file;
            if (bin >= 0 && bin < numbins) {
                v[r] = spec[bin];
                v[r].y = -v[r].y;
            }
        }
#pragma unroll
        for (int r = 0; r < 8; r++)
            bfly1(v[r], v[r + 8]);
        dft16_rest(v);
        fft2048_mid(v, buf, j, tw2);   /* its first barrier covers tw2l too */
        float2 u[8];
#pragma unroll
        for (int r = 0; r < 8; r++)
            u[r] = lds[LPR(tid, 256 * r)];
        dft8_tw(u, tw3);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 8; r++)
            lds[LPR(tid, 256 * r)] = u[REV8(r)];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 16; r++) {
            D[r] = lds[LPR(j, 128 * r)];
            D[r].y = -D[r].y;
        }
    }

    /* this thread's half-bin pairs, 2 tid + 512 k - 2 hw from the segment's
     * first: byte offsets from the first tile's row */
    const long long tile_stride = (long long) nt * AGPU_ROWLEN;
    const long long tile0 = seg_hb >> AGPU_TILE_LOG2;
    const int e0 = (int) (seg_hb & (AGPU_TILE - 1));
    const int lim = (int) min((long long) uselen, hb_end - seg_hb);
    const unsigned next = 4u * (unsigned) (tile_stride - AGPU_TILE);   /* the next tile's row */
    unsigned off[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int q = 2 * tid + 512 * k - 2 * hw, e = e0 + q;   /* e: from the tile's start */
        off[k] = OFF_NONE;
        if (q >= 0 && q < lim)
            off[k] = 4u * (unsigned) e + (e < AGPU_TILE ? 0u : next);
    }
    /* the first half-bins of a tile (AGPU_HALO of them, or with BOUNDS the
     * first AGPU_BHALO groups) are repeated behind the previous tile's row:
     * does the segment touch any? */
    const int rep = BOUNDS ? AGPU_GROUP * AGPU_BHALO : AGPU_HALO;
    const bool halo = (e0 < rep && tile0 > 0) || e0 + lim > AGPU_TILE;
    const int eq = e0 + 2 * tid - 2 * hw;
    /* BOUNDS: lanes 2 i and 2 i + 1 hold one group of AGPU_GROUP half-bins
     * for each k; the even lane stores the bound for k = 2 m, the odd one
     * for k = 2 m + 1 */
    const int eg = e0 + 2 * (tid & ~1) + 512 * (tid & 1) - 2 * hw;
    unsigned goff[4];
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const int e = eg + 1024 * m, q = e - e0;
        goff[m] = OFF_NONE;
        if (BOUNDS && q >= 0 && q < lim)
            goff[m] = e < AGPU_TILE
                          ? 4u * AGPU_TILE + 2u * (unsigned) (e / AGPU_GROUP)
                          : 4u * (unsigned) tile_stride + 4u * AGPU_TILE +
                                2u * (unsigned) ((e - AGPU_TILE) / AGPU_GROUP);
    }
    float *trow = plane + tile0 * tile_stride + (long long) t0 * AGPU_ROWLEN;
    const float4 *Tt = (const float4 *) (T + (size_t) t0 * CORR_N + odd * FFT_HALF) + j;
    for (int t = t0; t < t1; t++) {
        float2 v[16];
        /* template product fused with the first radix-2 stage */
#pragma unroll
        for (int r = 0; r < 8; r++) {
            const float4 w = Tt[128 * r];
            const float2 d = D[r];
            float2 a = make_float2(__builtin_fmaf(-d.y, w.y, d.x * w.x),
                                   __builtin_fmaf(d.y, w.x, d.x * w.y));
            float2 b = D[r + 8];
            bfly(a, b, make_float2(w.z, w.w));
            v[r] = a;
            v[r + 8] = b;
        }
        dft16_rest(v);
        __syncthreads();   /* the previous template's last reads */
        fft2048_mid(v, buf, j, tw2);
        float2 u[8], o[8];
#pragma unroll
        for (int r = 0; r < 8; r++) {
            u[r] = lds[LPR(tid, 256 * r)];
            o[r] = lds[FFT_LDS + LPR(tid, 256 * r)];
        }
        dft8_tw(u, tw3);
        dft8_tw(o, tw3);
        const __amdgpu_buffer_rsrc_t row = plane_rsrc(trow);
        /* behind the previous tile's row (no tile before the first: nothing
         * is stored there, every offset is OFF_NONE) */
        const __amdgpu_buffer_rsrc_t prev =
            plane_rsrc(tile0 > 0 ? trow - tile_stride + AGPU_TILE : trow);
        float2 p[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float2 a = u[REV8(k)], b = o[REV8(k)];
            p[k] = make_float2(__builtin_fmaf(a.x, a.x, a.y * a.y),
                               __builtin_fmaf(b.x, b.x, b.y * b.y));
            store_pair(row, off[k], p[k]);
        }
        if (BOUNDS) {
            /* the group's largest power rounded up to 16 bits: an upper bound
             * that the harmonic sum looks at before it reads the powers.  By
             * their bits as signed numbers, which order like the powers.  A
             * positive NaN is above all and must not carry into the sign, so
             * the addition saturates; a negative one is below all, and a
             * group of nothing else becomes a NaN or 0: no cell of it can
             * cross, so either will do */
            int e = eg;
            asm volatile("" : "+v"(e));   /* see below */
#pragma unroll
            for (int m = 0; m < 4; m++) {
                int w[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int x = max(__float_as_int(p[2 * m + h].x),
                                      __float_as_int(p[2 * m + h].y));
                    w[h] = max(x, __builtin_amdgcn_update_dpp(
                                      0, x, 0xb1 /* lanes 1,0,3,2 */, 0xf, 0xf, true));
                }
                const unsigned bnd =
                    (unsigned) __builtin_elementwise_add_sat(tid & 1 ? w[1] : w[0], 0xffff) >> 16;
                store_bound(row, goff[m], bnd);
                if (halo) {
                    const unsigned g = (unsigned) (e + 1024 * m) / AGPU_GROUP;
                    const bool ok = goff[m] != OFF_NONE;
                    store_bound(prev, ok && tile0 > 0 && g < AGPU_BHALO ? 2 * (g + AGPU_TILE / AGPU_GROUP)
                                                           : OFF_NONE, bnd);
                    store_bound(row, ok && g - AGPU_TILE / AGPU_GROUP < AGPU_BHALO
                                         ? 4u * AGPU_TILE + 2 * g : OFF_NONE, bnd);
                }
            }
        } else if (halo) {
            /* kept out of the loop's invariants: more addresses held over the
             * loop would spill */
            int e = eq;
            asm volatile("" : "+v"(e));
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const unsigned x = (unsigned) (e + 512 * k);
                const bool ok = off[k] != OFF_NONE;
                store_pair(prev, ok && tile0 > 0 && x < AGPU_HALO ? 4 * x : OFF_NONE, p[k]);
                store_pair(row, ok && x - AGPU_TILE < AGPU_HALO ? 4 * x : OFF_NONE, p[k]);
            }
        }
        trow += AGPU_ROWLEN;
        Tt += CORR_N / 2;
    }
}

/* ------------------------------------------------------------------ */
/* Harmonic summing and thresholding                                    */
/* ------------------------------------------------------------------ */
#define HS_TPB 256
#define HS_WAVES (HS_TPB / 64)
#define HS_RT AGPU_HS_RT
#define HS_RT_ROW AGPU_HS_RT_ROW
#define HS_RT_SUB AGPU_HS_RT_SUB
#define HS_CT AGPU_HS_CT
#define HS_CPT 4
#define HS_CHUNK (HS_TPB * HS_CPT)
#define HB_CHUNK (64 * AGPU_GROUP)   /* half-bins per workgroup of k_harmbound */
#define HB_MINROWS 16                /* z rows, cells below which k_harmsum is faster */
#define HB_MINCELLS (1LL << 23)
#define HB_ROWS 64                   /* z rows per workgroup of k_harmbound at most */

__device__ __forceinline__ void emit_hit(const agpu_harmsum_args &a, int b, int s, int wi,
                                         int zi, int ii, float p)
{
    unsigned idx = atomicAdd(a.nhits, 1u);
    if (idx < a.cap) {
        agpu_hit h;
        h.block = b;
        h.stage = s;
        h.wi = wi;
        h.zi = zi;
        h.ii = ii;
        h.pow = p;
        a.hits[idx].h = h;
    }
}

/* 64-float wave loads that cover one chunk's sub-harmonic span for fraction
 * k/H (the span is at most CHUNK k/H + 1 half-bins), rounded up to a
 * multiple of the workgroup's waves so that every wave issues the same
 * loads without a bound check; the extra floats stay inside the tile row
 * and its halo. */
__host__ __device__ constexpr int hs_frac_wl_span(int k, int H)
{
    return (HS_CHUNK * k / H + 1 + 63) / 64;
}

__host__ __device__ constexpr int hs_frac_wl(int k, int H)
{
    return ((HS_CHUNK * k / H + 1 + 63) / 64 + HS_WAVES - 1) / HS_WAVES * HS_WAVES;
}

__host__ __device__ constexpr int hs_stage_wl(int S)
{
    int n = 0;
    for (int k = 1; k < (1 << S); k += 2)
        n += hs_frac_wl(k, 1 << S);
    return n;
}

/* first LDS wave-load slot (64 floats) of stage S; stages 1-3 are resident
 * together, stage 4 and stage 5 (32 harmonics) each reuse the buffer from
 * slot 0 */
__host__ __device__ constexpr int hs_stage_base(int S)
{
    int n = 0;
    for (int s = 1; s < S && s <= 4; s++)
        n += hs_stage_wl(s);
    return n;
}

__host__ __device__ constexpr int hs_max(int a, int b) { return a > b ? a : b; }

/* LDS wave-load slots of a search with NSTAGES stages */
__host__ __device__ constexpr int hs_lds_wl(int nstages)
{
    return nstages <= 4 ? hs_stage_base(nstages)
                        : hs_max(hs_max(hs_stage_base(4), hs_stage_wl(4)),
                                 nstages > 5 ? hs_stage_wl(5) : 0);
}
static_assert(hs_frac_wl(15, 16) * 64 <= AGPU_HALO && hs_frac_wl(31, 32) * 64 <= AGPU_HALO &&
                  hs_frac_wl(1, 2) * 64 <= AGPU_HALO,
              "every padded sub-harmonic span fits in a tile-row halo");

/* Index-rule variants of the harmonic sum:
 *   HS_STD   standard path, sub-harmonic half-bin rint((hb + rh_off) k / H)
 *            (src/accel_utils.c:59, 1042-1047 with the block start r on the
 *            half-bin grid);
 *   HS_INMEM in-memory path, (int)(hb k / H + 0.5) (src/accel_utils.c:1326);
 *   HS_FRAC  standard path with a block start r off the half-bin grid: the
 *            reference's FP64 expression rint(2 (startr + ii/2) k / H),
 *            evaluated per cell. */
#define HS_STD 0
#define HS_INMEM 1
#define HS_FRAC 2

/* rint (half-even) or, for HS_INMEM, (int)(x+0.5) of rh * k / 2^s.
 * 32-bit: the launcher checks that every rh * k fits. */
template <int MODE>
__host__ __device__ __forceinline__ int hs_round(int rh, int k, int s)
{
    const unsigned q = (unsigned) rh * (unsigned) k;
    const unsigned H = 1u << s;
    if (MODE == HS_INMEM)
        return (int) ((q + (H >> 1)) >> s);
    return (int) ((q + (H >> 1) - 1 + ((q >> s) & 1u)) >> s);
}

/* per-thread staging registers of one fraction: its wave loads are dealt
 * round-robin to the HS_WAVES waves */
__host__ __device__ constexpr int hs_frac_regs(int k, int H)
{
    return hs_frac_wl(k, H) / HS_WAVES;
}

__host__ __device__ constexpr int hs_stage_regs(int S)
{
    int n = 0;
    for (int k = 1; k < (1 << S); k += 2)
        n += hs_frac_regs(k, 1 << S);
    return n;
}

__host__ __device__ constexpr int hs_regs_upto(int S)   /* stages 1..S-1 */
{
    int n = 0;
    for (int s = 1; s < S; s++)
        n += hs_stage_regs(s);
    return n;
}

/* Load every sub-harmonic span of stage S for this chunk into registers:
 * wave load i (64 consecutive half-bins) goes to wave i % HS_WAVES.  The
 * span's plane offset is the chunk table's tile offset of its first
 * half-bin plus the row table's offset of its (w, z) row, both loaded as
 * scalars: every load is base + lane + immediate. */
template <int S>
__device__ __forceinline__ void hs_load(const agpu_harmsum_args &a, float *v, const long long *cb,
                                        const unsigned *rt, int wv, int lane)
{
    constexpr int H = 1 << S;
    constexpr int F0 = (H >> 1) - 1;   /* index of fraction 1/H */
    int r = 0;
#pragma unroll
    for (int k = 1; k < H; k += 2) {
        const int f = F0 + (k - 1) / 2;
        const float *b1 = a.plane + cb[1 + f] + rt[HS_RT_SUB + f];
        /* wave loads past the span's own (the padding to a multiple of the
         * waves) repeat its last one: cache hits, no extra HBM traffic */
        const int real = hs_frac_wl_span(k, H);
#pragma unroll
        for (int u = 0; u < hs_frac_regs(k, H); u++) {
            const int wl = min(wv + HS_WAVES * u, real - 1);
            v[r + u] = b1[wl * 64 + lane];
        }
        r += hs_frac_regs(k, H);
    }
}

template <int S>
__device__ __forceinline__ void hs_store(float *lds, int base, const float *v, int wv, int lane)
{
    constexpr int H = 1 << S;
    int r = 0, wl = base;
#pragma unroll
    for (int k = 1; k < H; k += 2) {
#pragma unroll
        for (int u = 0; u < hs_frac_regs(k, H); u++)
            lds[(wl + wv + HS_WAVES * u) * 64 + lane] = v[r + u];
        r += hs_frac_regs(k, H);
        wl += hs_frac_wl(k, H);
    }
}

/* Accumulate stage S from LDS, in the reference's fraction order.  nr[j]
 * is the LDS row of norm^2 values of cell j's block; clo[1 + f] the first
 * half-bin of fraction f's span. */
template <int S, int MODE>
__device__ __forceinline__ void hs_consume4(const agpu_harmsum_args &a, const float *lds,
                                            int base, const float *nr0, const float *nr1,
                                            const float *nr2, const float *nr3, const int *clo,
                                            int rh_first, const double *rf, float *acc)
{
    /* each normalised sub-harmonic power is rounded to FP32 before it is
     * added, as the reference adds stored FP32 planes
     * (src/accel_utils.c:1261-1282, 1312-1362): no fused multiply-add */
#pragma clang fp contract(off)
    static_assert(HS_CPT == 4, "four cells per thread");
    constexpr int H = 1 << S;
    constexpr int F0 = (H >> 1) - 1;
    int wl = base;
#pragma unroll
    for (int k = 1; k < H; k += 2) {
        const int f = F0 + (k - 1) / 2;
        const int lo = clo[1 + f];
        float nn[4];
        if (MODE != HS_INMEM) {
            nn[0] = nr0[1 + f];
            nn[1] = nr1[1 + f];
            nn[2] = nr2[1 + f];
            nn[3] = nr3[1 + f];
        }
        if (MODE == HS_FRAC) {
            /* rint((2 rf) (k / H)): the reference's rounding steps, FP64 */
            const double hf = (double) k / (double) H;
            const int top = hs_frac_wl(k, H) * 64 - 1;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                int o = (int) __builtin_rint((2.0 * rf[j]) * hf) - lo;
                o = o < 0 ? 0 : (o > top ? top : o);
                acc[j] = acc[j] + lds[wl * 64 + o] * nn[j];
            }
        } else {
            const int rs0 = hs_round<MODE>(rh_first + (MODE == HS_STD ? a.rh_off : 0), k, S);
            const int step = (HS_TPB / H) * k;   /* HS_TPB k / H, even */
            const float *lp = lds + wl * 64 + (rs0 - lo);
            if (MODE == HS_INMEM) {
                const float *np = a.nsq_hb + rs0;
#pragma unroll
                for (int j = 0; j < 4; j++)
                    nn[j] = np[j * step];
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                acc[j] = acc[j] + lp[j * step] * nn[j];
        }
        wl += hs_frac_wl(k, H);
    }
}

/* One workgroup = one (w,z) row x one chunk of 1024 fundamental half-bins,
 * 4 cells per thread (cell = chunk base + t + 256 j).  The grid is
 * (8 rows' slots x groups of 8 chunks): blockIdx.x = 8 row + c, chunk =
 * c_lo + 8 blockIdx.y + c.  Workgroups are dealt round-robin to the 8
 * XCDs in linear order, so every row of a chunk runs on one XCD, one row
 * after another, and the sub-harmonic rows that the rows of a chunk share
 * are read once into that XCD's L2.  Row and chunk descriptors (plane
 * offsets of every fraction's span) come from tables built with the
 * search, so the per-workgroup scalar work is a few loads and adds.  The
 * fundamental values and every sub-harmonic span of stages 1-4 are loaded
 * with plain global loads, all in flight at once.  The spans of stages 1-3
 * go to LDS; stage 4's wait in registers and take the same LDS once stages
 * 1-3 are summed.  A 32-harmonic search loads stage 5 in a third round.
 * Adding 256 to a fundamental half-bin adds an even 256 k / 2^s to the
 * rounded quotient, so one rounding per thread and fraction serves all 4
 * cells. */
template <int NSTAGES, int MODE>
__global__ __launch_bounds__(HS_TPB) void k_harmsum(agpu_harmsum_args a, int c_lo, int c_hi)
{
    __shared__ float s_norm[3 * 32];   /* norm^2 of blocks b0..b0+2 x fraction */
    constexpr int NWL = hs_lds_wl(NSTAGES);
    __shared__ float lds[(NWL > 0 ? NWL : 1) * 64];
    const int row = blockIdx.x >> 3;
    const int chunk = c_lo + 8 * (int) blockIdx.y + (int) (blockIdx.x & 7);
    if (chunk >= c_hi)
        return;
    const unsigned *rt = a.row_tab + (size_t) row * HS_RT;
    const long long *cb = a.chunk_base + (size_t) chunk * HS_CT;
    const int *clo = a.chunk_lo + (size_t) chunk * HS_CT;
    const int wi = (int) rt[0], zi = (int) rt[1];
    const int ncell = a.nblocks * a.corr_uselen;
    const int rh_c0 = ((int) (a.rh0 / HS_CHUNK) + chunk) * HS_CHUNK;
    const int cell0 = rh_c0 - (int) a.rh0;   /* negative in the first chunk */
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int cu = a.corr_uselen;
    const int b0 = cell0 > 0 ? cell0 / cu : 0;
    const int e1 = (b0 + 1) * cu, e2 = (b0 + 2) * cu;
    const int nfr = a.nfrac + 1;
    const float *prow = a.plane + cb[0] + rt[HS_RT_ROW];
    float fund[HS_CPT];
#pragma unroll
    for (int j = 0; j < HS_CPT; j++)
        fund[j] = prow[t + HS_TPB * j];
    constexpr int NREG = hs_regs_upto(NSTAGES < 5 ? NSTAGES : 5);
    float v[NREG > 0 ? NREG : 1];
    if (NSTAGES > 1) hs_load<1>(a, v + hs_regs_upto(1), cb, rt, wv, lane);
    if (NSTAGES > 2) hs_load<2>(a, v + hs_regs_upto(2), cb, rt, wv, lane);
    if (NSTAGES > 3) hs_load<3>(a, v + hs_regs_upto(3), cb, rt, wv, lane);
    if (NSTAGES > 4) hs_load<4>(a, v + hs_regs_upto(4), cb, rt, wv, lane);
    if (MODE != HS_INMEM && t < 3 * nfr) {
        const int bb = min(b0 + t / nfr, a.nblocks - 1);
        s_norm[(t / nfr) * 32 + t % nfr] = a.nsq[(size_t) bb * nfr + t % nfr];
    }
    if (NSTAGES > 1) hs_store<1>(lds, hs_stage_base(1), v + hs_regs_upto(1), wv, lane);
    if (NSTAGES > 2) hs_store<2>(lds, hs_stage_base(2), v + hs_regs_upto(2), wv, lane);
    if (NSTAGES > 3) hs_store<3>(lds, hs_stage_base(3), v + hs_regs_upto(3), wv, lane);
    /* cells outside [0, ncell) read valid plane memory (the chunk before the
     * first cell or the padding tile) and are never emitted */
    const int rh_first = rh_c0 + t;
    int nb[HS_CPT];      /* block offset (0..2) of the cell */
    float acc[HS_CPT];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < HS_CPT; j++) {
        const int c = cell0 + t + HS_TPB * j;
        nb[j] = (c >= e1) + (c >= e2);
    }
    /* HS_FRAC: each cell's start r + ii/2 in FP64 (src/accel_utils.c:1044) */
    double rf[HS_CPT];
#pragma unroll
    for (int j = 0; j < HS_CPT; j++) {
        rf[j] = 0.0;
        if (MODE == HS_FRAC) {
            const int c = cell0 + t + HS_TPB * j;
            const int b = min(b0 + nb[j], a.nblocks - 1);
            rf[j] = a.bstart[b] + (double) (c - b * cu) * 0.5;
        }
    }
#pragma unroll
    for (int j = 0; j < HS_CPT; j++) {
        const float nn = MODE == HS_INMEM ? a.nsq_hb[rh_first + HS_TPB * j]
                                          : s_norm[nb[j] * 32];
        acc[j] = fund[j] * nn;
    }
#define HS_EMIT(ST)                                                                    \
    {                                                                                  \
        const float cut_ = a.powcut[ST];                                               \
        const bool any_ = acc[0] > cut_ || acc[1] > cut_ || acc[2] > cut_ ||           \
                          acc[3] > cut_;                                               \
        if (__ballot(any_)) {                                                          \
            _Pragma("unroll") for (int j = 0; j < HS_CPT; j++) {                      \
                const int c = cell0 + t + HS_TPB * j;                                  \
                if (c >= 0 && c < ncell && acc[j] > cut_) {                            \
                    const int b = b0 + nb[j];                                          \
                    emit_hit(a, b, ST, wi, zi, c - b * cu, acc[j]);                    \
                }                                                                      \
            }                                                                          \
        }                                                                              \
    }
    HS_EMIT(0)
    /* per-cell norm row bases: cell j reads s_norm[nb[j]*32 + 1 + f] */
    const float *nrow0 = s_norm + nb[0] * 32;
    const float *nrow1 = s_norm + nb[1] * 32;
    const float *nrow2 = s_norm + nb[2] * 32;
    const float *nrow3 = s_norm + nb[3] * 32;
#define HS_STAGE(ST)                                                                   \
    hs_consume4<ST, MODE>(a, lds, hs_stage_base(ST), nrow0, nrow1, nrow2, nrow3, clo,  \
                          rh_first, rf, acc);                                         \
    HS_EMIT(ST)
    if (NSTAGES > 1) { HS_STAGE(1) }
    if (NSTAGES > 2) { HS_STAGE(2) }
    if (NSTAGES > 3) { HS_STAGE(3) }
    if (NSTAGES > 4) {
        /* stage 4's spans waited in registers; they take the LDS of
         * stages 1-3 once those are consumed */
        __syncthreads();
        hs_store<4>(lds, 0, v + hs_regs_upto(4), wv, lane);
        __syncthreads();
        hs_consume4<4, MODE>(a, lds, 0, nrow0, nrow1, nrow2, nrow3, clo, rh_first, rf, acc);
        HS_EMIT(4)
    }
    if (NSTAGES > 5) {
        float v5[hs_stage_regs(5)];
        hs_load<5>(a, v5, cb, rt, wv, lane);
        __syncthreads();   /* stages 1-4 are done with LDS */
        hs_store<5>(lds, 0, v5, wv, lane);
        __syncthreads();
        hs_consume4<5, MODE>(a, lds, 0, nrow0, nrow1, nrow2, nrow3, clo, rh_first, rf, acc);
        HS_EMIT(5)
    }
#undef HS_STAGE
#undef HS_EMIT
}

/* Sigma of every hit (src/accel_utils.c:1434-1437), one thread per hit:
 * FP64 Newton steps on log(erfc), ~1 us each on a host core, here all at
 * once behind the harmonic sum (~12 us for any count up to some thousands).
 * A fixed grid strides over the count that the sum left on the device. */
__global__ __launch_bounds__(64) void k_hit_sigmas(agpu_hitrec *hits, const unsigned *nhits,
                                                   unsigned cap, agpu_numindep ni)
{
    const unsigned n = min(*nhits, cap);
    for (unsigned i = blockIdx.x * 64 + threadIdx.x; i < n; i += gridDim.x * 64) {
        const agpu_hit h = hits[i].h;
        hits[i].sigma = (float) sigma_of_power(h.pow, 1 << h.stage, ni.n[h.stage]);
    }
}

/* ---- the harmonic sum over bounds ---- */

/* Largest norm^2 that the cells of each 256-half-bin chunk meet, per
 * fraction ([chunk][32], fundamental first), raised by 2^-18: the bounds'
 * multiply-adds round differently than the cells' products and sums (16
 * roundings of 2^-24 each at most).  A NaN norm is skipped (its cells cross
 * no threshold) unless all are NaN. */
template <int MODE>
__global__ void k_bound_norms(agpu_harmsum_args a, int c0, int nc, long long hb_end, float *nb)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int c = i >> 5, f = i & 31;
    if (c >= nc || f > a.nfrac)
        return;
    const int hb = (c0 + c) * HB_CHUNK;
    const int rh0 = (int) a.rh0, cu = a.corr_uselen;
    float m;
    if (MODE == HS_INMEM) {
        /* f = 2^(s-1) + (k-1)/2 for fraction k / 2^s; 0 is the fundamental */
        const int s = f ? 32 - __clz(f) : 0, k = f ? 2 * (f - (1 << (s - 1))) + 1 : 1;
        const int end = (int) hb_end - 1;
        const int lo = min(hs_round<HS_INMEM>(hb, k, s), end);
        const int hi = min(hs_round<HS_INMEM>(hb + HB_CHUNK - 1, k, s), end);
        /* a span shorter than a block meets at most two blocks on either
         * side of rh0, where the pre-population ends */
        m = fmaxf(a.nsq_hb[lo], a.nsq_hb[hi]);
        if (lo < rh0 && rh0 <= hi)
            m = fmaxf(m, fmaxf(a.nsq_hb[rh0 - 1], a.nsq_hb[rh0]));
    } else {
        const int nfr = a.nfrac + 1;
        const int b0 = min(max(hb - rh0, 0) / cu, a.nblocks - 1);
        const int b1 = min(max(hb + HB_CHUNK - 1 - rh0, 0) / cu, a.nblocks - 1);
        m = fmaxf(a.nsq[(size_t) b0 * nfr + f], a.nsq[(size_t) b1 * nfr + f]);
    }
    nb[(size_t) c * 32 + f] = m + m * 0x1p-18f;
}

/* Bounds at and past hb_end, which k_corr does not write: 0.  The chunk that
 * holds the last half-bin looks at them beside the bounds before hb_end, in
 * one maximum over a lane's 16 sums, so what an earlier user left in the
 * memory must not stand there (the bits of a negative sum exceed those of
 * every power and would hide the lane's other sums).  Once per plane:
 * nothing writes them later.  first: the first tile with such a slot, of its
 * own or of the next tile's first groups. */
__global__ __launch_bounds__(256) void k_clear_bounds(float *plane, long long tile_stride,
                                                      long long hb_end, long long first)
{
    const long long tile = first + blockIdx.y;
    unsigned short *b = (unsigned short *) (plane + tile * tile_stride +
                                            (long long) blockIdx.x * AGPU_ROWLEN + AGPU_TILE);
    for (int i = threadIdx.x; i < AGPU_TILE / AGPU_GROUP + AGPU_BHALO; i += 256)
        if (tile * AGPU_TILE + (long long) i * AGPU_GROUP >= hb_end)
            b[i] = 0;
}

/* Exact sums of 64 cells, lane l at fundamental half-bin hb + l, of every
 * z row z0 + i with bit i set in todo (not 0), straight from the raw plane:
 * the terms and their order are k_harmsum's.  The lanes of a fraction lie
 * in one tile or the next, so their offsets from the first lane's tile-row
 * fit 32 bits; offsets and norms serve all rows. */
template <int NSTAGES, int MODE>
__device__ __forceinline__ void hb_cells(const agpu_harmsum_args &a, long long tile_stride, int hb,
                                         int lane, int wi, int z0, unsigned long long todo)
{
#pragma clang fp contract(off)
    constexpr int NF = 1 << (NSTAGES - 1);
    const int rh = hb + lane, c = rh - (int) a.rh0;
    const bool in = c >= 0 && c < a.nblocks * a.corr_uselen;
    const int b = in ? c / a.corr_uselen : 0;
    const unsigned next = 4u * (unsigned) (tile_stride - AGPU_TILE);
    const char *base[NF];
    unsigned off[NF];
    float nn[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const int S = f ? 32 - __builtin_clz(f) : 0, k = f ? 2 * (f - (1 << S >> 1)) + 1 : 1;
        const int first = S ? hs_round<MODE>(hb, k, S) : hb;
        const int rs = S ? hs_round<MODE>(rh, k, S) : rh;
        const int t0 = first & ~(AGPU_TILE - 1);
        const unsigned x = (unsigned) (rs - t0);
        base[f] = (const char *) (a.plane + (t0 >> AGPU_TILE_LOG2) * tile_stride);
        off[f] = 4u * x + (x < AGPU_TILE ? 0u : next);
        nn[f] = MODE == HS_INMEM ? a.nsq_hb[rs] : a.nsq[(size_t) b * NF + f];
    }
    while (todo) {   /* two rows' loads in flight */
        int zi[2];
        zi[0] = z0 + (int) __ffsll(todo) - 1;
        todo &= todo - 1;
        const bool pair = todo != 0;
        zi[1] = pair ? z0 + (int) __ffsll(todo) - 1 : zi[0];
        todo &= todo - 1;   /* 0 stays 0 */
        float val[2][NF];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const unsigned *rt = a.row_tab + (size_t) (wi * a.numz + zi[h]) * HS_RT;
#pragma unroll
            for (int f = 0; f < NF; f++)
                val[h][f] = *(const float *) (base[f] +
                                              4 * (size_t) rt[f ? HS_RT_SUB + f - 1 : HS_RT_ROW] +
                                              off[f]);
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            float acc[NSTAGES];
            acc[0] = val[h][0] * nn[0];
            bool hit = acc[0] > a.powcut[0];
#pragma unroll
            for (int S = 1; S < NSTAGES; S++) {
                acc[S] = acc[S - 1];
#pragma unroll
                for (int f = 1 << (S - 1); f < (1 << S); f++)
                    acc[S] = acc[S] + val[h][f] * nn[f];
                hit |= acc[S] > a.powcut[S];
            }
            if (in && hit && (h == 0 || pair))
#pragma unroll
                for (int S = 0; S < NSTAGES; S++)
                    if (acc[S] > a.powcut[S])
                        emit_hit(a, b, S, wi, zi[h], c - b * a.corr_uselen, acc[S]);
        }
    }
}

/* ---- LDS tiles of the bounds ----
 * A workgroup looks through HB_CHUNK half-bins (64 groups) of up to HB_ROWS
 * consecutive z rows.  For fraction k / 2^s they meet 64 k / 2^s + 1 groups
 * (32 k / 2^s + 1 dwords of two, an odd stride) of at most
 * (HB_ROWS - 1) k / 2^s + 3 z rows: the map rounds k z / 2^s half away from
 * zero, so the ends move apart by less than two rows. */
__host__ __device__ constexpr int hb_dw(int k, int s) { return (32 * k >> s) + 1; }
__host__ __device__ constexpr int hb_nr(int k, int s)
{
    return s ? ((HB_ROWS - 1) * k >> s) + 3 : HB_ROWS;
}
/* lanes per row of a load: the power of two that holds the dwords */
__host__ __device__ constexpr int hb_lpr(int k, int s)
{
    int n = 1;
    while (n < (s ? hb_dw(k, s) : 32))
        n *= 2;
    return n;
}
__host__ __device__ constexpr int hb_loads(int k, int s)
{
    const int rpp = 256 / hb_lpr(k, s);
    return (hb_nr(k, s) + rpp - 1) / rpp;
}
/* dwords of the tiles of stages s0..s1 before fraction (k, s) */
__host__ __device__ constexpr int hb_base(int s0, int k, int s)
{
    int n = 0;
    for (int t = s0; t <= s; t++)
        for (int i = 1; i < (1 << t) + (t == 0); i += 2)
            if (t < s || i < k)
                n += hb_dw(i, t) * hb_nr(i, t);
    return n;
}
__host__ __device__ constexpr int hb_size(int s0, int s1) { return hb_base(s0, (1 << s1) + 1, s1); }
__host__ __device__ constexpr int hb_lds(int nstages)
{
    return hs_max(hb_size(0, nstages < 4 ? nstages - 1 : 3), nstages > 4 ? hb_size(4, 4) : 0);
}
__host__ __device__ constexpr int hb_nloads(int s0, int s1)
{
    int n = 0;
    for (int t = s0; t <= s1; t++)
        for (int i = 1; i < (1 << t) + (t == 0); i += 2)
            n += hb_loads(i, t);
    return n;
}
static_assert(hb_dw(15, 4) <= 32 && 2 * (AGPU_TILE / AGPU_GROUP + AGPU_BHALO) == 4 * AGPU_HALO &&
                  AGPU_BHALO >= 64 + 2,
              "a chunk's bounds lie in one tile-row and its replica");

/* The workgroup's loads of fraction k / 2^s into registers: thread t takes
 * dword t % lpr of row t / lpr (and 256 / lpr rows on). */
template <int K, int S>
__device__ __forceinline__ void hb_load(const agpu_harmsum_args &a, unsigned *v, int g0,
                                        long long tile_stride, const unsigned *rt0,
                                        const unsigned *rt1)
{
    constexpr int LPR = hb_lpr(K, S), RPP = 256 / LPR, F = S ? (1 << S >> 1) + (K - 1) / 2 : 0;
    const int J = g0 * K >> S;   /* exact: g0 is a multiple of 64 */
    const unsigned r0 = rt0[S ? HS_RT_SUB + F - 1 : HS_RT_ROW];
    const unsigned r1 = rt1[S ? HS_RT_SUB + F - 1 : HS_RT_ROW];
    const char *base = (const char *) (a.plane +
                                       (long long) (J >> (AGPU_TILE_LOG2 - AGPU_GROUP_LOG2)) *
                                           tile_stride + r0 + AGPU_TILE) +
                       2 * (J & (AGPU_TILE / AGPU_GROUP - 1));
    /* through a descriptor that ends with the last row: a load past it (or
     * of a dword past the row's) is out of range and returns 0 */
    const unsigned bytes = 4u * (r1 - r0 + hb_dw(K, S));
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void *) base, 0, (int) bytes, 0x00027000);
    const int dw = threadIdx.x % LPR, row = threadIdx.x / LPR;
    const unsigned off = S == 0 || dw < hb_dw(K, S)
                             ? 4u * (unsigned) (row * AGPU_ROWLEN + dw) : 0x80000000u;
#pragma unroll
    for (int u = 0; u < hb_loads(K, S); u++)
        v[u] = __builtin_amdgcn_raw_buffer_load_b32(rs, (int) (off + 4u * u * RPP * AGPU_ROWLEN),
                                                    0, 0);
}

template <int K, int S>
__device__ __forceinline__ void hb_store(unsigned *lds, const unsigned *v)
{
    constexpr int LPR = hb_lpr(K, S), RPP = 256 / LPR;
    const int dw = threadIdx.x % LPR, row = threadIdx.x / LPR;
#pragma unroll
    for (int u = 0; u < hb_loads(K, S); u++)
        if (row + u * RPP < hb_nr(K, S) && (S == 0 || dw < hb_dw(K, S)))
            lds[(row + u * RPP) * hb_dw(K, S) + dw] = v[u];
}

/* Adds fraction k / 2^s to the sums of this wave's 16 groups of this lane's
 * row.  p: the row's dwords from the wave's first group on (ODD: from the
 * group before it).  Which groups a sum meets is known at compile time. */
template <int K, int S, bool ODD>
__device__ __forceinline__ void hb_add(float *acc, const unsigned *p, float nn)
{
    constexpr int N = ((63 * K + (1 << S >> 1)) >> (S + AGPU_GROUP_LOG2)) + 1;   /* groups met */
    unsigned w[(N + 2) / 2], g[N];
#pragma unroll
    for (int i = 0; i < (N + ODD + 1) / 2; i++)
        w[i] = p[i];
#pragma unroll
    for (int j = 0; j < N; j++)   /* the upper group's low half only raises it */
        g[j] = (j + ODD) & 1 ? w[(j + ODD) / 2] : w[(j + ODD) / 2] << 16;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int j0 = (AGPU_GROUP * i * K) >> (S + AGPU_GROUP_LOG2);
        const int j1 = ((AGPU_GROUP * i + AGPU_GROUP - 1) * K + (1 << S >> 1)) >>
                       (S + AGPU_GROUP_LOG2);
        /* as integers: powers order like their bits, and an infinite or NaN
         * bound stays one */
        const unsigned m = j1 == j0 ? g[j0] : max(g[j0], g[j1]);
        acc[i] = S ? __builtin_fmaf(__uint_as_float(m), nn, acc[i]) : __uint_as_float(m) * nn;
    }
}

/* The sub-harmonic z row of row z (from the middle row) for fraction
 * k / 2^s, from the middle row: k z / 2^s rounded half away from zero, as
 * calc_required_z rounds it (src/accel_utils.c:65). */
__host__ __device__ __forceinline__ int hb_zmap(int z, int k, int s)
{
    const int m = z * k, h = 1 << s >> 1;
    return m < 0 ? -((h - m) >> s) : (h + m) >> s;
}

/* any of the 16 sums above the threshold, or NaN.  By their bits, which order
 * like the sums since none is negative (a NaN of either sign exceeds every
 * one): bounds are powers or NaN (k_corr), or 0 past the last half-bin
 * (k_clear_bounds), and norms are squares. */
__device__ __forceinline__ bool hb_over(const float *acc, float cut)
{
    unsigned m = __float_as_uint(acc[0]);
#pragma unroll
    for (int i = 1; i < 16; i++)
        m = max(m, __float_as_uint(acc[i]));
    return !(__uint_as_float(m) <= cut);
}

/* stage by stage, the fractions of a stage in order */
template <int K, int S>
__device__ __forceinline__ void hb_load_stage(const agpu_harmsum_args &a, unsigned *v, int g0,
                                              long long tile_stride, const unsigned *rt0,
                                              const unsigned *rt1)
{
    hb_load<K, S>(a, v, g0, tile_stride, rt0, rt1);
    if constexpr (K + 2 < (1 << S))
        hb_load_stage<K + 2, S>(a, v + hb_loads(K, S), g0, tile_stride, rt0, rt1);
}
template <int K, int S>
__device__ __forceinline__ void hb_store_stage(unsigned *lds, const unsigned *v)
{
    hb_store<K, S>(lds, v);
    if constexpr (K + 2 < (1 << S))
        hb_store_stage<K + 2, S>(lds + hb_dw(K, S) * hb_nr(K, S), v + hb_loads(K, S));
}
template <int K, int S, bool ODD>
__device__ __forceinline__ void hb_add_stage(float *acc, const unsigned *lds, const float *np,
                                             int z0, int z, int wv)
{
    constexpr int F = (1 << S >> 1) + (K - 1) / 2;
    const int zs = hb_zmap(z, K, S) - hb_zmap(z0, K, S);
    hb_add<K, S, ODD>(acc, lds + zs * hb_dw(K, S) + (wv * (16 * K >> S)) / 2, np[F]);
    if constexpr (K + 2 < (1 << S))
        hb_add_stage<K + 2, S, ODD>(acc, lds + hb_dw(K, S) * hb_nr(K, S), np, z0, z, wv);
}

/* The harmonic sum and threshold by bounds.  A workgroup takes 256
 * fundamental half-bins (64 groups of 4; a wave 16 groups) of up to 64
 * consecutive z rows (a lane one row).  Each lane sums, in place of the
 * powers, the largest power of the one or two groups that a group's cells
 * meet in every sub-harmonic (the 16-bit bounds that k_corr<true> wrote,
 * rounded up) times the largest norm: no sum of the group's cells exceeds
 * that at any stage.  Only where it exceeds the stage's threshold (or is
 * NaN) are the 64 cells around it summed exactly, from the raw plane.  Hits
 * are those of k_harmsum bit for bit: a cell that crosses is never skipped,
 * and every emitted sum is formed from the same terms in the same order.
 *
 * Lanes along z share sub-harmonic rows, groups along r share sub-harmonic
 * groups, so each bound is read once into LDS per workgroup ((k / H)^2 of
 * the fundamental's bytes per fraction), and which groups a sum meets is
 * the same for every row and chunk: the inner loop is LDS reads, maxima and
 * multiply-adds without any index arithmetic.
 *
 * 2^23 samples, zmax 200, 16 harmonics: 1.85 ms against k_harmsum's 7.4 (an
 * eighth of its 39 GB needed; 1.3 % of the 64-cell runs summed exactly);
 * 2^20, 201 x 31 templates, 8 harmonics: 2.5 ms against 14.4.  Bound: vector
 * and scalar issue (1.1 ms of it) and the latency of the two load-store-sum
 * phases at four waves per SIMD.  Chunks on other XCDs share the cache lines
 * of a sub-harmonic's bounds (12.3 GB fetched for 4.9); runs of 32 chunks per
 * XCD halve that and leave whole searches between 2 % slower and 1 % faster. */
template <int NSTAGES, int MODE>
__global__ __launch_bounds__(256) void k_harmbound(agpu_harmsum_args a, const float *nb,
                                                   int chunks, int zblocks, int zrows)
{
    __shared__ unsigned lds[hb_lds(NSTAGES)];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    /* all rows of a chunk run on one XCD (block ids are dealt round-robin to
     * the 8), so that row blocks which share sub-harmonic rows find them in
     * its L2 */
    const int rb = zblocks * a.numw;
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
    const int c = (local / rb) * 8 + xcd;        /* chunk, from the one of the first cell */
    const int wi = (local % rb) / zblocks, z0 = (local % rb) % zblocks * zrows;
    const int z1 = min(a.numz, z0 + zrows);
    if (c >= chunks)
        return;
    const int hb = ((int) a.rh0 / HB_CHUNK + c) * HB_CHUNK, g0 = hb / AGPU_GROUP;
    const long long tile_stride = (long long) a.numz * a.numw * AGPU_ROWLEN;
    const float *np = nb + (size_t) c * 32;
    /* the first and the last row's tables: where a fraction's rows begin and end */
    const unsigned *rt0 = a.row_tab + (size_t) (wi * a.numz + z0) * HS_RT;
    const unsigned *rt1 = a.row_tab + (size_t) (wi * a.numz + z1 - 1) * HS_RT;
    constexpr int LAST = NSTAGES < 4 ? NSTAGES - 1 : 3;
    {
        unsigned v[hb_nloads(0, LAST)];
        hb_load<1, 0>(a, v, g0, tile_stride, rt0, rt1);
        if constexpr (NSTAGES > 1)
            hb_load_stage<1, 1>(a, v + hb_nloads(0, 0), g0, tile_stride, rt0, rt1);
        if constexpr (NSTAGES > 2)
            hb_load_stage<1, 2>(a, v + hb_nloads(0, 1), g0, tile_stride, rt0, rt1);
        if constexpr (NSTAGES > 3)
            hb_load_stage<1, 3>(a, v + hb_nloads(0, 2), g0, tile_stride, rt0, rt1);
        hb_store<1, 0>(lds, v);
        if constexpr (NSTAGES > 1)
            hb_store_stage<1, 1>(lds + hb_base(0, 1, 1), v + hb_nloads(0, 0));
        if constexpr (NSTAGES > 2)
            hb_store_stage<1, 2>(lds + hb_base(0, 1, 2), v + hb_nloads(0, 1));
        if constexpr (NSTAGES > 3)
            hb_store_stage<1, 3>(lds + hb_base(0, 1, 3), v + hb_nloads(0, 2));
    }
    unsigned v4[NSTAGES > 4 ? hb_nloads(4, 4) : 1];
    if constexpr (NSTAGES > 4)   /* in flight while the stages before are summed */
        hb_load_stage<1, 4>(a, v4, g0, tile_stride, rt0, rt1);
    __syncthreads();
    const int z = min(z0 + lane, z1 - 1), mid = (a.numz - 1) / 2;
    float acc[16];
    hb_add<1, 0, false>(acc, lds + (z - z0) * hb_dw(1, 0) + wv * 8, np[0]);
    bool over = hb_over(acc, a.powcut[0]);
    if constexpr (NSTAGES > 1) {
        hb_add_stage<1, 1, false>(acc, lds + hb_base(0, 1, 1), np, z0 - mid, z - mid, wv);
        over |= hb_over(acc, a.powcut[1]);
    }
    if constexpr (NSTAGES > 2) {
        hb_add_stage<1, 2, false>(acc, lds + hb_base(0, 1, 2), np, z0 - mid, z - mid, wv);
        over |= hb_over(acc, a.powcut[2]);
    }
    if constexpr (NSTAGES > 3) {
        hb_add_stage<1, 3, false>(acc, lds + hb_base(0, 1, 3), np, z0 - mid, z - mid, wv);
        over |= hb_over(acc, a.powcut[3]);
    }
    if constexpr (NSTAGES > 4) {
        __syncthreads();
        hb_store_stage<1, 4>(lds, v4);
        __syncthreads();
        /* k groups per wave: an odd wave starts on an odd group */
        if (wv & 1)
            hb_add_stage<1, 4, true>(acc, lds, np, z0 - mid, z - mid, wv);
        else
            hb_add_stage<1, 4, false>(acc, lds, np, z0 - mid, z - mid, wv);
        over |= hb_over(acc, a.powcut[4]);
    }
    const unsigned long long todo = __ballot(over && z0 + lane < z1);
    if (todo)
        hb_cells<NSTAGES, MODE>(a, tile_stride, hb + 64 * wv, lane, wi, z0, todo);
}

/* z rows per workgroup: numz in equal blocks of at most HB_ROWS */
static int hb_zrows(int numz)
{
    const int n = (numz + HB_ROWS - 1) / HB_ROWS;
    return (numz + n - 1) / n;
}

/* First half-bin of a chunk's span for fraction k / 2^s.  HS_FRAC starts
 * one half-bin below the grid rule's: its lookups lie within
 * (hb - 1/2, hb + 2) k / H, so the span [lo, lo + CHUNK k / H + 4) holds
 * them, inside the hs_frac_wl slots (whose 64-float rounding leaves at
 * least 31 spare half-bins). */
static int hs_span_lo_host(int mode, int rh_off, int rh_c0, int k, int s)
{
    if (mode == HS_STD)
        return hs_round<HS_STD>(rh_c0 + rh_off, k, s);
    if (mode == HS_INMEM)
        return hs_round<HS_INMEM>(rh_c0, k, s);
    const int lo = hs_round<HS_STD>(rh_c0, k, s) - 1;
    return lo > 0 ? lo : 0;
}

/* ------------------------------------------------------------------ */
/* C ABI                                                                */
/* ------------------------------------------------------------------ */
extern "C" {

const char *agpu_last_error(void) { return g_err; }

int agpu_init(int device)
{
    int n = 0;
    AGPU_CHECK(hipGetDeviceCount(&n));
    if (device < 0 || device >= n)
        return fail("agpu_init: no such HIP device");
    AGPU_CHECK(hipSetDevice(device));
    return 0;
}

int agpu_device_name(char *buf, int len)
{
    hipDeviceProp_t p;
    int dev = 0;
    AGPU_CHECK(hipGetDevice(&dev));
    AGPU_CHECK(hipGetDeviceProperties(&p, dev));
    snprintf(buf, len, "%s (%s, %d CUs)", p.name, p.gcnArchName, p.multiProcessorCount);
    return 0;
}

/* ------------------------------------------------------------------ */
/* Device memory arena.  Freed device memory is not immediately cheap to  */
/* hand out again (the next large allocation can stall for seconds), and  */
/* every hipFree waits for the whole device.  A long-running caller (the  */
/* request loop) therefore reserves one block once and every allocation   */
/* is carved from it: best fit, free neighbours coalesced, 64 KiB units.  */
/* Without an arena, allocations go straight to hipMalloc / hipFree.     */
/* ------------------------------------------------------------------ */
#define ARENA_UNIT ((size_t) 64 << 10)

struct arena_seg {
    size_t off, len;
};

static pthread_mutex_t g_arena_mu = PTHREAD_MUTEX_INITIALIZER;
static char *g_arena = NULL;
static size_t g_arena_len = 0, g_arena_used = 0;
static arena_seg *g_free = NULL, *g_used = NULL;
static int g_nfree = 0, g_nused = 0, g_capfree = 0, g_capused = 0;

static void seg_push(arena_seg **v, int *n, int *cap, arena_seg s)
{
    if (*n == *cap) {
        *cap = *cap ? 2 * *cap : 64;
        *v = (arena_seg *) realloc(*v, sizeof(arena_seg) * *cap);
    }
    (*v)[(*n)++] = s;
}

int agpu_arena_init(size_t bytes)
{
    pthread_mutex_lock(&g_arena_mu);
    int rc = 0;
    if (g_arena) {
        rc = (g_arena_len >= bytes) ? 0 : -2;
        if (rc)
            snprintf(g_err, sizeof(g_err), "agpu_arena_init: an arena of %zu bytes exists",
                     g_arena_len);
    } else {
        bytes = (bytes + ARENA_UNIT - 1) / ARENA_UNIT * ARENA_UNIT;
        hipError_t e = hipMalloc((void **) &g_arena, bytes);
        if (e != hipSuccess) {
            snprintf(g_err, sizeof(g_err), "agpu_arena_init: hipMalloc(%zu): %s", bytes,
                     hipGetErrorString(e));
            g_arena = NULL;
            rc = -1;
        } else {
            g_arena_len = bytes;
            g_arena_used = 0;
            g_nfree = g_nused = 0;
            seg_push(&g_free, &g_nfree, &g_capfree, arena_seg{0, bytes});
        }
    }
    pthread_mutex_unlock(&g_arena_mu);
    return rc;
}

int agpu_arena_release(void)
{
    pthread_mutex_lock(&g_arena_mu);
    int rc = 0;
    if (g_arena && g_nused) {
        snprintf(g_err, sizeof(g_err), "agpu_arena_release: %d blocks still allocated", g_nused);
        rc = -2;
    } else if (g_arena) {
        (void) hipFree(g_arena);
        g_arena = NULL;
        g_arena_len = g_arena_used = 0;
        g_nfree = 0;
    }
    pthread_mutex_unlock(&g_arena_mu);
    return rc;
}

size_t agpu_arena_used(void)
{
    pthread_mutex_lock(&g_arena_mu);
    size_t u = g_arena_used;
    pthread_mutex_unlock(&g_arena_mu);
    return u;
}

int agpu_malloc(void **p, size_t bytes)
{
    pthread_mutex_lock(&g_arena_mu);
    if (!g_arena) {
        pthread_mutex_unlock(&g_arena_mu);
        AGPU_CHECK(hipMalloc(p, bytes));
        return 0;
    }
    const size_t len = (bytes + ARENA_UNIT - 1) / ARENA_UNIT * ARENA_UNIT;
    int best = -1;
    for (int i = 0; i < g_nfree; i++)
        if (g_free[i].len >= len && (best < 0 || g_free[i].len < g_free[best].len))
            best = i;
    if (best < 0) {
        pthread_mutex_unlock(&g_arena_mu);
        snprintf(g_err, sizeof(g_err), "device arena: no free block of %zu bytes", len);
        return -1;
    }
    arena_seg blk = {g_free[best].off, len};
    g_free[best].off += len;
    g_free[best].len -= len;
    if (g_free[best].len == 0)
        g_free[best] = g_free[--g_nfree];
    seg_push(&g_used, &g_nused, &g_capused, blk);
    g_arena_used += len;
    *p = g_arena + blk.off;
    pthread_mutex_unlock(&g_arena_mu);
    return 0;
}

int agpu_free(void *p)
{
    if (!p)
        return 0;
    pthread_mutex_lock(&g_arena_mu);
    if (g_arena && (char *) p >= g_arena && (char *) p < g_arena + g_arena_len) {
        const size_t off = (size_t) ((char *) p - g_arena);
        int u = -1;
        for (int i = 0; i < g_nused; i++)
            if (g_used[i].off == off) {
                u = i;
                break;
            }
        if (u < 0) {
            pthread_mutex_unlock(&g_arena_mu);
            return fail("device arena: free of an unknown block");
        }
        arena_seg blk = g_used[u];
        g_used[u] = g_used[--g_nused];
        g_arena_used -= blk.len;
        /* coalesce with the free blocks just before and after */
        for (int i = 0; i < g_nfree;) {
            if (g_free[i].off + g_free[i].len == blk.off) {
                blk.off = g_free[i].off;
                blk.len += g_free[i].len;
                g_free[i] = g_free[--g_nfree];
            } else if (blk.off + blk.len == g_free[i].off) {
                blk.len += g_free[i].len;
                g_free[i] = g_free[--g_nfree];
            } else {
                i++;
            }
        }
        seg_push(&g_free, &g_nfree, &g_capfree, blk);
        pthread_mutex_unlock(&g_arena_mu);
        return 0;
    }
    pthread_mutex_unlock(&g_arena_mu);
    AGPU_CHECK(hipFree(p));
    return 0;
}

int agpu_h2d(void *dst, const void *src, size_t bytes, void *stream)
{
    AGPU_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, (hipStream_t) stream));
    AGPU_CHECK(hipStreamSynchronize((hipStream_t) stream));
    return 0;
}

int agpu_d2h(void *dst, const void *src, size_t bytes, void *stream)
{
    AGPU_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, (hipStream_t) stream));
    AGPU_CHECK(hipStreamSynchronize((hipStream_t) stream));
    return 0;
}

int agpu_memset(void *p, int v, size_t bytes, void *stream)
{
    AGPU_CHECK(hipMemsetAsync(p, v, bytes, (hipStream_t) stream));
    return 0;
}

int agpu_stream_create(void **s)
{
    hipStream_t st;
    AGPU_CHECK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    *s = (void *) st;
    return 0;
}

int agpu_stream_wait_event(void *s, void *e)
{
    AGPU_CHECK(hipStreamWaitEvent((hipStream_t) s, (hipEvent_t) e, 0));
    return 0;
}

int agpu_stream_destroy(void *s)
{
    AGPU_CHECK(hipStreamDestroy((hipStream_t) s));
    return 0;
}

int agpu_stream_sync(void *s)
{
    AGPU_CHECK(hipStreamSynchronize((hipStream_t) s));
    return 0;
}

int agpu_event_create(void **e)
{
    hipEvent_t ev;
    AGPU_CHECK(hipEventCreate(&ev));
    *e = (void *) ev;
    return 0;
}

int agpu_event_destroy(void *e)
{
    AGPU_CHECK(hipEventDestroy((hipEvent_t) e));
    return 0;
}

int agpu_event_sync(void *e)
{
    AGPU_CHECK(hipEventSynchronize((hipEvent_t) e));
    return 0;
}

int agpu_event_record(void *e, void *stream)
{
    AGPU_CHECK(hipEventRecord((hipEvent_t) e, (hipStream_t) stream));
    return 0;
}

int agpu_event_elapsed(float *ms, void *start, void *stop)
{
    AGPU_CHECK(hipEventSynchronize((hipEvent_t) stop));
    AGPU_CHECK(hipEventElapsedTime(ms, (hipEvent_t) start, (hipEvent_t) stop));
    return 0;
}

/* Records a HIP failure in g_err and jumps to the function's cleanup. */
#define AGPU_TRY(call)                                                            \
    do {                                                                          \
        hipError_t e_ = (call);                                                   \
        if (e_ != hipSuccess) {                                                   \
            snprintf(g_err, sizeof(g_err), "%s:%d %s: %s", __FILE__, __LINE__,    \
                     #call, hipGetErrorString(e_));                               \
            goto cleanup;                                                         \
        }                                                                         \
    } while (0)

/* The taps of every template rounded to FP32, as the reference stores
 * gen_z_response / gen_w_response (src/responses.c:159-418): row t at
 * R + t*stride, zero past its numkern taps. */
__global__ void k_resp_round(const double2 *resp, const int *nks, int nkmax, int stride,
                             float2 *R)
{
    const int t = blockIdx.y;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= stride)
        return;
    float2 v = make_float2(0.0f, 0.0f);
    if (k < nks[t] && k < nkmax) {
        const double2 d = resp[(size_t) t * nkmax + k];
        v = make_float2((float) d.x, (float) d.y);
    }
    R[(size_t) t * stride + k] = v;
}

/* The response stage shared by the template bank (d_T, length L) and the
 * FP32 tap table (d_R, row stride Rstride); either may be NULL. */
static int gen_responses(const int *zs, const int *ws, const int *numkern, int nt, int L,
                         void *d_T, int Rstride, void *d_R, void *stream)
{
    hipStream_t st = (hipStream_t) stream;
    int rc = -1;
    int nkmax = 0, nw = 0, nptsmax = 0;
    /* scratch comes from agpu_malloc: inside a request loop's arena no
     * hipMalloc / hipFree (and no device-wide wait) happens here */
    int *d_z = NULL, *d_w = NULL, *d_nk = NULL, *d_np = NULL, *d_tl = NULL;
    double2 *d_resp = NULL;
    int *npts = (int *) malloc(sizeof(int) * nt);
    int *tlist = (int *) malloc(sizeof(int) * nt);
    if (!npts || !tlist) {
        snprintf(g_err, sizeof(g_err), "agpu_gen_templates: out of host memory");
        goto cleanup;
    }
    for (int t = 0; t < nt; t++) {
        if (numkern[t] <= 0 || numkern[t] % 4 || (d_T && numkern[t] > L) ||
            (d_R && numkern[t] > Rstride)) {
            snprintf(g_err, sizeof(g_err),
                     "agpu_gen_templates: kernel width must be a positive multiple of 4 <= L");
            goto cleanup;
        }
        if (numkern[t] > nkmax)
            nkmax = numkern[t];
        npts[t] = 0;
        if (abs(ws[t]) > 0) {
            /* src/responses.c:381-382: next2(6 hw + 200 + numkern/2) */
            long long want = 6LL * (numkern[t] / 4) + 200 + numkern[t] / 2, p2 = 1;
            while (p2 < want)
                p2 <<= 1;
            npts[t] = (int) p2;
            if (p2 > nptsmax)
                nptsmax = (int) p2;
            tlist[nw++] = t;
        }
    }
    if (nptsmax * (long long) sizeof(float) > 60 * 1024) {
        snprintf(g_err, sizeof(g_err), "agpu_gen_templates: jerk chirp longer than 15360 samples");
        goto cleanup;
    }
    if (agpu_malloc((void **) &d_z, sizeof(int) * nt) ||
        agpu_malloc((void **) &d_w, sizeof(int) * nt) ||
        agpu_malloc((void **) &d_nk, sizeof(int) * nt) ||
        agpu_malloc((void **) &d_np, sizeof(int) * nt) ||
        agpu_malloc((void **) &d_tl, sizeof(int) * (nw > 0 ? nw : 1)) ||
        agpu_malloc((void **) &d_resp, sizeof(double2) * (size_t) nt * nkmax))
        goto cleanup;
    AGPU_TRY(hipMemcpyAsync(d_z, zs, sizeof(int) * nt, hipMemcpyHostToDevice, st));
    AGPU_TRY(hipMemcpyAsync(d_w, ws, sizeof(int) * nt, hipMemcpyHostToDevice, st));
    AGPU_TRY(hipMemcpyAsync(d_nk, numkern, sizeof(int) * nt, hipMemcpyHostToDevice, st));
    AGPU_TRY(hipMemcpyAsync(d_np, npts, sizeof(int) * nt, hipMemcpyHostToDevice, st));
    if (nw)
        AGPU_TRY(hipMemcpyAsync(d_tl, tlist, sizeof(int) * nw, hipMemcpyHostToDevice, st));
    {
        /* z responses for every template; jerk templates then overwrite theirs */
        dim3 g1((nkmax + 255) / 256, nt);
        hipLaunchKernelGGL(k_resp_z, g1, dim3(256), 0, st, d_z, d_nk, nkmax, d_resp);
        AGPU_TRY(hipGetLastError());
        if (nw) {
            hipLaunchKernelGGL(k_resp_w, dim3(nw), dim3(256), sizeof(float) * nptsmax, st, d_z,
                               d_w, d_nk, d_np, d_tl, nkmax, d_resp);
            AGPU_TRY(hipGetLastError());
        }
        if (d_T) {
            dim3 g2(CORR_N / 2 / 256, nt);
            hipLaunchKernelGGL(k_template_dft, g2, dim3(256), 0, st, d_resp, d_nk, nkmax,
                               (float2 *) d_T);
            AGPU_TRY(hipGetLastError());
        }
        if (d_R) {
            dim3 g3((Rstride + 255) / 256, nt);
            hipLaunchKernelGGL(k_resp_round, g3, dim3(256), 0, st, d_resp, d_nk, nkmax, Rstride,
                               (float2 *) d_R);
            AGPU_TRY(hipGetLastError());
        }
    }
    rc = 0;
cleanup:
    /* the scratch may be returned only once the kernels that read it ended */
    if (hipStreamSynchronize(st) != hipSuccess && rc == 0) {
        snprintf(g_err, sizeof(g_err), "agpu_gen_templates: stream synchronisation failed");
        rc = -1;
    }
    agpu_free(d_z);
    agpu_free(d_w);
    agpu_free(d_nk);
    agpu_free(d_np);
    agpu_free(d_tl);
    agpu_free(d_resp);
    free(npts);
    free(tlist);
    return rc;
}

int agpu_gen_templates(const int *zs, const int *ws, const int *numkern, int nt, int L,
                       void *d_T, void *stream)
{
    if (nt <= 0 || L != CORR_N || nt > 65535 || !d_T)
        return fail("agpu_gen_templates: bad template count, or a length other than 4096");
    return gen_responses(zs, ws, numkern, nt, L, d_T, 0, NULL, stream);
}

int agpu_gen_response_taps(const int *zs, const int *ws, const int *numkern, int nt,
                           int stride, void *d_R, void *stream)
{
    if (nt <= 0 || stride <= 0 || nt > 65535 || !d_R)
        return fail("agpu_gen_response_taps: bad template count or stride");
    return gen_responses(zs, ws, numkern, nt, 0, NULL, stride, d_R, stream);
}

int agpu_block_norms(const void *d_spec, long long numbins, long long lobin_file,
                     const agpu_window *d_win, int nwin, int maxn, double *d_norm,
                     float *d_nsq, void *stream)
{
    if (nwin <= 0)
        return 0;
    if (maxn <= 0 || maxn > NORM_MAXN)
        return fail("agpu_block_norms: window longer than the LDS selection buffer");
    if (maxn <= NW_KPL * 64) {
        hipLaunchKernelGGL(k_block_norms_wave, dim3((unsigned) ((nwin + 3) / 4)), dim3(256), 0,
                           (hipStream_t) stream, (const float2 *) d_spec, numbins, lobin_file,
                           d_win, nwin, d_norm, d_nsq);
        AGPU_CHECK(hipGetLastError());
        return 0;
    }
    hipLaunchKernelGGL(k_block_norms, dim3(nwin), dim3(256), sizeof(unsigned) * maxn,
                       (hipStream_t) stream, (const float2 *) d_spec, numbins, lobin_file,
                       d_win, d_norm, d_nsq);
    AGPU_CHECK(hipGetLastError());
    return 0;
}

int agpu_block_norm1(const void *d_spec, long long numbins, long long lobin_file,
                     long long lobin, int numdata, double *d_norm, float *d_nsq, void *stream)
{
    if (numdata <= 0 || numdata > NORM_MAXN)
        return fail("agpu_block_norm1: window longer than the LDS selection buffer");
    hipLaunchKernelGGL(k_block_norm1, dim3(1), dim3(256), sizeof(unsigned) * numdata,
                       (hipStream_t) stream, (const float2 *) d_spec, numbins, lobin_file,
                       lobin, numdata, d_norm, d_nsq);
    AGPU_CHECK(hipGetLastError());
    return 0;
}

int agpu_correlate(const void *d_spec, long long numbins, long long lobin_file,
                   const void *d_T, int nt, int L, int hw, int uselen, long long hb_end,
                   float *d_plane, long long ntiles, int groups, long long seg_lo,
                   long long seg_hi, int bounds, void *stream)
{
    if (L != CORR_N)
        return fail("agpu_correlate: only L = 4096 is built");
    if (uselen <= 0 || uselen % 2 || uselen > L - 4 * hw + 1 || hb_end % 2)
        return fail("agpu_correlate: uselen must be even and <= L - 4*hw + 1");
    if (groups <= 0 || groups % 8)
        return fail("agpu_correlate: groups must be a positive multiple of 8");
    if (hb_end > ntiles * AGPU_TILE)
        return fail("agpu_correlate: plane tiles do not cover the half-bin range");
    long long nseg = (hb_end + uselen - 1) / uselen;
    if (seg_hi < 0 || seg_hi > nseg)
        seg_hi = nseg;
    if (seg_lo < 0 || seg_lo > seg_hi)
        return fail("agpu_correlate: bad segment range");
    if (seg_lo == seg_hi)
        return 0;
    int tpg = (nt + groups - 1) / groups;
    long long nblk = (seg_hi - seg_lo) * groups;
    if (nblk >= (1LL << 24))   /* a dispatch counts work-items in 32 bits */
        return fail("agpu_correlate: grid too large");
    if (bounds && (uselen % AGPU_GROUP || hw % 2))
        return fail("agpu_correlate: bounds need segments of whole groups");
    if (bounds)
        hipLaunchKernelGGL(k_corr<true>, dim3((unsigned) nblk), dim3(256), 0, (hipStream_t) stream,
                           (const float2 *) d_spec, numbins, lobin_file, (const float2 *) d_T, nt,
                           hw, uselen, hb_end, d_plane, groups, tpg, seg_lo, seg_hi - seg_lo);
    else
        hipLaunchKernelGGL(k_corr<false>, dim3((unsigned) nblk), dim3(256), 0,
                           (hipStream_t) stream, (const float2 *) d_spec, numbins, lobin_file,
                           (const float2 *) d_T, nt, hw, uselen, hb_end, d_plane, groups, tpg,
                           seg_lo, seg_hi - seg_lo);
    AGPU_CHECK(hipGetLastError());
    return 0;
}

long long agpu_harmsum_nchunks(const agpu_harmsum_args *a)
{
    const long long ncell = (long long) a->nblocks * a->corr_uselen;
    if (ncell <= 0)
        return 0;
    return (a->rh0 + ncell - 1) / HS_CHUNK - a->rh0 / HS_CHUNK + 1;
}

long long agpu_harmsum_chunk_hb(const agpu_harmsum_args *a, long long c)
{
    return (a->rh0 / HS_CHUNK + c) * HS_CHUNK;
}

int agpu_harmsum(const agpu_harmsum_args *a, long long c_lo, long long c_hi, void *stream)
{
    long long ncell = (long long) a->nblocks * a->corr_uselen;
    if (ncell <= 0)
        return 0;
    if (a->nstages < 1 || a->nstages > AGPU_MAX_STAGES)
        return fail("agpu_harmsum: 1..6 stages");
    if (a->nfrac + 1 > 32)
        return fail("agpu_harmsum: at most 31 sub-harmonic fractions");
    if (a->corr_uselen < HS_CHUNK / 2)
        return fail("agpu_harmsum: corr_uselen below 512 half-bins");
    if (a->inmem && !a->nsq_hb)
        return fail("agpu_harmsum: in-memory path needs the per-half-bin norm table");
    if (a->rh_off < 0 || a->rh_off > 1 || (a->inmem && (a->rh_off || a->bstart)))
        return fail("agpu_harmsum: sub-harmonic offset is 0 or 1 half-bin, standard path only");
    const long long rh_end = a->rh0 + ncell;
    if (a->ntiles < ((rh_end - 1) >> AGPU_TILE_LOG2) + 2 || a->ntiles * AGPU_TILE > 0x7fffffffLL)
        return fail("agpu_harmsum: plane tiles must pad the half-bin range by one tile "
                    "and stay below 2^31 half-bins");
    long long nchunks = (rh_end - 1) / HS_CHUNK - a->rh0 / HS_CHUNK + 1;
    if ((rh_end + HS_CHUNK) * (long long) ((1 << (a->nstages - 1)) - 1) > 0x7fffffffLL)
        return fail("agpu_harmsum: spectrum too long for 32-bit sub-harmonic indices "
                    "(half-bins x highest harmonic must stay below 2^31)");
    if (c_hi < 0 || c_hi > nchunks)
        c_hi = nchunks;
    if (c_lo < 0 || c_lo > c_hi)
        return fail("agpu_harmsum: bad chunk range");
    if (c_lo == c_hi)
        return 0;
    const long long rows = (long long) a->numz * a->numw;
    if (!a->row_tab || !a->chunk_base || !a->chunk_lo)
        return fail("agpu_harmsum: address tables missing");
    /* grid (8 rows' slots, groups of 8 chunks); each dimension stays far
     * below the dispatch packet's 32-bit work-item counts */
    if (8 * rows * HS_TPB > 0xffffffffLL || (c_hi - c_lo + 7) / 8 > 0xffffLL)
        return fail("agpu_harmsum: grid too large");
    dim3 grid((unsigned) (8 * rows), (unsigned) ((c_hi - c_lo + 7) / 8));
    hipStream_t st = (hipStream_t) stream;
    const int cl = (int) c_lo, ch = (int) c_hi;
#define HS_CASE(NS)                                                                         \
    case NS:                                                                                \
        if (a->inmem)                                                                       \
            hipLaunchKernelGGL((k_harmsum<NS, HS_INMEM>), grid, dim3(HS_TPB), 0, st, *a, cl,  \
                               ch);                                                         \
        else if (a->bstart)                                                                 \
            hipLaunchKernelGGL((k_harmsum<NS, HS_FRAC>), grid, dim3(HS_TPB), 0, st, *a, cl,   \
                               ch);                                                         \
        else                                                                                \
            hipLaunchKernelGGL((k_harmsum<NS, HS_STD>), grid, dim3(HS_TPB), 0, st, *a, cl,    \
                               ch);                                                         \
        break;
    switch (a->nstages) {
        HS_CASE(1)
        HS_CASE(2)
        HS_CASE(3)
        HS_CASE(4)
        HS_CASE(5)
        HS_CASE(6)
    }
#undef HS_CASE
    AGPU_CHECK(hipGetLastError());
    return 0;
}

/* Bounds pay
 *  - while few cells pass them: on whitened noise the bound of a sum of H
 *    powers is 2.13 H on average (the largest of 4 half-bins, or of 4 and 4)
 *    with a spread of 1.3 sqrt(H); with a threshold 2.3 spreads up a tenth
 *    of the 64-cell runs are summed exactly.  16 harmonics, 2^18 samples,
 *    zmax 100 (3.0 sqrt(H) up): 88 us against k_harmsum's 118; 2^19, zmax
 *    100 (3.3): 123 against 232; 2^21, zmax 100 (3.8): 345 against 1133.  The
 *    line is above the first: a spectrum's lines cross there before noise does
 *    (one every 32 bins, 2^23 samples, zmax 200: 5.3 ms against 4.3);
 *  - with rows for the lanes and workgroups for the device: 8 harmonics,
 *    2^21 samples, 5 rows 54 us against 37, 11 rows 56 against 62 (whole
 *    search 175 either way), 21 rows 59 against 105; 21 rows of 2^18
 *    half-bins 37 against 23, of 2^19 37 against 35, 51 rows of 2^18 43
 *    against 40: near 2^23 cells the two are alike. */
int agpu_harmbound_pays(int nstages, const float *powcut, int corr_uselen, int numz, int numw,
                        long long numhb, int nfrac, const int *zmap)
{
    if (nstages < 1 || nstages > 5 || corr_uselen < HS_CHUNK / 2 || numz < HB_MINROWS ||
        (long long) numz * numw * numhb < HB_MINCELLS)
        return 0;
    for (int s = 0; s < nstages; s++) {
        const double H = 1 << s;
        if (!(powcut[s] >= 2.13 * H + 3.1 * sqrt(H)))
            return 0;
    }
    /* the LDS tiles hold every row block's sub-harmonic rows */
    const int zrows = hb_zrows(numz);
    for (int f = 1; f <= nfrac; f++) {
        const int s = 32 - __builtin_clz(f), k = 2 * (f - (1 << (s - 1))) + 1;
        for (int z0 = 0; z0 < numz; z0 += zrows) {
            const int z1 = z0 + zrows < numz ? z0 + zrows : numz;
            const int *m = zmap + (size_t) (f - 1) * numz;
            for (int z = z0; z < z1; z++)
                if (m[z] != hb_zmap(z - (numz - 1) / 2, k, s) + (numz - 1) / 2)
                    return 0;
            if (m[z1 - 1] - m[z0] + 1 > hb_nr(k, s))
                return 0;
        }
    }
    return 1;
}

long long agpu_harmbound_chunks(const agpu_harmsum_args *a)
{
    const long long ncell = (long long) a->nblocks * a->corr_uselen;
    return ncell > 0 ? (a->rh0 + ncell - 1) / HB_CHUNK - a->rh0 / HB_CHUNK + 1 : 0;
}

int agpu_clear_bounds(float *d_plane, int nrows, long long ntiles, long long hb_end, void *stream)
{
    const long long own = hb_end >> AGPU_TILE_LOG2, first = own > 0 ? own - 1 : 0;
    if (!d_plane || nrows < 1 || hb_end < 0 || first >= ntiles || ntiles - first > 65535)
        return fail("agpu_clear_bounds: bad plane");
    hipLaunchKernelGGL(k_clear_bounds, dim3((unsigned) nrows, (unsigned) (ntiles - first)),
                       dim3(256), 0, (hipStream_t) stream, d_plane,
                       (long long) nrows * AGPU_ROWLEN, hb_end, first);
    AGPU_CHECK(hipGetLastError());
    return 0;
}

int agpu_bound_norms(const agpu_harmsum_args *a, long long hb_end, float *d_nb, void *stream)
{
    const long long nc = agpu_harmbound_chunks(a);
    if (nc <= 0)
        return 0;
    const int c0 = (int) (a->rh0 / HB_CHUNK);
    const dim3 grid((unsigned) ((nc * 32 + 255) / 256));
    if (a->inmem)
        hipLaunchKernelGGL(k_bound_norms<HS_INMEM>, grid, dim3(256), 0, (hipStream_t) stream, *a,
                           c0, (int) nc, hb_end, d_nb);
    else
        hipLaunchKernelGGL(k_bound_norms<HS_STD>, grid, dim3(256), 0, (hipStream_t) stream, *a, c0,
                           (int) nc, hb_end, d_nb);
    AGPU_CHECK(hipGetLastError());
    return 0;
}

int agpu_harmbound(const agpu_harmsum_args *a, const float *d_nb, void *stream)
{
    const long long ncell = (long long) a->nblocks * a->corr_uselen;
    if (ncell <= 0)
        return 0;
    if (a->nstages < 1 || a->nstages > 5 || a->nfrac + 1 != 1 << (a->nstages - 1) || a->bstart ||
        a->rh_off)
        return fail("agpu_harmbound: 1..5 stages, blocks that start on whole bins");
    if (a->corr_uselen < HS_CHUNK / 2)
        return fail("agpu_harmbound: corr_uselen below 512 half-bins");
    if (a->inmem && !a->nsq_hb)
        return fail("agpu_harmbound: in-memory path needs the per-half-bin norm table");
    const long long rh_end = a->rh0 + ncell;
    if (a->ntiles < ((rh_end - 1) >> AGPU_TILE_LOG2) + 2 || a->ntiles * AGPU_TILE > 0x7fffffffLL)
        return fail("agpu_harmbound: plane tiles must pad the half-bin range by one tile "
                    "and stay below 2^31 half-bins");
    if ((rh_end + HS_CHUNK) * (long long) ((1 << (a->nstages - 1)) - 1) > 0x7fffffffLL)
        return fail("agpu_harmbound: spectrum too long for 32-bit sub-harmonic indices "
                    "(half-bins x highest harmonic must stay below 2^31)");
    if (!a->row_tab)
        return fail("agpu_harmbound: row table missing");
    if ((long long) a->numz * a->numw * AGPU_ROWLEN > 0x3fffffffLL)
        return fail("agpu_harmbound: too many rows for 32-bit row offsets");
    const int zrows = hb_zrows(a->numz), zblocks = (a->numz + zrows - 1) / zrows;
    const long long nc = agpu_harmbound_chunks(a);
    const long long nblk = (nc + 7) / 8 * 8 * zblocks * a->numw;
    if (nblk >= (1LL << 24))   /* a dispatch counts work-items in 32 bits */
        return fail("agpu_harmbound: grid too large");
    const dim3 grid((unsigned) nblk);
    hipStream_t st = (hipStream_t) stream;
#define HB_CASE(NS)                                                                          \
    case NS:                                                                                 \
        if (a->inmem)                                                                        \
            hipLaunchKernelGGL((k_harmbound<NS, HS_INMEM>), grid, dim3(256), 0, st, *a, d_nb, \
                               (int) nc, zblocks, zrows);                                    \
        else                                                                                 \
            hipLaunchKernelGGL((k_harmbound<NS, HS_STD>), grid, dim3(256), 0, st, *a, d_nb,   \
                               (int) nc, zblocks, zrows);                                    \
        break;
    switch (a->nstages) {
        HB_CASE(1)
        HB_CASE(2)
        HB_CASE(3)
        HB_CASE(4)
        HB_CASE(5)
    }
#undef HB_CASE
    AGPU_CHECK(hipGetLastError());
    return 0;
}

int agpu_hit_sigmas(agpu_hitrec *d_hits, const unsigned *d_nhits, unsigned cap,
                    const agpu_numindep *ni, void *stream)
{
    hipLaunchKernelGGL(k_hit_sigmas, dim3(1024), dim3(64), 0, (hipStream_t) stream, d_hits,
                       d_nhits, cap, *ni);
    AGPU_CHECK(hipGetLastError());
    return 0;
}

int agpu_harmsum_row_table(int numz, int numw, int nfrac, const int *zmap, const int *wmap,
                           unsigned *out)
{
    const long long rows = (long long) numz * numw;
    if (nfrac > AGPU_MAX_FRACS - 1 || AGPU_HS_RT_SUB + nfrac > AGPU_HS_RT)
        return fail("agpu_harmsum_row_table: too many fractions");
    if (rows * AGPU_ROWLEN > 0xffffffffLL)
        return fail("agpu_harmsum_row_table: row offsets exceed 32 bits");
    for (long long r = 0; r < rows; r++) {
        const int wi = (int) (r / numz), zi = (int) (r % numz);
        unsigned *o = out + r * AGPU_HS_RT;
        memset(o, 0, sizeof(unsigned) * AGPU_HS_RT);
        o[0] = (unsigned) wi;
        o[1] = (unsigned) zi;
        o[AGPU_HS_RT_ROW] = (unsigned) (r * AGPU_ROWLEN);
        for (int f = 0; f < nfrac; f++) {
            const long long srow = (long long) wmap[f * numw + wi] * numz + zmap[f * numz + zi];
            o[AGPU_HS_RT_SUB + f] = (unsigned) (srow * AGPU_ROWLEN);
        }
    }
    return 0;
}

int agpu_harmsum_chunk_tables(int mode, int rh_off, long long rh0, long long nchunks,
                              int nstages, int nrows, long long *base, int *lo)
{
    if (mode < 0 || mode > 2 || nstages < 1 || nstages > AGPU_MAX_STAGES)
        return fail("agpu_harmsum_chunk_tables: bad mode or stage count");
    const long long tile_stride = (long long) nrows * AGPU_ROWLEN;
    for (long long c = 0; c < nchunks; c++) {
        long long *b = base + c * AGPU_HS_CT;
        int *l = lo + c * AGPU_HS_CT;
        memset(b, 0, sizeof(long long) * AGPU_HS_CT);
        memset(l, 0, sizeof(int) * AGPU_HS_CT);
        const long long rh_c0 = (rh0 / HS_CHUNK + c) * HS_CHUNK;
        if (rh_c0 > 0x7fffffffLL)
            return fail("agpu_harmsum_chunk_tables: half-bins beyond 2^31");
        b[0] = (rh_c0 >> AGPU_TILE_LOG2) * tile_stride + (rh_c0 & (AGPU_TILE - 1));
        l[0] = (int) rh_c0;
        int f = 0;
        for (int st = 1; st < nstages; st++)
            for (int k = 1; k < (1 << st); k += 2, f++) {
                const int x = hs_span_lo_host(mode, rh_off, (int) rh_c0, k, st);
                l[1 + f] = x;
                b[1 + f] = ((long long) x >> AGPU_TILE_LOG2) * tile_stride +
                           (x & (AGPU_TILE - 1));
            }
    }
    return 0;
}

int agpu_inmem_nsq_table(const float *d_nsq, int npre, int nblocks, long long rh0, int cu,
                         long long hb_end, float *d_out, void *stream)
{
    if (hb_end <= 0)
        return 0;
    long long nb = (hb_end + 255) / 256;
    hipLaunchKernelGGL(k_inmem_nsq_table, dim3((unsigned) nb), dim3(256), 0,
                       (hipStream_t) stream, d_nsq, npre, nblocks, rh0, cu, hb_end, d_out);
    AGPU_CHECK(hipGetLastError());
    return 0;
}

} /* extern "C" */
