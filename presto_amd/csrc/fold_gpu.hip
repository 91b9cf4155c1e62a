/*
 * fold_gpu.hip -- prepfold's fold of a time series for an ACCEL candidate
 * (prepfold -accelcand on a .dat), on the GPU.
 *
 * The reference (src/fold.c:46-107, 443-653; src/prepfold_pipeline.c:
 * 1375-1594) folds records of 1024 points one after another: each point
 * covers the phase interval between its start and end times, and its value
 * is "drizzled" over the profile bins that interval covers, in proportion
 * to the overlap.  Contributions first go to a buffer that is added to the
 * current sub-integration's profile each time one full turn of phase has
 * been added since the fold started (the buffer and the phase added carry
 * across records and sub-integrations); what the last, incomplete turn
 * holds is never added.
 *
 * Here every point is independent: its phase interval [phi(t), phi(t+dt))
 * comes from the FP64 phase polynomial, and each piece of it (split at bin
 * edges and at whole turns of the phase added since the start) goes to the
 * profile of the sub-integration during which its turn completes -- the
 * one whose end phase first reaches the turn's end.  One workgroup folds
 * one record (all its points lie in one sub-integration) into LDS
 * accumulators for that sub-integration and the next, with FP64 LDS atomics,
 * then adds them to the global profiles; turns that complete two or more
 * sub-integrations later (periods longer than a record) go straight to
 * global memory.  The sums are FP64, in an order that varies from run to
 * run in the last bits.
 */
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>
#include "agpu.h"

#define FD_TPB 256
#define FD_REC 1024            /* SUBSBLOCKLEN */
#define FD_LDS_MAXPROF 2048    /* profiles longer than this go to global atomics */

#define FD_CHECK(call)                                                            \
    do {                                                                          \
        hipError_t e_ = (call);                                                   \
        if (e_ != hipSuccess) {                                                   \
            char m_[512];                                                         \
            snprintf(m_, sizeof(m_), "%s:%d %s: %s", __FILE__, __LINE__, #call,   \
                     hipGetErrorString(e_));                                      \
            agpu_set_error(m_);                                                   \
            return -1;                                                            \
        }                                                                         \
    } while (0)

/* phase at time t: t (t (t fdd/6 + fd/2) + f) (src/fold.c:530, 557) */
__device__ static double fd_phase(double t, double f, double fd2, double fdd6)
{
    return t * (t * (t * fdd6 + fd2) + f);
}

__global__ __launch_bounds__(FD_TPB) void k_fold(agpu_fold_args a)
{
    __shared__ double acc[2 * FD_LDS_MAXPROF];
    __shared__ double red[2][FD_TPB / 64];
    const int rec = blockIdx.x;                  /* record */
    const int part = rec / a.rpp, jj = rec % a.rpp;
    const int n = a.proflen;
    const bool use_lds = n <= FD_LDS_MAXPROF;
    if (use_lds)
        for (int k = threadIdx.x; k < 2 * n; k += FD_TPB)
            acc[k] = 0.0;
    __syncthreads();
    const double proftime = FD_REC * a.dt;
    /* fold_time0 of the record, as src/prepfold_pipeline.c:1515, 1577 */
    const double tlo = (double) ((long long) part * a.rpp) * proftime + jj * proftime;
    const double fd2 = a.fd / 2.0, fdd6 = a.fdd / 6.0;
    const double phi0 = a.phi_start;
    double s1 = 0.0, s2 = 0.0;
    for (int l = threadIdx.x; l < FD_REC; l += FD_TPB) {
        const long long i = (long long) rec * FD_REC + l;
        const double x = a.series[i];
        s1 += x;
        s2 += x * x;
        const double t = tlo + l * a.dt, tn = tlo + (l + 1) * a.dt;
        const double ph = fd_phase(t, a.f, fd2, fdd6), phn = fd_phase(tn, a.f, fd2, fdd6);
        double dph = phn - ph;
        if (!(dph > 1e-12))
            continue;
        const double valperphs = x / dph;
        double lophase = ph - floor(ph);
        double u = ph - phi0;                 /* phase added before this point */
        double curbin = lophase * n;
        while (dph > 1e-12) {
            int ib = (int) floor(curbin + 1e-12);
            double dphs = ((ib + 1.0) - curbin) / n;
            ib %= n;
            if (dphs > dph)
                dphs = dph;
            /* split the piece [u, u + dphs) at whole turns of phase added */
            double lo = u;
            const double hi = u + dphs;
            while (lo < hi) {
                const double turn = floor(lo);
                const double end = fmin(hi, turn + 1.0);
                const double v = (end - lo) * valperphs;
                /* the sub-integration during which this turn completes */
                int tp = part;
                while (tp < a.npart && a.part_end[tp] < turn + 1.0)
                    tp++;
                if (tp < a.npart) {
                    if (use_lds && tp - part < 2)
                        atomicAdd(&acc[(tp - part) * n + ib], v);
                    else
                        atomicAdd(&a.rawfolds[(size_t) tp * n + ib], v);
                }
                lo = end;
            }
            u = hi;
            dph -= dphs;
            curbin += dphs * n;
        }
    }
    /* per-record sums of the data for the statistics */
    for (int off = 32; off > 0; off >>= 1) {
        s1 += __shfl_xor(s1, off);
        s2 += __shfl_xor(s2, off);
    }
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = s1;
        red[1][threadIdx.x >> 6] = s2;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double t1 = 0.0, t2 = 0.0;
        for (int w = 0; w < FD_TPB / 64; w++) {
            t1 += red[0][w];
            t2 += red[1][w];
        }
        a.recsums[2 * rec] = t1;
        a.recsums[2 * rec + 1] = t2;
    }
    if (use_lds)
        for (int k = threadIdx.x; k < 2 * n; k += FD_TPB) {
            const int tp = part + k / n;
            if (tp < a.npart && acc[k] != 0.0)
                atomicAdd(&a.rawfolds[(size_t) tp * n + k % n], acc[k]);
        }
}

extern "C" int agpu_fold(const agpu_fold_args *args, void *stream)
{
    if (args->npart < 1 || args->rpp < 1 || args->proflen < 2) {
        agpu_set_error("agpu_fold: bad sub-integration or profile size");
        return -1;
    }
    const long long nrec = (long long) args->npart * args->rpp;
    if (nrec > 0x7fffffffLL) {
        agpu_set_error("agpu_fold: too many records");
        return -1;
    }
    hipLaunchKernelGGL(k_fold, dim3((unsigned) nrec), dim3(FD_TPB), 0, (hipStream_t) stream,
                       *args);
    FD_CHECK(hipGetLastError());
    return 0;
}

/* prepfold's period / period-derivative search over the sub-integrations
 * of one subband (src/prepfold_pipeline.c:1696-1868; combine_profs,
 * src/fold.c:696-754; chisqr, src/characteristics.c:562-575).  In trial
 * (ip, ipd) of the launch's p-dotdot trial part ii is delayed by
 * fdotdot2phasedelay(fdotdots[ipdd], parttimes[ii]) proflen (0 without a
 * p-dotdot search) + fdot2phasedelay(fdots[ipd], parttimes[ii]) proflen +
 * ii tot / npart bins (tot = pstep (ip - centre)), the delay rounded to whole
 * bins as combine_profs does; the shifted profiles are summed per bin in
 * part order and the reduced chi-squared over the bins in order, so every
 * trial's value is the reference's operation for operation. */

/* the part of a delay that all periods of one p-dot share */
__device__ static double fs_base(const agpu_fold_search_args &a, int ipd, int ii)
{
#pragma clang fp contract(off)
    const double t = a.parttimes[ii];
    double pdd_delay = 0.0;
    if (a.fdotdots) {
        double pdd = a.fdotdots[a.ipdd] * t * t * t / 6.0;   /* fdotdot2phasedelay */
        if (pdd == -0)
            pdd = 0.0;
        pdd_delay = pdd * a.proflen;
    }
    double pd = a.fdots[ipd] * t * t / 2.0;   /* fdot2phasedelay */
    if (pd == -0)
        pd = 0.0;
    return pdd_delay + pd * a.proflen;
}

__device__ static int fs_offset(const agpu_fold_search_args &a, double base, int ii, int tot)
{
#pragma clang fp contract(off)
    const double delay = base + (double) (ii * tot) / a.npart;
    /* fmod(-delay, proflen).  Below 2^52 the remainder of the whole quotient
     * is exact in one fma, and so is the step that mends a quotient that the
     * product with the reciprocal rounded to the next whole number. */
    const double x = -delay, y = a.proflen, ax = fabs(x);
    double ld;
    if (ax < 4503599627370496.0) {
        double r = fma(-trunc(ax * (1.0 / y)), y, ax);
        if (r < 0.0)
            r += y;
        if (r >= y)
            r -= y;
        ld = x < 0.0 ? -r : r;
    } else
        ld = fmod(x, y);
    if (ld < 0.0)
        ld += a.proflen;
    return (int) (ld + 0.5);
}

/* reduced chi-squared of a summed profile, stored; its bits if it counts as
 * a maximum (above 0, not NaN) */
__device__ static unsigned long long fs_redchi(const agpu_fold_search_args &a, const double *prof,
                                               int ip, int ipd)
{
#pragma clang fp contract(off)
    double chi = 0.0;
#pragma unroll 8
    for (int k = 0; k < a.proflen; k++) {
        const double d = prof[k] - a.prof_avg;
        chi += d * d;
    }
    const double v = chi / a.prof_var / (a.proflen - 1.0);
    const size_t i = (size_t) ipd * a.numtrials + ip;
    a.redchi[i] = v;
    a.redchif[i] = (float) v;
    return v > 0.0 ? (unsigned long long) __double_as_longlong(v) : 0;
}

/* Tiles of FS_TR consecutive periods of one p-dot, dealt to as many
 * workgroups as are resident: each reads the folds into LDS once, and a
 * tile's serial sums over the bins run in FS_TR lanes at once.  One workgroup
 * per trial (k_fold_search) re-read the folds and summed in a single lane:
 * 136 us for 257 x 257 trials of 64 parts by 64 bins, here 83.  Bound by the
 * LDS reads of a sum (8 B per trial, part and bin: 30 us at 128 B a clock,
 * half as much again for the offsets) and by the latency of its chain, which
 * 16 waves per workgroup cover better than 4, and two workgroups a CU better
 * than one (97 us): the second launch bound holds the scalar registers to 8
 * waves per SIMD (106 of them allow 7, so one workgroup of 4 per SIMD). */
#define FS_TR 32
#define FS_TH 1024
#define FS_UN 8 /* parts per step of a sum: their loads are in flight together */
/* parts rounded up to whole steps, so that a trial's offsets are aligned */
static __host__ __device__ int fs_rows(int npart)
{
    return (npart + FS_UN - 1) & ~(FS_UN - 1);
}
static size_t fs_tile_lds(int npart, int proflen)
{
    return sizeof(double) * ((size_t) npart * proflen + (size_t) FS_TR * (proflen + 1) + npart) +
           sizeof(int) * (size_t) FS_TR * fs_rows(npart);
}

__global__ __launch_bounds__(FS_TH, 8) void k_fold_search_tile(agpu_fold_search_args a)
{
    extern __shared__ double fs_lds[];
    const int L = a.proflen, nt = a.numtrials, nr = fs_rows(a.npart);
    /* offs first: its rows are read in vectors */
    int *offs = (int *) fs_lds;
    double *folds = (double *) (offs + FS_TR * nr), *prof = folds + a.npart * L;
    double *base = prof + FS_TR * (L + 1);
    const int per = (nt + FS_TR - 1) / FS_TR;
    const int nl = a.npart * L;
    for (int i0 = threadIdx.x; i0 < nl; i0 += 8 * FS_TH) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; u++)
            v[u] = a.profs[min(i0 + u * FS_TH, nl - 1)];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (i0 + u * FS_TH < nl)
                folds[i0 + u * FS_TH] = v[u];
    }
    for (int t = blockIdx.x; t < per * nt; t += gridDim.x) {
        const int ipd = t / per, ip0 = (t - ipd * per) * FS_TR;
        for (int ii = threadIdx.x; ii < a.npart; ii += FS_TH)
            base[ii] = fs_base(a, ipd, ii);
        __syncthreads();
        for (int i = threadIdx.x; i < FS_TR * nr; i += FS_TH) {
            const int tr = i / nr, ii = i - tr * nr;
            const int tot = a.pstep * (ip0 + tr - (nt - 1) / 2);
            offs[i] = ii < a.npart ? fs_offset(a, base[ii], ii, tot) : 0;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < FS_TR * L; i += FS_TH) {
            const int tr = i / L, k = i - tr * L;
            const int *o = offs + tr * nr;
            const double *row = folds;
            double s = 0.0;
            int ii = 0;
            for (; ii + FS_UN <= a.npart; ii += FS_UN) {
                double v[FS_UN];
#pragma unroll
                for (int u = 0; u < FS_UN; u++) {
                    const unsigned j = (unsigned) (k + o[ii + u]);
                    v[u] = row[min(j, j - (unsigned) L)];
                    row += L;
                }
#pragma unroll
                for (int u = 0; u < FS_UN; u++)
                    s += v[u];
            }
            for (; ii < a.npart; ii++) {
                const unsigned j = (unsigned) (k + o[ii]);
                s += row[min(j, j - (unsigned) L)];
                row += L;
            }
            prof[tr * (L + 1) + k] = s;
        }
        __syncthreads();
        /* base, which the next tile writes meanwhile, is not read here; its
         * first barrier keeps prof and offs until this wave is through */
        if (threadIdx.x < 64) {
            const int tr = threadIdx.x;
            unsigned long long key = 0;
            if (tr < FS_TR && ip0 + tr < nt)
                key = fs_redchi(a, prof + tr * (L + 1), ip0 + tr, ipd);
            for (int d = 32; d >= 1; d >>= 1) {
                const unsigned long long o = __shfl_xor(key, d, 64);
                key = o > key ? o : key;
            }
            if (threadIdx.x == 0)
                a.tilemax[t] = key;
        }
    }
}

/* one workgroup per trial, where the folds do not fit in LDS */
__global__ __launch_bounds__(256) void k_fold_search(agpu_fold_search_args a)
{
    extern __shared__ double fs_lds[];
    double *prof = fs_lds;                     /* proflen */
    int *offs = (int *) (fs_lds + a.proflen);  /* npart */
    const int ip = blockIdx.x, ipd = blockIdx.y;
    const int L = a.proflen;
    const int tot = a.pstep * (ip - (a.numtrials - 1) / 2);
    for (int ii = threadIdx.x; ii < a.npart; ii += blockDim.x)
        offs[ii] = fs_offset(a, fs_base(a, ipd, ii), ii, tot);
    __syncthreads();
    for (int k = threadIdx.x; k < L; k += blockDim.x) {
        double s = 0.0;
        for (int ii = 0; ii < a.npart; ii++) {
            int j = k + offs[ii];
            if (j >= L)
                j -= L;
            s += a.profs[(size_t) ii * L + j];
        }
        prof[k] = s;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        a.tilemax[(size_t) ipd * gridDim.x + ip] = fs_redchi(a, prof, ip, ipd);
}

extern "C" int agpu_fold_tile(int npart, int proflen)
{
    return fs_tile_lds(npart, proflen) <= 64 * 1024 ? FS_TR : 1;
}

/* workgroups of the tile kernel that the current device holds at once: a
 * further one would read the folds again for tiles that a resident one could
 * take (32 parts by 64 bins, 1024 instead of 512 workgroups: 63 us against
 * 54, of which the second workgroup of a CU gives 8) */
extern "C" int agpu_fold_resident(int npart, int proflen)
{
    int dev = 0, ncu = 0, per_cu = 0;
    FD_CHECK(hipGetDevice(&dev));
    FD_CHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    FD_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_fold_search_tile, FS_TH,
                                                          fs_tile_lds(npart, proflen)));
    return ncu * (per_cu > 0 ? per_cu : 1);
}

extern "C" int agpu_fold_search(const agpu_fold_search_args *args, void *stream)
{
    if (args->npart < 1 || args->proflen < 2 || args->numtrials < 1 ||
        args->numtrials > 65535) {
        agpu_set_error("agpu_fold_search: bad sizes");
        return -1;
    }
    /* 64 KB keep two workgroups of a tile on a CU; beyond (64 parts of more
     * than 64 bins or so) the folds stay in L2 */
    if (agpu_fold_tile(args->npart, args->proflen) == FS_TR) {
        const long tiles = (long) ((args->numtrials + FS_TR - 1) / FS_TR) * args->numtrials;
        const long resident = agpu_fold_resident(args->npart, args->proflen);
        if (resident < 0)
            return -1;
        hipLaunchKernelGGL(k_fold_search_tile, dim3((unsigned) (tiles < resident ? tiles : resident)),
                           dim3(FS_TH), fs_tile_lds(args->npart, args->proflen),
                           (hipStream_t) stream, *args);
        FD_CHECK(hipGetLastError());
        return 0;
    }
    const size_t lds = sizeof(double) * (size_t) args->proflen +
                       sizeof(int) * (size_t) args->npart;
    if (lds > 64 * 1024) {
        agpu_set_error("agpu_fold_search: profile and parts too large for LDS");
        return -1;
    }
    hipLaunchKernelGGL(k_fold_search, dim3((unsigned) args->numtrials, (unsigned) args->numtrials),
                       dim3(64), lds, (hipStream_t) stream, *args);
    FD_CHECK(hipGetLastError());
    return 0;
}

/* The first trial that holds the largest redchi above 0.  Tiles lie in the
 * trials' order, so it is in the first tile that holds the maximum; one
 * workgroup reads the tiles' maxima, and no atomic on one address is left
 * for every tile of the search to wait on. */
__global__ __launch_bounds__(1024) void k_fold_first(const double *redchi,
                                                     const unsigned long long *tilemax,
                                                     unsigned long long ntiles, int numtrials,
                                                     int tile, unsigned long long *first)
{
    __shared__ unsigned long long smax[1024], sidx[1024];
    unsigned long long m = 0, at = 0;
    for (unsigned long long i = threadIdx.x; i < ntiles; i += 1024)
        if (tilemax[i] > m) {
            m = tilemax[i];
            at = i;
        }
    smax[threadIdx.x] = m;
    sidx[threadIdx.x] = at;
    __syncthreads();
    for (int d = 512; d >= 1; d >>= 1) {
        if (threadIdx.x < d) {
            const unsigned long long om = smax[threadIdx.x + d], oi = sidx[threadIdx.x + d];
            if (om > smax[threadIdx.x] ||
                (om == smax[threadIdx.x] && oi < sidx[threadIdx.x])) {
                smax[threadIdx.x] = om;
                sidx[threadIdx.x] = oi;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const unsigned long long per = (unsigned long long) ((numtrials + tile - 1) / tile);
        const unsigned long long row = sidx[0] / per;
        unsigned long long i = row * numtrials + sidx[0] % per * tile;
        if (smax[0])
            while ((unsigned long long) __double_as_longlong(redchi[i]) != smax[0])
                i++;
        *first = smax[0] ? i : 0;
    }
}

extern "C" int agpu_fold_first(const double *d_redchi, const unsigned long long *d_tilemax,
                               unsigned long long rows, int numtrials, int tile,
                               unsigned long long *d_first, void *stream)
{
    if (rows == 0 || numtrials < 1 || tile < 1) {
        agpu_set_error("agpu_fold_first: bad sizes");
        return -1;
    }
    hipLaunchKernelGGL(k_fold_first, dim3(1), dim3(1024), 0, (hipStream_t) stream, d_redchi,
                       d_tilemax, rows * (unsigned long long) ((numtrials + tile - 1) / tile),
                       numtrials, tile, d_first);
    FD_CHECK(hipGetLastError());
    return 0;
}
