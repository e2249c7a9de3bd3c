// CF -> SF transform and the Monte Carlo M0 moment on gfx950.
//
// CF -> SF (idct_cf_to_sf, src/hawaii.c:5569-5601): Connes apodization (src/hawaii.c:5401-5410), the
//   IDCT (src/hawaii.c:5478-5553) times tmax/pi*Yscale at nu_k = k pi/tmax*Xscale.
//
// M0 (calculate_M0, src/hawaii.c:1423-1491): every lane owns one Mersenne Twister stream
// (mt_seed32 seeding, state interleaved across lanes so equal draw indices coalesce) and
// runs the reference's candidate loop (q_generator, p_generator, Hamiltonian, reject, pair
// filter, dipole, Welford running mean / sum of squared deviations) over its quota.
// M2 (calculate_M2, src/hawaii.c:1524-1617) is the same loop with |d mu/dt|^2 as the value.
#include <hip/hip_runtime.h>

#include "hh_engine.h"
#include "hh_systems.h"

namespace hh {

constexpr double kPI = 3.14159265358979323846;

// ------------------------------------------------------------------ CF -> SF
// The reference packs the n apodized samples v into a Hermitian sequence of 2n complex values and keeps
// n of the transform's 2n values, which are real: sf_j ~ v_0 + 2 sum_k v_k cos(pi k (2j + 1) / 2n).
// That is a complex transform of n points (Makhoul 1980) of
//   V_k = e^{i pi k / 2n} (v_k - i v_{n-k}), v_n = 0,   x_j = sum_k V_k e^{2 pi i jk / n}
// whose real parts x_0, x_1, ... are sf_0, sf_2, ... and, from the end, sf_1, sf_3, ...  (The x are real, so
// n/2 points would do, for 2 us less of a call's 44 at n = 4096, but the imaginary parts take half of the
// rounding errors' squares with them: error in the 2-norm 2.5e-16 to 3.5e-16 from n = 2^10 to 2^20, against
// 1.8e-16 to 2.7e-16 here and 2.0e-16 to 2.8e-16 with radix-2 stages over the 2n points.)
//
// The points run as Stockham passes of radix R over global memory, each R-point transform in LDS by
// eight points per thread (radix 8, the last step 2, 4 or 8): one workgroup does it all up to
// n = 4096, beyond that it is as few passes as that allows (two up to n = 2^20).  The first pass makes
// the V_k from cf as it loads them, the last one writes sf in order, nu and the apodized cf.
// What bounds it: at n = 4096 the call's launch and wait and the instructions of one workgroup; at 2^20
// points two passes over 16 MiB with a sincospi per point and pass.  Radix-2 stages with a sincospi per
// butterfly took 65 us of kernels at n = 4096 and 245 us at 2^20; this takes
// 15 us and 33 us.
constexpr int kFftSingleLog = 12;   // one workgroup: 512 threads, 136 KiB of LDS
constexpr int kFftPassLog = 10;     // a pass of 4 columns: 512 threads, 88 KiB
constexpr int kFftColsLog = 2;      // columns of a workgroup: 64-byte rows of complex values
constexpr double kSqrtHalf = 0.70710678118654752440;

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b)
{
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 ctimes_i(double2 a) { return make_double2(-a.y, a.x); }
__device__ __forceinline__ double2 cispi(double x)
{
    double2 w;
    sincospi(x, &w.y, &w.x);
    return w;
}

// backward transforms (e^{+i}) of 2, 4 and 8 points, in place
__device__ __forceinline__ void dft4(double2& a, double2& b, double2& c, double2& d)
{
    const double2 s = cadd(a, c), t = csub(a, c), u = cadd(b, d), v = ctimes_i(csub(b, d));
    a = cadd(s, u);
    b = cadd(t, v);
    c = csub(s, u);
    d = csub(t, v);
}

__device__ __forceinline__ void dft8(double2* v)
{
    double2 e[4], o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        e[i] = cadd(v[i], v[i + 4]);
        o[i] = csub(v[i], v[i + 4]);
    }
    o[1] = make_double2((o[1].x - o[1].y) * kSqrtHalf, (o[1].x + o[1].y) * kSqrtHalf);
    o[2] = ctimes_i(o[2]);
    o[3] = make_double2(-(o[3].x + o[3].y) * kSqrtHalf, (o[3].x - o[3].y) * kSqrtHalf);
    dft4(e[0], e[1], e[2], e[3]);
    dft4(o[0], o[1], o[2], o[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = e[i];
        v[2 * i + 1] = o[i];
    }
}

// x (1 - r^2)^2, r = k/n (exact: n is a power of two), the window with its rounding error
__device__ __forceinline__ double connes(double x, long k, double inv_n)
{
    const double r = (double)k * inv_n, p = r * r, f = 1.0 - p;
    const double fl = (-p - (f - 1.0)) - fma(r, r, -p);
    const double g = f * f, gl = fma(f, f, -g) + 2.0 * f * fl;
    return fma(x, g, x * gl);
}

// One Stockham pass of radix R = 2^logr, after passes of a combined radix 2^logl, for the 2^logc columns
// of this workgroup.  A thread holds rows q = b + i R/8 of one column.
template <bool FIRST, bool LAST>
__global__ void __launch_bounds__(512) sf_pass_kernel(double* cf, const double2* __restrict__ in,
                                                       double2* __restrict__ out, double* __restrict__ nu,
                                                       double* __restrict__ sf, int logn, double dt, int logr, int logl,
                                                       int logc)
{
    extern __shared__ double2 sm[];
    const long n = 1L << logn;
    const int t = threadIdx.x, c = t & ((1 << logc) - 1), b = t >> logc, eighth = 1 << (logr - 3);
    const int logcols = logn - logr;
    const long L = 1L << logl;
    // Workgroups go to the eight XCDs in turn: neighbouring tiles, which share cache lines, go to one
    // (n = 2^20: 42 -> 33 us)
    const long tile = gridDim.x % 8 ? blockIdx.x : (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
    // a pass's columns j; in the last pass half of a workgroup's columns mirror the other half
    const int half = 1 << logc >> 1;
    long j;
    if (LAST && half)
        j = c < half ? tile * half + c : (1L << logcols) - 1 - (tile * half + c - half);
    else
        j = (tile << logc) + c;
    const long k0 = j & (L - 1);
    auto slot = [&](int q, int col) { return ((q + (q >> 3)) << logc) + col; };

    double2 v[8];
    if constexpr (FIRST) {
        const double inv_n = 1.0 / (double)n;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const long k = j + ((long)(b + i * eighth) << logcols);
            const double v0 = connes(cf[k], k, inv_n), v1 = k ? connes(cf[n - k], n - k, inv_n) : 0.0;
            v[i] = cmul(cispi((double)k * (0.5 * inv_n)), make_double2(v0, -v1));
        }
    } else {
        const double unit = 2.0 / (double)(L << logr);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int q = b + i * eighth;
            v[i] = cmul(in[j + ((long)q << logcols)], cispi((double)(q * k0) * unit));
        }
    }
    // the roots e^{2 pi i q / R} of the steps
    double2* root = sm + ((1 << logr) + (1 << (logr - 3)) << logc);
    const double rel = 2.0 / (double)(1 << logr);
    for (int q = t; q < 1 << logr; q += blockDim.x) root[q] = cispi((double)q * rel);

    for (int lg = 0;;) {
        const int rest = logr - lg;
        if (rest >= 3) {
            if (lg) {
                const int k = (b & ((1 << lg) - 1)) << (logr - lg - 3);
#pragma unroll
                for (int i = 1; i < 8; ++i) v[i] = cmul(v[i], root[i * k]);
            }
            dft8(v);
            if (rest == 3) break;
        } else {
            // radix 4 or 2: butterflies of the rows b + u R/8
            if (rest == 2) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
#pragma unroll
                    for (int i = 1; i < 4; ++i) v[2 * i + u] = cmul(v[2 * i + u], root[i * (b + u * eighth)]);
                    dft4(v[u], v[2 + u], v[4 + u], v[6 + u]);
                }
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const double2 x = cmul(v[4 + u], root[b + u * eighth]);
                    v[4 + u] = csub(v[u], x);
                    v[u] = cadd(v[u], x);
                }
            }
            break;
        }
        const int k = b & ((1 << lg) - 1), g = b >> lg;
        if (lg) __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; ++i) sm[slot((g << (lg + 3)) + k + (i << lg), c)] = v[i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = sm[slot(b + i * eighth, c)];
        lg += 3;
    }

    if constexpr (!LAST) {
        const long o = ((j >> logl) << (logl + logr)) + k0;
#pragma unroll
        for (int i = 0; i < 8; ++i) out[o + ((long)(b + i * eighth) << logl)] = v[i];
    } else {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; ++i) sm[slot(b + i * eighth, c)] = v[i];
        __syncthreads();
        const double LightSpeed_cm = 2.99792458e10, ATU = 2.4188843265857e-17;
        const double ADIPMOMU = 8.4783536255e-30, EPSILON0 = 8.8541878128e-12;
        const double Xscale = 1.0 / LightSpeed_cm / ATU / 2.0 / kPI;
        const double Yscale = ATU * ADIPMOMU * ADIPMOMU / (4.0 * kPI * EPSILON0);
        const double tmax = n * dt;
        // tmax / pi * Yscale / 2n with its rounding error
        const double q0 = tmax / kPI, q1 = fma(-q0, kPI, tmax) / kPI, inv2n = 0.5 / n;
        const double s0 = q0 * Yscale * inv2n, s1 = (fma(q0, Yscale, -(q0 * Yscale)) + q1 * Yscale) * inv2n;
        auto scaled = [&](double x) { return fma(x, s0, x * s1); };
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = t + i * blockDim.x;
            const int col = half ? e & (half - 1) : 0, q = half ? e >> (logc - 1) : e;
            long m = (half ? tile * half + col : 0) + ((long)q << logl);
            double y = sm[slot(q, col)].x, ym = sm[slot((1 << logr) - 1 - q, half + col)].x;
            if (m >= n / 2) {
                m = n - 1 - m;
                const double s = y;
                y = ym;
                ym = s;
            }
            sf[2 * m] = scaled(y);
            sf[2 * m + 1] = scaled(ym);
        }
        const double itmax = recip<double>(tmax);
#pragma unroll 4
        for (int i = 0; i < 8; ++i) {
            const long k = ((long)blockIdx.x * 8 + i) * blockDim.x + t;
            // Connes apodization of the input in place, as the reference does (src/hawaii.c:5581): no
            // workgroup reads cf any more
            const double r = divide<double>(dt * k, tmax, itmax);
            cf[k] *= (1.0 - r * r) * (1.0 - r * r);
            nu[k] = divide<double>(k * kPI, tmax, itmax) * Xscale;
        }
    }
}

// n = 2, 4: the cosine sum itself
__global__ void __launch_bounds__(64) sf_direct_kernel(double* cf, double* __restrict__ nu, double* __restrict__ sf,
                                                       int n, double dt)
{
    const int j = threadIdx.x;
    double x[4], acc = 0.0;
    for (int k = 0; k < n; ++k) x[k] = cf[k];
    __syncthreads();
    if (j >= n) return;
    for (int k = 0; k < n; ++k)
        acc += (k ? 2.0 : 1.0) * connes(x[k], k, 1.0 / n) * cospi((double)(k * (2 * j + 1)) / (2.0 * n));
    const double LightSpeed_cm = 2.99792458e10, ATU = 2.4188843265857e-17;
    const double ADIPMOMU = 8.4783536255e-30, EPSILON0 = 8.8541878128e-12;
    const double Xscale = 1.0 / LightSpeed_cm / ATU / 2.0 / kPI;
    const double Yscale = ATU * ADIPMOMU * ADIPMOMU / (4.0 * kPI * EPSILON0);
    const double tmax = n * dt, r = (dt * j) / (dt * n);
    cf[j] *= (1.0 - r * r) * (1.0 - r * r);
    nu[j] = j * kPI / tmax * Xscale;
    sf[j] = acc * (tmax / kPI * Yscale / (2.0 * n));
}

// Global passes of a transform of 2^logn points: as many as it takes at 2^kFftPassLog points each
int sf_passes(int logn) { return logn <= kFftSingleLog ? 1 : (logn + kFftPassLog - 1) / kFftPassLog; }

size_t sf_work_bytes(long n, int which)
{
    int logn = 0;
    while ((1L << logn) < n) ++logn;
    return sf_passes(logn) > 1 + which ? (size_t)n * sizeof(double2) : 0;
}

hipError_t run_cf_to_sf(double* cf, long n, double dt, double2* work_a, double2* work_b, double* nu, double* sf,
                        hipStream_t st)
{
    int logn = 0;
    while ((1L << logn) < n) ++logn;
    if (n <= 4) {
        hipLaunchKernelGGL(sf_direct_kernel, dim3(1), dim3(64), 0, st, cf, nu, sf, (int)n, dt);
        return hipGetLastError();
    }
    const int passes = sf_passes(logn);
    double2 *src = work_b, *dst = work_a;
    int logl = 0;
    for (int p = 0; p < passes; ++p) {
        const int logr = (logn - logl + passes - p - 1) / (passes - p), logc = passes == 1 ? 0 : kFftColsLog;
        const bool first = p == 0, last = p == passes - 1;
        auto k = first ? (last ? sf_pass_kernel<true, true> : sf_pass_kernel<true, false>)
                       : (last ? sf_pass_kernel<false, true> : sf_pass_kernel<false, false>);
        const int points = 1 << (logr + logc);
        const size_t lds = (size_t)(points + points / 8 + (1 << logr)) * sizeof(double2);
        if (lds > 65536) {
            const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     (int)lds);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(k, dim3((unsigned)(n >> (logr + logc))), dim3(points / 8), lds, st, cf, src, dst, nu,
                           sf, logn, dt, logr, logl, logc);
        logl += logr;
        double2* x = src;
        src = dst;
        dst = x;
    }
    return hipGetLastError();
}

// ------------------------------------------------------------------ CF -> SF without allocation
// The n-point work sequence of the transform lives in a file-scope device array instead of an
// engine-allocated buffer, for callers that cannot allocate (graph capture, tight serving loops).
// Every device holds its own copy; its address comes from hipGetSymbolAddress once per device
// (noalloc_scratch_address, at engine creation) and only that address is passed to kernels: the
// array's name in host code is a host-side stand-in, not a device address.  Calls that overlap on
// one device share the array and race.
__device__ __align__(256) double2 scratch[kCfToSfNoAllocMaxN];

hipError_t noalloc_scratch_address(void** ptr)
{
    return hipGetSymbolAddress(ptr, HIP_SYMBOL(scratch));
}

// ------------------------------------------------------------------ M0
constexpr int kMTN = 624, kMTM = 397;
constexpr int kMTBatch = 16;   // divides kMTN, below kMTN - kMTM
constexpr double kHkT = 4.3597447222071e-18 / 1.380649e-23;

// Stream state for lane s lives at st[i * nstreams + s].  The generator's next words are made kMTBatch at a
// time, where the reference's twist makes all kMTN: 33 loads in flight at once and one wait for them every
// 16 draws, which come from LDS, instead of a wait per draw and three per twisted word (with one wavefront
// per SIMD nothing else hides them; 4e6 He-Ar points of 65536 streams: 1535 -> 893 us, now bound by the
// candidates' own instructions).  Every candidate takes the same number of draws, so the lanes of a
// wavefront refill together and their loads stay coalesced.
struct LaneMt {
    uint32_t* st;
    long ns, s;
    int pos;           // draws taken of the present kMTN words
    uint32_t* ahead;   // this lane's words of the present batch, tempered, at stride 256
    __device__ uint32_t& w(int i) { return st[(long)i * ns + s]; }
    __device__ static uint32_t temper(uint32_t y)
    {
        y ^= y >> 11;
        y ^= (y << 7) & 0x9d2c5680u;
        y ^= (y << 15) & 0xefc60000u;
        return y ^ (y >> 18);
    }
    __device__ void refill()
    {
        if (pos == kMTN) pos = 0;
        uint32_t old[kMTBatch + 1], far[kMTBatch];
#pragma unroll
        for (int j = 0; j < kMTBatch; ++j) {
            old[j] = w(pos + j);
            const int f = pos + j + kMTM;
            far[j] = w(f < kMTN ? f : f - kMTN);
        }
        old[kMTBatch] = w(pos + kMTBatch < kMTN ? pos + kMTBatch : 0);
#pragma unroll
        for (int j = 0; j < kMTBatch; ++j) {
            const uint32_t y = (old[j] & 0x80000000u) | (old[j + 1] & 0x7fffffffu);
            const uint32_t x = far[j] ^ (y >> 1) ^ ((y & 1u) ? 0x9908b0dfu : 0u);
            w(pos + j) = x;
            ahead[j * 256] = temper(x);
        }
    }
    // the batch in use when the last launch ended: its words are in the state
    __device__ void resume()
    {
        const int b0 = pos / kMTBatch * kMTBatch;
        if (pos > b0)
            for (int j = 0; j < kMTBatch; ++j) ahead[j * 256] = temper(w(b0 + j));
    }
    __device__ double drand()
    {
        const int j = pos % kMTBatch;
        if (j == 0) refill();
        ++pos;
        return (double)ahead[j * 256] * (1.0 / 4294967296.0);
    }
};

__device__ double m0_normal(LaneMt& mt)
{
    for (;;) {
        const double U = mt.drand();
        const double V = mt.drand();
        const double logU = log(U);
        if (isnan(logU) || isinf(logU)) continue;
        return sqrt(-2 * logU) * cos(2.0 * kPI * V);
    }
}

// One launch draws candidates for every stream until it has its quota, hits the candidate
// limit, or (ticks > 0) the launch has run `ticks` wall-clock ticks; `init` seeds the streams.
// ORDER 0 averages |mu|^2 (M0), ORDER 2 |d mu/dt|^2 (M2).
template <int SYS, int ORDER>
__global__ void __launch_bounds__(256) m0_kernel(SysConst sc, M0Params p, uint32_t seed, long nstreams, long npoints,
                                                 uint32_t* __restrict__ state, M0Acc acc, int init, long long ticks)
{
    const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nstreams) return;
    const long long t_end = wall_clock64() + ticks;
    __shared__ uint32_t ahead[kMTBatch * 256];
    LaneMt mt{state, nstreams, s, 0, ahead + threadIdx.x};
    const long quota = npoints / nstreams + (s < npoints % nstreams ? 1 : 0);
    const long max_candidates = quota * 100000 + 100000;   // bounded even if nothing is ever accepted
    long candidates = 0, n = 0;
    double m = 0.0, q = 0.0;
    if (init) {
        uint32_t v = seed + (uint32_t)s;
        if (v == 0) v = 4357u;
        mt.w(0) = v;
        for (int i = 1; i < kMTN; ++i) mt.w(i) = v = 69069u * v;
    } else {
        mt.pos = acc.pos[s];
        mt.resume();
        m = acc.m[s];
        q = acc.q[s];
        n = acc.n[s];
        candidates = acc.cand[s];
    }
    const bool was_done = !init && (n >= quota || candidates >= max_candidates);
    double y[10];
    const double RMIN = p.Rmin, RMAX = p.Rmax, T = p.T;
    const double sqrt_MUKT = sqrt(sc.mu / kHkT * T);
    const double sqrt_IIKT = sqrt(sc.I / kHkT * T);
    const double M = 1.5 * exp(-p.pesmin * kHkT / T);
    while (n < quota && candidates < max_candidates) {
        if (ticks > 0 && wall_clock64() >= t_end) break;
        ++candidates;
        const double R3 = mt.drand() * (RMAX * RMAX * RMAX - RMIN * RMIN * RMIN) + RMIN * RMIN * RMIN;
        y[4] = pow(R3, 1.0 / 3.0);
        y[0] = mt.drand() * 2.0 * kPI;
        y[2] = acos(2.0 * mt.drand() - 1.0);
        if (SYS == SYS_CO2AR) {
            y[6] = mt.drand() * 2.0 * kPI;
            y[8] = acos(2.0 * mt.drand() - 1.0);
        }
        const double sinT = sin(y[2]);
        const double x0 = m0_normal(mt), x1 = m0_normal(mt), x2 = m0_normal(mt);
        y[1] = sqrt_MUKT * y[4] * sinT * x0;
        y[3] = sqrt_MUKT * y[4] * x1;
        y[5] = sqrt_MUKT * x2;
        if (SYS == SYS_CO2AR) {
            const double st = sin(y[8]);
            const double r0 = m0_normal(mt), r1 = m0_normal(mt);
            y[7] = sqrt_IIKT * st * r1;
            y[9] = sqrt_IIKT * r0;
        }
        // Hamiltonian before reject (src/hawaii.c:1456-1459), then reject (src/hawaii.c:1382-1421):
        // u is drawn first; K and V at the same point
        const double K = kinetic<SYS>(sc, y);
        const double V = pes_value<SYS, double>(sc, y);
        const double energy = K + V;
        const double u = mt.drand();
        const double weight = exp(-(K + V) * kHkT / T) / exp(-K * kHkT / T) / M;
        if (weight < u) continue;
        if (p.pair_state == 1 && energy < 0.0) continue;
        if (p.pair_state == 2 && energy > 0.0) continue;
        double f;
        if constexpr (ORDER == 2) {
            f = dipole_rate_sq<SYS>(sc, y);
        } else {
            double mu[3];
            dipole<SYS, double>(sc, y, mu);
            f = mu[0] * mu[0] + mu[1] * mu[1] + mu[2] * mu[2];
        }
        const double diff = f - m;
        m += diff / (n + 1.0);
        q += diff * diff * (n / (n + 1.0));
        ++n;
    }
    acc.m[s] = m;
    acc.q[s] = q;
    acc.n[s] = n;
    acc.cand[s] = candidates;
    acc.pos[s] = mt.pos;
    if (!was_done && (n >= quota || candidates >= max_candidates)) atomicAdd(acc.finished, 1);
}

hipError_t run_m0(int sys, const SysConst& sc, const M0Params& p, uint32_t seed, long nstreams, long npoints,
                  uint32_t* state, const M0Acc& acc, int init, long long ticks, hipStream_t st, int order)
{
    const unsigned grid = (unsigned)((nstreams + 255) / 256);
    auto k = sys == SYS_HEAR ? (order == 2 ? m0_kernel<SYS_HEAR, 2> : m0_kernel<SYS_HEAR, 0>)
                             : (order == 2 ? m0_kernel<SYS_CO2AR, 2> : m0_kernel<SYS_CO2AR, 0>);
    hipLaunchKernelGGL(k, dim3(grid), dim3(256), 0, st, sc, p, seed, nstreams, npoints, state, acc, init, ticks);
    return hipGetLastError();
}

}  // namespace hh
