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
// The packed sequence of 2n complex values goes through radix-2 Stockham stages, up to eleven of them in a
// pass over global memory, three at a time in registers with eight points per thread: one pass up to
// n = 1024, two up to n = 2^21, with the packing in the first one's loads and the scaling, nu and the
// apodized cf in the last one's stores.
//
// The butterflies and their roots are those of a transform that runs a stage at a time, bit for bit.  A
// transform of n points (the packed sequence is Hermitian) with radix-8 butterflies needs half of the time
// in the kernels at n = 2^20 and 2 us less of a call at n = 4096, with an error in the 2-norm that is the same
// within a tenth, 1.8e-16 to 2.8e-16 from n = 2^10 to 2^20; but where a long CF's peak is hundreds of times
// the spectrum's root mean square, the peak's roundings decide the far wing, and two such transforms
// differ there by up to 1e-13 of the root mean square.
//
// Bound by the butterflies' sincospi and the latency of the passes.  Kernels of a call, with a pass per stage
// (or one workgroup for all of them at n = 4096) before and now: n = 2^20 245 and 58 us, n = 4096 65 and
// 15 us.
constexpr int kFftPassLog = 11;     // stages of a pass: up to 4096 points in two or more columns, 512 threads, 72 KiB

constexpr double kLightSpeed_cm = 2.99792458e10, kATU = 2.4188843265857e-17;
constexpr double kADIPMOMU = 8.4783536255e-30, kEPSILON0 = 8.8541878128e-12;
constexpr double kSfXscale = 1.0 / kLightSpeed_cm / kATU / 2.0 / kPI;
constexpr double kSfYscale = kATU * kADIPMOMU * kADIPMOMU / (4.0 * kPI * kEPSILON0);

// nu_k, and the Connes apodization of the input in place, as the reference does (src/hawaii.c:5581): for
// the last pass, when nobody reads cf any more
__device__ __forceinline__ void sf_axis(double* cf, double* nu, long k, double dt, double tmax, double itmax)
{
    const double r = divide<double>(dt * k, tmax, itmax);
    cf[k] *= (1.0 - r * r) * (1.0 - r * r);
    nu[k] = divide<double>(k * kPI, tmax, itmax) * kSfXscale;
}

// One radix-2 butterfly with the root e^{i pi k/half}: a + w b, a - w b
__device__ __forceinline__ void butterfly(double2& a, double2& b, double k_over_half)
{
    double s, c;
    sincospi(k_over_half, &s, &c);
    const double2 wb = make_double2(b.x * c - b.y * s, b.x * s + b.y * c);
    const double2 u = a;
    a = make_double2(u.x + wb.x, u.y + wb.y);
    b = make_double2(u.x - wb.x, u.y - wb.y);
}

// logr radix-2 Stockham stages over M = 2n = 2^logm points, after logl of them, for the 2^logc columns of this
// workgroup: column j holds in[j + q M/R], R = 2^logr; its outputs are out[g L R + k0 + p L], L = 2^logl,
// k0 = j % L, g = j / L.  A thread holds rows q = b + i R/8.
template <bool FIRST, bool LAST>
__global__ void __launch_bounds__(512) sf_stages_kernel(double* cf, const double2* __restrict__ in,
                                                        double2* __restrict__ out, double* __restrict__ nu,
                                                        double* __restrict__ sf, int logm, double dt, int logr, int logl,
                                                        int logc)
{
    extern __shared__ double2 sm[];
    const long M = 1L << logm, n = M >> 1, L = 1L << logl;
    const int t = threadIdx.x, c = t & ((1 << logc) - 1), b = t >> logc, eighth = 1 << (logr - 3);
    const int logcols = logm - logr;
    // Workgroups go to the eight XCDs in turn: neighbouring tiles, which share cache lines, go to one
    const long tile = gridDim.x % 8 ? blockIdx.x : (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
    const long j = (tile << logc) + c, k0 = j & (L - 1);
    auto slot = [&](int q) { return ((q + (q >> 3)) << logc) + c; };
    const double tmax = dt * n;

    double2 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const long k = j + ((long)(b + i * eighth) << logcols);
        if constexpr (FIRST) {
            // the packed sequence: v_k e^{i pi k/2n}, 0 at n, -v_{2n-k} e^{i pi k/2n}
            const double inv2n = 1.0 / (2.0 * n);
            const long kk = k < n ? k : 2 * n - k;
            const double tc = dt * kk, r = tc / tmax;
            double x = 0.0;
            if (k != n) x = cf[kk] * ((1.0 - r * r) * (1.0 - r * r));
            if (k > n) x = -x;
            double sn, cs;
            sincospi((double)k / (2.0 * n), &sn, &cs);
            v[i] = make_double2(x * cs * inv2n, x * sn * inv2n);
        } else {
            v[i] = in[k];
        }
    }

    // a stage over the pairs of local position k' with `half` = 2^lg local, L 2^lg global: root (k0 + k' L) / (L 2^lg)
    auto root = [&](int kp, int lg) { return (double)(k0 + ((long)kp << logl)) * (1.0 / (double)(L << lg)); };
    for (int lg = 0;;) {
        const int rest = logr - lg;
        if (rest >= 3) {
            const int k = b & ((1 << lg) - 1), l = 1 << lg;
            const double ra = root(k, lg), rb0 = root(k, lg + 1), rb1 = root(k + l, lg + 1);
#pragma unroll
            for (int i = 0; i < 4; ++i) butterfly(v[i], v[i + 4], ra);
            // v[i]: first output of pair i, v[i + 4]: second (k' + l)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                butterfly(v[i], v[i + 2], rb0);
                butterfly(v[i + 4], v[i + 6], rb1);
            }
            butterfly(v[0], v[1], root(k, lg + 2));
            butterfly(v[4], v[5], root(k + l, lg + 2));
            butterfly(v[2], v[3], root(k + 2 * l, lg + 2));
            butterfly(v[6], v[7], root(k + 3 * l, lg + 2));
            // output s = u + 2 w + 4 x is at v[4 u + 2 w + x]
            double2 o[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) o[s] = v[4 * (s & 1) + 2 * ((s >> 1) & 1) + (s >> 2)];
#pragma unroll
            for (int s = 0; s < 8; ++s) v[s] = o[s];
            if (rest == 3) break;
        } else {
            if (rest == 2) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int k = b + u * eighth, l = 1 << lg;
                    double2 &e0 = v[u], &e1 = v[2 + u], &e2 = v[4 + u], &e3 = v[6 + u];
                    const double ra = root(k, lg);
                    butterfly(e0, e2, ra);
                    butterfly(e1, e3, ra);
                    butterfly(e0, e1, root(k, lg + 1));
                    butterfly(e2, e3, root(k + l, lg + 1));
                    const double2 x = e1;   // outputs 0, 2, 1, 3
                    e1 = e2;
                    e2 = x;
                }
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u) butterfly(v[u], v[4 + u], root(b + u * eighth, lg));
            }
            break;
        }
        const int k = b & ((1 << lg) - 1), g = b >> lg;
        if (lg) __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; ++i) sm[slot((g << (lg + 3)) + k + (i << lg))] = v[i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = sm[slot(b + i * eighth)];
        lg += 3;
    }

    if constexpr (!LAST) {
        const long o = ((j >> logl) << (logl + logr)) + k0;
#pragma unroll
        for (int i = 0; i < 8; ++i) out[o + ((long)(b + i * eighth) << logl)] = v[i];
    } else {
        const double tm = n * dt;
#pragma unroll
        for (int i = 0; i < 4; ++i)   // the first n outputs: rows below R/2
            sf[k0 + ((long)(b + i * eighth) << logl)] = v[i].x * tm / kPI * kSfYscale;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            sf_axis(cf, nu, ((long)blockIdx.x * 4 + i) * blockDim.x + t, dt, tm, recip<double>(tm));
    }
}

// n = 2: the cosine sum itself
__global__ void __launch_bounds__(64) sf_direct_kernel(double* cf, double* __restrict__ nu, double* __restrict__ sf,
                                                       double dt)
{
    const int j = threadIdx.x;
    const double x0 = cf[0], x1 = cf[1] * (0.75 * 0.75);   // the window at r = 0, 1/2
    __syncthreads();
    if (j >= 2) return;
    const double tmax = 2 * dt, c = 2.0 * x1 * cospi(0.25 * (2 * j + 1));
    sf[j] = 0.25 * (x0 + c) * tmax / kPI * kSfYscale;
    sf_axis(cf, nu, j, dt, tmax, recip<double>(tmax));
}

// Passes of the 2^logm-point transform: as many as it takes at 2^kFftPassLog points each
int sf_passes(int logm) { return (logm + kFftPassLog - 1) / kFftPassLog; }

int sf_log(long m)
{
    int l = 0;
    while ((1L << l) < m) ++l;
    return l;
}

size_t sf_work_bytes(long n, int which)
{
    return sf_passes(sf_log(2 * n)) > 1 + which ? (size_t)(2 * n) * sizeof(double2) : 0;
}

hipError_t run_cf_to_sf(double* cf, long n, double dt, double2* work_a, double2* work_b, double* nu, double* sf,
                        hipStream_t st)
{
    if (n == 2) {
        hipLaunchKernelGGL(sf_direct_kernel, dim3(1), dim3(64), 0, st, cf, nu, sf, dt);
        return hipGetLastError();
    }
    const int logm = sf_log(2 * n), passes = sf_passes(logm);
    double2 *src = work_b, *dst = work_a;
    int logl = 0;
    for (int p = 0; p < passes; ++p) {
        const int logr = (logm - logl + passes - p - 1) / (passes - p);
        // Columns of a workgroup.  512 threads hold two at eleven stages; with fewer stages 1, 2, 4, 8 and 16 columns
        // take 17.5, 17.7, 16.7, 16.5 and 17.3 us at n = 2^12, 33, 29, 31, 34 and 34 at 2^18, 412, 259, 220, 199
        // and 205 at 2^22
        const int logc = passes == 1 ? 0 : (logr == kFftPassLog ? 1 : 2);
        const bool first = p == 0, last = p == passes - 1;
        auto k = first ? (last ? sf_stages_kernel<true, true> : sf_stages_kernel<true, false>)
                       : (last ? sf_stages_kernel<false, true> : sf_stages_kernel<false, false>);
        const int points = 1 << (logr + logc);
        const size_t lds = (size_t)(points + points / 8) * sizeof(double2);
        if (lds > 65536) {
            const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(k, dim3((unsigned)(2 * n >> (logr + logc))), dim3(points / 8), lds, st, cf, src, dst, nu, sf,
                           logm, dt, logr, logl, logc);
        logl += logr;
        double2* x = src;
        src = dst;
        dst = x;
    }
    return hipGetLastError();
}

// ------------------------------------------------------------------ CF -> SF without allocation
// The 2n-point work sequence of the transform lives in a file-scope device array instead of an
// engine-allocated buffer, for callers that cannot allocate (graph capture, tight serving loops).
// Every device holds its own copy; its address comes from hipGetSymbolAddress once per device
// (noalloc_scratch_address, at engine creation) and only that address is passed to kernels: the
// array's name in host code is a host-side stand-in, not a device address.  Calls that overlap on
// one device share the array and race.
__device__ __align__(256) double2 scratch[2 * kCfToSfNoAllocMaxN];

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
