// Device code shared by the integrator kernels: one trajectory per lane (hh_kernels.hip) and one
// trajectory per 16-lane row (hh_rows.hip).  Both are compiled with FP contraction inside
// expressions only, so an expression written here is the same instructions in both and a
// trajectory's row is the same bits whichever kernel integrates it.
#pragma once
#include <hip/hip_runtime.h>

#include "dop853_coeffs.h"
#include "hh_engine.h"
#include "hh_systems.h"

namespace hh {

constexpr double kEPS = 2.220446049250313e-16;
constexpr int kMaxTotalSteps = 400000;   // attempts per item; the longest CO2-Ar items take ~6e3

// Dense output of coordinate c (state index 2c) at x = (t_k - t) / h of an accepted step:
// DOP853's 7th-order continuous extension (Hairer's contd8) in Horner form.
__device__ __forceinline__ double dense_value(const double (&F)[7], double y0, double x)
{
    const double omx = 1.0 - x;
    double v = F[5] + x * F[6];
    v = F[4] + omx * v;
    v = F[3] + x * v;
    v = F[2] + omx * v;
    v = F[1] + x * v;
    v = F[0] + omx * v;
    return y0 + x * v;
}

// CF value mu(0) . mu(t_k) of a sample
template <typename P>
__device__ __forceinline__ double cf_value(const double* mu0, const P (&m)[3])
{
    return mu0[0] * (double)m[0] + mu0[1] * (double)m[1] + mu0[2] * (double)m[2];
}

// Checks of one sample in the reference's order (src/hawaii.c:2181-2236): a NaN dipole, a
// huge CF value, a jump by more than 1e10 from the previous sample (from sample 2 on).  A
// PR/mu series (record 2) has no check that ends it: the reference skips a sample whose dipole
// is NaN and integrates on (src/hawaii.c:3664-3677), leaving that sample of its zeroed series at
// 0 (store_sample).
template <typename P>
__device__ __forceinline__ int sample_status(const P (&m)[3], double curr, double prev, int k, int record)
{
    if (record == 2) return ITEM_OK;
    if (isnan((double)m[0]) || isnan((double)m[1]) || isnan((double)m[2])) return ITEM_FAIL_DIPOLE_NAN;
    if (fabs(curr) > 1e100) return ITEM_FAIL_CF_HUGE;
    if (k > 1 && fabs(curr / prev) > 1e10) return ITEM_FAIL_CF_JUMP;
    return ITEM_OK;
}

// sample k of an item whose row starts at `row`: mu(0) . mu(t_k), or the three dipole
// components (rows [3][L]) when the job records the series
template <typename P>
__device__ __forceinline__ void store_sample(double* row, int L, int record, int k, const P (&m)[3], double curr)
{
    if (record) {
        const bool skip = record == 2 && (isnan((double)m[0]) || isnan((double)m[1]) || isnan((double)m[2]));
        row[k] = skip ? 0.0 : (double)m[0];
        row[L + k] = skip ? 0.0 : (double)m[1];
        row[2 * (long long)L + k] = skip ? 0.0 : (double)m[2];
    } else {
        row[k] = curr;
    }
}

enum StepOutcome : int { STEP_ENDED = 0, STEP_REJECTED = 1, STEP_ACCEPTED = 2 };

// Fields of a lane's step record (field f at arena slot 1 + f / N, component f % N), in pairs
// that one 16-byte access moves: the sample-time scalars [0, CF0), the CF scalars [CF0, YN),
// the coordinates at the step's end (used only for a sample at exactly t + h), then per
// coordinate c its value at the step's start followed by its seven dense-output coefficients
// (Y + 8c .. Y + 8c + 7).
template <int NQ>
struct StepRecord {
    static constexpr int T = 0, H = 1, TNEW = 2, DT = 3, K0 = 4, CF0 = 6, MU0 = 6, CURR = 9, ROW = 10, L = 11,
                         RECORD = 12, YN = 14, Y = YN + (NQ + 1) / 2 * 2, SIZE = Y + 8 * NQ;
};

// Memory written by one lane (LDS, the wavefront's arena block) is visible to the others
// after this; every lane of the wavefront executes it.  A wavefront's own memory operations
// are performed in order and its lanes share one vector L1, so the wavefront-scope fence only
// keeps the compiler from moving accesses across it (it emits no wait).
__device__ __forceinline__ void wave_share_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// CO2-Ar surface tables are staged into LDS once per workgroup: every right-hand side reads
// 6 Legendre slots x 8 coefficients at a lane-dependent radial branch.
template <int SYS, typename P>
__device__ __forceinline__ SysConst stage_tables(const SysConst& sc, Co2ArTables<P>* s_tab)
{
    SysConst out = sc;
    if constexpr (SYS == SYS_CO2AR) {
        const double* src = (const double*)sc.tables;
        double* dst = (double*)s_tab;
        for (unsigned i = threadIdx.x; i < sizeof(Co2ArTables<P>) / sizeof(double); i += blockDim.x) dst[i] = src[i];
        __syncthreads();
        out.tables = s_tab;
    }
    return out;
}

// ring slot of the job holding global item g: jobs [first_seq, last_seq] are in flight, their
// item ranges are consecutive and increasing with the sequence number
__device__ __forceinline__ int ring_job(const JobDesc* __restrict__ ring, const PoolCtl& c, unsigned long long g)
{
    long long lo = c.first_seq, hi = c.last_seq;
    while (lo < hi) {
        const long long mid = (lo + hi + 1) >> 1;
        if ((long long)g >= ring[mid % c.ring].item_begin)
            lo = mid;
        else
            hi = mid - 1;
    }
    return (int)(lo % c.ring);
}

}  // namespace hh
