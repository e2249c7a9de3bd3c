// Row kernel of the batched engine: one trajectory per DPP row (16 lanes) of a wavefront.
//
// The lane kernel (pool_cf_kernel, one trajectory per lane) needs 64 trajectories per wavefront
// and thousands of wavefronts to pay for its stage arena: a stage reads its tableau row's columns
// from memory, so one right-hand side takes 2.3 us however few lanes hold a trajectory.  Small
// requests, and the last few thousand trajectories of large ones, are then a chain of memory round
// trips.  Here lane i of a row holds component i of the state: the 16 stage vectors are 16
// registers of every lane, a tableau row is one FMA per non-zero column for all components at
// once, and the independent parts of a right-hand side run side by side in the row's lanes (the
// angles' sines and cosines, the reciprocals, the radial slots of CO2-Ar, the site pairs of
// CH4-CO2), exchanged with DPP row broadcasts; for He-Ar and CO2-Ar every lane forms its own component of
// Hamilton's equations.  What is serial (the FP64 Legendre recurrence, the sums in their order, all of
// CH4-CO2's equations) runs in every lane of the row.
//
// Every expression is the lane kernel's, in its order, so a trajectory's row is the same bits
// whichever kernel integrates it, and the two share the slot format: a slice of a pool can run on
// either.  The rows of a grid hold the slots of ranks 0, 1, ... of a repacked pool.
//
// Bound: a lone wavefront's instruction issue (one in 4.4 cycles).  1153 CO2-Ar trajectories in FP64
// (L = 1024): 42 ms on the lane kernel, 21 ms with every lane evaluating both series of a sincos and
// all components, 18 ms in this form with the stages in a loop and 15 with them unrolled; 4096 He-Ar
// ones (L = 2048) 7.4, 4.4, 4.2 and 3.3 ms.
#include <hip/hip_runtime.h>

#include <utility>

#include "hh_integrate.h"

namespace hh {

typedef unsigned int rw_v2u __attribute__((ext_vector_type(2)));

constexpr int kRowBlock = 256;   // four wavefronts share the CO2-Ar tables in LDS

// the value of lane L of the caller's row (row_newbcast); every lane of the row takes part
template <int L>
__device__ __forceinline__ int bcast(int v)
{
    return __builtin_amdgcn_mov_dpp(v, 0x150 + L, 0xf, 0xf, true);
}
template <int L>
__device__ __forceinline__ float bcast(float v)
{
    return __builtin_bit_cast(float, bcast<L>(__builtin_bit_cast(int, v)));
}
template <int L>
__device__ __forceinline__ double bcast(double v)
{
    const rw_v2u u = __builtin_bit_cast(rw_v2u, v);
    return __builtin_bit_cast(double, rw_v2u{(unsigned)bcast<L>((int)u.x), (unsigned)bcast<L>((int)u.y)});
}
template <int L>
__device__ __forceinline__ long long bcast(long long v)
{
    return __builtin_bit_cast(long long, bcast<L>(__builtin_bit_cast(double, v)));
}

// the value of another lane of the row by a DPP control: within pairs (even lane's, odd lane's, the
// partner's) or two lanes down
enum RowMove : int { PAIR_EVEN = 0xa0, PAIR_ODD = 0xf5, PAIR_SWAP = 0xb1, QUAD_SWAP2 = 0x4e, HALF_MIRROR = 0x141, DOWN2 = 0x112 };
template <int CTRL>
__device__ __forceinline__ float row_move(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double row_move(double v)
{
    const rw_v2u u = __builtin_bit_cast(rw_v2u, v);
    return __builtin_bit_cast(double, rw_v2u{(unsigned)__builtin_amdgcn_mov_dpp((int)u.x, CTRL, 0xf, 0xf, true),
                                             (unsigned)__builtin_amdgcn_mov_dpp((int)u.y, CTRL, 0xf, 0xf, true)});
}

// slot_sum of lanes 0..5's values (lanes 6 and 7 hold 0, lanes 8..15 the same again), in every lane
template <typename P>
__device__ __forceinline__ P row_slot_sum(P t)
{
    t += row_move<PAIR_SWAP>(t);
    t += row_move<QUAD_SWAP2>(t);
    return t + row_move<HALF_MIRROR>(t);
}

// out[i] = lane i's value, i < N
template <typename T, int N, int... I>
__device__ __forceinline__ void gather_impl(T v, T (&out)[N], std::integer_sequence<int, I...>)
{
    ((out[I] = bcast<I>(v)), ...);
}
template <typename T, int N>
__device__ __forceinline__ void gather(T v, T (&out)[N])
{
    gather_impl<T, N>(v, out, std::make_integer_sequence<int, N>{});
}

// CH4-CO2: v[comp] by selects; the empty asm keeps the values in registers (the compiler would turn the
// selects into an indexed load of an array in scratch)
template <int N>
__device__ __forceinline__ double pick(const double (&v)[N], int comp)
{
    double r = v[0];
#pragma unroll
    for (int i = 1; i < N; ++i) {
        double x = v[i];
        __asm__("" : "+v"(x));
        r = comp == i ? x : r;
    }
    return r;
}

// What a lane keeps for the whole kernel: its component, the coefficients of its half of the sine and
// cosine (even lanes the sine's series, odd lanes the cosine's), for FP32 CO2-Ar its slot's Legendre
// recurrence (the steps past the slot's order repeat the value), for CH4-CO2 its site pair (lane l < 15:
// CO2 site l / 5, CH4 site l % 5).
template <int SYS, typename P>
struct RowCtx {
    int lane, comp;      // lane of the row; component (the last one again past QP)
    double w[8];         // FP64 series in r^2, highest order last
    float wf[5];         // FP32 series
    double kin;          // the lane's constant factor: 1/mu or 1/I
    P alpha[SYS == SYS_CO2AR && sizeof(P) == 4 ? 5 : 1], beta[SYS == SYS_CO2AR && sizeof(P) == 4 ? 5 : 1], gamma[SYS == SYS_CO2AR && sizeof(P) == 4 ? 5 : 1];
    P sgn, s2, e4, h0, h1, h2;
    P* scratch;          // CH4-CO2: the row's LDS scratch [5][16]
};

template <int SYS, typename P>
__device__ __forceinline__ RowCtx<SYS, P> row_ctx(const SysConst& sc, P* scratch)
{
    RowCtx<SYS, P> cx{};
    cx.lane = (int)(threadIdx.x & 15);
    cx.comp = min(cx.lane, SysTraits<SYS>::QP - 1);
    cx.scratch = scratch;
    const bool odd = cx.lane & 1;
    // the coefficients of sincos_p
    constexpr double ws[8] = {-1.0 / 6, 1.0 / 120, -1.0 / 5040, 1.0 / 362880, -1.0 / 39916800, 1.0 / 6227020800.0,
                              -1.0 / 1307674368000.0, 1.0 / 355687428096000.0};
    constexpr double wc[8] = {-0.5, 1.0 / 24, -1.0 / 720, 1.0 / 40320, -1.0 / 3628800, 1.0 / 479001600.0,
                              -1.0 / 87178291200.0, 1.0 / 20922789888000.0};
    constexpr float fs[5] = {-1.0f / 6, 1.0f / 120, -1.0f / 5040, 1.0f / 362880, 0.0f};
    constexpr float fc[5] = {-0.5f, 1.0f / 24, -1.0f / 720, 1.0f / 40320, -1.0f / 3628800};
#pragma unroll
    for (int i = 0; i < 8; ++i) cx.w[i] = odd ? wc[i] : ws[i];
#pragma unroll
    for (int i = 0; i < 5; ++i) cx.wf[i] = odd ? fc[i] : fs[i];
    cx.kin = cx.lane >= 6 ? sc.iI : sc.imu;
    if constexpr (SYS == SYS_CO2AR && sizeof(P) == 4) {
        const int slot = cx.lane & 7;
#pragma unroll
        for (int t = 0; t < 5; ++t) {
            const LegendreEven k = legendre_even_step(t);
            cx.alpha[t] = t < slot ? P(k.alpha) : P(0);
            cx.beta[t] = t < slot ? P(k.beta) : P(-1);
            cx.gamma[t] = t < slot ? P(k.gamma) : P(0);
        }
    }
    if constexpr (SYS == SYS_CH4CO2) {
        using namespace ch4co2;
        const int l = min(cx.lane, 14), j = l / 5, i = l % 5;
        const P hs = P(kRCH / 1.7320508075688772);
#pragma unroll
        for (int q = 0; q < 15; ++q) {
            // the lane kernel's compile-time constants, picked by lane
            const int jj = q / 5, ii = q % 5, tj = jj == 0 ? 2 : 3, ti = ii == 0 ? 0 : 1;
            const double sig = 0.5 * (kSigma[ti] + kSigma[tj]) * kAng;
            const P s2 = P(sig * sig);
            const P e4 = P(4.0 * kWellScale * kKelvinHartree) * (P)__builtin_sqrt(kEpsilon[ti] * kEpsilon[tj]);
            const P h0 = ii == 0 ? P(0) : hs * P(kH[ii == 0 ? 0 : ii - 1][0]);
            const P h1 = ii == 0 ? P(0) : hs * P(kH[ii == 0 ? 0 : ii - 1][1]);
            const P h2 = ii == 0 ? P(0) : hs * P(kH[ii == 0 ? 0 : ii - 1][2]);
            if (q == 5 * j + i) {
                cx.sgn = jj == 0 ? P(0) : (jj == 1 ? P(1) : P(-1));
                cx.s2 = s2;
                cx.e4 = e4;
                cx.h0 = h0;
                cx.h1 = h1;
                cx.h2 = h2;
            }
        }
    }
    return cx;
}

// sincos_p of an angle that both lanes of a pair hold: the even lane gets the sine, the odd lane the
// cosine
template <int SYS, typename P>
__device__ __forceinline__ void row_sincos(const RowCtx<SYS, P>& cx, const Reduced& red, double& v)
{
    const bool odd = cx.lane & 1;
    const double r2 = red.r * red.r;
    double w = cx.w[6] + r2 * cx.w[7];
#pragma unroll
    for (int i = 5; i >= 0; --i) w = cx.w[i] + r2 * w;
    const double base = odd ? 1.0 : red.r;   // sin: r + (r r2) w, cos: 1 + r2 w
    v = base + base * r2 * w;
    const double other = row_move<PAIR_SWAP>(v);
    v = (red.q & 1) ? other : v;
    rw_v2u u = __builtin_bit_cast(rw_v2u, v);
    u.y ^= (unsigned)((red.q + (odd ? 1 : 0)) & 2) << 30;
    v = __builtin_bit_cast(double, u);
}

template <int SYS, typename P>
__device__ __forceinline__ void row_sincos(const RowCtx<SYS, P>& cx, const Reduced& red, float& v)
{
    const bool odd = cx.lane & 1;
    const float r = (float)red.r, r2 = r * r;
    float w = cx.wf[3] + r2 * cx.wf[4];
#pragma unroll
    for (int i = 2; i >= 0; --i) w = cx.wf[i] + r2 * w;
    const float base = odd ? 1.0f : r;
    v = base + base * r2 * w;
    const float other = row_move<PAIR_SWAP>(v);
    v = (red.q & 1) ? other : v;
    v = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) ^ ((unsigned)((red.q + (odd ? 1 : 0)) & 2) << 30));
}

// ------------------------------------------------------------------ right-hand sides
// The component of Hamilton's equations of the calling lane; y: the lane's component of the
// state.  noise as in rhs().  Coordinates sit in the even lanes, their momenta in the odd ones; each
// branch follows rhs<SYS, P> expression by expression.
template <int SYS, typename P>
__device__ __forceinline__ double row_rhs(const SysConst& sc, const RowCtx<SYS, P>& cx, double y, double& noise)
{
    noise = 0.0;
    const int lane = cx.lane;
    const bool odd = lane & 1;
    double ang = row_move<PAIR_EVEN>(y);              // the pair's coordinate in both lanes
    const double p_next = row_move<PAIR_ODD>(y);      // and its momentum
    if constexpr (SYS == SYS_CO2AR && sizeof(P) == 4) {
        const double d = bcast<0>(y) - bcast<6>(y);   // Phi - phi1
        ang = lane < 2 ? d : ang;
    }
    const Reduced red = reduce_pio2(ang);
    double t;                                         // even lane: sine, odd lane: cosine
    row_sincos(cx, red, t);
    P tp;                                             // and in the surfaces' precision
    if constexpr (sizeof(P) == 8)
        tp = t;
    else
        row_sincos(cx, red, tp);
    const double R = bcast<4>(y);
    // reciprocals of the sines and, in lane 4, of R; in both lanes of a pair
    const double rc = row_move<PAIR_EVEN>(recip<P>(lane == 4 ? y : t));
    const double iR = bcast<4>(rc), is = bcast<2>(rc);
    const double is2 = is * is, a = sc.imu * (iR * iR);
    const double rad = radial_rate(bcast<1>(y), bcast<3>(y), is2, a);
    if constexpr (SYS == SYS_CH4CO2) {
        Ch4Co2Frame<P> f;
        const double sT = bcast<2>(t), cT = bcast<3>(t), s1 = bcast<8>(t), c1 = bcast<9>(t);
        const double sp = bcast<10>(t), cp = bcast<11>(t), s2 = bcast<14>(t), c2 = bcast<15>(t);
        f.sP = bcast<0>(tp), f.cP = bcast<1>(tp), f.sf = bcast<6>(tp), f.cf = bcast<7>(tp);
        f.sP2 = bcast<12>(tp), f.cP2 = bcast<13>(tp);
        f.sT = (P)sT, f.cT = (P)cT, f.s1 = (P)s1, f.c1 = (P)c1, f.sp = (P)sp, f.cp = (P)cp, f.s2 = (P)s2, f.c2 = (P)c2;
        ch4co2_axes<P>(f);
        const P Rp = (P)R;
        P gs[3], gd[3], mag = P(0);
        {
            // the lane's site pair
            using namespace ch4co2;
            const P sgn = cx.sgn;
            const P X[3] = {Rp * f.a[0] + sgn * P(kRCO) * f.b[0], Rp * f.a[1] + sgn * P(kRCO) * f.b[1],
                            Rp * f.a[2] + sgn * P(kRCO) * f.b[2]};
            const P d0 = X[0] - cx.h0, d1 = X[1] - cx.h1, d2 = X[2] - cx.h2;
            const P r2 = d0 * d0 + d1 * d1 + d2 * d2;
            const P ir2 = recip_p(r2);
            const P sr2 = cx.s2 * ir2, sr6 = sr2 * sr2 * sr2, sr12 = sr6 * sr6;
            const P w = cx.e4 * (P(-12) * sr12 + P(6) * sr6) * ir2;   // (dV/dr) / r
            P* sm = cx.scratch;
            sm[lane] = w;
            sm[16 + lane] = d0;
            sm[32 + lane] = d1;
            sm[48 + lane] = d2;
            if constexpr (sizeof(P) == 4) sm[64 + lane] = fabs(d0) + fabs(d1) + fabs(d2);
            wave_share_sync();
            // lane 3 j + k sums component k of CO2 site j over the five CH4 sites, in site order
            const int jk = min(lane, 8), j = jk / 3, k = jk - 3 * j;
            P g = P(0);
#pragma unroll
            for (int i = 0; i < 5; ++i) g += sm[5 * j + i] * sm[16 + 16 * k + 5 * j + i];
            if constexpr (sizeof(P) == 4) {
#pragma unroll
                for (int q = 0; q < 15; ++q) mag += fabs(sm[q]) * sm[64 + q];
            }
            wave_share_sync();
            P gj[9];
            gather<P, 9>(g, gj);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                gs[q] = P(0);
                gd[q] = P(0);
                gs[q] += gj[q];
                gd[q] += P(0);
                gs[q] += gj[3 + q];
                gd[q] += gj[3 + q];
                gs[q] += gj[6 + q];
                gd[q] += -gj[6 + q];
            }
        }
        double dV[8];
        ch4co2_gradient<P>(f, Rp, gs, gd, dV);
        noise = ch4co2_noise<P>(Rp, mag);
        double yd[16];
        yd[4] = bcast<5>(y) * sc.imu;
        yd[5] = rad * iR - dV[2];
        yd[0] = bcast<1>(y) * a * is2;
        yd[1] = -dV[0];
        yd[2] = bcast<3>(y) * a;
        yd[3] = polar_rate(bcast<1>(y), cT, a, is2, is, dV[1]);
        const double m[6] = {0.0, bcast<7>(y), 0.0, bcast<9>(y), 0.0, bcast<11>(y)};
        // the rotor's 1/sin(theta1) is FP64 in both precisions
        rotor_rhs(sc.IR, sc.iIR, m, dV + 3, s1, c1, sp, cp, sizeof(P) == 8 ? bcast<8>(rc) : recip<double>(s1), yd + 6);
        linear_rotor_eom(bcast<13>(y), bcast<15>(y), c2, sc.iI, bcast<14>(rc), dV[6], dV[7], yd + 12);
        return pick<16>(yd, cx.comp);
    } else {
        double dV;                                    // odd lanes: dV/dq of their coordinate
        double irot2 = 1.0;                           // CO2-Ar: 1/sin^2(theta1)
        if constexpr (SYS == SYS_HEAR) {
            const double x = kHearB * R;
            const double arg = lane == 0 ? -x : -kHearA1 * R - kHearA2 * R * R;
            const double ex = exp(arg);
            const double dVR = hear_dV_exps(R, bcast<0>(ex), bcast<1>(ex), sizeof(P) == 8 ? iR : recip<double>(R));
            dV = lane == 5 ? dVR : 0.0;
        } else {
            const Co2ArTables<P>* tb = (const Co2ArTables<P>*)sc.tables;
            // the lane's radial slot: value and derivative
            const int b = co2ar_branch<P>(tb, R);
            const int slot = min(lane & 7, 5);
            P v, dv;
            if (b == 0) {
                const P r = (P)R;
                const P e = tb->pes_exp[slot][0] * exp(tb->pes_exp[slot][1] * r);
                v = e;
                dv = tb->pes_exp[slot][1] * e;
            } else {
                const P x = (P)(R - tb->center[b]);
                slot_eval<P>(tb->pes[b][slot], x, (P)iR, v, dv);
            }
            const double sT = bcast<2>(t), cT = bcast<3>(t), st = bcast<8>(t), ct = bcast<9>(t);
            P dVdR, dVdc;
            Co2ArAngles<P> g;
            if constexpr (sizeof(P) == 8) {
                g = co2ar_angles<P>(bcast<0>(tp), bcast<1>(tp), sT, cT, bcast<6>(tp), bcast<7>(tp), st, ct);
                P Pl[11], dPl[11];
                legendre10<P>(g.c, Pl, dPl);
                P vs[6], dvs[6];
                gather<P, 6>(v, vs);
                gather<P, 6>(dv, dvs);
                dVdR = dVdc = P(0);
#pragma unroll
                for (int q = 0; q < 6; ++q) {
                    const P tR = dvs[q] * Pl[2 * q], tc = vs[q] * dPl[2 * q];
                    dVdR += tR;
                    dVdc += tc;
                }
            } else {
                g = co2ar_angles_difference<P>(bcast<0>(tp), bcast<1>(tp), (P)sT, (P)cT, (P)st, (P)ct);
                // the slot's Legendre polynomial and its derivative (lanes 6 and 7 of each half: 0)
                const P z = g.c * g.c;
                P p0 = P(0), p1 = (lane & 7) < 6 ? P(1) : P(0), d0 = P(0), d1 = P(0);
#pragma unroll
                for (int q = 0; q < 5; ++q) legendre_step<P>(cx.alpha[q], cx.beta[q], cx.gamma[q], z, p0, p1, d0, d1);
                const P tR = dv * p1, tc = v * d1;
                dVdR = row_slot_sum<P>(tR);
                const P c2 = g.c + g.c, ac2 = fabs(c2);
                dVdc = row_slot_sum<P>(tc) * c2;
                noise = kF32NoiseUnits * (double)row_slot_sum<P>(fabs(tc) * ac2 + fabs(tR));
            }
            P gl = lane == 3 ? g.dTheta : g.dPhi;
            gl = lane == 9 ? g.dtheta : gl;
            gl = lane == 7 ? g.dphi : gl;
            const double gq = (double)(dVdc * gl);
            dV = lane == 5 ? (double)dVdR : gq;
            const double ist = bcast<8>(rc);
            irot2 = ist * ist;
        }
        // even lanes: p a is2, p a, p / mu, p iI ist2, p iI; a factor 1 leaves the product as it is
        const double ka = lane < 4 ? a : cx.kin;
        double kb = lane == 0 ? is2 : 1.0;
        kb = lane == 6 ? irot2 : kb;
        const double coord = p_next * ka * kb;
        // odd lanes: lanes 3 and 9 polar_rate (azimuthal momentum two lanes down, own cosine), lane 5 the
        // radial rate; lanes 1 and 7 (a cyclic and a surface-driven azimuth) -dV, whatever the reciprocal of their
        // azimuth's sine is (at 0 a product with it is no number)
        const double pa = row_move<DOWN2>(y);
        const double i2 = lane == 3 ? is2 : irot2;
        const double pol = pa * pa * t * ka * i2;
        const double num = lane == 5 ? rad : pol;
        const double mul = lane == 5 ? iR : rc;
        double momentum = num * mul - dV;
        momentum = (lane == 1 || lane == 7) ? -dV : momentum;
        return odd ? momentum : coord;
    }
}

// ------------------------------------------------------------------ a row's trajectory
// y and K are the lane's component; everything else is the same in the 16 lanes of the row
struct RowItem {
    double y;
    double t, h, E0;
    double mx, my, mz;               // mu(0)
    double prev, curr;
    double dt, rtol, atol, Rcut;   // of the job, kept in registers
    double* row;
    long long local;
    int L, max_steps, record;
    int job, k, steps, total_steps, nrhs, reject, active;
};

__device__ __forceinline__ void row_job(const JobDesc& jb, RowItem& it)
{
    it.dt = jb.dt;
    it.rtol = jb.rtol;
    it.atol = jb.atol;
    it.Rcut = jb.Rcut;
    it.L = jb.L;
    it.max_steps = jb.max_steps;
    it.record = jb.record;
    it.row = jb.rows + it.local * (long long)jb.L * row_width(jb.record);
}

// finish_item of the lane kernel, by the row's first lane
__device__ __forceinline__ void row_finish(const JobDesc& jb, int lane, RowItem& it, int status, int last, float drift)
{
    if (lane == 0) {
        jb.len[it.local] = last + 1;
        jb.status[it.local] = status;
        if (jb.map) {
            jb.nrhs[it.local] += it.nrhs;
            atomicAdd(jb.orbit_nrhs, (unsigned long long)it.nrhs);
        } else
            jb.nrhs[it.local] = it.nrhs;
        jb.e_drift[it.local] = drift;
        if (jb.done) atomicAdd(jb.done, 1);
        if (jb.pool_done) atomicAdd(jb.pool_done, 1ull);
    }
    it.active = 0;
}

// sum over the components, in their order, of the squares of the lanes' values
template <int N>
__device__ __forceinline__ double sum_squares(double q)
{
    double v[N], acc = 0.0;
    gather<double, N>(q, v);
#pragma unroll
    for (int i = 0; i < N; ++i) acc += v[i] * v[i];
    return acc;
}

// The lane's stage values K0..K15, each a variable of its own: as an array they become one 32-register
// vector, which this compiler (ROCm 7.2) updates wrongly across the divergent branches of a step.
struct Stages {
    double k0, k1, k2, k3, k4, k5, k6, k7, k8, k9, k10, k11, k12, k13, k14, k15;
    template <int I>
    __device__ __forceinline__ double& at()
    {
        if constexpr (I == 0) return k0;
        else if constexpr (I == 1) return k1;
        else if constexpr (I == 2) return k2;
        else if constexpr (I == 3) return k3;
        else if constexpr (I == 4) return k4;
        else if constexpr (I == 5) return k5;
        else if constexpr (I == 6) return k6;
        else if constexpr (I == 7) return k7;
        else if constexpr (I == 8) return k8;
        else if constexpr (I == 9) return k9;
        else if constexpr (I == 10) return k10;
        else if constexpr (I == 11) return k11;
        else if constexpr (I == 12) return k12;
        else if constexpr (I == 13) return k13;
        else if constexpr (I == 14) return k14;
        else return k15;
    }
};

// tableau row R (its columns those of row C) applied to the lane's stage values, from column q on
template <int C, int R, int Q = 0>
__device__ __forceinline__ double stage_sum(Stages& K, double acc = 0.0)
{
    if constexpr (Q == DOP853_SP_NNZ[C]) {
        return acc;
    } else {
        acc += DOP853_SP_VAL[R][Q] * K.at<DOP853_SP_COL[C][Q]>();
        return stage_sum<C, R, Q + 1>(K, acc);
    }
}

__device__ __forceinline__ double stage_dot(Stages& K, int s)
{
    switch (s) {
    case 1: return stage_sum<1, 1>(K);
    case 2: return stage_sum<2, 2>(K);
    case 3: return stage_sum<3, 3>(K);
    case 4: return stage_sum<4, 4>(K);
    case 5: return stage_sum<5, 5>(K);
    case 6: return stage_sum<6, 6>(K);
    case 7: return stage_sum<7, 7>(K);
    case 8: return stage_sum<8, 8>(K);
    case 9: return stage_sum<9, 9>(K);
    case 10: return stage_sum<10, 10>(K);
    case 11: return stage_sum<11, 11>(K);
    case 12: return stage_sum<12, 12>(K);
    case 13: return stage_sum<13, 13>(K);
    case 14: return stage_sum<14, 14>(K);
    default: return stage_sum<15, 15>(K);
    }
}

template <int S0, int S1>
__device__ __forceinline__ void stage_store(Stages& K, int s, double k)
{
    K.at<S0>() = s == S0 ? k : K.at<S0>();
    if constexpr (S0 < S1) stage_store<S0 + 1, S1>(K, s, k);
}

// Stages S..S1: K_s = f(y + h sum_m A[s][m] K_m).  Unrolled, the tableau's columns and coefficients are
// immediates and no stage is selected at run time: 4096 He-Ar trajectories 4.2 -> 3.3 ms, 1153 FP64
// CO2-Ar ones 18.0 -> 15.2.  CH4-CO2's right-hand side is too long for that (15 copies of it leave the
// instruction cache: 12289 trajectories 108 -> 454 ms), so its stages run in a loop.
template <int SYS, typename P, int S, int S1>
__device__ __forceinline__ void row_stages(const SysConst& sc, const RowCtx<SYS, P>& cx, double y, double h, Stages& K,
                                           double& noise)
{
    if constexpr (SYS == SYS_CH4CO2) {
#pragma unroll 1
        for (int s = S; s <= S1; ++s) {
            double yt = stage_dot(K, s);
            yt = y + h * yt;
            double nz;
            const double k = row_rhs<SYS, P>(sc, cx, yt, nz);
            noise = fmax(noise, nz);
            stage_store<S, S1>(K, s, k);
        }
    } else {
        double yt = stage_sum<S, S>(K);
        yt = y + h * yt;
        double nz;
        K.at<S>() = row_rhs<SYS, P>(sc, cx, yt, nz);
        noise = fmax(noise, nz);
        if constexpr (S < S1) row_stages<SYS, P, S + 1, S1>(sc, cx, y, h, K, noise);
    }
}

// init_item of the lane kernel: the initial condition, mu(0), sample 0, H(0), f(y0), Hairer's HINIT
template <int SYS, typename P>
__device__ __forceinline__ bool row_init(const SysConst& sc, const RowCtx<SYS, P>& cx, const JobDesc& jb, int j,
                                         long long local, RowItem& it, Stages& K)
{
    constexpr int N = SysTraits<SYS>::QP;
    it.job = j;
    it.local = jb.map ? (long long)jb.map[local] : local;
    row_job(jb, it);
    const long long traj = it.local / jb.halves;
    const bool back = (it.local % jb.halves) == 1;
    const double v = jb.ic[(long long)cx.comp * jb.ntraj + traj];
    it.y = (back && (cx.comp & 1)) ? -v : v;
    double yv[N];
    gather<double, N>(it.y, yv);
    if constexpr (SYS == SYS_CH4CO2) {
        if (cx.lane < N && !(cx.lane & 1)) it.row[cx.lane >> 1] = it.y;
        it.mx = it.my = it.mz = 0.0;
    } else {
        P m[3];
        dipole<SYS, P>(sc, yv, m);
        it.mx = m[0];
        it.my = m[1];
        it.mz = m[2];
        if (cx.lane == 0) {
            if (it.record) {
                it.row[0] = it.mx;
                it.row[it.L] = it.my;
                it.row[2 * (long long)it.L] = it.mz;
            } else {
                it.row[0] = it.mx * it.mx + it.my * it.my + it.mz * it.mz;
            }
        }
    }
    it.E0 = hamiltonian<SYS, P>(sc, yv);
    it.t = 0.0;
    it.k = 1;
    it.steps = 0;
    it.total_steps = 0;
    it.reject = 0;
    it.nrhs = 0;
    it.prev = 0.0;
    it.curr = 0.0;
    it.active = 1;
    if (it.L <= 1) {
        row_finish(jb, cx.lane, it, ITEM_OK, 0, 0.0f);
        return false;
    }
    // Hairer's HINIT (initial_step)
    const double hmax = (it.L - 1) * it.dt;
    const double sk = it.atol + it.rtol * fabs(it.y);
    double y1 = it.y, h = 0.0, dnf = 0.0, nz;
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
        const double f = row_rhs<SYS, P>(sc, cx, y1, nz);
        if (pass == 0) {
            K.k0 = f;
            dnf = sum_squares<N>(f / sk);
            const double dny = sum_squares<N>(it.y / sk);
            h = (dnf <= 1e-10 || dny <= 1e-10) ? 1e-6 : sqrt(dny / dnf) * 0.01;
            h = fmin(h, hmax);
            y1 = it.y + h * f;
        } else {
            double der2 = sum_squares<N>((f - K.k0) / sk);
            der2 = sqrt(der2) / h;
            const double der12 = fmax(fabs(der2), sqrt(dnf));
            const double h1 = (der12 <= 1e-15) ? fmax(1e-6, fabs(h) * 1e-3) : sqrt(sqrt(sqrt(0.01 / der12)));
            h = fmin(fmin(100.0 * fabs(h), h1), hmax);
        }
    }
    it.nrhs = 2;
    it.h = h;
    return true;
}

// ------------------------------------------------------------------ samples
// The wavefront evaluates the pending samples of its four rows 64 at a time, as shared_samples of
// the lane kernel; the rows' step records lie in LDS.
template <int NQ>
struct RowShare {
    double rec[4][StepRecord<NQ>::SIZE];
    double last[4];
    int fail[4];
};

template <int SYS, typename P>
__device__ __forceinline__ void row_samples(const SysConst& sc, RowShare<SysTraits<SYS>::QP / 2>& ws, int n)
{
    constexpr int N = SysTraits<SYS>::QP, NQ = N / 2;
    using R = StepRecord<NQ>;
    const int lane = (int)__lane_id();
    const int n0 = __builtin_amdgcn_readlane(n, 0), n1 = __builtin_amdgcn_readlane(n, 16);
    const int n2 = __builtin_amdgcn_readlane(n, 32), n3 = __builtin_amdgcn_readlane(n, 48);
    const int p1 = n0, p2 = n0 + n1, p3 = p2 + n2, total = p3 + n3;
    if (total == 0) return;
    if (lane < 4) ws.fail[lane] = 0x7fffffff;
    wave_share_sync();
    double carry = 0.0;
#pragma unroll 1
    for (int base = 0; base < total; base += 64) {
        const int g = base + lane;
        const bool valid = g < total;
        int owner = 0, q = 0, k = 0, cnt = 0, record = 0;
        double curr = 0.0, prev_start = 0.0;
        double* row = nullptr;
        int rowL = 0;
        P m[3] = {P(0), P(0), P(0)};
        if (valid) {
            owner = g < p1 ? 0 : (g < p2 ? 1 : (g < p3 ? 2 : 3));
            const int first = owner == 0 ? 0 : (owner == 1 ? p1 : (owner == 2 ? p2 : p3));
            cnt = owner == 0 ? n0 : (owner == 1 ? n1 : (owner == 2 ? n2 : n3));
            q = g - first;
            const double* r = ws.rec[owner];
            k = (int)r[R::K0] + q;
            const double tk = k * r[R::DT];
            double ys[N];
#pragma unroll
            for (int i = 1; i < N; i += 2) ys[i] = 0.0;
            if (tk == r[R::TNEW]) {
#pragma unroll
                for (int c = 0; c < NQ; ++c) ys[2 * c] = r[R::YN + c];
            } else {
                const double x = sizeof(P) == 4 ? (tk - r[R::T]) * rcp_nr(r[R::H]) : (tk - r[R::T]) / r[R::H];
#pragma unroll
                for (int c = 0; c < NQ; ++c) {
                    const double* f = r + R::Y + 8 * c;
                    const double F[7] = {f[1], f[2], f[3], f[4], f[5], f[6], f[7]};
                    ys[2 * c] = dense_value(F, f[0], x);
                }
            }
            row = __builtin_bit_cast(double*, r[R::ROW]);
            rowL = (int)r[R::L];
            record = (int)r[R::RECORD];
            if constexpr (SYS == SYS_CH4CO2) {
#pragma unroll
                for (int c = 0; c < NQ; ++c) row[(long long)k * NQ + c] = ys[2 * c];
            } else {
                dipole<SYS, P>(sc, ys, m);
                const double mu0[3] = {r[R::MU0], r[R::MU0 + 1], r[R::MU0 + 2]};
                curr = cf_value<P>(mu0, m);
            }
            prev_start = r[R::CURR];
        }
        const double up = __shfl_up(curr, 1, 64);
        const double prev = q == 0 ? prev_start : (lane > 0 ? up : carry);
        carry = __shfl(curr, 63, 64);
        if (valid && SYS != SYS_CH4CO2) {
            const int st = sample_status<P>(m, curr, prev, k, record);
            if (st != ITEM_OK) atomicMin(&ws.fail[owner], (q << 3) | st);
        }
        wave_share_sync();
        if (valid) {
            if (SYS != SYS_CH4CO2 && q < (ws.fail[owner] >> 3)) store_sample<P>(row, rowL, record, k, m, curr);
            if (q == cnt - 1) ws.last[owner] = curr;
        }
    }
    wave_share_sync();
}

// One attempted DOP853 step of every row of the wavefront (dop853_attempt, dop853_step_shared and
// advance of the lane kernel)
template <int SYS, typename P>
__device__ __forceinline__ void row_step(const SysConst& sc, const RowCtx<SYS, P>& cx, const JobDesc* __restrict__ ring,
                                         RowItem& it, Stages& K, RowShare<SysTraits<SYS>::QP / 2>& ws)
{
    constexpr int N = SysTraits<SYS>::QP, NQ = N / 2;
    using R = StepRecord<NQ>;
    const int row = (int)(__lane_id() >> 4);
    double yn = 0.0, h = 0.0, fac11 = 0.0;
    int outcome = STEP_ENDED, n = 0;
    bool end = false;
    if (it.active) {
        const double tend = (it.L - 1) * it.dt;
        if (it.steps >= it.max_steps || ++it.total_steps > kMaxTotalSteps) {
            row_finish(ring[it.job], cx.lane, it, ITEM_FAIL_STEPS, it.k - 1, 0.0f);
        } else if (0.1 * fabs(it.h) <= fabs(it.t) * kEPS) {
            row_finish(ring[it.job], cx.lane, it, ITEM_FAIL_STEPSIZE, it.k - 1, 0.0f);
        } else {
            h = it.h;
            if (it.t + 1.01 * h - tend > 0.0) h = tend - it.t;
            double noise = 0.0;
            row_stages<SYS, P, 1, 12>(sc, cx, it.y, h, K, noise);
            it.nrhs += 12;
            const double be0 = stage_sum<DOP853_ROW_B, DOP853_ROW_B>(K), be1 = stage_sum<DOP853_ROW_B, DOP853_ROW_E5>(K);
            const double be2 = stage_sum<DOP853_ROW_B, DOP853_ROW_E3>(K);
            const double floor_p = fabs(h) * noise;
            yn = it.y + h * be0;
            const double sk = it.atol + it.rtol * fmax(fabs(it.y), fabs(yn)) + ((cx.comp & 1) ? floor_p : 0.0);
            const double isk = recip<P>(sk);
            double err = sum_squares<N>(divide<P>(be1, sk, isk));
            const double err2 = sum_squares<N>(divide<P>(be2, sk, isk));
            double deno = err + 0.01 * err2;
            if (deno <= 0.0) deno = 1.0;
            err = fabs(h) * err * sqrt(1.0 / (N * deno));
            fac11 = sqrt(sqrt(sqrt(err)));
            if (!(err == err) || !(h == h)) {
                row_finish(ring[it.job], cx.lane, it, ITEM_FAIL_STEPSIZE, it.k - 1, 0.0f);
            } else if (err > 1.0) {
                it.h = h / fmin(1.0 / 0.333, fac11 / 0.9);
                it.reject = 1;
                outcome = STEP_REJECTED;
            } else {
                ++it.steps;
                outcome = STEP_ACCEPTED;
                const double tnew = it.t + h;
                if (it.k < it.L && it.k * it.dt <= tnew) {
                    double nz_dense = 0.0;
                    row_stages<SYS, P, 13, 15>(sc, cx, it.y, h, K, nz_dense);
                    it.nrhs += 3;
                    double F[7];
                    const double dy = yn - it.y;
                    F[0] = dy;
                    F[1] = h * K.k0 - dy;
                    F[2] = 2.0 * dy - h * (K.k12 + K.k0);
                    F[3] = h * stage_sum<DOP853_ROW_D, DOP853_ROW_D>(K);
                    F[4] = h * stage_sum<DOP853_ROW_D, DOP853_ROW_D + 1>(K);
                    F[5] = h * stage_sum<DOP853_ROW_D, DOP853_ROW_D + 2>(K);
                    F[6] = h * stage_sum<DOP853_ROW_D, DOP853_ROW_D + 3>(K);
                    // the samples of the step, up to the one that ends the item
                    double FR[7];
#pragma unroll
                    for (int d = 0; d < 7; ++d) FR[d] = bcast<4>(F[d]);
                    const double R0 = bcast<4>(it.y), R1 = bcast<4>(yn);
                    double span = 0.0;
#pragma unroll
                    for (int d = 0; d < 7; ++d) span += fabs(FR[d]);
                    const double rmax = R0 + span * (1.0 + 1e-12) + 1e-12 * fabs(R0);
                    if (rmax < it.Rcut && R1 < it.Rcut) {
                        int kf = (int)fmin(floor(tnew / it.dt), (double)(it.L - 1));
                        while (kf + 1 <= it.L - 1 && (kf + 1) * it.dt <= tnew) ++kf;
                        while (kf > it.k && kf * it.dt > tnew) --kf;
                        n = kf - it.k + 1;
                        end = kf + 1 >= it.L;
                    } else {
                        for (int k = it.k; k < it.L && k * it.dt <= tnew; ++k) {
                            ++n;
                            const double tk = k * it.dt;
                            const double Rk = tk == tnew ? R1 : dense_value(FR, R0, (tk - it.t) / h);
                            if (Rk > it.Rcut || k + 1 >= it.L) {
                                end = true;
                                break;
                            }
                        }
                    }
                    double* r = ws.rec[row];
                    if (cx.lane < N && !(cx.lane & 1)) {
                        const int c = cx.lane >> 1;
                        r[R::YN + c] = yn;
                        r[R::Y + 8 * c] = it.y;
#pragma unroll
                        for (int d = 0; d < 7; ++d) r[R::Y + 8 * c + 1 + d] = F[d];
                    }
                    if (cx.lane == 1) {
                        r[R::T] = it.t;
                        r[R::H] = h;
                        r[R::TNEW] = tnew;
                        r[R::DT] = it.dt;
                        r[R::K0] = (double)it.k;
                    } else if (cx.lane == 3) {
                        r[R::MU0] = it.mx;
                        r[R::MU0 + 1] = it.my;
                        r[R::MU0 + 2] = it.mz;
                        r[R::CURR] = it.curr;
                        r[R::ROW] = __builtin_bit_cast(double, it.row);
                        r[R::L] = (double)it.L;
                        r[R::RECORD] = (double)it.record;
                    }
                }
            }
        }
    }
    row_samples<SYS, P>(sc, ws, n);
    if (outcome != STEP_ACCEPTED) return;
    if (n > 0) {
        const int f = ws.fail[row];
        if (f != 0x7fffffff) {
            row_finish(ring[it.job], cx.lane, it, f & 7, it.k + (f >> 3) - 1, 0.0f);
            return;
        }
        it.steps = 0;
        if (end) {
            double yv[N];
            gather<double, N>(yn, yv);
            const float drift = (float)fabs(hamiltonian<SYS, P>(sc, yv) - it.E0);
            row_finish(ring[it.job], cx.lane, it, ITEM_OK, it.k + n - 1, drift);
            return;
        }
        it.k += n;
        it.prev = it.curr;
        it.curr = ws.last[row];
    }
    if constexpr (sizeof(P) == 4) {
        if (bcast<5>(it.y) > 0.0 && bcast<5>(yn) <= 0.0) {
            const JobDesc& jb = ring[it.job];
            if (jb.orbit_items) {
                if (cx.lane == 0) {
                    const int at = atomicAdd(jb.orbit_count, 1);
                    jb.orbit_items[at] = (int)it.local;
                }
                row_finish(jb, cx.lane, it, ITEM_ORBIT, it.k - 1, 0.0f);
                return;
            }
        }
    }
    // advance: y <- y_new, f(y) <- K12 (first-same-as-last), the next step size
    const double tend = (it.L - 1) * it.dt;
    it.y = yn;
    K.k0 = K.k12;
    it.t = it.t + h;
    const double fac = fmax(1.0 / 6.0, fmin(1.0 / 0.333, fac11 / 0.9));
    double hnew = h / fac;
    if (fabs(hnew) > tend) hnew = tend;
    if (it.reject) {
        hnew = fmin(fabs(hnew), fabs(h));
        it.reject = 0;
    }
    it.h = hnew;
}

// ------------------------------------------------------------------ the kernel
// Row r of wavefront w of the grid holds the pool slot of rank r * (wavefronts) + w, so few
// trajectories spread one per wavefront; rank q is slot (q % W) * 64 + q / W of the pool's W
// wavefronts (repack_move_kernel).  Rows r < rows_used refill from the queue.
template <int SYS, typename P, int W>
__global__ void __launch_bounds__(kRowBlock, W) row_cf_kernel(SysConst sc, const JobDesc* __restrict__ ring, PoolCtl ctl,
                                                              LaneSlots sl, int rows_used)
{
    constexpr int N = SysTraits<SYS>::QP, NQ = N / 2;
    __shared__ Co2ArTables<P> s_tab;
    __shared__ RowShare<NQ> s_share[kRowBlock / 64];
    __shared__ P s_scratch[SYS == SYS_CH4CO2 ? kRowBlock / 16 : 1][5 * 16];
    const SysConst scl = stage_tables<SYS, P>(sc, &s_tab);
    const int wave = (int)(threadIdx.x >> 6);
    RowShare<NQ>& share = s_share[wave];
    const RowCtx<SYS, P> cx = row_ctx<SYS, P>(scl, s_scratch[SYS == SYS_CH4CO2 ? threadIdx.x >> 4 : 0]);
    const int row = (int)((threadIdx.x & 63) >> 4);
    const long long waves = (long long)gridDim.x * (kRowBlock / 64);
    const long long rank = row * waves + (long long)blockIdx.x * (kRowBlock / 64) + wave;
    const long long S = sl.S, W64 = S / 64;
    const long long slot = (rank % W64) * 64 + rank / W64;
    const bool mine = rank < S;
    const long long t_end = wall_clock64() + ctl.ticks;
    RowItem it{};
    Stages K{};
    it.job = mine ? sl.i[slot] : -1;
    it.active = it.job >= 0;
    if (it.active) {
        it.y = sl.d[cx.comp * S + slot];
        K.k0 = sl.d[(N + cx.comp) * S + slot];
        const double* d = sl.d + 2 * N * S + slot;
        it.t = d[0];
        it.h = d[S];
        it.E0 = d[2 * S];
        it.mx = d[3 * S];
        it.my = d[4 * S];
        it.mz = d[5 * S];
        it.prev = d[6 * S];
        it.curr = d[7 * S];
        it.k = sl.i[S + slot];
        it.steps = sl.i[2 * S + slot];
        it.total_steps = sl.i[3 * S + slot];
        it.nrhs = sl.i[4 * S + slot];
        it.reject = sl.i[5 * S + slot];
        it.local = sl.local[slot];
        row_job(ring[it.job], it);
    }
    bool queue_open = mine && row < rows_used;
    for (;;) {
        if (wall_clock64() >= t_end) break;
        if (!it.active && queue_open) {
            bool got = false;
            while (!got) {
                long long g = -1;
                if (cx.lane == 0 &&
                    __hip_atomic_load(ctl.next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < ctl.total)
                    g = (long long)atomicAdd(ctl.next, 1ull);
                g = bcast<0>(g);
                if (g < 0 || (unsigned long long)g >= ctl.total) break;
                int j = ring_job(ring, ctl, (unsigned long long)g);
                unsigned long long item = (unsigned long long)g;
                if (ring[j].order) {
                    item = (unsigned long long)(ring[j].order_base + ring[j].order[g - ring[j].order_base]);
                    j = ring_job(ring, ctl, item);
                }
                got = row_init<SYS, P>(scl, cx, ring[j], j, (long long)item - ring[j].item_begin, it, K);
            }
            queue_open = got;
        }
        if (__ballot(it.active) == 0) break;
        row_step<SYS, P>(scl, cx, ring, it, K, share);
    }
    if (!mine) return;
    if (!it.active) {
        if (cx.lane == 0) sl.i[slot] = -1;
        return;
    }
    if (cx.lane < N) {
        sl.d[cx.comp * S + slot] = it.y;
        sl.d[(N + cx.comp) * S + slot] = K.k0;
    }
    if (cx.lane == 0) {
        double* d = sl.d + 2 * N * S + slot;
        d[0] = it.t;
        d[S] = it.h;
        d[2 * S] = it.E0;
        d[3 * S] = it.mx;
        d[4 * S] = it.my;
        d[5 * S] = it.mz;
        d[6 * S] = it.prev;
        d[7 * S] = it.curr;
        sl.i[slot] = it.job;
        sl.i[S + slot] = it.k;
        sl.i[2 * S + slot] = it.steps;
        sl.i[3 * S + slot] = it.total_steps;
        sl.i[4 * S + slot] = it.nrhs;
        sl.i[5 * S + slot] = it.reject;
        sl.local[slot] = it.local;
    }
}

template <int SYS, typename P, int W>
static hipError_t launch_rows(const SysConst& sc, const JobDesc* ring, const PoolCtl& ctl, const LaneSlots& sl, int wgs,
                              int rows_used, hipStream_t st)
{
    hipLaunchKernelGGL((row_cf_kernel<SYS, P, W>), dim3((unsigned)wgs), dim3(kRowBlock), 0, st, sc, ring, ctl, sl,
                       rows_used);
    return hipGetLastError();
}

// one slice of a pool on the row kernel: wgs workgroups of 16 rows, rows_used rows of a wavefront
// take new items; the pool's live slots are ranks below 16 wgs
hipError_t run_rows(int sys, bool mixed, const SysConst& sc, const JobDesc* ring, const PoolCtl& ctl, const LaneSlots& sl,
                    int wgs, int rows_used, hipStream_t st)
{
    if (wgs < 1 || rows_used < 1 || rows_used > 4) return hipErrorInvalidValue;
    if (sys == SYS_CH4CO2)
        return mixed ? launch_rows<SYS_CH4CO2, float, 2>(sc, ring, ctl, sl, wgs, rows_used, st)
                     : launch_rows<SYS_CH4CO2, double, 2>(sc, ring, ctl, sl, wgs, rows_used, st);
    if (sys == SYS_HEAR)
        return mixed ? launch_rows<SYS_HEAR, float, 2>(sc, ring, ctl, sl, wgs, rows_used, st)
                     : launch_rows<SYS_HEAR, double, 2>(sc, ring, ctl, sl, wgs, rows_used, st);
    return mixed ? launch_rows<SYS_CO2AR, float, 2>(sc, ring, ctl, sl, wgs, rows_used, st)
                 : launch_rows<SYS_CO2AR, double, 2>(sc, ring, ctl, sl, wgs, rows_used, st);
}

}  // namespace hh
