// Generated by hawaiihybrid_amd/data/gen_pip_n2ar.py -- do not edit.
// Permutation-invariant polynomial bases of the N2-Ar PIP-NN surfaces, evaluated in
// blocks of 16 (the k-blocks of the first network layer).  Each polynomial is the orbit
// sum of one monomial of the distance variables y under the basis' permutation group;
// the order is the reference's (PES-IDS/c_basis_2_1_4_purify.cc:3-24; dipole bases
// PES-IDS/c_basis_1_1_2_1_3_purify.cc, c_basis_2_1_1_1_3_purify.cc,
// c_basis_2_2_1_3_purify.cc concatenated as PES-IDS/ai_ids_n2_ar_pip_nn.cpp:41-48).
#pragma once
#include <hip/hip_runtime.h>

#define HH_PIP_FN __host__ __device__ __forceinline__

namespace hh {

HH_PIP_FN float pip_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
HH_PIP_FN double pip_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }

constexpr int kPipPes = 17;
constexpr int kPipDip = 308;

// 17 polynomials in 2 blocks of 16 (zero-padded)
template <typename T>
HH_PIP_FN void pip_n2ar_pes_block(int kb, const T* __restrict__ y, T* __restrict__ p)
{
    switch (kb) {
    case 0:
        p[0] = y[1] + y[2];
        p[1] = y[1]*y[2];
        p[2] = y[0]*y[1] + y[0]*y[2];
        p[3] = y[1]*y[1] + y[2]*y[2];
        p[4] = y[0]*y[1]*y[2];
        p[5] = y[1]*y[1]*y[2] + y[1]*y[2]*y[2];
        p[6] = y[0]*y[1]*y[1] + y[0]*y[2]*y[2];
        p[7] = y[0]*y[0]*y[1] + y[0]*y[0]*y[2];
        p[8] = y[1]*y[1]*y[1] + y[2]*y[2]*y[2];
        p[9] = y[0]*y[1]*y[1]*y[2] + y[0]*y[1]*y[2]*y[2];
        p[10] = y[0]*y[0]*y[1]*y[2];
        p[11] = y[1]*y[1]*y[2]*y[2];
        p[12] = y[1]*y[1]*y[1]*y[2] + y[1]*y[2]*y[2]*y[2];
        p[13] = y[0]*y[1]*y[1]*y[1] + y[0]*y[2]*y[2]*y[2];
        p[14] = y[0]*y[0]*y[1]*y[1] + y[0]*y[0]*y[2]*y[2];
        p[15] = y[0]*y[0]*y[0]*y[1] + y[0]*y[0]*y[0]*y[2];
        break;
    case 1:
        p[0] = y[1]*y[1]*y[1]*y[1] + y[2]*y[2]*y[2]*y[2];
        p[1] = T(0);
        p[2] = T(0);
        p[3] = T(0);
        p[4] = T(0);
        p[5] = T(0);
        p[6] = T(0);
        p[7] = T(0);
        p[8] = T(0);
        p[9] = T(0);
        p[10] = T(0);
        p[11] = T(0);
        p[12] = T(0);
        p[13] = T(0);
        p[14] = T(0);
        p[15] = T(0);
        break;
    default:
        break;
    }
}

// 308 polynomials in 20 blocks of 16 (zero-padded)
template <typename T>
HH_PIP_FN void pip_n2ar_dip_block(int kb, const T* __restrict__ y, T* __restrict__ p)
{
    switch (kb) {
    case 0:
        p[0] = T(0);
        p[1] = y[8] + y[9];
        p[2] = y[6];
        p[3] = y[3];
        p[4] = y[8]*y[9];
        p[5] = pip_fma(y[7], y[9], y[7]*y[8]);
        p[6] = pip_fma(y[6], y[9], y[6]*y[8]);
        p[7] = y[6]*y[7];
        p[8] = pip_fma(y[4], y[9], y[5]*y[8]);
        p[9] = pip_fma(y[5], y[9], y[4]*y[8]);
        p[10] = pip_fma(y[4], y[6], y[5]*y[6]);
        p[11] = pip_fma(y[3], y[9], y[3]*y[8]);
        p[12] = y[3]*y[7];
        p[13] = y[3]*y[6];
        p[14] = pip_fma(y[3], y[5], y[3]*y[4]);
        p[15] = pip_fma(y[1], y[9], y[2]*y[8]);
        break;
    case 1:
        p[0] = pip_fma(y[2], y[9], y[1]*y[8]);
        p[1] = pip_fma(y[1], y[6], y[2]*y[6]);
        p[2] = pip_fma(y[2], y[3], y[1]*y[3]);
        p[3] = pip_fma(y[0], y[9], y[0]*y[8]);
        p[4] = y[0]*y[6];
        p[5] = y[0]*y[3];
        p[6] = pip_fma(y[9], y[9], y[8]*y[8]);
        p[7] = y[6]*y[6];
        p[8] = y[3]*y[3];
        p[9] = y[7]*y[8]*y[9];
        p[10] = y[6]*y[8]*y[9];
        p[11] = pip_fma(y[6]*y[7], y[8], y[6]*y[7]*y[9]);
        p[12] = pip_fma(y[4]*y[8], y[9], y[5]*y[8]*y[9]);
        p[13] = pip_fma(y[4]*y[7], y[9], y[5]*y[7]*y[8]);
        p[14] = pip_fma(y[4]*y[7], y[8], y[5]*y[7]*y[9]);
        p[15] = pip_fma(y[4]*y[6], y[9], y[5]*y[6]*y[8]);
        break;
    case 2:
        p[0] = pip_fma(y[4]*y[6], y[8], y[5]*y[6]*y[9]);
        p[1] = pip_fma(y[4]*y[6], y[7], y[5]*y[6]*y[7]);
        p[2] = pip_fma(y[4]*y[5], y[8], y[4]*y[5]*y[9]);
        p[3] = y[4]*y[5]*y[6];
        p[4] = y[3]*y[8]*y[9];
        p[5] = pip_fma(y[3]*y[7], y[8], y[3]*y[7]*y[9]);
        p[6] = pip_fma(y[3]*y[6], y[8], y[3]*y[6]*y[9]);
        p[7] = y[3]*y[6]*y[7];
        p[8] = pip_fma(y[3]*y[4], y[9], y[3]*y[5]*y[8]);
        p[9] = pip_fma(y[3]*y[4], y[8], y[3]*y[5]*y[9]);
        p[10] = pip_fma(y[3]*y[4], y[7], y[3]*y[5]*y[7]);
        p[11] = pip_fma(y[3]*y[4], y[6], y[3]*y[5]*y[6]);
        p[12] = y[3]*y[4]*y[5];
        p[13] = pip_fma(y[1]*y[8], y[9], y[2]*y[8]*y[9]);
        p[14] = pip_fma(y[1]*y[7], y[9], y[2]*y[7]*y[8]);
        p[15] = pip_fma(y[1]*y[7], y[8], y[2]*y[7]*y[9]);
        break;
    case 3:
        p[0] = pip_fma(y[1]*y[6], y[9], y[2]*y[6]*y[8]);
        p[1] = pip_fma(y[1]*y[6], y[8], y[2]*y[6]*y[9]);
        p[2] = pip_fma(y[1]*y[6], y[7], y[2]*y[6]*y[7]);
        p[3] = pip_fma(y[1]*y[5], y[9], y[2]*y[4]*y[8]);
        p[4] = pip_fma(y[1]*y[5], y[8], y[2]*y[4]*y[9]);
        p[5] = pip_fma(y[1]*y[5], y[6], y[2]*y[4]*y[6]);
        p[6] = pip_fma(y[1]*y[4], y[9], y[2]*y[5]*y[8]);
        p[7] = pip_fma(y[1]*y[4], y[8], y[2]*y[5]*y[9]);
        p[8] = pip_fma(y[1]*y[4], y[6], y[2]*y[5]*y[6]);
        p[9] = pip_fma(y[1]*y[3], y[9], y[2]*y[3]*y[8]);
        p[10] = pip_fma(y[1]*y[3], y[8], y[2]*y[3]*y[9]);
        p[11] = pip_fma(y[1]*y[3], y[7], y[2]*y[3]*y[7]);
        p[12] = pip_fma(y[1]*y[3], y[6], y[2]*y[3]*y[6]);
        p[13] = pip_fma(y[1]*y[3], y[5], y[2]*y[3]*y[4]);
        p[14] = pip_fma(y[1]*y[3], y[4], y[2]*y[3]*y[5]);
        p[15] = pip_fma(y[1]*y[2], y[9], y[1]*y[2]*y[8]);
        break;
    case 4:
        p[0] = y[1]*y[2]*y[6];
        p[1] = y[1]*y[2]*y[3];
        p[2] = y[0]*y[8]*y[9];
        p[3] = pip_fma(y[0]*y[7], y[8], y[0]*y[7]*y[9]);
        p[4] = pip_fma(y[0]*y[6], y[8], y[0]*y[6]*y[9]);
        p[5] = y[0]*y[6]*y[7];
        p[6] = pip_fma(y[0]*y[4], y[9], y[0]*y[5]*y[8]);
        p[7] = pip_fma(y[0]*y[4], y[8], y[0]*y[5]*y[9]);
        p[8] = pip_fma(y[0]*y[4], y[6], y[0]*y[5]*y[6]);
        p[9] = pip_fma(y[0]*y[3], y[8], y[0]*y[3]*y[9]);
        p[10] = y[0]*y[3]*y[7];
        p[11] = y[0]*y[3]*y[6];
        p[12] = pip_fma(y[0]*y[3], y[4], y[0]*y[3]*y[5]);
        p[13] = pip_fma(y[0]*y[1], y[9], y[0]*y[2]*y[8]);
        p[14] = pip_fma(y[0]*y[1], y[8], y[0]*y[2]*y[9]);
        p[15] = pip_fma(y[0]*y[1], y[6], y[0]*y[2]*y[6]);
        break;
    case 5:
        p[0] = pip_fma(y[0]*y[1], y[3], y[0]*y[2]*y[3]);
        p[1] = pip_fma(y[8]*y[8], y[9], y[8]*y[9]*y[9]);
        p[2] = pip_fma(y[7]*y[8], y[8], y[7]*y[9]*y[9]);
        p[3] = pip_fma(y[7]*y[7], y[8], y[7]*y[7]*y[9]);
        p[4] = pip_fma(y[6]*y[8], y[8], y[6]*y[9]*y[9]);
        p[5] = y[6]*y[7]*y[7];
        p[6] = pip_fma(y[6]*y[6], y[8], y[6]*y[6]*y[9]);
        p[7] = y[6]*y[6]*y[7];
        p[8] = pip_fma(y[4]*y[9], y[9], y[5]*y[8]*y[8]);
        p[9] = pip_fma(y[4]*y[8], y[8], y[5]*y[9]*y[9]);
        p[10] = pip_fma(y[4]*y[6], y[6], y[5]*y[6]*y[6]);
        p[11] = pip_fma(y[4]*y[4], y[9], y[5]*y[5]*y[8]);
        p[12] = pip_fma(y[4]*y[4], y[8], y[5]*y[5]*y[9]);
        p[13] = pip_fma(y[4]*y[4], y[6], y[5]*y[5]*y[6]);
        p[14] = pip_fma(y[3]*y[9], y[9], y[3]*y[8]*y[8]);
        p[15] = y[3]*y[7]*y[7];
        break;
    case 6:
        p[0] = y[3]*y[6]*y[6];
        p[1] = pip_fma(y[3]*y[4], y[4], y[3]*y[5]*y[5]);
        p[2] = pip_fma(y[3]*y[3], y[8], y[3]*y[3]*y[9]);
        p[3] = y[3]*y[3]*y[7];
        p[4] = y[3]*y[3]*y[6];
        p[5] = pip_fma(y[3]*y[3], y[4], y[3]*y[3]*y[5]);
        p[6] = pip_fma(y[1]*y[9], y[9], y[2]*y[8]*y[8]);
        p[7] = pip_fma(y[1]*y[8], y[8], y[2]*y[9]*y[9]);
        p[8] = pip_fma(y[1]*y[6], y[6], y[2]*y[6]*y[6]);
        p[9] = pip_fma(y[1]*y[3], y[3], y[2]*y[3]*y[3]);
        p[10] = pip_fma(y[1]*y[1], y[9], y[2]*y[2]*y[8]);
        p[11] = pip_fma(y[1]*y[1], y[8], y[2]*y[2]*y[9]);
        p[12] = pip_fma(y[1]*y[1], y[6], y[2]*y[2]*y[6]);
        p[13] = pip_fma(y[1]*y[1], y[3], y[2]*y[2]*y[3]);
        p[14] = pip_fma(y[0]*y[8], y[8], y[0]*y[9]*y[9]);
        p[15] = y[0]*y[6]*y[6];
        break;
    case 7:
        p[0] = y[0]*y[3]*y[3];
        p[1] = pip_fma(y[0]*y[0], y[8], y[0]*y[0]*y[9]);
        p[2] = y[0]*y[0]*y[6];
        p[3] = y[0]*y[0]*y[3];
        p[4] = pip_fma(y[8]*y[8], y[8], y[9]*y[9]*y[9]);
        p[5] = y[6]*y[6]*y[6];
        p[6] = y[3]*y[3]*y[3];
        p[7] = T(0);
        p[8] = y[9];
        p[9] = y[8];
        p[10] = y[3] + y[6];
        p[11] = y[8]*y[9];
        p[12] = y[7]*y[9];
        p[13] = y[7]*y[8];
        p[14] = pip_fma(y[3], y[9], y[6]*y[9]);
        p[15] = pip_fma(y[3], y[8], y[6]*y[8]);
        break;
    case 8:
        p[0] = pip_fma(y[6], y[7], y[3]*y[7]);
        p[1] = y[3]*y[6];
        p[2] = pip_fma(y[2], y[9], y[5]*y[9]);
        p[3] = pip_fma(y[2], y[8], y[5]*y[8]);
        p[4] = pip_fma(y[2], y[6], y[3]*y[5]);
        p[5] = pip_fma(y[5], y[6], y[2]*y[3]);
        p[6] = pip_fma(y[1], y[9], y[4]*y[9]);
        p[7] = pip_fma(y[1], y[8], y[4]*y[8]);
        p[8] = pip_fma(y[1], y[6], y[3]*y[4]);
        p[9] = pip_fma(y[4], y[6], y[1]*y[3]);
        p[10] = y[0]*y[9];
        p[11] = y[0]*y[8];
        p[12] = pip_fma(y[0], y[6], y[0]*y[3]);
        p[13] = y[9]*y[9];
        p[14] = y[8]*y[8];
        p[15] = pip_fma(y[6], y[6], y[3]*y[3]);
        break;
    case 9:
        p[0] = y[7]*y[8]*y[9];
        p[1] = pip_fma(y[3]*y[8], y[9], y[6]*y[8]*y[9]);
        p[2] = pip_fma(y[3]*y[7], y[9], y[6]*y[7]*y[9]);
        p[3] = pip_fma(y[3]*y[7], y[8], y[6]*y[7]*y[8]);
        p[4] = y[3]*y[6]*y[9];
        p[5] = y[3]*y[6]*y[8];
        p[6] = y[3]*y[6]*y[7];
        p[7] = pip_fma(y[2]*y[8], y[9], y[5]*y[8]*y[9]);
        p[8] = pip_fma(y[2]*y[7], y[9], y[5]*y[7]*y[9]);
        p[9] = pip_fma(y[2]*y[7], y[8], y[5]*y[7]*y[8]);
        p[10] = pip_fma(y[2]*y[6], y[9], y[3]*y[5]*y[9]);
        p[11] = pip_fma(y[2]*y[6], y[8], y[3]*y[5]*y[8]);
        p[12] = pip_fma(y[2]*y[6], y[7], y[3]*y[5]*y[7]);
        p[13] = y[2]*y[5]*y[9];
        p[14] = y[2]*y[5]*y[8];
        p[15] = pip_fma(y[2]*y[3], y[9], y[5]*y[6]*y[9]);
        break;
    case 10:
        p[0] = pip_fma(y[2]*y[3], y[8], y[5]*y[6]*y[8]);
        p[1] = pip_fma(y[2]*y[3], y[7], y[5]*y[6]*y[7]);
        p[2] = pip_fma(y[2]*y[3], y[6], y[3]*y[5]*y[6]);
        p[3] = pip_fma(y[2]*y[3], y[5], y[2]*y[5]*y[6]);
        p[4] = pip_fma(y[1]*y[8], y[9], y[4]*y[8]*y[9]);
        p[5] = pip_fma(y[1]*y[7], y[9], y[4]*y[7]*y[9]);
        p[6] = pip_fma(y[1]*y[7], y[8], y[4]*y[7]*y[8]);
        p[7] = pip_fma(y[1]*y[6], y[9], y[3]*y[4]*y[9]);
        p[8] = pip_fma(y[1]*y[6], y[8], y[3]*y[4]*y[8]);
        p[9] = pip_fma(y[1]*y[6], y[7], y[3]*y[4]*y[7]);
        p[10] = pip_fma(y[1]*y[5], y[9], y[2]*y[4]*y[9]);
        p[11] = pip_fma(y[1]*y[5], y[8], y[2]*y[4]*y[8]);
        p[12] = pip_fma(y[1]*y[5], y[6], y[2]*y[3]*y[4]);
        p[13] = y[1]*y[4]*y[9];
        p[14] = y[1]*y[4]*y[8];
        p[15] = pip_fma(y[1]*y[3], y[9], y[4]*y[6]*y[9]);
        break;
    case 11:
        p[0] = pip_fma(y[1]*y[3], y[8], y[4]*y[6]*y[8]);
        p[1] = pip_fma(y[1]*y[3], y[7], y[4]*y[6]*y[7]);
        p[2] = pip_fma(y[1]*y[3], y[6], y[3]*y[4]*y[6]);
        p[3] = pip_fma(y[1]*y[3], y[5], y[2]*y[4]*y[6]);
        p[4] = pip_fma(y[1]*y[3], y[4], y[1]*y[4]*y[6]);
        p[5] = pip_fma(y[1]*y[2], y[9], y[4]*y[5]*y[9]);
        p[6] = pip_fma(y[4]*y[5], y[8], y[1]*y[2]*y[8]);
        p[7] = pip_fma(y[1]*y[2], y[6], y[3]*y[4]*y[5]);
        p[8] = pip_fma(y[1]*y[2], y[3], y[4]*y[5]*y[6]);
        p[9] = y[0]*y[8]*y[9];
        p[10] = y[0]*y[7]*y[9];
        p[11] = y[0]*y[7]*y[8];
        p[12] = pip_fma(y[0]*y[3], y[9], y[0]*y[6]*y[9]);
        p[13] = pip_fma(y[0]*y[3], y[8], y[0]*y[6]*y[8]);
        p[14] = pip_fma(y[0]*y[3], y[7], y[0]*y[6]*y[7]);
        p[15] = y[0]*y[3]*y[6];
        break;
    case 12:
        p[0] = pip_fma(y[0]*y[2], y[9], y[0]*y[5]*y[9]);
        p[1] = pip_fma(y[0]*y[2], y[8], y[0]*y[5]*y[8]);
        p[2] = pip_fma(y[0]*y[2], y[6], y[0]*y[3]*y[5]);
        p[3] = pip_fma(y[0]*y[2], y[3], y[0]*y[5]*y[6]);
        p[4] = pip_fma(y[0]*y[1], y[9], y[0]*y[4]*y[9]);
        p[5] = pip_fma(y[0]*y[1], y[8], y[0]*y[4]*y[8]);
        p[6] = pip_fma(y[0]*y[1], y[6], y[0]*y[3]*y[4]);
        p[7] = pip_fma(y[0]*y[1], y[3], y[0]*y[4]*y[6]);
        p[8] = y[8]*y[9]*y[9];
        p[9] = y[8]*y[8]*y[9];
        p[10] = y[7]*y[9]*y[9];
        p[11] = y[7]*y[8]*y[8];
        p[12] = y[7]*y[7]*y[9];
        p[13] = y[7]*y[7]*y[8];
        p[14] = pip_fma(y[3]*y[9], y[9], y[6]*y[9]*y[9]);
        p[15] = pip_fma(y[6]*y[8], y[8], y[3]*y[8]*y[8]);
        break;
    case 13:
        p[0] = pip_fma(y[3]*y[7], y[7], y[6]*y[7]*y[7]);
        p[1] = pip_fma(y[3]*y[3], y[9], y[6]*y[6]*y[9]);
        p[2] = pip_fma(y[3]*y[3], y[8], y[6]*y[6]*y[8]);
        p[3] = pip_fma(y[3]*y[3], y[7], y[6]*y[6]*y[7]);
        p[4] = pip_fma(y[3]*y[3], y[6], y[3]*y[6]*y[6]);
        p[5] = pip_fma(y[2]*y[9], y[9], y[5]*y[9]*y[9]);
        p[6] = pip_fma(y[2]*y[8], y[8], y[5]*y[8]*y[8]);
        p[7] = pip_fma(y[2]*y[6], y[6], y[3]*y[3]*y[5]);
        p[8] = pip_fma(y[2]*y[3], y[3], y[5]*y[6]*y[6]);
        p[9] = pip_fma(y[2]*y[2], y[9], y[5]*y[5]*y[9]);
        p[10] = pip_fma(y[2]*y[2], y[8], y[5]*y[5]*y[8]);
        p[11] = pip_fma(y[2]*y[2], y[6], y[3]*y[5]*y[5]);
        p[12] = pip_fma(y[2]*y[2], y[3], y[5]*y[5]*y[6]);
        p[13] = pip_fma(y[1]*y[9], y[9], y[4]*y[9]*y[9]);
        p[14] = pip_fma(y[1]*y[8], y[8], y[4]*y[8]*y[8]);
        p[15] = pip_fma(y[1]*y[6], y[6], y[3]*y[3]*y[4]);
        break;
    case 14:
        p[0] = pip_fma(y[1]*y[3], y[3], y[4]*y[6]*y[6]);
        p[1] = pip_fma(y[1]*y[1], y[9], y[4]*y[4]*y[9]);
        p[2] = pip_fma(y[1]*y[1], y[8], y[4]*y[4]*y[8]);
        p[3] = pip_fma(y[1]*y[1], y[6], y[3]*y[4]*y[4]);
        p[4] = pip_fma(y[1]*y[1], y[3], y[4]*y[4]*y[6]);
        p[5] = y[0]*y[9]*y[9];
        p[6] = y[0]*y[8]*y[8];
        p[7] = pip_fma(y[0]*y[3], y[3], y[0]*y[6]*y[6]);
        p[8] = y[0]*y[0]*y[9];
        p[9] = y[0]*y[0]*y[8];
        p[10] = pip_fma(y[0]*y[0], y[3], y[0]*y[0]*y[6]);
        p[11] = y[9]*y[9]*y[9];
        p[12] = y[8]*y[8]*y[8];
        p[13] = pip_fma(y[3]*y[3], y[3], y[6]*y[6]*y[6]);
        p[14] = T(0);
        p[15] = y[8] + y[9];
        break;
    case 15:
        p[0] = y[3] + y[6];
        p[1] = y[8]*y[9];
        p[2] = pip_fma(y[7], y[9], y[7]*y[8]);
        p[3] = pip_fma(y[6], y[9], pip_fma(y[6], y[8], pip_fma(y[3], y[9], y[3]*y[8])));
        p[4] = pip_fma(y[6], y[7], y[3]*y[7]);
        p[5] = y[3]*y[6];
        p[6] = pip_fma(y[5], y[8], pip_fma(y[4], y[9], pip_fma(y[1], y[9], y[2]*y[8])));
        p[7] = pip_fma(y[5], y[9], pip_fma(y[4], y[8], pip_fma(y[2], y[9], y[1]*y[8])));
        p[8] = pip_fma(y[3], y[5], pip_fma(y[3], y[4], pip_fma(y[1], y[6], y[2]*y[6])));
        p[9] = pip_fma(y[5], y[6], pip_fma(y[4], y[6], pip_fma(y[2], y[3], y[1]*y[3])));
        p[10] = pip_fma(y[0], y[9], y[0]*y[8]);
        p[11] = pip_fma(y[0], y[6], y[0]*y[3]);
        p[12] = pip_fma(y[9], y[9], y[8]*y[8]);
        p[13] = pip_fma(y[6], y[6], y[3]*y[3]);
        p[14] = y[7]*y[8]*y[9];
        p[15] = pip_fma(y[3]*y[8], y[9], y[6]*y[8]*y[9]);
        break;
    case 16:
        p[0] = pip_fma(y[6]*y[7], y[9], pip_fma(y[6]*y[7], y[8], pip_fma(y[3]*y[7], y[8], y[3]*y[7]*y[9])));
        p[1] = pip_fma(y[3]*y[6], y[8], y[3]*y[6]*y[9]);
        p[2] = y[3]*y[6]*y[7];
        p[3] = pip_fma(y[5]*y[8], y[9], pip_fma(y[4]*y[8], y[9], pip_fma(y[1]*y[8], y[9], y[2]*y[8]*y[9])));
        p[4] = pip_fma(y[5]*y[7], y[8], pip_fma(y[4]*y[7], y[9], pip_fma(y[1]*y[7], y[9], y[2]*y[7]*y[8])));
        p[5] = pip_fma(y[5]*y[7], y[9], pip_fma(y[4]*y[7], y[8], pip_fma(y[1]*y[7], y[8], y[2]*y[7]*y[9])));
        p[6] = pip_fma(y[3]*y[5], y[8], pip_fma(y[3]*y[4], y[9], pip_fma(y[1]*y[6], y[9], y[2]*y[6]*y[8])));
        p[7] = pip_fma(y[3]*y[5], y[9], pip_fma(y[3]*y[4], y[8], pip_fma(y[1]*y[6], y[8], y[2]*y[6]*y[9])));
        p[8] = pip_fma(y[3]*y[5], y[7], pip_fma(y[3]*y[4], y[7], pip_fma(y[1]*y[6], y[7], y[2]*y[6]*y[7])));
        p[9] = pip_fma(y[2]*y[4], y[9], pip_fma(y[2]*y[4], y[8], pip_fma(y[1]*y[5], y[8], y[1]*y[5]*y[9])));
        p[10] = pip_fma(y[1]*y[4], y[9], y[2]*y[5]*y[8]);
        p[11] = pip_fma(y[1]*y[4], y[8], y[2]*y[5]*y[9]);
        p[12] = pip_fma(y[5]*y[6], y[8], pip_fma(y[4]*y[6], y[9], pip_fma(y[1]*y[3], y[9], y[2]*y[3]*y[8])));
        p[13] = pip_fma(y[5]*y[6], y[9], pip_fma(y[4]*y[6], y[8], pip_fma(y[1]*y[3], y[8], y[2]*y[3]*y[9])));
        p[14] = pip_fma(y[5]*y[6], y[7], pip_fma(y[4]*y[6], y[7], pip_fma(y[1]*y[3], y[7], y[2]*y[3]*y[7])));
        p[15] = pip_fma(y[3]*y[5], y[6], pip_fma(y[3]*y[4], y[6], pip_fma(y[1]*y[3], y[6], y[2]*y[3]*y[6])));
        break;
    case 17:
        p[0] = pip_fma(y[2]*y[4], y[6], pip_fma(y[2]*y[3], y[4], pip_fma(y[1]*y[3], y[5], y[1]*y[5]*y[6])));
        p[1] = pip_fma(y[2]*y[5], y[6], pip_fma(y[2]*y[3], y[5], pip_fma(y[1]*y[3], y[4], y[1]*y[4]*y[6])));
        p[2] = pip_fma(y[4]*y[5], y[9], pip_fma(y[4]*y[5], y[8], pip_fma(y[1]*y[2], y[9], y[1]*y[2]*y[8])));
        p[3] = pip_fma(y[1]*y[2], y[6], y[3]*y[4]*y[5]);
        p[4] = pip_fma(y[1]*y[2], y[3], y[4]*y[5]*y[6]);
        p[5] = y[0]*y[8]*y[9];
        p[6] = pip_fma(y[0]*y[7], y[8], y[0]*y[7]*y[9]);
        p[7] = pip_fma(y[0]*y[6], y[9], pip_fma(y[0]*y[6], y[8], pip_fma(y[0]*y[3], y[8], y[0]*y[3]*y[9])));
        p[8] = pip_fma(y[0]*y[3], y[7], y[0]*y[6]*y[7]);
        p[9] = y[0]*y[3]*y[6];
        p[10] = pip_fma(y[0]*y[5], y[8], pip_fma(y[0]*y[4], y[9], pip_fma(y[0]*y[1], y[9], y[0]*y[2]*y[8])));
        p[11] = pip_fma(y[0]*y[5], y[9], pip_fma(y[0]*y[4], y[8], pip_fma(y[0]*y[1], y[8], y[0]*y[2]*y[9])));
        p[12] = pip_fma(y[0]*y[3], y[5], pip_fma(y[0]*y[3], y[4], pip_fma(y[0]*y[1], y[6], y[0]*y[2]*y[6])));
        p[13] = pip_fma(y[0]*y[5], y[6], pip_fma(y[0]*y[4], y[6], pip_fma(y[0]*y[1], y[3], y[0]*y[2]*y[3])));
        p[14] = pip_fma(y[8]*y[8], y[9], y[8]*y[9]*y[9]);
        p[15] = pip_fma(y[7]*y[8], y[8], y[7]*y[9]*y[9]);
        break;
    case 18:
        p[0] = pip_fma(y[7]*y[7], y[8], y[7]*y[7]*y[9]);
        p[1] = pip_fma(y[6]*y[9], y[9], pip_fma(y[6]*y[8], y[8], pip_fma(y[3]*y[9], y[9], y[3]*y[8]*y[8])));
        p[2] = pip_fma(y[3]*y[7], y[7], y[6]*y[7]*y[7]);
        p[3] = pip_fma(y[6]*y[6], y[9], pip_fma(y[6]*y[6], y[8], pip_fma(y[3]*y[3], y[8], y[3]*y[3]*y[9])));
        p[4] = pip_fma(y[3]*y[3], y[7], y[6]*y[6]*y[7]);
        p[5] = pip_fma(y[3]*y[3], y[6], y[3]*y[6]*y[6]);
        p[6] = pip_fma(y[5]*y[8], y[8], pip_fma(y[4]*y[9], y[9], pip_fma(y[1]*y[9], y[9], y[2]*y[8]*y[8])));
        p[7] = pip_fma(y[5]*y[9], y[9], pip_fma(y[4]*y[8], y[8], pip_fma(y[1]*y[8], y[8], y[2]*y[9]*y[9])));
        p[8] = pip_fma(y[3]*y[3], y[5], pip_fma(y[3]*y[3], y[4], pip_fma(y[1]*y[6], y[6], y[2]*y[6]*y[6])));
        p[9] = pip_fma(y[5]*y[6], y[6], pip_fma(y[4]*y[6], y[6], pip_fma(y[1]*y[3], y[3], y[2]*y[3]*y[3])));
        p[10] = pip_fma(y[5]*y[5], y[8], pip_fma(y[4]*y[4], y[9], pip_fma(y[1]*y[1], y[9], y[2]*y[2]*y[8])));
        p[11] = pip_fma(y[5]*y[5], y[9], pip_fma(y[4]*y[4], y[8], pip_fma(y[1]*y[1], y[8], y[2]*y[2]*y[9])));
        p[12] = pip_fma(y[3]*y[5], y[5], pip_fma(y[3]*y[4], y[4], pip_fma(y[1]*y[1], y[6], y[2]*y[2]*y[6])));
        p[13] = pip_fma(y[5]*y[5], y[6], pip_fma(y[4]*y[4], y[6], pip_fma(y[1]*y[1], y[3], y[2]*y[2]*y[3])));
        p[14] = pip_fma(y[0]*y[8], y[8], y[0]*y[9]*y[9]);
        p[15] = pip_fma(y[0]*y[3], y[3], y[0]*y[6]*y[6]);
        break;
    case 19:
        p[0] = pip_fma(y[0]*y[0], y[8], y[0]*y[0]*y[9]);
        p[1] = pip_fma(y[0]*y[0], y[3], y[0]*y[0]*y[6]);
        p[2] = pip_fma(y[8]*y[8], y[8], y[9]*y[9]*y[9]);
        p[3] = pip_fma(y[3]*y[3], y[3], y[6]*y[6]*y[6]);
        p[4] = T(0);
        p[5] = T(0);
        p[6] = T(0);
        p[7] = T(0);
        p[8] = T(0);
        p[9] = T(0);
        p[10] = T(0);
        p[11] = T(0);
        p[12] = T(0);
        p[13] = T(0);
        p[14] = T(0);
        p[15] = T(0);
        break;
    default:
        break;
    }
}

}  // namespace hh
