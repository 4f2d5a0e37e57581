// Line transforms whose length, line count and strides are known at compile
// time, on radices 8, 4, 2, 5 in a fixed order: every index map is a shift or a
// multiply-shift, the strides fold into the LDS offsets and a thread holds only
// the butterflies it owns.
//
// The 128^2 and 160^2 planes and the x lines of 128, 160 and (six types) 256
// points run on these; fft_line.h runs everything else.  The line: at
// these sizes one workgroup fills a CU's LDS or registers and short stages of
// radix 8 and below, with their smaller register need, beat the longer
// radices that win elsewhere.  Measured, these against fft_line.h compiled for the same
// sizes: c2r of 160^2 planes, four types 140 against 161 us, x lines of
// 160^3, four types 55 against 63 us and of 256^3, six types 517 against 610
// us; 128^3, four types c2r 47.7 against 48.5 us.
#pragma once
#include "common.h"
#include "fft_line.h"

namespace hymd::ct {

constexpr int kMaxStages = 8;

template <int R>
__device__ __forceinline__ void small_dft(float2 (&u)[8], float sgn);

template <>
__device__ __forceinline__ void small_dft<2>(float2 (&u)[8], float) {
    float2 a = u[0], b = u[1];
    u[0] = cadd(a, b);
    u[1] = csub(a, b);
}

template <>
__device__ __forceinline__ void small_dft<4>(float2 (&u)[8], float sgn) {
    float2 t0 = cadd(u[0], u[2]), t1 = csub(u[0], u[2]);
    float2 t2 = cadd(u[1], u[3]), t3 = cmul_i(csub(u[1], u[3]), sgn);
    u[0] = cadd(t0, t2);
    u[1] = cadd(t1, t3);
    u[2] = csub(t0, t2);
    u[3] = csub(t1, t3);
}

template <>
__device__ __forceinline__ void small_dft<5>(float2 (&u)[8], float sgn) {
    const float c1 = 0.30901699437494742410f;   // cos(2pi/5)
    const float c2 = -0.80901699437494742410f;  // cos(4pi/5)
    const float s1 = 0.95105651629515357212f;   // sin(2pi/5)
    const float s2 = 0.58778525229247312917f;   // sin(4pi/5)
    float2 a1 = cadd(u[1], u[4]), b1 = csub(u[1], u[4]);
    float2 a2 = cadd(u[2], u[3]), b2 = csub(u[2], u[3]);
    float2 m1 = make_float2(u[0].x + c1 * a1.x + c2 * a2.x, u[0].y + c1 * a1.y + c2 * a2.y);
    float2 m2 = make_float2(u[0].x + c2 * a1.x + c1 * a2.x, u[0].y + c2 * a1.y + c1 * a2.y);
    float2 n1 = cmul_i(make_float2(s1 * b1.x + s2 * b2.x, s1 * b1.y + s2 * b2.y), sgn);
    float2 n2 = cmul_i(make_float2(s2 * b1.x - s1 * b2.x, s2 * b1.y - s1 * b2.y), sgn);
    u[0] = cadd(u[0], cadd(a1, a2));
    u[1] = cadd(m1, n1);
    u[4] = csub(m1, n1);
    u[2] = cadd(m2, n2);
    u[3] = csub(m2, n2);
}

template <>
__device__ __forceinline__ void small_dft<8>(float2 (&u)[8], float sgn) {
    const float r = 0.70710678118654752440f;
    float2 e[8] = {u[0], u[2], u[4], u[6], u[0], u[0], u[0], u[0]};
    float2 o[8] = {u[1], u[3], u[5], u[7], u[0], u[0], u[0], u[0]};
    small_dft<4>(e, sgn);
    small_dft<4>(o, sgn);
    // w^j o_j, w = exp(sgn 2 pi i / 8)
    float2 w1 = cscale(cadd(o[1], cmul_i(o[1], sgn)), r);
    float2 w2 = cmul_i(o[2], sgn);
    float2 w3 = cscale(csub(cmul_i(o[3], sgn), o[3]), r);
    u[0] = cadd(e[0], o[0]);
    u[4] = csub(e[0], o[0]);
    u[1] = cadd(e[1], w1);
    u[5] = csub(e[1], w1);
    u[2] = cadd(e[2], w2);
    u[6] = csub(e[2], w2);
    u[3] = cadd(e[3], w3);
    u[7] = csub(e[3], w3);
}

struct StagePlan {
    int ns;
    int r[kMaxStages], p[kMaxStages], twoff[kMaxStages];
};

// radices largest first: 8s, then one 4 / 4+4 / 2 for the power-of-two
// remainder, then 5s (ns = 0 if n is not 2^a 5^c)
constexpr StagePlan make_stage_plan(int n) {
    StagePlan sp{};
    int rs[kMaxStages] = {};
    int cnt = 0, a = 0;
    while (n % 2 == 0) {
        n /= 2;
        ++a;
    }
    int eights = a / 3;
    const int rem = a % 3;
    int tail[2] = {0, 0}, nt = 0;
    if (rem == 1 && eights > 0) {
        --eights;
        tail[nt++] = 4;
        tail[nt++] = 4;
    } else if (rem == 1) {
        tail[nt++] = 2;
    } else if (rem == 2) {
        tail[nt++] = 4;
    }
    for (int i = 0; i < eights; ++i) rs[cnt++] = 8;
    for (int i = 0; i < nt; ++i) rs[cnt++] = tail[i];
    while (n % 5 == 0) {
        n /= 5;
        rs[cnt++] = 5;
    }
    if (n != 1 || cnt > kMaxStages) return sp;
    int p = 1, off = 0;
    for (int i = 0; i < cnt; ++i) {
        sp.r[i] = rs[i];
        sp.p[i] = p;
        sp.twoff[i] = off;
        off += p * (rs[i] - 1);
        p *= rs[i];
    }
    sp.ns = cnt;
    return sp;
}

template <int N>
struct CtPlan {
    static constexpr StagePlan v = make_stage_plan(N);
};

template <int R, int P, int N, int NLINES, int SE, int SL, int NT, int SGN>
__device__ __forceinline__ void stockham_inplace_ct(float2 *buf, const float2 *__restrict__ tw) {
    constexpr int NR = N / R, TOTAL = NLINES * NR, KB = (TOTAL + NT - 1) / NT;
    constexpr float sgn = (float)SGN;
    float2 u[KB][8];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
        const int b = threadIdx.x + kb * NT;
        if (TOTAL % NT != 0 && b >= TOTAL) continue;
        const int i = b / NLINES, l = b - i * NLINES, k = i % P;
        const float2 *src = buf + l * SL + i * SE;
#pragma unroll
        for (int j = 0; j < R; ++j) u[kb][j] = src[j * NR * SE];
        if (P > 1) {
#pragma unroll
            for (int j = 1; j < R; ++j) {
                float2 w = tw[k * (R - 1) + j - 1];
                if (SGN > 0) w.y = -w.y;
                u[kb][j] = cmul(u[kb][j], w);
            }
        }
        small_dft<R>(u[kb], sgn);
    }
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
        const int b = threadIdx.x + kb * NT;
        if (TOTAL % NT != 0 && b >= TOTAL) continue;
        const int i = b / NLINES, l = b - i * NLINES, q = i / P, k = i - q * P;
        float2 *dst = buf + l * SL + (q * P * R + k) * SE;
#pragma unroll
        for (int j = 0; j < R; ++j) dst[j * P * SE] = u[kb][j];
    }
    __syncthreads();
}

// Stage 0 of fft_inplace_ct (P = 1, no twiddles) with its inputs from
// ld(line, element) (global memory) instead of buf: the load pass of the
// plane kernels and the first LDS round trip become one.  buf is only
// written, then a barrier; fft_inplace_ct<..., 1> runs the other stages.
// I_FAST: consecutive threads take consecutive butterflies of one line
// (the global reads of a line stored contiguously coalesce), else
// consecutive lines (lines stored side by side).
template <int N, int NLINES, int SE, int SL, int NT, int SGN, bool I_FAST = false, class Load>
__device__ __forceinline__ void fft_first_ct(float2 *buf, Load ld) {
    constexpr StagePlan sp = CtPlan<N>::v;
    static_assert(sp.ns >= 1, "no stage plan");
    constexpr int R = sp.r[0], NR = N / R, TOTAL = NLINES * NR, KB = (TOTAL + NT - 1) / NT;
    constexpr float sgn = (float)SGN;
    float2 u[KB][8];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
        const int b = threadIdx.x + kb * NT;
        if (TOTAL % NT != 0 && b >= TOTAL) continue;
        const int i = I_FAST ? b % NR : b / NLINES, l = I_FAST ? b / NR : b - i * NLINES;
#pragma unroll
        for (int j = 0; j < R; ++j) u[kb][j] = ld(l, i + j * NR);
        small_dft<R>(u[kb], sgn);
        float2 *dst = buf + l * SL + i * R * SE;
#pragma unroll
        for (int j = 0; j < R; ++j) dst[j * SE] = u[kb][j];
    }
    __syncthreads();
}

// Stage 0 of fft_inplace_ct with its inputs formed by ld(line, element)
// from buf itself (a pass that would otherwise write buf first, such as the
// real-FFT split): every input is read before the barrier, every output
// written after it.
template <int N, int NLINES, int SE, int SL, int NT, int SGN, bool I_FAST, class Load>
__device__ __forceinline__ void fft_first_ct_inplace(float2 *buf, Load ld) {
    constexpr StagePlan sp = CtPlan<N>::v;
    static_assert(sp.ns >= 1, "no stage plan");
    constexpr int R = sp.r[0], NR = N / R, TOTAL = NLINES * NR, KB = (TOTAL + NT - 1) / NT;
    constexpr float sgn = (float)SGN;
    float2 u[KB][8];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
        const int b = threadIdx.x + kb * NT;
        if (TOTAL % NT != 0 && b >= TOTAL) continue;
        const int i = I_FAST ? b % NR : b / NLINES, l = I_FAST ? b / NR : b - i * NLINES;
#pragma unroll
        for (int j = 0; j < R; ++j) u[kb][j] = ld(l, i + j * NR);
        small_dft<R>(u[kb], sgn);
    }
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
        const int b = threadIdx.x + kb * NT;
        if (TOTAL % NT != 0 && b >= TOTAL) continue;
        const int i = I_FAST ? b % NR : b / NLINES, l = I_FAST ? b / NR : b - i * NLINES;
        float2 *dst = buf + l * SL + i * R * SE;
#pragma unroll
        for (int j = 0; j < R; ++j) dst[j * SE] = u[kb][j];
    }
    __syncthreads();
}

template <int N, int NLINES, int SE, int SL, int NT, int SGN, int S = 0, int SEND = CtPlan<N>::v.ns>
__device__ __forceinline__ void fft_inplace_ct(float2 *buf, const float2 *__restrict__ tw) {
    constexpr StagePlan sp = CtPlan<N>::v;
    if constexpr (S < SEND) {
        stockham_inplace_ct<sp.r[S], sp.p[S], N, NLINES, SE, SL, NT, SGN>(buf, tw + sp.twoff[S]);
        fft_inplace_ct<N, NLINES, SE, SL, NT, SGN, S + 1, SEND>(buf, tw);
    }
}

// The last stage of fft_inplace_ct (q = 0: output element k + j P) with its
// outputs to st(line, element, value) (global memory) instead of buf: the
// store pass and the last LDS round trip become one.  buf is only read.
template <int N, int NLINES, int SE, int SL, int NT, int SGN, bool I_FAST, class Store>
__device__ __forceinline__ void fft_last_ct(const float2 *buf, const float2 *__restrict__ tw, Store st) {
    constexpr StagePlan sp = CtPlan<N>::v;
    static_assert(sp.ns >= 1, "no stage plan");
    constexpr int S = sp.ns - 1, R = sp.r[S], P = sp.p[S], NR = N / R, TOTAL = NLINES * NR,
                  KB = (TOTAL + NT - 1) / NT;
    static_assert(P == NR, "the last stage spans the line");
    constexpr float sgn = (float)SGN;
    const float2 *tws = tw + sp.twoff[S];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
        const int b = threadIdx.x + kb * NT;
        if (TOTAL % NT != 0 && b >= TOTAL) continue;
        const int i = I_FAST ? b % NR : b / NLINES, l = I_FAST ? b / NR : b - i * NLINES;
        const float2 *src = buf + l * SL + i * SE;
        float2 u[8];
#pragma unroll
        for (int j = 0; j < R; ++j) u[j] = src[j * NR * SE];
        if (P > 1) {
#pragma unroll
            for (int j = 1; j < R; ++j) {
                float2 w = tws[i * (R - 1) + j - 1];
                if (SGN > 0) w.y = -w.y;
                u[j] = cmul(u[j], w);
            }
        }
        small_dft<R>(u, sgn);
#pragma unroll
        for (int j = 0; j < R; ++j) st(l, i + j * P, u[j]);
    }
}

}  // namespace hymd::ct
