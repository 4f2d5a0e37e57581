// Line transforms for n = 2^a 3^b 5^c with radices up to 16, held in registers.
//
// What bounds the transforms of this path is neither flops nor HBM but the
// passes over LDS between the stages and the index arithmetic around them, so
// a line takes as few stages as possible.  With radices up to 10, as the line
// and plane passes take them: two to 100 points but for 75 and 96, three to
// 1000 but for 375, 625, 675, 750, 768, 864, 960 and 972; the x-line pass of one
// and two types ends with a radix up to 16 and takes two to 160 points.  The
// first stage reads its elements from wherever they are (global memory, or LDS
// through an element-wise map), the last one hands its outputs to a store
// functor, and only the values between two stages cross LDS.  Butterfly indices
// are split by a float reciprocal (exact below 2^22, see divq), five
// full-rate instructions where an integer multiply-high takes three quarter-rate
// ones.
//
// Stage s of radix R after sub-transforms of size p (self-sorting Stockham):
// butterfly i of n/R, k = i mod p, reads x[i + j n/R], multiplies by
// exp(-+2 pi i jk/(pR)), applies the R-point DFT and writes
// y[(i - k) R + k + j p].
#pragma once
#include <type_traits>
#include <utility>

#include "common.h"

namespace hymd {

constexpr int kMaxLineStages = 4;

// Radices of an n-point line, none above `most`: the fewest stages, among
// those the smallest largest radix (registers), then the smallest second one,
// and so on; larger radices first (the first stage has no twiddles).
// ns = 0: no such plan.
struct LineRadices {
    int ns;
    int r[kMaxLineStages];
};

constexpr bool line_radices_find(LineRadices &p, int depth, int stages, int rest, int most) {
    if (depth == stages) return rest == 1;
    for (int r = 2; r <= most; ++r) {
        if (r == 7 || r == 11 || r == 13 || r == 14 || rest % r != 0) continue;
        p.r[depth] = r;
        if (line_radices_find(p, depth + 1, stages, rest / r, r)) return true;
    }
    return false;
}

constexpr LineRadices line_radices(int n, int most) {
    LineRadices p{};
    for (int stages = 1; stages <= kMaxLineStages; ++stages)
        if (line_radices_find(p, 0, stages, n, most)) {
            p.ns = stages;
            return p;
        }
    return p;
}

// One stage: radix, sub-transform size, butterflies per line, twiddle offset.
struct LineStage {
    int R, p, nr, tw;
    float inv_p, inv_nr;
};

// A line with its plan known on the host only.
struct LineAxis {
    int n, ns;
    LineStage st[kMaxLineStages];
};

// q = b / d for 0 <= b < 2^22 and inv = 1.0f / d: (b + 0.5) / d lies at least
// 0.5 / d from an integer, and the two roundings, of 2^-24 each, move it by
// less than (b + 0.5) / d * 2^-23 (1 + 2^-24), which stays below 0.5 / d while
// b + 1 <= 2^22.
__device__ __forceinline__ int divq(int b, float inv) { return (int)(((float)b + 0.5f) * inv); }

// ---------------------------------------------------------------------------
// R-point DFTs in registers, SGN = -1 forward, +1 inverse
// ---------------------------------------------------------------------------
namespace dft {

// cos and sin of 2 pi m / n at compile time (Taylor series of the angle in
// [-pi, pi], 30 terms: below FP64 rounding)
constexpr double series(double x, bool odd) {
    double term = odd ? x : 1.0, sum = term;
    for (int k = odd ? 2 : 1; k < 60; k += 2) {
        term = -term * x * x / ((double)k * (double)(k + 1));
        sum += term;
    }
    return sum;
}
constexpr double angle(int m, int n) {
    const double a = 6.283185307179586476925286766559 * (double)(m % n) / (double)n;
    return a > 3.141592653589793238462643383280 ? a - 6.283185307179586476925286766559 : a;
}
constexpr double ccos(int m, int n) { return series(angle(m, n), false); }
constexpr double csin(int m, int n) { return series(angle(m, n), true); }

constexpr int inverse_mod(int a, int m) {
    for (int x = 1; x < m; ++x)
        if ((a * x) % m == 1) return x;
    return 0;
}

template <int R, int SGN>
struct Dft;

template <int SGN>
struct Dft<1, SGN> {
    static __device__ __forceinline__ void run(float2 (&)[1]) {}
};

template <int SGN>
struct Dft<2, SGN> {
    static __device__ __forceinline__ void run(float2 (&u)[2]) {
        const float2 a = u[0], b = u[1];
        u[0] = cadd(a, b);
        u[1] = csub(a, b);
    }
};

template <int SGN>
struct Dft<3, SGN> {
    static __device__ __forceinline__ void run(float2 (&u)[3]) {
        constexpr float h = (float)SGN * 0.86602540378443864676f;  // sqrt(3)/2
        const float2 t = cadd(u[1], u[2]);
        const float2 m = make_float2(u[0].x - 0.5f * t.x, u[0].y - 0.5f * t.y);
        const float2 s = cmul_i(csub(u[1], u[2]), h);
        u[0] = cadd(u[0], t);
        u[1] = cadd(m, s);
        u[2] = csub(m, s);
    }
};

template <int SGN>
struct Dft<4, SGN> {
    static __device__ __forceinline__ void run(float2 (&u)[4]) {
        const float2 t0 = cadd(u[0], u[2]), t1 = csub(u[0], u[2]);
        const float2 t2 = cadd(u[1], u[3]), t3 = cmul_i(csub(u[1], u[3]), (float)SGN);
        u[0] = cadd(t0, t2);
        u[1] = cadd(t1, t3);
        u[2] = csub(t0, t2);
        u[3] = csub(t1, t3);
    }
};

template <int SGN>
struct Dft<5, SGN> {
    static __device__ __forceinline__ void run(float2 (&u)[5]) {
        constexpr float c1 = 0.30901699437494742410f, c2 = -0.80901699437494742410f;  // cos 72, cos 144
        constexpr float s1 = 0.95105651629515357212f, s2 = 0.58778525229247312917f;   // sin 72, sin 144
        const float2 a1 = cadd(u[1], u[4]), b1 = csub(u[1], u[4]);
        const float2 a2 = cadd(u[2], u[3]), b2 = csub(u[2], u[3]);
        const float2 m1 = make_float2(u[0].x + c1 * a1.x + c2 * a2.x, u[0].y + c1 * a1.y + c2 * a2.y);
        const float2 m2 = make_float2(u[0].x + c2 * a1.x + c1 * a2.x, u[0].y + c2 * a1.y + c1 * a2.y);
        const float2 n1 = cmul_i(make_float2(s1 * b1.x + s2 * b2.x, s1 * b1.y + s2 * b2.y), (float)SGN);
        const float2 n2 = cmul_i(make_float2(s2 * b1.x - s1 * b2.x, s2 * b1.y - s1 * b2.y), (float)SGN);
        u[0] = cadd(u[0], cadd(a1, a2));
        u[1] = cadd(m1, n1);
        u[4] = csub(m1, n1);
        u[2] = cadd(m2, n2);
        u[3] = csub(m2, n2);
    }
};

// A B points, A and B coprime: the prime-factor map n = B n1 + A n2,
// k = B (B^-1 mod A) k1 + A (A^-1 mod B) k2 (mod AB) turns the transform
// into an A x B one without twiddles (Good 1958).
template <int A, int B, int SGN>
__device__ __forceinline__ void coprime(float2 (&u)[A * B]) {
    constexpr int N = A * B, eb = B * inverse_mod(B % A, A), ea = A * inverse_mod(A % B, B);
    float2 t[N];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
        float2 v[A];
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) v[n1] = u[(B * n1 + A * n2) % N];
        Dft<A, SGN>::run(v);
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) t[k1 * B + n2] = v[k1];
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        float2 v[B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) v[n2] = t[k1 * B + n2];
        Dft<B, SGN>::run(v);
#pragma unroll
        for (int k2 = 0; k2 < B; ++k2) u[(eb * k1 + ea * k2) % N] = v[k2];
    }
}

// multiplication by exp(SGN 2 pi i M / N), the quarter and eighth turns cheaply
template <int M, int N, int SGN>
__device__ __forceinline__ float2 turn(float2 v) {
    if constexpr (M % N == 0) return v;
    else if constexpr (4 * M == N) return cmul_i(v, (float)SGN);
    else {
        constexpr float c = (float)ccos(M, N), s = (float)SGN * (float)csin(M, N);
        return make_float2(v.x * c - v.y * s, v.x * s + v.y * c);
    }
}

// A B points by one decimation step: n = B n1 + n2, k = k1 + A k2
template <int A, int B, int SGN, int N2, int... K1>
__device__ __forceinline__ void column(const float2 (&u)[A * B], float2 (&t)[A * B],
                                       std::integer_sequence<int, K1...>) {
    float2 v[A];
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) v[n1] = u[B * n1 + N2];
    Dft<A, SGN>::run(v);
    ((t[K1 * B + N2] = turn<N2 * K1, A * B, SGN>(v[K1])), ...);
}
template <int A, int B, int SGN, int... N2>
__device__ __forceinline__ void columns(const float2 (&u)[A * B], float2 (&t)[A * B],
                                        std::integer_sequence<int, N2...>) {
    (column<A, B, SGN, N2>(u, t, std::make_integer_sequence<int, A>{}), ...);
}
template <int A, int B, int SGN>
__device__ __forceinline__ void split(float2 (&u)[A * B]) {
    float2 t[A * B];
    columns<A, B, SGN>(u, t, std::make_integer_sequence<int, B>{});
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        float2 v[B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) v[n2] = t[k1 * B + n2];
        Dft<B, SGN>::run(v);
#pragma unroll
        for (int k2 = 0; k2 < B; ++k2) u[k1 + A * k2] = v[k2];
    }
}

template <int SGN>
struct Dft<6, SGN> {
    static __device__ __forceinline__ void run(float2 (&u)[6]) { coprime<2, 3, SGN>(u); }
};
template <int SGN>
struct Dft<8, SGN> {
    static __device__ __forceinline__ void run(float2 (&u)[8]) { split<2, 4, SGN>(u); }
};
template <int SGN>
struct Dft<9, SGN> {
    static __device__ __forceinline__ void run(float2 (&u)[9]) { split<3, 3, SGN>(u); }
};
template <int SGN>
struct Dft<10, SGN> {
    static __device__ __forceinline__ void run(float2 (&u)[10]) { coprime<2, 5, SGN>(u); }
};
template <int SGN>
struct Dft<12, SGN> {
    static __device__ __forceinline__ void run(float2 (&u)[12]) { coprime<3, 4, SGN>(u); }
};
template <int SGN>
struct Dft<15, SGN> {
    static __device__ __forceinline__ void run(float2 (&u)[15]) { coprime<3, 5, SGN>(u); }
};
template <int SGN>
struct Dft<16, SGN> {
    static __device__ __forceinline__ void run(float2 (&u)[16]) { split<4, 4, SGN>(u); }
};

}  // namespace dft

// Calls op(std::integral_constant<int, R>) for a radix R <= MAXR <= 10 of the plans.
template <int MAXR, class Op>
__device__ __forceinline__ void with_radix(int R, Op &&op) {
    static_assert(MAXR <= 10, "radices of a stage that goes through LDS");
    if constexpr (MAXR > 8) {
        if (R == 9) return op(std::integral_constant<int, 9>{});
        if (R == 10) return op(std::integral_constant<int, 10>{});
    }
    if constexpr (MAXR > 6) {
        if (R == 8) return op(std::integral_constant<int, 8>{});
    }
    switch (R) {
        case 2: return op(std::integral_constant<int, 2>{});
        case 3: return op(std::integral_constant<int, 3>{});
        case 4: return op(std::integral_constant<int, 4>{});
        case 5: return op(std::integral_constant<int, 5>{});
        default: return op(std::integral_constant<int, 6>{});
    }
}

// What the stage functions take: an axis (its first, last, middle and later
// stages handed to f(radix constant, stage)), the lines of a workgroup and the
// stages in one of two forms: known at launch (the AxisRt and LinesRt of any
// mesh) or at compile time (AxisCt and LinesCt: every index map and LDS
// offset folds, which the most used meshes are worth).
template <int MAXR>
struct AxisRt {
    const LineAxis &a;
    static constexpr bool kCt = false;
    __device__ int n() const { return a.n; }
    __device__ int last_twiddles() const { return a.st[a.ns - 1].tw; }
    __device__ bool single() const { return a.ns == 1; }
    template <class F>
    __device__ __forceinline__ void stage(int s, F f) const {
        const LineStage st = a.st[s];
        with_radix<MAXR>(st.R, [&](auto r) { f(r, st); });
    }
    template <class F>
    __device__ __forceinline__ void first(F f) const { stage(0, f); }
    template <class F>
    __device__ __forceinline__ void last(F f) const { stage(a.ns - 1, f); }
    template <class F>
    __device__ __forceinline__ void middle(F f) const {
        for (int s = 1; s < a.ns - 1; ++s) stage(s, f);
    }
    template <class F>
    __device__ __forceinline__ void later(F f) const {
        for (int s = 1; s < a.ns; ++s) stage(s, f);
    }
};

template <int R_, int P, int N, int TW>
struct StageCt {
    static constexpr int R = R_, p = P, nr = N / R_, tw = TW;
};

// The axis of radices R... in this order.
template <int... R>
struct AxisList {
    static constexpr int ns = sizeof...(R);
    static constexpr int r[ns] = {R...};
    static constexpr int N = (R * ...);
    static constexpr bool kCt = true;
    static constexpr int p_of(int s) {
        int p = 1;
        for (int i = 0; i < s; ++i) p *= r[i];
        return p;
    }
    static constexpr int tw_of(int s) {
        int t = 0;
        for (int i = 0; i < s; ++i) t += p_of(i) * (r[i] - 1);
        return t;
    }
    static_assert(ns >= 2 && ns <= kMaxLineStages, "compile-time lines take two to four stages");
    __device__ static constexpr int n() { return N; }
    __device__ static constexpr bool single() { return false; }
    __device__ static constexpr int last_twiddles() { return tw_of(ns - 1); }
    template <int S, class F>
    __device__ __forceinline__ static void stage(F f) {
        f(std::integral_constant<int, r[S]>{}, StageCt<r[S], p_of(S), N, tw_of(S)>{});
    }
    template <class F>
    __device__ __forceinline__ void first(F f) const { stage<0>(f); }
    template <class F>
    __device__ __forceinline__ void last(F f) const { stage<ns - 1>(f); }
    template <class F>
    __device__ __forceinline__ void middle(F f) const {
        if constexpr (ns > 2) stage<1>(f);
        if constexpr (ns > 3) stage<2>(f);
    }
    template <class F>
    __device__ __forceinline__ void later(F f) const {
        middle(f);
        last(f);
    }
};

// The axis of line_radices(N, MAXR).
template <int N, int MAXR, class S>
struct AxisOf;
template <int N, int MAXR, int... I>
struct AxisOf<N, MAXR, std::integer_sequence<int, I...>> {
    static constexpr LineRadices v = line_radices(N, MAXR);
    using type = AxisList<v.r[I]...>;
};
template <int N, int MAXR>
using AxisCt = typename AxisOf<N, MAXR, std::make_integer_sequence<int, line_radices(N, MAXR).ns>>::type;

// `count` lines, element e of line l at buf[l * sl + e * se], worked on by
// nt() threads.  held: butterflies a thread holds in an in-place stage (at
// most ELEMS values, or as many as there are); batch: butterflies whose loads
// a first stage issues together (two where one large plane has a CU to
// itself and its own waves must cover the latency).
template <int ELEMS>
struct LinesRt {
    static constexpr bool kCt = false;
    int count, se, sl;
    float inv_count;
    __device__ static int nt() { return (int)blockDim.x; }
    template <int R, class St>
    static constexpr int held() { return ELEMS / R > 0 ? ELEMS / R : 1; }
    template <int R, class St>
    static constexpr int batch() { return ELEMS > 16 ? 2 : 1; }
};

template <int COUNT, int SE, int SL, int NT>
struct LinesCt {
    static constexpr bool kCt = true;
    static constexpr int count = COUNT, se = SE, sl = SL;
    __device__ static constexpr int nt() { return NT; }
    template <int R, class St>
    static constexpr int held() { return (COUNT * St::nr + NT - 1) / NT; }
    template <int R, class St>
    static constexpr int batch() { return held<R, St>(); }
};

template <int R, int SGN>
__device__ __forceinline__ void twiddle(float2 (&u)[R], const float2 *__restrict__ tw, int k) {
#pragma unroll
    for (int j = 1; j < R; ++j) {
        float2 w = tw[k * (R - 1) + j - 1];
        if (SGN > 0) w.y = -w.y;
        u[j] = cmul(u[j], w);
    }
}

// Butterfly b of a stage: line l, index i.  ROWS: consecutive threads take
// consecutive butterflies of a line (a line's elements are neighbours in
// global memory), else consecutive lines.
template <bool ROWS, class L, class St>
__device__ __forceinline__ void butterfly_of(int b, const L &lines, const St &st, int &l, int &i) {
    if constexpr (L::kCt) {
        l = ROWS ? b / st.nr : b % L::count;
        i = ROWS ? b % st.nr : b / L::count;
    } else if (ROWS) {
        l = divq(b, st.inv_nr);
        i = b - l * st.nr;
    } else {
        i = divq(b, lines.inv_count);
        l = b - i * lines.count;
    }
}

template <class St>
__device__ __forceinline__ int within(int i, const St &st) {  // i mod p
    if constexpr (std::is_same<St, LineStage>::value) return i - divq(i, st.inv_p) * st.p;
    else return i % St::p;
}

// First stage, results to buf (only written).  ld(line, i) gives an accessor
// whose value at d is element i + d: what depends on the line and i is formed
// once per butterfly, and d is uniform.
template <int SGN, bool ROWS, class Ax, class L, class Load>
__device__ __forceinline__ void line_first(float2 *buf, const L &lines, const Ax &ax, Load ld) {
    ax.first([&](auto r, const auto &st) {
        constexpr int R = decltype(r)::value, B = L::template batch<R, std::decay_t<decltype(st)>>();
        const int total = lines.count * st.nr;
        for (int b0 = threadIdx.x; b0 < total; b0 += B * L::nt()) {
            float2 u[B][R];
#pragma unroll
            for (int q = 0; q < B; ++q) {
                const int b = b0 + q * L::nt();
                if (B > 1 && b >= total) break;
                int l, i;
                butterfly_of<ROWS>(b, lines, st, l, i);
                const auto from = ld(l, i);
#pragma unroll
                for (int j = 0; j < R; ++j) u[q][j] = from(j * st.nr);
            }
#pragma unroll
            for (int q = 0; q < B; ++q) {
                const int b = b0 + q * L::nt();
                if (B > 1 && b >= total) break;
                int l, i;
                butterfly_of<ROWS>(b, lines, st, l, i);
                dft::Dft<R, SGN>::run(u[q]);
                float2 *d = buf + l * lines.sl + i * R * lines.se;
#pragma unroll
                for (int j = 0; j < R; ++j) d[j * lines.se] = u[q][j];
            }
        }
    });
}

// A stage in place (buf read, barrier, buf written, barrier).  FIRST: the
// stage's elements come from ld (as for line_first), which reads buf as it
// likes; else they are buf's own, with twiddles.
template <int SGN, bool ROWS, bool FIRST, class R_, class L, class St, class Load>
__device__ __forceinline__ void stage_inplace(R_, float2 *buf, const L &lines, const St &st,
                                              const float2 *__restrict__ tw, Load ld) {
    constexpr int R = R_::value, KB = L::template held<R, St>();
    const int total = lines.count * st.nr;
    float2 u[KB][R];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
        const int b = threadIdx.x + kb * L::nt();
        if (b >= total) break;
        int l, i;
        butterfly_of<ROWS>(b, lines, st, l, i);
        if constexpr (FIRST) {
            const auto from = ld(l, i);
#pragma unroll
            for (int j = 0; j < R; ++j) u[kb][j] = from(j * st.nr);
        } else {
            const float2 *s = buf + l * lines.sl + i * lines.se;
            const int step = st.nr * lines.se;
#pragma unroll
            for (int j = 0; j < R; ++j) u[kb][j] = s[j * step];
            twiddle<R, SGN>(u[kb], tw + st.tw, within(i, st));
        }
        dft::Dft<R, SGN>::run(u[kb]);
    }
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
        const int b = threadIdx.x + kb * L::nt();
        if (b >= total) break;
        int l, i;
        butterfly_of<ROWS>(b, lines, st, l, i);
        const int k = FIRST ? 0 : within(i, st);
        float2 *d = buf + l * lines.sl + ((i - k) * R + k) * lines.se;
        const int step = (FIRST ? 1 : st.p) * lines.se;
#pragma unroll
        for (int j = 0; j < R; ++j) d[j * step] = u[kb][j];
    }
    __syncthreads();
}

struct NoLoad {};

// The first stage in place, from ld.
template <int SGN, bool ROWS, class Ax, class L, class Load>
__device__ __forceinline__ void line_first_inplace(float2 *buf, const L &lines, const Ax &ax, Load ld) {
    ax.first([&](auto r, const auto &st) { stage_inplace<SGN, ROWS, true>(r, buf, lines, st, nullptr, ld); });
}

// Every stage after the first, in place (barrier after the first included).
template <int SGN, bool ROWS, class Ax, class L>
__device__ __forceinline__ void line_later(float2 *buf, const L &lines, const Ax &ax, const float2 *__restrict__ tw) {
    __syncthreads();
    ax.later([&](auto r, const auto &st) { stage_inplace<SGN, ROWS, false>(r, buf, lines, st, tw, NoLoad{}); });
}

// The stages after the first (barrier included), the last one with its
// outputs to store(line, i), an accessor called with (d, value of element
// i + d); the middle ones take consecutive lines.  An axis of one stage (a
// prime length) hands its values over.
template <int SGN, bool ROWS, class Ax, class L, class Store>
__device__ __forceinline__ void line_rest(float2 *buf, const L &lines, const Ax &ax, const float2 *__restrict__ tw,
                                          Store store) {
    __syncthreads();
    ax.middle([&](auto r, const auto &st) { stage_inplace<SGN, false, false>(r, buf, lines, st, tw, NoLoad{}); });
    if (ax.single()) {
        const int total = lines.count * ax.n();
        const float inv = 1.0f / (float)ax.n();
        for (int b = threadIdx.x; b < total; b += L::nt()) {
            const int l = divq(b, inv), e = b - l * ax.n();
            store(l, e)(0, buf[l * lines.sl + e * lines.se]);
        }
        return;
    }
    ax.last([&](auto r, const auto &st) {
        constexpr int R = decltype(r)::value;
        const int total = lines.count * st.nr;
        for (int b = threadIdx.x; b < total; b += L::nt()) {
            int l, i;
            butterfly_of<ROWS>(b, lines, st, l, i);
            const float2 *s = buf + l * lines.sl + i * lines.se;
            const int step = st.nr * lines.se;
            float2 u[R];
#pragma unroll
            for (int j = 0; j < R; ++j) u[j] = s[j * step];
            twiddle<R, SGN>(u, tw + st.tw, i);
            dft::Dft<R, SGN>::run(u);
            const auto to = store(l, i);
#pragma unroll
            for (int j = 0; j < R; ++j) to(j * st.p, u[j]);
        }
    });
}

}  // namespace hymd
