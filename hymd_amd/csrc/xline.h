// x-line pass: forward x transform, k-space pass and inverse x transforms of
// the field update (or of PME) in one kernel.
//
// A workgroup owns W consecutive (y, k_z) lines of all T spectra after their
// z and y passes.  k_y and k_z are constant along a line, so the x-inverse of
// -i k_d V_t for d = y, z is -i k_d times the x-inverse of V_t: per line and
// type two inverse transforms are needed, of -i k_x V_t -> out[t] and of V_t
// -> out[T + t]; the y-z passes apply -i k_y and -i k_z.
//
// The forward plan ends with radix R2 and the inverse plan starts with it, so
// the thread that forms a butterfly of the forward's last stage holds exactly
// the elements of one butterfly of the inverse's first stage: last stage,
// k-space mixing of the T types and first inverse stage run in registers (T R2
// complex values), and a line crosses LDS once on the way in and once per
// inverse transform.  Before, with the k-space pass between two whole LDS
// transforms of four or five stages and 16 values held per thread, the pass
// took 32 us at 100^3, T = 4 and 41 us for the PME of 150 x 144 x 160, bound by
// LDS passes and index arithmetic, not by its 8 T Gc + 16 T Gc bytes.
#pragma once
#include "fft.h"
#include "field_dev.h"

namespace hymd {

constexpr int kXlineThreads = 512;
constexpr int kXlineRadix = 10;  // largest radix of the stages that go through LDS
constexpr int kXlineElems = 16;  // values per thread of a middle stage
constexpr size_t kXlineLdsBytes = 150 * 1024;

// Lines, threads and plan (index into FftPlan::xl) of an x-line workgroup;
// W = 0: the pass does not take this mesh and number of types.
struct XlineShape {
    int W = 0, threads = 0, plan = 0;
    bool fixed = false;  // the pass of xline_fixed.hip
};
// want: lines wanted (0: any; others than the fixed pass has are the general
// pass's, where they fit); fixed: the pass of xline_fixed.hip may be taken (it
// makes the 2T inverse transforms and energies only).
XlineShape xline_shape(const FftPlan &plan, int T, int want, bool fixed);

// Lines per workgroup of the pass on fft_ct.h, 0 where there is none: x edges
// of 128 and 160 with up to four types, and 256 with one or with five and
// more, where the general pass has 2 lines (16-byte runs): 256^3, forces of 5,
// 7 and 8 types 2586, 3587 and 4934 us there, 1726, 2391 and 2955 here.
inline int xline_fixed_lines(int n, int T, int want) {
    if (n == 128 && T <= 4) return T <= 2 ? 16 : 8;
    if (n == 160 && T <= 4) return T <= 2 ? 8 : 4;
    if (n == 256 && T == 1) return 8;
    return n == 256 && T >= 5 && T <= 8 ? (want == 4 && T == 6 ? 4 : 8) : 0;
}

// Whether W lines per workgroup (runs of 8 W bytes) are too few for the pass,
// so that the separate passes (16 lines each) are the faster ones.  densities:
// the job writes spectra or densities too; transformed: it starts from held
// spectra; else it makes the force grids only.  The whole call with the pass /
// separate, us:
//   W = 1: 216^3, T = 8 2316 / 2093; 240^3, T = 8 2978 / 2643; up to two types
//     keep it: 900 x 96 x 96, T = 1 251 / 263.
//   W = 2: T = 8, 144^3 639 / 580, 160^3 687 / 645, 200^3 1539 / 1560; with
//     densities it goes either way (144^3 828 / 771, 160 x 180 x 216 1595 / 1620,
//     192^3 1603 / 1687) and they keep it, as fewer types do: T = 6, 216^3 1460 /
//     1608, 240^3 1819 / 2002.
//   Rows of 129 elements in multiples of 64, where the x stride is 2^k 129
//   elements and the pass moves 0.8 to 1.6 TB/s against 1.7 to 2.0 on every other
//   plane measured (64 to 256 rows of 33 to 161 elements; the strides seem to
//   meet on few memory channels):
//     W = 2: T = 6, 192 x 256 x 256 2305 / 1735, 240 x 256 x 256 2668 / 2228.
//     W = 4: T = 4, 192 x 256 x 256 1123 / 1175; T = 6, 100 x 256 x 256 908 / 938;
//       but where the types lie 2^k 129 elements apart as well T = 8, 128 x 256 x
//       256 2000 / 1563, T = 6, 96 x 256 x 256 951 / 896, and on long lines of
//       three types and more T = 4, 288 x 256 x 256 1945 / 1846, 320 x 256 x 256
//       2121 / 2003, 270 x 256 x 256 1731 / 1714 (T = 2, 400 x 256 x 256 1287 / 1461).
//     Held spectra, W = 2, 256^3, T = 6 2488 / 1653; W = 4, 192 x 256 x 256,
//       T = 4 874 / 825; with densities, 288 x 256 x 256, T = 4 2429 / 2306.
inline bool xline_narrow(const Mesh &m, int T, int W, bool densities, bool transformed) {
    const bool more = densities || transformed;
    const bool few_channels = m.zh == 129 && m.my % 64 == 0;
    const int least = more || (T >= 3 && m.mx >= 256) || (T >= 6 && m.mx % 32 == 0) ? 4 : 2;
    return (W == 1 && T >= 3) || (W == 2 && T >= 8 && !densities) || (few_channels && W <= least);
}

struct XlineJob {
    int T = 1;
    const float2 *spec = nullptr;  // T spectra after the z and y passes
    bool transformed = false;      // they are x-transformed too
    float2 *out = nullptr;         // 2T: IFFT_x(-i k_x V_t), IFFT_x(V_t)
    float2 *phif = nullptr;        // T filtered spectra H rho_t / G, or null
    float2 *phix = nullptr;        // T: IFFT_x of those, or null
    KGeom g;
    FieldK p{};
    bool pme = false;
    PmeK pk{};
    double *partials = nullptr;    // energy partial per workgroup, or null
};
// Runs the pass; *nblocks workgroups (partials).
int xline_pass(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int *nblocks, hipStream_t s);
// its part for T types: one per source file so that they compile side by side
using XlineLaunch = int(const FftPlan &, const XlineShape &, const XlineJob &, int, hipStream_t);
XlineLaunch xline_pass_fixed, xline_pass_pme, xline_pass_1, xline_pass_2, xline_pass_3, xline_pass_4, xline_pass_5, xline_pass_6,
    xline_pass_7, xline_pass_8;

struct XlineArgs {
    int plane;                     // lines in all
    float inv_zh;                  // 1 / (Mz/2+1)
    int transformed;
    const float2 *twf, *twi;
};

// Line geometry of a workgroup: lengths, forward and inverse axis.
struct XlineRt {
    static constexpr int threads = kXlineThreads;
    int n, W, wshift, ld;
    float inv_lines;               // 1 / (T W)
    LineAxis f, i;
    __device__ AxisRt<kXlineRadix> fwd() const { return {f}; }
    __device__ AxisRt<kXlineRadix> inv() const { return {i}; }
    template <int T>
    __device__ LinesRt<kXlineElems> lines() const { return {T * W, 1, ld, inv_lines}; }
};

// Sum of one double over the workgroup, in a fixed order, into *out.
__device__ __forceinline__ void block_sum_store(double v, double *out) {
    __shared__ double red[kXlineThreads / 64];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += red[w];
        *out = t;
    }
}

// A copy of v that the compiler takes for a new value: what is derived from it
// is formed where it is used instead of being kept across the phases of the
// kernel (the element indices and k_x of R2 elements would hold 40 registers).
__device__ __forceinline__ int fresh(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// Waves per SIMD that the registers allow: four where they suffice; the 15 and
// 16 elements of psi and of -i k_x psi of a PME thread spilled 36 to 60 bytes a
// lane at four (150 x 144 x 160 21.0 us), and are faster at three (18.4).
constexpr int xline_waves(int T, int R2, bool pme) {
    return T * R2 > 16 ? 1 : (pme && R2 > 12 ? 3 : 4);
}

template <int T, int R2, bool PME, class G>
__global__ void __launch_bounds__(G::threads, xline_waves(T, R2, PME))
    xline_kernel(const float2 *__restrict__ spec, float2 *__restrict__ out, float2 *__restrict__ phif,
                 float2 *__restrict__ phix, XlineArgs a, G geo, KGeom g, FieldK p, PmeK pk,
                 double *__restrict__ partials) {
    extern __shared__ double smem_d[];
    const int n = geo.n, W = geo.W, ld = geo.ld, nr2 = n / R2;
    double *ex = smem_d;                          // filter factor exp(-sigma^2 k_x^2 / 2) of element e
    float2 *twf = (float2 *)(ex + n), *twi = twf + n;
    float2 *D = twi + n;                          // line (t W + l) at D + (t W + l) ld
    const int line0 = (int)xcd_block(blockIdx.x, gridDim.x) * W;
    const int wv = min(W, a.plane - line0);
    const double half_s2 = -0.5 * (PME ? pk.sigma2 : p.sigma2);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        if (i < n - 1) {
            twf[i] = a.twf[i];
            twi[i] = a.twi[i];
        }
        const double kx = g.kfac[0] * (2 * i < n ? i : i - n);
        ex[i] = exp(half_s2 * (kx * kx));
    }
    const auto lines = geo.template lines<T>();
    const auto af = geo.fwd();
    const auto ai = geo.inv();
    if (!a.transformed) {
        line_first<-1, false>(D, lines, af, [&](int ln, int e) {
            const int ll = ln & (W - 1);
            const float2 *q = spec + (int64_t)(ln >> geo.wshift) * g.gc + (int64_t)e * a.plane + line0 + ll;
            const bool ok = ll < wv;
            return [q, ok, &a](int d) { return ok ? q[(int64_t)d * a.plane] : make_float2(0.f, 0.f); };
        });
        __syncthreads();
        af.middle([&](auto r, const auto &st) { stage_inplace<-1, false, false>(r, D, lines, st, twf, NoLoad{}); });
    } else {
        __syncthreads();
    }
    // the forward transform's last stage: u[t][j] is element i + j n / R2 of line l, type t
    const int l = (int)threadIdx.x & (W - 1), i = (int)threadIdx.x >> geo.wshift;
    const bool active = i < nr2;
    float2 u[T][R2];
    if (active) {
        const float2 *tw = twf + af.last_twiddles();
#pragma unroll
        for (int t = 0; t < T; ++t) {
            if (a.transformed) {
#pragma unroll
                for (int j = 0; j < R2; ++j)
                    u[t][j] = l < wv ? spec[(int64_t)t * g.gc + (int64_t)(i + j * nr2) * a.plane + line0 + l]
                                     : make_float2(0.f, 0.f);
            } else {
                const float2 *s = D + (t * W + l) * ld + i;
#pragma unroll
                for (int j = 0; j < R2; ++j) u[t][j] = s[j * nr2];
                twiddle<R2, -1>(u[t], tw, i);
                dft::Dft<R2, -1>::run(u[t]);
            }
        }
    }
    const int line = min(line0 + l, a.plane - 1), iy = divq(line, a.inv_zh), iz = line - iy * g.zh;
    const double ky = g.kfac[1] * (2 * iy < g.my ? iy : iy - g.my), kz = g.kfac[2] * iz;
    const double kyz2 = ky * ky + kz * kz, eyz = exp(half_s2 * kyz2);
    const double wgt = (iz == 0 || 2 * iz == g.mz) ? 1.0 : 2.0;
    // k_x of element e of the derivative (zero on the Nyquist plane)
    auto kdx = [&](int e) -> float { return 2 * e == n ? 0.f : (float)(g.kfac[0] * (2 * e < n ? e : e - n)); };
    double energy = 0.0;
    float2 dx[PME ? R2 : 1];  // PME: -i k_x psi
    if constexpr (PME) {
        // psi = 4 pi k_e / eps H rho / |k|^2 (|k|^2 := 1 at k = 0) and -i k_x psi, in FP64
        if (active) {
#pragma unroll
            for (int j = 0; j < R2; ++j) {
                const int e = fresh(i) + j * nr2;
                const double kx = g.kfac[0] * (2 * e < n ? e : e - n);
                double k2 = kx * kx + kyz2;
                if (line0 + l == 0 && e == 0) k2 = 1.0;
                const double f = pk.four_pi_elec * (ex[e] * eyz) / k2;
                const double rx = (double)u[0][j].x * pk.inv_g, ry = (double)u[0][j].y * pk.inv_g;
                const double px = f * rx, py = f * ry, kd = 2 * e == n ? 0.0 : kx;
                if (l < wv) energy += 0.5 * wgt * (rx * px + ry * py);
                u[0][j] = make_float2((float)px, (float)py);
                dx[j] = make_float2((float)(kd * py), (float)(-kd * px));
            }
        }
    } else {
        if (active) {
#pragma unroll
            for (int j = 0; j < R2; ++j) {
                const int e = fresh(i) + j * nr2;
                const float H = (float)(ex[e] * eyz);
                const float hn = (float)((double)H * p.inv_g);
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    u[t][j] = cscale(u[t][j], hn);
                    if (phif && l < wv) phif[(int64_t)t * g.gc + (int64_t)e * a.plane + line0 + l] = u[t][j];
                }
                if (p.want_energy && l < wv) {
                    double en = 0.0;
#pragma unroll
                    for (int t = 0; t < T; ++t)
#pragma unroll
                        for (int s = 0; s < T; ++s)
                            en += 0.5 * p.Ad[t * HYMD_MAX_TYPES + s] *
                                  ((double)u[t][j].x * (double)u[s][j].x + (double)u[t][j].y * (double)u[s][j].y);
                    en *= wgt;
                    if (line0 + l == 0 && e == 0) {
#pragma unroll
                        for (int t = 0; t < T; ++t) en += p.b[t] * (double)u[t][j].x;
                        en += p.c0;
                    }
                    energy += en;
                }
            }
        }
    }
    // the inverse transforms, family by family (one copy of the code): 0 the
    // filtered spectra themselves, 1 -i k_x V_t, 2 V_t
#pragma unroll 1
    for (int f = phix ? 0 : 1; f < 3; ++f) {
        if (!PME && f == 1 && active) {  // u <- V
#pragma unroll
            for (int j = 0; j < R2; ++j) {
                const int e = fresh(i) + j * nr2;
                const float H = (float)(ex[e] * eyz);
                float2 v[T];
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    v[t] = make_float2(0.f, 0.f);
#pragma unroll
                    for (int s = 0; s < T; ++s) {
                        const float A = p.Af[t * HYMD_MAX_TYPES + s];
                        v[t].x += A * u[s][j].x;
                        v[t].y += A * u[s][j].y;
                    }
                    v[t] = cscale(v[t], H);
                    if (line0 + l == 0 && e == 0) v[t].x += (float)p.b[t];
                }
#pragma unroll
                for (int t = 0; t < T; ++t) u[t][j] = v[t];
            }
        }
        __syncthreads();  // the last reads of D are done
        if (active) {
            float kx[R2];
            const int fi = fresh(i);
#pragma unroll
            for (int j = 0; j < R2; ++j) kx[j] = !PME && f == 1 ? kdx(fi + j * nr2) : 0.f;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                float2 c[R2];
#pragma unroll
                for (int j = 0; j < R2; ++j) {
                    if constexpr (PME) c[j] = f == 1 ? dx[j] : u[t][j];
                    else c[j] = f == 1 ? make_float2(kx[j] * u[t][j].y, -kx[j] * u[t][j].x) : u[t][j];
                }
                dft::Dft<R2, 1>::run(c);
                float2 *d = D + (t * W + l) * ld + i * R2;
#pragma unroll
                for (int j = 0; j < R2; ++j) d[j] = c[j];
            }
        }
        float2 *dst = f == 0 ? phix : out + (f == 2 ? (int64_t)T * g.gc : 0);
        line_rest<1, false>(D, lines, ai, twi, [&](int ln, int e) {
            const int ll = ln & (W - 1);
            float2 *q = dst + (int64_t)(ln >> geo.wshift) * g.gc + (int64_t)e * a.plane + line0 + ll;
            const bool ok = ll < wv;
            return [q, ok, &a](int d, float2 w) {
                if (ok) q[(int64_t)d * a.plane] = w;
            };
        });
    }
    if (partials) {
        __syncthreads();
        block_sum_store(energy, partials + blockIdx.x);
    }
}

// LDS bytes of a workgroup of W lines of n points and T types.
inline size_t xline_lds(int n, int T, int W) {
    return (sizeof(double) + 2 * sizeof(float2)) * (size_t)n + sizeof(float2) * (size_t)T * W * (n | 1);
}

template <int T, int R2, bool PME, class G>
int launch_xline_geo(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, const G &geo,
                     hipStream_t s) {
    const XlineAxes &x = plan.xl[sh.plan];
    const size_t lds = xline_lds(plan.mesh.mx, T, sh.W);
    static bool done = false;  // the opt-in is per kernel and process
    if (!done && lds > 64 * 1024) {
        HYMD_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&xline_kernel<T, R2, PME, G>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)kXlineLdsBytes));
        done = true;
    }
    const XlineArgs a{job.g.my * job.g.zh, 1.0f / (float)job.g.zh, job.transformed ? 1 : 0, x.twf, x.twi};
    xline_kernel<T, R2, PME, G><<<blocks, sh.threads, lds, s>>>(job.spec, job.out, job.phif, job.phix, a, geo, job.g,
                                                                job.p, job.pk, job.partials);
    HYMD_HIP(hipGetLastError());
    return HYMD_OK;
}

template <int T, int R2, bool PME>
int launch_xline(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, hipStream_t s) {
    const XlineAxes &x = plan.xl[sh.plan];
    const int n = plan.mesh.mx;
    int wshift = 0;
    while ((1 << wshift) < sh.W) ++wshift;
    const XlineRt geo{n, sh.W, wshift, n | 1, 1.0f / (float)(T * sh.W), x.fwd, x.inv};
    return launch_xline_geo<T, R2, PME>(plan, sh, job, blocks, geo, s);
}

// The launch for the plan's last radix among RS.
template <int T, bool PME, int... RS>
int launch_xline_radix(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, hipStream_t s) {
    const LineAxis &ax = plan.xl[sh.plan].fwd;
    const int R = ax.st[ax.ns - 1].R;
    int st = HYMD_ERR_UNSUPPORTED;
    if (!((R == RS && ((st = launch_xline<T, RS, PME>(plan, sh, job, blocks, s)), true)) || ...))
        set_error("no x-line pass for %d types with last radix %d", T, R);
    return st;
}

}  // namespace hymd
