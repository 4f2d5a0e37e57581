// x-line pass (xline.h) of the x edges that fft_ct.h takes: forward x
// transform, k-space pass and the two inverse transforms per type of one
// (y, k_z) line set in one LDS buffer of T W lines; V_t waits in registers
// (PMAX positions per thread) while the -i k_x V_t family is transformed and
// stored.
#include "fft_ct.h"
#include "xline.h"

namespace hymd {

// T_ types, W_ lines per workgroup of N points.
template <int T_, int N, int W_>
struct XlineFixed {
    static constexpr int n = N, W = W_, T = T_, ld = N + 1;
    static constexpr int wshift = W_ == 1 ? 0 : W_ == 2 ? 1 : W_ == 4 ? 2 : W_ == 8 ? 3 : 4;
    // the transforms with the first stage's inputs from ld(line, e) / the last
    // stage's outputs to st(line, e, value), line = t W + l
    template <int SGN, int NT, class Load>
    __device__ void fft_from(float2 *D, const float2 *tw, Load ld) const {
        ct::fft_first_ct<N, T_ * W_, 1, N + 1, NT, SGN>(D, ld);
        ct::fft_inplace_ct<N, T_ * W_, 1, N + 1, NT, SGN, 1>(D, tw);
    }
    template <int SGN, int NT, class Store>
    __device__ void fft_to(float2 *D, const float2 *tw, Store st) const {
        ct::fft_inplace_ct<N, T_ * W_, 1, N + 1, NT, SGN, 0, ct::CtPlan<N>::v.ns - 1>(D, tw);
        ct::fft_last_ct<N, T_ * W_, 1, N + 1, NT, SGN, false>(D, tw, st);
    }
};

// PME (T = 1): the k-space pass is pme_kspace_kernel's (psi = 4 pi elec H
// rho~ / |k|^2 with the same FP64 arithmetic); outputs -i k_x psi and psi.
template <int MAXT, int NT, class G, bool PME = false>
__global__ void __launch_bounds__(NT) xline_fixed_kernel(const float2 *__restrict__ spec, float2 *__restrict__ out,
                                                         KGeom g, FieldK p, G geo,
                                                         const float2 *__restrict__ tw_glob,
                                                         double *__restrict__ partials, PmeK pk) {
    constexpr int PMAX = 16 / MAXT;
    extern __shared__ float2 smem[];
    const int n = geo.n;  // Mx
    const int W = geo.W, wshift = geo.wshift;
    const int T = geo.T;
    const int ld = geo.ld;
    float2 *tw = smem;
    float2 *D = tw + n;  // line (t W + l) at D + (t W + l) ld
    const int plane = g.my * g.zh;
    const int line0 = (int)xcd_block(blockIdx.x, gridDim.x) * W;
    const int wv = min(W, plane - line0);
    for (int i = threadIdx.x; i < n - 1; i += NT) tw[i] = tw_glob[i];
    // the forward transform's first stage reads the lines from global memory
    geo.template fft_from<-1, NT>(D, tw, [&](int line, int e) -> float2 {
        const int t = line >> wshift, l = line & (W - 1);
        return l < wv ? spec[(int64_t)t * g.gc + (int64_t)e * plane + line0 + l] : make_float2(0.f, 0.f);
    });
    // k-space pass (the arithmetic of field_kspace_kernel): V_t kept in
    // registers, -i k_x V_t written back in place
    double e_acc[1] = {0.0};
    float2 hold[PMAX][MAXT];
#pragma unroll
    for (int j = 0; j < PMAX; ++j) {
        const int pos = threadIdx.x + j * NT;
        const int l = pos & (W - 1), e = pos >> wshift;
        if (pos >= W * n || l >= wv) {
#pragma unroll
            for (int t = 0; t < MAXT; ++t) hold[j][t] = make_float2(0.f, 0.f);
            continue;
        }
        const int64_t kk = (int64_t)e * plane + line0 + l;
        double k[3], kd[3], wgt;
        kvec(g, kk, k, kd, wgt);
        if constexpr (PME) {
            double k2 = k[0] * k[0] + k[1] * k[1] + k[2] * k[2];
            const double H = exp(-0.5 * pk.sigma2 * k2);
            if (kk == 0) k2 = 1.0;
            const float2 sp = D[l * ld + e];
            const double rx = (double)sp.x * pk.inv_g, ry = (double)sp.y * pk.inv_g;
            const double f = pk.four_pi_elec * H / k2;
            const double px = f * rx, py = f * ry;
            e_acc[0] += 0.5 * wgt * (rx * px + ry * py);
            hold[j][0] = make_float2((float)px, (float)py);
            D[l * ld + e] = make_float2((float)(kd[0] * py), (float)(-kd[0] * px));
            continue;
        }
        const double k2 = k[0] * k[0] + k[1] * k[1] + k[2] * k[2];
        const float H = (float)exp(-0.5 * p.sigma2 * k2);
        const float hn = (float)((double)H * p.inv_g);
        float2 ph[MAXT];
#pragma unroll
        for (int t = 0; t < MAXT; ++t) ph[t] = t < T ? cscale(D[(t * W + l) * ld + e], hn) : make_float2(0.f, 0.f);
        if (p.want_energy) {
            double en = 0.0;
#pragma unroll
            for (int t = 0; t < MAXT; ++t) {
                if (t >= T) continue;
#pragma unroll
                for (int u = 0; u < MAXT; ++u) {
                    if (u >= T) continue;
                    en += 0.5 * p.Ad[t * HYMD_MAX_TYPES + u] *
                          ((double)ph[t].x * (double)ph[u].x + (double)ph[t].y * (double)ph[u].y);
                }
            }
            en *= wgt;
            if (kk == 0) {
#pragma unroll
                for (int t = 0; t < MAXT; ++t)
                    if (t < T) en += p.b[t] * (double)ph[t].x;
                en += p.c0;
            }
            e_acc[0] += en;
        }
        const float kx = (float)kd[0];
#pragma unroll
        for (int t = 0; t < MAXT; ++t) {
            float2 v = make_float2(0.f, 0.f);
#pragma unroll
            for (int u = 0; u < MAXT; ++u)
                if (u < T) {
                    const float a = (float)p.Ad[t * HYMD_MAX_TYPES + u];
                    v.x += a * ph[u].x;
                    v.y += a * ph[u].y;
                }
            v = cscale(v, H);
            if (kk == 0) v.x += (float)p.b[t];
            hold[j][t] = v;
            if (t < T) D[(t * W + l) * ld + e] = make_float2(kx * v.y, -kx * v.x);
        }
    }
    __syncthreads();
    // the inverse transforms' last stage writes the lines to global memory
    geo.template fft_to<1, NT>(D, tw, [&](int line, int e, float2 v) {
        const int t = line >> wshift, l = line & (W - 1);
        if (l < wv) out[(int64_t)t * g.gc + (int64_t)e * plane + line0 + l] = v;
    });
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PMAX; ++j) {
        const int pos = threadIdx.x + j * NT;
        if (pos >= W * n) continue;
        const int l = pos & (W - 1), e = pos >> wshift;
#pragma unroll
        for (int t = 0; t < MAXT; ++t)
            if (t < T) D[(t * W + l) * ld + e] = hold[j][t];
    }
    __syncthreads();
    geo.template fft_to<1, NT>(D, tw, [&](int line, int e, float2 v) {
        const int t = line >> wshift, l = line & (W - 1);
        if (l < wv) out[(int64_t)(T + t) * g.gc + (int64_t)e * plane + line0 + l] = v;
    });
    if (partials) block_reduce_store<1, NT>(e_acc, partials + blockIdx.x);
}

template <int MAXT, int NT, int T, int N, int W, bool PME>
static int launch_fixed(const FftPlan &plan, const XlineJob &job, int blocks, hipStream_t s) {
    using G = XlineFixed<T, N, W>;
    static_assert(T <= MAXT && W * N <= NT * (16 / MAXT), "every position of the W lines is held by a thread");
    const size_t lds = sizeof(float2) * ((size_t)N + (size_t)T * W * (N + 1));
    static bool done = false;  // the opt-in is per kernel and process
    if (!done && lds > 64 * 1024) {
        HYMD_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&xline_fixed_kernel<MAXT, NT, G, PME>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)kXlineLdsBytes));
        done = true;
    }
    xline_fixed_kernel<MAXT, NT, G, PME>
        <<<blocks, NT, lds, s>>>(job.spec, job.out, job.g, job.p, G{}, plan.fx, job.partials, job.pk);
    HYMD_HIP(hipGetLastError());
    return HYMD_OK;
}

int xline_pass_fixed(const FftPlan &plan, const XlineShape &sh, const XlineJob &job, int blocks, hipStream_t s) {
    const int n = plan.mesh.mx;
#define HYMD_FIXED(NX, TT, WW, MT, NT)                                \
    if (n == NX && job.T == TT && sh.W == WW && !job.pme)             \
        return launch_fixed<MT, NT, TT, NX, WW, false>(plan, job, blocks, s);
    // 512 threads at 128 points, twice the waves in flight (128^3, T = 4 33.6 ->
    // 29.8 us); at 160 that made the peptide step slower
    HYMD_FIXED(128, 1, 16, 2, 512)
    HYMD_FIXED(128, 2, 16, 2, 512)
    HYMD_FIXED(128, 3, 8, 4, 512)
    HYMD_FIXED(128, 4, 8, 4, 512)
    HYMD_FIXED(160, 1, 8, 2, 256)
    HYMD_FIXED(160, 2, 8, 2, 256)
    HYMD_FIXED(160, 3, 4, 4, 256)
    HYMD_FIXED(160, 4, 4, 4, 256)
    HYMD_FIXED(256, 1, 8, 2, 256)
    HYMD_FIXED(256, 5, 8, 8, 1024)
    HYMD_FIXED(256, 6, 8, 8, 1024)
    HYMD_FIXED(256, 7, 8, 8, 1024)
    HYMD_FIXED(256, 8, 8, 8, 1024)
    HYMD_FIXED(256, 6, 4, 8, 512)
#undef HYMD_FIXED
    if (n == 128 && job.pme) return launch_fixed<2, 512, 1, 128, 16, true>(plan, job, blocks, s);
    if (n == 160 && job.pme) return launch_fixed<2, 256, 1, 160, 8, true>(plan, job, blocks, s);
    if (n == 256 && job.pme) return launch_fixed<2, 256, 1, 256, 8, true>(plan, job, blocks, s);
    set_error("no fixed x-line pass for %d types of %d points", job.T, n);
    return HYMD_ERR_UNSUPPORTED;
}

}  // namespace hymd
