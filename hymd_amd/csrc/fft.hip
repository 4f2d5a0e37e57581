// FFT kernels: packed r2c / c2r along z, complex passes along y and x.
#include <algorithm>
#include <cmath>
#include <vector>

#include "fft.h"
#include "fft_ct.h"

namespace hymd {

// ---------------------------------------------------------------------------
// plans
// ---------------------------------------------------------------------------

constexpr int kCus = 256;
constexpr int kLineRadix = 10;      // largest radix of a line's stages
// values per thread of an in-place stage: of the line passes, of the z rows'
// kernels (2048 values on 256 threads), of a large plane
constexpr int kLineElems = 16;
constexpr int kRowElems = 12;
constexpr int kPlaneElemsBig = 24;

// The stages of a plan; their forward twiddles appended to `host`.
static LineAxis make_line(int n, const LineRadices &rs, std::vector<float2> &host) {
    LineAxis ax{};
    ax.n = n;
    ax.ns = rs.ns;
    int p = 1, off = 0;
    for (int s = 0; s < ax.ns; ++s) {
        const int R = rs.r[s];
        ax.st[s] = LineStage{R, p, n / R, off, 1.0f / (float)p, 1.0f / (float)(n / R)};
        for (int k = 0; k < p; ++k)
            for (int j = 1; j < R; ++j) {
                const double ang = -2.0 * M_PI * (double)(j * k) / (double)(p * R);
                host.push_back(make_float2((float)cos(ang), (float)sin(ang)));
            }
        off += p * (R - 1);
        p *= R;
    }
    return ax;
}

// The forward radices of an x-line pass whose last one is at most `cap`:
// fewest stages, then the first of `last` that allows them (a small last radix
// means many threads per line and few registers, radix 2 and 3 gain little);
// ns = 0 for a line of one stage.
static LineRadices xline_radices(int n, int cap) {
    static const int last[] = {4, 5, 6, 8, 3, 10, 12, 15, 16};
    for (int stages = 2; stages <= kMaxLineStages; ++stages)
        for (int r : last) {
            LineRadices p{};
            if (r > cap || n % r != 0 || n == r || !line_radices_find(p, 0, stages - 1, n / r, kLineRadix)) continue;
            p.r[stages - 1] = r;
            p.ns = stages;
            return p;
        }
    return LineRadices{};
}

// Whether the stages [first, last) run in place on nlines lines fit `threads`
// threads of at most `elems` values.
static bool stages_fit(const LineAxis &ax, int nlines, int threads, int elems, int first, int last) {
    for (int s = first; s < last; ++s)
        if ((int64_t)nlines * ax.st[s].nr > (int64_t)threads * std::max(1, elems / ax.st[s].R)) return false;
    return true;
}

static bool line_fits(const LineAxis &ax, int nlines, int threads, int elems) {
    return stages_fit(ax, nlines, threads, elems, 0, ax.ns);
}

// Lines per workgroup of a strided pass: 16 (128 contiguous bytes per element
// row), fewer where the middle stages or LDS do not take them.
static int strided_width(const LineAxis &ax) {
    for (int W = 16; W > 1; W >>= 1) {
        const size_t lds = sizeof(float2) * ((size_t)ax.n + (size_t)W * (ax.n | 1));
        if (lds <= 64 * 1024 && (ax.ns <= 2 || line_fits(ax, W, kBlock, kLineElems))) return W;
    }
    return 1;
}

static bool plane_fits(const FftPlan &plan, int threads, int elems) {
    return line_fits(plan.ly, plan.mesh.zh, threads, elems) && line_fits(plan.lzh, plan.mesh.my, threads, elems);
}

// The same for one direction: its first axis' first stage and its second axis'
// last one do not run in place (an axis of one stage runs that one).
static bool plane_fits(const FftPlan &plan, int threads, int elems, bool inverse) {
    const LineAxis &a = inverse ? plan.ly : plan.lzh, &b = inverse ? plan.lzh : plan.ly;
    const int na = inverse ? plan.mesh.zh : plan.mesh.my, nb = inverse ? plan.mesh.my : plan.mesh.zh;
    return stages_fit(a, na, threads, elems, 1, a.ns) &&
           stages_fit(b, nb, threads, elems, 0, std::max(1, b.ns - 1));
}

// Whether the y-z planes have a kernel compiled for their size (with_plane).
static bool plane_ct(const Mesh &m) {
    return m.my == m.mz && (m.my == 48 || m.my == 64 || m.my == 96);
}

// Whether they run on the fixed radices of fft_ct.h.
static bool plane_fixed(const Mesh &m) { return m.my == m.mz && (m.my == 128 || m.my == 160); }

// Twiddles of the stages of fft_ct.h for n points (128, 160 or 256), appended to host.
static void fixed_tables(int n, std::vector<float2> &host) {
    const ct::StagePlan sp = ct::make_stage_plan(n);
    LineRadices rs{};
    rs.ns = sp.ns;
    for (int s = 0; s < sp.ns; ++s) rs.r[s] = sp.r[s];
    make_line(n, rs, host);
}

// The x and y edges taken: those whose lines, 16 at a time (8 from 256 points
// on, 4 from 512), fit 64 KB twice; 250, 486, 500 and above 909 are not.
static bool edge_taken(int n) {
    const int W = n >= 512 ? 4 : (n >= 256 ? 8 : 16);
    return sizeof(float2) * ((size_t)n + 2 * (size_t)W * (n + 1)) <= 64 * 1024;
}

int fft_plan_init(FftPlan &plan, const Mesh &mesh) {
    plan.mesh = mesh;
    if (mesh.mz % 2 != 0) {
        set_error("mesh edge along z must be even (got %d)", mesh.mz);
        return HYMD_ERR_UNSUPPORTED;
    }
    const int nh = mesh.mz / 2;
    std::vector<float2> host;
    size_t at[4 + 2 * kXlinePlans];
    const int len[3] = {mesh.mx, mesh.my, nh};
    LineAxis *axis[3] = {&plan.lx, &plan.ly, &plan.lzh};
    for (int d = 0; d < 3; ++d) {
        const LineRadices rs = line_radices(len[d], kLineRadix);
        if (rs.ns == 0) {
            set_error("FFT length %d is not of the form 2^a 3^b 5^c", len[d]);
            return HYMD_ERR_UNSUPPORTED;
        }
        at[d] = host.size();
        *axis[d] = make_line(len[d], rs, host);
    }
    at[3] = host.size();
    for (int k = 0; k < mesh.zh; ++k) {
        const double ang = -2.0 * M_PI * (double)k / (double)mesh.mz;
        host.push_back(make_float2((float)cos(ang), (float)sin(ang)));
    }
    for (int c = 0; c < kXlinePlans; ++c) {
        // T = 1, 2; 3; 4; 5; 6; 7, 8 (the launches of xline*.hip list what can come out): T times the
        // last radix complex values sit in registers, at most 40
        static const int cap[kXlinePlans] = {16, 8, 6, 6, 5, 5};
        const LineRadices f = xline_radices(mesh.mx, cap[c]);
        LineRadices r = f;
        std::reverse(r.r, r.r + r.ns);
        at[4 + 2 * c] = host.size();
        plan.xl[c].fwd = make_line(mesh.mx, f, host);
        at[5 + 2 * c] = host.size();
        plan.xl[c].inv = make_line(mesh.mx, r, host);
    }
    const size_t fx = host.size();
    if (xline_fixed_edge(mesh.mx)) fixed_tables(mesh.mx, host);
    const size_t fy = host.size();
    if (plane_fixed(mesh)) fixed_tables(mesh.my, host);
    const size_t fzh = host.size();
    if (plane_fixed(mesh)) fixed_tables(nh, host);
    HYMD_TRY(plan.tables.reserve(sizeof(float2) * host.size()));
    HYMD_HIP(hipMemcpy(plan.tables.ptr, host.data(), sizeof(float2) * host.size(), hipMemcpyHostToDevice));
    const float2 *base = (const float2 *)plan.tables.ptr;
    plan.tx = base + at[0];
    plan.ty = base + at[1];
    plan.tzh = base + at[2];
    plan.post = base + at[3];
    plan.fx = base + fx;
    plan.fy = base + fy;
    plan.fzh = base + fzh;
    for (int c = 0; c < kXlinePlans; ++c) {
        plan.xl[c].twf = base + at[4 + 2 * c];
        plan.xl[c].twi = base + at[5 + 2 * c];
    }
    plan.wx = strided_width(plan.lx);
    plan.wy = strided_width(plan.ly);
    plan.wz = std::max(1, 2048 / nh);
    while (plan.wz > 1 && !line_fits(plan.lzh, plan.wz, kBlock, kRowElems)) plan.wz /= 2;
    plan.zhs = mesh.zh | 1;
    // y-z plane kernels: twiddles (y, z half), post twiddles, one My x zh plane
    plan.lds_plane = sizeof(float2) * ((size_t)mesh.my + (size_t)nh + (size_t)mesh.zh + (size_t)mesh.my * plan.zhs);
    if (plan.lds_plane > kPlaneLdsBytes || !plane_fits(plan, 1024, kPlaneElemsBig)) plan.lds_plane = 0;
    if (!edge_taken(mesh.mx) || !edge_taken(mesh.my)) {
        set_error("mesh too large for the LDS-staged FFT");
        return HYMD_ERR_UNSUPPORTED;
    }
    return HYMD_OK;
}

// ---------------------------------------------------------------------------
// shared element maps
// ---------------------------------------------------------------------------

// The real-FFT split of rows of packed transforms Z (indices mod nh):
// X[m] = (Z[m] + Z*[nh-m])/2 + post[m] (Z[m] - Z*[nh-m])/(2i), post[m] =
// exp(-2 pi i m / Mz), of the row `off` elements on.
struct RealSplit {
    const float2 *a, *c;
    float2 w;
    __device__ RealSplit(const float2 *row, const float2 *post, int m, int nh)
        : a(row + (m == nh ? 0 : m)), c(row + (m == 0 ? 0 : nh - m)), w(post[m]) {}
    __device__ float2 operator()(int off) const {
        const float2 zm = a[off], zc = cconj(c[off]);
        return cadd(cscale(cadd(zm, zc), 0.5f), cmul(w, cmul_i(csub(zm, zc), -0.5f)));
    }
};

// -i k v for a derivative factor k, zero on its Nyquist plane, in FP32 or (wide)
// in FP64
__device__ __forceinline__ float2 mul_minus_i(float2 v, double k, bool nyquist, bool wide) {
    if (wide) {
        const double kd = nyquist ? 0.0 : k;
        return make_float2((float)(kd * (double)v.y), (float)(-kd * (double)v.x));
    }
    const float kd = nyquist ? 0.f : (float)k;
    return make_float2(kd * v.y, -kd * v.x);
}

// Its inverse: Z'[m] = (X[m] + X*[nh-m]) + i conj(post[m]) (X[m] - X*[nh-m])
__device__ __forceinline__ float2 real_join(const float2 *row, const float2 *post, int m, int nh) {
    const float2 xm = row[m], xc = cconj(row[nh - m]);
    return cadd(cadd(xm, xc), cmul_i(cmul(cconj(post[m]), csub(xm, xc)), 1.f));
}

// One grid of a YzJob: where it comes from and goes to.
struct YzGrid {
    const float2 *src;
    float *dst;
    bool dy, dz, wide;
    double kfy, kfz;
};

// kinds: the job's grids of one type in order, 3 bits each (0-2 gradient
// along x, y, z; 3 real_v; 4 real2)
// grid0: the first grid of a launch that takes some of them (the line passes).
struct YzArgs {
    YzJob job;
    int nkinds, kinds, grid0;
    int64_t g, gc;
};

// Grid d of type t (counted through the systems).
__device__ __forceinline__ YzGrid yz_grid(const YzArgs &a, int t, int d) {
    const int kind = (a.kinds >> (3 * d)) & 7;
    const int sys = a.job.systems > 1 ? t / a.job.T : 0;
    YzGrid q;
    q.src = kind == 4 ? a.job.in2 + (int64_t)t * a.gc
                      : a.job.in + (int64_t)(sys * a.job.T + t + (kind == 0 ? 0 : a.job.T)) * a.gc;
    q.dst = kind == 4 ? a.job.real2 + (int64_t)t * a.g
                      : (kind == 3 ? a.job.real_v + (int64_t)t * a.g : a.job.force + (int64_t)(3 * t + kind) * a.g);
    q.dy = kind == 1;
    q.dz = kind == 2;
    q.wide = a.job.wide;
    q.kfy = a.job.kf ? a.job.kf[sys].x : a.job.kfy;
    q.kfz = a.job.kf ? a.job.kf[sys].y : a.job.kfz;
    return q;
}

static YzArgs yz_args(const FftPlan &plan, const YzJob &job) {
    YzArgs a{job, 0, 0, 0, plan.mesh.g, plan.mesh.gc};
    auto add = [&](int kind) { a.kinds |= kind << (3 * a.nkinds++); };
    if (job.force)
        for (int k = 0; k < 3; ++k) add(k);
    if (job.real_v) add(3);
    if (job.real2) add(4);
    return a;
}

// What a YzJob's grid makes of element (y, kz) on its way into the y
// transform: -i k_y v or -i k_z v for those gradients (k_z is constant along
// the y line, so its factor commutes with the transform; both zero on their
// Nyquist planes).
struct YzFactor {
    bool dy, dz, wide, nyquist;
    int y, my;
    double kfy, kz;
    __device__ YzFactor(const YzGrid &q, int y_, int m, int my_, int nh)
        : dy(q.dy), dz(q.dz), wide(q.wide), nyquist(m == nh), y(y_), my(my_), kfy(q.kfy), kz(q.kfz * m) {}
    __device__ float2 operator()(float2 v, int d) const {
        if (dy) {
            const int yy = y + d;
            return mul_minus_i(v, kfy * (2 * yy < my ? yy : yy - my), 2 * yy == my, wide);
        }
        return dz ? mul_minus_i(v, kz, nyquist, wide) : v;
    }
};

// ---------------------------------------------------------------------------
// y-z plane kernels: one workgroup per (x-plane, grid) holds the plane's My x
// (Mz/2+1) half spectrum in LDS (row stride zhs, odd: a column's elements hit
// different banks) and runs the z and y transforms there.  Each transform's
// first and last stages read and write global memory where the plane enters
// and leaves, and the real-FFT split / join is formed element by element in
// the stage that follows it, so with two-stage axes a plane crosses LDS three
// times.
// ---------------------------------------------------------------------------
struct PlaneTables {
    const float2 *twy, *twz, *post;
};

// Any mesh: sizes, plans and strides known at launch.
template <int ELEMS>
struct PlaneRt {
    static constexpr int threads = 1024, waves = ELEMS <= 16 ? 6 : 4;  // 80 and 128 registers
    int mx, my, nh, zh, zhs;
    float inv_my, inv_zh;
    LineAxis ay, az;
    PlaneTables t;
    using L = LinesRt<ELEMS>;
    __device__ AxisRt<kLineRadix> y() const { return {ay}; }
    __device__ AxisRt<kLineRadix> z() const { return {az}; }
    __device__ L rows() const { return L{my, 1, zhs, inv_my}; }
    __device__ L cols() const { return L{zh, zhs, 1, inv_zh}; }
    __device__ static int nt() { return (int)blockDim.x; }
};

// My x Mz at compile time, NT threads held to WAVES waves per SIMD.
template <int MY, int MZ, int NT, int WAVES = 1>
struct PlaneCt {
    static constexpr int threads = NT, waves = WAVES;
    static constexpr int my = MY, nh = MZ / 2, zh = MZ / 2 + 1, zhs = zh | 1;
    int mx;
    PlaneTables t;
    __device__ AxisCt<MY, kLineRadix> y() const { return {}; }
    __device__ AxisCt<MZ / 2, kLineRadix> z() const { return {}; }
    __device__ LinesCt<MY, 1, zhs, NT> rows() const { return {}; }
    __device__ LinesCt<zh, zhs, 1, NT> cols() const { return {}; }
    __device__ static constexpr int nt() { return NT; }
};

// The planes of fft_ct.h, NT threads held to at least WPE waves per SIMD (the
// register budget).  160 x 160 (a 104 KB plane: one workgroup per CU) runs 16
// waves per CU instead of 8 with 512 threads; 128 x 128 (66.5 KB: two per CU)
// 32 instead of 16 when held to 64 VGPRs (WPE 8; the c2r pass then keeps 12
// B/lane in scratch and is still faster: 0.3637 -> 0.3616 ms per lipid/water
// outer step).
template <int MY, int MZ, int NT, int WPE>
struct PlaneFixed {
    static constexpr int threads = NT, waves = WPE;
    static constexpr int my = MY, nh = MZ / 2, zh = MZ / 2 + 1;
    int mx;
    PlaneTables t;
    __device__ static constexpr int nt() { return NT; }
};

struct PlaneLds {
    float2 *twy, *twz, *post, *D;
};

template <class G>
__device__ __forceinline__ PlaneLds plane_lds(float2 *smem, const G &g) {
    PlaneLds s{smem, smem + g.my, smem + g.my + g.nh, smem + g.my + g.nh + g.zh};
    for (int i = threadIdx.x; i < g.my - 1; i += G::nt()) s.twy[i] = g.t.twy[i];
    for (int i = threadIdx.x; i < g.nh - 1; i += G::nt()) s.twz[i] = g.t.twz[i];
    for (int i = threadIdx.x; i < g.zh; i += G::nt()) s.post[i] = g.t.post[i];
    return s;
}

// forward: My rows of Mz reals -> packed complex FFT of Mz/2 per row + split
// -> FFT along y of the Mz/2+1 columns -> out plane
template <class G>
__global__ void __launch_bounds__(G::threads, G::waves) r2c_zy_plane_kernel(const float *__restrict__ in,
                                                                            float2 *__restrict__ out, G g) {
    extern __shared__ float2 smem[];
    const PlaneLds s = plane_lds(smem, g);
    const unsigned flat = xcd_block(blockIdx.x, gridDim.x);  // grid * Mx + x
    const float2 *src = reinterpret_cast<const float2 *>(in) + (int64_t)flat * g.my * g.nh;
    float2 *dst = out + (int64_t)flat * g.my * g.zh;
    line_first<-1, true>(s.D, g.rows(), g.z(), [&](int y, int k) {
        const float2 *q = src + y * g.nh + k;
        return [q](int d) { return q[d]; };
    });
    line_later<-1, false>(s.D, g.rows(), g.z(), s.twz);
    line_first_inplace<-1, false>(s.D, g.cols(), g.y(), [&](int kz, int y) {
        const RealSplit q(s.D + y * g.zhs, s.post, kz, g.nh);
        return [q, &g](int d) { return q(d * g.zhs); };
    });
    line_rest<-1, false>(s.D, g.cols(), g.y(), s.twy, [&](int kz, int y) {
        float2 *q = dst + y * g.zh + kz;
        return [q, &g](int d, float2 v) { q[d * g.zh] = v; };
    });
}

// inverse: the planes of a YzJob.  Block (t Mx + x) nkinds + d: the planes
// that read in[T + t] are neighbours, so L2 serves all reads but the first.
template <class G>
__global__ void __launch_bounds__(G::threads, G::waves) c2r_yz_plane_kernel(YzArgs a, G g) {
    extern __shared__ float2 smem[];
    const PlaneLds s = plane_lds(smem, g);
    const int flat = (int)xcd_block(blockIdx.x, gridDim.x);
    const int rest = flat / a.nkinds, t = rest / g.mx, x = rest - t * g.mx;
    const YzGrid q = yz_grid(a, t, flat - rest * a.nkinds);
    const float2 *src = q.src + (int64_t)x * g.my * g.zh;
    float2 *dst = reinterpret_cast<float2 *>(q.dst) + (int64_t)x * g.my * g.nh;
    line_first<1, false>(s.D, g.cols(), g.y(), [&](int kz, int y) {
        const float2 *p = src + y * g.zh + kz;
        const YzFactor w(q, y, kz, g.my, g.nh);
        return [p, w, &g](int d) { return w(p[d * g.zh], d); };
    });
    line_later<1, false>(s.D, g.cols(), g.y(), s.twy);
    line_first_inplace<1, false>(s.D, g.rows(), g.z(),
                                 [&](int y, int m) {
        const float2 *row = s.D + y * g.zhs;
        return [row, m, &s, &g](int d) { return real_join(row, s.post, m + d, g.nh); };
    });
    const float scale = a.job.scale;
    line_rest<1, true>(s.D, g.rows(), g.z(), s.twz, [&](int y, int k) {
        float2 *p = dst + y * g.nh + k;
        return [p, scale](int d, float2 v) { p[d] = make_float2(v.x * scale, v.y * scale); };
    });
}

// The same two passes on fft_ct.h (row stride zh, odd at these sizes).
template <int MY, int MZ, int NT, int WPE>
__global__ void __launch_bounds__(NT, WPE)
    r2c_zy_plane_kernel_fixed(const float *__restrict__ in, float2 *__restrict__ out, PlaneFixed<MY, MZ, NT, WPE> g) {
    extern __shared__ float2 smem[];
    constexpr int my = MY, nh = MZ / 2, zh = MZ / 2 + 1;
    const PlaneLds s = plane_lds(smem, g);
    const unsigned flat = xcd_block(blockIdx.x, gridDim.x);  // grid * Mx + x
    const float2 *src = reinterpret_cast<const float2 *>(in) + (int64_t)flat * my * nh;
    float2 *dst = out + (int64_t)flat * my * zh;
    ct::fft_first_ct<nh, MY, 1, zh, NT, -1, true>(s.D, [&](int y, int k) -> float2 { return src[y * nh + k]; });
    ct::fft_inplace_ct<nh, MY, 1, zh, NT, -1, 1>(s.D, s.twz);
    ct::fft_first_ct_inplace<MY, zh, zh, 1, NT, -1, false>(s.D, [&](int kz, int y) -> float2 {
        const float2 *row = s.D + y * zh;
        const float2 zm = row[kz == nh ? 0 : kz], zc = row[kz == 0 ? 0 : nh - kz];
        const float2 a = cscale(cadd(zm, cconj(zc)), 0.5f);
        const float2 b = cmul_i(csub(zm, cconj(zc)), -0.5f);
        return cadd(a, cmul(s.post[kz], b));
    });
    ct::fft_inplace_ct<MY, zh, zh, 1, NT, -1, 1, ct::CtPlan<MY>::v.ns - 1>(s.D, s.twy);
    ct::fft_last_ct<MY, zh, zh, 1, NT, -1, false>(s.D, s.twy,
                                                  [&](int kz, int y, float2 v) { dst[y * zh + kz] = v; });
}

// WIDE: of the job (in FP64 where the job asks, by a kernel of its own: as a
// runtime choice it cost the 128^2 planes 2 %).
template <int MY, int MZ, int NT, int WPE, bool WIDE>
__global__ void __launch_bounds__(NT, WPE) c2r_yz_plane_kernel_fixed(YzArgs a, PlaneFixed<MY, MZ, NT, WPE> g) {
    extern __shared__ float2 smem[];
    constexpr int my = MY, mz = MZ, nh = MZ / 2, zh = MZ / 2 + 1;
    const PlaneLds s = plane_lds(smem, g);
    const int flat = (int)xcd_block(blockIdx.x, gridDim.x);
    const int rest = flat / a.nkinds, t = rest / g.mx, x = rest - t * g.mx;
    const YzGrid q = yz_grid(a, t, flat - rest * a.nkinds);
    const float2 *src = q.src + (int64_t)x * my * zh;
    ct::fft_first_ct<MY, zh, zh, 1, NT, 1>(s.D, [&](int kz, int y) -> float2 {
        float2 w = src[y * zh + kz];
        if (q.dy) {  // row y: k_y, zero on the Nyquist row
            const int ny = 2 * y < my ? y : y - my;
            w = mul_minus_i(w, q.kfy * ny, 2 * y == my, WIDE);
        }
        return w;
    });
    ct::fft_inplace_ct<MY, zh, zh, 1, NT, 1, 1>(s.D, s.twy);
    float2 *dst = reinterpret_cast<float2 *>(q.dst) + (int64_t)x * my * nh;
    const float scale = a.job.scale;
    ct::fft_first_ct_inplace<nh, MY, 1, zh, NT, 1, true>(s.D, [&](int y, int m) -> float2 {
        const float2 *row = s.D + y * zh;
        const int p = nh - m;
        float2 xm = row[m], xp = row[p];
        if (q.dz) {  // column kz: k_z, zero on the Nyquist column
            xm = mul_minus_i(xm, q.kfz * m, 2 * m == mz, WIDE);
            xp = mul_minus_i(xp, q.kfz * p, 2 * p == mz, WIDE);
        }
        const float2 sm = cadd(xm, cconj(xp));
        const float2 df = cmul(cconj(s.post[m]), csub(xm, cconj(xp)));
        return cadd(sm, cmul_i(df, 1.f));
    });
    ct::fft_inplace_ct<nh, MY, 1, zh, NT, 1, 1, ct::CtPlan<nh>::v.ns - 1>(s.D, s.twz);
    ct::fft_last_ct<nh, MY, 1, zh, NT, 1, true>(
        s.D, s.twz, [&](int y, int k, float2 v) { dst[y * nh + k] = make_float2(v.x * scale, v.y * scale); });
}

// The plane kernels of a geometry.
template <class G>
static constexpr auto r2c_plane(const G &) { return &r2c_zy_plane_kernel<G>; }
template <class G>
static constexpr auto c2r_plane(const G &, bool) { return &c2r_yz_plane_kernel<G>; }
template <int MY, int MZ, int NT, int WPE>
static constexpr auto r2c_plane(const PlaneFixed<MY, MZ, NT, WPE> &) { return &r2c_zy_plane_kernel_fixed<MY, MZ, NT, WPE>; }
template <int MY, int MZ, int NT, int WPE>
static constexpr auto c2r_plane(const PlaneFixed<MY, MZ, NT, WPE> &, bool wide) {
    return wide ? &c2r_yz_plane_kernel_fixed<MY, MZ, NT, WPE, true> : &c2r_yz_plane_kernel_fixed<MY, MZ, NT, WPE, false>;
}

// ---------------------------------------------------------------------------
// line passes: z rows (contiguous) and strided lines
// ---------------------------------------------------------------------------

// W rows of Mz reals per workgroup, any Mz or a compile-time one.
struct RowsRt {
    int nh, zh, zhs, W;
    float inv_zh;
    LineAxis az;
    const float2 *twz, *post;
    __device__ AxisRt<kLineRadix> z() const { return {az}; }
    __device__ LinesRt<kRowElems> lines(int wv) const { return {wv, 1, zhs, 1.0f / (float)wv}; }
    __device__ int row_of(int idx) const { return divq(idx, inv_zh); }
};

template <int MZ, int W_>
struct RowsCt {
    static constexpr int nh = MZ / 2, zh = MZ / 2 + 1, zhs = zh | 1, W = W_;
    const float2 *twz, *post;
    __device__ AxisCt<MZ / 2, kLineRadix> z() const { return {}; }
    __device__ LinesCt<W_, 1, zhs, kBlock> lines(int) const { return {}; }  // rows beyond the last are zero
    __device__ int row_of(int idx) const { return idx / zh; }
};

// z pass, real -> half spectrum
template <class G>
__global__ void __launch_bounds__(kBlock) r2c_z_kernel(const float *__restrict__ in, float2 *__restrict__ out,
                                                       int64_t rows, G g) {
    extern __shared__ float2 smem[];
    float2 *tw = smem, *post = tw + g.nh, *A = post + g.zh;  // W rows at stride zhs
    for (int i = threadIdx.x; i < g.nh - 1; i += kBlock) tw[i] = g.twz[i];
    for (int i = threadIdx.x; i < g.zh; i += kBlock) post[i] = g.post[i];
    const int64_t row0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * g.W;
    const int wv = (int)(rows - row0 < g.W ? rows - row0 : g.W);
    const float2 *src = reinterpret_cast<const float2 *>(in) + row0 * g.nh;
    float2 *dst = out + row0 * g.zh;
    line_first<-1, true>(A, g.lines(wv), g.z(),
                         [&](int l, int k) {
        const float2 *q = src + l * g.nh + k;
        const bool ok = l < wv;
        return [q, ok](int d) { return ok ? q[d] : make_float2(0.f, 0.f); };
    });
    line_later<-1, false>(A, g.lines(wv), g.z(), tw);
    for (int idx = threadIdx.x; idx < wv * g.zh; idx += kBlock) {
        const int l = g.row_of(idx), m = idx - l * g.zh;
        dst[idx] = RealSplit(A + l * g.zhs, post, m, g.nh)(0);
    }
}

// z pass of a YzJob, half spectrum -> real: block (grid, W rows), the
// y-transformed spectra in tmp, grid t nkinds + d at tmp + (it - grid0) gc.
template <class G>
__global__ void __launch_bounds__(kBlock) c2r_z_kernel(const float2 *__restrict__ tmp, YzArgs a, int64_t rows,
                                                       int blocks, G g) {
    extern __shared__ float2 smem[];
    float2 *tw = smem, *post = tw + g.nh, *A = post + g.zh;  // W rows at stride zhs
    for (int i = threadIdx.x; i < g.nh - 1; i += kBlock) tw[i] = g.twz[i];
    for (int i = threadIdx.x; i < g.zh; i += kBlock) post[i] = g.post[i];
    const int flat = (int)xcd_block(blockIdx.x, gridDim.x);
    const int local = flat / blocks, grid = a.grid0 + local, t = grid / a.nkinds;
    const YzGrid q = yz_grid(a, t, grid - t * a.nkinds);
    const int64_t row0 = (int64_t)(flat - local * blocks) * g.W;
    const int wv = (int)(rows - row0 < g.W ? rows - row0 : g.W);
    const float2 *src = tmp + (int64_t)local * a.gc + row0 * g.zh;
    float2 *dst = reinterpret_cast<float2 *>(q.dst) + row0 * g.nh;
    const int total = wv * g.zh;
    for (int i0 = threadIdx.x; i0 < g.W * g.zh; i0 += kBlock * kLoadBatch) {
        float2 v[kLoadBatch];
#pragma unroll
        for (int j = 0; j < kLoadBatch; ++j) {
            const int idx = i0 + j * kBlock;
            v[j] = idx < total ? src[idx] : make_float2(0.f, 0.f);
        }
#pragma unroll
        for (int j = 0; j < kLoadBatch; ++j) {
            const int idx = i0 + j * kBlock;
            if (idx < g.W * g.zh) A[idx + (g.zhs == g.zh ? 0 : g.row_of(idx))] = v[j];
        }
    }
    __syncthreads();
    line_first_inplace<1, true>(A, g.lines(wv), g.z(),
                                [&](int l, int m) {
        const float2 *row = A + l * g.zhs;
        return [row, m, post, &g](int d) { return real_join(row, post, m + d, g.nh); };
    });
    const float scale = a.job.scale;
    line_rest<1, true>(A, g.lines(wv), g.z(), tw, [&](int l, int k) {
        float2 *q = dst + l * g.nh + k;
        const bool ok = l < wv;
        return [q, ok, scale](int d, float2 v) {
            if (ok) q[d] = make_float2(v.x * scale, v.y * scale);
        };
    });
}

// Strided lines of one grid: line l at (l / inner) * outer + (l % inner),
// element e at es more; W consecutive lines per workgroup (neighbours in
// memory except at `inner` boundaries).
struct Strided {
    int nlines, inner, W, blocks;  // blocks: workgroups per grid
    int64_t outer, es;
    float inv_inner;
};

__device__ __forceinline__ int64_t strided_base(const Strided &q, int line) {
    const int o = divq(line, q.inv_inner);
    return (int64_t)o * q.outer + (line - o * q.inner);
}

// The axis of a strided pass, any length or N points with W lines of NT threads.
struct StridedRt {
    static constexpr int threads = kBlock;
    int n;
    LineAxis a;
    const float2 *tw;
    __device__ AxisRt<kLineRadix> axis() const { return {a}; }
    __device__ LinesRt<kLineElems> lines(int wv) const { return {wv, 1, n | 1, 1.0f / (float)wv}; }
    __device__ static int nt() { return kBlock; }
};

template <int N, int W, int NT>
struct StridedCt {
    static constexpr int threads = NT, n = N;
    const float2 *tw;
    __device__ AxisCt<N, kLineRadix> axis() const { return {}; }
    __device__ LinesCt<W, 1, N | 1, NT> lines(int) const { return {}; }
    __device__ static constexpr int nt() { return NT; }
};

// In-place complex pass along a strided axis.
template <int SGN, class G>
__global__ void __launch_bounds__(G::threads) fft_strided_kernel(float2 *__restrict__ data, int64_t gc, Strided q,
                                                                 G g) {
    extern __shared__ float2 smem[];
    float2 *tw = smem, *A = tw + g.n;  // W lines at an odd stride
    for (int i = threadIdx.x; i < g.n - 1; i += G::nt()) tw[i] = g.tw[i];
    const int flat = (int)xcd_block(blockIdx.x, gridDim.x);
    const int grid = flat / q.blocks, line0 = (flat - grid * q.blocks) * q.W;
    const int wv = min(q.W, q.nlines - line0);
    line_first<SGN, false>(A, g.lines(wv), g.axis(), [&](int l, int e) {
        const float2 *p = data + (int64_t)grid * gc + strided_base(q, line0 + l) + (int64_t)e * q.es;
        const bool ok = l < wv;
        return [p, ok, &q](int d) { return ok ? p[(int64_t)d * q.es] : make_float2(0.f, 0.f); };
    });
    line_rest<SGN, false>(A, g.lines(wv), g.axis(), tw, [&](int l, int e) {
        float2 *p = data + (int64_t)grid * gc + strided_base(q, line0 + l) + (int64_t)e * q.es;
        const bool ok = l < wv;
        return [p, ok, &q](int d, float2 v) {
            if (ok) p[(int64_t)d * q.es] = v;
        };
    });
}

// Out-of-place inverse y pass of a YzJob into tmp, laid out as c2r_z_kernel reads it.
template <class G>
__global__ void __launch_bounds__(G::threads) fft_y_multi_kernel(float2 *__restrict__ tmp, YzArgs a, Strided q, G g) {
    extern __shared__ float2 smem[];
    float2 *tw = smem, *A = tw + g.n;
    for (int i = threadIdx.x; i < g.n - 1; i += G::nt()) tw[i] = g.tw[i];
    const int flat = (int)xcd_block(blockIdx.x, gridDim.x);
    const int local = flat / q.blocks, line0 = (flat - local * q.blocks) * q.W;
    const int grid = a.grid0 + local, t = grid / a.nkinds;
    const YzGrid y = yz_grid(a, t, grid - t * a.nkinds);
    float2 *dst = tmp + (int64_t)local * a.gc;
    const int wv = min(q.W, q.nlines - line0);
    line_first<1, false>(A, g.lines(wv), g.axis(), [&](int l, int e) {
        const int line = line0 + l, x = divq(line, q.inv_inner), kz = line - x * q.inner;
        const float2 *p = y.src + (int64_t)x * q.outer + kz + (int64_t)e * q.es;
        const YzFactor w(y, e, kz, g.n, q.inner - 1);
        const bool ok = l < wv;
        return [p, w, ok, &q](int d) { return ok ? w(p[(int64_t)d * q.es], d) : make_float2(0.f, 0.f); };
    });
    line_rest<1, false>(A, g.lines(wv), g.axis(), tw, [&](int l, int e) {
        float2 *p = dst + strided_base(q, line0 + l) + (int64_t)e * q.es;
        const bool ok = l < wv;
        return [p, ok, &q](int d, float2 v) {
            if (ok) p[(int64_t)d * q.es] = v;
        };
    });
}

// ---------------------------------------------------------------------------
// launches
// ---------------------------------------------------------------------------
static size_t z_lds(const FftPlan &plan) {
    return sizeof(float2) * ((size_t)plan.lzh.n + plan.mesh.zh + (size_t)plan.wz * plan.zhs);
}

// Threads and register block of a plane kernel: the fewest turns, times the
// rounds of butterflies in a turn weighted with their radix.  Turns are the
// planes over those the chip works on at a time, half way to whole; a CU holds
// as many planes as LDS takes and as its SIMDs have registers for: PlaneRt::waves each, of which a workgroup takes a
// quarter of its wavefronts, rounded up (so whole quarters are tried; and five
// wavefronts of the smaller block, of which four workgroups were seen to fit).
// A turn also costs about 35 rounds of radix 1 of its own: loads, stores,
// barriers.  Gradient grids (c2r), the choice against the best of the others
// tried (4 to 16 wavefronts of both blocks): 100^3, four types 28.0 / 33 us,
// 96 x 200 x 96 61 / 69, 128 x 120 x 144, six types 103 / 118.  A rule that
// counted 24 wavefronts per CU however they fall on the SIMDs took 13 of the
// smaller block for planes of 75 to 81 KB, one plane per CU: 72 and 119 us in
// the last two, and 17.8 us, now 13.9, for r2c of four grids of 100^3.
static PlaneShape plane_shape(const FftPlan &plan, int64_t planes, bool inverse) {
    const int in_lds = (int)(160 * 1024 / plan.lds_plane);
    PlaneShape best;
    double best_cost = 0.0;
    for (int w : {1, 2, 3, 4, 5, 8, 12, 16})
        for (int elems : {kLineElems, kPlaneElemsBig}) {
            const bool small = elems == kLineElems;
            const int waves = small ? PlaneRt<kLineElems>::waves : PlaneRt<kPlaneElemsBig>::waves;
            const int k = std::min(in_lds, w == 5 && small ? 4 : waves / ((w + 3) / 4));
            if (k < 1 || !plane_fits(plan, 64 * w, elems, inverse)) continue;
            int rounds = 35;
            for (const LineAxis *ax : {&plan.ly, &plan.lzh})
                for (int s = 0; s < ax->ns; ++s) {
                    const int lines = ax == &plan.ly ? plan.mesh.zh : plan.mesh.my;
                    rounds += (lines * ax->st[s].nr + 64 * w - 1) / (64 * w) * ax->st[s].R;
                }
            const double turns = (double)planes / (kCus * k), whole = std::ceil(turns);
            const double cost = rounds * (turns < 1.0 ? 1.0 : 0.5 * (turns + whole));
            if (!best.threads || cost < best_cost) {
                best = PlaneShape{64 * w, elems};
                best_cost = cost;
            }
        }
    return best;
}

// Opt in to more than 64 KiB of dynamic LDS (once per kernel and process).
template <class K>
static int lds_opt_in(K kernel, bool &done) {
    if (!done) {
        HYMD_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)kPlaneLdsBytes));
        done = true;
    }
    return HYMD_OK;
}

// Calls f(geometry, threads) with the plane geometry for `planes` planes of
// the plan in one direction: compile-time for the planes of the cubic meshes
// listed, whose sizes the package's workloads use, else the general one.  Four
// types, c2r and r2c: 128^2 on fft_ct.h 48 us against 68 for the general form
// (c2r), 96^2 23.9 and 11.6 against 28.5 and 14.0, 64^2 9.3 and 6.0 against 11.1
// and 8.4, 48^2 7.2 and 4.8 against 8.8 and 6.8; whole updates 5 to 9 %.
template <class F>
static int with_plane(const FftPlan &plan, int64_t planes, bool inverse, F &&f) {
    const Mesh &m = plan.mesh;
    const PlaneTables t{plan.ty, plan.tzh, plan.post}, tf{plan.fy, plan.fzh, plan.post};
    if (plane_fixed(m) && m.my == 128) return f(PlaneFixed<128, 128, 1024, 8>{m.mx, tf}, 1024);
    if (plane_fixed(m)) return f(PlaneFixed<160, 160, 1024, 1>{m.mx, tf}, 1024);
    if (plane_ct(m)) {
        switch (m.my) {
            case 48: return f(PlaneCt<48, 48, 512>{m.mx, t}, 512);
            case 64: return f(PlaneCt<64, 64, 512>{m.mx, t}, 512);
            default: return f(PlaneCt<96, 96, 512>{m.mx, t}, 512);
        }
    }
    const PlaneShape sh = plane_shape(plan, planes, inverse);
    const float iy = 1.0f / (float)m.my, iz = 1.0f / (float)m.zh;
    if (sh.elems == kLineElems)
        return f(PlaneRt<kLineElems>{m.mx, m.my, m.mz / 2, m.zh, plan.zhs, iy, iz, plan.ly, plan.lzh, t}, sh.threads);
    return f(PlaneRt<kPlaneElemsBig>{m.mx, m.my, m.mz / 2, m.zh, plan.zhs, iy, iz, plan.ly, plan.lzh, t}, sh.threads);
}

// Calls f(geometry) with the z rows of the plan.
template <class F>
static int with_rows(const FftPlan &plan, F &&f) {
    const Mesh &m = plan.mesh;
    if (m.mz == 256 && plan.wz == 16) return f(RowsCt<256, 16>{plan.tzh, plan.post});
    return f(RowsRt{m.mz / 2, m.zh, plan.zhs, plan.wz, 1.0f / (float)m.zh, plan.lzh, plan.tzh, plan.post});
}

// 256-point lines: 16 per workgroup (128-byte row segments) for batches of 4
// grids or more, else 8.
static Strided strided_lines(const FftPlan &plan, int axis, int batch) {
    const Mesh &m = plan.mesh;
    Strided q;
    q.nlines = axis == 1 ? m.mx * m.zh : m.my * m.zh;  // (x, kz) lines, or (y, kz) ones
    q.inner = axis == 1 ? m.zh : q.nlines;
    q.outer = axis == 1 ? (int64_t)m.my * m.zh : 0;
    q.es = q.inner;
    q.W = axis == 1 ? plan.wy : plan.wx;
    if ((axis == 1 ? m.my : m.mx) == 256 && batch < 4) q.W = 8;
    q.blocks = (q.nlines + q.W - 1) / q.W;
    q.inv_inner = 1.0f / (float)q.inner;
    return q;
}

static size_t strided_lds(const LineAxis &ax, int W) { return sizeof(float2) * ((size_t)ax.n + (size_t)W * (ax.n | 1)); }

// Calls f(geometry) for a strided axis with W lines per workgroup.
template <class F>
static int with_strided(const FftPlan &plan, int axis, int W, F &&f) {
    const LineAxis &ax = axis == 1 ? plan.ly : plan.lx;
    const float2 *tw = axis == 1 ? plan.ty : plan.tx;
    if (ax.n == 256 && W == 16) return f(StridedCt<256, 16, 2 * kBlock>{tw});
    if (ax.n == 256 && W == 8) return f(StridedCt<256, 8, kBlock>{tw});
    return f(StridedRt{ax.n, ax, tw});
}

static int launch_strided(const FftPlan &plan, float2 *data, int batch, int axis, float sgn, hipStream_t s) {
    const Strided q = strided_lines(plan, axis, batch);
    const size_t lds = strided_lds(axis == 1 ? plan.ly : plan.lx, q.W);
    const int blocks = q.blocks * batch;
    return with_strided(plan, axis, q.W, [&](auto g) -> int {
        using G = decltype(g);
        if (sgn < 0.f)
            fft_strided_kernel<-1, G><<<blocks, G::threads, lds, s>>>(data, plan.mesh.gc, q, g);
        else
            fft_strided_kernel<1, G><<<blocks, G::threads, lds, s>>>(data, plan.mesh.gc, q, g);
        HYMD_HIP(hipGetLastError());
        return HYMD_OK;
    });
}

int fft_forward_x(const FftPlan &plan, float2 *data, int batch, hipStream_t s) {
    return launch_strided(plan, data, batch, 0, -1.f, s);
}

int fft_inverse_x(const FftPlan &plan, float2 *data, int batch, hipStream_t s) {
    return launch_strided(plan, data, batch, 0, 1.f, s);
}

int fft_r2c_zy(const FftPlan &plan, const float *in, float2 *out, int batch, hipStream_t s) {
    const Mesh &m = plan.mesh;
    if (plan.lds_plane) {
        const int blocks = m.mx * batch;
        return with_plane(plan, blocks, false, [&](auto g, int threads) -> int {
            using G = decltype(g);
            static bool done = false;
            if (plan.lds_plane > 64 * 1024) HYMD_TRY(lds_opt_in(r2c_plane(g), done));
            r2c_plane(g)<<<blocks, threads, plan.lds_plane, s>>>(in, out, g);
            HYMD_HIP(hipGetLastError());
            return HYMD_OK;
        });
    }
    const int64_t rows = (int64_t)m.mx * m.my * batch;
    HYMD_TRY(with_rows(plan, [&](auto g) -> int {
        using G = decltype(g);
        r2c_z_kernel<G><<<(unsigned)((rows + plan.wz - 1) / plan.wz), kBlock, z_lds(plan), s>>>(in, out, rows, g);
        HYMD_HIP(hipGetLastError());
        return HYMD_OK;
    }));
    return launch_strided(plan, out, batch, 1, -1.f, s);
}

int fft_r2c_real(const FftPlan &plan, const float *in, float2 *out, int batch, hipStream_t s) {
    HYMD_TRY(fft_r2c_zy(plan, in, out, batch, s));
    return fft_forward_x(plan, out, batch, s);
}

// The line passes take this many of a job's grids at a time: all, up to five
// per type, while that is 4 GB of scratch at most, then as many as 4 GB hold and
// at least one per type.  Several goes cost the ends of their launches: 256^3,
// six types, force grids 2072 us, one per type at a time 2146.
int fft_yz_tmp(const FftPlan &plan, const YzJob &job) {
    if (plan.lds_plane) return 0;
    const int64_t some = (int64_t(4) << 30) / ((int64_t)sizeof(float2) * plan.mesh.gc);
    const int64_t types = (int64_t)job.T * job.systems;
    return (int)std::min(std::max(some, types), types * yz_args(plan, job).nkinds);
}

// The z pass of `grids` of a job's grids, whose y-transformed spectra are in tmp.
static int launch_z_inverse(const FftPlan &plan, const YzArgs &a, int grids, const float2 *tmp, hipStream_t s) {
    const int64_t rows = (int64_t)plan.mesh.mx * plan.mesh.my;
    const int blocks = (int)((rows + plan.wz - 1) / plan.wz);
    return with_rows(plan, [&](auto g) -> int {
        using G = decltype(g);
        c2r_z_kernel<G><<<blocks * grids, kBlock, z_lds(plan), s>>>(tmp, a, rows, blocks, g);
        HYMD_HIP(hipGetLastError());
        return HYMD_OK;
    });
}

int fft_yz_multi(const FftPlan &plan, const YzJob &job, float2 *tmp, hipStream_t s) {
    const YzArgs a = yz_args(plan, job);
    const int grids = job.T * job.systems * a.nkinds;
    if (grids == 0) return HYMD_OK;
    if (plan.lds_plane) {
        const int blocks = plan.mesh.mx * grids;
        return with_plane(plan, blocks, true, [&](auto g, int threads) -> int {
            using G = decltype(g);
            static bool done[2] = {false, false};
            const auto kernel = c2r_plane(g, job.wide);
            if (plan.lds_plane > 64 * 1024) HYMD_TRY(lds_opt_in(kernel, done[job.wide]));
            kernel<<<blocks, threads, plan.lds_plane, s>>>(a, g);
            HYMD_HIP(hipGetLastError());
            return HYMD_OK;
        });
    }
    HYMD_REQUIRE(tmp, "planes that do not fit in LDS need the line passes' scratch");
    const Strided q = strided_lines(plan, 1, 1);
    const int step = fft_yz_tmp(plan, job);
    YzArgs b = a;
    for (b.grid0 = 0; b.grid0 < grids; b.grid0 += step) {
        const int some = std::min(step, grids - b.grid0);
        HYMD_TRY(with_strided(plan, 1, q.W, [&](auto g) -> int {
            using G = decltype(g);
            fft_y_multi_kernel<G><<<q.blocks * some, G::threads, strided_lds(plan.ly, q.W), s>>>(tmp, b, q, g);
            HYMD_HIP(hipGetLastError());
            return HYMD_OK;
        }));
        HYMD_TRY(launch_z_inverse(plan, b, some, tmp, s));
    }
    return HYMD_OK;
}

int fft_c2r_yz(const FftPlan &plan, float2 *in, float *out, int batch, float scale, hipStream_t s) {
    YzJob job;
    job.T = batch;
    job.in2 = in;
    job.real2 = out;
    job.scale = scale;
    if (plan.lds_plane) return fft_yz_multi(plan, job, nullptr, s);
    HYMD_TRY(launch_strided(plan, in, batch, 1, 1.f, s));  // y in place, then the z pass from there
    return launch_z_inverse(plan, yz_args(plan, job), batch, in, s);
}

int fft_c2r(const FftPlan &plan, float2 *data, float *out, int batch, float scale, hipStream_t s) {
    HYMD_TRY(fft_inverse_x(plan, data, batch, s));
    return fft_c2r_yz(plan, data, out, batch, scale, s);
}

}  // namespace hymd
