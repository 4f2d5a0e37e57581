// Batched mixed-radix FFT for mesh edges 2^a 3^b 5^c, staged in LDS (fft_line.h).
//
// 3-D real transforms (unnormalised, numpy sign convention):
//   r2c: z rows -> packed complex FFT of length Mz/2 + split (post twiddles),
//        then complex passes along y and x;
//   c2r: the same in reverse.
#pragma once
#include "common.h"
#include "fft_line.h"

namespace hymd {

// Loads are issued kLoadBatch at a time per thread (all in flight before the
// first LDS store) so that every wave keeps several HBM requests outstanding.
constexpr int kLoadBatch = 8;
constexpr size_t kPlaneLdsBytes = 150 * 1024;  // of the 160 KiB a gfx950 workgroup may use

// Threads per workgroup and values per thread of a plane kernel.
struct PlaneShape {
    int threads = 0, elems = 0;
};

// The x axis of an x-line pass: the forward plan's last radix is the inverse
// plan's first and at most what the registers hold for T types, T times over.
struct XlineAxes {
    LineAxis fwd, inv;
    const float2 *twf, *twi;
};
constexpr int kXlinePlans = 6;
inline int xline_plan_of(int T) { return T <= 2 ? 0 : (T <= 6 ? T - 2 : 5); }

struct FftPlan {
    Mesh mesh;
    LineAxis lx, ly, lzh;        // x, y full axes; z half-length packed axis
    XlineAxes xl[kXlinePlans];   // by xline_plan_of(T)
    DevBuf tables;               // their forward twiddles and exp(-2 pi i k / Mz), k = 0..Mz/2
    const float2 *tx, *ty, *tzh, *post;  // into tables
    const float2 *fx, *fy, *fzh;         // there, the twiddles of fft_ct.h where it runs
    int wx, wy, wz;              // lines per workgroup of the line passes
    int zhs;                     // LDS stride of a half-spectrum row (odd)
    size_t lds_plane;            // y-z plane kernels (0: planes do not fit, separate passes)
};

// x edges whose lines have kernels on fft_ct.h
inline bool xline_fixed_edge(int mx) { return mx == 128 || mx == 160 || mx == 256; }

int fft_plan_init(FftPlan &plan, const Mesh &mesh);

// What an inverse y-z pass makes of spectra whose x transform is done, per
// type t < T; every list that is null is left out:
//   force[3t + d]  gradient grids from in[t] = IFFT_x(-i k_x V_t) (d = 0) and
//                  in[T + t] = IFFT_x(V_t) (times -i k_y, -i k_z)
//   real_v[t]      the grid of in[T + t] itself
//   real2[t]       the grid of in2[t]
// (k_y = kfy n_y, k_z = kfz n_z, zero on Nyquist planes, multiplied in FP32, or
// with `wide` in FP64 and rounded once); all times scale.
// Several systems of the same mesh and T follow each other in every list
// (in: 2T spectra each), with their factors (kfy, kfz) in kf on the device.
struct YzJob {
    int T = 0, systems = 1;
    const double2 *kf = nullptr;
    const float2 *in = nullptr, *in2 = nullptr;
    float *force = nullptr, *real_v = nullptr, *real2 = nullptr;
    double kfy = 0.0, kfz = 0.0;
    bool wide = false;
    float scale = 1.f;
};

// 3-D real transforms of `batch` consecutive grids (unnormalised).  Where a
// My x (Mz/2+1) plane fits in LDS the z and y passes run as one plane kernel
// per (x-plane, grid), otherwise as separate line passes.
//   r2c:   fft_r2c_zy (z r2c + y) then fft_forward_x;  fft_r2c_real = both
//   c2r:   fft_inverse_x then fft_c2r_yz (y + z c2r);  fft_c2r = both.  The
//          spectra passed in may be overwritten.
int fft_r2c_zy(const FftPlan &plan, const float *in, float2 *out, int batch, hipStream_t s);
int fft_forward_x(const FftPlan &plan, float2 *data, int batch, hipStream_t s);
int fft_r2c_real(const FftPlan &plan, const float *in, float2 *out, int batch, hipStream_t s);
int fft_inverse_x(const FftPlan &plan, float2 *data, int batch, hipStream_t s);
int fft_c2r_yz(const FftPlan &plan, float2 *in, float *out, int batch, float scale, hipStream_t s);
int fft_c2r(const FftPlan &plan, float2 *data, float *out, int batch, float scale, hipStream_t s);
// The grids of `job`.  Where the planes do not fit in LDS, tmp holds one half
// spectrum for each of the grids made at a time (fft_yz_tmp of them; 0: none
// needed).
int fft_yz_multi(const FftPlan &plan, const YzJob &job, float2 *tmp, hipStream_t s);
int fft_yz_tmp(const FftPlan &plan, const YzJob &job);

}  // namespace hymd
