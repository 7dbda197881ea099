// Projector grid of a reference map on the GPU: MyProjector::computeFourierTransformMap
// (src/reconstruct.cpp:106-223) with griddingCorrect (src/reconstruct.cpp:61-103).
//
//   pad    : map / sinc^2(r / (ori * pf)) (trilinear interpolator, r > 0), zero-padded to pf*ori per axis
//            at the centred position and circularly shifted by pf*ori/2 (centerFFT3D/2D forward,
//            src/reconstruct.h:103-180): one thread per map voxel, FP64.
//   FFT    : hipFFT D2Z (FP64), then / (number of real samples) as normalizeComplex does
//            (src/fft_base.cpp:103-109).
//   window : coefficients with |k|^2 <= (pf r_max)^2, times pf^3 ori (3D) or pf^2 (2D), into the
//            [pad][pad][pad/2+1] grid (FP32 for the projector, FP64 when the caller asks for it), and the
//            shell power sum / count (block sums in LDS, one FP64 atomic per shell per block).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_util.h"
#include "kernels.h"

namespace rome {

namespace {

__global__ void k_fm_pad(const double* __restrict__ vol, int ori, int padori, int dim3, int do_gridding, int pf,
                         double* __restrict__ Mc, double* __restrict__ corrected) {
    const size_t n = dim3 ? (size_t)ori * ori * ori : (size_t)ori * ori;
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    const int j = (int)(idx % ori);
    const int i = (int)((idx / ori) % ori);
    const int k = dim3 ? (int)(idx / ((size_t)ori * ori)) : 0;
    const int sh = -(int)((float)ori / 2.0f);
    double v = vol[idx];
    if (do_gridding) {
        const int x = j + sh, y = i + sh, z = dim3 ? k + sh : 0;
        const double r = sqrt((double)(x * x + y * y + z * z));
        if (r > 0.) {
            const double rval = r / (double)(ori * pf);
            const double sinc = sin(3.14159265358979323846 * rval) / (3.14159265358979323846 * rval);
            v /= sinc * sinc;
        }
    }
    if (corrected) corrected[idx] = v;
    // centred padding offset, then the forward centring shift by padori/2
    const int off = sh + (int)((float)padori / 2.0f);
    const int s = padori / 2;
    const int jp = (j + off + s) % padori, ip = (i + off + s) % padori;
    if (dim3) {
        const int kp = (k + off + s) % padori;
        Mc[((size_t)kp * padori + ip) * padori + jp] = v;
    } else {
        Mc[(size_t)ip * padori + jp] = v;
    }
}

constexpr int kFmShells = 520;  // ori/2 + 1 for ori up to 1038

// One wave per grid row (z, y), lanes consecutive x, blocks striding over the rows: every grid element is written
// once, value or zero (no clearing pass), and equal shells, neighbouring lanes, are added up by shuffles before one
// LDS atomic each.  (A thread per transform element with two LDS atomics, most of a wave on two addresses, and a
// flush per 256 elements took 1.46 ms for 192^3 and needed 0.7 GB cleared first.)
__global__ __launch_bounds__(256) void k_fm_window(const double2* __restrict__ F, int padori, int dim3, int pf,
                                                   int r_max, int pad, int oriF, double size3, double normfft,
                                                   double2* __restrict__ grid64, float2* __restrict__ grid32,
                                                   double* __restrict__ pw, double* __restrict__ cnt) {
    __shared__ double s_pw[kFmShells], s_cnt[kFmShells];
    for (int q = threadIdx.x; q < oriF; q += blockDim.x) s_pw[q] = s_cnt[q] = 0.;
    __syncthreads();
    const int padoriF = padori / 2 + 1, padF = pad / 2 + 1, c = (int)((float)pad / 2.0f), lane = threadIdx.x & 63;
    const int max_r2 = r_max * r_max * pf * pf, rows = (dim3 ? pad : 1) * pad;
    for (int row = blockIdx.x * 4 + (threadIdx.x >> 6); row < rows; row += gridDim.x * 4) {
        const int z = row / pad, y = row - z * pad;
        const int kp = dim3 ? z - c : 0, ip = y - c;
        // the transform holds the signed indices -(padori - padoriF) .. padoriF - 1
        const bool have = kp >= padoriF - padori && kp < padoriF && ip >= padoriF - padori && ip < padoriF;
        const int k = kp < 0 ? kp + padori : kp, i = ip < 0 ? ip + padori : ip;
        const double2* Fr = F + ((size_t)k * padori + i) * padoriF;
        for (int x0 = 0; x0 < padF; x0 += 64) {
            const int x = x0 + lane, r2 = kp * kp + ip * ip + x * x;
            const bool in = have && x < padoriF && x < padF && r2 <= max_r2;
            double re = 0., im = 0.;
            int ires = -1;
            if (in) {
                const double2 f = Fr[x];
                re = (f.x / size3) * normfft;
                im = (f.y / size3) * normfft;
                ires = (int)round(sqrt((double)r2) / pf);
            }
            if (x < padF) {
                const size_t g = (size_t)row * padF + x;
                if (grid64) grid64[g] = make_double2(re, im);
                grid32[g] = make_float2((float)re, (float)im);
            }
            shell_add(ires, (re * re + im * im) / 2., s_pw, s_cnt);
        }
    }
    __syncthreads();
    for (int q = threadIdx.x; q < oriF; q += blockDim.x)
        if (s_cnt[q] != 0.) {
            atomicAdd(&pw[q], s_pw[q]);
            atomicAdd(&cnt[q], s_cnt[q]);
        }
}

}  // namespace

hipError_t launch_fm_pad(hipStream_t s, const double* vol, int ori, int padori, int dim3, int do_gridding, int pf,
                         double* Mc, double* corrected) {
    const size_t n = dim3 ? (size_t)ori * ori * ori : (size_t)ori * ori;
    k_fm_pad<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(vol, ori, padori, dim3, do_gridding, pf, Mc, corrected);
    return hipGetLastError();
}

hipError_t launch_fm_window(hipStream_t s, const double2* F, int padori, int dim3, int pf, int r_max, int pad,
                            int oriF, double normfft, double2* grid64, float2* grid32, double* pw, double* cnt) {
    if (oriF > kFmShells) return hipErrorInvalidValue;
    const int rows = (dim3 ? pad : 1) * pad;
    const double size3 = dim3 ? (double)padori * padori * padori : (double)padori * padori;
    k_fm_window<<<(unsigned)std::min((rows + 3) / 4, 1024), 256, 0, s>>>(F, padori, dim3, pf, r_max, pad, oriF, size3, normfft,
                                                           grid64, grid32, pw, cnt);
    return hipGetLastError();
}

}  // namespace rome
