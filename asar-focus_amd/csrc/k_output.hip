// Output conditioning (the step after the focusing path): the SLC as big-endian int16 I/Q records and the
// detected image as uint16 dB records, each record led by a zeroed MDS record header
// (envisat_format/src/envisat_format_kernels.cu:28-114).
#include <cmath>

#include "kernels.h"

namespace asarf {

constexpr int kOutThreads = 256;

// float -> integer the way the reference's device casts behave: truncation toward zero, saturating at the
// destination range, NaN -> 0
__device__ __forceinline__ int sat_trunc(float v, float lo, float hi) {
    if (!(v == v)) return 0;
    v = fminf(fmaxf(v, lo), hi);
    return (int)v;  // |v| <= 65535: exact truncation
}

// Every lane converts kPix adjacent pixels: 16 bytes of a record, whose pitch (17-byte ASAR header + pixels) leaves them
// at any address, with one unaligned 16-byte store and 16-byte loads at the row's own alignment. (One pixel a lane and
// byte stores: SLC of 30000 x 5095 396 us, detected 10200 x 7031 168 us; the copies of their bytes take 363 and 85 us.)
struct __attribute__((packed, aligned(1))) Bytes16 {
    unsigned w[4];
};
struct __attribute__((packed, aligned(4))) Floats4 {
    float v[4];
};
__device__ __forceinline__ void zero_header(const OutputArgs& a, unsigned char* rec) {
    if (blockIdx.x == 0)
        for (int h = threadIdx.x; h < a.header; h += kOutThreads) rec[h] = 0;
}

// CalibrateClampToBigEndian (:28-68): record y = header zero bytes, then x_size pixels of (I, Q) as big-endian
// int16 of clamp(value * calibration).
__device__ __forceinline__ unsigned slc_pixel(float2 v, float calibration) {
    const int i = sat_trunc(v.x * calibration, -32768.f, 32767.f);
    const int q = sat_trunc(v.y * calibration, -32768.f, 32767.f);
    return __builtin_bswap32(((unsigned)(i & 0xFFFF) << 16) | (unsigned)(q & 0xFFFF));  // bytes I high, I low, Q high, Q low
}
__global__ __launch_bounds__(kOutThreads) void k_condition_slc(OutputArgs a) {
    constexpr int kPix = 4;
    const int x = (blockIdx.x * kOutThreads + threadIdx.x) * kPix;
    const int y = blockIdx.y;
    unsigned char* rec = a.dest + (long)y * a.record_bytes;
    zero_header(a, rec);
    if (x >= a.x_size) return;
    const float2* in = a.slc + (long)y * a.x_stride + x;
    unsigned char* p = rec + a.header + 4 * x;
    if (x + kPix <= a.x_size) {
        const Floats4 f0 = *reinterpret_cast<const Floats4*>(in), f1 = *reinterpret_cast<const Floats4*>(in + 2);
        Bytes16 o;
        o.w[0] = slc_pixel(make_float2(f0.v[0], f0.v[1]), a.calibration);
        o.w[1] = slc_pixel(make_float2(f0.v[2], f0.v[3]), a.calibration);
        o.w[2] = slc_pixel(make_float2(f1.v[0], f1.v[1]), a.calibration);
        o.w[3] = slc_pixel(make_float2(f1.v[2], f1.v[3]), a.calibration);
        *reinterpret_cast<Bytes16*>(p) = o;
        return;
    }
    for (int k = 0; x + k < a.x_size; ++k) {
        const unsigned u = slc_pixel(in[k], a.calibration);
        for (int b = 0; b < 4; ++b) p[4 * k + b] = (unsigned char)(u >> (8 * b));
    }
}

// CalibrateClampToBigEndianDetected (:70-98): record y = header zero bytes, then x_size uint16 of
// 10 log10(value * calibration) in single precision, saturated to [0, 65535] (negative and NaN -> 0). The
// reference stores these low byte first (its detected kernel does not byte-swap, despite its name); so does this.
__device__ __forceinline__ unsigned detected_pixel(float v, float calibration) {
    return (unsigned)sat_trunc(10.0f * log10f(v * calibration), 0.f, 65535.f);
}
__global__ __launch_bounds__(kOutThreads) void k_condition_detected(OutputArgs a) {
    constexpr int kPix = 8;
    const int x = (blockIdx.x * kOutThreads + threadIdx.x) * kPix;
    const int y = blockIdx.y;
    unsigned char* rec = a.dest + (long)y * a.record_bytes;
    zero_header(a, rec);
    if (x >= a.x_size) return;
    const float* in = a.det + (long)y * a.x_stride + x;
    unsigned char* p = rec + a.header + 2 * x;
    if (x + kPix <= a.x_size) {
        const Floats4 f[2] = {*reinterpret_cast<const Floats4*>(in), *reinterpret_cast<const Floats4*>(in + 4)};
        Bytes16 o;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            o.w[k] = detected_pixel(f[k >> 1].v[2 * (k & 1)], a.calibration) |
                     detected_pixel(f[k >> 1].v[2 * (k & 1) + 1], a.calibration) << 16;
        *reinterpret_cast<Bytes16*>(p) = o;
        return;
    }
    for (int k = 0; x + k < a.x_size; ++k) {
        const unsigned u = detected_pixel(in[k], a.calibration);
        p[2 * k] = (unsigned char)(u & 0xFF);
        p[2 * k + 1] = (unsigned char)(u >> 8);
    }
}

hipError_t launch_condition(const OutputArgs& a, int detected, hipStream_t s) {
    const int per = kOutThreads * (detected ? 8 : 4);
    const dim3 grid((a.x_size + per - 1) / per, a.y_size);
    if (detected)
        hipLaunchKernelGGL(k_condition_detected, grid, dim3(kOutThreads), 0, s, a);
    else
        hipLaunchKernelGGL(k_condition_slc, grid, dim3(kOutThreads), 0, s, a);
    return hipGetLastError();
}

}  // namespace asarf
