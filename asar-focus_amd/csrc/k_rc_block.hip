// Range compression in blocks of a line: the compiled block lengths, the choice among them and the launch
// (rc_block.h holds the kernel).
#include "rc_block.h"

namespace asarf {

// Compiled lengths: N, lanes, waves per SIMD asked of the compiler, radices. One list per compilation unit. (6144 meets
// its six waves by spilling 7 registers for cf32 lines, 21 for the other formats; the other lengths do without.)
#define ASARF_RC_BLOCKS_0(X) X(1024, 64, 4, 16, 16, 4) X(1536, 128, 5, 16, 16, 6) X(2048, 128, 4, 16, 16, 8)
#define ASARF_RC_BLOCKS_1(X) X(2560, 256, 5, 16, 16, 10) X(3072, 256, 5, 16, 16, 12)
#define ASARF_RC_BLOCKS_2(X) X(4096, 256, 4, 16, 16, 16) X(6144, 512, 6, 8, 8, 8, 12)

#ifndef ASARF_RC_BLOCK_UNIT
#define ASARF_RC_BLOCK_UNIT 0
#endif
#define ASARF_RC_CAT_(a, b) a##b
#define ASARF_RC_CAT(a, b) ASARF_RC_CAT_(a, b)

bool ASARF_RC_CAT(launch_rc_block_, ASARF_RC_BLOCK_UNIT)(const RcArgs& a, int fmt, int n, hipStream_t s, hipError_t* err) {
    switch (n) {
#define ASARF_RC_CASE(N, T, W, ...) \
    case N: *err = rcblock::launch<N, T, W, RadixSeq<__VA_ARGS__>>(a, fmt, s); return true;
        ASARF_RC_CAT(ASARF_RC_BLOCKS_, ASARF_RC_BLOCK_UNIT)(ASARF_RC_CASE)
#undef ASARF_RC_CASE
        default: return false;
    }
}

#if ASARF_RC_BLOCK_UNIT == 0

bool launch_rc_block_1(const RcArgs& a, int fmt, int n, hipStream_t s, hipError_t* err);
bool launch_rc_block_2(const RcArgs& a, int fmt, int n, hipStream_t s, hipError_t* err);

#define ASARF_RC_ALL(X) ASARF_RC_BLOCKS_0(X) ASARF_RC_BLOCKS_1(X) ASARF_RC_BLOCKS_2(X)

hipError_t launch_rc_block(const RcArgs& a, int fmt, int n, hipStream_t s) {
    if (fmt != RAW_CF32 && fmt != RAW_U8 && fmt != RAW_I8 && fmt != RAW_ERS_LINES && fmt != RAW_ASAR_FBAQ4)
        return hipErrorInvalidValue;
    if (fmt == RAW_ASAR_FBAQ4 && !a.lines.lut) return hipErrorInvalidValue;
    if (!a.rc_tw || !a.hconj || a.blocks < 1 || a.block_step < 1 || a.rows < 1) return hipErrorInvalidValue;
    // blocks of one line overlap on the input side: several per line only out of place
    if (a.blocks > 1 && a.in == static_cast<const void*>(a.out)) return hipErrorInvalidValue;
    hipError_t err = hipErrorInvalidValue;
    if (launch_rc_block_0(a, fmt, n, s, &err) || launch_rc_block_1(a, fmt, n, s, &err) ||
        launch_rc_block_2(a, fmt, n, s, &err))
        return err;
    return hipErrorInvalidValue;
}

// A forward and an inverse transform of n points return their input times n and this: the rounded constants of the
// butterflies lie inside the unit circle more often than outside it (the eighth and the sixteenth roots of unity by
// 1.7e-8 and 2.9e-8), which shrinks every line alike and would not average out of a multilooked intensity. Measured
// on random lines; the spectrum, formed in FP64, takes it back. (5616 samples: error against FP64 1.82e-7 -> 1.68e-7.)
static double round_trip_gain(int n) {
    switch (n) {
        case 1024: return 1.0 - 5.45e-8;
        case 1536: return 1.0 - 7.26e-8;
        case 2048: return 1.0 - 6.47e-8;
        case 2560: return 1.0 - 3.21e-8;
        case 3072: return 1.0 - 7.43e-8;
        case 4096: return 1.0 - 7.95e-8;
        default: return 1.0 - 6.95e-8;  // 6144
    }
}

// conj(FFT_n(chirp)) * scale, one bin per wave: the chirp is short, so the sums are formed directly in FP64 (nc * n terms,
// about 10 us) and rounded once, which the FP32 transform of the padded chirp was not.
__global__ __launch_bounds__(256) void k_rc_block_spectrum(const float2* chirp, int nc, int n, int m, double scale,
                                                           float2* out) {
    const int lane = threadIdx.x & 63;
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6);  // n is a multiple of 4
    const int k = (i >> 1) % m + (2 * (i / (2 * m)) + (i & 1)) * m;
    double re = 0.0, im = 0.0;
    for (int t = lane; t < nc; t += 64) {
        double sn, cs;
        sincospi(2.0 * (double)((long)t * k % n) / (double)n, &sn, &cs);
        const double x = chirp[t].x, y = -chirp[t].y;
        re += x * cs - y * sn;
        im += x * sn + y * cs;
    }
    for (int o = 32; o > 0; o >>= 1) {
        re += __shfl_xor(re, o);
        im += __shfl_xor(im, o);
    }
    if (lane == 0) out[i] = make_float2((float)(re * scale), (float)(im * scale));
}

hipError_t launch_rc_block_spectrum(const float2* chirp, int nc, int n, float2* out, hipStream_t s) {
    int radix[kMaxPasses];
    const int np = rc_block_radices(n, radix);
    if (np == 0 || nc < 1 || nc > n) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_rc_block_spectrum, dim3(n / 4), dim3(256), 0, s, chirp, nc, n, n / radix[np - 1],
                       1.0 / (n * round_trip_gain(n)), out);
    return hipGetLastError();
}

int rc_block_radices(int n, int* radices) {
    switch (n) {
#define ASARF_RC_RADIX(N, T, W, ...) \
    case N: return rcblock::fill_seq<RadixSeq<__VA_ARGS__>>(radices);
        ASARF_RC_ALL(ASARF_RC_RADIX)
#undef ASARF_RC_RADIX
        default: return 0;
    }
}

// Time of one block with the device full, in ns (measured on lines of 1200 to 5616 u8 and i8 samples). A line costs its
// number of blocks times this, so short chirps favour the lengths with the best rate per sample (1024 to 4096) and
// their overlap decides among them: 5616 samples with a 521-sample chirp take 2 x 3072 (140 us per 8000 lines; 4 x 2048
// 165, 2 x 4096 168, 1 x 6144 193, the transform of the padded line of 6144 it replaces 207), with a 704-sample chirp
// 4 x 2048 (157; 2 x 4096 164, 1 x 6144 188, the padded line of 6400 291), and 4937 samples with 463 take 3 x 2048 (120;
// the runtime-radix padded line of 5600 it replaces 761).
static float block_ns(int n) {
    switch (n) {
        case 1024: return 2.15f;
        case 1536: return 4.15f;
        case 2048: return 5.05f;
        case 2560: return 7.4f;
        case 3072: return 8.4f;
        case 4096: return 10.3f;
        default: return 23.5f;  // 6144
    }
}

bool rc_block_choose(int nr, int nc, bool single, RcBlock* out, int only) {
    static const int lengths[] = {
#define ASARF_RC_ITEM(N, ...) N,
        ASARF_RC_ALL(ASARF_RC_ITEM)
#undef ASARF_RC_ITEM
    };
    const int nrv = nr - nc;
    float best = 0.f;
    out->n = 0;
    for (const int n : lengths) {
        const int step = n - nc + 1;
        if (step < 1 || (only > 0 && n != only)) continue;
        const int blocks = (nrv + step - 1) / step;
        if (single && blocks > 1) continue;
        const float cost = (float)blocks * block_ns(n);
        if (out->n == 0 || cost < best) {
            best = cost;
            *out = RcBlock{n, blocks, step};
        }
    }
    // chirps nearly as long as the longest block would run in many blocks of few kept samples; the runtime-radix
    // transform of the padded line costs about 13 ns per 1000 samples
    return out->n > 0 && best <= 0.013f * (float)(nr + nc);
}

#endif

}  // namespace asarf
