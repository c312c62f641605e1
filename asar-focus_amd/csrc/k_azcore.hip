// Fused azimuth core: forward pass B of the azimuth FFT, 16-tap sinc RCMC, azimuth matched filter and the
// inverse pass B', one workgroup per (k1 group, tile of columns), out of place (pass-A output -> pass-B' output).
//
// With the four-step split N = N1*N2, pass A leaves group k1's length-N2 transform inputs in the contiguous rows
// k1*N2 + m; pass B turns them into the bins k1 + N1*k2 (k2 < N2) of those rows. RCMC interpolates along range
// within one bin and the matched filter is pointwise, so a workgroup that transforms its k1 group for its
// columns plus a range halo can correct the bins in LDS and run the inverse length-N2 transform before anything
// returns to HBM: the spectrum makes one round trip to HBM instead of three (B out, RCMC in and out, B' in).
//   staged columns:    [x0 - 7, x0 + 73)    (80: the 14 taps with nonzero window weight reach x + p - 7 .. x + p + 6)
//   produced columns:  [x0, x0 + 64) for shifts p <= 3, [x0, x0 + 56) for p <= 8 = kAzCoreReach
// The bound on the shift comes from the device (ColConst), so every workgroup picks its tile width from it; the grid
// covers the narrow tiles and the surplus workgroups of the wide ones exit at once.
//
// What bounds it: vector issue (an instruction on every SIMD cycle; counted with transcendentals as two, 1.1), about
// half of it RCMC and matched filter, half the transforms. So that
// * a transform is 8 lanes per column and all 80 columns run at once on 640 of the 768 lanes. 768: a workgroup's waves
//   go to the SIMDs in order, so two workgroups of 640 lanes put 6 waves on two SIMDs and 4 on the others (1.02 ms on the
//   ASAR scene against 0.84 ms); the two waves that only take part in phase 2 change places from workgroup to workgroup;
// * the tile of up to 120 bins leaves room for two workgroups per CU (with 88 columns, 112 bins held one: 28672 x 4926
//   1.53 ms, now 0.83);
// * the twiddles W_N2^(r j) of both directions are one table of N2 entries in LDS (the inverse reads it transposed), and
//   the inter-pass twiddles W_N^(k1 n) of the workgroup's k1 are another, instead of powers and two-level lookups;
// * the band test, the aliasing and the phase work on whole bins: integers and one FP64 product chain per pixel.
// Together 17 % fewer vector instructions (617 M -> 510 M on the ASAR scene, 30240 = 288 x 105, 5095 columns): 1.02 ->
// 0.85 ms (0.85 to 0.89 from one card to the next). A copy of its bytes takes 0.49 ms.
// Phases:
//   1. forward transforms of the staged columns, bins left in the tile;
//   2. RCMC + matched filter: lane (wave w, column c) produces bins w, w + 12, ... of column c (a wave reads
//      consecutive tile columns of one bin row); results held in registers until every tap is read, then
//      written over the produced columns;
//   3. inverse transforms of the produced columns, inverse inter-pass twiddle, store.
#include "interp.h"
#include "kernels.h"

namespace asarf {

constexpr int kAcLanes = 8;                          // lanes per column transform
constexpr int kAcLeft = 7;                           // first produced column inside the tile
constexpr int kAcCols = 80;                          // staged columns per tile
constexpr int kAcThreads = 768;
constexpr int kAcWaves = kAcThreads / 64;
static_assert(kAcCols * kAcLanes <= kAcThreads, "one batch of column transforms");
constexpr int kAcPitch = kAcCols + 1;
constexpr int kAcNarrowReach = 3;                    // largest shift of 64-column tiles
constexpr int kAcNarrow = 64, kAcWide = 56;          // produced columns per tile
static_assert(kAcLeft + kAcNarrow + 6 + kAcNarrowReach <= kAcCols && kAcLeft + kAcWide + 6 + kAzCoreReach <= kAcCols,
              "the staged columns hold every tap");

// Butterflies j = lane + i * 8 of a pass with M of them; lanes past the last one work on a copy of it, and one that is
// past the end for the whole wave is skipped.
template <int M, class F>
__device__ __forceinline__ void each_butterfly(int lane, F&& f) {
    constexpr int NB = (M + kAcLanes - 1) / kAcLanes;
    static_for<0, NB>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        if ((i + 1) * kAcLanes <= M || wave_any(lane + i * kAcLanes < M)) {
            const int j = lane + i * kAcLanes;
            f(ic, (i + 1) * kAcLanes <= M ? j : min(j, M - 1), j < M);
        }
    });
}

constexpr int core_elems(int r0, int r1) {
    const int a = (r1 + kAcLanes - 1) / kAcLanes * r0, b = (r0 + kAcLanes - 1) / kAcLanes * r1;
    return a > b ? a : b;
}

// Waves per SIMD asked of the compiler: two workgroups per CU where their tiles fit. (90, 100 and 120 bins meet it by
// spilling 7, 21 and 21 registers, 20 to 36 bytes a lane; the other lengths do without.)
constexpr int core_waves(int n2) {
    return (size_t)n2 * (kAcPitch + 2) * sizeof(float2) <= 80 * 1024 ? 2 * kAcWaves / 4 : (kAcWaves + 3) / 4;
}

template <int N2, int R0, int R1>
__global__ __launch_bounds__(kAcThreads) __attribute__((amdgpu_waves_per_eu(core_waves(N2)))) void k_az_core(AzCoreArgs a) {
    static_assert(R0 * R1 == N2, "radices must factor N2");
    constexpr int E = core_elems(R0, R1);
    extern __shared__ float2 lds[];
    const int reach = a.reach ? *a.reach : a.reach_value;
    if (a.gated && reach > kAzCoreReach) return;
    const int width = reach <= kAcNarrowReach ? kAcNarrow : kAcWide;
    const int ntiles = (a.col1 - a.col0 + width - 1) / width;
    const int items = a.n1 * ntiles;
    // XCD-aware work order: workgroups are dealt to the 8 XCDs round robin, so consecutive work items
    // (neighbouring tiles of one k1 group, whose staged halos overlap) are given to the same XCD and its L2
    const int per_xcd = (items + 7) / 8;
    const int w = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if ((int)(blockIdx.x / 8) >= per_xcd || w >= items) return;
    const int k1 = w / ntiles;
    const int x0 = a.col0 + (w - k1 * ntiles) * width;
    const int tid = (int)((threadIdx.x + 128 * ((blockIdx.x >> 3) & 1)) % kAcThreads);
    float2* tl = lds;                  // [N2][kAcPitch]
    float2* tw = lds + N2 * kAcPitch;  // tw[r * R0 + j] = W_N2^(r j), r < R1, j < R0
    float2* tk = tw + N2;              // tk[n] = W_nbins^(k1 n)
    for (int i = tid; i < N2; i += kAcThreads) {
        tw[i] = a.tw2[(i / R0) * (i % R0)];
        tk[i] = a.tw_full[k1 * i];  // k1 * i < n1 * n2
    }
    const int c = tid % kAcCols, lane = tid / kAcCols;  // transform phases: column, lane of its transform
    const bool fwd = lane < kAcLanes;
    const long row0 = (long)k1 * N2;
    float2 v[E];

    // ---- 1. forward pass B of the staged columns (columns outside the image are zero, never read as taps)
    {
        const int x = x0 - kAcLeft + c;
        const bool ok = x >= 0 && x < a.nrv;
        const float2* in = a.in + row0 * a.stride;  // the same for every lane
        const unsigned stride = (unsigned)a.stride;
        const unsigned xc = ok ? x : 0;
        if (fwd) each_butterfly<R1>(lane, [&](auto ic, int j, bool) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                const float2 s = (in + (size_t)(r * R1) * stride)[(unsigned)j * stride + xc];
                v[decltype(ic)::value * R0 + r] = ok ? s : make_float2(0.f, 0.f);
            }
        });
        float2* col = tl + c;
        if (fwd) each_butterfly<R1>(lane, [&](auto ic, int j, bool valid) __attribute__((always_inline)) {
            float2* u = &v[decltype(ic)::value * R0];
            Dft<R0, false>::run(u);
            if (valid) {
#pragma unroll
                for (int r = 0; r < R0; ++r) col[(j * R0 + r) * kAcPitch] = u[r];
            }
        });
        __syncthreads();
        if (fwd) each_butterfly<R0>(lane, [&](auto ic, int j, bool) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < R1; ++r) v[decltype(ic)::value * R1 + r] = col[(j + r * R0) * kAcPitch];
        });
        __syncthreads();  // every element of the column is read before the bins overwrite it
        if (fwd) each_butterfly<R0>(lane, [&](auto ic, int j, bool valid) __attribute__((always_inline)) {
            float2* u = &v[decltype(ic)::value * R1];
#pragma unroll
            for (int r = 1; r < R1; ++r) u[r] = cmul(u[r], tw[r * R0 + j]);
            Dft<R1, false>::run(u);
            if (valid) {
#pragma unroll
                for (int r = 0; r < R1; ++r) col[(j + r * R0) * kAcPitch] = u[r];
            }
        });
    }
    __syncthreads();

    // ---- 2. RCMC + matched filter of the produced columns (k_rcmc_tile's pixel, on whole bins)
    {
        const int cw = tid & 63;
        const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int xc = x0 + cw;
        const ColConst cc = a.col[min(xc, a.nrv - 1)];
        const double m2 = 2.0 * (double)cc.m_dc;
        const int n = a.nbins, hb = a.half_bins;
        const bool wrap = 2 * hb >= n;  // a band of the whole PRF or more: the phase's offset wraps on its own
        float ws[16];  // signed window (-1)^i w[i]
#pragma unroll
        for (int i = 0; i < 16; ++i) ws[i] = (i & 1) ? -a.window[i] : a.window[i];
        constexpr int NR = (N2 + kAcWaves - 1) / kAcWaves;
        float2 res[NR];
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int m = wv + kAcWaves * i;
            if (m >= N2) break;
            const int k = k1 + a.n1 * m;
            const int kb = k < n / 2 ? k : k - n;  // signed bin
            int mn = kb > cc.alias_hi ? kb - n : kb;
            mn = kb < cc.alias_lo ? kb + n : mn;
            const int mo = mn - cc.m_dc;  // bins from the quantised centroid
            float2 val = make_float2(0.f, 0.f);
            // outside the azimuth band the matched filter zeroes the pixel: skip its interpolation
            if ((unsigned)(mo + hb) <= 2u * (unsigned)hb) {
                const double fn = (double)mn;
                const double shift = cc.shift_b2 * fn * fn;
                const double p = floor(shift + 0.5);  // round half away from zero: shift >= 0
                const int pi = (int)fmin(p, 4096.0);
                const int cx = xc + pi;
                if (!(cx - 8 < 0 || cx + 8 >= a.nrv)) {
                    const float d = (float)(shift - p);
                    // the tile width guarantees that the taps are staged; the clamp only keeps them inside the tile
                    const float2* tap = tl + m * kAcPitch + min(kAcLeft + cw + pi - 8, kAcCols - 15);
                    val = (d == 0.0f) ? tap[8] : sinc16_interior(tap, ws, d);
                }
                int mc = mo;
                if (wrap) {
                    mc = kb - cc.m_dc;
                    mc = 2 * mc > n ? mc - n : 2 * mc < -n ? mc + n : mc;
                }
                const double md = (double)mc;
                const double turns = cc.turns_b2 * fma(md, md, m2 * (double)kb);
                const float fr = (float)(turns - rint(turns));
                float sn, cs;
                sincos_turns(fr, &sn, &cs);
                val = make_float2(val.x * cs + val.y * sn, val.y * cs - val.x * sn);
            }
            res[i] = val;
        }
        __syncthreads();  // every tap is read before the produced columns are overwritten
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int m = wv + kAcWaves * i;
            if (m >= N2) break;
            tl[m * kAcPitch + kAcLeft + cw] = res[i];
        }
    }
    __syncthreads();

    // ---- 3. inverse pass B' of the produced columns, inverse inter-pass twiddle, store
    {
        const int ci = tid & 63, li = tid >> 6;  // 64 columns, 8 lanes each: the last four waves only reach the barriers
        const bool act = li < kAcLanes;
        float2* col = tl + kAcLeft + ci;
        if (act) {
            each_butterfly<R0>(li, [&](auto ic, int j, bool) __attribute__((always_inline)) {
#pragma unroll
                for (int r = 0; r < R1; ++r) v[decltype(ic)::value * R1 + r] = col[(j + r * R0) * kAcPitch];
            });
        }
        __syncthreads();  // every element of the column is read before the exchange overwrites it
        if (act) {
            each_butterfly<R0>(li, [&](auto ic, int j, bool valid) __attribute__((always_inline)) {
                float2* u = &v[decltype(ic)::value * R1];
                Dft<R1, true>::run(u);
                if (valid) {
#pragma unroll
                    for (int r = 0; r < R1; ++r) col[(j * R1 + r) * kAcPitch] = u[r];
                }
            });
        }
        __syncthreads();
        const int x = x0 + ci;
        const bool ok = act && ci < width && x < a.col1;
        if (act) {
            float2* out = a.out + row0 * a.stride;
            const unsigned stride = (unsigned)a.stride;
            each_butterfly<R1>(li, [&](auto, int j, bool valid) __attribute__((always_inline)) {
                float2 u[R0];
#pragma unroll
                for (int r = 0; r < R0; ++r) u[r] = col[(j + r * R1) * kAcPitch];
#pragma unroll
                for (int r = 1; r < R0; ++r) u[r] = cmulc(u[r], tw[j * R0 + r]);
                Dft<R0, true>::run(u);
                if (ok && valid) {
#pragma unroll
                    for (int r = 0; r < R0; ++r)
                        (out + (size_t)(r * R1) * stride)[(unsigned)j * stride + (unsigned)x] =
                            cmulc(u[r], tk[j + r * R1]);
                }
            });
        }
    }
}

size_t az_core_lds_bytes(int n2) { return sizeof(float2) * (size_t)(n2 * (kAcPitch + 2)); }

int az_core_tile_columns() { return kAcNarrow; }

int az_core_half_bins(double beta, int nbins) {
    return (int)std::floor(std::fmin(0.5 * beta, 1.0) * (double)nbins + 1e-9);
}

template <int N2, int R0, int R1>
static hipError_t core_launch(const AzCoreArgs& a, size_t lds, bool prepare, hipStream_t s) {
    if (prepare)
        return hipFuncSetAttribute((const void*)k_az_core<N2, R0, R1>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)lds);
    // enough workgroups for the narrower tiles, in whole rounds over the XCDs
    const long items = (long)a.n1 * ((a.col1 - a.col0 + kAcWide - 1) / kAcWide);
    hipLaunchKernelGGL((k_az_core<N2, R0, R1>), dim3((unsigned)((items + 7) / 8 * 8)), dim3(kAcThreads), lds, s, a);
    return hipGetLastError();
}

// Second-pass lengths with a compiled core and their radix sequences, in the planner's order of preference (the
// split of the azimuth FFT takes the first whose first-pass length has a compile-time column kernel). 84, 90, 96
// and 98 were measured on the production scenes; the others cover the azimuth lengths those four do not divide
// (powers of two, 3^a 5^b, ...). 63 and 49 come last, for the lengths that none of the others divides: azimuth passes
// of 3087 = 49 x 63 lines by 4912 columns 278 us with the separate kernels, 203 with the core; of 12005 = 245 x 49
// 1092 and 818. From 125 on the tile takes more than half a CU's LDS (one workgroup per CU).
#define ASARF_AZ_CORE_LENGTHS(X)                                                                                  \
    X(84, 12, 7) X(90, 9, 10) X(98, 7, 14) X(96, 8, 12) X(80, 10, 8) X(100, 10, 10) X(72, 9, 8) X(105, 15, 7)     \
    X(81, 9, 9) X(112, 16, 7) X(64, 8, 8) X(120, 12, 10) X(75, 15, 5) X(126, 14, 9) X(128, 16, 8) X(125, 25, 5)   \
    X(63, 9, 7) X(49, 7, 7)

bool az_core_supported(int n2) {
    switch (n2) {
#define ASARF_AZ_LABEL(N, ...) case N:
        ASARF_AZ_CORE_LENGTHS(ASARF_AZ_LABEL)
#undef ASARF_AZ_LABEL
            return true;
        default:
            return false;
    }
}

int az_core_lengths(int* out, int capacity) {
    static const int lengths[] = {
#define ASARF_AZ_ITEM(N, ...) N,
        ASARF_AZ_CORE_LENGTHS(ASARF_AZ_ITEM)
#undef ASARF_AZ_ITEM
    };
    const int n = (int)(sizeof(lengths) / sizeof(lengths[0]));
    for (int i = 0; i < n && i < capacity; ++i) out[i] = lengths[i];
    return n;
}

static hipError_t core_dispatch(const AzCoreArgs& a, int n2, bool prepare, hipStream_t s) {
    const size_t lds = az_core_lds_bytes(n2);
    if (lds > max_lds_bytes()) return hipErrorInvalidValue;
    switch (n2) {
#define ASARF_AZ_LAUNCH(N, ...) \
    case N: return core_launch<N, __VA_ARGS__>(a, lds, prepare, s);
        ASARF_AZ_CORE_LENGTHS(ASARF_AZ_LAUNCH)
#undef ASARF_AZ_LAUNCH
        default: return hipErrorInvalidValue;
    }
}

// Raises the kernel's dynamic LDS limit (once per plan, outside any graph capture).
hipError_t az_core_prepare(int n2) {
    AzCoreArgs a{};
    return core_dispatch(a, n2, true, nullptr);
}

hipError_t launch_az_core(const AzCoreArgs& a, int n2, hipStream_t s) {
    if (!a.in || !a.out || a.in == a.out || a.n1 <= 0 || a.col1 <= a.col0) return hipErrorInvalidValue;
    // the interpolation skips taps 0 and 15 (sinc16_interior): their window weights must be zero
    if (!(std::fabs(a.window[0]) < 1e-12f && std::fabs(a.window[15]) < 1e-12f)) return hipErrorInvalidValue;
    return core_dispatch(a, n2, false, s);
}

}  // namespace asarf
